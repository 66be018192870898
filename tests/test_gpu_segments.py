"""Trajectories in segments against the same particles integrated in order on
the device: equal in every bit where a photon's phase depends on the last bit."""
import numpy as np
import pytest

gpu = pytest.mark.gpu


def scene(field):
    from oscars_amd.sr import sr
    from tests.common import EPU, UNDULATOR
    s = sr()
    z0 = -1.5 if field == "epu" else -1.0
    s.set_particle_beam(energy_GeV=3, x0=[0, 0, z0], d0=[0, 0, 1], current=0.5)
    if field == "epu":
        s.add_bfield_epu(**EPU)
    else:
        s.add_bfield_undulator(**UNDULATOR)
    if field == "pair":
        s.add_bfield_gaussian(bfield=[0.02, 0, 0], sigma=[0, 0, 0.2], translation=[0, 0, 0.3])
    return s, z0


def electrons(s, z0, n, npoints, span, seed):
    """Electrons of a beam: a little off the axis, in angle and in energy."""
    from oscars_amd import geometry as G
    r = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        g = 3.0 * (1 + 9e-4 * r.standard_normal()) / (1e-9 * 9.10938356e-31 * G.C ** 2 / 1.602176462e-19)
        b = np.sqrt(1 - 1 / g ** 2)
        ax, ay = 2.5e-5 * r.standard_normal(), 3e-6 * r.standard_normal()
        s.set_particle([3.7e-5 * r.standard_normal(), 2.5e-6 * r.standard_normal(), z0],
                       [b * np.sin(ax), b * np.sin(ay), b * np.sqrt(1 - np.sin(ax) ** 2 - np.sin(ay) ** 2)])
        out.append(s._om_particle(s._particle, ctstart=0, ctstop=span, npoints=npoints))
    return out


@gpu
@pytest.mark.parametrize("field,npoints,span", [("epu", 40001, 3.0), ("pair", 8001, 2.0), ("planar", 4001, 2.0)])
def test_accepted_joins_are_exact_along(field, npoints, span):
    """More particles in a call than are cut into segments (512 of a length) are
    integrated in order; the first 40 of them again, each alone.  z and beta_z in
    every bit, however many rounds a chain took to settle; across, a join may be
    off by 2^-62 c or 2^-51 of the velocity itself (6.5e-11 m/s, over at most
    1e-8 s), at most 1700 joins: 2e-15 m."""
    s, z0 = scene(field)
    dev = s._device()
    parts = electrons(s, z0, 40, npoints, span, 4)
    dev.trajectories(s._fields, parts + [parts[0]] * 490)
    order = [dev.trajectory(i)[:2] for i in range(len(parts))]
    in_order = [dev.trajectory_rounds(i) for i in (0, 39, 529)]
    rounds = []
    for part, (t, p) in zip(parts, order):
        dev.trajectories(s._fields, [part])
        t1, p1, _ = dev.trajectory(0)
        assert np.array_equal(t1, t)
        assert np.array_equal(p1[:, 2], p[:, 2]) and np.array_equal(p1[:, 5], p[:, 5])
        assert np.max(np.abs(p1[:, :2] - p[:, :2])) < 2e-15
        rounds.append(dev.trajectory_rounds(0))
    print("%s: %s rounds" % (field, sorted(r[0] for r in rounds)))
    assert in_order == [(0, 0)] * 3 and all(r[0] > 1 and r[1] == 0 for r in rounds)
