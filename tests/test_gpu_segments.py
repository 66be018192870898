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


@gpu
def test_strong_fields_settle():
    """Chains that take more rounds than an ordinary one has: 3 GeV in a 10 T
    wiggler and 100 MeV in 0.3 T, with points for 60 and 96 rounds.  Equal to the
    integration in order as above."""
    from oscars_amd.sr import sr
    more = 0
    for energy, b, period, n_periods in ((3.0, 10.0, 0.5, 3), (0.1, 0.3, 0.049, 31)):
        s = sr()
        s.set_particle_beam(energy_GeV=energy, x0=[1e-5, 0, -1], d0=[1e-5, 2e-5, 1], current=0.5)
        s.add_bfield_undulator(bfield=[0, b, 0], period=[0, 0, period], nperiods=n_periods)
        dev = s._device()
        for npoints in (8001, 12001, 40001, 60001):
            part = s._om_particle(s._particle, ctstart=0, ctstop=2.0, npoints=npoints)
            dev.trajectory_limits(rounds=0)
            dev.trajectories(s._fields, [part])
            t, p = knots(dev, 0)
            dev.trajectory_limits()
            dev.trajectories(s._fields, [part])
            t1, p1 = knots(dev, 0)
            rounds = dev.trajectory_rounds(0)
            print("%g GeV, %g T, %d points: %d rounds" % (energy, b, npoints, rounds[0]))
            more += rounds[0] > 32
            assert np.array_equal(t1, t) and np.max(np.abs(p1[:, 2] - p[:, 2])) < 1e-19
            assert np.array_equal(p1[:, 5], p[:, 5]) and np.max(np.abs(p1[:, :2] - p[:, :2])) < 2e-15
    assert more > 0


def knots(dev, i):
    return dev.trajectory(i)[:2]


@gpu
@pytest.mark.parametrize("limits", [dict(rounds=0), dict(rounds=3), dict(polls=0)])
def test_chains_given_up_are_integrated_in_order(limits):
    """No chain cut, none settled after three rounds, and workgroups that do not
    wait for each other (so that every chain of more than one gives up): the
    integration in order takes over, in every bit.  The last particle's backward
    chain is one workgroup, accepted while its forward one is given up; and the
    next integration, with the default limits, is in segments again."""
    s, z0 = scene("planar")
    dev = s._device()
    parts = electrons(s, z0, 4, 6001, 2.0, 8)
    parts[2].ctstart = -1.0
    parts[3].ctstart = -0.1
    try:
        dev.trajectories(s._fields, [parts[i % 4] for i in range(520)])
        order = [knots(dev, i) for i in range(4)]
        assert [dev.trajectory_rounds(i) for i in range(4)] == [(0, 0)] * 4
        for k in range(2):
            dev.trajectory_limits(**limits)
            dev.trajectories(s._fields, parts)
            assert [dev.trajectory_rounds(i) for i in range(4)] == [(0, 0)] * 4
            for i, (t, p) in enumerate(order):
                t1, p1 = knots(dev, i)
                assert np.array_equal(t1, t) and np.array_equal(p1, p)
            dev.trajectory_limits()
            dev.trajectories(s._fields, parts)
            assert all(dev.trajectory_rounds(i)[0] > 3 for i in range(4))
            assert [dev.trajectory_rounds(i)[1] > 0 for i in range(4)] == [False, False, True, True]
            for i, (t, p) in enumerate(order):
                assert np.array_equal(knots(dev, i)[1][:, 2], p[:, 2])
    finally:
        dev.trajectory_limits()
    with pytest.raises(Exception):
        dev.trajectory_limits(rounds=97)


@gpu
def test_chains_given_up_in_a_replayed_graph():
    """A batch's graph integrates its particles in every replay: given up in each,
    and then, captured again with the default limits, in segments in each.  The
    sums agree to rounding with every replay."""
    from oscars_amd import multiparticle as M
    s, z0 = scene("planar")
    dev = s._device()
    parts = electrons(s, z0, 3, 6001, 2.0, 9)
    reqs = [(np.array([[0.0, 0.0, 30.0], [2e-4, 1e-4, 30.0]]), np.linspace(140.0, 300.0, 40))]

    class Held(M.BatchedFlux):
        def __init__(self):
            self.dev = dev
            dev.trajectories(s._fields, parts)
            dev.batch_setup(reqs, [0, 0, 0], [1.0, 1.0, 1.0], [0.0] * 6, dev.conv(mode="tiled"))
    b = Held()
    try:
        first = b.run(recompute_trajectories=False)[0][0]
        for limits, cut in ((dict(polls=0), False), ({}, True), (dict(rounds=2), False), ({}, True)):
            dev.trajectory_limits(**limits)
            for _ in range(3):
                out = b.run(recompute_trajectories=True)[0][0]
                assert [dev.trajectory_rounds(i)[0] > 0 for i in range(3)] == [cut] * 3
                assert np.max(np.abs(out - first)) < 1e-12 * np.max(first)
    finally:
        dev.trajectory_limits()


@gpu
@pytest.mark.parametrize("backward", [False, True])
def test_halved_steps_are_never_in_segments(backward):
    """A particle whose steps meet |beta| >= 1 and are halved, among 2000 steps,
    beside one that flies away from the field: the first is integrated in order,
    the second in segments, and both are the oracle's in every bit (a uniform
    box: no transcendental function enters)."""
    from oracle.pyoracle import Oracle
    from oscars_amd.sr import sr
    sign = -1.0 if backward else 1.0

    def setup(x, z0):
        x.set_particle_beam(energy_GeV=3, x0=[0, 0, z0], d0=[0, 0, 1], current=0.5)
        x.add_bfield_uniform(bfield=[0.5, 10.0, 0], width=[0, 0, 20.0], translation=[0, 0, 0])
        x.set_ctstartstop(-10000 if backward else 0, 0.0 if backward else 10000)
        x.set_npoints_trajectory(2001)
    s, away = sr(), sr()
    setup(s, -15 * sign)
    setup(away, 15 * sign)
    dev = s._device()
    dev.trajectories(s._fields, [s._om_particle(s._particle), away._om_particle(away._particle)])
    rounds = [dev.trajectory_rounds(i) for i in range(2)]
    assert rounds[0] == (0, 0) and rounds[1][1 if backward else 0] > 0
    for i, z0 in enumerate((-15 * sign, 15 * sign)):
        o = Oracle(nthreads=1)
        setup(o, z0)
        T = o.calculate_trajectory()
        assert (o.halvings()[0] > 0) == (i == 0)
        t, p = knots(dev, i)
        assert np.array_equal(t, T.t) and np.array_equal(p, T.p), i
