"""Batched multi-particle sums (one persistent launch, HIP graph replay)
against the oracle summing the same explicit particles one by one.

Particles are drawn from the Gaussian beam with uneven trajectory windows;
three requests differ in grid size and energy count.  FP64 (tiled) must agree
to 1e-9 per point, mixed precision to 1e-5 (denominator floored at 1e-6 of
each request's maximum)."""
import numpy as np
import pytest

from tests.common import UNDULATOR, rel_err

gpu = pytest.mark.gpu


def scenario(n_particles=6, seed=11):
    from oscars_amd import multiparticle as M
    from oscars_amd import beam as B
    rng = np.random.Generator(np.random.PCG64(seed))
    beam = M.config_beam()
    parts = B.sample_particles(beam, n_particles, rng=rng)
    windows = M.uneven_windows(parts, rng, npts_range=(3001, 6001))
    obs_a = np.array([[0.0, 0.0, 30.0]])
    obs_b = np.array([[x, y, 30.0] for x in (-0.001, 0.0, 0.001) for y in (-0.0005, 0.0005)])
    obs_c = np.array([[0.0005, 0.0002, 20.0], [-0.0003, 0.0, 25.0]])
    reqs = [(obs_a, np.linspace(120.0, 900.0, 70)), (obs_b, np.linspace(140.0, 480.0, 64)),
            (obs_c, np.array([150.0, 151.0, 300.0, 455.5, 610.0]))]
    req_of, weights = M.assign_round_robin(n_particles, len(reqs))
    return parts, windows, reqs, req_of, weights


def oracle_sums(parts, windows, reqs, req_of, weights):
    from oracle.pyoracle import Oracle
    outs = [np.zeros((len(o), len(e))) for o, e in reqs]
    for p, (a, b, n), r, w in zip(parts, windows, req_of, weights):
        o = Oracle(nthreads=8)
        o.set_particle_beam(energy_GeV=3, x0=[0, 0, -1], d0=[0, 0, 1], current=0.5)
        o.add_bfield_undulator(**UNDULATOR)
        o.set_particle(p.x0, p.b0, 0.0)
        o.set_ctstartstop(a, b)
        o.set_npoints_trajectory(n)
        obs, e = reqs[r]
        for k, ob in enumerate(obs):
            v, lev, conv, ef = o.spectrum(ob, e, carry_quirk=False)
            assert conv.all()
            outs[r][k] += w * v
    return outs


@pytest.fixture(scope="module")
def batch_case():
    parts, windows, reqs, req_of, weights = scenario()
    ref = oracle_sums(parts, windows, reqs, req_of, weights)
    return parts, windows, reqs, req_of, weights, ref


@gpu
@pytest.mark.parametrize("mode,tol", [("tiled", 1e-9), ("mixed", 1e-5)])
def test_batched_flux_matches_oracle(batch_case, mode, tol):
    from oscars_amd import _lib
    from oscars_amd import multiparticle as M
    from oscars_amd.sr import sr
    parts, windows, reqs, req_of, weights, ref = batch_case
    s = sr()
    s.add_bfield_undulator(**UNDULATOR)
    dev = s._device()
    bf = M.BatchedFlux(dev, s._fields, parts, windows, reqs, req_of, weights, mode=mode)
    outs, st = bf.run(recompute_trajectories=False)
    assert st["n_unconverged"] == 0
    for r in range(len(reqs)):
        e = rel_err(outs[r], ref[r], 1e-6)
        print("%s request %d: max rel err %.3e" % (mode, r, e))
        assert e < tol
    # graph replay with trajectory recomputation gives the same sums
    outs2, st2 = bf.run(recompute_trajectories=True)
    outs3, st3 = bf.run(recompute_trajectories=True)
    for r in range(len(reqs)):
        assert rel_err(outs2[r], outs[r], 1e-6) < 1e-12
        assert rel_err(outs3[r], outs[r], 1e-6) < 1e-12
    assert st2["evals"] == st["evals"] == st3["evals"]


@gpu
def test_batch_tuner_keeps_results(batch_case):
    from oscars_amd import multiparticle as M
    from oscars_amd.sr import sr
    parts, windows, reqs, req_of, weights, ref = batch_case
    s = sr()
    s.add_bfield_undulator(**UNDULATOR)
    dev = s._device()
    bf = M.BatchedFlux(dev, s._fields, parts, windows, reqs, req_of, weights, mode="tiled")
    best, times = bf.tune(candidates=(1, 2, 4), sample_items=50)
    assert best in (1, 2, 4) and len(times) == 3
    outs, st = bf.run(recompute_trajectories=False)
    for r in range(len(reqs)):
        assert rel_err(outs[r], ref[r], 1e-6) < 1e-9


@gpu
@pytest.mark.parametrize("mode,tol", [("tiled", 1e-9), ("mixed", 1e-5)])
def test_batch_hand_over_tuner_keeps_results(batch_case, mode, tol):
    """The hand-over level tuner times every candidate on the whole launch and
    keeps the fastest; whichever it keeps, the sums stay within the bar."""
    from oscars_amd import multiparticle as M
    from oscars_amd.sr import sr
    parts, windows, reqs, req_of, weights, ref = batch_case
    s = sr()
    s.add_bfield_undulator(**UNDULATOR)
    dev = s._device()
    bf = M.BatchedFlux(dev, s._fields, parts, windows, reqs, req_of, weights, mode=mode)
    best, times = bf.tune_deep((0, 10, 12))
    print("%s hand-over tuner: %s -> %d" % (mode, times, best))
    assert best in (0, 10, 12) and len(times) == 3
    outs, st = bf.run(recompute_trajectories=False)
    assert st["n_unconverged"] == 0
    for r in range(len(reqs)):
        assert rel_err(outs[r], ref[r], 1e-6) < tol
    with pytest.raises(Exception):
        bf.tune_deep((5,))


@gpu
def test_sr_nparticles_batched_matches_particle_loop():
    """sr.calculate_spectrum(nparticles=N): the batched tiled path against the
    per-particle plain loop over the same sampled particles."""
    from oscars_amd.sr import sr
    from oscars_amd import multiparticle as M
    s = sr()
    b = M.config_beam()
    s.set_particle_beam(energy_GeV=3, x0=[0, 0, -1], d0=[0, 0, 1], current=0.5, sigma_energy_GeV=b["sigma_energy_GeV"],
                        beta=b["beta"], alpha=b["alpha"], emittance=b["emittance"])
    s.add_bfield_undulator(**UNDULATOR)
    s.set_ctstartstop(0, 2)
    s.set_npoints_trajectory(6001)
    s.set_seed(5)
    a = np.array([v for _, v in s.calculate_spectrum(obs=[0, 0, 30], energy_range_eV=[140, 600], npoints=100,
                                                      nparticles=5, mode="tiled")])
    s.set_seed(5)
    c = np.array([v for _, v in s.calculate_spectrum(obs=[0, 0, 30], energy_range_eV=[140, 600], npoints=100,
                                                      nparticles=5, mode="plain")])
    e = rel_err(a, c, 1e-6)
    print("batched vs loop: %.3e" % e)
    assert e < 1e-9


@gpu
@pytest.mark.parametrize("mode,tol", [("tiled", 1e-9), ("mixed", 1e-5)])
def test_batched_hand_over_matches_oracle(batch_case, mode, tol):
    """deep_level=10: every point still active at level 10 leaves its unit in a
    group and goes on level by level (and, mixed, its borderline points by the
    FP64 recheck kernel) instead of inside its unit.
    Same bar against the oracle, same evaluation count as the default."""
    from oscars_amd import multiparticle as M
    from oscars_amd.sr import sr
    parts, windows, reqs, req_of, weights, ref = batch_case
    s = sr()
    s.add_bfield_undulator(**UNDULATOR)
    dev = s._device()
    base = M.BatchedFlux(dev, s._fields, parts, windows, reqs, req_of, weights, mode=mode)
    _, st0 = base.run(recompute_trajectories=False)
    bf = M.BatchedFlux(dev, s._fields, parts, windows, reqs, req_of, weights, mode=mode, deep_level=10)
    outs, st = bf.run(recompute_trajectories=False)
    _, cnt, _ = dev.batch_profile(False)
    print("%s deep_level 10: handed over %d, listed for the recheck kernel %d, rechecked in unit %d"
          % (mode, cnt["handed_over"], cnt["fix_listed"], cnt["rechecked_in_unit"]))
    assert cnt["handed_over"] > 0
    assert st["evals"] == st0["evals"] and st["n_unconverged"] == 0
    for r in range(len(reqs)):
        e = rel_err(outs[r], ref[r], 1e-6)
        print("%s deep_level 10 request %d: max rel err %.3e" % (mode, r, e))
        assert e < tol


@gpu
@pytest.mark.parametrize("deep_level", [0, 10])
def test_batched_mixed_levels_match_fp64(deep_level):
    """Mixed batch against the FP64 batch on a denser case: identical levels
    (equal evaluation counts: borderline points are recomputed in FP64 inside
    the same graph, in their unit or, for points handed over at deep_level (0: at
    level 12 here), by the recheck kernel) and per-point agreement to 1e-5."""
    from oscars_amd import multiparticle as M
    from oscars_amd.sr import sr
    parts, windows, _, _, _ = scenario(n_particles=24, seed=7)
    grid = np.array([[x, y, 30.0] for x in np.linspace(-0.002, 0.002, 5) for y in np.linspace(-0.001, 0.001, 5)])
    reqs = [(grid, np.linspace(140.0, 600.0, 256)), (grid[::3], np.linspace(440.0, 470.0, 100))]
    req_of, weights = M.assign_round_robin(len(parts), len(reqs))
    s = sr()
    s.add_bfield_undulator(**UNDULATOR)
    dev = s._device()
    res = {}
    for mode in ("tiled", "mixed"):
        bf = M.BatchedFlux(dev, s._fields, parts, windows, reqs, req_of, weights, mode=mode, deep_level=deep_level)
        res[mode] = bf.run(recompute_trajectories=False)
    (o64, s64), (o32, s32) = res["tiled"], res["mixed"]
    errs = [rel_err(a, b, 1e-6) for a, b in zip(o32, o64)]
    print("mixed batch (deep level %d): evals %g (fp64 %g), points rechecked %d, max rel err %.3e"
          % (deep_level, s32["evals"], s64["evals"], s32["n_rechecked"], max(errs)))
    assert s32["evals"] == s64["evals"]
    assert max(errs) < 1e-5


@gpu
def test_hand_over_level_has_one_meaning(batch_case):
    """deep_level 0 is the rule's level and a negative one none, in the set-up and
    in the tuner, whose choice can be given back to the set-up."""
    from oscars_amd import multiparticle as M
    from oscars_amd.sr import sr
    parts, windows, reqs, req_of, weights, ref = batch_case
    s = sr()
    s.add_bfield_undulator(**UNDULATOR)
    dev = s._device()

    def handed(deep):
        bf = M.BatchedFlux(dev, s._fields, parts, windows, reqs, req_of, weights, mode="tiled", precision=1e-3,
                           deep_level=deep)
        return bf, dev.batch_profile(False)[1]["handed_over"]
    n = {deep: handed(deep)[1] for deep in (0, 12, -1, 27)}
    assert n[0] == n[12] > 0 and n[-1] == n[27] == 0
    bf, _ = handed(9)
    for deep in (0, 12, -1):
        best, times = bf.tune_deep((deep,))
        assert best == deep and list(times) == [deep]
        assert dev.batch_profile(False)[1]["handed_over"] == n[deep]
    for bad in (1, 8):
        with pytest.raises(Exception):
            bf.tune_deep((bad,))
        with pytest.raises(Exception):
            handed(bad)


@gpu
def test_batched_mixed_levels_in_their_unit():
    """As above with every point finished in its unit, its FP64 recheck included."""
    test_batched_mixed_levels_match_fp64(-1)


@gpu
def test_small_batch_takes_little_memory(batch_case):
    """The groups handed over and their partial sums are sized by what the batch
    can hand over, and are left out where nothing is handed over, until the tuner
    asks for a level: 70 + 384 + 10 points, 4.8 KB a group and 4 KB for each of its
    256 slices, once (tiled: 10 groups, 10 MB); beside them 17 MB of wave scratch,
    1 MB of rows and a margin of 16 MB for allocation in blocks."""
    import torch
    from oscars_amd import _lib
    from oscars_amd import multiparticle as M
    from oscars_amd.sr import sr
    parts, windows, reqs, req_of, weights, ref = batch_case
    s = sr()
    s.add_bfield_undulator(**UNDULATOR)
    parts, windows, req_of, weights = parts[:3], windows[:3], req_of[:3], weights[:3]
    for deep, most in ((-1, 34e6), (0, 45e6)):
        dev = _lib.Device(0)
        dev.trajectories(s._fields, M.om_particles(parts, windows))
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info(0)[0]
        dev.batch_setup(reqs, req_of, weights, [0.0] * 6, dev.conv(mode="tiled"), 1, 10, deep)
        used = free - torch.cuda.mem_get_info(0)[0]
        print("deep_level %d: %.1f MB" % (deep, used / 1e6))
        assert used < most
        first, _ = dev.batch_run(False)
        best, _ = dev.batch_tune_deep((9, 12))
        outs, st = dev.batch_run(False)
        assert st["n_unconverged"] == 0
        assert all(rel_err(a, b, 1e-6) < 1e-11 for a, b in zip(outs, first))
        assert dev.batch_profile(False)[1]["handed_over"] > 0 or best == 12


@gpu
@pytest.mark.parametrize("mode", ["tiled", "mixed"])
@pytest.mark.parametrize("groups", [4, 40, 1416])
def test_batch_groups_run_out(mode, groups):
    """Fewer groups than the units ask for at the hand-over level: those that find
    none keep their energies; and just enough for them (12 x 25 x 4 + 12 x 9 x 2),
    so that the points of the recomputation list go on in its kernel.  Equal evaluation counts and, over several replays, the same values as
    with everything left in its unit (the sums' order: 2^16 terms, 1e-11; mixed
    sums carry 4.8e-9 in their sines and cosines, 1e-6)."""
    from oscars_amd import multiparticle as M
    from oscars_amd.sr import sr
    parts, windows, _, _, _ = scenario(n_particles=24, seed=7)
    grid = np.array([[x, y, 30.0] for x in np.linspace(-0.002, 0.002, 5) for y in np.linspace(-0.001, 0.001, 5)])
    reqs = [(grid, np.linspace(140.0, 600.0, 256)), (grid[::3], np.linspace(440.0, 470.0, 100))]
    req_of, weights = M.assign_round_robin(len(parts), len(reqs))
    s = sr()
    s.add_bfield_undulator(**UNDULATOR)
    dev = s._device()

    def batch(deep, limit):
        dev.batch_limits(limit)
        try:
            return M.BatchedFlux(dev, s._fields, parts, windows, reqs, req_of, weights, mode=mode, deep_level=deep)
        finally:
            dev.batch_limits()
    ref, st = batch(-1, -1).run(recompute_trajectories=False)
    batch(9, -1)
    all_handed = dev.batch_profile(False)[1]["handed_over"]
    b = batch(9, groups)
    cnt = dev.batch_profile(False)[1]
    print("%s, %d groups: handed over %d of %d, listed for the recheck kernel %d, rechecked in unit %d"
          % (mode, groups, cnt["handed_over"], all_handed, cnt["fix_listed"], cnt["rechecked_in_unit"]))
    assert 0 < cnt["handed_over"] <= 64 * groups and (cnt["handed_over"] < all_handed) == (groups < 1416)
    assert cnt["fix_listed"] > 0 or mode == "tiled" or groups < 1416  # (which units find a group varies)
    for k in range(3):
        outs, st1 = b.run(recompute_trajectories=k == 2)
        assert st1["evals"] == st["evals"] and st1["n_unconverged"] == st["n_unconverged"] == 0
        assert all(rel_err(x, y, 1e-6) < (1e-11 if mode == "tiled" else 1e-6) for x, y in zip(outs, ref))
