"""The kernels' tilings at the sizes where they change or end: results at the
edges of a tile, at remainders, and on both sides of every size rule, against
the oracle and against the same points in calls of another size."""
import numpy as np
import pytest

from tests.common import epu, planar, rel_err

gpu = pytest.mark.gpu


@pytest.fixture(scope="module")
def epu_pair():
    from oracle.pyoracle import Oracle
    from oscars_amd.sr import sr
    o, s = Oracle(nthreads=8), sr()
    for x in (o, s):
        epu(x, 8001)
        x.calculate_trajectory()
    return o, s._device()


def _scatter(n, half, z, seed=5):
    r = np.random.default_rng(seed)
    return np.column_stack([r.uniform(-half, half, (n, 2)), np.full(n, z)])


@gpu
@pytest.mark.parametrize("n", [1, 2, 63, 65, 4096, 4097, 32767, 32769, 32775])
def test_power_density_sizes(epu_pair, n):
    """One, two and eight points per wave (up to 4096, 32768 and beyond), with
    remainders.  Against the oracle to 1e-9 (1 - N.B = 1e-8 carries 1e-8 of
    rounding per sample; measured 1e-13), levels identical; the variants' sums
    differ in their order only: 2^13 terms, 2^13 u = 1e-12."""
    o, dev = epu_pair
    obs = _scatter(n, 0.03, 20.0)
    nrm = np.random.default_rng(6).normal(size=(n, 3)) * 0.2 + [0, 0, 1]
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    conv = dev.conv(precision=1e-4)  # several levels by lists of the points still running
    v, lev, cv, _ = dev.power_density_surface(0, obs, nrm, 1, conv)
    vm, levm, cvm, _ = dev.power_density_surface(0, obs, nrm, 1, dev.conv(precision=1e-4, mode="mixed"))
    k = np.unique(np.linspace(0, n - 1, 9).astype(int))
    ov, olev, _ = o.power_density_surface(obs[k], nrm[k], directional=True, precision=1e-4, carry_quirk=False)
    assert np.array_equal(lev[k], olev) and rel_err(v[k], ov, 1e-6) < 1e-9
    few, fewlev, _, _ = dev.power_density_surface(0, obs[-5:], nrm[-5:], 1, conv)
    assert np.array_equal(lev[-5:], fewlev) and rel_err(v[-5:], few) < 1e-12
    assert np.array_equal(lev, levm) and np.array_equal(cv, cvm)
    assert rel_err(vm, v, 1e-6) < 1e-5


@gpu
@pytest.mark.parametrize("z", [1e120, 1e153, 2e154, 1e160, 1e300])
def test_power_density_far_away(epu_pair, z):
    """Points so far that |R|^2 is near the largest double or overflows: the
    oracle's value (0 where it overflows, as the term is divided by infinity) and
    its level, in a few points and in as many as take several to a wave."""
    o, dev = epu_pair
    obs = np.column_stack([np.zeros((5000, 2)), np.full(5000, z)])
    obs[:, 0] = 1e-3 * z * np.linspace(-1, 1, 5000)
    ov, olev, oconv = o.power_density_surface(obs[:2], np.array([[0, 0, 1.0]] * 2), directional=True, precision=0.01,
                                              carry_quirk=False)
    for n in (2, 5000):
        v, lev, cv, _ = dev.power_density(0, obs[:n], [0.0, 0.0, 1.0], True, dev.conv(precision=0.01))
        assert np.isfinite(v).all() and np.allclose(v[:2], ov, rtol=1e-9, atol=0)
        assert np.array_equal(lev[:2], olev) and np.array_equal(cv[:2], np.asarray(oconv, dtype=cv.dtype))


def _field(x, name):
    from tests.common import EPU, UNDULATOR
    if name == "epu":
        x.add_bfield_epu(**EPU)
    elif name == "map":
        from oscars_amd import adjoint as A
        x.add_bfield_grid([0, 0, -1.0], [0, 0, 5e-4], [1, 1, 4001], A.undulator_pole_map(4001, -1.0, 5e-4))
    else:
        bf = dict(x=[1, 0, 0], xy=[0.5, 1, 0], tapered=[0, 1, 0], pair=[0, 1, 0]).get(name, [0, 1, 0])
        x.add_bfield_undulator(**dict(UNDULATOR, bfield=bf), **(dict(taper=0.05) if name == "tapered" else {}))
        if name == "pair":
            x.add_bfield_gaussian(bfield=[0.05, 0, 0], sigma=[0, 0, 0.2], translation=[0, 0, 0.3])


@gpu
@pytest.mark.parametrize("field", ["y", "x", "xy", "tapered", "epu", "map", "pair"])
def test_trajectory_in_segments(field):
    """Chains cut into segments and joined, one to 53 workgroups long, with
    remainders, T0 at the start, inside and at the end of the window, beside
    chains of one step; every one accepted, none left to the integration in order.
    Against the oracle's integration in order: times equal; positions
    along the trajectory within two units in the last place of 1 m (2^-52: the
    joins agree to a fraction of one), transverse ones and velocities to 1e-12 of
    their largest value (the device's sine differs from the C library's in the
    last bit; with integration in order on the device the bar is the same)."""
    from oracle.pyoracle import Oracle
    from oscars_amd.sr import sr
    windows = [(0, 2, 20001), (0, 0.15, 1500), (0, 0.1500001, 1502), (0, 0.3841, 3842), (-1, 1, 20001),
               (-0.7, 0.1, 8002), (-1, 0, 6000), (0, 1.3, 1701)]

    def setup(x):
        x.set_particle_beam(energy_GeV=3, x0=[1e-5, 0, -0.6], d0=[1e-5, 2e-5, 1], current=0.5)
        _field(x, field)

    s = sr()
    setup(s)
    dev = s._device()
    dev.trajectories(s._fields, [s._om_particle(s._particle, ctstart=a, ctstop=b, npoints=n) for a, b, n in windows])
    for i, (a, b, n) in enumerate(windows):
        o = Oracle(nthreads=1)
        setup(o)
        o.set_ctstartstop(a, b)
        o.set_npoints_trajectory(n)
        T = o.calculate_trajectory()
        t, p, _ = dev.trajectory(i)
        rounds = dev.trajectory_rounds(i)
        assert rounds[0] > 0 and (rounds[1] > 0) == (a < 0), (a, b, n, rounds)
        scale = np.max(np.abs(T.p), axis=0)
        scale[scale == 0] = 1
        err = np.max(np.abs(p - T.p) / scale, axis=0)
        assert np.array_equal(t, T.t), (a, b, n)
        assert np.max(np.abs(p[:, 2] - T.p[:, 2])) <= 2.0 ** -52 and np.max(err) < 1e-12, (a, b, n, err)


@gpu
def test_many_trajectories_in_segments():
    """More chains than workgroups are given out to: one workgroup a chain, no
    waiting between them.  The same particles in one call and alone (53
    workgroups): z within two units in the last place of 1 m, the rest to 1e-12
    of its largest value."""
    from oscars_amd.sr import sr
    from tests.common import UNDULATOR
    s = sr()
    s.set_particle_beam(energy_GeV=3, x0=[0, 0, -1], d0=[0, 0, 1], current=0.5)
    s.add_bfield_undulator(**UNDULATOR)
    r = np.random.default_rng(3)
    parts = []
    for i in range(150):
        s.set_particle([2e-5 * r.standard_normal(), 0, -1], [2e-5 * r.standard_normal(), 0, 0.99999998])
        parts.append(s._om_particle(s._particle, ctstart=-0.05, ctstop=1.9, npoints=int(r.integers(1600, 20001))))
    dev = s._device()
    dev.trajectories(s._fields, parts)
    many = [dev.trajectory(i) for i in (0, 74, 149)]
    assert all(min(dev.trajectory_rounds(i)) > 0 for i in range(150))
    for (t, p, _), i in zip(many, (0, 74, 149)):
        dev.trajectories(s._fields, [parts[i]])
        t1, p1, _ = dev.trajectory(0)
        scale = np.maximum(np.max(np.abs(p1), axis=0), 1e-300)
        assert np.array_equal(t, t1) and np.max(np.abs(p[:, 2] - p1[:, 2])) <= 2.0 ** -52
        assert np.max(np.abs(p - p1) / scale) < 1e-12


@gpu
@pytest.mark.parametrize("mode", ["tiled", "mixed"])
def test_batch_levels_handed_over(mode):
    """Energies handed over at level 9 in groups of 1, 63, 64, 64 + 1 and
    64 + 64 + 2, some to levels beyond the stored rows, against the same batch
    with no hand-over: equal evaluation counts (identical levels), and values to
    1e-11 (the order of up to 2^16 terms' sums: 2^16 u; 1e-6 for the mixed sums,
    whose sines and cosines carry 4.8e-9), over several replays of the graph."""
    from oscars_amd import multiparticle as M
    from oscars_amd.sr import sr
    from tests.common import UNDULATOR
    s = sr()
    s.add_bfield_undulator(**UNDULATOR)
    rng = np.random.default_rng(2)
    from oscars_amd import beam as B
    parts = B.sample_particles(M.config_beam(), 5, rng=rng)
    windows = M.uneven_windows(parts, rng, npts_range=(2001, 6001))
    grid = np.array([[x, 2e-4, 30.0] for x in (-3e-3, 0.0, 1e-3)])
    reqs = [(grid, np.linspace(150.0, 900.0, n)) for n in (1, 63, 64, 65, 130)]
    out = {}
    for deep in (27, 9):
        b = M.BatchedFlux(s._device(), s._fields, parts, windows, reqs, np.arange(5), np.ones(5), mode=mode,
                          precision=2e-3, level_cap=11, deep_level=deep)
        runs = [b.run(recompute_trajectories=k > 0) for k in range(3)]
        for o, st in runs[1:]:
            assert st["evals"] == runs[0][1]["evals"] and st["n_unconverged"] == 0
            assert all(rel_err(a, c) < 1e-12 for a, c in zip(o, runs[0][0]))
        out[deep] = runs[0]
        _, cnt, _ = s._device().batch_profile(False)
        assert (cnt["handed_over"] > 0) == (deep == 9)
    assert out[27][1]["evals"] == out[9][1]["evals"] > 323 * 3 * (2 ** 11 - 1)
    for a, c in zip(out[9][0], out[27][0]):
        assert rel_err(a, c, 1e-6) < (1e-11 if mode == "tiled" else 1e-6)


@gpu
@pytest.mark.parametrize("mode,tol", [("tiled", 1e-9), ("mixed", 1e-5), ("plain", 1e-9), ("point_mixed", 1e-5)])
@pytest.mark.parametrize("shape", [(1, 1), (1, 63), (1, 64), (1, 65), (3, 130), (41, 3), (512, 65), (1025, 64),
                                   (16384, 1), (16385, 1)])
def test_flux_request_shapes(epu_pair, mode, tol, shape):
    """Requests on both sides of the rules that choose the kernels (1024 groups of
    one observation point and 64 energies; 16384 points), with groups of 1, 63,
    64, 64 + 1 energies.  Three observation points against the plain path's values
    in a call of their own, levels identical, and against the oracle (1e-9 in FP64; 1e-5 mixed, whose sines and cosines carry
    4.8e-9)."""
    o, dev = epu_pair
    n_obs, n_e = shape
    obs = _scatter(n_obs, 0.002, 20.0, seed=n_obs)
    e = np.linspace(120.0, 700.0, n_e)
    conv = dev.conv(precision=5e-3, mode=mode)
    v, lev, cv, _, st = dev.flux(0, obs, e, [0.0] * 6, conv)
    assert cv.all() and st["n_unconverged"] == 0
    k = np.unique(np.array([0, n_obs // 2, n_obs - 1]))
    pv, plev, _, _, _ = dev.flux(0, obs[k], e, [0.0] * 6, dev.conv(precision=5e-3, mode="plain"))
    v, lev = v.reshape(n_obs, n_e)[k], lev.reshape(n_obs, n_e)[k]
    assert np.array_equal(lev.ravel(), plev) and rel_err(v.ravel(), pv, 1e-6) < tol
    je = np.unique(np.array([0, n_e // 2, n_e - 1]))
    for j in je:
        ov, olev, _, _ = o.flux_points(obs[k], float(e[j]), precision=5e-3, carry_quirk=False)
        assert np.array_equal(lev[:, j], olev) and rel_err(v[:, j], ov, 1e-6) < tol


@gpu
@pytest.mark.parametrize("mode,tol", [("tiled", 1e-9), ("mixed", 1e-5)])
@pytest.mark.parametrize("shape", [(1, 65), (5, 3)])
def test_flux_deep_levels(epu_pair, mode, tol, shape):
    """Small requests whose energies stop at levels 9 to 15, through the levels
    the host looks between: against the plain path's values (tolerances as
    above), levels identical."""
    o, dev = epu_pair
    n_obs, n_e = shape
    obs = _scatter(n_obs, 0.002, 20.0, seed=n_obs)
    e = np.linspace(400.0, 6000.0, n_e)
    kw = dict(precision=1e-6, max_level=15, max_level_extended=15)
    v, lev, cv, _, _ = dev.flux(0, obs, e, [0.0] * 6, dev.conv(mode=mode, **kw))
    pv, plev, pcv, _, _ = dev.flux(0, obs, e, [0.0] * 6, dev.conv(mode="plain", **kw))
    assert np.array_equal(lev, plev) and np.array_equal(cv, pcv) and lev.max() >= 14
    assert rel_err(v, pv, 1e-6) < tol


@gpu
@pytest.mark.parametrize("mode,tol", [("tiled", 1e-9), ("mixed", 1e-5)])
@pytest.mark.parametrize("n_obs,n_e,far", [(1024, 64, [0.02]), (1000, 3, [0.015, 0.03]), (97, 650, [0.02, 0.02]),
                                           (1, 65, [0.02])])
def test_flux_stragglers(epu_pair, mode, tol, n_obs, n_e, far):
    """Requests of up to 1024 groups of which one or two observation points go on
    beyond level 13, through the tiles listed for them: whole ones, remainders,
    and energies packed across a point's groups.  Against the plain path's values
    in a call of their own (tolerances as above), levels identical."""
    o, dev = epu_pair
    obs = _scatter(n_obs, 0.0005, 20.0, seed=n_obs)
    at = np.linspace(0, n_obs - 1, len(far) + 2).astype(int)[1:-1]
    obs[at, 0] = far
    e = np.linspace(600.0, 3000.0, n_e)
    kw = dict(precision=3e-3, max_level=16, max_level_extended=16)
    v, lev, cv, _, _ = dev.flux(0, obs, e, [0.0] * 6, dev.conv(mode=mode, **kw))
    v, lev, cv = (x.reshape(n_obs, n_e) for x in (v, lev, cv))
    assert np.all(lev[at].max(axis=1) > 13)
    k = np.unique(np.concatenate([at, [0, n_obs - 1]]))
    pv, plev, pcv, _, _ = dev.flux(0, obs[k], e, [0.0] * 6, dev.conv(mode="plain", **kw))
    pv, plev, pcv = (x.reshape(len(k), n_e) for x in (pv, plev, pcv))
    assert np.array_equal(lev[k], plev) and np.array_equal(cv[k], pcv)
    assert all(rel_err(v[i], pv[j], 1e-6) < tol for j, i in enumerate(k))


@gpu
@pytest.mark.parametrize("level", [0, 1, 2, 7, 8, 9, 10])
def test_power_density_stl_caps(tmp_path, level):
    """Levels on both sides of the first ones summed as one (0..8), down to
    levels of fewer samples than the waves that share them: the oracle on the
    device's own trajectory takes the same occlusion decisions, values to 1e-12
    (sums of at most 2047 positive terms in another order), and levels where they
    stopped before the cap."""
    from oracle.pyoracle import Trajectory
    from oscars_amd import io as IO
    from tests.common import stl_scene
    from tests.test_gpu_power import _pair
    scene = stl_scene(str(tmp_path))
    o, s = _pair(planar, 2001)
    for k, (path, scale, tr) in enumerate(scene):
        s.add_stl(path, scale=scale, translation=tr, name="s%d" % k)
    v = np.array([r[1] for r in s.calculate_power_density_stl(max_level=level)])
    tri = np.concatenate([IO.read_stl(p, sc, t) for p, sc, t in scene])
    o.traj = Trajectory(*s._device().trajectory(0))
    ov, olev, oconv = o.power_density_stl(tri, max_level=level, carry_quirk=False)
    done = np.asarray(oconv, dtype=bool)
    assert np.array_equal(np.asarray(s._last_conv, dtype=bool), done)
    assert np.array_equal(s._last_levels[done], olev[done]) and rel_err(v, ov, 1e-6) < 1e-12


@gpu
@pytest.mark.parametrize("npts", [66, 127, 2049, 8194])
def test_adjoint_segments(npts):
    """Reverse passes of fewer segments than the chain has groups, of about one
    a group, and of the most there are (2048) with a short last one: the angle
    gradients against 4th-order differences of the long-double forward (1e-4, as
    at 4001 points)."""
    from oracle.pyoracle import fdref_flux
    from oscars_amd import _lib
    from oscars_amd import adjoint as A
    from oscars_amd import geometry as G
    n, z0, dz = 1001, -0.4, 8e-4
    samples = np.zeros((n, 3))
    z = z0 + dz * np.arange(n)
    samples[:, 1] = 0.05 * np.sin(2 * np.pi * z / 0.2) * np.exp(-(z / 0.2) ** 2)
    obs = np.array([[0.001, 0.0005, 30.0], [-0.0007, 0.001, 30.0]])
    e = np.array([20.0, 31.0])
    prob = A.FieldMapProblem(_lib.Device(0), [0, 0, z0], [0, 0, dz], [1, 1, n], 3.0, [0, 0, -0.5], 0.0, 1.0, npts, obs,
                             e, 10)
    prob.forward(samples, (0.0, 0.0))
    w = np.array([[1.0, -0.4], [0.7, 0.2]])
    _, ga, _ = prob.backward(w)
    p0 = G.ideal_particle("electron", 3.0, [0, 0, -0.5], [0, 0, 1], 0.0, 0.5)

    def loss(ang):
        b0, _, _ = A.beta0_from_angles(p0.b0, ang[0], ang[1])
        return float(np.sum(w * fdref_flux(samples, z0, dz, [0, 0, -0.5], b0, 0.5, 0.0, 1.0, npts, obs, e, 10,
                                           long_double=True)))
    for k in range(2):
        def at(d):
            return loss([d if j == k else 0.0 for j in range(2)])
        fd = (-at(2e-7) + 8 * at(1e-7) - 8 * at(-1e-7) + at(-2e-7)) / 1.2e-6
        print("npts %d angle %d: adjoint %.10e differences %.10e" % (npts, k, ga[k], fd))
        assert abs(ga[k] - fd) < 1e-4 * abs(fd)


@gpu
@pytest.mark.parametrize("mode", ["plain", "tiled"])
def test_level_rows_of_many_particles(mode):
    """Of more than 2048 particles a sum keeps the level rows it needs, here to level
    9 or 10 of most (1023 or 2047 rows of 80 bytes; 250 KB a particle on average
    with the deeper ones and the allocations rounded up), and not 1.3 MB.  The
    same sums as of a particle alone, whose levels to 13 are summed before the
    host looks (the same additions, so equal but for the sums of slices: 1e-12)."""
    import torch
    from oscars_amd import _lib
    from oscars_amd.sr import sr
    from tests.common import UNDULATOR
    s = sr()
    s.set_particle_beam(energy_GeV=3, x0=[0, 0, -0.1], d0=[0, 0, 1], current=0.5)
    s.add_bfield_undulator(**UNDULATOR)
    r = np.random.default_rng(1)
    parts = []
    for i in range(2100):
        s.set_particle([1e-5 * r.standard_normal(), 0, -0.1], [2e-5 * r.standard_normal(), 0, 0.99999998])
        parts.append(s._om_particle(s._particle, ctstart=0, ctstop=0.2, npoints=301))
    obs, e = np.array([[1e-4, 0.0, 30.0]]), np.linspace(100.0, 400.0, 3)
    dev, one = _lib.Device(0), _lib.Device(0)
    dev.trajectories(s._fields, parts)
    conv = dev.conv(precision=0.05, mode=mode)
    dev.flux(0, obs, e, [0.0] * 6, conv)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info(0)[0]
    res = [dev.flux(i, obs, e, [0.0] * 6, conv) for i in range(2100)]
    used = free - torch.cuda.mem_get_info(0)[0]
    print("%s: %.0f KB a particle" % (mode, used / 2099e3))
    assert np.median([x[1].max() for x in res]) <= 10 and used < 2100 * 500e3
    for i in (0, 1049, 2099):
        one.trajectories(s._fields, [parts[i]])
        v, lev, cv, _, _ = one.flux(0, obs, e, [0.0] * 6, conv)
        assert np.array_equal(lev, res[i][1]) and np.array_equal(cv, res[i][2]) and rel_err(res[i][0], v) < 1e-12


def _spline(t, y):
    """Second derivatives of the clamped spline (include/TOMATH.h:141-203), the
    sweep in order, in the device's order of operations."""
    n = len(t)
    sig = (t[1:-1] - t[:-2]) / (t[2:] - t[:-2])
    w = ((y[2:] - y[1:-1]) / (t[2:] - t[1:-1])[:, None] - (y[1:-1] - y[:-2]) / (t[1:-1] - t[:-2])[:, None])
    w = w * 6. / (t[2:] - t[:-2])[:, None]
    pv, u, out = np.full(n, -0.5), np.zeros_like(y), np.zeros_like(y)
    for i in range(1, n - 1):
        p = sig[i - 1] * pv[i - 1] + 2.0
        pv[i] = (sig[i - 1] - 1.) / p
        u[i] = (w[i - 1] - sig[i - 1] * u[i - 1]) / p
    out[n - 1] = (0.0 - u[n - 2] * 0.5) / (pv[n - 2] * 0.5 + 1.)
    for i in range(n - 2, -1, -1):
        out[i] = pv[i] * out[i + 1] + u[i]
    return out


@gpu
@pytest.mark.parametrize("total,run", [(7000, 1), (14000, 2), (28000, 4), (240000, 32)])
def test_spline_runs(total, run):
    """The splines of many particles, whose knots a lane takes in runs of 1 to 32:
    runs that end inside a particle and go on in the next, or hold several whole
    ones, and particles of 3 knots up to many runs.  Against the sweep in order:
    the run-ups of 64 knots leave 0.27^64 = 4e-37 of a channel's scale, so that
    only entries of that size and their roundings differ (1e-19 of the scale)."""
    from oscars_amd.sr import sr
    s = sr()
    planar(s, 301)
    lengths = [3, 4, 5, 31, 32, 33, 63, 64, 65, 66, 129, 301, 3, 3, 1400, 34]
    while sum(lengths) < total - 1400:
        lengths.append(lengths[(len(lengths) * 7) % 16])
    assert min(32, -(-9 * sum(lengths) // 65536)) == run
    r = np.random.default_rng(total)
    parts = []
    for n in lengths:
        s.set_particle([1e-5 * r.standard_normal(), 0, -1], [2e-5 * r.standard_normal(), 1e-5, 0.9999999])
        parts.append(s._om_particle(s._particle, ctstart=0, ctstop=2.0, npoints=n))
    dev = s._device()
    dev.trajectories(s._fields, parts)
    n_knots = 0
    for i in list(range(min(48, len(parts)))) + [len(parts) - 1]:
        t, p, ypp = dev.trajectory(i)
        ref = _spline(t, p)
        n_knots += len(t)
        assert np.all(np.abs(ypp - ref) <= 1e-19 * np.abs(ref).max(axis=0)), (i, len(t))
    print("%d particles, %d knots, %d compared" % (len(parts), sum(lengths), n_knots))
