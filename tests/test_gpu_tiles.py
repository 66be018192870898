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
