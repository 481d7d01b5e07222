"""Critical stretches down to the rounding of a length: which bonds break is
exactly what the oracle's rounded stretch says, also where an ulp of a length
is not small against the threshold."""
import numpy as np
import pytest

import oracle
from probabilistic_peridynamics_amd import _lib, configs
from probabilistic_peridynamics_amd import integrators as it

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    try:
        ok = _lib.device_count() > 0
    except OSError:
        ok = False
    if not ok:
        pytest.fail("no HIP device: the gpu tests need an MI355X")


@pytest.mark.parametrize("tension", [False, True])
@pytest.mark.parametrize("s0", [1e-16, 3e-15, 1e-12, 1e-8])
def test_small_critical_stretches(s0, tension):
    w = configs.beam_vv(shape=(13, 7, 6))
    n, k = w.nlist.shape
    rng = np.random.default_rng(2)
    u = rng.normal(scale=s0 * w.extra["dx"], size=(n, 3))
    zeros = np.zeros_like(w.bc_types)
    integ = it.EulerHIP(2e-15)
    integ.build(n, 3, k, w.coords, w.volume, w.family, zeros, w.bc_values,
                zeros, w.force_bc_values, None, None, None)
    integ.set_break_mode(tension)
    integ.create_buffers(w.nlist, w.n_neigh, w.bond_stiffness, s0, None, u,
                         None, None, None, None, None, None, 1, 1)
    integ(0.0, 0.0)
    got = integ.write(None, None, None, None, None, None, None, None)
    want = w.nlist.copy()
    for i, row in enumerate(w.nlist):
        for c, j in enumerate(row):
            if j < 0:
                continue
            s = oracle.cl_strain(u[i], u[j], w.coords[i], w.coords[j])[0]
            if not ((s if tension else abs(s)) < s0):
                want[i, c] = -1
    broken = int((w.nlist >= 0).sum() - (want >= 0).sum())
    assert 0 < broken < (w.nlist >= 0).sum()
    np.testing.assert_array_equal(got[6], want)
