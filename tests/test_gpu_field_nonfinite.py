"""A node without live bonds feels no force whatever its stiffness: with c_i
infinite or NaN its empty and broken slots add nothing, in both break modes
and with corrections, and the rest of the body steps as without that node."""
import numpy as np
import pytest

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


@pytest.mark.parametrize("corrected", [False, True])
@pytest.mark.parametrize("tension", [False, True])
@pytest.mark.parametrize("c_alone", [np.inf, -np.inf, np.nan])
def test_nodes_without_bonds(c_alone, tension, corrected):
    w = configs.beam_vv(shape=(13, 6, 5))
    n, k = w.nlist.shape
    alone = np.array([3, 140, n - 1])
    rng = np.random.default_rng(6)
    nl = np.where(np.isin(w.nlist, alone), -1, w.nlist)
    nl[alone] = -1
    nn = (nl >= 0).sum(axis=1).astype(np.int32)
    u = rng.normal(scale=2e-3 * w.extra["dx"], size=(n, 3))
    corr = rng.uniform(0.5, 2.0, (n, k)) if corrected else None
    out = []
    for c in (1.0, c_alone):
        field = w.bond_stiffness * np.random.default_rng(3).uniform(0.5, 2, n)
        field[alone] = c
        integ = it.EulerHIP(2e-15)
        integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                    w.bc_values, np.zeros_like(w.force_bc_types),
                    w.force_bc_values, corr, None, None)
        integ.set_node_stiffness(field)
        integ.set_break_mode(tension)
        integ.create_buffers(nl, nn, w.bond_stiffness, w.critical_stretch,
                             None, u, None, None, None, None, None, None, 1,
                             1)
        integ.run(4, np.full(4, 1e-6), np.ones(4))
        out.append(integ.write(None, None, None, None, None, None, None,
                               None))
    assert np.all(out[1][3][alone] == 0.0)
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
