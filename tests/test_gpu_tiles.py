"""Meshes of one to six tiles per CU, on both sides of each limit: the tiles
are an even number per CU, with and without groups, and the state after a few
steps is bitwise that of other tiles, in the slot layout and in the exact
order."""
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


def _run(w, exact, tile, group):
    n, k = w.nlist.shape
    integ = it.Euler(2e-15) if exact else it.EulerHIP(2e-15)
    integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                w.bc_values, w.force_bc_types, w.force_bc_values, None, None,
                None)
    integ.set_launch(4, tile)
    integ.set_groups(group)
    u = np.random.default_rng(4).normal(scale=2e-3 * w.extra["dx"],
                                        size=(n, 3))
    integ.create_buffers(w.nlist, w.n_neigh, w.bond_stiffness,
                         w.critical_stretch, None, u, None, None, None, None,
                         None, None, 1, 1)
    integ.run(3, np.full(3, 1e-6), np.ones(3))
    return integ.tile_stats()["ntiles"], integ.write(
        None, None, None, None, None, None, None, None)


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("shape,per_cu", [
    ((64, 3, 1), 1), ((181, 181, 1), 1), ((182, 181, 1), 2),
    ((256, 256, 1), 2), ((257, 256, 1), 3), ((390, 391, 1), 5),
    ((423, 425, 1), 6)])
def test_tiles_spread_over_the_cus(shape, per_cu, exact):
    cus = 256
    w = configs.beam_vv(shape=shape, layout="compact" if exact else "slot")
    n = w.nlist.shape[0]
    assert -(-n // (128 * cus)) == per_cu
    group = np.minimum(np.arange(n) * 3 // n, 2).astype(np.int32)
    group[: n // 5] = 7
    _, want = _run(w, exact, 64, None)
    for g in (None, group):
        ntiles, got = _run(w, exact, 128, g)
        if n > 48 * cus and (g is None or n % (128 * cus)):
            limit = per_cu + (g is not None and n > per_cu * 128 * cus - 512)
            assert ntiles <= limit * cus
            assert ntiles > (per_cu - 1) * cus
        if per_cu <= 5 and g is None and n > 48 * cus:
            assert ntiles > per_cu * cus - 16
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)
