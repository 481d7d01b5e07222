"""The step kernel's narrow halo form (scalar stiffness, more than two tiles
per CU, halos of at most 959 entries) against the wide one, bitwise: tiles of
128 nodes run the one and tiles of 256, whose blocks are too large for it, the
other.  Each integrator and break mode, bonds breaking, halos far below and at
the capacity (where tiles are cut to it), and a mesh whose tiles would be cut
too often."""
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


def _run(w, kind, tile, tension):
    n, k = w.nlist.shape
    dens = None
    if kind == "euler":
        integ = it.EulerHIP(2e-15)
    else:
        dens = w.densities
        integ = (it.VelocityVerletHIP if kind == "verlet"
                 else it.EulerCromerHIP)(2.5e6, 1e-8)
    integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                w.bc_values, w.force_bc_types, w.force_bc_values, None, None,
                dens)
    integ.set_launch(4, tile)
    integ.set_break_mode(tension)
    rng = np.random.default_rng(4)
    u = rng.normal(scale=2e-3 * w.extra["dx"], size=(n, 3))
    ud = rng.normal(scale=1e-2, size=(n, 3))
    integ.create_buffers(w.nlist, w.n_neigh, w.bond_stiffness,
                         w.critical_stretch, None, u, ud, None, None, None,
                         None, None, 1, 1)
    integ.run(3, np.full(3, 1e-6), np.ones(3))
    return integ.tile_stats(), integ.write(
        None, None, None, None, None, None, None, None)


@pytest.mark.parametrize("shape,kind,tension,most", [
    ((300, 230, 1), "cromer", False, 400), ((300, 230, 1), "euler", True, 400),
    ((130, 24, 22), "verlet", False, 959), ((190, 23, 22), "euler", False, 959),
    ((190, 23, 22), "cromer", True, 959), ((212, 29, 31), "verlet", False,
                                           1279)])
def test_narrow_equals_wide(shape, kind, tension, most):
    w = configs.beam_vv(shape=shape)
    ns, narrow = _run(w, kind, 128, tension)
    ws, wide = _run(w, kind, 256, tension)
    assert ns["ntiles"] > 2 * 256 and ns["hstride"] <= most
    assert narrow[7].sum() < w.n_neigh.sum()
    for a, b in zip(narrow, wide):
        np.testing.assert_array_equal(a, b)
