"""pd_create_buffers again on one simulation against a fresh simulation,
bitwise: with the same bonds (whose tiles and slots are kept), after bonds
broke and regimes moved, with other state and other damage-model values, with
one bond fewer, with starting regimes, with another launch shape, and in the
exact order -- each call right after any other."""
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


def _workload(model):
    shape = (23, 7, 6)
    if model == "nlin":
        return configs.composite_ec(shape=shape)
    return configs.beam_vv(shape=shape, layout="compact" if model in (
        "cython", "cython_fast") else "slot")


def _make(model, w):
    n, k = w.nlist.shape
    dens = bt = corr = None
    if model in ("cython", "cython_fast"):
        integ = it.Euler(2e-15, exact_order=model == "cython")
    elif model == "field":
        integ = it.EulerHIP(2e-15)
    else:
        dens = w.densities
        integ = it.EulerCromerHIP(2.5e6, 1e-8)
        bt = w.bond_types
        if model == "corr":
            corr = np.random.default_rng(2).uniform(0.5, 2.0, (n, k))
    integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                w.bc_values, w.force_bc_types, w.force_bc_values, corr, bt,
                dens)
    if model == "field":
        integ.set_node_stiffness(
            w.bond_stiffness
            * np.random.default_rng(3).uniform(0.5, 2.0, n))
    return integ


def _start(integ, w, variant, model):
    """One of the ways to start; returns its argument set's launch shape."""
    n, k = w.nlist.shape
    dx = w.extra["dx"]
    rng = np.random.default_rng(variant)
    # stretches around s0 (0.005) and the regimes' breakpoints
    u = rng.normal(scale=2e-3 * dx, size=(n, 3)) if variant != 1 else None
    ud = rng.normal(scale=1e-2, size=(n, 3)) if variant % 2 else None
    nl, nn = w.nlist.copy(), w.n_neigh.copy()
    scale = 1.0 + 0.25 * variant
    regimes = None
    if variant == 2:  # one bond fewer, in both its rows
        i, j = 40, int(nl[40, 3])
        for a, b in ((i, j), (j, i)):
            p = int(np.flatnonzero(nl[a, :nn[a]] == b)[0])
            nl[a, p:nn[a] - 1] = nl[a, p + 1:nn[a]].copy()
            nl[a, nn[a] - 1] = 0 if integ.context is None else -1
            nn[a] -= 1
    if variant == 3 and w.nregimes > 1:
        regimes = rng.integers(0, 2, nl.shape).astype(np.int32)
    if model not in ("cython", "cython_fast"):
        integ.set_launch(4, 64 if variant == 4 else 128)
    integ.create_buffers(nl, nn, np.asarray(w.bond_stiffness) * scale,
                         np.asarray(w.critical_stretch) * scale,
                         None if w.plus_cs is None else w.plus_cs * scale
                         * scale, u, ud, None, None, None, None, regimes,
                         w.nregimes, w.nbond_types)


def _result(integ, w):
    integ.run(4, np.full(4, 1e-6), np.ones(4))
    out = integ.write(None, None, None, None, None, None, None, None)
    return list(out) + ([integ.regimes()] if w.nregimes > 1 else [])


@pytest.mark.parametrize("model", ["cython", "cython_fast", "field", "corr",
                                   "nlin"])
def test_restarts_equal_fresh_simulations(model):
    w = _workload(model)
    fresh = {}
    for v in range(5):
        integ = _make(model, w)
        _start(integ, w, v, model)
        fresh[v] = _result(integ, w)
        del integ
    lost = w.n_neigh.sum() - fresh[0][7].sum()
    assert lost > 0  # bonds break between the restarts
    integ = _make(model, w)
    for v in (0, 0, 1, 0, 2, 2, 0, 3, 0, 4, 4, 1, 3, 3, 2, 4, 0):
        _start(integ, w, v, model)
        for got, want in zip(_result(integ, w), fresh[v]):
            np.testing.assert_array_equal(got, want)
