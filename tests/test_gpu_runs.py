"""A run stores force, body_force, u (slot layout) and Euler-Cromer's udd of
its last step only: a run, a run as a graph, runs cut in pieces and a recorded
run leave every array bitwise as single steps do, for each integrator and
layout and for run lengths of 1, 2 and more."""
import numpy as np
import pytest

from probabilistic_peridynamics_amd import _lib, configs
from probabilistic_peridynamics_amd import integrators as it

pytestmark = pytest.mark.gpu

STEPS = 22  # graphs of 2, 8, 8 and 4 steps; of 1; of 2; of 2 and 1 ...


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    try:
        ok = _lib.device_count() > 0
    except OSError:
        ok = False
    if not ok:
        pytest.fail("no HIP device: the gpu tests need an MI355X")


def _make(model):
    shape = (23, 7, 6)
    w = (configs.composite_ec(shape=shape) if model == "nlin" else
         configs.beam_vv(shape=shape, layout="compact" if model in (
             "cython", "cython_fast") else "slot"))
    n, k = w.nlist.shape
    rng = np.random.default_rng(5)
    force_bc = np.zeros((n, 3), dtype=w.force_bc_types.dtype)
    force_bc[rng.random(n) < 0.2] = 1
    fv = rng.normal(scale=1e3, size=(n, 3))
    dens = bt = None
    if model in ("cython", "cython_fast"):
        integ = it.Euler(2e-15, exact_order=model == "cython")
    elif model == "euler":
        integ = it.EulerHIP(2e-15)
    elif model == "verlet":
        integ, dens = it.VelocityVerletHIP(2.5e6, 1e-8), w.densities
    else:
        integ, dens = it.EulerCromerHIP(2.5e6, 1e-8), w.densities
        bt = w.bond_types
    integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                w.bc_values, force_bc, fv, None, bt, dens)
    u = rng.normal(scale=2e-3 * w.extra["dx"], size=(n, 3))
    integ.create_buffers(w.nlist, w.n_neigh, w.bond_stiffness,
                         w.critical_stretch, w.plus_cs, u,
                         rng.normal(scale=1e-2, size=(n, 3)), None, None,
                         None, None, None, w.nregimes, w.nbond_types)
    return integ


def _arrays(integ):
    return integ.write(None, None, None, None, None, None, None, None)


def _check(got, want):
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("cut", [(STEPS,), (1, 2, 3, STEPS - 6)])
@pytest.mark.parametrize("model", ["cython", "cython_fast", "euler", "verlet",
                                   "nlin"])
def test_runs_equal_single_steps(model, cut):
    d, f = 1e-6 * np.arange(1, STEPS + 1), np.linspace(0.5, 2, STEPS)
    single = _make(model)
    for s in range(STEPS):
        single(d[s], f[s])
    want = _arrays(single)
    assert np.any(want[3] != 0.0)
    # the Cython path's class returns the body_force array that it was given
    assert model.startswith("cython") or np.any(want[4] != want[3])
    for name in ("run", "run_graph"):
        integ, at = _make(model), 0
        for m in cut:
            getattr(integ, name)(m, d[at:at + m], f[at:at + m])
            at += m
        _check(_arrays(integ), want)


@pytest.mark.parametrize("every", [1, 3, 20])
def test_recorded_runs_equal_recorded_steps(every):
    """Checkpoints and the replay between them."""
    d, f = 1e-6 * np.arange(1, STEPS + 1), np.linspace(0.5, 2, STEPS)
    out = []
    for whole in (False, True):
        integ = _make("euler")
        n = integ.nnodes
        integ.set_node_stiffness(
            np.random.default_rng(3).uniform(0.5e18, 1e18, n))
        integ.adjoint_start(STEPS, checkpoint_every=every)
        if whole:
            integ.run(STEPS, d, f)
        else:
            for s in range(STEPS):
                integ(d[s], f[s])
        before = _arrays(integ)
        grad = integ.adjoint_backward(np.ones((n, 3)))
        _check(_arrays(integ), before)
        out.append(list(before) + [np.asarray(grad)])
        assert np.any(out[-1][-1] != 0.0)
    _check(out[1], out[0])
