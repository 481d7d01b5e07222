"""A recording that keeps u of every step and one that keeps checkpoints (more
steps than 32 times its checkpoints and a segment) give bitwise the same
gradient and end state, with bonds breaking; a field or a launch shape that is
set after the recording is the one that the backward pass replays or
refuses."""
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


def _make(scale, seed=3):
    """(integrator, fields c) with displacements of `scale` grid spacings
    (2e-3 breaks bonds, whose critical stretch is 0.005)."""
    w = configs.beam_vv(shape=(19, 6, 5))
    n, k = w.nlist.shape
    integ = it.EulerHIP(2e-15)
    integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                w.bc_values, w.force_bc_types, w.force_bc_values, None, None,
                None)
    rng = np.random.default_rng(seed)
    cs = w.bond_stiffness * rng.uniform(0.5, 2.0, (2, n))
    integ.set_node_stiffness(cs[0])
    u = rng.normal(scale=scale * w.extra["dx"], size=(n, 3))
    integ.create_buffers(w.nlist, w.n_neigh, w.bond_stiffness,
                         w.critical_stretch, None, u, None, None, None, None,
                         None, None, 1, 1)
    return integ, cs


def _state(integ):
    return integ.write(None, None, None, None, None, None, None, None)


@pytest.mark.parametrize("steps,every", [(4200, 64), (4705, 99)])
def test_checkpoints_equal_every_step(steps, every):
    out = []
    for e in (every, steps):
        assert (steps > 32 * (-(-steps // e) + e)) == (e == every)
        integ, _ = _make(2e-3)
        live = _state(integ)[7].sum()
        integ.adjoint_start(steps, checkpoint_every=e)
        integ.run(steps - 5, 1e-9 * np.arange(steps - 5), np.ones(steps - 5))
        integ.run(5, np.full(5, 1e-6), np.ones(5))
        before = _state(integ)
        assert before[7].sum() < live
        dL = np.random.default_rng(1).normal(size=before[0].shape)
        grads = [integ.adjoint_backward(dL) for _ in range(2)]
        after = _state(integ)
        np.testing.assert_array_equal(grads[0], grads[1])
        assert np.any(grads[0] != 0.0) and np.all(np.isfinite(grads[0]))
        for a, b in zip(after, before):
            np.testing.assert_array_equal(a, b)
        integ.run(3, np.full(3, 1e-6), np.ones(3))  # and goes on from there
        out.append(list(before) + [grads[0]] + list(_state(integ)))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_backward_takes_what_was_set_after_the_recording():
    steps, grads = 9, []
    for change in (False, True):
        integ, cs = _make(1e-5)
        if not change:
            integ.set_node_stiffness(cs[1])
        integ.adjoint_start(steps, checkpoint_every=steps)
        integ.run(steps, np.zeros(steps), np.ones(steps))
        u = _state(integ)[0]
        if change:
            integ.set_node_stiffness(cs[1])
        grads.append(integ.adjoint_backward(np.ones(u.shape)))
        np.testing.assert_array_equal(_state(integ)[0], u)
    np.testing.assert_array_equal(*grads)
    integ.set_launch(4, 64)  # as a step: re-tile first
    with pytest.raises(_lib.PDError):
        integ.adjoint_backward(np.ones(u.shape))
