"""Recordings held to their checkpoints: no more memory than the interval
asks for, the same gradient and state bitwise, and back again."""
import numpy as np
import pytest

from probabilistic_peridynamics_amd import adjoint
from test_gpu_recording import _make, _state

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip_device")]


def _free():
    import torch
    return torch.cuda.mem_get_info(0)[0]


def _recording(integ, steps, every):
    integ.adjoint_start(steps, checkpoint_every=every)
    integ.run(steps - 3, 1e-9 * np.arange(steps - 3), np.ones(steps - 3))
    integ.run(3, np.full(3, 1e-6), np.ones(3))
    before = _state(integ)
    dL = np.random.default_rng(1).normal(size=before[0].shape)
    grad = integ.adjoint_backward(dL)
    for a, b in zip(_state(integ), before):
        np.testing.assert_array_equal(a, b)
    return list(before) + [grad]


@pytest.mark.parametrize("steps,every", [(22, 1), (22, 3), (22, 20), (40, 40),
                                         (300, 16)])
def test_checkpoints_give_what_every_step_gives(steps, every):
    out = []
    for keep in (True, False):
        integ, _ = _make(2e-3)
        integ.adjoint_keep(keep)
        live = _state(integ)[7].sum()
        out.append(_recording(integ, steps, every))
        assert out[-1][7].sum() < live and np.any(out[-1][-1] != 0.0)
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_memory_is_that_of_the_checkpoints():
    steps, every = 10000, 400
    integ, _ = _make(1e-5)
    n, slots = integ.nnodes, integ.tile_stats()["slots"]
    integ.adjoint_keep(False)
    base = _free()
    # 14 bytes a slot, 256 a node, 24 a node for a checkpoint and a step of a
    # segment; buffers are given out in pieces of 2 MiB
    asked = 14 * slots + n * (256 + 24 * (steps // every + every))
    for keep in (False, True, False):
        integ.adjoint_keep(keep)
        integ.adjoint_start(steps, checkpoint_every=every)
        taken = base - _free()
        if keep:
            assert taken > 24 * n * steps
        else:
            assert taken < asked + 24 * 2 ** 21
    integ.adjoint_stop()


def test_solvers_can_be_held_to_their_checkpoints():
    from test_adjoint_ref import adjoint_workload
    w = adjoint_workload(shape=(16, 5, 5), seed=0)
    grads = []
    for keep in (True, False):
        solver = adjoint.StiffnessAdjoint(w, 40, checkpoint_every=16,
                                          keep_every_step=keep)
        u = solver.forward(w.extra["g"])
        grads.append(solver.backward(np.ones_like(u)))
    np.testing.assert_array_equal(*grads)
