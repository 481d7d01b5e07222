"""Calls that fail on their way: what they leave is what was there before, or
the whole result, or is refused until the buffers are made anew -- never a
displacement of one step beside the bonds of another.

Failures of HIP calls are made by a small library that stands before the HIP
runtime in a process of its own and reports an error, without calling on, at
the given call of the given function."""
import json
import subprocess
import sys

import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip_device")]

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
typedef struct { unsigned x, y, z; } dim;
static int left[5], pending;
void shim_arm(int which, int calls) { left[which] = calls; pending = 0; }
static int now(int which) { return left[which] > 0 && --left[which] == 0; }
int hipGraphInstantiate(void *e, void *g, void *n, char *b, size_t s)
{
    if (now(0))
        return 2;
    int (*f)(void *, void *, void *, char *, size_t) =
        dlsym(RTLD_NEXT, "hipGraphInstantiate");
    return f(e, g, n, b, s);
}
int hipGraphLaunch(void *e, void *s)
{
    if (now(1))
        return 2;
    int (*f)(void *, void *) = dlsym(RTLD_NEXT, "hipGraphLaunch");
    return f(e, s);
}
int hipLaunchKernel(const void *k, dim g, dim b, void **a, size_t m, void *s)
{
    if (now(2))
        return pending = 2;
    int (*f)(const void *, dim, dim, void **, size_t, void *) =
        dlsym(RTLD_NEXT, "hipLaunchKernel");
    return f(k, g, b, a, m, s);
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st)
{
    if (now(3))
        return 2;
    int (*f)(void *, const void *, size_t, int, void *) =
        dlsym(RTLD_NEXT, "hipMemcpyAsync");
    return f(d, s, n, kind, st);
}
int hipMalloc(void **p, size_t n)
{
    if (now(4))
        return 2;
    int (*f)(void **, size_t) = dlsym(RTLD_NEXT, "hipMalloc");
    return f(p, n);
}
int hipGetLastError(void)
{
    int (*f)(void) = dlsym(RTLD_NEXT, "hipGetLastError");
    const int e = pending ? pending : f();
    pending = 0;
    return e;
}
"""

CHILD = r"""
import ctypes, json, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = sys.argv[2:4]
import numpy as np
from probabilistic_peridynamics_amd import _lib
from test_gpu_runs import _arrays, _make
which, calls, method = json.loads(sys.argv[4])
STEPS = 22
d, f = 1e-6 * np.arange(1, STEPS + 1), np.linspace(0.5, 2, STEPS)
integ = _make("euler")
start = _arrays(integ)
integ.run(STEPS, d, f)
want = _arrays(integ)
same = lambda a, b: all(np.array_equal(x, y) for x, y in zip(a, b))


def refused(call, *args):
    try:
        call(*args)
    except _lib.PDError as e:
        return e.code
    return 0


fresh = _make("euler")
shim.shim_arm(which, calls)
out = {"call": refused(getattr(fresh, method), STEPS, d, f)}
shim.shim_arm(which, 0)
out["write"] = refused(_arrays, fresh)
if not out["write"]:
    got = _arrays(fresh)
    out["state"] = ("whole" if same(got, want) else
                    "start" if same(got, start) else "neither")
else:
    out["others"] = [refused(call, *a) for call, a in (
        (fresh.run, (1, d[:1], f[:1])), (fresh, (0.0, 0.0)),
        (fresh.monitor, ()), (fresh.write_device, ()),
        (fresh.adjoint_start, (2,)), (fresh.regimes, ()),
        (fresh.live_bonds, ()))]
w = __import__("test_gpu_runs").configs.beam_vv(shape=(23, 7, 6))
n = fresh.nnodes
rng = np.random.default_rng(5)
rng.random(n), rng.normal(size=(n, 3))
u = rng.normal(scale=2e-3 * w.extra["dx"], size=(n, 3))
fresh.create_buffers(w.nlist, w.n_neigh, w.bond_stiffness,
                     w.critical_stretch, w.plus_cs, u,
                     rng.normal(scale=1e-2, size=(n, 3)), None, None, None,
                     None, None, 1, 1)
getattr(fresh, method)(STEPS, d, f)
out["again"] = same(_arrays(fresh), want)
print("RESULT", json.dumps(out), flush=True)
"""

INSTANTIATE, GRAPH, KERNEL, COPY, MALLOC = 0, 1, 2, 3, 4

HEAD = r"""
import ctypes, json, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = sys.argv[2:4]
import numpy as np
from probabilistic_peridynamics_amd import _lib
from test_gpu_recording import _make, _state
which, calls, what = json.loads(sys.argv[4])


def refused(call, *args):
    try:
        call(*args)
    except _lib.PDError as e:
        return e.code
    return 0


"""

RECORDED_STEP = HEAD + r"""
integ, _ = _make(2e-3)
integ.adjoint_keep(what)
integ.adjoint_start(4, checkpoint_every=1)
shim.shim_arm(which, calls)
out = [refused(integ, 1e-6, 1.0) for _ in range(2)]
shim.shim_arm(which, 0)
out += [refused(_state, integ), refused(integ, 1e-6, 1.0)]
print("RESULT", json.dumps(out), flush=True)
"""

CHANGED_MODEL = HEAD + r"""
if what == "order":
    integ = __import__("test_gpu_runs")._make("cython")
    call, args = integ.set_exact_order, (False,)
else:
    integ, cs = _make(2e-3)
    call, args = integ.set_node_stiffness, (cs[1],)
shim.shim_arm(which, calls)
out = [refused(call, *args)]
shim.shim_arm(which, 0)
out += [refused(_state, integ), refused(integ, 0.0, 0.0)]
print("RESULT", json.dumps(out), flush=True)
"""

MONITOR = HEAD + r"""
integ, _ = _make(2e-3)
integ(1e-6, 1.0)
shim.shim_arm(which, calls)
out = [refused(integ.monitor)]
shim.shim_arm(which, 0)
fresh, _ = _make(2e-3)
fresh(1e-6, 1.0)
out.append(integ.monitor() == fresh.monitor())
print("RESULT", json.dumps(out), flush=True)
"""

TIPS = HEAD + r"""
integ, _ = _make(2e-3)
integ(1e-6, 1.0)
tips = {"a": [(3, 0), (7, 2)], "b": [(0, 1)]}
shim.shim_arm(which, calls)
out = [refused(integ.set_tips, tips)]
shim.shim_arm(which, 0)
fresh, _ = _make(2e-3)
fresh(1e-6, 1.0)
fresh.set_tips(tips)
out.append(integ.monitor() == fresh.monitor())
print("RESULT", json.dumps(out), flush=True)
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(d / "shim.so"),
                    str(d / "shim.c"), "-Wl,--no-as-needed",
                    "-L/opt/rocm/lib", "-lamdhip64", "-ldl"], check=True)
    return d / "shim.so"


def _child(shim, code, which, calls, what):
    from conftest import ROOT, TESTS
    r = subprocess.run(
        [sys.executable, "-c", code, str(shim), str(ROOT), str(TESTS),
         json.dumps([which, calls, what])],
        capture_output=True, text=True, timeout=100)
    line = [x for x in r.stdout.splitlines() if x.startswith("RESULT")]
    assert r.returncode == 0 and line, r.stdout + r.stderr
    return json.loads(line[0][len("RESULT"):])


def _after_failure(shim, which, calls, method):
    out = _child(shim, CHILD, which, calls, method)
    assert out["again"]  # new buffers, and all is well
    return out


@pytest.mark.parametrize("which,calls,method", [
    (INSTANTIATE, 1, "run_graph"), (GRAPH, 1, "run_graph"),
    (KERNEL, 1, "run_graph"), (KERNEL, 1, "run")])
def test_a_run_that_fails_at_once_leaves_the_state(shim, which, calls,
                                                   method):
    out = _after_failure(shim, which, calls, method)
    assert out["call"] == -2 and out["state"] == "start"


@pytest.mark.parametrize("which,calls", [(INSTANTIATE, 3), (KERNEL, 6)])
def test_a_graph_that_cannot_be_made_is_run_as_launches(shim, which, calls):
    out = _after_failure(shim, which, calls, "run_graph")
    assert out["call"] == 0 and out["state"] == "whole"


@pytest.mark.parametrize("which,calls,method", [
    (GRAPH, 3, "run_graph"), (KERNEL, 6, "run"), (KERNEL, 6, "timed_run")])
def test_a_run_that_fails_on_its_way_is_not_read(shim, which, calls, method):
    out = _after_failure(shim, which, calls, method)
    assert out["call"] == -2 and out["write"] == -4
    assert out["others"] == [-4] * 7


@pytest.mark.parametrize("keep", [True, False])
def test_a_step_whose_recording_fails_is_not_read(shim, keep):
    """The copy of u that a recorded step makes after its launch, at the
    second step."""
    out = _child(shim, RECORDED_STEP, COPY, 2, keep)
    assert out == [0, -2, -4, -4]


@pytest.mark.parametrize("which,what", [(MALLOC, "field"), (KERNEL, "field"),
                                        (KERNEL, "order")])
def test_a_model_that_changed_half_is_not_stepped(shim, which, what):
    out = _child(shim, CHANGED_MODEL, which, 1, what)
    assert out == [-2, -4, -4]


@pytest.mark.parametrize("calls", [1, 2])
def test_memory_that_was_refused_is_asked_for_again(shim, calls):
    assert _child(shim, MONITOR, MALLOC, calls, None) == [-2, True]


@pytest.mark.parametrize("calls", [1, 2])
def test_tips_that_got_no_memory_are_asked_for_again(shim, calls):
    assert _child(shim, TIPS, MALLOC, calls, None) == [-2, True]


def test_refused_lists_leave_the_tiles_and_their_shape():
    """Bonds too many for a tile's halo are refused after the next tiling's
    shape is known: the steps go on with the one that there is."""
    from probabilistic_peridynamics_amd import _lib, configs
    from probabilistic_peridynamics_amd import integrators as it
    w = configs.beam_vv(shape=(14, 10, 10))
    n, k = w.nnodes, 1408
    nl = np.full((n, k), -1, np.int32)
    nl[:, :w.nlist.shape[1]] = w.nlist
    u = np.random.default_rng(1).normal(scale=2e-3 * w.extra["dx"],
                                        size=(n, 3))
    wide = nl.copy()
    wide[0, :1300] = np.arange(1, 1301)
    out = []
    for refuse in (False, True):
        integ = it.EulerHIP(2e-15)
        integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                    w.bc_values, w.force_bc_types, w.force_bc_values, None,
                    None, None)
        integ.set_launch(4, 64)
        args = (w.bond_stiffness, w.critical_stretch, None, u, None, None,
                None, None, None, None, 1, 1)
        integ.create_buffers(nl, w.n_neigh, *args)
        integ.set_launch(8, 64)
        if refuse:
            with pytest.raises(_lib.PDError) as e:
                integ.create_buffers(wide, w.n_neigh, *args)
            assert e.value.code == _lib.PD_E_LIMIT
        integ.run(3, np.full(3, 1e-6), np.ones(3))
        out.append(integ.write(None, None, None, None, None, None, None,
                               None))
    assert np.any(out[0][3] != 0.0)
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("every", [3, 9])
def test_a_backward_pass_that_is_refused_leaves_the_state(every):
    """A tile size set after the recording, which a replay would need."""
    from probabilistic_peridynamics_amd import _lib
    from test_gpu_recording import _make, _state
    integ, _ = _make(2e-3)
    integ.adjoint_start(9, checkpoint_every=every)
    integ.run(9, np.full(9, 1e-6), np.ones(9))
    before = _state(integ)
    integ.set_launch(4, 64)
    with pytest.raises(_lib.PDError) as e:
        integ.adjoint_backward(np.ones(before[0].shape))
    assert e.value.code == _lib.PD_E_STATE
    for a, b in zip(_state(integ), before):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("steps,every", [(1, 1), (1, 5), (9, 1)])
def test_a_backward_pass_that_replays_nothing_needs_no_tiles(steps, every):
    from test_gpu_recording import _make, _state
    grads = []
    for later in (False, True):
        integ, _ = _make(2e-3)
        integ.adjoint_start(steps, checkpoint_every=every)
        integ.run(steps, np.full(steps, 1e-6), np.ones(steps))
        before = _state(integ)
        if later:
            integ.set_launch(4, 64)
        dL = np.random.default_rng(1).normal(size=before[0].shape)
        grads.append(integ.adjoint_backward(dL))
        for a, b in zip(_state(integ), before):
            np.testing.assert_array_equal(a, b)
    assert np.any(grads[0] != 0.0)
    # the lanes of the default shape may be others: the sums' order
    np.testing.assert_allclose(grads[1], grads[0], rtol=0,
                               atol=1e-10 * np.abs(grads[0]).max())


@pytest.mark.parametrize("every", [3, 9])
def test_a_backward_pass_without_its_field_is_refused(every):
    """The field cleared after the recording; set again, the pass is that of
    a recording whose field was set anew."""
    from probabilistic_peridynamics_amd import _lib
    from test_gpu_recording import _make, _state
    grads = []
    for cleared in (False, True):
        integ, cs = _make(2e-3)
        integ.adjoint_start(9, checkpoint_every=every)
        integ.run(9, np.full(9, 1e-6), np.ones(9))
        before = _state(integ)
        dL = np.random.default_rng(1).normal(size=before[0].shape)
        if cleared:
            integ.set_node_stiffness(None)
            with pytest.raises(_lib.PDError) as e:
                integ.adjoint_backward(dL)
            assert e.value.code == _lib.PD_E_STATE
            for a, b in zip(_state(integ), before):
                np.testing.assert_array_equal(a, b)
        integ.set_node_stiffness(cs[0])
        grads.append(integ.adjoint_backward(dL))
    assert np.any(grads[0] != 0.0)
    np.testing.assert_array_equal(*grads)
