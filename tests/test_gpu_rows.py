"""Rows of every length against the oracle: stars of 1 to 40 bonds in one
mesh, so that rows end anywhere in a round of a node's lanes (and rows of
several rounds share tiles and wavefronts with rows of one bond), for each
variant of the step kernel and each number of lanes per node; and the same
stars at a scale outside the range in which the kernel's fast bond test is
exact, where every bond takes the exact path.

Lists, regimes and damage identical; u and force to the repository's parity
bounds (rows of at most 40 terms, three steps: rounding is below 1e-13)."""
import numpy as np
import pytest

import oracle
import pdcases as pc
from probabilistic_peridynamics_amd import _lib
from probabilistic_peridynamics_amd import integrators as it

pytestmark = pytest.mark.gpu

S0 = 0.01


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    try:
        ok = _lib.device_count() > 0
    except OSError:
        ok = False
    if not ok:
        pytest.fail("no HIP device: the gpu tests need an MI355X")


def _stars(scale, compact, seed=5, most=40):
    """Star s has s + 1 leaves; numbered in a random order."""
    rng = np.random.default_rng(seed)
    coords, edges = [], []
    for s in range(most):
        hub = len(coords)
        centre = np.array([4.0 * (s % 7), 4.0 * (s // 7), 1.0])
        coords.append(centre)
        for _ in range(s + 1):
            d = rng.normal(size=3)
            d *= rng.uniform(0.6, 1.4) / np.linalg.norm(d)
            edges.append((hub, len(coords)))
            coords.append(centre + d)
    n = len(coords)
    name = rng.permutation(n)
    x = np.empty((n, 3))
    x[name] = np.array(coords)
    rows = [[] for _ in range(n)]
    for a, b in edges:
        rows[name[a]].append(int(name[b]))
        rows[name[b]].append(int(name[a]))
    fam = np.array([len(r) for r in rows], dtype=np.int32)
    k = int(fam.max()) if compact else 1 << (int(fam.max()) - 1).bit_length()
    nl = np.full((n, k), 0 if compact else -1, dtype=np.int32)
    for i, r in enumerate(rows):
        nl[i, :len(r)] = sorted(r)
    u = rng.normal(scale=0.6 * S0, size=(n, 3))
    return x * scale, u * scale, fam, nl


@pytest.mark.parametrize("scale", [1.0, 1e-92])
@pytest.mark.parametrize("lanes", [1, 2, 4, 8])
@pytest.mark.parametrize("model", ["cython", "euler", "tension", "corr",
                                   "field", "nlin"])
def test_rows_of_every_length(model, lanes, scale):
    x, u0, fam, nl = _stars(scale, model == "cython")
    n, k = nl.shape
    rng = np.random.default_rng(7)
    vol = rng.uniform(0.5, 1.5, n)
    bct = np.zeros((n, 3), np.int32)
    bcv = np.zeros((n, 3))
    dt = 2e-4 * scale  # moves of a few per cent of s0 a step
    z = np.zeros((n, 3))
    corr = types = pcs = cnode = None
    stiff, crit, reg, kinds = 1.0, S0, 1, 1
    if model == "corr":
        corr = np.where(nl >= 0, rng.uniform(0.5, 2.0, nl.shape), 0.0)
    elif model == "field":
        cnode = rng.uniform(0.5, 2.0, n)
    elif model == "nlin":
        reg, kinds = 3, 2
        types = np.where(nl >= 0, rng.integers(0, 2, nl.shape), 0).astype(
            np.int32)
        stiff = np.array([[1.0, 0.6, 0.1], [2.0, 1.0, 0.5]])
        crit = S0 * np.array([[0.3, 0.7, 1.0], [0.2, 0.5, 1.2]])
        pcs = np.zeros((2, 3))
        for r in (1, 2):
            pcs[:, r] = (pcs[:, r - 1] + stiff[:, r - 1] * crit[:, r - 1]
                         - stiff[:, r] * crit[:, r - 1])
    if model == "cython":
        integ = it.Euler(dt, exact_order=False)
        ref = oracle.CythonEuler(dt, x, vol, fam, bct, bcv, bct, bcv, nl,
                                 fam, stiff, crit, u=u0)
    else:
        integ = it.EulerHIP(dt)
        ref = oracle.SlotStepper(
            0, dt, x, vol, fam, bct, bcv, bct, bcv, nl, stiff, crit,
            stiffness_corrections=corr, bond_types=types, plus_cs=pcs,
            nregimes=reg, cnode=cnode, tension_only=model == "tension",
            u=u0)
    integ.build(n, 3, k, x, vol, fam, bct, bcv, bct, bcv, corr, types, None)
    integ.set_launch(lanes, 64)
    integ.set_break_mode(model == "tension")
    if cnode is not None:
        integ.set_node_stiffness(cnode)
    integ.create_buffers(nl, fam.copy(), stiff, crit, pcs, u0, z, z, z, z,
                         np.zeros(n), None, reg, kinds)
    broken = 0
    for _ in range(3):
        integ(0.0, 0.0)
        ref(0.0, 0.0)
        u, _, _, force, _, dmg, lists, nn = integ.write(
            None, None, None, None, None, None, None, None)
        if model == "cython":
            rn, rd = ref.n_neigh, ref.damage()
        else:
            rn, rd = ref.connectivity()
        np.testing.assert_array_equal(lists, ref.nlist)
        np.testing.assert_array_equal(nn, rn)
        np.testing.assert_array_equal(dmg, rd)
        if reg > 1:
            np.testing.assert_array_equal(integ.regimes(), ref.regimes)
        assert pc.rel_l2(u / scale, ref.u / scale) < 1e-10
        assert pc.rel_l2(force, ref.force) < 1e-9
        broken = int(fam.sum() - np.sum(nn))
    assert 0 < broken < fam.sum() / 2


@pytest.mark.parametrize("scale", [1.0, 1e-92])
@pytest.mark.parametrize("most", [40, 185])
@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("fast_first", [False, True])
def test_exact_order_rows_of_every_length(fast_first, tile, most, scale):
    """The exact-order step on the same stars, bitwise: fold lists of every
    length, split anywhere between lower and upper neighbours (the numbering
    is random), with bonds breaking in both parts.  ``fast_first`` runs the
    first, breaking step in the fast order, whose broken bonds the fold lists
    made for the exact order must leave out.  185 stars (17,390 nodes) take
    tiles of more than 64 nodes where these are allowed, and with them four
    lanes per node instead of eight."""
    x, u0, fam, nl = _stars(scale, True, seed=8, most=most)
    n, k = nl.shape
    vol = np.random.default_rng(9).uniform(0.5, 1.5, n)
    bct = np.zeros((n, 3), np.int32)
    bcv = np.zeros((n, 3))
    dt = 2e-4 * scale
    z = np.zeros((n, 3))
    integ = it.Euler(dt, exact_order=not fast_first)
    integ.build(n, 3, k, x, vol, fam, bct, bcv, bct, bcv, None, None, None)
    integ.set_launch(4, tile)
    integ.create_buffers(nl, fam.copy(), 1.0, S0, None, u0, z, z, z, z,
                         np.zeros(n), None, 1, 1)
    ref = oracle.CythonEuler(dt, x, vol, fam, bct, bcv, bct, bcv, nl, fam,
                             1.0, S0, u=u0)
    for s in range(3):
        integ(0.0, 0.0)
        ref(0.0, 0.0)
        if fast_first and s == 0:
            integ.set_exact_order(True)
            continue
        u, _, _, force, _, dmg, lists, nn = integ.write(
            None, None, None, None, None, None, None, None)
        np.testing.assert_array_equal(lists, ref.nlist)
        np.testing.assert_array_equal(nn, ref.n_neigh)
        np.testing.assert_array_equal(dmg, ref.damage())
        if fast_first:
            assert pc.rel_l2(u / scale, ref.u / scale) < 1e-10
            assert pc.rel_l2(force, ref.force) < 1e-9
        else:
            np.testing.assert_array_equal(u, ref.u)
            np.testing.assert_array_equal(force, ref.force)
    assert 0 < int(fam.sum() - nn.sum()) < fam.sum() / 2
