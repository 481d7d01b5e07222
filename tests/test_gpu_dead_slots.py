"""Broken and empty slots add nothing, whatever the correction, the damage
tables or the node's own values hold: infinities and NaN reach only live
bonds."""
import numpy as np
import pytest

import oracle
import pdcases as pc
from probabilistic_peridynamics_amd import configs
from probabilistic_peridynamics_amd import integrators as it

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip_device")]

RTOL = 1e-10  # u against the oracle, relative L2; forces 1e-9
BAD = [np.inf, -np.inf, np.nan]


def _arrays(integ):
    return integ.write(None, None, None, None, None, None, None, None)


def _oracle_parity(integ, ref, steps):
    d, f = 1e-8 * np.arange(1, steps + 1), np.linspace(0.5, 2, steps)
    integ.run(steps, d, f)
    for s in range(steps):
        ref(d[s], f[s])
    u, _, _, force, _, _, nl, _ = _arrays(integ)
    assert np.all(np.isfinite(ref.force)) and np.any(ref.force != 0.0)
    np.testing.assert_array_equal(nl, ref.nlist)
    assert pc.rel_l2(u, ref.u) < RTOL
    assert pc.rel_l2(force, ref.force) < 10 * RTOL


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("model", ["scalar", "tension", "field", "nlin"])
def test_corrections_of_broken_bonds(model, bad):
    """Every bond that breaks in the first step carries one that is not
    finite."""
    nlin, tension = model == "nlin", model == "tension"
    w = (configs.composite_ec if nlin else configs.beam_vv)(shape=(13, 6, 5))
    n, k = w.nlist.shape
    rng = np.random.default_rng(6)
    u = rng.normal(scale=(4e-3 if nlin else 2e-3) * w.extra["dx"],
                   size=(n, 3))
    corr = rng.uniform(0.5, 2.0, (n, k))
    field = w.bond_stiffness * rng.uniform(0.5, 2, n) if model == "field" \
        else None
    # the n-linear bonds start in their last regime, so that some break at once
    reg = np.full((n, k), 2, np.int32) if nlin else None
    dens, bt = (w.densities, w.bond_types) if nlin else (None, None)

    def reference():
        return oracle.SlotStepper(
            1 if nlin else 0, 1e-8 if nlin else 2e-15, w.coords, w.volume,
            w.family, w.bc_types, w.bc_values, w.force_bc_types,
            w.force_bc_values, w.nlist, w.bond_stiffness, w.critical_stretch,
            damping=2.5e6 if nlin else 0.0, densities=dens,
            stiffness_corrections=corr, bond_types=bt, regimes=reg,
            plus_cs=w.plus_cs, nregimes=w.nregimes, cnode=field,
            tension_only=tension, u=u)

    first = reference()
    first(1e-8, 0.5)
    gone = (w.nlist >= 0) & (first.nlist < 0)
    assert gone.sum() > 100
    corr[gone] = bad
    integ = (it.EulerCromerHIP(2.5e6, 1e-8) if nlin else it.EulerHIP(2e-15))
    integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                w.bc_values, w.force_bc_types, w.force_bc_values, corr, bt,
                dens)
    integ.set_node_stiffness(field)
    integ.set_break_mode(tension)
    for _ in range(2):  # as set up, and restarted on the same bonds
        integ.create_buffers(w.nlist, w.n_neigh, w.bond_stiffness,
                             w.critical_stretch, w.plus_cs, u, None, None,
                             None, None, None, reg, w.nregimes, w.nbond_types)
        _oracle_parity(integ, reference(), 4)


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("where", ["bond_stiffness", "plus_cs"])
@pytest.mark.parametrize("given", ["at set-up", "at a restart"])
def test_damage_tables_of_unused_types(given, where, bad):
    """Type 0, whose row of the tables padding slots name, has no bond."""
    w = configs.composite_ec(shape=(13, 6, 5))
    n, k = w.nlist.shape
    bt = np.where(w.nlist >= 0, w.bond_types + 1, 0).astype(np.int32)
    tables = {name: np.vstack([t[:1], t]) for name, t in (
        ("bond_stiffness", w.bond_stiffness), ("plus_cs", w.plus_cs),
        ("critical_stretch", w.critical_stretch))}
    u = np.random.default_rng(6).normal(scale=2e-3 * w.extra["dx"],
                                        size=(n, 3))
    integ = it.EulerCromerHIP(2.5e6, 1e-8)
    integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                w.bc_values, w.force_bc_types, w.force_bc_values, None, bt,
                w.densities)
    for finite in ([True, False, True] if given == "at a restart"
                   else [False]):
        t = {name: a.copy() for name, a in tables.items()}
        if not finite:
            t[where][0] = bad
        integ.create_buffers(w.nlist, w.n_neigh, t["bond_stiffness"],
                             t["critical_stretch"], t["plus_cs"], u, None,
                             None, None, None, None, None, 3, 4)
        ref = oracle.SlotStepper(
            1, 1e-8, w.coords, w.volume, w.family, w.bc_types, w.bc_values,
            w.force_bc_types, w.force_bc_values, w.nlist, t["bond_stiffness"],
            t["critical_stretch"], damping=2.5e6, densities=w.densities,
            bond_types=bt, plus_cs=t["plus_cs"], nregimes=3, u=u)
        _oracle_parity(integ, ref, 6)


def _gradient(w, u, dL, c=None, volume=None, nlist=None, lanes=4, coords=None):
    """dL/dc after six recorded steps, and the arrays they leave."""
    n, k = w.nlist.shape
    nl = w.nlist if nlist is None else nlist
    integ = it.EulerHIP(2e-15)
    integ.build(n, 3, k, w.coords if coords is None else coords,
                w.volume if volume is None else volume, w.family,
                np.zeros_like(w.bc_types), w.bc_values, w.force_bc_types,
                w.force_bc_values, None, None, None)
    integ.set_launch(lanes, 128)
    integ.set_node_stiffness(c)
    integ.create_buffers(nl, (nl >= 0).sum(axis=1).astype(np.int32),
                         w.bond_stiffness, w.critical_stretch, None, u, None,
                         None, None, None, None, None, 1, 1)
    integ.adjoint_start(6, checkpoint_every=6)
    integ.run(6, np.zeros(6), np.ones(6))
    return integ.adjoint_backward(dL), _arrays(integ)


@pytest.mark.parametrize("lanes", [1, 4, 8])
@pytest.mark.parametrize("what", ["c", "dL_du", "u", "volume"])
def test_gradient_of_nodes_without_bonds(what, lanes):
    """Their own values reach neither their own gradient nor a neighbour's."""
    w = configs.beam_vv(shape=(13, 6, 5))
    n = w.nnodes
    alone = np.array([3, 140, n - 1])
    nl = np.where(np.isin(w.nlist, alone), -1, w.nlist)
    nl[alone] = -1
    rng = np.random.default_rng(6)
    args = dict(u=rng.normal(scale=2e-3 * w.extra["dx"], size=(n, 3)),
                dL_du=rng.normal(size=(n, 3)), volume=w.volume,
                c=w.bond_stiffness * rng.uniform(0.5, 2, n))
    grads = []
    for value in [1.0] + BAD:
        a = {name: v.copy() for name, v in args.items()}
        a[what][alone] = value
        g, end = _gradient(w, a["u"], a["dL_du"], a["c"], a["volume"], nl,
                           lanes)
        assert end[7].sum() < (nl >= 0).sum()  # bonds break on the way
        grads.append(g)
    assert np.all(np.isfinite(grads[0])) and np.any(grads[0] != 0.0)
    assert np.all(grads[0][alone] == 0.0)
    for g in grads[1:]:
        np.testing.assert_array_equal(g, grads[0])


@pytest.mark.parametrize("lanes", [1, 4, 8])
def test_gradient_with_a_bond_of_no_length(lanes):
    """Its stretch is NaN or infinite, so the first step breaks it: the
    gradient is that of the body without it."""
    w = configs.beam_vv(shape=(13, 6, 5))
    n = w.nnodes
    i = 140
    j = int(w.nlist[i, 5])
    coords = w.coords.copy()
    coords[j] = coords[i]
    without = w.nlist.copy()
    for a, b in ((i, j), (j, i)):
        without[a][without[a] == b] = -1
    rng = np.random.default_rng(6)
    u = rng.normal(scale=1e-3 * w.extra["dx"], size=(n, 3))
    dL = rng.normal(size=(n, 3))
    c = w.bond_stiffness * rng.uniform(0.5, 2, n)
    got, end = _gradient(w, u, dL, c, lanes=lanes, coords=coords)
    want, end2 = _gradient(w, u, dL, c, nlist=without, lanes=lanes,
                           coords=coords)
    np.testing.assert_array_equal(end[6], end2[6])
    assert np.all(np.isfinite(want)) and np.any(want != 0.0)
    assert pc.rel_l2(got, want) < RTOL


def test_broken_nlinear_bonds_cost_no_more_than_live_ones():
    """A body all of whose bonds broke past their last regime against the
    same body whole, timed in turn."""
    w = configs.composite_ec(shape=(120, 24, 24))
    n, k = w.nlist.shape
    zeros = np.zeros((n, 3), np.int32)
    sims = []
    for torn in (False, True):
        integ = it.EulerCromerHIP(2.5e6, 1e-14)
        integ.build(n, 3, k, w.coords, w.volume, w.family, zeros, w.bc_values,
                    zeros, w.force_bc_values, None, w.bond_types, w.densities)
        u = (2.0 * w.coords if torn else
             np.random.default_rng(1).normal(scale=1e-5 * w.extra["dx"],
                                             size=(n, 3)))
        integ.create_buffers(w.nlist, w.n_neigh, w.bond_stiffness,
                             w.critical_stretch, w.plus_cs, u, None, None,
                             None, None, None, None, 3, 3)
        integ.run(6, np.zeros(6), np.zeros(6))
        assert integ.live_bonds() == (0 if torn else w.n_neigh.sum())
        sims.append(integ)
    best = [1e9, 1e9]
    for rep in range(60):  # fifteen times, and more on a noisy machine
        if rep >= 15 and best[1] < 1.05 * best[0]:
            break
        for q, integ in enumerate(sims):
            best[q] = min(best[q], integ.timed_run(40, np.zeros(40),
                                                   np.zeros(40)))
    print("whole, torn:", best)
    assert best[1] < 1.05 * best[0]
