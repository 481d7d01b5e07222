"""n-linear tables near the largest double: the step scales them by powers of
two, which must not make infinite what the force itself holds."""
import numpy as np
import pytest

import oracle
import pdcases as pc
from probabilistic_peridynamics_amd import configs
from probabilistic_peridynamics_amd import integrators as it

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip_device")]

MOST = np.finfo(np.float64).max


@pytest.mark.parametrize("corrections", [False, True])
@pytest.mark.parametrize("name,value", [
    ("bond_stiffness", MOST), ("bond_stiffness", -1e308),
    ("bond_stiffness", MOST / 4), ("plus_cs", MOST), ("plus_cs", -1e308)])
def test_forces_of_huge_tables(name, value, corrections):
    """The force of one step, finite in the oracle, at 1e-9 of its norm (as
    the damage model's other parity tests)."""
    w = configs.composite_ec(shape=(13, 6, 5))
    n, k = w.nlist.shape
    rng = np.random.default_rng(6)
    tables = {"bond_stiffness": w.bond_stiffness.copy(),
              "plus_cs": w.plus_cs.copy()}
    tables[name][1, 0] = value
    u = rng.normal(scale=2e-4 * w.extra["dx"], size=(n, 3))
    # plus_cs / l V stays finite, summed over a node's bonds
    volume = np.full(n, 1e-9)
    corr = rng.uniform(0.25, 0.9, (n, k)) if corrections else None
    integ = it.EulerCromerHIP(2.5e6, 0.0)
    integ.build(n, 3, k, w.coords, volume, w.family, w.bc_types, w.bc_values,
                w.force_bc_types, w.force_bc_values, corr, w.bond_types,
                w.densities)
    ref = oracle.SlotStepper(
        1, 0.0, w.coords, volume, w.family, w.bc_types, w.bc_values,
        w.force_bc_types, w.force_bc_values, w.nlist,
        tables["bond_stiffness"], w.critical_stretch, damping=2.5e6,
        densities=w.densities, stiffness_corrections=corr,
        bond_types=w.bond_types, plus_cs=tables["plus_cs"],
        nregimes=w.nregimes, u=u)
    ref(0.0, 0.0)
    assert np.all(np.isfinite(ref.force)) and np.abs(ref.force).max() > 1e290
    integ.create_buffers(w.nlist, w.n_neigh, tables["bond_stiffness"],
                         w.critical_stretch, tables["plus_cs"], u, None, None,
                         None, None, None, None, w.nregimes, w.nbond_types)
    integ(0.0, 0.0)
    _, _, _, force, _, _, nl, _ = integ.write(None, None, None, None, None,
                                              None, None, None)
    np.testing.assert_array_equal(nl, ref.nlist)
    big = np.abs(ref.force).max()
    assert pc.rel_l2(force / big, ref.force / big) < 1e-9
