"""Buffers that are created anew hold the new state: force and body force of
the run before are gone, whether the bonds are the same or others."""
import numpy as np
import pytest

from probabilistic_peridynamics_amd import configs
from probabilistic_peridynamics_amd import integrators as it

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip_device")]


@pytest.mark.parametrize("layout", ["slot", "compact"])
@pytest.mark.parametrize("others", [False, True])
def test_no_force_of_the_run_before(layout, others):
    w = configs.beam_vv(shape=(13, 6, 5), layout=layout)
    n, k = w.nlist.shape
    rng = np.random.default_rng(2)
    # a body force on some nodes, whose force and body_force differ
    fbt = np.zeros((n, 3), w.force_bc_types.dtype)
    fbt[rng.random(n) < 0.2] = 1
    integ = it.EulerHIP(2e-15) if layout == "slot" else it.Euler(2e-15)
    integ.build(n, 3, k, w.coords, w.volume, w.family, w.bc_types,
                w.bc_values, fbt, np.ones((n, 3)), None, None, None)
    nl, nn = w.nlist.copy(), w.n_neigh.copy()
    u = rng.normal(scale=1e-3 * w.extra["dx"], size=(n, 3))

    def create():
        integ.create_buffers(nl, nn, w.bond_stiffness, w.critical_stretch,
                             None, u, None, None, None, None, None, None, 1,
                             1)
        return integ.write(*[np.full((n, 3), 7.0) for _ in range(5)], None,
                           None, None)

    create()
    integ(0.0, 1.0)
    assert np.any(integ.write(*[None] * 8)[3] != 0.0)
    if others:  # the last node without bonds: other rows, other tiles
        last = int(nn[n - 1])
        for j in w.nlist[n - 1, :last]:
            row = list(nl[j, :nn[j]])
            row.remove(n - 1)
            nl[j] = -1 if layout == "slot" else 0
            nl[j, :len(row)] = row
            nn[j] -= 1
        nl[n - 1] = -1 if layout == "slot" else 0
        nn[n - 1] = 0
    got = create()
    np.testing.assert_array_equal(got[0], u)
    np.testing.assert_array_equal(got[3], 0.0)
    np.testing.assert_array_equal(got[4], 0.0)
