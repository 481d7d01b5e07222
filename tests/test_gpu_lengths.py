"""Bond lengths and stretches of the step that sums in any order: correctly
rounded lengths, and break decisions that equal the rounded stretch's."""
import math
from fractions import Fraction

import numpy as np
import pytest

import oracle
from probabilistic_peridynamics_amd import _lib
from probabilistic_peridynamics_amd import integrators as it
from test_gpu_parity import _bond_batch

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip_device")]


def _pairs(layout, tension, s0, ui, uj, r0i, r0j, k=1.0):
    """One step of a body of bonds that share no node: (broken, force)."""
    m = len(r0i)
    n = 2 * m
    coords, u = np.empty((n, 3)), np.empty((n, 3))
    coords[0::2], coords[1::2], u[0::2], u[1::2] = r0i, r0j, ui, uj
    other = (np.arange(n) ^ 1).astype(np.int32)[:, None]
    ones, zeros = np.ones(n, np.int32), np.zeros((n, 3), np.int32)
    integ = (it.EulerHIP(1e-9) if layout == "slot" else
             it.Euler(1e-9, exact_order=False))
    integ.build(n, 3, 1, coords, np.ones(n), ones, zeros, u * 0, zeros, u * 0,
                None, None, None)
    integ.set_break_mode(tension)
    integ.create_buffers(other, ones, k, s0, None, u, None, None, None, None,
                         None, None, 1, 1)
    integ(0.0, 0.0)
    _, _, _, force, _, _, _, nn = integ.write(None, None, None, None, None,
                                              None, None, None)
    return nn[0::2] == 0, force


def _hard_squares():
    """Doubles q in [1, 4) whose root lies just above the middle between two
    doubles: q = (M^2 + r)/2^106 for an odd M of 54 bits and a small r, so
    that the root is M 2^-53 (1 + r/(2 M^2)), by r 2^-56 to r 2^-55 ulp off
    the middle.  r from 512 on: 7e-15 ulp, above what the error of the last
    correction's factor (5.4e-15, of half an ulp) does to the root."""
    out = []
    for r in range(519, 1 << 14, 8):  # -r is 1 modulo 8, a square mod 2^k
        for k in (54, 55):
            x = 1  # x^2 = -r modulo 2^k, bit by bit
            for b in range(3, k):
                if (x * x + r) >> b & 1:
                    x += 1 << (b - 1)
            for m in (x, -x, x + (1 << (k - 1)), -x + (1 << (k - 1))):
                m = m % (1 << k) % (1 << 54)
                q, rest = divmod(m * m + r, 1 << k)
                if rest == 0 and m >> 53 == 1 and 52 <= math.log2(q) < 53:
                    out.append(math.ldexp(q, k - 106))
    return out


def _vector(q, fused):
    """(x, y) whose computed squared length is exactly q: x^2 + y^2, or
    contracted as fma(x, x, y*y); y is small."""
    x = math.sqrt(q)
    square = lambda v: Fraction(v) ** 2 if fused else Fraction(v * v)
    while square(x) > Fraction(q):
        x = math.nextafter(x, 0.0) if hasattr(math, "nextafter") else float(
            np.nextafter(x, 0.0))
    y = math.sqrt(float(Fraction(q) - square(x)))
    got = float(square(x) + Fraction(y * y))
    return (x, y) if got == q else None


@pytest.mark.parametrize("layout", ["slot", "compact"])
def test_hard_lengths_are_rounded_correctly(layout):
    """A bond at rest whose length's rounding is hard to get: strained by
    nothing, it exerts no force."""
    r0j, uj = [], []
    for q in _hard_squares():
        v = _vector(q, layout == "slot")
        length = math.sqrt(q)
        # the reference length is a double whose computed square has that
        # double as its root, far from a middle
        root = Fraction(length * length) - Fraction(length) ** 2
        off = root / (2 * Fraction(length)) / Fraction(math.ulp(length))
        if v is None or abs(abs(off) - Fraction(1, 2)) < Fraction(1, 1000):
            continue
        r0j.append((length, 0.0, 0.0))
        uj.append((v[0] - length, v[1], 0.0))
    r0j, uj = np.array(r0j), np.array(uj)
    assert len(r0j) > 1000
    z = np.zeros_like(r0j)
    broken, force = _pairs(layout, False, 0.5, z, uj, z, r0j)
    assert not broken.any()
    np.testing.assert_array_equal(force, 0.0)


@pytest.mark.parametrize("opencl", [False, True])
@pytest.mark.parametrize("tension", [False, True])
def test_bond_check_is_the_step(tension, opencl):
    """pd_bond_check against steps of a body of such bonds and the oracle,
    with stretches within ulps of the threshold; from the stretch on at which
    the step divides (|s| >= 1/2), its working stretch is the divided one."""
    for s0, far in ((0.005, 0.02), (10.0, 0.9), (1e-13, 3e-13)):
        ri, rj, r0i, r0j = _bond_batch(seed=int(opencl), n=5000, s0=s0)
        rng = np.random.default_rng(9)
        target = rng.uniform(-far, far, len(ri))
        near = rng.random(len(ri)) < 0.33
        target[near] = rng.choice([-1, 1], near.sum()) * min(s0, far) * (
            1 + rng.integers(-8, 9, near.sum()) * 2.0 ** -52)
        d0 = r0j - r0i
        ui = rng.normal(scale=1e-3 * min(1, s0), size=ri.shape)
        uj = ui + d0 * target[:, None]
        ri, rj = (ui, uj) if opencl else (r0i + ui, r0j + uj)
        got = _lib.bond_check(ri, rj, r0i, r0j, s0, tension_only=tension,
                              opencl=opencl)
        s = np.array([oracle.cl_strain(*b)[0] if opencl else
                      oracle.strain(*b) for b in zip(ri, rj, r0i, r0j)])
        want = ~(s < s0) if tension else ~(np.abs(s) < s0)
        np.testing.assert_array_equal(got["s_exact"], s)
        np.testing.assert_array_equal(got["broken"].astype(bool), want)
        divided = np.abs(s) >= 0.5
        np.testing.assert_array_equal(got["s"][divided], s[divided])
        broken, _ = _pairs("slot" if opencl else "compact", tension, s0, ui,
                           uj, r0i, r0j)
        np.testing.assert_array_equal(broken, want)
        assert s0 == 10.0 or 0 < want.sum() < len(want)
        assert s0 != 10.0 or divided.sum() > 100
