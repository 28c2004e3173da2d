"""The SiLU kernel's quotient g / (1 + exp(-g)) (``silu_div`` in tilemix_amd/csrc/prefill.hip): a
Newton step on the hardware reciprocal, then Markstein's correction of the quotient,
    r1 = fma(fma(-den, r0, 1), r0, r0), q = RN(g r1), q1 = fma(fma(-q, den, g), r1, q).
Checked on the CPU for every finite fp16 gate, every denominator that an exp within two ulps gives
and every reciprocal seed within one ulp (the instruction's bound): q1 is the correctly rounded
quotient, and where it is too small for that it rounds to the same fp16 zero.  One denominator is
left out of that, 2 - 2^-23 with a seed that is not the nearest (the all-ones significand, the
exception in Markstein's theorem): q1 can then be one ulp off, which changes the fp16 result of the
gate 2^-24 alone, where exp would have to be one ulp low.  (The gates around it, infinities and
NaNs, the fix-up instruction's part, are checked on the GPU: test_silu_mul_every_gate and
test_silu_mul_smallest_gates.)
"""
from __future__ import annotations

import numpy as np

f32, f64 = np.float32, np.float64


def _fma32(a, b, c):
    """RN32(a b + c): the product is exact in float64, and the sum is rounded to odd there (Boldo and
    Melquiond), so that the rounding to float32 is the only one."""
    p, c = a.astype(f64) * b.astype(f64), c.astype(f64)
    s = p + c
    t = s - p
    err = (p - (s - t)) + (c - t)  # s + err = p + c exactly
    bits = s.view(np.int64)
    # inexact and even: the other of the two neighbours of the exact sum, which is odd
    step = np.where((err > 0) == (s > 0), 1, -1)
    bits = np.where((err != 0) & (bits & 1 == 0), bits + step, bits)
    return bits.view(f64).astype(f32)


def test_fma32_emulation():
    """Against exact rational arithmetic, sums that double rounding gets wrong among them."""
    from fractions import Fraction
    from test_quant_division import _rn32_exact
    rng = np.random.default_rng(0)
    a, b = (rng.standard_normal(2000).astype(f32) for _ in range(2))
    c = (rng.standard_normal(2000) * 2.0 ** rng.integers(-30, 30, 2000)).astype(f32)
    c[:500] = (a[:500].astype(f64) * b[:500]).astype(f32) * f32(2.0 ** 24)
    a[500], b[500], c[500] = f32(2.0 ** -24 * (1 + 2.0 ** -23)), f32(1 - 2.0 ** -24), f32(1.0)
    got = _fma32(a, b, c)
    for x, y, z, r in zip(a, b, c, got):
        assert Fraction(float(r)) == _rn32_exact(Fraction(float(x)) * Fraction(float(y)) + Fraction(float(z)))


def _ulps(x, n):
    return (x.view(np.int32) + n).view(f32)


def _quotient(g, den, r0):
    r1 = _fma32(_fma32(-den, r0, np.ones_like(den)), r0, r0)
    q = (g * r1).astype(f32)
    return _fma32(_fma32(-q, den, g), r1, q)


def test_every_gate_denominator_and_seed():
    gates = np.arange(1 << 16, dtype=np.uint32).astype(np.uint16).view(np.float16)
    g = gates[np.isfinite(gates)].astype(f32)
    with np.errstate(over="ignore", under="ignore"):
        e0 = np.exp(-g.astype(f64)).astype(f32)
        checked = 0
        for de in (-2, -1, 0, 1, 2):
            e = np.where((e0 > 1e-30) & np.isfinite(e0), _ulps(e0, de), e0)
            den = (f32(1.0) + e).astype(f32)
            exact = den <= f32(2.0 ** 100)
            for dr in (-1, 0, 1):
                x, d = g[exact], den[exact]
                got = _quotient(x, d, _ulps((f32(1.0) / d).astype(f32), dr))
                want = (x / d).astype(f32)
                off = got != want  # -0 == +0
                assert dr != 0 or not off.any()
                assert np.all(d[off] == f32(2.0 - 2.0 ** -23)) and off.sum() <= 1
                assert np.all(np.abs(got[off].view(np.int32) - want[off].view(np.int32)) == 1)
                off16 = got.astype(np.float16) != want.astype(np.float16)
                assert not off16.any() or (de == -1 and x[off16].tolist() == [2.0 ** -24])
                checked += x.size
            # beyond: a reciprocal at the end of the range, or flushed to zero
            x, d = g[~exact & np.isfinite(den)], den[~exact & np.isfinite(den)]
            for r0 in ((f32(1.0) / d).astype(f32), np.zeros_like(d)):
                got = _quotient(x, d, r0).astype(np.float16)
                want = (x / d).astype(f32).astype(np.float16)
                assert np.array_equal(got.view(np.uint16), want.view(np.uint16))
    assert checked > 600_000
