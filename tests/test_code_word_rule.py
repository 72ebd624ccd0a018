"""CPU: the rounding rule of the KV writers (csrc/device_common.hpp code_words),
restated in numpy, gives the codes of the correctly rounded quotient
rint(fl(x / s)) for fp16 x with |x| <= absmax and s = fl(absmax / qmax), for
every reciprocal within 1 ulp of 1 / s. fma(x, r, c) is computed in float64
from the exact product (11 + 24 bits) and rounded once to float32."""
from __future__ import annotations

import numpy as np

F = np.float32
MAGIC = 12582912.0
WINDOW = {7: 2.0 ** -18, 127: 2.0 ** -14}


def _round_to_magic(z):
    """fl32(z + MAGIC) for |z| < 2^22: z rounded to an integer, half to even
    (the float64 sum below could round z's tail away first, so rint)."""
    return np.rint(z)


def _codes(x, s, r, qmax, fallback=True):
    z = x.astype(np.float64) * r.astype(np.float64)            # exact: 35 bits
    k = _round_to_magic(z)
    d = np.abs((z - k).astype(F))                              # fma(x, r, -k), rounded once
    if not fallback:
        return k
    near = d >= F(0.5 - WINDOW[qmax])
    return np.where(near, np.rint((x.astype(F) / s).astype(F)), k)


def _cases(rng, qmax, n=300_000):
    """fp16 maxima over the whole range and values up to them: random ones,
    the multiples nearest to half-integer quotients, and their neighbours."""
    amax = rng.integers(1, 0x7C00, n).astype(np.uint16).view(np.float16)
    s = np.maximum((amax.astype(F) / F(qmax)).astype(F), F(1e-8))
    half = (rng.integers(-qmax, qmax, n) + 0.5) * s.astype(np.float64)
    near = half.astype(np.float16)
    xs = [near, np.nextafter(near, np.float16(np.inf)), np.nextafter(near, np.float16(-np.inf)),
          (rng.uniform(-1, 1, n) * amax.astype(np.float64)).astype(np.float16), amax, -amax,
          (amax.astype(np.float64) / 2).astype(np.float16)]
    x = np.concatenate(xs)
    a = np.tile(amax, len(xs))
    x = np.where(np.abs(x) <= a, x, a)
    return x, np.tile(s, len(xs)), a


def test_codes_equal_the_correctly_rounded_quotients():
    rng = np.random.default_rng(11)
    for qmax in (7, 127):
        x, s, _ = _cases(rng, qmax)
        want = np.rint((x.astype(F) / s).astype(F))
        assert np.abs(want).max() == qmax    # no clamp needed
        r0 = (F(1.0) / s).astype(F)
        for shift in (-1, 0, 1):
            r = r0 if shift == 0 else np.nextafter(r0, F(np.inf) if shift > 0 else F(-np.inf)).astype(F)
            assert np.array_equal(_codes(x, s, r, qmax), want), (qmax, shift)


def test_planted_no_fallback_fails():
    rng = np.random.default_rng(12)
    for qmax in (7, 127):
        x, s, _ = _cases(rng, qmax)
        r = np.nextafter((F(1.0) / s).astype(F), F(np.inf)).astype(F)
        assert not np.array_equal(_codes(x, s, r, qmax, fallback=False), np.rint((x.astype(F) / s).astype(F)))


def test_magic_word_holds_the_code_bits():
    """The low byte / nibble of fl32(code + MAGIC) is the two's complement code,
    and of the fp32 form of every fp16 NaN and of the default NaN is 0."""
    k = np.arange(-127, 128)
    bits = (k.astype(F) + F(MAGIC)).view(np.uint32)
    assert np.array_equal(bits & 0xFF, (k & 0xFF).astype(np.uint32))
    nan = np.concatenate([np.arange(0x7C01, 0x8000), np.arange(0xFC01, 0x10000)]).astype(np.uint16)
    f32 = (((nan.astype(np.uint32) & 0x8000) << 16) | 0x7F800000 | ((nan.astype(np.uint32) & 0x3FF) << 13))
    assert not (f32 & 0xFF).any() and not (np.array([0x7FC00000, 0xFFC00000]) & 0xFF).any()
