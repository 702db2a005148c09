"""The two roundings that many kernels share (csrc/kernels/common.h): quotients by
a shared divisor in fused steps, against plain division, on the CPU; and f32 to
bf16, against the oracle's integer form, on the GPU."""
import numpy as np
import pytest

import catena_amd as ca
import oracle


def _fma(a, b, c):
    """RN(a * b + c) of float32 arrays, one rounding: the product is exact in
    float64, the sum is rounded there to odd (the low bit set when anything was
    cut off), which leaves the rounding to float32 correct, subnormals too."""
    p, c = a.astype(np.float64) * b.astype(np.float64), c.astype(np.float64)
    s = p + c
    t = s - p
    e = (p - (s - t)) + (c - t)  # the part of the sum that s has lost (TwoSum)
    bits = s.view(np.int64)
    away = (e > 0) == (s > 0)    # |exact| lies above |s|
    bits = np.where((e != 0) & (bits & 1 == 0), bits + np.where(away, 1, -1), bits)
    return bits.view(np.float64).astype(np.float32)


def _shared_quotient(a, b):
    """divide_shared's steps; b > 0"""
    hi = np.float32(1) / b
    lo = (_fma(-b, hi, np.ones_like(b)) * hi).astype(np.float32)
    q = _fma(a, hi, (a * lo).astype(np.float32))
    return _fma(_fma(-b, q, a), hi, q)


def test_fma_model():
    """The model against exact integers: operands of 24-bit mantissas near one
    another's magnitude, where every rounding case occurs."""
    from fractions import Fraction
    rng = np.random.default_rng(1)
    n = 4000
    a, b = (rng.integers(1 << 23, 1 << 24, n).astype(np.float32) for _ in range(2))
    c = (-(a.astype(np.float64) * b) * rng.choice([0.5, 1, 1.0001, 2], n)).astype(np.float32)
    got = _fma(a, b, c)
    for x, y, z, g in zip(a, b, c, got):
        exact = Fraction(float(x)) * Fraction(float(y)) + Fraction(float(z))
        err = abs(Fraction(float(g)) - exact)
        for near in (np.nextafter(g, np.float32(np.inf)), np.nextafter(g, np.float32(-np.inf))):
            d = abs(Fraction(float(near)) - exact)
            assert err < d or (err == d and not g.view(np.uint32) & 1)


# the bounds that divide_shared's fast path states
B_EXP, A_EXP = (-20, 20), (-98, 100)


def test_shared_divisor_quotients():
    """Correctly rounded over the whole range of the fast path: extreme mantissas
    at every pair of edge exponents, quotients beside ties and beside floats,
    and random pairs."""
    rng = np.random.default_rng(2)
    edge = np.concatenate([np.arange(8), (1 << 23) - 1 - np.arange(8), (1 << 22) + np.arange(-4, 4), rng.integers(0, 1 << 23, 40)])
    mant = (1 + edge / 2.0 ** 23).astype(np.float64)
    total = 0
    with np.errstate(under="ignore"):
        for eb in (-20, -19, -1, 0, 1, 19):
            for ea in (-98, -97, -60, -1, 0, 1, 60, 98, 99):
                a, b = np.meshgrid(mant * 2.0 ** ea, mant * 2.0 ** eb)
                a, b = a.astype(np.float32).ravel(), b.astype(np.float32).ravel()
                assert np.array_equal(_shared_quotient(a, b).view(np.uint32), (a / b).view(np.uint32)), (ea, eb)
                total += a.size
        one = np.full(edge.size, 2.0 ** 20, np.float32)  # the top of b's range itself
        a = (mant * 2.0 ** -98).astype(np.float32)
        assert np.array_equal(_shared_quotient(a, one).view(np.uint32), (a / one).view(np.uint32))
        for _ in range(8):
            n = 1 << 19
            b = ((1 + rng.integers(0, 1 << 23, n) / 2.0 ** 23) * 2.0 ** rng.integers(B_EXP[0], B_EXP[1], n)).astype(np.float32)
            q = 1 + rng.integers(0, 1 << 24, n) / 2.0 ** 24  # floats and the ties between them
            a = (b.astype(np.float64) * q * 2.0 ** rng.integers(-70, 70, n)).astype(np.float32)
            a = np.nextafter(a, np.where(rng.random(n) < 0.5, np.float32(np.inf), np.float32(0))) if _ % 2 else a
            a = (a * rng.choice([-1, 1], n)).astype(np.float32)
            assert np.array_equal(_shared_quotient(a, b).view(np.uint32), (a / b).view(np.uint32))
            a = ((1 + rng.integers(0, 1 << 23, n) / 2.0 ** 23) * 2.0 ** rng.integers(A_EXP[0], A_EXP[1], n)).astype(np.float32)
            assert np.array_equal(_shared_quotient(a, b).view(np.uint32), (a / b).view(np.uint32))
            total += 2 * n
    assert total > 8e6


def _conversion_inputs():
    """Every high half with the low halves around the tie and around a float."""
    low = np.array([0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF, 0x5555, 0xC3A1], np.uint32)
    return ((np.arange(1 << 16, dtype=np.uint32)[:, None] << 16) | low[None]).reshape(-1).view(np.float32)


@pytest.mark.gpu
def test_bf16_conversion_of_every_high_half():
    """The bits of the oracle's integer form, signs and payloads of NaNs
    included: the v rows that rope_qkv_bf16 stores are converted and nothing
    else."""
    ca.init(0)
    x, heads = _conversion_inputs(), 16
    rows = x.size // (heads * 128)
    qkv = np.zeros((rows, 3, heads * 128), np.float32)
    qkv[:, 2] = x.reshape(rows, -1)
    print(f"[gpu-case] bf16 conversion of {x.size} values", flush=True)
    vc, kc, q = (ca.Buffer(heads * rows * 128 * 2) for _ in range(3))
    ca.rope_qkv_bf16(ca.Buffer.from_array(qkv), ca.Buffer.from_array(np.zeros(64, np.float32)),
                     ca.Buffer.from_array(np.array([rows], np.uint32)), q, kc, vc, 1, rows, heads, 128, rows)
    got = vc.read(np.uint16, (heads, rows, 128)).transpose(1, 0, 2).reshape(-1)
    assert np.array_equal(got, oracle.f32_to_bf16_bits_np(x))


@pytest.mark.gpu
def test_bf16_conversion_in_pairs():
    """The same for two values an instruction, as products are stored: rows whose
    sum is one f32 value in three bf16 parts, exact in any order."""
    ca.init(0)
    x = _conversion_inputs()
    x = x[np.isfinite(x) & (np.abs(x) >= np.float32(2.0 ** -100)) & (np.abs(x) < np.float32(2.0 ** 127))]
    x = x[:x.size // 16 * 16]
    parts, rest = [], x
    for _ in range(3):
        head = (rest.view(np.uint32) & 0xFFFF0000).view(np.float32)
        parts.append((head.view(np.uint32) >> 16).astype(np.uint16))
        rest = rest - head
    assert not rest.any()
    a16 = np.zeros((x.size, 8), np.uint16)
    a16[:, 1], a16[:, 4], a16[:, 6] = parts
    one = np.full((8, 8), 0x3F80, np.uint16)
    print(f"[gpu-case] bf16 conversion in pairs of {x.size} values", flush=True)
    ab, bb = ca.Buffer.from_array(a16), ca.Buffer.from_array(one)
    c32, c16 = ca.Buffer(x.size * 32), ca.Buffer(x.size * 16)
    ca.gemm_bf16(ab, bb, c32, x.size, 8, 8, out_f32=True)
    ca.gemm_bf16(ab, bb, c16, x.size, 8, 8)
    assert np.array_equal(c32.read(np.float32, (x.size, 8)), np.repeat(x[:, None], 8, 1))
    assert np.array_equal(c16.read(np.uint16, (x.size, 8)), np.repeat(oracle.f32_to_bf16_bits_np(x)[:, None], 8, 1))
