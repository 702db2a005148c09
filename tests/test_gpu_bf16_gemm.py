"""GPU parity of the bf16 MFMA GEMM (tile, edge and decode kernels).

The MFMA datapath sums in its own order, so against the reference-order
sequential oracle the check is an error bound, stated here:

  f32 output:  |C_gpu - C_exact| <= 8 * (K/32 + 1) * u * sum_k |A_ik B_kj|
               (K/32 dependent MFMA accumulation steps, each rounding to f32
               a bounded number of times; u = 2^-24; C_exact in float64);
  bf16 output: |C16_gpu - C16_oracle| <= delta + 1 ulp_bf16, with delta the
               f32-level distance bound above plus the oracle's own sequential
               bound K * u * sum|A B|.

Alongside it, the bf16 output must be bitwise RNE(f32 output) of the same
kernel (same accumulation order), and results are bitwise identical from run
to run (fixed tile->workgroup map, fixed K order, no atomics).
"""
import math

import numpy as np
import pytest

import catena_amd as ca
import oracle
from gpu_util import U, as_f32, bf16_ulp_diff, bf16_ulp_of, captured, dev_normal_bf16, gemm_within_bound, hash_bits, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _init():
    say("init device 0")
    ca.init(0)


def _inputs(n, m, k, seed, wscale=1.0):
    a = dev_normal_bf16(n * k, seed, 0, 1.0)
    b = dev_normal_bf16(k * m, seed, 1, wscale)
    return a, b, a.read(np.uint16, (n, k)), b.read(np.uint16, (k, m))


def _check(a16, b16, got32, got16, rows=None):
    af = as_f32(a16).astype(np.float64)
    bf = as_f32(b16).astype(np.float64)
    if rows is not None:
        af = af[rows]
    k = a16.shape[1]
    exact = af @ bf
    absprod = np.abs(af) @ np.abs(bf)
    mfma_bound = 8 * (k / 32 + 1) * U * absprod
    seq32, seq16 = oracle.matmul_bf16(a16, b16, rows=rows)
    stats = {}
    if got32 is not None:
        err = np.abs(got32.astype(np.float64) - exact)
        assert np.all(err <= mfma_bound), float((err / np.maximum(mfma_bound, 1e-300)).max())
        stats["f32_max_err_over_u_absprod"] = float((err / (U * np.maximum(absprod, 1e-300))).max())
        stats["f32_bitwise_equal_to_sequential_frac"] = float(np.mean(got32 == seq32))
    if got16 is not None:
        delta = mfma_bound + k * U * absprod
        g = as_f32(got16).astype(np.float64)
        s = as_f32(seq16).astype(np.float64)
        tol = delta + bf16_ulp_of(np.maximum(np.abs(g), np.abs(s)))
        assert np.all(np.abs(g - s) <= tol)
        ulps = bf16_ulp_diff(got16, seq16)
        stats["bf16_max_ulp_vs_sequential"] = int(ulps.max())
        stats["bf16_equal_frac"] = float(np.mean(ulps == 0))
        stats["bf16_le1ulp_frac"] = float(np.mean(ulps <= 1))
    print("[bf16-gemm-stats]", stats, flush=True)
    return stats


# few tiles (general kernels); 256 x 256 tiles with 32-k stages; with 64-k stages
@pytest.mark.parametrize("n,m,k,tiled", [(256, 256, 64, False), (512, 256, 1024, False), (256, 768, 320, False),
                                         (4096, 2304, 128, True), (2560, 2048, 64, True), (2560, 2048, 192, True)])
def test_tile_kernel_full_compare(n, m, k, tiled):
    assert (ca.gemm_bf16_plan(n, m, k)[2:] == (0, 0)) == tiled
    say(f"bf16 gemm tile {n}x{m}x{k}")
    a, b, a16, b16 = _inputs(n, m, k, seed=100 + n + m + k)
    c32, c16 = ca.Buffer(n * m * 4), ca.Buffer(n * m * 2)
    ca.gemm_bf16(a, b, c32, n, m, k, out_f32=True)
    ca.gemm_bf16(a, b, c16, n, m, k, out_f32=False)
    g32, g16 = c32.read(np.float32, (n, m)), c16.read(np.uint16, (n, m))
    assert np.array_equal(g16, oracle.f32_to_bf16_bits_np(g32))
    _check(a16, b16, g32, g16)


def test_tile_widths_give_identical_bits():
    """The 256 x 256 and 256 x 128 tile kernels and the general ones keep the
    same per-accumulator k32 order, so a cell's bits do not depend on which one
    computed it: of 2304 columns, 4096 rows take 256 x 256 tiles (144 of them;
    the 288 narrow ones would be two rounds of the chip), their first 2304 rows
    alone 256 x 128 tiles (one round), their first 512 the general kernels."""
    n, m, k = 4096, 2304, 1024
    say(f"bf16 gemm tile widths {n}x{m}x{k} vs 2304 and 512 rows")
    assert [ca.gemm_bf16_plan(r, m, k)[2:] == (0, 0) for r in (n, 2304, 512)] == [True, True, False]
    a, b, _, _ = _inputs(n, m, k, seed=901)
    for out_f32, dt, es in ((False, np.uint16, 2), (True, np.uint32, 4)):
        full = ca.Buffer(n * m * es)
        ca.gemm_bf16(a, b, full, n, m, k, out_f32=out_f32)
        for rows in (2304, 512):
            part = ca.Buffer(rows * m * es)
            ca.gemm_bf16(a, b, part, rows, m, k, out_f32=out_f32)
            assert np.array_equal(full.read(dt, (n, m))[:rows], part.read(dt, (rows, m)))


# 12 narrow tiles: general kernels on both sides; 160 and 320: the 64-k kernel
# against 256 x 128 and 256 x 256 tiles
@pytest.mark.parametrize("n,m,k", [(512, 768, 4160), (2560, 2048, 448), (5120, 2048, 192)])
def test_k64_kernel_equals_k32_kernel_on_zero_padded_k(n, m, k):
    """K % 128 != 0 takes the two-stage 64-k kernel, K % 128 == 0 the
    four-stage 32-k kernel; both add k32 MFMA steps in ascending order, so
    padding K with 64 zero columns of A (and zero rows of B) gives the same
    bits: the extra steps add exact zeros to nonzero sums."""
    kp = k + 64
    assert (ca.gemm_bf16_plan(n, m, k)[2:] == (0, 0)) == (n >= 2560) == (ca.gemm_bf16_plan(n, m, kp)[2:] == (0, 0))
    rng = np.random.default_rng(902)
    a32 = rng.normal(0, 1, (n, k)).astype(np.float32)
    b32 = rng.normal(0, 1, (k, m)).astype(np.float32)
    a16, b16 = oracle.f32_to_bf16_bits_np(a32), oracle.f32_to_bf16_bits_np(b32)
    ap = np.zeros((n, kp), np.uint16)
    ap[:, :k] = a16
    bp = np.zeros((kp, m), np.uint16)
    bp[:k] = b16
    say(f"bf16 gemm 64-k kernel {n}x{m}x{k} vs 32-k kernel on K={kp}")
    outs = []
    for aa, bb, kk in ((a16, b16, k), (ap, bp, kp)):
        c32 = ca.Buffer(n * m * 4)
        ca.gemm_bf16(ca.Buffer.from_array(aa), ca.Buffer.from_array(bb), c32, n, m, kk, out_f32=True)
        outs.append(c32.read(np.uint32, (n, m)))
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("n,m,k,tiled", [(256, 384, 256, False), (512, 128, 1152, False), (2560, 1664, 256, True)])
def test_narrow_tile_kernel_full_compare(n, m, k, tiled):
    """N % 256 == 128: of the tile kernels only the 256 x 128 one applies (few
    tiles go to the general kernels)."""
    assert (ca.gemm_bf16_plan(n, m, k)[2:] == (0, 0)) == tiled
    say(f"bf16 gemm 256x128 tiles {n}x{m}x{k}")
    a, b, a16, b16 = _inputs(n, m, k, seed=400 + n + m + k)
    c32, c16 = ca.Buffer(n * m * 4), ca.Buffer(n * m * 2)
    ca.gemm_bf16(a, b, c32, n, m, k, out_f32=True)
    ca.gemm_bf16(a, b, c16, n, m, k, out_f32=False)
    g32, g16 = c32.read(np.float32, (n, m)), c16.read(np.uint16, (n, m))
    assert np.array_equal(g16, oracle.f32_to_bf16_bits_np(g32))
    _check(a16, b16, g32, g16)


@pytest.mark.parametrize("n,m,k", [(1, 1, 1), (17, 9, 5), (300, 200, 100), (257, 513, 72),
                                   (64, 64, 63)])
@pytest.mark.parametrize("graph", [False, True])
def test_edge_kernel_full_compare(n, m, k, graph):
    """Sizes no tile divides: the general kernels, and, captured into a graph,
    where rows off 16 bytes cannot be packed, the bounds-checked kernel."""
    say(f"bf16 gemm edge {n}x{m}x{k} graph {graph}")
    a, b, a16, b16 = _inputs(n, m, k, seed=200 + n + m + k)
    if graph:  # one element off 16 bytes
        a = ca.Buffer.from_array(np.concatenate([np.zeros(1, np.uint16), a16.reshape(-1)]))
    ap = a.ptr + 2 if graph else a
    c32, c16 = ca.Buffer(n * m * 4), ca.Buffer(n * m * 2)
    for c in (c32, c16):
        run = lambda: ca.gemm_bf16(ap, b, c, n, m, k, out_f32=c is c32)  # noqa: E731,B023
        (captured(run) if graph else run)()
    g32, g16 = c32.read(np.float32, (n, m)), c16.read(np.uint16, (n, m))
    assert np.array_equal(g16, oracle.f32_to_bf16_bits_np(g32))
    _check(a16, b16, g32, g16)


def test_gemm_4096_full_compare_and_run_to_run():
    """The C2 workload (4096^3, N(0,1) bf16 inputs from seed 3): every one of
    the 16.8M output cells against the sequential-order oracle
    (catena-lang/src/codegen/ops/reducec.rs:73-130 on widened bf16), under
    the error bound above and a stated max-ULP bound, and bitwise run to run.

    Max-ULP bound.  With d = (8 (K/32 + 1) + K) u sum|A B| the f32-level
    distance bound of the GPU and oracle values, the two bf16 results of a
    cell differ by at most 1 + ceil(d / ulp) bf16 ulps, ulp the bf16 spacing
    at the smaller of the two magnitudes.  That bound grows with the cell's
    condition kappa = sum|A B| / |C|: d <= 5128 u kappa |C| and ulp >=
    2^-8 (1 - 5128 u kappa) |C|, so at most 1 + ceil(256 * 5128 u kappa /
    (1 - 5128 u kappa)) ulps -- 7 ulps for kappa <= 64 (N(0,1) data puts
    about half the cells there; the rest sit near a cancellation, |C| << sum
    |A B|).  Asserted: every cell within its own bound, every cell with
    kappa <= 64 within 7 ulps; printed: the max ulps overall and per kappa
    band and the identical fraction."""
    n = m = k = 4096
    say("bf16 gemm 4096^3")
    a, b, a16, b16 = _inputs(n, m, k, seed=3)
    c16 = ca.Buffer(n * m * 2)
    c32 = ca.Buffer(n * m * 4)
    ca.gemm_bf16(a, b, c16, n, m, k)
    first = c16.read(np.uint16, (n, m))
    say("bf16 gemm 4096^3 run-to-run x5")
    for _ in range(5):
        ca.gemm_bf16(a, b, c16, n, m, k)
        assert hash_bits(c16.read(np.uint16)) == hash_bits(first)
    ca.gemm_bf16(a, b, c32, n, m, k, out_f32=True)
    g32 = c32.read(np.float32, (n, m))
    assert np.array_equal(first, oracle.f32_to_bf16_bits_np(g32))
    say("bf16 gemm 4096^3: sequential oracle over all rows")
    seq32, seq16 = oracle.matmul_bf16(a16, b16)
    af = as_f32(a16).astype(np.float64)
    bf = as_f32(b16).astype(np.float64)
    exact = af @ bf
    absprod = np.abs(af) @ np.abs(bf)
    del af, bf
    # f32 output: the MFMA-order bound against the exact product
    mfma_bound = 8 * (k / 32 + 1) * U * absprod
    assert np.all(np.abs(g32.astype(np.float64) - exact) <= mfma_bound)
    # bf16 output against the sequential oracle's bf16
    delta = mfma_bound + k * U * absprod
    g = as_f32(first).astype(np.float64)
    sq = as_f32(seq16).astype(np.float64)
    spacing = bf16_ulp_of(np.minimum(np.abs(g), np.abs(sq)))
    ulps = bf16_ulp_diff(first, seq16)
    ulp_bound = 1 + np.ceil(delta / spacing)
    assert np.all(ulps <= ulp_bound), int((ulps - ulp_bound).max())
    kappa = absprod / np.maximum(np.abs(exact), 1e-300)
    well = kappa <= 64
    c = (8 * (k / 32 + 1) + k) * U * 64
    assert 1 + math.ceil(256 * c / (1 - c)) == 7
    assert ulps[well].max() <= 7
    stats = {
        "cells": int(ulps.size),
        "bf16_max_ulp": int(ulps.max()),
        "bf16_max_ulp_kappa_le_64": int(ulps[well].max()),
        "kappa_le_64_frac": float(well.mean()),
        "bf16_max_ulp_kappa_le_1024": int(ulps[kappa <= 1024].max()),
        "kappa_le_1024_frac": float((kappa <= 1024).mean()),
        "bf16_identical_frac": float(np.mean(ulps == 0)),
        "bf16_le1ulp_frac": float(np.mean(ulps <= 1)),
        "f32_identical_to_sequential_frac": float(np.mean(g32 == seq32)),
        "f32_max_err_over_bound": float((np.abs(g32.astype(np.float64) - exact) / mfma_bound).max()),
    }
    print("[bf16-gemm-4096-stats]", stats, flush=True)


@pytest.mark.parametrize("mrows,n,k", [(16, 11008, 4096), (16, 4096, 11008), (1, 4096, 4096),
                                       (7, 1024, 960), (16, 128, 32), (5, 136, 8),
                                       (16, 256, 16384), (3, 136, 20000)])
def test_decode_kernel_full_compare(mrows, n, k):
    """Whole-output comparison with the oracle under the stated bound, f32
    and bf16 outputs consistent, bits run to run.  The last two shapes split
    K into 64 and 79 k groups, so the reduction launch adds its partials in
    several batches of loads (and the second one over a ragged column
    block)."""
    say(f"bf16 decode gemm M={mrows} N={n} K={k}")
    a, b, a16, b16 = _inputs(mrows, n, k, seed=300 + mrows + n + k, wscale=0.02)
    c16 = ca.Buffer(mrows * n * 2)
    c32 = ca.Buffer(mrows * n * 4)
    ca.gemm_bf16(a, b, c16, mrows, n, k)
    ca.gemm_bf16(a, b, c32, mrows, n, k, out_f32=True)
    g16 = c16.read(np.uint16, (mrows, n))
    g32 = c32.read(np.float32, (mrows, n))
    assert np.array_equal(g16, oracle.f32_to_bf16_bits_np(g32))
    _check(a16, b16, g32, g16)
    h = hash_bits(g16)
    for _ in range(3):
        ca.gemm_bf16(a, b, c16, mrows, n, k)
        assert hash_bits(c16.read(np.uint16)) == h


def test_decode_and_tile_kernels_random_shapes():
    """Seeded random shapes through gemm_bf16: 16 decode shapes (M <= 16; N
    and K multiples of 8, so both the streamed path (K % 32 == 0) and the
    register path, ragged column blocks and one to many k groups) and 12
    wider ones (M > 16: general kernels), each against the oracle under the stated bound, f32 and bf16
    outputs consistent and bitwise run to run."""
    rng = np.random.default_rng(777)
    shapes = []
    for _ in range(16):
        m_rows = int(rng.integers(1, 17))
        n = 8 * int(rng.integers(1, 400))
        k = 8 * int(rng.integers(1, 800))
        if rng.random() < 0.5:
            k = 32 * max(1, k // 32)
        shapes.append((m_rows, n, k))
    for _ in range(12):
        m_rows = int(rng.integers(17, 600))
        n = int(rng.integers(1, 600))
        k = int(rng.integers(1, 600))
        if rng.random() < 0.5:
            m_rows, n, k = 256 * int(rng.integers(1, 3)), 128 * int(rng.integers(1, 5)), 128 * int(rng.integers(1, 5))
        shapes.append((m_rows, n, k))
    for i, (m_rows, n, k) in enumerate(shapes):
        say(f"bf16 gemm random shape M={m_rows} N={n} K={k}")
        a, b, a16, b16 = _inputs(m_rows, n, k, seed=1000 + i, wscale=0.02 if m_rows <= 16 else 1.0)
        c16, c32 = ca.Buffer(m_rows * n * 2), ca.Buffer(m_rows * n * 4)
        ca.gemm_bf16(a, b, c16, m_rows, n, k)
        ca.gemm_bf16(a, b, c32, m_rows, n, k, out_f32=True)
        g16, g32 = c16.read(np.uint16, (m_rows, n)), c32.read(np.float32, (m_rows, n))
        assert np.array_equal(g16, oracle.f32_to_bf16_bits_np(g32)), (m_rows, n, k)
        _check(a16, b16, g32, g16)
        ca.gemm_bf16(a, b, c16, m_rows, n, k)
        assert np.array_equal(c16.read(np.uint16, (m_rows, n)), g16), (m_rows, n, k)


def test_program_bf16_matmul():
    rt = ca.Runtime([])
    n, m, k = 32, 40, 24
    rng = np.random.default_rng(4)
    a16 = oracle.f32_to_bf16_bits_np(rng.integers(-4, 5, (n, k)).astype(np.float32))
    b16 = oracle.f32_to_bf16_bits_np(rng.integers(-4, 5, (k, m)).astype(np.float32))
    abuf, bbuf = ca.Buffer.from_array(a16), ca.Buffer.from_array(b16)
    say("runtime exec bf16.matmul.row-major.via-mem")
    [res] = rt.exec("bf16.matmul.row-major.via-mem",
                    [ca.Value.mem(abuf.mem), ca.Value.mem(bbuf.mem)] +
                    [ca.Value.u64(x) for x in (n, m, k, n * k, k * m, n * m)], 1)
    got = ca.mem_to_array(res.get(), np.uint16).reshape(n, m)
    # small integers: every partial sum is exact, so any order gives the oracle's bits
    assert np.array_equal(got, oracle.matmul_bf16(a16, b16)[1])
    ca.mem_free(res.get())


def test_decode_register_path():
    """The register-transpose decode path, taken when K % 32 != 0: same
    contract (bound, f32/bf16 consistency, run to run)."""
    mrows, n, k = 16, 4096, 2056
    say(f"bf16 decode gemm register path M={mrows} N={n} K={k}")
    a, b, a16, b16 = _inputs(mrows, n, k, seed=91, wscale=0.02)
    c16, c32 = ca.Buffer(mrows * n * 2), ca.Buffer(mrows * n * 4)
    ca.gemm_bf16(a, b, c16, mrows, n, k)
    ca.gemm_bf16(a, b, c32, mrows, n, k, out_f32=True)
    g16, g32 = c16.read(np.uint16, (mrows, n)), c32.read(np.float32, (mrows, n))
    assert np.array_equal(g16, oracle.f32_to_bf16_bits_np(g32))
    _check(a16, b16, g32, g16)
    ca.gemm_bf16(a, b, c16, mrows, n, k)
    assert np.array_equal(c16.read(np.uint16, (mrows, n)), g16)


@pytest.mark.parametrize("n,m,k", [(256, 1024, 2048), (2048, 8192, 256), (512, 384, 128)])
def test_gemm_swiglu_epilogue_equals_gemm_then_silu(n, m, k):
    """The SwiGLU-fused tile GEMM (256 x 128 tiles for the first and third
    shape, 256 x 256 for the second, as the plain GEMM would choose) gives
    the bits of the f32 GEMM followed by catena_mi355x_silu_mul_bf16 with
    group 64."""
    a = dev_normal_bf16(n * k, 31 + n + k, 0, 1.0)
    b = dev_normal_bf16(k * m, 31 + n + k, 1, 1.0)
    say(f"bf16 GEMM + SwiGLU n={n} m={m} k={k}")
    act = ca.Buffer(n * (m // 2) * 2)
    ca.gemm_bf16_silu(a, b, act, n, m, k)
    gu = ca.Buffer(n * m * 4)
    ca.gemm_bf16(a, b, gu, n, m, k, out_f32=True)
    want = ca.Buffer(n * (m // 2) * 2)
    ca.silu_mul_bf16(gu, want, n, m // 2, 64)
    assert np.array_equal(act.read(np.uint16), want.read(np.uint16))


def test_gemm_swiglu_rejects_untiled_shapes():
    a = dev_normal_bf16(256 * 256, 5, 0, 1.0)
    b = dev_normal_bf16(256 * 256, 5, 1, 1.0)
    act = ca.Buffer(256 * 128 * 2)
    with pytest.raises(ca.CatenaError):
        ca.gemm_bf16_silu(a, b, act, 100, 256, 256)
    with pytest.raises(ca.CatenaError):
        ca.gemm_bf16_silu(a, b, act, 256, 256, 96)


def test_gemm_swiglu_special_values():
    """NaN, +-inf and overflowing products in the gate and up columns: the
    fused epilogue gives the bits of the f32 GEMM followed by silu_mul."""
    n, m, k = 256, 512, 128
    rng = np.random.default_rng(41)
    a32 = rng.normal(0, 1, (n, k)).astype(np.float32)
    a32[3, 7] = np.nan                  # row 3: NaN everywhere
    a32[5, :] = 3e38                    # row 5: products overflow to +-inf
    a32[9, 0] = np.inf                  # row 9: +-inf or NaN (inf * 0)
    a32[11, :] = 0.0                    # row 11: exact zeros (silu(+0) * up)
    b32 = rng.normal(0, 1, (k, m)).astype(np.float32)
    b32[0, 64:128] = 0.0                # up columns of group 0 see inf * 0 = NaN on row 9
    a = ca.Buffer.from_array(oracle.f32_to_bf16_bits_np(a32))
    b = ca.Buffer.from_array(oracle.f32_to_bf16_bits_np(b32))
    say("bf16 GEMM + SwiGLU special values")
    act = ca.Buffer(n * (m // 2) * 2)
    ca.gemm_bf16_silu(a, b, act, n, m, k)
    gu = ca.Buffer(n * m * 4)
    ca.gemm_bf16(a, b, gu, n, m, k, out_f32=True)
    want = ca.Buffer(n * (m // 2) * 2)
    ca.silu_mul_bf16(gu, want, n, m // 2, 64)
    g16, w16 = act.read(np.uint16), want.read(np.uint16)
    assert np.array_equal(g16, w16), int(np.sum(g16 != w16))
    g = gu.read(np.float32, (n, m))
    assert np.isnan(g[3]).all() and not np.isfinite(g[5]).all() and np.isnan(g[9, 64:128]).all()


@pytest.mark.parametrize("B,Tq,H,L,k,lens", [
    (2, 128, 2, 300, 256, [128, 300]),        # empty cache; a cached prefix of 172
    (1, 256, 3, 200, 128, [256]),             # rows 200..255 past the cache end: q only
    (4, 64, 1, 128, 384, [64, 10, 128, 100]),  # lens < Tq: no cache row for batch 1
    (256, 1, 2, 64, 128, "random"),           # decode-shaped rows, lens 0 .. 80
])
def test_gemm_rope_qkv_fused_equals_gemm_then_rope(B, Tq, H, L, k, lens):
    """The RoPE-fused q / k / v projection (the decoder's prefill W_qkv) gives
    the bits of the f32 GEMM followed by catena_mi355x_rope_qkv_bf16: q for
    every row, cache rows only at positions in [0, L), every other cache
    element untouched -- with cached prefixes, rows past the cache end and
    sequences shorter than Tq."""
    D, R = 128, B * Tq
    m = 3 * H * D
    if lens == "random":
        lens = np.random.default_rng(B + L).integers(0, 81, B).tolist()
    a = dev_normal_bf16(R * k, 17 + k, 0, 1.0)
    w = dev_normal_bf16(k * m, 17 + k, 1, 0.2)
    inv = ca.Buffer.from_array(ca.rope_inv_freq(D, 10000.0))
    tab = ca.Buffer(L * D * 4)
    ca.rope_table_f32(inv, tab, L, D)
    lb = ca.Buffer.from_array(np.array(lens, np.uint32))
    sentinel = np.full(B * H * L * D, 0xABCD, np.uint16)
    caches = [ca.Buffer.from_array(sentinel) for _ in range(4)]
    q_f, q_u = ca.Buffer(R * H * D * 2), ca.Buffer(R * H * D * 2)
    say(f"fused q/k/v + RoPE B={B} Tq={Tq} H={H} L={L} k={k} lens={lens[:6]}")
    ca.gemm_bf16_rope_qkv(a, w, tab, lb, q_f, caches[0], caches[1], B, Tq, H, L, k)
    qkv = ca.Buffer(R * m * 4)
    ca.gemm_bf16(a, w, qkv, R, m, k, out_f32=True)
    ca.rope_qkv_bf16(qkv, inv, lb, q_u, caches[2], caches[3], B, Tq, H, D, L)
    assert np.array_equal(q_f.read(np.uint16), q_u.read(np.uint16))
    for got, want in ((caches[0], caches[2]), (caches[1], caches[3])):
        g, w_ = got.read(np.uint16, (B, H, L, D)), want.read(np.uint16, (B, H, L, D))
        assert np.array_equal(g, w_), int(np.sum(g != w_))
    written = (caches[2].read(np.uint16, (B, H, L, D)) != 0xABCD).any(axis=(1, 3))
    for b, n_ in enumerate(lens):  # the positions a row of batch b lands on
        want = np.zeros(L, bool)
        if n_ >= Tq:
            want[n_ - Tq:min(n_, L)] = True
        assert np.array_equal(written[b], want), b


def test_gemm_rope_qkv_rejects_untiled_shapes():
    a, w = ca.Buffer(256 * 256 * 2), ca.Buffer(256 * 384 * 2)
    tab, lb = ca.Buffer(64 * 128 * 4), ca.Buffer(4 * 4)
    q, kc, vc = ca.Buffer(256 * 128 * 2), ca.Buffer(4 * 64 * 128 * 2), ca.Buffer(4 * 64 * 128 * 2)
    with pytest.raises(ca.CatenaError):
        ca.gemm_bf16_rope_qkv(a, w, tab, lb, q, kc, vc, 2, 100, 1, 64, 256)  # rows % 256
    with pytest.raises(ca.CatenaError):
        ca.gemm_bf16_rope_qkv(a, w, tab, lb, q, kc, vc, 1, 256, 1, 64, 96)   # k % 128


@pytest.mark.parametrize("n,m,k,splits", [(256, 256, 256, 2), (256, 4096, 11008, 2),
                                          (512, 512, 1536, 3), (256, 256, 128, 1)])
def test_gemm_ksplit_parts_equal_gemm_of_each_k_range(n, m, k, splits):
    """parts[z] of the k-split GEMM (the decoder's prefill W_down) is bitwise
    the f32 GEMM of the z-th k range, and their ascending sum is within the
    bf16 GEMM bound of the whole product."""
    rng = np.random.default_rng(n + k + splits)
    a16 = oracle.f32_to_bf16_bits_np(rng.standard_normal((n, k)).astype(np.float32))
    b16 = oracle.f32_to_bf16_bits_np((rng.standard_normal((k, m)) * 0.1).astype(np.float32))
    parts = ca.Buffer(splits * n * m * 4)
    say(f"k-split GEMM n={n} m={m} k={k} splits={splits}")
    ca.gemm_bf16_ksplit_f32(ca.Buffer.from_array(a16), ca.Buffer.from_array(b16), parts, n, m, k,
                            splits)
    got = parts.read(np.float32, (splits, n, m))
    kl = k // splits
    for z in range(splits):
        az = ca.Buffer.from_array(np.ascontiguousarray(a16[:, z * kl:(z + 1) * kl]))
        bz = ca.Buffer.from_array(np.ascontiguousarray(b16[z * kl:(z + 1) * kl]))
        cz = ca.Buffer(n * m * 4)
        ca.gemm_bf16(az, bz, cz, n, m, kl, out_f32=True)
        assert np.array_equal(got[z].view(np.uint32), cz.read(np.uint32, (n, m))), z
    total = got[0].copy()
    for z in range(1, splits):
        total = total + got[z]
    rows = np.arange(0, n, max(1, n // 16))
    gemm_within_bound(a16[rows], b16, total[rows])


def test_gemm_ksplit_rejects_untiled_shapes():
    a, b, p = ca.Buffer(256 * 384 * 2), ca.Buffer(384 * 256 * 2), ca.Buffer(2 * 256 * 256 * 4)
    with pytest.raises(ca.CatenaError):
        ca.gemm_bf16_ksplit_f32(a, b, p, 256, 256, 384, 2)   # k % 256
    with pytest.raises(ca.CatenaError):
        ca.gemm_bf16_ksplit_f32(a, b, p, 256, 256, 384, 0)   # splits == 0


def _lm_head_case(x16, w16, n, m, k):
    """The fused LM head (catena_mi355x_gemm_bf16_argmax): its logits within
    the GEMM bound where finite, and every index equal to the oracle's
    tensor.argmax-f32 of the GPU's own logits row."""
    xb, wb = ca.Buffer.from_array(x16), ca.Buffer.from_array(w16)
    c = ca.Buffer(n * m * 4)
    idx = ca.Buffer(n * 4)
    ca.gemm_bf16_argmax(xb, wb, c, idx, n, m, k)
    logits = c.read(np.float32, (n, m))
    got = idx.read(np.uint32)
    want = [oracle.argmax_f32(logits[r]) for r in range(n)]
    assert list(got) == want, (list(got), want)
    return logits, got


def test_lm_head_argmax_nan_tie_and_zero_patterns():
    """Logit patterns for the per-block summaries and their composition
    across 128-column blocks (ragged last block): an exact tie between two
    blocks (duplicated weight columns: the earlier wins), NaN columns at a
    block boundary with the maximum after them, NaN in the last column (the
    answer), every logit +0 or -0, and rows with different maxima."""
    n, k = 8, 256
    m = 128 * 20 + 64
    rng = np.random.default_rng(23)
    x = rng.normal(0, 1, (n, k)).astype(np.float32)
    w = rng.normal(0, 0.05, (k, m)).astype(np.float32)
    w[:, 1000] = w[:, 400] = rng.normal(0, 1, k).astype(np.float32)  # the same dominant column twice
    x16 = oracle.f32_to_bf16_bits_np(x)

    say("LM head argmax: tie across blocks")
    w16 = oracle.f32_to_bf16_bits_np(w)
    logits, got = _lm_head_case(x16, w16, n, m, k)
    gemm_within_bound(x16, w16, logits)
    assert 1000 not in got  # its twin, column 400, comes first

    say("LM head argmax: NaN at a block boundary, the maximum after it")
    wn = w.copy()
    wn[3, 127] = wn[5, 128] = np.nan
    wn[:, 2000] = 4 * w[:, 1000]
    _lm_head_case(x16, oracle.f32_to_bf16_bits_np(wn), n, m, k)

    say("LM head argmax: NaN in the last column")
    wl = w.copy()
    wl[7, m - 1] = np.nan
    wl[7, 130] = np.nan
    _, got = _lm_head_case(x16, oracle.f32_to_bf16_bits_np(wl), n, m, k)
    assert list(got) == [m - 1] * n

    say("LM head argmax: all logits zero")
    wz = np.zeros((k, m), np.float32)
    _, got = _lm_head_case(x16, oracle.f32_to_bf16_bits_np(wz), n, m, k)

    say("LM head argmax: 8 x 32000 x 2048 against the plain GEMM")
    a, b, a16, b16 = _inputs(8, 32000, 2048, 29)
    c = ca.Buffer(8 * 32000 * 4)
    idx = ca.Buffer(8 * 4)
    ca.gemm_bf16_argmax(a, b, c, idx, 8, 32000, 2048)
    plain = ca.Buffer(8 * 32000 * 4)
    ca.gemm_bf16(a, b, plain, 8, 32000, 2048, out_f32=True)
    lg = c.read(np.float32, (8, 32000))
    assert np.array_equal(lg.view(np.uint32), plain.read(np.float32, (8, 32000)).view(np.uint32))
    assert list(idx.read(np.uint32)) == [oracle.argmax_f32(lg[r]) for r in range(8)]
