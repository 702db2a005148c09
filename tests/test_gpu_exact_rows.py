"""The exact-order f32 GEMM's row forms (A by scalar loads) at the sizes where
they and the 16 x 16 tiles change over, bitwise against the oracle's ascending
chain, with operands at any 4-byte address between NaNs."""
import numpy as np
import pytest

import catena_amd as ca
import oracle
from gpu_util import say

pytestmark = pytest.mark.gpu

SPECIALS = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-20, -1e-20, 3e-39, 1.0, -2.5], np.float32)


def _placed(a, shift_bytes):
    raw = np.full(a.nbytes + 1024, 0xFF, np.uint8)  # all-ones words are NaNs
    raw[256 + shift_bytes:256 + shift_bytes + a.nbytes] = np.ascontiguousarray(a).view(np.uint8).reshape(-1)
    buf = ca.Buffer.from_array(raw)
    return buf, buf.ptr + 256 + shift_bytes


def _check(n, m, k, shift=0, special=False):
    rng = np.random.default_rng(n + 3 * m + 7 * k + shift)
    a = rng.uniform(-1, 1, (n, k)).astype(np.float32)
    b = rng.uniform(-1, 1, (k, m)).astype(np.float32)
    if special:
        for x in (a, b):
            hit = rng.random(x.shape) < 0.01
            x[hit] = rng.choice(SPECIALS, int(hit.sum()))
        b[:, :3] *= np.float32(1e-19)
    say(f"gemm f32 exact rows {n}x{m}x{k} shift {shift} special {special}")
    (ab, ap), (bb, bp) = _placed(a, shift), _placed(b, shift)
    fill = 0xA5
    cb = ca.Buffer.from_array(np.full(n * m * 4 + 512, fill, np.uint8))
    ca.gemm_f32_exact(ap, bp, cb.ptr + 256, n, m, k)
    raw = cb.read(np.uint8)
    assert np.all(raw[:256] == fill) and np.all(raw[-256:] == fill)
    got, want = raw[256:-256].copy().view(np.float32).reshape(n, m), oracle.matmul_f32(a, b)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


# 2 x 1: more than 256 tiles of 16 x 16 and fewer than 600 workgroups of 4 x 1;
# 4 x 1; 8 x 2 from 700 workgroups on; one row or column past a wave's
@pytest.mark.parametrize("n,m,k", [
    (257, 257, 1), (272, 257, 7), (273, 259, 16), (300, 301, 17), (1000, 70, 33), (70, 1000, 47), (5, 20000, 31),
    (385, 1537, 15), (400, 1600, 16), (401, 1601, 48), (9600, 63, 19), (9601, 65, 16),
    (1089, 2561, 8), (1120, 2560, 9), (33, 90000, 7), (1121, 2562, 24),
    (512, 512, 16), (512, 516, 16), (516, 512, 32),
    # 8 x 2 with few k (below half a tile of rows) and with remainders of 0, 1, 7 k
    (32, 90000, 7), (17, 90001, 8), (31, 90001, 9), (1089, 2561, 40), (1120, 2560, 41), (1121, 2562, 55),
    # 64 x 64 tiles: few k, at and past a slab of 16; 4 x 1 at 64 columns and 16 x 16 at 16, next to them
    (1280, 1025, 15), (1281, 1088, 1), (1536, 2047, 23), (2049, 1537, 31), (1537, 2048, 24), (20000, 64, 33), (20000, 65, 33),
    (30001, 16, 48), (30001, 16, 33), (30001, 17, 48), (70000, 1, 65), ((1 << 20) - 15, 3, 32), ((1 << 20) + 21, 1, 33),
    # two tiles for each of 256 CUs (three past 3 MiB of operands), 6.5 of the DPP form
    (512, 256, 17), (513, 255, 17), (522, 256, 1011), (522, 256, 1010), (769, 250, 801), (1664, 256, 16), (1665, 256, 16)])
def test_row_forms(n, m, k):
    _check(n, m, k)


@pytest.mark.parametrize("n,m,k", [(300, 301, 50), (401, 1601, 37), (1089, 2561, 21), (1089, 2561, 45), (1025, 1345, 33)])
@pytest.mark.parametrize("shift,special", [(4, False), (12, True), (0, True), (2, False)])
def test_addresses_and_special_values(n, m, k, shift, special):
    _check(n, m, k, shift, special)


# the forms' ranges: 16 x 16 tiles, 2 x 1, 4 x 1, 8 x 2
@pytest.mark.parametrize("n,m", [(1, 1), (33, 31), (300, 301), (401, 1601), (1121, 2562)])
def test_empty_fold(n, m):
    """k == 0: every cell is the fold's start, +0; the operands may be null."""
    say(f"gemm f32 exact empty fold {n}x{m}")
    cb = ca.Buffer.from_array(np.full(n * m * 4 + 512, 0xA5, np.uint8))
    ca.gemm_f32_exact(0, 0, cb.ptr + 256, n, m, 0)
    raw = cb.read(np.uint8)
    assert not raw[256:-256].any()
    assert np.all(raw[:256] == 0xA5) and np.all(raw[-256:] == 0xA5)


@pytest.mark.parametrize("n,m,k", [(2, (1 << 25) + 3, 3), (65, (1 << 25) + 64, 1)])
def test_past_32_bit_offsets(n, m, k):
    """Rows wider than the row forms' offsets: 64 x 64 tiles."""
    say(f"gemm f32 exact {n}x{m}x{k}")
    rng = np.random.default_rng(k)
    one = rng.uniform(-1, 1, 999983).astype(np.float32)
    a, b = rng.uniform(-1, 1, (n, k)).astype(np.float32), np.resize(one, (k, m))
    ab, bb, cb = ca.Buffer.from_array(a), ca.Buffer.from_array(b), ca.Buffer(n * m * 4)
    ca.gemm_f32_exact(ab, bb, cb, n, m, k)
    for i in sorted({0, 1, n - 1}):
        want = np.zeros(m, np.float32)
        for kk in range(k):
            want = want + a[i, kk] * b[kk]
        assert np.array_equal(cb.read(np.uint32, (m,), offset=i * m * 4), want.view(np.uint32)), i
