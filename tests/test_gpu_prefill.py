"""The block-of-16-queries attention at the sizes where its form changes (four
or eight waves, one or two launches, one query per workgroup): every form gives
the bits of the one-query kernels on each query's prefix."""
import math

import numpy as np
import pytest

import catena_amd as ca
import oracle
from gpu_util import say

pytestmark = pytest.mark.gpu

D = 128
SCALE = 1.0 / math.sqrt(D)


def _causal(q16, kb, vb, lens, L, out_f32):
    B, Tq, H, _ = q16.shape
    qb, lb = ca.Buffer.from_array(q16), ca.Buffer.from_array(np.asarray(lens, np.uint32))
    fill = 0xA5
    ob = ca.Buffer.from_array(np.full(q16.size * (4 if out_f32 else 2) + 512, fill, np.uint8))
    ca.attn_causal_bf16(qb, kb, vb, lb, ob.ptr + 256, B, Tq, H, L, D, SCALE, out_f32=out_f32)
    raw = ob.read(np.uint8)
    assert np.all(raw[:256] == fill) and np.all(raw[-256:] == fill)
    return raw[256:-256].copy().view(np.uint32 if out_f32 else np.uint16).reshape(q16.shape)


def _inputs(B, Tq, H, L, seed, special):
    rng = np.random.default_rng(seed)
    mk = lambda *s: rng.normal(0, 1, s).astype(np.float32)  # noqa: E731
    q, k, v = mk(B, Tq, H, D), mk(B, H, L, D), mk(B, H, L, D)
    if special:
        # head 0: a NaN key; head 1: NaN, infinite and denormal values; head 2:
        # all scores equal; head 3: a query and keys outside the exact range of
        # the matrix-core fold
        k[:, 0, L // 3, 5] = np.nan
        v[:, 1, L // 2, 7], v[:, 1, L // 4, 9], v[:, 1, 3, :] = np.nan, -np.inf, 1e-39
        k[:, 2] = 0.0
        q[:, Tq // 2, 3, 11], k[:, 3, L // 5, :] = 1e-30, 1e25
    return (oracle.f32_to_bf16_bits_np(x) for x in (q, k, v))


# (B, Tq, H, max_len, cached before): grids of 65 .. 512 blocks and more, rows
# at 704 / 705, 1088 / 1089 and 2304 / 2305, partial last blocks, two launches
@pytest.mark.parametrize("B,Tq,H,L,pfx", [
    (1, 257, 4, 300, 0), (2, 129, 4, 640, 400), (1, 520, 16, 704, 100), (1, 520, 16, 705, 100),
    (2, 270, 16, 704, 434), (1, 100, 10, 1088, 900), (1, 100, 10, 1089, 900), (1, 600, 16, 1100, 500),
    (1, 300, 4, 2304, 2000), (1, 300, 4, 2305, 2000), (1, 64, 16, 90, 0), (1, 65, 16, 90, 0), (1, 1100, 8, 1150, 40),
    # past 1088 rows: at and past the fewest queries that take blocks
    (1, 300, 10, 1089, 700), (1, 300, 10, 2304, 2000), (1, 64, 40, 1100, 1000), (1, 64, 41, 1100, 1000),
    (8, 8, 31, 1200, 1100), (8, 8, 32, 1200, 1100), (4, 9, 60, 1190, 1100), (3, 33, 25, 1300, 1200), (3, 33, 26, 1300, 1200)])
@pytest.mark.parametrize("special", [False, True])
def test_every_form_equals_the_one_query_kernel(B, Tq, H, L, pfx, special):
    q16, k16, v16 = _inputs(B, Tq, H, L, B + Tq + H + L + pfx, special)
    kb, vb = ca.Buffer.from_array(k16), ca.Buffer.from_array(v16)
    lens = [min(L, pfx + Tq) - 3 * b for b in range(B)]
    say(f"causal attention B={B} Tq={Tq} H={H} L={L} lens={lens} special={special}")
    got = _causal(q16, kb, vb, lens, L, True)
    got16 = _causal(q16, kb, vb, lens, L, False)
    nan = np.isnan(got.view(np.float32))
    assert np.array_equal(got16[~nan], oracle.f32_to_bf16_bits_np(got.view(np.float32))[~nan])
    # seven queries at a time take the one-query kernels
    starts = sorted({0, 7, Tq // 3, Tq // 2, max(0, Tq - 23), Tq - 7})
    for t0 in starts:
        sub = np.ascontiguousarray(q16[:, t0:t0 + 7])
        after = Tq - t0 - sub.shape[1]
        want = _causal(sub, kb, vb, [max(0, n - after) for n in lens], L, True)
        a, b = got[:, t0:t0 + 7], want
        an, bn = np.isnan(a.view(np.float32)), np.isnan(b.view(np.float32))
        assert np.array_equal(an, bn), t0
        assert np.array_equal(a[~an], b[~bn]), t0
