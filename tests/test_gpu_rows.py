"""Row folds that keep rows in LDS (softmax one and four rows to a workgroup,
RMSNorm and f32 sums four): the sizes where the forms change over and their
edges, bitwise against the oracle, rows at any 4-byte address, in place, with
the values that steer the fold."""
import numpy as np
import pytest

import catena_amd as ca
import oracle
from oracle import decoder as od
from gpu_util import say

pytestmark = pytest.mark.gpu

INF, NAN = np.float32(np.inf), np.float32(np.nan)


def _same(got, want):
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


def _rows(rows, n, seed):
    """Normal values; a few rows hold what the maximum treats specially."""
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((rows, n)) * 3).astype(np.float32)
    special = [
        lambda r: np.full_like(r, -INF),
        lambda r: np.where(np.arange(n) % 3 == 0, np.float32(-0.0), np.float32(0.0)).astype(np.float32),
        lambda r: np.where(np.arange(n) == n - 1, NAN, r),
        lambda r: np.where(np.arange(n) == n // 2, NAN, r),
        lambda r: np.full_like(r, NAN),
        lambda r: np.where(np.arange(n) == n // 3, INF, r),
        lambda r: np.full_like(r, 1e-42),
        lambda r: np.minimum(r, np.float32(0.0)),
        # quotients outside the bounds of the shared-divisor division
        lambda r: r * np.float32(1e-33),
        lambda r: r * np.float32(10.0) ** (-(np.arange(n) % 44)).astype(np.float32),
        lambda r: r * np.float32(1e12),
        lambda r: np.where(np.arange(n) % 5 == 0, np.float32(-0.0), r),
    ]
    at = rng.permutation(rows)[:len(special)]
    for i, f in zip(at, special):
        x[i] = f(x[i]).astype(np.float32)
    return x, sorted(set(at.tolist()) | {0, rows - 1} | set(rng.integers(0, rows, 6).tolist()))


def _placed(x, shift):
    raw = np.full(x.nbytes + 512, 0xFF, np.uint8)  # all-ones words are NaNs
    raw[256 + shift:256 + shift + x.nbytes] = x.view(np.uint8).reshape(-1)
    buf = ca.Buffer.from_array(raw)
    return buf, buf.ptr + 256 + shift


# rows: one short of, at, and past six to a CU (1536 on 256 CUs); n: chunk edges
# of the folds, ragged, the longest rows of the four-row (9088) and one-row LDS
# forms (40944) and the next ones
@pytest.mark.parametrize("rows,n", [(1, 1), (3, 2), (5, 33), (9, 511), (1535, 64), (1536, 64), (1537, 65), (1541, 512),
                                    (1539, 516), (1537, 1028), (1537, 2047), (2, 9088), (3, 9089), (2, 40944),
                                    (2, 40945),
                                    # one row a CU: LDS up to three rounds; two: up to three and past eight rows a CU
                                    (768, 20448), (769, 20449), (1536, 13652), (1537, 13653), (2049, 13652)])
@pytest.mark.parametrize("shift", [0, 4])
def test_softmax(rows, n, shift):
    say(f"softmax rows {rows} n {n} shift {shift}")
    x, look = _rows(rows, n, rows * 7 + n)
    buf, p = _placed(x, shift)
    y = ca.Buffer.from_array(np.full(x.nbytes + 512, 0xA5, np.uint8))
    ca.softmax_f32(p, y.ptr + 256 + shift, rows, n)
    raw = y.read(np.uint8)
    assert (raw[:256 + shift] == 0xA5).all() and (raw[256 + shift + x.nbytes:] == 0xA5).all()
    got = raw[256 + shift:256 + shift + x.nbytes].view(np.float32).reshape(rows, n)
    for i in look:
        _same(got[i], oracle.softmax_f32(x[i]))
    ca.softmax_f32(p, p, rows, n)  # in place
    again = buf.read(np.uint8)[256 + shift:256 + shift + x.nbytes].view(np.float32).reshape(rows, n)
    _same(again, got)


@pytest.mark.parametrize("rows,n", [(1, 0), (1, 1), (7, 3), (6, 2048), (5, 513), (1025, 8192), (4099, 36), (9, 9088),
                                    (9, 9089), (1025, 6001), (3072, 2816), (3073, 2816), (3073, 2818), (4097, 2224), (4097, 2272)])
@pytest.mark.parametrize("shift", [0, 4])
def test_sum(rows, n, shift):
    say(f"sum rows {rows} n {n} shift {shift}")
    x, look = _rows(rows, n, rows * 5 + n) if n else (np.zeros((rows, 0), np.float32), [0])
    _, p = _placed(x, shift)
    for fn, ref in ((ca.sum_f32, lambda r: np.float32(oracle.fold_sum_f32(r))),
                    (ca.mean_f32, lambda r: np.float32(oracle.fold_sum_f32(r)) / np.float32(n))):
        out = ca.Buffer.from_array(np.full(rows + 2, 7.0, np.float32))
        fn(p, out.ptr + 4, rows, n)
        got = out.read(np.float32)
        assert got[0] == 7.0 and got[-1] == 7.0
        with np.errstate(invalid="ignore"):
            for i in look:
                _same(got[1 + i:2 + i], np.array([ref(x[i])], np.float32))


@pytest.mark.parametrize("rows,n", [(2048, 64), (2049, 64), (2051, 65), (2050, 2044), (2049, 514), (1281, 4096),
                                    (1282, 4093)])
def test_rmsnorm(rows, n):
    say(f"rmsnorm rows {rows} n {n}")
    x, look = _rows(rows, n, rows * 3 + n)
    xb, y = ca.Buffer.from_array(x), ca.Buffer.from_array(np.full(rows * n + 64, 7.0, np.float32))
    ca.rmsnorm_f32(xb, y, rows, n)
    got = y.read(np.float32)
    assert (got[rows * n:] == 7.0).all()
    got = got[:rows * n].reshape(rows, n)
    for i in look:
        _same(got[i], oracle.rmsnorm_f32(x[i]))


@pytest.mark.parametrize("rows,n", [(2305, 256), (2305, 260), (2305, 1024), (2305, 1030), (2305, 514), (2305, 1023), (3200, 1030),
                                    (2305, 1596), (2305, 2044), (2500, 2048), (1300, 4096), (2049, 4096)])
@pytest.mark.parametrize("parts", ["resid", "index", "both"])
def test_residual_rmsnorm_bf16(rows, n, parts):
    """The same norm with the residual add, the gather of rows, and both
    outputs, against the one-row form (fewer rows at a time)."""
    say(f"residual rmsnorm {rows} x {n} {parts}")
    x, _ = _rows(rows, n, n)
    rng = np.random.default_rng(n + 1)
    r = rng.standard_normal((rows, n)).astype(np.float32)
    idx = rng.permutation(rows).astype(np.uint32)
    xb, rb = ca.Buffer.from_array(x), None if parts == "index" else ca.Buffer.from_array(r)

    def run(index):
        m = len(index)
        h = ca.Buffer.from_array(np.zeros(m * n, np.float32))
        y = ca.Buffer.from_array(np.zeros(m * n, np.uint16))
        ca.residual_rmsnorm_bf16(xb, rb, ca.Buffer.from_array(index), h, y, m, n)
        return h.read(np.uint32).reshape(m, n), y.read(np.uint16).reshape(m, n)

    index = np.arange(rows, dtype=np.uint32) if parts == "resid" else idx
    h, y = run(index)
    if parts == "resid":  # and without the index
        h2, y2 = ca.Buffer.from_array(np.zeros(rows * n, np.float32)), ca.Buffer.from_array(np.zeros(rows * n, np.uint16))
        ca.residual_rmsnorm_bf16(xb, rb, None, h2, y2, rows, n)
        assert np.array_equal(h2.read(np.uint32).reshape(rows, n), h)
        assert np.array_equal(y2.read(np.uint16).reshape(rows, n), y)
    for a in range(0, rows, 1000):
        hs, ys = run(index[a:a + 1000])
        assert np.array_equal(h[a:a + 1000], hs) and np.array_equal(y[a:a + 1000], ys)


# whole and partial 512-value chunks, the longest rows of the bf16 form and the
# next ones (general form)
@pytest.mark.parametrize("heads,vocab", [(1, 8), (1, 2056), (5, 1032), (16, 2104), (40, 1032), (41, 8)])
def test_embed_norm_table(heads, vocab):
    d = 128 * heads
    say(f"normalized embedding table {vocab} x {d}")
    x, _ = _rows(vocab, d, vocab + d)
    bits = oracle.f32_to_bf16_bits_np(x).reshape(vocab, d)
    dec = ca.Decoder(d, heads, 128, 1, vocab, 1, 16)
    dec.init_weights(seed=1, std=0.02)
    ca.mem_write(dec.tensor(ca.DEC_EMBED), bits)
    dec.prefill(ca.Buffer.from_array(np.zeros((1, 1), np.uint32)), 1, 1, ca.Buffer(4))
    tab = dec.read(ca.DEC_EMBED_NORM, np.uint16).reshape(vocab + 1, d)
    dec.close()
    want = od.residual_rmsnorm_bf16((bits.astype(np.uint32) << 16).view(np.float32))[1]
    as_f32 = lambda u: (u.astype(np.uint32) << 16).view(np.float32)  # noqa: E731
    _same(as_f32(tab[:vocab]), as_f32(want.reshape(vocab, d)))
    assert np.isnan(as_f32(tab[vocab])).all()
