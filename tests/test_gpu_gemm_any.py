"""gemm_bf16 on shapes and addresses no aligned tile kernel takes: the general
tile kernels, their k groups, the packing of rows that do not start on 16
bytes, and the kernel that needs neither, at the sizes where they change."""
import numpy as np
import pytest

import catena_amd as ca
import oracle
from gpu_util import as_f32, captured, gemm_within_bound, say

pytestmark = pytest.mark.gpu

NAN16 = 0x7FC1  # what surrounds every operand: a value read past one shows in the product


def _placed(bits: np.ndarray, shift: int):
    """`bits` in a device buffer of NaNs, `shift` elements past a 256-byte line."""
    flat = np.full(bits.size + 512, NAN16, np.uint16)
    flat[128 + shift:128 + shift + bits.size] = bits.reshape(-1)
    buf = ca.Buffer.from_array(flat)
    return buf, buf.ptr + 2 * (128 + shift)


def _product(a16, b16, out_f32, shifts=(0, 0, 0)):
    """gemm_bf16 into the middle of a buffer whose other bytes must not move."""
    n, k = a16.shape
    m = b16.shape[1]
    es = 4 if out_f32 else 2
    (ab, ap), (bb, bp) = _placed(a16, shifts[0]), _placed(b16, shifts[1])
    pad, fill = 256 + es * shifts[2], 0xA5
    cb = ca.Buffer.from_array(np.full(n * m * es + 512 + es * shifts[2], fill, np.uint8))
    ca.gemm_bf16(ap, bp, cb.ptr + pad, n, m, k, out_f32=out_f32)
    raw = cb.read(np.uint8)
    got = raw[pad:pad + n * m * es].copy().view(np.float32 if out_f32 else np.uint16).reshape(n, m)
    assert np.all(raw[:pad] == fill) and np.all(raw[pad + n * m * es:] == fill)
    return got


def _inputs(n, m, k, seed):
    rng = np.random.default_rng(seed)
    return (oracle.f32_to_bf16_bits_np(rng.normal(0, 1, (n, k)).astype(np.float32)),
            oracle.f32_to_bf16_bits_np(rng.normal(0, 1, (k, m)).astype(np.float32)))


def _check(n, m, k, shifts=(0, 0, 0)):
    say(f"bf16 gemm general {n}x{m}x{k} shifts {shifts}")
    a16, b16 = _inputs(n, m, k, n + 3 * m + 7 * k)
    g32 = _product(a16, b16, True, shifts)
    gemm_within_bound(a16, b16, g32)
    g16 = _product(a16, b16, False, shifts)
    assert np.array_equal(g16, oracle.f32_to_bf16_bits_np(g32))
    assert np.array_equal(_product(a16, b16, True, shifts).view(np.uint32), g32.view(np.uint32))
    return a16, b16, g32


# rows at the edges of 32, 64, 128 and 256-row tiles; widths and depths one off
# a tile, a 16-byte chunk, a k step; from one tile to several rounds of them
@pytest.mark.parametrize("n,m,k", [
    (17, 8, 8), (31, 40, 32), (32, 32, 40), (33, 64, 120), (63, 72, 136), (64, 128, 96), (65, 136, 264),
    (127, 248, 512), (129, 264, 1032), (255, 520, 96), (257, 256, 160), (513, 1032, 1000), (1000, 2056, 72),
    (700, 3000, 232), (1, 1, 1), (3, 7, 1000), (16, 9, 64), (5, 64, 9), (40, 33, 31), (100, 127, 129),
    (257, 511, 255), (300, 1000, 2), (643, 10944, 136), (766, 11050, 137), (965, 10944, 136), (967, 10947, 129),
    (20, 4096, 3), (256, 256, 128), (256, 384, 256), (512, 512, 640), (48, 4096, 2888)])
def test_general_shapes(n, m, k):
    _check(n, m, k)


# every tile, stored four or eight columns at a time and by the element
@pytest.mark.parametrize("n,m,k,tile", [
    (30, 79, 79, (32, 32)), (17, 248, 12, (32, 32)), (37, 4241, 80, (32, 64)), (33, 4172, 76, (32, 64)),
    (78, 5591, 67, (64, 64)), (69, 5488, 77, (64, 64)), (2051, 109, 9, (64, 128)), (40, 4316, 15, (64, 128)),
    (1869, 2342, 8, (128, 128)), (666, 5908, 8, (128, 128)), (2122, 5457, 43, (128, 192)), (2009, 6096, 8, (128, 192)),
    (1483, 5917, 8, (192, 128)), (1670, 4736, 8, (192, 128)), (1745, 2398, 9, (256, 256)), (726, 5380, 9, (256, 256)),
    (1000, 6144, 2048, (128, 128))])
def test_each_tile(n, m, k, tile):
    assert ca.gemm_bf16_plan(n, m, k) == (1, k) + tile
    _check(n, m, k)


# the 256 x 256 tile with ragged edges (the tile the host's estimate takes for
# these): 1, 15, 16, 17 rows in the last tile; 1, 15, 17 k rows in the last slab
# and slabs past k; B packed, A packed, both, none
@pytest.mark.parametrize("n,m,k", [(257, 13567, 1), (271, 14976, 1), (272, 14720, 1), (273, 14593, 1), (1025, 11648, 33),
                                   (1040, 10990, 33), (1537, 7681, 47), (1537, 7552, 49), (1281, 6138, 81),
                                   (1025, 11007, 64), (1025, 7432, 96)])
def test_ragged_256_tile(n, m, k):
    assert ca.gemm_bf16_plan(n, m, k)[2:] == (256, 256)
    # what the packed operands of a longer product leave in the scratch memory:
    # a row read past one of this product's shows as a NaN
    nan = np.full((n, k + 39), NAN16, np.uint16), np.full((k + 39, m), NAN16, np.uint16)
    _product(*nan, True)
    _check(n, m, k)


@pytest.mark.parametrize("shifts", [(1, 0, 0), (0, 1, 0), (0, 0, 1)])
def test_ragged_256_tile_unaligned(shifts):
    assert ca.gemm_bf16_plan(1025, 7432, 96)[2:] == (256, 256)
    _check(1025, 7432, 96, shifts)


# few tiles and a deep k: folded as 2 .. 16 k groups, the last one shorter
@pytest.mark.parametrize("n,m,k", [(17, 256, 8192), (24, 96, 4104), (48, 2048, 2888), (64, 512, 8200), (100, 1024, 5000),
                                   (33, 64, 16384), (20, 60, 4099), (48, 4096, 6024), (999, 2048, 5632)])
def test_k_groups(n, m, k):
    assert ca.gemm_bf16_plan(n, m, k)[0] > 1
    _check(n, m, k)
    _check(n, m, k, (0, 0, 1))  # the groups' sum stored by the element


# every address a caller may pass: 2, 4 and 8-byte aligned operands and outputs
@pytest.mark.parametrize("shifts", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (3, 5, 7), (4, 2, 2), (8, 8, 4)])
@pytest.mark.parametrize("n,m,k", [(8, 136, 64), (130, 264, 192), (256, 256, 128)])
def test_unaligned_operands(n, m, k, shifts):
    _check(n, m, k, shifts)


# the padded product's depth and narrow tiles: 32-k stages on narrow (129 .. 256)
# and on wide tiles (257 .. 512), 64-k stages (160 and more)
@pytest.mark.parametrize("n,m,k,pk,tiles", [
    (999, 768, 256, 256, 129), (999, 768, 256, 256, 257), (200, 1024, 544, 640, 129), (200, 1024, 544, 576, 160),
    (333, 1536, 160, 256, 257), (333, 1536, 160, 192, 160), (1000, 2048, 96, 128, 257), (1000, 1920, 96, 128, 129)])
def test_unsplit_bits_equal_the_aligned_kernels(n, m, k, pk, tiles):
    """A product that is not split has the bits of the same product padded to
    whole tiles, and repeated until the tile kernels take it: rows and k rows of
    zeros change no other cell's MFMA steps."""
    a16, b16, g32 = _check(n, m, k)
    assert ca.gemm_bf16_plan(n, m, k)[0] == 1
    pn = -(-n // 256) * 256
    ap, bp = np.zeros((pn, pk), np.uint16), np.zeros((pk, m), np.uint16)
    ap[:n, :k], bp[:k] = a16, b16
    copies = -(-tiles // (pn // 256 * -(-m // 128)))
    say(f"bf16 gemm padded {copies} x {pn}x{m}x{pk}")
    assert ca.gemm_bf16_plan(copies * pn, m, pk)[2:] == (0, 0)
    full = _product(np.concatenate([ap] * copies), bp, True)[:n]
    assert np.array_equal(full.view(np.uint32), g32.view(np.uint32))


def test_special_values_stay_in_their_row_and_column():
    """An infinity or NaN of row i reaches row i only, also where k ends inside
    a k step and the next row's values lie behind it (and so for columns)."""
    n, m, k = 70, 200, 72
    a16, b16 = _inputs(n, m, k, 5)
    clean = _product(a16, b16, True)
    a16[10, 0], a16[41, k - 1], b16[3, 77] = 0x7F80, 0x7FC0, 0xFF80
    got = _product(a16, b16, True)
    hit = np.zeros((n, m), bool)
    hit[[10, 41]], hit[:, 77] = True, True
    assert not np.isfinite(got[hit]).any()
    assert np.array_equal(got[~hit].view(np.uint32), clean[~hit].view(np.uint32))


def test_strides_past_the_32_bit_offsets():
    """k past 2^22: the kernel with 64-bit addressing (small integers: every
    partial sum exact, so any order gives the same bits)."""
    n, m, k = 17, 8, (1 << 22) + 64
    rng = np.random.default_rng(9)
    a16 = oracle.f32_to_bf16_bits_np(rng.integers(-1, 2, (n, k)).astype(np.float32))
    b16 = oracle.f32_to_bf16_bits_np(rng.integers(-1, 2, (k, m)).astype(np.float32))
    say(f"bf16 gemm {n}x{m}x{k}")
    want = as_f32(a16) @ as_f32(b16).astype(np.float64)
    assert np.array_equal(_product(a16, b16, True), want)
    assert np.array_equal(_product(a16, b16, False), oracle.f32_to_bf16_bits_np(want.astype(np.float32)))


@pytest.mark.parametrize("n,m", [(1, 1), (3, 7), (8, 128), (16, 9), (17, 8), (32, 32), (33, 31), (256, 256), (1000, 2056)])
@pytest.mark.parametrize("out_f32", [True, False])
def test_empty_fold(n, m, out_f32):
    """k == 0: every element is the fold's start, +0; the operands may be null."""
    es = 4 if out_f32 else 2
    say(f"bf16 gemm empty fold {n}x{m} f32 {out_f32}")
    cb = ca.Buffer.from_array(np.full(n * m * es + 512, 0xA5, np.uint8))
    ca.gemm_bf16(0, 0, cb.ptr + 256, n, m, 0, out_f32=out_f32)
    raw = cb.read(np.uint8)
    assert not raw[256:-256].any()
    assert np.all(raw[:256] == 0xA5) and np.all(raw[-256:] == 0xA5)


# whole tiles (one fold), k groups, the 256 x 256 tile, packed operands
ORDERED = [(256, 256, 8192), (512, 768, 4160), (17, 256, 8192), (64, 512, 8200), (100, 1024, 5000), (20, 60, 4099),
           (40, 777, 2072), (999, 2048, 5632), (1025, 7432, 96)]


@pytest.mark.parametrize("n,m,k", ORDERED)
def test_same_bits_at_any_address(n, m, k):
    """The order of a sum is the shape's, not the pointers'."""
    say(f"bf16 gemm at several addresses {n}x{m}x{k} plan {ca.gemm_bf16_plan(n, m, k)}")
    a16, b16 = _inputs(n, m, k, n + m + k)
    want = _product(a16, b16, True)
    gemm_within_bound(a16, b16, want)
    want16 = oracle.f32_to_bf16_bits_np(want)
    for shifts in [(1, 0, 0), (0, 1, 0), (0, 0, 1), (4, 4, 1), (5, 3, 2)]:
        assert np.array_equal(_product(a16, b16, True, shifts).view(np.uint32), want.view(np.uint32)), shifts
        assert np.array_equal(_product(a16, b16, False, shifts), want16), shifts


@pytest.mark.parametrize("n,m,k", ORDERED)
@pytest.mark.parametrize("shifts", [(0, 0, 0), (1, 0, 0), (3, 5, 1)])
@pytest.mark.parametrize("out_f32", [True, False])
def test_captured_bits_equal_eager(n, m, k, shifts, out_f32):
    """A graph takes no scratch memory: groups fold in sequence, unaligned
    operands on the kernel that loads by the element; the bits are the same, on
    every replay, whatever eager products do to the scratch in between."""
    say(f"bf16 gemm captured {n}x{m}x{k} shifts {shifts} f32 {out_f32}")
    a16, b16 = _inputs(n, m, k, n + m + k)
    es = 4 if out_f32 else 2
    (_ab, ap), (_bb, bp) = _placed(a16, shifts[0]), _placed(b16, shifts[1])
    cb, eager = (ca.Buffer.from_array(np.full(n * m * es + 64, 0xA5, np.uint8)) for _ in range(2))
    off = es * shifts[2]
    replay = captured(lambda: ca.gemm_bf16(ap, bp, cb.ptr + off, n, m, k, out_f32=out_f32))
    other = _inputs(33, 1024, 4099, 1)
    for _ in range(3):
        replay()
        ca.gemm_bf16(ap, bp, eager.ptr + off, n, m, k, out_f32=out_f32)
        assert np.array_equal(cb.read(np.uint8), eager.read(np.uint8))
        cb.write(np.full(n * m * es + 64, 0xA5, np.uint8))
        _product(*other, True)


def test_same_bits_without_scratch():
    """Operands whose packed copies pass the scratch limit: the groups on the
    kernel that loads by the element.  64 x 64 x 2^22 from aligned operands, from
    one unaligned (packed) and from both (1 GiB and more)."""
    n = m = 64
    k = 1 << 22
    say(f"bf16 gemm {n}x{m}x{k} without scratch")
    assert ca.gemm_bf16_plan(n, m, k)[0] > 1
    size = n * k
    rng = np.random.default_rng(4)
    one = oracle.f32_to_bf16_bits_np(rng.normal(0, 1, 999983).astype(np.float32))  # a prime: no two rows alike
    a16, b16 = np.resize(one, size), np.resize(one[::-1], size)
    flat = np.full(size + 128, NAN16, np.uint16)

    def place(x, shift):
        flat[:] = NAN16
        flat[64 + shift:64 + shift + size] = x
        buf = ca.Buffer.from_array(flat)
        return buf, buf.ptr + 2 * (64 + shift)
    out = []
    for sa, sb in [(0, 0), (0, 1), (1, 1)]:
        (_a, ap), (_b, bp) = place(a16, sa), place(b16, sb)
        for es in (4, 2):
            cb = ca.Buffer(n * m * es)
            ca.gemm_bf16(ap, bp, cb, n, m, k, out_f32=es == 4)
            out.append(cb.read(np.uint32 if es == 4 else np.uint16, (n, m)))
    assert np.isfinite(out[0].view(np.float32)).all() and np.any(out[0])
    for got in out[2::2]:
        assert np.array_equal(got, out[0])
    for got in out[1::2]:
        assert np.array_equal(got, oracle.f32_to_bf16_bits_np(out[0].view(np.float32)))


def test_scratch_is_given_back():
    """Packed operands sit in a block of their own, which catena_pool_trim
    returns; the next product takes a new one."""
    n, m, k = 70, 2049, 4099
    a16, b16 = _inputs(n, m, k, 11)
    want = _product(a16, b16, True)
    say("scratch given back")
    live = ca.pool_stats()["bytes_live"]
    ca.lib().catena_pool_trim()
    assert ca.pool_stats()["bytes_live"] <= live - k * m * 2
    assert ca.pool_stats()["bytes_cached"] == 0
    assert np.array_equal(_product(a16, b16, True).view(np.uint32), want.view(np.uint32))


def test_captured_decode_product_outlives_larger_products():
    """A graph of the decode GEMM holds the address of its partials: products
    that need more scratch, and a trim, leave that block where it is."""
    n, m, k = 8, 4096, 11008
    assert ca.gemm_bf16_decode_plan(n, m, k)[0] > 1
    a16, b16 = _inputs(n, m, k, 12)
    ab, bb, cb = ca.Buffer.from_array(a16), ca.Buffer.from_array(b16), ca.Buffer(n * m * 4)
    ca.gemm_bf16(ab, bb, cb, n, m, k, out_f32=True)  # sizes the block
    want = cb.read(np.uint32)
    say("decode gemm captured, larger products between replays")
    replay = captured(lambda: ca.gemm_bf16(ab, bb, cb, n, m, k, out_f32=True))
    big = _inputs(65, 8193, 4099, 13)
    for _ in range(3):
        _product(*big, True)
        ca.lib().catena_pool_trim()
        # what would now sit where the block was
        held = [ca.Buffer.from_array(np.full(1 << s, 0xA5, np.uint8)) for s in range(18, 25)]
        cb.write(np.zeros(n * m, np.float32))
        replay()
        assert np.array_equal(cb.read(np.uint32), want)
        for h in held:
            assert np.all(h.read(np.uint8) == 0xA5)
