// bf16 GEMM on gfx950 MFMA for every shape the 256-row tile kernels do not
// take or would leave most CUs idle on: few rows, ragged rows and columns,
// any K.
//
// Contraction and order are those of gemm_bf16_k32.hip (reference semantics:
// catena-lang/stdlib/matrix.hex:236-327 on bf16 inputs widened exactly, f32
// accumulation, NN row-major): K ascending in v_mfma_f32_16x16x32_bf16 steps,
// one owner per output tile, so with splits == 1 every output element has the
// tile kernels' bits, whatever tile computes it.  With splits > 1 (grid.y)
// split z folds k in [z k_len, (z + 1) k_len) in that order into its own f32
// partial P[z] = [M][N], and a second launch adds them in ascending z; the
// split is a function of the shape alone.  No atomics.  The seq kernels fold
// the same groups one after the other in one workgroup and add each to the
// sum of those before it: the same bits where no memory for partials may be
// taken.
//
// Operands: A [M] rows of stride lda, B [K] rows of stride ldb, both strides
// multiples of 8 elements and both pointers 16-byte aligned (the host packs an
// operand that is neither).  Columns K .. of A's last 8-element chunk, when K
// % 8 != 0, are zeros (the pack writes them); nothing is assumed past a chunk.
//
// Layout: BM x BN output tile, WM x WN waves, stages of KS 32-k slabs in LDS,
// filled by 16-byte direct-to-LDS buffer loads.  Each load instruction (1 KiB)
// has its own descriptor whose record count ends at the operand's last row, so
// rows past M and k rows past K arrive as zeros without touching memory; a
// chunk of A past K gets an offset outside the descriptor.  Columns past N
// read the next row's values and are not stored.
// Swizzles: A [BM][64 B] as in gemm_bf16_k32.hip; B [32][2 BN B], chunk p of
// row k holds global chunk p ^ hB(k), where hB spreads the 16 rows of a
// transposing read over the 256-byte bank space for the row length at hand.
// What bounds it: the 128 x 128 tile (two workgroups to a CU) its LDS reads, 8
// KiB per 16 MFMAs of a wave; the small tiles the latency of a stage, so they
// fold four slabs to a barrier; few rows over a deep K the stream of B, hence
// the k groups.  Measured against the bounds-checked register-staged kernel
// (gemm_bf16.hip) that took these shapes: 1000 x 6144 x 2048 f32 out 416 -> 33
// us (770 TFLOP/s), 64 x 4096 x 11008 bf16 out 1658 -> 22.2 us with 8 k groups
// (4.1 TB/s; 38 us whole), 999 x 2048 x 5632 1300 -> 40 us.  Tried for the 128
// x 128 tile at 1000 x 6144 x 2048: stages of one slab, 4 deep 40 us, 3 deep
// 38; eight waves 37; the 256 x 128 kernel 36.
// The 192 x 128 and 128 x 192 tiles (also two workgroups to a CU, exactly its
// LDS) read 20 % less LDS per MFMA and fill rounds that 128 x 128 leaves half
// empty: 1340 x 6400 x 1408 46.3 -> 36.7 us, 1119 x 8320 x 4096 107 -> 88, 2816 x
// 10368 x 1920 149 -> 120, 999 x 11264 x 2048 60.9 -> 52.9.  Tried beside them
// and no better over 150 shapes: 128 x 192 in eight waves, three or four stages
// (one workgroup to a CU), 256 x 192, fragments double-buffered in registers.
// One barrier per stage: it follows the wait for the stage's loads and frees
// the buffer read one stage earlier, which the loads of stage t + S - 1 then
// fill, so S - 1 stages are in flight while one is multiplied.
#include "common.h"

namespace {
constexpr int BK = 32;
constexpr int kRsrcWord3 = 0x00020000;  // raw buffer, 32-bit access
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) i16x4_t lds_i16x4;

template <int BN>
CATENA_DEV uint32_t hB(uint32_t k) {
  if (BN == 128) return 2u * ((k & 3u) | (((k >> 3) & 1u) << 2));  // 256-byte rows: all alias
  if (BN == 64 || BN == 192) return 2u * (((k >> 1) & 1u) | (((k >> 3) & 1u) << 1));  // 128- and 384-byte rows: row parity picks the half
  return 2u * ((k >> 3) & 1u);                                     // 64-byte rows: k & 3 picks the quarter
}

CATENA_DEV bf16x8_t cat_bf16(i16x4_t lo, i16x4_t hi) {
  typedef short i16x8_t __attribute__((ext_vector_type(8)));
  i16x8_t v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8_t, v);
}

// Workgroup -> tile: each XCD takes a contiguous share of the tiles (workgroup
// ids go to the 8 XCDs round robin), walked in groups of 4 tile rows.
CATENA_DEV void tile_of(uint32_t bid, uint32_t tiles_m, uint32_t tiles_n, uint32_t& tm, uint32_t& tn) {
  const uint32_t total = tiles_m * tiles_n, q = total / 8u, rem = total % 8u, x = bid % 8u;
  bid = x * q + (x < rem ? x : rem) + bid / 8u;
  const uint32_t GROUP_M = 4, in_group = GROUP_M * tiles_n;
  const uint32_t first_m = bid / in_group * GROUP_M;
  const uint32_t gsize = tiles_m - first_m < GROUP_M ? tiles_m - first_m : GROUP_M;
  const uint32_t r = bid % in_group;
  tm = first_m + r % gsize;
  tn = r / gsize;
}

#define CATENA_WAIT_VMCNT(n) \
  __builtin_amdgcn_s_waitcnt((((n) & 15) | (((n) >> 4) << 14)) | 0x0070 | 0x0F00)

// Bytes of a descriptor that covers `n` elements (0 when n <= 0), in 31 bits
CATENA_DEV int records(int64_t n) {
  const int64_t b = n * 2;
  return b <= 0 ? 0 : b > 0x7FFFFFF0ll ? 0x7FFFFFF0 : (int)b;
}

template <int BM, int BN, int WM, int WN, int KS, int S, bool OUT_BF16, bool SEQ = false>
CATENA_DEV void gemm_any_body(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                              void* __restrict__ C, uint64_t M, uint64_t N, uint64_t K_all,
                              uint64_t lda, uint64_t ldb, uint64_t k_len, uint32_t vec) {
  constexpr int WAVES = WM * WN;
  constexpr int WI = BM / WM / 16, WJ = BN / WN / 16;  // 16 x 16 blocks per wave
  constexpr int A_ST = BM * BK, B_ST = BK * BN, ST = KS * (A_ST + B_ST);  // elements
  constexpr int A_INS = BM / 16, B_INS = BN / 16;      // 1-KiB loads per slab
  static_assert(KS * A_INS % WAVES == 0 && KS * B_INS % WAVES == 0, "whole loads per wave");
  constexpr int LA = KS * A_INS / WAVES, LB = KS * B_INS / WAVES, LOADS = LA + LB;  // per wave and stage
  constexpr int BL = BN / 8;                           // 16-byte chunks per B row
  extern __shared__ __attribute__((aligned(1024))) uint16_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  uint32_t tm, tn;
  tile_of(blockIdx.x, (uint32_t)((M + BM - 1) / BM), (uint32_t)((N + BN - 1) / BN), tm, tn);
  const uint64_t m0 = (uint64_t)tm * BM, n0 = (uint64_t)tn * BN;
  uint64_t kbeg = SEQ ? 0 : (uint64_t)blockIdx.y * k_len;
  int64_t kend = (int64_t)(kbeg + k_len < K_all ? kbeg + k_len : K_all);

  // Load l of a wave: A load x = wave LA + l is rows 16 (x % A_INS) .. +15 of
  // slab x / A_INS; B load x = wave LB + l rows BR (x % B_INS) .. of slab
  // x / B_INS.  Lane offsets (bytes from the stage's first element) and, for
  // A, the lane's k within the stage.
  uint32_t aoff[LA], boff[LB];
  int ak[LA];
#pragma unroll
  for (int l = 0; l < LA; ++l) {
    const int x = wave * LA + l;
    const uint32_t r = 16 * (x % A_INS) + ((uint32_t)lane >> 2);
    ak[l] = x / A_INS * BK + 8 * (int)((uint32_t)(lane & 3) ^ ((r >> 1) & 3u));
    aoff[l] = (uint32_t)((r * lda + ak[l]) * 2);
  }
#pragma unroll
  for (int l = 0; l < LB; ++l) {
    const int x = wave * LB + l;
    const uint32_t ch = 64 * (x % B_INS) + (uint32_t)lane;  // 16-byte chunk of the slab
    const uint32_t kr = ch / BL, q = ch % BL ^ hB<BN>(kr);  // its row, the global chunk it holds
    boff[l] = (uint32_t)(((x / B_INS * BK + kr) * ldb + 8 * q) * 2);
  }
  auto a_dst = [&](int buf, int l) {
    const int x = wave * LA + l;
    return (lds_void*)(smem + buf * ST + x / A_INS * (A_ST + B_ST) + x % A_INS * 16 * BK);
  };
  auto b_dst = [&](int buf, int l) {
    const int x = wave * LB + l;
    return (lds_void*)(smem + buf * ST + x / B_INS * (A_ST + B_ST) + A_ST + x % B_INS * 512);
  };
  auto issue = [&](int64_t k0, int buf) {  // the stage at k0 into buffer buf
    const int64_t left = kend - k0;        // k rows left (<= 0: every load brings zeros)
    const int64_t kl = left > 0 ? k0 : 0;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(A + m0 * lda + kl), (short)0,
        left > 0 ? records((int64_t)((M - m0) * lda) - kl) : 0, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(B + kl * ldb + n0), (short)0, left > 0 ? records(left * (int64_t)ldb - (int64_t)n0) : 0,
        kRsrcWord3);
    const int lim = left < KS * BK ? (int)left : KS * BK;
#pragma unroll
    for (int l = 0; l < LA; ++l)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, a_dst(buf, l), 16, ak[l] < lim ? (int)aoff[l] : 0x7FFFFFF0, 0,
                                               0, 0);
#pragma unroll
    for (int l = 0; l < LB; ++l)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, b_dst(buf, l), 16, (int)boff[l], 0, 0, 0);
  };

  // Fragment read bases (bytes within a slab), as in gemm_bf16_k32.hip
  const int G = lane >> 4, s = lane & 15;
  const uint32_t a_lds = (wm * 16 * WI + s) * BK * 2 + 16 * ((uint32_t)G ^ ((uint32_t)(s >> 1) & 3u));
  const uint32_t b_krow = 8 * G + (s >> 2);
  uint32_t b_lds[WJ][2];
#pragma unroll
  for (int j = 0; j < WJ; ++j) {
    const uint32_t col = wn * 16 * WJ + 16 * j + 4 * (s & 3);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      b_lds[j][h] = A_ST * 2 + (b_krow + 4 * h) * BN * 2 + 16 * ((col >> 3) ^ hB<BN>(b_krow + 4 * h)) + 2 * (col & 7);
  }

  f32x4_t acc[WI][WJ];
  f32x4_t sum[SEQ ? WI : 1][SEQ ? WJ : 1];  // of the groups before this one
  for (;;) {
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int64_t kspan = kend - (int64_t)kbeg;
    const uint64_t nt = kspan > 0 ? (uint64_t)(kspan + KS * BK - 1) / (KS * BK) : 0;
#pragma unroll
    for (int t = 0; t < S - 1; ++t) issue((int64_t)kbeg + t * KS * BK, t);
    int buf = 0;
    for (uint64_t t = 0; t < nt; ++t) {
      CATENA_WAIT_VMCNT(LOADS * (S - 2));  // this wave's loads of stage t have landed
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();        // every wave's have, and stage t - 1 is read
      asm volatile("" ::: "memory");
      issue((int64_t)kbeg + (int64_t)(t + S - 1) * KS * BK, buf == 0 ? S - 1 : buf - 1);
      const char* st = reinterpret_cast<const char*>(smem + buf * ST);
#pragma unroll
      for (int u = 0; u < KS; ++u) {
        const char* sl = st + u * (A_ST + B_ST) * 2;
        bf16x8_t fa[WI], fb[WJ];
#pragma unroll
        for (int i = 0; i < WI; ++i)
          fa[i] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(sl + a_lds + i * 16 * BK * 2));
#pragma unroll
        for (int j = 0; j < WJ; ++j)
          fb[j] = cat_bf16(__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(sl + b_lds[j][0])),
                           __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(sl + b_lds[j][1])));
#pragma unroll
        for (int j = 0; j < WJ; ++j)
#pragma unroll
          for (int i = 0; i < WI; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the buffer is read before the next barrier
      buf = buf + 1 == S ? 0 : buf + 1;
    }
    CATENA_WAIT_VMCNT(0);  // no LDS writes outstanding past this point
    if constexpr (!SEQ) {
      break;
    } else {
#pragma unroll
      for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int j = 0; j < WJ; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[i][j][q] = sum[i][j][q] = kbeg ? sum[i][j][q] + acc[i][j][q] : acc[i][j][q];
      kbeg += k_len;
      if (kbeg >= K_all) break;
      kend = (int64_t)(kbeg + k_len < K_all ? kbeg + k_len : K_all);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();  // every wave has read this group's stages
      asm volatile("" ::: "memory");
    }
  }

  // acc[i][j] lane (G, s) holds C[row 16 i + s][cols 16 j + 4G .. +3]; vec: N
  // and C's address let four columns be stored at once
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const uint64_t gr = m0 + wm * 16 * WI + 16 * i + s;
    if (gr >= M) continue;
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const uint64_t gc = n0 + wn * 16 * WJ + 16 * j + 4 * G;
      const f32x4_t v = acc[i][j];
      if (OUT_BF16) {
        uint16_t* c = static_cast<uint16_t*>(C) + gr * N + gc;
        if (vec) {
          if (gc < N) *reinterpret_cast<uint2*>(c) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (gc + q < N) c[q] = (uint16_t)f32_to_bf16_bits(v[q]);
        }
      } else {
        float* c = static_cast<float*>(C) + ((SEQ ? 0 : (uint64_t)blockIdx.y * M) + gr) * N + gc;
        if (vec) {
          if (gc < N) *reinterpret_cast<f32x4_t*>(c) = v;
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (gc + q < N) c[q] = v[q];
        }
      }
    }
  }
}
}  // namespace

// grid (tiles, splits), or tiles where SEQ; block 64 WM WN, dynamic LDS S KS (BM +
// BN) 64 B
#define CATENA_GEMM_ANY(NAME, SEQ, BM, BN, WM, WN, KS, S)                                                \
  extern "C" __global__ __launch_bounds__(64 * WM * WN) void catena_gemm_bf16_any_##NAME##_f32out(       \
      const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, void* __restrict__ C, uint64_t M,  \
      uint64_t N, uint64_t K, uint64_t lda, uint64_t ldb, uint64_t k_len, uint32_t vec) {                \
    gemm_any_body<BM, BN, WM, WN, KS, S, false, SEQ>(A, B, C, M, N, K, lda, ldb, k_len, vec);            \
  }                                                                                                      \
  extern "C" __global__ __launch_bounds__(64 * WM * WN) void catena_gemm_bf16_any_##NAME##_bf16out(      \
      const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, void* __restrict__ C, uint64_t M,  \
      uint64_t N, uint64_t K, uint64_t lda, uint64_t ldb, uint64_t k_len, uint32_t vec) {                \
    gemm_any_body<BM, BN, WM, WN, KS, S, true, SEQ>(A, B, C, M, N, K, lda, ldb, k_len, vec);             \
  }

CATENA_GEMM_ANY(192x128, false, 192, 128, 2, 2, 2, 2)
CATENA_GEMM_ANY(128x192, false, 128, 192, 2, 2, 2, 2)
CATENA_GEMM_ANY(128x128, false, 128, 128, 2, 2, 2, 2)
CATENA_GEMM_ANY(64x128, false, 64, 128, 2, 2, 2, 3)
CATENA_GEMM_ANY(64x64, false, 64, 64, 2, 2, 4, 2)
CATENA_GEMM_ANY(32x64, false, 32, 64, 1, 4, 4, 6)
CATENA_GEMM_ANY(32x32, false, 32, 32, 2, 2, 4, 4)
CATENA_GEMM_ANY(64x64_seq, true, 64, 64, 2, 2, 4, 2)
CATENA_GEMM_ANY(32x32_seq, true, 32, 32, 2, 2, 4, 4)

// An operand whose rows do not start on 16 bytes, copied to rows of ld
// elements (a multiple of 8) with zeros past its columns: dst[r][0 .. ld).
// One 8-element chunk per thread, chunks in order, so both sides are streamed;
// a whole chunk is one unaligned 16-byte load.
extern "C" __global__ __launch_bounds__(256) void catena_pack_rows_bf16(const uint16_t* __restrict__ src,
                                                                        uint64_t rows, uint64_t cols,
                                                                        uint16_t* __restrict__ dst, uint64_t ld) {
  const uint64_t per = ld / 8, total = rows * per;
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (uint64_t)gridDim.x * 256) {
    const uint64_t r = i / per, c = 8 * (i % per);
    const uint16_t* p = src + r * cols + c;
    u32x4_t w = {0u, 0u, 0u, 0u};
    if (c + 8 <= cols) {
      __builtin_memcpy(&w, p, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (c + e < cols) w[e >> 1] |= (uint32_t)p[e] << (16 * (e & 1));
    }
    *reinterpret_cast<u32x4_t*>(dst + r * ld + c) = w;
  }
}
