// Kernel ABI: shape checks, kernel selection and launches.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#include "internal.h"

using namespace catena;

namespace {
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

uint64_t ceil_div(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// 256 x 128 tiles instead of 256 x 256: measured on the box, a round of
// 256 x 128 tiles (one per CU) takes ~0.6 of a round of 256 x 256 tiles at the
// same K, so the narrow tiles win when the wide ones leave CUs idle (W_o and
// W_down of the C5 prefill: 128 wide tiles for 256 CUs, 52.6 -> 37.6 us and
// 124 -> 93 us) and lose on full rounds (4096^3: 115 -> 138 us).
bool prefer_n128(uint64_t rows, uint64_t cols, int cu_count) {
  const uint64_t cus = cu_count > 0 ? (uint64_t)cu_count : 256;
  const uint64_t wide = (rows / 256) * (cols / 256);
  const uint64_t narrow = (rows / 256) * (cols / 128);
  const double r_wide = (double)ceil_div(wide, cus), r_narrow = (double)ceil_div(narrow, cus);
  return 0.62 * r_narrow < r_wide;
}

// Column blocks x k groups the decode kernel spreads a weight over: the
// MI355X's 256 CUs, one 4-wave workgroup per CU.  A constant, not the
// device's CU count: the k grouping fixes which partial sums are added
// together, so it must depend on the shape alone for the bits to be the same
// on every device (a partitioned MI355X shows fewer CUs).
constexpr uint64_t kDecodeSpread = 256;

// k per wave for the decode kernel, in whole 32-k MFMA steps, from (N, K)
// only.  Streaming path (K % 32 == 0, one 4-wave workgroup per CU for its
// 144 KiB LDS ring; each wave keeps 36 KiB in flight): the fewest k groups
// that still give each of the 256 CUs a workgroup, so one round of
// workgroups streams the weight and few partials are added, but no fewer
// than 8 steps per wave, or 2 when the weight is at most 16 MiB: such a
// kernel is bound by latency, not by HBM, and more workgroups shorten each
// stream (measured: 8 x 2048 x 2048 takes 7.5 us at 2 steps per wave against
// 9.4 us at 8; the C3 shapes and the larger decoder projections are fastest
// at the 8-step floor or within 0.5 us of it).  Register path (K % 32 != 0):
// ~1500 waves.
uint32_t decode_kw(uint64_t n_cols, uint64_t k, bool regs_path) {
  const uint64_t blocks = ceil_div(n_cols, 128);
  uint64_t kw;
  if (!regs_path) {
    // at least 8 steps of 32 k per wave: shorter chunks pay the ring's fill
    // and the partials' reduction more often than they gain in spread
    const uint64_t groups = blocks >= kDecodeSpread ? 1 : kDecodeSpread / blocks;
    kw = ceil_div(k, 4 * groups);
    kw = ceil_div(kw, 32) * 32;
    const uint64_t min_kw = n_cols * k * 2 <= (16ull << 20) ? 64 : 256;
    if (kw < min_kw) kw = min_kw;
  } else {
    kw = ceil_div(k * blocks, 1536);
    kw = ceil_div(kw, 32) * 32;
    if (kw < 64) kw = 64;
  }
  if (kw > k) kw = ceil_div(k, 32) * 32;
  return (uint32_t)kw;
}
// The tile kernels of a product, with what the choice between them weighs.
// `alone` and `shared`: microseconds per 32-k slab of one workgroup that has
// its CU to itself, and of each of the `fit` workgroups that share a CU;
// `stream`: GB/s at which one CU brings a weight in from HBM (the narrower
// the tile's rows, the less).  Fitted to timings over n = 17 .. 4000, widths
// 256 .. 11264 and depths 512 .. 11008, 1 to 16 k groups.  On 110 other products
// of n = 17 .. 4000, widths 256 .. 11008 and depths 128 .. 11008, with every tile
// and number of groups timed, the choice takes 3.6 % more than the fastest on
// average and 18 % at worst, of which the timing's spread is up to 10, and 6.5 %
// less than the fastest undivided one.
struct GemmTile {
  KernelId f32, bf16;
  uint32_t bm, bn, waves, stages, stage_k, fit;
  double alone, shared, stream;
};
constexpr GemmTile kGemmTiles[] = {
    {KernelId::GemmBf16Any192x128F32, KernelId::GemmBf16Any192x128Bf16, 192, 128, 4, 2, 64, 2, 0.44, 0.27, 36.3},
    {KernelId::GemmBf16Any128x192F32, KernelId::GemmBf16Any128x192Bf16, 128, 192, 4, 2, 64, 2, 0.46, 0.29, 36.3},
    {KernelId::GemmBf16Any128x128F32, KernelId::GemmBf16Any128x128Bf16, 128, 128, 4, 2, 64, 2, 0.358, 0.211, 36.3},
    {KernelId::GemmBf16Any64x128F32, KernelId::GemmBf16Any64x128Bf16, 64, 128, 4, 3, 64, 2, 0.217, 0.158, 36.3},
    {KernelId::GemmBf16Any64x64F32, KernelId::GemmBf16Any64x64Bf16, 64, 64, 4, 2, 128, 2, 0.169, 0.105, 33.5},
    {KernelId::GemmBf16Any32x64F32, KernelId::GemmBf16Any32x64Bf16, 32, 64, 4, 6, 128, 1, 0.120, 0.120, 33.5},
    {KernelId::GemmBf16Any32x32F32, KernelId::GemmBf16Any32x32Bf16, 32, 32, 4, 4, 128, 2, 0.075, 0.067, 24.8},
    {KernelId::GemmBf16K32EdgeF32, KernelId::GemmBf16K32EdgeBf16, 256, 256, 8, 4, 32, 1, 0.705, 0.705, 36.3},
};
constexpr int kTileRagged256 = 7;
// the two of them that fold groups in sequence, and that form's kernels
constexpr int kTileSeq64 = 4, kTileSeq32 = 6;
// k groups a product may be split into (with 1: whole)
constexpr uint32_t kGemmSplits[] = {1, 2, 3, 4, 6, 8, 12, 16};
// row strides up to which the general kernels' 32-bit offsets reach (a stage
// of 128 rows)
constexpr uint64_t kGemmMaxStride = 1ull << 22;
// most scratch one product takes: packed operands and partials (a product
// that needs more runs on the kernel that needs none)
constexpr uint64_t kGemmScratchMax = 1ull << 30;

// k per group, in whole stages
uint64_t gemm_k_len(uint64_t k, uint32_t splits, uint32_t stage_k) {
  return ceil_div(ceil_div(k, splits), stage_k) * stage_k;
}

// Estimated microseconds.  A function of the shape alone (kDecodeSpread
// stands for the CUs), so that the k groups, which fix the order of a sum,
// are the same on every device.
double gemm_cost(const GemmTile& t, uint64_t n, uint64_t m, uint64_t k, uint32_t splits) {
  const double wgs = (double)ceil_div(n, t.bm) * (double)ceil_div(m, t.bn) * splits;
  const double per_cu = std::ceil(wgs / kDecodeSpread);
  const double whole = std::floor(per_cu / t.fit) * t.fit, left = per_cu - whole;
  const double slab = whole * t.shared + (left > 0 ? std::max(t.alone, left * t.shared) : 0.0);
  const double fold = (double)gemm_k_len(k, splits, t.stage_k) / 32 * slab;
  const double weight = 2.0 * (double)k * (double)m / (std::min(wgs, (double)kDecodeSpread) * t.stream * 1e3);
  const double out = 4.0 * (double)n * (double)m / 4.8e6;  // one f32 pass over the output
  double us = 2.5 + std::max(fold, weight) + out * splits;
  if (splits > 1) us += 2.8 + out * (splits + 1);  // the launch that adds the partials
  return us;
}

struct GemmPlan {
  int tile = 0;
  uint32_t splits = 1;
  double us = 0;
};
// ragged256: the 256 x 256 kernel may run (A's rows hold whole 32-k slabs, as
// they do when k % 32 == 0 or when k % 8 != 0, which packs them).  k > 0
// when may_split (an empty fold has no groups).
GemmPlan gemm_plan(uint64_t n, uint64_t m, uint64_t k, bool ragged256, bool may_split) {
  GemmPlan best;
  best.us = -1;
  for (int i = 0; i < (int)(sizeof(kGemmTiles) / sizeof(kGemmTiles[0])); ++i) {
    const GemmTile& t = kGemmTiles[i];
    if (i == kTileRagged256 && !ragged256) continue;
    if (ceil_div(n, t.bm) * ceil_div(m, t.bn) > 0x7FFFFFFFull) continue;
    for (uint32_t s : kGemmSplits) {
      if (s > 1 && (!may_split || i == kTileRagged256 || n * m * 4 * s > kGemmScratchMax / 4 ||
                    ceil_div(k, gemm_k_len(k, s, t.stage_k)) != s))
        continue;
      const double us = gemm_cost(t, n, m, k, s);
      if (best.us < 0 || us < best.us) best = GemmPlan{i, s, us};
    }
  }
  return best;
}

// The 32-k stage kernels need K % 128 == 0 (whole groups of 4 stages); they
// address A's 256-row tile and B's 32-row slab with 32-bit buffer offsets.
bool k32_stages(uint64_t m, uint64_t k) {
  return k % 128 == 0 && k > 0 && k <= (1ull << 22) && m <= (1ull << 24);
}
// Shapes of whole 256-row tiles.  They are never split into k groups: their
// order is the one the decoder's fused projections share.
bool whole_tiles(uint64_t n, uint64_t m, uint64_t k) {
  return k > 0 && n % 256 == 0 && ((m % 256 == 0 && k % 64 == 0) || (m % 128 == 0 && k32_stages(m, k)));
}
// The general kernels' 32-bit offsets reach these row strides
bool strides_fit(uint64_t m, uint64_t k) { return k <= kGemmMaxStride && m <= kGemmMaxStride; }
// Whole tiles that the 256-row tile kernels take when the pointers are aligned.
// Up to 128 of the narrow tiles half the CUs would be idle: then the general
// kernels' smaller tiles are faster (256 x 2048 x 2048: 16 narrow tiles take 38
// us, 256 tiles of 32 x 64 10 us; 512 x 8192 x 4096, 128: 48 / 45; past it they are
// not: 3328 x 1280 x 1408, 130: 22.3 / 23.3; 512 x 9728 x 768, 152: 14.0 / 16.8; 768
// x 6272 x 128, 147: 7.9 / 9.0).  The 64-k stage kernel, on wide tiles alone, is
// passed up to 159 (1536 x 2816 x 1600, 132: 39.5 / 25.4).
bool tile_kernels(uint64_t n, uint64_t m, uint64_t k) {
  const uint64_t few = k32_stages(m, k) ? 128 : 159;
  return whole_tiles(n, m, k) && !((n / 256) * ceil_div(m, 128) <= few && strides_fit(m, k));
}

// The k groups of a general product and the tile they are folded on: what
// fixes the order of its sums, so a function of (n, m, k) alone, never of
// addresses, of scratch memory or of stream capture.
GemmPlan gemm_order(uint64_t n, uint64_t m, uint64_t k, bool may_split) {
  const bool splittable = may_split && k > 0 && n * m % 4 == 0 && strides_fit(m, k) && !whole_tiles(n, m, k);
  return gemm_plan(n, m, k, k > 0 && (k % 32 == 0 || k % 8 != 0), splittable);
}

// Y = P[0] + P[1] + ... + P[S-1] in ascending order, f32 or bf16
int reduce_parts(const float* P, uint64_t S, uint64_t elems, void* Y, bool bf16) {
  uint64_t stride4 = elems / 4;
  uint32_t S32 = (uint32_t)S, b = bf16 ? 1u : 0u;
  void* args[] = {&P, &stride4, &S32, &Y, &elems, &b};
  return launch(KernelId::DecodeReduce, dim3((unsigned)ceil_div(elems, 1024)), dim3(256), 0, args);
}

int pack_rows(const uint16_t* src, uint64_t rows, uint64_t cols, uint16_t* dst, uint64_t ld) {
  const uint64_t g = ceil_div(rows * (ld / 8), 256);
  void* args[] = {&src, &rows, &cols, &dst, &ld};
  return launch(KernelId::PackRowsBf16, dim3((unsigned)(g < 16384 ? g : 16384)), dim3(256), 0, args);
}
}  // namespace

namespace catena {

uint64_t decode_partials_bytes(uint64_t n, uint64_t m, uint64_t k, uint32_t* k_groups) {
  const uint32_t kw = decode_kw(m, k, k % 32 != 0);
  const uint64_t S = ceil_div(ceil_div(k, kw), 4);
  if (k_groups) *k_groups = S > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)S;
  return S > 1 ? S * n * m * sizeof(float) : 0;
}

int gemm_bf16_decode(const uint16_t* a, const uint16_t* b, void* c, uint64_t n, uint64_t m,
                     uint64_t k, DecodeEpilogue epi, const DecodeEpiArgs& ep, void* scratch,
                     uint64_t scratch_bytes, bool whole_k) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0 || m == 0) return CATENA_OK;
  if (n > 16 || k == 0 || m % 8 != 0 || k % 8 != 0 || !aligned16(a) || !aligned16(b) ||
      !aligned16(c))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "decode GEMM shape or alignment");
  Device& d = device();
  const uint32_t M = (uint32_t)n;
  // streaming ring (4 waves x 4 stages x 9 KiB) when K % 32 == 0, else the
  // register path with the reduction buffers only (4 x 8 KiB wave sums + the
  // 16 x 132 f32 tile)
  const bool regs_path = k % 32 != 0;
  if (ep.x_sums && (regs_path || !ep.x_rows_out || !aligned16(ep.x_sums) || ep.x_sums_blocks == 0 ||
                    ep.x_sums_cols == 0 || ep.x_sums_cols >= 0x7FFFFFFFull ||
                    (uint64_t)n * ep.x_sums_blocks * 16 >= (1ull << 31)))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "decode GEMM token composition operands");
  const uint32_t kw =
      whole_k && !regs_path ? (uint32_t)(ceil_div(ceil_div(k, 4), 32) * 32) : decode_kw(m, k, regs_path);
  const uint64_t chunks = ceil_div(k, kw);
  const uint64_t S = ceil_div(chunks, 4);
  const uint64_t gx = ceil_div(m, 128);
  if (S > 65535 || gx > Device::kTicketsGemm)
    return fail(CATENA_ERR_UNSUPPORTED, "decode GEMM grid too large");
  KernelId id = KernelId::GemmBf16DecodeF32;
  DecodeEpiArgs e = ep;
  switch (epi) {
    case DecodeEpilogue::StoreF32: break;
    case DecodeEpilogue::StoreBf16: id = KernelId::GemmBf16DecodeBf16; break;
    case DecodeEpilogue::Rope:
      if (e.heads == 0 || m != 3ull * e.heads * 128 || !e.q_out || !e.k_cache || !e.v_cache ||
          !e.lens || !e.inv_freq)
        return fail(CATENA_ERR_INVALID_ARGUMENT, "rope epilogue operands");
      id = KernelId::GemmBf16DecodeRope;
      break;
    case DecodeEpilogue::Silu:
      if (m % 128 != 0 || !e.act) return fail(CATENA_ERR_INVALID_ARGUMENT, "silu epilogue operands");
      id = KernelId::GemmBf16DecodeSilu;
      break;
    case DecodeEpilogue::Partials:
      id = KernelId::GemmBf16DecodeParts;
      break;
    case DecodeEpilogue::Argmax:
      if ((!e.idx && !e.arg_defer) || m >= 0x7FFFFFFFull)
        return fail(CATENA_ERR_INVALID_ARGUMENT, "argmax epilogue operands");
      if (n * gx * 16 > Device::kRowPartialBytes)
        return fail(CATENA_ERR_UNSUPPORTED, "argmax epilogue over %llu column blocks",
                    (unsigned long long)gx);
      e.arg_ticket = d.misc_tickets();
      if (!e.arg_partials) e.arg_partials = static_cast<uint32_t*>(d.row_partials());
      else if (!aligned16(e.arg_partials))
        return fail(CATENA_ERR_INVALID_ARGUMENT, "argmax summaries must be 16-byte aligned");
      id = KernelId::GemmBf16DecodeArgmax;
      break;
  }
  float* P = nullptr;
  std::lock_guard<std::mutex> ws_guard(d.ws_mu);  // the workspace block stays ours until launched
  if (S > 1) {
    // the partials are addressed through one buffer descriptor with 32-bit
    // byte offsets
    const uint64_t pbytes = S * M * m * sizeof(float);
    if (pbytes >= (1ull << 31))
      return fail(CATENA_ERR_UNSUPPORTED, "decode GEMM partials exceed 2 GiB (%llu k groups)",
                  (unsigned long long)S);
    if (scratch) {
      // caller-provided scratch (the allocation-free entry point)
      if (pbytes > scratch_bytes)
        return fail(CATENA_ERR_UNSUPPORTED,
                    "decode GEMM partials need %llu B of scratch, more than the %llu B available",
                    (unsigned long long)pbytes, (unsigned long long)scratch_bytes);
      P = static_cast<float*>(scratch);
    } else {
      void* ws = nullptr;
      st = workspace(d.ws_decode, pbytes, &ws);
      if (st) return st;
      P = static_cast<float*>(ws);
    }
  }
  const uint16_t* X = a;
  const uint16_t* W = b;
  void* Y = c;
  uint64_t N = m, K = k;
  uint32_t* tickets = d.gemm_tickets();
  uint32_t stream_lds = regs_path ? 0u : 1u;
  const size_t lds = stream_lds ? 4 * 4 * 9216 : 4 * 8 * 64 * 16 + 16 * 132 * 4;
  void* args[] = {&X, &W, &Y, &P, &tickets, (void*)&M, &N, &K, (void*)&kw, &stream_lds, &e};
  if (lds > d.max_lds) return fail(CATENA_ERR_UNSUPPORTED, "decode GEMM needs %zu B of LDS", lds);
  if (S > 1 && (epi == DecodeEpilogue::StoreF32 || epi == DecodeEpilogue::StoreBf16)) {
    // plain output: the partials kernel (W streamed non-temporally, as the
    // plain-output kernels do), then the reduction as a launch of its own
    // (the same adds in the same order, ordered by the launch boundary
    // instead of a completion ticket)
    st = launch(KernelId::GemmBf16DecodePartsNt, dim3((unsigned)gx, (unsigned)S), dim3(256), lds, args);
    if (st) return st;
    return reduce_parts(P, S, (uint64_t)M * m, Y, epi == DecodeEpilogue::StoreBf16);
  }
  return launch(id, dim3((unsigned)gx, (unsigned)S), dim3(256), lds, args);
}

int argmax_compose(const uint32_t* sums, uint32_t n, uint32_t blocks, uint64_t cols, uint32_t* idx) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0) return CATENA_OK;
  if (!sums || !idx || n > 16 || blocks == 0 || cols == 0 || cols >= 0x7FFFFFFFull ||
      (uint64_t)n * blocks * 16 >= (1ull << 31))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "argmax composition operands");
  void* args[] = {&sums, &n, &blocks, &cols, &idx};
  return launch(KernelId::ArgmaxCompose, dim3(1), dim3(256), 0, args);
}

int gemm_bf16_decode_parts(const uint16_t* a, const uint16_t* b, float* parts, uint64_t parts_bytes,
                           uint64_t n, uint64_t m, uint64_t k, uint32_t* k_groups,
                           const DecodeEpiArgs& gather) {
  if (!parts || !k_groups) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  uint32_t S = 0;
  decode_partials_bytes(n, m, k, &S);
  *k_groups = S > 0 ? S : 1;
  if ((uint64_t)*k_groups * n * m * sizeof(float) > parts_bytes)
    return fail(CATENA_ERR_UNSUPPORTED, "decode GEMM partials need %llu B",
                (unsigned long long)((uint64_t)*k_groups * n * m * sizeof(float)));
  // S > 1: the partials go to P = parts; S = 1: the product goes to Y = parts
  // (gather: only its X-row fields are read)
  DecodeEpiArgs e;
  e.x_rows = gather.x_rows;
  e.x_rows_limit = gather.x_rows_limit;
  e.x_sums = gather.x_sums;
  e.x_sums_blocks = gather.x_sums_blocks;
  e.x_sums_cols = gather.x_sums_cols;
  e.x_rows_out = gather.x_rows_out;
  return gemm_bf16_decode(a, b, parts, n, m, k, DecodeEpilogue::Partials, e, parts, parts_bytes);
}

bool attn_few_fits(uint32_t batch, uint32_t tq, uint32_t heads, uint32_t max_len) {
  const uint64_t nq = (uint64_t)batch * tq * heads;
  return nq > 0 && nq <= kAttnFewMaxQueries && tq < 8 && max_len >= 64 &&
         attn_few_lds_bytes(max_len) <= device().max_lds;
}

int attn_few_launch(const uint16_t* q, const uint16_t* k, const uint16_t* v, const uint32_t* lens,
                    void* o, uint32_t batch, uint32_t tq, uint32_t heads, uint32_t max_len,
                    float scale, bool out_f32, const FewQkvArgs& qkv) {
  const uint64_t nq = (uint64_t)batch * tq * heads;
  if (!attn_few_fits(batch, tq, heads, max_len)) return -1;
  if (qkv.parts && (tq != 1 || qkv.n_parts == 0 || !qkv.rope_tab || !qkv.q_out || !qkv.k_cache ||
                    !qkv.v_cache || qkv.part_stride < (uint64_t)batch * 3 * heads * 128))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "attention q/k/v partials operands");
  FewQkvArgs a = qkv;
  void* args[] = {&q, &k, &v, &lens, &o, &heads, &max_len, &tq, &scale, &a};
  // up to 128 pairs: two workgroups per pair (each makes all the scores and
  // adds one half of the output columns), so that 2 x pairs CUs stream K
  // and V instead of one per pair
  if (nq <= kAttnFewSplitMaxQueries)
    return launch(out_f32 ? KernelId::AttnFewSplitD128F32 : KernelId::AttnFewSplitD128Bf16,
                  dim3((unsigned)(2 * nq)), dim3(448), attn_few_split_lds_bytes(max_len), args);
  return launch(out_f32 ? KernelId::AttnFewD128F32 : KernelId::AttnFewD128Bf16, dim3((unsigned)nq),
                dim3(512), attn_few_lds_bytes(max_len), args);
}

bool gemm_bf16_silu_fits(uint64_t n, uint64_t m, uint64_t k, const void* a, const void* b,
                         const void* act) {
  return n % 256 == 0 && m % 128 == 0 && k % 128 == 0 && k > 0 && k <= (1ull << 22) &&
         m <= (1ull << 24) && aligned16(a) && aligned16(b) && aligned16(act) &&
         (n / 256) * (m / 128) <= 0x7FFFFFFFull;
}

bool gemm_bf16_rope_fits(uint64_t rows, uint64_t k, uint32_t tq, uint32_t heads, const void* a,
                         const void* w, const void* q_out, const void* kc, const void* vc,
                         const void* tab) {
  const uint64_t m = 3ull * heads * 128;
  return tq > 0 && heads > 0 && rows % 256 == 0 && rows % tq == 0 && k % 128 == 0 && k > 0 &&
         k <= (1ull << 22) && m <= (1ull << 24) && aligned16(a) && aligned16(w) && aligned16(q_out) &&
         aligned16(kc) && aligned16(vc) && aligned16(tab) && (rows / 256) * (m / 128) <= 0x7FFFFFFFull;
}

bool gemm_bf16_ksplit_fits(uint64_t n, uint64_t m, uint64_t k, uint32_t splits, const void* a,
                           const void* b, const void* parts) {
  return splits > 0 && splits <= 64 && n % 256 == 0 && m % 256 == 0 && k > 0 &&
         k % (128ull * splits) == 0 && k <= (1ull << 22) && m <= (1ull << 24) && aligned16(a) &&
         aligned16(b) && aligned16(parts) && (n / 256) * (m / 256) <= 0x7FFFFFFFull;
}

int gemm_bf16_f32_ksplit(const uint16_t* a, const uint16_t* b, float* parts, uint64_t n, uint64_t m,
                         uint64_t k, uint32_t splits) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0 || m == 0) return CATENA_OK;
  if (!a || !b || !parts) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (!gemm_bf16_ksplit_fits(n, m, k, splits, a, b, parts))
    return fail(CATENA_ERR_UNSUPPORTED, "k-split GEMM: shape or alignment not taken");
  const size_t lds = 4ull * (256 + 256) * 32 * sizeof(uint16_t);
  if (lds > device().max_lds) return fail(CATENA_ERR_UNSUPPORTED, "device LDS %zu < %zu", device().max_lds, lds);
  uint64_t k_len = k / splits;
  void* args[] = {&a, &b, &parts, &n, &m, &k, &k_len};
  return launch(KernelId::GemmBf16K32F32Parts, dim3((unsigned)((n / 256) * (m / 256)), splits), dim3(512), lds,
                args);
}

int gemm_bf16_rope_qkv(const uint16_t* a, const uint16_t* w, const float* tab, const uint32_t* lens,
                       uint16_t* q_out, uint16_t* kc, uint16_t* vc, uint64_t rows, uint64_t k,
                       uint32_t tq, uint32_t heads, uint32_t max_len) {
  int st = ensure_init();
  if (st) return st;
  if (rows == 0) return CATENA_OK;
  if (!a || !w || !tab || !lens || !q_out || !kc || !vc)
    return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (!gemm_bf16_rope_fits(rows, k, tq, heads, a, w, q_out, kc, vc, tab))
    return fail(CATENA_ERR_UNSUPPORTED, "fused q / k / v projection: shape or alignment not taken");
  // the stages (4 x (256 + 128) x 32 bf16) hold the epilogue's staging,
  // 8 waves x 64 rows x 128 bytes
  const size_t lds = 4ull * (256 + 128) * 32 * sizeof(uint16_t);
  if (lds > device().max_lds) return fail(CATENA_ERR_UNSUPPORTED, "device LDS %zu < %zu", device().max_lds, lds);
  uint64_t n = rows, m = 3ull * heads * 128;
  const uint64_t grid = (n / 256) * (m / 128);
  void* args[] = {&a, &w, &n, &m, &k, &tab, &lens, &q_out, &kc, &vc, &tq, &heads, &max_len};
  return launch(KernelId::GemmBf16K32N128Rope, dim3((unsigned)grid), dim3(512), lds, args);
}

// bf16 product of any shape.  Every kernel below adds the same 32-k MFMA
// steps in the same ascending order per output element, so which one runs
// never changes the bits.  Ragged shapes with few tiles are folded as k groups
// whose f32 sums are added in ascending order (gemm_order); may_split = false
// keeps the one order throughout (the decoder).
int gemm_bf16(const uint16_t* a, const uint16_t* b, void* c, uint64_t n, uint64_t m, uint64_t k,
              int out_f32, bool may_split) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0 || m == 0) return CATENA_OK;
  if (!c || (k > 0 && (!a || !b))) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  Device& d = device();

  // decode shape: <= 16 rows of activations against a K x N weight
  if (n <= 16 && k > 0 && m % 8 == 0 && k % 8 == 0 && aligned16(a) && aligned16(b) &&
      aligned16(c))
    return gemm_bf16_decode(a, b, c, n, m, k,
                            out_f32 ? DecodeEpilogue::StoreF32 : DecodeEpilogue::StoreBf16,
                            DecodeEpiArgs{}, nullptr, 0);

  const bool ptr_ok = aligned16(a) && aligned16(b) && aligned16(c);
  const uint64_t tiles = ceil_div(n, 256) * ceil_div(m, 256);
  if (ceil_div(n, 256) * ceil_div(m, 128) > 0x7FFFFFFFu)
    return fail(CATENA_ERR_UNSUPPORTED, "matrix too large");
  // Aligned shapes: direct-to-LDS kernels (8 waves): the four-stage 32-k
  // kernel on 256 x 256 tiles, or on 256 x 128 tiles when N % 256 == 128 or
  // when that takes fewer rounds of the chip; the two-stage 64-k kernel when
  // K % 128 != 0.
  if (ptr_ok && tile_kernels(n, m, k)) {
    void* args[] = {&a, &b, &c, &n, &m, &k};
    KernelId id;
    size_t lds;
    uint64_t grid;
    if (k32_stages(m, k) && (m % 256 != 0 || prefer_n128(n, m, d.cu_count))) {
      id = out_f32 ? KernelId::GemmBf16K32N128F32 : KernelId::GemmBf16K32N128Bf16;
      lds = 4ull * (256 + 128) * 32 * sizeof(uint16_t);  // 98304 B
      grid = (n / 256) * (m / 128);
    } else if (k32_stages(m, k)) {
      id = out_f32 ? KernelId::GemmBf16K32F32 : KernelId::GemmBf16K32Bf16;
      lds = 4ull * (256 + 256) * 32 * sizeof(uint16_t);  // 131072 B
      grid = tiles;
    } else {
      id = out_f32 ? KernelId::GemmBf16LdsF32 : KernelId::GemmBf16LdsBf16;
      lds = 2ull * (256 * 64 + 64 * 256) * sizeof(uint16_t);  // 131072 B
      grid = tiles;
    }
    if (lds > d.max_lds) return fail(CATENA_ERR_UNSUPPORTED, "device LDS %zu < %zu", d.max_lds, lds);
    return launch(id, dim3((unsigned)grid), dim3(512), lds, args);
  }

  // General shapes.  An operand whose rows do not all start on 16 bytes is
  // packed into the library's scratch first (A's rows to whole 32-k slabs);
  // partials of k groups go there too.  Where there is no scratch -- the
  // stream is being captured (a graph would keep the address, and growing the
  // block is not allowed), the product would need too much, or the device has
  // none left -- the groups are folded in sequence, and a product that needs
  // packing runs on the bounds-checked kernel of gemm_bf16.hip, which also
  // takes strides past the 32-bit offsets here.  None of that changes the bits.
  const bool pack_a = k > 0 && (k % 8 != 0 || !aligned16(a));
  const bool pack_b = k > 0 && (m % 8 != 0 || !aligned16(b));
  const GemmPlan order = gemm_order(n, m, k, may_split);
  uint64_t k_len = order.splits > 1 ? gemm_k_len(k, order.splits, kGemmTiles[order.tile].stage_k) : k;
  if (strides_fit(m, k)) {
    const uint64_t lda = pack_a ? ceil_div(k, 32) * 32 : k, ldb = pack_b ? ceil_div(m, 8) * 8 : m;
    const uint64_t a_bytes = pack_a ? ceil_div(n * lda * 2, 256) * 256 : 0;
    const uint64_t b_bytes = pack_b ? ceil_div(k * ldb * 2, 256) * 256 : 0;
    const uint64_t part_bytes = order.splits > 1 ? order.splits * n * m * 4 : 0;
    std::unique_lock<std::mutex> ws_guard(d.ws_mu, std::defer_lock);
    char* ws = nullptr;
    bool with_parts = part_bytes > 0;
    if (a_bytes + b_bytes + part_bytes > 0) {
      hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
      const bool live = hipStreamIsCapturing(d.stream, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone;
      ws_guard.lock();  // the block stays ours until everything is launched
      // with the partials, or the packed operands alone
      for (const uint64_t need : {a_bytes + b_bytes + part_bytes, a_bytes + b_bytes}) {
        if (live && need > 0 && need <= kGemmScratchMax) {
          void* w = nullptr;
          if (workspace(d.ws_general, need, &w) == CATENA_OK) {
            ws = static_cast<char*>(w);
            break;
          }
          clear_error();  // no scratch is no failure
        }
        with_parts = false;
      }
    }
    if (ws || !(pack_a || pack_b)) {
      const uint16_t *pa = a, *pb = b;
      if (pack_a) {
        st = pack_rows(a, n, k, reinterpret_cast<uint16_t*>(ws), lda);
        if (st) return st;
        pa = reinterpret_cast<uint16_t*>(ws);
      }
      if (pack_b) {
        st = pack_rows(b, k, m, reinterpret_cast<uint16_t*>(ws + a_bytes), ldb);
        if (st) return st;
        pb = reinterpret_cast<uint16_t*>(ws + a_bytes);
      }
      const bool seq = order.splits > 1 && !with_parts;
      int tile = order.tile;
      if (seq)
        tile = gemm_cost(kGemmTiles[kTileSeq32], n, m, k, 1) < gemm_cost(kGemmTiles[kTileSeq64], n, m, k, 1) ? kTileSeq32
                                                                                                           : kTileSeq64;
      const GemmTile& t = kGemmTiles[tile];
      const size_t lds = (size_t)t.stages * t.stage_k * (t.bm + t.bn) * sizeof(uint16_t);
      if (lds > d.max_lds) return fail(CATENA_ERR_UNSUPPORTED, "device LDS %zu < %zu", d.max_lds, lds);
      const dim3 grid((unsigned)(ceil_div(n, t.bm) * ceil_div(m, t.bn)), with_parts ? order.splits : 1);
      float* parts = with_parts ? reinterpret_cast<float*>(ws + a_bytes + b_bytes) : nullptr;
      void* out = parts ? parts : c;
      const bool store_f32 = out_f32 || parts;
      KernelId id = store_f32 ? t.f32 : t.bf16;
      if (seq && tile == kTileSeq64) id = out_f32 ? KernelId::GemmBf16Any64x64SeqF32 : KernelId::GemmBf16Any64x64SeqBf16;
      if (seq && tile == kTileSeq32) id = out_f32 ? KernelId::GemmBf16Any32x32SeqF32 : KernelId::GemmBf16Any32x32SeqBf16;
      // four columns to a store of the general kernels, eight bf16 ones to one of the 256 x 256 kernel's
      uint32_t vec = (parts || aligned16(c)) && m % (tile == kTileRagged256 && !store_f32 ? 8 : 4) == 0;
      uint64_t sa = lda, sb = ldb;
      void* any_args[] = {&pa, &pb, &out, &n, &m, &k, &sa, &sb, &k_len, &vec};
      void* edge_args[] = {&pa, &pb, &out, &n, &m, &k, &sa, &sb, &vec};
      st = launch(id, grid, dim3(64 * t.waves), lds, tile == kTileRagged256 ? edge_args : any_args);
      if (st || !parts) return st;
      return reduce_parts(parts, order.splits, n * m, c, !out_f32);
    }
  }
  if (order.splits > 1) {
    void* args[] = {&a, &b, &c, &n, &m, &k, &k_len};
    const size_t lds = 2ull * (256 + 128) * 72 * sizeof(uint16_t);  // 110592 B
    if (lds > d.max_lds) return fail(CATENA_ERR_UNSUPPORTED, "device LDS %zu < %zu", d.max_lds, lds);
    return launch(out_f32 ? KernelId::GemmBf16EdgeGroupsF32 : KernelId::GemmBf16EdgeGroupsBf16,
                  dim3((unsigned)(ceil_div(n, 256) * ceil_div(m, 128))), dim3(256), lds, args);
  }
  void* args[] = {&a, &b, &c, &n, &m, &k};
  const size_t lds = 2ull * 2 * 256 * 72 * sizeof(uint16_t);  // 147456 B
  if (lds > d.max_lds) return fail(CATENA_ERR_UNSUPPORTED, "device LDS %zu < %zu", d.max_lds, lds);
  return launch(out_f32 ? KernelId::GemmBf16EdgeF32 : KernelId::GemmBf16EdgeBf16,
                dim3((unsigned)tiles), dim3(256), lds, args);
}

}  // namespace catena

extern "C" {

int catena_mi355x_gemm_f32_exact(const float* a, const float* b, float* c, uint64_t n, uint64_t m,
                                 uint64_t k) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0 || m == 0) return CATENA_OK;
  if (!c || (k > 0 && (!a || !b))) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  void* args[] = {&a, &b, &c, &n, &m, &k};
  // Every cell is the same k-ascending chain in every form, so the choice
  // never changes the bits.
  const uint64_t gx = ceil_div(m, 64), gy = ceil_div(n, 64), t64 = gx * gy, S = kDecodeSpread;
  if (t64 >= S && (gx > 0x7FFFFFFFu || gy > 65535u)) return fail(CATENA_ERR_UNSUPPORTED, "matrix too large");
  const uint64_t t16 = ceil_div(m, 16) * ceil_div(n, 16);
  const bool words = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 3u) == 0;
  // 16 columns or fewer: a 16 x 16 tile idles none of a wave's lanes that a form
  // 64 or 128 columns wide does not idle too (65536 x 4 x 64: 7 us by DPP, 12 through
  // LDS, 15 with 4 x 1, 26 with 8 x 2, 16 with 64 x 64 tiles)
  const bool narrow = m <= 16 && k >= 32;
  // One cell per thread on 16 x 16 tiles, A by DPP row broadcast and B through
  // LDS (k % 16 == 0, 16-byte rows of B, 31-bit buffer offsets): up to 6.5 tiles
  // for each CU (1792 x 192 x 1728, 1344 tiles: 54 us against 65 with 2 x 1; 576 x
  // 1088 x 896, 2448: 47 against 42 with 4 x 1).  Else A and B both through LDS up
  // to two tiles for each CU, to three where the operands outgrow an XCD's L2,
  // which the row forms feel first (192 x 960 x 1103, 720 tiles: 36 us against 42
  // with 2 x 1; 192 x 734 x 681, 552 tiles: 24 against 19).
  if ((t16 <= 13 * S / 2 || narrow) && k > 0 && k % 16 == 0 && m % 4 == 0 && aligned16(b) && words &&
      (n + 16) * k * 4 < (1ull << 31) && (k + 256) * m * 4 < (1ull << 31) && ceil_div(n, 16) <= 65535)
    return launch(KernelId::GemmF32ExactQ16, dim3((unsigned)ceil_div(m, 16), (unsigned)ceil_div(n, 16)), dim3(256),
                  256 * 16 * 4, args);
  const bool past_l2 = n + m > (3ull << 20) / 4 / (k > 0 ? k : 1);
  const bool small = t16 <= (past_l2 ? 3 : 2) * S || narrow;
  // The row forms take word-aligned operands within the offsets below.
  const bool reach = words && k < (1ull << 26) && m < (1ull << 25);
  // 64 x 64 tiles through LDS: what the row forms cannot take, from 320 tiles on
  // (operands off by 2 bytes, 1280 x 1280 x 512, 400 tiles: 94 us against 119 on 16 x
  // 16; 1024^3, 256: 228 against 153; 1024 x 1024 x 64: 13 against 15), and where
  // those are slower:
  //   * few k, whose remainder they fold one by one behind its loads (2560 x 2560 x
  //     15: 10.5 us against 13.0 with 8 x 2; x 24, no remainder: 13.4 against 13.5;
  //     1280 x 1280 x 12: 5.3 against 6.3 with 4 x 1; x 16: 5.8 against 4.6), but not
  //     below half a tile of rows (16 x 2^22 x 8: 162 against 117);
  //   * an operand past the 256 MiB cache that the narrow side makes them read again
  //     (131072 x 64 x 1000: 423 us against 610 with 4 x 1; 64 x 2^22 x 64: 968 against
  //     1028), from eight tiles for each CU (20000 x 128 x 8000, 626: 1997 against 1001).
  const bool few_k = (k < 16 && t64 >= 5 * S / 4) || (k < 32 && (k < 24 || k % 8 != 0) && t64 >= 3 * S);
  const bool reread = t64 >= 8 * S && ((m <= 128 && n * k > (64ull << 20)) || (n <= 64 && k * m > (64ull << 20)));
  if (reach ? !small && n > 32 && (few_k || reread) : t64 > 5 * S / 4 || (t64 >= S && k < 128))
    return launch(KernelId::GemmF32ExactT64, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, args);
  if (small || !reach) {
    if (t16 > 0x7FFFFFFFu) return fail(CATENA_ERR_UNSUPPORTED, "matrix too large");
    return launch(KernelId::GemmF32ExactT16, dim3((unsigned)t16), dim3(256), 0, args);
  }
  // Rows and columns per lane: 8 x 2 from 700 workgroups on (2.7 waves per
  // SIMD: 1800 x 1700 x 1500, 798 of them, 233 us against 243 with 4 x 1; 1500^3,
  // 564, 197 against 172) and past 64 columns, where its second ones are not idle
  // (65536 x 64 x 256: 88 us against 49 with 4 x 1), 4 x 1 from 600 on (300 x 2000 x
  // 500, 608: 21.6 us against 26.9 with 2 x 1; 1024 x 512 x 1024, 512: 48 against 42),
  // else 2 x 1.
  const uint64_t g82 = ceil_div(m, 128) * ceil_div(n, 32), g41 = gx * ceil_div(n, 16), g21 = gx * ceil_div(n, 8);
  const KernelId id = g82 >= 700 && m > 64 ? KernelId::GemmF32Exact8x2
                      : g41 >= 600         ? KernelId::GemmF32Exact4x1
                                           : KernelId::GemmF32Exact2x1;
  const uint64_t grid = id == KernelId::GemmF32Exact8x2 ? g82 : id == KernelId::GemmF32Exact4x1 ? g41 : g21;
  if (grid > 0x7FFFFFFFu) return fail(CATENA_ERR_UNSUPPORTED, "matrix too large");
  uint32_t m32 = (uint32_t)m, k32 = (uint32_t)k;
  void* rargs[] = {&a, &b, &c, &n, &m32, &k32};
  return launch(id, dim3((unsigned)grid), dim3(256), 0, rargs);
}

int catena_mi355x_gemm_bf16(const uint16_t* a, const uint16_t* b, void* c, uint64_t n, uint64_t m,
                            uint64_t k, int out_f32) {
  return gemm_bf16(a, b, c, n, m, k, out_f32, true);
}

int catena_mi355x_gemm_bf16_silu(const uint16_t* a, const uint16_t* b, uint16_t* act, uint64_t n,
                                 uint64_t m, uint64_t k) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0 || m == 0) return CATENA_OK;
  if (!act || (k > 0 && (!a || !b))) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (!gemm_bf16_silu_fits(n, m, k, a, b, act))
    return fail(CATENA_ERR_UNSUPPORTED,
                "SwiGLU GEMM needs n %% 256 == 0, m %% 128 == 0, k %% 128 == 0 (k <= 2^22, m <= 2^24) "
                "and 16-byte aligned pointers");
  Device& d = device();
  // the tile width the plain GEMM would take for this shape (same bits)
  const bool narrow = m % 256 != 0 || prefer_n128(n, m, d.cu_count);
  const size_t stages = narrow ? 4ull * (256 + 128) * 32 * sizeof(uint16_t)   // 98304 B
                               : 4ull * (256 + 256) * 32 * sizeof(uint16_t);  // 131072 B
  const size_t slots = 4ull * (narrow ? 64 : 128) * 68 * sizeof(float);        // up-column hand-over
  const size_t lds = stages > slots ? stages : slots;
  if (lds > d.max_lds) return fail(CATENA_ERR_UNSUPPORTED, "device LDS %zu < %zu", d.max_lds, lds);
  const uint64_t grid = narrow ? (n / 256) * (m / 128) : (n / 256) * (m / 256);
  void* args[] = {&a, &b, &act, &n, &m, &k};
  return launch(narrow ? KernelId::GemmBf16K32N128Silu : KernelId::GemmBf16K32Silu, dim3((unsigned)grid),
                dim3(512), lds, args);
}

int catena_mi355x_gemm_bf16_rope_qkv(const uint16_t* a, const uint16_t* w, const float* rope_tab,
                                     const uint32_t* lens, uint16_t* q, uint16_t* k_cache,
                                     uint16_t* v_cache, uint32_t batch, uint32_t tq, uint32_t heads,
                                     uint32_t max_len, uint64_t k) {
  int st = ensure_init();
  if (st) return st;
  const uint64_t rows = (uint64_t)batch * tq;
  if (rows == 0 || heads == 0) return CATENA_OK;
  if (!a || !w || !rope_tab || !lens || !q || !k_cache || !v_cache)
    return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (!gemm_bf16_rope_fits(rows, k, tq, heads, a, w, q, k_cache, v_cache, rope_tab))
    return fail(CATENA_ERR_UNSUPPORTED,
                "fused q / k / v projection needs batch * tq %% 256 == 0, k %% 128 == 0 (k <= 2^22) "
                "and 16-byte aligned pointers");
  return gemm_bf16_rope_qkv(a, w, rope_tab, lens, q, k_cache, v_cache, rows, k, tq, heads, max_len);
}

int catena_mi355x_gemm_bf16_ksplit_f32(const uint16_t* a, const uint16_t* b, float* parts,
                                       uint64_t n, uint64_t m, uint64_t k, uint32_t splits) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0 || m == 0) return CATENA_OK;
  if (!a || !b || !parts) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (!gemm_bf16_ksplit_fits(n, m, k, splits, a, b, parts))
    return fail(CATENA_ERR_UNSUPPORTED,
                "k-split GEMM needs 1 <= splits <= 64, n %% 256 == 0, m %% 256 == 0, "
                "k %% (128 splits) == 0 (k <= 2^22) and 16-byte aligned pointers");
  return gemm_bf16_f32_ksplit(a, b, parts, n, m, k, splits);
}

int catena_mi355x_gemm_bf16_argmax(const uint16_t* a, const uint16_t* b, float* c, uint32_t* idx,
                                   uint64_t n, uint64_t m, uint64_t k) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0 || m == 0) return CATENA_OK;
  if (!a || !b || !c || !idx) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  DecodeEpiArgs e;
  e.idx = idx;
  return gemm_bf16_decode(a, b, c, n, m, k, DecodeEpilogue::Argmax, e);
}

int catena_mi355x_attn_decode_bf16(const uint16_t* q, const uint16_t* k, const uint16_t* v,
                                   const uint32_t* lens, float* o, uint32_t batch, uint32_t heads,
                                   uint32_t max_len, uint32_t head_dim, float scale) {
  int st = ensure_init();
  if (st) return st;
  if (head_dim != 128)
    return fail(CATENA_ERR_UNSUPPORTED, "attention head_dim %u unsupported (only 128)", head_dim);
  const uint64_t bh = (uint64_t)batch * heads;
  if (bh == 0) return CATENA_OK;
  if (!q || !lens || !o || (max_len > 0 && (!k || !v)))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (!aligned16(k) || !aligned16(v))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "K/V caches must be 16-byte aligned");
  if (bh > 0x7FFFFFFFu) return fail(CATENA_ERR_UNSUPPORTED, "too many heads");
  Device& d = device();
  const size_t lds = attn_lds_bytes(max_len);
  if (lds > d.max_lds)
    return fail(CATENA_ERR_UNSUPPORTED, "max_len %u needs %zu B of LDS (device has %zu)", max_len,
                lds, d.max_lds);
  // few (batch, head) pairs: the eight-wave kernel spreads each over a CU
  st = attn_few_launch(q, k, v, lens, o, batch, 1, heads, max_len, scale, true);
  if (st >= 0) return st;
  void* args[] = {&q, &k, &v, &lens, &o, &heads, &max_len, &scale};
  return launch(KernelId::AttnDecodeD128, dim3((unsigned)bh), dim3(256), lds, args);
}

int catena_mi355x_softmax_f32(const float* x, float* y, uint64_t rows, uint64_t n) {
  int st = ensure_init();
  if (st) return st;
  if (rows == 0 || n == 0) return CATENA_OK;
  if (!x || !y) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (n >= 0x7FFFFFFFull) return fail(CATENA_ERR_UNSUPPORTED, "softmax length too large");
  if (rows > 0x7FFFFFFFull) return fail(CATENA_ERR_UNSUPPORTED, "too many rows");
  // Rows that fit LDS: one to a workgroup while the latency of a row is what
  // counts, four once the folds' adds do (a wave's add advances four rows): from
  // six rows a CU, where three such workgroups fit one.  Measured, one against
  // four: 1024 x 2048 11.6 / 12.7 us, 2048 x 2048 21.0 / 18.7, 16384 x 512 36.1 /
  // 24.2, 4096 x 4096 58.9 / 59.4, 8192 x 6000 173 / 302.  Longer rows: one row
  // per workgroup through memory.  So too when LDS holds one or two rows a CU and
  // that takes more than three rounds, since the form through memory folds eight
  // rows a CU at a time (LDS against memory: 768 x 30000 252 / 274 us, 800 331 / 276,
  // 4096 1439 / 950 at 32768; 1536 x 16384 152 / 164, 2048 201 / 178); two rows a CU
  // and more than eight are its streams' time again, and LDS reads x once (8192 x
  // 16384 792 / 870).
  const bool vec = n % 4 == 0 && aligned16(x) && aligned16(y);
  uint32_t n32 = (uint32_t)n, slot = rows4_slot(n);
  void* lds_args[] = {&x, &y, &rows, &n32, &slot};
  if (slot && rows4_per_cu(slot) >= 3 && rows >= 6ull * (unsigned)device().cu_count)
    return launch(vec ? KernelId::SoftmaxRows4Vec : KernelId::SoftmaxRows4, dim3((unsigned)ceil_div(rows, 4)),
                  dim3(256), 4 * (size_t)slot * sizeof(float), lds_args);
  const uint64_t row_lds = ceil_div(n, 4) * 4 * sizeof(float), cus = (unsigned)device().cu_count;
  const uint64_t fit = lds_fit(row_lds + 64);
  if (fit >= 3 || (fit > 0 && rows <= 3 * fit * cus) || (fit == 2 && rows > 8 * cus))
    return launch(vec ? KernelId::SoftmaxRowVec : KernelId::SoftmaxRow, dim3((unsigned)rows), dim3(256),
                  row_lds, lds_args);
  void* args[] = {&x, &y, &n};
  return launch(KernelId::SoftmaxRows, dim3((unsigned)rows), dim3(256), 0, args);
}

int catena_mi355x_exp_approx_f32(const float* x, float* y, uint64_t n) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0) return CATENA_OK;
  if (!x || !y) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  const uint64_t g = ceil_div(n, 256);
  if (g > 0x7FFFFFFFull) return fail(CATENA_ERR_UNSUPPORTED, "too many elements");
  void* args[] = {&x, &y, &n};
  return launch(KernelId::ExpApprox, dim3((unsigned)g), dim3(256), 0, args);
}

int catena_mi355x_map_f32(uint32_t op, const float* x, float* y, uint64_t n) {
  if (op > CATENA_MAP_SIN_APPROX_FULL) return fail(CATENA_ERR_INVALID_ARGUMENT, "unknown map op %u", op);
  int st = ensure_init();
  if (st) return st;
  if (n == 0) return CATENA_OK;
  if (!x || !y) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  const uint64_t g = ceil_div(n, 256);
  if (g > 0x7FFFFFFFull) return fail(CATENA_ERR_UNSUPPORTED, "too many elements");
  void* args[] = {&x, &y, &n, &op};
  return launch(KernelId::MapF32, dim3((unsigned)g), dim3(256), 0, args);
}

int catena_mi355x_fill_normal_bf16(uint16_t* out, uint64_t n, uint64_t seed, uint64_t stream,
                                   float scale) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0) return CATENA_OK;
  if (!out) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  const uint64_t g = ceil_div(n, 256);
  if (g > 0x7FFFFFFFull) return fail(CATENA_ERR_UNSUPPORTED, "too many elements");
  void* args[] = {&out, &n, &seed, &stream, &scale};
  return launch(KernelId::FillNormalBf16, dim3((unsigned)g), dim3(256), 0, args);
}

int catena_mi355x_fill_uniform_f32(float* out, uint64_t n, uint64_t seed, uint64_t stream) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0) return CATENA_OK;
  if (!out) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  const uint64_t g = ceil_div(n, 256);
  if (g > 0x7FFFFFFFull) return fail(CATENA_ERR_UNSUPPORTED, "too many elements");
  void* args[] = {&out, &n, &seed, &stream};
  return launch(KernelId::FillUniformF32, dim3((unsigned)g), dim3(256), 0, args);
}

int catena_mi355x_gemm_bf16_decode_plan(uint64_t n, uint64_t m, uint64_t k, uint32_t* k_groups,
                                        uint64_t* partials_bytes) {
  if (!k_groups || !partials_bytes) return fail(CATENA_ERR_INVALID_ARGUMENT, "null output");
  *k_groups = 0;
  *partials_bytes = 0;
  if (n == 0 || n > 16 || m == 0 || k == 0 || m % 8 != 0 || k % 8 != 0)
    return fail(CATENA_ERR_INVALID_ARGUMENT,
                "not a decode-GEMM shape (1 <= n <= 16, m %% 8 == 0, k %% 8 == 0, k > 0)");
  *partials_bytes = decode_partials_bytes(n, m, k, k_groups);
  return CATENA_OK;
}

int catena_mi355x_gemm_bf16_plan(uint64_t n, uint64_t m, uint64_t k, uint32_t* k_groups,
                                 uint64_t* group_k, uint32_t* tile_rows, uint32_t* tile_cols) {
  if (!k_groups || !group_k || !tile_rows || !tile_cols)
    return fail(CATENA_ERR_INVALID_ARGUMENT, "null output");
  *k_groups = 1;
  *group_k = k;
  *tile_rows = *tile_cols = 0;
  if (n == 0 || m == 0 || tile_kernels(n, m, k) || !strides_fit(m, k)) return CATENA_OK;
  const GemmPlan p = gemm_order(n, m, k, true);
  if (p.splits > 1) {
    *k_groups = p.splits;
    *group_k = gemm_k_len(k, p.splits, kGemmTiles[p.tile].stage_k);
  }
  *tile_rows = kGemmTiles[p.tile].bm;
  *tile_cols = kGemmTiles[p.tile].bn;
  return CATENA_OK;
}

int catena_mi355x_copy_bytes(void* dst, const void* src, uint64_t n) {
  int st = ensure_init();
  if (st) return st;
  if (n == 0) return CATENA_OK;
  if (!dst || !src) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (n % 16 != 0 || !aligned16(dst) || !aligned16(src))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "copy needs 16-byte aligned pointers and size");
  uint64_t n16 = n / 16;
  const uint64_t g = ceil_div(n16, 256) < 8192 ? ceil_div(n16, 256) : 8192;
  void* args[] = {&dst, &src, &n16};
  return launch(KernelId::Copy16, dim3((unsigned)g), dim3(256), 0, args);
}

}  // extern "C"
