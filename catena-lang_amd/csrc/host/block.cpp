// Kernel ABI of the decoder-block pieces (block.hip, causal attention) and
// the program ABI of the two stdlib ops they mirror (nn.rmsnorm,
// tensor.argmax-f32).
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

// Four rows of an RMSNorm to a workgroup, or one: once there are more rows than
// one round of one-row workgroups takes, and two of the larger ones fit a CU,
// four while their rounds, each longer than a one-row round, are fewer by more
// than that.  A round of fours takes 1.5 of the others when the row alone is
// read, 1.75 with an index, a table or a second output (extra 1), for which a
// lane has fewer loads in flight, about 2 with a residual (extra 2); rows under
// 1600 values, three or more of whose rounds go into one of fours, always win.
// Measured, one against four, us:
//   rows alone   4096 x 2048 24.2 / 17.3, 4096 x 3584 49 / 42, 6200 x 3584 66 / 76
//   index        4096 x 2048 25.3 / 20.5, 4097 x 2048 25.5 / 27.0, 8192 x 3072 68 / 75
//   residual     4096 x 2048 28.8 / 24.5, 8192 x 2048 45.1 / 46.4, 2049 x 2048 17.3 /
//                18.2, 8192 x 1536 38 / 35, 4096 x 4096 68 / 64, 4097 x 4096 70 / 76
// Rows of n % 4 != 0 go value by value in the four-row form: with anything
// beside them only short ones, of more than 1024 values where that fills half a
// round of fours or all of one (4096 x 1030 20.1 / 17.4, 6200 x 1030 28.0 / 30.6,
// 16384 x 1030 60 / 53, 4097 x 2050 36 / 49).
static bool rms_rows4(uint64_t rows, uint64_t n, uint32_t slot, int extra) {
  const uint64_t cus = (unsigned)device().cu_count;
  const uint64_t round1 = cus * std::min<uint64_t>(8, lds_fit(rmsnorm_lds_bytes(n)));
  const uint64_t round4 = cus * 4 * std::min<uint64_t>(8, rows4_per_cu(slot));
  if (rows <= round1 || rows4_per_cu(slot) < 2) return false;
  if (n % 4 != 0 && extra)
    return n <= 1024 || (n <= 1536 && (rows >= round4 || (2 * rows >= 3 * round1 && 2 * rows <= round4)));
  if (n < 1600) return true;
  const uint64_t c1 = ceil_div(rows, round1), c4 = ceil_div(rows, round4);
  if (extra < 2) return extra == 0 ? 3 * c4 < 2 * c1 : 7 * c4 < 4 * c1;
  return c4 == 1 ? n >= 2500 || 5 * rows >= 3 * round4 : n >= 3500 && 19 * c4 < 10 * c1;
}

int rmsnorm_launch(const float* x, const float* resid, const uint32_t* row_index, float* h_out,
                   float* y_f32, uint16_t* y_bf16, uint64_t rows, uint64_t n,
                   const uint32_t* tokens = nullptr, const uint16_t* table = nullptr,
                   uint32_t vocab = 0, uint32_t resid_parts = 1, uint64_t resid_stride = 0,
                   float* resid_out = nullptr) {
  int st = ensure_init();
  if (st) return st;
  if (rows == 0 || n == 0) return CATENA_OK;
  // input rows: x, or the embedding gather (tokens into table), or the
  // table's own rows (neither x nor tokens)
  if ((!x && !table) || (!y_f32 && !y_bf16)) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if ((tokens || !x) && (!table || (n % 4 == 0 && (reinterpret_cast<uintptr_t>(table) & 7u))))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "embedding table missing or misaligned");
  if (rows > 0x7FFFFFFFull || n > 0xFFFFFFFFull)
    return fail(CATENA_ERR_UNSUPPORTED, "rmsnorm shape too large");
  if (n % 4 == 0) {
    const void* ptrs[] = {x, resid, h_out, y_f32, resid_out};
    for (const void* p : ptrs)
      if (p && !aligned16(p))
        return fail(CATENA_ERR_INVALID_ARGUMENT, "rmsnorm rows must be 16-byte aligned");
    if (y_bf16 && (reinterpret_cast<uintptr_t>(y_bf16) & 7u))
      return fail(CATENA_ERR_INVALID_ARGUMENT, "rmsnorm bf16 output must be 8-byte aligned");
  }
  const uint64_t n_pad = (n + 3) & ~3ull;
  const size_t lds = 2 * n_pad * sizeof(float);  // dynamic part
  if (rmsnorm_lds_bytes(n) > device().max_lds)
    return fail(CATENA_ERR_UNSUPPORTED, "rmsnorm row of %llu needs %zu B of LDS",
                (unsigned long long)n, rmsnorm_lds_bytes(n));
  if (resid_parts == 0 || (resid_parts > 1 && (!resid || (n % 4 == 0 && resid_stride % 4 != 0))))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "rmsnorm residual partials");
  uint32_t n32 = (uint32_t)n, rows32 = (uint32_t)rows;
  // Four rows to a workgroup (their folds then cost the VALU a quarter)?
  uint32_t slot = rows4_slot(n);
  if (slot && !rms_rows4(rows, n, slot, resid ? 2 : h_out || row_index || !x ? 1 : 0)) slot = 0;
  void* args[] = {&x,     &resid, &row_index,   &h_out,        &y_f32,     &y_bf16, &n32, &tokens,
                  &table, &vocab, &resid_parts, &resid_stride, &resid_out, &rows32, &slot};
  if (slot)
    return launch(KernelId::RmsnormRows4, dim3((unsigned)ceil_div(rows, 4)), dim3(256),
                  4 * (size_t)slot * sizeof(float), args);
  return launch(KernelId::RmsnormRows, dim3((unsigned)rows), dim3(256), lds, args);
}
}  // namespace

namespace catena {
int embed_rmsnorm_bf16(const uint32_t* tokens, const uint16_t* table, uint32_t vocab,
                       float* x_out, uint16_t* y, uint64_t rows, uint64_t n) {
  if (!tokens || !y) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  return rmsnorm_launch(nullptr, nullptr, nullptr, x_out, nullptr, y, rows, n, tokens, table, vocab);
}

int embed_residual_rmsnorm_bf16(const uint32_t* tokens, const uint16_t* table, uint32_t vocab,
                                const float* resid, float* h_out, uint16_t* y, uint64_t rows,
                                uint64_t n, uint32_t resid_parts, float* resid_out) {
  if (!tokens || !resid || !y) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  return rmsnorm_launch(nullptr, resid, nullptr, h_out, nullptr, y, rows, n, tokens, table, vocab,
                        resid_parts, rows * n, resid_out);
}

int residual_parts_rmsnorm_bf16(const float* x, const float* resid, uint32_t resid_parts,
                                float* resid_out, const uint32_t* row_index, float* h_out,
                                uint16_t* y, uint64_t rows, uint64_t resid_rows, uint64_t n) {
  if (!x || !resid || !y) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  return rmsnorm_launch(x, resid, row_index, h_out, nullptr, y, rows, n, nullptr, nullptr, 0,
                        resid_parts, resid_rows * n, resid_out);
}

int embed_norm_table_bf16(const uint16_t* table, uint32_t vocab, uint16_t* y, uint64_t n) {
  if (!table || !y) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  // bf16 rows in LDS while at least four of the kernel's waves fit a CU (n up to
  // 5120); below that, or off 16 bytes, the general form
  int st = ensure_init();
  if (st) return st;
  const uint64_t lds = ceil_div(n, 512) * 4096;
  if (n > 0 && n % 8 == 0 && aligned16(table) && aligned16(y) && lds * 4 <= device().max_lds) {
    uint32_t n32 = (uint32_t)n;
    void* args[] = {&table, &y, &vocab, &n32};
    return launch(KernelId::EmbedNormTable, dim3((unsigned)(((uint64_t)vocab + 4) / 4)), dim3(64), lds, args);
  }
  return rmsnorm_launch(nullptr, nullptr, nullptr, nullptr, nullptr, y, (uint64_t)vocab + 1, n, nullptr,
                        table, vocab);
}

int rope_table_f32(const float* inv_freq, float* tab, uint32_t positions, uint32_t half) {
  int st = ensure_init();
  if (st) return st;
  if (!inv_freq || !tab) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (positions == 0 || half == 0) return CATENA_OK;
  if (positions > 65535) return fail(CATENA_ERR_UNSUPPORTED, "rope table of %u positions", positions);
  void* args[] = {&inv_freq, &tab, &positions, &half};
  return launch(KernelId::RopeTable, dim3((unsigned)ceil_div(half, 256), positions), dim3(256), 0, args);
}
}  // namespace catena

extern "C" {

int catena_mi355x_attn_causal_bf16(const uint16_t* q, const uint16_t* k, const uint16_t* v,
                                   const uint32_t* lens, void* o, uint32_t batch, uint32_t tq,
                                   uint32_t heads, uint32_t max_len, uint32_t head_dim,
                                   float scale, int out_f32) {
  return catena::attn_causal(q, k, v, lens, o, batch, tq, heads, max_len, max_len, head_dim, scale,
                             out_f32);
}
}  // extern "C"

namespace catena {
int attn_causal(const uint16_t* q, const uint16_t* k, const uint16_t* v, const uint32_t* lens,
                void* o, uint32_t batch, uint32_t tq, uint32_t heads, uint32_t max_len,
                uint32_t len_bound, uint32_t head_dim, float scale, int out_f32) {
  int st = ensure_init();
  if (st) return st;
  if (head_dim != 128)
    return fail(CATENA_ERR_UNSUPPORTED, "attention head_dim %u unsupported (only 128)", head_dim);
  const uint64_t blocks = (uint64_t)batch * tq * heads;
  if (blocks == 0) return CATENA_OK;
  if (!q || !lens || !o || (max_len > 0 && (!k || !v)))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (!aligned16(k) || !aligned16(v))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "K/V caches must be 16-byte aligned");
  if (blocks > 0x7FFFFFFFu) return fail(CATENA_ERR_UNSUPPORTED, "too many queries");
  // Many queries per sequence: the block-of-16-queries kernels, which read
  // each K / V row once per block and hold a block's scores in LDS, one row
  // per key up to the longest prefix (bounded by len_bound: every lens[b] <=
  // len_bound, and by max_len).  All of them, and the one-query-per-workgroup
  // kernel, give the same bits.
  //   * at most 64 blocks: one query per workgroup, since 16 times as many
  //     workgroups then still find CUs (128 queries x 8 heads over 1028 keys:
  //     56 us against 64 in 64 blocks; 200 queries, 104 blocks: 98 against 67).
  //     Past 1088 rows a CU holds one block, whose time falls less than in half
  //     from 16 queries to 8, and the one-query form's grows with the queries
  //     alone: the two meet at 1984 queries in blocks of 8 and 2560 in blocks of
  //     16 (2048 rows, one query / blocks: 128 pairs x 8 queries 96 / 184 us, x 16
  //     188 / 238, x 20 235 / 237, x 24 275 / 236; 256 pairs x 8 203 / 193).
  //     Both as long as the one-query workgroups, whose LDS holds max_len scores,
  //     take two rounds of the chip at most (a one-layer prompt of 64 tokens x 16
  //     heads in a cache of 32768 rows, one to a CU: 99 us against 91; of 33: 91 /
  //     88; of 16: 88 / 95; of 64 in 8192 rows, three to a CU: 88 / 91);
  //   * four waves while at least three workgroups share a CU (up to 704
  //     rows) and there are more than two for each CU; eight otherwise, which
  //     finish a block sooner and keep a CU busier where two blocks or one
  //     fit (336 blocks of 333 x 400: 30 us against 34; 1408 of 700 x 828: 275
  //     against 300; 2000 of 2000 x 2048: 470 against 583);
  //   * up to 1088 rows two workgroups share a CU, up to 2304 one fits.  When
  //     blocks with at most 1088 rows alone fill the chip's 512 places, they
  //     get a launch with that buffer (500 queries after 500 cached, in 1100:
  //     608 us against 824).
  const uint32_t rows_bound = len_bound < max_len ? len_bound : max_len;
  auto pf_lds = [](uint32_t waves, uint32_t rows) {
    return 16 * 136 * 2 + 3 * 16 * 4 + (size_t)3 * waves * 16 * 4 + (size_t)ceil_div(rows, 64) * 64 * 17 * 4;
  };
  const uint64_t bh = (uint64_t)batch * heads, grid = bh * ceil_div(tq, 16);
  const uint32_t nqb = (uint32_t)ceil_div(tq, 16);
  const bool few = bh * tq <= 2ull * (unsigned)device().cu_count * (device().max_lds / attn_lds_bytes(max_len)) &&
                   (grid <= 64 || (rows_bound > 1088 && bh * tq <= 1408 + 72ull * std::min(tq, 16u)));
  if (tq >= 8 && !few && aligned16(q) && pf_lds(8, rows_bound) <= device().max_lds) {
    if (grid > 0x7FFFFFFFu) return fail(CATENA_ERR_UNSUPPORTED, "too many query blocks");
    // keys the queries before block qb may see: the last of them is followed
    // by tq - 16 qb others
    auto rows_before = [&](uint32_t qb) {
      const uint64_t later = tq - std::min<uint64_t>(tq, 16ull * qb);
      return rows_bound > later ? (uint32_t)(rows_bound - later) : 0u;
    };
    auto blocks_of = [&](uint32_t waves, uint32_t qb0, uint32_t n) {
      const KernelId id = waves == 4 ? (out_f32 ? KernelId::AttnPrefillD128F32 : KernelId::AttnPrefillD128Bf16)
                                     : (out_f32 ? KernelId::AttnPrefillW8D128F32 : KernelId::AttnPrefillW8D128Bf16);
      void* pargs[] = {&q, &k, &v, &lens, &o, &batch, &heads, &max_len, &tq, &scale, &qb0, &n};
      return launch(id, dim3((unsigned)(bh * n)), dim3(64 * waves), pf_lds(waves, rows_before(qb0 + n)), pargs);
    };
    if (rows_bound <= 704 && grid > 512) return blocks_of(4, 0, nqb);
    uint32_t split = 0;  // query blocks below it have at most 1088 rows
    if (rows_bound > 1088) {
      while (split < nqb && rows_before(split + 1) <= 1088) ++split;
      if (split * bh < 512) split = 0;
    }
    st = blocks_of(8, split, nqb - split);
    if (st || split == 0) return st;
    return blocks_of(8, 0, split);
  }
  const size_t lds = attn_lds_bytes(max_len);
  if (lds > device().max_lds)
    return fail(CATENA_ERR_UNSUPPORTED, "max_len %u needs %zu B of LDS (device has %zu)", max_len,
                lds, device().max_lds);
  // few (query, head) pairs: the eight-wave kernel spreads each over a CU
  int split = attn_few_launch(q, k, v, lens, o, batch, tq, heads, max_len, scale, out_f32 != 0);
  if (split >= 0) return split;
  void* args[] = {&q, &k, &v, &lens, &o, &heads, &max_len, &tq, &scale};
  return launch(out_f32 ? KernelId::AttnCausalD128F32 : KernelId::AttnCausalD128Bf16,
                dim3((unsigned)blocks), dim3(256), lds, args);
}
}  // namespace catena

extern "C" {

int catena_mi355x_rmsnorm_f32(const float* x, float* y, uint64_t rows, uint64_t n) {
  if (x && x == y) return fail(CATENA_ERR_INVALID_ARGUMENT, "rmsnorm output may not alias input");
  return rmsnorm_launch(x, nullptr, nullptr, nullptr, y, nullptr, rows, n);
}

int catena_mi355x_residual_rmsnorm_bf16(const float* x, const float* resid,
                                        const uint32_t* row_index, float* h_out, uint16_t* y,
                                        uint64_t rows, uint64_t n) {
  if (!y) return fail(CATENA_ERR_INVALID_ARGUMENT, "null output");
  return rmsnorm_launch(x, resid, row_index, h_out, nullptr, y, rows, n);
}

int catena_mi355x_embed_bf16(const uint32_t* tokens, const uint16_t* table, float* x,
                             uint64_t rows, uint32_t vocab, uint32_t d) {
  int st = ensure_init();
  if (st) return st;
  if (rows == 0 || d == 0) return CATENA_OK;
  if (!tokens || !x || (vocab > 0 && !table)) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (d % 8 != 0 || !aligned16(table) || !aligned16(x))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "embedding needs d %% 8 == 0 and 16-byte aligned rows");
  if (rows > 65535) return fail(CATENA_ERR_UNSUPPORTED, "embedding of more than 65535 rows");
  void* args[] = {&tokens, &table, &x, &vocab, &d};
  return launch(KernelId::EmbedRowsBf16, dim3((unsigned)ceil_div(d, 2048), (unsigned)rows),
                dim3(256), 0, args);
}

int catena_mi355x_rope_inv_freq(float* out_host, uint32_t head_dim, double base) {
  if (!out_host || head_dim == 0 || head_dim % 2 != 0)
    return fail(CATENA_ERR_INVALID_ARGUMENT, "rope needs an even head_dim and an output");
  for (uint32_t i = 0; i < head_dim / 2; ++i)
    out_host[i] = (float)(1.0 / std::pow(base, (2.0 * i) / head_dim));
  return CATENA_OK;
}

int catena_mi355x_rope_table_f32(const float* inv_freq, float* tab, uint32_t positions,
                                 uint32_t head_dim) {
  if (head_dim % 2 != 0) return fail(CATENA_ERR_INVALID_ARGUMENT, "rope needs an even head_dim");
  return rope_table_f32(inv_freq, tab, positions, head_dim / 2);
}

int catena_mi355x_rope_qkv_bf16(const float* qkv, const float* inv_freq, const uint32_t* lens,
                                uint16_t* q, uint16_t* k_cache, uint16_t* v_cache,
                                uint32_t batch, uint32_t tq, uint32_t heads, uint32_t head_dim,
                                uint32_t max_len) {
  int st = ensure_init();
  if (st) return st;
  const uint64_t rows = (uint64_t)batch * tq;
  if (rows == 0 || heads == 0) return CATENA_OK;
  if (head_dim == 0 || head_dim % 2 != 0)
    return fail(CATENA_ERR_INVALID_ARGUMENT, "rope needs an even head_dim");
  if (!qkv || !inv_freq || !lens || !q || !k_cache || !v_cache)
    return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  const uint64_t threads = rows * heads * (head_dim / 2);
  if (rows > 0xFFFFFFFFull || ceil_div(threads, 256) > 0x7FFFFFFFull)
    return fail(CATENA_ERR_UNSUPPORTED, "rope shape too large");
  uint32_t R = (uint32_t)rows;
  void* args[] = {&qkv, &inv_freq, &lens, &q, &k_cache, &v_cache, &R, &tq, &heads, &head_dim,
                  &max_len};
  return launch(KernelId::RopeQkvStore, dim3((unsigned)ceil_div(threads, 256)), dim3(256), 0, args);
}

int catena_mi355x_silu_mul_bf16(const float* gu, uint16_t* out, uint64_t rows, uint32_t ffn,
                                uint32_t group) {
  int st = ensure_init();
  if (st) return st;
  if (rows == 0 || ffn == 0) return CATENA_OK;
  if (!gu || !out) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (ffn % 4 != 0 || !aligned16(gu) || (reinterpret_cast<uintptr_t>(out) & 7u))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "silu_mul needs F %% 4 == 0 and aligned rows");
  if (group != 0 && (group % 4 != 0 || ffn % group != 0))
    return fail(CATENA_ERR_INVALID_ARGUMENT, "silu_mul group must divide F and be a multiple of 4");
  if (rows > 65535) return fail(CATENA_ERR_UNSUPPORTED, "silu_mul of more than 65535 rows");
  void* args[] = {&gu, &out, &ffn, &group};
  return launch(KernelId::SiluMulBf16, dim3((unsigned)ceil_div(ffn, 1024), (unsigned)rows),
                dim3(256), 0, args);
}

int catena_mi355x_argmax_f32(const float* x, uint32_t* idx, uint64_t rows, uint64_t n) {
  int st = ensure_init();
  if (st) return st;
  if (rows == 0) return CATENA_OK;
  if (!idx || (n > 0 && !x)) return fail(CATENA_ERR_INVALID_ARGUMENT, "null operand");
  if (rows > 0x7FFFFFFFull || n >= 0x7FFFFFFFull)
    return fail(CATENA_ERR_UNSUPPORTED, "argmax shape too large");
  if (rows > 65535) return fail(CATENA_ERR_UNSUPPORTED, "argmax of more than 65535 rows");
  // Chunks of 4096 elements per workgroup (fewer, longer ones when the
  // per-row partials would not fit the library's scratch).
  const Device& d = device();
  const uint64_t max_parts = Device::kRowPartialBytes / 12;
  uint64_t chunk = 4096;
  if (rows > Device::kTicketsRows) {
    chunk = n > 0 ? n : 1;  // one workgroup per row: no ticket needed
  } else {
    while (rows * ceil_div(n, chunk) > max_parts) chunk *= 2;
  }
  const uint64_t chunks = n > 0 ? ceil_div(n, chunk) : 1;
  uint32_t n32 = (uint32_t)n, chunk32 = (uint32_t)chunk;
  uint32_t* tickets = d.row_tickets();
  uint32_t* partials = static_cast<uint32_t*>(d.row_partials());
  void* args[] = {&x, &idx, &n32, &chunk32, &tickets, &partials};
  return launch(KernelId::ArgmaxRowsF32, dim3((unsigned)chunks, (unsigned)rows), dim3(256), 0, args);
}

// ---------------------------------------------------------------- programs

void program_nn_rmsnorm(catena_mem_t x, catena_mem_t* out) {
  const uint64_t n = x.len / 4;  // mem.cast.f32
  catena_mem_t y{nullptr, 0};
  if (catena_mem_alloc(n * 4, &y) != CATENA_OK) trap_gpu("output allocation");
  if (n > 0) {
    if (catena_mi355x_rmsnorm_f32(static_cast<const float*>(x.data), static_cast<float*>(y.data), 1,
                                  n) != CATENA_OK)
      trap_gpu("nn.rmsnorm");
    if (catena_mi355x_synchronize() != CATENA_OK) trap_gpu("synchronize");
  }
  *out = y;
}

void program_tensor_argmax_f32(catena_mem_t x, uint64_t* out) {
  const uint64_t n = x.len / 4;
  if (n == 0) trap_assert("u64.assert-nz: argmax of an empty buffer");
  catena_mem_t idx{nullptr, 0};
  if (catena_mem_alloc(4, &idx) != CATENA_OK) trap_gpu("output allocation");
  if (catena_mi355x_argmax_f32(static_cast<const float*>(x.data), static_cast<uint32_t*>(idx.data), 1,
                               n) != CATENA_OK)
    trap_gpu("tensor.argmax-f32");
  uint32_t host = 0;
  if (catena_mem_read(idx, 0, &host, 4) != CATENA_OK) trap_gpu("download");
  catena_mem_free(&idx);
  *out = host;
}

}  // extern "C"
