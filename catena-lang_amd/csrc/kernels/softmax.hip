// nn.softmax, math.exp-approx and the scalar stdlib maps as device kernels.
//
// nn.softmax (catena-lang/stdlib/nn.hex:93-122) over each of `rows` f32
// vectors of length n:
//   max   = f32.max-env fold from -inf          (catena-lang/stdlib/sum.hex:73-84)
//   denom = f32.add-env fold from +0 of exp~(x_i - max)   (nn.hex:59-72)
//   out_i = exp~(x_i - max) / denom                        (nn.hex:75-90)
// The reference runs both folds serially on the host (the entry is host-only
// because it contains a materialize).  Rows that fit LDS: softmax_lds_body below.
// Longer ones: one workgroup per row computes the max with the exact parallel
// form of the fold (FirstMax, common.h), writes exp~ values to the output, folds
// the denominator in ascending order as one lane-to-lane chain in wave 0
// (serial_sum_wave), and divides in place.  Both are bitwise the sequential
// result.
#include "common.h"

namespace {
CATENA_DEV int wave_max_i32(int v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    int o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

CATENA_DEV FirstMax wave_first_max(FirstMax a) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    FirstMax b;
    b.v = __shfl_xor(a.v, off, 64);
    b.i = (uint32_t)__shfl_xor((int)a.i, off, 64);
    a = first_max_combine(a, b);
  }
  return a;
}
}  // namespace

extern "C" __global__ __launch_bounds__(256) void catena_softmax_rows_f32(
    const float* __restrict__ x, float* __restrict__ y, uint64_t n) {
  __shared__ int red_i[4];
  __shared__ float red_v[4];
  __shared__ uint32_t red_u[4];
  __shared__ float den_s;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* xr = x + (uint64_t)blockIdx.x * n;
  float* yr = y + (uint64_t)blockIdx.x * n;

  // index arithmetic of FirstMax is 32-bit; the host rejects n >= 2^32 - 1
  int lastnan = -1;
  for (uint64_t t = tid; t < n; t += 256)
    if (xr[t] != xr[t]) lastnan = (int)t;
  lastnan = wave_max_i32(lastnan);
  if (lane == 0) red_i[wave] = lastnan;
  __syncthreads();
  int J = red_i[0];
  for (int w = 1; w < 4; ++w) J = red_i[w] > J ? red_i[w] : J;

  FirstMax fm{__uint_as_float(0xFF800000u), 0xFFFFFFFFu};
  for (uint64_t t = tid; t < n; t += 256)
    if ((int64_t)t > J) fm = first_max_combine(fm, FirstMax{xr[t], (uint32_t)t});
  fm = wave_first_max(fm);
  if (lane == 0) {
    red_v[wave] = fm.v;
    red_u[wave] = fm.i;
  }
  __syncthreads();
  FirstMax all{red_v[0], red_u[0]};
  for (int w = 1; w < 4; ++w) all = first_max_combine(all, FirstMax{red_v[w], red_u[w]});
  float mx;
  if (n > 0 && J == (int64_t)n - 1)
    mx = xr[n - 1];
  else
    mx = (all.i == 0xFFFFFFFFu) ? __uint_as_float(0xFF800000u) : all.v;
  __syncthreads();  // x[n-1] is read above; y may alias x

  for (uint64_t t = tid; t < n; t += 256) {
    const float shifted = xr[t] - mx;
    yr[t] = exp_approx(shifted);
  }
  __syncthreads();
  if (tid < 64) {
    // den = (((0 + e_0) + e_1) + ...), ascending, as one lane-to-lane chain
    const float den = serial_sum_wave(yr, (uint32_t)n);
    if (tid == 0) den_s = den;
  }
  __syncthreads();
  const float den = den_s;
  for (uint64_t t = tid; t < n; t += 256) yr[t] = yr[t] / den;
}

// The same for rows that fit LDS: a row is read once and written once and kept
// in LDS between, one row to a workgroup, or (ROWS == 4) a wave to a row and
// wave 0 folds the four denominators together (serial_sum_rows4).
// The maximum: when a row holds no NaN, the fold's result is the largest value
// (of zeros the first one, whose sign changes no output: x - 0 is x, and exp~ of
// either zero is the same); a row with a NaN takes the exact parallel form over
// LDS, all of the row's threads together.  VEC: n % 4 == 0 and 16-byte aligned
// rows.
// What bounds the four-row form: at 4096 x 2048 it is one round of workgroups,
// so its phases follow one another: both passes over memory about 13 us, exp~
// and the division (35 and 12 instructions per value) about 7, the chain of adds
// 4.3 us of latency; 50 -> 27 us on one box against the form above, which reads
// x three times and its exp~ values back from memory (16384 x 512 59 -> 24, 1000
// x 8191 80 -> 54).  The one-row form has 256 threads for the row and the same
// chain: 1 x 2048 14.5 -> 7.4 us, 1 x 8192 51 -> 23, 1024 x 2048 17.7 -> 11.6.
namespace {
template <int ROWS, bool VEC>
CATENA_DEV void softmax_lds_body(const float* x, float* y, uint64_t rows, uint32_t n, uint32_t slot) {
  constexpr uint32_t T = 256 / ROWS;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float den_s[ROWS], top_s[4];
  __shared__ int nan_s[4];
  __shared__ uint32_t at_s[4];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, tid = threadIdx.x % T;
  float* s = reinterpret_cast<float*>(smem) + (ROWS == 4 ? wave * slot : 0);
  const uint64_t row = (uint64_t)blockIdx.x * ROWS + (ROWS == 4 ? wave : 0);
  const bool live = ROWS == 1 || row < rows;
  const float* xr = x + row * n;
  const float lowest = __uint_as_float(0xFF800000u);
  float top = lowest;
  bool isnan = false;
  if (live)
    row_to_lds<ROWS, VEC>(xr, s, n, [&](float v) {
      isnan |= v != v;
      top = __builtin_fmaxf(top, v);  // a NaN leaves it
    });
  // the wave's largest value: inclusive scans within rows of 16 lanes, rows
  // joined through row_bcast 15 and 31, lane 63's result for all
#define CATENA_DPP_FMAX(ctrl, lanes)                                                                              \
  top = __builtin_fmaxf(top, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(top), __float_as_int(top), \
                                                                        (ctrl), (lanes), 0xF, false)))
  CATENA_DPP_FMAX(0x111, 0xF);
  CATENA_DPP_FMAX(0x112, 0xF);
  CATENA_DPP_FMAX(0x114, 0xF);
  CATENA_DPP_FMAX(0x118, 0xF);
  CATENA_DPP_FMAX(0x142, 0xA);
  CATENA_DPP_FMAX(0x143, 0xC);
#undef CATENA_DPP_FMAX
  float mx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(top), 63));
  bool anynan = __builtin_amdgcn_ballot_w64(isnan) != 0;
  if (ROWS == 1) {
    if (lane == 0) {
      top_s[wave] = mx;
      nan_s[wave] = anynan;
    }
    __syncthreads();
    mx = __builtin_fmaxf(__builtin_fmaxf(top_s[0], top_s[1]), __builtin_fmaxf(top_s[2], top_s[3]));
    anynan = (nan_s[0] | nan_s[1] | nan_s[2] | nan_s[3]) != 0;
  }
  if (anynan) {  // the same for every thread of the row
    int lastnan = -1;
    for (uint32_t t = tid; t < n; t += T)
      if (s[row_at<ROWS>(t)] != s[row_at<ROWS>(t)]) lastnan = (int)t;
    lastnan = wave_max_i32(lastnan);
    if (ROWS == 1) {
      __syncthreads();  // top_s and nan_s have been read
      if (lane == 0) nan_s[wave] = lastnan;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < 4; ++w) lastnan = nan_s[w] > lastnan ? nan_s[w] : lastnan;
    }
    if (lastnan == (int)n - 1) {
      mx = s[row_at<ROWS>(n - 1)];
    } else {
      FirstMax fm{lowest, 0xFFFFFFFFu};
      for (uint32_t t = lastnan + 1 + tid; t < n; t += T)
        fm = first_max_combine(fm, FirstMax{s[row_at<ROWS>(t)], t});
      fm = wave_first_max(fm);
      if (ROWS == 1) {
        if (lane == 0) {
          top_s[wave] = fm.v;
          at_s[wave] = fm.i;
        }
        __syncthreads();
        fm = FirstMax{top_s[0], at_s[0]};
#pragma unroll
        for (int w = 1; w < 4; ++w) fm = first_max_combine(fm, FirstMax{top_s[w], at_s[w]});
      }
      mx = fm.i == 0xFFFFFFFFu ? lowest : fm.v;
    }
    if (ROWS == 1) __syncthreads();  // every wave has read the row
  }
  if (live) {
    for (uint32_t i = tid; i < (n + 3) / 4; i += T) {
      f32x4_t* p = reinterpret_cast<f32x4_t*>(s + row_at<ROWS>(4 * i));
      f32x4_t q = *p;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float shifted = q[c] - mx;
        const float e = exp_approx(shifted);
        q[c] = VEC || 4 * i + c < n ? e : 0.0f;  // the slots past the row: +0
      }
      *p = q;
    }
  }
  __syncthreads();
  if (wave == 0) {
    const float den = rows_fold<ROWS, false>(reinterpret_cast<float*>(smem), slot, (n + 3u) & ~3u);
    if (lane % (64 / ROWS) == 0) den_s[lane / (64 / ROWS)] = den;
  }
  __syncthreads();
  if (!live) return;
  const SharedDivisor den = shared_divisor(den_s[ROWS == 4 ? wave : 0]);
  float* yr = y + row * n;
  if (VEC) {
    for (uint32_t i = tid; i < n / 4; i += T) {
      const f32x4_t e = *reinterpret_cast<const f32x4_t*>(s + row_at<ROWS>(4 * i));
      float q[4] = {e[0], e[1], e[2], e[3]};
      divide_shared(q, den);
      reinterpret_cast<f32x4_t*>(yr)[i] = f32x4_t{q[0], q[1], q[2], q[3]};
    }
  } else {
    for (uint32_t i = tid; i < n; i += T) {
      float q[1] = {s[row_at<ROWS>(i)]};
      divide_shared(q, den);
      yr[i] = q[0];
    }
  }
}
}  // namespace

#define CATENA_SOFTMAX_LDS(name, ROWS, VEC)                                                                      \
  extern "C" __global__ __launch_bounds__(256) void name(const float* x, float* y, uint64_t rows, uint32_t n,   \
                                                         uint32_t slot) {                                       \
    softmax_lds_body<ROWS, VEC>(x, y, rows, n, slot);                                                            \
  }
// grid = rows, block = 256, dynamic LDS = slot floats (n rounded up to 4)
CATENA_SOFTMAX_LDS(catena_softmax_row_vec_f32, 1, true)
CATENA_SOFTMAX_LDS(catena_softmax_row_f32, 1, false)
// grid = ceil(rows / 4), block = 256, dynamic LDS = 4 slots of `slot` floats
// (slot % 4 == 0, at least pad32 of n rounded up to 4)
CATENA_SOFTMAX_LDS(catena_softmax_rows4_vec_f32, 4, true)
CATENA_SOFTMAX_LDS(catena_softmax_rows4_f32, 4, false)
#undef CATENA_SOFTMAX_LDS

// math.exp-approx applied elementwise (catena-lang/stdlib/math.hex:185-199).
extern "C" __global__ __launch_bounds__(256) void catena_exp_approx_f32(
    const float* __restrict__ x, float* __restrict__ y, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) y[i] = exp_approx(x[i]);
}

// The scalar stdlib programs applied elementwise, one device function each
// (common.h), selected by `op` (catena_map_op_t; uniform across the grid):
//   0 math.exp-approx       catena-lang/stdlib/math.hex:185-199
//   1 math.sqrt             catena-lang/stdlib/math.hex:235-272
//   2 nn.sigmoid            catena-lang/stdlib/nn.hex:1-12
//   3 nn.silu               catena-lang/stdlib/nn.hex:15-21
//   4 math.sin-approx       catena-lang/stdlib/math.hex:1-23
//   5 math.cos-approx       catena-lang/stdlib/math.hex:25-47
//   6 math.sin-approx-full  catena-lang/stdlib/math.hex:49-103
// The host rejects any other op before the launch.
extern "C" __global__ __launch_bounds__(256) void catena_map_f32(
    const float* __restrict__ x, float* __restrict__ y, uint64_t n, uint32_t op) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float v = x[i];
  float r;
  switch (op) {
    case 0: r = exp_approx(v); break;
    case 1: r = sqrt_newton(v); break;
    case 2: r = sigmoid_approx(v); break;
    case 3: r = silu_approx(v); break;
    case 4: r = sin_taylor(v); break;
    case 5: r = cos_taylor(v); break;
    default: r = sin_full(v); break;
  }
  y[i] = r;
}
