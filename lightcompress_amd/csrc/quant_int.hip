// Integer quantizer for gfx950: row-wise min/max -> scale/zero -> quantize ->
// dequantize / integer codes in ONE pass over HBM (skeleton in rowquant.h).
//
// Replaces the ~9 eager torch kernels behind
//   IntegerQuantizer.get_tensor_qparams / quant / dequant / quant_dequant /
//   fake_quant_*_dynamic|static / real_quant_weight_dynamic|static
// (llmc/compression/quantization/quant.py:134-145, 544-558, 689-716, 753-952).
//
// A "row" is one row of the reshaped tensor (quant.py:611-641): a group of
// `group_size` weights (per_group), a whole weight row (per_channel), a token
// (per_token) or a head (per_head).
//
// Arithmetic contract (bit-exact with the reference's torch op sequence):
//   fp32 rows : every step is one IEEE fp32 op (true division, rintf).
//   bf16 rows : every step is computed in fp32 and rounded to bf16 (RNE)
//               before the next step, as torch does for bf16 tensors.
//   fp16 rows : the same with fp16 roundings (the per-row parameters through true divisions).
// The per-element division x/s is evaluated as x*(1/s) with an exactness
// guard: whenever the approximate quotient is close enough to a rounding
// boundary that the IEEE quotient could round differently, the lane falls
// back to the true division.  Both paths give the same bits by construction.
#include "intop.h"

namespace {
using namespace lcq;

template <int BF>
int run(const void* x, int64_t rows, int64_t cols, float qmin, float qmax, int flags, float osf, void* dq,
        void* codes, int code_dtype, void* scales, void* zeros, hipStream_t st) {
  const bool big = (qmax > 256.0f) || (qmin < -256.0f);
  if (big || (flags & LCQ_FLAG_NO_ROUND_ZP))
    return dispatch_rows(x, rows, cols, dq, codes, scales, zeros,
                         make_op<IntOp<BF, false>>(qmin, qmax, flags, osf, code_dtype), true, st);
  // the common storage formats get kernels with the store path fixed at compile time
  #define LCQ_RUN(CDV) return dispatch_rows(x, rows, cols, dq, codes, scales, zeros, \
                         make_op<IntOp<BF, true, false, CDV>>(qmin, qmax, flags, osf, code_dtype), false, st)
  switch (code_dtype) {
    case LCQ_CODE_NONE: LCQ_RUN(LCQ_CODE_NONE);
    case LCQ_CODE_U8: LCQ_RUN(LCQ_CODE_U8);
    case LCQ_CODE_I32: LCQ_RUN(LCQ_CODE_I32);
    case LCQ_CODE_CT4: LCQ_RUN(LCQ_CODE_CT4);
    case LCQ_CODE_CT8: LCQ_RUN(LCQ_CODE_CT8);
    default: LCQ_RUN(-1);
  }
  #undef LCQ_RUN
}

// get_minmax_range (row-wise), quant.py:141-143
template <int BF>
__global__ __launch_bounds__(256) void minmax_rows_kernel(const void* __restrict__ x, int64_t rows, int64_t cols,
                                                          void* __restrict__ mn_out, void* __restrict__ mx_out) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= rows) return;
  float mn = __builtin_inff(), mx = -__builtin_inff();
  for (int64_t j = lane; j < cols; j += 64) {
    const float v = load_scalar<BF>(x, row * cols + j);
    mn = nan_min(mn, v); mx = nan_max(mx, v);
  }
  mn = team_reduce<64, false>(mn);
  mx = team_reduce<64, true>(mx);
  if (lane == 0) { store_scalar<BF>(mn_out, row, mn); store_scalar<BF>(mx_out, row, mx); }
}

// per_tensor range, quant.py:135-137: stage 1 writes one (min,max) per workgroup
template <int BF>
__global__ __launch_bounds__(256) void minmax_all_stage1(const void* __restrict__ x, int64_t n, float* __restrict__ part) {
  __shared__ float sm[8];
  float mn = __builtin_inff(), mx = -__builtin_inff();
  for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < n; j += (int64_t)gridDim.x * 256) {
    const float v = load_scalar<BF>(x, j);
    mn = nan_min(mn, v); mx = nan_max(mx, v);
  }
  mn = block_reduce<false>(mn, sm);
  mx = block_reduce<true>(mx, sm);
  if (threadIdx.x == 0) { part[2 * blockIdx.x] = mn; part[2 * blockIdx.x + 1] = mx; }
}
template <int BF>
__global__ __launch_bounds__(256) void minmax_all_stage2(const float* __restrict__ part, int nparts,
                                                         void* __restrict__ mn_out, void* __restrict__ mx_out) {
  __shared__ float sm[8];
  float mn = __builtin_inff(), mx = -__builtin_inff();
  for (int j = threadIdx.x; j < nparts; j += 256) { mn = nan_min(mn, part[2 * j]); mx = nan_max(mx, part[2 * j + 1]); }
  mn = block_reduce<false>(mn, sm);
  mx = block_reduce<true>(mx, sm);
  if (threadIdx.x == 0) { store_scalar<BF>(mn_out, 0, mn); store_scalar<BF>(mx_out, 0, mx); }
}

// get_qparams on explicit ranges, quant.py:544-558
template <int BF>
__global__ void qparams_kernel(const void* __restrict__ mn, const void* __restrict__ mx, int64_t n,
                               void* __restrict__ scales, void* __restrict__ zeros, IntOp<BF, false> op) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const IntRow p = op.make(load_scalar<BF>(mn, i), load_scalar<BF>(mx, i));
  op.store_qp(scales, zeros, i, p);
}

// 16-bit rows with fp32 parameters per row (calibrated ranges are fp32, quant.py:147-205): torch promotes every operation
// to fp32 and the caller casts the result back, so this reads 16-bit chunks, computes as fp32 rows do and rounds once.
// HBM-bound; the rows are not reduced over, so chunks are independent (row = chunk / chunks per row).
template <int BF>
__global__ __launch_bounds__(256) void static_promoted_kernel(const u32x4* __restrict__ x, int64_t nchunks, int cpr,
                                                              const void* __restrict__ scales, const void* __restrict__ zeros,
                                                              void* __restrict__ dq, void* __restrict__ codes, IntOp<0, true> op) {
  for (int64_t ch = (int64_t)blockIdx.x * 256 + threadIdx.x; ch < nchunks; ch += (int64_t)gridDim.x * 256) {
    const u32x4 raw = __builtin_nontemporal_load(x + ch);
    const IntRow p = op.load(scales, zeros, op.scalar_qp ? 0 : (int64_t)((uint64_t)ch / (uint32_t)cpr));
    float v[8], q[8];
    unpack<BF>(raw, v);
    if (!codes) {
      op.template fused_dq<4>(v, q, p);
      op.template fused_dq<4>(v + 4, q + 4, p);
      __builtin_nontemporal_store(pack_rne<BF>(q), (u32x4*)dq + ch);
      continue;
    }
    op.template codes<4>(v, q, p);
    op.template codes<4>(v + 4, q + 4, p);
    store_codes(op, codes, ch * 8, q);
    store_codes(op, codes, ch * 8 + 4, q + 4);
    if (dq) {
      #pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = op.deq_raw(q[i], p);
      __builtin_nontemporal_store(pack_rne<BF>(v), (u32x4*)dq + ch);
    }
  }
}

// dequant, quant.py:709-711, on stored float codes
template <int BF>
__global__ __launch_bounds__(256) void dequant_kernel(const void* __restrict__ q, int64_t rows, int64_t cols,
                                                      const void* __restrict__ scales, const void* __restrict__ zeros,
                                                      void* __restrict__ out, int scalar_qp, int scale_f32, float osf) {
  const int64_t n = rows * cols;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
    const int64_t row = scalar_qp ? 0 : e / cols;
    // fp32 parameters (0-dim next to a 16-bit tensor) are rounded to the row type where they meet the rows
    const float s = scale_f32 ? ((const float*)scales)[row] : load_scalar<BF>(scales, row);
    const float z = !zeros ? 0.0f : (scale_f32 ? rnd<BF>(((const float*)zeros)[row]) : load_scalar<BF>(zeros, row));
    const float d = rnd<BF>(load_scalar<BF>(q, e) - z);
    store_scalar<BF>(out, e, rnd<BF>(d * rnd<BF>(s * osf)));
  }
}

// get_mse_range, quant.py:147-205: per row, shrink steps i = 0 .. steps-1 with p = 1 - i / grid:
//   xmin = p * cur_min, xmax = p * cur_max;  err = sum_j |quant_dequant(x_j; xmin, xmax) - x_j| ^ norm
//   err < best  ->  best = err, cur_min = xmin, cur_max = xmax
// cur_min / cur_max start as the row's min / max and - as in the reference, whose best_min_val / best_max_val
// alias the range tensors - are the values the NEXT step shrinks.  All arithmetic in fp32 (tensor.float()).

// err of one row, a wave per row: IEEE quotients and powf, lane l adds columns l, l + 64, ... in order.  This sum defines
// which step wins; every path below takes the decisions it takes.
template <int BF>
__device__ __forceinline__ float mse_row_error(const void* __restrict__ x, int64_t row, int64_t cols, const IntRow& prm, float norm,
                                               const IntOp<0, false>& op, int lane) {
  float err = 0.0f;
  #pragma unroll 1
  for (int64_t j = lane; j < cols; j += 64) {
    const float v = load_scalar<BF>(x, row * cols + j);
    const float d = fabsf(op.deq(op.code(v, prm), prm) - v);
    err += __builtin_powf(d, norm);
  }
  return team_sum<64>(err);
}

// One wave per row; the row is re-read from L1/L2 on every step.
template <int BF>
__global__ __launch_bounds__(256) void mse_range_kernel(const void* __restrict__ x, int64_t rows, int64_t cols, int steps,
                                                        int grid_n, float norm, IntOp<0, false> op,
                                                        float* __restrict__ mn_out, float* __restrict__ mx_out) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  float mn = __builtin_inff(), mx = -__builtin_inff();
  for (int64_t j = lane; j < cols; j += 64) {
    const float v = load_scalar<BF>(x, row * cols + j);
    mn = nan_min(mn, v); mx = nan_max(mx, v);
  }
  float cur_min = team_reduce<64, false>(mn), cur_max = team_reduce<64, true>(mx);
  float best = __builtin_inff();
  for (int i = 0; i < steps; ++i) {
    const float p = (float)(1.0 - (double)i / (double)grid_n);
    const float xmin = p * cur_min, xmax = p * cur_max;
    const float err = mse_row_error<BF>(x, row, cols, op.make(xmin, xmax), norm, op, lane);
    if (err < best) { best = err; cur_min = xmin; cur_max = xmax; }
  }
  if (lane == 0) { mn_out[row] = cur_min; mx_out[row] = cur_max; }
}

// The same search with the row in registers, for rounded zero points: TEAM lanes (256: a workgroup) share a row, PER
// elements each.  A step's error is first estimated:
//   * t = x * (1/s) instead of x / s: a quotient within 2 ulp of a half-integer may round to the other neighbour, both
//     of which are half a step away from x;
//   * |d| ^ norm = 2 ^ (norm log2 |d|) through v_log / v_exp; x and s are scaled by the power of two that brings the row's
//     largest value to [1, 2), so |log2| stays small and nothing underflows.  The factor is common to all steps of a row and
//     positive, so it changes no comparison;
//   * every term is >= 0 and fp32 sums of such terms never shrink, so a part of the estimate that is far enough above the
//     best one decides a step: first the error of the two extremes alone (most steps behind the best one lose by what they
//     clip there), then after every quarter of the elements.  A wave goes on to the next step when all its rows are decided;
//   * the steps that are left only shrink the range further (it changes when one of them wins).  Quantized values end at
//     xmax + s / 2 and xmin - s / 2 at the latest (symmetric: at qmax s and qmin s; a zero point is rounded, and clamped
//     towards the range), which moves towards zero from step to step, so once what the ends alone clip there (less MSE_SLACK
//     for the roundings of either evaluation, |x| < 2) is more than the best error for all rows of a wave, it is done: after
//     28 of 80 steps on average.  Not where a later step's range would be clamped at 1e-5, which widens it again;
//   * elements past the row's end are zeros: with qmin <= z <= qmax they quantize to themselves and add nothing.
// The estimate and mse_row_error differ by a relative delta at most (mse_margin below).  Where `margin` cannot tell the two
// steps apart, the wave evaluates mse_row_error for both of them, so the range is always the one mse_range_kernel finds: an
// estimate that decides ties by itself picked another range for one group in 16000.  A step with the scale and zero point of
// the best one (a clamped scale) has its error and is not better.  Rows whose largest value is below `small` or above
// `large`, where powers of the unscaled errors may under- or overflow, are always evaluated, and so are estimates below
// MSE_SMALL, next to which underflowed terms might count: small = 2^(-68 / norm), 2^-28 for 2.4, leaves MSE_SMALL small^norm = 2^-91,
// 2^21 times the 2^-112 that 2^14 underflowed terms can come to; large = 2^(113 / norm - 1), 2^46 for 2.4, keeps 2^14 terms of at
// most (2 large)^norm below 2^127.  In a row with an infinity or a NaN the error of every step is NaN: it keeps its range.
// What bounds it: nine instructions per element and step, two of them transcendental (60 vector cycles for 64 elements), over
// the 20 steps' worth of elements that the slowest row of a wave needs.  4096 x 4096 bf16 in groups of 128, 80 steps, 4 bits:
// 1864 us re-reading, 497 with the row in registers, 225 with the steps cut short and near-ties evaluated, 183 with the last
// steps left out, 179 on four lanes a row; 8 bits 62 -> 19 (4096 rows of 4096: 381 -> 350 and 102 -> 65).
constexpr float MSE_SMALL = 1.1920929e-7f;                   // 2^-23, in units of (largest value of the row, 1 .. 2) ^ norm
constexpr float MSE_SLACK = 2e-5f;
template <int BF, int TEAM, int PER>
__global__ __launch_bounds__(256) void mse_range_team_kernel(const void* __restrict__ x, int64_t rows, int cols, int vec, int steps,
                                                             int grid_n, float norm, float margin, float small, float large, IntOp<0, false> op,
                                                             float* __restrict__ mn_out, float* __restrict__ mx_out) {
  constexpr int N = Vec<BF>::N;
  constexpr bool BLOCK = TEAM > 64;
  constexpr int SUB = BLOCK ? 64 : TEAM;                     // lanes of a wave that share a row
  __shared__ float shrink[256];                              // p of every step (a double division each)
  __shared__ float sm[8];
  for (int i = threadIdx.x; i < steps; i += 256) shrink[i] = (float)(1.0 - (double)i / (double)grid_n);
  __syncthreads();
  const int64_t row_ = ((int64_t)blockIdx.x * 256 + threadIdx.x) / TEAM;
  const int64_t row = row_ < rows ? row_ : rows - 1;         // surplus teams repeat the last row and store nothing
  const int t = threadIdx.x % TEAM, lane = threadIdx.x & 63;
  float v[PER], mn = __builtin_inff(), mx = -__builtin_inff();
  if (vec) {
    #pragma unroll
    for (int c = 0; c < PER / N; ++c) {                      // chunks dealt out round robin: whole lines per instruction
      const int col = (c * TEAM + t) * N;
      u32x4 raw = {0, 0, 0, 0};
      if (col < cols) raw = *(const u32x4*)((const char*)x + (row * cols + col) * (BF ? 2 : 4));
      unpack<BF>(raw, v + c * N);
      if (col < cols)
        #pragma unroll
        for (int i = 0; i < N; ++i) { mn = nan_min(mn, v[c * N + i]); mx = nan_max(mx, v[c * N + i]); }
    }
  } else {
    #pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int col = i * TEAM + t;
      v[i] = 0.0f;
      if (col < cols) { v[i] = load_scalar<BF>(x, row * cols + col); mn = nan_min(mn, v[i]); mx = nan_max(mx, v[i]); }
    }
  }
  if constexpr (BLOCK) block_range(mn, mx, sm);
  else team_range<TEAM>(mn, mx);
  const auto row_sum = [&](float e) {                        // the same value in every lane of the row
    if constexpr (!BLOCK) return team_sum<TEAM>(e);
    e = team_sum<64>(e);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = e;
    __syncthreads();
    return (sm[0] + sm[1]) + (sm[2] + sm[3]);
  };
  float cur_min = mn, cur_max = mx;
  // 2^k with 2^k max|x| in [1, 2)
  const float big = fmaxf(fabsf(mn), fabsf(mx));
  const bool live = row_ < rows && mn > -__builtin_inff() && mx < __builtin_inff();       // (NaN: false)
  const bool regular = live && big >= small && big <= large;
  const int e = regular ? (int)(f2u(big) >> 23) : 127;
  const float up = u2f((uint32_t)(254 - e) << 23), down = u2f((uint32_t)e << 23);
  #pragma unroll
  for (int i = 0; i < PER; ++i) v[i] *= up;
  const float top = mx * up, bottom = mn * up, last_p = shrink[steps - 1];
  const auto power = [&](float d) { return __builtin_amdgcn_exp2f(norm * __builtin_amdgcn_logf(fabsf(d))); };
  // an estimate above `hi` cannot beat the best step, one below `lo` does
  float hi = live ? __builtin_inff() : -1.0f, lo = regular ? __builtin_inff() : -__builtin_inff();
  float best = __builtin_inff(), best_s = -1.0f, best_z = 0.0f;        // mse_row_error of the best step (if `have`), its parameters
  bool have = true;                                          // before the first step: infinity
  #pragma unroll 1
  for (int i = 0; i < steps; ++i) {
    const float p = shrink[i];
    const float xmin = p * cur_min, xmax = p * cur_max;
    const IntRow prm = op.make(xmin, xmax);
    const float s = prm.s * up, r = prm.r * down;
    const auto add = [&](float w, float sum) {
      const float q = __builtin_amdgcn_fmed3f(rintf(w * r), prm.lo, prm.hi);
      const float d = q * s - w;                             // (both operations rounded, as in deq)
      return sum + power(d);
    };
    if (__all(fmaxf(add(top, 0.0f), add(bottom, 0.0f)) > hi)) {                // (a workgroup's lanes all hold the same two)
      // what this and every later step clip at the ends, from above (see the comment)
      const float slack = op.sym ? 0.0f : 0.5f * s;
      const float over = fmaxf(top - ((op.sym ? op.qmax * s : xmax * up) + slack) - MSE_SLACK, 0.0f);
      const float under = fmaxf((op.sym ? op.qmin * s : xmin * up) - slack - bottom - MSE_SLACK, 0.0f);
      const float smallest = last_p * (op.sym ? fmaxf(fabsf(cur_min), fabsf(cur_max)) : cur_max - cur_min);
      if (__all((smallest > 2e-5f && power(over) + power(under) > hi) || hi < 0.0f)) break;
      continue;
    }
    float err = 0.0f, sum = 0.0f;
    #pragma unroll
    for (int quarter = 0; quarter < 4; ++quarter) {
      #pragma unroll
      for (int j = quarter * (PER / 4); j < (quarter + 1) * (PER / 4); ++j) err = add(v[j], err);
      sum = row_sum(err);
      if (quarter < 3 && __all(sum > hi)) break;
    }
    bool better = sum < lo;
    const bool close = live && !better && !(sum > hi) && !(prm.s == best_s && prm.z == best_z);
    float exact = 0.0f;
    for (uint64_t need = __ballot(close && lane % SUB == 0); need; need &= need - 1) {
      const int src = __builtin_ctzll(need);
      const auto of = [&](float f) { return u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(f), src)); };
      const int64_t r_ = BLOCK ? (int64_t)blockIdx.x : ((int64_t)blockIdx.x * 256 + (threadIdx.x & ~63) + src) / TEAM;
      const float en = mse_row_error<BF>(x, r_, cols, op.make(of(xmin), of(xmax)), norm, op, lane);
      float eb = of(best);
      if (!__builtin_amdgcn_readlane((int)have, src)) eb = mse_row_error<BF>(x, r_, cols, op.make(of(cur_min), of(cur_max)), norm, op, lane);
      if (lane / SUB == src / SUB) { exact = en; best = eb; have = true; }
    }
    if (close) better = exact < best;
    if (better) {
      cur_min = xmin; cur_max = xmax;
      best_s = prm.s; best_z = prm.z;
      have = close;
      if (close) best = exact;
      if (regular) {
        hi = fmaxf(sum * (1.0f + margin), MSE_SMALL);
        lo = sum >= MSE_SMALL ? sum * (1.0f - margin) : -__builtin_inff();
      }
    }
  }
  if (t == 0 && row_ < rows) { mn_out[row] = cur_min; mx_out[row] = cur_max; }
}

// Two estimates that differ by more than this tell which of the two errors is larger.  delta bounds the relative difference
// between an estimate and mse_row_error:
//   powers   v_log is good to an ulp of |log2 d| < 32 (2^-19), times norm, and the product to half an ulp of 128 (2^-18), both
//            times ln 2; v_exp and powf to an ulp each;
//   ties     where x * (1/s) and x / s round to different integers, |x/s| is within |x/s| 2^-22 of a half-integer and both
//            errors are s / 2 to (levels + 1) 2^-19.5, levels = qmax - qmin >= |x/s| - 1/2; norm times that for the power;
//   sums     of non-negative terms: 2^-24 for every addition a term goes through, in either order.
// (1 + delta) / (1 - delta) on either side: 2.5 delta.
float mse_margin(int64_t cols, int per, float levels, float norm) {
  const float delta = norm * 1.33e-6f + 2.65e-6f + 5e-7f + norm * (levels + 1.0f) * 1.35e-6f + (float)(cols / 64 + per + 16) * 6e-8f;
  return 2.5f * delta;
}

template <int BF>
int run_mse(const void* x, int64_t rows, int64_t cols, int steps, int grid_n, float norm, const IntOp<0, false>& op,
            float* min_out, float* max_out, hipStream_t st) {
  constexpr int N = Vec<BF>::N;
  const int vec = cols % N == 0 && (uintptr_t)x % 16 == 0;
  #define LCQ_MSE(T, P) do { const int64_t grid = (rows * T + 255) / 256; if (grid > 0x7fffffff) return LCQ_EINVAL; \
    mse_range_team_kernel<BF, T, P><<<dim3((unsigned)grid), dim3(256), 0, st>>>(x, rows, (int)cols, vec, steps, grid_n, norm, \
        mse_margin(cols, P, op.qrange, norm), ldexpf(1.0f, -(int)(68.0f / norm)), ldexpf(1.0f, (int)(113.0f / norm) - 1), op, min_out, max_out); \
    return LCQ_OK; } while (0)
  if (op.round_zp && op.qmin <= 0.0f && op.qmax >= 0.0f && op.qrange <= 512.0f && norm > 2.0f && norm <= 4.0f && steps <= 256) {
    // Many elements per lane amortise the step's row arithmetic, but below 20000 rows such waves are too few to fill the
    // chip and their steps one after the other are what takes the time: bf16 rows of 128 on 16 / 4 / 2 lanes take 26 / 38 /
    // 38 us at 4096 rows, 42 / 41 / 42 at 16384, - / 54 / 59 at 32768, - / 174 / 181 at 131072 (4 bits, symmetric)
    if (cols <= 32) LCQ_MSE(4, 8);
    if (cols <= 128 && rows < 20000) LCQ_MSE(16, 8);
    if (cols <= 64) LCQ_MSE(4, 16);
    if (cols <= 128) LCQ_MSE(4, 32);
    if (cols <= 512) LCQ_MSE(16, 32);
    if (cols <= 4096) LCQ_MSE(64, 64);
    if (cols <= 16384) LCQ_MSE(256, 64);
  }
  #undef LCQ_MSE
  const int64_t grid = (rows + 3) / 4;
  if (grid > 0x7fffffff) return LCQ_EINVAL;
  mse_range_kernel<BF><<<dim3((unsigned)grid), dim3(256), 0, st>>>(x, rows, cols, steps, grid_n, norm, op, min_out, max_out);
  return LCQ_OK;
}

// One proximal iteration of the HQQ zero-point solver (optimize_weights_proximal, quant.py:587-609):
//   W_q = clamp(round(x * inv_s + z), qmin, qmax);  W_r = (W_q - z) / inv_s;  W_e = shrink(x - W_r)
//   z'  = mean(W_q - (x - W_e) * inv_s)  per row;   abs_err = sum |x - W_r|  per row
// with inv_s = 1 / s and shrink(d) = sign(d) * relu(|d| - inv_beta * |d|^(p-1))  (p == 1: |d| - inv_beta).
// One pass over x; LANES lanes share a row and combine their partial sums with a DPP butterfly.
template <int LANES>
__global__ __launch_bounds__(256) void hqq_step_kernel(const float* __restrict__ x, long long rows, int cols,
                                                       const float* __restrict__ scales, const float* __restrict__ zeros_in,
                                                       float* __restrict__ zeros_out, float* __restrict__ abs_err,
                                                       float* __restrict__ scales_rt, float inv_beta, float p, float qmin,
                                                       float qmax) {
  const int lane = threadIdx.x % LANES;
  const long long row = (long long)blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
  const bool ok = row < rows;
  const long long r = ok ? row : 0;
  const float inv_s = 1.0f / scales[r];
  const float z = zeros_in ? zeros_in[r] : 0.0f;
  const float* xr = x + r * cols;
  float acc_z = 0.0f, acc_e = 0.0f;
  for (int c = lane; c < cols; c += LANES) {
    const float v = xr[c];
    const float wq = __builtin_amdgcn_fmed3f(rintf(v * inv_s + z), qmin, qmax);
    const float wr = (wq - z) / inv_s;
    const float d = v - wr;
    const float ad = fabsf(d);
    const float thr = (p == 1.0f) ? inv_beta : inv_beta * powf(ad, p - 1.0f);
    const float mag = fmaxf(ad - thr, 0.0f);
    const float sgn = (d > 0.0f) ? 1.0f : ((d < 0.0f) ? -1.0f : 0.0f);
    const float we = sgn * mag;
    acc_z += wq - (v - we) * inv_s;
    acc_e += ad;
  }
  acc_z = team_sum<LANES>(acc_z);
  acc_e = team_sum<LANES>(acc_e);
  if (ok && lane == 0) {
    zeros_out[row] = acc_z * (1.0f / (float)cols);      // torch.mean on the GPU: the sum times an fp32 factor
    abs_err[row] = acc_e;
    if (scales_rt) scales_rt[row] = 1.0f / inv_s;
  }
}

}  // namespace

extern "C" {

int lcq_quant_int(const void* x, int dtype, int64_t rows, int64_t cols, float qmin, float qmax, int flags,
                  float out_scale_factor, void* dq, void* codes, int code_dtype, void* scales, void* zeros,
                  void* stream) {
  if (!x || rows < 0 || cols <= 0 || (!scales && (flags & LCQ_FLAG_STATIC))) return LCQ_EINVAL;
  if (rows == 0) return LCQ_OK;
  if (codes && !(code_dtype == LCQ_CODE_U8 || code_dtype == LCQ_CODE_I8 || code_dtype == LCQ_CODE_I32 ||
                 code_dtype == LCQ_CODE_SAME || code_dtype == LCQ_CODE_CT4 || code_dtype == LCQ_CODE_CT8)) return LCQ_EDTYPE;
  if (!(qmax > qmin)) return LCQ_EINVAL;
  if (codes && code_dtype == LCQ_CODE_CT4) {
    // only the vectorised kernels store nibbles: 16-byte chunks, codes + 8 within a nibble
    if (qmin < -8.0f || qmax > 7.0f || (flags & LCQ_FLAG_NO_ROUND_ZP) || cols % 8 != 0) return LCQ_EINVAL;
    if ((((uintptr_t)x | (uintptr_t)dq) % 16) != 0 || ((uintptr_t)codes % 4) != 0) return LCQ_EALIGN;
  }
  if (codes && code_dtype == LCQ_CODE_CT8 && (qmin < -128.0f || qmax > 127.0f || cols % 4 != 0)) return LCQ_EINVAL;
  if ((flags & LCQ_FLAG_SCALES_F16) && (flags & LCQ_FLAG_STATIC)) return LCQ_EINVAL;
  if ((flags & LCQ_FLAG_SCALAR_QP) && !(flags & LCQ_FLAG_STATIC)) return LCQ_EINVAL;
  if ((flags & LCQ_FLAG_SCALE_F32) && !(flags & LCQ_FLAG_STATIC)) return LCQ_EINVAL;
  if (!codes) code_dtype = LCQ_CODE_NONE;
  hipStream_t st = (hipStream_t)stream;
  if (flags & LCQ_FLAG_PROMOTED) {
    if (dtype != LCQ_BF16 && dtype != LCQ_F16) return LCQ_EDTYPE;
    if (!(flags & LCQ_FLAG_STATIC) || (flags & (LCQ_FLAG_NO_ROUND_ZP | LCQ_FLAG_SCALE_F32)) || qmax > 256.0f || qmin < -256.0f) return LCQ_EINVAL;
    if (codes && code_dtype != LCQ_CODE_U8 && code_dtype != LCQ_CODE_I8 && code_dtype != LCQ_CODE_I32) return LCQ_EDTYPE;
    if (cols % 8 != 0 || cols / 8 > 0x7fffffff || (((uintptr_t)x | (uintptr_t)dq | (uintptr_t)codes) % 16) != 0) return LCQ_EALIGN;
    const auto op = make_op<IntOp<0, true>>(qmin, qmax, flags, out_scale_factor, code_dtype);
    const int64_t nchunks = rows * (cols / 8);
    const int64_t grid = nchunks > (int64_t)262144 * 256 ? 262144 : (nchunks + 255) / 256;
    if (dtype == LCQ_BF16) static_promoted_kernel<ROW_BF16><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const u32x4*)x, nchunks, (int)(cols / 8), scales, zeros, dq, codes, op);
    else static_promoted_kernel<ROW_F16><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const u32x4*)x, nchunks, (int)(cols / 8), scales, zeros, dq, codes, op);
    LCQ_CHECK_LAUNCH();
    return LCQ_OK;
  }
  int rc;
  if (dtype == LCQ_F32) rc = run<false>(x, rows, cols, qmin, qmax, flags, out_scale_factor, dq, codes, code_dtype, scales, zeros, st);
  else if (dtype == LCQ_BF16) rc = run<true>(x, rows, cols, qmin, qmax, flags, out_scale_factor, dq, codes, code_dtype, scales, zeros, st);
  else if (dtype == LCQ_F16) rc = run<ROW_F16>(x, rows, cols, qmin, qmax, flags, out_scale_factor, dq, codes, code_dtype, scales, zeros, st);
  else return LCQ_EDTYPE;
  if (rc != LCQ_OK) return rc;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_mse_range(const void* x, int dtype, int64_t rows, int64_t cols, float qmin, float qmax, int flags, int steps,
                  int grid_n, float norm, float* min_out, float* max_out, void* stream) {
  if (!x || !min_out || !max_out || rows <= 0 || cols <= 0 || steps <= 0 || grid_n <= 0) return LCQ_EINVAL;
  if (!(qmax > qmin) || (flags & LCQ_FLAG_STATIC)) return LCQ_EINVAL;
  auto op = make_op<IntOp<false, false>>(qmin, qmax, flags, 1.0f, LCQ_CODE_NONE);
  hipStream_t st = (hipStream_t)stream;
  int rc;
  if (dtype == LCQ_F32) rc = run_mse<false>(x, rows, cols, steps, grid_n, norm, op, min_out, max_out, st);
  else if (dtype == LCQ_BF16) rc = run_mse<true>(x, rows, cols, steps, grid_n, norm, op, min_out, max_out, st);
  else if (dtype == LCQ_F16) rc = run_mse<ROW_F16>(x, rows, cols, steps, grid_n, norm, op, min_out, max_out, st);
  else return LCQ_EDTYPE;
  if (rc != LCQ_OK) return rc;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_hqq_step(const float* x, int64_t rows, int64_t cols, const float* scales, const float* zeros_in, float* zeros_out,
                 float* abs_err_rowsum, float* scales_roundtrip, float inv_beta, float lp_norm, float qmin, float qmax,
                 void* stream) {
  if (!x || !scales || !zeros_out || !abs_err_rowsum || rows <= 0 || cols <= 0 || cols > 0x7fffffff) return LCQ_EINVAL;
  if (!(qmax > qmin) || zeros_in == zeros_out) return LCQ_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (cols <= 256) {
    const int64_t grid = (rows + 15) / 16;
    if (grid > 0x7fffffff) return LCQ_EINVAL;
    hqq_step_kernel<16><<<dim3((unsigned)grid), dim3(256), 0, st>>>(x, rows, (int)cols, scales, zeros_in, zeros_out,
                                                                     abs_err_rowsum, scales_roundtrip, inv_beta, lp_norm, qmin, qmax);
  } else {
    const int64_t grid = (rows + 3) / 4;
    if (grid > 0x7fffffff) return LCQ_EINVAL;
    hqq_step_kernel<64><<<dim3((unsigned)grid), dim3(256), 0, st>>>(x, rows, (int)cols, scales, zeros_in, zeros_out,
                                                                     abs_err_rowsum, scales_roundtrip, inv_beta, lp_norm, qmin, qmax);
  }
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_awq_scale_quant(const void* w, int dtype, int64_t R, int64_t K, const void* colscale, int group_size,
                        float qmin, float qmax, int flags, void* out, void* stream) {
  if (!w || !colscale || !out || R <= 0 || K <= 0 || K > 0x7fffffff) return LCQ_EINVAL;
  if (!(qmax > qmin) || (flags & (LCQ_FLAG_STATIC | LCQ_FLAG_NO_ROUND_ZP))) return LCQ_EINVAL;
  if (qmax > 256.0f || qmin < -256.0f) return LCQ_EINVAL;
  const int64_t cols = group_size > 0 ? group_size : K;
  if (K % cols != 0) return LCQ_EINVAL;
  const int64_t rows = R * (K / cols);
  const int n = dtype == LCQ_F32 ? 4 : 8;
  if (cols % n != 0 || K % n != 0 || ((uintptr_t)colscale % 16) != 0) return LCQ_EALIGN;
  hipStream_t st = (hipStream_t)stream;
  int rc;
  // the group scales / zeros stay in registers: fake_quantize_weight does not return them
  if (dtype == LCQ_F32) {
    auto op = make_op<IntOp<false, true, true>>(qmin, qmax, flags, 1.0f, LCQ_CODE_NONE);
    op.colscale = colscale; op.wrow_cols = (int)K; op.is_static = 0;
    rc = dispatch_rows(w, rows, cols, out, (void*)nullptr, (void*)nullptr, (void*)nullptr, op, false, st);
  } else if (dtype == LCQ_BF16) {
    auto op = make_op<IntOp<true, true, true>>(qmin, qmax, flags, 1.0f, LCQ_CODE_NONE);
    op.colscale = colscale; op.wrow_cols = (int)K; op.is_static = 0;
    rc = dispatch_rows(w, rows, cols, out, (void*)nullptr, (void*)nullptr, (void*)nullptr, op, false, st);
  } else if (dtype == LCQ_F16) {
    auto op = make_op<IntOp<ROW_F16, true, true>>(qmin, qmax, flags, 1.0f, LCQ_CODE_NONE);
    op.colscale = colscale; op.wrow_cols = (int)K; op.is_static = 0;
    rc = dispatch_rows(w, rows, cols, out, (void*)nullptr, (void*)nullptr, (void*)nullptr, op, false, st);
  } else return LCQ_EDTYPE;
  if (rc != LCQ_OK) return rc;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_minmax_rows(const void* x, int dtype, int64_t rows, int64_t cols, void* min_out, void* max_out, void* stream) {
  if (!x || !min_out || !max_out || rows < 0 || cols <= 0) return LCQ_EINVAL;
  if (rows == 0) return LCQ_OK;
  const int64_t grid = (rows + 3) / 4;
  if (grid > 0x7fffffff) return LCQ_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == LCQ_F32) minmax_rows_kernel<false><<<dim3((unsigned)grid), dim3(256), 0, st>>>(x, rows, cols, min_out, max_out);
  else if (dtype == LCQ_BF16) minmax_rows_kernel<true><<<dim3((unsigned)grid), dim3(256), 0, st>>>(x, rows, cols, min_out, max_out);
  else if (dtype == LCQ_F16) minmax_rows_kernel<ROW_F16><<<dim3((unsigned)grid), dim3(256), 0, st>>>(x, rows, cols, min_out, max_out);
  else return LCQ_EDTYPE;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int64_t lcq_minmax_all_workspace_bytes(void) { return 2 * 2048 * sizeof(float); }

int lcq_minmax_all(const void* x, int dtype, int64_t n, void* min_out, void* max_out, void* workspace, void* stream) {
  if (!x || !min_out || !max_out || !workspace || n <= 0) return LCQ_EINVAL;
  int64_t blocks = (n + 256 * 16 - 1) / (256 * 16);
  if (blocks > 2048) blocks = 2048;
  hipStream_t st = (hipStream_t)stream;
  float* part = (float*)workspace;
  if (dtype == LCQ_F32) {
    minmax_all_stage1<false><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(x, n, part);
    minmax_all_stage2<false><<<dim3(1), dim3(256), 0, st>>>(part, (int)blocks, min_out, max_out);
  } else if (dtype == LCQ_BF16) {
    minmax_all_stage1<true><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(x, n, part);
    minmax_all_stage2<true><<<dim3(1), dim3(256), 0, st>>>(part, (int)blocks, min_out, max_out);
  } else if (dtype == LCQ_F16) {
    minmax_all_stage1<ROW_F16><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(x, n, part);
    minmax_all_stage2<ROW_F16><<<dim3(1), dim3(256), 0, st>>>(part, (int)blocks, min_out, max_out);
  } else return LCQ_EDTYPE;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_qparams_int(const void* min_in, const void* max_in, int dtype, int64_t n, float qmin, float qmax, int flags,
                    void* scales, void* zeros, void* stream) {
  if (!min_in || !max_in || !scales || n <= 0) return LCQ_EINVAL;
  const int64_t grid = (n + 255) / 256;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == LCQ_F32)
    qparams_kernel<false><<<dim3((unsigned)grid), dim3(256), 0, st>>>(
        min_in, max_in, n, scales, zeros, make_op<IntOp<false, false>>(qmin, qmax, flags, 1.0f, LCQ_CODE_NONE));
  else if (dtype == LCQ_BF16)
    qparams_kernel<true><<<dim3((unsigned)grid), dim3(256), 0, st>>>(
        min_in, max_in, n, scales, zeros, make_op<IntOp<true, false>>(qmin, qmax, flags, 1.0f, LCQ_CODE_NONE));
  else if (dtype == LCQ_F16)
    qparams_kernel<ROW_F16><<<dim3((unsigned)grid), dim3(256), 0, st>>>(
        min_in, max_in, n, scales, zeros, make_op<IntOp<ROW_F16, false>>(qmin, qmax, flags, 1.0f, LCQ_CODE_NONE));
  else return LCQ_EDTYPE;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_dequant_int(const void* q, int dtype, int64_t rows, int64_t cols, const void* scales, const void* zeros,
                    int flags, float out_scale_factor, void* out, void* stream) {
  if (!q || !scales || !out || rows < 0 || cols <= 0) return LCQ_EINVAL;
  if (rows == 0) return LCQ_OK;
  const int scalar_qp = (flags & LCQ_FLAG_SCALAR_QP) != 0;
  const int scale_f32 = (flags & LCQ_FLAG_SCALE_F32) != 0;
  int64_t grid = (rows * cols + 255) / 256;
  if (grid > 65536) grid = 65536;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == LCQ_F32) dequant_kernel<false><<<dim3((unsigned)grid), dim3(256), 0, st>>>(q, rows, cols, scales, zeros, out, scalar_qp, scale_f32, out_scale_factor);
  else if (dtype == LCQ_BF16) dequant_kernel<true><<<dim3((unsigned)grid), dim3(256), 0, st>>>(q, rows, cols, scales, zeros, out, scalar_qp, scale_f32, out_scale_factor);
  else if (dtype == LCQ_F16) dequant_kernel<ROW_F16><<<dim3((unsigned)grid), dim3(256), 0, st>>>(q, rows, cols, scales, zeros, out, scalar_qp, scale_f32, out_scale_factor);
  else return LCQ_EDTYPE;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

}  // extern "C"
