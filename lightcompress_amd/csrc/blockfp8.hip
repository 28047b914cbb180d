// Block-wise float8 (e4m3) casts for gfx950: one fp32 scale per 128x128 weight block or per
// 128-element activation block.
//
// Replaces the reference's Triton kernels weight_cast_to_fp8 / weight_cast_to_bf16 / act_quant
// (llmc/compression/quantization/kernel.py:7-138) and its non-Hopper fallback through
// FloatQuantizer(granularity='per_block') (quant.py:20-45, 138-140, 634-638, 1194-1220):
//   s = max|x| / 448        (fallback: clamp(max|x|, 1e-5) / 448, LCQ_FLAG_CLAMP_RANGE)
//   y = float8_e4m3fn(x / s)   in fp32 arithmetic whatever the input type
//   back:  out = float(y) * s
// Rounding to float8 is the hardware convert (round to nearest even, what Triton's and torch's casts
// do); LCQ_FLAG_TIE_AWAY nudges exact ties one ulp outwards first (the add-half-then-truncate model of
// float_quantize).
#include "rowquant.h"

namespace {
using namespace lcq;

constexpr int BS = 128;

// x / s for a divisor that many elements share, correctly rounded without the division sequence: with y = RN(1/s) the product
// q0 = x y is within 2 ulp, one residual step makes it faithful and a second one exact (Markstein, IBM J. R&D 34(1), 1990;
// the residuals are exact).  Five full-rate instructions; a guarded product needs as many to find out whether it may stay, and
// values below the minimum normal, where the grid's midpoints are not a bit pattern, went through the division sequence.
// Scales outside 2^-60 .. 2^60 (an infinite or NaN block, a block of subnormals) divide.
struct Divisor {
  float s, y;
  bool fast;
  __device__ __forceinline__ explicit Divisor(float s_) : s(s_), fast(s_ > 8.6736174e-19f && s_ < 1.1529215e18f) {
    const float y0 = __builtin_amdgcn_rcpf(s);
    y = __builtin_fmaf(__builtin_fmaf(-s, y0, 1.0f), y0, y0);
  }
  __device__ __forceinline__ float quotient(float x) const {
    if (__builtin_expect(!fast, 0)) return x / s;
    float q = x * y;                                         // (s q - x taken off, not x - s q added: that way -0 / s stays -0)
    q = __builtin_fmaf(-__builtin_fmaf(s, q, -x), y, q);
    return __builtin_fmaf(-__builtin_fmaf(s, q, -x), y, q);
  }
};

// value handed to the float8 convert.  model = false: x / s itself (Triton / torch cast: one rounding, to
// nearest even, done by the convert).  model = true: the FloatQuantizer route, "x / s + 0" rounded by the
// float_quantize model first - add-half-then-truncate on the fp32 mantissa (ties away; tie_even: to even),
// and below the minimum normal 2^-6 the same on |t| + 2^-6 (whose fp32 addition already rounds once) - so the
// convert only re-encodes an exact grid value.
__device__ __forceinline__ float fp8_input(float x, const Divisor& d, bool tie_away, bool model) {
  float t = d.quotient(x);
  if (!model) return t;
  t = t + 0.0f;                                             // "+ zeros": -0 becomes +0
  if (fabsf(t) >= 0.015625f) {
    if (tie_away && (f2u(t) & 0xfffffu) == 0x80000u) t = u2f(f2u(t) + 1u);   // an exact tie: push it outwards
    return t;
  }
  if (!(fabsf(t) == fabsf(t))) return t;                    // NaN
  const uint32_t b = f2u(fabsf(t) + 0.015625f);
  const uint32_t rb = tie_away ? (b + 0x80000u) & 0xfff00000u : (b + 0x7ffffu + ((b >> 20) & 1u)) & 0xfff00000u;
  return __builtin_copysignf(u2f(rb) - 0.015625f, t);
}

struct BlkArgs {
  const void* x; uint8_t* y; float* scales;
  int64_t M, N;
  int nbn, clamp_range, tie_away;
};

// One workgroup of 512 per 128x128 block: 2048 (bf16) / 4096 (fp32) 16-byte chunks, 4 / 8 per thread in registers.  HBM-bound
// beyond a few thousand blocks; at 2112 x 7168 (952 blocks, less than four per CU) the latency of load - reduce - store: 16.7 us
// with 256 lanes per block and guarded quotients, 11.8 so (7.5 at the rate of a plain stream).
template <bool BF>
__global__ __launch_bounds__(512) void block_quant_kernel(BlkArgs a) {
  constexpr int N = Vec<BF>::N, CPR = BS / N, PER = BS * CPR / 512;
  __shared__ float sm[8];
  const int bm = blockIdx.y, bn = blockIdx.x;
  u32x4 raw[PER];
  bool ok[PER];
  float amax = 0.0f;
  #pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int ci = threadIdx.x + k * 512, r = ci / CPR, c = ci % CPR;
    const int64_t row = (int64_t)bm * BS + r, col = (int64_t)bn * BS + c * N;
    ok[k] = row < a.M && col < a.N;
    raw[k] = ok[k] ? __builtin_nontemporal_load((const u32x4*)a.x + (row * a.N + col) / N) : u32x4{0, 0, 0, 0};
  }
  #pragma unroll
  for (int k = 0; k < PER; ++k) {
    float v[N];
    unpack<BF>(raw[k], v);
    #pragma unroll
    for (int i = 0; i < N; i += 2) amax = nan_max(nan_max(amax, fabsf(v[i])), fabsf(v[i + 1]));
  }
  amax = team_reduce<64, true>(amax);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = amax;
  __syncthreads();
  #pragma unroll
  for (int w = 0; w < 8; ++w) amax = nan_max(amax, sm[w]);
  if (a.clamp_range) amax = nan_max(amax, 1e-5f);
  const float s = amax / 448.0f;
  const Divisor div(s);
  if (threadIdx.x == 0) a.scales[(int64_t)bm * a.nbn + bn] = s;
  #pragma unroll
  for (int k = 0; k < PER; ++k) {
    if (!ok[k]) continue;
    const int ci = threadIdx.x + k * 512, rr = ci / CPR, c = ci % CPR;
    const int64_t row = (int64_t)bm * BS + rr, col = (int64_t)bn * BS + c * N;
    float v[N];
    unpack<BF>(raw[k], v);
    #pragma unroll
    for (int i = 0; i < N; ++i) v[i] = fp8_input(v[i], div, a.tie_away, a.clamp_range);
    uint32_t w[N / 4];
    #pragma unroll
    for (int q = 0; q < N / 4; ++q) {
      int u = 0;
      u = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * q], v[4 * q + 1], u, false);
      u = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * q + 2], v[4 * q + 3], u, true);
      w[q] = (uint32_t)u;
    }
    uint8_t* dst = a.y + row * a.N + col;
    if constexpr (N == 8) *(u32x2*)dst = u32x2{w[0], w[1]};
    else *(uint32_t*)dst = w[0];
  }
}

// activations: one 128-element block per 16-lane (bf16) / 32-lane (fp32) team, one chunk per lane
template <bool BF>
__global__ __launch_bounds__(256) void act_quant_kernel(const u32x4* __restrict__ x, int64_t nblocks, uint8_t* __restrict__ y,
                                                        float* __restrict__ scales, int clamp_range, int tie_away) {
  constexpr int N = Vec<BF>::N, TEAM = BS / N;
  const int64_t blk = ((int64_t)blockIdx.x * 256 + threadIdx.x) / TEAM;
  const int t = threadIdx.x % TEAM;
  const bool okb = blk < nblocks;
  const u32x4 raw = okb ? __builtin_nontemporal_load(x + blk * TEAM + t) : u32x4{0, 0, 0, 0};
  float v[N];
  unpack<BF>(raw, v);
  float amax = 0.0f;
  #pragma unroll
  for (int i = 0; i < N; ++i) amax = nan_max(amax, fabsf(v[i]));
  amax = team_reduce<TEAM, true>(amax);
  if (clamp_range) amax = nan_max(amax, 1e-5f);
  const float s = amax / 448.0f;
  const Divisor div(s);
  if (!okb) return;
  if (t == 0) scales[blk] = s;
  #pragma unroll
  for (int i = 0; i < N; ++i) v[i] = fp8_input(v[i], div, tie_away, clamp_range);
  uint32_t w[N / 4];
  #pragma unroll
  for (int q = 0; q < N / 4; ++q) {
    int u = 0;
    u = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * q], v[4 * q + 1], u, false);
    u = __builtin_amdgcn_cvt_pk_fp8_f32(v[4 * q + 2], v[4 * q + 3], u, true);
    w[q] = (uint32_t)u;
  }
  uint8_t* dst = y + (blk * TEAM + t) * N;
  if constexpr (N == 8) *(u32x2*)dst = u32x2{w[0], w[1]};
  else *(uint32_t*)dst = w[0];
}

// out = float(y) * s[block]: a lane takes W float8 of each of two rows of one block row, so that its output is one 16-byte piece
// next to its neighbours'; the lanes are numbered along the pieces of a row pair, then down, so none is idle whatever the width
// (a workgroup per 256 pieces of a row left most of it idle on narrow matrices).  HBM-bound: 2112 x 7168 to fp32 (76 MB) 14.4 us
// with eight float8 per lane, two half-line stores and a 64-bit division per chunk, 12.3 so (one, four and eight rows: 12.4, 12.3,
// 12.5); 131072 x 128 to bf16 8.6 (8.7, 8.8, 8.9).
constexpr int DQ_ROWS = 2;
template <int OUT>   // LCQ_F32 | LCQ_BF16
__global__ __launch_bounds__(256) void block_dequant_kernel(const uint8_t* __restrict__ y, const float* __restrict__ scales,
                                                            int64_t M, int64_t N, int nbn, uint32_t pieces, void* __restrict__ out) {
  constexpr int W = OUT == LCQ_BF16 ? 8 : 4;
  const uint32_t lane = blockIdx.x * 256u + threadIdx.x, group = lane / pieces;
  const int64_t col = (int64_t)(lane - group * pieces) * W, row0 = (int64_t)group * DQ_ROWS;
  if (row0 >= M) return;
  const float s = scales[(row0 / BS) * nbn + col / BS];
  uint32_t w[DQ_ROWS][W / 4];
  #pragma unroll
  for (int r = 0; r < DQ_ROWS; ++r)
    if (row0 + r < M) {
      if constexpr (W == 8) { const u32x2 v = *(const u32x2*)(y + (row0 + r) * N + col); w[r][0] = v[0]; w[r][W / 4 - 1] = v[1]; }
      else w[r][0] = *(const uint32_t*)(y + (row0 + r) * N + col);
    }
  #pragma unroll
  for (int r = 0; r < DQ_ROWS; ++r)
    if (row0 + r < M) {
      float v[W];
      #pragma unroll
      for (int q = 0; q < W / 4; ++q) {
        const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[r][q], false), hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[r][q], true);
        v[4 * q] = lo[0] * s; v[4 * q + 1] = lo[1] * s; v[4 * q + 2] = hi[0] * s; v[4 * q + 3] = hi[1] * s;
      }
      u32x4* const dst = (u32x4*)((char*)out + ((row0 + r) * N + col) * (OUT == LCQ_BF16 ? 2 : 4));
      if constexpr (OUT == LCQ_BF16) *dst = pack_rne<true>(v);
      else *dst = u32x4{f2u(v[0]), f2u(v[1]), f2u(v[2]), f2u(v[3])};
    }
}

}  // namespace

extern "C" {

int lcq_fp8_block_quant(const void* x, int dtype, int64_t M, int64_t N, int block_rows, int flags, void* y, float* scales,
                        void* stream) {
  if (!x || !y || !scales || M <= 0 || N <= 0) return LCQ_EINVAL;
  if (dtype != LCQ_F32 && dtype != LCQ_BF16) return LCQ_EDTYPE;
  if (block_rows != 1 && block_rows != BS) return LCQ_EINVAL;
  const int n = dtype == LCQ_BF16 ? 8 : 4;
  if (N % n != 0 || ((uintptr_t)x % 16) != 0 || ((uintptr_t)y % 8) != 0) return LCQ_EALIGN;
  hipStream_t st = (hipStream_t)stream;
  const int clamp_range = (flags & LCQ_FLAG_CLAMP_RANGE) != 0, tie_away = (flags & LCQ_FLAG_TIE_AWAY) != 0;
  if (block_rows == 1) {
    if (N % BS != 0) return LCQ_EINVAL;
    const int64_t nblocks = M * (N / BS);
    const int team = BS / n;
    const int64_t grid = (nblocks * team + 255) / 256;
    if (grid > 0x7fffffff) return LCQ_EINVAL;
    if (dtype == LCQ_BF16) act_quant_kernel<true><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const u32x4*)x, nblocks, (uint8_t*)y, scales, clamp_range, tie_away);
    else act_quant_kernel<false><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const u32x4*)x, nblocks, (uint8_t*)y, scales, clamp_range, tie_away);
  } else {
    BlkArgs a;
    a.x = x; a.y = (uint8_t*)y; a.scales = scales; a.M = M; a.N = N;
    a.nbn = (int)((N + BS - 1) / BS); a.clamp_range = clamp_range; a.tie_away = tie_away;
    const dim3 grid((unsigned)a.nbn, (unsigned)((M + BS - 1) / BS));
    if (grid.y > 65535) return LCQ_EINVAL;
    if (dtype == LCQ_BF16) block_quant_kernel<true><<<grid, dim3(512), 0, st>>>(a);
    else block_quant_kernel<false><<<grid, dim3(512), 0, st>>>(a);
  }
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_fp8_block_dequant(const void* y, const float* scales, int64_t M, int64_t N, void* out, int out_dtype, void* stream) {
  if (!y || !scales || !out || M <= 0 || N <= 0) return LCQ_EINVAL;
  if (N % 8 != 0 || ((uintptr_t)y % 8) != 0 || ((uintptr_t)out % 16) != 0) return LCQ_EALIGN;
  const int nbn = (int)((N + BS - 1) / BS);
  if (out_dtype != LCQ_BF16 && out_dtype != LCQ_F32) return LCQ_EDTYPE;
  const int64_t pieces = N / (out_dtype == LCQ_BF16 ? 8 : 4);
  hipStream_t st = (hipStream_t)stream;
  // lanes are numbered in 32 bits: whole block rows per launch (one, but for matrices of more than 3e10 elements)
  const int64_t most = (int64_t)0xffffff00 / (pieces * (BS / DQ_ROWS)) * BS;
  if (most == 0) return LCQ_EINVAL;
  for (int64_t m0 = 0; m0 < M; m0 += most) {
    const int64_t m = M - m0 < most ? M - m0 : most;
    const dim3 grid((unsigned)((pieces * ((m + DQ_ROWS - 1) / DQ_ROWS) + 255) / 256));
    const uint8_t* src = (const uint8_t*)y + m0 * N;
    const float* sc = scales + m0 / BS * nbn;
    if (out_dtype == LCQ_BF16) block_dequant_kernel<LCQ_BF16><<<grid, dim3(256), 0, st>>>(src, sc, m, N, nbn, (uint32_t)pieces, (uint16_t*)out + m0 * N);
    else block_dequant_kernel<LCQ_F32><<<grid, dim3(256), 0, st>>>(src, sc, m, N, nbn, (uint32_t)pieces, (float*)out + m0 * N);
  }
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

}  // extern "C"
