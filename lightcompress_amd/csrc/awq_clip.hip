// AWQ weight-clip search for gfx950.
//
// Replaces AutoClipper.auto_clip_layer / fake_quantize_weight (clip_version v1, weight-only;
// llmc/compression/quantization/auto_clip.py:83-191, 258-262) and apply_clip v1 (:194-211).
// For every (output row r, group g) the reference tries n_steps shrunken ranges
//   max_i = org_max * (1 - i/n_grid),  min_i = org_min * (1 - i/n_grid)      (or -max_i)
// fake-quantizes clamp(w, min_i, max_i) and keeps the range whose per-group partial outputs
//   out[r, t, g] = sum_j x[t, g, j] * w_q[r, g, j]
// are closest (mean over the sampled tokens t of the squared difference) to those of the
// original weights.  It materialises [256, T, G, 128] products per shrink step; here a wave keeps
// 32 rows of one group in registers, derives the bf16 weight DIFFERENCE of every step there and
// multiplies it with the group's token tile (LDS) on bf16 MFMA:
//   err_i[r] = mean_t ( sum_j x[t, j] * (fq_i(w) - w)[r, j] )^2
// The reference rounds both dot products to bf16 before subtracting them; that rounding noise
// (2^-9 of the outputs) is not reproduced, the decision rule is: errors are rounded to bf16 and
// compared with <, so the first minimum wins exactly as `err_mean < min_errs` does.
//
// GEMM shape per wave and step: tokens (M, from LDS) x 32 weight rows (N, registers) x 128 (K).
// With v_mfma_f32_32x32x16_bf16 lane (h = lane/32, c = lane%32) supplies token c / weight row c
// and k = 16 ks + 8 h .. +7 of k-step ks; accumulator register r holds token 8(r/4)+4h+r%4 of
// weight row c, so the sum over tokens is a sum over a lane's registers plus its partner lane.
#include "intop.h"

namespace {
using namespace lcq;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int CG = 128;                  // group size
constexpr int TS = 512;                  // tokens per LDS pass
constexpr int PITCH = CG * 2 + 16;       // bytes per token row in LDS (16-byte skew against bank conflicts)
constexpr int ROWS_PER_WG = 256;         // 8 waves x 32 rows

__global__ __launch_bounds__(512, 1) void awq_clip_kernel(const uint16_t* __restrict__ w, const uint16_t* __restrict__ x,
                                                          int R, int K, int T, int n_grid, int n_steps, int clip_sym,
                                                          IntOp<true, true> op, uint16_t* __restrict__ best_max,
                                                          uint16_t* __restrict__ best_min, float* __restrict__ errs) {
  __shared__ __attribute__((aligned(16))) char lds[TS * PITCH];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, c = lane & 31;
  const int gi = blockIdx.y, G = K / CG;
  const int row = blockIdx.x * ROWS_PER_WG + wave * 32 + c;
  const bool row_ok = row < R;
  const int npass = (T + TS - 1) / TS;

  auto load_tokens = [&](int t0) {                          // tokens t0 .. t0+TS of group gi -> LDS, zero past T
    const int c16 = tid & 15, tr = tid >> 4;
    #pragma unroll 4
    for (int it = 0; it < TS / 32; ++it) {
      const int t = it * 32 + tr;
      u32x4 v = {0, 0, 0, 0};
      if (t0 + t < T) v = *(const u32x4*)(x + (int64_t)(t0 + t) * K + gi * CG + c16 * 8);
      *(u32x4*)(lds + t * PITCH + c16 * 16) = v;
    }
  };

  // this lane's 64 weights of row `row`: j = 16 ks + 8 h + i
  u32x4 wf[8];
  #pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    wf[ks] = u32x4{0, 0, 0, 0};
    if (row_ok) wf[ks] = *(const u32x4*)(w + (int64_t)row * K + gi * CG + 16 * ks + 8 * h);
  }
  float mn = __builtin_inff(), mx = -__builtin_inff();
  #pragma unroll
  for (int ks = 0; ks < 8; ++ks) chunk_minmax<IntOp<true, true>>(wf[ks], mn, mx);
  mn = nan_min(mn, __shfl_xor(mn, 32));
  mx = nan_max(mx, __shfl_xor(mx, 32));
  const float org_min = mn;
  const float org_max = clip_sym ? nan_max(fabsf(mn), fabsf(mx)) : mx;       // w.abs().amax when clip_sym

  if (npass == 1) { load_tokens(0); __syncthreads(); }

  float best = 998244352.0f;                                // bf16(1e9), min_errs = ones_like * 1e9
  float bmax = org_max, bmin = org_min;
  for (int s = 0; s < n_steps; ++s) {
    const float fs = (float)(1.0 - (double)s / (double)n_grid);
    const float max_s = rnd<true>(org_max * fs);
    const float min_s = clip_sym ? -max_s : rnd<true>(org_min * fs);
    // range of the clamped group = clamped range (clamp is monotone)
    const IntRow p = op.make(fminf(fmaxf(mn, min_s), max_s), fminf(fmaxf(mx, min_s), max_s));
    u32x4 bfrag[8];
    #pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      float wv[8], cv[8], d[8];
      unpack<true>(wf[ks], wv);
      #pragma unroll
      for (int i = 0; i < 8; ++i) cv[i] = fminf(fmaxf(wv[i], min_s), max_s);
      op.template fused_dq<8>(cv, d, p);
      #pragma unroll
      for (int i = 0; i < 8; i += 2) rnd_pair<true>(d[i], d[i + 1]);           // fake-quantized weight (bf16)
      #pragma unroll
      for (int i = 0; i < 8; ++i) d[i] -= wv[i];                               // exact in fp32
      bfrag[ks] = pack_rne<true>(d);
    }
    float e = 0.0f;
    for (int ps = 0; ps < npass; ++ps) {
      if (npass > 1) { __syncthreads(); load_tokens(ps * TS); __syncthreads(); }
      const int nt = min(TS, T - ps * TS);
      for (int tb = 0; tb * 32 < nt; ++tb) {
        f32x16 acc;
        #pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
        const char* a0 = lds + (tb * 32 + c) * PITCH + 16 * h;
        #pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
          const u32x4 a = *(const u32x4*)(a0 + 32 * ks);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, bfrag[ks]),
                                                        acc, 0, 0, 0);
        }
        #pragma unroll
        for (int r = 0; r < 16; ++r) e = __builtin_fmaf(acc[r], acc[r], e);
      }
    }
    e += __shfl_xor(e, 32);
    const float mean = e * (1.0f / (float)T);       // torch's GPU mean: the sum times an fp32 factor
    if (errs && row_ok && h == 0) errs[((int64_t)row * G + gi) * n_steps + s] = mean;
    const float eb = rnd<true>(mean);
    if (eb < best) { best = eb; bmax = max_s; bmin = min_s; }
  }
  if (row_ok && h == 0) {
    best_max[(int64_t)row * G + gi] = (uint16_t)(f2u(bmax) >> 16);
    best_min[(int64_t)row * G + gi] = (uint16_t)(f2u(bmin) >> 16);
  }
}

template <int BF>
__global__ __launch_bounds__(256) void clamp_groups_kernel(const u32x4* __restrict__ w, int64_t nchunks, int cpg,
                                                           const void* __restrict__ lo, const void* __restrict__ hi,
                                                           u32x4* __restrict__ out) {
  constexpr int N = Vec<BF>::N;
  for (int64_t ch = (int64_t)blockIdx.x * 256 + threadIdx.x; ch < nchunks; ch += (int64_t)gridDim.x * 256) {
    const int64_t grp = ch / cpg;
    const float l = load_scalar<BF>(lo, grp), u = load_scalar<BF>(hi, grp);
    float v[N];
    unpack<BF>(w[ch], v);
    #pragma unroll
    for (int i = 0; i < N; ++i) v[i] = nan_min(nan_max(v[i], l), u);          // torch.clamp: min(max(x, lo), hi)
    out[ch] = pack<BF>(v);
  }
}

// the same clamp element by element, for group sizes that do not fill 16-byte chunks
template <int BF>
__global__ __launch_bounds__(256) void clamp_groups_scalar_kernel(const void* __restrict__ w, int64_t n, int gs,
                                                                  const void* __restrict__ lo, const void* __restrict__ hi,
                                                                  void* __restrict__ out) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int64_t grp = i / gs;
    store_scalar<BF>(out, i, nan_min(nan_max(load_scalar<BF>(w, i), load_scalar<BF>(lo, grp)), load_scalar<BF>(hi, grp)));
  }
}

// The reference's rounding sequence on the matrix pipe (bf16).
//
//   dot(t, r) = sum_j round(x[t, j] * w[r, j])      every product rounded to the tensors' type, fp32 sums
//
// The rounding of every product keeps the contraction itself off the matrix pipe, but not its two halves:
//   products  v_mfma_f32_32x32x4_2b with ONE non-zero k slot per block is an outer product: block 0 gives x[t, j] w[r, j],
//             block 1 gives x[t, j+1] w[r, j+1] for 32 tokens x 32 rows (exact in fp32), in the same registers of both blocks;
//   rounding  one v_cvt_pk per pair (j, j+1): 16 instructions for 2048 products, all the vector pipe has to do;
//   sums      16 rounded values of a lane (four columns of four tokens) are its share of the dense operand of
//             v_smfmac_f32_16x16x64, whose other operand is sparse: two of four values.  That one holds ones where a value belongs
//             to an output and nothing elsewhere: 1024 values meet their sums in 16 cycles, where a dense instruction takes 512.
// Layouts: products leave lane l with row l % 32 and tokens 8 (i / 4) + 4 (l / 32) + i % 4 in register i.  Lane l supplies the
// values k = 8 (l / 16) .. + 7 and 32 + 8 (l / 16) .. + 7 of column l % 16 of the dense operand, and the sparse one holds the values
// k = 16 (l / 16) .. + 15 of row l % 16, two of every four.  Row 4 h + o adds what the lanes of quarter h hold of output o, and the
// accumulator has rows 4 (l / 16) + i of column l % 16 in register i: sum[q][i] of a lane is its own product register 4 q + i.
// What bounds it: 2 x 64 + 4 x 16 matrix-pipe cycles per 4096 products, and 32 conversions of 4 cycles each (half the rate of other
// vector instructions) that only partly run beside them: two waves per SIMD take 302 cycles (328 with the pairs added by four
// v_mfma_f32_16x16x32 per 2048 products, 256 matrix cycles).  v_mfma_f32_32x32x1 and v_dot2_f32_bf16 would do the same sums, but
// neither overlaps with vector instructions on this chip, and moving a quarter of the sums to the vector pipe made it 13 % slower.
// Measured: 4096 x 11008, 512 tokens, 10 steps, all errors: 8.57 ms with those, 7.95 so; the products one after the other in the
// same registers, or conversions between the sums instead of ahead of them, are slower still.
typedef __attribute__((ext_vector_type(4))) short i16x4;
typedef __attribute__((ext_vector_type(32))) float f32x32;
typedef __attribute__((ext_vector_type(16))) __bf16 bf16x16;
typedef __attribute__((ext_vector_type(8))) uint32_t u32x8;

__device__ __forceinline__ f32x32 outer_products(u32x2 a, u32x2 b) {
  f32x32 z;
  #pragma unroll
  for (int i = 0; i < 32; ++i) z[i] = 0.0f;
  return __builtin_amdgcn_mfma_f32_32x32x4bf16_1k(__builtin_bit_cast(i16x4, a), __builtin_bit_cast(i16x4, b), z, 0, 0, 0);
}
// The sparse operand: where this lane's share holds ones, and which two of every four values they stand for.
// Outputs 0 and 1 of a lane are in its values 0 .. 7, two and three in 8 .. 15; an even one in the first two of every four.
struct Sums { u32x4 ones; int places; };
__device__ __forceinline__ Sums sums_of_own_values(int lane) {
  const int h = (lane >> 2) & 3, o = lane & 3, quarter = lane >> 4;         // row l % 16 = 4 h + o of the operand
  const uint32_t one = quarter == (h >> 1) + (o & 2) ? 0x3f803f80u : 0u, first = (h & 1) ? 0u : one, second = (h & 1) ? one : 0u;
  return Sums{u32x4{first, first, second, second}, (o & 1) ? 0xeeee : 0x4444};
}
__device__ __forceinline__ f32x4 add_values(const u32x8& values, const Sums& to, f32x4 c) {
  return __builtin_amdgcn_smfmac_f32_16x16x64_bf16(__builtin_bit_cast(bf16x8, to.ones), __builtin_bit_cast(bf16x16, values), c, to.places, 0, 0);
}

constexpr int GT = 32;                   // tokens and rows of one wave's tile
template <int GS> constexpr int gd_pitch() { return GS * 2 + 16; }     // bytes per LDS row (16-byte skew)
// sum[4] of a tile: a = the tokens' GS columns (lane l: token l % 32), wrow = row l % 32 in LDS.  The products of the next
// column pair are issued before the current ones are rounded: the empty asm keeps that order (without it the compiler
// runs the two one after the other in the same registers).
template <int GS>
__device__ __forceinline__ void dots_tile(const u32x4* a, const char* wrow, uint32_t mask, const Sums& to, f32x4* sum) {
  #pragma unroll
  for (int q = 0; q < 4; ++q) sum[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  u32x4 b = *(const u32x4*)wrow, ahead = *(const u32x4*)(wrow + 16);
  const auto products = [&](int i) {                        // columns 2 i (block 0) and 2 i + 1 (block 1)
    const int p = i & 3;
    if (p == 0 && i > 0) {
      asm volatile("" : "+v"(ahead));                       // (or the load moves to where it is used: 1 %)
      b = ahead;
      if (i + 4 < GS / 2) ahead = *(const u32x4*)(wrow + 4 * (i + 4));
    }
    const u32x4 av = a[i >> 2];
    const uint32_t w = b[p] & mask;
    return outer_products(p < 2 ? u32x2{av[0], av[1]} : u32x2{av[2], av[3]}, (p & 1) ? u32x2{0, w} : u32x2{w, 0});
  };
  f32x32 d[2];
  d[0] = products(0);
  u32x8 pr[4];                                              // four columns (2 i .. 2 i + 3) of the four tokens of product register 4 q + k
  #pragma unroll
  for (int q = 0; q < 4; ++q) pr[q] = u32x8{0, 0, 0, 0, 0, 0, 0, 0};
  #pragma unroll
  for (int i = 0; i < GS / 2; ++i) {
    f32x32& cur = d[i & 1];
    if (i + 1 < GS / 2) {
      d[(i + 1) & 1] = products(i + 1);
      asm volatile("" : "+v"(d[0]), "+v"(d[1]));
    }
    #pragma unroll
    for (int q = 0; q < 4; ++q)
      #pragma unroll
      for (int k = 0; k < 4; ++k) pr[q][4 * (k >> 1) + 2 * (i & 1) + (k & 1)] = bf16_pack_rne(cur[4 * q + k], cur[16 + 4 * q + k]);
    asm volatile("" : "+v"(pr[0]), "+v"(pr[1]), "+v"(pr[2]), "+v"(pr[3]));
    if (i & 1) {
      #pragma unroll
      for (int q = 0; q < 4; ++q) sum[q] = add_values(pr[q], to, sum[q]);
    }
  }
}

// A column of the dense operand in add_values holds the values of four lanes (l % 16), kept apart by the zeros of the other one, and
// 0 * infinity is NaN: an infinite or NaN product (an infinite or NaN weight, a product beyond the largest bf16 number) turns the sums
// of those lanes into NaN as well.  So a lane with a sum that is not finite adds its products up again one by one:
// x: the group's columns of token 0, w: where the weights of the lane's row lie in LDS.  Off the path of finite tiles, which pay for
// the test alone.
template <int GS>
__device__ __forceinline__ void redo_sums_that_are_not_finite(const uint16_t* __restrict__ x, int64_t K, int t0, int T, const char* w, int lane,
                                                              f32x4* sum) {
  float m = 0.0f;
  #pragma unroll
  for (int q = 0; q < 4; ++q)
    #pragma unroll
    for (int i = 0; i < 4; i += 2) m = nan_max(nan_max(m, fabsf(sum[q][i])), fabsf(sum[q][i + 1]));
  if (__builtin_expect(m < __builtin_inff(), 1)) return;
  const int tok = t0 + 4 * (lane >> 5);
  #pragma unroll
  for (int q = 0; q < 4; ++q) sum[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  #pragma unroll 1
  for (int j = 0; j < GS; ++j) {
    const float wv = u2f((uint32_t)*(const uint16_t*)(w + 2 * j) << 16);
    #pragma unroll
    for (int q = 0; q < 4; ++q)
      #pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = tok + 8 * q + i;
        const float xv = t < T ? u2f((uint32_t)x[(int64_t)t * K + j] << 16) : 0.0f;
        sum[q][i] += rnd<true>(xv * wv);
      }
  }
}

// the columns of one token; a token past T: zeros, which add nothing
template <int GS>
__device__ __forceinline__ void load_token(const uint16_t* __restrict__ x, int64_t K, int T, int t, u32x4* a) {
  const bool ok = t < T;
  const uint16_t* xr = x + (ok ? t : 0) * K;
  #pragma unroll
  for (int c = 0; c < GS / 8; ++c) { a[c] = *(const u32x4*)(xr + 8 * c); if (!ok) a[c] = u32x4{0, 0, 0, 0}; }
}
__device__ __forceinline__ void round_sums(f32x4* v) {
  #pragma unroll
  for (int q = 0; q < 4; ++q)
    #pragma unroll
    for (int i = 0; i < 4; i += 2) {
      float o0 = v[q][i], o1 = v[q][i + 1];
      rnd_pair<true>(o0, o1);
      v[q][i] = o0; v[q][i + 1] = o1;
    }
}
// the rounded sums of a lane as 32 bytes in two pieces (tokens 0 .. 7 and 8 .. 15 of the lane), the pieces of the 64 lanes side by side
constexpr int ORG_HALF = 64 * 16;
__device__ __forceinline__ void store_org(char* at, const f32x4* v) {
  #pragma unroll
  for (int p = 0; p < 2; ++p)
    *(u32x4*)(at + p * ORG_HALF) = u32x4{bf16_pack(v[2 * p][0], v[2 * p][1]), bf16_pack(v[2 * p][2], v[2 * p][3]),
                                         bf16_pack(v[2 * p + 1][0], v[2 * p + 1][1]), bf16_pack(v[2 * p + 1][2], v[2 * p + 1][3])};
}
__device__ __forceinline__ void load_org(const char* at, f32x4* v) {
  #pragma unroll
  for (int p = 0; p < 2; ++p) {
    const u32x4 raw = *(const u32x4*)(at + p * ORG_HALF);
    #pragma unroll
    for (int d = 0; d < 4; ++d) { v[2 * p + d / 2][2 * (d & 1)] = u2f(raw[d] << 16); v[2 * p + d / 2][2 * (d & 1) + 1] = u2f(raw[d] & 0xffff0000u); }
  }
}
// v of lane l + v of lane l ^ 32
__device__ __forceinline__ float both_halves(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(f2u(v), f2u(v), false, false);
  return u2f(s[0]) + u2f(s[1]);
}
// the error of the lane's row over the 32 tokens of the tile; org rounded
__device__ __forceinline__ float tile_error(const f32x4* cur, const f32x4* org) {
  float e[2] = {0.0f, 0.0f};
  #pragma unroll
  for (int q = 0; q < 4; ++q)
    #pragma unroll
    for (int i = 0; i < 4; i += 2) {
      float c0 = cur[q][i], c1 = cur[q][i + 1];
      rnd_pair<true>(c0, c1);
      c0 -= org[q][i]; c1 -= org[q][i + 1];
      rnd_pair<true>(c0, c1);
      c0 *= c0; c1 *= c1;
      rnd_pair<true>(c0, c1);
      e[0] += c0; e[1] += c1;
    }
  return both_halves(e[0] + e[1]);
}

__device__ __forceinline__ float shrunk(float v, int s, int n_grid) { return rnd<true>(v * (float)(1.0 - (double)s / (double)n_grid)); }

// 32 rows of one group to LDS: version 0 as they are, version s + 1 clamped to the range of step s and fake-quantized.
template <int GS>
__device__ __forceinline__ void make_versions(char* smem, const uint16_t* __restrict__ w, int R, int K, int r0, int g, int n_grid, int n_steps,
                                              int clip_sym, const IntOp<true, true>& op) {
  constexpr int PITCH_W = gd_pitch<GS>(), TEAM = GS / 8, VERSION = GT * PITCH_W;
  const int tid = threadIdx.x;
  for (int ch = tid; ch < GT * TEAM; ch += blockDim.x) {                 // one 16-byte chunk per thread (and turn)
    const int row = ch / TEAM, c = ch % TEAM;
    u32x4 raw = {0, 0, 0, 0};
    if (r0 + row < R) raw = *(const u32x4*)(w + (int64_t)(r0 + row) * K + g * GS + c * 8);
    char* dst = smem + row * PITCH_W + c * 16;
    *(u32x4*)dst = raw;
    float v[8], mn = __builtin_inff(), mx = -__builtin_inff();
    unpack<true>(raw, v);
    chunk_minmax<IntOp<true, true>>(raw, mn, mx);
    team_range<TEAM>(mn, mx);
    const float org_max = clip_sym ? nan_max(fabsf(mx), fabsf(mn)) : mx;
    for (int s = 0; s < n_steps; ++s) {
      const float hi = shrunk(org_max, s, n_grid), lo = clip_sym ? -hi : shrunk(mn, s, n_grid);
      const IntRow p = op.make(nan_min(nan_max(mn, lo), hi), nan_min(nan_max(mx, lo), hi));   // range of the clamped group
      float cv[8], d[8];
      #pragma unroll
      for (int i = 0; i < 8; ++i) cv[i] = nan_min(nan_max(v[i], lo), hi);
      op.template fused_dq<8>(cv, d, p);
      *(u32x4*)(dst + (s + 1) * VERSION) = pack_rne<true>(d);
    }
  }
}

// The whole search of AutoClipper.auto_clip_layer (v1, weight-only, bf16, groups of GS columns) in one launch: a workgroup
// owns 32 rows of one group, keeps the original and the n_steps clamped-and-quantized versions of them in LDS, and every
// wave runs all versions over its 32-token tiles; neither the candidates nor the [R, G, T] products reach memory.
template <int GS>
__global__ __launch_bounds__(512, 2) void clip_search_kernel(const uint16_t* __restrict__ w, const uint16_t* __restrict__ x,
                                                             int R, int K, int T, int n_grid, int n_steps, int clip_sym,
                                                             IntOp<true, true> op, uint16_t* __restrict__ best_max,
                                                             uint16_t* __restrict__ best_min, float* __restrict__ errs) {
  constexpr int PITCH_W = gd_pitch<GS>(), TEAM = GS / 8, VERSION = GT * PITCH_W;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* const esum = (float*)(smem + (n_steps + 1) * VERSION);          // [waves][n_steps][32]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
  const int G = K / GS, g = blockIdx.x % G, r0 = (blockIdx.x / G) * GT;
  const auto shrink = [&](float v, int s) { return shrunk(v, s, n_grid); };

  for (int i = tid; i < waves * n_steps * GT; i += blockDim.x) esum[i] = 0.0f;
  make_versions<GS>(smem, w, R, K, r0, g, n_grid, n_steps, clip_sym, op);
  __syncthreads();

  const uint32_t mask = lane < 32 ? 0xffffu : 0xffff0000u;
  const Sums to = sums_of_own_values(lane);
  const char* wrow = smem + (lane & 31) * PITCH_W;
  for (int t0 = wave * GT; t0 < T; t0 += waves * GT) {
    u32x4 a[GS / 8];
    load_token<GS>(x + g * GS, K, T, t0 + (lane & 31), a);
    f32x4 org[4], cur[4];
    dots_tile<GS>(a, wrow, mask, to, org);
    redo_sums_that_are_not_finite<GS>(x + g * GS, K, t0, T, wrow, lane, org);
    round_sums(org);
    #pragma unroll 1
    for (int s = 0; s < n_steps; ++s) {
      dots_tile<GS>(a, wrow + (s + 1) * VERSION, mask, to, cur);
      redo_sums_that_are_not_finite<GS>(x + g * GS, K, t0, T, wrow + (s + 1) * VERSION, lane, cur);
      const float e = tile_error(cur, org);
      if (lane < GT) esum[(wave * n_steps + s) * GT + lane] += e;
    }
  }
  __syncthreads();
  // err_mean < min_errs, step by step: the first minimum below 1e9 wins, NaN never does
  if (tid < GT && r0 + tid < R) {
    const int row = tid;
    float mn = __builtin_inff(), mx = -__builtin_inff();
    for (int c = 0; c < TEAM; ++c) chunk_minmax<IntOp<true, true>>(*(const u32x4*)(smem + row * PITCH_W + c * 16), mn, mx);
    const float org_max = clip_sym ? nan_max(fabsf(mx), fabsf(mn)) : mx;
    float best = 998244352.0f, bmax = org_max, bmin = mn;                 // bf16(1e9)
    const int64_t at = (int64_t)(r0 + row) * G + g;
    for (int s = 0; s < n_steps; ++s) {
      float e = 0.0f;
      for (int wv = 0; wv < waves; ++wv) e += esum[(wv * n_steps + s) * GT + row];
      e = rnd<true>(e * (1.0f / (float)T));                              // torch's mean: the sum times an fp32 factor
      if (errs) errs[at * n_steps + s] = e;
      const float hi = shrink(org_max, s), lo = clip_sym ? -hi : shrink(mn, s);
      if (e < best) { best = e; bmax = hi; bmin = lo; }
    }
    best_max[at] = (uint16_t)(f2u(bmax) >> 16);
    best_min[at] = (uint16_t)(f2u(bmin) >> 16);
  }
}

// The same search without the errors of steps that cannot win (errs == NULL, at most two tiles of tokens per wave).
//
// The rounded original sums o_t are computed as above; a step's sums only up to their roundings, as plain matrix products:
//   a_t = sum_j x w_s - o_t,   |e_t - a_t| <= b_t = u (sum_j |x w_s| + |sum_j x w_s| + |a_t|)
// (every product, the sum and the difference are rounded once, each by at most 2^-8 / (1 + 2^-8) of itself; CLIP_U adds what these
// roundings do to each other, 2 u of u, and 2.5e-3 u for the fp32 sums of either side), so
//   sum_t max(|a_t| - b_t, 0)^2 <= sum_t e_t^2 <= sum_t (|a_t| + b_t)^2.
// A step whose lower bound is above the smallest upper bound of its row by more than what rounding the squares (2^-8 either way)
// and the mean (a bf16 step, 2^-7) can make up for neither wins nor ties (CLIP_MARGIN).  The other steps of rows with more than one of
// them are evaluated as above, 32 (step, row) pairs to a tile whatever rows and steps they come from: first the most promising step of
// each row (its exact sum decides again, with nothing of the bounds' slack on its side), then the others on half of the tokens, where
// exact sums and the bounds of the rest decide once more.  Rows that are not plain (a bound that is not finite, or below
// CLIP_SMALL where underflow might count, or near the 1e9 the search starts from) have every step evaluated.
// Measured (an MLP's Linears as above, all three without errors, 10 steps): 25.7 -> 17.9 ms; 3.7 of 10 steps are evaluated (5.6 without the
// first step ahead of the others: 21.0 ms; a second and a third step by itself: 19.2, 20.7, a pass costs its tiles however few rows
// it still has), the matrix pipes are busy in 45 % of the cycles (the making of the versions, estimates and decisions are not
// overlapped by another workgroup: one fills the LDS).  One step at a time in the estimates, and decisions by a single wave: 1.6 ms
// more.  Four waves per SIMD, tokens read as they are used so that 128 registers hold it: 23.0 against 21.0 ms, the conversions of
// two waves already fill the vector pipe beside the products.
constexpr float CLIP_U = 3.95e-3f, CLIP_MARGIN = 1.02f, CLIP_SMALL = 1e-25f;
template <int GS> constexpr size_t clip_pruned_lds(int n_steps, int waves, int rounds) {
  return (size_t)(n_steps + 1) * GT * gd_pitch<GS>() + (size_t)rounds * waves * GT * GT * 2 + (size_t)waves * n_steps * GT * 8 +
         (size_t)(rounds + 1) * n_steps * GT * 8 + (size_t)(n_steps + 1) * GT * 2 + GT * 4 + 16;
}

template <int GS>
__global__ __launch_bounds__(512, 2) void clip_search_pruned_kernel(const uint16_t* __restrict__ w, const uint16_t* __restrict__ x,
                                                                    int R, int K, int T, int n_grid, int n_steps, int clip_sym,
                                                                    IntOp<true, true> op, uint16_t* __restrict__ best_max,
                                                                    uint16_t* __restrict__ best_min) {
  constexpr int PITCH_W = gd_pitch<GS>(), TEAM = GS / 8, VERSION = GT * PITCH_W;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
  const int rounds = (T + waves * GT - 1) / (waves * GT), pairs = n_steps * GT;
  const int G = K / GS, g = blockIdx.x % G, r0 = (blockIdx.x / G) * GT;
  char* const orgs = smem + (n_steps + 1) * VERSION;                     // [tiles] rounded sums of the original weights (store_org)
  float* const part = (float*)(orgs + rounds * waves * 2 * ORG_HALF);    // [waves][pairs] bounds; later [waves][pairs] exact sums
  float* const tab = part + waves * pairs * 2;                           // [rounds][pairs] lower, upper
  float* const bounds = tab + rounds * pairs * 2;                        // [pairs] lower, upper
  uint16_t* const list = (uint16_t*)(bounds + pairs * 2);                // (step, row) = entry / 32, entry % 32
  uint32_t* const masks = (uint32_t*)(list + pairs + GT);                // steps of a row that may still win, the step evaluated first (from bit LEAD on); FOUND: the one left wins
  int* const count = (int*)(masks + GT);
  const uint16_t* const xg = x + g * GS;
  constexpr uint32_t FOUND = 1u << 31;
  constexpr int LEAD = 24;

  make_versions<GS>(smem, w, R, K, r0, g, n_grid, n_steps, clip_sym, op);
  __syncthreads();

  const uint32_t mask = lane < 32 ? 0xffffu : 0xffff0000u;
  const Sums to = sums_of_own_values(lane);
  const int h = lane >> 5, c = lane & 31;
  for (int k = 0; k < rounds; ++k) {
    const int t0 = (k * waves + wave) * GT;
    if (t0 < T) {
      u32x4 a[GS / 8];
      load_token<GS>(xg, K, T, t0 + c, a);
      // v_mfma_f32_32x32x16: lane (h, c) supplies token / row c and columns 16 ks + 8 h .. + 7; register r holds token
      // 8 (r / 4) + 4 h + r % 4 of row c, as the exact sums do
      f32x4 org[4];
      dots_tile<GS>(a, smem + c * PITCH_W, mask, to, org);
      redo_sums_that_are_not_finite<GS>(xg, K, t0, T, smem + c * PITCH_W, lane, org);
      round_sums(org);
      store_org(orgs + (k * waves + wave) * 2 * ORG_HALF + lane * 16, org);
      u32x4 ax[GS / 16];
      #pragma unroll
      for (int ks = 0; ks < GS / 16; ++ks)
        #pragma unroll
        for (int d = 0; d < 4; ++d) ax[ks][d] = h ? a[2 * ks + 1][d] : a[2 * ks][d];
      // two steps at a time: four independent chains of matrix instructions
      #pragma unroll 1
      for (int s = 0; s < n_steps; s += 2) {
        const char* wr[2];
        f32x16 sum[2], mag[2];
        #pragma unroll
        for (int v = 0; v < 2; ++v) {
          wr[v] = smem + (min(s + v, n_steps - 1) + 1) * VERSION + c * PITCH_W + 16 * h;
          #pragma unroll
          for (int r = 0; r < 16; ++r) { sum[v][r] = 0.0f; mag[v][r] = 0.0f; }
        }
        #pragma unroll
        for (int ks = 0; ks < GS / 16; ++ks) {
          u32x4 aa;
          #pragma unroll
          for (int d = 0; d < 4; ++d) aa[d] = ax[ks][d] & 0x7fff7fffu;
          #pragma unroll
          for (int v = 0; v < 2; ++v) {
            const u32x4 b = *(const u32x4*)(wr[v] + 32 * ks);
            u32x4 ab;
            #pragma unroll
            for (int d = 0; d < 4; ++d) ab[d] = b[d] & 0x7fff7fffu;
            sum[v] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ax[ks]), __builtin_bit_cast(bf16x8, b), sum[v], 0, 0, 0);
            mag[v] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, aa), __builtin_bit_cast(bf16x8, ab), mag[v], 0, 0, 0);
          }
        }
        #pragma unroll
        for (int v = 0; v < 2; ++v) {
          float lo = 0.0f, hi = 0.0f;
          #pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float d = fabsf(sum[v][r] - org[r >> 2][r & 3]), b = CLIP_U * ((mag[v][r] + fabsf(sum[v][r])) + d);
            const float l = fmaxf(d - b, 0.0f), u = d + b;
            lo = __builtin_fmaf(l, l, lo);
            hi = __builtin_fmaf(u, u, hi);
          }
          lo = both_halves(lo);
          hi = both_halves(hi);
          if (h == 0 && s + v < n_steps) *(f32x2*)(part + 2 * ((wave * n_steps + s + v) * GT + c)) = f32x2{lo, hi};
        }
      }
    } else {
      for (int i = lane; i < pairs; i += 64) *(f32x2*)(part + 2 * (wave * pairs + i)) = f32x2{0.0f, 0.0f};
    }
    __syncthreads();
    for (int i = tid; i < pairs; i += blockDim.x) {
      float lo = 0.0f, hi = 0.0f;
      for (int v = 0; v < waves; ++v) { lo += part[2 * (v * pairs + i)]; hi += part[2 * (v * pairs + i) + 1]; }
      *(f32x2*)(tab + 2 * (k * pairs + i)) = f32x2{lo, hi};
    }
    __syncthreads();
  }

  // Which steps may still win: masks and the list of pairs to go on with.  Before anything is evaluated (!led) that is the most
  // promising step of each row; then, with that one evaluated and `done` rounds of tokens of the others, the others.
  const auto decide = [&](bool led, int done) {
    for (int i = tid; i < pairs; i += blockDim.x) {                      // bounds of every pair
      float e = 0.0f, lo = 0.0f, hi = 0.0f;
      if (led)
        for (int v = 0; v < waves; ++v) e += part[v * pairs + i];
      if (!led || ((masks[i % GT] >> LEAD) & 31) != (uint32_t)(i / GT))
        for (int k = done; k < rounds; ++k) { lo += tab[2 * (k * pairs + i)]; hi += tab[2 * (k * pairs + i) + 1]; }
      lo += e; hi += e;
      *(f32x2*)(bounds + 2 * i) = f32x2{lo * (1.0f - 1e-4f), hi * (1.0f + 1e-4f)};              // (their own fp32 sums)
    }
    __syncthreads();
    if (wave != 0) return;
    uint32_t go = 0;
    if (lane < GT && r0 + lane < R) {
      const uint32_t all = (1u << n_steps) - 1, was = led ? masks[lane] : all, cand = was & all;
      if (!(was & FOUND)) {
        f32x2 bnd[LCQ_CLIP_MAX_STEPS];
        #pragma unroll
        for (int s = 0; s < LCQ_CLIP_MAX_STEPS; ++s) {
          bnd[s] = f32x2{0.0f, __builtin_inff()};
          if (s < n_steps) bnd[s] = *(const f32x2*)(bounds + 2 * (s * GT + lane));
        }
        float best = __builtin_inff();
        bool plain = true;
        #pragma unroll
        for (int s = 0; s < LCQ_CLIP_MAX_STEPS; ++s)
          if ((cand >> s) & 1) {
            plain = plain && bnd[s][1] < 1e38f;                          // (NaN: false)
            best = fminf(best, bnd[s][1]);
          }
        plain = plain && best > CLIP_SMALL && best < 9e8f * (float)T;
        uint32_t alive = cand;
        if (plain)
          #pragma unroll
          for (int s = 0; s < LCQ_CLIP_MAX_STEPS; ++s)
            if (bnd[s][0] > best * CLIP_MARGIN) alive &= ~(1u << s);
        const bool found = plain && (alive & (alive - 1)) == 0;          // needs no more sums
        int lead = (was >> LEAD) & 31;
        if (!led) {
          lead = __builtin_ctz(alive);                                   // (the best step is never ruled out: not empty)
          float least = __builtin_inff();
          #pragma unroll
          for (int s = 0; s < LCQ_CLIP_MAX_STEPS; ++s)
            if ((alive >> s) & 1 && bnd[s][0] + bnd[s][1] < least) { least = bnd[s][0] + bnd[s][1]; lead = s; }
        }
        masks[lane] = alive | (uint32_t)lead << LEAD | (found ? FOUND : 0);
        if (!found) go = led ? alive & ~(1u << lead) : 1u << lead;
      }
    }
    int n = 0;
    for (int s = 0; s < n_steps; ++s) {
      const bool on = (go >> s) & 1;
      const uint64_t b = __ballot(on);
      if (on) list[n + __popcll(b & ((1ull << lane) - 1))] = (uint16_t)(s * GT + lane);
      n += __popcll(b);
    }
    if (lane < GT && n + lane < (n + GT - 1) / GT * GT) list[n + lane] = 0;               // (the last tile's surplus lanes)
    if (lane == 0) *count = n;
  };
  decide(false, 0);
  __syncthreads();
  for (int i = tid; i < waves * pairs; i += blockDim.x) part[i] = 0.0f;  // from here on: exact sums
  __syncthreads();
  for (int pass = 0; pass < 2 * rounds; ++pass) {                        // all tokens of the first step, then round by round the others
    const int k = pass < rounds ? pass : pass - rounds;
    const int t0 = (k * waves + wave) * GT, n = *count;
    if (t0 < T && n > 0) {
      u32x4 a[GS / 8];
      load_token<GS>(xg, K, T, t0 + c, a);
      #pragma unroll 1
      for (int p = 0; p < n; p += GT) {
        const int mine = list[p + c];
        const char* const wrow = smem + ((mine >> 5) + 1) * VERSION + (mine & 31) * PITCH_W;
        f32x4 org[4], cur[4];
        dots_tile<GS>(a, wrow, mask, to, cur);
        redo_sums_that_are_not_finite<GS>(xg, K, t0, T, wrow, lane, cur);
        load_org(orgs + (k * waves + wave) * 2 * ORG_HALF + ((mine & 31) + 32 * h) * 16, org);
        const float e = tile_error(cur, org);
        if (h == 0 && p + c < n) part[wave * pairs + mine] += e;
      }
    }
    __syncthreads();
    if (pass + 1 >= rounds && pass + 1 < 2 * rounds) {
      decide(true, pass + 1 - rounds);
      __syncthreads();
    }
  }
  // err_mean < min_errs over the steps that are left: the first minimum below 1e9 wins, NaN never does
  if (tid < GT && r0 + tid < R) {
    const int row = tid;
    float mn = __builtin_inff(), mx = -__builtin_inff();
    for (int ch = 0; ch < TEAM; ++ch) chunk_minmax<IntOp<true, true>>(*(const u32x4*)(smem + row * PITCH_W + ch * 16), mn, mx);
    const float org_max = clip_sym ? nan_max(fabsf(mx), fabsf(mn)) : mx;
    float best = 998244352.0f, bmax = org_max, bmin = mn;                 // bf16(1e9)
    const uint32_t alive = masks[row];
    for (int s = 0; s < n_steps; ++s) {
      if (!((alive >> s) & 1)) continue;
      float e = 0.0f;
      for (int v = 0; v < waves; ++v) e += part[v * pairs + s * GT + row];
      e = rnd<true>(e * (1.0f / (float)T));                              // torch's mean: the sum times an fp32 factor
      const float hi = shrunk(org_max, s, n_grid), lo = clip_sym ? -hi : shrunk(mn, s, n_grid);
      if (e < best || (alive & FOUND)) { best = e; bmax = hi; bmin = lo; }
    }
    const int64_t at = (int64_t)(r0 + row) * G + g;
    best_max[at] = (uint16_t)(f2u(bmax) >> 16);
    best_min[at] = (uint16_t)(f2u(bmin) >> 16);
  }
}

// out[r, g, t] = round( sum_j round(x[t, g*gs + j] * w[r, g*gs + j]) ): the reference's (x * w).sum(dim=-1) of
// auto_clip.py:141,160 on x [1, T, G, gs] and w [R, 1, G, gs] - the product tensor is materialised in the tensors'
// type there (every product rounded), the sum accumulates in fp32 and rounds once.  General in the group size, the
// element type and which tensors are multiplied, so it serves every configuration the MFMA search kernel leaves out
// (activation fake-quant, learnable ranges, other group sizes) and reproduces the reference's rounding sequence.
// With `org` (the same sums for the original weights) the sums are not stored; the kernel goes on to
//   err[r, g] = round( mean_t round( round(out - org)^2 ) )                    (auto_clip.py:163)
// One workgroup: 64 rows x one group, looping over 64-token tiles and 128-column chunks staged in LDS as fp32; thread
// (ty, tx) = (tid / 16, tid % 16) owns rows ty + 16 a and tokens tx + 16 b (a, b = 0..3): 8 LDS reads per 16 products.
constexpr int GD_J = 128, GD_P = GD_J + 1, GD_M = 64;
template <int BF>
__device__ __forceinline__ void gd_stage(float (*S)[GD_P], const void* __restrict__ src, int row0, int nrows, int K,
                                         int64_t col0, int nj, bool vec, int tid) {
  constexpr int N = Vec<BF>::N;
  if (vec) {                                                // 16-byte pieces: K, the group offset and nj are multiples of N
    for (int e = tid; e < GD_M * (GD_J / N); e += 256) {
      const int rr = e / (GD_J / N), c = (e % (GD_J / N)) * N;
      float v[N];
      #pragma unroll
      for (int i = 0; i < N; ++i) v[i] = 0.0f;
      if (rr + row0 < nrows && c < nj) {
        const char* p = (const char*)src + ((int64_t)(row0 + rr) * K + col0 + c) * (BF ? 2 : 4);
        unpack<BF>(*(const u32x4*)p, v);
      }
      #pragma unroll
      for (int i = 0; i < N; ++i) S[rr][c + i] = v[i];
    }
  } else {
    for (int e = tid; e < GD_M * GD_J; e += 256) {
      const int rr = e / GD_J, j = e % GD_J;
      S[rr][j] = (j < nj && row0 + rr < nrows) ? load_scalar<BF>(src, (int64_t)(row0 + rr) * K + col0 + j) : 0.0f;
    }
  }
}

template <int BF>
__global__ __launch_bounds__(256) void group_dots_kernel(const void* __restrict__ x, const void* __restrict__ w, int R, int K,
                                                         int T, int gs, int vec, void* __restrict__ out,
                                                         const void* __restrict__ org, void* __restrict__ err) {
  __shared__ float Xs[GD_M][GD_P], Ws[GD_M][GD_P];
  const int tid = threadIdx.x, G = K / gs, g = blockIdx.y;
  const int r0 = blockIdx.x * GD_M, ty = tid >> 4, tx = tid & 15;
  const bool one_chunk = gs <= GD_J;
  float esum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (one_chunk) gd_stage<BF>(Ws, w, r0, R, K, (int64_t)g * gs, gs, vec, tid);
  for (int t0 = 0; t0 < T; t0 += GD_M) {
    float acc[4][4];
    #pragma unroll
    for (int a = 0; a < 4; ++a)
      #pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = 0.0f;
    for (int j0 = 0; j0 < gs; j0 += GD_J) {
      const int nj = min(GD_J, gs - j0);
      __syncthreads();
      gd_stage<BF>(Xs, x, t0, T, K, (int64_t)g * gs + j0, nj, vec, tid);
      if (!one_chunk) gd_stage<BF>(Ws, w, r0, R, K, (int64_t)g * gs + j0, nj, vec, tid);
      __syncthreads();
      for (int j = 0; j < nj; ++j) {
        float wv[4], xv[4];
        #pragma unroll
        for (int a = 0; a < 4; ++a) wv[a] = Ws[ty + 16 * a][j];
        #pragma unroll
        for (int b = 0; b < 4; ++b) xv[b] = Xs[tx + 16 * b][j];
        #pragma unroll
        for (int a = 0; a < 4; ++a)
          #pragma unroll
          for (int b = 0; b < 4; b += 2) {
            float p0 = xv[b] * wv[a], p1 = xv[b + 1] * wv[a];
            rnd_pair<BF>(p0, p1);
            acc[a][b] += p0;
            acc[a][b + 1] += p1;
          }
      }
    }
    #pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int r = r0 + ty + 16 * a;
      #pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int t = t0 + tx + 16 * b;
        if (r < R && t < T) {
          const int64_t at = ((int64_t)r * G + g) * T + t;
          const float v = rnd_e<BF>(acc[a][b]);
          if (org) {
            const float d = rnd_e<BF>(v - load_scalar<BF>(org, at));
            esum[a] += rnd_e<BF>(d * d);
          } else {
            store_scalar<BF>(out, at, v);
          }
        }
      }
    }
  }
  if (org) {
    #pragma unroll
    for (int a = 0; a < 4; ++a) {
      const float s = team_sum<16>(esum[a]);
      const int r = r0 + ty + 16 * a;
      if (tx == 0 && r < R) store_scalar<BF>(err, (int64_t)r * G + g, rnd_e<BF>(s * (1.0f / (float)T)));
    }
  }
}

}  // namespace

extern "C" {

int lcq_group_dots(const void* x, const void* w, int dtype, int64_t R, int64_t K, int64_t T, int group_size, void* out,
                   const void* org, void* err, void* stream) {
  if (!x || !w || R <= 0 || K <= 0 || T <= 0 || group_size <= 0 || K % group_size != 0) return LCQ_EINVAL;
  if ((org && !err) || (!org && !out)) return LCQ_EINVAL;
  if (R > 0x7fffffff || K > 0x7fffffff || T > 0x7fffffff || K / group_size > 65535) return LCQ_EINVAL;
  if (dtype != LCQ_BF16 && dtype != LCQ_F32 && dtype != LCQ_F16) return LCQ_EDTYPE;
  const int n = dtype == LCQ_F32 ? 4 : 8;
  const int vec = (K % n == 0 && group_size % n == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0) ? 1 : 0;
  const dim3 grid((unsigned)((R + GD_M - 1) / GD_M), (unsigned)(K / group_size));
  hipStream_t st = (hipStream_t)stream;
  if (dtype == LCQ_BF16)
    group_dots_kernel<true><<<grid, dim3(256), 0, st>>>(x, w, (int)R, (int)K, (int)T, group_size, vec, out, org, err);
  else if (dtype == LCQ_F16)
    group_dots_kernel<ROW_F16><<<grid, dim3(256), 0, st>>>(x, w, (int)R, (int)K, (int)T, group_size, vec, out, org, err);
  else
    group_dots_kernel<false><<<grid, dim3(256), 0, st>>>(x, w, (int)R, (int)K, (int)T, group_size, vec, out, org, err);
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_awq_clip_search(const void* w, const void* x, int64_t R, int64_t K, int64_t T, int n_grid, int n_steps,
                        int clip_sym, float qmin, float qmax, int flags, void* best_max, void* best_min, float* errs,
                        void* stream) {
  if (!w || !x || !best_max || !best_min || R <= 0 || K <= 0 || T <= 0) return LCQ_EINVAL;
  if (K % CG != 0 || K > 0x7fffffff / 2 || R > 0x7fffffff || T > 0x7fffffff) return LCQ_EINVAL;
  if (n_grid <= 0 || n_steps <= 0 || n_steps > n_grid) return LCQ_EINVAL;
  if (!(qmax > qmin) || qmax > 256.0f || qmin < -256.0f || (flags & (LCQ_FLAG_STATIC | LCQ_FLAG_NO_ROUND_ZP))) return LCQ_EINVAL;
  if ((((uintptr_t)w | (uintptr_t)x) % 16) != 0) return LCQ_EALIGN;
  const auto op = make_op<IntOp<true, true>>(qmin, qmax, flags, 1.0f, LCQ_CODE_NONE);
  const dim3 grid((unsigned)((R + ROWS_PER_WG - 1) / ROWS_PER_WG), (unsigned)(K / CG));
  awq_clip_kernel<<<grid, dim3(512), 0, (hipStream_t)stream>>>((const uint16_t*)w, (const uint16_t*)x, (int)R, (int)K,
                                                               (int)T, n_grid, n_steps, clip_sym, op, (uint16_t*)best_max,
                                                               (uint16_t*)best_min, errs);
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_clip_search_exact(const void* w, const void* x, int64_t R, int64_t K, int64_t T, int group_size, int n_grid,
                          int n_steps, int clip_sym, float qmin, float qmax, int flags, void* best_max, void* best_min,
                          float* errs, void* stream) {
  if (!w || !x || !best_max || !best_min || R <= 0 || K <= 0 || T <= 0) return LCQ_EINVAL;
  if ((group_size != 32 && group_size != 64 && group_size != 128) || K % group_size != 0) return LCQ_EINVAL;
  if (K > 0x7fffffff / 2 || R > 0x7fffffff || T > 0x7fffffff) return LCQ_EINVAL;
  if (n_grid <= 0 || n_steps <= 0 || n_steps > n_grid || n_steps > LCQ_CLIP_MAX_STEPS) return LCQ_EINVAL;
  if (!(qmax > qmin) || qmax > 256.0f || qmin < -256.0f || (flags & (LCQ_FLAG_STATIC | LCQ_FLAG_NO_ROUND_ZP))) return LCQ_EINVAL;
  if ((((uintptr_t)w | (uintptr_t)x) % 16) != 0) return LCQ_EALIGN;
  const auto op = make_op<IntOp<true, true>>(qmin, qmax, flags, 1.0f, LCQ_CODE_NONE);
  const int64_t grid = ((R + GT - 1) / GT) * (K / group_size);
  if (grid > 0x7fffffff) return LCQ_EINVAL;
  // one wave per 32 tokens up to eight (two per SIMD: one wave's conversions run under the other's matrix instructions)
  const int waves = T > 4 * GT ? 8 : (T > 2 * GT ? 4 : 2);
  hipStream_t st = (hipStream_t)stream;
  const int rounds = (int)((T + waves * GT - 1) / (waves * GT));
  constexpr size_t LDS = 160 * 1024;
  #define LCQ_CLIP_LAUNCH(KERNEL, BYTES, ...) do { \
    /* on every call, for it belongs to the current device; the same value always, for another thread may set it too */ \
    if (BYTES > 64 * 1024 && hipFuncSetAttribute((const void*)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) != hipSuccess) return LCQ_ELAUNCH; \
    KERNEL<<<dim3((unsigned)grid), dim3(64 * waves), BYTES, st>>>((const uint16_t*)w, (const uint16_t*)x, (int)R, (int)K, (int)T, n_grid, \
        n_steps, clip_sym, op, (uint16_t*)best_max, (uint16_t*)best_min __VA_ARGS__); } while (0)
  // without errors, and with few enough tokens and steps that the original sums and the bounds of all steps fit LDS (T <= 512,
  // 10 steps at groups of 128): only the steps that may win
  #define LCQ_CLIP(GS) do { \
    const size_t pruned = clip_pruned_lds<GS>(n_steps, waves, rounds < 2 ? rounds : 2); \
    if (!errs && rounds <= 2 && pruned <= LDS) LCQ_CLIP_LAUNCH(clip_search_pruned_kernel<GS>, pruned); \
    else { \
      const size_t lds = (size_t)(n_steps + 1) * GT * gd_pitch<GS>() + (size_t)waves * n_steps * GT * 4; \
      LCQ_CLIP_LAUNCH(clip_search_kernel<GS>, lds, , errs); } } while (0)
  if (group_size == 128) LCQ_CLIP(128); else if (group_size == 64) LCQ_CLIP(64); else LCQ_CLIP(32);
  #undef LCQ_CLIP
  #undef LCQ_CLIP_LAUNCH
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_clamp_groups(const void* w, int dtype, int64_t R, int64_t K, int group_size, const void* lo, const void* hi,
                     void* out, void* stream) {
  if (!w || !lo || !hi || !out || R <= 0 || K <= 0 || group_size <= 0 || K % group_size != 0) return LCQ_EINVAL;
  if (dtype != LCQ_F32 && dtype != LCQ_BF16 && dtype != LCQ_F16) return LCQ_EDTYPE;
  const int n = dtype == LCQ_F32 ? 4 : 8;
  hipStream_t st = (hipStream_t)stream;
  if (group_size % n != 0 || (((uintptr_t)w | (uintptr_t)out) % 16) != 0) {
    int64_t grid = (R * K + 255) / 256;
    if (grid > 262144) grid = 262144;
    if (dtype == LCQ_BF16) clamp_groups_scalar_kernel<true><<<dim3((unsigned)grid), dim3(256), 0, st>>>(w, R * K, group_size, lo, hi, out);
    else if (dtype == LCQ_F16) clamp_groups_scalar_kernel<ROW_F16><<<dim3((unsigned)grid), dim3(256), 0, st>>>(w, R * K, group_size, lo, hi, out);
    else clamp_groups_scalar_kernel<false><<<dim3((unsigned)grid), dim3(256), 0, st>>>(w, R * K, group_size, lo, hi, out);
    LCQ_CHECK_LAUNCH();
    return LCQ_OK;
  }
  const int64_t nchunks = R * K / n;
  int64_t grid = (nchunks + 255) / 256;
  if (grid > 262144) grid = 262144;
  if (dtype == LCQ_BF16) clamp_groups_kernel<true><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const u32x4*)w, nchunks, group_size / n, lo, hi, (u32x4*)out);
  else if (dtype == LCQ_F16) clamp_groups_kernel<ROW_F16><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const u32x4*)w, nchunks, group_size / n, lo, hi, (u32x4*)out);
  else clamp_groups_kernel<false><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const u32x4*)w, nchunks, group_size / n, lo, hi, (u32x4*)out);
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

}  // extern "C"
