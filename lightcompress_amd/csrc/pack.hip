// int4 / int8 code packing for gfx950.
//
//  * lcq_pack_ct      : compressed-tensors "pack-quantized" layout used by the
//                       vLLM / SGLang / LightLLM exporters
//                       (VllmRealQuantLinear.pack, module_utils.py:929-955):
//                       u = uint8(code + 2^(bits-1)); word j of a row holds
//                       u[pf*j + i] << (bits*i), pf = 32 / bits, tail zero-padded.
//                       The reference round-trips through numpy on the host.
//  * lcq_pack_awq     : AutoAWQ / MLC "gemm_pack" layout
//                       (AutoawqRealQuantLinear.gemm_pack, module_utils.py:1097-1158):
//                       iw[r,k] = int(round((w[r,k] + z*s) / s)) with fp16 scales,
//                       NOT clamped; qweight[k, c] = OR_i iw[8c+order[i], k] << 4i,
//                       order = 0,2,4,6,1,3,5,7; qzeros likewise; scales -> fp16 [K/g, R].
//                       The reference loops over K columns and R/8 x 8 nibbles in Python.
//  * lcq_quant_pack_awq: the same with the scales and zero points found on the way (real_quant_weight_dynamic,
//                       quant.py:915-952, whose codes this layout does not use).
// Byte shuffles: one read of the codes / weights, one write of the packed words.
#include "intop.h"

namespace {

template <typename CodeT>
__global__ __launch_bounds__(256) void pack_ct_kernel(const CodeT* __restrict__ codes, int64_t R, int64_t K, int bits,
                                                      int64_t words_per_row, uint32_t* __restrict__ packed) {
  const int pf = 32 / bits;
  const int offset = 1 << (bits - 1);
  const int64_t total = R * words_per_row;
  for (int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x; w < total; w += (int64_t)gridDim.x * 256) {
    const int64_t r = w / words_per_row, j = w % words_per_row;
    const CodeT* src = codes + r * K + j * pf;
    uint32_t acc = 0;
    if (sizeof(CodeT) == 4 && pf == 8 && (j + 1) * pf <= K && (K % 4) == 0) {
      const u32x4 a = *(const u32x4*)src, b = *(const u32x4*)(src + 4);
      #pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc |= ((a[i] + (uint32_t)offset) & 0xffu) << (4 * i);
        acc |= ((b[i] + (uint32_t)offset) & 0xffu) << (4 * (i + 4));
      }
    } else {
      for (int i = 0; i < pf; ++i) {
        const int64_t col = j * pf + i;
        if (col < K) acc |= (((uint32_t)(int32_t)src[i] + (uint32_t)offset) & 0xffu) << (bits * i);
      }
    }
    packed[w] = acc;
  }
}

template <int WDT> __device__ __forceinline__ float load_w(const void* w, int64_t i);
template <> __device__ __forceinline__ float load_w<LCQ_F32>(const void* w, int64_t i) { return ((const float*)w)[i]; }
template <> __device__ __forceinline__ float load_w<LCQ_BF16>(const void* w, int64_t i) { return u2f((uint32_t)((const uint16_t*)w)[i] << 16); }
template <> __device__ __forceinline__ float load_w<LCQ_F16>(const void* w, int64_t i) { return (float)((const _Float16*)w)[i]; }

// Eight rows x eight columns per lane: the eight nibbles of a word (one column, rows 8c .. 8c+7) meet in one lane, so the words
// are built in registers; GS / 8 lanes hold a group's columns and reduce its ranges (DYN) over their team, then each works out
// the parameters of one of the rows and leaves them in LDS for the others (worked out by every lane they are a third of all
// instructions).  A workgroup of 512 lanes owns 8 * 512 / TEAM rows of one group; its words go through LDS so that they leave
// as whole lines.
// (x + z*s) / s: the product with the reciprocal and one residual step.  That is the correctly rounded quotient: the residual is
// exact, the step leaves an error of 2^-21 ulp, and a quotient by a number of 11 significant bits (s is fp16) is never closer
// than 2^-12 ulp to a rounding midpoint.  (A guard and a division where it fails, as in the quantizers, would run in every wave
// here: bf16 weights hit half-integers exactly, x = s / 2 is one.)  v + 1.5 * 2^23 leaves its integer in the low mantissa bits,
// which are shifted to the nibble and added up (the bias is linear modulo 2^32 and comes off once per word); integers outside
// 0 .. 15 are ORed unmasked as in the reference.
// 11008 x 4096 bf16 in groups of 128: the range, the codes nobody reads and a packing pass with a division and a 2-byte load
// per element took 43 + 139 us; this takes 27, of which 19 are the bytes at the rate of a plain stream (42 with a guard and
// divisions in place of the residual step, 15 against 24 vector instructions per element).
template <int WDT, int GS, bool DYN>
__global__ __launch_bounds__(512) void pack_awq_team_kernel(const void* __restrict__ w, const void* __restrict__ scales,
                                                            const int32_t* __restrict__ zeros, int64_t R, int64_t K,
                                                            lcq::IntOp<WDT, true> op, uint32_t* __restrict__ qweight,
                                                            _Float16* __restrict__ scales_out, uint32_t* __restrict__ qzeros) {
  using namespace lcq;
  constexpr int TEAM = GS / 8, OCT = 512 / TEAM, CPL = 8 / Vec<WDT>::N;     // row octets per workgroup; 16-byte chunks per lane and row
  constexpr int ROWS = (8 + TEAM - 1) / TEAM;                // rows whose parameters a lane works out
  __shared__ uint32_t words[GS][OCT + 1];
  __shared__ f32x4 prm[OCT][8];                              // fp16 scale, z * scale, 1 / scale, zero point
  const int t = threadIdx.x % TEAM, oct = threadIdx.x / TEAM;
  const int64_t g = blockIdx.x, G = K / GS, c0 = (int64_t)blockIdx.y * OCT;
  const bool ok = c0 + oct < R / 8;
  const int64_t c = ok ? c0 + oct : R / 8 - 1;               // surplus teams repeat the last octet and store nothing
  u32x4 raw[8][CPL];
  #pragma unroll
  for (int i = 0; i < 8; ++i)
    #pragma unroll
    for (int k = 0; k < CPL; ++k)
      raw[i][k] = __builtin_nontemporal_load((const u32x4*)((const char*)w + ((8 * c + i) * K + g * GS + 8 * t) * (WDT ? 2 : 4)) + k);
  float mn[ROWS], mx[ROWS];                                  // of rows t % 8 (, t + 4)
  if constexpr (DYN) {
    #pragma unroll
    for (int i = 0; i < 8; ++i) {
      float lo = __builtin_inff(), hi = -__builtin_inff();
      #pragma unroll
      for (int k = 0; k < CPL; ++k) chunk_minmax<IntOp<WDT, true>>(raw[i][k], lo, hi);
      team_range<TEAM>(lo, hi);
      #pragma unroll
      for (int j = 0; j < ROWS; ++j)
        if ((t + j * TEAM) % 8 == i) { mn[j] = lo; mx[j] = hi; }
    }
  }
  #pragma unroll
  for (int j = 0; j < ROWS; ++j) {
    const int i = (t + j * TEAM) % 8;
    float s, z;
    if constexpr (DYN) {
      const IntRow p = op.make(mn[j], mx[j]);
      s = p.s; z = (float)(int32_t)p.z;
    } else {
      s = load_scalar<WDT>(scales, (8 * c + i) * G + g);
      z = (float)zeros[(8 * c + i) * G + g];
    }
    const float s16 = f16_round(s);
    prm[oct][i] = f32x4{s16, f16_round(z * s16), __builtin_amdgcn_rcpf(s16), z};   // (16 lanes: written twice, the same)
  }
  __syncthreads();
  uint32_t acc[8] = {0, 0, 0, 0, 0, 0, 0, 0}, odd[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  #pragma unroll
  for (int i = 0; i < 8; ++i) {
    const f32x4 p = prm[oct][i];
    const float s16 = p[0], sz = p[1], r = p[2];
    const int nib = 4 * ((i & 1) ? 4 + i / 2 : i / 2);       // order 0,2,4,6,1,3,5,7 read backwards
    float x[8], tq[8], v[8], lo = __builtin_inff(), hi = -__builtin_inff();
    #pragma unroll
    for (int k = 0; k < CPL; ++k) unpack<WDT>(raw[i][k], x + k * Vec<WDT>::N);
    #pragma unroll
    for (int k = 0; k < 8; ++k) {
      // bf16 / fp32 next to fp16 promote to fp32; fp16 tensors round the sum and the quotient
      x[k] = WDT == LCQ_F16 ? rnd<ROW_F16>(x[k] + sz) : x[k] + sz;
      const float q = x[k] * r;
      tq[k] = __builtin_fmaf(__builtin_fmaf(-s16, q, x[k]), r, q);
    }
    if constexpr (WDT == LCQ_F16)
      #pragma unroll
      for (int k = 0; k < 8; k += 2) rnd_pair<ROW_F16>(tq[k], tq[k + 1]);
    #pragma unroll
    for (int k = 0; k < 8; k += 2) {
      v[k] = tq[k] + RINT_BIAS; v[k + 1] = tq[k + 1] + RINT_BIAS;
      lo = nan_min(nan_min(lo, tq[k]), tq[k + 1]);
      hi = nan_max(nan_max(hi, tq[k]), tq[k + 1]);
    }
    if (__builtin_expect(!(lo > -0.5f && hi < 15.5f && s16 > 1e-7f), 0)) {
      const bool divide = !(lo > -1024.0f && hi < 1024.0f && s16 > 1e-7f);
      #pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (divide) {
          tq[k] = x[k] / s16;
          if constexpr (WDT == LCQ_F16) tq[k] = rnd<ROW_F16>(tq[k]);
        }
        odd[k] |= (uint32_t)(int32_t)rintf(tq[k]) << nib;
        v[k] = RINT_BIAS;
      }
    }
    #pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = (f2u(v[k]) << nib) + acc[k];
  }
  #pragma unroll
  for (int k = 0; k < 8; ++k) words[8 * t + k][oct] = (acc[k] - (uint32_t)RINT_BIAS_BITS * 0x11111111u) | odd[k];
  if (t == 0 && ok) {
    uint32_t h[4], zacc = 0;
    #pragma unroll
    for (int i = 0; i < 4; ++i)
      h[i] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)prm[oct][2 * i][0]) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)prm[oct][2 * i + 1][0]) << 16);
    #pragma unroll
    for (int i = 0; i < 8; ++i) zacc |= (uint32_t)(int32_t)prm[oct][i][3] << (4 * ((i & 1) ? 4 + i / 2 : i / 2));
    *(u32x4*)(scales_out + g * R + 8 * c) = u32x4{h[0], h[1], h[2], h[3]};
    qzeros[g * (R / 8) + c] = zacc;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < GS * OCT; e += 512) {
    const int k = e / OCT, o = e % OCT;
    if (c0 + o < R / 8) qweight[(g * GS + k) * (R / 8) + c0 + o] = words[k][o];
  }
}

constexpr int AWQ_TR = 256;   // output channels per tile
constexpr int AWQ_TK = 32;    // input channels per tile
constexpr int AWQ_PITCH = AWQ_TR + 1;

// one tile: iw for AWQ_TR rows x AWQ_TK columns through LDS, then R/8 words per column
template <int WDT>
__global__ __launch_bounds__(256) void pack_awq_kernel(const void* __restrict__ w, const void* __restrict__ scales,
                                                       const int32_t* __restrict__ zeros, int64_t R, int64_t K, int g,
                                                       int32_t* __restrict__ qweight) {
  extern __shared__ int32_t tile[];                         // [AWQ_TK][AWQ_PITCH]
  const int64_t r0 = (int64_t)blockIdx.y * AWQ_TR, k0 = (int64_t)blockIdx.x * AWQ_TK;
  const int64_t G = K / g;
  const int tk = threadIdx.x & 31, tr = threadIdx.x >> 5;
  for (int rr = tr; rr < AWQ_TR; rr += 8) {
    const int64_t r = r0 + rr, k = k0 + tk;
    int32_t iw = 0;
    if (r < R && k < K) {
      const int64_t gi = r * G + k / g;
      const float s16 = f16_round(load_w<WDT>(scales, gi));            // scales.to(float16)
      const float sz = f16_round((float)zeros[gi] * s16);              // zeros * scales, fp16 result
      const float x = load_w<WDT>(w, r * K + k);
      float t;
      if (WDT == LCQ_F16) t = f16_round(f16_round(x + sz) / s16);      // all-fp16 tensor ops
      else t = (x + sz) / s16;                                         // promoted to fp32
      iw = (int32_t)rintf(t);
    }
    tile[tk * AWQ_PITCH + rr] = iw;
  }
  __syncthreads();
  const int order[8] = {0, 2, 4, 6, 1, 3, 5, 7};
  const int c = threadIdx.x & 31;
  for (int kk = threadIdx.x >> 5; kk < AWQ_TK; kk += 8) {
    const int64_t k = k0 + kk;
    const int64_t cg = r0 / 8 + c;
    if (k < K && cg < R / 8) {
      uint32_t acc = 0;
      #pragma unroll
      for (int i = 0; i < 8; ++i) acc |= (uint32_t)tile[kk * AWQ_PITCH + 8 * c + order[i]] << (4 * i);
      qweight[k * (R / 8) + cg] = (int32_t)acc;
    }
  }
}

template <int WDT>
__global__ __launch_bounds__(256) void pack_awq_qparams_kernel(const void* __restrict__ scales, const int32_t* __restrict__ zeros,
                                                               int64_t R, int64_t G, uint16_t* __restrict__ scales_out,
                                                               int32_t* __restrict__ qzeros) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < G * R) {                                          // scales.t().contiguous().to(float16)
    const int64_t gi = i / R, r = i % R;
    const _Float16 h = (_Float16)load_w<WDT>(scales, r * G + gi);
    scales_out[i] = __builtin_bit_cast(uint16_t, h);
  }
  if (i < G * (R / 8)) {
    const int order[8] = {0, 2, 4, 6, 1, 3, 5, 7};
    const int64_t gi = i / (R / 8), c = i % (R / 8);
    uint32_t acc = 0;
    #pragma unroll
    for (int j = 0; j < 8; ++j) acc |= (uint32_t)zeros[(8 * c + order[j]) * G + gi] << (4 * j);
    qzeros[i] = (int32_t)acc;
  }
}

bool awq_team_applies(const void* w, int64_t R, int64_t K, int gs, const void* s16) {
  return (gs == 32 || gs == 64 || gs == 128) && R % 8 == 0 && K % gs == 0 && R <= (int64_t)65535 * 256 && K <= 0x7fffffff && ((uintptr_t)w % 16) == 0 && ((uintptr_t)s16 % 16) == 0;
}
template <int WDT, bool DYN>
void launch_awq_team(const void* w, const void* scales, const int32_t* zeros, int64_t R, int64_t K, int gs, float qmin, float qmax,
                     int32_t* qweight, void* s16, int32_t* qzeros, hipStream_t st) {
  const auto op = lcq::make_op<lcq::IntOp<WDT, true>>(qmin, qmax, 0, 1.0f, LCQ_CODE_NONE);
  const int64_t octs = 512 / (gs / 8);
  const dim3 grid((unsigned)(K / gs), (unsigned)((R / 8 + octs - 1) / octs));        // neighbouring workgroups read the same rows
  #define LCQ_AWQ(GS) pack_awq_team_kernel<WDT, GS, DYN><<<grid, dim3(512), 0, st>>>(w, scales, zeros, R, K, op, (uint32_t*)qweight, (_Float16*)s16, (uint32_t*)qzeros)
  if (gs == 128) LCQ_AWQ(128); else if (gs == 64) LCQ_AWQ(64); else LCQ_AWQ(32);
  #undef LCQ_AWQ
}

}  // namespace

extern "C" {

int lcq_pack_ct(const void* codes, int code_dtype, int64_t R, int64_t K, int bits, int32_t* packed, void* stream) {
  if (!codes || !packed || R < 0 || K <= 0) return LCQ_EINVAL;
  if (bits != 4 && bits != 8 && bits != 2 && bits != 16) return LCQ_EINVAL;
  if (R == 0) return LCQ_OK;
  const int pf = 32 / bits;
  const int64_t wpr = (K + pf - 1) / pf;
  int64_t grid = (R * wpr + 255) / 256;
  if (grid > 1 << 20) grid = 1 << 20;
  hipStream_t st = (hipStream_t)stream;
  if (code_dtype == LCQ_CODE_I32) pack_ct_kernel<int32_t><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const int32_t*)codes, R, K, bits, wpr, (uint32_t*)packed);
  else if (code_dtype == LCQ_CODE_I8) pack_ct_kernel<int8_t><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const int8_t*)codes, R, K, bits, wpr, (uint32_t*)packed);
  else if (code_dtype == LCQ_CODE_U8) pack_ct_kernel<uint8_t><<<dim3((unsigned)grid), dim3(256), 0, st>>>((const uint8_t*)codes, R, K, bits, wpr, (uint32_t*)packed);
  else return LCQ_EDTYPE;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_quant_pack_awq(const void* w, int dtype, int64_t R, int64_t K, int group_size, float qmin, float qmax,
                       int32_t* qweight, void* scales_f16_out, int32_t* qzeros, void* stream) {
  if (!w || !qweight || !scales_f16_out || !qzeros || R <= 0 || K <= 0) return LCQ_EINVAL;
  if (!awq_team_applies(w, R, K, group_size, scales_f16_out) || R % 32 != 0) return LCQ_EINVAL;
  if (!(qmax > qmin) || qmax > 256.0f || qmin < -256.0f) return LCQ_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == LCQ_F32) launch_awq_team<LCQ_F32, true>(w, nullptr, nullptr, R, K, group_size, qmin, qmax, qweight, scales_f16_out, qzeros, st);
  else if (dtype == LCQ_BF16) launch_awq_team<LCQ_BF16, true>(w, nullptr, nullptr, R, K, group_size, qmin, qmax, qweight, scales_f16_out, qzeros, st);
  else if (dtype == LCQ_F16) launch_awq_team<LCQ_F16, true>(w, nullptr, nullptr, R, K, group_size, qmin, qmax, qweight, scales_f16_out, qzeros, st);
  else return LCQ_EDTYPE;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_pack_awq(const void* w, int dtype, const void* scales, const int32_t* zeros, int64_t R, int64_t K, int group_size,
                 int32_t* qweight, void* scales_f16_out, int32_t* qzeros, void* stream) {
  if (!w || !scales || !zeros || !qweight || !scales_f16_out || !qzeros) return LCQ_EINVAL;
  if (R <= 0 || K <= 0 || group_size <= 0 || K % group_size != 0 || R % 32 != 0) return LCQ_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (awq_team_applies(w, R, K, group_size, scales_f16_out)) {
    if (dtype == LCQ_F32) launch_awq_team<LCQ_F32, false>(w, scales, zeros, R, K, group_size, 0, 15, qweight, scales_f16_out, qzeros, st);
    else if (dtype == LCQ_BF16) launch_awq_team<LCQ_BF16, false>(w, scales, zeros, R, K, group_size, 0, 15, qweight, scales_f16_out, qzeros, st);
    else if (dtype == LCQ_F16) launch_awq_team<LCQ_F16, false>(w, scales, zeros, R, K, group_size, 0, 15, qweight, scales_f16_out, qzeros, st);
    else return LCQ_EDTYPE;
    LCQ_CHECK_LAUNCH();
    return LCQ_OK;
  }
  const dim3 grid((unsigned)((K + AWQ_TK - 1) / AWQ_TK), (unsigned)((R + AWQ_TR - 1) / AWQ_TR));
  const size_t lds = (size_t)AWQ_TK * AWQ_PITCH * sizeof(int32_t);
  const int64_t G = K / group_size;
  const int64_t n = G * R;
  const unsigned g2 = (unsigned)((n + 255) / 256);
  if (dtype == LCQ_F32) {
    pack_awq_kernel<LCQ_F32><<<grid, dim3(256), lds, st>>>(w, scales, zeros, R, K, group_size, qweight);
    pack_awq_qparams_kernel<LCQ_F32><<<dim3(g2), dim3(256), 0, st>>>(scales, zeros, R, G, (uint16_t*)scales_f16_out, qzeros);
  } else if (dtype == LCQ_BF16) {
    pack_awq_kernel<LCQ_BF16><<<grid, dim3(256), lds, st>>>(w, scales, zeros, R, K, group_size, qweight);
    pack_awq_qparams_kernel<LCQ_BF16><<<dim3(g2), dim3(256), 0, st>>>(scales, zeros, R, G, (uint16_t*)scales_f16_out, qzeros);
  } else if (dtype == LCQ_F16) {
    pack_awq_kernel<LCQ_F16><<<grid, dim3(256), lds, st>>>(w, scales, zeros, R, K, group_size, qweight);
    pack_awq_qparams_kernel<LCQ_F16><<<dim3(g2), dim3(256), 0, st>>>(scales, zeros, R, G, (uint16_t*)scales_f16_out, qzeros);
  } else return LCQ_EDTYPE;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

}  // extern "C"
