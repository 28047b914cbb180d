// GPTQ lazy-batch column loop for gfx950.
//
// Replaces GPTQ.weight_transform (llmc/compression/quantization/gptq.py:198-244)
// together with search_column_qparams (:358-366):
//   for each block of `blocksize` columns:
//     for each column i:  (group boundary -> refresh scale/zero from W[:, i:i+g])
//        q = quant_dequant(w);  tmp[:, i] = w;  Losses[:, i] = (w-q)^2 / (2 d^2)
//        err = (w-q)/d;  W1[:, i:] -= err (x) Hinv1[i, i:];  Err1[:, i] = err
//     W[:, i2:] -= Err1 @ Hinv[i1:i2, i2:]
// The reference issues >= 5 tiny launches per column; here one launch runs the
// 128 sequential columns of a block and fp32-MFMA launches apply the deferred
// update.  The update entry point takes any (contraction range, column range),
// so the host can defer a second time: update only the next few blocks after
// every block and everything behind them once per 1024 columns, which reads
// and writes the bulk of W eight times less often.
//
// Block kernel layout: 16 lanes share one weight row, lane t starts with columns 8t..8t+7 of the
// block in registers; a wave therefore carries 4 rows and a 256-thread workgroup 16.  Every lane
// evaluates the quantizer on its own register (same instruction stream), the owner's error is
// broadcast inside the 16-lane team, and all lanes apply the rank-1 update to their 8 columns from
// the Hinv block held in LDS.  Per-group min/max are 16-lane DPP butterflies.
//
// With R = 4096 rows the kernel has one wave per SIMD on the whole chip, so its run time is the
// length of the per-column dependency chain times 128.  That chain is kept to about ten VALU
// operations:
//  * the quotient w/s goes through the group's reciprocal; an octet (8 columns) in which an owner
//    comes within 2^-11 of a rounding boundary is replayed with true divisions;
//  * (w-q)/d goes through a reciprocal of the diagonal prepared in LDS (at most one ulp from the
//    quotient; it only perturbs later columns, never the rounding of this one);
//  * the registers rotate by one lane after every octet, so the owner is always lane 0 and the
//    broadcast of the error is a DPP row_share:0 instead of an LDS permute, while the loop over
//    octets stays rolled (fully unrolled it is 126 KB of straight-line code that runs at
//    instruction-fetch speed);
//  * the octet's rows of U are fetched from LDS ahead of the chain, and because U is stored zero
//    below the diagonal no update needs a mask;
//  * tmp / (w-q) / err rotate along and are stored once at the end, 32 bytes per lane: a store
//    inside the loop would make every later wait on a load cover it too.
#include <type_traits>

#include "gemm_f32.h"
#include "gemm_s3p.h"
#include "launch_rules.h"
#include "lcq_internal.h"

namespace {
using namespace lcq;

constexpr int BS = 128;          // columns per block (lazy batch)
// Hinv1 in LDS: a row holds, for each of the 16 lanes of a team, the first four of the lane's eight columns at
// float 4 t and the other four at UH + 4 t, so the two 16-byte reads of a team are each one contiguous run (no bank
// conflicts); the second half starts 4 floats past a multiple of 64 so that a wave's 16-byte stores, which alternate
// between the halves while the block is loaded, do not collide either.
constexpr int UH = 68;           // offset of the second halves inside a row
constexpr int UP = 136;          // row pitch (floats)
__device__ __forceinline__ int us_col(int c) { return ((c & 4) ? UH : 0) + 4 * (c >> 3) + (c & 3); }

struct LoopArgs {
  float* W; float* tmp; float* Losses; float* Err; const float* U;
  const float* W0;      // the weights before the loop, or null: Err then receives q - W0 instead of the errors (see lcq_chol_block_factor)
  float* scales; float* zeros; const int* gidx;
  long long R; int K, Kq, i1, count, g, G, ldErr;      // Kq: columns that are quantized (K unless outlier columns are kept)
  float qmin, qmax;
  int sym, is_static, aligned;
  int nrz;              // round_zp=False: un-rounded zero point inside the rounding, scale clamped at 1e-9 (quant.py:556-557, 702-706)
};

// DPP moves inside every 16-lane row: the value of lane 0, and the value of the next lane (rotation by one)
__device__ __forceinline__ float row16_first(float v) {
  return u2f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f2u(v), 0x150, 0xf, 0xf, true));          // row_share:0
}
__device__ __forceinline__ float row16_next(float v) {
  return u2f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f2u(v), 0x12F, 0xf, 0xf, true));          // row_ror:15
}

struct ColQ {           // quantizer of the column being processed
  float s, z, r;        // scale, zero point, 1/s
  float lo, hi;         // qmin - z, qmax - z: clamp(round(t) + z, qmin, qmax) - z == clamp(round(t), lo, hi) for integral z
  bool fast;            // x * r may stand for x / s (guarded) and lo / hi are exact
};
__device__ __forceinline__ ColQ make_colq(float s, float z, float qmin, float qmax, bool nrz = false) {
  ColQ q;
  q.s = s; q.z = z;
  q.r = __builtin_amdgcn_rcpf(s);
  q.lo = qmin - z; q.hi = qmax - z;
  const float a = fabsf(s);
  q.fast = (a > 8.6736174e-19f) & (a < 1.1529215e18f) & (rintf(z) == z) & (fabsf(z) <= 512.0f) & (fabsf(qmin) <= 512.0f) &
           (fabsf(qmax) <= 512.0f) & !nrz;
  return q;
}

// scale and zero point of a group with this range
__device__ __forceinline__ void group_params(const LoopArgs& a, float mn, float mx, float& s, float& z) {
  if (a.sym) {
    s = fmaxf(fmaxf(fabsf(mx), fabsf(mn)), 1e-5f) / a.qmax;
    z = 0.0f;
  } else {
    s = fmaxf(mx - mn, 1e-5f) / (a.qmax - a.qmin);
    z = a.nrz ? a.qmin - mn / s : fminf(fmaxf(a.qmin - rintf(mn / s), a.qmin), a.qmax);
  }
}

// A group opens at column idx: scale and zero point from the range of W[row, idx : min(idx+g, K)] as it is in
// memory now -- trailing updates of earlier blocks applied, this block's own updates not (gptq.py:216-222 reads
// W, not W1).
// `held`: the team's registers when they are exactly that range (group = block, nothing updated yet).
__device__ __forceinline__ ColQ open_group(const LoopArgs& a, int idx, int lane, long long row, bool row_ok, long long rbase,
                                           const float (&held)[8], bool use_held) {
  const int end = min(idx + a.g, a.Kq);
  float mn = __builtin_inff(), mx = -__builtin_inff();
  if (use_held) {
    #pragma unroll
    for (int c = 0; c < 8; ++c) { mn = nan_min(mn, held[c]); mx = nan_max(mx, held[c]); }      // NaN-propagating like torch.amin / amax
  } else {
    for (int col = idx + lane; col < end; col += 16) {
      const float v = a.W[rbase + col];
      mn = nan_min(mn, v); mx = nan_max(mx, v);
    }
  }
  mn = team_reduce<16, false>(mn);
  mx = team_reduce<16, true>(mx);
  float s, z;
  group_params(a, mn, mx, s, z);
  if (row_ok && lane == 0) {
    a.scales[row * a.G + idx / a.g] = s;
    if (!a.sym) a.zeros[row * a.G + idx / a.g] = z;
  }
  return make_colq(s, z, a.qmin, a.qmax, a.nrz);
}

// STATIC: scales / zero points are given (per group, or per column through gidx).  OCT: every group starts on
// a multiple of 8 columns, so groups open only between octets and the 8 columns of an octet are straight-line code.
// RW rows per workgroup (16 lanes each): 16, or 32 for launches of many rows (one copy of Hinv1 in LDS then serves
// eight waves, and two such workgroups put four waves on every SIMD instead of two).
template <bool STATIC, bool OCT, int RW>
__global__ __launch_bounds__(16 * RW) void gptq_block_kernel(LoopArgs a) {
  constexpr int NT = 16 * RW;                    // threads
  constexpr int ROWS_PER_WG = RW;
  constexpr int NP = OCT ? 16 : BS;              // parameter slots of a row: one per octet, or one per column
  __shared__ float Us[BS * UP];                  // Hinv1 = U[i1:i2, i1:i2] above the diagonal, zero everywhere else (us_col layout)
  __shared__ float Rd[BS];                       // 1 / U[i, i]
  __shared__ float Dg[BS];                       // U[i, i]
  __shared__ float Ps[STATIC ? 1 : ROWS_PER_WG * NP], Pz[STATIC ? 1 : ROWS_PER_WG * NP];   // scale, zero point in force
  const int tid = threadIdx.x;
  // full block and 16-byte aligned rows (the entry point checks the base pointers): vector loads and stores
  const bool vec = (a.count == BS) && (a.K % 4 == 0) && (a.i1 % 4 == 0) && a.aligned;
  // The diagonal is zero in LDS as well: a column's own update would only turn it into its quantized value, which
  // nothing reads.  Left alone, the register of a finished column keeps the weight as it was when the column was
  // quantized, which is the `tmp` output, and (w - q), err and the loss are recomputed from it once, after the loop.
  if (vec) {
    // all 16 loads of the thread in flight at once: one after the other they are 16 memory latencies,
    // which used to be most of the kernel's run time
    constexpr int NL = BS * BS / 4 / NT;
    f32x4 v[NL];
    #pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int e = tid + NT * j, r = e >> 5, c = (e & 31) * 4;
      v[j] = *(const f32x4*)(a.U + (long long)(a.i1 + r) * a.K + a.i1 + c);
    }
    #pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int e = tid + NT * j, r = e >> 5, c = (e & 31) * 4;
      #pragma unroll
      for (int k = 0; k < 4; ++k) if (c + k <= r) v[j][k] = 0.0f;
      *(f32x4*)(Us + r * UP + us_col(c)) = v[j];
    }
  } else {
    for (int e = tid; e < BS * BS / 4; e += NT) {
      const int r = (e * 4) / BS, c = (e * 4) % BS;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (r < a.count) {
        const float* p = a.U + (long long)(a.i1 + r) * a.K + a.i1 + c;
        #pragma unroll
        for (int k = 0; k < 4; ++k) if (c + k < a.count && c + k > r) v[k] = p[k];
      }
      *(f32x4*)(Us + r * UP + us_col(c)) = v;
    }
  }
  if (tid < BS) {
    const float d = (tid < a.count) ? a.U[(long long)(a.i1 + tid) * a.K + a.i1 + tid] : 1.0f;
    Dg[tid] = d;
    Rd[tid] = (tid < a.count) ? 1.0f / d : 0.0f;
  }

  const int lane = tid & 15;                     // physical lane inside the row's team
  const int prow = tid >> 4;                     // the team's row inside the workgroup
  const long long row = (long long)blockIdx.x * ROWS_PER_WG + prow;
  const bool row_ok = row < a.R;
  const long long rbase = (row_ok ? row : 0) * a.K;

  // lane t starts with columns 8t..8t+7 (and, for static groups, their scales and zero points)
  float w[8], ss[8], zz[8];
  if (vec) {                                     // rows of W / tmp / Losses are 16-byte aligned at the block's columns
    const f32x4 lo4 = *(const f32x4*)(a.W + rbase + a.i1 + 8 * lane), hi4 = *(const f32x4*)(a.W + rbase + a.i1 + 8 * lane + 4);
    #pragma unroll
    for (int k = 0; k < 4; ++k) { w[k] = row_ok ? lo4[k] : 0.0f; w[4 + k] = row_ok ? hi4[k] : 0.0f; }
  }
  #pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int col = 8 * lane + c;
    if (!vec) w[c] = (row_ok && col < a.count) ? a.W[rbase + a.i1 + col] : 0.0f;
    ss[c] = 1.0f; zz[c] = 0.0f;
    if (STATIC && col < a.count) {
      const int idx = a.i1 + col;
      const int gi = a.gidx ? a.gidx[idx] : (a.g > 0 ? idx / a.g : 0);
      ss[c] = a.scales[(row_ok ? row : 0) * a.G + gi];
      zz[c] = a.sym ? 0.0f : a.zeros[(row_ok ? row : 0) * a.G + gi];
    }
  }
  ColQ q = make_colq(1.0f, 0.0f, a.qmin, a.qmax);
  int nextb = 0x7fffffff;
  if (!STATIC) {
    nextb = (a.i1 + a.g - 1) / a.g * a.g;
    if (a.i1 % a.g != 0)                         // the block starts inside a group opened by an earlier block
      q = make_colq(a.scales[(row_ok ? row : 0) * a.G + a.i1 / a.g], a.sym ? 0.0f : a.zeros[(row_ok ? row : 0) * a.G + a.i1 / a.g], a.qmin, a.qmax,
                    a.nrz);
  }
  __syncthreads();

  // Octet `to` = columns 8*to .. 8*to+7.  After every octet the registers rotate by one lane inside the team, so
  // the owner of the current octet is always lane 0 (a constant DPP source) and lane p holds the columns of
  // team member (p + to) mod 16.  After the last octet lane p therefore holds the finished columns of octet
  // (p + n_oct) mod 16, eight consecutive columns, and stores them once.  (Stores inside the loop would make every
  // later wait on a load wait for them too.)
  // A lone wave per SIMD issues about one instruction every ten cycles whatever the instruction is, so the run time
  // is the number of instructions per column, not the length of the dependency chain: the loop body holds the
  // chain, the eight fused multiply-adds of the rank-1 update and nothing else.
  const bool first = lane == 0;
  int n_oct = 0;
  for (int to = 0; to < 16; ++to) {
    if (8 * to >= a.count) break;
    ++n_oct;
    // the octet's 8 rows of U (this lane's 8 columns of each) and reciprocal diagonals, fetched ahead of the
    // dependency chain; rows past `count` are zero in LDS, so the 8 columns need no bound check
    const float* ucol = Us + (8 * to) * UP + 4 * ((lane + to) & 15);
    f32x4 u0[8], u1[8];
    #pragma unroll
    for (int c = 0; c < 8; ++c) {
      u0[c] = *(const f32x4*)(ucol + c * UP);
      u1[c] = *(const f32x4*)(ucol + c * UP + UH);
    }
    const f32x4 rda = *(const f32x4*)(Rd + 8 * to), rdb = *(const f32x4*)(Rd + 8 * to + 4);
    const float rd[8] = {rda[0], rda[1], rda[2], rda[3], rdb[0], rdb[1], rdb[2], rdb[3]};
    if (!STATIC && OCT) {
      if (a.i1 + 8 * to == nextb) {
        nextb += a.g;
        q = open_group(a, a.i1 + 8 * to, lane, row, row_ok, rbase, w, to == 0 && a.g == BS && a.count == BS);
      }
      if (first) { Ps[prow * NP + to] = q.s; Pz[prow * NP + to] = q.z; }
    }
    // 8 columns.  Each: quantize-dequantize like clamp(round(w / s) + z, qmin, qmax), (q - z) * s in fp32 (only
    // lane 0's result is used), err = (w - q) / d, rank-1 update of the lane's 8 columns.  U is strictly upper
    // triangular in LDS, so the column itself and the columns left of it see a zero factor and need no mask.
    // The first pass takes the quotient through the reciprocal and only notes how close an owner's product came to
    // a rounding boundary: within 2^-11 product and quotient may round apart, and the wave runs the octet again
    // from the saved registers with true divisions.  (Beyond +-1024 both round outside the clamp range, which
    // make_colq keeps within +-1024 for `fast` parameters; an infinite or NaN product makes the distance NaN.)
    // That keeps every branch out of the chain.
    auto octet = [&](auto exact_tag) -> bool {
      constexpr bool EXACT = decltype(exact_tag)::value;
      float margin = 0.5f;                                  // smallest distance of a product from a rounding boundary
      #pragma unroll
      for (int c = 0; c < 8; ++c) {
        if (STATIC) {
          q = make_colq(ss[c], zz[c], a.qmin, a.qmax, a.nrz);               // lane 0: the parameters of this column
          if (!EXACT) margin = q.fast ? margin : 0.0f;
        } else if (!OCT) {
          if (a.i1 + 8 * to + c == nextb && 8 * to + c < a.count) {
            nextb += a.g;
            q = open_group(a, a.i1 + 8 * to + c, lane, row, row_ok, rbase, w, false);
          }
          if (first) { Ps[prow * NP + 8 * to + c] = q.s; Pz[prow * NP + 8 * to + c] = q.z; }
        }
        const float wv = w[c];
        float diff;
        if (EXACT) {
          const float code = a.nrz ? rintf(wv / fmaxf(q.s, 1e-9f) + q.z) : rintf(wv / q.s) + q.z;
          diff = wv - (__builtin_amdgcn_fmed3f(code, a.qmin, a.qmax) - q.z) * q.s;
        } else {
          const float t = wv * q.r, rt = rintf(t);
          margin = nan_min(margin, fabsf(fabsf(t - rt) - 0.5f));
          diff = wv - __builtin_amdgcn_fmed3f(rt, q.lo, q.hi) * q.s;
        }
        const float eb = row16_first(diff * rd[c]);
        #pragma unroll
        for (int k = 0; k < 4; ++k) {
          w[k] = __builtin_fmaf(-eb, u0[c][k], w[k]);
          w[4 + k] = __builtin_fmaf(-eb, u1[c][k], w[4 + k]);
        }
      }
      if (EXACT) return false;
      return first & !((margin > 4.8828125e-04f) & (STATIC || q.fast));
    };
    if (STATIC || OCT) {
      float saved[8];
      #pragma unroll
      for (int c = 0; c < 8; ++c) saved[c] = w[c];
      const bool unsure = octet(std::false_type{});
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(unsure) != 0, 0)) {
        #pragma unroll
        for (int c = 0; c < 8; ++c) w[c] = saved[c];
        octet(std::true_type{});
      }
    } else {
      octet(std::true_type{});          // groups may open inside the octet: no replay, divide throughout
    }
    #pragma unroll
    for (int c = 0; c < 8; ++c) {
      w[c] = row16_next(w[c]);
      if (STATIC) { ss[c] = row16_next(ss[c]); zz[c] = row16_next(zz[c]); }
    }
  }

  // Outputs of the lane's eight finished columns.  w still holds each column as it was when it was quantized; the
  // quantized value, with true divisions, is the one the loop used (its reciprocal form is only taken where it
  // rounds like the division), and err = (w - q) * (1 / d) as in the loop.
  const int oct = (lane + n_oct) & 15;                      // the octet whose columns this lane holds now
  if (row_ok && 8 * oct < a.count) {
    float o_err[8], loss[8];
    #pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int col = 8 * oct + c;
      float s_, z_;
      if (STATIC) { s_ = ss[c]; z_ = zz[c]; }
      else { s_ = Ps[prow * NP + (OCT ? oct : col)]; z_ = Pz[prow * NP + (OCT ? oct : col)]; }
      if (col >= a.count) { s_ = 1.0f; z_ = 0.0f; }
      const float wv = w[c];
      const float code = a.nrz ? rintf(wv / fmaxf(s_, 1e-9f) + z_) : rintf(wv / s_) + z_;
      const float qdq = (__builtin_amdgcn_fmed3f(code, a.qmin, a.qmax) - z_) * s_;
      const float diff = wv - qdq;
      o_err[c] = diff * Rd[col];
      if (a.W0) o_err[c] = (col < a.count) ? qdq - a.W0[rbase + a.i1 + col] : 0.0f;
      const float d = Dg[col];
      loss[c] = (diff * diff) / (2.0f * (d * d));
    }
    if (vec) {
      float* pt = a.tmp + rbase + a.i1 + 8 * oct;
      float* pl = a.Losses + rbase + a.i1 + 8 * oct;
      *(f32x4*)pt = f32x4{w[0], w[1], w[2], w[3]};
      *(f32x4*)(pt + 4) = f32x4{w[4], w[5], w[6], w[7]};
      *(f32x4*)pl = f32x4{loss[0], loss[1], loss[2], loss[3]};
      *(f32x4*)(pl + 4) = f32x4{loss[4], loss[5], loss[6], loss[7]};
    }
    float* pe = a.Err + row * a.ldErr + 8 * oct;
    if (vec && a.ldErr % 4 == 0 && (reinterpret_cast<uintptr_t>(a.Err) & 15) == 0) {
      *(f32x4*)pe = f32x4{o_err[0], o_err[1], o_err[2], o_err[3]};
      *(f32x4*)(pe + 4) = f32x4{o_err[4], o_err[5], o_err[6], o_err[7]};
    } else {
      #pragma unroll
      for (int c = 0; c < 8; ++c) if (8 * oct + c < a.count) pe[c] = o_err[c];
    }
    if (!vec) {
      #pragma unroll
      for (int c = 0; c < 8; ++c) {
        const int col = 8 * oct + c;
        if (col < a.count) {
          a.tmp[rbase + a.i1 + col] = w[c];
          a.Losses[rbase + a.i1 + col] = loss[c];
        }
      }
    }
  }
}

// The same block for its most frequent forms (gptq_by_panels): 128 whole columns, groups of 16, 32, 64 or 128 of them that open inside the
// block or parameters that are given for groups of whole panels or rows, rounded zero points.  What the kernel above spends its time on are
// instructions: sixteen lanes share a row, so a column's quantization is issued once per four rows, and its update takes eight
// multiply-adds.  Here a wave quantizes 64 rows, one per lane:
//   * the chain wave (0) takes 16 columns from LDS and goes through them without a barrier.  A column is about nine instructions and at
//     most four v_mfma_f32_4x4x1_16b: with ONE block of the A operand (four columns of a row of U) broadcast to all 16 (cbsz = 4, abid),
//     an instruction updates four columns of 64 rows;
//   * the update waves (1, 2, 3, 5) hold 16 rows each in 16 x 16 tiles, the accumulators of v_mfma_f32_16x16x4f32.  They apply the
//     errors of a finished panel first to the next panel's columns and hand those over, then to the rest beside the chain of the next
//     panel.  Two barriers per panel;
//   * waves 4, 6 and 7 bring U to LDS; 6 and 7 then write the outputs of a finished panel.  The chain wave keeps its SIMD to itself:
//     beside an update wave its products wait for the other's, 32 cycles each, and a panel takes up to 2400 cycles instead of 1340.
// The ranges of all groups are known before the first column (groups are read from W as it is in memory).
// Quotients go through the group's reciprocal as above.  Where a product is closer to a rounding boundary than twice what its error can be,
// |t| 2^-22 for |t| up to the code range + 1, the wave runs the panel again with true divisions.  With 1024 products per panel that
// is 1 to 2 % of the panels at 4 bits, 12 to 22 % at 8 (4096 rows: 14.8 and 16.1 us per block; 16.5 by the kernel above), 40 % at codes of
// +-512, and beyond those, where reciprocals are not used, all of them (19.3 us; 24.3 by the kernel above, which divides then too).
// (The 2^-11 of the kernel above, for codes up to 1024, would be one of 1000 products.)
// Bound by the chain: eight times 1340 cycles for its columns and 1050 to 1650 for the handing over, behind 7200 (64 rows) to 8700 (4096) for
// the ranges and U.
// R = 64: 14.2 -> 12.8 us per block, 1000: 15.6 -> 13.7, 4096: 17.3 -> 14.9, 6144: 20.3 -> 16.1, 14336: 29.7 -> 21.3, 28672: 49.5 -> 31.7
// (two workgroups per CU).  The chain wave bringing in the errors of the panel before by itself, 64 more matrix instructions, cost 700
// cycles per panel instead of the 500 of the handing over.
constexpr int PT = 20;           // row pitch of a 16 x 16 tile and of the panel: 16-byte rows, 16 rows of 4 lanes in different banks
struct PanelLds {
  float U[36][16][PT];           // tiles (p, j), j >= p, of Hinv1; zero on and below the diagonal
  float Pn[64][PT];              // the panel on its way to the chain wave
  float E[64][PT];               // -err of the finished panel
  float Wq[64][PT], Dq[64][PT];  // its weights as they were quantized, and what they became
  float Rd[BS], Dg[BS];          // 1 / U[i, i], U[i, i]
  f32x4 pa[8][64];               // per panel and row: s, 1 / s, qmin - z, qmax - z
  f32x2 pb[8][64];               // z, distance from a rounding boundary that is enough
};
__device__ __forceinline__ constexpr int panel_tile(int p, int j) { return 8 * p - p * (p - 1) / 2 + j - p; }

// c + a b over 16 of the contraction, k = 4 (l / 16) + e in instruction e
__device__ __forceinline__ f32x4 panel_mac(const f32x4& a, const f32x4& b, f32x4 c) {
  #pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
  return c;
}
// columns 16 j .. of the rows of U that belong to panel p, as the first operand
__device__ __forceinline__ f32x4 panel_u(const PanelLds& s, int p, int j, int m, int g) {
  f32x4 v;
  #pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = s.U[panel_tile(p, j)][4 * g + e][m];
  return v;
}

// the 16 columns of a panel, in order: w -> as quantized, dq: quantized and back, e = -err.  EXACT: true divisions.  Returns the smallest distance of a product
// from a rounding boundary, NaN if a product was not finite.
// An update covers four columns, and U is zero up to the column itself: what has been quantized stays as it was while the errors are
// finite.  Zero times an infinite or NaN error is NaN, in the finished columns of the four as well as in those behind, whose products then
// are NaN: such panels run again, and EXACT keeps every column as it found it.
template <bool EXACT>
__device__ __forceinline__ float panel_chain(const LoopArgs& a, f32x4 (&w)[4], float (&dq)[16], float (&e)[16], const float (&u)[16], const f32x4 (&nrd)[4],
                                             const f32x4& pa, float z) {
  float margin = 0.5f;
  f32x4 found[4];
  #pragma unroll
  for (int j = 0; j < 16; ++j) {
    const float x = w[j >> 2][j & 3];
    if (EXACT) {
      found[j >> 2][j & 3] = x;
      const float code = rintf(x / pa[0]) + z;
      dq[j] = (__builtin_amdgcn_fmed3f(code, a.qmin, a.qmax) - z) * pa[0];
    } else {
      const float t = x * pa[1], rt = rintf(t);
      margin = nan_min(margin, fabsf(fabsf(t - rt) - 0.5f));
      dq[j] = __builtin_amdgcn_fmed3f(rt, pa[2], pa[3]) * pa[0];
    }
    e[j] = (x - dq[j]) * nrd[j >> 2][j & 3];
    if (j < 3) w[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(u[j], e[j], w[0], 4, 0, 0);
    if (j < 7) w[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(u[j], e[j], w[1], 4, 1, 0);
    if (j < 11) w[2] = __builtin_amdgcn_mfma_f32_4x4x1f32(u[j], e[j], w[2], 4, 2, 0);
    if (j < 15) w[3] = __builtin_amdgcn_mfma_f32_4x4x1f32(u[j], e[j], w[3], 4, 3, 0);
  }
  if (EXACT) {
    #pragma unroll
    for (int b = 0; b < 4; ++b) w[b] = found[b];
  }
  return margin;
}

__global__ __launch_bounds__(512) void gptq_panel_kernel(LoopArgs a) {
  __shared__ __align__(16) PanelLds s;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int id = __builtin_amdgcn_readfirstlane(tid >> 6);
  int last = 8;
  asm volatile("" : "+s"(last));                            // (or the loops over the panels are unrolled, and wait for instruction fetches)
  if (id == 4 || id >= 6) {
    // rows of panels 0, 5, 7 / 1, 4, 6 / 2, 3 of Hinv1: 12, 13 and 11 tiles, all loads in flight
    const int p0 = id == 4 ? 0 : id - 5, p1 = 5 - p0, p2 = p0 == 2 ? 8 : 7 - p0, n0 = 8 - p0, n1 = n0 + 8 - p1;
    const int panels = p0 | p1 << 4 | p2 << 8, starts = n0 << 4 | n1 << 8;    // (nibbles instead of selects: those became memory)
    const int r = lane >> 2, c = 4 * (lane & 3);
    f32x4 v[13];
    const auto tile_of = [=](int q, int& p, int& j) {
      const int at = 4 * ((q >= n0) + (q >= n1));
      p = (panels >> at) & 15;
      j = p + q - ((starts >> at) & 15);
      return p < 8 && j < 8;
    };
    #pragma unroll
    for (int q = 0; q < 13; ++q) {
      int p, j;
      if (!tile_of(q, p, j)) p = j = 7;
      v[q] = *(const f32x4*)(a.U + (long long)(a.i1 + 16 * p + r) * a.K + a.i1 + 16 * j + c);
    }
    #pragma unroll
    for (int q = 0; q < 13; ++q) {
      int p, j;
      if (!tile_of(q, p, j)) continue;
      #pragma unroll
      for (int e = 0; e < 4; ++e) v[q][e] = p == j && c + e <= r ? 0.0f : v[q][e];
      *(f32x4*)(s.U[panel_tile(p, j)][r] + c) = v[q];
    }
    __syncthreads();
    if (id == 4) return;
    // waves 6 and 7: the outputs of panel P - 1 beside the chain of panel P, two tiles of 16 rows each
    long long at[2], to[2];
    bool row_ok[2];
    #pragma unroll
    for (int h = 0; h < 2; ++h) {
      const long long row = (long long)blockIdx.x * 64 + 32 * (id - 6) + 16 * h + m;
      row_ok[h] = row < a.R;
      at[h] = (row_ok[h] ? row : a.R - 1) * a.K + a.i1 + 4 * g;
      to[h] = row * a.ldErr + 4 * g;
    }
    const auto fetch = [&](int Q, f32x4 (&w0)[2]) __attribute__((always_inline)) {
      if (a.W0)
        #pragma unroll
        for (int h = 0; h < 2; ++h) w0[h] = *(const f32x4*)(a.W0 + at[h] + 16 * Q);
    };
    const auto outputs = [&](int Q, const f32x4 (&w0)[2]) __attribute__((always_inline)) {
      const int col = 16 * Q;
      const f32x4 rd = *(const f32x4*)(s.Rd + col + 4 * g), d = *(const f32x4*)(s.Dg + col + 4 * g);
      #pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = 32 * (id - 6) + 16 * h + m;
        const f32x4 wq = *(const f32x4*)(s.Wq[row] + 4 * g), dq = *(const f32x4*)(s.Dq[row] + 4 * g);
        f32x4 out, loss;
        #pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float diff = wq[e] - dq[e];
          out[e] = a.W0 ? dq[e] - w0[h][e] : diff * rd[e];
          loss[e] = (diff * diff) / (2.0f * (d[e] * d[e]));
        }
        if (row_ok[h]) {
          *(f32x4*)(a.tmp + at[h] + col) = wq;
          *(f32x4*)(a.Losses + at[h] + col) = loss;
          *(f32x4*)(a.Err + to[h] + col) = out;
        }
      }
    };
    // W0 comes a panel or two ahead, into registers of its own for even and odd panels: a copy of them would wait for the loads, and
    // for the stores in front of them, before the barrier
    f32x4 even[2] = {}, odd[2] = {};
    fetch(0, even);
    #pragma unroll 1
    for (int P = 0; P < last; P += 2) {
      if (P > 0) outputs(P - 1, odd);
      fetch(P + 1, odd);
      __syncthreads();
      __syncthreads();                                      // panel P is done
      outputs(P, even);
      if (P < 6) fetch(P + 2, even);
      __syncthreads();
      __syncthreads();
    }
    outputs(7, odd);
    return;
  }
  if (id == 0) {
    #pragma unroll
    for (int c = lane; c < BS; c += 64) {
      const float d = a.U[(long long)(a.i1 + c) * a.K + a.i1 + c];
      s.Dg[c] = d;
      s.Rd[c] = 1.0f / d;
    }
    __syncthreads();
    f32x4 pa = {1.0f, 1.0f, 0.0f, 0.0f}, nrd[4];
    f32x2 pb = {0.0f, 0.0f};
    float u[16], dq[16], e[16];
    const auto fetch = [&](int P) {
      #pragma unroll
      for (int j = 0; j < 16; ++j) u[j] = s.U[panel_tile(P, P)][j][m];
      #pragma unroll
      for (int b = 0; b < 4; ++b) nrd[b] = -*(const f32x4*)(s.Rd + 16 * P + 4 * b);
      pa = s.pa[P][lane];
      pb = s.pb[P][lane];
    };
    fetch(0);
    #pragma unroll 1
    for (int P = 0; P < last; ++P) {
      f32x4 w[4], kept[4];
      #pragma unroll
      for (int b = 0; b < 4; ++b) kept[b] = w[b] = *(const f32x4*)(s.Pn[lane] + 4 * b);
      const bool unsure = !(panel_chain<false>(a, w, dq, e, u, nrd, pa, pb[0]) > pb[1]);
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(unsure) != 0, 0)) {
        #pragma unroll
        for (int b = 0; b < 4; ++b) w[b] = kept[b];
        panel_chain<true>(a, w, dq, e, u, nrd, pa, pb[0]);
      }
      #pragma unroll
      for (int b = 0; b < 4; ++b) *(f32x4*)(s.E[lane] + 4 * b) = f32x4{e[4 * b], e[4 * b + 1], e[4 * b + 2], e[4 * b + 3]};
      __syncthreads();                                      // E holds panel P
      // beside the handing over
      #pragma unroll
      for (int b = 0; b < 4; ++b) {
        *(f32x4*)(s.Wq[lane] + 4 * b) = w[b];
        *(f32x4*)(s.Dq[lane] + 4 * b) = f32x4{dq[4 * b], dq[4 * b + 1], dq[4 * b + 2], dq[4 * b + 3]};
      }
      if (P < 7) fetch(P + 1);
      __syncthreads();                                      // Wq and Dq hold panel P, Pn panel P + 1
    }
    return;
  }

  const int wave = id == 5 ? 0 : id;
  const long long row = (long long)blockIdx.x * 64 + 16 * wave + m;
  const bool row_ok = row < a.R;
  const long long at = (row_ok ? row : a.R - 1) * a.K + a.i1;
  // tile j of this wave's 16 rows, transposed: lane element e is row m, column 16 j + 4 g + e
  f32x4 t[8];
  #pragma unroll
  for (int j = 0; j < 8; ++j) t[j] = *(const f32x4*)(a.W + at + 16 * j + 4 * g);
  *(f32x4*)(s.Pn[16 * wave + m] + 4 * g) = t[0];
  {
    // ranges of the groups: over a lane's elements, its tiles, and the four lanes of a row
    const int gt = a.is_static ? 1 : a.g >> 4, sh = 31 - __builtin_clz(gt);   // panels per group, a power of two
    float mn[8], mx[8], sc = 1.0f, z = 0.0f, mine[2] = {}, zero[2] = {};      // a lane's parameters are those of panels g and g + 4
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      mn[j] = nan_min(nan_min(t[j][0], t[j][1]), nan_min(t[j][2], t[j][3]));
      mx[j] = nan_max(nan_max(t[j][0], t[j][1]), nan_max(t[j][2], t[j][3]));
    }
    #pragma unroll
    for (int span = 1; span < 8; span *= 2)
      if (span < gt)
        #pragma unroll
        for (int j = 0; j < 8; j += 2 * span) { mn[j] = nan_min(mn[j], mn[j + span]); mx[j] = nan_max(mx[j], mx[j + span]); }
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (a.is_static) {
        const long long from = (row_ok ? row : a.R - 1) * a.G + (a.g > 0 ? (a.i1 + 16 * j) / a.g : 0);
        sc = a.scales[from];
        z = a.sym ? 0.0f : a.zeros[from];
      } else if ((j & (gt - 1)) == 0) {
        float lo = nan_min(mn[j], lane_xor<16>(mn[j])), hi = nan_max(mx[j], lane_xor<16>(mx[j]));
        lo = nan_min(lo, lane_xor<32>(lo));
        hi = nan_max(hi, lane_xor<32>(hi));
        group_params(a, lo, hi, sc, z);
        if (g == 0 && row_ok) {
          const long long to = row * a.G + (a.i1 >> 4 >> sh) + (j >> sh);
          a.scales[to] = sc;
          if (!a.sym) a.zeros[to] = z;
        }
      }
      mine[j >> 2] = g == (j & 3) ? sc : mine[j >> 2];
      zero[j >> 2] = g == (j & 3) ? z : zero[j >> 2];
    }
    #pragma unroll
    for (int h = 0; h < 2; ++h) {
      const ColQ q = make_colq(mine[h], zero[h], a.qmin, a.qmax);
      s.pa[4 * h + g][16 * wave + m] = f32x4{q.s, q.r, q.lo, q.hi};
      s.pb[4 * h + g][16 * wave + m] = f32x2{q.z, q.fast ? (fmaxf(fabsf(q.lo), fabsf(q.hi)) + 1.0f) * 4.76837158e-7f : __builtin_inff()};
    }
  }
  __syncthreads();                                          // U, the first panel and the parameters
  #pragma unroll
  for (int k = 0; k < 7; ++k) t[k] = t[k + 1];              // from here on t[0] is the panel after the one in the chain
  f32x4 err = {0.0f, 0.0f, 0.0f, 0.0f};
  #pragma unroll 1
  for (int P = 0; P < last; ++P) {
    f32x4 u[6], next = {0.0f, 0.0f, 0.0f, 0.0f};
    if (P < 7) next = panel_u(s, P, P + 1, m, g);
    if (P > 0) {                                            // panel P - 1 on the tiles behind
      #pragma unroll
      for (int k = 0; k < 6; ++k) u[k] = panel_u(s, P - 1, min(P + 1 + k, 7), m, g);
      #pragma unroll
      for (int k = 0; k < 6; ++k)
        if (k < 7 - P) t[k] = panel_mac(u[k], err, t[k]);
    }
    __syncthreads();                                        // E holds panel P
    err = *(const f32x4*)(s.E[16 * wave + m] + 4 * g);
    if (P < 7) {
      t[0] = panel_mac(next, err, t[0]);
      *(f32x4*)(s.Pn[16 * wave + m] + 4 * g) = t[0];
    }
    __syncthreads();                                        // Wq and Dq hold panel P, Pn panel P + 1
    #pragma unroll
    for (int k = 0; k < 6; ++k) t[k] = t[k + 1];
  }
}

}  // namespace

extern "C" {

int lcq_gptq_block(float* W, float* tmp, float* Losses, float* Err, int64_t ldErr, const float* U, const float* W0, int64_t R,
                   int64_t K, int64_t n_quant, int64_t i1, int count, int group_size, float qmin, float qmax, int flags, float* scales, float* zeros,
                   const int32_t* gidx, int64_t G, void* stream) {
  if (!W || !tmp || !Losses || !Err || !U || !scales || ldErr < count || ldErr > 0x7fffffff) return LCQ_EINVAL;
  if (R <= 0 || K <= 0 || K > 0x7fffffff || i1 < 0 || count <= 0 || count > BS) return LCQ_EINVAL;
  if (n_quant <= 0 || n_quant > K || i1 + count > n_quant) return LCQ_EINVAL;
  if (!(qmax > qmin) || G <= 0) return LCQ_EINVAL;
  const int is_static = (flags & LCQ_FLAG_STATIC) != 0;
  const int sym = (flags & LCQ_FLAG_SYM) != 0;
  if (!is_static && (group_size <= 0 || G < (n_quant + group_size - 1) / group_size)) return LCQ_EINVAL;
  if (!sym && !zeros) return LCQ_EINVAL;
  LoopArgs a;
  a.W = W; a.tmp = tmp; a.Losses = Losses; a.Err = Err; a.U = U; a.W0 = W0;
  a.scales = scales; a.zeros = zeros; a.gidx = gidx;
  a.R = R; a.K = (int)K; a.Kq = (int)n_quant; a.i1 = (int)i1; a.count = count; a.g = group_size; a.G = (int)G;
  a.qmin = qmin; a.qmax = qmax; a.sym = sym; a.is_static = is_static; a.ldErr = (int)ldErr;
  a.nrz = (flags & LCQ_FLAG_NO_ROUND_ZP) != 0;
  a.aligned = ((reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(tmp) | reinterpret_cast<uintptr_t>(Losses) |
                reinterpret_cast<uintptr_t>(U)) & 15) == 0;
  const bool oct = !is_static && group_size % 8 == 0 && i1 % 8 == 0;
  hipStream_t st = (hipStream_t)stream;
  const bool on16 = a.aligned && (((uintptr_t)Err | (uintptr_t)W0) & 15) == 0;
  if (gptq_by_panels(is_static, gidx != nullptr, !a.nrz, group_size, R, K, i1, count, ldErr, on16, qmin, qmax)) {
    gptq_panel_kernel<<<dim3((unsigned)((R + 63) / 64)), dim3(512), 0, st>>>(a);
    LCQ_CHECK_LAUNCH();
    return LCQ_OK;
  }
  // The other forms.  From 6144 rows on, 32 rows per workgroup: one copy of Hinv1 in LDS (70 KB) per eight waves, so that the two
  // workgroups a CU holds put four waves on every SIMD (R = 28672: 57 -> 48 us per block, 14336: 35 -> 29, 6144:
  // 20 -> 19; at 4096 rows, one workgroup per CU either way, the smaller workgroup is faster, 17 against 19 us).
  // The rows do not interact: the results are the same bit for bit.
  if (R >= 6144 && (is_static || oct) && !(flags & LCQ_FLAG_ROWS16)) {
    const unsigned grid = (unsigned)((R + 31) / 32);
    if (is_static) gptq_block_kernel<true, true, 32><<<dim3(grid), dim3(512), 0, st>>>(a);
    else gptq_block_kernel<false, true, 32><<<dim3(grid), dim3(512), 0, st>>>(a);
  } else {
    const unsigned grid = (unsigned)((R + 15) / 16);
    if (is_static) gptq_block_kernel<true, true, 16><<<dim3(grid), dim3(256), 0, st>>>(a);
    else if (oct) gptq_block_kernel<false, true, 16><<<dim3(grid), dim3(256), 0, st>>>(a);
    else gptq_block_kernel<false, false, 16><<<dim3(grid), dim3(256), 0, st>>>(a);
  }
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_gptq_trailing(float* W, const float* Err, int64_t ldErr, const float* U, int64_t R, int64_t K, int64_t k1,
                      int64_t k2, int64_t j1, int64_t j2, void* stream) {
  if (!W || !Err || !U || R <= 0 || K <= 0 || K > 0x7fffffff || R > 0x7fffffff) return LCQ_EINVAL;
  if (k1 < 0 || k2 <= k1 || k2 > K || j1 < k2 || j2 < j1 || j2 > K || ldErr < k2 - k1 || ldErr > 0x7fffffff) return LCQ_EINVAL;
  if (j1 == j2) return LCQ_OK;
  // W[:, j1:j2] -= Err[:, :k2-k1] @ U[k1:k2, j1:j2]
  GemmProblem g{Err, U + k1 * K + j1, W + j1, (int)R, (int)(j2 - j1), (int)(k2 - k1), (int)ldErr, (int)K, (int)K};
  launch_gemm<false>(g, -1.0f, 1.0f, 0, (hipStream_t)stream);
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

// The operands split once (gemm_s3p.h) where that pays; the same bits either way.
int64_t lcq_gptq_trailing_workspace_bytes(int64_t R, int64_t K, int64_t k1, int64_t k2, int64_t j1, int64_t j2) {
  if (R <= 0 || R > (1 << 24) || K <= 0 || K > (1 << 20) || k1 < 0 || k2 <= k1 || k2 > j1 || j2 > K || j2 <= j1) return 0;
  if (!g_gemm_split.load(std::memory_order_relaxed) || !s3p_depth(k2 - k1) || !s3p_pays(R, j2 - j1, s3p_tiles(R, j2 - j1))) return 0;
  return s3p_bytes(R, k2 - k1) + s3p_bytes(j2 - j1, k2 - k1);
}

int lcq_gptq_trailing_deep(float* W, const float* Err, int64_t ldErr, const float* U, int64_t R, int64_t K, int64_t k1, int64_t k2,
                           int64_t j1, int64_t j2, void* workspace, int64_t workspace_bytes, void* stream) {
  const int64_t need = lcq_gptq_trailing_workspace_bytes(R, K, k1, k2, j1, j2);
  if (need == 0 || !W || !Err || !U || ldErr < k2 - k1 || !s3p_operand(Err, ldErr, k2 - k1))
    return lcq_gptq_trailing(W, Err, ldErr, U, R, K, k1, k2, j1, j2, stream);
  if (!workspace || workspace_bytes < need) return LCQ_EWORKSPACE;
  if (((uintptr_t)workspace % 16) != 0) return LCQ_EALIGN;
  const int Kc = (int)(k2 - k1), N = (int)(j2 - j1);
  hipStream_t st = (hipStream_t)stream;
  const S3POperand a(workspace, R), b((char*)workspace + s3p_bytes(R, Kc), N);
  s3p_pack<false>(Err, ldErr, (int)R, Kc, a, st);
  s3p_pack<true>(U + k1 * K + j1, K, N, Kc, b, st);
  s3p_multiply<false>(a, b, W + j1, (int)K, (int)R, N, Kc, st);
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

}  // extern "C"
