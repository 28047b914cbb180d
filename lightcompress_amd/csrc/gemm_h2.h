// fp32 products as three fp16 products, for the large launches of the Cholesky chain and of the column loop.
//
//   x = hi + lo,  hi = fp16(s x), lo = fp16(s x - hi)       s a power of two per row of A and per column of B
// carries x to 2^-23 of itself (hi, 11 bits, leaves a residual of at most 2^-11 |x|, whose last bit lo loses where it has more
// than 11), as long as x is above 2^-17 of the largest value of its row, and to 2^-40 of that value below; a b = lo hi + hi lo +
// hi hi, the dropped lo lo being at most 2^-22 of the product.  Three matrix instructions accumulate in fp32 where the three-way
// bf16 split takes six, so the sum is rounded half as often.  The operands' part does not grow with the depth (some 7e-8 of the
// norm, the three-way split's is 1e-8), the sum's does: from 512 on the result is closer to fp64 than the three-way split's
// (below), which is closer than the fp32 pipe's; at 256 a few large products per element (exp(2 N) of a normal N as elements of
// both) leave 1.6e-7 against 0.8e-7.  Shallower products stay with the three-way split.
//
// The operands are split once (h2_pack_kernel), not by every tile that reads them, into the order the matrix pipe reads:
//   planes[k / 16][hi, lo][row / 32][(k / 8) % 2][row % 32][k % 8]        1 KiB per operand of v_mfma_f32_32x32x16_f16
// and the product is the Hessian kernel's (hessian_packed_kernel) with its 32 tokens replaced by the two planes of 16 k:
// 256 x 256 tiles, four waves of 128 x 128, direct loads to four LDS stages, operands double-buffered in registers.  Per 16 k a
// wave reads 16 operands for 48 matrix instructions, a third less LDS traffic and two thirds of the loads per instruction.
// Measured with the packing (us, three-way bf16 split on 128 x 128 tiles -> this): 28672 x 3072 x 1024 1015 -> 539, 4096 x 13312 x
// 1024 641 -> 352, lower triangle of 13824 x 13824 x 512 655 -> 343 (335, 317 and 286 TFLOP/s of fp32 products).  Relative error
// against fp64 of a 4096 x 5000 x 1024 product: 3.6e-7, bf16 split 4.9e-7, fp32 pipe 5.7e-7.  What bounds it: reading and writing
// C, 512 KB per tile that no second workgroup overlaps, a quarter of the time at Kc = 1024; the matrix pipes the rest.
#pragma once
#include "common.h"

namespace lcq {

typedef __attribute__((ext_vector_type(8))) _Float16 h2_f16x8;
typedef __attribute__((ext_vector_type(16))) float h2_f32x16;

constexpr int H2_T = 256;                           // tile of C
constexpr int H2_STAGES = 4, H2_HALF = 16384, H2_STAGE = 2 * H2_HALF;
constexpr int H2_MAX_K = 1024;

inline int64_t h2_rows(int64_t rows) { return (rows + H2_T - 1) / H2_T * H2_T; }
// planes and scales of one operand
inline int64_t h2_bytes(int64_t rows, int64_t Kc) { return h2_rows(rows) * (Kc * 4 + 4); }

// 32 rows of an operand per workgroup: src[row * ld + k], or src[k * ld + row] (T).  Rows past `rows` are zeros.
template <bool T, int STEPS>
__global__ __launch_bounds__(256) void h2_pack_kernel(const float* __restrict__ src, long long ld, int rows, int Kc, int blocks,
                                                      uint16_t* __restrict__ planes, float* __restrict__ unscale) {
  __shared__ float red[4][32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, kh = lane >> 5;
  const int row = blockIdx.x * 32 + r, n = Kc / 16;
  float v[STEPS][8], m = 0.0f;                      // steps wave, wave + 4, ...
  #pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int step = wave + 4 * i;
    const long long k = 16 * step + 8 * kh;
    #pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] = 0.0f;
    if (step < n && row < rows) {
      if constexpr (T) {
        #pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = src[(k + e) * ld + row];
      } else {
        const f32x4* const p = (const f32x4*)(src + row * ld + k);
        const f32x4 a = p[0], b = p[1];
        #pragma unroll
        for (int e = 0; e < 4; ++e) { v[i][e] = a[e]; v[i][4 + e] = b[e]; }
      }
    }
  }
  #pragma unroll
  for (int i = 0; i < STEPS; ++i)
    #pragma unroll
    for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(v[i][e]));
  m = fmaxf(m, __shfl_xor(m, 32));
  if (kh == 0) red[wave][r] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0][r], red[1][r]), fmaxf(red[2][r], red[3][r]));
  // s = 2^(14 - e), 2^e <= m < 2^(e + 1): the largest value lands in [2^14, 2^15).  (No scale for rows of zeros or with infinities.)
  int e = m < __builtin_inff() && m > 0.0f ? (int)(f2u(m) >> 23) - 127 : 14;
  if (e < -100) e = -100;
  const float s = u2f((uint32_t)(127 + 14 - e) << 23);
  if (wave == 0 && kh == 0) unscale[row] = u2f((uint32_t)(127 - 14 + e) << 23);
  #pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int step = wave + 4 * i;
    if (step < n) {
      h2_f16x8 hi, lo;
      #pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float x = v[i][c] * s;
        hi[c] = (_Float16)x;
        lo[c] = (_Float16)(x - (float)hi[c]);
      }
      uint16_t* const out = planes + ((long long)step * 2 * blocks + blockIdx.x) * 512 + lane * 8;
      *(h2_f16x8*)out = hi;
      *(h2_f16x8*)(out + (long long)blocks * 512) = lo;
    }
  }
}

struct H2Gemm {
  const uint16_t *A, *B;                            // planes
  const float *ua, *ub;                             // 1 / s of the rows of A, the columns of B
  float* C;
  int blocksA, blocksB, ldc, M, N, Kc;
};

// C -= A B.  LOWER: the tiles that reach the lower triangle of a square C, a 1-D grid over 4 x 4 super-blocks;
// else a 2-D grid.  EDGE: M or N not in whole tiles.  Kc % 32 == 0.
template <bool EDGE, bool LOWER>
__global__ __launch_bounds__(256, 1) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_h2_kernel(H2Gemm g, int gx, int gy) {
  typedef const __attribute__((address_space(3))) char* lds_ptr;
  typedef const __attribute__((address_space(3))) h2_f16x8* lds_frag;
  __shared__ __attribute__((aligned(1024))) char lds[H2_STAGES * H2_STAGE];
  // XCD x (blocks b % 8 == x) works through a contiguous range of the tile order, in super-blocks of 4 x 4 tiles
  int ti, tj;
  if constexpr (LOWER) {
    const int total = gridDim.x, lin = blockIdx.x, v = (lin & 7) * (total >> 3) + (lin >> 3);     // 16 tiles per super-block
    const int sb = v >> 4, t = v & 15;
    int sr = (int)((__builtin_sqrtf(8.0f * (float)sb + 1.0f) - 1.0f) * 0.5f);
    while (sr * (sr + 1) / 2 > sb) --sr;
    while ((sr + 1) * (sr + 2) / 2 <= sb) ++sr;
    ti = sr * 4 + (t >> 2);
    tj = (sb - sr * (sr + 1) / 2) * 4 + (t & 3);
    if (ti >= gy || tj > ti) return;
  } else {
    const int total = gx * gy, base = total >> 3, rem = total & 7, lin = blockIdx.x, x = lin & 7;
    int v = x * base + min(x, rem) + (lin >> 3);
    const int r0 = v / (4 * gx) * 4, nr = min(4, gy - r0);
    v -= r0 * gx;
    const int sc = min(v / (nr * 4), (gx - 1) / 4), nc = min(4, gx - sc * 4);
    v -= sc * nr * 4;
    ti = r0 + v / nc;
    tj = sc * 4 + v % nc;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 1, wc = wave & 1;
  const int steps = g.Kc / 16;                      // an even number of slabs of 16 k
  const int64_t slabA = (int64_t)g.blocksA * 1024, slabB = (int64_t)g.blocksB * 1024;       // elements
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds;
  const lds_ptr readA = (lds_ptr)lds + lane * 16 + wr * 4096, readB = (lds_ptr)lds + H2_HALF + lane * 16 + wc * 4096;
  uint32_t gof[8];                                  // this wave's pieces of a slab: plane c / 8, block c % 8 of A, then of B
  #pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int c = wave * 4 + p;
    gof[p] = ((c >> 3) * g.blocksA + ti * 8 + (c & 7)) * 1024u + lane * 16;
    gof[4 + p] = ((c >> 3) * g.blocksB + tj * 8 + (c & 7)) * 1024u + lane * 16;
  }
  const auto gload = [&](const uint16_t* a, const uint16_t* b, uint32_t dst, int p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 ::"s"(dst + (p >> 2) * H2_HALF + (p & 3) * 1024), "v"(gof[p]), "s"(p < 4 ? a : b) : "memory");
  };
  h2_f32x16 acc[4][4];
  #pragma unroll
  for (int i = 0; i < 4; ++i)
    #pragma unroll
    for (int j = 0; j < 4; ++j)
      #pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  h2_f16x8 fr[2][16];                               // two sets of operands: A hi 0..3, A lo 4..7, B hi 8..11, B lo 12..15
  const auto rd = [&](int set, int f, uint32_t stage) {
    fr[set][f] = *(lds_frag)((f < 8 ? readA : readB) + stage + ((f >> 2) & 1) * 8192 + (f & 3) * 1024);
  };
  constexpr int ORDER[16] = {8, 4, 5, 6, 7, 9, 10, 11, 0, 1, 2, 3, 12, 13, 14, 15};        // as the products need them

  // Past the last slab a load fetches the first one again (its stage is never read): the number in flight is always the same.
  #pragma unroll
  for (int s = 0; s < H2_STAGES; ++s) {
    const int at = s < steps ? s : 0;
    #pragma unroll
    for (int p = 0; p < 8; ++p) gload(g.A + at * slabA, g.B + at * slabB, lds0 + s * H2_STAGE + wave * 4096, p);
  }
  constexpr int FIRST = (H2_STAGES - 1) * 8, LATER = (H2_STAGES - 2) * 8;
  __builtin_amdgcn_s_waitcnt(0x0F70 | (FIRST & 15) | ((FIRST >> 4) << 14));
  __syncthreads();
  #pragma unroll
  for (int f = 0; f < 16; ++f) rd(0, ORDER[f], 0);
  int s = 0;
  uint32_t cur = 0;
  __builtin_amdgcn_sched_barrier(0);
  const auto half = [&](int set) __attribute__((always_inline)) {
    // slab s is in every wave's registers (its stage takes slab s + 4), slab s + 1 has landed
    __builtin_amdgcn_s_waitcnt(0x0070 | (LATER & 15) | ((LATER >> 4) << 14));
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t nxt = (cur == (H2_STAGES - 1) * H2_STAGE) ? 0 : cur + H2_STAGE;
    const int at = s + H2_STAGES < steps ? s + H2_STAGES : 0;
    const uint16_t* const a = g.A + at * slabA;
    const uint16_t* const b = g.B + at * slabB;
    #pragma unroll
    for (int m = 0; m < 48; ++m) {
      // 16 products lo hi, 16 hi lo, 16 hi hi
      const int i = m & 3, j = (m >> 2) & 3, fa = m < 16 ? 4 + i : i, fb = m < 16 || m >= 32 ? 8 + j : 12 + j;
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[set][fa], fr[set][fb], acc[i][j], 0, 0, 0);
      if (m % 3 != 2 && m < 24) rd(set ^ 1, ORDER[(m / 3) * 2 + m % 3], nxt);
      if (m % 6 == 5) gload(a, b, lds0 + cur + wave * 4096, m / 6);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = nxt;
    ++s;
  };
  do {                                              // (at least two slabs)
    half(0);
    half(1);
  } while (s < steps);
  __builtin_amdgcn_s_waitcnt(0x0070);               // nothing may still be on its way to LDS when the workgroup ends

  // accumulator register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32
  const int row = wr * 128 + 4 * (lane >> 5), col = wc * 128 + (lane & 31);
  char* const out = (char*)(g.C + (int64_t)(ti * H2_T) * g.ldc + tj * H2_T);
  const uint32_t pitch = 4u * (uint32_t)g.ldc, at0 = row * pitch + 4 * col;
  const int rows = EDGE ? g.M - (ti * H2_T + row) : H2_T, cols = EDGE ? g.N - (tj * H2_T + col) : H2_T;
  const auto inside = [&](int i, int j, int r) { return !EDGE || (i * 32 + 8 * (r >> 2) + (r & 3) < rows && j * 32 < cols); };
  float uc[4];
  #pragma unroll
  for (int j = 0; j < 4; ++j) uc[j] = g.ub[tj * H2_T + col + j * 32];
  #pragma unroll
  for (int i = 0; i < 4; ++i) {
    // (the accumulators stay where they are until their turn: copied out together they would not fit the other registers)
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]));
    float old[4][16], ur[16];
    uint32_t off[16];                               // 32-bit offsets from the tile's corner; j * 128 goes into the instruction
    #pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 u = *(const f32x4*)(g.ua + ti * H2_T + row + i * 32 + 8 * q);
      #pragma unroll
      for (int c = 0; c < 4; ++c) { ur[4 * q + c] = u[c]; off[4 * q + c] = at0 + (i * 32 + 8 * q + c) * pitch; }
    }
    #pragma unroll
    for (int r = 0; r < 16; ++r)
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (EDGE) old[j][r] = *(const float*)(out + (inside(i, j, r) ? off[r] + j * 128 : 0u));     // (all loads in flight)
        else old[j][r] = *(const float*)(out + (uint64_t)off[r] + j * 128);
      }
    #pragma unroll
    for (int r = 0; r < 16; ++r)
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float w = old[j][r] - acc[i][j][r] * ur[r] * uc[j];
        if (inside(i, j, r)) *(float*)(out + (uint64_t)off[r] + j * 128) = w;
      }
  }
}

// Operands in memory of h2_bytes(rows, Kc), 16-byte aligned.
struct H2Operand {
  uint16_t* planes;
  float* unscale;
  int blocks;
  H2Operand(void* p, int64_t rows, int64_t Kc)
      : planes((uint16_t*)p), unscale((float*)(planes + h2_rows(rows) * Kc * 2)), blocks((int)(h2_rows(rows) / 32)) {}
};
template <bool T>
inline void h2_pack(const float* src, int64_t ld, int rows, int Kc, const H2Operand& o, hipStream_t st) {
  if (Kc <= 512) h2_pack_kernel<T, 8><<<dim3((unsigned)o.blocks), dim3(256), 0, st>>>(src, ld, rows, Kc, o.blocks, o.planes, o.unscale);
  else h2_pack_kernel<T, 16><<<dim3((unsigned)o.blocks), dim3(256), 0, st>>>(src, ld, rows, Kc, o.blocks, o.planes, o.unscale);
}

// May a row-major operand [rows, Kc] be packed?  (One given as [Kc, rows] only needs the depth.)
inline bool h2_depth(int64_t Kc) { return Kc % 64 == 0 && Kc >= 512 && Kc <= H2_MAX_K; }      // (why 512: at the top)
inline bool h2_operand(const float* p, int64_t ld, int64_t Kc) { return h2_depth(Kc) && ld % 4 == 0 && (uintptr_t)p % 16 == 0; }
inline int64_t h2_tiles(int64_t M, int64_t N) { return ((M + H2_T - 1) / H2_T) * ((N + H2_T - 1) / H2_T); }

// C [M, N] -= A B^T, A's rows from row0A on (a multiple of 32), B's from row0B on.  LOWER: M == N, the tiles on and below the
// diagonal.
template <bool LOWER>
inline void h2_multiply(const H2Operand& a, int row0A, const H2Operand& b, int row0B, float* C, int ldc, int M, int N, int Kc,
                        hipStream_t st) {
  H2Gemm g;
  g.A = a.planes + (int64_t)(row0A / 32) * 512; g.B = b.planes + (int64_t)(row0B / 32) * 512;
  g.ua = a.unscale + row0A; g.ub = b.unscale + row0B;
  g.blocksA = a.blocks; g.blocksB = b.blocks;
  g.C = C; g.ldc = ldc; g.M = M; g.N = N; g.Kc = Kc;
  const int gx = (N + H2_T - 1) / H2_T, gy = (M + H2_T - 1) / H2_T, nsb = (gy + 3) / 4;
  const unsigned grid = LOWER ? (unsigned)(16 * (nsb * (nsb + 1) / 2)) : (unsigned)(gx * gy);
  if (M % H2_T != 0 || N % H2_T != 0) gemm_h2_kernel<true, LOWER><<<dim3(grid), dim3(256), 0, st>>>(g, gx, gy);
  else gemm_h2_kernel<false, LOWER><<<dim3(grid), dim3(256), 0, st>>>(g, gx, gy);
}

}  // namespace lcq
