// The three-way bf16 product of gemm_f32.h on operands that are split once, for the large launches of the Cholesky chain and of
// the column loop.
//
// The split (s3_split) and the six partial products per 16 k, in their order, are gemm_tile_s3's, and an element of C is one chain
// over all k either way: the results are the same bit for bit.  What differs is who splits.  There every tile splits the operands
// it reads; here s3p_pack_kernel does it once, into the order the matrix pipe reads:
//   planes[k / 16][hi, mid, lo][row / 32][(k / 8) % 2][row % 32][k % 8]        1 KiB per operand of v_mfma_f32_32x32x16_bf16
// and the product is the Hessian kernel's (hessian_packed_kernel) with its 32 tokens replaced by the three planes of 16 k:
// 256 x 256 tiles, four waves of 128 x 128, direct loads to three LDS stages of 48 KB.  Per 16 k a wave reads 24 operands for 96
// matrix instructions.
// Measured with the packing (us, split by the tiles -> this): 28672 x 3072 x 1024 1055 -> 891, 4096 x 13312 x 1024 666 -> 571,
// 14336 x 2048 x 512 212 -> 166; Cholesky chain of K = 14336 12.3 -> 11.2 ms.  What bounds it: the matrix pipes (1.2 PFLOP/s of
// bf16 products), and reading and writing C, 512 KB per tile that no second workgroup overlaps.
#pragma once
#include "gemm_f32.h"

namespace lcq {

constexpr int S3P_T = 256;                          // tile of C
constexpr int S3P_STAGES = 3, S3P_HALF = 3 * 8192, S3P_STAGE = 2 * S3P_HALF;
constexpr int S3P_MAX_K = 1024;

inline int64_t s3p_rows(int64_t rows) { return (rows + S3P_T - 1) / S3P_T * S3P_T; }
// planes of one operand
inline int64_t s3p_bytes(int64_t rows, int64_t Kc) { return s3p_rows(rows) * Kc * 6; }

// 32 rows of an operand per workgroup, every fourth step of 16 k per wave: src[row * ld + k], or src[k * ld + row] (T).  Rows
// past `rows` are zeros.
template <bool T>
__global__ __launch_bounds__(256) void s3p_pack_kernel(const float* __restrict__ src, long long ld, int rows, int Kc, int blocks,
                                                       uint16_t* __restrict__ planes) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, kh = lane >> 5;
  const int row = blockIdx.x * 32 + r, n = Kc / 16;
  #pragma unroll 4
  for (int step = wave; step < n; step += 4) {
    const long long k = 16 * step + 8 * kh;
    f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f}, b = a;
    if (row < rows) {
      if constexpr (T) {
        #pragma unroll
        for (int e = 0; e < 4; ++e) { a[e] = src[(k + e) * ld + row]; b[e] = src[(k + 4 + e) * ld + row]; }
      } else {
        const f32x4* const p = (const f32x4*)(src + row * ld + k);
        a = p[0]; b = p[1];
      }
    }
    u32x2 h[2], m[2], l[2];
    s3_split(a, h[0], m[0], l[0]);
    s3_split(b, h[1], m[1], l[1]);
    uint16_t* const out = planes + ((long long)step * 3 * blocks + blockIdx.x) * 512 + lane * 8;
    *(u32x4*)out = u32x4{h[0][0], h[0][1], h[1][0], h[1][1]};
    *(u32x4*)(out + (long long)blocks * 512) = u32x4{m[0][0], m[0][1], m[1][0], m[1][1]};
    *(u32x4*)(out + (long long)blocks * 1024) = u32x4{l[0][0], l[0][1], l[1][0], l[1][1]};
  }
}

struct S3PGemm {
  const uint16_t *A, *B;                            // planes
  float* C;
  int blocksA, blocksB, ldc, M, N, Kc;
};

// C -= A B.  LOWER: the tiles that reach the lower triangle of a square C, a 1-D grid over 4 x 4 super-blocks;
// else a 2-D grid.  EDGE: M or N not in whole tiles.  Kc % 32 == 0.
template <bool EDGE, bool LOWER>
__global__ __launch_bounds__(256, 1) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_s3p_kernel(S3PGemm g, int gx, int gy) {
  typedef const __attribute__((address_space(3))) char* lds_ptr;
  typedef const __attribute__((address_space(3))) s3_bf16x8* lds_frag;
  __shared__ __attribute__((aligned(1024))) char lds[S3P_STAGES * S3P_STAGE];
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
  const int64_t slabA = (int64_t)g.blocksA * 1536, slabB = (int64_t)g.blocksB * 1536;       // elements
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds;
  const lds_ptr readA = (lds_ptr)lds + lane * 16 + wr * 4096, readB = (lds_ptr)lds + S3P_HALF + lane * 16 + wc * 4096;
  uint32_t gof[12];                                 // this wave's pieces of a slab: plane c / 8, block c % 8 of A, then of B
  #pragma unroll
  for (int p = 0; p < 6; ++p) {
    const int c = wave * 6 + p;
    gof[p] = ((uint32_t)(c >> 3) * g.blocksA + ti * 8 + (c & 7)) * 1024u + lane * 16;
    gof[6 + p] = ((uint32_t)(c >> 3) * g.blocksB + tj * 8 + (c & 7)) * 1024u + lane * 16;
  }
  const auto gload = [&](const uint16_t* a, const uint16_t* b, uint32_t dst, int p) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 ::"s"(dst + (p < 6 ? p * 1024 : S3P_HALF + (p - 6) * 1024)), "v"(gof[p]), "s"(p < 6 ? a : b) : "memory");
  };
  f32x16 acc[4][4];
  #pragma unroll
  for (int i = 0; i < 4; ++i)
    #pragma unroll
    for (int j = 0; j < 4; ++j)
      #pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  s3_bf16x8 fr[2][24];                              // two sets of operands: A hi 0..3, mid 4..7, lo 8..11, B hi 12..15, mid 16..19, lo 20..23
  const auto rd = [&](int set, int f, uint32_t stage) {
    const int q = f < 12 ? f : f - 12;
    fr[set][f] = *(lds_frag)((f < 12 ? readA : readB) + stage + (q >> 2) * 8192 + (q & 3) * 1024);
  };
  constexpr int FA[6] = {8, 0, 4, 4, 0, 0}, FB[6] = {12, 20, 16, 12, 16, 12};              // lo hi, hi lo, mid mid, mid hi, hi mid, hi hi

  // Past the last slab a load fetches the first one again (its stage is never read): the number in flight is always the same.
  #pragma unroll
  for (int s = 0; s < S3P_STAGES; ++s) {
    const int at = s < steps ? s : 0;
    #pragma unroll
    for (int p = 0; p < 12; ++p) gload(g.A + at * slabA, g.B + at * slabB, lds0 + s * S3P_STAGE + wave * 6144, p);
  }
  constexpr int FIRST = (S3P_STAGES - 1) * 12, LATER = (S3P_STAGES - 2) * 12;
  __builtin_amdgcn_s_waitcnt(0x0F70 | (FIRST & 15) | ((FIRST >> 4) << 14));
  __syncthreads();
  #pragma unroll
  for (int f = 0; f < 24; ++f) rd(0, f, 0);
  int s = 0;
  uint32_t cur = 0;
  __builtin_amdgcn_sched_barrier(0);
  const auto half = [&](int set) __attribute__((always_inline)) {
    // slab s is in every wave's registers (its stage takes slab s + 3), slab s + 1 has landed
    __builtin_amdgcn_s_waitcnt(0x0070 | (LATER & 15) | ((LATER >> 4) << 14));
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t nxt = (cur == (S3P_STAGES - 1) * S3P_STAGE) ? 0 : cur + S3P_STAGE;
    const int at = s + S3P_STAGES < steps ? s + S3P_STAGES : 0;
    const uint16_t* const a = g.A + at * slabA;
    const uint16_t* const b = g.B + at * slabB;
    #pragma unroll
    for (int m = 0; m < 96; ++m) {
      const int i = m & 3, j = (m >> 2) & 3, t = m >> 4;
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[set][FA[t] + i], fr[set][FB[t] + j], acc[i][j], 0, 0, 0);
      if (m >= 32 && m < 80 && !(m & 1)) rd(set ^ 1, (m - 32) / 2, nxt);   // (behind the products with lo: its registers are free)
      if (m % 8 == 7) gload(a, b, lds0 + cur + wave * 6144, m / 8);
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
  char* const out = (char*)(g.C + (int64_t)(ti * S3P_T) * g.ldc + tj * S3P_T);
  const uint32_t pitch = 4u * (uint32_t)g.ldc, at0 = row * pitch + 4 * col;
  const int rows = EDGE ? g.M - (ti * S3P_T + row) : S3P_T, cols = EDGE ? g.N - (tj * S3P_T + col) : S3P_T;
  const auto inside = [&](int i, int j, int r) { return !EDGE || (i * 32 + 8 * (r >> 2) + (r & 3) < rows && j * 32 < cols); };
  #pragma unroll
  for (int i = 0; i < 4; ++i) {
    // (the accumulators stay where they are until their turn: copied out together they would not fit the other registers)
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]));
    float old[4][16];
    uint32_t off[16];                               // 32-bit offsets from the tile's corner; j * 128 goes into the instruction
    #pragma unroll
    for (int r = 0; r < 16; ++r) off[r] = at0 + (i * 32 + 8 * (r >> 2) + (r & 3)) * pitch;
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
        const float w = old[j][r] - acc[i][j][r];
        if (inside(i, j, r)) *(float*)(out + (uint64_t)off[r] + j * 128) = w;
      }
  }
}

// Operands in memory of s3p_bytes(rows, Kc), 16-byte aligned.
struct S3POperand {
  uint16_t* planes;
  int blocks;
  S3POperand(void* p, int64_t rows) : planes((uint16_t*)p), blocks((int)(s3p_rows(rows) / 32)) {}
};
template <bool T>
inline void s3p_pack(const float* src, int64_t ld, int rows, int Kc, const S3POperand& o, hipStream_t st) {
  s3p_pack_kernel<T><<<dim3((unsigned)o.blocks), dim3(256), 0, st>>>(src, ld, rows, Kc, o.blocks, o.planes);
}

// (Depths from 512 on: the shallower launches of the chain and of the loop are narrow ones.)  May a row-major operand [rows, Kc] be packed?  (One given as [Kc, rows] only needs the depth.)
inline bool s3p_depth(int64_t Kc) { return Kc % 64 == 0 && Kc >= 512 && Kc <= S3P_MAX_K; }
inline bool s3p_operand(const float* p, int64_t ld, int64_t Kc) { return s3p_depth(Kc) && ld % 4 == 0 && (uintptr_t)p % 16 == 0; }
// Up to 128 of the 256 x 256 tiles the 128 x 128 tiles of gemm_s3_kernel are one round of its two workgroups per CU and
// faster (us, theirs against these): 4096 x 2048 x 1024, 128 tiles, 102 / 125; 4096 x 2304, 144 tiles, 161 / 126; 4096 x 4096,
// 256 tiles, 197 / 170; 4096 x 4352, 272 tiles, 262 / 260; 4096 x 8192 385 / 325.  With a short side packing the long one costs
// more than is won: 28672 x 512 x 1024 183 / 210, 14336 x 768 x 1024 173 / 148.  At a depth of 512 the lines are the same.
inline bool s3p_pays(int64_t M, int64_t N, int64_t tiles) { return tiles > 128 && M > 512 && N > 512; }
inline int64_t s3p_tiles(int64_t M, int64_t N) { return ((M + S3P_T - 1) / S3P_T) * ((N + S3P_T - 1) / S3P_T); }

// C [M, N] -= A B^T.  LOWER: M == N, the tiles on and below the diagonal.
template <bool LOWER>
inline void s3p_multiply(const S3POperand& a, const S3POperand& b, float* C, int ldc, int M, int N, int Kc, hipStream_t st) {
  const S3PGemm g{a.planes, b.planes, C, a.blocks, b.blocks, ldc, M, N, Kc};
  const int gx = (N + S3P_T - 1) / S3P_T, gy = (M + S3P_T - 1) / S3P_T, nsb = (gy + 3) / 4;
  const unsigned grid = LOWER ? (unsigned)(16 * (nsb * (nsb + 1) / 2)) : (unsigned)(gx * gy);
  if (M % S3P_T != 0 || N % S3P_T != 0) gemm_s3p_kernel<true, LOWER><<<dim3(grid), dim3(256), 0, st>>>(g, gx, gy);
  else gemm_s3p_kernel<false, LOWER><<<dim3(grid), dim3(256), 0, st>>>(g, gx, gy);
}

}  // namespace lcq
