// Damped Cholesky chain of GPTQ for gfx950.
//
// Replaces, in GPTQ.process_hessian_and_weights (gptq.py:139-141, 150-153, 169-174):
//   dead = diag(H) == 0; H[dead, dead] = 1; W[:, dead] = 0
//   H = H[perm][:, perm]
//   H += percdamp * mean(diag(H)) * I
//   H = cholesky(H); H = cholesky_inverse(H); H = cholesky(H, upper=True)
// The result U is upper triangular with U^T U = (H + damp I)^-1.
//
// Instead of three factorizations (4/3 K^3 flop) the chain is computed as
//   J H J = L L^T  (J = index reversal, L lower)   ->   U = J L^-1 J,
// one Cholesky plus one triangular inverse (2/3 K^3 flop): L^-1 lower with a
// positive diagonal, reversed on both axes, is upper triangular and
// (J L^-1 J)^T (J L^-1 J) = J (L L^T)^-1 J = H^-1, so it IS the unique upper
// Cholesky factor of H^-1.
//
// Kernels
//   diag_prep      diagonal scan: dead columns, mean(diag) -> damp
//   build          gather  A[a][b] = H[p(K-1-a)][p(K-1-b)] (+damp on the diagonal), a >= b
//   potrf_diag     128x128 diagonal block in LDS: L11 and L11^-1 (one workgroup)
//   gemm_f32       fp32 MFMA: panel solve  A21 <- A21 L11^-T  and trailing  A22 -= A21 A21^T
//   (batched)      triangular inverse by pairwise merging of inverted diagonal
//                  blocks: [[A,0],[B,C]]^-1 = [[A^-1,0],[-C^-1 B A^-1, C^-1]]
//   scatter        U[i][j] = Linv[K-1-i][K-1-j], j >= i; zeros below the diagonal
#include <mutex>
#include <type_traits>
#include "gemm_f32.h"
#include "gemm_s3p.h"
#include "lcq_internal.h"

namespace lcq {
std::atomic<int> g_gemm_split{1};
}

namespace {
using namespace lcq;

constexpr int NB = 128;

struct PrepScalars {
  float damp;
  int status;      // 0 ok, 1 non-positive pivot met
};

// one workgroup: dead-column fix on the diagonal, damp = percdamp * mean(diag)
__global__ __launch_bounds__(1024) void diag_prep_kernel(float* __restrict__ H, int K, float percdamp,
                                                         uint8_t* __restrict__ dead, PrepScalars* sc) {
  __shared__ float part[16];
  float s = 0.0f;
  for (int j = threadIdx.x; j < K; j += 1024) {
    float d = H[(long long)j * K + j];
    const bool is_dead = (d == 0.0f);
    if (is_dead) { d = 1.0f; H[(long long)j * K + j] = 1.0f; }
    dead[j] = is_dead;
    s += d;
  }
  s = team_sum<64>(s);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.0f;
    for (int i = 0; i < 16; ++i) t += part[i];
    sc->damp = percdamp * (t * (1.0f / (float)K));     // torch.mean on the GPU: the sum times an fp32 factor
    sc->status = 0;
  }
}

// W[:, dead] = 0
__global__ __launch_bounds__(256) void apply_dead_kernel(float* __restrict__ W, long long R, int K,
                                                         const uint8_t* __restrict__ dead) {
  const long long n = R * K;
  for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long long)gridDim.x * 256)
    if (dead[e % K]) W[e] = 0.0f;
}

// W[r, j] = dead[c] ? 0 : float(w[r, c]),  c = perm ? perm[j] : j   -- the weight clone, fp32 cast, dead-column
// zeroing and act-order gather of process_hessian_and_weights (gptq.py:133-141, 150-151) in one pass.  A workgroup
// takes 4 rows; without a permutation reads and writes are both coalesced.
template <int DT>
__device__ __forceinline__ float load_w(const void* w, long long i) {
  if (DT == LCQ_F32) return ((const float*)w)[i];
  if (DT == LCQ_BF16) return u2f((uint32_t)((const uint16_t*)w)[i] << 16);
  return (float)((const _Float16*)w)[i];
}
template <int DT>
__global__ __launch_bounds__(256) void prepare_w_kernel(const void* __restrict__ w, long long R, int K,
                                                        const long long* __restrict__ perm,
                                                        const uint8_t* __restrict__ dead, float* __restrict__ out) {
  for (long long row = (long long)blockIdx.x * 4; row < R && row < (long long)blockIdx.x * 4 + 4; ++row) {
    for (int j = threadIdx.x; j < K; j += 256) {
      const long long c = perm ? perm[j] : j;
      float v = load_w<DT>(w, row * K + c);
      if (dead && dead[c]) v = 0.0f;
      out[row * K + j] = v;
    }
  }
}
// The same without a permutation, 16 bytes per lane (K in whole chunks, everything aligned): four rows per workgroup.
template <int DT>
__global__ __launch_bounds__(256) void prepare_w_vec_kernel(const u32x4* __restrict__ w, long long R, int K,
                                                            const uint8_t* __restrict__ dead, f32x4* __restrict__ out) {
  constexpr int N = DT == LCQ_F32 ? 4 : 8;
  const long long row0 = (long long)blockIdx.x * 4;
  const int cpr = K / N, n = (R - row0 < 4 ? (int)(R - row0) : 4) * cpr;
  for (int e = threadIdx.x; e < n; e += 256) {
    const long long at = row0 * cpr + e;
    const u32x4 raw = w[at];
    float v[N];
    #pragma unroll
    for (int i = 0; i < N; ++i) v[i] = load_w<DT>(&raw, i);
    if (dead) {
      const uint8_t* d = dead + (long long)(e % cpr) * N;
      #pragma unroll
      for (int i = 0; i < N; ++i) v[i] = d[i] ? 0.0f : v[i];
    }
    #pragma unroll
    for (int i = 0; i < N; i += 4) out[at * (N / 4) + i / 4] = f32x4{v[i], v[i + 1], v[i + 2], v[i + 3]};
  }
}
// `n` pieces to LDS, eight loads in flight per thread (one load at a time is a memory latency per piece and thread).
template <int THREADS, class V>
__device__ __forceinline__ void pieces_to_lds(V* to, const V* from, int n) {
  int i0 = threadIdx.x;
  for (; i0 + 7 * THREADS < n; i0 += 8 * THREADS) {
    V v[8];
    #pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = from[i0 + k * THREADS];
    #pragma unroll
    for (int k = 0; k < 8; ++k) to[i0 + k * THREADS] = v[k];
  }
  for (; i0 < n; i0 += 2 * THREADS) {
    const bool two = i0 + THREADS < n;
    const V v = from[i0], w = from[two ? i0 + THREADS : i0];
    to[i0] = v;
    if (two) to[i0 + THREADS] = w;
  }
}
// Row-major elements to LDS (`to` on 16 bytes): 16 bytes per thread, or element by element where they do not start on 16 bytes.
template <int THREADS, class E>
__device__ __forceinline__ void rows_to_lds(E* to, const E* from, int n) {
  if ((((uintptr_t)from) & 15) != 0) { pieces_to_lds<THREADS>(to, from, n); return; }
  constexpr int PER = 16 / (int)sizeof(E);
  pieces_to_lds<THREADS>((u32x4*)to, (const u32x4*)from, n / PER);
  for (int i = n / PER * PER + threadIdx.x; i < n; i += THREADS) to[i] = from[i];
}

// The same with a permutation: a gather inside every row.  From memory that is one 64-byte sector per element; here
// the workgroup's rows (`rows` of them, as many as fit 64 KB) come in as they lie, and the gather reads LDS, four columns per thread
// where K allows it.  The permutation is read once per workgroup and column.
// HBM-bound: 14336 x 4096 bf16 91 -> 68 us, 4096 x 14336 fp32 251 -> 110 (one load in flight per thread and 4-byte stores before).
template <int DT>
__global__ __launch_bounds__(512) void prepare_w_gather_kernel(const void* __restrict__ w, long long R, int K, int rows,
                                                               const long long* __restrict__ perm,
                                                               const uint8_t* __restrict__ dead, float* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char staged[];
  typedef typename std::conditional<DT == LCQ_F32, float, uint16_t>::type Element;
  const long long row0 = (long long)blockIdx.x * rows;
  const int n = (int)((R - row0 < rows) ? (R - row0) : rows);
  rows_to_lds<512>((Element*)staged, (const Element*)w + row0 * K, n * K);
  __syncthreads();
  if (K % 4 == 0 && (((uintptr_t)out) & 15) == 0) {
    for (int j = 4 * threadIdx.x; j < K; j += 2048) {
      int c[4];
      bool dz[4];
      #pragma unroll
      for (int e = 0; e < 4; ++e) { c[e] = (int)perm[j + e]; dz[e] = dead && dead[c[e]]; }
      for (int r = 0; r < n; ++r) {
        f32x4 v;
        #pragma unroll
        for (int e = 0; e < 4; ++e) { const float x = load_w<DT>(staged, (long long)(r * K + c[e])); v[e] = dz[e] ? 0.0f : x; }
        *(f32x4*)(out + (row0 + r) * K + j) = v;
      }
    }
    return;
  }
  for (int j = threadIdx.x; j < K; j += 512) {
    const long long c = perm[j];
    const bool dz = dead && dead[c];
    for (int r = 0; r < n; ++r) {
      const float v = load_w<DT>(staged, (long long)r * K + c);
      out[(row0 + r) * K + j] = dz ? 0.0f : v;
    }
  }
}

// A (lower triangle, reversed + permuted + damped); strict upper triangle zeroed
__global__ __launch_bounds__(256) void build_kernel(const float* __restrict__ H, int K, const long long* __restrict__ perm,
                                                    const PrepScalars* __restrict__ sc, float* __restrict__ A) {
  const int a = blockIdx.y;
  const int b = blockIdx.x * 256 + threadIdx.x;
  if (b >= K) return;
  float v = 0.0f;
  if (b <= a) {
    long long i = K - 1 - a, j = K - 1 - b;
    if (perm) { i = perm[i]; j = perm[j]; }
    const long long lo = i < j ? i : j, hi = i < j ? j : i;     // H is valid on and above the diagonal
    v = H[lo * K + hi];
    if (a == b) v += sc->damp;
  }
  A[(long long)a * K + b] = v;
}

// The same from a fully symmetric H and with a permutation: row a of A draws on row perm[K-1-a] of H only, which
// comes in as it lies (16 bytes per lane) and is gathered from LDS.  (Picking H[min][max] from memory, as build_kernel
// does, walks down a column of H for half of the entries: one 64-byte sector per element.)
// HBM-bound at large K: K = 14336 567 -> 298 us, 8192 121 -> 96, 4096 22.0 -> 18.5, 2048 10.3 -> 7.8, 1280 6.5 -> 6.0 (256 threads, one load in flight, the
// permutation read behind the row and 4-byte stores before; kernel traces).
// V: K a multiple of 4, at most 4 Q THREADS, and H on 16 bytes: a thread's pieces of the row and its columns of the permutation are all in flight (the
// permutation first: it waits for nothing), no more threads or columns than a row has.  (512 threads for 16384 columns, whatever K: 7.6 us at 1280, 15.3 at
// 3000, where 6.5 and 13.9 were taken before.)  Otherwise a column per thread, Q of the permutation in flight, rows that may start off 16 bytes, then
// staged by 4: K = 2047 8.9 us (9.0 before; 15.3 staged byte by byte), 4095 24.4 (24.4; 41), 14335 406 (1040; 700).
template <bool V, int THREADS, int Q>
__global__ __launch_bounds__(THREADS) void build_gather_kernel(const float* __restrict__ H, int K, const long long* __restrict__ perm,
                                                               const PrepScalars* __restrict__ sc, float* __restrict__ A) {
  extern __shared__ __align__(16) float hrow[];
  const int a = blockIdx.x;
  const float damp = sc->damp;
  if constexpr (V) {
    int c[Q][4];
    #pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int b = 4 * (threadIdx.x + THREADS * q);
      if (b < K && b <= a)
        #pragma unroll
        for (int e = 0; e < 4; ++e) c[q][e] = (int)perm[K - 1 - b - e];
    }
    const float* const row = H + perm[K - 1 - a] * (long long)K;
    f32x4 piece[Q];
    #pragma unroll
    for (int q = 0; q < Q; ++q) piece[q] = *(const f32x4*)(row + min(4 * (int)(threadIdx.x + THREADS * q), K - 4));
    #pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int b = 4 * (threadIdx.x + THREADS * q);
      if (b < K) *(f32x4*)(hrow + b) = piece[q];
    }
    __syncthreads();
    #pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int b = 4 * (threadIdx.x + THREADS * q);
      if (b < K) {
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        if (b <= a)
          #pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float h = hrow[c[q][e]];                  // (columns past the diagonal too: every entry of perm is one of H)
            v[e] = b + e < a ? h : b + e == a ? h + damp : 0.0f;
          }
        *(f32x4*)(A + (long long)a * K + b) = v;
      }
    }
  } else {
    rows_to_lds<THREADS>(hrow, H + perm[K - 1 - a] * (long long)K, K);
    __syncthreads();
    for (int b0 = threadIdx.x; b0 < K; b0 += Q * THREADS) {
      int c[Q];
      #pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int b = b0 + THREADS * q;
        if (b < K && b <= a) c[q] = (int)perm[K - 1 - b];
      }
      #pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int b = b0 + THREADS * q;
        if (b < K) A[(long long)a * K + b] = b > a ? 0.0f : b == a ? hrow[c[q]] + damp : hrow[c[q]];
      }
    }
  }
}
// K <= 16384: a row of H fits the 64 KB of LDS a workgroup may ask for
static void launch_build_gather(const float* H, int K, const long long* perm, const PrepScalars* sc, float* A, hipStream_t st) {
  const dim3 grid((unsigned)K);
  const size_t lds = (size_t)K * 4;
  if (K % 4 != 0 || ((uintptr_t)H & 15) != 0) {
    if (K <= 4096) build_gather_kernel<false, 256, 4><<<grid, dim3(256), lds, st>>>(H, K, perm, sc, A);
    else build_gather_kernel<false, 512, 4><<<grid, dim3(512), lds, st>>>(H, K, perm, sc, A);
  }
  else if (K <= 1024) build_gather_kernel<true, 256, 1><<<grid, dim3(256), lds, st>>>(H, K, perm, sc, A);
  else if (K <= 2048) build_gather_kernel<true, 256, 2><<<grid, dim3(256), lds, st>>>(H, K, perm, sc, A);
  else if (K <= 4096) build_gather_kernel<true, 512, 2><<<grid, dim3(512), lds, st>>>(H, K, perm, sc, A);
  else if (K <= 8192) build_gather_kernel<true, 512, 4><<<grid, dim3(512), lds, st>>>(H, K, perm, sc, A);
  else build_gather_kernel<true, 512, 8><<<grid, dim3(512), lds, st>>>(H, K, perm, sc, A);
}

// Diagonal block: Cholesky factor L11 of a 128x128 block and the inverse of L11, one workgroup of 8 waves.
// A wave that is alone on its SIMD issues about one instruction per 8 cycles, so what counts is how many instructions the serial
// part needs.  The 128 columns are 8 panels of 16; everything that is not the pivot chain of a panel runs on the fp32 matrix pipe:
//   * the panel waves (4, 6, 7) take a panel from LDS with one row per lane and factor it without barriers.  A column costs one
//     v_readlane (the pivot), a reciprocal square root, one product and at most four v_mfma_f32_4x4x1_16b: 16 blocks of 4 x 4 are
//     64 rows x 4 columns, and with the A operand of ONE block broadcast to all of them (cbsz = 4, abid = the quad of lanes that
//     holds the rows these columns belong to) one instruction is the rank-1 update of four columns for all rows of the wave.
//     The rows of an identity ride along behind the panel's: they come out as the transposed inverse of its 16 x 16 block.
//   * the update waves (1, 2, 3, 5) hold the lower triangle behind in 16 x 16 tiles, the accumulators of v_mfma_f32_16x16x4f32
//     (wave u tile rows u and 7 - u).  They apply a finished panel first to the next panel's columns, hand those over, and do the
//     rest of the update while the panel waves are factoring (a right-looking update with look-ahead; two barriers per panel).
//   * They also build the inverse beside the panels, a column block j per wave and half: X_Pj = -X_PP T_Pj goes to memory, and from the
//     registers it is in to the rows below, T_rj += L_rP X_Pj: products that do not wait for one another.  Behind the last
//     panel only X_7j is left.  (T of a row summed up when its turn comes, one chain of up to 28 products: 1.5 us more per block.)
// Contractions take k = 4 (l / 16) + i in instruction i, so an operand is one 16-byte read of a row and an accumulator is the B
// operand of the next product as it stands.  The panels and tiles hold -A, so that updates add.
// Bound by the serial chain of one wave's instructions: 12.5 us per block (26.4 us with updates of 8 x 8 values per thread, 240
// v_readlane / v_fma per panel and the inverse by three levels of merges at the end).
constexpr int LP = NB + 4;       // row pitch of the LDS matrices (16-byte aligned rows, 4-bank skew)
constexpr int PP = 16 + 4;       // row pitch of the panel

struct PotrfLds {
  float L[NB][LP];       // L row-major, below the 16 x 16 diagonal blocks
  float XT[8][16][PP];   // the inverted diagonal blocks, transposed: XT[i][c][r] = X(16 i + r, 16 i + c), X = L^-1
  float Pn[NB + 16][PP]; // - the panel on its way to the panel waves, and behind it - the identity
};

__device__ __forceinline__ float rdlane(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// Panel P: columns 16 P .. +15.  Lanes 0 .. 15 of every panel wave hold the panel's own 16 rows (pivots and multipliers come from
// there), the other 48 lanes the rows behind them and then 16 rows of the identity, dealt to as many waves as they need.
// `least` gathers the pivots (NaN stays).
__device__ __forceinline__ void potrf_panel(PotrfLds& s, int P, int w, int lane, float& least) {
  #pragma clang fp contract(fast)   // the residual of the reciprocal square root as FMAs
  const int behind = NB - 16 * P - 16;                      // rows behind the panel's own
  const int q = lane - 16 + 48 * w;                         // this lane's row among those and the identity's
  const bool own = lane < 16, rest = !own && q < behind, unit = !own && q >= behind && q < behind + 16;
  const float* const from = s.Pn[own ? 16 * P + lane : 16 * P + 16 + q];        // (the identity follows row 127)
  f32x4 n[4];
  #pragma unroll
  for (int b = 0; b < 4; ++b) n[b] = *(const f32x4*)((own || rest || unit ? from : s.Pn[0]) + 4 * b);
  f32x4 l[4];
  #pragma unroll
  for (int j = 0; j < 16; ++j) {
    const float x = n[j >> 2][j & 3], piv = -rdlane(x, j);
    least = nan_min(least, piv);
    const float r = __builtin_amdgcn_rsqf(piv);             // 1/sqrt(pivot), one Newton step to full precision
    const float v = x * -(r + (0.5f * r) * (1.0f - (piv * r) * r));
    l[j >> 2][j & 3] = v;                                   // (own rows above the diagonal hold garbage; nothing reads it)
    // columns from j + 1 on; those of j's own four that are done pick up garbage
    if (j < 3) n[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(v, v, n[0], 4, 0, 0);
    if (j < 7) n[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(v, v, n[1], 4, 1, 0);
    if (j < 11) n[2] = __builtin_amdgcn_mfma_f32_4x4x1f32(v, v, n[2], 4, 2, 0);
    if (j < 15) n[3] = __builtin_amdgcn_mfma_f32_4x4x1f32(v, v, n[3], 4, 3, 0);
  }
  if (rest || unit) {
    float* const to = rest ? &s.L[16 * P + 16 + q][16 * P] : s.XT[P][q - behind];
    #pragma unroll
    for (int b = 0; b < 4; ++b) *(f32x4*)(to + 4 * b) = l[b];
  }
}

// c + sum over 16 of the contraction: a and b as read from rows (lane l: row l % 16, k = 4 (l / 16) + i in element i)
__device__ __forceinline__ f32x4 potrf_mac(const f32x4& a, const f32x4& b, f32x4 c) {
  #pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}

// What an update wave holds: tile rows u (`top`) and 7 - u (`bottom`), tile (i, j) transposed: lane element e is row 16 i + l % 16, column
// 16 j + 4 (l / 16) + e; and what the rows below still lack of column blocks u and 7 - u of the inverse, T[.][r] = sum L_rk X_kj.
struct PotrfTiles { f32x4 top[4], bottom[8], T[2][8]; };

// the columns of panel J to the panel waves
template <int J>
__device__ __forceinline__ void potrf_publish(PotrfLds& s, const PotrfTiles& t, int u, int m, int g) {
  if constexpr (J < 4) { if (u >= J) *(f32x4*)(s.Pn[16 * u + m] + 4 * g) = t.top[J]; }
  if (7 - u >= J) *(f32x4*)(s.Pn[16 * (7 - u) + m] + 4 * g) = t.bottom[J];
}

// Column block j of the inverse, beside panel I + 1: X_Ij of tile row I, whose own block has been inverted, and its part in the rows below
// (l[r]: row r of L's panel I, as the first operand).
template <int I>
__device__ __forceinline__ void potrf_inverse(const PotrfLds& s, f32x4 (&T)[8], int j, const f32x4 (&x)[2], const f32x4 (&l)[8], int nb,
                                              float* __restrict__ Dinv, int m, int g) {
  if (I < j) return;
  f32x4 v;                                                  // X_Ij: rows 4 g + e, column m
  if (I == j) {
    v = x[1];
    #pragma unroll
    for (int r = I + 1; r < 8; ++r) T[r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  } else {
    v = -potrf_mac(x[0], T[I], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
  }
  #pragma unroll
  for (int e = 0; e < 4; ++e)                               // (the padding's diagonal is no part of the inverse)
    Dinv[(16 * I + 4 * g + e) * NB + 16 * j + m] = 16 * I + 4 * g + e < nb ? v[e] : 0.0f;
  #pragma unroll
  for (int e = 0; e < 4; ++e)
    #pragma unroll
    for (int r = I + 1; r < 8; ++r) T[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(l[r][e], v[e], T[r], 0, 0, 0);
}

// what an update wave does with panel P once that is complete, but for the next panel's columns
template <int P>
__device__ __forceinline__ void potrf_rest(const PotrfLds& s, PotrfTiles& t, int u, int nb, float* __restrict__ Dinv, int m, int g) {
  f32x4 l[8], x[2];                                         // rows of L's panel P; X_PP(m, 4 g + e) and X_PP(4 g + e, m)
  #pragma unroll
  for (int r = P + 1; r < 8; ++r) l[r] = *(const f32x4*)(s.L[16 * r + m] + 16 * P + 4 * g);
  const f32x4 hi = *(const f32x4*)(s.L[16 * (7 - u) + m] + 16 * P + 4 * g);
  const f32x4 lo = *(const f32x4*)(s.L[16 * u + m] + 16 * P + 4 * g);         // (used only where u > P)
  #pragma unroll
  for (int e = 0; e < 4; ++e) x[0][e] = s.XT[P][4 * g + e][m];
  x[1] = *(const f32x4*)(s.XT[P][m] + 4 * g);
  #pragma unroll
  for (int j = P + 2; j < 8; ++j) {
    if (j <= 7 - u) t.bottom[j] = potrf_mac(l[j], hi, t.bottom[j]);
    if (j < 4 && j <= u) t.top[j & 3] = potrf_mac(l[j], lo, t.top[j & 3]);
  }
  potrf_inverse<P>(s, t.T[0], u, x, l, nb, Dinv, m, g);
  potrf_inverse<P>(s, t.T[1], 7 - u, x, l, nb, Dinv, m, g);
}

template <int P>
__device__ __forceinline__ void potrf_phase(PotrfLds& s, PotrfTiles& t, int u, int nb, float* __restrict__ Dinv, int m, int g) {
  __syncthreads();                                          // Pn holds panel P
  if constexpr (P > 0) potrf_rest<P - 1>(s, t, u, nb, Dinv, m, g);
  __syncthreads();                                          // L of panel P and its inverted block are complete
  if constexpr (P < 7) {
    const f32x4 a = *(const f32x4*)(s.L[16 * (P + 1) + m] + 16 * P + 4 * g);
    const f32x4 hi = *(const f32x4*)(s.L[16 * (7 - u) + m] + 16 * P + 4 * g), lo = *(const f32x4*)(s.L[16 * u + m] + 16 * P + 4 * g);
    if (P + 1 <= 7 - u) t.bottom[P + 1] = potrf_mac(a, hi, t.bottom[P + 1]);
    if constexpr (P < 3) { if (P + 1 <= u) t.top[P + 1] = potrf_mac(a, lo, t.top[P + 1]); }
    potrf_publish<P + 1>(s, t, u, m, g);
  }
}

__global__ __launch_bounds__(512) void potrf_diag_kernel(const float* __restrict__ Ablk, int lda, int nb,
                                                         float* __restrict__ Dinv, PrepScalars* sc) {
  __shared__ __align__(16) PotrfLds s;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int panels = 8;
  asm volatile("" : "+s"(panels));                          // (or the loops over the panels are unrolled, and wait for instruction fetches)
  if (wave == 0 || wave == 4 || wave >= 6) {
    if (wave == 0) {                                        // the tiles above the diagonal are zeros
      for (int r = 0; r < NB - 16; r += 2) {
        const int row = r + (lane >> 5), c4 = (lane & 31) * 4;
        if (c4 >= (row & ~15) + 16) *(f32x4*)(Dinv + row * NB + c4) = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
    if (wave == 6) {
      #pragma unroll
      for (int e = 0; e < 4; ++e) s.Pn[NB + m][4 * g + e] = 4 * g + e == m ? -1.0f : 0.0f;
    }
    float least = __builtin_inff();
    const int w = wave == 0 ? 3 : wave == 4 ? 0 : wave - 5;                   // wave 0 has no rows: NB <= 3 x 48
    #pragma unroll 1
    for (int P = 0; P < panels; ++P) {
      __syncthreads();
      if (48 * w < NB - 16 * P) potrf_panel(s, P, w, lane, least);
      __syncthreads();
    }
    if (wave == 4 && lane == 0 && !(least > 0.0f)) sc->status = 1;
    return;
  }
  // the busiest first, on the SIMD that panels leave first; the two that share one are among the others (u in the order 5, 1, 2, 3:
  // 1 us more per block)
  const int u = wave == 3 ? 0 : wave == 1 ? 1 : wave == 5 ? 2 : 3;
  PotrfTiles t;
  // a whole block: plain loads, all in flight (those above the diagonal are never used)
  if (nb == NB && lda % 4 == 0 && ((uintptr_t)Ablk & 15) == 0) {
    const float* const pt = Ablk + (long long)(16 * u + m) * lda + 4 * g;
    const float* const pb = Ablk + (long long)(16 * (7 - u) + m) * lda + 4 * g;
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < 4) t.top[j & 3] = *(const f32x4*)(pt + 16 * j);
      t.bottom[j] = *(const f32x4*)(pb + 16 * j);
    }
  } else {
    const auto load = [&](int i, int j, f32x4& v) {
      const int r = 16 * i + m, c = 16 * j + 4 * g;
      #pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (r < nb && c + e <= r) ? Ablk[(long long)r * lda + c + e] : (r == c + e) ? 1.0f : 0.0f;   // pad with identity
    };
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < 4) load(u, j, t.top[j & 3]);
      load(7 - u, j, t.bottom[j]);
    }
  }
  #pragma unroll
  for (int j = 0; j < 8; ++j)
    #pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (j < 4) t.top[j & 3][e] = (j < u || 4 * g + e <= m) ? -t.top[j & 3][e] : 0.0f;
      t.bottom[j][e] = (j < 7 - u || 4 * g + e <= m) ? -t.bottom[j][e] : 0.0f;
    }
  potrf_publish<0>(s, t, u, m, g);
  potrf_phase<0>(s, t, u, nb, Dinv, m, g);
  potrf_phase<1>(s, t, u, nb, Dinv, m, g);
  potrf_phase<2>(s, t, u, nb, Dinv, m, g);
  potrf_phase<3>(s, t, u, nb, Dinv, m, g);
  potrf_phase<4>(s, t, u, nb, Dinv, m, g);
  potrf_phase<5>(s, t, u, nb, Dinv, m, g);
  potrf_phase<6>(s, t, u, nb, Dinv, m, g);
  potrf_phase<7>(s, t, u, nb, Dinv, m, g);
  potrf_rest<7>(s, t, u, nb, Dinv, m, g);
  // (L itself is not written back: everything after this kernel works with the inverse, the solved panels and the
  // blocks behind them; place_diag_kernel puts the inverse where the block was.)
}

// copy the inverted diagonal blocks into place, eight rows per workgroup
__global__ __launch_bounds__(256) void place_diag_kernel(float* __restrict__ A, int K, const float* __restrict__ Dinv) {
  const int blk = blockIdx.x, k0 = blk * NB;
  const int nb = min(NB, K - k0);
  const float* D = Dinv + (long long)blk * NB * NB;
  for (int e = threadIdx.x; e < 8 * NB; e += 256) {
    const int r = blockIdx.y * 8 + e / NB, c = e % NB;
    if (r < nb && c < nb) A[(long long)(k0 + r) * K + k0 + c] = D[r * NB + c];
  }
}

// U[i][j] = Linv[K-1-i][K-1-j], zeros below the diagonal.  With `Dinv` (K in whole blocks) the diagonal blocks come from there.
// V: four columns per thread (K a multiple of 4, U on 16 bytes): K = 14336 412 -> 187 us,
// 4096 28 -> 16, which workgroups of 256 single elements took to start.
template <bool V>
__global__ __launch_bounds__(256) void scatter_kernel(const float* __restrict__ Linv, int K, const float* __restrict__ Dinv,
                                                      float* __restrict__ U) {
  const int i = blockIdx.y, a = K - 1 - i;
  const int j = (blockIdx.x * 256 + threadIdx.x) * (V ? 4 : 1);
  if (j >= K) return;
  if constexpr (V) {
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (j + 3 >= i) {
      const int b = K - 4 - j;                              // columns b .. b + 3, the last one first
      const f32x4 x = *(const f32x4*)(Dinv && a / NB == b / NB ? Dinv + (long long)a * NB + b % NB : Linv + (long long)a * K + b);
      #pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = j + e >= i ? x[3 - e] : 0.0f;
    }
    *(f32x4*)(U + (long long)i * K + j) = v;
  } else {
    const int b = K - 1 - j;
    float v = 0.0f;
    if (j >= i) v = (Dinv && a / NB == b / NB) ? Dinv[(long long)a * NB + b % NB] : Linv[(long long)a * K + b];
    U[(long long)i * K + j] = v;
  }
}
static void launch_scatter(const float* Linv, int K, const float* Dinv, float* U, hipStream_t st) {
  if (K % 4 == 0 && ((uintptr_t)U & 15) == 0) scatter_kernel<true><<<dim3((unsigned)((K + 1023) / 1024), (unsigned)K), dim3(256), 0, st>>>(Linv, K, Dinv, U);
  else scatter_kernel<false><<<dim3((unsigned)((K + 255) / 256), (unsigned)K), dim3(256), 0, st>>>(Linv, K, Dinv, U);
}

}  // namespace

// super-panels of the factorization, and the workspace in front of the packed one
constexpr int NBO = 4 * NB;
static int64_t chol_base_bytes(int64_t K, int64_t nblk) {
  return (K * K * 4 + nblk * NB * NB * 4 + ((K + 255) / 256) * 256 + 256 + 255) / 256 * 256;
}

extern "C" {

int64_t lcq_chol_inv_upper_workspace_bytes(int64_t K) {
  const int64_t nblk = (K + NB - 1) / NB;
  return chol_base_bytes(K, nblk) + s3p_bytes(K, NBO);
}

int lcq_set_gemm_split(int on) {
  return g_gemm_split.exchange(on ? 1 : 0);
}

int lcq_gptq_prepare_weights(const void* w, int dtype, int64_t R, int64_t K, const int64_t* perm, const uint8_t* dead,
                             float* out, void* stream) {
  if (!w || !out || R <= 0 || K <= 0 || K > 0x7fffffff || (const void*)out == w) return LCQ_EINVAL;
  const int64_t grid = (R + 3) / 4;
  if (grid > 0x7fffffff) return LCQ_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  const long long* p = (const long long*)perm;
  const int es = dtype == LCQ_F32 ? 4 : 2;
  if (p && K * es <= 65536 && (dtype == LCQ_F32 || dtype == LCQ_BF16 || dtype == LCQ_F16)) {   // gather through LDS
    int rows = (int)(65536 / (K * es));
    if (rows > 8) rows = 8;
    const int64_t g = (R + rows - 1) / rows;
    if (g > 0x7fffffff) return LCQ_EINVAL;
    const size_t lds = (size_t)rows * K * es;
    if (dtype == LCQ_F32) prepare_w_gather_kernel<LCQ_F32><<<dim3((unsigned)g), dim3(512), lds, st>>>(w, R, (int)K, rows, p, dead, out);
    else if (dtype == LCQ_BF16) prepare_w_gather_kernel<LCQ_BF16><<<dim3((unsigned)g), dim3(512), lds, st>>>(w, R, (int)K, rows, p, dead, out);
    else prepare_w_gather_kernel<LCQ_F16><<<dim3((unsigned)g), dim3(512), lds, st>>>(w, R, (int)K, rows, p, dead, out);
  }
  else if (!p && K % 8 == 0 && K <= (1 << 28) && ((uintptr_t)w & 15) == 0 && ((uintptr_t)out & 15) == 0 &&
           (dtype == LCQ_F32 || dtype == LCQ_BF16 || dtype == LCQ_F16)) {
    const u32x4* src = (const u32x4*)w;
    f32x4* dst = (f32x4*)out;
    if (dtype == LCQ_F32) prepare_w_vec_kernel<LCQ_F32><<<dim3((unsigned)grid), dim3(256), 0, st>>>(src, R, (int)K, dead, dst);
    else if (dtype == LCQ_BF16) prepare_w_vec_kernel<LCQ_BF16><<<dim3((unsigned)grid), dim3(256), 0, st>>>(src, R, (int)K, dead, dst);
    else prepare_w_vec_kernel<LCQ_F16><<<dim3((unsigned)grid), dim3(256), 0, st>>>(src, R, (int)K, dead, dst);
  }
  else if (dtype == LCQ_F32) prepare_w_kernel<LCQ_F32><<<dim3((unsigned)grid), dim3(256), 0, st>>>(w, R, (int)K, p, dead, out);
  else if (dtype == LCQ_BF16) prepare_w_kernel<LCQ_BF16><<<dim3((unsigned)grid), dim3(256), 0, st>>>(w, R, (int)K, p, dead, out);
  else if (dtype == LCQ_F16) prepare_w_kernel<LCQ_F16><<<dim3((unsigned)grid), dim3(256), 0, st>>>(w, R, (int)K, p, dead, out);
  else return LCQ_EDTYPE;
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

// A second stream per (device, caller's stream) for the deep trailing updates of long chains, with the two events that
// order it against the caller's stream.  Created on first use, kept until the process ends.
struct SideLane { int dev; hipStream_t caller; hipStream_t side; hipEvent_t fork, join; };
static SideLane g_lanes[16];
static int g_nlanes = 0;
static std::mutex g_lane_mu;
static std::atomic<int> g_lookahead{1};
static SideLane* side_lane(hipStream_t st) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lock(g_lane_mu);
  for (int i = 0; i < g_nlanes; ++i)
    if (g_lanes[i].dev == dev && g_lanes[i].caller == st) return &g_lanes[i];
  if (g_nlanes == 16) return nullptr;
  SideLane l{dev, st, nullptr, nullptr, nullptr};
  if (hipStreamCreateWithFlags(&l.side, hipStreamNonBlocking) != hipSuccess) return nullptr;       // default priority
  if (hipEventCreateWithFlags(&l.fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&l.join, hipEventDisableTiming) != hipSuccess) return nullptr;
  g_lanes[g_nlanes] = l;
  return &g_lanes[g_nlanes++];
}

// The chain behind lcq_chol_inv_upper (blocks_only = false) and lcq_chol_block_factor (true).
static int chol_chain(float* H, int64_t K64, const int64_t* perm, float percdamp, float* W, int64_t R, float* U,
                      void* workspace, int64_t workspace_bytes, int* status, void* stream, bool blocks_only) {
  if (!H || !U || !workspace || K64 <= 0 || K64 > 65536 || R < 0) return LCQ_EINVAL;
  if (blocks_only && K64 % NB != 0) return LCQ_EINVAL;     // the blocks of the reversed matrix must be the loop's blocks
  if (workspace_bytes < lcq_chol_inv_upper_workspace_bytes(K64)) return LCQ_EWORKSPACE;
  if (((uintptr_t)workspace % 16) != 0) return LCQ_EALIGN;
  const int K = (int)K64;
  const int nblk = (K + NB - 1) / NB;
  hipStream_t st = (hipStream_t)stream;
  float* A = (float*)workspace;
  float* Dinv = A + (long long)K * K;
  uint8_t* dead = (uint8_t*)(Dinv + (long long)nblk * NB * NB);
  PrepScalars* sc = (PrepScalars*)(dead + ((K + 255) / 256) * 256);
  void* const panel_space = (char*)workspace + chol_base_bytes(K, nblk);     // the current super-panel for the deep updates

  diag_prep_kernel<<<dim3(1), dim3(1024), 0, st>>>(H, K, percdamp, dead, sc);
  if (W && R > 0) {
    long long g = ((long long)R * K + 255) / 256;
    if (g > 65536) g = 65536;
    apply_dead_kernel<<<dim3((unsigned)g), dim3(256), 0, st>>>(W, R, K, dead);
  }
  if (perm && K <= 16384) {
    if (lcq_symmetrize(H, K, stream) != LCQ_OK) return LCQ_ELAUNCH;
    launch_build_gather(H, K, (const long long*)perm, sc, A, st);
  } else {
    build_kernel<<<dim3((unsigned)((K + 255) / 256), (unsigned)K), dim3(256), 0, st>>>(H, K, (const long long*)perm, sc, A);
  }

  // Blocked right-looking Cholesky with two block sizes: 128-column panels are factored one by
  // one, but their trailing update is applied only inside the current 512-column super-panel;
  // the rest of the matrix is updated once per super-panel with a 512-deep contraction, which
  // cuts the read-modify-write traffic on the trailing matrix fourfold.
  // The last 1024 columns are one super-panel: their rank-128 updates stay launches of about 5 us, while the 512-deep update that they
  // replace runs on 10 to 36 of 256 CUs (32 us).  K = 1024: 213 us with 512 columns, 189 so; 2048: 484 and 460; 4096: 1099 and 1074.
  // (1536 and 2048 columns: 2048 443 and 439, 4096 1057 and 1053; 14336 the same within 1 %.)
  constexpr int TAIL = 8 * NB;
  const auto super_end = [&](int o0) { return K - o0 <= TAIL ? K : o0 + NBO; };
  // Long chains: the deep update behind a super-panel is split into the columns of the NEXT super-panel (on the
  // caller's stream, the panels that follow need it) and everything behind those (on the side stream, beside those
  // panels: a few narrow launches that leave the chip to it).  The next deep update touches that region again and
  // waits for it.
  SideLane* lane = (g_lookahead.load() && K >= 8192) ? side_lane(st) : nullptr;
  // The update of rows and columns from `from` on by the super-panel [o0, o1).
  const auto deep_update = [&](int o0, int o1, int from, hipStream_t on) {
    const float* P = A + (long long)from * K + o0;
    float* C = A + (long long)from * K + from;
    const int rows = K - from, n = (rows + S3P_T - 1) / S3P_T;
    if (g_gemm_split.load() != 0 && o1 - o0 == NBO && s3p_pays(rows, rows, (int64_t)n * (n + 1) / 2) && s3p_operand(P, K, NBO)) {
      const S3POperand panel(panel_space, rows);    // (all deep updates of a chain are on one stream)
      s3p_pack<false>(P, K, rows, NBO, panel, on);
      s3p_multiply<true>(panel, panel, C, K, rows, rows, NBO, on);
    } else {
      launch_gemm<true>(GemmProblem{P, P, C, rows, rows, o1 - o0, K, K, K}, -1.0f, 1.0f, GEMM_LOWER_TILES, on);
    }
  };
  bool pending = false;
  for (int o0 = 0, o1; o0 < K; o0 = o1) {
    o1 = super_end(o0);
    for (int k0 = o0; k0 < o1; k0 += NB) {
      const int b = k0 / NB, nb = (K - k0 < NB) ? (K - k0) : NB;
      float* Akk = A + (long long)k0 * K + k0;
      float* Db = Dinv + (long long)b * NB * NB;
      potrf_diag_kernel<<<dim3(1), dim3(512), 0, st>>>(Akk, K, nb, Db, sc);
      const int k1 = k0 + nb, M = K - k1;
      if (M > 0) {
        float* A21 = A + (long long)k1 * K + k0;
        launch_gemm<true>(GemmProblem{A21, Db, A21, M, nb, nb, K, NB, K}, 1.0f, 0.0f, 0, st);       // A21 L11^-T
        if (o1 > k1)                                                                              // inside the super-panel
          launch_gemm<true>(GemmProblem{A21, A21, A + (long long)k1 * K + k1, M, o1 - k1, nb, K, K, K}, -1.0f, 1.0f,
                            GEMM_LOWER_TILES, st);
      }
    }
    if (o1 < K && lane) {
      const int o2 = super_end(o1);
      const float* P = A + (long long)o1 * K + o0;
      if (pending && hipStreamWaitEvent(st, lane->join, 0) != hipSuccess) return LCQ_ELAUNCH;
      pending = false;
      if (hipEventRecord(lane->fork, st) != hipSuccess) return LCQ_ELAUNCH;           // the panels of this super-panel
      launch_gemm<true>(GemmProblem{P, P, A + (long long)o1 * K + o1, K - o1, o2 - o1, o1 - o0, K, K, K}, -1.0f, 1.0f,
                        GEMM_LOWER_TILES, st);
      if (o2 < K) {
        if (hipStreamWaitEvent(lane->side, lane->fork, 0) != hipSuccess) return LCQ_ELAUNCH;
        deep_update(o0, o1, o2, lane->side);
        if (hipEventRecord(lane->join, lane->side) != hipSuccess) return LCQ_ELAUNCH;
        pending = true;
      }
    } else if (o1 < K) {                                                                          // everything behind it
      deep_update(o0, o1, o1, st);
    }
  }
  if (pending && hipStreamWaitEvent(st, lane->join, 0) != hipSuccess) return LCQ_ELAUNCH;

  if (blocks_only) {
    // No triangular inverse.  With M = J L J (H_d = M M^T, M upper triangular; J reverses the order) the inverse
    // factor is U = M^-1, and the column loop needs of it only (a) the diagonal blocks U_bb = (M_bb)^-1, which drive
    // the recurrence inside a block, and (b) something that carries a block's effect to the columns behind it.  From
    // E U = W - Q (E the loop's errors, Q the quantized weights, W the weights before the loop) follows
    //   W[:, b] as the loop finds it at block b  =  W0[:, b] + sum_{p<b} (W0 - Q)[:, p] M[p, b] U_bb,
    // so with P[p, b] = M[p, b] U_bb above the diagonal blocks and P[b, b] = U_bb the loop runs unchanged on P if a
    // block hands (Q - W0) instead of its errors to the deferred update.  In the reversed order that is every
    // sub-diagonal panel of L times the inverse of its diagonal block, which the factorization has already: one
    // batched product instead of the log2(K/128) merge levels of the inverse (K^3/3 flop).
    for (int b0 = 0; b0 + 1 < nblk; b0 += GEMM_MAX_BATCH) {
      const int np = (nblk - 1 - b0 < GEMM_MAX_BATCH) ? (nblk - 1 - b0) : GEMM_MAX_BATCH;
      GemmBatch bt;
      int maxM = 0;
      for (int q = 0; q < np; ++q) {
        const int b = b0 + q, k0 = b * NB, k1 = k0 + NB;
        bt.offA[q] = (long long)k1 * K + k0; bt.offB[q] = (long long)b * NB * NB; bt.offC[q] = bt.offA[q];
        bt.M[q] = K - k1; bt.N[q] = NB; bt.Kc[q] = NB;
        if (K - k1 > maxM) maxM = K - k1;
      }
      // Short tiles with all operands in flight while the launch leaves CUs idle, 128-row tiles when it fills the chip.
      // K = 1024: 9.3 us with 32 rows (23.5 with 128); 2176: 18.0 with 64 (25.0); 3072: 29.4 (32.0); 4096: 42.6 (41.4).
      const int tm = nblk <= 16 ? 32 : nblk <= 24 ? 64 : GT;
      const dim3 grid(1, (unsigned)((maxM + tm - 1) / tm), (unsigned)np);
      if (tm == 32) gemm_f32_batched_kernel<false, 32, true><<<grid, dim3(256), 0, st>>>(A, K, Dinv, NB, A, K, bt, 1.0f, 0.0f, 0);
      else if (tm == 64) gemm_f32_batched_kernel<false, 64, true><<<grid, dim3(256), 0, st>>>(A, K, Dinv, NB, A, K, bt, 1.0f, 0.0f, 0);
      else gemm_f32_batched_kernel<false><<<grid, dim3(256), 0, st>>>(A, K, Dinv, NB, A, K, bt, 1.0f, 0.0f, 0);
    }
    launch_scatter(A, K, Dinv, U, st);
    if (status)
      (void)hipMemcpyAsync(status, &sc->status, sizeof(int), hipMemcpyDeviceToDevice, st);
    LCQ_CHECK_LAUNCH();
    return LCQ_OK;
  }

  // triangular inverse: inverted diagonal blocks, then pairwise merges
  place_diag_kernel<<<dim3((unsigned)nblk, NB / 8), dim3(256), 0, st>>>(A, K, Dinv);
  int nseg = nblk;
  int seg_start[512], seg_size[512];
  if (nblk > 512) return LCQ_EINVAL;
  for (int b = 0; b < nblk; ++b) { seg_start[b] = b * NB; seg_size[b] = (K - b * NB < NB) ? (K - b * NB) : NB; }
  float* T = U;                                  // scratch until the final scatter
  while (nseg > 1) {
    const int npairs = nseg / 2;
    for (int p0 = 0; p0 < npairs; p0 += GEMM_MAX_BATCH) {
      const int np = (npairs - p0 < GEMM_MAX_BATCH) ? (npairs - p0) : GEMM_MAX_BATCH;
      GemmBatch b1, b2;
      int maxM = 0, maxN = 0;
      for (int q = 0; q < np; ++q) {
        const int sa = seg_start[2 * (p0 + q)], na = seg_size[2 * (p0 + q)];
        const int sc_ = seg_start[2 * (p0 + q) + 1], nc = seg_size[2 * (p0 + q) + 1];
        const long long offBlk = (long long)sc_ * K + sa;          // B block (rows of C-part, cols of A-part)
        // T1 = B * Ainv
        b1.offA[q] = offBlk; b1.offB[q] = (long long)sa * K + sa; b1.offC[q] = offBlk;
        b1.M[q] = nc; b1.N[q] = na; b1.Kc[q] = na;
        // X = -Cinv * T1
        b2.offA[q] = (long long)sc_ * K + sc_; b2.offB[q] = offBlk; b2.offC[q] = offBlk;
        b2.M[q] = nc; b2.N[q] = na; b2.Kc[q] = nc;
        if (nc > maxM) maxM = nc;
        if (na > maxN) maxN = na;
      }
      const dim3 grid((unsigned)((maxN + GT - 1) / GT), (unsigned)((maxM + GT - 1) / GT), (unsigned)np);
      if (g_gemm_split.load() && ((long long)grid.x * grid.y * grid.z > 256 || maxN >= 256)) {      // long contractions
        gemm_s3_batched_kernel<false><<<grid, dim3(256), 0, st>>>(A, K, A, K, T, K, b1, 1.0f, 0.0f, GEMM_K_FROM_N);
        gemm_s3_batched_kernel<false><<<grid, dim3(256), 0, st>>>(A, K, T, K, A, K, b2, -1.0f, 0.0f, GEMM_K_TO_M);
      } else {
        gemm_f32_batched_kernel<false><<<grid, dim3(256), 0, st>>>(A, K, A, K, T, K, b1, 1.0f, 0.0f, GEMM_K_FROM_N);
        gemm_f32_batched_kernel<false><<<grid, dim3(256), 0, st>>>(A, K, T, K, A, K, b2, -1.0f, 0.0f, GEMM_K_TO_M);
      }
    }
    int w = 0;
    for (int p = 0; p < npairs; ++p) {
      seg_start[w] = seg_start[2 * p];
      seg_size[w] = seg_size[2 * p] + seg_size[2 * p + 1];
      ++w;
    }
    if (nseg & 1) { seg_start[w] = seg_start[nseg - 1]; seg_size[w] = seg_size[nseg - 1]; ++w; }
    nseg = w;
  }

  launch_scatter(A, K, nullptr, U, st);
  if (status)
    (void)hipMemcpyAsync(status, &sc->status, sizeof(int), hipMemcpyDeviceToDevice, st);
  LCQ_CHECK_LAUNCH();
  return LCQ_OK;
}

int lcq_set_chain_lookahead(int on) {
  return g_lookahead.exchange(on ? 1 : 0);
}

int lcq_chol_inv_upper(float* H, int64_t K, const int64_t* perm, float percdamp, float* W, int64_t R, float* U,
                       void* workspace, int64_t workspace_bytes, int* status, void* stream) {
  return chol_chain(H, K, perm, percdamp, W, R, U, workspace, workspace_bytes, status, stream, false);
}

int lcq_chol_block_factor(float* H, int64_t K, const int64_t* perm, float percdamp, float* W, int64_t R, float* P,
                          void* workspace, int64_t workspace_bytes, int* status, void* stream) {
  return chol_chain(H, K, perm, percdamp, W, R, P, workspace, workspace_bytes, status, stream, true);
}

}  // extern "C"
