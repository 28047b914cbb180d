// Rules by which an entry point takes one of several kernels, as functions of sizes, types and alignment alone.  Plain C++: they can
// be checked without a GPU and without a HIP compiler.
#pragma once

namespace lcq {

// Products with a contraction of exactly 128 (gemm_f32.h): C = alpha A op(B) + beta C.
//   solve   C = A B^T of 128 columns (C may be A)
//   waves   C -= A op(B), one wave per 16 x 32 of C; leaves out the tiles above the diagonal where `lower` asks for it
//   stream  C -= A B, a wave per 64 columns streams rows; every tile
//   none    the general kernels, which leave them out too
// The line between waves and stream is 1024 tiles of 16 x 64, a stream's one tile per wave (measured beside the launches).
enum class Rank128 { none, solve, waves, stream };
inline Rank128 rank128_form(bool b_t, long long M, long long N, float alpha, float beta, bool in_place, bool lower) {
  if (b_t && alpha == 1.0f && beta == 0.0f && N == 128) return Rank128::solve;
  if (alpha != -1.0f || beta != 1.0f || in_place) return Rank128::none;
  if (b_t || ((M + 15) / 16) * ((N + 63) / 64) <= 1024) return Rank128::waves;
  return lower ? Rank128::none : Rank128::stream;
}

// Column loop (gptq_loop.hip): does a block run by panels of 64 rows?  Whole blocks of 128 columns on 16 bytes (`on16`: all pointers),
// rounded zero points, and parameters that change at the starts of 16-column panels only: searched for groups that open inside the
// block, or given for groups of whole panels or for rows.
// Codes of 9 and 10 bits (all of them within +-512, beyond that both kernels divide everywhere) stay with sixteen lanes per row where the
// panels that run again with divisions cost more than a wave of 64 rows gains.  How many do grows with the code range and with the rows
// of a wave; the gain is smaller for long groups, and sixteen lanes lose beyond one workgroup per CU (4096 rows).  us per block by panels
// / by sixteen lanes, 9 | 10 bits, symmetric:
//   rows          64                      256                     1000                    4096                    5120
//   g = 32    13.7 / 15.3 | 14.6 / 15.4   14.7 / 15.8 | 15.8 / 15.8   15.8 / 16.5 | 16.7 / 16.5   17.1 / 17.9 | 17.9 / 17.9   17.5 / 21.4 | 18.3 / 21.4
//   g = 64    13.8 / 14.8 | 14.5 / 14.8   14.7 / 15.3 | 15.9 / 15.3   15.6 / 16.1 | 16.6 / 16.0   17.0 / 17.3 | 18.0 / 17.4   17.5 / 20.5 | 18.4 / 20.5
//   g = 128   13.3 / 14.0 | 14.6 / 14.2   14.8 / 14.4 | 15.9 / 14.6   15.7 / 15.3 | 16.7 / 15.3   17.0 / 16.5 | 18.0 / 16.6   17.5 / 19.9 | 18.3 / 19.9
// (8 bits, g = 128: 13.3 / 14.1, 14.1 / 14.5, 14.9 / 15.3, 16.2 / 16.5, 16.8 / 19.8; given parameters, 10 bits, 4096 rows: 18.0 / 20.8.)
inline bool gptq_by_panels(bool is_static, bool has_gidx, bool rounded, int group, long long R, long long K, long long i1, int count, long long ldErr,
                           bool on16, float qmin, float qmax) {
  const bool whole = is_static ? !has_gidx && (group <= 0 || group % 16 == 0) : group == 16 || group == 32 || group == 64 || group == 128;
  if (!whole || !rounded || count != 128 || i1 % 128 != 0 || K % 4 != 0 || ldErr % 4 != 0 || !on16) return false;
  const float codes = qmax - qmin + 1.0f;
  const bool divides = qmin < -512.0f || qmin > 512.0f || qmax < -512.0f || qmax > 512.0f;
  return is_static || divides || codes * group < 65536.0f || codes * R <= 32768.0f || R > 4096;
}

}  // namespace lcq
