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

}  // namespace lcq
