// How a LayerNorm row lies over lanes, and its arithmetic: shared by the stand-alone kernels (layernorm.hip)
// and by the single track's stage (single_stage.h), so that both give the same bits.
#pragma once
#include "common.h"

namespace ptx {

// A group of G lanes owns a row, each lane NCHUNK vectors: columns (c * G + lane) * VEC.  The first layout that
// holds a row's vectors is taken.
#define PTX_LN_LAYOUTS(X) \
  X(1, 1) X(2, 1) X(4, 1) X(8, 1) X(16, 1) X(32, 1) X(16, 2) X(16, 3) X(64, 1) X(64, 2) X(64, 4) X(64, 8)

struct LnLayout {
  int g, nc;
};
inline LnLayout ln_layout(int n_vectors) {
#define PTX_LN_PICK(G, NC) \
  if (n_vectors <= (G) * (NC)) return LnLayout{G, NC};
  PTX_LN_LAYOUTS(PTX_LN_PICK)
#undef PTX_LN_PICK
  return LnLayout{0, 0};
}
constexpr int kLnChunks = 3;   // most chunks ln_four_rows takes

// (one rounding for gamma and beta, whatever the surrounding code lets the compiler contract)
__device__ __forceinline__ float ln_affine(float x, float mean, float rstd, float gamma, float beta) {
  return __builtin_fmaf((x - mean) * rstd, gamma, beta);
}

// LayerNorm of rows row0 .. row0 + 3 of x [rows][cols], by one wave.  16-byte vectors; cols a multiple of them,
// layout.nc <= kLnChunks.
template <typename T>
__device__ __forceinline__ void ln_four_rows(const T* x, T* y, const T* gamma, const T* beta, int rows, int cols, int row0,
                                             float eps, LnLayout l, int lane) {
  constexpr int VEC = 16 / (int)sizeof(T);
  typedef __attribute__((ext_vector_type(VEC))) T V;
  const int sub = lane & (l.g - 1), grp = lane / l.g, at_once = kWave / l.g;
  const float inv_n = 1.0f / (float)cols;
  V raw[4][kLnChunks], gm[kLnChunks], bt[kLnChunks];
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int64_t row = min(row0 + min(it * at_once + grp, 3), rows - 1);
#pragma unroll
    for (int c = 0; c < kLnChunks; ++c) {
      const int col = (c * l.g + sub) * VEC;
      raw[it][c] = *reinterpret_cast<const V*>(x + row * cols + (col < cols ? col : 0));
    }
  }
#pragma unroll
  for (int c = 0; c < kLnChunks; ++c) {
    const int col = (c * l.g + sub) * VEC < cols ? (c * l.g + sub) * VEC : 0;
    if (gamma) gm[c] = *reinterpret_cast<const V*>(gamma + col);
    if (beta) bt[c] = *reinterpret_cast<const V*>(beta + col);
  }
  // (the four rows' exchanges side by side: each waits for the one before)
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f}, q[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int it = 0; it < 4; ++it)
#pragma unroll
    for (int c = 0; c < kLnChunks; ++c)
      if ((c * l.g + sub) * VEC < cols) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) s[it] += (float)raw[it][c][e];
      }
  for (int m = l.g >> 1; m >= 1; m >>= 1)
#pragma unroll
    for (int it = 0; it < 4; ++it) s[it] += __shfl_xor(s[it], m, 64);
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    s[it] *= inv_n;
#pragma unroll
    for (int c = 0; c < kLnChunks; ++c)
      if ((c * l.g + sub) * VEC < cols) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const float d = (float)raw[it][c][e] - s[it];
          q[it] = __builtin_fmaf(d, d, q[it]);
        }
      }
  }
  for (int m = l.g >> 1; m >= 1; m >>= 1)
#pragma unroll
    for (int it = 0; it < 4; ++it) q[it] += __shfl_xor(q[it], m, 64);
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const float rstd = rsqrtf(fmaxf(q[it] * inv_n, 0.0f) + eps);
    const int r = it * at_once + grp;
    if (r >= 4 || row0 + r >= rows) continue;
#pragma unroll
    for (int c = 0; c < kLnChunks; ++c) {
      const int col = (c * l.g + sub) * VEC;
      if (col < cols) {
        V o;
#pragma unroll
        for (int e = 0; e < VEC; ++e)
          o[e] = (T)ln_affine((float)raw[it][c][e], s[it], rstd, gamma ? (float)gm[c][e] : 1.0f, beta ? (float)bt[c][e] : 0.0f);
        *reinterpret_cast<V*>(y + (int64_t)(row0 + r) * cols + col) = o;
      }
    }
  }
}

}  // namespace ptx
