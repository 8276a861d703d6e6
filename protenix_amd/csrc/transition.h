// What the two transition kernels (transition.hip, transition_small.hip) share.
#pragma once
#include "common.h"
#include "kernels.h"

namespace ptx {

struct PairBiasArgs {
  const void *gamma, *beta, *w;   // LayerNorm of the bias (either may be null), W [heads][c]
  void* out;                      // [heads][n_rows], fp32 or T
  int heads, out_f32;
  float eps;
};

struct AttnOutArgs {
  const void* o;             // attention output, head-major [4][n_rows][32], T, rows in the attention's order
  const void *gamma, *beta;  // the attention's LayerNorm (either may be null)
  RowMap omap;               // row of x -> element offset of its 32 channels inside a head's plane of o
  float eps;
};
constexpr int kAoChunks = 3;   // chunks of 24 fragments that hold the 64 fragments of W_g and W_o

// The transition on few rows (transition_small.hip); arguments as the fused kernel's.  Returns
// false where the fused kernel is to be launched instead.  carry (PB and AO): a stage of the single track on operands of type
// TZ, run by the launch's first workgroups.
template <typename T, int KS, typename TZ, bool PB, bool AO>
bool transition_small(const TZ* x, const T* gamma, const T* beta, const T* packed, TZ* out, int64_t n_rows, int n_chunks,
                      int add_residual, float eps, const PairBiasArgs& pb, const AttnOutArgs& ao, hipStream_t stream,
                      const SingleStage* carry = nullptr);

}  // namespace ptx
