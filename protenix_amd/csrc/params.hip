// Parameters on their way into the kernels: any number of vectors and matrices converted (fp32 <-> bf16) and
// gathered, or laid out as a linear stage's fragments (single_stage.h), in one launch.  What a plan needs before
// its first call: one conversion per parameter was some thirty launches a block, 0.4 ms of host time on new weights.
// Bound by launches at every size met (a block's parameters are 2 - 12 MB, 3 - 15 us).
#include "common.h"
#include "kernels.h"

namespace ptx {

namespace {
constexpr int kParamsPerLaunch = 56;   // (kernel arguments: 4 KB at most)
constexpr int kParamWork = 2048;       // elements per workgroup
struct ParamList {
  Param p[kParamsPerLaunch];
  int first[kParamsPerLaunch + 1];     // first workgroup of each
  int count;
};
static_assert(sizeof(ParamList) <= 3584, "kernel arguments");
}  // namespace

__global__ __launch_bounds__(256) void param_pack_kernel(ParamList l) {
  int i = 0;
  while (i + 1 < l.count && (int)blockIdx.x >= l.first[i + 1]) ++i;
  const Param p = l.p[i];
  const int64_t n = p.rows * p.cols, base = (int64_t)(blockIdx.x - l.first[i]) * kParamWork;
  const int steps = p.cols >> 5, ve = p.dst_bits16 ? 8 : 4;
#pragma unroll
  for (int j = 0; j < kParamWork / 256; ++j) {
    const int64_t e = base + j * 256 + threadIdx.x;
    if (e >= n) return;
    int64_t s = e;
    if (p.fragments) {   // [16 rows][32 columns][piece][lane][ve]: lane % 16 <-> row, ve * (lane / 16) + 4 * ve * piece <-> column
      const int v = (int)(e % ve), lane = (int)(e / ve) & 63;
      const int64_t q = e / (64 * ve);
      const int pieces = 8 / ve, piece = (int)(q % pieces);
      const int64_t step = q / pieces % steps, cb = q / pieces / steps;
      s = (cb * 16 + (lane & 15)) * p.cols + step * 32 + 4 * ve * piece + ve * (lane >> 4) + v;
    }
    const float x = p.src_bits16 ? to_f32(((const bf16_t*)p.src)[s]) : ((const float*)p.src)[s];
    if (p.dst_bits16) ((bf16_t*)p.dst)[e] = from_f32<bf16_t>(x);
    else ((float*)p.dst)[e] = x;
  }
}

int param_pack(const Param* p, int count, hipStream_t stream) {
  for (int i = 0; i < count;) {
    ParamList l;
    l.count = 0;
    int wgs = 0;
    for (; i < count && l.count < kParamsPerLaunch; ++i) {
      const int w = (int)((p[i].rows * p[i].cols + kParamWork - 1) / kParamWork);
      if (w == 0) continue;
      l.p[l.count] = p[i];
      l.first[l.count++] = wgs;
      wgs += w;
    }
    if (wgs) param_pack_kernel<<<dim3((unsigned)wgs), dim3(256), 0, stream>>>(l);
  }
  return 0;
}

}  // namespace ptx
