// Launches of the single-representation track's stages (single_stage.h) on their own: for callers of one
// layer at a time, and for the last block of a stack, which has no pair kernels left to ride on.
#include "single_stage.h"

namespace ptx {

template <typename T>
__global__ __launch_bounds__(kStageWaves * 64, 3) void single_stage_kernel(SingleStage p) {
  __shared__ __attribute__((aligned(16))) char smem[kStageLds];
  single_stage<T>(p, blockIdx.x, smem);
}

// A linear stage takes the smallest tile (16 x 16, 16 x 32, 32 x 32) that makes at most this many workgroups, counted
// in whole sets of eight column tiles: they then fit beside a small pair kernel's own (three workgroups per
// compute unit).  (Launched are the tiles there are: 147456 rows, 128 -> 16 in fp32 231 us with empty workgroups up
// to whole sets, 33 without.)
constexpr int kStageTiles = 320;

int single_stage_layernorm(SingleStage* s, const void* x, const void* gamma, const void* beta, void* y, int rows, int cols,
                           float eps, bool bits16) {
  *s = SingleStage{};
  const int vec = bits16 ? 8 : 4;
  const LnLayout l = ln_layout(cols / vec);
  if (cols % vec || l.nc < 1 || l.nc > kLnChunks) return -1;
  s->kind = rows > 0 ? kStageLayerNorm : kStageNone;
  s->n_work = (rows + 15) / 16;
  s->bits16 = bits16;
  s->rows = rows;
  s->x = x;
  s->w = gamma;
  s->w2 = beta;
  s->out = y;
  s->k = cols;
  s->ln_g = l.g;
  s->ln_nc = l.nc;
  s->eps = eps;
  return 0;
}

void single_stage_linear(SingleStage* s, const void* x, const void* w, const void* w2, const void* bias, int bias_cols,
                         const void* res, void* out, void* out_t, int split_col, int64_t ldt, int rows, int k, int n_out,
                         bool bits16, int packed) {
  *s = SingleStage{};
  s->bits16 = bits16;
  s->packed = packed;
  s->x = x;
  s->w = w;
  s->w2 = w2;
  s->bias = bias;
  s->bias_cols = bias_cols;
  s->res = res;
  s->out = out;
  s->out_t = out_t;
  s->split_col = split_col < n_out ? split_col : n_out;
  s->ldo = s->split_col;
  s->ldt = ldt;
  s->rows = rows;
  s->k = k;
  s->n_out = n_out;
  const int64_t span = s->split_col < n_out && ldt > rows ? ldt : rows;
  for (s->tile = 1;; ++s->tile) {
    const int rm = s->tile == 3 ? 32 : 16, cn = s->tile == 1 ? 16 : 32;
    s->row_blocks = (int)((span + rm - 1) / rm);
    const int cols = (n_out + cn - 1) / cn;
    s->n_work = cols * s->row_blocks;
    for (s->set_shift = 3; s->set_shift > 0 && cols % (1 << s->set_shift); --s->set_shift) {}
    if (s->tile == 3 || (cols + 7) / 8 * 8 * s->row_blocks <= kStageTiles) break;
  }
  s->kind = s->n_work == 0 || rows == 0 ? kStageNone : w2 ? kStageSwiGLU : kStageLinear;
}

void single_stage_attention(SingleStage* s, const void* q, const void* k, const void* vt, const void* gate, const void* bias,
                            int bias_f32, void* out, int n, int heads, int d, int64_t ld, int64_t ldt, int64_t ldo,
                            float scale, bool bits16) {
  *s = SingleStage{};
  s->kind = n == 0 || heads == 0 ? kStageNone : kStageAttention;
  s->n_work = (n + 31) / 32 * heads;
  s->bits16 = bits16;
  s->rows = n;
  s->x = q;
  s->w = k;
  s->w2 = vt;
  s->gate = gate;
  s->bias = bias;
  s->bias_f32 = bias_f32;
  s->bias_vec = (n % 8 == 0) && (((uintptr_t)bias & 15) == 0);
  s->out = out;
  s->ld = ld;
  s->ldt = ldt;
  s->ldo = ldo;
  s->heads = heads;
  s->d = d;
  s->scale = scale;
}

int single_stage_run(const SingleStage* s, hipStream_t stream) {
  if (s->kind == kStageNone) return 0;
  const dim3 grid((unsigned)s->n_work), block(kStageWaves * 64);
  if (s->bits16) single_stage_kernel<bf16_t><<<grid, block, 0, stream>>>(*s);
  else single_stage_kernel<float><<<grid, block, 0, stream>>>(*s);
  return 0;
}

}  // namespace ptx
