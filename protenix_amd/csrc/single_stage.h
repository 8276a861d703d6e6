// The stages of the single-representation track, as device code that runs in a launch of its own
// (single.hip) or on extra workgroups of a pair-tensor kernel (pairproj.hip: "carried").  The track is
// a thousandth of a block's work in seven dependent stages; as launches on a second stream they cost
// the block 25 to 65 us (93 to 512 tokens: the caches' write-backs and invalidations at every kernel's
// ends, and the waits between the streams), carried they need no launch and no wait, because the pair
// kernels they ride on are already in order.
//
//   layernorm   out = LayerNorm(x)
//   linear      out = [res +] x W^T [+ bias], optionally with a tail of the output columns stored
//               transposed (the attention's V^T); or, SwiGLU, out = silu(x W_a^T) * (x W_b^T)
//   attention   flash-style softmax(q k^T * scale + bias) v per head, gated by sigmoid(g), logits
//               never materialised
//
// A stage is a set of independent workgroups of four waves; operands go from global memory (L2-resident
// at these sizes) straight into MFMA fragments.
#pragma once
#include "common.h"
#include "kernels.h"
#include "lnrow.h"

namespace ptx {

constexpr int kStageWaves = 4;
// LDS of a stage: the waves' partial results, up to 32 registers per lane (SwiGLU in tiles of 32 x 32)
constexpr int kStageLds = kStageWaves * 32 * kWave * 4;

// acc[16 x 16] += A[16 x 32] B[32 x 16]: lane l supplies row (column) l % 16, K-slots 8 * (l / 16) .. + 7, and receives
// column l % 16, rows 4 * (l / 16) + register.
__device__ __forceinline__ void mma16(f32x4& acc, bf16x8 a, bf16x8 b) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ void mma16(f32x4& acc, f32x8 a, f32x8 b) {
#pragma unroll
  for (int t = 0; t < 8; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], acc, 0, 0, 0);
}

// One workgroup per tile of 16 RM rows x 16 CN columns; its four waves each take a quarter of K and the partial
// tiles are summed through LDS in wave order.  Few rows take the smallest tiles: the fp32 matrix pipes of 36
// compute units would be busy for 5 us with 93 x 384 outputs in tiles of 32 x 32 at K = 1536, and a wave's share of
// the weights (which come from memory: a block's 12 MB pass through once per block) can be requested
// as a whole before anything else is waited for.
template <typename T, bool SWIGLU, int RM, int CN>
__device__ __forceinline__ void linear_stage(const SingleStage& p, int wg, char* smem) {
  typedef typename Vec8<T>::type V8;
  typedef typename Vec4<T>::type V4;
  constexpr int NM = SWIGLU ? 2 : 1, NB = RM * CN;   // matrices; 16 x 16 blocks of the tile
  static_assert(NM * NB <= 8, "LDS of the partial sums");
  constexpr int KC = NB == 1 ? (SWIGLU ? 3 : 4) : 2;   // K steps requested together
  float (*part)[4 * NM * NB][kWave] = reinterpret_cast<float (*)[4 * NM * NB][kWave]>(smem);       // [wave][register][lane]
  const int lane = threadIdx.x & 63, ln = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Sets of eight column blocks (or fewer, see single_stage_linear): all row blocks of a column block on one XCD, whose L2 then
  // fetches those weights once.
  const int per_set = p.row_blocks << p.set_shift;
  const int set = wg / per_set, in_set = wg - set * per_set;
  const int rb = in_set >> p.set_shift, cb = (set << p.set_shift) + in_set - (rb << p.set_shift);
  const int row0 = rb * 16 * RM, col0 = cb * 16 * CN;
  const bool transposed = !SWIGLU && col0 >= p.split_col;   // the same for the whole workgroup
  // K steps of 32 (k is a multiple of 16), an equal share per wave.  A lane's 8 elements of a step are 16-byte pieces
  // VE * g of every 4 * VE elements, so that a load instruction covers 64 contiguous bytes of each of its 16 rows.
  constexpr int VE = 16 / (int)sizeof(T), PIECES = 8 / VE;
  const int steps = (p.k + 31) >> 5;
  const T* xp[RM];
  const T* wp[NM][CN];
#pragma unroll
  for (int a = 0; a < RM; ++a) xp[a] = (const T*)p.x + (int64_t)min(row0 + 16 * a + ln, p.rows - 1) * p.k;
  // weights: rows like x's, or packed [column block][step][piece][lane][VE]
#pragma unroll
  for (int b = 0; b < CN; ++b) {
    const int64_t wr = p.packed ? (int64_t)min(col0 + 16 * b, p.n_out - 16) * p.k + lane * VE : (int64_t)min(col0 + 16 * b + ln, p.n_out - 1) * p.k;
    wp[0][b] = (const T*)p.w + wr;
    if (SWIGLU) wp[NM - 1][b] = (const T*)p.w2 + wr;
  }
  auto k_of = [&](int s, int pc) { return min(32 * min(s, steps - 1) + 4 * VE * pc + VE * g, p.k - VE); };   // (clamped: beyond the slice, a valid one)
  auto load_row = [&](const T* row, int s) {
    V8 v;
    u32x4_t* d = reinterpret_cast<u32x4_t*>(&v);
#pragma unroll
    for (int pc = 0; pc < PIECES; ++pc) d[pc] = *reinterpret_cast<const u32x4_t*>(row + k_of(s, pc));
    return v;
  };
  auto load_packed = [&](const T* base, int s) {
    V8 v;
    u32x4_t* d = reinterpret_cast<u32x4_t*>(&v);
#pragma unroll
    for (int pc = 0; pc < PIECES; ++pc) d[pc] = *reinterpret_cast<const u32x4_t*>(base + min(s, steps - 1) * 512 + pc * 256);
    return v;
  };
  const int per_wave = (steps + kStageWaves - 1) / kStageWaves;
  const int s_begin = wave * per_wave, s_end = min(steps, s_begin + per_wave);
  V8 xa[KC][RM], wa[KC][NM][CN];
  auto load_w = [&](int s0) {
#pragma unroll
    for (int s = 0; s < KC; ++s)
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int b = 0; b < CN; ++b) wa[s][m][b] = p.packed ? load_packed(wp[m][b], s0 + s) : load_row(wp[m][b], s0 + s);
  };
  auto load_x = [&](int s0) {
#pragma unroll
    for (int s = 0; s < KC; ++s)
#pragma unroll
      for (int a = 0; a < RM; ++a) xa[s][a] = load_row(xp[a], s0 + s);
  };
  load_w(s_begin);
  load_x(s_begin);

  f32x4 acc[NM][RM][CN];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int a = 0; a < RM; ++a)
#pragma unroll
      for (int b = 0; b < CN; ++b) acc[m][a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = s_begin; s0 < s_end;) {
#pragma unroll
    for (int s = 0; s < KC; ++s) {
      if (s0 + s >= s_end) break;
      if (32 * (s0 + s) + 32 > p.k) {   // a last step of 16
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          if (32 * (s0 + s) + 4 * VE * (t / VE) + VE * g < p.k) continue;
#pragma unroll
          for (int a = 0; a < RM; ++a) xa[s][a][t] = (T)0.0f;
#pragma unroll
          for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int b = 0; b < CN; ++b) wa[s][m][b][t] = (T)0.0f;
        }
      }
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int a = 0; a < RM; ++a)
#pragma unroll
          for (int b = 0; b < CN; ++b) {
            if (!SWIGLU && transposed) mma16(acc[m][a][b], xa[s][a], wa[s][m][b]);   // lane <-> column, register <-> row
            else mma16(acc[m][a][b], wa[s][m][b], xa[s][a]);                          // lane <-> row, register <-> column
          }
    }
    s0 += KC;
    if (s0 < s_end) {
      load_w(s0);
      load_x(s0);
    }
  }
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int a = 0; a < RM; ++a)
#pragma unroll
      for (int b = 0; b < CN; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[wave][4 * (NB * m + CN * a + b) + e][lane] = acc[m][a][b][e];
  __syncthreads();

  // wave w finishes block w
  if (wave >= NB) return;
  const int ba = wave / CN, bb = wave - ba * CN;
  f32x4 y[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    y[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < kStageWaves; ++w)
#pragma unroll
      for (int e = 0; e < 4; ++e) y[m][e] += part[w][4 * (NB * m + wave) + e][lane];
  }
  if (!transposed) {
    const int row = row0 + 16 * ba + ln, col = col0 + 16 * bb + 4 * g;
    if (row < p.rows && col < p.n_out) {   // (n_out is a multiple of 4)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (SWIGLU) {
          // a and b rounded to T first, as the two linear layers of the reference do
          const float av = to_f32(from_f32<T>(y[0][e])), bv = to_f32(from_f32<T>(y[NM - 1][e]));
          y[0][e] = to_f32(from_f32<T>(av * sigmoidf_fast(av))) * bv;
        } else if (p.bias && col + e < p.bias_cols) {
          y[0][e] += to_f32(((const T*)p.bias)[col + e]);
        }
      }
      if (p.res) {
        const f32x4 rv = to_f32(*reinterpret_cast<const V4*>((const T*)p.res + (int64_t)row * p.n_out + col));
#pragma unroll
        for (int e = 0; e < 4; ++e) y[0][e] = to_f32(from_f32<T>(y[0][e])) + rv[e];
      }
      *reinterpret_cast<V4*>((T*)p.out + (int64_t)row * p.ldo + col) = from_f32<T>(y[0]);
    }
  } else {
    const int col = col0 + 16 * bb + ln, row = row0 + 16 * ba + 4 * g;
    if (col < p.n_out && row < p.ldt) {   // (ldt is a multiple of 4)
#pragma unroll
      for (int e = 0; e < 4; ++e) y[0][e] = row + e < p.rows ? y[0][e] : 0.0f;
      *reinterpret_cast<V4*>((T*)p.out_t + (int64_t)(col - p.split_col) * p.ldt + row) = from_f32<T>(y[0]);
    }
  }
}

template <typename T> __device__ __forceinline__ typename Vec8<T>::type zero8() {
  typename Vec8<T>::type z;
#pragma unroll
  for (int t = 0; t < 8; ++t) z[t] = (T)0.0f;
  return z;
}

// MFMA row m of a 32-key block stands for key 16*(m>>4) + 8*((m>>2)&1) + 4*((m>>3)&1) + (m&3), which makes
// accumulator registers 8*ks .. 8*ks+7 of half-wave g hold keys 16*ks + 8*g .. +7: the probabilities feed
// P.V as its B operand without a shuffle, and bias and V^T loads are runs of 8 consecutive keys.
__device__ __forceinline__ int key_of_mfma_row(int m) {
  return 16 * (m >> 4) + 8 * ((m >> 2) & 1) + 4 * ((m >> 3) & 1) + (m & 3);
}

// One workgroup per (32 queries, head); its kStageWaves waves take every kStageWaves-th block of
// 32 keys each and merge their partial results through LDS in a fixed order: the chain of
// dependent loads a wave walks through is a quarter as long.
template <typename T>
__device__ __forceinline__ void attention_stage(const SingleStage& p, int wg, char* smem) {
  typedef typename Vec8<T>::type V8;
  typedef typename Vec4<T>::type V4;
  constexpr float kL2e = 1.4426950408889634f;
  float (*part_o)[16][kWave] = reinterpret_cast<float (*)[16][kWave]>(smem);
  float (*part_ml)[2][kWave] = reinterpret_cast<float (*)[2][kWave]>(smem + kStageWaves * 16 * kWave * 4);
  const int lane = threadIdx.x & 63, ln = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = p.rows, d = p.d;
  const int q_blocks = (n + 31) >> 5;
  const int h = wg / q_blocks, q0 = (wg - h * q_blocks) * 32;
  const int qi = min(q0 + ln, n - 1);
  const T* qp = (const T*)p.x + (int64_t)qi * p.ld + h * d;
  // q fragments (B operand: lane <-> query, slots <-> channels 16*kk + 8*g .. +7), in log2 units
  V8 qf[2];
  const float qs = p.scale * kL2e;
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    qf[kk] = zero8<T>();
    if (16 * kk + 8 * g < d) {
      f32x8 v = to_f32(load8<T>(qp + 16 * kk + 8 * g));
#pragma unroll
      for (int t = 0; t < 8; ++t) v[t] *= qs;
      qf[kk] = from_f32<T>(v);
    }
  }
  const int krow = key_of_mfma_row(ln);
  const T* kbase = (const T*)p.w + h * d;
  const T* vrow = (const T*)p.w2 + (int64_t)(h * d + min(ln, d - 1)) * p.ldt;
  const float* bf = (const float*)p.bias + ((int64_t)h * n + qi) * n;
  const T* bt = (const T*)p.bias + ((int64_t)h * n + qi) * n;

  f32x16 acc_o;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc_o[r] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;

  for (int key0 = 32 * wave; key0 < n; key0 += 32 * kStageWaves) {
    const bool tail = key0 + 32 > n;   // the same for the whole wave
    // K fragments (A operand: lane <-> key, slots <-> channels)
    const T* kp = kbase + (int64_t)min(key0 + krow, n - 1) * p.ld;
    V8 kf[2], vf[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      kf[kk] = zero8<T>();
      if (16 * kk + 8 * g < d) kf[kk] = load8<T>(kp + 16 * kk + 8 * g);
    }
    // V^T fragments (A operand: lane <-> channel, slots <-> keys key0 + 16*ks + 8*g .. +7)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      vf[ks] = zero8<T>();
      if (ln < d) vf[ks] = load8<T>(vrow + key0 + 16 * ks + 8 * g);
    }
    // logits start from the bias: registers 8*ks + t <-> keys key0 + 16*ks + 8*g + t
    f32x16 s;
    if (p.bias && !tail && p.bias_vec) {
      // (n is a multiple of 8: the 8-key runs are 16-byte aligned vectors)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int key = key0 + 16 * ks + 8 * g;
        f32x8 b;
        if (p.bias_f32) {
          const f32x4 b0 = *reinterpret_cast<const f32x4*>(bf + key);
          const f32x4 b1 = *reinterpret_cast<const f32x4*>(bf + key + 4);
          b = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
        } else {
          b = to_f32(load8<T>(bt + key));
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) s[8 * ks + t] = b[t] * kL2e;
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const int key = key0 + 16 * ks + 8 * g + t;
          float b = 0.0f;
          if (p.bias) {
            const int kc = min(key, n - 1);
            b = p.bias_f32 ? bf[kc] : to_f32(bt[kc]);
          }
          s[8 * ks + t] = b * kL2e;
        }
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) mma32(s, kf[kk], qf[kk]);
    if (tail) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int t = 0; t < 8; ++t)
          if (key0 + 16 * ks + 8 * g + t >= n) s[8 * ks + t] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, swap32(mx));
    const float m_new = fmaxf(m_run, mx);     // finite: every block holds at least one key
    const float alpha = fast_exp2(m_run - m_new);
    m_run = m_new;
    float psum = 0.0f;
    V8 pf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      f32x8 p8;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        p8[t] = fast_exp2(s[8 * ks + t] - m_new);
        psum += p8[t];
      }
      pf[ks] = from_f32<T>(p8);
    }
    l_run = l_run * alpha + psum;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc_o[r] *= alpha;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) mma32(acc_o, vf[ks], pf[ks]);   // lane <-> query, register <-> channel
  }

  // merge the waves' partial results (a wave without key blocks contributes m = -inf, l = 0)
  l_run += swap32(l_run);
#pragma unroll
  for (int r = 0; r < 16; ++r) part_o[wave][r][lane] = acc_o[r];
  part_ml[wave][0][lane] = m_run;
  part_ml[wave][1][lane] = l_run;
  __syncthreads();
  if (wave != 0) return;
  float m_all = part_ml[0][0][lane];
#pragma unroll
  for (int w = 1; w < kStageWaves; ++w) m_all = fmaxf(m_all, part_ml[w][0][lane]);
  l_run = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc_o[r] = 0.0f;
#pragma unroll
  for (int w = 0; w < kStageWaves; ++w) {
    const float f = fast_exp2(part_ml[w][0][lane] - m_all);   // wave 0 always has a block: m_all is finite
    l_run += part_ml[w][1][lane] * f;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc_o[r] += part_o[w][r][lane] * f;
  }
  const float inv = fast_rcp(l_run);
  if (q0 + ln < n) {
    const T* gp = p.gate ? (const T*)p.gate + (int64_t)qi * p.ld + h * d : nullptr;
    T* op = (T*)p.out + (int64_t)qi * p.ldo + h * d;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const int c0 = 8 * a + 4 * g;
      if (c0 < d) {   // (d is a multiple of 4)
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = to_f32(from_f32<T>(acc_o[4 * a + e] * inv));
        if (gp) {
          const f32x4 gv = to_f32(*reinterpret_cast<const V4*>(gp + c0));
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] *= to_f32(from_f32<T>(sigmoidf_fast(gv[e])));
        }
        *reinterpret_cast<V4*>(op + c0) = from_f32<T>(v);
      }
    }
  }
}

// 16 rows per workgroup, four per wave.  (Taken into the linear stages that follow - statistics per tile, rows
// normalised on their way into the fragments - it made each of them 3.5 us longer and saved no launch.)
template <typename T>
__device__ __forceinline__ void layernorm_stage(const SingleStage& p, int wg) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  ln_four_rows<T>((const T*)p.x, (T*)p.out, (const T*)p.w, (const T*)p.w2, p.rows, p.k, wg * 16 + wave * 4, p.eps,
                  LnLayout{p.ln_g, p.ln_nc}, threadIdx.x & 63);
}

template <typename T>
__device__ __forceinline__ void single_stage(const SingleStage& p, int wg, char* smem) {
  if (wg >= p.n_work) return;   // (the count is rounded up, see SingleStage)
  if (p.kind == kStageAttention) {
    attention_stage<T>(p, wg, smem);
  } else if (p.kind == kStageLayerNorm) {
    layernorm_stage<T>(p, wg);
  } else if (p.kind == kStageSwiGLU) {
    if (p.tile == 1) linear_stage<T, true, 1, 1>(p, wg, smem);
    else if (p.tile == 2) linear_stage<T, true, 1, 2>(p, wg, smem);
    else linear_stage<T, true, 2, 2>(p, wg, smem);
  } else {
    if (p.tile == 1) linear_stage<T, false, 1, 1>(p, wg, smem);
    else if (p.tile == 2) linear_stage<T, false, 1, 2>(p, wg, smem);
    else linear_stage<T, false, 2, 2>(p, wg, smem);
  }
}

}  // namespace ptx
