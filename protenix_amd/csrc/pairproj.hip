// The row-local stages of the triangle updates on packed weights: LayerNorm + projections
// (trimul_in, triattn_in), and the output stages (trimul_out, triattn_out).
//
// A workgroup of four waves takes a tile of 32 * RBW pair-tensor rows.  Its rows are read once, in
// whole cache lines (8 lanes per row), normalised in fp32 and parked in LDS as MFMA operand
// fragments; after one barrier every wave multiplies them by its own share of the output columns.
// The weights were packed into fragment order beforehand (pair_pack), so a fragment is one
// contiguous 1 KB load from the L2 into registers, used for all of the tile's row blocks: no LDS
// traffic for them, and no barrier in the loop.  (The L2s deliver a buffer that all compute units
// read at 28 - 31 TB/s: 128 KB of weights per 64 rows are 42 us per launch at N = 768, under
// the 120 us that the pair tensor's own bytes take.  Read from row-major weights, a fragment touches 32
// cache lines per load instruction and costs the first-level cache four times as much.)
// Short workgroups, three or four of them per compute unit at different points of their lives,
// take the place of the resident kernels of rowgemm.hip: those hold 128 KB of weights per compute unit
// and two waves per SIMD, need eight row tiles per compute unit to have something for every wave, and end
// in a partial round of tiles.  They serve callers that hand in row-major weights and, out of the packed
// buffer, the large calls named at pp_resident().
#include "common.h"
#include "kernels.h"
#include "rowpieces.h"
#include "single_stage.h"
#include <algorithm>

namespace ptx {

namespace {

constexpr int kPpWaves = 4;
static_assert(kPpWaves == kStageWaves, "workgroups of both kinds in one launch");
constexpr int cmax(int a, int b) { return a > b ? a : b; }
// The launch's first `carried` workgroups run a stage of the single track (not on rows of 64 channels: no stack
// of that width has one, and the attention's kernel would spill).
#define PTX_CARRIED_STAGE()                          \
  if constexpr (KS > 4) {                            \
    if (blockIdx.x < carried) {                      \
      single_stage<TZ>(carry, blockIdx.x, smem);     \
      return;                                        \
    }                                                \
  }                                                  \
  const uint32_t block = blockIdx.x - carried, blocks = gridDim.x - carried

// Waves per SIMD that the register allocator leaves room for: three in 16-bit arithmetic (168 registers; the carried
// stages alone take 148), two on rows of 256 channels and in fp32.  Without that bound the carried stages take 32
// registers of the accumulation file on top of the kernel's 240 and one workgroup is left per compute unit
// (triattn_in on rows of 256 channels, 600 tokens: 566 us per launch; with two 377).
template <typename T, int KS> constexpr int kPpMinWaves = sizeof(T) == 2 && KS <= 8 ? 3 : 2;

// Hidden widths (see Widths in rowgemm.hip): 128 for rows of at most 128 channels, else the row width.
template <int KS> struct PpWidths {
  static constexpr int SL = KS > 8 ? KS : 8;
  static constexpr int HIDDEN = 16 * SL;
  static constexpr int HEADS = HIDDEN / 32;
};

// Which logical rows a tile of ROWS rows stands for.  linear: ROWS consecutive rows p = i * n + j (n is a multiple
// of the 16-byte vector length, so that vectors of consecutive rows stay inside one i); otherwise ROWS
// positions j of one i, the last tile of an i partial.
struct TileRows {
  static constexpr bool kPatch = false;
  int64_t p0;
  int i0, j0, n;
  int64_t n_rows;
  bool linear;
  __device__ __forceinline__ bool at(int r, int& i, int& j) const {
    if (linear) {
      const int64_t p = p0 + r;
      const bool ok = p < n_rows;
      const uint32_t pc = (uint32_t)(ok ? p : n_rows - 1);
      i = pc / (uint32_t)n;
      j = pc - i * (uint32_t)n;
      return ok;
    }
    i = i0;
    j = min(j0 + r, n - 1);
    return j0 + r < n;
  }
};
__device__ __forceinline__ TileRows tile_rows(int64_t tile, int rows, int n, int tiles_per_i) {
  TileRows t;
  t.n = n;
  t.n_rows = (int64_t)n * n;
  t.linear = tiles_per_i == 0;
  t.p0 = tile * rows;
  t.i0 = t.linear ? 0 : (int)((uint32_t)tile / (uint32_t)tiles_per_i);
  t.j0 = t.linear ? 0 : ((int)tile - t.i0 * tiles_per_i) * rows;
  return t;
}

struct ProjInParams {
  const void* x;          // pair tensor; logical row (i, j) at i * si + j * sj
  int64_t si, sj;
  const void *gamma, *beta;
  float eps;
  const void* packed;     // weight fragments (pair_pack)
  void* out[5];           // trimul_in: a, b; triattn_in: q, k, v^T, gate (or null), bias
  const void* mask;       // trimul_in: value of (i, k) at i * mi + k * mk, or null
  int64_t mi, mk;
  int n, pitch, backward;
  int tiles_per_i;        // triattn_in: 0 = linear tiles
  int heads;
  int slices;             // workgroups per tile, each with its share of the output columns (see in_slices)
  unsigned tiles;
  unsigned work;          // trimul_in: workgroups before those that write zeros only
  int share;              // trimul_in: a wave's chunks per slice
  float q_scale;
};

}  // namespace

// The output columns of a triangle multiplication's projection: a, b[c][i][k] = mask * sigmoid(gate) * projection in the
// contraction's fragment order, from the normalised rows in LDS of a patch of 4 * RBW outer indices i x 8 inner indices
// k, which makes a row block's 32 values of one channel 64 contiguous bytes.
template <typename T, int KS, int RBW, bool APART = false>
struct MulColumns {
  typedef typename Vec8<T>::type V8;
  typedef typename VecE<T>::type VE_t;
  typedef Cfg<T> C;
  static constexpr int CPM = PpWidths<KS>::HIDDEN / 32;    // chunks (of 32 channels) per operand
  static constexpr int CHW = 2 * CPM / kPpWaves;           // chunks per wave, all slices
  static constexpr int kStage = kPpWaves * 32 * C::PITCH * (int)sizeof(T) + 128 * RBW;   // LDS beside the rows': staging tiles, mask
  V8 w[2][KS];
  __device__ __forceinline__ void load_w(const ProjInParams& p, int ch, int lane) {
    const T* packed = (const T*)p.packed;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) w[t][kk] = packed_frag<T>(packed, (ch * 2 + t) * KS + kk, lane);
  }
  static __device__ __forceinline__ float* mask_of(char* stage_lds) { return reinterpret_cast<float*>(stage_lds + kStage - 128 * RBW); }
  // the patch's mask into LDS
  static __device__ __forceinline__ void put_mask(const ProjInParams& p, char* stage_lds, int pi0, int pk0) {
    if (threadIdx.x < 32 * RBW) {
      const int n = p.n, i = min(pi0 + (int)(threadIdx.x >> 3), n - 1), k = pk0 + (int)(threadIdx.x & 7);
      float mv = 1.0f;
      if (p.mask) mv = to_f32(((const T*)p.mask)[i * p.mi + min(k, n - 1) * p.mk]);
      mask_of(stage_lds)[threadIdx.x] = k < n ? mv : 0.0f;   // (the contraction relies on zeros between n and the pitch)
    }
  }
  // Patches along the inner index: whole K steps of the contraction.
  static __host__ __device__ __forceinline__ uint32_t patches_k(int n) { return 2 * ((uint32_t)(n + 15) >> 4); }
  // The K steps that hold nothing but the zeros up to the pitch, whole fragments: 16 channels of one operand and row block a
  // workgroup.  (As patches, which write 64 bytes at a time, they cost both multiplications 3 us of 72 at 200 tokens.)
  static int zero_groups(int n, int pitch) { return (pitch >> 4) > (n + 15) >> 4 ? ((n + 31) >> 5) * (2 * PpWidths<KS>::HIDDEN / 16) : 0; }
  static __device__ __forceinline__ void put_zeros(const ProjInParams& p, uint32_t group, int wave, int lane) {
    const int n_rb = (p.n + 31) >> 5, n_ks = p.pitch >> 4, ks0 = (p.n + 15) >> 4;
    const uint32_t per_rb = 2 * PpWidths<KS>::HIDDEN / 16, rb = group / per_rb;
    const int ch0 = (int)(group - rb * per_rb) * 16;
    T* const operand = (T*)(ch0 < PpWidths<KS>::HIDDEN ? p.out[0] : p.out[1]);
    VE_t zero;
#pragma unroll
    for (int t = 0; t < C::VE; ++t) zero[t] = (T)0.0f;
#pragma unroll 1
    for (int c = wave; c < 16; c += kPpWaves) {
      T* dst = operand + trimul_frag_offset((ch0 + c) % PpWidths<KS>::HIDDEN, (int)rb, ks0, n_rb, n_ks) + lane * C::VE;
      for (int e = 0; e < (n_ks - ks0) * kFragElems; e += kWave * C::VE) *reinterpret_cast<VE_t*>(dst + e) = zero;
    }
  }
  // chunks c_begin .. c_end - 1 of the wave's; the first one's weights have been requested
  __device__ __forceinline__ void run(const ProjInParams& p, const char* frag, char* stage_lds, int pi0, int pk0, int c_begin, int c_end, int wave,
                                      int lane) {
    T (*stage)[32 * C::PITCH] = reinterpret_cast<T (*)[32 * C::PITCH]>(stage_lds);
    const float* const lmask = mask_of(stage_lds);
    T* const out_a = (T*)p.out[0];
    T* const out_b = (T*)p.out[1];
    const int n = p.n, g = lane >> 5;
    T* st = stage[wave];
    const int n_rb = (n + 31) >> 5, n_ks = p.pitch >> 4;
    // this lane's vector of row block 0 inside a channel block's planes
    uint32_t rel[C::NPASS];
#pragma unroll
    for (int ps = 0; ps < C::NPASS; ++ps) {
      int chn, r0;
      stage_coord<T>(ps, lane, chn, r0);
      const int i = pi0 + (r0 >> 3);
      rel[ps] = (uint32_t)(trimul_frag_offset(chn, i >> 5, pk0 >> 4, n_rb, n_ks) + ((pk0 >> 3) & 1) * 256 + (i & 31) * 8 + (r0 & 7));
    }
#pragma unroll
    for (int c = 0; c < CHW; ++c) {
      if (c < c_begin || c >= c_end) continue;
      const int ch = wave * CHW + c;
      T* outp = (ch < CPM ? out_a : out_b) + trimul_frag_offset((ch % CPM) * 32, 0, 0, n_rb, n_ks);
#pragma unroll
      for (int rb = 0; rb < RBW; ++rb) {
        f32x16 acc[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
          const V8 xv = FragLds<T, KS>::get(frag, rb, kk, lane);
          mma32(acc[0], xv, w[0][kk]);   // lane <-> channel, register <-> row
          mma32(acc[1], xv, w[1][kk]);
        }
        // (APART: the products stay together; mixed with the staging below they take 138 registers from two row blocks of 16-bit rows and
        // leave three waves per SIMD instead of four.  us for both multiplications of bf16 rows, so / as here: 300 tokens 137 / 135, 352
        // 167 / 163, 387 218 / 214, 440 256 / 251)
        if constexpr (APART) __builtin_amdgcn_sched_barrier(0);
        if (rb == RBW - 1 && c + 1 < CHW && c + 1 < c_end) load_w(p, ch + 1, lane);
        float vals[16];
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
          const f32x4 m4 = *reinterpret_cast<const f32x4*>(&lmask[rb * 32 + 8 * qd + 4 * g]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * qd + e;
            vals[r] = m4[e] * sigmoidf_fast(acc[1][r]) * acc[0][r];
          }
        }
        wave_lds_sync();
        stage_put<T>(st, vals, lane);
        wave_lds_sync();
        // row block rb: outer indices 4 rb .. 4 rb + 3 further on; a patch of 4 RBW outer indices lies in one block of 32
#pragma unroll
        for (int ps = 0; ps < C::NPASS; ++ps) {
          int chn, r0;
          stage_coord<T>(ps, lane, chn, r0);
          *reinterpret_cast<VE_t*>(outp + rel[ps] + rb * 32) = stage_get_vec<T>(st, chn, r0);
        }
      }
    }
  }
};

// Tiles in the order of the memory rows they read.
template <typename T, typename TZ, int KS, int RBW>
__global__ __launch_bounds__(kPpWaves * 64, (kPpMinWaves<T, KS>)) void pp_trimul_in_kernel(ProjInParams p, SingleStage carry, unsigned carried) {
  typedef MulColumns<T, KS, RBW, sizeof(T) == 2 && sizeof(TZ) == 2 && RBW == 2> Columns;
  constexpr int kFrag = RBW * FragLds<T, KS>::ROWBLOCK;
  __shared__ __attribute__((aligned(16))) char smem[cmax(kFrag + Columns::kStage, kStageLds)];
  PTX_CARRIED_STAGE();
  char* const frag = smem;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = p.n;
  const uint32_t n_kb = Columns::patches_k(n), n_ip = (uint32_t)(n + 4 * RBW - 1) / (4 * RBW);
  if (block >= p.work) {
    Columns::put_zeros(p, block - p.work, wave, lane);
    return;
  }
  // (slices: of one row block only, see in_slices; fp32 rows keep their bounds, which cost them no wave: 440 tokens 351 us with, 356 without)
  constexpr bool kSliced = RBW == 1 || sizeof(TZ) == 4;
  // back to front behind a kernel that wrote the pair tensor front to back (the tail is what the memory-side cache still holds)
  const uint32_t tiles = p.tiles, slice = kSliced ? (block >= tiles) + (block >= 2 * tiles) + (block >= 3 * tiles) : 0u;
  const uint32_t bx = xcd_run(block - slice * tiles, tiles), tile = p.backward ? tiles - 1 - bx : bx;
  int pi0, pk0;
  if (p.backward) {   // incoming: the inner index is the slow one of z
    const uint32_t kb = tile / n_ip;
    pk0 = kb * 8;
    pi0 = (tile - kb * n_ip) * (4 * RBW);
  } else {
    const uint32_t ip = tile / n_kb;
    pi0 = ip * (4 * RBW);
    pk0 = (tile - ip * n_kb) * 8;
  }
  const int c_begin = kSliced ? slice * p.share : 0, c_end = kSliced ? c_begin + p.share : Columns::CHW;   // this slice's chunks of every wave
  Columns columns;
  typename RowPieces<TZ, KS>::V raw[RBW][RowPieces<TZ, KS>::NP];
  norm_rows<T, TZ, KS, RBW>(
      frag, (const TZ*)p.x,
      [&](int r) {
        const int i = min(pi0 + (r >> 3), n - 1), k = min(pk0 + (r & 7), n - 1);
        return i * p.si + k * p.sj;
      },
      (const T*)p.gamma, (const T*)p.beta, p.eps, wave, lane, raw);
  columns.load_w(p, wave * Columns::CHW + c_begin, lane);
  Columns::put_mask(p, smem + kFrag, pi0, pk0);
  __syncthreads();
  columns.run(p, frag, smem + kFrag, pi0, pk0, c_begin, c_end, wave, lane);
}

// The output columns of an attention projection: q (scaled), K, V^T, triangle bias and (GATE) sigmoid(gate) in the attention
// core's layouts, from a tile's normalised rows in LDS.  The waves take pairs of 32-column tiles in turn.  Rows: where
// the tile's rows lie, at(row, i, j); runs of VE rows from a multiple of VE on are consecutive j of one i.
template <typename T, int KS, int RBW, bool GATE>
struct AttnColumns {
  typedef typename Vec8<T>::type V8;
  typedef typename VecE<T>::type VE_t;
  typedef Cfg<T> C;
  static constexpr int HP = PpWidths<KS>::HEADS / 2;            // pairs of heads
  static constexpr int NPAIR = (GATE ? 4 : 3) * HP + 1;         // q, k, v (, gate): HP pairs of tiles each; the bias: one tile
  static constexpr int kStage = kPpWaves * 2 * 32 * C::PITCH * (int)sizeof(T);   // LDS beside the rows'
  V8 w[2][KS];
  __device__ __forceinline__ void load_w(const ProjInParams& p, int pair, int lane) {   // pair -> tiles 2 pair, 2 pair + 1 (the bias' tile twice)
    const T* packed = (const T*)p.packed;
    const int t0 = pair < NPAIR - 1 ? 2 * pair : 8 * HP, t1 = pair < NPAIR - 1 ? t0 + 1 : t0;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      w[0][kk] = packed_frag<T>(packed, t0 * KS + kk, lane);
      w[1][kk] = packed_frag<T>(packed, t1 * KS + kk, lane);
    }
  }
  // (the weights of pair `first` have been requested)
  template <typename Rows>
  __device__ __forceinline__ void run(const ProjInParams& p, const char* frag, char* stage_lds, const Rows tr, int first, int step, int wave, int lane) {
    T* const q_out = (T*)p.out[0];
    T* const gate_out = (T*)p.out[3];
    T (*stage)[2][32 * C::PITCH] = reinterpret_cast<T (*)[2][32 * C::PITCH]>(stage_lds);
    const int n = p.n;
    const int64_t n_rows = (int64_t)n * n;
    const int key_tiles = p.pitch >> 6, q_blocks = (n + 31) >> 5;
    const int64_t head_plane = (int64_t)n * key_tiles * kAttnTileElems;
#pragma unroll 1
    for (int pair = first; pair < NPAIR; pair += step) {
      const int which = pair < NPAIR - 1 ? pair / HP : 4;   // 0 q, 1 k, 2 v, 3 gate, 4 bias
      const int h0 = (pair % HP) * 2;
#pragma unroll
      for (int rb = 0; rb < RBW; ++rb) {
        f32x16 acc[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.0f;
        if (which == 2 || which == 4) {
#pragma unroll
          for (int kk = 0; kk < KS; ++kk) {
            const V8 xv = FragLds<T, KS>::get(frag, rb, kk, lane);
            mma32(acc[0], xv, w[0][kk]);   // lane <-> channel, register <-> row
            mma32(acc[1], xv, w[1][kk]);
          }
        } else {
#pragma unroll
          for (int kk = 0; kk < KS; ++kk) {
            const V8 xv = FragLds<T, KS>::get(frag, rb, kk, lane);
            mma32(acc[0], w[0][kk], xv);   // lane <-> row, register <-> channel
            mma32(acc[1], w[1][kk], xv);
          }
        }
        if (rb == RBW - 1 && pair + step < NPAIR) load_w(p, pair + step, lane);
        wave_lds_sync();
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          float vals[16];
          if (which == 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) vals[r] = to_f32(from_f32<T>(acc[t][r])) * p.q_scale;
          } else if (which == 4) {
#pragma unroll
            for (int r = 0; r < 16; ++r) vals[r] = acc[t][r] * 1.4426950408889634f;   // the core works in log2 units
          } else if (GATE && which == 3) {
#pragma unroll
            for (int r = 0; r < 16; ++r) vals[r] = sigmoidf_fast(acc[t][r]);
          } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) vals[r] = acc[t][r];
          }
          stage_put<T>(stage[wave][t], vals, lane);
        }
        wave_lds_sync();
        if (which == 2 || which == 4) {
          // vectors of VE consecutive keys of one i
          const int v0 = (lane % C::LPM) * C::VE;
          int i, j;
          const bool ok = tr.at(rb * 32 + v0, i, j);
          if (which == 2) {
            T* outp = (T*)p.out[2] + attn_v_offset(0, i, j, 0, n, key_tiles);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
              for (int ps = 0; ps < C::NPASS; ++ps) {
                int chn, r0;
                stage_coord<T>(ps, lane, chn, r0);
                if (ok) *reinterpret_cast<VE_t*>(outp + (h0 + t) * head_plane + chn * 8) = stage_get_vec<T>(stage[wave][t], chn, r0);
              }
          } else {
            T* outp = (T*)p.out[4];
#pragma unroll
            for (int ps = 0; ps < C::NPASS; ++ps) {
              int chn, r0;
              stage_coord<T>(ps, lane, chn, r0);
              if (ok && chn < p.heads)
                *reinterpret_cast<VE_t*>(outp + attn_b_offset(chn, i, j, q_blocks, key_tiles)) = stage_get_vec<T>(stage[wave][0], chn, r0);
            }
          }
        } else {
#pragma unroll
          for (int ps = 0; ps < C::NPASS; ++ps) {
            int mj, m0;
            stage_coord<T>(ps, lane, mj, m0);
            int i, j;
            const bool ok = tr.at(rb * 32 + mj, i, j);
            if (which == 1) {
              T* outp = (T*)p.out[1] + attn_k_offset(0, i, j, m0, n, key_tiles);
#pragma unroll
              for (int t = 0; t < 2; ++t)
                if (ok) *reinterpret_cast<VE_t*>(outp + (h0 + t) * head_plane) = stage_get_vec<T>(stage[wave][t], mj, m0);
            } else {
              T* outp = (GATE && which == 3 ? gate_out : q_out) + ((int64_t)i * n + j) * 32 + m0;
#pragma unroll
              for (int t = 0; t < 2; ++t)
                if (ok) *reinterpret_cast<VE_t*>(outp + (int64_t)(h0 + t) * n_rows * 32) = stage_get_vec<T>(stage[wave][t], mj, m0);
            }
          }
        }
      }
    }
  }
};

// q (scaled), K, V^T, triangle bias and (GATE) sigmoid(gate) in the attention core's layouts.
template <typename T, typename TZ, int KS, int RBW, bool GATE>
__global__ __launch_bounds__(kPpWaves * 64, (kPpMinWaves<T, KS>)) void pp_triattn_in_kernel(ProjInParams p, SingleStage carry, unsigned carried) {
  typedef AttnColumns<T, KS, RBW, GATE> Columns;
  constexpr int kFrag = RBW * FragLds<T, KS>::ROWBLOCK;
  __shared__ __attribute__((aligned(16))) char smem[cmax(kFrag + Columns::kStage, kStageLds)];
  PTX_CARRIED_STAGE();
  char* const frag = smem;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t tiles = p.tiles, slice = (block >= tiles) + (block >= 2 * tiles) + (block >= 3 * tiles);
  const uint32_t bx = xcd_run(block - slice * tiles, tiles);
  const int64_t tile = p.backward ? tiles - 1 - bx : bx;
  const TileRows tr = tile_rows(tile, 32 * RBW, p.n, p.tiles_per_i);
  Columns columns;
  typename RowPieces<TZ, KS>::V raw[RBW][RowPieces<TZ, KS>::NP];
  norm_rows<T, TZ, KS, RBW>(
      frag, (const TZ*)p.x,
      [&](int r) {
        int i, j;
        tr.at(r, i, j);
        return i * p.si + j * p.sj;
      },
      (const T*)p.gamma, (const T*)p.beta, p.eps, wave, lane, raw);
  const int first = wave + kPpWaves * (int)slice;
  columns.load_w(p, min(first, Columns::NPAIR - 1), lane);
  __syncthreads();
  columns.run(p, frag, smem + kFrag, tr, first, kPpWaves * p.slices, wave, lane);
}

namespace {
struct ProjOutParams {
  const void* z;          // pair tensor: LayerNorm input and residual; row (i, j) at i * si + j * sj (also of out)
  int64_t si, sj;
  const void *gamma, *beta;     // LayerNorm of z (trimul_out; triattn_out with the gate formed here)
  const void *gamma2, *beta2;   // trimul_out: LayerNorm of the triangle product
  float eps;
  const void* packed;     // weight fragments of this stage
  const void* packed_g;   // triattn_out: fragments of the gate's weights
  const void* x;          // trimul_out: triangle product [hidden][n][ldx]; triattn_out: attention output [heads][n * n][32]
  int ldx;
  void* out;
  int n, add_residual, tiles_per_i;
};
}  // namespace

// Element offset of a tile's row in z and out, or -1; clamped: past the end that of a row the tile has.
template <typename Rows> struct ZRow {
  const ProjOutParams& p;
  const Rows& tr;
  __device__ __forceinline__ int64_t operator()(int r) const {
    int i, j;
    const bool ok = tr.at(r, i, j);
    const int64_t o = i * p.si + j * p.sj;
    return ok ? o : -1;
  }
  __device__ __forceinline__ int64_t clamped(int r) const {
    int i, j;
    tr.at(r, i, j);
    return i * p.si + j * p.sj;
  }
};

// The update (W_z LN_out(x)) * sigmoid(W_g LN_in(z)) of a tile, left in LDS (returned) with the raw rows of z in registers;
// a barrier is due before it is read.
template <typename T, typename TZ, int KS, int RBW> struct MulOut {
  static constexpr int SL = PpWidths<KS>::SL, HIDDEN = PpWidths<KS>::HIDDEN, NOB = KS / 2;
  static constexpr int XP = 32 * RBW + 4;   // pitch of the triangle product's tile (elements)
  static constexpr int kXt = (int)sizeof(T) * HIDDEN * XP, kUpd = (int)sizeof(T) * 32 * RBW * kUpdPitch<KS>;
  static constexpr int kFrag = RBW * FragLds<T, KS>::ROWBLOCK, kFrag2 = RBW * FragLds<T, SL>::ROWBLOCK;
  static constexpr int kLds = kFrag + kFrag2 + cmax(kXt, kUpd);
  template <typename Rows>
  static __device__ __forceinline__ T* run(const ProjOutParams& p, const Rows& tr, char* smem, int wave, int lane,
                                           typename RowPieces<TZ, KS>::V (&raw)[RBW][RowPieces<TZ, KS>::NP]) {
    typedef typename Vec8<T>::type V8;
    typedef typename VecE<T>::type VE_t;
    typedef Cfg<T> C;
    char* const frag = smem;
    char* const frag2 = smem + kFrag;
    char* const scratch = smem + kFrag + kFrag2;
    const int n = p.n;
    const T* packed = (const T*)p.packed;

    // the triangle product's rows of every channel: vectors of VE rows, or for a patch of 8 i x 4 * RBW j of XE of
    // an i's j, in which order they then lie in LDS
    constexpr bool kPatch = Rows::kPatch;
    constexpr int JW = 4 * RBW, XE = kPatch && JW < C::VE ? JW : C::VE;
    typedef typename std::conditional<XE == C::VE, VE_t, u32x2>::type X_t;
    static_assert(sizeof(X_t) == XE * sizeof(T), "one vector");
    auto x_pos = [](int r) { return kPatch ? (r & 7) * JW + (r >> 3) : r; };
    constexpr int VPC = 32 * RBW / XE, NV = HIDDEN * VPC / (kPpWaves * 64);
    const int v0 = (threadIdx.x % VPC) * XE, c0 = threadIdx.x / VPC;
    X_t xv[NV];
    {
      int i, j;
      tr.at(kPatch ? (v0 % JW) * 8 + v0 / JW : v0, i, j);
      if (kPatch) j &= ~(XE - 1);   // (clamped to n - 1: the vector that holds it)
      // (a tile past the end of a plane re-reads its last vector: those rows are not stored)
      const int64_t off = min((int64_t)i * p.ldx + j, (int64_t)n * p.ldx - XE) & ~(int64_t)(XE - 1);
      const T* src = (const T*)p.x + off;
      const int64_t plane = (int64_t)n * p.ldx;
#pragma unroll
      for (int q = 0; q < NV; ++q) xv[q] = *reinterpret_cast<const X_t*>(src + (c0 + q * (kPpWaves * 64 / VPC)) * plane);
    }
    const ZRow<Rows> z_row{p, tr};
    norm_rows<T, TZ, KS, RBW>(
        frag, (const TZ*)p.z, [&](int r) { return z_row.clamped(r); }, (const T*)p.gamma, (const T*)p.beta, p.eps,
        wave, lane, raw);
    T* xt = reinterpret_cast<T*>(scratch);
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      u32x2* d = reinterpret_cast<u32x2*>(xt + (c0 + q * (kPpWaves * 64 / VPC)) * XP + v0);
      const u32x2* s = reinterpret_cast<const u32x2*>(&xv[q]);
      d[0] = s[0];
      if (sizeof(X_t) == 16) d[1] = s[sizeof(X_t) / 8 - 1];
    }
    __syncthreads();
    {
      typedef RowPieces<T, SL> RP;
      constexpr int PE = RP::PE, NP = RP::NP;
      const int j = lane & 7, r8 = wave * 8 + (lane >> 3);
      float gm[NP][PE], bt[NP][PE];
      load_affine_pieces<T, PE, NP>((const T*)p.gamma2, (const T*)p.beta2, j, gm, bt);
#pragma unroll
      for (int rb = 0; rb < RBW; ++rb) {
        float v[NP][PE];
#pragma unroll
        for (int q = 0; q < NP; ++q)
#pragma unroll
          for (int t = 0; t < PE; ++t) v[q][t] = to_f32(xt[(PE * (j + 8 * q) + t) * XP + x_pos(rb * 32 + r8)]);
        normalize_pieces<PE, NP>(v, gm, bt, p.eps);
#pragma unroll
        for (int q = 0; q < NP; ++q) put_piece<T, SL, PE>(frag2, rb, r8, j + 8 * q, v[q]);
      }
    }
    V8 wz[SL], wg[KS];
    auto load_w = [&](int ob) {
#pragma unroll
      for (int kk = 0; kk < SL; ++kk) wz[kk] = packed_frag<T>(packed, ob * (SL + KS) + kk, lane);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) wg[kk] = packed_frag<T>(packed, ob * (SL + KS) + SL + kk, lane);
    };
    if (wave < NOB) load_w(wave);
    __syncthreads();   // both operand tiles are complete, and the product's tile has been read
    T* upd = reinterpret_cast<T*>(scratch);
#pragma unroll
    for (int ob = wave; ob < NOB; ob += kPpWaves) {
#pragma unroll
      for (int rb = 0; rb < RBW; ++rb) {
        f32x16 az, ag;
#pragma unroll
        for (int r = 0; r < 16; ++r) az[r] = ag[r] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < SL; ++kk) mma32(az, wz[kk], FragLds<T, SL>::get(frag2, rb, kk, lane));
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) mma32(ag, wg[kk], FragLds<T, KS>::get(frag, rb, kk, lane));
        if (rb == RBW - 1 && ob + kPpWaves < NOB) load_w(ob + kPpWaves);
        float vals[16];
#pragma unroll
        for (int r = 0; r < 16; ++r)   // linear_z's output rounded to T, times the gate, rounded to T
          vals[r] = to_f32(from_f32<T>(az[r])) * sigmoidf_fast(ag[r]);
        put_update<T, KS>(upd, rb, ob, vals, lane);
      }
    }
    return upd;
  }
};

// out = [z +] (W_z LN_out(x)) * sigmoid(W_g LN_in(z)); out may be z.
template <typename T, typename TZ, int KS, int RBW>
__global__ __launch_bounds__(kPpWaves * 64, (kPpMinWaves<T, KS>)) void pp_trimul_out_kernel(ProjOutParams p, SingleStage carry, unsigned carried) {
  typedef MulOut<T, TZ, KS, RBW> Out;
  __shared__ __attribute__((aligned(16))) char smem[cmax(Out::kLds, kStageLds)];
  PTX_CARRIED_STAGE();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const TileRows tr = tile_rows(xcd_run(block, blocks), 32 * RBW, p.n, p.tiles_per_i);
  typename RowPieces<TZ, KS>::V raw[RBW][RowPieces<TZ, KS>::NP];
  const T* upd = Out::run(p, tr, smem, wave, lane, raw);
  __syncthreads();
  store_rows<T, TZ, KS, RBW>((TZ*)p.out, ZRow<TileRows>{p, tr}, upd, wave, lane, p.add_residual, raw);
}

// Row of the attention output that belongs to a tile's row (past the end: a valid one).
__device__ __forceinline__ int64_t o_row(const TileRows& tr, int r, int n) { return min(tr.p0 + r, (int64_t)n * n - 1); }

// The update W_o (gate * o) of a tile, as above.
// GATE: gate = sigmoid(W_g LN(z)) formed here (16-bit arithmetic; wave = head, and head + 4
// on rows of 256 channels), otherwise o arrives gated.  out may be z.  The gate formed here is neither written nor
// read: on rows of 64 / 256 channels, whose gates are twice / as wide as their rows, one update (projection, core,
// output) takes 270
// instead of 281 us at 512 tokens / 1169 instead of 1207 at 600 (per launch: 63 + 156 + 51, was 80 + 165 + 36; 323 + 571 + 275,
// was 392 + 603 + 212; 256 channels at 96 / 200 / 400 / 800 tokens: 43 / 118 / 481 / 2242, was 44 / 113 / 487 / 2349).  Two row
// blocks per workgroup on 256 channels: 292 us at 600, 43 instead of 32 at 200.
template <typename T, typename TZ, int KS, bool GATE, int RBW> struct AttnOut {
  static constexpr int SL = PpWidths<KS>::SL, NOB = KS / 2;
  static_assert(!GATE || sizeof(T) == 2, "gate formed here: 16-bit arithmetic");
  static constexpr int kFrag = GATE ? RBW * FragLds<T, KS>::ROWBLOCK : 16, kUpd = (int)sizeof(T) * 32 * RBW * kUpdPitch<KS>;
  static constexpr int kScratch = cmax(kFrag, kUpd);   // the normalised rows, then the update
  static constexpr int kLds = kScratch + RBW * FragLds<T, SL>::ROWBLOCK;
  template <typename Rows>
  static __device__ __forceinline__ T* run(const ProjOutParams& p, const Rows& tr, char* smem, int wave, int lane,
                                           typename RowPieces<TZ, KS>::V (&raw)[RBW][RowPieces<TZ, KS>::NP]) {
    typedef typename Vec8<T>::type V8;
    char* const scratch = smem;
    char* const fo = smem + kScratch;
    const int n = p.n, nl = lane & 31, g = lane >> 5;
    const int64_t n_rows = (int64_t)n * n;
    const T* packed = (const T*)p.packed;
    V8 w[SL];
    auto load_w = [&](int ob) {
#pragma unroll
      for (int kk = 0; kk < SL; ++kk) w[kk] = packed_frag<T>(packed, ob * SL + kk, lane);
    };
    // this wave's share of the attention output: heads wave, wave + 4, .. as fragments
    constexpr int HPW = PpWidths<KS>::HEADS / kPpWaves;
    V8 of[RBW][HPW][2];
#pragma unroll
    for (int rb = 0; rb < RBW; ++rb) {
      const int64_t pr = o_row(tr, rb * 32 + nl, p.n);
#pragma unroll
      for (int q = 0; q < HPW; ++q)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          of[rb][q][u] = load8<T>((const T*)p.x + ((int64_t)(wave + 4 * q) * n_rows + pr) * 32 + 16 * u + 8 * g);
    }
    const ZRow<Rows> z_row{p, tr};
    auto z_row0 = [&](int r) { return z_row.clamped(r); };
    if constexpr (GATE) {
      // (all of a wave's gate weights under the LayerNorm, the output's first under the last head's products: fetched
      // when needed, one after the other, they cost rows of 256 channels three waits instead of one)
      V8 wg[HPW][KS];
#pragma unroll
      for (int q = 0; q < HPW; ++q)
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) wg[q][kk] = packed_frag<T>((const T*)p.packed_g, (wave + 4 * q) * KS + kk, lane);
      norm_rows<T, TZ, KS, RBW>(scratch, (const TZ*)p.z, z_row0, (const T*)p.gamma, (const T*)p.beta, p.eps, wave, lane, raw);
      if (HPW == 1 && wave < NOB) load_w(wave);
      __syncthreads();
#pragma unroll
      for (int q = 0; q < HPW; ++q)
#pragma unroll
      for (int rb = 0; rb < RBW; ++rb) {
        f32x16 ag;
#pragma unroll
        for (int r = 0; r < 16; ++r) ag[r] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) mma32(ag, wg[q][kk], FragLds<T, KS>::get(scratch, rb, kk, lane));
        if (HPW > 1 && rb == RBW - 1 && q == HPW - 2) load_w(wave);
        // (weight rows packed so that registers 8 u + t are the channels 16 u + 8 g + t of the lane's own fragments;
        // gate and gated output rounded to T like the reference's sigmoid(linear_g(x)) and o * g)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const f32x8 ov = to_f32(of[rb][q][u]);
          f32x8 gated;
#pragma unroll
          for (int t = 0; t < 8; ++t) gated[t] = ov[t] * to_f32(from_f32<T>(sigmoidf_fast(ag[8 * u + t])));
          of[rb][q][u] = from_f32<T>(gated);
        }
      }
    } else {
      if (wave < NOB) load_w(wave);
      if (p.add_residual) {
        typedef RowPieces<TZ, KS> RP;
#pragma unroll
        for (int rb = 0; rb < RBW; ++rb) {
          const TZ* rp = (const TZ*)p.z + z_row0(rb * 32 + wave * 8 + (lane >> 3)) + RP::PE * (lane & 7);
#pragma unroll
          for (int q = 0; q < RP::NP; ++q) raw[rb][q] = *reinterpret_cast<const typename RP::V*>(rp + 8 * RP::PE * q);
        }
      }
    }
#pragma unroll
    for (int rb = 0; rb < RBW; ++rb)
#pragma unroll
      for (int q = 0; q < HPW; ++q)
#pragma unroll
        for (int u = 0; u < 2; ++u) FragLds<T, SL>::put(fo, rb, nl, 2 * (2 * (wave + 4 * q) + u) + g, of[rb][q][u]);
    __syncthreads();   // (and the normalised rows have been read)
    T* upd = reinterpret_cast<T*>(scratch);
#pragma unroll
    for (int ob = wave; ob < NOB; ob += kPpWaves) {
#pragma unroll
      for (int rb = 0; rb < RBW; ++rb) {
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < SL; ++kk) mma32(acc, w[kk], FragLds<T, SL>::get(fo, rb, kk, lane));
        if (rb == RBW - 1 && ob + kPpWaves < NOB) load_w(ob + kPpWaves);
        float vals[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) vals[r] = acc[r];
        put_update<T, KS>(upd, rb, ob, vals, lane);   // (rounded to T, as the module's output is)
      }
    }
    return upd;
  }
};

template <typename T, typename TZ, int KS, bool GATE, int RBW>
__global__ __launch_bounds__(kPpWaves * 64, (kPpMinWaves<T, KS>)) void pp_triattn_out_kernel(ProjOutParams p, SingleStage carry, unsigned carried) {
  typedef AttnOut<T, TZ, KS, GATE, RBW> Out;
  __shared__ __attribute__((aligned(16))) char smem[cmax(Out::kLds, kStageLds)];
  PTX_CARRIED_STAGE();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const TileRows tr = tile_rows(xcd_run(block, blocks), 32 * RBW, p.n, 0);
  typename RowPieces<TZ, KS>::V raw[RBW][RowPieces<TZ, KS>::NP];
  const T* upd = Out::run(p, tr, smem, wave, lane, raw);
  __syncthreads();
  store_rows<T, TZ, KS, RBW>((TZ*)p.out, ZRow<TileRows>{p, tr}, upd, wave, lane, p.add_residual, raw);
}

// ---- an output stage and the projection that reads its rows next, in one launch -------------------------
// A patch of 8 x 4 * RBW positions, for a projection that reads the pair tensor transposed (the ending node, the incoming
// multiplication): its logical rows (i, j) are z[j][i]; 8 consecutive j of one i follow each other.
struct PatchRows {
  int i0, j0, n;
  __device__ __forceinline__ bool at(int r, int& i, int& j) const {   // of the projection
    i = min(i0 + (r >> 3), n - 1);
    j = min(j0 + (r & 7), n - 1);
    return i0 + (r >> 3) < n && j0 + (r & 7) < n;
  }
};
struct PatchRowsT {   // the same positions as rows of z
  static constexpr bool kPatch = true;
  PatchRows t;
  __device__ __forceinline__ bool at(int r, int& i, int& j) const { return t.at(r, j, i); }
};
__device__ __forceinline__ int64_t o_row(const PatchRowsT& tr, int r, int n) {
  int i, j;
  tr.at(r, i, j);
  return (int64_t)i * n + j;
}

// z' = z + update (stored), and its rows, as stored, normalised with the next stage's parameters into `frag`.
template <typename T, typename TZ, int KS, int RBW, typename Off>
__device__ __forceinline__ void store_and_norm_rows(char* frag, TZ* out, Off off, const T* upd, const T* gamma, const T* beta, float eps, int wave,
                                                    int lane, typename RowPieces<TZ, KS>::V (&raw)[RBW][RowPieces<TZ, KS>::NP]) {
  typedef RowPieces<TZ, KS> RP;
  constexpr int PE = RP::PE, NP = RP::NP;
  const int j = lane & 7, r8 = wave * 8 + (lane >> 3);
  float gm[NP][PE], bt[NP][PE];
  load_affine_pieces<T, PE, NP>(gamma, beta, j, gm, bt);
  __syncthreads();   // (the update is complete, and what lay in `frag` has been read)
  store_rows<T, TZ, KS, RBW>(out, off, upd, wave, lane, 1, raw);
#pragma unroll
  for (int rb = 0; rb < RBW; ++rb) {
    float v[NP][PE];
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int t = 0; t < PE; ++t) v[q][t] = to_f32(raw[rb][q][t]);
    normalize_pieces<PE, NP>(v, gm, bt, eps);
#pragma unroll
    for (int q = 0; q < NP; ++q) put_piece<T, KS, PE>(frag, rb, r8, j + 8 * q, v[q]);
  }
}

// The output stage of a triangle multiplication and the projection of the starting node behind it: z' is read by nothing in
// between.
template <typename T, typename TZ, int KS, int RBW>
__global__ __launch_bounds__(kPpWaves * 64, (kPpMinWaves<T, KS>)) void pp_mul_out_attn_in_kernel(ProjOutParams p, ProjInParams pi, SingleStage carry,
                                                                                                unsigned carried) {
  typedef MulOut<T, TZ, KS, RBW> Out;
  typedef AttnColumns<T, KS, RBW, false> Columns;
  __shared__ __attribute__((aligned(16))) char smem[cmax(cmax(Out::kLds, Out::kFrag + Columns::kStage), kStageLds)];
  PTX_CARRIED_STAGE();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const TileRows tr = tile_rows(xcd_run(block, blocks), 32 * RBW, p.n, p.tiles_per_i);
  typename RowPieces<TZ, KS>::V raw[RBW][RowPieces<TZ, KS>::NP];
  const T* upd = Out::run(p, tr, smem, wave, lane, raw);
  store_and_norm_rows<T, TZ, KS, RBW>(smem, (TZ*)p.out, ZRow<TileRows>{p, tr}, upd, (const T*)pi.gamma, (const T*)pi.beta, pi.eps, wave, lane, raw);
  Columns columns;
  columns.load_w(pi, wave, lane);
  __syncthreads();
  columns.run(pi, smem, smem + Out::kFrag, tr, wave, kPpWaves, wave, lane);
}

// The output stage of the outgoing triangle multiplication and the projection of the incoming one behind it.
template <typename T, typename TZ, int KS, int RBW>
__global__ __launch_bounds__(kPpWaves * 64, (kPpMinWaves<T, KS>)) void pp_mul_out_mul_in_kernel(ProjOutParams p, ProjInParams pi, SingleStage carry,
                                                                                               unsigned carried) {
  typedef MulOut<T, TZ, KS, RBW> Out;
  typedef MulColumns<T, KS, RBW> Columns;
  __shared__ __attribute__((aligned(16))) char smem[cmax(cmax(Out::kLds, Out::kFrag + Columns::kStage), kStageLds)];
  PTX_CARRIED_STAGE();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t n_ip = (uint32_t)(p.n + 4 * RBW - 1) / (4 * RBW), work = n_ip * Columns::patches_k(p.n);
  if (block >= work) {
    Columns::put_zeros(pi, block - work, wave, lane);
    return;
  }
  const uint32_t tile = xcd_run(block, work), kb = tile / n_ip;
  const PatchRows tr = {(int)(tile - kb * n_ip) * (4 * RBW), (int)kb * 8, p.n};
  const PatchRowsT trt = {tr};
  typename RowPieces<TZ, KS>::V raw[RBW][RowPieces<TZ, KS>::NP];
  const T* upd = Out::run(p, trt, smem, wave, lane, raw);
  store_and_norm_rows<T, TZ, KS, RBW>(smem, (TZ*)p.out, ZRow<PatchRowsT>{p, trt}, upd, (const T*)pi.gamma, (const T*)pi.beta, pi.eps, wave, lane, raw);
  Columns columns;
  columns.load_w(pi, wave * Columns::CHW, lane);
  __syncthreads();
  Columns::put_mask(pi, smem + Out::kFrag, tr.i0, tr.j0);   // (over the update)
  __syncthreads();
  columns.run(pi, smem, smem + Out::kFrag, tr.i0, tr.j0, 0, Columns::CHW, wave, lane);
}

// The output stage of a starting node and the projection of the ending node behind it.
template <typename T, typename TZ, int KS, int RBW>
__global__ __launch_bounds__(kPpWaves * 64, (kPpMinWaves<T, KS>)) void pp_attn_out_attn_in_kernel(ProjOutParams p, ProjInParams pi, SingleStage carry,
                                                                                                 unsigned carried) {
  typedef AttnOut<T, TZ, KS, true, RBW> Out;
  typedef AttnColumns<T, KS, RBW, false> Columns;
  // the next stage's rows: behind the update, which other waves may still read, and the staging tiles
  constexpr int kNorm = cmax(Out::kScratch, Columns::kStage);
  __shared__ __attribute__((aligned(16))) char smem[cmax(kNorm + RBW * FragLds<T, KS>::ROWBLOCK, cmax(Out::kLds, kStageLds))];
  PTX_CARRIED_STAGE();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t n_ip = (uint32_t)(p.n + 4 * RBW - 1) / (4 * RBW), tile = xcd_run(block, blocks), jb = tile / n_ip;
  const PatchRows tr = {(int)(tile - jb * n_ip) * (4 * RBW), (int)jb * 8, p.n};
  const PatchRowsT trt = {tr};
  typename RowPieces<TZ, KS>::V raw[RBW][RowPieces<TZ, KS>::NP];
  const T* upd = Out::run(p, trt, smem, wave, lane, raw);
  store_and_norm_rows<T, TZ, KS, RBW>(smem + kNorm, (TZ*)p.out, ZRow<PatchRowsT>{p, trt}, upd, (const T*)pi.gamma, (const T*)pi.beta, pi.eps,
                                      wave, lane, raw);
  Columns columns;
  columns.load_w(pi, wave, lane);
  __syncthreads();
  columns.run(pi, smem + kNorm, smem, tr, wave, kPpWaves, wave, lane);
}
// ---------------------------------------------------------------------------
// Weight packing: every 32-row tile of the matrices as KS (or more) fragments, one lane's 8
// elements in 16-byte pieces [fragment][piece][lane].
// ---------------------------------------------------------------------------
namespace {
struct PackTile {
  const void* w;
  int row0, n_out, ldw, ksteps, frag0, perm;
  int raw;   // where the matrix is also kept row-major (elements; 0: not kept)
};
constexpr int kMaxPackTiles = 52;
struct PackList {
  PackTile t[kMaxPackTiles];
};
}  // namespace

template <typename T>
__global__ __launch_bounds__(256) void pair_pack_kernel(PackList list, T* __restrict__ packed) {
  const PackTile t = list.t[blockIdx.x];
  const int lane = threadIdx.x & 63;
  int m = lane & 31;
  if (t.perm) m = 16 * (m >> 4) + 8 * ((m >> 2) & 1) + 4 * ((m >> 3) & 1) + (m & 3);
  const T* row = (const T*)t.w + (int64_t)min(t.row0 + m, t.n_out - 1) * t.ldw + 8 * (lane >> 5);
  constexpr int PIECES = (int)sizeof(T) / 2;
  for (int kk = threadIdx.x >> 6; kk < t.ksteps; kk += 4) {
    typename Vec8<T>::type v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = row[16 * kk + e];
    const u32x4_t* s = reinterpret_cast<const u32x4_t*>(&v);
    u32x4_t* d = reinterpret_cast<u32x4_t*>(packed + (int64_t)(t.frag0 + kk) * kFragElems) + lane;
#pragma unroll
    for (int pc = 0; pc < PIECES; ++pc) d[pc * kWave] = s[pc];
    if (t.raw && t.row0 + m < t.n_out)
      store8<T>(packed + t.raw + (int64_t)(t.row0 + m) * t.ldw + 16 * kk + 8 * (lane >> 5), v);
  }
}

// On rows of 128 channels in 16-bit arithmetic the packed weights are followed by the matrices as they are, for the
// kernels of rowgemm.hip and attnout.hip, which keep them in LDS (resident_rows): as many bytes again.
static int64_t trimul_frag_elems(int c_z, int hidden) { return 5 * (int64_t)c_z * hidden + (int64_t)c_z * c_z; }
static int64_t triattn_frag_elems(int c_z, int heads) { return (int64_t)(4 * heads + 1) * 32 * c_z + (int64_t)c_z * heads * 32; }
static bool keeps_rows(int c_z, int hidden, bool bits16) { return bits16 && c_z == 128 && hidden == 128; }
constexpr int kMat = 128 * 128;   // such a matrix

int64_t pp_trimul_packed_elems(int c_z, int hidden, bool bits16) {
  return trimul_frag_elems(c_z, hidden) + (keeps_rows(c_z, hidden, bits16) ? 6 * kMat : 0);
}

template <typename T>
int pp_trimul_pack(const void* w_ap, const void* w_ag, const void* w_bp, const void* w_bg, const void* w_z,
                   const void* w_g, void* packed, int c_z, int hidden, hipStream_t stream) {
  PackList l;
  int nt = 0, f = 0;
  const int ks = c_z / 16, sl = hidden / 16, rows0 = (int)trimul_frag_elems(c_z, hidden);
  auto raw = [&](int i) { return keeps_rows(c_z, hidden, sizeof(T) == 2) ? rows0 + i * kMat : 0; };
  for (int op = 0; op < 2; ++op)
    for (int cb = 0; cb < hidden / 32; ++cb)
      for (int t = 0; t < 2; ++t) {
        l.t[nt++] = PackTile{op ? (t ? w_bg : w_bp) : (t ? w_ag : w_ap), 32 * cb, hidden, c_z, ks, f, 0, raw(2 * op + t)};
        f += ks;
      }
  for (int ob = 0; ob < c_z / 32; ++ob) {
    l.t[nt++] = PackTile{w_z, 32 * ob, c_z, hidden, sl, f, 0, raw(4)};
    l.t[nt++] = PackTile{w_g, 32 * ob, c_z, c_z, ks, f + sl, 0, raw(5)};
    f += sl + ks;
  }
  pair_pack_kernel<T><<<dim3(nt), dim3(256), 0, stream>>>(l, (T*)packed);
  return 0;
}

int64_t pp_triattn_packed_elems(int c_z, int heads, bool bits16) {
  return triattn_frag_elems(c_z, heads) + (keeps_rows(c_z, heads * 32, bits16) ? 5 * kMat + 4 * 128 : 0);
}

template <typename T>
int pp_triattn_pack(const void* w_q, const void* w_k, const void* w_v, const void* w_g, const void* w_b,
                    const void* w_o, void* packed, int c_z, int heads, hipStream_t stream) {
  PackList l;
  int nt = 0, f = 0;
  const int ks = c_z / 16, sl = heads * 2, rows0 = (int)triattn_frag_elems(c_z, heads);
  auto raw = [&](int i) { return keeps_rows(c_z, heads * 32, sizeof(T) == 2) ? rows0 + i * kMat : 0; };   // q, k, v, g, o, bias
  // (the gate formed in the output kernel: its rows permuted, see pp_triattn_out_kernel)
  const bool late = pp_late_gate(c_z, heads, sizeof(T) == 2);
  const void* m[4] = {w_q, w_k, w_v, w_g};
  for (int which = 0; which < 4; ++which)
    for (int h = 0; h < heads; ++h) {
      l.t[nt++] = PackTile{m[which], 32 * h, heads * 32, c_z, ks, f, which == 3 && late, raw(which)};
      f += ks;
    }
  l.t[nt++] = PackTile{w_b, 0, heads, c_z, ks, f, 0, raw(5)};
  f += ks;
  for (int ob = 0; ob < c_z / 32; ++ob) {
    l.t[nt++] = PackTile{w_o, 32 * ob, c_z, heads * 32, sl, f, 0, raw(4)};
    f += sl;
  }
  pair_pack_kernel<T><<<dim3(nt), dim3(256), 0, stream>>>(l, (T*)packed);
  return 0;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// Row blocks (of 32 rows) per workgroup, by the launch's number of rows.  More of them share the
// weights a wave fetches; fewer leave more workgroups and more of them per compute unit.  Lines from
// sweeps over n (us per launch, fp32 rows; c = channels):
//   trimul_in   c = 128: 1 / 2 at n = 128: 8.0 / 8.5, at 192: 14.5 / 13.8; 2 / 4 at 387: 41 / 43, 512: 62 / 61,
//               768: 184 / 157; c = 256: 1 / 2 at 128: 23 / 18, 2 / 4 at 256: 69 / 54, 600: 373 / 295
//   triattn_in  c = 128: as trimul_in for 1 / 2; 2 / 4 at 768: 180 / 181; c = 64: 2 / 4 at 512: 98 / 88;
//               c = 256: 1 / 2 at 128: 29 / 25, 2 / 4 at 600: 356 / 434 (registers)
//   trimul_out  c = 128: 1 / 2 at 387: 41 / 43, 512: 68 / 65, 768: 186 / 162; c = 64 at 512: 39 / 43; c = 256 at 600: 292 / 352
//   triattn_out c = 128: 1 / 2 at 256: 17.4 / 17.4, 387: 34.8 / 33.7, 768: 170 / 140; c = 64, 256: no gain
// 32-bit arithmetic: one (twice the registers per fragment).
static int in_row_blocks(int64_t rows, int ks, bool attention) {
  if (rows < (ks > 8 ? 96 * 96 : 160 * 160)) return 1;
  const int64_t four = attention ? (ks == 4 ? 400 * 400 : INT64_MAX) : (ks > 8 ? 200 * 200 : 448 * 448);
  return rows >= four ? 4 : 2;
}
static int out_row_blocks(int64_t rows, int ks, bool attention) {
  return ks == 8 && rows >= (attention ? 320 * 320 : 448 * 448) ? 2 : 1;
}

// Large calls on rows of 128 channels in 16-bit arithmetic take the kernels that keep all of the weights in LDS, one
// workgroup per compute unit (rowgemm.hip, attnout.hip), where those are faster: there the weights, which every tile here
// fetches from the L2, weigh as much as the rows. Only where 8 divides n (their 16-byte accesses) and no stage of the
// single track rides along.  us per launch, here / resident.  16-bit rows: trimul_in 640 tokens 94 / 100, 768 132 / 127, 1024
// 264 / 219, 1536 523 / 478; trimul_out 448 44.1 / 43.5, 512 55 / 52, 768 121 / 113, 1536 465 / 426; triattn_in 256 21.5 / 23.2,
// 384 34.8 / 33.6, 512 74 / 62, 768 162 / 149, 1536 632 / 592; triattn_out 640 75 / 78, 768 106 / 106, 1024 186 / 182, 1536
// 415 / 399.
// fp32 rows (within a stack): triattn_in 448 62 / 62, 512 86 / 78, 640 125 / 112, 768 182 / 167, 1024 324 / 299, 1536 722 / 694,
// 2048 1243 / 1262; trimul_in 1024 272 / 271, 1536 571 / 594, 2048 1183 / 1066 (1984 and 2304: the same block either way);
// trimul_out and triattn_out are faster here at every size (768: 151 / 154, 132 / 145).
bool pp_resident(RowStage stage, int n, int c_z, int hidden, bool bits16, bool rows16) {
  constexpr int kFrom16[4] = {704, 480, 352, 896};
  if (!keeps_rows(c_z, hidden, bits16) || n % 8 != 0) return false;
  if (rows16) return n >= kFrom16[stage];
  return stage == kTriAttnInStage ? n >= 480 && n < 1792 : stage == kTriMulInStage && n >= 2048;
}
template <typename T, typename TZ>
static bool resident_rows(RowStage stage, int n, int c_z, int hidden, const SingleStage* carry) {
  return pp_resident(stage, n, c_z, hidden, sizeof(T) == 2, sizeof(TZ) == 2) && !(carry && carry->kind != kStageNone);
}

// Workgroups per tile of a projection.  Where the tiles leave compute units idle, each takes a share of the output
// columns (and normalises the rows again): a wave then works through one set of columns instead of two or three.  fp32,
// whose sets take 4 us of matrix pipe each, up to three and a half workgroups per compute unit.  us, without / with: one
// fp32 block at 48 tokens 209 / 181, 64 215 / 195, 93 333 / 317 (128, which stays as it is: 347 / 352); two blocks of 256 channels at 64
// tokens 342 / 316; 16 blocks under autocast at 40 tokens 1230 / 1209, 64 1328 / 1316 (up to four workgroups per compute unit: 128
// 2000 / 2030, 160 2789 / 2843).
static int in_slices(int64_t tiles, int most, bool bits16) {
  int s = 1;
  while (s < most && tiles * (s + 1) <= (bits16 ? 256 : 900)) ++s;
  return s;
}

template <typename T, typename TZ, int KS>
static int pp_trimul_in_ks(ProjInParams p, const SingleStage* carry, hipStream_t stream) {
  typedef MulColumns<T, KS, 1> Columns;   // (its numbers of workgroups do not depend on the row blocks)
  const int rbw = sizeof(T) == 2 ? in_row_blocks((int64_t)p.n * p.n, KS, false) : 1;
  static const SingleStage none = {};
  if (carry && KS <= 4) single_stage_run(carry, stream);
  if (!carry || KS <= 4) carry = &none;
  const unsigned carried = single_stage_groups(carry);
  const unsigned tiles = (unsigned)((p.n + 4 * rbw - 1) / (4 * rbw)) * Columns::patches_k(p.n);
  constexpr int kChunks = PpWidths<KS>::HIDDEN / 64;   // per wave
  p.slices = rbw == 1 ? in_slices(tiles, kChunks, sizeof(T) == 2) : 1;
  if (kChunks % p.slices) --p.slices;   // (2 or 4 chunks: equal shares)
  p.tiles = tiles;
  p.share = kChunks / p.slices;
  p.work = tiles * p.slices;
  const dim3 grid(carried + p.work + Columns::zero_groups(p.n, p.pitch)), block(kPpWaves * 64);
  if constexpr (sizeof(T) == 2) {
    if (rbw == 4) {
      pp_trimul_in_kernel<T, TZ, KS, 4><<<grid, block, 0, stream>>>(p, *carry, carried);
      return 0;
    }
    if (rbw == 2) {
      pp_trimul_in_kernel<T, TZ, KS, 2><<<grid, block, 0, stream>>>(p, *carry, carried);
      return 0;
    }
  }
  pp_trimul_in_kernel<T, TZ, KS, 1><<<grid, block, 0, stream>>>(p, *carry, carried);
  return 0;
}

template <typename T, typename TZ>
int pp_trimul_in(const void* z, const void* mask, const void* ln_w, const void* ln_b, const void* packed, void* a,
                 void* b, int n, int c_z, int k_pitch, int incoming, float eps, const SingleStage* carry, hipStream_t stream) {
  if constexpr (sizeof(T) == 2) {
    if (resident_rows<T, TZ>(kTriMulInStage, n, c_z, 128, carry)) {
      const T* m = (const T*)packed + trimul_frag_elems(128, 128);
      return trimul_project<T, TZ>(z, mask, ln_w, ln_b, m, m + kMat, m + 2 * kMat, m + 3 * kMat, a, b, n, c_z, k_pitch, incoming,
                                   eps, stream);
    }
  }
  ProjInParams p = {};
  p.x = z;
  p.si = incoming ? c_z : (int64_t)n * c_z;
  p.sj = incoming ? (int64_t)n * c_z : c_z;
  p.gamma = ln_w;
  p.beta = ln_b;
  p.eps = eps;
  p.packed = packed;
  p.out[0] = a;
  p.out[1] = b;
  p.mask = mask;
  p.mi = incoming ? 1 : n;
  p.mk = incoming ? n : 1;
  p.n = n;
  p.pitch = k_pitch;
  p.backward = incoming != 0;
  if (c_z == 64) return pp_trimul_in_ks<T, TZ, 4>(p, carry, stream);
  if (c_z == 256) {
    if constexpr (sizeof(T) == 2) return pp_trimul_in_ks<T, TZ, 16>(p, carry, stream);
    else return -1;
  }
  return pp_trimul_in_ks<T, TZ, 8>(p, carry, stream);
}

template <typename T, typename TZ, int KS, bool GATE>
static int pp_triattn_in_ks(ProjInParams p, const SingleStage* carry, hipStream_t stream) {
  const int rbw = sizeof(T) == 2 ? in_row_blocks((int64_t)p.n * p.n, KS, true) : 1;
  const int rows = 32 * rbw;
  p.tiles_per_i = p.n % Cfg<T>::VE == 0 ? 0 : (p.n + rows - 1) / rows;
  const int64_t tiles = p.tiles_per_i ? (int64_t)p.n * p.tiles_per_i : ((int64_t)p.n * p.n + rows - 1) / rows;
  static const SingleStage none = {};
  if (carry && KS <= 4) single_stage_run(carry, stream);
  if (!carry || KS <= 4) carry = &none;
  const unsigned carried = single_stage_groups(carry);
  p.slices = in_slices(tiles, ((GATE ? 4 : 3) * PpWidths<KS>::HEADS / 2 + kPpWaves) / kPpWaves, sizeof(T) == 2);
  p.tiles = (unsigned)tiles;
  const dim3 grid(carried + p.tiles * p.slices), block(kPpWaves * 64);
  if constexpr (sizeof(T) == 2) {
    if constexpr (KS == 4) {
      if (rbw == 4) {
        pp_triattn_in_kernel<T, TZ, KS, 4, GATE><<<grid, block, 0, stream>>>(p, *carry, carried);
        return 0;
      }
    }
    if (rbw == 2) {
      pp_triattn_in_kernel<T, TZ, KS, 2, GATE><<<grid, block, 0, stream>>>(p, *carry, carried);
      return 0;
    }
  }
  pp_triattn_in_kernel<T, TZ, KS, 1, GATE><<<grid, block, 0, stream>>>(p, *carry, carried);
  return 0;
}

template <typename T, typename TZ>
int pp_triattn_in(const void* z, const void* ln_w, const void* ln_b, const void* packed, void* q, void* k, void* vt,
                  void* g, void* tri_bias, int n, int c_z, int heads, int key_pitch, int transposed, float eps,
                  const SingleStage* carry, hipStream_t stream) {
  if constexpr (sizeof(T) == 2) {
    if (resident_rows<T, TZ>(kTriAttnInStage, n, c_z, heads * 32, carry)) {
      const T* m = (const T*)packed + triattn_frag_elems(128, 4);
      return triattn_project<T, TZ>(z, ln_w, ln_b, m, m + kMat, m + 2 * kMat, m + 3 * kMat, m + 5 * kMat, q, k, vt, nullptr,
                                    tri_bias, n, c_z, heads, 32, key_pitch, transposed, eps, stream);
    }
  }
  ProjInParams p = {};
  p.x = z;
  p.si = transposed ? c_z : (int64_t)n * c_z;
  p.sj = transposed ? (int64_t)n * c_z : c_z;
  p.gamma = ln_w;
  p.beta = ln_b;
  p.eps = eps;
  p.packed = packed;
  p.out[0] = q; p.out[1] = k; p.out[2] = vt; p.out[3] = g; p.out[4] = tri_bias;
  p.n = n;
  p.pitch = key_pitch;
  p.backward = 1;
  p.heads = heads;
  p.q_scale = 1.4426950408889634f / sqrtf(32.0f);   // log2(e) / sqrt(d), see triattn.hip
  if (c_z == 64) return pp_triattn_in_ks<T, TZ, 4, sizeof(T) == 4>(p, carry, stream);
  if (c_z == 256) {
    if constexpr (sizeof(T) == 2) return pp_triattn_in_ks<T, TZ, 16, false>(p, carry, stream);
    else return -1;
  }
  if constexpr (sizeof(T) == 2) return pp_triattn_in_ks<T, TZ, 8, false>(p, carry, stream);
  else return pp_triattn_in_ks<T, TZ, 8, true>(p, carry, stream);
}

template <typename T, typename TZ, int KS>
static int pp_trimul_out_ks(ProjOutParams p, const SingleStage* carry, hipStream_t stream) {
  const int rbw = sizeof(T) == 2 ? out_row_blocks((int64_t)p.n * p.n, KS, false) : 1, rows = 32 * rbw;
  p.tiles_per_i = p.ldx == p.n && p.n % Cfg<T>::VE == 0 ? 0 : (p.n + rows - 1) / rows;
  const int64_t tiles = p.tiles_per_i ? (int64_t)p.n * p.tiles_per_i : ((int64_t)p.n * p.n + rows - 1) / rows;
  static const SingleStage none = {};
  if (carry && KS <= 4) single_stage_run(carry, stream);
  if (!carry || KS <= 4) carry = &none;
  const unsigned carried = single_stage_groups(carry);
  const dim3 grid(carried + (unsigned)tiles), block(kPpWaves * 64);
  if constexpr (sizeof(T) == 2 && KS == 8) {
    if (rbw == 2) {
      pp_trimul_out_kernel<T, TZ, KS, 2><<<grid, block, 0, stream>>>(p, *carry, carried);
      return 0;
    }
  }
  pp_trimul_out_kernel<T, TZ, KS, 1><<<grid, block, 0, stream>>>(p, *carry, carried);
  return 0;
}

template <typename T, typename TZ, int KS, bool GATE>
static int pp_triattn_out_ks(const ProjOutParams& p, const SingleStage* carry, hipStream_t stream) {
  const int rbw = sizeof(T) == 2 ? out_row_blocks((int64_t)p.n * p.n, KS, true) : 1, rows = 32 * rbw;
  static const SingleStage none = {};
  if (carry && KS <= 4) single_stage_run(carry, stream);
  if (!carry || KS <= 4) carry = &none;
  const unsigned carried = single_stage_groups(carry);
  const dim3 grid(carried + (unsigned)(((int64_t)p.n * p.n + rows - 1) / rows)), block(kPpWaves * 64);
  if constexpr (sizeof(T) == 2 && KS == 8) {
    if (rbw == 2) {
      pp_triattn_out_kernel<T, TZ, KS, GATE, 2><<<grid, block, 0, stream>>>(p, *carry, carried);
      return 0;
    }
  }
  pp_triattn_out_kernel<T, TZ, KS, GATE, 1><<<grid, block, 0, stream>>>(p, *carry, carried);
  return 0;
}

template <typename T, typename TZ>
int pp_trimul_out(const void* x, int ldx, const void* z, const void* ln_in_w, const void* ln_in_b,
                  const void* ln_out_w, const void* ln_out_b, const void* packed, void* out, int n, int c_z,
                  int hidden, int add_residual, float eps, const SingleStage* carry, hipStream_t stream) {
  if constexpr (sizeof(T) == 2) {
    if (ldx == n && resident_rows<T, TZ>(kTriMulOutStage, n, c_z, hidden, carry)) {
      const T* m = (const T*)packed + trimul_frag_elems(128, 128);
      return trimul_output<T, TZ>(x, z, ln_in_w, ln_in_b, ln_out_w, ln_out_b, m + 4 * kMat, m + 5 * kMat, out, n, c_z,
                                  add_residual, eps, stream);
    }
  }
  ProjOutParams p = {};
  p.z = z;
  p.si = (int64_t)n * c_z;
  p.sj = c_z;
  p.gamma = ln_in_w;
  p.beta = ln_in_b;
  p.gamma2 = ln_out_w;
  p.beta2 = ln_out_b;
  p.eps = eps;
  p.packed = (const T*)packed + (int64_t)4 * c_z * hidden;
  p.x = x;
  p.ldx = ldx;
  p.out = out;
  p.n = n;
  p.add_residual = add_residual;
  if (c_z == 64) return pp_trimul_out_ks<T, TZ, 4>(p, carry, stream);
  if (c_z == 256) {
    if constexpr (sizeof(T) == 2) return pp_trimul_out_ks<T, TZ, 16>(p, carry, stream);
    else return -1;
  }
  return pp_trimul_out_ks<T, TZ, 8>(p, carry, stream);
}

template <typename T, typename TZ>
int pp_triattn_out(const void* o, const void* z, const void* ln_w, const void* ln_b, const void* packed, void* out,
                   int n, int c_z, int heads, int transposed, int add_residual, float eps, const SingleStage* carry, hipStream_t stream) {
  if constexpr (sizeof(T) == 2) {
    if (resident_rows<T, TZ>(kTriAttnOutStage, n, c_z, heads * 32, carry)) {
      const T* m = (const T*)packed + triattn_frag_elems(128, 4);
      return triattn_gate_output<TZ>(o, z, ln_w, ln_b, m + 3 * kMat, m + 4 * kMat, out, n, transposed, add_residual, eps, stream);
    }
  }
  ProjOutParams p = {};
  p.z = z;
  p.si = transposed ? c_z : (int64_t)n * c_z;
  p.sj = transposed ? (int64_t)n * c_z : c_z;
  p.gamma = ln_w;
  p.beta = ln_b;
  p.eps = eps;
  p.packed = (const T*)packed + (int64_t)(4 * heads + 1) * 32 * c_z;
  p.packed_g = (const T*)packed + (int64_t)3 * heads * 32 * c_z;
  p.x = o;
  p.out = out;
  p.n = n;
  p.add_residual = add_residual;
  if (c_z == 64) return pp_triattn_out_ks<T, TZ, 4, sizeof(T) == 2>(p, carry, stream);
  if (c_z == 256) {
    if constexpr (sizeof(T) == 2) return pp_triattn_out_ks<T, TZ, 16, true>(p, carry, stream);
    else return -1;
  }
  return pp_triattn_out_ks<T, TZ, 8, sizeof(T) == 2>(p, carry, stream);
}

// ---- an output stage with the next projection ----
// Where the two stages are faster in one launch.  They save a launch, its wait for the rows and one reading of the pair
// tensor, and give up the kernel with all weights in LDS that a projection by itself may take (pp_resident), on rows of 64 and 128
// channels tiles of four row blocks, on 256 tiles of two; the ending node's patches read the attention output and the rows in
// shorter runs.  us per block, no / the first / both pairs joined: 128 channels, fp32 rows, 64 tokens 85.1 / 84.1 / 79.2, 93 119 / 116 / 110, 160 173
// / 169 / 164, 256 300 / 290 / 278, 387 739 / 723 / 714, 512 1115 / 1109 / 1102, 576 1421 / 1409 / 1429, 640 1774 / 1775 / 1789, 768 2601 / 2596 /
// 2613, 1500 (no such kernel) 13264 / 13160 / 13226, 2048 27462 / 27528 / 27682; 16-bit rows, 256 262 / 259 / 251, 440 769 / 750 / 747, 480 918 / 922 / 924, 768
// 2354 / 2402 / 2437; 64 channels, 128 101 / 97 / 94, 512 790 / 792 / 790, 1200 6191 / 6171 / 6147, 1500 10724 / 10774 / 10803; 256 channels, 96 240 / 234 / 228, 256
// 715 / 715 / 714, 300 1114 / 1133 / 1139.
// The two multiplications (up to 256 tokens, where the products take the operands of any patch order from the L2), us per block
// without / with: 40 tokens 74.5 / 68.6, 93 110 / 102, 128 118 / 115, 200 226 / 216, 256 276 / 275; without a single track 200 221 / 213, 256
// 263 / 257; 64 channels 64 60 / 57, 200 169 / 165.
bool pp_joined(int pair, int n, int c_z, int hidden, bool rows16) {
  if (pair == 0) return n <= 256 && c_z <= 128;
  if (c_z == 256) return n <= 256;
  if (c_z == 64) return n <= 1280;
  const bool first = n < (rows16 ? 480 : 528) || (n < 1792 && !pp_resident(kTriAttnInStage, n, c_z, hidden, true, rows16));
  return first && (pair == 1 || n < 600);
}
static int merged_row_blocks(int64_t rows, int ks) { return ks <= 8 && rows >= 160 * 160 ? 2 : 1; }

static void attn_in_params(ProjInParams& p, const void* ln_w, const void* ln_b, const void* packed, void* q, void* k, void* vt, void* tri_bias,
                           int n, int heads, int key_pitch, float eps) {
  p.gamma = ln_w;
  p.beta = ln_b;
  p.eps = eps;
  p.packed = packed;
  p.out[0] = q; p.out[1] = k; p.out[2] = vt; p.out[4] = tri_bias;
  p.n = n;
  p.pitch = key_pitch;
  p.heads = heads;
  p.q_scale = 1.4426950408889634f / sqrtf(32.0f);   // log2(e) / sqrt(d), see triattn.hip
}

template <typename TZ, int KS>
static void mul_out_attn_in_ks(ProjOutParams p, const ProjInParams& pi, const SingleStage* carry, hipStream_t stream) {
  const int rbw = merged_row_blocks((int64_t)p.n * p.n, KS), rows = 32 * rbw;
  p.tiles_per_i = p.ldx == p.n && p.n % Cfg<bf16_t>::VE == 0 ? 0 : (p.n + rows - 1) / rows;
  const int64_t tiles = p.tiles_per_i ? (int64_t)p.n * p.tiles_per_i : ((int64_t)p.n * p.n + rows - 1) / rows;
  static const SingleStage none = {};
  if (carry && KS <= 4) single_stage_run(carry, stream);
  if (!carry || KS <= 4) carry = &none;
  const unsigned carried = single_stage_groups(carry);
  const dim3 grid(carried + (unsigned)tiles), block(kPpWaves * 64);
  if constexpr (KS <= 8) {
    if (rbw == 2) {
      pp_mul_out_attn_in_kernel<bf16_t, TZ, KS, 2><<<grid, block, 0, stream>>>(p, pi, *carry, carried);
      return;
    }
  }
  pp_mul_out_attn_in_kernel<bf16_t, TZ, KS, 1><<<grid, block, 0, stream>>>(p, pi, *carry, carried);
}

template <typename TZ, int KS>
static void attn_out_attn_in_ks(const ProjOutParams& p, const ProjInParams& pi, const SingleStage* carry, hipStream_t stream) {
  const int rbw = merged_row_blocks((int64_t)p.n * p.n, KS);
  static const SingleStage none = {};
  if (carry && KS <= 4) single_stage_run(carry, stream);
  if (!carry || KS <= 4) carry = &none;
  const unsigned carried = single_stage_groups(carry);
  const dim3 grid(carried + (unsigned)((p.n + 4 * rbw - 1) / (4 * rbw)) * (unsigned)((p.n + 7) / 8)), block(kPpWaves * 64);
  if constexpr (KS <= 8) {
    if (rbw == 2) {
      pp_attn_out_attn_in_kernel<bf16_t, TZ, KS, 2><<<grid, block, 0, stream>>>(p, pi, *carry, carried);
      return;
    }
  }
  pp_attn_out_attn_in_kernel<bf16_t, TZ, KS, 1><<<grid, block, 0, stream>>>(p, pi, *carry, carried);
}

template <typename TZ>
int pp_trimul_out_triattn_in(const void* x, int ldx, const void* z, const void* ln_in_w, const void* ln_in_b, const void* ln_out_w,
                             const void* ln_out_b, const void* packed, void* out, const void* att_ln_w, const void* att_ln_b,
                             const void* att_packed, void* q, void* k, void* vt, void* tri_bias, int n, int c_z, int hidden, int heads,
                             int key_pitch, float eps, const SingleStage* carry, hipStream_t stream) {
  ProjOutParams p = {};
  p.z = z;
  p.si = (int64_t)n * c_z;
  p.sj = c_z;
  p.gamma = ln_in_w;
  p.beta = ln_in_b;
  p.gamma2 = ln_out_w;
  p.beta2 = ln_out_b;
  p.eps = eps;
  p.packed = (const bf16_t*)packed + (int64_t)4 * c_z * hidden;
  p.x = x;
  p.ldx = ldx;
  p.out = out;
  p.n = n;
  p.add_residual = 1;
  ProjInParams pi = {};
  attn_in_params(pi, att_ln_w, att_ln_b, att_packed, q, k, vt, tri_bias, n, heads, key_pitch, eps);
  if (c_z == 64) mul_out_attn_in_ks<TZ, 4>(p, pi, carry, stream);
  else if (c_z == 256) mul_out_attn_in_ks<TZ, 16>(p, pi, carry, stream);
  else mul_out_attn_in_ks<TZ, 8>(p, pi, carry, stream);
  return 0;
}

template <typename TZ>
int pp_triattn_out_triattn_in(const void* o, const void* z, const void* ln_w, const void* ln_b, const void* packed, void* out,
                              const void* next_ln_w, const void* next_ln_b, const void* next_packed, void* q, void* k, void* vt,
                              void* tri_bias, int n, int c_z, int heads, int key_pitch, float eps, const SingleStage* carry,
                              hipStream_t stream) {
  ProjOutParams p = {};
  p.z = z;
  p.si = (int64_t)n * c_z;
  p.sj = c_z;
  p.gamma = ln_w;
  p.beta = ln_b;
  p.eps = eps;
  p.packed = (const bf16_t*)packed + (int64_t)(4 * heads + 1) * 32 * c_z;
  p.packed_g = (const bf16_t*)packed + (int64_t)3 * heads * 32 * c_z;
  p.x = o;
  p.out = out;
  p.n = n;
  p.add_residual = 1;
  ProjInParams pi = {};
  attn_in_params(pi, next_ln_w, next_ln_b, next_packed, q, k, vt, tri_bias, n, heads, key_pitch, eps);
  if (c_z == 64) attn_out_attn_in_ks<TZ, 4>(p, pi, carry, stream);
  else if (c_z == 256) attn_out_attn_in_ks<TZ, 16>(p, pi, carry, stream);
  else attn_out_attn_in_ks<TZ, 8>(p, pi, carry, stream);
  return 0;
}
template <typename TZ, int KS>
static void mul_out_mul_in_ks(const ProjOutParams& p, const ProjInParams& pi, const SingleStage* carry, hipStream_t stream) {
  const int rbw = merged_row_blocks((int64_t)p.n * p.n, KS);
  static const SingleStage none = {};
  if (carry && KS <= 4) single_stage_run(carry, stream);
  if (!carry || KS <= 4) carry = &none;
  const unsigned carried = single_stage_groups(carry);
  typedef MulColumns<bf16_t, KS, 1> Columns;
  const unsigned work = (unsigned)((p.n + 4 * rbw - 1) / (4 * rbw)) * Columns::patches_k(p.n);
  const dim3 grid(carried + work + Columns::zero_groups(pi.n, pi.pitch)), block(kPpWaves * 64);
  if (rbw == 2) pp_mul_out_mul_in_kernel<bf16_t, TZ, KS, 2><<<grid, block, 0, stream>>>(p, pi, *carry, carried);
  else pp_mul_out_mul_in_kernel<bf16_t, TZ, KS, 1><<<grid, block, 0, stream>>>(p, pi, *carry, carried);
}

template <typename TZ>
int pp_trimul_out_trimul_in(const void* x, int ldx, const void* z, const void* mask, const void* ln_in_w, const void* ln_in_b,
                            const void* ln_out_w, const void* ln_out_b, const void* packed, void* out, const void* next_ln_w,
                            const void* next_ln_b, const void* next_packed, void* a, void* b, int n, int c_z, int hidden, int k_pitch,
                            float eps, const SingleStage* carry, hipStream_t stream) {
  ProjOutParams p = {};
  p.z = z;
  p.si = (int64_t)n * c_z;
  p.sj = c_z;
  p.gamma = ln_in_w;
  p.beta = ln_in_b;
  p.gamma2 = ln_out_w;
  p.beta2 = ln_out_b;
  p.eps = eps;
  p.packed = (const bf16_t*)packed + (int64_t)4 * c_z * hidden;
  p.x = x;
  p.ldx = ldx;
  p.out = out;
  p.n = n;
  p.add_residual = 1;
  ProjInParams pi = {};
  pi.gamma = next_ln_w;
  pi.beta = next_ln_b;
  pi.eps = eps;
  pi.packed = next_packed;
  pi.out[0] = a;
  pi.out[1] = b;
  pi.mask = mask;
  pi.mi = 1;
  pi.mk = n;
  pi.n = n;
  pi.pitch = k_pitch;
  if (c_z == 64) mul_out_mul_in_ks<TZ, 4>(p, pi, carry, stream);
  else if (c_z == 128) mul_out_mul_in_ks<TZ, 8>(p, pi, carry, stream);
  else return -1;
  return 0;
}
#define PTX_INSTANTIATE_MERGED(TZ)                                                                                    \
  template int pp_trimul_out_trimul_in<TZ>(const void*, int, const void*, const void*, const void*, const void*,      \
                                           const void*, const void*, const void*, void*, const void*, const void*,    \
                                           const void*, void*, void*, int, int, int, int, float, const SingleStage*,  \
                                           hipStream_t);                                                              \
  template int pp_trimul_out_triattn_in<TZ>(const void*, int, const void*, const void*, const void*, const void*,     \
                                            const void*, const void*, void*, const void*, const void*, const void*,   \
                                            void*, void*, void*, void*, int, int, int, int, int, float,               \
                                            const SingleStage*, hipStream_t);                                         \
  template int pp_triattn_out_triattn_in<TZ>(const void*, const void*, const void*, const void*, const void*, void*,  \
                                             const void*, const void*, const void*, void*, void*, void*, void*, int,  \
                                             int, int, int, float, const SingleStage*, hipStream_t);
PTX_INSTANTIATE_MERGED(float)
PTX_INSTANTIATE_MERGED(bf16_t)
#undef PTX_INSTANTIATE_MERGED

#define PTX_INSTANTIATE_PACK(T)                                                                                        \
  template int pp_trimul_pack<T>(const void*, const void*, const void*, const void*, const void*, const void*, void*, \
                                 int, int, hipStream_t);                                                              \
  template int pp_triattn_pack<T>(const void*, const void*, const void*, const void*, const void*, const void*,       \
                                  void*, int, int, hipStream_t);
PTX_INSTANTIATE_PACK(float)
PTX_INSTANTIATE_PACK(bf16_t)
#undef PTX_INSTANTIATE_PACK
#define PTX_INSTANTIATE(T, TZ)                                                                                        \
  template int pp_trimul_in<T, TZ>(const void*, const void*, const void*, const void*, const void*, void*, void*,    \
                                   int, int, int, int, float, const SingleStage*, hipStream_t);                                          \
  template int pp_triattn_in<T, TZ>(const void*, const void*, const void*, const void*, void*, void*, void*, void*,  \
                                    void*, int, int, int, int, int, float, const SingleStage*, hipStream_t);                             \
  template int pp_trimul_out<T, TZ>(const void*, int, const void*, const void*, const void*, const void*,            \
                                    const void*, const void*, void*, int, int, int, int, float, const SingleStage*, hipStream_t);        \
  template int pp_triattn_out<T, TZ>(const void*, const void*, const void*, const void*, const void*, void*, int,    \
                                     int, int, int, int, float, const SingleStage*, hipStream_t);
PTX_INSTANTIATE(float, float)
PTX_INSTANTIATE(bf16_t, bf16_t)
PTX_INSTANTIATE(bf16_t, float)
#undef PTX_INSTANTIATE

}  // namespace ptx
