// Triangle attention core: flash-style online softmax on MFMA, the N^3 logits
// are never written anywhere.
//
// One workgroup (4 or 8 waves) owns one row i, or two, of one head h and 128 or 256 queries; each
// wave owns 32 queries and walks over the keys in staged tiles of 64, which it
// processes as two halves of 32 keys (16 logit registers at a time: four waves
// fit a SIMD).  Per half:
//   S^T[key][query]  = K Q^T + bias     2 + 2 MFMA
//   online softmax along keys = along the registers of a lane (+ one exchange
//   with the other half-wave), because MFMA puts the query on the lane
//   O^T[d][query]   += V^T P^T          2 MFMA, P^T taken straight from the S^T
//   accumulators with no shuffle
// MFMA row m of half u is mapped to key 32*((m>>2)&1) + 16*u + 4*(m>>3) + (m&3),
// which makes register r of half-wave g hold key 32*g + 16*u + r: 16 consecutive
// keys -> 16-byte bias loads, and 8 consecutive keys per P.V operand slot group.
// The triangle bias is the initial value of the S^T accumulators (converted to fp32 if it
// is stored in 16 bits).  q and the bias are stored multiplied by log2(e) (by the projection
// kernel), so on the common path the vector ALU executes per logit one conversion, one exp2,
// half a packed bf16 convert and half a dot2 (the row sum).
// K and V^T tiles are shared by the waves through LDS in fragment order (two tiles, one barrier per
// tile; 16-bit tiles arrive by direct-to-LDS loads); the bias tile is private to a wave
// and read straight from global (L2-resident: workgroups are numbered so that
// one XCD works on one head at a time).
//
// Mask semantics follow the reference's fp32 arithmetic exactly: on tiles that
// contain a masked (or out-of-range) key the logit is (q.k + inf*(mask-1)) +
// bias in that order on the vector ALU, so -1e9 absorbs small logits and a fully
// masked row averages v over all keys (which a launch on a range of rows finds out beforehand, see
// triattn_uniform_kernel); tiles whose keys are all unmasked take the matrix-pipe path above.
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "single_stage.h"

namespace ptx {

constexpr int kD = 32;          // head dim
constexpr int kKeyTile = 64;
constexpr float kLog2e = 1.4426950408889634f;
// half_row: code paths, and the largest per-lane probability sum of a half tile (16 values) the
// optimistic paths accept
enum { kOptimistic = 0, kClassic = 1, kMasked = 2, kOptimisticZero = 3 };
constexpr float kOptimisticLimit = 1.0e12f;
constexpr float kLn2 = 0.6931471805599453f;
// fast_tile: sums of a lane's first 16 probabilities against the reference 0 for which kClassic is sure to choose that reference
// as well: the largest logit lies within 14 of 0 if the sum is below e^14 and above 16 e^-14, with a margin for rounding.
constexpr float kNearZeroLow = 2.0e-5f, kNearZeroHigh = 1.0e6f;
// kClassic: a running maximum no larger than this (natural units, all lanes of the wave) is
// replaced by the reference 0, which makes exp2() of the raw logit the probability
constexpr float kZeroReferenceLimit = 14.0f;

// Addressing of q / gate / o and the optional outputs (see the kernel's header comment).
struct AttnAux {
  int64_t sh, si, sj;     // element strides of q, gate, o: head, row, query
  int n_rows;
  int mask_is_bias;
  float* lse;             // or null
  int64_t lh, li, lj;     // element strides of lse: head, row, query
  int row0, row_end;      // rows row0 .. row_end-1 are this launch's (a launch may cover a range)
  int n_keys;             // keys 0 .. n_keys-1 take part (n_keys <= n; the rest count as masked)
  float uniform_limit;    // > 0: triattn_uniform_kernel has looked at the launch's rows, with that limit
};

// Rows whose keys are all masked by the same -inf: (q.k - inf) + bias is -inf, whatever q.k and the bias are, as long as both
// are below half of the last place of inf, and then every key has the same weight and every query gets the mean of V.  This kernel finds
// out, in front of a masked launch on a range of rows (the padded ones), and leaves what it found where the output of
// those rows goes: in the first query's place of every block of 32 the mean (its first channel NaN where the row is not
// such a row: a key that is not masked, or |q| |k| too large), in the second's 0, or infinity if a |bias| of the block's
// queries is too large.  The masked kernel's workgroups look there first (uniform_rows) and either store the mean or do their work.
// Reads K, V and q of the rows once and the bias once, where the masked path reads the bias for every row: 64 padded rows of 2048
// keys, 4 heads: 27 + 19 us in place of 380; 32 of 384 5.8 + 5.1 in place of 16.8.
// Where the first key of a row is not masked nothing else of it is read, and where that of the last row is not (a launch on
// other rows than padded ones), neither is the bias: 192 valid rows of 384 45 -> 35 us, 384 of 768 230 -> 207.
__global__ __launch_bounds__(256) void triattn_uniform_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
                                                              const bf16_t* __restrict__ vt, const bf16_t* __restrict__ bias,
                                                              const bf16_t* __restrict__ mask, bf16_t* __restrict__ o, int n, int heads,
                                                              int key_pitch, int mask_transposed, int row0, int row_count, float limit) {
  typedef Vec8<bf16_t>::type V8;
  __shared__ float red[4][36];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = lane & 31, g = lane >> 5;
  const int key_tiles = key_pitch >> 6, q_blocks = (n + 31) >> 5;
  auto max_of_all = [&](float v) {   // (fmaxf passes over NaN: those are found one by one and count as infinite)
#pragma unroll
    for (int d = 32; d; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    return v;
  };
  if ((int)blockIdx.x >= row_count * heads) {   // the bias of 32 queries of a head
    const int item = (int)blockIdx.x - row_count * heads, h = item / q_blocks, qb = item - h * q_blocks;
    const bf16_t* const tiles = bias + ((int64_t)h * q_blocks + qb) * key_tiles * kAttnTileElems + lane * 8;
    const bool q_ok = 32 * qb + ln < n;
    const int i_last = row0 + row_count - 1;
    float most = to_f32(mask[mask_transposed ? (int64_t)i_last : (int64_t)i_last * n]) == 0.0f ? 0.0f : INFINITY;
    for (int t = wave; t * 64 < n && most < INFINITY; t += 4)
#pragma unroll
      for (int f = 0; f < 4; ++f) {   // fragment (u, c) = f: keys 32 g + 16 u + 8 c .. + 7
        const f32x8 b = to_f32(load8<bf16_t>(tiles + (int64_t)t * kAttnTileElems + f * 512));
        const int key = t * 64 + 32 * g + 16 * (f >> 1) + 8 * (f & 1);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (q_ok && key + e < n) most = fabsf(b[e]) < limit ? most : INFINITY;   // (a NaN is not)
      }
    most = max_of_all(most);
    if (lane == 0) red[wave][0] = most;
    __syncthreads();
    most = fmaxf(fmaxf(red[0][0], red[1][0]), fmaxf(red[2][0], red[3][0]));
    if (32 * qb + 1 < n)
      for (int r = threadIdx.x; r < row_count; r += 256)
        *reinterpret_cast<float*>(o + (((int64_t)h * n + row0 + r) * n + 32 * qb + 1) * kD) = most;
    return;
  }
  const int h = (int)blockIdx.x / row_count, i = row0 + (int)blockIdx.x - h * row_count;
  const bool valid = !(to_f32(mask[mask_transposed ? (int64_t)i : (int64_t)i * n]) == 0.0f);
  if (valid) {
    for (int qb = threadIdx.x; qb < q_blocks; qb += 256) o[(((int64_t)h * n + i) * n + 32 * qb) * kD] = (bf16_t)NAN;
    return;
  }
  float k2 = 0.0f, q2 = 0.0f, vsum = 0.0f;
  bool bad = false;
  const bf16_t* const kt = k + ((int64_t)h * n + i) * key_tiles * kAttnTileElems + lane * 8;
  const bf16_t* const vtt = vt + ((int64_t)h * n + i) * key_tiles * kAttnTileElems + lane * 8;
#pragma unroll 2
  for (int t = wave; t * 64 < n; t += 4) {
    V8 kf[4], vf[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      kf[f] = load8<bf16_t>(kt + (int64_t)t * kAttnTileElems + f * 512);
      vf[f] = load8<bf16_t>(vtt + (int64_t)t * kAttnTileElems + f * 512);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      // K fragments (u, 0 / 1): MFMA row ln, half of the key's channels each half-wave
      float s2 = 0.0f;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const f32x8 x = to_f32(kf[2 * u + kk]);
#pragma unroll
        for (int e = 0; e < 8; ++e) s2 += x[e] * x[e];
      }
      s2 += swap32(s2);
      if (t * 64 + 32 * ((ln >> 2) & 1) + 16 * u + 4 * (ln >> 3) + (ln & 3) < n) {
        bad |= !(s2 < INFINITY);
        k2 = fmaxf(k2, s2);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {   // V^T fragments (u, s): channel ln
        const f32x8 x = to_f32(vf[2 * u + s]);
        const int key = t * 64 + 32 * g + 16 * u + 8 * s;
#pragma unroll
        for (int e = 0; e < 8; ++e) vsum += key + e < n ? x[e] : 0.0f;
      }
    }
  }
  const bf16_t* const qrow = q + ((int64_t)h * n + i) * n * kD;
  constexpr int U = 8;   // loads under way
  for (int j0 = 0; j0 < n; j0 += 64 * U) {   // four lanes to a query; beyond n the last one again
    V8 x8[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x8[u] = load8<bf16_t>(qrow + (int64_t)min(j0 + 64 * u + (int)(threadIdx.x >> 2), n - 1) * kD + 8 * (threadIdx.x & 3));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const f32x8 x = to_f32(x8[u]);
      float s2 = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) s2 += x[e] * x[e];
      s2 += __shfl_xor(s2, 1, 64);
      s2 += __shfl_xor(s2, 2, 64);
      bad |= !(s2 < INFINITY);
      q2 = fmaxf(q2, s2);
    }
  }
  for (int j0 = threadIdx.x; j0 < n; j0 += 256 * U) {
    bf16_t m[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = min(j0 + 256 * u, n - 1);
      m[u] = mask_transposed ? mask[(int64_t)j * n + i] : mask[(int64_t)i * n + j];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) bad |= !(to_f32(m[u]) == 0.0f);
  }
  vsum += swap32(vsum);
  k2 = max_of_all(bad ? INFINITY : k2);
  q2 = max_of_all(q2);
  if (g == 0) red[wave][ln] = vsum;
  if (lane == 0) {
    red[wave][32] = k2;
    red[wave][33] = q2;
  }
  __syncthreads();
  k2 = fmaxf(fmaxf(red[0][32], red[1][32]), fmaxf(red[2][32], red[3][32]));
  q2 = fmaxf(fmaxf(red[0][33], red[1][33]), fmaxf(red[2][33], red[3][33]));
  const bool uniform = k2 * q2 < limit * limit;   // |q.k| <= |q| |k|
  const float inv = fast_rcp((float)n);
  V8 mean;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int c = 8 * (threadIdx.x & 3) + e;
    mean[e] = from_f32<bf16_t>(uniform || c ? (red[0][c] + red[1][c] + red[2][c] + red[3][c]) * inv : NAN);
  }
  for (int qb = threadIdx.x >> 2; qb < q_blocks; qb += 64)
    store8<bf16_t>(o + (((int64_t)h * n + i) * n + 32 * qb) * kD + 8 * (threadIdx.x & 3), mean);
}

// Rows of the pair tensor handled by one wave: R = 1 or 2, chosen per launch (triattn_fwd_ex).

// NWQ waves per workgroup (4 or 8), each with 32 queries: the workgroup's waves share the staged
// K / V^T tiles, so with 8 every wave moves one fragment per tile instead of two.
// n: queries = keys per row; ax.n_rows: rows (= n for a whole pair tensor, fewer for a chunk of
// rows).  q, gate and o are addressed through the element strides in `ax` (head, row, query; 32
// contiguous channels at each position); gate may be null (no gating).  mask: per (row, key),
// 0/1 values turned into inf*(mask-1), or with ax.mask_is_bias an additive bias used as it is.
// ax.lse: optional log2-sum-exp2 of the logits per (head, row, query).
// MK: kMaskGiven, or no mask (its own instantiations: a mask of all ones is passed as none by
// the host side).  Without a mask nothing of the masked path is left in the kernel; a last,
// partial key tile takes the same paths as the others with the logits of the keys beyond
// n_keys set to -inf (kMaskTail; kMaskNone where the keys fill whole tiles).
enum { kMaskNone = 0, kMaskTail = 1, kMaskGiven = 2 };
// TS: the launch's first `carried` workgroups run a stage of the single track on operands of that type (void: none; with one three waves
// per SIMD instead of four).
// STD: K and V as the operator's callers have them, [row][position][head][32] (addressed like q), and q not yet multiplied by
// log2 e: K rows find their fragments by the lanes' addresses, V tiles lie row-major in LDS and are turned when they
// are read.  (Repacked by kernels of their own, q, K and V cost 44 us at 384 rows of 384 positions and 4 heads, next to 86 of
// the core.)
template <typename T, int R, int NWQ, int MK, typename TS, bool STD = false>
__global__ __launch_bounds__((NWQ * 64), (sizeof(T) == 2 ? (!std::is_void<TS>::value ? 3 : R == 1 ? 16 / NWQ : 4) : 2)) void triattn_fwd_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ vt,
    const T* gate, const T* __restrict__ bias, const T* __restrict__ mask,
    T* o, int n, int heads, int key_pitch, int mask_transposed, float inf,
    int n_qtiles, int n_rowgroups, int64_t total_items, AttnAux ax, SingleStage carry, unsigned carried) {
  typedef typename Vec8<T>::type V8;
  typedef typename Vec4<T>::type V4;
  constexpr bool kCarries = !std::is_void<TS>::value;
  static_assert(!kCarries || (sizeof(T) == 2 && R == 1 && NWQ == kStageWaves), "the small launches");
  // two key tiles x R rows: iteration t reads tile t while tile t+1 is written
  __shared__ V8 lds_kv[kCarries ? 4 : 2][R][8][kWave];     // fragments 0-3: K (u,kk); 4-7: V^T (u,s)
  if constexpr (kCarries) {
    static_assert(!kCarries || sizeof(lds_kv) >= kStageLds, "the stage's LDS");
    if (blockIdx.x < carried) {
      single_stage<TS>(carry, blockIdx.x, reinterpret_cast<char*>(lds_kv));
      return;
    }
  }
  const unsigned block = blockIdx.x - carried;
  __shared__ __attribute__((aligned(16))) float lds_mb[2][R][kKeyTile];  // mask bias per key

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31, g = lane >> 5;

  // Work item -> (h, row group, query tile), h-major, one contiguous span per XCD
  // (workgroups are dealt round-robin to the 8 XCDs).
  const int64_t per_xcd = (total_items + 7) / 8;
  const int64_t item = (int64_t)(block & 7) * per_xcd + (block >> 3);
  if (item >= total_items) return;
  const int qt = (int)(item % n_qtiles);
  const int i0 = ax.row0 + (int)((item / n_qtiles) % n_rowgroups) * R;   // first of this workgroup's R rows
  const int h = (int)(item / ((int64_t)n_qtiles * n_rowgroups));

  if constexpr (MK == kMaskGiven && !STD && !kCarries && R == 1 && sizeof(T) == 2) {
    if (ax.uniform_limit > 0.0f) {   // (what triattn_uniform_kernel left; nobody else's output lies here)
      const int first = qt * NWQ * 32, blocks = min(NWQ, (n - first + 31) >> 5);
      T* const rows = o + h * ax.sh + i0 * ax.si + (int64_t)first * kD;
      const V8 mean = load8<T>(rows + 8 * (lane & 3));
      bool uniform = !(to_f32(rows[0]) != to_f32(rows[0]));
      for (int b = 0; b < blocks; ++b)
        uniform &= first + 32 * b + 1 < n && *reinterpret_cast<const float*>(rows + (32 * b + 1) * kD) < ax.uniform_limit;
      if (__builtin_amdgcn_readfirstlane(uniform)) {   // the same for all lanes of the workgroup
        __syncthreads();   // (every wave has read)
        for (int r = threadIdx.x >> 2; r < 32 * blocks && first + r < n; r += NWQ * 16) store8<T>(rows + r * kD + 8 * (lane & 3), mean);
        return;
      }
    }
  }
  const int q0 = (qt * NWQ + wave) * 32;   // first query of this wave
  const int key_tiles = key_pitch >> 6;
  const int q_blocks = (n + 31) >> 5;
  const int nk = ax.n_keys;
  const int n_tiles = (nk + kKeyTile - 1) / kKeyTile;
  constexpr bool has_mask = MK == kMaskGiven;
  // Operand tiles in fragment order (common.h): 2048 elements per key tile, this lane's
  // 8 elements of fragment f at f*512 + lane*8.  Rows beyond n re-read row n-1, a wave whose
  // queries all lie beyond n re-reads the last query block; nothing of either is stored.
  const T* b_tiles = bias + ((int64_t)h * q_blocks + min(q0 >> 5, q_blocks - 1)) * key_tiles * kAttnTileElems + lane * 8;
  const int qi = min(q0 + ln, n - 1);
  const int n_rows = ax.n_rows;
  // Lanes whose query lies beyond n compute on whatever the bias workspace holds there; they
  // store nothing, and they are kept out of the wave-wide decisions below so that the path a
  // wave takes (and with it the rounding of its valid queries) never depends on that content.
  const bool q_ok = q0 + ln < n;
  // (as a lane mask: wave-wide decisions are ballots of the condition alone, combined with this
  // mask on the scalar unit; a wave with none only helps to stage)
  uint64_t q_ok_mask = __builtin_amdgcn_ballot_w64(q_ok);

  // Q fragments (B operand): lane <-> query, slots <-> d = 16*kk + 8*g + t
  V8 qf[R][2];
  int64_t qrow[R];                       // head-major q / gate / o row of this lane's query
#pragma unroll
  for (int r = 0; r < R; ++r) {
    qrow[r] = h * ax.sh + min(i0 + r, ax.row_end - 1) * ax.si + qi * ax.sj;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      qf[r][kk] = load8<T>(q + qrow[r] + 16 * kk + 8 * g);
      if constexpr (STD) {
        f32x8 v = to_f32(qf[r][kk]);
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] *= kLog2e;
        qf[r][kk] = from_f32<T>(v);
      }
    }
  }

  // ---- cooperative tile loader: 8*R fragments per key tile, 8*R / NWQ per wave ----
  // 16-bit: direct-to-LDS loads (a fragment's LDS image is its global image: no registers, no LDS writes and, with
  // a scalar base, no vector arithmetic); fp32: through registers.  fetch() only issues loads; what looks at a loaded value
  // (mask -> additive bias, zeroing of V^T beyond n_keys) happens in stash(), one tile of work later.
  // Keys beyond n_keys hold garbage (or, below n, keys that are left out) in K, removed by the -inf mask bias, and
  // are zeroed in V^T (0 * garbage must stay 0).
  constexpr bool kDirect = sizeof(T) == 2;
  constexpr bool kFast = sizeof(T) == 2;
  static_assert(!has_mask || R == 1, "a mask is looked at for one row per workgroup");
  __shared__ int lds_vote[2][kFast ? NWQ : 1];
  constexpr int FPW = 8 * R / NWQ;   // fragments each wave moves per tile, of one operand and row
  static_assert(FPW >= 1 && FPW <= 4, "a wave's fragments are consecutive in memory");
  const int fid0 = wave * FPW, fr = fid0 >> 3, f0 = fid0 & 7;   // row, first fragment
  static_assert(!STD || kDirect, "standard layouts: 16-bit");
  const T* const kv_base = STD ? (f0 < 4 ? k : vt) + h * ax.sh + min(i0 + fr, ax.row_end - 1) * ax.si
                               : (f0 < 4 ? k : vt) + ((int64_t)h * n_rows + min(i0 + fr, ax.row_end - 1)) * key_tiles * kAttnTileElems + (f0 & 3) * 512;
  // STD: this lane's key within the tile and its channels, of the wave's fragment j
  auto std_place = [&](int j, int& key, int& d) {
    const int f = (f0 + j) & 3;
    if (f0 < 4) {   // K fragment (u, kk) = f: MFMA row lane % 32 (see the top), half-wave's channels
      const int m = lane & 31;
      key = 32 * ((m >> 2) & 1) + 16 * (f >> 1) + 4 * (m >> 3) + (m & 3);
      d = 16 * (f & 1) + 8 * g;
    } else {        // V: 16 rows of 64 bytes
      key = 16 * f + (lane >> 2);
      d = 8 * (lane & 3);
    }
  };
  V8 pre[kDirect ? 1 : FPW];
  T pre_mv;
  // mask value of key kc for this wave's row: m_base[kc * m_stride]
  const int m_row = min(i0 + min(wave, R - 1), ax.row_end - 1);
  const unsigned m_stride = mask_transposed ? n : 1;
  const T* m_base = has_mask ? mask + (mask_transposed ? (int64_t)m_row : (int64_t)m_row * n) : nullptr;
  auto fetch = [&](int tile) {
    const T* src = kv_base + (int64_t)tile * kAttnTileElems;
    if constexpr (STD) {
      const uint64_t base = uniform64((uint64_t)kv_base);
      const uint32_t dst = lds_address(&lds_kv[tile & 1][fr][f0][0]);
#pragma unroll
      for (int j = 0; j < FPW; ++j) {
        int key, d;
        std_place(j, key, d);   // (keys beyond n: the last one, left out below)
        load_to_lds16_s<0>(base, (uint32_t)(min(tile * kKeyTile + key, n - 1) * (int)ax.sj + d) * (uint32_t)sizeof(T), dst + j * 1024);
      }
    } else if constexpr (kDirect) {
      const uint64_t base = uniform64((uint64_t)src);
      const uint32_t dst = lds_address(&lds_kv[tile & 1][fr][f0][0]), off = lane * 16;
      load_to_lds16_s<0>(base, off, dst);
      if constexpr (FPW > 1) load_to_lds16_s<1024>(base, off, dst);
      if constexpr (FPW > 2) load_to_lds16_s<2048>(base, off, dst);
      if constexpr (FPW > 3) load_to_lds16_s<3072>(base, off, dst);
    } else {
#pragma unroll
      for (int j = 0; j < FPW; ++j) pre[j] = load8<T>(src + j * 512 + lane * 8);
    }
    // wave w < R publishes the mask bias of row i0 + w; all waves load (uniform load count)
    if constexpr (has_mask) {
      const int kc = min(tile * kKeyTile + lane, n - 1);
      pre_mv = m_base[__umul24(kc, m_stride)];   // both below 2^15
    }
  };
  // all loads, in a form that the compiler counts by (it knows nothing of the direct-to-LDS loads)
  auto landed = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
    asm volatile("" ::: "memory");
  };
  auto stash = [&](int tile) {
    const int buf = tile & 1;
    const int key0 = tile * kKeyTile;
    const bool tail = MK != kMaskNone && key0 + kKeyTile > nk;   // uniform (kMaskNone: whole tiles only)
    if constexpr (kDirect) landed();
    if (!kDirect || tail) {
#pragma unroll
      for (int j = 0; j < FPW; ++j) {
        V8 v;
        if constexpr (kDirect) v = lds_kv[buf][fr][f0 + j][lane];
        else v = pre[j];
        if (STD && tail && f0 >= 4) {
          int key, d;
          std_place(j, key, d);
#pragma unroll
          for (int t = 0; t < 8; ++t) v[t] = key0 + key < nk ? v[t] : (T)0.0f;
        } else if (tail && f0 >= 4) {
          // V^T fragment (u, s): slots <-> keys 32g + 16u + 8s + t
          const int f = f0 + j, koff = key0 + 32 * g + 16 * ((f >> 1) & 1) + 8 * (f & 1);
#pragma unroll
          for (int t = 0; t < 8; ++t) v[t] = koff + t < nk ? v[t] : (T)0.0f;
        }
        lds_kv[buf][fr][f0 + j][lane] = v;
      }
    }
    if constexpr (has_mask) {
      if (wave < R) {
        const float mb = ax.mask_is_bias ? to_f32(pre_mv) : inf * (to_f32(pre_mv) - 1.0f);
        lds_mb[buf][wave][lane] = key0 + lane < nk ? mb : 0.0f;   // (beyond n_keys: see TAIL)
      }
    }
  };

  // ---- per-wave bias tile: lane <-> query, [u][c] = keys key0 + 32g + 16u + 8c .. +7 ----
  auto fetch_bias_half = [&](int tile, int u, V8 (&dst)[2]) {
    const T* bp = b_tiles + (int64_t)min(tile, n_tiles - 1) * kAttnTileElems + u * 1024;
#pragma unroll
    for (int c = 0; c < 2; ++c) dst[c] = load8<T>(bp + c * 512);
  };
  auto fetch_bias = [&](int tile, V8 (&dst)[2][2]) {
#pragma unroll
    for (int u = 0; u < 2; ++u) fetch_bias_half(tile, u, dst[u]);
  };

  // V^T fragment (u, c) of row r: keys 32g + 16u + 8c .. + 7 of channel lane % 32
  auto v_frag = [&](int buf, int r, int u, int c) -> V8 {
    if constexpr (STD)
      return load8_turned(reinterpret_cast<const T*>(&lds_kv[buf][r][4][0]), 32, 32 * g + 16 * u + 8 * c, 16 * ((lane >> 4) & 1), lane);
    else
      return lds_kv[buf][r][4 + u * 2 + c][lane];
  };
  f32x16 acc_o[R];                // O^T per row
  float m_run[R], l_run[R];       // running max (natural units) and denominator (this lane's keys)
  auto reset = [&](float reference) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int e = 0; e < 16; ++e) acc_o[r][e] = 0.0f;
      m_run[r] = reference;
      l_run[r] = 0.0f;
    }
  };

  // One half of a key tile: logits, online softmax, P^T.  `tb` was fetched one tile ago.
  // Complete instantiations, so that the rarer paths share no code with - and cannot be
  // speculated into - the common one:
  //   kOptimistic  The softmax reference m_run only has to keep exp() in
  //                range, so it is NOT updated: probabilities are taken against the reference
  //                left by earlier tiles, no tile maximum is formed and O, l are not rescaled.
  //                If a probability sum leaves the safe range (a logit ~28 above the
  //                reference, or no reference yet), nothing has been committed and the half
  //                is redone by kClassic.  Returns false in that case (same in all lanes).
  //   kOptimisticZero  the common path: the same with the reference 0 in all lanes.  q and
  //                the triangle bias arrive multiplied by log2(e), so the matrix pipe's
  //                result IS the exponent: one v_exp_f32 per logit and no other arithmetic.
  //   kClassic     running maximum, rescale of O and l (first tile, or redo).  A maximum of
  //                modest size is replaced by the reference 0 (any reference is exact as long
  //                as exp() stays in range), which puts the row on the kOptimisticZero path.
  //   kMasked      tiles with a masked or out-of-range key: the reference's exact fp32
  //                order (q.k + mask_bias) + triangle_bias.
  // A path works on one 32-key half u of the staged tile (keys 32g + 16u + 0..15 of half-wave
  // g): 16 logit registers instead of 32, which lets four waves share a SIMD (a wave issues a
  // vector instruction only every ~9 cycles; it takes several to keep the vector unit busy).
  // What a path hands to the commit point of its half: P^T as the B operand of P.V, this
  // lane's probability sum, and the factor by which O and l shrink first (1 unless the
  // reference moved).
  struct HalfOut {
    V8 pf[2];
    float psum, alpha;
  };
  // P^T of a half from its exponentials, and their sum over this lane's keys.
  auto probabilities = [&](const f32x16& s, V8 (&pf)[2]) -> float {
    float psum = 0.0f;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      f32x8 p8;
#pragma unroll
      for (int t = 0; t < 8; ++t) p8[t] = s[8 * c + t];
      pf[c] = from_f32<T>(p8);
      if constexpr (sizeof(T) == 2) {
        bf16x2 ones;
        ones[0] = (__bf16)1.0f;
        ones[1] = (__bf16)1.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          bf16x2 pr;
          pr[0] = pf[c][2 * t];
          pr[1] = pf[c][2 * t + 1];
          psum = __builtin_amdgcn_fdot2_f32_bf16(pr, ones, psum, false);
        }
      } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) psum += p8[t];
      }
    }
    return psum;
  };
  // TAIL: the tile holds keys beyond n_keys; their logits, whatever was made of the K rows and
  // mask values found there, are replaced by -inf before the softmax (weight zero).  The other
  // keys of such a tile take the same path as in any other tile, so a mask of all ones gives
  // the bits that no mask gives.
  // `r`: which of the wave's R rows; `tbf`: the half's bias tile in fp32 (converted once per
  // half, for all R rows: they share the query block and with it the bias).
  auto half_row = [&](auto mode_tag, auto tail_tag, int r, int buf, int u, int key0, V8 (&tbh)[2],
                      const f32x16& tbf, HalfOut& out) -> bool {
    constexpr int MODE = decltype(mode_tag)::value;
    constexpr bool MASKED = MODE == kMasked;
    constexpr bool TAIL = decltype(tail_tag)::value;
    V8 kf[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) kf[kk] = lds_kv[buf][r][u * 2 + kk][lane];
    f32x16 s;
    if constexpr (!MASKED) {
      // S^T starts from the bias, the C operand of the first product: register e of this lane
      // <-> element e of its 16 stored values (16-bit: one conversion per logit, which with
      // four waves per SIMD costs less than adding the bias on the matrix pipe)
      s = tbf;
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = 0.0f;
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) mma32(s, kf[kk], qf[r][kk]);
    if constexpr (MASKED) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const f32x8 b = to_f32(tbh[c]);
        const f32x4 m0 = *reinterpret_cast<const f32x4*>(&lds_mb[buf][r][32 * g + 16 * u + 8 * c]);
        const f32x4 m1 = *reinterpret_cast<const f32x4*>(&lds_mb[buf][r][32 * g + 16 * u + 8 * c + 4]);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const float mbv = t < 4 ? m0[t & 3] : m1[t & 3];
          s[8 * c + t] = (s[8 * c + t] * kLn2 + mbv) + b[t] * kLn2;
        }
      }
    }
    if constexpr (TAIL) {
      const int kfirst = key0 + 32 * g + 16 * u;   // register e <-> key kfirst + e
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = kfirst + e < nk ? s[e] : -INFINITY;
    }
    float alpha = 1.0f;
    if constexpr (MODE == kClassic || MODE == kMasked) {
      float mx[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) mx[j] = fmaxf(s[2 * j], s[2 * j + 1]);
      float mt = fmaxf(fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3])),
                       fmaxf(fmaxf(mx[4], mx[5]), fmaxf(mx[6], mx[7])));
      mt = fmaxf(mt, swap32(mt));
      if (!MASKED) mt *= kLn2;
      // (a half whose keys all lie beyond n has mt = -inf: the reference stays where it is)
      float m_new = fmaxf(m_run[r], mt);
      if (!MASKED && (__builtin_amdgcn_ballot_w64(!(fabsf(m_new) < kZeroReferenceLimit)) & q_ok_mask) == 0ull) m_new = 0.0f;
      alpha = m_new == -INFINITY ? 1.0f : fast_exp2((m_run[r] - m_new) * kLog2e);
      m_run[r] = m_new;
    }
    if constexpr (MODE == kOptimisticZero) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = fast_exp2(s[e]);
    } else if constexpr (!MASKED) {
      // (as below: no key with a finite logit yet; one rounding, in every instantiation)
      const float mref = fmaxf(m_run[r], -2.0e38f);
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = fast_exp2(__builtin_fmaf(mref, -kLog2e, s[e]));
    } else {
      // (no key with a finite logit yet: -inf minus a finite stand-in is -inf, weight 0, where
      // -inf minus -inf would not be a number)
      const float mref = fmaxf(m_run[r], -3.0e38f);
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = fast_exp2((s[e] - mref) * kLog2e);
    }
    const float psum = probabilities(s, out.pf);
    if constexpr (MODE == kOptimistic || MODE == kOptimisticZero) {
      if ((__builtin_amdgcn_ballot_w64(!(psum < kOptimisticLimit)) & q_ok_mask) != 0ull) return false;
    }
    out.psum = psum;
    out.alpha = alpha;
    return true;
  };
  auto bias_of = [](const V8 (&raw)[2]) {
    const f32x8 b0 = to_f32(raw[0]), b1 = to_f32(raw[1]);
    return __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
  };
  auto process_tile = [&](auto tail_tag, int tile, V8 (&tb)[2][2]) {
    constexpr bool LAST_PARTIAL = decltype(tail_tag)::value;   // the one tile with keys beyond n_keys
    const int buf = tile & 1;
    const int key0 = tile * kKeyTile;
    // keys of the tile with a non-zero mask bias, per row, as a lane mask (key <-> lane); half
    // u's keys are the lanes with bit 4 == u
    uint64_t mb_mask[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      mb_mask[r] = 0ull;
      if constexpr (has_mask) mb_mask[r] = __builtin_amdgcn_ballot_w64(lds_mb[buf][r][lane] != 0.0f);
    }
    // keys of this tile that take part (uniform; 64 or more: all).  Half u holds the keys
    // 16u .. 16u+15 and 32+16u .. 32+16u+15 of the tile: complete from 48 + 16u keys on, empty
    // (and left out altogether) up to 16u.
    const int tile_keys = LAST_PARTIAL ? nk - key0 : kKeyTile;
    // A wave whose queries all lie beyond the launch's range only helps to stage the tiles (the
    // bias loads below stay unconditional: both paths then leave the same loads in flight).
    if (q_ok_mask != 0ull) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const bool tail_tile = LAST_PARTIAL && tile_keys < 48 + 16 * u;
      if (LAST_PARTIAL && tile_keys <= 16 * u) continue;
      const f32x16 tbf = bias_of(tb[u]);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        // the unmasked paths of one half: optimistic against the reference the earlier tiles
        // left, classic if there is none yet or the optimistic one had to give up
        auto unmasked_half = [&](auto ttag, HalfOut& out) -> bool {
          bool done = false;
          if (tile != 0 || u != 0) {
            if ((__builtin_amdgcn_ballot_w64(m_run[r] != 0.0f) & q_ok_mask) == 0ull)
              done = half_row(std::integral_constant<int, kOptimisticZero>{}, ttag, r, buf, u, key0, tb[u], tbf, out);
            else
              done = half_row(std::integral_constant<int, kOptimistic>{}, ttag, r, buf, u, key0, tb[u], tbf, out);
          }
          if (!done) half_row(std::integral_constant<int, kClassic>{}, ttag, r, buf, u, key0, tb[u], tbf, out);
          return !done;   // classic: O and l are rescaled first
        };
        HalfOut out;
        bool rescale = true;
        // this half's keys are those of lanes with bit 4 == u
        if (has_mask && (mb_mask[r] & (u ? 0xffff0000ffff0000ull : 0x0000ffff0000ffffull)) != 0ull) {
          if (tail_tile) half_row(std::integral_constant<int, kMasked>{}, std::true_type{}, r, buf, u, key0, tb[u], tbf, out);
          else half_row(std::integral_constant<int, kMasked>{}, std::false_type{}, r, buf, u, key0, tb[u], tbf, out);
        } else if (tail_tile) {
          rescale = unmasked_half(std::true_type{}, out);
        } else {
          rescale = unmasked_half(std::false_type{}, out);
        }
        if (rescale) {
#pragma unroll
          for (int e = 0; e < 16; ++e) acc_o[r][e] *= out.alpha;
          l_run[r] *= out.alpha;
        }
        l_run[r] += out.psum;
#pragma unroll
        for (int c = 0; c < 2; ++c) mma32(acc_o[r], v_frag(buf, r, u, c), out.pf[c]);
      }
    }
    }
  };
  // whether the sums of all this wave's rows and queries lie in a range (a NaN does not)
  auto all_between = [&](float low, float high) {
    uint64_t out = 0ull;
#pragma unroll
    for (int r = 0; r < R; ++r) out |= __builtin_amdgcn_ballot_w64(!(l_run[r] > low && l_run[r] < high));
    return (out & q_ok_mask) == 0ull;
  };
  // The common path (16-bit; tiles without a masked key): the reference is 0 in all lanes and stays it, and nothing looks at the sums on the way,
  // so that a tile is one stretch of instructions without a branch.  All rows' logits of a half are formed before the first
  // row's exponentials, which run under the second row's products, and the second's under the first's P.V.  The bias of the next tile is
  // requested as soon as this one's is converted: half a step of work or more lies between every load and its wait.  What a
  // row does is what half_row's kOptimisticZero does, bit for bit.
  // us per launch, 4 heads, with a check and a branch per row and half / this: n = 128 6.1 / 5.9, 256 22.4 / 22.1, 272 34.6 / 31.3, 384
  // 55.6 / 51.8, 387 74.6 / 68.0, 600 224 / 203, 768 381 / 358, 1024 859 / 803, 1280 1642 / 1551, 2048
  // 6558 / 6107.  What is left at 768 is 402 ns a tile and wave, where the tile's 8 MFMAs and 88 vector instructions alone take 265 ns
  // at four waves per SIMD (two pipes that overlap by half).  Tried and no better: two chains of dot2; s_setprio
  // around the logits' products; the next (half, row)'s logits ahead of this one's exponentials (14 spills: 768 353 -> 473).
  // `first_tag`: tile 0.  Returns false, after its first half, where that leaves a row a reference other than 0.
  auto fast_tile = [&](auto tail_tag, auto first_tag, int tile, V8 (&tb)[2][2]) -> bool {
    constexpr bool TAIL = decltype(tail_tag)::value, FIRST = decltype(first_tag)::value;
    const int buf = tile & 1;
    bool near_zero = true;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (TAIL && nk - tile * kKeyTile <= 16 * u) continue;   // (the half has no keys)
      if (FIRST && R == 2 && !near_zero) continue;   // (of one row, a small launch: a branch more than it saves)
      f32x16 tbf = bias_of(tb[u]);
      asm volatile("" : "+v"(tbf) :: "memory");   // (converted before its registers are loaded again)
      fetch_bias_half(tile + 1, u, tb[u]);
      asm volatile("" ::: "memory");
      V8 kf[R][2];
      f32x16 s[R];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) kf[r][kk] = lds_kv[buf][r][u * 2 + kk][lane];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        s[r] = tbf;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) mma32(s[r], kf[r][kk], qf[r][kk]);
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        V8 pf[2], vf[2];   // (V ahead of the exponentials)
#pragma unroll
        for (int c = 0; c < 2; ++c) vf[c] = v_frag(buf, r, u, c);
        if constexpr (TAIL) {
          const int kfirst = tile * kKeyTile + 32 * g + 16 * u;   // register e <-> key kfirst + e
#pragma unroll
          for (int e = 0; e < 16; ++e) s[r][e] = kfirst + e < nk ? s[r][e] : -INFINITY;
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) s[r][e] = fast_exp2(s[r][e]);
        l_run[r] += probabilities(s[r], pf);
#pragma unroll
        for (int c = 0; c < 2; ++c) mma32(acc_o[r], vf[c], pf[c]);
      }
      if constexpr (FIRST) {
        if (u == 0) near_zero = all_between(kNearZeroLow, kNearZeroHigh);
      }
    }
    return near_zero;
  };
  // Tile t+1 travels while tile t is processed; its bias tile is requested into the bias registers once tile t has
  // consumed them, behind the wait for tile t+1 (fast_tile: in mid-tile).
  V8 tbias[2][2];
  auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  auto start = [&] {
    fetch(0);
    fetch_bias(0, tbias);
    stash(0);
    barrier();
  };
  auto step = [&](auto tail_tag, int tile) {
    const bool more = tile + 1 < n_tiles;
    if constexpr (kDirect) landed();   // (the bias: ahead of loads that the compiler does not count)
    if (more) fetch(tile + 1);
    process_tile(tail_tag, tile, tbias);
    if (more) {
      stash(tile + 1);
      fetch_bias(tile + 1, tbias);
    }
    barrier();
  };
  auto fast_step = [&](auto tail_tag, auto first_tag, int tile) -> bool {
    const bool more = tile + 1 < n_tiles;
    if (more) fetch(tile + 1);
    const bool near_zero = q_ok_mask == 0ull || fast_tile(tail_tag, first_tag, tile, tbias);
    if (more) stash(tile + 1);
    landed();   // (the bias)
    return near_zero;
  };
  // the tiles whose keys all take part, in a loop that knows nothing of a partial tile (with
  // its tests in the loop every tile was 7 % slower), then the partial one if there is one
  const int n_full = MK == kMaskNone ? n_tiles : nk / kKeyTile;
  // What process_tile makes of a row is what counts: it depends on that row's 32 queries alone, and fast_tile does the same, bit for bit,
  // as long as the row keeps the reference 0.  A workgroup whose rows all take it in their first half tile walks by
  // fast_tile, up to a masked key, any other by process_tile from tile 0 on.  That no sum has reached the limit at which half_row
  // would have left the reference 0 is looked at where the fast walk ends; waves with such a sum start again by process_tile.
  // us per launch, 768 tokens, 4 heads, with the checks of process_tile throughout / so: logits with a deviation of 1.2 381 / 358; of 4
  // 412 / 431, 8 425 / 445, 12 442 / 457, 40 561 / 575 (tile 0 twice); a logit of 41 (the limit is some 27) that first appears in the
  // last tile, for every query 406 / 713 (everything twice), for one in each 128 397 / 543.  Tried: the checks in fast_tile, ahead of
  // each half's P.V: such logits 380, all others 4 % longer; a look in every fourth tile: all 1 % longer.
  int first = 0;   // tiles that are done
  reset(-INFINITY);
  start();
  if constexpr (kFast) {
    // whether it holds for one of the workgroup's waves; also the barrier of a step
    auto vote = [&](int which, bool v) {
      lds_vote[which][wave] = v;   // (the same from all lanes)
      barrier();
      int any = 0;
#pragma unroll
      for (int w = 0; w < NWQ; ++w) any |= lds_vote[which][w];
      return __builtin_amdgcn_readfirstlane(any) != 0;
    };
    // a key of the (staged) tile is masked: the same for all waves, whose row is the same
    auto masked = [&](int tile) { return has_mask && __builtin_amdgcn_ballot_w64(lds_mb[tile & 1][0][lane] != 0.0f) != 0ull; };
    const std::false_type no;
    const std::true_type yes;
    bool again = false;
    if (n_full > 0 && !masked(0)) {
      again = vote(0, !fast_step(no, yes, 0));
      first = 1;
      if (!again) {
        int tile = 1;
        for (; tile < n_full; ++tile) {
          if (masked(tile)) break;
          fast_step(no, no, tile);
          barrier();
        }
        first = has_mask ? tile : n_tiles;
        if constexpr (MK != kMaskNone) {
          if (n_full < n_tiles && (!has_mask || (tile == n_full && !masked(n_full)))) {
            fast_step(yes, no, n_full);
            first = n_tiles;
          }
        }
        const bool out = !all_between(0.0f, kOptimisticLimit);
        again = vote(1, out);
        if (again && !out && first == n_tiles) q_ok_mask = 0ull;   // (done: in the second walk it only helps to stage)
      }
    }
    if (again) {
      first = 0;
      if (q_ok_mask != 0ull) reset(-INFINITY);
      start();
    }
    if (first > 0 || (again && q_ok_mask == 0ull)) {
#pragma unroll
      for (int r = 0; r < R; ++r) m_run[r] = 0.0f;
    }
  }
  for (int tile = first; tile < n_full; ++tile) step(std::false_type{}, tile);
  if constexpr (MK != kMaskNone) {
    if (first < n_tiles && n_full < n_tiles) step(std::true_type{}, n_full);
  }

  // ---- normalise, gate, store: lane <-> query, register e <-> d = acc_row(e, g) ----
  // o may alias gate: every gate load is issued before the first store.
  // (the row offsets are formed again from a laundered query index: kept across the key loop
  // they cost two registers of a budget that has none to spare)
  int qi_again = qi;
  asm volatile("" : "+v"(qi_again));
#pragma unroll
  for (int r = 0; r < R; ++r) qrow[r] = h * ax.sh + min(i0 + r, ax.row_end - 1) * ax.si + qi_again * ax.sj;
  f32x4 gv[R][4];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      gv[r][c] = f32x4{1.0f, 1.0f, 1.0f, 1.0f};
      if (gate) gv[r][c] = to_f32(*reinterpret_cast<const V4*>(gate + qrow[r] + 4 * g + 8 * c));
    }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float l_tot = l_run[r] + swap32(l_run[r]);
    const float inv = fast_rcp(l_tot);
    if (ax.lse && g == 0 && q0 + ln < n && i0 + r < ax.row_end)
      ax.lse[h * ax.lh + (int64_t)(i0 + r) * ax.li + (int64_t)qi_again * ax.lj] =
          m_run[r] * kLog2e + __builtin_amdgcn_logf(l_tot);   // v_log_f32 is log2
    if (q0 + ln < n && i0 + r < ax.row_end) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        f32x4 ov;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          // attention output rounded to T before the gate multiply, as the reference does
          ov[t] = to_f32(from_f32<T>(acc_o[r][4 * c + t] * inv)) * gv[r][c][t];
        }
        *reinterpret_cast<V4*>(o + qrow[r] + 4 * g + 8 * c) = from_f32<T>(ov);
      }
    }
  }
}

constexpr int kTwoRowsFrom = 272;   // (see triattn_fwd_ex)

// workgroups of four waves that take one row each
static int64_t one_row_groups(int n_rows, int n, int heads) { return (int64_t)heads * n_rows * ((n + 127) / 128); }

// Where the core reads standard layouts: with one row per wave (with two, the lanes' addresses take registers that it does not
// have).  Two rows per wave on repacked operands gain less than the repacking costs.  us, the operator's forward without Bias1, 4 heads,
// S rows of S positions, repacked / as they are: 352 92 / 65, 384 101 / 73, 512 198 / 144, 640 334 / 298, 768 516 / 474, 1024 1089 / 1072, 1536
// 3268 / 3273; 64 rows of 384 32 / 19, of 768 58 / 48.  Beyond,
// where the rows are few one is taken per wave either way: 2 rows of 1536 68 / 42, 8 of 2048 (512 workgroups of four waves) 92 / 72, 4 of 4096
// (512) 264 / 255, 7 of 4096 (896) 270 / 304: there repacked operands go to workgroups of eight.
bool triattn_fwd_standard(int n_rows, int n, int heads, bool masked) {
  return masked || n < 1536 || one_row_groups(n_rows, n, heads) <= 512;
}

// (one row and four waves at those sizes, and workgroups to spare)
bool triattn_fwd_carries(int n, bool bits16) { return bits16 && n <= 256; }

template <typename T>
int triattn_fwd(const T* q, const T* k, const T* vt, const T* g, const T* tri_bias, const T* mask,
                T* o, int n, int heads, int key_pitch, int mask_transposed, float inf,
                int row_begin, int row_count, int n_keys, const SingleStage* carry, hipStream_t stream) {
  // head-major q, gate, o of a whole pair tensor: [heads][n][n][32]
  AttnAux ax = {};
  ax.sh = (int64_t)n * n * kD;
  ax.si = (int64_t)n * kD;
  ax.sj = kD;
  ax.n_rows = n;
  return triattn_fwd_ex<T>(q, k, vt, g, tri_bias, mask, o, n, n, heads, key_pitch, mask_transposed, inf,
                           0, ax.sh, ax.si, ax.sj, nullptr, 0, 0, 0, row_begin, row_count, n_keys, carry, stream);
}

template <typename T>
int triattn_fwd_ex(const T* q, const T* k, const T* vt, const T* g, const T* tri_bias,
                   const T* mask, T* o, int n_rows, int n, int heads, int key_pitch,
                   int mask_transposed, float inf, int mask_is_bias, int64_t sh, int64_t si,
                   int64_t sj, float* lse, int64_t lh, int64_t li, int64_t lj, int row_begin,
                   int row_count, int n_keys, const SingleStage* carry, hipStream_t stream, bool standard) {
  const bool empty = n == 0 || n_rows == 0 || row_count == 0 || heads == 0;
  if (carry && (empty || !triattn_fwd_carries(n, sizeof(T) == 2))) {
    single_stage_run(carry, stream);
    carry = nullptr;
  }
  if (empty) return 0;
  AttnAux ax = {sh, si, sj, n_rows, mask_is_bias, lse, lh, li, lj, row_begin, row_begin + row_count, n_keys, 0.0f};
  // A masked launch on the last rows: those are the padded rows of a batch, as a rule.  (Not where o holds the gate, and in
  // the layout of the pair tensor's attention only.)  Up to 256 tokens a second launch costs more than it saves.  us for n / 8 padded rows,
  // 4 heads, masked path / with it: n = 128 5.4 / 7.8, 200 7.7 / 8.1, 256 8.2 / 8.4, 288 12.0 / 8.7, 320 11.7 / 8.9, 352 17.4 / 9.0; half of the rows,
  // none of them padded: 256 12.6 / 15.9, 288 24.6 / 26.0, 352 33.8 / 34.8, 512 67.9 / 67.2.
  if constexpr (sizeof(T) == 2) {
    if (mask && n > 256 && row_begin > 0 && row_begin + row_count == n && !mask_is_bias && !g && !lse && n_rows == n && n_keys == n && inf > 0.0f && inf < 1.0e30f && sj == kD &&
        si == (int64_t)n * kD && sh == n * si) {
      // half of inf's last place is at least inf * 2^-25; q and the bias are in units of ln 2
      ax.uniform_limit = 0.99f * 0x1p-25f * inf * kLog2e;
      triattn_uniform_kernel<<<dim3((unsigned)(row_count * heads + heads * ((n + 31) >> 5))), dim3(256), 0, stream>>>(
          q, k, vt, tri_bias, mask, o, n, heads, key_pitch, mask_transposed, row_begin, row_count, ax.uniform_limit);
    }
  }
  // Two rows per wave (16-bit, no mask): the two rows share the query block and with it the bias tile - one load
  // and one conversion per logit for both, half the bias stream from the L2 - at 128 registers, so that four waves
  // still share a SIMD (a mask belongs to a row: one row per workgroup, 120 registers).  Below 272 tokens the pairs of rows leave too few
  // workgroups.  us per launch, 4 heads, one row / two rows (four waves each): n = 200 17.2 / 17.5, 256 20.9 / 21.1, 288 34.1 / 33.2, 300 36.7 /
  // 35.0, 320 35.8 / 34.1, 336 44.6 / 40.6, 350 50.7 / 46.4.
  // Nor do they pay where one row per wave takes a single round of the machine, 1024 workgroups of four waves (a range of few rows): 272
  // tokens, 64 rows (768 workgroups) 9.9 / 11.6, 85 (1020) 11.7 / 14.3, 100 15.2 / 14.7; 768, 2 rows 10.3 / 13.9, 32 18.4 / 21.2, 43 (1032)
  // 32.2 / 28.5; 1024, 32 rows (1024) 29.7 / 29.0; 2048, 8 rows 31.9 / 46.3.
  const bool two_rows = sizeof(T) == 2 && !mask && n >= kTwoRowsFrom && one_row_groups(row_count, n, heads) >= 1024 && !standard;
  // Eight waves share the staged K / V tiles of long rows.  Two rows: where that leaves no more waves without queries than four do (they
  // skip the arithmetic and only help to stage the tiles) and the keys fill whole tiles (with a partial one its registers
  // spill): four / eight 768 338 / 346, 1024 755 / 765, 1100 1001 / 1080, 1200 1346 / 1441, 1280 1475 / 1467, 1536 2509 / 2459, 2048
  // 5909 / 5775.  One row: +2 % at n = 768, even at 1024, -2.6 % at 1536.
  const bool wide = sizeof(T) == 2 && (mask || !standard) && (two_rows ? n > 1056 && (n + 127) / 128 % 2 == 0 && n_keys % kKeyTile == 0
                                                : (n % 256 == 0 && n >= 1536) || n >= 2048);
  const int mk = mask ? kMaskGiven : n_keys % kKeyTile ? kMaskTail : kMaskNone;
  const int n_qtiles = wide ? (n + 255) / 256 : (n + 127) / 128;
  const int R = two_rows ? 2 : 1;
  const int n_rowgroups = (row_count + R - 1) / R;
  const int64_t total = (int64_t)heads * n_rowgroups * n_qtiles;
  const int64_t per_xcd = (total + 7) / 8;
#define PTX_ATTN_LAUNCH_T(RR, NWQ, MK, ...)                                                                  \
  triattn_fwd_kernel<T, RR, NWQ, MK, __VA_ARGS__><<<dim3(carried + (unsigned)(per_xcd * 8)), dim3(NWQ * 64), 0, stream>>>( \
      q, k, vt, g, tri_bias, mask, o, n, heads, key_pitch, mask_transposed, inf, n_qtiles,                   \
      n_rowgroups, total, ax, carried ? *carry : SingleStage{}, carried)
#define PTX_ATTN_LAUNCH_R(RR, NWQ, MK) PTX_ATTN_LAUNCH_T(RR, NWQ, MK, void)
  const unsigned carried = single_stage_groups(carry);
  if constexpr (sizeof(T) == 2) {
    if (carried) {
#define PTX_ATTN_LAUNCH_C(TS)                                              \
  do {                                                                     \
    if (mk == kMaskGiven) PTX_ATTN_LAUNCH_T(1, 4, kMaskGiven, TS);         \
    else if (mk == kMaskTail) PTX_ATTN_LAUNCH_T(1, 4, kMaskTail, TS);      \
    else PTX_ATTN_LAUNCH_T(1, 4, kMaskNone, TS);                           \
  } while (0)
      if (carry->bits16) PTX_ATTN_LAUNCH_C(bf16_t);
      else PTX_ATTN_LAUNCH_C(float);
#undef PTX_ATTN_LAUNCH_C
      return 0;
    }
  }
  if constexpr (sizeof(T) == 2) {
    if (standard) {
      // (without a mask four waves: beyond 1535 positions triattn_fwd_standard() leaves few rows only)
      if (mk == kMaskGiven && wide) PTX_ATTN_LAUNCH_T(1, 8, kMaskGiven, void, true);
      else if (mk == kMaskGiven) PTX_ATTN_LAUNCH_T(1, 4, kMaskGiven, void, true);
      else if (mk == kMaskTail) PTX_ATTN_LAUNCH_T(1, 4, kMaskTail, void, true);
      else PTX_ATTN_LAUNCH_T(1, 4, kMaskNone, void, true);
      return 0;
    }
  }
#define PTX_ATTN_LAUNCH(RR, MK)                \
  do {                                         \
    if (wide) PTX_ATTN_LAUNCH_R(RR, 8, MK);    \
    else PTX_ATTN_LAUNCH_R(RR, 4, MK);         \
  } while (0)
  if (two_rows) {
    if constexpr (sizeof(T) == 2) {
      if (mk == kMaskTail) PTX_ATTN_LAUNCH_R(2, 4, kMaskTail);
      else PTX_ATTN_LAUNCH(2, kMaskNone);
    }
  } else if (mk == kMaskGiven) {
    PTX_ATTN_LAUNCH(1, kMaskGiven);
  } else if (mk == kMaskTail) {
    PTX_ATTN_LAUNCH(1, kMaskTail);
  } else {
    PTX_ATTN_LAUNCH(1, kMaskNone);
  }
#undef PTX_ATTN_LAUNCH
#undef PTX_ATTN_LAUNCH_R
#undef PTX_ATTN_LAUNCH_T
  return 0;
}

#define PTX_INSTANTIATE_EX(T)                                                                     \
  template int triattn_fwd_ex<T>(const T*, const T*, const T*, const T*, const T*, const T*, T*,  \
                                 int, int, int, int, int, float, int, int64_t, int64_t, int64_t,  \
                                 float*, int64_t, int64_t, int64_t, int, int, int, const SingleStage*, hipStream_t, bool);
PTX_INSTANTIATE_EX(float)
PTX_INSTANTIATE_EX(bf16_t)
#undef PTX_INSTANTIATE_EX
template int triattn_fwd<float>(const float*, const float*, const float*, const float*,
                                const float*, const float*, float*, int, int, int, int, float,
                                int, int, int, const SingleStage*, hipStream_t);
template int triattn_fwd<bf16_t>(const bf16_t*, const bf16_t*, const bf16_t*, const bf16_t*,
                                 const bf16_t*, const bf16_t*, bf16_t*, int, int, int, int, float,
                                 int, int, int, const SingleStage*, hipStream_t);

}  // namespace ptx
