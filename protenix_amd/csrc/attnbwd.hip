// Backward of the fused attention operator on standard-layout tensors
// (the contract of tri_attention/op.py:79-163 and tri_attention/backward.py:27-609 of the
// reference): given Q (already scaled), K, V, O, dO [rows][S][H][32], Bias1 [rows][S],
// Bias2 [H][S][S] and the forward's M = log2 sum_k 2^(logit * log2 e) [rows][S][H], with
//   P = 2^(S log2 e - M),  S = Q K^T + Bias1 + Bias2,  Delta = rowsum(O * dO),
//   dS = P * (dO V^T - Delta)
// it produces  dV = P^T dO,  dK = dS^T Q,  dQ = dS K,  dBias2[h] = sum over rows of dS.
// Two kernels where a workgroup takes a whole row (rows_at_once) - dQ, dK and dV, and dBias2 -, else three: dQ, dK / dV, dBias2.
// The first forms Delta (the reference's preprocess kernel) and leaves it for the others; P is recomputed, the
// logits are never stored.  One wave owns a 32 x 32 block of (query, key) pairs and walks over
// the other index; every product runs on MFMA with fp32 accumulation (conventions of
// common.h).  The register <-> index permutation of single.hip makes the recomputed P and dS
// usable as MFMA operands as they sit in the accumulators.
// What bounds these kernels is the operand stream out of L2 (6 to 8 KB per block pair when
// every wave fetches its own) and the cache lines each load touches, so the four waves of a
// workgroup take neighbouring blocks and share the tiles that walk: the workgroup loads each
// tile once, one step ahead, into registers, parks it in LDS row-major, and every wave reads
// its MFMA fragments from there - also those a product needs with the walking index in the K
// slots (K^T for dQ, Q^T and dO^T for dK / dV), which 16-bit tiles give through the
// transposing LDS load and fp32 tiles through a transposed copy.
#include <algorithm>
#include <type_traits>
#include "common.h"
#include "kernels.h"
#include "rowtile.h"

namespace ptx {

namespace {

constexpr float kBwdLog2e = 1.4426950408889634f;
constexpr int kTP = 40;   // pitch of the LDS tiles (elements): 16-byte aligned rows, spread over banks

struct BwdParams {
  const void *q, *k, *v, *o, *dout, *b1, *b2;
  const float* lse;
  float* delta;
  void *dq, *dk, *dv, *db2;
  int n_rows, s, heads;
  float* parts;     // dBias2's partial sums [slice][H][S][S], or null: one slice, written as it is
  int slices;
};

// Work item of this workgroup in a grid of `items` rounded up to a multiple of 8: one contiguous span per XCD
// (workgroups are dealt round-robin to the 8 XCDs), so that the heads and blocks of a row, which read the same
// cache lines, share an L2.
__device__ __forceinline__ uint32_t xcd_item(uint32_t items) {
  return (blockIdx.x & 7) * ((items + 7) / 8) + (blockIdx.x >> 3);
}

__device__ __forceinline__ int perm_row(int m) {   // MFMA row m of a 32-block <-> index in the block
  return 16 * (m >> 4) + 8 * ((m >> 2) & 1) + 4 * ((m >> 3) & 1) + (m & 3);
}
__device__ __forceinline__ int64_t elem(const BwdParams& p, int i, int pos, int h) {
  return (((int64_t)i * p.s + pos) * p.heads + h) * 32;
}
// index (within a 32-block) that accumulator register r of half-wave g stands for
__device__ __forceinline__ int reg_index(int r, int g) { return 16 * (r >> 3) + 8 * g + (r & 7); }

template <typename T> __device__ __forceinline__ typename Vec8<T>::type zero_frag() {
  typename Vec8<T>::type z;
#pragma unroll
  for (int t = 0; t < 8; ++t) z[t] = (T)0.0f;
  return z;
}

// 8 consecutive bias values starting at key block `kb` (a multiple of 8) of a row of `s` keys.
// vec (s % 8 == 0): a block of 8 keys is inside the row or outside as a whole, and an outside block is
// read from the row's last one (the caller masks it).  Otherwise rows start at any element: a whole block is one load
// of the element type's alignment (the hardware's vector loads take any; eight loads of one element
// took dQ 595 us and dK/dV 551 at 500 tokens, 4 heads, bf16, now 323 and 395), the row's last, partial block one load per element.
template <typename T>
__device__ __forceinline__ typename Vec8<T>::type load_bias8_raw(const T* row, int kb, int s,
                                                                bool vec) {
  if (vec) return load8<T>(row + min(kb, s - 8));
  typename Vec8<T>::type v;
  if (kb + 8 <= s) {
    __builtin_memcpy(&v, row + kb, sizeof(v));
  } else {
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = row[min(kb + t, s - 1)];
  }
  return v;
}
template <typename T>
__device__ __forceinline__ f32x8 load_bias8(const T* row, int kb, int s, bool vec) {
  return to_f32(load_bias8_raw<T>(row, kb, s, vec));
}

}  // namespace

// 16-bit kernels double-buffer their shared tiles (one barrier a step) and are held to the
// registers of three waves per SIMD; fp32 tiles are twice as
// large and stay single-buffered (two barriers a step).
template <typename T, bool VEC> struct BwdCfg {
  static constexpr int kBuffers = sizeof(T) == 2 ? 2 : 1;
  // (the second argument of __launch_bounds__: waves per SIMD the register budget allows for)
  static constexpr int kMinWaves = sizeof(T) == 2 ? 3 : 1;
};

// 16-bit tiles are parked in LDS row-major only; an operand that a product needs with the
// tile's rows in the K slots is read with the transposing LDS load of gfx950 (load8_turned in
// common.h).  fp32 has no such load and keeps transposed copies of its tiles.
template <typename T> struct Turned {
  static constexpr bool value = sizeof(T) == 2;
};
__device__ __forceinline__ f32x8 load8_turned(const float*, int, int, int, int) { return f32x8{}; }   // (never called)

// -inf as the lowest finite value, so that a product with 0 is 0 (a NaN's row is NaN throughout by its log-sum-exp).
__device__ __forceinline__ Vec8<bf16_t>::type finite_low(Vec8<bf16_t>::type x) {
  typedef uint16_t U8 __attribute__((ext_vector_type(8)));
  return __builtin_bit_cast(Vec8<bf16_t>::type, __builtin_elementwise_min(__builtin_bit_cast(U8, x), (U8)0xff7f));
}

// The workgroup's 256 threads load two [32 rows][32 channels] tiles (rows `pos0 ..` of tensors
// a and b at (row i, head h)): thread t takes 8 channels of one row of one tile.
template <typename T> struct TilePiece {
  typename Vec8<T>::type v;
  __device__ __forceinline__ void fetch(const BwdParams& p, const void* a, const void* b, int i,
                                        int pos0, int h, int tid) {
    const int row = min(pos0 + ((tid & 127) >> 2), p.s - 1);
    v = load8<T>((const T*)(tid >> 7 ? b : a) + elem(p, i, row, h) + 8 * (tid & 3));
  }
  // row-major into rm[tid >> 7]; the first n_tr tiles also transposed ([channel][row]) into
  // tr + (tid >> 7) * 32 * kTP
  __device__ __forceinline__ void park(T (*rm)[32 * kTP], T* tr, int n_tr, int tid) const {
    const int which = tid >> 7, row = (tid & 127) >> 2, c0 = 8 * (tid & 3);
    store8<T>(&rm[which][row * kTP + c0], v);
    if (which < n_tr) {
#pragma unroll
      for (int t = 0; t < 8; ++t) tr[which * 32 * kTP + (c0 + t) * kTP + row] = v[t];
    }
  }
};

// dQ: a workgroup takes 128 queries of one (row, head), a wave 32 of them, and walks over the
// key blocks; K, V and K^T are shared.  Works on S^T: lane <-> query, register <-> key, so the
// biases arrive as 8 consecutive keys per load and the row statistics are per-lane scalars.
// The biases are the initial value of the S^T accumulator and -Delta that of dP^T, so that a
// logit costs one multiply-add, one exponential and one multiply.  Lanes whose query lies
// beyond s repeat query s - 1 and store nothing; keys beyond s exist in the last block only,
// which has its own copy of the step.  The shared tiles are double-buffered: one barrier a step.
template <typename T, bool VEC>
__global__ __launch_bounds__(256, (BwdCfg<T, VEC>::kMinWaves)) void attn_bwd_dq_kernel(BwdParams p) {
  typedef typename Vec8<T>::type V8;
  typedef typename Vec4<T>::type V4;
  constexpr int NB = BwdCfg<T, VEC>::kBuffers;
  __shared__ __attribute__((aligned(32))) T rm[NB][2][32 * kTP];   // K, V
  constexpr bool TURN = Turned<T>::value;
  __shared__ __attribute__((aligned(32))) T tr[TURN ? 8 : NB * 32 * kTP];   // K^T (fp32 only)
  __shared__ __attribute__((aligned(32))) T b2s[NB][128 * kTP];    // Bias2 of the 128 queries x 32 keys
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, ln = lane & 31, g = lane >> 5;
  const int s = p.s, H = p.heads;
  constexpr bool vec = VEC;   // rows of s keys are 8-aligned
  const uint32_t n_wg = ((uint32_t)s + 127) / 128, items = n_wg * (uint32_t)H * (uint32_t)p.n_rows, item = xcd_item(items);
  if (item >= items) return;
  const int wg = item % n_wg, h = item / n_wg % H, i = item / n_wg / H;
  const int q0 = (wg * 4 + wave) * 32;
  const int qi = min(q0 + ln, s - 1);
  const bool q_ok = q0 + ln < s;
  // (without a Bias1 the loads go to a row of Bias2 and count for nothing: a load under a
  // branch would make every wait for memory a wait for all of it)
  const T* b1row = p.b1 ? (const T*)p.b1 + (int64_t)i * s : (const T*)p.b2 + (int64_t)h * s * s;
  const float b1on = p.b1 ? 1.0f : 0.0f;
  // 16-bit: the biases reach the S^T accumulator on the matrix pipe, which these kernels leave
  // idle four fifths of the time, instead of being converted and added on the vector ALU:
  //   Bias2  S^T += E * B2, B2 the block's [key][query] values as they lie in LDS for this
  //          lane's query (B operand: slots <-> keys), E the 0/1 matrix that sends key j to
  //          the accumulator row that stands for it (row m <-> key perm_row(m)), -inf as the lowest finite value;
  //   Bias1  S^T += b * 1^T: Bias1 of the row's key in K slot 0 of one more product, against
  //          a B operand with 1 in that slot (0 without a Bias1).  Products with 1 are exact.
  constexpr bool MMB = sizeof(T) == 2;
  V8 e_frag[2], one_frag;
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int t = 0; t < 8; ++t) e_frag[kk][t] = (T)(perm_row(ln) == 16 * kk + 8 * g + t ? 1.0f : 0.0f);
#pragma unroll
  for (int t = 0; t < 8; ++t) one_frag[t] = (T)(t == 0 && g == 0 ? b1on : 0.0f);

  V8 qf[2], dof[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    qf[kk] = load8<T>((const T*)p.q + elem(p, i, qi, h) + 16 * kk + 8 * g);
    dof[kk] = load8<T>((const T*)p.dout + elem(p, i, qi, h) + 16 * kk + 8 * g);
  }
  const float neg_mq = -p.lse[((int64_t)i * s + qi) * H + h];
  // Delta = sum_d O * dO of this lane's query, formed here (the lane holds half of the query's
  // channels, the other half-wave the rest) and left in p.delta for the two kernels that follow
  float delta = 0.0f;
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const f32x8 of = to_f32(load8<T>((const T*)p.o + elem(p, i, qi, h) + 16 * kk + 8 * g));
    const f32x8 df = to_f32(dof[kk]);
#pragma unroll
    for (int t = 0; t < 8; ++t) delta += of[t] * df[t];
  }
  delta += swap32(delta);
  if (g == 0 && q_ok) p.delta[((int64_t)i * s + qi) * H + h] = delta;
  const float neg_dq = -delta;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;

  // Bias2 comes in through LDS like the tiles: four neighbouring lanes read the 64 bytes a
  // query's row has for the block (a lane reading 16 bytes of its own query's row touches as
  // many cache lines per load as it has lanes, and the texture path was busy 96 % of the time).
  TilePiece<T> piece;
  V8 b1n[2], b2n[2];
  T b1m = (T)0.0f;   // (16-bit) Bias1 of key perm_row(ln) of the block
  const int b2col = 8 * (tid & 3);
  const T* b2rows[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
    b2rows[j] = (const T*)p.b2 + ((int64_t)h * s + min(wg * 128 + 64 * j + (tid >> 2), s - 1)) * s;
  // (the compiler barriers keep the loads where they are written, a step ahead of their use:
  // left alone, the compiler moves them down to the use and waits there)
  auto fetch = [&](int key0) {
    piece.fetch(p, p.k, p.v, i, key0, h, tid);
#pragma unroll
    for (int j = 0; j < 2; ++j) b2n[j] = load_bias8_raw<T>(b2rows[j], key0 + b2col, s, vec);
    asm volatile("" ::: "memory");
  };
  auto park = [&](int buf) {
    piece.park(rm[buf], tr + (TURN ? 0 : buf * 32 * kTP), TURN ? 0 : 1, tid);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (MMB) b2n[j] = finite_low(b2n[j]);
      store8<T>(&b2s[buf][(64 * j + (tid >> 2)) * kTP + b2col], b2n[j]);
    }
  };
  auto fetch_bias = [&](int key0) {
    if (MMB) {
      b1m = b1row[min(key0 + perm_row(ln), s - 1)];
    } else {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) b1n[ks] = load_bias8_raw<T>(b1row, key0 + 16 * ks + 8 * g, s, vec);
    }
    asm volatile("" ::: "memory");
  };
  // one block of 32 keys out of buffer `buf`; TAIL: the block holds keys beyond s.  The biases
  // of the next block are requested as soon as this block's sit in the accumulator.
  auto step = [&](auto tail_tag, int buf, int key0, int next_key0) {
    constexpr bool TAIL = decltype(tail_tag)::value;
    V8 kf[2], vf[2], ktf[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      kf[kk] = load8<T>(&rm[buf][0][perm_row(ln) * kTP + 16 * kk + 8 * g]);
      vf[kk] = load8<T>(&rm[buf][1][perm_row(ln) * kTP + 16 * kk + 8 * g]);
      ktf[kk] = TURN ? load8_turned(rm[buf][0], kTP, 16 * kk + 8 * g, 16 * ((lane >> 4) & 1), lane)
                     : load8<T>(&tr[TURN ? 0 : buf * 32 * kTP + ln * kTP + 16 * kk + 8 * g]);
    }
    f32x16 st, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) dp[r] = neg_dq;
    if constexpr (MMB) {
      V8 b1a;
#pragma unroll
      for (int t = 0; t < 8; ++t) b1a[t] = (T)0.0f;
      b1a[0] = (g == 0 && b1on != 0.0f) ? b1m : (T)0.0f;
      V8 b2v[2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) b2v[ks] = load8<T>(&b2s[buf][(32 * wave + ln) * kTP + 16 * ks + 8 * g]);
      fetch_bias(next_key0);
#pragma unroll
      for (int r = 0; r < 16; ++r) st[r] = 0.0f;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) mma32(st, kf[kk], qf[kk]);      // S^T[key][query]
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) mma32(st, e_frag[kk], b2v[kk]);  // + Bias2
      mma32(st, b1a, one_frag);                                        // + Bias1
    } else {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const f32x8 b1f = to_f32(b1n[ks]);
        const f32x8 b2f = to_f32(load8<T>(&b2s[buf][(32 * wave + ln) * kTP + 16 * ks + 8 * g]));
#pragma unroll
        for (int t = 0; t < 8; ++t) st[8 * ks + t] = (b1on != 0.0f ? b1f[t] : 0.0f) + b2f[t];   // (not b1f * b1on: -inf)
      }
      fetch_bias(next_key0);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) mma32(st, kf[kk], qf[kk]);    // S^T[key][query] (+ biases)
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) mma32(dp, vf[kk], dof[kk]);   // dP^T[key][query] - Delta
    V8 dsf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      f32x8 ds;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int r = 8 * ks + t;
        float pr = fast_exp2(st[r] * kBwdLog2e + neg_mq);
        if (TAIL) pr = key0 + reg_index(r, g) < s ? pr : 0.0f;
        ds[t] = pr * dp[r];
      }
      dsf[ks] = from_f32<T>(ds);
    }
    // dQ^T[d][query] += K^T[d][key] dS^T[key][query]: lane <-> query, register <-> d
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) mma32(acc, ktf[ks], dsf[ks]);
  };

  // Block t is computed out of buffer t & 1 while block t + 1 waits in registers (fetched a
  // step earlier) and is parked into the other buffer, which every wave has left at the
  // barrier that ended step t - 1.
  const int n_steps = (s + 31) >> 5;
  const int n_full = s >> 5;
  fetch(0);
  fetch_bias(0);
  park(0);
  __syncthreads();
  fetch(min(1, n_steps - 1) * 32);
  for (int t = 0; t < n_full; ++t) {
    step(std::false_type{}, t % NB, t * 32, min(t + 1, n_steps - 1) * 32);
    if (NB == 1) __syncthreads();
    park((t + 1) % NB);
    __syncthreads();
    fetch(min(t + 2, n_steps - 1) * 32);
  }
  if (n_full < n_steps) step(std::true_type{}, n_full % NB, n_full * 32, n_full * 32);
  if (q_ok) {
    T* dst = (T*)p.dq + elem(p, i, qi, h);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[4 * a + e];
      *reinterpret_cast<V4*>(dst + 8 * a + 4 * g) = from_f32<T>(v);
    }
  }
}

// dK and dV: a workgroup takes 128 keys of one (row, head), a wave 32 of them, and walks over
// the query blocks; Q, dO, their transposes and the queries' statistics are shared.  Works on
// S (not S^T): lane <-> key, register <-> query.  Bias2 is loaded along the queries' rows (8
// keys per load) and turned on its way through LDS; with Bias1 added it is the initial value
// of the S accumulator, -Delta that of dP.  Lanes whose key lies beyond s
// repeat key s - 1 and store nothing; queries beyond s exist in the last block only, which has
// its own copy of the step.  Everything shared is double-buffered: one barrier a step.
template <typename T, bool VEC>
__global__ __launch_bounds__(256, (BwdCfg<T, VEC>::kMinWaves)) void attn_bwd_kv_kernel(BwdParams p) {
  typedef typename Vec8<T>::type V8;
  typedef typename Vec4<T>::type V4;
  constexpr int NB = BwdCfg<T, VEC>::kBuffers;
  __shared__ __attribute__((aligned(32))) T rm[NB][2][32 * kTP];    // Q, dO
  constexpr bool TURN = Turned<T>::value;
  __shared__ __attribute__((aligned(32))) T tr[TURN ? 8 : NB * 2 * 32 * kTP];   // Q^T, dO^T (fp32 only)
  // Bias2 of the step: fp32 per wave as [key][query]; 16-bit one tile [query][128 keys] for
  // the workgroup, as it was loaded
  constexpr int kB2P = 136;   // pitch of the 16-bit tile (elements)
  __shared__ __attribute__((aligned(32))) T b2t[NB][TURN ? 32 * kB2P : 4 * 32 * kTP];
  __shared__ __attribute__((aligned(32))) float stats[NB][2][32];   // -log-sum-exp, -Delta of the 32 queries
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, ln = lane & 31, g = lane >> 5;
  const int s = p.s, H = p.heads;
  constexpr bool vec = VEC;
  const uint32_t n_wg = ((uint32_t)s + 127) / 128, items = n_wg * (uint32_t)H * (uint32_t)p.n_rows, item = xcd_item(items);
  if (item >= items) return;
  const int wg = item % n_wg, h = item / n_wg % H, i = item / n_wg / H;
  const int key0 = (wg * 4 + wave) * 32;
  const int kc = min(key0 + ln, s - 1);
  const bool k_ok = key0 + ln < s;
  V8 kf[2], vf[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    kf[kk] = load8<T>((const T*)p.k + elem(p, i, kc, h) + 16 * kk + 8 * g);
    vf[kk] = load8<T>((const T*)p.v + elem(p, i, kc, h) + 16 * kk + 8 * g);
  }
  const float b1v = p.b1 ? to_f32(((const T*)p.b1)[(int64_t)i * s + kc]) : 0.0f;
  const float* stat_src = g == 0 ? p.lse : p.delta;   // every wave fetches, wave 0 publishes
  f32x16 acc_dk, acc_dv;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc_dk[r] = acc_dv[r] = 0.0f;

  TilePiece<T> piece;
  float stat = 0.0f;
  // fp32: lane (ln, g) loads Bias2 of query q0 + ln for this wave's keys key0 + 16 g .. + 15.
  // 16-bit: thread t loads keys 8 (t & 7) .. + 7 of both halves of the workgroup's 128 keys for
  // query q0 + (t >> 3): eight neighbouring lanes read one 128-byte line (a lane per query
  // touches as many lines per load as it has lanes).
  V8 b2a, b2b;
  const int b2q = TURN ? tid >> 3 : ln;
  const int b2k = TURN ? wg * 128 + 8 * (tid & 7) : key0 + 16 * g;
  auto fetch = [&](int q0) {
    piece.fetch(p, p.q, p.dout, i, q0, h, tid);
    stat = stat_src[((int64_t)i * s + min(q0 + ln, s - 1)) * H + h];
    const T* b2row = (const T*)p.b2 + ((int64_t)h * s + min(q0 + b2q, s - 1)) * s;
    b2a = load_bias8_raw<T>(b2row, b2k, s, vec);
    b2b = load_bias8_raw<T>(b2row, b2k + (TURN ? 64 : 8), s, vec);
    asm volatile("" ::: "memory");   // the loads are issued here, a step ahead of their use
  };
  auto park = [&](int buf) {
    piece.park(rm[buf], tr + (TURN ? 0 : buf * 2 * 32 * kTP), TURN ? 0 : 2, tid);
    if (wave == 0) stats[buf][g][ln] = -stat;
    if (TURN) {
      store8<T>(&b2t[buf][b2q * kB2P + 8 * (tid & 7)], b2a);
      store8<T>(&b2t[buf][b2q * kB2P + 8 * (tid & 7) + 64], b2b);
    } else {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        b2t[buf][wave * 32 * kTP + (16 * g + t) * kTP + ln] = b2a[t];
        b2t[buf][wave * 32 * kTP + (16 * g + 8 + t) * kTP + ln] = b2b[t];
      }
    }
  };
  // one block of 32 queries out of buffer `buf`; TAIL: the block holds queries beyond s
  auto step = [&](auto tail_tag, int buf, int q0) {
    constexpr bool TAIL = decltype(tail_tag)::value;
    V8 qf[2], dof[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      qf[kk] = load8<T>(&rm[buf][0][perm_row(ln) * kTP + 16 * kk + 8 * g]);
      dof[kk] = load8<T>(&rm[buf][1][perm_row(ln) * kTP + 16 * kk + 8 * g]);
    }
    f32x16 sm, dp;
    f32x8 nlse[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int qb = 16 * ks + 8 * g;   // queries q0 + qb .. + 7 sit in registers 8 ks .. 8 ks + 7
      nlse[ks] = *reinterpret_cast<const f32x8*>(&stats[buf][0][qb]);
      const f32x8 ndel = *reinterpret_cast<const f32x8*>(&stats[buf][1][qb]);
      const f32x8 b28 = to_f32(TURN ? load8_turned(b2t[buf], kB2P, qb, 32 * wave + 16 * ((lane >> 4) & 1), lane)
                                    : load8<T>(&b2t[buf][wave * 32 * kTP + ln * kTP + qb]));
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        sm[8 * ks + t] = b1v + b28[t];
        dp[8 * ks + t] = ndel[t];
      }
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      mma32(sm, qf[kk], kf[kk]);    // S[query][key] (+ biases): lane <-> key, register <-> query
      mma32(dp, dof[kk], vf[kk]);   // dP[query][key] - Delta
    }
    V8 pf[2], dsf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int qb = 16 * ks + 8 * g;
      f32x8 pv, dv;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const int r = 8 * ks + t;
        float pr = fast_exp2(sm[r] * kBwdLog2e + nlse[ks][t]);
        if (TAIL) pr = q0 + qb + t < s ? pr : 0.0f;
        pv[t] = pr;
        dv[t] = pr * dp[r];
      }
      pf[ks] = from_f32<T>(pv);
      dsf[ks] = from_f32<T>(dv);
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const V8 qtf = TURN ? load8_turned(rm[buf][0], kTP, 16 * ks + 8 * g, 16 * ((lane >> 4) & 1), lane)
                          : load8<T>(&tr[TURN ? 0 : (buf * 2 + 0) * 32 * kTP + ln * kTP + 16 * ks + 8 * g]);
      const V8 dotf = TURN ? load8_turned(rm[buf][1], kTP, 16 * ks + 8 * g, 16 * ((lane >> 4) & 1), lane)
                           : load8<T>(&tr[TURN ? 0 : (buf * 2 + 1) * 32 * kTP + ln * kTP + 16 * ks + 8 * g]);
      mma32(acc_dv, dotf, pf[ks]);    // dV^T[d][key] += dO^T[d][query] P[query][key]
      mma32(acc_dk, qtf, dsf[ks]);    // dK^T[d][key] += Q^T[d][query] dS[query][key]
    }
  };

  // Block t is computed out of buffer t & 1 while block t + 1 waits in registers (fetched a
  // step earlier) and is parked into the other buffer, which every wave has left at the
  // barrier that ended step t - 1.
  const int n_steps = (s + 31) >> 5;
  const int n_full = s >> 5;
  fetch(0);
  park(0);
  __syncthreads();
  fetch(min(1, n_steps - 1) * 32);
  for (int t = 0; t < n_full; ++t) {
    step(std::false_type{}, t % NB, t * 32);
    if (NB == 1) __syncthreads();
    park((t + 1) % NB);
    __syncthreads();
    fetch(min(t + 2, n_steps - 1) * 32);
  }
  if (n_full < n_steps) step(std::true_type{}, n_full % NB, n_full * 32);
  if (k_ok) {
    T* dk = (T*)p.dk + elem(p, i, kc, h);
    T* dv = (T*)p.dv + elem(p, i, kc, h);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      f32x4 x, y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = acc_dk[4 * a + e];
        y[e] = acc_dv[4 * a + e];
      }
      *reinterpret_cast<V4*>(dk + 8 * a + 4 * g) = from_f32<T>(x);
      *reinterpret_cast<V4*>(dv + 8 * a + 4 * g) = from_f32<T>(y);
    }
  }
}

// LDS tiles of 32 channels, 16-bit: rows of 64 bytes, their four 16-byte pieces exchanged by bits 2 and 3 of the row, so that
// neither eight rows' pieces (vector reads and writes) nor four rows' halves (turning reads) meet in a bank.
__device__ __forceinline__ int piece_at(int row, int piece) { return row * 32 + ((piece ^ ((row >> 2) & 3)) << 3); }

// Eight elements of this lane's column out of such a tile, rows 16 ks + 8 g .. + 7 (g = lane / 32), column 16 (lane / 16 % 2) + lane % 16
struct TurnedAt {
  int lo, hi;   // of the rows' first and second four
  __device__ explicit TurnedAt(int lane) {
    const int row = 8 * (lane >> 5) + ((lane & 15) >> 2), piece = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), e = 4 * (lane & 1);
    lo = piece_at(row, piece) + e;
    hi = piece_at(row + 4, piece) + e;
  }
  __device__ __forceinline__ bf16x8 load(const bf16_t* tile, int ks) const {
    typedef short v4s __attribute__((ext_vector_type(4)));
    typedef short v8s __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) v4s* LdsV4;
    const v4s a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4)(tile + lo + 512 * ks));
    const v4s b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsV4)(tile + hi + 512 * ks));
    return __builtin_bit_cast(bf16x8, (v8s)__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
  }
};

// dQ, dK and dV in one pass, 16-bit, rows of at most 32 NW NBK positions: a workgroup takes one (row, head), a wave NBK blocks of
// 32 keys (every NW-th), and all walk over the query blocks.  Logits and dP are formed once instead of once for dQ and
// once for dK / dV.  Works on S like the dK / dV kernel (lane <-> key, register <-> query); dQ contracts over the keys, so
// a block's dS goes through LDS once more and is turned on its way out, and the waves' dQ of a query block, each over its own
// keys, are added through LDS in wave order.  Bias2 reaches the S accumulator on the matrix pipe, S += B2 * 1, from fragments
// loaded along the queries' rows; Bias1 is the accumulator's initial value, and -inf for keys beyond s.
// At 384 rows of 384 positions and 4 heads (us per launch, parts left out in turn): 42 are the workgroups' beginnings and ends, K, V, dK and dV
// at the memory's rate; of the 135 of the walk the products alone take 40, Bias2's loads 28, the operands out of LDS 24, the
// statistics 11, the exponentials 7, dS' way through LDS 5: two waves per SIMD (the accumulators of all its keys are registers) hide
// little of one under the other.  Hence: O and the log-sum-exp come in along the walk, where Delta is formed, and not ahead of it (O, dO
// and 384 log-sum-exps first: 75 us of beginnings and ends); K and V are requested in one go; dK and dV leave as whole rows of 64
// bytes through LDS (as pieces of 8 bytes from the accumulators 56); Q and dO fragments are read again for every block, since kept across
// the blocks they spill.  203 us before, 177 with these; 109 + 126 in two kernels.  Tried without gain: V out of the caches instead of
// registers, dQ's product a block behind, Bias2 laid out in fragments by a launch of its own (170 + 5 us).
template <int NW, int NBK>
__global__ __launch_bounds__(NW * 64, NBK == 1 ? 3 : 2) void attn_bwd_row_kernel(BwdParams p) {
  typedef bf16_t T;
  typedef Vec8<T>::type V8;
  typedef Vec4<T>::type V4;
  constexpr int KB = NW * NBK, kExWave = 16 * kWave * 4;   // bytes of a wave's partial dQ
  static_assert(2 * 1024 * (int)sizeof(T) <= kExWave, "a wave's dS tile, and a block's dK and dV on their way out, fit its place for dQ");
  __shared__ __attribute__((aligned(32))) T kt[KB][1024];      // K, row-major, read by the wave that owns the block
  __shared__ __attribute__((aligned(32))) T rm[2][2][1024];      // Q, dO of the step
  __shared__ f32x8 stats[2][2][4];   // -log-sum-exp, -Delta of the step's queries
  // two of them, for a step and the next: a wave's dS tile, later its partial dQ
  __shared__ __attribute__((aligned(32))) char ex[2][NW][kExWave];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 31, g = lane >> 5;
  const int s = p.s, H = p.heads;
  const uint32_t items = (uint32_t)H * (uint32_t)p.n_rows, item = xcd_item(items);
  if (item >= items) return;
  const int h = item % H, i = item / H;

  // this wave's keys (all loads in front of the first wait; without a Bias1 they read Bias2, which counts for nothing)
  V8 vf[NBK][2], k_in[NBK][2];
  T b1_in[NBK];
  float b1v[NBK];
  f32x16 acc_dk[NBK], acc_dv[NBK];
  const T* const b1_src = p.b1 ? (const T*)p.b1 + (int64_t)i * s : (const T*)p.b2;
#pragma unroll
  for (int b = 0; b < NBK; ++b) {
    const int kc = min((b * NW + wave) * 32 + ln, s - 1);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      k_in[b][kk] = load8<T>((const T*)p.k + elem(p, i, kc, h) + 16 * kk + 8 * g);
      vf[b][kk] = load8<T>((const T*)p.v + elem(p, i, kc, h) + 16 * kk + 8 * g);
    }
    b1_in[b] = b1_src[kc];
  }
  asm volatile("" ::: "memory");
#pragma unroll
  for (int b = 0; b < NBK; ++b) {
    b1v[b] = (b * NW + wave) * 32 + ln >= s ? -INFINITY : p.b1 ? to_f32(b1_in[b]) : 0.0f;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) store8<T>(&kt[b * NW + wave][piece_at(ln, 2 * kk + g)], k_in[b][kk]);
#pragma unroll
    for (int r = 0; r < 16; ++r) acc_dk[b][r] = acc_dv[b][r] = 0.0f;
  }
  // the unit matrix as the other operand of Bias2's product (slot <-> key of the block, lane <-> key)
  V8 one[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int t = 0; t < 8; ++t) one[kk][t] = (T)(ln == 16 * kk + 8 * g + t ? 1.0f : 0.0f);

  const int n_steps = (s + 31) >> 5;
  const TurnedAt turned(lane);
  // Q and dO tiles: the first 256 threads, 8 channels of one row of one tile each, a step ahead (positions of a row times
  // heads and channels stay below 2^31).  The threads of dO also take O and form Delta = sum_d O * dO on the way, four lanes
  // to a query, left in p.delta for the dBias2 kernel.
  const bool of_dout = wave >> 1 & 1;   // (the same for a wave)
  V8 piece, o_piece;
  float lse_piece;
  const int64_t row_at = elem(p, i, 0, h);
  const T* const tile_src = (const T*)(of_dout ? p.dout : p.q) + row_at;
  const T* const o_src = (const T*)(of_dout ? p.o : p.q) + row_at;
  const int64_t stat_at = (int64_t)i * s * H + h;
  const int tile_row = (tid & 127) >> 2, tile_col = 8 * (tid & 3), tile_at = piece_at(tile_row, tid & 3);
  auto fetch = [&](int t) {
    if (NW == 4 || wave < 4) {
      const uint32_t at = (uint32_t)min(t * 32 + tile_row, s - 1) * (uint32_t)H;
      piece = load8<T>(tile_src + (at * 32 + tile_col));
      o_piece = load8<T>(o_src + (at * 32 + tile_col));
      lse_piece = p.lse[stat_at + at];
    }
  };
  auto park = [&](int t) {
    if (NW == 4 || wave < 4) {
      store8<T>(&rm[t & 1][of_dout][tile_at], piece);
      if (of_dout) {
        const f32x8 of = to_f32(o_piece), df = to_f32(piece);
        float d = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) d += of[e] * df[e];
        d += __shfl_xor(d, 1, 64);
        d += __shfl_xor(d, 2, 64);
        const int q = t * 32 + tile_row;
        if ((tid & 3) == 0) {
          reinterpret_cast<float*>(stats[t & 1][0])[tile_row] = q < s ? -lse_piece : -INFINITY;   // (beyond s: probability 0)
          reinterpret_cast<float*>(stats[t & 1][1])[tile_row] = -d;
          if (q < s) p.delta[stat_at + (uint32_t)q * (uint32_t)H] = d;
        }
      }
    }
  };
  // Bias2 fragments of block b at step t: lane <-> query perm_row(ln), slots <-> 8 keys; one block ahead.  Rows start at any
  // element.  The last 8 keys are read again for those beyond, and moved down (zeros above: -inf plus whatever lies there
  // might not be -inf).
  const T* b2h = (const T*)p.b2 + (int64_t)h * s * s;
  const int b2q = perm_row(ln);
  V8 b2n[2];
  auto fetch_bias = [&](int t, int b) {
    const int key0 = (b * NW + wave) * 32;
    const uint32_t row = (uint32_t)min(t * 32 + b2q, s - 1) * (uint32_t)s;
    if (key0 + 32 <= s) {   // the same for the whole wave
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) __builtin_memcpy(&b2n[kk], b2h + (row + (uint32_t)(key0 + 16 * kk + 8 * g)), sizeof(V8));
    } else {
      int part0 = key0;
      asm volatile("" : "+s"(part0));   // (nothing of it is formed ahead of the walk: no registers for it)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int kb = part0 + 16 * kk + 8 * g, from = min(kb, s - 8);
        unsigned __int128 v;
        __builtin_memcpy(&v, b2h + (row + (uint32_t)from), sizeof(v));
        v = kb >= s ? 0 : v >> (16 * (kb - from));
        __builtin_memcpy(&b2n[kk], &v, sizeof(v));
      }
    }
  };
  fetch(0);
  fetch_bias(0, 0);
  park(0);
  __syncthreads();
  for (int t = 0; t < n_steps; ++t) {
    const int buf = t & 1;
    fetch(t + 1);
    asm volatile("" ::: "memory");   // (issued here, a step ahead of their use)
    T* const ds_tile = reinterpret_cast<T*>(&ex[buf][wave][0]);
    f32x16 dq;
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[r] = 0.0f;
#pragma unroll
    for (int b = 0; b < NBK; ++b) {
      const int blk = b * NW + wave;
      // (opaque offsets: what all steps or all blocks read alike would be kept in registers that are not there)
      int kt_off = blk * 1024, rm_off = buf * 2048, st_off = buf * 8;
      asm volatile("" : "+v"(kt_off), "+v"(rm_off), "+v"(st_off));
      const T* const kb = &kt[0][0] + kt_off;
      const T* const qd = &rm[0][0][0] + rm_off;
      f32x16 sm, dp;
      float b1 = b1v[b];
      asm volatile("" : "+v"(b1));   // (sixteen registers with the same value, per block)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sm[r] = b1;
        dp[r] = stats[0][1][st_off + 2 * (r >> 3) + g][r & 7];
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) mma32(sm, finite_low(b2n[kk]), one[kk]);   // Bias1 + Bias2
      __builtin_amdgcn_sched_barrier(0);
      fetch_bias(b + 1 < NBK ? t : t + 1, b + 1 < NBK ? b + 1 : 0);
      asm volatile("" ::: "memory");
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        mma32(sm, load8<T>(qd + piece_at(b2q, 2 * kk + g)), load8<T>(kb + piece_at(ln, 2 * kk + g)));   // S[query][key] (+ biases)
        mma32(dp, load8<T>(qd + 1024 + piece_at(b2q, 2 * kk + g)), vf[b][kk]);                           // dP[query][key] - Delta
      }
      __builtin_amdgcn_sched_barrier(0);
      V8 pf[2], dsf[2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const f32x8 nl = stats[0][0][st_off + 2 * ks + g];
        f32x8 pv, dv;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int r = 8 * ks + e;
          const float pr = fast_exp2(sm[r] * kBwdLog2e + nl[e]);
          pv[e] = pr;
          dv[e] = pr * dp[r];
        }
        pf[ks] = from_f32<T>(pv);
        dsf[ks] = from_f32<T>(dv);
        store8<T>(ds_tile + piece_at(ln, 2 * ks + g), dsf[ks]);   // [key][query]
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        mma32(acc_dv[b], turned.load(qd + 1024, ks), pf[ks]);    // dV^T[d][key] += dO^T P
        mma32(acc_dk[b], turned.load(qd, ks), dsf[ks]);   // dK^T[d][key] += Q^T dS
      }
      __builtin_amdgcn_sched_barrier(0);
      wave_lds_sync();
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)   // dQ^T[d][query] += K^T dS^T
        mma32(dq, turned.load(kb, ks), turned.load(ds_tile, ks));
      wave_lds_sync();
    }
    {
      float* d = reinterpret_cast<float*>(&ex[buf][wave][0]) + lane;
#pragma unroll
      for (int r = 0; r < 16; ++r) d[r * kWave] = dq[r];
    }
    park(t + 1);
    // the waves' dQ of this step and the next step's tiles are complete; the other pair of places was read before the
    // last barrier
    __syncthreads();
    if (wave < 4) {   // wave w: registers 4 w .. 4 w + 3, channels 8 w + 4 g .. + 3 of the lane's query
      f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += reinterpret_cast<const float*>(&ex[buf][w][0])[(4 * wave + e) * kWave + lane];
      const int q = t * 32 + ln;
      if (q < s) *reinterpret_cast<V4*>((T*)p.dq + elem(p, i, q, h) + 8 * wave + 4 * g) = from_f32<T>(sum);
    }
  }
  // dK and dV, a block at a time through the place of this wave's partial dQ that the last step left alone: four lanes to a
  // key store its 64 bytes (from the accumulators they would be pieces of 8)
  T* const out_tile = reinterpret_cast<T*>(&ex[n_steps & 1][wave][0]);
#pragma unroll
  for (int b = 0; b < NBK; ++b) {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      f32x4 x, y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = acc_dk[b][4 * a + e];
        y[e] = acc_dv[b][4 * a + e];
      }
      *reinterpret_cast<V4*>(out_tile + piece_at(ln, a) + 4 * g) = from_f32<T>(x);
      *reinterpret_cast<V4*>(out_tile + 1024 + piece_at(ln, a) + 4 * g) = from_f32<T>(y);
    }
    wave_lds_sync();
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int row = 16 * half + (lane >> 2), key = (b * NW + wave) * 32 + row;
      const V8 x = load8<T>(out_tile + piece_at(row, lane & 3)), y = load8<T>(out_tile + 1024 + piece_at(row, lane & 3));
      if (key < s) {
        const int64_t at = elem(p, i, key, h) + 8 * (lane & 3);
        store8<T>((T*)p.dk + at, x);
        store8<T>((T*)p.dv + at, y);
      }
    }
    wave_lds_sync();
  }
}

// Whether a workgroup takes whole rows (attn_bwd_row_kernel): 16-bit rows whose accumulators for dK and dV fit the registers
// of eight waves, at least one vector long, and enough of them.  A (row, head) is one workgroup, whatever its length: what
// these cost is rounds of the machine - 512 of four waves with two or three blocks each, 256 of eight waves -, where the kernels
// of 128 queries or keys a workgroup, two to six of them for a pair, fill it sooner.  So as many pairs are asked for, round by round, as
// give the others a round more (256 workgroups; three to a pair: from 171 pairs on, from 342).
// us for dQ, dK and dV, by themselves | so, 4 heads, (rows, positions):
//   one block a wave: (1, 128) 11.5 | 8.9, (256, 128) 31.8 | 25.0
//   two: (32, 136) 13.5 | 15.2, (32, 256) 17.4 | 20.7, (34, 136) 17.7 | 15.2, (36, 200) 20.2 | 19.3, (36, 256) 22.7 | 20.9, (112, 200) 38.5 | 29.0,
//     (130, 200) 43.0 | 45.0, (160, 200) 45.5 | 44.8
//   three, 8 divides the positions: (1, 384) 20.5 | 38.8, (48, 384) 40 | 46, (84, 264) 41 | 45, (84, 384) 57 | 59, (88, 264) 48.4 | 45.1, (88, 384)
//     63.3 | 59.9, (130, 384) 86 | 100, (160, 384) 104 | 100, (192, 384) 115 | 101; otherwise: (40, 300) 31.8 | 35.7, (47, 300) 39.9 | 36.7, (72, 300) 54 | 49,
//     (130, 300) 81.5 | 84.8, (144, 300) 86 | 84
//   eight waves: (48, 400) 45 | 41, (80, 400) 69 | 78, (96, 400) 81 | 79, (48, 512) 57 | 48, (96, 512) 103 | 93, (48, 520) 70 | 70, (80, 520) 108 | 136, (96, 520)
//     128 | 137, (112, 520) 141 | 138, (160, 520) 203 | 205, (64, 640) 98 | 86, (96, 640) 153 | 166, (112, 640) 177 | 167, (48, 768) 115 | 99, (80, 768) 184 | 195,
//     (96, 768) 217 | 196
// The operator forward and backward: 384 rows of 384, 390 | 355; 768 of 768, 3054 | 2735.
template <typename T>
bool rows_at_once(const BwdParams& p) {
  if (sizeof(T) != 2 || p.s < 8 || p.s > 768) return false;
  if (p.s <= 128) return true;
  const int64_t pairs = (int64_t)p.heads * p.n_rows;
  if (p.s <= 256) return pairs > 128;
  if (p.s <= 384) return pairs >= (p.s % 8 == 0 ? 342 : 171) + 290 * ((pairs - 1) / 512);
  return pairs >= (p.s > 512 && p.s <= 640 ? 216 : 192) * ((pairs + 255) / 256);
}

// dBias2, the walk: a workgroup takes a tile of queries x keys of one head and walks over the rows, whose Q, dO, K and V tiles its waves
// share.  Works on S^T like dQ.  Bias2 itself does not change along the walk and stays in registers; a row's Bias1 is added to it for the
// initial value of the S^T accumulator, -Delta is that of dP^T.  Nothing in the walk looks at s: queries and keys beyond it repeat the last
// one, and what accumulates for them is not stored.
// The walk is cut into slices of rows: 384 tokens and 4 heads are 96 workgroups (of three waves; a compute unit holds twelve waves), every
// one a serial chain over 384 rows.  Slices write fp32 partial sums that
// attn_bwd_db2_sum_kernel adds in order (no atomics).  A slice's workgroups all go to one XCD
// (workgroups are dealt to the XCDs in turn, and the slice is the fastest index), whose L2 then fetches the slice's rows
// once; with a slice's workgroups on all eight the rows come through the memory-side cache eight times.  us at 384 rows,
// 384 tokens, 4 heads, bf16, tiles of 64 x 64: one slice 312; seven slices, spread 165 with the sum; eight, one per XCD, 107 + 4.

// What a lane holds of a 32 x 32 block of dBias2: keys key0 + 16 ks + 8 g .. + 7 of query qi, in acc[8 ks ..]
template <typename T>
__device__ __forceinline__ void db2_store(const BwdParams& p, int slice, int h, int qi, int key0, int g, const f32x16& acc) {
  const int s = p.s;
  const bool vec = (s & 7) == 0;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int kb = key0 + 16 * ks + 8 * g;
    f32x8 v;
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = acc[8 * ks + t];
    if (p.parts) {
      float* const dst = p.parts + (((int64_t)slice * p.heads + h) * s + qi) * s;
      if (vec) {
        if (kb < s) store8<float>(dst + kb, v);
      } else {
#pragma unroll
        for (int t = 0; t < 8; ++t)
          if (kb + t < s) dst[kb + t] = v[t];
      }
    } else {
      T* const dst = (T*)p.db2 + ((int64_t)h * s + qi) * s;
      if (vec) {
        if (kb < s) store8<T>(dst + kb, from_f32<T>(v));
      } else {
#pragma unroll
        for (int t = 0; t < 8; ++t)
          if (kb + t < s) dst[kb + t] = from_f32<T>(v[t]);
      }
    }
  }
}

// 16-bit: NWQ waves, each 32 queries x NB blocks of 32 keys that share the query's operands and statistics; the next row's tiles
// travel by direct-to-LDS loads while a row is computed.  A lane's place in LDS is fixed by the instruction, so the exchange
// of pieces (piece_at) is one of the global addresses.
// Bound by what a compute unit issues, its LDS and the way of the tiles there together: with two blocks and four waves 67 vector instructions
// and 5 MFMA per block, and 9 KB through LDS.  In tiles of 64 x 64, a block a wave, with the tiles through registers, they were 82, 5
// and 12 KB (figures: db2_walk).  Two waves per SIMD of twice the registers: 123 us against 98 at 384 positions; sixteen slices instead
// of eight: 100 - 117.
template <int NWQ, int NB>
__global__ __launch_bounds__(NWQ * 64, 3) void attn_bwd_db2_kernel(BwdParams p) {
  typedef bf16_t T;
  typedef Vec8<T>::type V8;
  constexpr int kQ = 32 * NWQ, kKeys = 32 * NB;
  __shared__ __attribute__((aligned(32))) T tiles[2][(2 * kQ + 2 * kKeys) * 32];   // Q, dO, K, V
  constexpr int kDo = kQ * 32, kK = 2 * kQ * 32, kV = kK + kKeys * 32;               // where they start
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 31, g = lane >> 5;
  const int s = p.s, H = p.heads;
  const int q_tiles = (s + kQ - 1) / kQ, k_tiles = (s + kKeys - 1) / kKeys, slice = blockIdx.x % p.slices;
  // One slice: workgroups in turn put the query tiles on the XCDs in turn, and where their number shares little with 8 every XCD
  // fetches all of a row; neighbours then stay on one (figures: db2_walk).
  const bool spans = p.slices == 1 && (q_tiles & 3) != 0;
  const int pair = spans ? xcd_item((uint32_t)q_tiles * (uint32_t)k_tiles * (uint32_t)H) : blockIdx.x / p.slices;
  if (pair >= q_tiles * k_tiles * H) return;
  const int row_begin = (int)((int64_t)p.n_rows * slice / p.slices), row_end = (int)((int64_t)p.n_rows * (slice + 1) / p.slices);
  const int qs0 = pair % q_tiles * kQ, ks0 = pair / q_tiles % k_tiles * kKeys, h = pair / q_tiles / k_tiles;
  const int q0 = qs0 + 32 * wave, qi = min(q0 + ln, s - 1);
  const bool vec = (s & 7) == 0;
  const T* const b2row = (const T*)p.b2 + ((int64_t)h * s + qi) * s;
  f32x16 b2acc[NB], acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const f32x8 lo = load_bias8<T>(b2row, ks0 + 32 * b + 8 * g, s, vec), hi = load_bias8<T>(b2row, ks0 + 32 * b + 16 + 8 * g, s, vec);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      b2acc[b][r] = r < 8 ? lo[r & 7] : hi[r & 7];
      acc[b][r] = 0.0f;
    }
  }
  // Bias1 reaches the accumulator on the matrix pipe (see the dQ kernel): one value per lane, that of the key its accumulator row
  // stands for, in K slot 0 of one more product.  (Without a Bias1 the loads go to Bias2's row and count for nothing.)
  const T* const b1base = p.b1 ? (const T*)p.b1 : b2row;
  const int64_t b1pitch = p.b1 ? s : 0;
  const bool b1on = p.b1 != nullptr;
  unsigned off_b1[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) off_b1[b] = min(ks0 + 32 * b + perm_row(ln), s - 1);
  V8 one_frag = zero_frag<T>();
  one_frag[0] = (T)(g == 0 && b1on ? 1.0f : 0.0f);

  // This wave's share of a row's tiles: 16 rows of 64 bytes an instruction, two of Q's and dO's 2 NWQ, its part of K's and V's four
  // (three waves load one of those twice, to the same place).  A row moves the base address, the same for all lanes.
  constexpr int kKv = (2 * NB + NWQ - 1) / NWQ;
  const int piece8 = 8 * ((lane & 3) ^ ((lane >> 4) & 3));
  auto tile_offset = [&](int pos) { return (((uint32_t)min(pos + (lane >> 2), s - 1) * H + h) * 32 + piece8) * (uint32_t)sizeof(T); };
  uint32_t off_q[2], off_k[kKv];
  int kv_at[kKv];
#pragma unroll
  for (int j = 0; j < 2; ++j) off_q[j] = tile_offset(qs0 + 16 * (wave + NWQ * j));
#pragma unroll
  for (int j = 0; j < kKv; ++j) {
    kv_at[j] = min(wave + NWQ * j, 2 * NB - 1);
    off_k[j] = tile_offset(ks0 + 16 * kv_at[j]);
  }
  const int64_t row_elems = (int64_t)s * H * 32, row_stats = (int64_t)s * H;
  const unsigned off_stat = (unsigned)qi * H + h;
  float mq_n, dq_n;
  T b1_n[NB];
  auto fetch = [&](int i) {
    T* const t = tiles[i & 1];
    mq_n = (p.lse + i * row_stats)[off_stat];
    dq_n = (p.delta + i * row_stats)[off_stat];
    const T* const b1row = b1base + i * b1pitch;
#pragma unroll
    for (int b = 0; b < NB; ++b) b1_n[b] = b1row[off_b1[b]];
    const uint64_t qa = (uint64_t)((const T*)p.q + i * row_elems), da = (uint64_t)((const T*)p.dout + i * row_elems);
    const uint64_t ka = (uint64_t)((const T*)p.k + i * row_elems), va = (uint64_t)((const T*)p.v + i * row_elems);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      load_to_lds16_s<0>(qa, off_q[j], lds_address(t + (wave + NWQ * j) * 512));
      load_to_lds16_s<0>(da, off_q[j], lds_address(t + kDo + (wave + NWQ * j) * 512));
    }
#pragma unroll
    for (int j = 0; j < kKv; ++j) {
      load_to_lds16_s<0>(ka, off_k[j], lds_address(t + kK + kv_at[j] * 512));
      load_to_lds16_s<0>(va, off_k[j], lds_address(t + kV + kv_at[j] * 512));
    }
  };
  // Row i is computed out of buffer i & 1 while row i + 1 travels into the other one, which every wave left at the last barrier.
  const int last = row_end - 1;
  fetch(row_begin);
  ring_barrier<0>();
  for (int i = row_begin; i < row_end; ++i) {
    const float neg_mq = -mq_n, neg_dq = -dq_n;
    T b1[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) b1[b] = b1_n[b];
    if (i < last) fetch(i + 1);
    const T* const t = tiles[i & 1];
    V8 qf[2], dof[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      qf[kk] = load8<T>(t + piece_at(32 * wave + ln, 2 * kk + g));
      dof[kk] = load8<T>(t + kDo + piece_at(32 * wave + ln, 2 * kk + g));
    }
    f32x16 ndq;
#pragma unroll
    for (int r = 0; r < 16; ++r) ndq[r] = neg_dq;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      V8 b1a = zero_frag<T>();
      b1a[0] = g == 0 && b1on ? b1[b] : (T)0.0f;
      f32x16 st = b2acc[b], dp = ndq;
      if (b) __builtin_amdgcn_sched_barrier(0);   // (one block after the other: both blocks' logits at once are registers that are not there)
      mma32(st, b1a, one_frag);   // Bias2 + Bias1
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const V8 kf = load8<T>(t + kK + piece_at(32 * b + perm_row(ln), 2 * kk + g));
        const V8 vf = load8<T>(t + kV + piece_at(32 * b + perm_row(ln), 2 * kk + g));
        mma32(st, kf, qf[kk]);    // S^T[key][query] (+ biases)
        mma32(dp, vf, dof[kk]);   // dP^T[key][query] - Delta
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[b][r] += fast_exp2(st[r] * kBwdLog2e + neg_mq) * dp[r];
    }
    ring_barrier<0>();
  }
  if (q0 + ln < s) {
#pragma unroll
    for (int b = 0; b < NB; ++b) db2_store<T>(p, slice, h, qi, ks0 + 32 * b, g, acc[b]);
  }
}

// fp32: four waves, tiles of 64 queries x 64 keys, a 32 x 32 quadrant each; one buffer, through registers.
template <bool VEC>
__global__ __launch_bounds__(256, 1) void attn_bwd_db2_fp32_kernel(BwdParams p) {
  typedef float T;
  typedef Vec8<T>::type V8;
  __shared__ __attribute__((aligned(32))) T tiles[4][64 * kTP];   // Q, dO (64 queries), K, V (64 keys)
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, ln = lane & 31, g = lane >> 5;
  const int s = p.s, H = p.heads;
  const int slice = blockIdx.x % p.slices, pair = blockIdx.x / p.slices, tiles_s = (s + 63) / 64;
  const int row_begin = (int)((int64_t)p.n_rows * slice / p.slices), row_end = (int)((int64_t)p.n_rows * (slice + 1) / p.slices);
  const int qs0 = pair % tiles_s * 64, ks0 = pair / tiles_s % tiles_s * 64, h = pair / tiles_s / tiles_s;
  const int wq = wave >> 1, wk = wave & 1;
  const int q0 = qs0 + 32 * wq, key0 = ks0 + 32 * wk;
  const int qi = min(q0 + ln, s - 1);
  const bool q_ok = q0 + ln < s;
  const T* b2row = (const T*)p.b2 + ((int64_t)h * s + qi) * s;
  f32x8 b2f[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) b2f[ks] = load_bias8<T>(b2row, key0 + 16 * ks + 8 * g, s, VEC);
  // (without a Bias1 the loads go to Bias2's row and count for nothing: no load under a branch)
  const T* b1base = p.b1 ? (const T*)p.b1 : b2row;
  const int64_t b1pitch = p.b1 ? s : 0;
  const bool b1on = p.b1 != nullptr;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;

  // thread t: 8 channels (t & 3) of row t >> 2 of each of the four 64-row tiles.  Along the
  // walk only the row's base address changes, the same for all lanes: what a lane adds to it
  // is formed once.
  const int crow = tid >> 2, cc = 8 * (tid & 3), park_at = crow * kTP + cc;
  const unsigned off_q = ((unsigned)min(qs0 + crow, s - 1) * H + h) * 32 + cc;
  const unsigned off_k = ((unsigned)min(ks0 + crow, s - 1) * H + h) * 32 + cc;
  const unsigned off_stat = (unsigned)qi * H + h;
  unsigned off_b1[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) off_b1[ks] = VEC ? min(key0 + 16 * ks + 8 * g, s - 8) : 0;
  const int64_t row_elems = (int64_t)s * H * 32, row_stats = (int64_t)s * H;
  V8 piece[4], b1n[2];
  float mq_n = 0.0f, dq_n = 0.0f;
  auto fetch = [&](int i) {
    piece[0] = load8<T>((const T*)p.q + i * row_elems + off_q);
    piece[1] = load8<T>((const T*)p.dout + i * row_elems + off_q);
    piece[2] = load8<T>((const T*)p.k + i * row_elems + off_k);
    piece[3] = load8<T>((const T*)p.v + i * row_elems + off_k);
    mq_n = (p.lse + i * row_stats)[off_stat];
    dq_n = (p.delta + i * row_stats)[off_stat];
    const T* b1row = b1base + i * b1pitch;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      b1n[ks] = VEC ? load8<T>(b1row + off_b1[ks]) : load_bias8_raw<T>(b1row, key0 + 16 * ks + 8 * g, s, false);
  };
  const int last = row_end - 1;
  fetch(row_begin);
#pragma unroll
  for (int w = 0; w < 4; ++w) store8<T>(&tiles[w][park_at], piece[w]);
  float neg_mq = -mq_n, neg_dq = -dq_n;
  V8 b1c[2] = {b1n[0], b1n[1]};
  __syncthreads();
  for (int i = row_begin; i < row_end; ++i) {
    fetch(min(i + 1, last));
    asm volatile("" ::: "memory");   // the loads are issued here, a step ahead of their use
    f32x16 st, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) dp[r] = neg_dq;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const f32x8 b1f = to_f32(b1c[ks]);
#pragma unroll
      for (int t = 0; t < 8; ++t) st[8 * ks + t] = (b1on ? b1f[t] : 0.0f) + b2f[ks][t];
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = 16 * kk + 8 * g;
      const V8 qf = load8<T>(&tiles[0][(32 * wq + ln) * kTP + c]), dof = load8<T>(&tiles[1][(32 * wq + ln) * kTP + c]);
      const V8 kf = load8<T>(&tiles[2][(32 * wk + perm_row(ln)) * kTP + c]), vf = load8<T>(&tiles[3][(32 * wk + perm_row(ln)) * kTP + c]);
      mma32(st, kf, qf);    // S^T[key][query] (+ biases)
      mma32(dp, vf, dof);   // dP^T[key][query] - Delta
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] += fast_exp2(st[r] * kBwdLog2e + neg_mq) * dp[r];
    __syncthreads();
    // the next row: tiles into LDS, its statistics and Bias1 into this step's places
#pragma unroll
    for (int w = 0; w < 4; ++w) store8<T>(&tiles[w][park_at], piece[w]);
    neg_mq = -mq_n;
    neg_dq = -dq_n;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) b1c[ks] = b1n[ks];
    __syncthreads();
  }
  if (q_ok) db2_store<T>(p, slice, h, qi, key0, g, acc);
}

// dBias2 = the slices' partial sums added in order, V values per thread (4 where the values of a slice are
// whole vectors).  Reads what the kernel before it left in the caches: 19 MB at 384 tokens, 4 us.
template <typename T, int V>
__global__ __launch_bounds__(256) void attn_bwd_db2_sum_kernel(const float* __restrict__ parts, T* __restrict__ db2, int slices, int64_t n) {
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (e >= n) return;
  if constexpr (V == 4) {
    f32x4 sum = *reinterpret_cast<const f32x4*>(parts + e);
    for (int sl = 1; sl < slices; ++sl) sum += *reinterpret_cast<const f32x4*>(parts + sl * n + e);
    *reinterpret_cast<typename Vec4<T>::type*>(db2 + e) = from_f32<T>(sum);
  } else {
    float sum = parts[e];
    for (int sl = 1; sl < slices; ++sl) sum += parts[sl * n + e];
    db2[e] = from_f32<T>(sum);
  }
}

// Slices of rows of dBias2's walk: eight, one per XCD, or as many more (multiples of eight) as 64 x 64 tiles make 1024 of, of at least
// 8 rows, as long as the partial sums (4 S^2 H bytes per slice, written and read once) stay within 128 MB.  16-bit, up to 100 blocks of
// 32 x 32: as many as make some 2300 blocks, one for 16 rows and eight more at most: there every block is a wave by itself (db2_walk),
// of which a SIMD takes two in little more than the time of one, and what more slices save on the walk goes into their sums.  us, slices by
// 64 x 64 tiles / by blocks, 4 heads: 256 rows of 64 19.5 / 18.6, 512 of 64 25.9 / 23.7, 512 of 96 31.0 / 25.7, 200 of 128 20.8 / 17.0, 512
// of 128 33.3 / 26.7, 768 of 128 37.4 / 33.0, 160 of 160 21.0 / 18.0, 320 of 160 31.3 / 25.4; above 100: 512 of 128 with 8 heads 42.3 / 47.9, 448
// of 224 46.3 / 50.5.
int triattn_bwd_slices(int n_rows, int s, int heads, bool bits16) {
  const int64_t tiles = (s + 63) / 64, pairs = tiles * tiles * heads, blocks = (int64_t)((s + 31) / 32) * ((s + 31) / 32) * heads;
  if (pairs <= 0 || n_rows <= 0) return 1;
  int64_t want = bits16 && blocks <= 100 ? std::min<int64_t>(2304 / blocks, n_rows / 16 + 8) : 1024 / pairs;
  want = std::min<int64_t>(std::max<int64_t>(8, want), n_rows / 8);
  if (want > 8) want &= ~(int64_t)7;
  return want > 1 && want * heads * s * s * 4 <= (int64_t)128 << 20 ? (int)want : 1;
}

// dBias2's walk, 16-bit: waves of a workgroup and blocks of a wave.  A small one is a chain of rows, whose length counts: up to two
// 32 x 32 blocks for every SIMD, two waves of one block each (a SIMD holds three; 2048 blocks: 256 rows of 256 in 8 slices 34.2 us,
// four waves of two 38.1; 2304: 12 rows of 768 17.9 / 17.2).  Beyond, two blocks a wave, four waves or three; the work of a
// compute unit is that of the workgroups it gets, in turn or at once, so the fullest one's waves count, and four do in the time of
// three what loads a quarter less.  us at S rows of S positions, 4 heads, 64 x 64 tiles of four waves (before) / two waves of one block /
// three of two / four of two: S = 64 7.4 / 5.6 / 8.7 / 9.0, 96 9.6 / 8.8 / 12.3 / 12.6, 160 15.2 / 13.6 / 16.4 / 17.6, 192 18.1 / 21.4 / 18.9 / 20.1, 256
// 30.7 / 39 / 31 / 27.5, 288 50.8 / 54 / 45.2 / 48, 320 59.8 / 79 / 63 / 53, 352 87.8 / 96 / 74.4 / 77, 384 107 / 126 / 88 / 94, 416 139 / 172 / 138 / 132,
// 512 222 / 324 / 250 / 215, 640 471 / 927 / 476 / 393, 768 781 / - / 763 / 659.
template <typename T>
static void db2_walk(const BwdParams& p, hipStream_t stream) {
  const auto groups = [&](int queries, int keys) {
    return (unsigned)((p.s + queries - 1) / queries) * (unsigned)((p.s + keys - 1) / keys) * (unsigned)p.heads * (unsigned)p.slices;
  };
  if constexpr (sizeof(T) == 2) {
    // (with one slice spans of whole workgroups per XCD, see the kernel.  us, 64 rows, 4 heads, in turn / in spans: S = 1050 171 / 138, 1100 201 / 132,
    // 1280 185 / 162, 1300 260 / 198; the query tiles a multiple of four, 1500 233 / 251, 2048 365 / 477; 3 rows of 600 7.5 / 6.6)
    const auto grid = [&](int queries, int keys) { return dim3((groups(queries, keys) + 7) / 8 * 8); };
    const int64_t three = (int64_t)((groups(96, 64) + 255) / 256) * 3, four = (int64_t)((groups(128, 64) + 255) / 256) * 4;
    if (groups(32, 32) <= 2048) attn_bwd_db2_kernel<2, 1><<<grid(64, 32), dim3(128), 0, stream>>>(p);
    else if (4 * four > 5 * three) attn_bwd_db2_kernel<3, 2><<<grid(96, 64), dim3(192), 0, stream>>>(p);
    else attn_bwd_db2_kernel<4, 2><<<grid(128, 64), dim3(256), 0, stream>>>(p);
  } else {
    const dim3 grid(groups(64, 64));
    if ((p.s & 7) == 0) attn_bwd_db2_fp32_kernel<true><<<grid, dim3(256), 0, stream>>>(p);
    else attn_bwd_db2_fp32_kernel<false><<<grid, dim3(256), 0, stream>>>(p);
  }
}

template <typename T>
static void db2_sum(const BwdParams& p, int slices, hipStream_t stream) {
  const int64_t n = (int64_t)p.heads * p.s * p.s;
  const bool vec = n % 4 == 0 && (uintptr_t)p.db2 % (4 * sizeof(T)) == 0 && (uintptr_t)p.parts % 16 == 0;
  const unsigned blocks = (unsigned)((n / (vec ? 4 : 1) + 255) / 256);
  if (vec) attn_bwd_db2_sum_kernel<T, 4><<<dim3(blocks), dim3(256), 0, stream>>>(p.parts, (T*)p.db2, slices, n);
  else attn_bwd_db2_sum_kernel<T, 1><<<dim3(blocks), dim3(256), 0, stream>>>(p.parts, (T*)p.db2, slices, n);
}

template <typename T>
int triattn_bwd(const void* q, const void* k, const void* v, const void* b1, const void* b2,
                const void* o, const float* lse, const void* dout, void* dq, void* dk, void* dv,
                void* db2, float* delta, float* parts, int n_rows, int s, int heads, hipStream_t stream) {
  if (n_rows == 0 || s == 0 || heads == 0) return 0;
  const int slices = parts && db2 ? triattn_bwd_slices(n_rows, s, heads, sizeof(T) == 2) : 1;
  BwdParams p = {q, k, v, o, dout, b1, b2, lse, delta, dq, dk, dv, db2, n_rows, s, heads, slices > 1 ? parts : nullptr, slices};
  const dim3 walk(((unsigned)((s + 127) / 128) * heads * n_rows + 7) / 8 * 8);
  const bool joint = rows_at_once<T>(p);
  if constexpr (sizeof(T) == 2) if (joint) {
    const dim3 grid(((unsigned)heads * n_rows + 7) / 8 * 8);
    if (s <= 128) attn_bwd_row_kernel<4, 1><<<grid, dim3(256), 0, stream>>>(p);
    else if (s <= 256) attn_bwd_row_kernel<4, 2><<<grid, dim3(256), 0, stream>>>(p);
    else if (s <= 384) attn_bwd_row_kernel<4, 3><<<grid, dim3(256), 0, stream>>>(p);
    else if (s <= 512) attn_bwd_row_kernel<8, 2><<<grid, dim3(512), 0, stream>>>(p);
    else attn_bwd_row_kernel<8, 3><<<grid, dim3(512), 0, stream>>>(p);
  }
  if (!joint) {
    if ((s & 7) == 0) {
      attn_bwd_dq_kernel<T, true><<<walk, dim3(256), 0, stream>>>(p);   // (writes Delta: first)
      attn_bwd_kv_kernel<T, true><<<walk, dim3(256), 0, stream>>>(p);
    } else {
      attn_bwd_dq_kernel<T, false><<<walk, dim3(256), 0, stream>>>(p);
      attn_bwd_kv_kernel<T, false><<<walk, dim3(256), 0, stream>>>(p);
    }
  }
  if (db2) db2_walk<T>(p, stream);
  if (slices > 1) db2_sum<T>(p, slices, stream);
  return 0;
}

template int triattn_bwd<float>(const void*, const void*, const void*, const void*, const void*,
                                const void*, const float*, const void*, void*, void*, void*, void*,
                                float*, float*, int, int, int, hipStream_t);
template int triattn_bwd<bf16_t>(const void*, const void*, const void*, const void*, const void*,
                                 const void*, const float*, const void*, void*, void*, void*, void*,
                                 float*, float*, int, int, int, hipStream_t);

}  // namespace ptx
