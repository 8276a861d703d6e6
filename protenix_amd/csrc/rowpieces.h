// Helpers of the kernels in which a workgroup shares a tile of pair-tensor rows (pairproj.hip,
// transition_small.hip): rows read in whole lines by 8 lanes each, normalised rows parked in LDS as
// MFMA operand fragments, packed weight fragments straight from memory, updates collected in LDS and
// added to the raw rows in registers.
#pragma once
#include "common.h"
#include "rowtile.h"

namespace ptx {

// ---- normalised rows in LDS -------------------------------------------------------------
// Row block rb, 8-channel group c8, 16-byte piece: one plane of 32 rows x 16 bytes.  A fragment
// read (K step kk: groups 2 kk + lane / 32, lane % 32 = row) is two contiguous halves of planes;
// the plane pitch spreads the writes (8 neighbouring lanes hold 8 groups of one row).
constexpr int kPlanePitch = 32 * 16 + 32;
template <typename T, int KS> struct FragLds {
  static constexpr int PIECES = (int)sizeof(T) / 2;
  static constexpr int ROWBLOCK = 2 * KS * PIECES * kPlanePitch;   // bytes per 32 rows
  static __device__ __forceinline__ void put(char* base, int rb, int row, int c8, typename Vec8<T>::type v) {
    const u32x4_t* s = reinterpret_cast<const u32x4_t*>(&v);
    char* d = base + rb * ROWBLOCK + c8 * PIECES * kPlanePitch + row * 16;
#pragma unroll
    for (int pc = 0; pc < PIECES; ++pc) *reinterpret_cast<u32x4_t*>(d + pc * kPlanePitch) = s[pc];
  }
  static __device__ __forceinline__ typename Vec8<T>::type get(const char* base, int rb, int kk, int lane) {
    typename Vec8<T>::type v;
    u32x4_t* d = reinterpret_cast<u32x4_t*>(&v);
    const char* s = base + rb * ROWBLOCK + (2 * kk + (lane >> 5)) * PIECES * kPlanePitch + (lane & 31) * 16;
#pragma unroll
    for (int pc = 0; pc < PIECES; ++pc) d[pc] = *reinterpret_cast<const u32x4_t*>(s + pc * kPlanePitch);
    return v;
  }
};

// Fragment `f` of a packed weight set: [fragment][16-byte piece][lane].
template <typename T>
__device__ __forceinline__ typename Vec8<T>::type packed_frag(const T* packed, int f, int lane) {
  constexpr int PIECES = (int)sizeof(T) / 2;
  typename Vec8<T>::type v;
  u32x4_t* d = reinterpret_cast<u32x4_t*>(&v);
  const u32x4_t* s = reinterpret_cast<const u32x4_t*>(packed + (int64_t)f * kFragElems) + lane;
#pragma unroll
  for (int pc = 0; pc < PIECES; ++pc) d[pc] = s[pc * kWave];
  return v;
}

// A row in 8 neighbouring lanes: lane j holds the 16-byte pieces j, j + 8, .. of the stored row (PE
// channels each), so that every access covers whole 128-byte lines.
template <typename TZ, int KS> struct RowPieces {
  static constexpr int PE = 16 / (int)sizeof(TZ);
  static constexpr int NP = 16 * KS / (8 * PE);   // pieces per lane
  typedef typename VecE<TZ>::type V;
};

// LayerNorm of such a row (statistics in fp32, two passes) with this lane's gamma / beta.
template <int PE, int NP>
__device__ __forceinline__ void normalize_pieces(float (&v)[NP][PE], const float (&gm)[NP][PE], const float (&bt)[NP][PE], float eps) {
  float s = 0.0f;
#pragma unroll
  for (int q = 0; q < NP; ++q)
#pragma unroll
    for (int t = 0; t < PE; ++t) s += v[q][t];
  const float mean = lane_group_sum<8>(s) * (1.0f / (8 * NP * PE));
  float d2 = 0.0f;
#pragma unroll
  for (int q = 0; q < NP; ++q)
#pragma unroll
    for (int t = 0; t < PE; ++t) {
      const float d = v[q][t] - mean;
      d2 += d * d;
    }
  const float rstd = rsqrtf(lane_group_sum<8>(d2) * (1.0f / (8 * NP * PE)) + eps);
#pragma unroll
  for (int q = 0; q < NP; ++q)
#pragma unroll
    for (int t = 0; t < PE; ++t) v[q][t] = (v[q][t] - mean) * rstd * gm[q][t] + bt[q][t];
}

template <typename T, int PE, int NP>
__device__ __forceinline__ void load_affine_pieces(const T* gamma, const T* beta, int j, float (&gm)[NP][PE], float (&bt)[NP][PE]) {
  const T* gp = (gamma ? gamma : default_gamma<T>()) + PE * j;
  const T* bp = (beta ? beta : default_beta<T>()) + PE * j;
#pragma unroll
  for (int q = 0; q < NP; ++q)
#pragma unroll
    for (int e = 0; e < PE; e += 4) {
      const f32x4 g4 = to_f32(*reinterpret_cast<const typename Vec4<T>::type*>(gp + 8 * PE * q + e));
      const f32x4 b4 = to_f32(*reinterpret_cast<const typename Vec4<T>::type*>(bp + 8 * PE * q + e));
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        gm[q][e + t] = g4[t];
        bt[q][e + t] = b4[t];
      }
    }
}

// Piece (PE values) number c / PE of a row into the fragment tile, rounded to T.
template <typename T, int KS, int PE>
__device__ __forceinline__ void put_piece(char* frag, int rb, int row, int piece, const float (&v)[PE]) {
  if constexpr (PE == 8) {
    f32x8 f;
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] = v[t];
    FragLds<T, KS>::put(frag, rb, row, piece, from_f32<T>(f));
  } else {
    const typename Vec4<T>::type h = from_f32<T>(f32x4{v[0], v[1], v[2], v[3]});
    char* d = frag + rb * FragLds<T, KS>::ROWBLOCK;
    if constexpr (sizeof(T) == 2)   // half of a group's 16 bytes
      *reinterpret_cast<typename Vec4<T>::type*>(d + (piece >> 1) * kPlanePitch + row * 16 + 8 * (piece & 1)) = h;
    else
      *reinterpret_cast<typename Vec4<T>::type*>(d + piece * kPlanePitch + row * 16) = h;
  }
}

// The tile's rows, normalised, into LDS; the raw pieces stay in `raw` (row rb * 32 + 8 * wave + lane / 8).
// off(r): element offset of row r of the tile.
template <typename T, typename TZ, int KS, int RBW, typename Off>
__device__ __forceinline__ void norm_rows(char* frag, const TZ* x, Off off, const T* gamma, const T* beta, float eps,
                                          int wave, int lane,
                                          typename RowPieces<TZ, KS>::V (&raw)[RBW][RowPieces<TZ, KS>::NP]) {
  typedef RowPieces<TZ, KS> RP;
  constexpr int PE = RP::PE, NP = RP::NP;
  const int j = lane & 7, r8 = wave * 8 + (lane >> 3);
#pragma unroll
  for (int rb = 0; rb < RBW; ++rb) {
    const TZ* rp = x + off(rb * 32 + r8) + PE * j;
#pragma unroll
    for (int q = 0; q < NP; ++q) raw[rb][q] = *reinterpret_cast<const typename RP::V*>(rp + 8 * PE * q);
  }
  float gm[NP][PE], bt[NP][PE];
  load_affine_pieces<T, PE, NP>(gamma, beta, j, gm, bt);
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

// The update of the tile's rows (T, [32 RBW][16 KS] at a pitch of kUpdPitch<KS>) added to the raw rows norm_rows() left
// in registers (or stored as it is) and written in the same layout: whole lines.  `raw` then holds the rows as stored.
template <int KS> constexpr int kUpdPitch = 16 * KS + 8;
template <typename T, typename TZ, int KS, int RBW, typename Off>
__device__ __forceinline__ void store_rows(TZ* out, Off off, const T* upd, int wave, int lane, int add,
                                           typename RowPieces<TZ, KS>::V (&raw)[RBW][RowPieces<TZ, KS>::NP]) {
  typedef RowPieces<TZ, KS> RP;
  constexpr int PE = RP::PE, NP = RP::NP;
  const int j = lane & 7, r8 = wave * 8 + (lane >> 3);
#pragma unroll
  for (int rb = 0; rb < RBW; ++rb) {
    const int64_t o = off(rb * 32 + r8);
    const T* up = upd + (rb * 32 + r8) * kUpdPitch<KS> + PE * j;
    if (o >= 0) {
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        typename RP::V v;
#pragma unroll
        for (int e = 0; e < PE; e += 4) {
          const f32x4 u = to_f32(*reinterpret_cast<const typename Vec4<T>::type*>(up + 8 * PE * q + e));
#pragma unroll
          for (int t = 0; t < 4; ++t) v[e + t] = from_f32<TZ>(add ? to_f32(raw[rb][q][e + t]) + u[t] : u[t]);
        }
        *reinterpret_cast<typename RP::V*>(out + o + PE * j + 8 * PE * q) = v;
        raw[rb][q] = v;
      }
    }
  }
}

// One 32 x 32 result tile (lane <-> row, register <-> column) into the update's tile.
template <typename T, int KS>
__device__ __forceinline__ void put_update(T* upd, int rb, int ob, const float (&vals)[16], int lane) {
  T* d = upd + (rb * 32 + (lane & 31)) * kUpdPitch<KS> + ob * 32 + 4 * (lane >> 5);
#pragma unroll
  for (int qd = 0; qd < 4; ++qd)
    *reinterpret_cast<typename Vec4<T>::type*>(d + 8 * qd) =
        from_f32<T>(f32x4{vals[4 * qd], vals[4 * qd + 1], vals[4 * qd + 2], vals[4 * qd + 3]});
}

// Workgroups are dealt round-robin to the 8 XCDs: runs of four neighbouring tiles go to one XCD, whose L2
// then sees both halves of the 128-byte lines that two tiles of 32 16-bit values share.
__device__ __forceinline__ uint32_t xcd_run(uint32_t b, uint32_t n) {
  constexpr uint32_t RUN = 4;
  const uint32_t base = b / (8 * RUN) * (8 * RUN), o = b - base;
  return base + 8 * RUN <= n ? base + (o & 7) * RUN + (o >> 3) : b;
}

}  // namespace ptx
