// The transition (and the stages fused with it, see transition.hip) on few rows.
//
// The kernel of transition.hip gives a wave 32 rows and the whole hidden dimension: 16 chunks one
// after the other, 28 us however few the rows.  Here a workgroup takes 32 rows and its four waves split
// the hidden dimension: each walks every fourth chunk of 32 and the partial output tiles
// meet in LDS, added in wave order.  The weights, packed as fragments of 1 KB, go from the L2 straight to
// registers, W_a / W_b of a wave's next chunk under the activation and second product of this
// one: 384 KB per 32 rows, which the L2s deliver at some 28 TB/s, so the form pays as long as that
// stays below what the fused kernel's walk takes (see transition_small at the end).
#include "common.h"
#include "kernels.h"
#include "rowpieces.h"
#include "single_stage.h"
#include "transition.h"
#include <type_traits>

namespace ptx {

constexpr int kTsWaves = 4;

template <typename T, int KS, typename TZ, bool PB, bool AO>
__global__ __launch_bounds__(kTsWaves * 64, (sizeof(T) == 2 && KS <= 8 ? 2 : 1)) void transition_small_kernel(
    const TZ* x, const T* __restrict__ gamma, const T* __restrict__ beta, const T* __restrict__ packed, TZ* out,
    int64_t n_rows, int n_chunks, int add_residual, float eps, PairBiasArgs pb, AttnOutArgs ao, SingleStage carry, unsigned carried) {
  typedef typename Vec8<T>::type V8;
  typedef RowPieces<TZ, KS> RP;
  constexpr int NOB = KS / 2, FRAGS = 3 * KS, kCx = 16 * KS, PE = RP::PE, NP = RP::NP, NW = kTsWaves;
  static_assert(!AO || (KS == 8 && sizeof(T) == 2), "attention-output prologue: rows of 128 channels, 16-bit arithmetic");
  static_assert(!PB || (KS == 8 && sizeof(T) == 2), "pair bias: rows of 128 channels, 16-bit arithmetic");
  constexpr int kFrag = FragLds<T, KS>::ROWBLOCK;
  constexpr int kUpd = (int)sizeof(T) * 32 * kUpdPitch<KS>;
  // the normalised rows, later the update; the partial output tiles, before them the gated attention output
  __shared__ __attribute__((aligned(16))) char frag[kFrag > kUpd ? kFrag : kUpd];
  __shared__ __attribute__((aligned(16))) float part[NW][NOB][16][kWave];
  static_assert(!AO || sizeof(part) >= (size_t)FragLds<T, KS>::ROWBLOCK + kUpd, "the prologue's tiles fit the partial sums' place");
  // The first `carried` workgroups run a stage of the single track (the form that a block with one launches).
  if constexpr (PB && AO) {
    static_assert(!(PB && AO) || sizeof(part) >= kStageLds, "the stage's LDS");
    if (blockIdx.x < carried) {
      single_stage<TZ>(carry, blockIdx.x, reinterpret_cast<char*>(part));
      return;
    }
  }
  const uint32_t block = blockIdx.x - carried, blocks = gridDim.x - carried;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nl = lane & 31, g = lane >> 5, j8 = lane & 7, r8 = wave * 8 + (lane >> 3);
  // (back to front: the kernel before this one wrote the pair tensor front to back)
  const int64_t row0 = (int64_t)(blocks - 1 - xcd_run(block, blocks)) * 32;
  const T* tpacked = packed + (AO ? (int64_t)kAoChunks * FRAGS * kFragElems : 0);
  auto x_row = [&](int r) -> int64_t { return row0 + r < n_rows ? (row0 + r) * kCx : -1; };
  auto x_row0 = [&](int r) -> int64_t { return min(row0 + r, n_rows - 1) * kCx; };

  typename RP::V raw[1][NP];   // the rows (AO: after the attention's update)
  if constexpr (AO) {
    char* fo = reinterpret_cast<char*>(part);
    T* aupd = reinterpret_cast<T*>(fo + FragLds<T, KS>::ROWBLOCK);
    V8 of[2], wg[KS], wo[KS];
    {
      const T* op = (const T*)ao.o + ao.omap(min(row0 + nl, n_rows - 1)) + (int64_t)wave * n_rows * 32 + 8 * g;
#pragma unroll
      for (int u = 0; u < 2; ++u) of[u] = load8<T>(op + 16 * u);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) wg[kk] = packed_frag<T>(packed, 8 * wave + kk, lane);
      norm_rows<T, TZ, KS, 1>(frag, x, x_row0, (const T*)ao.gamma, (const T*)ao.beta, ao.eps, wave, lane, raw);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) wo[kk] = packed_frag<T>(packed, 32 + 8 * wave + kk, lane);
    }
    __syncthreads();
    {
      // gate of head `wave`, as in pp_triattn_out_kernel
      f32x16 ag;
#pragma unroll
      for (int r = 0; r < 16; ++r) ag[r] = 0.0f;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) mma32(ag, wg[kk], FragLds<T, KS>::get(frag, 0, kk, lane));
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const f32x8 ov = to_f32(of[u]);
        f32x8 gated;
#pragma unroll
        for (int t = 0; t < 8; ++t) gated[t] = ov[t] * to_f32(from_f32<T>(sigmoidf_fast(ag[8 * u + t])));
        FragLds<T, KS>::put(fo, 0, nl, 2 * (2 * wave + u) + g, from_f32<T>(gated));
      }
    }
    __syncthreads();
    {
      // output block `wave`: the update, rounded to T (registers 8 u + t <-> channels 16 u + 8 g + t of the block)
      f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) mma32(acc, wo[kk], FragLds<T, KS>::get(fo, 0, kk, lane));
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        f32x8 a8;
#pragma unroll
        for (int t = 0; t < 8; ++t) a8[t] = acc[8 * u + t];
        store8<T>(aupd + nl * kUpdPitch<KS> + 32 * wave + 16 * u + 8 * g, from_f32<T>(a8));
      }
    }
    __syncthreads();
    {
      // x' = x + update as stored, in place of x; its LayerNorm into the fragment tile
      float v[NP][PE], gm[NP][PE], bt[NP][PE];
      load_affine_pieces<T, PE, NP>(gamma, beta, j8, gm, bt);
#pragma unroll
      for (int q = 0; q < NP; ++q)
#pragma unroll
        for (int e = 0; e < PE; ++e) {
          raw[0][q][e] = from_f32<TZ>(to_f32(raw[0][q][e]) + to_f32(aupd[r8 * kUpdPitch<KS> + PE * (j8 + 8 * q) + e]));
          v[q][e] = to_f32(raw[0][q][e]);
        }
      normalize_pieces<PE, NP>(v, gm, bt, eps);
#pragma unroll
      for (int q = 0; q < NP; ++q) put_piece<T, KS, PE>(frag, 0, r8, j8 + 8 * q, v[q]);
    }
  } else {
    norm_rows<T, TZ, KS, 1>(frag, x, x_row0, gamma, beta, eps, wave, lane, raw);
  }

  // this wave's chunks of the hidden dimension
  V8 wa[KS], wb[KS], wo[KS];
  auto load_ab = [&](int j) {
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      wa[kk] = load8<T>(tpacked + ((int64_t)j * FRAGS + kk) * kFragElems + lane * 8);
      wb[kk] = load8<T>(tpacked + ((int64_t)j * FRAGS + KS + kk) * kFragElems + lane * 8);
    }
  };
  auto load_o = [&](int j) {
#pragma unroll
    for (int f = 0; f < KS; ++f) wo[f] = load8<T>(tpacked + ((int64_t)j * FRAGS + 2 * KS + f) * kFragElems + lane * 8);
  };
  const int j_first = min(wave, n_chunks - 1);
  load_ab(j_first);
  load_o(j_first);
  f32x16 acc_o[NOB];
#pragma unroll
  for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc_o[ob][r] = 0.0f;
  __syncthreads();
  for (int j = wave; j < n_chunks; j += NW) {
    const int jn = min(j + NW, n_chunks - 1);   // (past the end: a valid chunk that is not used)
    f32x16 a, b;
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = b[r] = 0.0f;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      const V8 xv = FragLds<T, KS>::get(frag, 0, kk, lane);
      mma32(a, wa[kk], xv);   // lane <-> row, register <-> hidden
      mma32(b, wb[kk], xv);
    }
    load_ab(jn);
    V8 hf[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) hf[r >> 3][r & 7] = from_f32<T>(a[r] * b[r] * sigmoidf_fast(a[r]));
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int ob = 0; ob < NOB; ++ob) mma32(acc_o[ob], wo[2 * ob + u], hf[u]);
    load_o(jn);
  }
#pragma unroll
  for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][ob][r][lane] = acc_o[ob][r];
  __syncthreads();
  // sums in wave order: every wave finishes a quarter of the output registers
  T* upd = reinterpret_cast<T*>(frag);
  constexpr int QUADS = NOB * 4 / NW;   // register quads (4 neighbouring columns) per wave
#pragma unroll
  for (int q = 0; q < QUADS; ++q) {
    const int qq = wave * QUADS + q, ob = qq >> 2, qd = qq & 3;
    f32x4 s;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[e] = part[0][ob][4 * qd + e][lane];
#pragma unroll
      for (int w = 1; w < NW; ++w) s[e] += part[w][ob][4 * qd + e][lane];
    }
    *reinterpret_cast<typename Vec4<T>::type*>(upd + nl * kUpdPitch<KS> + ob * 32 + 8 * qd + 4 * g) = from_f32<T>(s);
  }
  __syncthreads();
  if (!PB) {
    store_rows<T, TZ, KS, 1>(out, x_row, upd, wave, lane, add_residual, raw);
    return;
  }
  if constexpr (PB) {
    // the finished rows, as stored, normalised for the pair bias
    char* fpb = reinterpret_cast<char*>(part);
    {
      const int64_t o = x_row(r8);
      float v[NP][PE], gm[NP][PE], bt[NP][PE];
      load_affine_pieces<T, PE, NP>((const T*)pb.gamma, (const T*)pb.beta, j8, gm, bt);
#pragma unroll
      for (int q = 0; q < NP; ++q) {
        typename RP::V d;
#pragma unroll
        for (int e = 0; e < PE; ++e) {
          const float u = to_f32(upd[r8 * kUpdPitch<KS> + PE * (j8 + 8 * q) + e]);
          d[e] = from_f32<TZ>(add_residual ? to_f32(raw[0][q][e]) + u : u);
          v[q][e] = to_f32(d[e]);
        }
        if (o >= 0) *reinterpret_cast<typename RP::V*>(out + o + PE * (j8 + 8 * q)) = d;
      }
      normalize_pieces<PE, NP>(v, gm, bt, pb.eps);
#pragma unroll
      for (int q = 0; q < NP; ++q) put_piece<T, KS, PE>(fpb, 0, r8, j8 + 8 * q, v[q]);
    }
    V8 wp[KS];   // rows beyond `heads` repeat the last head: not stored
    const T* wrow = (const T*)pb.w + min(nl, pb.heads - 1) * kCx + 8 * g;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) wp[kk] = load8<T>(wrow + 16 * kk);
    __syncthreads();
    {
      f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) mma32(acc, wp[kk], FragLds<T, KS>::get(fpb, 0, kk, lane));   // lane <-> row, register <-> head
      if (row0 + nl < n_rows) {
#pragma unroll
        for (int qd = 0; qd < 4; ++qd)
          if (qd == wave) {   // every wave stores a quarter of the heads
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int head = acc_row(4 * qd + e, g);
              if (head < pb.heads) {
                if (pb.out_f32) ((float*)pb.out)[(int64_t)head * n_rows + row0 + nl] = acc[4 * qd + e];
                else ((T*)pb.out)[(int64_t)head * n_rows + row0 + nl] = from_f32<T>(acc[4 * qd + e]);
              }
            }
          }
      }
    }
  }
}

static bool takes_split(int64_t n_rows, int ks, bool bits16) {
  // us per launch, fused / split (fp32 rows where the arithmetic is 16-bit):
  //   c = 128, 16-bit (with the attention's output and the pair bias): 27.4 / 12.4 at 64^2 rows, 27.6 / 18.9 at 93^2,
  //     28.2 / 20.0 at 128^2, 42.8 / 43.8 at 192^2: the fused kernel is flat up to 256 workgroups of 128 rows
  //   c = 64: 11.5 / 4.4 at 64^2, 11.8 / 5.5 at 128^2, 13.5 / 13.7 at 256^2
  //   c = 128, fp32: 104 / 34 at 64^2, 104 / 66 at 128^2, 209 / 161 at 192^2, 212 / 255 at 256^2, 418 / 410 at 320^2: one
  //     workgroup of the fused kernel per compute unit, whole rounds of 32768 rows; c = 256 likewise: 53 / 25 at
  //     64^2, 56 / 51 at 128^2, 114 / 117 at 192^2, 128 / 185 at 256^2
  // (Eight waves per workgroup: 14.1 at 64^2, 26.8 at 128^2.)
  const double rounds = (double)((n_rows + 32767) / 32768);
  if (!bits16) return 10.0 + 0.0038 * (double)n_rows < 104.0 * rounds;
  if (ks == 16) return 3.0 + 0.003 * (double)n_rows < 56.0 * rounds;
  return n_rows <= (ks == 4 ? 60000 : 21500);
}

// Two workgroups per compute unit: where a stage's (some two hundred of its own, with as much LDS) would make another round they
// are launched apart (128 tokens: a block of 119 us took 125).
bool transition_carries(int64_t n_rows) {
  constexpr int64_t kRound = 512, kStage = 200;
  const int64_t blocks = (n_rows + 31) / 32;
  return takes_split(n_rows, 8, true) && (blocks + kStage + kRound - 1) / kRound == (blocks + kRound - 1) / kRound;
}

template <typename T, int KS, typename TZ, bool PB, bool AO>
bool transition_small(const TZ* x, const T* gamma, const T* beta, const T* packed, TZ* out, int64_t n_rows, int n_chunks,
                      int add_residual, float eps, const PairBiasArgs& pb, const AttnOutArgs& ao, hipStream_t stream, const SingleStage* carry) {
  if (!takes_split(n_rows, KS, sizeof(T) == 2)) return false;
  static const SingleStage none = {};
  if (!carry) carry = &none;
  const unsigned carried = PB && AO ? single_stage_groups(carry) : 0u;
  transition_small_kernel<T, KS, TZ, PB, AO><<<dim3(carried + (unsigned)((n_rows + 31) / 32)), dim3(kTsWaves * 64), 0, stream>>>(
      x, gamma, beta, packed, out, n_rows, n_chunks, add_residual, eps, pb, ao, *carry, carried);
  return true;
}

#define PTX_INSTANTIATE(T, KS, TZ, PB, AO)                                                                            \
  template bool transition_small<T, KS, TZ, PB, AO>(const TZ*, const T*, const T*, const T*, TZ*, int64_t, int, int,  \
                                                    float, const PairBiasArgs&, const AttnOutArgs&, hipStream_t, const SingleStage*);
PTX_INSTANTIATE(float, 4, float, false, false)
PTX_INSTANTIATE(float, 8, float, false, false)
PTX_INSTANTIATE(bf16_t, 4, bf16_t, false, false)
PTX_INSTANTIATE(bf16_t, 4, float, false, false)
PTX_INSTANTIATE(bf16_t, 16, bf16_t, false, false)
PTX_INSTANTIATE(bf16_t, 16, float, false, false)
PTX_INSTANTIATE(bf16_t, 8, bf16_t, false, false)
PTX_INSTANTIATE(bf16_t, 8, float, false, false)
PTX_INSTANTIATE(bf16_t, 8, bf16_t, true, false)
PTX_INSTANTIATE(bf16_t, 8, float, true, false)
PTX_INSTANTIATE(bf16_t, 8, bf16_t, false, true)
PTX_INSTANTIATE(bf16_t, 8, float, false, true)
PTX_INSTANTIATE(bf16_t, 8, bf16_t, true, true)
PTX_INSTANTIATE(bf16_t, 8, float, true, true)
#undef PTX_INSTANTIATE

}  // namespace ptx
