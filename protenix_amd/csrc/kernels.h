// Host-callable launchers, one per kernel family; api.hip validates arguments
// and dispatches on dtype.  c_z / c: channels of a pair-tensor row: 64 or 128 (hidden
// widths - c_hidden_mul, heads * d - of 128), or 256 in bf16 (hidden widths of 256).  All return 0 after enqueueing on `stream`.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ptx {

// T: arithmetic / weight / workspace type.  TZ (where present): storage type of the pair
// tensor rows the kernel reads (z, x) and of the residual stream it writes (out): T, or float
// with T = bf16 (the fp32 residual stream of autocast inference; rows of 64 or 128 channels).
template <typename T>
int layernorm_fwd(const T* x, const T* gamma, const T* beta, T* y, float* mean, float* rstd,
                  int64_t rows, int cols, float eps, hipStream_t stream);
// LayerNorm backward: dx always; dgamma / dbeta when non-null, through `workspace`
// (layernorm_bwd_workspace_elems fp32 elements).
int64_t layernorm_bwd_workspace_elems(int64_t rows, int cols);
template <typename T>
int layernorm_bwd(const T* dout, const T* x, const float* mean, const float* rstd, const T* gamma,
                  T* dx, T* dgamma, T* dbeta, float* workspace, int64_t rows, int cols,
                  hipStream_t stream);

template <typename T, typename TZ = T>
int trimul_project(const void* z, const void* mask, const void* ln_w, const void* ln_b,
                   const void* w_ap, const void* w_ag, const void* w_bp, const void* w_bg, void* a,
                   void* b, int n, int c_z, int k_pitch, int incoming, float eps,
                   hipStream_t stream);
template <typename T, typename TZ = T>
int trimul_output(const void* x, const void* z, const void* ln_in_w, const void* ln_in_b,
                  const void* ln_out_w, const void* ln_out_b, const void* w_z, const void* w_g,
                  void* out, int n, int c_z, int add_residual, float eps, hipStream_t stream);
template <typename T, typename TZ = T>
int triattn_project(const void* z, const void* ln_w, const void* ln_b, const void* w_q,
                    const void* w_k, const void* w_v, const void* w_g, const void* w_b, void* q,
                    void* k, void* vt, void* g, void* tri_bias, int n, int c_z, int heads, int d,
                    int key_pitch, int transposed, float eps, hipStream_t stream);
template <typename T, typename TZ = T>
int triattn_output(const void* o, const void* w_o, const void* z, void* out, int n, int c_z,
                   int transposed, int add_residual, hipStream_t stream);
// out = [z +] W_o (sigmoid(W_g LN(z)) * o) on rows of 128 channels, 4 heads, 16-bit arithmetic:
// the last stage of the triangle attention with the gate formed here (o ungated, head-major).
template <typename TZ>
int triattn_gate_output(const void* o, const void* z, const void* ln_w, const void* ln_b,
                        const void* w_g, const void* w_o, void* out, int n, int transposed,
                        int add_residual, float eps, hipStream_t stream);
// transition weights -> fragment-ordered chunks of 32 hidden (3 * n_factor*c * c elements)
template <typename T>
int transition_pack(const void* w_a, const void* w_b, const void* w_o, void* packed, int c,
                    int n_factor, hipStream_t stream);
template <typename T, typename TZ = T>
int transition_fwd(const void* x, const void* ln_w, const void* ln_b, const void* packed,
                   void* out, int64_t rows, int c, int n_factor, int add_residual, float eps,
                   hipStream_t stream);
struct SingleStage;
// The transition on rows of 128 channels (16-bit arithmetic) with the pair bias of the single
// attention, bias[h][row] = (W LN_pb(out[row]))[h], formed from the finished rows in its epilogue.
template <typename T, typename TZ = T>
int transition_pair_bias_fwd(const void* x, const void* ln_w, const void* ln_b, const void* packed,
                             void* out, int64_t rows, int n_factor, int add_residual, float eps,
                             const void* pb_ln_w, const void* pb_ln_b, const void* pb_w,
                             void* bias, int heads, int bias_f32, float pb_eps,
                             hipStream_t stream);
// The last stage of a triangle attention (as triattn_gate_output, residual added) and the pair
// transition that follows it (as transition_fwd / transition_pair_bias_fwd, residual added) in
// one launch on rows of 128 channels, 16-bit arithmetic: out = z' + transition(z'),
// z' = z + W_o (sigmoid(W_g LN_att(z)) * o).  `packed` holds both stages' weights
// (triattn_output_transition_pack); pb_w null: no pair bias.
int64_t triattn_output_transition_packed_elems(int n_factor);
template <typename T>
int triattn_output_transition_pack(const void* w_g, const void* w_o, const void* w_a,
                                   const void* w_b, const void* w_to, void* packed, int n_factor,
                                   hipStream_t stream);
template <typename T, typename TZ = T>
int triattn_output_transition_fwd(const void* o, const void* z, const void* att_ln_w,
                                  const void* att_ln_b, const void* packed, const void* ln_w,
                                  const void* ln_b, void* out, int n, int transposed, int n_factor,
                                  float att_eps, float eps, const void* pb_ln_w, const void* pb_ln_b,
                                  const void* pb_w, void* bias, int heads, int bias_f32, float pb_eps,
                                  hipStream_t stream, const SingleStage* carry = nullptr);
// Whether that launch, with a pair bias, runs a carried stage along its own workgroups (else in front).
bool transition_carries(int64_t n_rows);
template <typename T, typename TZ = T>
int pair_bias_fwd(const void* z, const void* ln_w, const void* ln_b, const void* w, void* bias,
                  int n, int c_z, int heads, int out_f32, float eps, hipStream_t stream);

// One stage of the single-representation track (single_stage.h): filled by the functions below, run by single_stage_run
// in a launch of its own or carried by one of the pp_* launches.
enum { kStageNone = 0, kStageLinear = 1, kStageSwiGLU = 2, kStageAttention = 3, kStageLayerNorm = 4 };
struct SingleStage {
  int kind, n_work;       // n_work workgroups
  int packed;             // linear: w, w2 in fragment order (single_stage.h; n_out % 16 == 0, k % 32 == 0)
  int tile, row_blocks;   // linear: tiles of 16 x 16, 16 x 32, 32 x 32 (1, 2, 3); tiles over the rows
  int set_shift;          // linear: column tiles go to the XCDs in sets of 1 << set_shift
  int bits16;             // operands bf16, else fp32
  int rows;               // layernorm, linear: rows of x; attention: queries = keys
  const void* x;          // layernorm, linear: [rows][k]; attention: q, rows of pitch ld
  const void* w;          // layernorm: gamma or null; linear: [n_out][k]; attention: k, rows of pitch ld
  const void* w2;         // layernorm: beta or null; SwiGLU: the second matrix; attention: V^T [heads * d][ldt], keys beyond `rows` hold zeros
  const void* bias;       // linear: [bias_cols] or null, added to output columns < bias_cols; attention: [heads][n][n] or null
  const void* res;        // [rows][n_out] or null
  const void* gate;       // attention: gate logits, rows of pitch ld, or null
  void* out;              // rows of pitch ldo: output columns < split_col
  void* out_t;            // [n_out - split_col][ldt]: output columns >= split_col, transposed; rows in [rows, ldt) written as zeros
  int64_t ld, ldo, ldt;
  int k, n_out, split_col, bias_cols;   // split_col: a multiple of 32, or n_out (nothing is transposed)
  int ln_g, ln_nc;        // layernorm: how rows lie over lanes (lnrow.h)
  float eps;
  int heads, d, bias_f32, bias_vec;     // bias_vec: rows of the bias can be read as 16-byte vectors
  float scale;
};
// workgroups a launch gives the stage: whole rounds over the 8 XCDs, so that the others keep their places
inline unsigned single_stage_groups(const SingleStage* s) { return s && s->kind ? (unsigned)(s->n_work + 7) / 8 * 8 : 0u; }
// 0, or -1 where the rows do not fit the stage
int single_stage_layernorm(SingleStage* s, const void* x, const void* gamma, const void* beta, void* y, int rows, int cols,
                           float eps, bool bits16);
void single_stage_linear(SingleStage* s, const void* x, const void* w, const void* w2, const void* bias, int bias_cols,
                         const void* res, void* out, void* out_t, int split_col, int64_t ldt, int rows, int k, int n_out,
                         bool bits16, int packed);
void single_stage_attention(SingleStage* s, const void* q, const void* k, const void* vt, const void* gate, const void* bias,
                            int bias_f32, void* out, int n, int heads, int d, int64_t ld, int64_t ldt, int64_t ldo,
                            float scale, bool bits16);
int single_stage_run(const SingleStage* s, hipStream_t stream);

// x[c][i][j] = sum_k a[c][i][k] * b[c][j][k] for `batch` independent products;
// a, b rows have pitch k_pitch (a multiple of 64, >= n), x is [batch][n][ldx].
// carry: null, or a stage of the single track that the launch's first workgroups run (it must not depend on the launch), where
// nt_gemm_carries(); elsewhere the stage is launched in front.
bool nt_gemm_carries(int n, bool bits16);
template <typename T>
int nt_gemm_batched(const T* a, const T* b, T* x, int n, int ldx, int k_pitch, int batch, const SingleStage* carry, hipStream_t stream);

// A parameter on its way into the kernels (params.hip): src, dst bf16 or fp32 as the flags say, dst [rows][cols] like src or,
// fragments, in the order of a linear stage's packed weights (rows % 16 == 0, cols % 32 == 0).
struct Param {
  const void* src;
  void* dst;
  int64_t rows;
  int cols;
  bool src_bits16, dst_bits16, fragments;
};
int param_pack(const Param* p, int count, hipStream_t stream);

// The row-local stages of the triangle updates on packed weights (pairproj.hip).  carry: null, or a stage of the single
// track on operands of type TZ that this launch's first workgroups run (it must not depend on the launch).
// Whether the attention's gate is formed by the output stage (no gate tensor exists then).
inline bool pp_late_gate(int c_z, int heads, bool bits16) { return bits16 && heads == (c_z == 256 ? 8 : 4); }
// Whether such a stage, with nothing to carry, takes the kernel that holds all of its weights in LDS.
enum RowStage { kTriMulInStage, kTriMulOutStage, kTriAttnInStage, kTriAttnOutStage };
bool pp_resident(RowStage stage, int n, int c_z, int hidden, bool bits16, bool rows16);
int64_t pp_trimul_packed_elems(int c_z, int hidden, bool bits16);
template <typename T>
int pp_trimul_pack(const void* w_ap, const void* w_ag, const void* w_bp, const void* w_bg, const void* w_z,
                   const void* w_g, void* packed, int c_z, int hidden, hipStream_t stream);
int64_t pp_triattn_packed_elems(int c_z, int heads, bool bits16);
template <typename T>
int pp_triattn_pack(const void* w_q, const void* w_k, const void* w_v, const void* w_g, const void* w_b,
                    const void* w_o, void* packed, int c_z, int heads, hipStream_t stream);
template <typename T, typename TZ = T>
int pp_trimul_in(const void* z, const void* mask, const void* ln_w, const void* ln_b, const void* packed, void* a,
                 void* b, int n, int c_z, int k_pitch, int incoming, float eps, const SingleStage* carry, hipStream_t stream);
template <typename T, typename TZ = T>
int pp_triattn_in(const void* z, const void* ln_w, const void* ln_b, const void* packed, void* q, void* k, void* vt,
                  void* g, void* tri_bias, int n, int c_z, int heads, int key_pitch, int transposed, float eps,
                  const SingleStage* carry, hipStream_t stream);
// x [hidden][n][ldx]: ldx = n, or n rounded up to a multiple of 8 (rows of any n then start aligned)
template <typename T, typename TZ = T>
int pp_trimul_out(const void* x, int ldx, const void* z, const void* ln_in_w, const void* ln_in_b,
                  const void* ln_out_w, const void* ln_out_b, const void* packed, void* out, int n, int c_z,
                  int hidden, int add_residual, float eps, const SingleStage* carry, hipStream_t stream);
template <typename T, typename TZ = T>
int pp_triattn_out(const void* o, const void* z, const void* ln_w, const void* ln_b, const void* packed, void* out,
                   int n, int c_z, int heads, int transposed, int add_residual, float eps, const SingleStage* carry,
                   hipStream_t stream);
// Whether a triangle update's output stage and the projection behind it are faster in
// one launch, in 16-bit arithmetic; pair: 0 the outgoing multiplication -> the incoming one, 1 the incoming multiplication -> the
// starting node, 2 the starting -> the ending node.
bool pp_joined(int pair, int n, int c_z, int hidden, bool rows16);
// An output stage and the projection that reads its rows next, in one launch (16-bit arithmetic, residual added; attentions'
// projections write no gate): these pairs.
template <typename TZ>
int pp_trimul_out_trimul_in(const void* x, int ldx, const void* z, const void* mask, const void* ln_in_w, const void* ln_in_b,
                            const void* ln_out_w, const void* ln_out_b, const void* packed, void* out, const void* next_ln_w,
                            const void* next_ln_b, const void* next_packed, void* a, void* b, int n, int c_z, int hidden, int k_pitch,
                            float eps, const SingleStage* carry, hipStream_t stream);
template <typename TZ>
int pp_trimul_out_triattn_in(const void* x, int ldx, const void* z, const void* ln_in_w, const void* ln_in_b, const void* ln_out_w,
                             const void* ln_out_b, const void* packed, void* out, const void* att_ln_w, const void* att_ln_b,
                             const void* att_packed, void* q, void* k, void* vt, void* tri_bias, int n, int c_z, int hidden, int heads,
                             int key_pitch, float eps, const SingleStage* carry, hipStream_t stream);
template <typename TZ>
int pp_triattn_out_triattn_in(const void* o, const void* z, const void* ln_w, const void* ln_b, const void* packed, void* out,
                              const void* next_ln_w, const void* next_ln_b, const void* next_packed, void* q, void* k, void* vt,
                              void* tri_bias, int n, int c_z, int heads, int key_pitch, float eps, const SingleStage* carry,
                              hipStream_t stream);

// Flash-style triangle attention core (see triattn.hip).
template <typename T>
int triattn_fwd(const T* q, const T* k, const T* vt, const T* g, const T* tri_bias, const T* mask,
                T* o, int n, int heads, int key_pitch, int mask_transposed, float inf,
                int row_begin, int row_count, int n_keys, const SingleStage* carry, hipStream_t stream);
// carry: null, or a stage of the single track that the launch's first workgroups run where triattn_fwd_carries(); elsewhere it
// is launched in front.
bool triattn_fwd_carries(int n, bool bits16);
// The same core on n_rows rows of n queries / keys, with q / g / o addressed through element
// strides (head, row, query), an optional gate (g may be null), the mask either 0/1 values or
// (mask_is_bias) an additive bias per (row, key), and an optional log2-sum-exp2 output.
// The launch covers rows row_begin .. row_begin + row_count - 1 and lets keys 0 .. n_keys - 1
// take part (keys beyond count as masked: weight exactly zero).  standard (16-bit): k and vt are K and V addressed by q's
// strides, and q is not yet in log2 units; where triattn_fwd_standard().
bool triattn_fwd_standard(int n_rows, int n, int heads, bool masked);
template <typename T>
int triattn_fwd_ex(const T* q, const T* k, const T* vt, const T* g, const T* tri_bias,
                   const T* mask, T* o, int n_rows, int n, int heads, int key_pitch,
                   int mask_transposed, float inf, int mask_is_bias, int64_t sh, int64_t si,
                   int64_t sj, float* lse, int64_t lh, int64_t li, int64_t lj, int row_begin,
                   int row_count, int n_keys, const SingleStage* carry, hipStream_t stream, bool standard = false);
// Standard-layout K, V [n_rows][n][heads][32] and bias [heads][n][n] -> the core's fragment-
// ordered K, V^T and bias (bias and nothing else multiplied by log2(e)); q [n_rows][n][heads][32]
// -> qs, the same layout multiplied by log2(e).  q = null: the bias only.
template <typename T>
int triattn_pack(const T* q, const T* k, const T* v, const T* bias2, T* qs, T* kf, T* vtf, T* bf,
                 int n_rows, int n, int heads, int key_pitch, hipStream_t stream);
// Backward of the standard-layout attention operator: dQ, dK, dV [n_rows][s][heads][32] and,
// when db2 is given, dBias2 [heads][s][s], from Q (scaled), K, V, O, dO, the biases and the
// forward's log2-sum-exp2; delta [n_rows][s][heads] is fp32 scratch; parts: fp32 scratch of
// triattn_bwd_slices() * heads * s * s elements for the partial sums of dBias2, or null (one slice).
int triattn_bwd_slices(int n_rows, int s, int heads, bool bits16);
template <typename T>
int triattn_bwd(const void* q, const void* k, const void* v, const void* b1, const void* b2,
                const void* o, const float* lse, const void* dout, void* dq, void* dk, void* dv,
                void* db2, float* delta, float* parts, int n_rows, int s, int heads, hipStream_t stream);

// Streams `bytes` (a multiple of 16) from src to dst; src null: write-only, dst null: read-only.
int hbm_stream(const void* src, void* dst, int64_t bytes, int nontemporal, hipStream_t stream);

}  // namespace ptx
