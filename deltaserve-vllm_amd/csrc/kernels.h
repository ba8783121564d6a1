// Internal launch API of the backward's HIP kernels (not part of the C-ABI).
#pragma once

#include "../../include/dsb.h"
#include "dsb_common.h"

namespace dsb {

// ---- norm_rope.hip
hipError_t rmsnorm_fwd(const bf16* x, long ldx, const bf16* w, bf16* y, long ldy, int rows,
                       const int* rows_dev, int D, float eps, hipStream_t s);
// out = bf16(o), o = rmsnorm_backward(x, g, w) + (resid | resid32), and the
// fp32 o into out32 when set (resid and resid32 share the row stride ldr,
// out and out32 the row stride ldo). An fp32 g may be gparts planes, gplane
// elements apart, whose sum is the gradient.
hipError_t rmsnorm_bwd(const bf16* x, long ldx, const void* g, bool g_f32, long ldg,
                       const bf16* w, const bf16* resid, long ldr, bf16* out, long ldo,
                       int rows, const int* rows_dev, int D, float eps, hipStream_t s,
                       const float* resid32 = nullptr, float* out32 = nullptr, int gparts = 1,
                       long gplane = 0);
hipError_t rope_table(const int* pos, int n, const int* n_dev, const float* inv_freq,
                      int half, float* cosb, float* sinb, hipStream_t s);
// q heads of a row at in / pre (row stride ldin / ldp); k heads at ink / prek
// (stride ldk / ldpk), by default right after the q heads of the same row.
// hd: head_dim, 128 or 64 (cos/sin rows of hd/2).
hipError_t rope_fwd(const bf16* in, long ldin, bf16* out, long ldout, const float* cosb,
                    const float* sinb, int n, const int* n_dev, int Hq, int Hkv, int hd,
                    const bf16* qn_w, const bf16* kn_w, float eps, hipStream_t s,
                    const bf16* ink = nullptr, long ldk = 0);
hipError_t rope_bwd(bf16* g, long ldg, const bf16* pre, long ldp, const float* cosb,
                    const float* sinb, int n, const int* n_dev, int Hq, int Hkv, int hd,
                    const bf16* qn_w, const bf16* kn_w, float eps, hipStream_t s,
                    const bf16* prek = nullptr, long ldpk = 0, const float* kv_part = nullptr,
                    int hs = 1);
hipError_t swiglu_h(const bf16* gu, long ldgu, bf16* h, long ldh, int n, const int* n_dev,
                    int I, hipStream_t s);

// ---- attention.hip
// Packed varlen causal GQA attention, head_dim 128 or 64. `tiles` holds one int4
// (seq_start, seq_len, tile_start, 0) per 128-token tile of every sequence;
// `ntiles_dev` is the live tile count (grid is sized for `max_tiles`).
struct AttnArgs {
  const bf16* q; long ldq;   // [n, Hq*hd] (post-RoPE)
  const bf16* k; long ldk;   // [n, Hkv*hd] (post-RoPE)
  const bf16* v; long ldv;   // [n, Hkv*hd]
  bf16* ctx; long ldc;       // fwd out [n, Hq*hd]
  float* o32;                // fwd out fp32 copy of ctx, ld = ldo32; null: none
  long ldo32;
  bf16* ores;                // fwd out bf16(O − bf16(O)), the rounding residual of
                             // ctx (ld = ldc); dsum then takes O = ctx + ores.
                             // With neither copy dsum takes O from the bf16 ctx.
  float* lse;                // [Hq, ld_stat] log2-domain row log-sum-exp
  float* dsum;               // [Hq, ld_stat] rowsum(dO ∘ O), written by attn_dsum
  long ld_stat;
  const bf16* dout; long lddo;  // bwd in: grad of ctx
  bf16* dq; long lddq;       // bwd out
  bf16* dk; long lddk;
  bf16* dv; long lddv;
  const int4* tiles;          // {start, L, t0, 0} per 128-row tile, heaviest query tile first
  const int4* tiles_k;        // the same tiles, heaviest key tile first (dK/dV pass)
  const int* ntiles_dev;
  int max_tiles;
  int Hq, Hkv;
  int hd = 128;                          // head_dim: 128 or 64
  float scale = 0.08838834764831845f;    // 1/sqrt(hd)
  const int* n_dev;  // live token count (the dK/dV head-split sum reads it)
  int n;
  // fp32 workspace for the dK/dV pass's head split (null: none), at least
  // (Hq / Hkv) · n · 2 · Hkv·hd floats when the split applies
  float* kv_part = nullptr;
  long kv_part_elems = 0;
  bool kv_defer = false;  // the caller adds a head split's partials (rope_bwd)
};
hipError_t attn_fwd(const AttnArgs& a, hipStream_t s);
hipError_t attn_bwd(const AttnArgs& a, hipStream_t s);  // attn_dsum, dQ, dK/dV in order
// dsum for every live row and q-head; the dQ and dK/dV passes read it
hipError_t attn_dsum(const AttnArgs& a, hipStream_t s);
hipError_t attn_bwd_dkdv(const AttnArgs& a, hipStream_t s);
// q-head slices the dK/dV pass splits into (1: none) when kv_part_elems
// holds the partials; attn_bwd_dkdv takes the split when kv_part is set
int attn_dkdv_head_split(const AttnArgs& a);
hipError_t attn_bwd_dq(const AttnArgs& a, hipStream_t s);

// ---- lora.hip
struct CastJob {
  const float* src;
  bf16* dst;
  int rows, cols;   // source shape
  int ld_src, ld_dst;
  int transpose;    // dst[c, r] = src[r, c]
  float scale;
  float clamp;      // > 0: clamp the scaled value to [-clamp, clamp] before the cast
};
hipError_t lora_cast(const CastJob* jobs_dev, const int2* chunks_dev, int nchunks,
                     hipStream_t s);
// Z[t, j] = sum_k X[t, k] · B[j, k] for t < n, j < R; bf16 out.
struct SkinnyArgs {
  const bf16* X; long ldx;
  const bf16* B; long ldb;
  int R, K;
  bf16* Z; long ldz;
  int n; const int* n_dev;
  // fp32 workspace of part_elems floats for a K split (null: no split)
  float* part = nullptr;
  long part_elems = 0;
};
// K slices for a (1: none): short token ranges whose blocks would leave most
// CUs idle split K when part_elems holds slices · n · R partials; lora_skinny
// takes the split when a.part is set
int lora_skinny_split(const SkinnyArgs& a);
hipError_t lora_skinny(const SkinnyArgs& a, hipStream_t s);
// Up to kSkinnyBatch independent products of one n and R: one launch where they take the
// same block shape and none splits K, else one after the other.
constexpr int kSkinnyBatch = 3;
hipError_t lora_skinny(const SkinnyArgs* a, int count, hipStream_t s);
// out[j, c] (or out[c, j] when transposed) = scale · sum_t P[t, j] * X[t, c],
// t < n. Output rows j are split into groups of `rg` written to outs[j / rg].
struct TnArgs {
  const bf16* P; long ldp;
  const bf16* X; long ldx;
  int R, C;
  int n; const int* n_dev;
  float* work;     // [nsplit, C, R]
  int nsplit;
  float* outs[3];
  int rg;
  int transpose_out;
  float scale;
  // rows of each group that are stored (0: rg) and, transposed, the output
  // row pitch: a rank padded to a multiple of 8 stores only the adapter's r
  int rv = 0;
};
hipError_t lora_tn(const TnArgs& a, hipStream_t s);
// Up to kTnBatch TN passes (each its own P, X, R, C, outputs and work region;
// one token-split count) in one launch plus one reduction launch.
constexpr int kTnBatch = 12;
struct TnBatch {
  TnArgs a[kTnBatch];
  int count;
  int b0[kTnBatch + 1];
  long r0[kTnBatch + 1];
};
hipError_t lora_tn_batch(const TnArgs* a, int count, hipStream_t s);
// One pass over G [n, C] for the two rank-r products that read it
// (ops.py:142 grad_Z = gy @ (s·B) and ops.py:144 grad_B = s · gy.t() @ Z):
//   Y[t, j] = bf16(sum_c G[t, c]·W[j, c])          (W = (s·B)ᵀ [R2, C])
//   out[c, j] = scale · sum_t P[t, j]·G[t, c]      (P = Z [n, R1], out = grad_B)
// The same pass serves grad_A = grad_Zᵀ·h with Z = h·Aᵀ (W = A, P = grad_Z,
// out[j, c] when transpose_out = 0).
// R1 = 16·RB1 and R2 = 16·RB2 with RB1, RB2 in {1, 2}; C a multiple of 8.
// work holds ceil(C/512)·n_alloc·R2 + nsplit·C·R1 floats.
struct DualArgs {
  const bf16* X; long ldx;  // G
  const bf16* P; long ldp;  // Z
  const bf16* W; long ldw;  // (s·B)ᵀ
  int R1, R2, C;
  int n; const int* n_dev;
  int n_alloc;              // row stride of the Y partials (n <= n_alloc)
  int nsplit;
  float* work;
  bf16* Y; long ldy;
  float* out; float scale;  // out[c, j] (row pitch rv), or out[j, c] when !transpose_out
  int transpose_out;
  int rv = 0;               // rows j < rv are stored (0: R1)
};
// Up to 3 passes with the same R1, R2, n and nsplit in one launch (plus one
// launch for all their reductions); each a[i].work is its own region.
hipError_t lora_dual(const DualArgs* a, int count, hipStream_t s);
bool lora_dual_supported(int R1, int R2, int C);

// ---- head.hip
// Of a run of vocabulary columns of one row, the target column left out: the
// softmax reference, Σ exp(logit − ref) and the same sum of bf16-rounded terms.
struct CEStat {
  float ref, sum, rsum;
};
struct HeadArgs {
  const bf16* normed; long ldh;   // [n, D]
  const bf16* W;                  // [V, D]
  const int64_t* ids;             // [n] token ids
  const int* pred;                // [n] 1 where row t predicts ids[t + 1]
  int* err;                       // bit 1: a target id outside [0, V)
  int* labels;                    // [n] target id or -1 (head_init)
  int n; const int* n_dev;
  int D, V;
  CEStat* stats;                  // [n_cap, ntn] per run of ce_bn columns
  int ntn;                        // ceil(V / ce_bn)
  int ce_bn, ce_cfg;              // run width and tile of the logits product (head_plan)
  int dh_cfg, dh_ks;              // tile and K slices of the dH product (head_plan)
  float* tgt_logit;               // [n_cap] from the logits product
  float* lse;                     // [n_cap] row LSE (natural log), after the last chunk
  float* run_m;                   // [n_cap] the row's softmax reference M
  float* run_l;                   // [n_cap] running Σ exp(logit − run_m), target left out
  float* run_r;                   // [n_cap] the same sum of P as stored (bf16)
  float* alpha;                   // [n_cap] the dH accumulator's factor for the chunk
  float* loss_row;                // [n_cap]
  float* loss_out;                // scalar: sum(loss_row)/n_valid
  const float* inv_nvalid;        // device scalar 1/n_valid (0 when none)
  bf16* dlog; int vchunk;         // [n_cap, vchunk] bf16 probabilities of one product
                                  // pair's columns; vchunk a multiple of 256
  float* dH;                      // [n, D] fp32
  // head_part_elems floats when dh_ks > 1: the dH product's accumulators, one
  // per K slice, live from the first chunk to the finalize
  float* part = nullptr;
  float* tail_part = nullptr;     // partials of a tail split of the dH product (null: none)
  long tail_elems = 0;
  int ncu = 0;                    // compute units (tail split; 0: none)
};
// Tiles, K slices and the statistics' layout for a's n, D, V and vchunk
// (gemm_cfg: forced tile of the dH product, -1 by cost; can_split: a.part will
// be provided); then head_init (after
// the final norm), per chunk c0 (a multiple of vchunk) head_prob (logits,
// statistics and probabilities), head_rescale (softmax reference) and
// head_chunk_dh (dH·α + P·W), and head_finalize after the last (dH, LSE, loss).
void head_plan(HeadArgs& a, int gemm_cfg, bool can_split);
long head_part_elems(const HeadArgs& a);
int head_num_chunks(const HeadArgs& a);
// Vocabulary chunks per logits / dH product pair where the chunk width is the default
int head_group(int n, int V, int vchunk);
hipError_t head_fwd_bwd(const HeadArgs& a, hipStream_t s);
hipError_t head_init(const HeadArgs& a, hipStream_t s);
hipError_t head_prob(const HeadArgs& a, int c0, hipStream_t s);
hipError_t head_rescale(const HeadArgs& a, int c0, hipStream_t s);
hipError_t head_chunk_dh(const HeadArgs& a, int c0, hipStream_t s);
hipError_t head_finalize(const HeadArgs& a, hipStream_t s);
// K splits over the tiles of the dH product's partly filled last round (1: none)
int head_dh_tail(const HeadArgs& a, int c0, int* tail);

// ---- optim.hip
struct OptTensor {
  float* w;
  float* g;
  float* m;
  float* v;
  int numel;
  int layer;
};
struct OptHyper {
  float lr, beta1, beta2, eps, wd, bc1, bc2, max_norm;
};
hipError_t clip_adamw(const OptTensor* tensors_dev, const int2* chunks_dev, int nchunks,
                      const int2* layer_chunks_dev, int nlayers, float* partial,
                      float* sq_layer, const OptHyper* hyper_dev, int do_clip, hipStream_t s);

// ---- capture.hip (forward-side save into the activation store)
hipError_t save_rows(const void* x, long ldx, const void* r, long ldr, long x_rows, int dtype,
                     const int64_t* src, const int64_t* dst, int count, int width, bf16* buf,
                     long ldbuf, long buf_rows, hipStream_t s);
hipError_t save_ids(const int64_t* ids, long ids_len, const int64_t* src, const int64_t* dst, int count,
                    int64_t* out, long out_len, hipStream_t s);

}  // namespace dsb
