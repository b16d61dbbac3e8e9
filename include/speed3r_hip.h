/*
 * speed3r_hip.h -- C ABI of the MI355X (gfx950) implementation of Speed3R's global
 * top-k block-sparse attention path.
 *
 * The reference implements this path in Python + Triton and has no FFI of its own; each
 * entry point below replaces the Python-level call named in its comment (paths relative to
 * the reference root).  All tensors are device pointers; strides are in ELEMENTS; the last
 * (head_dim) stride of every q/k/v/o tensor is 1.  Launches are asynchronous on `stream`
 * (a hipStream_t passed as void*; NULL = the default stream).  Every function returns
 * S3R_OK or a negative error code and never throws; s3r_last_error() gives the message of
 * the calling thread's last failure.  No entry point allocates memory.  State kept between calls: the
 * S3R_B16_KERNEL environment switch (read once, on first use) and the built-in score buffer of
 * s3r_compressed_attn_topk_static; nothing else.
 */
#ifndef SPEED3R_HIP_H
#define SPEED3R_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* element types of q/k/v/o/gate tensors ("I/O dtype") */
#define S3R_F32 0
#define S3R_BF16 1
#define S3R_F16 2

#define S3R_OK 0
#define S3R_ERR_BAD_ARG (-1)     /* null pointer, non-positive size, misaligned pointer/stride */
#define S3R_ERR_UNSUPPORTED (-2) /* shape/dtype outside what the kernels are built for */
#define S3R_ERR_HIP (-3)         /* a HIP runtime call or launch failed */

/* Library identification, e.g. "speed3r_hip 0.1 gfx950". */
const char* s3r_version(void);
/* Message of the calling thread's most recent failing call ("" if none). */
const char* s3r_last_error(void);
/* Bit set of optional features built into this library. */
#define S3R_CAP_FUSED_TOPK 1 /* s3r_compressed_attn_topk selects without a scores buffer */
int s3r_capabilities(void);

/*
 * Block mean-pooling: y[b,h,j,:] = mean over tokens [j*block, min((j+1)*block, N)) of x[b,h,t,:].
 * Replaces F.avg_pool1d(kernel=stride=block) in pi3/models/layers/sparse_attention.py:97-99
 * (applied there to the packed qkv; pass H = 3*heads with the packed strides to pool all
 * three at once).  fp32 accumulation, result rounded to `dtype`.  y is [B,H,ceil(N/block),D]
 * with its own strides.  A ragged tail block is a mean over its valid tokens.
 * Requires D*sizeof(elt) to be a power-of-two multiple of 16 bytes up to 1024, and 16-byte
 * aligned pointers/strides.
 */
int s3r_pool_mean(const void* x, void* y, int B, int H, int64_t N, int D, int block,
                  int64_t sxb, int64_t sxh, int64_t sxn,
                  int64_t syb, int64_t syh, int64_t syn,
                  int dtype, void* stream);
/* The same for q, k and v of one shape in one launch; y: contiguous [3,B,H,ceil(N/block),D]. */
int s3r_pool_means3(const void* q, const void* k, const void* v, void* y, int B, int H, int64_t N, int D, int block,
                    int64_t sqb, int64_t sqh, int64_t sqn, int64_t skb, int64_t skh, int64_t skn,
                    int64_t svb, int64_t svh, int64_t svn, int dtype, void* stream);

/*
 * Compressed-branch attention with top-k block selection.
 * Replaces flash_attn_topk_func / forward_with_topk / _fwd_kernel_with_topk
 * (pi3/models/sparse_attn/flash_attention_topk.py:22-200,633-668), non-causal, no bias.
 *   o[b,h,i,:]   = softmax_j(scale * q[i].k[j]) v[j]          (I/O dtype)
 *   lse[b,h,i]   = log sum_j exp(scale * q[i].k[j])           (fp32, optional, [B,H,Lq] contiguous)
 *   topk_idx[b,h,i,0..K-1] = columns of the K largest raw UNSCALED fp32 q[i].k[j], ordered by
 *       descending 64-bit key (sortable(bits(s)) << 32 | Lk-1-j): descending score, equal
 *       scores lowest column first; if Lk < K the trailing slots hold Lk-1.
 *       (int32, optional, [B,H,Lq,K] contiguous)
 *   scores[b,h,i,j] = raw fp32 q[i].k[j]                      (optional, [B,H,Lq,Lk] contiguous)
 * When `scores` is given the indices are computed from exactly those stored values, so
 * s3r_topk_rows() on `scores` reproduces `topk_idx` bit for bit.  When `scores` is NULL the
 * scores never reach HBM: the attention output comes from a dense sweep of the selection
 * kernel and the indices from a top-k-only kernel that recomputes the scores on chip
 * (bf16/fp16, D == 64, K in {1,2,4,8,16,32}, Lk <= 2^21; two launches on `stream`).  `o` (and then `v`)
 * may be NULL when only the indices are wanted (MFMA path), `topk_idx` may be NULL when only the
 * attention is: a caller with two streams runs the two halves side by side.
 * Requires D <= 64 (D == 64 for the MFMA path), K a power of two <= 64.
 */
int s3r_compressed_attn_topk(const void* q, const void* k, const void* v,
                             void* o, float* lse, int32_t* topk_idx, float* scores,
                             int B, int H, int Lq, int Lk, int D, int K,
                             int64_t sqb, int64_t sqh, int64_t sqm,
                             int64_t skb, int64_t skh, int64_t skn,
                             int64_t svb, int64_t svh, int64_t svn,
                             int64_t sob, int64_t soh, int64_t som,
                             float softmax_scale, int dtype, void* stream);
/* Whether the indices without a score buffer come from the kernel for short lists of keys, which keeps a row's scores in LDS, and the
 * attention output with them in one launch (else from the one that sweeps over the keys twice, and a dense sweep); the same indices
 * either way.  batch_heads = B*H. */
int s3r_topk_in_lds(int64_t batch_heads, int64_t Lq, int64_t Lk, int K);

/*
 * The causal variant of s3r_compressed_attn_topk: the IS_CAUSAL branches of _fwd_kernel_with_topk
 * (flash_attention_topk.py:71,93), which the reference layer never takes (it calls with causal=False).
 * Query i (row i of its 64-row block m = i / 64) sees the keys below end_n = min((m + 1) * 64, Lk) only:
 *   o, lse:   softmax over the keys j <= i;
 *   topk_idx: the K largest of the keys j < end_n, where a key j > i has the score -inf (it ranks below every finite
 *             score, lowest column first, as the reference's integer keys order it); if end_n < K the trailing slots
 *             hold end_n - 1;
 *   scores:   [B,H,Lq,Lk] fp32 work buffer, required with `topk_idx` (row i: raw scores of the keys j < end_n with
 *             -inf for j > i; columns from end_n on are not written).
 * Any I/O dtype, D <= 64, K a power of two <= 64; runs the generic (non-MFMA) kernels.  The reference's backward
 * ignores `causal` (flash_attention_topk.py:653-666 calls _flash_attn_backward without it), so s3r_attn_bwd on the
 * lse of this call reproduces the reference's gradients as they are.
 */
int s3r_compressed_attn_topk_causal(const void* q, const void* k, const void* v,
                                    void* o, float* lse, int32_t* topk_idx, float* scores,
                                    int B, int H, int Lq, int Lk, int D, int K,
                                    int64_t sqb, int64_t sqh, int64_t sqm,
                                    int64_t skb, int64_t skh, int64_t skn,
                                    int64_t svb, int64_t svh, int64_t svn,
                                    int64_t sob, int64_t soh, int64_t som,
                                    float softmax_scale, int dtype, void* stream);

/*
 * s3r_compressed_attn_topk with its score buffer built into the library: allocates nothing.
 * No counterpart in the reference.  For callers that cannot allocate device memory: code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc.  It is the `scores != NULL` path of
 * s3r_compressed_attn_topk (any I/O dtype, any K a power of two <= 64; indices selected from exactly the stored
 * fp32 scores, so results equal that call bit for bit) with the B*H*Lq*Lk scores held in a file-scope device array
 * of S3R_STATIC_SCORES_MAX floats (96 MiB per GPU the library runs on, kept until the process ends).  Larger
 * problems return S3R_ERR_UNSUPPORTED.  `o` and `topk_idx` are both required.  The first call on a device looks up
 * that device's copy of the array (no allocation; make it outside a graph capture).  All calls on one GPU share
 * the array: calls that overlap on one GPU (two streams, two threads) race; calls on one stream do not.
 */
#define S3R_STATIC_SCORES_MAX (24u * 1024u * 1024u)
int s3r_compressed_attn_topk_static(const void* q, const void* k, const void* v,
                                    void* o, float* lse, int32_t* topk_idx,
                                    int B, int H, int Lq, int Lk, int D, int K,
                                    int64_t sqb, int64_t sqh, int64_t sqm,
                                    int64_t skb, int64_t skh, int64_t skn,
                                    int64_t svb, int64_t svh, int64_t svn,
                                    int64_t sob, int64_t soh, int64_t som,
                                    float softmax_scale, int dtype, void* stream);

/*
 * Row-wise exact top-k of a materialised fp32 score matrix (same ordering rule as above).
 * Stands for the streaming bitonic top-k inside _fwd_kernel_with_topk
 * (flash_attention_topk.py:112-132,145-152; topk_utils.py:11-23,438-501).
 * scores: `rows` rows of `cols` floats, row r at scores + r*row_stride; idx: [rows, K] int32.
 * 1 <= K <= 64.
 */
int s3r_topk_rows(const float* scores, int32_t* idx, int64_t rows, int cols, int64_t row_stride,
                  int K, void* stream);

/*
 * Selection-branch attention: every `block`-row query block attends to the K key blocks its
 * index row lists, in list order.
 * Replaces topk_blocksparse_attention / _topk_blocksparse_attention_fwd /
 * block_sparse_forward_kernel (pi3/models/sparse_attn/topk_blocksparse_attention.py:35-128,
 * 852-904,1093-1121).
 *   idx: int32 [B,H,ceil(N/block),K] (strides sib,sih,sim; last stride 1), block units;
 *        entries < 0 or with idx*block >= N are skipped; duplicates are attended twice.
 *   o:   I/O dtype [B,H,N,D];  lse: optional fp32 [B,H,N] contiguous.
 * Keys beyond N in a partial last block are masked out; a query block with no valid entry
 * gives zeros.  block in {4,16,32,64}, D <= 64 (MFMA paths: block 64 or 16, D == 64, bf16/fp16, K <= 64).
 * Rounding points of the 64-token MFMA kernel: with lse == NULL the queries are multiplied by
 * softmax_scale * log2(e) once and rounded to the I/O dtype, and the fp32 scores of those queries are exponents of two
 * (the reference scales each fp32 score, :100); a query block whose scaled scores leave [-20, 20] (bf16) is recomputed
 * with the reference's per-score scaling.  With lse != NULL (a forward whose backward will recompute the probabilities
 * from lse) every score is scaled in fp32 as in the reference.
 * The reference's larger blocks (128, 256; topk_blocksparse_attention.py:862) are the caller's to rewrite, as the
 * Python operator does: the list of a query block serves each of its 64-row parts, a listed key block j becomes the
 * entries r*j .. r*j+r-1 (r = block/64), and the call is made with block 64 and K*r entries per row.
 */
int s3r_select_attn(const void* q, const void* k, const void* v, const int32_t* idx,
                    void* o, float* lse,
                    int B, int H, int64_t N, int D, int block, int K,
                    int64_t sqb, int64_t sqh, int64_t sqn,
                    int64_t skb, int64_t skh, int64_t skn,
                    int64_t svb, int64_t svh, int64_t svn,
                    int64_t sob, int64_t soh, int64_t son,
                    int64_t sib, int64_t sih, int64_t sim,
                    float softmax_scale, int dtype, void* stream);

/*
 * Selection-branch attention with the gated merge in its epilogue: the selection output never
 * goes to memory; the kernel writes
 *   out[b,n,h*D+d] = gate[b,h,n,0]*o_cmp[b,h,n/block,d] + gate[b,h,n,1]*o_sel[b,h,n,d]
 * 16-token blocks, and fp32: with the rounding points of s3r_gated_merge (o_sel, each product and the sum rounded to the I/O
 * dtype), so the result equals s3r_select_attn followed by s3r_gated_merge bit for bit.  64-token blocks of 16-bit types: the expression
 * is evaluated in fp32 on the unrounded selection output and rounded ONCE (at most four rounding steps of the I/O dtype,
 * taken on |gate0 o_cmp| + |gate1 o_sel|, away from the two-call result, on the side of the exact value).
 * Replaces topk_blocksparse_attention (pi3/models/sparse_attn/topk_blocksparse_attention.py:1093-1121)
 * together with the merge expression of pi3/models/layers/sparse_attention.py:127-136.
 * Arguments as in s3r_select_attn and s3r_gated_merge; out is contiguous [B,N,H*D].
 * Only for the MFMA paths (D == 64, block == 64 or 16, fp32 also 32, 16-byte aligned tensors); other
 * shapes return S3R_ERR_UNSUPPORTED and the caller runs the two operators one after the other.
 */
int s3r_select_attn_merge(const void* q, const void* k, const void* v, const int32_t* idx,
                          const void* o_cmp, const void* gate, void* out,
                          int B, int H, int64_t N, int D, int block, int K,
                          int64_t sqb, int64_t sqh, int64_t sqn,
                          int64_t skb, int64_t skh, int64_t skn,
                          int64_t svb, int64_t svh, int64_t svn,
                          int64_t sib, int64_t sih, int64_t sim,
                          int64_t scb, int64_t sch, int64_t scm,
                          int64_t sgb, int64_t sgh, int64_t sgn,
                          float softmax_scale, int dtype, void* stream);

/*
 * qk-LayerNorm and 2-D rotary embedding of one [B,H,N,64] tensor (q or k) in one pass:
 *   y = RoPE2D(LayerNorm(x) rounded to the I/O dtype, pos)
 * Replaces self.q_norm / self.k_norm, the cast and self.rope of the reference layer
 * (pi3/models/layers/sparse_attention.py:103-110,120-124) and RoPE2D.forward
 * (pi3/models/layers/pos_embed.py:112-159).
 *   x: strides sxb,sxh,sxn (last stride 1; the packed projection can be passed as a view); y: contiguous.
 *   pos: int32 (y,x) per token, strides spb,spn (pair contiguous), or NULL for no rotation.
 *   cos_tab, sin_tab: I/O dtype [P,16], row p = cos/sin of the angles p * base^(-2i/32), i = 0..15, with the
 *     angles rounded to the I/O dtype first (the reference's table); positions are clamped to [0,P-1].
 *   ln_w, ln_b: I/O dtype [64] LayerNorm weight and bias, ln_w NULL for no normalisation (ln_b optional).
 * Products and sum of the rotation are rounded to the I/O dtype like the reference's eager expression.  The row
 * statistics are fp32; 1/sqrt(var + eps) comes from the hardware's reciprocal square root (1 ulp), so for 16-bit I/O
 * a value may land on the neighbouring representable number of the eager result (as it may from the order of the sums).
 */
int s3r_norm_rope(const void* x, void* y, const int32_t* pos, const void* cos_tab, const void* sin_tab, int P,
                  const void* ln_w, const void* ln_b, float eps,
                  int B, int H, int64_t N, int D,
                  int64_t sxb, int64_t sxh, int64_t sxn, int64_t spb, int64_t spn,
                  int dtype, void* stream);

/*
 * The layer's pre-pass over the packed q/k/v projection in ONE kernel: block means of the raw q, k, v rows (the
 * compressed branch's inputs) and qk-LayerNorm + 2-D rotary embedding of the full-token q and k, each input row read once.
 * Replaces F.avg_pool1d on the raw projection, the three .contiguous() copies, q_norm / k_norm with their casts and
 * the two rope calls on the full tokens (pi3/models/layers/sparse_attention.py:97-99,115-124).  Same bits as
 * s3r_pool_mean on q, k, v followed by s3r_norm_rope on q and k.
 *   q, k, v: [B,H,N,64] views with common strides sxb,sxh,sxn (last stride 1), e.g. the three sections of the packed
 *     [B,N,3*H*64] projection; v is only read (the attention kernels take it in place).
 *   q_out, k_out: contiguous [B,H,N,64];  qc, kc, vc: contiguous [B,H,ceil(N/block),64] (a ragged last block is a mean
 *     over its valid tokens).
 *   pos, cos_tab, sin_tab, P, eps and the LayerNorm parameters (qn_* for q, kn_* for k; both NULL for no norm) as in
 *     s3r_norm_rope.
 */
int s3r_qkv_prepass(const void* q, const void* k, const void* v, void* q_out, void* k_out, void* qc, void* kc, void* vc,
                    const int32_t* pos, const void* cos_tab, const void* sin_tab, int P,
                    const void* qn_w, const void* qn_b, const void* kn_w, const void* kn_b, float eps,
                    int B, int H, int64_t N, int D, int block,
                    int64_t sxb, int64_t sxh, int64_t sxn, int64_t spb, int64_t spn, int dtype, void* stream);

/*
 * The same pass with everything the layer needs of it, in an argument block:
 *   q_out, k_out (both or neither): the full-token q and k after norm and rotation, contiguous [B,H,N,64].
 *   q_pool, k_pool, v_pool (all or none): the block means, contiguous [B,H,ceil(N/block),64]; with finish_pooled q_pool and
 *     k_pool are normalised and rotated too, at the truncated mean position of their block's tokens (the reference's pooled
 *     tokens, pi3/models/layers/sparse_attention.py:97-110); q_raw, k_raw (optional): their values before that.
 *   positions: (y,x) pairs, int32 or int64 (positions_int64), strides in elements, or NULL.
 *   cos_table, sin_table: [table_rows,16] in the I/O dtype as in s3r_norm_rope.  inv_freq (optional, [16] fp32): positions
 *     at or beyond table_rows get cosine and sine of round(position * inv_freq); without it they are clamped.  Positions below
 *     zero are clamped too, or, with inv_freq and signed_positions, get their own angles like those.
 *   norm parameters in the I/O dtype, or fp32 with norm_fp32 (used unrounded).
 */
typedef struct s3r_prepass_args {
  const void *q, *k, *v;
  void *q_out, *k_out;
  void *q_pool, *k_pool, *v_pool;
  void *q_raw, *k_raw;
  const void* positions;
  const void *cos_table, *sin_table;
  const float* inv_freq;
  const void *q_norm_weight, *q_norm_bias, *k_norm_weight, *k_norm_bias;
  int64_t N, stride_b, stride_h, stride_n, pos_stride_b, pos_stride_n;
  int B, H, head_dim, block, table_rows, positions_int64, norm_fp32, finish_pooled, signed_positions, dtype;
  float eps;
} s3r_prepass_args;

int s3r_layer_prepass(const s3r_prepass_args* args, void* stream);

/*
 * Gradient of that pass (bf16/fp16, blocks of at most 64 tokens): from the gradients of q_out, k_out, v [B,H,N,64] and of
 * the finished q_pool, k_pool, v_pool (all contiguous, I/O dtype) those of the raw projection, written through
 * dx_q, dx_k, dx_v with the strides of q, k, v, and, where there is a norm, norm_grads [4,64] fp32: q_norm weight, bias,
 * k_norm weight, bias.  args as in the forward call (its outputs q_raw, k_raw are read); workspace: fp32
 * [workspace_rows,256] (768 rows fill the chip), any contents.
 */
int s3r_layer_prepass_bwd(const s3r_prepass_args* args, const void* dq, const void* dk, const void* dv, const void* dq_pool,
                          const void* dk_pool, const void* dv_pool, void* dx_q, void* dx_k, void* dx_v, float* norm_grads,
                          float* workspace, int workspace_rows, void* stream);

/*
 * Gradient of the gated merge (bf16/fp16, head_dim 64): dout [B,N,H*64], o_cmp [B,H,ceil(N/block),64], o_sel [B,H,N,64]
 * contiguous, gate [B,H,N,2] with strides sgb,sgh,sgn (pair contiguous) -> d_o_cmp, d_o_sel (as o_cmp, o_sel), d_gate
 * [B,N,H,2], and the row sums delta_cmp = <d_o_cmp, o_cmp> [B,H,ceil(N/block)], delta_sel = <d_o_sel, o_sel> [B,H,N] (fp32)
 * that s3r_attn_bwd takes.  Sums in fp32, every result rounded once.
 */
int s3r_gated_merge_bwd(const void* dout, const void* o_cmp, const void* o_sel, const void* gate, void* d_o_cmp, void* d_o_sel,
                        void* d_gate, float* delta_cmp, float* delta_sel, int B, int H, int64_t N, int D, int block,
                        int64_t sgb, int64_t sgh, int64_t sgn, int dtype, void* stream);

/*
 * LayerNorm over the channels of token rows:  y[r,:] = (x[r,:] - mean_r) * rstd_r * w + b, fp32 statistics, one
 * rounding to the I/O dtype.  Replaces, for inference, the nn.LayerNorm modules in front of the attention layers and
 * the MLPs (norm1 / norm2, pi3/models/layers/block.py:281,296,312,315).
 *   x, y: [rows, C] in the I/O dtype with row strides sx, sy (elements; multiples of 16 bytes); w, b: [C] (b may be
 *   NULL).  C: a multiple of 16 bytes worth of elements, at most 4096 (two-byte types) or 2048 (fp32).
 */
int s3r_layer_norm(const void* x, void* y, const void* w, const void* b, float eps, int64_t rows, int C,
                   int64_t sx, int64_t sy, int dtype, void* stream);

/*
 * Residual and the norm behind it:  s[r,:] = x[r,:] + gamma * a[r,:] rounded to the I/O dtype, y = LayerNorm(s) as
 * s3r_layer_norm computes it.  The add (LayerScale with gamma, pi3/models/layers/block.py:281,296) and the next norm
 * in one pass.  x, a, s, y: contiguous [rows, C], s and y apart from x and a; gamma, w, b: [C], gamma and b may be NULL.
 */
int s3r_add_layer_norm(const void* x, const void* a, const void* gamma, void* s, void* y, const void* w, const void* b, float eps,
                       int64_t rows, int C, int dtype, void* stream);

/*
 * A linear layer of the inference paths  y[r,:] = act(x[r,:] W^T + bias)  (the projections around the attention,
 * pi3/models/layers/sparse_attention.py:93,140, and the MLPs); fp32 sums, bias and activation in fp32, one rounding.
 *   x: [M, K], w: [N, K], y: [M, N] with row strides ldx, ldw, ldy (elements); bias: [N] or NULL; bf16 / fp16, K a multiple of
 *   128, N of 8; x, w, y and their rows multiples of 16 bytes, bias of 8.
 */
#define S3R_ACT_NONE 0
#define S3R_ACT_GELU 1 /* exact: x/2 (1 + erf(x / sqrt 2)) */
int s3r_linear(const void* x, const void* w, const void* bias, void* y, int64_t M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldy,
               int activation, int dtype, void* stream);

/*
 * Gradients of a linear layer's parameters over many rows:  dw = dy^T x [N, C],  db = the sums of dy over the rows [N], or NULL;
 * fp32 sums, one rounding, the same bits for the same inputs.
 *   dy: [M, N], x: [M, C] with row strides lddy, ldx (elements); dw, db contiguous; workspace: as many floats as
 *   s3r_linear_wgrad_workspace says; bf16 / fp16, N and C multiples of 8, C > 768 with db; dy, x, dw, the workspace and the rows of
 *   dy and x multiples of 16 bytes.
 */
int64_t s3r_linear_wgrad_workspace(int64_t M, int N, int C, int64_t lddy, int64_t ldx);
int s3r_linear_wgrad(const void* dy, const void* x, void* dw, void* db, float* workspace, int64_t M, int N, int C, int64_t lddy, int64_t ldx,
                     int dtype, void* stream);

/*
 * s3r_linear and s3r_layer_prepass in one: the layer's projection  [q | k | v] = x W^T + bias  and, of it,
 * q and k after LayerNorm and RoPE2D, v, and the finished block means (sparse_attention.py:93-110,115-124).
 *   x: [B*N, C] rows of stride ldx, w: [3*C, C] of stride ldw, bias: [3*C] or NULL, C = 64 H; v_out: contiguous [B,H,N,64];
 *   a: as for s3r_layer_prepass (q, k, v and the strides are not read): q_out, k_out, positions and tables are required,
 *   the three means and the norms optional; means only with norms, `finish_pooled` and without q_raw, k_raw; not with inv_freq and
 *   signed_positions.
 * bf16 / fp16, an even number of heads, block 16 or 64; several sequences: 256 tokens or more each, with means a multiple of
 * the block.  gate_out (or NULL): [B*N, gate_outputs], what s3r_gate gives for x, gate_w ([gate_outputs, C]) and gate_bias (or
 * NULL); a multiple of 4 outputs up to 32.  Rounding: the projection to the I/O dtype, then once at the end (s3r_layer_prepass also rounds in between).
 */
int s3r_qkv_project(const void* x, const void* w, const void* bias, int64_t ldx, int64_t ldw, void* v_out, const struct s3r_prepass_args* a,
                    const void* gate_w, const void* gate_bias, void* gate_out, int gate_outputs, void* stream);
/* Whether s3r_qkv_project computes the gate of `rows` = B*N rows and H heads in time that it leaves idle (else s3r_gate is as good). */
int s3r_qkv_project_gate_rides(int64_t rows, int H);

/*
 * The attention layer's inference (pi3/models/layers/sparse_attention.py:90-141) in one call: s3r_qkv_project with its gate,
 * s3r_compressed_attn_topk with indices, s3r_gate where that does not ride, s3r_select_attn_merge and, with proj_w, s3r_linear, one after
 * the other on `stream`: the same results.  Few tokens wait for the host, which makes one call instead of five.
 *   a: as for s3r_qkv_project with means and norms, but its outputs (q_out .. v_pool) are not read: they lie in `workspace`,
 *   s3r_attention_layer_workspace bytes at a multiple of 256; gate_w: [2 H, C]; proj_w: [C, C] or NULL (out is then the merged
 *   branches); out: contiguous [B*N, C]; all weights contiguous, 16-byte aligned, in a->dtype.
 * K: 1, 2, 4, 8, 16 or 32; softmax_scale > 0; B H up to 65535.  The gate: 2 H outputs a multiple of 4 up to 32 that ride, or H a
 * multiple of 4 up to 16.
 */
int64_t s3r_attention_layer_workspace(int B, int H, int64_t N, int block, int K, int with_projection);
int s3r_attention_layer(const void* x, const void* qkv_w, const void* qkv_bias, const void* gate_w, const void* gate_bias,
                        const void* proj_w, const void* proj_bias, void* out, void* workspace, int64_t workspace_bytes,
                        const struct s3r_prepass_args* a, int K, float softmax_scale, void* stream);

/*
 * The layer's gate  out[r,:] = sigmoid(x[r,:] W^T + bias)  (pi3/models/layers/sparse_attention.py:88,127); fp32 sums, the
 * product with its bias and the sigmoid each rounded to the I/O dtype.
 *   x: contiguous [rows, C], w: contiguous [O, C], bias: [O] or NULL, out: contiguous [rows, O]; bf16 / fp16, C a multiple of
 *   256 up to 1024, O even, up to 32.
 */
int s3r_gate(const void* x, const void* w, const void* bias, void* out, int64_t rows, int C, int O, int dtype, void* stream);

/*
 * Gated merge of the two branches, written in the [B,N,H*D] layout the output projection
 * reads:  out[b,n,h*D+d] = gate[b,h,n,0]*o_cmp[b,h,n/block,d] + gate[b,h,n,1]*o_sel[b,h,n,d].
 * Replaces the einops/broadcast expression in pi3/models/layers/sparse_attention.py:127-136.
 * Each product and the sum are rounded to the I/O dtype, like the eager expression.
 * gate strides sgb,sgh,sgn address the pair (last stride 1); out is contiguous.
 */
int s3r_gated_merge(const void* o_cmp, const void* o_sel, const void* gate, void* out,
                    int B, int H, int64_t N, int D, int block,
                    int64_t scb, int64_t sch, int64_t scm,
                    int64_t ssb, int64_t ssh, int64_t ssn,
                    int64_t sgb, int64_t sgh, int64_t sgn,
                    int dtype, void* stream);

/*
 * Backward of the two attention operators (bf16/fp16, head_dim 64; selection blocks of 64 or 16 tokens, `block`
 * is ignored when idx == NULL).
 * Replaces _topk_blocksparse_attention_bwd (pi3/models/sparse_attn/topk_blocksparse_attention.py:907-1038, kernels
 * backward_sum_o_do :132-170, backward_dkdv :558-712, backward_dq :722-850) and, with idx == NULL (every key tile),
 * _flash_attn_backward (pi3/models/sparse_attn/flash_attention_topk.py:204-630).
 *
 * s3r_attn_bwd_delta:  delta[b,h,n] = sum_d o[b,h,n,d] * dout[b,h,n,d]  (fp32, contiguous [B,H,N]).
 * s3r_attn_bwd: with P = exp(scale * q k^T - lse) over the keys the forward attended to,
 *   dv = P^T dout,  dS = scale * P * (dout v^T - delta),  dq = dS k,  dk = dS^T q;
 *   P and dS are rounded to the I/O dtype before the products, accumulation is fp32 (for dk in bf16 the
 *   rounded factor is dS / scale and the scale multiplies the fp32 sum: the same relative rounding).
 *   lse: the forward's optional output (natural log, scaled scores), fp32 [B,H,Lq] contiguous.
 *   idx: the forward's block indices [B,H,ceil(Lq/block),K] (strides sib,sih,sim), or NULL for dense attention.
 *   kq_list, kq_off (needed for dk/dv when idx is given): for every (b,h) the query-block ids that list key block j,
 *     one entry per occurrence, ascending, are kq_list[(b*H+h)*list_stride + kq_off[(b*H+h)*(nkb+1) + j] ...
 *     kq_off[... + j+1]), nkb = ceil(Lk/block); entries of idx that are < 0 or >= nkb appear in no list
 *     (reference count_query_fixedlen / reorder_topk_idx_fixedlen, :423-554).  The kernels add up in the order of the list.
 *   dq (layout strides sdq*), dk, dv (sdk*, sdv*): I/O dtype; dq == NULL or dk == dv == NULL skips that kernel.
 *   Every row of dq, dk, dv inside the tensors is written (zeros where nothing attends).
 * s3r_attn_bwd_from_output: the same with delta computed on the way, from the forward's output o (layout strides so*): delta is
 *   [B,H,Lq] fp32 that the call fills.  dq is required.
 */
/*
 * Key-centric lists for s3r_attn_bwd from the forward's index tensor.
 * Replaces count_query_fixedlen, the stable argsort and reorder_topk_idx_fixedlen of the reference's backward
 * (pi3/models/sparse_attn/topk_blocksparse_attention.py:423-554).
 *   idx: [B,H,nqb,K] int32 (strides sib,sih,sim, last dimension contiguous); nkb: number of key blocks.
 *   kq_off: [B,H,nkb+1] int32, contiguous; kq_list: [B,H,list_stride] int32, list_stride >= nqb*K.
 * Block j's list of (b,h) = kq_list[(b*H+h)*list_stride + kq_off[..j] ... kq_off[..j+1]): the query-block ids whose
 * index row names j, one entry per occurrence, ascending.  Entries of idx < 0 or >= nkb appear in no list; the part
 * of kq_list behind kq_off[..nkb] is left as it was.  No workspace; the result does not depend on the run.
 */
int s3r_key_block_lists(const int32_t* idx, int32_t* kq_list, int32_t* kq_off, int B, int H, int64_t nqb, int K, int64_t nkb,
                        int64_t sib, int64_t sih, int64_t sim, int64_t list_stride, void* stream);
int s3r_attn_bwd_delta(const void* o, const void* dout, float* delta, int B, int H, int64_t N, int D,
                       int64_t sob, int64_t soh, int64_t son, int64_t sdb, int64_t sdh, int64_t sdn,
                       int dtype, void* stream);
int s3r_attn_bwd(const void* q, const void* k, const void* v, const void* dout, const float* lse, const float* delta,
                 const int32_t* idx, const int32_t* kq_list, const int32_t* kq_off, int64_t list_stride,
                 void* dq, void* dk, void* dv,
                 int B, int H, int64_t Lq, int64_t Lk, int D, int block, int K,
                 int64_t sqb, int64_t sqh, int64_t sqm, int64_t skb, int64_t skh, int64_t skn,
                 int64_t svb, int64_t svh, int64_t svn, int64_t sgb, int64_t sgh, int64_t sgm,
                 int64_t sdqb, int64_t sdqh, int64_t sdqm, int64_t sdkb, int64_t sdkh, int64_t sdkn,
                 int64_t sdvb, int64_t sdvh, int64_t sdvn, int64_t sib, int64_t sih, int64_t sim,
                 float softmax_scale, int dtype, void* stream);
int s3r_attn_bwd_from_output(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                             const void* o, int64_t sob, int64_t soh, int64_t som, float* delta,
                             const int32_t* idx, const int32_t* kq_list, const int32_t* kq_off, int64_t list_stride,
                             void* dq, void* dk, void* dv,
                             int B, int H, int64_t Lq, int64_t Lk, int D, int block, int K,
                             int64_t sqb, int64_t sqh, int64_t sqm, int64_t skb, int64_t skh, int64_t skn,
                             int64_t svb, int64_t svh, int64_t svn, int64_t sgb, int64_t sgh, int64_t sgm,
                             int64_t sdqb, int64_t sdqh, int64_t sdqm, int64_t sdkb, int64_t sdkh, int64_t sdkn,
                             int64_t sdvb, int64_t sdvh, int64_t sdvn, int64_t sib, int64_t sih, int64_t sim,
                             float softmax_scale, int dtype, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* SPEED3R_HIP_H */
