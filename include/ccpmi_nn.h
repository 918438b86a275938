/*
 * ccpmi_nn — kernels of the contact-map surrogate (no counterpart in ccp).
 *
 * A 1-D convolutional encoder over the binned het/LAD sequence with a
 * pairwise outer-product head. Two sets of kernels compute it: single
 * operations (a strided batched BF16 GEMM on the matrix cores with FP32
 * accumulation, and the element-wise steps around it), for a caller's own
 * composition, and the network's own kernels further down, which fuse them
 * and give the same bits in outputs and weight gradients. Activations are stored
 * channel-major: x[c, b L + l] for channel c, sample b, bin l. BF16 values
 * are passed as raw 16-bit words (void pointers). Every call is
 * asynchronous on `stream` (a hipStream_t) and returns 0, 1 for bad sizes,
 * or 2 for a launch failure.
 */
#ifndef CCPMI_NN_H
#define CCPMI_NN_H

#ifdef __cplusplus
extern "C" {
#endif

/* C[b](m, n) = alpha sum_k A[b](m, k) B[b](k, n) + beta C[b](m, n), with
 * X[b](i, j) at X + b sxb + i sxi + j sxj; A, B BF16. The result is written
 * to C (FP32, may be NULL when beta = 0) and/or Cb (BF16). */
int ccp_nn_gemm(const void *A, const void *B, float *C, void *Cb, int M, int N, int K, int batch, long sab, long sam,
                long sak, long sbb, long sbk, long sbn, long scb, long scm, long scn, float alpha, float beta,
                void *stream);
/* kernel-3, padding-1 convolution as a GEMM: cols[(c 3 + t), p] = x[c, p + t - 1] within each sample */
int ccp_nn_im2col(const void *x, void *cols, int C, int Bn, int L, void *stream);
/* its adjoint: dx = col2im(dcols) + beta dx */
int ccp_nn_col2im(const float *dcols, float *dx, int C, int Bn, int L, float beta, void *stream);
/* pre += bias (per channel); y = gelu(pre) + res (res may be NULL); y FP32 (may be NULL) and yb BF16 */
int ccp_nn_bias_gelu(float *pre, const float *bias, const float *res, float *y, void *yb, int C, long P,
                     void *stream);
/* g = dy gelu'(pre) (FP32 and BF16); dbias += sum over positions */
int ccp_nn_gelu_back(const float *pre, const float *dy, float *g, void *gb, float *dbias, int C, long P,
                     void *stream);
/* pred[b](i, j) = (raw[b](i, j) + raw[b](j, i)) / 2 + dist[|i - j|] + c0[0] */
int ccp_nn_pair_map(const float *raw, const float *dist, const float *c0, float *pred, int L, int Bn, void *stream);
/* w * mean squared error over i <= j; gradients of raw (FP32, BF16), dist and c0 (accumulated); loss += */
int ccp_nn_pair_loss(const float *pred, const float *target, float *gS, float *graw, void *grawb, float *gdist,
                     float *gc0, float *loss, int L, int Bn, float w, void *stream);
int ccp_nn_mean_pool(const float *h, float *pooled, void *pooledb, int C, int Bn, int L, void *stream);
int ccp_nn_pool_back(const float *dpooled, float *dh, int C, int Bn, int L, void *stream);
/* pred += bias; w * mean squared error; g = dLoss/dpred (FP32, BF16); dbias += ; loss += */
int ccp_nn_rd_loss(float *pred, const float *bias, const float *target, float *g, void *gb, float *dbias, float *loss,
                   int O, int Bn, float w, void *stream);
int ccp_nn_cast_bf16(const float *x, void *y, long n, void *stream);
/* AdamW step t (1-based) on FP32 parameters; pb receives the BF16 copy (may be NULL) */
int ccp_nn_adamw(float *p, const float *g, float *m, float *v, void *pb, long n, float lr, float b1, float b2,
                 float eps, float wd, int t, void *stream);

/* ---- the network's own kernels ----
 * Positions are p = b L + l, P = B L. BF16 activations and gradients come as
 * channel rows [C][Ps], Ps = P rounded up to 16, zero beyond P, and as position
 * rows [P][Cs], Cs at least C rounded up to the K tile of what reads them (16
 * channels for a convolution, 64 for the heads, 32 backward), zero beyond C.
 * FP32 ones are [C][Ps].
 * All pointers are 16-byte aligned device memory. */

/* x[c, p] FP32 -> channel rows xb (may be NULL) and position rows xt; *loss = 0
 * when given */
int ccp_nn_input(const float *x, void *xb, void *xt, int C, int Cs, int P, int Ps, float *loss, void *stream);

/* A layer's forward product (M rows). conv: kernel-3 convolution of X with
 * the packed weights A0 [M rounded to 64][Kp], Kp = 3 (C rounded up to 16);
 * pre = product + bias, y = gelu(pre) + res (res, pre may be NULL); y in
 * FP32, in BF16 as ob (channel rows, may be NULL) and ot (position rows of
 * Os). Otherwise the plain product of A0 (rows below M0) and A1 (the others),
 * Kp = C rounded up to 64, to ob and ot, the rows from M0 on at column O1 of
 * the position rows. */
typedef struct ccp_nn_fwd_args {
  const unsigned short *A0, *A1, *X;
  const float *bias, *res;
  float *pre, *y;
  unsigned short *ob, *ot;
  int M, M0, Kp, Cs, P, Ps, L, Os, O1;
} ccp_nn_fwd_args;
int ccp_nn_fwd(const ccp_nn_fwd_args *a, int conv, void *stream);

/* pair map of ccp_nn_pair_map, straight from position rows holding U in
 * columns [0, d) and V in [d, 2 d) (d a multiple of 16, zero where unused) */
int ccp_nn_pair(const void *uv, int d, const float *dist, const float *c0, float *S, int L, int B, float alpha,
                void *stream);
/* mean over each sample's L positions, summed in order, as pb [C][Bs] and pt [B][Cs] */
int ccp_nn_pool(const float *h, void *pb, void *pt, int C, int B, int L, int Ps, int Bs, int Cs, void *stream);
/* C[m][n] = sum over k of A[m][k] B[n][k]: few rows, K a multiple of 16, leading dimensions lda, ldb (multiples of 8), ldc */
int ccp_nn_small(const void *A, const void *B, float *C, int M, int N, int K, int lda, int ldb, int ldc, void *stream);

/* ccp_nn_pair_loss with the raw map's gradient as BF16 rows of Ls entries (L
 * rounded up to 8, zero beyond L) and per (sample, band) partials of gdist (L
 * each) and gc0; ccp_nn_pair_bands(L) bands a sample. loss += */
int ccp_nn_pair_bands(int L);
int ccp_nn_pair_grad(const float *pred, const float *target, void *graw, float *gdist, float *gc0, float *loss, int L,
                     int Ls, int B, float w, void *stream);
/* ccp_nn_rd_loss with the gradient as gb [O][Bs] and gt [Bn][Os], dbias summed in a fixed order */
int ccp_nn_rd_grad(float *pred, const float *bias, const float *target, void *gb, void *gt, float *dbias, float *loss,
                   int O, int Bn, int Bs, int Os, float w, void *stream);
/* gradients of U and V (uvb: their 2 d channel rows) from the raw map's
 * (symmetric), as 2 d channel rows db and position rows dt of 2 ds */
int ccp_nn_duv(const void *uvb, const void *graw, void *db, void *dt, int d, int ds, int L, int Ls, int B, int Ps,
               float alpha, void *stream);

/* Gradient of a layer's activations, times gelu'(pre), as channel rows gb and
 * position rows gt of Cs; its sums over 128-position tiles as partials dbias
 * [ceil(P / 128)][C]. W: packed [taps][Cr][Kr], Cr = C rounded up to 64, Kr the
 * contraction rounded up to 32. head: from the gradients of U and V (position
 * rows G, V at column V1; W two matrices) and dpooled; otherwise the adjoint of
 * the next layer's convolution added to dh. dh written when keep. */
typedef struct ccp_nn_back_args {
  const unsigned short *W, *G;
  const float *dpooled, *pre;
  float *dh;
  unsigned short *gb, *gt;
  float *dbias;
  int C, Cs, Cr, Kr, Gs, P, Ps, L, B, V1, keep;
} ccp_nn_back_args;
int ccp_nn_back(const ccp_nn_back_args *a, int head, void *stream);

/* Weight gradients of n_jobs products in one launch (tables in device memory):
 * dst[m][taps c + t] += sum over p of G[m, p] X[c, p + t - 1] (taps 3, nothing
 * across a sample's ends) or G[m, p] X[c, p] (taps 1), p < P, rows of Ps (P
 * rounded up to 16, below 2^26, zero beyond P); rows from M0 on go to dst1.
 * first: each job's first tile, jobs in order, ccp_nn_wgrad_tiles of each,
 * n_tiles in all. */
typedef struct ccp_nn_wgrad_job {
  const void *G, *X;
  float *dst0, *dst1;
  int M, M0, C, taps, P, Ps;
} ccp_nn_wgrad_job;
int ccp_nn_wgrad_tiles(int M, int C);
int ccp_nn_wgrad(const ccp_nn_wgrad_job *tab, const int *first, int n_jobs, int n_tiles, int L, void *stream);
/* the same where a job's rows have 2^26 entries or more (addresses of 64 bits) */
int ccp_nn_wgrad_far(const ccp_nn_wgrad_job *tab, const int *first, int n_jobs, int n_tiles, int L, void *stream);

/* dst[i] += sum over parts of src[k stride + i], i < n, for n segments of a
 * table in device memory, in a fixed order */
typedef struct ccp_nn_segment {
  const float *src;
  float *dst;
  long n, stride;
  long parts;
} ccp_nn_segment;
int ccp_nn_reduce(const ccp_nn_segment *seg, int n, void *stream);

/* BF16 copies of n weight matrices w [M][taps C] (table in device memory): wb
 * as it is, fwd [.][Kp] for ccp_nn_fwd (may be NULL), back [taps][Cr][Kr] for
 * ccp_nn_back (may be NULL); entries outside are left as they are */
typedef struct ccp_nn_weight {
  const float *w;
  void *wb, *fwd, *back;
  int M, C, taps, Kp, Cr, Kr;
} ccp_nn_weight;
int ccp_nn_pack(const ccp_nn_weight *tab, int n, void *stream);

/* ccp_nn_adamw over one flat run of n parameters, decay on the first n_decay */
int ccp_nn_adamw_flat(float *p, const float *g, float *m, float *v, long n, long n_decay, float lr, float b1, float b2,
                      float eps, float wd, int t, void *stream);

#ifdef __cplusplus
}
#endif

#endif
