// gfx950 kernels of the contact-map surrogate: a strided, batched BF16 GEMM
// on the matrix cores (v_mfma_f32_32x32x16 bf16, FP32 accumulation) and the
// element-wise pieces of a 1-D convolutional encoder with a pairwise
// outer-product head (im2col / col2im, bias + GELU and its derivative, the
// symmetric pair map, pooling, losses, AdamW).
//
// Matrices are addressed by element strides, so one GEMM covers every
// transpose the forward and backward passes need:
//   C[b](m, n) = alpha * sum_k A[b](m, k) B[b](k, n) + beta * C[b](m, n)
// with A[b](m, k) = A[b * sab + m * sam + k * sak] and likewise for B and C.

#include "ccpmi_nn.h"

#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint16_t f2bf(float f) {
  // round to nearest even; NaN stays NaN
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// Block tile 64 x 64 (four wavefronts of 32 x 32), K tile 32: two
// v_mfma_f32_32x32x16_bf16 per wavefront per K tile.
constexpr int TM = 64, TN = 64, TK = 32, GEMM_THREADS = 256;
// LDS rows: 32 K values plus 8 of padding (80 bytes), so the 16-byte reads
// of the 32 rows one MFMA operand takes spread over the banks
constexpr int TKP = TK + 8;

// Eight elements along K of one row (A) or column (B) of the tile, for the
// staging thread: one 16-byte load when they are contiguous and aligned in
// memory, else eight loads (zero outside the matrix).
__device__ __forceinline__ uint4 load8(const uint16_t *__restrict__ P, long base, long sk, int row_ok, int k,
                                       int K) {
  if (row_ok && sk == 1 && k + 8 <= K && ((uintptr_t)(P + base + k) & 15u) == 0)
    return *(const uint4 *)(P + base + k);
  uint16_t v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (row_ok && k + j < K) ? P[base + (long)(k + j) * sk] : (uint16_t)0;
  uint4 r;
  r.x = v[0] | (uint32_t)v[1] << 16;
  r.y = v[2] | (uint32_t)v[3] << 16;
  r.z = v[4] | (uint32_t)v[5] << 16;
  r.w = v[6] | (uint32_t)v[7] << 16;
  return r;
}

__global__ __launch_bounds__(GEMM_THREADS) void k_gemm(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                                                       float *C, uint16_t *Cb, int M, int N, int K, long sab,
                                                       long sam, long sak, long sbb, long sbk, long sbn, long scb,
                                                       long scm, long scn, float alpha, float beta) {
  // A tile by row (m, k) and B tile by column (n, k): a lane's eight K values
  // of either operand are one 16-byte LDS read
  __shared__ __align__(16) uint16_t As[TM][TKP];
  __shared__ __align__(16) uint16_t Bs[TN][TKP];
  const int b = blockIdx.z;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  A += (long)b * sab;
  B += (long)b * sbb;
  // staging: each thread one row (column) and one group of eight K values.
  // When the matrix is contiguous along M (N), consecutive threads take
  // consecutive rows, so each of the eight element loads is coalesced;
  // otherwise four threads cover one row's 32 K values.
  const bool a_rows = sam == 1 && sak != 1;
  const int am = a_rows ? tid & 63 : tid >> 2, ak = a_rows ? (tid >> 6) * 8 : (tid & 3) * 8;
  const bool b_cols = sbn == 1 && sbk != 1;
  const int bn = b_cols ? tid & 63 : tid >> 2, bk = b_cols ? (tid >> 6) * 8 : (tid & 3) * 8;
  const int gm = m0 + am, hn = n0 + bn;
  const long abase = (long)gm * sam, bbase = (long)hn * sbn;
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  for (int k0 = 0; k0 < K; k0 += TK) {
    const uint4 av = load8(A, abase, sak, gm < M, k0 + ak, K);
    const uint4 bv = load8(B, bbase, sbk, hn < N, k0 + bk, K);
    *(uint4 *)&As[am][ak] = av;
    *(uint4 *)&Bs[bn][bk] = bv;
    __syncthreads();
    // lane l holds A(row l % 32, k 8 (l / 32) + j) and B(k 8 (l / 32) + j, col l % 32), j = 0..7
    const int r = lane & 31, kq = 8 * (lane >> 5);
#pragma unroll
    for (int ks = 0; ks < TK; ks += 16) {
      const bf16x8 af = *(const bf16x8 *)&As[wm + r][ks + kq];
      const bf16x8 bfr = *(const bf16x8 *)&Bs[wn + r][ks + kq];
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bfr, acc, 0, 0, 0);
    }
    __syncthreads();
  }
  // D element v of lane l: row 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32
  const int col = n0 + wn + (lane & 31);
  if (col >= N) return;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = m0 + wm + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
    if (row >= M) continue;
    const long o = (long)b * scb + (long)row * scm + (long)col * scn;
    float out = alpha * acc[v];
    if (beta != 0.0f) out += beta * C[o];
    if (C) C[o] = out;
    if (Cb) Cb[o] = f2bf(out);
  }
}

constexpr int EW = 256;
inline unsigned grid_for(long n) { return (unsigned)((n + EW - 1) / EW); }

// cols[(c 3 + t), b L + l] = x[c, b L + l + t - 1] (zero outside the sequence)
__global__ void k_im2col(const uint16_t *x, uint16_t *cols, int C, int Bn, int L) {
  const long P = (long)Bn * L, n = (long)C * 3 * P;
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i >= n) return;
  const long p = i % P;
  const int row = (int)(i / P), c = row / 3, t = row % 3;
  const int l = (int)(p % L), src = l + t - 1;
  cols[i] = (src >= 0 && src < L) ? x[(long)c * P + p + (t - 1)] : (uint16_t)0;
}

// dx[c, b L + l] = sum_t dcols[(c 3 + t), b L + l - t + 1]
__global__ void k_col2im(const float *dcols, float *dx, int C, int Bn, int L, float beta) {
  const long P = (long)Bn * L, n = (long)C * P;
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i >= n) return;
  const int c = (int)(i / P);
  const long p = i % P;
  const int l = (int)(p % L);
  float s = 0.0f;
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const int dst = l - t + 1;
    if (dst >= 0 && dst < L) s += dcols[(long)(c * 3 + t) * P + p - t + 1];
  }
  dx[i] = s + (beta != 0.0f ? beta * dx[i] : 0.0f);
}

__device__ __forceinline__ float gelu(float x) {
  const float k = 0.7978845608f; // sqrt(2 / pi)
  return 0.5f * x * (1.0f + tanhf(k * (x + 0.044715f * x * x * x)));
}
__device__ __forceinline__ float gelu_grad(float x) {
  const float k = 0.7978845608f;
  const float u = k * (x + 0.044715f * x * x * x), t = tanhf(u);
  return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * k * (1.0f + 3.0f * 0.044715f * x * x);
}

// pre[c, p] += bias[c]; y = gelu(pre) (+ res when given); y in FP32 and BF16
__global__ void k_bias_gelu(float *pre, const float *bias, const float *res, float *y, uint16_t *yb, int C, long P) {
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i >= (long)C * P) return;
  const float v = pre[i] + bias[i / P];
  pre[i] = v;
  float o = gelu(v);
  if (res) o += res[i];
  if (y) y[i] = o;
  yb[i] = f2bf(o);
}

// g = dy * gelu'(pre), in FP32 and BF16; dbias[c] accumulates over p
__global__ void k_gelu_back(const float *pre, const float *dy, float *g, uint16_t *gb, float *dbias, int C, long P) {
  const int c = blockIdx.y;
  float part = 0.0f;
  for (long p = (long)blockIdx.x * EW + threadIdx.x; p < P; p += (long)gridDim.x * EW) {
    const long i = (long)c * P + p;
    const float v = dy[i] * gelu_grad(pre[i]);
    g[i] = v;
    gb[i] = f2bf(v);
    part += v;
  }
  __shared__ float red[EW];
  red[threadIdx.x] = part;
  __syncthreads();
  for (int o = EW / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(dbias + c, red[0]);
}

// Pair map of sample b: S = (M + M^T) / 2 + dist[|i - j|] + c0, with
// M = raw[b] (L x L); pred written in FP32.
__global__ void k_pair_map(const float *raw, const float *dist, const float *c0, float *pred, int L, int Bn) {
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i >= (long)Bn * L * L) return;
  const int b = (int)(i / ((long)L * L)), r = (int)((i / L) % L), c = (int)(i % L);
  const float *M = raw + (long)b * L * L;
  const int d = r > c ? r - c : c - r;
  pred[i] = 0.5f * (M[(long)r * L + c] + M[(long)c * L + r]) + dist[d] + c0[0];
}

// Loss of the pair maps over the pairs r <= c (mean squared error against
// target, weight w) and its gradient. gS(r, c) = dLoss/dS for r <= c; the
// raw map M enters S(lo, hi) as (M(lo, hi) + M(hi, lo)) / 2, so
// graw(r, c) = gS(lo, hi) / 2 off the diagonal and gS(r, r) on it. One block
// per row (b, r); the block's squared errors are summed into loss[0].
__global__ void k_pair_loss(const float *pred, const float *target, float *gS, float *graw, uint16_t *grawb,
                            float *loss, int L, int Bn, float w) {
  const long row = blockIdx.x; // b L + r
  const int r = (int)(row % L);
  const long base = (row - r) * L; // start of sample b
  const float count = (float)Bn * L * (L + 1) / 2;
  float sq = 0.0f;
  for (int c = threadIdx.x; c < L; c += blockDim.x) {
    const int lo = r < c ? r : c, hi = r < c ? c : r;
    const long u = base + (long)lo * L + hi;
    const float e = pred[u] - target[u];
    const float g = 2.0f * w * e / count;
    const float gr = (r == c) ? g : 0.5f * g;
    const long i = row * L + c;
    graw[i] = gr;
    grawb[i] = f2bf(gr);
    if (r <= c) {
      gS[i] = g;
      sq += w * e * e / count;
    } else {
      gS[i] = 0.0f;
    }
  }
  __shared__ float red[EW];
  red[threadIdx.x] = sq;
  __syncthreads();
  for (int o = EW / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

// gdist[d] = sum over samples and rows of gS(r, r + d); gc0 = sum of all.
__global__ void k_pair_reduce(const float *gS, float *gdist, float *gc0, int L, int Bn) {
  const int d = blockIdx.x;
  float s = 0.0f;
  const long n = (long)Bn * (L - d);
  for (long k = threadIdx.x; k < n; k += blockDim.x) {
    const long b = k / (L - d);
    const int r = (int)(k % (L - d));
    s += gS[(b * L + r) * L + r + d];
  }
  __shared__ float red[EW];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = EW / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    gdist[d] += red[0];
    atomicAdd(gc0, red[0]);
  }
}

// pooled[c, b] = mean over l of h[c, b L + l], FP32 and BF16
__global__ void k_mean_pool(const float *h, float *pooled, uint16_t *pooledb, int C, int Bn, int L) {
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i >= (long)C * Bn) return;
  const int c = (int)(i / Bn), b = (int)(i % Bn);
  const float *row = h + (long)c * Bn * L + (long)b * L;
  float s = 0.0f;
  for (int l = 0; l < L; ++l) s += row[l];
  s /= (float)L;
  pooled[i] = s;
  pooledb[i] = f2bf(s);
}

// dh[c, b L + l] += dpooled[c, b] / L
__global__ void k_pool_back(const float *dpooled, float *dh, int C, int Bn, int L) {
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i >= (long)C * Bn * L) return;
  const long P = (long)Bn * L;
  const int c = (int)(i / P), b = (int)((i % P) / L);
  dh[i] += dpooled[(long)c * Bn + b] / (float)L;
}

// Radial head: pred[o, b] += bias[o]; loss of w * mean squared error
// against target; g = dLoss/dpred (FP32, BF16); dbias accumulates. One block.
__global__ void k_rd_loss(float *pred, const float *bias, const float *target, float *g, uint16_t *gb, float *dbias,
                          float *loss, int O, int Bn, float w) {
  float sq = 0.0f;
  const float count = (float)O * Bn;
  for (int i = threadIdx.x; i < O * Bn; i += blockDim.x) {
    const int o = i / Bn;
    const float v = pred[i] + bias[o];
    pred[i] = v;
    const float e = v - target[i];
    const float gi = 2.0f * w * e / count;
    g[i] = gi;
    gb[i] = f2bf(gi);
    sq += w * e * e / count;
    atomicAdd(dbias + o, gi);
  }
  __shared__ float red[EW];
  red[threadIdx.x] = sq;
  __syncthreads();
  for (int o = EW / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}

__global__ void k_cast(const float *x, uint16_t *y, long n) {
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

// AdamW (Loshchilov & Hutter) with bias correction; writes the BF16 copy.
__global__ void k_adamw(float *p, const float *g, float *m, float *v, uint16_t *pb, long n, float lr, float b1,
                        float b2, float eps, float wd, float c1, float c2) {
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  float pi = p[i] * (1.0f - lr * wd);
  pi -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  p[i] = pi;
  if (pb) pb[i] = f2bf(pi);
}


// ---------------------------------------------------------------- network kernels
// The encoder and its heads on buffers laid out for them. A position is
// p = b L + l, P = B L of them. BF16 activations and gradients exist twice, as
// channel rows [C][Ps] (contiguous along the positions, Ps = P rounded up to
// 16, zero beyond P) and as position rows [P][Cs] (Cs = C rounded up to whole
// K tiles, zero beyond C), because the products contract over channels in one direction and
// over positions in the other: every operand row is then contiguous along the
// contraction and 16-byte aligned, whatever C, L and B are. Weights are packed
// to match (k_pack): forward [M rounded to 64][K rounded up, K = taps x
// channels], backward [tap][C rounded to 64][M rounded to 32], zero outside.
//
// Every product contracts in the order and the groups of 16 of k_gemm over an
// im2col matrix (k = 3 c + t forward, the channels per tap backward, the
// positions for the weights), so the results are its bits. (A network's
// outputs jump by 1e-5 when one BF16 weight or activation rounds the other
// way, so sums in another order show after a training step.)

__device__ __forceinline__ bf16x8 frag(const uint16_t *row, int k) { return *(const bf16x8 *)(row + k); }

// a + b, not fused with the product that made a: the residual is added to the
// rounded activation
__device__ __forceinline__ float add_alone(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

// K tiles in registers ahead of the one in LDS: a tile's MFMAs take 0.1 to 0.2
// us and its loads, of what another XCD has just written, up to 1 us. The loads
// of a ring are issued by every lane in every round, with their addresses
// clamped into the arrays (what a clamped lane reads is masked, or belongs to
// a row or column that is not stored): behind a condition the compiler cannot
// count what is in flight, and waits for all of it at each use.
constexpr int AHEAD = 4;
// f(place in the ring, tile) for n tiles, whole rounds of the ring without a
// condition between their tiles
template <int RING, class F> __device__ __forceinline__ void in_rounds(int n, F &&f) {
  int k = 0;
  for (; k + RING <= n; k += RING)
#pragma unroll
    for (int i = 0; i < RING; ++i) f(i, k + i);
#pragma unroll
  for (int i = 0; i < RING; ++i)
    if (k + i < n) f(i, k + i);
}

// threads of k_fwd and k_back: eight wavefronts, two per SIMD, one 32 x 32 block
// of the tile each (with four of 32 x 64 the epilogues' tanh chains had no
// second wavefront to fill in: 23 and 22 us instead of 19 and 18)
constexpr int NET_THREADS = 512;

// 16 bytes in registers (a vector type: arrays of the struct uint4 filled by
// plain copies ended up in scratch memory)
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 zero4() { return u32x4{0u, 0u, 0u, 0u}; }

// x[c, p] in FP32 -> both BF16 layouts of the first layer's input; the
// loss starts at zero when given
__global__ void k_input(const float *x, uint16_t *xb, uint16_t *xt, int C, int Cs, int P, int Ps, float *loss) {
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i == 0 && loss) *loss = 0.0f;
  if (i >= (long)C * P) return;
  const int c = (int)(i / P), p = (int)(i % P);
  const uint16_t v = f2bf(x[i]);
  if (xb) xb[(long)c * Ps + p] = v;
  xt[(long)p * Cs + c] = v;
}

// Forward product of one layer: M output channels x P positions.
// CONV: the kernel-3 convolution, taken straight from the position rows of
// the neighbours (no im2col matrix: it was written and read once per layer,
// 2 x 12.6 MB at 256 channels x 8192 positions), with bias, GELU and the
// residual in the epilogue. Otherwise a plain product over the channels
// (the heads' U and V).
// 64 x 128 tile per workgroup, 256 workgroups at 256 x 8192. 256 channels x 8192 positions, K = 768: im2col
// 13.3 + product 18.9 + bias and GELU 9.1 us -> 18.5 us.
template <bool CONV> __global__ __launch_bounds__(NET_THREADS) void k_fwd(ccp_nn_fwd_args g) {
  constexpr int BM = 64, BN = 128, KT = CONV ? 48 : 64, CH = CONV ? 16 : 64, ST = KT + 8;
  constexpr int NA = BM * KT / 8, RA = (NA + NET_THREADS - 1) / NET_THREADS; // 16-byte pieces of A, per thread
  constexpr int RB = BN * KT / 8 / NET_THREADS;                              // and of B (not CONV)
  constexpr int TS = BM + 4;                              // output rows staged for [P][Os]
  __shared__ __align__(16) uint16_t lds[2 * (BM + BN) * ST];
  static_assert(BN * TS <= (BM + BN) * ST, "the staged output fits one buffer's memory");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = (wave >> 2) * 32, wn = (wave & 3) * 32;
  struct {
    u32x4 a[RA];
    std::conditional_t<CONV, u32x2, u32x4> b[CONV ? 3 : RB];
  } ring[AHEAD];
  // CONV: this thread's position and which four of the tile's 16 channels
  const int bp = min(n0 + (tid >> 2), g.P - 1), bc = (tid & 3) * 4;
  const int bl = bp % g.L;
  const bool left = bl > 0, right = bl + 1 < g.L;
  auto load = [&](auto &t, int kt) {
#pragma unroll
    for (int u = 0; u < RA; ++u) {
      const int e = min(tid + u * NET_THREADS, NA - 1), m = m0 + e / (KT / 8), k = kt * KT + e % (KT / 8) * 8;
      // (CONV has one weight matrix, padded to whole tiles of rows)
      const uint16_t *a = CONV || m < g.M0 ? g.A0 + (long)m * g.Kp : g.A1 + (long)(min(m, g.M - 1) - g.M0) * g.Kp;
      t.a[u] = *(const u32x4 *)(a + k);
    }
    if constexpr (CONV) {
      const uint16_t *x = g.X + (long)bp * g.Cs + kt * CH + bc;
      t.b[0] = *(const u32x2 *)(x - (left ? g.Cs : 0));
      t.b[1] = *(const u32x2 *)x;
      t.b[2] = *(const u32x2 *)(x + (right ? g.Cs : 0));
    } else {
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        const int e = tid + u * NET_THREADS, p = min(n0 + e / (KT / 8), g.P - 1);
        t.b[u] = *(const u32x4 *)(g.X + (long)p * g.Cs + kt * CH + e % (KT / 8) * 8);
      }
    }
  };
  auto store = [&](const auto &t, uint16_t *As) {
    uint16_t *Bs = As + BM * ST;
#pragma unroll
    for (int u = 0; u < RA; ++u) {
      const int e = tid + u * NET_THREADS;
      if (e < NA) *(u32x4 *)(As + e / (KT / 8) * ST + e % (KT / 8) * 8) = t.a[u];
    }
    if constexpr (CONV) {
      // taps a, b, d of channels 0..3 interleaved: a0 b0 d0 a1 b1 d1 ...
      const u32x2 none = {0u, 0u}, x = left ? t.b[0] : none, y = right ? t.b[2] : none;
      const uint32_t a[2] = {x.x, x.y}, b[2] = {t.b[1].x, t.b[1].y}, d[2] = {y.x, y.y};
      uint32_t o[6];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        o[3 * i] = (a[i] & 0xffffu) | (b[i] << 16);
        o[3 * i + 1] = (d[i] & 0xffffu) | (a[i] & 0xffff0000u);
        o[3 * i + 2] = (b[i] >> 16) | (d[i] & 0xffff0000u);
      }
      u32x2 *w = (u32x2 *)(Bs + (tid >> 2) * ST + bc * 3);
#pragma unroll
      for (int i = 0; i < 3; ++i) w[i] = u32x2{o[2 * i], o[2 * i + 1]};
    } else {
#pragma unroll
      for (int u = 0; u < RB; ++u) {
        const int e = tid + u * NET_THREADS;
        *(u32x4 *)(Bs + e / (KT / 8) * ST + e % (KT / 8) * 8) = t.b[u];
      }
    }
  };
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  const int nk = g.Kp / KT, r = lane & 31, kq = 8 * (lane >> 5);
  // What the epilogue adds, before the loop: a load behind a store waits for
  // the store too, and one such wait per element was most of the kernel's time.
  float bias[16], res[16];
  if constexpr (CONV) {
    const float *from = g.res ? g.res : g.y; // (not added without g.res)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = min(m0 + wm + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3), g.M - 1);
      bias[v] = g.bias[m];
      res[v] = from[(long)m * g.Ps + min(n0 + wn + r, g.P - 1)];
    }
  }
#pragma unroll
  for (int d = 0; d < AHEAD; ++d) load(ring[d], min(d, nk - 1));
  // (a buffer is written again two tiles on, behind the barrier of the tile between)
  in_rounds<AHEAD>(nk, [&](int d, int kt) {
    uint16_t *As = lds + (d & 1) * (BM + BN) * ST, *Bs = As + BM * ST;
    store(ring[d], As);
    __syncthreads();
    load(ring[d], min(kt + AHEAD, nk - 1));
#pragma unroll
    for (int ks = 0; ks < KT; ks += 16)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(As + (wm + r) * ST, ks + kq), frag(Bs + (wn + r) * ST, ks + kq),
                                                    acc, 0, 0, 0);
  });
  __syncthreads();
  // D element v of lane l: row 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32.
  // The four rows of a v / 4 are staged together for the position rows.
  const int n = wn + r, p = n0 + n;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint16_t h[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int v = 4 * q + u, m = m0 + wm + 8 * q + 4 * (lane >> 5) + u;
      float o = acc[v], pre = 0.0f;
      if constexpr (CONV) {
        pre = o + bias[v];
        o = gelu(pre);
        if (g.res) o = add_alone(o, res[v]);
      }
      h[u] = m < g.M ? f2bf(o) : (uint16_t)0;
      if (p < g.P && m < g.M) {
        const long i = (long)m * g.Ps + p;
        if constexpr (CONV) {
          if (g.pre) g.pre[i] = pre;
          g.y[i] = o;
        }
        if (g.ob) g.ob[i] = h[u];
      }
    }
    *(u32x2 *)(lds + n * TS + wm + 8 * q + 4 * (lane >> 5)) =
        u32x2{h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16};
  }
  __syncthreads();
  if constexpr (CONV) {
    for (int e = tid; e < BN * BM / 4; e += NET_THREADS) {
      const int n = e / (BM / 4), m = m0 + e % (BM / 4) * 4, p = n0 + n;
      if (p < g.P && m < g.Os) *(u32x2 *)(g.ot + (long)p * g.Os + m) = *(const u32x2 *)(lds + n * TS + (m - m0));
    }
  } else {
    // (rows from M0 on go to column O1 of the position rows)
    for (int e = tid; e < BN * BM; e += NET_THREADS) {
      const int n = e / BM, m = m0 + e % BM, p = n0 + n;
      if (p < g.P && m < g.M) g.ot[(long)p * g.Os + (m < g.M0 ? m : g.O1 + m - g.M0)] = lds[n * TS + (m - m0)];
    }
  }
}

// Contact map of sample b from the position rows of U (columns 0 .. d) and V
// (columns ds ..): S = (M + M^T) / 2 + dist[|i - j|] + c0, M = alpha U^T V.
// One 32 x 32 block of S per wavefront; the transposed block is a second
// product with U and V exchanged (the same products in the same order), so M
// is neither stored nor read back. 64 samples of 128 x 128, d = 64: 8.1 -> 7.6 us
// with the distance terms loaded ahead and four groups in flight, not two.
struct PairFrags {
  bf16x8 ui, vi, uj, vj;
};
__global__ __launch_bounds__(256) void k_pair(const uint16_t *__restrict__ uv, int ds, int Os, const float *dist,
                                              const float *c0, float *S, int L, float alpha) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nt = (L + 31) / 32, t = blockIdx.x * 4 + wave;
  if (t >= nt * nt) return;
  const int i0 = t / nt * 32, j0 = t % nt * 32, b = blockIdx.y;
  const int r = lane & 31, kq = 8 * (lane >> 5);
  const long p0 = (long)b * L;
  // (rows past the sample's last: its values, for results that are not stored)
  const uint16_t *ri = uv + (p0 + min(i0 + r, L - 1)) * Os + kq, *rj = uv + (p0 + min(j0 + r, L - 1)) * Os + kq;
  f32x16 m, mt;
#pragma unroll
  for (int v = 0; v < 16; ++v) m[v] = mt[v] = 0.0f;
  const int nk = ds / 16;
  PairFrags ring[4];
  auto load = [&](PairFrags &t, int k) {
    t.ui = *(const bf16x8 *)(ri + 16 * k);
    t.vi = *(const bf16x8 *)(ri + ds + 16 * k);
    t.uj = *(const bf16x8 *)(rj + 16 * k);
    t.vj = *(const bf16x8 *)(rj + ds + 16 * k);
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) load(ring[i], min(i, nk - 1));
  // the distance terms before the stores: a load behind a store waits for it
  const int col = j0 + r;
  const float c = c0[0];
  float far[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int d = i0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3) - col;
    far[v] = dist[min(d < 0 ? -d : d, L - 1)];
  }
  in_rounds<4>(nk, [&](int i, int k) {
    m = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i].ui, ring[i].vj, m, 0, 0, 0);
    mt = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i].vi, ring[i].uj, mt, 0, 0, 0);
    load(ring[i], min(k + 4, nk - 1));
  });
  if (col >= L) return;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = i0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
    if (row >= L) continue;
    const float a = alpha * m[v], at_ = alpha * mt[v];
    S[((long)b * L + row) * L + col] = 0.5f * (a + at_) + far[v] + c;
  }
}

// mean over l of h[c, b L + l], summed in order, in BF16 as pb[C][Bs] and pt[B][Cs].
// A workgroup brings POOL_ROWS of the rows (c, b) into LDS in whole lines,
// then one lane adds each. 16384 rows of 128: 4.6 us (a lane reading its own row
// 18 us; with two 64-bit divisions for each value's place 9.5 us).
constexpr int POOL_ROWS = 32, POOL_SEG = 128;
__global__ __launch_bounds__(256) void k_pool(const float *h, uint16_t *pb, uint16_t *pt, int C, int B, int L, int Ps,
                                              int Bs, int Cs) {
  __shared__ float s[POOL_ROWS][POOL_SEG + 1];
  __shared__ long place[POOL_ROWS]; // of a row's first value
  const long rows = (long)C * B, r0 = (long)blockIdx.x * POOL_ROWS;
  float sum = 0.0f;
  if (threadIdx.x < POOL_ROWS) {
    const long i = min(r0 + (long)threadIdx.x, rows - 1);
    place[threadIdx.x] = i / B * Ps + i % B * L;
  }
  for (int l0 = 0; l0 < L; l0 += POOL_SEG) {
    const int n = min(POOL_SEG, L - l0);
    __syncthreads();
    // all of a thread's values in flight together (places past a row's end: its
    // last value, which is not added)
    constexpr int STEP = 256 / POOL_SEG, EACH = POOL_ROWS / STEP;
    const int l = threadIdx.x % POOL_SEG, row = threadIdx.x / POOL_SEG;
    float v[EACH];
#pragma unroll
    for (int k = 0; k < EACH; ++k) v[k] = h[place[row + k * STEP] + min(l0 + l, L - 1)];
#pragma unroll
    for (int k = 0; k < EACH; ++k) s[row + k * STEP][l] = v[k];
    __syncthreads();
    if (threadIdx.x < POOL_ROWS) {
      int l = 0;
      for (; l + 16 <= n; l += 16) {
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = s[threadIdx.x][l + j];
#pragma unroll
        for (int j = 0; j < 16; ++j) sum += v[j];
      }
      for (; l < n; ++l) sum += s[threadIdx.x][l];
    }
  }
  const long i = r0 + threadIdx.x;
  if (threadIdx.x >= POOL_ROWS || i >= rows) return;
  sum /= (float)L;
  const int c = (int)(i / B), b = (int)(i % B);
  pb[(long)c * Bs + b] = pt[(long)b * Cs + c] = f2bf(sum);
}

// C[m][n] = sum over k of A[m][k] B[n][k] for the radial head (rows of K, a
// multiple of 16, zero where unused; C's rows ldc apart): one 32 x 32 block per
// wavefront, operands straight from memory, four groups of 16 ahead. (k_gemm
// takes 11 us for 32 x 64 outputs, one workgroup's chain of loads; this 4.1.)
__global__ __launch_bounds__(64) void k_small(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B, float *C,
                                              int M, int N, int K, int lda, int ldb, int ldc) {
  const int lane = threadIdx.x, r = lane & 31, kq = 8 * (lane >> 5);
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
  const uint16_t *a = A + (long)min(m0 + r, M - 1) * lda + kq, *b = B + (long)min(n0 + r, N - 1) * ldb + kq;
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  struct {
    bf16x8 x, y;
  } ring[4];
  auto load = [&](auto &t, int k) {
    t.x = *(const bf16x8 *)(a + 16 * k);
    t.y = *(const bf16x8 *)(b + 16 * k);
  };
  const int nk = K / 16;
#pragma unroll
  for (int i = 0; i < 4; ++i) load(ring[i], min(i, nk - 1));
  in_rounds<4>(nk, [&](int i, int k) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i].x, ring[i].y, acc, 0, 0, 0);
    load(ring[i], min(k + 4, nk - 1));
  });
  const int n = n0 + r;
  if (n >= N) return;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int m = m0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
    if (m < M) C[(long)m * ldc + n] = acc[v];
  }
}

// Loss of the pair maps over the pairs r <= c (mean squared error, weight w)
// and its gradient with respect to the raw map, dLoss/dM(r, c) = g(lo, hi) / 2
// off the diagonal and g(r, r) on it, as BF16 rows of Ls entries; the sums of
// g along each diagonal of the band as a partial of gdist. One workgroup per
// sample and band of PL_ROWS rows. A lane takes one diagonal for the upper
// triangle (consecutive lanes read consecutive columns), or one column for
// the lower one, whose PL_ROWS values lie side by side in that column's row:
// at 128 bins each of 256 lanes has one of them, 14.6 us for 64 samples (16.3
// with the columns behind the diagonals on half the lanes).
constexpr int PL_ROWS = 16;
__global__ __launch_bounds__(256) void k_pair_grad(const float *pred, const float *target, uint16_t *graw, float *gdist,
                                                   float *gc0, float *loss, int L, int Ls, int B, float w) {
  const int b = blockIdx.y, r0 = blockIdx.x * PL_ROWS, r1 = min(r0 + PL_ROWS, L);
  const long base = (long)b * L * L;
  const float count = (float)B * L * (L + 1) / 2;
  float sq = 0.0f, all = 0.0f;
  float *gd = gdist + ((long)b * gridDim.x + blockIdx.x) * L;
  // (a band's values are loaded together: places past the sample's last are
  // read from it and left out)
  float x[PL_ROWS], y[PL_ROWS];
  // the band's diagonals, then its columns, from the next whole wavefront on
  const int cols = (L + 63) / 64 * 64;
  for (int e = threadIdx.x; e < cols + r1; e += 256) {
    if (e < cols) {
      const int d = e;
      if (d >= L) continue;
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < PL_ROWS; ++i) {
        const long u = base + (long)min(r0 + i, L - 1) * L + min(r0 + i + d, L - 1);
        x[i] = pred[u];
        y[i] = target[u];
      }
#pragma unroll
      for (int i = 0; i < PL_ROWS; ++i) {
        const int r = r0 + i;
        if (r + d >= L) continue;
        const float e = x[i] - y[i];
        const float g = 2.0f * w * e / count;
        sum += g;
        sq += w * e * e / count;
        graw[((long)b * L + r) * Ls + r + d] = f2bf(d == 0 ? g : 0.5f * g);
      }
      gd[d] = sum;
      all += sum;
    } else {
      const int c = e - cols;
#pragma unroll
      for (int i = 0; i < PL_ROWS; ++i) {
        const long u = base + (long)c * L + min(r0 + i, L - 1);
        x[i] = pred[u];
        y[i] = target[u];
      }
#pragma unroll
      for (int i = 0; i < PL_ROWS; ++i) {
        const int r = r0 + i;
        if (r <= c || r >= r1) continue;
        const float e = x[i] - y[i];
        const float g = 2.0f * w * e / count;
        graw[((long)b * L + r) * Ls + c] = f2bf(0.5f * g);
      }
    }
  }
  __shared__ float red[2][EW];
  red[0][threadIdx.x] = sq;
  red[1][threadIdx.x] = all;
  __syncthreads();
  for (int o = EW / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      red[0][threadIdx.x] += red[0][threadIdx.x + o];
      red[1][threadIdx.x] += red[1][threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    atomicAdd(loss, red[0][0]);
    gc0[(long)b * gridDim.x + blockIdx.x] = red[1][0];
  }
}

// Radial head as k_rd_loss, one wavefront per output: the bias gradient of an
// output is one sum (2048 atomics on 32 words took 37 us, this 4.9 us).
__global__ __launch_bounds__(1024) void k_rd_grad(float *pred, const float *bias, const float *target, uint16_t *gb,
                                                  uint16_t *gt, float *dbias, float *loss, int O, int Bn, int Bs,
                                                  int Os, float w) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float count = (float)O * Bn;
  float sq = 0.0f;
  for (int o = wave; o < O; o += 16) {
    float sum = 0.0f;
    for (int b = lane; b < Bn; b += 64) {
      const int i = o * Bn + b;
      const float v = pred[i] + bias[o];
      pred[i] = v;
      const float e = v - target[i];
      const float gi = 2.0f * w * e / count;
      gb[(long)o * Bs + b] = gt[(long)b * Os + o] = f2bf(gi);
      sq += w * e * e / count;
      sum += gi;
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) sum += __shfl_xor(sum, s);
    if (lane == 0) dbias[o] += sum;
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) sq += __shfl_xor(sq, s);
  __shared__ float red[16];
  if (lane == 0) red[wave] = sq;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.0f;
    for (int k = 0; k < 16; ++k) t += red[k];
    atomicAdd(loss, t);
  }
}

// Gradients of U and V of sample b: dU(c, i) = alpha sum_j V(c, j) graw(i, j)
// in rows 0 .. d, dV(c, j) = alpha sum_i U(c, i) graw(i, j) in rows d .. 2 d
// (graw is symmetric, so both contract along its rows, of Ls = L rounded up to
// 8 entries). uvb holds U then V as [2 d][Ps]. One 32 x 32 block per
// wavefront, operands straight from memory (a sample's 32 KB are read by its
// few wavefronts only); 16-byte loads where samples are whole groups of 16.
__global__ __launch_bounds__(256) void k_duv(const uint16_t *__restrict__ uvb, const uint16_t *__restrict__ graw,
                                             uint16_t *db, uint16_t *dt, int d, int ds, int L, int Ls, int Ps, int Os,
                                             float alpha) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nm = (2 * d + 31) / 32, nn = (L + 31) / 32, t = blockIdx.x * 4 + wave;
  if (t >= nm * nn) return;
  const int m0 = t / nn * 32, n0 = t % nn * 32, b = blockIdx.y;
  const int r = lane & 31, kq = 8 * (lane >> 5);
  const int m = m0 + r, n = n0 + r;
  // row m of the result takes row (m + d) mod 2 d of U, V (rows and columns
  // past the last: its values, for results that are not stored)
  const int mc = min(m, 2 * d - 1);
  const uint16_t *a = uvb + (long)(mc < d ? mc + d : mc - d) * Ps + (long)b * L;
  const uint16_t *q = graw + ((long)b * L + min(n, L - 1)) * Ls;
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  const int nk = (L + 15) / 16;
  if (L % 16 == 0) {
    struct {
      bf16x8 x, y;
    } ring[4];
    auto load = [&](auto &t, int k) {
      t.x = *(const bf16x8 *)(a + 16 * k + kq);
      t.y = *(const bf16x8 *)(q + 16 * k + kq);
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) load(ring[i], min(i, nk - 1));
    in_rounds<4>(nk, [&](int i, int k) {
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ring[i].x, ring[i].y, acc, 0, 0, 0);
      load(ring[i], min(k + 4, nk - 1));
    });
  } else {
    union Frag {
      uint16_t e[8];
      bf16x8 f;
    };
    for (int k = 0; k < nk; ++k) {
      Frag x, y;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int i = 16 * k + kq + j;
        x.e[j] = i < L ? a[i] : (uint16_t)0;
        y.e[j] = i < L ? q[i] : (uint16_t)0;
      }
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.f, y.f, acc, 0, 0, 0);
    }
  }
  if (n >= L) return;
  const long p = (long)b * L + n;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = m0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
    if (row >= 2 * d) continue;
    const uint16_t h = f2bf(alpha * acc[v]);
    db[(long)row * Ps + p] = h;
    dt[p * Os + (row < d ? row : ds + row - d)] = h;
  }
}

// Gradient with respect to a layer's activations h (C channels x P
// positions), with the layer's GELU derivative and bias gradient in the
// epilogue.
// HEAD: dh = Wv^T dV + Wu^T dU + dpooled / L; otherwise dh += the adjoint of
// the next layer's convolution, one accumulator per tap (source position
// p + 1 - t, nothing across a sample's ends), added in tap order. Then
// g = dh gelu'(pre) in both BF16 layouts, and the sums of g over the tile's
// positions as a partial of the bias gradient.
// Without it each layer's product wrote 3 C x P floats (25 MB at 256 x 8192)
// for col2im to read back, and the derivative was another pass:
// 39 + 10.4 + 27.6 us -> 17.5 us.
template <bool HEAD> __global__ __launch_bounds__(NET_THREADS) void k_back(ccp_nn_back_args g) {
  constexpr int BM = 64, BN = 128, KT = 32, ST = KT + 8, NT = HEAD ? 2 : 3, TS = BM + 4;
  constexpr int ROWS = HEAD ? 2 * BN : BN + 2; // rows of G staged: both halves, or one more on each side
  constexpr int NA = NT * BM * KT / 8, RA = (NA + NET_THREADS - 1) / NET_THREADS;
  constexpr int NB = ROWS * KT / 8, RB = (NB + NET_THREADS - 1) / NET_THREADS;
  constexpr int BUF = (NT * BM + ROWS) * ST;
  __shared__ __align__(16) uint16_t lds[2 * BUF];
  __shared__ float s_bias[4][BM];
  static_assert(BN * TS <= BUF, "the staged output fits one buffer's memory");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int wm = (wave >> 2) * 32, wn = (wave & 3) * 32;
  struct {
    u32x4 a[RA], b[RB];
  } ring[AHEAD];
  auto load = [&](auto &t, int kt) {
#pragma unroll
    for (int u = 0; u < RA; ++u) {
      const int e = min(tid + u * NET_THREADS, NA - 1), row = e / (KT / 8), k = e % (KT / 8) * 8;
      t.a[u] = *(const u32x4 *)(g.W + ((long)(row / BM) * g.Cr + m0 + row % BM) * g.Kr + kt * KT + k);
    }
#pragma unroll
    for (int u = 0; u < RB; ++u) {
      const int e = min(tid + u * NET_THREADS, NB - 1), row = e / (KT / 8), k = kt * KT + e % (KT / 8) * 8;
      const int p = min(max(n0 + (HEAD ? row % BN : row - 1), 0), g.P - 1);
      t.b[u] = *(const u32x4 *)(g.G + (long)p * g.Gs + (HEAD && row >= BN ? g.V1 : 0) + k);
    }
  };
  f32x16 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;
  const int nk = g.Kr / KT, r = lane & 31, kq = 8 * (lane >> 5);
  // whether the source of the first (p + 1) and the last tap (p - 1) lies in the sample
  const int l = (n0 + wn + r) % g.L;
  const bool edge[2] = {l + 1 < g.L, l > 0};
  // the epilogue's inputs, ahead of its stores (see k_fwd)
  float pre[16], add[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int c = min(m0 + wm + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3), g.C - 1), p = min(n0 + wn + r, g.P - 1);
    pre[v] = g.pre[(long)c * g.Ps + p];
    add[v] = HEAD ? g.dpooled[(long)c * g.B + p / g.L] : g.dh[(long)c * g.Ps + p];
  }
#pragma unroll
  for (int d = 0; d < AHEAD; ++d) load(ring[d], min(d, nk - 1));
  in_rounds<AHEAD>(nk, [&](int i, int kt) {
    uint16_t *As = lds + (i & 1) * BUF, *Bs = As + NT * BM * ST;
#pragma unroll
    for (int u = 0; u < RA; ++u) {
      const int e = tid + u * NET_THREADS;
      if (e < NA) *(u32x4 *)(As + e / (KT / 8) * ST + e % (KT / 8) * 8) = ring[i].a[u];
    }
#pragma unroll
    for (int u = 0; u < RB; ++u) {
      const int e = tid + u * NET_THREADS;
      if (e < NB) *(u32x4 *)(Bs + e / (KT / 8) * ST + e % (KT / 8) * 8) = ring[i].b[u];
    }
    __syncthreads();
    load(ring[i], min(kt + AHEAD, nk - 1));
#pragma unroll
    for (int ks = 0; ks < KT; ks += 16)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        bf16x8 x = frag(Bs + (wn + r + (HEAD ? t * BN : 2 - t)) * ST, ks + kq);
        if (!HEAD && t != 1) {
          const bf16x8 none = {};
          x = edge[t == 0 ? 0 : 1] ? x : none;
        }
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(As + (t * BM + wm + r) * ST, ks + kq), x, acc[t], 0, 0, 0);
      }
  });
  __syncthreads();
  float part[16];
  const int n = wn + r, p = n0 + n;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint16_t h[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int v = 4 * q + u, c = m0 + wm + 8 * q + 4 * (lane >> 5) + u;
      const bool ok = p < g.P && c < g.C;
      float d;
      if constexpr (HEAD) {
        d = acc[1][v] + acc[0][v];
        d += add[v] / (float)g.L;
      } else {
        d = acc[0][v];
        d += acc[1][v];
        d += acc[2][v];
        d += add[v];
      }
      const float gi = d * gelu_grad(pre[v]);
      part[v] = ok ? gi : 0.0f;
      h[u] = c < g.C ? f2bf(gi) : (uint16_t)0;
      if (ok) {
        const long i = (long)c * g.Ps + p;
        if (g.keep) g.dh[i] = d;
        g.gb[i] = h[u];
      }
    }
    *(u32x2 *)(lds + n * TS + wm + 8 * q + 4 * (lane >> 5)) =
        u32x2{h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16};
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    float s = part[v];
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (r == 0) s_bias[wave & 3][wm + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)] = s;
  }
  __syncthreads();
  if (tid < BM && m0 + tid < g.C) g.dbias[(long)blockIdx.x * g.C + m0 + tid] = (s_bias[0][tid] + s_bias[1][tid]) + (s_bias[2][tid] + s_bias[3][tid]);
  for (int e = tid; e < BN * BM / 4; e += NET_THREADS) {
    const int n = e / (BM / 4), m = m0 + e % (BM / 4) * 4, p = n0 + n;
    if (p < g.P && m < g.Cs) *(u32x2 *)(g.gt + (long)p * g.Cs + m) = *(const u32x2 *)(lds + n * TS + (m - m0));
  }
}

// Weight gradients of every layer in one launch (table): dst[m][TAPS c + t] +=
// sum over p of G[m, p] X[c, p + t - 1] (three taps, nothing across a sample's
// ends) or G[m, p] X[c, p] (one). One wavefront takes 32 rows m and 32 channels
// c, all taps: both operands' rows are contiguous along p, so a lane's eight
// values of a group of 16 positions are one 16-byte load into the registers
// the MFMA reads, and the neighbours' taps are that load shifted by one
// element, the odd one from the other half of the wavefront. No LDS: staged
// through it, one tap per wavefront, the tiles' reads alone were twice its
// bandwidth. A wavefront's sums are a chain of P / 16 MFMAs a tap (32 cycles
// each); the loads of WG_AHEAD groups are in flight.
// A layer alone is 64 such chains on 1024 SIMDs, but no gradient is needed
// before the optimizer, so all layers and the heads go together. The positions
// are not split: that would fill the chip from one layer, but change the order
// of the sums. 256 channels x 8192 positions, six layers and the heads:
// 6 x 165 us (k_gemm, 48 workgroups gathering two bytes at a time) -> 95 us.
constexpr int WG_AHEAD = 8;
// (pointers from a table are generic ones to the compiler, whose loads count
// with the LDS ones and cannot be waited for one by one)
typedef __attribute__((address_space(1))) uint8_t global_u8;
typedef __attribute__((address_space(1))) uint16_t global_u16;
typedef __attribute__((address_space(1))) float global_f32;
typedef __attribute__((address_space(1))) u32x4 global_u32x4;
__device__ __forceinline__ uint32_t other_half(uint32_t v) { return (uint32_t)__shfl_xor((int)v, 32); }
// ALIGNED: samples of a multiple of 8 positions. OFF: the lane's byte offset
// from a tile's first row, 32 bits on a scalar base so that a load needs no
// address arithmetic, while 31 rows lie within them (Ps below 2^26)
template <int TAPS, bool ALIGNED, class OFF>
__device__ __forceinline__ void wgrad_tile(const ccp_nn_wgrad_job &J, int m0, int c0, int L) {
  const int P = J.P, Ps = J.Ps;
  const int lane = threadIdx.x, r = lane & 31, half = lane >> 5;
  // this lane's offset from the tile's first row of each matrix (rows past the
  // last: its values, for results that are not stored)
  const OFF go = ((OFF)(min(m0 + r, J.M - 1) - m0) * (OFF)Ps + 8u * half) * 2u;
  const OFF xo = ((OFF)(min(c0 + r, J.C - 1) - c0) * (OFF)Ps + 8u * half) * 2u;
  const global_u16 *G = (const global_u16 *)J.G + (long)m0 * Ps, *X = (const global_u16 *)J.X + (long)c0 * Ps;
  union Frag {
    u32x4 u;
    uint16_t e[8];
    bf16x8 f;
  };
  f32x16 acc[TAPS];
#pragma unroll
  for (int t = 0; t < TAPS; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;
  Frag a[WG_AHEAD], b[WG_AHEAD];
  uint32_t next[WG_AHEAD]; // three taps: the element after the lane's own eight
  const int groups = (P + 15) / 16;
  // (the element after the last position is masked: the row's padding, or past
  // the last row of all the position's own element)
  auto load = [&](int i, int k) {
    const global_u8 *g = (const global_u8 *)(G + 16 * k), *x = (const global_u8 *)(X + 16 * k);
    a[i].u = *(const global_u32x4 *)(g + go);
    b[i].u = *(const global_u32x4 *)(x + xo);
    if (TAPS == 3) next[i] = *(const global_u16 *)(x + (16 * k + 16 < Ps ? 16 : 14) + xo);
  };
#pragma unroll
  for (int i = 0; i < WG_AHEAD; ++i) load(i, min(i, groups - 1));
  uint32_t last = 0; // element before the group, in the lower half
  int l0 = 8 * half % L;  // place of the lane's first element in its sample
  const int step = 16 % L;
  in_rounds<WG_AHEAD>(groups, [&](int i, int k) {
    if constexpr (TAPS == 3) {
      const u32x4 x = b[i].u;
      // upper half: the element before is the lower half's last one; lower
      // half: the element after is the upper half's first one, the element
      // before the upper half's last one of the group before
      const uint32_t sw = other_half(x.w >> 16 | x.x << 16);
      const uint32_t before = half ? sw & 0xffffu : last, after = half ? next[i] : sw >> 16;
      last = sw & 0xffffu;
      Frag lo, hi;
      lo.u = u32x4{x.x << 16 | before, x.y << 16 | x.x >> 16, x.z << 16 | x.y >> 16, x.w << 16 | x.z >> 16};
      hi.u = u32x4{x.x >> 16 | x.y << 16, x.y >> 16 | x.z << 16, x.z >> 16 | x.w << 16,
                        x.w >> 16 | after << 16};
      if (ALIGNED) { // a sample starts only at a lane's first element and ends only at its last
        if (l0 == 0) lo.u.x &= 0xffff0000u;
        if (l0 + 8 == L) hi.u.w &= 0xffffu;
      } else {
        int l = l0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          lo.e[j] = l == 0 ? (uint16_t)0 : lo.e[j];
          hi.e[j] = l == L - 1 ? (uint16_t)0 : hi.e[j];
          l = l + 1 == L ? 0 : l + 1;
        }
      }
      l0 += step;
      l0 = l0 >= L ? l0 - L : l0;
      acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i].f, lo.f, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i].f, b[i].f, acc[1], 0, 0, 0);
      acc[2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i].f, hi.f, acc[2], 0, 0, 0);
    } else {
      acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i].f, b[i].f, acc[0], 0, 0, 0);
    }
    load(i, min(k + WG_AHEAD, groups - 1));
  });
  const int N = TAPS * J.C, n = TAPS * (c0 + r);
  if (c0 + r >= J.C) return;
  float old[TAPS][16];
#pragma unroll
  for (int t = 0; t < TAPS; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = m0 + 8 * (v >> 2) + 4 * half + (v & 3);
      const int mc = min(m, J.M - 1);
      const global_f32 *d = (const global_f32 *)(mc < J.M0 ? J.dst0 + (long)mc * N : J.dst1 + (long)(mc - J.M0) * N);
      old[t][v] = d[n + t];
    }
#pragma unroll
  for (int t = 0; t < TAPS; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = m0 + 8 * (v >> 2) + 4 * half + (v & 3);
      global_f32 *d = (global_f32 *)(m < J.M0 ? J.dst0 + (long)m * N : J.dst1 + (long)(m - J.M0) * N);
      if (m < J.M) d[n + t] = acc[t][v] + old[t][v];
    }
}
template <class OFF>
__global__ __launch_bounds__(64) void k_wgrad(const ccp_nn_wgrad_job *tab, const int *first, int n_jobs, int L) {
  // Workgroups go round-robin over the 8 XCDs: each XCD takes a run of tiles,
  // so the rows that a layer's tiles share stay in one or two L2s.
  const int n_wg = (int)gridDim.x, x = (int)blockIdx.x % 8, q = n_wg / 8, rem = n_wg % 8;
  const int bid = (x < rem ? x * (q + 1) : rem * (q + 1) + (x - rem) * q) + (int)blockIdx.x / 8;
  int job = 0;
  while (job + 1 < n_jobs && bid >= first[job + 1]) ++job;
  const ccp_nn_wgrad_job J = tab[job];
  const int nc = (J.C + 31) / 32, tile = bid - first[job];
  const int m0 = tile / nc * 32, c0 = tile % nc * 32;
  if (J.taps == 1) wgrad_tile<1, true, OFF>(J, m0, c0, L);
  else if (L % 8 == 0) wgrad_tile<3, true, OFF>(J, m0, c0, L);
  else wgrad_tile<3, false, OFF>(J, m0, c0, L);
}

// dst[i] += sum over parts of src[s stride + i], for every segment of the
// table (blockIdx.y): 64 results per workgroup, sixteen lanes each taking
// every sixteenth part, in a fixed order.
__global__ __launch_bounds__(1024) void k_reduce(const ccp_nn_segment *seg) {
  const ccp_nn_segment s = seg[blockIdx.y];
  const int q = threadIdx.x >> 6, k = threadIdx.x & 63;
  __shared__ float red[16][64];
  for (long i0 = (long)blockIdx.x * 64; i0 < s.n; i0 += (long)gridDim.x * 64) {
    const long i = i0 + k;
    float v = 0.0f;
    if (i < s.n) {
      long u = q;
      for (; u + 48 < s.parts; u += 64) {
        const float a = s.src[u * s.stride + i], b = s.src[(u + 16) * s.stride + i],
                    c = s.src[(u + 32) * s.stride + i], d = s.src[(u + 48) * s.stride + i];
        v += (a + b) + (c + d);
      }
      for (; u < s.parts; u += 16) v += s.src[u * s.stride + i];
    }
    __syncthreads();
    red[q][k] = v;
    __syncthreads();
    if (q == 0 && i < s.n) {
      float t = 0.0f;
#pragma unroll
      for (int w = 0; w < 16; ++w) t += red[w][k];
      s.dst[i] += t;
    }
  }
}

// BF16 copies of every weight matrix (table, blockIdx.y): as it is, packed
// for k_fwd and packed for k_back, which is the transpose: tiles of 64 rows x
// 48 columns through LDS, so that both ends are read and written in runs.
constexpr int PK_M = 64, PK_K = 48;
__global__ __launch_bounds__(256) void k_pack(const ccp_nn_weight *tab) {
  const ccp_nn_weight t = tab[blockIdx.y];
  const int K = t.taps * t.C, nk = (K + PK_K - 1) / PK_K, tiles = nk * ((t.M + PK_M - 1) / PK_M);
  __shared__ uint16_t s[PK_K][PK_M + 2];
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const int m0 = tile / nk * PK_M, k0 = tile % nk * PK_K;
    __syncthreads();
    for (int e = threadIdx.x; e < PK_M * PK_K; e += 256) {
      const int m = m0 + e / PK_K, k = k0 + e % PK_K;
      if (m >= t.M || k >= K) continue;
      const uint16_t h = f2bf(t.w[(long)m * K + k]);
      ((uint16_t *)t.wb)[(long)m * K + k] = h;
      if (t.fwd) ((uint16_t *)t.fwd)[(long)m * t.Kp + k] = h;
      s[e % PK_K][e / PK_K] = h;
    }
    __syncthreads();
    if (!t.back) continue;
    for (int e = threadIdx.x; e < PK_M * PK_K; e += 256) {
      const int m = m0 + e % PK_M, k = k0 + e / PK_M;
      if (m < t.M && k < K)
        ((uint16_t *)t.back)[((long)(k % t.taps) * t.Cr + k / t.taps) * t.Kr + m] = s[e / PK_M][e % PK_M];
    }
  }
}

// launch(first sample, samples) for B samples, as many as a grid's second
// dimension takes at a time
template <class F> void in_samples(int B, F &&launch) {
  constexpr int MOST = 65535;
  for (int b = 0; b < B; b += MOST) launch((long)b, (unsigned)(B - b < MOST ? B - b : MOST));
}

// k_adamw over one flat run of parameters, decay on the first n_decay
__global__ void k_adamw_flat(float *p, const float *g, float *m, float *v, long n, long n_decay, float lr, float b1,
                             float b2, float eps, float wd, float c1, float c2) {
  const long i = (long)blockIdx.x * EW + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  float pi = p[i] * (1.0f - lr * (i < n_decay ? wd : 0.0f));
  pi -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  p[i] = pi;
}

} // namespace

extern "C" {

int ccp_nn_gemm(const void *A, const void *B, float *C, void *Cb, int M, int N, int K, int batch, long sab, long sam,
                long sak, long sbb, long sbk, long sbn, long scb, long scm, long scn, float alpha, float beta,
                void *stream) {
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0 || (!C && !Cb) || (beta != 0.0f && !C)) return 1;
  const dim3 grid((unsigned)((N + TN - 1) / TN), (unsigned)((M + TM - 1) / TM), (unsigned)batch);
  k_gemm<<<grid, GEMM_THREADS, 0, (hipStream_t)stream>>>((const uint16_t *)A, (const uint16_t *)B, C,
                                                         (uint16_t *)Cb, M, N, K, sab, sam, sak, sbb, sbk, sbn, scb,
                                                         scm, scn, alpha, beta);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_im2col(const void *x, void *cols, int C, int Bn, int L, void *stream) {
  const long n = (long)C * 3 * Bn * L;
  k_im2col<<<grid_for(n), EW, 0, (hipStream_t)stream>>>((const uint16_t *)x, (uint16_t *)cols, C, Bn, L);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_col2im(const float *dcols, float *dx, int C, int Bn, int L, float beta, void *stream) {
  const long n = (long)C * Bn * L;
  k_col2im<<<grid_for(n), EW, 0, (hipStream_t)stream>>>(dcols, dx, C, Bn, L, beta);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_bias_gelu(float *pre, const float *bias, const float *res, float *y, void *yb, int C, long P,
                     void *stream) {
  k_bias_gelu<<<grid_for((long)C * P), EW, 0, (hipStream_t)stream>>>(pre, bias, res, y, (uint16_t *)yb, C, P);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_gelu_back(const float *pre, const float *dy, float *g, void *gb, float *dbias, int C, long P,
                     void *stream) {
  const unsigned bx = (unsigned)((P + EW - 1) / EW < 64 ? (P + EW - 1) / EW : 64);
  k_gelu_back<<<dim3(bx, (unsigned)C), EW, 0, (hipStream_t)stream>>>(pre, dy, g, (uint16_t *)gb, dbias, C, P);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_pair_map(const float *raw, const float *dist, const float *c0, float *pred, int L, int Bn, void *stream) {
  k_pair_map<<<grid_for((long)Bn * L * L), EW, 0, (hipStream_t)stream>>>(raw, dist, c0, pred, L, Bn);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_pair_loss(const float *pred, const float *target, float *gS, float *graw, void *grawb, float *gdist,
                     float *gc0, float *loss, int L, int Bn, float w, void *stream) {
  k_pair_loss<<<(unsigned)(Bn * L), EW, 0, (hipStream_t)stream>>>(pred, target, gS, graw, (uint16_t *)grawb, loss, L,
                                                                  Bn, w);
  k_pair_reduce<<<(unsigned)L, EW, 0, (hipStream_t)stream>>>(gS, gdist, gc0, L, Bn);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_mean_pool(const float *h, float *pooled, void *pooledb, int C, int Bn, int L, void *stream) {
  k_mean_pool<<<grid_for((long)C * Bn), EW, 0, (hipStream_t)stream>>>(h, pooled, (uint16_t *)pooledb, C, Bn, L);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_pool_back(const float *dpooled, float *dh, int C, int Bn, int L, void *stream) {
  k_pool_back<<<grid_for((long)C * Bn * L), EW, 0, (hipStream_t)stream>>>(dpooled, dh, C, Bn, L);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_rd_loss(float *pred, const float *bias, const float *target, float *g, void *gb, float *dbias, float *loss,
                   int O, int Bn, float w, void *stream) {
  k_rd_loss<<<1, EW, 0, (hipStream_t)stream>>>(pred, bias, target, g, (uint16_t *)gb, dbias, loss, O, Bn, w);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_cast_bf16(const float *x, void *y, long n, void *stream) {
  k_cast<<<grid_for(n), EW, 0, (hipStream_t)stream>>>(x, (uint16_t *)y, n);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_adamw(float *p, const float *g, float *m, float *v, void *pb, long n, float lr, float b1, float b2,
                 float eps, float wd, int t, void *stream) {
  const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
  k_adamw<<<grid_for(n), EW, 0, (hipStream_t)stream>>>(p, g, m, v, (uint16_t *)pb, n, lr, b1, b2, eps, wd, c1, c2);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

// ---- network kernels
int ccp_nn_input(const float *x, void *xb, void *xt, int C, int Cs, int P, int Ps, float *loss, void *stream) {
  if (C <= 0 || P <= 0 || !x || !xt || Ps % 16 || Ps < P || Cs % 16 || Cs < C) return 1;
  k_input<<<grid_for((long)C * P), EW, 0, (hipStream_t)stream>>>(x, (uint16_t *)xb, (uint16_t *)xt, C, Cs, P, Ps, loss);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_fwd(const ccp_nn_fwd_args *a, int conv, void *stream) {
  if (!a || a->M <= 0 || a->P <= 0 || a->L <= 0 || a->Ps < a->P || a->Cs % 8 || a->Kp <= 0 ||
      a->Kp % (conv ? 48 : 64) || a->Cs < (conv ? a->Kp / 3 : a->Kp) || !a->A0 || !a->X || !a->ot || a->Os % 4)
    return 1;
  if (conv ? !a->y || !a->bias || a->Os < a->M : a->M0 <= 0 || a->M0 > a->M || (a->M0 < a->M && !a->A1)) return 1;
  const dim3 grid((unsigned)((a->P + 127) / 128), (unsigned)((a->M + 63) / 64));
  if (conv) k_fwd<true><<<grid, NET_THREADS, 0, (hipStream_t)stream>>>(*a);
  else k_fwd<false><<<grid, NET_THREADS, 0, (hipStream_t)stream>>>(*a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_pair(const void *uv, int d, const float *dist, const float *c0, float *S, int L, int B, float alpha,
                void *stream) {
  if (d <= 0 || d % 16 || L <= 0 || B <= 0) return 1;
  const unsigned nt = (unsigned)((L + 31) / 32);
  in_samples(B, [&](long b, unsigned n) {
    k_pair<<<dim3((nt * nt + 3) / 4, n), 256, 0, (hipStream_t)stream>>>((const uint16_t *)uv + b * L * 2 * d, d, 2 * d,
                                                                       dist, c0, S + b * L * L, L, alpha);
  });
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_pool(const float *h, void *pb, void *pt, int C, int B, int L, int Ps, int Bs, int Cs, void *stream) {
  if (C <= 0 || B <= 0 || L <= 0 || Ps < (long)B * L || Bs < B || Cs < C) return 1;
  const long rows = (long)C * B;
  k_pool<<<(unsigned)((rows + POOL_ROWS - 1) / POOL_ROWS), 256, 0, (hipStream_t)stream>>>(
      h, (uint16_t *)pb, (uint16_t *)pt, C, B, L, Ps, Bs, Cs);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_small(const void *A, const void *B, float *C, int M, int N, int K, int lda, int ldb, int ldc, void *stream) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 16 || lda < K || ldb < K || lda % 8 || ldb % 8 || ldc < N) return 1;
  k_small<<<dim3((unsigned)((N + 31) / 32), (unsigned)((M + 31) / 32)), 64, 0, (hipStream_t)stream>>>(
      (const uint16_t *)A, (const uint16_t *)B, C, M, N, K, lda, ldb, ldc);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_pair_bands(int L) { return (L + PL_ROWS - 1) / PL_ROWS; }

int ccp_nn_pair_grad(const float *pred, const float *target, void *graw, float *gdist, float *gc0, float *loss, int L,
                     int Ls, int B, float w, void *stream) {
  if (L <= 0 || Ls % 8 || Ls < L || B <= 0) return 1;
  const int bands = ccp_nn_pair_bands(L);
  in_samples(B, [&](long b, unsigned n) {
    k_pair_grad<<<dim3((unsigned)bands, n), EW, 0, (hipStream_t)stream>>>(
        pred + b * L * L, target + b * L * L, (uint16_t *)graw + b * L * Ls, gdist + b * bands * L, gc0 + b * bands,
        loss, L, Ls, B, w);
  });
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_rd_grad(float *pred, const float *bias, const float *target, void *gb, void *gt, float *dbias, float *loss,
                   int O, int Bn, int Bs, int Os, float w, void *stream) {
  if (O <= 0 || Bn <= 0 || Bs < Bn || Os < O) return 1;
  k_rd_grad<<<1, 1024, 0, (hipStream_t)stream>>>(pred, bias, target, (uint16_t *)gb, (uint16_t *)gt, dbias, loss, O, Bn,
                                                 Bs, Os, w);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_duv(const void *uvb, const void *graw, void *db, void *dt, int d, int ds, int L, int Ls, int B, int Ps,
               float alpha, void *stream) {
  if (d <= 0 || ds % 8 || ds < d || L <= 0 || Ls % 8 || Ls < L || B <= 0 || Ps % 8 || Ps < (long)B * L) return 1;
  const unsigned blocks = (unsigned)((2 * d + 31) / 32 * ((L + 31) / 32));
  in_samples(B, [&](long b, unsigned n) {
    k_duv<<<dim3((blocks + 3) / 4, n), 256, 0, (hipStream_t)stream>>>(
        (const uint16_t *)uvb + b * L, (const uint16_t *)graw + b * L * Ls, (uint16_t *)db + b * L,
        (uint16_t *)dt + b * L * 2 * ds, d, ds, L, Ls, Ps, 2 * ds, alpha);
  });
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_back(const ccp_nn_back_args *a, int head, void *stream) {
  if (!a || a->C <= 0 || a->P <= 0 || a->L <= 0 || a->Ps < a->P || a->Gs % 8 || a->Cs % 8 || a->Cs < a->C ||
      a->Cr % 64 || a->Cr < a->C || a->Kr <= 0 || a->Kr % 32 || !a->dh ||
      (head ? !a->dpooled || a->B <= 0 || a->V1 < a->Kr || a->V1 % 8 || a->V1 + a->Kr > a->Gs : a->Kr > a->Gs))
    return 1;
  const dim3 grid((unsigned)((a->P + 127) / 128), (unsigned)((a->C + 63) / 64));
  if (head) k_back<true><<<grid, NET_THREADS, 0, (hipStream_t)stream>>>(*a);
  else k_back<false><<<grid, NET_THREADS, 0, (hipStream_t)stream>>>(*a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_wgrad_tiles(int M, int C) { return (M + 31) / 32 * ((C + 31) / 32); }

int ccp_nn_wgrad(const ccp_nn_wgrad_job *tab, const int *first, int n_jobs, int n_tiles, int L, void *stream) {
  if (!tab || !first || n_jobs <= 0 || n_tiles <= 0 || L <= 0) return 1;
  k_wgrad<uint32_t><<<(unsigned)n_tiles, 64, 0, (hipStream_t)stream>>>(tab, first, n_jobs, L);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_wgrad_far(const ccp_nn_wgrad_job *tab, const int *first, int n_jobs, int n_tiles, int L, void *stream) {
  if (!tab || !first || n_jobs <= 0 || n_tiles <= 0 || L <= 0) return 1;
  k_wgrad<uint64_t><<<(unsigned)n_tiles, 64, 0, (hipStream_t)stream>>>(tab, first, n_jobs, L);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_reduce(const ccp_nn_segment *seg, int n, void *stream) {
  if (!seg || n <= 0) return 1;
  k_reduce<<<dim3(8, (unsigned)n), 1024, 0, (hipStream_t)stream>>>(seg);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_pack(const ccp_nn_weight *tab, int n, void *stream) {
  if (!tab || n <= 0) return 1;
  k_pack<<<dim3(64, (unsigned)n), 256, 0, (hipStream_t)stream>>>(tab);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int ccp_nn_adamw_flat(float *p, const float *g, float *m, float *v, long n, long n_decay, float lr, float b1, float b2,
                      float eps, float wd, int t, void *stream) {
  if (n <= 0 || n_decay < 0 || n_decay > n) return 1;
  const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
  k_adamw_flat<<<grid_for(n), EW, 0, (hipStream_t)stream>>>(p, g, m, v, n, n_decay, lr, b1, b2, eps, wd, c1, c2);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

} // extern "C"
