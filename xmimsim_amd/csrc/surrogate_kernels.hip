/*
 * surrogate_kernels.hip -- gfx950 kernels of the net-line surrogate: a
 * multilayer perceptron (log composition/thickness/density/energy -> log net
 * line intensities) trained on spectra of the GPU Monte Carlo.
 *
 * Every product is one kernel shape, C[M x N] = A[M x K] * B[N x K]^T with both
 * operands K-contiguous BF16 and FP32 accumulation on the matrix cores
 * (v_mfma_f32_16x16x32_bf16).  The forward pass, the input gradient and the
 * weight gradient are all of this form because each activation and gradient is
 * stored both row-major and transposed by the epilogue that produces it.
 *
 * Tiles of 64 or 128 rows and columns per workgroup of four wave64s, K in steps
 * of 64 through double-buffered LDS (k_sg_gemm_nt).  The ensemble members run
 * side by side in one launch.  Sizes must be multiples of 64 (M, N and K); the
 * host checks this.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "surrogate_kernels.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define SG_TK 64 /* contraction step: 128 bytes of an operand's row */

/* bf16 <-> f32 with round-to-nearest-even, written out so that the host and the
 * device round identically (NaN is not produced by these kernels) */
__device__ __forceinline__ uint16_t sg_f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
/* One tile of C = A B^T: BM x BN per workgroup of four wave64s (2 x 2 waves of
 * BM/2 x BN/2, each a grid of 16 x 16 MFMA blocks), K in steps of 64 through
 * two LDS buffers: the next step's operands are loaded from global memory
 * into registers while the matrix cores work on the current ones, and stored
 * into the other buffer afterwards, so one barrier per step suffices.  An LDS
 * row is 128 bytes, its 16-byte pieces exchanged by the low bits of the row, so
 * that eight rows of an operand read lie in different banks.
 *
 * The workgroups of a group read one operand panel together: the column tiles
 * of a row panel of A, or (weight gradient) all tiles of one part of the
 * contraction.  Consecutive workgroups go to the eight XCDs in turn, so a
 * group's members are taken eight apart and share an L2.
 *
 * What bounds it is the memory side, not the matrix cores: 128 x 128 tiles
 * halve the operand traffic of 64 x 64, the bf16 results and their transposes
 * leave through LDS in rows of 16-byte pieces instead of 2 and 8 bytes a lane.
 * The gradient of the activation is formed beside the activation (one erf) and
 * stored in place of the pre-activation, and the gradient's column sums (the
 * bias gradient) are formed here per wave's rows, so that the f32 gradient is
 * not stored at all. */
template <int EPI, int BM, int BN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BM == 128 ? (BN == 128 ? 2 : 3) : 4, BM == 128 ? (BN == 128 ? 2 : 3) : 4)))
k_sg_gemm_nt(int M, int N, int nx, int ny, int K, const uint16_t *A, long lda, long s_a, const uint16_t *B, long ldb,
             long s_b, SgEpiArgs e) {
  constexpr int WM = BM / 2, WN = BN / 2, FI = WM / 16, FJ = WN / 16;
  constexpr int LA = BM * SG_TK / 8 / 256, LB = BN * SG_TK / 8 / 256; /* 16-byte loads per thread */
  constexpr int SH = BN + 8, ST = BM + 8;                             /* epilogue rows: 16 bytes of padding */
  constexpr int BUF = (BM + BN) * SG_TK;
  constexpr bool STAGE = EPI == SG_EPI_HIDDEN || EPI == SG_EPI_DX;
  constexpr int LDS = STAGE && BM * SH + BN * ST > 2 * BUF ? BM * SH + BN * ST : 2 * BUF;
  __shared__ __attribute__((aligned(16))) uint16_t lds[LDS];
  /* this workgroup's tile: member `in` of group `grp` */
  const int gs = EPI == SG_EPI_DW ? nx * ny : nx, total = (int)gridDim.x, L = (int)blockIdx.x;
  const bool xcd = total % (8 * gs) == 0;
  const int in = xcd ? (L >> 3) % gs : L % gs, grp = xcd ? (L & 7) + 8 * ((L >> 3) / gs) : L / gs;
  const int m0 = (EPI == SG_EPI_DW ? in / nx : grp % ny) * BM, n0 = (EPI == SG_EPI_DW ? in % nx : in) * BN;
  const int net = EPI == SG_EPI_DW ? grp / e.splits : grp / ny;
  const int split = EPI == SG_EPI_DW ? grp % e.splits : 0;
  A += (size_t)net * s_a + (size_t)split * K;
  B += (size_t)net * s_b + (size_t)split * K;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = (wave >> 1) * WM, wc = (wave & 1) * WN;
  f32x4 acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; i++)
#pragma unroll
    for (int j = 0; j < FJ; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  /* global -> LDS: load q of a thread moves the 16-byte piece t % 8 of row
   * t / 8, t = tid + 256 q, i.e. row tid / 8 + 32 q.  The pieces in flight are
   * named one by one: an array of them ends up in LDS or copied register by
   * register, with a wait after each load */
  const int lrow = tid >> 3, lpc = (tid & 7) * 8, lds_at = lrow * SG_TK + (((tid & 7) ^ (lrow & 7)) * 8);
  const uint16_t *ga = A + (size_t)(m0 + lrow) * lda + lpc, *gb = B + (size_t)(n0 + lrow) * ldb + lpc;
  const size_t a32 = 32 * (size_t)lda, b32 = 32 * (size_t)ldb;
  uint4 a0, a1, a2, a3, b0, b1, b2, b3;
#define SG_LOAD(k0)                                      \
  do {                                                   \
    a0 = *(const uint4 *)(ga + (k0));                    \
    a1 = *(const uint4 *)(ga + (k0) + a32);              \
    if constexpr (LA > 2) {                              \
      a2 = *(const uint4 *)(ga + (k0) + 2 * a32);        \
      a3 = *(const uint4 *)(ga + (k0) + 3 * a32);        \
    }                                                    \
    b0 = *(const uint4 *)(gb + (k0));                    \
    b1 = *(const uint4 *)(gb + (k0) + b32);              \
    if constexpr (LB > 2) {                              \
      b2 = *(const uint4 *)(gb + (k0) + 2 * b32);        \
      b3 = *(const uint4 *)(gb + (k0) + 3 * b32);        \
    }                                                    \
  } while (0)
#define SG_STORE(buf)                                              \
  do {                                                             \
    uint16_t *as_ = lds + (buf) * BUF + lds_at, *bs_ = as_ + BM * SG_TK; \
    *(uint4 *)(as_) = a0;                                          \
    *(uint4 *)(as_ + 32 * SG_TK) = a1;                             \
    if constexpr (LA > 2) {                                        \
      *(uint4 *)(as_ + 64 * SG_TK) = a2;                           \
      *(uint4 *)(as_ + 96 * SG_TK) = a3;                           \
    }                                                              \
    *(uint4 *)(bs_) = b0;                                          \
    *(uint4 *)(bs_ + 32 * SG_TK) = b1;                             \
    if constexpr (LB > 2) {                                        \
      *(uint4 *)(bs_ + 64 * SG_TK) = b2;                           \
      *(uint4 *)(bs_ + 96 * SG_TK) = b3;                           \
    }                                                              \
  } while (0)
  const int nk = K / SG_TK;
  SG_LOAD(0);
  SG_STORE(0);
  __syncthreads();
  /* operands: lane l holds row (l % 16) and the 8 consecutive k of group l / 16;
   * A and B use the same k assignment, so the contraction is complete */
  const int fr = lane & 15, fg = lane >> 4;
  for (int kt = 0; kt < nk; kt++) {
    const uint16_t *as = lds + (kt & 1) * BUF, *bs = as + BM * SG_TK;
    if (kt + 1 < nk) SG_LOAD((kt + 1) * SG_TK);
#pragma unroll
    for (int kk = 0; kk < SG_TK / 8; kk += 4) {
      bf16x8 a[FI], b[FJ];
      const int piece = ((kk + fg) ^ (fr & 7)) * 8; /* tile rows start at multiples of 16 */
#pragma unroll
      for (int i = 0; i < FI; i++) a[i] = *(const bf16x8 *)(as + (wr + i * 16 + fr) * SG_TK + piece);
#pragma unroll
      for (int j = 0; j < FJ; j++) b[j] = *(const bf16x8 *)(bs + (wc + j * 16 + fr) * SG_TK + piece);
#pragma unroll
      for (int i = 0; i < FI; i++)
#pragma unroll
        for (int j = 0; j < FJ; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) SG_STORE((kt & 1) ^ 1);
    __syncthreads();
  }
#undef SG_LOAD
#undef SG_STORE
  /* result layout of a 16 x 16 block: lane l holds column l % 16, rows 4 (l / 16) + v */
  float *cf = e.cf ? e.cf + (size_t)net * e.s_cf + (size_t)split * e.s_split : nullptr;
  const float *dprev = EPI == SG_EPI_DX ? e.dprev + (size_t)net * e.s_dprev : nullptr;
  uint16_t *hs = lds, *ts = lds + BM * SH;
#pragma unroll
  for (int j = 0; j < FJ; j++) {
    const int lc = wc + j * 16 + fr, col = n0 + lc;
    const float bias = EPI == SG_EPI_HIDDEN || EPI == SG_EPI_OUT ? e.bias[(size_t)net * e.s_bias + col] : 0.0f;
    float cs = 0.0f;
#pragma unroll
    for (int i = 0; i < FI; i++) {
      const int lr = wr + i * 16 + fg * 4;
      uint16_t hv[4];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const size_t o = (size_t)(m0 + lr + v) * N + col;
        const float x = acc[i][j][v];
        if (EPI == SG_EPI_HIDDEN) {
          const float z = x + bias, er = 1.0f + erff(z * 0.70710678118654752f);
          hv[v] = sg_f2bf(0.5f * z * er);
          if (cf) cf[o] = 0.5f * er + z * 0.39894228040143268f * expf(-0.5f * z * z);
        } else if (EPI == SG_EPI_OUT) {
          cf[o] = x + bias;
        } else if (EPI == SG_EPI_DX) {
          const float g = x * dprev[o];
          cs += g;
          hv[v] = sg_f2bf(g);
        } else {
          cf[o] = x;
        }
      }
      if (STAGE) {
#pragma unroll
        for (int v = 0; v < 4; v++) hs[(lr + v) * SH + lc] = hv[v];
        *(uint2 *)(ts + lc * ST + lr) =
            make_uint2((uint32_t)hv[0] | ((uint32_t)hv[1] << 16), (uint32_t)hv[2] | ((uint32_t)hv[3] << 16));
      }
    }
    if (EPI == SG_EPI_DX) {
      /* the wave's rows of this column: lanes l, l + 16, l + 32, l + 48 */
      cs += __shfl_xor(cs, 16);
      cs += __shfl_xor(cs, 32);
      if (fg == 0) e.cs[((size_t)net * (M / WM) + (m0 + wr) / WM) * N + col] = cs;
    }
  }
  if (STAGE) {
    __syncthreads();
    uint16_t *cb = e.cb + (size_t)net * e.s_cb;
#pragma unroll
    for (int t = tid; t < BM * BN / 8; t += 256) {
      const int r = t / (BN / 8), c = (t % (BN / 8)) * 8;
      *(uint4 *)(cb + (size_t)(m0 + r) * N + n0 + c) = *(const uint4 *)(hs + r * SH + c);
    }
    if (e.ct) {
      uint16_t *ct = e.ct + (size_t)net * e.s_ct;
#pragma unroll
      for (int t = tid; t < BM * BN / 8; t += 256) {
        const int c = t / (BM / 8), r = (t % (BM / 8)) * 8;
        *(uint4 *)(ct + (size_t)(n0 + c) * M + m0 + r) = *(const uint4 *)(ts + c * ST + r);
      }
    }
  }
}

/* f32 [rows x cols] -> bf16 row-major [rows x ld] (zero padded) and its
 * transpose [ld x rows]; one thread per padded element */
__global__ void k_sg_pack(int rows, int cols, int ld, const float *X, uint16_t *Xb, uint16_t *XbT) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)rows * ld) return;
  const int r = (int)(idx / ld), c = (int)(idx % ld);
  const uint16_t h = c < cols ? sg_f2bf(X[(size_t)r * cols + c]) : (uint16_t)0;
  Xb[idx] = h;
  if (XbT) XbT[(size_t)c * rows + r] = h;
}

/* masked mean-square loss of the output layer and its gradient:
 * dY = 2 (Y - T) mask / count, stored bf16 and transposed bf16, with its
 * column sums per 64 rows (cs); loss partials per (net, workgroup) */
__global__ void __launch_bounds__(256) k_sg_loss(int rows, int N, int nets, const float *Y, const float *T,
                                                  const float *Mk, float inv_count, const unsigned int *count,
                                                  uint16_t *Gb, uint16_t *GT, float *cs, float *partial) {
  const int net = blockIdx.y;
  /* with a device count (mask entries of the batch), the same rounding as the host's (float)(1.0 / count) */
  if (count) inv_count = *count ? (float)(1.0 / (double)*count) : 0.0f;
  const size_t base = (size_t)net * rows * N;
  __shared__ uint16_t tile[64][66];
  __shared__ float csum[4][64];
  float s = 0.0f;
  /* 64 x 64 tiles (rows and N are multiples of 64), this block's in turn:
   * row-major results straight out, the transpose through LDS */
  const int tc = N / 64, ntiles = (rows / 64) * tc;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const int r0 = (t / tc) * 64, c0 = (t % tc) * 64;
    float gs = 0.0f; /* this thread's column, every fourth row */
#pragma unroll 8
    for (int q = 0; q < 16; q++) {
      const int k = (int)threadIdx.x + 256 * q, rr = k >> 6, cc = k & 63;
      const size_t idx = (size_t)(r0 + rr) * N + c0 + cc;
      const float d = (Y[base + idx] - T[idx]) * Mk[idx];
      s += d * d;
      const float g = 2.0f * d * inv_count;
      gs += g;
      const uint16_t gb = sg_f2bf(g);
      Gb[base + idx] = gb;
      tile[rr][cc] = gb;
    }
    csum[threadIdx.x >> 6][threadIdx.x & 63] = gs;
    __syncthreads();
    if (threadIdx.x < 64)
      cs[((size_t)net * (rows / 64) + r0 / 64) * N + c0 + threadIdx.x] =
          (csum[0][threadIdx.x] + csum[1][threadIdx.x]) + (csum[2][threadIdx.x] + csum[3][threadIdx.x]);
    for (int k = threadIdx.x; k < 64 * 64; k += 256) {
      const int cc = k >> 6, rr = k & 63;
      GT[base + (size_t)(c0 + cc) * rows + r0 + rr] = tile[rr][cc];
    }
    __syncthreads();
  }
  /* fixed-order block sum */
  __shared__ float red[256];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[(size_t)net * gridDim.x + blockIdx.x] = red[0];
}

/* one mini-batch, rows idx[0..batch) of the resident data, in one launch.  The
 * first xr x xc workgroups take 64 x 64 tiles of the inputs: packed to bf16,
 * row-major (zero padded to ld) and transposed through LDS so that both stores
 * are coalesced.  The others take the targets and the mask in f32 and count
 * the mask's entries. */
#define SG_GATHER_BLOCKS 512
__global__ void __launch_bounds__(256) k_sg_gather(int batch, int in_f, int ld, int out_f, int xr, int xc, const int *idx,
                                                    const float *Xall, const float *Tall, const float *Mall, uint16_t *Xb,
                                                    uint16_t *XbT, float *T, float *Mk, unsigned int *count) {
  if ((int)blockIdx.x < xr * xc) {
    __shared__ uint16_t tile[64][66];
    const int r0 = (int)blockIdx.x / xc * 64, c0 = (int)blockIdx.x % xc * 64;
#pragma unroll
    for (int q = 0; q < 16; q++) { /* all loads of the tile in flight */
      const int k = (int)threadIdx.x + 256 * q, rr = k >> 6, cc = k & 63, r = r0 + rr, c = c0 + cc;
      uint16_t h = 0;
      if (r < batch && c < in_f) h = sg_f2bf(Xall[(size_t)idx[r] * in_f + c]);
      if (r < batch && c < ld) Xb[(size_t)r * ld + c] = h;
      tile[rr][cc] = h;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int k = (int)threadIdx.x + 256 * q, cc = k >> 6, rr = k & 63, r = r0 + rr, c = c0 + cc;
      if (r < batch && c < ld) XbT[(size_t)c * batch + r] = tile[rr][cc];
    }
    return;
  }
  const unsigned b0 = blockIdx.x - (unsigned)(xr * xc);
  const unsigned w4 = (unsigned)out_f / 4, n4 = (unsigned)batch * w4; /* out_f is a multiple of 64 */
  unsigned int on = 0;
#pragma unroll 2
  for (unsigned i = b0 * 256 + threadIdx.x; i < n4; i += SG_GATHER_BLOCKS * 256) {
    const unsigned r = i / w4, c = i - r * w4;
    const size_t src = (size_t)idx[r] * w4 + c;
    const float4 m = ((const float4 *)Mall)[src];
    ((float4 *)T)[i] = ((const float4 *)Tall)[src];
    ((float4 *)Mk)[i] = m;
    on += (m.x != 0.0f) + (m.y != 0.0f) + (m.z != 0.0f) + (m.w != 0.0f);
  }
  /* one atomic per workgroup: thousands on one address would serialise */
  __shared__ unsigned int red[4];
  unsigned int w = on;
  for (int off = 32; off > 0; off >>= 1) w += __shfl_xor(w, off);
  if (__lane_id() == 0) red[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(count, red[0] + red[1] + red[2] + red[3]);
}

/* the sum of n parts (1 .. SG_MAX_SPLITS) a stride apart, in order, every
 * load issued before the first is used */
__device__ __forceinline__ float4 sg_add4(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
__device__ __forceinline__ float4 sg_sum_parts4(const float *p, int n, size_t stride) {
  static_assert(SG_MAX_SPLITS == 8, "eight parts are named");
  const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 g0 = *(const float4 *)p, g1 = z, g2 = z, g3 = z, g4 = z, g5 = z, g6 = z, g7 = z;
  if (n > 1) g1 = *(const float4 *)(p + stride);
  if (n > 2) g2 = *(const float4 *)(p + 2 * stride);
  if (n > 3) g3 = *(const float4 *)(p + 3 * stride);
  if (n > 4) g4 = *(const float4 *)(p + 4 * stride);
  if (n > 5) g5 = *(const float4 *)(p + 5 * stride);
  if (n > 6) g6 = *(const float4 *)(p + 6 * stride);
  if (n > 7) g7 = *(const float4 *)(p + 7 * stride);
  return sg_add4(sg_add4(sg_add4(sg_add4(sg_add4(sg_add4(sg_add4(g0, g1), g2), g3), g4), g5), g6), g7);
}

/* bias gradients 16 blk .. 16 blk + 15 (of nets x N) from their row parts
 * cs[net][chunks][N], returned by threads 0 to 15: sixteen threads a column take
 * every sixteenth part, summed in order (one thread a column waits for its
 * 64 parts one by one: 50 us) */
__device__ __forceinline__ float sg_bias_sum(const float *cs, int N, int chunks, int blk) {
  __shared__ float red[16][17];
  const int c = (int)threadIdx.x & 15, t = (int)threadIdx.x >> 4, i = blk * 16 + c;
  const float *p = cs + (size_t)(i / N) * chunks * N + i % N;
  float s = 0.0f;
#pragma unroll 4
  for (int k = t; k < chunks; k += 16) s += p[(size_t)k * N];
  red[t][c] = s;
  __syncthreads();
  float r = 0.0f;
  if (threadIdx.x < 16)
    for (int k = 0; k < 16; k++) r += red[k][threadIdx.x];
  return r;
}

__device__ __forceinline__ float sg_adam_one(const SgAdamArgs &a, float g, float *p, float *m, float *v) {
  const float mi = a.b1 * *m + (1.0f - a.b1) * g;
  const float vi = a.b2 * *v + (1.0f - a.b2) * g * g;
  *m = mi;
  *v = vi;
  return *p = *p - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
}

/* Adam (Kingma & Ba 2015) on the f32 master parameters of several layers in
 * one launch, and the weights' bf16 copy (row-major [N x K]) and transpose
 * [K x N].  The gradients come in parts (of the contraction for a weight, of
 * the rows for a bias) that are summed here in order.  The first workgroups
 * take the biases, 16 each; every other one a 64 x 64 tile of a weight, whose
 * transpose leaves through LDS.  Bound by memory: 28 bytes a parameter and
 * four per further part.  The five layers of the 4 x 512-wide ensemble: 38.6 us
 * (ten launches of 7.6 us, and 5 x 25 us for the bias sums, a layer at a time). */
__global__ void __launch_bounds__(256) k_sg_adam(SgAdamArgs a) {
  __shared__ uint16_t tile[64][66];
  int blk = (int)blockIdx.x, l = 0;
  if (blk < a.bias_blocks) {
    while (blk >= a.layer[l].nb_blocks) blk -= a.layer[l++].nb_blocks;
    const SgAdamLayer &y = a.layer[l];
    const float g = sg_bias_sum(y.cs, y.N, y.chunks, blk);
    const int i = blk * 16 + (int)threadIdx.x;
    if (threadIdx.x < 16) sg_adam_one(a, g, y.b + i, y.mb + i, y.vb + i);
    return;
  }
  blk -= a.bias_blocks;
  while (blk >= a.layer[l].nw_blocks) blk -= a.layer[l++].nw_blocks;
  const SgAdamLayer &y = a.layer[l];
  const int tk = y.K / 64, per = tk * (y.N / 64);
  const int net = blk / per, r0 = (blk % per) / tk * 64, c0 = (blk % tk) * 64;
  const size_t base = (size_t)net * y.N * y.K;
#pragma unroll 2
  for (int q = 0; q < 4; q++) {
    const int k = (int)threadIdx.x + 256 * q, rr = k >> 4, cc = (k & 15) * 4;
    const size_t i = base + (size_t)(r0 + rr) * y.K + c0 + cc;
    const float4 g = sg_sum_parts4(y.gW + i, y.splits, y.s_split);
    float4 p = *(const float4 *)(y.W + i), m = *(const float4 *)(y.mW + i), v = *(const float4 *)(y.vW + i);
    const uint16_t h0 = sg_f2bf(sg_adam_one(a, g.x, &p.x, &m.x, &v.x)), h1 = sg_f2bf(sg_adam_one(a, g.y, &p.y, &m.y, &v.y)),
                   h2 = sg_f2bf(sg_adam_one(a, g.z, &p.z, &m.z, &v.z)), h3 = sg_f2bf(sg_adam_one(a, g.w, &p.w, &m.w, &v.w));
    *(float4 *)(y.W + i) = p;
    *(float4 *)(y.mW + i) = m;
    *(float4 *)(y.vW + i) = v;
    *(uint2 *)(y.Wb + i) = make_uint2((uint32_t)h0 | ((uint32_t)h1 << 16), (uint32_t)h2 | ((uint32_t)h3 << 16));
    tile[rr][cc] = h0;
    tile[rr][cc + 1] = h1;
    tile[rr][cc + 2] = h2;
    tile[rr][cc + 3] = h3;
  }
  __syncthreads();
  for (int k = threadIdx.x; k < 64 * 64; k += 256)
    y.WT[base + (size_t)(c0 + (k >> 6)) * y.N + r0 + (k & 63)] = tile[k & 63][k >> 6];
}

/* the parts of 4 n values summed into the first, in order */
__global__ void k_sg_sum(size_t n, int parts, size_t stride, float *p) {
  const size_t i = 4 * ((size_t)blockIdx.x * blockDim.x + threadIdx.x);
  if (i < 4 * n) *(float4 *)(p + i) = sg_sum_parts4(p + i, parts, stride);
}

/* bias gradients db[net][N] (sg_bias_sum) */
__global__ void __launch_bounds__(256) k_sg_bias_grad(int N, int chunks, const float *cs, float *db) {
  const float g = sg_bias_sum(cs, N, chunks, (int)blockIdx.x);
  if (threadIdx.x < 16) db[blockIdx.x * 16 + threadIdx.x] = g;
}

/* bf16 copy (row-major [N x K] per net) and its transpose from f32 parameters */
__global__ void k_sg_refresh(size_t n, int N, int K, const float *p, uint16_t *pb, uint16_t *pt) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t per = (size_t)N * K;
  const size_t net = i / per, rem = i % per;
  const int r = (int)(rem / K), c = (int)(rem % K);
  const uint16_t h = sg_f2bf(p[i]);
  pb[i] = h;
  pt[net * per + (size_t)c * N + r] = h;
}

/* ------------------------------------------------------------------------ */

extern "C" {

hipError_t sg_launch_refresh(size_t n, int N, int K, const float *p, uint16_t *pb, uint16_t *pt, hipStream_t st) {
  hipLaunchKernelGGL(k_sg_refresh, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, N, K, p, pb, pt);
  return hipGetLastError();
}

/* 128 x 128 tiles where the sizes allow and the launch still brings two
 * workgroups (one round) to each of the 256 compute units, 64 x 64 elsewhere.
 * Hidden layer of 4 nets, 4096 x 512 x 512, forward and input gradient: 29.7
 * and 26.9 us against 30.2 and 30.7 (128 x 64 33.8 and 33.1; at the first
 * 64 x 64 kernel 35.5 and 59.9); its output layer of 256 columns, 256
 * workgroups of 128 x 128, 17.0 against 15.7. */
static int tile_of(int nets, int M, int N) {
  return M % 128 == 0 && N % 128 == 0 && (long)(M / 128) * (N / 128) * nets >= 512 ? 128 : 64;
}

/* parts of the weight gradient's contraction: its few tiles (128 x 64) leave
 * most of the chip idle over a batch of thousands; as many parts, up to
 * SG_MAX_SPLITS, as bring 512 workgroups and divide the batch's steps.  512 x
 * 512 x 4096 of 4 nets: 56.1 us in one part of 64 x 64 tiles, 19.0 in four
 * (31.9 in two, 17.0 in eight of 128 x 128, whose sum costs the update more) */
int sg_dw_splits(int nets, int M, int N, int rows) {
  const long tiles = (long)(M % 128 ? M / 64 : M / 128) * (N / 64) * nets;
  int s = 1;
  while (2 * s <= SG_MAX_SPLITS && 2 * s * tiles <= 512 && (rows / SG_TK) % (2 * s) == 0) s *= 2;
  return s;
}

int sg_dx_chunk(int nets, int M, int N) { return tile_of(nets, M, N) / 2; }

hipError_t sg_launch_gemm(int epi, int nets, int M, int N, int K, const uint16_t *A, long lda, long s_a,
                          const uint16_t *B, long ldb, long s_b, const SgEpiArgs *a, hipStream_t st) {
  const bool dw = epi == SG_EPI_DW;
  const int bm = dw ? (M % 128 ? 64 : 128) : tile_of(nets, M, N), bn = dw ? 64 : bm;
  const int nx = N / bn, ny = M / bm, nz = nets * (dw ? a->splits : 1);
  if (dw) K /= a->splits;
#define SG_GEMM(E, BM, BN)                                                                                            \
  hipLaunchKernelGGL((k_sg_gemm_nt<E, BM, BN>), dim3((unsigned)(nx * ny * nz)), dim3(256), 0, st, M, N, nx, ny, K, A, \
                     lda, s_a, B, ldb, s_b, *a)
#define SG_TILE(E)                           \
  do {                                       \
    if (bm == 128) SG_GEMM(E, 128, 128);     \
    else SG_GEMM(E, 64, 64);                 \
  } while (0)
  switch (epi) {
    case SG_EPI_HIDDEN: SG_TILE(SG_EPI_HIDDEN); break;
    case SG_EPI_OUT: SG_TILE(SG_EPI_OUT); break;
    case SG_EPI_DX: SG_TILE(SG_EPI_DX); break;
    default:
      if (bm == 128) SG_GEMM(SG_EPI_DW, 128, 64);
      else SG_GEMM(SG_EPI_DW, 64, 64);
      break;
  }
#undef SG_TILE
#undef SG_GEMM
  return hipGetLastError();
}

hipError_t sg_launch_pack(int rows, int cols, int ld, const float *X, uint16_t *Xb, uint16_t *XbT, hipStream_t st) {
  size_t n = (size_t)rows * ld;
  hipLaunchKernelGGL(k_sg_pack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, rows, cols, ld, X, Xb, XbT);
  return hipGetLastError();
}

hipError_t sg_launch_loss(int rows, int N, int nets, const float *Y, const float *T, const float *Mk, float inv_count,
                          const unsigned int *count, uint16_t *Gb, uint16_t *GT, float *cs, float *partial, int blocks,
                          hipStream_t st) {
  hipLaunchKernelGGL(k_sg_loss, dim3(blocks, nets), dim3(256), 0, st, rows, N, nets, Y, T, Mk, inv_count, count, Gb, GT,
                     cs, partial);
  return hipGetLastError();
}

hipError_t sg_launch_gather(int batch, int in_f, int ld, int out_f, const int *idx, const float *Xall, const float *Tall,
                            const float *Mall, uint16_t *Xb, uint16_t *XbT, float *T, float *Mk, unsigned int *count,
                            hipStream_t st) {
  const int xr = (batch + 63) / 64, xc = (ld + 63) / 64;
  hipLaunchKernelGGL(k_sg_gather, dim3((unsigned)(xr * xc + SG_GATHER_BLOCKS)), dim3(256), 0, st, batch, in_f, ld, out_f,
                     xr, xc, idx, Xall, Tall, Mall, Xb, XbT, T, Mk, count);
  return hipGetLastError();
}

hipError_t sg_launch_adam(SgAdamArgs *a, int n_layers, hipStream_t st) {
  int nw = 0;
  a->bias_blocks = 0;
  for (int l = 0; l < n_layers; l++) {
    SgAdamLayer &y = a->layer[l];
    y.nb_blocks = a->nets * y.N / 16; /* widths are multiples of 64 */
    y.nw_blocks = a->nets * (y.N / 64) * (y.K / 64);
    a->bias_blocks += y.nb_blocks;
    nw += y.nw_blocks;
  }
  hipLaunchKernelGGL(k_sg_adam, dim3((unsigned)(a->bias_blocks + nw)), dim3(256), 0, st, *a);
  return hipGetLastError();
}

hipError_t sg_launch_sum(size_t n, int parts, size_t stride, float *p, hipStream_t st) {
  n /= 4; /* weights come in tiles of 64 x 64 */
  hipLaunchKernelGGL(k_sg_sum, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, parts, stride, p);
  return hipGetLastError();
}

hipError_t sg_launch_bias_grad(int nets, int N, int chunks, const float *cs, float *db, hipStream_t st) {
  hipLaunchKernelGGL(k_sg_bias_grad, dim3((unsigned)(nets * N / 16)), dim3(256), 0, st, N, chunks, cs, db);
  return hipGetLastError();
}

} /* extern "C" */
