/*
 * surrogate_kernels.h -- launch interface between the surrogate's host code
 * (surrogate_host.cpp) and its gfx950 kernels (surrogate_kernels.hip).
 */
#ifndef XMIMSIM_AMD_SURROGATE_KERNELS_H
#define XMIMSIM_AMD_SURROGATE_KERNELS_H

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

/* epilogue kinds of sg_launch_gemm */
#define SG_EPI_HIDDEN 0 /* z = acc + b -> cf (f32), gelu(z) -> cb (bf16) and ct (bf16, transposed) */
#define SG_EPI_OUT 1    /* acc + b -> cf (f32) */
#define SG_EPI_DX 2     /* acc * gelu'(zprev) -> cf (f32), cb (bf16), ct (bf16, transposed) */
#define SG_EPI_DW 3     /* acc -> cf (f32) */

typedef struct SgEpiArgs {
  const float *bias;
  long s_bias;        /* per-net strides (elements) */
  float *cf;
  long s_cf;
  uint16_t *cb;
  long s_cb;
  uint16_t *ct;
  long s_ct;
  const float *dprev; /* SG_EPI_DX: activation gradient [M x N] */
  long s_dprev;
  float *cs;          /* SG_EPI_DX: column sums of the result per sg_dx_chunk rows, [net][chunk][N] */
  int splits;         /* SG_EPI_DW: parts of the contraction (sg_dw_splits), s_split floats apart in cf */
  long s_split;
} SgEpiArgs;

#define SG_MAX_SPLITS 8

/* one layer of the Adam update: gradients as `splits` parts of gW and
 * `chunks` row parts of the bias gradient in cs[net][chunks][N] */
typedef struct SgAdamLayer {
  int N, K, splits, chunks, nb_blocks, nw_blocks;
  size_t s_split;
  const float *gW, *cs;
  float *W, *mW, *vW, *b, *mb, *vb;
  uint16_t *Wb, *WT;
} SgAdamLayer;

#define SG_ADAM_LAYERS 8 /* of one launch */
typedef struct SgAdamArgs {
  int nets, bias_blocks;
  float lr, b1, b2, eps, c1, c2;
  SgAdamLayer layer[SG_ADAM_LAYERS];
} SgAdamArgs;

#ifdef __cplusplus
extern "C" {
#endif
/* C[M x N] = A[M x K] * B[N x K]^T per net (gridDim.z = nets); M, N and K
 * multiples of 64, lda/ldb multiples of 8 */
hipError_t sg_launch_gemm(int epi, int nets, int M, int N, int K, const uint16_t *A, long lda, long s_a,
                          const uint16_t *B, long ldb, long s_b, const SgEpiArgs *a, hipStream_t st);
hipError_t sg_launch_pack(int rows, int cols, int ld, const float *X, uint16_t *Xb, uint16_t *XbT, hipStream_t st);
/* inv_count scales the gradient; a non-NULL count (device) overrides it with 1 / *count */
hipError_t sg_launch_loss(int rows, int N, int nets, const float *Y, const float *T, const float *Mk, float inv_count,
                          const unsigned int *count, uint16_t *Gb, uint16_t *GT, float *cs, float *partial, int blocks,
                          hipStream_t st);
/* parts of the weight gradient [M x N] over `rows` (rows == 0: the most any batch takes) */
int sg_dw_splits(int nets, int M, int N, int rows);
/* rows per column sum of an SG_EPI_DX product [M x N] */
int sg_dx_chunk(int nets, int M, int N);
hipError_t sg_launch_sum(size_t n, int parts, size_t stride, float *p, hipStream_t st);
hipError_t sg_launch_bias_grad(int nets, int N, int chunks, const float *cs, float *db, hipStream_t st);
/* mini-batch rows idx[batch] of the resident data into the packed inputs, targets, mask; count += mask entries */
hipError_t sg_launch_gather(int batch, int in_f, int ld, int out_f, const int *idx, const float *Xall, const float *Tall,
                            const float *Mall, uint16_t *Xb, uint16_t *XbT, float *T, float *Mk, unsigned int *count,
                            hipStream_t st);
hipError_t sg_launch_refresh(size_t n, int N, int K, const float *p, uint16_t *pb, uint16_t *pt, hipStream_t st);
hipError_t sg_launch_adam(SgAdamArgs *a, int n_layers, hipStream_t st);
#ifdef __cplusplus
}
#endif

#endif
