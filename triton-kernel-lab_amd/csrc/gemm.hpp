// Internal interface between the GEMM entry point (gemm.hip) and its buffer->LDS DMA
// fast path (gemm_dma.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace tk {

namespace gemm_dma {

// How the operands are stored, BLAS letters: N row-major, T transposed. NN: A [M][K], B [K][N];
// NT: A [M][K], B [N][K]; TN: A [K][M], B [K][N].
enum class Layout { NN, NT, TN };

struct Plan {
  Layout layout;
  bool swap;      // compute C^T = B^T A^T (both operands transposed)
  bool k_tail;    // K may end inside a 32-wide K tile
  int64_t lda, ldb;  // row strides of the stored matrices, in elements (after the swap)
};

// True when the DMA kernels handle this problem: f16/bf16 operands, each stored with one unit
// stride, a contiguous extent and a row stride that are multiples of 8 elements, a 16-byte
// aligned base and a byte extent below 2 GiB.
bool plan(const void* a, const void* b, int64_t m, int64_t n, int64_t k, int64_t stride_am,
          int64_t stride_ak, int64_t stride_bk, int64_t stride_bn, Plan* plan);

}  // namespace gemm_dma

// True when that is a row-major problem with K a multiple of 32 (the fused kernels' contract).
bool gemm_dma_applies(const void* a, const void* b, int64_t m, int64_t n, int64_t k,
                      int64_t stride_am, int64_t stride_ak, int64_t stride_bk, int64_t stride_bn);

// Enqueues the DMA kernel for a plan; arguments are checked by the caller. With `row_scale`
// (float32[m], row-major problems only) row m of C is round(row_scale[m] * acc).
void gemm_dma_launch(const gemm_dma::Plan& plan, int dtype, const void* a, const void* b, void* c,
                     int64_t m, int64_t n, int64_t k, int64_t stride_cm, int64_t stride_cn,
                     hipStream_t stream, const float* row_scale = nullptr);

// Enqueues the split-K kernels (gemm_tile_kernels.hpp), plain, row-scaled (row_scale) or SwiGLU
// (b_up), with `partial` holding splits * m * n float32 sums (twice that for SwiGLU); strides:
// am, ak, bk, bn, up k, up n, cm, cn. False when the DMA kernels do not handle the problem.
bool gemm_split_launch(int dtype, const void* a, const void* b, const void* b_up,
                       const float* row_scale, void* c, float* partial, int64_t m, int64_t n,
                       int64_t k, int64_t splits, const int64_t* strides, hipStream_t stream);

// Enqueues the SwiGLU-fused DMA kernel: y = swiglu(value = a * b_up, gate = a * b_gate),
// both weights [K, N] row-major; each must satisfy gemm_dma_applies with `a`.
void gemm_swiglu_dma_launch(int dtype, const void* a, const void* b_gate, const void* b_up,
                            void* y, int64_t m, int64_t n, int64_t k, int64_t stride_am,
                            int64_t stride_gk, int64_t stride_uk, int64_t stride_ym,
                            int64_t stride_yn, hipStream_t stream);

}  // namespace tk
