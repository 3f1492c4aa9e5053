// The small-tile DMA GEMM kernels for bfloat16.
#include "gemm_tile_kernels.hpp"

namespace tk {
namespace gemm_dma {

template void launch_tile<__bf16>(int, Variant, const Plan&, const void*, const void*, const void*,
                               void*, const Problem&, hipStream_t);
template void launch_split<__bf16>(Variant, const Plan&, const void*, const void*, const void*,
                                void*, const Problem&, int, hipStream_t);

}  // namespace gemm_dma
}  // namespace tk
