// The small-tile DMA GEMM kernels for float16.
#include "gemm_tile_kernels.hpp"

namespace tk {
namespace gemm_dma {

template void launch_tile<_Float16>(int, Variant, const Plan&, const void*, const void*, const void*,
                               void*, const Problem&, hipStream_t);
template void launch_split<_Float16>(Variant, const Plan&, const void*, const void*, const void*,
                                 void*, const Problem&, int, hipStream_t);

}  // namespace gemm_dma
}  // namespace tk
