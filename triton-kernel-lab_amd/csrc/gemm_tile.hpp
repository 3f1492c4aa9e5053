// Interface of the small-tile DMA GEMM kernels (gemm_tile_kernels.hpp; one translation unit per
// dtype instantiates them).
#pragma once
#include "gemm_device.hpp"

namespace tk {
namespace gemm_dma {

enum class Variant { kPlain, kRowScale, kSwiGLU };

// Block tiles (rows x columns of the A and B tiles; with SwiGLU half of the columns are gate
// and half up columns).
struct Tile {
  int m, n;
};
constexpr Tile kTiles[] = {{256, 256}, {256, 128}, {128, 256}, {192, 192}, {128, 192},
                           {192, 128}, {128, 128}, {128, 64},  {64, 128},  {64, 64}};
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);

// Index of the tile for a problem (0 of kTiles is the 256 x 256 kernel of gemm_dma.hip). Every
// tile sums K in the same order, so the choice of a tile never changes a result; splitting K
// (launch_split) does.
int pick_tile(const Tile* tiles, int count, int64_t m, int64_t n, int64_t k, Variant variant);

// Enqueues the small-tile kernel `tile` (1 ..) for a problem whose tile counts are filled in.
template <typename T>
void launch_tile(int tile, Variant variant, const Plan& plan, const void* a, const void* b,
                 const void* b2, void* c, const Problem& p, hipStream_t stream);

// Enqueues the split-K kernels: 64 x 64 tiles (64 x 128 for SwiGLU: 64 output columns) of a problem
// whose tile counts, partial and split_tiles are filled in, `splits` runs of K tiles.
template <typename T>
void launch_split(Variant variant, const Plan& plan, const void* a, const void* b, const void* b2,
                  void* c, const Problem& p, int splits, hipStream_t stream);

}  // namespace gemm_dma
}  // namespace tk
