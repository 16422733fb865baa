// Weight-gradient GEMM of the MaskedFFN backward with one operand read where it lies: the rows of
// H, dt1 or dt3 (routed order) are the contraction rows, turned into MFMA operands by the transposing
// LDS read; the other operand is the 64-padded transpose of the gathered x or g.
#include "gemm_tiles.hpp"

namespace ffnk {

template <class Tiles>
static hipError_t launch_tile(int tile, const SplitKArgs& g, hipStream_t stream) {
  switch (tile) {
    case TILE_256x256_W8: return launch_grouped_splitk<typename Tiles::T0>(g, stream);
    case TILE_256x256_W4: return launch_grouped_splitk<typename Tiles::T1>(g, stream);
    case TILE_64x128_R3:
    case TILE_128x256_R3:  // no such weight-gradient tile
    case TILE_128x128_R4:  // no ring here: the group's last slab is cleared in LDS
    case TILE_128x128_W4: return launch_grouped_splitk<typename Tiles::T2>(g, stream);
    case TILE_SMALL_W4: return launch_grouped_splitk<typename Tiles::T3>(g, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_splitk_gemm_kmajor(int tile, const SplitKArgs& g, hipStream_t stream) {
  const bool along_r = g.out[0] != nullptr && g.out_sr == 1 && g.out_sc != 1;  // partials are contiguous along the columns
  return along_r ? launch_tile<KMajorDwTiles<false>>(tile, g, stream) : launch_tile<KMajorDwTiles<true>>(tile, g, stream);
}

}  // namespace ffnk
