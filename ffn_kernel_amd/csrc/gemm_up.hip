// MaskedFFN up-projection with the SwiGLU epilogue: gathered A rows, H written in routed order.
#include "gemm_tiles.hpp"

namespace ffnk {

hipError_t launch_up_gemm(int tile, bool direct, const GemmArgs& g, hipStream_t stream) {
  if (tile == TILE_MIXED_W4) {
    if (!direct) return hipErrorInvalidValue;
    return launch_routed_mixed<DualTiles<true>::T1, DualTiles<true>::Short, DualTiles<true>::Quarter>(g, stream);
  }
  return direct ? dispatch_tile_with_tail<DualTiles<true>>(tile, g, stream)
                : dispatch_tile<DualTiles<false>>(tile, g, stream);
}

TileGeom tile_geom(int tile, bool dual) {
  switch (tile) {
    case TILE_256x256_W8: return {256, dual ? 128 : 256, 2, 4};
    case TILE_256x256_W4: return {256, dual ? 128 : 256, 2, 2};
    case TILE_128x128_W4:
    case TILE_128x128_R4: return {128, dual ? 64 : 128, 2, 2};
    case TILE_128x256_R3: return {128, dual ? 128 : 256, 2, 2};
    case TILE_64x128_R3: return {64, dual ? 64 : 128, 2, 2};
    case TILE_192x256_W4: return dual ? TileGeom{128, 128, 2, 2} : TileGeom{192, 256, 2, 2};
    case TILE_160x256_W4: return dual ? TileGeom{128, 128, 2, 2} : TileGeom{160, 256, 2, 2};
    default: return dual ? TileGeom{64, 64, 2, 2} : TileGeom{128, 64, 2, 2};
  }
}

}  // namespace ffnk
