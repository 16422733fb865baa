// Weight-gradient GEMM of the MaskedFFN backward with one operand read where it lies: the rows of
// H, dt1 or dt3 (routed order) are the contraction rows, turned into MFMA operands by the transposing
// LDS read; the other operand is the 64-padded transpose of the gathered x or g.
#include "gemm_tiles.hpp"

namespace ffnk {

// The layer's three weight gradients in one launch: a launch of its own for each is a ramp up, a last partial round and a gap on
// the stream three times over, and as many launches for the host.  MaskedFFN forward + backward over 60 drawn layers: 4.0 % less
// time in the geometric mean on the tiles of three launches, 4.6 % on tiles and split factors picked for the three together (d =
// 1728, h = 4992, M = 2682 568 -> 481 us, d = 1664, h = 5184, M = 97 137 -> 126, d = 6528, h = 14336, M = 6755 9100 -> 9188).
struct DwBatch {
  SplitKArgs s[kDwBatch];
  int along_r;  // bit i: s[i] stores runs along r (KMajorDwTiles<false>)
  int blocks;   // workgroups per GEMM, a multiple of the XCD count
};

template <class AlongR, class AlongC>
__global__ __launch_bounds__(AlongC::NT) void dw_batch_kernel(const DwBatch b) {
  static_assert(AlongR::LDS_BYTES == AlongC::LDS_BYTES && AlongR::NT == AlongC::NT && kDwBatch == 3, "the same tile");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[AlongC::LDS_BYTES];
  const int which = (int)blockIdx.x / b.blocks, bid = (int)blockIdx.x - which * b.blocks;
  // Selected member by member: an index into the kernel's arguments would put them in scratch memory.
  auto pick = [&](auto first, auto second, auto third) { return which == 0 ? first : which == 1 ? second : third; };
  SplitKArgs s = b.s[0];
  s.A = pick(b.s[0].A, b.s[1].A, b.s[2].A);
  s.lda = pick(b.s[0].lda, b.s[1].lda, b.s[2].lda);
  s.B = pick(b.s[0].B, b.s[1].B, b.s[2].B);
  s.ldb = pick(b.s[0].ldb, b.s[1].ldb, b.s[2].ldb);
  s.out[0] = pick(b.s[0].out[0], b.s[1].out[0], b.s[2].out[0]);
  s.out[1] = pick(b.s[0].out[1], b.s[1].out[1], b.s[2].out[1]);
  s.out_sr = pick(b.s[0].out_sr, b.s[1].out_sr, b.s[2].out_sr);
  s.out_sc = pick(b.s[0].out_sc, b.s[1].out_sc, b.s[2].out_sc);
  if ((b.along_r >> which) & 1) grouped_splitk_body<AlongR>(s, lds, bid);
  else grouped_splitk_body<AlongC>(s, lds, bid);
}

template <class AlongR, class AlongC>
static hipError_t launch_batch(DwBatch& b, hipStream_t stream) {
  for (const SplitKArgs& s : b.s)
    if (s.R % 8 != 0 || s.lda * (kBK * 2) + 2 * (int64_t)s.R >= ((int64_t)1 << 32)) return hipErrorInvalidValue;
  b.blocks = dw_blocks(cdiv(b.s[0].R, AlongC::BN), cdiv(b.s[0].Cc, AlongC::BM), 1);
  hipLaunchKernelGGL((dw_batch_kernel<AlongR, AlongC>), dim3(kDwBatch * b.blocks), dim3(AlongC::NT), 0, stream, b);
  return hipGetLastError();
}

hipError_t launch_dw_batch_kmajor(int tile, const SplitKArgs (&g)[kDwBatch], hipStream_t stream) {
  using R = KMajorDwTiles<false>;
  using C = KMajorDwTiles<true>;
  DwBatch b;
  b.along_r = 0;
  for (int i = 0; i < kDwBatch; ++i) {
    if (g[i].R <= 0 || g[i].Cc <= 0 || g[i].R != g[0].R || g[i].Cc != g[0].Cc || g[i].splits != 1 || g[i].out[0] == nullptr)
      return hipErrorInvalidValue;
    b.s[i] = g[i];
    b.along_r |= (g[i].out_sr == 1 && g[i].out_sc != 1) << i;
  }
  switch (tile) {
    case TILE_256x256_W8: return launch_batch<R::T0, C::T0>(b, stream);
    case TILE_256x256_W4: return launch_batch<R::T1, C::T1>(b, stream);
    case TILE_SMALL_W4: return launch_batch<R::T3, C::T3>(b, stream);
    case TILE_64x128_R3:
    case TILE_128x256_R3:  // no such weight-gradient tile
    case TILE_128x128_R4:  // no ring here: the group's last slab is cleared in LDS
    case TILE_128x128_W4: return launch_batch<R::T2, C::T2>(b, stream);
    default: return hipErrorInvalidValue;
  }
}

// One weight gradient, its contraction cut into ranges (fp32 partials, contiguous along the columns).
hipError_t launch_splitk_gemm_kmajor(int tile, const SplitKArgs& g, hipStream_t stream) {
  using C = KMajorDwTiles<true>;
  if (g.out[0] != nullptr) return hipErrorInvalidValue;  // launch_dw_batch_kmajor
  switch (tile) {
    case TILE_256x256_W8: return launch_grouped_splitk<C::T0>(g, stream);
    case TILE_256x256_W4: return launch_grouped_splitk<C::T1>(g, stream);
    case TILE_SMALL_W4: return launch_grouped_splitk<C::T3>(g, stream);
    case TILE_64x128_R3:
    case TILE_128x256_R3:
    case TILE_128x128_R4:
    case TILE_128x128_W4: return launch_grouped_splitk<C::T2>(g, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ffnk
