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
__device__ __forceinline__ void dw_batch_body(const DwBatch& b, uint8_t* lds, const int block) {
  static_assert(AlongR::LDS_BYTES == AlongC::LDS_BYTES && AlongR::NT == AlongC::NT && kDwBatch == 3, "the same tile");
  const int which = block / b.blocks, bid = block - which * b.blocks;
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
__global__ __launch_bounds__(AlongC::NT) void dw_batch_kernel(const DwBatch b) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[AlongC::LDS_BYTES];
  dw_batch_body<AlongR, AlongC>(b, lds, (int)blockIdx.x);
}

// The layer's dx GEMM ahead of them in the same launch: its few, long workgroups start first, the weight gradients' many short ones
// fill the CUs around them.
template <class Dx, class AlongR, class AlongC>
__global__ __launch_bounds__(AlongC::NT) void dx_dw_batch_kernel(const GemmArgs gx, const DwBatch b, const int dx_blocks) {
  static_assert(Dx::NT == AlongC::NT, "one workgroup size");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[Dx::LDS_BYTES > AlongC::LDS_BYTES ? Dx::LDS_BYTES : AlongC::LDS_BYTES];
  if ((int)blockIdx.x < dx_blocks) routed_gemm_body<Dx>(gx, lds, (int)blockIdx.x);
  else dw_batch_body<AlongR, AlongC>(b, lds, (int)blockIdx.x - dx_blocks);
}

static bool fill_batch(const SplitKArgs (&g)[kDwBatch], int bm, int bn, DwBatch* b) {
  b->along_r = 0;
  for (int i = 0; i < kDwBatch; ++i) {
    const SplitKArgs& s = g[i];
    if (s.R <= 0 || s.Cc <= 0 || s.R != g[0].R || s.Cc != g[0].Cc || s.splits != 1 || s.out[0] == nullptr) return false;
    if (s.R % 8 != 0 || s.lda * (kBK * 2) + 2 * (int64_t)s.R >= ((int64_t)1 << 32)) return false;
    b->s[i] = s;
    b->along_r |= (s.out_sr == 1 && s.out_sc != 1) << i;
  }
  b->blocks = dw_blocks(cdiv(g[0].R, bn), cdiv(g[0].Cc, bm), 1);
  return true;
}

template <class AlongR, class AlongC>
static hipError_t launch_batch(const SplitKArgs (&g)[kDwBatch], hipStream_t stream) {
  DwBatch b;
  if (!fill_batch(g, AlongC::BM, AlongC::BN, &b)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((dw_batch_kernel<AlongR, AlongC>), dim3(kDwBatch * b.blocks), dim3(AlongC::NT), 0, stream, b);
  return hipGetLastError();
}

hipError_t launch_dx_dw_batch_kmajor(const GemmArgs& gx, const SplitKArgs (&g)[kDwBatch], hipStream_t stream) {
  using Dx = KMajorTiles<false, true>::T0;
  using R = KMajorDwTiles<false>::T0;
  using C = KMajorDwTiles<true>::T0;
  DwBatch b;
  if (gx.M <= 0 || gx.N <= 0 || gx.splits != 1 || gx.tail_mode != 0 || gx.P_tail != nullptr || !routed_gemm_args_ok<Dx>(gx) || !fill_batch(g, C::BM, C::BN, &b))
    return hipErrorInvalidValue;
  const int dx_blocks = routed_gemm_grid<Dx>(gx.M, gx.N);  // a multiple of the XCD count
  hipLaunchKernelGGL((dx_dw_batch_kernel<Dx, R, C>), dim3(dx_blocks + kDwBatch * b.blocks), dim3(C::NT), 0, stream, gx, b, dx_blocks);
  return hipGetLastError();
}

hipError_t launch_dw_batch_kmajor(int tile, const SplitKArgs (&g)[kDwBatch], hipStream_t stream) {
  using R = KMajorDwTiles<false>;
  using C = KMajorDwTiles<true>;
  switch (tile) {
    case TILE_256x256_W8: return launch_batch<R::T0, C::T0>(g, stream);
    case TILE_256x256_W4: return launch_batch<R::T1, C::T1>(g, stream);
    case TILE_SMALL_W4: return launch_batch<R::T3, C::T3>(g, stream);
    case TILE_64x128_R3:
    case TILE_128x256_R3:  // no such weight-gradient tile
    case TILE_128x128_R4:  // no ring here: the group's last slab is cleared in LDS
    case TILE_128x128_W4: return launch_batch<R::T2, C::T2>(g, stream);
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
