// Tile order of the routed GEMMs, shared by the GEMM kernel and the reduce pass of its split tail.
#pragma once
#include "common.hpp"

namespace ffnk {

constexpr int kXcds = 8;             // MI355X: 8 XCDs, workgroups are dealt to them round-robin
constexpr int kCusPerChip = 256;
constexpr int kTailSlots = 256;      // (tile, K range) pairs of a split tail never exceed one per CU
constexpr int kTailMaxSplits = 16;

// Contractions that the direct kernels can load: whole 64-element slabs, or 16-byte pieces of at least one slab, whose first
// slab is loaded whole from the contraction's start (clear_head): under 64 elements that load would run past the rows.
__host__ __device__ inline bool direct_slabs_ok(int K) { return K > 0 && (K % 64 == 0 || (K % 8 == 0 && K >= 64)); }

constexpr int kEvenGroups = 3;    // see routed_tile_coord
constexpr int kEvenGroupMin = 6;  // 6 x 5 tiles on the 32 CUs of an XCD load the fewest panels

struct TileCoord {
  int grp;      // 0 = visual, 1 = text
  int row0;     // first routed position of the tile
  int row_end;  // end of the tile's group
  int n0;       // first output column
};

// Tiles are bm rows x bn output columns; M-tiles never straddle the two groups.
__host__ __device__ inline int routed_tile_count(int n_vis, int M, int N, int bm, int bn) {
  return (cdiv(n_vis, bm) + cdiv(M - n_vis, bm)) * cdiv(N, bn);
}

// Split-K factor of a launch: `splits` where the two groups have cdiv(M, bm) M-tiles between them, else (one more) splits_more.
__host__ __device__ inline int routed_splits(int n_vis, int M, int bm, int splits, int splits_more) {
  return cdiv(n_vis, bm) + cdiv(M - n_vis, bm) > cdiv(M, bm) ? splits_more : splits;
}

// Position L of the order -> tile.  The order walks super-groups of M-tiles column by column, so that tiles sharing A rows /
// B columns are neighbours.  Above kEvenGroups * group_m M-tiles: super-groups of group_m M-tiles from the first tile on.  Up to
// there, where the edges of the super-groups weigh more: super-groups of one modality's M-tiles only (two modalities share
// no weight panel), at most group_m each (or kEvenGroupMin), the modality's M-tiles dealt evenly to them.  MaskedFFN at
// d = 4096, h = 14336: forward at M = 1411 (three M-tiles of each modality) 507.5 -> 501.7 us, the backward's dx GEMM at
// M = 4096 (eight of each; before, all sixteen were one super-group and 41 % of its L2 requests missed, now 33 %) 775 -> 706 us;
// forward at M = 902, d = 7296 and at M = 4381, d = 1728: 1.0-1.5 % faster.  Dealt evenly at any size, M = 32768 lost 1.5 %.
__host__ __device__ inline TileCoord routed_tile_coord(int L, int n_vis, int M, int N, int bm, int bn, int group_m) {
  const int tiles_v = cdiv(n_vis, bm);
  const int tiles_m = tiles_v + cdiv(M - n_vis, bm);
  const int tiles_n = cdiv(N, bn);
  int first_m, gsz;
  if (tiles_m > kEvenGroups * group_m) {
    first_m = L / (group_m * tiles_n) * group_m;
    gsz = group_m < tiles_m - first_m ? group_m : tiles_m - first_m;
  } else {
    const bool visual = L < tiles_v * tiles_n;
    first_m = visual ? 0 : tiles_v;                         // first M-tile of the modality
    gsz = visual ? tiles_v : tiles_m - tiles_v;             // ... and how many it has
    const int cap = group_m > kEvenGroupMin ? group_m : kEvenGroupMin;
    if (gsz > cap) {  // (divisions of a few hundred cycles each, ahead of a tile's first load)
      const int own = gsz, base = first_m, groups = cdiv(own, cap);
      const int s = ((L / tiles_n - base + 1) * groups - 1) / own;  // the super-group [s * own / groups, (s + 1) * own / groups) with this row
      first_m = base + s * own / groups;
      gsz = base + (s + 1) * own / groups - first_m;
    }
  }
  L -= first_m * tiles_n;
  const int tile_m = first_m + L % gsz;
  const int tile_n = L / gsz;
  TileCoord t;
  t.grp = tile_m < tiles_v ? 0 : 1;
  t.row0 = t.grp == 0 ? tile_m * bm : n_vis + (tile_m - tiles_v) * bm;
  t.row_end = t.grp == 0 ? n_vis : M;
  t.n0 = tile_n * bn;
  return t;
}

// Weight-gradient GEMMs: [groups][splits][tiles_r x tiles_c].  Workgroup b runs on XCD b % 8, and every XCD takes an eighth of
// EACH group's order, the group with more rows first: the two groups' tiles cost what the groups have rows, and a group
// without any only stores zeros.  One order over both groups dealt an absent modality's zeros to four XCDs and all of the products
// to the other four: forward + backward of one modality, MaskedFFN M = 3806, d = 2112, h = 6400 1364 -> 1105 us, MaskedLinear
// M = 6638, K = 1920, N = 3712 414 -> 329 us; both modalities present within 1.5 % (d = 4096, h = 14336, M = 4096 3834 -> 3783).
// Inside a group a K range's tiles stay together (tiles of different ranges share nothing), and inside a range the order walks super-groups of kDwGroup row tiles column by
// column, so the 32 tiles that an XCD runs at a time are 8 x 4 of them and load 12 panels per slab.  With the row tiles of
// the whole output walked first, 32 of a long column ran at a time and loaded 33: the MaskedFFN's weight gradients at
// M = 4096, d = 4096, h = 14336 missed L2 with 47 % of their requests and moved 4.5 TB/s; with the super-groups 20 % miss,
// 500 -> 475 us per launch, and MaskedLinear's backward at K = N = 2048 ... 6000 gains 1.5-3 %.
constexpr int kDwGroup = 8;
struct DwTileCoord {
  int grp, split, tile_r, tile_c;  // grp < 0: a surplus workgroup
};
inline int dw_blocks(int64_t tiles_r, int64_t tiles_c, int splits) {
  return (int)(2 * kXcds * cdiv64(tiles_r * tiles_c * splits, kXcds));
}
__host__ __device__ inline DwTileCoord dw_tile_coord(int bid, int tiles_r, int tiles_c, int splits, int n_vis, int M) {
  DwTileCoord t{-1, 0, 0, 0};
  const int tiles = tiles_r * tiles_c;
  const int per_xcd = cdiv(tiles * splits, kXcds);
  int slot = bid / kXcds;
  const int second = slot >= per_xcd ? 1 : 0;
  slot -= second * per_xcd;
  int L = (bid % kXcds) * per_xcd + slot;
  if (slot >= per_xcd || L >= tiles * splits) return t;
  t.grp = (n_vis * 2 >= M ? 0 : 1) ^ second;
  t.split = L / tiles;
  L -= t.split * tiles;
  const int width = kDwGroup * tiles_c;
  const int first_r = (L / width) * kDwGroup;
  const int gsz = kDwGroup < tiles_r - first_r ? kDwGroup : tiles_r - first_r;
  t.tile_r = first_r + (L % width) % gsz;
  t.tile_c = (L % width) / gsz;
  return t;
}

// Tiles of the whole rounds of a launch whose remainder runs as smaller tiles (GemmArgs::tail_mode 1 and 2).  Up to half a
// round the remainder's 128-row tiles, two to a CU, are one round of their own at 0.6 of the big tile's time (SwiGLU GEMM,
// K = 4096: 62 us against 103); past half a round they are two, and the big tile's round is the shorter one.
__host__ __device__ inline int whole_round_tiles(int total) {
  const int rest = total % kCusPerChip;
  return rest > kCusPerChip / 2 ? total : total - rest;
}

// Split tail: the tiles past the last whole round of kCusPerChip are each cut into this many K
// ranges, so that the (tile, range) pairs fill about one round; ranges keep at least 8 slabs.
__host__ __device__ inline int tail_split_factor(int n_tail, int slabs) {
  if (n_tail <= 0) return 1;
  int s = kTailSlots / n_tail;
  if (s > kTailMaxSplits) s = kTailMaxSplits;
  if (s > slabs / 8) s = slabs / 8;
  if (s < 1) s = 1;
  return cdiv(slabs, cdiv(slabs, s));  // no empty range
}

}  // namespace ffnk
