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
struct OrderPos {
  int tile_m, tile_n;
};
__host__ __device__ inline OrderPos order_pos(int L, int tiles_v, int tiles_m, int tiles_n, int group_m) {
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
  return {first_m + L % gsz, L / gsz};
}
__host__ __device__ inline TileCoord routed_tile_coord(int L, int n_vis, int M, int N, int bm, int bn, int group_m) {
  const int tiles_v = cdiv(n_vis, bm);
  const OrderPos at = order_pos(L, tiles_v, tiles_v + cdiv(M - n_vis, bm), cdiv(N, bn), group_m);
  TileCoord t;
  t.grp = at.tile_m < tiles_v ? 0 : 1;
  t.row0 = t.grp == 0 ? at.tile_m * bm : n_vis + (at.tile_m - tiles_v) * bm;
  t.row_end = t.grp == 0 ? n_vis : M;
  t.n0 = at.tile_n * bn;
  return t;
}

// Taller tiles among the others of a launch (192 rows among 128 or 160, 224 among 192) where those end just past a whole round of
// the chip - as the tiles of two modalities do whenever the rows of both together fill whole rounds: one M-tile goes, and its rows
// are spread over taller ones of its modality.  (65 x 8 tiles of 128x128 on 512 places ran the last 8 by themselves, 13 of 31 us at
// K = 1024, 20 of 51 at K = 2048.)  Rows of both modalities mixed, weights not in a cache, us: 128x128 tiles, M = 16384, K = N = 512
// 20.9 -> 15.2, M = 32768 33.9 -> 29.8; 128x256 tiles, M = 8192, N = 1024, K = 4096 95.6 -> 74.4, M = 2048, K = N = 4096 98.0 -> 77.7,
// M = 4096, K = 6144, N = 2048 144.4 -> 105.7.  A mask that leaves whole rounds (one modality alone) runs up to 1 % slower than on the
// kernel of one height, 128x128 tiles over K = 512 in two rounds 2.5 % (M = 32768 29.3 -> 30.0).
struct StretchShape {
  int base, tall;  // rows of a tile
  int slots;       // workgroups that the chip runs at once
};
struct Stretch {
  int tiles_v, tiles_x;  // M-tiles by modality
  int tall_v, tall_x;    // ... the first of them taller
};
// One M-tile less of tiles_m fits the whole rounds, and what is past them is no more than an eighth of a round (past that the
// 256-row tiles are the faster ones).
__host__ __device__ inline bool stretch_fits(int64_t tiles_m, int64_t tiles_n, int slots) {
  const int64_t tiles = tiles_m * tiles_n, rest = tiles % slots;
  return rest > 0 && rest < tiles && rest <= tiles_n && rest <= slots / 8;
}
// ... for some split of M rows, which has cdiv(M, base) M-tiles or one more (with their own split-K factors).
inline bool may_stretch(int64_t M, int64_t tiles_n, const StretchShape& shape, int splits = 1, int splits_more = 1) {
  const int64_t tiles_m = cdiv64(M, shape.base);
  return stretch_fits(tiles_m, tiles_n * splits, shape.slots) || stretch_fits(tiles_m + 1, tiles_n * splits_more, shape.slots);
}
// tiles_n: workgroups per M-tile (column tiles times K ranges).
__host__ __device__ inline Stretch stretch_rows(int n_vis, int M, int tiles_n, const StretchShape& shape) {
  const Stretch s{cdiv(n_vis, shape.base), cdiv(M - n_vis, shape.base), 0, 0};
  if (!stretch_fits(s.tiles_v + s.tiles_x, tiles_n, shape.slots)) return s;
  // The last M-tile of the modality that takes the fewer taller ones for it.
  const int more = shape.tall - shape.base, left_v = s.tiles_v - 1, left_x = s.tiles_x - 1;
  const int tall_v = cdiv(n_vis - left_v * shape.base, more), tall_x = cdiv(M - n_vis - left_x * shape.base, more);
  const bool can_v = tall_v <= left_v, can_x = tall_x <= left_x;
  if (can_v && (!can_x || tall_v <= tall_x)) return {left_v, s.tiles_x, tall_v, 0};
  if (can_x) return {s.tiles_v, left_x, 0, tall_x};
  return s;
}
__host__ __device__ inline TileCoord stretch_tile_coord(int L, const Stretch& s, int n_vis, int M, int tiles_n, int bn, int group_m,
                                                        const StretchShape& shape, bool* is_tall) {
  const OrderPos at = order_pos(L, s.tiles_v, s.tiles_v + s.tiles_x, tiles_n, group_m);
  TileCoord t;
  t.grp = at.tile_m < s.tiles_v ? 0 : 1;
  const int m = t.grp == 0 ? at.tile_m : at.tile_m - s.tiles_v, tall = t.grp == 0 ? s.tall_v : s.tall_x;
  *is_tall = m < tall;
  t.row0 = (t.grp == 0 ? 0 : n_vis) + m * shape.base + (m < tall ? m : tall) * (shape.tall - shape.base);
  t.row_end = t.grp == 0 ? n_vis : M;
  t.n0 = at.tile_n * bn;
  return t;
}

// Tiles of two heights in one launch, 256 rows ("tall") and 160 ("short", 11/16 of a tall one's time), chosen on the device from
// the modalities' rows: all tall, or per modality the numbers of either that cost the least - whichever the chip is done with
// earlier.  Tall tiles past the last whole round run as two short ones where those and the other short ones are one round.
// The SwiGLU GEMM over 1353 drawn shapes of 0.5 - 30 rounds that the time model gives to 256x256 tiles, caches not flushed, against
// those tiles with their remainder as 128x128 ones in a second launch (which takes 5 us where it is empty): 4.9 % less time in the
// geometric mean (8.5 % below a round, 5.8 % up to two, 4.1 % up to four, 2.3 % up to eight), 79 % of them faster.  Caches flushed,
// 3000 others: 3.5 % less, 1.8 % of them more than 3 % slower (the worst 13 %): calls whose rows end just past a whole round, where
// the mask decides which side wins.  M = 300 (150 + 150), K = 4096, 14336 columns: 122.7 -> 111.3 us, the MaskedFFN call 207 -> 184;
// M = 499, K = 5696, 16192 columns 278 -> 200.
constexpr int kTallRows = 256, kShortRows = 160, kQuarterRows = 64, kTallCost = 256, kShortCost = 176;
// A column's weight panel from memory, by the whole chip: 512 bytes per element of the contraction at 6.2 TB/s against the tall
// tile's 1.056 us per 64 of them.  Tiles of both heights of one modality read it twice (they run at different times).
constexpr int kColumnCost64 = 85;  // in 64ths
struct MixedRows {
  int tall, shrt;
};
// The cheapest: whole tall tiles, and the rest as one short tile, as two with the last tall one, or as a tall one.  (Three and
// more short tiles are never cheaper than tall ones that hold as many rows.)
__host__ __device__ inline MixedRows mixed_rows(int rows) {
  static_assert(2 * kShortCost < 2 * kTallCost && kShortCost < kTallCost && 3 * kShortCost > 2 * kTallCost, "costs");
  const int whole = rows / kTallRows, rest = rows % kTallRows;
  if (rest == 0) return {whole, 0};
  if (whole > 0 && rest <= 2 * kShortRows - kTallRows) return {whole - 1, 2};
  return rest <= kShortRows ? MixedRows{whole, 1} : MixedRows{whole + 1, 0};
}
// Into how many pieces the tall tiles past the last whole round are cut: two short ones each where those and the other short ones are
// one round, four of kQuarterRows behind whole rounds where those are one.  A round of such pieces, which share every column's weight
// panel, ends in 0.4 (64 of them) to 0.6 (256) of a tall one's time against 0.7 for two short ones each: MaskedFFN with 1 to 64 tiles past
// whole rounds, whole call, halves -> quarters: d = 1024, h = 2368, M = 6959 (20) 112.6 -> 107.6 us, d = 2048, h = 4480, M = 3818 (13)
// 196.6 -> 188.7, d = 1536, h = 3456, M = 2383 (14) 100.5 -> 96.4, d = 4096, h = 8192, M = 1280 (64) 224.6 -> 218.8.
__host__ __device__ inline int mixed_pieces(int tall, int shrt) {
  const int rest = tall % kCusPerChip;
  if (rest == 0) return 1;
  if (shrt == 0 && tall > rest && 4 * rest <= kCusPerChip) return 4;
  return 2 * rest + shrt <= kCusPerChip ? 2 : 1;
}
// When the last CU is done: tall tiles first, a CU that is free takes the next tile.  Quarters at the price of halves: at their own,
// tiles of one height were taken where two heights are the faster (d = 3072, h = 8256, M = 1872, spans 301 us against 283; of 240 calls of
// 60 layers 24 then ran more than 1 % slower than without quarters, the worst 7 %, and 10 so, the worst 2 %; as many gained).
__host__ __device__ inline int mixed_time(int tall, int shrt) {
  static_assert(kTallCost == kCusPerChip, "a shift less");
  const int rest = tall % kCusPerChip, done = tall - rest;
  if (mixed_pieces(tall, shrt) > 1) return done + kShortCost;
  if (rest == 0) return done + cdiv(shrt, kCusPerChip) * kShortCost;
  if (shrt <= kCusPerChip - rest) return done + kTallCost;
  return done + (rest * kTallCost + shrt * kShortCost) / kCusPerChip + kShortCost / 2;  // (the last tiles of a CU end anywhere in half a tile)
}
// The same with `reads` modalities' weights read from memory: of the shorter of the two times, 11/16 is not hidden (as fitted for
// the time model: kDualCost.hidden).
__host__ __device__ inline int mixed_time(const MixedRows& v, const MixedRows& x, int tiles_n) {
  const int reads = (v.tall > 0) + (v.shrt > 0) + (x.tall > 0) + (x.shrt > 0);
  const int tiles = mixed_time((v.tall + x.tall) * tiles_n, (v.shrt + x.shrt) * tiles_n), bytes = reads * tiles_n * kColumnCost64 / 64;
  return tiles > bytes ? tiles + bytes * 11 / 16 : bytes + tiles * 11 / 16;
}
// The tiles of either modality for n_vis and M - n_vis rows.
__host__ __device__ inline void mixed_choice(int n_vis, int M, int tiles_n, MixedRows* v, MixedRows* x) {
  *v = mixed_rows(n_vis);
  *x = mixed_rows(M - n_vis);
  const MixedRows all_v{cdiv(n_vis, kTallRows), 0}, all_x{cdiv(M - n_vis, kTallRows), 0};
  if (mixed_time(all_v, all_x, tiles_n) <= mixed_time(*v, *x, tiles_n)) {
    *v = all_v;
    *x = all_x;
  }
}
// Workgroups of a launch, for any split of M rows.
inline int mixed_blocks(int M, int N, int bn) {
  const int64_t tiles = (int64_t)(cdiv(M, kTallRows) + 1) * cdiv(N, bn) + kCusPerChip * 3 / 4;  // with the other pieces of cut tiles
  return kXcds * (int)(cdiv64(tiles, kXcds) + 1);
}
// Tile of workgroup `bid`; grp < 0: a surplus workgroup.  Every XCD takes an eighth of the tall tiles' order, then an eighth of the
// short ones'; an order walks the M-tiles of one height and modality in super-groups of `group`, column by column, so that the tiles
// of a column share the weight panel.
__host__ __device__ inline TileCoord mixed_tile_coord(int bid, int n_vis, int M, int N, int bn, int group, bool* is_tall, bool* is_quarter = nullptr) {
  TileCoord t{-1, 0, 0, 0};
  const int tiles_n = cdiv(N, bn);
  MixedRows v, x;
  mixed_choice(n_vis, M, tiles_n, &v, &x);
  const int tall = (v.tall + x.tall) * tiles_n, shrt = (v.shrt + x.shrt) * tiles_n;
  const int cut = mixed_pieces(tall, shrt);
  const int whole = cut > 1 ? tall / kCusPerChip * kCusPerChip : tall;  // tall tiles that run as such
  const int pieces = cut * (tall - whole);
  const int per_tall = cdiv(whole, kXcds), per_short = cdiv(pieces + shrt, kXcds);
  int slot = bid / kXcds;
  *is_tall = slot < per_tall;
  if (!*is_tall) slot -= per_tall;
  const int per = *is_tall ? per_tall : per_short;
  int L = (bid % kXcds) * per + slot;
  if (slot >= per || L >= (*is_tall ? whole : pieces + shrt)) return t;
  const bool piece = !*is_tall && L < pieces;
  const int part = piece ? L & (cut - 1) : 0;
  if (piece) L = whole + (cut == 4 ? L / 4 : L / 2);
  else if (!*is_tall) L -= pieces;
  const bool quarter = piece && cut == 4;
  if (is_quarter != nullptr) *is_quarter = quarter;
  const bool of_tall = *is_tall || piece;
  const int own_v = of_tall ? v.tall : v.shrt, own_x = of_tall ? x.tall : x.shrt;  // M-tiles of this height by modality
  const int grp = L < own_v * tiles_n ? 0 : 1;
  if (grp == 1) L -= own_v * tiles_n;
  const int own = grp == 0 ? own_v : own_x;
  int first = 0, gsz = own;  // super-group of M-tiles, dealt evenly (routed_tile_coord)
  if (own > group) {
    const int groups = cdiv(own, group), s = ((L / tiles_n + 1) * groups - 1) / own;
    first = s * own / groups;
    gsz = (s + 1) * own / groups - first;
    L -= first * tiles_n;
  }
  const int begin = grp == 0 ? 0 : n_vis, end = grp == 0 ? n_vis : M;
  t.row0 = begin + (of_tall ? 0 : (grp == 0 ? v.tall : x.tall) * kTallRows) + (first + L % gsz) * (of_tall ? kTallRows : kShortRows);
  t.row_end = piece && t.row0 + kTallRows < end ? t.row0 + kTallRows : end;
  t.row0 += part * (quarter ? kQuarterRows : kShortRows);
  if (quarter && t.row0 + kQuarterRows < t.row_end) t.row_end = t.row0 + kQuarterRows;
  t.n0 = (L / gsz) * bn;
  if (t.row0 < t.row_end) t.grp = grp;
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
