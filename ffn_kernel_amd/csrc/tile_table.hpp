// gfx950 tile table: which kernel family and macro tile each (op, M, K, N) uses.
//
// The reference looks its tile up with find_spec(table, M // 1024) in A100-tuned JSON files
// holding one entry each (ffn_kernel/utils.py:3-5, ffn_kernel/bf16_linear_fwd.json,
// bf16_ffn_fwd.json, bf16_linear_bwd.json).  On MI355X the choice is driven by how many
// workgroups a shape yields against 256 CUs, so the table is keyed on the real extents.
#pragma once
#include "launch.hpp"
#include "common.hpp"
#include "gemm_sched.hpp"

namespace ffnk {

constexpr int kCus = 256;

// Smallest M for which the LDS-tiled path is used by the FFN forward; below it the
// weight-streaming kernels win because the op is bound by reading the weights once.
constexpr int kStreamMaxM = 64;

struct TileChoice {
  int tile;    // TileId
  int splits;  // split-K factor (weight-gradient GEMM only)
  bool tuned;  // the pair is a measured plan (as timed by the tuner), not the rules' guess
};

// Contractions that the direct kernels run: whole 64-element slabs, or 16-byte pieces with the first slab partly ahead of
// the contraction (clear_head in gemm_nt.hpp).  Under 128 elements the part ahead is a third of the work and more, and the
// register-staged loop stays.
constexpr int kRaggedMinK = 128;
inline bool direct_contraction(int64_t K) { return K > 0 && (K % 64 == 0 || (K % 8 == 0 && K >= kRaggedMinK)); }

// The direct global->LDS path addresses operands with 32-bit byte offsets: from the start of A when its rows are gathered,
// from the tile's first row otherwise (at most 256 rows away).  The base of a contraction that is no whole number of slabs
// lies 2 * (-K mod 64) bytes ahead of the operand (clear_head), and the offsets past slab 0 are larger by as much.
inline bool direct_ok(int64_t K, int64_t gathered_rows, int64_t lda, int64_t ldb) {
  constexpr int64_t k4g = (int64_t)1 << 32;
  if (!direct_contraction(K)) return false;
  const int64_t ahead = 2 * (round_up64(K, 64) - K);
  if (gathered_rows > 0 && gathered_rows * lda * 2 + ahead >= k4g) return false;
  return 256 * lda * 2 + ahead < k4g && 256 * ldb * 2 + ahead < k4g;
}

// Measured plans.  `python -m ffn_kernel_amd.tune --emit` times every candidate (tile x split-K factor)
// per operation, shape and M bucket on the GPU and writes tile_table_gen.hpp: one entry wherever the best
// candidate beat the rules and the cost model below by a margin.  The pick_* functions consult these
// entries first (exact contraction / output extents, M inside the bucket) and fall back to the rules.
// This is what the reference's find_spec/*.py searches and bf16_*.json tables are to its kernels
// (find_spec/find.py:18-64, ffn_kernel/utils.py:3-5).
enum TunedOp : int {
  TUNED_PLAIN = 0,   // MaskedLinear forward (gathered rows in, scattered rows out; whole-call timing): k = contraction, n = output columns
  TUNED_DUAL = 1,    // SwiGLU GEMM: k = contraction (d), n = output columns (h)
  TUNED_SPLITK = 2,  // weight-gradient GEMM: k = R (rows of the in-place operand), n = Cc
  TUNED_DOWN = 3,    // MaskedFFN down projection (routed-order rows in, scattered out; stage timing): k = contraction (h), n = output columns (d)
  TUNED_NONE = -1,   // a GEMM the tuner does not measure (the backward's dx GEMMs): no measured plans
};
struct TunedPlan {
  int op;            // TunedOp, -1 ends the table
  int m_lo, m_hi;    // rows M of the call, inclusive
  int k, n;
  int tile, splits;
  int group_m;       // M-tiles per super-group of the tile order (GemmArgs::group_m); 0 = the tile's own
};
}  // namespace ffnk
#include "tile_table_gen.hpp"
namespace ffnk {

inline const TunedPlan* tuned_plan(int op, int64_t M, int64_t k, int64_t n) {
  for (const TunedPlan* p = kTunedPlans; p->op >= 0; ++p)
    if (p->op == op && p->k == k && p->n == n && M >= p->m_lo && M <= p->m_hi) return p;
  return nullptr;
}

// Super-group size of a measured plan for this operation and shape, 0 where there is none (the tile's own then).
inline int tuned_group_m(int op, int64_t M, int64_t k, int64_t n) {
  const TunedPlan* t = tuned_plan(op, M, k, n);
  return t ? t->group_m : 0;
}

// Tile and split-K factor of a routed GEMM.  The visual and the text rows each end in a partial tile, so a call has
// cdiv(M, block_m) M-tiles or one more, which only the device knows: `splits` is for the one count and `splits_more` for
// the other (the kernel and the reduce pass pick by counts[]); either both are 1 or neither is.
struct RoutedPlan {
  int tile;
  int splits;
  int splits_more;
};

// Time of a direct-path GEMM in us, fitted to every tile and split factor at drawn shapes, up to four sets of weights in turn
// (600 MB of them, where the layer is that large), one or both modalities present: 8000 SwiGLU GEMMs (M = 33 ... 8192,
// d = 1024 ... 8192, h = 2 ... 3.5 d) and 8000 single-weight GEMMs (M = 9 ... 12000, K = 128 ... 28672, N = 512 ... 8192), a
// quarter of them off multiples of 64; rms error 7 %.  A round of the chip takes base + slabs * per_slab.  A partial round
// takes a part of it that depends on the workgroups of the fullest CU: `first` (the launch is less than a round) and `again`
// (behind whole rounds) hold, per number of workgroups, the part just past the number below it and the part when every CU
// has as many.  The weights arrive at `tbs` TB/s, token rows and results at `io`; of the products' and the weights' times the
// smaller is partly hidden behind the larger.  Where K % 64 != 0 the rows of a packed operand start anywhere in a 128-byte
// line and every 128-byte piece of a slab lies in two lines: a slab takes `ragged` times as long, the more the fewer flops the
// tile has per byte it loads.
// Without the steps by workgroups per CU (a partial round taken as linear in them) and with the likelier M-tile count alone,
// the plans were 2.8 % (single weight) and 4.7 % (SwiGLU) behind the best of each shape in the geometric mean, and more than
// 8 % behind the rules by tile count below in 2.9 % and 5.1 % of 3900 / 4500 shapes that no fit has seen (K = 11392, N = 4544,
// M = 403: 127 us, rules 84); with both, 1.5 % and 3.8 % behind the best, 22 % and 14 % ahead of the rules, and more than 8 %
// behind them in 0.8 % and 2.8 % (K = 11392, N = 4544, M = 403: 75 us).
constexpr int kMaxPerCu = 3;
struct TileCost {
  int tile, per_cu;
  double base, per_slab, tbs, ragged;
  double first[2 * kMaxPerCu], again[2 * kMaxPerCu];
};
struct GemmCost {
  double launch, hidden, io, tail;   // tail: the second launch of a big tile's remainder
  double reduce, reduce_tbs;         // split plans: the reduce pass, and the partials' way out and back
};
// (The SwiGLU GEMM's four-wave 256x256 tile is priced as whole rounds and a remainder launch.  Up to eight rounds it runs beside
// 160-row tiles in one launch instead, 3.5 % faster on drawn shapes: the plan takes it somewhat less often than it could.)
constexpr GemmCost kDualCost = {4.073, 0.683, 3.0, 3.968, 0.0, 1.0}, kPlainCost = {5.448, 0.32, 11.972, 17.518, 2.151, 7.525};
constexpr TileCost kDualCosts[] = {
    {TILE_256x256_W4, 1, 8.145, 1.056, 9.0, 1.319, {0.956, 1.0}, {1.003, 1.0}},
    {TILE_128x128_W4, 2, 0.64, 0.853, 8.894, 1.277, {0.825, 0.841, 1.012, 1.0}, {0.762, 0.857, 0.862, 1.0}},
    {TILE_SMALL_W4, 3, 0.0, 0.899, 7.554, 1.341, {0.648, 0.74, 0.779, 0.77, 1.105, 1.0}, {0.434, 0.556, 0.638, 0.704, 0.962, 1.0}},
    {TILE_128x128_R4, 1, 2.181, 0.436, 9.0, 1.464, {1.015, 1.0}, {0.899, 1.0}},
    {TILE_128x256_R3, 1, 2.476, 0.724, 9.0, 1.486, {0.982, 1.0}, {0.907, 1.0}},
    {TILE_64x128_R3, 2, 0.0, 0.612, 7.659, 1.469, {0.679, 0.65, 1.124, 1.0}, {0.531, 0.606, 0.99, 1.0}}};
constexpr TileCost kPlainCosts[] = {
    {TILE_256x256_W8, 1, 4.964, 1.261, 6.216, 1.106, {0.772, 1.0}, {0.886, 1.0}},
    {TILE_256x256_W4, 1, 12.067, 1.188, 4.001, 1.117, {0.769, 1.0}, {0.207, 1.0}},
    {TILE_128x128_W4, 2, 3.08, 0.874, 5.329, 1.234, {0.51, 0.714, 0.862, 1.0}, {0.565, 0.691, 0.867, 1.0}},
    {TILE_SMALL_W4, 3, 1.882, 0.891, 5.278, 1.235, {0.327, 0.581, 0.598, 0.682, 0.939, 1.0}, {0.339, 0.404, 0.517, 0.642, 0.899, 1.0}},
    {TILE_128x128_R4, 1, 3.892, 0.417, 6.008, 1.352, {0.642, 1.0}, {0.826, 1.0}},
    {TILE_128x256_R3, 1, 6.127, 0.679, 5.596, 1.317, {0.694, 1.0}, {0.825, 1.0}},
    {TILE_64x128_R3, 2, 2.924, 0.519, 5.577, 1.38, {0.404, 0.589, 0.868, 1.0}, {0.425, 0.499, 0.808, 1.0}},
    // (forward GEMMs only; 6700 measurements at 400 shapes of their own, 7.5 and 8 % rms, GemmCost as it is)
    {TILE_192x256_W4, 1, 5.102, 0.879, 6.529, 1.258, {0.845, 1.0}, {0.929, 1.0}},
    {TILE_160x256_W4, 1, 4.303, 0.784, 6.305, 1.307, {0.814, 1.0}, {0.852, 1.0}}};

// Single-weight tiles that may have taller ones among them (stretch_rows), and the part of a round that what is just past the whole
// rounds then takes.  Measured 0.05 - 0.27 (128x128) and 0.04 - 0.26 (128x256) at K = 512 ... 8192; for the other two it is what the taller
// tile has more rows.
struct StretchCost {
  StretchShape shape;
  double part;
};
inline StretchCost stretch_cost(int tile) {
  switch (tile) {
    case TILE_128x128_W4: return {{128, 192, 2 * kCus}, 0.17};
    case TILE_128x256_R3: return {{128, 192, kCus}, 0.21};
    case TILE_160x256_W4: return {{160, 192, kCus}, 0.17};
    case TILE_192x256_W4: return {{192, 224, kCus}, 0.17};
    default: return {{0, 0, 0}, 0.0};
  }
}

// Part of a round that `rest` workgroups take on per_cu slots of every CU.
inline double round_part(const double* knots, int64_t rest) {
  const int n = (int)cdiv64(rest, kCus);
  const double lo = knots[2 * (n - 1)], hi = knots[2 * n - 1];
  return lo + (hi - lo) * ((double)rest / (double)kCus - (double)(n - 1));
}

// The time of one tile's launches, for any M-tile count, split factor and number of modalities: what these share is taken out here, as
// a plan prices some three hundred of them.
struct TileTimer {
  const TileCost& c;
  const GemmCost& g;
  const bool dual;
  const int64_t M, n_out;
  const TileGeom geom;
  const int tiles_n, slots, slabs;
  const double slow;      // a slab's time against one of whole lines
  const double per_slab, io;
  double weights[2];      // one modality, both
  const StretchCost stretched;

  TileTimer(const TileCost& cost, bool dual_, int64_t M_, int64_t n_out_, int64_t K)
      : c(cost), g(dual_ ? kDualCost : kPlainCost), dual(dual_), M(M_), n_out(n_out_), geom(tile_geom(cost.tile, dual_)),
        tiles_n((int)cdiv64(n_out_, geom.block_n_out)), slots(kCus * cost.per_cu), slabs((int)cdiv64(K, 64)),
        slow(K % 64 == 0 ? 1.0 : cost.ragged), per_slab(cost.per_slab * slow),
        io(g.launch + (double)M_ * (double)(K + n_out_) * 2.0e-6 / g.io),
        stretched(dual_ ? StretchCost{} : stretch_cost(cost.tile)) {
    for (int m = 1; m <= 2; ++m) weights[m - 1] = m * (dual ? 2.0 : 1.0) * (double)K * (double)n_out * 2.0e-6 / c.tbs;
  }
  // The rounds of the chip.  `range`: slabs of a K range.
  double rounds(int tiles_m, int splits, int range, bool stretch) const {
    const int64_t tiles = (int64_t)tiles_m * tiles_n * splits;
    const int64_t full = tiles < (int64_t)1 << 31 ? (int64_t)((uint32_t)tiles / (uint32_t)slots) : tiles / slots;
    const int64_t rest = tiles - full * slots;
    const double round = c.base + per_slab * (double)range;
    double time = (double)full * round;
    if (rest > 0) {
      if (stretch && stretched.part > 0.0 && stretch_fits(tiles_m, (int64_t)tiles_n * splits, stretched.shape.slots)) {
        time += round * stretched.part;
      } else if (!is_big_tile(c.tile) || splits > 1 || full == 0 || (dual && rest > slots / 2)) {  // whole_round_tiles
        time += round * round_part(full > 0 ? c.again : c.first, rest);
      } else if (dual) {  // four 128-row tiles for each of the remainder
        const TileCost& s = kDualCosts[1];
        const double small = s.base + (slow == 1.0 ? s.per_slab : s.per_slab * s.ragged) * (double)slabs;
        time += g.tail + small * round_part(s.first, 4 * rest);
      } else {            // split tail
        time += g.tail + c.base + per_slab * (double)slabs / (double)tail_split_factor((int)rest, slabs);
      }
    }
    return time;
  }
  double total(double rounds, int modalities, int splits) const {
    const double w = weights[modalities - 1];
    double time = io + (rounds > w ? rounds + g.hidden * w : w + g.hidden * rounds);
    if (splits > 1) time += g.reduce + (double)splits * (double)M * (double)n_out * 8.0e-6 / g.reduce_tbs;
    return time;
  }
  int range(int splits) const { return cdiv(slabs, splits); }
  double time(int tiles_m, int modalities, int splits, bool stretch) const {
    return total(rounds(tiles_m, splits, range(splits), stretch), modalities, splits);
  }
};

// Split factors the cost model considers: whole 64-element slabs, at least four to a range, no empty range.
inline bool routed_split_ok(int64_t K, int s) {
  const int64_t nk = cdiv64(K, 64);
  return s == 1 || (nk / s >= 4 && cdiv64(nk, cdiv64(nk, s)) == s);
}

// What a plan is chosen by.  With both modalities present the rows of the two make cdiv(M, block_m) M-tiles or one more, and
// where that starts another round the times differ by up to a half.  One more it is at (M / block_m rounded up) *
// ((M - 1) mod block_m) of the M - 1 ways to split M; masks that set every row by itself split M about evenly.  The score is
// the product of three times: over all splits (weight 1), at an even split (weight 2), of one modality alone (weight 2).
inline int even_deviation(int64_t M) {  // a third of sqrt(M): how far such a mask is off an even split
  int dev = 0;
  while ((dev + 1) * (dev + 1) * 9 <= M) ++dev;
  return dev;
}
inline bool even_split_has_one_more(int64_t M, int64_t bm) {
  const int64_t dev = even_deviation(M);
  const int64_t visual = (M + 1) / 2 + dev < M ? (M + 1) / 2 + dev : M;
  return cdiv64(visual, bm) + cdiv64(M - visual, bm) > cdiv64(M, bm);
}
inline double plan_score(const TileTimer& t, bool even_more, int splits, int splits_more, bool stretch) {
  const int64_t M = t.M, bm = t.geom.block_m, less = cdiv64(M, bm);
  const double p = M > 1 ? (double)(less * ((M - 1) % bm)) / (double)(M - 1) : 0.0;
  const double rounds = t.rounds((int)less, splits, t.range(splits), stretch);
  const double both = t.total(rounds, 2, splits), one = t.total(rounds, 1, splits);
  const double more = t.time((int)less + 1, 2, splits_more, stretch);
  const double even = even_more ? more : both;
  return ((1.0 - p) * both + p * more) * even * even * one * one;
}
inline double plan_score(const TileCost& c, bool dual, int64_t M, int64_t n_out, int64_t K, int splits, int splits_more, bool stretch = true) {
  const TileTimer t(c, dual, M, n_out, K);
  return plan_score(t, even_split_has_one_more(M, t.geom.block_m), splits, splits_more, stretch);
}

// The rules by tile count: where the model does not apply, and what its plan has to beat.
inline int rule_tile(int64_t M, int64_t n_out, bool dual, int64_t K) {
  auto tiles = [&](int tile) {
    const TileGeom t = tile_geom(tile, dual);
    return cdiv64(M, t.block_m) * cdiv64(n_out, t.block_n_out);
  };
  // Past two rounds of the chip, four 128x128-per-wave wavefronts lead for the SwiGLU kernel at 128 rows x
  // 128x128 (a third fewer LDS reads per flop; measured 4 % faster at M = 32768, d = 4096, h = 14336); so do the
  // single-weight kernels over a long contraction (1-2.5 % faster at K = 4096 and 14336, N = 4096, M >= 16384),
  // which otherwise keep eight wavefronts of 128x64 (less exposed when K is short).
  if (tiles(TILE_256x256_W8) >= 2 * kCus) return dual || (K >= 4096 && K % 64 == 0) ? TILE_256x256_W4 : TILE_256x256_W8;
  if (tiles(TILE_128x128_W4) >= kCus) return TILE_128x128_W4;
  return TILE_SMALL_W4;
}

inline RoutedPlan rule_plan(int64_t M, int64_t n_out, int64_t K);

inline int max_splits(const RoutedPlan& p) { return p.splits > p.splits_more ? p.splits : p.splits_more; }
// fp32 workspace of a plan: the partials of all rows where K is split for the whole GEMM, or the kTailSlots tiles of the split
// tail of an unsplit 256x256 tile - only a launch of more than one round has one.
inline size_t plan_partial_bytes(const RoutedPlan& p, int64_t M, int64_t n_out, int64_t K) {
  if (p.splits > 1) return ws_align((size_t)max_splits(p) * M * n_out * 4);
  return is_big_tile(p.tile) && direct_contraction(K) && (cdiv64(M, 256) + 1) * cdiv64(n_out, 256) > kCus
             ? ws_align((size_t)kTailSlots * 256 * 256 * 4) : 0;
}

// The plan with the smallest score among all tiles and split factors.  `forward`: a GEMM over row-major weights that scatters its
// rows (CanStretch), which has the 192- and 160-row tiles too.  `split`: N % 4 == 0 and the reduce pass takes M; `room`:
// bytes that the caller has for partials.  The rules' plan stays unless the model sees a gain of kModelMargin, near which its
// choice is as often the slower one (MaskedFFN d = 1024, h = 2048, M = 8192, runs of both modalities: 133 us with the model's
// 256x256 tiles under the down projection, 129 with the rules' 128x128): without it 6.0 % of the SwiGLU and 2.1 % of the
// single-weight shapes ran more than 3 % slower than on the rules' plan, with it 5.1 % and 1.7 %.
constexpr double kModelMargin = 1.03;
// A plan on 192- or 160-row tiles replaces another, up to two rounds of the chip, where the model sees it 7 % ahead over the splits
// of the rows, no slower with one modality and nowhere kModelMargin behind (the model puts 256- and 128-row tiles 2 - 6 % above
// what they take, those two 1 %).  6452 drawn single-weight GEMMs with such a plan, three masks each, timed against the plans without:
// 1.13 times as fast in the geometric mean with one modality and with both, 1.1 % of the calls more than 3 % slower (4.5 % below 12
// slabs), 0.02 % more than 10 %.  At 16 splits of the rows instead of kSplitsOfRows, none of them even, 81 more had one: 8 % of their
// calls more than 3 % slower, the worst by half (K = 3584, N = 6400, M = 1936, even splits: a twelfth M-tile, a second round).  Between
// two and three rounds 1.03, with 23 % more than 3 % slower; by the score alone 12 % more than 3 % slower, and 4 % more than 8 %.
constexpr double kForwardGain = 0.93;
constexpr int kSplitsOfRows = 64;
constexpr size_t kAnyRoom = ~(size_t)0;
inline RoutedPlan compute_model_plan(bool dual, int64_t M, int64_t n_out, int64_t K, bool split, size_t room = kAnyRoom, bool forward = true) {
  constexpr int kSplits[] = {2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16}, kMaxCosts = 9;
  static_assert(sizeof(kPlainCosts) / sizeof(TileCost) <= kMaxCosts && sizeof(kDualCosts) / sizeof(TileCost) <= kMaxCosts, "tiles");
  const TileCost* costs = dual ? kDualCosts : kPlainCosts;
  const int n_costs = dual ? (int)(sizeof(kDualCosts) / sizeof(TileCost)) : (int)(sizeof(kPlainCosts) / sizeof(TileCost));
  const RoutedPlan rule = dual ? RoutedPlan{rule_tile(M, n_out, true, K), 1, 1} : rule_plan(M, n_out, K);
  RoutedPlan p{TILE_SMALL_W4, 1, 1};
  double best = -1.0, keep = -1.0;
  auto fits = [&](const RoutedPlan& q) { return dual || plan_partial_bytes(q, M, n_out, K) <= room; };
  // The factors that this contraction and room allow, and the slabs of a range.
  int factors[sizeof(kSplits) / sizeof(int)], ranges[sizeof(kSplits) / sizeof(int)], n_factors = 0;
  if (!dual && split)
    for (const int k : kSplits)
      if (routed_split_ok(K, k) && fits({TILE_SMALL_W4, k, k})) {
        factors[n_factors] = k;
        ranges[n_factors++] = (int)cdiv64(cdiv64(K, 64), k);
      }
  // The best factors of a tile for each M-tile count; either both are split or neither is (1: none fits).
  auto best_split = [&](const TileTimer& t, bool stretch) {
    const int less = (int)cdiv64(M, t.geom.block_m);
    int s = 1, s_more = 1;
    double t_less = 0.0, t_more = 0.0;
    for (int i = 0; i < n_factors; ++i) {
      const int k = factors[i];
      const double rounds = t.rounds(less, k, ranges[i], stretch);
      const double a = t.total(rounds, 2, k) * t.total(rounds, 1, k);
      const double b = t.total(t.rounds(less + 1, k, ranges[i], stretch), 2, k);
      if (s == 1 || a < t_less) { t_less = a; s = k; }
      if (s_more == 1 || b < t_more) { t_more = b; s_more = k; }
    }
    return RoutedPlan{t.c.tile, s, s_more};
  };
  for (int i = 0; i < n_costs; ++i) {
    const TileCost& c = costs[i];
    if (forward_only(c.tile)) continue;
    const TileTimer t(c, dual, M, n_out, K);
    const bool even_more = even_split_has_one_more(M, t.geom.block_m);
    auto consider = [&](const RoutedPlan& q) {
      if (!fits(q)) return;
      const double score = plan_score(t, even_more, q.splits, q.splits_more, false);
      if (best < 0.0 || score < best) {
        best = score;
        p = q;
      }
    };
    consider({c.tile, 1, 1});
    if (n_factors > 0 && c.tile != TILE_256x256_W4) consider(best_split(t, false));
    if (c.tile == rule.tile && (rule.splits == 1 || split) && fits(rule)) keep = plan_score(t, even_more, rule.splits, rule.splits_more, false);
  }
  constexpr double m = kModelMargin * kModelMargin * kModelMargin * kModelMargin * kModelMargin;  // a score is five times long
  if (keep > 0.0 && keep < best * m) p = rule;
  if (dual || !forward) return p;
  // The heights between 128 and 256 rows, where they lead at nearly every split of the rows (kForwardGain).
  auto cost = [&](int tile) -> const TileCost& {
    int i = 0;
    while (costs[i].tile != tile) ++i;
    return costs[i];
  };
  RoutedPlan between = p;
  best = -1.0;
  for (int i = 0; i < n_costs; ++i) {
    const TileCost& c = costs[i];
    if (!forward_only(c.tile)) continue;
    const TileTimer t(c, false, M, n_out, K);
    const bool even_more = even_split_has_one_more(M, t.geom.block_m);
    const int64_t tiles = cdiv64(M, t.geom.block_m) * t.tiles_n;
    if (tiles > 2 * kCus) continue;
    for (int split_too = 0; split_too <= (n_factors > 0 ? 1 : 0); ++split_too) {
      const RoutedPlan q = split_too ? best_split(t, true) : RoutedPlan{c.tile, 1, 1};
      if (tiles * q.splits > 2 * kCus || !fits(q)) continue;
      const double score = plan_score(t, even_more, q.splits, q.splits_more, true);
      if (best < 0.0 || score < best) {
        best = score;
        between = q;
      }
    }
  }
  if (best < 0.0) return p;
  // A plan's times by M-tile count and stretch: four numbers, whatever the split of the rows.
  struct Times {
    TileTimer t;
    RoutedPlan q;
    int less;
    bool fits[2];
    double at[2][2];
    Times(const TileCost& c, const RoutedPlan& plan, int64_t M, int64_t n_out, int64_t K)
        : t(c, false, M, n_out, K), q(plan), less((int)cdiv64(M, t.geom.block_m)) {
      for (int more = 0; more < 2; ++more) {
        const int splits = more ? q.splits_more : q.splits;
        fits[more] = t.stretched.part > 0.0 && stretch_fits(less + more, (int64_t)t.tiles_n * splits, t.stretched.shape.slots);
        for (int stretch = 0; stretch <= (fits[more] ? 1 : 0); ++stretch) at[more][stretch] = t.time(less + more, 2, splits, stretch != 0);
      }
    }
    double time(int n_vis) const {
      const int bm = t.geom.block_m, M = (int)t.M, more = cdiv(n_vis, bm) + cdiv(M - n_vis, bm) - less;
      if (!fits[more]) return at[more][0];
      const Stretch s = stretch_rows(n_vis, M, t.tiles_n * (more ? q.splits_more : q.splits), t.stretched.shape);
      return at[more][s.tall_v + s.tall_x > 0 ? 1 : 0];
    }
    double one_modality() const {
      const bool stretch = fits[0] && stretch_rows((int)t.M, (int)t.M, t.tiles_n * q.splits, t.stretched.shape).tall_v > 0;
      return t.time(less, 1, q.splits, stretch);
    }
  };
  const Times a(cost(p.tile), p, M, n_out, K), b(cost(between.tile), between, M, n_out, K);
  const double one = b.one_modality() / a.one_modality();
  if (one > 1.0) return p;
  // About even splits (a mask that sets every row by itself is off by sqrt(M) / 2), where two partial M-tiles are one too many for a
  // whole round more often than elsewhere ...
  for (int i = -4; i <= 4; ++i) {
    const int off = (int)(M / 2) + i * even_deviation(M) / 2, n_vis = off < 1 ? 1 : off < M ? off : (int)M - 1;
    if (b.time(n_vis) >= kModelMargin * a.time(n_vis)) return p;
  }
  // ... and from one end to the other, no two with the same remainder.
  double product = one, gain = kForwardGain;
  for (int i = 1; i < kSplitsOfRows; ++i) {
    const int64_t at = M * i / kSplitsOfRows + i * 37 % 61, n_vis = at < 1 ? 1 : at < M ? at : M - 1;
    const double r = b.time((int)n_vis) / a.time((int)n_vis);
    if (r >= kModelMargin) return p;
    product *= r;
    gain *= kForwardGain;
  }
  return product < gain ? between : p;
}

// The model is a pure function of the extents and takes host time: 2.7 us at K = N = 1024, 4.4 at 2048, 7.5 at K = 14336, N = 4096 for
// a single-weight forward (7.4, 10.9 and 15.7 with every time priced from its extents alone), 0.6 for SwiGLU; every thread keeps the last
// plans.  Extents are mostly multiples of 32 and more: the slot comes from the top of a product, where all their bits arrive.
inline unsigned model_plan_slot(bool dual, int64_t M, int64_t n_out, int64_t K, bool split, size_t room, bool forward = true) {
  constexpr uint64_t kMul = 0x9E3779B97F4A7C15ull;
  uint64_t x = (uint64_t)M;
  for (const uint64_t v : {(uint64_t)n_out, (uint64_t)K, (uint64_t)room * 8 + (forward ? 0 : 4) + (dual ? 2 : 0) + (split ? 1 : 0)}) x = (x ^ (x >> 29)) * kMul + v;
  return (unsigned)((x ^ (x >> 32)) * kMul >> 59);
}
inline RoutedPlan model_routed_plan(bool dual, int64_t M, int64_t n_out, int64_t K, bool split, size_t room = kAnyRoom, bool forward = true) {
  struct Entry {
    int64_t M = -1, n_out, K;
    bool dual, split, forward;
    size_t room;
    RoutedPlan plan;
  };
  static thread_local Entry memo[32];
  Entry& e = memo[model_plan_slot(dual, M, n_out, K, split, room, forward)];
  if (e.M != M || e.n_out != n_out || e.K != K || e.dual != dual || e.split != split || e.forward != forward || e.room != room)
    e = Entry{M, n_out, K, dual, split, forward, room, compute_model_plan(dual, M, n_out, K, split, room, forward)};
  return e.plan;
}

// Where the model applies: up to two rounds of 256x256 tiles; past them the rule below takes that tile.
inline bool model_applies(bool dual, int64_t M, int64_t n_out, int64_t K) {
  const TileGeom t = tile_geom(TILE_256x256_W8, dual);
  return M > 0 && n_out > 0 && direct_contraction(K) && cdiv64(M, t.block_m) * cdiv64(n_out, t.block_n_out) < 2 * kCus;
}

// Routed GEMM over M rows and n_out output columns (K: the contraction, 0 = not known to the caller).
// `op`: whose measured plans apply (TUNED_NONE: none; the tuner times each operation with its own gather /
// scatter pattern and its own launches around the GEMM, so one operation's plan says nothing about another's).
inline int pick_routed_tile(int64_t M, int64_t n_out, bool dual, int64_t K = 0, bool use_table = true,
                            int op = TUNED_PLAIN) {
  if (use_table && K > 0 && (dual || op != TUNED_NONE)) {
    if (const TunedPlan* t = tuned_plan(dual ? TUNED_DUAL : op, M, K, n_out))
      if (dual || t->splits == 1) return t->tile;
  }
  if (dual && model_applies(true, M, n_out, K)) return model_routed_plan(true, M, n_out, K, false).tile;
  return rule_tile(M, n_out, dual, K);
}

// What the model's plan has to beat, and where the model does not apply: when the output yields fewer
// tiles than the chip has workgroup slots and the contraction is long, cutting K into `splits` ranges of whole 64-element
// slabs fills the chip, at the price of fp32 partials (4 * splits * M * n_out bytes written, then read by the reduce pass):
//   time = rounds * (5 us + slabs_per_range * t_slab) + splits * M * n_out * 8 bytes / 4 TB/s
//   rounds = ceil(tiles * splits / slots),  slots = 256 CUs * workgroups per CU by LDS use,
//   t_slab = 1.2 us for the 256x256 tile, 0.8 us for the 128x128 and 128x64 tiles.
// The unsplit 256x256 tile is priced with its split tail.  Limited to M <= 4096 (above it the tiles fill the chip).
inline double routed_plan_cost(int64_t M, int64_t n_out, int64_t K, int tile, int splits) {
  const TileGeom t = tile_geom(tile, false);
  const int64_t tiles = (cdiv64(M, t.block_m) + 1) * cdiv64(n_out, t.block_n_out);
  const int64_t slots = (int64_t)kCus * (tile == TILE_SMALL_W4 ? 3 : tile == TILE_128x128_W4 ? 2 : 1);
  const double t_slab = (tile == TILE_256x256_W8 || tile == TILE_256x256_W4) ? 1.2 : tile == TILE_128x128_R4 ? 0.4 : 0.8;
  const int64_t slabs = cdiv64(cdiv64(K, 64), splits);
  const double reduce = splits > 1 ? (double)splits * (double)M * (double)n_out * 8.0 / 4.0e6 : 0.0;
  if (tile == TILE_256x256_W8 && splits == 1 && direct_contraction(K) && tiles > slots) {
    // Unsplit 256x256 tiles past one round: the launcher runs the whole rounds, then the remaining tiles
    // cut into K ranges (split tail) - a fraction of a round, a second launch and a small reduce pass.
    const int64_t tail = tiles % slots;
    double c = (double)(tiles / slots) * (5.0 + (double)slabs * t_slab);
    if (tail > 0) c += 15.0 + (double)cdiv64(slabs, tail_split_factor((int)tail, (int)slabs)) * t_slab;
    return c;
  }
  return (double)cdiv64(tiles * splits, slots) * (5.0 + (double)slabs * t_slab) + reduce;
}

// Best split for a given tile: ranges of at least 8 slabs, no empty range.
inline int pick_routed_splits(int64_t M, int64_t n_out, int64_t K, int tile) {
  if (M > 4096 || !direct_contraction(K) || tile == TILE_256x256_W4) return 1;
  const int64_t nk = cdiv64(K, 64);
  int best = 1;
  double best_cost = routed_plan_cost(M, n_out, K, tile, 1);
  for (int s = 2; s <= 16 && nk / s >= 8; ++s) {
    if (cdiv64(nk, cdiv64(nk, s)) != s) continue;  // would leave an empty range
    const double c = routed_plan_cost(M, n_out, K, tile, s);
    if (c < best_cost) {
      best_cost = c;
      best = s;
    }
  }
  return best;
}

inline RoutedPlan rule_plan(int64_t M, int64_t n_out, int64_t K) {
  RoutedPlan p;
  p.tile = rule_tile(M, n_out, false, K);
  p.splits = p.splits_more = 1;
  if (M > 4096 || !direct_contraction(K)) return p;
  double best_cost = 0.0;
  const int cand[3] = {TILE_256x256_W8, TILE_128x128_W4, TILE_SMALL_W4};
  for (int i = 0; i < 3; ++i) {
    const int s = pick_routed_splits(M, n_out, K, cand[i]);
    const double c = routed_plan_cost(M, n_out, K, cand[i], s);
    if (i == 0 || c < best_cost) {
      best_cost = c;
      p.tile = cand[i];
      p.splits = p.splits_more = s;
    }
  }
  return p;
}

inline RoutedPlan pick_routed_plan(int64_t M, int64_t n_out, int64_t K, bool use_table = true, int op = TUNED_DOWN) {
  RoutedPlan p;
  if (use_table && op != TUNED_NONE)
    if (const TunedPlan* t = tuned_plan(op, M, K, n_out)) {
      p.tile = t->tile;
      p.splits = p.splits_more = (direct_contraction(K) && M < 65536 && n_out % 4 == 0) ? t->splits : 1;
      return p;
    }
  if (op != TUNED_NONE && model_applies(false, M, n_out, K)) return model_routed_plan(false, M, n_out, K, M < 65536 && n_out % 4 == 0);
  return rule_plan(M, n_out, K);
}

// Weight-gradient GEMM: two [R, Cc] outputs, contraction over about M / 2 rows each; `batch` of them in one launch.
inline TileChoice pick_splitk_tile(int64_t M, int64_t R, int64_t Cc, bool use_table = true, int batch = 1) {
  TileChoice c;
  c.tuned = false;
  if (use_table)
    if (const TunedPlan* t = tuned_plan(TUNED_SPLITK, M, R, Cc)) {
      c.tile = t->tile;
      c.splits = t->splits;
      c.tuned = true;
      return c;
    }
  // Large outputs: the 256x256 tile fills the chip on its own, no split needed (and the GEMM then
  // stores bf16 directly, without partials or a reduce pass).
  if (batch * 2 * cdiv64(R, 256) * cdiv64(Cc, 256) >= 2 * kCus) {
    c.tile = TILE_256x256_W8;
    c.splits = 1;
    return c;
  }
  c.tile = TILE_128x128_W4;
  const int64_t tiles = batch * 2 * cdiv64(R, 128) * cdiv64(Cc, 128);
  int64_t s = cdiv64(2 * kCus, tiles);            // aim at two workgroups per CU ...
  const int64_t slabs = cdiv64(cdiv64(M, 2), 64);  // 64-row slabs per group at an even split
  // ... with at least 16 slabs to each range: below that the partials and the reduce pass cost more than the idle CUs
  // (K = N = 1024, M = 256 ... 1024: one range is 20-30 % faster than the two to four that fill the chip)
  if (s > slabs / 16) s = slabs / 16;
  if (s > 16) s = 16;
  if (s < 1) s = 1;
  c.splits = (int)s;
  return c;
}

// Decode shapes: the streaming kernels need whole 128-element K chunks in both projections.
inline bool stream_shape_ok(int64_t M, int64_t d, int64_t h) {
  return M >= 1 && M <= kStreamMaxM && d >= 128 && h >= 128 && d % 128 == 0 && h % 128 == 0 && d % 16 == 0;
}

// Split-K factor of the streamed down-projection.  A workgroup covers `rows_per_block` weight rows
// x one K range that its `waves` wavefronts share.  Aim at about 16 wavefronts per CU and per
// modality, keep at least four 128-element chunks per wavefront, prefer a split that gives every
// wavefront the same number of chunks.  1 means no cross-workgroup split: the kernel then stores
// the output itself and no reduce pass runs.
inline int stream_down_splits(int64_t d, int64_t h, int rows_per_block, int waves) {
  const int64_t row_blocks = cdiv64(d, rows_per_block);
  const int64_t chunks = h / 128;
  int64_t s = cdiv64((int64_t)16 * kCus, row_blocks * waves);
  if (s > chunks / (4 * waves)) s = chunks / (4 * waves);
  if (s > 16) s = 16;
  if (s < 1) s = 1;
  for (int64_t c = s; c >= 1 && c * 2 > s; --c)
    if (chunks % (c * waves) == 0) return (int)c;
  return (int)s;
}

}  // namespace ffnk
