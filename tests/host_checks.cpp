// Host-side rules of the library behind C names, for tests/test_host_rules.py: they decide which kernel a call runs, and
// none of them touches a GPU.  Compiled for the host and linked with the library's objects.
#include "../ffn_kernel_amd/csrc/launch.hpp"
#include "../ffn_kernel_amd/csrc/tile_table.hpp"

using namespace ffnk;

extern "C" {

int hc_direct_ok(int64_t K, int64_t gathered_rows, int64_t lda, int64_t ldb) { return direct_ok(K, gathered_rows, lda, ldb); }

// {tile, splits, splits_more} of a single-weight GEMM whose caller has `room` bytes for partials; what a plan needs; its score.
void hc_plan(int64_t M, int64_t N, int64_t K, size_t room, int* out) {
  const RoutedPlan p = compute_model_plan(false, M, N, K, true, room);
  out[0] = p.tile; out[1] = p.splits; out[2] = p.splits_more;
}
size_t hc_plan_bytes(int64_t M, int64_t N, int64_t K, int tile, int splits, int splits_more) {
  return plan_partial_bytes({tile, splits, splits_more}, M, N, K);
}
double hc_plan_score(int64_t M, int64_t N, int64_t K, int tile, int splits, int splits_more) {
  for (const TileCost& c : kPlainCosts)
    if (c.tile == tile && routed_split_ok(K, splits) && routed_split_ok(K, splits_more) && (tile != TILE_256x256_W4 || splits == 1))
      return plan_score(c, false, M, N, K, splits, splits_more);
  return -1.0;
}

// Workgroups of a weight-gradient launch; the tile of workgroup `bid`: {group, range, row tile, column tile}, group -1: none.
int hc_dw_blocks(int tiles_r, int tiles_c, int splits) { return dw_blocks(tiles_r, tiles_c, splits); }
void hc_dw_tile(int bid, int tiles_r, int tiles_c, int splits, int n_vis, int M, int* out) {
  const DwTileCoord t = dw_tile_coord(bid, tiles_r, tiles_c, splits, n_vis, M);
  out[0] = t.grp; out[1] = t.split; out[2] = t.tile_r; out[3] = t.tile_c;
}

// Workgroups of a launch on tiles of two heights; the tile of workgroup `bid`: {group, first row, end, first column}, group -1: none.
int hc_mixed_blocks(int M, int N, int bn) { return mixed_blocks(M, N, bn); }
void hc_mixed_tile(int bid, int n_vis, int M, int N, int bn, int group, int* out) {
  bool tall;
  const TileCoord t = mixed_tile_coord(bid, n_vis, M, N, bn, group, &tall);
  const int end = t.row0 + (tall ? kTallRows : kShortRows);
  out[0] = t.grp; out[1] = t.row0; out[2] = end < t.row_end ? end : t.row_end; out[3] = t.n0;
}

int hc_mixed_time(int tall, int shrt) { return mixed_time(tall, shrt); }
void hc_mixed_choice(int n_vis, int M, int tiles_n, int* out) {
  MixedRows v, x;
  mixed_choice(n_vis, M, tiles_n, &v, &x);
  out[0] = v.tall; out[1] = v.shrt; out[2] = x.tall; out[3] = x.shrt;
}

// Tiles of a launch with taller tiles among the others: how many; tile L: {group, first row, end, first column}.
int hc_may_stretch(int M, int tiles_n, int base, int tall, int slots) { return may_stretch(M, tiles_n, {base, tall, slots}) ? 1 : 0; }
int hc_stretch_tiles(int n_vis, int M, int tiles_n, int base, int tall, int slots) {
  const Stretch s = stretch_rows(n_vis, M, tiles_n, {base, tall, slots});
  return (s.tiles_v + s.tiles_x) * tiles_n;
}
void hc_stretch_tile(int L, int n_vis, int M, int tiles_n, int base, int tall, int slots, int bn, int group, int* out) {
  const StretchShape shape{base, tall, slots};
  const Stretch s = stretch_rows(n_vis, M, tiles_n, shape);
  bool is_tall;
  const TileCoord t = stretch_tile_coord(L, s, n_vis, M, tiles_n, bn, group, shape, &is_tall);
  const int end = t.row0 + (is_tall ? tall : base);
  out[0] = t.grp; out[1] = t.row0; out[2] = end < t.row_end ? end : t.row_end; out[3] = t.n0;
}

unsigned hc_plan_slot(int dual, int64_t M, int64_t N, int64_t K) { return model_plan_slot(dual != 0, M, N, K, !dual, kAnyRoom); }

// hipError_t of a launcher for operands it refuses before it launches anything (the operands are never read).
// form: 0 linear, 1 SwiGLU, 2 down, 3 gather, 4 ... 6 the K-major forms of 0, 2 and 3, 7 and 8 the fused backward (two
// stages, ring), 9 the same with the weight gradients in place.
int hc_launch(int form, int tile, int M, int N, int K, int split_tail) {
  static uint16_t operand[8] __attribute__((aligned(16)));
  static float partials[4];
  GemmArgs g;
  g.A = operand; g.lda = K; g.B0[0] = g.B0[1] = g.B1[0] = g.B1[1] = operand; g.ldb = form >= 4 ? N : K;
  g.C = operand; g.ldc = N; g.perm = nullptr; g.counts = nullptr; g.M = M; g.N = N; g.K = K;
  g.P_tail = split_tail ? partials : nullptr;
  SplitKArgs w;
  w.A = w.B = operand; w.lda = w.ldb = 128; w.P = partials; w.counts = nullptr; w.M = M; w.R = w.Cc = 64; w.splits = 1;
  GatherDwArgs gw;
  gw.G = gw.X = operand; gw.ldg = gw.ldx = 64; gw.perm = nullptr; gw.counts = nullptr; gw.s = w;
  switch (form) {
    case 0: return launch_linear_gemm(tile, true, g, nullptr);
    case 1: return launch_up_gemm(tile, true, g, nullptr);
    case 2: return launch_down_gemm(tile, true, g, nullptr);
    case 3: return launch_gather_gemm(tile, true, g, nullptr);
    case 4: return launch_linear_gemm_kmajor(tile, g, nullptr);
    case 5: return launch_down_gemm_kmajor(tile, g, nullptr);
    case 6: return launch_gather_gemm_kmajor(tile, g, nullptr);
    case 7: return launch_fused_bwd(g, w, false, nullptr);
    case 8: return launch_fused_bwd(g, w, true, nullptr);
    default: return launch_fused_bwd_gather(g, gw, nullptr);
  }
}

}  // extern "C"
