// C ABI of libffnk (declared in include/ffnk.h): argument checks, workspace carving, path
// selection and kernel sequencing.  Nothing here allocates, frees or synchronises.
#include "../../include/ffnk.h"

#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <atomic>

#include "common.hpp"
#include "launch.hpp"
#include "tile_table.hpp"
#include "gemm_sched.hpp"

using namespace ffnk;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  snprintf(g_err, sizeof(g_err), "%s: %s", what, hipGetErrorString(e));
  return (int)e;
}

#define FFNK_HIP(expr, what)                       \
  do {                                             \
    hipError_t e__ = (expr);                       \
    if (e__ != hipSuccess) return hip_fail(e__, what); \
  } while (0)

// Row limit.  The row partition runs in one launch of at most 256 blocks (route.hip), each of which
// counts the whole mask once: 256 * M bytes of L2 / HBM reads, 4 GB and about a millisecond at 2^24 rows -
// linear in M, and small against any GEMM over that many rows.  The tile counts and workspace offsets
// derived from M stay inside 32-bit grids up to here for every N the column limit admits.
constexpr int64_t kMaxRows = (int64_t)1 << 24;
constexpr int64_t kMaxCols = (int64_t)1 << 24;

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool aligned2(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 1) == 0; }

int check_extents(int64_t M, int64_t K, int64_t N) {
  if (M < 0 || K < 0 || N < 0) return fail(FFNK_E_SHAPE, "negative extent M=%lld K=%lld N=%lld", (long long)M, (long long)K, (long long)N);
  if (M > kMaxRows) return fail(FFNK_E_SHAPE, "M=%lld exceeds %lld rows", (long long)M, (long long)kMaxRows);
  if (K > kMaxCols || N > kMaxCols) return fail(FFNK_E_SHAPE, "K=%lld or N=%lld exceeds %lld", (long long)K, (long long)N, (long long)kMaxCols);
  return FFNK_OK;
}

// Workspace regions.
struct RouteWs {
  int32_t* perm;
  int32_t* counts;
  size_t bytes;
};
size_t route_ws_bytes(int64_t M) { return ws_align((size_t)M * 4) + ws_align(8); }
RouteWs carve_route(uint8_t* ws, int64_t M) {
  RouteWs r;
  r.perm = reinterpret_cast<int32_t*>(ws);
  r.counts = reinterpret_cast<int32_t*>(ws + ws_align((size_t)M * 4));
  r.bytes = route_ws_bytes(M);
  return r;
}

// Tuner overrides, see ffnk_debug_force_tile / ffnk_debug_force_splits.
std::atomic<int> g_force_tile{-1};    // 0..4, 6, 7, 16, 17: that tile; -1: table, then rules; -2: rules only
std::atomic<int> g_force_splits{-1};  // >= 1: that split-K factor where a GEMM can be split
std::atomic<int> g_force_group_m{0};      // >= 1: M-tiles per super-group in the tile order of every routed GEMM
std::atomic<int> g_force_bwd_gather{-1};  // MaskedLinear backward: 1 = weight gradients from g and x in place, 0 = from transposes, -1 = plan

// Pseudo tile id of a measured weight-gradient plan: g and x read where they lie (gemm_dw_gather.hpp) on the 128x128 tile.
constexpr int kTileGatherDw = 5;

bool can_force(int tile) { return (tile >= 0 && tile < TILE_COUNT && tile != kTileGatherDw) || forward_only(tile); }
int forced_forward_tile() {
  const int t = g_force_tile.load(std::memory_order_relaxed);
  return can_force(t) ? t : -1;
}
// ... in every GEMM but the forward's single-weight ones, which alone have the 192- and 160-row tiles.
int forced_tile() {
  const int t = forced_forward_tile();
  return forward_only(t) ? TILE_128x256_R3 : t;
}
bool use_tuned() { return g_force_tile.load(std::memory_order_relaxed) != -2; }
// GemmArgs::group_m of a routed GEMM: the forced value, else the measured plan's, else 0 (the tile's own).
int plan_group_m(int op, int64_t M, int64_t k, int64_t n) {
  if (const int f = g_force_group_m.load(std::memory_order_relaxed); f > 0) return f;
  return use_tuned() && op != TUNED_NONE ? tuned_group_m(op, M, k, n) : 0;
}
int forced_splits() {
  const int s = g_force_splits.load(std::memory_order_relaxed);
  return (s >= 1 && s <= 16) ? s : -1;
}

int64_t padded_rows(int64_t M) { return round_up64(M, 64) + 64; }  // >= pad64(nv) + pad64(M - nv)

// The row partition a call works with: the caller's (ffnk_routing_t, made by ffnk_route for the same mask
// and M) or, without one, the workspace's own region.
struct Routing {
  const int32_t* perm;
  const int32_t* counts;
  const uint8_t* mask = nullptr;  // the call's first GEMM makes it (GemmArgs::mask)
};
// `make`: the caller's is still to be made, and left there for the calls behind this one.  `in_gemm`: the call's first GEMM can
// make a partition; a launch of its own at the head of the call does where it cannot.
int resolve_routing(const ffnk_routing_t* rt, bool make, const RouteWs& r, const uint8_t* mask, int64_t M, bool in_gemm, hipStream_t stream,
                    Routing* out) {
  int32_t *perm = r.perm, *counts = r.counts;
  if (rt != nullptr) {
    if (!rt->perm || !rt->counts) return fail(FFNK_E_NULL, "routing: perm or counts is NULL");
    perm = const_cast<int32_t*>(rt->perm);
    counts = const_cast<int32_t*>(rt->counts);
  }
  out->perm = perm;
  out->counts = counts;
  if (rt != nullptr && !make) return FFNK_OK;
  if (in_gemm) out->mask = mask;
  else FFNK_HIP(launch_route(mask, (int)M, perm, counts, stream), "route kernel");
  return FFNK_OK;
}
// Paths without a partition of their own leave the caller's all the same.
int leave_routing(const ffnk_routing_t* rt, bool make, const uint8_t* mask, int64_t M, hipStream_t stream) {
  Routing unused;
  return make ? resolve_routing(rt, true, RouteWs{}, mask, M, false, stream, &unused) : FFNK_OK;
}
// A call that leaves the partition does so whatever its other extents are.
int check_made(const ffnk_routing_t* made, const uint8_t* mask, int64_t M) {
  if (!made || !made->perm || !made->counts) return fail(FFNK_E_NULL, "made, its perm or its counts is NULL");
  return !mask && M > 0 ? fail(FFNK_E_NULL, "mask is NULL") : FFNK_OK;
}
// The first GEMM of a forward makes the partition (GemmArgs::mask): one launch, results by whole 16-byte chunks, up to one and a half
// rounds of the chip.  Every workgroup then counts the mask, 0.7 us more than it takes to read a partition (64x128 tiles at
// M = 2048, 1 us for a 256x256 tile at M = 8192), against 3 to 4 us for the launch on the device and as much again on the host:
// MaskedLinear, masks of both modalities, K = N = 1024, M = 2048 17.8 -> 14.0 us, M = 3001, K = 2056, N = 1544 38.8 -> 36.6; forward +
// backward at K = N = 1024, M = 8192 and MaskedFFN d = 4096, h = 14336, M = 300 level (the runs' spread).  Past that every tile pays:
// MaskedFFN d = 1024, h = 2048, M = 8192 (2.1 rounds) 133.7 -> 135.3, d = 4096, h = 14336, M = 1411 (2.6) 474.7 -> 475.3.
bool gemm_routes(int tile, bool direct, bool dual, int splits, int64_t M, int64_t N, const uint8_t* mask, const uint16_t* C, int64_t ldc) {
  if (!direct || M > kScanMaxRows || !aligned16(mask) || !aligned16(C) || N % 8 != 0 || ldc % 8 != 0) return false;
  const TileGeom t = tile_geom(tile == TILE_MIXED_W4 ? TILE_256x256_W4 : tile, dual);
  const int64_t tiles = (cdiv64(M, t.block_m) + 1) * cdiv64(N, t.block_n_out) * splits;
  if (is_big_tile(tile) && splits == 1 && tiles > kCus) return false;  // (a second launch for the remainder: dispatch_tile_with_tail)
  if (tile == TILE_256x256_W4 && !dual) return false;                  // (RoutedGemmCfg::SELF_ROUTED)
  const int per_cu = tile == TILE_SMALL_W4 ? 3 : tile == TILE_128x128_W4 || tile == TILE_64x128_R3 ? 2 : 1;
  return 2 * tiles <= 3 * (int64_t)kCus * per_cu;
}

struct BwdPlan {
  bool dw_k_contig;  // dW memory is [N, K] (k contiguous): R = N, Cc = K
  int64_t R, Cc;
  TileChoice tc;
  bool gather;       // weight gradients from g and x in place, where the call's operands allow it (gather_dw_ok)
  int64_t ldt;       // row stride of the transposed operands
  size_t off_wt, off_gt, off_xt, off_p, total;
};
BwdPlan plan_bwd(int64_t M, int64_t K, int64_t N, bool dw_k_contig) {
  BwdPlan p;
  p.dw_k_contig = dw_k_contig;
  p.R = dw_k_contig ? N : K;
  p.Cc = dw_k_contig ? K : N;
  p.tc = pick_splitk_tile(M, p.R, p.Cc, use_tuned());
  // A measured plan names the form (5: in place; 0 / 2 / 4: from transposes).  Where nothing was measured: the in-place
  // form saves a launch and the transposes' 4 * M * (K + N) bytes of traffic, and its two-stage loop runs the GEMM's
  // M * K * N products about 15 % slower than the tiles that read transposes; on this part the two balance near
  // K * N / (K + N) = 1600 (K = N: faster by 19 % at 1024, 15 % at 2048, slower by 9 % at 4096).
  // Up to 1024 rows the transposes are a launch that moves next to nothing, and the in-place form wins at every size
  // (by 4-8 % at K = N = 4096, 8-33 % at 8192).
  p.gather = p.tc.tuned ? p.tc.tile == kTileGatherDw : (K * N <= 1536 * (K + N) || M <= 1024);
  if (p.tc.tile == kTileGatherDw) p.tc.tile = TILE_128x128_W4;
  if (forced_tile() >= 0) {
    p.tc.tile = forced_tile();
    p.gather = false;
  }
  if (const int fg = g_force_bwd_gather.load(std::memory_order_relaxed); fg >= 0) p.gather = fg == 1;
  if (forced_splits() >= 1) p.tc.splits = forced_splits();
  p.ldt = padded_rows(M);
  size_t o = route_ws_bytes(M);
  p.off_wt = o; o += 2 * ws_align((size_t)K * N * 2);
  p.off_gt = o; o += ws_align((size_t)N * p.ldt * 2);
  p.off_xt = o; o += ws_align((size_t)K * p.ldt * 2);
  p.off_p = o;  o += ws_align((size_t)2 * p.tc.splits * K * N * 4);
  p.total = o;
  return p;
}

// T13 and DH end in 64 rows of padding: the weight-gradient GEMMs load them in whole 64-row slabs (and
// clear what lies past a group's end before using it).
constexpr int kBwdPadRows = 64;

// MaskedFFN backward workspace: route | T13 [M + 64, 2 * half], half = h or h rounded up to 64 | DH [M + 64, h] | W2^T, U2^T [h, d] | [W1^T|W3^T],
// [U1^T|U3^T] [d, 2h] | g^T, x^T [d, ldt] | H^T, dt1^T, dt3^T [h, ldt] | fp32 split-K partials.
struct FfnBwdPlan {
  BwdPlan up, dn;  // weight-gradient GEMM shapes: up = dW1/dW3 (K = d, N = h), dn = dW2 (K = h, N = d)
  int64_t ldt;
  size_t w2t_bytes;  // room at off_w2t: the W2^T / U2^T copies, or the dx GEMM's partials / split tail after them
  size_t off_t13, off_dh, off_w2t, off_w13t, off_gt, off_xt, off_ht, off_d1t, off_d3t, off_p, total;
};
// Which of the optional regions a call touches (decided from strides and alignment, the same way by the
// planner and by the backward itself): copies of the down / up weights for layouts the K-major kernels do not
// read in place, and transposes of H, dt1, dt3 when their rows do not fit 32-bit slab offsets.
struct FfnBwdPaths {
  bool w2_copy = true, w13_copy = true, acts_in_place = false, dx_direct = false;
  int64_t half = 0;  // columns from dt1 to dt3 in T13: h, or the next multiple of 64 where the up weights are read in place
};
constexpr FfnBwdPaths kFfnBwdWorstCase{};
// Tile and split of the in-place path (H, dt1, dt3 read where they lie): the three GEMMs fill the chip together, unsplit in one
// launch.  The measured plans are MaskedLinear's, of single launches.
TileChoice ffn_bwd_in_place_choice(int64_t M, int64_t d, int64_t h) {
  TileChoice tc = pick_splitk_tile(M, h, d, false, kDwBatch);
  if (forced_splits() >= 1) tc.splits = forced_splits();
  return tc;
}
// Tile and split of the dx GEMM (2h-long contraction) and the bytes of partials or split tail it wants.
RoutedPlan ffn_bwd_dx_plan(int64_t M, int64_t d, int64_t contraction, bool dx_direct, size_t room, size_t* need);
FfnBwdPlan plan_ffn_bwd(int64_t M, int64_t d, int64_t h, bool dup_k_contig, bool ddn_k_contig,
                        const FfnBwdPaths& paths = kFfnBwdWorstCase) {
  FfnBwdPlan p;
  p.up = plan_bwd(M, d, h, dup_k_contig);
  p.dn = plan_bwd(M, h, d, ddn_k_contig);
  p.ldt = padded_rows(M);
  int splits = p.up.tc.splits > p.dn.tc.splits ? p.up.tc.splits : p.dn.tc.splits;
  if (paths.acts_in_place) splits = ffn_bwd_in_place_choice(M, d, h).splits;
  const size_t w2_copies = 2 * ws_align((size_t)h * d * 2);
  // The dx GEMM's partials (or split tail) live where the copies would, as far as they fit there - the same bound
  // whether or not the copies are made, so that the dx GEMM's plan does not depend on the layout.
  size_t dx_need = 0;
  ffn_bwd_dx_plan(M, d, 2 * (paths.half > 0 ? paths.half : h), paths.dx_direct, w2_copies, &dx_need);
  p.w2t_bytes = paths.w2_copy ? w2_copies : ws_align(dx_need);
  size_t o = route_ws_bytes(M);
  p.off_t13 = o;  o += ws_align((size_t)(M + kBwdPadRows) * 2 * round_up64(h, 64) * 2);
  p.off_dh = o;   o += ws_align((size_t)(M + kBwdPadRows) * h * 2);
  p.off_w2t = o;  o += p.w2t_bytes;
  p.off_w13t = o; o += paths.w13_copy ? 2 * ws_align((size_t)d * 2 * h * 2) : 0;
  p.off_gt = o;   o += ws_align((size_t)d * p.ldt * 2);
  p.off_xt = o;   o += ws_align((size_t)d * p.ldt * 2);
  p.off_ht = o;   o += paths.acts_in_place ? 0 : ws_align((size_t)h * p.ldt * 2);
  p.off_d1t = o;  o += paths.acts_in_place ? 0 : ws_align((size_t)h * p.ldt * 2);
  p.off_d3t = o;  o += paths.acts_in_place ? 0 : ws_align((size_t)h * p.ldt * 2);
  p.off_p = o;    o += (paths.acts_in_place && splits == 1) ? 0 : ws_align((size_t)2 * splits * d * h * 4);
  p.total = o;
  return p;
}

// The K-major kernels read a weight where the backward finds it: [K, N] rows of the contraction, N
// contiguous, row stride ldb.  Slabs are addressed with 32-bit byte offsets from their first row.
bool kmajor_ok(int64_t K, int64_t N, int64_t ldb, const void* w0, const void* w1) {
  constexpr int64_t k4g = (int64_t)1 << 32;
  return direct_contraction(K) && N >= 8 && N % 8 == 0 && ldb % 8 == 0 && ldb >= N && aligned16(w0) && aligned16(w1) &&
         ldb * 128 + 2 * N < k4g;
}

// Scratch of ffnk_masked_ffn_fwd_static: one copy per GPU, held from the moment the library's code
// object is loaded there until the process ends.  The name is a host-side stand-in, not a device
// address: host code only ever uses the per-device address that static_scratch() looks up.
static __device__ __align__(256) unsigned char scratch[FFNK_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// Address of `scratch` on the GPU that holds `on_device` (the call's output): each GPU has its own copy
// of the array at its own address, and the kernels run where their operands live, which need not be the
// calling thread's current device.  Looked up once per device, with that device current (two threads that
// race here both get the same answer).
int static_scratch(const void* on_device, void** out) {
  hipPointerAttribute_t attr;
  if (hipPointerGetAttributes(&attr, on_device) != hipSuccess || attr.type != hipMemoryTypeDevice) {
    (void)hipGetLastError();  // the query's own error must not surface in a later call
    return fail(FFNK_E_NULL, "ffnk_masked_ffn_fwd_static: out is not device memory");
  }
  const int dev = attr.device;
  if (dev < 0 || dev >= kMaxDevices) return fail(FFNK_E_SHAPE, "device index %d outside [0, %d)", dev, kMaxDevices);
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    int cur = -1;
    FFNK_HIP(hipGetDevice(&cur), "hipGetDevice");
    if (cur != dev) FFNK_HIP(hipSetDevice(dev), "hipSetDevice");
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != dev) FFNK_HIP(hipSetDevice(cur), "hipSetDevice");
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (p == nullptr) return fail(FFNK_E_NULL, "static scratch has no address on device %d", dev);
    g_scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return FFNK_OK;
}

int routed_tile(int64_t M, int64_t n_out, bool dual, int64_t K = 0, int op = TUNED_PLAIN) {
  const int f = forced_tile();
  return f >= 0 ? f : pick_routed_tile(M, n_out, dual, K, use_tuned(), op);
}

// Whole extents off the dot kernels' 512-element slices at M <= 8, against the LDS-transposed streams.  Up to four rows the
// dot-product streams lead wherever there is a stream to speak of: 1410 drawn MaskedFFN calls of d * h >= 2^21 took 1.05 ... 1.7
// times as long on the others, the worst of them 0.97.  Five rows and more are eight dot products per weight, and the cut
// last slice of a short contraction weighs more.  10317 drawn MaskedLinear calls, caches flushed, time on the others over time
// here: up to 4096 weight rows 1.26 - 1.45 for K <= 4096, 0.98 - 1.24 above; more rows 0.82 - 1.03 up to K = 5120 (worst 0.60)
// and 0.99 - 1.13 above it.
constexpr int64_t kDotMinWeight = (int64_t)1 << 21, kDotManyRowsN = 4352, kDotManyRowsK = 5120;
bool whole_dot_pays(int64_t M, int64_t K, int64_t N) {
  return K * N >= kDotMinWeight && (M <= 4 || stream_dot_ok((int)M, (int)K) || N <= kDotManyRowsN || K > kDotManyRowsK);
}
bool use_stream_path(int64_t M, int64_t d, int64_t h) { return stream_shape_ok(M, d, h); }

// Kernels of the two projections of a streamed forward: fragment-layout streams (extents under 1024), contiguous-row
// dot-product streams (M <= 8), LDS-transposed MFMA streams.
enum { STREAM_FRAG, STREAM_DOT, STREAM_TILE };
struct StreamKinds { int up, down; };

StreamKinds stream_kinds_any(int64_t M, int64_t d, int64_t h) {
  return {stream_dot_any_ok((int)M, (int)d) ? STREAM_DOT : STREAM_TILE, stream_dot_any_ok((int)M, (int)h) ? STREAM_DOT : STREAM_TILE};
}
// Above 32 rows, time on the tiled GEMMs over time on the streams, geometric means over 7000 drawn shapes, caches flushed (both
// modalities / one), by K * N.  33 - 48 rows: MaskedFFN 1.06 - 1.24 / 1.15 - 1.31 up to 2^25, 1.07 - 1.13 / 0.95 - 1.08 past it;
// MaskedLinear 1.10 - 1.24 / 1.01 - 1.14 and 1.06 - 1.11 / 0.95 - 0.97.  49 - 64 rows up to 2^25: MaskedFFN 1.04 - 1.20 /
// 1.10 - 1.26, MaskedLinear 1.01 - 1.20 / 0.99 - 1.12; past it the GEMMs lead with one modality (d=5832 h=11784 M=64 133
// against 139 us, d=4160 h=12480 77 against 86).
bool ragged_stream_pays(int64_t M, int64_t K, int64_t N) { return M <= 48 || K * N <= ((int64_t)1 << 25); }

// Extents that are multiples of 8 but not of 128 run on the streams too, except in the forward that keeps its
// pre-activations (ffnk_masked_ffn_can_save).  Against the tiled GEMMs, which wait for a slab of weights per barrier and have
// few workgroups at these sizes (us, GEMM -> streams, caches flushed): one modality d=2104 h=7176 M=1 46.6 -> 25.7, d=5832
// h=11784 M=3 115 -> 81, M=8 116 -> 92, M=13 119 -> 115, linear K=2056 N=1544 M=1 14.0 -> 6.1; both modalities d=5832 h=11784
// M=3 124 -> 84, M=8 206 -> 151, M=13 208 -> 171, d=3008 h=9024 M=40 94 -> 82.
bool use_ragged_stream(int64_t M, int64_t d, int64_t h) {
  return M >= 1 && M <= kStreamMaxM && d <= kMaxCols && h <= kMaxCols && !use_stream_path(M, d, h) && forced_tile() < 0 &&
         stream_tile_any_ok((int)M, (int)d, (int)h) && ragged_stream_pays(M, d, h);
}

StreamKinds stream_kinds(int64_t M, int64_t d, int64_t h) {
  if (!use_stream_path(M, d, h)) return stream_kinds_any(M, d, h);
  if (stream_dot_ok((int)M, (int)d) && stream_dot_ok((int)M, (int)h)) return {STREAM_DOT, STREAM_DOT};
  if (!stream_tile_ok((int)M, (int)d, (int)h)) return {STREAM_FRAG, STREAM_FRAG};
  StreamKinds kinds = stream_kinds_any(M, d, h);
  if (!whole_dot_pays(M, d, h)) kinds.up = STREAM_TILE;
  if (!whole_dot_pays(M, h, d)) kinds.down = STREAM_TILE;
  return kinds;
}

int down_splits(int64_t M, int64_t d, int64_t h) {
  const int kind = stream_kinds(M, d, h).down;
  if (kind == STREAM_DOT) return 1;
  if (kind == STREAM_TILE) {
    // a forced factor (tuner) where every K range keeps the kernel's minimum of eight 128-element chunks
    const int fs = forced_splits(), chunks = (int)cdiv64(h, 128);
    if (fs >= 1 && chunks - (int)cdiv64(chunks, fs) * (fs - 1) >= 8) return fs;
    return stream_tile_down_splits((int)M, (int)d, (int)h);
  }
  return stream_down_splits(d, h, stream_rows_per_block((int)M, false), stream_waves_per_block((int)M, false));
}

// Split-K factor of the down projection on the LDS-tiled path (1: none).
// Tile and split-K factor of the down projection on the LDS-tiled path (a forced tile keeps its own
// best split).
// `op`: whose measured plans apply (TunedOp).
RoutedPlan down_plan(int64_t M, int64_t d, int64_t h, int op = TUNED_DOWN) {
  RoutedPlan p;
  if (const int f = op == TUNED_NONE ? forced_tile() : forced_forward_tile(); f >= 0) {
    p.tile = f;
    p.splits = p.splits_more = pick_routed_splits(M, d, h, p.tile);
  } else {
    p = pick_routed_plan(M, d, h, use_tuned(), op);
  }
  // a forced split-K factor: whole 64-element slabs, no empty range, what the reduce pass can address
  if (const int fs = forced_splits(); fs >= 1 && direct_contraction(h) && M < 65536 && cdiv64(cdiv64(h, 64), cdiv64(cdiv64(h, 64), fs)) == fs &&
      p.tile != TILE_256x256_W4)
    p.splits = p.splits_more = fs;
  return p;
}
// Workspace of the MaskedFFN forward without partials: the row partition and the [M, h] bf16 intermediate in routed order.
size_t ffn_fixed_bytes(int64_t M, int64_t h) { return route_ws_bytes(M) + ws_align((size_t)M * round_up64(h, 8) * 2); }
// The MaskedFFN forward's down projection: the model's plan where the caller's workspace is sized for it, the best of the plans
// that fit where it is not (the static entry point).
RoutedPlan ffn_down_plan(int64_t M, int64_t d, int64_t h, size_t ws_limit = kAnyRoom) {
  const RoutedPlan p = down_plan(M, d, h);
  const size_t fixed = ffn_fixed_bytes(M, h);
  if (forced_tile() >= 0 || forced_splits() >= 1 || fixed >= ws_limit || plan_partial_bytes(p, M, d, h) <= ws_limit - fixed) return p;
  return model_routed_plan(false, M, d, h, M < 65536 && d % 4 == 0, ws_limit - fixed);
}
// The SwiGLU GEMM's plan is the four-wave 256x256 tile, and it has up to eight rounds of the chip: that tile beside 160-row ones in
// one launch (mixed_rows), also where it is forced, so that what the tuner times is what a plan of it runs.  Past that the two
// launches of whole rounds and remainder are the faster (M = 32768, d = 4096, h = 14336, 56 rounds: 7834 us against 8002;
// M = 23225, d = 2624, h = 8512, one modality, 24 rounds: 2241 against 2281).
bool up_two_heights(int tile, bool direct, int64_t M, int64_t h) {
  return tile == TILE_256x256_W4 && direct && cdiv64(M, kTallRows) * cdiv64(h, 128) <= 8 * kCus;
}
// Tile of an unsplit GEMM of the backward: the time model's, although it was fitted to row-major weights - over 2320 drawn GEMMs
// on K-major weights (M = 65 ... 16384, up to two rounds of 256x256 tiles and past them) its plans are 1.8 % (MaskedLinear's
// dx), 2.9 % (dh) and 3.0 % (the feed-forward dx, K split) behind the best of all tiles and split factors in the geometric mean,
// the rules by tile count, which these GEMMs ran on before, 32, 23 and 17 %.
int bwd_tile(int64_t M, int64_t n_out, int64_t K, bool direct) {
  if (forced_tile() < 0 && direct && model_applies(false, M, n_out, K)) return model_routed_plan(false, M, n_out, K, false, kAnyRoom, false).tile;
  return routed_tile(M, n_out, false, 0, TUNED_NONE);
}
// dx GEMM of the MaskedFFN backward: few output tiles over a contraction of 2h (or 2 * half), so K is split like the forward's
// down projection when the fp32 partials fit `room`; an unsplit big tile wants room for its split tail instead.
RoutedPlan ffn_bwd_dx_plan(int64_t M, int64_t d, int64_t contraction, bool dx_direct, size_t room, size_t* need) {
  // No measured plans: they are timings of other kernels (the forward's down projection reads K-contiguous weights through
  // another loop).
  RoutedPlan dxp = down_plan(M, d, contraction, TUNED_NONE);
  if (forced_tile() < 0 && forced_splits() < 1 && dx_direct && model_applies(false, M, d, contraction))
    dxp = model_routed_plan(false, M, d, contraction, M < 65536, room, false);
  if (!dx_direct || (size_t)max_splits(dxp) * M * d * 4 > room) {
    dxp.splits = dxp.splits_more = 1;
    dxp.tile = routed_tile(M, d, false, 0, TUNED_NONE);
  }
  size_t n = 0;
  if (dxp.splits > 1) n = (size_t)max_splits(dxp) * M * d * 4;
  else if (dx_direct && is_big_tile(dxp.tile) && (size_t)kTailSlots * 256 * 256 * 4 <= room) n = (size_t)kTailSlots * 256 * 256 * 4;
  if (need) *need = n;
  return dxp;
}
// The dx GEMM (plan dxp) in one launch with the weight gradients, uncut: where both run on 256x256 tiles, dx's own rounds would be
// less than 0.7 full - a split tail or K ranges, and a reduce pass - and its workgroups are done in 3/4 of the time of all work
// spread over the chip (a tile costs its slabs and about eight more).  Forward + backward, apart -> beside, of 34 drawn layers those
// inside these lines: 2.2 to 5.0 % less where dx fills half a round or a little more than whole ones (d = 4184, h = 13480, M = 1995
// 2214 -> 2108 us, d = 4160, h = 9024, M = 1284 1006 -> 967, d = 5760, h = 14336, M = 2589 3462 -> 3359), none slower; M = 4096,
// d = 4096, h = 14336 3553 -> 3552.  Outside: fuller rounds up to 2.2 % more (d = 4288, h = 14208, M = 7144 6317 -> 6458), 9/10 of
// the time and more +-0.5 %; below ten slabs per weight-gradient tile those are bound by their stores and slow dx down (d = 6976,
// h = 23232, M = 471 1817 -> 2066).
bool ffn_bwd_dx_beside_dw(int64_t M, int64_t d, int64_t h, int64_t contraction, const RoutedPlan& dxp, const TileChoice& dw) {
  constexpr int64_t kFixed = 8, kDwSlabs = 10;
  if (!is_big_tile(dxp.tile) || dw.tile != TILE_256x256_W8 || dw.splits != 1 || forced_splits() > 1) return false;
  const int64_t tiles_n = cdiv64(d, 256), dx_tiles = (cdiv64(M, 256) + 1) * tiles_n, dw_tiles = 2 * kDwBatch * cdiv64(h, 256) * tiles_n;
  const int64_t slabs = contraction / 64, dw_slabs = cdiv64(M, 128), rounds = cdiv64(dx_tiles, kCus);
  return dw_slabs >= kDwSlabs && 10 * dx_tiles < 7 * rounds * kCus &&
         4 * rounds * (slabs + kFixed) * kCus <= 3 * (dx_tiles * (slabs + kFixed) + dw_tiles * (dw_slabs + kFixed));
}
// Paths of the MaskedFFN backward for one layout: which weights are read in place and which copied, and whether
// H, dt1, dt3 are read in place by the weight-gradient GEMMs.  The backward and the lean workspace query both ask
// here, so that the regions a call touches are the regions its plan holds.
FfnBwdPaths ffn_bwd_paths(int64_t M, int64_t d, int64_t h, int64_t g_stride_m, int64_t up_stride_n, int64_t down_stride_k,
                          int64_t down_stride_n, const uint16_t* W1, const uint16_t* W3, const uint16_t* U1,
                          const uint16_t* U3, const uint16_t* W2, const uint16_t* U2, bool* w2_direct_out = nullptr,
                          bool* w2_kmajor_out = nullptr, bool* w13_kmajor_out = nullptr) {
  const int64_t half = round_up64(h, 64);
  const bool w2_direct = down_stride_n == 1 && down_stride_k % 8 == 0 && down_stride_k >= d && aligned16(W2) && aligned16(U2);
  // The forward's layout ([d, h] rows, h contiguous) is K-major for the dh GEMM: read in place.
  const bool w2_kmajor = !w2_direct && down_stride_k == 1 && kmajor_ok(d, h, down_stride_n, W2, U2) &&
                         direct_ok(d, M, g_stride_m, 8);
  // The up-projection weights ([h, d] rows, d contiguous) are K-major for the dx GEMM: the contraction
  // runs through the gate weight's rows and on into the up weight's, each padded to whole slabs (GemmArgs::k_rows; T13's rows
  // are padded alike).  With copies of the four weights for h off multiples of 64, forward + backward took (us, copies -> in
  // place): d = 6744, h = 16008, M = 389 1914 -> 1226 (one modality), d = 4824, h = 10736, M = 159 909 -> 654, d = 4408, h = 13192,
  // M = 3021 3763 -> 3172, d = 1880, h = 5144, M = 1883 589 -> 511.
  const bool w13_kmajor = kmajor_ok(2 * half, d, up_stride_n, W1, W3) && aligned16(U1) && aligned16(U3) && direct_ok(2 * half, 0, 2 * half, 8);
  FfnBwdPaths paths;
  paths.w2_copy = !(w2_direct || w2_kmajor);
  paths.w13_copy = !w13_kmajor;
  paths.half = w13_kmajor ? half : h;
  const int64_t ld13 = 2 * paths.half;
  paths.acts_in_place = ld13 * 128 + 2 * h < ((int64_t)1 << 32);
  paths.dx_direct = w13_kmajor || direct_ok(2 * h, 0, ld13, ld13);
  if (w2_direct_out) *w2_direct_out = w2_direct;
  if (w2_kmajor_out) *w2_kmajor_out = w2_kmajor;
  if (w13_kmajor_out) *w13_kmajor_out = w13_kmajor;
  return paths;
}

// MaskedLinear forward at decode sizes: 0 = LDS-tiled GEMM, 1 = dot-product streams (M <= 8),
// 2 = LDS-transposed streams (M <= 64).  The op is bound by reading each weight once.
int linear_stream_kind(int64_t M, int64_t K, int64_t N) {
  if (M < 1 || M > kStreamMaxM || K > kMaxCols || N > kMaxCols) return 0;
  if (stream_dot_ok((int)M, (int)K)) return 1;
  const bool whole = stream_tile_down_ok((int)M, (int)N, (int)K);
  if (stream_dot_any_ok((int)M, (int)K) && (whole ? whole_dot_pays(M, K, N) : forced_tile() < 0)) return 1;
  if (whole) return 2;
  return forced_tile() < 0 && stream_tile_down_any_ok((int)M, (int)N, (int)K) && ragged_stream_pays(M, K, N) ? 2 : 0;
}
int linear_stream_splits(int64_t M, int64_t K, int64_t N) {
  return linear_stream_kind(M, K, N) == 2 ? stream_tile_down_splits((int)M, (int)N, (int)K) : 1;
}

// MaskedLinear forward: the table's tile unless cutting K pays (few output tiles, long contraction).
RoutedPlan linear_plan(int64_t M, int64_t K, int64_t N) {
  RoutedPlan p = down_plan(M, N, K, TUNED_PLAIN);
  if (N % 4 != 0) p.splits = p.splits_more = 1;  // the reduce pass moves four columns per thread
  return p;
}
// fp32 partials of the tiled MaskedLinear forward: split-K for the whole GEMM, or the split tail of
// the 256x256 tile.
size_t linear_partial_bytes(int64_t M, int64_t K, int64_t N) {
  return plan_partial_bytes(linear_plan(M, K, N), M, N, K);
}
// Workspace of the MaskedFFN forward with at most `ws_limit` bytes for it: partition, intermediate, and the fp32 partials of the
// down projection where it is split (the larger need where strides or saved pre-activations send a ragged shape to the GEMMs).
size_t ffn_fwd_bytes(int64_t M, int64_t d, int64_t h, size_t ws_limit = kAnyRoom) {
  const size_t fixed = ffn_fixed_bytes(M, h);
  if (use_stream_path(M, d, h)) return fixed + ws_align((size_t)down_splits(M, d, h) * M * d * 4);
  size_t part = plan_partial_bytes(ffn_down_plan(M, d, h, ws_limit), M, d, h);
  if (use_ragged_stream(M, d, h)) {
    const int s = down_splits(M, d, h);  // (a forced factor may be larger than the rule's)
    const size_t streamed = s > 1 ? ws_align((size_t)s * M * d * 4) : 0;
    if (streamed > part) part = streamed;
  }
  return fixed + part;
}

// Split-K factor of the weight-gradient GEMM when it shares a launch with the dx GEMM (both on 128x128
// tiles, two workgroups per CU).  The weight-gradient workgroups are few and long, the dx workgroups many
// and short and fill the CUs the others leave: the launch lasts as long as the longer of the two, in
// 64-row slabs of 0.8 us (a 128x128 tile's slab behind two LDS stages waits on its loads: measured).  Unsplit (no
// partials, no reduce pass, one launch fewer) unless cutting the contraction shortens the estimate by more than 35 %
// (K = N = 1024: at M = 8192, estimate 0.75, two or three ranges measure between 7 % slower and 16 % faster than one
// depending on the mask; at M = 16384, estimate 0.63, 17-26 % faster); never more ranges than the plan sized the
// partials for.
int fused_bwd_splits(int64_t M, int64_t K, int64_t N, int plan_splits) {
  const double slots = 2.0 * kCus, t_slab = 0.8;
  const double dw_tiles = 2.0 * (double)cdiv64(N, 128) * (double)cdiv64(K, 128);
  const double dx_units = (double)(cdiv64(M, 128) + 1) * (double)cdiv64(K, 128) * (double)cdiv64(N, 64);
  auto estimate = [&](int s) {
    const double dw_wgs = dw_tiles * s;
    const double dw_slabs = (double)cdiv64(cdiv64(M, 2 * 64), s) * (double)cdiv64((int64_t)dw_wgs, (int64_t)slots);
    const double rest = slots - dw_wgs > slots / 8 ? slots - dw_wgs : slots / 8;
    const double t = (dw_slabs > dx_units / rest ? dw_slabs : dx_units / rest) * t_slab;
    return s == 1 ? t : t + 4.0 + (double)s * 2.0 * (double)K * (double)N * 8.0 / 4.0e6;  // launch + partials at 4 TB/s
  };
  const double unsplit = estimate(1);
  int best = 1;
  double best_t = unsplit;
  for (int s = 2; s <= plan_splits; ++s) {
    const double t = estimate(s);
    if (t < best_t) {
      best = s;
      best_t = t;
    }
  }
  return best_t < 0.65 * unsplit ? best : 1;
}

// Whether the MaskedLinear backward runs its two GEMMs in one launch, and the split-K factor its
// weight-gradient GEMM is really launched with.  A measured plan and a forced factor are used as they are
// (that is what the tuner timed); only a factor the rules guessed goes through the fused launch's own model.
// The fused launch is one decision: it runs when the weights are readable in place and both GEMMs are on a 128x128
// tile; the weight-gradient plan (rules, measured plan or forced tile) says which of the two - two LDS stages, or
// the ring of four - and the dx GEMM follows it.
bool is_128_tile(int tile) { return tile == TILE_128x128_W4 || tile == TILE_128x128_R4; }
// The in-place weight-gradient GEMM addresses token rows with 32-bit byte offsets and moves 8-column chunks.
// (16-byte aligned in memory, so row strides are multiples of 8 as well).
bool gather_dw_ok(int64_t M, int64_t K, int64_t N, const void* g, int64_t g_stride_m, const void* x, int64_t x_stride_m) {
  constexpr int64_t k4g = (int64_t)1 << 32;
  return M > 0 && K >= 8 && N >= 8 && K % 8 == 0 && N % 8 == 0 && g_stride_m % 8 == 0 && x_stride_m % 8 == 0 &&
         M * g_stride_m * 2 + 2 * N < k4g && M * x_stride_m * 2 + 2 * K < k4g &&
         ((reinterpret_cast<uintptr_t>(g) | reinterpret_cast<uintptr_t>(x)) & 15) == 0;
}
// One launch for both GEMMs: the dx GEMM on a 128x128 tile over weights read in place, and the weight gradients on the
// same tile (the in-place form has no other).
bool bwd_is_fused(int64_t M, int64_t K, const BwdPlan& p, bool w_kmajor, bool in_place) {
  return w_kmajor && is_128_tile(routed_tile(M, K, false, 0, TUNED_NONE)) && (in_place || is_128_tile(p.tc.tile));
}
int bwd_dw_launch_splits(int64_t M, int64_t K, int64_t N, const BwdPlan& p, bool fused) {
  if (!fused || p.tc.tuned || forced_splits() >= 1) return p.tc.splits;
  return fused_bwd_splits(M, K, N, p.tc.splits);
}

// The feed-forward backward's dx and (where H, dt1 and dt3 are read in place) weight-gradient GEMMs.
struct FfnBwdGemms {
  RoutedPlan dx;
  size_t dx_need;  // bytes of partials or split tail, if dx has a launch of its own
  TileChoice dw{};
  bool beside = false;
};
FfnBwdGemms ffn_bwd_gemms(int64_t M, int64_t d, int64_t h, const FfnBwdPaths& paths, bool w13_kmajor) {
  FfnBwdGemms g;
  const int64_t contraction = 2 * paths.half;
  g.dx = ffn_bwd_dx_plan(M, d, contraction, paths.dx_direct, 2 * ws_align((size_t)h * d * 2), &g.dx_need);
  if (paths.acts_in_place) {
    g.dw = ffn_bwd_in_place_choice(M, d, h);
    if (forced_tile() >= 0) g.dw.tile = forced_tile();
    g.beside = w13_kmajor && ffn_bwd_dx_beside_dw(M, d, h, contraction, g.dx, g.dw);
  }
  return g;
}

int linear_fwd_impl(const uint16_t* x, int64_t x_stride_m, const uint16_t* Wv, const uint16_t* Wt, int64_t w_stride_k,
                    int64_t w_stride_n, const uint8_t* mask, uint16_t* y, int64_t y_stride_m, int64_t M, int64_t K, int64_t N, void* ws,
                    size_t ws_bytes, void* stream_, const ffnk_routing_t* routing, bool make) {
  hipStream_t stream = (hipStream_t)stream_;
  if (int e = check_extents(M, K, N)) return e;
  if (M == 0 || N == 0) return leave_routing(routing, make, mask, M, stream);
  if (!x && K > 0) return fail(FFNK_E_NULL, "x is NULL");
  if ((!Wv || !Wt) && K > 0) return fail(FFNK_E_NULL, "weight pointer is NULL");
  if (!mask || !y) return fail(FFNK_E_NULL, "mask or y is NULL");
  if (!aligned2(x) || !aligned2(Wv) || !aligned2(Wt) || !aligned2(y)) return fail(FFNK_E_ALIGN, "bf16 pointer not 2-byte aligned");
  if (y_stride_m < N) return fail(FFNK_E_STRIDE, "y_stride_m=%lld < N=%lld", (long long)y_stride_m, (long long)N);

  const bool fast = K > 0 && K % 8 == 0 && x_stride_m % 8 == 0 && x_stride_m >= K && aligned16(x) &&
                    w_stride_k == 1 && w_stride_n % 8 == 0 && w_stride_n >= K && aligned16(Wv) && aligned16(Wt);
  if (!fast) {
    GenericLinearArgs a;
    a.x = x; a.sxm = x_stride_m; a.sxk = 1;
    a.W[0] = Wv; a.W[1] = Wt; a.swk = w_stride_k; a.swn = w_stride_n;
    a.mask = mask; a.y = y; a.sym = y_stride_m; a.syn = 1;
    a.M = (int)M; a.K = (int)K; a.N = (int)N;
    FFNK_HIP(launch_generic_linear(a, stream), "generic linear kernel");
    return leave_routing(routing, make, mask, M, stream);
  }
  const size_t need = ffnk_workspace_bytes(FFNK_OP_LINEAR_FWD, M, K, N);
  if (ws_bytes < need || !ws) return fail(FFNK_E_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, need);
  if (!aligned16(ws)) return fail(FFNK_E_ALIGN, "workspace not 16-byte aligned");
  const RouteWs r = carve_route(static_cast<uint8_t*>(ws), M);
  const bool far_rows = M * x_stride_m >= ((int64_t)1 << 30);  // past the LDS-transposed streams' 32-bit offsets
  const int kind = linear_stream_kind(M, K, N);
  if (kind && !(kind == 2 && far_rows && !stream_tile_down_ok((int)M, (int)N, (int)K))) {
    // Decode sizes: the weight-streaming kernels of the FFN's down projection, fed token rows in
    // token order; they route from the mask themselves.
    if (kind == 2 && far_rows)
      return fail(FFNK_E_STRIDE, "x_stride_m=%lld: the decode kernels address the token rows with 32-bit offsets",
                  (long long)x_stride_m);
    const int splits = linear_stream_splits(M, K, N);
    StreamArgs a;
    a.X = x; a.ldx = x_stride_m; a.gather_x = 1; a.mask = mask; a.M = (int)M;
    a.W0[0] = Wv; a.W0[1] = Wt; a.W1[0] = a.W1[1] = nullptr; a.ldw = w_stride_n;
    a.Nrows = (int)N; a.K = (int)K; a.splits = splits; a.H = nullptr; a.ldh = 0;
    a.P = splits > 1 ? reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + r.bytes) : nullptr;
    a.out = y; a.ldo = y_stride_m;
    FFNK_HIP(kind == 1 ? launch_stream_dot_down(a, stream) : launch_stream_tile_down(a, stream), "streaming linear");
    if (splits > 1)
      FFNK_HIP(launch_stream_reduce(a.P, splits, (int)M, (int)N, mask, y, y_stride_m, stream), "streaming reduce");
    return leave_routing(routing, make, mask, M, stream);
  }
  const bool direct = direct_ok(K, M, x_stride_m, w_stride_n);
  RoutedPlan plan = linear_plan(M, K, N);
  if (!direct) {
    plan.splits = plan.splits_more = 1;
    plan.tile = routed_tile(M, N, false, K);
  }
  Routing rt;
  const bool in_gemm = gemm_routes(plan.tile, direct, false, max_splits(plan), M, N, mask, y, y_stride_m);
  if (int e = resolve_routing(routing, make, r, mask, M, in_gemm, stream, &rt)) return e;
  GemmArgs g;
  g.A = x; g.lda = x_stride_m;
  g.B0[0] = Wv; g.B0[1] = Wt; g.B1[0] = g.B1[1] = nullptr; g.ldb = w_stride_n;
  g.C = y; g.ldc = y_stride_m;
  g.perm = rt.perm; g.counts = rt.counts; g.mask = rt.mask;
  g.M = (int)M; g.N = (int)N; g.K = (int)K; g.group_m = plan_group_m(TUNED_PLAIN, M, K, N);
  if (plan.splits > 1) {
    g.splits = plan.splits;
    g.splits_more = plan.splits_more;
    g.P = reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + r.bytes);
  } else if (direct && is_big_tile(plan.tile)) {
    g.P_tail = reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + r.bytes);
  }
  FFNK_HIP(launch_linear_gemm(plan.tile, direct, g, stream), "linear GEMM");
  if (plan.splits > 1)
    FFNK_HIP(launch_routed_reduce(g.P, plan.splits, plan.splits_more, tile_geom(plan.tile, false).block_m, (int)M, (int)N, rt.counts,
                                  rt.perm, y, y_stride_m, stream), "linear reduce");
  return FFNK_OK;
}

}  // namespace

extern "C" {

int ffnk_version(void) { return FFNK_VERSION; }

int ffnk_debug_force_tile(int tile) {
  return g_force_tile.exchange(can_force(tile) || tile == -2 ? tile : -1);
}

int ffnk_debug_force_group_m(int group_m) { return g_force_group_m.exchange(group_m >= 1 && group_m <= 64 ? group_m : 0); }

int ffnk_debug_force_bwd_gather(int on) { return g_force_bwd_gather.exchange((on == 0 || on == 1) ? on : -1); }

int ffnk_debug_force_splits(int splits) { return g_force_splits.exchange((splits >= 1 && splits <= 16) ? splits : -1); }

const char* ffnk_last_error(void) { return g_err; }

int ffnk_route(const uint8_t* mask, int64_t M, int32_t* perm, int32_t* counts, void* stream) {
  if (int e = check_extents(M, 0, 0)) return e;
  if (!counts || (M > 0 && (!mask || !perm))) return fail(FFNK_E_NULL, "ffnk_route: NULL pointer");
  FFNK_HIP(launch_route(mask, (int)M, perm, counts, (hipStream_t)stream), "route kernel");
  return FFNK_OK;
}

size_t ffnk_workspace_bytes(int op, int64_t M, int64_t K, int64_t N) {
  if (M < 0 || K < 0 || N < 0 || M > kMaxRows || K > kMaxCols || N > kMaxCols) return (size_t)-1;
  switch (op) {
    case FFNK_OP_LINEAR_FWD: {
      // perm + counts + the fp32 split-K partials where the GEMM (or the streamed projection) is split
      if (linear_stream_kind(M, K, N)) {
        const int splits = linear_stream_splits(M, K, N);
        const size_t part = splits > 1 ? ws_align((size_t)splits * M * N * 4) : 0;
        // (a row stride past the streams' 32-bit offsets sends a ragged shape to the tiled GEMM)
        const size_t tiled = stream_tile_down_ok((int)M, (int)N, (int)K) ? 0 : linear_partial_bytes(M, K, N);
        return route_ws_bytes(M) + (part > tiled ? part : tiled);
      }
      return route_ws_bytes(M) + linear_partial_bytes(M, K, N);
    }
    case FFNK_OP_FFN_FWD: return ffn_fwd_bytes(M, K, N);
    case FFNK_OP_LINEAR_BWD: {
      const BwdPlan a = plan_bwd(M, K, N, true), b = plan_bwd(M, K, N, false);
      return a.total > b.total ? a.total : b.total;
    }
    case FFNK_OP_FFN_BWD: {
      size_t best = 0;
      for (int i = 0; i < 4; ++i) {
        const size_t t = plan_ffn_bwd(M, K, N, (i & 1) != 0, (i & 2) != 0).total;
        if (t > best) best = t;
      }
      return best;
    }
    default:
      return (size_t)-1;
  }
}

size_t ffnk_workspace_bytes_ffn_bwd(int64_t M, int64_t d, int64_t h, int64_t g_stride_m, int64_t up_stride_n,
                                    int64_t down_stride_k, int64_t down_stride_n, int64_t dup_stride_k,
                                    int64_t ddown_stride_k) {
  if (M < 0 || d <= 0 || h <= 0 || M > kMaxRows || d > kMaxCols || h > kMaxCols) return (size_t)-1;
  const FfnBwdPaths paths = ffn_bwd_paths(M, d, h, g_stride_m, up_stride_n, down_stride_k, down_stride_n, nullptr, nullptr,
                                          nullptr, nullptr, nullptr, nullptr);
  return plan_ffn_bwd(M, d, h, dup_stride_k == 1, ddown_stride_k == 1, paths).total;
}

int ffnk_tile_config(int op, int64_t M, int64_t K, int64_t N, ffnk_tile_config_t* out) {
  if (!out) return fail(FFNK_E_NULL, "ffnk_tile_config: out is NULL");
  if (int e = check_extents(M, K, N)) return e;
  memset(out, 0, sizeof(*out));
  int tile;
  bool dual = false;
  int64_t contraction;
  int splits = 1;
  bool in_place = false;
  switch (op) {
    case FFNK_OP_LINEAR_FWD: { const RoutedPlan lp = linear_plan(M, K, N); tile = lp.tile; splits = max_splits(lp); contraction = K; break; }
    case FFNK_OP_FFN_FWD:
    case FFNK_OP_FFN_UP: tile = routed_tile(M, N, true, K); dual = true; contraction = K; break;
    case FFNK_OP_FFN_DOWN: tile = ffn_down_plan(M, K, N).tile; contraction = N; break;  // out cols = d = K, contraction h = N
    case FFNK_OP_LINEAR_BWD:
    case FFNK_OP_BWD_DX:
    case FFNK_OP_BWD_DW: {
      // As launched for the reference's layout (nn.Linear.weight.T views, contiguous g): weights read in place.
      const BwdPlan bp = plan_bwd(M, K, N, true);
      const bool w_kmajor = K >= 8 && K % 8 == 0 && direct_ok(N, M, N, 8);
      in_place = bp.gather && gather_dw_ok(M, K, N, nullptr, N, nullptr, K);
      const bool fused = bwd_is_fused(M, K, bp, w_kmajor, in_place);
      if (op == FFNK_OP_BWD_DW) {
        tile = in_place ? TILE_128x128_W4 : bp.tc.tile; contraction = M;
        splits = bwd_dw_launch_splits(M, K, N, bp, fused);
      } else {
        tile = fused ? routed_tile(M, K, false, 0, TUNED_NONE) : bwd_tile(M, K, N, w_kmajor); contraction = N;
        in_place = false;
      }
      break;
    }
    default: return fail(FFNK_E_OP, "unknown op %d", op);
  }
  // (the weight-gradient GEMM contracts over whole slabs, padded or cleared, whatever M is)
  const bool direct = op == FFNK_OP_BWD_DW ? contraction > 0 : direct_contraction(contraction);
  // Kernels without the two ring tiles of three stages run the two-stage tiles in their place.
  const bool kmajor_dx = op == FFNK_OP_LINEAR_BWD || op == FFNK_OP_BWD_DX;
  if (!direct || op == FFNK_OP_BWD_DW) {
    if (tile == TILE_128x256_R3 || forward_only(tile)) tile = TILE_128x128_W4;
    if (tile == TILE_64x128_R3) tile = op == FFNK_OP_BWD_DW ? TILE_128x128_W4 : TILE_SMALL_W4;
  }
  if (!direct && tile == TILE_256x256_W4) tile = TILE_256x256_W8;  // the four-wave tile runs on the direct path only
  const TileGeom gm = tile_geom(tile, dual);
  const bool stream = (op == FFNK_OP_FFN_FWD || op == FFNK_OP_FFN_UP || op == FFNK_OP_FFN_DOWN) && (use_stream_path(M, K, N) || use_ragged_stream(M, K, N));
  out->path = stream ? FFNK_PATH_STREAM : FFNK_PATH_MFMA_TILED;
  out->block_m = gm.block_m;
  out->block_n = gm.block_n_out;
  out->block_k = 64;
  out->waves_m = gm.waves_m;
  out->waves_n = gm.waves_n;
  // the plan's super-group size, else the tile's own: 8 for the SwiGLU GEMM and over K-major weights (the backward's
  // dx GEMM in the usual layout), 4 for the other single-weight GEMMs
  int plan_gm = 0;
  switch (op) {
    case FFNK_OP_LINEAR_FWD: plan_gm = plan_group_m(TUNED_PLAIN, M, K, N); break;
    case FFNK_OP_FFN_FWD:
    case FFNK_OP_FFN_UP: plan_gm = plan_group_m(TUNED_DUAL, M, K, N); break;
    case FFNK_OP_FFN_DOWN: plan_gm = plan_group_m(TUNED_DOWN, M, N, K); break;
    default: plan_gm = plan_group_m(TUNED_NONE, M, K, N); break;
  }
  out->group_m = plan_gm > 0 ? plan_gm : (dual || kmajor_dx) ? 8 : 4;
  out->split_k = splits;
  out->direct_lds = (direct || in_place) ? 1 : 0;
  out->in_place = in_place ? 1 : 0;
  // 4: ring of four stages (128x128); 3: token panel in three stages, weight panel in two (single-weight 256x256 tiles)
  out->lds_stages = !(direct || in_place) ? 2 : tile == TILE_128x128_R4 ? 4 : (tile == TILE_128x256_R3 || tile == TILE_64x128_R3 || forward_only(tile)) ? 3 : (is_big_tile(tile) && !dual) ? 3 : 2;
  if (op == FFNK_OP_FFN_DOWN && !stream) out->split_k = max_splits(ffn_down_plan(M, K, N));
  if (op == FFNK_OP_LINEAR_FWD && linear_stream_kind(M, K, N)) {
    out->path = FFNK_PATH_STREAM;
    out->waves_m = out->waves_n = 1;
    out->group_m = 1;
    if (linear_stream_kind(M, K, N) == 1) {
      out->block_m = (int)M;
      out->block_n = stream_dot_rows_per_block((int)N, false, (int)K);
      out->block_k = 512 * stream_dot_slices_per_wave((int)K);
      out->split_k = stream_dot_waves((int)K);
      out->lds_stages = 0;
      out->direct_lds = 0;
    } else {
      out->block_m = 16 * (int)cdiv64(M, 16);
      out->block_n = stream_tile_rows_per_block((int)M, false);
      out->waves_n = stream_tile_waves((int)M, (int)N, (int)K, false);
      out->block_k = 128;
      out->lds_stages = stream_tile_depth((int)M, false);
      out->direct_lds = stream_tile_direct((int)M, false);
      out->split_k = linear_stream_splits(M, K, N);
    }
    return FFNK_OK;
  }
  if (stream) {
    // Streaming kernels: a workgroup is 16 * RT weight rows x one K range whose four wavefronts
    // take a quarter each; operands go global -> registers, no LDS staging.
    const bool up = op != FFNK_OP_FFN_DOWN;
    out->block_m = 16 * (int)cdiv64(M, 16);
    out->block_n = stream_rows_per_block((int)M, up);
    out->block_k = stream_chunk_k((int)M, up);
    out->waves_m = 1;
    out->waves_n = 1;
    out->lds_stages = 0;
    out->group_m = 1;
    out->split_k = stream_waves_per_block((int)M, up) * (up ? 1 : down_splits(M, K, N));
    out->direct_lds = 0;
    const StreamKinds kinds = stream_kinds(M, K, N);
    const int kind = up ? kinds.up : kinds.down;
    if (kind == STREAM_TILE) {
      // LDS-transposed streams: block_n weight rows (of each matrix) x 128-element chunks, three in flight
      out->block_n = stream_tile_rows_per_block((int)M, up);
      out->waves_n = stream_tile_waves((int)M, (int)(up ? N : K), (int)(up ? K : N), up);
      out->block_k = 128;
      out->lds_stages = stream_tile_depth((int)M, up);
      out->direct_lds = stream_tile_direct((int)M, up);
      out->split_k = up ? 1 : down_splits(M, K, N);
    }
    if (kind == STREAM_DOT) {
      // dot-product streams: a workgroup is block_n weight rows x all of K, one wavefront per
      // block_k-element slice of K
      const int64_t contr = up ? K : N;
      out->block_m = (int)M;
      out->block_n = stream_dot_rows_per_block((int)(up ? N : K), up, (int)contr);
      out->block_k = 512 * stream_dot_slices_per_wave((int)contr);
      out->split_k = stream_dot_waves((int)contr);
    }
  }
  return FFNK_OK;
}

int ffnk_debug_ffn_joint(int64_t M, int64_t d, int64_t h) {
  if (int e = check_extents(M, d, h)) return e;
  int joint = 0;
  if (!use_stream_path(M, d, h) && d % 8 == 0 && up_two_heights(routed_tile(M, h, true, d), direct_ok(d, M, d, d), M, h)) joint |= 1;
  if (M > 0 && d > 0 && h > 0 && d % 8 == 0 && h % 8 == 0) {
    bool w13_kmajor = false;
    const FfnBwdPaths paths = ffn_bwd_paths(M, d, h, d, d, 1, h, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, &w13_kmajor);
    if (ffn_bwd_gemms(M, d, h, paths, w13_kmajor).beside) joint |= 2;
  }
  return joint;
}

int ffnk_masked_linear_fwd(const uint16_t* x, int64_t x_stride_m, const uint16_t* Wv, const uint16_t* Wt,
                           int64_t w_stride_k, int64_t w_stride_n, const uint8_t* mask, uint16_t* y,
                           int64_t y_stride_m, int64_t M, int64_t K, int64_t N, void* ws, size_t ws_bytes,
                           void* stream_) {
  return ffnk_masked_linear_fwd_routed(x, x_stride_m, Wv, Wt, w_stride_k, w_stride_n, mask, y, y_stride_m, M, K, N, ws,
                                       ws_bytes, stream_, nullptr);
}

int ffnk_masked_linear_fwd_routed(const uint16_t* x, int64_t x_stride_m, const uint16_t* Wv, const uint16_t* Wt,
                                  int64_t w_stride_k, int64_t w_stride_n, const uint8_t* mask, uint16_t* y,
                                  int64_t y_stride_m, int64_t M, int64_t K, int64_t N, void* ws, size_t ws_bytes,
                                  void* stream_, const ffnk_routing_t* routing) {
  return linear_fwd_impl(x, x_stride_m, Wv, Wt, w_stride_k, w_stride_n, mask, y, y_stride_m, M, K, N, ws, ws_bytes, stream_, routing, false);
}

int ffnk_masked_linear_fwd_routing(const uint16_t* x, int64_t x_stride_m, const uint16_t* Wv, const uint16_t* Wt,
                                   int64_t w_stride_k, int64_t w_stride_n, const uint8_t* mask, uint16_t* y,
                                   int64_t y_stride_m, int64_t M, int64_t K, int64_t N, void* ws, size_t ws_bytes,
                                   void* stream_, const ffnk_routing_t* made) {
  if (int e = check_made(made, mask, M)) return e;
  return linear_fwd_impl(x, x_stride_m, Wv, Wt, w_stride_k, w_stride_n, mask, y, y_stride_m, M, K, N, ws, ws_bytes, stream_, made, true);
}

int ffnk_masked_ffn_fwd(const uint16_t* x, int64_t x_stride_m, const uint16_t* W1, const uint16_t* W3,
                        const uint16_t* U1, const uint16_t* U3, int64_t up_stride_k, int64_t up_stride_n,
                        const uint16_t* W2, const uint16_t* U2, int64_t down_stride_k, int64_t down_stride_n,
                        const uint8_t* mask, uint16_t* out, int64_t out_stride_m, int64_t M, int64_t d,
                        int64_t h, void* ws, size_t ws_bytes, void* stream_) {
  return ffnk_masked_ffn_fwd_ev(x, x_stride_m, W1, W3, U1, U3, up_stride_k, up_stride_n, W2, U2, down_stride_k,
                                down_stride_n, mask, out, out_stride_m, M, d, h, ws, ws_bytes, stream_, nullptr);
}

}  // extern "C"

namespace {

// Forward shared by the entry points.  pre != NULL: also store the two pre-activations (routed order,
// [M, 2h], gate | up) for a later ffnk_masked_ffn_bwd_saved; only the LDS-tiled path can do that.
int ffn_fwd_impl(const uint16_t* x, int64_t x_stride_m, const uint16_t* W1, const uint16_t* W3, const uint16_t* U1,
                 const uint16_t* U3, int64_t up_stride_k, int64_t up_stride_n, const uint16_t* W2, const uint16_t* U2,
                 int64_t down_stride_k, int64_t down_stride_n, const uint8_t* mask, uint16_t* out, int64_t out_stride_m,
                 uint16_t* pre, int64_t pre_stride_m, int64_t M, int64_t d, int64_t h, void* ws, size_t ws_bytes,
                 void* stream_, void* const* events, const ffnk_routing_t* routing = nullptr, size_t ws_limit = kAnyRoom, bool make = false) {
  hipStream_t stream = (hipStream_t)stream_;
  auto mark = [&](int i) -> hipError_t {
    if (events && events[i]) return hipEventRecord((hipEvent_t)events[i], stream);
    return hipSuccess;
  };
  if (int e = check_extents(M, d, h)) return e;
  if (M == 0 || d == 0) return leave_routing(routing, make, mask, M, stream);
  if (!x || !mask || !out) return fail(FFNK_E_NULL, "x, mask or out is NULL");
  if (h > 0 && (!W1 || !W3 || !U1 || !U3 || !W2 || !U2)) return fail(FFNK_E_NULL, "weight pointer is NULL");
  if (!aligned2(x) || !aligned2(out) || !aligned2(W1) || !aligned2(W3) || !aligned2(U1) || !aligned2(U3) ||
      !aligned2(W2) || !aligned2(U2))
    return fail(FFNK_E_ALIGN, "bf16 pointer not 2-byte aligned");
  if (out_stride_m < d) return fail(FFNK_E_STRIDE, "out_stride_m=%lld < d=%lld", (long long)out_stride_m, (long long)d);
  if (pre != nullptr) {
    if (!ffnk_masked_ffn_can_save(M, d, h))
      return fail(FFNK_E_STRIDE, "MaskedFFN forward: pre-activations can only be saved on the LDS-tiled path "
                                 "(ffnk_masked_ffn_can_save)");
    if (pre_stride_m < 2 * h || pre_stride_m % 8 != 0 || !aligned16(pre))
      return fail(FFNK_E_STRIDE, "pre_stride_m=%lld: need >= 2h, a multiple of 8, and 16-byte aligned rows",
                  (long long)pre_stride_m);
  }
  const size_t need = ffn_fwd_bytes(M, d, h, ws_limit);
  if (ws_bytes < need || !ws) return fail(FFNK_E_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, need);
  if (!aligned16(ws)) return fail(FFNK_E_ALIGN, "workspace not 16-byte aligned");

  uint8_t* wsb = static_cast<uint8_t*>(ws);
  const RouteWs r = carve_route(wsb, M);
  uint16_t* H = reinterpret_cast<uint16_t*>(wsb + r.bytes);
  const int64_t ldh = round_up64(h, 8);

  const bool fast = d % 8 == 0 && h > 0 && h % 8 == 0 && x_stride_m % 8 == 0 && x_stride_m >= d && aligned16(x) &&
                    up_stride_k == 1 && up_stride_n % 8 == 0 && up_stride_n >= d && down_stride_k == 1 &&
                    down_stride_n % 8 == 0 && down_stride_n >= h && aligned16(W1) && aligned16(W3) &&
                    aligned16(U1) && aligned16(U3) && aligned16(W2) && aligned16(U2);
  if (pre != nullptr && !fast)
    return fail(FFNK_E_STRIDE, "MaskedFFN forward: saving the pre-activations needs the fast layout (16-byte aligned, "
                               "K-contiguous operands)");
  if (!fast) {
    // Token-order intermediate, then the generic routed linear on it.
    GenericUpArgs u;
    u.x = x; u.sxm = x_stride_m;
    u.G[0] = W1; u.G[1] = U1; u.U[0] = W3; u.U[1] = U3; u.swk = up_stride_k; u.swn = up_stride_n;
    u.mask = mask; u.H = H; u.ldh = ldh;
    u.M = (int)M; u.K = (int)d; u.N = (int)h;
    FFNK_HIP(mark(0), "event record");
    FFNK_HIP(launch_generic_up(u, stream), "generic up kernel");
    FFNK_HIP(mark(1), "event record");
    GenericLinearArgs a;
    a.x = H; a.sxm = ldh; a.sxk = 1;
    a.W[0] = W2; a.W[1] = U2; a.swk = down_stride_k; a.swn = down_stride_n;
    a.mask = mask; a.y = out; a.sym = out_stride_m; a.syn = 1;
    a.M = (int)M; a.K = (int)h; a.N = (int)d;
    FFNK_HIP(launch_generic_linear(a, stream), "generic down kernel");
    FFNK_HIP(mark(2), "event record");
    return leave_routing(routing, make, mask, M, stream);
  }

  const bool far_rows = M * x_stride_m >= ((int64_t)1 << 30);  // past the LDS-transposed streams' 32-bit offsets
  if (use_stream_path(M, d, h) ||
      (pre == nullptr && use_ragged_stream(M, d, h) && !(far_rows && stream_kinds(M, d, h).up == STREAM_TILE))) {
    float* P = reinterpret_cast<float*>(wsb + r.bytes + ws_align((size_t)M * ldh * 2));
    const int splits = down_splits(M, d, h);
    FFNK_HIP(mark(0), "event record");
    StreamArgs u;
    u.X = x; u.ldx = x_stride_m; u.gather_x = 1; u.mask = mask; u.M = (int)M;
    u.W0[0] = W1; u.W0[1] = U1; u.W1[0] = W3; u.W1[1] = U3; u.ldw = up_stride_n;
    u.Nrows = (int)h; u.K = (int)d; u.splits = 1; u.H = H; u.ldh = ldh; u.P = nullptr; u.out = nullptr; u.ldo = 0;
    const StreamKinds kinds = stream_kinds(M, d, h);
    if (kinds.up == STREAM_TILE && far_rows)
      return fail(FFNK_E_STRIDE, "x_stride_m=%lld: the decode kernels address the token rows with 32-bit offsets",
                  (long long)x_stride_m);
    FFNK_HIP(kinds.up == STREAM_DOT ? launch_stream_dot_up(u, stream)
             : kinds.up == STREAM_TILE ? launch_stream_tile_up(u, stream) : launch_stream_up(u, stream),
             "streaming up-projection");
    FFNK_HIP(mark(1), "event record");
    StreamArgs dn;
    dn.X = H; dn.ldx = ldh; dn.gather_x = 0; dn.mask = mask; dn.M = (int)M;
    dn.W0[0] = W2; dn.W0[1] = U2; dn.W1[0] = dn.W1[1] = nullptr; dn.ldw = down_stride_n;
    dn.Nrows = (int)d; dn.K = (int)h; dn.splits = splits; dn.H = nullptr; dn.ldh = 0;
    dn.P = splits > 1 ? P : nullptr; dn.out = out; dn.ldo = out_stride_m;
    FFNK_HIP(kinds.down == STREAM_DOT ? launch_stream_dot_down(dn, stream)
             : kinds.down == STREAM_TILE ? launch_stream_tile_down(dn, stream) : launch_stream_down(dn, stream),
             "streaming down-projection");
    if (splits > 1)
      FFNK_HIP(launch_stream_reduce(P, splits, (int)M, (int)d, mask, out, out_stride_m, stream), "streaming reduce");
    FFNK_HIP(mark(2), "event record");
    return leave_routing(routing, make, mask, M, stream);
  }

  const bool up_direct = direct_ok(d, M, x_stride_m, up_stride_n);
  int up_tile = routed_tile(M, h, true, d);
  if (up_two_heights(up_tile, up_direct, M, h)) up_tile = TILE_MIXED_W4;
  Routing rt;
  const bool in_gemm = gemm_routes(up_tile, up_direct, true, 1, M, h, mask, H, ldh);
  if (int e = resolve_routing(routing, make, r, mask, M, in_gemm, stream, &rt)) return e;
  FFNK_HIP(mark(0), "event record");
  GemmArgs up;
  up.A = x; up.lda = x_stride_m;
  up.B0[0] = W1; up.B0[1] = U1; up.B1[0] = W3; up.B1[1] = U3; up.ldb = up_stride_n;
  up.C = H; up.ldc = ldh;
  up.perm = rt.perm; up.counts = rt.counts; up.mask = rt.mask;
  up.M = (int)M; up.N = (int)h; up.K = (int)d; up.group_m = plan_group_m(TUNED_DUAL, M, d, h);
  up.C_pre = pre; up.ldc_pre = pre_stride_m;
  FFNK_HIP(launch_up_gemm(up_tile, up_direct, up, stream), "up-projection GEMM");
  FFNK_HIP(mark(1), "event record");
  GemmArgs dn;
  dn.A = H; dn.lda = ldh;
  dn.B0[0] = W2; dn.B0[1] = U2; dn.B1[0] = dn.B1[1] = nullptr; dn.ldb = down_stride_n;
  dn.C = out; dn.ldc = out_stride_m;
  dn.perm = rt.perm; dn.counts = rt.counts;
  dn.M = (int)M; dn.N = (int)d; dn.K = (int)h; dn.group_m = plan_group_m(TUNED_DOWN, M, h, d);
  const bool dn_direct = direct_ok(h, 0, ldh, down_stride_n);
  RoutedPlan dn_plan = ffn_down_plan(M, d, h, ws_limit);
  if (!dn_direct) dn_plan.splits = dn_plan.splits_more = 1;
  float* partials = reinterpret_cast<float*>(wsb + r.bytes + ws_align((size_t)M * ldh * 2));
  if (dn_plan.splits > 1) {
    dn.splits = dn_plan.splits;
    dn.splits_more = dn_plan.splits_more;
    dn.P = partials;
  } else if (dn_direct && is_big_tile(dn_plan.tile)) {
    dn.P_tail = partials;  // the last, partial round of 256x256 tiles runs cut into K ranges
  }
  FFNK_HIP(launch_down_gemm(dn_plan.tile, dn_direct, dn, stream), "down-projection GEMM");
  if (dn_plan.splits > 1)
    FFNK_HIP(launch_routed_reduce(dn.P, dn_plan.splits, dn_plan.splits_more, tile_geom(dn_plan.tile, false).block_m, (int)M, (int)d,
                                  rt.counts, rt.perm, out, out_stride_m, stream), "down-projection reduce");
  FFNK_HIP(mark(2), "event record");
  return FFNK_OK;
}

}  // namespace

extern "C" {

int ffnk_masked_ffn_fwd_ev(const uint16_t* x, int64_t x_stride_m, const uint16_t* W1, const uint16_t* W3,
                           const uint16_t* U1, const uint16_t* U3, int64_t up_stride_k, int64_t up_stride_n,
                           const uint16_t* W2, const uint16_t* U2, int64_t down_stride_k, int64_t down_stride_n,
                           const uint8_t* mask, uint16_t* out, int64_t out_stride_m, int64_t M, int64_t d,
                           int64_t h, void* ws, size_t ws_bytes, void* stream_, void* const* events) {
  return ffn_fwd_impl(x, x_stride_m, W1, W3, U1, U3, up_stride_k, up_stride_n, W2, U2, down_stride_k, down_stride_n, mask,
                      out, out_stride_m, nullptr, 0, M, d, h, ws, ws_bytes, stream_, events);
}

int ffnk_masked_ffn_fwd_static(const uint16_t* x, int64_t x_stride_m, const uint16_t* W1, const uint16_t* W3,
                               const uint16_t* U1, const uint16_t* U3, int64_t up_stride_k, int64_t up_stride_n,
                               const uint16_t* W2, const uint16_t* U2, int64_t down_stride_k, int64_t down_stride_n,
                               const uint8_t* mask, uint16_t* out, int64_t out_stride_m, int64_t M, int64_t d,
                               int64_t h, void* stream_) {
  if (int e = check_extents(M, d, h)) return e;
  const size_t need = ffn_fwd_bytes(M, d, h, FFNK_STATIC_SCRATCH_BYTES);
  if (need > (size_t)FFNK_STATIC_SCRATCH_BYTES)
    return fail(FFNK_E_WORKSPACE, "ffnk_masked_ffn_fwd_static: M=%lld d=%lld h=%lld needs %zu bytes of scratch, the static "
                                  "buffer holds %zu; use ffnk_masked_ffn_fwd with a workspace",
                (long long)M, (long long)d, (long long)h, need, (size_t)FFNK_STATIC_SCRATCH_BYTES);
  if (M == 0 || d == 0) return FFNK_OK;
  if (!out) return fail(FFNK_E_NULL, "x, mask or out is NULL");
  void* ws = nullptr;
  if (int e = static_scratch(out, &ws)) return e;
  // Nothing in the scratch has to start at zero: every region the forward reads (perm, counts, the
  // intermediate, the fp32 partials) is written by an earlier kernel of the same call.
  return ffn_fwd_impl(x, x_stride_m, W1, W3, U1, U3, up_stride_k, up_stride_n, W2, U2, down_stride_k, down_stride_n, mask,
                      out, out_stride_m, nullptr, 0, M, d, h, ws, (size_t)FFNK_STATIC_SCRATCH_BYTES, stream_, nullptr, nullptr, FFNK_STATIC_SCRATCH_BYTES);
}

int ffnk_masked_ffn_fwd_routed(const uint16_t* x, int64_t x_stride_m, const uint16_t* W1, const uint16_t* W3,
                               const uint16_t* U1, const uint16_t* U3, int64_t up_stride_k, int64_t up_stride_n,
                               const uint16_t* W2, const uint16_t* U2, int64_t down_stride_k, int64_t down_stride_n,
                               const uint8_t* mask, uint16_t* out, int64_t out_stride_m, uint16_t* pre,
                               int64_t pre_stride_m, int64_t M, int64_t d, int64_t h, void* ws, size_t ws_bytes,
                               void* stream_, const ffnk_routing_t* routing) {
  return ffn_fwd_impl(x, x_stride_m, W1, W3, U1, U3, up_stride_k, up_stride_n, W2, U2, down_stride_k, down_stride_n, mask,
                      out, out_stride_m, pre, pre_stride_m, M, d, h, ws, ws_bytes, stream_, nullptr, routing);
}

int ffnk_masked_ffn_fwd_routing(const uint16_t* x, int64_t x_stride_m, const uint16_t* W1, const uint16_t* W3,
                               const uint16_t* U1, const uint16_t* U3, int64_t up_stride_k, int64_t up_stride_n,
                               const uint16_t* W2, const uint16_t* U2, int64_t down_stride_k, int64_t down_stride_n,
                               const uint8_t* mask, uint16_t* out, int64_t out_stride_m, uint16_t* pre,
                               int64_t pre_stride_m, int64_t M, int64_t d, int64_t h, void* ws, size_t ws_bytes,
                               void* stream_, const ffnk_routing_t* made) {
  if (int e = check_made(made, mask, M)) return e;
  return ffn_fwd_impl(x, x_stride_m, W1, W3, U1, U3, up_stride_k, up_stride_n, W2, U2, down_stride_k, down_stride_n, mask,
                      out, out_stride_m, pre, pre_stride_m, M, d, h, ws, ws_bytes, stream_, nullptr, made, kAnyRoom, true);
}

int ffnk_masked_ffn_can_save(int64_t M, int64_t d, int64_t h) {
  return (M > 0 && d > 0 && h > 0 && d % 8 == 0 && h % 8 == 0 && !use_stream_path(M, d, h)) ? 1 : 0;
}

int ffnk_masked_ffn_fwd_save(const uint16_t* x, int64_t x_stride_m, const uint16_t* W1, const uint16_t* W3,
                             const uint16_t* U1, const uint16_t* U3, int64_t up_stride_k, int64_t up_stride_n,
                             const uint16_t* W2, const uint16_t* U2, int64_t down_stride_k, int64_t down_stride_n,
                             const uint8_t* mask, uint16_t* out, int64_t out_stride_m, uint16_t* pre,
                             int64_t pre_stride_m, int64_t M, int64_t d, int64_t h, void* ws, size_t ws_bytes,
                             void* stream_) {
  if (!pre) return fail(FFNK_E_NULL, "pre is NULL");
  return ffn_fwd_impl(x, x_stride_m, W1, W3, U1, U3, up_stride_k, up_stride_n, W2, U2, down_stride_k, down_stride_n, mask,
                      out, out_stride_m, pre, pre_stride_m, M, d, h, ws, ws_bytes, stream_, nullptr);
}

int ffnk_masked_linear_bwd(const uint16_t* g, int64_t g_stride_m, const uint16_t* x, int64_t x_stride_m,
                           const uint16_t* Wv, const uint16_t* Wt, int64_t w_stride_k, int64_t w_stride_n,
                           const uint8_t* mask, uint16_t* dx, int64_t dx_stride_m, uint16_t* dWv, uint16_t* dWt,
                           int64_t dw_stride_k, int64_t dw_stride_n, int64_t M, int64_t K, int64_t N, void* ws,
                           size_t ws_bytes, void* stream_) {
  return ffnk_masked_linear_bwd_routed(g, g_stride_m, x, x_stride_m, Wv, Wt, w_stride_k, w_stride_n, mask, dx, dx_stride_m,
                                       dWv, dWt, dw_stride_k, dw_stride_n, M, K, N, ws, ws_bytes, stream_, nullptr);
}

int ffnk_masked_linear_bwd_routed(const uint16_t* g, int64_t g_stride_m, const uint16_t* x, int64_t x_stride_m,
                                  const uint16_t* Wv, const uint16_t* Wt, int64_t w_stride_k, int64_t w_stride_n,
                                  const uint8_t* mask, uint16_t* dx, int64_t dx_stride_m, uint16_t* dWv, uint16_t* dWt,
                                  int64_t dw_stride_k, int64_t dw_stride_n, int64_t M, int64_t K, int64_t N, void* ws,
                                  size_t ws_bytes, void* stream_, const ffnk_routing_t* routing) {
  hipStream_t stream = (hipStream_t)stream_;
  if (int e = check_extents(M, K, N)) return e;
  if (K == 0) return FFNK_OK;  // dx and dW are empty
  if (M > 0 && (!mask || !dx || !x)) return fail(FFNK_E_NULL, "mask, x or dx is NULL");
  if (M > 0 && N > 0 && (!g || !Wv || !Wt)) return fail(FFNK_E_NULL, "g or weight pointer is NULL");
  if (N > 0 && (!dWv || !dWt)) return fail(FFNK_E_NULL, "dW pointer is NULL");
  if (!aligned2(g) || !aligned2(x) || !aligned2(Wv) || !aligned2(Wt) || !aligned2(dx) || !aligned2(dWv) || !aligned2(dWt))
    return fail(FFNK_E_ALIGN, "bf16 pointer not 2-byte aligned");
  if (dx_stride_m < K) return fail(FFNK_E_STRIDE, "dx_stride_m=%lld < K=%lld", (long long)dx_stride_m, (long long)K);

  const bool fast = M > 0 && N > 0 && K % 8 == 0 && N % 8 == 0 && g_stride_m % 8 == 0 && g_stride_m >= N &&
                    x_stride_m % 8 == 0 && x_stride_m >= K && aligned16(g) && aligned16(x) &&
                    direct_ok(64, 0, padded_rows(M), padded_rows(M));  // transposed operands have M-long rows
  if (!fast) {
    GenericBwdArgs a;
    a.g = g; a.sgm = g_stride_m; a.x = x; a.sxm = x_stride_m;
    a.W[0] = Wv; a.W[1] = Wt; a.swk = w_stride_k; a.swn = w_stride_n;
    a.mask = mask; a.dx = dx; a.sdxm = dx_stride_m;
    a.dW[0] = dWv; a.dW[1] = dWt; a.sdk = dw_stride_k; a.sdn = dw_stride_n;
    a.M = (int)M; a.K = (int)K; a.N = (int)N;
    FFNK_HIP(launch_generic_bwd(a, stream), "generic backward kernels");
    return FFNK_OK;
  }

  const BwdPlan p = plan_bwd(M, K, N, dw_stride_k == 1);
  if (ws_bytes < p.total || !ws) return fail(FFNK_E_WORKSPACE, "workspace %zu < %zu bytes", ws_bytes, p.total);
  if (!aligned16(ws)) return fail(FFNK_E_ALIGN, "workspace not 16-byte aligned");
  uint8_t* wsb = static_cast<uint8_t*>(ws);
  const RouteWs r = carve_route(wsb, M);
  Routing rt;
  if (int e = resolve_routing(routing, false, r, mask, M, false, stream, &rt)) return e;

  // ---- dx = gather(g) @ W_g^T, contraction over N: needs the weights as [K, N] rows, N contiguous ----
  const uint16_t* wt[2] = {Wv, Wt};
  int64_t ldw = w_stride_k;
  const bool w_direct = w_stride_n == 1 && w_stride_k % 8 == 0 && w_stride_k >= N && aligned16(Wv) && aligned16(Wt);
  // The forward's layout ([N, K] rows, K contiguous) is K-major for this GEMM: no copy either.
  const bool w_kmajor = !w_direct && w_stride_k == 1 && kmajor_ok(N, K, w_stride_n, Wv, Wt) && direct_ok(N, M, g_stride_m, 8);
  if (w_kmajor) {
    ldw = w_stride_n;
  } else if (!w_direct) {
    uint16_t* c0 = reinterpret_cast<uint16_t*>(wsb + p.off_wt);
    uint16_t* c1 = reinterpret_cast<uint16_t*>(wsb + p.off_wt + ws_align((size_t)K * N * 2));
    FFNK_HIP(launch_strided_copy2d(Wv, w_stride_k, w_stride_n, c0, N, (int)K, (int)N, stream), "weight transpose");
    FFNK_HIP(launch_strided_copy2d(Wt, w_stride_k, w_stride_n, c1, N, (int)K, (int)N, stream), "weight transpose");
    wt[0] = c0; wt[1] = c1; ldw = N;
  }
  GemmArgs a;
  a.A = g; a.lda = g_stride_m;
  a.B0[0] = wt[0]; a.B0[1] = wt[1]; a.B1[0] = a.B1[1] = nullptr; a.ldb = ldw;
  a.C = dx; a.ldc = dx_stride_m;
  a.perm = rt.perm; a.counts = rt.counts;
  a.M = (int)M; a.N = (int)K; a.K = (int)N; a.group_m = plan_group_m(TUNED_NONE, M, N, K);
  const bool dx_direct = w_kmajor || direct_ok(N, M, g_stride_m, ldw);
  // Both GEMMs on the 128x128 tile and the weights readable in place: one launch runs the two side by
  // side (after the transposes it depends on), see below.
  const bool gather = p.gather && gather_dw_ok(M, K, N, g, g_stride_m, x, x_stride_m);
  const bool fused = bwd_is_fused(M, K, p, w_kmajor, gather);
  if (!fused) {
    const int dx_tile = bwd_tile(M, K, N, dx_direct);
    if (w_kmajor) FFNK_HIP(launch_linear_gemm_kmajor(dx_tile, a, stream), "dx GEMM");
    else FFNK_HIP(launch_linear_gemm(dx_tile, dx_direct, a, stream), "dx GEMM");
  }

  // ---- dW_g = x_g^T g_g, contraction over the rows of group g ----
  float* P = reinterpret_cast<float*>(wsb + p.off_p);
  SplitKArgs s;
  s.P = P; s.counts = rt.counts; s.M = (int)M;
  s.R = (int)p.R; s.Cc = (int)p.Cc; s.splits = p.tc.splits;
  const int64_t sr = p.dw_k_contig ? dw_stride_n : dw_stride_k;
  const int64_t sc = p.dw_k_contig ? dw_stride_k : dw_stride_n;
  s.splits = bwd_dw_launch_splits(M, K, N, p, fused);
  if (s.splits == 1) { s.out[0] = dWv; s.out[1] = dWt; s.out_sr = sr; s.out_sc = sc; }
  if (gather) {
    // g and x read where they lie: the row operand of the output is g when dW's memory is [N, K], x otherwise
    GatherDwArgs gw;
    gw.G = p.dw_k_contig ? g : x; gw.ldg = p.dw_k_contig ? g_stride_m : x_stride_m;
    gw.X = p.dw_k_contig ? x : g; gw.ldx = p.dw_k_contig ? x_stride_m : g_stride_m;
    gw.perm = rt.perm; gw.counts = rt.counts;
    s.A = s.B = nullptr; s.lda = s.ldb = 0;
    gw.s = s;
    if (fused) FFNK_HIP(launch_fused_bwd_gather(a, gw, stream), "fused dx / dW GEMM");
    else FFNK_HIP(launch_gathered_dw(gw, stream), "dW GEMM");
  } else {
    uint16_t* GT = reinterpret_cast<uint16_t*>(wsb + p.off_gt);  // [N, ldt]
    uint16_t* XT = reinterpret_cast<uint16_t*>(wsb + p.off_xt);  // [K, ldt]
    FFNK_HIP(launch_gather_transpose2(g, g_stride_m, (int)N, GT, x, x_stride_m, (int)K, XT, p.ldt, rt.perm, rt.counts,
                                      (int)M, stream), "g / x transpose");
    s.A = p.dw_k_contig ? GT : XT; s.lda = p.ldt;
    s.B = p.dw_k_contig ? XT : GT; s.ldb = p.ldt;
    if (fused) FFNK_HIP(launch_fused_bwd(a, s, p.tc.tile == TILE_128x128_R4, stream), "fused dx / dW GEMM");
    else FFNK_HIP(launch_splitk_gemm(p.tc.tile, s, stream), "dW split-K GEMM");
  }
  if (s.splits > 1)
    FFNK_HIP(launch_splitk_reduce(P, s.splits, (int)p.R, (int)p.Cc, dWv, dWt, sr, sc, stream), "dW reduce");
  return FFNK_OK;
}

}  // extern "C"

namespace {

// Backward shared by the entry points.  pre != NULL: the pre-activations a forward saved
// (ffnk_masked_ffn_fwd_save, same mask), read-only; NULL: recompute them with two routed GEMMs.
int ffn_bwd_impl(const uint16_t* g, int64_t g_stride_m, const uint16_t* x, int64_t x_stride_m, const uint16_t* W1,
                 const uint16_t* W3, const uint16_t* U1, const uint16_t* U3, int64_t up_stride_k, int64_t up_stride_n,
                 const uint16_t* W2, const uint16_t* U2, int64_t down_stride_k, int64_t down_stride_n,
                 const uint8_t* mask, const uint16_t* pre, int64_t pre_stride_m, uint16_t* dx, int64_t dx_stride_m,
                 uint16_t* dW1, uint16_t* dW3, uint16_t* dU1, uint16_t* dU3, int64_t dup_stride_k, int64_t dup_stride_n,
                 uint16_t* dW2, uint16_t* dU2, int64_t ddown_stride_k, int64_t ddown_stride_n, int64_t M, int64_t d,
                 int64_t h, void* ws, size_t ws_bytes, void* stream_, const ffnk_routing_t* routing = nullptr) {
  hipStream_t stream = (hipStream_t)stream_;
  if (pre != nullptr && (pre_stride_m < 2 * h || pre_stride_m % 8 != 0 || !aligned16(pre)))
    return fail(FFNK_E_STRIDE, "pre_stride_m=%lld: need >= 2h, a multiple of 8, and 16-byte aligned rows",
                (long long)pre_stride_m);
  if (int e = check_extents(M, d, h)) return e;
  if (d == 0 || h == 0) return fail(FFNK_E_SHAPE, "MaskedFFN backward needs d > 0 and h > 0");
  if (!W1 || !W3 || !U1 || !U3 || !W2 || !U2 || !dW1 || !dW3 || !dU1 || !dU3 || !dW2 || !dU2)
    return fail(FFNK_E_NULL, "weight or weight-gradient pointer is NULL");
  if (M > 0 && (!g || !x || !mask || !dx)) return fail(FFNK_E_NULL, "g, x, mask or dx is NULL");
  if (dx_stride_m < d) return fail(FFNK_E_STRIDE, "dx_stride_m=%lld < d=%lld", (long long)dx_stride_m, (long long)d);
  const bool ok = d % 8 == 0 && h % 8 == 0 && g_stride_m % 8 == 0 && g_stride_m >= d && x_stride_m % 8 == 0 &&
                  x_stride_m >= d && (M == 0 || (aligned16(g) && aligned16(x))) && up_stride_k == 1 &&
                  up_stride_n % 8 == 0 && up_stride_n >= d && aligned16(W1) && aligned16(W3) && aligned16(U1) &&
                  aligned16(U3) && aligned2(W2) && aligned2(U2) && aligned2(dx) && aligned2(dW1) && aligned2(dW3) &&
                  aligned2(dU1) && aligned2(dU3) && aligned2(dW2) && aligned2(dU2) &&
                  direct_ok(64, 0, padded_rows(M), padded_rows(M));
  if (!ok)
    return fail(FFNK_E_STRIDE, "MaskedFFN backward: d, h and the row strides must be multiples of 8, rows 16-byte "
                               "aligned and the up-projection weights K-contiguous (up_stride_k == 1)");
  // Which optional regions this layout needs (ffnk_workspace_bytes_ffn_bwd asks the same function).
  bool w2_direct = false, w2_kmajor = false, w13_kmajor = false;
  const FfnBwdPaths paths = ffn_bwd_paths(M, d, h, g_stride_m, up_stride_n, down_stride_k, down_stride_n, W1, W3, U1, U3, W2,
                                          U2, &w2_direct, &w2_kmajor, &w13_kmajor);
  const int64_t half = paths.half, ld13 = 2 * half;
  const FfnBwdPlan p = plan_ffn_bwd(M, d, h, dup_stride_k == 1, ddown_stride_k == 1, paths);
  if (ws_bytes < p.total || !ws)
    return fail(FFNK_E_WORKSPACE, "workspace %zu < %zu bytes (ffnk_workspace_bytes_ffn_bwd sizes it for aligned pointers; "
                                  "ffnk_workspace_bytes(FFNK_OP_FFN_BWD) for any layout)", ws_bytes, p.total);
  if (!aligned16(ws)) return fail(FFNK_E_ALIGN, "workspace not 16-byte aligned");
  uint8_t* wsb = static_cast<uint8_t*>(ws);
  const RouteWs r = carve_route(wsb, M);
  uint16_t* T13 = reinterpret_cast<uint16_t*>(wsb + p.off_t13);
  uint16_t* DH = reinterpret_cast<uint16_t*>(wsb + p.off_dh);
  Routing rt;
  if (int e = resolve_routing(routing, false, r, mask, M, false, stream, &rt)) return e;

  // ---- pre-activations, routed order: T13[:, 0:h] = x A1, T13[:, half:half + h] = x A3 ----
  GemmArgs a;
  a.A = x; a.lda = x_stride_m;
  a.B1[0] = a.B1[1] = nullptr; a.ldb = up_stride_n;
  a.ldc = ld13; a.perm = rt.perm; a.counts = rt.counts;
  a.M = (int)M; a.N = (int)h; a.K = (int)d; a.group_m = plan_group_m(TUNED_NONE, M, d, h);
  const bool up_direct = direct_ok(d, M, x_stride_m, up_stride_n);
  if (pre == nullptr) {
    a.B0[0] = W1; a.B0[1] = U1; a.C = T13;
    FFNK_HIP(launch_gather_gemm(routed_tile(M, h, false), up_direct, a, stream), "t1 GEMM");
    a.B0[0] = W3; a.B0[1] = U3; a.C = T13 + half;
    FFNK_HIP(launch_gather_gemm(routed_tile(M, h, false), up_direct, a, stream), "t3 GEMM");
  }

  // ---- dh = gather(g) @ A2^T, and on its tiles T13 <- (dt1 | dt3), DH <- the SwiGLU intermediate: contraction over d needs the
  // down weights as [h, d] rows ----
  const uint16_t* w2t[2] = {W2, U2};
  int64_t ld2 = down_stride_k;
  if (w2_kmajor) {
    ld2 = down_stride_n;
  } else if (!w2_direct) {
    uint16_t* c0 = reinterpret_cast<uint16_t*>(wsb + p.off_w2t);
    uint16_t* c1 = reinterpret_cast<uint16_t*>(wsb + p.off_w2t + ws_align((size_t)h * d * 2));
    FFNK_HIP(launch_strided_copy2d(W2, down_stride_k, down_stride_n, c0, d, (int)h, (int)d, stream), "weight transpose");
    FFNK_HIP(launch_strided_copy2d(U2, down_stride_k, down_stride_n, c1, d, (int)h, (int)d, stream), "weight transpose");
    w2t[0] = c0; w2t[1] = c1; ld2 = d;
  }
  a.A = g; a.lda = g_stride_m; a.B0[0] = w2t[0]; a.B0[1] = w2t[1]; a.ldb = ld2;
  a.C = DH; a.ldc = h;
  a.pre = pre ? pre : T13; a.ld_pre = pre ? pre_stride_m : ld13; a.half_pre = (int)(pre ? h : half);
  a.T13 = T13; a.ld13 = ld13; a.half = (int)half;
  const bool dh_direct = w2_kmajor || direct_ok(d, M, g_stride_m, ld2);
  const int dh_tile = bwd_tile(M, h, d, dh_direct);
  if (w2_kmajor) FFNK_HIP(launch_gather_gemm_kmajor(dh_tile, a, stream), "dh GEMM");
  else FFNK_HIP(launch_gather_gemm(dh_tile, dh_direct, a, stream), "dh GEMM");

  // ---- dx = (dt1 | dt3) @ (A1^T | A3^T)^T: one GEMM over the concatenated contraction ----
  // In place over the K-major up-projection weights, or over one [d, 2h] copy per modality.
  GemmArgs b;
  b.A = T13; b.lda = ld13;
  if (w13_kmajor) {
    b.B0[0] = W1; b.B0[1] = U1; b.B1[0] = W3; b.B1[1] = U3; b.ldb = up_stride_n;
    b.k_switch = (int)half;
    b.k_rows = (int)h;
  } else {
    uint16_t* w13[2] = {reinterpret_cast<uint16_t*>(wsb + p.off_w13t),
                        reinterpret_cast<uint16_t*>(wsb + p.off_w13t + ws_align((size_t)d * 2 * h * 2))};
    FFNK_HIP(launch_strided_copy2d(W1, up_stride_k, up_stride_n, w13[0], ld13, (int)d, (int)h, stream), "weight transpose");
    FFNK_HIP(launch_strided_copy2d(W3, up_stride_k, up_stride_n, w13[0] + h, ld13, (int)d, (int)h, stream), "weight transpose");
    FFNK_HIP(launch_strided_copy2d(U1, up_stride_k, up_stride_n, w13[1], ld13, (int)d, (int)h, stream), "weight transpose");
    FFNK_HIP(launch_strided_copy2d(U3, up_stride_k, up_stride_n, w13[1] + h, ld13, (int)d, (int)h, stream), "weight transpose");
    b.B0[0] = w13[0]; b.B0[1] = w13[1]; b.B1[0] = b.B1[1] = nullptr; b.ldb = ld13;
  }
  b.C = dx; b.ldc = dx_stride_m; b.perm = rt.perm; b.counts = rt.counts;
  b.M = (int)M; b.N = (int)d; b.K = (int)ld13; b.group_m = plan_group_m(TUNED_NONE, M, ld13, d);
  // Few output tiles over a 2h-long contraction: split K like the forward's down projection.  The
  // fp32 partials live where the W2^T copies were (dead since the dh GEMM), if they fit there.
  const bool dx_direct = paths.dx_direct;
  const FfnBwdGemms gemms = ffn_bwd_gemms(M, d, h, paths, w13_kmajor);
  const RoutedPlan& dxp = gemms.dx;
  const size_t dx_need = gemms.dx_need;
  if (dx_need > p.w2t_bytes) return fail(FFNK_E_WORKSPACE, "internal: dx partials %zu > %zu planned", dx_need, p.w2t_bytes);
  if (!gemms.beside) {
    if (dxp.splits > 1) {
      b.splits = dxp.splits;
      b.splits_more = dxp.splits_more;
      b.P = reinterpret_cast<float*>(wsb + p.off_w2t);
    } else if (dx_need > 0) {
      b.P_tail = reinterpret_cast<float*>(wsb + p.off_w2t);  // split tail of the last, partial round
    }
    if (w13_kmajor) FFNK_HIP(launch_down_gemm_kmajor(dxp.tile, b, stream), "dx GEMM");
    else FFNK_HIP(launch_down_gemm(dxp.tile, dx_direct, b, stream), "dx GEMM");
    if (dxp.splits > 1)
      FFNK_HIP(launch_routed_reduce(b.P, dxp.splits, dxp.splits_more, tile_geom(dxp.tile, false).block_m, (int)M, (int)d, rt.counts, rt.perm,
                                    dx, dx_stride_m, stream), "dx reduce");
  }

  // ---- weight gradients: contraction over the rows of each group.  x and g are gathered into
  // 64-padded transposes; H, dt1 and dt3 (routed order already) are read in place by the K-major
  // kernels, or transposed as well when their row strides do not fit 32-bit slab offsets. ----
  uint16_t* GT = reinterpret_cast<uint16_t*>(wsb + p.off_gt);    // [d, ldt]
  uint16_t* XT = reinterpret_cast<uint16_t*>(wsb + p.off_xt);    // [d, ldt]
  float* P = reinterpret_cast<float*>(wsb + p.off_p);
  const bool in_place = paths.acts_in_place;
  if (in_place) {
    FFNK_HIP(launch_gather_transpose2(g, g_stride_m, (int)d, GT, x, x_stride_m, (int)d, XT, p.ldt, rt.perm, rt.counts, (int)M,
                                      stream, false, false), "g / x transpose");
    const TileChoice& tc = gemms.dw;
    // out[r * sr + c * sc]: r runs over h (the in-place operand's columns), c over d
    auto weight_grad = [&](const uint16_t* rows, int64_t ld_rows, const uint16_t* cT, uint16_t* o0, uint16_t* o1, int64_t sr, int64_t sc) {
      SplitKArgs s;
      s.A = rows; s.lda = ld_rows;
      s.B = cT; s.ldb = p.ldt;
      s.P = P; s.counts = rt.counts; s.M = (int)M;
      s.R = (int)h; s.Cc = (int)d; s.splits = tc.splits;
      s.out[0] = o0; s.out[1] = o1; s.out_sr = sr; s.out_sc = sc;
      return s;
    };
    const SplitKArgs dw[kDwBatch] = {weight_grad(DH, h, GT, dW2, dU2, ddown_stride_k, ddown_stride_n),
                                     weight_grad(T13, ld13, XT, dW1, dU1, dup_stride_n, dup_stride_k),
                                     weight_grad(T13 + half, ld13, XT, dW3, dU3, dup_stride_n, dup_stride_k)};
    if (gemms.beside) {
      FFNK_HIP(launch_dx_dw_batch_kmajor(b, dw, stream), "dx / dW GEMMs");
      return FFNK_OK;
    }
    if (tc.splits == 1) {
      FFNK_HIP(launch_dw_batch_kmajor(tc.tile, dw, stream), "dW GEMMs");
      return FFNK_OK;
    }
    for (SplitKArgs s : dw) {
      uint16_t *o0 = s.out[0], *o1 = s.out[1];
      s.out[0] = s.out[1] = nullptr;
      FFNK_HIP(launch_splitk_gemm_kmajor(tc.tile, s, stream), "dW split-K GEMM");
      FFNK_HIP(launch_splitk_reduce(P, tc.splits, (int)h, (int)d, o0, o1, s.out_sr, s.out_sc, stream), "dW reduce");
    }
    return FFNK_OK;
  }
  uint16_t* HT = reinterpret_cast<uint16_t*>(wsb + p.off_ht);    // [h, ldt]
  uint16_t* D1T = reinterpret_cast<uint16_t*>(wsb + p.off_d1t);  // [h, ldt]
  uint16_t* D3T = reinterpret_cast<uint16_t*>(wsb + p.off_d3t);  // [h, ldt]
  FFNK_HIP(launch_gather_transpose2(g, g_stride_m, (int)d, GT, DH, h, (int)h, HT, p.ldt, rt.perm, rt.counts, (int)M,
                                    stream, false, true), "g / intermediate transpose");
  FFNK_HIP(launch_gather_transpose2(x, x_stride_m, (int)d, XT, T13, ld13, (int)h, D1T, p.ldt, rt.perm, rt.counts,
                                    (int)M, stream, false, true), "x / dt1 transpose");
  FFNK_HIP(launch_gather_transpose2(T13 + half, ld13, (int)h, D3T, nullptr, 0, 0, nullptr, p.ldt, rt.perm, rt.counts,
                                    (int)M, stream, true, false), "dt3 transpose");
  auto weight_grad = [&](const BwdPlan& q, const uint16_t* gT, const uint16_t* xT, uint16_t* o0, uint16_t* o1,
                         int64_t sk, int64_t sn) -> int {
    SplitKArgs s;
    s.A = q.dw_k_contig ? gT : xT; s.lda = p.ldt;
    s.B = q.dw_k_contig ? xT : gT; s.ldb = p.ldt;
    s.P = P; s.counts = rt.counts; s.M = (int)M;
    s.R = (int)q.R; s.Cc = (int)q.Cc; s.splits = q.tc.splits;
    const int64_t sr = q.dw_k_contig ? sn : sk, sc = q.dw_k_contig ? sk : sn;
    if (q.tc.splits == 1) { s.out[0] = o0; s.out[1] = o1; s.out_sr = sr; s.out_sc = sc; }
    FFNK_HIP(launch_splitk_gemm(q.tc.tile, s, stream), "dW split-K GEMM");
    if (q.tc.splits > 1)
      FFNK_HIP(launch_splitk_reduce(P, q.tc.splits, (int)q.R, (int)q.Cc, o0, o1, sr, sc, stream), "dW reduce");
    return FFNK_OK;
  };
  if (int e = weight_grad(p.dn, GT, HT, dW2, dU2, ddown_stride_k, ddown_stride_n)) return e;
  if (int e = weight_grad(p.up, D1T, XT, dW1, dU1, dup_stride_k, dup_stride_n)) return e;
  if (int e = weight_grad(p.up, D3T, XT, dW3, dU3, dup_stride_k, dup_stride_n)) return e;
  return FFNK_OK;
}

}  // namespace

extern "C" {

int ffnk_masked_ffn_bwd(const uint16_t* g, int64_t g_stride_m, const uint16_t* x, int64_t x_stride_m,
                        const uint16_t* W1, const uint16_t* W3, const uint16_t* U1, const uint16_t* U3,
                        int64_t up_stride_k, int64_t up_stride_n, const uint16_t* W2, const uint16_t* U2,
                        int64_t down_stride_k, int64_t down_stride_n, const uint8_t* mask, uint16_t* dx,
                        int64_t dx_stride_m, uint16_t* dW1, uint16_t* dW3, uint16_t* dU1, uint16_t* dU3,
                        int64_t dup_stride_k, int64_t dup_stride_n, uint16_t* dW2, uint16_t* dU2,
                        int64_t ddown_stride_k, int64_t ddown_stride_n, int64_t M, int64_t d, int64_t h, void* ws,
                        size_t ws_bytes, void* stream_) {
  return ffn_bwd_impl(g, g_stride_m, x, x_stride_m, W1, W3, U1, U3, up_stride_k, up_stride_n, W2, U2, down_stride_k,
                      down_stride_n, mask, nullptr, 0, dx, dx_stride_m, dW1, dW3, dU1, dU3, dup_stride_k, dup_stride_n,
                      dW2, dU2, ddown_stride_k, ddown_stride_n, M, d, h, ws, ws_bytes, stream_);
}

int ffnk_masked_ffn_bwd_routed(const uint16_t* g, int64_t g_stride_m, const uint16_t* x, int64_t x_stride_m,
                               const uint16_t* W1, const uint16_t* W3, const uint16_t* U1, const uint16_t* U3,
                               int64_t up_stride_k, int64_t up_stride_n, const uint16_t* W2, const uint16_t* U2,
                               int64_t down_stride_k, int64_t down_stride_n, const uint8_t* mask, const uint16_t* pre,
                               int64_t pre_stride_m, uint16_t* dx, int64_t dx_stride_m, uint16_t* dW1, uint16_t* dW3,
                               uint16_t* dU1, uint16_t* dU3, int64_t dup_stride_k, int64_t dup_stride_n, uint16_t* dW2,
                               uint16_t* dU2, int64_t ddown_stride_k, int64_t ddown_stride_n, int64_t M, int64_t d,
                               int64_t h, void* ws, size_t ws_bytes, void* stream_, const ffnk_routing_t* routing) {
  return ffn_bwd_impl(g, g_stride_m, x, x_stride_m, W1, W3, U1, U3, up_stride_k, up_stride_n, W2, U2, down_stride_k,
                      down_stride_n, mask, pre, pre_stride_m, dx, dx_stride_m, dW1, dW3, dU1, dU3, dup_stride_k,
                      dup_stride_n, dW2, dU2, ddown_stride_k, ddown_stride_n, M, d, h, ws, ws_bytes, stream_, routing);
}

int ffnk_masked_ffn_bwd_saved(const uint16_t* g, int64_t g_stride_m, const uint16_t* x, int64_t x_stride_m,
                              const uint16_t* W1, const uint16_t* W3, const uint16_t* U1, const uint16_t* U3,
                              int64_t up_stride_k, int64_t up_stride_n, const uint16_t* W2, const uint16_t* U2,
                              int64_t down_stride_k, int64_t down_stride_n, const uint8_t* mask, const uint16_t* pre,
                              int64_t pre_stride_m, uint16_t* dx, int64_t dx_stride_m, uint16_t* dW1, uint16_t* dW3,
                              uint16_t* dU1, uint16_t* dU3, int64_t dup_stride_k, int64_t dup_stride_n, uint16_t* dW2,
                              uint16_t* dU2, int64_t ddown_stride_k, int64_t ddown_stride_n, int64_t M, int64_t d,
                              int64_t h, void* ws, size_t ws_bytes, void* stream_) {
  if (M > 0 && !pre) return fail(FFNK_E_NULL, "pre is NULL");
  return ffn_bwd_impl(g, g_stride_m, x, x_stride_m, W1, W3, U1, U3, up_stride_k, up_stride_n, W2, U2, down_stride_k,
                      down_stride_n, mask, pre, pre_stride_m, dx, dx_stride_m, dW1, dW3, dU1, dU3, dup_stride_k,
                      dup_stride_n, dW2, dU2, ddown_stride_k, ddown_stride_n, M, d, h, ws, ws_bytes, stream_);
}

}  // extern "C"
