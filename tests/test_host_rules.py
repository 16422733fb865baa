"""The rules that choose a kernel for a call, and the launchers' own checks, run on the host without a GPU."""
import ctypes
import random
import shutil
import subprocess
from pathlib import Path

import pytest

from ffn_kernel_amd import build

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="session")
def rules(tmp_path_factory):
    objs = sorted(build.OBJ_DIR.glob("*.o"))
    if len(objs) != len(list(build.CSRC.glob("*.hip"))):
        build.build_library(verbose=False)
        objs = sorted(build.OBJ_DIR.glob("*.o"))
    so = tmp_path_factory.mktemp("host") / "host_checks.so"
    cmd = [shutil.which("hipcc") or "/opt/rocm/bin/hipcc", "--offload-host-only", "-x", "hip", "-std=c++17", "-O1", "-fPIC", "-c",
           str(HERE / "host_checks.cpp"), "-o", str(so.with_suffix(".o"))]
    subprocess.run(cmd, check=True, capture_output=True)
    subprocess.run(["g++", "-shared", "-o", str(so), str(so.with_suffix(".o")), *map(str, objs), "-L/opt/rocm/lib", "-lamdhip64"],
                   check=True, capture_output=True)
    lib = ctypes.CDLL(str(so))
    lib.hc_direct_ok.argtypes = [ctypes.c_int64] * 4
    lib.hc_plan_slot.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3
    lib.hc_plan.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_size_t, ctypes.POINTER(ctypes.c_int)]
    lib.hc_plan_bytes.argtypes = lib.hc_plan_score.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int] * 3
    lib.hc_plan_bytes.restype, lib.hc_plan_score.restype = ctypes.c_size_t, ctypes.c_double
    return lib


def _last_byte(M, K, lda):
    """End of the furthest 16-byte load of the gathered operand, from the base the direct kernels use (gemm_nt.hpp: the base
    is -K mod 64 elements ahead; a lane's offset is its row and piece, a slab's the scalar offset)."""
    slabs = -(-K // 64)
    return (M - 1) * lda * 2 + 7 * 16 + (slabs - 1) * 128 + 16


# K = 149640: 56 elements past the last whole slab but one; M * K = 2^31 - 8.  Rows as packed, and further apart.
@pytest.mark.parametrize("M,K,lda", [(14351, 149640, 149640), (14351, 149632, 149632), (1 << 20, 2040, 2040), ((1 << 20) + 4096, 2040, 2040),
                                     (131071, 4104, 16384), (65536, 32760, 32760), (65544, 32760, 32760)])
def test_direct_offsets_fit_32_bits(rules, M, K, lda):
    if rules.hc_direct_ok(K, M, lda, K):
        assert _last_byte(M, K, lda) <= (1 << 32) - 1
    assert rules.hc_direct_ok(K, M // 2, lda, K)  # well inside: the direct path


INVALID_VALUE = 1  # hipErrorInvalidValue


@pytest.fixture
def refused(rules):
    """Launcher calls that must be refused; on a machine with a GPU they are not tried."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("a launcher that let the call through would launch it")
    return lambda *a: rules.hc_launch(*a) == INVALID_VALUE


# A split tail exists for single-weight tiles that scatter their rows: with its workspace set, the others would leave half of
# the tiles past the last whole round to a launch that does not come.
@pytest.mark.parametrize("form", [1, 3, 6])
@pytest.mark.parametrize("tile", [0, 1])
def test_split_tail_is_refused_where_there_is_none(refused, form, tile):
    assert refused(form, tile, 20 * 256, 20 * 256, 64, 1)


# Under one slab the direct kernels' first load would pass the rows' ends: only whole slabs and 64 elements or more.
@pytest.mark.parametrize("K", [-64, 0, 8, 48, 56, 68, 130])
def test_direct_launchers_refuse_short_contractions(refused, K):
    for form in range(10):
        for tile in (0, 1, 2, 3, 4, 6, 7) if form < 7 else (2,):
            assert refused(form, tile, 64, 64, K, 0), (form, tile)


# Row counts at which the plan on the left took 1.2 ... 1.5 times as long as the rules' plan on the right (weights cold; us as
# measured): unsplit 64x128 tiles of long contractions, 256-row tiles whose count passes a round for some masks.
@pytest.mark.parametrize("dual,M,K,N,slow,us,rules_us", [
    (False, 403, 11392, 4544, (7, 1), 127, 84), (False, 2127, 1216, 7104, (0, 1), 78, 52), (False, 466, 10112, 3968, (7, 1), 110, 75),
    (False, 3448, 6208, 520, (3, 1), 57, 43), (False, 1571, 5376, 2472, (3, 1), 81, 62), (False, 333, 9344, 3456, (7, 1), 64, 49),
    (False, 81, 3648, 4608, (7, 1), 30, 23), (False, 1247, 7040, 3264, (6, 1), 95, 76),
    (True, 1059, 1248, 3256, (6, 1), 47, 31), (True, 791, 1088, 2240, (4, 1), 27, 19), (True, 88, 2552, 8232, (6, 1), 69, 48),
    (True, 335, 4256, 9120, (1, 1), 109, 77), (True, 730, 1440, 4904, (1, 1), 52, 38)])
def test_plans_measured_slow_are_not_chosen(dual, M, K, N, slow, us, rules_us):
    from ffn_kernel_amd import _lib, tune
    cfg = _lib.tile_config(_lib.OP_FFN_UP if dual else _lib.OP_LINEAR_FWD, M, K, N)
    assert (tune._tile_id(cfg, dual), cfg["split_k"]) != slow


# Whole extents off the dot kernels' 512-element slices: up to four rows the dot-product streams, above that where the weight
# rows are few or the contraction is long (others took up to 1.6 times as long on them).
@pytest.mark.parametrize("M,d,h,up_dot,down_dot", [(4, 2176, 7296, True, True), (5, 2176, 7296, False, True), (8, 5120 - 128, 8320, False, True),
                                                   (8, 5120 + 128, 8320, True, True), (8, 1152, 2176, True, True), (8, 1152, 4864, False, True),
                                                   (8, 1024, 22528, True, False)])
def test_dot_streams_where_they_lead(M, d, h, up_dot, down_dot):
    from ffn_kernel_amd import _lib
    for op, dot in ((_lib.OP_FFN_UP, up_dot), (_lib.OP_FFN_DOWN, down_dot)):
        cfg = _lib.tile_config(op, M, d, h)
        assert cfg["path"] == _lib.PATH_STREAM and (cfg["block_m"] == M) == dot
    lin = _lib.tile_config(_lib.OP_LINEAR_FWD, M, d, h)
    assert lin["path"] == _lib.PATH_STREAM and (lin["block_m"] == M) == up_dot


# Ragged extents above 32 rows: streams up to 48 rows whatever the weights, up to 2^25 elements of them at 49 ... 64.
@pytest.mark.parametrize("M,K,N,stream", [(33, 5832, 11784, True), (48, 5832, 11784, True), (49, 5832, 11784, False), (64, 5832, 11784, False),
                                          (64, 4104, 8168, True), (48, 8168, 8168, True), (49, 8168, 8168, False)])
def test_ragged_streams_where_they_lead(M, K, N, stream):
    from ffn_kernel_amd import _lib
    for op in (_lib.OP_LINEAR_FWD, _lib.OP_FFN_UP, _lib.OP_FFN_DOWN):
        assert (_lib.tile_config(op, M, K, N)["path"] == _lib.PATH_STREAM) == stream


# The down projection of a MaskedFFN forward whose best plan does not fit the static scratch beside the intermediate, over whole
# slabs and off them: that plan on a caller's workspace, the best of those that fit on the scratch.  (M=724: taken before.)
@pytest.mark.parametrize("M,d,h", [(397, 6584, 22040), (1189, 3144, 10576), (1016, 1968, 6288), (724, 3584, 7488), (800, 4096, 14336), (301, 8192, 28672)])
def test_down_projection_plan_within_the_static_scratch(rules, M, d, h):
    from ffn_kernel_amd import _lib, tune
    fixed = _lib.workspace_bytes(_lib.OP_LINEAR_FWD, M, 72, 4) + -(-M * h * 2 // 256) * 256  # partition (a GEMM without partials) and intermediate
    room = _lib.STATIC_SCRATCH_BYTES - fixed
    plan = (ctypes.c_int * 3)()
    rules.hc_plan(M, d, h, ctypes.c_size_t(-1).value, plan)
    cfg = _lib.tile_config(_lib.OP_FFN_DOWN, M, d, h)
    assert (tune._tile_id(cfg, False), cfg["split_k"]) == (plan[0], max(plan[1:]))
    assert _lib.workspace_bytes(_lib.OP_FFN_FWD, M, d, h) == fixed + rules.hc_plan_bytes(M, d, h, *plan) > _lib.STATIC_SCRATCH_BYTES
    rules.hc_plan(M, d, h, room, plan)
    assert rules.hc_plan_bytes(M, d, h, *plan) <= room
    score = rules.hc_plan_score(M, d, h, *plan)
    for tile in tune.TILES:
        for s in range(1, 17):
            for more in ({1} if s == 1 else range(2, 17)):
                other = rules.hc_plan_score(M, d, h, tile, s, more)
                if other > 0 and rules.hc_plan_bytes(M, d, h, tile, s, more) <= room:
                    assert score <= other * 1.03 ** 5


@pytest.mark.parametrize("M,d,h,taken", [(397, 6584, 22040, True), (724, 3584, 7488, True), (414, 4480, 13824, True), (256, 4096, 14336, True),
                                         (1170, 4096, 14336, True), (1171, 4096, 14336, False), (32768, 4096, 14336, False)])
def test_static_entry_point_takes_what_leaves_room_for_the_intermediate(M, d, h, taken):
    """The size check comes before any pointer is looked at: FFNK_E_WORKSPACE, or FFNK_E_NULL for the missing output."""
    from ffn_kernel_amd import _lib
    rc = _lib.load().ffnk_masked_ffn_fwd_static(0, d, 0, 0, 0, 0, 1, d, 0, 0, 1, h, 0, 0, d, M, d, h, 0)
    assert rc == (-1 if taken else -5)


def test_plans_of_a_model_keep_their_own_slots(rules):
    """The projections of a layer at one row count: eight keys thrown into 32 slots meet seven of them on average."""
    gen = random.Random(7)
    distinct = []
    for _ in range(500):
        M, widths = gen.randrange(65, 8192), [64 * gen.randrange(8, 256) for _ in range(4)]
        keys = {(gen.random() < 0.25, gen.choice(widths), gen.choice(widths)) for _ in range(8)}
        distinct.append(len({rules.hc_plan_slot(int(d), M, n, k) for d, n, k in keys}) / len(keys))
    assert sum(distinct) / len(distinct) > 0.85


# Weight-gradient launches: fewer tiles than XCDs, ragged super-groups, several K ranges; either group the larger one.
@pytest.mark.parametrize("tiles_r,tiles_c,splits", [(1, 1, 1), (3, 2, 1), (9, 5, 1), (8, 8, 3), (17, 6, 2)])
@pytest.mark.parametrize("n_vis,M", [(0, 70), (70, 70), (30, 70), (35, 70)])
def test_weight_gradient_order(rules, tiles_r, tiles_c, splits, n_vis, M):
    """Every tile of both groups once; every XCD an equal share of each group, the larger group first."""
    t = (ctypes.c_int * 4)()
    seen, per_xcd = [], {}
    for b in range(rules.hc_dw_blocks(tiles_r, tiles_c, splits)):
        rules.hc_dw_tile(b, tiles_r, tiles_c, splits, n_vis, M, t)
        if t[0] >= 0:
            seen.append(tuple(t))
            per_xcd.setdefault(b % 8, []).append(t[0])
    assert sorted(seen) == sorted((g, s, r, c) for g in (0, 1) for s in range(splits) for r in range(tiles_r) for c in range(tiles_c))
    larger = 0 if 2 * n_vis >= M else 1
    share = -(-tiles_r * tiles_c * splits // 8)
    for groups in per_xcd.values():
        assert groups.count(0) == groups.count(1) <= share
        assert groups == sorted(groups, key=lambda g: g != larger)


# Rows of a modality at the edges of what tall and short tiles hold, either modality absent; columns that make less than a round
# of tiles, just past one (the rest as halves), several.
@pytest.mark.parametrize("n_vis", [0, 1, 159, 160, 161, 256, 257, 320, 321, 416, 576, 577, 672, 835, 1500, 2060, 4700])
@pytest.mark.parametrize("n_text", [0, 160, 262, 480, 1025])
def test_tiles_of_two_heights_cover_every_row(rules, n_vis, n_text):
    """Every row of either modality in one tile of every column, no tile astride the modalities."""
    M, bn = n_vis + n_text, 128
    t = (ctypes.c_int * 4)()
    for tiles_n in (5, 43, 90, 129, 258) if M else ():
        covered = {}
        for b in range(rules.hc_mixed_blocks(M, tiles_n * bn - 120, bn)):
            rules.hc_mixed_tile(b, n_vis, M, tiles_n * bn - 120, bn, 8, t)
            grp, row0, end, n0 = t
            if grp == -1:
                continue
            assert grp == (0 if row0 < n_vis else 1) and row0 < end <= (n_vis if grp == 0 else M)
            covered.setdefault(n0, []).append((row0, end))
        assert sorted(covered) == list(range(0, tiles_n * bn, bn))
        for tiles in covered.values():
            tiles.sort()
            assert tiles[0][0] == 0 and tiles[-1][1] == M and all(a[1] == b[0] for a, b in zip(tiles, tiles[1:]))


@pytest.mark.parametrize("group", [1, 2, 3, 8, 64])
@pytest.mark.parametrize("n_vis,M", [(0, 2560), (1285, 4000)])
def test_tiles_of_two_heights_in_super_groups(rules, group, n_vis, M):
    """Every tile once whatever the super-group size, and an XCD's whole tall tiles of a modality at most that many to a column."""
    bn, N, t = 128, 29 * 128, (ctypes.c_int * 4)()
    tiles, longest, per_xcd = set(), 0, {}
    for b in range(rules.hc_mixed_blocks(M, N, bn)):
        rules.hc_mixed_tile(b, n_vis, M, N, bn, group, t)
        if t[0] >= 0:
            assert tuple(t) not in tiles
            tiles.add(tuple(t))
            if t[2] - t[1] > 160:
                per_xcd.setdefault(b % 8, []).append((t[0], t[3]))
    assert sum((end - row0) * min(bn, N - n0) for _, row0, end, n0 in tiles) == M * N
    for order in per_xcd.values():
        run = 1
        for prev, cur in zip(order, order[1:]):
            run = run + 1 if cur == prev else 1
            longest = max(longest, run)
    assert min(group, 4) <= longest <= group


# The four-wave 256x256 tile of the SwiGLU GEMM, planned or forced (as the tuner times it): beside 160-row tiles up to eight rounds.
@pytest.mark.parametrize("tile,M,d,h,joint", [(-1, 300, 4096, 14336, 1), (-1, 32768, 4096, 14336, 0), (1, 300, 136, 264, 1), (0, 300, 4096, 14336, 0),
                                              (1, 4096, 64, 16384, 1), (1, 4097, 64, 16384, 0), (1, 300, 72, 264, 0)])
def test_where_tiles_of_two_heights_run(tile, M, d, h, joint):
    from ffn_kernel_amd import _lib
    lib = _lib.load()
    lib.ffnk_debug_force_tile(tile)
    try:
        assert lib.ffnk_debug_ffn_joint(M, d, h) & 1 == joint
    finally:
        lib.ffnk_debug_force_tile(-1)


# The feed-forward backward's dx beside the weight gradients (tile 0 forced: both on 256x256 tiles), either side of each line: ten
# slabs per weight-gradient tile, 0.7 of dx's rounds filled, 3/4 of the time of all work; not in K ranges, not on other tiles, and
# the layers that the lines were drawn by.
@pytest.mark.parametrize("tile,splits,M,d,h,joint", [
    (0, -1, 1152, 7424, 4096, 0), (0, -1, 1153, 7424, 4096, 2), (0, -1, 2560, 4096, 1024, 2), (0, -1, 2561, 4096, 1024, 0),
    (0, -1, 2304, 3072, 4096, 0), (0, -1, 2305, 3072, 4096, 2), (0, 2, 2500, 4096, 1024, 0), (2, -1, 2500, 4096, 1024, 0),
    (-1, -1, 4096, 4096, 14336, 2), (-1, -1, 1995, 4184, 13480, 2), (-1, -1, 7144, 4288, 14208, 0), (-1, -1, 471, 6976, 23232, 0)])
def test_where_dx_runs_beside_the_weight_gradients(tile, splits, M, d, h, joint):
    from ffn_kernel_amd import _lib
    lib = _lib.load()
    lib.ffnk_debug_force_tile(tile)
    lib.ffnk_debug_force_splits(splits)
    try:
        assert lib.ffnk_debug_ffn_joint(M, d, h) & 2 == joint
    finally:
        lib.ffnk_debug_force_tile(-1)
        lib.ffnk_debug_force_splits(-1)


def test_the_swiglu_derivative_divides(tmp_path):
    """The sigmoid of the feed-forward backward is a correctly rounded division, as it was in a pass of its own: one for each of the
    eight values, none left to the bare reciprocal (v_rcp_f32, one ulp)."""
    src = tmp_path / "derivative.hip"
    src.write_text(f'#include "{build.CSRC}/common.hpp"\n'
                   "__global__ void derivative(const uint4* in, uint4* out) {\n"
                   "  ffnk::swiglu_bwd(in[0], in[1], in[2], out, out + 1, out + 2);\n}\n")
    asm = subprocess.run([shutil.which("hipcc") or "/opt/rocm/bin/hipcc", *build.HIPCC_FLAGS, "--cuda-device-only", "-S", str(src), "-o", "-"],
                         check=True, capture_output=True, text=True).stdout
    assert [asm.count(i) for i in ("v_rcp_f32", "v_div_fmas_f32", "v_div_fixup_f32")] == [8, 8, 8]


# 192- and 160-row tiles where one more M-tile, at a few splits of the rows, is a second round: the tiles that were there before.
@pytest.mark.parametrize("M,K,N", [(1936, 3584, 6400), (2320, 3584, 5376), (2145, 2688, 5504), (396, 5128, 6984)])
def test_no_second_round_at_some_splits_of_the_rows(rules, M, K, N):
    out = (ctypes.c_int * 3)()
    rules.hc_plan(M, N, K, 2 ** 64 - 1, out)
    assert out[0] not in (16, 17)


# The heights are chosen as if tiles past whole rounds were cut in two wherever they are cut (176 of a tall tile's 256).
def test_quarters_are_priced_as_halves(rules):
    assert {rules.hc_mixed_time(256 + rest, 0) for rest in range(1, 129)} == {256 + 176}


# The cases that a lower price moved to tiles of one height: two heights again (tall, short M-tiles of either modality).
@pytest.mark.parametrize("M,n_vis,h,heights", [(1024, 518, 14336, (1, 2, 2, 0)), (4339, 2231, 7296, (9, 0, 7, 2)), (3172, 1610, 7104, (6, 1, 5, 2))])
def test_two_heights_where_they_are_faster(rules, M, n_vis, h, heights):
    out = (ctypes.c_int * 4)()
    rules.hc_mixed_choice(n_vis, M, -(-h // 128), out)
    assert tuple(out) == heights


# Taller tiles among the others of a launch: every result in one tile, no more tiles than without, whole rounds where one
# M-tile less makes them, and no stretch that the host's launch does not allow for.
@pytest.mark.parametrize("base,tall", [(128, 192), (160, 192), (192, 224)])
@pytest.mark.parametrize("tiles_n,slots,tiles_m", [(8, 512, 64), (8, 256, 32), (32, 256, 8), (64, 512, 8), (20, 256, 12), (3, 512, 170), (128, 256, 4), (256, 256, 1)])
def test_stretched_tiles_cover_the_output(rules, base, tall, tiles_n, slots, tiles_m):
    t = (ctypes.c_int * 4)()
    stretched, whole = 0, tiles_m * base
    for M in (whole, whole - 1, whole + 1, whole + 60, whole + 65, whole - base + 1):
        splits = {0, 1, M, M - 1, M // 2, 64, 65, base - 1, base, base + 1, tall, tall + 1, M - 64, M - tall}
        splits |= {M // 2 + i for i in (-70, -64, 1, 31, 32, 33, 60, 63, 64, 65, base - 1)}
        for n_vis in sorted(v for v in splits if 0 <= v <= M):
            plain = (-(-n_vis // base) + -(-(M - n_vis) // base)) * tiles_n
            count = rules.hc_stretch_tiles(n_vis, M, tiles_n, base, tall, slots)
            assert count in (plain, plain - tiles_n)
            if count < plain:
                stretched += 1
                assert rules.hc_may_stretch(M, tiles_n, base, tall, slots) and plain // slots > (count - 1) // slots
            rows = {}
            for L in range(count):
                rules.hc_stretch_tile(L, n_vis, M, tiles_n, base, tall, slots, 128, 4, t)
                assert 0 <= t[1] < t[2] <= (n_vis if t[0] == 0 else M) and (t[0] == 0 or t[1] >= n_vis)
                rows.setdefault(t[3], []).append((t[1], t[2]))
            assert sorted(rows) == [n * 128 for n in range(tiles_n)]
            for spans in rows.values():
                spans.sort()
                assert spans[0][0] == 0 and spans[-1][1] == M and all(a[1] == b[0] for a, b in zip(spans, spans[1:]))
    assert stretched > 0 or tiles_n > slots // 8
