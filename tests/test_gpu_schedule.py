"""Tile orders and launch splits of the GEMMs, at the sizes where they can go wrong, against the row-select form in
double precision computed with torch on the GPU."""
import pytest
import torch

from ffn_kernel_amd import MaskedFFN, MaskedLinear, _lib
from ffn_kernel_amd.ops import masked_ffn_backward, masked_ffn_forward, masked_linear_backward
from helpers import assert_close, assert_close_pipeline, note
from oracle import modules as om

pytestmark = pytest.mark.gpu


def make_linear(dev, nv, nt, K, N, seed):
    """x, [N, K] weights, a shuffled mask with nv visual and nt text rows, and an upstream gradient."""
    gen = torch.Generator(device=dev).manual_seed(seed)
    M = nv + nt
    mask = (torch.arange(M, device=dev) < nv)[torch.randperm(M, generator=gen, device=dev)]
    rnd = lambda r, c, std: (torch.randn(r, c, generator=gen, device=dev) * std).to(torch.bfloat16)
    return rnd(M, K, 1.0), rnd(N, K, 0.05), rnd(N, K, 0.05), mask, rnd(M, N, 1.0)


@pytest.fixture
def forced():
    """Forced tile / split for one test; back to the table afterwards."""
    lib = _lib.load()

    def force(tile=-1, splits=-1):
        lib.ffnk_debug_force_tile(tile)
        lib.ffnk_debug_force_splits(splits)
    try:
        yield force
    finally:
        lib.ffnk_debug_force_tile(-1)
        lib.ffnk_debug_force_splits(-1)


# M-tiles (of 256 rows) per modality around the edges of the even super-groups: one super-group, one of each modality, two
# uneven ones, one modality absent, the last count that is dealt evenly (12 = 3 * 4) and the first that is not.
@pytest.mark.parametrize("tiles_v,tiles_t", [(1, 0), (0, 6), (3, 3), (7, 2), (0, 7), (9, 3), (6, 7), (12, 13)])
def test_super_groups_cover_every_tile(dev, forced, tiles_v, tiles_t):
    nv, nt = max(0, tiles_v * 256 - 100), max(0, tiles_t * 256 - 7)
    note(f"super-groups: {nv} visual, {nt} text rows")
    x, Wv, Wt, mask, _ = make_linear(dev, nv, nt, 64, 520, seed=tiles_v * 32 + tiles_t)
    forced(tile=0, splits=1)
    y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
    forced()
    ref = torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T)
    assert_close(y, ref.cpu(), "y")


# Row tiles of a weight gradient (128 or 256 columns of g): below, at and past a super-group of eight, split and not.
@pytest.mark.parametrize("tile,splits", [(0, 1), (2, 3), (2, 1)])
@pytest.mark.parametrize("N", [7 * 128 - 8, 8 * 128, 9 * 128 + 8, 17 * 128 + 40])
def test_weight_gradient_super_groups(dev, forced, tile, splits, N):
    note(f"weight-gradient order: N={N} tile={tile} splits={splits}")
    x, Wv, Wt, mask, g = make_linear(dev, 300, 201, 264, N, seed=N)
    forced(tile, splits)
    dx, dv, dt = masked_linear_backward(g, x, Wv.T, Wt.T, mask)
    forced()
    gd, xd, mv = g.double(), x.double(), mask.double()[:, None]
    assert_close(dv.T, ((gd * mv).T @ xd).cpu(), "dWv")
    assert_close(dt.T, ((gd * (1 - mv)).T @ xd).cpu(), "dWt")
    assert_close(dx, torch.where(mask[:, None], gd @ Wv.double(), gd @ Wt.double()).cpu(), "dx")


def select_ffn(x, W, mask):
    """SwiGLU feed-forward, row-select form in double precision, the intermediate rounded to bf16 once as it is stored."""
    out = torch.empty_like(x, dtype=torch.float64)
    for sel, g, d, u in ((mask, 0, 1, 2), (~mask, 3, 4, 5)):
        xs = x[sel].double()
        t1 = xs @ W[g].double().T
        mid = (t1 * torch.sigmoid(t1) * (xs @ W[u].double().T)).to(torch.bfloat16).double()
        out[sel] = mid @ W[d].double().T
    return out


# The ring tiles of 128 x 256 and 64 x 128: contractions of fewer slabs than stages, exactly as many and more; single rows,
# whole tiles, one row past them; columns below and past a tile; cut into K ranges with and without a remainder.
@pytest.mark.parametrize("tile", [6, 7])
@pytest.mark.parametrize("nv,nt,K,N,splits", [(1, 1, 64, 8, 1), (128, 64, 128, 256, 1), (129, 0, 192, 264, 1), (0, 257, 256, 136, 1),
                                              (65, 63, 1024, 520, 3), (200, 130, 1536, 128, 5)])
def test_ring_tiles(dev, forced, tile, nv, nt, K, N, splits):
    note(f"ring tile {tile}: nv={nv} nt={nt} K={K} N={N} splits={splits}")
    x, Wv, Wt, mask, g = make_linear(dev, nv, nt, K, N, seed=K + N)
    forced(tile, splits)
    y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
    dx = masked_linear_backward(g, x, Wv.T, Wt.T, mask)[0]  # over K-major weights, contraction N
    h = 136  # M, d, h beyond the decode kernels' shapes: h is no multiple of 128
    gen = torch.Generator(device=dev).manual_seed(3)
    W = [(torch.randn(*s, generator=gen, device=dev) * 0.05).to(torch.bfloat16) for s in ((h, K), (K, h), (h, K)) * 2]
    out = MaskedFFN.apply(x, *[w.T for w in W], mask)
    forced()
    assert_close(y, torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T).cpu(), "y")
    assert_close(dx, torch.where(mask[:, None], g.double() @ Wv.double(), g.double() @ Wt.double()).cpu(), "dx")
    assert_close(out, select_ffn(x, W, mask).cpu(), "ffn")


# The split factor depends on the number of M-tiles, which only the device knows: as many as the rows need, or one more.
@pytest.mark.parametrize("nv", [0, 128, 150, 199, 200])
@pytest.mark.parametrize("K,N", [(4096, 512), (8192, 1024)])
def test_split_factor_by_row_tiles(dev, nv, K, N):
    note(f"split factor: nv={nv} of 200, K={K} N={N}")
    assert _lib.tile_config(_lib.OP_LINEAR_FWD, 200, K, N)["split_k"] > 1
    x, Wv, Wt, mask, _ = make_linear(dev, nv, 200 - nv, K, N, seed=nv)
    y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
    assert_close(y, torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T).cpu(), "y")


# The remainder of a launch on 256-row SwiGLU tiles: exactly half a round (256 + 128 tiles), one tile past it (256 + 129: another
# whole round), and one tile past a round; the same past eight rounds, below which the four-wave tile runs beside 160-row ones.
# d = 64, h = 128 * tiles_n columns.
@pytest.mark.parametrize("tiles_m,h", [(6, 64 * 128), (55, 7 * 128), (257, 128), (17, 128 * 128), (311, 7 * 128), (683, 3 * 128)])
def test_whole_rounds_and_remainder(dev, forced, tiles_m, h):
    note(f"remainder of whole rounds: {tiles_m} M-tiles, h={h}")
    x, _, _, mask, _ = make_linear(dev, 256 * 2, 256 * (tiles_m - 2) - 5, 64, 8, seed=tiles_m)
    gen = torch.Generator(device=dev).manual_seed(5)
    W = [(torch.randn(*s, generator=gen, device=dev) * 0.05).to(torch.bfloat16) for s in ((h, 64), (64, h), (h, 64)) * 2]
    forced(1)
    assert _lib.load().ffnk_debug_ffn_joint(x.shape[0], 64, h) & 1 == (tiles_m * h <= 8 * 256 * 128)
    out = MaskedFFN.apply(x, *[w.T for w in W], mask)
    forced()
    assert_close(out, select_ffn(x, W, mask).cpu(), "ffn")


def ffn_case(dev, nv, nt, d, h, seed):
    x, _, _, mask, _ = make_linear(dev, nv, nt, d, 8, seed)
    gen = torch.Generator(device=dev).manual_seed(seed + 1)
    W = [(torch.randn(*s, generator=gen, device=dev) * 0.05).to(torch.bfloat16) for s in ((h, d), (d, h), (h, d)) * 2]
    return x, W, mask, torch.randn(nv + nt, d, generator=gen, device=dev).to(torch.bfloat16)


def assert_ffn_backward(x, W, mask, g, what):
    """Gradients of the feed-forward layer against the chain rule in double precision with the same bf16 storage points."""
    views = [w.T for w in W]
    out, pre = masked_ffn_forward(x, *views, mask, save_pre=True)
    got = masked_ffn_backward(g, x, *views, mask, pre=pre)
    dx, dW = om.ffn_backward_select(g.cpu(), x.cpu(), dict(zip(("w1", "w2", "w3", "u1", "u2", "u3"), (w.cpu() for w in W))), mask.cpu(),
                                    torch.float64, round_intermediates=True)
    assert_close_pipeline(got[0], dx, f"{what}: dx")
    for i, k in enumerate(("w1", "w2", "w3", "u1", "u2", "u3")):
        assert_close_pipeline(got[1 + i].T, dW[k], f"{what}: d{k}")


# The ring tiles of three stages over K-major weights (dh and dx): contractions of fewer slabs than stages and more, through
# both up-projection weights (h a multiple of 64) or over copies of them, ragged rows and columns, single rows, cut into ranges.
@pytest.mark.parametrize("tile", [6, 7])
@pytest.mark.parametrize("nv,nt,d,h,splits", [(1, 69, 64, 64, 1), (128, 64, 128, 320, 1), (129, 0, 264, 192, 1), (65, 130, 520, 136, 1),
                                              (200, 130, 136, 1024, 3)])
def test_backward_ring_tiles(dev, forced, tile, nv, nt, d, h, splits):
    note(f"backward ring tile {tile}: nv={nv} nt={nt} d={d} h={h} splits={splits}")
    case = ffn_case(dev, nv, nt, d, h, seed=d + h)
    forced(tile, splits)
    assert_ffn_backward(*case, f"tile {tile}")


# dx of the feed-forward layer on its own plan, a contraction of 2h cut by the number of row tiles: as many as the rows need, or
# one more.
@pytest.mark.parametrize("nv", [0, 64, 100, 199, 200])
def test_backward_split_factor_by_row_tiles(dev, nv):
    note(f"backward split factor: nv={nv} of 200")
    assert_ffn_backward(*ffn_case(dev, nv, 200 - nv, 512, 2048, seed=nv), f"nv {nv}")


# dx over up-projection weights whose rows end inside a slab: less than a slab, one row group short of whole slabs, one past, on
# every tile and cut into ranges (whose ends may be either weight's ragged slab).  What lies behind the weights is NaN.
@pytest.mark.parametrize("tile,splits", [(-1, -1), (0, 1), (1, 1), (2, 1), (3, 1), (4, 1), (6, 1), (7, 1), (2, 3), (7, 5)])
@pytest.mark.parametrize("h", [8, 72, 200, 312, 1016])
def test_backward_ragged_intermediate(dev, forced, tile, splits, h):
    note(f"backward ragged intermediate: h={h} tile={tile} splits={splits}")
    x, W, mask, g = ffn_case(dev, 90, 75, 136, h, seed=h)
    for i in (0, 2, 3, 5):
        behind = torch.full((h + 64, 136), float("nan"), dtype=torch.bfloat16, device=dev)
        behind[:h] = W[i]
        W[i] = behind[:h]
    forced(tile, splits)
    assert_ffn_backward(x, W, mask, g, f"h {h} tile {tile}")


# The SwiGLU GEMM on tiles of two heights in one launch: rows of a modality that fill a short tile, that one row more does not,
# that are two short tiles, a tall one and the rest; one modality; several super-groups.  Contractions of one slab, of fewer than
# the short tile's stages, ragged ones; columns of whole rounds, just past one (the rest as halves) and a ragged last tile.
@pytest.mark.parametrize("nv,nt,h", [(1, 511, 32768), (160, 352, 32768), (161, 256, 33000), (262, 157, 32776), (576, 835, 11528),
                                     (0, 700, 24576), (2060, 100, 7432), (256, 256, 32896)])
@pytest.mark.parametrize("d", [64, 128, 200, 328])
def test_tiles_of_two_heights(dev, nv, nt, h, d):
    note(f"tiles of two heights: nv={nv} nt={nt} h={h} d={d}")
    cfg = _lib.tile_config(_lib.OP_FFN_UP, nv + nt, d, h)
    assert (cfg["block_m"], cfg["waves_m"] * cfg["waves_n"]) == (256, 4) and _lib.load().ffnk_debug_ffn_joint(nv + nt, d, h) & 1
    x, W, mask, _ = ffn_case(dev, nv, nt, d, h, seed=h + d)
    W = [w * 0.5 for w in W]
    out, pre = masked_ffn_forward(x, *[w.T for w in W], mask, save_pre=True)
    assert_close(out, select_ffn(x, W, mask).cpu(), "out")
    assert torch.equal(out, masked_ffn_forward(x, *[w.T for w in W], mask))
    order = torch.cat([mask.nonzero(), (~mask).nonzero()]).flatten()
    xs, m = x[order].double(), mask[order][:, None]
    for half, (v, t) in enumerate(((W[0], W[3]), (W[2], W[5]))):
        assert_close(pre[:, half * h:(half + 1) * h], torch.where(m, xs @ v.double().T, xs @ t.double().T).cpu(), f"pre {half}")


# The order of that launch in super-groups of other sizes: the same tiles, the same sums.
@pytest.mark.parametrize("group", [1, 3, 64])
def test_tiles_of_two_heights_in_super_groups(dev, group):
    note(f"tiles of two heights: super-groups of {group}")
    lib = _lib.load()
    x, W, mask, _ = ffn_case(dev, 2060, 100, 128, 7432, seed=9)
    out = masked_ffn_forward(x, *[w.T for w in W], mask)
    try:
        lib.ffnk_debug_force_group_m(group)
        assert _lib.tile_config(_lib.OP_FFN_UP, 2160, 128, 7432)["group_m"] == group
        other = masked_ffn_forward(x, *[w.T for w in W], mask)
    finally:
        lib.ffnk_debug_force_group_m(0)
    assert torch.equal(out, other)


# The SwiGLU derivative on the dh GEMM's tiles: row and column edges of every tile, halves padded to whole slabs (h = 328, 72) and
# not, pre-activations kept by a forward (also in rows wider than they are) and recomputed in place; down weights in both layouts.
@pytest.mark.parametrize("tile", [-1, 0, 1, 2, 3, 4, 6, 7])
@pytest.mark.parametrize("nv,nt,d,h", [(1, 66, 136, 72), (130, 257, 128, 328), (0, 300, 200, 512)])
def test_swiglu_backward_in_the_epilogue(dev, forced, tile, nv, nt, d, h):
    note(f"SwiGLU backward in the epilogue: nv={nv} nt={nt} d={d} h={h} tile={tile}")
    x, W, mask, g = ffn_case(dev, nv, nt, d, h, seed=d + h)
    forced(tile)
    assert_ffn_backward(x, W, mask, g, f"tile {tile}")
    for views in ([w.T for w in W], [w.T.contiguous() if i % 3 == 1 else w.T for i, w in enumerate(W)]):
        _, pre = masked_ffn_forward(x, *views, mask, save_pre=True)
        wide = torch.full((nv + nt, 2 * h + 24), float("nan"), dtype=torch.bfloat16, device=dev)
        wide[:, :2 * h] = pre
        kept = masked_ffn_backward(g, x, *views, mask, pre=pre)
        for other in (masked_ffn_backward(g, x, *views, mask, pre=wide[:, :2 * h]), masked_ffn_backward(g, x, *views, mask)):
            assert all(torch.equal(a, b) for a, b in zip(kept, other))


# dx in one launch with the weight gradients on 256x256 tiles: ragged extents, rows of both modalities, of one, and a single one.
@pytest.mark.parametrize("nv,nt,d,h", [(1200, 1301, 3080, 1000), (0, 2500, 4096, 1024), (1599, 1, 4104, 1032)])
def test_dx_beside_the_weight_gradients(dev, forced, nv, nt, d, h):
    note(f"dx beside dW: nv={nv} nt={nt} d={d} h={h}")
    case = ffn_case(dev, nv, nt, d, h, seed=d + h)
    forced(0)
    assert _lib.load().ffnk_debug_ffn_joint(nv + nt, d, h) & 2
    assert_ffn_backward(*case, "one launch")


# 192-row tiles among 128-row ones (csrc/gemm_sched.hpp: stretch_rows): a round of the chip and one M-tile more, the last M-tile of
# the stretched modality at one row, at the edges of what one and two taller tiles hold, whole, and in either modality; contraction
# of a few slabs, whole and ragged.
@pytest.mark.parametrize("tile,N", [(2, 8192), (6, 8192)])
@pytest.mark.parametrize("K", [192, 328])
@pytest.mark.parametrize("nv,nt", [(513, 511), (576, 448), (577, 447), (448, 576), (447, 577), (639, 385), (1000, 24), (0, 1025), (1025, 0)])
def test_stretched_tiles(dev, forced, tile, N, K, nv, nt):
    note(f"192-row tiles among 128-row ones: tile={tile} K={K} {nv} visual, {nt} text rows")
    x, Wv, Wt, mask, _ = make_linear(dev, nv, nt, K, N, seed=nv + K)
    forced(tile=tile, splits=1)
    y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
    forced()
    ref = torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T)
    assert_close(y, ref.cpu(), "y")


# The same on 160-row tiles (192-row ones among them) and 192-row tiles (224), unsplit and cut into two K ranges, where the last M-tile
# takes one to six taller ones, and where a modality has too few M-tiles for that.
@pytest.mark.parametrize("tile,base", [(16, 192), (17, 160)])
@pytest.mark.parametrize("N,splits,K", [(8192, 1, 328), (4096, 2, 712)])
@pytest.mark.parametrize("more", [0, 1, 32, 33, 100, 150, 300])
def test_stretched_tiles_between(dev, forced, tile, base, N, splits, K, more):
    nv = 4 * base + more
    nt = 8 * base - nv
    note(f"tiles between 128 and 256 rows: tile={tile} K={K} splits={splits} {nv} visual, {nt} text rows")
    x, Wv, Wt, mask, _ = make_linear(dev, nv, nt, K, N, seed=nv + K)
    forced(tile=tile, splits=splits)
    y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
    forced()
    ref = torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T)
    assert_close(y, ref.cpu(), "y")


@pytest.mark.parametrize("tile", [16, 17])
@pytest.mark.parametrize("nv,nt", [(1, 0), (0, 159), (161, 192), (193, 1), (400, 225)])
def test_tiles_between_at_few_rows(dev, forced, tile, nv, nt):
    note(f"tiles between 128 and 256 rows: tile={tile} {nv} visual, {nt} text rows")
    x, Wv, Wt, mask, _ = make_linear(dev, nv + 64, nt, 192, 264, seed=nv)
    forced(tile=tile, splits=1)
    y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
    forced()
    ref = torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T)
    assert_close(y, ref.cpu(), "y")


@pytest.mark.parametrize("tile", [2, 6, 16, 17])
def test_stretched_down_projection(dev, forced, tile):
    nv, nt, d, h = 540, 484, 8192, 192
    note(f"192-row tiles in the down projection: tile={tile}")
    x, _, _, mask, _ = make_linear(dev, nv, nt, d, 8, seed=5)
    gen = torch.Generator(device=dev).manual_seed(6)
    w = [(torch.randn(*s, generator=gen, device=dev) * 0.02).bfloat16() for s in [(h, d), (d, h), (h, d)] * 2]
    forced(tile=tile, splits=1)
    y = MaskedFFN.apply(x, *(v.T for v in w), mask)
    forced()

    def half(w1, w2, w3):
        g, u = x.double() @ w1.double().T, x.double() @ w3.double().T
        return (torch.nn.functional.silu(g) * u).bfloat16().double() @ w2.double().T

    assert_close(y, torch.where(mask[:, None], half(*w[:3]), half(*w[3:])).cpu(), "y")


# 256-row tiles of the SwiGLU GEMM past a whole round, cut into 64-row pieces (mixed_pieces): a few tiles and a quarter of a round, a
# last column tile that is half full, modalities that end at the edges of a piece, pre-activations kept or not.
@pytest.mark.parametrize("nv,nt,h", [(1500, 0, 5440), (760, 740, 5504), (0, 1473, 5504), (1281, 200, 5504), (1217, 0, 8192), (513, 705, 8128)])
@pytest.mark.parametrize("save", [False, True])
def test_swiglu_tiles_in_quarters(dev, forced, nv, nt, h, save):
    d = 128
    note(f"SwiGLU tiles in quarters: {nv} visual, {nt} text rows, h={h} save={save}")
    x, _, _, mask, _ = make_linear(dev, nv, nt, d, 8, seed=nv + h)
    gen = torch.Generator(device=dev).manual_seed(h)
    w = [(torch.randn(*s, generator=gen, device=dev) * 0.05).bfloat16() for s in [(h, d), (d, h), (h, d)] * 2]
    forced(tile=1)
    y = masked_ffn_forward(x, *(v.T for v in w), mask, save_pre=save)
    forced()

    def half(w1, w2, w3):
        g, u = x.double() @ w1.double().T, x.double() @ w3.double().T
        return (torch.nn.functional.silu(g) * u).bfloat16().double() @ w2.double().T

    assert_close(y[0] if save else y, torch.where(mask[:, None], half(*w[:3]), half(*w[3:])).cpu(), "y")
    if save:
        order = torch.cat([mask.nonzero()[:, 0], (~mask).nonzero()[:, 0]])
        pre = torch.where(mask[:, None], x.double() @ torch.cat([w[0], w[2]]).double().T, x.double() @ torch.cat([w[3], w[5]]).double().T)
        assert_close(y[1], pre[order].cpu(), "pre")
