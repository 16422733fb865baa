"""Contractions that are no whole number of 64-element slabs (the first one overlaps the second), against the
row-select form in double precision computed with torch on the GPU."""
import pytest
import torch

from ffn_kernel_amd import MaskedLinear, _lib
from ffn_kernel_amd.ops import masked_ffn_backward, masked_ffn_forward, masked_linear_backward
from ffn_kernel_amd import workloads as wl
from helpers import assert_close, assert_close_pipeline, note
from oracle import cref
from oracle import modules as om

pytestmark = pytest.mark.gpu


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


def linear_case(dev, M, K, N, p, seed):
    gen = torch.Generator(device=dev).manual_seed(seed)
    rnd = lambda r, c, std: (torch.randn(r, c, generator=gen, device=dev) * std).to(torch.bfloat16)
    mask = torch.rand(M, generator=gen, device=dev) < p
    return rnd(M, K, 1.0), rnd(N, K, 0.05), rnd(N, K, 0.05), mask, rnd(M, N, 1.0)


# Under 128 (register-staged), two slabs, three, four and five slabs with 8 ... 56 elements in the first, and 33.
@pytest.mark.parametrize("K,N", [(120, 136), (136, 200), (184, 184), (248, 72), (264, 328), (2056, 264)])
@pytest.mark.parametrize("tile,splits", [(-1, -1), (0, 1), (1, 1), (2, 1), (3, 1), (4, 1), (6, 1), (7, 1), (2, 2), (4, 2), (0, 2)])
def test_linear_fwd_bwd(dev, forced, tile, splits, K, N):
    note(f"ragged linear fwd + bwd K={K} N={N} tile={tile} splits={splits}")
    x, Wv, Wt, mask, g = linear_case(dev, 301, K, N, 0.45, seed=K + N)
    forced(tile, splits)
    if tile in (6, 7) and N >= 128:  # dx on the ring tiles of three stages themselves
        cfg = _lib.tile_config(_lib.OP_BWD_DX, 301, K, N)
        assert (cfg["block_m"], cfg["lds_stages"]) == ((128, 64)[tile - 6], 3)
    y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
    dx, dv, dt = masked_linear_backward(g, x, Wv.T, Wt.T, mask)
    forced()
    m = mask[:, None]
    assert_close(y, torch.where(m, x.double() @ Wv.double().T, x.double() @ Wt.double().T).cpu(), "y")
    assert_close(dx, torch.where(m, g.double() @ Wv.double(), g.double() @ Wt.double()).cpu(), "dx")
    gv = g.double() * m
    assert_close(dv.T, (gv.T @ x.double()).cpu(), "dWv")
    assert_close(dt.T, ((g.double() - gv).T @ x.double()).cpu(), "dWt")


@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4, 6, 7])
def test_what_lies_ahead_of_a_row_never_counts(dev, forced, tile):
    """Slab 0 would start ahead of the contraction, where the row before ends: non-finite values there stay in their own row of
    the output (token rows, weight rows) and of dx (weight rows of the K-major panel, token rows of g)."""
    note(f"ragged linear: non-finite neighbours, tile={tile}")
    K, N, M = 200, 264, 260
    x, Wv, Wt, mask, g = linear_case(dev, M, K, N, 0.5, seed=5)
    x[40, -64:] = float("nan")
    Wv[70, -64:] = float("inf")
    g[90, -64:] = float("nan")
    forced(tile, 1)
    y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
    dx = masked_linear_backward(g, x, Wt.T, Wt.T, mask)[0]
    forced()
    rows, cols = torch.arange(M, device=dev) != 40, torch.arange(N, device=dev) != 70
    ref = torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T)
    assert_close(y[rows][:, cols], ref[rows][:, cols].cpu(), "y")
    rows = torch.arange(M, device=dev) != 90
    assert_close(dx[rows], (g.double() @ Wt.double())[rows].cpu(), "dx")


# 17 and 19 column tiles of 256 over 16 row tiles: past one round of the chip, the remainder as a split tail.
@pytest.mark.parametrize("K", [1032, 1080])
def test_split_tail(dev, forced, K):
    note(f"ragged linear: split tail K={K}")
    x, Wv, Wt, mask, _ = linear_case(dev, 4000, K, 4400, 0.5, seed=K)
    for tile in (0, 1):
        forced(tile, 1)
        y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
        forced()
        assert_close(y, torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T).cpu(), f"tile {tile}")


@pytest.mark.parametrize("tile", [-1, 0, 1, 2, 3, 4, 6, 7])
@pytest.mark.parametrize("M,d,h", [(300, 136, 264), (180, 200, 392), (300, 192, 328), (300, 264, 256)])
def test_ffn_fwd_bwd(dev, forced, tile, M, d, h):
    note(f"ragged ffn fwd + bwd M={M} d={d} h={h} tile={tile}")
    gen = torch.Generator().manual_seed(M + d)
    w = wl.make_ffn("t", M, d, h, torch.rand(M, generator=gen) < 0.4, seed=h, w_std=0.05)
    g = torch.randn(M, d, generator=gen).to(torch.bfloat16)
    dw = w.to(dev)
    forced(tile)
    out, pre = masked_ffn_forward(*dw.op_args(), save_pre=True)
    grads_saved = masked_ffn_backward(g.to(dev), *dw.op_args(), pre=pre)
    grads = masked_ffn_backward(g.to(dev), *dw.op_args())
    torch.cuda.synchronize()
    forced()
    assert_close(out, cref.ffn_fwd(w.x, w.W, w.mask, round_mid=True), "ffn out")
    rdx, rdW = om.ffn_backward_select(g, w.x, w.W, w.mask, torch.float64, round_intermediates=True)
    for got in (grads, grads_saved):
        assert_close_pipeline(got[0], rdx, "dx")
        for i, k in enumerate(("w1", "w2", "w3", "u1", "u2", "u3")):
            assert_close_pipeline(got[1 + i].T, rdW[k], f"d{k}")
