"""Outputs with a row stride of their own: every tile stores its results where they belong and nothing beside them, whichever way
they leave the kernel - whole 16-byte chunks of a row, or runs of four where the output is not made of such chunks."""
import pytest
import torch

from ffn_kernel_amd import _lib
from helpers import assert_close, note

pytestmark = pytest.mark.gpu
MARK = -77.0


def canvas(rows, cols, ahead, pad, dev):
    """(buffer, view): a [rows, cols] view `ahead` elements into a marked buffer whose rows are cols + pad apart."""
    buf = torch.full((ahead + rows * (cols + pad),), MARK, dtype=torch.bfloat16, device=dev)
    return buf, buf[ahead:].view(rows, cols + pad)[:, :cols]


def untouched(buf, view):
    view.fill_(MARK)
    return bool((buf == MARK).all())


def rnd(gen, r, c, std, dev):
    return (torch.randn(r, c, generator=gen, device=dev) * std).to(torch.bfloat16)


@pytest.fixture
def forced():
    lib = _lib.load()
    try:
        yield lambda tile: lib.ffnk_debug_force_tile(tile)
    finally:
        lib.ffnk_debug_force_tile(-1)


# One chunk of columns, a ragged last tile, one past a tile; whole chunks at an offset, a start or a stride that is none, columns
# that are none.
LAYOUTS = [(8, 0, 0), (136, 0, 8), (264, 8, 24), (264, 4, 0), (136, 0, 4), (132, 0, 4), (100, 0, 0)]


@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4, 6, 7])
@pytest.mark.parametrize("N,ahead,pad", LAYOUTS)
def test_linear_forward_rows(dev, forced, tile, N, ahead, pad):
    note(f"output rows: tile {tile} N={N} ahead={ahead} pad={pad}")
    M, K = 333, 192
    gen = torch.Generator(device=dev).manual_seed(N + ahead)
    x, Wv, Wt = rnd(gen, M, K, 1.0, dev), rnd(gen, N, K, 0.05, dev), rnd(gen, N, K, 0.05, dev)
    mask = torch.rand(M, generator=gen, device=dev) < 0.4
    buf, y = canvas(M, N, ahead, pad, dev)
    forced(tile)
    ws = torch.empty(_lib.workspace_bytes(_lib.OP_LINEAR_FWD, M, K, N), dtype=torch.uint8, device=dev)
    rc = _lib.load().ffnk_masked_linear_fwd(x.data_ptr(), K, Wv.data_ptr(), Wt.data_ptr(), 1, K, mask.data_ptr(), y.data_ptr(),
                                            N + pad, M, K, N, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "linear")
    assert_close(y, torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T).cpu(), "y")
    assert untouched(buf, y)


@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4, 6, 7])
@pytest.mark.parametrize("h,pad", [(136, 0), (264, 8), (72, 16)])
def test_saved_pre_activations(dev, forced, tile, h, pad):
    """Gate and up pre-activations beside the forward's result, in routed order."""
    note(f"saved pre-activations: tile {tile} h={h} pad={pad}")
    M, d = 261, 128
    gen = torch.Generator(device=dev).manual_seed(h)
    x = rnd(gen, M, d, 1.0, dev)
    W = [rnd(gen, *s, 0.05, dev) for s in ((h, d), (d, h), (h, d)) * 2]
    mask = torch.rand(M, generator=gen, device=dev) < 0.5
    buf, pre = canvas(M, 2 * h, 0, pad, dev)
    out = torch.empty(M, d, dtype=torch.bfloat16, device=dev)
    forced(tile)
    ws = torch.empty(_lib.workspace_bytes(_lib.OP_FFN_FWD, M, d, h), dtype=torch.uint8, device=dev)
    p = [w.data_ptr() for w in W]
    rc = _lib.load().ffnk_masked_ffn_fwd_save(x.data_ptr(), d, p[0], p[2], p[3], p[5], 1, d, p[1], p[4], 1, h, mask.data_ptr(),
                                              out.data_ptr(), d, pre.data_ptr(), 2 * h + pad, M, d, h, ws.data_ptr(), ws.numel(),
                                              torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "ffn")
    order = torch.cat([mask.nonzero(), (~mask).nonzero()]).flatten()
    xs, m = x[order].double(), mask[order][:, None]
    assert_close(pre[:, :h], torch.where(m, xs @ W[0].double().T, xs @ W[3].double().T).cpu(), "gate")
    assert_close(pre[:, h:], torch.where(m, xs @ W[2].double().T, xs @ W[5].double().T).cpu(), "up")
    assert untouched(buf, pre)


# Weight gradients in every layout: contiguous along the input features (nn.Linear) or along the output features, rows further
# apart than they are long, rows that are no whole chunks.
@pytest.mark.parametrize("tile", [-1, 0, 1, 2, 3, 4])
@pytest.mark.parametrize("K,N,pad,k_contig", [(72, 264, 8, True), (136, 264, 0, True), (264, 136, 8, False), (136, 72, 4, True)])
def test_weight_gradient_rows(dev, forced, tile, K, N, pad, k_contig):
    note(f"weight-gradient rows: tile {tile} K={K} N={N} pad={pad} k_contig={k_contig}")
    M = 200
    gen = torch.Generator(device=dev).manual_seed(K + N)
    x, g = rnd(gen, M, K, 1.0, dev), rnd(gen, M, N, 1.0, dev)
    Wv, Wt = rnd(gen, N, K, 0.05, dev), rnd(gen, N, K, 0.05, dev)
    mask = torch.rand(M, generator=gen, device=dev) < 0.5
    rows, cols = (N, K) if k_contig else (K, N)
    bufs, views = zip(*(canvas(rows, cols, 0, pad, dev) for _ in range(2)))
    dx = torch.empty(M, K, dtype=torch.bfloat16, device=dev)
    sk, sn = (1, cols + pad) if k_contig else (cols + pad, 1)
    forced(tile)
    ws = torch.empty(_lib.workspace_bytes(_lib.OP_LINEAR_BWD, M, K, N), dtype=torch.uint8, device=dev)
    rc = _lib.load().ffnk_masked_linear_bwd(g.data_ptr(), N, x.data_ptr(), K, Wv.data_ptr(), Wt.data_ptr(), 1, K, mask.data_ptr(),
                                            dx.data_ptr(), K, views[0].data_ptr(), views[1].data_ptr(), sk, sn, M, K, N,
                                            ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "linear backward")
    for view, buf, sel in zip(views, bufs, (mask, ~mask)):
        ref = (g.double() * sel[:, None]).T @ x.double()
        assert_close(view if k_contig else view.T, ref.cpu(), "dW")
        assert untouched(buf, view)
