"""Decode sizes (M <= 64) over extents that are multiples of 8 but not of 128: the weight streams with a last K slice or
chunk cut short and a last row block that overlaps the one before it."""
import pytest
import torch

from ffn_kernel_amd import MaskedFFN, MaskedLinear, _lib
from ffn_kernel_amd import workloads as wl
from ffn_kernel_amd.ops import masked_ffn_backward, masked_ffn_forward
from helpers import assert_close, assert_close_pipeline, note
from oracle import cref
from oracle import modules as om

pytestmark = pytest.mark.gpu


def framed(t):
    """t as a column slice of a wider tensor of NaNs: a load past a row's ends shows up in the result."""
    wide = torch.full((t.shape[0], t.shape[1] + 16), float("nan"), dtype=t.dtype, device=t.device)
    wide[:, 8:-8] = t
    return wide[:, 8:-8]


# 8, 64 and 120 elements past a chunk of 128 and a slice of 512; 1 and 2 slices per wavefront, up to 16 wavefronts; row
# counts of 8 ... 56 past a block; M at the edges of the kernels' token-row tiles.
@pytest.mark.parametrize("M,p", [(1, 0.0), (2, 0.5), (3, 1.0), (5, 0.5), (8, 0.6), (9, 0.5), (16, 1.0), (17, 0.5), (33, 0.0),
                                 (48, 1.0), (64, 0.5), (64, 1.0)])
@pytest.mark.parametrize("K,N", [(520, 72), (904, 72), (1088, 200), (1144, 136), (2056, 1544), (4104, 328), (15880, 120)])
def test_linear(dev, M, p, K, N):
    note(f"ragged decode linear M={M} K={K} N={N} p={p}")
    streamed = M <= 8 or K > 896
    assert (_lib.tile_config(_lib.OP_LINEAR_FWD, M, K, N)["path"] == _lib.PATH_STREAM) == streamed
    gen = torch.Generator(device=dev).manual_seed(M * K + N)
    rnd = lambda r, c, std: (torch.randn(r, c, generator=gen, device=dev) * std).to(torch.bfloat16)
    x, Wv, Wt = rnd(M, K, 1.0), rnd(N, K, 0.03), rnd(N, K, 0.03)
    mask = torch.rand(M, generator=gen, device=dev) < p
    ref = torch.where(mask[:, None], x.double() @ Wv.double().T, x.double() @ Wt.double().T)
    y = MaskedLinear.apply(framed(x), framed(Wv).T, framed(Wt).T, mask)
    assert_close(y, ref.cpu(), "y")
    assert torch.equal(y, MaskedLinear.apply(x, Wv.T, Wt.T, mask))
    # a non-finite weight or token value stays in its column or row, and is counted once: inf, not NaN
    x, Wv, Wt = x.abs() + 0.125, Wv.clone(), Wt.clone()
    for at in (0, K - 120, K - 8, K - 1):
        Wv[:, at] = Wt[:, at] = 0.0
        Wv[7, at] = Wt[7, at] = float("inf")
    y = MaskedLinear.apply(x, Wv.T, Wt.T, mask)
    assert torch.isposinf(y[:, 7]).all() and torch.isfinite(y[:, :7]).all() and torch.isfinite(y[:, 8:]).all()


def test_token_rows_far_apart(dev):
    """Row strides past the LDS-transposed streams' 32-bit offsets run on the tiled GEMM, as they did before."""
    note("ragged decode, 2^26 elements between token rows")
    M, K, N = 16, 904, 72
    x = torch.empty(M, 1 << 26, dtype=torch.bfloat16, device=dev)[:, :K]
    gen = torch.Generator(device=dev).manual_seed(1)
    x.copy_(torch.randn(M, K, generator=gen, device=dev))
    W = [(torch.randn(N, K, generator=gen, device=dev) * 0.03).to(torch.bfloat16) for _ in range(2)]
    mask = torch.arange(M, device=dev) % 3 == 0
    ref = torch.where(mask[:, None], x.double() @ W[0].double().T, x.double() @ W[1].double().T)
    assert_close(MaskedLinear.apply(x, W[0].T, W[1].T, mask), ref.cpu(), "y")


# Whole 128-element chunks off the dot kernels' slices: each projection on its own kernel (22528: past 16 wavefronts).
@pytest.mark.parametrize("M,kind", [(1, "visual"), (5, "bernoulli"), (8, "bernoulli")])
@pytest.mark.parametrize("d,h", [(1152, 2176), (1664, 4224), (1024, 22528)])
def test_ffn_whole_chunks(dev, M, kind, d, h):
    note(f"decode ffn on the dot streams M={M} kind={kind} d={d} h={h}")
    up, down = (_lib.tile_config(op, M, d, h) for op in (_lib.OP_FFN_UP, _lib.OP_FFN_DOWN))
    assert up["block_m"] == M and (down["block_m"] == M) == (h <= 16384)
    w = wl.cfg5_ffn_decode(M, kind, seed=120 + M, d=d, h=h)
    out = MaskedFFN.apply(*w.to(dev).op_args())
    assert_close(out, cref.ffn_fwd(w.x, w.W, w.mask, round_mid=True), f"decode {M} {kind}")


@pytest.mark.parametrize("M,kind", [(1, "text"), (4, "bernoulli"), (7, "visual"), (8, "bernoulli"), (9, "bernoulli"),
                                    (31, "visual"), (40, "bernoulli"), (64, "bernoulli"), (64, "text")])
@pytest.mark.parametrize("d,h", [(904, 1000), (1096, 2200), (1088, 1856), (1024, 2120), (1984, 1024)])
def test_ffn(dev, M, kind, d, h):
    note(f"ragged decode ffn M={M} kind={kind} d={d} h={h}")
    assert _lib.tile_config(_lib.OP_FFN_UP, M, d, h)["path"] == _lib.PATH_STREAM
    w = wl.cfg5_ffn_decode(M, kind, seed=90 + M, d=d, h=h)
    w = wl.FFNWorkload(w.name, w.x, {k: (v.float() * 1.5).to(torch.bfloat16) for k, v in w.W.items()}, w.mask)
    out = MaskedFFN.apply(*w.to(dev).op_args())
    assert_close(out, cref.ffn_fwd(w.x, w.W, w.mask, round_mid=True), f"ragged decode {M} {kind}")
    assert torch.equal(out, MaskedFFN.apply(*w.to(dev).op_args()))
    if kind != "bernoulli":
        W = dict(w.W)
        for k in (("u1", "u2", "u3") if kind == "visual" else ("w1", "w2", "w3")):
            W[k] = torch.full_like(W[k], float("nan"))
        assert torch.equal(MaskedFFN.apply(*wl.FFNWorkload("p", w.x, W, w.mask).to(dev).op_args()), out)


def test_training_forward_keeps_its_pre_activations(dev):
    """A training step of few rows over such extents still saves t1 | t3 (on the tiled GEMMs)."""
    note("ragged decode-sized training step")
    M, d, h = 40, 1096, 2200
    assert _lib.load().ffnk_masked_ffn_can_save(M, d, h) == 1
    gen = torch.Generator().manual_seed(3)
    w = wl.make_ffn("t", M, d, h, torch.rand(M, generator=gen) < 0.4, seed=h, w_std=0.03)
    g = torch.randn(M, d, generator=gen).to(torch.bfloat16)
    dw = w.to(dev)
    out, pre = masked_ffn_forward(*dw.op_args(), save_pre=True)
    assert pre is not None
    grads = masked_ffn_backward(g.to(dev), *dw.op_args(), pre=pre)
    assert_close(out, cref.ffn_fwd(w.x, w.W, w.mask, round_mid=True), "ffn out")
    rdx, rdW = om.ffn_backward_select(g, w.x, w.W, w.mask, torch.float64, round_intermediates=True)
    assert_close_pipeline(grads[0], rdx, "dx")
    for i, k in enumerate(("w1", "w2", "w3", "u1", "u2", "u3")):
        assert_close_pipeline(grads[1 + i].T, rdW[k], f"d{k}")
