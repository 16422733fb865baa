"""Forward GEMMs that make the row partition themselves (csrc/route_rows.hpp), against the partition of ffnk_route and the same
GEMM reading it: the same integers, the same results bit for bit, at the edges of a thread's word, a wave's segment, a tile and
the row limit, with masks that leave words empty or full, and with masks the GEMMs leave to ffnk_route (past the limit, off
16-byte alignment)."""
import ctypes

import pytest
import torch

from ffn_kernel_amd import _lib
from helpers import note

pytestmark = pytest.mark.gpu

MASKS = ("mixed", "spans", "visual", "text", "first", "last", "sparse")


def make_mask(kind, M):
    gen = torch.Generator().manual_seed(M)
    mask = torch.zeros(M, dtype=torch.bool)
    if kind == "mixed":
        mask = torch.rand(M, generator=gen) < 0.5
    elif kind == "spans":
        mask = (torch.arange(M) // 100) % 2 == 1
    elif kind == "visual":
        mask[:] = True
    elif kind == "first":
        mask[0] = True
    elif kind == "last":
        mask[-1] = True
    elif kind == "sparse":
        mask = torch.rand(M, generator=gen) < 0.02
    return mask


class _Part:
    def __init__(self, M, dev):
        self.perm = torch.full((M,), -1, dtype=torch.int32, device=dev)
        self.counts = torch.full((2,), -1, dtype=torch.int32, device=dev)
        self.struct = _lib.RoutingStruct(self.perm.data_ptr(), self.counts.data_ptr())


def _randn(shape, seed, dev):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * 0.05).bfloat16().to(dev)


def _check_same(name, call, mask, dev):
    """call(entry suffix, partition) -> output."""
    M = mask.numel()
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    want, got = _Part(M, dev), _Part(M, dev)
    _lib.check(lib.ffnk_route(mask.data_ptr(), M, want.perm.data_ptr(), want.counts.data_ptr(), stream), "ffnk_route")
    ref = call("routed", want)
    out = call("routing", got)
    plain = call(None, None)
    torch.cuda.synchronize()
    assert torch.equal(got.counts, want.counts), name
    assert torch.equal(got.perm, want.perm), name
    assert torch.equal(out, ref) and torch.equal(plain, ref), name


def _linear(x, W, mask, N):
    M, K = x.shape
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream

    def call(suffix, part):
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=x.device)
        ws = torch.empty(max(_lib.workspace_bytes(_lib.OP_LINEAR_FWD, M, K, N), 16), dtype=torch.uint8, device=x.device)
        args = (x.data_ptr(), K, W[0].data_ptr(), W[1].data_ptr(), 1, K, mask.data_ptr(), y.data_ptr(), N, M, K, N, ws.data_ptr(), ws.numel(), stream)
        fn = lib.ffnk_masked_linear_fwd if suffix is None else getattr(lib, f"ffnk_masked_linear_fwd_{suffix}")
        _lib.check(fn(*args) if part is None else fn(*args, ctypes.byref(part.struct)), "linear")
        return y

    return call


@pytest.mark.parametrize("tile", [-1, 0, 2, 3, 4, 6, 7, 16, 17])
@pytest.mark.parametrize("M", [65, 129, 257, 700, 2047, 2049, 4097, 8191, 8192, 8193])
def test_linear_forward_makes_the_partition(dev, M, tile):
    K, N = 192, 256
    x, W = _randn((M, K), 1, dev), [_randn((N, K), 2, dev), _randn((N, K), 3, dev)]
    old = _lib.load().ffnk_debug_force_tile(tile)
    try:
        for kind in MASKS:
            note(f"self-routed linear M={M} tile={tile} mask={kind}")
            mask = make_mask(kind, M).to(dev)
            _check_same(kind, _linear(x, W, mask, N), mask, dev)
    finally:
        _lib.load().ffnk_debug_force_tile(old)


# Launches with taller tiles among the others (csrc/gemm_sched.hpp: stretch_rows): a round of the chip and one M-tile more, the last
# M-tile of either modality spread over one taller tile, several and as many as there are, and of a modality with too few.
@pytest.mark.parametrize("tile,base,N,splits,K", [(2, 128, 8192, 1, 192), (6, 128, 8192, 1, 192), (6, 128, 4096, 2, 712),
                                                  (16, 192, 8192, 1, 192), (17, 160, 8192, 1, 192), (17, 160, 4096, 2, 712)])
def test_stretched_forward_makes_the_partition(dev, tile, base, N, splits, K):
    M = 8 * base
    x, W = _randn((M, K), 1, dev), [_randn((N, K), 2, dev), _randn((N, K), 3, dev)]
    old = _lib.load().ffnk_debug_force_tile(tile), _lib.load().ffnk_debug_force_splits(splits)
    try:
        for n_vis in (1, base, base + 1, 4 * base - 100, 4 * base - 1, 4 * base, 4 * base + 1, 4 * base + 33, 4 * base + 100, M - base - 1, M - 1, M):
            note(f"self-routed linear with taller tiles, tile={tile} splits={splits} {n_vis} of {M} visual")
            mask = (torch.randperm(M, generator=torch.Generator().manual_seed(n_vis)) < n_vis).to(dev)
            _check_same(str(n_vis), _linear(x, W, mask, N), mask, dev)
    finally:
        _lib.load().ffnk_debug_force_tile(old[0])
        _lib.load().ffnk_debug_force_splits(old[1])


def test_split_contraction_and_unaligned_mask(dev):
    M, K, N = 333, 4096, 256
    x, W = _randn((M, K), 1, dev), [_randn((N, K), 2, dev), _randn((N, K), 3, dev)]
    assert _lib.tile_config(_lib.OP_LINEAR_FWD, M, K, N)["split_k"] > 1
    for offset in (0, 16, 1, 7):
        for kind in MASKS:
            note(f"self-routed linear, K split, mask={kind} offset={offset}")
            room = torch.zeros(M + 64, dtype=torch.bool, device=dev)
            mask = room[offset:offset + M]
            mask.copy_(make_mask(kind, M))
            room[offset + M:] = True  # rows past the mask's end count as nothing
            _check_same(kind, _linear(x, W, mask, N), mask, dev)


@pytest.mark.parametrize("tile", [-1, 0, 1, 2, 3, 4, 6, 7])
@pytest.mark.parametrize("M", [65, 161, 300, 1411, 2048])
def test_ffn_forward_makes_the_partition(dev, M, tile):
    d, h = 256, 512
    x = _randn((M, d), 1, dev)
    up, down = [_randn((h, d), 2 + i, dev) for i in range(4)], [_randn((d, h), 6 + i, dev) for i in range(2)]
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    old = lib.ffnk_debug_force_tile(tile)

    def call(suffix, part):
        y = torch.full((M, d), float("nan"), dtype=torch.bfloat16, device=dev)
        ws = torch.empty(_lib.workspace_bytes(_lib.OP_FFN_FWD, M, d, h), dtype=torch.uint8, device=dev)
        head = (x.data_ptr(), d, *(w.data_ptr() for w in up), 1, d, *(w.data_ptr() for w in down), 1, h, mask.data_ptr(), y.data_ptr(), d)
        tail = (M, d, h, ws.data_ptr(), ws.numel(), stream)
        if part is None:
            _lib.check(lib.ffnk_masked_ffn_fwd(*head, *tail), "ffn")
        else:
            _lib.check(getattr(lib, f"ffnk_masked_ffn_fwd_{suffix}")(*head, None, 0, *tail, ctypes.byref(part.struct)), "ffn")
        return y

    try:
        for kind in MASKS:
            note(f"self-routed FFN M={M} tile={tile} mask={kind}")
            mask = make_mask(kind, M).to(dev)
            _check_same(kind, call, mask, dev)
    finally:
        lib.ffnk_debug_force_tile(old)


def test_decode_sizes_and_odd_layouts_leave_it_too(dev):
    """Paths that need no partition of their own still fill the caller's."""
    for M, K, N in ((40, 256, 256), (200, 36, 40)):
        note(f"linear M={M} K={K} N={N}: partition left by a path without one")
        x, W = _randn((M, K), 1, dev), [_randn((N, K), 2, dev), _randn((N, K), 3, dev)]
        mask = make_mask("mixed", M).to(dev)
        _check_same(f"{M}", _linear(x, W, mask, N), mask, dev)
