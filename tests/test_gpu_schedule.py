"""Tile orders and launch splits of the GEMMs, at the sizes where they can go wrong, against the row-select form in
double precision computed with torch on the GPU."""
import pytest
import torch

from ffn_kernel_amd import MaskedLinear, _lib
from ffn_kernel_amd.ops import masked_linear_backward
from helpers import assert_close, note

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
