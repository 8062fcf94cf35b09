"""Products of many rows through the loop of wide.h: every number of blocks a tile can have, more and fewer steps than its rings
hold, ragged rows and columns, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from socrates_amd.kernels import HipKernels
    return HipKernels(torch.bfloat16, DEV)


def rnd(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).bfloat16().to(DEV)


@pytest.mark.parametrize("counts", [[33, 96, 97, 160], [161, 224, 225, 288], [289, 2305, 1, 32]])
@pytest.mark.parametrize("K", [64, 576])
@pytest.mark.parametrize("by_token", [True, False])
def test_places_in_blocks_of_32(ops, counts, K, by_token):
    """An expert's places are cut into tiles in blocks of 32; each tile's block count has a loop of its own. K roundings of
    float32 at the sum of sizes are the bound."""
    E, M, n = len(counts), sum(counts), 264
    order = torch.randperm(M, generator=torch.Generator().manual_seed(1))
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[order].int().view(M, 1).contiguous().to(DEV)
    runs = ops.moe_sort(idx, E, 256)
    x, w = rnd((M, K), 2), rnd((E, n, K), 3, 0.3)
    got = ops.grouped_linear(x, w, runs, by_token, out_dtype=torch.float32).double()
    place, expert = runs.place.long(), idx[:, 0].long()
    for e in range(E):
        at = (expert == e).nonzero()[:, 0]
        rows = (x[at] if by_token else x[place[at]]).double()
        slack = rows.abs() @ w[e].double().abs().T * K * 2.0 ** -24
        assert ((got[place[at]] - rows @ w[e].double().T).abs() <= slack + 1e-6).all()


def test_short_sums_keep_smaller_tiles(ops):
    """Tiles of 256 from 14 places per expert where both sums have 512 terms, from 160 otherwise."""
    x = rnd((64, 512), 1)
    for d, ff, m, tile in ((512, 512, 13, 16), (512, 512, 14, 256), (512, 448, 47, 16), (512, 448, 48, 128), (512, 448, 160, 256)):
        assert ops._expert_tile(x, m * 4, 4, d, ff, rnd((4, 2 * ff, d), 2)) == tile
