"""Products per expert in tiles of up to 256 places: runs around whole tiles and their halves and quarters, outputs that are no
multiple of a block, sums of one step of 64 and of several, against float64."""

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


COUNTS = [[1, 0, 257, 64], [512, 513, 31, 16], [65, 192, 193, 129], [4097, 0, 0, 3]]


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("K,n", [(64, 40), (128, 130), (192, 257), (320, 512)])
@pytest.mark.parametrize("form", ["plain", "float32", "squared", "glu"])
def test_tiles_of_256_places(ops, counts, K, n, form):
    E, M = len(counts), sum(counts)
    order = torch.randperm(M, generator=torch.Generator().manual_seed(1))
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[order].int().view(M, 1).contiguous().to(DEV)
    runs = ops.moe_sort(idx, E, 256)
    x, w = rnd((M, K), 2), rnd((E, 2 * n if form == "glu" else n, K), 3, 0.3)
    glu = (7.0, 1.702) if form == "glu" else None
    got = ops.grouped_linear(x, w, runs, True, glu=glu, squared=form == "squared",
                             out_dtype=torch.float32 if form == "float32" else None).double()
    place, expert = runs.place.long(), idx[:, 0].long()
    assert torch.equal(place.sort().values, torch.arange(M, device=DEV))
    want = torch.empty_like(got)
    slack = torch.zeros_like(got)                        # of float32 sums: K roundings of the sum of sizes
    for e in range(E):
        at = (expert == e).nonzero()[:, 0]
        y, size = x[at].double() @ w[e].double().T, (x[at].double().abs() @ w[e].double().abs().T) * K * 2.0 ** -24
        if form == "glu":
            g, u = y[:, :n].float().bfloat16().double().clamp(max=7.0), y[:, n:].float().bfloat16().double().clamp(-7.0, 7.0)
            size = 2.0 ** -7 * ((g.abs() + 1) * (u.abs() + 1))       # gate and up are rounded to bfloat16: one step either way
            y = g * torch.sigmoid(1.702 * g) * (u + 1)
        elif form == "squared":
            size = 2 * y.abs() * size + size * size
            y = y.clamp(min=0) ** 2
        want[place[at]], slack[place[at]] = y, size
    if form != "float32":
        slack = slack + 2.0 ** -8 * want.abs()
    assert ((got - want).abs() <= slack + 1e-6).all(), float(((got - want).abs() - slack).max())


def test_which_tiles(ops):
    x, w = rnd((64, 128), 1), rnd((4, 64, 128), 2)
    assert [ops._expert_tile(x, m * 4, 4, 128, 64, w) for m in (47, 48, 159, 160)] == [16, 128, 128, 256]
    assert ops._expert_tile(x, 4000, 4, 128, 72, w) == 128 and ops._expert_tile(x, 4000, 4, 128, 66, w) == 16
    shifted = torch.empty(w.numel() + 1, dtype=w.dtype, device=DEV)[1:].view_as(w)
    assert ops._expert_tile(x, 4000, 4, 128, 64, shifted) == 128


@pytest.mark.parametrize("top", [1, 2, 4, 8])
@pytest.mark.parametrize("N,d", [(1, 4), (3, 1020), (5, 1024), (7, 1028), (2, 2562), (300, 2560)])
@pytest.mark.parametrize("extra,skip", [(False, False), (True, False), (True, True)])
def test_weighted_sums_of_experts(ops, top, N, d, extra, skip):
    """Rows of whole and broken runs of four, one workgroup and several, with a shared expert behind a gate, and with
    pairs that stand for the token itself. ``top`` + 1 roundings of float32 at sums of the sizes are the bound."""
    from types import SimpleNamespace
    g = torch.Generator().manual_seed(d + top)
    place = torch.randperm(N * top, generator=g).int()
    if skip:
        place[::3] = -1
    y, weight = torch.randn((N * top, d), generator=g), torch.rand((N, top), generator=g)
    own, shared, gate = rnd((N, d), 5), rnd((N, d), 6), torch.randn((N, 3), generator=g)
    got = ops.moe_combine(y.to(DEV), SimpleNamespace(place=place.to(DEV)), weight.to(DEV), shared if extra else None,
                          gate.to(DEV)[:, 1] if extra else None, own if skip else None).double().cpu()
    rows = torch.where(place[:, None] >= 0, y[place.clamp(min=0).long()].double(), own.cpu().double().repeat_interleave(top, 0))
    terms = weight.double()[:, :, None] * rows.view(N, top, d)
    if extra:
        terms = torch.cat([terms, (gate[:, 1].double().sigmoid()[:, None] * shared.cpu().double())[:, None]], 1)
    # (the gate's sigmoid in float32: a few roundings of it)
    assert ((got - terms.sum(1)).abs() <= (top + 6) * 2.0 ** -24 * terms.abs().sum(1) + 1e-30).all()
