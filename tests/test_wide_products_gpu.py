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


FORMS = [(8, 8, 0), (8, 8, 1), (6, 8, 0), (6, 8, 1), (5, 8, 0), (4, 8, 0), (4, 8, 1), (3, 8, 0), (2, 8, 0), (8, 4, 0), (8, 6, 0), (6, 6, 0),
         (8, 5, 0), (4, 6, 0), (5, 5, 0), (4, 5, 0), (4, 4, 0), (3, 5, 0)]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("M,N,K", [(65, 264, 64), (257, 1096, 320), (700, 3080, 448)])
def test_whole_and_partial_sums(ops, form, M, N, K):
    """Tiles with one row or a few columns, more tiles than an XCD has in a round, fewer and more steps than the rings hold, parts
    of unequal length. K roundings of float32 at the sum of sizes, and the result's own, are the bound."""
    x, w = rnd((M, K), 1), rnd((N, K), 2, 0.3)
    want, slack = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T * K * 2.0 ** -24 + 1e-6
    for parts in (1, 2, 3):
        if parts > K // 64:
            continue
        got = ops._wide_product(form + (parts,), x, w, torch.float32)
        assert ((got.double() - want).abs() <= slack).all()
        rounded = ops._wide_product(form + (parts,), x, w, torch.bfloat16)
        assert torch.equal(rounded, got.bfloat16())
        if parts > 1:
            sums = ops._wide_product(form + (parts,), x, w, torch.bfloat16, partial=True)
            assert sums.shape == (parts, M, N) and torch.equal(sum(sums[1:], sums[0]), got)


@pytest.mark.parametrize("form", [f for f in FORMS if f[1] % 4 == 0])
@pytest.mark.parametrize("M,ff,K", [(65, 144, 64), (300, 1552, 320)])
def test_activations_in_the_epilogue(ops, form, M, ff, K):
    """Gate and up rows that alternate by 16 or lie in halves; both products are rounded to bfloat16 (a step either way where a
    float32 sum lies near the middle), the activation's own error is below the result's rounding."""
    x, gate, up = rnd((M, K), 1), rnd((ff, K), 2, K ** -0.5), rnd((ff, K), 3, K ** -0.5)
    g, u = (x.double() @ t.double().T for t in (gate, up))
    apart = torch.cat([gate, up]).contiguous()
    mixed = torch.stack([gate.view(ff // 16, 16, K), up.view(ff // 16, 16, K)], 1).reshape(2 * ff, K).contiguous()
    gg, uu = (t.float().bfloat16().double() for t in (g, u))
    size = 2.0 ** -7 * (gg.abs() + 1) * (uu.abs() + 2)
    limit = 0.7
    want = {ops.WIDE_SILU: torch.nn.functional.silu(gg) * uu,
            ops.WIDE_GATED: gg.clamp(max=limit) * torch.sigmoid(1.702 * gg.clamp(max=limit)) * (uu.clamp(-limit, limit) + 1),
            ops.WIDE_GELU: torch.nn.functional.gelu(gg, approximate="tanh") * uu}
    for act, y in want.items():
        a = ops._wide_product(form + (1,), x, mixed, torch.bfloat16, act=act, gate=(limit, 1.702, 1.0))
        b = ops._wide_product(form + (1,), x, apart, torch.bfloat16, act=act, halves=True, gate=(limit, 1.702, 1.0))
        assert torch.equal(a, b) and ((a.double() - y).abs() <= size + 2.0 ** -8 * y.abs()).all(), act
    y = ops._wide_product(form + (1,), x, apart, torch.bfloat16, act=ops.WIDE_SQUARED)
    both = torch.cat([gg, uu], 1)
    assert ((y.double() - both.clamp(min=0) ** 2).abs() <= 2.0 ** -6 * both ** 2 + 1e-4).all()


def test_what_is_not_finite_stays_where_it_was(ops):
    """Infinities and NaN in a gate or an up row come out as the activation of plain rows has them."""
    M, ff, K = 70, 64, 64
    x, w = rnd((M, K), 1), rnd((2 * ff, K), 2, 0.1)
    x[3, 5], x[4, 6], x[5, 7] = float("inf"), float("nan"), -float("inf")
    both = torch.mm(x.float(), w.float().T).bfloat16()
    got = ops._wide_product((2, 8, 0, 1), x, w, torch.bfloat16, act=ops.WIDE_SILU, halves=True)
    want = ops.swiglu(both)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    got = ops._wide_product((2, 8, 0, 1), x, w, torch.bfloat16, act=ops.WIDE_GELU, halves=True)
    assert torch.equal(got.isnan(), ops.glu_gelu(both, ff).isnan())


def test_which_products_are_wide(ops):
    """Rows, outputs, operations and alignment decide; what the kernel does not take goes the way it went."""
    form = ops._wide_form
    assert form(64, 2560, 9728) is None and form(65, 2560, 9728) is not None and form(65, 248, 9728) is None
    # whole sums: from 1 billion operations on, but not from 7 to 15
    assert [form(m, 2560, 2560) is not None for m in (76, 77, 534, 535, 1144, 1145)] == [False, True, True, False, False, True]
    assert form(65, 2560, 2560, 0, True)[3] > 1
    assert form(2048, 2560, 2592) is None and form(2048, 2564, 2560) is None and form(65, 19456, 2560, ops.WIDE_SILU) is None
    x, w = rnd((70, 4096), 1), rnd((264, 4096), 2, 0.02)
    shifted = torch.empty(w.numel() + 1, dtype=w.dtype, device=DEV)[1:].view_as(w).copy_(w)
    for weight, name in ((w, "wide"), (shifted, "library")):
        ops.forms.clear()
        y = ops.linear(x, weight)
        assert ops.forms[name] == 1 and torch.allclose(y.double(), x.double() @ w.double().T, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("kind,rows", [("gated", 1024), ("gelu", 1024), ("squared", 512)])
def test_activated_products_where_they_are_long_enough(ops, kind, rows):
    x, w = rnd((4100, 1024), 1), rnd((rows, 1024), 2, 1024 ** -0.5)
    both = ops.linear(x, w)
    want = {"gated": lambda: ops.glu_clamped(both, 0.7, 1.702), "gelu": lambda: ops.glu_gelu(both, 512), "squared": lambda: ops.relu_squared(both)}[kind]()
    got = ops.linear_activated(x, w, kind, 0.7, 1.702)
    # a product whose float32 sum lies between two bfloat16 values may round to either: a step of gate and of up
    torch.testing.assert_close(got.float(), want.float(), atol=2e-2, rtol=2e-2)
    assert ops.linear_activated(x[:70].contiguous(), w, kind) is None      # 0.07 to 0.15 billion


@pytest.mark.parametrize("tiles", [205, 305, 405, 505, 605, 705, 805, 905, 308, 408, 508])
@pytest.mark.parametrize("M,N,K", [(1, 4, 64), (33, 81, 128), (145, 644, 192), (70, 1000, 832)])
def test_float32_products_whose_waves_share_k(ops, tiles, M, N, K):
    """One chunk per wave and several, an even and an odd number of them, a tile's first row or column alone, parts of K. K roundings
    of float32 at the sum of sizes are the bound."""
    x, w = (torch.randn(s, generator=torch.Generator().manual_seed(s[0])).to(DEV) for s in ((M, K), (N, K)))
    want, slack = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T * K * 2.0 ** -24 + 1e-12
    for splits in (1, 2, 3):
        if splits > 1 and (N % 4 or -(-(K // 64) // splits) * (splits - 1) >= K // 64):
            continue
        got = ops._linear_f32(x, w, torch.float32, False, tiles, splits)
        assert ((got.double() - want).abs() <= slack).all()
        assert torch.equal(ops._linear_f32(x, w, torch.bfloat16, False, tiles, splits), got.bfloat16())
        if splits > 1:
            parts = ops._linear_f32(x, w, torch.float32, True, tiles, splits)
            assert parts.shape == (splits, M, N) and torch.equal(sum(parts[1:], parts[0]), got)
