"""Pozalorn on the GPU: every new HIP kernel against its stand-in from odd sizes and non-zero states, then the
kernels under the framework's step function, cache manager, scheduler and entry points, in float32 and
bfloat16, against the plain implementation in ``plain_pozalorn``: the same small models and cuts as on the
CPU, captured decode steps, greedy generation through ``Engine`` and the trace runner as a user starts it."""

import json
import subprocess
import sys
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import plain_pozalorn as plain
from helpers import make_runner, random_prompts, replay, trace_mixed, trace_portions, trace_tail_decode
from pozalorn_models import (BLOCK, CUTS, MODELS, STRETCH, attention, check_trace, compare, dense, drawn_model, gla, lightning, model,
                             oracle, parallel, read_folder, rot, row_errors, window, write_model)
from torch_kernels import TorchKernels

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parents[1]
DEV = "cuda:0"
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16}
# in units of the logits' spread per position; bfloat16: (every row, nine rows in ten)
TOL = {"float32": 3e-4, "bfloat16": (0.35, 0.06)}


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    base = tmp_path_factory.mktemp("pozalorn_gpu")
    return {name: write_model(base / name, made, seed=i + 1) for i, (name, made) in enumerate(MODELS.items())}


@pytest.fixture(scope="module")
def kernel_sets():
    from socrates_amd.kernels import HipKernels
    return {name: HipKernels(dt, DEV) for name, dt in DTYPES.items()}


def _close(got, want, dtype, what, scale=1.0):
    tol = dict(atol=2e-5 * scale, rtol=2e-5) if dtype == "float32" else dict(atol=2e-2 * scale, rtol=2e-2)
    torch.testing.assert_close(got.float().cpu(), want.float().cpu(), msg=lambda m: f"{what} ({dtype}): {m}", **tol)


def _ctx(lengths, rows, starts, dev):
    """A step's context for kernels that walk sequences: tokens of several sequences one after the other."""
    q = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    pos = np.concatenate([np.arange(s, s + n) for s, n in zip(starts, lengths)]).astype(np.int32)
    trow = np.concatenate([np.full(n, r) for r, n in zip(rows, lengths)]).astype(np.int32)
    t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int32, device=dev)      # noqa: E731
    return SimpleNamespace(n_seqs=len(lengths), n_tokens=int(q[-1]), seq_qstart=t(q), seq_rows=t(rows), positions=t(pos),
                           token_rows=t(trow), max_q_len=int(max(lengths)), seq_ctx=t([s + n for s, n in zip(starts, lengths)]),
                           max_ctx_len=int(max(s + n for s, n in zip(starts, lengths))))


# ---- each kernel against its stand-in ----------------------------------------------------------------------
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("H,D,Dv", [(3, 20, 28), (1, 48, 80), (4, 8, 8), (2, 64, 40), (2, 128, 64), (1, 200, 16), (6, 32, 32), (2, 128, 256)])
@pytest.mark.parametrize("lengths", [[9, 1, 2, 15], [37, 1, 2, 170]])
def test_linear_attention_kernel(kernel_sets, dtype, channel, H, D, Dv, lengths):
    """A decay per head over activated q, k, v and a decay per token and key channel, from a state that is not
    zero, several sequences of unequal length side by side, single tokens among them."""
    ops, dt = kernel_sets[dtype], DTYPES[dtype]
    ref = TorchKernels(dt, DEV)
    g = torch.Generator(device="cpu").manual_seed(H * D + Dv)
    rows, starts = [2, 0, 3, 1], [5, 300, 0, 41]
    ctx = _ctx(lengths, rows, starts, DEV)
    N, ld = ctx.n_tokens, 7 + H * (2 * D + 2 * Dv)
    x = (torch.randn(N, ld, generator=g) * 0.7).to(dt).to(DEV)
    cols = (7 + H * Dv, 7 + H * Dv + H * D, 7 + H * Dv + 2 * H * D)
    decays = None if channel else torch.tensor([0.9, 0.99, 1.0, 0.5, 0.8, 0.999][:H], dtype=torch.float32, device=DEV)
    z = (torch.randn(N, H * D, generator=g) * 2).to(DEV) if channel else None
    zb = (2 + torch.randn(H * D, generator=g)).to(DEV) if channel else None
    state = torch.randn(5, 3 + H * D * Dv, generator=g).to(DEV)
    s1, s2 = state.clone(), state.clone()
    got = ops.linear_attention(x, cols, H, D, Dv, D ** -0.5, not channel, decays, z, zb, 16.0, s1, 3, ctx)
    want = ref.linear_attention(x, cols, H, D, Dv, D ** -0.5, not channel, decays, z, zb, 16.0, s2, 3, ctx)
    assert got.dtype == torch.float32
    torch.testing.assert_close(got.cpu(), want.float().cpu(), atol=3e-4, rtol=3e-4)
    torch.testing.assert_close(s1.cpu(), s2.cpu(), atol=3e-4, rtol=3e-4)
    assert torch.equal(s1[4], state[4]) and torch.equal(s1[:, :3], state[:, :3])       # rows and columns that are not the step's


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("norm", ["head", "whole", None])
@pytest.mark.parametrize("Hq,Hkv,D,Dv,rotary,turned", [(4, 2, 24, 12, 8, True), (3, 1, 16, 16, 16, False), (2, 2, 40, 64, 0, True),
                                                       (8, 8, 48, 32, 24, False), (1, 1, 200, 256, 100, True), (8, 2, 64, 64, 64, True)])
def test_window_prepare_kernel(kernel_sets, dtype, norm, Hq, Hkv, D, Dv, rotary, turned):
    """Biases, norms per head or over the whole projection, the rotation of q and k over part of a head, the values
    turned over all of theirs, keys and values written to the tokens' places in pages of 4; then the result of a
    head cut back to the values' size and turned back."""
    from socrates_amd.cache.manager import PagedSlot
    from socrates_amd.config.specs import PairRopeSpec
    ops, dt = kernel_sets[dtype], DTYPES[dtype]
    ref = TorchKernels(dt, DEV)
    g = torch.Generator(device="cpu").manual_seed(D + Dv)
    P = (max(D, Dv) + 15) // 16 * 16
    lengths, rows, starts = [9, 1, 14], [1, 2, 0], [3, 17, 0]
    ctx = _ctx(lengths, rows, starts, DEV)
    N, ld = ctx.n_tokens, 5 + Hq * D + Hkv * (D + Dv) + 3
    x = torch.randn(N, ld, generator=g).to(dt).to(DEV)
    cols = (5, 5 + Hq * D, 5 + Hq * D + Hkv * D)
    bias = (0.5 * torch.randn(ld, generator=g)).to(DEV) if Hq != 3 else None
    sizes = {"head": (D, D), "whole": (Hq * D, Hkv * D), None: (1, 1)}[norm]
    qg, kg = [(1 + 0.3 * torch.randn(n, generator=g)).to(DEV) for n in sizes]
    inv_freq = None
    if rotary:
        inv_freq = torch.tensor(PairRopeSpec(dims=rotary, base=500.0, stretch=STRETCH).frequencies(), dtype=torch.float64).float().to(DEV)
    vfreq = (500.0 ** (-2.0 * torch.arange(Dv // 2, dtype=torch.float64) / Dv)).float().to(DEV) if turned else None
    table = torch.zeros(4, 8, dtype=torch.int32, device=DEV)
    table[:3, :6] = torch.arange(1, 19, dtype=torch.int32, device=DEV).view(3, 6)
    outs = []
    for o in (ops, ref):
        slot = PagedSlot(torch.full((19, Hkv, 4, P), 7.0, dtype=dt, device=DEV), torch.full((19, Hkv, 4, P), 7.0, dtype=dt, device=DEV),
                         table, 4, None)
        q = o.window_prepare(x, cols, Hq, Hkv, D, Dv, P, bias, qg if norm else None, kg if norm else None, norm, 1e-5, inv_freq, rotary,
                             vfreq, ctx.positions, ctx.token_rows, slot)
        outs.append((q, slot.k, slot.v))
    for a, b, what in zip(outs[0], outs[1], ("q", "keys", "values")):
        _close(a, b, dtype, what, scale=3.0)
    assert float(outs[0][1][0].float().abs().max()) == 7.0                  # the null page is nobody's
    o = torch.randn(N, Hq * P, generator=g).to(dt).to(DEV)
    for f in (vfreq, None):
        _close(ops.turn_back(o, Hq, P, Dv, f, ctx.positions), ref.turn_back(o, Hq, P, Dv, f, ctx.positions), dtype, "turned back")


def _pooled_slot(dt, Hkv, P, bs, per, rows, pages, g):
    from socrates_amd.cache.manager import PagedSlot
    table = torch.arange(1, 1 + rows * pages, dtype=torch.int32, device=DEV).view(rows, pages)
    table = torch.cat([table, torch.zeros(1, pages, dtype=torch.int32, device=DEV)]).contiguous()
    mpages = max(1, -(-(pages * bs // per) // bs))
    mtable = torch.arange(1, 1 + rows * mpages, dtype=torch.int32, device=DEV).view(rows, mpages).flip(0)
    mtable = torch.cat([mtable, torch.zeros(1, mpages, dtype=torch.int32, device=DEV)]).contiguous()
    k = (torch.randn(1 + rows * pages, Hkv, bs, P, generator=g) * 0.8).to(dt).to(DEV)
    v = torch.randn(1 + rows * pages, Hkv, bs, P, generator=g).to(dt).to(DEV)
    mk = torch.full((1 + rows * mpages, Hkv, bs, P), 5.0, dtype=dt, device=DEV)
    means = PagedSlot(mk, mk.clone(), mtable, bs, None)
    return PagedSlot(k, v, table, bs, None, pooled=means, pool=per)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("window,per,bs", [(5, 4, 4), (7, 3, 4), (40, 16, 16), (3, 1, 4), (6, 7, 4), (9, 5, 16), (88, 8, 16)])
def test_pooled_blocks_in_the_attention_kernels(kernel_sets, dtype, window, per, bs):
    """The means of the blocks that a step completes, from the pages (blocks that span pages, pages that span
    blocks), then the paged-attention kernel with the visible means in front of the window, against the stand-in:
    queries in front of, at and behind the position where a block comes into sight, with and without key splits,
    a long portion, portions behind cached tokens and single tokens."""
    ops, dt = kernel_sets[dtype], DTYPES[dtype]
    ref = TorchKernels(dt, DEV)
    g = torch.Generator(device="cpu").manual_seed(window * 10 + per)
    Hq, Hkv, P = 4, 2, 32
    pages = 256 // bs
    slot = _pooled_slot(dt, Hkv, P, bs, per, 4, pages, g)
    other = _pooled_slot(dt, Hkv, P, bs, per, 4, pages, torch.Generator(device="cpu").manual_seed(window * 10 + per))
    # the means of everything that came before this step, then this step's
    lengths, rows, starts = [200, 1, 1, 37], [0, 1, 2, 3], [0, 159, 2 * per - 1, 100]
    before = _ctx([s for s in starts if s], [r for r, s in zip(rows, starts) if s], [0 for s in starts if s], DEV)
    ctx = _ctx(lengths, rows, starts, DEV)
    for o, s in ((ops, slot), (ref, other)):
        o.pool_blocks(s, before)
        o.pool_blocks(s, ctx)
    _close(slot.pooled.k, other.pooled.k, dtype, "mean keys")
    _close(slot.pooled.v, other.pooled.v, dtype, "mean values")
    assert float(slot.pooled.k[0].float().abs().max()) == 5.0                 # the null page is nobody's
    q = torch.randn(ctx.n_tokens, Hq, P, generator=g).to(dt).to(DEV)
    for terms in ({"pooled": other}, {"pooled": other, "sinks": torch.tensor([0.5, -1.0, 2.0, 0.0], device=DEV)}):
        want = ref.paged_attention(q, other, ctx, 0.4, window, terms=terms)
        mine = dict(terms, pooled=slot)
        for splits in (None, (16, 16)):
            ops.attention_splits = splits
            try:
                got = ops.paged_attention(q, slot, ctx, 0.4, window, terms=mine)
            finally:
                ops.attention_splits = None
            _close(got, want, dtype, f"window {window}, blocks of {per}, splits {splits}")
    without = ref.paged_attention(q, other, ctx, 0.4, window)
    assert not torch.allclose(without.float(), want.float(), atol=0.05)


@pytest.mark.parametrize("row_tiles", [None, 1, 2, 32])
@pytest.mark.parametrize("window,per,P,G", [(40, 7, 32, 2), (100, 16, 64, 1), (64, 64, 128, 4), (7, 1, 48, 2), (500, 3, 64, 2), (33, 100, 32, 1),
                                           (88, 8, 64, 2)])
def test_prompt_attention_on_the_matrix_cores_sees_the_pooled_blocks(kernel_sets, window, per, P, G, row_tiles):
    """Long portions go to the kernel that shares its key tiles among four waves: the means of the blocks before the
    window in tiles of their own in front of the window's, with and without a learned sink per head, rows of several
    sequences (one from position 0, one behind 300 cached tokens, single tokens beside them), every form of the
    kernel, against the stand-in."""
    ops, dt = kernel_sets["bfloat16"], torch.bfloat16
    if row_tiles == 32 and P % 32:
        pytest.skip("32-row products take head sizes in steps of 32")
    ref = TorchKernels(dt, DEV)
    g = torch.Generator(device="cpu").manual_seed(window + per)
    Hkv, bs = 2, 16
    Hq = Hkv * G
    lengths, rows, starts = [700, 1, 230, 1, 17], [0, 1, 2, 3, 4], [0, 59, 300, 5, 140]
    ctx = _ctx(lengths, rows, starts, DEV)
    slot = _pooled_slot(dt, Hkv, P, bs, per, 5, 48, g)
    # the means of all complete blocks, whatever they hold: from the pages
    everything = _ctx([s + n for s, n in zip(starts, lengths)], rows, [0] * 5, DEV)
    ref.pool_blocks(slot, everything)
    q = torch.randn(ctx.n_tokens, Hq, P, generator=g).to(dt).to(DEV)
    sinks = torch.randn(Hq, generator=g).to(DEV) * 2
    for terms in ({"pooled": slot}, {"pooled": slot, "sinks": sinks}, {"sinks": sinks}):
        want = ref.paged_attention(q, slot, ctx, 0.3, window, terms=terms)
        ops.attention_row_tiles = row_tiles
        try:
            got = ops.paged_attention(q, slot, ctx, 0.3, window, terms=terms)
            kernel = ops.last_attention_kernel
        finally:
            ops.attention_row_tiles = None
        assert kernel[0] == ("workgroup" if row_tiles else kernel[0])
        _close(got, want, "bfloat16", f"window {window}, blocks of {per}, {sorted(terms)}, row tiles {row_tiles} ({kernel})")
    plain_window = ref.paged_attention(q, slot, ctx, 0.3, window)
    assert not torch.allclose(plain_window.float(), want.float(), atol=0.05)


@pytest.mark.parametrize("dtype", list(DTYPES))
def test_small_kernels(kernel_sets, dtype):
    ops, dt = kernel_sets[dtype], DTYPES[dtype]
    ref = TorchKernels(dt, DEV)
    g = torch.Generator(device="cpu").manual_seed(8)
    x = (torch.randn(33, 2 * 77 + 3, generator=g) * 2).to(dt).to(DEV)
    _close(ops.glu_gelu(x, 77), ref.glu_gelu(x, 77), dtype, "gelu gate")
    gain = (1 + 0.3 * torch.randn(77, generator=g)).to(DEV)
    bias = torch.randn(77, generator=g).to(DEV)
    for wide in (False, True):
        a = torch.randn(33, 77, generator=g).to(torch.float32 if wide else dt).to(DEV)
        b = torch.randn(33, 77, generator=g).to(dt if wide else torch.float32).to(DEV)
        for bb, bi in ((b, bias), (None, bias), (b, None)):
            got, want = ops.scaled_sum(a, 0.8, bb, 1.1, bi), ref.scaled_sum(a, 0.8, bb, 1.1, bi)
            assert got.dtype == torch.float32
            torch.testing.assert_close(got.cpu(), want.float().cpu(), atol=1e-5, rtol=1e-5)
        # a branch's result normed and added to the stream, with the cast for the next product
        r1 = torch.randn(33, 77, generator=g).to(DEV)
        r2 = r1.clone()
        _close(ops.norm_add_cast(r1, a, gain, 1e-5), ref.norm_add_cast(r2, a, gain, 1e-5), dtype, "norm, sum and cast")
        torch.testing.assert_close(r1.cpu(), r2.cpu(), atol=2e-5 if dtype == "float32" or wide else 2e-2, rtol=1e-5)
        assert ops.norm_add_cast(r1, a, gain, 1e-5, cast=False) is None
    # results by depth
    r = torch.randn(33, 77, generator=g).to(DEV)
    k1, c1 = ops.depth_begin(r.clone(), 4, cast=True)
    k2, c2 = ref.depth_begin(r.clone(), 4, cast=True)
    _close(c1, c2, dtype, "the stream, cast")
    for count, w in ((1, [0.3, -0.7]), (2, [0.1, 0.2, 0.5]), (3, [1.0, 0.0, -0.5, 0.25])):
        w = torch.tensor(w, device=DEV)
        a, b = torch.randn(33, 77, generator=g).to(DEV), None
        b = a.clone()
        _close(ops.depth_average(a, k1, count, w), ref.depth_average(b, k2, count, w), dtype, "weighted sum over depth")
        torch.testing.assert_close(a.cpu(), b.cpu(), atol=1e-5, rtol=1e-5)
        torch.testing.assert_close(k1[:count + 1].cpu(), k2[:count + 1].cpu(), atol=0, rtol=0)       # what has been filed so far
    # a branch's norm and sum with the weighted sum over depth behind it, in one kernel; rows of 77 and of 2,560 elements
    for d in (77, 2560):
        r = torch.randn(9, d, generator=g).to(DEV)
        gain_d = (1 + 0.3 * torch.randn(d, generator=g)).to(DEV)
        k1, k2 = ops.depth_begin(r.clone(), 5), ref.depth_begin(r.clone(), 5)
        for count, w in ((1, [0.3, -0.7]), (2, [0.1, 0.2, 0.5]), (3, [1.0, 0.0, -0.5, 0.25]), (4, [0.2, 0.2, 0.2, 0.2, 0.2])):
            w = torch.tensor(w, device=DEV)
            for wide in (False, True):
                y = torch.randn(9, d, generator=g).to(torch.float32 if wide else dt).to(DEV)
                a = torch.randn(9, d, generator=g).to(DEV)
                b = a.clone()
                got = ops.norm_add_cast(a, y, gain_d, 1e-5, cast=True, depth=(k1, count, w))
                want = ref.norm_add_cast(b, y, gain_d, 1e-5, cast=True, depth=(k2, count, w))
                _close(got, want, dtype, "norm, sum and the sum over depth")
                torch.testing.assert_close(a.cpu(), b.cpu(), atol=2e-5, rtol=1e-5)
                torch.testing.assert_close(k1[:count + 1].cpu(), k2[:count + 1].cpu(), atol=2e-5, rtol=1e-5)
    # the group norm with a sigmoid gate behind it
    y = torch.randn(33, 96, generator=g).to(DEV)
    zz = torch.randn(33, 96 + 5, generator=g).to(dt).to(DEV)
    gg = (1 + 0.3 * torch.randn(96, generator=g)).to(DEV)
    for groups in (1, 3):
        for sig in (True, False):
            _close(ops.gated_group_norm(y, zz, gg, groups, 1e-5, gate_first=False, sigmoid=sig),
                   ref.gated_group_norm(y, zz, gg, groups, 1e-5, gate_first=False, sigmoid=sig), dtype, "gated norm")


# ---- the models, cut in every way ------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("cut", list(CUTS))
@pytest.mark.parametrize("name", list(MODELS))
def test_cuts_match_the_plain_model(folders, kernel_sets, name, cut, dtype):
    cfg = MODELS[name][0]
    prompts = random_prompts([3, 41, 70, 26, 1, 58], cfg["vocab"], seed=7)
    pool = dict(num_blocks=4 * (-(-72 // BLOCK[name]))) if cut == "mixed" else {}
    check_trace(folders[name], kernel_sets[dtype], prompts, CUTS[cut](prompts), TOL[dtype], block_size=BLOCK[name], max_len=128,
                what=f"{name} {cut} {dtype}", graphs=4 if cut in ("tail", "mixed") else 0, **pool)


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("seed", range(24))
def test_drawn_configurations(tmp_path, kernel_sets, seed, dtype):
    """Configurations drawn from everything config.json can say, each under one way of cutting its requests,
    captured decode steps included. Such models can be touchy (a width of 24, a sharp softmax, a decay of one): in
    bfloat16 a request is judged against what rounding alone does to it, which the stand-in kernels in bfloat16 on
    the CPU say (they round where the HIP kernels round): within three times that, per request, for the worst row
    and for nine rows in ten."""
    made = drawn_model(seed)
    folder = write_model(tmp_path / "m", made, seed=100 + seed)
    prompts = random_prompts([23, 1, 40, 9], made[0]["vocab"], seed=seed)
    block = [2, 4, 16][seed % 3]
    cut = CUTS[["mixed", "portions", "tail"][seed % 3]]
    runner = make_runner(folder, kernel_sets[dtype], max_rows=4, max_len=64, block_size=block)
    if seed % 2:
        runner.enable_graphs(4)
    got = replay(runner, cut(prompts))
    want = oracle(folder, prompts)
    if dtype == "float32":
        for i in range(len(prompts)):
            compare(got[f"r{i}"], want[i], 1e-3, f"drawn {seed} {dtype} request {i}")
        return
    rounded = replay(make_runner(folder, TorchKernels(torch.bfloat16, "cpu"), max_rows=4, max_len=64, block_size=block), cut(prompts))
    for i in range(len(prompts)):
        mine, noise = row_errors(got[f"r{i}"], want[i]), row_errors(rounded[f"r{i}"], want[i])
        nine = max(1, int(0.9 * mine.numel()))
        assert float(mine.max()) <= 3 * float(noise.max()) + 0.03, f"drawn {seed} request {i}: {float(mine.max()):.3g} against {float(noise.max()):.3g}"
        assert float(mine.kthvalue(nine).values) <= 3 * float(noise.kthvalue(nine).values) + 0.03, f"drawn {seed} request {i}, nine rows in ten"


@pytest.mark.parametrize("dtype", list(DTYPES))
def test_a_wider_model_with_long_prompts(tmp_path, kernel_sets, dtype):
    """Width 320, five layers, keys of 80 beside values of 48 and of 32 beside 112, states of 64 x 96 and 128 x 32,
    windows of 100, 37 and 300 with blocks of 16 and 10, prompts of up to 700 tokens: decoded at the end, mixed,
    and in portions of 2 to 200 tokens, through captured decode steps."""
    made = model(320, 500, [parallel(window(10, 5, 80, 48, 100, rot(40, 40000.0, (3.0, 1.0, 4.0, 256)), scale=0.1),
                                     lightning(5, 64, 96, (0.9, 0.97, 0.99, 0.995, 0.999)), 0.7, 1.2),
                            gla(5, 64, 96, 12.0, rank=16),
                            attention(4, 1, 32, 112, size=37, pool=10, rotation=rot(32, 300000.0, (6.0, 1.0, 4.0, 128)), scale=0.2),
                            attention(5, 5, 64, 48, size=300, pool=16, rotation=rot(64, 1e6), scale=0.12),
                            gla(2, 128, 32, 4.0, rank=7)],
                 [dense(520), dense(100), None, dense(640), dense(320)])
    folder = write_model(tmp_path / "m", made, seed=5)
    prompts = random_prompts([700, 333, 64, 150], made[0]["vocab"], seed=6)
    want = oracle(folder, prompts)
    for name, steps in (("tail", trace_tail_decode(prompts, 40)), ("mixed", trace_mixed(prompts, seed=7)),
                        ("portions", trace_portions(prompts, seed=8, sizes=(2, 3, 64, 65, 128, 200)))):
        runner = make_runner(folder, kernel_sets[dtype], max_rows=4, max_len=768, block_size=16, num_blocks=4 * 48)
        runner.enable_graphs(4)
        got = replay(runner, steps)
        for i in range(len(prompts)):
            compare(got[f"r{i}"], want[i], TOL[dtype], f"{name} {dtype} request {i}")


@pytest.mark.parametrize("row_tiles", [1, 2, 32])
def test_long_portions_through_the_prompt_kernel_on_the_matrix_cores(tmp_path, kernel_sets, row_tiles):
    """bfloat16 steps whose long portions are sent to the prompt kernel on the matrix cores (by an override: models this
    small have too few rows for it otherwise), with the cache manager's own pages, tables and pages of means: a
    learned sink in one layer, pooled blocks in the other, whole prompts, portions behind cached tokens and single
    tokens beside them, against the plain model."""
    ops = kernel_sets["bfloat16"]
    made = model(128, 300, [parallel(window(6, 3, 64, 32, 80, rot(48, 20000.0, (3.0, 1.0, 8.0, 512)), scale=0.15),
                                     lightning(2, 32, 48, (0.9, 0.99)), 0.7, 1.2),
                            attention(6, 2, 32, 64, size=56, pool=24, rotation=rot(32, 300000.0, (6.0, 1.0, 4.0, 256)), scale=0.2),
                            gla(2, 32, 48, 8.0, rank=8)],
                 [dense(256), dense(192), None])
    folder = write_model(tmp_path / "m", made, seed=61)
    prompts = random_prompts([400, 150, 333], made[0]["vocab"], seed=62)
    want = oracle(folder, prompts)
    ops.attention_row_tiles = row_tiles
    try:
        for name, steps in (("whole", CUTS["whole"](prompts)), ("mixed", trace_mixed(prompts, seed=63)),
                            ("portions", trace_portions(prompts, seed=64, sizes=(17, 64, 65, 128, 200)))):
            runner = make_runner(folder, ops, max_rows=4, max_len=448, block_size=16)
            got = replay(runner, steps)
            if name != "mixed":
                assert ops.last_attention_kernel == ("workgroup", row_tiles)
            for i in range(len(prompts)):
                compare(got[f"r{i}"], want[i], TOL["bfloat16"], f"{name}, row tiles {row_tiles}, request {i}")
    finally:
        ops.attention_row_tiles = None


@pytest.mark.parametrize("dtype", list(DTYPES))
def test_edges_and_long_decoding(tmp_path, kernel_sets, dtype):
    """A window of 6 before which blocks of 4 come into sight, beside a window of 5 with sinks (in float32 under a
    sharp softmax, so the key at an edge often carries the weight; in bfloat16 a flatter one, where rounding moves
    little), pages of 4, 150 tokens decoded one by one from captured steps: the windows pass over decoded tokens,
    pages behind them come back, the means stay."""
    scale = 2.0 if dtype == "float32" else 0.4
    made = model(48, 50, [attention(2, 1, 16, 8, size=6, pool=4, rotation=rot(8, 1000.0, STRETCH), scale=scale),
                          parallel(window(4, 2, 12, 8, 5, rot(6, 1000.0), scale=scale), lightning(2, 16, 24, (0.99, 0.9)), 1.2, 0.5)],
                 [dense(64), None])
    folder = write_model(tmp_path / "m", made, seed=21)
    prompts = random_prompts([160], made[0]["vocab"], seed=22)
    want = oracle(folder, prompts)
    runner = make_runner(folder, kernel_sets[dtype], max_rows=2, max_len=192, block_size=4, num_blocks=8)
    runner.enable_graphs(2)
    got = replay(runner, trace_tail_decode(prompts, 150))
    compare(got["r0"], want[0], TOL[dtype], "decoded behind the windows")
    # the test sees an edge that is one off: the plain model with such constants is far outside the limits
    pcfg, w = read_folder(folder)
    for layer, key, other in ((0, "size", 7), (0, "pool", 3), (1, "size", 4)):
        m = pcfg["layers"][layer]["mixer"]
        mask = (m["left"] if layer else m)["mask"]
        was, mask[key] = mask[key], other
        with pytest.raises(AssertionError):
            compare(plain.forward(pcfg, w, prompts[0]).float(), want[0], TOL[dtype])
        mask[key] = was


@pytest.mark.parametrize("dtype", list(DTYPES))
def test_captured_decode_steps_equal_eager_ones(folders, kernel_sets, dtype):
    cfg = MODELS["A"][0]
    prompts = random_prompts([30, 45, 9], cfg["vocab"], seed=31)
    steps = trace_mixed(prompts, seed=32, max_live=3, prefill_frac=0.3)
    eager = replay(make_runner(folders["A"], kernel_sets[dtype], max_len=64, block_size=4), steps)
    runner = make_runner(folders["A"], kernel_sets[dtype], max_len=64, block_size=4)
    runner.enable_graphs(4)
    assert runner.graphs_refused is None and runner.model.capturable
    captured = replay(runner, steps)
    assert runner._graphs, "no decode step was captured"
    for rid in eager:
        torch.testing.assert_close(captured[rid], eager[rid], atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("name", ["A", "pooled", "B"])
def test_greedy_generation_through_the_engine(folders, name):
    """``Engine(folder)`` finds the model class by config.json; float32 greedy tokens are the plain model's,
    with more requests than rows, so rows, states and pages are used again."""
    from socrates_amd.engine import Engine
    cfg, w = read_folder(folders[name])
    prompts = random_prompts([5, 17, 33, 2, 21, 11], cfg["vocab"], seed=41)
    want = [plain.greedy(cfg, w, p, 8) for p in prompts]
    engine = Engine(str(folders[name]), device=DEV, dtype=torch.float32, max_batch=3, max_len=64, max_new_tokens=8,
                    block_size=BLOCK[name], chunk=16)
    assert engine.generate(prompts, max_new_tokens=8) == want
    engine.cache.check()


def test_command_line(tmp_path, folders):
    """``python -m socrates_amd.generate`` on a model folder, and with ``--random-weights`` on a configuration alone
    (it writes a seeded random model into --model; the rank of the decays' inner projections, which only a tensor's
    shape says, is made up): float32 greedy tokens are the plain model's."""
    cfg, w = read_folder(folders["A"])
    prompts = random_prompts([5, 17], cfg["vocab"], seed=2)
    want = [plain.greedy(cfg, w, p, 5) for p in prompts]
    cmd = [sys.executable, "-m", "socrates_amd.generate", "--model", str(folders["A"]), "--dtype", "float32",
           "--max-new-tokens", "5", "--max-len", "64", "--max-batch", "2", "--block-size", "4"]
    for p in prompts:
        cmd += ["--prompt-ids", ",".join(map(str, p))]
    proc = subprocess.run(cmd, capture_output=True, text=True, timeout=300, cwd=str(ROOT))
    assert proc.returncode == 0, proc.stderr[-2000:]
    lines = proc.stdout.strip().split("\n")
    shown = [l for i, l in enumerate(lines) if i > 0 and lines[i - 1].startswith("> ")]
    assert shown == [" ".join(map(str, x)) for x in want]
    (tmp_path / "config.json").write_text(json.dumps(MODELS["B"][0]))
    made = tmp_path / "made"
    cmd = [sys.executable, "-m", "socrates_amd.generate", "--model", str(made), "--random-weights", str(tmp_path / "config.json"),
           "--seed", "4", "--dtype", "float32", "--max-new-tokens", "4", "--max-len", "64", "--max-batch", "2",
           "--prompt-ids", "7,100,12,5,9"]
    proc = subprocess.run(cmd, capture_output=True, text=True, timeout=300, cwd=str(ROOT))
    assert proc.returncode == 0, proc.stderr[-2000:]
    cfg, w = read_folder(made)
    assert cfg == MODELS["B"][0] and w["l2.mix.a1"].shape[1] == cfg["width"]
    lines = proc.stdout.strip().split("\n")
    shown = [l for i, l in enumerate(lines) if i > 0 and lines[i - 1].startswith("> ")]
    assert shown == [" ".join(map(str, plain.greedy(cfg, w, [7, 100, 12, 5, 9], 4)))]


def test_trace_runner_on_a_model_folder(tmp_path, folders):
    cfg = MODELS["B"][0]
    prompts = random_prompts([70, 33, 100, 12, 64], cfg["vocab"], seed=51)
    want = oracle(folders["B"], prompts)
    steps = trace_mixed(prompts, seed=52)
    lines, wanted, fed = [], [], {}
    for n, (entries, ends) in enumerate(steps):
        lines.append(json.dumps({"step": n, "entries": [{"id": r, "tokens": t, "want": w} for r, t, w in entries], "end": ends}))
        here = []
        for r, t, w in entries:
            here.append((int(r[1:]), [fed.get(r, 0) + j for j in w]))
            fed[r] = fed.get(r, 0) + len(t)
        wanted.append(here)
    max_tokens = sum(-(-len(p) // 64) * 64 for p in sorted(prompts, key=len)[-4:])
    for dtype in DTYPES:
        out = tmp_path / dtype
        proc = subprocess.run([sys.executable, str(ROOT / "bin" / "trace_run"), "--model", str(folders["B"]), "--dtype", dtype,
                               "--out", str(out), "--max-tokens", str(max_tokens)], input="\n".join(lines) + "\n",
                              capture_output=True, text=True, timeout=600)
        assert proc.returncode == 0, proc.stderr[-2000:]
        assert proc.stdout.split("\n")[:-1] == [f"done {i}" for i in range(len(lines))]
        for n, here in enumerate(wanted):
            rows = sum(len(pos) for _, pos in here)
            if rows:
                got = torch.from_numpy(np.fromfile(out / f"{n}.f32", dtype="<f4").reshape(rows, cfg["vocab"]).copy())
                compare(got, torch.cat([want[i][pos] for i, pos in here]), TOL[dtype], f"step {n} {dtype}")


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("N,ff,ld", [(1, 8, 16), (3, 2056, 4112), (70, 72, 160), (5, 72, 150), (5, 76, 152)])
def test_gelu_gate_in_runs_of_eight(kernel_sets, dtype, N, ff, ld):
    """Rows in steps of eight elements and rows that are not, one workgroup and several, against float64."""
    ops, dt = kernel_sets[dtype], DTYPES[dtype]
    x = torch.randn((N, ld), generator=torch.Generator().manual_seed(ff)).to(dt).to(DEV)
    g, u = x[:, :ff].double(), x[:, ff:2 * ff].double()
    want = torch.nn.functional.gelu(g, approximate="tanh") * u
    # 1 + tanh loses the low bits where tanh is near -1: steps of 2^-24 of g u, a few of them
    slack = 8 * 2.0 ** -24 * (g * u).abs() + (2.0 ** -8 if dt == torch.bfloat16 else 0.0) * want.abs()
    assert ((ops.glu_gelu(x, ff).double() - want).abs() <= slack + 1e-30).all()


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("N,ff,ld", [(63, 8192, 16384), (64, 8192, 16384), (65, 8200, 16416), (64, 8192, 16388), (64, 8196, 16400)])
def test_gelu_gate_of_many_rows(kernel_sets, dtype, N, ff, ld):
    """Around the number of elements from which a lane takes eight, with rows that it may not read so; each row's bits are those
    of the row alone, which a lane per element makes."""
    ops = kernel_sets[dtype]
    x = torch.randn((N, ld), generator=torch.Generator().manual_seed(N)).to(DTYPES[dtype]).to(DEV)
    got = ops.glu_gelu(x, ff)
    for n in (0, 1, N // 2, N - 1):
        assert torch.equal(got[n], ops.glu_gelu(x[n:n + 1].contiguous(), ff)[0])
    g, u = x[:, :ff].double(), x[:, ff:2 * ff].double()
    want = torch.nn.functional.gelu(g, approximate="tanh") * u
    slack = 8 * 2.0 ** -24 * (g * u).abs() + (2.0 ** -8 if dtype == "bfloat16" else 0.0) * want.abs()
    assert ((got.double() - want).abs() <= slack + 1e-30).all()
