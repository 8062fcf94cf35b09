"""Prompt attention with 32 rows per wave in tiles of 64 keys: every head size it is built for, pages of any size, portions that
start anywhere, windows, kept first keys, a soft cap, against float64."""

import math
from ctypes import c_float, c_int

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from socrates_amd.kernels import HipKernels
    return HipKernels(torch.bfloat16, DEV)


@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("BS", [5, 8, 64])
@pytest.mark.parametrize("start,T,window,keep,cap", [(0, 1, 0, 0, 0.0), (0, 130, 0, 0, 0.0), (63, 97, 0, 0, 3.0), (200, 70, 90, 0, 0.0),
                                                     (300, 66, 65, 7, 0.0), (70, 140, -64, 0, 0.0)])
def test_tiles_of_64_keys(ops, D, BS, start, T, window, keep, cap):
    Hkv, G = 2, 3                                        # three heads in a group of four rows
    Hq, n = Hkv * G, start + T
    pages = -(-n // BS)
    gen = torch.Generator().manual_seed(D + BS + T)
    q = torch.randn((T, Hq, D), generator=gen).bfloat16().to(DEV)
    k, v = ((torch.randn((pages + 2, Hkv, BS, D), generator=gen)).bfloat16().to(DEV) for _ in range(2))
    order = torch.randperm(pages, generator=gen).int().to(DEV) + 2
    k[0], v[0], k[1], v[1] = (float("nan") for _ in range(4))     # pages of no row
    rows = torch.zeros(T, dtype=torch.int32, device=DEV)
    positions = torch.arange(start, n, dtype=torch.int32, device=DEV)
    kk = k[order.long()].permute(1, 0, 2, 3).reshape(Hkv, pages * BS, D)[:, :n].double()
    vv = v[order.long()].permute(1, 0, 2, 3).reshape(Hkv, pages * BS, D)[:, :n].double()
    for pool in (k, v):                                  # what lies behind the last token is not read as a value
        pool[order[-1].long(), :, (n - 1) % BS + 1:] = float("nan")
    i, j = torch.arange(start, n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    seen = j <= i
    if window > 0:
        seen = seen & ((i - j < window) | (j < keep))
    elif window < 0:
        seen = seen & (i // -window == j // -window)
    s = torch.einsum("thd,hjd->htj", q.double(), kk.repeat_interleave(G, 0)) * D ** -0.5
    if cap:
        s = cap * torch.tanh(s / cap)
    p = torch.softmax(s.masked_fill(~seen, -math.inf), -1)
    values = vv.repeat_interleave(G, 0)
    want = (p @ values).transpose(0, 1)
    # weights are rounded to bfloat16 before the second product (scores carry float32 sums of D terms, exponentials a unit in the
    # last place), the result once more
    slack = ((2.0 ** -8 + 2e-5 * D ** 0.5) * (p @ values.abs()).transpose(0, 1) + 2.0 ** -8 * want.abs()) + 1e-6
    lib = ops._attention_lib(D)
    tokens = 32                                          # 4 waves of 32 rows, four rows a token
    blocks = torch.tensor([[t, min(tokens, T - t)] for t in range(0, T, tokens)], dtype=torch.int32, device=DEV)
    for form in (32, 64):
        if form == 64 and keep:
            continue                                     # refused: no kept keys with key halves
        out = torch.full_like(q, float("nan"))
        from socrates_amd.kernels.common import _ptr
        err = lib.soc_paged_attention_prefill(
            _ptr(q), _ptr(k), _ptr(v), _ptr(order), c_int(pages), _ptr(rows), _ptr(positions), _ptr(blocks), c_int(len(blocks)),
            _ptr(out), c_int(T), c_int(Hq), c_int(Hkv), c_int(BS), c_float(D ** -0.5), c_int(window), c_int(form), c_int(2),
            c_int(keep), c_int(0), None, None, None, None, c_int(0), c_int(0), c_float(cap), ops._stream())
        assert err == 0 and ((out.double() - want).abs() <= slack).all(), (form, float(((out.double() - want).abs() - slack).max()))


def test_which_form_a_portion_takes(ops):
    """512 tokens of eight kv heads are 128 workgroups of 32 rows a wave: keys in two halves; fewer take 16 rows a wave or key
    splits, kept first keys four waves from 256 workgroups on."""
    from types import SimpleNamespace

    import numpy as np
    Hkv, G, D, BS = 8, 4, 128, 16
    for T, want in ((511, None), (512, ("workgroup", 64)), (3071, ("workgroup", 64)), (3072, ("workgroup", 32))):
        pages = -(-T // BS)
        q = torch.randn((T, Hkv * G, D), generator=torch.Generator().manual_seed(1)).bfloat16().to(DEV)
        k, v = (torch.randn((pages, Hkv, BS, D), generator=torch.Generator().manual_seed(s)).bfloat16().to(DEV) for s in (2, 3))
        table = torch.arange(pages, dtype=torch.int32, device=DEV)[None]
        slot = SimpleNamespace(k=k, v=v, block_table=table, block_size=BS)
        starts = torch.tensor([0, T], dtype=torch.int32)
        ctx = SimpleNamespace(token_rows=torch.zeros(T, dtype=torch.int32, device=DEV), positions=torch.arange(T, dtype=torch.int32, device=DEV),
                              max_ctx_len=T, max_q_len=T, n_seqs=1, seq_qstart=starts.to(DEV),
                              host={"seq_qstart": np.array([0, T], dtype=np.int32)})
        out = ops.paged_attention(q, slot, ctx, D ** -0.5)
        assert (ops.last_attention_kernel == want) if want else ops.last_attention_kernel != ("workgroup", 64), (T, ops.last_attention_kernel)
        i = torch.tensor([0, 1, T // 2, T - 1], device=DEV)
        kk, vv = (t.permute(1, 0, 2, 3).reshape(Hkv, -1, D)[:, :T].double().repeat_interleave(G, 0) for t in (k, v))
        s = (torch.einsum("thd,hjd->htj", q[i].double(), kk) * D ** -0.5).masked_fill(torch.arange(T, device=DEV)[None] > i[:, None], -math.inf)
        expect = (torch.softmax(s, -1) @ vv).transpose(0, 1)
        torch.testing.assert_close(out.view(T, -1, D)[i].double(), expect, atol=2e-2, rtol=2e-2)
