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
