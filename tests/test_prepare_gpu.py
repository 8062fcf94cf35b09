"""Heads of prompts prepared a token per workgroup, against the general kernels on the same rows (which a step of few tokens takes)."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from socrates_amd.kernels import HipKernels
    return HipKernels(torch.bfloat16, DEV)


def rnd(shape, seed, dtype=torch.bfloat16):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


def slot(pages, Hkv, BS, D, rows):
    k, v = (torch.zeros((pages, Hkv, BS, D), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    table = torch.randperm(pages, generator=torch.Generator().manual_seed(3)).int().view(rows, -1).contiguous().to(DEV)
    return SimpleNamespace(k=k, v=v, block_table=table, block_size=BS)


def same(a, b):
    """The sums of squares are added in another order: a result may round to the neighbouring bfloat16."""
    torch.testing.assert_close(a.float(), b.float(), atol=2.0 ** -9, rtol=2.0 ** -7)


def compare(call, N, Hkv, BS, D):
    """One call of all N tokens against calls of 200 (under the 256 from which a workgroup takes a token)."""
    pages = 2 * (-(-N // BS))
    whole, parts = slot(pages, Hkv, BS, D, 2), slot(pages, Hkv, BS, D, 2)
    q = call(slice(0, N), whole)
    p = torch.cat([call(slice(lo, min(N, lo + 200)), parts) for lo in range(0, N, 200)])
    same(q, p)
    same(whole.k, parts.k)
    same(whole.v, parts.v)
    assert whole.k.abs().sum() > 0 and whole.v.abs().sum() > 0


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Hq,Hkv,rot,norm,blend", [(1, 1, 0, False, False), (5, 3, 32, True, True), (32, 8, 64, True, True), (7, 7, 64, False, True)])
def test_turned_halves(ops, D, Hq, Hkv, rot, norm, blend):
    N, BS = 300, 7
    x = rnd((N, (Hq + 2 * Hkv) * D + 24), 1)
    gains = [1 + 0.2 * rnd((D,), s, torch.float32) for s in (2, 3)] if norm else [None, None]
    first, lam = rnd((N, Hkv * D + 8), 4), torch.tensor([0.3], device=DEV)
    freq = 10000.0 ** (-torch.arange(rot // 2, device=DEV) / max(1, rot // 2))
    pos, rows = (torch.arange(N, device=DEV, dtype=torch.int32) + 5) % N, (torch.arange(N, device=DEV, dtype=torch.int32) % 2)
    cols = (8, 8 + Hq * D, 16 + (Hq + Hkv) * D)
    compare(lambda at, to: ops.attn_prepare(x[at].contiguous(), cols, Hq, Hkv, D, D, D, *gains, 1e-6, freq, rot, pos[at].contiguous(), rows[at].contiguous(),
                                            to, first[at][:, 8:] if blend else None, lam if blend else None), N, Hkv, BS, D)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("norm", [None, "head", "whole"])
@pytest.mark.parametrize("Hq,Hkv,rot,bias,turned", [(1, 1, 0, False, False), (5, 3, 34, True, True), (32, 8, 64, True, False), (6, 2, 62, False, True)])
def test_turned_pairs(ops, D, norm, Hq, Hkv, rot, bias, turned):
    N, BS = 300, 16
    x = rnd((N, (Hq + 2 * Hkv) * D), 1)
    b = rnd((x.shape[1],), 5, torch.float32) if bias else None
    sizes = {None: (0, 0), "head": (D, D), "whole": (Hq * D, Hkv * D)}[norm]
    gains = [1 + 0.2 * rnd((s,), 2, torch.float32) if s else None for s in sizes]
    freq = 10000.0 ** (-torch.arange(rot // 2, device=DEV) / max(1, rot // 2))
    value_freq = 500.0 ** (-torch.arange(D // 2, device=DEV) / (D // 2)) if turned else None
    pos, rows = (torch.arange(N, device=DEV, dtype=torch.int32) + 5) % N, (torch.arange(N, device=DEV, dtype=torch.int32) % 2)
    cols = (0, Hq * D, (Hq + Hkv) * D)
    compare(lambda at, to: ops.window_prepare(x[at].contiguous(), cols, Hq, Hkv, D, D, D, b, *gains, norm, 1e-6, freq, rot, value_freq,
                                              pos[at].contiguous(), rows[at].contiguous(), to), N, Hkv, BS, D)


@pytest.mark.parametrize("N,H,P,Dv", [(1, 1, 8, 8), (3, 5, 128, 96), (40, 32, 128, 128)])
def test_gates_and_turns_of_eight(ops, N, H, P, Dv):
    o, g = rnd((N, H, P), 1), rnd((N, H + 3), 2)
    flat = o.view(N, H * P)
    got = ops.head_gate(flat, H, P, Dv, g[:, 1:1 + H]).view(N, H, Dv).float()
    want = o[..., :Dv].double() * torch.sigmoid(g[:, 1:1 + H].double())[..., None]
    torch.testing.assert_close(got.double(), want, atol=1e-6, rtol=2.0 ** -8)
    assert torch.equal(ops.head_gate(flat, H, P, Dv, None).view(N, H, Dv), o[..., :Dv])
    pos, freq = torch.arange(N, device=DEV, dtype=torch.int32) * 7, 500.0 ** (-torch.arange(Dv // 2, device=DEV) / (Dv // 2))
    got = ops.turn_back(flat, H, P, Dv, freq, pos).view(N, H, Dv // 2, 2).double()
    ang = (pos.float()[:, None] * freq[None]).double()[:, None]
    a, b = o[..., 0:Dv:2].double(), o[..., 1:Dv:2].double()
    want = torch.stack([a * ang.cos() + b * ang.sin(), b * ang.cos() - a * ang.sin()], -1)
    size = torch.stack([a.abs() + b.abs()] * 2, -1)
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * size).all()
