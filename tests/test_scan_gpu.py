"""The recurrences with a matrix state taken 64 tokens at a time, against float64 token by token and against the
walk: portions around whole chunks and runs of 16 tokens, sizes that are no multiple of a tile, decays of one, of
almost nothing and of zero, states that are not zero, and the chunks taken in several rounds."""

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16}


@pytest.fixture(scope="module")
def kernel_sets():
    from socrates_amd.kernels import HipKernels
    return {n: HipKernels(dt, DEV) for n, dt in DTYPES.items()}


def step_of(lengths):
    starts = torch.tensor([0] + lengths).cumsum(0)
    return SimpleNamespace(n_seqs=len(lengths), max_q_len=max(lengths), n_tokens=int(starts[-1]), seq_qstart=starts.int().to(DEV),
                           seq_rows=torch.arange(len(lengths)).flip(0).int().to(DEV), positions=torch.arange(int(starts[-1])).int().to(DEV))


def rnd(shape, dtype, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype).to(DEV)


def decays_of(shape, seed):
    """Most between 0.3 and 1; some 1, some 1e-30, some 0."""
    g = torch.Generator().manual_seed(seed)
    a = torch.rand(shape, generator=g) * 0.7 + 0.3
    for share, value in ((0.2, 1.0), (0.01, 1e-30), (0.01, 0.0)):
        a[torch.rand(shape, generator=g) < share] = value
    return a.to(DEV)


def walk64(ctx, q, k, v, a, S, bonus=None, take=None, skip=None):
    """q, k, a [N, H, D], v [N, H, Dv], S [rows, H, D, Dv], all float64; S is moved on in place."""
    out = torch.empty_like(v)
    starts, rows = ctx.seq_qstart.tolist(), ctx.seq_rows.tolist()
    for i, row in enumerate(rows):
        for n in range(starts[i], starts[i + 1]):
            add = k[n][:, :, None] * v[n][:, None]
            if bonus is None:
                S[row] = a[n][:, :, None] * S[row] + add
                out[n] = (q[n][:, None] @ S[row])[:, 0]
            else:
                out[n] = (q[n][:, None] @ (S[row] + bonus[:, :, None] * add))[:, 0]
                S[row] = a[n][:, :, None] * S[row] + add
    return out if skip is None else out + skip[:, None] * v


LENGTHS = [[64, 63, 1], [65, 16, 17, 200], [129], [256, 5], [7]]


def check(ops, call, want, S0, S1, slack=2e-7):
    """In chunks as close to float64 as the walk, or within a few roundings (2^-24 each) of the sums; the same in rounds."""
    got = {}
    for name, settings in (("walk", dict(scan_from=0)), ("chunks", dict(scan_from=1)), ("rounds", dict(scan_from=1, scan_scratch=1))):
        for s, v in settings.items():
            setattr(ops, s, v)
        try:
            state = S0.clone()
            ops.forms.clear()
            got[name] = (call(state), state)
            assert ops.forms["scan"] == (name != "walk")
        finally:
            for s in settings:
                delattr(ops, s)
    for i, exact in enumerate((want, S1)):
        def off(name):
            return float((got[name][i].double().reshape(exact.shape) - exact).norm() / exact.norm())
        assert off("chunks") <= 1.5 * off("walk") + slack, (off("chunks"), off("walk"))
        assert torch.equal(got["chunks"][i], got["rounds"][i])


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("H,D,Dv", [(2, 64, 64), (1, 128, 256), (3, 20, 33), (1, 100, 65)])
@pytest.mark.parametrize("kind", ["head", "channel", "prepared"])
@pytest.mark.parametrize("lead", [5, 0])
def test_linear_attention_in_chunks(kernel_sets, dtype, lengths, H, D, Dv, kind, lead):
    """``lead``: columns of a row before the queries; with 5 nothing starts on four elements, with none (and rows in steps of
    eight) everything may, up to an odd number of value columns beside one of ones."""
    ops, dt, ctx = kernel_sets[dtype], DTYPES[dtype], step_of(lengths)
    N = ctx.n_tokens
    x = rnd((N, lead + 2 * H * D + H * Dv + (0 if lead else -(2 * H * D + H * Dv) % 8)), dt, 1, 0.5)
    cols = (lead, lead + H * D, lead + 2 * H * D)
    q, k = (x[:, c:c + H * D].double().view(N, H, D) for c in cols[:2])
    v = x[:, cols[2]:cols[2] + H * Dv].double().view(N, H, Dv)
    S0 = rnd((len(lengths), 3 + H * D * Dv), torch.float32, 2)
    S = S0[:, 3:].double().view(-1, H, D, Dv).clone()
    if kind == "head":
        decays = decays_of((H,), 5)
        silu = torch.nn.functional.silu
        want = walk64(ctx, silu(q) * 0.3, silu(k), silu(v), decays.double()[None, :, None].expand(N, H, D), S)
        args, more = (0.3, True, decays, None, None, 1.0), {}
    elif kind == "channel":
        z, zb = rnd((N, H * D), torch.float32, 3, 8.0), rnd((H * D,), torch.float32, 4)
        a = torch.exp(torch.nn.functional.logsigmoid(z.double() + zb.double()) / 4.0).view(N, H, D)
        want = walk64(ctx, q * 0.3, k, v, a, S)
        args, more = (0.3, False, None, z, zb, 4.0), {}
    else:
        a = decays_of((N, H, D), 6)
        prepared = torch.stack([q.float(), k.float(), a], 1).view(N, 3, H * D).contiguous()
        ones = 1
        v = torch.cat([x[:, cols[2]:cols[2] + H * (Dv - 1)].double().view(N, H, Dv - 1), torch.ones(N, H, 1, dtype=torch.float64, device=DEV)], -1)
        want = walk64(ctx, q, k, v, a.double(), S)
        args, more = (1.0, False, None, None, None, 1.0), dict(prepared=prepared, ones=ones)

    def call(state):
        return ops.linear_attention(x, cols, H, D, Dv, *args, state, 3, ctx, **more)
    check(ops, call, want.reshape(N, -1), S0, torch.cat([S0[:, :3].double(), S.reshape(len(lengths), -1)], 1))


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("H,D", [(3, 64), (1, 128), (2, 36)])
def test_bonus_recurrence_in_chunks(kernel_sets, dtype, lengths, H, D):
    ops, dt, ctx = kernel_sets[dtype], DTYPES[dtype], step_of(lengths)
    N, C = ctx.n_tokens, H * D
    r, k, v = (rnd((N, C), dt, i, 0.5) for i in range(3))
    decay, bonus = decays_of((N, C), 7), rnd((H, D), torch.float32, 8)
    S0 = rnd((len(lengths), C * D), torch.float32, 9)
    S = S0.double().view(-1, H, D, D).clone()
    want = walk64(ctx, *(t.double().view(N, H, D) for t in (r, k, v, decay)), S, bonus=bonus.double())
    kept = ops.gated_group_norm
    ops.gated_group_norm = lambda raw, *a, **kw: raw           # the recurrence alone
    try:
        check(ops, lambda state: ops.wkv(r, k, v, decay, v, bonus, bonus.view(-1), 1e-5, H, state, 0, ctx), want.reshape(N, C), S0,
              S.reshape(len(lengths), -1))
    finally:
        ops.gated_group_norm = kept


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("H,P,Ns,G", [(4, 64, 128, 1), (2, 33, 20, 2), (6, 24, 64, 3)])
def test_step_size_recurrence_in_chunks(kernel_sets, dtype, lengths, H, P, Ns, G):
    ops, dt, ctx = kernel_sets[dtype], DTYPES[dtype], step_of(lengths)
    N = ctx.n_tokens
    xbc, raw = rnd((N, H * P + 2 * G * Ns), dt, 1, 0.5), rnd((N, H), torch.float32, 2, 2.0)
    bias, a_log, skip = rnd((H,), torch.float32, 3), rnd((H,), torch.float32, 4), rnd((H,), torch.float32, 5)
    step = torch.nn.functional.softplus(raw.double() + bias.double(), threshold=1e9)
    decay = torch.exp(-torch.exp(a_log.double()) * step)[..., None].expand(N, H, Ns)
    x = xbc[:, :H * P].double().view(N, H, P)
    B, C = (xbc[:, H * P + i * G * Ns:H * P + (i + 1) * G * Ns].double().view(N, G, Ns).repeat_interleave(H // G, 1) for i in range(2))
    S0 = rnd((len(lengths), H * Ns * P), torch.float32, 6)
    S = S0.double().view(-1, H, Ns, P).clone()
    want = walk64(ctx, C, B * step[..., None], x, decay, S, skip=skip.double())
    check(ops, lambda state: ops.ssd(xbc, raw, bias, a_log, skip, H, P, Ns, G, state, 0, ctx), want.reshape(N, -1), S0,
          S.reshape(len(lengths), -1))


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("H,D,Dv,rot", [(2, 128, 128, 128), (3, 20, 28, 12), (1, 48, 80, 0)])
def test_retention_in_chunks(kernel_sets, dtype, H, D, Dv, rot):
    ops, dt, ctx = kernel_sets[dtype], DTYPES[dtype], step_of([65, 16, 17, 200])
    N = ctx.n_tokens
    x = rnd((N, 2 * H * D + H * Dv), dt, 1, 0.5)
    inv_freq = (1e4 ** (-torch.arange(rot // 2).double() * 2 / max(rot, 1))).float().to(DEV) if rot else None
    decays = torch.tensor([0.9, 1.0, 0.0][:H], device=DEV)
    S0 = rnd((4, H * D * Dv), torch.float32, 2)
    S = S0.double().view(-1, H, D, Dv).clone()
    q, k = (x[:, i * H * D:(i + 1) * H * D].double().view(N, H, D) for i in range(2))
    if rot:
        angle = (ctx.positions.float()[:, None] * inv_freq[None]).double()[:, None]          # the angle itself is float32
        def turn(t):
            a, b = t[..., :rot // 2], t[..., rot // 2:rot]
            return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin(), t[..., rot:]], -1)
        q, k = turn(q), turn(k)
    v = x[:, 2 * H * D:].double().view(N, H, Dv)
    want = walk64(ctx, q, k * D ** -0.5, v, decays.double()[None, :, None].expand(N, H, D), S)
    check(ops, lambda state: ops.retention(x, (0, H * D, 2 * H * D), H, D, Dv, inv_freq, rot, D ** -0.5, decays, state, 0, ctx),
          want.reshape(N, -1), S0, S.reshape(4, -1))


def delta64(ctx, qk, v, gates, G, H, D, Dv, S0):
    """(results [N, H, Dv], states [rows, H, D, Dv]) of the gated delta rule in float64."""
    N = v.shape[0]
    S = S0.double().view(-1, H, Dv, D).transpose(2, 3).clone()
    want = torch.empty(N, H, Dv, dtype=torch.float64, device=DEV)
    starts, (g, beta) = ctx.seq_qstart.tolist(), gates.double().unbind(-1)
    q64, k64 = (t.double()[..., :D].repeat_interleave(H // G, 1) for t in qk.unbind(1))
    for i, row in enumerate(ctx.seq_rows.tolist()):
        for n in range(starts[i], starts[i + 1]):
            S[row] = g[n][:, None, None] * S[row]
            u = beta[n][:, None] * (v[n].double().view(H, Dv) - (k64[n][:, None] @ S[row])[:, 0])
            S[row] = S[row] + k64[n][:, :, None] * u[:, None]
            want[n] = (q64[n][:, None] @ S[row])[:, 0]
    return want, S


def delta_rule(ops, ctx, qk, v, gates, G, H, D, Dv, state):
    """The recurrence behind its preparation, in chunks where ``ops.scan_from`` says so."""
    from socrates_amd.kernels.common import _check, _ptr
    from ctypes import c_int
    N, Dp = v.shape[0], qk.shape[-1]
    out = torch.empty((N, H * Dv), device=DEV)
    stride = ops._state(state, 0, H * D * Dv, ctx)
    if ops._in_chunks(ctx, D):
        return ops._delta_scan(qk, v, gates, G, H, D, Dv, Dp, state, stride, 0, ctx, N, out)
    _check(ops._delta().soc_delta_walk(_ptr(qk), _ptr(v), _ptr(gates), c_int(G), c_int(H), c_int(D), c_int(Dv), c_int(Dp), _ptr(state),
                                       stride, c_int(0), _ptr(ctx.seq_qstart), _ptr(ctx.seq_rows), _ptr(out), c_int(ctx.n_seqs),
                                       c_int(ops.code), ops._stream()), "delta_walk")
    return out


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("G,H,D,Dv", [(1, 2, 128, 128), (2, 2, 64, 33), (3, 9, 20, 72), (1, 1, 100, 16)])
@pytest.mark.parametrize("alike", [False, True])
def test_delta_rule_in_chunks(kernel_sets, dtype, lengths, G, H, D, Dv, alike):
    """``alike``: keys that nearly repeat with a step size of almost one, so that a token's correction leans on all
    the ones before it in its chunk."""
    ops, dt, ctx = kernel_sets[dtype], DTYPES[dtype], step_of(lengths)
    N, Dp = ctx.n_tokens, (D + 63) // 64 * 64
    qk = torch.zeros(N, 2, G, Dp, device=DEV)
    qk[..., :D] = rnd((N, 2, G, D), torch.float32, 1) * (0.3 if alike else 1.0) + (rnd((1, 2, G, D), torch.float32, 2) if alike else 0.0)
    qk /= qk.norm(dim=-1, keepdim=True)
    v = rnd((N, H * Dv), dt, 3)
    g = decays_of((N, H), 4)
    beta = torch.rand((N, H), generator=torch.Generator().manual_seed(5)).to(DEV)
    if alike:
        g, beta = g.clamp(min=0.3), beta * 0.05 + 0.95
    gates = torch.stack([g, beta], -1).contiguous()
    S0 = rnd((len(lengths), H * D * Dv), torch.float32, 6)
    want, S = delta64(ctx, qk, v, gates, G, H, D, Dv, S0)

    def call(state):
        return delta_rule(ops, ctx, qk, v, gates, G, H, D, Dv, state)
    check(ops, call, want.reshape(N, -1), S0, S.transpose(2, 3).reshape(len(lengths), -1))


def in_earnest(ops, dt, kind, N):
    """(call, exact results, exact states, states before) of one sequence with the values that the layers meet: decays of a
    4B-sized model's heads, vectors behind activations, unit keys that have nothing in common or nearly repeat."""
    ctx, silu, D = step_of([N]), torch.nn.functional.silu, 128
    uniform = lambda shape, seed, lo, hi: (torch.rand(shape, generator=torch.Generator().manual_seed(seed)) * (hi - lo) + lo).to(DEV)
    f32 = torch.float32
    H = {"gated": 10, "prepared": 4, "bonus": 20, "step": 40}.get(kind, 10)
    if kind in ("retention", "lightning", "gated", "prepared"):
        Dv = 128 if kind in ("retention", "lightning") else 257 if kind == "prepared" else 256
        ones = int(kind == "prepared")
        x = rnd((N, 2 * H * D + H * (Dv - ones)), dt, 1, 0.5)
        cols = (0, H * D, 2 * H * D)
        q, k = (x[:, i * H * D:(i + 1) * H * D].double().view(N, H, D) for i in range(2))
        v = x[:, 2 * H * D:].double().view(N, H, Dv - ones)
        S0 = rnd((1, H * D * Dv), f32, 2)
        decays = torch.tensor([1.0 - 2.0 ** (-5 - 4 * h / H) for h in range(H)], device=DEV)
        a, scale = decays.double()[None, :, None].expand(N, H, D), D ** -0.5
        if kind == "retention":
            k = k * scale
            call = lambda state: ops.retention(x, cols, H, D, Dv, None, 0, scale, decays, state, 0, ctx)
        elif kind == "lightning":
            q, k, v = silu(q) * scale, silu(k), silu(v)
            call = lambda state: ops.linear_attention(x, cols, H, D, Dv, scale, True, decays, None, None, 1.0, state, 0, ctx)
        elif kind == "gated":
            z, zb = rnd((N, H * D), f32, 3), rnd((H * D,), f32, 4) + 2.0
            q, a = q * scale, torch.exp(torch.nn.functional.logsigmoid(z.double() + zb.double()) / 16.0).view(N, H, D)
            call = lambda state: ops.linear_attention(x, cols, H, D, Dv, scale, False, None, z, zb, 16.0, state, 0, ctx)
        else:
            gate = uniform((N, H, 1), 3, 0.8, 1.0).expand(N, H, D)
            prepared = torch.stack([q.float(), k.float(), gate], 1).view(N, 3, H * D).contiguous()
            a, v = gate.double(), torch.cat([v, torch.ones(N, H, 1, dtype=torch.float64, device=DEV)], -1)
            call = lambda state: ops.linear_attention(x, cols, H, D, Dv, 1.0, False, None, None, None, 1.0, state, 0, ctx,
                                                      prepared=prepared, ones=1)
        S = S0.double().view(1, H, D, Dv).clone()
        want = walk64(ctx, q, k, v, a, S)
    elif kind == "bonus":
        D = 64
        r, k, v = (rnd((N, H * D), dt, i, 0.5) for i in range(3))
        decay = torch.exp(-torch.exp(uniform((1, H * D), 3, -6.0, 0.0) + rnd((N, H * D), f32, 4, 0.3)))
        bonus, S0 = rnd((H, D), f32, 5, 0.5), rnd((1, H * D * D), f32, 2)
        S = S0.double().view(1, H, D, D).clone()
        want = walk64(ctx, *(t.double().view(N, H, D) for t in (r, k, v, decay)), S, bonus=bonus.double())
        call = lambda state: ops.wkv(r, k, v, decay, v, bonus, bonus.view(-1), 1e-5, H, state, 0, ctx)
    elif kind == "step":
        P = 64
        xbc, raw = silu(rnd((N, H * P + 2 * D), f32, 1)).to(dt), rnd((N, H), f32, 2)
        bias, a_log, skip = uniform((H,), 3, -6.9, -2.3).exp().expm1().log(), uniform((H,), 4, 1.0, 16.0).log(), 1.0 + rnd((H,), f32, 5, 0.05)
        step = torch.nn.functional.softplus(raw.double() + bias.double(), threshold=1e9)
        decay = torch.exp(-torch.exp(a_log.double()) * step)[..., None].expand(N, H, D)
        B, C = (xbc[:, H * P + i * D:H * P + (i + 1) * D].double().view(N, 1, D).expand(N, H, D) for i in range(2))
        S0 = rnd((1, H * D * P), f32, 2, 0.3)
        S = S0.double().view(1, H, D, P).clone()
        want = walk64(ctx, C, B * step[..., None], xbc[:, :H * P].double().view(N, H, P), decay, S, skip=skip.double())
        call = lambda state: ops.ssd(xbc, raw, bias, a_log, skip, H, P, D, 1, state, 0, ctx)
    else:
        y = rnd((N, 2, H, D), f32, 1)
        if kind == "delta":
            y, beta = silu(y), torch.sigmoid(rnd((N, H), f32, 5))
            g = torch.exp(-uniform((1, H), 4, 1.0, 16.0) * torch.exp(uniform((N, H), 6, -6.9, -2.3)))
        else:
            y, beta = 0.3 * y + rnd((1, 2, H, D), f32, 7), uniform((N, H), 5, 0.95, 1.0)
            g = uniform((N, H), 6, 0.3 if kind == "delta, alike" else 0.999, 1.0)
        qk = y / y.norm(dim=-1, keepdim=True)
        v, gates, S0 = rnd((N, H * D), dt, 3), torch.stack([g, beta], -1).contiguous(), rnd((1, H * D * D), f32, 2)
        call = lambda state: delta_rule(ops, ctx, qk, v, gates, H, H, D, D, state)
        want, S = delta64(ctx, qk, v, gates, H, H, D, D, S0)
        S = S.transpose(2, 3)
    return call, want.reshape(N, -1), S.reshape(1, -1), S0


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("kind", ["retention", "lightning", "gated", "prepared", "bonus", "step", "delta", "delta, alike", "delta, alike and kept"])
def test_no_further_off_than_the_walk(kernel_sets, dtype, kind):
    """1,000 tokens at real head sizes. Both errors are norms over a hundred thousand roundings and more, so they repeat to a
    few per cent; states right behind a nearly repeated key are at a single rounding either way (0.65e-7 against 0.6e-7)."""
    ops = kernel_sets[dtype]
    call, want, S, S0 = in_earnest(ops, DTYPES[dtype], kind, 1000)
    kept, off = ops.gated_group_norm, {}
    ops.gated_group_norm = lambda raw, *a, **kw: raw           # the recurrence alone
    try:
        for name, least in (("walk", 0), ("chunks", 1)):
            ops.scan_from, state = least, S0.clone()
            got = call(state)
            off[name] = [float((t.double().reshape(e.shape) - e).norm() / e.norm()) for t, e in ((got, want), (state, S))]
    finally:
        ops.gated_group_norm = kept
        del ops.scan_from
    for walk, chunks in zip(off["walk"], off["chunks"]):
        assert chunks <= 1.15 * walk, off


def test_from_which_portion_on(kernel_sets):
    ops = kernel_sets["float32"]
    assert [ops._in_chunks(SimpleNamespace(max_q_len=n), D) for n, D in ((1, 64), (159, 64), (160, 64), (4000, 128), (4000, 129))] == [
        False, False, True, True, False]
    delta = lambda lengths, D=128: ops._delta_in_chunks(SimpleNamespace(max_q_len=max(lengths)), sum(lengths), D, 20, 128)
    assert [delta([n]) for n in (1, 255, 256, 3000)] == [False, False, True, True] and not delta([3000], 129)
    assert [delta([n] * 2) for n in (256, 500, 1000)] == [False, True, True]             # side by side the walks cost little more
    assert not delta([500] * 3) and delta([1000] * 3) and not delta([1000] * 5) and delta([2000] + [1] * 20)


KINDS = ["retention", "lightning", "gated", "prepared", "bonus", "step", "delta"]


def layer(ops, dt, kind, ctx):
    """(call of one recurrence, its queries, keys, values and decays (views, None: a constant), elements of a row's state)."""
    N, H, D = ctx.n_tokens, 2, {"delta": 36, "bonus": 20}.get(kind, 72)
    f32 = torch.float32
    if kind in ("bonus", "delta"):
        q, k, v = (rnd((N, H * D), dt, i, 0.5) for i in range(3))
        decay = decays_of((N, H * D), 4)
    elif kind == "step":
        xbc, decay = rnd((N, H * 40 + 2 * D), dt, 1, 0.5), rnd((N, H), f32, 2)
        v, k, q = xbc[:, :H * 40], xbc[:, H * 40:H * 40 + D], xbc[:, H * 40 + D:]
    else:
        x, decay = rnd((N, 3 * H * D), dt, 1, 0.5), rnd((N, H * D), f32, 3)
        q, k, v = (x[:, i * H * D:(i + 1) * H * D] for i in range(3))
    if kind == "prepared":
        given = torch.stack([q.float(), k.float(), decays_of((N, H * D), 4)], 1).contiguous()
        q, k, decay = given.unbind(1)
    one, per_head = rnd((H,), f32, 6), torch.tensor([0.9, 0.5], device=DEV)
    if kind == "delta":
        x, decay = torch.cat([q, k, v], 1), rnd((N, 2 * H), f32, 3)          # the second half: logits of the decays
        q, k, v = (x[:, i * H * D:(i + 1) * H * D] for i in range(3))
        taps = rnd((3 * H * D, 4), f32, 5)
    calls = {"retention": lambda s: ops.retention(x, (0, H * D, 2 * H * D), H, D, D, None, 0, 0.1, per_head, s, 0, ctx),
             "lightning": lambda s: ops.linear_attention(x, (0, H * D, 2 * H * D), H, D, D, 0.1, True, per_head, None, None, 1.0, s, 0, ctx),
             "gated": lambda s: ops.linear_attention(x, (0, H * D, 2 * H * D), H, D, D, 0.1, False, None, decay, torch.zeros(H * D, device=DEV), 4.0, s, 0, ctx),
             "prepared": lambda s: ops.linear_attention(x, (0, 0, 2 * H * D), H, D, D + 1, 1.0, False, None, None, None, 1.0, s, 0, ctx, prepared=given, ones=1),
             "bonus": lambda s: ops.wkv(q, k, v, decay, v, rnd((H, D), f32, 8), rnd((H * D,), f32, 8), 1e-5, H, s, 0, ctx),
             "step": lambda s: ops.ssd(xbc, decay, one, one, one, H, 40, D, 1, s, 0, ctx),
             "delta": lambda s: ops.delta_rule(x, 0, H, H, D, D, taps, 1.0, 1e-6, decay, one, one, s, 0, 9 * H * D, ctx)}
    parts = {"q": q, "k": k, "v": v, "decay": None if kind in ("retention", "lightning") else decay}
    return calls[kind], parts, H * D * {"prepared": D + 1, "step": 40, "delta": D + 9}.get(kind, D)


# (token, what is not finite there): in the first and the last place of a run, in a run's middle, in the last token
BROKEN = {"results": [(3, "v", float("inf")), (79, "v", float("nan")), (200, "q", float("nan"))],
          "keys": [(37, "k", float("inf")), (95, "v", float("-inf")), (170, "k", float("nan"))],
          "steps": [(64, "decay", float("nan")), (81, "k", float("nan")), (130, "decay", float("nan"))]}


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("where", list(BROKEN))
@pytest.mark.parametrize("kind", KINDS)
def test_what_is_not_finite_touches_no_earlier_token(kernel_sets, dtype, where, kind):
    """Results and states that the walk leaves finite are finite in chunks too, and what they are without (the 16 sums of a run
    with such a value are added up in another order: 16 roundings of 2^-24 of the largest)."""
    ops, dt, ctx = kernel_sets[dtype], DTYPES[dtype], step_of([65, 16, 17, 200])
    call, parts, size = layer(ops, dt, kind, ctx)
    kept = ops.gated_group_norm
    ops.gated_group_norm = lambda raw, *a, **kw: raw

    def run(least):
        state = rnd((4, size), torch.float32, 9)
        ops.scan_from = ops.delta_scan_from = least
        return call(state), state
    try:
        sound = run(1)
        spoiled = 0
        for token, what, value in BROKEN[where]:
            if parts[what] is not None:
                parts[what][token, token % parts[what].shape[1]] = value
                spoiled += 1
        walk, chunks = run(0), run(1)
    finally:
        ops.gated_group_norm = kept
        del ops.scan_from, ops.delta_scan_from
    for a, b, c in zip(walk, chunks, sound):
        fine = a.isfinite()
        assert (not spoiled or not fine.all()) and fine.any()
        assert torch.equal(b.isfinite(), fine)
        assert float((b[fine] - c[fine]).abs().max()) <= 16 * 2.0 ** -24 * float(c.abs().max())


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("rounds", [False, True])
@pytest.mark.parametrize("kind", KINDS)
def test_short_sequences_walk_beside_long_ones(kernel_sets, dtype, rounds, kind):
    """Decoding rows and short portions before, between and behind portions in chunks, more than a wave looks at in one go:
    the short ones' results and states are the walk's bits, the long ones' those of a step that is in chunks whole."""
    lengths = [1] * 40 + [300, 1, 9] + [1] * 30 + [129, 1, 17, 400] + [1] * 3
    ops, dt, ctx = kernel_sets[dtype], DTYPES[dtype], step_of(lengths)
    call, _, size = layer(ops, dt, kind, ctx)
    kept, got = ops.gated_group_norm, {}
    ops.gated_group_norm = lambda raw, *a, **kw: raw
    if rounds:
        ops.scan_scratch = 1
    try:
        for name, least in (("walk", 0), ("whole", 1), ("split", 1)):
            ops.scan_from = ops.delta_scan_from = least
            if name == "split":
                ops._chunks_from = lambda *a, **kw: 100
                ctx.host = {"seq_qstart": ctx.seq_qstart.cpu().numpy()}
            state = rnd((len(lengths), size), torch.float32, 9)
            got[name] = call(state), state
    finally:
        ops.gated_group_norm = kept
        for n in ("scan_from", "delta_scan_from", "_chunks_from", "scan_scratch"):
            vars(ops).pop(n, None)
    starts, rows = ctx.seq_qstart.tolist(), ctx.seq_rows.tolist()
    for i, n in enumerate(lengths):
        like = got["whole" if n >= 100 else "walk"]
        assert torch.equal(got["split"][0][starts[i]:starts[i + 1]], like[0][starts[i]:starts[i + 1]]), (i, n)
        assert torch.equal(got["split"][1][rows[i]], like[1][rows[i]]), (i, n)
