"""The steps that a program on this engine has it run, one case each, for timing and for checking.

A pass is one call of ``ModelRunner.step``: the call behind ``Engine.step``, ``Engine.generate`` and
``bin/trace_run``. ``mode`` says what the step holds: whole prompts (``prefill``), one further token of every
request behind its context (``decode``, replayed from a captured graph as the engine does), or one portion of a
prompt beside decoding rows (``mixed``). A decoding row is put back by one token after its pass, so that every
pass runs the same positions. Models have the layer sizes of the presets and of the benchmark, some with fewer
layers; the weights are random with the spread that such weights have after training where that matters (decays,
step sizes, routers that are sure of their choice).

``exact`` computes the same logits in float64 with plain torch operations, whole sequences from position 0.
"""

import math
import zlib

import torch

F64 = torch.float64
DEVICE = "cuda:0"
VOCAB = 151936
CLUSTERS = 32        # kinds of tokens that routed models tell apart
POSITIONS = 4096     # learned positions of the model that has them


def listed():
    return [
        # one user, one chat: every token waits for the whole model
        {"name": "decode_1", "model": "qwen3-4b", "layers": 36, "dtype": "bfloat16", "mode": "decode", "rows": 1, "context": 700},
        # the benchmark's headline: 8 requests behind 2,048 tokens
        {"name": "decode_8", "model": "qwen3-4b", "layers": 36, "dtype": "bfloat16", "mode": "decode", "rows": 8, "context": 2048},
        # a full server: 64 requests of uneven lengths
        {"name": "decode_64", "model": "qwen3-4b", "layers": 12, "dtype": "bfloat16", "mode": "decode", "rows": 64, "context": 2011},
        # few requests behind long documents: the cache is most of what is read
        {"name": "decode_long", "model": "qwen3-4b", "layers": 12, "dtype": "bfloat16", "mode": "decode", "rows": 3, "context": 15000},
        # one prompt of 2,048 tokens in one step, the benchmark's prefill
        {"name": "prefill_2048", "model": "qwen3-4b", "layers": 36, "dtype": "bfloat16", "mode": "prefill", "rows": 1, "context": 2048},
        # the serving workload: a portion of a prompt beside decoding rows, at the larger model's layer sizes
        {"name": "mixed_50", "model": "qwen3-8b", "layers": 12, "dtype": "bfloat16", "mode": "mixed", "rows": 50, "context": 1500, "portion": 1981},
        # short prompts together, in the float32 mode that results are compared in
        {"name": "short_float32", "model": "qwen3-4b", "layers": 4, "dtype": "float32", "mode": "prefill", "rows": 3, "context": 61},
        # prompts of the architectures with recurrent layers: time mixing, state space and latent attention
        {"name": "mitisun_prefill", "model": "mitisun", "layers": 6, "dtype": "bfloat16", "mode": "prefill", "rows": 1, "context": 2048},
        # retention, windowed attention and routed experts, uneven prompts in one step
        {"name": "tedulorn_prefill", "model": "tedulorn", "layers": 6, "dtype": "bfloat16", "mode": "prefill", "rows": 3, "context": 1100},
        # gated linear and lightning attention
        {"name": "pozalorn_prefill", "model": "pozalorn", "layers": 8, "dtype": "bfloat16", "mode": "prefill", "rows": 1, "context": 2048},
        # the gated delta rule beside chunked attention, a long prompt
        {"name": "nebutar_prefill", "model": "nebutar", "layers": 4, "dtype": "bfloat16", "mode": "prefill", "rows": 1, "context": 3000},
        # decoding with states, windows and experts
        {"name": "tedulorn_decode", "model": "tedulorn", "layers": 6, "dtype": "bfloat16", "mode": "decode", "rows": 8, "context": 1500},
    ]


def draw(rng):
    def log_uniform(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice(["qwen3-4b", "qwen3-4b", "qwen3-4b", "qwen3-8b", "mitisun", "tedulorn", "pozalorn", "nebutar"])
    layers = {"qwen3-4b": 12, "qwen3-8b": 12, "mitisun": 6, "tedulorn": 6, "pozalorn": 8, "nebutar": 4}[model]
    case = {"model": model, "layers": layers, "dtype": "bfloat16"}
    if model.startswith("qwen3"):
        case["mode"] = rng.choice(["decode", "decode", "prefill", "mixed"])
        if case["mode"] == "prefill" and rng.random() < 0.25:
            case["dtype"], case["layers"] = "float32", 4
    else:
        case["mode"] = rng.choice(["prefill", "prefill", "decode"])
    if case["mode"] == "decode":
        case["rows"] = log_uniform(1, 64 if model.startswith("qwen3") else 16)
        case["context"] = log_uniform(20, max(64, min(15000 if model.startswith("qwen3") else 2500, 60000 // case["rows"])))
    elif case["mode"] == "prefill":
        case["rows"] = rng.choice([1, 1, 2, 3, 5])
        longest = 200 if case["dtype"] == "float32" else 3000
        case["context"] = log_uniform(8, longest // (1 if case["rows"] == 1 else 2))
    else:
        case["rows"] = log_uniform(2, 60)
        case["context"] = log_uniform(100, 2000)
        case["portion"] = log_uniform(16, 2000)
    return case


# ---- models ------------------------------------------------------------------------------------------
def _qwen3(preset, layers):
    import json

    from socrates_amd.config import preset_path
    return dict(json.loads(preset_path(preset).read_text()), num_hidden_layers=layers)


def _mitisun(layers):
    kinds = [{"type": "wkv", "mixer": {"heads": 40, "dim": 64, "decay_rank": 64}},
             {"type": "mamba2", "mixer": {"heads": 80, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}},
             {"type": "latent_attention", "mixer": {"heads": 20, "dim": 128, "rot_dim": 32, "vdim": 128, "kv_rank": 96, "q_rank": 640,
                                                    "scale": 160 ** -0.5, "rot": {"base": 10000.0, "dims": 32}, "mask": {"size": 1024}}}]
    out = [{"type": kinds[i % 3]["type"], "mixer": dict(kinds[i % 3]["mixer"]), "mlp": {"kind": "dense", "ff": 9728, "limit": 7.0}}
           for i in range(layers)]
    for i in range(5, layers, 6):
        out[i]["mixer"]["kv_from"] = i - 3
    return {"architecture": "Mitisun", "vocab": VOCAB, "width": 2560, "layers": out, "norm": {"eps": 1e-6}, "residual_mult": 0.5}


def _tedulorn(layers):
    attention = {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": {"base": 1000000.0, "dims": 64},
                 "mask": {"size": 1024, "keep_first": 4}, "v_mix": True}
    retention = {"heads": 20, "dim": 128, "vdim": 128, "rot": {"base": 10000.0, "dims": 128},
                 "decay": [1.0 - 2.0 ** (-5 - 4 * h / 20) for h in range(20)]}
    moe = {"kind": "moe", "expert": {"ff": 2432, "limit": 7.0}, "shared": {"ff": 2432, "limit": 7.0},
           "router": {"experts": 32, "top": 4, "groups": {"count": 4, "keep": 2}}}
    out = [{"type": "retention" if i % 3 == 2 else "attention", "mixer": dict(retention if i % 3 == 2 else attention),
            "mlp": {"kind": "dense", "ff": 9728} if i == 0 else moe} for i in range(layers)]
    return {"architecture": "Tedulorn", "vocab": VOCAB, "width": 2560, "layers": out, "norm": {"eps": 1e-6},
            "embedding": {"scale": 50.0}, "token_side": {"dim": 64}}


def _pozalorn(layers):
    rot = {"base": 1000000.0, "dims": 128, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}
    left = {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": rot, "mask": {"size": 1024}}
    right = {"heads": 20, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-5 - 4 * h / 20) for h in range(20)]}
    gla = {"type": "gla", "mixer": {"heads": 10, "dim": 128, "vdim": 256, "tau": 16.0}}
    kinds = [{"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 0.7, "right_scale": 0.7}}, gla, gla,
             {"type": "attention", "mixer": dict(left, mask={"size": 1024, "pool": 64})}]
    out = [{"type": kinds[i % 4]["type"], "mixer": dict(kinds[i % 4]["mixer"]), "mlp": {"kind": "dense", "ff": 9728}} for i in range(layers)]
    return {"architecture": "Pozalorn", "vocab": VOCAB, "width": 2560, "layers": out, "norm": {"eps": 1e-6}}


def _nebutar(layers):
    layer = {"type": "parallel",
             "mixer": {"left": {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "softcap": 50.0, "mask": {"size": 1024}},
                       "right": {"heads": 20, "kv_heads": 10, "dim": 128, "vdim": 128, "conv": 4}, "left_scale": 0.7, "right_scale": 0.7},
             "mlp": {"kind": "moe", "expert": {"ff": 2432}, "router": {"experts": 32, "identity": 4, "top": 4}}}
    return {"architecture": "Nebutar", "vocab": VOCAB, "width": 2560, "layers": [layer] * layers, "norm": {"eps": 1e-6},
            "embedding": {"scale": 50.0}, "max_positions": POSITIONS, "streams": 4}


def _config(case):
    if case["model"].startswith("qwen3"):
        return _qwen3(case["model"], case["layers"])
    return {"mitisun": _mitisun, "tedulorn": _tedulorn, "pozalorn": _pozalorn, "nebutar": _nebutar}[case["model"]](case["layers"])


# ---- weights: each tensor from its name and the seed ------------------------------------------------------
class _Weights:
    def __init__(self, case, seed):
        self.seed, self.dtype = seed, getattr(torch, case["dtype"])
        self.model, self.layers = case["model"], case["layers"]
        self.routed = self.model in ("tedulorn", "nebutar")

    def _gen(self, name, device=DEVICE):
        return torch.Generator(device=device).manual_seed(zlib.crc32(f"{self.seed}/{name}".encode()))

    def _normal(self, name, shape):
        return torch.randn(shape, generator=self._gen(name), device=DEVICE)

    def _uniform(self, name, shape, lo, hi):
        return torch.rand(shape, generator=self._gen(name), device=DEVICE) * (hi - lo) + lo

    def _centers(self, d):
        return torch.nn.functional.normalize(self._normal("centers", (CLUSTERS, d)), dim=-1)

    def _router(self, name, shape):
        """Every kind of token has four experts that it wants far more than the others."""
        E, d = shape
        gen = self._gen(name, "cpu")
        want = torch.zeros(E, CLUSTERS)
        for c in range(CLUSTERS):
            if E % 4 == 0 and E == 32:                # four groups, experts are taken from two
                a, b = torch.randperm(4, generator=gen)[:2].tolist()
                p, q = torch.randperm(8, generator=gen), torch.randperm(8, generator=gen)
                chosen = [8 * a + int(p[0]), 8 * b + int(q[0]), 8 * a + int(p[1]), 8 * b + int(q[1])]
            else:
                chosen = torch.randperm(E, generator=gen)[:4].tolist()
            for e, strength in zip(chosen, (1.0, 0.9, 0.8, 0.7)):
                want[e, c] = strength
        return 0.28 * want.to(DEVICE) @ self._centers(d)

    def __call__(self, name, shape, vector=False):
        """A matrix in the model's dtype, or a float32 vector."""
        shape, last = tuple(shape), name.rsplit(".", 1)[-1]
        if not vector:
            if last == "router":
                t = self._router(name, shape)
            elif name == "embed" and self.routed:
                t = self._normal(name, shape).mul_(0.0174)
                kind = torch.arange(shape[0], device=DEVICE) % CLUSTERS
                t.add_((self._centers(shape[1]) * (0.01 * math.sqrt(shape[1])))[kind])
            elif name in ("embed", "model.embed_tokens.weight"):
                t = self._normal(name, shape).mul_(1.0 if name == "embed" else 0.5)
            elif name.endswith(("o_proj.weight", "down_proj.weight")):     # scaled by depth, as such models are set up
                t = self._normal(name, shape).mul_(0.02 / math.sqrt(2 * self.layers))
            else:
                t = self._normal(name, shape).mul_(0.02)
            return t.to(self.dtype)
        if last == "A_log":
            return self._uniform(name, shape, 1.0, 16.0).log()
        if last == "dt_bias":                          # a softplus of it lies between 0.001 and 0.1
            return self._uniform(name, shape, math.log(0.001), math.log(0.1)).exp().expm1().log()
        if ".mu." in name:
            return self._uniform(name, shape, 0.0, 1.0)
        if last == "w0":
            return self._uniform(name, shape, -6.0, 0.0)
        if name.endswith("a2.b"):
            return self._normal(name, shape) + 2.0
        if name.endswith("conv"):
            return self._normal(name, shape).mul_(0.4)
        if last in ("b", "correction"):
            return self._normal(name, shape).mul_(0.01)
        if last in ("u", "sink"):
            return self._normal(name, shape).mul_(0.5)
        if last == "vmix":
            return self._uniform(name, shape, 0.2, 0.5)
        if last == "dwa":
            t = self._normal(name, shape).mul_(0.05)
            t[-1] += 1.0
            return t
        if last == "in":
            return self._normal(name, shape).mul_(0.02) + 0.25
        if last == "mix" and len(shape) == 2:
            return self._normal(name, shape).mul_(0.02) + torch.eye(shape[0], device=DEVICE)
        t = 1.0 + self._normal(name, shape).mul_(0.05)         # gains, skips, streams' shares of a result
        closing = {"mitisun": ("norm1b", "norm2b"), "pozalorn": ("norm1", "norm2")}.get(self.model, ())
        return t.mul_(0.5) if last in closing else t           # gains of a branch's result


# ---- inputs ----------------------------------------------------------------------------------------------
def _lengths(case):
    """Tokens before (decode, mixed) or in (prefill) each row's pass, falling from ``context`` to an eighth of it."""
    rows, longest = case["rows"], case["context"]
    return [max(1, longest - longest * 7 * i // (8 * rows)) for i in range(rows)]


def _tokens(case, seed):
    """Per request (tokens before the pass, tokens of the pass)."""
    gen = torch.Generator().manual_seed(zlib.crc32(f"{seed}/tokens".encode()))

    def some(n):
        return torch.randint(VOCAB, (n,), generator=gen).tolist()
    if case["mode"] == "prefill":
        return [([], some(n)) for n in _lengths(case)]
    out = [(some(n), some(1)) for n in _lengths(case)]
    if case["mode"] == "mixed":
        out.append((some(case["context"] // 2), some(case["portion"])))
    return out


def _plan(case):
    from socrates_amd.config import config_class_for
    cfg = _config(case)
    return config_class_for((cfg.get("architectures") or [cfg.get("architecture")])[0]).from_dict(cfg).plan()


class _State(dict):
    """Gives the copies of weights that the kernel set made for its products back with the model."""

    def __del__(self):
        self["runner"].ops.forget_packed()


def prepare(case, seed):
    from socrates_amd.cache import CacheManager, blocks_for
    from socrates_amd.engine import ModelRunner
    from socrates_amd.engine.batch import StepEntry
    from socrates_amd.kernels import HipKernels
    from socrates_amd.parts import DecoderModel, cache_needs, expected_tensors

    plan, dtype, draw_tensor = _plan(case), getattr(torch, case["dtype"]), _Weights(case, seed)
    weights = {name: draw_tensor(name, decl.made_up_shape() if -1 in decl.shape else decl.shape, decl.kind == "vector")
               for name, decl in expected_tensors(plan).items()}
    model = DecoderModel(plan, weights, HipKernels(dtype, DEVICE))
    del weights
    tokens = _tokens(case, seed)
    longest = max(len(a) + len(b) for a, b in tokens) + 16
    cache = CacheManager(cache_needs(plan), max_rows=len(tokens), max_len=longest, block_size=16,
                         num_blocks=sum(blocks_for(len(a) + len(b) + 16, 16) for a, b in tokens), dtype=dtype, device=DEVICE)
    runner = ModelRunner(model, cache)
    state = _State(runner=runner, mode=case["mode"], tokens=[b for _, b in tokens])
    if case["mode"] == "prefill":
        return state
    rows = [cache.open_row() for _ in tokens]
    held = 1 if case["mode"] == "decode" else 0        # the last token before the pass is decoded, as in serving
    left = [(r, a[:len(a) - held]) for r, (a, _) in zip(rows, tokens)]
    while any(a for _, a in left):
        entries, room = [], 8192
        for i, (r, a) in enumerate(left):
            n = min(len(a), room)
            if n:
                entries.append(StepEntry(r, a[:n], []))
                left[i], room = (r, a[n:]), room - n
        runner.step(entries[:-1] + [StepEntry(entries[-1].row, entries[-1].tokens, [0])])
    if held:
        runner.enable_graphs(len(rows))
        runner.step([StepEntry(r, a[-1:], [0]) for r, (a, _) in zip(rows, tokens)])
    state["entries"] = [StepEntry(r, b, [len(b) - 1]) for r, (_, b) in zip(rows, tokens)]
    return state


def run(state):
    from socrates_amd.engine.batch import StepEntry
    runner = state["runner"]
    cache = runner.cache
    if state["mode"] == "prefill":
        rows = [cache.open_row() for _ in state["tokens"]]
        logits = runner.step([StepEntry(r, b, [len(b) - 1]) for r, b in zip(rows, state["tokens"])])
        for r in rows:
            cache.close_row(r)
        return logits
    logits = runner.step(state["entries"], borrow=True)
    for e in state["entries"]:
        cache.advance(e.row, -len(e.tokens))
    return logits


# ---- what a pass cannot do without ---------------------------------------------------------------------------
def work(case):
    from socrates_amd.parts import expected_tensors
    item = 2 if case["dtype"] == "bfloat16" else 4
    requests = [(0, n) for n in _lengths(case)] if case["mode"] == "prefill" else [(n, 1) for n in _lengths(case)]
    if case["mode"] == "mixed":
        requests.append((case["context"] // 2, case["portion"]))
    new, rows = sum(n for _, n in requests), len(requests)
    cfg = _config(case)
    size = {name: math.prod(decl.made_up_shape() if -1 in decl.shape else decl.shape) for name, decl in expected_tensors(_plan(case)).items()}
    tied = "head" not in size and "lm_head.weight" not in size
    nbytes, flops = 4.0 * rows * VOCAB, 0.0
    for name, n in size.items():
        expert = ".e" in name and ".mlp." in name
        if "embed" in name and "side" not in name:
            nbytes += item * n if tied else 0
            flops += 2.0 * n * rows if tied else 0
        elif name in ("head", "lm_head.weight"):
            nbytes += item * n
            flops += 2.0 * n * rows
        elif name not in ("pos", "side.embed"):
            nbytes += item * n * (min(1.0, 4 * new / 32) if expert else 1.0)
            flops += 2.0 * n * new * (4 / 32 if expert else 1.0)

    def attention(heads, kv_heads, dim, vdim, window, kept_dim=None):
        """Keys and values read once per request and written once per token; scores and sums of the visible keys."""
        b = f = 0.0
        per_key = kept_dim if kept_dim is not None else kv_heads * (dim + vdim)
        for past, n in requests:
            reach = min(past + n, window) if n == 1 else min(past, window)
            b += item * per_key * (reach + n)
            f += 2.0 * heads * (dim + vdim) * sum(min(p + 1, window) for p in range(past, past + n))
        return b, f

    def recurrence(heads, dim, vdim):
        return 2.0 * 4 * heads * dim * vdim * rows, 4.0 * heads * dim * vdim * new

    far = 1 << 30
    if case["model"].startswith("qwen3"):
        b, f = attention(cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["head_dim"], far)
        return {"bytes": nbytes + case["layers"] * b, "flops": flops + case["layers"] * f}
    for layer in cfg["layers"]:
        m, kind = layer["mixer"], layer["type"]
        parts = [("attention", m["left"]), ("state", m["right"])] if kind == "parallel" else [
            ({"latent_attention": "latent", "attention": "attention"}.get(kind, "state"), m)]
        for part, m in parts:
            if part == "state":
                b, f = recurrence(m["heads"], m.get("state", m.get("dim")), m.get("vdim", m.get("dim")))
            elif part == "latent":
                b, f = attention(m["heads"], 1, m["kv_rank"] + m["rot_dim"], m["kv_rank"], m["mask"]["size"], m["kv_rank"] + m["rot_dim"])
            else:
                b, f = attention(m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["mask"]["size"])
            nbytes, flops = nbytes + b, flops + f
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Float32 sums of up to 9,728 terms are 6e-6 off the exact logits. In bfloat16 the same sums in another order (the
    kernel set's other forms of its products and norms) move the logits by 0.004 to 0.009, at most 0.04 of their root
    mean square: a rounding that falls the other way decides many after it."""
    if case["dtype"] == "float32":
        return {"rel": 3e-5, "max": 3e-4}
    return {"rel": 0.03, "max": 0.16}


# ---- the same in float64, without the package ------------------------------------------------------------------
def _rms(x, eps):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _turn(x, freq, pairs, sign=1.0):
    """x [T, H, D] turned by position * freq over the first 2 len(freq) elements: neighbours (pairs) or halves."""
    n = 2 * len(freq)
    a = sign * torch.arange(x.shape[0], device=x.device, dtype=F64)[:, None] * freq[None]
    c, s = a.cos()[:, None], a.sin()[:, None]
    out = x.clone()
    u, v = (x[..., 0:n:2], x[..., 1:n:2]) if pairs else (x[..., :n // 2], x[..., n // 2:n])
    p, q = u * c - v * s, v * c + u * s
    if pairs:
        out[..., 0:n:2], out[..., 1:n:2] = p, q
    else:
        out[..., :n // 2], out[..., n // 2:n] = p, q
    return out


def _freq(rot, dims=None):
    dims = dims or rot["dims"]
    f = torch.tensor([rot["base"] ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=F64, device=DEVICE)
    sc = rot.get("scaling")
    if sc:
        wave = 2.0 * math.pi / f
        s = ((sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
        f = (1.0 - s) * f / sc["factor"] + s * f
    return f


def _attend(q, k, v, scale, seen, cap=None, sink=None, block=1024):
    """q [T, H, D], k [J, G, D], v [J, G, Dv]; ``seen(i)`` [len(i), J]; ``sink`` [H]: one more score without a value."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=F64, device=q.device)
    for lo in range(0, T, block):
        hide = ~seen(torch.arange(lo, min(lo + block, T), device=q.device)[:, None])
        for h in range(H):
            s = (q[lo:lo + block, h] @ k[:, h // (H // G)].T) * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            s = s.masked_fill_(hide, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[h].expand(s.shape[0], 1)], dim=1)
            p = torch.softmax(s, dim=-1)
            out[lo:lo + block, h] = p[:, :k.shape[0]] @ v[:, h // (H // G)]
    return out


def _seen(T, window=None, keep=0, chunk=None):
    j = torch.arange(T, device=DEVICE)[None]

    def seen(i):
        ok = j <= i
        if window is not None:
            ok = ok & ((i - j < window) | (j < keep))
        return ok & (i // chunk == j // chunk) if chunk else ok
    return seen


def _walk(q, k, v, decay):
    """S <- decay_t S + k_t v_t^T, o_t = S^T q_t: q, k [T, H, D], v [T, H, Dv], decay broadcast to [T, H, D]."""
    S = torch.zeros(q.shape[1], q.shape[2], v.shape[2], dtype=F64, device=q.device)
    out = []
    for q_t, k_t, v_t, d_t in zip(q, k, v, decay.expand(q.shape)):
        S = d_t[..., None] * S + k_t[..., None] * v_t[:, None]
        out.append((q_t[:, None] @ S)[:, 0])
    return torch.stack(out)


def _conv(x, taps, bias=0.0):
    n = taps.shape[1]
    padded = torch.cat([x.new_zeros(n - 1, x.shape[1]), x])
    return sum(padded[j:j + x.shape[0]] * taps[:, j] for j in range(n)) + bias


class _Plain:
    """``M`` draws a matrix, ``V`` a vector, in float64. x [N, d] holds the whole sequences one behind the other;
    what mixes tokens is run per sequence (``each``)."""

    def __init__(self, case, seed):
        draw_tensor = _Weights(case, seed)
        self.cfg = _config(case)
        self.M = lambda name, *shape: draw_tensor(name, shape).to(F64)
        self.V = lambda name, *shape: draw_tensor(name, shape, True).to(F64)
        self.ids = [torch.tensor(a + b, device=DEVICE) for a, b in _tokens(case, seed)]
        self.all = torch.cat(self.ids)
        self.ends = torch.tensor([len(i) for i in self.ids]).cumsum(0).tolist()
        self.d = 2560 if case["model"] != "qwen3-8b" else 4096

    def each(self, f, *tensors):
        n = [len(i) for i in self.ids]
        return torch.cat([f(*parts) for parts in zip(*(t.split(n) for t in tensors))])

    def embed(self, name, scale=1.0):
        return self.M(name, VOCAB, self.d)[self.all] * scale

    def last(self, x):
        return x[[e - 1 for e in self.ends]]

    # -- Qwen3
    def qwen3(self):
        c, d, M, V = self.cfg, self.d, self.M, self.V
        H, G, D, ff, eps = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["intermediate_size"], c["rms_norm_eps"]
        freq = _freq({"base": c["rope_theta"], "dims": D})
        x = self.embed("model.embed_tokens.weight")
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            a, m = p + "self_attn.", p + "mlp."
            h = _rms(x, eps) * V(p + "input_layernorm.weight", d)
            q = _rms((h @ M(a + "q_proj.weight", H * D, d).T).view(-1, H, D), eps) * V(a + "q_norm.weight", D)
            k = _rms((h @ M(a + "k_proj.weight", G * D, d).T).view(-1, G, D), eps) * V(a + "k_norm.weight", D)
            v = (h @ M(a + "v_proj.weight", G * D, d).T).view(-1, G, D)
            o = self.each(lambda q, k, v: _attend(_turn(q, freq, False), _turn(k, freq, False), v, D ** -0.5, _seen(len(q))), q, k, v)
            x = x + o.reshape(-1, H * D) @ M(a + "o_proj.weight", d, H * D).T
            h = _rms(x, eps) * V(p + "post_attention_layernorm.weight", d)
            x = x + (_silu(h @ M(m + "gate_proj.weight", ff, d).T) * (h @ M(m + "up_proj.weight", ff, d).T)) @ M(m + "down_proj.weight", d, ff).T
        x = _rms(self.last(x), eps) * V("model.norm.weight", d)
        return x @ M("model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight", VOCAB, d).T

    # -- Mitisun
    def wkv(self, h, p, m, eps):
        H, D, d, r, M, V = m["heads"], m["dim"], self.d, m["decay_rank"], self.M, self.V

        def before(h):
            return torch.cat([torch.zeros_like(h[:1]), h[:-1]])
        diff = self.each(before, h) - h
        mix = {s: h + diff * V(f"{p}mu.{s}", d) for s in "rkvgw"}
        q, k, v = ((mix[s] @ M(p + s, H * D, d).T).view(-1, H, D) for s in "rkv")
        gate = _silu(mix["g"] @ M(p + "g", H * D, d).T)
        w = torch.tanh(mix["w"] @ M(p + "w1", r, d).T) @ M(p + "w2", H * D, r).T + V(p + "w0", H * D)
        decay, u = torch.exp(-torch.exp(w)).view(-1, H, D), V(p + "u", H, D)

        def walk(q, k, v, decay):
            S = torch.zeros(H, D, D, dtype=F64, device=q.device)
            out = []
            for q_t, k_t, v_t, d_t in zip(q, k, v, decay):
                kv = k_t[..., None] * v_t[:, None]
                out.append((q_t[:, None] @ (S + u[..., None] * kv))[:, 0])
                S = d_t[..., None] * S + kv
            return torch.stack(out)
        o = _rms(self.each(walk, q, k, v, decay), eps).reshape(-1, H * D) * V(p + "norm", H * D)
        return (o * gate) @ M(p + "o", d, H * D).T

    def mamba2(self, h, p, m, eps):
        H, P, N, d, M, V = m["heads"], m["vdim"], m["state"], self.d, self.M, self.V
        inner = H * P
        z, xbc, dt = (h @ M(p + "in", 2 * inner + 2 * N + H, d).T).split([inner, inner + 2 * N, H], dim=-1)
        taps, bias = V(p + "conv", inner + 2 * N, m["conv"]), V(p + "conv.b", inner + 2 * N)
        x, B, C = _silu(self.each(lambda x: _conv(x, taps, bias), xbc)).split([inner, N, N], dim=-1)
        x, dt = x.reshape(-1, H, P), torch.nn.functional.softplus(dt + V(p + "dt_bias", H))
        decay = torch.exp(-torch.exp(V(p + "A_log", H)) * dt)[..., None]
        B, C = (t[:, None].expand(-1, H, N) for t in (B, C))
        y = self.each(_walk, C, B * dt[..., None], x, decay.expand(-1, H, N)) + V(p + "D", H)[:, None] * x
        y = _rms(y.reshape(-1, inner) * _silu(z), eps) * V(p + "norm", inner)
        return y @ M(p + "o", d, inner).T

    def latent(self, h, p, m, eps, kept, source):
        H, D, R, Dv, K, Q, d, M, V = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], m["q_rank"], self.d, self.M, self.V
        freq = _freq(m["rot"])
        if source is None:
            down = h @ M(p + "dkv", K + R, d).T
            turned = self.each(lambda t: _turn(t[:, None], freq, True)[:, 0], down[:, K:])
            source = kept[p] = (_rms(down[:, :K], eps) * V(p + "dkv.norm", K), turned)
        q = ((_rms(h @ M(p + "dq", Q, d).T, eps) * V(p + "dq.norm", Q)) @ M(p + "uq", H * (D + R), Q).T).view(-1, H, D + R)
        k = (source[0] @ M(p + "uk", H * D, K).T).view(-1, H, D)
        v = (source[0] @ M(p + "uv", H * Dv, K).T).view(-1, H, Dv)
        k = torch.cat([k, source[1][:, None].expand(-1, H, R)], dim=-1)

        def attend(q, k, v):
            q = torch.cat([q[..., :D], _turn(q[..., D:], freq, True)], dim=-1)
            return _attend(q, k, v, m["scale"], _seen(len(q), m["mask"]["size"]))
        return self.each(attend, q, k, v).reshape(-1, H * Dv) @ M(p + "o", d, H * Dv).T

    def clamped(self, h, p, ff, limit, act=1.702):
        g = (h @ self.M(p + "gate", ff, self.d).T).clamp(max=limit)
        u = (h @ self.M(p + "up", ff, self.d).T).clamp(-limit, limit)
        return (g * torch.sigmoid(act * g) * (u + 1)) @ self.M(p + "down", self.d, ff).T

    def mitisun(self):
        c, d, M, V, eps = self.cfg, self.d, self.M, self.V, self.cfg["norm"]["eps"]
        x, kept = self.embed("embed"), {}
        for i, layer in enumerate(c["layers"]):
            L, m = f"l{i}.", layer["mixer"]
            h = _rms(x, eps) * V(L + "norm1")
            if layer["type"] == "latent_attention":
                a = self.latent(h, L + "mix.", m, eps, kept, kept[f"l{m['kv_from']}.mix."] if "kv_from" in m else None)
            else:
                a = getattr(self, layer["type"])(h, L + "mix.", m, eps)
            a = a * torch.sigmoid(h @ M(L + "rg1", d, d).T + V(L + "rg1.b", d))
            x = x + c["residual_mult"] * _rms(a, eps) * V(L + "norm1b")
            h = _rms(x, eps) * V(L + "norm2")
            f = self.clamped(h, L + "mlp.", layer["mlp"]["ff"], layer["mlp"]["limit"])
            f = f * torch.sigmoid(h @ M(L + "rg2", d, d).T + V(L + "rg2.b", d))
            x = x + c["residual_mult"] * _rms(f, eps) * V(L + "norm2b")
        return (_rms(self.last(x), eps) * V("final.norm")) @ M("head", VOCAB, d).T

    # -- Tedulorn
    def retention(self, h, p, m, eps):
        H, D, Dv, d, M = m["heads"], m["dim"], m["vdim"], self.d, self.M
        freq = _freq(m["rot"])
        q, k = (self.each(lambda t: _turn(t, freq, False), (h @ M(p + s, H * D, d).T).view(-1, H, D)) for s in "qk")
        v = (h @ M(p + "v", H * Dv, d).T).view(-1, H, Dv)
        decay = torch.tensor(m["decay"], dtype=F64, device=DEVICE)[None, :, None].expand(q.shape)
        o = _rms(self.each(_walk, q, k * D ** -0.5, v, decay), eps).reshape(-1, H * Dv)
        return (o * _silu(h @ M(p + "g", H * Dv, d).T)) @ M(p + "o", d, H * Dv).T

    def kept_attention(self, h, p, m, eps, first):
        H, G, D, Dv, d, M, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"], self.d, self.M, self.V
        freq, mask = _freq(m["rot"]), m["mask"]
        q = _rms((h @ M(p + "q", H * D, d).T).view(-1, H, D), eps) * V(p + "q.norm", D)
        k = _rms((h @ M(p + "k", G * D, d).T).view(-1, G, D), eps) * V(p + "k.norm", D)
        own = v = (h @ M(p + "v", G * Dv, d).T).view(-1, G, Dv)
        if first is not None:
            lam = V(p + "vmix")
            v = (1.0 - lam) * v + lam * first
        zero = torch.zeros(H, dtype=F64, device=DEVICE)
        o = self.each(lambda q, k, v: _attend(_turn(q, freq, False), _turn(k, freq, False), v, m["scale"],
                                              _seen(len(q), mask["size"], mask["keep_first"]), sink=zero), q, k, v)
        o = o * torch.sigmoid(h @ M(p + "g", H, d).T)[:, :, None]
        return o.reshape(-1, H * Dv) @ M(p + "o", d, H * Dv).T, own if first is None else first

    def routed(self, h, p, mlp, one):
        r = mlp["router"]
        E, same = r["experts"], r.get("identity", 0)
        s = torch.softmax(h @ self.M(p + "router", E + same, self.d).T, dim=-1)
        choice = s + self.V(p + "correction", E + same)
        groups = r.get("groups")
        if groups:
            per = E // groups["count"]
            best = choice.view(-1, groups["count"], per).amax(-1).topk(groups["keep"], dim=-1).indices
            allowed = torch.zeros(len(h), groups["count"], dtype=torch.bool, device=DEVICE).scatter_(1, best, True)
            choice = choice.masked_fill(~allowed.repeat_interleave(per, dim=1), -math.inf)
        chosen = choice.topk(r["top"], dim=-1).indices
        picked = s.gather(1, chosen)
        if groups:
            picked = picked / (picked.sum(-1, keepdim=True) + 1e-20)
        w = torch.zeros_like(s).scatter_(1, chosen, picked)
        y = h * w[:, E:].sum(-1, keepdim=True)
        for e in range(E):
            at = w[:, e].nonzero()[:, 0]
            if len(at):
                y[at] += w[at, e, None] * one(h[at], f"{p}e{e}.")
        return y

    def tedulorn(self):
        c, d, M, V, eps = self.cfg, self.d, self.M, self.V, self.cfg["norm"]["eps"]
        x, first, side = self.embed("embed", c["embedding"]["scale"]), None, c["token_side"]["dim"]
        sides = M("side.embed", VOCAB, side * len(c["layers"]))[self.all]
        for i, layer in enumerate(c["layers"]):
            L, mlp = f"l{i}.", layer["mlp"]
            h = _rms(x, eps) * V(L + "norm1", d)
            if layer["type"] == "retention":
                x = x + self.retention(h, L + "mix.", layer["mixer"], eps)
            else:
                y, first = self.kept_attention(h, L + "mix.", layer["mixer"], eps, first)
                x = x + y
            h = _rms(x, eps) * V(L + "norm2", d)
            if mlp["kind"] == "dense":
                x = x + torch.relu(h @ M(L + "mlp.up", mlp["ff"], d).T) ** 2 @ M(L + "mlp.down", d, mlp["ff"]).T
            else:
                def one(h, p):
                    return self.clamped(h, p, mlp["expert"]["ff"], mlp["expert"]["limit"])
                x = x + self.routed(h, L + "mlp.", mlp, one) + one(h, L + "mlp.shared.")
            y = (_gelu(x @ M(L + "side.gate", side, d).T) * sides[:, i * side:(i + 1) * side]) @ M(L + "side.proj", d, side).T
            x = x + _rms(y, eps) * V(L + "side.norm", d)
        return (_rms(self.last(x), eps) * V("final.norm", d)) @ M("head", VOCAB, d).T

    # -- Pozalorn
    def gla(self, h, p, m, eps):
        H, D, Dv, d, M, V = m["heads"], m["dim"], m["vdim"], self.d, self.M, self.V
        q, k = ((h @ M(p + s, H * D, d).T).view(-1, H, D) for s in "qk")
        v = (h @ M(p + "v", H * Dv, d).T).view(-1, H, Dv)
        z = (h @ M(p + "a1", 16, d).T) @ M(p + "a2", H * D, 16).T + V(p + "a2.b", H * D)
        alpha = torch.sigmoid(z).pow(1.0 / m["tau"]).view(-1, H, D)
        o = _rms(self.each(_walk, q * D ** -0.5, k, v, alpha), eps) * V(p + "norm", Dv)
        return (o.reshape(-1, H * Dv) * _silu(h @ M(p + "g", H * Dv, d).T)) @ M(p + "o", d, H * Dv).T

    def lightning(self, h, p, m, eps):
        H, D, Dv, d, M, V = m["heads"], m["dim"], m["vdim"], self.d, self.M, self.V
        q, k, v = (_silu(h @ M(p + s, H * D, d).T).view(-1, H, D) for s in "qkv")
        decay = torch.tensor(m["decay"], dtype=F64, device=DEVICE)[None, :, None].expand(q.shape)
        o = self.each(_walk, q, k, v, decay).reshape(-1, H * Dv)
        return (_rms(o, eps) * V(p + "norm", H * Dv) * torch.sigmoid(h @ M(p + "g", H * Dv, d).T)) @ M(p + "o", d, H * Dv).T

    def window(self, h, p, m, eps):
        """With a sink and norms per head, or with block means before the window and norms over the projections."""
        H, G, D, Dv, d, M, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"], self.d, self.M, self.V
        size, pool, freq = m["mask"]["size"], m["mask"].get("pool", 0), _freq(m["rot"])
        q = h @ M(p + "q", H * D, d).T + V(p + "q.b", H * D)
        k = h @ M(p + "k", G * D, d).T + V(p + "k.b", G * D)
        v = (h @ M(p + "v", G * Dv, d).T + V(p + "v.b", G * Dv)).view(-1, G, Dv)
        if pool:
            q, k = ((_rms(t, eps) * V(f"{p}{s}.norm", n * D)).view(-1, n, D) for t, s, n in ((q, "q", H), (k, "k", G)))
            vfreq = _freq({"base": m["rot"]["base"], "dims": Dv})

            def attend(q, k, v):
                T, B = len(q), len(q) // pool
                k, v = _turn(k, freq, True), _turn(v, vfreq, True)
                means = [t[:B * pool].view(B, pool, G, t.shape[2]).mean(1) for t in (k, v)]
                near, last = _seen(T, size), torch.arange(B, device=DEVICE)[None] * pool + pool - 1
                o = _attend(_turn(q, freq, True), torch.cat([k, means[0]]), torch.cat([v, means[1]]), m["scale"],
                            lambda i: torch.cat([near(i), last <= i - size], dim=1))
                return _turn(o, vfreq, True, -1.0)
            return self.each(attend, q, k, v).reshape(-1, H * Dv) @ M(p + "o", d, H * Dv).T
        q, k = (_rms(t.view(-1, n, D), eps) * V(f"{p}{s}.norm", D) for t, s, n in ((q, "q", H), (k, "k", G)))
        sink = V(p + "sink", H)
        o = self.each(lambda q, k, v: _attend(_turn(q, freq, True), _turn(k, freq, True), v, m["scale"], _seen(len(q), size), sink=sink), q, k, v)
        return o.reshape(-1, H * Dv) @ M(p + "o", d, H * Dv).T + V(p + "o.b", d)

    def pozalorn(self):
        c, d, M, V, eps = self.cfg, self.d, self.M, self.V, self.cfg["norm"]["eps"]
        x = self.embed("embed")
        results = [x]
        for i, layer in enumerate(c["layers"]):
            L, m = f"l{i}.", layer["mixer"]
            if layer["type"] == "parallel":
                y = m["left_scale"] * self.window(x, L + "mix.left.", m["left"], eps) + m["right_scale"] * self.lightning(x, L + "mix.right.", m["right"], eps)
            else:
                y = (self.gla if layer["type"] == "gla" else self.window)(x, L + "mix.", m, eps)
            x = x + _rms(y, eps) * V(L + "norm1", d)
            ff = layer["mlp"]["ff"]
            y = (_gelu(x @ M(L + "mlp.gate", ff, d).T) * (x @ M(L + "mlp.up", ff, d).T)) @ M(L + "mlp.down", d, ff).T
            results.append(x + _rms(y, eps) * V(L + "norm2", d))
            share = V(L + "dwa", i + 2)
            x = sum(share[j] * r for j, r in enumerate(results))
        return (_rms(self.last(x), eps) * V("final.norm", d)) @ M("head", VOCAB, d).T

    # -- Nebutar
    def centred(self, x, name, eps):
        x = x - x.mean(-1, keepdim=True)
        return _rms(x, eps) * self.V(name, self.d) + self.V(name + ".b", self.d)

    def chunked(self, h, p, m):
        H, G, D, Dv, d, M = m["heads"], m["kv_heads"], m["dim"], m["vdim"], self.d, self.M
        q = (h @ M(p + "q", H * D, d).T).view(-1, H, D)
        k, v = (h @ M(p + "k", G * D, d).T).view(-1, G, D), (h @ M(p + "v", G * Dv, d).T).view(-1, G, Dv)
        o = self.each(lambda q, k, v: _attend(q, k, v, m["scale"], _seen(len(q), chunk=m["mask"]["size"]), cap=m["softcap"]), q, k, v)
        return o.reshape(-1, H * Dv) @ M(p + "o", d, H * Dv).T

    def delta(self, h, p, m, eps):
        H, G, D, Dv, n, d, M, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["conv"], self.d, self.M, self.V

        def projected(s, width):
            taps = V(f"{p}{s}.conv", width, n)
            return _silu(self.each(lambda x: _conv(x, taps), h @ M(p + s, width, d).T))
        q, k = (projected(s, G * D).view(-1, G, D) for s in "qk")
        v = projected("v", H * Dv).view(-1, H, Dv)
        q, k = (t / torch.sqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        q, k = (t.repeat_interleave(H // G, dim=1) for t in (q * D ** -0.5, k))
        beta = torch.sigmoid(h @ M(p + "b", H, d).T)
        g = torch.exp(-torch.exp(V(p + "A_log", H)) * torch.nn.functional.softplus(h @ M(p + "a", H, d).T + V(p + "dt_bias", H)))

        def walk(q, k, v, g, beta):
            S = torch.zeros(H, D, Dv, dtype=F64, device=q.device)
            out = []
            for q_t, k_t, v_t, g_t, b_t in zip(q, k, v, g[..., None, None], beta[..., None]):
                S = g_t * S
                u = b_t * (v_t - (k_t[:, None] @ S)[:, 0])
                S = S + k_t[..., None] * u[:, None]
                out.append((q_t[:, None] @ S)[:, 0])
            return torch.stack(out)
        o = _rms(self.each(walk, q, k, v, g, beta), eps) * V(p + "norm", Dv)
        return (o.reshape(-1, H * Dv) * _silu(h @ M(p + "g", H * Dv, d).T)) @ M(p + "o", d, H * Dv).T

    def nebutar(self):
        c, d, M, V, eps = self.cfg, self.d, self.M, self.V, self.cfg["norm"]["eps"]
        pos = M("pos", c["max_positions"], d)
        x = (self.embed("embed", c["embedding"]["scale"]) + torch.cat([pos[:len(i)] for i in self.ids]))[None].repeat(c["streams"], 1, 1)

        def through(x, p, f):
            n = c["streams"]
            y = f(torch.einsum("a,atd->td", V(p + "in", n), x))
            return torch.einsum("ab,atd->btd", V(p + "mix", n, n), x) + V(p + "out", n).view(-1, 1, 1) * y
        for i, layer in enumerate(c["layers"]):
            L, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]

            def mixer(u):
                h = self.centred(u, L + "norm1", eps)
                return m["left_scale"] * self.chunked(h, L + "mix.left.", m["left"]) + m["right_scale"] * self.delta(h, L + "mix.right.", m["right"], eps)

            def one(h, p):
                ff = mlp["expert"]["ff"]
                return (_silu(h @ M(p + "gate", ff, d).T) * (h @ M(p + "up", ff, d).T)) @ M(p + "down", d, ff).T
            x = through(x, L + "hc1.", mixer)
            x = through(x, L + "hc2.", lambda u: self.routed(self.centred(u, L + "norm2", eps), L + "mlp.", mlp, one))
        return self.centred(self.last(x.sum(0)), "final.norm", eps) @ M("embed", VOCAB, d).T


def exact(case, seed):
    with torch.no_grad():
        plain = _Plain(case, seed)
        return getattr(plain, "qwen3" if case["model"].startswith("qwen3") else case["model"])()
