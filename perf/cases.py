"""Performance cases: the work that a training program has this package do.

Each case is one call (forward and backward) through the public entry points,
on the inputs a program has in hand before it.  ``listed()`` names the cases,
``draw`` makes others of the same ranges, ``exact`` restates each of them in
64-bit torch.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64

NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
       -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
       0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
       0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)
INT4 = tuple(float(i - 8) for i in range(16))

Q, K, V, O = (f"self_attn.{p}_proj" for p in "qkvo")
GATE, UP, DOWN = (f"mlp.{p}_proj" for p in ("gate", "up", "down"))
ALL7 = (Q, K, V, O, GATE, UP, DOWN)
QVO = (Q, V, O)

YARN = {"rope_type": "yarn", "rope_theta": 10000.0, "factor": 40.0,
        "original_max_position_embeddings": 4096, "beta_fast": 32, "beta_slow": 1, "mscale": 1.0,
        "mscale_all_dim": 1.0}


def listed():
    return [
        # the smallest step a program takes: a unit-sized layer (tests, debug
        # runs), where launches and host work count
        {"name": "layer_tiny", "kind": "layer", "H": 256, "I": 688, "heads": 4, "kv": 4, "D": 64,
         "B": 2, "S": 128, "rank": 8, "codec": "nf4-g128", "targets": "all", "qk_norm": False,
         "padded": False, "layers": 1, "stream": False},
        # the headline: one Llama-3-8B decoder layer, forward + recompute + backward
        {"name": "layer_llama8b", "kind": "layer", "H": 4096, "I": 14336, "heads": 32, "kv": 8,
         "D": 128, "B": 1, "S": 2048, "rank": 16, "codec": "nf4-g128", "targets": "all",
         "qk_norm": False, "padded": False, "layers": 1, "stream": False},
        # a batch of chat rows of unequal length: right padding, an odd row
        # length, int4 storage, the default q/v/o adapters, Qwen3's q/k norms
        {"name": "layer_qwen3_padded", "kind": "layer", "H": 4096, "I": 12288, "heads": 32,
         "kv": 8, "D": 128, "B": 3, "S": 701, "rank": 8, "codec": "int4-sym-g128",
         "targets": "qvo", "qk_norm": True, "padded": True, "layers": 1, "stream": False},
        # four layers streamed from pinned host memory through two slots, as a
        # model larger than its device budget runs
        {"name": "stream_llama8b", "kind": "layer", "H": 4096, "I": 14336, "heads": 32, "kv": 8,
         "D": 128, "B": 1, "S": 2048, "rank": 16, "codec": "nf4-g128", "targets": "all",
         "qk_norm": False, "padded": False, "layers": 4, "stream": True},
        # one adapted projection on a short prompt: the fewest rows a GEMM sees
        {"name": "linear_short", "kind": "linear", "M": 77, "N": 14336, "K": 4096, "rank": 16,
         "residual": True},
        # a bitsandbytes NF4 + double-quantisation matrix under a frozen linear
        {"name": "linear_nf4_state", "kind": "nf4_state", "M": 1000, "N": 14336, "K": 4096},
        # grouped-query attention at the streamed model's sequence length
        {"name": "attention_gqa", "kind": "attention", "B": 1, "S": 4096, "heads": 32, "kv": 8,
         "D": 128, "padded": False},
        # small heads, ragged right-padded rows
        {"name": "attention_d64_padded", "kind": "attention", "B": 4, "S": 333, "heads": 16,
         "kv": 4, "D": 64, "padded": True},
        # a DeepSeek-V3 decoder layer with multi-head latent attention and a dense MLP
        {"name": "layer_mla", "kind": "mla", "H": 7168, "heads": 128, "q_rank": 1536,
         "kv_rank": 512, "I": 12288, "B": 1, "S": 2048, "rank": 8},
        # mixture-of-experts feed-forwards: ~256 rows an expert with adapters
        # on the experts, and ~64 rows an expert with a shared expert
        {"name": "moe_qwen3", "kind": "moe", "H": 2048, "I": 768, "E": 128, "k": 8, "T": 4096,
         "rank": 8},
        {"name": "moe_deepseek", "kind": "deepseek_moe", "H": 7168, "I": 2048, "E": 256, "k": 8,
         "groups": 8, "group_k": 4, "T": 2048, "rank": 8},
        # final norm, head and loss over a whole sequence with its gradient
        {"name": "terminal_qwen3", "kind": "terminal", "H": 4096, "V": 151936, "S": 4096,
         "chunk": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "stream", "linear", "nf4_state", "attention", "mla",
                       "moe", "deepseek_moe", "terminal"])
    if kind in ("layer", "stream"):
        H = rng.choice([1024, 2048, 2560, 4096])
        D = rng.choice([64, 128])
        heads = H // D
        stream = kind == "stream"
        return {"kind": "layer", "H": H, "I": 8 * _log(rng, H // 4, H // 2), "heads": heads,
                "kv": heads // rng.choice([1, 2, 4]), "D": D, "B": rng.choice([1, 2, 3]),
                "S": _log(rng, 40, 1000), "rank": rng.choice([4, 8, 16, 21]),
                "codec": rng.choice(["nf4-g128", "int4-sym-g128"]),
                "targets": rng.choice(["all", "qvo"]), "qk_norm": rng.random() < 0.5,
                "padded": rng.random() < 0.5, "layers": 3 if stream else 1, "stream": stream}
    if kind == "linear":
        return {"kind": "linear", "M": _log(rng, 8, 6000), "N": 8 * _log(rng, 128, 3584),
                "K": 128 * _log(rng, 8, 112), "rank": rng.choice([0, 3, 8, 16, 32]),
                "residual": rng.random() < 0.5}
    if kind == "nf4_state":
        return {"kind": "nf4_state", "M": _log(rng, 8, 6000), "N": 8 * _log(rng, 128, 3584),
                "K": 64 * _log(rng, 16, 224)}
    if kind == "attention":
        kv = rng.choice([2, 4, 8])
        return {"kind": "attention", "B": rng.choice([1, 2, 3]), "S": _log(rng, 30, 3000),
                "heads": kv * rng.choice([1, 2, 4]), "kv": kv, "D": rng.choice([64, 128]),
                "padded": rng.random() < 0.5}
    if kind == "mla":
        return {"kind": "mla", "H": rng.choice([2048, 4096, 7168]),
                "heads": rng.choice([16, 32, 64, 128]), "q_rank": rng.choice([768, 1536]),
                "kv_rank": 512, "I": 128 * _log(rng, 16, 96), "B": rng.choice([1, 2]),
                "S": _log(rng, 60, 1000), "rank": rng.choice([8, 16])}
    if kind == "moe":
        return {"kind": "moe", "H": 128 * _log(rng, 8, 24), "I": 128 * _log(rng, 3, 12),
                "E": rng.choice([16, 64, 100, 128]), "k": rng.choice([2, 4, 8]),
                "T": _log(rng, 60, 4500), "rank": rng.choice([0, 4, 8])}
    if kind == "deepseek_moe":
        return {"kind": "deepseek_moe", "H": 128 * _log(rng, 16, 56), "I": 128 * _log(rng, 6, 16),
                "E": rng.choice([64, 128, 256]), "k": rng.choice([4, 6, 8]), "groups": 8,
                "group_k": rng.choice([3, 4]), "T": _log(rng, 60, 2048), "rank": 8}
    S = _log(rng, 60, 4000)
    return {"kind": "terminal", "H": 256 * _log(rng, 4, 16), "V": 8 * _log(rng, 4000, 16000),
            "S": S, "chunk": rng.choice([256, 1024, 4096])}


# --------------------------------------------------------------- raw inputs
# Everything below that begins with an underscore and takes a generator makes
# plain tensors on the GPU; prepare() hands them to the package and exact()
# to the 64-bit restatement.
def _dev():
    return torch.device("cuda:0")


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed) * 2654435761 % (1 << 62) + 1)


def _randn(g, *shape, std=1.0, dtype=BF):
    return (torch.randn(*shape, generator=g, device=_dev()) * std).to(dtype)


def _quantise(g, numel, codec, std=0.02, step=1 << 27):
    """N(0, std) weights stored 4-bit: codes (two a byte, low nibble first) and
    one fp32 scale per 128."""
    payload = torch.empty(numel // 2, dtype=torch.uint8, device=_dev())
    scales = torch.empty(numel // 128, dtype=F32, device=_dev())
    mids = torch.tensor([(a + b) / 2 for a, b in zip(NF4, NF4[1:])], device=_dev())
    for at in range(0, numel, step):
        n = min(step, numel - at)
        w = torch.randn(n, generator=g, device=_dev()).mul_(std).view(-1, 128)
        amax = w.abs().amax(1)
        if codec == "nf4-g128":
            scale = amax
            codes = torch.bucketize(w.div_(scale[:, None]), mids, out_int32=True).to(torch.uint8)
        else:
            scale = amax / 7
            codes = (w.div_(scale[:, None]).round_() + 8).to(torch.uint8)
        scales[at // 128:(at + n) // 128] = scale
        pair = codes.view(-1, 2)
        payload[at // 2:(at + n) // 2] = pair[:, 0] | (pair[:, 1] << 4)
    return payload, scales


def _decode64(payload, scales, shape, codec, group=128, high_first=False):
    """bf16(codebook[code] * scale) of every weight, in float64."""
    cb = torch.tensor(NF4 if codec == "nf4-g128" else INT4, dtype=F32, device=payload.device)
    lo, hi = payload & 15, payload >> 4
    codes = torch.stack((hi, lo) if high_first else (lo, hi), 1).view(-1).long()
    numel = math.prod(shape)
    w = cb[codes[:numel]]
    w = w * scales.repeat_interleave(group)[:numel]
    return w.to(BF).to(F64).view(shape)


def _adapter(g, rank, fin, fout):
    return (_randn(g, rank, fin, std=0.02, dtype=F32), _randn(g, fout, rank, std=0.02, dtype=F32))


def _lengths(case):
    """Valid prefix of each right-padded row, or None."""
    if not case["padded"]:
        return None
    B, S = case["B"], case["S"]
    return [S if b == 0 else max(1, S - (b * S) // 5) for b in range(B)]


def _layer_shapes(c):
    H, I, D = c["H"], c["I"], c["D"]
    return {Q: (c["heads"] * D, H), K: (c["kv"] * D, H), V: (c["kv"] * D, H),
            O: (H, c["heads"] * D), GATE: (I, H), UP: (I, H), DOWN: (H, I)}


def _layer_inputs(c, seed):
    g = _gen(seed)
    layers = []
    targets = ALL7 if c["targets"] == "all" else QVO
    for _ in range(c["layers"]):
        w = {}
        for n, s in _layer_shapes(c).items():
            numel = s[0] * s[1]
            p, sc = _quantise(g, -(-numel // 128) * 128, c["codec"])
            if numel % 128:  # the last group's padding holds zeros (code 7 or 8)
                zero = 7 if c["codec"] == "nf4-g128" else 8
                p[numel // 2:] = zero | (zero << 4)
            w[n] = (p, sc, s)
        norms = {"input_layernorm.weight": 1 + _randn(g, c["H"], std=0.05, dtype=F32),
                 "post_attention_layernorm.weight": 1 + _randn(g, c["H"], std=0.05, dtype=F32)}
        if c["qk_norm"]:
            norms["self_attn.q_norm.weight"] = 1 + _randn(g, c["D"], std=0.1, dtype=F32)
            norms["self_attn.k_norm.weight"] = 1 + _randn(g, c["D"], std=0.1, dtype=F32)
        ab = {t: _adapter(g, c["rank"], _layer_shapes(c)[t][1], _layer_shapes(c)[t][0])
              for t in targets}
        layers.append((w, {k: v.to(BF) for k, v in norms.items()}, ab))
    x = _randn(g, c["B"], c["S"], c["H"])
    dy = _randn(g, c["B"], c["S"], c["H"])
    return layers, x, dy


def _record(spec_shape, codec, payload, scales):
    from spilltune_amd import codecs
    spec = {"version": 1, "shape": list(spec_shape), "dtype": "bfloat16", "codec": codec,
            "group_size": codecs.GROUP, "numel": math.prod(spec_shape)}
    return codecs.Record(spec, {"payload": payload.cpu(), "scales": scales.cpu()})


def _lora_objects(index, shapes, ab, alpha, rank, targets):
    from spilltune_amd.lora import create_lora_for_block
    adapters = create_lora_for_block(index, "full_attention", shapes, rank=rank, alpha=alpha,
                                     device=_dev(), targets=targets)
    with torch.no_grad():
        for t, p in adapters.items():
            p.A.copy_(ab[t][0])
            p.B.copy_(ab[t][1])
    return adapters


def _prepare_layer(c, seed):
    from spilltune_amd import slots
    from spilltune_amd.dense import dense_block, lora_kwargs, positions_and_masks
    layers, x, dy = _layer_inputs(c, seed)
    blocks = []
    for i, (w, norms, ab) in enumerate(layers):
        host, specs = {}, {}
        for n, (p, s, shape) in w.items():
            rec = _record(shape, c["codec"], p, s)
            specs[f"{n}.weight"] = {"spec": rec.spec, "parts": {}}
            for part, t in rec.parts.items():
                host[f"@{n}.weight/{part}"] = t
                specs[f"{n}.weight"]["parts"][part] = f"@{n}.weight/{part}"
        host.update({k: v.cpu() for k, v in norms.items()})
        adapters = _lora_objects(i, _layer_shapes(c), ab, 2.0 * c["rank"], c["rank"], tuple(ab))
        kwargs = {"heads": c["heads"], "kv_heads": c["kv"], "head_dim": c["D"], "eps": 1e-5,
                  **lora_kwargs(adapters)}
        if c["qk_norm"]:
            kwargs["qk_norm"] = True
        blocks.append(slots.BlockPlan(i, "full_attention", dense_block, kwargs, host, adapters,
                                      specs))
    if c["stream"]:
        session = slots.Q4SlotSession(blocks, _dev(), host_budget_bytes=1 << 40,
                                      device_budget_bytes=1 << 40, slots=2)
    else:
        session = slots.ResidentSession(blocks, _dev())
    valid = torch.ones(c["B"], c["S"], dtype=torch.bool)
    for b, n in enumerate(_lengths(c) or []):
        valid[b, n:] = False
    rot, mask = positions_and_masks(valid, head_dim=c["D"], theta=500000.0, device=_dev())
    return {"blocks": blocks, "session": session, "rot": rot, "mask": mask, "x": x, "dy": dy}


def _run_layer(s):
    from spilltune_amd.recompute import streaming_block
    x = s["x"].detach().requires_grad_(True)
    h = x
    with s["session"].run():
        for b in s["blocks"]:
            h = streaming_block(h, s["rot"], s["mask"], b.functional, b.kwargs,
                                s["session"].reloader(b), b.adapters, b.index)
        h.backward(s["dy"])
    out = {"out": h.detach(), "dx": x.grad}
    for b in s["blocks"]:
        for n, p in b.adapters.items():
            out[f"{b.index}:{n}.A"] = p.grad_A
            out[f"{b.index}:{n}.B"] = p.grad_B
    return out


# --------------------------------------------------------------- 64-bit pieces
def _rms64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(F64)


def _rotate64(t, cos, sin):
    half = t.shape[-1] // 2
    return t * cos + torch.cat((-t[..., half:], t[..., :half]), -1) * sin


def _tables(S, dim, inverse, amplitude=1.0):
    """The bf16 rotary tables of positions 0..S-1 as float64 [S, dim]."""
    phase = torch.arange(S, device=_dev()).float()[:, None] * inverse[None, :]
    phase = torch.cat((phase, phase), -1)
    return (phase.cos() * amplitude).to(BF).to(F64), (phase.sin() * amplitude).to(BF).to(F64)


def _attend64(q, k, v, scale, lengths=None):
    """Causal attention [B,H,S,*] in float64, one (row, head) group at a time;
    a differentiable result."""
    B, H, S, _ = q.shape
    rep = H // k.shape[1]
    causal = torch.ones(S, S, dtype=torch.bool, device=q.device).tril()
    step = max(1, int(2e8) // (S * S))
    rows = []
    for b in range(B):
        keep = causal if lengths is None else causal & (
            torch.arange(S, device=q.device)[None, :] < lengths[b])
        parts = []
        for h in range(0, H, step):
            hs = torch.arange(h, min(h + step, H), device=q.device)
            qq, kk, vv = q[b, hs], k[b, hs // rep], v[b, hs // rep]
            sc = (qq @ kk.transpose(1, 2).contiguous()) * scale
            p = torch.softmax(sc.masked_fill(~keep, -1e300), -1)
            parts.append(p @ vv)
        rows.append(torch.cat(parts, 0))
    return torch.stack(rows)


def _lin64(x, w, ab=None, scale=2.0):
    y = x @ w.t()
    return y if ab is None else y + scale * (x @ ab[0].t()) @ ab[1].t()


def _exact_layer(c, seed):
    layers, x, dy = _layer_inputs(c, seed)
    B, S, H = x.shape
    D, heads, kv = c["D"], c["heads"], c["kv"]
    inv = 1.0 / 500000.0 ** (torch.arange(0, D, 2, device=_dev()).float() / D)
    cos, sin = _tables(S, D, inv)
    leaves = {"x": x.to(F64).requires_grad_(True)}
    h = leaves["x"]
    for i, (w, norms, ab) in enumerate(layers):
        W = {n: _decode64(p, s, shape, c["codec"]) for n, (p, s, shape) in w.items()}
        L = {}
        for t, (a, b) in ab.items():
            L[t] = (a.to(F64).requires_grad_(True), b.to(F64).requires_grad_(True))
            leaves[f"{i}:{t}.A"], leaves[f"{i}:{t}.B"] = L[t]
        xn = _rms64(h, norms["input_layernorm.weight"], 1e-5)

        def proj(t, name, n):
            return _lin64(t, W[name], L.get(name)).view(B, S, n, D)
        q, k, v = proj(xn, Q, heads), proj(xn, K, kv), proj(xn, V, kv)
        if c["qk_norm"]:
            q = _rms64(q, norms["self_attn.q_norm.weight"], 1e-5)
            k = _rms64(k, norms["self_attn.k_norm.weight"], 1e-5)
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
        a = _attend64(_rotate64(q, cos, sin), _rotate64(k, cos, sin), v, D ** -0.5, _lengths(c))
        h = h + _lin64(a.transpose(1, 2).reshape(B, S, heads * D), W[O], L.get(O))
        xn = _rms64(h, norms["post_attention_layernorm.weight"], 1e-5)
        act = F.silu(_lin64(xn, W[GATE], L.get(GATE))) * _lin64(xn, W[UP], L.get(UP))
        h = h + _lin64(act, W[DOWN], L.get(DOWN))
    grads = torch.autograd.grad(h, list(leaves.values()), dy.to(F64))
    out = dict(zip(leaves, grads))
    return {"out": h.detach(), "dx": out.pop("x"), **out}


# --------------------------------------------------------------- one projection
class _Lora:
    def __init__(self, A, B, rank):
        self.A, self.B, self.rank, self.scale = A, B, rank, 2.0


def _linear_inputs(c, seed):
    g = _gen(seed)
    M, N, Kd = c["M"], c["N"], c["K"]
    p, s = _quantise(g, N * Kd, "nf4-g128")
    ab = _adapter(g, c["rank"], Kd, N) if c["rank"] else None
    res = _randn(g, M, N) if c["residual"] else None
    return p, s, ab, res, _randn(g, M, Kd), _randn(g, M, N)


def _prepare_linear(c, seed):
    from spilltune_amd import ops
    p, s, ab, res, x, dy = _linear_inputs(c, seed)
    lora = None if ab is None else _Lora(ab[0].requires_grad_(True), ab[1].requires_grad_(True),
                                         c["rank"])
    return {"w": ops.Q4Weight(p, s, (c["N"], c["K"]), "nf4-g128"), "lora": lora, "res": res,
            "x": x, "dy": dy}


def _run_linear(s):
    from spilltune_amd import ops
    x = s["x"].detach().requires_grad_(True)
    lora = s["lora"]
    y = ops.q4_lora_linear(x, s["w"], None if lora is None else [lora], residual=s["res"])
    if lora is None:
        (dx,) = torch.autograd.grad(y, [x], s["dy"])
        return {"y": y.detach(), "dx": dx}
    dx, da, db = torch.autograd.grad(y, [x, lora.A, lora.B], s["dy"])
    return {"y": y.detach(), "dx": dx, "dA": da, "dB": db}


def _exact_linear(c, seed):
    p, s, ab, res, x, dy = _linear_inputs(c, seed)
    W = _decode64(p, s, (c["N"], c["K"]), "nf4-g128")
    x, dy = x.to(F64), dy.to(F64)
    y, dx = x @ W.t(), dy @ W
    out = {}
    if ab is not None:
        A, B = ab[0].to(F64), ab[1].to(F64)
        t, dt = x @ A.t(), 2.0 * dy @ B
        y, dx = y + 2.0 * t @ B.t(), dx + dt @ A
        out = {"dA": dt.t() @ x, "dB": 2.0 * dy.t() @ t}
    return {"y": y if res is None else y + res.to(F64), "dx": dx, **out}


def _nf4_inputs(c, seed):
    """A double-quantised state: uint8 block statistics (one per 64 weights)
    against a 256-entry map, one fp32 scale per 256 blocks, one offset."""
    g = _gen(seed)
    M, N, Kd = c["M"], c["N"], c["K"]
    numel = N * Kd
    blocks = -(-numel // 64)
    payload = torch.randint(0, 256, (numel // 2,), dtype=torch.uint8, device=_dev(), generator=g)
    absmax = torch.randint(0, 256, (blocks,), dtype=torch.uint8, device=_dev(), generator=g)
    nested = 0.01 + 0.005 * torch.rand(-(-blocks // 256), device=_dev(), generator=g)
    nmap = torch.linspace(-1.0, 1.0, 256, device=_dev())
    offset = 0.046875
    scales = nmap[absmax.long()] * nested.repeat_interleave(256)[:blocks] + offset
    x = _randn(g, 1, M, Kd)
    return payload, absmax, nested, nmap, offset, scales, x, _randn(g, 1, M, N)


def _prepare_nf4(c, seed):
    from spilltune_amd import nf4_state
    payload, absmax, nested, nmap, offset, _, x, dy = _nf4_inputs(c, seed)
    meta = {"quant_type": "nf4", "blocksize": 64, "dtype": "bfloat16", "shape": [c["N"], c["K"]],
            "nested_blocksize": 256, "nested_dtype": "float32", "nested_offset": offset}
    parts = {"absmax": absmax.cpu(), "nested_absmax": nested.cpu(),
             "nested_quant_map": nmap.cpu(), "quant_map": torch.tensor(NF4),
             nf4_state.PACKED_STATE_KEY: nf4_state.pack_metadata(meta)}
    state = nf4_state.PinnedNF4State(payload.cpu().view(-1, 1), parts).stage(_dev())
    return {"state": state, "x": x, "dy": dy}


def _run_nf4(s):
    from spilltune_amd import nf4_state
    x = s["x"].detach().requires_grad_(True)
    y = nf4_state.linear_cuda(x, s["state"])
    (dx,) = torch.autograd.grad(y, [x], s["dy"])
    return {"y": y.detach(), "dx": dx}


def _exact_nf4(c, seed):
    payload, _, _, _, _, scales, x, dy = _nf4_inputs(c, seed)
    W = _decode64(payload, scales, (c["N"], c["K"]), "nf4-g128", 64, True)
    return {"y": x.to(F64) @ W.t(), "dx": dy.to(F64) @ W}


# --------------------------------------------------------------- attention
def _attention_inputs(c, seed):
    g = _gen(seed)
    B, S, D = c["B"], c["S"], c["D"]
    q = _randn(g, B, c["heads"], S, D)
    k, v = (_randn(g, B, c["kv"], S, D) for _ in range(2))
    return q, k, v, _randn(g, B, S, c["heads"] * D)


def _prepare_attention(c, seed):
    q, k, v, do = _attention_inputs(c, seed)
    n = _lengths(c)
    lengths = None if n is None else torch.tensor(n, dtype=torch.int32, device=_dev())
    return {"q": q, "k": k, "v": v, "do": do, "lengths": lengths, "D": c["D"]}


def _run_attention(s):
    from spilltune_amd import ops
    q, k, v = (s[n].detach().requires_grad_(True) for n in "qkv")
    out = ops.causal_attention(q, k, v, ops.attention_scale(s["D"]), s["lengths"])
    dq, dk, dv = torch.autograd.grad(out, [q, k, v], s["do"])
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}


def _exact_attention(c, seed):
    q, k, v, do = _attention_inputs(c, seed)
    q, k, v = (t.to(F64).requires_grad_(True) for t in (q, k, v))
    out = _attend64(q, k, v, c["D"] ** -0.5, _lengths(c)).transpose(1, 2).reshape(do.shape)
    dq, dk, dv = torch.autograd.grad(out, [q, k, v], do.to(F64))
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}


# --------------------------------------------------------------- MLA layer
NOPE, ROPE, VDIM = 128, 64, 128
MLA_TARGETS = ("self_attn.q_a_proj", "self_attn.q_b_proj", "self_attn.kv_a_proj_with_mqa",
               "self_attn.kv_b_proj", O)


def _mla_shapes(c):
    H, heads = c["H"], c["heads"]
    return {"self_attn.q_a_proj": (c["q_rank"], H),
            "self_attn.q_b_proj": (heads * (NOPE + ROPE), c["q_rank"]),
            "self_attn.kv_a_proj_with_mqa": (c["kv_rank"] + ROPE, H),
            "self_attn.kv_b_proj": (heads * (NOPE + VDIM), c["kv_rank"]),
            O: (H, heads * VDIM), GATE: (c["I"], H), UP: (c["I"], H), DOWN: (H, c["I"])}


def _mla_inputs(c, seed):
    g = _gen(seed)
    w = {n: (*_quantise(g, s[0] * s[1], "nf4-g128"), s) for n, s in _mla_shapes(c).items()}
    norms = {n: (1 + _randn(g, d, std=0.05, dtype=F32)).to(BF) for n, d in (
        ("input_layernorm.weight", c["H"]), ("post_attention_layernorm.weight", c["H"]),
        ("self_attn.q_a_layernorm.weight", c["q_rank"]),
        ("self_attn.kv_a_layernorm.weight", c["kv_rank"]))}
    ab = {t: _adapter(g, c["rank"], _mla_shapes(c)[t][1], _mla_shapes(c)[t][0])
          for t in MLA_TARGETS}
    return w, norms, ab, _randn(g, c["B"], c["S"], c["H"]), _randn(g, c["B"], c["S"], c["H"])


def _yarn_scale():
    m = 0.1 * math.log(YARN["factor"]) + 1.0
    return (NOPE + ROPE) ** -0.5 * m * m


def _prepare_mla(c, seed):
    from spilltune_amd import deepseek, slots
    w, norms, ab, x, dy = _mla_inputs(c, seed)
    weights = {f"{n}.weight": _record(s, "nf4-g128", p, sc) for n, (p, sc, s) in w.items()}
    weights.update({n: t.cpu() for n, t in norms.items()})
    params = {"heads": c["heads"], "nope": NOPE, "rope": ROPE, "value": VDIM,
              "kv_rank": c["kv_rank"], "q_rank": c["q_rank"], "eps": 1e-6,
              "attention_scale": deepseek.attention_scale(NOPE, ROPE, YARN), "interleave": True,
              "moe": False}
    block = deepseek.make_deepseek_block(0, weights, codec="nf4-g128", parameters=params,
                                         rank=c["rank"], alpha=2.0 * c["rank"], device=_dev())
    with torch.no_grad():
        for t, p in block.adapters.items():
            p.A.copy_(ab[t][0])
            p.B.copy_(ab[t][1])
    rot, mask = deepseek.positions_and_masks(torch.ones(c["B"], c["S"], dtype=torch.bool),
                                             rope=YARN, rope_dim=ROPE, device=_dev())
    return {"blocks": [block], "session": slots.ResidentSession([block], _dev()), "rot": rot,
            "mask": mask, "x": x, "dy": dy}


def _yarn_tables(S):
    """YaRN's frequencies: a ramp from interpolated to plain between the
    dimensions that turn beta_fast and beta_slow times over the original
    context; its amplitude is 1 (mscale and mscale_all_dim are equal)."""
    base, orig = YARN["rope_theta"], YARN["original_max_position_embeddings"]
    freq = base ** (torch.arange(0, ROPE, 2, device=_dev()).float() / ROPE)

    def dim_of(turns):
        return ROPE * math.log(orig / (turns * 2 * math.pi)) / (2 * math.log(base))
    lo, hi = math.floor(dim_of(YARN["beta_fast"])), math.ceil(dim_of(YARN["beta_slow"]))
    lo, hi = max(lo, 0), min(hi, ROPE - 1)
    ramp = ((torch.arange(ROPE // 2, device=_dev()).float() - lo) / (hi - lo)).clamp(0, 1)
    keep = 1 - ramp
    return _tables(S, ROPE, (1.0 / (YARN["factor"] * freq)) * (1 - keep) + (1.0 / freq) * keep)


def _exact_mla(c, seed):
    w, norms, ab, x, dy = _mla_inputs(c, seed)
    B, S, H = x.shape
    heads = c["heads"]
    cos, sin = _yarn_tables(S)
    W = {n: _decode64(p, sc, s, "nf4-g128") for n, (p, sc, s) in w.items()}
    leaves = {"x": x.to(F64).requires_grad_(True)}
    L = {}
    for t, (a, b) in ab.items():
        L[t] = (a.to(F64).requires_grad_(True), b.to(F64).requires_grad_(True))
        leaves[f"0:{t}.A"], leaves[f"0:{t}.B"] = L[t]
    h = leaves["x"]

    def pairs(t):  # interleaved pairs to halves, then the rotation
        d = t.shape[-1]
        t = t.view(*t.shape[:-1], d // 2, 2).transpose(-1, -2).reshape(t.shape)
        return _rotate64(t, cos, sin)
    xn = _rms64(h, norms["input_layernorm.weight"], 1e-6)
    qa = _lin64(xn, W["self_attn.q_a_proj"], L["self_attn.q_a_proj"])
    comp = _lin64(xn, W["self_attn.kv_a_proj_with_mqa"], L["self_attn.kv_a_proj_with_mqa"])
    q = _lin64(_rms64(qa, norms["self_attn.q_a_layernorm.weight"], 1e-6),
               W["self_attn.q_b_proj"], L["self_attn.q_b_proj"])
    kvn = _rms64(comp[..., :c["kv_rank"]], norms["self_attn.kv_a_layernorm.weight"], 1e-6)
    kv = _lin64(kvn, W["self_attn.kv_b_proj"], L["self_attn.kv_b_proj"])
    q = q.view(B, S, heads, NOPE + ROPE).transpose(1, 2)
    kv = kv.view(B, S, heads, NOPE + VDIM).transpose(1, 2)
    kr = pairs(comp[..., c["kv_rank"]:].unsqueeze(1)).expand(B, heads, S, ROPE)
    Qh = torch.cat((q[..., :NOPE], pairs(q[..., NOPE:])), -1)
    Kh = torch.cat((kv[..., :NOPE], kr), -1)
    a = _attend64(Qh, Kh, kv[..., NOPE:], _yarn_scale())
    h = h + _lin64(a.transpose(1, 2).reshape(B, S, heads * VDIM), W[O], L[O])
    xn = _rms64(h, norms["post_attention_layernorm.weight"], 1e-6)
    h = h + (F.silu(xn @ W[GATE].t()) * (xn @ W[UP].t())) @ W[DOWN].t()
    grads = dict(zip(leaves, torch.autograd.grad(h, list(leaves.values()), dy.to(F64))))
    return {"out": h.detach(), "dx": grads.pop("x"), **grads}


# --------------------------------------------------------------- MoE
def _moe_inputs(c, seed):
    g = _gen(seed)
    H, I, E, T, r = c["H"], c["I"], c["E"], c["T"], c["rank"]
    deep = c["kind"] == "deepseek_moe"
    router = _randn(g, E, H, std=H ** -0.5)
    bias = _randn(g, E, std=0.01, dtype=F32)
    gu, dn = _quantise(g, E * 2 * I * H, "nf4-g128"), _quantise(g, E * H * I, "nf4-g128")
    lora = {}
    if deep:
        sgu, sdn = _quantise(g, 2 * I * H, "nf4-g128"), _quantise(g, H * I, "nf4-g128")
        lora = {"gate": _adapter(g, r, H, I), "up": _adapter(g, r, H, I),
                "down": _adapter(g, r, I, H)}
    else:
        sgu = sdn = None
        if r:
            lora = {"gu": (_randn(g, E, 2 * r, H, std=0.02, dtype=F32),
                           _randn(g, E, 2 * I, r, std=0.02, dtype=F32)),
                    "down": (_randn(g, E, r, I, std=0.02, dtype=F32),
                             _randn(g, E, H, r, std=0.02, dtype=F32))}
    return router, bias, gu, dn, sgu, sdn, lora, _randn(g, T, H), _randn(g, T, H)


def _prepare_moe(c, seed):
    from spilltune_amd import moe, ops
    router, bias, gu, dn, sgu, sdn, lora, x, dy = _moe_inputs(c, seed)
    H, I, E, r = c["H"], c["I"], c["E"], c["rank"]
    weights = {"mlp.gate.weight": router,
               "mlp.experts.gate_up_proj": moe.Q4Experts(*gu, E, 2 * I, H, "nf4-g128"),
               "mlp.experts.down_proj": moe.Q4Experts(*dn, E, H, I, "nf4-g128")}
    state = {"c": dict(c), "w": weights, "x": x, "dy": dy, "leaves": {}}
    if c["kind"] == "deepseek_moe":
        weights["mlp.gate.e_score_correction_bias"] = bias
        hp, hs = I * H // 2, I * H // 128
        pre = "mlp.shared_experts."
        weights[pre + "gate_proj.weight"] = ops.Q4Weight(sgu[0][:hp], sgu[1][:hs], (I, H), "nf4-g128")
        weights[pre + "up_proj.weight"] = ops.Q4Weight(sgu[0][hp:], sgu[1][hs:], (I, H), "nf4-g128")
        weights[pre + "down_proj.weight"] = ops.Q4Weight(*sdn, (H, I), "nf4-g128")
        state["shared"] = {n: _Lora(a.requires_grad_(True), b.requires_grad_(True), r)
                           for n, (a, b) in lora.items()}
        for n, l in state["shared"].items():
            state["leaves"][n + ".A"], state["leaves"][n + ".B"] = l.A, l.B
    elif r:
        mk = lambda n, fin, fout, seg, ab: moe.ExpertLoRA(  # noqa: E731
            n, r, 2.0 * r, E, fin, fout, seg, ab[0], ab[1])
        state["gu"] = mk("mlp.experts.gate_up_proj", H, 2 * I, 2, lora["gu"])
        state["down"] = mk("mlp.experts.down_proj", I, H, 1, lora["down"])
        for n in ("gu", "down"):
            state["leaves"][n + ".A"], state["leaves"][n + ".B"] = state[n].A, state[n].B
    return state


def _run_moe(s):
    from spilltune_amd import moe
    c = s["c"]
    x = s["x"].detach().requires_grad_(True)
    if c["kind"] == "deepseek_moe":
        out = moe.deepseek_moe_feed_forward(
            x, s["w"], num_experts=c["E"], top_k=c["k"], groups=c["groups"],
            group_k=c["group_k"], normalize=True, scale=2.5, lora_shared=s["shared"])
    else:
        out = moe.moe_feed_forward(x, s["w"], num_experts=c["E"], top_k=c["k"],
                                   norm_topk_prob=True, lora_gate_up=s.get("gu"),
                                   lora_down=s.get("down"))
    grads = torch.autograd.grad(out, [x, *s["leaves"].values()], s["dy"])
    return {"out": out.detach(), "dx": grads[0], **dict(zip(s["leaves"], grads[1:]))}


def _exact_moe(c, seed):
    router, bias, gu, dn, sgu, sdn, lora, x, dy = _moe_inputs(c, seed)
    H, I, E, T, k = c["H"], c["I"], c["E"], c["T"], c["k"]
    deep = c["kind"] == "deepseek_moe"
    leaves = {"x": x.to(F64).requires_grad_(True)}
    L = {}
    for n, (a, b) in lora.items():
        L[n] = (a.to(F64).requires_grad_(True), b.to(F64).requires_grad_(True))
        leaves[n + ".A"], leaves[n + ".B"] = L[n]
    # routing on a leaf of its own: its gradient is added to the experts' below
    logits = leaves["x"] @ router.to(F64).t()
    with torch.no_grad():  # the picks, as the stored types decide them
        if deep:
            pick = torch.sigmoid(logits) + bias.to(F64)
            best = pick.view(T, c["groups"], -1).topk(2, -1)[0].sum(-1)
            allowed = torch.zeros_like(best, dtype=torch.bool).scatter_(
                1, best.topk(c["group_k"], -1)[1], True)
            pick = pick.masked_fill(~allowed.repeat_interleave(E // c["groups"], 1), -1e300)
            idx = pick.topk(k, -1)[1]
        else:  # bf16 logits: ties go to the lower expert
            idx = torch.sort(logits.to(BF).to(F64), dim=-1, descending=True, stable=True)[1][:, :k]
    if deep:
        wts = torch.sigmoid(logits).gather(1, idx)
        wts = 2.5 * wts / wts.sum(-1, keepdim=True)
    else:
        wts = torch.softmax(logits, -1).gather(1, idx)
        wts = wts / wts.sum(-1, keepdim=True)
    g_out = dy.to(F64)
    grads = {n: torch.zeros_like(t) for n, t in leaves.items()}
    out = torch.zeros(T, H, dtype=F64, device=_dev())
    wleaf = wts.detach().requires_grad_(True)
    gw = torch.zeros_like(wts)
    for e in range(E):
        tok, slot = (idx == e).nonzero(as_tuple=True)
        if not tok.numel():
            continue
        ge = slice(e * 2 * I * H // 2, (e + 1) * 2 * I * H // 2)
        gs = slice(e * 2 * I * H // 128, (e + 1) * 2 * I * H // 128)
        de = slice(e * I * H // 2, (e + 1) * I * H // 2)
        ds = slice(e * I * H // 128, (e + 1) * I * H // 128)
        Wg = _decode64(gu[0][ge], gu[1][gs], (2 * I, H), "nf4-g128")
        Wd = _decode64(dn[0][de], dn[1][ds], (H, I), "nf4-g128")
        xe = leaves["x"].detach()[tok].requires_grad_(True)
        y = xe @ Wg.t()
        own = []
        if "gu" in L:
            r = c["rank"]
            own = [t.detach()[e].requires_grad_(True) for n in ("gu", "down") for t in L[n]]
            A, B, Ad, Bd = own
            y = y + 2.0 * torch.cat((xe @ A[:r].t() @ B[:I].t(), xe @ A[r:].t() @ B[I:].t()), 1)
        act = F.silu(y[:, :I]) * y[:, I:]
        z = act @ Wd.t()
        if own:
            z = z + 2.0 * act @ Ad.t() @ Bd.t()
        wl = wleaf[tok, slot].detach().requires_grad_(True)
        z = z * wl[:, None]
        out.index_add_(0, tok, z.detach())
        got = torch.autograd.grad(z, [xe, wl, *own], g_out[tok])
        grads["x"].index_add_(0, tok, got[0])
        gw[tok, slot] = got[1]
        if own:
            for n, t in zip(("gu.A", "gu.B", "down.A", "down.B"), got[2:]):
                grads[n][e] = t
    (gr,) = torch.autograd.grad(wts, [leaves["x"]], gw)
    grads["x"] += gr
    if deep:
        Wg = _decode64(*sgu, (2 * I, H), "nf4-g128")
        Wd = _decode64(*sdn, (H, I), "nf4-g128")
        xs = leaves["x"]
        act = F.silu(_lin64(xs, Wg[:I], L["gate"])) * _lin64(xs, Wg[I:], L["up"])
        z = _lin64(act, Wd, L["down"])
        got = torch.autograd.grad(z, list(leaves.values()), g_out)
        out += z.detach()
        for n, t in zip(leaves, got):
            grads[n] += t
    return {"out": out, "dx": grads.pop("x"), **grads}


# --------------------------------------------------------------- terminal
def _terminal_inputs(c, seed):
    g = _gen(seed)
    S, H, Vv = c["S"], c["H"], c["V"]
    h = _randn(g, 1, S, H)
    norm = (1 + _randn(g, H, std=0.05, dtype=F32)).to(BF)
    head = _randn(g, Vv, H, std=0.02)
    labels = torch.randint(0, Vv, (1, S), device=_dev(), generator=g)
    labels[:, : S // 8] = -100  # the prompt's tokens are not supervised
    return h, norm, head, labels


def _prepare_terminal(c, seed):
    h, norm, head, labels = _terminal_inputs(c, seed)
    labels = labels.cpu()
    return {"h": h, "norm": norm, "head": head, "labels": labels, "chunk": c["chunk"],
            "count": int((labels[:, 1:] != -100).sum())}


def _run_terminal(s):
    from spilltune_amd import ops
    h = s["h"].detach().requires_grad_(True)
    B, S, H = h.shape
    normalized = ops.rms_norm(h.reshape(B * S, H), s["norm"], 1e-6).view(B, S, H)
    loss = ops.chunked_causal_loss(
        normalized, s["head"], s["labels"], normalization=s["count"], token_chunk=s["chunk"],
        supervised_chunks=ops.supervised_chunk_intervals(s["labels"], s["chunk"]))
    (g,) = torch.autograd.grad(loss, h)
    return {"loss": loss.detach(), "dh": g}


def _exact_terminal(c, seed):
    h, norm, head, labels = _terminal_inputs(c, seed)
    h = h.to(F64).requires_grad_(True)
    n = _rms64(h, norm, 1e-6)[0, :-1]
    target = labels[0, 1:]
    count = int((target != -100).sum())
    W = head.to(F64)
    loss, gn = torch.zeros((), dtype=F64, device=_dev()), torch.zeros_like(n)
    for at in range(0, n.shape[0], 1024):
        leaf = n[at:at + 1024].detach().requires_grad_(True)
        part = F.cross_entropy(leaf @ W.t(), target[at:at + 1024], ignore_index=-100,
                               reduction="sum") / count
        (gn[at:at + 1024],) = torch.autograd.grad(part, leaf)
        loss += part.detach()
    (g,) = torch.autograd.grad(n, h, gn)
    return {"loss": loss, "dh": g}


# --------------------------------------------------------------- the interface
_PREPARE = {"layer": _prepare_layer, "linear": _prepare_linear, "nf4_state": _prepare_nf4,
            "attention": _prepare_attention, "mla": _prepare_mla, "moe": _prepare_moe,
            "deepseek_moe": _prepare_moe, "terminal": _prepare_terminal}
_RUN = {"layer": _run_layer, "linear": _run_linear, "nf4_state": _run_nf4,
        "attention": _run_attention, "mla": _run_layer, "moe": _run_moe,
        "deepseek_moe": _run_moe, "terminal": _run_terminal}
_EXACT = {"layer": _exact_layer, "linear": _exact_linear, "nf4_state": _exact_nf4,
          "attention": _exact_attention, "mla": _exact_mla, "moe": _exact_moe,
          "deepseek_moe": _exact_moe, "terminal": _exact_terminal}


def prepare(case, seed):
    return {"kind": case["kind"], "state": _PREPARE[case["kind"]](case, seed)}


def run(state):
    return _RUN[state["kind"]](state["state"])


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


Q4BYTES = 0.5 + 4 / 128  # a code and its share of the scale


def work(case):
    """Bytes: weights, inputs, upstream gradients read once and outputs written
    once.  Flops: the products of the forward, the recomputation that the
    layer step is defined by, and the input and adapter gradients."""
    c, kind = case, case["kind"]
    if kind in ("layer", "mla"):
        shapes = _layer_shapes(c) if kind == "layer" else _mla_shapes(c)
        M, P = c["B"] * c["S"], sum(n * k for n, k in shapes.values())
        targets = MLA_TARGETS if kind == "mla" else ALL7 if c["targets"] == "all" else QVO
        nk = sum(sum(shapes[t]) for t in targets)
        dq, dv = (NOPE + ROPE, VDIM) if kind == "mla" else (c["D"], c["D"])
        # causal half; QK and PV twice (forward, recomputation), five products backward
        pairs = c["B"] * c["heads"] * c["S"] ** 2 / 2
        att = pairs * 2 * (2 * (dq + dv) + 3 * dq + 2 * dv)
        n = c.get("layers", 1)
        flops = n * (6 * M * P + att + 2 * M * c["rank"] * nk * 4)
        return {"bytes": n * (P * Q4BYTES + 8 * c["rank"] * nk) + 8 * M * c["H"], "flops": flops}
    if kind in ("linear", "nf4_state"):
        M, N, Kd = c["M"], c["N"], c["K"]
        r = c.get("rank", 0)
        q = Q4BYTES if kind == "linear" else 0.5 + 4 / 64
        res = 2 * M * N if c.get("residual") else 0
        return {"bytes": N * Kd * q + 4 * M * (N + Kd) + res + 8 * r * (N + Kd),
                "flops": 4 * M * N * Kd + 8 * M * r * (N + Kd)}
    if kind == "attention":
        B, S, D = c["B"], c["S"], c["D"]
        pairs = B * c["heads"] * S * S / 2
        return {"bytes": 2 * B * S * D * (4 * c["heads"] + 4 * c["kv"]), "flops": pairs * 2 * 7 * D}
    if kind in ("moe", "deepseek_moe"):
        H, I, T, r = c["H"], c["I"], c["T"], c["rank"]
        R, nk = T * c["k"], (H + 2 * I) + (I + H)
        hit = min(c["E"], R)  # experts that can be hit
        flops = 4 * R * 3 * H * I + 4 * T * H * c["E"]
        wbytes = hit * 3 * H * I * Q4BYTES
        if kind == "deepseek_moe":
            return {"bytes": wbytes + 8 * T * H + 3 * H * I * Q4BYTES + 8 * r * nk,
                    "flops": flops + 4 * T * 3 * H * I + 8 * T * r * nk}
        return {"bytes": wbytes + 8 * T * H + 8 * c["E"] * r * nk, "flops": flops + 8 * R * r * nk}
    S, H, Vv = c["S"], c["H"], c["V"]
    return {"bytes": 2 * Vv * H + 4 * S * H, "flops": 4 * S * H * Vv}


def tolerance(case):
    """About four times what the path differs by from ``exact``: bf16 results
    of fp32 sums, the layers' through several roundings."""
    return {"layer": {"rel": 0.03}, "mla": {"rel": 0.03}, "linear": {"rel": 0.01},
            "nf4_state": {"rel": 0.01}, "attention": {"rel": 0.01}, "moe": {"rel": 0.02},
            "deepseek_moe": {"rel": 0.02}, "terminal": {"rel": 0.015}}[case["kind"]]
