"""Performance cases of the Gated DeltaNet path and the attention ops beside it.

Each case is one call of a public entry point as a serving program makes it:
prompts (prefill), chunks of prompts over a cached prefix, decode steps, and the
whole layer.  Sizes are those of the benchmark and the tests of this
repository (GDN heads 16 / 32 of 128, hidden 2048, attention heads 16 / 2 of
256, vision heads of 72, 16-token pages) and of one tensor-parallel half of
them.  ``listed()`` holds the fixed cases, ``draw`` more of the same ranges.

Inputs are drawn on the GPU from the seed alone.  ``exact`` restates each op
in float64 with plain torch, without this repository's code and without the
roundings between the stages of a layer.
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
CONV_W = 4
HEAD = 128  # GDN head dim
PAGE = 16


def listed() -> list[dict]:
    return [
        # one user's chat: a decode step of one sequence through a GDN layer, where latency and launches count
        dict(name="layer_decode_1", kind="layer", seqs=0, lo=0, hi=0, len_seed=0, decode=1, slots=16, hk=16, hv=32),
        # an ordinary serving batch's decode step through a GDN layer
        dict(name="layer_decode_64", kind="layer", seqs=0, lo=0, hi=0, len_seed=0, decode=64, slots=96, hk=16, hv=32),
        # a scheduler's mixed batch: four prompts and the decode tokens of the running sequences in one call
        dict(name="layer_mixed", kind="layer", seqs=4, lo=2048, hi=2048, len_seed=0, decode=128, slots=160, hk=16,
             hv=32),
        # one prompt of ordinary length through the chunked rule, odd size
        dict(name="gdn_prefill_1", kind="gdn_prefill", seqs=1, lo=2943, hi=2943, len_seed=0, hk=16, hv=32,
             dtype="bf16"),
        # a full prefill batch of ragged prompts (the benchmark's headline range)
        dict(name="gdn_prefill_16", kind="gdn_prefill", seqs=16, lo=512, hi=4096, len_seed=3, hk=16, hv=32,
             dtype="bf16"),
        # many one-chunk pieces, as a chunked-prefill scheduler with a small budget sends them
        dict(name="gdn_prefill_short", kind="gdn_prefill", seqs=512, lo=64, hi=64, len_seed=0, hk=16, hv=32,
             dtype="bf16"),
        # the recurrent decode step of a large batch
        dict(name="gdn_decode_256", kind="gdn_decode", seqs=256, hk=16, hv=32, dtype="bf16"),
        # the convolution of a prefill batch
        dict(name="conv_prefill", kind="conv_prefill", seqs=8, lo=256, hi=4096, len_seed=5, channels=8192,
             dtype="bf16"),
        # an attention layer's prefill of ragged prompts
        dict(name="attn_prefill_16", kind="attn_prefill", seqs=16, lo=512, hi=4096, len_seed=3, hq=16, hkv=2, dim=256,
             causal=True, dtype="bf16"),
        # the vision tower: images of different sizes, bidirectional, head dim 72
        dict(name="attn_vision", kind="attn_prefill", seqs=6, lo=256, hi=4096, len_seed=7, hq=16, hkv=16, dim=72,
             causal=False, dtype="bf16"),
        # chunks of long prompts over what is already in the paged cache
        dict(name="attn_paged_prefill", kind="attn_paged_prefill", seqs=4, lo=256, hi=2048, prefix=16384, len_seed=9,
             hq=16, hkv=2, dim=256, dtype="bf16"),
        # decode of a batch with long, uneven contexts
        dict(name="attn_decode_32", kind="attn_decode", seqs=32, lo=1024, hi=16384, len_seed=11, hq=16, hkv=2,
             dim=256, dtype="bf16"),
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    """A whole number in [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng: random.Random) -> dict:
    """One more case.  Token counts stay at or below the listed cases'."""
    kind = rng.choice(["layer_decode", "layer_mixed", "gdn_prefill", "gdn_prefill", "gdn_short", "gdn_decode",
                       "conv_prefill", "attn_prefill", "vision", "attn_paged_prefill", "attn_decode", "attn_decode"])
    hk, hv = rng.choice([(16, 32), (16, 32), (16, 32), (8, 16), (16, 16)])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    ls = rng.randrange(1 << 20)
    if kind == "layer_decode":
        n = _log(rng, 1, 256)
        return dict(kind="layer", seqs=0, lo=0, hi=0, len_seed=ls, decode=n, slots=n + rng.randint(0, 64), hk=hk,
                    hv=hv)
    if kind == "layer_mixed":
        hi = _log(rng, 64, 4096)
        seqs = max(1, min(_log(rng, 1, 16), 8192 // hi))
        n = rng.choice([0, _log(rng, 1, 128)])
        return dict(kind="layer", seqs=seqs, lo=max(1, hi // 4), hi=hi, len_seed=ls, decode=n,
                    slots=seqs + n + rng.randint(0, 32), hk=hk, hv=hv)
    if kind == "gdn_prefill":
        hi = _log(rng, 128, 8192)
        seqs = max(1, min(_log(rng, 1, 16), 32768 // hi))
        return dict(kind="gdn_prefill", seqs=seqs, lo=max(1, hi // 8), hi=hi, len_seed=ls, hk=hk, hv=hv,
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]) if seqs * hi <= 8192 else dtype)
    if kind == "gdn_short":
        hi = _log(rng, 16, 256)
        seqs = max(1, min(_log(rng, 16, 512), 32768 // hi))
        return dict(kind="gdn_prefill", seqs=seqs, lo=1, hi=hi, len_seed=ls, hk=hk, hv=hv, dtype=dtype)
    if kind == "gdn_decode":
        return dict(kind="gdn_decode", seqs=_log(rng, 1, 256), hk=hk, hv=hv, dtype=dtype)
    if kind == "conv_prefill":
        hi = _log(rng, 64, 4096)
        seqs = max(1, min(_log(rng, 1, 32), 20480 // hi))
        return dict(kind="conv_prefill", seqs=seqs, lo=max(1, hi // 16), hi=hi, len_seed=ls,
                    channels=2 * hk * HEAD + hv * HEAD, dtype=dtype)
    if kind == "attn_prefill":
        hi = _log(rng, 64, 8192)
        seqs = max(1, min(_log(rng, 1, 16), 32768 // hi, 80_000_000 // (hi * hi)))
        hq, hkv, dim = rng.choice([(16, 2, 256), (16, 2, 256), (8, 1, 256), (16, 4, 128), (16, 16, 64)])
        return dict(kind="attn_prefill", seqs=seqs, lo=max(1, hi // 8), hi=hi, len_seed=ls, hq=hq, hkv=hkv, dim=dim,
                    causal=True, dtype=dtype)
    if kind == "vision":
        hi = _log(rng, 64, 4096)
        seqs = max(1, min(_log(rng, 1, 16), 16384 // hi))
        return dict(kind="attn_prefill", seqs=seqs, lo=max(1, hi // 4), hi=hi, len_seed=ls, hq=16, hkv=16, dim=72,
                    causal=False, dtype=dtype)
    hq, hkv, dim = rng.choice([(16, 2, 256), (16, 2, 256), (8, 1, 256), (16, 4, 128)])
    if kind == "attn_paged_prefill":
        hi, prefix = _log(rng, 16, 2048), _log(rng, 64, 16384)
        seqs = max(1, min(_log(rng, 1, 16), 45_000_000 // (hi * (prefix + hi))))
        return dict(kind="attn_paged_prefill", seqs=seqs, lo=max(1, hi // 8), hi=hi, prefix=prefix, len_seed=ls,
                    hq=hq, hkv=hkv, dim=dim, dtype=dtype)
    hi = _log(rng, 64, 32768)
    seqs = max(1, min(_log(rng, 1, 256), 524288 // hi))
    return dict(kind="attn_decode", seqs=seqs, lo=max(1, hi // 8), hi=hi, len_seed=ls, hq=hq, hkv=hkv, dim=dim,
                dtype=dtype)


# ---- sizes ---------------------------------------------------------------------------


def _lengths(c: dict) -> list[int]:
    r = random.Random(c["len_seed"])
    return [r.randint(c["lo"], c["hi"]) for _ in range(c["seqs"])]


def _prefixes(c: dict) -> list[int]:
    r = random.Random(c["len_seed"] + 1)
    return [r.randint(0, c["prefix"]) for _ in range(c["seqs"])]


def _cu(lens: list[int]) -> list[int]:
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu


# ---- inputs --------------------------------------------------------------------------


class _Inputs:
    """Seeded draws on the GPU."""

    def __init__(self, seed: int):
        self.dev = torch.device("cuda:0")
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)
        self.cpu = random.Random(seed)

    def normal(self, *shape, std: float = 1.0) -> torch.Tensor:
        return torch.randn(*shape, generator=self.gen, device=self.dev) * std

    def slots(self, n: int, of: int) -> torch.Tensor:
        return torch.tensor(self.cpu.sample(range(of), n), dtype=torch.int32, device=self.dev)

    def ints(self, values) -> torch.Tensor:
        return torch.tensor(values, dtype=torch.int32, device=self.dev)


def _gdn_qkvgb(i: _Inputs, T: int, c: dict):
    """Inputs as the layer makes them: q, k of unit norm, log-decay below zero, beta in (0, 1)."""
    dt = DTYPES[c["dtype"]]
    q = F.normalize(i.normal(T, c["hk"], HEAD), dim=-1).to(dt)
    k = F.normalize(i.normal(T, c["hk"], HEAD), dim=-1).to(dt)
    v = i.normal(T, c["hv"], HEAD).to(dt)
    g = -F.softplus(i.normal(T, c["hv"]))
    beta = torch.sigmoid(i.normal(T, c["hv"]))
    return q, k, v, g, beta


def _paged(i: _Inputs, c: dict, ctx: list[int], new: int):
    """A paged cache of exactly the pages these contexts take, pages in random order."""
    dt = DTYPES[c["dtype"]]
    pages = [-(-n // PAGE) for n in ctx]
    total = sum(pages) + 3
    kc = i.normal(total, PAGE, c["hkv"], c["dim"]).to(dt)
    vc = i.normal(total, PAGE, c["hkv"], c["dim"]).to(dt)
    order = list(range(total))
    i.cpu.shuffle(order)
    rows, at = [], 0
    for p in pages:
        rows.append(order[at: at + p] + [-1] * (max(pages) - p))
        at += p
    q = i.normal(new, c["hq"], c["dim"]).to(dt)
    return dict(q=q, k_cache=kc, v_cache=vc, tables=i.ints(rows), ctx=i.ints(ctx), scale=c["dim"] ** -0.5)


def _inputs(c: dict, seed: int) -> dict:
    i = _Inputs(seed)
    kind = c["kind"]
    if kind == "layer":
        hidden, hk, hv = 2048, c["hk"], c["hv"]
        lens = _lengths(c)
        T, conv = sum(lens) + c["decode"], (2 * hk + hv) * HEAD
        n = len(lens) + c["decode"]
        return dict(
            x=i.normal(T, hidden).bfloat16(),
            in_proj=i.normal(conv + hv * HEAD + 2 * hv, hidden, std=0.02).bfloat16(),
            conv_w=i.normal(conv, CONV_W, std=0.5).bfloat16(),
            out_proj=i.normal(hidden, hv * HEAD, std=0.02).bfloat16(),
            A_log=torch.log(torch.rand(hv, generator=i.gen, device=i.dev) * 15 + 1),
            dt_bias=torch.ones(hv, device=i.dev), norm_w=torch.ones(HEAD, device=i.dev),
            conv_state=i.normal(c["slots"], CONV_W - 1, conv).bfloat16(),
            state=i.normal(c["slots"], hv, HEAD, HEAD, std=0.1),
            conv_idx=i.slots(n, c["slots"]), idx=i.slots(n, c["slots"]), cu=i.ints(_cu(lens)))
    if kind == "gdn_prefill":
        lens = _lengths(c)
        q, k, v, g, beta = _gdn_qkvgb(i, sum(lens), c)
        slots = len(lens) + 4
        return dict(q=q, k=k, v=v, g=g, beta=beta, state=i.normal(slots, c["hv"], HEAD, HEAD, std=0.1),
                    idx=i.slots(len(lens), slots), cu=i.ints(_cu(lens)))
    if kind == "gdn_decode":
        n = c["seqs"]
        slots = n + 8
        q, k, v, g, beta = _gdn_qkvgb(i, n, c)
        return dict(q=q, k=k, v=v, g=g, beta=beta, state=i.normal(slots, c["hv"], HEAD, HEAD, std=0.1),
                    idx=i.slots(n, slots))
    if kind == "conv_prefill":
        dt, lens = DTYPES[c["dtype"]], _lengths(c)
        slots = len(lens) + 8
        return dict(x=i.normal(sum(lens), c["channels"]).to(dt), w=i.normal(c["channels"], CONV_W, std=0.5).to(dt),
                    state=i.normal(slots, CONV_W - 1, c["channels"]), idx=i.slots(len(lens), slots),
                    cu=i.ints(_cu(lens)))
    if kind == "attn_prefill":
        dt, lens = DTYPES[c["dtype"]], _lengths(c)
        T = sum(lens)
        return dict(q=i.normal(T, c["hq"], c["dim"]).to(dt), k=i.normal(T, c["hkv"], c["dim"]).to(dt),
                    v=i.normal(T, c["hkv"], c["dim"]).to(dt), cu=i.ints(_cu(lens)), scale=c["dim"] ** -0.5,
                    longest=max(lens))
    if kind == "attn_paged_prefill":
        lens = _lengths(c)
        d = _paged(i, c, [p + n for p, n in zip(_prefixes(c), lens)], sum(lens))
        return dict(d, cu=i.ints(_cu(lens)), longest=max(lens))
    if kind == "attn_decode":
        return _paged(i, c, _lengths(c), c["seqs"])
    raise ValueError(kind)


def prepare(case: dict, seed: int) -> dict:
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "layer":
        from myvllm_amd.cache import LinearAttentionCache
        from myvllm_amd.layer import GatedDeltaNet

        hk, hv = case["hk"], case["hv"]
        dev = s["x"].device
        layer = GatedDeltaNet(2048, hk, hv, HEAD, HEAD, CONV_W, device=dev)
        cache = LinearAttentionCache(1, case["slots"], CONV_W, HEAD, HEAD, hk, hv, torch.bfloat16, dev)
        with torch.no_grad():
            for p, name in ((layer.in_proj, "in_proj"), (layer.conv1d_weight, "conv_w"), (layer.out_proj, "out_proj"),
                            (layer.A_log, "A_log"), (layer.dt_bias, "dt_bias"), (layer.norm_weight, "norm_w")):
                p.copy_(s.pop(name))
        layer.conv_state, layer.recurrent_state = cache.layer(0)
        layer.conv_state.copy_(s.pop("conv_state"))
        layer.recurrent_state.copy_(s.pop("state"))
        s["layer"] = layer
    return s


def run(s: dict):
    import myvllm_amd as ops

    c = s["case"]
    kind = c["kind"]
    if kind == "layer":
        layer = s["layer"]
        with torch.no_grad():
            out = layer(s["x"], s["cu"], s["conv_idx"], s["idx"], num_decode_tokens=c["decode"])
        return {"out": out, "conv_state": layer.conv_state, "state": layer.recurrent_state}
    if kind == "gdn_prefill":
        o = ops.chunk_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], s["idx"], s["cu"])
        return {"o": o, "state": s["state"]}
    if kind == "gdn_decode":
        o = ops.recurrent_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], s["idx"])
        return {"o": o, "state": s["state"]}
    if kind == "conv_prefill":
        y = ops.causal_conv1d_fn(s["x"], s["w"], s["state"], s["idx"], s["cu"])
        return {"y": y, "state": s["state"]}
    if kind == "attn_prefill":
        return {"o": ops.flash_attention_prefill(s["q"], s["k"], s["v"], s["cu"], s["scale"], c["hq"], c["hkv"],
                                                 c["dim"], c["dim"], c["causal"], max_seqlen=s["longest"])}
    if kind == "attn_paged_prefill":
        return {"o": ops.paged_flash_attention_prefill(s["q"], s["k_cache"], s["v_cache"], s["tables"], s["ctx"],
                                                       s["cu"], None, s["scale"], PAGE, max_seqlen=s["longest"])}
    return {"o": ops.paged_flash_attention_decode(s["q"], s["k_cache"], s["v_cache"], s["tables"], s["ctx"],
                                                  s["scale"], PAGE)}


# ---- what a pass cannot do without ---------------------------------------------------


def _gdn_flops(T: int, hk: int, hv: int) -> int:
    """The chunked rule at 64-token chunks: K K^T and Q K^T per k-head; w, u, P v', w S, k^T v', q S per v-head."""
    C, D = 64, HEAD
    return 2 * T * (2 * C * D * hk + (2 * C * D + C * D + 3 * D * D) * hv)


def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    es = 4 if c.get("dtype") == "fp32" else 2
    if kind == "layer":
        hidden, hk, hv = 2048, c["hk"], c["hv"]
        lens, n = _lengths(c), c["decode"]
        T, conv = sum(lens) + n, (2 * hk + hv) * HEAD
        rows = conv + hv * HEAD + 2 * hv
        weights = (rows * hidden + hidden * hv * HEAD + conv * CONV_W) * 2
        states = (len(lens) + n) * (hv * HEAD * HEAD * 8 + (CONV_W - 1) * conv * 4)
        return {"bytes": weights + states + T * hidden * 4,
                "flops": 2 * T * hidden * (rows + hv * HEAD) + _gdn_flops(sum(lens), hk, hv)
                + n * 6 * hv * HEAD * HEAD}
    if kind in ("gdn_prefill", "gdn_decode"):
        hk, hv = c["hk"], c["hv"]
        n = c["seqs"]
        T = n if kind == "gdn_decode" else sum(_lengths(c))
        b = T * ((2 * hk + 2 * hv) * HEAD * es + hv * 8) + n * hv * HEAD * HEAD * 8
        return {"bytes": b, "flops": 6 * T * hv * HEAD * HEAD if kind == "gdn_decode" else _gdn_flops(T, hk, hv)}
    if kind == "conv_prefill":
        T, D = sum(_lengths(c)), c["channels"]
        return {"bytes": 2 * T * D * es + D * CONV_W * es + c["seqs"] * (CONV_W - 1) * D * 8,
                "flops": T * D * 2 * CONV_W}
    lens = _lengths(c)
    hq, hkv, D = c["hq"], c["hkv"], c["dim"]
    if kind == "attn_prefill":
        T = sum(lens)
        pairs = sum(n * (n + 1) // 2 if c["causal"] else n * n for n in lens)
        return {"bytes": T * (2 * hq + 2 * hkv) * D * es, "flops": 4 * D * hq * pairs}
    if kind == "attn_paged_prefill":
        T, pre = sum(lens), _prefixes(c)
        pairs = sum(n * p + n * (n + 1) // 2 for n, p in zip(lens, pre))
        keys = T + sum(pre)
        return {"bytes": (T * 2 * hq + keys * 2 * hkv) * D * es + keys // PAGE * 4, "flops": 4 * D * hq * pairs}
    keys = sum(lens)
    return {"bytes": (c["seqs"] * 2 * hq + keys * 2 * hkv) * D * es + keys // PAGE * 4, "flops": 4 * D * hq * keys}


def tolerance(case: dict) -> dict:
    """Relative error norms, about four times what the ops show against float64: they round their
    16-bit outputs (and attention its probabilities) once after float32 sums, 1.7e-3 to 2.3e-3 in
    bf16 and an eighth of it in fp16; fp32 runs on fp16 q and k, 2.2e-4; the layer rounds after
    every stage, 5e-3."""
    if case["kind"] == "layer":
        return {"rel": 2e-2, "max": 0.6}
    if case["dtype"] in ("fp16", "fp32"):
        return {"rel": 1.2e-3, "max": 4e-2}
    return {"rel": 8e-3, "max": 0.2}


# ---- the same in 64 bits -------------------------------------------------------------


def _delta_rule(q, k, v, g, beta, S, scale):
    """One sequence in chunks of 64: q, k (L, Hk, K), v (L, Hv, V), g, beta (L, Hv), S (Hv, K, V); o and S."""
    C, L, hv = 64, v.shape[0], v.shape[1]
    r = hv // q.shape[1]
    pad = -L % C

    def heads(x):  # (L, H, ...) -> (H, chunks, C, ...)
        x = torch.cat([x, x.new_zeros((pad,) + tuple(x.shape[1:]))]).unflatten(0, (-1, C))
        return x.movedim(2, 0).contiguous()

    Q = heads(q).repeat_interleave(r, 0)
    K = heads(k).repeat_interleave(r, 0)
    V, b = heads(v), heads(beta)
    gam = heads(g).cumsum(-1)
    Kt = K.transpose(-1, -2).contiguous()
    diff = gam[..., :, None] - gam[..., None, :]
    low = torch.ones(C, C, dtype=torch.bool, device=v.device).tril()
    dec = torch.exp(diff.masked_fill(~low, -math.inf))
    eye = torch.eye(C, dtype=v.dtype, device=v.device)
    A = (b[..., None] * (K @ Kt) * dec).tril(-1)
    # (I + A)^-1 of a nilpotent A: the product of (I + N^(2^j)) with N = -A, j = 0..5
    N = -A
    T = eye + N
    for _ in range(5):
        N = N @ N
        T = T + T @ N
    eg = torch.exp(gam)
    W = T @ ((b * eg)[..., None] * K)
    U = T @ (b[..., None] * V)
    P = (Q @ Kt) * dec
    last = gam[..., -1]
    Kd = (K * torch.exp(last[..., None] - gam)[..., None]).transpose(-1, -2).contiguous()
    Qe = Q * eg[..., None]
    O = torch.empty_like(V)
    for n in range(V.shape[1]):
        X = U[:, n] - W[:, n] @ S
        O[:, n] = scale * (Qe[:, n] @ S + P[:, n] @ X)
        S = torch.exp(last[:, n])[:, None, None] * S + Kd[:, n] @ X
    return O.flatten(1, 2)[:, :L].transpose(0, 1), S


def _rules(q, k, v, g, beta, state, slots, cu, scale):
    o = torch.zeros_like(v)
    if len(slots) > 1 and all(cu[n + 1] - cu[n] == cu[1] for n in range(len(slots))) and cu[1] <= 64:
        # equal one-chunk sequences side by side: sequences become heads of one call
        n, L = len(slots), cu[1]
        side = lambda x: x[:cu[-1]].unflatten(0, (n, L)).transpose(0, 1).flatten(1, 2)  # noqa: E731
        idx = torch.tensor(slots, device=v.device)
        oo, S = _delta_rule(side(q), side(k), side(v), side(g), side(beta), state[idx].flatten(0, 1), scale)
        o[:cu[-1]] = oo.unflatten(1, (n, -1)).transpose(0, 1).flatten(0, 1)
        state[idx] = S.unflatten(0, (n, -1))
        return o
    for n, slot in enumerate(slots):
        a, b = cu[n], cu[n + 1]
        o[a:b], state[slot] = _delta_rule(q[a:b], k[a:b], v[a:b], g[a:b], beta[a:b], state[slot], scale)
    return o


def _recurrent(q, k, v, g, beta, state, idx, scale):
    """One token of every sequence."""
    r = v.shape[1] // q.shape[1]
    q, k = q.repeat_interleave(r, 1), k.repeat_interleave(r, 1)
    i = idx.long()
    S = state[i] * torch.exp(g)[..., None, None]
    d = beta[..., None] * (v - (k[..., None] * S).sum(-2))
    S = S + k[..., None] * d[..., None, :]
    state[i] = S
    return ((q * scale)[..., None] * S).sum(-2)


def _conv(x, w, state, slots, cu):
    y = torch.zeros_like(x)
    W = w.shape[1]
    for n, slot in enumerate(slots):
        a, b = cu[n], cu[n + 1]
        xt = torch.cat([state[slot], x[a:b]])
        acc = sum(w[:, j] * xt[j: j + b - a] for j in range(W))
        y[a:b] = F.silu(acc)
        state[slot] = xt[-(W - 1):]
    return y


def _attend(q, k, v, scale, causal):
    """q (n, Hq, D) at the last n of the m keys k, v (m, Hkv, D)."""
    n, hq, _ = q.shape
    m, hkv, _ = k.shape
    o = torch.empty_like(q)
    r = hq // hkv
    for h in range(hkv):
        kt = k[:, h].t().contiguous()
        vh = v[:, h].contiguous()
        for a in range(0, n, 1024):
            e = min(n, a + 1024)
            s = (q[a:e, h * r: (h + 1) * r].reshape(-1, q.shape[-1]) @ kt).unflatten(0, (e - a, r)) * scale
            if causal:
                pos = torch.arange(a, e, device=q.device) + (m - n)
                s = s.masked_fill((torch.arange(m, device=q.device) > pos[:, None])[:, None], -math.inf)
            p = torch.softmax(s, -1)
            o[a:e, h * r: (h + 1) * r] = (p.flatten(0, 1) @ vh).unflatten(0, (e - a, r))
    return o


def exact(case: dict, seed: int):
    c, kind = case, case["kind"]
    s = {k: v.double() if isinstance(v, torch.Tensor) and v.is_floating_point() else v
         for k, v in _inputs(case, seed).items()}
    scale = HEAD ** -0.5
    if kind == "gdn_prefill":
        o = _rules(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], s["idx"].tolist(), s["cu"].tolist(), scale)
        return {"o": o, "state": s["state"]}
    if kind == "gdn_decode":
        o = _recurrent(s["q"], s["k"], s["v"], s["g"], s["beta"], s["state"], s["idx"], scale)
        return {"o": o, "state": s["state"]}
    if kind == "conv_prefill":
        y = _conv(s["x"], s["w"], s["state"], s["idx"].tolist(), s["cu"].tolist())
        return {"y": y, "state": s["state"]}
    if kind == "attn_prefill":
        cu = s["cu"].tolist()
        return {"o": torch.cat([_attend(s["q"][a:b], s["k"][a:b], s["v"][a:b], s["scale"], c["causal"])
                                for a, b in zip(cu, cu[1:])])}
    if kind in ("attn_paged_prefill", "attn_decode"):
        cu = s["cu"].tolist() if "cu" in s else list(range(c["seqs"] + 1))
        out = []
        for n, m in enumerate(s["ctx"].tolist()):
            pages = s["tables"][n, : -(-m // PAGE)].long()
            k, v = (s[x][pages].flatten(0, 1)[:m] for x in ("k_cache", "v_cache"))
            out.append(_attend(s["q"][cu[n]: cu[n + 1]], k, v, s["scale"], True))
        return {"o": torch.cat(out)}
    # the layer
    hk, hv, n = c["hk"], c["hv"], c["decode"]
    cu = s["cu"].tolist()
    Tp, Np = cu[-1], len(cu) - 1
    kd, vd = hk * HEAD, hv * HEAD
    qkv, z, b, a = torch.split(s["x"] @ s["in_proj"].t().contiguous(), [2 * kd + vd, vd, hv, hv], dim=1)
    g = -torch.exp(s["A_log"]) * F.softplus(a + s["dt_bias"])
    beta = torch.sigmoid(b)
    cslots, slots = s["conv_idx"].tolist(), s["idx"].tolist()
    y = _conv(qkv, s["conv_w"], s["conv_state"], cslots, cu + [Tp + 1 + j for j in range(n)])
    q, k, v = torch.split(y, [kd, kd, vd], dim=1)
    l2 = lambda t: t * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k, v = l2(q.unflatten(1, (hk, HEAD))), l2(k.unflatten(1, (hk, HEAD))), v.unflatten(1, (hv, HEAD))
    o = torch.empty_like(v)
    if Np:
        o[:Tp] = _rules(q[:Tp], k[:Tp], v[:Tp], g[:Tp], beta[:Tp], s["state"], slots[:Np], cu, scale)
    if n:
        o[Tp:] = _recurrent(q[Tp:], k[Tp:], v[Tp:], g[Tp:], beta[Tp:], s["state"], s["idx"][Np:], scale)
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-6) * s["norm_w"] * F.silu(z.unflatten(1, (hv, HEAD)))
    return {"out": o.flatten(1) @ s["out_proj"].t().contiguous(), "conv_state": s["conv_state"], "state": s["state"]}
