"""Performance cases: the calls a program that keeps its KV cache packed makes, over the sizes it makes them at.

Every case goes through the public Python API (``torque_hip``): the cache classes, the packed-attention operators
and the attention adapter.  ``kind`` names the call:

* ``decode``: ``TorqueKVCacheMLX.decode_mlx`` over a filled cache, one query token for all layers and heads -- the
  call of the synthetic and qwen-decode benchmarks and of every decoded token;
* ``append_decode``: one decode step of a loop, the new token packed and attended to in the same call
  (``ops.packed_decode_append``, which the adapter's one-token step and ``decode_append`` make);
* ``prefill``: a prompt's keys and values into a cache that is used again (``reset`` and ``append_many_mlx``);
* ``strategy_op``: the stateless ``split_batched`` operator, one row per head;
* ``attention_layer``: a whole gated attention layer through ``TorqueQwenAttention``, a prompt chunk followed by
  decoded tokens.

Inputs follow the benchmark: fp16 (or float32) normal queries, keys and values, keys scaled by one log-normal factor
per channel, Gaussian Lloyd-Max codebooks.
"""

from __future__ import annotations

import math
import sys
from functools import lru_cache
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "torque-mlx_amd"))

import torque_hip as tq  # noqa: E402
from torque_hip import ops, qwen_torch  # noqa: E402

ROTATION_SEED = 0
SIZES = {"f16": 2, "f32": 4}


def listed():
    return [
        # the first tokens of a chat on a model without grouped queries: latency and launches
        dict(name="decode_short", kind="decode", bits=4, dim=128, layers=1, kv=8, group=1, seq=512, dtype="f16", rms=False),
        # the benchmark's headline shape: one layer, 32K tokens of context
        dict(name="decode_32k", kind="decode", bits=4, dim=128, layers=1, kv=8, group=4, seq=32768, dtype="f16", rms=False),
        # long context at the widest head
        dict(name="decode_128k_d256", kind="decode", bits=4, dim=256, layers=1, kv=2, group=4, seq=131072, dtype="f16", rms=False),
        # eight query heads to a KV head, a context that fills no whole block
        dict(name="decode_gqa8_ragged", kind="decode", bits=4, dim=128, layers=1, kv=4, group=8, seq=30001, dtype="f16", rms=False),
        # the smallest codes the cache is kept in without losing much, 3 bits: codes cross word boundaries
        dict(name="decode_3bit", kind="decode", bits=3, dim=128, layers=1, kv=8, group=4, seq=32768, dtype="f16", rms=False),
        # per-vector scales, for rows whose norms differ
        dict(name="decode_scaled", kind="decode", bits=4, dim=128, layers=1, kv=8, group=4, seq=16384, dtype="f32", rms=True),
        # one decode call for every layer of a model, as the qwen-decode benchmark makes it
        dict(name="decode_24_layers", kind="decode", bits=4, dim=256, layers=24, kv=4, group=4, seq=8192, dtype="f16", rms=False),
        # the same at a long context: the largest call
        dict(name="decode_24_layers_32k", kind="decode", bits=4, dim=128, layers=24, kv=8, group=4, seq=32768, dtype="f16", rms=False),
        # one layer's step of a decode loop: the new token packed and attended to, some way past a round length
        dict(name="append_decode_8k", kind="append_decode", bits=4, dim=256, layers=1, kv=4, group=4, seq=8259, dtype="f16"),
        # a prompt packed into one layer's cache, odd in every size
        dict(name="prefill_chunk", kind="prefill", bits=3, dim=64, layers=1, kv=4, seq=1999, dtype="f32", rms=False),
        # a long prompt packed for every layer of a model
        dict(name="prefill_24_layers", kind="prefill", bits=4, dim=128, layers=24, kv=8, seq=8192, dtype="f16", rms=False),
        # a whole attention layer: a prompt chunk, then a few decoded tokens
        dict(name="attention_layer", kind="attention_layer", bits=4, dim=256, hidden=2048, kv=4, group=4, seq=1024, tokens=8),
    ]


LARGEST_BYTES = 850e6  # packed K and V of the largest decode, dense K and V of the largest prefill


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "append_decode", "prefill", "prefill", "strategy_op", "attention_layer"])
    bits, dim, dtype = rng.choice([2, 3, 4, 4]), rng.choice([64, 128, 256]), rng.choice(["f16", "f16", "f32"])
    kv, group = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 4, 4, 5, 6, 7, 8])
    layers = rng.choice([1, 1, 1, _log_uniform(rng, 2, 24)])
    if kind == "attention_layer":
        return dict(kind=kind, bits=bits, dim=dim, hidden=rng.choice([1024, 1536, 2048]), kv=kv, group=rng.choice([1, 2, 4, 8]),
                    seq=_log_uniform(rng, 32, 1500), tokens=rng.randint(1, 12))
    seq = _log_uniform(rng, 100, 131072)
    rms = rng.random() < 0.15
    if kind == "prefill":
        seq = max(1, min(seq, int(LARGEST_BYTES / (2 * layers * kv * dim * SIZES[dtype]))))
        return dict(kind=kind, bits=bits, dim=dim, layers=layers, kv=kv, seq=seq, dtype=dtype, rms=rms)
    if kind == "strategy_op":  # one row of packed codes per head
        rows = kv * rng.choice([1, 2, 4])
        return dict(kind=kind, bits=bits, dim=dim, layers=1, kv=rows, group=1, seq=min(seq, 32768), dtype="f32", rms=False)
    if kind == "append_decode":
        return dict(kind=kind, bits=bits, dim=dim, layers=1, kv=kv, group=group, seq=min(seq, 65536), dtype=dtype)
    seq = max(1, min(seq, int(LARGEST_BYTES / (layers * kv * dim * bits / 4))))
    return dict(kind=kind, bits=bits, dim=dim, layers=layers, kv=kv, group=group, seq=seq, dtype=dtype, rms=rms)


# ------------------------------------------------------------------ inputs


@lru_cache(maxsize=None)
def _centroids(bits, seed):
    """Lloyd-Max centroids of seeded normal samples."""
    rng = np.random.default_rng(1000 + seed)
    x = np.sort(rng.normal(size=50_000)).astype(np.float64)
    c = np.quantile(x, (np.arange(1 << bits) + 0.5) / (1 << bits))
    for _ in range(60):
        at = np.searchsorted(x, (c[:-1] + c[1:]) / 2)
        c = np.array([part.mean() for part in np.split(x, at)])
    return c.astype(np.float32)


def _codebooks(bits):
    return tq.Codebook(bits, _centroids(bits, 0)), tq.Codebook(bits, _centroids(bits, 1))


def _boundaries(c):
    return ((c[:-1] + c[1:]) / np.float32(2)).astype(np.float32)


def _signs(dim):
    """The rotation's sign vectors, (left, right), as a seed defines them."""
    rng = np.random.default_rng(ROTATION_SEED)
    pm = np.array([-1.0, 1.0], dtype=np.float32)
    return rng.choice(pm, size=dim), rng.choice(pm, size=dim)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, shape, dtype="f32"):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float16 if dtype == "f16" else torch.float32)


def _kv_rows(g, case, seq):
    """Keys and values [L, Hkv, seq, D]; with per-vector scales, rows of differing norms."""
    shape = (case["layers"], case["kv"], seq, case["dim"])
    k, v = _randn(g, shape, case["dtype"]), _randn(g, shape, case["dtype"])
    k *= torch.exp(_randn(g, (shape[0], shape[1], 1, shape[3]))).to(k.dtype)
    if case.get("rms"):
        for x in (k, v):
            x *= torch.exp(0.5 * _randn(g, (shape[0], shape[1], seq, 1))).to(x.dtype)
    return k, v


def _cache(case, capacity, **kwargs):
    config = tq.TorqueConfig(bit_width=case["bits"], head_dim=case["dim"], num_layers=case.get("layers", 1), kv_heads=case["kv"],
                             rotation_seed=ROTATION_SEED, scale_mode="rms" if case.get("rms") else "none")
    kc, vc = _codebooks(case["bits"])
    return tq.TorqueKVCacheMLX(config=config, key_codebook=kc, value_codebook=vc, initial_capacity=capacity, **kwargs)


def _decode_inputs(case, seed):
    g = _generator(seed)
    q = _randn(g, (case["layers"], case["kv"] * case["group"], case["dim"]), case["dtype"])
    k, v = _kv_rows(g, case, case["seq"])
    return q, k, v


def _step_inputs(case, seed):
    q, k, v = _decode_inputs(case, seed)
    nk, nv = _kv_rows(_generator(seed + 7_000_000), case, 1)
    return q, k, v, nk, nv


class _Attention(torch.nn.Module):
    """A gated attention layer's weights, shaped as the adapter takes them."""

    def __init__(self, w, head_dim):
        super().__init__()
        self.head_dim = head_dim

        def linear(x):
            m = torch.nn.Linear(x.shape[1], x.shape[0], bias=False, device=x.device, dtype=x.dtype)
            m.weight = torch.nn.Parameter(x.clone(), requires_grad=False)
            return m

        self.q_proj, self.k_proj, self.v_proj, self.o_proj = (linear(w[n]) for n in ("q", "k", "v", "o"))
        self.q_norm, self.k_norm = _Norm(w["qn"]), _Norm(w["kn"])


class _Norm(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = torch.nn.Parameter(weight.clone(), requires_grad=False)

    def forward(self, x):
        y = x.float()
        return (y * torch.rsqrt(y.pow(2).mean(-1, keepdim=True) + 1e-6)).to(x.dtype) * self.weight


def _layer_inputs(case, seed):
    g = _generator(seed)
    hd, hidden, hq, total = case["dim"], case["hidden"], case["kv"] * case["group"], case["seq"] + case["tokens"]
    shapes = {"q": (2 * hq * hd, hidden), "k": (case["kv"] * hd, hidden), "v": (case["kv"] * hd, hidden), "o": (hidden, hq * hd)}
    w = {n: (_randn(g, s) / math.sqrt(s[1])).to(torch.bfloat16) for n, s in shapes.items()}
    w["qn"], w["kn"] = ((1 + 0.1 * _randn(g, (hd,))).to(torch.bfloat16) for _ in range(2))
    hidden_states = _randn(g, (1, total, hidden)).to(torch.bfloat16)
    rotary = hd // 4
    inv = 1.0 / 10000.0 ** (torch.arange(0, rotary, 2, device="cuda", dtype=torch.float32) / rotary)
    angle = torch.arange(total, device="cuda", dtype=torch.float32)[:, None] * inv[None]
    angle = torch.cat([angle, angle], dim=-1)[None]
    return w, hidden_states, angle.cos(), angle.sin()


# ------------------------------------------------------------------ the calls


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        q, k, v = _decode_inputs(case, seed)
        cache = _cache(case, case["seq"])
        cache.append_many_mlx(key=k, value=v)
        return {"kind": kind, "cache": cache, "q": q}
    if kind == "prefill":
        k, v = _kv_rows(_generator(seed), case, case["seq"])
        return {"kind": kind, "cache": _cache(case, case["seq"]), "k": k, "v": v}
    if kind in ("strategy_op", "append_decode"):
        kc, vc = (torch.from_numpy(c.centroids).cuda() for c in _codebooks(case["bits"]))
        kb, vb = (torch.from_numpy(_boundaries(c.centroids)).cuda() for c in _codebooks(case["bits"]))
        pack = dict(bit_width=case["bits"], head_dim=case["dim"])
        words = case["dim"] * case["bits"] // 32
    if kind == "strategy_op":
        q, k, v = _decode_inputs(case, seed)
        codes = ops.quantize_and_pack_rows_dual(k.reshape(-1, case["dim"]), v.reshape(-1, case["dim"]), kb, vb, **pack)
        k_codes, v_codes = (c.view(torch.int32).reshape(case["kv"], case["seq"], words) for c in codes)
        return {"kind": kind, "args": (q[0], k_codes, v_codes, kc, vc), "kwargs": pack}
    if kind == "append_decode":
        q, k, v, nk, nv = _step_inputs(case, seed)
        cache = _cache(case, case["seq"] + 64)  # a loop's slab has room for the tokens to come
        cache.append_many_mlx(key=k, value=v)
        left, right = (torch.from_numpy(s).cuda() for s in _signs(case["dim"]))
        k_codes, v_codes = (c.view(torch.int32) for c in cache.state)
        kwargs = dict(num_layers=1, query_heads=case["kv"] * case["group"], kv_heads=case["kv"], head_dim=case["dim"],
                      bit_width=case["bits"], key_codes=k_codes, value_codes=v_codes, capacity=case["seq"] + 64, seq_len=case["seq"],
                      key_centroids=kc, value_centroids=vc, key_boundaries=kb, value_boundaries=vb, signs_left=left,
                      signs_right=right, rotate_query=True, inverse_output=True)
        return {"kind": kind, "args": (q, nk[:, :, 0].contiguous(), nv[:, :, 0].contiguous()), "kwargs": kwargs}
    w, hidden_states, cos, sin = _layer_inputs(case, seed)
    layer = torch.nn.Module()
    layer.self_attn = _Attention(w, case["dim"])
    kc, vc = _codebooks(case["bits"])
    cache = qwen_torch.build_qwen_torque_cache(bit_width=case["bits"], head_dim=case["dim"], kv_heads=case["kv"],
                                               rotation_seed=ROTATION_SEED, key_codebook=kc, value_codebook=vc,
                                               initial_capacity=case["seq"] + case["tokens"])
    left, right = _signs(case["dim"])
    rotation = tq.RotationSpec(head_dim=case["dim"], signs_left=left, signs_right=right)
    adapter = qwen_torch.patch_vo_only_qwen_attention(layer, rotation=rotation, cache=cache)
    at = [slice(0, case["seq"])] + [slice(case["seq"] + t, case["seq"] + t + 1) for t in range(case["tokens"])]
    return {"kind": kind, "adapter": adapter, "steps": [(hidden_states[:, s], (cos[:, s], sin[:, s])) for s in at]}


def run(state):
    kind = state["kind"]
    if kind == "decode":
        return state["cache"].decode_mlx(query=state["q"], return_numpy=False)
    if kind == "append_decode":
        kw = state["kwargs"]
        return ops.packed_decode_append(*state["args"], **kw), kw["key_codes"], kw["value_codes"]
    if kind == "prefill":
        state["cache"].reset()
        state["cache"].append_many_mlx(key=state["k"], value=state["v"])
        return [c.view(torch.int32) for c in state["cache"].state]
    if kind == "strategy_op":
        return ops.decode_packed_attention_split_batched(*state["args"], **state["kwargs"])
    adapter = state["adapter"]
    with torch.no_grad():
        adapter.cache.torque_cache.reset()  # a new request
        return [adapter(h, pos)[0] for h, pos in state["steps"]]


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    d, kv = case["dim"], case["kv"]
    if case["kind"] == "prefill":
        rows = 2 * case["layers"] * kv * case["seq"]
        out = rows * (d * case["bits"] / 8 + (4 if case["rms"] else 0))
        return {"bytes": rows * d * SIZES[case["dtype"]] + out, "flops": rows * d * (math.log2(d) + 4 + case["bits"])}
    if case["kind"] == "attention_layer":
        hq, n, total = kv * case["group"], case["seq"], case["seq"] + case["tokens"]
        weights = case["hidden"] * d * (3 * hq + 2 * kv)
        flops = 2 * weights * total + 2 * hq * d * n * n + 4 * hq * d * n * case["tokens"]
        return {"bytes": 2 * weights * (1 + case["tokens"]) + 4 * case["hidden"] * total
                + case["tokens"] * n * kv * d * case["bits"] / 4, "flops": flops}
    hq, rows = case["layers"] * kv * case["group"], case["layers"] * kv * case["seq"]
    new = case["kind"] == "append_decode"
    codes = 2 * rows * (d * case["bits"] / 8 + (4 if case.get("rms") else 0))
    return {"bytes": codes + hq * d * (SIZES[case["dtype"]] + 4) + (2 * kv * d * (SIZES[case["dtype"]] + case["bits"] / 8) if new else 0),
            "flops": 4.0 * case["group"] * rows * d}


def tolerance(case):
    if case["kind"] == "prefill":
        return "exact"  # packed codes
    if case["kind"] == "attention_layer":
        # bf16 projections: 0.5 % for the prompt chunk, and 3 to 5 % against 64 bits for the decoded tokens, whose
        # codes move where a key's rounding takes it over a boundary
        return {"rel": 3e-2}
    # float32 sums in another order, or f16 hi/lo split products summed in float32: 2e-7 to 3.2e-6 against 64 bits
    return {"rel": 8e-6, "max": 1e-4}


# ------------------------------------------------------------------ the same in 64 bits


def _transform(x):
    """Walsh-Hadamard transform of the last axis, in x's own precision."""
    d, s = x.shape[-1], 1
    while s < d:
        y = x.reshape(*x.shape[:-1], d // (2 * s), 2, s)
        x = torch.stack((y[..., 0, :] + y[..., 1, :], y[..., 0, :] - y[..., 1, :]), dim=-2).reshape(x.shape)
        s *= 2
    return x


def _rotate(x, first, second):
    """second * H (first * x) / sqrt(D) in x's own precision; float32 here gives the cache's rotation bit for bit."""
    first, second = (torch.from_numpy(s).to(x.device, x.dtype) for s in (first, second))
    root = torch.full((1,), math.sqrt(x.shape[-1]), device=x.device, dtype=x.dtype)
    return _transform(x * first) / root * second


def _stored(rows, centroids, signs, rms, rotate=True):
    """What the packed cache holds of float32 rows, in 64 bits: the centroids of the rotated rows' codes."""
    if rotate:
        rows = _rotate(rows.float(), signs[1], signs[0])
    scale = 1.0
    if rms:
        scale = rows.double().pow(2).mean(-1, keepdim=True).sqrt().float()
        rows = rows / scale
        scale = scale.double()
    c = torch.from_numpy(centroids).to(rows.device)
    codes = torch.bucketize(rows.contiguous(), torch.from_numpy(_boundaries(centroids)).to(rows.device))
    return c.double()[codes] * scale


def _attend(q, k, v):
    """Attention of float64 queries [G, D] over [S, D]."""
    s = torch.matmul(k, q.t().contiguous()) / math.sqrt(q.shape[-1])
    return torch.matmul(torch.softmax(s, dim=0).t().contiguous(), v)


def exact(case, seed):
    kind = case["kind"]
    if kind == "prefill":
        return None  # packed codes: whole numbers
    ck, cv = _centroids(case["bits"], 0), _centroids(case["bits"], 1)
    signs = _signs(case["dim"])
    if kind == "attention_layer":
        return _exact_layer(case, seed, ck, cv, signs)
    if kind == "append_decode":
        q, k, v, nk, nv = _step_inputs(case, seed)
        k, v = torch.cat([k, nk], dim=2), torch.cat([v, nv], dim=2)
    else:
        q, k, v = _decode_inputs(case, seed)
    rotate, group = kind != "strategy_op", case["group"]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for layer in range(case["layers"]):
        for h in range(case["kv"]):
            mine = slice(h * group, (h + 1) * group)
            x = q[layer, mine].double()
            x = _rotate(x, signs[1], signs[0]) if rotate else x
            y = _attend(x, _stored(k[layer, h], ck, signs, case.get("rms"), rotate), _stored(v[layer, h], cv, signs, case.get("rms"), rotate))
            out[layer, mine] = _rotate(y, signs[0], signs[1]) if rotate else y
    if kind == "strategy_op":
        return out[0]
    return (out, None, None) if kind == "append_decode" else out


def _exact_layer(case, seed, ck, cv, signs):
    w, x, cos, sin = _layer_inputs(case, seed)
    w, x, cos, sin = {n: t.double() for n, t in w.items()}, x[0].double(), cos[0].double(), sin[0].double()
    hd, kv, group, n, total = case["dim"], case["kv"], case["group"], case["seq"], case["seq"] + case["tokens"]
    r = cos.shape[-1]

    def norm(t, weight):
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6) * weight

    def rotary(t):  # [T, H, D]
        a, rest = t[..., :r], t[..., r:]
        half = torch.cat((-a[..., r // 2:], a[..., : r // 2]), dim=-1)
        return torch.cat((a * cos[:, None] + half * sin[:, None], rest), dim=-1)

    q, gate = torch.chunk(torch.matmul(x, w["q"].t()).reshape(total, kv * group, 2 * hd), 2, dim=-1)
    q = rotary(norm(q, w["qn"]))
    k = rotary(norm(torch.matmul(x, w["k"].t()).reshape(total, kv, hd), w["kn"]))
    v = torch.matmul(x, w["v"].t()).reshape(total, kv, hd)
    attended = torch.empty(total, kv * group, hd, dtype=torch.float64, device=x.device)
    hidden = torch.ones(n, n, dtype=torch.bool, device=x.device).triu(1)
    for h in range(kv):
        kh, vh = k[:, h].contiguous(), v[:, h].contiguous()
        ks = _stored(kh.float(), ck, signs, False)
        vs = _stored(_rotate(vh, signs[1], signs[0]).float(), cv, signs, False, rotate=False)
        for j in range(h * group, (h + 1) * group):
            s = torch.matmul(q[:n, j].contiguous(), kh[:n].t().contiguous()) / math.sqrt(hd)
            attended[:n, j] = torch.matmul(torch.softmax(s.masked_fill(hidden, -math.inf), dim=-1), vh[:n])
        for t in range(n, total):
            y = _attend(_rotate(q[t, h * group : (h + 1) * group].contiguous(), signs[1], signs[0]), ks[: t + 1], vs[: t + 1])
            attended[t, h * group : (h + 1) * group] = _rotate(y, signs[0], signs[1])
    out = torch.matmul((attended * torch.sigmoid(gate)).reshape(total, -1), w["o"].t())[None]
    return [out[:, :n]] + [out[:, t : t + 1] for t in range(n, total)]
