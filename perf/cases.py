"""Workloads this framework is used for, as calls through its public entry
points: MoE blocks at every batch size a server forms, decode steps, prompt
prefill and the plugin product.

A case is a dict of plain values.  ``kind`` is the path it takes:

* ``block``    ``HbmExpertStore.layer_ffn_batch`` on LAYERS layers in turn, as
               a host that keeps its own attention runs them (one call per
               layer, so that each call meets weights that no cache holds);
* ``step``     ``HipDecoder.decode_layers_batch``: one decode step of a batch
               of sequences over their caches, through a few layers of the
               model, optionally with the lm_head;
* ``prefill``  ``HipDecoder.prefill_layers``: a whole prompt, its cache rows
               and the last position's logits;
* ``gemm``     ``HipBackend.q4_gemm``: one Q4 matrix against T tokens, the
               plugin product.

Models are those of the repository's benchmark: Qwen3-30B-A3B- and
OLMoE-1B-7B-shaped blocks and a Qwen3-8B-shaped dense decoder.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from joule_amd.backend import HipBackend
from joule_amd.decoder import DecoderShape, DecoderWeights, HipDecoder, KVCacheSet, rope_tables
from joule_amd.dense import DenseFfnStore, dense_ffn_shape
from joule_amd.moe import OLMOE, QWEN3, HbmExpertStore
from joule_amd.q4_store import record_sizes
from joule_amd.synth import bf16_round, decoder_weights, fill_kv, torch_store, zipf_bias

LAYERS = 4                      # layers of a block case's store, called in turn
MODEL_LAYERS = 2                # layers of a step or prefill case
V = 151936                      # Qwen3's vocabulary
MOE = {"qwen3": QWEN3, "olmoe": OLMOE}
DENSE_D, DENSE_M, DENSE_H, DENSE_KH = 4096, 12288, 32, 8


def listed() -> list[dict]:
    return [
        # one user's chat: a single token per step, where launches and
        # round trips count
        {"name": "block_qwen3_b1", "kind": "block", "model": "qwen3", "group": 64, "tokens": 1, "zipf": False,
         "router": "bf16"},
        # the headline decode batch
        {"name": "block_qwen3_b8", "kind": "block", "model": "qwen3", "group": 64, "tokens": 8, "zipf": False,
         "router": "bf16"},
        # a few users of the other model family, with its float32 router
        # table and the smaller Q4 group
        {"name": "block_olmoe_b3_g32", "kind": "block", "model": "olmoe", "group": 32, "tokens": 3, "zipf": False,
         "router": "f32"},
        # a busy server's decode batch: every expert active, few tokens each
        {"name": "block_qwen3_b52", "kind": "block", "model": "qwen3", "group": 64, "tokens": 52, "zipf": False,
         "router": "bf16"},
        # a short prompt's chunk
        {"name": "block_olmoe_t203", "kind": "block", "model": "olmoe", "group": 64, "tokens": 203, "zipf": False,
         "router": "bf16"},
        # a full prefill chunk with the skewed routing of real text
        {"name": "block_qwen3_t509_zipf", "kind": "block", "model": "qwen3", "group": 64, "tokens": 509, "zipf": True,
         "router": "bf16"},
        # decode of 8 sequences in the middle of long answers
        {"name": "step_qwen3_b8", "kind": "step", "model": "qwen3", "tokens": 8, "context": 2048, "kv": "bf16",
         "logits": False},
        # a dense model, three sequences, the whole step with its logits
        {"name": "step_dense_b3", "kind": "step", "model": "dense", "tokens": 3, "context": 1000, "kv": "bf16",
         "logits": True},
        # the benchmark's prompt
        {"name": "prefill_qwen3_t512", "kind": "prefill", "model": "qwen3", "tokens": 512, "kv": "bf16"},
        # a long, ragged prompt: later chunks read the rows of earlier ones
        {"name": "prefill_qwen3_t1531", "kind": "prefill", "model": "qwen3", "tokens": 1531, "kv": "bf16"},
        # a short prompt of the dense model
        {"name": "prefill_dense_t301", "kind": "prefill", "model": "dense", "tokens": 301, "kv": "bf16"},
        # a host that brings its own driver and calls the plugin product
        {"name": "gemm_t37", "kind": "gemm", "rows": 768, "cols": 2048, "group": 64, "tokens": 37},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["block", "block", "block", "step", "step", "prefill", "prefill", "gemm"])
    if kind == "block":
        return {"kind": "block", "model": rng.choice(["qwen3", "qwen3", "olmoe"]), "group": rng.choice([64, 64, 32]),
                "tokens": _log_int(rng, 1, 512), "zipf": rng.random() < 0.4, "router": rng.choice(["bf16", "f32"])}
    if kind == "step":
        return {"kind": "step", "model": rng.choice(["qwen3", "qwen3", "dense"]), "tokens": _log_int(rng, 1, 12),
                "context": _log_int(rng, 24, 3000), "kv": rng.choice(["bf16", "bf16", "f32"]),
                "logits": rng.random() < 0.3}
    if kind == "prefill":
        model, kv = rng.choice([("qwen3", "bf16"), ("qwen3", "bf16"), ("qwen3", "f32"), ("dense", "bf16")])
        top = {("qwen3", "bf16"): 1500, ("qwen3", "f32"): 700, ("dense", "bf16"): 400}[model, kv]
        return {"kind": "prefill", "model": model, "tokens": _log_int(rng, 20, top), "kv": kv}
    rows, cols = rng.choice([(768, 2048), (2048, 768), (1024, 2048), (2048, 1024)])
    return {"kind": "gemm", "rows": rows, "cols": cols, "group": rng.choice([64, 64, 32]),
            "tokens": _log_int(rng, 1, 512)}


# ------------------------------------------------------------------- inputs


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(gen, *shape) -> torch.Tensor:
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _router(gen, shape, layers: int, zipf: bool, f32: bool, seed: int) -> torch.Tensor:
    """Router table [layers, E, d]: N(0, 0.02), as bf16 values unless f32;
    with zipf, column 0 carries the bias that skews the experts' shares."""
    w = _randn(gen, layers, shape.E, shape.d) * 0.02
    if not f32:
        w = w.to(torch.bfloat16).float()
    if zipf:
        for l in range(layers):
            bias = zipf_bias(shape.E, alpha=0.28, seed=4000 + seed + l)
            w[l, :, 0] = torch.from_numpy(bf16_round(bias / np.float32(4.0))).cuda()
    return w.contiguous()


def _moe_store(case, seed: int, layers: int):
    shape, group = MOE[case["model"]], case.get("group", 64)
    blob, offsets = torch_store(shape, layers, group, seed=100_000 + 64 * seed)
    store = HbmExpertStore(shape, layers, blob, offsets, group)
    gate = _router(_gen(seed * 7 + 1), shape, layers, case.get("zipf", False), case.get("router") == "f32", seed)
    store.set_router(gate)
    return store, gate


def _shape(case, max_t: int) -> DecoderShape:
    if case["model"] == "dense":
        return DecoderShape(n_layers=MODEL_LAYERS, moe=dense_ffn_shape(DENSE_D, DENSE_M), n_heads=DENSE_H,
                            n_kv=DENSE_KH, maxT=max_t, V=V, name="dense")
    return DecoderShape(n_layers=MODEL_LAYERS, moe=QWEN3, n_heads=32, n_kv=4, maxT=max_t, V=V, name="qwen3")


def _decoder(case, seed: int, max_t: int, lm: bool, embed: bool):
    shape = _shape(case, max_t)
    if case["model"] == "dense":
        store = DenseFfnStore(DENSE_D, DENSE_M, MODEL_LAYERS)
        gate = None
    else:
        store, gate = _moe_store(case, seed, MODEL_LAYERS)
    t = decoder_weights(shape, seed=seed * 7 + 2, norm_jitter=0.1)
    gen = _gen(seed * 7 + 3)
    if embed:
        t["embed"] = _randn(gen, V, shape.d).to(torch.bfloat16)
    dec = HipDecoder(store, DecoderWeights(shape, **t))
    lm_w = None
    if lm:
        lm_w = (_randn(gen, V, shape.d) * 0.02).to(torch.bfloat16)
        dec.set_lm_head(lm_w)
    return dec, t, gate, lm_w


def _kv_type(case):
    return torch.float32 if case["kv"] == "f32" else torch.bfloat16


def _positions(case, seed: int) -> list[int]:
    """The sequences' lengths differ: each within the last fifth below the
    case's context."""
    rng = np.random.default_rng(seed + 17)
    c = case["context"]
    return [c] + [int(c - rng.integers(0, max(1, c // 5))) for _ in range(case["tokens"] - 1)]


def _max_t(case) -> int:
    n = case["context"] + 1 if case["kind"] == "step" else case["tokens"]
    return (n + 127) // 128 * 128


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "block":
        shape = MOE[case["model"]]
        store, gate = _moe_store(case, seed, LAYERS)
        store.reserve(case["tokens"])
        x = _randn(_gen(seed * 7 + 4), case["tokens"], shape.d)
        if case["zipf"]:
            x[:, 0] = 4.0
        s.update(store=store, gate=gate, x=x.contiguous())
    elif kind == "step":
        dec, t, gate, lm = _decoder(case, seed, _max_t(case), case["logits"], False)
        kv = KVCacheSet(dec.shape, case["tokens"], dtype=_kv_type(case))
        fill_kv(kv.data, seed=50_000 + 64 * seed)
        x = _randn(_gen(seed * 7 + 4), case["tokens"], dec.shape.d)
        pos = _positions(case, seed)
        s.update(dec=dec, t=t, gate=gate, lm=lm, kv=kv, x=x, pos=pos, hidden=torch.empty_like(x),
                 logits=torch.empty((case["tokens"], V), device="cuda") if case["logits"] else None,
                 rows=[kv.data[b, :, :, p] for b, p in enumerate(pos)])
    elif kind == "prefill":
        dec, t, gate, lm = _decoder(case, seed, _max_t(case), True, True)
        kv = KVCacheSet(dec.shape, 1, dtype=_kv_type(case))
        tok = torch.randint(0, V, (case["tokens"],), generator=_gen(seed * 7 + 4), device="cuda", dtype=torch.int32)
        s.update(dec=dec, t=t, gate=gate, lm=lm, kv=kv, tok=tok, logits=torch.empty(V, device="cuda"),
                 rows=kv.data[0, :, :, :case["tokens"]])
    else:
        m, d, g = case["rows"], case["cols"], case["group"]
        gen = _gen(seed * 7 + 4)
        packed = torch.randint(0, 256, (m * d // 2,), generator=gen, device="cuda", dtype=torch.uint8)
        scales = (torch.rand(m * d // g, generator=gen, device="cuda") * 0.01 + 0.002).to(torch.float16)
        s.update(backend=HipBackend(), packed=packed, scales=scales.view(torch.int16), m=m, d=d, group=g,
                 X=_randn(gen, case["tokens"], d), out=torch.empty((case["tokens"], m), device="cuda"))
    return s


def run(state: dict):
    kind = state["kind"]
    if kind == "block":
        return [state["store"].layer_ffn_batch(l, state["x"]) for l in range(LAYERS)]
    if kind == "step":
        state["dec"].decode_layers_batch(state["x"], state["pos"], state["kv"], hidden=state["hidden"],
                                         logits=state["logits"])
        out = [state["hidden"], *state["rows"]]
        return out if state["logits"] is None else out + [state["logits"]]
    if kind == "prefill":
        state["dec"].prefill_layers(state["tok"], state["kv"], 0, state["logits"])
        return [state["logits"], state["rows"]]
    state["backend"].q4_gemm(state["out"], state["X"], state["packed"], state["scales"], state["m"], state["d"],
                             state["group"])
    return state["out"]


# --------------------------------------------------------------------- work


def _expert_bytes(shape, group: int) -> int:
    return sum(sum(record_sizes(r, c, group)) for r, c in ((shape.m, shape.d), (shape.m, shape.d), (shape.d, shape.m)))


def _block_work(shape, group: int, B: int, router_bytes: int) -> tuple[float, float]:
    """Bytes and flops of one MoE block: the experts B tokens reach when each
    takes top-k of E alike, the router table, x in and out."""
    active = shape.E * (1.0 - (1.0 - shape.topk / shape.E) ** B)
    by = active * _expert_bytes(shape, group) + shape.E * shape.d * router_bytes + 2 * B * shape.d * 4
    fl = 2.0 * B * shape.d * shape.E + 6.0 * B * shape.topk * shape.d * shape.m
    return by, fl


def _layer_work(case, B: int, kv_read: int, pairs: int) -> tuple[float, float]:
    """One decoder layer of B tokens that reads kv_read cache rows and forms
    `pairs` (query, position) products."""
    sh = _shape(case, 128)
    d, hd, H, KH = sh.d, sh.hd, sh.n_heads, sh.n_kv
    proj = (H + 2 * KH) * hd * d + d * H * hd
    row = 2 * KH * hd * (4 if case["kv"] == "f32" else 2)
    by = 2.0 * proj + kv_read * row + B * row
    fl = 2.0 * B * proj + 4.0 * pairs * H * hd
    if case["model"] == "dense":
        return by + 2.0 * 3 * DENSE_D * DENSE_M, fl + 6.0 * B * DENSE_D * DENSE_M
    mb, mf = _block_work(QWEN3, 64, B, 2)
    return by + mb, fl + mf


def work(case: dict) -> dict:
    kind, B = case["kind"], case["tokens"]
    if kind == "block":
        by, fl = _block_work(MOE[case["model"]], case["group"], B, 4 if case["router"] == "f32" else 2)
        return {"bytes": LAYERS * by, "flops": LAYERS * fl}
    if kind == "gemm":
        sb, pb = record_sizes(case["rows"], case["cols"], case["group"])
        return {"bytes": sb + pb + 4 * B * (case["rows"] + case["cols"]), "flops": 2.0 * B * case["rows"] * case["cols"]}
    d = _shape(case, 128).d
    if kind == "step":
        n = int(B * (case["context"] + 1) * 0.9)
        by, fl = _layer_work(case, B, n, n)
        lm = B if case["logits"] else 0
    else:
        # the prompt's own rows are read once, after they are written
        by, fl = _layer_work(case, B, B, B * (B + 1) // 2)
        lm = 1
    by, fl = by * MODEL_LAYERS + 8.0 * B * d, fl * MODEL_LAYERS
    if lm:
        by += 2.0 * V * d + 4.0 * lm * V
        fl += 2.0 * lm * V * d
    return {"bytes": by, "flops": fl}


def tolerance(case: dict) -> dict:
    # Measured against float64 (exact below) and stated at about four times
    # that: the expert product rounds activations to 15 or 16 bits of their
    # group's largest value, bf16 cache rows differ by their last bit.
    if case["kind"] in ("block", "gemm"):
        return {"rel": 2e-4}
    return {"rel": 1e-2}


# ----------------------------------------------------------- float64 results


def _dequant(packed, scales, rows: int, cols: int, group: int) -> torch.Tensor:
    p = packed.view(-1, 1).to(torch.int16)
    q = torch.cat([p & 15, p >> 4], dim=1).view(rows, cols // group, group) - 8
    return (q.double() * scales.view(torch.float16).double().view(rows, cols // group, 1)).view(rows, cols)


def _moe64(store, gate, l: int, x: torch.Tensor) -> torch.Tensor:
    """The MoE block of layer l on float64 tokens x."""
    sh, g = store.shape, store.group
    p = torch.softmax(x @ gate[l].double().T, dim=1)
    w, idx = torch.topk(p, sh.topk, dim=1)
    if sh.renorm:
        w = w / w.sum(dim=1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(sh.E):
        tok, slot = torch.where(idx == e)
        if tok.numel() == 0:
            continue
        (gs, gp, _), (us, up, _), (ds, dp, _) = store.ensure(l, e)
        xe = x[tok]
        act = torch.nn.functional.silu(xe @ _dequant(gp, gs, sh.m, sh.d, g).T) * (
            xe @ _dequant(up, us, sh.m, sh.d, g).T)
        out.index_add_(0, tok, w[tok, slot].unsqueeze(1) * (act @ _dequant(dp, ds, sh.d, sh.m, g).T))
    return out


def _rms64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(dim=-1, keepdim=True) + eps) * w.double()


def _rope64(x, cos, sin):
    h = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., h:], x[..., :h]], dim=-1) * sin


@functools.lru_cache(maxsize=4)
def _rope(max_t: int, hd: int, theta: float):
    return tuple(torch.from_numpy(a).cuda().double() for a in rope_tables(max_t, hd, theta))


def _model64(s, x, pos, cache_of):
    """Every layer on float64 tokens x at positions pos: (final-normed
    hidden, appended k and v rows [layer][2][token, KH, hd]).  cache_of(l, b)
    gives token b's float64 (k, v) with the call's own rows in place."""
    dec, t = s["dec"], s["t"]
    sh = dec.shape
    H, KH, hd = sh.n_heads, sh.n_kv, sh.hd
    cos, sin = (c[torch.as_tensor(pos, device="cuda")].unsqueeze(1) for c in _rope(sh.maxT, hd, sh.theta))
    B, new = x.shape[0], []
    h = x
    for l in range(sh.n_layers):
        n = _rms64(h, t["norm1"][l], sh.eps)
        q = (n @ t["wq"][l].double().T).view(B, H, hd)
        k = (n @ t["wk"][l].double().T).view(B, KH, hd)
        v = (n @ t["wv"][l].double().T).view(B, KH, hd)
        q = _rope64(_rms64(q, t["qn"][l], sh.eps), cos, sin)
        k = _rope64(_rms64(k, t["kn"][l], sh.eps), cos, sin)
        # attention reads the rows as the cache holds them
        new.append((k, v))
        kc, vc = (a.to(s["kv"].data.dtype).double() for a in (k, v))
        att = cache_of(l, q.view(B, KH, H // KH, hd) * hd ** -0.5, kc, vc)
        h = h + att.reshape(B, H * hd) @ t["wo"][l].double().T
        n = _rms64(h, t["norm2"][l], sh.eps)
        if sh.moe.E == 0:
            a = torch.nn.functional.silu(n @ t["w1"][l].double().T) * (n @ t["w2"][l].double().T)
            h = h + a @ t["w3"][l].double().T
        else:
            h = h + _moe64(dec.store, s["gate"], l, n)
    return _rms64(h, t["final_norm"], sh.eps), new


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "block":
        return [_moe64(s["store"], s["gate"], l, s["x"].double()) for l in range(LAYERS)]
    if kind == "gemm":
        return s["X"].double() @ _dequant(s["packed"], s["scales"], s["m"], s["d"], s["group"]).T
    if kind == "step":
        pos, data = s["pos"], s["kv"].data

        def attend(l, q, kc, vc):
            out = torch.empty_like(q)
            for b, p in enumerate(pos):
                K = torch.cat([data[b, l, 0, :p].double(), kc[b:b + 1]])
                W = torch.cat([data[b, l, 1, :p].double(), vc[b:b + 1]])
                pr = torch.softmax(torch.einsum("kqd,tkd->kqt", q[b], K), dim=-1)
                out[b] = torch.einsum("kqt,tkd->kqd", pr, W)
            return out

        hid, new = _model64(s, s["x"].double(), pos, attend)
        rows = [torch.stack([torch.stack([k[b], v[b]]) for k, v in new]) for b in range(len(pos))]
        out = [hid, *rows]
        return out if s["lm"] is None else out + [hid @ s["lm"].double().T]
    T = case["tokens"]
    mask = torch.full((T, T), float("-inf"), device="cuda", dtype=torch.float64).triu(1)

    def attend(l, q, kc, vc):
        out = torch.empty_like(q)
        for kh in range(q.shape[1]):
            for i in range(q.shape[2]):
                out[:, kh, i] = torch.softmax(q[:, kh, i] @ kc[:, kh].T.contiguous() + mask, dim=-1) @ vc[:, kh]
        return out

    x = s["t"]["embed"][s["tok"].long()].double()
    hid, new = _model64(s, x, list(range(T)), attend)
    rows = torch.stack([torch.stack([k, v]) for k, v in new])
    return [hid[-1] @ s["lm"].double().T, rows]
