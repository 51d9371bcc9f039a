"""The work that performance is measured on: what a program that decodes, verifies, prefills and
scores with this package's attention has it do, through the public entry points.

Five kinds of case, over the head layouts that the tests and the benchmark use:
  decode   one step of T tokens per row onto a filled cache (ops.attn_decode_append): single-token
           decode, the speculative verify step (T = 2 .. 16), rows of one length or of their own,
           sliding windows;
  prefill  a prompt, or one chunk of a long one at an offset: the cache write (ops.kv_append) and
           the causal attention over it (ops.attn_prefill), with windows and packed documents;
  layer    sleuth_amd.attention.Attention called eagerly with a cache, its projections included;
  graph    one replayed decode or verify step of a whole small model (GraphDecoder), logits out.
"""

import functools
import math

import torch
import torch.nn.functional as F

from sleuth_amd import ops
from sleuth_amd.attention import Attention
from sleuth_amd.config import ModelConfig
from sleuth_amd.generate import GraphDecoder
from sleuth_amd.kv_cache import KVCache
from sleuth_amd.model import Transformer
from sleuth_amd.rope import rope_tables

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
EPS = 1e-6
THETA = 1e6


def listed():
    return [
        # the smallest call: one token of generate() in an eager layer, batch 1, a short context
        dict(name="layer_decode_b1", kind="layer", dtype="bf16", B=1, T=1, H=16, K=8, D=128, d_model=1024,
             offset=211, cap=4096),
        # one token of a whole small model through the recorded graph (launches back to back)
        dict(name="graph_step", kind="graph", dtype="bf16", T=1, H=16, K=8, D=128, d_model=1024, layers=4,
             hidden=3072, vocab=8192, offset=701, cap=4096),
        # a serving batch of equal lengths, small heads (the 12 q / 4 KV, head dim 64 layout)
        dict(name="decode_batch", kind="decode", dtype="bf16", B=16, T=1, H=12, K=4, D=64, keys=2049, cap=2176,
             ragged=False, window=0),
        # a large serving batch of ragged lengths: the largest decode step
        dict(name="decode_ragged", kind="decode", dtype="bf16", B=64, T=1, H=16, K=8, D=128, keys=32768, cap=32768,
             ragged=True, window=0),
        # speculative verify of 3 guesses on a sliding-window layer, one KV head of 256
        dict(name="verify_window", kind="decode", dtype="bf16", B=8, T=4, H=8, K=1, D=256, keys=8196, cap=8448,
             ragged=False, window=1024),
        # speculative verify of 4 guesses, two query heads per KV head, fp16
        dict(name="verify_gqa", kind="decode", dtype="fp16", B=8, T=5, H=16, K=8, D=128, keys=6005, cap=8192,
             ragged=False, window=0),
        # a short prompt of odd length in an eager layer
        dict(name="layer_prompt", kind="layer", dtype="bf16", B=1, T=333, H=16, K=8, D=128, d_model=1024,
             offset=0, cap=4096),
        # one 512-token chunk of a long prompt, its prefix already cached
        dict(name="prefill_chunk", kind="prefill", dtype="bf16", B=1, T=512, H=16, K=8, D=128, offset=15360,
             cap=32768, window=0, docs=0),
        # a batch of whole prompts: the largest prefill
        dict(name="prefill_batch", kind="prefill", dtype="bf16", B=4, T=4096, H=16, K=8, D=128, offset=0,
             cap=4096, window=0, docs=0),
        # a whole prompt on a layer with one KV head of 512
        dict(name="prefill_wide", kind="prefill", dtype="bf16", B=1, T=3001, H=16, K=1, D=512, offset=0,
             cap=4096, window=0, docs=0),
        # scoring packed windows: documents of a few hundred tokens, head dim 256, fp16
        dict(name="prefill_docs", kind="prefill", dtype="fp16", B=4, T=2048, H=8, K=4, D=256, offset=0,
             cap=2048, window=0, docs=500),
        # full precision: the small 8 q / 4 KV head layout in fp32
        dict(name="layer_fp32", kind="layer", dtype="fp32", B=2, T=1025, H=8, K=4, D=32, d_model=256,
             offset=0, cap=2048),
    ]


# ---------------------------------------------------------------- more cases of the same ranges
_HEADS = [(16, 8, 128), (16, 8, 128), (12, 4, 64), (32, 8, 128), (8, 1, 256), (8, 4, 256), (16, 16, 64),
          (28, 4, 128), (16, 1, 512)]
_MAX_BYTES, _MAX_FLOPS, _MAX_FLOPS_FP32 = 3.8e9, 2.6e11, 4e9


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "layer", "layer", "graph"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    H, K, D = rng.choice(_HEADS)
    if kind == "decode":
        T = rng.choice([1, 1, 1, 2, 3, 4, 5, 8, 9, 16])
        keys = max(T + 1, _log(rng, 150, 32768))
        return dict(kind=kind, dtype=dtype, B=_log(rng, 1, 64), T=T, H=H, K=K, D=D, keys=keys,
                    cap=_log(rng, keys, min(32768, 4 * keys)), ragged=rng.random() < 0.4,
                    window=rng.choice([0, 0, 0, 512, 1024]))
    if kind == "prefill":
        T = _log(rng, 17, 4096)
        offset = rng.choice([0, 0, _log(rng, 64, 24000)])
        docs = _log(rng, 100, 1500) if offset == 0 and rng.random() < 0.3 else 0
        return dict(kind=kind, dtype=dtype, B=_log(rng, 1, 8) if offset == 0 else 1, T=T, H=H, K=K, D=D,
                    offset=offset, cap=_log(rng, offset + T, 2 * (offset + T)),
                    window=0 if docs else rng.choice([0, 0, 0, 512, 1024]), docs=docs)
    if kind == "layer":
        if rng.random() < 0.4:   # full precision
            H, K, D = rng.choice([(8, 4, 32), (8, 4, 64), (16, 8, 128)])
            dtype = "fp32"
        T = rng.choice([1, 1, 5, _log(rng, 17, 2048), _log(rng, 17, 2048)])
        offset = rng.choice([0, _log(rng, 16, 4096)]) if T > 1 else _log(rng, 16, 4096)
        return dict(kind=kind, dtype=dtype, B=_log(rng, 1, 8), T=T, H=H, K=K, D=D,
                    d_model=256 if D == 32 else 1024, offset=offset, cap=max(4096, offset + T + 64))
    H, K, D = rng.choice([(16, 8, 128), (12, 4, 64), (8, 1, 256)])
    T = rng.choice([1, 1, 5])
    return dict(kind=kind, dtype=dtype, T=T, H=H, K=K, D=D, d_model=1024, layers=rng.choice([2, 4]), hidden=3072,
                vocab=8192, offset=_log(rng, 30, 4000), cap=4096 + 64)


def draw(rng):
    while True:
        c = _draw_once(rng)
        w = work(c)
        if w["bytes"] <= _MAX_BYTES and w["flops"] <= (_MAX_FLOPS_FP32 if c["dtype"] == "fp32" else _MAX_FLOPS):
            return c


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, shape, dtype, scale=1.0):
    """Normal values of the dtype, made in slices of the first axis (no fp32 copy of a whole cache)."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    for part in out if out.numel() > 1 << 26 else [out]:
        part.copy_(torch.randn(part.shape, generator=g, device="cuda") * scale)
    return out


def _gain(g, D):
    """q/k norm gains as trained ones are: near 1.3, so that scores have a standard deviation above 1."""
    return 1.3 + 0.15 * torch.randn(D, generator=g, device="cuda")


def _lengths(case, seed):
    """Tokens stored per row once the step's T are in: one length, or log-uniform-ish ragged ones."""
    if not case["ragged"]:
        return [case["keys"]] * case["B"]
    g = torch.Generator().manual_seed(1234)   # one set of lengths per case: seeds change the data, not the work
    lo = min(case["keys"], max(case["T"] + 1, case["keys"] // 32))
    return torch.randint(lo, case["keys"] + 1, (case["B"],), generator=g).tolist()


def _doc_starts(case):
    """[B][T] first position of each token's document: runs of about `docs` tokens."""
    g = torch.Generator().manual_seed(4321)
    rows = []
    for _ in range(case["B"]):
        starts, at = [], 0
        while at < case["T"]:
            n = min(int(torch.randint(max(1, case["docs"] // 3), 2 * case["docs"], (1,), generator=g)), case["T"] - at)
            starts += [at] * n
            at += n
        rows.append(starts)
    return rows


def _split(y, case):
    """q, k, v [B, heads, T, D] as views of the fused projection's rows [B, T, (H + 2K) D]."""
    B, T, H, K, D = (case[n] for n in "BTHKD")
    q, k, v = y.split([H * D, K * D, K * D], -1)
    return (q.view(B, T, H, D).transpose(1, 2), k.view(B, T, K, D).transpose(1, 2),
            v.view(B, T, K, D).transpose(1, 2))


def _model_config(case):
    return ModelConfig(vocab_size=case.get("vocab", 16), d_model=case["d_model"], n_layers=case.get("layers", 1),
                       n_heads=case["H"], head_size=case["D"], n_kv_heads=case["K"], norm_eps=EPS,
                       rope_theta=THETA, max_seq_len=case["cap"], qk_norm=True, ffn_hidden=case.get("hidden", 0))


@torch.no_grad()
def prepare(case, seed):
    g, dt, kind = _gen(seed), DTYPES[case["dtype"]], case["kind"]
    s = {"case": case}
    if kind in ("decode", "prefill"):
        B, T, H, K, D, cap = (case[n] for n in ("B", "T", "H", "K", "D", "cap"))
        s["kc"], s["vc"] = _randn(g, (B, K, cap, D), dt, 1.3), _randn(g, (B, K, cap, D), dt)
        s["q"], s["k"], s["v"] = _split(_randn(g, (B, T, (H + 2 * K) * D), dt), case)
        s["qw"], s["kw"] = _gain(g, D), _gain(g, D)
        cos, sin = (t.cuda() for t in rope_tables(D, cap, THETA))
        if kind == "prefill":
            o = case["offset"]
            s["cos"], s["sin"] = cos[o:o + T], sin[o:o + T]
            s["docs"] = torch.tensor(_doc_starts(case), dtype=torch.int32, device="cuda") if case["docs"] else None
        else:
            base = [n - T for n in _lengths(case, seed)]
            if case["ragged"]:
                s["row_pos"] = torch.tensor(base, dtype=torch.int32, device="cuda")
                at = s["row_pos"].long()[:, None] + torch.arange(T, device="cuda")
                s["cos"], s["sin"] = cos[at], sin[at]
            else:
                s["cos"], s["sin"] = cos[base[0]:base[0] + T], sin[base[0]:base[0] + T]
            s["base"] = base
        return s
    devs = [torch.cuda.current_device()]
    with torch.random.fork_rng(devices=devs):
        torch.manual_seed(seed)
        with torch.device("cuda"):
            net = Transformer(_model_config(case)) if kind == "graph" else Attention(_model_config(case), 0)
    for name, p in net.named_parameters():
        if name.endswith(("q_norm.weight", "k_norm.weight")):
            p.copy_(_gain(g, case["D"]))
    net = net.to(dt).eval()
    s["net"] = net
    T, o = case["T"], case["offset"]
    if kind == "layer":
        s["x"] = _randn(g, (case["B"], T, case["d_model"]), dt)
        s["cache"] = KVCache([(case["K"], case["D"])], case["B"], case["cap"], "cuda", dt)
        s["cache"].k[0].copy_(_randn(g, s["cache"].k[0].shape, dt, 1.3))
        s["cache"].v[0].copy_(_randn(g, s["cache"].v[0].shape, dt, 0.5))
        s["cache"].pos = o
        cos, sin = (t.cuda() for t in rope_tables(case["D"], case["cap"], THETA))
        s["cos"], s["sin"] = cos[o:o + T], sin[o:o + T]
        return s
    s["prompt"] = torch.randint(case["vocab"], (1, o), generator=g, device="cuda")
    s["ids"] = torch.randint(case["vocab"], (T,), generator=g, device="cuda")
    s["dec"] = GraphDecoder(net, case["cap"], dt, T)
    net(s["prompt"], cache=s["dec"].cache)   # the prompt's prefill, then the graph is recorded once
    run(s)
    return s


# ---------------------------------------------------------------- one pass
@torch.no_grad()
def run(s):
    case = s["case"]
    if case["kind"] == "layer":
        s["cache"].pos = case["offset"]
        return {"y": s["net"](s["x"], s["cos"], s["sin"], s["cache"]), "k": s["cache"].k[0], "v": s["cache"].v[0]}
    if case["kind"] == "graph":
        dec = s["dec"]
        dec.cache.pos = case["offset"]
        return {"logits": dec.step(s["ids"]) if case["T"] == 1 else dec.verify(s["ids"]),
                "k": dec.cache.k[-1], "v": dec.cache.v[-1]}
    scale = case["D"] ** -0.5
    norm = dict(eps=EPS, cos=s["cos"], sin=s["sin"])
    if case["kind"] == "decode":
        where = dict(row_pos=s["row_pos"], max_kv_len=max(s["base"]) + case["T"]) if case["ragged"] else \
            dict(pos=s["base"][0])
        y = ops.attn_decode_append(s["q"], s["k"], s["v"], s["kc"], s["vc"], scale=scale, window=case["window"],
                                   q_weight=s["qw"], k_weight=s["kw"], norm_q=True, norm_k=True, **norm, **where)
    else:
        ops.kv_append(s["k"], s["v"], s["kc"], s["vc"], pos=case["offset"], k_weight=s["kw"], norm_k=True, **norm)
        y = ops.attn_prefill(s["q"], s["kc"], s["vc"], scale=scale, offset=case["offset"], window=case["window"],
                             q_weight=s["qw"], norm_q=True, doc_start=s["docs"], check_doc_start=False, **norm)
    return {"y": y, "k": s["kc"], "v": s["vc"]}


# ---------------------------------------------------------------- what a pass cannot do without
def _seen(base, T, window):
    """(query, key) pairs of T queries at base ..., and the keys that any of them sees."""
    pairs = sum(min(base + t + 1, window or base + t + 1) for t in range(T))
    keys = base + T if not window else min(base + T, window + T - 1)
    return pairs, keys


def work(case):
    e = torch.finfo(DTYPES[case["dtype"]]).bits // 8
    T, H, K, D, B = case["T"], case["H"], case["K"], case["D"], case.get("B", 1)
    if case["kind"] == "decode":
        rows = [_seen(n - T, T, case["window"]) for n in _lengths(case, 0)]
    elif case["kind"] == "prefill" and case["docs"]:
        rows = [(sum(t - d + 1 for t, d in enumerate(r)), T) for r in _doc_starts(case)]
    else:
        rows = [_seen(case["offset"], T, case.get("window", 0))] * B
    pairs, keys = sum(r[0] for r in rows), sum(r[1] for r in rows)
    # K and V of the visible keys, of which the new ones come from the projections; the new rows into
    # the cache; q in, the output out
    attn_bytes = e * D * (2 * K * keys + 2 * K * B * T + 2 * H * B * T)
    attn_flops = 4 * D * H * pairs
    if case["kind"] in ("decode", "prefill"):
        return {"bytes": attn_bytes, "flops": attn_flops}
    d = case["d_model"]
    weights = d * D * (2 * H + 2 * K)
    if case["kind"] == "layer":   # x in and y out; q, k, v and the heads' outputs need not leave the chip
        return {"bytes": e * (weights + 2 * B * T * d + D * (2 * K * keys + 2 * K * B * T)),
                "flops": attn_flops + 2 * B * T * weights}
    per_layer = weights + 3 * d * case["hidden"]
    n = case["layers"]
    return {"bytes": e * (n * (per_layer + D * (2 * K * keys + 2 * K * T)) + d * case["vocab"] + T * case["vocab"]),
            "flops": n * (attn_flops + 2 * T * per_layer) + 2 * T * d * case["vocab"]}


def tolerance(case):
    # Seen against 64 bits: 3-4e-3 in bf16 and 4-5e-4 in fp16 from the roundings of the outputs, of q
    # and k after RoPE and (in the matrix-core kernels) of the softmax weights, 5e-3 with a layer's
    # projections rounded too, 1.6e-2 at the logits of a four-layer model, 7e-7 in fp32. Two correct
    # implementations differ by about as much as each is off.
    rel = {"graph": {"bf16": 0.03, "fp16": 0.004}, "layer": {"bf16": 0.012, "fp16": 0.0015, "fp32": 1e-5}}.get(
        case["kind"], {"bf16": 8e-3, "fp16": 1e-3})[case["dtype"]]
    return {"rel": rel, "max": min(0.9, 12 * rel)}


# ---------------------------------------------------------------- the same in 64 bits
def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


@functools.lru_cache(maxsize=1)
def _tables(D):
    return [t.cuda() for t in rope_tables(D, 1 << 15, THETA)]


def _rope64(pos, D):
    """The rows of the fp32 tables that the inputs hold, as 64-bit values."""
    cos, sin = _tables(D)
    return cos[pos].double(), sin[pos].double()


def _rotate(x, cos, sin):
    a, b = x.chunk(2, -1)
    return x * cos + torch.cat([-b, a], -1) * sin


def _attend(q, k, v, base, window=0, docs=None):
    """q [H, T, D] at positions base ..., k/v [K, S, D], 64 bits -> [T, H, D]."""
    H, T, D = q.shape
    qpos = base + torch.arange(T, device=q.device)[:, None]
    kpos = torch.arange(k.shape[1], device=q.device)[None, :]
    hide = kpos > qpos
    if window:
        hide = hide | (qpos - kpos >= window)
    if docs is not None:
        hide = hide | (kpos < docs[:, None])
    out = torch.empty(T, H, D, dtype=torch.float64, device=q.device)
    for h in range(H):
        kv = h * k.shape[0] // H
        p = (q[h] @ k[kv].T * D ** -0.5).masked_fill(hide, -math.inf).softmax(-1)
        out[:, h] = p @ v[kv]
    return out


def _layer64(at, x, kc, vc, o, D):
    """One attention layer in 64 bits; kc/vc [B, K, S, D] hold the prefix and take the new rows."""
    B, T, _ = x.shape
    pos = o + torch.arange(T, device=x.device)
    cos, sin = _rope64(pos, D)
    heads = lambda m: (x @ m.weight.double().T).view(B, T, -1, D).transpose(1, 2)  # noqa: E731
    q = _rotate(_norm(heads(at.q_proj), at.q_norm.weight), cos, sin)
    kc[:, :, o:o + T] = _rotate(_norm(heads(at.k_proj), at.k_norm.weight), cos, sin)
    vc[:, :, o:o + T] = heads(at.v_proj)
    y = torch.stack([_attend(q[b], kc[b, :, :o + T], vc[b, :, :o + T], o) for b in range(B)])
    return y.reshape(B, T, -1) @ at.o_proj.weight.double().T


@torch.no_grad()
def exact(case, seed):
    s = prepare(case, seed)
    T, D = case["T"], case["D"]
    if case["kind"] == "layer":
        kc, vc = s["cache"].k[0].double(), s["cache"].v[0].double()
        return {"y": _layer64(s["net"], s["x"].double(), kc, vc, case["offset"], D), "k": kc, "v": vc}
    if case["kind"] == "graph":
        net, n = s["net"], case["offset"] + T
        x = net.tok_emb.weight.double()[torch.cat([s["prompt"][0], s["ids"]])][None]
        for b in net.blocks:
            kc = torch.zeros(1, case["K"], n, D, dtype=torch.float64, device="cuda")
            x = x + _layer64(b.attn, _norm(x, b.norm1.weight), kc, torch.zeros_like(kc), 0, D)
            h = _norm(x, b.norm2.weight)
            m = b.mlp
            x = x + (F.silu(h @ m.gate.weight.double().T) * (h @ m.up.weight.double().T)) @ m.down.weight.double().T
        logits = _norm(x, net.norm_f.weight) @ net.lm_head.weight.double().T
        return {"logits": logits[0, -T:], "k": None, "v": None}
    out = torch.empty(case["B"], T, case["H"], D, dtype=torch.float64, device="cuda")
    big = s["kc"].numel() > 1 << 28
    caches = (None, None) if big else (s["kc"].double(), s["vc"].double())
    for b in range(case["B"]):
        o = s["base"][b] if case["kind"] == "decode" else case["offset"]
        cos, sin = _rope64(o + torch.arange(T, device="cuda"), D)
        q = _rotate(_norm(s["q"][b].double(), s["qw"]), cos, sin)
        k, v = s["kc"][b, :, :o + T].double(), s["vc"][b, :, :o + T].double()
        k[:, o:] = _rotate(_norm(s["k"][b].double(), s["kw"]), cos, sin)
        v[:, o:] = s["v"][b].double()
        docs = s["docs"][b] if case["kind"] == "prefill" and case["docs"] else None
        out[b] = _attend(q, k, v, o, case.get("window", 0), docs)
        if not big:
            caches[0][b, :, :o + T], caches[1][b, :, :o + T] = k, v
    return {"y": out, "k": caches[0], "v": caches[1]}
