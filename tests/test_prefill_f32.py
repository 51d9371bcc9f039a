"""fp32 prefill on matrix cores (forge_attn_prefill_f32): results at the edges of its tiles, parts and
windows, its error against 64 bits beside the split-K path's, and the module's route to it."""

from __future__ import annotations

import math

import pytest
import torch

import oracle
from conftest import gpu_available
from helpers import gen, max_abs, randn, scale_of, tables, tol
from sleuth_amd import _lib

DEV = "cuda"
F32 = torch.float32


def test_rejections():
    """Each bad argument alone, everything else in order, is named by the error."""
    lib = _lib.lib()
    size = lib.forge_attn_prefill_f32_workspace_bytes
    assert size(1, 20, 8, 4, 32, 4000, 0) > 0 and size(8, 2048, 8, 4, 32, 0, 0) == 0
    assert size(1, 20, 8, 4, 256, 4000, 0) == 0 and size(1, 20, 8, 3, 32, 4000, 0) == 0
    ok = dict(D=32, K=4, q=4096, w=None, sqt=256, sks=32, offset=0, window=0, out=4096, ws=None)

    def call(**kw):
        a = {**ok, **kw}
        return lib.forge_attn_prefill_f32(1, 20, 8, a["K"], a["D"], a["q"], 0, 32, a["sqt"], a["w"], 1e-6, 0, None, None, 0,
                                          4096, 4096, 0, 32, a["sks"], a["offset"], a["window"], 1.0, a["out"], 0, 256, 32,
                                          a["ws"], 0, None)

    for kw, why in ((dict(out=None), "null"), (dict(q=None), "null"), (dict(D=256), "head dim"), (dict(K=3), "multiple of the KV"),
                    (dict(q=4100), "16-byte aligned"), (dict(out=4104), "16-byte aligned"), (dict(w=4100), "16-byte aligned"),
                    (dict(ws=4104), "16-byte aligned"), (dict(sks=34), "multiples of 16 bytes"),
                    (dict(sqt=258), "multiples of 16 bytes"), (dict(offset=-1), "offset"), (dict(window=-1), "window"),
                    (dict(offset=2 ** 31 - 276), "31 bits"), (dict(sks=28), "2^31 bytes"), (dict(offset=2 ** 24), "2^31 bytes"),
                    (dict(sks=2 ** 21), "stride too large"), (dict(sks=2 ** 20, offset=300), "2^31 bytes")):
        assert call(**kw) < 0, kw
        assert why in lib.forge_last_error().decode(), (kw, lib.forge_last_error())


def test_what_it_supports():
    """The rule sends every call that the kernel would refuse the split-K way."""
    from sleuth_amd import ops

    q, odd = torch.zeros(1, 4, 20, 32), torch.zeros(33)[1:]
    k = torch.empty_strided((1, 2, 40, 32), (80 * 2 ** 20, 40 * 2 ** 20, 2 ** 20, 1), device="meta")
    ok = lambda **kw: ops.prefill_f32_supported(q, **kw)  # noqa: E731
    assert ok() and ok(q_weight=torch.zeros(32), k=torch.zeros(1, 2, 40, 32), offset=20)
    assert not ok(q_weight=odd) and not ok(cos=odd[None].expand(20, 32))
    assert ok(k=k, offset=20) and not ok(k=k, offset=236)         # 2^20 * 4 * (offset + 20 + 256) < 2^31 or not
    assert not ok(k=k[..., :1, :].expand(1, 2, 40, 32))           # one row for every key
    assert not ops.prefill_f32_supported(q.half()) and not ops.prefill_f32_supported(torch.zeros(1, 4, 20, 256))


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("B,T,H,K,D,offset,window", [
    (1, 1, 4, 4, 32, 0, 0),          # one query, one key
    (2, 17, 8, 4, 32, 0, 0), (1, 32, 8, 4, 32, 0, 0), (1, 33, 8, 4, 64, 95, 0), (2, 129, 4, 2, 32, 127, 0),
    (1, 200, 6, 2, 64, 0, 50),       # windows shorter and longer than a wave's tile, starting inside one
    (1, 300, 4, 1, 128, 77, 200), (1, 150, 4, 4, 32, 1000, 1),
    (1, 20, 4, 2, 32, 4000, 0), (1, 40, 4, 2, 128, 2500, 0),   # key-split
    (3, 257, 16, 8, 128, 0, 0),
])
def test_fp32_prefill(B, T, H, K, D, offset, window):
    from sleuth_amd import ops

    S = offset + T
    g = gen(T + D + offset)
    q = randn(g, B, T, H, D).transpose(1, 2)
    w = 1 + 0.1 * randn(g, D)
    kc, vc = randn(g, B, K, S + 40, D), randn(g, B, K, S + 40, D)
    kc[:, :, S:] = float("nan")      # positions past the call's last key are never used
    vc[:, :, S:] = float("nan")
    cos, sin = (t[offset:S] for t in tables(D, S, 1e4))
    qn = oracle.head_norm_rope(q, w, 1e-6, cos, sin)
    ref = oracle.sdpa(qn.double(), kc[:, :, :S].double(), vc[:, :, :S].double(), offset, window, scale_of(D))
    dev = [t.to(DEV) for t in (q, kc, vc, w, cos, sin)]
    kw = dict(scale=scale_of(D), window=window, q_weight=dev[3], eps=1e-6, norm_q=True, cos=dev[4], sin=dev[5])
    got = ops.attn_prefill_f32(*dev[:3], offset=offset, **kw)
    assert max_abs(got.cpu().transpose(1, 2), ref.float()) <= tol(F32)
    # no less exact than the split-K path: both are within a few units of 2^-24 of 64 bits (2-norm), so a
    # factor of 1.3 covers what the draw of one case moves
    old = ops.attn_decode(*dev[:3], pos=offset, **kw)
    err = lambda y: ((y.cpu().transpose(1, 2).double() - ref).norm() / ref.norm()).item()  # noqa: E731
    assert err(got) <= 1.3 * max(err(old), 2.0 ** -24)


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("scale", [0.0, -0.3, 4.0])
def test_fp32_prefill_scales(scale):
    """Equal, reversed and very peaked weights (scores move the reference maximum often)."""
    from sleuth_amd import ops

    g = gen(7)
    q, k, v = randn(g, 1, 4, 100, 32), randn(g, 1, 2, 100, 32), randn(g, 1, 2, 100, 32)
    s = q.double() @ k.double().repeat_interleave(2, 1).transpose(-1, -2) * scale
    s = s.masked_fill(~torch.ones(100, 100, dtype=torch.bool).tril(), -math.inf)
    ref = (s.softmax(-1) @ v.double().repeat_interleave(2, 1)).transpose(1, 2)
    got = ops.attn_prefill_f32(q.to(DEV), k.to(DEV), v.to(DEV), scale=scale)
    assert max_abs(got.cpu(), ref.float()) <= tol(F32)


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
def test_module_takes_fp32_prompts_to_it_and_unaligned_tables_elsewhere(monkeypatch):
    from sleuth_amd import ops
    from sleuth_amd.attention import Attention
    from sleuth_amd.config import ModelConfig
    from sleuth_amd.kv_cache import KVCache

    torch.manual_seed(3)
    cfg = ModelConfig(vocab_size=16, d_model=128, n_layers=1, n_heads=4, n_kv_heads=2, qk_norm=True, max_seq_len=256)
    a = Attention(cfg, 0).to(DEV).eval()
    x = torch.randn(2, 60, 128, device=DEV)
    cos, sin = (t[:60].to(DEV) for t in tables(32, 64, 1e4))
    odd = [torch.empty(60 * 32 + 1, device=DEV)[1:].view(60, 32).copy_(t) for t in (cos, sin)]
    outs, calls, fn = [], [], ops.attn_prefill_f32
    monkeypatch.setattr(ops, "attn_prefill_f32", lambda *a, **kw: calls.append(1) or fn(*a, **kw))
    with torch.no_grad():
        for c, s in ((cos, sin), odd):
            cache = KVCache([(2, 32)], 2, 128, DEV, F32)
            outs.append((a(x, c, s, cache), cache.k[0].clone(), len(calls)))
    assert [o[2] for o in outs] == [1, 1]
    assert torch.equal(outs[0][1], outs[1][1])
    assert max_abs(outs[0][0], outs[1][0]) <= 1e-5   # fp32 sums in another order


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("what", ["gain", "slab"])
def test_module_takes_unaligned_gains_and_wide_slabs_the_split_k_way(monkeypatch, what):
    """A q_norm weight that is a view into a flat buffer, and a cache whose rows lie so far apart that
    only its own rows fit 2^31 bytes, give what an aligned gain and a dense cache give."""
    from host_protocol import HostKVCache
    from sleuth_amd import ops
    from sleuth_amd.attention import Attention
    from sleuth_amd.config import ModelConfig

    torch.manual_seed(4)
    cfg = ModelConfig(vocab_size=16, d_model=128, n_layers=1, n_heads=4, n_kv_heads=2, qk_norm=True, max_seq_len=64)
    a = Attention(cfg, 0).to(DEV).eval()
    a.q_norm.weight.data.copy_(torch.linspace(0.8, 1.2, 32))
    x = torch.randn(1, 60, 128, device=DEV)
    cos, sin = (t[:60].to(DEV) for t in tables(32, 64, 1e4))
    calls, fn = [], ops.attn_prefill_f32
    monkeypatch.setattr(ops, "attn_prefill_f32", lambda *a, **kw: calls.append(1) or fn(*a, **kw))

    def run():
        calls.clear()
        with torch.no_grad():
            return a(x, cos, sin, cache), cache.k[0].clone(), len(calls)

    cache = HostKVCache([(2, 32)], 1, 60, DEV, F32)
    want = run()
    if what == "gain":
        flat = torch.empty(33, device=DEV)
        flat[1:] = a.q_norm.weight.detach()
        a.q_norm.weight.data = flat[1:]
    else:
        row = 2 ** 21       # floats: 61 rows span 0.5 GB, 316 of them 2.7 GB
        for kv in (cache.k, cache.v):
            kv[0] = torch.zeros(60 * row, device=DEV).as_strided((1, 2, 60, 32), (64, 32, row, 1))
    got = run()
    assert (want[2], got[2]) == (1, 0)
    assert torch.equal(want[1], got[1]) and max_abs(want[0], got[0]) <= 1e-5   # fp32 sums in another order


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("T,offset,taken", [(17, 0, 0), (20, 28, 0), (48, 0, 0), (49, 0, 1), (17, 32, 1)])
def test_module_keeps_few_keys_on_the_split_k_path(monkeypatch, T, offset, taken):
    """Up to 48 keys, where the matrix-core kernel's sums are no more exact: the split-K call's own bits."""
    from sleuth_amd import ops
    from sleuth_amd.attention import Attention
    from sleuth_amd.config import ModelConfig
    from sleuth_amd.kv_cache import KVCache

    torch.manual_seed(5)
    cfg = ModelConfig(vocab_size=16, d_model=128, n_layers=1, n_heads=4, n_kv_heads=2, qk_norm=True, max_seq_len=64)
    a = Attention(cfg, 0).to(DEV).eval()
    x = torch.randn(1, T, 128, device=DEV)
    cos, sin = (t[offset:offset + T].to(DEV) for t in tables(32, 64, 1e4))
    outs, calls, fn = [], [], ops.attn_prefill_f32
    monkeypatch.setattr(ops, "attn_prefill_f32", lambda *a, **kw: calls.append(1) or fn(*a, **kw))
    for least in (ops.PREFILL_F32_MIN_KEYS, 1000):
        monkeypatch.setattr(ops, "PREFILL_F32_MIN_KEYS", least)
        cache = KVCache([(2, 32)], 1, 64, DEV, F32)
        cache.pos = offset
        with torch.no_grad():
            outs.append(a(x, cos, sin, cache))
    assert len(calls) == taken
    assert max_abs(*outs) <= 1e-5 and (taken or torch.equal(*outs))   # fp32 sums in another order, or the same
