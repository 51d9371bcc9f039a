"""forge_linear_small, the projections of a decode or verify step, against torch in 64 bits with the
eager layers' roundings, and the block's use of it."""

from __future__ import annotations

import types

import pytest
import torch
import torch.nn.functional as F

from conftest import gpu_available
from helpers import gen, randn
from sleuth_amd import _lib

DEV = "cuda"
needs_gpu = pytest.mark.skipif(not gpu_available(), reason="needs a GPU")


def test_rejections():
    lib = _lib.lib()

    def call(dtype=_lib.BF16, M=1, N=16, K=64, x=4096, sx=64, w=4096, w2=None, sw=64, bias=None, gain=None, gd=0, out=None):
        return lib.forge_linear_small(dtype, M, N, K, x, sx, w, w2, sw, bias, gain, gd, 0, 0.0, None, 0, out, N, None)

    for kw in (dict(), dict(dtype=_lib.F32), dict(M=17), dict(M=0), dict(K=48), dict(x=4098), dict(sw=60), dict(M=2, sx=56),
               dict(w2=4096, bias=4096),
               dict(gain=4096, gd=_lib.F16)):
        assert call(**{"out": 4096 if kw else None, **kw}) < 0


def test_rows_up_to_which_the_launch_is_taken():
    """Shapes measured on either side of the rule's lines (N, K -> rows per form)."""
    rows = _lib.lib().forge_linear_small_rows
    want = {   # plain, residual, norm, gated
        (4096, 1024): (16, 16, 16, 16), (1024, 3072): (16, 16, 16, 16), (4096, 4096): (16, 16, 16, 16),
        (8192, 2048): (16, 16, 16, 16), (10240, 768): (12, 12, 16, 16), (9216, 1024): (16, 16, 16, 16), (12288, 1024): (16, 16, 16, 16), (6144, 4096): (0, 0, 8, 16), (5120, 5120): (0, 0, 0, 4),
        (4096, 14336): (0, 4, 0, 0), (4096, 16384): (0, 0, 0, 0), (14336, 4096): (0, 0, 4, 8), (28672, 8192): (0, 0, 0, 4),
        (32768, 2048): (0, 0, 16, 0), (151936, 1024): (0, 0, 16, 0), (128256, 4096): (0, 0, 0, 0),
        (163840, 2048): (0, 0, 4, 0), (131072, 512): (0, 0, 0, 0), (65536, 128): (0, 0, 0, 0), (16403, 64): (16, 16, 16, 16)}
    for (N, K), w in want.items():
        assert (rows(N, K, 0, 0, 0), rows(N, K, 0, 0, 1), rows(N, K, 1, 0, 0)) == w[:3], (N, K)
        if N < 16403:
            assert rows(N, K, 1, 1, 0) == w[3], (N, K)
    assert rows(0, 64, 0, 0, 0) == rows(64, 48, 0, 0, 0) == rows(64, 0, 1, 1, 0) == 0


@pytest.mark.gpu
@needs_gpu
def test_torch_takes_the_shapes_that_it_is_faster_at():
    """A layer of a wide model: the rule's rows go through the kernel, one more through torch."""
    from sleuth_amd import ops

    x, w = torch.randn(9, 4096, device=DEV).bfloat16(), torch.randn(6144, 4096, device=DEV).bfloat16()
    gain = torch.ones(4096, device=DEV)
    kw = dict(gain=gain, eps=1e-6, norm=True)
    assert ops.linear_small(x[:8], w, **kw) is not None and ops.linear_small(x, w, **kw) is None
    assert ops.linear_small(x[:1], w) is None


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("N,K", [(1, 32), (17, 96), (100, 1024), (40, 2048), (40, 3072), (256, 3104), (16403, 64), (16384, 288)])
@pytest.mark.parametrize("form", ["plain", "bias", "norm", "norm+residual", "swiglu", "norm+swiglu"])
def test_linear_small(dtype, M, N, K, form):
    from sleuth_amd import ops

    g = gen(N + K + M)
    x = randn(g, M, K, dtype=dtype)
    w, u = (randn(g, N, K, dtype=dtype) * 0.05 for _ in range(2))
    bias, res, gain = randn(g, N, dtype=dtype), randn(g, M, N, dtype=dtype), 1 + 0.1 * randn(g, K)
    rnd = lambda t: t.to(dtype).double()  # noqa: E731
    xn = x.double()
    if "norm" in form:
        xn = rnd(xn * torch.rsqrt(xn.square().mean(-1, keepdim=True) + 1e-6) * gain.double())
    y = xn @ w.double().T
    if form == "bias":
        y = y + bias.double()
    if "swiglu" in form:
        y = rnd(F.silu(rnd(y))) * rnd(xn @ u.double().T)
    if "residual" in form:
        y = rnd(y) + res.double()
    d = lambda t: t.to(DEV)  # noqa: E731
    kw = dict(w_up=d(u) if "swiglu" in form else None, gain=d(gain) if "norm" in form else None, eps=1e-6,
              norm="norm" in form, residual=d(res) if "residual" in form else None)
    call = lambda rows, **o: ops.linear_small(d(x)[rows].contiguous(), d(w), d(bias) if form == "bias" else None,  # noqa: E731
                                              **{**kw, **o})
    got = call(slice(None))
    # relative to the value, a rounding moves it by at most 2^-p (p = 8, 11: half a spacing), and by
    # twice that against the reference's where fp32 and 64 bits fall on either side of an edge; a
    # single value (M = N = 1) can meet that at each of its roundings: of x, gate, silu, up, the
    # product before the sum, and the result (whose reference is not rounded: 2^-p)
    ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    inner = {"plain": 0, "bias": 0, "norm": 1, "norm+residual": 2, "swiglu": 3, "norm+swiglu": 4}[form]
    err = (got.cpu().double() - y).norm() / y.norm()
    assert err.item() <= ulp * (1 + 2 * inner)
    if "norm" in form:                        # a gain of x's type, read as it is
        low = d(gain).to(dtype)
        assert torch.equal(call(slice(None), gain=low), call(slice(None), gain=low.float()))
    one = call(slice(M - 1, M), residual=d(res)[M - 1:] if "residual" in form else None)
    assert torch.equal(one, got[M - 1:])      # a row does not depend on the others


@pytest.mark.gpu
@needs_gpu
def test_declines_what_stands_between_the_call_and_the_memory():
    """Forward-mode tangents, tensor subclasses, tracing, function and dispatch modes: torch's own call."""
    import torch.autograd.forward_ad as fwd
    from torch.utils._python_dispatch import TorchDispatchMode
    from sleuth_amd import ops

    class Sub(torch.nn.Parameter):
        pass

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x, w = torch.ones(1, 64, dtype=torch.bfloat16, device=DEV), torch.ones(16, 64, dtype=torch.bfloat16, device=DEV)
    with torch.no_grad():
        assert ops.linear_small(x, w) is not None and ops.linear_small(x, torch.nn.Parameter(w)) is not None
        assert ops.linear_small(x, Sub(w)) is None
        with fwd.dual_level():
            assert ops.linear_small(fwd.make_dual(x, x), w) is None
            assert ops.linear_small(x, fwd.make_dual(w, w)) is None
        for mode in (Mode(), torch.overrides.BaseTorchFunctionMode()):
            with mode:
                assert ops.linear_small(x, w) is None
        seen = []
        torch.jit.trace(lambda t: seen.append(ops.linear_small(t, w)) or t + 1, x, check_trace=False)
        assert seen == [None]


def _model(**kw):
    from sleuth_amd.config import ModelConfig
    from sleuth_amd.model import Transformer

    torch.manual_seed(5)
    cfg = ModelConfig(vocab_size=128, d_model=128, n_layers=2, n_heads=4, n_kv_heads=2, qk_norm=True, max_seq_len=128,
                      ffn_hidden=160, init_std=0.05, **kw)
    return Transformer(cfg).to(DEV, torch.bfloat16).eval()


def _block_and_step():
    """A block on the CPU, and a stand-in for the one GPU row that its dispatch looks at."""
    from sleuth_amd.config import ModelConfig
    from sleuth_amd.model import Block

    cfg = ModelConfig(vocab_size=16, d_model=64, n_layers=1, n_heads=2, n_kv_heads=1, max_seq_len=32, ffn_hidden=64)
    return Block(cfg, 0), types.SimpleNamespace(numel=lambda: 64, shape=(1, 1, 64), is_cuda=True)


@torch.no_grad()
def test_what_stands_in_for_a_tap_turns_the_fused_step_off():
    blk, x = _block_and_step()
    assert blk._small_step(x)
    for name in ("tap_attn_out", "tap_resid_post"):
        tap = getattr(blk, name)
        for register in (tap.register_forward_hook, tap.register_forward_pre_hook):
            h = register(lambda *a: None)
            assert not blk._small_step(x)
            h.remove()
        tap.listeners.append(lambda name, t: None)
        assert not blk._small_step(x)
        tap.listeners.clear()
        tap.forward = lambda t: 2 * t
        assert not blk._small_step(x)
        del tap.forward
        setattr(blk, name, torch.nn.Dropout(0.5))
        assert not blk._small_step(x)
        setattr(blk, name, tap)
        assert blk._small_step(x)


@torch.no_grad()
def test_what_stands_in_for_a_class_turns_the_fused_step_off(monkeypatch):
    import functools

    from sleuth_amd.attention import Attention
    from sleuth_amd.model import SwiGLU
    from sleuth_amd.norm import RMSNorm

    blk, x = _block_and_step()
    for cls in (Attention, SwiGLU, RMSNorm, torch.nn.Linear, type(blk.tap_attn_out)):
        own = cls.forward
        for other in (lambda self, *a, **kw: None, functools.wraps(own)(lambda self, *a, **kw: own(self, *a, **kw)),
                      functools.partialmethod(own)):
            with monkeypatch.context() as m:
                m.setattr(cls, "forward", other)
                assert not blk._small_step(x), cls
    for name in ("__call__", "_call_impl"):
        with monkeypatch.context() as m:
            m.setattr(torch.nn.Module, name, lambda self, *a, **kw: None)
            assert not blk._small_step(x)
    assert blk._small_step(x)
    for part in (blk.attn, blk.mlp, blk.norm1, blk.mlp.down):
        part.compile()
        assert not blk._small_step(x)
        part._compiled_call_impl = None
    assert blk._small_step(x)


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("T", [1, 5])
def test_block_step_and_what_turns_its_fusion_off(T, monkeypatch):
    """A decode/verify step takes four fused launches per block (and one for the head); a hook, a
    listener, a replaced forward, autograd or a prompt keep the modules' own calls, with equal
    logits up to bf16 roundings."""
    from sleuth_amd import ops
    from sleuth_amd.kv_cache import KVCache
    from sleuth_amd.taps import listen

    m = _model()
    prompt, ids = torch.randint(0, 128, (1, 40), device=DEV), torch.randint(0, 128, (1, T), device=DEV)
    calls, fn = [], ops.linear_small
    monkeypatch.setattr(ops, "linear_small", lambda *a, **kw: calls.append(1) or fn(*a, **kw))

    @torch.no_grad()
    def step():
        cache = KVCache.for_model(m, 1)
        m(prompt, cache=cache)
        calls.clear()
        return m(ids, cache=cache).logits.float(), len(calls)

    step()
    fused, n = step()
    assert n == 2 * 4 + 1
    blk = m.blocks[0]

    def same(want):
        y, k = step()
        assert k == want and ((y - fused).norm() / fused.norm()).item() <= 0.03   # two layers of bf16 roundings
    seen = []
    h = blk.norm2.register_forward_hook(lambda mod, a, out: seen.append(out.shape))
    same(5 + 2)                                  # the other block and the head; this one's q/k/v and o_proj
    assert len(seen) == 2                        # the prompt and the step
    h.remove()
    with listen(m, {"blocks.0.resid_post": lambda name, x: seen.append(1)}):
        same(5 + 2)
    for name in ("tap_attn_out", "tap_resid_post"):
        seen.clear()
        h = getattr(blk, name).register_forward_hook(lambda mod, a, out: seen.append(out.shape))
        same(5 + 2)
        assert len(seen) == 2                    # the prompt and the step
        h.remove()
    tap, blk.tap_attn_out = blk.tap_attn_out, torch.nn.Identity()
    same(5 + 2)
    blk.tap_attn_out = tap
    blk.mlp.forward = type(blk.mlp).forward.__get__(blk.mlp)
    same(5 + 2)
    del blk.mlp.forward
    calls.clear()
    m(ids).logits.sum().backward()               # autograd: none
    assert not calls and m.blocks[0].mlp.down.weight.grad is not None


@pytest.mark.gpu
@needs_gpu
def test_recorded_step_reads_the_norm_gains_live():
    """A recorded step multiplies by the norms' parameters themselves: gains changed in place between
    replays count at once, and no copy of them is freed under the graph."""
    from sleuth_amd.generate import GraphDecoder
    from sleuth_amd.kv_cache import KVCache

    m = _model()
    prompt, ids = torch.randint(0, 128, (1, 40), device=DEV), torch.randint(0, 128, (1,), device=DEV)
    dec = GraphDecoder(m, 64, torch.bfloat16)

    @torch.no_grad()
    def both():
        dec.cache.reset()
        m(prompt, cache=dec.cache)
        got = dec.step(ids).clone()
        cache = KVCache.for_model(m, 1)
        m(prompt, cache=cache)
        want = m(ids[None], cache=cache).logits[0]
        return got.float(), want.float()

    both()
    for scale in (0.5, 3.0):
        with torch.no_grad():
            for n in (m.blocks[0].norm1, m.blocks[1].norm2, m.norm_f):
                n.weight.copy_(torch.linspace(0.5, 1.5, n.weight.numel(), device=DEV) * scale)
        got, want = both()
        assert ((got - want).norm() / want.norm()).item() <= 0.03   # two layers of bf16 roundings
