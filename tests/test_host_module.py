"""The native host module (csrc/host.cpp): it declines what it does not take, and the calls that it takes
give the Python way's results bit for bit, errors included."""

from __future__ import annotations

import sys
import threading
import time
import types

import pytest
import torch

from conftest import gpu_available
from helpers import gen, qkv_proj_views, randn, tables
from sleuth_amd import _lib, ops

DEV = "cuda"
needs_gpu = pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
DECLINE = types.SimpleNamespace(**{n: (lambda *a: None) for n in ("decode_append", "kv_append", "prefill", "linear_small")})


def test_declines_what_is_no_plain_gpu_tensor():
    h = _lib.host()
    t, i = torch.zeros(1, 2, 1, 64), torch.zeros(1, dtype=torch.long)
    for bad in (t, None, 3, "x", [t]):
        assert h.decode_append({}, bad, t, t, t, t, 1.0, 0, None, None, None, 0, None, None, 1e-6, False, False, False, None,
                               None, 0) is None
        assert h.kv_append(bad, t, t, t, 0, None, 1e-6, False, False, None, None) is None
        assert h.prefill(bad, t, t, 1.0, 0, 0, None, 1e-6, False, None, None) is None
        assert h.linear_small(bad, t[0, :, 0], None, None, None, 0.0, False, None) is None
        assert h.tensors_are((bad,), (id(bad),), ((0, 0),), t) is None
    with pytest.raises(TypeError):
        h.kv_append(t, i)


class Recorder:
    """The native module, with what its functions returned: taken (a result or a status) or declined."""

    def __init__(self):
        self.taken = []

    def __getattr__(self, name):
        fn = getattr(_lib.host(), name)

        def call(*a):
            r = fn(*a)
            self.taken.append(r is not None)
            return r
        return call


def _both(monkeypatch, call, taken=None):
    """call() the Python way and the native way: results, or the errors' types and texts. taken: whether the
    native functions take the calls, one value each."""
    out, rec = [], Recorder()
    for native in (False, True):
        with monkeypatch.context() as m:
            m.setattr(ops, "host", (lambda: rec) if native else lambda: DECLINE)
            try:
                out.append(call())
            except Exception as e:   # compared, not swallowed
                out.append((type(e), str(e)))
    assert taken is None or rec.taken == taken, (rec.taken, taken)
    return out


def _equal(a, b):
    if isinstance(a, torch.Tensor):
        return isinstance(b, torch.Tensor) and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)
    return a == b if not isinstance(a, (list, tuple)) or isinstance(a[0], type) else \
        len(a) == len(b) and all(_equal(x, y) for x, y in zip(a, b))


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("where", ["pos", "pos_dev", "row_pos", "none"])
@pytest.mark.parametrize("T,H,K,D,window", [(1, 4, 2, 64, 0), (5, 8, 2, 128, 40), (3, 8, 1, 256, 0), (20, 4, 4, 32, 0)])
def test_decode_append_equals_the_python_way(monkeypatch, dtype, where, T, H, K, D, window):
    B, L = 2, 300
    g = gen(T + D)
    q, k, v = (t.to(DEV) for t in qkv_proj_views(g, B, T, H, K, D, dtype))
    cache = randn(g, 2, B, L, K, D, dtype=dtype).transpose(2, 3).to(DEV)     # [2, B, K, L, D], heads inside the rows
    cos, sin = (t[:B * T].view(B, T, D).to(DEV) for t in tables(D, 64, 1e4))
    kw = {"pos": dict(pos=250), "pos_dev": dict(pos_dev=torch.tensor([250], device=DEV)),
          "row_pos": dict(row_pos=torch.tensor([250, 3], dtype=torch.int32, device=DEV)), "none": {}}[where]
    w = torch.linspace(0.9, 1.1, D, device=DEV)
    f32 = dtype == torch.float32
    # the native way takes what needs no conversion (once the stream has its workspace) and leaves the rest
    for tab, gain, norm, plain in ((dict(cos=cos, sin=sin), w, True, True), (dict(cos=cos[0], sin=sin[0]), w.to(dtype), True, f32),
                                   ({}, None, False, True), (dict(cos=cos[:, :, ::1].double(), sin=sin.double()), None, True, False),
                                   (dict(cos=cos), w, True, False),
                                   (dict(cos=cos[:, :1], sin=sin[:, :1]), w, True, T == 1)):
        def call():
            kc, vc = cache[0].clone(memory_format=torch.preserve_format), cache[1].clone(memory_format=torch.preserve_format)
            y = ops.attn_decode_append(q, k, v, kc, vc, scale=0.1, window=window, q_weight=gain, k_weight=gain, norm_q=norm,
                                       norm_k=norm, norm_v=norm, **tab, **kw)
            return [y, kc, vc]
        a, b = _both(monkeypatch, call, [plain])
        assert _equal(a, b), (a, b)


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_prefill_and_append_equal_the_python_way(monkeypatch, dtype):
    B, T, H, K, D, L = 2, 40, 4, 2, 64, 200
    g = gen(3)
    q, k, v = (t.to(DEV) for t in qkv_proj_views(g, B, T, H, K, D, dtype))
    kc0, vc0 = (randn(g, B, K, L, D, dtype=dtype).to(DEV) for _ in range(2))
    cos, sin = (t[100:100 + T].to(DEV) for t in tables(D, 200, 1e4))
    w = torch.linspace(0.9, 1.1, D, device=DEV)
    fn = ops.attn_prefill_f32 if dtype == torch.float32 else ops.attn_prefill
    for off, kk, extra, taken in ((100, k, {}, [True, True]), (100, k.to(torch.float16), {}, [False, True]),
                                  (190, k, {}, [True]), (100, k[..., :32], {}, [False]), (100, k, dict(window=30), [True, True]),
                                  (0, k, dict(cos=cos, sin=sin), [True, True]), (-1, k, {}, [True])):
        def call():
            kc, vc = kc0.clone(), vc0.clone()
            ops.kv_append(kk, v, kc, vc, pos=off, k_weight=w, norm_k=True, cos=cos, sin=sin)
            y = fn(q, kc, vc, scale=0.2, offset=off, q_weight=w, norm_q=True, **extra)
            return [y, kc, vc]
        a, b = _both(monkeypatch, call, taken)
        assert _equal(a, b), (off, extra, a, b)
    for off in (161, 2 ** 31, 2 ** 63 - 20):     # past the keys' end, also where the end wraps
        a, b = _both(monkeypatch, lambda: fn(q, kc0, vc0, scale=0.2, offset=off), [False])
        assert a == b and a[0] is ValueError, (off, a, b)


@pytest.mark.gpu
@needs_gpu
def test_streams_and_threads_have_workspaces_of_their_own():
    """Split-K decodes in two threads, each on its own stream, many at once: every result equals the
    one made alone (a shared workspace would mix their partials)."""
    g = gen(4)
    sets = []
    for _ in range(2):
        q, k, v = (t.to(DEV) for t in qkv_proj_views(g, 4, 1, 8, 2, 128, torch.bfloat16))
        sets.append((q, k, v, randn(g, 4, 2, 3000, 128, dtype=torch.bfloat16).to(DEV),
                     randn(g, 4, 2, 3000, 128, dtype=torch.bfloat16).to(DEV)))
    call = lambda s: ops.attn_decode_append(*s, scale=0.1, pos=2900, chunk=256)  # noqa: E731
    want = [call(s) for s in sets]
    torch.cuda.synchronize()
    got = [[], []]

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            got[i] = [call(sets[i]) for _ in range(50)]
            torch.cuda.current_stream().synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(len(got[i]) == 50 and all(torch.equal(y, want[i]) for y in got[i]) for i in range(2))


@pytest.mark.gpu
@needs_gpu
def test_launches_give_up_the_gil():
    """With the interpreter's own switching all but off, a waiting thread runs only if the native calls
    give the GIL up around their launches."""
    k = torch.zeros(1, 1, 1, 64, dtype=torch.bfloat16, device=DEV)
    (kc, vc), append = torch.zeros(2, 1, 1, 4, 64, dtype=torch.bfloat16, device=DEV), ops.host().kv_append
    started, ran, interval = threading.Event(), [], sys.getswitchinterval()

    def other():
        started.set()
        time.sleep(0.01)       # until the loop below holds the GIL
        ran.append(1)

    thread = threading.Thread(target=other)
    try:
        thread.start()
        started.wait()
        sys.setswitchinterval(1000.0)
        for n in range(30000):
            assert append(k, k, kc, vc, 0, None, 0.0, False, False, None, None) == 0   # (no torch call beside it)
            if ran:
                break
        assert ran
    finally:
        sys.setswitchinterval(interval)
        thread.join()
        torch.cuda.synchronize()


@pytest.mark.gpu
@needs_gpu
@pytest.mark.parametrize("native", [False, True])
def test_a_streams_workspace_is_out_of_the_table_during_a_call(monkeypatch, native):
    """Threads on one stream: while a call launches, the table must not hand its buffer to another."""
    g = gen(6)
    q, k, v = (t.to(DEV) for t in qkv_proj_views(g, 1, 1, 4, 2, 64, torch.bfloat16))
    kc, vc = (randn(g, 1, 2, 3000, 64, dtype=torch.bfloat16).to(DEV) for _ in range(2))
    call = lambda: ops.attn_decode_append(q, k, v, kc, vc, scale=0.1, pos=2900, chunk=256)  # noqa: E731
    key = (torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream)
    ops._STREAM_WS.pop(key, None)
    want = call()
    buf = ops._STREAM_WS[key]
    if native:
        # the native call takes the buffer and puts it back: nothing else of the table changes
        others = {("other", i): torch.zeros(1) for i in range(3)}
        table = {key: buf, **others}
        monkeypatch.setattr(ops, "_STREAM_WS", table)
        assert torch.equal(call(), want)
        assert list(table)[-1] == key and table[key] is buf and len(table) == 4
    else:
        monkeypatch.setattr(ops, "host", lambda: DECLINE)
        fn, during = _lib.lib().forge_attn_decode_append, []

        class Lib:
            def __getattr__(self, name):
                real = getattr(_lib.lib(), name)
                return (lambda *a: during.append(key in ops._STREAM_WS) or fn(*a)) if name == fn.__name__ else real
        monkeypatch.setattr(ops, "lib", Lib)
        assert torch.equal(call(), want)
        assert during == [False] and ops._STREAM_WS[key] is buf
