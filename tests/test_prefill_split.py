"""The key-split prefill launch (forge_attn_prefill_ws): when it splits, and its results at the
edges of its parts, tiles and windows against the oracle and the unsplit launch."""

from __future__ import annotations

import types

import pytest
import torch

import oracle
from conftest import gpu_available
from helpers import gen, max_abs, randn, scale_of, tables, tol
from sleuth_amd import _lib

DEV = "cuda"


def _bytes(B, T, H, K, D, offset, window=0, dtype=_lib.BF16):
    return _lib.lib().forge_attn_prefill_workspace_bytes(dtype, B, T, H, K, D, offset, window)


def test_split_rule():
    """Chunks of long prompts split (each partial: D + 2 floats per row and part); launches that
    fill the CUs do not, nor short prompts, and refused shapes need nothing."""
    row = 512 * 16
    need = _bytes(1, 512, 16, 8, 128, 15360)
    parts = need // (row * (128 + 2) * 4)
    assert 2 <= parts <= 32 and need == parts * row * 4 * (128 + 2)
    assert _bytes(1, 64, 16, 8, 128, 1000) > 0 and _bytes(1, 600, 16, 1, 512, 8000) > 0
    assert _bytes(4, 4096, 16, 8, 128, 0) == 0      # 2,048 query tiles
    assert _bytes(1, 2048, 16, 8, 128, 0) == 0      # the partials would cost what the split saves
    assert _bytes(1, 333, 16, 8, 128, 0) == 0
    assert _bytes(1, 512, 16, 8, 128, 15360, window=64) == 0   # few keys per query
    assert _bytes(1, 512, 16, 8, 128, 15360, dtype=_lib.F32) == 0
    assert _bytes(1, 512, 16, 8, 32, 15360) == 0 and _bytes(1, 512, 16, 3, 128, 15360) == 0


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("docs,name", [(False, "forge_attn_prefill"), (True, "forge_attn_prefill_docs")])
def test_a_rejected_call_names_its_entry_point(docs, name):
    from sleuth_amd import ops

    q, k = (torch.zeros(1, 2, 20, 64, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    odd = torch.zeros(1281, device=DEV)[1:].view(20, 64)       # tables the kernel refuses: not 16-byte aligned
    starts = torch.zeros(1, 20, dtype=torch.int32, device=DEV) if docs else None
    with pytest.raises(_lib.ForgeError, match=name + r"\b"):
        ops.attn_prefill(q, k, k, scale=1.0, cos=odd, sin=odd, doc_start=starts)


def test_workspace_too_small_is_rejected():
    lib = _lib.lib()
    need = _bytes(1, 512, 16, 8, 128, 15360)
    args = [_lib.BF16, 1, 512, 16, 8, 128, 4096, 0, 128, 2048, None, 1e-6, 0, None, None, 0, 4096, 4096, 0, 128, 1024,
            15360, 0, 1.0, None, 0, 4096, 0, 128, 2048]
    assert lib.forge_attn_prefill_ws(*args, 4096, need - 1, None) < 0
    assert b"workspace" in lib.forge_last_error()
    assert lib.forge_attn_prefill_ws(*args, 4104, need, None) < 0


CASES = [
    # dtype, B, T, H, K, D, offset, window: one query; one tile and a query; odd group; windows
    # whose first part starts inside a tile and whose parts hold no key of some queries; hd 512 with
    # two heads per block and (odd group) one
    (torch.bfloat16, 1, 1, 4, 2, 128, 4095, 0),
    (torch.bfloat16, 1, 17, 16, 8, 128, 3001, 0),
    (torch.float16, 1, 129, 6, 2, 64, 2500, 0),
    (torch.bfloat16, 2, 200, 3, 3, 128, 1900, 0),
    (torch.float16, 1, 257, 4, 1, 256, 1500, 0),
    (torch.bfloat16, 1, 1800, 8, 4, 256, 0, 0),
    (torch.bfloat16, 1, 130, 4, 2, 128, 5000, 1500),
    (torch.float16, 1, 640, 4, 4, 64, 1000, 700),
    (torch.bfloat16, 1, 65, 4, 1, 512, 1777, 0),
    (torch.float16, 1, 33, 3, 1, 512, 2000, 900),
]


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("case", range(len(CASES)))
def test_split_prefill_against_oracle(case):
    from sleuth_amd import ops

    dtype, B, T, H, K, D, offset, window = CASES[case]
    S = offset + T
    g = gen(900 + case)
    q = randn(g, B, T, H, D, dtype=dtype).transpose(1, 2)
    w = (1 + 0.1 * randn(g, D)).to(dtype)
    kc, vc = randn(g, B, K, S + 3, D, dtype=dtype), randn(g, B, K, S + 3, D, dtype=dtype)
    vc[:, :, S:] = 1e4                     # positions past the call's last key are never read
    cos, sin = (t[offset:S] for t in tables(D, S, 1e4))
    qn = oracle.head_norm_rope(q, w, 1e-6, cos, sin)
    ref = oracle.sdpa(qn.float(), kc[:, :, :S].float(), vc[:, :, :S].float(), offset, window, scale_of(D))
    dev = [t.to(DEV) for t in (q, kc, vc, w, cos, sin)]
    kw = dict(q_weight=dev[3], eps=1e-6, norm_q=True, cos=dev[4], sin=dev[5], scale=scale_of(D), offset=offset,
              window=window)
    assert _bytes(B, T, H, K, D, offset, window, _lib.BF16) > 0
    got = ops.attn_prefill(*dev[:3], **kw)
    assert max_abs(got.cpu().transpose(1, 2), ref) <= tol(dtype)
    # the unsplit launch (documents are never split; starts of 0 hide nothing): both round the
    # weights and the outputs once to the dtype, so each is within 2 * 2^-p of exact in 2-norm
    # (p = 9 in bf16, 12 in fp16)
    whole = ops.attn_prefill(*dev[:3], doc_start=torch.zeros(B, T, dtype=torch.int32, device=DEV), **kw).float()
    eps = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    assert ((got.float() - whole).norm() / whole.norm()).item() <= 4 * eps
    assert torch.equal(ops.attn_prefill(*dev[:3], **kw), got)


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
def test_split_prefill_under_graph_capture():
    """The partials' workspace belongs to the graph: replays on new inputs equal the eager calls."""
    from sleuth_amd import ops

    B, T, H, K, D, offset = 1, 96, 8, 4, 128, 3000
    g = gen(950)
    q = randn(g, B, H, T, D, dtype=torch.bfloat16).to(DEV)
    kc, vc = (randn(g, B, K, offset + T, D, dtype=torch.bfloat16).to(DEV) for _ in range(2))
    call = lambda: ops.attn_prefill(q, kc, vc, scale=scale_of(D), offset=offset)  # noqa: E731
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for seed in range(3):
        q.copy_(randn(gen(960 + seed), B, H, T, D, dtype=torch.bfloat16))
        want = call()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("dtype,window,docs", [(torch.bfloat16, 0, False), (torch.float16, 300, False),
                                               (torch.bfloat16, 0, True)])
def test_wide_prefill_with_four_heads_per_block(dtype, window, docs):
    """Head dim 512 with enough query tiles for four heads per block (eight waves): 701 queries (a
    last tile of 29), raw q with norm and RoPE, two KV heads of eight query heads each."""
    from sleuth_amd import ops

    B, T, H, K, D = 3, 701, 16, 2, 512
    g = gen(980)
    q = randn(g, B, T, H, D, dtype=dtype).transpose(1, 2)
    w = (1 + 0.1 * randn(g, D)).to(dtype)
    k, v = randn(g, B, K, T, D, dtype=dtype), randn(g, B, K, T, D, dtype=dtype)
    cos, sin = tables(D, T, 1e4)
    starts = torch.tensor([0] * 100 + [100] * 301 + [401] * 300, dtype=torch.int32)[None].expand(B, T).contiguous()
    qn = oracle.head_norm_rope(q, w, 1e-6, cos, sin)
    same = (starts[:, :, None] == starts[:, None, :])[:, None] if docs else None
    ref = oracle.sdpa(qn.float(), k.float(), v.float(), 0, window, scale_of(D), same_doc=same)
    got = ops.attn_prefill(q.to(DEV), k.to(DEV), v.to(DEV), scale=scale_of(D), window=window, q_weight=w.to(DEV),
                           eps=1e-6, norm_q=True, cos=cos.to(DEV), sin=sin.to(DEV),
                           doc_start=starts.to(DEV) if docs else None)
    assert max_abs(got.cpu().transpose(1, 2), ref) <= tol(dtype)


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("native", [True, False])
def test_without_memory_for_the_partials_the_launch_is_not_split(monkeypatch, native):
    """With the process's memory limited to what it holds and room for the output, a call that would
    split gives the unsplit launch's result (forge_attn_prefill, which has no workspace)."""
    from sleuth_amd import ops

    B, T, H, K, D, offset = 1, 1024, 16, 8, 128, 15360
    g = gen(970)
    q = randn(g, B, T, H, D, dtype=torch.bfloat16).transpose(1, 2).to(DEV)
    kc, vc = (randn(g, B, K, offset + T, D, dtype=torch.bfloat16).to(DEV) for _ in range(2))
    room = 24 << 20              # a 20 MB segment of the allocator for the output (4 MB)
    assert _bytes(B, T, H, K, D, offset) > room
    call = lambda: ops.attn_prefill(q, kc, vc, scale=scale_of(D), offset=offset)  # noqa: E731
    split, want = call(), torch.empty(B, T, H, D, dtype=torch.bfloat16, device=DEV)
    if not native:
        monkeypatch.setattr(ops, "host", lambda: types.SimpleNamespace(prefill=lambda *a: None))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    limit = (torch.cuda.memory_reserved() + room) / torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction(limit)
        got = call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    _lib.check(_lib.lib().forge_attn_prefill(
        _lib.BF16, B, T, H, K, D, q.data_ptr(), *q.stride()[:3], None, 1e-6, 0, None, None, 0, kc.data_ptr(),
        vc.data_ptr(), *kc.stride()[:3], offset, 0, scale_of(D), want.data_ptr(), *want.stride()[:3],
        torch.cuda.current_stream().cuda_stream), "forge_attn_prefill")
    assert torch.equal(got, want) and not torch.equal(got, split)


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("B,T,window,docs", [(5, 1900, 0, True), (6, 1400, 512, False)])
def test_rows_do_not_depend_on_the_blocks_a_cu_holds(B, T, window, docs):
    """Head dim 64 with 900 and 792 blocks (three per CU): every row as in a call of its own."""
    from sleuth_amd import ops

    H, K, D = 12, 4, 64
    g = gen(990)
    q = randn(g, B, T, H, D, dtype=torch.bfloat16).transpose(1, 2).to(DEV)
    k, v = (randn(g, B, K, T, D, dtype=torch.bfloat16).to(DEV) for _ in range(2))
    starts = torch.tensor([0] * 700 + [700] * (T - 700), dtype=torch.int32, device=DEV)[None].expand(B, T).contiguous()
    call = lambda r: ops.attn_prefill(q[r], k[r], v[r], scale=scale_of(D), window=window,  # noqa: E731
                                      doc_start=starts[r] if docs else None)
    got = call(slice(None))
    assert docs or _bytes(1, T, H, K, D, 0, window) == 0     # a row alone is not split
    for b in range(B):
        assert torch.equal(call(slice(b, b + 1)), got[b:b + 1])


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("docs", [False, True])
def test_entry_points_without_a_workspace(docs):
    """forge_attn_prefill at a shape that the call with a workspace splits, and forge_attn_prefill_docs, as a
    C caller makes them, against the oracle."""
    B, T, H, K, D, offset = 1, 200, 8, 4, 128, 0 if docs else 2500
    S = offset + T
    g = gen(1000)
    q = randn(g, B, T, H, D, dtype=torch.bfloat16).transpose(1, 2)
    k, v = (randn(g, B, K, S, D, dtype=torch.bfloat16) for _ in range(2))
    starts = torch.tensor([0] * 70 + [70] * 130, dtype=torch.int32)[None].contiguous()
    same = (starts[:, :, None] == starts[:, None, :])[:, None] if docs else None
    ref = oracle.sdpa(q.float(), k.float(), v.float(), offset, 0, scale_of(D), same_doc=same)
    dq, dk, dv, ds = (t.to(DEV) for t in (q, k, v, starts))
    out = torch.empty(B, T, H, D, dtype=torch.bfloat16, device=DEV)
    args = [_lib.BF16, B, T, H, K, D, dq.data_ptr(), *dq.stride()[:3], None, 1e-6, 0, None, None, 0, dk.data_ptr(), dv.data_ptr(),
            *dk.stride()[:3], offset, 0, scale_of(D)]
    stream = torch.cuda.current_stream().cuda_stream
    if docs:
        st = _lib.lib().forge_attn_prefill_docs(*args, ds.data_ptr(), T, out.data_ptr(), *out.stride()[:3], stream)
    else:
        assert _bytes(B, T, H, K, D, offset) > 0
        st = _lib.lib().forge_attn_prefill(*args, out.data_ptr(), *out.stride()[:3], stream)
    assert st == 0
    assert max_abs(out.cpu().transpose(1, 2), ref) <= tol(torch.bfloat16)
