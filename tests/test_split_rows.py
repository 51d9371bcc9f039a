"""Row blocks of the split-K kernel: every block size (1 to 8 rows, equal blocks beyond) gives each row
the bits of its own single-token decode, and the oracle's values."""

from __future__ import annotations

import pytest
import torch

import oracle
from conftest import gpu_available
from helpers import gen, max_abs, randn, scale_of, tol

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]
DEV = "cuda"


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 64), (torch.float32, 32), (torch.bfloat16, 512)])
@pytest.mark.parametrize("G,T", [(1, 3), (1, 5), (3, 1), (3, 2), (1, 7), (3, 3), (2, 5), (1, 11), (2, 9), (3, 7)])
@pytest.mark.parametrize("ragged", [False, True])
def test_rows_per_block(dtype, D, G, T, ragged):
    from sleuth_amd import ops

    B, K, L, chunk = 2, 2, 700, 128 if D < 512 else 64
    g = gen(100 * G + T)
    q = randn(g, B, G * K, T, D, dtype=dtype)
    kc, vc = randn(g, B, K, L, D, dtype=dtype), randn(g, B, K, L, D, dtype=dtype)
    lens = [600, 333] if ragged else [600, 600]
    chunk = max(chunk, 256 // max(1, D // (4 if dtype == torch.float32 else 8)) * 2)
    dev = [t.to(DEV) for t in (q, kc, vc)]

    def call(t0, n):
        at = [x + t0 for x in lens]
        where = dict(row_pos=torch.tensor(at, dtype=torch.int32, device=DEV), max_kv_len=L) if ragged else dict(pos=at[0])
        return ops.attn_decode(dev[0][:, :, t0:t0 + n], *dev[1:], scale=scale_of(D), chunk=chunk, **where)
    got = call(0, T)
    for t in range(T):
        assert torch.equal(call(t, 1), got[:, t:t + 1]), t
    for b in range(B):
        S = lens[b] + T
        ref = oracle.sdpa(q[b:b + 1].float(), kc[b:b + 1, :, :S].float(), vc[b:b + 1, :, :S].float(), lens[b], 0, scale_of(D))
        assert max_abs(got[b:b + 1].cpu().transpose(1, 2), ref) <= tol(dtype)
