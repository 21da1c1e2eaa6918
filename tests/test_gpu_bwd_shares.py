"""GPU parity of the backward whose dK/dV key blocks are dealt out in shares:
against the whole-block grid (the C entry with no workspace past the row arrays)
and the oracle. Shapes: shares of odd and single tiles, a group of one and of
three heads, blocks without any query, a cached prefix, head_dims that pad.
"""
import math

import pytest
import torch

from helpers import ATOL
from oracle.attention import causal_attention_backward

pytestmark = pytest.mark.gpu


def _whole_blocks(q, k, v, out, lse, do, off):
    from llm_cuda import _native as nat
    from llm_cuda.kernels import _ops

    B, Hq, Sq, D = q.shape
    Hkv, Skv = k.shape[1], k.shape[2]
    lib = nat.load()
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    ws = torch.empty(lib.lc_prefill_attn_bwd_workspace_bytes(B, Hq, Sq), dtype=torch.uint8,
                     device=q.device)
    st = [_ops._i64arr(t.stride()) for t in (q, k, v, out, do, dq, dk, dv)]
    rc = lib.lc_prefill_attn_bwd(
        *(t.data_ptr() for t in (q, k, v, out, lse, do, dq, dk, dv)), B, Hq, Hkv, Sq, Skv, D, *st,
        off, None, None, 0, 1.0 / math.sqrt(D), ws.data_ptr(), ws.numel(), nat.lc_dtype(q),
        nat.stream_ptr(q.device))
    nat.check(rc, "lc_prefill_attn_bwd")
    return dq, dk, dv


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,off,D,dtype", [
    (1, 4, 1, 700, 700, 0, 128, torch.bfloat16),
    (1, 3, 1, 450, 450, 0, 64, torch.float16),
    (1, 3, 3, 1000, 1000, 0, 96, torch.bfloat16),
    (2, 8, 2, 333, 600, 267, 128, torch.float16),
    (1, 8, 2, 260, 700, 100, 128, torch.bfloat16),  # keys past 360 are never seen
])
def test_dkv_shares(cuda, B, Hq, Hkv, Sq, Skv, off, D, dtype):
    from llm_cuda import _native as nat
    from llm_cuda.kernels import _ops

    g = torch.Generator().manual_seed(Sq + D)
    q, k, v, do = (torch.randn(s, generator=g).to(dtype).to(cuda) for s in (
        (B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D), (B, Hq, Sq, D)))
    assert nat.load().lc_prefill_attn_bwd_split_bytes(B, Hq, Hkv, Sq, Skv, D, off, 0,
                                                      nat.lc_dtype(q)) > 0
    out, lse = _ops.prefill_attention(q, k, v, q_offset=off, return_lse=True)
    got = _ops.prefill_attention_backward(q, k, v, out, lse, do, q_offset=off)
    whole = _whole_blocks(q, k, v, out, lse, do, off)
    ref = causal_attention_backward(q.cpu(), k.cpu(), v.cpu(), do.cpu(), q_offset=off)
    assert torch.equal(got[0], whole[0])
    for name, x, w, r in zip(("dq", "dk", "dv"), got, whole, ref):
        bound = ATOL[dtype] * max(1.0, r.abs().max().item())
        assert (x.float().cpu() - r.float()).abs().max().item() <= bound, name
        # the same products in fp32, added in another order, then one rounding
        ulp = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
        assert ((x.float() - w.float()).abs()
                <= ulp * w.float().abs() + 1e-4 * w.float().abs().max()).all(), name
