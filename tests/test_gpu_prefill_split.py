"""GPU parity of prefill calls whose keys are split into ranges (few row groups
over many keys): against float64, and the ranges' edges against the unsplit
kernel (the C entry without a workspace)."""
import math

import pytest
import torch

from helpers import ATOL

pytestmark = pytest.mark.gpu


def _inputs(B, Hq, Hkv, Sq, Skv, D, dtype, device):
    g = torch.Generator().manual_seed(Sq + Skv)
    return tuple(torch.randn(s, generator=g).to(dtype).to(device) for s in (
        (B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)))


def _unsplit(q, k, v, off):
    """lc_prefill_attn_fwd: the entry that has no workspace and never splits."""
    from llm_cuda import _native as nat
    from llm_cuda.kernels import _ops

    B, Hq, Sq, D = q.shape
    out = torch.empty_like(q)
    lse = torch.empty(B, Hq, Sq, dtype=torch.float32, device=q.device)
    st = [_ops._i64arr(t.stride()) for t in (q, k, v, out)]
    rc = nat.load().lc_prefill_attn_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr(), B, Hq,
        k.shape[1], Sq, k.shape[2], D, *st, off, None, None, 0, None, 1.0 / math.sqrt(D),
        nat.lc_dtype(q), nat.stream_ptr(q.device))
    nat.check(rc, "lc_prefill_attn_fwd")
    return out, lse


# Sq 1 and partial row groups; keys that end inside a tile and inside a range;
# q_offset short of the keys (trailing keys unseen), so the last range is empty
# for some rows; the diagonal crossing several ranges (Sq 1500); three head groups.
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,off,D,dtype", [
    (1, 8, 2, 1, 1985, 1984, 128, torch.bfloat16),
    (1, 8, 2, 16, 4000, 3984, 64, torch.float16),
    (2, 8, 2, 33, 2111, 2078, 128, torch.bfloat16),
    (1, 8, 2, 100, 3000, 1950, 128, torch.float16),
    (1, 4, 1, 1500, 2100, 600, 128, torch.bfloat16),
    (1, 6, 2, 70, 2500, 2430, 96, torch.bfloat16),
])
def test_split_prefill(cuda, B, Hq, Hkv, Sq, Skv, off, D, dtype):
    from llm_cuda import _native as nat
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    q, k, v = _inputs(B, Hq, Hkv, Sq, Skv, D, dtype, cuda)
    assert nat.load().lc_prefill_attn_workspace_bytes(B, Hq, Hkv, Sq, Skv, D, off, 0,
                                                      nat.lc_dtype(q)) > 0
    out, lse = triton_fused_causal_attention(q, k, v, return_lse=True, q_offset=off)
    g = Hq // Hkv
    s = q.double() @ k.double().repeat_interleave(g, 1).transpose(-1, -2) / math.sqrt(D)
    seen = torch.arange(Skv, device=cuda) <= torch.arange(Sq, device=cuda).view(-1, 1) + off
    s = s.masked_fill(~seen, -math.inf)
    ref = torch.softmax(s, -1) @ v.double().repeat_interleave(g, 1)
    assert (out.double() - ref).abs().max().item() <= ATOL[dtype]
    # an fp32 sum of at most Skv terms and a few roundings of the merge
    ref_lse = torch.logsumexp(s, -1)
    assert (lse.double() - ref_lse).abs().max().item() <= Skv * 2.0 ** -24 + 1e-5
    out1, lse1 = _unsplit(q, k, v, off)
    assert (lse - lse1).abs().max().item() <= Skv * 2.0 ** -23 + 1e-5
    assert (out.float() - out1.float()).abs().max().item() <= ATOL[dtype]


def test_split_prefill_strided_views(cuda):
    """q, k and v as projection views, k and v cut from longer rows, a batch that
    shares its keys."""
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    B, Hq, Hkv, Sq, Skv, D = 2, 8, 2, 50, 2200, 64
    g = torch.Generator().manual_seed(4)
    q = torch.randn(B, Sq, Hq, D, generator=g).bfloat16().to(cuda).transpose(1, 2)
    kv = torch.randn(1, Skv, 2 * Hkv, D + 8, generator=g).bfloat16().to(cuda).transpose(1, 2)
    k, v = (t[..., 8:].expand(B, -1, -1, -1) for t in (kv[:, :Hkv], kv[:, Hkv:]))
    out, lse = triton_fused_causal_attention(q, k, v, return_lse=True, q_offset=Skv - Sq)
    ref, rlse = _unsplit(q.contiguous(), k.contiguous(), v.contiguous(), Skv - Sq)
    assert (lse - rlse).abs().max().item() <= Skv * 2.0 ** -23 + 1e-5
    assert (out.float() - ref.float()).abs().max().item() <= ATOL[torch.bfloat16]


def test_split_prefill_replays_from_a_graph(cuda):
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    q, k, v = _inputs(1, 8, 2, 40, 3000, 128, torch.bfloat16, cuda)
    run = lambda: triton_fused_causal_attention(q, k, v, return_lse=True, q_offset=2960)  # noqa: E731
    ref = run()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, ref))
        run()


# A NaN or inf in one K row of a range (seen by all rows; by the last 20 only; in
# the first and in the last tile of a range), in one element of V, in a Q row.
@pytest.mark.parametrize("where,value", [
    ("k 1000", math.nan), ("k 2980", math.nan), ("k 0", math.nan), ("k 511", math.nan),
    ("k 1000", math.inf), ("v 700", math.nan), ("q 7", math.nan), ("q 7", math.inf)])
def test_split_prefill_keeps_what_is_not_finite(cuda, where, value):
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    B, Hq, Hkv, Sq, Skv, D = 1, 8, 2, 40, 3000, 128
    q, k, v = _inputs(B, Hq, Hkv, Sq, Skv, D, torch.bfloat16, cuda)
    name, row = where.split()
    if name == "v":
        v[0, 1, int(row), 3] = value
    else:
        dict(q=q, k=k)[name][0, 1, int(row)] = value
    out, lse = triton_fused_causal_attention(q, k, v, return_lse=True, q_offset=Skv - Sq)
    ref, rlse = _unsplit(q, k, v, Skv - Sq)
    assert not ref.isfinite().all()
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(lse.isinf(), rlse.isinf())
    fine = ref.isfinite()
    assert (out.float() - ref.float())[fine].abs().max().item() <= ATOL[torch.bfloat16]
