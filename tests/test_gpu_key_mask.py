"""GPU parity of key masks ([B, 1, 1, Skv]: staged in LDS, added to the scaled
scores) against float64 and against the same mask written out per row ([B, 1, Sq,
Skv], the row-bias kernel, whose arithmetic is the same): padding values of every
usual size, mixed ones, rows with no real key and with no key at all, odd lengths,
a cached prefix, the most keys LDS holds with the first count past it, and the
gradients of a left-padded batch.
"""
import math

import pytest
import torch

from helpers import ATOL

pytestmark = pytest.mark.gpu


def _mask(kind, B, Skv, dtype, g):
    m = torch.zeros(B, 1, 1, Skv)
    n = max(1, Skv // 3)
    if kind == "mixed":  # ordinary biases, -1e4, -1e9, the type's lowest and -inf
        m = 2.0 * torch.randn(m.shape, generator=g)
        m[..., 1::5], m[..., 2::7] = -1e4, -1e9
        m[..., 3::11], m[..., 4::13] = torch.finfo(dtype).min, -math.inf
    else:
        m[0, ..., :n] = {"min": torch.finfo(dtype).min, "1e4": -1e4, "1e9": -1e9,
                         "inf": -math.inf}[kind]
    return m.to(dtype)


def _reference(q, k, v, mask, off):
    g = q.shape[1] // k.shape[1]
    s = q.double() @ k.double().repeat_interleave(g, 1).transpose(-1, -2) / math.sqrt(q.shape[-1])
    # (masks below -1e30 act as -1e30; the scores next to them vanish as in fp32)
    s = (s + mask.double().clamp(min=-1e30)).masked_fill(mask.double() == -math.inf, -math.inf)
    Sq, Skv = s.shape[-2:]
    seen = (torch.arange(Skv, device=q.device)
            <= torch.arange(Sq, device=q.device).view(-1, 1) + off)
    s = s.masked_fill(~seen, -math.inf)
    p = torch.softmax(s, -1)
    return torch.nan_to_num(p, nan=0.0) @ v.double().repeat_interleave(g, 1)


@pytest.mark.parametrize("kind", ["min", "1e4", "1e9", "inf", "mixed"])
@pytest.mark.parametrize("Sq,Skv,D,dtype,mdt", [
    (200, 200, 128, torch.bfloat16, torch.bfloat16),
    (77, 133, 64, torch.float16, torch.float32),
    (2, 65, 128, torch.bfloat16, torch.float32),
    # one query row: expand keeps its stride, so the row-bias kernel on both sides
    (1, 65, 128, torch.bfloat16, torch.float32),
])
def test_key_mask(cuda, kind, Sq, Skv, D, dtype, mdt):
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    B, Hq, Hkv, off = 2, 8, 2, Skv - Sq
    g = torch.Generator().manual_seed(Skv)
    q, k, v = (torch.randn(s, generator=g).to(dtype).to(cuda) for s in (
        (B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)))
    mask = _mask(kind, B, Skv, mdt, g).to(cuda)
    out, lse = triton_fused_causal_attention(q, k, v, mask, return_lse=True, q_offset=off)
    rows, rlse = triton_fused_causal_attention(
        q, k, v, mask.expand(B, 1, Sq, Skv).contiguous(), return_lse=True, q_offset=off)
    assert torch.equal(out, rows) and torch.equal(lse, rlse)
    if kind != "1e9" and kind != "mixed":  # (at -1e9 the fp32 scores keep a few bits)
        assert (out.double() - _reference(q, k, v, mask, off)).abs().max().item() <= ATOL[dtype]


@pytest.mark.parametrize("form", ["batch of one", "every other", "one value", "odd start"])
def test_key_mask_forms(cuda, form):
    """Masks that broadcast or stride: one for the batch, a strided row, a single
    value for every key, rows from an odd element on; views of q, k and v."""
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    B, Hq, Hkv, S, D, dtype = 2, 8, 2, 150, 64, torch.bfloat16
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(B, S, h, D, generator=g).to(dtype).to(cuda).transpose(1, 2)
               for h in (Hq, Hkv, Hkv))
    m = torch.zeros(B, 1, 1, 2 * S + 1, dtype=dtype, device=cuda)
    m[0, ..., :80] = torch.finfo(dtype).min
    m[1, ..., ::3] = -2.5
    mask = {"batch of one": m[:1, ..., :S], "every other": m[..., :2 * S:2],
            "one value": m[1:, ..., :1], "odd start": m[..., 1:S + 1]}[form]
    out = triton_fused_causal_attention(q, k, v, mask)
    ref = _reference(q, k, v, mask.expand(B, 1, 1, S), 0)
    assert (out.double() - ref).abs().max().item() <= ATOL[dtype]


@pytest.mark.parametrize("value", ["min", -math.inf])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D", [
    (3, 8, 2, 400, 400, 128),   # 6 units: the plain unit order
    (2, 16, 8, 300, 450, 64),   # 16 units dealt over the XCDs, a cached prefix
])
def test_masked_ends_are_left_out(cuda, value, B, Hq, Hkv, Sq, Skv, D):
    """Padding of several tiles at both ends: rows before, on and after the kept
    keys, a sequence with one kept key and one with none masked."""
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    dtype, off = torch.bfloat16, Skv - Sq
    g = torch.Generator().manual_seed(Skv)
    q, k, v = (torch.randn(s, generator=g).to(dtype).to(cuda) for s in (
        (B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)))
    mask = torch.zeros(B, 1, 1, Skv)
    low = torch.finfo(dtype).min if value == "min" else value
    mask[0, ..., :197] = mask[0, ..., 330:] = low
    mask[1] = low
    mask[1, ..., 131] = 0.25
    mask = mask.to(dtype).to(cuda)
    out, lse = triton_fused_causal_attention(q, k, v, mask, return_lse=True, q_offset=off)
    assert (out.double() - _reference(q, k, v, mask, off)).abs().max().item() <= ATOL[dtype]
    rows, rlse = triton_fused_causal_attention(
        q, k, v, mask.expand(B, 1, Sq, Skv).contiguous(), return_lse=True, q_offset=off)
    assert torch.equal(out, rows) and torch.equal(lse, rlse)


@pytest.mark.parametrize("Skv", [4096, 4097])
def test_key_mask_at_the_most_keys_staged(cuda, Skv):
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    B, Hq, Hkv, Sq, D, dtype = 1, 4, 1, 40, 128, torch.bfloat16
    g = torch.Generator().manual_seed(Skv)
    q, k, v = (torch.randn(s, generator=g).to(dtype).to(cuda) for s in (
        (B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D)))
    mask = _mask("min", B, Skv, dtype, g).to(cuda)
    out = triton_fused_causal_attention(q, k, v, mask, q_offset=Skv - Sq)
    ref = _reference(q, k, v, mask, Skv - Sq)
    assert (out.double() - ref).abs().max().item() <= ATOL[dtype]


@pytest.mark.parametrize("value,D,dtype", [
    (value, D, dtype) for value in ("min", -1e9, -1e20)
    for D, dtype in ((40, torch.bfloat16), (56, torch.bfloat16), (64, torch.float16),
                     (104, torch.bfloat16), (112, torch.float16), (128, torch.bfloat16),
                     (64, torch.float32))
    if value != -1e20 or dtype != torch.float16])  # (-1e20: not a float16 value)
def test_left_padded_gradients(cuda, value, D, dtype):
    """A training step over a left-padded batch, no gradient arriving at the pad
    rows (all of whose keys are masked): the gradients are those of the prompts
    alone, zero at the pads, and those of the mask written out per row."""
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    B, Hq, Hkv, S, pads = 2, 4, 2, 150, (90, 0)
    g = torch.Generator().manual_seed(D)
    mdt = torch.float32 if dtype == torch.float16 and value == -1e9 else dtype
    low = torch.finfo(mdt).min if value == "min" else value
    q, k, v, dout = (torch.randn(s, generator=g).to(dtype).to(cuda) for s in (
        (B, Hq, S, D), (B, Hkv, S, D), (B, Hkv, S, D), (B, Hq, S, D)))
    mask = torch.zeros(B, 1, 1, S)
    for b, n in enumerate(pads):
        mask[b, ..., :n] = low
        dout[b, :, :n] = 0
    mask = mask.to(mdt).to(cuda)

    def step(m):
        ins = [t.clone().requires_grad_(True) for t in (q, k, v)]
        out, lse = triton_fused_causal_attention(*ins, m, return_lse=True)
        return (out.detach(), lse) + torch.autograd.grad(out, ins, dout)

    keys, rows = step(mask), step(mask.expand(B, 1, S, S).contiguous())
    assert all(torch.equal(a, b) for a, b in zip(keys, rows))
    for b, n in enumerate(pads):
        assert all((t[b, :, :n] == 0).all() for t in keys[2:])
        ins = [t[b:b + 1, :, n:].double().requires_grad_(True) for t in (q, k, v)]
        rep = [ins[0]] + [t.repeat_interleave(Hq // Hkv, 1) for t in ins[1:]]
        s = rep[0] @ rep[1].transpose(-1, -2) / math.sqrt(D)
        ones = torch.ones(S - n, S - n, dtype=torch.bool, device=cuda)
        out = torch.softmax(s.masked_fill(ones.triu(1), -math.inf), -1) @ rep[2]
        ref = torch.autograd.grad(out, ins, dout[b:b + 1, :, n:].double())
        for got, want in zip(keys[2:], ref):
            err = (got[b:b + 1, :, n:].double() - want).abs().max().item()
            assert err <= ATOL[dtype] * max(1.0, want.abs().max().item())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bias", [-65504.0, -1e6])
def test_scores_next_to_a_large_bias_round_once(cuda, D, bias):
    """Every key with the same large bias: the softmax is the unmasked one, from
    scores that round once at the bias's size. A step of u there is an rms error
    of u / sqrt(12) in the exponent, ln 2 times that in a weight and in the
    output's norm (1.5 of it allowed), beside 2^-11 for the weights in f16."""
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    B, Hq, Hkv, S = 1, 8, 2, 300
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(s, generator=g).half().to(cuda) for s in (
        (B, Hq, S, D), (B, Hkv, S, D), (B, Hkv, S, D)))
    mask = torch.full((B, 1, 1, S), bias, device=cuda)
    out, lse = triton_fused_causal_attention(q, k, v, mask, return_lse=True)
    rows, rlse = triton_fused_causal_attention(q, k, v, mask.expand(B, 1, S, S).contiguous(),
                                               return_lse=True)
    assert torch.equal(out, rows) and torch.equal(lse, rlse)
    ref = _reference(q, k, v, torch.zeros_like(mask), 0)
    u = 2.0 ** (math.floor(math.log2(-bias * math.log2(math.e))) - 23)
    bound = 1.5 * math.log(2) * u / math.sqrt(12) + 2.0 ** -11
    assert ((out.double() - ref).norm() / ref.norm()).item() <= bound
