"""GPU parity of the fp32 MFMA attention kernels, forward and backward, against
float64 autograd of a dense causal softmax: edges of the 32-row tiles and of the
four waves' round (128 rows), the smallest calls, head_dims that pad each tile
width, group sizes, cached prefixes and masks.

Bound: each output is a few chained sums of at most D + Skv fp32 terms, so its
error is within (D + Skv) 2^-23 of the largest value (rounding errors of one
sign throughout).
"""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, do, q_offset, mask):
    q, k, v = (t.detach().cpu().double().requires_grad_(True) for t in (q, k, v))
    g = q.shape[1] // k.shape[1]
    kk, vv = (t.repeat_interleave(g, dim=1) for t in (k, v))
    s = q @ kk.transpose(-1, -2) / math.sqrt(q.shape[-1])
    if mask is not None:
        s = s + mask.cpu().double()
    Sq, Skv = s.shape[-2:]
    seen = torch.arange(Skv).view(1, -1) <= torch.arange(Sq).view(-1, 1) + q_offset
    s = s.masked_fill(~seen, -math.inf)
    out = torch.softmax(s, -1) @ vv
    grads = torch.autograd.grad(out, (q, k, v), do.cpu().double())
    return (out.detach(), torch.logsumexp(s, -1).detach(), *grads)


def _inputs(B, Hq, Hkv, Sq, Skv, D, device, seed=0):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(s, generator=g).to(device) for s in (
        (B, Hq, Sq, D), (B, Hkv, Skv, D), (B, Hkv, Skv, D), (B, Hq, Sq, D)))


def _run(q, k, v, do, q_offset=0, mask=None):
    from llm_cuda.kernels.triton.attention import triton_fused_causal_attention

    q, k, v = (t.clone().requires_grad_(True) for t in (q, k, v))
    out, lse = triton_fused_causal_attention(q, k, v, mask, return_lse=True, q_offset=q_offset)
    return (out.detach(), lse, *torch.autograd.grad(out, (q, k, v), do))


def _check(got, ref, D, Skv):
    for name, x, r in zip(("out", "lse", "dq", "dk", "dv"), got, ref):
        bound = (D + Skv) * 2.0 ** -23 * max(1.0, r.abs().max().item())
        err = (x.cpu().double() - r).abs().max().item()
        assert err <= bound, f"{name}: {err:.3e} > {bound:.3e}"


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Skv,D", [
    (1, 1, 1, 1, 1, 4), (2, 4, 2, 31, 31, 20), (1, 2, 2, 32, 32, 32), (1, 4, 1, 33, 33, 36),
    (2, 3, 1, 127, 127, 64), (1, 2, 1, 128, 128, 64), (1, 6, 2, 129, 129, 100),
    (1, 2, 2, 161, 161, 128), (1, 4, 4, 5, 133, 64), (1, 2, 1, 40, 300, 128),
])
def test_f32_attention_matches_float64(cuda, B, Hq, Hkv, Sq, Skv, D):
    q, k, v, do = _inputs(B, Hq, Hkv, Sq, Skv, D, cuda, seed=Sq + D)
    _check(_run(q, k, v, do, Skv - Sq), _reference(q, k, v, do, Skv - Sq, None), D, Skv)


@pytest.mark.parametrize("D", [20, 64, 128])
def test_f32_attention_layouts(cuda, D):
    """Rows of odd strides from an odd element on (4-byte aligned only), projection
    views, a batch that shares its keys (stride 0), and a strided gradient."""
    B, Hq, Hkv, S = 2, 4, 2, 70
    g = torch.Generator().manual_seed(D)
    q = torch.randn(B, Hq, S, D + 3, generator=g).to(cuda)[..., 1:D + 1]
    k = torch.randn(1, Hkv, S, D + 5, generator=g).to(cuda)[..., 3:D + 3].expand(B, -1, -1, -1)
    v = torch.randn(B, S, Hkv, D, generator=g).to(cuda).transpose(1, 2)
    do = torch.randn(B, S, Hq, D + 1, generator=g).to(cuda)[..., 1:].transpose(1, 2)
    from llm_cuda.kernels import _ops

    out, lse = _ops.prefill_attention(q, k, v, return_lse=True)
    grads = _ops.prefill_attention_backward(q, k, v, out, lse, do)
    ref = _reference(q, k, v, do, 0, None)
    _check((out, lse, *grads), ref, D, S)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_f32_attention_with_mask(cuda, D):
    B, H, S = 2, 4, 150
    q, k, v, do = _inputs(B, H, 2, S, S, D, cuda, seed=D)
    g = torch.Generator().manual_seed(D)
    mask = torch.randn(B, 1, S, S, generator=g)
    mask[torch.rand(mask.shape, generator=g) < 0.2] = -math.inf
    mask[..., 0] = 0.0  # every row keeps a key
    _check(_run(q, k, v, do, mask=mask.to(cuda)), _reference(q, k, v, do, 0, mask), D, S)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("bad", [math.inf, math.nan])
def test_f32_masked_pairs_touch_no_nonfinite_value(cuda, D, bad):
    """A key that a query does not see, and a query that does not see a key, add
    nothing to it even where their values are infinite or NaN (such a tile sums
    its pairs in another order, so within the bound rather than bit for bit)."""
    S, at = 70, 40
    bound = (D + S) * 2.0 ** -23 * 8.0  # gradients of at most 8 here
    q, k, v, do = _inputs(1, 2, 1, S, S, D, cuda, seed=D)
    ref = _run(q[:, :, :at], k[:, :, :at], v[:, :, :at], do[:, :, :at])
    k2, v2 = k.clone(), v.clone()
    k2[:, :, at:, 1] = bad
    v2[:, :, at:, 2] = bad
    got = _run(q, k2, v2, do)
    for x, r in zip(got[:3], ref[:3]):  # rows before the bad keys: out, lse, dq
        assert (x[:, :, :at] - r).abs().max().item() <= bound
    q2, do2 = q.clone(), do.clone()
    q2[:, :, :at, 1] = bad
    do2[:, :, :at, 2] = bad
    got = _run(q2, k, v, do2)
    ref = _run(q, k, v, do)
    for x, r in zip(got[3:], ref[3:]):  # keys after the bad queries: dk, dv
        assert (x[:, :, at:] - r[:, :, at:]).abs().max().item() <= bound


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("S,Skv", [(50, 90), (33, 64), (1, 40)])
@pytest.mark.parametrize("bad", [math.inf, math.nan])
def test_f32_keys_that_no_query_sees(cuda, bad, S, Skv, masked):
    """Infinite or NaN values of keys past every query's view (the unused end of a
    buffer) in the query rows' last, partial tile: their gradients are zero, the
    others those of the visible keys alone."""
    bound = (32 + Skv) * 2.0 ** -23 * 8.0
    q, k, v, do = _inputs(1, 2, 1, S, Skv, 32, cuda, seed=S)
    mask = torch.zeros(1, 1, S, Skv, device=cuda) if masked else None
    ref = _run(q, k[:, :, :S], v[:, :, :S], do)
    k[:, :, S:] = bad
    v[:, :, S:, 3] = bad
    got = _run(q, k, v, do, mask=mask)
    for x, r in zip(got, ref):
        assert (x[:, :, :S] - r).abs().max().item() <= bound
    assert all((x[:, :, S:] == 0).all() for x in got[3:])
