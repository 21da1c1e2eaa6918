"""GPU parity of the small fp32 projections (lc_linear_f32) against float64: edges
of the 32 x 32 tiles, K remainders of the 8 waves' shares, strided rows, and the
calls the rule leaves to torch.

Bound: a sum of K fp32 products, K 2^-23 of the largest value's scale.
"""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (1, 4, 4), (2, 512, 256), (31, 36, 12), (32, 32, 64), (33, 100, 68), (128, 256, 688),
    (65, 1376, 256), (3, 8, 768), (256, 1024, 20)])
@pytest.mark.parametrize("strided", [False, True])
def test_linear_f32_matches_float64(cuda, M, N, K, strided):
    from llm_cuda.kernels import _ops

    g = torch.Generator().manual_seed(M + N + K)
    pad = 12 if strided else 0
    x = torch.randn(M, K + pad, generator=g).to(cuda)[:, :K]
    w = torch.randn(N, K + pad, generator=g).to(cuda)[:, :K]
    assert _ops.linear_f32_applies(x, w)
    y = _ops.linear_f32(x, w)
    ref = F.linear(x.double(), w.double())
    assert (y.double() - ref).abs().max().item() <= K * 2.0 ** -23 * max(1.0, ref.abs().max().item())
    assert torch.equal(_ops.linear(x.view(1, M, K) if not strided else x, w).view(M, N), y)


def test_linear_f32_leaves_other_calls_to_torch(cuda):
    from llm_cuda.kernels import _ops

    x, w = torch.randn(4, 64, device=cuda), torch.randn(32, 64, device=cuda)
    assert _ops.linear_f32_applies(x, w)
    assert not _ops.linear_f32_applies(x.bfloat16(), w.bfloat16())
    assert not _ops.linear_f32_applies(x, w.requires_grad_(True))
    w = w.detach()
    assert not _ops.linear_f32_applies(x.expand(4096, 4, 64), w)      # too many tiles
    assert not _ops.linear_f32_applies(x[:, :62], w[:, :62])          # K % 4
    assert not _ops.linear_f32_applies(x, w.t().contiguous().t())     # column-major weight
    assert not _ops.linear_f32_applies(x[:0], w)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert _ops.linear(x, w).dtype == torch.bfloat16
    lin = torch.nn.Linear(64, 32, bias=False, device=cuda).requires_grad_(False)
    lin.register_forward_hook(lambda m, i, o: o + 1)
    assert torch.equal(_ops.project(x, lin), F.linear(x, lin.weight) + 1)


@pytest.mark.parametrize("where", ["instance", "class", "backward hook"])
def test_project_calls_what_replaced_the_forward(cuda, where, monkeypatch):
    """A wrapper's own forward (offloading, adapters, quantisation) runs."""
    from llm_cuda.kernels import _ops

    x = torch.randn(4, 64, device=cuda)
    lin = torch.nn.Linear(64, 32, bias=False, device=cuda).requires_grad_(False)
    assert torch.equal(_ops.project(x, lin), _ops.linear_f32(x, lin.weight))
    if where == "backward hook":
        lin.register_full_backward_hook(lambda m, gi, go: None)
        assert not _ops._is_plain_linear(lin)
        return
    plain = F.linear(x, lin.weight)
    if where == "instance":
        own = lin.forward
        lin.forward = lambda t: own(t) + 1
    else:
        monkeypatch.setattr(torch.nn.Linear, "forward", lambda m, t: F.linear(t, m.weight) + 1)
    assert torch.equal(_ops.project(x, lin), plain + 1)


def test_linear_stays_with_torch_where_its_calls_are_followed(cuda):
    """Forward-mode tangents, FLOP counters, function modes, vmap and traces."""
    from torch.autograd import forward_ad
    from torch.utils.flop_counter import FlopCounterMode

    from llm_cuda.kernels import _ops

    x, w, t = (torch.randn(s, 64, device=cuda) for s in (4, 32, 32))
    assert _ops.linear_f32_applies(x, w)
    with forward_ad.dual_level():
        tangent = forward_ad.unpack_dual(_ops.linear(x, forward_ad.make_dual(w, t))).tangent
        assert torch.equal(tangent, F.linear(x, t))
    with FlopCounterMode(display=False) as flops:
        _ops.linear(x, w)
    assert flops.get_total_flops() == 2 * 4 * 32 * 64

    class Seen(torch.overrides.TorchFunctionMode):
        calls = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.calls.append(func)
            return func(*args, **(kwargs or {}))

    with Seen():
        _ops.linear(x, w)
    assert F.linear in Seen.calls
    xs = torch.stack((x, 2 * x))
    assert torch.allclose(torch.func.vmap(lambda u: _ops.linear(u, w))(xs), F.linear(xs, w))
    traced = torch.jit.trace(lambda u: _ops.linear(u, w), x)
    assert torch.allclose(traced(3 * x), F.linear(3 * x, w), atol=1e-4)
    assert _ops.linear_f32_applies(x, w)


def test_project_of_a_sparse_weight(cuda):
    """A pruned weight, which F.linear takes (CSR has no strides to ask for)."""
    from llm_cuda.kernels import _ops

    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(4, 64, generator=g).to(cuda), torch.randn(32, 64, generator=g).to(cuda)
    for sparse in (w.to_sparse_csr(), w.to_sparse()):
        lin = torch.nn.Linear(64, 32, bias=False, device=cuda)
        lin.weight = torch.nn.Parameter(sparse, requires_grad=False)
        assert not _ops.linear_f32_applies(x, lin.weight)
        assert torch.equal(_ops.project(x, lin), F.linear(x, sparse))
    assert not _ops.linear_f32_applies(x.to_sparse_csr(), w)
