"""GPU parity of the workgroup splits over 16-token pages (two page lookups per
32-token step): lengths on every side of a half step, a half whose page entry is
invalid, the longest-first order, more splits than the rule's, against float64;
and against the per-lane lookup kernel (which a call with a zero mask takes).
"""
import math

import pytest
import torch

from helpers import ATOL

pytestmark = pytest.mark.gpu


def _call(lens, Hq, Hkv, D, dtype, device, bad=()):
    g = torch.Generator().manual_seed(len(lens) + D)
    pages = [-(-n // 16) for n in lens]
    perm = torch.randperm(sum(pages) + 3, generator=g).to(torch.int32)
    bt = torch.full((len(lens), max(pages) + 1), -1, dtype=torch.int32)
    o = 0
    for b, n in enumerate(pages):
        bt[b, :n] = perm[o:o + n]
        o += n
    for b, page in bad:
        bt[b, page] = -1
    n = sum(pages) + 3
    kp, vp = (torch.randn(n, Hkv, 16, D, generator=g).to(dtype).to(device) for _ in range(2))
    q = torch.randn(len(lens), Hq, 1, D, generator=g).to(dtype).to(device)
    return q, kp, vp, bt.to(device), torch.tensor(lens, dtype=torch.int32, device=device)


def _reference(q, kp, vp, bt, sl):
    B, Hq, _, D = q.shape
    Hkv = kp.shape[1]
    out = torch.zeros(B, Hq, 1, D, dtype=torch.float64, device=q.device)
    lse = torch.full((B, Hq), -math.inf, dtype=torch.float64, device=q.device)
    for b in range(B):
        n = int(sl[b])
        tok = torch.arange(n, device=q.device)
        page = bt[b].long()[tok // 16]
        ok = page >= 0
        if not ok.any():
            continue
        k = kp[page[ok], :, (tok % 16)[ok]].double().transpose(0, 1)
        v = vp[page[ok], :, (tok % 16)[ok]].double().transpose(0, 1)
        s = q[b].view(Hkv, Hq // Hkv, D).double() @ k.transpose(1, 2) / math.sqrt(D)
        out[b] = (torch.softmax(s, -1) @ v).view(Hq, 1, D)
        lse[b] = torch.logsumexp(s, -1).view(Hq)
    return out, lse


@pytest.mark.parametrize("lens,Hq,Hkv,D,dtype,bad,split", [
    ([0, 1, 15, 16, 17, 31, 32, 33], 8, 2, 128, torch.bfloat16, (), None),
    ([700, 513, 80], 8, 2, 64, torch.float16, ((0, 3), (0, 4), (1, 31)), 768),
    ([1900, 1033, 80], 8, 2, 64, torch.float16, ((0, 3), (0, 40), (1, 64)), 192),
    ([2500] + [100 * i + 7 for i in range(39)], 32, 8, 128, torch.bfloat16, ((5, 0),), None),
    ([300, 47], 40, 2, 256, torch.float16, (), 320),   # two head groups
    ([2047, 900], 4, 1, 96, torch.bfloat16, ((0, 127),), 256),
    ([7900, 60], 4, 2, 128, torch.bfloat16, (), 7936),  # the longest single split
])
def test_page16_decode(cuda, lens, Hq, Hkv, D, dtype, bad, split):
    from llm_cuda.kernels.triton.decode_attention import paged_decode_attention

    from llm_cuda.kernels import _ops

    args = _call(lens, Hq, Hkv, D, dtype, cuda, bad)
    capacity, units = args[3].shape[1] * 16, len(lens) * Hkv * -(-(Hq // Hkv) // 16)
    used = split or _ops.choose_split_tokens(len(lens), Hkv, Hq // Hkv, capacity, 16, D)
    assert _ops.takes_workgroup_splits(units, used, -(-capacity // used), 16, D, capacity)
    out, lse = paged_decode_attention(*args, return_lse=True, split_tokens=split)
    ref, ref_lse = _reference(*args)
    assert (out.double() - ref).abs().max().item() <= ATOL[dtype]
    live = torch.isfinite(ref_lse)
    assert torch.equal(torch.isfinite(lse), live)
    # an fp32 sum over at most max(lens) terms
    assert (lse.double() - ref_lse)[live].abs().max().item() <= max(lens) * 2.0 ** -24 + 1e-5
    zero = torch.zeros(len(lens), 1, 1, max(lens), device=cuda)
    lanes, llse = paged_decode_attention(*args, return_lse=True, attention_mask=zero)
    assert (out.float() - lanes.float()).abs().max().item() <= ATOL[dtype]
    assert (lse - llse)[live].abs().max().item() <= max(lens) * 2.0 ** -23 + 1e-5


@pytest.mark.parametrize("lens,columns,split,Hq,Hkv,D,dtype", [
    ([900, 1, 0, 255], 600, 320, 8, 2, 128, torch.bfloat16),      # parts of a step a wave
    ([257, 512, 2049, 4097], 2000, 2048, 16, 4, 64, torch.float16),  # one token into another part
    ([3000], 1875, 1024, 4, 1, 256, torch.bfloat16),
    ([1700, 33] * 20, 520, 2816, 8, 2, 96, torch.float16),
])
def test_page16_short_sequences_in_a_wide_table(cuda, lens, columns, split, Hq, Hkv, D,
                                                    dtype):
    """Each sequence is cut by its own length, whatever the table's capacity: as in
    a table of just its pages."""
    from llm_cuda.kernels import _ops
    from llm_cuda.kernels.triton.decode_attention import paged_decode_attention

    q, kp, vp, bt, sl = args = _call(lens, Hq, Hkv, D, dtype, cuda)
    wide = torch.full((len(lens), columns), -1, dtype=torch.int32, device=cuda)
    wide[:, :bt.shape[1]] = bt
    units, capacity = len(lens) * Hkv, columns * 16
    n = -(-capacity // split)
    assert n > 1 and units * n <= 256
    assert _ops.takes_workgroup_splits(units, split, n, 16, D, capacity)
    out, lse = paged_decode_attention(q, kp, vp, wide, sl, return_lse=True, split_tokens=split)
    ref, ref_lse = _reference(*args)
    assert (out.double() - ref).abs().max().item() <= ATOL[dtype]
    live = torch.isfinite(ref_lse)
    assert torch.equal(torch.isfinite(lse), live)
    assert (lse.double() - ref_lse)[live].abs().max().item() <= max(lens) * 2.0 ** -24 + 1e-5
