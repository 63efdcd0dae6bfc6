"""Prefill attention where a launch has few workgroups: each wave's rows are other ones than in a
full launch, their sums the same."""
import math

import pytest
import torch

from distributed_llm_inferencing_amd import ops

HD, BS = 128, 16


def _case(gpu, n, ctx, hq, hkv):
    g = torch.Generator(device=gpu).manual_seed(n + ctx)
    r = lambda *s: torch.randn(*s, device=gpu, generator=g).bfloat16()  # noqa: E731
    nb = -(-ctx // BS)
    kc, vc = r(nb, hkv, BS, HD), r(nb, hkv, BS, HD)
    bt = torch.randperm(nb, device=gpu, generator=g).int().view(1, nb)
    return r(n, (hq + 2 * hkv) * HD), kc, vc, bt


def _paged(q, kc, vc, bt, n, ctx, hq, hkv, seqs):
    cu = torch.arange(seqs + 1, device=q.device, dtype=torch.int32) * n
    cl = torch.full((seqs,), ctx, device=q.device, dtype=torch.int32)
    return ops.prefill_attention_paged(q.repeat(seqs, 1), cu, n, cl, bt.repeat(seqs, 1).contiguous(), kc, vc, hq,
                                       hkv, HD, 1 / math.sqrt(HD))


# half blocks of 128 rows: an odd and an even number, one row in the last; up to 4 heads (another
# grid); alone (paired) and as often as fills the chip (not paired): the same bits in every copy
@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv", [(32, 8), (4, 2)])
@pytest.mark.parametrize("n", [256, 257, 384, 385, 640, 1000, 2048])
def test_paired_row_blocks(gpu, n, hq, hkv):
    blocks = -(-n // 256)
    seqs = 256 // (blocks * hq) + 1
    old = ops.prefill_long_min_len(1)
    try:
        q = _case(gpu, n, n, hq, hkv)[0]
        one = torch.tensor([0, n], device=gpu, dtype=torch.int32)
        many = torch.arange(seqs + 1, device=gpu, dtype=torch.int32) * n
        a = ops.prefill_attention(q, one, n, hq, hkv, HD, 1 / math.sqrt(HD))
        b = ops.prefill_attention(q.repeat(seqs, 1), many, n, hq, hkv, HD, 1 / math.sqrt(HD))
        assert torch.equal(b.view(seqs, n, -1), a.expand(seqs, -1, -1))
        x = (*_case(gpu, n, n + 333, hq, hkv), n, n + 333, hq, hkv)
        assert torch.equal(_paged(*x, seqs).view(seqs, n, -1), _paged(*x, 1).expand(seqs, -1, -1))
    finally:
        ops.prefill_long_min_len(old)
