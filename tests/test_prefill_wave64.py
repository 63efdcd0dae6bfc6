"""Prefill attention with 64 query rows a wave against the kernel of 32 rows a wave, whose sums it repeats in the same
order: equal to the bit, at the edges of its waves, tiles and workgroups, and in whatever a cache holds past a context."""
import math

import pytest
import torch

from distributed_llm_inferencing_amd import ops

HD = 128
# enough sequences for more than 256 workgroups
EDGES = [1, 2, 63, 64, 65, 127, 128, 129, 191, 193, 255, 256, 257, 300, 449, 511, 512, 513, 700]


@pytest.fixture
def both(gpu):
    """A call on either kernel: (64 rows a wave, 32 rows a wave). The launcher's own rule says that they are; where not
    even the first is (taken False), both are calls of the latter."""
    from distributed_llm_inferencing_amd.ops import _native
    lib = _native.require_native()

    def run(call, lens, hq, qkv, block=0, taken=True):
        takes = lambda: bool(lib.dli_prefill_takes_wave64(sum(lens), len(lens), max(lens), hq, HD, qkv.stride(0), block))
        assert len(qkv) == sum(lens)
        old = ops.prefill_wave64_min_len(1), ops.prefill_long_min_len(1)
        try:
            assert takes() == taken
            new = call()
            ops.prefill_wave64_min_len(1 << 30)
            assert not takes()
            return new, call()
        finally:
            ops.prefill_wave64_min_len(old[0])
            ops.prefill_long_min_len(old[1])
    return run


def cumulated(lens, gpu):
    return torch.tensor([0, *lens]).cumsum(0).to(gpu, torch.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,times,wide", [(32, 8, 1, 0), (8, 8, 2, 0), (5, 1, 3, 64), (4, 2, 4, 0), (1, 1, 14, 8)])
def test_rows_of_the_activation(gpu, both, hq, hkv, times, wide):
    g = torch.Generator(device=gpu).manual_seed(hq)
    lens = EDGES * times
    qkv = torch.randn(sum(lens), (hq + 2 * hkv) * HD + wide, device=gpu, generator=g).bfloat16()
    cu = cumulated(lens, gpu)
    new, old = both(lambda: ops.prefill_attention(qkv, cu, max(lens), hq, hkv, HD, HD ** -0.5), lens, hq, qkv)
    assert torch.equal(new, old)
    # the last sequence against 64 bits: bf16 queries, keys, values and weights, half an ulp (2^-9) each
    n = lens[-1]
    q, k, v = (t.double().view(n, -1, HD) for t in qkv[-n:, :(hq + 2 * hkv) * HD].split([hq * HD, hkv * HD, hkv * HD], 1))
    k, v = (t.repeat_interleave(hq // hkv, 1) for t in (k, v))
    s = torch.einsum("qhd,khd->hqk", q, k) / math.sqrt(HD)
    s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=gpu).triu(1), -math.inf).softmax(-1)
    want = torch.einsum("hqk,khd->qhd", s, v).reshape(n, -1)
    assert float((new[-n:].double() - want).norm() / want.norm()) < 2.0 ** -8


# what lies behind a sequence, in the next one or past the last: a weight of zero would not keep a NaN or an infinity out
@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 4)])
def test_rows_behind_a_sequence(gpu, both, hq, hkv):
    lens = [n for edge in EDGES for n in (edge, 70)] + [449, 70, 300]
    ends = torch.tensor([0, *lens]).cumsum(0).tolist()
    held = torch.randn(ends[-1] + 256, (hq + 2 * hkv) * HD, device=gpu, generator=torch.Generator(device=gpu).manual_seed(hq)).bfloat16()
    qkv = held[:ends[-1]]
    call = lambda: ops.prefill_attention(qkv, cumulated(lens, gpu), max(lens), hq, hkv, HD, HD ** -0.5)
    clean = both(call, lens, hq, qkv)
    for i, (a, b) in enumerate(zip(ends[1::2], [*ends[2::2], len(held)])):
        held[a:b, hq * HD:] = (float("nan"), float("inf"), -float("inf"))[i % 3]
    for got, want in zip(both(call, lens, hq, qkv), clean):
        for a, b in zip(ends[0::2], ends[1::2]):
            assert torch.equal(got[a:b], want[a:b]) and torch.isfinite(got[a:b].float()).all(), (a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("block", [16, 64, 8, 48])          # the last two are the other kernel's
def test_blocks_of_the_cache(gpu, both, block):
    g = torch.Generator(device=gpu).manual_seed(block)
    hq, hkv = 8, 2
    lens = EDGES
    before = [(0, 1, 15, 16, 17, 63, 64, 100, 333)[i % 9] for i in range(len(lens))]
    ctx = [a + b for a, b in zip(lens, before)]
    blocks = [-(-c // block) for c in ctx]
    caches = torch.full((2, sum(blocks) + 1, hkv, block, HD), float("nan"), device=gpu).bfloat16()
    order = torch.randperm(sum(blocks), generator=torch.Generator().manual_seed(1)).tolist()
    table = torch.zeros(len(lens), max(blocks) + 1, dtype=torch.int32)
    for i, c in enumerate(ctx):
        for b in range(blocks[i]):
            table[i, b] = order.pop()
            n = min(block, c - b * block)
            caches[:, table[i, b], :, :n] = torch.randn(2, hkv, n, HD, device=gpu, generator=g).bfloat16()
    qkv = torch.randn(sum(lens), (hq + 2 * hkv) * HD, device=gpu, generator=g).bfloat16()
    new, old = both(lambda: ops.prefill_attention_paged(
        qkv, cumulated(lens, gpu), max(lens), torch.tensor(ctx, device=gpu, dtype=torch.int32), table.to(gpu), caches[0], caches[1],
        hq, hkv, HD, HD ** -0.5), lens, hq, qkv, block, taken=block in (16, 64))
    assert torch.equal(new, old) and torch.isfinite(new.float()).all()


# a running maximum that rises by more than the threshold in tile after tile, falls, and scores of equal size
@pytest.mark.gpu
def test_rising_scores(gpu, both):
    hq = hkv = 4
    lens = [513] * 30
    qkv = torch.zeros(sum(lens), 3 * hq * HD, device=gpu)
    at = torch.cat([torch.arange(n) for n in lens]).to(gpu).float()
    qkv[:, :hq * HD:HD] = 1.0                               # one dimension of the queries; keys by position
    for h, k in enumerate((at * 0.5, -at * 0.5, torch.sin(at) * 40, torch.zeros_like(at))):
        qkv[:, hq * HD + h * HD] = k
    qkv[:, 2 * hq * HD:] = torch.randn(sum(lens), hq * HD, device=gpu, generator=torch.Generator(device=gpu).manual_seed(5))
    qkv = qkv.bfloat16()
    new, old = both(lambda: ops.prefill_attention(qkv, cumulated(lens, gpu), 513, hq, hkv, HD, 1.0), lens, hq, qkv)
    assert torch.equal(new, old) and torch.isfinite(new.float()).all()


# which launches take it: by the longest sequence and by what stands beside it (measured on both kernels, us)
@pytest.mark.parametrize("lens,hq,paged,taken", [
    ([2500], 32, False, True), ([2048], 32, False, False), ([2047] * 8, 32, False, False), ([2048] * 7, 32, False, True),
    ([2100] + [353, 489, 330, 341, 433, 294, 207], 32, False, False),       # 76 / 80
    ([2048] + [40] * 60, 32, False, False), ([2048] + [40] * 60, 8, False, False),      # 178 / 210
    ([4096] + [300] * 7, 32, False, True), ([2100, 300], 32, False, True),              # 179 / 171, 62 / 57
    ([2100] + [300] * 7, 8, False, True), ([2100] + [300] * 7, 64, False, False),       # 59 / 54, 136 / 145
    ([8192] + [300] * 31, 32, False, True),
    ([4096], 32, True, True), ([2048] * 4, 32, True, True), ([2048, 300], 32, True, True),
    ([2048, 40], 32, True, False), ([2048] + [300] * 7, 32, True, False)])              # 217 / 263
def test_choice_by_the_mix_of_lengths(lens, hq, paged, taken):
    from distributed_llm_inferencing_amd.ops import _native
    takes = _native.require_native().dli_prefill_takes_wave64
    assert takes(sum(lens), len(lens), max(lens), hq, HD, (hq + 16) * HD, 16 if paged else 0) == taken
    assert not takes(sum(lens), len(lens), max(lens), hq, 64, (hq + 16) * 64, 16 if paged else 0)
    assert not paged or not takes(sum(lens), len(lens), max(lens), hq, HD, 0, 48)
    try:
        assert ops.prefill_wave64_min_len(1) == 2048
        assert takes(sum(lens), len(lens), max(lens), hq, HD, (hq + 16) * HD, 16 if paged else 0) == (lens != [2048])
    finally:
        ops.prefill_wave64_min_len(2048)
