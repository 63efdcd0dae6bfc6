"""Prefill attention of up to a workgroup a CU, whose waves take 32 rows of a half block and 32 of its counterpart from the
sequence's end: equal to the bit to the kernel of 32 rows a wave, at the edges of waves, half blocks and key tiles, of
the windows in which block ids are held (15 tiles of 64 keys), and in whatever lies behind keys and rows."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops

HD = 128


def taken(lens, hq, row_stride, block=0):
    from distributed_llm_inferencing_amd.ops import _native
    return bool(_native.require_native().dli_prefill_pairs_wave64(len(lens), max(lens), hq, HD, row_stride, block))


def other(call):
    old = ops.prefill_wave64_min_len(1 << 30)
    try:
        return call()
    finally:
        ops.prefill_wave64_min_len(old)


def cumulated(lens, gpu):
    return torch.tensor([0, *lens]).cumsum(0).to(gpu, torch.int32)


# an odd and an even number of half blocks, one row in the last wave, half block and block; beside the longest, one half block,
# two and three
LENS = [[600], [700, 300, 1, 64], [640, 383, 384], [641, 32, 33, 129], [768, 257], [769, 512], [700, 256, 255], [1025], [2048]]


@pytest.mark.gpu
@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("hq,hkv,wide", [(32, 8, 0), (8, 8, 8), (5, 1, 0), (4, 2, 64)])
def test_rows_of_the_activation(gpu, lens, hq, hkv, wide):
    if -(-max(lens) // 256) * hq * len(lens) > 256:
        lens = lens[:1]
    g = torch.Generator(device=gpu).manual_seed(sum(lens))
    held = torch.randn(sum(lens) + 256, (hq + 2 * hkv) * HD + wide, device=gpu, generator=g).bfloat16()
    held[sum(lens):] = float("nan")                         # behind the last row
    qkv = held[:sum(lens)]
    assert taken(lens, hq, qkv.stride(0))
    # output rows that are 8-byte aligned
    outs = [torch.full((sum(lens) + 64, hq * HD + 4), 7.0, device=gpu).bfloat16() for _ in range(2)]
    call = lambda out: ops.prefill_attention(qkv, cumulated(lens, gpu), max(lens), hq, hkv, HD, HD ** -0.5,  # noqa: E731
                                             out=out[:sum(lens), 4:])
    call(outs[0])
    other(lambda: call(outs[1]))
    assert torch.equal(outs[0], outs[1]) and torch.isfinite(outs[0].float()).all()
    assert torch.all(outs[0][sum(lens):] == 7) and torch.all(outs[0][:, :4] == 7)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,before", [
    ([257], [0]), ([300, 1, 64], [0, 895, 896]), ([383, 384], [577, 576]), ([513, 32], [447, 3000]), ([512, 40], [512, 1921]),
    ([700, 256, 5], [0, 704, 2047]), ([2048], [0]), ([2048], [897])])
@pytest.mark.parametrize("block", [16, 64, 256, 8, 24])     # the last two are the other kernel's
@pytest.mark.parametrize("hq,hkv", [(32, 8), (4, 4)])
def test_blocks_of_the_cache(gpu, lens, before, block, hq, hkv):
    if -(-max(lens) // 256) * hq * len(lens) > 256:
        lens, before = lens[:2], before[:2]
    g = torch.Generator(device=gpu).manual_seed(sum(lens) + block)
    ctx = [a + b for a, b in zip(lens, before)]
    need = [-(-c // block) for c in ctx]
    caches = torch.full((2, sum(need) + 1, hkv, block, HD), float("nan"), device=gpu).bfloat16()
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(1)).tolist()
    table = torch.full((len(lens), max(need)), sum(need), dtype=torch.int32)
    for i, c in enumerate(ctx):
        for b in range(need[i]):
            table[i, b] = order.pop()
            n = min(block, c - b * block)
            caches[:, table[i, b], :, :n] = torch.randn(2, hkv, n, HD, device=gpu, generator=g).bfloat16()
    qkv = torch.randn(sum(lens), (hq + 2 * hkv) * HD, device=gpu, generator=g).bfloat16()
    assert taken(lens, hq, qkv.stride(0), block) == (block in (16, 64, 256))
    call = lambda x: ops.prefill_attention_paged(x, cumulated(lens, gpu), max(lens),  # noqa: E731
                                                 torch.tensor(ctx, device=gpu, dtype=torch.int32), table.to(gpu), caches[0],
                                                 caches[1], hq, hkv, HD, HD ** -0.5)
    new = call(qkv)
    assert torch.equal(new, other(lambda: call(qkv))) and torch.isfinite(new.float()).all()
    for at in (4, 2, 1):                                    # rows of whole dwords, and of none: the other kernel's too
        odd = torch.zeros(sum(lens), qkv.shape[1] + at, device=gpu).bfloat16()[:, at:]
        odd.copy_(qkv)
        assert taken(lens, hq, odd.stride(0), block) == (block in (16, 64, 256) and at > 1)
        assert torch.equal(new, call(odd))


# scores whose maximum rises by more than the threshold in tile after tile, falls, and is equal, on both blocks of rows
@pytest.mark.gpu
def test_rising_scores(gpu):
    hq = hkv = 4
    n = 1000
    qkv = torch.zeros(n, 3 * hq * HD, device=gpu)
    at = torch.arange(n, device=gpu).float()
    qkv[:, :hq * HD:HD] = 1.0
    for h, k in enumerate((at * 0.5, -at * 0.5, torch.sin(at) * 40, torch.zeros_like(at))):
        qkv[:, hq * HD + h * HD] = k
    qkv[:, 2 * hq * HD:] = torch.randn(n, hq * HD, device=gpu, generator=torch.Generator(device=gpu).manual_seed(5))
    qkv = qkv.bfloat16()
    call = lambda: ops.prefill_attention(qkv, cumulated([n], gpu), n, hq, hkv, HD, 1.0)  # noqa: E731
    new = call()
    assert taken([n], hq, qkv.stride(0)) and torch.equal(new, other(call)) and torch.isfinite(new.float()).all()


@pytest.mark.parametrize("lens,hq,block,expected", [
    ([257], 32, 16, True), ([256], 32, 16, False), ([600], 32, 0, True), ([599], 32, 0, False), ([2048], 32, 16, True), ([2049], 32, 16, False), ([2048], 32, 0, True),
    ([512] * 4, 32, 32, True), ([512] * 5, 32, 32, False), ([2048], 32, 8, False), ([2048], 32, 24, False)])
def test_choice(lens, hq, block, expected):
    assert taken(lens, hq, (hq + 16) * HD, block) == expected


# in the cache's launches rows of whole dwords, however they are aligned; in the activation's, whatever keys and values are read by
@pytest.mark.parametrize("more,paged", [(0, True), (4, True), (2, True), (1, False)])
def test_alignment(more, paged):
    assert taken([300], 32, 48 * HD + more, 16) == paged and taken([600], 32, 48 * HD + more, 0)


# rows so far apart that 32 of them, a wave's queries, leave the kernel's 32-bit offsets are the other kernel's
@pytest.mark.parametrize("block", [0, 16])
def test_rows_far_apart(block):
    from distributed_llm_inferencing_amd.ops import _native
    lib = _native.require_native()
    assert taken([600], 4, 1 << 20, block) and not taken([600], 4, 1 << 25, block)
    assert lib.dli_prefill_takes_wave64(4100, 1, 4100, 32, HD, 1 << 17, block)
    assert not lib.dli_prefill_takes_wave64(4100, 1, 4100, 32, HD, 1 << 25, block)
