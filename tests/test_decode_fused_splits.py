"""Decode attention with several KV splits fused to the QKV reduce, rotation and cache write, against the
three kernels it replaces."""
import math

import pytest
import torch

from distributed_llm_inferencing_amd import ops
from distributed_llm_inferencing_amd.ops import gemm as G
from distributed_llm_inferencing_amd.ops import reference as R

HD, BS, HKV = 128, 16, 8


# one token; a split's edge and either side; a short last split; a long
# context among short ones; a padded row (0: no slot); more sequences than one scan covers; as many as take no splits
@pytest.mark.gpu
@pytest.mark.parametrize("hq", (8, 32, 128))
@pytest.mark.parametrize("tile,splits", ((0, 1), (0, 2), (0, 4), (30, 2)))
@pytest.mark.parametrize("lens,limit", (
    ([1], 2048), ([64], 2048), ([65], 2048), ([129], 1024), ([2047, 0, 5, 33], 2048), ([4000] + [70] * 5, 4096),
    ([700, 701, 690, 720], 1024), ([(7 * i) % 190 + 1 for i in range(70)], 1024), ([(37 * i) % 901 for i in range(260)], 1024)))
def test_fused_splits_match_separate_kernels(gpu, hq, tile, splits, lens, limit):
    B, K, N = len(lens), 512, (hq + 2 * HKV) * HD
    if tile == 30 and B > G.GEMV_MAX_M:
        pytest.skip("weight stream of up to 4 rows")
    assert (ops.decode_num_splits(B, HKV, limit) > 1) == (B < 256)
    g = torch.Generator(device=gpu).manual_seed(hq + B)
    width = -(-limit // BS)
    need = [-(-n // BS) for n in lens]
    perm = torch.randperm(sum(need) + 3, device=gpu, generator=g).to(torch.int32)
    tables = torch.zeros(B, width, dtype=torch.int32, device=gpu)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = perm[at:at + n]
        at += n
    ctx = torch.tensor(lens, dtype=torch.int32, device=gpu)
    pos = (ctx - 1).clamp(min=0)
    slots = torch.where(ctx > 0, tables.gather(1, (pos // BS).long()[:, None])[:, 0] * BS + pos % BS, -1).to(torch.int32)
    kc, vc = (torch.randn(len(perm), HKV, BS, HD, device=gpu, generator=g).bfloat16() for _ in range(2))
    cs = R.rope_cos_sin(limit, HD, 10000.0, device=gpu)
    x = torch.randn(B, K, device=gpu, generator=g).bfloat16()
    w = (torch.randn(N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    kept = dict(G._plan_cache)
    try:
        plan = G.GemmPlan("dli", tile, splits)
        G.set_plan(B, N, K, "splitk", plan)
        if splits == 1:
            G.set_plan(B, N, K, "none", plan)
        k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
        qkv = ops.linear_rope_cache(x, w, pos, slots, cs, k1, v1, hq, HKV, HD)
        want = ops.decode_attention(qkv, k1, v1, tables, ctx, limit, hq, HKV, HD, 1 / math.sqrt(HD))
        got = ops.linear_rope_attention(x, w, pos, slots, cs, k2, v2, tables, ctx, limit, hq, HKV, HD,
                                        1 / math.sqrt(HD))
    finally:
        G.clear_plans()
        G._plan_cache.update(kept)
    # the rotation's products and difference may be contracted differently: a key or query element that
    # lies between two bf16 values falls to either side, one ulp (2^-7 of it at most), the rest is equal;
    # where the difference cancels, what is left is the products' rounding: 2^-23 of |a cos| + |b sin| <= 16
    assert torch.equal(v1, v2)
    apart = (k1.float() - k2.float()).abs()
    assert bool((apart <= 2.0 ** -7 * k1.float().abs() + 2.0 ** -19).all()) and int((apart > 0).sum()) <= 2 + B * HKV * HD // 1000
    # a few elements of a score's 128 move by 2^-8: the softmax's weights by less than 1 %
    live = ctx > 0
    assert float((got[live].float() - want[live].float()).norm() / want[live].float().norm()) < 2.0 ** -8
