"""Prefill attention of prompts of up to 32 tokens, on tiles of 32 keys: every packing of query heads into workgroups, rows that
end inside a wave's 16 and at its edge, outputs at any alignment and nothing written beside them."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[32] * 3, [31, 1, 17], [16, 16, 15], [1], [33, 32, 5]])     # the last on tiles of 64
@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 2), (9, 3)])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("at", [0, 8, 3])
def test_short_prompts(gpu, lens, hq, hkv, hd, at):
    g = torch.Generator(device=gpu).manual_seed(sum(lens) + hd)
    T, wide = sum(lens), (hq + 2 * hkv) * hd
    held = torch.randn(T + 64, wide, device=gpu, generator=g).bfloat16()
    held[T:] = float("nan")                                 # behind the last row
    qkv = held[:T]
    cu = torch.tensor([0, *lens]).cumsum(0).to(gpu, torch.int32)
    out = torch.full((T + 32, hq * hd + at), 7.0, device=gpu).bfloat16()
    ops.prefill_attention(qkv, cu, max(lens), hq, hkv, hd, hd ** -0.5, out=out[:T, at:])
    assert torch.all(out[T:] == 7) and torch.all(out[:, :at] == 7)
    for a, n in zip(cu.tolist(), lens):
        q, k, v = (t.double().view(n, -1, hd) for t in qkv[a:a + n].split([hq * hd, hkv * hd, hkv * hd], 1))
        k, v = (t.repeat_interleave(hq // hkv, 1) for t in (k, v))
        s = (q.permute(1, 0, 2) @ k.permute(1, 2, 0).contiguous()) * hd ** -0.5
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=gpu).triu(1), float("-inf")).softmax(-1)
        want = (s @ v.permute(1, 0, 2).contiguous()).permute(1, 0, 2).reshape(n, -1)
        # weights and outputs rounded to bf16, half an ulp (2^-9) each
        assert float((out[a:a + n, at:].double() - want).norm() / want.norm()) < 2 * 2.0 ** -9
