"""Latent attention over portions with expanded keys and values against float64: portions from the start
and from the middle of a sequence, single tokens among them, windows, shuffled pages, head gates; and
the rule that chooses between this form and the absorbed one."""
import pytest
import torch

from distributed_llm_inferencing_amd.ops import hybrid as H

F64 = torch.float64


@pytest.mark.gpu
@pytest.mark.parametrize("lens,before", [([64], [0]), ([300, 1, 255], [0, 900, 33]),
                                         ([257, 64, 7, 512], [0, 129, 0, 1000])])
@pytest.mark.parametrize("window,gated", [(1 << 30, True), (100, False)])
def test_expanded_latent_attention(gpu, lens, before, window, gated):
    heads, d, dr, dv, r, block = 3, 128, 64, 128, 192, 16
    scale, g = (d + dr) ** -0.5, torch.Generator().manual_seed(sum(lens) + window % 7)
    T, ctx = sum(lens), [a + b for a, b in zip(lens, before)]
    need = [-(-c // block) for c in ctx]
    perm, bt, o = torch.randperm(sum(need) + 2, generator=g).int(), torch.zeros(len(lens), max(need)).int(), 0
    for s, n in enumerate(need):
        bt[s, :n] = perm[o:o + n]
        o += n
    cache = torch.randn(len(perm) * block, r + dr, generator=g).bfloat16()
    q = torch.randn(T, heads, d, generator=g).bfloat16()
    qf = torch.randn(T, heads, r + dr, generator=g).bfloat16()
    w = (torch.randn(heads * (d + dv), r, generator=g) * r ** -0.5).bfloat16()
    gates = torch.randn(T, heads + 2, generator=g)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist()).int()
    cuc = torch.tensor([0] + torch.tensor(ctx).cumsum(0).tolist()).int()
    pos = torch.cat([torch.arange(n) + b for n, b in zip(lens, before)]).int()
    want = torch.zeros(T, heads, dv, dtype=F64)
    for s, n in enumerate(lens):
        j = torch.arange(ctx[s])
        row = cache[bt[s].long()[j // block] * block + j % block].to(F64)
        kv = row[:, :r] @ w.to(F64).t()
        k = torch.cat([kv[:, :heads * d].view(-1, heads, d), row[:, None, r:].expand(-1, heads, -1)], 2)
        v = kv[:, heads * d:].view(-1, heads, dv)
        t = slice(int(cu[s]), int(cu[s + 1]))
        qq = torch.cat([q[t], qf[t][:, :, r:]], 2).to(F64)
        sc = torch.einsum("thd,jhd->htj", qq, k) * scale
        far = pos[t].long()[:, None] - j[None]
        p = sc.masked_fill(((far < 0) | (far >= window))[None], float("-inf")).softmax(-1)
        want[t] = torch.einsum("htj,jhd->thd", p, v)
    if gated:
        want = want * torch.sigmoid(gates[:, 1:1 + heads].to(F64))[:, :, None]
    dev = lambda x: x.to(gpu)  # noqa: E731
    got = H.expanded_latent_attention(dev(q), dev(qf)[:, :, r:], dev(cache), dev(w), heads, r, dev(cu), max(lens),
                                      dev(pos), dev(bt), block, dev(cuc), int(cuc[-1]), max(ctx), min(window, max(ctx)),
                                      scale, dev(gates)[:, 1:1 + heads] if gated else None)
    got = got.view(T, heads, dv).to(F64).cpu()
    assert torch.isfinite(got).all()
    # expanded keys (a score's error grows with its size: logits of about 1.2 here) and values, weights
    # and outputs rounded to bf16, half an ulp (2^-9) each
    assert float((got - want).norm() / want.norm()) < 4 * 2.0 ** -9


def test_expansion_rule():
    def pays(lens, before, width=8192):
        ctx = [a + b for a, b in zip(lens, before)]
        pairs = sum(-(-n // 16) * 16 * c - n * (n - 1) // 2 for n, c in zip(lens, ctx))
        return H.latent_expansion_pays(sum(lens), max(lens), sum(ctx), pairs, width)
    assert pays([2048] * 4, [0] * 4) and pays([64] * 32, [0] * 32)       # whole prompts
    assert pays([512], [4096])                                           # a portion of a long one
    assert pays([512] + [1] * 64, [2048] + [1000] * 64)                  # ... beside decode rows
    assert not pays([1] * 64, [1000] * 64)                               # decode rows
    assert not pays([37] + [1] * 64, [0] + [1000] * 64)                  # a short prompt beside them
    assert not pays([64], [4096])
    assert not pays([4096] * 64, [0] * 64)                               # an expansion of over 2 GiB
