"""Latent attention over portions with expanded keys and values against float64: portions from the start
and from the middle of a sequence, single tokens among them, windows, shuffled pages, head gates; and
the rule that chooses between this form and the absorbed one."""
import numpy as np
import pytest
import torch

from distributed_llm_inferencing_amd.ops import hybrid as H

F64 = torch.float64


@pytest.mark.gpu
@pytest.mark.parametrize("lens,before", [([64], [0]), ([300, 1, 255], [0, 900, 33]),
                                         ([257, 64, 7, 512], [0, 129, 0, 1000])])
@pytest.mark.parametrize("window,gated", [(1 << 30, True), (100, False)])
def test_expanded_latent_attention(gpu, lens, before, window, gated):
    check(gpu, lens, before, window, gated, [a + b for a, b in zip(lens, before)])


@pytest.mark.gpu
@pytest.mark.parametrize("lens,before", [([300, 1, 255], [0, 900, 33]), ([257, 64, 7, 512], [0, 129, 0, 1000]),
                                         ([1, 1, 700, 1], [0, 64, 3000, 5000])])
@pytest.mark.parametrize("window", [1, 64, 100, 1500])
def test_only_what_a_window_shows_is_expanded(gpu, lens, before, window):
    rows, _ = H.visible_context(np.array(lens), np.array(lens) + np.array(before), window)
    check(gpu, lens, before, window, False, rows.tolist())


def check(gpu, lens, before, window, gated, rows):
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
    cuc = torch.tensor([0] + torch.tensor(rows).cumsum(0).tolist()).int()
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
                                      dev(pos), dev(bt), block, dev(cuc), int(cuc[-1]), max(rows), min(window, max(ctx)),
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


def visible(lens, before, window):
    lens = np.array(lens, dtype=np.int64)
    return H.visible_context(lens, lens + np.array(before, dtype=np.int64), window)


@pytest.mark.parametrize("window", [1, 15, 16, 17, 100, 1024, 1 << 30])
@pytest.mark.parametrize("more", [0, 17])                   # few tiles, and more than a key split takes
def test_visible_context(window, more):
    lens, before = [1, 0, 16, 17, 100, 5, 1], [0, 7, 0, 3, 1 << 17, 95, 1023]
    lens, before = lens + [1] * more, before + [300] * more
    rows, pairs = visible(lens, before, window)
    xcd = [0] * 8
    for s, (n, b, r) in enumerate(zip(lens, before, rows)):
        seen = [(max(0, p - window + 1), p) for p in range(b, b + n)]
        assert r == (n + b - min(lo for lo, _ in seen) if seen else 0)
        for t in range(0, n, 16):
            xcd[(s * 7 + t // 16) % 8] += seen[t:t + 16][-1][1] + 1 - seen[t][0]
    assert pairs == (128 * max(xcd) if more else 16 * sum(xcd))


def test_expansion_counts_what_a_window_shows():
    def pays(lens, before, window):
        rows, pairs = visible(lens, before, window)
        return H.latent_expansion_pays(sum(lens), max(lens), int(rows.sum()), pairs, 8192)
    for before in (8000, 65024, 200000):
        # a portion of a long prompt expands a window more than itself, not the prompt anew
        rows, pairs = visible([512], [before], 1024)
        assert rows.tolist() == [1535] and pairs == visible([512], [1024], 1024)[1]
        assert pays([512], [before], 1024)
    assert not pays([64], [65024], 1024)
    rows, _ = visible([512] + [1] * 64, [65024] + [20000] * 64, 1024)
    assert rows.tolist() == [1535] + [1024] * 64
    # single tokens beside a portion: 10.1 ms absorbed, 1.2 expanded (2.8 and 0.5 at 256)
    for window in (64, 256, 1024, 1 << 30):
        assert pays([512] + [1] * 64, [2000] + [1000] * 64, window)


def test_the_pairs_are_asked_for_only_where_they_decide():
    def never():
        raise AssertionError
    assert H.latent_expansion_pays(2048, 2048, 2048, never, 8192)         # a whole prompt
    assert not H.latent_expansion_pays(33, 33, 33, never, 8192)
    assert not H.latent_expansion_pays(64, 64, 4160, lambda: 64 * 4160, 8192)
    assert H.latent_expansion_pays(512, 512, 4608, lambda: 512 * 4608, 8192)


def test_cumulative_rows_of_a_step():
    from distributed_llm_inferencing_amd.models.mixers import StepView

    def view(lens, before):
        cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32)
        lens = np.array(lens, dtype=np.int64)
        return StepView(cu, int(lens.max()), cu, cu, cu, 16, None, 1 << 30, lens, lens + np.array(before))
    whole = view([5, 0, 70], [0, 0, 0])
    assert whole.cu_visible(64) is whole.cu_seqlens and whole.cu_visible(1) is whole.cu_seqlens
    part = view([5, 70, 0], [3, 40, 9])
    assert part.cu_visible(10).tolist() == [0, 8, 87, 87] and part.cu_visible(1).tolist() == [0, 5, 75, 75]
