"""The portions' form of attention with mixed heads (32 heads of 128 channels): against the fp32
reference over a paged cache, at lengths around its 16-query and 32-key tiles, windows shorter and
longer than the context, portions that start inside a context, every number of key heads it takes, with
and without slopes, gate (per channel and per head) and output scale."""
import pytest
import torch

from distributed_llm_inferencing_amd.ops import hybrid as H
from distributed_llm_inferencing_amd.ops import reference as R

pytestmark = pytest.mark.gpu
HEADS, D, BS = 32, 128, 16


@pytest.mark.parametrize("G,window,slopes,gate,scale_out", [
    (8, 1 << 12, True, "channel", 1.0),          # (past 4081: one value tile a wave)
    (8, 100, True, "channel", 1.0), (8, 33, False, None, 0.7),
    (4, 70, True, "head", 1.0), (1, 1000, True, None, 1.0), (2, 16, False, "channel", 1.0)])
@pytest.mark.parametrize("parts", [
    # (tokens before the portion, tokens of the portion); query tiles are counted by the longest
    [(0, 1025)], [(0, 17), (5, 1), (31, 33), (400, 700), (0, 300)], [(47, 1), (1, 1040)],
    [(31 * i, 1) for i in range(20)]])
def test_matches_reference(G, window, slopes, gate, scale_out, parts):
    g = torch.Generator().manual_seed(window + len(parts))
    ctx = [a + b for a, b in parts]
    T = sum(b for _, b in parts)
    nb = [-(-n // BS) for n in ctx]
    slots = (sum(nb) + 1) * BS
    kc, vc = (torch.randn(slots, G * D, generator=g).bfloat16() for _ in range(2))
    ids, at = torch.randperm(sum(nb) + 1, generator=g).int(), 0
    tables = torch.zeros(len(parts), max(nb), dtype=torch.int32)
    for s, n in enumerate(nb):
        tables[s, :n] = ids[at:at + n]
        at += n
    q = torch.randn(T, HEADS * D, generator=g).bfloat16()
    pos = torch.cat([torch.arange(a, a + b) for a, b in parts]).int()
    cu = torch.tensor([0] + [b for _, b in parts]).cumsum(0).int()
    talk = (torch.eye(HEADS) + 0.2 * torch.randn(HEADS, HEADS, generator=g)).bfloat16().float()
    sl = torch.pow(2.0, -8.0 * torch.arange(1, HEADS + 1) / HEADS) if slopes else None
    width = {"channel": HEADS * D, "head": HEADS, None: 0}[gate]
    gt = torch.randn(T, width + 3, generator=g)[:, :width] if gate else None
    args = dict(slopes=sl, talk=talk, gate=gt, head_gate=gate == "head", out_scale=scale_out)
    want = R.window_attention(q.float(), kc.float(), vc.float(), D, D, HEADS, G, cu, pos, tables, BS,
                              window, D ** -0.5, out_dtype=torch.float32, **args)
    dev = {n: v.cuda() if torch.is_tensor(v) else v for n, v in args.items()}
    got = H.window_attention(q.cuda(), kc.cuda(), vc.cuda(), D, D, HEADS, G, cu.cuda(),
                             max(b for _, b in parts), pos.cuda(), tables.cuda(), BS, window,
                             D ** -0.5, **dev).float().cpu()
    # a head's weights sum to 1 and are rounded to bf16, as the mixed ones are: 2^-8 of
    # sum_g |talk_hg| max|v| at the most, and the result's own rounding
    bound = 2 ** -8 * float(talk.abs().sum(1).max()) * float(vc.float().abs().max()) * scale_out
    assert (got - want).abs().max() <= bound + 2 ** -8 * float(want.abs().max())
    assert float((got - want).norm() / want.norm()) < 2 ** -7
