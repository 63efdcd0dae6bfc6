"""Decode attention whose KV splits are dealt from the step's actual contexts: ragged, near-equal,
empty and very long contexts, batches of more than one register's and more than four registers' lanes,
slot counts that are no power of two and more than 64, against the fp32 reference of the same cache."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops

pytestmark = pytest.mark.gpu
HD, BS = 128, 16


def reference(q, kc, vc, tables, lens, scale):
    out = []
    for b, n in enumerate(lens):
        if n == 0:
            out.append(torch.zeros_like(q[b]))
            continue
        nb = -(-n // BS)
        k = kc[tables[b, :nb].long()].transpose(1, 2).reshape(nb * BS, -1, HD)[:n]
        v = vc[tables[b, :nb].long()].transpose(1, 2).reshape(nb * BS, -1, HD)[:n]
        g = q.shape[1] // k.shape[1]
        k, v = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
        p = torch.softmax((q[b][:, None] * k.transpose(0, 1)).sum(-1) * scale, -1)
        out.append((p[..., None] * v.transpose(0, 1)).sum(1))
    return torch.stack(out)


CASES = {
    "one long among short": [5] * 20 + [4100] + [33] * 9,
    "ragged": [int(40 * 1.16 ** i) for i in range(30)],
    "near equal": [500 + 3 * i for i in range(40)],
    "equal, whole tiles": [512] * 12,
    "empty rows": [0, 700, 0, 64, 0],
    "all empty": [0, 0, 0],
    "a token": [1],
    "70 rows": [(37 * i) % 400 + 1 for i in range(70)],
    "300 rows": [(53 * i) % 180 + 1 for i in range(300)],
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("hq,hkv", [(8, 2), (16, 1)])
@pytest.mark.parametrize("splits", [None, 2, 5, 64, 100])
def test_contexts_dealt_to_splits(name, hq, hkv, splits):
    lens = CASES[name]
    torch.manual_seed(len(lens))
    B, longest = len(lens), max(lens)
    nb = [-(-n // BS) for n in lens]
    total = sum(nb) + 1
    kc, vc = (torch.randn(total, hkv, BS, HD, device="cuda").bfloat16() for _ in range(2))
    ids, at = torch.randperm(total).int(), 0
    tables = torch.zeros(B, max(1, -(-longest // BS)), dtype=torch.int32)
    for b, n in enumerate(nb):
        tables[b, :n] = ids[at:at + n]
        at += n
    tables = tables.cuda()
    qkv = torch.randn(B, (hq + 2 * hkv) * HD, device="cuda").bfloat16()
    ctx = torch.tensor(lens, dtype=torch.int32, device="cuda")
    # a slot table may be wider than the contexts in it
    for bound in (max(1, longest), 8192):
        ops.G.workspace(qkv.device, 1 << 20).fill_(0xff)      # stale partials are NaN
        got = ops.decode_attention(qkv, kc, vc, tables, ctx, bound, hq, hkv, HD, HD ** -0.5,
                                   num_splits=splits).view(B, hq, HD).float()
        want = reference(qkv[:, :hq * HD].view(B, hq, HD).float(), kc.float(), vc.float(), tables,
                         lens, HD ** -0.5)
        # probabilities are rounded to bf16 (2^-9 relative) before the value sum, whose terms are at
        # most |v| < 6 with weights summing to 1, and the result is rounded to bf16
        assert (got - want).abs().max() <= 6 * 2 ** -9 + 2 ** -8 * want.abs().max()


@pytest.mark.parametrize("B,bound", [(24, 32768), (64, 16384), (8, 65536)])
def test_a_wide_table_does_not_change_the_split(B, bound):
    """The bound is a table's width: contexts of 100 tokens take two slots at most, whatever it is,
    and nothing is written for the others."""
    hq, hkv = 32, 8
    splits = ops.decode_num_splits(B, hkv, bound)
    assert splits > 4 and bound // splits >= 768
    kc, vc = (torch.randn(B * 7, hkv, BS, HD, device="cuda").bfloat16() for _ in range(2))
    tables = torch.zeros(B, bound // BS, dtype=torch.int32, device="cuda")
    tables[:, :7] = torch.arange(B * 7, device="cuda").view(B, 7)
    qkv = torch.randn(B, (hq + 2 * hkv) * HD, device="cuda").bfloat16()
    ctx = torch.full((B,), 100, dtype=torch.int32, device="cuda")
    used = B * hq * splits * (HD + 2) * 4
    ws = ops.G.workspace(qkv.device, used)
    ws.fill_(0xff)
    got = ops.decode_attention(qkv, kc, vc, tables, ctx, bound, hq, hkv, HD, HD ** -0.5)
    partials = ws[:B * hq * splits * HD * 4].view(torch.int32).view(B * hq, splits, HD)
    assert (partials[:, 2:] == -1).all()
    want = reference(qkv[:, :hq * HD].view(B, hq, HD).float(), kc.float(), vc.float(), tables[:, :7],
                     [100] * B, HD ** -0.5)
    assert (got.view(B, hq, HD).float() - want).abs().max() <= 6 * 2 ** -9 + 2 ** -8 * want.abs().max()


@pytest.mark.parametrize("splits", [2, 3, 5, 17, 21, 64])
def test_infinite_values_stay_infinite(splits):
    """A value that overflowed bf16 in the first or the last split: its channel is infinite and no other
    one is touched, whatever the number of splits leaves of the reduce's batches."""
    hq, hkv, n = 4, 1, 64 * splits
    kc = torch.randn(n // BS, hkv, BS, HD, device="cuda").bfloat16()
    vc = torch.randn_like(kc)
    vc[0, 0, 0, 5] = float("inf")
    vc[-1, 0, 0, 9] = float("-inf")
    tables = torch.arange(n // BS, device="cuda", dtype=torch.int32)[None]
    qkv = 0.1 * torch.randn(1, (hq + 2 * hkv) * HD, device="cuda").bfloat16()
    ctx = torch.tensor([n], dtype=torch.int32, device="cuda")
    got = ops.decode_attention(qkv, kc, vc, tables, ctx, n, hq, hkv, HD, HD ** -0.5,
                               num_splits=splits).view(hq, HD).float()
    assert (got[:, 5] == float("inf")).all() and (got[:, 9] == float("-inf")).all()
    rest = [c for c in range(HD) if c not in (5, 9)]
    assert torch.isfinite(got[:, rest]).all()
