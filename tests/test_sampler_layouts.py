"""The sampler's pick depends on a row's values, not on where they lie: rows of distinct logits in
random order, in descending order and with the largest ones in a single thread's columns (which the
selection by per-thread lists cannot take, so the radix select runs) give the same sampled values."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [7, 64, 300, 1000, 4097, 32000, 128256])
@pytest.mark.parametrize("B", [3, 12])
def test_same_values_in_any_layout(V, B, dtype):
    g = torch.Generator().manual_seed(V + B)
    n = min(V, 1 << 12)                          # distinct in either type, ties only at the bottom
    top = torch.arange(0x3f80 + n, 0x3f80, -1, dtype=torch.int32)
    vals = (top << 16).view(torch.float32).log2() if dtype == torch.float32 else \
        top.to(torch.int16).view(torch.bfloat16).float().log2().to(torch.bfloat16)
    if dtype == torch.bfloat16:
        vals = torch.unique(vals).flip(0)
    rest = torch.full((V - len(vals),), -30.0, dtype=dtype)
    down = torch.cat([vals, rest])               # descending
    mixed = down[torch.randperm(V, generator=g)]
    step = 512 * 16 // down.element_size()       # columns of one thread: 16 bytes every step
    per = 16 // down.element_size()
    own = torch.tensor([c for c in range(V) if c % step < per])
    packed = torch.empty_like(down)
    other = torch.ones(V, dtype=torch.bool)
    other[own] = False
    packed[own] = down[:len(own)]
    packed[other] = down[len(own):]
    for T, K, P in ((1.0, 50, 0.9), (20.0, 50, 1.0), (20.0, 1, 1.0), (20.0, 7, 1.0), (50.0, 100, 0.95),
                    (50.0, 129, 1.0), (50.0, 200, 0.99), (50.0, 256, 1.0), (50.0, 257, 1.0)):
        seeds = torch.arange(B, dtype=torch.int64, device="cuda") * 77 + K
        got = []
        for row in (mixed, down, packed):
            x = row[None].repeat(B, 1).cuda()
            tok = ops.sample(x, torch.full((B,), T, device="cuda"),
                             torch.full((B,), K, dtype=torch.int32, device="cuda"),
                             torch.full((B,), P, device="cuda"), seeds)
            got.append(x.gather(1, tok.long()[:, None]).cpu())
            assert (got[-1] >= down[min(K, V) - 1]).all(), (T, K, P)
        assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2]), (T, K, P)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [8191, 8192, 16384, 32768, 32776, 128256, 128257])
def test_rows_that_rise_with_the_index(V, dtype):
    """The threshold comes from a sample that is spread over the row, at sizes around those where it is
    the whole row, a half and a quarter; rows of odd lengths are not aligned."""
    B = 12
    g = torch.Generator().manual_seed(V)
    x = (torch.randn(V, generator=g) + torch.linspace(0, 8, V)).to(dtype)
    order = torch.randperm(V, generator=g)
    for K, P in ((1, 1.0), (50, 0.9), (64, 1.0), (65, 1.0), (128, 0.95), (129, 1.0), (256, 1.0)):
        picked = []
        for row in (x, x.flip(0), x[order]):
            rows = row[None].repeat(B, 1).cuda()
            tok = ops.sample(rows, torch.full((B,), 3.0, device="cuda"), torch.full((B,), K, dtype=torch.int32, device="cuda"),
                             torch.full((B,), P, device="cuda"), torch.arange(B, dtype=torch.int64, device="cuda") * 77 + K)
            picked.append(rows.gather(1, tok.long()[:, None]).cpu())
            assert (picked[-1] >= x.sort(descending=True).values[K - 1]).all(), (K, P)
        if dtype == torch.float32:               # (bf16 values tie, and ties count in the top k)
            assert torch.equal(picked[0], picked[1]) and torch.equal(picked[0], picked[2]), (K, P)
