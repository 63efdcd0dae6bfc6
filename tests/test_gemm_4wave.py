"""The 4-wave GEMM kernel at the edges of what it distinguishes: one to five K-tiles (two are staged ahead), columns
that end in a quad, an octet or neither, outputs whose rows lie apart or are not aligned, K split into slices, and
groups of rows, empty ones and more than a wave's lanes of them among these."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops
from distributed_llm_inferencing_amd.ops import gemm as G

# fp32 sums of exact products of up to 1280 values: 1e-5; bf16 results are rounded once, half an ulp (2^-9) a value
BOUND = {True: 1e-5, False: 2.0 ** -8}
TILES = [45]


def operands(gpu, M, N, K, seed, groups=1):
    g = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.randn(M, K, device=gpu, generator=g).bfloat16()
    w = (torch.randn(groups * N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    return x, w.view(groups, N, K)


def expected(x, w, epi, bias=None):
    want = x.double() @ w.double().t()
    if epi in G.PAIR_EPIS:
        gate, up = want.view(len(x), -1, 2, 16).unbind(2)
        act = torch.nn.functional.silu(gate) if epi == "silu_mul" else torch.nn.functional.gelu(gate, approximate="tanh")
        return (act * up).reshape(len(x), -1)
    if epi.startswith("bias"):
        want = want + bias.double()
    return torch.nn.functional.gelu(want, approximate="tanh") if epi == "bias_gelu" else want


def off(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,splits", [
    (1, 8, 64, 1), (256, 256, 128, 1), (257, 264, 192, 1), (511, 260, 320, 1), (300, 1001, 256, 1), (40, 520, 64, 1),
    (300, 520, 128, 2), (513, 1028, 384, 2), (300, 257, 640, 2), (700, 4104, 1280, 4), (2600, 8200, 64, 1), (5000, 4104, 192, 1)])
def test_products(gpu, M, N, K, splits, tile):
    x, w = operands(gpu, M, N, K, M + N + K)
    bias = torch.randn(N, device=gpu).bfloat16()
    for epi in ("none", "f32", "bias", "bias_gelu", "silu_mul"):
        if epi == "silu_mul" and N % 64:
            continue
        b = bias if epi.startswith("bias") else None
        got = ops._gemm_native(x, w[0], epi, bias=b, plan=G.GemmPlan("dli", tile, splits))
        assert off(got, expected(x, w[0], epi, bias)) < BOUND[epi == "f32"], epi


# outputs inside a wider buffer, whole and odd offsets: nothing beside the product is written
@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,wide,at", [(300, 264, 512, 8), (300, 264, 516, 4), (257, 260, 301, 3), (513, 512, 520, 0)])
@pytest.mark.parametrize("epi", ["none", "f32"])
def test_outputs_inside_wider_rows(gpu, M, N, wide, at, epi, tile):
    x, w = operands(gpu, M, N, 192, M + wide)
    whole = torch.full((M, wide), 7.0, device=gpu, dtype=torch.float32 if epi == "f32" else torch.bfloat16)
    ops._gemm_native(x, w[0], epi, out=whole[:, at:at + N], plan=G.GemmPlan("dli", tile, 1))
    assert off(whole[:, at:at + N], expected(x, w[0], epi)) < BOUND[epi == "f32"]
    assert torch.all(whole[:, :at] == 7) and torch.all(whole[:, at + N:] == 7)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("groups,splits", [(1, 1), (5, 1), (5, 2), (64, 1), (70, 1), (131, 1)])
@pytest.mark.parametrize("epi", ["none", "silu_mul"])
def test_groups_of_rows(gpu, groups, splits, epi, tile):
    N, K = 576, 256
    sizes = [(0, 37, 300, 1, 256, 0, 513)[i % 7] for i in range(groups)] if groups > 1 else [300]
    sizes[-1] = 0 if groups == 70 else sizes[-1]
    ends = torch.tensor([0, *sizes]).cumsum(0)
    x, w = operands(gpu, int(ends[-1]), N, K, groups, groups)
    got = ops._gemm_native(x, w, epi, plan=G.GemmPlan("dli", tile, splits), groups=groups,
                           group_off=ends.to(gpu, torch.int32), rows_per_group=len(x))
    want = torch.cat([expected(x[a:b], w[e], epi) for e, (a, b) in enumerate(zip(ends[:-1], ends[1:])) if b > a])
    assert off(got, want) < BOUND[False]


# sums that overflow and NaN, through the SiLU too
@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
def test_values_at_the_limits(gpu, tile):
    x = torch.zeros(300, 128, device=gpu).bfloat16()
    w = torch.zeros(64, 128, device=gpu).bfloat16()
    w[:16, 0] = w[:16, 2] = w[16:32, 1] = 1             # gates: twice column 0 of x, ups: column 1
    gates = [3e38, -3e38, float("nan"), 1.5e38, -1.5e38, -45.0, 45.0, 0.0, -0.0]
    for i, v in enumerate(gates):
        x[i, 0] = x[i, 2] = v
        x[i, 1] = 1
    got = ops._gemm_native(x, w, "silu_mul", plan=G.GemmPlan("dli", tile, 1))[:len(gates), 0].float().tolist()
    assert got[0] == float("inf") and got[3] > 2.9e38 and got[6] == 90.0 and got[7] == got[8] == 0
    assert got[1] != got[1] and got[2] != got[2]        # -inf / inf, NaN
    assert abs(got[4]) < 1e-30 and abs(got[5]) < 1e-30
