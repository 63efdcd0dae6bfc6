"""The 4-wave GEMM kernel at the edges of what it distinguishes: one to five K-tiles (two are staged ahead), columns
that end in a quad, an octet or neither, outputs whose rows lie apart or are not aligned, K split into slices, and
groups of rows, empty ones and more than a wave's lanes of them among these."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops
from distributed_llm_inferencing_amd.ops import gemm as G
from test_head_maxima import block_keys

# fp32 sums of exact products of up to 1280 values: 1e-5; bf16 results are rounded once, half an ulp (2^-9) a value
BOUND = {True: 1e-5, False: 2.0 ** -8}
TILES = [45, 22, 28]      # 256 columns, by rounds of the chip, 128


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


# partial sums in 16 bits on tiles of every width that tile 22 takes; half an ulp (2^-11) of each of the slices, whose
# squares add up to the sum's; nothing behind the last slab
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,splits,width", [
    (300, 15000, 256, 2, 256), (300, 12808, 256, 2, 224), (512, 6144, 1024, 4, 192), (300, 10244, 384, 2, 192),
    (512, 4096, 1024, 4, 128), (257, 1001, 512, 8, 128), (300, 9000, 256, 2, 160)])
@pytest.mark.parametrize("tile", [22, 28])
def test_partial_sums_in_16_bits(gpu, M, N, K, splits, width, tile):
    x, w = operands(gpu, M, N, K, M + N)
    from distributed_llm_inferencing_amd.ops import _native
    assert _native.require_native().dli_gemm_4w_width(tile, G.EPI["slab16"], M, N, splits) == (128 if tile == 28 else width)
    held = torch.full((splits * M + 256, N), 7.0, device=gpu, dtype=torch.float16)
    ws, behind = held[:splits * M].view(splits, M, N), held[splits * M:]
    ops._native_call("dli_gemm", ops._p(x), K, ops._p(w), K, None, N, M, N, K, G.EPI["slab16"], tile, splits, None,
                     ops._p(ws), None, 1, ops._st())
    assert off(ws.double().sum(0) * 16, expected(x, w[0], "none")) < 2.0 ** -11 and torch.all(behind == 7)


# outputs inside a wider buffer, whole and odd offsets: nothing beside the product is written, nor behind it, where a tile's
# rows go on (up to 255 of them)
@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,wide,at", [(300, 264, 512, 8), (300, 264, 516, 4), (257, 260, 301, 3), (513, 512, 520, 0),
                                         (1, 264, 512, 8), (17, 264, 264, 0), (300, 30000, 30000, 0), (257, 1000, 1000, 0)])
@pytest.mark.parametrize("epi", ["none", "f32"])
def test_outputs_inside_wider_rows(gpu, M, N, wide, at, epi, tile):
    x, w = operands(gpu, M, N, 192, M + wide)
    whole = torch.full((M + 256, wide), 7.0, device=gpu, dtype=torch.float32 if epi == "f32" else torch.bfloat16)
    ops._gemm_native(x, w[0], epi, out=whole[:M, at:at + N], plan=G.GemmPlan("dli", tile, 1))
    assert off(whole[:M, at:at + N], expected(x, w[0], epi)) < BOUND[epi == "f32"]
    whole[:M, at:at + N] = 7
    assert torch.all(whole == 7)


# fp32 partial sums: nothing behind the last slab
@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,splits", [(1, 264, 128, 2), (17, 260, 256, 4), (257, 1001, 512, 8), (300, 1000, 384, 2)])
def test_partial_sums(gpu, M, N, K, splits, tile):
    x, w = operands(gpu, M, N, K, M + N)
    held = torch.full((splits * M + 256, N), 7.0, device=gpu)
    ops._native_call("dli_gemm", ops._p(x), K, ops._p(w), K, None, N, M, N, K, G.EPI["none"], tile, splits, None,
                     ops._p(held), None, 1, ops._st())
    assert off(held[:splits * M].view(splits, M, N).double().sum(0), expected(x, w[0], "none")) < BOUND[True]
    assert torch.all(held[splits * M:] == 7)


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


# the LM head of a plan on tile 22 writes block maxima too, as tile 55 (the same kernel); they are exact
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(300, 1000, 512), (257, 20000, 256), (300, 24000, 128), (300, 30720, 512), (300, 1000, 192)])
def test_block_maxima_of_the_head(gpu, monkeypatch, M, N, K):
    x, w = operands(gpu, M, N, K, M + N)
    monkeypatch.setattr(G, "row_cut", lambda *a: 0)
    monkeypatch.setattr(G, "plan", lambda *a, **k: G.GemmPlan("dli", 22, 1))
    logits, top = ops.head(x, w[0])
    assert off(logits, expected(x, w[0], "f32")) < BOUND[True]
    assert (top is None) == (K % 128 != 0)               # tile 55 takes whole pairs of K-tiles
    assert top is None or torch.equal(top[0], block_keys(logits, top[1]))


# SiLU and GELU pairs divide as the other kernels do, to the bit: 4 million gates given to 24 bits (three bf16 values each,
# which one product adds up), of which a quotient off by an ulp of fp32 would round some 30 to another bf16 value
@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("epi", ["silu_mul", "gelu_mul"])
def test_quotients(gpu, epi, tile):
    if tile == 45 and epi == "gelu_mul":
        tile = 55
    M, gates, K = 32768, 128, 512
    g = torch.Generator(device=gpu).manual_seed(7)
    left = torch.randn(M, gates, device=gpu, generator=g) * torch.tensor([1.0, 4.0, 40.0, 0.01], device=gpu).repeat(gates // 4)
    x = torch.zeros(M, K, device=gpu).bfloat16()
    for i in range(3):
        x[:, i:3 * gates:3] = left.bfloat16()
        left = left - x[:, i:3 * gates:3].float()
    x[:, 3 * gates] = torch.rand(M, device=gpu, generator=g).bfloat16() + 0.5
    w = torch.zeros(gates // 16, 2, 16, K, device=gpu).bfloat16()
    for j in range(gates):
        w[j // 16, 0, j % 16, 3 * j:3 * j + 3] = 1
    w[:, 1, :, 3 * gates] = 1
    w = w.view(2 * gates, K)
    got, other = (ops._gemm_native(x, w, epi, plan=G.GemmPlan("dli", t, 1)) for t in (tile, 13))
    assert torch.equal(got, other)


# the kernel stores partial sums in one way: a product that should use another is refused, not run as if it did
@pytest.mark.gpu
@pytest.mark.parametrize("family", [None, 2])
def test_other_store_modes_are_refused(gpu, family):
    from distributed_llm_inferencing_amd.ops import _native
    lib = _native.require_native()
    x, w = operands(gpu, 300, 512, 256, 1)
    setter = lib.dli_gemm_set_slab_store if family is None else lambda m: lib.dli_gemm_set_slab_store_family(family, m)
    before = [ops._gemm_native(x, w[0], "f32", plan=G.GemmPlan("dli", t, 2)) for t in TILES]
    assert setter(2) == 0
    try:
        for tile in TILES:
            with pytest.raises(RuntimeError):
                ops._gemm_native(x, w[0], "f32", plan=G.GemmPlan("dli", tile, 2))
            ops._gemm_native(x, w[0], "f32", plan=G.GemmPlan("dli", tile, 1))
    finally:
        assert setter(0) == 2
    assert all(torch.equal(b, ops._gemm_native(x, w[0], "f32", plan=G.GemmPlan("dli", t, 2))) for b, t in zip(before, TILES))
