"""The weight-streaming GEMM tiles (2 to 128 rows): the fitted plans at each side of their lines, and every
tile against float64 at the sizes where it can go wrong."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops
from distributed_llm_inferencing_amd.ops import gemm as G
from distributed_llm_inferencing_amd.ops.reference import interleave_gate_up


@pytest.mark.parametrize("M,N,K,epi,tile,splits", [
    # 32, 64 and 128 columns, each where it fills three quarters of the chip; below, 64 and K split
    (5, 6112, 4096, "f32", 62, 2), (32, 6144, 4096, "f32", 60, 1), (32, 6144, 4160, "f32", 61, 1), (24, 12224, 4096, "f32", 60, 1),
    (24, 12288, 4096, "f32", 62, 1), (24, 24448, 4096, "silu_mul", 62, 1), (24, 24480, 4096, "silu_mul", 61, 1),
    (33, 4096, 4096, "f32", 64, 4), (33, 8192, 4096, "f32", 69, 1), (64, 16384, 4160, "f32", 64, 1), (64, 28672, 4096, "silu_mul", 63, 1),
    (65, 4096, 4096, "f32", 70, 4), (65, 3008, 4096, "f32", 5, 4), (96, 8192, 4096, "f32", 72, 1), (96, 28672, 4096, "silu_mul", 66, 1),
    (97, 4096, 4096, "f32", 6, 4), (128, 4096, 14336, "f32", 7, 8), (97, 12288, 4096, "f32", 71, 1), (97, 28672, 4096, "silu_mul", 67, 1),
    (24, 128256, 4096, "f32", 62, 1), (64, 128256, 4096, "f32", 65, 1), (65, 128256, 4096, "f32", 68, 1), (129, 4096, 4096, "f32", 1, 8),
    # short K is not split, but where a fused reduce follows
    (24, 4096, 1024, "f32", 62, 1), (24, 4096, 1024, "splitk", 62, 2), (24, 4096, 768, "splitk", 62, 1),
    # narrow weights: the 64-column tile with 3 stages
    (97, 3072, 768, "bias_gelu", 5, 1), (128, 5120, 1024, "f32", 5, 1), (97, 4096, 1088, "f32", 6, 1), (96, 3072, 768, "f32", 70, 1),
    (33, 256, 1024, "bias_gelu", 5, 4), (64, 96, 4096, "f32", 5, 8), (33, 64, 768, "none", 5, 1), (32, 256, 1024, "f32", 62, 1),
    (33, 257, 1024, "f32", 64, 1), (128, 256, 2048, "f32", 5, 4),
    # up to 4 rows stay on the plain weight stream
    (5, 28672, 4096, "silu_mul", 61, 1), (4, 28672, 4096, "silu_mul", 31, 1), (4, 4096, 4096, "f32", 30, 2),
    (1, 28672, 4096, "silu_mul", 29, 1)])
def test_fitted_plan(M, N, K, epi, tile, splits):
    assert G._heuristic(M, N, K, epi) == G.GemmPlan("dli", tile, splits)


def test_every_candidate_fits_its_rows_and_k():
    for M in (1, 2, 3, 4, 5, 16, 17, 32, 33, 64, 65, 96, 97, 128, 129, 512):
        for K in (64, 192, 768, 4096, 4160):
            for epi in ("f32", "splitk", "silu_mul", "none"):
                for p in G.candidate_plans(M, 4096, K, epi):
                    if p.tile in G.STREAM_TILES:
                        bm, _, step = G.STREAM_TILES[p.tile]
                        assert K % (step * p.splits) == 0 and 2 <= M <= bm
                        assert M > G.GEMV_MAX_M or epi not in ("splitk", "none")


# Sums are fp32 in up to 64 steps of 32 exact products (1e-6); bf16 results are rounded once, half an ulp
# (2^-9) a value; fp16 partial sums likewise (2^-11 each)
@pytest.mark.gpu
@pytest.mark.parametrize("tile", sorted(G.STREAM_TILES))
@pytest.mark.parametrize("rows", ["one", "full", "two rows of tiles"])
def test_tiles_match_float64(gpu, tile, rows):
    bm, bn, step = G.STREAM_TILES[tile]
    M = {"one": 1, "full": bm, "two rows of tiles": bm + 3}[rows]
    g = torch.Generator(device=gpu).manual_seed(tile)
    for N, K, epi, splits in ((bn + 3, step, "f32", 1), (3 * bn - 1, 2 * step, "none", 1), (96, 3 * step, "silu_mul", 1),
                              (5 * bn + 32, 9 * step, "silu_mul", 1), (bn * 2, 8 * step, "f32", 4),
                              (260, 4 * step, "slab16", 2), (bn + 16, 5 * step, "bias_gelu", 1)):
        x = torch.randn(M, K, device=gpu, generator=g).bfloat16()
        w = (torch.randn(N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
        bias = torch.randn(N, device=gpu, generator=g).bfloat16() if epi == "bias_gelu" else None
        want, plan, tol = x.double() @ w.double().t(), G.GemmPlan("dli", tile, splits), 2.0 ** -8
        if epi == "slab16":
            ws = torch.full((splits, M, N), 7.0, dtype=torch.float16, device=gpu)
            ops._native_call("dli_gemm", x.data_ptr(), K, w.data_ptr(), K, None, N, M, N, K, G.EPI[epi], tile, splits,
                             None, ws.data_ptr(), None, 1, ops._st())
            got, tol = ws.double().sum(0) * 16, 2.0 ** -10
        else:
            if epi == "silu_mul":
                gate, up = want[:, :N // 2], want[:, N // 2:]
                want, w = torch.nn.functional.silu(gate) * up, interleave_gate_up(w[:N // 2], w[N // 2:]).contiguous()
            elif bias is not None:
                want = torch.nn.functional.gelu(want + bias.double(), approximate="tanh")
            got = ops._gemm_native(x, w, epi, bias=bias, plan=plan).double()
            tol = 1e-5 if epi == "f32" else tol
        err = float((got - want).norm() / want.norm())
        assert err < tol, (N, K, epi, splits, err)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", (60, 61, 63, 66))
def test_grouped_tiles_match_float64(gpu, tile):
    """Experts of no, one, a full tile's and more rows, gathered and in place."""
    bm, _, step = G.STREAM_TILES[tile]
    counts, K, N = [3, 0, bm, 1, bm + 5], 2 * step, 160
    off = [sum(counts[:i]) for i in range(len(counts) + 1)]
    g = torch.Generator(device=gpu).manual_seed(tile)
    x = torch.randn(off[-1], K, device=gpu, generator=g).bfloat16()
    w = (torch.randn(len(counts), N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    offs = torch.tensor(off, dtype=torch.int32, device=gpu)
    want = torch.cat([x[a:b].double() @ w[e].double().t() for e, (a, b) in enumerate(zip(off, off[1:]))])
    got = ops._gemm_native(x, w, "none", plan=G.GemmPlan("dli", tile, 1), groups=len(counts), group_off=offs,
                           rows_per_group=off[-1]).double()
    assert float((got - want).norm() / want.norm()) < 2.0 ** -8
    rows = torch.randperm(off[-1], device=gpu, generator=g).to(torch.int32)
    out = torch.empty(off[-1], N // 2, dtype=torch.bfloat16, device=gpu)
    ops._native_call("dli_gemm_grouped_gather", x.data_ptr(), K, w.data_ptr(), K, out.data_ptr(), N // 2, off[-1], N, K,
                     tile, rows.data_ptr(), offs.data_ptr(), len(counts), ops._st())
    want = torch.cat([x[rows[a:b].long()].double() @ w[e].double().t() for e, (a, b) in enumerate(zip(off, off[1:]))])
    want = want.view(off[-1], N // 32, 2, 16)
    want = (torch.nn.functional.silu(want[:, :, 0]) * want[:, :, 1]).reshape(off[-1], N // 2)
    assert float((out.double() - want).norm() / want.norm()) < 2.0 ** -8


@pytest.mark.parametrize("M,N,K,cut", [
    (4104, 4096, 4096, 4096), (4224, 4096, 4096, 4096), (4225, 4096, 4096, 0), (4096, 4096, 4096, 0), (4353, 4096, 4096, 0),
    (8199, 28672, 4096, 8192), (4104, 6144, 4096, 0), (8199, 6144, 4096, 8192), (1312, 12288, 4096, 1280),
    (513, 28672, 4096, 0), (640, 32000, 4096, 0), (769, 32000, 4096, 0), (1025, 32000, 4096, 1024),
    (513, 65536, 4096, 0), (300, 32768, 4096, 0), (2049, 128256, 4096, 0), (4104, 4096, 512, 0), (4104, 4096, 4104, 0)])
def test_rows_that_would_begin_a_round_run_apart(M, N, K, cut):
    assert G.row_cut(M, N, K) == cut


@pytest.mark.gpu
@pytest.mark.parametrize("rest", (1, 3, 33, 128))
@pytest.mark.parametrize("epi", ("f32", "none", "silu_mul", "bias_gelu", "gelu_mul"))
def test_products_cut_by_rows(gpu, rest, epi):
    M, N, K = 4096 + rest, 4096, 1024
    kept = dict(G._plan_cache), set(G._tuned)
    G.clear_plans()
    assert G.row_cut(M, N, K) == 4096
    g = torch.Generator(device=gpu).manual_seed(rest)
    x = torch.randn(M, 2 * K, device=gpu, generator=g).bfloat16()[:, K:]      # (rows of a wider tensor)
    w = (torch.randn(N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    bias = torch.randn(N, device=gpu, generator=g).bfloat16() if epi == "bias_gelu" else None
    want = x.double() @ w.double().t()
    if epi in G.PAIR_EPIS:
        act = torch.nn.functional.silu if epi == "silu_mul" else lambda v: torch.nn.functional.gelu(v, approximate="tanh")
        want, w = act(want[:, :N // 2]) * want[:, N // 2:], interleave_gate_up(w[:N // 2], w[N // 2:]).contiguous()
    elif bias is not None:
        want = torch.nn.functional.gelu(want + bias.double(), approximate="tanh")
    try:
        got = ops.linear(x, w, bias, epi=epi).double()
    finally:
        G.clear_plans()
        G._plan_cache.update(kept[0])
        G._tuned.update(kept[1])
    tol = 1e-5 if epi == "f32" else 2.0 ** -8
    for rows in (slice(0, 4096), slice(4096, M)):
        assert float((got[rows] - want[rows]).norm() / want[rows].norm()) < tol
