"""Products added into their output by the 4-wave kernel's epilogue (EPI "res_add"), and linear_add_rmsnorm's choice of it."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops
from distributed_llm_inferencing_amd.ops import gemm as G


def call(x, w, out, tile, splits=1, n=None):
    """dli_gemm's status."""
    from distributed_llm_inferencing_amd.ops import _native as N
    ws = torch.empty(splits * x.shape[0] * w.shape[0] * 4, dtype=torch.uint8, device=x.device)
    return N.require_native().dli_gemm(
        ops._p(x), x.stride(0), ops._p(w), w.stride(0), ops._p(out), out.stride(0), x.shape[0], n or w.shape[0], x.shape[1],
        G.EPI["res_add"], tile, splits, None, ops._p(ws), None, 1, ops._st())


def close(got, x, w, before):
    """Within an fp32 sum's error (K products of relative 2^-24 each) and one rounding to bf16 of 64 bits: half a unit in
    the last of 8 significant bits is up to 2^-8 of a number just above a power of two."""
    ref = before.double() + x.double() @ w.double().t()
    size = before.double().abs() + x.double().abs() @ w.double().abs().t()
    return bool(((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + (x.shape[1] + 1) * 2.0 ** -24 * size).all())


SIZES = [(1, 8, 64), (17, 24, 128), (128, 264, 64), (129, 136, 192), (255, 248, 256), (256, 256, 128), (257, 1000, 128),
         (300, 520, 640), (700, 4104, 256), (2112, 4096, 128), (257, 24008, 192), (300, 28008, 128), (513, 32776, 64)]


# the sizes below are on tiles of every width that the kernel has
def test_widths():
    from distributed_llm_inferencing_amd.ops import _native as N
    width = lambda tile: {N.require_native().dli_gemm_4w_width(tile, G.EPI["res_add"], m, n, 1) for m, n, _ in SIZES}
    assert width(22) == {128, 160, 192, 224, 256} and width(55) == {160, 192, 256} and width(28) == {128} and width(45) == {256}


# edges of the 256-row tile and its waves, of 16 columns and each tile width, K of one, two, three and more K-tiles.
# A tile's rows past the product's, up to 255, are kept off what follows it by a descriptor's range
@pytest.mark.gpu
@pytest.mark.parametrize("tile", [45, 22, 28, 55])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_sums(gpu, tile, M, N, K):
    if tile == 55 and K % 128:
        K += 64
    g = torch.Generator(device=gpu).manual_seed(M)
    x = torch.randn(M, K, device=gpu, generator=g).bfloat16()
    w = torch.randn(N, K, device=gpu, generator=g).bfloat16()
    held = torch.randn(M + 257, N + 16, device=gpu, generator=g).bfloat16()
    before = held.clone()
    assert call(x, w, held[1:, 8:], tile) == 0
    assert close(held[1:M + 1, 8:N + 8], x, w, before[1:M + 1, 8:N + 8])
    held[1:M + 1, 8:N + 8] = before[1:M + 1, 8:N + 8]
    assert torch.equal(held, before)                       # nothing beside the output


@pytest.mark.gpu
def test_refused(gpu):
    x, w = torch.zeros(64, 128, device=gpu).bfloat16(), torch.zeros(64, 128, device=gpu).bfloat16()
    out = torch.ones(64, 80, device=gpu).bfloat16()
    assert call(x, w, out, 45, splits=2) != 0
    assert call(x, w, out[:, 4:], 45) != 0                  # rows that are not 16-byte aligned
    assert call(x, w, out, 45, n=60) != 0                   # columns in part of 8
    assert call(x, w, out[:, :76].contiguous(), 45) != 0    # rows in part of 8
    assert call(x, w, out, 2) != 0                          # a kernel without it
    torch.cuda.synchronize()
    assert bool((out == 1).all())


# rows that the rule takes, with a cut, and calls that stay with the separate add: few rows, a residual that is not
# aligned, columns in part of 8, a split plan
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,off,taken", [(4096, 4096, 256, 0, True), (8199, 4096, 7168, 0, True), (512, 4096, 256, 0, False),
                                             (4096, 4096, 256, 4, False), (4096, 4100, 256, 0, False), (1100, 4096, 4096, 0, False)])
@pytest.mark.parametrize("norm", [True, False])
def test_linear_add_rmsnorm(gpu, monkeypatch, M, N, K, off, taken, norm):
    g = torch.Generator(device=gpu).manual_seed(N + K)
    x = torch.randn(M, K, device=gpu, generator=g).bfloat16()
    w = (torch.randn(N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    nw = torch.randn(N, device=gpu, generator=g).bfloat16()
    residual = torch.randn(M * N + off, device=gpu, generator=g).bfloat16()[off:].view(M, N)
    before = residual.clone()
    assert (G.row_cut(M, N, K) > 0) == (M == 8199)
    norm = norm and N % 8 == 0                              # (what the norm takes)
    assert ops._add_product(x, w, residual, None) == taken  # its own decision
    residual.copy_(before)
    h = ops.linear_add_rmsnorm(x, w, residual, nw if norm else None, 1e-5)
    if taken:
        rows = slice(M - 300, M)                            # (the cut's both sides)
        want = before[rows].float() + x[rows].float() @ w.float().t()
        # the sum rounded to bf16, behind the cut the product too: 2^-8 of each
        assert bool(((residual[rows].float() - want).abs()
                     <= 2.0 ** -8 * (want.abs() + (want - before[rows].float()).abs()) + 1e-4).all())
    else:
        monkeypatch.setattr(ops, "_add_product", lambda *a: False)
        normed = ops.linear_add_rmsnorm(x, w, before, nw if norm else None, 1e-5)
        assert torch.equal(residual, before)
    if not norm:
        assert h is None
    else:
        assert torch.equal(h, ops.rmsnorm(residual, nw, 1e-5) if taken else normed)


# the add inside the product stores tiles while others are read: not where the residual is an operand, or shares bytes
# with one, nor where it lies elsewhere
@pytest.mark.parametrize("K", [1024, 4096])
def test_operands_apart_from_the_residual(monkeypatch, K):
    calls = []
    monkeypatch.setattr(ops, "_use_native", lambda t: True)
    monkeypatch.setattr(ops, "_gemm_native", lambda *a, **k: calls.append(a))
    monkeypatch.setattr(G, "row_cut", lambda *a: 0)
    monkeypatch.setattr(G, "plan", lambda *a: G.GemmPlan("dli", 22, 1))
    M, N = 1024, 1024
    held = torch.zeros(3 * M * K).bfloat16()
    residual, w = held[:M * N].view(M, N), torch.zeros(N, K).bfloat16()
    for at, x in ((0, held[:M * K]), (8, held[8:M * K + 8]), (M * N - 8, held[M * N - 8:M * N - 8 + M * K])):
        assert not ops._add_product(x.view(M, K), w, residual, None) and not calls, at
    assert not ops._add_product(torch.zeros(M, K).bfloat16(), held[M * N - 8:M * N - 8 + N * K].view(N, K), residual, None)
    assert not ops._add_product(torch.zeros(M, K).bfloat16(), w, residual.to("meta"), None) and not calls
    assert ops._add_product(held[M * N:M * N + M * K].view(M, K), w, residual, None) and calls


@pytest.mark.gpu
@pytest.mark.parametrize("norm", [True, False])
def test_a_residual_that_is_the_input(gpu, norm):
    g = torch.Generator(device=gpu).manual_seed(3)
    x = torch.randn(4096, 4096, device=gpu, generator=g).bfloat16()
    w = (torch.randn(4096, 4096, device=gpu, generator=g) / 64).bfloat16()
    nw = torch.ones(4096, device=gpu).bfloat16() if norm else None
    want = x + ops.linear(x, w)
    ops.linear_add_rmsnorm(x, w, x, nw, 1e-5)
    assert torch.equal(x, want)
