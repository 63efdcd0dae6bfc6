"""Tiles of 192 and 320 rows of the 4-wave kernel, which tiles 22 and 55 take where they fill the rounds better: every shape
sums a product's terms in the order that the 256 x 256 tile (45) does, so that results are equal to the bit."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops
from distributed_llm_inferencing_amd.ops import gemm as G
from test_head_maxima import block_keys

# every shape (rows, columns of a tile), whole and partial tiles, one to three a workgroup; 24 to 33 K-tiles
CASES = [(1, 520, 1536, 1, 192), (193, 1032, 1600, 1, 192), (300, 16392, 1536, 1, 192), (1281, 6152, 1664, 1, 192),
         (321, 24584, 1536, 1, 192), (1281, 20488, 1536, 1, 192), (577, 12904, 1600, 1, 320), (577, 17032, 1536, 1, 320),
         (300, 1001, 1536, 1, 192), (321, 16385, 2112, 1, 192), (577, 17041, 1536, 1, 320)]
SPLIT = [(65, 520, 1536, 2, 192), (300, 4104, 2048, 4, 192), (321, 8200, 2048, 4, 192), (65, 12296, 2048, 4, 192),
         (300, 6152, 2048, 4, 320), (577, 4104, 2048, 4, 320), (300, 8201, 1536, 2, 192)]


def rows(tile, epi, M, N, K, splits):
    from distributed_llm_inferencing_amd.ops import _native
    return _native.require_native().dli_gemm_4w_rows(tile, G.EPI[epi], M, N, K, splits)


def operands(dev, M, N, K):
    g = torch.Generator(device=dev).manual_seed(M + N)
    return (torch.randn(M, K, device=dev, generator=g).bfloat16(),
            (torch.randn(N, K, device=dev, generator=g) * K ** -0.5).bfloat16())


def call(x, w, out, epi, tile, splits=1, ws=None):
    from distributed_llm_inferencing_amd.ops import _native
    assert _native.require_native().dli_gemm(
        ops._p(x), x.stride(0), ops._p(w), w.stride(0), ops._p(out), w.shape[0] if out is None else out.stride(0), x.shape[0],
        w.shape[0], x.shape[1], G.EPI[epi], tile, splits, None, ops._p(ws), None, 1, ops._st()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [22, 55])
@pytest.mark.parametrize("M,N,K,splits,tall", CASES)
def test_outputs(gpu, M, N, K, splits, tall, tile):
    if tile == 55:
        K += K % 128
    x, w = operands(gpu, M, N, K)
    want = x.double() @ w.double().t()
    for epi in ("none", "f32", "silu_mul", "gelu_mul", "res_add"):
        if epi in G.PAIR_EPIS:
            n = N // 64 * 64
            wide, other = n // 2, 28 if epi == "gelu_mul" else 45   # (45 has no GELU pairs: 28, of 256 x 128, does)
        else:
            n, wide, other = N, N, 45
        if epi == "res_add" and N % 8:
            continue
        assert rows(tile, epi, M, n, K, 1) == tall and rows(other, epi, M, n, K, 1) == 256
        held = torch.full((M + 330, wide + 8), 0.5, device=gpu, dtype=torch.float32 if epi == "f32" else torch.bfloat16)
        ref = held.clone()
        call(x, w[:n], held[:M, :wide], epi, tile)
        call(x, w[:n], ref[:M, :wide], epi, other)
        assert torch.equal(held, ref), epi                  # (nothing beside or behind the output either)
        if epi == "gelu_mul":
            gate, up = want[:, :n].view(M, -1, 2, 16).unbind(2)
            exact = (torch.nn.functional.gelu(gate, approximate="tanh") * up).reshape(M, -1)
            # a rounding to bf16 is 2^-9 of the value at most, the norm of all less
            assert float((held[:M, :wide].double() - exact).norm() / exact.norm()) < 2.0 ** -8
        if epi == "f32":
            assert float((ref[:M, :wide].double() - want).norm() / want.norm()) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,splits,tall", SPLIT)
def test_partial_sums(gpu, M, N, K, splits, tall):
    x, w = operands(gpu, M, N, K)
    for epi, dt, other in (("none", torch.float32, 45), ("slab16", torch.float16, 28)):
        assert rows(22, epi, M, N, K, splits) == tall
        held = torch.full((splits * M + 330, N), 7.0, device=gpu, dtype=dt)
        ref = held.clone()
        call(x, w, None, epi, 22, splits, held)
        call(x, w, None, epi, other, splits, ref)
        assert torch.equal(held, ref) and bool((held[splits * M:] == 7).all()) and not bool((held[:splits * M] == 7).all())


# rows so far apart that 320 of them leave the kernel's 32-bit offsets stay on tiles of 256
@pytest.mark.gpu
@pytest.mark.parametrize("stride", [(1 << 21) - 8, 1 << 21, (1 << 22) - 8])
def test_rows_far_apart(gpu, stride):
    M, N, K = 600, 12296, 1536
    x, w = operands(gpu, M, N, K)
    far = torch.empty(M * stride, device=gpu, dtype=torch.bfloat16).view(M, stride)[:, :K]
    far.copy_(x)
    a, b = (torch.empty(M, N, device=gpu) for _ in range(2))
    call(far, w, a, "f32", 22)
    call(x, w, b, "f32", 45)
    assert torch.equal(a, b)


# where the taller or wider tile would move as many bytes for fewer products, those of 256 rows stay (2 to 14 % ahead there)
@pytest.mark.parametrize("epi,M,N,K,splits,tall", [
    ("silu_mul", 820, 8192, 5120, 1, 256), ("none", 640, 14336, 14336, 1, 256), ("res_add", 640, 32000, 14336, 1, 256),
    ("silu_mul", 777, 22016, 11008, 1, 256), ("slab16", 777, 2048, 8192, 4, 256),
    ("none", 777, 8192, 2048, 1, 256), ("silu_mul", 2112, 28672, 4096, 1, 192), ("res_add", 1100, 4096, 14336, 1, 192),
    ("res_add", 5000, 4096, 14336, 1, 320)])
def test_choice(epi, M, N, K, splits, tall):
    assert rows(22, epi, M, N, K, splits) == tall


# short K, groups, biases and the other tiles keep 256 rows, and so does a head with block maxima
def test_what_stays():
    assert rows(22, "none", 300, 1000, 1472, 1) == 256 and rows(22, "none", 300, 1000, 4096, 16) == 256
    assert rows(45, "none", 300, 1000, 4096, 1) == 256 and rows(28, "none", 300, 1000, 4096, 1) == 256
    assert rows(22, "bias", 300, 1000, 4096, 1) == 256


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(300, 30720, 2048), (577, 17032, 1536)])
def test_block_maxima_of_the_head(gpu, monkeypatch, M, N, K):
    x, w = operands(gpu, M, N, K)
    assert rows(55, "f32", M, N, K, 1) != 256
    monkeypatch.setattr(G, "row_cut", lambda *a: 0)
    monkeypatch.setattr(G, "plan", lambda *a, **k: G.GemmPlan("dli", 55, 1))
    logits, top = ops.head(x, w)
    assert torch.equal(top[0], block_keys(logits, top[1]))
