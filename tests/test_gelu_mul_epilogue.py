"""gelu(gate) * up in the GEMM epilogue and over an interleaved fp32 projection, against float64."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops
from distributed_llm_inferencing_amd.ops import gemm as G
from distributed_llm_inferencing_amd.ops import hybrid as H
from distributed_llm_inferencing_amd.ops.reference import interleave_gate_up


def case(M, F, K, device):
    g = torch.Generator().manual_seed(M + F)
    x = torch.randn(M, K, generator=g).bfloat16()
    gate, up = ((torch.randn(F, K, generator=g) * s * K ** -0.5).bfloat16() for s in (3.0, 1.0))
    a, u = x.double() @ gate.double().t(), x.double() @ up.double().t()
    want = torch.nn.functional.gelu(a, approximate="tanh") * u
    return x.to(device), interleave_gate_up(gate, up).contiguous().to(device), want


# the product's terms are exact in fp32 and its sum of K terms is good to about 1e-6; the result is
# rounded to bf16 once, half an ulp (2^-9) a value
def close(got, want):
    assert float((got.double().cpu() - want).norm() / want.norm()) < 2.0 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("tile,splits", [(0, 1), (0, 2), (1, 4), (2, 1), (13, 1), (22, 1), (22, 2), (26, 1), (28, 2),
                                         (55, 1)])
@pytest.mark.parametrize("M", [5, 70, 300])
def test_epilogue(gpu, tile, splits, M):
    x, w, want = case(M, 448, 256, gpu)
    close(ops._gemm_native(x, w, "gelu_mul", plan=G.GemmPlan("dli", tile, splits)), want)


@pytest.mark.gpu
@pytest.mark.parametrize("M,F", [(1, 32), (4, 448), (33, 16)])
def test_interleaved_projection(gpu, M, F):
    x, w, want = case(M, F, 128, gpu)
    close(H.act_mul(H.linear_any(x, w), F, torch.bfloat16, "gelu_mul_pairs"), want)


def test_cpu_forms():
    x, w, want = case(7, 32, 64, "cpu")
    close(ops.linear(x, w, epi="gelu_mul"), want)
    close(H.act_mul(H.linear_any(x, w), 32, torch.bfloat16, "gelu_mul_pairs"), want)
