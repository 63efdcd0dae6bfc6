"""Portions whose full blocks take a loop of their own (heads of 128 channels, column blocks of 128), against the float64 walk:
portions around the shortest that take it, last blocks of 1, 15 and 16 tokens behind it, shorter portions beside
them, a whole column block beside a narrower one, and decays that leave the range of fp32; heads that cannot take it; and the
matrix memory's gates at the edges of a lane's tokens and of a pass."""
import pytest
import torch

from test_recurrence_chunks import check


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["hgrn2", "gla", "lightning", "mlstm"])
@pytest.mark.parametrize("lens", [[95, 80], [96, 64, 97], [127, 3], [128, 16, 81], [129, 112, 143]])
@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_around_the_shortest(gpu, mode, lens, strong, dtype):
    n = len(lens)
    check(gpu, mode, 128, 128, strong, dtype, lens, [4, 1, 0][:n], [0, 1, 0][:n])


@pytest.mark.gpu
@pytest.mark.parametrize("dv", [200, 256])
@pytest.mark.parametrize("lens", [[131, 20], [700]])
def test_column_blocks(gpu, dv, lens):
    check(gpu, "lightning", 128, dv, False, torch.float32, lens, [2, 5][:len(lens)], [0, 1][:len(lens)])


# the gates' maximum: 33 tokens a lane, 2112 a pass
@pytest.mark.gpu
@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("lens", [[2112, 33], [2113, 34, 1], [32, 66, 67], [512, 513]])
def test_gates_of_the_matrix_memory(gpu, strong, lens):
    n = len(lens)
    check(gpu, "mlstm", 128, 128, strong, torch.float32, lens, [3, 0, 2][:n], [0, 1, 0][:n])


# narrower heads, columns short of a block and rows past 24 bits keep the kernels of the general loop alone
@pytest.mark.parametrize("mode,tokens,d,dv,stride,expected", [
    (0, 96, 128, 128, 4096, 1), (0, 95, 128, 128, 4096, 0), (3, 127, 128, 128, 4096, 0), (3, 128, 128, 128, 4096, 1),
    (2, 4000, 128, 200, 4096, 1), (0, 4000, 96, 96, 4096, 0), (1, 4000, 112, 128, 4096, 0), (0, 4000, 128, 64, 4096, 0),
    (3, 4000, 100, 100, 4096, 0), (1, 4000, 128, 128, 1 << 24, 0)])
def test_choice(mode, tokens, d, dv, stride, expected):
    from distributed_llm_inferencing_amd.ops import _native
    assert _native.require_native().dli_recurrence_long(mode, tokens, d, dv, stride, 4096, 4096) == expected


# wide heads that are no whole tile, portions cut and whole
@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["hgrn2", "gla", "lightning", "mlstm"])
@pytest.mark.parametrize("d,dv", [(96, 96), (112, 128), (128, 64)])
@pytest.mark.parametrize("lens", [[129, 33, 144], [700, 5]])
def test_wide_heads_of_no_whole_tile(gpu, mode, d, dv, lens):
    n = len(lens)
    check(gpu, mode, d, dv, True, torch.float32, lens, [2, 0, 4][:n], [0, 1, 0][:n])


# the number of segments: of equal portions, of few and of many ragged ones, where every number was timed (within 12 % of the best
# one's time; the numbers left out are up to four times that)
@pytest.mark.parametrize("heads,d,dv,lens,good", [
    (32, 128, 128, [2048] * 4, (2, 4)), (32, 128, 128, [256] * 32, (1,)), (32, 128, 128, [8000], (8,)),
    (16, 32, 32, [1994, 2512, 3165, 3988], (8, 9, 10, 11, 13, 14, 15, 16)), (16, 64, 64, [1060, 1395, 1836, 2417, 3181], range(7, 17)),
    (32, 128, 128, [152, 172, 194, 220, 248, 281, 317, 358, 405, 458], (1,)),
    (32, 128, 128, [671, 798, 949, 1129, 1343], (2, 4, 5, 6, 8, 9, 10))])
def test_segments(heads, d, dv, lens, good):
    from distributed_llm_inferencing_amd.ops import _native
    width = 32 if d <= 32 else 64 if d <= 64 else 128
    unit = 4 * heads * len(lens) * (width * 128 + 256)      # bytes of one segment a portion: states, decays and normalisers
    nb = _native.require_native().dli_recurrence_workspace_bytes(0, len(lens), max(lens), sum(lens), 1, heads, d, dv)
    assert nb % unit == 0 and max(1, nb // unit) in good
