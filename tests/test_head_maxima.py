"""The LM head's block maxima and the sampler that reads them."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops
from distributed_llm_inferencing_amd.ops import _native as N
from distributed_llm_inferencing_amd.ops import gemm as G


def keys_of(x):
    """Order-preserving int64 keys of fp32 values."""
    u = x.view(torch.int32).long() & 0xffffffff
    return torch.where(u >> 31 == 1, u ^ 0xffffffff, u | 0x80000000)


def block_keys(x, bw):
    B, V = x.shape
    k = torch.zeros(B, -(-V // bw) * bw, dtype=torch.int64, device=x.device)
    k[:, :V] = keys_of(x)
    k = k.view(B, -1, bw).amax(-1)
    return torch.where(k >= 1 << 31, k - (1 << 32), k).int().contiguous()


# a kernel of each family and width; rows and columns that end inside a tile (the keys are exact: the
# products are neither zero nor NaN), and the logits those of the kernel without keys
@pytest.mark.gpu
@pytest.mark.parametrize("tile,M", [(30, 1), (30, 3), (31, 4), (32, 1), (60, 5), (61, 32), (62, 17), (63, 64),
                                    (64, 33), (65, 40), (66, 96), (67, 100), (68, 128), (69, 64), (70, 70),
                                    (71, 65), (72, 128), (55, 200), (55, 512), (55, 300)])
@pytest.mark.parametrize("Nn", [1000, 4096, 9992])
def test_keys_are_the_blocks_maxima(gpu, tile, M, Nn, monkeypatch):
    g = torch.Generator(device=gpu).manual_seed(tile + M + Nn)
    h = torch.randn(M, 512, device=gpu, generator=g).bfloat16()
    w = (torch.randn(Nn, 512, device=gpu, generator=g) * 0.05).bfloat16()
    plan = G.GemmPlan("dli", tile, 1)
    monkeypatch.setattr(G, "row_cut", lambda *a: 0)
    monkeypatch.setattr(G, "plan", lambda *a, **k: plan)
    lg, top = ops.head(h, w)
    assert torch.equal(lg, ops._gemm_native(h, w, "f32", plan=plan))
    keys, bw = top
    assert torch.equal(keys, block_keys(lg, bw))
    t = torch.full((M,), 0.8, device=gpu)
    args = (t, torch.full((M,), 20, device=gpu, dtype=torch.int32), torch.full((M,), 0.95, device=gpu),
            torch.arange(M, device=gpu, dtype=torch.int64))
    assert torch.equal(ops.sample(lg, *args, maxima=top), ops.sample(lg, *args))


def _rows(V, gpu):
    g = torch.Generator(device=gpu).manual_seed(V)
    x = torch.randn(14, V, device=gpu, generator=g) * 3
    x[1] = x[1].bfloat16().float()                         # ties
    x[2] = 1.5                                             # one value
    x[3] = torch.arange(V, device=gpu) * 1e-3              # rises: the large ones in a few blocks
    x[4] = -x[3]
    x[5] = -float("inf")
    x[5, V // 2] = 0.25
    x[6, ::7] = float("inf")
    x[7] = 0.0
    x[7, 1::2] = -0.0
    x[8] = -1.0
    x[8, V // 3:V // 3 + 2] = torch.tensor([-0.0, 0.0], device=gpu)
    x[9, V - 1] = 50.0
    x[10, 5] = float("nan")
    x[11, 5::9] = -float("nan")
    x[12] = -float("inf")
    x[13, :64] = 40.0                                      # a block of ties
    return x


# every way to sample, on rows with ties, infinities, zeros of both signs and NaNs: the tokens that
# the whole row gives. 24 columns: fewer blocks than the bound needs
@pytest.mark.gpu
@pytest.mark.parametrize("V,bw", [(32000, 64), (32000, 16), (128256, 128), (4096, 32), (1000, 80), (24, 16)])
def test_tokens_are_those_of_the_whole_row(gpu, V, bw):
    x = _rows(V, gpu)
    B = x.shape[0]
    keys = block_keys(x, bw)
    for T, K, P in ((0.0, 0, 1.0), (1.0, 1, 1.0), (0.8, 50, 0.95), (1.3, 2, 1.0), (0.7, 200, 0.9), (1.0, 256, 1.0),
                    (1.0, 300, 0.8), (0.9, 0, 0.9), (1.0, 0, 1.0)):
        a = (torch.full((B,), T, device=gpu), torch.full((B,), K, device=gpu, dtype=torch.int32),
             torch.full((B,), P, device=gpu))
        for s in range(3):
            seeds = torch.arange(B, device=gpu, dtype=torch.int64) + 100 * s
            # 9 rows and more sample in one pass over the row, as the blocks' sampler does where it must
            want = ops.sample(x, *a, seeds)
            got = ops.sample(x, *a, seeds, maxima=(keys, bw))
            assert torch.equal(got, want), (T, K, P, (got != want).nonzero().flatten().tolist())


@pytest.mark.gpu
def test_a_replaced_sampler_has_plain_logits(gpu, monkeypatch):
    from distributed_llm_inferencing_amd.models.model import TransformerLM

    class Forced(TransformerLM):
        def sample(self, logits, b, generator=None):
            logits[:, 7] = 1e9
            return super().sample(logits, b, generator)
    x = torch.zeros(3, 64, device=gpu)
    one = torch.ones(3, device=gpu)
    b = type("B", (), dict(temperature=one, top_k=(5 * one).int(), top_p=0.9 * one, seeds=one.long()))
    top = (block_keys(x, 16), 16)
    assert Forced.sample_head(object.__new__(Forced), x, b, top).tolist() == [7] * 3

    class Capped(TransformerLM):
        def head_logits(self, h):
            return torch.tanh(super().head_logits(h))
    m = object.__new__(Capped)
    m.params, m.cfg = {"lm_head": torch.ones(64, 512, device=gpu).bfloat16()}, type("C", (), dict(tie_embeddings=False))
    lg, none = m.head(torch.ones(2, 512, device=gpu).bfloat16())
    assert none is None and lg.max().item() == 1.0
    assert TransformerLM.sample_head(object.__new__(TransformerLM), x, b, (block_keys(x, 16), 16)).tolist() == [7] * 3


@pytest.mark.gpu
def test_refused_shapes(gpu):
    lib = N.require_native()
    assert lib.dli_gemm_head_block(56, 1, 4096) == 0 and lib.dli_gemm_head_block(22, 512, 4096) == 0
    assert lib.dli_gemm_head_block(63, 64, 4098) == 0 and lib.dli_gemm_head_block(30, 5, 4096) == 0
    h, w = torch.zeros(2, 512, device=gpu).bfloat16(), torch.zeros(64, 512, device=gpu).bfloat16()
    o, k = torch.zeros(2, 64, device=gpu), torch.zeros(2, 4, device=gpu, dtype=torch.int32)
    assert lib.dli_gemm_head(ops._p(h), 512, ops._p(w), 512, ops._p(o), 64, 2, 64, 512, 22, ops._p(k), ops._st())


# logits of another type (half the bytes that the kernel would read), candidates of a sliced head, keys of other
# rows, other blocks, another type or place
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_maxima_of_other_logits_are_refused(device):
    B, V, bw = 2, 64, 16
    x, one = torch.randn(B, V, device=device), torch.ones(B, device=device)
    keys = torch.zeros(B, V // bw, device=device, dtype=torch.int32)
    args = (one, (5 * one).int(), 0.9 * one, one.long())
    ids = torch.arange(V, device=device, dtype=torch.int32).expand(B, V)
    for logits, top, more in ((x.bfloat16(), (keys, bw), {}), (x.half(), (keys, bw), {}), (x, (keys, bw), dict(ids=ids)),
                              (x, (keys[:1], bw), {}), (x, (keys, 32), {}), (x, (keys, 0), {}), (x, (keys.long(), bw), {}),
                              (x, (keys.t().contiguous().t(), bw), {}), (x.t().contiguous().t(), (keys, bw), {})):
        with pytest.raises(ValueError):
            ops.sample(logits, *args, maxima=top, **more)
    if device != "cpu":
        with pytest.raises(ValueError):
            ops.sample(x, *args, maxima=(keys.cpu(), bw))


# operands that do not match never reach the tuned head, whose kernel takes their word for it
def test_a_mismatched_head_weight_is_left_to_the_general_product(monkeypatch):
    from distributed_llm_inferencing_amd.models import hybrid
    calls = []
    monkeypatch.setattr(hybrid.ops, "head", lambda h, w: calls.append("tuned"))
    monkeypatch.setattr(hybrid.H, "linear_any", lambda h, w, **k: calls.append("general"))
    m = object.__new__(hybrid.HybridLM)
    h = torch.zeros(2, 128).bfloat16()
    for w, want in ((torch.zeros(64, 128).bfloat16(), "tuned"), (torch.zeros(64, 128), "general"),
                    (torch.zeros(64, 64).bfloat16(), "general"), (torch.zeros(64, 256).bfloat16(), "general"),
                    (torch.zeros(128, 64).bfloat16().t(), "general")):
        m.params = {"lm_head": w}
        m.head(h)
        assert calls.pop() == want and not calls
