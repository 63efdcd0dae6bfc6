"""T4 model-level tests on the GPU: HIP path vs fp32 reference, graph == eager."""
import pytest
import torch

from distributed_llm_inferencing_amd.engine import SamplingParams
from distributed_llm_inferencing_amd.engine.llm_engine import LLMEngine
from distributed_llm_inferencing_amd.models import get_config
from distributed_llm_inferencing_amd.models.weights import from_hf_state_dict

from hf_helpers import hf_model, our_last_logits

pytestmark = pytest.mark.gpu
IDS = [5, 17, 99, 3, 250, 7, 8, 1000, 42, 11, 600, 3, 3, 9]


@pytest.mark.parametrize("name", ["llama-tiny", "llama-tiny128", "gpt2-tiny", "mixtral-tiny"])
def test_gpu_logits_close_to_hf_fp32(gpu, name):
    torch.manual_seed(0)
    cfg = get_config(name)
    hm = hf_model(cfg)
    with torch.no_grad():
        ref = hm(torch.tensor([IDS])).logits[0, -1]
    params = from_hf_state_dict(cfg, hm.state_dict(), dtype=torch.bfloat16)
    params = {k: v.to(gpu) for k, v in params.items()}
    ours = our_last_logits(cfg, params, IDS, device=gpu).cpu()
    err = (ours - ref).abs().max().item()
    assert err < 0.05 * ref.abs().max().item() + 0.02, err
    assert ours.argmax() == ref.argmax() or (ref.topk(2).values.diff().abs() < 0.05).item()


@pytest.mark.parametrize("name", ["llama-tiny", "gpt2-tiny", "mixtral-tiny"])
def test_graph_decode_equals_eager(gpu, name, monkeypatch):
    # same GEMM plans on both sides (capture would otherwise autotune between the runs and
    # change split-K summation order)
    monkeypatch.setenv("DLI_GEMM_AUTOTUNE", "0")
    prompts = [IDS[:5], IDS[:9], IDS[3:14], IDS[:2]]
    sp = SamplingParams(max_length=40, temperature=0.8, top_k=50, top_p=0.95, seed=123,
                        ignore_eos=True)
    outs = []
    for graphs in (False, True):
        eng = LLMEngine(name, device="cuda", max_batch=8, max_model_len=128, num_blocks=64,
                        use_graphs=graphs, seed=3)
        outs.append([o.output_ids for o in eng.generate(prompts, sp)])
    assert outs[0] == outs[1]


def test_continuous_batching_is_batch_invariant(gpu):
    """A request's sampled tokens do not depend on what else is in the batch (per-request
    Philox seeds) — greedy and sampled."""
    eng = LLMEngine("llama-tiny", device="cuda", max_batch=16, max_model_len=128, num_blocks=128,
                    seed=4)
    sp = SamplingParams(max_length=30, seed=77, ignore_eos=True)
    alone = eng.generate([IDS[:6]], sp)[0].output_ids
    many = eng.generate([IDS[:3], IDS[:6], IDS[2:12], IDS[:6]], sp)
    assert many[1].output_ids == alone


@pytest.mark.parametrize("name", ["llama-tiny", "llama-tiny128"])
def test_batch1_deferred_norm_decode(gpu, name, monkeypatch):
    """Batch-1 decode on the reduce-free GEMV chain (O / down add into the residual in their
    epilogue, the next GEMV normalises in its prologue: models/model.py ``defer``) against
    the split-K + reduce path: every step's logits agree until the first differing token,
    and there the reference's top two logits are a near tie (the paths differ only in fp32
    summation order, so a token can flip only where two logits are within rounding)."""
    from distributed_llm_inferencing_amd import ops
    from distributed_llm_inferencing_amd.models.model import TransformerLM
    from distributed_llm_inferencing_amd.ops import gemm as G
    monkeypatch.setenv("DLI_GEMM_AUTOTUNE", "0")
    calls, logits = [], []
    real = ops.linear_residual
    monkeypatch.setattr(ops, "linear_residual", lambda *a, **k: (calls.append(1), real(*a, **k)))
    real_sample = TransformerLM.sample

    def spy(self, lg, b, generator=None):
        logits.append(lg.float().cpu())
        return real_sample(self, lg, b, generator=generator)
    monkeypatch.setattr(TransformerLM, "sample", spy)
    sp = SamplingParams(max_length=40, do_sample=False, ignore_eos=True)

    def run(defer, prompt):
        monkeypatch.setattr(G, "DEFER_NORM", defer)
        G.clear_plans()
        calls.clear(), logits.clear()
        eng = LLMEngine(name, device="cuda", max_batch=4, max_model_len=128, num_blocks=64,
                        seed=5, use_graphs=False)
        toks = eng.generate([prompt], sp)[0].output_ids
        assert bool(calls) == defer
        return toks, list(logits)
    for prompt in (IDS[:6], IDS[2:13]):
        t1, l1 = run(True, prompt)
        t0, l0 = run(False, prompt)
        assert len(t1) == len(t0) and len(l1) == len(l0) >= len(t0)
        n = next((i for i, (a, b) in enumerate(zip(t1, t0)) if a != b), len(t0))
        for i in range(min(n + 1, len(l0))):
            err = (l1[i] - l0[i]).abs().max().item()
            assert err < 0.02 * l0[i].abs().max().item() + 0.02, (i, err)
        if n < len(t0):
            top = l0[n][0].topk(2).values
            assert (top[0] - top[1]).item() < 0.02 * top[0].abs().item() + 0.02, (n, top)


def test_llama3_8b_smoke(gpu):
    eng = LLMEngine("llama3-8b", device="cuda", max_batch=4, max_model_len=256,
                    num_blocks=64, seed=0)
    outs = eng.generate(["The MI355X has 288 GB of HBM3E"], SamplingParams(max_length=40))
    assert len(outs[0].output_ids) == 40 - len(outs[0].prompt_ids)
    assert all(0 <= t < eng.cfg.vocab_size for t in outs[0].output_ids)


@pytest.mark.parametrize("n", [2, 4])
def test_loopback_pipeline_on_gpu_matches_single_stage(gpu, n):
    """All stages on cuda:0 (loopback transport): graphs on non-first stages, metadata
    round-trips, microbatch schedule — token-identical to the single-stage engine."""
    from distributed_llm_inferencing_amd.parallel.pipeline import LocalPipeline
    prompts = [IDS[:5], IDS[:9], IDS[3:14], IDS[:2], IDS[1:4]]
    for sp in (SamplingParams(max_length=30, do_sample=False, ignore_eos=True),
               SamplingParams(max_length=30, seed=9, ignore_eos=True)):
        ref = LLMEngine("llama-tiny", device="cuda", max_batch=8, max_model_len=128,
                        num_blocks=64, seed=2).generate(prompts, sp)
        pp = LocalPipeline("llama-tiny", n, device="cuda", max_batch=8, max_model_len=128,
                           num_blocks=64, seed=2)
        assert [o.all_ids for o in pp.generate(prompts, sp)] == [o.all_ids for o in ref]


@pytest.mark.parametrize("name", ["llama3-70b", "mixtral-8x7b"])
def test_real_shape_layers_close_to_hf_fp32(gpu, name):
    """Llama-3-70B and Mixtral-8x7B at their real layer shapes (hidden 8192 / 64 heads / GQA 8
    / FFN 28672; hidden 4096 / 8 experts x FFN 14336, top-2) and real vocabularies, 2 layers
    each: prefill logits of the HIP path vs HF transformers in fp32 on the same weights."""
    torch.manual_seed(0)
    cfg = get_config(name, num_layers=2)
    with torch.device(gpu):
        hm = hf_model(cfg)
    ids = IDS + [1234, 4321, 777]
    with torch.no_grad():
        ref = hm(torch.tensor([ids], device=gpu)).logits[0, -1].float().cpu()
        params = from_hf_state_dict(cfg, hm.state_dict(), dtype=torch.bfloat16)
    del hm
    params = {k: v.to(gpu) for k, v in params.items()}
    ours = our_last_logits(cfg, params, ids, device=gpu).float().cpu()
    err = (ours - ref).abs().max().item()
    assert err < 0.05 * ref.abs().max().item() + 0.02, err


@pytest.mark.parametrize("name", ["llama3-70b", "mixtral-8x7b"])
def test_real_shape_engine_decode(gpu, name, monkeypatch):
    """The serving path at real layer shapes (2 layers): continuous batching, graph-captured
    decode with autotuned GEMM plans and fused split-K reduces (N = 8192 rows for 70B),
    grouped expert GEMMs (Mixtral); graph decode equals eager decode token for token."""
    monkeypatch.setenv("DLI_GEMM_AUTOTUNE", "0")      # same GEMM plans on both sides
    prompts = [IDS[:5], IDS[:9], IDS[3:14]]
    sp = SamplingParams(max_length=24, seed=5, ignore_eos=True)
    outs = []
    for graphs in (False, True):
        eng = LLMEngine(name, device="cuda", max_batch=4, max_model_len=64, num_blocks=64,
                        num_layers=2, use_graphs=graphs, seed=1)
        outs.append([o.output_ids for o in eng.generate(prompts, sp)])
        assert all(len(o) == 24 - len(p) for o, p in zip(outs[-1], prompts))
        del eng
        torch.cuda.empty_cache()
    assert outs[0] == outs[1]


def _fp32_top2(eng, prefix):
    """Top-2 logits of the next token after ``prefix`` under the fp32 CPU reference of
    ``eng``'s weights (the same bf16 parameters, computed exactly in fp32)."""
    from distributed_llm_inferencing_amd.models.model import TransformerLM
    params = {k: v.float().cpu() for k, v in eng.model.params.items()}
    lm = TransformerLM(eng.cfg, params, device="cpu")
    ref = LLMEngine(eng.cfg, device="cpu", dtype=torch.float32, max_batch=1, max_model_len=128,
                    num_blocks=16, lm=lm)
    seen = []
    real = TransformerLM.sample

    def spy(self, lg, b, generator=None):
        seen.append(lg.float())
        return real(self, lg, b, generator=generator)
    TransformerLM.sample = spy
    try:
        ref.generate([prefix], SamplingParams(max_length=len(prefix) + 1, do_sample=False,
                                              ignore_eos=True))
    finally:
        TransformerLM.sample = real
    return seen[0][0].topk(2).values


def test_full_gpt2_on_tuned_plans(gpu, monkeypatch):
    """GPT-2 at its full size (biased products, K = 768, a head of 50257 columns): captured decode steps on
    timed plans give the tokens of eager steps on the fitted ones, but where the exact model is undecided
    (sums in another order: at the first differing token the fp32 reference's top two nearly tie)."""
    from distributed_llm_inferencing_amd.ops import gemm as G
    prompts, outs = [IDS[:5], IDS[:9], IDS[3:14]], []
    sp = SamplingParams(max_length=24, do_sample=False, ignore_eos=True)
    for tuned in (False, True):
        monkeypatch.setenv("DLI_GEMM_AUTOTUNE", "1" if tuned else "0")
        G.clear_plans()
        eng = LLMEngine("gpt2", device="cuda", max_batch=4, max_model_len=64, num_blocks=64, use_graphs=tuned,
                        seed=3)
        outs.append([o.all_ids for o in eng.generate(prompts, sp)])
        assert all(len(o) == 24 and max(o) < eng.cfg.vocab_size for o in outs[-1])
    assert any(k[3] == "bias_gelu" for k in G._tuned)
    G.clear_plans()
    for a, b in zip(*outs):
        if a != b:
            n = next(i for i, (x, y) in enumerate(zip(a, b)) if x != y)
            top = _fp32_top2(eng, a[:n])
            assert (top[0] - top[1]).item() < 0.01 * top[0].abs().item() + 0.01, (n, top)


def test_mixed_steps_token_identical_on_gpu(gpu, monkeypatch):
    """Prompts arriving while others decode: the mixed prefill+decode steps (decode rows on
    the decode kernel, prompt rows on the paged prefill kernel, one GEMM pass) give the
    tokens of the engine without mixed steps — greedy, graphs, lookahead and the reduce-free
    batch-1 chain (``DEFER_NORM``) all on, heuristic plans (no autotune), so the result does
    not depend on what an earlier test left in the plan cache. The two engines run the
    same math in different fp32 summation orders (a mixed step's decode rows take the MFMA
    tiles; a decode-only step of <= 4 rows the weight-streaming GEMVs), so a request may
    differ only where the exact model is undecided: at its first differing token the fp32
    reference's top-two logits are a near tie; and at most one request of the eight differs.
    (Token identity would hold only on plans that earlier tests had autotuned.)"""
    from distributed_llm_inferencing_amd.ops import gemm as G
    monkeypatch.setenv("DLI_GEMM_AUTOTUNE", "0")
    assert G.DEFER_NORM
    waves = [[IDS[:5], IDS[:9], IDS[3:14]], [IDS[:2], IDS[1:4]], [IDS[2:11]]]
    sp = SamplingParams(max_length=40, do_sample=False, ignore_eos=True)
    res, engs = [], []
    for mixed in (False, True):
        G.clear_plans()
        eng = LLMEngine("llama-tiny", device="cuda", max_batch=8, max_model_len=128,
                        num_blocks=64, seed=2, mixed_steps=mixed)
        outs, rids = {}, []
        for w, wave in enumerate(waves):
            rids += [eng.add_request(p, sp) for p in wave]
            for _ in range(2):
                for o in eng.step():
                    outs[o.request_id] = o
        while eng.has_work():
            for o in eng.step():
                outs[o.request_id] = o
        res.append([outs[r].all_ids for r in rids])
        assert (eng.stats.mixed_steps > 0) == mixed
        engs.append(eng)
    G.clear_plans()
    differ = [(a, b) for a, b in zip(res[0], res[1]) if a != b]
    assert len(differ) <= 1, len(differ)
    for a, b in differ:
        n = next(i for i, (x, y) in enumerate(zip(a, b)) if x != y)
        top = _fp32_top2(engs[0], a[:n])
        assert (top[0] - top[1]).item() < 0.01 * top[0].abs().item() + 0.01, (n, top)
