"""Automatic prefix caching:
full KV blocks are published under chain hashes of their tokens; a later request with the
same prefix maps those blocks (refcounted) and prefills only its remaining tokens as a chunk
over the paged cache. Outputs must be token-identical to an engine without the cache, also
when cached blocks are evicted under memory pressure and after preemption."""
import numpy as np
import torch

from distributed_llm_inferencing_amd.engine import SamplingParams
from distributed_llm_inferencing_amd.engine.llm_engine import LLMEngine
from distributed_llm_inferencing_amd.runtime import BlockManager

SYS = list(range(300, 300 + 45))                  # shared "system prompt" (2 full blocks + 13)


def _engine(cache: bool, **kw):
    kw.setdefault("num_blocks", 256)
    e = LLMEngine("llama-tiny", device="cpu", dtype=torch.float32, max_batch=8,
                  max_model_len=256, **kw)
    e.scheduler.prefix_caching = cache
    return e


def test_block_manager_refcounts_and_eviction():
    bm = BlockManager(6, 4)
    assert bm.ensure(1, 12)                       # 3 blocks
    h = np.array([11, 22, 33], np.uint64)
    assert bm.register_prefix(1, h) == 3
    assert bm.num_cached == 3
    assert bm.match_prefix(2, h[:2]) == 2         # shares 2 blocks
    assert bm.table(2) == bm.table(1)[:2]
    assert bm.num_free == 3
    bm.free(1)                                    # block 3 cached + evictable, 1-2 still used
    assert bm.num_free == 4 and bm.num_cached == 3
    assert bm.ensure(3, 16)                       # takes the 3 free + evicts the cached one
    assert bm.num_cached == 2 and bm.num_free == 0
    bm.free(2)
    assert bm.num_free == 2                       # both back as evictable cached blocks
    assert bm.match_prefix(4, h) == 2             # the evicted third block is gone
    assert bm.prefix_hits == 4


def test_prefix_cache_token_identical():
    greedy = SamplingParams(max_length=80, do_sample=False, ignore_eos=True)
    sampled = SamplingParams(max_length=80, seed=11, ignore_eos=True)
    tails = [[1, 2, 3], [4, 5, 6, 7, 8, 9], list(range(40, 60)), [9] * 30]
    for sp in (greedy, sampled):
        ref = _engine(False)
        eng = _engine(True)
        want = [o.all_ids for o in ref.generate([SYS + [7]], sp)]
        want += [o.all_ids for o in ref.generate([SYS + t for t in tails], sp)]
        got = [o.all_ids for o in eng.generate([SYS + [7]], sp)]
        hits0 = eng.scheduler.prefix_hit_tokens
        got += [o.all_ids for o in eng.generate([SYS + t for t in tails], sp)]
        assert got == want
        assert hits0 == 0
        assert eng.scheduler.prefix_hit_tokens == 4 * 32       # 2 blocks x 4 requests
        assert ref.scheduler.prefix_hit_tokens == 0
        # the same prompt again: everything but the last (partial) block comes from cache
        again = eng.generate([SYS + tails[3]], sp)[0].all_ids
        assert again == want[-1]


def test_prefix_cache_under_pressure_and_preemption():
    sp = SamplingParams(max_length=110, do_sample=False, ignore_eos=True)
    prompts = [SYS + [i] * (3 + i) for i in range(7)]
    ref = _engine(False)
    want = [o.all_ids for o in ref.generate(prompts, sp)]
    eng = _engine(True, num_blocks=30, max_prefill_tokens=64)    # forces eviction/preemption
    got = []
    for i in range(0, 7, 2):                                      # arrivals in waves
        got += [o.all_ids for o in eng.generate(prompts[i:i + 2], sp)]
    assert got == want
    assert eng.scheduler.prefix_hit_tokens > 0
