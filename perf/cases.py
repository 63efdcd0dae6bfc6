"""Workloads of the serving engine, for timing and for comparing one revision's outputs with another's.

A case is one step of an ``LLMEngine`` (prefill of whole prompts, decode of a running batch, or a
mixed step) for one model family at real layer sizes and four layers, random weights. ``prepare``
does what a serving process does before the step: it keeps the weights, admits the requests and runs
the steps that come before; ``run`` is the step itself through the engine's runner (metadata upload,
model, LM head, sampler; decode steps replay the captured graph). Outputs are the logits of every
sequence's last token and the caches and recurrent states that the step writes. The sampled tokens
are left out: one of two nearly equal logits wins by rounding.
"""
from __future__ import annotations

import functools
import math
import random
import zlib

import numpy as np
import torch

from distributed_llm_inferencing_amd.engine import SamplingParams
from distributed_llm_inferencing_amd.engine.llm_engine import LLMEngine
from distributed_llm_inferencing_amd.models import model_class, weights
from distributed_llm_inferencing_amd.models.configs import LayerSpec, get_config, hybrid_config

DEVICE = "cuda:0"
LAYERS = 4
BLOCK = 16
BUCKETS = (1, 2, 4, 8, 16, 24, 32, 48, 64, 96, 128, 160, 192, 256, 320, 384, 448, 512)


# ----------------------------------------------------------------------------- the cases
def listed():
    return [
        # one user, a short chat turn: the batch-1 step whose latency a single user sees
        _case("llama-decode-1", "llama", "decode", 1, 75, 75),
        # the throughput benchmark's running batch: 512 requests of at most 100 tokens
        _case("llama-decode-512", "llama", "decode", 512, 33, 99),
        # long conversations and documents beside short ones, few at a time
        _case("llama-decode-ragged", "llama", "decode", 24, 500, 8000),
        # the throughput benchmark's admission wave: 512 prompts of 32 tokens
        _case("llama-prefill-wave", "llama", "prefill", 512, 32, 32),
        # one document near the model's context length: time to first token
        _case("llama-prefill-long", "llama", "prefill", 1, 7993, 7993),
        # a busy server: a running batch with the second 2048-token portion of a long prompt
        _case("llama-mixed", "llama", "mixed", 64, 100, 1500, prompt=6001, chunk=2048),
        # routed experts: a mid-sized running batch, and a wave of ragged prompts
        _case("mixtral-decode-64", "mixtral", "decode", 64, 200, 1900),
        _case("mixtral-prefill", "mixtral", "prefill", 8, 300, 2000),
        # the layer-list designs at their benchmark's sizes (4 x 2048 prompts, batch 64 at ~1000
        # tokens), and ragged prompts of odd lengths
        _case("buborax-prefill", "buborax", "prefill", 4, 2048, 2048),
        _case("risutar-prefill", "risutar", "prefill", 6, 301, 3000),
        _case("lapunex-prefill", "lapunex", "prefill", 5, 900, 2601),
        _case("lapunex-decode-64", "lapunex", "decode", 64, 984, 984),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    model = rng.choice(("llama", "llama", "llama", "mixtral", "buborax", "risutar", "lapunex"))
    kind = rng.choice(("prefill", "decode", "mixed") if model == "llama" else ("prefill", "decode"))
    if kind == "prefill":
        seqs = log(1, 256)
        longest = log(33, min(8000, 9000 // seqs)) if seqs <= 256 else 33
        c = _case(None, model, kind, seqs, max(17, longest // rng.choice((1, 2, 6))), longest)
    elif kind == "decode":
        seqs = log(1, 512 if model in ("llama", "mixtral") else 96)
        longest = log(48, min(8000, 50000 // seqs))
        c = _case(None, model, kind, seqs, max(33, longest // rng.choice((1, 3, 12))), longest)
    else:
        seqs, longest, chunk = log(4, 256), 0, rng.choice((512, 1024, 2048))
        longest = log(48, min(4000, 50000 // seqs))
        c = _case(None, model, kind, seqs, max(33, longest // 4), longest, prompt=2 * chunk + log(16, 4000),
                  chunk=chunk)
    c["shortest"] = min(c["shortest"], c["longest"])
    return c


def _case(name, model, kind, seqs, shortest, longest, **more):
    c = {"name": name, "model": model, "kind": kind, "seqs": seqs, "shortest": shortest,
         "longest": longest, **more}
    if name is None:
        del c["name"]
    return c


def _lengths(case):
    """Context lengths of the step's sequences, its new tokens included, spread evenly over their
    logarithm in an order of no meaning; a mixed step's last one is the long prompt's."""
    n, a, b = case["seqs"], case["shortest"], case["longest"]
    ls = [int(round(a * (b / a) ** (i / max(1, n - 1)))) for i in range(n)] if a < b else [b] * n
    random.Random(n).shuffle(ls)
    return ls + ([2 * case["chunk"]] if case["kind"] == "mixed" else [])


def _new_tokens(case):
    ls = _lengths(case)
    if case["kind"] == "prefill":
        return ls
    return [1] * case["seqs"] + ([case["chunk"]] if case["kind"] == "mixed" else [])


# ----------------------------------------------------------------------------- models
D, FF, VOCAB, HEADS, GROUPS, HD = 4096, 14336, 32000, 32, 8, 128
LATENT = dict(heads=HEADS, kv_heads=1, dim=HD, vdim=HD, scale=(HD + 64) ** -0.5, rot_dim=64,
              kv_rank=512, rot_dims=64, rot_base=10000.0)
DECAYS = tuple(1.0 - 2.0 ** (-1.0 - 7.0 * h / (HEADS - 1)) for h in range(HEADS))
BIGRAM = (65521, 31, 17)
CAP, STREAMS, ALPHA, SIDE, TAU, RANK, QRANK = 15.0, 3, 2.0, 32, 8.0, 32, 1536
YARN = (4.0, 8192.0, 16.0, 2.0)


@functools.lru_cache(maxsize=None)
def _config(model):
    if model == "llama":
        return get_config("llama3-8b", LAYERS)
    if model == "mixtral":
        return get_config("mixtral-8x7b", LAYERS)
    if model == "buborax":
        att = LayerSpec("attention", heads=HEADS, kv_heads=GROUPS, dim=HD, vdim=HD, window=1024,
                        scale=HD ** -0.5, ff=FF)
        return hybrid_config("buborax-4096", D, VOCAB, (
            att, LayerSpec("hgrn2", heads=HEADS, dim=HD, vdim=HD, ff=FF),
            LayerSpec("latent_attention", window=1024, ff=FF, **LATENT), att),
            loop=(1, 3, 2), norm_groups=4, residual_mult=0.7)
    ff = dict(ff=FF, ff_kind="gated_silu")
    if model == "risutar":
        gla = LayerSpec("gla", heads=HEADS, dim=HD, vdim=HD, tau=TAU, decay_rank=RANK, **ff)
        lat = dict(window=1 << 30, q_rank=QRANK, head_gate=True, rot_half=True, **LATENT, **ff)
        return hybrid_config("risutar-4096", D, VOCAB, (
            gla, LayerSpec("latent_attention", **lat), LayerSpec("latent_attention", kv_from=1, **lat),
            gla), arch="risutar", max_position=1 << 15, norm_eps=1e-6, post_norm=True,
            postln_alpha=ALPHA, bigram=BIGRAM, side_dim=SIDE)
    light = LayerSpec("lightning", heads=HEADS, dim=HD, vdim=HD, decays=DECAYS, **ff)
    par = LayerSpec("parallel", heads=HEADS, kv_heads=GROUPS, dim=HD, vdim=HD, left=LayerSpec(
        "sink_attention", heads=HEADS, kv_heads=GROUPS, dim=HD, vdim=HD, scale=HD ** -0.5, rot_dims=64,
        rot_base=10000.0, window=1 << 30, rot_scaling=YARN),
        right=LayerSpec("mlstm", heads=HEADS // 2, dim=HD, vdim=HD, gate_cap=CAP), left_scale=0.7,
        right_scale=0.6, **ff)
    return hybrid_config("lapunex-4096", D, VOCAB, (light, par, light, par), arch="lapunex",
                         max_position=1 << 15, norm_eps=1e-6, embed_scale=8.0, streams=STREAMS,
                         norm_offset=1.0, loop_entry=False)


class _Made(dict):
    """Checkpoint tensors by name: bf16 values that depend on the name alone."""

    def put(self, name, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        g = torch.Generator(device=DEVICE)
        g.manual_seed(zlib.crc32(name.encode()))
        t = torch.empty(shape, dtype=torch.bfloat16, device=DEVICE).normal_(mean, std, generator=g)
        self[name] = t.to(dtype)

    def mat(self, name, rows, cols, gain=1.0):
        self.put(name, (rows, cols), gain * cols ** -0.5)


def _checkpoint(model):
    """Trained-like scales: unit activations into every projection, each sublayer adding about half
    of what the stream holds, slow and fast decays."""
    m, cfg = _Made(), _config(model)
    V = cfg.vocab_size
    if model in ("llama", "mixtral"):
        m.put("model.embed_tokens.weight", (V, D))
        m.put("model.norm.weight", (D,), 0.1, 1.0)
        m.mat("lm_head.weight", V, D)
        for i in range(LAYERS):
            p = f"model.layers.{i}."
            for n in ("input_layernorm", "post_attention_layernorm"):
                m.put(f"{p}{n}.weight", (D,), 0.1, 1.0)
            for n, rows, gain in (("q", HEADS * HD, 1.0), ("k", GROUPS * HD, 1.0),
                                  ("v", GROUPS * HD, 1.0), ("o", D, 0.5)):
                m.mat(f"{p}self_attn.{n}_proj.weight", rows, HEADS * HD if n == "o" else D, gain)
            if model == "llama":
                _glu(m, p + "mlp.{}_proj.weight", ("gate", "up", "down"), 0.5)
                continue
            for e in range(cfg.num_experts):
                _glu(m, f"{p}block_sparse_moe.experts.{e}." + "{}.weight", ("w1", "w3", "w2"), 0.5)
        if model == "mixtral":
            # a trained router decides clearly: every token's embedding leans towards two experts
            E = cfg.num_experts
            m.put("toward", (E, D))
            lean = m.pop("toward")
            g = torch.Generator(device=DEVICE)
            g.manual_seed(1)
            two = torch.rand(V, E, device=DEVICE, generator=g).topk(2).indices
            m["model.embed_tokens.weight"] += 0.35 * lean[two[:, 0]] + 0.25 * lean[two[:, 1]]
            for i in range(LAYERS):
                m[f"model.layers.{i}.block_sparse_moe.gate.weight"] = lean * (4.0 / D)
        return m
    m.put("embed", (V, D), 0.125 if model == "lapunex" else 1.0)
    m.mat("head", V, D)
    m.put("final.norm", (D,), 0.1, 1.0 - cfg.norm_offset)
    if model == "buborax":
        m.mat("loop.in", D, 2 * D)
        m.put("loop.step", (cfg.loop[2], D), 0.3)
    if model == "risutar":
        m.put("final.norm.b", (D,), 0.1)
        m.put("bigram", (BIGRAM[0] + 1, D), 0.5)
        m.put("side.embed", (V, SIDE * LAYERS))
    for i, s in enumerate(cfg.layer_specs):
        a, x = f"l{i}.", f"l{i}.mix."
        for n in ("norm1", "norm2"):
            m.put(a + n, (D,), 0.1, 1.0 - cfg.norm_offset)
            if model == "risutar":
                m.put(f"{a}{n}.b", (D,), 0.1)
        _glu(m, a + "mlp.{}", ("gate", "up", "down"), 0.5)
        if model == "risutar":
            m.mat(a + "side.gate", SIDE, D)
            m.mat(a + "side.proj", D, SIDE)
            m.put(a + "side.norm", (D,), 0.05, 0.3)
        if model == "lapunex":
            for q in "12":
                m.put(f"{a}hc{q}.in", (STREAMS,), 0.1, 1.0 / STREAMS, torch.float32)
                m.put(f"{a}hc{q}.out", (STREAMS,), 0.2, 1.0, torch.float32)
                m.put(f"{a}hc{q}.mix", (STREAMS, STREAMS), 0.1, 0.0, torch.float32)
                m[f"{a}hc{q}.mix"] += torch.eye(STREAMS, device=DEVICE)
        for n, rows in _projections(s):
            m.mat(x + n, rows, {"uq": QRANK, "a2": RANK, "uk": s.kv_rank, "uv": s.kv_rank}.get(n, D))
        if s.kind == "parallel":
            m.put(x + "left.q.norm", (HEADS * HD,), 0.1, 1.0)
            m.put(x + "left.k.norm", (GROUPS * HD,), 0.1, 1.0)
            m.put(x + "left.sink", (HEADS,), 1.0, 0.0, torch.float32)
            m.put(x + "right.norm", (HEADS // 2 * HD,), 0.1, 1.0)
            m.put(x + "right.i.b", (HEADS // 2,), 0.5, -1.0, torch.float32)
            m.put(x + "right.f.b", (HEADS // 2,), 1.0, 3.0, torch.float32)
            m.mat(x + "left.o", D, HEADS * HD, 0.5)
            m.mat(x + "right.o", D, HEADS // 2 * HD, 0.5)
            continue
        m.mat(x + "o", D, HEADS * HD, 0.5)
        if s.kind == "attention":
            m.put(x + "q.norm", (HD,), 0.2, 1.0)
            m.put(x + "k.norm", (HD,), 0.2, 1.0)
            m.put(x + "talk", (HEADS, HEADS), 0.2, 0.0, torch.float32)
            m[x + "talk"] += torch.eye(HEADS, device=DEVICE)
        elif s.kind == "hgrn2":
            m.put(x + "f.b", (HEADS * HD,), 1.0)
            m.put(x + "lower", (HEADS * HD,), 1.0)
            m[x + "lower"] = (0.95 * torch.sigmoid(m[x + "lower"].float())).to(torch.bfloat16)
            m.put(x + "norm", (HD,), 0.2, 1.0)
        elif s.kind == "latent_attention":
            if s.kv_from < 0:
                m.put(x + "dkv.norm", (s.kv_rank,), 0.1, 1.0)
            if s.q_rank:
                m.put(x + "dq.norm", (QRANK,), 0.1, 1.0)
        elif s.kind == "gla":
            m.put(x + "a2.b", (HEADS * HD,), 2.0, 1.0)
            m.put(x + "norm", (HD,), 0.2, 1.0)
        elif s.kind == "lightning":
            m.put(x + "norm", (HEADS * HD,), 0.1, 1.0)
    return m


def _glu(m, pattern, names, gain):
    for n, rows, cols, g in ((names[0], FF, D, 1.0), (names[1], FF, D, 1.0), (names[2], D, FF, gain)):
        m.mat(pattern.format(n), rows, cols, g)


def _projections(s):
    """(checkpoint name, rows) of a design layer's projections but the output's."""
    q, kv = HEADS * HD, GROUPS * HD
    if s.kind == "attention":
        return [("q", q), ("k", kv), ("g", q)]
    if s.kind == "hgrn2":
        return [("q", q), ("f", q), ("v", q)]
    if s.kind == "gla":
        return [("q", q), ("k", q), ("v", q), ("g", q), ("a1", RANK), ("a2", q)]
    if s.kind == "lightning":
        return [("q", q), ("k", q), ("v", q), ("g", q)]
    if s.kind == "parallel":
        return ([("left." + n, r) for n, r in (("q", q), ("k", kv), ("v", kv), ("g", HEADS))]
                + [("right." + n, q // 2) for n in "qkvg"] + [("right.i", HEADS // 2), ("right.f", HEADS // 2)])
    up = [("uk", HEADS * HD), ("uv", HEADS * HD)]
    if s.q_rank:
        return ([("dq", QRANK), ("uq", HEADS * (HD + s.rot_dim)), ("g", HEADS)] + up
                + ([("dkv", s.kv_rank + s.rot_dim)] if s.kv_from < 0 else []))
    return [("q", HEADS * (HD + s.rot_dim)), ("dkv", s.kv_rank + s.rot_dim)] + up


@functools.lru_cache(maxsize=None)
def _model(model):
    """The model with its weights, which a serving process loads once. It keeps the logits that its
    step function made beside the tokens that it samples from them."""
    cfg, sd = _config(model), _checkpoint(model)
    read = {"buborax": weights.from_buborax_state_dict, "risutar": weights.from_risutar_state_dict,
            "lapunex": weights.from_lapunex_state_dict}.get(model, weights.from_hf_state_dict)
    params = read(cfg, sd)
    if model == "risutar":
        cfg, params = params
    lm = model_class(cfg)(cfg, params, device=DEVICE)
    forward = lm.forward

    def keeping_logits(batch, caches, hidden=None, return_logits=False):
        tokens, lm.step_logits = forward(batch, caches, hidden=hidden, return_logits=True)
        return (tokens, lm.step_logits) if return_logits else tokens
    lm.forward = keeping_logits
    return lm


# ----------------------------------------------------------------------------- a pass
def _tokens(case, seed):
    """Every sequence's token ids up to and with the step's new ones."""
    rng = np.random.default_rng(seed)
    ls = _lengths(case)
    if case["kind"] == "mixed":
        ls = ls[:-1] + [max(case["prompt"], ls[-1])]
    return [rng.integers(0, _config(case["model"]).vocab_size, n) for n in ls]


def prepare(case, seed):
    lm, ids, ls = _model(case["model"]), _tokens(case, seed), _lengths(case)
    kind, n = case["kind"], case["seqs"]
    # decode rows stand one token (a mixed step's: one more, for the portion before) past the prompt
    behind = {"prefill": 0, "decode": 1, "mixed": 2}[kind]
    total = sum(len(t) for t in ids) + 16 * len(ids)
    eng = LLMEngine(lm.cfg, device=DEVICE, lm=lm, max_batch=next(b for b in BUCKETS if b >= len(ids)),
                    max_model_len=max(2048, max(len(t) for t in ids) + 16), block_size=BLOCK,
                    num_blocks=total // BLOCK + 2 * len(ids) + 8, max_prefill_tokens=total,
                    use_graphs=kind == "decode", lookahead=False)
    more = SamplingParams(max_new_tokens=16, ignore_eos=True, seed=7)
    for t, length in zip(ids[:n], ls):
        eng.add_request(t[:length - behind].tolist(), more)

    def plan():
        meta = eng.plan_step()      # its input ids, but the dictated ones where it would feed samples
        starts = np.cumsum(meta.seq_lens) - meta.seq_lens
        rows = np.repeat(np.asarray(meta.seq_ids), meta.seq_lens)
        assert len(rows) == len(meta.positions) and len(starts) == len(meta.seq_ids)
        meta.input_ids = np.asarray([ids[s][p] for s, p in zip(rows, meta.positions)], np.int32)
        return meta

    meta = plan()
    if kind != "prefill":
        eng.finish_step(meta)
        if kind == "mixed":
            eng.scheduler.max_prefill_tokens = case["chunk"]
            eng.scheduler.admit_window_s = 0.0      # the prompt has waited its turn
            eng.add_request(ids[-1].tolist(), more)
            eng.finish_step(plan())
        meta = plan()
    assert len(meta.seq_ids) == len(ls) and meta.num_tokens == sum(_new_tokens(case))
    state = {"runner": eng.runner, "meta": meta, "lm": lm, "logits": None, "cache": _cache(eng.kv), "engine": eng}
    if kind == "decode":
        eng.runner.capture([next(b for b in BUCKETS if b >= n)])
        state["logits"] = lm.step_logits[:n]
    return state


def _cache(kv):
    if hasattr(kv, "entries"):
        return list({t.data_ptr(): t for e in kv.entries for t in e}.values())
    return [kv.k, kv.v]


def run(state):
    state["runner"].run(state["meta"])
    logits = state["logits"]
    return {"logits": state["lm"].step_logits if logits is None else logits, "cache": state["cache"]}


# ----------------------------------------------------------------------------- what a pass needs
def work(case):
    cfg, ls, new = _config(case["model"]), _lengths(case), _new_tokens(case)
    T, S = sum(new), len(new)
    pairs = lambda w: sum(sum(min(p + 1, w) for p in range(l - n, l)) for l, n in zip(ls, new))  # noqa: E731
    reach = lambda w: sum(min(l, n + w) for l, n in zip(ls, new))  # noqa: E731
    bytes_ = T * D * 2 + S * cfg.vocab_size * 4 + cfg.vocab_size * D * 2
    flops = 2.0 * S * D * cfg.vocab_size
    glu, everything = 3 * D * FF, 1 << 40
    if case["model"] in ("llama", "mixtral"):
        top, E = (cfg.top_k_experts, cfg.num_experts) if cfg.is_moe else (1, 1)
        att = (2 * HEADS + 2 * GROUPS) * HD * D
        bytes_ += LAYERS * (2 * (att + min(E, T * top) * glu) + 4 * GROUPS * HD * reach(everything))
        flops += LAYERS * (2.0 * T * (att + top * glu) + 4.0 * HEADS * HD * pairs(everything))
        return {"bytes": bytes_, "flops": flops}
    if cfg.loop:
        bytes_ += 4 * D * D
        flops += cfg.loop[2] * 4.0 * T * D * D
    for li, _, _ in cfg.layer_runs():
        s = cfg.layer_specs[li]
        mats = [r * {"uq": QRANK, "a2": RANK, "uk": s.kv_rank, "uv": s.kv_rank}.get(n, D)
                for n, r in _projections(s)] + [HEADS * HD * D * (1.5 if s.kind == "parallel" else 1)]
        flops += 2.0 * T * (sum(mats) + glu)
        bytes_ += 2 * (sum(mats) + glu)
        w = min(s.window, everything) if s.kind in ("attention", "latent_attention") else everything
        if s.kind in ("hgrn2", "gla", "lightning", "parallel"):
            state = (HEADS // 2 if s.kind == "parallel" else HEADS) * HD * HD
            flops += 4.0 * T * state
            bytes_ += S * state * 4 * (1 if case["kind"] == "prefill" else 2)
        if s.kind in ("attention", "parallel"):
            flops += (4.0 * HD + (2.0 * HEADS if s.kind == "attention" else 0)) * HEADS * pairs(w)
            bytes_ += 4 * GROUPS * HD * reach(w)
        elif s.kind == "latent_attention":
            flops += 2.0 * (2 * HD + s.rot_dim) * HEADS * pairs(w)
            bytes_ += 2 * (s.kv_rank + s.rot_dim) * reach(w)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """bf16 operands and caches through four to six layers with fp32 sums, norms and states: four
    times the measured distance from 64 bits (0.006 where the residual stream is bf16, 0.0028 where
    it is fp32); the largest differences of a few million values lie at six times the mean ones."""
    return {"rel": 0.024, "max": 0.2} if case["model"] in ("llama", "mixtral") else {"rel": 0.012, "max": 0.1}


# ----------------------------------------------------------------------------- in 64 bits
def exact(case, seed):
    sd, cfg, ls = _checkpoint(case["model"]), _config(case["model"]), _lengths(case)
    ids = [torch.from_numpy(t[:n]).to(DEVICE) for t, n in zip(_tokens(case, seed), ls)]
    with torch.no_grad():
        f = _Exact(sd, cfg, ids)
        x = {"llama": f.transformer, "mixtral": f.transformer, "buborax": f.buborax,
             "risutar": f.risutar, "lapunex": f.lapunex}[case["model"]]()
    return {"logits": x, "cache": None}


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


class _Exact:
    """The models over whole sequences in float64, packed rows [T, D]; logits of the last rows."""

    def __init__(self, sd, cfg, ids):
        self.sd, self.cfg, self.eps = sd, cfg, cfg.norm_eps
        self.n = [len(t) for t in ids]
        self.at = np.concatenate([[0], np.cumsum(self.n)]).tolist()
        self.tok = torch.cat(ids)
        self.prev = torch.cat([torch.cat([t.new_tensor([-1]), t[:-1]]) for t in ids])
        self.pos = torch.cat([torch.arange(len(t), device=DEVICE) for t in ids]).double()
        self.last = torch.tensor([b - 1 for b in self.at[1:]], device=DEVICE)

    def w(self, name):
        return self.sd[name].double()

    def lin(self, x, name):
        w = self.w(name).t()
        return torch.cat([c @ w for c in x.split(8192)])

    def glu(self, x, pattern, names, act):
        g, u, d = (self.w(pattern.format(n)).t() for n in names)
        return torch.cat([(act(c @ g) * (c @ u)) @ d for c in x.split(4096)]) if len(x) else x

    def attend(self, q, k, v, scale, window=1 << 40, slopes=None, talk=None, sink=None):
        """q [T, H, d], k [T, Gk, d], v [T, G, dv] -> [T, H, dv], every sequence by itself."""
        H = q.shape[1]
        out = []
        for a, b in zip(self.at, self.at[1:]):
            kk = k[a:b].repeat_interleave(H // k.shape[1], 1).permute(1, 2, 0).contiguous()
            vv = v[a:b].repeat_interleave(H // v.shape[1], 1).permute(1, 0, 2).contiguous()
            for r in range(a, b, 1024):
                e = min(b, r + 1024)
                lo = max(0, r - a - min(window, 1 << 30) + 1)
                s = (q[r:e].permute(1, 0, 2) @ kk[:, :, lo:e - a]) * scale
                far = self.pos[r:e, None] - self.pos[None, a + lo:e]
                if slopes is not None:
                    s -= slopes[:, None, None] * far
                s.masked_fill_(((far < 0) | (far >= window))[None], -math.inf)
                if sink is not None:
                    s = torch.cat([s, sink[:, None, None].expand(H, e - r, 1)], 2)
                p = s.softmax(-1)
                p = p[:, :, :-1] if sink is not None else p
                if talk is not None:
                    p = (talk @ p.reshape(H, -1)).view_as(p)
                out.append((p @ vv[:, lo:e - a]).permute(1, 0, 2))
        return torch.cat(out)

    def walk(self, step, *rows):
        """Applies ``step(t, *rows at t)`` over time to all sequences at once; rows [T, ...]."""
        S, n = len(self.n), max(self.n)
        idx = torch.zeros(S, n, dtype=torch.long, device=DEVICE)
        for s, (a, b) in enumerate(zip(self.at, self.at[1:])):
            idx[s] = a + torch.arange(n, device=DEVICE).clamp(max=b - a - 1)
        got = torch.stack([step(*(r[idx[:, t]] for r in rows)) for t in range(n)], 1)
        return torch.cat([got[s, :m] for s, m in enumerate(self.n)])

    def rotate(self, x, freq, adjacent=False, factor=1.0):
        n = 2 * len(freq)
        ang = self.pos[:, None] * freq[None]
        c, s = (ang.cos() * factor)[:, None], (ang.sin() * factor)[:, None]
        out = x.clone()
        i = (slice(0, n, 2), slice(1, n, 2)) if adjacent else (slice(0, n // 2), slice(n // 2, n))
        a, b = x[..., i[0]], x[..., i[1]]
        out[..., i[0]], out[..., i[1]] = a * c - b * s, b * c + a * s
        return out

    def freq(self, dims, base):
        return base ** (-2.0 * torch.arange(dims // 2, device=DEVICE, dtype=torch.float64) / dims)

    def heads(self, x, n=HEADS):
        return x.view(x.shape[0], n, -1)

    def transformer(self):
        cfg, x = self.cfg, self.w("model.embed_tokens.weight")[self.tok]
        f = self.freq(HD, cfg.rope_theta)
        for i in range(LAYERS):
            p = f"model.layers.{i}."
            h = _rms(x, self.eps) * self.w(p + "input_layernorm.weight")
            q, k, v = (self.heads(self.lin(h, f"{p}self_attn.{n}_proj.weight"), c)
                       for n, c in (("q", HEADS), ("k", GROUPS), ("v", GROUPS)))
            o = self.attend(self.rotate(q, f), self.rotate(k, f), v, HD ** -0.5)
            x = x + self.lin(o.reshape(len(x), -1), p + "self_attn.o_proj.weight")
            h = _rms(x, self.eps) * self.w(p + "post_attention_layernorm.weight")
            if not cfg.is_moe:
                x = x + self.glu(h, p + "mlp.{}_proj.weight", ("gate", "up", "down"), _silu)
                continue
            p += "block_sparse_moe."
            top = self.lin(h, p + "gate.weight").topk(cfg.top_k_experts)
            share = top.values.softmax(-1)
            for e in range(cfg.num_experts):
                r, j = (top.indices == e).nonzero(as_tuple=True)
                x = x.index_add(0, r, share[r, j, None] * self.glu(
                    h[r], f"{p}experts.{e}." + "{}.weight", ("w1", "w3", "w2"), _silu))
        h = _rms(x[self.last], self.eps) * self.w("model.norm.weight")
        return self.lin(h, "lm_head.weight")

    def group_norm(self, x, name):
        g = self.cfg.norm_groups
        return _rms(x.view(len(x), g, -1), self.eps).reshape_as(x) * self.w(name)

    def latent_kv(self, h, p, s):
        kv = self.lin(h, p + "dkv")
        c = _rms(kv[:, :s.kv_rank], self.eps) * self.w(p + "dkv.norm")
        return c, self.rotate(kv[:, None, s.kv_rank:], self.freq(s.rot_dims, s.rot_base), not s.rot_half)

    def latent(self, q, kv, p, s):
        c, kr = kv
        qr = self.rotate(q[..., HD:], self.freq(s.rot_dims, s.rot_base), not s.rot_half)
        k = torch.cat([self.heads(self.lin(c, p + "uk")), kr.expand(-1, HEADS, -1)], 2)
        return self.attend(torch.cat([q[..., :HD], qr], 2), k, self.heads(self.lin(c, p + "uv")),
                           s.scale, s.window)

    def buborax(self):
        cfg, x = self.cfg, self.w("embed")[self.tok]
        x0, m = x, cfg.residual_mult
        slopes = 2.0 ** (-8.0 * torch.arange(1, HEADS + 1, device=DEVICE, dtype=torch.float64) / HEADS)
        for li, t, first in cfg.layer_runs():
            s, p = cfg.layer_specs[li], f"l{li}.mix."
            if first:
                x = self.lin(torch.cat([x, x0], 1), "loop.in") + self.w("loop.step")[t]
            h = self.group_norm(x, f"l{li}.norm1")
            if s.kind == "attention":
                k = self.heads(self.lin(h, p + "k"), GROUPS)
                y = self.attend(_rms(self.heads(self.lin(h, p + "q")), self.eps) * self.w(p + "q.norm"),
                                _rms(k, self.eps) * self.w(p + "k.norm"), k, s.scale, s.window, slopes,
                                self.w(p + "talk"))
                y = y.reshape_as(h) * torch.sigmoid(self.lin(h, p + "g"))
            elif s.kind == "hgrn2":
                low = self.w(p + "lower")
                f = low + (1.0 - low) * torch.sigmoid(self.lin(h, p + "f") + self.w(p + "f.b"))
                f = self.heads(f)
                y = self.linear_attention(_silu(self.heads(self.lin(h, p + "q"))), 1.0 - f,
                                          self.heads(self.lin(h, p + "v")), f)
                y = _rms(y, self.eps) * self.w(p + "norm")
            else:
                y = self.latent(self.heads(self.lin(h, p + "q")), self.latent_kv(h, p, s), p, s)
            x = x + m * self.lin(y.reshape_as(h), p + "o")
            h = self.group_norm(x, f"l{li}.norm2")
            x = x + m * self.glu(h, f"l{li}.mlp." + "{}", ("gate", "up", "down"), _gelu)
        return self.lin(self.group_norm(x[self.last], "final.norm"), "head")

    def linear_attention(self, q, k, v, decay):
        """S = decay S + k v^T, o = S^T q over time; decay [T, H, d] or [T, H, 1]."""
        S = torch.zeros(len(self.n), q.shape[1], HD, HD, dtype=torch.float64, device=DEVICE)

        def step(q, k, v, a):
            S.mul_(a[..., None]).addcmul_(k[..., None], v[..., None, :])
            return (q[..., None, :] @ S)[..., 0, :]
        return self.walk(step, q, k, v, decay)

    def risutar(self):
        cfg, eps = self.cfg, self.eps

        def ln(x, n):
            x = x - x.mean(-1, keepdim=True)
            return _rms(x, eps) * self.w(n) + self.w(n + ".b")
        row = (self.prev * BIGRAM[1] + self.tok * BIGRAM[2]) % BIGRAM[0]
        x = self.w("embed")[self.tok] + self.w("bigram")[torch.where(self.prev < 0, BIGRAM[0], row)]
        kv = None
        for li, s in enumerate(cfg.layer_specs):
            a, p = f"l{li}.", f"l{li}.mix."
            if s.kind == "gla":
                z = self.lin(self.lin(x, p + "a1"), p + "a2") + self.w(p + "a2.b")
                y = self.linear_attention(self.heads(self.lin(x, p + "q")) * HD ** -0.5,
                                          self.heads(self.lin(x, p + "k")), self.heads(self.lin(x, p + "v")),
                                          self.heads(torch.sigmoid(z) ** (1.0 / TAU)))
                y = (_rms(y, eps) * self.w(p + "norm")).reshape_as(x) * _silu(self.lin(x, p + "g"))
            else:
                kv = self.latent_kv(x, p, s) if s.kv_from < 0 else kv
                q = self.lin(_rms(self.lin(x, p + "dq"), eps) * self.w(p + "dq.norm"), p + "uq")
                y = self.latent(self.heads(q), kv, p, s) * torch.sigmoid(self.lin(x, p + "g"))[..., None]
            x = ln(ALPHA * x + self.lin(y.reshape_as(x), p + "o"), a + "norm1")
            x = ln(ALPHA * x + self.glu(x, a + "mlp.{}", ("gate", "up", "down"), _silu), a + "norm2")
            e = self.w("side.embed")[self.tok][:, li * SIDE:(li + 1) * SIDE]
            y = self.lin(_gelu(self.lin(x, a + "side.gate")) * e, a + "side.proj")
            x = x + _rms(y, eps) * self.w(a + "side.norm")
        return self.lin(ln(x[self.last], "final.norm"), "head")

    def lapunex(self):
        cfg, eps = self.cfg, self.eps
        norm = lambda x, n: _rms(x, eps) * (1.0 + self.w(n))  # noqa: E731
        xs = [self.w("embed")[self.tok] * cfg.embed_scale] * STREAMS
        for li, s in enumerate(cfg.layer_specs):
            a, p = f"l{li}.", f"l{li}.mix."
            for q in "12":
                read, out, mix = (self.w(f"{a}hc{q}.{n}").tolist() for n in ("in", "out", "mix"))
                h = norm(sum(c * x for c, x in zip(read, xs)), f"{a}norm{q}")
                if q == "2":
                    y = self.glu(h, a + "mlp.{}", ("gate", "up", "down"), _silu)
                elif s.kind == "lightning":
                    y = self.linear_attention(*(self.heads(_silu(self.lin(h, p + n))) for n in "qkv"),
                                              torch.tensor(DECAYS, device=DEVICE, dtype=torch.float64)
                                              .view(1, HEADS, 1).expand(len(h), -1, 1))
                    y = _rms(y.reshape_as(h), eps) * self.w(p + "norm") * torch.sigmoid(self.lin(h, p + "g"))
                    y = self.lin(y, p + "o")
                else:
                    y = (s.left_scale * self.lin(self.sink_attention(h, p + "left.", s.left), p + "left.o")
                         + s.right_scale * self.lin(self.memory(h, p + "right."), p + "right.o"))
                xs = [sum(mix[i][j] * xs[i] for i in range(STREAMS)) + out[j] * y for j in range(STREAMS)]
        return self.lin(norm(sum(xs)[self.last], "final.norm"), "head")

    def sink_attention(self, h, p, s):
        factor, orig, fast, slow = YARN
        dims, base = s.rot_dims, s.rot_base
        f = self.freq(dims, base)
        at = lambda turns: dims * math.log(orig / (2 * math.pi * turns)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(at(fast)), 0), min(math.ceil(at(slow)), dims - 1)
        ramp = ((torch.arange(dims // 2, device=DEVICE, dtype=torch.float64) - lo) / max(hi - lo, 1e-3)).clamp(0, 1)
        f, grow = f / factor * ramp + f * (1 - ramp), 0.1 * math.log(factor) + 1.0
        q, k = (self.rotate(self.heads(_rms(self.lin(h, p + n), self.eps) * self.w(f"{p}{n}.norm"), c), f,
                            False, grow) for n, c in (("q", HEADS), ("k", GROUPS)))
        o = self.attend(q, k, self.heads(self.lin(h, p + "v"), GROUPS), s.scale, sink=self.w(p + "sink"))
        return (o * torch.sigmoid(self.lin(h, p + "g"))[..., None]).reshape(len(h), -1)

    def memory(self, h, p):
        n = HEADS // 2
        q, k, v = (self.heads(self.lin(h, p + c), n) for c in "qkv")
        i, f = (CAP * torch.tanh((self.lin(h, p + c) + self.w(f"{p}{c}.b")) / CAP) for c in "if")
        f = torch.nn.functional.logsigmoid(f)
        S = torch.zeros(len(self.n), n, HD, HD + 1, dtype=torch.float64, device=DEVICE)
        m = torch.zeros(len(self.n), n, dtype=torch.float64, device=DEVICE)

        def step(q, k, v, i, f):
            top = torch.maximum(f + m, i)
            S.mul_((f + m - top).exp()[..., None, None])
            S.addcmul_((k * (i - top).exp()[..., None])[..., None], v[..., None, :])
            m.copy_(top)
            r = (q[..., None, :] @ S)[..., 0, :]
            return r[..., :HD] / (torch.maximum(r[..., HD:].abs(), (-top).exp()[..., None]) + 1e-6)
        one = torch.ones(len(h), n, 1, dtype=torch.float64, device=DEVICE)
        y = _rms(self.walk(step, q * HD ** -0.5, k, torch.cat([v, one], 2), i, f), self.eps)
        return y.reshape(len(h), -1) * self.w(p + "norm") * torch.sigmoid(self.lin(h, p + "g"))
