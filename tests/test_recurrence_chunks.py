"""Portions of the linear recurrences (ops.hybrid.hgrn2 / gla / lightning / mlstm) against a float64
walk: block edges (16 tokens), heads narrower than a tile, several column blocks, continued states,
padding rows, and decays so strong that a block's product leaves the range of fp32."""
import pytest
import torch
import torch.nn.functional as F

from distributed_llm_inferencing_amd.ops import hybrid as H

F64 = torch.float64


def rms(x, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def oracle(mode, proj, extra, state, nstate, lens, slots, first, heads, d, dv, eps):
    """(rows [T, heads * dv], new states) in float64."""
    proj, state = proj.to(F64), state.to(F64).clone()
    nstate = nstate.to(F64).clone() if nstate is not None else None
    ex = {k: (v.to(F64) if isinstance(v, torch.Tensor) else v) for k, v in extra.items()}
    out, t0, hd = torch.zeros(proj.shape[0], heads * dv, dtype=F64), 0, heads * d
    for s, n in enumerate(lens):
        p = proj[t0:t0 + n]
        q, k = p[:, :hd].view(n, heads, d), p[:, hd:2 * hd].view(n, heads, d)
        v = p[:, 2 * hd:2 * hd + heads * dv].view(n, heads, dv)
        g = p[:, 2 * hd + heads * dv:2 * hd + 2 * heads * dv].view(n, heads, dv)
        one = torch.ones(n, heads, 1, dtype=F64)
        if mode == "hgrn2":
            lo = ex["lower"].view(heads, d)
            a = lo + (1 - lo) * torch.sigmoid(k + ex["bias"].view(heads, d))
            q, k, b = F.silu(q), 1 - a, one
        elif mode == "gla":
            a = torch.exp(F.logsigmoid(ex["z"][t0:t0 + n] + ex["bias"]) / ex["tau"]).view(n, heads, d)
            q, b = q * d ** -0.5, one
        elif mode == "lightning":
            q, k, v = F.silu(q), F.silu(k), F.silu(v)
            a, b = ex["decays"].view(1, heads, 1) * one, one
        else:
            o0, cap = 2 * hd + 2 * heads * dv, ex["cap"]
            ig = cap * torch.tanh((p[:, o0:o0 + heads] + ex["if_b"][:heads]) / cap)
            fg = F.logsigmoid(cap * torch.tanh((p[:, o0 + heads:o0 + 2 * heads] + ex["if_b"][heads:]) / cap))
            q = q * d ** -0.5
        if slots[s] < 0:
            t0 += n
            continue
        S = state[slots[s]] * (0.0 if first[s] else 1.0)
        if mode == "mlstm":
            nv, m = nstate[slots[s]][:, :d] * (0.0 if first[s] else 1.0), nstate[slots[s]][:, d] * (0.0 if first[s] else 1.0)
        for t in range(n):
            if mode == "mlstm":
                m1 = torch.maximum(fg[t] + m, ig[t])
                at, bt, m = torch.exp(fg[t] + m - m1)[:, None], torch.exp(ig[t] - m1)[:, None], m1
                nv = at * nv + bt * k[t]
            else:
                at, bt = a[t], b[t]
            S = at[:, :, None] * S + (bt * k[t])[:, :, None] * v[t][:, None, :]
            o = torch.einsum("hdv,hd->hv", S, q[t])
            if mode == "mlstm":
                o = o / (torch.maximum((nv * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6)[:, None]
                o = rms(o, eps) * ex["norm"].view(heads, dv) * torch.sigmoid(g[t]) * ex["scale"]
            elif mode != "lightning":
                o = rms(o, eps) * ex["norm"] * (F.silu(g[t]) if mode == "gla" else 1.0)
            out[t0 + t] = o.reshape(-1)
        state[slots[s]] = S
        if mode == "mlstm":
            nstate[slots[s]] = torch.cat([nv, m[:, None]], 1)
        t0 += n
    return out, state, nstate


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["hgrn2", "gla", "lightning", "mlstm"])
@pytest.mark.parametrize("d,dv,strong", [(128, 128, False), (128, 128, True), (64, 48, True),
                                         (24, 20, False), (16, 128, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_portions_match_a_float64_walk(gpu, mode, d, dv, strong, dtype):
    if mode == "lightning" and dv == 48:
        dv = 200                                     # raw read-outs: more than one column block
    check(gpu, mode, d, dv, strong, dtype, [1, 16, 0, 17, 100, 33, 5], [4, 0, 1, 2, 5, 3, -1],
          [0, 1, 0, 0, 1, 0, 0])


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["hgrn2", "gla", "lightning", "mlstm"])
@pytest.mark.parametrize("d,dv,strong", [(128, 128, False), (32, 48, True)])
@pytest.mark.parametrize("lens,slots,first", [
    # segments of 144 tokens: last ones of 1 and 16 tokens, portions of one segment and of exactly
    # one, new and continued states, padding
    ([289, 144, 704, 1, 400, 145], [4, 0, 1, 2, -1, 3], [0, 1, 0, 0, 1, 1]),
    ([1500], [3], [0]), ([1500], [3], [1])])
def test_portions_cut_in_segments(gpu, mode, d, dv, strong, lens, slots, first):
    if mode == "lightning" and dv == 48:
        dv = 200
    check(gpu, mode, d, dv, strong, torch.float32, lens, slots, first)


def check(gpu, mode, d, dv, strong, dtype, lens, slots, first):
    heads, eps = 3, 1e-6
    g = torch.Generator().manual_seed(d * 7 + dv + strong)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    T, wide = sum(lens), 2 * heads * (d + dv) + 2 * heads
    proj = rnd(T, wide + 3)[:, :wide]                # rows of a wider buffer
    extra = {"norm": (1 + 0.2 * rnd(heads * dv if mode == "mlstm" else dv)).to(dtype)}
    if mode == "hgrn2":
        low = torch.rand(heads * d, generator=g) * (0.0 if strong else 0.9)
        extra.update(lower=low.to(dtype), bias=(rnd(heads * d) - (6.0 if strong else 0.0)).to(dtype))
    elif mode == "gla":
        z = rnd(T, heads * d) * 3
        if strong:                                   # some channels forget everything at once
            z[:, ::5] -= 300.0
            z[7::11] -= 900.0
        extra.update(z=z, bias=rnd(heads * d).to(dtype), tau=8.0)
    elif mode == "lightning":
        extra["decays"] = torch.tensor([1e-3, 0.5, 1.0] if strong else [0.7, 0.97, 0.999])
    else:
        if strong:
            proj[5::9, -2 * heads:] *= 30.0          # gates slam shut and open
        extra.update(if_b=torch.cat([rnd(heads) - 1, rnd(heads) + 3]), cap=15.0, scale=0.6)
    state = rnd(6, heads, d, dv)
    nstate = torch.cat([rnd(6, heads, d), rnd(6, heads, 1).abs()], 2) if mode == "mlstm" else None
    want, want_s, want_n = oracle(mode, proj, extra, state, nstate, lens, slots, first, heads, d, dv, eps)
    pos = torch.cat([torch.arange(n) + (0 if f else 9) for n, f in zip(lens, first)]).int()
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist()).int()

    def step(device):
        ex = {k: (v.to(device) if isinstance(v, torch.Tensor) else v) for k, v in extra.items()}
        pd = torch.full((T, wide + 3), float("nan"), device=device)[:, :wide]
        pd.copy_(proj)
        st, ns = state.to(device, copy=True), nstate.to(device, copy=True) if nstate is not None else None
        tail = (torch.tensor(slots).int().to(device), cu.to(device), max(lens), pos.to(device), heads, d, dv)
        if mode == "hgrn2":
            got = H.hgrn2(pd, ex["bias"], ex["lower"], ex["norm"], eps, st, *tail)
        elif mode == "gla":
            got = H.gla(pd, ex["z"], ex["bias"], 8.0, ex["norm"], eps, st, *tail)
        elif mode == "lightning":
            got = H.lightning(pd, ex["decays"], st, *tail)
        else:
            got = torch.empty(T, heads * dv + 8, dtype=dtype, device=device)[:, 4:4 + heads * dv]
            H.mlstm(pd, ex["if_b"], 15.0, ex["norm"], eps, st, ns, *tail, got, 0.6)
        return got, st, ns

    def off(a, b):
        a, b = a.cpu().to(F64), b.to(F64)
        assert torch.isfinite(a).all()
        return float((a - b).norm() / b.norm())
    got, st, ns = step(gpu)
    walk, _, _ = step(torch.device("cpu"))           # the same step token by token in fp32
    # fp32 sums of at most 128 + 16 products and products of at most 16 decays: some 1e-6; bf16
    # rows add a rounding of at most 2^-9 of every value. A normed read-out may be what a cancelled
    # sum left over (one surviving token whose key and query are nearly orthogonal): its error is
    # bounded by the sum's terms, not by its value, and the fp32 walk shows how far that goes.
    assert off(got, want) < (3e-3 if got.dtype == torch.bfloat16 else max(1e-5, 4 * off(walk, want)))
    assert off(st, want_s) < 1e-5
    if ns is not None:
        assert off(ns, want_n) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["hgrn2", "gla", "lightning", "mlstm"])
@pytest.mark.parametrize("d,dv,known", [(128, 128, False), (64, 64, True), (24, 20, False)])
def test_a_short_sequence_does_not_feel_its_neighbours(gpu, mode, d, dv, known):
    """Single tokens and portions of one step, each alone and all together: a sequence runs the form of
    its own length, so that its rows and its state are the same to the bit (at d = 128 GLA's portions of
    2 tokens and more run the blocks' form beside longer ones)."""
    heads, dtype = 48, torch.bfloat16                 # (few heads: one round of blocks takes them all)
    lens, rnd = [1, 40, 1, 5, 33, 1, 15], lambda *s: torch.randn(*s, device=gpu)
    if mode == "gla" and d > 64:
        lens[3] = lens[6] = 1
    T, S = sum(lens), len(lens)
    proj, z = rnd(T, 2 * heads * (d + dv) + 2 * heads), rnd(T, heads * d)
    bias, low = rnd(heads * d).to(dtype), torch.rand(heads * d, device=gpu).to(dtype)
    nw = rnd(heads * dv if mode == "mlstm" else dv).to(dtype)
    ifb, decays = torch.cat([rnd(heads) - 1, rnd(heads) + 3]), torch.linspace(0.5, 0.99, heads, device=gpu)
    state, nstate = rnd(S, heads, d, dv), rnd(S, heads, d + 1).abs()

    def step(which):
        rows = torch.cat([torch.arange(sum(lens[:s]), sum(lens[:s + 1])) for s in which]).to(gpu)
        ls = [lens[s] for s in which]
        st, ns = state.clone(), nstate.clone()
        cu = torch.tensor([0] + ls).cumsum(0).int().to(gpu)
        pos = torch.cat([torch.arange(n) + 9 for n in ls]).int().to(gpu)
        tail = (torch.tensor(which).int().to(gpu), cu, max(ls), pos, heads, d, dv)
        more = dict(min_seqlen=min(ls)) if known else {}
        p = proj[rows].contiguous()
        if mode == "hgrn2":
            got = H.hgrn2(p, bias, low, nw, 1e-6, st, *tail, **more)
        elif mode == "gla":
            got = H.gla(p, z[rows].contiguous(), bias, 8.0, nw, 1e-6, st, *tail, **more)
        elif mode == "lightning":
            got = H.lightning(p, decays, st, *tail, **more)
        else:
            got = torch.full((len(rows), heads * dv), float("nan"), dtype=dtype, device=gpu)
            H.mlstm(p, ifb, 15.0, nw, 1e-6, st, ns, *tail, got, 0.6, **more)
        return got, st, ns
    got, st, ns = step(list(range(S)))
    assert torch.isfinite(got).all()
    for s in range(S):
        if lens[s] == 1 and (mode == "hgrn2" or mode == "gla" and d <= 64):
            continue                              # alone a decode step, whose sums are dealt otherwise
        alone, sa, na = step([s])
        at = sum(lens[:s])
        assert torch.equal(got[at:at + lens[s]], alone), lens[s]
        assert torch.equal(st[s], sa[s]) and torch.equal(ns[s], na[s]), lens[s]


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["hgrn2", "gla", "lightning", "mlstm"])
@pytest.mark.parametrize("d,dv", [(128, 128), (24, 20)])
@pytest.mark.parametrize("what", [float("nan"), float("inf")])
@pytest.mark.parametrize("part", ["key", "value"])
def test_no_token_feels_a_later_one(gpu, mode, d, dv, what, part):
    """A key or value that is not finite changes nothing before its own token, in its block of 16 either."""
    heads, T, bad = 2, 60, 37
    rnd = lambda *s: torch.randn(*s, device=gpu)  # noqa: E731
    proj, z, state, nstate = rnd(T, 2 * heads * (d + dv) + 2 * heads), rnd(T, heads * d), rnd(1, heads, d, dv), rnd(1, heads, d + 1).abs()
    bias, low, nw = rnd(heads * d), torch.rand(heads * d, device=gpu), rnd(heads * dv if mode == "mlstm" else dv)
    ifb, decays = torch.cat([rnd(heads) - 1, rnd(heads) + 3]), torch.tensor([0.5, 0.99], device=gpu)
    tail = (torch.zeros(1, dtype=torch.int32, device=gpu), torch.tensor([0, T]).int().to(gpu), T,
            torch.arange(T, device=gpu).int() + 3, heads, d, dv)

    def step(p):
        st, ns = state.clone(), nstate.clone()
        if mode == "hgrn2":
            return H.hgrn2(p, bias, low, nw, 1e-6, st, *tail), st
        if mode == "gla":
            return H.gla(p, z, bias, 8.0, nw, 1e-6, st, *tail), st
        if mode == "lightning":
            return H.lightning(p, decays, st, *tail), st
        got = torch.empty(T, heads * dv, device=gpu)
        H.mlstm(p, ifb, 15.0, nw, 1e-6, st, ns, *tail, got, 0.6)
        return got, st
    good, _ = step(proj)
    proj[bad, heads * d + 3 if part == "key" else 2 * heads * d + 3] = what
    got, st = step(proj)
    assert torch.isfinite(got[:bad]).all()
    # (fp32 sums of 16 terms in another order)
    assert (got[:bad] - good[:bad]).abs().max() <= 1e-5 * good.abs().max()
    if not (mode == "hgrn2" and part == "key" and what == float("inf")):        # (a saturated gate)
        assert not torch.isfinite(got[bad]).all() and not torch.isfinite(st).all()


def test_blocks_rule():
    G, X, L, M = H._CHUNK_GLA, H._CHUNK_HGRN2, H._CHUNK_FIXED, H._CHUNK_MLSTM

    def least(mode, lens, heads, d):
        return H.chunk_min_tokens(mode, len(lens), sum(lens), max(lens), min(lens) < 16, heads, d)
    for mode in (G, X, L, M):
        assert least(mode, [8000], 8, 64) == least(mode, [16] * 4, 32, 64) == 16     # CUs are left over
        assert least(mode, [20] * 64, 32, 64) > 40 and least(mode, [32] * 256, 16, 32) > 32
        assert least(mode, [1] * 16 + [2048], 8, 128) == 1            # one round of workgroups
        assert least(mode, [1] * 64 + [512], 32, 64) in (16, 32)      # one portion beside single tokens
    assert [least(m, [20] * 64, 32, 128) for m in (X, G, L, M)] == [32, 2, 32, 16]
    assert [least(m, [1] * 64 + [512], 32, 128) for m in (X, G, L, M)] == [32, 2, 32, 16]
