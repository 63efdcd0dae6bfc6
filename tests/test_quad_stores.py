"""Kernels that store four columns at a time where every row takes it, and one by one elsewhere."""
import pytest
import torch

from distributed_llm_inferencing_amd.ops import hybrid
from distributed_llm_inferencing_amd.ops import hybrid as H


# N a multiple of 4, of 2, odd; rows of the output 16 bytes apart and not; an output that starts off 16 bytes.
# bf16 products summed in fp32: K terms of at most |a||b|, 2^-24 each, and bf16's own rounding
@pytest.mark.gpu
@pytest.mark.parametrize("N", [4096, 68, 30, 33])
@pytest.mark.parametrize("K", [32, 96, 7])
@pytest.mark.parametrize("pad,off", [(0, 0), (4, 0), (3, 0), (4, 1)])
@pytest.mark.parametrize("f32", [True, False])
def test_rank_products(gpu, N, K, pad, off, f32):
    g = torch.Generator(device=gpu).manual_seed(N + K)
    M = 70
    x, w = (torch.randn(r, K, device=gpu, generator=g).bfloat16() for r in (M, N))
    whole = torch.full((M, N + pad + off), 7.0, device=gpu, dtype=torch.float32 if f32 else torch.bfloat16)
    out = whole[:, off:off + N]
    H.linear_any(x, w, out_f32=f32, out=out)
    want = x.double() @ w.double().T
    bound = (x.double().abs() @ w.double().abs().T) * K * 2.0 ** -24 + (0 if f32 else want.abs() * 2.0 ** -8)
    assert bool(((out.double() - want).abs() <= bound).all())
    assert bool((whole[:, :off] == 7).all()) and bool((whole[:, off + N:] == 7).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dim", [40, 30, 4096])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hashed", [True, False])
@pytest.mark.parametrize("many", [False, True])            # (from 2^19 elements in pieces)
def test_bigram_rows(gpu, dim, dtype, hashed, many):
    g = torch.Generator(device=gpu).manual_seed(dim)
    T = -(-(1 << 19) // dim) if many else 65
    t, b = (torch.randn(r, dim, device=gpu, generator=g).to(dtype) for r in (31, 18))
    ids = torch.randint(0, 31, (T,), device=gpu, generator=g, dtype=torch.int32)
    prev = torch.randint(-1, 31, (T,), device=gpu, generator=g, dtype=torch.int32)
    x, xs = H.embedding_bigram(ids, prev if hashed else None, t, b if hashed else None, 17, 29, 5)
    want = t[ids.long()].float()
    if hashed:
        row = torch.where(prev < 0, 17, (prev.long() * 29 + ids.long() * 5) % 17)
        want = want + b[row].float()
    assert torch.equal(x, want) and torch.equal(xs, want.to(dtype))


# groups of whole quads and not, against float64: the sums' and products' rounding, and the output's
@pytest.mark.gpu
@pytest.mark.parametrize("dim,groups", [(4096, 4), (4096, 1), (40, 2), (60, 4), (48, 3), (4096, 64), (30, 5), (36, 6)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [3, 1030])
def test_grouped_norm(gpu, dim, groups, dtype, rows):
    g = torch.Generator(device=gpu).manual_seed(dim + groups)
    x, y = (torch.randn(rows, dim, device=gpu, generator=g) for _ in range(2))
    w = torch.randn(dim, device=gpu, generator=g).to(dtype)
    new = x.double() + 0.7 * y.double()
    v = new.view(rows, groups, -1)
    want = (v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-5)).view(rows, dim) * (w.double() + 0.5) * 1.25
    h = H.resadd_groupnorm(x, y, w, groups, 1e-5, mult=0.7, gain=1.25, w_offset=0.5)
    assert torch.allclose(x.double(), new, rtol=0, atol=float(new.abs().max()) * 2.0 ** -22)
    # a group's sum of squares: dim / groups terms of one sign, half of that in the root; five roundings after
    rel = (dim / groups / 2 + 8) * 2.0 ** -24 + (2.0 ** -8 if dtype == torch.bfloat16 else 0)
    assert bool(((h.double() - want).abs() <= rel * want.abs() + 2.0 ** -21 * (w.double().abs() + 0.5)).all())


# the pieces' form (rows 16 bytes apart) and the general one (rows 4 bytes off) against float64: the split
# halves and the interleaved pairs, part of the tail rotated, none of it, a cache of another layer, unused slots
@pytest.mark.gpu
@pytest.mark.parametrize("H,d,dr,r,rot", [(32, 128, 64, 512, 64), (3, 8, 16, 20, 8), (2, 4, 8, 4, 0), (2, 8, 12, 12, 6)])
@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("own", [True, False])
@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_latent_rows(gpu, H, d, dr, r, rot, half, own, pad, dtype):
    g = torch.Generator(device=gpu).manual_seed(d + r + rot)
    T = 9
    q = torch.randn(T, H * (d + dr) + 4 * pad + pad, device=gpu, generator=g)[:, pad:pad + H * (d + dr)]
    kv = torch.randn(T, r + dr + 4 * pad + pad, device=gpu, generator=g)[:, pad:pad + r + dr] if own else None
    w = torch.randn(r, device=gpu, generator=g).to(dtype)
    freq = torch.rand(max(rot // 2, 1), device=gpu, generator=g).double()
    pos = torch.randint(0, 5000, (T,), device=gpu, generator=g, dtype=torch.int32)
    slots = torch.arange(T, device=gpu, dtype=torch.int32) * 2
    slots[4] = -1
    cache = torch.full((2 * T, r + dr), 7.0, device=gpu, dtype=dtype)
    want = cache.double().cpu()
    qn, qf = hybrid.latent_prepare(q, kv, w, 1e-5, H, d, dr, r, rot, freq, pos, slots, cache, dtype, half)
    c = lambda t: None if t is None else t.double().cpu()  # noqa: E731
    tail = lambda v: rotated(v, pos.double().cpu(), freq.cpu(), rot, half)  # noqa: E731
    qq = c(q).reshape(T, H, d + dr)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    near = lambda a, b: bool(((c(a) - b).abs() <= ulp * b.abs() + 2.0 ** -20).all())  # noqa: E731
    assert near(qn, qq[:, :, :d]) and near(qf[:, :, r:], tail(qq[:, :, d:]))
    if own:
        lat = c(kv)[:, :r] * torch.rsqrt(c(kv)[:, :r].pow(2).mean(-1, keepdim=True) + 1e-5) * c(w)
        ok = (slots >= 0).cpu()
        want[slots.cpu()[ok].long()] = torch.cat([lat, tail(c(kv)[:, None, r:])[:, 0]], 1)[ok]
    assert near(cache, want)


def rotated(v, pos, freq, rot, half):
    """v float64 [T, H, dr]: the first rot dims turned by pos * freq."""
    out = v.clone()
    if not rot:
        return out
    a = pos[:, None, None] * freq[None, None, :rot // 2]
    co, si = a.cos().float().double(), a.sin().float().double()
    x, y = (v[..., :rot // 2], v[..., rot // 2:rot]) if half else (v[..., 0:rot:2], v[..., 1:rot:2])
    first, second = x * co - y * si, y * co + x * si
    if half:
        out[..., :rot // 2], out[..., rot // 2:rot] = first, second
    else:
        out[..., 0:rot:2], out[..., 1:rot:2] = first, second
    return out


# rows in a workgroup's registers (1024 to 4096 columns in quads) and the forms around it; several parts, gates
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1020, 1024, 1028, 1030, 2052, 4096, 4100])
@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("rows", [3, 601])
@pytest.mark.parametrize("gated", [False, True])
def test_column_norm(gpu, n, groups, rows, gated):
    g = torch.Generator(device=gpu).manual_seed(n + rows)
    x = torch.randn(rows, n * groups, device=gpu, generator=g)
    gate = torch.randn(rows, n * groups, device=gpu, generator=g) if gated else None
    w = torch.randn(n * groups, device=gpu, generator=g).bfloat16()
    got = hybrid.rmsnorm_cols(x, w, 1e-5, gate=gate, groups=groups)
    v = x.double().view(rows, groups, n)
    want = (v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-5)).view(rows, -1) * w.double()
    if gated:
        want = want * torch.sigmoid(gate.double())
    # bf16's rounding; the sum's and the few products' before it are 2^-24 each
    assert bool(((got.double() - want).abs() <= (2.0 ** -8 + 2.0 ** -12) * want.abs() + 1e-30).all())
