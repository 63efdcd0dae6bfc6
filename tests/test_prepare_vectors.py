"""The 16-byte forms of the attention prologues and of the loop entry's concatenation against the plain
reference, at widths that they take and ones that they leave to the column-at-a-time forms, with rows of
a wider buffer, padding tokens and positions far into a context."""
import pytest
import torch

from distributed_llm_inferencing_amd.ops import hybrid as H
from distributed_llm_inferencing_amd.ops import reference as R

pytestmark = pytest.mark.gpu


def close(a, b, dtype):
    # fp32: sums of at most 512 squares in another order, some 1e-6 of a norm; bf16: the rounding of a
    # value that differs by that much may fall to the neighbour, 2^-8
    a, b = a.float().cpu(), b.float().cpu()
    assert (a - b).abs().max() <= (2 ** -8 if dtype == torch.bfloat16 else 4e-6) * max(1.0, float(b.abs().max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,G,d,pad", [(32, 8, 128, 0), (5, 1, 64, 4), (3, 3, 256, 8), (40, 2, 4, 0),
                                           (7, 2, 96, 0), (4, 2, 30, 0), (4, 2, 128, 3)])
def test_attn_prepare(heads, G, d, pad, dtype):
    g = torch.Generator().manual_seed(d + heads)
    T, W = 9, (heads + G) * d
    proj = torch.randn(T, W + pad, generator=g)
    qw, kw = (torch.randn(d, generator=g).to(dtype) for _ in range(2))
    slots = torch.tensor([3, -1, 0, 7, 1, -1, 9, 4, 2]).int()
    kc, vc = (torch.full((10, G * d), 5.0, dtype=dtype) for _ in range(2))
    kd, vd = kc.cuda(), vc.cuda()
    want = R.attn_prepare(proj[:, :W], qw, kw, 1e-6, heads, G, d, kc, vc, slots, dtype)
    got = H.attn_prepare(proj.cuda()[:, :W], qw.cuda(), kw.cuda(), 1e-6, heads, G, d, kd, vd, slots.cuda())
    for a, b in ((got, want), (kd, kc), (vd, vc)):
        close(a, b, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,heads,G,d,pad", [(511, 32, 8, 128, 0), (513, 32, 8, 128, 4), (1707, 5, 1, 64, 4),
                                             (1639, 16, 4, 256, 0), (245, 40, 2, 4, 0), (1600, 16, 5, 32, 8)])
def test_attn_prepare_of_many_rows(T, heads, G, d, pad, dtype):
    """On both sides of the number of rows from which the 16-byte form runs."""
    g = torch.Generator().manual_seed(T)
    W = (heads + G) * d
    proj = torch.randn(T, W + pad, generator=g)
    qw, kw = (torch.randn(d, generator=g).to(dtype) for _ in range(2))
    slots = torch.randperm(T + 3, generator=g)[:T].int()
    slots[::7] = -1
    kc, vc = (torch.full((T + 3, G * d), 5.0, dtype=dtype) for _ in range(2))
    kd, vd = kc.cuda(), vc.cuda()
    want = R.attn_prepare(proj[:, :W], qw, kw, 1e-6, heads, G, d, kc, vc, slots, dtype)
    got = H.attn_prepare(proj.cuda()[:, :W], qw.cuda(), kw.cuda(), 1e-6, heads, G, d, kd, vd, slots.cuda())
    for a, b in ((got, want), (kd, kc), (vd, vc)):
        close(a, b, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,d,dr,r,rot,pad", [(32, 128, 64, 512, 64, 0), (3, 20, 12, 36, 6, 4),
                                                  (2, 64, 32, 48, 0, 0), (4, 16, 10, 48, 8, 0), (1, 8, 4, 4, 2, 1)])
def test_mla_prepare(heads, d, dr, r, rot, pad, dtype):
    g = torch.Generator().manual_seed(d + heads)
    T, W = 6, heads * (d + dr) + r + dr
    proj = torch.randn(T, W + pad, generator=g)
    cw = torch.randn(r, generator=g).to(dtype)
    # the reference rounds the angles to fp32: position * 2^-24 radians, below 5e-7 at these
    slots, pos = torch.tensor([3, -1, 0, 7, 1, 2]).int(), torch.tensor([0, 1, 5, 3, 6, 7]).int()
    inv = torch.pow(10000.0, -torch.arange(max(1, rot // 2)).double() / max(1, rot // 2))
    cache = torch.full((8, r + dr), 5.0, dtype=dtype)
    cd = cache.cuda()
    wn, wr = R.mla_prepare(proj[:, :W], cw, 1e-6, heads, d, dr, r, rot, inv, pos, slots, cache, dtype)
    gn, gf = H.mla_prepare(proj.cuda()[:, :W], cw.cuda(), 1e-6, heads, d, dr, r, rot, inv.cuda(), pos.cuda(),
                           slots.cuda(), cd)
    for a, b in ((gn, wn), (gf[:, :, r:], wr), (cd, cache)):
        close(a.reshape(-1), b.reshape(-1), dtype)
    # far into a context, the angles in double
    pos = torch.tensor([4000, 31000, 131071, 17, 70000, 9]).int()
    _, gf = H.mla_prepare(proj.cuda()[:, :W], cw.cuda(), 1e-6, heads, d, dr, r, rot, inv.cuda(), pos.cuda(),
                          slots.cuda(), cd)
    x = proj[:, :heads * (d + dr)].view(T, heads, d + dr)[:, :, d:]
    want, w = x.double().clone(), (pos.double()[:, None] * inv)[:, None, :rot // 2]
    even, odd = x[..., 0:rot:2].double(), x[..., 1:rot:2].double()
    want[..., 0:rot:2], want[..., 1:rot:2] = even * w.cos() - odd * w.sin(), odd * w.cos() + even * w.sin()
    close(gf[:, :, r:], want, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [4, 33, 1024, 4100])
def test_concat_cast(D, dtype):
    a, b = torch.randn(5, D), torch.randn(5, D)
    assert torch.equal(H.concat_cast(a.cuda(), b.cuda(), dtype).cpu(), torch.cat([a, b], 1).to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,D", [(159, 1028), (160, 1028), (170, 4100), (300, 33)])
def test_concat_cast_of_many_rows(T, D, dtype):
    a, b = torch.randn(T, D), torch.randn(T, D)
    assert torch.equal(H.concat_cast(a.cuda(), b.cuda(), dtype).cpu(), torch.cat([a, b], 1).to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,G,d,dv,rot,pad", [(32, 8, 128, 128, 64, 4), (4, 2, 24, 20, 24, 0), (4, 1, 32, 8, 8, 0),
                                                  (6, 3, 64, 64, 0, 0), (4, 2, 24, 20, 20, 0), (4, 2, 24, 18, 8, 1)])
def test_sink_prepare(heads, G, d, dv, rot, pad, dtype):
    g = torch.Generator().manual_seed(d + rot)
    T, W = 6, (heads + G) * d + G * dv
    proj = torch.randn(T, W + pad, generator=g)
    qw, kw = (torch.randn(n * d, generator=g).to(dtype) for n in (heads, G))
    slots, pos = torch.tensor([3, -1, 0, 7, 1, 2]).int(), torch.tensor([0, 1, 5, 4000, 31000, 7]).int()
    freq = torch.pow(10000.0, -torch.arange(max(1, rot // 2)).double() / max(1, rot // 2))
    kc, vc = torch.full((8, G * d), 5.0, dtype=dtype), torch.full((8, G * dv), 5.0, dtype=dtype)
    kd, vd = kc.cuda(), vc.cuda()
    want = R.sink_prepare(proj[:, :W], qw, kw, 1e-6, heads, G, d, dv, rot, freq[:rot // 2], 1.3, pos, kc, vc,
                          slots, dtype)
    got = H.sink_prepare(proj.cuda()[:, :W], qw.cuda(), kw.cuda(), 1e-6, heads, G, d, dv, rot, freq.cuda(), 1.3,
                         pos.cuda(), kd, vd, slots.cuda())
    for a, b in ((got, want), (kd, kc), (vd, vc)):
        close(a.reshape(-1), b.reshape(-1), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,groups,gated,pad", [(4096, 1, True, 4), (1024, 3, True, 0), (2052, 1, False, 0), (4100, 1, True, 0),
                                                (1030, 2, True, 0), (3000, 1, True, 3)])
def test_rmsnorm_of_few_wide_rows(n, groups, gated, pad, dtype):
    T, W = 5, n * groups
    src, gate = torch.randn(T, W + pad)[:, :W], torch.randn(T, W + pad)[:, :W]
    w = torch.randn(W).to(dtype)
    want = torch.cat([R.rmsnorm_cols(src[:, i * n:(i + 1) * n], w[i * n:(i + 1) * n], 1e-6, torch.float32,
                                     gate[:, i * n:(i + 1) * n] if gated else None) for i in range(groups)], 1) * 0.5

    def wide(x):                                 # rows of a wider buffer there too
        b = torch.zeros(T, W + pad, device="cuda")
        b[:, :W] = x.cuda()
        return b[:, :W]
    got = H.rmsnorm_cols(wide(src), w.cuda(), 1e-6, gate=wide(gate) if gated else None, groups=groups, out_scale=0.5)
    close(got, want, dtype)
