"""Decode steps of the scalar-decay recurrences (one token a sequence, ops.hybrid.lightning / mlstm) against
float64, and the partial sums that the stream and post-norm kernels add up."""
import pytest
import torch

from distributed_llm_inferencing_amd.ops import hybrid as H

CAP, EPS = 15.0, 1e-6


def _step(mode, d, heads, n, gpu, dtype, pad):
    g = torch.Generator(device=gpu).manual_seed(d + heads + n)
    r = lambda *s: torch.randn(*s, device=gpu, generator=g)  # noqa: E731
    width = (4 * d + 2) * heads if mode == "mlstm" else 4 * d * heads
    proj = r(n, width + pad)[:, :width]
    slots = torch.randperm(n + 2, device=gpu, generator=g)[:n].to(torch.int32)
    slots[n // 2] = -1                                    # a padding row of a captured step
    pos = torch.randint(1, 50, (n,), device=gpu, generator=g, dtype=torch.int32)
    pos[0] = 0                                            # starts from zeros whatever its slot held
    cu = torch.arange(n + 1, device=gpu, dtype=torch.int32)
    state, mstate = r(n + 2, heads, d, d), r(n + 2, heads, d + 1)
    q, k, v = (proj[:, i * heads * d:(i + 1) * heads * d].view(n, heads, d).double() for i in range(3))
    use = slots.clamp(min=0).long()
    live = (pos > 0).double().view(n, 1, 1)
    S = state.double()[use] * live[..., None]
    if mode == "lightning":
        decay = torch.linspace(0.3, 0.999, heads, device=gpu)
        silu = torch.nn.functional.silu
        q, k, v = silu(q), silu(k), silu(v)
        S = decay.double().view(1, heads, 1, 1) * S + k[..., None] * v[..., None, :]
        want = (q[..., None, :] @ S)[..., 0, :].reshape(n, -1)
        got = H.lightning(proj, decay, state, slots, cu, 1, pos, heads, d, d)
        tol = 1e-5                                        # fp32 sums of d products
    else:
        b, w = r(2 * heads), r(heads * d).to(dtype)
        i, f = (CAP * torch.tanh((proj[:, o:o + heads].double() + c.double()) / CAP)
                for o, c in ((4 * heads * d, b[:heads]), (4 * heads * d + heads, b[heads:])))
        f = torch.nn.functional.logsigmoid(f)
        m = mstate.double()[use][..., d] * live[..., 0]
        nv = mstate.double()[use][..., :d] * live
        top = torch.maximum(f + m, i)
        a, e = (f + m - top).exp()[..., None], (i - top).exp()[..., None]
        S, nv = a[..., None] * S + (e * k)[..., None] * v[..., None, :], a * nv + e * k
        q = q * d ** -0.5
        o = (q[..., None, :] @ S)[..., 0, :] / (torch.maximum((nv * q).sum(-1).abs(), (-top).exp())[..., None] + 1e-6)
        o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS)
        gate = torch.sigmoid(proj[:, 3 * heads * d:4 * heads * d].double())
        want = o.reshape(n, -1) * w.double() * gate * 0.6
        got = torch.empty(n, heads * d + 8, dtype=dtype, device=gpu)[:, :heads * d]
        H.mlstm(proj, b, CAP, w, EPS, state, mstate, slots, cu, 1, pos, heads, d, d, got, 0.6)
        tol = 2e-5 if dtype == torch.float32 else 2.0 ** -8
        kept = slots >= 0
        assert float((mstate.double()[use][kept][..., :d] - nv[kept]).norm() / nv[kept].norm()) < 1e-5
        assert torch.allclose(mstate.double()[use][kept][..., d], top[kept], rtol=1e-5, atol=1e-5)
    kept = slots >= 0
    assert bool((got[~kept] == 0).all())
    assert float((got[kept].double() - want[kept]).norm() / want[kept].norm()) < tol
    assert float((state.double()[use][kept] - S[kept]).norm() / S[kept].norm()) < 1e-6 * d ** 0.5


# 64 and 128: the step's own kernel; rows 4 bytes off (pad 1) and other widths: the general one
@pytest.mark.gpu
@pytest.mark.parametrize("mode,dtype", [("lightning", torch.float32), ("mlstm", torch.float32), ("mlstm", torch.bfloat16)])
@pytest.mark.parametrize("d,heads,n,pad", [(128, 1, 2, 0), (128, 16, 5, 0), (64, 3, 70, 0), (64, 4, 3, 1), (32, 2, 3, 0)])
def test_step_matches_float64(gpu, mode, dtype, d, heads, n, pad):
    _step(mode, d, heads, n, gpu, dtype, pad)


# sums of up to 4 fp32 numbers in either order
@pytest.mark.gpu
@pytest.mark.parametrize("dim", (4096, 64, 30))
@pytest.mark.parametrize("splits", (2, 4))
def test_partial_sums_are_added(gpu, dim, splits):
    g = torch.Generator(device=gpu).manual_seed(dim)
    r = lambda *s: torch.randn(*s, device=gpu, generator=g)  # noqa: E731
    T, w = 5, r(dim).bfloat16()
    y = r(splits, T, dim)
    for ns in (1, 2, 3, 4, 6):
        xs, prev, read = r(T, ns, dim), r(ns * (ns + 2)), r(ns)
        a, b = xs.clone(), xs.clone()
        ha = H.hyper_mix(a, y, prev, read, w, 1e-6, 1.0)
        hb = H.hyper_mix(b, y.sum(0), prev, read, w, 1e-6, 1.0)
        want = torch.einsum("tsd,sr->trd", xs.double(), prev[2 * ns:].double().view(ns, ns)) + (
            prev[ns:2 * ns].double()[None, :, None] * y.double().sum(0)[:, None])
        assert torch.allclose(a.double(), want, rtol=1e-5, atol=1e-5 * float(want.abs().max()))
        assert torch.allclose(a, b, rtol=1e-5, atol=1e-5) and torch.allclose(ha.float(), hb.float(), rtol=2e-2, atol=2e-2)
    x, bias = r(T, dim), r(dim).bfloat16()
    a, b = x.clone(), x.clone()
    ha, hb = H.postnorm(a, y, w, bias, 1e-6, 2.0), H.postnorm(b, y.sum(0), w, bias, 1e-6, 2.0)
    assert torch.allclose(a, b, rtol=1e-4, atol=1e-4) and torch.allclose(ha.float(), hb.float(), rtol=2e-2, atol=2e-2)
