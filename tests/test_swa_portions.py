"""Portions of sliding-window attention whose tiles are staged by sixteens of cache rows: windows and kept tokens at every
alignment to them, blocks that the form takes and that it does not, cache rows behind a sequence's last that hold NaN."""
import re
import subprocess

import pytest
import torch

from distributed_llm_inferencing_amd import build
from distributed_llm_inferencing_amd.ops import hybrid as H
from distributed_llm_inferencing_amd.ops import reference as R


def run(gpu, lens, before, block, window, keep, d=128, dv=128, G=2, wide=0):
    heads, scale = 4, d ** -0.5
    g = torch.Generator().manual_seed(sum(lens) + block + keep)
    S, T, ctx = len(lens), sum(lens), [a + b for a, b in zip(lens, before)]
    need = [-(-c // block) for c in ctx]
    perm = torch.randperm(sum(need) + 1, generator=g).int()
    bt, o = torch.full((S, max(need)), int(perm[-1]), dtype=torch.int32), 0
    for s, n in enumerate(need):
        bt[s, :n] = perm[o:o + n]
        o += n
    kc, vc = (torch.full((len(perm) * block, G * w + wide), float("nan")).bfloat16() for w in (d, dv))
    for s, n in enumerate(ctx):
        j = torch.arange(n)
        rows = bt[s].long()[j // block] * block + j % block
        kc[rows] = torch.randn(n, kc.shape[1], generator=g).bfloat16()
        vc[rows] = torch.randn(n, vc.shape[1], generator=g).bfloat16()
    q = torch.randn(T, heads * d, generator=g).bfloat16()
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist()).int()
    pos = torch.cat([torch.arange(n) + b for n, b in zip(lens, before)]).int()
    want = R.window_attention(q, kc.nan_to_num(0)[:, :G * d], vc.nan_to_num(0)[:, :G * dv], d, dv, heads, G, cu, pos, bt, block,
                              window, scale, out_dtype=torch.float32, keep_first=keep).double()
    kg, vg = kc.to(gpu)[:, :G * d], vc.to(gpu)[:, :G * dv]
    got = H.window_attention(q.to(gpu), kg, vg, d, dv, heads, G, cu.to(gpu), max(lens), pos.to(gpu), bt.to(gpu), block, window,
                             scale, keep_first=keep).double().cpu()
    assert torch.isfinite(got).all()
    # weights and outputs rounded to bf16, half an ulp (2^-9) each
    assert float((got - want).norm() / want.norm()) < 2 * 2.0 ** -9


@pytest.mark.gpu
@pytest.mark.parametrize("keep", [0, 1, 15, 16, 17, 64, 65, 200])
@pytest.mark.parametrize("window", [1, 16, 63, 100, 257, 1 << 30])
def test_windows_and_kept_tokens(gpu, window, keep):
    run(gpu, [192, 300, 1, 513], [0, 37, 400, 160], 16, window, keep)


@pytest.mark.gpu
@pytest.mark.parametrize("block", [1, 8, 16, 24, 32, 48, 256])
@pytest.mark.parametrize("window,keep", [(1 << 30, 0), (90, 5)])
def test_blocks(gpu, block, window, keep):
    run(gpu, [193, 260, 7], [0, 33, 511], block, window, keep)


@pytest.mark.gpu
@pytest.mark.parametrize("d,dv", [(64, 64), (64, 128), (96, 192), (128, 256)])
@pytest.mark.parametrize("window,keep", [(1 << 30, 0), (100, 3)])
def test_widths(gpu, d, dv, window, keep):
    run(gpu, [200, 333], [10, 77], 16, window, keep, d, dv, wide=8)


def form(block, width, window, keep, d=128, dv=128, G=2):
    """How the kernel finds its tiles: 2 by sixteens of rows, 1 by a table of rows, 0 by the block table."""
    from distributed_llm_inferencing_amd.ops import _native
    return _native.require_native().dli_swa_portion_form(d, dv, G * d, G * dv, block, min(window, width * block), keep)


# contexts past the tables beside the tiles: 6144 keys row by row (fewer at 128 + 256 wide), 65536 by sixteens at 128 + 256; and to them
@pytest.mark.gpu
@pytest.mark.parametrize("block,before,window,keep,d,dv,found", [
    (16, 70000, 1 << 30, 0, 128, 128, 2), (16, 70000, 1 << 30, 0, 128, 256, 0), (256, 64000, 1 << 30, 0, 128, 256, 2), (24, 5600, 1 << 30, 0, 128, 128, 1),
    (24, 6500, 1 << 30, 0, 128, 128, 0), (8, 7000, 1 << 30, 0, 64, 64, 0), (8, 7000, 1 << 30, 70, 96, 192, 0), (24, 9000, 6000, 20, 64, 128, 0),
    (8, 3500, 1 << 30, 0, 128, 256, 1), (8, 4100, 1 << 30, 5, 128, 256, 0), (1, 300, 250, 40, 128, 128, 1)])
def test_long_contexts(gpu, block, before, window, keep, d, dv, found):
    lens = [260, 193]
    assert form(block, -(-(before + 260) // block), window, keep, d, dv) == found
    run(gpu, lens, [before, before // 3], block, window, keep, d, dv)


# the expanded latent form's rows: NaN behind each sequence's, windows at every alignment
@pytest.mark.gpu
@pytest.mark.parametrize("window", [1, 50, 64, 129, 1 << 30])
@pytest.mark.parametrize("lens,before", [([64], [0]), ([300, 1, 255], [100, 9, 33]), ([513, 65], [0, 700])])
def test_shared_tails(gpu, lens, before, window):
    heads, d, dr = 3, 128, 64
    g = torch.Generator(device=gpu).manual_seed(sum(lens))
    ctx = [a + b for a, b in zip(lens, before)]
    T, rows, scale = sum(lens), sum(ctx), (d + dr) ** -0.5
    rnd = lambda *s: torch.randn(*s, device=gpu, generator=g).bfloat16()  # noqa: E731
    q, q2, kv, k2 = rnd(T, heads, d), rnd(T, heads, dr), rnd(rows + 70, heads * 2 * d), rnd(rows + 70, 8 + dr)
    kv[rows:] = k2[rows:] = float("nan")
    cu, cuc = (torch.tensor([0] + torch.tensor(x).cumsum(0).tolist(), dtype=torch.int32, device=gpu) for x in (lens, ctx))
    pos = torch.cat([torch.arange(n) + b for n, b in zip(lens, before)]).int().to(gpu)
    out = torch.zeros(T, heads * d, device=gpu).bfloat16()
    v, tail = kv[:, heads * d:], k2[:, 8:]
    H._call("dli_shared_tail_attention", H._p(q), heads * d, H._p(q2), heads * dr, dr, H._p(kv), kv.stride(0), H._p(tail),
            tail.stride(0), H._p(v), kv.stride(0), H._p(out), heads * d, H._p(cu), H._p(pos), H._p(cuc), len(lens), max(lens),
            heads, d, dr, d, window, scale, None, 0, H._st())
    for s, n in enumerate(lens):
        t, r = slice(int(cu[s]), int(cu[s + 1])), slice(int(cuc[s]), int(cuc[s + 1]))
        k = torch.cat([kv[r, :heads * d].view(-1, heads, d), k2[r, None, 8:].expand(-1, heads, -1)], 2).double()
        far = pos[t].long()[:, None] - torch.arange(ctx[s], device=gpu)[None]
        sc = (torch.cat([q[t], q2[t]], 2).double().permute(1, 0, 2) @ k.permute(1, 2, 0).contiguous()) * scale
        p = sc.masked_fill(((far < 0) | (far >= window))[None], float("-inf")).softmax(-1)
        want = (p @ v[r].view(-1, heads, d).double().permute(1, 0, 2).contiguous()).permute(1, 0, 2).reshape(n, -1)
        assert float((out[t].double() - want).norm() / want.norm()) < 2 * 2.0 ** -9


# no form spills registers, whose traffic would pass the counted waits for the tiles (11 to 14 % where one did), but that of the row
# table at 128 + 256 wide, which is ahead of the general mask in windows even so
def test_registers(tmp_path):
    src = build.CSRC / "kernels" / "swa_attention.hip"
    r = subprocess.run([build._hipcc(), *build.KERNEL_FLAGS, build._REMARKS, "-I", str(src.parent), "--offload-device-only", "-S", str(src),
                        "-o", str(tmp_path / "k.s")], check=True, capture_output=True, text=True)
    scratch = dict(re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)", r.stderr, re.S))
    assert sum("swa_prefill32" in k for k in scratch) >= 11
    assert [k for k, n in scratch.items() if n != "0" and "swa_prefill32_kernelILi128ELi0ELi256ELi1E" not in k] == []
