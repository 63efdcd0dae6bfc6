"""The fitted GEMM plans for steps above the decode sizes (ops.gemm.plan): each side of every line, and
the products that run on them against float64."""
import pytest
import torch

from distributed_llm_inferencing_amd import ops
from distributed_llm_inferencing_amd.ops import gemm as G
from distributed_llm_inferencing_amd.ops.reference import interleave_gate_up


@pytest.fixture(autouse=True)
def fitted():
    """No tuned or pinned plan while a test runs."""
    kept = dict(G._plan_cache), set(G._tuned)
    G.clear_plans()
    yield
    G.clear_plans()
    G._plan_cache.update(kept[0])
    G._tuned.update(kept[1])


@pytest.mark.parametrize("M,N,K,epi,tile,splits", [
    # fp32 outputs: half-width tiles where they fill the chip unsplit, else K split as for bf16
    (1100, 4096, 4096, "f32", 28, 1), (2048, 4096, 6144, "f32", 28, 1), (520, 8192, 4096, "f32", 28, 1),
    (1024, 4096, 4096, "f32", 22, 4), (1100, 4096, 14336, "f32", 22, 2), (1100, 4096, 6272, "f32", 22, 2),
    (1100, 4096, 6208, "f32", 22, 1), (2049, 4096, 4096, "f32", 55, 1), (520, 12288, 4096, "f32", 22, 1),
    # the persistent kernel: from 1024 rows, K in whole pairs of steps, long K for few rows only
    (1023, 28672, 4096, "none", 22, 1), (1024, 28672, 4096, "none", 55, 1), (8192, 4096, 4160, "none", 22, 1),
    (4095, 4096, 14336, "none", 55, 1), (4096, 4096, 14336, "none", 22, 1), (16384, 16384, 4096, "none", 55, 1),
    # not with a bias, nor for a pairing epilogue over short K (but several rounds of tiles of 1024)
    (4096, 3072, 768, "bias_gelu", 22, 1), (8192, 12288, 4096, "bias_gelu", 22, 1),
    (4096, 2304, 768, "bias", 22, 1), (1024, 8192, 1024, "silu_mul", 22, 1), (8192, 8192, 1024, "silu_mul", 55, 1),
    (8192, 8192, 512, "silu_mul", 22, 1), (1024, 8192, 4096, "silu_mul", 55, 1), (1024, 8192, 2048, "gelu_mul", 22, 1),
    (1024, 8224, 1024, "silu_mul", 55, 1),
    # the head over a wave's last rows: 256x256 tiles above 384 rows, below in nearly full rounds
    (512, 128256, 4096, "f32", 22, 1), (385, 102400, 768, "f32", 22, 1), (257, 128256, 4096, "f32", 22, 1),
    (384, 102400, 4096, "f32", 2, 1), (300, 128256, 1024, "f32", 2, 1), (512, 65280, 4096, "f32", 2, 1)])
def test_fitted_plan(M, N, K, epi, tile, splits):
    assert G.plan(M, N, K, epi) == G.GemmPlan("dli", tile, splits)


def test_a_fitted_plan_is_of_its_own_rows_and_a_pinned_one_of_its_bucket():
    assert G._bucket(1100) == G._bucket(2048)
    assert G.plan(1100, 4096, 14336, "none").splits == 2
    assert G.plan(2048, 4096, 14336, "none").splits == 2
    assert G.plan(1024, 4096, 14336, "none").splits == 4
    assert G.plan(2049, 4096, 14336, "none") == G.GemmPlan("dli", 55, 1)       # the bucket of 4096
    assert G.plan(4096, 4096, 14336, "none") == G.GemmPlan("dli", 22, 1)
    G.set_plan(4096, 4096, 14336, "none", G.GemmPlan("dli", 34, 1))
    for rows in (2049, 3000, 4096):
        assert G.plan(rows, 4096, 14336, "none") == G.GemmPlan("dli", 34, 1)
    assert G.plan(2048, 4096, 14336, "none").splits == 2


# sizes with partial tiles in both directions; the sums are fp32 in 64 to 4096 steps of 32 exact products
# (1e-6), bf16 results are rounded once, half an ulp (2^-9) a value
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,epi", [
    (1100, 4000, 2048, "f32"), (1025, 4104, 4096, "f32"), (1030, 4096, 14336, "f32"), (1500, 1032, 6208, "f32"),
    (2100, 4104, 1024, "f32"), (300, 65544, 2048, "f32"), (400, 65544, 768, "f32"), (1100, 2312, 768, "bias"),
    (1100, 3080, 768, "bias_gelu"), (1030, 8224, 1024, "silu_mul"), (1030, 8256, 1024, "silu_mul"), (4100, 4160, 1024, "gelu_mul")])
def test_products_on_fitted_plans(gpu, M, N, K, epi):
    g = torch.Generator(device=gpu).manual_seed(M + N)
    x, w = (torch.randn(r, K, device=gpu, generator=g).bfloat16() for r in (M, N))
    w = w * K ** -0.5
    bias = torch.randn(N, device=gpu, generator=g).bfloat16() if epi.startswith("bias") else None
    pairs = epi in G.PAIR_EPIS
    want = x.double() @ w.double().t()
    if epi.startswith("bias"):
        want += bias.double()
    if epi == "bias_gelu":
        want = torch.nn.functional.gelu(want, approximate="tanh")
    if pairs:
        gate, up = want[:, :N // 2], want[:, N // 2:]
        act = torch.nn.functional.silu(gate) if epi == "silu_mul" else torch.nn.functional.gelu(
            gate, approximate="tanh")
        want, w = act * up, interleave_gate_up(w[:N // 2], w[N // 2:]).contiguous()
    got = ops.linear(x, w, bias, epi=epi)
    assert got.shape == want.shape and got.dtype == (torch.float32 if epi == "f32" else torch.bfloat16)
    assert float((got.double() - want).norm() / want.norm()) < (1e-5 if epi == "f32" else 2.0 ** -8)


@pytest.mark.gpu
def test_persistent_tile_widths_are_the_kernels(gpu):
    from distributed_llm_inferencing_amd.ops import _native
    width = _native.require_native().dli_gemm_4w_width
    for M in (1, 256, 257, 1290, 2112, 2816, 4352, 5000, 8199):
        for N in (32, 160, 4096, 4100, 6144, 14336, 28672):
            for pairs in (False, True):
                assert G.persistent_width(M, N, pairs, G.device_cus()) == width(
                    55, G.EPI["silu_mul" if pairs else "none"], M, N, 1), (M, N, pairs)


# 17 x 16 = 272 tiles of 256 columns: a second round of 256 CUs, hardly filled, but one of 272 and of 304
def test_persistent_width_goes_by_the_devices_cus(monkeypatch):
    assert [G.persistent_width(4352, 4096, False, cus) for cus in (256, 272, 304)] == [160, 256, 256]
    for cus, tile in ((256, 55), (304, 22)):
        monkeypatch.setattr(G, "device_cus", lambda: cus)
        G._heuristic.cache_clear()
        assert G._heuristic(4352, 4096, 14336, "f32").tile == tile
    G._heuristic.cache_clear()


# every width of the persistent kernel's tiles, with partial tiles in both directions, two to twenty K-tiles and
# one to three tiles a workgroup; tolerances as above
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,epi,width", [
    (1290, 4100, 128, "f32", 160), (2300, 4090, 640, "none", 160), (4300, 4096, 256, "f32", 160), (300, 1000, 1280, "f32", 160),
    (2810, 4104, 384, "f32", 192), (5000, 4096, 128, "none", 192), (900, 10400, 256, "f32", 192), (1270, 28672, 128, "silu_mul", 192),
    (1270, 28704, 256, "gelu_mul", 192), (9216, 4096, 128, "f32", 256), (300, 1024, 128, "silu_mul", 192)])
def test_persistent_tiles_of_every_width(gpu, M, N, K, epi, width):
    pairs = epi in G.PAIR_EPIS
    assert G.persistent_width(M, N, pairs) == width
    g = torch.Generator(device=gpu).manual_seed(M + N)
    x, w = (torch.randn(r, K, device=gpu, generator=g).bfloat16() for r in (M, N))
    w = w * K ** -0.5
    want = x.double() @ w.double().t()
    if pairs:
        gate, up = want.view(M, N // 32, 2, 16).unbind(2)
        act = torch.nn.functional.silu(gate) if epi == "silu_mul" else torch.nn.functional.gelu(gate, approximate="tanh")
        want = (act * up).reshape(M, N // 2)
    got = ops._gemm_native(x, w, epi, plan=G.GemmPlan("dli", 55, 1)).double()
    assert float((got - want).norm() / want.norm()) < (1e-5 if epi == "f32" else 2.0 ** -8)


class OnGpu:
    """A CPU tensor that says it is on the GPU."""
    is_cuda = True

    def __init__(self, t):
        self.t = t

    def __getattr__(self, name):
        return getattr(self.t, name)


# a split product's operands go to the kernel by address: those that do not match go to linear_any, which raises
def test_partial_sums_of_mismatched_operands_are_refused(monkeypatch):
    from distributed_llm_inferencing_amd.ops import hybrid as H
    calls = []
    monkeypatch.setattr(H._gemm, "plan", lambda *a: G.GemmPlan("dli", 22, 2))
    monkeypatch.setattr(H._gemm, "workspace", lambda device, nbytes: torch.empty(nbytes, dtype=torch.uint8))
    monkeypatch.setattr(H, "_call", lambda *a: calls.append(a[0]))
    monkeypatch.setattr(H, "_st", lambda: None)
    x = OnGpu(torch.zeros(8, 128).bfloat16())
    assert H.linear_out(x, torch.zeros(64, 128).bfloat16()).shape == (2, 8, 64) and calls.pop() == "dli_gemm"
    for w in (torch.zeros(64, 128), torch.zeros(64, 64).bfloat16(), torch.zeros(64, 256).bfloat16()):
        with pytest.raises(ValueError):
            H.linear_out(x, w)
    assert not calls


# the timing of a product with a bias reads one: an address of none is a fault on the GPU (a width of K that gives
# candidates, as GPT-2's 768 does and its tiny variant's does not)
@pytest.mark.parametrize("epi", ["bias", "bias_gelu", "clamp_mul", "f32"])
@pytest.mark.parametrize("M,N,K", [(1, 96, 768), (64, 96, 768), (2048, 256, 768)])
@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_timed_products_have_their_bias(device, monkeypatch, epi, M, N, K):
    seen = []
    native = ops._gemm_native

    def product(x, w, epi, bias=None, plan=None, **more):
        seen.append(None if bias is None else (bias.numel(), bias.dtype, bias.device.type))
        if device != "cpu":
            assert seen[-1] is not None or epi == "f32"
            native(x, w, epi, bias=bias, plan=plan, **more)
    monkeypatch.setattr(ops, "_gemm_native", product)
    if device == "cpu":
        monkeypatch.setattr(ops, "benchmark", lambda run, **k: (run(), 1.0)[1])
    w = torch.ones(N, K, device=device).bfloat16()
    more = dict(candidates=G.prefill_candidates) if M > 1024 else {}
    got = G.autotune([(M, N, K, epi)], {(N, K): w}, torch.device(device), iters=1, cold_bytes=1, **more)
    want = {"clamp_mul": (1, torch.float32, device), "f32": None}.get(epi, (N, torch.bfloat16, device))
    assert seen and all(s == want for s in seen) and (M, N, K, epi) in got


def test_a_missing_bias_is_refused(monkeypatch):
    monkeypatch.setattr(ops, "_native_call", lambda *a: pytest.fail("reached the kernel"))
    x, w = torch.zeros(8, 768).bfloat16(), torch.zeros(96, 768).bfloat16()
    for epi in ("bias", "bias_gelu", "clamp_mul"):
        with pytest.raises(ValueError):
            ops._gemm_native(x, w, epi, plan=G.GemmPlan("dli", 5, 1))


@pytest.mark.gpu
def test_the_library_refuses_a_missing_bias(gpu):
    from distributed_llm_inferencing_amd.ops import _native
    lib = _native.require_native()
    x, w, o = (torch.zeros(r, 768, device=gpu).bfloat16() for r in (8, 96, 8))
    for tile in (0, 22, 34, 45, 30, 55, 62):
        for epi in ("bias", "bias_gelu"):
            assert lib.dli_gemm(ops._p(x), 768, ops._p(w), 768, ops._p(o), 96, 4, 96, 768, G.EPI[epi], tile, 1, None,
                                None, None, 1, ops._st()) != 0


# rows that the 4-wave kernel does not reach by its offsets (expanded, windows of a signal, very far apart) go to it as a
# copy, one row with its length for a stride; other kernels take them as they are
@pytest.mark.parametrize("tile,copied", [(22, True), (28, True), (45, True), (55, True), (26, False), (2, False)])
def test_rows_of_any_stride(monkeypatch, tile, copied):
    calls = []
    monkeypatch.setattr(ops, "_native_call", lambda name, *a: calls.append(a[:4]))
    monkeypatch.setattr(ops, "_st", lambda: None)
    plan, w = G.GemmPlan("dli", tile, 1), torch.zeros(32, 128).bfloat16()
    signal = torch.zeros(4096).bfloat16()
    for x in (w[:1].expand(16, 128), signal.as_strided((16, 128), (40, 1)), signal.as_strided((16, 128), (200, 1)), w[:, :128]):
        ops._gemm_native(x, w, "none", plan=plan)
        a, lda, _, ldw = calls.pop()
        assert (a, lda) == ((x.data_ptr(), x.stride(0)) if not copied or x.stride(0) >= 128 else (a, 128)) and ldw == 128
        assert (a == x.data_ptr()) == (not copied or x.stride(0) >= 128)
        ops._gemm_native(w, x[:16], "none", plan=plan)
        assert calls.pop()[3] == (max(x.stride(0), 128) if copied else x.stride(0))
    ops._gemm_native(signal.as_strided((1, 128), (1, 1)), w, "none", plan=plan)
    assert calls.pop()[:2] == (signal.data_ptr(), 128 if copied else 1)
    monkeypatch.setattr(G, "MAX_4W_STRIDE", 200)
    far = signal.as_strided((16, 128), (200, 1))
    assert G.spaced(far, far, tile)[1::2] == ((128, 128) if copied else (200, 200))


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [22, 28, 45, 55])
@pytest.mark.parametrize("stride", [0, 8, 40, 120])
def test_products_of_overlapping_rows(gpu, tile, stride):
    signal = torch.randn(300 * 120 + 128, device=gpu, generator=torch.Generator(device=gpu).manual_seed(1)).bfloat16()
    x = signal.as_strided((300, 128), (stride, 1))
    w = torch.randn(264, 128, device=gpu, generator=torch.Generator(device=gpu).manual_seed(2)).bfloat16()
    plan = G.GemmPlan("dli", tile, 1)
    for a, b in ((x, w), (w, x)):
        assert torch.equal(ops._gemm_native(a, b, "f32", plan=plan), ops._gemm_native(a.contiguous(), b.contiguous(), "f32", plan=plan))
