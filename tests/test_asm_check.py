"""The build's look through the assembly of kernels whose matrix products are asm statements, which hipcc pads nothing
for: what it finds, what it lets pass, and the kernels themselves."""
import re
import subprocess

import pytest

from distributed_llm_inferencing_amd import asm_check, build

PRODUCT = "v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], a[16:19], a[0:15]"
REQUEST = "buffer_load_dwordx4 v156, s[40:43], s78 offen lds"
SMALL = "v_mfma_f32_16x16x32_bf16 v[8:11], v[0:3], v[4:7], 0"


def function(*lines):
    return "\t.type\tk,@function\nk:\n" + "\n".join(lines) + "\n\ts_endpgm\n.Lfunc_end0:\n"


# 12 wait states behind the 32x32 product, 8 behind the 16x16 one, on any path; 2 from an operand's write to its product
@pytest.mark.parametrize("lines,ok", [
    ([PRODUCT, "s_nop 10", "v_accvgpr_read_b32 v0, a15"], False),
    ([PRODUCT, "s_nop 11", "v_accvgpr_read_b32 v0, a15"], True),
    ([PRODUCT, "s_nop 3", "v_accvgpr_read_b32 v0, a16"], True),
    ([PRODUCT, "v_accvgpr_write_b32 a3, v9"], False),
    ([PRODUCT, PRODUCT, "s_nop 11", "v_accvgpr_read_b32 v0, a0"], True),
    ([PRODUCT, "v_mfma_f32_32x32x16_bf16 a[32:47], v[0:3], a[12:15], a[32:47]"], False),
    ([SMALL, "s_nop 6", "global_store_dwordx4 v12, v[8:11], s[0:1]"], False),
    ([SMALL, "s_nop 7", "global_store_dwordx4 v12, v[8:11], s[0:1]"], True),
    ([PRODUCT, "s_cbranch_scc0 .LBB0_1", "s_nop 15", ".LBB0_1:", "v_accvgpr_read_b32 v0, a0"], False),
    ([PRODUCT, "s_branch .LBB0_2", ".LBB0_1:", "v_accvgpr_read_b32 v0, a0", ".LBB0_2:", "s_nop 15"], True),
    ([".LBB0_1:", "v_accvgpr_read_b32 v0, a0", "s_nop 15", PRODUCT, "s_cbranch_vccnz .LBB0_1"], False),
    (["v_cvt_pk_bf16_f32 v3, v20, v21", "s_nop 0", PRODUCT], False),
    (["v_cvt_pk_bf16_f32 v3, v20, v21", "s_nop 1", PRODUCT], True),
    # a scalar from a vector instruction: 5 to the memory instruction that reads it
    (["v_readfirstlane_b32 s40, v148", "s_and_b32 s41, s2, 0xffff", "s_add_i32 s2, s49, s56", "s_mov_b32 m0, s2", "s_nop 0", REQUEST], False),
    (["v_readfirstlane_b32 s40, v148", "s_nop 4", REQUEST], True),
    (["v_readlane_b32 s78, v148, 3", "s_nop 2", REQUEST], False),
    (["s_mov_b32 s40, s2", REQUEST], True),
    (["v_readfirstlane_b32 s40, v148", "s_add_i32 s40, s40, s2"], True),
    (["v_div_scale_f32 v133, s[0:1], v132, v132, 1.0", "global_store_dword v12, v133, s[4:5]"], True),
    (["v_div_scale_f32 v133, s[4:5], v132, v132, 1.0", "global_store_dword v12, v133, s[4:5]"], False),
])
def test_what_is_found(lines, ok):
    if ok:
        asm_check.check(function(*lines), "k.hip")
    else:
        with pytest.raises(RuntimeError, match="k.hip: 1 hazards"):
            asm_check.check(function(*lines), "k.hip")


def test_kernels_with_asm_products_are_looked_through():
    named = {s.name for s in build._group_sources("kernels")[0] if build.has_asm_mfma(s)}
    assert {"attention_prefill_long.hip", "attention_prefill_pairs.hip", "gemm4w.hip", "gemm4w_narrow.hip", "gemm4w_rows192.hip",
            "gemm4w_rows320.hip"} <= named
    with pytest.raises(RuntimeError, match="8 B/lane"):
        build.check_scratch("x: remark: Function Name: _Z19prefill_long_kernelILi0EEv\nx: remark: ScratchSize [bytes/lane]: 8\n", "x")


def assembly(name, tmp_path):
    src, out = build.CSRC / "kernels" / name, tmp_path / "k.s"
    subprocess.run([build._hipcc(), *build.KERNEL_FLAGS, "-I", str(src.parent), "--offload-device-only", "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    return out.read_text()


@pytest.mark.parametrize("src", ["attention_prefill_long.hip", "attention_prefill_pairs.hip"])
def test_long_attention(src, tmp_path):
    text = assembly(src, tmp_path)
    assert sum(fn.name.startswith("_Z19prefill_long_kernel") for fn in asm_check.functions(text)) == 2
    asm_check.check(text, src)


# hipcc does not count LDS-DMA that is asked for in asm statements: what it waits for, and where, is only its own loads' business. So
# the source itself waits for a tile's values between their request and the transposed reads of them, in every iteration
def test_values_of_the_mixing_attention_are_waited_for(tmp_path):
    text = assembly("mix_attention.hip", tmp_path)
    asked = re.sub(r"#ASMSTART\n\ts_waitcnt vmcnt\(0\)", "#ASMSTART\n\ts_asked", text)
    forms = [fn for fn in asm_check.functions(asked) if "mix_attention_kernelILb0E" in fn.name]
    assert len(forms) == 2                                  # one value tile a wave, and two

    def unwaited(fn, at):
        """The transposed reads that can follow ``at`` without such a wait."""
        seen, todo = set(), list(fn.following(at))
        while todo:
            n = todo.pop()
            if n not in seen and fn.code[n][0] != "s_asked":
                seen.add(n)
                todo += fn.following(n)
        return {n for n in seen if fn.code[n][0].startswith("ds_read_b64_tr")}

    for fn in forms:
        where = lambda name: [n for n, c in enumerate(fn.code) if c[0].startswith(name)]  # noqa: E731
        reads, requests = where("ds_read_b64_tr"), where("global_load_lds")
        assert reads and requests and not unwaited(fn, 0)
        assert all(min(unwaited(fn, n), default=n + 1) > n for n in reads)      # (nor once round the loop)
        if "ILb0ELi1E" in fn.name:                          # (two tiles: the reads behind a request are of the other one)
            assert not any(unwaited(fn, n) for n in requests)


# an output gate's four rows are asked for together: hipcc waits for all loads in flight ahead of each where a condition stands before it
def test_gate_rows_of_the_matrix_memory(tmp_path):
    text = assembly("recurrent_chunk.hip", tmp_path)
    forms = [fn for fn in asm_check.functions(text) if re.search(r"recurrence_chunk_kernelI[tf]Li\d+ELi3ELb0ELb0E", fn.name)]
    assert len(forms) == 6                                  # three widths, outputs in 16 and in 32 bits
    for fn in forms:
        starts, waited = set(fn.labels.values()), 0
        loop = [n for n, c in enumerate(fn.code) if c[0] == "s_barrier"][1]
        for n, (name, _, _) in enumerate(fn.code):
            if n < loop or not name.startswith("global_load"):
                continue
            n -= 1
            while fn.code[n][0] != "s_waitcnt" and n + 1 not in starts and not fn.code[n][0].startswith(("s_cbranch", "global_", "ds_")):
                n -= 1
            waited += fn.code[n][0] == "s_waitcnt" and "vmcnt(0)" in " ".join(fn.code[n][1])
        assert waited <= 1, fn.name
