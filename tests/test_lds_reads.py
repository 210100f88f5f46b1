"""Reads of LDS that a kernel writes as instructions are unknown to the compiler, which takes their registers as filled at
once: nothing may touch these before the wait that the kernel writes behind them, and no branch may lie between, where the
compiler is free to move registers.  The device code of the sources that write such reads is compiled to text and looked
over, in straight lines; no GPU is needed."""
import re

import pytest

FUNCTION = re.compile(r"^(\w+):\s*; @\S+\n(.*?)^\.Lfunc_end", re.S | re.M)


def _registers(text):
    found = {(kind, int(n)) for kind, n in re.findall(r"\b([va])(\d+)\b", text)}
    for kind, first, last in re.findall(r"\b([va])\[(\d+):(\d+)\]", text):
        found |= {(kind, n) for n in range(int(first), int(last) + 1)}
    return found


def unwaited(assembly, kernel):
    """(reads written as instructions, what happens to their registers before a wait covers them) of the named kernel's
    instances."""
    reads, faults = 0, []
    for name, body in FUNCTION.findall(assembly):
        if kernel not in name:
            continue
        pending, written = [], False                # registers of the reads under way, oldest first (none: the compiler's own)
        for line in body.split("\n"):
            if "#ASMSTART" in line or "#ASMEND" in line:
                written = "#ASMSTART" in line
                continue
            line = line.split(";")[0].strip()
            if not line or (line.startswith(".") and not line.endswith(":")):
                continue
            if line.endswith(":") or line.startswith(("s_cbranch", "s_branch")):
                if any(pending):
                    faults.append(f"{name}: {line} with reads under way")
                continue
            wait = re.match(r"s_waitcnt.*?lgkmcnt\((\d+)\)", line)
            if wait:                                # LDS answers in order
                pending = pending[max(0, len(pending) - int(wait[1])):]
                continue
            if any(regs & _registers(line) for regs in pending):
                faults.append(f"{name}: {line} before the wait")
            if line.startswith("ds_"):
                own = written and line.startswith("ds_read")
                reads += own
                pending.append(_registers(line.split(",")[0]) if own else set())
    return reads, faults


@pytest.mark.parametrize("source, kernel", [("gemm.hip", "gemm_fma_flow_kernel"),
                                            ("grouped_gemm.hip", "grouped_gemm_tile_kernel"),
                                            ("latent_attention.hip", "latent_attention_prompt_kernel"),
                                            ("gemm_mfma.hip", "gemm_tile_kernel"),
                                            ("gemm_mfma.hip", "gemm_small_tile_kernel"),
                                            ("gemm_mfma.hip", "gemm_rows_kernel"),
                                            ("attention_mfma.hip", "attention_prefill_kernel"),
                                            ("attention_mfma.hip", "attention_decode_kernel"),
                                            ("state_space.hip", "state_space_walk_kernel")])
def test_nothing_comes_between_a_read_and_its_wait(device_code, source, kernel):
    reads, faults = unwaited(device_code(source, "float32" if source == "gemm.hip" else "bfloat16"), kernel)
    assert reads > 0 and not faults, faults[:5]


def test_the_look_finds_what_it_is_for():
    def text(*lines):
        return "kernel_a:    ; @kernel_a\n" + "\n".join(lines) + "\n.Lfunc_end0:\n"
    read = ["\t;#ASMSTART", "\tds_read_b128 v[4:7], v1 offset:16", "\t;#ASMEND"]
    assert unwaited(text(*read, "\ts_waitcnt lgkmcnt(0)", "\tv_mov_b32 v9, v4"), "kernel") == (1, [])
    assert len(unwaited(text(*read, "\tv_mov_b32 v9, v6", "\ts_waitcnt lgkmcnt(0)"), "kernel")[1]) == 1
    assert len(unwaited(text(*read, "\ts_cbranch_scc0 .LBB0_3", "\ts_waitcnt lgkmcnt(0)"), "kernel")[1]) == 1
    younger = [line.replace("[4:7]", "[8:11]") for line in read]
    assert unwaited(text(*read, *younger, "\ts_waitcnt lgkmcnt(1)", "\tv_mov_b32 v9999, v5"), "kernel") == (2, [])
    assert len(unwaited(text(*read, *younger, "\ts_waitcnt lgkmcnt(1)", "\tv_mov_b32 v1, v9"), "kernel")[1]) == 1
