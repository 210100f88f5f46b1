"""What the device code shows of kernels whose speed rests on it: how many waves a SIMD holds, and how outputs are stored."""
import re

import pytest


def functions(assembly, kernel):
    """{an instance of the kernel: its instructions}."""
    found = {name: body for name, body in re.findall(r"^(\w+):\s*; @\S+\n(.*?)^\.Lfunc_end", assembly, re.S | re.M) if kernel in name}
    assert found
    return found


@pytest.mark.parametrize("source, kernel, most", [("attention_mfma.hip", "attention_combine_kernel", 128)])
def test_registers_leave_room_for_the_waves(device_code, source, kernel, most):
    """A SIMD has 512 registers a lane and hands them out to a wave in eights, so 128 are four waves."""
    seen = 0
    for note in re.findall(r"- \.agpr_count:.*?\.wavefront_size:", device_code(source), re.S):
        field = {k: v for k, v in re.findall(r"\.(\w+):\s+(\S+)", note)}
        if kernel in field["symbol"]:
            seen += 1
            assert int(field["vgpr_count"]) <= most and int(field["private_segment_fixed_size"]) == 0, field
    assert seen


def test_sums_of_segments_leave_the_tiles_across_lanes(device_code):
    """A 16-byte store whose lanes hold four columns of sixteen rows each meets 64 lines, four stores of 4 bytes whose lanes hold
    sixteen columns meet 16: each tile has a form whose 32-bit values (segments' sums, rows added into) leave that way."""
    across = 0
    for name, body in functions(device_code("gemm_mfma.hip"), "gemm_tile_kernel").items():
        stores = set(re.findall(r"\b(global_store_\w+)", body))
        across += "global_store_dword" in stores and not stores & {"global_store_dwordx2", "global_store_dwordx4"}
    assert across >= 5                # 256 columns, gated and not, 192, and kept ones, gated and not


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_32_bit_products_of_few_rows_spill_nothing(device_code, dtype):
    seen = set()
    for note in re.findall(r"- \.agpr_count:.*?\.wavefront_size:", device_code("gemm.hip", dtype), re.S):
        field = {k: v for k, v in re.findall(r"\.(\w+):\s+(\S+)", note)}
        kernel = re.search(r"gemm_fma_(few_rows|by_chain)_kernel", field["symbol"])
        if kernel:
            seen.add(kernel[1])
            assert int(field["vgpr_spill_count"]) == 0 and int(field["private_segment_fixed_size"]) == 0, field
    assert seen == {"few_rows", "by_chain"}
