"""The build's check of the kernels' registers and occupancy (csrc/check_usage.awk): what it passes and what it stops."""
import os
import subprocess

import pytest

AWK = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-llm_amd", "csrc", "check_usage.awk")


def accepted(kernel, vgprs, occupancy):
    remarks = (f"x.hip:1:1: remark: Function Name: _ZN12_GLOBAL__N_1{len(kernel)}{kernel}EPKi [-R]\n"
               f"x.hip:1:1: remark:     VGPRs: {vgprs} [-R]\n"
               f"x.hip:1:1: remark:     Occupancy [waves/SIMD]: {occupancy} [-R]\n")
    r = subprocess.run(["awk", "-f", AWK], input=remarks, capture_output=True, text=True)
    assert (r.returncode == 0) == (r.stdout == "")
    return r.returncode == 0


@pytest.mark.parametrize("kernel,vgprs,occupancy", [("spmm_stream_kernel", 250, 2), ("spmm_group_kernel", 168, 3),
                                                    ("spmm_wide_kernel", 234, 2), ("spmm_quarter_kernel", 218, 1), ("encode_tiles_kernel", 79, 6)])
def test_a_kernel_below_its_occupancy_stops_the_build(kernel, vgprs, occupancy):
    assert accepted(kernel, vgprs, occupancy)
    assert not accepted(kernel, vgprs, occupancy - 1)


@pytest.mark.parametrize("kernel,vgprs,occupancy", [("spmm_group_kernel", 169, 3), ("spmm_wide_kernel", 241, 2), ("spmm_quarter_kernel", 233, 1), ("spmm_even_kernel", 233, 1)])
def test_a_kernel_with_more_registers_than_measured_stops_the_build(kernel, vgprs, occupancy):
    assert not accepted(kernel, vgprs, occupancy)
