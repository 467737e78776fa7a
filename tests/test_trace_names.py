"""trace_summary.short(): the names of a kernel trace against those of the solver's launch
accounting, for every SpMV kernel the library was built with."""
import os
import re
import shutil
import subprocess

import pytest
from conftest import PKG


def test_names_as_the_launch_accounting():
    from trace_summary import short

    pre = "void xh::(anonymous namespace)::"
    tail = "(unsigned int const*, xh::(anonymous namespace)::GridCol const*, double const*)"
    for trace, want in (
            ("k_spmv<double, unsigned short, 32, 6, 8>", "k_spmv<double,u16,32,OP_CHEB>"),
            ("k_spmv<double, unsigned int, 8, 2, 16>", "k_spmv<double,u32,8,OP_RESID,16>"),
            ("k_spmv<double, xh::(anonymous namespace)::GridCol, 8, 3, 8>",
             "k_spmv<double,grid,8,OP_DOT1>"),
            ("k_spmv_wave<float, unsigned short, 1, 2, 4>", "k_spmv_wave<float,u16,1,OP_RESID,4>"),
            ("k_spmv_wave<double, unsigned int, 64, 12, 16>",
             "k_spmv_wave<double,u32,64,OP_CHEBR,16>"),
            ("k_spmv_sweep<double, 32, 4>", "k_spmv_sweep<double,32,OP_DOT3>"),
            ("k_spmv_st7<double, 32, 6>", "k_spmv_st7<double,32,OP_CHEB>"),
            ("k_vec<32, 1>", "k_vec<32,V_XR_UPDATE>")):
        assert short(pre + trace + tail) == want


def test_every_built_spmv_kernel_has_a_name():
    from trace_summary import short

    if shutil.which("nm") is None:
        pytest.skip("nm not found")
    out = subprocess.run(["nm", "-C", os.path.join(PKG, "lib", "libxamg_hip.so")],
                         capture_output=True, text=True, check=True).stdout
    names = {m.group(1) for m in re.finditer(r"__device_stub__(k_spmv[^\n]*)", out)}
    assert len(names) > 300
    for n in names:
        assert re.search(r"<(double|float),((u8|u16|u32|grid),)?\d+,OP_\w+(,\d+)?>$", short(n)), n
