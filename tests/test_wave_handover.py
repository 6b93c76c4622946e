"""Data that one wave hands to another of its workgroup in LDS: the count that
announces it has to be stored with release and read with acquire order at
workgroup scope, or nothing orders the data behind it.  Checked on the device
code before any optimisation, as compiled for gfx950."""
import os
import re
import subprocess

import pytest

from openrcwa_amd import build


@pytest.mark.parametrize("source", ["eig.hip", "rcwa_kernels.hip", "blas.hip", "smatrix.hip"])
def test_workgroup_atomics_order_what_they_announce(tmp_path, source):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    ir = tmp_path / "device.ll"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-Xclang",
                    "-disable-llvm-passes", "-S", "-emit-llvm", "-x", "hip",
                    os.path.join(build.CSRC, source), "-o", str(ir)], check=True,
                   capture_output=True)
    found = re.findall(r'\b(load|store) atomic .*syncscope\("workgroup"\) (\w+)', ir.read_text())
    order = {"load": "acquire", "store": "release"}
    assert all(how == order[op] for op, how in found), sorted(set(found))
    if source == "eig.hip":
        assert {op for op, _ in found} == {"load", "store"}
