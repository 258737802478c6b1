"""Kernels whose wavefronts bounce activations through LDS of their own have no workgroup barrier between a lane's stores and the reads of other
lanes' data: both must be held in place by a wavefront fence and barrier, or nothing but alias analysis keeps the compiler from moving one past
the other.  Checked on the IR in front of the optimiser, where the function that bounces is one of its own for every instantiation."""
import os
import re
import subprocess

import pytest

from vllm_amd import build as vbuild

ORDER = "lds_lanes_in_order"


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc"), reason="no hipcc")
@pytest.mark.parametrize("kernel", ["rows", "decode", "skinny"])
def test_private_bounce_is_ordered(tmp_path, kernel):
    out = tmp_path / "k.ll"
    cmd = [vbuild.hipcc_path()] + [f for f in vbuild.HIPCC_FLAGS if f not in ("-shared", "-fPIC")] + [
        "--cuda-device-only", "-Xclang", "-disable-llvm-passes", "-emit-llvm", "-S", os.path.join(vbuild.CSRC, f"gemm_{kernel}.hip"), "-o", str(out)]
    subprocess.run(cmd, check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    kernels, ordered = set(), set()
    for body in re.split(r"\n(?=define )", out.read_text()):
        head = body.split("{", 1)[0]
        if ORDER in head:
            assert re.search(r'fence syncscope\("wavefront"\) acq_rel', body) and "llvm.amdgcn.wave.barrier" in body
        name = re.search(rf"@_Z(Z?)N5w4a16\d+{kernel}_kernelI((?:L[ib]\d+E)+)E", head)
        if not name:
            continue
        if not name.group(1):
            kernels.add(name.group(2))
        elif ORDER in body:
            at = [m.start() for m in re.finditer(rf"call [^\n]*{ORDER}", body)]
            stores = [m.start() for m in re.finditer(r"store <4 x i32>", body)]
            reads = [m.start() for m in re.finditer(r"load i32, ptr [^\n]*, align 4, !tbaa", body)]
            assert len(at) == 1 and stores[0] < at[0] and any(at[0] < r for r in reads), head
            ordered.add(name.group(2))
    assert len(kernels) >= 16
    assert ordered == kernels
