"""The reaction kernels' multi-instruction DPP statements where operands hold
the same value: an instruction of a statement may not read a register that an
earlier one of it has written, other than its own accumulator (compiled for the
device, the assembly read; nothing runs)."""
import os
import re
import subprocess

import pytest

from pflotran_amd import build

PROBE = """
#define PFX_REACT_PART 9   // no instantiation
#include "pfx_react.hip"
extern "C" __global__ void probe_self(double *p) {
  double *q = p + threadIdx.x;
  double a = q[0], b = q[64], c = q[128], d = q[192];
  fmac_bcast_self<3, 15, 15>(a, a, b, c, d);
  q[0] = a; q[64] = b; q[128] = c; q[192] = d;
}
extern "C" __global__ void probe_four(double *p) {
  double *q = p + threadIdx.x;
  double a = q[0], b = q[64], c = q[128], d = q[192];
  fmac_bcast4<5, 15, 15>(b, a, c, b, a, c, b, d, a);
  q[0] = a; q[64] = b; q[128] = c; q[192] = d;
}
"""


def test_operands_of_one_statement_do_not_overlap(tmp_path):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(PROBE)
    cmd = build.hipcc_cmd(str(out), str(src))
    cmd[cmd.index("-c")] = "-S"
    subprocess.run(cmd + ["--offload-device-only", "-I", build.CSRC], check=True, capture_output=True)
    found = 0
    for statement in re.findall(r"ASMSTART\n(.*?)ASMEND", out.read_text(), flags=re.S):
        ops = re.findall(r"v_fmac_f64_dpp (v\[\d+:\d+\]), (v\[\d+:\d+\]), (v\[\d+:\d+\])", statement)
        written = set()
        for dst, src0, src1 in ops:
            assert dst not in written and src0 not in written and src1 not in written, statement
            written.add(dst)
        found += len(ops) == 4
    assert found == 2
