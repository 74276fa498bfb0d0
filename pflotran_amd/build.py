"""Build libpfx_chem.so (HIP, gfx950) in-tree with hipcc.

    python -m pflotran_amd.build
"""
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libpfx_chem.so")
ARCH = os.environ.get("PFX_OFFLOAD_ARCH", "gfx950")


def units(defines=()):
    """(source, defines) of every object: the reaction kernels' instantiations
    are split into parts of their own, so that the objects compile in parallel.
    The profiling build (PFX_SECTION_TIMERS) keeps them in one, with one set of
    counters."""
    parts = [()] if "PFX_SECTION_TIMERS" in defines else [(f"PFX_REACT_PART={p}",) for p in (2, 3, 1, 0)]
    return [("pfx_react.hip", tuple(defines) + p) for p in parts] + [
        (s, tuple(defines)) for s in ("pfx_api.hip", "pfx_mlp.hip", "pfx_gi.hip", "pfx_krylov.hip")]


def hipcc_cmd(out, source, defines=()):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    return [hipcc, f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC"] + [f"-D{d}" for d in defines] + [
            # no packed-FP32 instructions in device code
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
            "-Wall", "-Wno-unused-variable", "-Wno-unused-but-set-variable",
            "-c", os.path.join(CSRC, source), "-o", out]


def build(verbose=True, out=LIB, defines=()):
    with tempfile.TemporaryDirectory(prefix="pfx_build_") as tmp:
        objs, running = [], []
        for k, (source, unit_defines) in enumerate(units(defines)):
            objs.append(os.path.join(tmp, f"{k}.o"))
            cmd = hipcc_cmd(objs[-1], source, unit_defines)
            if verbose:
                print(" ".join(cmd), flush=True)
            running.append((cmd, subprocess.Popen(cmd)))
        failed = [cmd for cmd, p in running if p.wait() != 0]
        if failed:
            raise subprocess.CalledProcessError(1, failed[0])
        link = [running[0][0][0], f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", out + ".tmp"] + objs
        subprocess.run(link, check=True)
    os.replace(out + ".tmp", out)
    return out


if __name__ == "__main__":
    build()
    sys.exit(0)
