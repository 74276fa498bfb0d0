"""The objects of the library, in the product build and in the profiling
build: together they define every C entry of the reaction kernels' file that the
build has, once (the host side preprocessed; nothing is compiled)."""
import os
import subprocess

import pytest

from pflotran_amd import build


@pytest.mark.parametrize("defines,entries", [((), {"pfx_scr_bytes": 1, "pfx_section_cycles": 0}),
                                             (("PFX_SECTION_TIMERS",), {"pfx_scr_bytes": 1, "pfx_section_cycles": 1})])
def test_entries_are_defined_once(defines, entries):
    if not os.path.exists(os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")):
        pytest.skip("no hipcc")
    text = ""
    for source, unit_defines in build.units(defines):
        if source != "pfx_react.hip":
            continue
        cmd = build.hipcc_cmd("-", source, unit_defines)
        cmd[cmd.index("-c")] = "-E"
        text += subprocess.run(cmd + ["-P", "--offload-host-only"], check=True, capture_output=True, text=True).stdout
    for name, count in entries.items():
        assert text.count(f'extern "C" int {name}(') == count, name
    for kernel in ("pfx_react_zones_kernel<1, false>", "pfx_react_zones_kernel<1, true>"):
        assert text.count(kernel) == 1
    for lanes in (8, 16, 32):
        assert text.count(f"pfx_react_kernel<{lanes}, PFX_MODE_AUX, 1,") == 1


def test_product_build_covers_every_source():
    for defines in ((), ("PFX_SECTION_TIMERS",)):
        names = {source for source, _ in build.units(defines)}
        assert names == {f for f in os.listdir(build.CSRC) if f.endswith(".hip")}
