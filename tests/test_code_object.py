"""The built gfx950 code object, by its own metadata (CPU only): no kernel spills
registers to memory or has a stack, and the projection tiles bounded for two or
three workgroups a CU leave each of them the LDS for it."""
import re
import subprocess

import g4a

LLVM = "/opt/rocm/llvm/bin/"
LDS = 160 * 1024  # of a CU


def _kernels(tmp_path):
    co = tmp_path / "kernels.co"
    subprocess.run([LLVM + "clang-offload-bundler", "--unbundle", "--type=o", f"--input={g4a.HSACO_PATH}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={co}"], check=True)
    notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(co)], check=True, capture_output=True, text=True).stdout
    kernels = {}
    for block in notes.split("- .agpr_count:")[1:]:
        field = dict(re.findall(r"\n    \.(\w+): +(\S+)", block))
        kernels[field["name"]] = field
    return kernels


def test_no_kernel_spills_and_bounded_workgroups_fit(tmp_path):
    kernels = _kernels(tmp_path)
    assert "g4a_decode_d256_g8" in kernels and "g4a_linear_mm_0_b4_mode0" in kernels
    spilled = {n: (k["vgpr_spill_count"], k["private_segment_fixed_size"]) for n, k in kernels.items()
               if k["vgpr_spill_count"] != "0" or k["private_segment_fixed_size"] != "0"}
    assert not spilled
    for form, workgroups in ((1, 2), (3, 2), (4, 3)):
        for n, k in kernels.items():
            # (form 3 of two weights is bounded for one)
            if n.startswith(f"g4a_linear_mm_{form}_") and not (form == 3 and n.endswith("mode1")):
                assert workgroups * int(k["group_segment_fixed_size"]) <= LDS, n
