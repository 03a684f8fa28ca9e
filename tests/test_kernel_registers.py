"""Registers of the Kaczmarz kernels, from the compiler's resource report: how
many workgroups share a CU depends on them (512 registers per SIMD lane, four
SIMDs per CU)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# kernel, at most so many registers: kLeanSlots leaves room for two workgroups of
# 512 threads with variable lanes (FP32: beside two with uniform lanes), kFewSlots
# for five of 256 threads in FP64 and FP32 (8 and 16 entries a lane)
LIMITS = [("k_kacz_flow_vl<512, float, float, true, kLeanSlots>", 96),
          ("k_kacz_flow_vl<512, double, double, true, kLeanSlots>", 128),
          ("k_kacz_flow<512, 4, 16, float, float, true, kLeanSlots>", 80),
          ("k_kacz_flow<512, 4, 16, double, double, true, kLeanSlots>", 128),
          ("k_kacz_bundle<256, 1, 8, double, double, false, kFewSlots>", 96),
          ("k_kacz_bundle<256, 1, 8, float, float, false, kFewSlots>", 72),
          ("k_kacz_bundle<256, 2, 16, float, float, false, kFewSlots>", 102),
          ("k_kacz_flow<256, 2, 16, float, float, false, kFewSlots>", 102)]


def test_registers_leave_room_for_several_workgroups(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    src = tmp_path / "kernels.hip"
    src.write_text('#include "bundle_exec.hpp"\nnamespace race {\nconst void* volatile kernels[] = {\n'
                   + "".join(f"    reinterpret_cast<const void*>(&{k}),\n" for k, _ in LIMITS) + "};\n}\n")
    r = subprocess.run([hipcc, "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only",
                        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-Rpass-analysis=kernel-resource-usage", "-I", os.path.join(ROOT, "race_amd", "csrc"),
                        "-c", str(src), "-o", str(tmp_path / "kernels.o")],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    seen = {}
    for block in r.stderr.split("Function Name: ")[1:]:
        name = block.split()[0]
        seen[name] = (int(re.search(r" VGPRs: (\d+)", block).group(1)), int(re.search(r"VGPRs Spill: (\d+)", block).group(1)))
    slots = {"kLeanSlots": 2, "kFewSlots": 4}
    code = {"float": "f", "double": "d", "true": "Lb1E", "false": "Lb0E"}
    for kernel, limit in LIMITS:
        name, args = re.match(r"(\w+)<(.*)>", kernel).groups()
        mangled = "".join(code.get(a) or f"Li{slots.get(a, a)}E" for a in args.split(", "))
        found = [v for k, v in seen.items() if f"{len(name)}{name}I{mangled}E" in k]
        assert len(found) == 1, (kernel, sorted(seen))
        assert found[0][0] <= limit and found[0][1] == 0, (kernel, found)
