"""Register, LDS and scratch budget of the kernels (CPU: compiles the sources
for gfx950 and reads the compiler's resource report).

The stage kernels are tuned for a number of workgroups resident per CU, which
their registers and their LDS have to allow together: FP64 k_rhs_tiled four in
3D (0.676 -> 0.510 ms per launch at 128^3 when it went from three), FP32 five,
k_rhs_wide three, k_rhs_small two in FP32 (its dispatch counts on them).  A
change that crosses one of those lines must show up here rather than in the
benchmark.  None of the 20 uses scratch memory: the runtime sets that up at a
kernel's first launch on a stream."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def resources(src_name, tmp_path):
    from smaug_amd.build import HIPCC_FLAGS

    flags = [f for f in HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    src = os.path.join(ROOT, "smaug_amd", "csrc", src_name)
    p = subprocess.run([HIPCC, *flags, "--cuda-device-only", "-c", src, "-o", str(tmp_path / "k.o"),
                        "-Rpass-analysis=kernel-resource-usage"], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr[-3000:]
    report = {}
    name = None
    for line in p.stderr.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        if m:
            name = m.group(1)
            report[name] = {}
            continue
        m = re.search(r"remark:\s+(VGPRs|AGPRs|ScratchSize \[bytes/lane\]|Occupancy \[waves/SIMD\]|LDS Size \[bytes/block\]): (\d+)", line)
        if m and name:
            report[name][m.group(1).split()[0]] = int(m.group(2))
    return report


# kernel (mangled name part): threads, workgroups a CU has to hold
LDS_PER_CU = 160 * 1024
STAGE_KERNELS = {
    "k_rhs_tiledILi3EdE": (256, 4),
    "k_rhs_tiledILi3EfE": (256, 5),
    "k_rhs_tiledILi3ENS_4DualEE": (512, 1),
    "k_rhs_tiledILi3ENS_5DualFEE": (512, 2),
    "k_rhs_tiledILi2EdE": (256, 4),
    "k_rhs_tiledILi2EfE": (256, 4),
    "k_rhs_tiledILi2ENS_4DualEE": (256, 2),
    "k_rhs_tiledILi2ENS_5DualFEE": (256, 4),
    "k_rhs_generalILi3EdE": (256, 4),
    "k_rhs_generalILi3EfE": (256, 5),
    "k_rhs_generalILi3ENS_4DualEE": (512, 1),
    "k_rhs_generalILi3ENS_5DualFEE": (512, 2),
    "k_rhs_generalILi2EdE": (256, 4),
    "k_rhs_generalILi2EfE": (256, 4),
    "k_rhs_generalILi2ENS_4DualEE": (256, 2),
    "k_rhs_generalILi2ENS_5DualFEE": (256, 4),
    "k_rhs_smallIdE": (256, 1),
    "k_rhs_smallIfE": (256, 2),
    "k_rhs_smallINS_5DualFEE": (256, 1),
    "k_rhs_wideE": (256, 3),
}


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_k_rhs_occupancy_and_scratch(tmp_path):
    from smaug_amd.build import ARCH

    assert ARCH == "gfx950"
    report = resources("smaug_rhs.hip", tmp_path)
    found = {}
    for part in STAGE_KERNELS:
        names = [k for k in report if part in k]
        assert len(names) == 1, (part, names)
        found[names[0]] = part
    assert set(found) == set(report), set(report) - set(found)  # every stage kernel is listed
    for name, part in found.items():
        v, (threads, groups) = report[name], STAGE_KERNELS[part]
        assert v["ScratchSize"] == 0, (part, v)
        assert v["Occupancy"] * 4 * 64 >= groups * threads, (part, v)
        assert v["LDS"] * groups <= LDS_PER_CU, (part, v)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_adjoint_kernels_plain_registers(tmp_path):
    """The adjoint kernels use no accumulation registers and no scratch and
    keep at least three wavefronts per SIMD (each term group is its own
    launch so no instantiation needs the register file of a whole step)."""
    report = resources("smaug_adj.hip", tmp_path)
    assert len(report) > 10
    for k, v in report.items():
        assert v.get("AGPRs", 0) == 0, (k, v)
        assert v["ScratchSize"] == 0, (k, v)
        assert v["Occupancy"] >= 3, (k, v)
