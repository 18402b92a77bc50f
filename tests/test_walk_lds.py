"""The 20-state walks' workgroups that a CU gets fit its LDS together, with the
dynamic LDS of their slots and what the built kernels declare besides
(group_segment_fixed_size of the code object).  CPU only."""
import os
import shutil
import subprocess

import pytest

from code_object import kernels

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIP_INCLUDE = "/opt/rocm/include"
CUS, LDS_PER_CU, PIECE = 256, 160 * 1024, 1280


@pytest.fixture(scope="module")
def fixed_lds(tmp_path_factory):
    field = "group_segment_fixed_size"
    return {n: f[field] for n, f in kernels(tmp_path_factory.mktemp("codeobj"), field).items() if field in f}


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.isdir(HIP_INCLUDE):
        pytest.skip("g++ or the HIP headers are not available")
    exe = str(tmp_path_factory.mktemp("lds") / "walk_lds_check")
    csrc = os.path.join(ROOT, "netrax_amd", "csrc")
    subprocess.run([gxx, "-std=c++17", "-O1", f"-I{HIP_INCLUDE}", "-D__HIP_PLATFORM_AMD__",
                    os.path.join(HERE, "walk_lds_check.cpp"), os.path.join(csrc, "schedule.cpp"),
                    os.path.join(csrc, "dag.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("ncat", [1, 2, 4, 8])
def test_planned_workgroups_fit_a_cu(fixed_lds, planner, ncat, fp32):
    forward = f"k_forward_mfmaILi{ncat}ELi4E" if fp32 else f"k_forward_level_aaILi{ncat}E"
    reverse = f"k_adjoint_mfmaILi{ncat}E" if fp32 else f"k_adjoint_level_aaILi{ncat}E"
    fixed = []
    for fragment in (forward, reverse):
        hits = [size for name, size in fixed_lds.items() if fragment in name]
        assert len(hits) == 1, fragment
        fixed.append(hits[0])
    # waves of a CU by the kernels' registers (forward: workgroups of ncat waves)
    most = [max(1, (16 if fp32 else 12) // ncat), 12 if fp32 else 8]
    sites = list(range(64, 70000, 64))
    text = "".join(f"{ncat} {int(fp32)} {n}\n" for n in sites)
    lines = subprocess.run([planner], input=text, check=True, capture_output=True, text=True).stdout.split("\n")
    for n, line in zip(sites, lines):
        got = [int(x) for x in line.split()]
        for i, groups in enumerate((n // 16, n // 16 * ncat)):
            per_cu = min(most[i], -(-groups // CUS))
            slots, dynamic = got[2 * i], got[2 * i + 1]
            held = -(-(dynamic + fixed[i]) // PIECE) * PIECE
            assert slots == 2 or held * per_cu <= LDS_PER_CU, (n, i, got, fixed)
