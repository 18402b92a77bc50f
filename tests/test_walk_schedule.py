"""The 4-state walks' schedule (netrax_amd/csrc/schedule.cpp) checked on
the CPU: tests/walk_check.cpp replays the depth-first op order and the LDS
slots of the forward and reverse walks (a slot holds the row that is read
from it, HBM rows are loaded, one op ahead, after they are complete, first and accumulated
deliveries), whole and cut into launches as under a memory budget, for every
slot count.  A memory budget that the order by levels can meet can be met
in the depth-first order too."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from netrax_amd.network import parse_newick, random_network

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SAMPLES = os.path.join(HERE, "golden", "sample_networks")
HIP_INCLUDE = "/opt/rocm/include"
CASES = [(s, p) for s in (2, 3, 4, 5, 6, 8, 14, 32) for p in (1, 2, 3, 7, 1 << 20)]


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.isdir(HIP_INCLUDE):
        pytest.skip("g++ or the HIP headers are not available")
    exe = str(tmp_path_factory.mktemp("walk") / "walk_check")
    csrc = os.path.join(ROOT, "netrax_amd", "csrc")
    cmd = [gxx, "-std=c++17", "-O1", f"-I{HIP_INCLUDE}", "-D__HIP_PLATFORM_AMD__",
           os.path.join(HERE, "walk_check.cpp"), os.path.join(csrc, "schedule.cpp"),
           os.path.join(csrc, "dag.cpp"), "-o", exe]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    return exe


def _run(exe, net):
    head = [net.n_nodes, net.n_tips, net.root, len(net.edge_parent), len(net.retic_first_edge)]
    body = [*head, *net.edge_parent, *net.edge_child, *net.retic_first_edge, *net.retic_second_edge]
    text = " ".join(str(int(x)) for x in body) + "\n" + "\n".join(" ".join(map(str, c)) for c in CASES) + "\n"
    r = subprocess.run([exe], input=text, capture_output=True, text=True, timeout=120)
    lines = r.stdout.strip().split("\n")
    assert r.returncode == 0 and len(lines) == len(CASES) + 1 and all(x.startswith("ok") for x in lines[:-1]), r.stdout
    depth_first, by_level = (int(x) for x in lines[-1].split()[1:])
    return depth_first, by_level, [int(x.split()[4]) for x in lines[:-1]]


@pytest.mark.parametrize("name", sorted(f for f in os.listdir(SAMPLES) if f.endswith(".nw")))
def test_walks_of_reference_sample_networks(checker, name):
    with open(os.path.join(SAMPLES, name)) as f:
        net = parse_newick(f.read().strip())
    depth_first, by_level, _ = _run(checker, net)
    assert depth_first <= by_level, (depth_first, by_level)


def test_walks_of_random_networks(checker):
    rng = np.random.default_rng(77)
    handoffs = 0
    for _ in range(40):
        net = random_network(int(rng.integers(3, 90)), int(rng.integers(0, 7)), rng)
        depth_first, by_level, n = _run(checker, net)
        assert depth_first <= by_level, (depth_first, by_level)
        handoffs += sum(n)
    assert handoffs > 0
