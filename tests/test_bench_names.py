"""The kernels that bench.py reports on are kernels of the built library."""
import pytest

import bench
from code_object import kernels


@pytest.fixture(scope="module")
def names(tmp_path_factory):
    return list(kernels(tmp_path_factory.mktemp("codeobj"), "vgpr_count"))


@pytest.mark.parametrize("ncat", [1, 4, 8])
@pytest.mark.parametrize("sites", [64, 41408, 65536, 1 << 20])
@pytest.mark.parametrize("group", [2, 3, 4, 8])
def test_batched_kernels_exist(names, group, sites, ncat):
    for step in ("forward", "adjoint"):
        name = bench.batched_kernel(step, group, sites, ncat)
        stem, args = name[:-1].split("<")
        mangled = stem + "I" + "".join(f"Li{int(a)}E" for a in args.split(",")) + "E"
        assert any(mangled in n for n in names), name


def test_reported_kernels_of_the_headline_workload(names):
    class Stats:
        fwd_op_bytes, adj_bytes, n_sites_padded = 1e9, 2e9, 41408

    res = dict(stats=Stats, fwd_ms_per_eval=0.1, fwd_launches_per_eval=1, adj_ms_per_eval=0.2, adj_launches_per_eval=1)
    for tuning in (None, {"group_width": 4, "tile_sites": 64, "row_lanes": 1},
                   {"group_width": 3, "tile_sites": 32, "row_lanes": 2}):
        for t in (0.1, 0.3):
            r = bench.roofline(dict(res, fwd_ms_per_eval=t, tuning=tuning))
            assert r["traffic"], r["kernel"]  # a kernel that the committed counters were taken of
