"""The kernels the benchmark names, and the traffic summaries it looks up for them, belong to kernels that
the library has."""
import glob
import os
import re

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# the first name of a kernel's form after each __global__ (its launch bounds hold none)
KERNELS = {name for path in glob.glob(os.path.join(ROOT, "utttcompanion_amd", "csrc", "*.hip"))
           for name in re.findall(r"__global__.*?\b(k_\w+)\(", open(path).read(), re.S)}


def test_update_phases_name_kernels_of_the_library():
    assert "k_update_write" in KERNELS and "k_chain_apply_wide" in KERNELS
    for phase in bench.PHASES:
        assert phase.split(" ")[0] in KERNELS, phase


def test_traffic_summaries_belong_to_kernels_of_the_library():
    found = 0
    for path in glob.glob(os.path.join(ROOT, "profiles", "*_traffic.md")):
        for name in re.findall(r"^traffic_bytes_per_launch (\w+):", open(path).read(), re.M):
            assert name in KERNELS, (path, name)
            found += 1
    for path in glob.glob(os.path.join(ROOT, "profiles", "k_*_traffic.md")):
        name = re.match(r"(k_\w+)_c\d_traffic\.md", os.path.basename(path)).group(1)
        assert any(k.startswith(name) for k in KERNELS), path
        found += 1
    assert found > 0
    assert bench.measured_traffic("k_update_write") == 614102957
    assert bench.measured_traffic("k_apply") is None
