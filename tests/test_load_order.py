"""The waits that count vector loads by hand, checked in the compiled code (no GPU needed).

A wave waits for its direct-to-LDS loads with s_waitcnt vmcnt(N), where N counts the younger loads that may
stay in flight.  Some of those are plain loads that the compiler places: were one of them moved out of
the stretch between the loads waited for and the wait, the wait would let the former through early."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "utttcompanion_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")


def kernels(source, tmp_path):
    """Of every kernel of a source: its stretches of code between barriers, each a list of the loads
    ("lds" or "plain") and wait counts (int) in it, and whether a barrier ended it."""
    asm = tmp_path / "k.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--offload-device-only", "-S", os.path.join(CSRC, source), "-o", str(asm)],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    found, now = {}, None
    for line in asm.read_text().splitlines():
        m = re.match(r"(_Z\w+):", line)
        if m:
            now = found.setdefault(m.group(1), [[]])
        elif now is not None:
            op = line.strip()
            if op.startswith(("buffer_load", "global_load")):
                now[-1].append("lds" if op.endswith(" lds") else "plain")
            elif m := re.match(r"s_waitcnt vmcnt\((\d+)\)", op):
                now[-1].append(int(m.group(1)))
            elif op.startswith("s_barrier"):
                now.append([])
            elif op.startswith(".Lfunc_end"):
                now = None
    return found


@pytest.mark.parametrize("source, name, plain, lds", [
    ("update_mm.hip", "k_update_back", 4, 2),
    ("readout_mm.hip", r"k_readout_mmILb[01]EfLi2ELi2ELi1ELi3E", 8, 2),  # the small fp32 tile, two steps ahead
])
def test_steps_ahead_are_the_last_loads_before_the_wait(source, name, plain, lds, tmp_path):
    """Each wait that leaves one step's loads in flight follows on exactly that step's loads."""
    seen = 0
    for kernel, stretches in kernels(source, tmp_path).items():
        if not re.search(name, kernel):
            continue
        for s in stretches[:-1]:  # the barrier that ends a stretch directly follows the hand-counted wait
            if s and s[-1] == plain + lds:
                loads = [x for x in s if not isinstance(x, int)][-(plain + lds):]
                assert (loads.count("plain"), loads.count("lds")) == (plain, lds), (kernel, s)
                seen += 1
    assert seen >= 4  # the first step and the loop's, of two kernels


def test_state_loads_stay_between_the_slabs_and_the_wait(tmp_path):
    """The state write waits for its slabs with its eight state loads in flight."""
    seen = 0
    for kernel, stretches in kernels("update_mm.hip", tmp_path).items():
        if not re.search(r"k_update_writeILNS0_9WriteFormE[12]E", kernel):
            continue
        first = stretches[0]
        last_lds = max(i for i, x in enumerate(first) if x == "lds")
        after = first[last_lds + 1:]
        waits = [i for i, x in enumerate(after) if x in (8, 12)]
        assert waits, (kernel, first)
        assert all(after[:i].count("plain") >= 8 for i in waits), (kernel, first)
        # one block's slabs (two pieces of each operand), and another's
        assert first.count("lds") == 8
        seen += 1
    assert seen == 2
