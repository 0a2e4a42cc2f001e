"""How much of a run of pairs the neighbor list's emit may write (csrc/nlist_run.h), for lists that run past
the output by more than 32 bits of components: compiled and evaluated on the host."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "molnex_amd", "csrc")


@pytest.mark.parametrize("first,pairs,capacity,want", [
    (0, 32, 32, 96), (0, 32, 1 << 40, 96), (31, 5, 32, 3), (32, 5, 32, 0), (33, 5, 32, 0), (0, 0, 8, 0),
    ((1 << 40) - 2, 32, 1 << 40, 6),
    # 3 (capacity - first) below -2^31, where it once wrapped to a positive count
    (715_827_883, 32, 0, 0), (900_000_000, 32, 1000, 0), (1_431_655_765, 1, 0, 0), (1 << 40, 32, 7, 0),
])
def test_components_within_the_output(first, pairs, capacity, want, tmp_path):
    src = tmp_path / "run.cpp"
    src.write_text('#include "nlist_run.h"\n'
                   f"static_assert(mnx::run_components(INT64_C({first}), {pairs}, INT64_C({capacity})) == {want});\n")
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", f"-I{CSRC}", str(src)], check=True, timeout=60)

