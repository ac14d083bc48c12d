"""The device layout of a scene's trees (yrh_internal.h LayOutArena) on the
host: where its parts lie, and how large they may be."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")

PROGRAM = r"""
#include "yrh_internal.h"
#include <cstdio>
#include <cstdlib>
using namespace yrh;
int main(int argc, char** argv) {
    ArenaLayout a;
    const bool fits = LayOutArena(atoll(argv[1]), atoll(argv[2]), atoll(argv[3]), atoll(argv[4]), a);
    std::printf("%d %lld %lld %lld %lld", fits, (long long)a.slots, (long long)a.tlas_nodes, (long long)a.instances,
                (long long)a.units);
}
"""


@pytest.fixture(scope="module")
def layout(tmp_path_factory):
    d = tmp_path_factory.mktemp("arena")
    (d / "layout.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "yaoray_amd", "csrc"), "-I" + os.path.join(ROOT, "include"), "-w",
                    "-c", str(d / "layout.cpp"), "-o", str(d / "layout.o")], check=True)
    subprocess.run(["g++", str(d / "layout.o"), "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-o",
                    str(d / "layout")], check=True)

    def run(*counts):
        out = subprocess.run([str(d / "layout"), *map(str, counts)], check=True, capture_output=True, text=True).stdout
        return [int(x) for x in out.split()]

    return run


MAX_SLOT = 2**27 - 1


def test_parts_follow_each_other(layout):
    assert layout(1, 3, 2, 4) == [1, 4, 16, 24, 44]  # TLAS nodes on 64-byte lines
    assert layout(0, 1, 0, 0) == [1, 0, 4, 4, 4]
    assert layout(0, 0, 0, 0) == [1, 0, 0, 0, 0]


@pytest.mark.parametrize("counts, fits", [
    # The largest binary trees over disjoint leaves: MAX_SLOT slots in the
    # BLASes (or the flat tree) and as many in the TLAS, one per leaf.
    ((MAX_SLOT - 1, MAX_SLOT, 0, 0), 1),
    ((MAX_SLOT - 1, MAX_SLOT, MAX_SLOT - 1, MAX_SLOT), 1),
    ((1, 2, MAX_SLOT - 1, MAX_SLOT), 1),
    # Past what a code can name.
    ((2**29 + 1, 0, 0, 0), 0),
    ((2**28 + 1, 0, 1, 1), 0),
    ((MAX_SLOT - 1, MAX_SLOT, MAX_SLOT + 8, MAX_SLOT), 0),
])
def test_limits(layout, counts, fits):
    assert layout(*counts)[0] == fits
