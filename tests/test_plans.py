"""CPU checks of the launch arithmetic that kernels and host code share
(diskmule_amd/csrc/dm_plan.h): the header is compiled with the host compiler
and its functions are run over whole ranges of sizes."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include "dm_plan.h"
extern "C" {
uint32_t experts_grid(uint32_t cus, uint32_t pairs) { return dm::experts_grid(cus, pairs); }
uint32_t experts_share(uint32_t grid, uint32_t entries) { return dm::experts_share(grid, entries); }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plans")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "diskmule_amd", "csrc"), str(d / "shim.cpp"), "-o", str(d / "shim.so")],
                   check=True)
    lib = ctypes.CDLL(str(d / "shim.so"))
    for name in ("experts_grid", "experts_share"):
        getattr(lib, name).restype = ctypes.c_uint32
    return lib


def test_every_grouped_expert_entry_has_workgroups(plan):
    """Whatever the CU count (a partition may show 32 or fewer) and however
    the pairs fall on experts (1 to `pairs` entries), every entry is some
    workgroup's, each entry's workgroups are numbered 0 .. share - 1, and a
    whole MI355X keeps two workgroups per CU."""
    for cus in (1, 4, 16, 31, 32, 38, 64, 80, 128, 256, 304):
        for pairs in range(1, 129):
            grid = plan.experts_grid(cus, pairs)
            assert grid >= 2 * cus
            for entries in range(1, pairs + 1):
                share = plan.experts_share(grid, entries)
                assert share >= 1 and (entries - 1) * share + share - 1 < grid, (cus, pairs, entries)
    assert all(plan.experts_grid(256, pairs) == 512 for pairs in range(1, 129))
