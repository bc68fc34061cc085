"""The rules that choose an FP8 kernel and its shape (fp8_plan.h: sizes only, no
device), compiled for the host."""

from __future__ import annotations

import ctypes
import subprocess

import pytest

from conftest import REPO

SOURCE = """
#include "fp8_plan.h"
extern "C" {
long from(long rows, long blocks, int outs, int bf16) { return plm::panel_from(rows, blocks, outs, bf16); }
long mlp_from(long hidden, long inter, int bf16) { return plm::panel_mlp_from(hidden, inter, bf16); }
int tiles(long m, int one_plane) { return plm::panel_tiles(m, one_plane); }
int wr(long rows, int silu, long x_tiles, int waves, int cus) { return plm::panel_plan(rows, silu, x_tiles, waves, cus).wr; }
int splits(long rows, int silu, long x_tiles, int waves, int cus) {
    return plm::panel_plan(rows, silu, x_tiles, waves, cus).splits;
}
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    folder = tmp_path_factory.mktemp("plan")
    (folder / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{REPO / 'pocketlm_amd' / 'csrc'}",
                    str(folder / "plan.cpp"), "-o", str(folder / "plan.so")], check=True)
    lib = ctypes.CDLL(str(folder / "plan.so"))
    long, i = ctypes.c_long, ctypes.c_int
    for name, args in (("from", [long, long, i, i]), ("mlp_from", [long, long, i]), ("tiles", [long, i]),
                       ("wr", [long, i, long, i, i]), ("splits", [long, i, long, i, i])):
        getattr(lib, name).argtypes = args
        getattr(lib, name).restype = long
    return lib


@pytest.mark.parametrize("cus", [32, 64, 128, 256])
def test_panel_slots_are_split_only_where_the_split_kernel_runs(plan, cus):
    """The 128-row workgroups keep a tile's K slots together (launched several
    times over they would compute each tile that often), whatever the number
    of compute units; splits are at most the slots and keep the grid within
    two workgroups a unit and a tile."""
    seen = set()
    for rows in (16, 500, 2048, 7168, 24576):
        for m in (17, 65, 129, 512):
            for silu in (0, 1):
                for waves in (1, 4, 8, 16):
                    args = (rows, silu, plan.tiles(m, 1), waves, cus)
                    wr, splits = plan.wr(*args), plan.splits(*args)
                    seen.add((wr, splits > 1))
                    groups = -(-rows // (32 if silu else 64)) * (plan.tiles(m, 1) // 8)
                    assert wr in (1, 2) and 1 <= splits <= waves
                    assert splits == 1 or (wr == 1 and (splits - 1) * groups < 2 * cus)
    assert seen == {(2, False), (1, False), (1, True)}


def test_the_gpu_tests_shapes_reach_every_panel_instance(plan):
    from test_gpu_fp8_batch import LONG, LONG_LINEARS, LONG_MLPS

    seen = set()

    def add(kind, rows, silu, one_plane, waves):
        args = (rows, silu, plan.tiles(LONG, one_plane), waves, 256)
        seen.add((kind, plan.wr(*args), plan.splits(*args) > 1))

    for bf16 in (0, 1):
        for rows, cols in LONG_LINEARS:
            blocks = -(-cols // 128)
            assert LONG >= getattr(plan, "from")(rows, blocks, 1, bf16), (rows, cols)
            add(("linear", bf16), rows, 0, bf16, min(blocks, 8))
        for inter, hid in LONG_MLPS:
            assert LONG >= plan.mlp_from(hid, inter, bf16), (inter, hid)
            add(("gate_up", bf16), inter, 1, bf16, min(-(-hid // 128), 4))
            add("down", hid, 0, 0, min(-(-inter // 128), 16))
    kinds = [("linear", 0), ("linear", 1), ("gate_up", 0), ("gate_up", 1), "down"]
    assert seen == {(k, wr, split) for k in kinds for wr, split in ((2, False), (1, False), (1, True))}
