"""The plan of a decode attention whose workgroups wait for each other (plan_attn_share, ts_share.h): whatever the device
holds, a whole one or a part of it, all workgroups of the launch are resident at once, or nobody waits."""

import ctypes
import os
import subprocess

import pytest

from tokenselect_amd import build

SOURCE = """
#include "ts_share.h"
extern "C" void plan(int batch, int heads, int kv_heads, int max_sel, int cus, int half, int full, int* out) {
  const ts::AttnShare s = ts::plan_attn_share(batch, heads, kv_heads, max_sel, ts::AttnRoom{cus, half, full});
  out[0] = s.nsplit, out[1] = s.half, out[2] = s.parts, out[3] = s.cols, out[4] = (int)s.parts_magic, out[5] = (int)s.bytes;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    at = tmp_path_factory.mktemp("share")
    (at / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", f"-I{build.CSRC}", str(at / "plan.cpp"), "-o",
                    str(at / "plan.so")], check=True, capture_output=True)
    lib = ctypes.CDLL(os.fspath(at / "plan.so"))

    def call(batch, heads, kv_heads, max_sel, cus, half, full):
        out = (ctypes.c_int * 6)()
        lib.plan(batch, heads, kv_heads, max_sel, cus, half, full, out)
        return dict(zip(("nsplit", "half", "parts", "cols", "magic", "bytes"), out))
    return call


@pytest.mark.parametrize("cus", [256, 128, 64, 32, 0])
@pytest.mark.parametrize("per_cu", [(2, 2), (2, 1), (1, 1), (3, 4)], ids=str)
def test_all_that_wait_are_resident(plan, cus, per_cu):
    shared = 0
    for batch in (1, 2, 3, 4, 8, 31):
        for kv_heads in (1, 2, 4, 8):
            for group in range(1, 9):
                for max_sel in (1, 63, 640, 641, 2688, 2689, 4736, 5120, 8832):
                    room = [n * cus for n in per_cu]
                    s = plan(batch, group * kv_heads, kv_heads, max_sel, cus, *room)
                    grid = batch * kv_heads * s["nsplit"]
                    if not s["nsplit"]:
                        continue
                    shared += 1
                    assert grid <= (min(cus, room[0]) if s["half"] else min(2 * cus, room[1])), (batch, group, kv_heads, max_sel)
                    # and they cover the list, each word has one reader, and every column of a head one workgroup
                    if s["half"]:
                        assert s["nsplit"] * 64 >= max_sel
                    assert 10 <= s["nsplit"] <= 80 and s["nsplit"] >= group * s["parts"]
                    assert s["parts"] * s["cols"] >= 64
                    for x in range(256):
                        assert x * s["magic"] >> 16 == x // s["parts"]
                    assert s["bytes"] == grid * group * (64 + s["parts"]) * 8
    assert (shared > 0) == (cus > 0)


def test_the_whole_device(plan):
    """What the figures of the plan's comment were measured with; and what becomes of it on a quarter of the device."""
    whole, quarter = (256, 512, 512), (64, 128, 128)
    assert [plan(1, 28, 4, 2688, *whole)[x] for x in ("nsplit", "half")] == [42, 1]
    assert [plan(1, 32, 8, 2688, *whole)[x] for x in ("nsplit", "half")] == [21, 0]
    assert [plan(8, 28, 4, 2688, *whole)[x] for x in ("nsplit", "half")] == [14, 0]
    assert plan(8, 32, 8, 2688, *whole)["nsplit"] == 0
    assert [plan(1, 28, 4, 2688, *quarter)[x] for x in ("nsplit", "half")] == [21, 0]
    assert [plan(1, 32, 8, 2688, *quarter)[x] for x in ("nsplit", "half")] == [14, 0]
    assert plan(2, 32, 8, 2688, *quarter)["nsplit"] == 0
