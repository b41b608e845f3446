"""As test_prefill_hazards_cpu, for the attention in workgroups of 256 columns (ts_prefill_shared.hip)."""

import os
import re
import subprocess

import pytest

from test_prefill_hazards_cpu import _hazards, _parse
from tokenselect_amd import build


@pytest.mark.parametrize("kind", ["as built", "free"])
def test_output_products_keep_their_distance(tmp_path, kind):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    text = open(os.path.join(build.CSRC, "ts_prefill_shared.hip")).read()
    if kind == "free":
        text = re.sub(r"__builtin_amdgcn_sched_(group_)?barrier\([^;]*;", ";", text)
        assert "sched_barrier" not in text
    src, out = tmp_path / "shared.hip", tmp_path / "shared.s"
    src.write_text(text.replace('#include "', f'#include "{build.CSRC}/'))
    subprocess.run([build.HIPCC, *build.CXXFLAGS, *build.SOURCE_FLAGS["ts_prefill_shared.hip"], "-S",
                    "--offload-device-only", str(src), "-o", str(out)], check=True, capture_output=True)
    kernels = _parse(out.read_text())
    assert len(kernels) == 2                                   # with and without a cap
    for name, kernel in kernels.items():
        assert sum(i[3] and i[4] for i in kernel) >= 4 * 32, name
        assert _hazards(kernel) == [], name


def test_what_is_asked_for_ahead_is_bounded_by_the_lanes_offset(tmp_path):
    """Tiles past the end of the staging area are asked for ahead: it is the buffer's size that keeps those loads off the
    memory behind it, and a buffer's size bounds the lanes' offset and the instruction's, not the scalar one."""
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path / "shared.s"
    subprocess.run([build.HIPCC, *build.CXXFLAGS, *build.SOURCE_FLAGS["ts_prefill_shared.hip"], "-S", "--offload-device-only",
                    os.path.join(build.CSRC, "ts_prefill_shared.hip"), "-o", str(out)], check=True, capture_output=True)
    loads = [line.split() for line in out.read_text().splitlines() if re.match(r"\s*buffer_load\w* .*\blds\b", line)]
    assert len(loads) >= 2 * 2 * 7                             # kernels, halves, and three and four packages' halves
    for load in loads:
        assert "offen" in load and load[3] == "0", " ".join(load)
