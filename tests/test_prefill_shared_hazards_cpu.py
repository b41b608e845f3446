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
