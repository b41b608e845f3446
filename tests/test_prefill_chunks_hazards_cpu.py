"""As test_prefill_hazards_cpu, for the same attention over several chunks (ts_prefill_chunks.hip)."""

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
    text = open(os.path.join(build.CSRC, "ts_prefill_chunks.hip")).read()
    assert text.count('#include "ts_prefill.hip"') == 1
    text = text.replace('#include "ts_prefill.hip"', open(os.path.join(build.CSRC, "ts_prefill.hip")).read())
    if kind == "free":
        text = re.sub(r"__builtin_amdgcn_sched_(group_)?barrier\([^;]*;", ";", text)
        assert "sched_barrier" not in text
    src, out = tmp_path / "chunks.hip", tmp_path / "chunks.s"
    src.write_text(text.replace('#include "', f'#include "{build.CSRC}/'))
    subprocess.run([build.HIPCC, *build.CXXFLAGS, *build.SOURCE_FLAGS["ts_prefill_chunks.hip"], "-S",
                    "--offload-device-only", str(src), "-o", str(out)], check=True, capture_output=True)
    kernels = _parse(out.read_text())
    assert len(kernels) == 16                                  # 1 to 8 heads per KV head, with and without a cap
    for name, kernel in kernels.items():
        assert sum(i[3] and i[4] for i in kernel) >= 64, name
        assert _hazards(kernel) == [], name
