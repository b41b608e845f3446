"""What the built kernels take of a CU, from the notes the compiler leaves in the library."""

import os
import re
import struct
import subprocess

import pytest

from tokenselect_amd import _lib, build

LLVM = os.path.join(build.ROCM, "llvm", "bin")
LDS = 160 * 1024  # of a CU


def _kernels(tmp_path):
    """Name -> bytes of LDS that the kernel has before any it is launched with."""
    fat = tmp_path / "fat"
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={fat}", _lib.LIB_PATH, str(tmp_path / "rest")],
                   check=True, capture_output=True)
    data, found = fat.read_bytes(), {}
    for bundle in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = bundle.start() + 32
        for _ in range(struct.unpack_from("<Q", data, bundle.start() + 24)[0]):
            offset, size, name = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + name]
            at += 24 + name
            if build.ARCH.encode() not in target:
                continue
            (tmp_path / "code").write_bytes(data[bundle.start() + offset:bundle.start() + offset + size])
            notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(tmp_path / "code")], check=True, capture_output=True,
                                   text=True).stdout
            for kernel in re.split(r"\n  - ", notes)[1:]:
                symbol, lds = (re.search(rf"\.{key}:\s+(\S+)", kernel) for key in ("name", "group_segment_fixed_size"))
                if symbol and lds:
                    found[symbol[1]] = int(lds[1])
    return found


def test_a_fused_selection_fits_beside_its_largest_stage(tmp_path):
    """Whichever head shape and form: what does not fit has no fused selection at all, and only the capacity query says so."""
    if not (os.path.exists(f"{LLVM}/llvm-objcopy") and os.path.exists(f"{LLVM}/llvm-readelf")):
        pytest.skip("no llvm tools")
    if not os.path.exists(_lib.LIB_PATH):
        build.build(verbose=False)
    source = open(os.path.join(build.CSRC, "ts_score.hip")).read()
    stage = int(re.search(r"kFusedLargeStageBytes = (\d+) \* 1024", source)[1]) * 1024
    # score_kernel<KV heads, group, false, 2 to 4>
    fused = {name: lds for name, lds in _kernels(tmp_path).items() if re.search(r"score_kernelILi\dELi\dELb0ELi[234]E", name)}
    assert len(fused) == 4 * 8 * 3
    for name, lds in fused.items():
        assert lds + stage <= LDS, (name, lds)
