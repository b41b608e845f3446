"""The prefill attention's output products are assembly whose registers the compiler's hazard
handling does not see.  Its listing, for every head group and both logit forms, is searched for a
result that is used, or an operand that is written, too close to such a product: as the library
is built, and once more without the scheduling barriers of the source, where only the order of
the values themselves keeps the two apart."""

import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from tokenselect_amd import build

# Instructions between a 16x16x32 product and a use of its result, and between a vector
# instruction and a product that reads its result: what the compiler itself leaves (s_nop 7, and
# two) where it sees both.
RESULT, OPERAND = 8, 2


def _registers(token):
    m = re.fullmatch(r"-?\|?([av])(?:(\d+)|\[(\d+):(\d+)\])\|?", token)
    if not m:
        return set()
    lo, hi = (m[2], m[2]) if m[2] else (m[3], m[4])
    return {(m[1], i) for i in range(int(lo), int(hi) + 1)}


def _parse(listing):
    """Kernel name -> its instructions: (text, written, read, matrix, by hand, idle, predecessors)."""
    kernels, name, by_hand = {}, None, False
    for line in listing.splitlines():
        if re.match(r"_Z\w+:", line):
            name = line.split(":")[0]
            kernels[name], labels, jumps, open_labels, falls = [], {}, [], [], False
            kernels[name + " flow"] = (labels, jumps)
        if name is None:
            continue
        if "ASMSTART" in line or "ASMEND" in line:
            by_hand = "ASMSTART" in line
            continue
        m = re.match(r"(\.L\w+):", line)
        if m:
            open_labels.append(m[1])
            continue
        text = line.split(";")[0].strip()
        if line.startswith(".Lfunc_end"):
            name = None
            continue
        if not text or text[0] in "._" or text.endswith(":") or not line.startswith("\t"):
            continue
        op, _, rest = text.partition(" ")
        op = op.split("\t")[0]
        rest = text[len(op):]
        tokens = [t.split()[0] for t in re.split(r",(?![^\[]*\])", rest) if t.split()]
        stores = "store" in op or op.startswith("ds_write")
        written = set() if stores or not tokens else _registers(tokens[0])
        read = set().union(*(_registers(t) for t in (tokens if stores else tokens[1:]))) if tokens else set()
        here = kernels[name]
        for label in open_labels:
            labels[label] = len(here)
        open_labels = []
        before = [len(here) - 1] if falls else []
        if "branch" in op:
            jumps.append((len(here), tokens[-1]))
        falls = op not in ("s_branch", "s_endpgm")
        idle = int(tokens[0]) + 1 if op == "s_nop" else 1
        here.append((text, written, read, "mfma" in op, by_hand, idle, before))
    for key in [k for k in kernels if not k.endswith(" flow")]:
        labels, jumps = kernels.pop(key + " flow")
        for at, label in jumps:
            if label in labels and labels[label] < len(kernels[key]):
                kernels[key][labels[label]][6].append(at)
    return {k: v for k, v in kernels.items() if any(i[3] and i[4] for i in v)}


def _hazards(kernel):
    found = []
    for text, written, read, matrix, by_hand, _, before in kernel:
        product = matrix and by_hand
        todo, seen = [(p, 0) for p in before], {}
        while todo:
            at, between = todo.pop()
            if between >= RESULT or seen.get(at, RESULT) <= between:
                continue
            seen[at] = between
            other, other_written, _, other_matrix, other_hand, idle, other_before = kernel[at]
            if other_matrix and other_hand and other_written & (read | written) and \
                    not (product and other_written == written and not other_written & _operands(text)):
                found.append((other, text, between))
            if product and between < OPERAND and other.startswith("v_") and not other_matrix and other_written & read:
                found.append((other, text, between))
            todo += [(p, between + idle) for p in other_before]
    return found


def _operands(text):
    """The two operands of a product beside its accumulator."""
    tokens = [t.strip() for t in re.split(r",(?![^\[]*\])", text.split(None, 1)[1])]
    return _registers(tokens[1]) | _registers(tokens[2])


def test_the_search_finds_planted_hazards():
    product = "\t;ASMSTART\n\tv_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]\n\t;ASMEND\n"

    def count(before, after, loop=False):
        text = "_Zk:\n" + (".LBB0_1:\n" if loop else "") + before + product + after
        return len(_hazards(_parse(text + ("\ts_cbranch_scc1 .LBB0_1\n" if loop else "") +
                                   "\ts_endpgm\n.Lfunc_end0:\n")["_Zk"]))

    assert count("", product) == 0
    assert count("", "\ts_nop 7\n\tv_accvgpr_read_b32 v9, a3\n") == 0
    assert count("", "\ts_nop 6\n\tv_accvgpr_read_b32 v9, a3\n") == 1
    assert count("", "\tv_accvgpr_write_b32 a1, v9\n") == 1
    assert count("", "\tds_write_b128 v20, a[0:3]\n") == 1
    assert count("\tv_mov_b32_e32 v5, v9\n\ts_nop 0\n", "") == 1
    assert count("\tv_mov_b32_e32 v5, v9\n\ts_nop 1\n", "") == 0
    assert count("\tv_mov_b32_e32 v9, v5\n", "\ts_nop 7\n", loop=True) == 0
    assert count("\tv_accvgpr_read_b32 v9, a3\n", "\ts_nop 5\n", loop=True) == 1   # (round the loop)
    assert count("\tv_accvgpr_read_b32 v9, a3\n", "\ts_nop 6\n", loop=True) == 0


def test_output_products_keep_their_distance(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    source = open(os.path.join(build.CSRC, "ts_prefill.hip")).read()
    free = re.sub(r"__builtin_amdgcn_sched_(group_)?barrier\([^;]*;", ";", source)
    assert "sched_barrier" in source and "sched_barrier" not in free

    def listing(kind, text):
        src, out = tmp_path / f"{kind}.hip", tmp_path / f"{kind}.s"
        src.write_text(text.replace('#include "', f'#include "{build.CSRC}/'))
        subprocess.run([build.HIPCC, *build.CXXFLAGS, *build.SOURCE_FLAGS["ts_prefill.hip"], "-S",
                        "--offload-device-only", str(src), "-o", str(out)], check=True, capture_output=True)
        return _parse(out.read_text())

    with ThreadPoolExecutor(2) as pool:
        listings = pool.map(lambda kind: (kind, listing(*kind)), [("as built", source), ("free", free)])
    for (kind, _), kernels in listings:
        assert len(kernels) == 16, kind                        # 1 to 8 heads per KV head, with and without a cap
        for name, kernel in kernels.items():
            assert sum(i[3] and i[4] for i in kernel) >= 64, name
            assert _hazards(kernel) == [], (kind, name)
