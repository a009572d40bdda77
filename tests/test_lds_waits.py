"""Rows that come to LDS by copies of other waves replace what a wave has read: every read of
LDS has returned ahead of a barrier. Nothing at run time shows it (a copy takes longer than
a read), so the compiled kernels are looked at."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

HIP = Path(__file__).resolve().parents[1] / "bloombee_amd" / "ops" / "hip"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def blocks(kernel):
    """{label: (lines, labels that follow)} of a kernel's assembly; "" is its entry."""
    out, name, lines, to = {}, "", [], []
    for line in kernel:
        label = re.match(r"(\.LBB\S*):", line)
        if label:
            out[name] = lines, to + [label[1]]
            name, lines, to = label[1], [], []
            continue
        line = line.split(";")[0].strip()
        if re.match(r"s_c?branch", line):
            to.append(line.split()[-1])
            if line.startswith("s_branch"):     # what follows has a label of its own
                out[name] = lines, to
                name, lines, to = f"behind {len(out)}", [], []
            continue
        lines.append(line)
    out[name] = lines, to
    return out


def early_barriers(kernel):
    """Barriers that a read of LDS may be on its way at."""
    graph = blocks(kernel)
    pending, todo, found = {}, [("", False)], set()
    while todo:
        name, reads = todo.pop()
        if name not in graph or pending.get(name, -1) >= reads:
            continue
        pending[name] = reads
        lines, to = graph[name]
        for i, line in enumerate(lines):
            if line.startswith("ds_read"):
                reads = True
            elif re.match(r"s_waitcnt\b.*lgkmcnt\(0\)", line):
                reads = False
            elif line.startswith("s_barrier") and reads:
                found.add((name, i))
        todo += [(t, reads) for t in to]
    return found


def kernels(tmp_path, source):
    (tmp_path / "all.hip").write_text(source)
    subprocess.run(
        [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "--offload-device-only", "-S",
         "-w", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", str(HIP),
         str(tmp_path / "all.hip"), "-o", str(tmp_path / "all.s")], check=True)
    out, body = {}, None
    for line in (tmp_path / "all.s").read_text().splitlines():
        start = re.match(r"(_Z\w+):", line)
        if start:
            body = out.setdefault(start[1], [])
        elif line.startswith(".Lfunc_end"):
            body = None
        elif body is not None:
            body.append(line)
    return out


@pytest.mark.parametrize("D", [64, 128])
def test_training_attention(tmp_path, D):
    if not Path(HIPCC).exists():
        pytest.skip("no compiler for the device")
    found = kernels(tmp_path, '#include "attn_train.hip"\n' + "".join(
        f"template __global__ void attn_train_{k}kernel<{D}>(TrainAttnArgs);\n"
        for k in ("", "dq_", "dkv_")))
    found = {n: k for n, k in found.items() if "attn_train" in n}
    assert len(found) == 3
    for name, kernel in found.items():
        assert sum("s_barrier" in line for line in kernel) >= 2
        assert not early_barriers(kernel), name


def test_a_read_that_is_waited_for_behind_the_barrier():
    late = [".LBB0_1:", "s_barrier", "s_waitcnt lgkmcnt(0)", "ds_read_b128 v[0:3], v4",
            "s_waitcnt vmcnt(2)", "s_cbranch_scc1 .LBB0_1", "s_endpgm"]
    assert early_barriers(late) == {(".LBB0_1", 0)}
    late[4] = "s_waitcnt vmcnt(2) lgkmcnt(0)"
    assert not early_barriers(late)
