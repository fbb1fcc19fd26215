"""The order of the LDS DMA copies ahead of a counted wait, read from the compiled device IR (CPU).

The three-buffer kernels (k_mx_gemm with three buffers, k_mx_head_ring) send
the copies of steps 0 and 1 before their loop, and step 0 then waits until no
more than one step's copies are outstanding.  Memory counters complete in issue
order, so that wait covers step 0's copies only if all of them are issued before
any of step 1's; the two steps fill different LDS arrays, so nothing but a
scheduling fence keeps the compiler from mixing them.  It needs hipcc, not a GPU.
"""

from __future__ import annotations

import re
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT / "maple-flash-dgx-spark_amd"))
import build as libbuild  # noqa: E402


def prologues(ir: str, pattern: str) -> dict[str, str]:
    """Per kernel: its LDS copies (L) and scheduling fences (F) before the first wait, in order."""
    res: dict[str, str] = {}
    name, open_ = None, False
    for line in ir.splitlines():
        m = re.match(r"define .*@(\S+?)\(", line)
        if m:
            name, open_ = m.group(1), True
            if re.search(pattern, name):
                res[name] = ""
            continue
        if name not in res or not open_ or " call " not in line:
            continue
        if re.search(r"load\.(async\.)?(to\.)?lds", line):
            res[name] += "L"
        elif "sched.barrier" in line:
            res[name] += "F"
        elif "s.waitcnt" in line:
            open_ = False
    return res


@pytest.mark.skipif(not (Path(libbuild.HIPCC).exists() or shutil.which("hipcc")), reason="hipcc not found")
@pytest.mark.parametrize("src,pattern,kernels", [("mx_gemm.hip", r"k_mx_gemmILi\dELi\d+ELi3E", 4),
                                                 ("mx_head.hip", r"k_mx_head_ring", 2)])
def test_two_steps_copies_are_fenced(src, pattern, kernels, tmp_path):
    out = tmp_path / (src + ".ll")
    flags = [f for f in libbuild.FLAGS if f != "-fPIC"]
    cmd = [libbuild.HIPCC, *flags, "--cuda-device-only", "-S", "-emit-llvm", str(libbuild.CSRC / src), "-o", str(out)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    found = prologues(out.read_text(), pattern)
    assert len(found) == kernels, sorted(found)
    for name, seq in found.items():
        n = seq.count("L") // 2
        assert n > 0 and re.fullmatch(f"F+L{{{n}}}F+L{{{n}}}F+", seq), f"{name}: {seq}"
