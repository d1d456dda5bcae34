"""The lane-read builtins return int: an unsigned lane value widened straight from one is sign-extended.

Compiles every device source that names such a builtin for syntax only, with the sign-conversion warning, and
looks at the warnings on the lines that name one."""
import concurrent.futures as cf
import pathlib
import re
import shutil
import subprocess

import pytest

REPO = pathlib.Path(__file__).resolve().parents[1]
CSRC = REPO / "luisacompute-parallelprimitive_amd" / "csrc"
READS = "__builtin_amdgcn_read"
WIDENED = re.compile(r"^(\S+?):(\d+):\d+: warning: implicit conversion changes signedness: 'int' to '(?:const )?(?:uint64_t|size_t|unsigned long)")


def widened_reads(src: pathlib.Path) -> set[str]:
    res = subprocess.run([shutil.which("hipcc") or "/opt/rocm/bin/hipcc", "-x", "hip", "-std=c++20", "--offload-arch=gfx950",
                          "--cuda-device-only", "-fsyntax-only", "-Wsign-conversion", f"-I{REPO / 'include'}", src.name],
                         cwd=CSRC, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    found = set()
    for line in res.stderr.splitlines():
        m = WIDENED.match(line)
        if m:
            text = (CSRC / m[1]).read_text().splitlines()[int(m[2]) - 1]
            if READS in text:
                found.add(f"{m[1]}:{m[2]}: {text.strip()}")
    return found


def test_no_lane_read_is_widened():
    if not (shutil.which("hipcc") or pathlib.Path("/opt/rocm/bin/hipcc").exists()):
        pytest.skip("needs hipcc")
    sources = [p for p in sorted(CSRC.glob("*.hip")) if READS in p.read_text()
               or any(READS in (CSRC / h).read_text() for h in re.findall(r'#include "(\w+\.hpp)"', p.read_text()))]
    with cf.ThreadPoolExecutor(4) as pool:
        found = set().union(*pool.map(widened_reads, sources))
    assert not found, "\n".join(sorted(found))
