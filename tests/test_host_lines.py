"""Line kernels of the assembly (ifem_amd/csrc/lines.hpp) compiled for the
host, one thread per lane of a workgroup, in every configuration that the
library launches: degrees and rules, scalar and vector, FP64 with and without
right-hand side and FP32, own rows, rows shared with other patches (with and
without position maps), prescribed values, and work lists of a batch.

The address sanitizer bounds every access to the records, tables, equation
numbers and the matrix; the thread sanitizer sees two lanes that touch one LDS
value without a barrier between them.  K and b equal direct quadrature over the
elements: sums of some thousand products, 1e-12 of the largest entry (FP32 1e-5).
"""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "ifem_amd", "csrc")
CLANG = "/opt/rocm/llvm/bin/clang++"
CONFIGS = [(1, 2, 1), (1, 2, 3), (1, 3, 1), (1, 3, 3), (2, 3, 1), (2, 3, 3)]
SANITIZERS = {"address": ["-fsanitize=address,bounds"], "thread": ["-fsanitize=thread"]}
# the barriers are the same in every configuration
PROGRAMS = [("address", c) for c in CONFIGS] + [("thread", c) for c in CONFIGS[:2]]

# fp32, rhs, accum, elements, row segments, fixed functions, prescribed values
CASES = [
    (0, 1, 0, (3, 13, 1), 1, 2, 0),   # several line groups, the last one short
    (0, 1, 0, (5, 3, 1), 3, 3, 1),    # segments that start inside an element's rows
    (0, 0, 0, (1, 1, 1), 1, 0, 0),
    (0, 1, 0, (3, 2, 1), 4, 2, 0),    # one row per segment
    (0, 1, 2, (3, 9, 1), 2, 3, 1),
    (0, 0, 1, (2, 2, 2), 2, 2, 1),
    (1, 0, 0, (3, 8, 2), 2, 1, 0),
    (1, 0, 2, (2, 2, 2), 1, 3, 0),
]
BATCH = [(0, 1, 3, (3, 10, 1), 2, 0, 0), (1, 0, 3, (3, 9, 1), 2, 3, 0)]


def _cases(config, sanitizer):
    out = list(CASES) + (BATCH if config in ((1, 2, 1), (2, 3, 1)) else [])
    if config[2] == 3:  # one line per group: fewer lines
        out = [(*c[:3], (c[3][0], (c[3][1] + 3) // 4, c[3][2]), *c[4:]) for c in out]
    if config == (2, 3, 3):  # FP32 of this one has a kernel of its own
        out = [c for c in out if not c[0]]
    return out[1::2] if sanitizer == "thread" else out


@pytest.fixture(scope="module")
def programs(tmp_path_factory):
    """{(sanitizer, config): executable}, compiled side by side.  The copies of
    the kernel headers lose their inline assembly: a wait for LDS, which the
    host's barrier includes."""
    if not os.path.exists(CLANG):
        pytest.skip("no host clang with sanitizers")
    d = tmp_path_factory.mktemp("host_lines")
    shutil.copytree(os.path.join(HERE, "host_lines"), d, dirs_exist_ok=True)
    shutil.copy(os.path.join(CSRC, "asmargs.hpp"), d)
    with open(os.path.join(CSRC, "lines.hpp")) as f:
        text = f.read()
    assert "asm volatile" in text
    (d / "lines.hpp").write_text(re.sub(r"asm volatile\([^;]*\);", "", text))

    def build(key):
        san, config = key
        exe = str(d / ("%s_%d%d%d" % (san, *config)))
        r = subprocess.run([CLANG, "-std=c++20", "-O1", "-w",
                            *SANITIZERS[san], "-DCONFIG=CASE(%d, %d, %d)" % config, f"-I{d}",
                            str(d / "main.cpp"), "-o", exe, "-lpthread"],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-3000:]
        return key, exe
    with ThreadPoolExecutor(8) as ex:
        return dict(ex.map(build, PROGRAMS))


def _run(exe, args):
    r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=120)
    return r.returncode, r.stdout + r.stderr[-2000:]


@pytest.mark.parametrize("sanitizer,config", PROGRAMS,
                         ids=lambda v: v if isinstance(v, str) else "p%d_ng%d_nc%d" % v)
def test_line_kernels_on_the_host(programs, sanitizer, config):
    cases = [(*config, *c[:3], *c[3], *c[4:]) for c in _cases(config, sanitizer)]
    with ThreadPoolExecutor(4) as ex:
        for args, (rc, out) in zip(cases, ex.map(
                lambda a: _run(programs[sanitizer, config], a), cases)):
            assert rc == 0 and out.strip().endswith("ok"), (args, out)


def test_records_of_a_very_long_line(programs):
    """4,000,000 x 11 x 1 elements: the records of one group of lines span
    2.5e9 values, more than a 32-bit offset holds."""
    rc, out = _run(programs["address", (1, 2, 1)], ["long"])
    assert rc == 0, out
