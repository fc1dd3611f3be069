"""Index arithmetic of the kernels (csrc/hip/ranges.hpp) compiled for the host, against
Python's integers, up to the largest counts that an int holds."""
import shutil
import subprocess
from pathlib import Path

import pytest

HIP = Path(__file__).resolve().parents[1] / "spsim_amd" / "csrc" / "hip"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")


def _run(tmp_path, body, args):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include <cstdio>\n#include <cstdlib>\n#include "ranges.hpp"\nint main(int argc, char **argv) {\n'
                   "  auto arg = [&](int i) { return atoi(argv[i]); };\n" + body + "\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=undefined",
                    "-fno-sanitize-recover=undefined", f"-I{HIP}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    return [int(x) for x in r.stdout.split()]


@pytest.mark.parametrize("count,n", [(0, 1), (1, 4), (1000, 7), (8_500_000, 512), (17_000_000, 256),
                                     (2**31 - 1, 4), (2**31 - 1, 1024)])
def test_ranges_cover_the_count(tmp_path, count, n):
    """A molecule of 17 million atoms, half of them in one cell: 8.5 million atoms
    in some 250 ranges, whose products with the range's number pass 2^31."""
    got = _run(tmp_path, "  for (int k = 0; k <= arg(2); ++k) printf(\"%d\\n\", spsim::range_begin(arg(1), k, arg(2)));",
               [count, n])
    assert got == [count * k // n for k in range(n + 1)]
    assert got[0] == 0 and got[-1] == count
