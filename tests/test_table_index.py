"""The row a pair kernel reads from a table stays inside it for every grid
index: whatever the conversion of a distance that is no number gives, too.
The device header's own function, compiled for the host."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROGRAM = r"""
#include <cstdio>
#include "qmc_dev.h"
int main() {
  const int idx[] = {INT_MIN, INT_MIN + 1, -1000000, -2, -1, 0, 1, 99, 100, 101, 102, 1000000, INT_MAX - 1, INT_MAX};
  const int ngs[] = {0, 1, 100, 101, 200};
  for (int ng : ngs)
    for (int i : idx) printf("%d %d %u\n", ng, i, tab_index(i, ng));
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_every_index_reads_a_row_of_the_table(tmp_path):
    src, exe = tmp_path / "t.hip", tmp_path / "t"
    src.write_text("#include <climits>\n" + PROGRAM)
    subprocess.run([HIPCC, "-std=c++17", "--offload-host-only", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "2degas_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, stdout=subprocess.PIPE).stdout.decode().split()
    rows = [tuple(int(v) for v in out[k:k + 3]) for k in range(0, len(out), 3)]
    assert len(rows) == 5 * 14
    for ng, i, row in rows:
        assert 0 <= row <= ng
        if 0 <= i <= ng:
            assert row == i
