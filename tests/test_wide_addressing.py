"""Where the one-pass kernel reads x (wide_row_chunks of lowbit_gemv_wide.h, compiled for the host): the rows of four, clamped to the
last one, at rows of any length that a weight may have - three of them are 2^32 elements and more from K = 1431655766 on."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ipex-llm_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
PROGRAM = """
#include <hip/hip_runtime.h>
#include "lowbit_gemv_wide.h"
#include <cstdio>
int main() {
    for (int K : {128, 4096, 11008, 1073741824, 1431655680, 1431655808, 2147483520})
        for (int left = 0; left < 64; left++)
            for (int xrow = 0; xrow < 4; xrow++)
                printf("%d %d %d %u\\n", K, left, xrow, lowbit::wide_row_chunks(xrow, left, K));
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_rows_of_any_length(tmp_path):
    source, program = str(tmp_path / "rows.hip"), str(tmp_path / "rows")
    with open(source, "w") as f:
        f.write(PROGRAM)
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-w", "-I", CSRC, source, "-o", program], check=True)
    lines = subprocess.run([program], capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(lines) == 7 * 64 * 4
    for line in lines:
        k, left, xrow, at = map(int, line.split())
        assert at * 8 == min(xrow, left) * k
