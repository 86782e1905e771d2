"""Rows per block of mid-sized batches (batch_spread_rows), on the host."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "lattice_boltzmann_parallel_solver_amd", "csrc")

DRIVER = r"""
#include <cstdio>

#include "lbm_batch_tables.h"

int main() {
    int rows, threads, k, f64, cus;
    long long total;
    while (std::scanf("%d %d %d %d %lld %d", &rows, &threads, &k, &f64, &total, &cus) == 6)
        std::printf("%d\n", lbm::batch_spread_rows(rows, threads, k, f64 != 0, total, cus));
    return 0;
}
"""


def test_spread_rows(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ missing")
    src = tmp_path / "spread.cpp"
    src.write_text(DRIVER)
    exe = str(tmp_path / "spread")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, "-o", exe, str(src),
                    os.path.join(CSRC, "lbm_batch_tables.cpp")], check=True)
    cases = [  # rows asked, threads, k, FP64, rows in the batch, CUs -> rows
        (8, 256, 2, 0, 180000, 256, 8), (32, 512, 3, 0, 180000, 256, 32), (32, 576, 2, 0, 180000, 256, 32),
        (8, 256, 2, 0, 15473, 256, 3), (30, 512, 3, 0, 15473, 256, 10), (30, 576, 2, 0, 15473, 256, 7),
        (8, 256, 2, 1, 15473, 256, 8), (8, 256, 2, 1, 12000, 256, 5), (32, 576, 2, 1, 30142, 256, 32), (30, 576, 2, 1, 15473, 256, 15), (2, 256, 2, 0, 2462, 256, 2),
        (1, 256, 2, 0, 300, 256, 1), (5, 256, 2, 0, 5819, 256, 2), (8, 64, 2, 0, 0, 0, 2),
    ]
    text = "".join(" ".join(str(v) for v in c[:-1]) + "\n" for c in cases)
    out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split()
    assert [int(v) for v in out] == [c[-1] for c in cases]
