"""weightsFitRegisters (cusync_amd/csrc/gemm_resident.h), host code only: which output projections hold their weights in registers."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# rows, hidden, heads of 128, taken
CASES = [
    # what it is for, and what the registers and the CUs hold
    (1, 12288, 12, 1), (16, 12288, 12, 1), (64, 12288, 12, 1), (112, 12288, 12, 1), (113, 12288, 12, 0), (16, 12288, 13, 0), (16, 8064, 12, 0),
    (16, 16384, 12, 1), (16, 16392, 12, 0),
    # where 64x192 tiles do the projection: behind them with short K and from 65 rows on
    (112, 9216, 8, 1), (64, 9216, 7, 1), (65, 9216, 7, 0), (96, 12288, 6, 0), (64, 15360, 4, 1), (65, 15360, 4, 0), (16, 12288, 3, 1), (17, 12288, 3, 0), (1, 12288, 2, 0),
    # other widths: never behind from 33 rows on, but for the shortest K; 17 to 32 rows cost the 32-row tiles nothing
    (112, 8192, 12, 1), (112, 16384, 5, 1), (32, 16384, 5, 1), (33, 16384, 4, 1), (32, 16384, 4, 0), (32, 16384, 3, 0), (16, 16384, 3, 1), (16, 16384, 2, 0), (33, 16384, 2, 1),
    (33, 16384, 1, 0), (33, 10240, 1, 1), (32, 10240, 4, 1), (17, 10240, 2, 0), (16, 10240, 2, 1), (16, 10240, 1, 0), (16, 8192, 1, 1), (17, 8192, 1, 0),
]

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "gemm_resident.h"
int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3)
    std::printf("%d\n", (int)cusync::gemm::weightsFitRegisters((uint32_t)std::atoi(argv[i]), (uint32_t)std::atoi(argv[i + 1]), 128u * (uint32_t)std::atoi(argv[i + 2]), 256));
  return 0;
}
"""


def test_which_projections_hold_their_weights_in_registers(tmp_path):
    (tmp_path / "choice.cpp").write_text(SRC)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "cusync_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                           str(tmp_path / "choice.cpp"), "-o", str(tmp_path / "choice")])
    args = [str(v) for c in CASES for v in c[:3]]
    got = subprocess.run([str(tmp_path / "choice")] + args, capture_output=True, text=True, check=True).stdout.split()
    assert [(c[:3], int(g)) for c, g in zip(CASES, got)] == [(c[:3], c[3]) for c in CASES]
