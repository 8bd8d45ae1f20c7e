"""The outer-block kernel's scratch: what different workgroups write without an
order between them lies apart.  Workgroup 2 keeps the passes' factors, workgroups
0 and 1 publish blocks, and workgroup 0's column-wise refactorization of a
rejected block has its Gram and T there; a rejection is not ordered after
workgroup 2's stores.  Compiles the layout's constants on the CPU."""
import itertools
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rnp2_amd", "csrc")
MAIN = """
#include <cstdio>
#include "rnpx_cqr_layout.hpp"
using namespace rnpx::blk;
int main() {
  std::printf("factors %d %d\\n", kR, kRSize);
  std::printf("published %d %d\\n", kU1i, kPublishedEnd - kU1i);
  std::printf("gram %d %d\\n", kGram, 128 * 128);
  std::printf("tfactor %d %d\\n", kTFactor, 128 * 128);
  std::printf("row %d %d\\n", kRow, 2 * 128);
  std::printf("all 0 %d\\n", kScratch);
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not available")
def test_regions_are_disjoint(tmp_path):
    src, exe = tmp_path / "layout.cpp", tmp_path / "layout"
    src.write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    regions = {k: (int(o), int(o) + int(n)) for k, o, n in (line.split() for line in out.splitlines())}
    whole = regions.pop("all")
    for (a, x), (b, y) in itertools.combinations(regions.items(), 2):
        assert x[1] <= y[0] or y[1] <= x[0], (a, x, b, y)
    assert all(whole[0] <= r[0] < r[1] <= whole[1] for r in regions.values())


def test_kernel_takes_its_offsets_from_the_layout():
    s = open(os.path.join(CSRC, "rnpx_cqr.hip")).read()
    for name, field in (("kBR", "kR"), ("kBU1i", "kU1i"), ("kBD2", "kD2"), ("kBG", "kGram"), ("kBTF", "kTFactor"), ("kBRow", "kRow")):
        assert f"{name} = blk::{field}" in s
