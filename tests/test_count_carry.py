"""The 32-bit counts of the q_inv histograms in LDS (count_carry in
csrc/hbt_device.h): past 2^32 in one bin of one block they carry into the 64-bit
histograms, to which the block adds what is left at its end.  Run on the host with
plain adds, from counts near the wrap; a count that drops the carry (the planted
mistake) must come out short."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "hadronic_afterburner_toolkit_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include <cstdio>
#include "hbt_device.h"
using namespace hbt;
int main(int argc, char **) {
    const bool plant = argc > 1;
    int bad = 0;
    for (unsigned before : {0u, 1u, 0x7fffffffu, 0xfffffff0u, 0xfffffffeu, 0xffffffffu})
        for (int n : {0, 1, 2, 17, 1000}) {
            unsigned lo = before;
            unsigned long long total = 5;
            for (int k = 0; k < n; k++)
                count_carry(&lo, &total, [](unsigned *p) { return (*p)++; },
                            [&](unsigned long long *p, unsigned long long v) { *p += plant ? 0 : v; });
            total += lo;
            bad += total != 5ull + before + (unsigned long long)n;
        }
    std::printf("bad %d\n", bad);
    return 0;
}
"""


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")
def test_counts_carry(tmp_path):
    src = tmp_path / "cc.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "cc"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-x", "hip", "--cuda-host-only", f"-I{CSRC}",
                    str(src), "-o", str(exe)], check=True, timeout=300, capture_output=True)

    def bad(*args):
        r = subprocess.run([str(exe), *args], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout + r.stderr
        return int(r.stdout.split()[1])

    assert bad() == 0
    assert bad("plant") > 0
