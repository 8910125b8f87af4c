"""CPU check that the down kernel stays inside its dynamic LDS: every index that
its threads form while they stage n slots' rows and their run sums
(down_lds.h, which the launch sizes the allocation by and the kernel indexes
by), for one to nine slots and every width of the one-type path (inter <= 512),
lies inside the allocation, rows and sums apart, and all of both are written."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "roaster_amd", "csrc")

PROGRAM = r"""
#include <stdio.h>
#include <vector>
#include "down_lds.h"
int main()
{
    for (int n = 1; n <= 9; n++)
        for (int I = 256; I <= 512; I += 256) {
            const DownLds S = { n, I };
            std::vector<char> lds(S.bytes() / 4, 0);
            for (int tid = 0; tid < 256; tid++)
                for (int k = 0; k < 5; k++)
                    for (int f = 0; f < 4; f++) {
                        const int at = 4 * S.unit(tid + 256 * k) + f;
                        if (at < 0 || at >= S.sums_at()) return printf("row store %d of n %d I %d\n", at, n, I), 1;
                        lds[at] = 1;
                    }
            for (int r = 0; r < S.sums(); r++) {
                if (r * 16 + 16 > S.sums_at()) return printf("run %d of n %d I %d\n", r, n, I), 1;
                if (S.sums_at() + r >= (int)lds.size()) return printf("sum %d of n %d I %d\n", r, n, I), 1;
                lds[S.sums_at() + r] = 1;
            }
            for (char c : lds)
                if (!c) return printf("n %d I %d not all written\n", n, I), 1;
        }
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_staging_stays_inside(tmp_path):
    src, exe = tmp_path / "lds.cpp", tmp_path / "lds"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-O1", "-I", CSRC, "-o", str(exe), str(src)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


def test_kernel_and_launch_use_that_layout():
    """The one-type path indexes its rows and sums by the launch's own slot count:
    nothing in it is written for nine slots whatever the call has."""
    with open(os.path.join(CSRC, "decode.hip")) as f:
        text = f.read()
    body = re.search(r"void down_one_token\(.*?\n}\n", text, re.S).group(0)
    assert "9 * I" not in body and "9 * (I" not in body and "9 * ngroups" not in body
    assert "DownLds{ nslot, A.I }.bytes()" in text
