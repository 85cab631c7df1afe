"""Layout of the masked products (csrc/spk_prodlay.hpp, compiled here for the host): a
column with products is read at its own place, a column without any at a stored place
of a kept column, on every grid of powers of two."""
import os
import shutil
import subprocess

import pytest

from spkmod import REPO

CSRC = os.path.join(REPO, "spooky-git_amd", "csrc")
CXX = os.environ.get("CXX", "g++")

pytestmark = pytest.mark.skipif(shutil.which(CXX) is None, reason="no host compiler")

MAIN = r"""
#include <cstdio>
#include "spk_prodlay.hpp"
using namespace spk;
int main() {
    long long bad = 0;
    for (int ny = 2; ny <= 2048; ny *= 2)
        for (int nz = 2; nz <= 1024; nz *= 2)
            for (int pad = 0; pad < 2; pad++) {
                const int nzh = nz / 2 + 1;
                ProdLay l;  // |k| <= 2/3 (n / 2 - 1) is kept
                l.kc = 2 * (nz / 2 - 1) / 3 + 1;
                l.jc = 2 * (ny / 2 - 1) / 3;
                l.nskip = ny - (2 * l.jc + 1);
                l.kp = l.kc + pad;
                l.xs = (long long)ny * l.kp;
                int rows = 0;
                for (int j = 0; j < ny; j++) {
                    const int r = prod_row(l, j);
                    if (r >= 0 && r != rows++) bad++;
                    for (int k = 0; k < nzh; k++) {
                        const int p = prod_column(l, nzh, j, k);
                        if (p < 0 || p / l.kp >= 2 * l.jc + 1 || p % l.kp >= l.kc) bad++;
                        if (r >= 0 && k < l.kc && p != r * l.kp + k) bad++;
                    }
                }
                if (rows != 2 * l.jc + 1) bad++;
            }
    const ProdLay full = {3, 3, 8, 0, 24};  // no mask
    for (int j = 0; j < 8; j++)
        for (int k = 0; k < 3; k++)
            if (prod_column(full, 3, j, k) != 3 * j + k) bad++;
    printf("%lld\n", bad);
    return 0;
}
"""


def test_places_of_columns(tmp_path):
    src, exe = tmp_path / "lay.cpp", tmp_path / "lay"
    src.write_text(MAIN)
    subprocess.run([CXX, "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, check=True)
    assert int(r.stdout) == 0
