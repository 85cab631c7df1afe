"""Addresses of a closure brick's halo (csrc/spk_halo.hpp, compiled here for the
host) against the wrapped point index in 64 bits, for bricks at every face, edge
and corner and inside, up to the largest grid spk_closure_create accepts: there a
field holds 2^32 chunks of 16 bytes."""
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
#include <cstdlib>
#include "spk_halo.hpp"
using namespace spk;
int main(int, char **argv) {
    const int n = atoi(argv[1]), nq = atoi(argv[2]);
    const long long P = (long long)n * n * n * nq;
    const int xs[] = {0, 4, n / 8 * 4, n - 8, n - 4}, zs[] = {0, n / 64 * 32, n - 32};
    long long bad = 0;
    for (int x0 : xs)
        for (int y0 : xs)
            for (int z0 : zs)
                for (int c = 0; c < HX * HY * HZ * nq; c++) {
                    const int at[1] = {halo_place(c, n, nq)};
                    unsigned o[1];
                    halo_chunks(at, o, n, nq, x0, y0, z0);
                    const int hp = c / nq;
                    const long long gx = (x0 + hp / (HZ * HY) - 1 + n) % n, gy = (y0 + hp / HZ % HY - 1 + n) % n,
                                    gz = (z0 + hp % HZ - 1 + n) % n;
                    const long long want = ((gx * n + gy) * n + gz) * nq + c % nq;
                    const long long got = o[0];
                    if (got != want || got < 0 || got >= P) bad++;
                }
    printf("%lld\n", bad);
    return 0;
}
"""


@pytest.mark.parametrize("n", [32, 64, 128, 800, 832, 896, 1024])
@pytest.mark.parametrize("nq", [2, 4])
def test_halo_chunks(tmp_path, n, nq):
    src, exe = tmp_path / "halo.cpp", tmp_path / "halo"
    src.write_text(MAIN)
    subprocess.run([CXX, "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe), str(n), str(nq)], capture_output=True, text=True, check=True)
    assert int(r.stdout) == 0
