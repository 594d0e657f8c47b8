"""How a training batch is split for its weight gradients (threepoint_amd/csrc/tp_mlp_split.h): the workspace holds
tp_wgrad_max_splits(capacity) blocks per layer, and a batch of any size up to the capacity must fit into it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "tp_mlp_split.h"
#include <cstdio>
int main()
{
    int most = 0;  // splits of the batches up to M
    for (int M = 64; M <= 1 << 22; M += 64) {
        const TpWgradSplit s = tp_wgrad_split(M);
        most = s.n > most ? s.n : most;
        // the kernel's stages: whole multiples of 32 rows, which cover the batch, none of them empty
        const bool covers = s.rows > 0 && s.rows % 32 == 0 && (long long)s.rows * s.n >= M && (long long)s.rows * (s.n - 1) < M;
        if (!covers || most > tp_wgrad_max_splits(M)) {
            std::printf("M %d: %d splits of %d rows; batches up to here take %d, the workspace holds %d\n", M, s.n, s.rows,
                        most, tp_wgrad_max_splits(M));
            return 1;
        }
    }
    return 0;
}
"""


def test_splits_of_every_batch_fit_the_workspace(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    (tmp_path / "t.cpp").write_text(SRC)
    subprocess.run([cxx, "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "threepoint_amd", "csrc"),
                    str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
