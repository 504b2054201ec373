"""Which kernel the multi-step LSTM launches of test_gpu_cell.py take: the header with the rule, compiled for the host."""
import os
import shutil
import subprocess

import pytest

from tests import test_gpu_cell

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tilesparsity_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "tw_lstm_form.h"
int main(int argc, char **argv)
{
    for (int i = 1; i + 4 < argc; i += 5)
        std::printf("%d\n", (int)tw::lstm_rows_in_lds(std::atoi(argv[i]), std::atoi(argv[i + 1]), std::atoi(argv[i + 2]), std::atoi(argv[i + 3]),
                                                   std::atoi(argv[i + 4])));
}
"""


def parameters(test):
    for mark in test.pytestmark:
        if mark.name == "parametrize" and "," in mark.args[0]:
            names = mark.args[0].split(",")
            return [dict(zip(names, values)) for values in mark.args[1]]


def test_both_kernels_are_tested(tmp_path):
    """The launches that say that they keep the rows of A in LDS do (with the 150 kept rows a tile that each asserts), the others do not."""
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "form.cpp", tmp_path / "form"
    src.write_text(PROGRAM)
    subprocess.run([compiler, "-std=c++17", "-O1", "-I", CSRC, "-o", str(exe), str(src)], check=True)

    def in_lds(cases):
        args = [str(v) for I, H, M, T, kept in cases for v in (I + H, H, M, T, kept)]
        return subprocess.run([str(exe)] + args, stdout=subprocess.PIPE, text=True, check=True).stdout.split()
    with_rows = [(p["I"], p["H"], p["M"], p["T"], 150) for p in parameters(test_gpu_cell.test_multi_step_launch_with_its_rows_in_lds)]
    with_rows += [(256, 1024, 40, 24, 150), (256, 1024, 72, 24, 150)]  # (non-finite values; in a graph)
    assert len(with_rows) == 7 and in_lds(with_rows) == ["1"] * 7
    others = [(48, p["H"], p["M"], 4, 512) for p in parameters(test_gpu_cell.test_multi_step_launch_places)]
    others += [(128, 256, 96, 5, 512), (192, 512, 120, 6, 512)]        # (in a graph; without the first look)
    assert in_lds(others) == ["0"] * len(others)
    # one below each line
    assert in_lds([(256, 1024, 40, 23, 150), (256, 1024, 40, 24, 149), (256, 1024, 1, 24, 150), (1025, 1024, 40, 24, 150), (0, 1024, 40, 24, 150),
                   (256, 1056, 40, 24, 150), (256, 992, 40, 31, 150), (256, 992, 32, 32, 150), (1000, 512, 33, 32, 295), (256, 480, 40, 32, 480)]) == ["0"] * 10
    assert in_lds([(1024, 1024, 2, 24, 150), (256, 992, 33, 32, 150), (1000, 512, 33, 32, 296)]) == ["1"] * 3
