"""The work queues of the streaming kernels, walked on the CPU: the header that the kernels and their launches are built
from is compiled for the host with a program that enumerates every queue."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tilesparsity_amd", "csrc")

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <vector>
namespace tw { constexpr int kXcd = 8, kBalColumns = 4; }
#include "tw_queue.h"
using namespace tw;
struct Args {
    int32_t n_mblk, n_pipe_u, n_all_u, n_own, n_last, last_x, last_r, n_lead_items, n_col_mblk, n_col_items, n_rest_items, rb_major;
    int32_t n_bal, bal_first[kBalColumns + 1], bal_rows[kBalColumns];
};
static int walk(const Args &a, bool owned, bool by_rows)
{
    std::vector<int> seen((size_t)a.n_all_u * a.n_mblk, 0);
    std::vector<int> owner(a.n_mblk, -1);
    for (int x = 0; x < kXcd; ++x) {
        const int len = queue_length(a, x);
        int last = -1;
        for (int q = 0; q < len; ++q) {
            const Work w = queue_entry(a, x, q, len, 256);
            if (w.col < 0 || w.col >= a.n_all_u || w.m0 < 0 || w.m0 % 256 || w.m0 / 256 >= a.n_mblk || w.rows != 256)
                return 1;
            const int m = w.m0 / 256;
            ++seen[(size_t)w.col * a.n_mblk + m];
            if (q % (2 * a.n_pipe_u + !a.n_pipe_u) == 0 && q <= a.n_lead_items) // (a group of two row blocks, and what comes behind them)
                last = -1;
            if (!by_rows && w.col < last) // heaviest columns first
                return 2;
            last = w.col;
            if (w.col < a.n_pipe_u && owned) {
                if (owner[m] == -1)
                    owner[m] = x;
                else if (owner[m] != x)
                    owner[m] = -2;
            }
        }
        for (int q = len; q < len + 5; ++q)
            if (queue_entry(a, x, q, len, 256).col != a.n_all_u)
                return 3;
    }
    for (int n : seen)
        if (n != 1)
            return 4;
    int shared = 0;
    for (int o : owner)
        shared += o == -2;
    return owned && shared > a.n_mblk % kXcd ? 5 : 0; // (all others have one die)
}
int main()
{
    long n = 0;
    for (int mblk = 1; mblk < 70; ++mblk)
        for (int pipe : {0, 1, 2, 3, 5, 8, 13, 40})
            for (int other : {0, 1, 3, 9})
                for (int order = 0; order < 3; ++order)
                    for (long wgs : {1l, 8l, 32l, 256l, 100000l}) {
                        Args a{};
                        a.n_mblk = mblk;
                        a.n_pipe_u = pipe;
                        a.n_all_u = pipe + other;
                        if (!a.n_all_u)
                            continue;
                        lay_queues(a, order == 1, wgs);
                        if (order == 2)
                            order_by_row_blocks(a);
                        const int bad = walk(a, order == 1, order == 2);
                        if (bad) {
                            std::printf("%d: %d row blocks, %d + %d columns, order %d, %ld workgroups\n", bad, mblk, pipe, other, order, wgs);
                            return 1;
                        }
                        ++n;
                    }
    // the largest launch: the last entry of every queue, and what a workgroup draws behind it
    Args a{};
    a.n_mblk = 0x7fffffff / 31;
    a.n_pipe_u = 30;
    a.n_all_u = 31;
    for (int owned = 0; owned < 2; ++owned) {
        lay_queues(a, owned, 256);
        for (int x = 0; x < kXcd; ++x) {
            const int len = queue_length(a, x);
            const Work w = queue_entry(a, x, len - 1, len, 1);
            if (w.col != 30 || w.m0 < a.n_mblk - 2 * kXcd || w.m0 >= a.n_mblk || queue_entry(a, x, len + 4096, len, 1).col != 31) {
                std::printf("largest %d %d: %d %d\n", owned, x, w.col, w.m0);
                return 1;
            }
        }
    }
    std::printf("ok %ld\n", n);
    return 0;
}
"""


def test_every_item_is_in_one_queue_once(tmp_path):
    """Every item in exactly one queue, nothing behind a queue's end, the columns in their order, and no more row blocks
    that several dies work on than those nobody owns."""
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "queues.cpp", tmp_path / "queues"
    src.write_text(PROGRAM)
    subprocess.run([compiler, "-std=c++17", "-O1", "-Wno-unknown-pragmas", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert res.returncode == 0 and res.stdout.startswith("ok"), res.stdout
