"""The workgroups of the kernel for few rows, walked on the CPU: the header that the kernel and its launch are built from is
compiled for the host with a program that enumerates what they take."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tilesparsity_amd", "csrc")
HEAD = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>
namespace tw { constexpr int kXcd = 8; constexpr int64_t kMaxGridThreads = 0xFFFFFFFFll; }
#include "tw_few_rows.h"
using namespace tw;
"""

FILLS = HEAD + r"""
int main()
{
    // every item of a fill once, the launch as large as it likes and cut to a few workgroups
    for (int n_tiles : {0, 1, 2, 7, 40})
        for (int M : {1, 32, 33, 64, 65, 1000})
            for (int rm = 0; rm < 2; ++rm)
                for (int most : {0, 1, 3, 16, 17}) {
                    SkinnyWork w{};
                    skinny_fill(&w, n_tiles, M, rm, 512);
                    if (most && w.fill_wgs > most)
                        w.fill_wgs = most;
                    std::vector<int> seen((size_t)n_tiles * w.n_fillblk, 0);
                    for (int wg = 0; wg < w.fill_wgs; ++wg)
                        for (FillPlace at = fill_first(w, wg); at.z < n_tiles; at = fill_next(w, at))
                            ++seen.at((size_t)at.z * w.n_fillblk + at.blk);
                    for (int n : seen)
                        if (n != 1)
                            return std::printf("%d tiles, M %d, row-major %d, %d workgroups: %d\n", n_tiles, M, rm, w.fill_wgs, n);
                }
    // more than 2^31 items, and a product that leaves the fill seven workgroups: the places of some workgroups against their numbers
    for (int rm = 0; rm < 2; ++rm)
        for (int n_tiles : {16384, 65536, 1 << 20})
            for (int M : {1 << 20, (8 << 20) + 1, 0x7fffffff})
                for (int gemm : {0, 8, 8388600}) {
                    SkinnyWork w{};
                    w.gemm_wgs = gemm;
                    skinny_fill(&w, n_tiles, M, rm, 512);
                    const int64_t items = (int64_t)n_tiles * w.n_fillblk;
                    if (w.fill_wgs < 1 || ((int64_t)gemm + w.fill_wgs) * 512 > kMaxGridThreads)
                        return std::printf("%d workgroups left\n", w.fill_wgs);
                    for (int wg : {0, w.fill_wgs / 2, w.fill_wgs - 1}) {
                        int64_t i = wg;
                        FillPlace at = fill_first(w, wg);
                        for (int n = 0; n < 100000 && i < items; ++n, i += w.fill_wgs, at = fill_next(w, at))
                            if (at.z != i / w.n_fillblk || at.blk != i % w.n_fillblk || at.z >= n_tiles)
                                return std::printf("item %lld of %lld: %d %d\n", (long long)i, (long long)items, at.z, at.blk);
                        if (i >= items && at.z < n_tiles)
                            return std::printf("%lld items, and one more: %d %d\n", (long long)items, at.z, at.blk);
                    }
                }
    // the workgroups that multiply never take all of a launch
    for (int units = 1; units < 100; ++units)
        for (int M = 1; M > 0 && M < 0x7fffffff - (M >> 3) - 1000; M += (M >> 3) + 997) {
            SkinnyWork w{};
            const int64_t wgs = skinny_work(units, 128, M, &w);
            if (wgs >= 0 && (wgs % 8 || wgs * 512 > kMaxGridThreads || kMaxGridThreads / 512 - wgs < 1))
                return std::printf("%d units, M %d: %lld\n", units, M, (long long)wgs);
        }
    std::printf("ok\n");
    return 0;
}
"""

FORM = HEAD + r"""
int main(int argc, char **argv) // units, columns of the widest, row-major, M ...: a line of columns and rows of a workgroup for each M
{
    for (int i = 4; i < argc; ++i) {
        SkinnyWork w{};
        int64_t wgs;
        const SkinnyForm f = skinny_form(std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[i]), std::atoi(argv[3]), 256, &w, &wgs);
        if (wgs < 0 || w.n_rowblk != (std::atoi(argv[i]) + f.rows - 1) / f.rows)
            return 1;
        std::printf("%d %d\n", f.cols, f.rows);
    }
    return 0;
}
"""


def build(tmp_path, program):
    compiler = shutil.which("g++")
    if compiler is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "few.cpp", tmp_path / "few"
    src.write_text(program)
    subprocess.run([compiler, "-std=c++17", "-O1", "-Wno-unknown-pragmas", "-fsanitize=undefined", "-fno-sanitize-recover=undefined",
                    "-I", CSRC, "-o", str(exe), str(src)], check=True)
    return str(exe)


def test_every_block_of_pruned_columns_is_filled_once(tmp_path):
    """Also where they number 2^31 and more, and beside a product of as many workgroups as a launch takes."""
    res = subprocess.run([build(tmp_path, FILLS)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0 and res.stdout == "ok\n", res.stdout


def test_what_the_tests_on_the_gpu_launch(tmp_path):
    """Row blocks of 8, 16 and 32 rows are each among the launches of test_gpu_gemm.py's
    test_row_major_blocks_of_fewer_rows and test_k_major_blocks_of_fewer_rows, on the 256 compute units of an MI355X."""
    exe = build(tmp_path, FORM)
    rows = [1, 7, 8, 9, 16, 17, 24, 33, 130]
    for row_major, widths in ((1, (96, 2048)), (0, (96, 1024, 4096))):
        seen = set()
        for N in widths:
            cols = round(min(N, 128) * 0.9)
            out = subprocess.run([exe, str(-(-N // 128)), str(cols), str(row_major)] + [str(m) for m in rows],
                                 stdout=subprocess.PIPE, text=True, check=True).stdout
            seen |= {tuple(map(int, line.split())) for line in out.splitlines()}
        assert seen == {(32, 8), (32, 16), (64, 32)} | (set() if row_major else {(32, 32)}), (row_major, seen)


@pytest.mark.gpu
def test_compute_units_of_the_device(tw):
    """What the forms above are worked out for."""
    import torch
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
