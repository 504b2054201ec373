// How a launch of the kernel for few rows (tw_gemm_skinny_kernel) is cut into workgroups: what the host works out and a workgroup reads its
// place from, arithmetic on sizes alone.
#ifndef TW_FEW_ROWS_H
#define TW_FEW_ROWS_H

#include <algorithm>
#include <cstdint>

#ifdef __HIPCC__
#define TW_FEW_ROWS_FN __host__ __device__ __forceinline__
#else
#define TW_FEW_ROWS_FN inline // (a host program that walks the workgroups)
#endif

namespace tw {

constexpr int kSkRows = 32;                            // rows m of a workgroup (or eight or sixteen)
constexpr int kSkCols = 64;                            // compact columns of a workgroup, or half of them
constexpr int sk_fill_rows(bool rm) { return rm ? 32 : 64; } // rows m of a tile's pruned columns that a workgroup fills
struct SkinnyWork {
    int32_t n_units, n_rowblk;
    int32_t pieces, piece_shift; // of a unit: 1, 2 or 4, and its logarithm
    int32_t grouped;       // items of a row block in whole groups of eight units
    int32_t grouped_items; // n_rowblk times that
    uint32_t magic;        // 2^32 / grouped, rounded up
    int32_t left;          // units left over
    int32_t dies_per_unit; // kXcd / left
    int32_t gemm_wgs;      // workgroups that multiply; those behind them fill pruned columns
    int32_t fill_wgs, n_fillblk; // so many, sk_fill_rows rows of a tile at a time
};

// The kernel's work on M rows in blocks of `rows`, in pieces of `cols` columns (64 or 32), for units of up to `unit_cols` columns, and its number of
// workgroups, or -1 where that is more than it numbers: it divides a workgroup's number by `grouped` with a multiplication, exact while
// number * grouped stays below 2^32.
inline int64_t skinny_work(int n_units, int unit_cols, int M, SkinnyWork *w, int cols = kSkCols, int rows = kSkRows)
{
    w->n_units = n_units;
    w->piece_shift = unit_cols > 2 * cols ? 2 : unit_cols > cols ? 1 : 0;
    w->pieces = 1 << w->piece_shift;
    w->n_rowblk = (int32_t)(((int64_t)M + rows - 1) / rows);
    w->left = n_units % kXcd;
    w->dies_per_unit = w->left ? kXcd / w->left : 1;
    const int64_t grouped = (int64_t)(n_units - w->left) * w->pieces, grouped_items = grouped * w->n_rowblk;
    const int64_t left_items = w->left ? (int64_t)kXcd * w->pieces * ((w->n_rowblk + w->dies_per_unit - 1) / w->dies_per_unit) : 0;
    if ((grouped_items + left_items) * 64 * 8 > kMaxGridThreads || grouped_items * grouped >= (1ll << 32))
        return -1;
    w->grouped = (int32_t)grouped;
    w->grouped_items = (int32_t)grouped_items;
    w->magic = grouped ? (uint32_t)(((1ull << 32) + grouped - 1) / grouped) : 0u;
    return grouped_items + left_items;
}

// Workgroups on the die that has most of them.
inline int64_t skinny_per_die(const SkinnyWork &w)
{
    return (int64_t)w.grouped / kXcd * w.n_rowblk + (w.left ? (int64_t)w.pieces * ((w.n_rowblk + w.dies_per_unit - 1) / w.dies_per_unit) : 0);
}

// The form a launch takes on `cu` compute units: columns and rows of a workgroup; `w` and the number of workgroups go with it (-1: too many).
struct SkinnyForm {
    int32_t cols, rows;
};
// Pieces of 32 columns while no compute unit gets two workgroups: a workgroup on a compute unit of its own is bound by what
// that fetches (50 bytes a clock, 12 KB a step of 64 columns, 8 KB of 32), and the other compute units are idle.  us with
// pieces of 64 and of 32, K-major and row-major: M 64, K 4608, N 512, half the rows kept 6.5 and 5.0, 12.9 and 12.3; M 64,
// K 2304, N 256 4.6 and 3.8, 8.1 and 7.7; M 256, K 4096, N 1024 (256 workgroups) 5.1 and 4.7, 9.5 and 9.5; four waves,
// M 128, K 768, N 768 3.1 and 2.8, 4.5 and 4.1.  From 288 workgroups on 1.02 - 1.20 of the time, and 1.05 - 1.49.
// Eight or sixteen rows a workgroup instead of 32 while there is a compute unit for each workgroup.  The sums are the same, bit for bit.  us with
// 32 rows and this way, one plan again and again, 80 plans in turn, and 600 (operands out of the L2s, beside them, and of memory):
// Row-major A: a kept row is a load of its own for every m, so that a workgroup is as long as its rows are many (32 loads a step of 64 kept
// rows, of which each holds the address pipe as long as one of 1 KB).  M 1, K 3072, N 768, a quarter kept 6.0 and 3.4, 6.9 and 3.8, 7.9 and 4.7; M 128 (sixteen
// rows) 6.5 and 4.6, 7.3 and 5.1, 8.7 and 6.0; M 64, K 4608, N 512, 0.6 kept 14.0 and 6.2, 17.7 and 8.0, 18.1 and 8.0; 42 problems 0.58 of the time in the
// mean and 0.74 at most, with 80 plans 0.62 and 0.79.
// K-major A: a step of A is one or two loads instead of four, stored and read that much shorter.  M 1, K 3072, N 768, 0.6 kept 4.9 and 3.7, 6.7 and 6.0, 7.5 and 6.8;
// M 32, K 8192, N 1024 7.6 and 6.8, 15.9 and 13.5, 15.8 and 13.4; M 48, K 4096, N 512, a quarter kept 3.6 and 3.4, 4.8 and 4.5, 6.3 and 5.8; 22 problems 0.89 in the
// mean, worst 1.02, with 80 plans 0.94 and 1.03 (N 128, 0.1 kept: 3.32 and 3.41).  Here only up to 5/8 of the compute units: each workgroup asks for
// as many lines of A as one of 32 rows did, and with more of them the L2 falls behind: M 64, K 3072, N 768 (256 workgroups) 4.6 and 5.5 from the L2s, 7.7 and 7.0
// with 80 plans; 385 workgroups and more 1.3 - 1.8 and 1.1 - 1.5 of the time.
inline SkinnyForm skinny_form(int n_units, int unit_cols, int M, bool rm, int cu, SkinnyWork *w, int64_t *wgs)
{
    SkinnyForm f{kSkCols, kSkRows};
    *wgs = skinny_work(n_units, unit_cols, M, w);
    SkinnyWork other;
    const int64_t narrow = skinny_work(n_units, unit_cols, M, &other, kSkCols / 2);
    if (*wgs < 0 || narrow < 0 || skinny_per_die(other) * kXcd > cu)
        return f;
    f.cols = kSkCols / 2;
    *w = other;
    *wgs = narrow;
    for (int rows = 8; rows < kSkRows; rows *= 2) {
        const int64_t n = skinny_work(n_units, unit_cols, M, &other, kSkCols / 2, rows);
        if (n >= 0 && skinny_per_die(other) * kXcd <= (rm ? cu : cu * 5 / 8)) {
            f.rows = rows;
            *w = other;
            *wgs = n;
            break;
        }
    }
    return f;
}

// The workgroups that fill the pruned columns of `n_tiles` tiles, behind w->gemm_wgs of `threads` threads.  A launch of as many workgroups as
// it takes loops over the rest; some are always left, since those that multiply come in eights and 8 * n * 512 is never the limit itself.
inline void skinny_fill(SkinnyWork *w, int n_tiles, int M, bool rm, int threads)
{
    w->n_fillblk = (int32_t)(((int64_t)M + sk_fill_rows(rm) - 1) / sk_fill_rows(rm));
    w->fill_wgs = (int32_t)std::min<int64_t>((int64_t)n_tiles * w->n_fillblk, kMaxGridThreads / threads - w->gemm_wgs);
}

// One of their items: block `blk` of the rows of tile z.  The items number n_tiles * n_fillblk, which can be 2^31 and more: a workgroup goes
// from one to the next by tiles and row blocks instead of by number.  (The step is worked out here rather than brought along: with two more members the
// compiler reads this struct behind the test for a fill, a trip of its own for the product: 0 - 3 % of a launch, and 1 - 2.5 % in the mean where they are asked for ahead of it.)
struct FillPlace {
    int32_t z, blk;
};
TW_FEW_ROWS_FN FillPlace fill_first(const SkinnyWork &w, int wg)
{
    const int z = wg / w.n_fillblk;
    return FillPlace{z, wg - z * w.n_fillblk};
}
TW_FEW_ROWS_FN FillPlace fill_next(const SkinnyWork &w, FillPlace at)
{
    const FillPlace step = fill_first(w, w.fill_wgs);
    at.z += step.z;
    at.blk += step.blk; // (n_fillblk is at most 2^26)
    if (at.blk >= w.n_fillblk) {
        at.blk -= w.n_fillblk;
        ++at.z;
    }
    return at;
}

} // namespace tw
#endif
