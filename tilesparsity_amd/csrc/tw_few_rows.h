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
    int32_t step_z, step_blk;    // fill_wgs as tiles and row blocks
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

// The workgroups that fill the pruned columns of `n_tiles` tiles, behind w->gemm_wgs of `threads` threads.  A launch of as many workgroups as
// it takes loops over the rest; some are always left, since those that multiply come in eights and 8 * n * 512 is never the limit itself.
inline void skinny_fill(SkinnyWork *w, int n_tiles, int M, bool rm, int threads)
{
    w->n_fillblk = (int32_t)(((int64_t)M + sk_fill_rows(rm) - 1) / sk_fill_rows(rm));
    w->fill_wgs = (int32_t)std::min<int64_t>((int64_t)n_tiles * w->n_fillblk, kMaxGridThreads / threads - w->gemm_wgs);
    w->step_z = w->fill_wgs / w->n_fillblk;
    w->step_blk = w->fill_wgs % w->n_fillblk;
}

// One of their items: block `blk` of the rows of tile z.  The items number n_tiles * n_fillblk, which can be 2^31 and more: a workgroup goes
// from one to the next by tiles and row blocks instead of by number (and divides once).
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
    at.z += w.step_z;
    at.blk += w.step_blk; // (n_fillblk is at most 2^26)
    if (at.blk >= w.n_fillblk) {
        at.blk -= w.n_fillblk;
        ++at.z;
    }
    return at;
}

} // namespace tw
#endif
