// The work queues of a streaming launch: what the host lays out and a workgroup reads an item's place from.
//
// The work of one launch is a matrix of items: `n_all_u` columns (pieces of units that have kept
// K rows first, heaviest first; then pieces of units without; then, with TW_PRUNED_ZERO, the tiles
// whose pruned columns are filled) by `n_mblk` blocks of BM rows.  It is handed out through
// kXcd queues, one per accelerator die: workgroup b runs on die b % kXcd and draws from that
// die's queue only, so the workgroups that share an L2 work on the same rows of A.  A queue owns `n_own` row
// blocks: first, where a workgroup has many items, in groups of kQueueGroup neighbouring row blocks, column after
// column of a group; then column after column over the n_last row blocks left of its own and a share of
// the row blocks that nobody owns; then its share of the columns without steps.  What follows the groups is one list
// for all queues that is dealt out in turn, entry j to queue j % kXcd: a column has n_col_mblk = kXcd * n_last +
// n_mblk - kXcd * n_own entries, of which the first kXcd * n_last are the kXcd owners' row blocks, one of each after the other.
#ifndef TW_QUEUE_H
#define TW_QUEUE_H

#include <cstdint>

#ifdef __HIPCC__
#define TW_QUEUE_FN __host__ __device__ __forceinline__
#else
#define TW_QUEUE_FN inline // (a host program that walks the queues)
#endif

namespace tw {

constexpr int kQueueGroup = 2;

// The entry of a queue: an item, or what stands for its end.
struct Work {
    int col;  // column of the item matrix, n_all_u past the end
    int m0;   // first row
    int rows; // rows [m0, m0 + rows) of A and C, cut at M by the caller
};

// The queues of the items in `a` (n_mblk, n_pipe_u, n_all_u) for `wgs` workgroups; `owned`: the dies own row blocks.
template <class Args> inline void lay_queues(Args &a, bool owned, int64_t wgs)
{
    a.n_own = owned ? a.n_mblk / kXcd : 0;
    const int groups = (int64_t)a.n_pipe_u * a.n_mblk >= 12 * wgs ? a.n_own / kQueueGroup : 0;
    a.n_last = groups > 1 ? a.n_own - (groups - 1) * kQueueGroup : a.n_own;
    // Every eighth row block, as the list deals them out, or neighbours: where a workgroup has few items the former is ahead
    // (M 8192, K 4096, N 1024, half the rows kept 41.2 -> 40.0 us), with the groups neighbours are (load-imbalance stress 348 -> 336).
    a.last_x = groups > 1 ? a.n_last : 1;
    a.last_r = groups > 1 ? 1 : kXcd;
    // (64 bits: a launch of too many items is refused later)
    a.n_lead_items = (int32_t)((int64_t)(a.n_own - a.n_last) * a.n_pipe_u);
    a.n_col_mblk = a.n_mblk - kXcd * (a.n_own - a.n_last);
    a.n_col_items = (int32_t)((int64_t)a.n_pipe_u * a.n_col_mblk);
    a.n_rest_items = (int32_t)(a.n_col_items + (int64_t)(a.n_all_u - a.n_pipe_u) * a.n_mblk);
    a.rb_major = 0;
}

// ... in another order, where nobody owns a row block: all columns of a row block (heaviest first) before the next
template <class Args> inline void order_by_row_blocks(Args &a)
{
    a.rb_major = 1;
    a.n_col_mblk = a.n_all_u;
    a.n_col_items = a.n_rest_items;
}

template <class Args> TW_QUEUE_FN int queue_length(const Args &p, int x)
{
    return p.n_lead_items + (int)(((uint32_t)p.n_rest_items + kXcd - 1 - x) / kXcd);
}

// Entry q of queue x, of `len` entries; bm: rows of a row block.  Every workgroup works its first entry out before its
// first load leaves, by code that comes from memory then: one division, whatever the part of the queue, and the end
// without it.  With a division for each part and the starts of the columns counted die by die, launches of one item a
// workgroup took up to a tenth longer (a quarter of the rows kept: M 4096, K 3072, N 768 15.4 us, 14.6 by this; M 8192, K 4096, N 1024
// 28.6 and 27.4; M 8192, K 4096, N 512 with a tenth 12.7 and 11.8), longer ones 1 - 3 % (VGG16 conv4_2 29.3 and 28.6).
template <class Args> TW_QUEUE_FN Work queue_entry(const Args &p, int x, int q, int len, int bm)
{
    Work w;
    w.col = p.n_all_u;
    w.m0 = 0;
    w.rows = bm;
    if (q >= len)
        return w;
    const bool lead = q < p.n_lead_items;
    uint32_t j = lead ? (uint32_t)q : (uint32_t)(q - p.n_lead_items) * kXcd + x;
    if (p.n_bal > 0) {
        // columns with row blocks of their own height: column u owns the items
        // bal_first[u] .. bal_first[u + 1] - 1 of the list
        int u = 0;
#pragma unroll
        for (int i = 1; i < kBalColumns; ++i)
            u += i < p.n_bal && (int)j >= p.bal_first[i];
        w.col = u;
        w.rows = p.bal_rows[u];
        w.m0 = ((int)j - p.bal_first[u]) * w.rows;
        return w;
    }
    uint32_t per = lead ? kQueueGroup * p.n_pipe_u : p.n_col_mblk;
    const bool fill = !lead && j >= (uint32_t)p.n_col_items; // a column without steps
    if (fill) {
        j -= p.n_col_items;
        per = p.n_mblk;
    }
    const int d = (int)(j / per), r = (int)(j - (uint32_t)d * per);
    int mblk = r;
    w.col = d;
    if (lead) {
        w.col = r / kQueueGroup;
        mblk = x * (p.n_own - p.n_last) + d * kQueueGroup + r % kQueueGroup;
    } else if (fill) {
        w.col += p.n_pipe_u;
    } else {
        if (r < p.n_last * kXcd)
            mblk = x * p.last_x + r / kXcd * p.last_r;
        mblk += (p.n_own - p.n_last) * kXcd;
    }
    if (p.rb_major) {
        w.col = r;
        mblk = d;
    }
    w.m0 = mblk * bm;
    return w;
}

} // namespace tw

#endif
