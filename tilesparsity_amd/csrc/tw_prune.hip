// TW mask producers on the GPU: network-global thresholds on per-tile row norms (and column
// norms) of the importance scores, as the reference's pruning scripts compute them with NumPy
// (Pruning/VGG/prune_algo.py:55-148; Pruning/BERT/utils/MyHook.py:226-313).
//
// The masks are integer results of floating-point comparisons, so every float operation here
// repeats NumPy's, in NumPy's order:
//   * a tile row norm is sqrt(add.reduce(x*x)) / width in float32, the sum being NumPy's
//     pairwise sum along the contiguous axis (8 running sums over blocks of up to 128 elements,
//     halves combined above that);
//   * a column norm accumulates the rows one after the other;
//   * np.percentile with linear interpolation: the two neighbouring order statistics are found
//     here with a radix select, and interpolated here in the arithmetic type NumPy would
//     use for the given kind of `q`;
//   * comparisons are strict.
// This file is compiled with floating-point contraction off (pragma below): a product and the sum
// that takes it stay two rounded operations, as in NumPy.  The __fmul_rn / __fadd_rn intrinsics
// would not do: their bodies live in a header outside the pragma and are fused after inlining.
// sqrtf and the division are the compiler's correctly rounded ones (the __fsqrt_rn / __fdiv_rn
// intrinsics map to the approximate hardware instructions).
#include "tw_device.h"

#include <cmath>
#include <condition_variable>
#include <cstring>
#include <iterator>
#include <mutex>

#pragma clang fp contract(off)

namespace tw {

// A pointer that comes out of a table in memory is not known to point to global memory, and a load
// through it is a flat one, which waits for LDS as well.
template <class T> __device__ __forceinline__ TW_GLOBAL(T) as_global(T *p) { return (TW_GLOBAL(T))p; }

// A load of data that nothing reads again soon (ONCE): it does not push other lines out of the caches.
template <bool ONCE, class T> __device__ __forceinline__ T load_global(TW_GLOBAL(const T) p)
{
    if constexpr (ONCE)
        return __builtin_nontemporal_load(p);
    else
        return *p;
}

// An entry, the same for all lanes, of a table that nobody writes while the kernel runs, through the scalar cache.  (In a kernel that
// stores, the compiler takes the vector path for it, and the wait for it there is one for every load in flight.)
template <class T> __device__ __forceinline__ T load_entry(const T *p)
{
    struct Words {
        uint32_t w[sizeof(T) / 4];
    } a;
    const auto *const src = (const __attribute__((address_space(4))) uint32_t *)(uintptr_t)p;
#pragma unroll
    for (size_t i = 0; i < sizeof(T) / 4; ++i)
        a.w[i] = src[i];
    return __builtin_bit_cast(T, a);
}

// NumPy's pairwise sum of the squares of n <= 128 terms, by a group of 8 adjacent lanes: lane j keeps
// NumPy's running sum r[j] (terms j, j+8, j+16, ...), the three shuffle steps are NumPy's
// ((r0+r1)+(r2+r3)) + ((r4+r5)+(r6+r7)), lane 0 then adds the n % 8 trailing terms.  The result
// is valid in lane 0 of the group.  All reads leave before the chain of additions starts.
__device__ __forceinline__ float pairwise_block(const float *x, int n, int l8)
{
    if (n < 8) {
        float r = 0.0f;
        for (int i = 0; i < n; ++i)
            r = r + x[i] * x[i];
        return r;
    }
    const int n8 = n >> 3;
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i)
        v[i] = x[(i < n8 ? i : 0) * 8 + l8]; // (the others are not added)
    float r = v[0] * v[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) {
        const float sq = v[i] * v[i];
        r = i < n8 ? r + sq : r;
    }
    r = r + __shfl_down(r, 1, 8);
    r = r + __shfl_down(r, 2, 8);
    r = r + __shfl_down(r, 4, 8);
    for (int i = n8 * 8; i < n; ++i)
        r = r + x[i] * x[i];
    return r;
}

// ... and for any n: halves (the first a multiple of 8) are summed separately and added.  PairWalk
// walks the blocks of that tree from left to right; `left` (kPairDepth floats of LDS for each group
// of eight lanes) holds the sums of the left halves whose right halves are still open, one per level,
// and bit d of `path` says that the walk is in the right half at level d.
constexpr int kPairDepth = 26; // 2^31 columns in blocks of 57 and more
struct PairWalk {
    int n, off, size; // all columns; the block the walk stands at
    uint32_t path = 0;
    int depth = 0;
    __device__ explicit PairWalk(int n_) : n(n_) { descend(); }
    __device__ void descend()
    {
        off = 0;
        size = n;
        for (int d = 0; d < depth; ++d) {
            const int n2 = size / 2 - size / 2 % 8;
            const bool right = path >> d & 1u;
            off += right ? n2 : 0;
            size = right ? size - n2 : n2;
        }
        for (; size > 128; ++depth)
            size = size / 2 - size / 2 % 8;
    }
    // takes the block's sum (lane 0 of the group); true, with everything in `sum`, after the last block
    __device__ bool add(float &sum, float *left, int l8)
    {
        for (; depth > 0 && (path >> (depth - 1) & 1u); --depth) {
            sum = left[depth - 1] + sum;
            path &= ~(1u << (depth - 1));
        }
        if (depth == 0)
            return true;
        if (l8 == 0)
            left[depth - 1] = sum;
        path |= 1u << (depth - 1);
        descend();
        return false;
    }
};

constexpr int kNormNotDivided = 1;   // norms are not divided by the tile width
constexpr int kPerTileThreshold = 2; // tile t compares with a threshold of its own (one layer only)

// One entry per layer of a producer call; all layers run in one launch per stage.  The host fills
// the table, and for the 2-D producer plan_2d_kernel fills in what depends on the kept columns
// (n_tiles, norms, rt_begin and the tile table itself).
struct PruneLayer {
    const float *score;
    uint8_t *mask;
    uint8_t *colkeep;     // nullptr: every column counts
    uint8_t *colout;      // the caller's copy of colkeep, or nullptr
    int32_t *tcol0;       // n_tiles + 1 entries, or nullptr: tiles of `granularity` columns
    float *norms;         // [n_tiles][K]
    int32_t K, N, n_tiles, granularity;
    int32_t flags;        // kNormNotDivided, kPerTileThreshold
    int32_t pad_;
    int64_t rt_begin;     // first (row block, tile) item of this layer in the launch-wide numbering
    int64_t el_begin;     // first workgroup of the mask fill likewise (kFillUnits of ceil(K/4) x ceil(N/16) units)
    int64_t col_begin;    // first column of this layer among the pooled column norms
};

__device__ __forceinline__ int tile_begin(const PruneLayer &L, int t)
{
    return L.tcol0 ? as_global(L.tcol0)[t] : min(t * L.granularity, L.N);
}

// The layer that owns item `idx`, given the layers' first items (`stride` bytes apart), for wave-uniform
// items: each lane of a wave keeps one layer's first item in a register, so a look-up is a ballot, and
// the first one a single trip to memory instead of a chain of dependent ones.
class LayerFinder {
public:
    __device__ LayerFinder(const int64_t *begin, size_t stride, int n_layers) : begin_(begin), stride_(stride), n_(n_layers)
    {
        mine_ = at(0);
    }
    __device__ int operator()(int64_t idx) const
    {
        int n = __popcll(__ballot(mine_ <= idx));
        for (int base = 64; base < n_ && n == base; base += 64) // (beyond 64 layers)
            n += __popcll(__ballot(at(base) <= idx));
        return __builtin_amdgcn_readfirstlane(n - 1);
    }

private:
    __device__ int64_t at(int base) const
    {
        const int l = base + (int)(threadIdx.x & 63);
        return l < n_ ? *(TW_GLOBAL(const int64_t))(reinterpret_cast<const char *>(begin_) + (size_t)l * stride_)
                      : (int64_t)0x7fffffffffffffff;
    }
    const int64_t *begin_;
    size_t stride_;
    int n_;
    int64_t mine_;
};

// norms[t*K + k] = ||score[k][tile t]|| / width, pruned columns counting as 0.  A workgroup takes
// one tile of up to 32 rows.  NumPy's order of summation gives every eighth column to one running
// sum, so lanes that read what they add would touch eight 32-byte pieces per load: instead the rows
// go through LDS a block of the sum (at most 128 columns) at a time, loaded along the row (16 bytes a
// lane where the rows are aligned), pruned columns replaced by zeros on the way, and eight lanes per
// row add from there.  The pitch of a staged row is 8 floats past 128, so the eight rows a wave adds
// at a time lie in eight different groups of banks.  The pointers out of the layer table are known to
// be global and no load is conditional: flat or predicated loads wait for each other.  Bound by the
// read: the feed-forward weights of twelve BERT-base layers (226 MB) in 40 us, 5.6 TB/s (a kernel
// that only reads them 35); 92 us when every lane loaded what it added.
constexpr int kNormRows = 32;     // rows of an item: eight lanes each
constexpr int kNormPitch = 136;   // floats; a block of 128 columns with up to 3 before it
template <bool ONCE>
__global__ void __launch_bounds__(256, 6)
    tile_row_norms_kernel(const PruneLayer *layers, int n_layers, const int64_t *n_items, int64_t first_item)
{
    __shared__ __align__(16) float stage[kNormRows * kNormPitch];
    __shared__ float s_left[kNormRows][kPairDepth];
    const int64_t item = first_item + blockIdx.x;
    if (n_items && item >= *n_items)
        return; // (a grid sized for the most tiles the layers can have)
    const PruneLayer L = layers[LayerFinder(&layers->rt_begin, sizeof(PruneLayer), n_layers)(item)];
    const uint32_t idx = (uint32_t)(item - L.rt_begin); // (a call has fewer than 2^31 items)
    const int rblk = (int)(idx / (uint32_t)L.n_tiles), t = (int)(idx - (uint32_t)rblk * (uint32_t)L.n_tiles);
    const int k0 = rblk * kNormRows, nr = min(kNormRows, L.K - k0);
    const int c0 = tile_begin(L, t), w = tile_begin(L, t + 1) - c0;
    const int tid = (int)threadIdx.x, l8 = tid & 7, grp = tid >> 3;
    TW_GLOBAL(const float) const src = as_global(L.score) + (int64_t)k0 * L.N;
    TW_GLOBAL(const uint8_t) const keep = as_global((const uint8_t *)L.colkeep);
    // rows whose starts are aligned are loaded from the 16-byte piece that holds the block's first
    // column to the one that holds its last (which does not reach past the row: N is a multiple of 4)
    const bool vec = (L.N & 3) == 0 && ((uintptr_t)L.score & 15) == 0;
    PairWalk walk(w);
    for (;;) {
        const int c = c0 + walk.off, n = walk.size;
        const int lead = vec ? c & 3 : 0;
        // (loads and LDS writes are unconditional, so that they all leave at once: rows past the
        // item's last repeat that one)
        if (vec) {
            const int r0 = tid >> 5, q0 = tid & 31, w4 = (lead + n + 3) >> 2;
            for (int q = q0; q < w4; q += 32) {
                const int cq = c - lead + q * 4;
                float4 v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    v[i] = __builtin_bit_cast(float4, load_global<ONCE>((TW_GLOBAL(const u32x4))(src + (int64_t)min(r0 + i * 8, nr - 1) * L.N + cq)));
                bool kp[4] = {true, true, true, true};
                if (keep) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        kp[e] = keep[cq + e] != 0;
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    *reinterpret_cast<float4 *>(stage + (r0 + i * 8) * kNormPitch + q * 4) =
                        float4{kp[0] ? v[i].x : 0.0f, kp[1] ? v[i].y : 0.0f, kp[2] ? v[i].z : 0.0f, kp[3] ? v[i].w : 0.0f};
            }
        } else {
            const int r0 = tid >> 6, q0 = tid & 63;
            for (int q = q0; q < n; q += 64) {
                const bool kp = !keep || keep[c + q];
                float v[kNormRows / 4];
#pragma unroll
                for (int i = 0; i < kNormRows / 4; ++i)
                    v[i] = load_global<ONCE>(src + (int64_t)min(r0 + i * 4, nr - 1) * L.N + c + q);
#pragma unroll
                for (int i = 0; i < kNormRows / 4; ++i)
                    stage[(r0 + i * 4) * kNormPitch + q] = kp ? v[i] : 0.0f;
            }
        }
        __syncthreads();
        float s = pairwise_block(stage + grp * kNormPitch + lead, n, l8); // (rows past the last: unused)
        if (walk.add(s, s_left[grp], l8)) {
            if (l8 == 0 && grp < nr) // both operations correctly rounded
                as_global(L.norms)[(int64_t)t * L.K + k0 + grp] = (L.flags & kNormNotDivided) ? sqrtf(s) : sqrtf(s) / (float)w;
            return;
        }
        __syncthreads(); // the stage is written again
    }
}

// cnorm[pooled c] = ||score[:, c]|| / K, the rows accumulated in order.  The chain of K additions
// per column is sequential by definition; everything around it is not: a workgroup takes 32
// columns; four waves load 64 rows at a time (eight such groups in flight in registers: 64 KB a
// workgroup, as much as hides the way to memory), square them and leave them in LDS as [column][row];
// a fifth adds, four rows per LDS read.
// All layers share one launch; a column block belongs to one layer (blk_begin: its first block).
// 26 us for the 126 MB of VGG16's layers (4.8 TB/s, the chain of 4608 additions being about as long);
// 117 us with a thread per column that loads 32 rows ahead of its additions.
struct ColLayer {
    const float *score;
    int32_t K, N;
    int64_t col_begin; // first column of this layer in the pooled numbering
    int64_t blk_begin; // first block of 32 columns likewise
};
constexpr int kColRows = 64, kColCols = 32, kColPitch = kColRows + 4, kColDeep = 8;
constexpr int kColThreads = 320; // four waves that load, one that adds
__global__ void __launch_bounds__(kColThreads) col_norms_kernel(const ColLayer *layers, int n_layers, float *cnorm, int64_t first_blk)
{
    __shared__ __align__(16) float sq[2][kColCols * kColPitch];
    const ColLayer L = layers[LayerFinder(&layers->blk_begin, sizeof(ColLayer), n_layers)(first_blk + blockIdx.x)];
    const int c0 = (int)(first_blk + blockIdx.x - L.blk_begin) * kColCols;
    const int tid = (int)threadIdx.x, col = tid & 31;
    const int K = L.K, N = L.N;
    const int n_grp = (K + kColRows * kColDeep - 1) / (kColRows * kColDeep) * kColDeep; // in whole rounds of kColDeep
    if (tid >= 256) { // the adding wave: lanes 0 - 31 and, as an unused copy, 32 - 63
        float acc = 0.0f;
        const float *const x = sq[0] + col * kColPitch;
        for (int g = 0; g < n_grp; ++g) {
            __syncthreads(); // group g is staged
            const float *const s = x + (g & 1) * (kColCols * kColPitch);
            float4 a[kColRows / 4];
#pragma unroll
            for (int j = 0; j < kColRows / 4; ++j)
                a[j] = *reinterpret_cast<const float4 *>(s + j * 4);
#pragma unroll
            for (int j = 0; j < kColRows / 4; ++j) {
                acc = acc + a[j].x;
                acc = acc + a[j].y;
                acc = acc + a[j].z;
                acc = acc + a[j].w;
            }
        }
        if (tid < 256 + kColCols && c0 + col < N)
            cnorm[L.col_begin + c0 + col] = sqrtf(acc) / (float)K;
        return;
    }
    const int r0 = tid >> 5;
    // (a column past the layer's last repeats that one and is dropped at the end)
    TW_GLOBAL(const float) const p = as_global(L.score) + min(c0 + col, N - 1);
    float v[kColDeep][8];
    auto load = [&](int g, float (&d)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            d[i] = p[(int64_t)min(g * kColRows + r0 + i * 8, K - 1) * N];
        }
    };
    // (groups past the last repeat its last row and count as zeros: no load is conditional, so the
    // waits for them are exact counts)
#pragma unroll
    for (int d = 0; d < kColDeep; ++d)
        load(d, v[d]);
    for (int g0 = 0; g0 < n_grp; g0 += kColDeep) {
#pragma unroll
        for (int d = 0; d < kColDeep; ++d) {
            const int g = g0 + d;
            // (the adding wave has read this stage: it read group g - 2 before barrier g - 1)
            float *const s = sq[d & 1];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float x = g * kColRows + r0 + i * 8 < K ? v[d][i] : 0.0f; // (a zero leaves a sum of squares alone)
                s[col * kColPitch + r0 + i * 8] = x * x;
            }
            load(g + kColDeep, v[d]);
            __syncthreads();
        }
    }
}

// order-preserving map float -> uint32
__device__ __forceinline__ uint32_t sort_key(float v)
{
    const uint32_t b = __float_as_uint(v);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_to_float(uint32_t key)
{
    return __uint_as_float((key & 0x80000000u) ? (key & 0x7FFFFFFFu) : ~key);
}

// np.percentile with linear interpolation, on the device: a radix select of the k-th smallest key in
// three passes over the values (11 + 11 + 10 bits of the key), and what the interpolation needs
// beside it, its upper neighbour, out of the same passes: the values above the digits fixed so far
// leave their minimum, those that share all digits but the last leave it in the last histogram.
// (A first digit of 11 bits - sign, exponent, two bits of mantissa - also spreads the values of a
// layer over a few dozen counters; with 8 bits, two octaves a digit, most lanes of a wave met in one
// or two LDS counters: 38 us a pass over 31.5 M values.)
// Pass p counts the values that agree with the digits before it; which digit holds the rank is
// worked out of the histogram by every workgroup of the next pass, and the threshold out of the
// last one by whatever uses it (threshold_of).
constexpr int kSelBins = 2048;
constexpr uint32_t kNanFrom = 0x7F800001u; // |x| from here on is no number
struct SelectHead {               // the wanted rank and the interpolation above it
    int64_t n;                    // number of values
    unsigned long long rank0;     // 0-based rank of the wanted value
    double gamma64;
    float gamma32;
    int32_t top;                  // the percentile is the largest value
    int32_t f64;                  // the interpolation runs in float64
    int32_t pad_;
};
struct SelectState {
    unsigned long long hist[3][kSelBins];
    SelectHead head;
    unsigned long long rank[3];   // rank among the values that match before pass p (from pass 1 on)
    uint32_t prefix[3];           // their common leading bits, as the value of the bits above pass p's digit
    uint32_t min_gt;              // smallest key above the group the passes so far narrowed down to (0xFFFFFFFF: none)
    // mixed masks: the selection first narrows the elements down to those between two values
    float lo, hi;                 // the bracket
    uint32_t cut[2][2];           // of an element without and with a mask byte: the first |x| whose score is inside it, the first beyond (as bits)
    float row_norm;               // what the norms of kept rows are above (masks out of norms; the sample's kernel leaves it)
    uint32_t room;                // values inside it that a wave can keep aside
    uint32_t key_base;            // the passes' digits are those of key - key_base,
    int32_t key_bits;             // which has this many bits (up to 22: two passes hold them all, the third has nothing to do)
    unsigned long long below;     // elements below the bracket,
    int32_t narrowed;             // and whether the selection runs over those inside only
};

// Rank and weight of np.percentile(v[0..n), q): with q_is_f64 == 0 (q was a Python number) the
// quantile q/100, the virtual index (n-1)*quantile and the interpolation are float32; with 1 (q was
// a NumPy float64) they are float64, only the difference of the two neighbours stays float32.
__device__ void select_rank(SelectHead *h, int64_t n, double q, int q_is_f64)
{
    int64_t lo;
    bool top;
    h->gamma32 = 0.0f;
    h->gamma64 = 0.0;
    if (q_is_f64) {
        const double quant = q / 100.0;
        const double virt = (double)(n - 1) * quant;
        top = virt >= (double)(n - 1);
        lo = top ? n - 1 : (int64_t)floor(virt);
        h->gamma64 = virt - floor(virt);
    } else {
        const float quant = (float)q / 100.0f;
        const float virt = (float)(n - 1) * quant;
        top = virt >= (float)(n - 1);
        lo = top ? n - 1 : (int64_t)floorf(virt);
        h->gamma32 = virt - floorf(virt);
    }
    h->n = n;
    h->top = top;
    h->f64 = q_is_f64;
    h->rank0 = (unsigned long long)min(lo, n - 1);
}
__device__ void select_begin(SelectState *st, int64_t n, double q, int q_is_f64)
{
    select_rank(&st->head, n, q, q_is_f64);
    st->min_gt = 0xFFFFFFFFu;
    st->lo = -INFINITY;
    st->hi = INFINITY;
    st->cut[0][0] = st->cut[1][0] = 0;
    st->cut[0][1] = st->cut[1][1] = kNanFrom;
    st->key_base = 0;
    st->key_bits = 32;
}

// The digits are those of key - base, for keys known to lie within `bits` bits above `base` (all keys:
// 0 and 32): 11 bits, 11 bits and what is left of them.
struct KeyRange {
    uint32_t base;
    int shift[3]; // of each pass's digit
    __device__ KeyRange(uint32_t base_, int bits) : base(base_), shift{max(bits - 11, 0), max(bits - 22, 0), 0} {}
    __device__ int lead_shift(int pass) const { return pass == 0 ? 32 : shift[pass - 1]; } // the digits before: key >> this
    __device__ uint32_t digit(int pass, uint32_t k) const
    {
        return (k >> shift[pass]) & (pass == 0 ? kSelBins - 1u : (1u << (shift[pass - 1] - shift[pass])) - 1u);
    }
};

// The digit of a finished pass whose counts (NB of them) hold `rank`, the rank among the values with
// that digit and how many those are, and (NEXT) the next digit any value has (0xFFFFFFFF: none); called by
// all NT threads of a workgroup, the same values come back to every one.  A rank that is not below the sum of
// the counts cannot happen; it comes back as kLostRank, which no later pass finds either, and ends the
// call with an error.
constexpr unsigned long long kLostRank = ~0ull;
struct Digit {
    unsigned long long rest, count;
    uint32_t digit, next;
};
// (T: what the counts are and, counts of a launch's values fitting one or the other, what they add up to)
template <int NT, int NB, bool NEXT = false, class T> __device__ Digit find_digit(const T *hist, unsigned long long rank)
{
    constexpr int PER = NB / NT;
    __shared__ T s_wave[NT / 64];
    __shared__ Digit s_d;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    T c[PER], sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i)
        c[i] = hist[tid * PER + i];
#pragma unroll
    for (int i = 0; i < PER; ++i)
        sum += c[i];
    T incl = wave_scan(sum);
    if (lane == 63)
        s_wave[wave] = incl;
    if (tid == 0)
        s_d = Digit{kLostRank, 1, (uint32_t)NB - 1u, 0xFFFFFFFFu};
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) // (all of them at once, not one after another)
        incl += w < wave ? s_wave[w] : 0;
    T before = incl - sum;
    uint32_t next = 0xFFFFFFFFu; // the first digit with a value and more than `rank` values before it
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        if (before <= rank && rank < (unsigned long long)before + c[i]) { // exactly one digit
            s_d.digit = tid * PER + i;
            s_d.rest = rank - before;
            s_d.count = c[i];
        }
        if (NEXT && before > rank && c[i])
            next = min(next, (uint32_t)(tid * PER + i));
        before += c[i];
    }
    if (NEXT) { // (one LDS atomic per wave: hundreds on one word take microseconds)
        next = wave_min(next);
        if (lane == 0 && next != 0xFFFFFFFFu)
            atomicMin(&s_d.next, next);
    }
    __syncthreads();
    const Digit d = s_d;
    __syncthreads(); // the shared words are written again by the next call
    return d;
}

// A threshold in both types; values of the type of NumPy's result are compared with it, strictly.
struct Threshold {
    double v64;
    float v32;
    bool f64;
    bool lost; // no value had the wanted rank
    __device__ bool passed_by(float v) const { return f64 ? (double)v > v64 : v > v32; }
    // the float that the same floats are above
    __device__ float in_float() const
    {
        const float near = (float)v64;
        return !f64 ? v32 : (double)near > v64 ? nextafterf(near, -INFINITY) : near;
    }
};

// NumPy's two-sided linear interpolation between the k-th smallest value a and its upper
// neighbour b (a again if it is repeated, or if the index is the last one): float32 throughout
// for a float32 gamma, float64 with a float32 difference b - a otherwise.
__device__ Threshold interpolate(const SelectHead *st, uint32_t key_a, uint32_t key_b)
{
    const float a = key_to_float(key_a);
    const float b = st->top || key_b == 0xFFFFFFFFu ? a : key_to_float(key_b);
    const float diff = b - a;
    if (st->f64) {
        const double g = st->gamma64;
        const double prod = g >= 0.5 ? (double)diff * (1.0 - g) : (double)diff * g;
        const double r = g >= 0.5 ? (double)b - prod : (double)a + prod;
        return Threshold{r, (float)r, true, false};
    }
    const float g = st->gamma32;
    const float prod = g >= 0.5f ? diff * (1.0f - g) : diff * g;
    const float r = g >= 0.5f ? b - prod : a + prod;
    return Threshold{(double)r, r, false, false};
}

// The threshold out of the counts of the finished last pass, by all NT threads of a workgroup: the key
// of the wanted value, and the key above it where that value is not repeated.  Whatever uses a
// threshold works it out itself: a kernel of its own for it, or a last workgroup of the last pass,
// is a chain of trips to memory of 5 to 10 us with the chip idle.
template <int NT> __device__ Threshold threshold_of(const SelectState *st)
{
    __shared__ Threshold s_t;
    const uint32_t min_gt = st->min_gt;
    const uint32_t base = st->key_base;
    const KeyRange range(base, st->key_bits);
    const bool two = st->key_bits <= 22;
    const uint32_t lead = two ? st->prefix[1] << range.lead_shift(1) : st->prefix[2] << range.lead_shift(2);
    const Digit d = two ? find_digit<NT, kSelBins, true>(st->hist[1], st->rank[1]) : find_digit<NT, 1024, true>(st->hist[2], st->rank[2]);
    if (threadIdx.x == 0) {
        const uint32_t key_a = base + (lead | d.digit);
        uint32_t key_b = key_a;
        if (d.rest + 1 >= d.count) // the wanted value is the last of its kind
            key_b = d.next != 0xFFFFFFFFu ? base + (lead | d.next) : min_gt;
        s_t = interpolate(&st->head, key_a, key_b);
        s_t.lost = d.rest == kLostRank;
    }
    __syncthreads();
    return s_t;
}

// Calls f(value) for every element of v[0..n) once, the first `workgroups` of blockIdx.x sharing the
// work: 16-byte loads over the aligned middle (four of them in flight per thread), single
// elements at the ragged ends.
template <class F> __device__ __forceinline__ void for_each_value(const float *v, int64_t n, int workgroups, F f)
{
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nthr = (int64_t)workgroups * blockDim.x;
    const int64_t head = min(n, (int64_t)((16 - ((uintptr_t)v & 15)) & 15) >> 2);
    const int64_t nvec = (n - head) >> 2;
    const float4 *v4 = reinterpret_cast<const float4 *>(v + head);
    int64_t i = tid;
    for (; i + 3 * nthr < nvec; i += 4 * nthr) {
        const float4 a = v4[i], b = v4[i + nthr], c = v4[i + 2 * nthr], d = v4[i + 3 * nthr];
        f(a.x); f(a.y); f(a.z); f(a.w);
        f(b.x); f(b.y); f(b.z); f(b.w);
        f(c.x); f(c.y); f(c.z); f(c.w);
        f(d.x); f(d.y); f(d.z); f(d.w);
    }
    for (; i < nvec; i += nthr) {
        const float4 a = v4[i];
        f(a.x); f(a.y); f(a.z); f(a.w);
    }
    // the elements before the first and after the last whole vector
    const int64_t tail0 = head + 4 * nvec;
    for (int64_t j = tid; j < head + (n - tail0); j += nthr)
        f(v[j < head ? j : tail0 + (j - head)]);
}

// One value of pass PASS: counted where it agrees with the digits before, remembered as the
// smallest above them where it lies above.
template <int PASS>
__device__ __forceinline__ void select_count(uint32_t key, const KeyRange &r, uint32_t prefix, unsigned int *s_h, uint32_t &mn)
{
    const uint32_t k = key - r.base;
    const uint32_t lead = PASS == 0 ? 0u : k >> r.lead_shift(PASS);
    if (PASS == 0 || lead == prefix)
        atomicAdd(&s_h[r.digit(PASS, k)], 1u);
    else if (lead > prefix)
        mn = min(mn, key);
}

// What a workgroup of pass PASS does before it counts: the digits so far (its first workgroup
// leaves them for the next pass), cleared counters.  rank0: the rank before the first pass.
template <int PASS, int NT>
__device__ void select_enter(SelectState *st, const KeyRange &range, unsigned int *s_h, uint32_t *s_min, unsigned long long rank0,
                             uint32_t &prefix, unsigned long long &rank)
{
    for (int i = (int)threadIdx.x; i < kSelBins; i += NT)
        s_h[i] = 0;
    if (threadIdx.x == 0)
        *s_min = 0xFFFFFFFFu;
    prefix = 0;
    rank = rank0;
    if (PASS > 0) {
        const Digit d = find_digit<NT, kSelBins>(st->hist[PASS > 0 ? PASS - 1 : 0], PASS == 2 ? st->rank[1] : rank0);
        prefix = PASS == 2 ? st->prefix[1] << (range.shift[0] - range.shift[1]) | d.digit : d.digit;
        rank = d.rest;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            st->prefix[PASS] = prefix;
            st->rank[PASS] = rank;
        }
    }
    __syncthreads();
}

// ... and after it has counted: its counts join those of the others.
template <int PASS, int NT> __device__ void select_leave(SelectState *st, unsigned int *s_h, uint32_t *s_min, uint32_t mn)
{
    if (PASS > 0) {
        mn = wave_min(mn);
        if ((threadIdx.x & 63) == 0 && mn != 0xFFFFFFFFu)
            atomicMin(s_min, mn);
    }
    __syncthreads();
    for (int i = (int)threadIdx.x; i < kSelBins; i += NT)
        if (s_h[i])
            atomicAdd(&st->hist[PASS][i], (unsigned long long)s_h[i]);
    if (PASS > 0 && threadIdx.x == 0 && *s_min != 0xFFFFFFFFu)
        atomicMin(&st->min_gt, *s_min);
}

// Pass PASS over v[0 .. st->n).  The selection works on segments of equal length laid end to end
// (one segment for the network-wide thresholds, one per tile for per-tile thresholds): segment g =
// blockIdx.y uses state st[g] and values v[g*n .. g*n+n).
template <int PASS> __global__ void __launch_bounds__(256) select_hist_kernel(const float *v, SelectState *st)
{
    __shared__ unsigned int s_h[kSelBins];
    __shared__ uint32_t s_min;
    st += blockIdx.y;
    const int64_t n = st->head.n;
    uint32_t prefix, mn = 0xFFFFFFFFu;
    unsigned long long rank;
    const KeyRange range(0, 32);
    select_enter<PASS, 256>(st, range, s_h, &s_min, st->head.rank0, prefix, rank);
    for_each_value(v + (int64_t)blockIdx.y * n, n, (int)gridDim.x, [&](float x) { select_count<PASS>(sort_key(x), range, prefix, s_h, mn); });
    select_leave<PASS, 256>(st, s_h, &s_min, mn);
}

// The selection in one workgroup and its LDS, for a few ten thousand values (the columns of a network, a
// sample).  The digits are those of the keys' own range, so that the values spread over all counters:
// lanes of a wave that meet in one LDS counter take turns.
template <class V> __device__ KeyRange key_range_in_block(V each)
{
    __shared__ uint32_t s_lo, s_hi;
    if (threadIdx.x == 0) {
        s_lo = 0xFFFFFFFFu;
        s_hi = 0;
    }
    __syncthreads();
    uint32_t lo = 0xFFFFFFFFu, hi = 0;
    each([&](uint32_t k) {
        lo = min(lo, k);
        hi = max(hi, k);
    });
    lo = wave_min(lo);
    hi = wave_max(hi);
    if ((threadIdx.x & 63) == 0) {
        atomicMin(&s_lo, lo);
        atomicMax(&s_hi, hi);
    }
    __syncthreads();
    return KeyRange(s_lo, s_hi > s_lo ? 32 - __clz(s_hi - s_lo) : 1);
}
// one pass: rank becomes the rank among the values that share the digits so far
template <int PASS, int NT, class V>
__device__ Digit count_in_block(V each, const KeyRange &range, unsigned long long &rank, uint32_t &prefix, unsigned int *s_h,
                                uint32_t &mn)
{
    for (int i = (int)threadIdx.x; i < kSelBins; i += NT)
        s_h[i] = 0;
    __syncthreads();
    each([&](uint32_t k) { select_count<PASS>(k, range, prefix, s_h, mn); });
    __syncthreads();
    const Digit d = find_digit<NT, PASS == 2 ? 1024 : kSelBins, PASS != 0>(s_h, rank);
    prefix = PASS == 0 ? d.digit : prefix << (range.lead_shift(PASS) - range.shift[PASS]) | d.digit;
    rank = d.rest;
    return d;
}
// (each(f): f of every key of this thread's)
template <int NT, class V> __device__ Threshold select_in_block(V each, const SelectHead *h, unsigned int *s_h)
{
    __shared__ uint32_t s_min;
    __shared__ Threshold s_t;
    if (threadIdx.x == 0)
        s_min = 0xFFFFFFFFu;
    const KeyRange range = key_range_in_block(each);
    uint32_t prefix = 0, mn = 0xFFFFFFFFu;
    unsigned long long rank = h->rank0;
    count_in_block<0, NT>(each, range, rank, prefix, s_h, mn);
    Digit d = count_in_block<1, NT>(each, range, rank, prefix, s_h, mn);
    if (range.shift[1] > 0) // (else two digits hold all of the range)
        d = count_in_block<2, NT>(each, range, rank, prefix, s_h, mn);
    mn = wave_min(mn);
    if ((threadIdx.x & 63) == 0)
        atomicMin(&s_min, mn);
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t a = range.base + prefix;
        s_t = interpolate(h, a, d.rest + 1 < d.count ? a : d.next != 0xFFFFFFFFu ? a - d.digit + d.next : s_min);
        s_t.lost = d.rest == kLostRank;
    }
    __syncthreads();
    return s_t;
}

// What a call leaves for the host in its page of pinned memory.
struct Mail {
    double thr_rows, thr_cols;
    int32_t lost; // cleared by the host, set by whoever's selection lost its rank
};

// the thresholds of several segments, or one that only the host wants
__global__ void __launch_bounds__(256) select_finish_kernel(const SelectState *st, Threshold *out, Mail *mail)
{
    const Threshold t = threshold_of<256>(st + blockIdx.x);
    if (threadIdx.x == 0) {
        out[blockIdx.x] = t;
        if (t.lost)
            mail->lost = 1;
    }
}

// One threshold per tile: workgroup t selects among the K norms of tile t, which it keeps in LDS.  The
// passes over all tiles with counters in memory took 49 KB of them a tile, cleared and read again for
// a few hundred norms: K 768, N 4096 in tiles of one column 245 against 861 us a call, in tiles of
// eight 63 against 145.  They remain for tiles of more than kTileSelect norms.
constexpr int kTileSelect = 8192;
template <int STAGE> __global__ void __launch_bounds__(256) tile_select_kernel(const float *norms, int K, double q, int q_is_f64,
                                                                               Threshold *out, Mail *mail, int64_t first_tile)
{
    __shared__ unsigned int s_h[kSelBins];
    __shared__ SelectHead s_head;
    __shared__ float s_v[STAGE];
    const int64_t tile = first_tile + blockIdx.x;
    const float *const v = norms + tile * K;
    const int tid = (int)threadIdx.x;
    for (int i0 = tid; i0 < K; i0 += 256 * 4) { // four loads in flight
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            x[e] = v[min(i0 + e * 256, K - 1)];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (i0 + e * 256 < K)
                s_v[i0 + e * 256] = x[e];
    }
    if (tid == 0)
        select_rank(&s_head, K, q, q_is_f64);
    __syncthreads();
    const Threshold t = select_in_block<256>(
        [&](auto f) {
            for (int i = tid; i < K; i += 256)
                f(sort_key(s_v[i]));
        },
        &s_head, s_h);
    if (tid == 0) {
        out[tile] = t;
        if (t.lost)
            mail->lost = 1;
    }
}

// Between the column stage and the row stage of the 2-D producer, one workgroup: the threshold over
// all column norms, the column masks, every layer's tiles (they end after every `granularity` kept
// columns) and where its norms and its row-norm items begin, and the state of the row selection.
// All on the device, so that the call needs no trip to the host between its stages.
// What bounds it is the chain of LDS trips and barriers of one workgroup: the keys stay in registers over the selection's
// passes, and all layers' columns are taken together in groups of 64, the waves a run of groups each, and then every group's
// tiles by a thread of its own from the sums of the groups before it.  VGG16's layers (8832 columns) 31 -> 22 us; in front of
// that a wave took a layer, group after group (N 4096: 64 times 570 cycles, 15 us).
constexpr int kPlanThreads = 1024;
constexpr int kPlanStage = 12288; // column norms kept in LDS; more of them are read from memory in every pass
constexpr int kPlanGroups = 2 * kPlanThreads; // groups of 64 columns at a time
__global__ void __launch_bounds__(kPlanThreads)
    plan_2d_kernel(PruneLayer *layers, int n_layers, const float *cnorm, int64_t n_cols, float *norms,
                   SelectState *st_rows, int64_t *n_items, double q, int q_is_f64, Mail *mail)
{
    __shared__ unsigned int s_h[kSelBins];
    __shared__ SelectHead s_head;
    __shared__ int64_t s_norm[kPlanThreads], s_item[kPlanThreads];
    __shared__ float s_cn[kPlanStage];
    __shared__ unsigned long long s_bits[kPlanGroups]; // which columns of a group are kept
    __shared__ uint16_t s_layer[kPlanGroups];
    __shared__ uint32_t s_first[kPlanThreads + 1];     // first group of each layer
    __shared__ uint32_t s_start[kPlanThreads];         // kept columns of the layers before it
    __shared__ uint32_t s_sum[kPlanThreads / 64];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool staged = n_cols <= kPlanStage;
    constexpr int PER = kPlanStage / kPlanThreads;
    float v[PER];
    if (staged) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
            v[i] = cnorm[min((int64_t)tid + i * kPlanThreads, n_cols - 1)];
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (tid + i * kPlanThreads < n_cols)
                s_cn[tid + i * kPlanThreads] = v[i];
    }
    if (tid == 0)
        select_rank(&s_head, n_cols, q, q_is_f64);
    __syncthreads();
    auto norm_of = [&](int64_t i) -> float {
        if (staged)
            return s_cn[i];
        return as_global(cnorm)[i];
    };
    const Threshold thr = select_in_block<kPlanThreads>(
        [&](auto f) {
            if (staged) {
#pragma unroll
                for (int i = 0; i < PER; ++i)
                    if (tid + i * kPlanThreads < n_cols)
                        f(sort_key(v[i]));
            } else {
                for (int i = tid; i < (int)n_cols; i += kPlanThreads)
                    f(sort_key(as_global(cnorm)[i]));
            }
        },
        &s_head, s_h);
    if (tid == 0) {
        mail->thr_cols = thr.v64;
        if (thr.lost)
            mail->lost = 1;
    }
    // sums over the threads up to this one (modulo 2^32: only differences are used), and over all
    auto scan = [&](uint32_t mine, uint32_t &total) {
        uint32_t incl = wave_scan(mine);
        if (lane == 63)
            s_sum[wave] = incl;
        __syncthreads();
        total = 0;
#pragma unroll
        for (int w = 0; w < kPlanThreads / 64; ++w) {
            incl += w < wave ? s_sum[w] : 0u;
            total += s_sum[w];
        }
        __syncthreads();
        return incl;
    };
    int64_t norm_carry = 0, item_carry = 0;
    for (int base = 0; base < n_layers; base += kPlanThreads) {
        const int cnt = min(kPlanThreads, n_layers - base);
        uint32_t n_groups;
        s_first[tid + 1] = scan(tid < cnt ? ((uint32_t)layers[base + tid].N + 63u) / 64u : 0u, n_groups);
        if (tid == 0)
            s_first[0] = 0;
        __syncthreads();
        uint32_t carry = 0; // kept columns of the groups before these
        for (uint32_t g0 = 0; g0 < n_groups; g0 += kPlanGroups) {
            const uint32_t ng = min((uint32_t)kPlanGroups, n_groups - g0);
            // ---- which columns are kept: a run of groups a wave
            const uint32_t run = (ng + kPlanThreads / 64 - 1) / (kPlanThreads / 64);
            const uint32_t begin = g0 + wave * run, stop = min(begin + run, g0 + ng);
            int l = 0;
            for (int step = kPlanThreads / 2; step > 0 && begin < stop; step >>= 1) // the layer of its first group
                l += l + step < cnt && s_first[l + step] <= begin ? step : 0;
            for (uint32_t g = begin; g < stop; ++l) {
                l = __builtin_amdgcn_readfirstlane(l);
                const PruneLayer &L = layers[base + l];
                const int64_t first = L.col_begin;
                TW_GLOBAL(uint8_t) const colkeep = as_global(L.colkeep);
                TW_GLOBAL(uint8_t) const colout = as_global(L.colout);
                const int N = L.N;
                const uint32_t l0 = s_first[l], l1 = min(s_first[l + 1], stop);
                for (; g < l1; ++g) {
                    const int c = (int)(g - l0) * 64 + lane;
                    const float x = c < N ? norm_of(first + c) : 0.0f;
                    const bool keep = c < N && thr.passed_by(x);
                    const unsigned long long b = __ballot(keep);
                    if (c < N) {
                        colkeep[c] = keep ? 1 : 0;
                        if (colout)
                            colout[c] = keep ? 1 : 0;
                    }
                    if (lane == 0) {
                        s_bits[g - g0] = b;
                        s_layer[g - g0] = (uint16_t)l;
                    }
                }
            }
            __syncthreads();
            // ---- kept columns before each group
            uint32_t at[2], in[2];
#pragma unroll
            for (int e = 0; e < 2; ++e)
                in[e] = (uint32_t)tid * 2 + e < ng ? (uint32_t)__popcll(s_bits[tid * 2 + e]) : 0u;
            uint32_t all;
            at[0] = carry + scan(in[0] + in[1], all) - in[0] - in[1];
            at[1] = at[0] + in[0];
            carry += all;
#pragma unroll
            for (int e = 0; e < 2; ++e)
                if ((uint32_t)tid * 2 + e < ng) {
                    const int gl = s_layer[tid * 2 + e];
                    if (s_first[gl] == g0 + tid * 2 + e)
                        s_start[gl] = at[e];
                }
            __syncthreads();
            // ---- the tiles that end in each group
#pragma unroll 1
            for (int e = 0; e < 2; ++e) {
                const uint32_t g = g0 + tid * 2 + e;
                if (g >= g0 + ng)
                    break;
                const int gl = s_layer[g - g0];
                PruneLayer &L = layers[base + gl];
                const int N = L.N, G = L.granularity, K = L.K;
                TW_GLOBAL(int32_t) const tcol0 = as_global(L.tcol0);
                const unsigned long long bits = s_bits[g - g0];
                const int before = (int)(at[e] - s_start[gl]), here = (int)in[e];
                int tile = before / G;
                for (int64_t need = (int64_t)(tile + 1) * G - before; need <= here; need += G) {
                    int pos = 0, n = (int)need; // the n-th kept column of the group
#pragma unroll
                    for (int half = 32; half > 0; half >>= 1) {
                        const int low = __popcll(bits >> pos & ((1ull << half) - 1ull));
                        pos += n > low ? half : 0;
                        n -= n > low ? low : 0;
                    }
                    ++tile;
                    const int c = (int)(g - s_first[gl]) * 64 + pos;
                    if (c + 1 < N)
                        tcol0[tile] = c + 1;
                }
                if (g + 1 == s_first[gl + 1]) {
                    // tiles that ended before the last column, and the one that takes the rest
                    const int kept = before + here;
                    const bool last_col_ends = kept > 0 && kept % G == 0 && (bits >> ((N - 1) & 63) & 1ull);
                    const int nt = kept / G - (last_col_ends ? 1 : 0) + 1;
                    tcol0[0] = 0;
                    tcol0[nt] = N;
                    L.n_tiles = nt;
                    s_norm[gl] = (int64_t)K * nt;
                    s_item[gl] = (int64_t)((K + kNormRows - 1) / kNormRows) * nt;
                }
            }
            __syncthreads();
        }
        const int64_t my_norm = tid < cnt ? s_norm[tid] : 0, my_item = tid < cnt ? s_item[tid] : 0;
        for (int off = 1; off < cnt; off <<= 1) { // inclusive sums over the layers
            const int64_t a = tid >= off && tid < cnt ? s_norm[tid - off] : 0;
            const int64_t b = tid >= off && tid < cnt ? s_item[tid - off] : 0;
            __syncthreads();
            if (tid < cnt) {
                s_norm[tid] += a;
                s_item[tid] += b;
            }
            __syncthreads();
        }
        if (tid < cnt) {
            layers[base + tid].norms = norms + norm_carry + s_norm[tid] - my_norm;
            layers[base + tid].rt_begin = item_carry + s_item[tid] - my_item;
        }
        norm_carry += s_norm[cnt - 1];
        item_carry += s_item[cnt - 1];
        __syncthreads();
    }
    if (tid == 0) {
        *n_items = item_carry;
        select_begin(st_rows, norm_carry, q, q_is_f64);
    }
}

// Start of a call: up to kBlobWords words of the call's tables, handed over in the kernel arguments, go
// to device memory, the histograms of `n_states` selections are cleared and, where n > 0, their ranks
// worked out.  One launch (or a few, for tables of more than some twenty layers) instead of a copy
// from host memory and the wait for it.
constexpr int kBlobWords = 960; // (a launch takes 4 KB of arguments)
struct Blob {
    uint32_t w[kBlobWords];
};
struct SetupSelect {
    SelectState *st;
    int64_t n;
    double q;
    int32_t n_states, q_is_f64;
    uint32_t room;
    int32_t pad_;
};
// (`a`, the words, is the kernel's first argument; by the launch's first `workgroups`)
__device__ __forceinline__ void prune_setup(uint32_t *dst, int words, const SetupSelect &first, const SetupSelect &second, int workgroups)
{
    const auto *src = (const __attribute__((address_space(4))) uint32_t *)__builtin_amdgcn_kernarg_segment_ptr();
    const int gtid = (int)(blockIdx.x * blockDim.x + threadIdx.x), nthr = workgroups * (int)blockDim.x;
    for (int i = gtid; i < words; i += nthr)
        dst[i] = src[i];
    auto begin = [&](const SetupSelect &p) {
        for (int g = 0; g < p.n_states; ++g) {
            for (int i = gtid; i < 3 * kSelBins; i += nthr)
                (&p.st[g].hist[0][0])[i] = 0;
            if (gtid == 0 && p.n > 0) {
                select_begin(&p.st[g], p.n, p.q, p.q_is_f64);
                p.st[g].room = p.room;
            }
        }
    };
    begin(first);
    begin(second);
}
__global__ void __launch_bounds__(256)
    prune_setup_kernel(const Blob a, uint32_t *dst, int words, const SetupSelect first, const SetupSelect second)
{
    prune_setup(dst, words, first, second, (int)gridDim.x);
}

// The same where every tile of every layer is one block of the sum whose rows are made of whole pieces of 16 bytes
// (queue_norms): the second item's rows are on their way while the first is added up (226 MB of BERT-base read past the
// caches: 37 us, 6.1 TB/s; four items 38, tile_row_norms_kernel 40; through the caches 43, 45 and 46).
// SETUP: the call's tables are in the arguments, and the first workgroups do on the side what prune_setup_kernel does, so that the call's
// first launch is the one that reads the scores (masks of twelve BERT-base feed-forward layers 119.6 -> 116.4 us; tables of more than kBlobWords
// words, and many selections to clear, keep the launch of their own).
constexpr int kNormItems = 2; // of a workgroup, in a row
struct NormTable { // on the device
    const PruneLayer *layers;
};
struct NormSetup {
    Blob a;
    uint32_t *dst;
    int32_t words, pad_;
    SetupSelect first, second;
};
constexpr int kNormSetupWgs = 16;
template <bool ONCE, bool SETUP>
__global__ void __launch_bounds__(256, 5)
    block_row_norms_kernel(const std::conditional_t<SETUP, NormSetup, NormTable> from, int n_layers, int64_t n_items, int64_t first_wg)
{
    __shared__ __align__(16) float stage[kNormRows * kNormPitch];
    const PruneLayer *layers;
    if constexpr (SETUP)
        layers = (const PruneLayer *)(uintptr_t)__builtin_amdgcn_kernarg_segment_ptr();
    else
        layers = from.layers;
    const LayerFinder find(&layers->rt_begin, sizeof(PruneLayer), n_layers);
    const int tid = (int)threadIdx.x, l8 = tid & 7, grp = tid >> 3, r0 = tid >> 5, q = tid & 31;
    struct Item {
        u32x4 v[4]; // the thread's pieces of rows r0 + 8 i
        TW_GLOBAL(float) out;
        int nr, w, divide;
    };
    auto fetch = [&](int64_t item, Item &d) {
        const PruneLayer L = load_entry(layers + find(item));
        const int K = L.K, N = L.N, G = L.granularity, n_tiles = L.n_tiles;
        const uint32_t idx = (uint32_t)(item - L.rt_begin); // (a call has fewer than 2^31 items)
        const int rblk = (int)(idx / (uint32_t)n_tiles), t = (int)(idx - (uint32_t)rblk * (uint32_t)n_tiles);
        const int k0 = rblk * kNormRows, c0 = t * G;
        d.nr = min(kNormRows, K - k0);
        d.w = min(G, N - c0);
        d.divide = !(L.flags & kNormNotDivided);
        d.out = as_global(L.norms) + (int64_t)t * K + k0;
        TW_GLOBAL(const float) const src = as_global(L.score) + (int64_t)k0 * N + c0 + min(q * 4, d.w - 4); // (pieces past the last repeat it)
#pragma unroll
        for (int i = 0; i < 4; ++i) // (so do rows)
            d.v[i] = load_global<ONCE>((TW_GLOBAL(const u32x4))(src + (int64_t)min(r0 + i * 8, d.nr - 1) * N));
    };
    auto add = [&](const Item &d) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<u32x4 *>(stage + (r0 + i * 8) * kNormPitch + q * 4) = d.v[i];
        TW_LDS_BARRIER();
        const float s = pairwise_block(stage + grp * kNormPitch, d.w, l8);
        if (l8 == 0 && grp < d.nr) // both operations correctly rounded
            d.out[grp] = d.divide ? sqrtf(s) / (float)d.w : sqrtf(s);
        TW_LDS_BARRIER(); // the stage is written again
    };
    const int64_t first = (first_wg + blockIdx.x) * kNormItems, last = n_items - 1;
    Item a, b;
    fetch(first, a);
    fetch(min(first + 1, last), b);
    add(a);
    if (first < last)
        add(b);
    if constexpr (SETUP) {
        if (first_wg == 0 && blockIdx.x < kNormSetupWgs)
            prune_setup(from.dst, from.words, from.first, from.second, min((int)gridDim.x, kNormSetupWgs));
    }
}

// mask[k][c] = (norm of row k in c's tile > threshold) and column c kept.  A unit of work is 16
// consecutive columns of four consecutive rows: one 16-byte store per row where the chunk is whole and
// aligned; a workgroup takes 1024 units of one layer, four per thread.  Where every chunk of the layer is whole
// and no tile narrower than one (but the last), a thread fetches what its four units need ahead of the
// threshold, which is 3 us of loads and barriers (57 MB of masks of twelve BERT-base feed-forward layers 16.6 -> 14.2 us, the
// 31 MB of VGG16 in tiles of kept columns 20.6 -> 12.7).
// The masks' addresses come with the launch, so that the caller can allocate them while the kernels before run (a
// network of more layers: in the table, at the start).
constexpr int kFillRows = 4, kFillUnits = 1024;
constexpr int kLateMasks = 128;
struct MaskTable {
    uint8_t *m[kLateMasks];
};
typedef float Norms4 __attribute__((ext_vector_type(4), aligned(4)));
__global__ void __launch_bounds__(256)
    fill_mask_kernel(const PruneLayer *layers, int n_layers, const SelectState *st, const Threshold *tile_thr, Mail *mail,
                     const MaskTable masks)
{
    const int layer = LayerFinder(&layers->el_begin, sizeof(PruneLayer), n_layers)(blockIdx.x);
    const PruneLayer L = layers[layer];
    TW_GLOBAL(uint8_t) const mask = as_global(n_layers <= kLateMasks ? masks.m[layer] : L.mask);
    const uint32_t cpr = (uint32_t)(L.N + 15) >> 4; // chunks per row
    const int64_t n_units = (int64_t)cpr * ((L.K + kFillRows - 1) / kFillRows);
    const int64_t first = (blockIdx.x - L.el_begin) * kFillUnits;
    TW_GLOBAL(const float) const norms = as_global((const float *)L.norms);
    TW_GLOBAL(const int32_t) const tcol0 = as_global((const int32_t *)L.tcol0);
    TW_GLOBAL(const uint8_t) const colkeep = as_global((const uint8_t *)L.colkeep);
    auto begin_of = [&](int t) { return tcol0 ? tcol0[t] : min(t * L.granularity, L.N); };
    // the tile of column c: start near where tiles of equal width would put it, then walk
    auto tile_of = [&](int c) {
        int t = tcol0 ? min(L.n_tiles - 1, (int)((float)c * (float)L.n_tiles / (float)L.N)) : c / L.granularity;
        if (tcol0) {
            while (tcol0[t] > c)
                --t;
            while (tcol0[t + 1] <= c)
                ++t;
        }
        return t;
    };
    // (a 32-bit division where the layer's units allow it: the 64-bit one is long)
    auto row_group = [&](int64_t unit) { return (unit >> 31) == 0 ? (int)((uint32_t)unit / cpr) : (int)(unit / cpr); };
    auto report = [&](const Threshold &t) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            mail->thr_rows = t.v64;
            if (t.lost)
                mail->lost = 1;
        }
    };
    constexpr int UNITS = kFillUnits / 256;
    if (!tile_thr && (L.N & 15) == 0 && L.granularity >= 16 && L.K >= kFillRows && (((uintptr_t)mask | (uintptr_t)L.colkeep) & 15) == 0) {
        // a chunk then lies in one tile or two; rows past the last are those before it once more (the same bytes)
        u32x4 cols[UNITS];
        Norms4 nv[UNITS][2];
        int cut[UNITS]; // columns of the chunk in the first of its tiles
        int64_t at[UNITS];
#pragma unroll
        for (int i = 0; i < UNITS; ++i) {
            const int64_t unit = min(first + i * 256 + (int64_t)threadIdx.x, n_units - 1);
            const int kg = row_group(unit);
            const int c0 = (int)(unit - (int64_t)kg * cpr) << 4, k0 = min(kg * kFillRows, L.K - kFillRows);
            const int t = tile_of(c0), end = begin_of(t + 1);
            cut[i] = min(end - c0, 16);
            at[i] = (int64_t)k0 * L.N + c0;
            const int64_t n0 = (int64_t)t * L.K + k0;
            nv[i][0] = *reinterpret_cast<TW_GLOBAL(const Norms4)>(norms + n0);
            nv[i][1] = *reinterpret_cast<TW_GLOBAL(const Norms4)>(norms + (cut[i] < 16 ? n0 + L.K : n0));
            cols[i] = colkeep ? *reinterpret_cast<TW_GLOBAL(const u32x4)>(colkeep + c0)
                              : u32x4{0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u};
        }
        const Threshold thr = threshold_of<256>(st);
        report(thr);
#pragma unroll
        for (int i = 0; i < UNITS; ++i) {
            if (first + i * 256 + (int64_t)threadIdx.x >= n_units)
                break;
            u32x4 one = cols[i], two = {0u, 0u, 0u, 0u}; // the kept columns of either tile
            if (cut[i] < 16) {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int n = min(max(cut[i] - w * 4, 0), 4);
                    two[w] = cols[i][w] & ~(uint32_t)((1ull << (n * 8)) - 1ull);
                    one[w] = cols[i][w] & ~two[w];
                }
            }
#pragma unroll
            for (int r = 0; r < kFillRows; ++r) {
                const uint32_t a = thr.passed_by(nv[i][0][r]) ? ~0u : 0u, b = thr.passed_by(nv[i][1][r]) ? ~0u : 0u;
                *(TW_GLOBAL(u32x4))(mask + at[i] + (int64_t)r * L.N) =
                    u32x4{(one.x & a) | (two.x & b), (one.y & a) | (two.y & b), (one.z & a) | (two.z & b), (one.w & a) | (two.w & b)};
            }
        }
        return;
    }
    const Threshold thr = tile_thr ? *tile_thr : threshold_of<256>(st); // (tile_thr: one per tile)
    report(thr);
#pragma unroll
    for (int i = 0; i < kFillUnits / 256; ++i) {
        const int64_t unit = first + i * 256 + threadIdx.x;
        if (unit >= n_units)
            break;
        const int kg = row_group(unit);
        const int c0 = (int)(unit - (int64_t)kg * cpr) << 4, n = min(16, L.N - c0), k0 = kg * kFillRows;
        uint32_t cols[4]; // the chunk's columns: a byte of 1 where kept
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            cols[w] = 0x01010101u;
            if (colkeep) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (!colkeep[min(c0 + w * 4 + e, L.N - 1)])
                        cols[w] &= ~(1u << (e * 8));
            }
        }
        int t = tile_of(c0);
        uint32_t out[kFillRows][4];
#pragma unroll
        for (int r = 0; r < kFillRows; ++r)
            out[r][0] = out[r][1] = out[r][2] = out[r][3] = 0u;
        for (int cb = c0; cb < c0 + n; ++t) { // the tiles the chunk touches: one, or a few
            const int ce = min(begin_of(t + 1), c0 + n);
            const Threshold tt = tile_thr ? tile_thr[t] : thr;
            float nv[kFillRows];
#pragma unroll
            for (int r = 0; r < kFillRows; ++r)
                nv[r] = norms[(int64_t)t * L.K + min(k0 + r, L.K - 1)];
            uint32_t in_tile[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int lo = min(max(cb - c0 - w * 4, 0), 4), hi = min(max(ce - c0 - w * 4, 0), 4);
                in_tile[w] = cols[w] & (uint32_t)((1ull << (hi * 8)) - 1ull) & ~(uint32_t)((1ull << (lo * 8)) - 1ull);
            }
#pragma unroll
            for (int r = 0; r < kFillRows; ++r) {
                const bool keep = tt.passed_by(nv[r]);
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    out[r][w] |= keep ? in_tile[w] : 0u;
            }
            cb = ce;
        }
#pragma unroll
        for (int r = 0; r < kFillRows; ++r) {
            if (k0 + r >= L.K)
                break;
            TW_GLOBAL(uint8_t) const dst = mask + (int64_t)(k0 + r) * L.N + c0;
            if (n == 16 && (((uintptr_t)dst) & 15) == 0) {
                *(TW_GLOBAL(u32x4))dst = u32x4{out[r][0], out[r][1], out[r][2], out[r][3]};
            } else {
                for (int e = 0; e < n; ++e)
                    dst[e] = (uint8_t)(out[r][e >> 2] >> ((e & 3) * 8));
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// mixed masks: a TW mask plus the largest remaining single elements

struct MixLayer {
    const float *score;
    const uint8_t *mask0; // the TW mask of the layer, or nullptr: an element is kept where the norm of its row of its tile passes
    const float *norms;   // [tiles][K]
    uint8_t *out;         // may be mask0 itself
    int64_t n;            // elements of the layer
    int64_t begin;        // its first element among all layers'
    int64_t item_begin;   // its first item in the launch-wide numbering
    double per_n;         // 1 / N
    float per_nf, per_g;  // 1 / N, 1 / G
    int32_t K, N, G;      // G: columns of a tile
    int32_t rows_on, cols_on; // 1024 / N, 1024 % N
    int32_t in_fours;     // whole items are worked off as vectors: score, masks and output are aligned alike, and (norms) no tile is
                          // narrower than three columns, so that four neighbours lie in two tiles or rows at most;
                          // 2: in one, rows and tiles being made of fours
};

// Where the mask bytes of the elements come from: the caller's masks; the norms of the tiles' rows and
// their threshold, for masks that nobody has written yet; a bit each that the narrowing pass has left.
// MIX_SPLIT: norms where four elements that are worked off together can lie in two tiles or rows (a kernel of its own, since a load on a
// condition is waited for on the spot).
enum MixSource { MIX_BYTES, MIX_NORMS, MIX_SPLIT, MIX_BITS };

// ||x|| of a single element (sqrt(x*x) / 1, the reference's norm over a tile of one column) minus 1
// where the TW mask already keeps it (prune_algo.py:159-161).  The square root of a rounded square
// is |x| again as long as the square is a normal number (or zero).
constexpr float kMixPlainMin = 1e-18f, kMixPlainMax = 1e18f;
__device__ __forceinline__ bool mix_plain(float ax) { return (ax >= kMixPlainMin && ax <= kMixPlainMax) || ax == 0.0f; }
__device__ __forceinline__ float mix_value(float x, uint32_t m0)
{
    float nrm = fabsf(x);
    if (!mix_plain(nrm)) {
        const float sq = x * x;
        nrm = sqrtf(sq);
    }
    return m0 ? nrm - 1.0f : nrm;
}

// The kernels of the mixed producer walk items of 4096 consecutive elements of a layer, sixteen per
// thread, as vectors where the layer allows it.  The element scores are worked
// out anew from weight and mask wherever they are needed rather than written to a pool and read back.  At
// four or five bytes an element the vector instructions count as much as the memory: ten per element
// are 8 us for 31.5 M elements.
constexpr int kMixItem = 4096;
struct MixFetched {
    TW_GLOBAL(const float) sc;
    TW_GLOBAL(const uint8_t) mk;
    uint8_t *out;
    int n;
    bool vec;
    float4 x[4];
    uint32_t m[4];   // mask bytes, any value but 0 counting as 1 (MIX_SPLIT: how many of the four have the first norm)
    float nv[4][2];  // MIX_NORMS: the norm of four elements; MIX_SPLIT: of the first and of the last
    uint32_t bits;   // MIX_BITS: the thread's sixteen elements
    const MixLayer *layer;
    int64_t e0;      // the item's first element
};
__device__ __forceinline__ bool mix_in_vectors(const MixLayer &L, int64_t e0) { return L.in_fours && L.n - e0 >= kMixItem; }
// Layers whose elements are placed in rows and tiles with a multiplication in float: (x + 0.5) / N is off by less than
// 0.5 / N for x below 2^22, and a product of two numbers below 2^24 is a full-rate instruction.
constexpr int kMixMaxN = 1 << 21, kMixMaxK = 1 << 23;
constexpr int64_t kMixMaxNorms = 1 << 29;
struct MixCell {
    uint32_t k, c; // row (from the layer's first), column
    __device__ MixCell(const MixLayer &L, int64_t e0, uint32_t more) // element e0 + more
    {
        uint32_t k0 = (uint32_t)((double)e0 * L.per_n); // e0 / N, or one off
        int32_t r0 = (int32_t)(e0 - (int64_t)k0 * L.N);
        if (r0 < 0) {
            --k0;
            r0 += L.N;
        } else if (r0 >= L.N) {
            ++k0;
            r0 -= L.N;
        }
        const uint32_t x = (uint32_t)r0 + more;
        const uint32_t q = (uint32_t)(((float)x + 0.5f) * L.per_nf);
        k = k0 + q;
        c = x - __umul24(q, (uint32_t)L.N);
    }
    __device__ void on_1024(const MixLayer &L)
    {
        k += L.rows_on;
        c += L.cols_on;
        if (c >= (uint32_t)L.N) {
            c -= L.N;
            ++k;
        }
    }
    __device__ uint32_t tile(const MixLayer &L) const { return (uint32_t)(((float)c + 0.5f) * L.per_g); }
    __device__ uint32_t norm(const MixLayer &L, uint32_t t) const { return __umul24(t, (uint32_t)L.K) + k; }
};
template <int SRC>
__device__ __forceinline__ void mix_fetch(const MixLayer *layer, int64_t item, const uint16_t *bits, const float *safe, MixFetched &d)
{
    const MixLayer L = load_entry(layer);
    const int64_t e0 = (item - L.item_begin) * kMixItem;
    d.n = (int)min((int64_t)kMixItem, L.n - e0);
    d.sc = as_global(L.score) + e0;
    d.mk = as_global(L.mask0) + e0;
    d.out = L.out + e0;
    d.vec = mix_in_vectors(L, e0);
    // (an item that cannot be loaded in vectors loads something else in its place: with no load on a
    // condition the waits for them are exact counts)
    TW_GLOBAL(const u32x4) const x = d.vec ? (TW_GLOBAL(const u32x4))d.sc : (TW_GLOBAL(const u32x4))safe;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        d.x[i] = __builtin_bit_cast(float4, x[threadIdx.x + i * 256]);
    if constexpr (SRC == MIX_BYTES) {
        TW_GLOBAL(const uint32_t) const m = d.vec ? (TW_GLOBAL(const uint32_t))d.mk : (TW_GLOBAL(const uint32_t))safe;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            d.m[i] = m[threadIdx.x + i * 256];
    } else if constexpr (SRC == MIX_BITS) {
        d.bits = as_global(bits)[item * 256 + threadIdx.x];
    } else {
        d.layer = layer;
        d.e0 = e0;
        TW_GLOBAL(const float) const nm = as_global(L.norms);
        MixCell p(L, e0, d.vec ? threadIdx.x * 4 : 0u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t t = p.tile(L), at = d.vec ? p.norm(L, t) : 0u; // (no branch: any norm will do)
            d.nv[i][0] = nm[at];
            if constexpr (SRC == MIX_SPLIT) {
                const uint32_t end = min((t + 1) * (uint32_t)L.G, (uint32_t)L.N); // of the tile
                d.m[i] = min(end - p.c, 4u);
                d.nv[i][1] = nm[d.vec && d.m[i] < 4 ? (end == (uint32_t)L.N ? p.k + 1 : at + L.K) : at];
            }
            p.on_1024(L);
        }
    }
}
// MIX_BITS: f(values, mask bytes, output, count) per four (or single) elements
template <class F> __device__ __forceinline__ void mix_apply(const MixFetched &d, F f)
{
    if (d.vec) {
        float ax[4][4];
        // largest and (zeros aside: 0 - 1 wraps) smallest of the sixteen, by the bits of |x|, where a NaN is
        // larger than every number
        uint32_t hi = 0u, lo_less_1 = 0xFFFFFFFFu;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            ax[i][0] = fabsf(d.x[i].x);
            ax[i][1] = fabsf(d.x[i].y);
            ax[i][2] = fabsf(d.x[i].z);
            ax[i][3] = fabsf(d.x[i].w);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t bits = __float_as_uint(ax[i][e]);
                hi = max(hi, bits);
                lo_less_1 = min(lo_less_1, bits - 1u);
            }
        }
        // mix_plain for all sixteen
        if (hi > __float_as_uint(kMixPlainMax) || lo_less_1 < __float_as_uint(kMixPlainMin) - 1u) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    ax[i][e] = mix_value(ax[i][e], 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float v[4];
            const uint32_t m = ((d.bits >> (i * 4) & 15u) * 0x204081u) & 0x01010101u;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] = ax[i][e] - (float)(m >> (e * 8) & 255u);
            f(v, m, d.out + (threadIdx.x + i * 256) * 4, 4);
        }
    } else {
        for (int i = (int)threadIdx.x, slot = 0; i < d.n; i += 256, ++slot) {
            const uint32_t m0 = d.bits >> slot & 1u;
            const float v[4] = {mix_value(d.sc[i], m0), 0.0f, 0.0f, 0.0f};
            f(v, m0, d.out + i, 1);
        }
    }
}
// an element's place in its item, from its wave and the ten bits that `place` and the element's number among the four
// (times 64) and its lane make
__device__ __forceinline__ int mix_place(bool vec, int wave, uint32_t code)
{
    const int thread = wave * 64 + (int)(code & 63u);
    return vec ? (thread + (int)(code >> 8 & 3u) * 256) * 4 + (int)(code >> 6 & 3u) : (int)(code >> 6 & 15u) * 256 + thread;
}
// All items of a launch, shared out over its workgroups, the next item's loads in flight while one is
// worked on: work(item, what was fetched for it).
// bits: MIX_BITS; safe: 16 KB of device memory that can be read; fetched(): once, after the first loads.
template <int SRC, class R, class F>
__device__ __forceinline__ void mix_for_each(const MixLayer *layers, int n_layers, int64_t n_items, const uint16_t *bits, const float *safe,
                                             R fetched, F work)
{
    const LayerFinder find(&layers->item_begin, sizeof(MixLayer), n_layers);
    MixFetched a, b;
    const int64_t step = gridDim.x, last = n_items - 1;
    int64_t item = blockIdx.x; // (a launch has at most n_items workgroups)
    mix_fetch<SRC>(layers + find(item), item, bits, safe, a);
    fetched();
    for (;;) {
        const int64_t i1 = min(item + step, last), i2 = min(item + 2 * step, last);
        mix_fetch<SRC>(layers + find(i1), i1, bits, safe, b);
        work(item, a);
        if (item + step > last)
            break;
        mix_fetch<SRC>(layers + find(i2), i2, bits, safe, a);
        work(item + step, b);
        item += 2 * step;
        if (item > last)
            break;
    }
}

// The selection over the element scores.  Three passes with a histogram over all elements cost three
// reads of everything and, most elements sharing a few dozen digits, as many conflicts in LDS (60, 90
// and 67 us over the 31.5 M elements of VGG16).  So the wanted value is bracketed first: 8192 elements
// drawn evenly (one at a random place of every stretch) give two keys between which it lies but for
// one case in a million, one pass over the elements counts what is below and keeps aside what is
// between (2 - 3 % of the elements), and the three passes run over what was kept.
// Where the bracket missed or does not fit - the counts tell, for certain - they run over the
// elements.  The narrowing pass also writes the masks: what lies outside the bracket is decided
// already, and the few per cent inside are marked one by one when the threshold is known, from the places kept
// beside their values.
// Over the elements of VGG16, masks out of norms: sample, bracket, narrowing, passes, marking 5 + 8 + 30 + 23 + 9 us; with those masks
// written and read and the elements read once more at the end 13 + 4 + 11 + 31 + 31 + 32, and the host's wait between the stages.
constexpr int kMixSamples = 8192;
constexpr int64_t kMixSampleFrom = 1 << 17; // fewer elements than this are all kept aside
template <int SRC>
__global__ void __launch_bounds__(256)
    mix_sample_kernel(const MixLayer *layers, int n_layers, int64_t total, const SelectState *st_rows, SelectState *st, uint32_t *sample, Mail *mail)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x); // kMixSamples threads
    const int64_t at = total / kMixSamples * i;
    uint32_t h = (uint32_t)i * 0x9E3779B9u;
    h = (h ^ (h >> 16)) * 0x85EBCA6Bu;
    h ^= h >> 13;
    const int64_t e = at + (int64_t)(h % (uint32_t)min(total / kMixSamples, (int64_t)0x7FFFFFFF));
    int lo = 0, hi = n_layers;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (layers[mid].begin <= e)
            lo = mid;
        else
            hi = mid;
    }
    const MixLayer &L = layers[lo];
    const int64_t j = e - L.begin;
    const float x = as_global(L.score)[j];
    uint32_t m0;
    if constexpr (SRC == MIX_NORMS) {
        int64_t k = (int64_t)((double)j * L.per_n);
        if (k * L.N > j)
            --k;
        else if ((k + 1) * L.N <= j)
            ++k;
        const float norm = as_global(L.norms)[(int64_t)((int)(j - k * L.N) / L.G) * L.K + k];
        const Threshold t = threshold_of<256>(st_rows);
        const float rows = t.in_float();
        m0 = norm > rows ? 1u : 0u;
        if (i == 0) {
            st->row_norm = rows;
            if (t.lost)
                mail->lost = 1;
        }
    } else {
        m0 = L.mask0[j];
    }
    sample[i] = sort_key(mix_value(x, m0));
}

// The bracket out of the sample, one workgroup: the sample's values five standard deviations of their
// rank to either side of the wanted one, widened to 22 bits of the sample's range.
constexpr int kBracketThreads = 1024;
__global__ void __launch_bounds__(kBracketThreads) mix_bracket_kernel(const uint32_t *sample, SelectState *st)
{
    constexpr int PER = kMixSamples / kBracketThreads;
    __shared__ unsigned int s_h[kSelBins];
    const int tid = (int)threadIdx.x;
    uint32_t key[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i)
        key[i] = sample[tid + i * kBracketThreads];
    const double f = (double)st->head.rank0 / (double)st->head.n;
    const double mid = f * kMixSamples, dev = 5.0 * sqrt((double)kMixSamples * f * (1.0 - f)) + 2.0;
    const double want[2] = {mid - dev, mid + dev};
    const KeyRange range = key_range_in_block([&](auto f) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
            f(key[i]);
    });
    // both edges out of one count of the first digit and one of the second, with counters for each: an edge is a chain of trips
    // through LDS and barriers, which is all that this kernel waits for (one edge after the other: 14.6 us, so 11, and 8 with the steps over a wave's lanes in registers)
    __shared__ unsigned int s_h2[kSelBins];
    bool inside[2];
    uint32_t prefix[2], edge[2];
    unsigned long long rank[2];
    for (int i = tid; i < kSelBins; i += kBracketThreads)
        s_h[i] = s_h2[i] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i)
        atomicAdd(&s_h[range.digit(0, key[i] - range.base)], 1u);
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        inside[w] = want[w] >= 0.0 && want[w] < (double)kMixSamples; // workgroup-uniform
        const Digit d = find_digit<kBracketThreads, kSelBins>(s_h, inside[w] ? (unsigned long long)want[w] : 0ull);
        prefix[w] = d.digit;
        rank[w] = d.rest;
    }
    for (int i = tid; i < kSelBins; i += kBracketThreads)
        s_h[i] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const uint32_t k = key[i] - range.base, lead = k >> range.lead_shift(1);
        if (lead == prefix[0])
            atomicAdd(&s_h[range.digit(1, k)], 1u);
        if (lead == prefix[1])
            atomicAdd(&s_h2[range.digit(1, k)], 1u);
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const Digit d = find_digit<kBracketThreads, kSelBins>(w ? s_h2 : s_h, rank[w]);
        const uint32_t both = prefix[w] << (range.lead_shift(1) - range.shift[1]) | d.digit;
        const unsigned long long at = ((unsigned long long)both + w) << range.shift[1];
        edge[w] = inside[w] ? (uint32_t)min((unsigned long long)range.base + at - w, 0xFFFFFFFFull) : w ? 0xFFFFFFFFu : 0u;
    }
    const float lo = edge[0] == 0u ? -INFINITY : key_to_float(edge[0]);
    const float hi = edge[1] == 0xFFFFFFFFu ? INFINITY : key_to_float(edge[1]);
    if (tid == 0) {
        st->lo = lo;
        st->hi = hi;
    }
    // (a score grows with |x|: which |x| are inside is one range for elements without a mask byte and one for those with.  A wave looks for
    // one end of one of them, 64 places at a time)
    const int wave = tid >> 6, lane = tid & 63;
    if (wave < 4) {
        const uint32_t m0 = wave & 1;
        auto from = [&](uint32_t u) {
            const float v = mix_value(__uint_as_float(u), m0);
            return u >= kNanFrom || !(wave >> 1 ? v <= hi : v < lo);
        };
        uint32_t first = 0;
#pragma unroll 1
        for (int s = 25; s >= 1; s -= 6)
            first += (uint32_t)__popcll(__ballot(!from(first + ((uint32_t)(lane + 1) << s) - 1u))) << s;
        first += (uint32_t)__popcll(__ballot(lane < 2 && !from(first + lane)));
        if (lane == 0)
            st->cut[m0][wave >> 1] = first;
    }
}

// Below, between, above.  Every wave of the launch keeps the values between, and where they are, in a piece
// of the candidates of its own and leaves its counts beside it: nothing is added up with atomics, of which the
// memory takes one in 15 ns on one address (a counter per workgroup that all add to was 25 us of this
// kernel, one per wave 90).  The masks leave with it, as if nothing between were above the threshold; and a bit for
// each element's mask0, which nobody can read any more where the masks are written in place, should the
// bracket have missed.
// The 31.5 M elements of VGG16 with masks out of norms 39 -> 30 us: reading them takes 22 (5.7 TB/s), the norms of their rows 2, the masks 3
// and the candidates 3 (and the norms' threshold 3 more where no sample's kernel has left it); before, every item waited for the next one's loads (its layer's entry
// and conditional loads of norms behind them), and 29 vector instructions an element were 24 us of every SIMD's time (17 now).
constexpr int kMixWgs = 1024, kMixWaves = kMixWgs * 4; // most workgroups and waves of a pass over the elements
struct MixCounts {
    uint32_t between, below;
};
template <int SRC>
__global__ void __launch_bounds__(256, 4)
    mix_narrow_kernel(const MixLayer *layers, int n_layers, int64_t n_items, const SelectState *st_rows, const SelectState *st, u32x2 *cand,
                      MixCounts *counts, uint16_t *bits, Mail *mail, int sampled)
{
    const float lo = st->lo, hi = st->hi;
    const uint32_t in0 = st->cut[0][0], up0 = st->cut[0][1], in1 = st->cut[1][0], up1 = st->cut[1][1];
    const uint32_t room = st->room;
    const int lane = (int)(threadIdx.x & 63);
    const int w = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    TW_GLOBAL(u32x2) const keep = as_global(cand) + (int64_t)w * room;
    __shared__ __align__(16) float s_v[kMixItem];
    constexpr uint32_t kFrom = 0x22000000u, kTo = 0x5D000000u; // 2^-59 and 2^59, as bits
    const bool plain = min(in0, in1) >= kFrom && max(up0, up1) <= kTo; // every candidate is: see mix_plain
    static_assert(kMixPlainMin < 0x1p-59f && kMixPlainMax > 0x1p59f, "within mix_plain's");
    uint32_t kept = 0, round = 0;            // wave-uniform
    uint32_t below = 0;                      // of the lane's elements
    uint32_t mine = 0, inside = 0;           // mask0 of the thread's sixteen elements of the item; which are candidates
    float rows = 0.0f;
    auto rows_of = [&]() {
        if constexpr (SRC != MIX_BYTES) {
            if (sampled) {
                rows = st->row_norm;
            } else {
                const Threshold t = threshold_of<256>(st_rows);
                if (blockIdx.x == 0 && threadIdx.x == 0 && t.lost)
                    mail->lost = 1;
                rows = t.in_float();
            }
        }
    };
    // Sixteen elements of a thread: |x|, as whole numbers, against the two ends of the bracket for an element of its kind.  A bit of
    // two registers for each, the last element first, and everything else out of those.
    auto narrow = [&](const MixFetched &d) {
        if (d.vec) {
            uint32_t mask[4], under_in = 0, under_up = 0, top = 0;
            mine = 0;
            auto test = [&](float x, uint32_t in, uint32_t up) { // (all three below 2^31: the difference's sign)
                const uint32_t u = __float_as_uint(x) & 0x7FFFFFFFu;
                under_in = __builtin_amdgcn_alignbit(under_in, u - in, 31);
                under_up = __builtin_amdgcn_alignbit(under_up, u - up, 31);
                top = max(top, u);
            };
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<float4 *>(s_v + (i * 256 + (int)threadIdx.x) * 4) = d.x[i];
            if constexpr (SRC == MIX_NORMS) { // four elements of one kind
#pragma unroll
                for (int i = 3; i >= 0; --i) {
                    const bool row = d.nv[i][0] > rows;
                    const uint32_t in = row ? in1 : in0, up = row ? up1 : up0;
                    mask[i] = row ? 0x01010101u : 0u;
                    mine = mine << 4 | (row ? 15u : 0u);
                    test(d.x[i].w, in, up);
                    test(d.x[i].z, in, up);
                    test(d.x[i].y, in, up);
                    test(d.x[i].x, in, up);
                }
            } else {
#pragma unroll
                for (int i = 3; i >= 0; --i) {
                    uint32_t m;
                    if constexpr (SRC == MIX_SPLIT) {
                        const uint32_t first = (uint32_t)((1ull << (d.m[i] * 8)) - 1ull); // bytes of the first tile
                        m = (d.nv[i][0] > rows ? first & 0x01010101u : 0u) | (d.nv[i][1] > rows ? ~first & 0x01010101u : 0u);
                    } else {
                        m = ((d.m[i] & 0x7F7F7F7Fu) + 0x7F7F7F7Fu | d.m[i]) >> 7 & 0x01010101u; // mask bytes that are not 0
                    }
                    mask[i] = m;
                    mine = mine << 4 | m * 0x10204080u >> 28;
                    const float x[4] = {d.x[i].x, d.x[i].y, d.x[i].z, d.x[i].w};
#pragma unroll
                    for (int e = 3; e >= 0; --e) {
                        const bool one = m >> (e * 8) & 1u;
                        test(x[e], one ? in1 : in0, one ? up1 : up0);
                    }
                }
            }
            below += (uint32_t)__popc(under_in);
            inside = under_up & ~under_in;
            uint32_t above = ~under_up;
            if (top >= kNanFrom) { // (what is no number is neither below nor inside nor above)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float x[4] = {d.x[i].x, d.x[i].y, d.x[i].z, d.x[i].w};
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        above &= ~((x[e] != x[e] ? 1u : 0u) << (i * 4 + e));
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *(TW_GLOBAL(uint32_t))(d.out + (threadIdx.x + i * 256) * 4) = mask[i] | __umul24(above >> (i * 4) & 15u, 0x204081u) & 0x01010101u;
        } else {
            mine = inside = 0;
            for (int i = (int)threadIdx.x, slot = 0; i < d.n; i += 256, ++slot) {
                uint32_t m0;
                if constexpr (SRC != MIX_BYTES) {
                    const MixCell p(*d.layer, d.e0, (uint32_t)i);
                    m0 = as_global(d.layer->norms)[p.norm(*d.layer, p.tile(*d.layer))] > rows ? 1u : 0u;
                } else {
                    m0 = d.mk[i] ? 1u : 0u;
                }
                const float x = d.sc[i], v = mix_value(x, m0);
                s_v[((slot >> 2) * 256 + (int)threadIdx.x) * 4 + (slot & 3)] = x;
                below += v < lo ? 1u : 0u;
                inside |= (v >= lo && v <= hi ? 1u : 0u) << slot;
                mine |= m0 << slot;
                as_global(d.out)[i] = m0 || v > hi ? 1 : 0;
            }
        }
    };
    // The candidates of an item, one of every lane that has one left at a time: a lane has half of one among its
    // sixteen elements, so that three or four rounds do for sixteen tests and as many stores (4 us less than a test behind each of
    // VGG16's 31.5 M elements).
    auto work = [&](int64_t item, const MixFetched &d) {
        narrow(d);
        for (;;) {
            const bool some = inside != 0;
            const unsigned long long in = __ballot(some);
            if (!in)
                break;
            const uint32_t slot = some ? (uint32_t)__builtin_ctz(inside) : 0u;
            const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(in >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)in, kept));
            if (some && at < room) { // (the count tells of an overflow)
                const float x = s_v[((slot >> 2) * 256 + threadIdx.x) * 4 + (slot & 3)];
                const uint32_t one = mine >> slot & 1u;
                const float v = plain ? fabsf(x) - (float)one : mix_value(x, one);
                keep[at] = u32x2{__float_as_uint(v), round << 10 | slot << 6 | (uint32_t)lane};
            }
            kept += __popcll(in);
            inside &= inside - 1;
        }
        as_global(bits)[item * 256 + threadIdx.x] = (uint16_t)mine;
        ++round;
    };
    mix_for_each<SRC>(layers, n_layers, n_items, nullptr, reinterpret_cast<const float *>(cand), rows_of, work);
    below = last_lane(wave_scan(below));
    if (lane == 0)
        counts[w] = MixCounts{kept, below};
}

// the counts of all waves of the narrowing pass added up, and whether every piece held its values; called by all 256
// threads of a workgroup
__device__ bool mix_totals(const MixCounts *counts, int waves, uint32_t room, unsigned long long &between, unsigned long long &below)
{
    __shared__ unsigned long long s_sum[2];
    __shared__ uint32_t s_most;
    if (threadIdx.x == 0) {
        s_sum[0] = s_sum[1] = 0;
        s_most = 0;
    }
    __syncthreads();
    unsigned long long a = 0, b = 0;
    uint32_t most = 0;
#pragma unroll
    for (int i = 0; i < kMixWaves / 256; ++i) {
        const int w = (int)threadIdx.x + i * 256;
        const MixCounts c = counts[min(w, waves - 1)];
        a += w < waves ? c.between : 0u;
        b += w < waves ? c.below : 0u;
        most = max(most, c.between);
    }
    a = wave_scan(a);
    b = wave_scan(b);
    most = wave_max(most);
    if ((threadIdx.x & 63) == 63) {
        atomicAdd(&s_sum[0], a);
        atomicAdd(&s_sum[1], b);
        atomicMax(&s_most, most);
    }
    __syncthreads();
    between = s_sum[0];
    below = s_sum[1];
    return s_most <= room;
}

constexpr int kMixHistWgs = 96; // workgroups that count what was kept (each adds up to 2048 counters to the others')
// A piece holds some two hundred values, and one piece after the other, each behind the load of its count, was eleven pairs of trips to memory.
// (What is left of a pass are the counts of all waves, the digits so far and the counters' atomics: with 48 workgroups 12 + 15 + 15 us,
// 96 11 + 10 + 11, and 5 for the third where two digits hold the bracket's range, 192 10 + 10 + 10, 256 12 + 10 + 10;
// with 96 and the first pieces on their way while those are looked at 9.5 + 9.)
constexpr int kMixPieces = 4; // at a time
static_assert(kMixWaves <= 64 * 4 * kMixHistWgs, "a lane for each piece of a wave");
template <int PASS>
__global__ void __launch_bounds__(256)
    mix_hist_kernel(const MixLayer *layers, int n_layers, int64_t n_items, SelectState *st, const u32x2 *cand,
                    const MixCounts *counts, int waves, const uint16_t *bits)
{
    if (PASS == 2 && st->key_bits <= 22)
        return; // (two digits hold all of the range)
    __shared__ unsigned int s_h[kSelBins];
    __shared__ uint32_t s_min;
    uint32_t prefix, mn = 0xFFFFFFFFu;
    unsigned long long rank;
    const unsigned long long want = st->head.rank0;
    const uint32_t room = st->room;
    // this wave's pieces (at most 64, see below): w0, w0 + per, ..; lane l has the count of number l
    const int per = min((int)gridDim.x, kMixHistWgs) * 4, w0 = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
    const int mine = w0 < min(per, waves) ? (waves - w0 + per - 1) / per : 0;
    const uint32_t held = lane < mine ? counts[w0 + lane * per].between : 0u;
    // Four pieces at a time, sixteen loads in flight; the first of them ahead of the counts of all waves and the digits so far
    TW_GLOBAL(const u32x2) v[kMixPieces];
    uint32_t n[kMixPieces];
    float x[kMixPieces][4];
    auto fetch = [&](int q0) {
#pragma unroll
        for (int q = 0; q < kMixPieces; ++q) {
            n[q] = q0 + q < mine ? (uint32_t)__builtin_amdgcn_readlane((int)held, q0 + q) : 0u;
            v[q] = as_global(cand) + (int64_t)(mine ? w0 + min(q0 + q, mine - 1) * per : 0) * room;
#pragma unroll
            for (int e = 0; e < 4; ++e) // (a piece that did not hold all of its values is not looked at)
                x[q][e] = __uint_as_float(v[q][min((uint32_t)(lane + e * 64), min(max(n[q], 1u), room) - 1u)].x);
        }
    };
    if (blockIdx.x < kMixHistWgs)
        fetch(0);
    unsigned long long n_cand, below;
    bool narrowed;
    if (PASS == 0) {
        const bool whole = mix_totals(counts, waves, room, n_cand, below);
        // the wanted value and the one above it lie inside the bracket, and all of that was kept
        narrowed = whole && below <= want && (want - below) + 1 < n_cand;
    } else {
        below = st->below;
        narrowed = st->narrowed != 0;
    }
    if (narrowed && blockIdx.x >= kMixHistWgs)
        return;
    // (-0 and +0 are one value to the comparisons with the bracket, and two keys)
    const uint32_t lo = narrowed ? sort_key(st->lo == 0.0f ? -0.0f : st->lo) : 0u;
    const uint32_t span = narrowed ? sort_key(st->hi == 0.0f ? 0.0f : st->hi) - lo : 0xFFFFFFFFu;
    const int key_bits = span ? 32 - __clz(span) : 1;
    const KeyRange range(lo, key_bits);
    select_enter<PASS, 256>(st, range, s_h, &s_min, narrowed ? want - below : want, prefix, rank);
    if (PASS == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
        st->key_base = lo;
        st->key_bits = key_bits;
        st->below = below;
        st->narrowed = narrowed;
    }
    if (narrowed) {
        for (int q0 = 0; q0 < mine; q0 += kMixPieces) {
            if (q0)
                fetch(q0);
#pragma unroll
            for (int q = 0; q < kMixPieces; ++q) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if ((uint32_t)(lane + e * 64) < n[q])
                        select_count<PASS>(sort_key(x[q][e]), range, prefix, s_h, mn);
                for (uint32_t i = 256 + lane; i < n[q]; i += 256) { // (the rest of a long one)
                    float y[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        y[e] = __uint_as_float(v[q][min(i + e * 64, n[q] - 1)].x);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (i + e * 64 < n[q])
                            select_count<PASS>(sort_key(y[e]), range, prefix, s_h, mn);
                }
            }
        }
    } else {
        auto count = [&](const float (&v)[4], uint32_t, uint8_t *, int cnt) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e < cnt)
                    select_count<PASS>(sort_key(v[e]), range, prefix, s_h, mn);
        };
        mix_for_each<MIX_BITS>(layers, n_layers, n_items, bits, reinterpret_cast<const float *>(cand), []() {},
                               [&](int64_t, const MixFetched &d) { mix_apply(d, count); });
    }
    select_leave<PASS, 256>(st, s_h, &s_min, mn);
}

constexpr int kMarkLayers = 128;
// out = mask0 | (score > threshold)   (prune_algo.py:171-176): the candidates above the threshold, a wave for each
// piece of them; all elements where the selection ran over all
__global__ void __launch_bounds__(256)
    mix_mark_kernel(const MixLayer *layers, int n_layers, int64_t n_items, const SelectState *st, const u32x2 *cand,
                    const MixCounts *counts, const uint16_t *bits, Mail *mail)
{
    // what a candidate's place is worked out from, for the first kMarkLayers layers: a look-up is a few reads of LDS then,
    // instead of as many trips to memory
    __shared__ int64_t s_item[kMarkLayers], s_n[kMarkLayers];
    __shared__ uint8_t *s_out[kMarkLayers];
    __shared__ int s_fours[kMarkLayers];
    const int staged = min(n_layers, kMarkLayers);
    for (int l = (int)threadIdx.x; l < staged; l += 256) {
        s_item[l] = layers[l].item_begin;
        s_n[l] = layers[l].n;
        s_out[l] = layers[l].out;
        s_fours[l] = layers[l].in_fours;
    }
    const Threshold thr = threshold_of<256>(st);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        mail->thr_rows = thr.v64;
        if (thr.lost)
            mail->lost = 1;
    }
    if (st->narrowed) { // (the grid is the narrowing pass's)
        const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
        const int64_t w = (int64_t)blockIdx.x * 4 + wave;
        const uint32_t room = st->room, n = counts[w].between;
        TW_GLOBAL(const u32x2) const v = as_global(cand) + w * room;
        for (uint32_t i0 = 0; i0 < n; i0 += 256) {
            u32x2 c[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                c[e] = v[min(i0 + e * 64 + lane, n - 1)];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (i0 + e * 64 + lane >= n || !thr.passed_by(__uint_as_float(c[e].x)))
                    continue;
                const int64_t item = blockIdx.x + (int64_t)(c[e].y >> 10) * gridDim.x;
                int lo = 0, hi = staged;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (s_item[mid] <= item)
                        lo = mid;
                    else
                        hi = mid;
                }
                int64_t e0 = (item - s_item[lo]) * kMixItem, left = s_n[lo] - e0;
                uint8_t *out = s_out[lo];
                int fours = s_fours[lo];
                if (left <= 0) { // (beyond the staged layers)
                    hi = n_layers;
                    while (hi - lo > 1) {
                        const int mid = (lo + hi) >> 1;
                        if (layers[mid].item_begin <= item)
                            lo = mid;
                        else
                            hi = mid;
                    }
                    e0 = (item - layers[lo].item_begin) * kMixItem;
                    left = layers[lo].n - e0;
                    out = layers[lo].out;
                    fours = layers[lo].in_fours;
                }
                as_global(out)[e0 + mix_place(fours && left >= kMixItem, wave, c[e].y)] = 1;
            }
        }
        return;
    }
    auto mark = [&](const float (&v)[4], uint32_t m, uint8_t *out, int cnt) {
        if (cnt == 4) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                m |= thr.passed_by(v[e]) ? 1u << (e * 8) : 0u;
            *(TW_GLOBAL(uint32_t))out = m;
        } else {
            *as_global(out) = (m || thr.passed_by(v[0])) ? 1 : 0;
        }
    };
    mix_for_each<MIX_BITS>(layers, n_layers, n_items, bits, reinterpret_cast<const float *>(cand), []() {},
                           [&](int64_t, const MixFetched &d) { mix_apply(d, mark); });
}

// ---------------------------------------------------------------------------------
// host side

namespace {

// Temporaries of one producer call come from a device buffer that is kept and grows (until
// tw_release_memory gives it back), so that a steady stream of calls does not pay for hipMalloc / hipFree,
// and its thresholds come back through a page of pinned host memory that its last kernel writes.  A call holds
// both for its duration, and one that finds them held waits (producer calls are serialised) - but never for a
// call that is in its caller's `ready`: that code may itself wait for this call (a lock of an interpreter), make
// a producer call or give memory back.  The second set is for a call that comes by then.
struct Kept {
    void *ws = nullptr;
    size_t size = 0;
    int device = -1; // the device the buffer lives on; calls on another device do not use it
    Mail *mail = nullptr;
    bool held = false;
    bool away = false; // held by a call that is in its caller's `ready`
    bool drop = false; // given back by tw_release_memory while it was held: freed when the call ends

    void give_back()
    {
        if (ws && hipFree(ws) != hipSuccess)
            (void)hipGetLastError();
        ws = nullptr;
        size = 0;
        device = -1; // the device of the next call
    }
};
// (held for a look at `g_kept` only; neither is destroyed when the process ends, whose other threads may still wait)
std::mutex &g_kept_mutex = *new std::mutex;
std::condition_variable &g_kept_free = *new std::condition_variable;
Kept g_kept[2];

class Arena {
public:
    // `s`: the stream the call queues its kernels on; the buffer is not handed to the next call
    // before that stream has run dry, whichever way the call ends (an error return after kernels
    // were queued included).
    explicit Arena(hipStream_t s) : stream_(s)
    {
        if (hipGetDevice(&device_) != hipSuccess)
            device_ = -2;
        std::unique_lock<std::mutex> lock(g_kept_mutex);
        for (;;) {
            Kept *k = g_kept, *const end = std::end(g_kept);
            while (k != end && k->held && k->away)
                ++k;
            if (k == end) // (a producer in the `ready` of one in the `ready` of another: memory of its own)
                break;
            if (!k->held) {
                kept_ = k;
                break;
            }
            g_kept_free.wait(lock);
        }
        kept_->held = true;
        if (kept_->device < 0)
            kept_->device = device_;
        usable_ = device_ == kept_->device;
    }
    ~Arena()
    {
        if (!idle_)
            (void)hipStreamSynchronize(stream_);
        for (void *p : extras_)
            (void)hipFree(p);
        if (kept_ == &own_) {
            if (own_.mail)
                (void)hipHostFree(own_.mail);
            return;
        }
        std::unique_lock<std::mutex> lock(g_kept_mutex);
        if (!kept_->drop && usable_ && need_ > kept_->size) { // grow for the next call
            lock.unlock();
            (void)hipFree(kept_->ws);
            kept_->ws = nullptr;
            kept_->size = 0;
            const size_t want = need_ + need_ / 2;
            if (hipMalloc(&kept_->ws, want) == hipSuccess) {
                kept_->size = want;
            } else {
                (void)hipGetLastError();
                kept_->ws = nullptr;
            }
            lock.lock();
        }
        if (kept_->drop)
            kept_->give_back();
        kept_->held = kept_->drop = false;
        lock.unlock();
        g_kept_free.notify_all();
    }
    Arena(const Arena &) = delete;
    Arena &operator=(const Arena &) = delete;
    // while code of the caller's runs: nobody waits for this call
    class Away {
    public:
        explicit Away(Arena *a) : kept_(a ? a->kept_ : nullptr) { set(true); }
        ~Away() { set(false); }
        Away(const Away &) = delete;
        Away &operator=(const Away &) = delete;

    private:
        void set(bool away)
        {
            if (!kept_)
                return;
            {
                std::lock_guard<std::mutex> lock(g_kept_mutex);
                kept_->away = away;
            }
            if (away)
                g_kept_free.notify_all();
        }
        Kept *const kept_;
    };
    void *alloc(size_t bytes)
    {
        bytes = (bytes + 255) / 256 * 256;
        need_ += bytes;
        if (usable_ && off_ + bytes <= kept_->size) {
            void *p = static_cast<char *>(kept_->ws) + off_;
            off_ += bytes;
            return p;
        }
        void *p = nullptr;
        if (hipMalloc(&p, bytes) != hipSuccess) {
            (void)hipGetLastError(); // (or the next call's check of its launches would find it)
            return nullptr;
        }
        extras_.push_back(p);
        return p;
    }
    template <class T> T *alloc_n(size_t n) { return static_cast<T *>(alloc(sizeof(T) * std::max<size_t>(n, 1))); }
    // the pinned page for this call, or nullptr
    Mail *mail()
    {
        if (!kept_->mail && hipHostMalloc((void **)&kept_->mail, 4096, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            kept_->mail = nullptr;
        }
        mail_ = kept_->mail;
        if (mail_)
            mail_->lost = 0;
        return mail_;
    }
    // waits for the call's kernels; nothing may be queued behind this
    int wait()
    {
        TW_HIP(hipStreamSynchronize(stream_));
        idle_ = true;
        if (mail_ && mail_->lost)
            return fail(TW_ERR_DEVICE, "radix select lost its rank");
        return TW_OK;
    }

private:
    hipStream_t stream_;
    Kept own_, *kept_ = &own_;
    int device_ = -1;
    bool usable_ = false, idle_ = false;
    Mail *mail_ = nullptr;
    size_t off_ = 0, need_ = 0;
    std::vector<void *> extras_;
};

// `bytes` of a host table to the device through kernel arguments, and the selections cleared
int put_table(const void *table, size_t bytes, void *dst, SetupSelect first, SetupSelect second, hipStream_t s)
{
    size_t off = 0;
    do {
        Blob a;
        const size_t take = std::min(bytes - off, sizeof(a.w));
        std::memcpy(a.w, static_cast<const char *>(table) + off, take);
        hipLaunchKernelGGL(prune_setup_kernel, dim3(first.n_states > 4 ? 128 : 16), dim3(256), 0, s, a,
                           reinterpret_cast<uint32_t *>(static_cast<char *>(dst) + off), (int)((take + 3) / 4), first, second);
        first.n_states = second.n_states = 0; // (the selections once)
        off += take;
    } while (off < bytes);
    TW_HIP(hipGetLastError());
    return TW_OK;
}
SetupSelect setup_of(SelectState *st, int n_states, int64_t n, double q, int q_is_f64, uint32_t room = 0)
{
    return SetupSelect{st, n, q, n_states, q_is_f64, room, 0};
}

int check_percentile(int64_t n, double q)
{
    if (n <= 0)
        return fail(TW_ERR_SHAPE, "percentile of an empty set");
    if (!(q >= 0.0 && q <= 100.0))
        return fail(TW_ERR_SHAPE, "percentile %g is outside [0, 100]", q);
    return TW_OK;
}

// The three passes over `n` values (at most, where the state holds the exact number) in each of
// n_segments segments.  Two workgroups per compute unit at most: every workgroup starts by
// working out a digit from 16 KB of counters and ends with an atomic on every counter it has used.
int queue_select(const float *d_v, int64_t n, SelectState *st, int n_segments, hipStream_t s)
{
    const int grid = (int)std::min<int64_t>(n_segments > 1 ? 64 : 256, (n + 4095) / 4096);
    const dim3 g(std::max(1, grid), n_segments);
    hipLaunchKernelGGL(select_hist_kernel<0>, g, dim3(256), 0, s, d_v, st);
    hipLaunchKernelGGL(select_hist_kernel<1>, g, dim3(256), 0, s, d_v, st);
    hipLaunchKernelGGL(select_hist_kernel<2>, g, dim3(256), 0, s, d_v, st);
    TW_HIP(hipGetLastError());
    return TW_OK;
}

// The caller's masks: there from the start, or (`ready`) once that has been called, when the first kernels are queued.
struct Masks {
    uint8_t *const *m;
    tw_masks_ready ready = nullptr;
    void *user = nullptr;

    // asks for them and checks them; `ar`: what the call holds
    int get(int n_layers, Arena *ar)
    {
        if (ready) {
            const Arena::Away away(ar);
            if (ready(user))
                return fail(TW_ERR_ALLOC, "the caller has no masks");
        }
        ready = nullptr;
        for (int l = 0; l < n_layers; ++l)
            if (!m[l])
                return fail(TW_ERR_NULL, "layer %d: scores or mask pointer is NULL", l);
        return TW_OK;
    }
};

int check_layers(int n_layers, const int32_t *K, const int32_t *N, const float *const *scores,
                 const Masks &masks, int granularity)
{
    if (n_layers <= 0 || granularity <= 0)
        return fail(TW_ERR_SHAPE, "n_layers=%d granularity=%d must be positive", n_layers,
                    granularity);
    if (!K || !N || !scores || !masks.m)
        return fail(TW_ERR_NULL, "K, N, scores or masks is NULL");
    for (int l = 0; l < n_layers; ++l) {
        if (K[l] <= 0 || N[l] <= 0)
            return fail(TW_ERR_SHAPE, "layer %d: K=%d N=%d must be positive", l, K[l], N[l]);
        if (!scores[l] || (!masks.ready && !masks.m[l]))
            return fail(TW_ERR_NULL, "layer %d: scores or mask pointer is NULL", l);
    }
    return TW_OK;
}

// The table of a call whose tiles are every `granularity` columns, or (2-D) at most that many tiles, found on
// the device.
struct CallTable {
    std::vector<PruneLayer> layers;
    int64_t n_norms = 0, n_items = 0, n_fill = 0, n_tcol = 0, n_cols = 0; // sums over the layers (upper bounds)
};
// A launch of 2^32 threads or more reports no error and runs nothing: as many launches as that asks for.
// launch(first workgroup, workgroups)
template <class F> void in_launches(int64_t workgroups, int threads, F launch)
{
    const int64_t most = kMaxGridThreads / threads;
    for (int64_t first = 0; first < workgroups; first += most)
        launch(first, dim3((unsigned)std::min(most, workgroups - first)));
}

CallTable make_table(int n_layers, const int32_t *K, const int32_t *N, const float *const *scores, int granularity, int flags)
{
    CallTable c;
    c.layers.resize(n_layers);
    for (int l = 0; l < n_layers; ++l) {
        PruneLayer &e = c.layers[l];
        std::memset(&e, 0, sizeof(e));
        e.score = scores[l];
        e.K = K[l];
        e.N = N[l];
        e.granularity = granularity;
        e.n_tiles = (int32_t)(((int64_t)N[l] + granularity - 1) / granularity);
        e.flags = flags;
        e.rt_begin = c.n_items;
        e.el_begin = c.n_fill;
        e.col_begin = c.n_cols;
        c.n_norms += (int64_t)e.K * e.n_tiles;
        c.n_items += (int64_t)((e.K + kNormRows - 1) / kNormRows) * e.n_tiles;
        c.n_fill += (((int64_t)e.K + kFillRows - 1) / kFillRows * (((int64_t)e.N + 15) / 16) + kFillUnits - 1) / kFillUnits;
        c.n_tcol += e.n_tiles + 1;
        c.n_cols += e.N;
    }
    return c;
}

// The row norms of all layers' tiles; n_items: tiles of kept columns, *n_items items of them.  `last`: the call does not read the
// scores again.  Scores that go far beyond the memory-side cache (256 MB) are then read past it: most of them would not stay there for
// whoever comes next.  The line is where that next one, a build of the layers' plans out of the same matrices, no longer loses what the
// masks gain (BERT-base layers, us with the loads through the caches and past them, masks and plans): 283 MB 146 + 1265 and 133 + 1282, 321 MB
// 160 + 1433 and 143 + 1449, 340 MB 166 + 1520 and 148 + 1530, 377 MB 178 + 1705 and 158 + 1705.  Below it the plans lose more (226 MB 112 + 988 and
// 113 + 1022), though masks of scores that were written just before gain from 208 MB on (226 MB 144 and 129).
constexpr int64_t kStayingBytes = 320 << 20;
// Tables that are not on the device yet, the layers' first.
struct Tables {
    const void *host;
    size_t bytes;
    void *dev;
    SetupSelect first, second;
};
int queue_norms(const CallTable &c, const PruneLayer *d_table, const int64_t *n_items, bool last, hipStream_t s, const Tables *tables = nullptr)
{
    bool blocks = n_items == nullptr;
    int64_t bytes = 0;
    for (const PruneLayer &e : c.layers)
        bytes += (int64_t)e.K * e.N * 4;
    const bool once = last && bytes > kStayingBytes;
    for (const PruneLayer &e : c.layers)
        blocks &= (e.N & 3) == 0 && (e.granularity & 3) == 0 && e.granularity <= 128 && ((uintptr_t)e.score & 15) == 0;
    const int n_layers = (int)c.layers.size();
    if (blocks && tables && tables->bytes <= sizeof(Blob) && tables->first.n_states <= 4) { // (more of them want more workgroups to clear them)
        NormSetup u;
        std::memcpy(u.a.w, tables->host, tables->bytes);
        u.dst = static_cast<uint32_t *>(tables->dev);
        u.words = (int32_t)((tables->bytes + 3) / 4);
        u.pad_ = 0;
        u.first = tables->first;
        u.second = tables->second;
        auto kernel = once ? block_row_norms_kernel<true, true> : block_row_norms_kernel<false, true>;
        in_launches((c.n_items + kNormItems - 1) / kNormItems, 256, [&](int64_t first, dim3 grid) {
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, u, n_layers, c.n_items, first);
        });
        TW_HIP(hipGetLastError());
        return TW_OK;
    }
    if (tables)
        if (const int st = put_table(tables->host, tables->bytes, tables->dev, tables->first, tables->second, s))
            return st;
    if (blocks) {
        auto kernel = once ? block_row_norms_kernel<true, false> : block_row_norms_kernel<false, false>;
        in_launches((c.n_items + kNormItems - 1) / kNormItems, 256, [&](int64_t first, dim3 grid) {
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, NormTable{d_table}, n_layers, c.n_items, first);
        });
    } else {
        auto kernel = once ? tile_row_norms_kernel<true> : tile_row_norms_kernel<false>;
        in_launches(c.n_items, 256, [&](int64_t first, dim3 grid) {
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, d_table, n_layers, n_items, first);
        });
    }
    TW_HIP(hipGetLastError());
    return TW_OK;
}

// masks of more layers than a launch takes addresses: into the table, before it goes to the device
int early_masks(CallTable &c, Masks &masks)
{
    const int n_layers = (int)c.layers.size();
    if (n_layers <= kLateMasks)
        return TW_OK;
    const int st = masks.get(n_layers, nullptr);
    for (int l = 0; !st && l < n_layers; ++l)
        c.layers[l].mask = masks.m[l];
    return st;
}
int queue_fill(const CallTable &c, Masks &masks, Arena &ar, const PruneLayer *d_table, const SelectState *d_st, const Threshold *d_tile_thr, Mail *mail,
               hipStream_t s)
{
    const int n_layers = (int)c.layers.size();
    const int st = masks.get(n_layers, &ar);
    if (st)
        return st;
    MaskTable m;
    std::memset(&m, 0, sizeof(m));
    for (int l = 0; l < std::min(n_layers, kLateMasks); ++l)
        m.m[l] = masks.m[l];
    hipLaunchKernelGGL(fill_mask_kernel, dim3((unsigned)c.n_fill), dim3(256), 0, s, d_table, n_layers, d_st, d_tile_thr, mail, m);
    TW_HIP(hipGetLastError());
    return TW_OK;
}

int too_large(int64_t workgroups)
{
    return workgroups > 0x7fffffff ? fail(TW_ERR_SHAPE, "%lld workgroups: a launch takes at most 2^31 - 1", (long long)workgroups)
                                   : TW_OK;
}

// tiles of `granularity` columns: norms of all layers into one pooled vector, one threshold (or, with
// kPerTileThreshold, one per tile of the only layer), masks.  *threshold receives it.  `last`: nobody reads the scores right after.
int uniform_rows(int n_layers, const int32_t *K, const int32_t *N, const float *const *scores, double q, int q_is_f64,
                 int granularity, Masks masks, double *threshold, hipStream_t s, int flags, bool last = true)
{
    CallTable c = make_table(n_layers, K, N, scores, granularity, flags);
    const bool per_tile = (flags & kPerTileThreshold) != 0;
    const int n_seg = per_tile ? c.layers[0].n_tiles : 1;
    const bool in_blocks = per_tile && K[0] <= kTileSelect; // a workgroup a tile, no counters in memory
    int st = check_percentile(c.n_norms / n_seg, q);
    if (!st)
        st = too_large(std::max(c.n_items, c.n_fill));
    if (!st)
        st = early_masks(c, masks);
    if (st)
        return st;
    Arena ar(s);
    float *d_norms = ar.alloc_n<float>(c.n_norms);
    PruneLayer *d_table = ar.alloc_n<PruneLayer>(n_layers);
    SelectState *d_st = ar.alloc_n<SelectState>(in_blocks ? 0 : n_seg);
    Threshold *d_tile_thr = per_tile ? ar.alloc_n<Threshold>(n_seg) : nullptr;
    Mail *mail = ar.mail();
    if (!d_norms || !d_table || !d_st || (per_tile && !d_tile_thr) || !mail)
        return fail(TW_ERR_ALLOC, "allocation of %lld norms failed", (long long)c.n_norms);
    int64_t off = 0;
    for (PruneLayer &e : c.layers) {
        e.norms = d_norms + off;
        off += (int64_t)e.K * e.n_tiles;
    }
    const Tables tables{c.layers.data(), sizeof(PruneLayer) * n_layers, d_table,
                        setup_of(d_st, in_blocks ? 0 : n_seg, c.n_norms / n_seg, q, q_is_f64), SetupSelect{}};
    st = queue_norms(c, d_table, nullptr, last, s, &tables);
    if (st)
        return st;
    // per-tile thresholds (one layer): every tile's K norms are one segment
    if (in_blocks) {
        auto kernel = K[0] <= 1024 ? tile_select_kernel<1024> : tile_select_kernel<kTileSelect>;
        in_launches(n_seg, 256, [&](int64_t first, dim3 grid) {
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, d_norms, K[0], q, q_is_f64, d_tile_thr, mail, first);
        });
    } else {
        st = queue_select(d_norms, c.n_norms / n_seg, d_st, n_seg, s);
        if (st)
            return st;
        if (per_tile)
            hipLaunchKernelGGL(select_finish_kernel, dim3(n_seg), dim3(256), 0, s, d_st, d_tile_thr, mail);
    }
    st = queue_fill(c, masks, ar, d_table, d_st, d_tile_thr, mail, s);
    if (st)
        return st;
    st = ar.wait();
    if (!st && threshold)
        *threshold = mail->thr_rows;
    return st;
}

// The second stage of the mixed producers (tw_mix_fn): its buffers, its table of the layers, and the launches behind it.
class MixCall {
public:
    // `masks0` or, where that is nullptr, `rows`: the table of a first stage whose masks nobody has written (norms and tiles)
    int plan(int n_layers, const int32_t *K, const int32_t *N, const float *const *scores, const uint8_t *const *masks0,
             const CallTable *rows, double q, int q_type)
    {
        layers_.resize(n_layers);
        for (int l = 0; l < n_layers; ++l) {
            MixLayer &e = layers_[l];
            std::memset(&e, 0, sizeof(e));
            e.score = scores[l];
            e.mask0 = masks0 ? masks0[l] : nullptr;
            e.n = (int64_t)K[l] * N[l];
            e.begin = total_;
            e.item_begin = n_items_;
            e.K = K[l];
            e.N = N[l];
            e.G = rows ? rows->layers[l].granularity : 1;
            e.per_n = 1.0 / N[l];
            e.per_nf = 1.0f / (float)N[l];
            e.per_g = 1.0f / (float)e.G;
            e.rows_on = kMixItem / 4 / N[l];
            e.cols_on = kMixItem / 4 % N[l];
            total_ += e.n;
            n_items_ += (e.n + kMixItem - 1) / kMixItem;
        }
        q_ = q;
        q_type_ = q_type;
        return check_percentile(total_, q);
    }
    void write_to(uint8_t *const *masks)
    {
        for (size_t l = 0; l < layers_.size(); ++l) {
            MixLayer &e = layers_[l];
            e.out = masks[l];
            const bool wide = e.mask0 || (e.G >= 3 && e.N >= 3 && (e.N % e.G == 0 || e.N % e.G >= 3));
            if (((uintptr_t)e.score & 15) == 0 && (((uintptr_t)e.mask0 | (uintptr_t)e.out) & 3) == 0 && wide)
                e.in_fours = e.N % 4 == 0 && e.G % 4 == 0 ? 2 : 1;
        }
    }
    int alloc(Arena &ar)
    {
        // room for the values inside the bracket: an eighth of the elements, and all of a small network's
        wgs_ = (int)std::min<int64_t>(n_items_, kMixWgs);
        const int64_t share = (n_items_ + wgs_ - 1) / wgs_ * (kMixItem / 4); // elements of a wave
        room_ = (uint32_t)(sampled() ? std::max<int64_t>(share / 8, 512) : share);
        d_cand_ = ar.alloc_n<u32x2>((size_t)wgs_ * 4 * room_);
        d_counts_ = ar.alloc_n<MixCounts>(wgs_ * 4);
        d_bits_ = ar.alloc_n<uint16_t>((size_t)n_items_ * 256);
        d_sample_ = ar.alloc_n<uint32_t>(kMixSamples);
        d_st_ = ar.alloc_n<SelectState>(1);
        if (!d_cand_ || !d_counts_ || !d_bits_ || !d_sample_ || !d_st_)
            return fail(TW_ERR_ALLOC, "allocation for %lld element scores failed", (long long)total_);
        return TW_OK;
    }
    bool sampled() const { return total_ > kMixSampleFrom; }
    size_t table_bytes() const { return sizeof(MixLayer) * layers_.size(); }
    std::vector<MixLayer> &table() { return layers_; }
    SetupSelect setup() const { return setup_of(d_st_, 1, total_, q_, q_type_, room_); }
    // behind put_table of the table (at d_layers on the device; where the masks are is not looked at) and, with SRC == MIX_NORMS, the
    // passes of the selection of `st_rows`
    template <int SRC> void queue_bracket(const MixLayer *d_layers, const SelectState *st_rows, Mail *mail, hipStream_t s)
    {
        if (!sampled())
            return;
        hipLaunchKernelGGL(mix_sample_kernel<SRC>, dim3(kMixSamples / 256), dim3(256), 0, s, d_layers, (int)layers_.size(), total_, st_rows,
                           d_st_, d_sample_, mail);
        hipLaunchKernelGGL(mix_bracket_kernel, dim3(1), dim3(kBracketThreads), 0, s, d_sample_, d_st_);
    }
    // behind that, and put_table of the table with the masks' places
    template <int SRC> int queue(const MixLayer *d_layers, const SelectState *st_rows, Mail *mail, hipStream_t s)
    {
        const int n_layers = (int)layers_.size(), waves = wgs_ * 4;
        bool split = false;
        for (const MixLayer &e : layers_)
            split |= e.in_fours == 1;
        auto narrow = SRC == MIX_NORMS && split ? mix_narrow_kernel<MIX_SPLIT> : mix_narrow_kernel<SRC>;
        hipLaunchKernelGGL(narrow, dim3(wgs_), dim3(256), 0, s, d_layers, n_layers, n_items_, st_rows, d_st_, d_cand_,
                           d_counts_, d_bits_, mail, sampled() ? 1 : 0);
        const dim3 grid((unsigned)std::min<int64_t>(n_items_, 512));
        hipLaunchKernelGGL(mix_hist_kernel<0>, grid, dim3(256), 0, s, d_layers, n_layers, n_items_, d_st_, d_cand_, d_counts_, waves,
                           d_bits_);
        hipLaunchKernelGGL(mix_hist_kernel<1>, grid, dim3(256), 0, s, d_layers, n_layers, n_items_, d_st_, d_cand_, d_counts_, waves,
                           d_bits_);
        hipLaunchKernelGGL(mix_hist_kernel<2>, grid, dim3(256), 0, s, d_layers, n_layers, n_items_, d_st_, d_cand_, d_counts_, waves,
                           d_bits_);
        hipLaunchKernelGGL(mix_mark_kernel, dim3(wgs_), dim3(256), 0, s, d_layers, n_layers, n_items_, d_st_, d_cand_,
                           d_counts_, d_bits_, mail);
        TW_HIP(hipGetLastError());
        return TW_OK;
    }

private:
    std::vector<MixLayer> layers_;
    int64_t total_ = 0, n_items_ = 0;
    double q_ = 0.0;
    int q_type_ = 0, wgs_ = 0;
    uint32_t room_ = 0;
    u32x2 *d_cand_ = nullptr;
    uint32_t *d_sample_ = nullptr;
    MixCounts *d_counts_ = nullptr;
    uint16_t *d_bits_ = nullptr;
    SelectState *d_st_ = nullptr;
};

} // namespace

void release_producer_memory()
{
    std::lock_guard<std::mutex> lock(g_kept_mutex);
    for (Kept &k : g_kept) {
        if (k.held)
            k.drop = true;
        else
            k.give_back();
    }
}

} // namespace tw

using namespace tw;

extern "C" {

int tw_tiles_every_g_columns(int N, int G, int32_t *tile_col0, int32_t *tile_width, int32_t *n_tiles)
{
    if (N <= 0 || G <= 0)
        return fail(TW_ERR_SHAPE, "N=%d G=%d must be positive", N, G);
    if (!tile_col0 || !tile_width || !n_tiles)
        return fail(TW_ERR_NULL, "an output pointer is NULL");
    int t = 0;
    for (int c = 0; c < N; c += G, ++t) {
        tile_col0[t] = c;
        tile_width[t] = std::min(G, N - c);
    }
    *n_tiles = t;
    return TW_OK;
}

int tw_tiles_every_g_kept_columns(int N, int G, const uint8_t *col_mask, int32_t *tile_col0,
                                  int32_t *tile_width, int32_t *n_tiles)
try {
    if (N <= 0 || G <= 0)
        return fail(TW_ERR_SHAPE, "N=%d G=%d must be positive", N, G);
    if (!col_mask || !tile_col0 || !tile_width || !n_tiles)
        return fail(TW_ERR_NULL, "a pointer is NULL");
    int t = 0, start = 0, kept = 0;
    for (int c = 0; c < N; ++c) {
        kept += col_mask[c] != 0;
        if (kept == G && c + 1 < N) {
            tile_col0[t] = start;
            tile_width[t] = c + 1 - start;
            ++t;
            start = c + 1;
            kept = 0;
        }
    }
    tile_col0[t] = start;
    tile_width[t] = N - start;
    *n_tiles = t + 1;
    return TW_OK;
}
TW_CATCH_TO_STATUS

int tw_prune_tile_row_norms(int K, int N, const float *scores, int n_tiles,
                            const int32_t *tile_col0, const int32_t *tile_width,
                            const uint8_t *col_keep, float *norms, void *stream)
try {
    if (K <= 0 || N <= 0 || n_tiles <= 0)
        return fail(TW_ERR_SHAPE, "K=%d N=%d n_tiles=%d must be positive", K, N, n_tiles);
    if (!scores || !tile_col0 || !tile_width || !norms)
        return fail(TW_ERR_NULL, "a pointer is NULL");
    std::vector<int32_t> tcol0(n_tiles + 1);
    int c = 0;
    for (int t = 0; t < n_tiles; ++t) {
        if (tile_col0[t] != c || tile_width[t] <= 0)
            return fail(TW_ERR_TILE_TABLE, "tile %d: col0=%d width=%d", t, tile_col0[t], tile_width[t]);
        tcol0[t] = c;
        c += tile_width[t];
    }
    if (c != N)
        return fail(TW_ERR_TILE_TABLE, "tiles cover %d columns, N=%d", c, N);
    tcol0[n_tiles] = N;
    const int64_t n_items = (int64_t)((K + kNormRows - 1) / kNormRows) * n_tiles;
    int st = too_large(n_items);
    if (st)
        return st;
    hipStream_t s = (hipStream_t)stream;
    Arena ar(s);
    int32_t *d_tab = ar.alloc_n<int32_t>(n_tiles + 1);
    PruneLayer *d_table = ar.alloc_n<PruneLayer>(1);
    if (!d_tab || !d_table)
        return fail(TW_ERR_ALLOC, "hipMalloc of the tile table failed");
    PruneLayer e;
    std::memset(&e, 0, sizeof(e));
    e.score = scores;
    e.colkeep = const_cast<uint8_t *>(col_keep); // (read only)
    e.tcol0 = d_tab;
    e.norms = norms;
    e.K = K;
    e.N = N;
    e.n_tiles = n_tiles;
    st = put_table(tcol0.data(), sizeof(int32_t) * (n_tiles + 1), d_tab, setup_of(nullptr, 0, 0, 0.0, 0), SetupSelect{}, s);
    if (!st)
        st = put_table(&e, sizeof(e), d_table, setup_of(nullptr, 0, 0, 0.0, 0), SetupSelect{}, s);
    if (st)
        return st;
    in_launches(n_items, 256, [&](int64_t first, dim3 grid) {
        hipLaunchKernelGGL(tile_row_norms_kernel<false>, grid, dim3(256), 0, s, d_table, 1, (const int64_t *)nullptr, first);
    });
    TW_HIP(hipGetLastError());
    return ar.wait();
}
TW_CATCH_TO_STATUS

int tw_prune_col_norms(int K, int N, const float *scores, float *norms, void *stream)
try {
    if (K <= 0 || N <= 0)
        return fail(TW_ERR_SHAPE, "K=%d N=%d must be positive", K, N);
    if (!scores || !norms)
        return fail(TW_ERR_NULL, "a pointer is NULL");
    hipStream_t s = (hipStream_t)stream;
    Arena ar(s);
    ColLayer *d_cl = ar.alloc_n<ColLayer>(1);
    if (!d_cl)
        return fail(TW_ERR_ALLOC, "hipMalloc of the layer table failed");
    const ColLayer cl{scores, K, N, 0, 0};
    const int st = put_table(&cl, sizeof(cl), d_cl, setup_of(nullptr, 0, 0, 0.0, 0), SetupSelect{}, s);
    if (st)
        return st;
    in_launches(((int64_t)N + kColCols - 1) / kColCols, kColThreads, [&](int64_t first, dim3 grid) {
        hipLaunchKernelGGL(col_norms_kernel, grid, dim3(kColThreads), 0, s, d_cl, 1, norms, first);
    });
    TW_HIP(hipGetLastError());
    return ar.wait();
}
TW_CATCH_TO_STATUS

int tw_percentile_linear(const float *values, int64_t n, double q, int q_type, double *result,
                         void *stream)
try {
    if (!values || !result)
        return fail(TW_ERR_NULL, "a pointer is NULL");
    if (q_type != TW_Q_F32 && q_type != TW_Q_F64)
        return fail(TW_ERR_LAYOUT, "q_type=%d: unknown", q_type);
    hipStream_t s = (hipStream_t)stream;
    int st = check_percentile(n, q);
    if (st)
        return st;
    Arena ar(s);
    SelectState *d_st = ar.alloc_n<SelectState>(1);
    Threshold *d_thr = ar.alloc_n<Threshold>(1);
    Mail *mail = ar.mail();
    if (!d_st || !d_thr || !mail)
        return fail(TW_ERR_ALLOC, "allocation of the selection state failed");
    st = put_table(nullptr, 0, d_st, setup_of(d_st, 1, n, q, q_type), SetupSelect{}, s);
    if (!st)
        st = queue_select(values, n, d_st, 1, s);
    if (st)
        return st;
    hipLaunchKernelGGL(select_finish_kernel, dim3(1), dim3(256), 0, s, d_st, d_thr, mail);
    TW_HIP(hipGetLastError());
    TW_HIP(hipMemcpyAsync(result, &d_thr->v64, sizeof(double), hipMemcpyDeviceToHost, s));
    return ar.wait();
}
TW_CATCH_TO_STATUS

int tw_prune_tiled_wise_1d_late(int n_layers, const int32_t *K, const int32_t *N,
                                const float *const *scores, double sparsity, int q_type,
                                int granularity, uint8_t *const *masks, tw_masks_ready ready, void *user, double *threshold, void *stream)
try {
    const Masks m{masks, ready, user};
    int st = check_layers(n_layers, K, N, scores, m, granularity);
    if (st)
        return st;
    if (q_type != TW_Q_F32 && q_type != TW_Q_F64)
        return fail(TW_ERR_LAYOUT, "q_type=%d: unknown", q_type);
    return uniform_rows(n_layers, K, N, scores, sparsity, q_type, granularity, m, threshold, (hipStream_t)stream, 0);
}
TW_CATCH_TO_STATUS

int tw_prune_tiled_wise_1d(int n_layers, const int32_t *K, const int32_t *N,
                           const float *const *scores, double sparsity, int q_type,
                           int granularity, uint8_t *const *masks, double *threshold, void *stream)
{
    return tw_prune_tiled_wise_1d_late(n_layers, K, N, scores, sparsity, q_type, granularity, masks, nullptr, nullptr, threshold, stream);
}

int tw_prune_granularity(int K, int N, const float *scores, double sparsity, int q_type,
                         int granularity, uint8_t *mask, void *stream)
try {
    const float *const sc[1] = {scores};
    uint8_t *const mk[1] = {mask};
    const Masks m{mk};
    int st = check_layers(1, &K, &N, sc, m, granularity);
    if (st)
        return st;
    if (q_type != TW_Q_F32 && q_type != TW_Q_F64)
        return fail(TW_ERR_LAYOUT, "q_type=%d: unknown", q_type);
    if (N % granularity != 0)
        return fail(TW_ERR_SHAPE, "N=%d is not a multiple of the granularity %d", N, granularity);
    return uniform_rows(1, &K, &N, sc, sparsity, q_type, granularity, m, nullptr, (hipStream_t)stream,
                        kNormNotDivided | kPerTileThreshold);
}
TW_CATCH_TO_STATUS

int tw_prune_tiled_wise_2d(int n_layers, const int32_t *K, const int32_t *N,
                           const float *const *scores, double sparsity, int q_type, int transform,
                           int granularity, uint8_t *const *masks, uint8_t *const *col_masks,
                           double *thresholds, void *stream)
{
    return tw_prune_tiled_wise_2d_late(n_layers, K, N, scores, sparsity, q_type, transform, granularity, masks, nullptr, nullptr, col_masks,
                                       thresholds, stream);
}

int tw_prune_tiled_wise_2d_late(int n_layers, const int32_t *K, const int32_t *N,
                                const float *const *scores, double sparsity, int q_type, int transform,
                                int granularity, uint8_t *const *masks, tw_masks_ready ready, void *user, uint8_t *const *col_masks,
                                double *thresholds, void *stream)
try {
    Masks m{masks, ready, user};
    int st = check_layers(n_layers, K, N, scores, m, granularity);
    if (st)
        return st;
    if (q_type != TW_Q_F32 && q_type != TW_Q_F64)
        return fail(TW_ERR_LAYOUT, "q_type=%d: unknown", q_type);
    hipStream_t s = (hipStream_t)stream;
    double q = sparsity;
    if (transform) {
        // the two prunings compose to `sparsity`; NumPy's result here is a float64
        if (!(sparsity >= 0.0 && sparsity <= 100.0))
            return fail(TW_ERR_SHAPE, "sparsity %g is outside [0, 100]", sparsity);
        q = 100.0 - std::sqrt(10000.0 - sparsity * 100.0);
        q_type = TW_Q_F64;
    }
    // columns: one pooled vector of column norms, one threshold; then, without a trip to the host,
    // the tiles and the rows
    CallTable c = make_table(n_layers, K, N, scores, granularity, 0);
    st = check_percentile(c.n_cols, q);
    if (!st)
        st = too_large(std::max({c.n_items, c.n_fill, c.n_cols}));
    if (!st)
        st = early_masks(c, m);
    if (st)
        return st;
    Arena ar(s);
    float *d_cnorm = ar.alloc_n<float>(c.n_cols);
    uint8_t *d_ckeep = ar.alloc_n<uint8_t>(c.n_cols);
    int32_t *d_tcol = ar.alloc_n<int32_t>(c.n_tcol);
    float *d_norms = ar.alloc_n<float>(c.n_norms);
    int64_t *d_items = ar.alloc_n<int64_t>(1);
    SelectState *d_st = ar.alloc_n<SelectState>(1);
    // both layer tables in one buffer: one upload
    const size_t table_bytes = sizeof(PruneLayer) * n_layers;
    char *d_tables = static_cast<char *>(ar.alloc(table_bytes + sizeof(ColLayer) * n_layers));
    Mail *mail = ar.mail();
    if (!d_cnorm || !d_ckeep || !d_tcol || !d_norms || !d_items || !d_st || !d_tables || !mail)
        return fail(TW_ERR_ALLOC, "allocation for %lld columns and %lld norms failed", (long long)c.n_cols, (long long)c.n_norms);
    PruneLayer *d_table = reinterpret_cast<PruneLayer *>(d_tables);
    ColLayer *d_cl = reinterpret_cast<ColLayer *>(d_tables + table_bytes);
    std::vector<char> both(table_bytes + sizeof(ColLayer) * n_layers);
    int64_t n_blk = 0, n_tcol = 0;
    for (int l = 0; l < n_layers; ++l) {
        PruneLayer &e = c.layers[l];
        e.colkeep = d_ckeep + e.col_begin;
        e.colout = col_masks ? col_masks[l] : nullptr;
        e.tcol0 = d_tcol + n_tcol;
        n_tcol += e.n_tiles + 1;
        const ColLayer cl{scores[l], K[l], N[l], e.col_begin, n_blk};
        std::memcpy(both.data() + table_bytes + sizeof(ColLayer) * l, &cl, sizeof(cl));
        n_blk += (N[l] + kColCols - 1) / kColCols;
    }
    std::memcpy(both.data(), c.layers.data(), table_bytes);
    st = put_table(both.data(), both.size(), d_tables, setup_of(d_st, 1, 0, q, q_type), SetupSelect{}, s);
    if (st)
        return st;
    in_launches(n_blk, kColThreads, [&](int64_t first, dim3 grid) {
        hipLaunchKernelGGL(col_norms_kernel, grid, dim3(kColThreads), 0, s, d_cl, n_layers, d_cnorm, first);
    });
    hipLaunchKernelGGL(plan_2d_kernel, dim3(1), dim3(kPlanThreads), 0, s, d_table, n_layers, d_cnorm, c.n_cols, d_norms,
                       d_st, d_items, q, q_type, mail);
    st = queue_norms(c, d_table, d_items, false, s);
    if (!st)
        st = queue_select(d_norms, c.n_norms, d_st, 1, s);
    if (st)
        return st;
    st = queue_fill(c, m, ar, d_table, d_st, nullptr, mail, s);
    if (st)
        return st;
    st = ar.wait();
    if (!st && thresholds) {
        thresholds[0] = mail->thr_cols;
        thresholds[1] = mail->thr_rows;
    }
    return st;
}
TW_CATCH_TO_STATUS

int tw_prune_mix(int n_layers, const int32_t *K, const int32_t *N, const float *const *scores,
                 const uint8_t *const *layer_masks, double g1percent, int q_type,
                 uint8_t *const *masks, double *threshold, void *stream)
try {
    int st = check_layers(n_layers, K, N, scores, Masks{masks}, 1);
    if (st)
        return st;
    if (!layer_masks)
        return fail(TW_ERR_NULL, "layer_masks is NULL");
    if (q_type != TW_Q_F32 && q_type != TW_Q_F64)
        return fail(TW_ERR_LAYOUT, "q_type=%d: unknown", q_type);
    for (int l = 0; l < n_layers; ++l)
        if (!layer_masks[l])
            return fail(TW_ERR_NULL, "layer %d: layer mask pointer is NULL", l);
    hipStream_t s = (hipStream_t)stream;
    MixCall mix;
    st = mix.plan(n_layers, K, N, scores, layer_masks, nullptr, 100.0 - g1percent, q_type);
    if (st)
        return st;
    mix.write_to(masks);
    Arena ar(s);
    st = mix.alloc(ar);
    MixLayer *d_layers = ar.alloc_n<MixLayer>(n_layers);
    Mail *mail = ar.mail();
    if (!st && (!d_layers || !mail))
        st = fail(TW_ERR_ALLOC, "allocation for %d layers failed", n_layers);
    if (!st)
        st = put_table(mix.table().data(), mix.table_bytes(), d_layers, mix.setup(), SetupSelect{}, s);
    if (!st) {
        mix.queue_bracket<MIX_BYTES>(d_layers, nullptr, mail, s);
        st = mix.queue<MIX_BYTES>(d_layers, nullptr, mail, s);
    }
    if (st)
        return st;
    st = ar.wait();
    if (!st && threshold)
        *threshold = mail->thr_rows;
    return st;
}
TW_CATCH_TO_STATUS

int tw_prune_tiled_wise_1d_mix_late(int n_layers, const int32_t *K, const int32_t *N, const float *const *scores, double sparsity,
                                    int q_type, int granularity, double g1percent, int g1_q_type, uint8_t *const *masks,
                                    tw_masks_ready ready, void *user, double *threshold, void *stream)
try {
    Masks m{masks, ready, user};
    int st = check_layers(n_layers, K, N, scores, m, granularity);
    if (st)
        return st;
    if ((q_type != TW_Q_F32 && q_type != TW_Q_F64) || (g1_q_type != TW_Q_F32 && g1_q_type != TW_Q_F64))
        return fail(TW_ERR_LAYOUT, "q_type=%d, %d: unknown", q_type, g1_q_type);
    for (int l = 0; l < n_layers; ++l)
        if (N[l] > kMixMaxN || K[l] > kMixMaxK || (N[l] + (int64_t)granularity - 1) / granularity * K[l] > kMixMaxNorms) { // one stage after the other
            st = m.get(n_layers, nullptr);
            if (!st)
                st = uniform_rows(n_layers, K, N, scores, sparsity, q_type, granularity, m, nullptr, (hipStream_t)stream, 0, false);
            return st ? st : tw_prune_mix(n_layers, K, N, scores, masks, g1percent, g1_q_type, masks, threshold, stream);
        }
    hipStream_t s = (hipStream_t)stream;
    CallTable c = make_table(n_layers, K, N, scores, granularity, 0);
    MixCall mix;
    st = check_percentile(c.n_norms, sparsity);
    if (!st)
        st = too_large(c.n_items);
    if (!st)
        st = mix.plan(n_layers, K, N, scores, nullptr, &c, 100.0 - g1percent, g1_q_type);
    if (st)
        return st;
    Arena ar(s);
    float *d_norms = ar.alloc_n<float>(c.n_norms);
    SelectState *d_st = ar.alloc_n<SelectState>(1);
    // both layer tables in one buffer: one upload
    const size_t table_bytes = sizeof(PruneLayer) * n_layers;
    char *d_tables = static_cast<char *>(ar.alloc(table_bytes + mix.table_bytes()));
    Mail *mail = ar.mail();
    if (!d_norms || !d_st || !d_tables || !mail)
        return fail(TW_ERR_ALLOC, "allocation of %lld norms failed", (long long)c.n_norms);
    st = mix.alloc(ar);
    if (st)
        return st;
    int64_t off = 0;
    for (int l = 0; l < n_layers; ++l) {
        c.layers[l].norms = d_norms + off;
        mix.table()[l].norms = d_norms + off;
        off += (int64_t)K[l] * c.layers[l].n_tiles;
    }
    PruneLayer *d_table = reinterpret_cast<PruneLayer *>(d_tables);
    MixLayer *d_layers = reinterpret_cast<MixLayer *>(d_tables + table_bytes);
    std::vector<char> both(table_bytes + mix.table_bytes());
    std::memcpy(both.data(), c.layers.data(), table_bytes);
    std::memcpy(both.data() + table_bytes, mix.table().data(), mix.table_bytes());
    const Tables tables{both.data(), both.size(), d_tables, setup_of(d_st, 1, c.n_norms, sparsity, q_type), mix.setup()};
    st = queue_norms(c, d_table, nullptr, false, s, &tables);
    if (!st)
        st = queue_select(d_norms, c.n_norms, d_st, 1, s);
    if (st)
        return st;
    // (everything that the masks' places are not needed for is on its way when the caller allocates them)
    mix.queue_bracket<MIX_NORMS>(d_layers, d_st, mail, s);
    st = m.get(n_layers, &ar);
    if (st)
        return st;
    mix.write_to(masks);
    st = put_table(mix.table().data(), mix.table_bytes(), d_layers, SetupSelect{}, SetupSelect{}, s);
    if (!st)
        st = mix.queue<MIX_NORMS>(d_layers, d_st, mail, s);
    if (st)
        return st;
    st = ar.wait();
    if (!st && threshold)
        *threshold = mail->thr_rows;
    return st;
}
TW_CATCH_TO_STATUS

int tw_prune_tiled_wise_1d_mix(int n_layers, const int32_t *K, const int32_t *N, const float *const *scores, double sparsity,
                               int q_type, int granularity, double g1percent, int g1_q_type, uint8_t *const *masks,
                               double *threshold, void *stream)
{
    return tw_prune_tiled_wise_1d_mix_late(n_layers, K, N, scores, sparsity, q_type, granularity, g1percent, g1_q_type, masks, nullptr,
                                           nullptr, threshold, stream);
}

} // extern "C"
