// Plan construction for libtwgemm: the integer mask -> kept lists -> relative
// offsets -> compaction pre-pass (HIP kernels), the MFMA-ordered weight packing,
// and the read-back used for bit-exact checks.
//
// Packed weight of tile t (K_t x N_t compact, padded to k_pad x n_pad, nblk = n_pad/32):
//   for 64-row step s, 32-column block nb, k16 step ks (0..3), lane l (0..63), e (0..7):
//     Bp[b_off + (((s * nblk + nb) * 4 + ks) * 64 + l) * 8 + e]
//        = compact[s*64 + ks*16 + (l/32)*8 + e][nb*32 + l%32]      (0 outside K_t x N_t)
// i.e. one MFMA B operand is 16 bytes per lane, 1 KiB contiguous per wave, and the whole
// block a 64-row main-loop step needs is one contiguous run of nblk * 4 KiB.
#include "tw_internal.h"
#include "tw_device.h"

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstring>
#include <map>
#include <mutex>

namespace tw {

constexpr int kPackKS = kBlockK / kMfmaK; // MFMA k steps per packed step

// One tile of a plan being built: its geometry, where its lists lie among the ones they are made from
// (kk_src, kn_src, pn_src) and where they go (kk_dst ...; see GemmArgs for the padded copies).
struct PlanTile {
    int32_t col0, k_kept, n_kept, k_pad, n_pad, n_pruned;
    int32_t kk_dst, kn_dst, pn_dst;
    int32_t kkp_dst, kkp_len;  // its stretch of the padded list of rows
    int32_t pad_;
    int64_t kk_src, kn_src, pn_src;
    int64_t b_off;
    int64_t src_off; // stream layout only: element offset of the tile in B_stream
};

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f)
{
    uint32_t x = __float_as_uint(f);
    if ((x & 0x7F800000u) == 0x7F800000u && (x & 0x007FFFFFu))
        return (uint16_t)((x >> 16) | 0x0040u);
    x += 0x7FFFu + ((x >> 16) & 1u);
    return (uint16_t)(x >> 16);
}

__device__ __forceinline__ uint16_t f32_to_f16_rne(float f)
{
    _Float16 h = (_Float16)f; // v_cvt_f16_f32, round to nearest even
    return __builtin_bit_cast(uint16_t, h);
}

__device__ __forceinline__ uint16_t cast16(float f, int dtype)
{
    return dtype == TW_BF16 ? f32_to_bf16_rne(f) : f32_to_f16_rne(f);
}

// ---------------------------------------------------------------------------------
// packing

// Group g of a tile's packed weight: eight k rows of one column, the sixteen bytes of one lane.
struct PackPos {
    int n, kk0; // compact column, first compact row
    bool any;   // inside the tile's packed weight
};
__device__ __forceinline__ PackPos pack_pos(const PlanTile &t, int64_t g)
{
    PackPos q;
    q.any = g < (int64_t)t.k_pad * t.n_pad / 8;
    const int lane = (int)(g & 63);
    const uint32_t blk = (uint32_t)(g >> 6); // ((step * nblk + nb) * kPackKS + ks)
    const uint32_t nblk = max(t.n_pad / kMfmaN, 1);
    const uint32_t step = blk / kPackKS / nblk;
    q.n = (int)(blk / kPackKS - step * nblk) * kMfmaN + (lane & 31);
    q.kk0 = (int)(step * kPackKS + blk % kPackKS) * kMfmaK + (lane >> 5) * 8;
    return q;
}
__device__ __forceinline__ void pack_put(uint16_t *Bp, const PlanTile &t, int64_t g, const uint16_t (&v)[8])
{
    uint4 out;
    out.x = v[0] | ((uint32_t)v[1] << 16);
    out.y = v[2] | ((uint32_t)v[3] << 16);
    out.z = v[4] | ((uint32_t)v[5] << 16);
    out.w = v[6] | ((uint32_t)v[7] << 16);
    *reinterpret_cast<uint4 *>(Bp + t.b_off + g * 8) = out;
}

// From the dense fp32 weight.  `mask` (optional, K x N bytes): elements whose mask byte is zero are
// stored as zeros (covering plans of masks that are not rows x columns per tile).
__device__ __forceinline__ void pack_dense(const PlanTile &t, int64_t g, const int32_t *kept_k, const int32_t *kept_n,
                                           const float *B, int N, int dtype, uint16_t *Bp, const uint8_t *mask)
{
    const PackPos q = pack_pos(t, g);
    if (!q.any)
        return;
    // (what lies past the lists' ends repeats their last entry: no load is on a condition, so the eight rows' numbers are on their way
    // together and then the eight weights; VGG16's layers 3.4 - 4.2 us, 6.6 - 7.4 with each behind the one before)
    const bool in = q.n < t.n_kept;
    const int64_t col = t.col0 + kept_n[t.kn_src + min(q.n, t.n_kept - 1)];
    int32_t row[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        row[e] = kept_k[t.kk_src + min(q.kk0 + e, t.k_kept - 1)];
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        f[e] = B[(int64_t)row[e] * N + col];
    if (mask) {
        uint8_t m[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            m[e] = mask[(int64_t)row[e] * N + col];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            f[e] = m[e] ? f[e] : 0.0f;
    }
    uint16_t v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        v[e] = cast16(in && q.kk0 + e < t.k_kept ? f[e] : 0.0f, dtype);
    pack_put(Bp, t, g, v);
}

// From the reference's compacted layout: tile column j, row i at Bs[src_off + j*K + i]
// (gen_masked_stream_weight, basic_nn.cu:765).
__device__ __forceinline__ void pack_stream(const PlanTile &t, int64_t g, const uint16_t *Bs, int K, uint16_t *Bp)
{
    const PackPos q = pack_pos(t, g);
    if (!q.any)
        return;
    const uint16_t *const src = Bs + t.src_off + (int64_t)min(q.n, t.n_kept - 1) * K;
    uint16_t v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        v[e] = src[min(q.kk0 + e, t.k_kept - 1)];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        v[e] = q.n < t.n_kept && q.kk0 + e < t.k_kept ? v[e] : (uint16_t)0;
    pack_put(Bp, t, g, v);
}

// Everything of a plan that is not known on the host.  Row t of the grid packs tile t's weight, row
// n_tiles + t writes its lists, the last row copies the tables the host has made (units, tiles, blocks and
// the PlanTile table itself) out of pinned host memory and clears the ticket slots.  The tiles of most
// plans fit the kernel arguments, and then this is one launch; a plan of more runs it twice, once for
// the lists and tables (a workgroup reads its tile's entry across the bus, next to its other first
// loads) and once for the weight, out of the table the first has copied.
constexpr int kArgTiles = 24;
struct BuildArgs {
    const PlanTile *tiles; // null: arg_tiles
    int32_t row0;          // first row of this launch
    int32_t n_tiles, K, N, dtype;
    const int32_t *kk, *kn, *pn; // lists the plan is made from
    const float *B;              // dense weight, or
    const uint16_t *Bs;          // compacted weight in the stream layout
    const uint8_t *mask;
    const uint4 *header; // host
    uint4 *header_dst;
    int32_t *kept_k, *rel_k, *kept_n, *rel_n, *pruned_n, *kept_k_pad;
    uint32_t *kept_pairs;
    int32_t *tickets;
    uint16_t *Bp;
    int32_t header_chunks; // of 16 bytes
    int32_t ticket_words;
    PlanTile arg_tiles[kArgTiles];
};
__device__ __forceinline__ PlanTile build_tile(const BuildArgs &a, int t)
{
    constexpr int W = sizeof(PlanTile) / 4;
    int32_t w[W];
    if (a.tiles) {
        const auto *g = (const __attribute__((address_space(4))) int32_t *)(uintptr_t)(a.tiles + t);
#pragma unroll
        for (int i = 0; i < W; ++i)
            w[i] = g[i];
    } else {
        const auto *ka = (const __attribute__((address_space(4))) int32_t *)__builtin_amdgcn_kernarg_segment_ptr();
#pragma unroll
        for (int i = 0; i < W; ++i)
            w[i] = ka[offsetof(BuildArgs, arg_tiles) / 4 + t * W + i];
    }
    PlanTile q;
    __builtin_memcpy(&q, w, sizeof(q));
    return q;
}
__global__ void __launch_bounds__(256) plan_build_kernel(const BuildArgs a)
{
    const int y = a.row0 + (int)blockIdx.y;
    const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
    if (y < a.n_tiles) {
        const PlanTile t = build_tile(a, y);
        const int64_t groups = (int64_t)t.k_pad * t.n_pad / 8;
        for (int64_t g = i0; g < groups; g += step) {
            if (a.B)
                pack_dense(t, g, a.kk, a.kn, a.B, a.N, a.dtype, a.Bp, a.mask);
            else
                pack_stream(t, g, a.Bs, a.K, a.Bp);
        }
        return;
    }
    if (y == 2 * a.n_tiles) {
        for (int64_t i = i0; i < a.header_chunks; i += step)
            a.header_dst[i] = a.header[i];
        for (int64_t i = i0; i < a.ticket_words; i += step)
            a.tickets[i] = 0;
        return;
    }
    // All lists of the tile together, an entry of each a thread, out of loads that wait for nothing but each other's addresses (a list
    // after the other was as many trips to memory).  An empty list's entry comes from another one and is dropped.
    const PlanTile t = build_tile(a, y - a.n_tiles);
    const int32_t *const kk = t.k_kept > 0 ? a.kk + t.kk_src : t.n_kept > 0 ? a.kn + t.kn_src : a.pn + t.pn_src;
    const int32_t *const kn = t.n_kept > 0 ? a.kn + t.kn_src : kk, *const pn = t.n_pruned > 0 ? a.pn + t.pn_src : kk;
    const int last_k = max(t.k_kept, 1) - 1, last_n = max(t.n_kept, 1) - 1, last_p = max(t.n_pruned, 1) - 1;
    const int kept = t.n_kept > 0 ? t.k_kept : 0; // of the pairs
    const int64_t longest = max(max(t.k_kept, t.kkp_len), max(t.n_kept, t.n_pruned));
    for (int64_t i = i0; i < longest; i += step) {
        // pairs of rows (GemmArgs::kept_pairs); the padding names row K there (a row of zeros behind the
        // A-stationary kernel's panel), not row 0.  A tile without columns has no unit and its list
        // counts as padding.
        const int in = (int)(i & 31), e = in >> 2, g16 = in & 3;
        const int lo = (int)(i >> 5) * 64 + g16 * 16 + (e >> 2) * 8 + (e & 3);
        const int k = kk[min(i, (int64_t)last_k)], c = kn[min(i, (int64_t)last_n)], z = pn[min(i, (int64_t)last_p)];
        const int k_lo = kk[min(lo, last_k)], k_hi = kk[min(lo + 4, last_k)];
        if (i < t.k_kept) {
            a.kept_k[t.kk_dst + i] = k;
            a.rel_k[t.kk_dst + i] = k - (int)i;
        }
        if (i < t.n_kept) {
            a.kept_n[t.kn_dst + i] = c;
            a.rel_n[t.kn_dst + i] = c - (int)i;
        }
        if (i < t.n_pruned)
            a.pruned_n[t.pn_dst + i] = z;
        if (i < t.kkp_len)
            a.kept_k_pad[t.kkp_dst + i] = i < t.k_kept ? k : 0;
        if (a.kept_pairs && i < t.kkp_len / 2)
            a.kept_pairs[t.kkp_dst / 2 + i] = (lo < kept ? (uint32_t)k_lo : (uint32_t)a.K) | (lo + 4 < kept ? (uint32_t)k_hi : (uint32_t)a.K) << 16;
    }
}
// Inverse of the packing into the reference's compacted layout at K*col0.
__global__ void unpack_stream_kernel(const PlanTile *tiles, const uint16_t *Bp, int K, uint16_t *Bs)
{
    const PlanTile t = tiles[blockIdx.y];
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const PackPos q = pack_pos(t, g);
    if (!q.any || q.n >= t.n_kept)
        return;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int kk = q.kk0 + e;
        if (kk < t.k_kept)
            Bs[(int64_t)(t.col0 + q.n) * K + kk] = Bp[t.b_off + g * 8 + e];
    }
}

// ---------------------------------------------------------------------------------
// mask -> flags -> lists  (integer pre-pass)

// A tile keeps row k where any byte of mask[k][its columns] is non-zero, and a column likewise.  Two
// kernels: mask_flags_kernel reads the mask once, mask_lists_kernel turns the flags into ascending
// lists.  Whether the mask is rows x columns in every tile needs no second pass over it: its non-zero
// elements lie in that product, so it is exactly when they are as many as rows times columns.

// Rows of one tile and slab, and what a slab of kFlagRows rows of it says about the columns.
constexpr int kFlagRows = 128;
constexpr int kMaxTileRows = 32768; // tiles of one launch, where they are the rows of its grid
constexpr int kFlagArgTiles = 64;   // tiles whose first columns fit the kernel arguments
struct FlagArgs {
    const uint8_t *mask;
    const int32_t *tcol0; // host memory (pinned): first column of each tile, N behind the last; null: arg_tcol0
    int32_t K, N, n_slabs, tile0;
    uint8_t *rowflag;     // [tile][K]
    uint8_t *colpart;     // per tile [slab][width, rounded up to 4], see colpart_at
    uint32_t *nnz;        // [tile][slab]: non-zero elements
    int32_t arg_tcol0[kFlagArgTiles + 1];
    __device__ int64_t colpart_at(int t, int c0) const { return (int64_t)(((int64_t)c0 + 3 * t + 3) & ~(int64_t)3) * n_slabs; }
};

// First column of tile t (uniform), out of the arguments of a kernel whose first one is `a`: a read of the host's memory across
// the bus, at the head of both kernels, takes 1.5 us.
__device__ __forceinline__ int flag_col0(const FlagArgs &a, int t)
{
    if (a.tcol0)
        return a.tcol0[t];
    const auto *ka = (const __attribute__((address_space(4))) int32_t *)__builtin_amdgcn_kernarg_segment_ptr();
    return ka[offsetof(FlagArgs, arg_tcol0) / 4 + t];
}

typedef uint32_t Flags __attribute__((ext_vector_type(4), aligned(1))); // sixteen bytes at any address

// Workgroup (slab, tile): kFlagRows rows of one tile, so every flag has one writer and nothing has to
// be cleared first.  Each row is taken by 8, 16 or 32 lanes (LG: 3, 4, 5) of 16 bytes (windows of 32 lanes for wider
// tiles), all loads of a window in flight at once; a row's lanes vote, the rows of a column are
// joined with shuffles and through LDS.  What the mask's rows are aligned to (UNIT bytes) and the lanes of a row are constants of each copy, and
// what lies past a row's end repeats its last bytes: with a branch around a load the compiler waits for each of them (VGG16's layers 3.8 -
// 6.2 us, 3.8 - 9 with those, and a mask off 4 bytes 256 loads of a byte).
template <int UNIT, int LG> __device__ __forceinline__ void flags_of_slab(const FlagArgs &a, int t, int c0, int w)
{
    __shared__ uint32_t s_col[4][128]; // per wave, a window's columns
    __shared__ uint32_t s_nnz;
    constexpr int lpr = 1 << LG, rpp = 256 >> LG, kPasses = kFlagRows / rpp; // rows the workgroup takes at a time
    const int slab = (int)blockIdx.x;
    const int k0 = slab * kFlagRows, nr = min(kFlagRows, a.K - k0);
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int a0 = UNIT == 0 ? c0 : c0 & -UNIT, chunks = (c0 + w - a0 + 15) >> 4;
    const int64_t last16 = (int64_t)a.K * a.N - 16; // the mask's last sixteen bytes
    const int l = tid & (lpr - 1), r0 = tid >> LG;
    const uint8_t *const base = a.mask + (int64_t)k0 * a.N;
    uint32_t row_any = 0; // bit p: row r0 + p * rpp has an element (this lane's chunks)
    uint32_t nnz = 0;
    if (tid == 0)
        s_nnz = 0;
    for (int win = 0; win * lpr < chunks; ++win) {
        const int cc = a0 + (win * lpr + l) * 16; // first column of this lane's chunk
        uint32_t v[kPasses][4];
#pragma unroll
        for (int p = 0; p < kPasses; ++p) {
            const uint8_t *const row = base + (int64_t)min(r0 + p * rpp, nr - 1) * a.N;
            if constexpr (UNIT == 16) {
                const uint4 x = *reinterpret_cast<const uint4 *>(row + min(cc, a.N - 16));
                v[p][0] = x.x, v[p][1] = x.y, v[p][2] = x.z, v[p][3] = x.w;
            } else if constexpr (UNIT == 4) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    v[p][j] = *reinterpret_cast<const uint32_t *>(row + min(cc + j * 4, a.N - 4));
            } else if constexpr (UNIT == 1) {
                const int64_t at = row - a.mask + cc;
                const Flags x = *reinterpret_cast<const Flags *>(a.mask + min(at, last16));
                v[p][0] = x.x, v[p][1] = x.y, v[p][2] = x.z, v[p][3] = x.w;
            } else { // (less than 16 bytes of mask)
                uint32_t x[16];
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    x[e] = row[min(cc + e, a.N - 1)];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    v[p][j] = x[j * 4] | x[j * 4 + 1] << 8 | x[j * 4 + 2] << 16 | x[j * 4 + 3] << 24;
            }
        }
        if (UNIT == 1 && (int64_t)(a.K - k0 - nr) * a.N < 16) { // what was read before its place, the mask ending there, moves down
#pragma unroll
            for (int p = 0; p < kPasses; ++p) {
                const int64_t over = (int64_t)(k0 + min(r0 + p * rpp, nr - 1)) * a.N + cc - last16;
                if (over > 0) {
                    const int by = (int)min(over, (int64_t)16) * 8;
                    unsigned long long lo = (unsigned long long)v[p][1] << 32 | v[p][0], hi = (unsigned long long)v[p][3] << 32 | v[p][2];
                    lo = by >= 64 ? (by >= 128 ? 0ull : hi >> (by - 64)) : lo >> by | hi << 1 << (63 - by);
                    hi = by >= 64 ? 0ull : hi >> by;
                    v[p][0] = (uint32_t)lo, v[p][1] = (uint32_t)(lo >> 32), v[p][2] = (uint32_t)hi, v[p][3] = (uint32_t)(hi >> 32);
                }
            }
        }
        uint32_t in_tile[4], acc[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int lo = min(max(c0 - cc - j * 4, 0), 4), hi = min(max(c0 + w - cc - j * 4, 0), 4);
            in_tile[j] = (uint32_t)((1ull << (hi * 8)) - 1ull) & ~(uint32_t)((1ull << (lo * 8)) - 1ull);
        }
#pragma unroll
        for (int p = 0; p < kPasses; ++p) {
            uint32_t any = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t x = r0 + p * rpp < nr ? v[p][j] & in_tile[j] : 0u;
                const uint32_t nz = ((x | ((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu)) >> 7) & 0x01010101u;
                any |= nz;
                acc[j] |= nz;
                nnz += __popc(nz);
            }
            row_any |= (any ? 1u : 0u) << p;
        }
        // the window's columns over all rows of the slab
#pragma unroll
        for (int j = 0; j < 4; ++j)
            for (int off = lpr; off < 64; off <<= 1)
                acc[j] |= __shfl_xor(acc[j], off);
        if (lane < lpr) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                s_col[wave][l * 4 + j] = acc[j];
        }
        __syncthreads();
        const int wp = (w + 3) & ~3; // width of the slab's row of column flags
        uint8_t *const part = a.colpart + a.colpart_at(t, c0) + (int64_t)slab * wp;
        for (int j = tid; j < lpr * 16; j += 256) {
            const int rel = a0 + win * lpr * 16 + j - c0;
            const uint32_t x = s_col[0][j >> 2] | s_col[1][j >> 2] | s_col[2][j >> 2] | s_col[3][j >> 2];
            if (rel >= 0 && rel < w)
                part[rel] = (uint8_t)(x >> ((j & 3) * 8));
        }
        __syncthreads();
    }
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        const unsigned long long votes = __ballot(row_any >> p & 1u);
        const unsigned long long mine = (lpr == 32 ? 0xFFFFFFFFull : (1ull << lpr) - 1ull) << (lane & -lpr);
        if (l == 0 && r0 + p * rpp < nr)
            a.rowflag[(int64_t)t * a.K + k0 + r0 + p * rpp] = (votes & mine) != 0ull;
    }
    nnz = wave_scan(nnz);
    if (lane == 63)
        atomicAdd(&s_nnz, nnz);
    __syncthreads();
    if (tid == 0)
        a.nnz[(int64_t)t * a.n_slabs + slab] = s_nnz;
}
__global__ void __launch_bounds__(256, 3) mask_flags_kernel(const FlagArgs a)
{
    const int t = a.tile0 + (int)blockIdx.y;
    const int c0 = flag_col0(a, t), w = flag_col0(a, t + 1) - c0;
    auto lanes_of = [&](auto unit) { // loads of 16 bytes, 4 or, at any address, 16 again
        constexpr int UNIT = decltype(unit)::value;
        const int chunks = (c0 + w - (c0 & -UNIT) + 15) >> 4;
        if (chunks <= 8)
            flags_of_slab<UNIT, 3>(a, t, c0, w);
        else if (chunks <= 16)
            flags_of_slab<UNIT, 4>(a, t, c0, w);
        else
            flags_of_slab<UNIT, 5>(a, t, c0, w);
    };
    if ((a.N & 15) == 0 && ((uintptr_t)a.mask & 15) == 0)
        lanes_of(std::integral_constant<int, 16>());
    else if ((a.N & 3) == 0 && ((uintptr_t)a.mask & 3) == 0)
        lanes_of(std::integral_constant<int, 4>());
    else if ((int64_t)a.K * a.N >= 16)
        lanes_of(std::integral_constant<int, 1>());
    else
        flags_of_slab<0, 3>(a, t, c0, w);
}

// What the host needs to know of a tile before it can lay the plan out, in pinned memory: kept rows, kept columns, the low and
// the high half of the number of non-zero elements, each with the build's number above it.  A word is written
// at once, so none of them has to wait for another on its way across the bus.
struct TileCounts {
    unsigned long long word[4];
};

// One workgroup per tile: ascending lists of the kept rows (at kk + t * K), of the kept columns and of
// the pruned ones (both at the tile's first column), and the counts.  Every thread takes a run of
// neighbouring flags, so one scan orders all of them.
constexpr int kListThreads = 512;
__global__ void __launch_bounds__(kListThreads)
    mask_lists_kernel(const FlagArgs a, int32_t *kk, int32_t *kn, int32_t *pn, TileCounts *counts, uint32_t stamp)
{
    constexpr int NW = kListThreads / 64;
    __shared__ int s_wave[NW];
    __shared__ uint32_t s_cols[kListThreads]; // flags of a window of four times as many columns
    __shared__ unsigned long long s_nnz;
    const int t = (int)blockIdx.x, tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c0 = flag_col0(a, t), w = flag_col0(a, t + 1) - c0;
    // position of this thread's first one among all ones of the workgroup, and their number
    auto scan = [&](int mine, int &total) {
        const int incl = (int)wave_scan((uint32_t)mine);
        if (lane == 63)
            s_wave[wave] = incl;
        __syncthreads();
        int before = incl - mine;
        total = 0;
#pragma unroll
        for (int v = 0; v < NW; ++v) {
            before += v < wave ? s_wave[v] : 0;
            total += s_wave[v];
        }
        __syncthreads();
        return before;
    };
    if (tid == 0)
        s_nnz = 0;
    // The first loads of everything leave together, none of them on a condition (VGG16's layers 4.0 - 5.5 us, 4.1 - 6.5 with one part's
    // behind another's and a flag at a time, each behind the one before).
    // sixteen rows' flags a thread (what lies behind a tile's last one stays inside the workspace)
    const uint8_t *const flag = a.rowflag + (int64_t)t * a.K;
    auto rows_per_thread = [&](int base) { return min(16, (a.K - base + kListThreads - 1) / kListThreads); };
    auto flags_of = [&](int base) { return *reinterpret_cast<const Flags *>(flag + min(base + tid * rows_per_thread(base), a.K - 1)); };
    Flags f = flags_of(0);
    const uint32_t nnz0 = a.nnz[(int64_t)t * a.n_slabs + min(tid, a.n_slabs - 1)];
    // What the slabs say about a window's columns: four of them a thread, 2^lg threads side by side, the slabs dealt out over the
    // groups, eight of them at a time.
    const int words = ((w + 3) & ~3) >> 2;
    const uint32_t *const part = reinterpret_cast<const uint32_t *>(a.colpart + a.colpart_at(t, c0));
    const int lg = words >= kListThreads ? 9 : words > 1 ? 32 - __clz(words - 1) : 0, groups = kListThreads >> lg;
    static_assert(kListThreads == 512, "a window is at most 2^9 words");
    const int cj = tid & ((1 << lg) - 1);
    auto eight_slabs = [&](int base, int slab, uint32_t (&v)[8]) {
        const uint32_t *const src = part + min(base + cj, words - 1);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = src[(int64_t)min(slab + i * groups, a.n_slabs - 1) * words];
    };
    uint32_t v0[8];
    eight_slabs(0, tid >> lg, v0);
    auto slabs_of = [&](int base, uint32_t x, int slab) {
        for (; slab < a.n_slabs; slab += 8 * groups) {
            uint32_t v[8];
            eight_slabs(base, slab, v);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                x |= v[i];
        }
        return x;
    };

    // rows
    int32_t *const rows = kk + (int64_t)t * a.K;
    int k_kept = 0;
    for (int base = 0; base < a.K; base += kListThreads * 16) { // sixteen rows a thread at a time
        const int run = rows_per_thread(base);
        const int first = base + tid * run;
        if (base > 0)
            f = flags_of(base);
        uint32_t bits = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            bits |= (f[i >> 2] >> (i & 3) * 8 & 1u) << i;
        bits &= (1u << max(min(run, a.K - first), 0)) - 1u;
        int total;
        int at = k_kept + scan(__popc(bits), total);
        for (; bits; bits &= bits - 1u)
            rows[at++] = first + __ffs(bits) - 1;
        k_kept += total;
    }
    uint32_t cols = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i)
        cols |= v0[i];
    cols = slabs_of(0, cols, (tid >> lg) + 8 * groups);
    unsigned long long nnz = tid < a.n_slabs ? nnz0 : 0u;
    for (int i = tid + kListThreads; i < a.n_slabs; i += kListThreads)
        nnz += a.nnz[(int64_t)t * a.n_slabs + i];
    nnz = wave_scan(nnz);
    if (lane == 63)
        atomicAdd(&s_nnz, nnz);

    // columns: kept where any slab says so
    int n_kept = 0;
    for (int base = 0; base < words; base += kListThreads) {
        const int nw = min(kListThreads, words - base);
        if (base > 0)
            cols = slabs_of(base, 0u, tid >> lg);
        s_cols[tid] = 0;
        __syncthreads();
        if (cj < nw && cols)
            atomicOr(&s_cols[cj], cols);
        __syncthreads();
        const int here = min(max(w - (base + tid) * 4, 0), 4); // columns of this word (what lies behind them was not written)
        const uint32_t x = (tid < nw ? s_cols[tid] : 0u) & (uint32_t)((1ull << (here * 8)) - 1ull);
        int total;
        int at = n_kept + scan(__popc(x), total);
        const int col = (base + tid) * 4;
        int pruned = col - at; // pruned columns before this word
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (tid >= nw || col + e >= w)
                break;
            if (x >> (e * 8) & 0xFFu)
                kn[c0 + at++] = col + e;
            else
                pn[c0 + pruned++] = col + e;
        }
        n_kept += total;
    }
    if (tid < 4) {
        const uint32_t v = tid == 0 ? (uint32_t)k_kept : tid == 1 ? (uint32_t)n_kept : tid == 2 ? (uint32_t)s_nnz : (uint32_t)(s_nnz >> 32);
        reinterpret_cast<volatile TileCounts *>(counts)[t].word[tid] = (unsigned long long)stamp << 32 | v;
    }
}

// ---------------------------------------------------------------------------------

static int round_up(int v, int m) { return (v + m - 1) / m * m; }

// Device memory of plans and of builds.  The runtime maps and unmaps pieces of more than a megabyte anew (25 us for a hipMalloc of 4 MB,
// 20 - 240 for its hipFree), and hipFree waits for the device whatever the size: a program that replaces its plans and has
// products of the new ones on their way stood there until they had run (14 VGG16 layers, masks, plans and first products
// 1066 us a pass with pieces of up to a megabyte left to the runtime, 912 this way).  So they are kept here when they are given back, up to
// kPoolBytes and kPoolPieces a process, and go to the next that asks for about as much on that device; at a bound the oldest are freed (a
// quarter of the pieces at a time: the first of those frees waits for the device), and all
// of it when an allocation fails or the host program asks for it (tw_release_memory).  Kernels of a plan that is destroyed may still be queued, on any
// stream or in a graph: its piece is handed out again only behind a wait for the whole device, made by
// the build that takes it (a build waits anyway) and not by the destruction, which may come in the
// middle of a stream capture.  Nor may that wait be hipDeviceSynchronize: it ends every capture under way
// in the process, whichever thread and mode it was begun in, and another thread may be capturing while
// this one builds.  hipFree waits for the device as well, by contract, and leaves the captures of other
// threads (and relaxed ones) alone, so the wait is the freeing of a small piece.
constexpr size_t kPoolBytes = 256u << 20, kPoolPieces = 512;
class DevicePool {
public:
    void *get(size_t bytes, int device)
    {
        {
            std::unique_lock<std::mutex> lock(mu_);
            size_t best = free_.size();
            for (size_t i = 0; i < free_.size(); ++i)
                if (free_[i].device == device && free_[i].bytes >= bytes && free_[i].bytes <= 2 * bytes &&
                    (best == free_.size() || free_[i].bytes < free_[best].bytes))
                    best = i;
            if (best < free_.size()) {
                const Piece p = free_[best];
                free_.erase(free_.begin() + best);
                held_ -= p.bytes;
                used_[p.ptr] = p.bytes;
                if (p.idle)
                    return p.ptr;
                const unsigned long long before = ++waits_;
                lock.unlock();
                const bool waited = wait_for_device();
                lock.lock();
                if (waited) {
                    for (Piece &q : free_) // what was given back before that wait
                        q.idle |= q.device == device && q.wait < before;
                    return p.ptr;
                }
                lock.unlock();
                put(p.ptr, device, false); // (a capture forbids to wait)
            }
        }
        void *p = nullptr;
        if (hipMalloc(&p, bytes) != hipSuccess) {
            (void)hipGetLastError();
            drop_all();
            if (hipMalloc(&p, bytes) != hipSuccess)
                return nullptr;
        }
        std::lock_guard<std::mutex> lock(mu_);
        used_[p] = bytes;
        return p;
    }
    // `device` is p's; no kernel uses `p` any more, or (idle == false) what is queued on the device may
    void put(void *p, int device, bool idle)
    {
        if (!p)
            return;
        std::vector<Piece> gone;
        {
            std::lock_guard<std::mutex> lock(mu_);
            auto it = used_.find(p);
            const size_t bytes = it != used_.end() ? it->second : 0;
            if (it != used_.end())
                used_.erase(it);
            if (bytes && bytes <= kPoolBytes) {
                // (the oldest: sizes that nobody asks for again would keep all others out)
                const size_t most = free_.size() < kPoolPieces ? free_.size() : kPoolPieces - kPoolPieces / 4;
                size_t n = 0;
                for (; n < free_.size() && (held_ + bytes > kPoolBytes || free_.size() - n > most); ++n)
                    held_ -= free_[n].bytes;
                gone.assign(free_.begin(), free_.begin() + n);
                free_.erase(free_.begin(), free_.begin() + n);
                free_.push_back(Piece{p, bytes, device, idle, waits_});
                held_ += bytes;
                p = nullptr;
            }
        }
        for (const Piece &q : gone)
            free_now(q.ptr);
        if (p)
            free_now(p);
    }
    // what is kept goes back to the device (hipFree waits for work still queued on a destroyed plan: not
    // under the lock, other threads build and destroy plans meanwhile)
    void drop_all()
    {
        std::vector<Piece> pieces;
        {
            std::lock_guard<std::mutex> lock(mu_);
            pieces.swap(free_);
            held_ = 0;
        }
        for (const Piece &p : pieces)
            free_now(p.ptr);
    }

private:
    // A plan may be destroyed in the middle of a capture, and hipFree in a thread's own mode ends that (or
    // any global one); in relaxed mode it does not.
    static void free_now(void *p)
    {
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        if (hipFree(p) != hipSuccess)
            (void)hipGetLastError();
        (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
    // everything queued on the current device has run; false where a capture forbids to wait
    static bool wait_for_device()
    {
        void *p = nullptr;
        if (hipMalloc(&p, 256) == hipSuccess && hipFree(p) == hipSuccess)
            return true;
        (void)hipGetLastError();
        return false;
    }
    struct Piece {
        void *ptr;
        size_t bytes;
        int device;
        bool idle;
        unsigned long long wait; // waits begun before it was given back
    };
    std::mutex mu_;
    std::vector<Piece> free_;
    std::map<void *, size_t> used_;
    size_t held_ = 0;
    unsigned long long waits_ = 0;
};
// (never destroyed: plans may be, by a host program's own destructors, after the library's)
static DevicePool &device_pool()
{
    static DevicePool *const pool = new DevicePool;
    return *pool;
}

// Pinned host memory of a build, on a list of a few pieces between builds.
class PinnedPool {
public:
    void *get(size_t bytes, size_t *size)
    {
        {
            std::lock_guard<std::mutex> lock(mu_);
            for (size_t i = 0; i < free_.size(); ++i)
                if (free_[i].second >= bytes) {
                    const auto p = free_[i];
                    free_.erase(free_.begin() + i);
                    *size = p.second;
                    return p.first;
                }
        }
        void *p = nullptr;
        *size = std::max<size_t>(bytes, 64 << 10);
        if (hipHostMalloc(&p, *size, hipHostMallocPortable) == hipSuccess)
            return p;
        (void)hipGetLastError(); // (or the next call's check of its launches would find it)
        return nullptr;
    }
    void put(void *p, size_t size)
    {
        if (!p)
            return;
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (size <= (1u << 20) && free_.size() < 8) {
                free_.emplace_back(p, size);
                return;
            }
        }
        (void)hipHostFree(p);
    }
    void drop_all()
    {
        std::vector<std::pair<void *, size_t>> pieces;
        {
            std::lock_guard<std::mutex> lock(mu_);
            pieces.swap(free_);
        }
        for (const auto &p : pieces)
            (void)hipHostFree(p.first);
    }

private:
    std::mutex mu_;
    std::vector<std::pair<void *, size_t>> free_;
};
static PinnedPool &pinned_pool()
{
    static PinnedPool *const pool = new PinnedPool;
    return *pool;
}

static void free_plan(tw_plan *p)
{
    if (!p)
        return;
    device_pool().put(p->d_slab, p->device, false);
    delete p;
}

// Owners of what a builder holds until it succeeds: whatever path leaves the builder (an error
// return, an exception on its way to the status conversion), its buffers and the half-built plan are
// released.  The stream of a build is waited for first: its kernels use them.
struct DeviceBuffer {
    void *ptr = nullptr;
    int device = 0;
    DeviceBuffer() = default;
    DeviceBuffer(const DeviceBuffer &) = delete;
    DeviceBuffer &operator=(const DeviceBuffer &) = delete;
    ~DeviceBuffer()
    {
        device_pool().put(ptr, device, true);
    }
    bool get(size_t bytes, int dev)
    {
        device = dev;
        ptr = device_pool().get(bytes, dev);
        return ptr != nullptr;
    }
};
struct PinnedBuffer {
    void *ptr = nullptr;
    size_t size = 0;
    PinnedBuffer() = default;
    PinnedBuffer(const PinnedBuffer &) = delete;
    PinnedBuffer &operator=(const PinnedBuffer &) = delete;
    ~PinnedBuffer()
    {
        pinned_pool().put(ptr, size);
    }
    bool get(size_t bytes)
    {
        ptr = pinned_pool().get(bytes, &size);
        return ptr != nullptr;
    }
};
struct StreamWait { // declared behind the buffers it protects
    hipStream_t s;
    bool done = false;
    ~StreamWait()
    {
        if (!done)
            (void)hipStreamSynchronize(s);
    }
};
struct PlanOwner {
    tw_plan *p = nullptr;
    PlanOwner() = default;
    PlanOwner(const PlanOwner &) = delete;
    PlanOwner &operator=(const PlanOwner &) = delete;
    ~PlanOwner()
    {
        if (p)
            free_plan(p);
    }
    tw_plan *release()
    {
        tw_plan *r = p;
        p = nullptr;
        return r;
    }
};

// What a plan is made from besides its counts (kept_k_ptr, kept_n_ptr): lists in device memory (tile
// t's kept rows at kk + kk_src[t], and so on) and one of the two forms of the weight.
struct PlanSource {
    const int32_t *kk = nullptr, *kn = nullptr, *pn = nullptr;
    std::vector<int64_t> kk_src, kn_src, pn_src;
    const float *B = nullptr;
    const uint8_t *mask = nullptr;
    const uint16_t *Bs = nullptr;
    const int64_t *off_B = nullptr;
};

// Lays out a plan whose tile table and counts are set, and builds everything it owns on the device
// with one launch on `s`; returns when that has run.
static int build_plan(tw_plan *p, const PlanSource &src, hipStream_t s)
{
    const int dst = prepare_device();
    if (dst != TW_OK)
        return dst;
    TW_HIP(hipGetDevice(&p->device));
    const int nt = p->n_tiles;
    p->k_pad.assign(nt, 0);
    p->n_pad.assign(nt, 0);
    p->b_off.assign(nt, 0);
    int64_t off = 0, kkp = 0, groups = 1, longest_list = 1;
    int32_t n_pruned = 0;
    std::vector<UnitDev> &units = p->h_units;
    std::vector<TileDev> ztiles;
    std::vector<PlanTile> tiles(nt);
    units.clear();
    p->max_unit_n = 0;
    p->n_halves = 0;
    for (int t = 0; t < nt; ++t) {
        const int kt = p->kept_k_ptr[t + 1] - p->kept_k_ptr[t];
        const int ntk = p->kept_n_ptr[t + 1] - p->kept_n_ptr[t];
        p->k_pad[t] = ntk > 0 ? round_up(kt, kBlockK) : 0;
        p->n_pad[t] = kt > 0 ? round_up(ntk, kMfmaN) : 0;
        if (p->k_pad[t] == 0 || p->n_pad[t] == 0) {
            // nothing to multiply; kept columns (if any) still receive alpha*0 + beta*C
            p->k_pad[t] = 0;
            p->n_pad[t] = ntk > 0 ? round_up(ntk, kMfmaN) : 0;
        }
        PlanTile &q = tiles[t];
        std::memset(&q, 0, sizeof(q));
        q.col0 = p->tile_col0[t];
        q.k_kept = kt;
        q.n_kept = ntk;
        q.k_pad = p->k_pad[t];
        q.n_pad = p->n_pad[t];
        q.n_pruned = p->tile_width[t] - ntk;
        q.kk_dst = p->kept_k_ptr[t];
        q.kn_dst = p->kept_n_ptr[t];
        q.pn_dst = n_pruned;
        // the padded list: the kernels prefetch it up to eight 64-row steps ahead
        q.kkp_dst = (int32_t)kkp;
        q.kkp_len = p->k_pad[t] + 8 * kBlockK;
        q.kk_src = src.kk_src[t];
        q.kn_src = src.kn_src[t];
        q.pn_src = src.pn_src[t];
        q.src_off = src.off_B ? src.off_B[t] : 0;
        kkp += q.kkp_len;
        longest_list = std::max<int64_t>(longest_list, std::max(q.kkp_len, p->tile_width[t]));
        q.b_off = p->b_off[t] = off; // (a multiple of 64 x 32 elements: every tile is 1 KiB aligned)
        off += (int64_t)p->k_pad[t] * p->n_pad[t];
        groups = std::max<int64_t>(groups, (int64_t)p->k_pad[t] * p->n_pad[t] / 8);
        for (int nc0 = 0; nc0 < ntk; nc0 += kMaxUnitN) {
            UnitDev u;
            u.col0 = p->tile_col0[t];
            u.k_kept = kt;
            u.k_pad = p->k_pad[t];
            u.n_cnt = std::min(kMaxUnitN, ntk - nc0);
            u.nb0 = nc0 / kMfmaN;
            u.nb_cnt = (u.n_cnt + kMfmaN - 1) / kMfmaN;
            u.kk_off = q.kkp_dst;
            u.kn_off = p->kept_n_ptr[t] + nc0;
            u.b_off = p->b_off[t];
            u.tile = t;
            u.nblk = p->n_pad[t] / kMfmaN;
            units.push_back(u);
            p->max_unit_n = std::max(p->max_unit_n, u.n_cnt);
            p->n_halves += (u.n_cnt + 63) / 64;
        }
        if (q.n_pruned > 0) {
            TileDev z;
            z.col0 = p->tile_col0[t];
            z.n_pruned = q.n_pruned;
            z.pn_off = n_pruned;
            z.pad_ = 0;
            ztiles.push_back(z);
            n_pruned += q.n_pruned;
        }
    }
    if (kkp > INT32_MAX)
        return fail(TW_ERR_SHAPE, "the plan keeps %lld rows in all its tiles: at most 2^31 - 1", (long long)kkp);
    // work queue order: heaviest kept-K first, ties keep a tile's pieces adjacent
    std::stable_sort(units.begin(), units.end(),
                     [](const UnitDev &a, const UnitDev &b) { return a.k_kept > b.k_kept; });
    p->packed_elems = off;
    p->n_units = (int)units.size();
    p->n_pipe_units = 0;
    for (const UnitDev &u : units)
        p->n_pipe_units += u.k_pad > 0;
    // nearly dense: kept rows summed over the tiles that keep any, against all K rows for each of
    // those tiles (a tile pruned away whole takes no part on either side)
    int64_t tiles_with_rows = 0;
    for (int t = 0; t < nt; ++t)
        tiles_with_rows += p->kept_k_ptr[t + 1] > p->kept_k_ptr[t];
    p->rows_shared = tiles_with_rows > 1 && p->n_pipe_units > 0 &&
                     (int64_t)p->kept_k_ptr[nt] * 10 >= (int64_t)p->K * tiles_with_rows * 9;
    p->n_zero_tiles = (int)ztiles.size();
    p->max_k_pad = 0;
    p->pipe_steps = 0;
    for (const UnitDev &u : units) {
        p->max_k_pad = std::max(p->max_k_pad, u.k_pad);
        p->pipe_steps += u.k_pad / kBlockK;
    }
    p->n_blocks = 0;
    p->blocks_per_unit = units.empty() ? 0 : units[0].nb_cnt;
    for (const UnitDev &u : units) {
        p->n_blocks += u.nb_cnt;
        if (u.nb_cnt != p->blocks_per_unit)
            p->blocks_per_unit = 0;
    }

    // One device allocation for everything the plan owns: the tables the host makes (one copy), then
    // what the kernel writes.
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    size_t at = 0;
    auto place = [&](size_t bytes) { // returns the 256-aligned offset
        const size_t o = at;
        at = up(at + std::max<size_t>(bytes, 4));
        return o;
    };
    const size_t o_units = place(units.size() * sizeof(UnitDev));
    const size_t o_ztiles = place(ztiles.size() * sizeof(TileDev));
    const size_t o_tiles = place(tiles.size() * sizeof(PlanTile));
    const size_t o_blocks = place(p->n_blocks * sizeof(int32_t));
    const size_t header_bytes = at;
    const size_t sk = p->kept_k_ptr[nt], sn = p->kept_n_ptr[nt];
    const size_t o_kk = place(sk * sizeof(int32_t)), o_rk = place(sk * sizeof(int32_t));
    const size_t o_kn = place(sn * sizeof(int32_t)), o_rn = place(sn * sizeof(int32_t));
    const size_t o_pruned = place(n_pruned * sizeof(int32_t));
    const size_t o_kkpad = place(kkp * sizeof(int32_t));
    const bool pairs = p->K < 0xFFFF;
    const size_t o_pairs = place(pairs ? kkp / 2 * sizeof(uint32_t) : 0);
    const int ticket_words = kTicketInts * (kTicketSlots + 1); // (the last: status words)
    const size_t o_tickets = place(ticket_words * sizeof(int32_t));
    at = (at + 1023) / 1024 * 1024;
    const size_t o_bp = place((size_t)std::max<int64_t>(p->packed_elems, 8) * 2);

    PinnedBuffer header;
    if (!header.get(header_bytes))
        return fail(TW_ERR_ALLOC, "hipHostMalloc of %zu bytes for the plan's tables failed", header_bytes);
    p->d_slab = device_pool().get(at, p->device);
    if (!p->d_slab)
        return fail(TW_ERR_ALLOC, "hipMalloc of %zu bytes for the plan failed", at);
    char *const slab = static_cast<char *>(p->d_slab), *const host = static_cast<char *>(header.ptr);
    std::memcpy(host + o_units, units.data(), units.size() * sizeof(UnitDev));
    std::memcpy(host + o_ztiles, ztiles.data(), ztiles.size() * sizeof(TileDev));
    std::memcpy(host + o_tiles, tiles.data(), tiles.size() * sizeof(PlanTile));
    int32_t *blocks = reinterpret_cast<int32_t *>(host + o_blocks);
    for (size_t ui = 0; ui < units.size(); ++ui)
        for (int nb = 0; nb < units[ui].nb_cnt; ++nb)
            *blocks++ = (int32_t)ui * 4 + nb;

    p->d_units = reinterpret_cast<UnitDev *>(slab + o_units);
    p->d_tiles = reinterpret_cast<TileDev *>(slab + o_ztiles);
    p->d_plan_tiles = slab + o_tiles;
    p->d_blocks = reinterpret_cast<int32_t *>(slab + o_blocks);
    p->d_kept_k = reinterpret_cast<int32_t *>(slab + o_kk);
    p->d_rel_k = reinterpret_cast<int32_t *>(slab + o_rk);
    p->d_kept_n = reinterpret_cast<int32_t *>(slab + o_kn);
    p->d_rel_n = reinterpret_cast<int32_t *>(slab + o_rn);
    p->d_pruned_n = reinterpret_cast<int32_t *>(slab + o_pruned);
    p->d_kept_k_pad = reinterpret_cast<int32_t *>(slab + o_kkpad);
    p->d_kept_pairs = pairs ? reinterpret_cast<uint32_t *>(slab + o_pairs) : nullptr;
    p->d_tickets = reinterpret_cast<int32_t *>(slab + o_tickets);
    p->d_Bp = slab + o_bp;

    BuildArgs a;
    a.n_tiles = nt;
    a.K = p->K;
    a.N = p->N;
    a.dtype = p->dtype;
    a.kk = src.kk;
    a.kn = src.kn;
    a.pn = src.pn;
    a.B = src.B;
    a.Bs = src.Bs;
    a.mask = src.mask;
    a.header = reinterpret_cast<const uint4 *>(host);
    a.header_dst = reinterpret_cast<uint4 *>(slab);
    a.kept_k = p->d_kept_k;
    a.rel_k = p->d_rel_k;
    a.kept_n = p->d_kept_n;
    a.rel_n = p->d_rel_n;
    a.pruned_n = p->d_pruned_n;
    a.kept_k_pad = p->d_kept_k_pad;
    a.kept_pairs = p->d_kept_pairs;
    a.tickets = p->d_tickets;
    a.Bp = static_cast<uint16_t *>(p->d_Bp);
    a.header_chunks = (int32_t)(header_bytes / 16);
    a.ticket_words = ticket_words;
    const unsigned gl = (unsigned)std::min<int64_t>((longest_list + 1023) / 1024, 1024);
    const unsigned gp = (unsigned)std::min<int64_t>((groups + 255) / 256, 4096);
    StreamWait wait{s};
    auto launch_rows = [&](unsigned gx, int begin, int end) { // (kMaxTileRows rows of a grid at a time)
        for (a.row0 = begin; a.row0 < end; a.row0 += kMaxTileRows)
            hipLaunchKernelGGL(plan_build_kernel, dim3(gx, std::min(end - a.row0, kMaxTileRows)), dim3(256), 0, s, a);
    };
    if (nt <= kArgTiles) {
        a.tiles = nullptr;
        std::memcpy(a.arg_tiles, tiles.data(), tiles.size() * sizeof(PlanTile));
        launch_rows(std::max(gl, gp), 0, 2 * nt + 1);
    } else {
        a.tiles = reinterpret_cast<const PlanTile *>(host + o_tiles);
        launch_rows(gl, nt, 2 * nt + 1);
        a.tiles = static_cast<const PlanTile *>(p->d_plan_tiles);
        launch_rows(gp, 0, nt);
    }
    TW_HIP(hipGetLastError());
    {
        // the CU count of a device does not change: ask once per device
        static std::mutex mu;
        static std::vector<int> cu_of;
        std::lock_guard<std::mutex> lock(mu);
        if ((int)cu_of.size() <= p->device)
            cu_of.resize(p->device + 1, 0);
        if (cu_of[p->device] == 0) {
            int n = 0;
            TW_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, p->device));
            cu_of[p->device] = n;
        }
        p->cu_count = cu_of[p->device];
    }
    const hipError_t e = hipStreamSynchronize(s);
    wait.done = true;
    if (e != hipSuccess)
        return fail(TW_ERR_DEVICE, "building the plan on the device failed: %s", hipGetErrorString(e));
    return TW_OK;
}

// The same from lists in host memory (tile t's kept rows kept_k_idx[kept_k_ptr[t] ..], likewise the
// columns), which are uploaded first.
static int build_plan_from_host_lists(tw_plan *p, const int32_t *kept_k_idx, const int32_t *kept_n_idx, PlanSource &src,
                                      hipStream_t s)
{
    const int nt = p->n_tiles;
    const size_t sk = p->kept_k_ptr[nt], sn = p->kept_n_ptr[nt];
    std::vector<int32_t> lists; // kept rows, kept columns, pruned columns
    lists.reserve(sk + p->N);
    lists.insert(lists.end(), kept_k_idx, kept_k_idx + sk);
    lists.insert(lists.end(), kept_n_idx, kept_n_idx + sn);
    src.kk_src.resize(nt);
    src.kn_src.resize(nt);
    src.pn_src.resize(nt);
    for (int t = 0; t < nt; ++t) {
        src.kk_src[t] = p->kept_k_ptr[t];
        src.kn_src[t] = p->kept_n_ptr[t];
        src.pn_src[t] = (int64_t)(lists.size() - sk - sn);
        int j = p->kept_n_ptr[t];
        for (int c = 0; c < p->tile_width[t]; ++c) {
            if (j < p->kept_n_ptr[t + 1] && kept_n_idx[j] == c)
                ++j;
            else
                lists.push_back(c);
        }
    }
    int dev = -1;
    TW_HIP(hipGetDevice(&dev));
    DeviceBuffer d_lists;
    const size_t bytes = std::max<size_t>(lists.size(), 1) * sizeof(int32_t);
    if (!d_lists.get(bytes, dev))
        return fail(TW_ERR_ALLOC, "hipMalloc of %zu bytes for the plan's lists failed", bytes);
    src.kk = static_cast<const int32_t *>(d_lists.ptr);
    src.kn = src.kk + sk;
    src.pn = src.kn + sn;
    if (!lists.empty())
        TW_HIP(hipMemcpy(d_lists.ptr, lists.data(), lists.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    return build_plan(p, src, s);
}

static int unpack_to_stream(const tw_plan *p, uint16_t *d_Bs, hipStream_t s)
{
    TW_HIP(hipMemsetAsync(d_Bs, 0, (size_t)p->K * p->N * 2, s));
    int64_t mg = 0;
    for (int t = 0; t < p->n_tiles; ++t)
        mg = std::max<int64_t>(mg, (int64_t)p->k_pad[t] * p->n_pad[t] / 8);
    if (mg > 0) {
        for (int t0 = 0; t0 < p->n_tiles; t0 += kMaxTileRows)
            hipLaunchKernelGGL(unpack_stream_kernel, dim3((unsigned)((mg + 255) / 256), std::min(p->n_tiles - t0, kMaxTileRows)),
                               dim3(256), 0, s, static_cast<const PlanTile *>(p->d_plan_tiles) + t0, (const uint16_t *)p->d_Bp,
                               p->K, d_Bs);
        TW_HIP(hipGetLastError());
    }
    TW_HIP(hipStreamSynchronize(s));
    return TW_OK;
}

static int check_dtype(int dtype)
{
    if (dtype != TW_F16 && dtype != TW_BF16)
        return fail(TW_ERR_DTYPE, "dtype %d is neither TW_F16 nor TW_BF16", dtype);
    return TW_OK;
}

} // namespace tw

using namespace tw;

extern "C" {

int tw_plan_create(int K, int N, int dtype, int n_tiles, const int32_t *tile_col0,
                   const int32_t *tile_width, const int32_t *kept_k_ptr, const int32_t *kept_k_idx,
                   const int32_t *kept_n_ptr, const int32_t *kept_n_idx, const float *B,
                   tw_plan **out)
try {
    if (!out)
        return fail(TW_ERR_NULL, "out is NULL");
    *out = nullptr;
    int st = check_dtype(dtype);
    if (st)
        return st;
    st = validate_lists(K, N, n_tiles, tile_col0, tile_width, kept_k_ptr, kept_k_idx, kept_n_ptr,
                        kept_n_idx);
    if (st)
        return st;
    if (!B)
        return fail(TW_ERR_NULL, "B is NULL");
    PlanOwner owner;
    tw_plan *p = owner.p = new (std::nothrow) tw_plan;
    if (!p)
        return fail(TW_ERR_ALLOC, "out of host memory");
    p->K = K;
    p->N = N;
    p->dtype = dtype;
    p->n_tiles = n_tiles;
    p->tile_col0.assign(tile_col0, tile_col0 + n_tiles);
    p->tile_width.assign(tile_width, tile_width + n_tiles);
    p->kept_k_ptr.assign(kept_k_ptr, kept_k_ptr + n_tiles + 1);
    p->kept_n_ptr.assign(kept_n_ptr, kept_n_ptr + n_tiles + 1);
    int dev = -1;
    TW_HIP(hipGetDevice(&dev));
    DeviceBuffer d_B;
    const size_t bytes = (size_t)K * N * sizeof(float);
    if (!d_B.get(bytes, dev))
        return fail(TW_ERR_ALLOC, "hipMalloc of %zu bytes for the weight upload failed", bytes);
    TW_HIP(hipMemcpy(d_B.ptr, B, bytes, hipMemcpyHostToDevice));
    PlanSource src;
    src.B = static_cast<const float *>(d_B.ptr);
    st = build_plan_from_host_lists(p, kept_k_idx, kept_n_idx, src, nullptr);
    if (st)
        return st;
    *out = owner.release();
    return TW_OK;
}
TW_CATCH_TO_STATUS

int tw_plan_create_dense(int K, int N, int G, int dtype, const float *B, tw_plan **out)
try {
    if (!out)
        return fail(TW_ERR_NULL, "out is NULL");
    *out = nullptr;
    if (K <= 0 || N <= 0 || G <= 0)
        return fail(TW_ERR_SHAPE, "K=%d N=%d G=%d must all be positive", K, N, G);
    const int nt = (N + G - 1) / G;
    std::vector<int32_t> col0(nt), width(nt), kp(nt + 1), np(nt + 1), ki, ni;
    ki.reserve((size_t)nt * K);
    ni.reserve(N);
    kp[0] = np[0] = 0;
    for (int t = 0; t < nt; ++t) {
        col0[t] = t * G;
        width[t] = std::min(G, N - t * G);
        for (int k = 0; k < K; ++k)
            ki.push_back(k);
        for (int c = 0; c < width[t]; ++c)
            ni.push_back(c);
        kp[t + 1] = (int32_t)ki.size();
        np[t + 1] = (int32_t)ni.size();
    }
    return tw_plan_create(K, N, dtype, nt, col0.data(), width.data(), kp.data(), ki.data(),
                          np.data(), ni.data(), B, out);
}
TW_CATCH_TO_STATUS

int tw_plan_from_mask(int K, int N, int G, int dtype, const uint8_t *mask, const float *B,
                      tw_plan **out)
try {
    if (!out)
        return fail(TW_ERR_NULL, "out is NULL");
    *out = nullptr;
    if (K <= 0 || N <= 0 || G <= 0)
        return fail(TW_ERR_SHAPE, "K=%d N=%d G=%d must all be positive", K, N, G);
    const int nt = (N + G - 1) / G;
    std::vector<int32_t> col0(nt), width(nt);
    for (int t = 0; t < nt; ++t) {
        col0[t] = t * G;
        width[t] = std::min(G, N - t * G);
    }
    return tw_plan_from_mask_tiles(K, N, dtype, nt, col0.data(), width.data(), mask, B, out);
}
TW_CATCH_TO_STATUS

// The pre-pass on device operands: d_mask is K x N bytes, d_B the fp32 weight, both row-major in
// device memory.  Temporaries (flags, counters, the tile table) share one allocation.
static int plan_from_device_mask(int K, int N, int dtype, int n_tiles, const int32_t *tile_col0,
                                 const int32_t *tile_width, const uint8_t *d_mask, const float *d_B,
                                 bool cover, hipStream_t s, tw_plan **out)
{
    if (!out)
        return fail(TW_ERR_NULL, "out is NULL");
    *out = nullptr;
    int st = check_dtype(dtype);
    if (st)
        return st;
    if (K <= 0 || N <= 0 || n_tiles <= 0)
        return fail(TW_ERR_SHAPE, "K=%d N=%d n_tiles=%d must all be positive", K, N, n_tiles);
    if (!d_mask || !d_B || !tile_col0 || !tile_width)
        return fail(TW_ERR_NULL, "mask, B or the tile table is NULL");
    const int nt = n_tiles;
    std::vector<int32_t> tcol0(nt + 1);
    {
        int c = 0;
        for (int t = 0; t < nt; ++t) {
            if (tile_col0[t] != c || tile_width[t] <= 0)
                return fail(TW_ERR_TILE_TABLE,
                            "tile %d: col0=%d width=%d, tiles must cover [0,N) in order without gaps",
                            t, tile_col0[t], tile_width[t]);
            tcol0[t] = c;
            c += tile_width[t];
        }
        if (c != N)
            return fail(TW_ERR_TILE_TABLE, "tiles cover %d columns, N=%d", c, N);
        tcol0[nt] = N;
    }

    // one allocation for all temporaries, carved at 256-byte boundaries
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    const int n_slabs = (K + kFlagRows - 1) / kFlagRows;
    const size_t o_rowflag = 0;
    const size_t o_colpart = o_rowflag + up((size_t)nt * K);
    const size_t o_nnz = o_colpart + up((size_t)(N + 3 * nt + 4) * n_slabs);
    const size_t o_kk = o_nnz + up(sizeof(uint32_t) * nt * n_slabs);
    const size_t o_kn = o_kk + up(sizeof(int32_t) * nt * K);
    const size_t o_pn = o_kn + up(sizeof(int32_t) * N);
    const size_t ws_bytes = o_pn + up(sizeof(int32_t) * N);
    int dev = -1;
    TW_HIP(hipGetDevice(&dev));
    // the workspace and the half-built plan are released on every way out of this function;
    // every kernel and copy runs on the caller's stream, which this function waits for
    DeviceBuffer ws_owner;
    PinnedBuffer pinned; // the counts, then the tile table
    PlanOwner owner;
    const size_t counts_bytes = up(sizeof(TileCounts) * nt);
    if (!ws_owner.get(ws_bytes, dev) || !pinned.get(counts_bytes + sizeof(int32_t) * (nt + 1)))
        return fail(TW_ERR_ALLOC, "allocation of %zu bytes for the pre-pass failed", ws_bytes);
    char *const ws = static_cast<char *>(ws_owner.ptr);
    volatile TileCounts *const counts = static_cast<volatile TileCounts *>(pinned.ptr);
    int32_t *const h_tcol0 = reinterpret_cast<int32_t *>(static_cast<char *>(pinned.ptr) + counts_bytes);
    FlagArgs fa;
    fa.tcol0 = nt <= kFlagArgTiles ? nullptr : h_tcol0;
    std::memcpy(nt <= kFlagArgTiles ? fa.arg_tcol0 : h_tcol0, tcol0.data(), sizeof(int32_t) * (nt + 1));
    // (never 0, and another number for every build, so that a stamp an earlier build left is not taken for this one's)
    static std::atomic<uint32_t> builds{0};
    uint32_t stamp = ++builds;
    if (stamp == 0)
        stamp = ++builds;
    for (int t = 0; t < nt; ++t)
        for (int i = 0; i < 4; ++i)
            counts[t].word[i] = 0;
    fa.mask = d_mask;
    fa.K = K;
    fa.N = N;
    fa.n_slabs = n_slabs;
    fa.rowflag = reinterpret_cast<uint8_t *>(ws + o_rowflag);
    fa.colpart = reinterpret_cast<uint8_t *>(ws + o_colpart);
    fa.nnz = reinterpret_cast<uint32_t *>(ws + o_nnz);
    int32_t *const kk = reinterpret_cast<int32_t *>(ws + o_kk);
    int32_t *const kn = reinterpret_cast<int32_t *>(ws + o_kn);
    int32_t *const pn = reinterpret_cast<int32_t *>(ws + o_pn);
    StreamWait wait{s};
    for (fa.tile0 = 0; fa.tile0 < nt; fa.tile0 += kMaxTileRows)
        hipLaunchKernelGGL(mask_flags_kernel, dim3(n_slabs, std::min(nt - fa.tile0, kMaxTileRows)), dim3(256), 0, s, fa);
    hipLaunchKernelGGL(mask_lists_kernel, dim3(nt), dim3(kListThreads), 0, s, fa, kk, kn, pn,
                       static_cast<TileCounts *>(pinned.ptr), stamp);
    TW_HIP(hipGetLastError());

    tw_plan *const p = owner.p = new (std::nothrow) tw_plan;
    if (!p)
        return fail(TW_ERR_ALLOC, "out of host memory");
    p->device = dev;
    p->K = K;
    p->N = N;
    p->dtype = dtype;
    p->n_tiles = nt;
    p->tile_col0.assign(tile_col0, tile_col0 + nt);
    p->tile_width.assign(tile_width, tile_width + nt);
    p->kept_k_ptr.assign(nt + 1, 0);
    p->kept_n_ptr.assign(nt + 1, 0);
    PlanSource src;
    src.kk = kk;
    src.kn = kn;
    src.pn = pn;
    src.kk_src.resize(nt);
    src.kn_src.resize(nt);
    src.pn_src.resize(nt);
    // The counts arrive in host memory tile by tile: looked at until they are there, which is some 5 us
    // sooner than the runtime's own wait notices the end of the stream.  The look is bounded by that
    // wait, taken after a while.
    unsigned long long mismatch = 0;
    int64_t sum_k = 0;
    for (int t = 0; t < nt; ++t) {
        uint32_t count[4];
        for (int i = 0; i < 4; ++i) {
            unsigned long long word;
            for (long spin = 0; (word = counts[t].word[i]) >> 32 != stamp; ++spin) {
                if (spin < 200000) {
                    __builtin_ia32_pause();
                    continue;
                }
                TW_HIP(hipStreamSynchronize(s));
                if (counts[t].word[i] >> 32 != stamp)
                    return fail(TW_ERR_DEVICE, "the pre-pass left no counts for tile %d", t);
            }
            count[i] = (uint32_t)word;
        }
        const int32_t rows = (int32_t)count[0], cols = (int32_t)count[1];
        mismatch += (unsigned long long)rows * (unsigned long long)cols - ((unsigned long long)count[3] << 32 | count[2]);
        sum_k += rows;
        p->kept_k_ptr[t + 1] = (int32_t)std::min<int64_t>(sum_k, INT32_MAX);
        p->kept_n_ptr[t + 1] = p->kept_n_ptr[t] + cols;
        src.kk_src[t] = (int64_t)t * K;
        src.kn_src[t] = src.pn_src[t] = tile_col0[t];
    }
    if (sum_k > INT32_MAX)
        return fail(TW_ERR_SHAPE, "K=%d rows in %d tiles are more than the pre-pass indexes", K, nt);
    if (mismatch != 0 && !cover) {
        return fail(TW_ERR_NOT_TW,
                    "%llu mask elements differ from (row kept) & (column kept) of their tile",
                    mismatch);
    }
    // rows and columns of a covering tile are the union of its elements: the elements the mask
    // drops inside that cover are stored as zeros
    src.B = d_B;
    src.mask = mismatch != 0 ? d_mask : nullptr;
    st = build_plan(p, src, s);
    if (st)
        return st;
    wait.done = true; // (the build has waited)
    *out = owner.release();
    return TW_OK;
}

// host operands: one upload buffer for the mask and the weight, then the device pre-pass
static int plan_from_mask_impl(int K, int N, int dtype, int n_tiles, const int32_t *tile_col0,
                               const int32_t *tile_width, const uint8_t *mask, const float *B,
                               bool cover, tw_plan **out)
{
    if (!out)
        return fail(TW_ERR_NULL, "out is NULL");
    *out = nullptr;
    if (int st = check_dtype(dtype))
        return st;
    if (K <= 0 || N <= 0 || n_tiles <= 0)
        return fail(TW_ERR_SHAPE, "K=%d N=%d n_tiles=%d must all be positive", K, N, n_tiles);
    if (!mask || !B || !tile_col0 || !tile_width)
        return fail(TW_ERR_NULL, "mask, B or the tile table is NULL");
    const size_t b_bytes = (size_t)K * N * sizeof(float), m_bytes = (size_t)K * N;
    int dev = -1;
    TW_HIP(hipGetDevice(&dev));
    DeviceBuffer upload_buf;
    if (!upload_buf.get(b_bytes + m_bytes, dev))
        return fail(TW_ERR_ALLOC, "hipMalloc of %zu bytes for the mask and weight upload failed",
                    b_bytes + m_bytes);
    char *const buf = static_cast<char *>(upload_buf.ptr);
    hipError_t e = hipMemcpy(buf, B, b_bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(buf + b_bytes, mask, m_bytes, hipMemcpyHostToDevice);
    return e == hipSuccess
               ? plan_from_device_mask(K, N, dtype, n_tiles, tile_col0, tile_width,
                                       reinterpret_cast<const uint8_t *>(buf + b_bytes),
                                       reinterpret_cast<const float *>(buf), cover, nullptr, out)
               : fail(TW_ERR_DEVICE, "mask / weight upload failed: %s", hipGetErrorString(e));
}

int tw_plan_from_device_mask(int K, int N, int dtype, int n_tiles, const int32_t *tile_col0,
                             const int32_t *tile_width, const uint8_t *mask, const float *B,
                             int cover, void *stream, tw_plan **out)
try {
    return plan_from_device_mask(K, N, dtype, n_tiles, tile_col0, tile_width, mask, B, cover != 0,
                                 (hipStream_t)stream, out);
}
TW_CATCH_TO_STATUS

int tw_plan_from_mask_tiles(int K, int N, int dtype, int n_tiles, const int32_t *tile_col0,
                            const int32_t *tile_width, const uint8_t *mask, const float *B,
                            tw_plan **out)
try {
    return plan_from_mask_impl(K, N, dtype, n_tiles, tile_col0, tile_width, mask, B, false, out);
}
TW_CATCH_TO_STATUS

int tw_plan_from_mask_cover(int K, int N, int dtype, int n_tiles, const int32_t *tile_col0,
                            const int32_t *tile_width, const uint8_t *mask, const float *B,
                            tw_plan **out)
try {
    return plan_from_mask_impl(K, N, dtype, n_tiles, tile_col0, tile_width, mask, B, true, out);
}
TW_CATCH_TO_STATUS

int tw_plan_from_export(int K, int N, int dtype, int n_kept_k, const int32_t *mask_i,
                        int n_kept_n, const int32_t *mask_o, const float *kernel, tw_plan **out)
try {
    if (!out)
        return fail(TW_ERR_NULL, "out is NULL");
    *out = nullptr;
    if (K <= 0 || N <= 0 || n_kept_k < 0 || n_kept_k > K || n_kept_n < 0 || n_kept_n > N)
        return fail(TW_ERR_SHAPE, "K=%d N=%d with %d kept rows and %d kept columns", K, N,
                    n_kept_k, n_kept_n);
    if ((n_kept_k > 0 && !mask_i) || (n_kept_n > 0 && !mask_o) ||
        (n_kept_k > 0 && n_kept_n > 0 && !kernel))
        return fail(TW_ERR_NULL, "mask_i, mask_o or kernel is NULL");
    std::vector<int32_t> kk((size_t)std::max(n_kept_k, 1)), kn((size_t)std::max(n_kept_n, 1));
    int st = tw_offsets_to_kept(mask_i, n_kept_k, K, kk.data());
    if (!st)
        st = tw_offsets_to_kept(mask_o, n_kept_n, N, kn.data());
    if (st)
        return st;
    // one tile over all columns: every unit of 128 compact columns shares the kept rows
    std::vector<float> B((size_t)K * N, 0.0f);
    for (int i = 0; i < n_kept_k; ++i) {
        float *dst = B.data() + (size_t)kk[i] * N;
        const float *src = kernel + (size_t)i * n_kept_n;
        for (int j = 0; j < n_kept_n; ++j)
            dst[kn[j]] = src[j];
    }
    const int32_t col0 = 0, width = N;
    const int32_t kp[2] = {0, n_kept_k}, np[2] = {0, n_kept_n};
    return tw_plan_create(K, N, dtype, 1, &col0, &width, kp, kk.data(), np, kn.data(), B.data(),
                          out);
}
TW_CATCH_TO_STATUS

int tw_plan_from_stream_operands(int M, int N, int K, int dtype, const void *B_stream,
                                 int block_num, const int32_t *N_cal, const int32_t *K_cal,
                                 const int32_t *const *mask_n, const int32_t *const *mask_k,
                                 const int64_t *off_B, const int64_t *off_C, tw_plan **out)
try {
    if (!out)
        return fail(TW_ERR_NULL, "out is NULL");
    *out = nullptr;
    int st = check_dtype(dtype);
    if (st)
        return st;
    if (M <= 0 || N <= 0 || K <= 0 || block_num <= 0)
        return fail(TW_ERR_SHAPE, "M=%d N=%d K=%d block_num=%d must all be positive", M, N, K,
                    block_num);
    if (!B_stream || !N_cal || !K_cal || !mask_n || !mask_k || !off_B || !off_C)
        return fail(TW_ERR_NULL, "an operand pointer is NULL");
    std::vector<int32_t> col0(block_num), width(block_num), kp(block_num + 1, 0),
        np(block_num + 1, 0), ki, ni;
    for (int t = 0; t < block_num; ++t) {
        if (off_C[t] % M != 0)
            return fail(TW_ERR_TILE_TABLE, "off_C[%d] = %lld is not a multiple of M", t,
                        (long long)off_C[t]);
        col0[t] = (int32_t)(off_C[t] / M);
        if (N_cal[t] < 0 || K_cal[t] < 0 || K_cal[t] > K)
            return fail(TW_ERR_SHAPE, "tile %d: N_cal=%d K_cal=%d", t, N_cal[t], K_cal[t]);
        if ((N_cal[t] > 0 && !mask_n[t]) || (K_cal[t] > 0 && !mask_k[t]))
            return fail(TW_ERR_NULL, "mask pointer of tile %d is NULL", t);
    }
    for (int t = 0; t < block_num; ++t) {
        const int next = t + 1 < block_num ? col0[t + 1] : N;
        width[t] = next - col0[t];
        if (width[t] <= 0 || N_cal[t] > width[t])
            return fail(TW_ERR_TILE_TABLE, "tile %d: width %d, N_cal %d", t, width[t], N_cal[t]);
        if (off_B[t] < 0 || off_B[t] + (int64_t)std::max(N_cal[t] - 1, 0) * K + K_cal[t] >
                                (int64_t)K * N)
            return fail(TW_ERR_SHAPE, "off_B[%d] = %lld leaves the K*N weight buffer", t,
                        (long long)off_B[t]);
        std::vector<int32_t> rel_k(K_cal[t]), rel_n(N_cal[t]);
        if (K_cal[t])
            TW_HIP(hipMemcpy(rel_k.data(), mask_k[t], sizeof(int32_t) * K_cal[t],
                             hipMemcpyDeviceToHost));
        if (N_cal[t])
            TW_HIP(hipMemcpy(rel_n.data(), mask_n[t], sizeof(int32_t) * N_cal[t],
                             hipMemcpyDeviceToHost));
        size_t k0 = ki.size(), n0 = ni.size();
        ki.resize(k0 + K_cal[t]);
        ni.resize(n0 + N_cal[t]);
        if ((st = tw_offsets_to_kept(rel_k.data(), K_cal[t], K, ki.data() + k0)) ||
            (st = tw_offsets_to_kept(rel_n.data(), N_cal[t], width[t], ni.data() + n0)))
            return st;
        kp[t + 1] = (int32_t)ki.size();
        np[t + 1] = (int32_t)ni.size();
    }
    st = validate_lists(K, N, block_num, col0.data(), width.data(), kp.data(), ki.data(), np.data(),
                        ni.data());
    if (st)
        return st;
    PlanOwner owner;
    tw_plan *p = owner.p = new (std::nothrow) tw_plan;
    if (!p)
        return fail(TW_ERR_ALLOC, "out of host memory");
    p->K = K;
    p->N = N;
    p->dtype = dtype;
    p->n_tiles = block_num;
    p->tile_col0 = col0;
    p->tile_width = width;
    p->kept_k_ptr = kp;
    p->kept_n_ptr = np;
    PlanSource src;
    src.Bs = static_cast<const uint16_t *>(B_stream);
    src.off_B = off_B;
    st = build_plan_from_host_lists(p, ki.data(), ni.data(), src, nullptr);
    if (st)
        return st;
    *out = owner.release();
    return TW_OK;
}
TW_CATCH_TO_STATUS

int tw_plan_info(const tw_plan *p, int64_t *info, int n_info)
{
    if (!p || !info)
        return fail(TW_ERR_NULL, "plan or info is NULL");
    int64_t v[12] = {0};
    v[0] = p->K;
    v[1] = p->N;
    v[2] = p->dtype;
    v[3] = p->n_tiles;
    for (int t = 0; t < p->n_tiles; ++t) {
        const int64_t kt = p->kept_k_ptr[t + 1] - p->kept_k_ptr[t];
        const int64_t nt = p->kept_n_ptr[t + 1] - p->kept_n_ptr[t];
        v[4] += kt;
        v[5] += nt;
        v[6] += kt * nt;
        v[8] = std::max(v[8], kt);
        v[9] = std::max(v[9], nt);
        v[10] += (kt * nt == 0);
        v[11] += p->tile_width[t];
    }
    v[7] = p->packed_elems * 2;
    for (int i = 0; i < n_info && i < 12; ++i)
        info[i] = v[i];
    return TW_OK;
}

int tw_plan_export(const tw_plan *p, int32_t *tile_col0, int32_t *tile_width, int32_t *kept_k_ptr,
                   int32_t *kept_k_idx, int32_t *mask_k_rel, int32_t *kept_n_ptr,
                   int32_t *kept_n_idx, int32_t *mask_n_rel, uint16_t *B_stream)
try {
    if (!p)
        return fail(TW_ERR_NULL, "plan is NULL");
    const int nt = p->n_tiles;
    if (tile_col0)
        memcpy(tile_col0, p->tile_col0.data(), sizeof(int32_t) * nt);
    if (tile_width)
        memcpy(tile_width, p->tile_width.data(), sizeof(int32_t) * nt);
    if (kept_k_ptr)
        memcpy(kept_k_ptr, p->kept_k_ptr.data(), sizeof(int32_t) * (nt + 1));
    if (kept_n_ptr)
        memcpy(kept_n_ptr, p->kept_n_ptr.data(), sizeof(int32_t) * (nt + 1));
    const size_t sk = p->kept_k_ptr[nt], sn = p->kept_n_ptr[nt];
    // the index lists come back from the device copies the kernels read
    if (kept_k_idx && sk)
        TW_HIP(hipMemcpy(kept_k_idx, p->d_kept_k, sizeof(int32_t) * sk, hipMemcpyDeviceToHost));
    if (mask_k_rel && sk)
        TW_HIP(hipMemcpy(mask_k_rel, p->d_rel_k, sizeof(int32_t) * sk, hipMemcpyDeviceToHost));
    if (kept_n_idx && sn)
        TW_HIP(hipMemcpy(kept_n_idx, p->d_kept_n, sizeof(int32_t) * sn, hipMemcpyDeviceToHost));
    if (mask_n_rel && sn)
        TW_HIP(hipMemcpy(mask_n_rel, p->d_rel_n, sizeof(int32_t) * sn, hipMemcpyDeviceToHost));
    if (B_stream) {
        int dev = -1;
        TW_HIP(hipGetDevice(&dev));
        DeviceBuffer d_Bs;
        const size_t bytes = (size_t)p->K * p->N * 2;
        if (!d_Bs.get(bytes, dev))
            return fail(TW_ERR_ALLOC, "hipMalloc of %zu bytes failed", bytes);
        if (int st = unpack_to_stream(p, static_cast<uint16_t *>(d_Bs.ptr), nullptr))
            return st;
        const hipError_t e = hipMemcpy(B_stream, d_Bs.ptr, bytes, hipMemcpyDeviceToHost);
        if (e != hipSuccess)
            return fail(TW_ERR_DEVICE, "read-back failed: %s", hipGetErrorString(e));
    }
    return TW_OK;
}
TW_CATCH_TO_STATUS

int tw_plan_destroy(tw_plan *plan)
{
    free_plan(plan);
    return TW_OK;
}

int tw_release_memory(void)
try {
    // (another stream, or another thread's, may be under capture)
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    device_pool().drop_all();
    pinned_pool().drop_all();
    release_producer_memory();
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    return TW_OK;
}
TW_CATCH_TO_STATUS

} // extern "C"
