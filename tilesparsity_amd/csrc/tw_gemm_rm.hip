// Row-major streaming kernel of the tile-wise-sparse GEMM: row-major A[M][lda] and C[M][ldc], the operands of the
// reference's Python operator (mask_dense, Pruning/BERT/utils/modeling.py:992-1007), mostly for a K too long for a panel
// of A in LDS.
//
// A kept row k of a tile is one 2-byte element per row m of a row-major A, and at a quarter kept every 64-byte piece of a
// row holds some, so nothing is gained by gathering from memory: a workgroup streams all of its rows of A through LDS, 128
// columns k at a time, and gathers there.  Before this kernel such operands were turned into K-major copies around the
// streaming kernel: three launches, of which the turning alone moved A twice.
//   K 3072, N 768, M 4096, a quarter kept, f16: 31.9 -> 17.0 us a call (the copies of A 11.4 and of C 4.7, the product
//   16.4); K 4608, N 512, M 12544: 82 -> 46; K 2304, N 512, M 16384: 57 -> 37.
// What bounds the first of these: 6300 cycles until the lists are there (arguments, unit, row numbers: trips to memory
// from cold caches, then the lists themselves), 24 chunks at 735 cycles (a wave's chain of about 70 instructions and 8
// MFMAs per record; the loads alone take 430, the multiplying side alone 600), 5000 to add up and store.  (The compiler keeps 53
// to 58 scalar registers of the unit and the arguments in lanes of a vector register across the loop; no scratch memory.)
//
//   work:  a workgroup takes 64 rows m and two units (four of at most 64 columns): with 256 columns the bytes a
//          compute unit fetches (128 K for A, 512 K_t for the weight) are near their least, while 4096 rows of 768 columns
//          still give 192 workgroups.  Four waves multiply, 64 rows x 128 columns each, two of them taking the groups
//          of 16 kept rows of a unit in turn; four waves load.
//   ring:  six chunks of A, [64 rows m][128 columns k], filled with loads that write LDS directly (buffer_load_dwordx4 ...
//          lds: 1 KiB, four rows, each).  The sixteen 16-byte pieces of a row lie in the order p ^ (m % 16), so that the 32
//          rows a read of one column touches fall into sixteen groups of banks instead of one, and rows m and m + 16
//          read the two columns of a pair in opposite order (25.0 -> 21.6 us when that came).
//   lists: the kept rows of a unit as records of 16: the place of each row's column inside the ring (chunk, piece,
//          element: 16 bits), the chunk that has to be there, where the weight is.  A group that spans more than two chunks
//          is cut into several records, the rows of the others named as a chunk of zeros: such a record multiplies what is
//          in the ring at its time.  A lane holds row m = lane % 32 of an MFMA operand and eight kept rows: eight 2-byte
//          LDS reads at place ^ (its own row's bits), for 32 more rows the same addresses plus a constant.
//   meet:  through words in LDS, no barrier in the loop: a loading wave says how far its chunks have landed, a
//          multiplying wave which chunk it is at, which frees the chunks before the one before.  The waves drift apart
//          and use the LDS pipe, the matrix cores and the loads at different times (a barrier per chunk: 21.6 us).  A loading
//          wave has one chunk of its own in flight: four waves that shared every chunk went one chunk at a time, 20.0.
//   sums:  in fp32 in the order of k within each of the two waves of a unit, then one addition: the last bit can differ
//          from the K-major kernels'.
//   output: the product is turned around (weight times A: a lane holds neighbouring columns of a row), the partial
//          products meet in LDS in the ring's place, and all eight waves add them up, finish and store 16-byte pieces of
//          rows where eight compact columns are an aligned octet of C, else element by element.
// Inf and NaN in rows of A that a tile prunes never reach its products: the reads name kept rows and zeros only.
#include "tw_device.h"

#include <algorithm>

namespace tw {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kRmRows = kRmRowsPerWg;         // rows m of a workgroup
constexpr int kRmChunk = 128;                 // columns k of a chunk
constexpr int kRmSlot = kRmRows * kRmChunk * 2; // bytes of a chunk
constexpr int kRmSlots = 6;                   // chunks of the ring; a chunk of zeros behind it
constexpr int kRmKeep = 2;                    // chunks a record of the list may span
constexpr int kRmMulWaves = 4, kRmLoadWaves = 4;
constexpr int kRmThreads = 64 * (kRmMulWaves + kRmLoadWaves);
constexpr int kRmCols = 256;                  // compact columns of a workgroup: two wide units or four narrow ones
constexpr int kRmW = 4;                       // records of weight a multiplying wave has in flight
constexpr int kRmRecord = 48;                 // bytes of a record: 16 places (2 bytes each), its chunk, a weight offset, its rows
constexpr int kRmMaxLds = 160 * 1024;
constexpr int kRmRsrcFlags = 0x00020000;      // word 3 of a raw buffer descriptor of this target

// LDS: column numbers, bias and flags; the ring and its zeros; the lists.  At the end the partial products, [row][column] in
// fp32, take the place of all but the first part.
constexpr int kRmFlags = kRmCols * 8;         // chunks landed (4), chunk at hand (4), lengths of the lists (4); words nobody reads
constexpr int kRmRing = 4096;
static_assert(kRmFlags + 64 + kRmMulWaves * 256 <= kRmRing, "columns, bias and flags fit ahead of the ring");
constexpr int kRmLists = kRmRing + (kRmSlots + 1) * kRmSlot;
constexpr int kRmPitch = kRmCols + 4;         // floats per row of a partial product
constexpr int kRmPart = kRmRows * kRmPitch;   // floats of one
// Units of at most 64 compact columns (`narrow`) have a multiplying wave each; of wider ones two waves share one and
// take its records in turn.
constexpr int rm_turns(bool narrow) { return narrow ? 1 : 2; }
constexpr int rm_units(bool narrow) { return kRmMulWaves / rm_turns(narrow); }
// Records of a list: one per group of 16 kept rows, one more each time a group is cut (at most once per chunk), and what
// the waves look ahead on either side.
__host__ __device__ constexpr int rm_list_records(int k_pad, int n_chunks, bool narrow)
{
    return k_pad / 16 + n_chunks + rm_turns(narrow) * (2 * kRmW + 1);
}
static bool rm_narrow(const tw_plan *plan) { return plan->max_unit_n <= 64; }
static int64_t rm_lds_bytes(const tw_plan *plan)
{
    const bool narrow = rm_narrow(plan);
    return std::max<int64_t>(kRmRing + rm_turns(narrow) * kRmPart * 4,
                             kRmLists + (int64_t)rm_units(narrow) * kRmRecord *
                                            rm_list_records(plan->max_k_pad, (plan->K + kRmChunk - 1) / kRmChunk, narrow));
}

// waits until at most N of the wave's loads are outstanding
template <int N> __device__ __forceinline__ void rm_wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

template <int DT, bool NARROW>
__global__ void __launch_bounds__(kRmThreads, 2)
    tw_gemm_rm_kernel(const GemmArgs p, int k_rows, int n_rowblk, int max_k_pad)
{
    using E = Elem<DT>;
    constexpr int T = rm_turns(NARROW);
    constexpr int CB = NARROW ? 2 : 4;       // 32-column blocks of a unit
    extern __shared__ __align__(1024) unsigned char rm_smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // (the grid is row blocks by groups of units, row blocks fastest: a multiple of eight of them puts the groups of a row
    // block on one die)
    const int rb = blockIdx.x, grp = blockIdx.y;
    if (rb >= n_rowblk)
        return;
    const int m0 = rb * kRmRows;
    const int m_cnt = min(kRmRows, p.M - m0);
    const int n_chunks = (k_rows + kRmChunk - 1) / kRmChunk;
    uint16_t *const C = reinterpret_cast<uint16_t *>(p.C);
    TW_LDS(volatile int) const landed = (TW_LDS(volatile int))(TW_LDS(unsigned char))(rm_smem + kRmFlags);
    TW_LDS(volatile int) const at_hand = landed + 4;
    TW_LDS(volatile int) const n_records = landed + 8;
    int *const col_s = reinterpret_cast<int *>(rm_smem); // columns of C, -1 for those the units do not have
    float *const bias_s = reinterpret_cast<float *>(rm_smem) + kRmCols;
    if (tid < 8)
        landed[tid] = tid < 4 ? tid : 0; // (the first chunk that is not there of each loading wave's)

    if (wave >= kRmMulWaves) {
        // ================= loading waves: a chunk in turn each ==============================
        const int w = wave - kRmMulWaves;
        const int lrow = lane >> 4, pos = lane & 15;
        const uint32_t lda_b = (uint32_t)p.lda * 2u;
        // (what lies past the last row of A, or past its end, arrives as zeros; columns past K are never read)
        const uint32_t a_bytes = (uint32_t)(m_cnt - 1) * lda_b + (uint32_t)((k_rows + 7) / 8) * 16u;
        const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(reinterpret_cast<const char *>(p.A) + (int64_t)m0 * p.lda * 2), 0, (int)a_bytes, kRmRsrcFlags);
        // Load j covers rows 4 j .. 4 j + 3: this lane's piece of row 4 j + lane / 16, j = 0 .. 3; 16 rows on the order
        // of the pieces repeats.
        uint32_t off[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            off[j] = (uint32_t)(j * 4 + lrow) * lda_b + (uint32_t)(pos ^ (j * 4 + lrow)) * 16u + (uint32_t)w * (kRmChunk * 2);
        TW_LDS(unsigned char) const ring = (TW_LDS(unsigned char))(rm_smem + kRmRing);
        bool lists = false;
        for (int c = w; c < n_chunks; c += kRmLoadWaves) {
            if (c >= kRmSlots) {
                // The chunk takes the place of the one kRmSlots back, once no wave needs that any more: a wave at a record
                // of chunk r needs r - kRmKeep + 1 on.
                while (!__all(at_hand[lane & 3] >= c - kRmSlots + kRmKeep))
                    __builtin_amdgcn_s_sleep(1);
            }
            TW_LDS(unsigned char) const dst = ring + c % kRmSlots * kRmSlot;
#pragma unroll
            for (int j = 0; j < kRmRows / 4; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (TW_LDS(void))(dst + j * 1024), 16,
                                                         (int)(off[j & 3] + (uint32_t)(j >> 2) * 16u * lda_b), 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                off[j] += kRmLoadWaves * kRmChunk * 2;
            if (!lists)
                TW_LDS_BARRIER(); // the lists are there, and the flags
            lists = true;
            rm_wait_loads<0>();
            if (lane == 0)
                landed[w] = c + kRmLoadWaves; // (the first of this wave's chunks that is not there)
        }
        if (!lists)
            TW_LDS_BARRIER(); // the lists are there, and the flags
        if (lane == 0)
            landed[w] = 0x7fffffff;
        TW_LDS_BARRIER(); // the ring is read no more
    } else {

    // ================= multiplying waves ====================================================
    const int uq = NARROW ? wave : wave >> 1, turn = NARROW ? 0 : wave & 1;
    const int ui = grp * rm_units(NARROW) + uq;
    UnitDev u{};
    const bool active = ui < p.n_gemm_u;
    if (active) {
        // (whole units: n_split is 1 here, and load_unit's division by it is not cheap)
        const auto *const src = p.n_arg_units ? (const __attribute__((address_space(4))) int32_t *)__builtin_amdgcn_kernarg_segment_ptr() +
                                                    offsetof(GemmArgs, arg_units) / 4 + ui * 12
                                              : (const __attribute__((address_space(4))) int32_t *)(uintptr_t)(p.units + ui);
        int32_t w[12];
#pragma unroll
        for (int i = 0; i < 12; ++i)
            w[i] = __builtin_amdgcn_readfirstlane(src[i]);
        __builtin_memcpy(&u, w, sizeof(UnitDev));
    }
    const int n16 = (u.k_kept + 15) / 16; // groups of 16 kept rows
    // record i of the list, i from -T * kRmW on
    TW_LDS(unsigned char) const list =
        (TW_LDS(unsigned char))(rm_smem + kRmLists) +
        (uq * rm_list_records(max_k_pad, n_chunks, NARROW) + T * kRmW) * kRmRecord;
    const int half16 = lane >> 5, mrow = lane & 31;
    if (turn == 0 && !active && lane == 0)
        n_records[uq] = 0;
    if (active && turn == 0) {
        // ---- the list: a record per group of 16 kept rows, lane by lane; a group that spans more than kRmKeep chunks gets
        // one for every kRmKeep of them, with the zeros' place for the rows of the others.  A record's last words
        // are its own chunk, the weight offset of the record T * kRmW on, and which of its rows are its own.
        constexpr uint32_t kZeros = kRmSlots * (kRmSlot / 2);
        constexpr uint32_t kNoWeight = 0xFFFFF000u; // (beyond the buffer, which delivers zeros)
        const int32_t *const kept = p.kept_k + u.kk_off;
        const uint32_t step_b = (uint32_t)u.nblk * 4096u;
        int n_rec = 0;
        for (int g0 = 0; g0 < n16; g0 += 64) {
            const int g = g0 + lane;
            uint32_t k[16];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int4 v = *reinterpret_cast<const int4 *>(kept + min(g, n16 - 1) * 16 + i * 4);
                k[4 * i] = v.x;
                k[4 * i + 1] = v.y;
                k[4 * i + 2] = v.z;
                k[4 * i + 3] = v.w;
            }
            const int rows = min(16, u.k_kept - g * 16); // (0 or less: no group of this lane's)
            const int first = (int)(k[0] / kRmChunk);
            int last = first;
#pragma unroll
            for (int i = 1; i < 16; ++i)
                last = i < rows ? (int)(k[i] / kRmChunk) : last;
            const int pieces = rows > 0 ? (last - first) / kRmKeep + 1 : 0;
            int before = pieces; // inclusive scan
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int v = __shfl_up(before, d);
                before += lane >= d ? v : 0;
            }
            const int total = __shfl(before, 63);
            for (int j = 0; j < pieces; ++j) {
                // a place: chunk's place in the ring, piece and element of the row, halved to fit 16 bits
                static_assert(kRmKeep == 2, "a record's rows are of two chunks");
                const int lo = first + j * kRmKeep, hi = min(last, lo + 1), slot = lo % kRmSlots;
                const uint32_t p_lo = (uint32_t)slot * (kRmSlot / 2), p_hi = slot + 1 < kRmSlots ? p_lo + kRmSlot / 2 : 0u;
                uint32_t w[8], there = 0;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int ch = (int)(k[i] / kRmChunk);
                    const bool in = i < rows && (ch == lo || ch == hi);
                    const uint32_t place = in ? (ch == lo ? p_lo : p_hi) + k[i] % kRmChunk : kZeros;
                    w[i >> 1] = i & 1 ? w[i >> 1] | place << 16 : place;
                    there |= in ? 1u << i : 0u;
                }
                TW_LDS(unsigned char) const rec = list + (n_rec + before - pieces + j) * kRmRecord;
                *(TW_LDS(u32x4))rec = u32x4{w[0], w[1], w[2], w[3]};
                *(TW_LDS(u32x4))(rec + 16) = u32x4{w[4], w[5], w[6], w[7]};
                *(TW_LDS(uint32_t))(rec + 32) = (uint32_t)hi;
                *(TW_LDS(uint32_t))(rec + 40) = pieces > 1 ? there : 0xFFFFu;
                *(TW_LDS(uint32_t))(rec + 36 - T * kRmW * kRmRecord) = (uint32_t)(g >> 2) * step_b + (uint32_t)(g & 3) * 1024u;
            }
            n_rec += total;
        }
        if (lane < T * (kRmW + 1)) { // past the end: zeros times zeros
            TW_LDS(unsigned char) const rec = list + (n_rec + lane) * kRmRecord;
            *(TW_LDS(u32x4))rec = *(TW_LDS(u32x4))(rec + 16) = u32x4{kZeros * 0x10001u, kZeros * 0x10001u, kZeros * 0x10001u, kZeros * 0x10001u};
            *(TW_LDS(uint32_t))(rec + 32) = 0u;
            *(TW_LDS(uint32_t))(rec + 36) = kNoWeight;
            *(TW_LDS(uint32_t))(rec + 40) = 0xFFFFu;
            *(TW_LDS(uint32_t))(rec + 36 - T * kRmW * kRmRecord) = kNoWeight;
        }
        if (lane == 0)
            n_records[uq] = n_rec;
    }
    if (turn == T - 1) {
#pragma unroll
        for (int i = lane; i < CB * 32; i += 64) {
            const bool in = active && i < u.n_cnt;
            const int c = in ? u.col0 + p.kept_n[u.kn_off + i] : -1;
            col_s[uq * (CB * 32) + i] = c;
            bias_s[uq * (CB * 32) + i] = in && p.bias ? p.bias[c] : 0.0f;
        }
    }
    // the chunk of zeros: what a place there can name is the piece m % 16 of row m
    if (tid < kRmRows)
        *reinterpret_cast<u32x4 *>(rm_smem + kRmRing + kRmSlots * kRmSlot + tid * (kRmChunk * 2) + (tid & 15) * 16) = u32x4{0u, 0u, 0u, 0u};
    f32x16 acc[CB][2];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                acc[cb][mi][r] = 0.0f;
    TW_LDS_BARRIER(); // the lists are there, and the flags
    const int n_rec = __builtin_amdgcn_readfirstlane(n_records[uq]);

    if (turn < n_rec) {
        const uint32_t mbits = (uint32_t)(mrow * (kRmChunk * 2) | (mrow & 15) << 4);
        const uint32_t mb2 = mbits >> 1 | mbits >> 1 << 16;
        const uint32_t ring0 = (uint32_t)(uintptr_t)(TW_LDS(unsigned char))(rm_smem + kRmRing);
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(reinterpret_cast<const char *>(p.Bp) + u.b_off * 2 + (int64_t)u.nb0 * 4096), 0,
            u.k_pad / kBlockK * u.nblk * 4096 - u.nb0 * 4096, kRmRsrcFlags);
        u32x4 wq[kRmW][CB];
        const uint32_t lane16 = (uint32_t)lane * 16u;
        auto fetch_w = [&](uint32_t off, u32x4 (&w)[CB]) {
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) // (a block the unit does not have repeats its first)
                w[cb] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (int)(off + lane16), cb < u.nb_cnt ? cb * 4096 : 0, 0));
        };
        // The places, the chunk and the weight offset of this wave's next record, read a record ahead.
        TW_LDS(unsigned char) at = list + turn * kRmRecord;
        u32x4 r_next = *(TW_LDS(const u32x4))(at + half16 * 16);
        u32x4 x_next = *(TW_LDS(const u32x4))(at + 32);
#pragma unroll
        for (int q = 0; q < kRmW; ++q) {
            fetch_w(*(TW_LDS(const uint32_t))(at + 36 + (q - kRmW) * T * kRmRecord), wq[q]);
            asm volatile("" ::: "memory"); // (in this order, for the waits' counts)
        }
        // where this lane says which chunk its wave is at: one lane where the loading waves look, the others beside each other
        TW_LDS(volatile int) const say = lane == 0 ? at_hand + wave : landed + 16 + wave * 64 + lane;
        // The 2-byte reads of a record are issued one record ahead of its products.  Rows 16 .. 31 read the two rows of a
        // pair in the other order: rows m and m + 16 of a column lie in the same banks.
        const uint32_t turn_r = mrow & 16 ? 0x01000302u : 0x03020100u, turn_e = mrow & 16 ? 0x01000504u : 0x05040100u;
        uint32_t e[2][8];
        uint32_t w_off, own; // of the record at hand: the weight offset it brings, its rows
        int seen = 0; // chunks known to have landed
        auto look = [&]() {
            const int l = landed[lane & 3];
            const int l2 = min(l, __builtin_amdgcn_mov_dpp(l, 0xB1, 0xF, 0xF, true));      // lanes 1 0 3 2
            return __builtin_amdgcn_readfirstlane(min(l2, __builtin_amdgcn_mov_dpp(l2, 0x4E, 0xF, 0xF, true))); // lanes 2 3 0 1
        };
        // the next record: its chunk awaited, the look ahead, the reads of its rows one pair after another
        auto open = [&]() {
            const u32x4 r = r_next;
            const int run = __builtin_amdgcn_readfirstlane((int)x_next.x);
            w_off = x_next.y;
            own = (uint32_t)__builtin_amdgcn_readfirstlane((int)x_next.z);
            *say = (int)x_next.x; // (what the records before this one read is in registers)
            while (seen <= run)
                seen = look();
            asm volatile("" ::: "memory"); // (no read of the ring before this)
            at += T * kRmRecord;
            r_next = *(TW_LDS(const u32x4))(at + half16 * 16);
            x_next = *(TW_LDS(const u32x4))(at + 32);
            return r;
        };
        auto read_pair = [&](const u32x4 &r, int i) {
            const uint32_t rx = __builtin_amdgcn_perm(r[i], r[i], turn_r) ^ mb2;
            uint32_t q0, q1;
            asm("v_mad_u32_u16 %0, %1, 2, %2" : "=v"(q0) : "v"(rx), "v"(ring0));
            asm("v_mad_u32_u16 %0, %1, 2, %2 op_sel:[1,0,0,0]" : "=v"(q1) : "v"(rx), "v"(ring0));
#pragma unroll
            for (int mi = 0; mi < 2; ++mi) {
                e[mi][2 * i] = *(TW_LDS(const uint16_t))(uintptr_t)(q0 + mi * 32 * kRmChunk * 2);
                e[mi][2 * i + 1] = *(TW_LDS(const uint16_t))(uintptr_t)(q1 + mi * 32 * kRmChunk * 2);
            }
        };
        {
            const u32x4 r = open();
#pragma unroll
            for (int i = 0; i < 4; ++i)
                read_pair(r, i);
        }
        // The products of the record whose reads are in e[] between the reads of the next one (past the list's end zeros
        // times zeros), then the weight of the one kRmW on.  Nothing here is conditional and nothing else goes to
        // memory: the waits for a record's weight are exact counts.
        auto step = [&](u32x4 (&w)[CB]) {
            u32x4 a[2];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int mi = 0; mi < 2; ++mi)
                    a[mi][i] = __builtin_amdgcn_perm(e[mi][2 * i + 1], e[mi][2 * i], turn_e);
            const uint32_t off = w_off;
            if (own != 0xFFFFu) { // a record of a cut group: zeros also for the weight of the rows of its others, which may be infinite
                const uint32_t mine = own >> (half16 * 8);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t keep = (mine >> (2 * i) & 1u ? 0xFFFFu : 0u) | (mine >> (2 * i + 1) & 1u ? 0xFFFF0000u : 0u);
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb)
                        w[cb][i] &= keep;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            const u32x4 r = open();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                read_pair(r, i);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = i * CB / 2; j < (i + 1) * CB / 2; ++j)
                    acc[j >> 1][j & 1] = E::mfma(w[j >> 1], a[j & 1], acc[j >> 1][j & 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
            fetch_w(off, w);
        };
        for (int v = turn; v < n_rec; v += T * kRmW) {
#pragma unroll
            for (int q = 0; q < kRmW; ++q)
                step(wq[q]);
        }
    }
    if (lane == 0)
        at_hand[wave] = 0x7fffffff;
    TW_LDS_BARRIER(); // the ring is read no more

    // ---- the (partial) products: a lane holds row mi * 32 + lane % 32, columns cb * 32 + r4 * 8 + lane / 32 * 4 + 0 .. 3
    TW_LDS(float) const part = (TW_LDS(float))(TW_LDS(unsigned char))(rm_smem + kRmRing) + turn * kRmPart + mrow * kRmPitch +
                               uq * (CB * 32) + half16 * 4;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                *(TW_LDS(f32x4))(part + mi * 32 * kRmPitch + cb * 32 + r4 * 8) =
                    f32x4{acc[cb][mi][r4 * 4], acc[cb][mi][r4 * 4 + 1], acc[cb][mi][r4 * 4 + 2], acc[cb][mi][r4 * 4 + 3]};
    }
    TW_LDS_BARRIER(); // the products are there

    // ---- All waves: alpha, beta * C, bias, activation, one rounding, in pieces of eight columns of a row.  (In a loop
    // that is not unrolled: every instruction of this part is fetched once, by waves that wait for it.)
    const int oct = tid % (kRmCols / 8);
    TW_LDS(const float) const sum0 = (TW_LDS(const float))(TW_LDS(unsigned char))(rm_smem + kRmRing) + oct * 8;
    int col[8];
    float bias[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        col[i] = col_s[oct * 8 + i];
        bias[i] = bias_s[oct * 8 + i];
    }
    const bool octet = (col[0] & 7) == 0 && col[7] == col[0] + 7; // (-1 is no multiple of eight)
#pragma unroll 1
    for (int row = tid / (kRmCols / 8); row < m_cnt; row += kRmThreads / (kRmCols / 8)) {
        uint16_t *const dst = C + (int64_t)(m0 + row) * p.ldc;
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i += 4) {
            f32x4 s = *(TW_LDS(const f32x4))(sum0 + row * kRmPitch + i);
            if (!NARROW)
                s += *(TW_LDS(const f32x4))(sum0 + kRmPart + row * kRmPitch + i);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[i + j] = p.alpha * s[j];
        }
        if (p.beta != 0.0f) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (col[i] >= 0)
                    v[i] += p.beta * E::from_bits(dst[col[i]]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] += bias[i];
        tw_activate_all(v, p.act);
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            h[i] = E::to_bits2(tw_fp32_value(v[2 * i]), tw_fp32_value(v[2 * i + 1]));
        if (octet) {
            *reinterpret_cast<u32x4 *>(dst + col[0]) = u32x4{h[0], h[1], h[2], h[3]};
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (col[i] >= 0)
                    dst[col[i]] = (uint16_t)(h[i >> 1] >> ((i & 1) * 16));
        }
    }
    // ---- TW_PRUNED_ZERO: pruned columns receive act(beta * C + bias); shared out over the
    // workgroups of a row block
    fill_rowmajor_tiles<DT, kRmThreads>(p, grp, (int)gridDim.y, m0, m0 + m_cnt, tid);
}

int rm_groups(const tw_plan *plan)
{
    const int units = rm_units(rm_narrow(plan));
    return (plan->n_units + units - 1) / units;
}

// Whether the kernel can take the call: its lists fit beside the ring, its offsets 32 bits, its blocks of rows (a row block
// to a die, see launch_rm_t) and groups of units the two dimensions of a grid.
constexpr int kRmMaxGroups = 65535;
bool rm_takes(const tw_plan *plan, int M, int64_t lda)
{
    return plan->n_units > 0 && rm_lds_bytes(plan) <= kRmMaxLds && lda * 2 * kRmRows < (1ll << 31) &&
           plan->packed_elems * 2 < (1ll << 31) && rm_groups(plan) <= kRmMaxGroups &&
           ((int64_t)M / kRmRows + kXcd) * kRmThreads <= kMaxGridThreads;
}

template <int DT, bool NARROW> static int launch_rm_t(const tw_plan *plan, const GemmArgs &a, hipStream_t s)
{
    const int n_rowblk = (a.M + kRmRows - 1) / kRmRows, n_groups = rm_groups(plan);
    // (a row block to a die where that leaves no die more than a tenth behind)
    const int padded = (n_rowblk + kXcd - 1) / kXcd * kXcd;
    const int gx = (int64_t)padded * 10 <= (int64_t)n_rowblk * 11 ? padded : n_rowblk;
    hipLaunchKernelGGL((tw_gemm_rm_kernel<DT, NARROW>), dim3((unsigned)gx, (unsigned)n_groups), dim3(kRmThreads),
                       (size_t)rm_lds_bytes(plan), s, a, plan->K, n_rowblk, plan->max_k_pad);
    TW_HIP(hipGetLastError());
    return TW_OK;
}

int launch_rm(const tw_plan *plan, const GemmArgs &a, hipStream_t s)
{
    if (plan->dtype == TW_F16)
        return rm_narrow(plan) ? launch_rm_t<TW_F16, true>(plan, a, s) : launch_rm_t<TW_F16, false>(plan, a, s);
    return rm_narrow(plan) ? launch_rm_t<TW_BF16, true>(plan, a, s) : launch_rm_t<TW_BF16, false>(plan, a, s);
}

// (set once per device by prepare_device: function attributes may not be set during a capture)
int prepare_rm()
{
    const void *kernels[] = {(const void *)tw_gemm_rm_kernel<TW_F16, false>, (const void *)tw_gemm_rm_kernel<TW_F16, true>,
                             (const void *)tw_gemm_rm_kernel<TW_BF16, false>, (const void *)tw_gemm_rm_kernel<TW_BF16, true>};
    for (const void *k : kernels)
        TW_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kRmMaxLds));
    return TW_OK;
}

} // namespace tw
