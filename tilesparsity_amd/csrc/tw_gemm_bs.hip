// Weight-stationary kernels of the tile-wise-sparse GEMM (TW_SHAPE_BS), for tiles that keep few
// rows under many rows of A: BERT-like layers at 75 % sparsity and more.  First the one of four multiplying waves
// (tw_gemm_bs_kernel, at most 192 kept rows), then its wider form of eight (tw_gemm_bw_kernel, at most 384).
//
// A workgroup takes one unit (up to 128 compact columns of a tile) and a range of rows of A.  Its
// four multiplying waves own one block of 32 compact columns each and keep that block's packed
// weight - every kept row of it - in registers for the whole range, so the weight is read once
// per workgroup and the steady state moves nothing but A in and C out.  A fifth wave only loads:
// it gathers the tile's kept rows of A, 64 rows m at a time, with loads that write straight into
// LDS (buffer_load_dwordx4 ... lds: no registers, no LDS write instructions), a step of 64 kept
// rows per stage of a ring of four, two steps ahead of the multiplying waves.  Its waits for a
// step count exactly the loads issued behind it.  (It issues no store: memory operations of a
// wave complete in order, and a store in front of a load keeps that load's completion back
// until memory has acknowledged the store; measured with the stores of C moved into this wave:
// 27 us on a problem that takes 13.)  Both sides meet at one barrier per step.  The reference's
// counterpart is the masked main loop (cutlass/gemm/gemm_mainloop.h:230-338) with its gathered
// global -> shared stage (cutlass/tile_iterator.h:786-816), which re-reads the weight tile for
// every 128 rows of A.
//
//   stage:  64 kept rows k x 64 rows m, row k at k * 128 bytes, no padding (a load writes 1 KiB
//           of consecutive LDS: 8 rows); the two 64-byte halves of a row are swapped in rows
//           with bit 1 set, so that the four rows a transposed read touches fall into four
//           different bank groups.  The swap happens on the global side: lane l of a load
//           fetches chunk (l % 8) ^ 4 of such a row.
//   edges:  A is addressed through a buffer descriptor; a lane's offset names its row k and
//           16-byte piece, the scalar offset the block's first row m.  A list of kept rows is
//           padded to whole steps: the padding gets an offset beyond the buffer, for which the
//           hardware delivers zeros, so that nothing of a row the tile does not keep ever
//           reaches a product.  Rows m beyond M fetch whatever follows (or zeros); the rows of
//           the product they feed are never stored.
//   ranges: the rows of A are cut into n_ranges ranges on 32-row boundaries; the workgroups of a
//           range run on one die (workgroup b runs on die b % 8), so that the units of a range
//           share its rows of A in that die's L2.
//   output: a wave turns its 64 x 32 product through its own piece of LDS (no barrier) and
//           stores 16-byte pieces of whole columns, as the other kernels do; same order of
//           summation, so the same bits.
// Takes a K-major A below 4 GiB, a K-major C, and beta == 0 (C is not read).
#include "tw_device.h"

#include <algorithm>
#include <type_traits>

namespace tw {

constexpr int kBsRows = 64;                       // rows of A per block of a range
constexpr int kBsMulWaves = 4;
constexpr int kBsLoadWave = kBsMulWaves;
constexpr int kBsWaves = kBsMulWaves + 1;
constexpr int kBsRing = 4;                        // stages
constexpr int kBsAhead = 2;                       // steps of loads in flight ahead of the multiplying waves
constexpr int kBsStage = kBlockK * kBsRows * 2;   // 8 KiB
constexpr int kBsCPitch = kBsRows + 4;            // elements per column of a wave's C stage
constexpr int kBsCStage = 32 * kBsCPitch * 2;     // bytes
constexpr int kBsPerCu = 2;                       // workgroups meant to share a compute unit
constexpr int kBsRsrcFlags = 0x00020000;          // word 3 of a raw buffer descriptor of this target
static_assert(kBsRing >= kBsAhead + 2, "a stage is refilled only after the step before last has been multiplied");
static_assert(kBsAhead == 2, "the loading wave's waits are written out for two steps ahead");
constexpr int kBsMaxSteps = 3;                    // steps of 64 kept rows the widest instantiation holds in registers
                                                  // (four: 64 more registers than a wave of four a SIMD has)

// the loading wave: waits until at most N of its loads are outstanding, then meets the other waves
template <int N> __device__ __forceinline__ void bs_wait_loads_and_meet()
{
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

// (at most 128 registers: the first SIMD of a compute unit holds two waves of each of its two
// workgroups; a third workgroup's five waves find no room on it)
template <int DT, int NS>
__global__ void __launch_bounds__(64 * kBsWaves, 4)
    tw_gemm_bs_kernel(const GemmArgs p, int n_units, int n_ranges, int row_units, int affine, uint32_t a_bytes,
                      uint32_t)
{
    using E = Elem<DT>;
    static_assert(NS >= 1 && NS <= kBsMaxSteps, "steps in registers");
    __shared__ __align__(1024) unsigned char ring[kBsRing * kBsStage];
    __shared__ __align__(16) unsigned char cstage[kBsMulWaves * kBsCStage];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroup -> (unit, range); with `affine` the ranges r = die (mod 8) sit on one die
    int ui, r;
    if (affine) {
        const int die = blockIdx.x % kXcd, i = blockIdx.x / kXcd;
        ui = i % n_units;
        r = die + kXcd * (i / n_units);
    } else {
        r = blockIdx.x % n_ranges;
        ui = blockIdx.x / n_ranges;
    }
    if (r >= n_ranges)
        return;
    const int m_lo = (int)((int64_t)r * row_units / n_ranges) * 32;
    const int m_hi = min((int)((int64_t)(r + 1) * row_units / n_ranges) * 32, p.M);
    if (m_lo >= m_hi)
        return;
    const UnitDev u = load_unit(p, ui);
    const int nsteps = u.k_pad / kBlockK; // <= NS (host check)
    const int n_mb = (m_hi - m_lo + kBsRows - 1) / kBsRows;
    const int total = n_mb * nsteps; // steps, and barriers, of the workgroup

    if (wave == kBsLoadWave) {
        // ================= the loading wave =================================================
        if (nsteps == 0)
            return;
        const int rr = lane >> 3, pos = lane & 7;
        const uint32_t lda_b = (uint32_t)p.lda * 2u;
        const __amdgpu_buffer_rsrc_t a_rsrc =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p.A), 0, (int)a_bytes, kBsRsrcFlags);
        // Load j of a step covers its kept rows 8 j .. 8 j + 7; lane l fetches 16 bytes of row
        // 8 j + l / 8 into LDS position l % 8 of that row.
        uint32_t off[NS][8];
        {
            // the row numbers: one load per step for the whole wave (lane l asks for row l of the
            // step; a step the unit does not have asks for its last one again), all in flight
            // together, then handed to the lanes that fetch the row
            int knum[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s)
                knum[s] = p.kept_k[u.kk_off + (s < nsteps ? s : nsteps - 1) * kBlockK + lane]; // the list is padded: in bounds
#pragma unroll
            for (int s = 0; s < NS; ++s) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int row = j * 8 + rr; // kept row of the step
                    const int chunk = pos ^ (((row >> 1) & 1) << 2);
                    const uint32_t k = (uint32_t)__shfl(knum[s], row);
                    off[s][j] = s * kBlockK + row < u.k_kept ? k * lda_b + (uint32_t)chunk * 16u : 0xFFFFFFF0u;
                }
            }
        }
        TW_LDS(unsigned char) const lds0 = (TW_LDS(unsigned char))ring;
        // Step gi is issued, then step gi - 2 handed over: behind its loads are those of the steps
        // issued since (two, fewer at the end of the range).
        int s_cur = 0, mb_cur = 0;
        for (int gi = 0; gi < total + kBsAhead; ++gi) {
            if (gi < total) {
                const int m0b = (m_lo + mb_cur * kBsRows) * 2;
                TW_LDS(unsigned char) const dst = lds0 + (gi % kBsRing) * kBsStage;
#define TW_BS_ISSUE(S)                                                                                      \
    _Pragma("unroll") for (int j = 0; j < 8; ++j) __builtin_amdgcn_raw_ptr_buffer_load_lds(                 \
        a_rsrc, (TW_LDS(void))(dst + j * 1024), 16, (int)off[(S) < NS ? (S) : 0][j], m0b, 0, 0)
                switch (s_cur) { // (the offsets of a step sit in registers: one copy of the loads per step)
                case 0:
                    TW_BS_ISSUE(0);
                    break;
                case 1:
                    TW_BS_ISSUE(1);
                    break;
                default:
                    TW_BS_ISSUE(2);
                    break;
                }
#undef TW_BS_ISSUE
                if (++s_cur == nsteps) {
                    s_cur = 0;
                    ++mb_cur;
                }
            }
            if (gi >= kBsAhead) {
                const int behind = min(gi, total - 1) - (gi - kBsAhead); // steps issued behind the one handed over
                if (behind >= 2)
                    bs_wait_loads_and_meet<16>();
                else if (behind == 1)
                    bs_wait_loads_and_meet<8>();
                else
                    bs_wait_loads_and_meet<0>();
            }
        }
        return;
    }

    // ================= multiplying waves ====================================================
    // A unit of at most 64 compact columns has two blocks: its four waves then take a block and
    // one 32-row half of the 64 rows each, instead of two waves taking a block and two idling.
    const bool narrow = u.nb_cnt <= 2;
    const int half = wave >> 1;
    const bool active = (narrow ? wave & 1 : wave) < u.nb_cnt;
    const int nb = active ? (narrow ? wave & 1 : wave) : 0;
    const int cnt = min(32, u.n_cnt - nb * 32); // compact columns of this wave's block
    const int L = lane & 15;
    const int j = lane & 31;
    // weight fragments of the block: every kept row, in registers
    u32x4 bq[NS][4];
    {
        const unsigned char *const bsrc = reinterpret_cast<const unsigned char *>(p.Bp) +
                                          (nsteps ? u.b_off * 2 + (int64_t)(u.nb0 + nb) * 4096 : 0) + lane * 16;
        const int64_t step_b = (int64_t)u.nblk * 4096;
        // (no branches: a step the unit does not have fetches its last one again and is never used;
        // a unit without kept rows owns no weight: it fetches the plan's first fragments)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int sc = s < nsteps ? s : max(nsteps - 1, 0);
#pragma unroll
            for (int k16 = 0; k16 < 4; ++k16)
                bq[s][k16] = *reinterpret_cast<const u32x4 *>(bsrc + sc * step_b + k16 * 1024);
        }
    }
    int out_col = u.col0 + p.kept_n[u.kn_off + nb * 32 + (j < cnt ? j : 0)];
    float out_bias = p.bias ? p.bias[out_col] : 0.0f;
    // Everything fetched so far is waited for here, before the loop over the range: inside it
    // the only memory operations of these waves are the output stores, and a wait placed there
    // for one of these loads would wait for the stores of the block before as well.
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int k16 = 0; k16 < 4; ++k16)
            asm volatile("" : "+v"(bq[s][k16]));
    asm volatile("" : "+v"(out_col), "+v"(out_bias));
    // this lane's address inside a stage for the transposed reads: row (lane / 32) * 8 + L / 4 of a
    // group of 16 kept rows, 8 bytes at m = (lane / 16 % 2) * 16 + (L % 4) * 4 of a 32-row half;
    // the halves of a row are swapped where bit 1 of the row is set
    const uint32_t swap = (uint32_t)((L >> 3) & 1);
    const uint32_t lane_row = (uint32_t)((lane >> 5) * 8 + (L >> 2)) * 128u + (uint32_t)(((lane >> 4) & 1) * 32 + (L & 3) * 8);
    const uint32_t lane_a[2] = {lane_row + swap * 64u, lane_row + (1u - swap) * 64u};
    TW_LDS(unsigned char) const lds0 = (TW_LDS(unsigned char))ring;
    uint16_t *const cst = reinterpret_cast<uint16_t *>(cstage + wave * kBsCStage);
    uint16_t *const C = reinterpret_cast<uint16_t *>(p.C);

    int g = 0; // flat step
    for (int mb = 0; mb < n_mb; ++mb) {
        f32x16 acc[2];
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[mi][e] = 0.0f;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (s < nsteps) {
                TW_LDS_BARRIER(); // the step is in its stage (and this wave's reads of the step before are over)
                if (active) {
                    TW_LDS(unsigned char) const st = lds0 + (g % kBsRing) * kBsStage;
#pragma unroll
                    for (int k16 = 0; k16 < 4; ++k16) {
#pragma unroll
                        for (int mi = 0; mi < 2; ++mi) {
                            if (narrow && mi != half)
                                continue;
                            TW_LDS(unsigned char) const q = st + lane_a[mi] + k16 * 2048;
                            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((TW_LDS(s16x4))q);
                            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((TW_LDS(s16x4))(q + 512));
                            const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
                            acc[mi] = E::mfma(u32x4{l2.x, l2.y, h2.x, h2.y}, bq[s][k16], acc[mi]);
                        }
                    }
                }
                ++g;
            }
        }
        if (!active)
            continue;
        // ---- the block's 64 x 32 product: alpha, bias, activation, one rounding; through the
        // wave's stage as [column][row m]; 16-byte stores of whole columns
        const int m0 = m_lo + mb * kBsRows;
        const int m_end = min(m0 + kBsRows, m_hi);
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[mi][e] = p.alpha * acc[mi][e] + out_bias;
        }
        if (p.act != TW_ACT_NONE) { // (tested once per block, not per element)
#pragma unroll
            for (int mi = 0; mi < 2; ++mi) {
                float v[16];
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    v[e] = acc[mi][e];
                tw_activate_all(v, p.act);
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    acc[mi][e] = v[e];
            }
        }
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                u32x2 pk;
                pk.x = E::to_bits2(tw_fp32_value(acc[mi][r4 * 4]), tw_fp32_value(acc[mi][r4 * 4 + 1]));
                pk.y = E::to_bits2(tw_fp32_value(acc[mi][r4 * 4 + 2]), tw_fp32_value(acc[mi][r4 * 4 + 3]));
                *reinterpret_cast<u32x2 *>(cst + j * kBsCPitch + mi * 32 + (lane >> 5) * 4 + r4 * 8) = pk;
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        // (what follows is worked out from the lane number anew in every block: kept across the
        // loop, these few values cost registers the widest instantiation does not have, and a
        // value parked in scratch memory comes back behind a wait for every store in flight)
        int ln = lane;
        asm volatile("" : "+v"(ln));
#pragma unroll
        for (int q = 0; q < 4; ++q) { // 32 columns x 8 chunks of 8 rows
            const int idx = ln + q * 64;
            const int jj = idx >> 3, ch = idx & 7;
            const int col = __shfl(out_col, jj);
            const u32x2 lo = *reinterpret_cast<const u32x2 *>(cst + jj * kBsCPitch + ch * 8);
            const u32x2 hi = *reinterpret_cast<const u32x2 *>(cst + jj * kBsCPitch + ch * 8 + 4);
            const int m = m0 + ch * 8;
            if (jj < cnt && (!narrow || (ch >> 2) == half))
                store_chunk(C + (int64_t)col * p.ldc + m, u32x4{lo.x, lo.y, hi.x, hi.y}, m, m_end,
                            p.store_through != 0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the stage is free again
    }

    // ---- TW_PRUNED_ZERO: the pruned columns of this unit's share of the tiles receive act(bias)
    // on the range's rows
    for (int z = ui; z < p.n_all_u - p.n_gemm_u; z += n_units)
        fill_kmajor<DT, 64 * kBsMulWaves>(p, p.act, fill_tile(p, z), m_lo, m_hi, tid, p.store_through != 0);
}

// ---------------------------------------------------------------------------------
// The same with eight multiplying waves, for tiles of up to 384 kept rows (instantiations of two, three, four and six steps).
// What bounds it is C on its way out (M 8192, N 4096: 64 MB, 14 us at 4.5 TB/s, what such stores alone reach) beside the
// gathered reads of A, and how well a block's epilogue hides beneath the next one's products.  A wave that holds 32 columns of
// four steps and multiplies 64 rows at a time has room for nobody beside it, so here eight waves multiply 32 rows x 32 columns
// each (the two of a block of columns hold its weight twice), two to four load, and one workgroup has the compute unit (168
// registers a wave).  Two waves a SIMD are too few to fill each other's waits, so a wave's own work is laid out to overlap:
// the vector instructions of a block's epilogue (GELU: 250 of them) stand between the products of the next block, which need
// the matrix pipe for 32 cycles each, and the reads of a product's rows three products ahead.  For that a block is one piece
// of straight code: all of its steps have landed when it begins (words in LDS instead of a barrier per step: a loading wave
// says which of its steps are there, a multiplying wave how many it has read), tiles with fewer steps multiply zeros in the
// missing ones, and the activation is a template argument.  The multiplying waves' memory queue holds stores only and nothing
// in the loop waits for it.
// A wave's 32 rows are 64 bytes of a column.  Where those are whole sectors of memory they are stored through to it; else they
// stay in L2, where a sector's two parts meet (`through`: M 5809, N 3515, two thirds of the columns 16 bytes off, 41.5 us
// through and 17 not; M 12516, N 7222 152 and 58; 1000 such problems 0.47 - 0.71 of what ran before, through 0.92 - 1.18).
// Stored a further block later through the stage that the two waves of a block of
// columns share, they go out as whole 128-byte lines (`lines`): ahead where C leaves the last-level cache (134 MB 61 -> 47.6
// us), level below (64 MB: 26.2 without, 26.8 with), crossing at 90 - 96 MB.
// Measured (bf16, us of a replayed graph, the panel kernel or the four-wave one -> this): M 8192, K 1024, N 4096, 256 kept rows
// 34.2 -> 26.2, with GELU 39.7 -> 32.5; M 12288 61.3 -> 37.0, with GELU 69.5 -> 43.5; M 4096, K 768, N 3072, 192 kept 15.1 ->
// 13.0, with GELU 16.9 -> 16.1.  Without activation and with ReLU bit for bit what those give; GELU and tanh of the same sum come
// from instructions in another order, within one unit in the last place of the result.
constexpr int kBwMulWaves = 8;
constexpr int bw_load_waves(int ns) { return ns <= 4 ? ns : 3; } // (three and four waves a SIMD have 168 and 128 registers)
constexpr int bw_threads(int ns) { return 64 * (kBwMulWaves + bw_load_waves(ns)); }
constexpr int kBwRing = 14;                          // stages of 8 KiB
constexpr int kBwCPitch = kBsRows + 4;               // elements per column of a C stage
constexpr int kBwCStage = 32 * kBwCPitch * 2;        // bytes; two of them for the two waves of a block of columns
constexpr int64_t kBwLineBytes = 90 << 20;           // outputs from here on are stored in whole lines
constexpr uint64_t kBwMaxBytes = 0xFFFF0000u;        // of C, which is stored through a buffer descriptor
constexpr int kBwSteps = 6;                          // most steps of an instantiation
constexpr uint32_t kBwNoRow = 0xFFFFFFFFu;           // (offsets of rows are multiples of 16)

template <int DT, int ACT, int NS>
__global__ void __launch_bounds__(bw_threads(NS), 3)
    tw_gemm_bw_kernel(const GemmArgs p, int n_units, int n_ranges, int row_units, int affine, uint32_t a_bytes,
                      uint32_t c_bytes, int lines, int through)
{
    using E = Elem<DT>;
    constexpr int LW = bw_load_waves(NS), SPW = NS / LW; // loading waves, steps of a block each
    static_assert(LW * SPW == NS, "whole steps a wave");
    __shared__ __align__(1024) unsigned char ring[kBwRing * kBsStage];
    __shared__ __align__(16) unsigned char cstage[kBwMulWaves * kBwCStage];
    __shared__ uint32_t row_off[NS * kBlockK]; // byte offset of each kept row in A, kBwNoRow for the list's padding
    __shared__ int flags[16];                  // first step that is not there of each loading wave's, steps each multiplying wave has read
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int ui, r;
    if (affine) {
        const int die = blockIdx.x % kXcd, i = blockIdx.x / kXcd;
        ui = i % n_units;
        r = die + kXcd * (i / n_units);
    } else {
        r = blockIdx.x % n_ranges;
        ui = blockIdx.x / n_ranges;
    }
    if (r >= n_ranges)
        return;
    const int m_lo = (int)((int64_t)r * row_units / n_ranges) * 32;
    const int m_hi = min((int)((int64_t)(r + 1) * row_units / n_ranges) * 32, p.M);
    if (m_lo >= m_hi)
        return;
    const UnitDev u = load_unit(p, ui);
    const int nsteps = u.k_pad / kBlockK; // <= NS (host check)
    const int n_mb = (m_hi - m_lo + kBsRows - 1) / kBsRows;
    TW_LDS(volatile int) const landed = (TW_LDS(volatile int))flags;
    TW_LDS(volatile int) const done = landed + 4;
    if (tid < 4 + kBwMulWaves)
        flags[tid] = tid < LW ? 0 : tid < 4 ? 0x7fffffff : 0;
    uint16_t *const C = reinterpret_cast<uint16_t *>(p.C);

    if (wave >= kBwMulWaves) {
        // ================= loading waves: the same SPW steps of every block each =============
        const int w = wave - kBwMulWaves;
        const uint32_t lda_b = (uint32_t)p.lda * 2u;
#pragma unroll
        for (int q = 0; q < SPW; ++q) {
            const int i = (w * SPW + q) * kBlockK + lane;
            row_off[i] = i < u.k_kept ? (uint32_t)p.kept_k[u.kk_off + i] * lda_b : kBwNoRow;
        }
        TW_LDS_BARRIER(); // the row offsets, and the flags
        const __amdgpu_buffer_rsrc_t a_rsrc =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p.A), 0, (int)a_bytes, kBsRsrcFlags);
        const int rr = lane >> 3, pos = lane & 7;
        // load j of a step covers its kept rows 8 j .. 8 j + 7, lane l 16 bytes of row 8 j + l / 8; halves swapped as above
        uint32_t off[SPW][8];
#pragma unroll
        for (int q = 0; q < SPW; ++q)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                // (a row that is not there: 16 bytes short of 4 GiB whatever the piece, beyond every buffer bs_takes admits)
                const uint32_t row = row_off[(w * SPW + q) * kBlockK + j * 8 + rr];
                off[q][j] = row == kBwNoRow ? 0xFFFFFFF0u : row + (uint32_t)(pos ^ ((rr >> 1 & 1) << 2)) * 16u;
            }
        TW_LDS(unsigned char) const lds0 = (TW_LDS(unsigned char))ring;
        // two blocks in flight: what a block takes to arrive is more than what it takes to multiply
        auto issue = [&](int mb) {
            const int m0b = (m_lo + mb * kBsRows) * 2;
#pragma unroll
            for (int q = 0; q < SPW; ++q) {
                const int g = mb * NS + w * SPW + q;
                if (g >= kBwRing)
                    while (!__all(done[lane & 7] > g - kBwRing))
                        __builtin_amdgcn_s_sleep(1);
                TW_LDS(unsigned char) const dst = lds0 + g % kBwRing * kBsStage;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (TW_LDS(void))(dst + j * 1024), 16, (int)off[q][j], m0b, 0, 0);
            }
        };
        issue(0);
        for (int mb = 0; mb < n_mb; ++mb) {
            if (NS <= kBwRing / 3 && mb + 1 < n_mb) { // (a block ahead of the one waited for, where three fit the ring)
                issue(mb + 1);
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 * SPW) : "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            if (lane == 0)
                landed[w] = (mb + 1) * NS;
            if (NS > kBwRing / 3 && mb + 1 < n_mb)
                issue(mb + 1);
        }
        return;
    }

    // ================= multiplying waves ====================================================
    const int cb = wave & 3, mi = wave >> 2;
    const bool active = cb < u.nb_cnt;
    const int nb = active ? cb : 0;
    const int cnt = min(32, u.n_cnt - nb * 32);
    const int L = lane & 15, j = lane & 31;
    TW_LDS_BARRIER(); // the row offsets, and the flags (before anything is fetched here: the loading waves stand behind it)
    const int out_n = p.kept_n[u.kn_off + nb * 32 + (j < cnt ? j : 0)];
    u32x4 bq[NS][4];
    {
        const unsigned char *const bsrc = reinterpret_cast<const unsigned char *>(p.Bp) +
                                          (nsteps ? u.b_off * 2 + (int64_t)(u.nb0 + nb) * 4096 : 0) + lane * 16;
        const int64_t step_b = (int64_t)u.nblk * 4096;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
#pragma unroll
            for (int k16 = 0; k16 < 4; ++k16) {
                bq[s][k16] = *reinterpret_cast<const u32x4 *>(bsrc + (s < nsteps ? s : 0) * step_b + k16 * 1024);
                if (s >= nsteps) // (zeros times zeros: the loading waves' rows there are beyond the buffer)
                    bq[s][k16] = u32x4{0u, 0u, 0u, 0u};
            }
        }
    }
    int out_col = u.col0 + out_n;
    float out_bias = p.bias ? p.bias[out_col] : 0.0f;
    const uint32_t swap = (uint32_t)((L >> 3) & 1);
    const uint32_t lane_a = (uint32_t)((lane >> 5) * 8 + (L >> 2)) * 128u + (uint32_t)(((lane >> 4) & 1) * 32 + (L & 3) * 8) +
                            (mi ? 1u - swap : swap) * 64u;
    TW_LDS(unsigned char) const lds0 = (TW_LDS(unsigned char))ring + lane_a;
    TW_LDS(unsigned char) const cst = (TW_LDS(unsigned char))cstage + cb * 2 * kBwCStage;
    int slot = 0;
    f32x16 acc{};
    // Both waves of a block of columns put their 32 rows of a product into one stage.  With `lines` each takes 16 of its columns
    // out, 64 rows, whole 128-byte lines of C, for which it waits until the other is as far; else each takes its own 32 rows out
    // again, 64 bytes a column.  This lane's two 16-byte pieces:
    const int jq[2] = {lines ? mi * 16 + (lane >> 3) : lane >> 2, lines ? mi * 16 + (lane >> 3) + 8 : (lane >> 2) + 16};
    const int row_q = lines ? (lane & 7) * 8 : mi * 32 + (lane & 3) * 8;
    uint32_t o_q[2]; // byte offset of the column, and of the row inside a block (set once the column numbers are there)
    // a block's epilogue goes to stage `parity`
    auto stage_put = [&](int parity, int r4, const float (&e)[4]) {
        *(TW_LDS(u32x2))(cst + parity * kBwCStage + (j * kBwCPitch + mi * 32 + (lane >> 5) * 4 + r4 * 8) * 2) =
            u32x2{E::to_bits2(e[0], e[1]), E::to_bits2(e[2], e[3])};
    };
    auto stage_get = [&](int parity, int q) {
        const u32x2 lo = *(TW_LDS(const u32x2))(cst + parity * kBwCStage + (jq[q] * kBwCPitch + row_q) * 2);
        const u32x2 hi = *(TW_LDS(const u32x2))(cst + parity * kBwCStage + (jq[q] * kBwCPitch + row_q + 4) * 2);
        return u32x4{lo.x, lo.y, hi.x, hi.y};
    };
    // the pieces of block mb, out of the stage, to C
    auto put = [&](int mb, const u32x4 (&v)[2]) {
        const int m0 = m_lo + mb * kBsRows;
        const int m_end = min(m0 + kBsRows, m_hi);
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (jq[q] < cnt)
                store_chunk(reinterpret_cast<uint16_t *>(reinterpret_cast<char *>(C) + o_q[q]) + m0, v[q], m0 + row_q, m_end,
                            through && p.store_through);
    };
    // The products of block mb, whose steps have landed.  Between them (`older` blocks before it: 0, 1, or 2 and more) the
    // epilogue of the block before (`prev`) goes to one stage, and the block before that from the other one to C: whole
    // blocks, through a buffer descriptor that drops the columns the unit does not have, and `through` to memory (as
    // store_chunk).  `land` is what the flags said in the middle of the block.
    const __amdgpu_buffer_rsrc_t c_rsrc = __builtin_amdgcn_make_buffer_rsrc(C + m_lo, 0, (int)c_bytes, kBsRsrcFlags);
    const bool other = lines && (lane & 4); // what this lane watches: the other wave, or the loads
    TW_LDS(volatile int) const flag = other ? done + (wave ^ 4) : landed + (lane & 3);
    const int flag_add = other ? NS : 0;
    int land = 0;
    auto block = [&](const f32x16 &prev, int mb, auto older_tag) {
        constexpr int OLDER = decltype(older_tag)::value;
        const int parity = (mb - 1) & 1;
        u32x4 out[2];
        f32x16 sum;
#pragma unroll
        for (int e = 0; e < 16; ++e)
            sum[e] = 0.0f;
        u32x4 af[NS * 4];
        auto fetch = [&](int i) {
            const int sl = slot + (i >> 2);
            TW_LDS(unsigned char) const st = lds0 + (sl >= kBwRing ? sl - kBwRing : sl) * kBsStage + (i & 3) * 2048;
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((TW_LDS(s16x4))(st));
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((TW_LDS(s16x4))(st + 512));
            const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
            af[i] = u32x4{l2.x, l2.y, h2.x, h2.y};
        };
        constexpr int AHEAD = NS == 6 ? 2 : 3; // (registers)
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            fetch(i);
        __builtin_amdgcn_sched_barrier(0);
        float epi[4];
#pragma unroll
        for (int i = 0; i < NS * 4; ++i) {
            if (i + AHEAD < NS * 4)
                fetch(i + AHEAD);
            if (i == NS)
                land = *flag;
            if (OLDER > 1 && (i == 2 || i == 3))
                out[i - 2] = stage_get(parity ^ 1, i - 2);
            sum = E::mfma(af[i], bq[i >> 2][i & 3], sum);
            if (OLDER > 1 && (i == NS * 4 - 2 || i == NS * 4 - 1)) {
                const int q = i - (NS * 4 - 2), row_b = (mb - 2) * kBsRows * 2;
                if (through)
                    __builtin_amdgcn_raw_buffer_store_b128(out[q], c_rsrc, (int)o_q[q], row_b, 1 | 2 | 16);
                else
                    __builtin_amdgcn_raw_buffer_store_b128(out[q], c_rsrc, (int)o_q[q], row_b, 0);
                // Two wait states before the data's registers are written again: the store is still reading them, and the compiler
                // adds none to a buffer store with a scalar offset (an instruction that wrote the second of the four
                // at once put its own result into C).
                asm volatile("s_nop 1" ::"v"(out[q]));
            }
            if constexpr (OLDER > 0) {
                // this product's share of the sixteen values of the block before; four of them go to the stage together
                constexpr int P = NS < 4 ? NS * 4 : 16;
#pragma unroll
                for (int e = 16 * i / P; e < 16 * (i + 1) / P && e < 16; ++e) {
                    epi[e & 3] = tw_fp32_value(tw_activate(p.alpha * prev[e] + out_bias, ACT));
                    if ((e & 3) == 3)
                        stage_put(parity, e >> 2, epi);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        slot += NS;
        slot = slot >= kBwRing ? slot - kBwRing : slot;
        return sum;
    };
    // All steps of block mb have landed, and with `lines` the other wave of these columns has the block before behind it (it
    // has put its rows of the one before that into the stage, and taken its columns of the one before that out of it).
    auto await = [&](int mb) {
        for (int l = land;; l = *flag)
            if (__all(l >= (mb + 1) * NS - flag_add))
                break;
        asm volatile("" ::: "memory"); // (no read of the stages before this)
    };
    // (every read of the block's stages has been waited for by its product)
    auto say = [&](int mb) {
        asm volatile("" ::: "memory");
        if (lane == 0)
            done[wave] = (mb + 1) * NS;
    };
    if (active) {
        await(0);
        acc = block(acc, 0, std::integral_constant<int, 0>());
        say(0);
        // (the weight has arrived: nothing in the loop waits for it, which would be to wait for stores as well)
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int k16 = 0; k16 < 4; ++k16)
                asm volatile("" : "+v"(bq[s][k16]));
        asm volatile("" : "+v"(out_col), "+v"(out_bias));
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t col = (uint32_t)__shfl(out_col, jq[q]);
            o_q[q] = jq[q] < cnt ? col * ((uint32_t)p.ldc * 2u) + (uint32_t)row_q * 2u : 0xFFFFFF00u;
        }
        if (n_mb > 1) {
            await(1);
            acc = block(acc, 1, std::integral_constant<int, 1>());
            say(1);
        }
        for (int mb = 2; mb < n_mb; ++mb) {
            await(mb);
            acc = block(acc, mb, std::integral_constant<int, 2>());
            say(mb);
        }
        while (lines && done[wave ^ 4] < n_mb * NS) // (the other wave has taken out what was in the last block's stage)
            ;
        asm volatile("" ::: "memory");
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] = tw_fp32_value(tw_activate(p.alpha * acc[r4 * 4 + e] + out_bias, ACT));
            stage_put((n_mb - 1) & 1, r4, v);
        }
        asm volatile("" ::: "memory");
        if (lane == 0)
            done[wave] = 0x7fffffff;
        while (lines && done[wave ^ 4] != 0x7fffffff)
            ;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        for (int mb = max(n_mb - 2, 0); mb < n_mb; ++mb) {
            const u32x4 out[2] = {stage_get(mb & 1, 0), stage_get(mb & 1, 1)};
            put(mb, out);
        }
    }
    if (lane == 0)
        done[wave] = 0x7fffffff;

    // ---- TW_PRUNED_ZERO: the pruned columns of this unit's share of the tiles receive act(bias)
    for (int z = ui; z < p.n_all_u - p.n_gemm_u; z += n_units)
        fill_kmajor<DT, 64 * kBwMulWaves>(p, ACT, fill_tile(p, z), m_lo, m_hi, tid, through && p.store_through);
}

bool bw_takes(const tw_plan *plan, int64_t lda, int64_t ldc, bool reads_c)
{
    if (reads_c || plan->n_units == 0 || plan->n_pipe_units == 0 || (int64_t)plan->n_units * 1024 > kMaxGridThreads)
        return false;
    // A is addressed, and C stored, through a buffer descriptor with 32-bit offsets
    return (uint64_t)plan->K * (uint64_t)lda * 2u < (1ull << 32) && plan->max_k_pad <= kBwSteps * kBlockK &&
           (uint64_t)plan->N * (uint64_t)ldc * 2u < kBwMaxBytes;
}

bool bs_takes(const tw_plan *plan, int64_t lda, int64_t ldc, bool reads_c)
{
    if (bw_takes(plan, lda, ldc, reads_c))
        return true;
    // (the four-wave kernel stores C by address: any size of it)
    return plan->max_k_pad <= kBsMaxSteps * kBlockK && bw_takes(plan, lda, 0, reads_c);
}

// ranges of rows of A a launch is cut into: as many as give every compute unit `per_cu`
// workgroups, a multiple of the number of dies (a range then lives on one die) or a divisor of it
int bs_ranges(const tw_plan *plan, int M, int per_cu)
{
    if (per_cu <= 0)
        per_cu = kBsPerCu;
    const int row_units = (M + 31) / 32;
    int r = std::max(1, plan->cu_count * per_cu / std::max(1, plan->n_units));
    r = std::min(r, std::max(1, row_units / 2)); // at least 64 rows a range
    if (r >= kXcd)
        r = r / kXcd * kXcd;
    else
        r = r >= 4 ? 4 : (r >= 2 ? 2 : 1);
    return r;
}

// the wider form's: as many as fit one workgroup on each compute unit; below the number of dies whatever that is
int bw_ranges(const tw_plan *plan, int M, int per_cu)
{
    const int r = std::min(std::max(1, plan->cu_count * std::max(1, per_cu) / std::max(1, plan->n_units)), std::max(1, (M + 31) / 64));
    return r >= kXcd ? r / kXcd * kXcd : r;
}

// share of the compute units the launch fills with one workgroup each, over a whole number of rounds
double bs_fill(const tw_plan *plan, int M)
{
    const int64_t wgs = (int64_t)plan->n_units * bw_ranges(plan, M, 1), cu = plan->cu_count;
    const int64_t rounds = (wgs + cu - 1) / cu;
    return (double)wgs / (double)(rounds * cu);
}

// whether every 32 rows of a column of C are whole 64-byte pieces of memory
bool bs_whole_sectors(const void *C, int64_t ldc) { return (((uintptr_t)C | (uintptr_t)ldc * 2u) & 63) == 0; }

template <int DT, int NS> static int launch_bs_t(const tw_plan *plan, const GemmArgs &a, int per_cu, hipStream_t s)
{
    const int n_ranges = bs_ranges(plan, a.M, per_cu);
    const int affine = n_ranges >= kXcd;
    const int64_t grid = affine ? (int64_t)kXcd * plan->n_units * (n_ranges / kXcd) : (int64_t)n_ranges * plan->n_units;
    if (grid > (int64_t)0x7fffffff)
        return fail(TW_ERR_SHAPE, "%lld workgroups (M=%d): a launch takes at most %lld", (long long)grid, a.M,
                    (long long)(int64_t)0x7fffffff);
    hipLaunchKernelGGL((tw_gemm_bs_kernel<DT, NS>), dim3((unsigned)grid), dim3(64 * kBsWaves), 0, s, a, plan->n_units,
                       n_ranges, (a.M + 31) / 32, affine, (uint32_t)((uint64_t)plan->K * (uint64_t)a.lda * 2u), 0u);
    TW_HIP(hipGetLastError());
    return TW_OK;
}

template <int DT, int NS> static int launch_bw(const tw_plan *plan, const GemmArgs &a, int per_cu, hipStream_t s)
{
    const int n_ranges = bw_ranges(plan, a.M, per_cu);
    const int affine = n_ranges >= kXcd;
    const int64_t grid = affine ? (int64_t)kXcd * plan->n_units * (n_ranges / kXcd) : (int64_t)n_ranges * plan->n_units;
    if (grid > (int64_t)0x7fffffff)
        return fail(TW_ERR_SHAPE, "%lld workgroups (M=%d): a launch takes at most %lld", (long long)grid, a.M,
                    (long long)(int64_t)0x7fffffff);
    const int whole = bs_whole_sectors(a.C, a.ldc);
    const auto kernel = a.act == TW_ACT_RELU   ? tw_gemm_bw_kernel<DT, TW_ACT_RELU, NS>
                        : a.act == TW_ACT_GELU ? tw_gemm_bw_kernel<DT, TW_ACT_GELU, NS>
                        : a.act == TW_ACT_TANH ? tw_gemm_bw_kernel<DT, TW_ACT_TANH, NS>
                                               : tw_gemm_bw_kernel<DT, TW_ACT_NONE, NS>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(bw_threads(NS)), 0, s, a, plan->n_units, n_ranges, (a.M + 31) / 32, affine,
                       (uint32_t)((uint64_t)plan->K * (uint64_t)a.lda * 2u), (uint32_t)((uint64_t)plan->N * (uint64_t)a.ldc * 2u),
                       whole && (int64_t)a.M * plan->N * 2 > kBwLineBytes, whole);
    TW_HIP(hipGetLastError());
    return TW_OK;
}

// Up to three steps either kernel takes the plan.  The one whose waves store 64 rows themselves is ahead without a long
// activation, where its workgroups, two to a compute unit, come out even, every 32 rows of a column of C are whole
// sectors of memory, and (us of it against the wider one, M 4096 .. 16384, N 900 .. 8192, 1500 problems)
// - one step, 32 to 90 MB of output (0.88 - 0.99 of the time in the mean of a size; N 4096, M 10240: 16.2 against 18.6; from
//   there on, where the wider one stores whole lines, 1.02 - 1.7), or to 128 MB where C's columns are a multiple of 16 KB apart
//   (N 8192, M 8192: 0.71; N 4096, M 16384: 0.83);
// - two steps, the same stride and 112 to 128 MB (N 4096, M 16384 40.9 against 48.3; M 16320 1.09; N 8192, M 8192 0.95; 256 MB 1.15).
// Three steps: the wider one (1.06 - 1.7, N 4096, M 14336 1.39).
bool bs_wide(const tw_plan *plan, int M, const void *C, int64_t ldc, int act)
{
    const int ns = std::max(1, plan->max_k_pad / kBlockK);
    if (ns > kBsMaxSteps)
        return true;
    if ((uint64_t)plan->N * (uint64_t)ldc * 2u >= kBwMaxBytes)
        return false;
    const int64_t mb = (int64_t)1 << 20, out_bytes = (int64_t)M * plan->N * 2, wgs2 = (int64_t)plan->n_units * bs_ranges(plan, M, 2);
    const int64_t slots2 = 2 * (int64_t)plan->cu_count, all2 = (wgs2 + slots2 - 1) / slots2 * slots2;
    if ((act != TW_ACT_NONE && act != TW_ACT_RELU) || wgs2 * 10 < all2 * 9 || !bs_whole_sectors(C, ldc))
        return true;
    const bool far_stride = ldc * 2 % 16384 == 0;
    if (ns == 1)
        return !(out_bytes >= 32 * mb && (out_bytes <= kBwLineBytes || (far_stride && out_bytes <= 128 * mb)));
    return !(ns == 2 && far_stride && out_bytes > 112 * mb && out_bytes <= 128 * mb);
}

int launch_bs(const tw_plan *plan, const GemmArgs &a, int per_cu, bool wide, hipStream_t s)
{
    // (per_cu <= 0: as many workgroups per compute unit as the kernel is built for)
    const int ns = std::max(1, plan->max_k_pad / kBlockK);
    const int pc = per_cu > 0 ? per_cu : kBsPerCu;
    const bool f16 = plan->dtype == TW_F16;
    if (!wide) {
        if (ns <= 2)
            return f16 ? launch_bs_t<TW_F16, 2>(plan, a, pc, s) : launch_bs_t<TW_BF16, 2>(plan, a, pc, s);
        return f16 ? launch_bs_t<TW_F16, 3>(plan, a, pc, s) : launch_bs_t<TW_BF16, 3>(plan, a, pc, s);
    }
    if (ns <= 2)
        return f16 ? launch_bw<TW_F16, 2>(plan, a, per_cu, s) : launch_bw<TW_BF16, 2>(plan, a, per_cu, s);
    if (ns == 3)
        return f16 ? launch_bw<TW_F16, 3>(plan, a, per_cu, s) : launch_bw<TW_BF16, 3>(plan, a, per_cu, s);
    if (ns == 4)
        return f16 ? launch_bw<TW_F16, 4>(plan, a, per_cu, s) : launch_bw<TW_BF16, 4>(plan, a, per_cu, s);
    return f16 ? launch_bw<TW_F16, 6>(plan, a, per_cu, s) : launch_bw<TW_BF16, 6>(plan, a, per_cu, s);
}

} // namespace tw
