// Device-side helpers shared by the GEMM kernels of libtwgemm: element types and MFMA wrappers,
// the output store, the fused epilogue's arithmetic, the unit descriptor fetch.
#pragma once

#include "tw_internal.h"

#include <cstddef>

namespace tw {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

#define TW_LDS(T) __attribute__((address_space(3))) T *
#define TW_GLOBAL(T) __attribute__((address_space(1))) T *

#ifndef TW_A_PAD
#define TW_A_PAD 32 // halfs of padding per staged A row: 64 B, so that the 4 rows x 2 column
                    // halves one transposed read touches fall into 8 distinct 32-byte bank groups
#endif

template <int DT> struct Elem;
template <> struct Elem<TW_F16> {
    static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t to_bits(float f)
    {
        return __builtin_bit_cast(uint16_t, (_Float16)f);
    }
    // two neighbours in one register: v_cvt_pk_f16_f32, nearest even
    static __device__ __forceinline__ uint32_t to_bits2(float lo, float hi)
    {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), f16x2));
    }
    static __device__ __forceinline__ float from_bits(uint16_t h)
    {
        return (float)__builtin_bit_cast(_Float16, h);
    }
};
template <> struct Elem<TW_BF16> {
    static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t to_bits(float f)
    {
        return __builtin_bit_cast(uint16_t, (__bf16)f); // v_cvt_pk_bf16_f32, nearest even
    }
    static __device__ __forceinline__ uint32_t to_bits2(float lo, float hi)
    {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
    }
    static __device__ __forceinline__ float from_bits(uint16_t h)
    {
        return __uint_as_float((uint32_t)h << 16);
    }
};

// 16-byte chunk of column c, rows m..m+7 of a K-major matrix, honouring the M edge.  With
// `through` the store writes through to memory (sc0 sc1) and does not linger in the caches (nt):
// C is written once and not read again by this launch, and lines left dirty in the L2s would
// otherwise all be written back after the last wave has ended, where nothing overlaps them.  A
// small output is better left in the L2s: that write-back is short then, and shorter than the
// last stores' way to memory.
__device__ __forceinline__ void store_chunk(uint16_t *dst, u32x4 v, int m, int M, bool through)
{
    if (m + 8 <= M) {
        if (through)
            asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt\n\ts_nop 1" ::"v"(dst), "v"(v) : "memory");
        else
            *reinterpret_cast<u32x4 *>(dst) = v;
    } else if (m < M) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        for (int e = 0; e < M - m; ++e)
            dst[e] = (uint16_t)(w[e >> 1] >> ((e & 1) * 16));
    }
}

// Activation of the fused epilogue (tw_gemm_ex): the activations the reference's dense layers
// can be given (get_activation, Pruning/BERT/utils/modeling.py:280-305); GELU in its tanh form
// (modeling.py:264-277).
__device__ __forceinline__ float tw_activate(float v, int act)
{
    if (act == TW_ACT_RELU)
        return v > 0.0f ? v : 0.0f;
    // v_exp_f32 (a power of two) and v_rcp_f32, 1 ulp each, with log2(e) folded into the constants:
    // exact limits at +-inf, ~1e-6 relative error in between, far below the 16-bit rounding.  An
    // epilogue is bound by these instructions once its stores are not (33.5 M GELUs are 0.5 M
    // wave-instructions of each kind, a quarter-rate one taking 16 cycles), so GELU is
    //   0.5 v (1 + tanh u) = v / (1 + exp(-2u)),  u = sqrt(2/pi) (v + 0.044715 v^3):
    // five full-rate instructions and the two quarter-rate ones.
    if (act == TW_ACT_GELU) {
        const float t = v * __builtin_fmaf(-0.1029432396f, v * v, -2.302208198f); // -2u log2(e)
        return v * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t));
    }
    if (act == TW_ACT_TANH)
        return 1.0f - 2.0f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(2.885390082f * v) + 1.0f);
    return v;
}
// the same for a handful of values with the test of `act` outside the loop over them
template <int N> __device__ __forceinline__ void tw_activate_all(float (&v)[N], int act)
{
    if (act == TW_ACT_RELU) {
#pragma unroll
        for (int e = 0; e < N; ++e)
            v[e] = tw_activate(v[e], TW_ACT_RELU);
    } else if (act == TW_ACT_GELU) {
#pragma unroll
        for (int e = 0; e < N; ++e)
            v[e] = tw_activate(v[e], TW_ACT_GELU);
    } else if (act == TW_ACT_TANH) {
#pragma unroll
        for (int e = 0; e < N; ++e)
            v[e] = tw_activate(v[e], TW_ACT_TANH);
    }
}
// The value of an output element is rounded to fp32 before it is rounded to 16 bits, in every
// kernel: left to itself the compiler turns "multiply, add, convert" into one fused instruction
// with a single rounding in some epilogues and not in others, and the kernels then differ in the
// last bit of about one element in twenty thousand.
__device__ __forceinline__ float tw_fp32_value(float v)
{
    asm volatile("" : "+v"(v));
    return v;
}
// alpha*acc + beta*C is already in `v`: adds the bias of column c and applies the activation
__device__ __forceinline__ float tw_finish(float v, const float *bias, int c, int act)
{
    if (bias)
        v += bias[c];
    return tw_activate(v, act);
}

// Piece `uv` of the unit table: unit uv / n_split, its columns [j * w, (j + 1) * w) with
// w = 32 * piece_nb and j = uv % n_split.  A piece beyond the unit's columns keeps valid
// offsets and has n_cnt == 0: it runs like any other and stores nothing.  The descriptor is
// workgroup-uniform and ends up in scalar registers.
__device__ __forceinline__ UnitDev unit_piece(const GemmArgs &p, int uv, int ui, const int32_t (&w)[12])
{
    static_assert(sizeof(UnitDev) == 48, "UnitDev is read as 12 words");
    UnitDev u;
    __builtin_memcpy(&u, w, sizeof(UnitDev));
    if (p.n_split > 1) {
        const int j = uv - ui * p.n_split;
        const int bps = p.piece_nb; // 32-column blocks per piece
        const int nb = min(max(u.nb_cnt - j * bps, 0), bps);
        const int nc = min(max(u.n_cnt - j * bps * kMfmaN, 0), bps * kMfmaN);
        if (nb > 0) {
            u.nb0 += j * bps;
            u.kn_off += j * bps * kMfmaN;
        }
        u.nb_cnt = nb;
        u.n_cnt = nc;
    }
    return u;
}
__device__ __forceinline__ UnitDev load_unit(const GemmArgs &p, int uv)
{
    const int ui = uv / p.n_split;
    int32_t w[12];
    if (p.n_arg_units) {
        // from the kernel-argument segment: scalar loads, no global round trip
        const auto *ka = (const __attribute__((address_space(4))) int32_t *)
            __builtin_amdgcn_kernarg_segment_ptr();
#pragma unroll
        for (int i = 0; i < 12; ++i)
            w[i] = ka[offsetof(GemmArgs, arg_units) / 4 + ui * 12 + i];
    } else {
        // the address is workgroup-uniform and the table is constant: scalar loads
        const auto *gu = (const __attribute__((address_space(4))) int32_t *)(uintptr_t)(p.units + ui);
#pragma unroll
        for (int i = 0; i < 12; ++i)
            w[i] = gu[i];
    }
#pragma unroll
    for (int i = 0; i < 12; ++i)
        w[i] = __builtin_amdgcn_readfirstlane(w[i]);
    return unit_piece(p, uv, ui, w);
}
// The same in two parts: word `lane` of the unit of piece `uv`, by a vector load, and the piece out of the wave's words.
__device__ __forceinline__ int unit_word(const GemmArgs &p, int uv, int lane)
{
    const int ui = uv / p.n_split;
    return reinterpret_cast<const int32_t *>(p.units + ui)[lane < 12 ? lane : 0];
}
__device__ __forceinline__ UnitDev unit_of_words(const GemmArgs &p, int uv, int words)
{
    int32_t w[12];
#pragma unroll
    for (int i = 0; i < 12; ++i)
        w[i] = __builtin_amdgcn_readlane(words, i);
    return unit_piece(p, uv, uv / p.n_split, w);
}

// Workgroup barrier for hand-overs through LDS only: waits for this wave's LDS operations, not
// for its global loads, stores or atomics in flight (which __syncthreads() would do for stores
// and atomics), so prefetched loads, the item's output stores and the ticket atomic keep flying.
#define TW_LDS_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

// Pruned columns (TW_PRUNED_ZERO) receive act(beta * C + bias).  A tile, its columns and their bias are a chain of three trips to memory, so
// four of them go together: of four tiles, or four stretches of one.  (With a column at a time per thread, and its bias read again for
// every row, what a fill added to the product was, in us, and is: M 6272, K 3072, N 768, half of the columns pruned, 256 x 64 streaming
// kernel 10.9 and 3.8; K 768, N 3072 row-major, A-stationary 26.6 and 10.1; M 1024 7.1 and 3.2; M 6272, K 4096, N 8192, row-major streaming 85 and 28;
// a tenth pruned, M 6272, K 3072, N 768 3.6 and 2.0.)

// Added where there is no bias: the zero that leaves every value as it is, -0 too.
constexpr float kNoBias = -0.0f;

// Tile z of the fill table, or, past the end, one without columns.
__device__ __forceinline__ TileDev fill_tile(const GemmArgs &p, int z)
{
    const int last = p.n_all_u - p.n_gemm_u - 1;
    const auto *const g = (const __attribute__((address_space(4))) int32_t *)(uintptr_t)(p.tiles + (z < last ? z : last));
    return TileDev{g[0], z <= last ? g[1] : 0, g[2], 0};
}
// K-major C, rows [m_lo, m_hi): pieces first[j] + tid, + stride .. of tile t[j], a piece being eight rows of a column.
template <int DT> __device__ __forceinline__ void fill_kmajor(const GemmArgs &p, int act, const TileDev (&t)[4], const int (&first)[4], int stride,
                                                              int m_lo, int m_hi, int tid, bool through)
{
    using E = Elem<DT>;
    if (m_hi <= m_lo)
        return;
    uint16_t *const C = reinterpret_cast<uint16_t *>(p.C);
    const uint32_t per_col = (uint32_t)(m_hi - m_lo + 7) / 8;
    int most = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        most = max(most, t[j].n_pruned * (int)per_col - first[j]);
    for (int k = tid; k < most; k += stride) {
        int c[4], m[4];
        float b[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t i = (uint32_t)(first[j] + k), q = i / per_col;
            const bool in = (int)q < t[j].n_pruned;
            c[j] = in ? t[j].col0 + p.pruned_n[t[j].pn_off + (in ? (int)q : 0)] : -1;
            m[j] = m_lo + (int)(i - q * per_col) * 8;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            b[j] = p.bias ? p.bias[max(c[j], 0)] : kNoBias;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (c[j] < 0)
                continue;
            uint16_t *const dst = C + (int64_t)c[j] * p.ldc + m[j];
            uint32_t h[4];
            if (p.beta == 0.0f) {
                const uint32_t v = E::to_bits(tw_activate(0.0f + b[j], act));
                h[0] = h[1] = h[2] = h[3] = v | v << 16;
            } else {
                h[0] = h[1] = h[2] = h[3] = 0u;
                for (int e = 0; e < 8 && m[j] + e < m_hi; ++e)
                    h[e >> 1] |= E::to_bits(tw_activate(p.beta * E::from_bits(dst[e]) + b[j], act)) << ((e & 1) * 16);
            }
            store_chunk(dst, u32x4{h[0], h[1], h[2], h[3]}, m[j], m_hi, through);
        }
    }
}
// one tile, by NT threads
template <int DT, int NT> __device__ __forceinline__ void fill_kmajor(const GemmArgs &p, int act, const TileDev &t, int m_lo, int m_hi, int tid, bool through)
{
    const TileDev same[4] = {t, t, t, t};
    const int first[4] = {0, NT, 2 * NT, 3 * NT};
    fill_kmajor<DT>(p, act, same, first, 4 * NT, m_lo, m_hi, tid, through);
}
// tiles z0, z0 + step, .. of the table
template <int DT, int NT> __device__ __forceinline__ void fill_kmajor_tiles(const GemmArgs &p, int z0, int step, int m_lo, int m_hi, int tid, bool through)
{
    const int n = p.n_all_u - p.n_gemm_u;
    const int first[4] = {0, 0, 0, 0};
    for (int z = z0; z < n; z += 4 * step) {
        const TileDev t[4] = {fill_tile(p, z), fill_tile(p, z + step), fill_tile(p, z + 2 * step), fill_tile(p, z + 3 * step)};
        fill_kmajor<DT>(p, p.act, t, first, NT, m_lo, m_hi, tid, through);
    }
}
// Row-major C, tiles z0, z0 + step, .. by NT threads: a lane keeps its column of each of four tiles, and with it the value where C is not
// read, and walks down the rows.
template <int DT, int NT> __device__ __forceinline__ void fill_rowmajor_tiles(const GemmArgs &p, int z0, int step, int m_lo, int m_hi, int tid)
{
    using E = Elem<DT>;
    uint16_t *const C = reinterpret_cast<uint16_t *>(p.C);
    const int n = p.n_all_u - p.n_gemm_u;
    for (int z = z0; z < n; z += 4 * step) {
        const TileDev t[4] = {fill_tile(p, z), fill_tile(p, z + step), fill_tile(p, z + 2 * step), fill_tile(p, z + 3 * step)};
        const int most = max(max(t[0].n_pruned, t[1].n_pruned), max(t[2].n_pruned, t[3].n_pruned));
        int lg = 0; // 2^lg columns side by side
        while (lg < 6 && 1 << lg < most)
            ++lg;
        for (int base = 0; base < most; base += 1 << lg) {
            const int q = base + (tid & ((1 << lg) - 1));
            int c[4];
            float b[4];
            uint16_t v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                c[j] = q < t[j].n_pruned ? t[j].col0 + p.pruned_n[t[j].pn_off + q] : -1;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                b[j] = p.bias ? p.bias[max(c[j], 0)] : kNoBias;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = (uint16_t)E::to_bits(tw_activate(0.0f + b[j], p.act));
            for (int m = m_lo + (tid >> lg); m < m_hi; m += NT >> lg) {
                uint16_t *const row = C + (int64_t)m * p.ldc;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (c[j] < 0)
                        continue;
                    row[c[j]] = p.beta == 0.0f ? v[j] : (uint16_t)E::to_bits(tw_activate(p.beta * E::from_bits(row[c[j]]) + b[j], p.act));
                }
            }
        }
    }
}

// Over the lanes of a wave, in registers: a step through LDS (__shfl) is some 60 cycles, and a selection or an ordered list is a chain of them.
// (row_shr 1, 2, 4, 8 inside rows of 16 lanes, then the last lane of a row to the next row, of the second row to the upper half; a lane
// that gets nothing keeps `none`)
template <class F> __device__ __forceinline__ uint32_t wave_steps(uint32_t x, uint32_t none, F f)
{
    x = f(x, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)x, 0x111, 0xF, 0xF, false));
    x = f(x, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)x, 0x112, 0xF, 0xF, false));
    x = f(x, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)x, 0x114, 0xF, 0xF, false));
    x = f(x, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)x, 0x118, 0xF, 0xF, false));
    x = f(x, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)x, 0x142, 0xA, 0xF, false));
    return f(x, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)x, 0x143, 0xC, 0xF, false));
}
__device__ __forceinline__ uint32_t last_lane(uint32_t x) { return (uint32_t)__builtin_amdgcn_readlane((int)x, 63); }
__device__ __forceinline__ uint32_t wave_min(uint32_t x)
{
    return last_lane(wave_steps(x, 0xFFFFFFFFu, [](uint32_t a, uint32_t b) { return min(a, b); }));
}
__device__ __forceinline__ uint32_t wave_max(uint32_t x)
{
    return last_lane(wave_steps(x, 0u, [](uint32_t a, uint32_t b) { return max(a, b); }));
}
// sums over the lanes up to this one
__device__ __forceinline__ uint32_t wave_scan(uint32_t x)
{
    return wave_steps(x, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ unsigned long long wave_scan(unsigned long long x)
{
    auto step = [&](auto ctrl, auto rows) {
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, decltype(ctrl)::value, decltype(rows)::value, 0xF, false);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(x >> 32), decltype(ctrl)::value, decltype(rows)::value, 0xF, false);
        x += (unsigned long long)hi << 32 | lo;
    };
    step(std::integral_constant<int, 0x111>(), std::integral_constant<int, 0xF>());
    step(std::integral_constant<int, 0x112>(), std::integral_constant<int, 0xF>());
    step(std::integral_constant<int, 0x114>(), std::integral_constant<int, 0xF>());
    step(std::integral_constant<int, 0x118>(), std::integral_constant<int, 0xF>());
    step(std::integral_constant<int, 0x142>(), std::integral_constant<int, 0xA>());
    step(std::integral_constant<int, 0x143>(), std::integral_constant<int, 0xC>());
    return x;
}

} // namespace tw
