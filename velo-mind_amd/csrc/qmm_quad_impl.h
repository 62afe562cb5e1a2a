// Quantized matmul for rows_m > 4 on gfx950 MFMA, weights straight from
// global memory into MFMA operand registers.
//
// C[M, N] = A[M, K] * W[K, N], W the reference's codes (N contiguous) and
// fp32 scales; fp32 accumulation.
//
// Operands
//   B   A lane loads 4 adjacent columns x 8 K rows of codes as dwords (INT8
//       eight, INT4 four, each a 128- or 64-byte run across the lanes of one
//       K group), and v_perm_b32 gathers each column's codes into the lane's
//       operand of one MFMA column tile: tile c of four holds columns 4 i + c.
//       So one set of loads feeds four MFMA column tiles, the weights never
//       pass through LDS, and a lane's results are four adjacent columns of
//       each of its rows (one 16-byte store).
//   A   fp32: two fp16 parts of a row scaled by a power of two, staged by a
//       prep kernel or a producer (a_split.h) in operand order (AM_PIECES) or
//       row-major (AM_ROWS).  (Splitting in this kernel instead, after every
//       workgroup has scanned A for its row maxima, is slower than the extra
//       launch: M = 16, K = 2048, N = 5632 INT4 12.6 us against 8.75.)
//       fp16, bf16: one part as it is, row-major (AM_ROWS) or in operand
//       order, times codes that are exact in the same type.
// Work
//   wave       BM = TILE * MT rows x NT = 4 * TILE columns over its own run of
//              32-row K chunks; waves split K, so the main loop has no barrier
//              and no LDS traffic
//   workgroup  W waves: NW side by side in N (large calls: A's lines are then
//              shared in L1), KW splitting K; the KW sums meet in LDS in wave
//              order
//   split      further K splits across workgroups; partial tiles go to the
//              stream's workspace and the last workgroup of a tile adds them
//              in split order (results do not depend on scheduling)
// Block scales multiply each 32-row chunk's fp32 sum, as the reference
// multiplies each block's (quantized_matmul.cpp:76-90); codes are exact in
// fp16.
// Shared by qmm_quad.hip (fp32) and qmm_quad_half.hip (fp16, bf16), which
// instantiate their kernels side by side.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

#include "a_split.h"
#include "qmm_kernels.h"
#include "vm_device.h"
#include "vm_internal.h"

namespace vmhip {
namespace {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));


enum AMode { AM_PIECES = 0, AM_ROWS = 1 };
// What A and C hold: fp32 (A as two fp16 parts), fp16 or bf16.
enum Elem { EL_F32 = 0, EL_F16 = 1, EL_BF16 = 2 };

template <int TILE>
struct Mfma;
template <>
struct Mfma<32> {
    using Acc = floatx16;
    static constexpr int kElems = 16;
    static constexpr int kK = 16;
    template <int EL>
    static __device__ __forceinline__ Acc run(half8v a, half8v b, Acc c) {
        if constexpr (EL == EL_BF16)
            return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                           c, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    // row of element v in lane group h
    static __device__ __forceinline__ int row(int v, int h) { return 8 * (v / 4) + 4 * h + v % 4; }
};
template <>
struct Mfma<16> {
    using Acc = floatx4;
    static constexpr int kElems = 4;
    static constexpr int kK = 32;
    template <int EL>
    static __device__ __forceinline__ Acc run(half8v a, half8v b, Acc c) {
        if constexpr (EL == EL_BF16)
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                           c, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int v, int h) { return 4 * h + v; }
};

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}

// INT8: codes of rows i and j (dword x, y: four columns each) of column C as
// two fp16: bytes [x.C, 0, y.C, 0] ^ 0x6480 = 1024 + 128 + code, minus 1152.
template <int C>
__device__ __forceinline__ uint32_t pair8(uint32_t x, uint32_t y) {
    const uint32_t t = perm(y, x, 0x0c000c00u | ((4u + C) << 16) | C) ^ 0x64806480u;
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, t) - half2v{1152.0f16, 1152.0f16});
}

// INT4: byte rows x, y (K rows 2i, 2i+1 and 2j, 2j+1; nibbles already ^ 8) of
// column C: the even rows (low nibbles) and the odd rows (high nibbles) as
// two fp16 each.  The high nibbles stay where they are: 1024 + 16 * nibble,
// times 1/16, minus 72 (exact in fp16).
// `magic` is 0x64006400 in a vector register: v_and_or_b32 takes one scalar.
template <int C>
__device__ __forceinline__ void pair4(uint32_t x, uint32_t y, uint32_t magic, uint32_t& even, uint32_t& odd) {
    const uint32_t t = perm(y, x, 0x0c000c00u | ((4u + C) << 16) | C);
    const half2v lo = __builtin_bit_cast(half2v, (t & 0x000F000Fu) | magic);
    const half2v hi = __builtin_bit_cast(half2v, (t & 0x00F000F0u) | magic);
    even = __builtin_bit_cast(uint32_t, lo - half2v{1032.0f16, 1032.0f16});
    odd = __builtin_bit_cast(uint32_t, hi * half2v{0.0625f16, 0.0625f16} + half2v{-72.0f16, -72.0f16});
}

// bf16: signed bytes of column C of x and y converted to fp32 (exact) and cut
// to their upper halves (exact: at most 8 significant bits).
template <int C>
__device__ __forceinline__ uint32_t pair_bf16(uint32_t x, uint32_t y) {
    const float fx = static_cast<float>(static_cast<int8_t>(x >> (8 * C)));
    const float fy = static_cast<float>(static_cast<int8_t>(y >> (8 * C)));
    return perm(__float_as_uint(fy), __float_as_uint(fx), 0x07060302u);
}

// The lane's eight codes of column C in the order k = 0, 4, 1, 5, 2, 6, 3, 7
// (the order A is staged in).
// (bf16 INT4: sixteen times the codes, taken out once per output).
template <int KIND, int EL, int C>
__device__ __forceinline__ half8v unpack_column(const uint32_t (&w)[KIND == 2 ? 4 : 8], uint32_t magic) {
    u32x4 o;
    if constexpr (KIND == 2 && EL == EL_BF16) {
        // each nibble at the top of a byte: a signed byte of 16 * code
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo[i] = (w[i] << 4) & 0xF0F0F0F0u;
            hi[i] = w[i] & 0xF0F0F0F0u;
        }
        o[0] = pair_bf16<C>(lo[0], lo[2]);
        o[1] = pair_bf16<C>(hi[0], hi[2]);
        o[2] = pair_bf16<C>(lo[1], lo[3]);
        o[3] = pair_bf16<C>(hi[1], hi[3]);
    } else if constexpr (EL == EL_BF16) {
        o[0] = pair_bf16<C>(w[0], w[4]);
        o[1] = pair_bf16<C>(w[1], w[5]);
        o[2] = pair_bf16<C>(w[2], w[6]);
        o[3] = pair_bf16<C>(w[3], w[7]);
    } else if constexpr (KIND == 2) {
        uint32_t e, d;
        pair4<C>(w[0], w[2], magic, e, d);
        o[0] = e;
        o[1] = d;
        pair4<C>(w[1], w[3], magic, e, d);
        o[2] = e;
        o[3] = d;
    } else {
        o[0] = pair8<C>(w[0], w[4]);
        o[1] = pair8<C>(w[1], w[5]);
        o[2] = pair8<C>(w[2], w[6]);
        o[3] = pair8<C>(w[3], w[7]);
    }
    return __builtin_bit_cast(half8v, o);
}

// Row-major 8-groups (k = 0..7) in the order the codes are unpacked.
__device__ __forceinline__ half8v piece_order(u32x4 v) {
    return __builtin_bit_cast(half8v, u32x4{perm(v[2], v[0], 0x05040100u), perm(v[2], v[0], 0x07060302u),
                                            perm(v[3], v[1], 0x05040100u), perm(v[3], v[1], 0x07060302u)});
}

template <int EL>
__device__ __forceinline__ float widen(uint32_t h) {   // the low 16 bits
    if constexpr (EL == EL_BF16) return __uint_as_float(h << 16);
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(h)));
}

struct QuadArgs {
    const void* a;
    const int* row_exp;
    const uint8_t* wq;
    const void* scale;
    void* c;
    float* partials;
    unsigned* counters;
    int m, k, n;
    int block_chunks;       // 32-row chunks per scale block
    int chunks;             // of K
    int chunks_per_wave;
    int tiles_n, tiles_m;
    int panel;              // row tiles of a panel
    uint32_t a_bytes, lo_offset, code_bytes, scale_bytes;
    int c_vec;
};

// KIND: 0 = INT8 per column, 1 = INT8 blockwise, 2 = INT4 blockwise.
template <int KIND, int TILE, int MT, int W, int NW, int AM, int EL, bool SH, int D>
struct QuadCfg {
    using M = Mfma<TILE>;
    static constexpr int PARTS = EL == EL_F32 ? 2 : 1;
    static constexpr int BM = TILE * MT;
    static constexpr int KW = W / NW;                     // waves that split K
    static constexpr int WT = 4 * TILE;                   // columns of a wave
    static constexpr int NT = NW * WT;                    // and of the workgroup
    // K rows per pipeline stage: a scale block's granularity, else one MFMA
    static constexpr int kChunk = KIND != 0 ? 32 : M::kK;
    static constexpr int Q = kChunk / M::kK;              // MFMA K steps per chunk
    static constexpr int kWords = KIND == 2 ? 4 : 8;
    static constexpr bool kBlock = KIND != 0;
    static constexpr int kItems = MT * M::kElems;         // float4 results per lane
    // items of a wave that meet in LDS at a time: all of them while 64 KB hold them
    static constexpr int kPhase = kItems * W * 1024 <= 64 * 1024 ? kItems : 64 / W;
    static constexpr int kLdsBytes = kPhase * W * 1024;
    static constexpr int kRegs = kItems * 4 + D * (MT * Q * 4 * PARTS + Q * kWords + (kBlock ? 4 : 0)) +
                                 (kBlock ? 2 * MT * M::kElems : 0) + Q * 8 + 16;
    static constexpr int kWavesPerEu = W >= 8 ? 2 : kRegs <= 256 ? 2 : 1;
    static_assert(kItems % kPhase == 0 && (kPhase % KW == 0 || kPhase < KW), "phases split the items, waves split a phase");
};

template <int KIND, int TILE, int MT, int W, int NW, int AM, int EL, bool SH, int D>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(QuadCfg<KIND, TILE, MT, W, NW, AM, EL, SH, D>::kWavesPerEu,
                                                                        QuadCfg<KIND, TILE, MT, W, NW, AM, EL, SH, D>::kWavesPerEu)))
void qmm_quad_kernel(const QuadArgs g) {
    using C = QuadCfg<KIND, TILE, MT, W, NW, AM, EL, SH, D>;
    using M = typename C::M;
    using Acc = typename M::Acc;
    constexpr int PARTS = C::PARTS;
    __shared__ __attribute__((aligned(16))) float4 red[C::kLdsBytes / 16];
    __shared__ unsigned ticket;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lc = lane % TILE;    // operand row of A, column quad of B
    const int lg = lane / TILE;    // 8-row K group
    // Grid over (split, row panel, tile column, tile row), row fastest;
    // workgroups go to the 8 XCDs round-robin by id, and renumbering gives each
    // XCD a contiguous run, so that the workgroups of one L2 share weight
    // columns and, in panels (launch_quad), A as well: a run over all rows of a
    // large A reads it whole from beyond the L2 (2048 rows of 2048 x 2048 INT8
    // 69.7 us in one panel, 49.3 in panels of 512 rows, 48.1 of 256).
    int lin = blockIdx.x;
    {
        const int full = static_cast<int>(gridDim.x) & ~7;
        if (lin < full) lin = (lin & 7) * (full >> 3) + (lin >> 3);
    }
    const int split = lin / (g.tiles_n * g.tiles_m);
    const int in_split = lin - split * g.tiles_n * g.tiles_m;
    int panel = 0, in_panel = in_split, panel_rows = g.tiles_m;
    if (EL == EL_F32 && g.panel < g.tiles_m) {   // (16-bit A: one panel)
        panel = in_split / (g.panel * g.tiles_n);
        in_panel = in_split - panel * g.panel * g.tiles_n;
        panel_rows = min(g.panel, g.tiles_m - panel * g.panel);
    }
    const int tile_x = in_panel / panel_rows;
    const int tile_y = panel * g.panel + in_panel - tile_x * panel_rows;
    const int splits = static_cast<int>(gridDim.x) / (g.tiles_n * g.tiles_m);
    const int n = g.n, m = g.m;
    const int m0 = tile_y * C::BM;
    // The lane's four columns; a quad that would cross the row's end moves
    // back to end with it (its first columns are then the quad before's).
    const int wn = wave % NW, wk = wave / NW;
    const int col = tile_x * C::NT + wn * C::WT + 4 * lc;
    const int cs = min(col, n - 4);
    const int c_begin = min((split * C::KW + wk) * g.chunks_per_wave, g.chunks);
    const int c_end = min(c_begin + g.chunks_per_wave, g.chunks);

    const __amdgpu_buffer_rsrc_t ars = buffer_rsrc(g.a, g.a_bytes);
    const __amdgpu_buffer_rsrc_t wrs = buffer_rsrc(g.wq, g.code_bytes);
    const __amdgpu_buffer_rsrc_t srs = buffer_rsrc(g.scale, g.scale_bytes);

    struct Stage {
        u32x4 a[MT][C::Q][PARTS];
        uint32_t w[C::Q][C::kWords];
        u32x4 s;
    };

    // Byte offsets of the lane's next loads, advanced by one chunk per load:
    // A pieces (rows past the matrix start past the buffer and read zeros),
    // codes, and the scale block of the next chunk.  Loads may run past the
    // wave's run, into rows that are not used, or past the buffers, which
    // reads zeros.
    constexpr uint32_t kKBytes = AM == AM_PIECES ? 64u : 2u;   // bytes from one k to the next (operand order: of 32 rows)
    uint32_t a_next[MT][PARTS];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int row = m0 + t * TILE + lc;
        uint32_t off;
        if constexpr (AM == AM_PIECES)
            off = static_cast<uint32_t>(row / 32) * static_cast<uint32_t>(g.k) * 64u + (row % 32) * 16u + lg * 512u +
                  static_cast<uint32_t>(c_begin) * (64u * C::kChunk);
        else
            off = (static_cast<uint32_t>(row) * static_cast<uint32_t>(g.k) + lg * 8u +
                   static_cast<uint32_t>(c_begin) * C::kChunk) * 2u;
#pragma unroll
        for (int p = 0; p < PARTS; ++p) a_next[t][p] = row < m ? off + p * g.lo_offset : g.a_bytes;
    }
    const uint32_t un = static_cast<uint32_t>(n);
    constexpr uint32_t kRowsPerChunk = KIND == 2 ? C::kChunk / 2 : C::kChunk;   // code byte rows
    uint32_t w_next = (static_cast<uint32_t>(c_begin) * kRowsPerChunk + C::kWords * lg) * un + cs;
    int blk = 0, blk_rem = 0;
    if constexpr (C::kBlock) {
        blk = __builtin_amdgcn_readfirstlane(c_begin / g.block_chunks);
        blk_rem = c_begin - blk * g.block_chunks;
    }

    auto load = [&](Stage& st) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int p = 0; p < PARTS; ++p) {
#pragma unroll
                for (int q = 0; q < C::Q; ++q) {
                    st.a[t][q][p] = buffer_load16(ars, a_next[t][p] + q * kKBytes * M::kK);
                }
                a_next[t][p] += kKBytes * C::kChunk;
            }
#pragma unroll
        for (int q = 0; q < C::Q; ++q)
#pragma unroll
            for (int i = 0; i < C::kWords; ++i)
                st.w[q][i] = buffer_load4(wrs, w_next + (q * (kRowsPerChunk / C::Q) + i) * un);
        w_next += kRowsPerChunk * un;
        if constexpr (C::kBlock) {
            if constexpr (SH) {
                const auto h = __builtin_amdgcn_raw_buffer_load_b64(
                    srs, static_cast<int>((static_cast<uint32_t>(blk) * un + cs) * 2u), 0, 0);
                st.s[0] = h[0];
                st.s[1] = h[1];
            } else {
                st.s = buffer_load16(srs, (static_cast<uint32_t>(blk) * un + cs) * 4u);
            }
            const int wrap = ++blk_rem == g.block_chunks ? 1 : 0;
            blk += wrap;
            blk_rem = wrap ? 0 : blk_rem;
        }
    };

    Acc acc[4][MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int e = 0; e < M::kElems; ++e) acc[c][t][e] = 0.0f;

    uint32_t magic = 0;
    if constexpr (KIND == 2 && EL != EL_BF16) asm("v_mov_b32 %0, 0x64006400" : "=v"(magic));
    // One column tile of a chunk: the codes of column c unpacked, then its MFMAs.
    struct Col {
        half8v b[C::Q];
    };
    auto unpack = [&](const Stage& st, Col& o, auto ic) {
#pragma unroll
        for (int q = 0; q < C::Q; ++q) {
            uint32_t w[C::kWords];
#pragma unroll
            for (int i = 0; i < C::kWords; ++i) w[i] = KIND == 2 && EL != EL_BF16 ? st.w[q][i] ^ 0x88888888u : st.w[q][i];
            o.b[q] = unpack_column<KIND, EL, decltype(ic)::value>(w, magic);
        }
    };
        // A's operands of a stage
    struct Operand {
        half8v v[MT][C::Q][PARTS];
    };
    auto operand = [&](const Stage& st, Operand& o) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int q = 0; q < C::Q; ++q) {
#pragma unroll
                    for (int p = 0; p < PARTS; ++p)
                        o.v[t][q][p] = AM == AM_PIECES ? __builtin_bit_cast(half8v, st.a[t][q][p]) : piece_order(st.a[t][q][p]);
            }
    };
    auto multiply = [&](const Operand& a, const Col& o, Acc* to) {
#pragma unroll
        for (int q = 0; q < C::Q; ++q)
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
#pragma unroll
                for (int t = 0; t < MT; ++t) to[t] = M::template run<EL>(a.v[t][q][p], o.b[q], to[t]);
    };
    auto scale_add = [&](const Stage& st, const Acc* part, int c) {
        const float s = SH ? widen<EL>(st.s[c / 2] >> (16 * (c % 2))) : __uint_as_float(st.s[c]);
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int e = 0; e < M::kElems; ++e) acc[c][t][e] = fmaf(part[t][e], s, acc[c][t][e]);
    };
    auto zero = [&](Acc* part) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int e = 0; e < M::kElems; ++e) part[t][e] = 0.0f;
    };
    // Instruction order of a region: its MFMAs, each followed by a share of
    // the VALU work and of the loads (left alone, the compiler issues the
    // loads of every stage together at the end of the loop body, which leaves
    // them no time to arrive).
    auto interleave = [&](auto mf, auto va, auto vm) {
        constexpr int kMf = decltype(mf)::value, kVa = decltype(va)::value, kVm = decltype(vm)::value;
#pragma unroll
        for (int i = 0; i < kMf; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
            for (int l = i * kVm / kMf; l < (i + 1) * kVm / kMf; ++l) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, kVa, 0);
        }
    };
    using std::integral_constant;
    constexpr int kColMfma = MT * PARTS * C::Q;
    constexpr int kLoads = MT * PARTS * C::Q + C::Q * C::kWords + (C::kBlock ? 1 : 0);
    Stage st[D];
    Col b0, b1;
    Acc p0[C::kBlock ? MT : 1], p1[C::kBlock ? MT : 1];
    // One stage: its four columns' MFMAs, the refill of the stage used before
    // it, and the first column of the stage after it unpacked.  Blockwise:
    // column c's products go to a fresh accumulator; while they run, column
    // c - 1's are scaled and added.
    auto step = [&](auto iu, auto refill) {
        constexpr int u = decltype(iu)::value;
        const Stage& cur = st[u];
        const Stage& next = st[(u + 1) % D];
        Operand a;
        operand(cur, a);
        if constexpr (decltype(refill)::value) load(st[(u + D - 1) % D]);
        if constexpr (C::kBlock) {
            zero(p0);
            multiply(a, b0, p0);
            unpack(cur, b1, integral_constant<int, 1>{});
            interleave(integral_constant<int, kColMfma>{}, integral_constant<int, 32 / kColMfma + 1>{},
                       integral_constant<int, kLoads>{});
            __builtin_amdgcn_sched_barrier(0);
            zero(p1);
            multiply(a, b1, p1);
            scale_add(cur, p0, 0);
            unpack(cur, b0, integral_constant<int, 2>{});
            interleave(integral_constant<int, kColMfma>{}, integral_constant<int, 7>{}, integral_constant<int, 0>{});
            __builtin_amdgcn_sched_barrier(0);
            zero(p0);
            multiply(a, b0, p0);
            scale_add(cur, p1, 1);
            unpack(cur, b1, integral_constant<int, 3>{});
            interleave(integral_constant<int, kColMfma>{}, integral_constant<int, 7>{}, integral_constant<int, 0>{});
            __builtin_amdgcn_sched_barrier(0);
            zero(p1);
            multiply(a, b1, p1);
            scale_add(cur, p0, 2);
            unpack(next, b0, integral_constant<int, 0>{});
            interleave(integral_constant<int, kColMfma>{}, integral_constant<int, 7>{}, integral_constant<int, 0>{});
            __builtin_amdgcn_sched_barrier(0);
            scale_add(cur, p1, 3);
        } else {
            multiply(a, b0, acc[0]);
            unpack(cur, b1, integral_constant<int, 1>{});
            multiply(a, b1, acc[1]);
            unpack(cur, b0, integral_constant<int, 2>{});
            multiply(a, b0, acc[2]);
            unpack(cur, b1, integral_constant<int, 3>{});
            multiply(a, b1, acc[3]);
            unpack(next, b0, integral_constant<int, 0>{});
            interleave(integral_constant<int, 4 * kColMfma>{}, integral_constant<int, 64 / (4 * kColMfma) + 1>{},
                       integral_constant<int, kLoads>{});
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    static_assert(D == 3 || D == 4, "the loop below");
    // D - 1 stages in flight ahead of the one in use
#pragma unroll
    for (int d = 0; d + 1 < D; ++d) load(st[d]);
    unpack(st[0], b0, integral_constant<int, 0>{});
    int left = c_end - c_begin;
    constexpr integral_constant<bool, true> kRefill{};
    for (; left >= D; left -= D) {
        step(integral_constant<int, 0>{}, kRefill);
        step(integral_constant<int, 1>{}, kRefill);
        if constexpr (D > 2) step(integral_constant<int, 2 % D>{}, kRefill);
        if constexpr (D > 3) step(integral_constant<int, 3 % D>{}, kRefill);
    }
    constexpr integral_constant<bool, false> kLast{};
    if (left > 0) step(integral_constant<int, 0>{}, kLast);
    if constexpr (D > 2)
        if (left > 1) step(integral_constant<int, 1>{}, kLast);
    if constexpr (D > 3)
        if (left > 2) step(integral_constant<int, 2 % D>{}, kLast);

    // ---- epilogue
    auto column_scale = [&]() {
        if constexpr (C::kBlock) {
            return make_float4(1.f, 1.f, 1.f, 1.f);
        } else if constexpr (SH) {
            const auto h = __builtin_amdgcn_raw_buffer_load_b64(srs, static_cast<int>(cs * 2), 0, 0);
            return make_float4(widen<EL>(h[0]), widen<EL>(h[0] >> 16), widen<EL>(h[1]), widen<EL>(h[1] >> 16));
        } else {
            return __builtin_bit_cast(float4, buffer_load16(srs, static_cast<uint32_t>(cs) * 4u));
        }
    };
    const float4 cscale = column_scale();
    // The outputs of one row: four adjacent columns, or the ones of a moved
    // quad that are the lane's own.
    bool lost = false;   // bf16: the lane stored an output that is no number
    auto store_row = [&](int row, const float4& v) {
        if (row >= m || col >= n) return;
        const int64_t at = static_cast<int64_t>(row) * n + cs;
        const float e[4] = {v.x, v.y, v.z, v.w};
        if constexpr (EL == EL_F32) {
            float* o = static_cast<float*>(g.c) + at;
            if (cs == col) {
                __builtin_memcpy(o, &v, 16);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (cs + j >= col) o[j] = e[j];
            }
        } else {
            uint16_t* o = static_cast<uint16_t*>(g.c) + at;
            uint16_t h[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) h[j] = EL == EL_BF16 ? f32_to_bf16_ref(e[j]) : f32_to_f16_ref(e[j]);
            if constexpr (EL == EL_BF16)
                lost = lost || !(fabsf(v.x) + fabsf(v.y) + fabsf(v.z) + fabsf(v.w) <= 3.4028235e38f);
            if (g.c_vec) {   // n % 4 == 0, 8-byte aligned C
                *reinterpret_cast<uint2*>(o) = make_uint2(h[0] | static_cast<uint32_t>(h[1]) << 16,
                                                          h[2] | static_cast<uint32_t>(h[3]) << 16);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (cs + j >= col) o[j] = h[j];
            }
        }
    };
    // partial tiles: [tile][split][item][lane] float4
    const int tile = tile_x * g.tiles_m + tile_y;
    const __amdgpu_buffer_rsrc_t prs =
        buffer_rsrc(g.partials + static_cast<int64_t>(tile * NW + wn) * splits * (C::kItems * 256), 0x7fffffff);
    constexpr int kOwn = (C::kPhase + C::KW - 1) / C::KW;   // items of a phase that a wave adds up
    // (unrolled: the results of a phase leave their registers with it)
#pragma unroll
    for (int ph = 0; ph < C::kItems; ph += C::kPhase) {
        if (ph) __syncthreads();
#pragma unroll
        for (int i = 0; i < C::kItems; ++i)
            if (i >= ph && i < ph + C::kPhase) {
                const int t = i / M::kElems, e = i % M::kElems;
                red[(wave * C::kPhase + (i - ph)) * 64 + lane] =
                    make_float4(acc[0][t][e], acc[1][t][e], acc[2][t][e], acc[3][t][e]);
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kOwn; ++j) {
            const int i = wk * kOwn + j;
            if (C::kPhase < C::KW && i >= C::kPhase) break;
            float4 v = red[(wn * C::kPhase + i) * 64 + lane];
#pragma unroll
            for (int w = 1; w < C::KW; ++w) {
                const float4 x = red[((w * NW + wn) * C::kPhase + i) * 64 + lane];
                v.x += x.x;
                v.y += x.y;
                v.z += x.z;
                v.w += x.w;
            }
            const int item = ph + i;
            const int row = m0 + (item / M::kElems) * TILE + M::row(item % M::kElems, lg);
            v = make_float4(v.x * cscale.x, v.y * cscale.y, v.z * cscale.z, v.w * cscale.w);
            if constexpr (EL == EL_F32) {   // 2^-x undoes the row's staging scale
                const int nx = row < m ? -g.row_exp[row] : 0;
                v = make_float4(ldexpf(v.x, nx), ldexpf(v.y, nx), ldexpf(v.z, nx), ldexpf(v.w, nx));
            } else if constexpr (KIND == 2 && EL == EL_BF16) {
                v = make_float4(v.x * 0.0625f, v.y * 0.0625f, v.z * 0.0625f, v.w * 0.0625f);   // the codes' factor 16
            }
            if (splits == 1) {
                store_row(row, v);
            } else if (row < m) {
                coherent_store16(prs, static_cast<uint32_t>((split * C::kItems + item) * 64 + lane) * 16u,
                                 __builtin_bit_cast(u32x4, v));
            }
        }
    }
    if (splits > 1) {
        publish_partials();
        __syncthreads();
        if (tid == 0) ticket = ticket_take(&g.counters[tile], static_cast<unsigned>(splits));
        __syncthreads();
        if (ticket != static_cast<unsigned>(splits - 1)) return;
        for (int item = wk; item < C::kItems; item += C::KW) {
            const int row = m0 + (item / M::kElems) * TILE + M::row(item % M::kElems, lg);
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            for (int s0 = 0; s0 < splits; s0 += 4) {
                u32x4 x[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    x[u] = s0 + u < splits && row < m
                               ? coherent_load16(prs, static_cast<uint32_t>(((s0 + u) * C::kItems + item) * 64 + lane) * 16u)
                               : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    v.x += __uint_as_float(x[u][0]);
                    v.y += __uint_as_float(x[u][1]);
                    v.z += __uint_as_float(x[u][2]);
                    v.w += __uint_as_float(x[u][3]);
                }
            }
            store_row(row, v);
        }
        if (tid == 0) __hip_atomic_store(&g.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // bf16 has fp32's range, so products with the codes (16 times them for
    // INT4) and their sums can leave fp32 although the outputs do not (|a|
    // from 2.6e36).  Infinities and NaN never turn back into numbers, so an
    // output that is a number is right; one that is not is summed again by
    // the lane that stored it, its row scaled as fp32 rows are when they are
    // staged (a row that itself holds an infinity or NaN stays as it is).
    // Nothing else pays for it (M = 333, 5632 x 2048 INT4 28.9 us with and
    // without); a pass over A for its row maxima would cost every call 2 us.
    if constexpr (EL == EL_BF16) {
        if (!lost) return;
        const int groups = g.chunks * (C::kChunk / 8);
#pragma unroll 1
        for (int item = 0; item < C::kItems; ++item) {
            const int owner = splits > 1 ? item % C::KW : item % C::kPhase / kOwn;
            const int row = m0 + (item / M::kElems) * TILE + M::row(item % M::kElems, lg);
            if (owner != wk || row >= m) continue;
            const uint16_t* c = static_cast<const uint16_t*>(g.c) + static_cast<int64_t>(row) * n + cs;
            bool number = true;
#pragma unroll
            for (int j = 0; j < 4; ++j) number = number && (cs + j < col || (c[j] & 0x7F80u) != 0x7F80u);
            if (number) continue;
            const uint32_t a_at = AM == AM_PIECES
                                      ? static_cast<uint32_t>(row / 32) * static_cast<uint32_t>(g.k) * 64u + (row % 32) * 16u
                                      : static_cast<uint32_t>(row) * static_cast<uint32_t>(g.k) * 2u;
            constexpr uint32_t kGroupBytes = AM == AM_PIECES ? 512u : 16u;
            float mx = 0.0f;
            bool special = false;
#pragma unroll 1
            for (int i = 0; i < groups; ++i) {
                const u32x4 w = buffer_load16(ars, a_at + i * kGroupBytes);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float lo = fabsf(widen<EL>(w[j])), hi = fabsf(widen<EL>(w[j] >> 16));
                    special = special || !(lo <= 3.4028235e38f) || !(hi <= 3.4028235e38f);
                    mx = fmaxf(mx, fmaxf(lo, hi));
                }
            }
            if (special) continue;
            const int x = a_row_exponent(mx);
            float total[4] = {0.f, 0.f, 0.f, 0.f}, part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int i = 0; i < groups; ++i) {
                const u32x4 w = buffer_load16(ars, a_at + i * kGroupBytes);
#pragma unroll
                for (int kk = 0; kk < 8; ++kk) {
                    // operand order holds k at position 2 (k % 4) + k / 4
                    const int p = AM == AM_PIECES ? 2 * (kk % 4) + kk / 4 : kk;
                    const float av = ldexpf(widen<EL>(w[p / 2] >> (16 * (p % 2))), x);
                    const uint32_t at = static_cast<uint32_t>(KIND == 2 ? 4 * i + kk / 2 : 8 * i + kk) * un + cs;
                    const uint32_t codes = buffer_load4(wrs, at);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int b = static_cast<int8_t>(codes >> (8 * j));
                        const int code = KIND != 2 ? b : kk % 2 ? b >> 4 : static_cast<int8_t>(b << 4) >> 4;
                        part[j] = fmaf(av, static_cast<float>(code), part[j]);
                    }
                }
                if (C::kBlock && i % 4 == 3) {   // a 32-row chunk
                    const uint32_t at = static_cast<uint32_t>(i / 4 / g.block_chunks) * un + cs;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float s = SH ? widen<EL>(__builtin_amdgcn_raw_buffer_load_b16(srs, static_cast<int>((at + j) * 2u), 0, 0))
                                           : __uint_as_float(buffer_load4(srs, (at + j) * 4u));
                        total[j] = fmaf(part[j], s, total[j]);
                        part[j] = 0.0f;
                    }
                }
            }
            const float4 f = column_scale();
            const float4 v = C::kBlock ? make_float4(total[0], total[1], total[2], total[3])
                                       : make_float4(part[0] * f.x, part[1] * f.y, part[2] * f.z, part[3] * f.w);
            store_row(row, make_float4(ldexpf(v.x, -x), ldexpf(v.y, -x), ldexpf(v.z, -x), ldexpf(v.w, -x)));
        }
    }
}

template <int KIND, int TILE, int MT, int W, int NW, int AM, int EL, bool SH, int D>
int launch_quad(const GemmOperands& o, int splits, hipStream_t stream) {
    using C = QuadCfg<KIND, TILE, MT, W, NW, AM, EL, SH, D>;
    QuadArgs g{};
    g.a = o.a;
    g.row_exp = o.row_exp;
    g.wq = o.wq;
    g.scale = o.scale;
    g.c = o.c;
    g.m = o.m;
    g.n = o.n;
    const int kp = (o.k + 31) / 32 * 32;   // operand order pads K with zeros
    g.k = AM == AM_PIECES ? kp : o.k;
    g.chunks = (o.k + C::kChunk - 1) / C::kChunk;
    g.block_chunks = KIND == 0 ? 1 : o.block_size / C::kChunk;
    g.tiles_n = (o.n + C::NT - 1) / C::NT;
    g.tiles_m = (o.m + C::BM - 1) / C::BM;
    const int units = splits * C::KW;
    g.chunks_per_wave = (g.chunks + units - 1) / units;
    splits = (g.chunks + g.chunks_per_wave * C::KW - 1) / (g.chunks_per_wave * C::KW);
    // Row tiles of a panel: of the tiles an XCD works on at a time, up to 32 (one
    // to a compute unit; counting two measured slower), p rows by 32 / p columns
    // read p row tiles of A and 32 / p column tiles of codes, least at p = sqrt(32
    // codes / A).  Panels of equal height, so that the last is not a short one.
    // One panel to 384 rows (192 rows of 4096 x 5632 INT8 33.7 us, 35.7 in two),
    // for 16-bit A, half the size (1024 rows of 4096 x 1024 bf16 INT4 24.9, 26.7;
    // of 2048 x 5632 54.2, 52.5), and for K splits, whose runs are short already
    // (1024 rows of 8192 x 256 INT8 in four splits 52, 61).
    int panels = 1;
    if (EL == EL_F32 && splits == 1 && o.m > 384) {
        const double tile_codes = C::NT * (KIND == 2 ? 0.5 : 1.0), tile_a = C::BM * 4.0;
        const double active = std::min(32.0, g.tiles_n * static_cast<double>(g.tiles_m) / 8);
        const int high = std::max(1, static_cast<int>(std::sqrt(active * tile_codes / tile_a) + 0.5));
        panels = std::max(1, (g.tiles_m + high / 2) / high);
    }
    g.panel = (g.tiles_m + panels - 1) / panels;
    Workspace ws{};
    const std::size_t tiles = static_cast<std::size_t>(g.tiles_n) * g.tiles_m;
    if (splits > 1) VM_TRY(get_workspace(stream, tiles * NW * splits * (C::kItems * 256), tiles, &ws));
    g.partials = ws.partials;
    g.counters = ws.counters;
    const int64_t rows = AM == AM_PIECES ? (static_cast<int64_t>(o.m) + 31) / 32 * 32 : o.m;
    g.lo_offset = static_cast<uint32_t>(rows * g.k * 2);
    g.a_bytes = static_cast<uint32_t>(rows * g.k * (EL == EL_F32 ? 4 : 2));
    const int64_t nblk = KIND == 0 ? 1 : (static_cast<int64_t>(o.k) + o.block_size - 1) / o.block_size;
    g.code_bytes = static_cast<uint32_t>((KIND == 2 ? (static_cast<int64_t>(o.k) + 1) / 2 : static_cast<int64_t>(o.k)) * o.n);
    g.scale_bytes = static_cast<uint32_t>(nblk * o.n * (SH ? 2 : 4));
    g.c_vec = o.n % 4 == 0 && reinterpret_cast<uintptr_t>(o.c) % 8 == 0 ? 1 : 0;
    hipLaunchKernelGGL((qmm_quad_kernel<KIND, TILE, MT, W, NW, AM, EL, SH, D>), dim3(static_cast<unsigned>(tiles * splits)),
                       dim3(64 * W), 0, stream, g);
    return check_launch("QuantizedMatMul", stream);
}

// Tile, waves and K splits of a call.
struct QuadConfig {
    int tile, mt, waves, splits;
    bool pair = false;   // two waves side by side in N, two in K
};

// Chosen from sweeps of every tile, wave count and 1 - 12 splits on MI355X
// over K x N = 576 x 1536 .. 8192 x 8192 and 2048 x 32000, 1 to 1024 rows,
// INT8 and INT4, fp32 and bf16 (weights warm; times are staging + GEMM):
//   * 16-row tiles (64 columns a wave) up to 16 rows, and up to 32 while the
//     codes are at most 16 MB: twice the tiles, no rows multiplied for
//     padding, and small calls are bound by latency (M = 32, 2048 x 5632 INT4
//     9.3 us, 32-row tiles 12.9).  Past 48 MB of codes (INT8 from 32 MB) the
//     128-byte code runs of the 128-column tiles count for more (M = 16,
//     8192 x 28672 INT4 46 us against 57).
//   * 64-row tiles for per-column INT8 whose 64 x 128 tiles number 170 or
//     more, where their padding adds less than an eighth: each unpacked
//     column feeds two row tiles (M = 512, 2048 x 11264 50.8 us against 59.7;
//     blockwise kinds lack the registers: M = 512, 2048 x 5632 INT4 46 us
//     against 36, and with 16-bit A, where they fit one wave per SIMD, 37
//     against 31, M = 333, 5632 x 2048 bf16 31.7 against 30.4).
//   * two waves side by side in N, sharing A's lines in L1, where the tiles are
//     many enough to do with two waves in K: blockwise above 512 rows from 600 tiles
//     of 32 x 256 (M = 1024, 2048 x 5632 INT4 76.5 -> 65.8 us; M = 512, 2048 x
//     11264 64.1 -> 61 to 66, 2048 x 5632 41 -> 43.5); 64-row tiles from 1024
//     where the wider ones, at two units of time each, take no more rounds of
//     the GPU (M = 1024, INT8: 1024 tiles of 576 x 8192 31.7 -> 29.8 us, of 2048 x
//     8192 69.8 -> 68.0; 768 tiles, 2048 rows of 2048 x 3072, would take four
//     rounds for three, 58.9 -> 63.3; below 1024 tiles either way within 5 %).
//   * eight waves per tile; four once the tiles alone fill the GPU (more than
//     260), or when a 16-row tile's K is too short for eight (576 x 1536).
//   * K splits only where the tiles leave compute units idle: 16-row tiles
//     until a wave holds at most 8 (INT4) or 4 (INT8) chunks of 32 rows or
//     about 60 workgroups run, wider tiles up to about 260 workgroups, never
//     below two chunks a wave (M = 64, 2048 x 2048 INT4: four splits 11.9 us,
//     one 14); at most six there, at most twelve on 16-row tiles.
// Where the staged A leaves the no-allocation entry point room in its static
// array, a call's fp32 partial tiles stay within it, so that all entry points
// choose alike; it refuses longer A, and takes no 16-bit calls, and these have
// all their splits (M = 512, 8192 x 512 INT8 33.6 us in four splits, 44.5 in one).
// VELOMIND_GEMM_WIDE="BM,BN,S,D[,G]" or VELOMIND_GEMM_CFG="BM,BN,S[,D]" force
// the row tile (16 up to BM = 16, per-column INT8 64 from BM = 128, else 32),
// paired waves with BN of 256 or more (64-row tiles and blockwise kinds), S
// splits and, with D or G of 2, eight waves (not 64-row tiles).
template <int KIND, int AM, int EL>
QuadConfig choose_quad(int m, int k, int n, std::size_t a_bytes) {
    const double code_bytes = (KIND == 2 ? 0.5 : 1.0) * k * n;
    const int chunks = (k + 31) / 32;
    auto tiles_of = [&](int bm, int bn) { return static_cast<long>((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
    QuadConfig c{32, 1, 8, 1};
    if ((m <= 16 && code_bytes <= (KIND == 2 ? 48e6 : 32e6)) || (m <= 32 && code_bytes <= 16e6)) {
        c.tile = 16;
        const long tiles = tiles_of(16, 64);
        if (chunks <= 20 || tiles >= 400) c.waves = 4;
        const long per_wave = KIND == 2 ? 8 : 4;
        long s = std::max((chunks + per_wave * c.waves - 1) / (per_wave * c.waves), 60 / tiles);
        s = std::min({s, 260 / tiles, static_cast<long>(chunks) / (2 * c.waves), 12L});
        c.splits = static_cast<int>(std::max(1L, s));
    } else {
        const long tiles64 = tiles_of(64, 128);
        if (KIND == 0 && AM == AM_PIECES && tiles64 >= 170 && (m + 63) / 64 * 64 <= (m + 31) / 32 * 36) {
            c.mt = 2;
            c.waves = 4;
            const long cus = 256, rounds = (tiles64 + cus - 1) / cus;
            c.pair = tiles64 >= 1024 && 2 * ((tiles_of(64, 256) + cus - 1) / cus) <= rounds;
        } else if (KIND != 0 && AM == AM_PIECES && m > 512 && tiles_of(32, 256) >= 600) {
            c.waves = 4;
            c.pair = true;
        } else {
            const long tiles = tiles_of(32, 128);
            if (tiles > 260) c.waves = 4;
            c.splits = static_cast<int>(std::max(1L, std::min({260 / tiles, static_cast<long>(chunks) / (2 * c.waves), 6L})));
        }
    }
    auto partials = [&](int s) {
        return s > 1 ? static_cast<double>(tiles_of(c.tile * c.mt, 4 * c.tile)) * s * c.tile * c.mt * 4 * c.tile * 4 : 0.0;
    };
    constexpr std::size_t kRoom = kStaticPartialBytes - 65536;
    if (EL == EL_F32 && a_bytes <= kRoom)
        while (c.splits > 1 && partials(c.splits) > static_cast<double>(kRoom - a_bytes)) --c.splits;
    int bm = 0, bn = 0, s = 0, d = 0, g = 0;
    const char* env = std::getenv("VELOMIND_GEMM_WIDE");
    int got = env ? std::sscanf(env, "%d,%d,%d,%d,%d", &bm, &bn, &s, &d, &g) : 0;
    if (got < 4 && (env = std::getenv("VELOMIND_GEMM_CFG"))) got = std::sscanf(env, "%d,%d,%d,%d", &bm, &bn, &s, &d);
    if (got >= 3 && bm >= 16 && s >= 1 && s <= 16) {
        c.tile = bm <= 16 ? 16 : 32;
        c.mt = bm >= 128 && KIND == 0 && AM == AM_PIECES ? 2 : 1;
        c.pair = bn >= 256 && AM == AM_PIECES && c.tile == 32 && (c.mt == 2 || KIND != 0);
        c.waves = c.mt == 1 && (d == 2 || g == 2) ? 8 : 4;
        c.splits = s;
    }
    return c;
}

template <int KIND, int AM, int EL, bool SH>
int launch_mode(const GemmOperands& o, hipStream_t s) {
    const std::size_t a_bytes = EL == EL_F32 ? a_stage_bytes(o.m, (o.k + 31) / 32 * 32, AM == AM_PIECES) : 0;
    const QuadConfig c = choose_quad<KIND, AM, EL>(o.m, o.k, o.n, a_bytes);
    if (c.tile == 16) {
        if (c.waves == 4) return launch_quad<KIND, 16, 1, 4, 1, AM, EL, SH, 3>(o, c.splits, s);
        return launch_quad<KIND, 16, 1, 8, 1, AM, EL, SH, 3>(o, c.splits, s);
    }
    if constexpr (AM == AM_PIECES) {
        if constexpr (KIND == 0)
            if (c.mt == 2)
                return c.pair ? launch_quad<KIND, 32, 2, 4, 2, AM, EL, SH, 4>(o, c.splits, s)
                              : launch_quad<KIND, 32, 2, 4, 1, AM, EL, SH, 4>(o, c.splits, s);
        if constexpr (KIND != 0)
            if (c.pair) return launch_quad<KIND, 32, 1, 4, 2, AM, EL, SH, 3>(o, c.splits, s);
    }
    if (c.waves == 4) return launch_quad<KIND, 32, 1, 4, 1, AM, EL, SH, 3>(o, c.splits, s);
    return launch_quad<KIND, 32, 1, 8, 1, AM, EL, SH, 3>(o, c.splits, s);
}

template <int AM, int EL, bool SH>
int launch_kind(const GemmOperands& o, hipStream_t s) {
    if (o.kind == 2) return launch_mode<2, AM, EL, SH>(o, s);
    if (o.kind == 1) return launch_mode<1, AM, EL, SH>(o, s);
    return launch_mode<0, AM, EL, SH>(o, s);
}

}  // namespace
}  // namespace vmhip
