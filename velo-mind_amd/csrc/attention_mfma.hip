// Attention with fp32 matrix cores: the resident decoder's prompts over its KV
// cache and FusedAttention's (fused_attention.cpp:20-139) with several query
// rows.
//
// A workgroup of four waves takes QR = 16 RW query rows of one head: wave w
// owns rows 16 (w % RW) .. +15 and, of the KS key groups, group w / RW: the
// blocks of KB keys whose number is w / RW modulo KS.  A wave reads its K and
// V blocks from global memory straight into MFMA operand registers, one
// block ahead, so the loop has no LDS traffic and no barrier, and two waves
// per SIMD hide each other's softmax; the groups' (max, sum, output) triples
// are merged through LDS at the end.  (Staging K and V in LDS for the whole
// workgroup took 20 us at 512 x 512, 15 heads of 64, most of it waiting at
// its two barriers per step; three-way bf16 splits of every operand on the
// 16-bit matrix cores there, 24 us: the splitting costs what it saves.)
// The grid is one-dimensional with the query tiles that see the most keys
// first, so the workgroups dispatched last are the short ones.
//
// v_mfma_f32_16x16x4_f32 (fp32 inputs and accumulation, so no precision is
// given up against the fp32 reference) holds A[i][k] in lane i + 16k,
// B[k][j] in lane j + 16k and D[i][j] in lane j + 16 (i / 4), element i % 4.
// Scores are computed transposed, S^T = K Q^T, four dims 16 c + 4 k + e at a
// time (lane group k holds four adjacent dims: one 16-byte load); lane (row r
// = lane % 16, group g = lane / 16) then holds row r's scores for keys 16b +
// 4g + e: exactly the A operand of P V once the product's reduction index is
// ordered as key(s, k) = 16 (s / 4) + 4k + s % 4 (the order of a sum's terms
// is free).  Output column j of MFMA tile db is dim 64 (db / 4) + 4 j + db %
// 4, so that a lane's four V operands of a key are one 16-byte load, and its
// results one 16-byte store.  Row statistics live in the lanes of row r
// (shared across the four groups); output row 4g + e fetches its factor from
// lane 4g + e.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "attention.h"
#include "vm_internal.h"

namespace vmhip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;

// e^x for x <= 0: 2^h with h = x log2 e rounded, times e^l for what the
// rounding and log2 e's own lost (the error of 2^h alone grows with |x|).
// NaN stays NaN; -inf gives 0.
__device__ __forceinline__ float exp_nonpos(float x) {
    constexpr float kLog2e = 1.44269504f, kLog2eLow = 1.92596299e-8f;
    const float h = x * kLog2e;
    const float l = fmaf(x, kLog2eLow, fmaf(x, kLog2e, -h));
    const float r = __builtin_amdgcn_exp2f(h);
    return x < -120.0f ? 0.0f : fmaf(r, l * 0.693147181f, r);
}

template <int D, int RW, int KS>
__global__ __launch_bounds__(kThreads, 2) void attention_mfma_kernel(const AttentionCall a, int fold) {
    static_assert(D == 64 || D == 128, "64-dim slabs");
    static_assert(RW * KS == 4 && KS > 1, "four waves");
    constexpr int H = D / 64;          // 64-dim slabs
    constexpr int KB = 32 / H;         // keys per block: K and V of two blocks fit the registers
    constexpr int NB = KB / 16;        // 16-key MFMA tiles of a block
    constexpr int NC = D / 16;         // 16-dim groups
    constexpr int NS = KB / 4;         // reduction steps of P V
    constexpr int QR = 16 * RW;        // query rows per workgroup
    const int tiles = (a.rows + QR - 1) / QR;
    const int bh_count = a.batch * a.heads;
    // Tiles in descending order of the keys they see; of a grid that fits the
    // GPU two workgroups to a compute unit, the second one per unit comes in
    // ascending order, so that a unit's two together see about as many as any
    // other's (512 cached rows, 32 heads: 24.6 -> 20.8 us).
    int order = static_cast<int>(blockIdx.x);
    if (fold > 0 && order >= fold) order = fold + static_cast<int>(gridDim.x) - 1 - order;
    const int bh = order % bh_count;
    const int bkv = bh / a.heads * a.kv_heads + bh % a.heads / (a.heads / a.kv_heads);
    const int r0 = (tiles - 1 - order / bh_count) * QR;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave % RW, kg = wave / RW;   // row block, key group
    const int lr = lane & 15, lg = lane >> 4;
    const int p0 = a.pos ? a.pos[0] : a.keys - a.rows;   // position of query row 0
    const int n_keys = a.pos ? min(p0 + a.rows, a.keys) : a.keys;
    const int qrow = r0 + 16 * wr + lr;       // the query row whose Q this lane holds
    const bool row_ok = qrow < a.rows;
    // keys <= my_last are visible to row qrow
    const int my_last = !row_ok ? -1 : a.causal ? min(p0 + qrow, n_keys - 1) : n_keys - 1;
    // keys past wave_last are masked for every row of the wave; up to
    // wave_first they are visible to every row
    const int row_end = min(r0 + 16 * wr + 15, a.rows - 1);
    const int wave_last = r0 + 16 * wr >= a.rows ? -1 : a.causal ? min(p0 + row_end, n_keys - 1) : n_keys - 1;
    const int wave_first = a.causal ? min(p0 + r0 + 16 * wr, n_keys - 1) : n_keys - 1;

    // Q operand: Q[qrow][16 c + 4 lg + e].
    float4 qf[NC];
    {
        const float* qp = a.q + (static_cast<int64_t>(bh) * a.rows + (row_ok ? qrow : 0)) * D + 4 * lg;
#pragma unroll
        for (int c = 0; c < NC; ++c)
            qf[c] = row_ok ? *reinterpret_cast<const float4*>(qp + 16 * c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    const float* kb = a.k + static_cast<int64_t>(bkv) * a.keys * D + 4 * lg;
    const float* vb = a.v + static_cast<int64_t>(bkv) * a.keys * D + 4 * lr;
    f32x4 acc[4 * H];   // O[row 4 lg + e][dim 64 (db / 4) + 4 lr + db % 4]
#pragma unroll
    for (int db = 0; db < 4 * H; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.0f;   // statistics of row lr of this wave

    struct Block {
        float4 k[NB][NC];   // K[k0 + 16 nb + lr][16 c + 4 lg ..]
        float4 v[NS][H];    // V[k0 + 16 (s / 4) + 4 lg + s % 4][64 h + 4 lr ..]
    };
    // Keys past the end read the last one; they are masked.
    auto load = [&](int k0, Block& b) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const float* p = kb + static_cast<int64_t>(min(k0 + 16 * nb + lr, n_keys - 1)) * D;
#pragma unroll
            for (int c = 0; c < NC; ++c) b.k[nb][c] = *reinterpret_cast<const float4*>(p + 16 * c);
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const float* p = vb + static_cast<int64_t>(min(k0 + 16 * (s / 4) + 4 * lg + s % 4, n_keys - 1)) * D;
#pragma unroll
            for (int h = 0; h < H; ++h) b.v[s][h] = *reinterpret_cast<const float4*>(p + 64 * h);
        }
    };
    auto compute = [&](int k0, const Block& b) {
        // S^T = K Q^T: per 16-key tile two accumulators in turn.
        f32x4 st[NB], su[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) st[nb] = su[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NC; ++c) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) st[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.k[nb][c].x, qf[c].x, st[nb], 0, 0, 0);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) su[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.k[nb][c].y, qf[c].y, su[nb], 0, 0, 0);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) st[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.k[nb][c].z, qf[c].z, st[nb], 0, 0, 0);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) su[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.k[nb][c].w, qf[c].w, su[nb], 0, 0, 0);
        }
        // Scale, mask (blocks that some row does not see whole), online softmax
        // of row lr.  A row that has seen nothing but -inf keeps the maximum
        // -inf and exponentiates against 0.
        const bool masked = k0 + KB - 1 > wave_first;
        float mt = -INFINITY;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = (st[nb][e] + su[nb][e]) * a.scale;
                if (masked) v = k0 + 16 * nb + 4 * lg + e <= my_last ? v : -INFINITY;
                st[nb][e] = v;
                mt = fmaxf(mt, v);
            }
        mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float m_new = fmaxf(m_run, mt);
        const float m_ref = m_new == -INFINITY ? 0.0f : m_new;
        const float alpha = exp_nonpos(m_run - m_ref);
        float lt = 0.0f;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                st[nb][e] = exp_nonpos(st[nb][e] - m_ref);
                lt += st[nb][e];
            }
        l_run = fmaf(l_run, alpha, lt);   // (this lane's keys; summed over the lane groups at the end)
        m_run = m_new;
        // Rescale the output rows 4 lg + e by their rows' factors.
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float ae = __shfl(alpha, 4 * lg + e, 64);
#pragma unroll
            for (int db = 0; db < 4 * H; ++db) acc[db][e] *= ae;
        }
        // O += P V.  A masked key's zero would turn an infinity or NaN of its
        // V into NaN: in a partly masked block such values are multiplied as
        // 0 and added for the rows that see them.
        bool special = false;
        if (masked) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const float4 v = b.v[s][h];   // x - x is 0 for finite x, NaN otherwise
                    special = special || !((v.x - v.x) + (v.y - v.y) + (v.z - v.z) + (v.w - v.w) == 0.0f);
                }
            special = __any(special);
        }
        if (!special) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const float p = st[s / 4][s % 4];
                    acc[4 * h + 0] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, b.v[s][h].x, acc[4 * h + 0], 0, 0, 0);
                    acc[4 * h + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, b.v[s][h].y, acc[4 * h + 1], 0, 0, 0);
                    acc[4 * h + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, b.v[s][h].z, acc[4 * h + 2], 0, 0, 0);
                    acc[4 * h + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, b.v[s][h].w, acc[4 * h + 3], 0, 0, 0);
                }
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const float p = st[s / 4][s % 4];
                    const float v[4] = {b.v[s][h].x, b.v[s][h].y, b.v[s][h].z, b.v[s][h].w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        acc[4 * h + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, v[i] - v[i] == 0.0f ? v[i] : 0.0f,
                                                                              acc[4 * h + i], 0, 0, 0);
                        for (int g = 0; g < 4; ++g) {
                            const int key = k0 + 16 * (s / 4) + 4 * g + s % 4;
                            const float vk = __shfl(v[i], lr + 16 * g, 64);
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const int row = r0 + 16 * wr + 4 * lg + e;
                                const float pk = __shfl(p, 4 * lg + e + 16 * g, 64);
                                const bool sees = row < a.rows && key < n_keys && (!a.causal || key <= p0 + row);
                                if (sees && !(vk - vk == 0.0f)) acc[4 * h + i][e] = fmaf(pk, vk, acc[4 * h + i][e]);
                            }
                        }
                    }
                }
        }
    };

    Block b0, b1;
    int k0 = kg * KB;
    if (k0 <= wave_last) {
        load(k0, b0);
        while (true) {
            load(k0 + KS * KB, b1);
            compute(k0, b0);
            k0 += KS * KB;
            if (k0 > wave_last) break;
            load(k0 + KS * KB, b0);
            compute(k0, b1);
            k0 += KS * KB;
            if (k0 > wave_last) break;
        }
    }
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);

    // Merge the key groups' triples into group 0 (fixed order: group 0, 1,
    // ..): m = max m_g, l = sum l_g e^(m_g - m), O = sum O_g e^(m_g - m).
    {
        __shared__ __align__(16) float so[(KS - 1) * RW * 16 * D];   // [KS - 1][RW][16 rows][D]
        __shared__ float sst[(KS - 1) * RW * 16 * 2];                // [KS - 1][RW][16 rows][2]
        if (kg > 0) {
            float* o = so + ((kg - 1) * RW + wr) * 16 * D;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int h = 0; h < H; ++h)
                    *reinterpret_cast<float4*>(o + (4 * lg + e) * D + 64 * h + 4 * lr) =
                        make_float4(acc[4 * h][e], acc[4 * h + 1][e], acc[4 * h + 2][e], acc[4 * h + 3][e]);
            if (lg == 0) {
                float* t = sst + (((kg - 1) * RW + wr) * 16 + lr) * 2;
                t[0] = m_run;
                t[1] = l_run;
            }
        }
        __syncthreads();
        if (kg > 0) return;
        float mg[KS], lgs[KS];
        mg[0] = m_run;
        lgs[0] = l_run;
#pragma unroll
        for (int g = 1; g < KS; ++g) {
            const float* t = sst + (((g - 1) * RW + wr) * 16 + lr) * 2;
            mg[g] = t[0];
            lgs[g] = t[1];
        }
        float m = mg[0];
#pragma unroll
        for (int g = 1; g < KS; ++g) m = fmaxf(m, mg[g]);
        const float m_ref = m == -INFINITY ? 0.0f : m;
        float fg[KS];
        float l = 0.0f;
#pragma unroll
        for (int g = 0; g < KS; ++g) {
            fg[g] = exp_nonpos(mg[g] - m_ref);
            l += lgs[g] * fg[g];
        }
        l_run = l;
        m_run = m;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float f0 = __shfl(fg[0], 4 * lg + e, 64);
#pragma unroll
            for (int db = 0; db < 4 * H; ++db) acc[db][e] *= f0;
#pragma unroll
            for (int g = 1; g < KS; ++g) {
                const float fe = __shfl(fg[g], 4 * lg + e, 64);
                const float* o = so + ((g - 1) * RW + wr) * 16 * D + (4 * lg + e) * D;
#pragma unroll
                for (int db = 0; db < 4 * H; ++db) acc[db][e] += o[64 * (db / 4) + 4 * lr + db % 4] * fe;
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float le = __shfl(l_run, 4 * lg + e, 64);
        const float me = __shfl(m_run, 4 * lg + e, 64);
        // a row whose every score is -inf has no softmax: NaN, as the
        // reference's 0 / 0
        const float inv = me == -INFINITY ? NAN : le > 0.0f ? 1.0f / le : 0.0f;
        const int row = r0 + 16 * wr + 4 * lg + e;
        if (row < a.rows) {
            float* o = a.o + row * a.out_row + bh * a.out_head + 4 * lr;
#pragma unroll
            for (int h = 0; h < H; ++h)
                *reinterpret_cast<float4*>(o + 64 * h) = make_float4(acc[4 * h][e] * inv, acc[4 * h + 1][e] * inv,
                                                                     acc[4 * h + 2][e] * inv, acc[4 * h + 3][e] * inv);
        }
    }
}

template <int D, int RW, int KS>
int launch(const AttentionCall& c, const char* op, hipStream_t stream) {
    const int64_t grid = static_cast<int64_t>((c.rows + 16 * RW - 1) / (16 * RW)) * c.batch * c.heads;
    const int cus = cu_count();
    const int fold = c.causal && grid > cus && grid <= 2 * cus ? cus : 0;
    hipLaunchKernelGGL((attention_mfma_kernel<D, RW, KS>), dim3(static_cast<unsigned>(grid)), dim3(kThreads), 0, stream, c,
                       fold);
    return check_launch(op, stream);
}

// Key groups per workgroup (64 / groups query rows each): four, which cut the
// last rows' chain of blocks the most, while the 16-row tiles are few enough
// that chains and not throughput bound the call, else two (sharing K and V
// lines in L1 between two row blocks).  MI355X: 512 x 512, 15 heads of 64 (480
// tiles) 14.4 us against 17.1 with two, 16 x 2000, 8 heads 28.7 against 52.8; 512
// cached rows, 32 heads of 64 (1024 tiles) 25.5 against 20.7, 1500 rows 122
// against 116; 150 x 498, 128 heads of 128 (1280 tiles) 68 against 81, 1000 x
// 1500, 64 heads (4032 tiles) 386 against 378.  One group (64 rows a
// workgroup, nothing to merge) is faster for 128 cached heads of 64 (700 rows
// 103 against 112) and slower below (512 rows, 48 heads 37.6 against 33.1).
int key_groups(const AttentionCall& c) {
    const int64_t tiles = (static_cast<int64_t>(c.rows) + 15) / 16 * c.batch * c.heads;
    return tiles <= (c.head_dim == 64 ? 512 : 2048) ? 4 : 2;
}

}  // namespace

bool attention_mfma_takes(const AttentionCall& c) {
    const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return (c.head_dim == 64 || c.head_dim == 128) && aligned(c.q) && aligned(c.k) && aligned(c.v) && aligned(c.o) &&
           (static_cast<int64_t>(c.rows) + 15) / 16 * c.batch * c.heads <= INT32_MAX;
}

int attention_mfma(const AttentionCall& c, const char* op, hipStream_t stream) {
    const bool four = key_groups(c) == 4;
    if (c.head_dim == 128) return four ? launch<128, 1, 4>(c, op, stream) : launch<128, 2, 2>(c, op, stream);
    return four ? launch<64, 1, 4>(c, op, stream) : launch<64, 2, 2>(c, op, stream);
}

}  // namespace vmhip
