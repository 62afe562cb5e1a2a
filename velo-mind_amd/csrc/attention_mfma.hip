// Attention with fp32 matrix cores: the resident decoder's prompts over its KV
// cache and FusedAttention's (fused_attention.cpp:20-139) with several query
// rows.
//
// A workgroup of four waves takes QR = 16 RW query rows of one head: wave w
// owns rows 16 (w % RW) .. +15 and key group w / RW of KS.  The keys go by
// in steps of KS 64-key tiles staged in LDS; group g runs its online
// softmax over tile g of each step, and the groups' (max, sum, output)
// triples are merged through LDS at the end.  Splitting the keys cuts the
// longest chain of dependent MFMAs (the last query rows see every key) by
// KS; the grid is one-dimensional with the query tiles that see the most
// keys first, so the workgroups dispatched last are the short ones.
//
// v_mfma_f32_16x16x4_f32 (fp32 inputs and accumulation, so no precision is
// given up against the fp32 reference) holds A[i][k] in lane i + 16k,
// B[k][j] in lane j + 16k and D[i][j] in lane j + 16 (i / 4), element i % 4.
// Scores are computed transposed, S^T = K Q^T, so lane (row r = lane % 16,
// group g = lane / 16) holds row r's scores for keys 16b + 4g + e: exactly
// the A operand of P V once the product's reduction index is ordered as
// key(s, k) = 16 (s / 4) + 4k + s % 4 (the order of a sum's terms is free).
// Output column j of MFMA tile db is dim 64 (db / 4) + 4 j + db % 4, so that
// a lane's four V operands of a key are one 16-byte LDS read, and its
// results one 16-byte store.  Four independent accumulators alternate in
// both products.  Row statistics live in the lanes of row r (shared across
// the four groups); output row 4g + e fetches its factor from lane 4g + e.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdlib>

#include "attention.h"
#include "vm_internal.h"

namespace vmhip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kTile = 64;   // keys per tile (one key group's share of a step)

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
__global__ __launch_bounds__(kThreads) void attention_mfma_kernel(const AttentionCall a) {
    static_assert(D == 64 || D == 128, "64-dim slabs, 16 dims per lane group");
    static_assert(RW * KS == 4, "four waves");
    constexpr int H = D / 64;          // 64-dim slabs
    constexpr int ST = kTile * KS;     // keys per step
    constexpr int PITCH = D + 4;       // LDS row pitch in floats (conflict-free 16-byte reads)
    constexpr int QR = 16 * RW;        // query rows per workgroup
    extern __shared__ __align__(16) float smem[];
    float* sk = smem;                  // [ST][PITCH]
    float* sv = smem + ST * PITCH;
    __shared__ int v_special[2];       // whether the step's V holds an infinity or NaN, by step parity
    const int tiles = (a.rows + QR - 1) / QR;
    const int bh_count = a.batch * a.heads;
    const int bh = static_cast<int>(blockIdx.x) % bh_count;
    const int bkv = bh / a.heads * a.kv_heads + bh % a.heads / (a.heads / a.kv_heads);
    const int r0 = (tiles - 1 - static_cast<int>(blockIdx.x) / bh_count) * QR;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
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

    // Q fragment: Q[qrow][64 h + 16 lg + s], s = 0..15.
    float4 qf[H][4];
    {
        const float* qp = a.q + (static_cast<int64_t>(bh) * a.rows + (row_ok ? qrow : 0)) * D + 16 * lg;
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                qf[h][c] = row_ok ? *reinterpret_cast<const float4*>(qp + 64 * h + 4 * c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // keys < wg_end reach some row of the tile
    const int wg_end = a.causal ? min(p0 + min(r0 + QR, a.rows), n_keys) : n_keys;
    const float* kb = a.k + static_cast<int64_t>(bkv) * a.keys * D;
    const float* vb = a.v + static_cast<int64_t>(bkv) * a.keys * D;
    f32x4 acc[4 * H];   // O[row 4 lg + e][dim 64 (db / 4) + 4 lr + db % 4]
#pragma unroll
    for (int db = 0; db < 4 * H; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.0f;   // statistics of row lr of this wave

    // K/V steps pass through registers one step ahead: the next step's
    // loads are issued as soon as the current one is in LDS, so they are in
    // flight during its scores and p . V.
    constexpr int kU = ST * D / 4 / kThreads;   // float4s of K (and of V) per thread per step
    float4 nk_reg[kU], nv_reg[kU];
    auto load_step = [&](int t0) {
        const int nkt = min(ST, n_keys - t0);
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int e = tid + u * kThreads;
            const int j = e / (D / 4), c = e - j * (D / 4);
            nk_reg[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            nv_reg[u] = nk_reg[u];
            if (j < nkt) {
                nk_reg[u] = *reinterpret_cast<const float4*>(kb + static_cast<int64_t>(t0 + j) * D + 4 * c);
                nv_reg[u] = *reinterpret_cast<const float4*>(vb + static_cast<int64_t>(t0 + j) * D + 4 * c);
            }
        }
    };
    if (tid < 2) v_special[tid] = 0;
    if (wg_end > 0) load_step(0);
    int parity = 0;
    for (int s0 = 0; s0 < wg_end; s0 += ST, parity ^= 1) {
        __syncthreads();   // the previous step is consumed
        bool special = false;
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int e = tid + u * kThreads;
            const int j = e / (D / 4), c = e - j * (D / 4);
            *reinterpret_cast<float4*>(sk + j * PITCH + 4 * c) = nk_reg[u];
            *reinterpret_cast<float4*>(sv + j * PITCH + 4 * c) = nv_reg[u];
            // x - x is 0 for finite x, NaN otherwise
            const float4 v = nv_reg[u];
            const float d = (v.x - v.x) + (v.y - v.y) + (v.z - v.z) + (v.w - v.w);
            special = special || !(d == 0.0f);
        }
        if (special) v_special[parity] = 1;
        if (s0 + ST < wg_end) load_step(s0 + ST);
        __syncthreads();
        if (tid == 0) v_special[parity ^ 1] = 0;   // the next step sets it after the next barrier

        const int k0 = s0 + kg * kTile;   // this key group's tile
        // a tile wholly past the wave's last visible key changes nothing
        if (k0 > wave_last) continue;
        const float* skt = sk + kg * kTile * PITCH;
        const float* svt = sv + kg * kTile * PITCH;

        // S^T = K Q^T for the four 16-key blocks.
        f32x4 st[4];
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) st[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float4 ka[4];
#pragma unroll
                for (int nb = 0; nb < 4; ++nb)
                    ka[nb] = *reinterpret_cast<const float4*>(skt + (16 * nb + lr) * PITCH + 64 * h + 16 * lg + 4 * c);
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) st[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[nb].x, qf[h][c].x, st[nb], 0, 0, 0);
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) st[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[nb].y, qf[h][c].y, st[nb], 0, 0, 0);
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) st[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[nb].z, qf[h][c].z, st[nb], 0, 0, 0);
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) st[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[nb].w, qf[h][c].w, st[nb], 0, 0, 0);
            }
        // Scale, mask (tiles that some row does not see whole), online softmax
        // of row lr.  A row that has seen nothing but -inf keeps the maximum
        // -inf and exponentiates against 0.
        const bool masked = k0 + kTile - 1 > wave_first || !row_ok;
        float mt = -INFINITY;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = st[nb][e] * a.scale;
                if (masked) v = k0 + 16 * nb + 4 * lg + e <= my_last ? v : -INFINITY;
                st[nb][e] = v;
                mt = fmaxf(mt, v);
            }
        mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float m_new = fmaxf(m_run, mt);
        const float m_ref = m_new == -INFINITY ? 0.0f : m_new;
        float lt = 0.0f;
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                st[nb][e] = exp_nonpos(st[nb][e] - m_ref);
                lt += st[nb][e];
            }
        lt += __shfl_xor(lt, 16, 64);
        lt += __shfl_xor(lt, 32, 64);
        const float alpha = exp_nonpos(m_run - m_ref);
        l_run = l_run * alpha + lt;
        m_run = m_new;
        // Rescale the output rows 4 lg + e by their rows' factors.
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float ae = __shfl(alpha, 4 * lg + e, 64);
#pragma unroll
            for (int db = 0; db < 4 * H; ++db) acc[db][e] *= ae;
        }
        // O += P V.  A masked key's zero would turn an infinity or NaN of its
        // V into NaN: a partly masked tile of a step with such values
        // multiplies them as 0 and adds them for the rows that see them below.
        const bool careful = v_special[parity] != 0 && k0 + kTile - 1 > wave_first;
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const float* vrow = svt + (16 * (s / 4) + 4 * lg + s % 4) * PITCH + 4 * lr;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                float4 bv = *reinterpret_cast<const float4*>(vrow + 64 * h);
                if (careful) {
                    bv.x = bv.x - bv.x == 0.0f ? bv.x : 0.0f;
                    bv.y = bv.y - bv.y == 0.0f ? bv.y : 0.0f;
                    bv.z = bv.z - bv.z == 0.0f ? bv.z : 0.0f;
                    bv.w = bv.w - bv.w == 0.0f ? bv.w : 0.0f;
                }
                const float p = st[s / 4][s % 4];
                acc[4 * h + 0] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, bv.x, acc[4 * h + 0], 0, 0, 0);
                acc[4 * h + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, bv.y, acc[4 * h + 1], 0, 0, 0);
                acc[4 * h + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, bv.z, acc[4 * h + 2], 0, 0, 0);
                acc[4 * h + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, bv.w, acc[4 * h + 3], 0, 0, 0);
            }
        }
        if (careful) {
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int s = 0; s < 16; ++s) {
                    const int key = 16 * (s / 4) + 4 * g + s % 4;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int row = r0 + 16 * wr + 4 * lg + e;
                        const float p = __shfl(st[s / 4][s % 4], 16 * g + 4 * lg + e, 64);
                        const bool sees = row < a.rows && k0 + key < n_keys && (!a.causal || k0 + key <= p0 + row);
#pragma unroll
                        for (int db = 0; db < 4 * H; ++db) {
                            const float v = svt[key * PITCH + 64 * (db / 4) + 4 * lr + db % 4];
                            if (sees && !(v - v == 0.0f)) acc[db][e] = fmaf(p, v, acc[db][e]);
                        }
                    }
                }
        }
    }

    // Merge the key groups' triples into group 0 (fixed order: group 0, 1,
    // ..): m = max m_g, l = sum l_g e^(m_g - m), O = sum O_g e^(m_g - m).
    if constexpr (KS > 1) {
        __syncthreads();   // every wave is past its last LDS read
        float* so = sk;                         // [KS - 1][RW][16 rows][D]
        float* sst = sv;                        // [KS - 1][RW][16 rows][2]
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
    constexpr int kLds = 2 * kTile * KS * (D + 4) * 4;
    auto kernel = attention_mfma_kernel<D, RW, KS>;
    // (above the 64 KB default; a refused attribute fails the launch)
    static const hipError_t lds_set = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (lds_set != hipSuccess) return fail_hip(lds_set, op);
    const int64_t grid = static_cast<int64_t>((c.rows + 16 * RW - 1) / (16 * RW)) * c.batch * c.heads;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kThreads), kLds, stream, c);
    return check_launch(op, stream);
}

// Key groups per workgroup (64 / groups query rows each), from sweeps on
// MI355X: one when a single tile holds the keys, or when one-group workgroups
// already number more than 512 (1000 x 1500, 64 heads of 128: 408 us, two
// groups 514); four when even 16-row tiles would leave compute units idle and
// the keys are many (16 x 2000, 8 heads of 64: 43 us, two groups 65, one 107;
// head_dim 128 lacks the LDS); two otherwise (512 x 512, 15 heads: 20.5 us,
// one group 31, four 23).  A cache's key count is on the device: its rows
// stand for it.  VELOMIND_ATTN_SPLIT = 1 or 2 overrides (sweeps).
int key_groups(const AttentionCall& c) {
    static const int forced = [] {
        const char* e = std::getenv("VELOMIND_ATTN_SPLIT");
        const int v = e ? std::atoi(e) : 0;
        return (v == 1 || v == 2) ? v : 0;
    }();
    if (forced) return forced;
    const int64_t bh = static_cast<int64_t>(c.batch) * c.heads;
    const int keys = c.pos ? c.rows : c.keys;
    if ((static_cast<int64_t>(c.rows) + 63) / 64 * bh > 512 || (keys <= kTile && !c.pos)) return 1;
    return c.head_dim == 64 && (static_cast<int64_t>(c.rows) + 15) / 16 * bh <= 256 && keys > 256 ? 4 : 2;
}

}  // namespace

bool attention_mfma_takes(const AttentionCall& c) {
    const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return (c.head_dim == 64 || c.head_dim == 128) && aligned(c.q) && aligned(c.k) && aligned(c.v) && aligned(c.o) &&
           (static_cast<int64_t>(c.rows) + 15) / 16 * c.batch * c.heads <= INT32_MAX;
}

int attention_mfma(const AttentionCall& c, const char* op, hipStream_t stream) {
    const int groups = key_groups(c);
    if (c.head_dim == 128)
        return groups == 1 ? launch<128, 4, 1>(c, op, stream) : launch<128, 2, 2>(c, op, stream);
    if (groups == 4) return launch<64, 1, 4>(c, op, stream);
    return groups == 1 ? launch<64, 4, 1>(c, op, stream) : launch<64, 2, 2>(c, op, stream);
}

}  // namespace vmhip
