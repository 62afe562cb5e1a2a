// Prefill-shaped (rows_m > 4, and any 16-bit) quantized matmul: which shapes
// the MFMA kernel (qmm_quad_impl.h) takes, and the staging of its
// activations.
//
// fp32 A is split once per call (the prep kernels, or its producer, see
// a_split.h): each row r is multiplied by 2^x_r, the power of two that puts
// its largest magnitude in [2^14, 2^15), and written as two fp16 parts
// hi = fp16(a * 2^x_r) and lo = fp16(a * 2^x_r - hi), so that hi + lo
// carries 22 significant bits of any finite fp32 row without overflow or
// underflow.  Both parts go through the MFMAs (products with the exact fp16
// codes are exact, accumulation is fp32), and the epilogue multiplies by
// 2^-x_r, which is exact: the activations are used at fp32-equivalent
// precision, and beyond fp32 accumulation the only rounding is A's split
// (relative 2^-22).  fp16 and bf16 A go through the MFMAs as they are.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>

#include "a_split.h"
#include "qmm_kernels.h"
#include "vm_device.h"
#include "vm_internal.h"

namespace vmhip {
namespace {

typedef _Float16 half8v __attribute__((ext_vector_type(8)));

// A [m, k] fp32 -> two fp16 parts with a power-of-two scale per row: x_r
// is chosen so that the largest finite |a[r, k]| * 2^x_r lies in [2^14, 2^15)
// (x_r = 0 where that is zero; an infinity or NaN goes into hi and reaches
// the output as the reference's fp32 arithmetic propagates it);
// hi = fp16(a * 2^x_r) and lo = fp16(a * 2^x_r - hi), the difference being
// exact in fp32.
// The parts go out in the operand order of v_mfma_f32_32x32x16_f16, so that one wave's operand for 32 rows and 16 k
// is 1 KB of consecutive memory: the 16 bytes lane l of the wave loads for
// row block b (rows 32b .. 32b + 31) and k block q (k 16q .. 16q + 15) --
// row 32b + l % 32, k 16q + 8 (l / 32) + 0..7 -- sit at half offset
// ((b * kp / 16 + q) * 64 + l) * 8, kp being k rounded up to 32 (zeros past
// k); lo follows hi after mp * kp halves, mp = m rounded up to 32.  Inside each 16-byte piece the halves are stored in
// the order k = 0, 4, 1, 5, 2, 6, 3, 7, the order in which the MFMA
// kernel's weight unpacking produces B (a dot product does not depend on
// the order of its terms, so A and B only have to agree).
//
// Workgroup r splits row r; rows of up to kSplitHeld groups of eight per
// thread stay in registers between the maximum and the split (one read of
// A), longer rows are read a second time (from L2).
constexpr int kSplitHeld = 3;   // k <= 6144 in one read

// Eight values of a row of k from column c, zeros past its end.
__device__ __forceinline__ void load8_tail(const float* src, int c, int k, float4& p, float4& q) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = c + i < k ? src[c + i] : 0.0f;
    p = make_float4(v[0], v[1], v[2], v[3]);
    q = make_float4(v[4], v[5], v[6], v[7]);
}

// PIECES: operand order; else row-major (k a multiple of 32).
template <bool PIECES>
__global__ __launch_bounds__(256) void gemm_prep_kernel(const float* __restrict__ a, _Float16* __restrict__ ah,
                                                        int* __restrict__ row_exp, int m, int k, int kp, int vec) {
    __shared__ float wmax[4];
    const int tid = threadIdx.x;
    const int row = static_cast<int>(blockIdx.x);
    const float* src = a + static_cast<int64_t>(row) * k;
    const int groups = kp >> 3;   // columns k .. kp - 1 are written as zeros
    const bool held = groups <= kSplitHeld * 256;
    auto load8 = [&](int g, float4& p, float4& q) {
        if (vec) {
            p = reinterpret_cast<const float4*>(src)[2 * g];
            q = reinterpret_cast<const float4*>(src)[2 * g + 1];
        } else {
            load8_tail(src, 8 * g, k, p, q);
        }
    };
    float4 keep[kSplitHeld][2];
    float mx = 0.0f;
    if (held) {
#pragma unroll
        for (int r = 0; r < kSplitHeld; ++r) {
            const int g = tid + r * 256;
            if (g < groups) {
                load8(g, keep[r][0], keep[r][1]);
            } else {
                keep[r][0] = make_float4(0.f, 0.f, 0.f, 0.f);
                keep[r][1] = keep[r][0];
            }
        }
#pragma unroll
        for (int r = 0; r < kSplitHeld; ++r) {
            a_scan4(keep[r][0], mx);
            a_scan4(keep[r][1], mx);
        }
    } else {
        for (int g = tid; g < groups; g += 256) {
            float4 p, q;
            load8(g, p, q);
            a_scan4(p, mx);
            a_scan4(q, mx);
        }
    }
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((tid & 63) == 0) wmax[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const int x = a_row_exponent(mx);
    if (tid == 0) row_exp[row] = x;
    const int64_t mp = PIECES ? (static_cast<int64_t>(m) + 31) / 32 * 32 : m;
    half8v* hi = reinterpret_cast<half8v*>(ah);
    half8v* lo = reinterpret_cast<half8v*>(ah + mp * kp);
    auto split = [&](int g, const float4& p, const float4& q) {
        half8v h, l;
        a_split8<PIECES>(p, q, x, h, l);
        const int64_t at = a_piece<PIECES>(row, g, kp);
        hi[at] = h;
        lo[at] = l;
    };
    if (held) {
#pragma unroll
        for (int r = 0; r < kSplitHeld; ++r) {
            const int g = tid + r * 256;
            if (g < groups) split(g, keep[r][0], keep[r][1]);
        }
    } else {
        for (int g = tid; g < groups; g += 256) {
            float4 p, q;
            load8(g, p, q);
            split(g, p, q);
        }
    }
}


// The prep for k <= 6144 (GT = ceil(k / 2048) groups of
// eight per thread and row): R = 8 / GT rows per workgroup, held in
// registers between their maxima and their split.  Operand order puts 32
// rows side by side in every 1 KB piece, so one row alone writes 16 bytes
// per 512-byte half-piece; R consecutive rows give each thread an R x
// 16-byte run.
template <int R, int GT>
__global__ __launch_bounds__(256) void gemm_prep_frag_kernel(const float* __restrict__ a, _Float16* __restrict__ ah,
                                                             int* __restrict__ row_exp, int m, int k, int kp, int vec) {
    __shared__ float wmax[4 * R];
    const int tid = threadIdx.x;
    const int wg = a_stage_wg(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
    const int row0 = wg * R;
    const int groups = kp >> 3;
    float4 v[R][GT][2];
    float mx[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float* src = a + static_cast<int64_t>(row0 + r) * k;
#pragma unroll
        for (int u = 0; u < GT; ++u) {
            const int g = tid + u * 256;
            if (row0 + r < m && g < groups) {
                if (vec) {
                    v[r][u][0] = reinterpret_cast<const float4*>(src)[2 * g];
                    v[r][u][1] = reinterpret_cast<const float4*>(src)[2 * g + 1];
                } else {
                    load8_tail(src, 8 * g, k, v[r][u][0], v[r][u][1]);
                }
            } else {
                v[r][u][0] = make_float4(0.f, 0.f, 0.f, 0.f);
                v[r][u][1] = v[r][u][0];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        mx[r] = 0.0f;
#pragma unroll
        for (int u = 0; u < GT; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) a_scan4(v[r][u][h], mx[r]);
        for (int off = 32; off > 0; off >>= 1) mx[r] = fmaxf(mx[r], __shfl_xor(mx[r], off));
    }
    if ((tid & 63) == 0)
#pragma unroll
        for (int r = 0; r < R; ++r) wmax[(tid >> 6) * R + r] = mx[r];
    __syncthreads();
    int x[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
        x[r] = a_row_exponent(fmaxf(fmaxf(wmax[r], wmax[R + r]), fmaxf(wmax[2 * R + r], wmax[3 * R + r])));
    if (tid < R && row0 + tid < m) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (r == tid) row_exp[row0 + r] = x[r];
    }
    const int64_t mp = (static_cast<int64_t>(m) + 31) / 32 * 32;
    half8v* hi = reinterpret_cast<half8v*>(ah);
    half8v* lo = reinterpret_cast<half8v*>(ah + mp * kp);
#pragma unroll
    for (int u = 0; u < GT; ++u) {
        const int g = tid + u * 256;
        if (g >= groups) break;
        // rows row0 .. row0 + R - 1 (one 32-row block) are consecutive 16-byte pieces
        const int64_t base = (static_cast<int64_t>(row0 / 32) * (kp / 16) + g / 2) * 64 + row0 % 32 + 32 * (g % 2);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (row0 + r >= m) break;
            half8v h, l;
            a_split8<true>(v[r][u][0], v[r][u][1], x[r], h, l);
            hi[base + r] = h;
            lo[base + r] = l;
        }
    }
}

// fp16 or bf16 rows [m, k] to operand order as they are (a copy, zeros past
// k): workgroup (block of 32 rows, 8 8-groups), thread (row, 8-group), in a
// one-dimensional grid (at most 2^18 workgroups by gemm_kind's limits, where
// either count alone can pass the 65535 of grid y).
// Threads of one 8-group write 512 consecutive bytes; a row's eight groups
// are one 128-byte read.
__global__ __launch_bounds__(256) void gemm_prep_half_kernel(const uint16_t* __restrict__ a, u32x4* __restrict__ out,
                                                             int m, int k, int kp, int vec) {
    __shared__ u32x4 tile[32][9];
    const unsigned g_blocks = (static_cast<unsigned>(kp) / 8 + 7) / 8;
    const int g0 = static_cast<int>(blockIdx.x % g_blocks) * 8;
    const int row0 = static_cast<int>(blockIdx.x / g_blocks) * 32;
    {
        const int r = threadIdx.x / 8, g = threadIdx.x % 8;
        const int c = 8 * (g0 + g);
        u32x4 v = {0u, 0u, 0u, 0u};
        if (row0 + r < m && c < k) {
            const uint16_t* src = a + static_cast<int64_t>(row0 + r) * k + c;
            if (vec) {
                v = *reinterpret_cast<const u32x4*>(src);
            } else {
                uint32_t e[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) e[i] = c + i < k ? src[i] : 0u;
                v = u32x4{e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16};
            }
        }
        // k = 0..7 to the order 0, 4, 1, 5, 2, 6, 3, 7
        tile[r][g] = u32x4{__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
                           __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
    }
    __syncthreads();
    const int r = threadIdx.x % 32, g = threadIdx.x / 32;
    if (8 * (g0 + g) < kp)
        out[static_cast<int64_t>(row0 / 32) * (kp / 8) * 32 + static_cast<int64_t>(g0 + g) * 32 + r] = tile[r][g];
}

}  // namespace

// Rows per workgroup of the operand-order prep: the most (up to 8 / GT,
// a power of two) that still leave at least kPrepMinWgs row workgroups.
// VELOMIND_PREP_MIN_WGS overrides the minimum (measurement sweeps).
constexpr int kPrepMinWgs = 256;

static int prep_rows_per_wg(int m, int gt) {
    if (gt > 3) return 0;
    int min_wgs = kPrepMinWgs;
    if (const char* env = std::getenv("VELOMIND_PREP_MIN_WGS")) min_wgs = std::max(0, std::atoi(env));
    int r = 8 / gt;
    if (r == 8 / 3) r = 2;
    while (r > 1 && (m + r - 1) / r < min_wgs) r /= 2;
    return r;
}

// Shapes the MFMA kernels take: any K, N of at least one 16-column group,
// scale blocks of whole 32-row chunks, 32-bit buffer offsets.  Operand order
// pads K to a multiple of 32 (kp) and M to a multiple of 32.
// VM_HIP_EUNSUPPORTED: another kernel takes the shape.
static int gemm_kind(int m, int k, int n, int quant_type, int block_size, int* kind) {
    if (n < 16) return VM_HIP_EUNSUPPORTED;
    const int64_t kp = (static_cast<int64_t>(k) + 31) / 32 * 32;
    if ((static_cast<int64_t>(m) + 31) / 32 * 32 * kp * 4 >= (int64_t(1) << 31) || kp * n >= (int64_t(1) << 31) ||
        static_cast<int64_t>(n) * 128 * 4 >= (int64_t(1) << 31) ||
        static_cast<int64_t>(m) * n * 4 * 16 >= (int64_t(1) << 40) ||
        ((static_cast<int64_t>(m) + 15) / 16) * ((n + 63) / 64) * 16 >= (int64_t(1) << 30))
        return VM_HIP_EUNSUPPORTED;
    *kind = quant_type == VM_HIP_QUANT_INT4 ? 2 : block_size > 0 ? 1 : 0;
    if (*kind != 0 && (block_size <= 0 || block_size % 32 != 0)) return VM_HIP_EUNSUPPORTED;
    return 0;
}

// The staged layouts of a shape for its producers: whole 32-row chunks of K
// and 16-column groups of N; few rows of per-column INT8 are staged
// row-major, everything else in operand order.
int gemm_plan(int m, int k, int n, int quant_type, int block_size, GemmPlan* plan) {
    if (m <= 4 || k % 32 != 0 || n % 16 != 0) return VM_HIP_EUNSUPPORTED;
    VM_TRY(gemm_kind(m, k, n, quant_type, block_size, &plan->kind));
    plan->pieces = plan->kind != 0 || m > 32;
    return 0;
}

int gemm_qmm_staged_f32(const GemmPlan& plan, const _Float16* ah, const int* row_exp,
                        const uint8_t* wq, const float* scale, float* c, int m, int k, int n, int block_size,
                        hipStream_t stream) {
    return quad_qmm_f32(GemmOperands{ah, plan.pieces ? 0 : 1, row_exp, wq, scale, false, c, m, k, n, block_size, plan.kind},
                        stream);
}

// Ragged calls so small that one launch with a thread per output, a serial
// chain over K, takes less than staging and GEMM, which take 7 to 8 us at any
// such size (generic / MFMA): per-column INT8 33 rows of 31 x 130 4.7 / 7.3 us,
// of 48 x 1027 6.4 / 7.7, of 63 x 130 7.7 / 7.7, of 63 x 65 6.6 / 7.4, of 80 x 31
// 7.1 / 7.7, 512 rows of 48 x 515 6.8 / 7.7, of 31 x 1027 8.1 / 8.1; INT4 33 rows
// of 33 x 130 6.4 / 8.1, of 45 x 17 7.2 / 7.9, of 48 x 130 8.4 / 7.9, 512 rows of
// 16 x 515 5.9 / 8.4, of 31 x 515 8.9 / 8.3.
static bool generic_is_faster(int kind, int m, int k, int n) {
    const double work = static_cast<double>(m) * n * k;
    if (kind == 0) return work <= 13e6 && (k <= 48 || (k <= 72 && n <= 80) || (k <= 80 && n <= 40));
    return work <= 4.4e6 && (k <= 40 || (k <= 46 && n <= 40));
}

int gemm_qmm_f32(const float* a, const uint8_t* wq, const float* scale, float* c, int m, int k, int n,
                 int quant_type, int block_size, hipStream_t stream) {
    // Operand order for every shape (it reads faster than rows: M = 16,
    // K = 2048, N = 5632 INT8 9.9 us against 10.8), K padded with zeros.
    GemmPlan plan;
    VM_TRY(gemm_kind(m, k, n, quant_type, block_size, &plan.kind));
    const int kp = (k + 31) / 32 * 32;
    // Few rows so long that operand order's 32 are more than the no-allocation
    // entry point's array holds: per-column INT8 takes them row by row (in
    // every entry point, so that all give the same bits).
    plan.pieces = !(plan.kind == 0 && m <= 32 && k % 32 == 0 && n % 16 == 0 &&
                    a_stage_bytes(m, kp, true) > kStaticPartialBytes);
    const std::size_t bytes = a_stage_bytes(m, kp, plan.pieces);
    // A ragged shape whose scratch is refused keeps the generic kernel, which
    // needs none.
    const bool ragged = k % 32 != 0 || n % 16 != 0;
    if (ragged && generic_is_faster(plan.kind, m, k, n)) return VM_HIP_EUNSUPPORTED;
    void* aux = nullptr;
    int rc = get_aux(stream, bytes, &aux);
    if (ragged && scratch_refused(rc)) return VM_HIP_EUNSUPPORTED;
    VM_TRY(rc);
    auto* ah = static_cast<_Float16*>(aux);
    auto* row_exp = reinterpret_cast<int*>(static_cast<char*>(aux) + a_stage_half_bytes(m, kp, plan.pieces));
    const int vec = k % 32 == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0 ? 1 : 0;
    const int gt = (kp / 8 + 255) / 256;
    const int rows_per_wg = prep_rows_per_wg(m, gt);
    if (!plan.pieces) {
        hipLaunchKernelGGL(gemm_prep_kernel<false>, dim3(m), dim3(256), 0, stream, a, ah, row_exp, m, k, kp, vec);
    } else
#define VM_PREP(RX, GX)                                                                                           \
    if (gt == GX && rows_per_wg == RX)                                                                            \
        hipLaunchKernelGGL((gemm_prep_frag_kernel<RX, GX>), dim3((m + RX - 1) / RX), dim3(256), 0, stream, a, ah, \
                           row_exp, m, k, kp, vec);                                                               \
    else
    VM_PREP(8, 1) VM_PREP(4, 1) VM_PREP(2, 1) VM_PREP(1, 1) VM_PREP(4, 2) VM_PREP(2, 2) VM_PREP(1, 2)
    VM_PREP(2, 3) VM_PREP(1, 3)
#undef VM_PREP
        hipLaunchKernelGGL(gemm_prep_kernel<true>, dim3(m), dim3(256), 0, stream, a, ah, row_exp, m, k, kp, vec);
    VM_TRY(check_launch("QuantizedMatMul", stream));
    rc = gemm_qmm_staged_f32(plan, ah, row_exp, wq, scale, c, m, k, n, block_size, stream);
    return ragged && scratch_refused(rc) ? VM_HIP_EUNSUPPORTED : rc;
}

constexpr int kHalfRowsDirect = 128;

int gemm_qmm_half(const uint16_t* a, bool bf16, const uint8_t* wq, const void* scale, bool scale_half, uint16_t* c,
                  int m, int k, int n, int quant_type, int block_size, hipStream_t stream) {
    GemmOperands o{a, 1, nullptr, wq, scale, scale_half, c, m, k, n, block_size, 0};
    // Scratch that cannot grow during graph capture leaves the call to the
    // staged fp32 form, whose buffer an earlier call may have sized.
    const auto refused = [](int rc) { return scratch_refused(rc) ? VM_HIP_EUNSUPPORTED : rc; };
    VM_TRY(gemm_kind(m, k, n, quant_type, block_size, &o.kind));
    const int kp = (k + 31) / 32 * 32;
    const bool aligned = reinterpret_cast<uintptr_t>(a) % 16 == 0;
    // Few rows are read where they lie (a row-major operand load touches one
    // line per row, but a second launch costs more: M = 64, 2048 x 5632 INT4
    // 11.6 us against 13.0, M = 128, 960 x 2560 8.0 against 9.6).
    if (k % 32 != 0 || !aligned || m > kHalfRowsDirect) {
        void* aux = nullptr;
        const int rc = get_aux(stream, a_stage_half_bytes(m, kp, true) / 2, &aux);
        if (rc != 0) return refused(rc);
        hipLaunchKernelGGL(gemm_prep_half_kernel, dim3((kp / 8 + 7) / 8 * ((m + 31) / 32)), dim3(256), 0, stream, a,
                           static_cast<u32x4*>(aux), m, k, kp, k % 8 == 0 && aligned ? 1 : 0);
        VM_TRY(check_launch("QuantizedMatMul", stream));
        o.a = aux;
        o.layout = 0;
    }
    return refused(quad_qmm_half(o, bf16, stream));
}

}  // namespace vmhip
