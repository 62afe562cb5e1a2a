// Weight packing on the device, bit-exact with the reference's host
// packers (src/quant.cpp:74-104 INT8, :125-175 INT4), plus the inverse
// maps and half->fp32 widening.
//
// Exactness: the scale is a correctly rounded fp32 division (max / 127 or
// max / 7; built with -fhip-fp32-correctly-rounded-divide-sqrt and without
// fast-math), the reciprocal is a correctly rounded 1 / scale that is then
// multiplied, roundf() rounds half away from zero, and the clamp and the
// int8 cast follow.  Only finite inputs are in the contract (the
// reference's float->int8 cast of NaN/Inf is undefined).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "vm_internal.h"

namespace vmhip {
namespace {

constexpr int kColsPerWg = 64;
constexpr int kRowGroups = 4;

// One workgroup owns 64 columns; 4 row groups find the column maxima
// together, then every thread quantizes its own rows.
__global__ __launch_bounds__(kColsPerWg * kRowGroups) void pack_int8_kernel(
    const float* __restrict__ w, int8_t* __restrict__ q, float* __restrict__ scale, int64_t rows,
    int64_t cols) {
    __shared__ float smax[kRowGroups][kColsPerWg];
    const int tx = threadIdx.x % kColsPerWg;
    const int ty = threadIdx.x / kColsPerWg;
    const int64_t c = static_cast<int64_t>(blockIdx.x) * kColsPerWg + tx;
    float m = 0.0f;
    if (c < cols) {
        for (int64_t r = ty; r < rows; r += kRowGroups) {
            const float v = fabsf(w[r * cols + c]);
            if (v > m) m = v;
        }
    }
    smax[ty][tx] = m;
    __syncthreads();
    float amax = smax[0][tx];
    for (int g = 1; g < kRowGroups; ++g) amax = smax[g][tx] > amax ? smax[g][tx] : amax;
    if (c >= cols) return;
    const float s = amax > 0.0f ? amax / 127.0f : 1.0f;
    const float inv = 1.0f / s;
    if (ty == 0) scale[c] = s;
    for (int64_t r = ty; r < rows; r += kRowGroups) {
        float v = roundf(w[r * cols + c] * inv);
        v = v < -127.0f ? -127.0f : (127.0f < v ? 127.0f : v);
        q[r * cols + c] = static_cast<int8_t>(v);
    }
}

// V adjacent columns of a row (16-byte loads with V = 4; V = 1 where cols
// or a pointer rules them out).
template <int V>
struct Columns {
    float e[V];
};

// Two-pass INT8 packing (a workgroup of the single-pass kernel scans all rows
// of 64 columns, a serial chain of loads that leaves the GPU mostly idle).
// Four waves of 64 V columns:
//   pass 1: the maximum |w| of the columns over a chunk of rows, kPackRows
//           loads in flight per wave, the waves' maxima joined in LDS, one
//           partial per chunk;
//   pass 2: a wave requests its kPackRows rows, then the column maxima are
//           joined from the partials (max is exact in any order) while those
//           are in flight, then quant.cpp's scale / reciprocal / round /
//           clamp, V codes per store.
// At most 32 chunks (pass 2 reads every partial).  Against one wave's columns
// per thread group and no join: 5632 x 2048 55.7 -> 32.1 us, 2048 x 5632 31.1
// -> 26.2; odd widths, 2048 x 5633, 280 -> 40.
// The comparison `v > m` skips NaN, as the single-pass kernel does.
constexpr int kPackRows = 16;
constexpr int kPackMaxChunks = 32;

template <int V>
__device__ __forceinline__ void load_rows(const float* __restrict__ w, int64_t r0, int64_t r1, int64_t cols, int64_t c,
                                          Columns<V> (&x)[kPackRows]) {
#pragma unroll
    for (int u = 0; u < kPackRows; ++u) {
        if (r0 + u < r1 && c < cols) {
            __builtin_memcpy(&x[u], __builtin_assume_aligned(w + (r0 + u) * cols + c, 4 * V), 4 * V);
        } else {
#pragma unroll
            for (int v = 0; v < V; ++v) x[u].e[v] = 0.0f;
        }
    }
}

// Column maxima of the four waves, joined in every wave.
template <int V>
__device__ __forceinline__ void join_max(float (&m)[V], float (*smax)[64][V], int wave, int lane) {
#pragma unroll
    for (int v = 0; v < V; ++v) smax[wave][lane][v] = m[v];
    __syncthreads();
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int v = 0; v < V; ++v) m[v] = smax[g][lane][v] > m[v] ? smax[g][lane][v] : m[v];
}

template <int V>
__global__ __launch_bounds__(256) void pack_int8_colmax_kernel(const float* __restrict__ w, float* __restrict__ part,
                                                               int64_t rows, int64_t cols, int64_t rows_per_chunk) {
    __shared__ float smax[4][64][V];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t c = (static_cast<int64_t>(blockIdx.x) * 64 + lane) * V;
    const int64_t r0 = static_cast<int64_t>(blockIdx.y) * rows_per_chunk;
    const int64_t r1 = min(rows, r0 + rows_per_chunk);
    float m[V] = {};
    for (int64_t r = r0 + wave * kPackRows; r < r1; r += 4 * kPackRows) {
        Columns<V> x[kPackRows];
        load_rows<V>(w, r, r1, cols, c, x);
#pragma unroll
        for (int u = 0; u < kPackRows; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v) m[v] = fabsf(x[u].e[v]) > m[v] ? fabsf(x[u].e[v]) : m[v];
    }
    join_max<V>(m, smax, wave, lane);
    if (wave == 0 && c < cols) {
#pragma unroll
        for (int v = 0; v < V; ++v) part[static_cast<int64_t>(blockIdx.y) * cols + c + v] = m[v];
    }
}

__device__ __forceinline__ uint32_t int8_code(float x, float inv) {
    float v = roundf(x * inv);
    v = v < -127.0f ? -127.0f : (127.0f < v ? 127.0f : v);
    return static_cast<uint32_t>(static_cast<uint8_t>(static_cast<int8_t>(v)));
}

template <int V>
__global__ __launch_bounds__(256) void pack_int8_quantize_kernel(const float* __restrict__ w,
                                                                 const float* __restrict__ part, int chunks,
                                                                 int8_t* __restrict__ q, float* __restrict__ scale,
                                                                 int64_t rows, int64_t cols) {
    __shared__ float smax[4][64][V];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t c = (static_cast<int64_t>(blockIdx.x) * 64 + lane) * V;
    const int64_t r0 = (static_cast<int64_t>(blockIdx.y) * 4 + wave) * kPackRows;
    Columns<V> x[kPackRows];
    load_rows<V>(w, r0, rows, cols, c, x);
    float m[V] = {};
#pragma unroll
    for (int i = 0; i < kPackMaxChunks / 4; ++i) {
        const int ch = wave + 4 * i;
        if (ch < chunks && c < cols) {
            Columns<V> p;
            __builtin_memcpy(&p, part + static_cast<int64_t>(ch) * cols + c, 4 * V);
#pragma unroll
            for (int v = 0; v < V; ++v) m[v] = p.e[v] > m[v] ? p.e[v] : m[v];
        }
    }
    join_max<V>(m, smax, wave, lane);
    if (c >= cols) return;
    float inv[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const float sc = m[v] > 0.0f ? m[v] / 127.0f : 1.0f;   // quant.cpp:94-96
        inv[v] = 1.0f / sc;
        if (blockIdx.y == 0 && wave == 0) scale[c + v] = sc;
    }
#pragma unroll
    for (int u = 0; u < kPackRows; ++u) {
        uint32_t b = 0;
#pragma unroll
        for (int v = 0; v < V; ++v) b |= int8_code(x[u].e[v], inv[v]) << (8 * v);
        if (r0 + u < rows) __builtin_memcpy(__builtin_assume_aligned(q + (r0 + u) * cols + c, V), &b, V);
    }
}

__device__ __forceinline__ unsigned int4_code(float x, float inv) {
    float v = roundf(x * inv);
    v = v < -8.0f ? -8.0f : (7.0f < v ? 7.0f : v);
    return static_cast<unsigned>(static_cast<int8_t>(v)) & 0xFu;
}

// INT4 blocks of 32 * G rows, G a power of two up to 4: bandwidth-bound, so
// the matrix is read once.  A thread holds 32 rows of V adjacent columns
// (all its loads in flight at once, 16 bytes each with V = 4), finds their
// maxima, the G waves of a block exchange theirs through LDS, and the held
// values are quantized and stored V packed bytes at a time.  Four waves
// cover 4 / G blocks.  2048 x 32000, blocks of 32: 67 us (4.4 TB/s; a
// copy reaches 5.1), against 113 with a thread per block and column, which
// reads 4 bytes a lane, twice.
template <int V, int G>
__global__ __launch_bounds__(256) void pack_int4_rows_kernel(const float* __restrict__ w, uint8_t* __restrict__ packed,
                                                             float* __restrict__ scale, int64_t rows, int64_t cols) {
    constexpr int R = 32;
    __shared__ float smax[4][64][V];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t c = (static_cast<int64_t>(blockIdx.x) * 64 + lane) * V;
    const int64_t r0 = (static_cast<int64_t>(blockIdx.y) * 4 + wave) * R;
    const bool in = c < cols;
    Columns<V> x[R];
    const float* src = w + r0 * cols + c;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (in && r0 + r < rows) {
            __builtin_memcpy(&x[r], __builtin_assume_aligned(src + r * cols, 4 * V), 4 * V);
        } else {
#pragma unroll
            for (int v = 0; v < V; ++v) x[r].e[v] = 0.0f;
        }
    }
    float amax[V];
#pragma unroll
    for (int v = 0; v < V; ++v) amax[v] = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int v = 0; v < V; ++v) amax[v] = fabsf(x[r].e[v]) > amax[v] ? fabsf(x[r].e[v]) : amax[v];   // skips NaN
    if constexpr (G > 1) {
#pragma unroll
        for (int v = 0; v < V; ++v) smax[wave][lane][v] = amax[v];
        __syncthreads();
        const int first = wave & ~(G - 1);
#pragma unroll
        for (int v = 0; v < V; ++v) {
            float m = smax[first][lane][v];
#pragma unroll
            for (int g = 1; g < G; ++g) m = smax[first + g][lane][v] > m ? smax[first + g][lane][v] : m;
            amax[v] = m;
        }
    }
    if (!in || r0 >= rows) return;
    Columns<V> s;
    float inv[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        s.e[v] = amax[v] > 0.0f ? amax[v] / 7.0f : 1.0f;
        inv[v] = 1.0f / s.e[v];
    }
    if (wave % G == 0)
        __builtin_memcpy(__builtin_assume_aligned(scale + r0 / (R * G) * cols + c, 4 * V), &s, 4 * V);
    uint8_t* dst = packed + r0 / 2 * cols + c;
#pragma unroll
    for (int r = 0; r < R; r += 2) {
        uint32_t b = 0;
#pragma unroll
        for (int v = 0; v < V; ++v)   // rows past the matrix hold zeros, code 0
            b |= (int4_code(x[r].e[v], inv[v]) | int4_code(x[r + 1].e[v], inv[v]) << 4) << (8 * v);
        if (r0 + r < rows) __builtin_memcpy(__builtin_assume_aligned(dst + r / 2 * cols, V), &b, V);
    }
}

// Any other block size: one thread per (scale block, column); blocks are even, so every packed
// byte belongs to exactly one thread.
__global__ __launch_bounds__(256) void pack_int4_kernel(const float* __restrict__ w,
                                                        uint8_t* __restrict__ packed,
                                                        float* __restrict__ scale, int64_t rows,
                                                        int64_t cols, int64_t block) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t b = blockIdx.y;
    if (c >= cols) return;
    const int64_t r0 = b * block;
    const int64_t r1 = r0 + block < rows ? r0 + block : rows;
    float amax = 0.0f;
    for (int64_t r = r0; r < r1; ++r) {
        const float v = fabsf(w[r * cols + c]);
        if (v > amax) amax = v;
    }
    const float s = amax > 0.0f ? amax / 7.0f : 1.0f;
    const float inv = 1.0f / s;
    scale[b * cols + c] = s;
    for (int64_t r = r0; r < r1; r += 2) {
        const unsigned lo = int4_code(w[r * cols + c], inv);
        const unsigned hi = (r + 1 < r1) ? int4_code(w[(r + 1) * cols + c], inv) : 0u;
        packed[(r / 2) * cols + c] = static_cast<uint8_t>(lo | (hi << 4));
    }
}

__global__ void dequant_int8_kernel(const int8_t* __restrict__ q, const float* __restrict__ scale,
                                    float* __restrict__ w, int64_t rows, int64_t cols) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= rows * cols) return;
    w[idx] = static_cast<float>(q[idx]) * scale[idx % cols];
}

__device__ __forceinline__ int nib(unsigned v) {
    v &= 0xFu;
    return (v & 8u) ? static_cast<int>(v) - 16 : static_cast<int>(v);
}

// Row r of block b reads the pair that the reference's block-local pair
// loop assigns to it (src/quant.cpp:197-205); for even blocks that is byte
// row r/2, nibble r%2.
__global__ void dequant_int4_kernel(const uint8_t* __restrict__ packed,
                                    const float* __restrict__ scale, float* __restrict__ w,
                                    int64_t rows, int64_t cols, int64_t block) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= rows * cols) return;
    const int64_t r = idx / cols;
    const int64_t c = idx - r * cols;
    const int64_t b = r / block;
    const int64_t r0 = b * block;
    const int64_t pair_row = r0 + ((r - r0) & ~int64_t(1));
    const unsigned byte = packed[(pair_row / 2) * cols + c];
    const int code = ((r - r0) & 1) ? nib(byte >> 4) : nib(byte);
    w[idx] = static_cast<float>(code) * scale[b * cols + c];
}

// dtype.h:21-51 (exact widening, NaN made quiet) and :91-95.
__global__ void half_to_f32_kernel(const uint16_t* __restrict__ src, float* __restrict__ dst,
                                   int64_t count, int is_bf16, float factor) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const uint32_t h = src[i];
    uint32_t f;
    if (is_bf16) {
        f = h << 16;
    } else {
        const uint32_t sign = (h & 0x8000u) << 16;
        const uint32_t e = (h >> 10) & 0x1Fu;
        uint32_t m = h & 0x3FFu;
        if (e == 0) {
            if (m == 0) {
                f = sign;
            } else {
                int ex = -14;
                while (!(m & 0x400u)) { m <<= 1; --ex; }
                f = sign | (static_cast<uint32_t>(ex + 127) << 23) | ((m & 0x3FFu) << 13);
            }
        } else if (e == 0x1F) {
            f = sign | 0x7F800000u | (m << 13) | (m ? 0x400000u : 0u);
        } else {
            f = sign | ((e + 112u) << 23) | (m << 13);
        }
    }
    dst[i] = factor == 1.0f ? __uint_as_float(f) : __uint_as_float(f) * factor;   // NaN bits stay at 1
}

unsigned grid_1d(int64_t count, int threads) {
    return static_cast<unsigned>((count + threads - 1) / threads);
}

}  // namespace
int half_to_f32_times(const uint16_t* src, bool bf16, float* dst, int64_t count, float factor, hipStream_t stream) {
    hipLaunchKernelGGL(half_to_f32_kernel, dim3(grid_1d(count, 256)), dim3(256), 0, stream, src, dst, count, bf16 ? 1 : 0,
                       factor);
    return check_launch("ConvertDtype", stream);
}

}  // namespace vmhip

using namespace vmhip;

extern "C" {

int vm_hip_pack_int8(const float* w, int8_t* q, float* scale, int64_t rows, int64_t cols,
                     void* stream) {
    if (rows < 0 || cols < 0) return fail_inval("vm_hip_pack_int8: negative shape");
    if (rows == 0 || cols == 0) return 0;  // quant.cpp:81-83
    if (!w || !q || !scale) return fail_inval("vm_hip_pack_int8: null pointer");
    VM_TRY(injected_failure("QuantizePack", "launch"));
    auto s = static_cast<hipStream_t>(stream);
    // Two passes for matrices wide and tall enough to fill the GPU, when the
    // stream is not being captured (the row partials use the stream's
    // workspace, sized here; refused memory leaves the single pass, which
    // needs none) and the second pass's grid holds the rows.
    // The single pass walks all rows of a column and is the faster one up to
    // about 108 of them (64 x 2049 6.7 us against 9.4, 100 x 515 9.4 and 9.8, 128 x
    // 515 11.4 and 9.9); four columns a lane pay from more than one workgroup of
    // the second pass per compute unit (1000 x 8192 18.8 us against 24.8 with one
    // column; 512 x 8192 12.9 and 12.6, 2048 x 2048 13.8 and 12.5, 512 x 516 17.6
    // and 10.1).
    const int64_t row_groups = (rows + 4 * kPackRows - 1) / (4 * kPackRows);
    const bool vec = cols % 4 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(q) % 4 == 0 && row_groups * ((cols + 255) / 256) > 256;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (s) (void)hipStreamIsCapturing(s, &cap);
    if (rows > 108 && cols >= 256 && row_groups <= 65535 && cap == hipStreamCaptureStatusNone) {
        const int64_t col_groups = (cols + (vec ? 255 : 63)) / (vec ? 256 : 64);
        // about 1024 workgroups, whole steps of 64 rows each
        int64_t chunks = std::min<int64_t>({(1024 + col_groups - 1) / col_groups, row_groups, kPackMaxChunks});
        const int64_t rpc = (row_groups + chunks - 1) / chunks * (4 * kPackRows);
        chunks = (rows + rpc - 1) / rpc;
        Workspace ws{};
        const int rc = get_workspace(s, static_cast<std::size_t>(chunks * cols), 0, &ws);
        if (rc != 0 && !scratch_refused(rc)) return rc;
        if (rc == 0) {
            const dim3 grid(static_cast<unsigned>(col_groups), static_cast<unsigned>(chunks));
            const dim3 grid2(static_cast<unsigned>(col_groups), static_cast<unsigned>(row_groups));
            if (vec) {
                hipLaunchKernelGGL(pack_int8_colmax_kernel<4>, grid, dim3(256), 0, s, w, ws.partials, rows, cols, rpc);
                hipLaunchKernelGGL(pack_int8_quantize_kernel<4>, grid2, dim3(256), 0, s, w, ws.partials,
                                   static_cast<int>(chunks), q, scale, rows, cols);
            } else {
                hipLaunchKernelGGL(pack_int8_colmax_kernel<1>, grid, dim3(256), 0, s, w, ws.partials, rows, cols, rpc);
                hipLaunchKernelGGL(pack_int8_quantize_kernel<1>, grid2, dim3(256), 0, s, w, ws.partials,
                                   static_cast<int>(chunks), q, scale, rows, cols);
            }
            return check_launch("QuantizePack", s);
        }
    }
    hipLaunchKernelGGL(pack_int8_kernel, dim3(grid_1d(cols, kColsPerWg)), dim3(kColsPerWg * kRowGroups),
                       0, s, w, q, scale, rows, cols);
    return check_launch("QuantizePack", s);
}

int vm_hip_pack_int4(const float* w, uint8_t* packed, float* scale, int64_t rows, int64_t cols,
                     int64_t block, void* stream) {
    if (rows < 0 || cols < 0) return fail_inval("vm_hip_pack_int4: negative shape");
    if (block <= 0) return fail_inval("vm_hip_pack_int4: block_size must be positive");
    if (block % 2 != 0) return fail_inval("vm_hip_pack_int4: block_size must be even");
    if (rows == 0 || cols == 0) return 0;
    if (!w || !packed || !scale) return fail_inval("vm_hip_pack_int4: null pointer");
    const int64_t nblk = (rows + block - 1) / block;
    if (nblk > 65535) return fail_inval("vm_hip_pack_int4: too many scale blocks");
    auto s = static_cast<hipStream_t>(stream);
    if (block == 32 || block == 64 || block == 128) {
        const bool vec = cols % 4 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                         reinterpret_cast<uintptr_t>(packed) % 4 == 0 && reinterpret_cast<uintptr_t>(scale) % 16 == 0;
        const int64_t groups = (rows + 127) / 128;   // (at most 65535, as the blocks above)
        // Four columns a lane where that still leaves a workgroup for every
        // compute unit; fewer are bound by one wave's 128 codes a lane and
        // take one column (blocks of 32: 2048 x 4096, 256 workgroups, 10.2 us
        // against 11.9 with one; 2048 x 2048 8.8 and 5.7, 512 x 1028 19.2 and 5.0).
        const bool wide = vec && groups * ((cols + 255) / 256) >= 256;
#define VM_PACK4(VX, GX)                                                                                             \
    hipLaunchKernelGGL((pack_int4_rows_kernel<VX, GX>), dim3(grid_1d(cols, 64 * VX), static_cast<unsigned>(groups)), \
                       dim3(256), 0, s, w, packed, scale, rows, cols)
        if (wide) {
            if (block == 32) VM_PACK4(4, 1);
            else if (block == 64) VM_PACK4(4, 2);
            else VM_PACK4(4, 4);
        } else {
            if (block == 32) VM_PACK4(1, 1);
            else if (block == 64) VM_PACK4(1, 2);
            else VM_PACK4(1, 4);
        }
#undef VM_PACK4
        return check_launch("QuantizePack", s);
    }
    hipLaunchKernelGGL(pack_int4_kernel, dim3(grid_1d(cols, 256), static_cast<unsigned>(nblk)), dim3(256),
                       0, s, w, packed, scale, rows, cols, block);
    return check_launch("QuantizePack", s);
}

int vm_hip_dequant_int8(const int8_t* q, const float* scale, float* w, int64_t rows, int64_t cols,
                        void* stream) {
    if (rows < 0 || cols < 0) return fail_inval("vm_hip_dequant_int8: negative shape");
    if (rows == 0 || cols == 0) return 0;
    if (!q || !scale || !w) return fail_inval("vm_hip_dequant_int8: null pointer");
    auto s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(dequant_int8_kernel, dim3(grid_1d(rows * cols, 256)), dim3(256), 0, s, q, scale,
                       w, rows, cols);
    return check_launch("Dequantize", s);
}

int vm_hip_dequant_int4(const uint8_t* packed, const float* scale, float* w, int64_t rows,
                        int64_t cols, int64_t block, void* stream) {
    if (rows < 0 || cols < 0) return fail_inval("vm_hip_dequant_int4: negative shape");
    if (block <= 0) return fail_inval("vm_hip_dequant_int4: block_size must be positive");
    if (rows == 0 || cols == 0) return 0;
    if (!packed || !scale || !w) return fail_inval("vm_hip_dequant_int4: null pointer");
    auto s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(dequant_int4_kernel, dim3(grid_1d(rows * cols, 256)), dim3(256), 0, s, packed,
                       scale, w, rows, cols, block);
    return check_launch("Dequantize", s);
}

int vm_hip_half_to_f32(const uint16_t* src, int src_dtype, float* dst, int64_t count, void* stream) {
    if (src_dtype != VM_HIP_DTYPE_F16 && src_dtype != VM_HIP_DTYPE_BF16)
        return fail_inval("vm_hip_half_to_f32: source dtype must be Float16 or BFloat16");
    if (count < 0) return fail_inval("vm_hip_half_to_f32: negative count");
    if (count == 0) return 0;
    if (!src || !dst) return fail_inval("vm_hip_half_to_f32: null pointer");
    return half_to_f32_times(src, src_dtype == VM_HIP_DTYPE_BF16, dst, count, 1.0f, static_cast<hipStream_t>(stream));
}

}  // extern "C"
