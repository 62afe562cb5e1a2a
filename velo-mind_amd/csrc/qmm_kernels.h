// Internal launchers shared between the libvmhip translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace vmhip {

// Decode-shaped GEMV for 1 <= m <= 4 rows (qmm_gemv.hip).  Returns
// VM_HIP_EUNSUPPORTED when the shape/alignment needs another kernel.  A
// non-null `addend` [m, n] is added to each output (addend + A x W, one fp32
// addition after the product's last rounding).  A non-null `a_up` [m, k]
// makes the activations the SwiGLU product silu_mul_f32(a, a_up).
int gemv_qmm_f32(const float* a, const uint8_t* wq, const float* scale, float* c, int m, int k,
                 int n, int quant_type, int block_size, hipStream_t stream, const float* addend = nullptr,
                 const float* a_up = nullptr);

// The same GEMV for `count` (<= 4) matrices sharing the activations, in one
// launch (qmm_gemv.hip); VM_HIP_EUNSUPPORTED when a member needs another
// kernel.
// With a non-null norm_w, each row of A is first RMS-normalized (the
// separate RMSNorm kernel's arithmetic, bit for bit): C_g = RMSNorm(A) x W_g.
int gemv_qmm_group_f32(const float* a, const uint8_t* const* wq, const float* const* scale, float* const* c,
                       const int* n, int count, int m, int k, int quant_type, int block_size, hipStream_t stream,
                       const float* norm_w = nullptr, float norm_eps = 0.0f);

// The kernels with fused extras (qmm_gemv_fx.hip), reached through the two
// functions above when an extra is non-null: addend (one matrix only),
// norm_w or a_up (not both).
int gemv_qmm_fx_f32(const float* a, const uint8_t* const* wq, const float* const* scale, float* const* c,
                    const int* n, int count, int m, int k, int quant_type, int block_size, hipStream_t stream,
                    const float* addend, const float* norm_w, float norm_eps, const float* a_up);

// Prefill-shaped MFMA GEMM for m > 4 rows (qmm_gemm.hip).
int gemm_qmm_f32(const float* a, const uint8_t* wq, const float* scale, float* c, int m, int k,
                 int n, int quant_type, int block_size, hipStream_t stream);

// The same for fp16 or bf16 activations and outputs (any m >= 1); scales fp32
// or, with scale_half, of the same 16-bit type.
int gemm_qmm_half(const uint16_t* a, bool bf16, const uint8_t* wq, const void* scale, bool scale_half, uint16_t* c,
                  int m, int k, int n, int quant_type, int block_size, hipStream_t stream);

// How the GEMM takes A staged by its producer: kind 0 = INT8 per column, 1 =
// INT8 blockwise, 2 = INT4; `pieces`: operand order (else row-major,
// a_split.h).  VM_HIP_EUNSUPPORTED for shapes whose producers write fp32
// (rows <= 4, K % 32, N % 16, sizes past 32-bit offsets); gemm_qmm_f32 and
// gemm_qmm_half stage ragged K and N themselves.
struct GemmPlan {
    int kind = 0;
    bool pieces = false;
};
int gemm_plan(int m, int k, int n, int quant_type, int block_size, GemmPlan* plan);
// One call of the MFMA kernel (qmm_quad_impl.h).
struct GemmOperands {
    const void* a;
    int layout;             // 0 operand order, 1 row-major
    const int* row_exp;     // fp32 only: the rows' staging exponents
    const uint8_t* wq;
    const void* scale;
    bool scale_half;        // scales of A's 16-bit type
    void* c;
    int m, k, n, block_size;
    int kind;               // 0 INT8 per column, 1 INT8 blockwise, 2 INT4
};
int quad_qmm_f32(const GemmOperands& o, hipStream_t stream);
int quad_qmm_half(const GemmOperands& o, bool bf16, hipStream_t stream);
// The GEMM on A staged by its producer (a_split.h layout for the plan).
int gemm_qmm_staged_f32(const GemmPlan& plan, const _Float16* ah, const int* row_exp, const uint8_t* wq,
                        const float* scale, float* c, int m, int k, int n, int block_size, hipStream_t stream);

// Any-shape reference-order kernel used for layouts the fast kernels do
// not cover (odd N, block sizes that are not multiples of 32).
int generic_qmm_f32(const float* a, const uint8_t* wq, const float* scale, float* c, int m, int k,
                    int n, int quant_type, int block_size, hipStream_t stream);

// Argument checks of vm_hip_qmm_f32 (0 or an error status).
int validate_qmm(const void* a, const int8_t* wq, const void* scale, const void* c, int64_t m, int64_t k,
                 int64_t n, int quant_type, int block_size);

// Routing behind vm_hip_qmm_f32 for validated arguments: GEMV (rows <= 4),
// MFMA GEMM (rows > 4) or the generic kernel.
int qmm_f32_impl(const float* a, const int8_t* wq, const float* scale, float* c, int64_t m, int64_t k,
                 int64_t n, int quant_type, int block_size, hipStream_t stream);

}  // namespace vmhip
