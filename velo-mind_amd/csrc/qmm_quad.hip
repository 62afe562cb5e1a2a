// The MFMA quantized matmul (qmm_quad_impl.h) for fp32 activations, staged
// as two fp16 parts.
#include "qmm_quad_impl.h"

namespace vmhip {

int quad_qmm_f32(const GemmOperands& o, hipStream_t s) {
    if (o.layout == AM_PIECES) return launch_kind<AM_PIECES, EL_F32, false>(o, s);
    // row-major parts are staged for per-column INT8 only (gemm_plan)
    return o.kind == 0 ? launch_mode<0, AM_ROWS, EL_F32, false>(o, s) : VM_HIP_EUNSUPPORTED;
}

}  // namespace vmhip
