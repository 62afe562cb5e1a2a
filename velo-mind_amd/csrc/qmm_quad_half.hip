// The MFMA quantized matmul (qmm_quad_impl.h) for fp16 and bf16 activations
// and outputs.
#include "qmm_quad_impl.h"

namespace vmhip {
namespace {

template <int EL>
int launch_half(const GemmOperands& o, hipStream_t s) {
    if (o.layout == AM_PIECES)
        return o.scale_half ? launch_kind<AM_PIECES, EL, true>(o, s) : launch_kind<AM_PIECES, EL, false>(o, s);
    return o.scale_half ? launch_kind<AM_ROWS, EL, true>(o, s) : launch_kind<AM_ROWS, EL, false>(o, s);
}

}  // namespace

int quad_qmm_half(const GemmOperands& o, bool bf16, hipStream_t s) {
    return bf16 ? launch_half<EL_BF16>(o, s) : launch_half<EL_F16>(o, s);
}

}  // namespace vmhip
