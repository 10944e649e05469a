// The guarded tiles with M- / N-major operands (gemm_mfma_w4_majors.hpp): f16 operands.
#include "gemm_mfma_w4_kernel.hpp"
#include "gemm_mfma_w4_majors.hpp"

namespace moye {

int32_t gemm_mfma_w4_majors_f16(int32_t out_dt, GemmForm form, const GemmArgs& a, GemmPlan& plan) {
    return out_dt == MOYE_F32 ? launch_majors_of<W4F16L, OutF32>(form, a, plan) : launch_majors_of<W4F16L, OutF16>(form, a, plan);
}

}  // namespace moye
