// The hand-ordered kernel's guarded tiles with operands that keep their M- (N-) major form in blocks of 64 rows (AMAJ / BMAJ = 2 of
// gemm_mfma_w4_kernel.hpp), one operand type to a translation unit: gemm_mfma_w4_majors_f16.hip, ..._bf16.hip.
#pragma once

#include "gemm_mfma_w4_kernel.hpp"
#include "gemm_plan.hpp"

namespace moye {

template <typename In, typename Out, int RING, int BM, int BN, int WGN = 4>
static int32_t launch_majors_tiles(GemmArgs a, GemmPlan& plan) {
    typedef std::conditional_t<RING == 2, In, W4Deep<In, RING>> L;
    a.tiles_m = (a.M + BM - 1) / BM;
    a.tiles_n = (a.N + BN - 1) / BN;
    const bool am = a.flags & kGemmAMajorM, bm = a.flags & kGemmBMajorN;
    return am && bm ? launch256_w4<L, Out, WGN, false, true, BM, 2, 2, false, false, false, BN>(a, plan)
           : am     ? launch256_w4<L, Out, WGN, false, true, BM, 2, 0, false, false, false, BN>(a, plan)
                    : launch256_w4<L, Out, WGN, false, true, BM, 0, 2, false, false, false, BN>(a, plan);
}

// Any M, N and K of whole 16-byte pieces (M and N only where that operand is M- or N-major), K of 64 and more; the 256 x 256 tile
// (GemmForm::kOther) without C, the others with any epilogue; results in f32 or the operands' type.
template <typename In, typename Out>
static int32_t launch_majors_of(GemmForm form, const GemmArgs& a, GemmPlan& plan) {
    switch (form) {
        case GemmForm::kTile128x64: return launch_majors_tiles<In, Out, 5, 128, 64, 2>(a, plan);
        case GemmForm::kTile128x128: return launch_majors_tiles<In, Out, 4, 128, 128>(a, plan);
        case GemmForm::kTile128x192: return launch_majors_tiles<In, Out, 3, 128, 192>(a, plan);
        case GemmForm::kTile192x128: return launch_majors_tiles<In, Out, 3, 192, 128>(a, plan);
        case GemmForm::kTile128x256: return launch_majors_tiles<In, Out, 3, 128, 256>(a, plan);
        default: return launch_majors_tiles<In, Out, 2, 256, 256>(a, plan);
    }
}

}  // namespace moye
