// The hand-ordered kernel (gemm_mfma_w4_kernel.hpp) on tiles between 128 x 64 and 128 x 256, whole-line stages in rings of three
// to five, one workgroup per CU: problems of few tiles, where 128 x 128 and 256 x 256 ones in two stages leave CUs idle or
// every k-step waits for the loads of the step before (two stages: a k-step takes a load's latency, 0.85 us for 128 x 128 tiles
// with a CU each; in a ring of four 0.4-0.54).  What bounds them then is neither pipe alone.  Cycles of a k-step, of which the MFMAs /
// the LDS's reads, by counters, bf16, K = 4096 or 8192: 128 x 128 1100, 512 / 395; 128 x 192 1500, 768 / 480; 192 x 128 1320, 768 / 540; 128 x 256
// 2060, 1024 / 530; bank conflicts 1 % of them.  A wave waits for loads, reads or the barrier for 24 to 29 % of its time, and for its turn
// to issue, with the other wave of its SIMD in the matrix pipe, for 42 to 50 %.  The schedule and the clock both cost.  1000 x 6144 x 4096, call after
// call, operands cached: 1168 cycles of a k-step, 768 of them MFMAs, at 1.87 GHz, 45.0 us; all-zero operands take the same cycles (1181) at 2.38 GHz, 37.6 us; with
// a B that is not cached 1316 cycles at 1.93 GHz, 49.1 us, 148 cycles more for its lines out of memory.  2048 x 4096 x 4096 on 128 x 256 tiles 1412 cycles (1024)
// at 1.85 GHz, zeros 1430 at 2.36, not cached 1489 at 1.81; 1536 x 3072 x 4096 on 192 x 128, 192 workgroups, 1187 (768) at 2.32, 1434 at 2.28 not cached.
// The ring is what fits beside nothing else in 160 KiB; four stages where three would do made no difference (128 x 192
// 50.3 / 51.0 us at 1000 x 6144 x 4096).  Eight waves against four: 128 x 128 a twelfth faster where operands are cached,
// 128 x 256 a twentieth, 128 x 192 the same; 128 x 64 has room for four.  Always the guarded form (ragged tiles, any D, a K tail):
// a round of tiles or two, where its 3 % are less than a second set of instances is worth.  The barrier sits before the last
// column's reads of the next stage (BAR < A0).
// us before / now, operands not cached, bf16: 1000 x 6144 x 4096 69.9 / 49.9 (cached 49.5 / 43.0), 512 x 8192 x 8192 unsplit 109.9 / 72.6,
// 300 x 7168 x 4096 59.8 / 32.8, 742 x 10496 x 5888 110.8 / 89.6, 1080 x 4352 x 1664 31.9 / 22.3.
#include "gemm_mfma_w4_kernel.hpp"
#include "gemm_plan.hpp"

namespace moye {

template <typename In, typename Out, int RING, int WGN, int BM, int BN>
static int32_t launch_tiles(GemmArgs a, GemmPlan& plan) {
    a.tiles_m = (a.M + BM - 1) / BM;
    a.tiles_n = (a.N + BN - 1) / BN;
    return launch256_w4<W4Deep<In, RING>, Out, WGN, false, true, BM, 0, 0, false, false, false, BN>(a, plan);
}

template <typename In, typename Out>
static int32_t launch_tiles_of(GemmForm form, const GemmArgs& a, GemmPlan& plan) {
    switch (form) {
        case GemmForm::kTile128x64: return launch_tiles<In, Out, 5, 2, 128, 64>(a, plan);
        case GemmForm::kTile128x128: return launch_tiles<In, Out, 4, 4, 128, 128>(a, plan);
        case GemmForm::kTile128x192: return launch_tiles<In, Out, 3, 4, 128, 192>(a, plan);
        case GemmForm::kTile192x128: return launch_tiles<In, Out, 3, 4, 192, 128>(a, plan);
        default: return launch_tiles<In, Out, 3, 4, 128, 256>(a, plan);
    }
}

template <typename In>
static int32_t launch_tiles_out(GemmForm form, int32_t out_dt, const GemmArgs& a, GemmPlan& plan) {
    switch (out_dt) {
        case MOYE_F32: return launch_tiles_of<In, OutF32>(form, a, plan);
        case MOYE_F16: return launch_tiles_of<In, OutF16>(form, a, plan);
        case MOYE_BF16: return launch_tiles_of<In, OutBF16>(form, a, plan);
        default: return fail(MOYE_ERR_UNSUPPORTED, "gemm!: MFMA kernels write f32, f16 or bf16, not %s", dtype_name(out_dt));
    }
}

// Any M and N, K a multiple of 16 bytes, pointers and pitches of A and B 16-byte aligned, rows that fit 32-bit lane offsets, any
// D with its unit stride along N, any epilogue (the caller has checked).
int32_t gemm_mfma_w4_tiles_dispatch(int32_t in_dt, int32_t out_dt, GemmForm form, GemmArgs a, GemmPlan& plan) {
    a.flags |= kGemmRagged;
    switch (in_dt) {
        case MOYE_F16: return launch_tiles_out<W4F16L>(form, out_dt, a, plan);
        case MOYE_BF16: return launch_tiles_out<W4BF16L>(form, out_dt, a, plan);
        case MOYE_F8E4M3: return launch_tiles_out<W4FP8L>(form, out_dt, a, plan);
        default: return fail(MOYE_ERR_UNSUPPORTED, "gemm!: the hand-ordered kernel's smaller tiles take f16, bf16 or fp8 operands, not %s", dtype_name(in_dt));
    }
}

}  // namespace moye
