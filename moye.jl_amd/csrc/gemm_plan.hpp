// Host-side choice of CTA tile and K ranges for a gemm! whose tile is left to the library and that does not fill the chip
// with 256 x 256 tiles: a small cost model instead of thresholds.  Its per-k-tile times are fitted to bf16 timings on one
// MI355X with a different B on every call (operands that stay in the 256 MiB memory-side cache between calls run the
// kernels with one workgroup per CU up to 1.4 times faster, which real callers with several weight matrices do not see);
// the number of compute units that share the work is an argument (DeviceShape::cus).
//
//   time = 3 us + k-tiles per workgroup x t(tile, workgroups resident on a CU) [x rounds] + second pass of a K split
//
// with k-tiles of 128 bytes of K and, per k-tile and workgroup,
//   128 x 128 tiles (gemm_mfma128.hip, two workgroups fit a CU):   0.85 us alone on its CU, 1.08 us with a neighbour
//   64 x 64 tiles (gemm_mfma.hip, four fit):                       0.48 / 0.73 / 0.86 / 1.00 us for 1 / 2 / 3 / 4 on a CU
// (512 x 8192 x 8192 on 256 workgroups of 128 x 128: 111.8 us, in two K ranges on 512: 89.4; 1024 x 4096 x 14336 on 256:
// 198.5; 2048 x 4096 x 4096 on 512: 72.3; 2048^3 on 1024 workgroups of 64 x 64: 33.0; 512 x 4096 x 4096 on 512: 49.8), and a
// second pass that moves the fp32 partial products at about 6 TB/s (they are still in the caches) after 3 us of launch.
// Ragged tiles cost the 128 x 128 kernel 15 % more; the 64 x 64 kernel has no ragged form.  fp32 operands have their own
// per-k-tile times.  Problems of at most one round of 256 x 256 tiles, and the rests of larger ones, are also priced on the forms
// of gemm_form_choose, whose formula and prices are their own.
#pragma once

#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace moye {

// Kernel forms that one price formula covers (gemm_form_us below); kOther: the forms and launches that the rest of this file
// and the dispatcher price.
enum class GemmForm { kOther, kBlock32x32, kBlock64x32, kBlock64x64, kTile128x64, kTile128x128, kTile128x192, kTile192x128, kTile128x256 };

struct TileChoice {
    int tile;   // 64, 128 or 256; 0 where `form` says what runs
    int split;  // K ranges
    double us;
    GemmForm form = GemmForm::kOther;
};

inline double gemm_plan_cost(int tile, int split, int64_t M, int64_t N, int64_t k_bytes, bool f32_in, int cus) {
    const int64_t tiles = ((M + tile - 1) / tile) * ((N + tile - 1) / tile), ctas = tiles * split;
    const int slots = tile == 128 ? 2 : 4;
    // per k-tile and workgroup with 1 .. slots workgroups resident on a CU.  fp32 operands run on v_mfma_f32_16x16x4_f32,
    // an eighth of the 16-bit rate per byte of K, and are bound by it (2048^3 on 256 workgroups of 128 x 128: 124.5 us;
    // 4096 x 2048 x 4096 on 512: 465 us; 2560^3 on 400: 291 us; 3072^3 on 576: 522 us; 1024^3 on 256 workgroups of
    // 64 x 64: 25.7 us; 2048^3 on 1024: 156 us; 3072^3 on 2304: 509 us)
    static const double t128_16[3] = {0, 0.85, 1.08}, t64_16[5] = {0, 0.48, 0.73, 0.86, 1.00};
    static const double t128_32[3] = {0, 1.92, 3.62}, t64_32[5] = {0, 0.71, 1.25, 1.80, 2.40};
    const double* t = tile == 128 ? (f32_in ? t128_32 : t128_16) : (f32_in ? t64_32 : t64_16);
    const double ktiles = (double)((k_bytes / split + 127) / 128);
    // whole rounds of cus x slots workgroups, then the rest with fewer neighbours
    const int64_t full = ctas / ((int64_t)cus * slots), rest = ctas % ((int64_t)cus * slots);
    double us = 3.0 + ktiles * ((double)full * t[slots] + (rest ? t[(rest + cus - 1) / cus] : 0.0));
    if (tile == 128 && (M % 128 || N % 128 || k_bytes % 128)) us *= 1.15;
    if (split > 1) us += 3.0 + (2.0 * split * 4.0 + 4.0) * (double)M * (double)N / 6.0e6;
    return us;
}

// `max_split` = 1 forbids K ranges (no workspace); `fixed_split` > 0 asks for the best tile for that many ranges (the
// dispatch after the split has been made: k_bytes is then the whole K again, so both calls price the same candidates).
inline TileChoice gemm_plan(int64_t M, int64_t N, int64_t k_bytes, bool f32_in, bool tile64_ok, int max_split, int cus,
                            int fixed_split = 0) {
    TileChoice best{128, fixed_split > 0 ? fixed_split : 1, 1e30};
    for (int tile : {128, 64}) {
        if (tile == 64 && !tile64_ok) continue;
        // (one row of tiles: the 64 x 64 kernel has nothing to share B with, and the model does not know
        // -- bf16 64 x 65536 x 2048: 51.9 us against 43.3 on 128 x 128 tiles; 64 x 32768 x 2048: 26.7 against 27.4)
        if (tile == 64 && M <= 64) continue;
        for (int s = 1; s <= 16; s *= 2) {
            if (fixed_split > 0 && s != fixed_split) continue;
            if (fixed_split <= 0 && s > 1) {
                // equal ranges of whole k-tiles, at least four of them
                if (s > max_split || k_bytes % s || (k_bytes / s) % 128 || k_bytes / s < 512) continue;
            }
            const double us = gemm_plan_cost(tile, s, M, N, k_bytes, f32_in, cus);
            if (us < best.us) best = TileChoice{tile, s, us};
        }
    }
    return best;
}

// The same problem on 256 x 256 tiles, one workgroup per CU: 9 us + per k-tile 1.44 us in a round that fills the chip,
// 1.30 us in one that fills half of it or less, linear in between (bf16, B not cached: 512 x 8192 x 8192 on 64 tiles 176 us,
// in two K ranges 109.1, in four 79.4; with B cached 0.98 us per k-tile up to half the chip: fp16 K = 4096, 144 tiles 73 us,
// 128 72); a quarter more for the guarded instance (130 x 32768 x 4096 on 128 ragged tiles: 99 us).  `split` K ranges:
// that many times the workgroups with a share of K each, and the second pass.
inline double gemm_plan_cost_256(int64_t M, int64_t N, int64_t k_bytes, bool f32_in, bool ragged, int cus, int split = 1) {
    const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256) * split, full = tiles / cus, rest = tiles % cus;
    const int half = cus / 2 > 0 ? cus / 2 : 1;
    const double ktiles = (double)((k_bytes / split + 127) / 128);
    // (fp32: 7.05 us per k-tile however many CUs are busy: the matrix pipe alone sets the pace; 4096^3 909 us,
    // 3072^3 on 144 tiles 687 us, 4096 x 2048 x 4096 on 128 tiles 913 us)
    const double t_full = f32_in ? 7.05 : 1.44;
    const double t_rest = rest == 0 ? 0.0 : f32_in ? 7.05 : rest <= half ? 1.30 : 1.30 + (double)(rest - half) / (double)half * 0.14;
    double us = 9.0 + 6.0 * (double)(full + (rest ? 1 : 0) - 1) + ktiles * ((double)full * t_full + t_rest);
    if (ragged) us *= 1.25;
    if (split > 1) us += 3.0 + (2.0 * split * 4.0 + 4.0) * (double)M * (double)N / 6.0e6;  // the second pass, as in gemm_plan_cost
    return us;
}

// The forms above against each other and against one launch of 256 x 256 tiles or of 128 x 128 ones two to a CU:
//
//   time = start + more x (rounds - 1) + k-tiles of a wave x (each x rounds + filled x rounds, the last one counted as far as it is full)
//
// fitted, per operand size, to 500 bf16, 300 fp8 and 150 fp32 problems of 65 to 4096 rows, 96 to 14336 columns and K from 64 to
// 8192, as the geometric mean of operands that are cached and operands that are not (the formula misses a time by 9 %, and
// what it picks takes 1.02 times what the best form takes).  A round is `slots` workgroups on every CU.  The short-M kernel's
// blocks (gemm_mfma_skinny.hip) divide K among the four waves of a workgroup and need no barrier: few elements.  The tiles of
// gemm_mfma_w4_tiles.hip have a CU's LDS to themselves and three to five stages in flight: few tiles, one round of them where one
// of the sizes comes out even.  Of nine sizes timed, these five and the three blocks leave 1 % to all nine.
struct FormPrice {
    GemmForm form;
    int tm, tn, slots, waves_k;
    double start, more, each, filled;
};
inline constexpr FormPrice kFormPrices16[] = {
    {GemmForm::kOther, 256, 256, 1, 1, 7.6, 8.4, 1.09, 0.385},       {GemmForm::kOther, 128, 128, 2, 1, 4.73, 3.13, 0.544, 0.502},
    {GemmForm::kBlock32x32, 32, 32, 2, 4, 3.40, 0.75, 0.19, 0.64},   {GemmForm::kBlock64x32, 64, 32, 1, 4, 3.63, 1.63, 0.47, 0.23},
    {GemmForm::kBlock64x64, 64, 64, 1, 4, 4.24, 2.73, 0.77, 0.12},
    {GemmForm::kTile128x64, 128, 64, 1, 1, 4.30, 2.91, 0.277, 0.063}, {GemmForm::kTile128x128, 128, 128, 1, 1, 4.33, 2.93, 0.385, 0.152},
    {GemmForm::kTile128x192, 128, 192, 1, 1, 5.61, 4.91, 0.464, 0.235}, {GemmForm::kTile192x128, 192, 128, 1, 1, 5.11, 4.30, 0.511, 0.168},
    {GemmForm::kTile128x256, 128, 256, 1, 1, 6.03, 4.83, 0.585, 0.269}};
inline double gemm_form_us(const FormPrice& f, int64_t M, int64_t N, int64_t k_bytes, int cus) {
    const int64_t wgs = ((M + f.tm - 1) / f.tm) * ((N + f.tn - 1) / f.tn), per = (int64_t)cus * f.slots, full = wgs / per, rest = wgs % per;
    const int64_t lines = (k_bytes + 127) / 128, kt = (lines + f.waves_k - 1) / f.waves_k;
    const double rounds = (double)(full + (rest ? 1 : 0));
    return f.start + f.more * (rounds - 1) + (double)kt * (f.each * rounds + f.filled * ((double)full + (double)rest / (double)per));
}
// `part`: what is left of a larger problem, for which the blocks are not looked at (a round of tiles wide or long, it has too many
// elements for them).  The cheapest form of the table, or kOther where one of the other two, or what `limit_us` stands for, is no dearer.
inline GemmForm gemm_form_choose(int64_t M, int64_t N, int64_t k_bytes, int elem_bytes, int cus, double limit_us, double* us, bool part = false) {
    static const FormPrice bits8[] = {
        {GemmForm::kOther, 256, 256, 1, 1, 7.7, 6.5, 1.04, 0.5},         {GemmForm::kOther, 128, 128, 2, 1, 4.76, 2.76, 0.514, 0.619},
        {GemmForm::kBlock32x32, 32, 32, 2, 4, 3.32, 0.79, 0.23, 0.67},   {GemmForm::kBlock64x32, 64, 32, 1, 4, 3.49, 1.61, 0.51, 0.38},
        {GemmForm::kBlock64x64, 64, 64, 1, 4, 3.96, 2.39, 0.99, 0.28},
        {GemmForm::kTile128x64, 128, 64, 1, 1, 4.07, 2.49, 0.29, 0.07},   {GemmForm::kTile128x128, 128, 128, 1, 1, 4.42, 2.78, 0.364, 0.188},
        {GemmForm::kTile128x192, 128, 192, 1, 1, 5.31, 4.70, 0.443, 0.375}, {GemmForm::kTile192x128, 192, 128, 1, 1, 4.93, 4.32, 0.469, 0.271},
        {GemmForm::kTile128x256, 128, 256, 1, 1, 5.59, 5.04, 0.581, 0.427}};
    // (fp32: the other forms' prices are those of gemm_plan_cost and gemm_plan_cost_256, which were fitted apart from these: the
    // blocks have to be a fifth cheaper)
    static const FormPrice bits32[] = {
        {GemmForm::kBlock32x32, 32, 32, 2, 4, 3.34, 1.60, 0.556, 0.766}, {GemmForm::kBlock64x32, 64, 32, 1, 4, 3.78, 2.46, 1.155, 0.119},
        {GemmForm::kBlock64x64, 64, 64, 1, 4, 5.31, 3.19, 2.09, 0.13}};
    GemmForm best = GemmForm::kOther;
    *us = elem_bytes == 4 ? 0.8 * limit_us : limit_us;
    // (more 256 x 256 tiles than CUs: the dispatcher may give the last round a launch of its own, which is not priced here; bf16
    // 2624 x 8896 x 3072 145 us so and 170 on 128 x 256 tiles; where one of these forms was cheaper it was by 5 %)
    if (((M + 255) / 256) * ((N + 255) / 256) > cus) return best;
    auto look = [&](const FormPrice* f, size_t n) {
        for (size_t i = 0; i < n; ++i) {
            if (part && f[i].waves_k > 1) continue;
            const double t = gemm_form_us(f[i], M, N, k_bytes, cus);
            if (t < *us) { *us = t; best = f[i].form; }
        }
    };
    if (elem_bytes == 2) look(kFormPrices16, sizeof kFormPrices16 / sizeof *kFormPrices16);
    else if (elem_bytes == 1) look(bits8, sizeof bits8 / sizeof *bits8);
    else look(bits32, sizeof bits32 / sizeof *bits32);
    return best;
}

// 16-bit operands that are not K-major on tiles that read them as they lie, in one launch: the cheapest of the tiles in deep rings and of
// 256 x 256 ones (guarded or whole, `two_stages`: 128 x 128 ones in two stages too, which take whole tiles only; `tile256`: 256 x 256 ones
// where there are no more of them than CUs).  Prices of K-major operands, which the transposing reads miss by little: bf16, operands not
// cached, us K-major / B N-major / A M-major / both: 2048 x 4096 x 4096 on 128 x 256 tiles 57.5 / 59.4 / 60.0 / 62.4, 1000 x 6144 x 4096 on
// 128 x 192 49.6 / 53.2 / 55.5 / 54.8, 1536 x 3072 x 4096 on 192 x 128 45.7 / 45.2 / - / 45.7.
inline const FormPrice* gemm_majors_form(int64_t M, int64_t N, int64_t k_bytes, int cus, bool tile256, bool two_stages, double* us) {
    const FormPrice* best = nullptr;
    *us = 1e30;
    for (const FormPrice& f : kFormPrices16) {
        if (f.waves_k > 1) continue;
        if (f.form == GemmForm::kOther && (f.tm == 256 ? !tile256 || ((M + 255) / 256) * ((N + 255) / 256) > cus : !two_stages)) continue;
        // (whole tiles in two stages run unguarded: they keep what is a tenth dearer)
        const double t = (f.form == GemmForm::kOther && f.tm == 128 ? 0.9 : 1.0) * gemm_form_us(f, M, N, k_bytes, cus);
        if (t < *us) { *us = t; best = &f; }
    }
    return best;
}
// Are K-major copies (`copied` elements of operands in all, one launch for each operand) and the cheapest K-major form the better plan?  The
// blocks, which divide K among four waves, have no form that reads operands otherwise: few elements and a long K (bf16 500 x 1000 x 1992, A
// M-major, 14.8 us so).  Beyond that copies are 5 us and twice the operands' bytes: 264 x 1024 x 1088 with B N-major 10.5 with a copy and blocks,
// 9.0 as it lies, 1000 x 6144 x 4096 69.2 / 53.2, both operands 76.8 / 54.8; 1088 x 1024 x 264 both 15.8 / 7.5.  `ragged_rows`: the other
// operand is K-major with a pitch of no whole lines, which costs the tiles 2 us more than the blocks (A M-major, 1000 x 520 x 1984 / 1992 15.5 /
// 17.3; 1992 with B N-major 18.2 with a copy, 19.2 as it lies).  Few tiles and long problems with a short K follow the prices like any other: both
// operands, copies / as they lie, 200 x 136 x 504 11.2 / 8.0, 408 x 96 x 1280 12.7 / 11.7, 28000 x 1208 x 520 81.9 / 66.0, 208 x 37432 x 960 63.9 / 32.4;
// of 66 such problems the one that prices send the slower way as it lies is 16848 x 3280 x 152 with A M-major, 57.4 / 59.5, and of fewer than 8 tiles of
// 128 x 128 with one operand to copy and a K under 500 they copy where that takes 0.3 to 2 us more (136 x 160 x 144 6.7 / 4.8).
inline bool gemm_majors_copies_pay(int64_t M, int64_t N, int64_t k_bytes, int64_t copied, int launches, bool ragged_rows, int cus) {
    double native, kmajor;
    gemm_majors_form(M, N, k_bytes, cus, true, false, &native);
    gemm_form_choose(M, N, k_bytes, 2, cus, 1e30, &kmajor);
    if (ragged_rows) native += 2.0;
    return kmajor + 2.5 * launches + 4.0 * (double)copied / 5.0e6 < native;
}

// Everything left to the library (tile, waves, K ranges): the cheapest of 64 x 64 / 128 x 128 tiles with 1 .. max_split K
// ranges and of unsplit 256 x 256 tiles, which are considered from a quarter of the CUs' worth of tiles on.  The one
// place where tile and K ranges are chosen together: the workspace sizing and the dispatcher both take their answer
// from here.  `transposed`: the kernels run N x M (a column-major D), and the forms, some with two different sides, are priced for
// that.  bf16, B not cached, us as M x N / as N x M: 1000 x 6144 x 4096 80 on 288 tiles of 128 x 192 / 52-59 on 256 of 192 x 128, 2048 x
// 3072 x 4096 79.5 / 52.5, 639 x 9216 x 1152 36.5 / 29.5 (with a row-major D 54, 52 and 29.5).
inline TileChoice gemm_choose(int64_t M, int64_t N, int64_t k_bytes, int elem_bytes, int max_split, int cus, bool forms, bool transposed) {
    const bool f32_in = elem_bytes == 4;
    TileChoice best = gemm_plan(M, N, k_bytes, f32_in, M % 64 == 0 && N % 64 == 0 && k_bytes % 128 == 0, max_split, cus);
    const bool ragged = M % 256 || N % 256 || k_bytes % 128;
    if (((M + 255) / 256) * ((N + 255) / 256) >= cus / 4) {
        const double us = gemm_plan_cost_256(M, N, k_bytes, f32_in, ragged, cus);
        if (us <= best.us) best = TileChoice{256, 1, us};
    }
    // few whole 256 x 256 tiles and a long K: K ranges that bring the workgroups up to one per CU at most (bf16, a B that is
    // not cached: 512 x 8192 x 8192 on 128 x 128 tiles 111.8 us, in two ranges 89.4, on 256 x 256 tiles in four ranges
    // 79.4; 1024 x 4096 x 14336 198.5 / 145.2 / 113.5)
    if (!ragged && !f32_in) {
        const int64_t tiles = (M / 256) * (N / 256);
        for (int s = 2; s <= max_split && tiles * s <= cus; s *= 2) {
            if (k_bytes % s || (k_bytes / s) % 128 || k_bytes / s < 512) continue;
            const double us = gemm_plan_cost_256(M, N, k_bytes, f32_in, false, cus, s);
            if (us < best.us) best = TileChoice{256, s, us};
        }
    }
    if (forms) {
        double us;
        const GemmForm form = gemm_form_choose(transposed ? N : M, transposed ? M : N, k_bytes, elem_bytes, cus, best.us, &us);
        if (form != GemmForm::kOther) best = TileChoice{0, 1, us, form};
    }
    return best;
}

// A short A (at most 64 rows, K in 16-byte pieces) goes to the kernel that streams B once and reads all of A per workgroup
// (gemm_mfma_skinny.hip) -- except more than 16 rows with many columns: that kernel then brings A out of the L2s as
// often as B out of memory and has one stage in flight per wave, which holds it near 5 TB/s of B, and 128 x 128 tiles,
// part empty as they are, take less once there are more of them than CUs (the hand-ordered instance with two workgroups
// on a CU) or, with a very short K, from three quarters of the CUs on.  bf16, us with a different B on every call (so
// that the memory-side cache does not serve it), that kernel / tiles: 64 x 65536 x 2048 63.8 / 47.1; 32 x 65536 x 2048
// 59.8 / 46.3; 64 x 36864 x 2048 44.9 / 40.0; 64 x 65536 x 4096 107.9 / 92.8; 64 x 65536 x 8192 201.3 / 181.5;
// 24 x 65536 x 1024 37.4 / 25.7; 64 x 262144 x 2048 265.0 / 209.7; 64 x 32768 x 1024 22.7 / 21.5; 64 x 24576 x 512
// 16.3 / 12.6.  But 64 x 32768 x 2048 32.7 / 36.7; 64 x 28672 x 8192 95.7 / 134.8; 48 x 49152 x 8192 132.8 / 149.3;
// 16 x 65536 x 2048 42.4 / 46 and 64 x 16384 x 2048 17.6 / 34.3.
// (fp32 operands stay on that kernel: their MFMA is slow enough for the empty part of a tile to cost more than it saves,
// 32 x 65536 x 1024 73.2 us against 138.5 on tiles, 64 x 65536 x 2048 165.2 against 252.3.)
inline bool gemm_short_m(int64_t M, int64_t N, int64_t k_bytes, bool f32_in, int cus) {
    if (M > 64 || k_bytes % 16) return false;
    if (M <= 16 || f32_in) return true;
    const int64_t tiles = (N + 127) / 128;
    if (tiles > cus) return !(k_bytes <= 8192 || (M > 48 && tiles >= 2 * (int64_t)cus));
    return !(4 * tiles >= 3 * (int64_t)cus && k_bytes <= 2048);
}

// The short-M kernel's workgroups take 8 to 64 rows of B, in eights, and all of A, one workgroup on a CU at a time (its rings
// fill the LDS), and a workgroup streams its rows at about 64 GB/s whatever the others do (56 with 48 and 64 rows of B,
// measured with long K).  A launch therefore takes as many rounds as its workgroups -- times the K ranges of a split -- need
// on the CUs: bf16, us with 32 / 48 / 64 rows: 64 x 12288 x 8192 59.0 / 39.2 / 44.1; 64 x 14336 x 4096 33.0 / 37.9 / 24.9;
// 64 x 8192 x 8192 30.9 / 34.0 / 41.3; 32 x 10240 x 8192 42.6 / 30.6 / 35.2; 32 x 20480 x 8192 66.2 / 59.5 / 69.5;
// 24 x 28672 x 4096 45.0 / 45.6 / 38.6; 16 x 14336 x 4096 20.5 / 27.2 / 19.3; 16 x 24576 x 4096 31.1 / 32.7 / 34.0.  But
// 64 x 4096 x 14336 42.0 unsplit on 256 workgroups of 16 rows, 47.0 in two K ranges on 512.  In microseconds:
// 4.5 (two launches of a split: 7.5, and never under 10.7) + the longer of all bytes at 6 TB/s and rounds x a workgroup's
// bytes at its rate.
inline double gemm_short_m_us(int64_t M, int64_t N, int64_t k_bytes, int cus, int rows, int split) {
    const int mt = (int)((M + 15) / 16);
    const int64_t wgs = (N + rows - 1) / rows * split, rounds = (wgs + cus - 1) / cus;
    const double wg_us = (double)(rows + 16 * mt) * ((double)k_bytes / split) / (rows > 32 ? 56.0e3 : 64.0e3);
    const double floor_us = (double)(N + M) * (double)k_bytes / 6.0e6;
    const double t = floor_us > (double)rounds * wg_us ? floor_us : (double)rounds * wg_us;
    if (split > 1) return 7.5 + t > 10.7 ? 7.5 + t : 10.7;
    return 4.5 + t;
}
// Rows of B per workgroup for a launch in `split` K ranges: the fewest rows of A and B that a CU reads in all its
// rounds, more rows at once on a tie.  (A is read in groups of eight rows.  Up to 16 rows of A two workgroups of 32 rows of B
// share a CU, which is worth 15 % from a second round on: 5 x 14336 x 8192 36.4 us against 38.5 with 64 rows; from a fifth
// on 22 %: 16 x 40960 x 4096 49.7 / 52.9, fp8 15 x 34304 x 4096 24.6 against 26.4 with 48.)  Whole MFMA blocks of 16 rows, or one of
// them half empty, its last eight rows neither read nor stored, where that leaves a CU 6 % less to read: bf16, not cached, us whole /
// half: 50 x 14336 x 4096 23.5 (64 rows) / 22.7 (56), 16 x 6144 x 8192 19.3 (32) / 17.2 (24), 40 x 10240 x 8192 32.6 (48) / 30.2 (40), 50 x 2048 x 4096
// 11.8 (16) / 10.5 (8), 16 x 20480 x 4096 29.1 / 27.7, 64 x 28672 x 8192 92.8 / 88.3.  Not with a few rows of A and long rows, which run at
// the memory's rate as they are (1 x 6144 x 16384 30.6 / 33.7, 1 x 5120 x 16384 28.2 / 28.9; but 1 x 5000 x 12288 22.1 / 20.1), nor
// 40 and 56 rows with rows under 2 KiB, where they win as often as they lose (40 x 14336 x 256 5.4 / 5.6, x 512 6.9 / 6.6, x 768 7.8 / 7.8; from 2 KiB
// on 40 x 9600 x 1536 9.6 / 9.3, 24 x 20480 x 2048 18.5 / 17.7, 24 x 14336 x 2040 19.5 / 19.1), or up to 4 KiB where two workgroups of 32 share a CU
// (12 x 19456 x 1536 12.7 / 13.5, x 2048 15.3 / 15.8, x 2056 24.9 / 24.3, x 2304 17.1 / 17.2, x 2560 20.1 / 19.2), nor 56 rows in several rounds beside more than 32 rows of A where rows are 4 KiB, more
// than 40 where they are 8 KiB: their lines at one k lie in few memory channels (N = 28672, M = 40 / 56 / 64: K = 2048 24.2 / 24.9, 26.4 / 27.6, 27.2 / 28.4,
// K = 4096 41.2 / 41.0, 44.9 / 45.8, 46.7 / 47.8; but K = 1536 21.3 / 20.8, 23.5 / 23.3, 24.2 / 24.2, 3072 35.7 / 34.8, 39.1 / 39.1, 40.5 / 40.5, 6144 64.1 / 63.6,
// 71.7 / 71.2, 75.0 / 73.8, 8192 76.1 / 75.9, 86.1 / 82.8, 90.5 / 84.6).  Eight rows in unsplit launches only.  `us` is the price with whole blocks, which the model was fitted to: on it K ranges are decided (16 x 2048 x 16384
// 22.2 unsplit with 16 rows, 19.9 with 8, 17.1 in two ranges).
inline int gemm_short_m_rows(int64_t M, int64_t N, int64_t k_bytes, int cus, int split, double* us = nullptr) {
    // (the host's time for a call of a few microseconds counts: no division where one round holds the workgroups)
    const int m8 = (int)((M + 7) / 8 * 8);
    auto rounds_of = [&](int r) {
        const int64_t wgs = (int64_t)(((uint32_t)N + (uint32_t)r - 1) / (uint32_t)r) * split;
        return wgs <= cus ? 1 : (wgs + cus - 1) / cus;
    };
    auto cost = [&](int r, int64_t rounds) { return (double)(rounds * (r + m8)) * (r > 32 || M > 16 || rounds == 1 ? 1.0 : rounds < 5 ? 0.85 : 0.78); };
    int best = 16;
    double least = cost(16, rounds_of(16));
    for (int r : {32, 48, 64}) {
        const double c = cost(r, rounds_of(r));
        if (c <= least) { best = r; least = c; }
    }
    if (us) *us = gemm_short_m_us(M, N, k_bytes, cus, best, split);
    least *= 0.94;
    const int whole = best;
    for (int r : {8, 24, 40, 56}) {
        if (r == 8 ? split > 1 : M <= 8 && k_bytes >= 28 * 1024) continue;
        const int64_t rounds = rounds_of(r);
        if (r >= 40 && (k_bytes < 2048 || (whole == 32 && k_bytes <= 4096))) continue;
        if (r == 56 && rounds > 1 && ((M > 32 && k_bytes == 4096) || (M > 40 && k_bytes == 8192))) continue;
        const double c = cost(r, rounds);
        if (c <= least) { best = r; least = c; }
    }
    return best;
}

// The hardware deals consecutive workgroups to the XCDs in turn.  Which of `n` tiles workgroup `bid` takes, so that each XCD gets one
// run of neighbouring tiles, the first n % xcds of them a tile more than the others.
constexpr int tile_in_xcd_runs(int bid, int n, int xcds) {
    const int xcd = bid % xcds, rest = n % xcds;
    return xcd * (n / xcds) + (xcd < rest ? xcd : rest) + bid / xcds;
}

}  // namespace moye
