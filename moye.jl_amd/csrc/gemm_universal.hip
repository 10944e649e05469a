// gemm! with the UniversalFMA atom on the device, arithmetic identical to the reference's:
//   d = (a * b) + c          (src/arch/mma/mma.jl:64, via src/traits/mma.jl:49-68)
// with `a * b` rounded in promote_type(TA, TB), the sum rounded in the accumulator type, never
// contracted into an fma, and k running ascending so every C element is the strict
// left-to-right sum the reference's loop nest produces (src/algorithm/blas.jl:63-67,83-85 inside
// the k-tile loop of test/device/matmul.jl:40-49).  The m/n visiting order and the CTA tile
// cannot change any element, so results are bit-identical to the CPU restatement for every
// tiling.  Any strides, any sizes (edges are predicated).
//
// This file is compiled with -ffp-contract=off.
#include "kernels.hpp"

namespace moye {

// (a NaN stays as it is; everything else through v_cvt_pk_bf16_f32, round to nearest even)
__device__ __forceinline__ float u_bf16_round(float f) {
    if (f != f) return f;
    return __uint_as_float((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f) << 16);
}

__device__ __forceinline__ float u_load(const void* p, int64_t i, int dt) {
    switch (dt) {
        case MOYE_F32: return static_cast<const float*>(p)[i];
        case MOYE_F16: return (float)static_cast<const _Float16*>(p)[i];
        default: return __uint_as_float((uint32_t)static_cast<const uint16_t*>(p)[i] << 16);  // bf16
    }
}

__device__ __forceinline__ void u_store(void* p, int64_t i, int dt, float v) {
    switch (dt) {
        case MOYE_F32: static_cast<float*>(p)[i] = v; break;
        case MOYE_F16: static_cast<_Float16*>(p)[i] = (_Float16)v; break;
        default: static_cast<uint16_t*>(p)[i] = (uint16_t)(__float_as_uint(u_bf16_round(v)) >> 16); break;
    }
}

// kProd / kAcc: 0 = fp32, 1 = fp16, 2 = bf16 — the type the product / the running sum is rounded in
// (fp16: the value is made opaque first; a product the compiler can see is rounded by v_fma_mixlo_f16 with an addend of +0,
// which turns a product of -0 into +0)
template <int kT>
__device__ __forceinline__ float round_in(float x) {
    if constexpr (kT == 1) {
        asm("" : "+v"(x));
        return (float)(_Float16)x;
    } else if constexpr (kT == 2) return u_bf16_round(x);
    else return x;
}

template <int BM, int BN, int BK, int TM, int TN, int kProd, int kAcc>
__global__ __launch_bounds__(256) void gemm_universal_fma(UArgs p) {
    static_assert((BM / TM) * (BN / TN) == 256, "256 threads per workgroup");
    __shared__ float sA[BK][BM + 1];
    __shared__ float sB[BK][BN + 1];
    const int tid = threadIdx.x;
    const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
    constexpr int TX = BM / TM, TY = BN / TN;
    const int tx = tid % TX, ty = tid / TX;

    float acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int m = m0 + tx + TX * i, n = n0 + ty + TY * j;
            acc[i][j] = (p.C && p.alpha == 1.0f && m < p.M && n < p.N)
                            ? u_load(p.C, m * p.sc_m + n * p.sc_n, p.c_dt) : 0.0f;
        }

    const bool a_kfast = p.sa_k == 1, b_kfast = p.sb_k == 1;
    // Operand stages go global -> registers -> LDS, and the registers of stage t+1 are filled while stage t is
    // multiplied: a small problem (few workgroups per CU) would otherwise wait out one global round trip per stage.
    constexpr int LA = (BM * BK + 255) / 256, LB = (BN * BK + 255) / 256;
    float ra[LA], rb[LB];
    auto fetch = [&](int k0) {
        const int kmax = min(BK, p.K - k0);
#pragma unroll
        for (int q = 0; q < LA; ++q) {
            const int idx = tid + 256 * q;
            const int m = a_kfast ? idx / BK : idx % BM, k = a_kfast ? idx % BK : idx / BM;
            ra[q] = 0.0f;
            if (idx < BM * BK && m0 + m < p.M && k < kmax) ra[q] = u_load(p.A, (int64_t)(m0 + m) * p.sa_m + (int64_t)(k0 + k) * p.sa_k, p.a_dt);
        }
#pragma unroll
        for (int q = 0; q < LB; ++q) {
            const int idx = tid + 256 * q;
            const int n = b_kfast ? idx / BK : idx % BN, k = b_kfast ? idx % BK : idx / BN;
            rb[q] = 0.0f;
            if (idx < BN * BK && n0 + n < p.N && k < kmax) rb[q] = u_load(p.B, (int64_t)(n0 + n) * p.sb_n + (int64_t)(k0 + k) * p.sb_k, p.b_dt);
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int q = 0; q < LA; ++q) {
            const int idx = tid + 256 * q;
            const int m = a_kfast ? idx / BK : idx % BM, k = a_kfast ? idx % BK : idx / BM;
            if (idx < BM * BK) sA[k][m] = ra[q];
        }
#pragma unroll
        for (int q = 0; q < LB; ++q) {
            const int idx = tid + 256 * q;
            const int n = b_kfast ? idx / BK : idx % BN, k = b_kfast ? idx % BK : idx / BN;
            if (idx < BN * BK) sB[k][n] = rb[q];
        }
    };
    auto k_step = [&](int k) {
        float a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = sA[k][tx + TX * i];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = sB[k][ty + TY * j];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const float prod = round_in<kProd>(__fmul_rn(a[i], b[j]));
                acc[i][j] = round_in<kAcc>(__fadd_rn(prod, acc[i][j]));
            }
    };
    if (p.K > 0) {
        fetch(0);
        stash();
    }
    __syncthreads();
    for (int k0 = 0; k0 < p.K; k0 += BK) {
        const int kmax = min(BK, p.K - k0);
        const bool more = k0 + BK < p.K;
        if (more) fetch(k0 + BK);  // in flight during the arithmetic below
        if (kmax == BK) {   // a whole stage: unrolled, so that the LDS reads of later k are in flight under the arithmetic
#pragma unroll
            for (int k = 0; k < BK; ++k) k_step(k);
        } else {
            for (int k = 0; k < kmax; ++k) k_step(k);
        }
        __syncthreads();           // everybody is done reading this stage
        if (more) {
            stash();
            __syncthreads();
        }
    }

#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int m = m0 + tx + TX * i, n = n0 + ty + TY * j;
            if (m < p.M && n < p.N) {
                float v = acc[i][j];
                if (p.alpha != 1.0f) {
                    v = __fmul_rn(p.alpha, v);
                    if (p.C) v = __fadd_rn(v, u_load(p.C, m * p.sc_m + n * p.sc_n, p.c_dt));
                }
                u_store(p.D, m * p.sd_m + n * p.sd_n, p.d_dt, v);
            }
        }
}

// The form for few elements: tiles of 16 TM x 16 TN elements of D, TM x TN to a lane (rows 16 apart), so that a small problem
// has a workgroup for every CU, and KB k to a stage.  Operands lie in LDS with k contiguous, rows KB + 4 floats apart: a lane's 128-bit read
// brings four k, sixteen neighbouring lanes read sixteen rows in sixteen different groups of four banks, and the writes
// (lanes along m or along k, whichever is contiguous in memory) spread over the banks.  Bound by latency at these sizes: a
// launch, a memory round trip per stage (the next stage's is under way during the arithmetic), K dependent additions.
// Against 32 x 32 tiles that read LDS value by value and told the types apart per element, us: fp32 256^3 17.4 -> 6.2, 64 x 64
// x 768 44.9 -> 12.4, 512^3 35.0 -> 21.2, 768^3 63.7 -> 49.4, 1024^3 102 -> 80; fp16 256^3 25.5 -> 7.1, 768^3 111 -> 94.
// The arithmetic is the kernel's above, element by element.
// kAny: operands of different types, told apart at run time
enum { kAny = -1 };
template <int kDt> struct URaw { typedef float type; };
template <> struct URaw<MOYE_F16> { typedef _Float16 type; };
template <> struct URaw<MOYE_BF16> { typedef uint16_t type; };
template <int kDt>
__device__ __forceinline__ typename URaw<kDt>::type u_raw(const void* p, int64_t i, int dt) {
    if constexpr (kDt == kAny) return u_load(p, i, dt);
    else return static_cast<const typename URaw<kDt>::type*>(p)[i];
}
template <int kDt>
__device__ __forceinline__ float u_widen(typename URaw<kDt>::type v) {
    if constexpr (kDt == MOYE_BF16) return __uint_as_float((uint32_t)v << 16);
    else return (float)v;
}
template <int TM, int TN, int KB, int kProd, int kAcc, int DA, int DB>
__global__ __launch_bounds__(256) void gemm_universal_fma_small(UArgs p) {
    constexpr int BM = 16 * TM, BN = 16 * TN, PITCH = KB + 4;
    constexpr int DD = kAcc == 1 ? MOYE_F16 : kAcc == 2 ? MOYE_BF16 : MOYE_F32;  // C and D
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) float sA[BM * PITCH];
    __shared__ __align__(16) float sB[BN * PITCH];
    const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
    const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
    const bool a_kfast = p.sa_k == 1, b_kfast = p.sb_k == 1;
    constexpr int LA = BM * KB / 256, LB = BN * KB / 256;
    // element q of this lane in a stage: along k where that is the contiguous index, else along m (n)
    auto place = [&](bool kfast, int rows, int q, int* row, int* k) {
        const int idx = tid + 256 * q;
        *row = kfast ? idx / KB : idx % rows;
        *k = kfast ? idx % KB : idx / rows;
    };
    typename URaw<DA>::type ra[LA];
    typename URaw<DB>::type rb[LB];
    // (beyond M, N and K the last element is read again: what is computed from it is not stored or not added)
    auto fetch = [&](int k0) {
        const int klast = p.K - 1 - k0;
#pragma unroll
        for (int q = 0; q < LA; ++q) {
            int m, k;
            place(a_kfast, BM, q, &m, &k);
            ra[q] = u_raw<DA>(p.A, (int64_t)min(m0 + m, p.M - 1) * p.sa_m + (int64_t)(k0 + min(k, klast)) * p.sa_k, p.a_dt);
        }
#pragma unroll
        for (int q = 0; q < LB; ++q) {
            int n, k;
            place(b_kfast, BN, q, &n, &k);
            rb[q] = u_raw<DB>(p.B, (int64_t)min(n0 + n, p.N - 1) * p.sb_n + (int64_t)(k0 + min(k, klast)) * p.sb_k, p.b_dt);
        }
    };
    float acc[TM][TN];
    if (p.K > 0) fetch(0);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int m = m0 + tx + 16 * i, n = n0 + ty + 16 * j;
            acc[i][j] = (p.C && p.alpha == 1.0f && m < p.M && n < p.N) ? u_load(p.C, m * p.sc_m + n * p.sc_n, DD) : 0.0f;
        }
    auto fma = [&](const float (&a)[TM], const float (&b)[TN]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = round_in<kAcc>(__fadd_rn(round_in<kProd>(__fmul_rn(a[i], b[j])), acc[i][j]));
    };
    const float* const a0 = sA + tx * PITCH;
    const float* const b0 = sB + ty * PITCH;
    // G k-quads in one set of registers
    constexpr int G = TM * TN == 1 ? 4 : TM * TN <= 4 ? 2 : 1;
    struct Frag {
        f32x4 a[G][TM], b[G][TN];
    };
    auto read = [&](Frag& f, int k) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
#pragma unroll
            for (int i = 0; i < TM; ++i) f.a[g][i] = *reinterpret_cast<const f32x4*>(a0 + 16 * i * PITCH + k + 4 * g);
#pragma unroll
            for (int j = 0; j < TN; ++j) f.b[g][j] = *reinterpret_cast<const f32x4*>(b0 + 16 * j * PITCH + k + 4 * g);
        }
    };
    auto work = [&](const Frag& f) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float a[TM], b[TN];
#pragma unroll
                for (int i = 0; i < TM; ++i) a[i] = f.a[g][i][e];
#pragma unroll
                for (int j = 0; j < TN; ++j) b[j] = f.b[g][j][e];
                fma(a, b);
            }
    };
    for (int k0 = 0; k0 < p.K; k0 += KB) {
        if (k0) __syncthreads();  // everybody is done reading the stage before this one
#pragma unroll
        for (int q = 0; q < LA; ++q) {
            int m, k;
            place(a_kfast, BM, q, &m, &k);
            sA[m * PITCH + k] = u_widen<DA>(ra[q]);
        }
#pragma unroll
        for (int q = 0; q < LB; ++q) {
            int n, k;
            place(b_kfast, BN, q, &n, &k);
            sB[n * PITCH + k] = u_widen<DB>(rb[q]);
        }
        __syncthreads();
        if (k0 + KB < p.K) fetch(k0 + KB);  // in flight during the arithmetic below
        const int kmax = min(KB, p.K - k0), whole = kmax / (8 * G) * (8 * G);
        // two sets of fragments: one is read while the other is worked on
        Frag f0, f1;
        if (whole) read(f0, 0);
#pragma unroll 1
        for (int k = 0; k < whole; k += 8 * G) {
            read(f1, k + 4 * G);
            __builtin_amdgcn_sched_barrier(0);
            work(f0);
            if (k + 8 * G < whole) read(f0, k + 8 * G);
            __builtin_amdgcn_sched_barrier(0);
            work(f1);
        }
#pragma unroll 1
        for (int k = whole; k < kmax; ++k) {
            float a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = a0[16 * i * PITCH + k];
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = b0[16 * j * PITCH + k];
            fma(a, b);
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int m = m0 + tx + 16 * i, n = n0 + ty + 16 * j;
            if (m < p.M && n < p.N) {
                float v = acc[i][j];
                if (p.alpha != 1.0f) {
                    v = __fmul_rn(p.alpha, v);
                    if (p.C) v = __fadd_rn(v, u_load(p.C, m * p.sc_m + n * p.sc_n, DD));
                }
                u_store(p.D, m * p.sd_m + n * p.sd_n, DD, v);
            }
        }
}

template <int TM, int TN, int KB>
static int32_t launch_small(const UArgs& a, int prod, int accT, hipStream_t st) {
    const dim3 grid((a.M + 16 * TM - 1) / (16 * TM), (a.N + 16 * TN - 1) / (16 * TN));
#define MOYE_U(P, Q, T) gemm_universal_fma_small<TM, TN, KB, P, Q, T, T><<<grid, 256, 0, st>>>(a)
    if (prod == 0 && accT == 0 && a.a_dt == MOYE_F32 && a.b_dt == MOYE_F32) MOYE_U(0, 0, MOYE_F32);
    else if (prod == 0 && accT == 0) MOYE_U(0, 0, kAny);
    else if (prod == 1 && accT == 0) MOYE_U(1, 0, MOYE_F16);
    else if (prod == 2 && accT == 0) MOYE_U(2, 0, MOYE_BF16);
    else if (prod == 1 && accT == 1) MOYE_U(1, 1, MOYE_F16);
    else if (prod == 2 && accT == 2) MOYE_U(2, 2, MOYE_BF16);
    else return fail(MOYE_ERR_UNSUPPORTED, "gemm!: UniversalFMA has no kernel for this type combination");
#undef MOYE_U
    MOYE_HIP_CHECK(hipGetLastError());
    return MOYE_OK;
}

template <int BM, int BN, int BK, int TM, int TN>
static int32_t launch_u(const UArgs& a, int prod, int accT, hipStream_t st) {
    const dim3 grid((a.M + BM - 1) / BM, (a.N + BN - 1) / BN);
#define MOYE_U(P, Q) gemm_universal_fma<BM, BN, BK, TM, TN, P, Q><<<grid, 256, 0, st>>>(a)
    if (prod == 0 && accT == 0) MOYE_U(0, 0);
    else if (prod == 1 && accT == 0) MOYE_U(1, 0);
    else if (prod == 2 && accT == 0) MOYE_U(2, 0);
    else if (prod == 1 && accT == 1) MOYE_U(1, 1);
    else if (prod == 2 && accT == 2) MOYE_U(2, 2);
    else return fail(MOYE_ERR_UNSUPPORTED, "gemm!: UniversalFMA has no kernel for this type combination");
#undef MOYE_U
    MOYE_HIP_CHECK(hipGetLastError());
    return MOYE_OK;
}

static int type_class(int dt) { return dt == MOYE_F16 ? 1 : dt == MOYE_BF16 ? 2 : 0; }

// the type of the product, promote_type(TA, TB): the narrow one only when both operands have it
static int product_class(const UArgs& a) { return type_class(a.a_dt) == type_class(a.b_dt) ? type_class(a.a_dt) : 0; }

int32_t gemm_universal_choose(int bm, int bn, int bk, const UArgs& a, int cus, UniversalTile* tile) {
    for (int dt : {a.a_dt, a.b_dt, a.d_dt, a.C ? a.c_dt : MOYE_F32})
        if (dt != MOYE_F32 && dt != MOYE_F16 && dt != MOYE_BF16)
            return fail(MOYE_ERR_UNSUPPORTED, "gemm!: UniversalFMA kernels take f32, f16 or bf16, not %s", dtype_name(dt));
    // the running sum lives in the accumulator type TC == TD
    const int accT = type_class(a.d_dt);
    if (accT != 0 && accT != product_class(a))
        return fail(MOYE_ERR_UNSUPPORTED, "gemm!: a %s accumulator needs %s operands", dtype_name(a.d_dt), dtype_name(a.d_dt));
    if (a.C && a.c_dt != a.d_dt)
        return fail(MOYE_ERR_UNSUPPORTED, "gemm!: C and D must have the same element type");
    if (bm == 0 && bn == 0) {
        // measured, fp32: 1024^3 runs at 21.0 / 11.8 / 5.0 TFLOP/s on 32 / 64 / 128 tiles, 2048^3 at 28.0 / 36.5 / 20.3,
        // 4096^3 at 29.9 / 39.3 / 40.1 (every tile gives the same bits: k ascends strictly whatever the tile)
        const bool small = (int64_t)a.M * a.N <= 1024 * 1024;
        bm = bn = small ? 32 : 64;
    }
    if (bk == 0) bk = 8;
    // bK of the caller's tile is how many k the reference's kernel stages per trip, and bM x bN what a workgroup computes; the
    // sum over k is strictly ascending and no element depends on another whatever they are.  The 32 x 32 tile runs the form
    // for few elements, on tiles of its own: the smaller, the more workgroups, the larger, the fewer LDS reads per product.
    // fp32, us, 16 x 16 / 32 x 32 / 64 x 32: 256^3 6.2 / 11.9 / 18.0; 512^3 21.2 / 22.2 / 32.3; 640^3 39.2 / 32.1 / 40.1; 768^3
    // 58.2 / 49.4 / 56.9; 1024^3 128.8 / 93.3 / 79.8; 30000 x 30 x 300 39.8 / 28.8 / 25.3.  64 x 32 and 64 x 64 (the kernel above) only
    // where their tiles are full: two workgroups of 64 x 32 to a CU in one round, or seven eighths of more rounds (3000 x 1000
    // x 500 180 / 113 / 106, but 1040 x 1000 x 200 31.9 / 22.8 / 30.0 and 64 x 64 39.0; 1500^2 x 300 86 / 55 / 61 / 67; 2048^2 x 200
    // 113 / 65 / 67 / 53), and a side of at most 16 or 32 takes tiles no wider than that (16 x 100000 x 256 50 / 61 / 116 / 103;
    // 32 x 32768 x 256 33.8 / 24.0 / 38.5 / 49.5).  A launch holds 65535 tiles along N.
    if (bm == 32 && bn == 32 && bk == 8) {
        auto tiles = [&](int64_t tm, int64_t tn) { return ((a.M + tm - 1) / tm) * ((a.N + tn - 1) / tn); };
        const int64_t t32 = tiles(32, 32), rounds = (tiles(64, 32) + 2 * cus - 1) / (2 * cus);
        auto full = [&](int64_t elements) { return 8 * (int64_t)a.M * a.N >= 7 * elements; };
        if ((t32 <= cus || a.M <= 16 || a.N <= 16) && a.N <= 16 * 65535) *tile = UniversalTile::k16x16;
        else if (a.N > 32 * 65535 || (t32 > 12 * cus && full(tiles(64, 64) * 64 * 64))) *tile = UniversalTile::k64x64;
        else if (t32 > 3 * cus && (rounds == 1 || full(rounds * 2 * cus * 64 * 32))) *tile = UniversalTile::k64x32;
        else *tile = UniversalTile::k32x32;
        return MOYE_OK;
    }
    if (bm == 64 && bn == 64 && bk == 8) *tile = UniversalTile::k64x64;
    else if (bm == 128 && bn == 128 && bk == 8) *tile = UniversalTile::k128x128;
    else return fail(MOYE_ERR_UNSUPPORTED, "gemm!: UniversalFMA CTA tile %dx%dx%d not built (32x32x8, 64x64x8, 128x128x8)", bm, bn, bk);
    return MOYE_OK;
}

const char* gemm_universal_name(UniversalTile tile) {
    switch (tile) {
        case UniversalTile::k16x16: return "gemm_universal_fma_small<16,16,64>";
        case UniversalTile::k32x32: return "gemm_universal_fma_small<32,32,32>";
        case UniversalTile::k64x32: return "gemm_universal_fma_small<64,32,64>";
        case UniversalTile::k64x64: return "gemm_universal_fma<64,64,8>";
        default: return "gemm_universal_fma<128,128,8>";
    }
}

int32_t gemm_universal_dispatch(UniversalTile tile, const UArgs& a, hipStream_t st) {
    const int prod = product_class(a), accT = type_class(a.d_dt);
    switch (tile) {
        case UniversalTile::k16x16: return launch_small<1, 1, 64>(a, prod, accT, st);
        case UniversalTile::k32x32: return launch_small<2, 2, 32>(a, prod, accT, st);
        case UniversalTile::k64x32: return launch_small<4, 2, 64>(a, prod, accT, st);
        case UniversalTile::k64x64: return launch_u<64, 64, 8, 4, 4>(a, prod, accT, st);
        default: return launch_u<128, 128, 8, 8, 8>(a, prod, accT, st);
    }
}

}  // namespace moye
