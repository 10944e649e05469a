// copyto! between arrays whose unit strides lie on different modes -- transposes, batches of them, with or without a
// conversion of the element type (src/algorithm/copy.jl:4-12,38-46 with the layouts of a transpose).
//
// src(i, j) at i + j * lds (i is the source's contiguous index), dst(i, j) at i * ldd + j; further modes count matrices.
// Any extents, pitches and element-aligned pointers: one launch, no strips.
#include <algorithm>

#include "copy_convert.hpp"
#include "copy_transpose.hpp"

namespace moye {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// one 128-bit access of an array that is only aligned to its elements (the part takes such accesses at any byte)
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));

// 4 x 4 bytes: o[e] holds byte e of r0, r1, r2, r3
__device__ __forceinline__ void transpose_bytes(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3, uint32_t (&o)[4]) {
    const uint32_t t0 = __builtin_amdgcn_perm(r1, r0, 0x05010400u), t1 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
    const uint32_t t2 = __builtin_amdgcn_perm(r3, r2, 0x05010400u), t3 = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
    o[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
    o[1] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
    o[2] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
    o[3] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
}

// element e (a constant) of a 16-byte piece, widened to fp32
template <int kSrc>
__device__ __forceinline__ float element_f32(const u32x4& v, int e) {
    if constexpr (kSrc == MOYE_F32) return __uint_as_float(v[e]);
    else if constexpr (kSrc == MOYE_F16) return (float)__builtin_bit_cast(_Float16, (uint16_t)(v[e / 2] >> (16 * (e % 2))));
    else if constexpr (kSrc == MOYE_BF16) return __uint_as_float(e % 2 ? v[e / 2] & 0xffff0000u : v[e / 2] << 16);
    else return f8e4m3_to_f32((uint8_t)(v[e / 4] >> (8 * (e % 4))));
}
// four bytes of results, rounded as store_from rounds them
template <int kDst, int N>
__device__ __forceinline__ uint32_t pack_f32(const float (&x)[N]) {
    if constexpr (kDst == MOYE_F32) {
        return __float_as_uint(x[0]);
    } else if constexpr (kDst == MOYE_F16) {
        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, f16x2{(_Float16)x[0], (_Float16)x[1]});
    } else if constexpr (kDst == MOYE_BF16) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)x[0], (__bf16)x[1]});
    } else {
        // (the instruction gives every NaN the same sign: only where a lane holds one are the bytes made one by one)
        const bool nan = __builtin_isunordered(x[0], x[1]) | __builtin_isunordered(x[2], x[3]);
        if (__builtin_expect(nan, 0))
            return f32_to_f8e4m3(x[0]) | ((uint32_t)f32_to_f8e4m3(x[1]) << 8) | ((uint32_t)f32_to_f8e4m3(x[2]) << 16) | ((uint32_t)f32_to_f8e4m3(x[3]) << 24);
        return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(x[2], x[3], __builtin_amdgcn_cvt_pk_fp8_f32(x[0], x[1], 0, false), true);
    }
}

// A block of Q rows (j) of 16 bytes (ES elements along i) -> ES pieces of 16 bytes, piece e holding element e of every row,
// converted.
template <int kSrc, int kDst, int SB, int DB>
__device__ __forceinline__ void turn_block(const u32x4 (&v)[16 / DB], u32x4 (&o)[16 / SB]) {
    constexpr int ES = 16 / SB, Q = 16 / DB;
    if constexpr (kSrc == kDst && SB == 1) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                uint32_t t[4];
                transpose_bytes(v[4 * g][c], v[4 * g + 1][c], v[4 * g + 2][c], v[4 * g + 3][c], t);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[4 * c + e][g] = t[e];
            }
    } else if constexpr (kSrc == kDst && SB == 2) {
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                o[2 * c][p] = __builtin_amdgcn_perm(v[2 * p + 1][c], v[2 * p][c], 0x05040100u);
                o[2 * c + 1][p] = __builtin_amdgcn_perm(v[2 * p + 1][c], v[2 * p][c], 0x07060302u);
            }
    } else if constexpr (kSrc == kDst && SB == 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = u32x4{v[0][e], v[1][e], v[2][e], v[3][e]};
    } else if constexpr (kSrc == kDst && SB == 8) {
#pragma unroll
        for (int e = 0; e < 2; ++e) o[e] = u32x4{v[0][2 * e], v[0][2 * e + 1], v[1][2 * e], v[1][2 * e + 1]};
    } else if constexpr (kSrc == MOYE_F64 || kDst == MOYE_F64) {
#pragma unroll
        for (int e = 0; e < ES; ++e) {
            char w[16];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                char x[SB];
                __builtin_memcpy(x, reinterpret_cast<const char*>(&v[q]) + e * SB, SB);
                store_from<kDst>(w + q * DB, load_as_f64<kSrc>(x), kSrc == MOYE_F64);
            }
            __builtin_memcpy(&o[e], w, 16);
        }
    } else {
#pragma unroll
        for (int e = 0; e < ES; ++e)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                float x[4 / DB];
#pragma unroll
                for (int k = 0; k < 4 / DB; ++k) x[k] = element_f32<kSrc>(v[w * (4 / DB) + k], e);
                o[e][w] = pack_f32<kDst>(x);
            }
    }
}

// A workgroup of T lanes moves a tile of TI (i) x TJ (j) elements.  A lane loads NB blocks of Q rows x 16 bytes, PI lanes
// side by side along a source row, turns each block in registers, so that what goes into LDS are whole 16-byte pieces of
// destination rows, and the lanes then read LDS rows back side by side and store 16 bytes each.  LDS: rows of JC 16-byte
// pieces, the piece's index XORed with bits of the row so that eight neighbouring lanes always touch eight different
// bank groups, on the way in (eight rows ES apart, one piece each) and out (eight pieces of one row).
//
// Edges: a lane whose 16 bytes would reach beyond a source row's end reads the row's last 16 bytes instead (some
// elements then come twice and are written to LDS twice, the same values); rows beyond nj are read from the last row and
// not stored; the piece that crosses the end of a destination row goes out element by element.
//
// Bound by memory, and by lines that two workgroups share where a pitch is no multiple of 128 bytes.  Against the kernels
// this one replaced (whole 64 x 64 patches; strips and unaligned pitches element by element), us before -> now:
// f32 16384^2 343 -> 341 (6.30 TB/s), 8192^2 121 -> 97, 16400 x 16392 421 -> 405, 10001 x 7003 1111 -> 134;
// f16 16384^2 192 -> 187, 6000 x 4096 24.1 -> 19.3, 10001 x 7003 1042 -> 75; [4,2000,32,128] -> [4,32,128,2000] 937 -> 28.4;
// NCHW -> NHWC 32 x 256 x 28 x 28 234 -> 7.5; bytes 16384^2 121 -> 103; 8-byte elements 8192^2 188 -> 180;
// f32 -> bf16 5000 x 3000 32.1 -> 21.3, 8192^2 80.8 -> 72.2.
template <int kSrc, int kDst, int SB, int DB, int PI, int NB, int T>
__global__ __launch_bounds__(T) void transpose_blocks(TransposeArgs a) {
    constexpr int ES = 16 / SB, Q = 16 / DB, NJ = T / PI, TI = PI * ES, JC = NJ * NB, TJ = JC * Q;
    const int sw = a.linear ? 0 : JC < 8 ? JC - 1 : 7;
    static_assert(T % JC == 0 && TI % (T / JC) == 0, "whole rows per pass");
    extern __shared__ u32x4 tile[];  // ES rows that are never read (see below), then TI rows, of JC pieces
    const char* src = a.src;
    char* dst = a.dst;
    {
        uint32_t rest = blockIdx.y + blockIdx.z * gridDim.y;
        if (rest >= a.batch) return;
#pragma unroll 1
        for (int m = 0; m < a.modes; ++m) {
            const uint32_t q = rest / a.extent[m], r = rest - q * a.extent[m];
            src += (int64_t)r * a.s_stride[m] * SB;
            dst += (int64_t)r * a.d_stride[m] * DB;
            rest = q;
        }
    }
    uint32_t bid = blockIdx.x;
    if (a.run > 1) {  // workgroup ids go to the XCDs in turn: `run` neighbouring tiles to each
        const uint32_t per = (uint32_t)(a.xcds * a.run), g = bid / per, r = bid - g * per;
        if ((g + 1) * per <= gridDim.x) bid = g * per + (r % (uint32_t)a.xcds) * (uint32_t)a.run + r / (uint32_t)a.xcds;
    }
    int ti, tj;
    if (a.band == 0) {
        tj = bid % (uint32_t)a.tiles_j;
        ti = bid / (uint32_t)a.tiles_j;
    } else {  // bands of `band` tile columns (j), the source's contiguous index fastest inside a band
        const uint32_t per = (uint32_t)a.band * (uint32_t)a.tiles_i, b = bid / per, r = bid - b * per;
        const uint32_t w = min((uint32_t)a.band, (uint32_t)a.tiles_j - b * (uint32_t)a.band);
        const uint32_t blk = r / ((uint32_t)a.band * w), q = r - blk * (uint32_t)a.band * w;
        const uint32_t h = min((uint32_t)a.band, (uint32_t)a.tiles_i - blk * (uint32_t)a.band);
        ti = (int)(blk * (uint32_t)a.band + q % h);
        tj = (int)(b * (uint32_t)a.band + q / h);
    }
    const int pi = threadIdx.x % PI, jr = threadIdx.x / PI;
    constexpr int RPP = T / JC;
    const int jc = threadIdx.x % JC, r0 = threadIdx.x / JC;
    const int iw = a.ni - ti * TI, jw = a.nj - tj * TJ;  // what is left of the two extents here
    // LDS rows are counted from ES on: a lane that was shifted back may write rows that belong to the tile before this one
    auto slot = [&](int row, int piece) -> u32x4& { return tile[row * JC + (piece ^ ((row / ES) & sw))]; };
    auto put = [&](int row0, const u32x4 (&v)[NB][Q]) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            u32x4 o[ES];
            turn_block<kSrc, kDst, SB, DB>(v[b], o);
#pragma unroll
            for (int e = 0; e < ES; ++e) slot(row0 + e, jr + NJ * b) = o[e];
        }
    };
    char* const d = dst + ((int64_t)(ti * TI + r0) * a.ldd + tj * TJ + Q * jc) * DB;
    if (iw >= TI && jw >= TJ) {
        const char* const s = src + ((int64_t)(tj * TJ + Q * jr) * a.lds + ti * TI + pi * ES) * SB;
        u32x4 v[NB][Q];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int q = 0; q < Q; ++q)
                v[b][q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(s + (int64_t)(Q * NJ * b + q) * a.lds * SB));
        put(ES + pi * ES, v);
        __syncthreads();
#pragma unroll
        for (int p = 0; p < TI / RPP; ++p)
            __builtin_nontemporal_store(slot(ES + r0 + RPP * p, jc), reinterpret_cast<u32x4_any*>(d + (int64_t)(RPP * p) * a.ldd * DB));
        return;
    }
    if (pi * ES < iw) {
        const int il = min(pi * ES, iw - ES);  // (below 0 where fewer than ES columns are left)
        const char* const s = src + ((int64_t)tj * TJ * a.lds + ti * TI + il) * SB;
        u32x4 v[NB][Q];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int j = min(Q * (jr + NJ * b) + q, jw - 1);
                v[b][q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(s + (int64_t)j * a.lds * SB));
            }
        put(ES + il, v);
    }
    __syncthreads();
    const int left = jw - Q * jc;
    if (left >= Q) {
#pragma unroll
        for (int p = 0; p < TI / RPP; ++p)
            if (r0 + RPP * p < iw)
                __builtin_nontemporal_store(slot(ES + r0 + RPP * p, jc), reinterpret_cast<u32x4_any*>(d + (int64_t)(RPP * p) * a.ldd * DB));
    } else if (left > 0) {
#pragma unroll 1
        for (int p = 0; r0 + RPP * p < min(iw, TI); ++p) {
            const u32x4 w = slot(ES + r0 + RPP * p, jc);
            char* const dr = d + (int64_t)(RPP * p) * a.ldd * DB;
#pragma unroll
            for (int q = 0; q < Q - 1; ++q)
                if (q < left) __builtin_memcpy(dr + q * DB, reinterpret_cast<const char*>(&w) + q * DB, DB);
        }
    }
}

template <int kSrc, int kDst, int SB, int DB, int PI, int NB, int T>
static int32_t launch_blocks(TransposeArgs a, int lds_request, hipStream_t st) {
    constexpr int ES = 16 / SB, Q = 16 / DB, NJ = T / PI, TI = PI * ES, TJ = NJ * NB * Q, kLds = (TI + ES) * TJ * DB;
    constexpr int kCap = 160 * 1024;  // all of a CU's LDS
    static_assert(kLds <= kCap, "the tile fits");
    auto kern = transpose_blocks<kSrc, kDst, SB, DB, PI, NB, T>;
    const int lds = std::max(kLds, lds_request);
    if (lds > 48 * 1024) {
        static LdsCap cap;
        if (int32_t e = raise_lds_cap(cap, reinterpret_cast<const void*>(kern), kCap)) return e;
    }
    a.tiles_i = (a.ni + TI - 1) / TI;
    a.tiles_j = (a.nj + TJ - 1) / TJ;
    const int64_t tiles = (int64_t)a.tiles_i * a.tiles_j;
    if (tiles >= ((int64_t)1 << 32) / T) return fail(MOYE_ERR_SHAPE, "copyto!: too many tiles for one launch (2^32 lanes)");
    const unsigned gy = std::min<unsigned>(a.batch, 32768u), gz = (a.batch + gy - 1) / gy;
    kern<<<dim3((unsigned)tiles, gy, gz), T, lds, st>>>(a);
    MOYE_HIP_CHECK(hipGetLastError());
    return MOYE_OK;
}

// Which tile.  Few elements: small tiles, so that there are workgroups for every CU (f16 1024^2: 3.6 us on 64 x 128, 4.3 on
// 64 x 256).  Rows that are whole 128-byte lines: tiles of 128-byte source runs, 512-byte destination runs (f16 8192^2 50.6
// us, 55.7 on 128 x 512; f32 8192^2 96.6, 108 on 64 x 256).  Anything else, and arrays far beyond the caches: the longest
// runs, whose ends are the smallest part of them (f16 10001 x 7003 77 us, 86 on 64 x 256).
template <int kSrc, int kDst, int SB, int DB>
static int32_t launch_shape(TransposeArgs a, hipStream_t st) {
    const int64_t n = (int64_t)a.ni * a.nj * a.batch, bytes = n * std::max(SB, DB);
    const bool lines = (a.lds * SB) % 128 == 0 && (a.ldd * DB) % 128 == 0;
    const bool few = n <= (2 << 20), huge = bytes >= ((int64_t)256 << 20);
    if constexpr (SB == 2 && DB == 2) {
        if (few) return launch_blocks<kSrc, kDst, 2, 2, 8, 1, 128>(a, 0, st);
        if (n <= (8 << 20)) return launch_blocks<kSrc, kDst, 2, 2, 16, 1, 256>(a, 0, st);
        if (lines && !huge) return launch_blocks<kSrc, kDst, 2, 2, 8, 1, 256>(a, 0, st);
        return launch_blocks<kSrc, kDst, 2, 2, 16, 2, 512>(a, 0, st);
    } else if constexpr (SB == 4 && DB == 4) {
        // (one workgroup per CU, for which the LDS request sees, where the array is far beyond the caches: 16384^2 341 us
        // against 344; and the tiles in plain order then: 341 against 357)
        const bool far = bytes >= ((int64_t)600 << 20);
        if (far && lines && a.band == 0) a.run = 1;
        if (far || (!lines && bytes >= ((int64_t)32 << 20))) return launch_blocks<kSrc, kDst, 4, 4, 16, 2, 512>(a, 96 * 1024, st);
        if (few || lines) return launch_blocks<kSrc, kDst, 4, 4, 8, 1, 256>(a, 0, st);
        return launch_blocks<kSrc, kDst, 4, 4, 16, 2, 256>(a, 0, st);
    } else if constexpr (SB == 1 && DB == 1) {
        if (n <= (6 << 20)) return launch_blocks<kSrc, kDst, 1, 1, 4, 1, 64>(a, 0, st);
        if (n <= (64 << 20)) return launch_blocks<kSrc, kDst, 1, 1, 16, 1, 256>(a, 0, st);
        return launch_blocks<kSrc, kDst, 1, 1, 8, 1, 256>(a, 0, st);
    } else if constexpr (SB == 8 && DB == 8) {
        if (bytes < ((int64_t)24 << 20)) return launch_blocks<kSrc, kDst, 8, 8, 16, 4, 256>(a, 0, st);
        return launch_blocks<kSrc, kDst, 8, 8, 32, 4, 512>(a, 96 * 1024, st);
    } else if constexpr (SB == 4 && DB == 2) {
        if (few) return launch_blocks<kSrc, kDst, 4, 2, 8, 1, 128>(a, 0, st);
        if (lines) return launch_blocks<kSrc, kDst, 4, 2, 16, 1, 512>(a, 0, st);
        return launch_blocks<kSrc, kDst, 4, 2, 16, 2, 512>(a, 0, st);
    } else if constexpr (SB == 2 && DB == 4) {
        if (few) return launch_blocks<kSrc, kDst, 2, 4, 8, 1, 128>(a, 0, st);
        if (lines && !huge) return launch_blocks<kSrc, kDst, 2, 4, 8, 1, 256>(a, 0, st);
        return launch_blocks<kSrc, kDst, 2, 4, 16, 2, 512>(a, 0, st);
    } else if constexpr (SB == 4 && DB == 1) {
        if (few) return launch_blocks<kSrc, kDst, 4, 1, 8, 1, 128>(a, 0, st);
        if (n <= (8 << 20)) return launch_blocks<kSrc, kDst, 4, 1, 16, 1, 256>(a, 0, st);
        return launch_blocks<kSrc, kDst, 4, 1, 16, 1, 512>(a, 0, st);
    } else if constexpr (SB == 2 && DB == 1) {
        if (n <= (8 << 20)) return launch_blocks<kSrc, kDst, 2, 1, 8, 1, 128>(a, 0, st);
        return launch_blocks<kSrc, kDst, 2, 1, 16, 1, 256>(a, 0, st);
    } else if constexpr (SB == 1) {  // runs of 64 or 128 bytes in, 512 or 1024 out
        return launch_blocks<kSrc, kDst, 1, DB, DB == 8 ? 4 : 8, 1, 256>(a, 0, st);
    } else if constexpr (SB == 8) {
        return launch_blocks<kSrc, kDst, 8, DB, 16, DB == 4 ? 2 : 1, 256>(a, 0, st);
    } else {
        static_assert(DB == 8, "every pair of sizes");
        return launch_blocks<kSrc, kDst, SB, 8, SB == 4 ? 16 : 8, SB == 4 ? 4 : 2, 256>(a, 0, st);
    }
}

template <int kSrc, int SB>
static int32_t launch_converting(int32_t dd, const TransposeArgs& a, hipStream_t st) {
    switch (dd) {
        case MOYE_F32: if constexpr (kSrc != MOYE_F32) return launch_shape<kSrc, MOYE_F32, SB, 4>(a, st); break;
        case MOYE_F16: if constexpr (kSrc != MOYE_F16) return launch_shape<kSrc, MOYE_F16, SB, 2>(a, st); break;
        case MOYE_BF16: if constexpr (kSrc != MOYE_BF16) return launch_shape<kSrc, MOYE_BF16, SB, 2>(a, st); break;
        case MOYE_F8E4M3: if constexpr (kSrc != MOYE_F8E4M3) return launch_shape<kSrc, MOYE_F8E4M3, SB, 1>(a, st); break;
        case MOYE_F64: if constexpr (kSrc != MOYE_F64) return launch_shape<kSrc, MOYE_F64, SB, 8>(a, st); break;
        default: break;
    }
    return fail(MOYE_ERR_UNSUPPORTED, "copyto!: no conversion between these element types");
}

bool transpose_plan(const moye_tensor& src, const moye_tensor& dst, bool same_bits, TransposeArgs* a) {
    const int sb = dtype_bytes(src.dtype), db = dtype_bytes(dst.dtype), r = src.rank;
    if (r != dst.rank || r < 2 || sb > 8 || db > 8 || (!same_bits && !(is_float_dtype(src.dtype) && is_float_dtype(dst.dtype)))) return false;
    int mi = -1, mj = -1;
    for (int m = 0; m < r; ++m) {
        if (src.shape[m] != dst.shape[m]) return false;
        if (src.shape[m] > 1 && src.stride[m] == 1 && mi < 0) mi = m;
        if (dst.shape[m] > 1 && dst.stride[m] == 1 && mj < 0) mj = m;
    }
    if (mi < 0 || mj < 0 || mi == mj) return false;
    *a = TransposeArgs{};
    const int64_t ni = src.shape[mi], nj = src.shape[mj];
    a->src = static_cast<const char*>(src.ptr);
    a->dst = static_cast<char*>(dst.ptr);
    a->lds = src.stride[mj];
    a->ldd = dst.stride[mi];
    // (fewer than 32 along either side leave most of a tile's lanes without work: element by element costs no more there)
    if (ni < 32 || nj < 32 || ni >= ((int64_t)1 << 31) || nj >= ((int64_t)1 << 31) || a->ldd < nj) return false;
    a->ni = (int32_t)ni;
    a->nj = (int32_t)nj;
    int64_t batch = 1;
    for (int m = 0; m < r; ++m) {
        if (m == mi || m == mj || src.shape[m] == 1) continue;
        if (src.shape[m] >= ((int64_t)1 << 31)) return false;
        a->extent[a->modes] = (uint32_t)src.shape[m];
        a->s_stride[a->modes] = src.stride[m];
        a->d_stride[a->modes] = dst.stride[m];
        ++a->modes;
        batch *= src.shape[m];
        if (batch >= ((int64_t)1 << 31)) return false;
    }
    a->batch = (uint32_t)batch;
    return true;
}

// Which order.  Destination rows first where the source's contiguous extent is at least the destination's: writes are the
// side that needs locality on this part (16384^2 f32: 341 us, 353 source rows first), else bands of 64 tile columns with
// the source's index fastest (4096 x 32768 f32 192 us, 202 the other way).  Four neighbouring tiles to an XCD, so that
// lines two of them share meet in one L2 (f32 8192^2 102.8 -> 96.6 us, 16400 x 16392 ~420 -> 405).
int32_t transpose_run(int32_t src_dt, int32_t dst_dt, bool same_bits, bool linear_lds, int xcds, TransposeArgs a, hipStream_t st) {
    a.band = a.ni >= a.nj || a.batch > 1 ? 0 : 64;
    a.xcds = xcds;
    a.run = 4;
    a.linear = linear_lds;
    if (same_bits) {
        switch (dtype_bytes(src_dt)) {
            case 1: return launch_shape<MOYE_U8, MOYE_U8, 1, 1>(a, st);
            case 2: return launch_shape<MOYE_U16, MOYE_U16, 2, 2>(a, st);
            case 4: return launch_shape<MOYE_U32, MOYE_U32, 4, 4>(a, st);
            default: return launch_shape<MOYE_U64, MOYE_U64, 8, 8>(a, st);
        }
    }
    switch (src_dt) {
        case MOYE_F32: return launch_converting<MOYE_F32, 4>(dst_dt, a, st);
        case MOYE_F16: return launch_converting<MOYE_F16, 2>(dst_dt, a, st);
        case MOYE_BF16: return launch_converting<MOYE_BF16, 2>(dst_dt, a, st);
        case MOYE_F8E4M3: return launch_converting<MOYE_F8E4M3, 1>(dst_dt, a, st);
        default: return launch_converting<MOYE_F64, 8>(dst_dt, a, st);
    }
}

}  // namespace moye
