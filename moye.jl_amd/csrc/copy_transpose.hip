// copyto! between arrays whose unit strides lie on different modes -- transposes, batches of them, with or without a
// conversion of the element type (src/algorithm/copy.jl:4-12,38-46 with the layouts of a transpose).
//
// src(i, j) at i + j * lds (i is the source's contiguous index), dst(i, j) at i * ldd + j; further modes count matrices.
// Any extents, pitches and element-aligned pointers: one launch, no strips.
#include <algorithm>
#include <initializer_list>

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
// four bytes of results, rounded as store_from rounds them; kFinite: none is a NaN
template <int kDst, bool kFinite = false, int N>
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
        // (the instruction gives every NaN the same sign)
        if constexpr (!kFinite)
            return f32_to_f8e4m3(x[0]) | ((uint32_t)f32_to_f8e4m3(x[1]) << 8) | ((uint32_t)f32_to_f8e4m3(x[2]) << 16) | ((uint32_t)f32_to_f8e4m3(x[3]) << 24);
        return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(x[2], x[3], __builtin_amdgcn_cvt_pk_fp8_f32(x[0], x[1], 0, false), true);
    }
}

// The first `left` elements of a piece, fewer than all: 8, 4, 2 and 1 bytes as they are needed (with one store per element bytes
// 1000 x 300 took 8.1 us, with these 6.8)
template <int DB>
__device__ __forceinline__ void store_first(char* p, u32x4 w, int left) {
    const int bytes = left * DB;
    if (bytes & 8) {
        __builtin_memcpy(p, &w, 8);
        p += 8;
        w[0] = w[2];
        w[1] = w[3];
    }
    if constexpr (DB <= 4) {
        if (bytes & 4) {
            __builtin_memcpy(p, &w, 4);
            p += 4;
            w[0] = w[1];
        }
    }
    if constexpr (DB <= 2) {
        if (bytes & 2) {
            __builtin_memcpy(p, &w, 2);
            p += 2;
            w[0] >>= 16;
        }
    }
    if constexpr (DB == 1) {
        if (bytes & 1) *p = (char)w[0];
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
        if constexpr (kDst == MOYE_F8E4M3) {  // (one test for a lane's block, not one for every four bytes of it)
            bool nan = false;
#pragma unroll
            for (int e = 0; e < ES; ++e)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    float x[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) x[k] = element_f32<kSrc>(v[4 * w + k], e);
                    nan |= __builtin_isunordered(x[0], x[1]) | __builtin_isunordered(x[2], x[3]);
                    o[e][w] = pack_f32<kDst, true>(x);
                }
            if (__builtin_expect(!nan, 1)) return;
        }
        if constexpr (kSrc == MOYE_F8E4M3) {
            // Two elements to an instruction (a lane's 128 conversions one by one were most of a small call: fp8 -> bf16 1024^2
            // 5.9 -> 3.6 us).  It makes every NaN negative: only a block with a positive one, 0x7f, goes the way below.
            uint32_t found = 0;
#pragma unroll
            for (int q = 0; q < Q; ++q)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const uint32_t t = v[q][c] ^ 0x7f7f7f7fu;
                    found |= (t - 0x01010101u) & ~t;  // bit 7 of the lowest byte that is zero
                }
            if (__builtin_expect((found & 0x80808080u) == 0, 1)) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        float x[4][4 / DB];
#pragma unroll
                        for (int k = 0; k < 4 / DB; ++k) {
                            const int row = w * (4 / DB) + k;
                            const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)v[row][c], false), hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)v[row][c], true);
                            x[0][k] = lo[0]; x[1][k] = lo[1]; x[2][k] = hi[0]; x[3][k] = hi[1];
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[4 * c + e][w] = pack_f32<kDst>(x[e]);
                    }
                return;
            }
        }
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
// not stored; the piece that crosses the end of a destination row goes out in halves.
//
// Bound by memory, and by lines that two workgroups share where a pitch is no multiple of 128 bytes.  Against the kernels
// this one replaced (whole 64 x 64 patches; strips and unaligned pitches element by element), us before -> now:
// f32 16384^2 343 -> 341 (6.30 TB/s), 8192^2 121 -> 97, 16400 x 16392 421 -> 405, 10001 x 7003 1111 -> 134;
// f16 16384^2 192 -> 187, 6000 x 4096 24.1 -> 19.3, 10001 x 7003 1042 -> 75; [4,2000,32,128] -> [4,32,128,2000] 937 -> 28.4;
// NCHW -> NHWC 32 x 256 x 28 x 28 234 -> 7.5; bytes 16384^2 121 -> 103; 8-byte elements 8192^2 188 -> 180;
// f32 -> bf16 5000 x 3000 32.1 -> 21.3, 8192^2 80.8 -> 72.2.
// kSkew: destination rows whose pitch is no whole lines: a workgroup's part of a row starts and ends on the row's own 128-byte
// boundaries, up to 127 bytes behind those of the tile, so that no line but a row's first and last is written by two
// workgroups, and every store is aligned.  1: pitches and addresses of whole pieces, 2: any.  It reads eight pieces' worth of source rows more, which its neighbour reads as well (skew_of: where, and what it measured).
// kKeep: bit 0: the source is read, bit 1: the destination is written through the caches in the ordinary way instead of with the
// non-temporal hint (launch_shape decides).
template <int kSrc, int kDst, int SB, int DB, int PI, int NB, int T, int kKeep, int kSkew>
__global__ __launch_bounds__(T) void transpose_blocks(TransposeArgs a) {
    constexpr int ES = 16 / SB, Q = 16 / DB, NJ = T / PI, TI = PI * ES, JC = NJ * NB, TJ = JC * Q;
    constexpr int JX = kSkew ? 8 : 0, JL = JC + JX;  // pieces of an LDS row
    static_assert(!kSkew || (NJ >= JX && JC % 8 == 0), "the pieces more come from one more block of the first lanes, and are swizzled among themselves");
    const int sw = a.linear ? 0 : JC < 8 ? JC - 1 : 7;
    static_assert(T % JC == 0 && TI % (T / JC) == 0, "whole rows per pass");
    extern __shared__ u32x4 tile[];  // ES rows that are never read (see below), then TI rows, of JL pieces
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
    auto slot = [&](int row, int piece) -> u32x4& { return tile[row * JL + (piece ^ ((row / ES) & sw))]; };
    auto load = [](const char* p) -> u32x4 {
        if constexpr (kKeep & 1) return *reinterpret_cast<const u32x4_any*>(p);
        else return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(p));
    };
    auto store = [](const u32x4& w, char* p) {
        if constexpr (kKeep & 2) *reinterpret_cast<u32x4_any*>(p) = w;
        else __builtin_nontemporal_store(w, reinterpret_cast<u32x4_any*>(p));
    };
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
    auto put1 = [&](int row0, const u32x4 (&v)[Q]) {  // the block behind the tile's (kSkew)
        u32x4 o[ES];
        turn_block<kSrc, kDst, SB, DB>(v, o);
#pragma unroll
        for (int e = 0; e < ES; ++e) slot(row0 + e, JC + jr) = o[e];
    };
    // bytes from the tile's start in row p of this lane's pass to the row's next whole line (the lanes of a wave share a row)
    static_assert(!kSkew || JC % 64 == 0, "a wave has one row");
    auto shift = [&](int p) { return kSkew ? __builtin_amdgcn_readfirstlane((int)(-reinterpret_cast<uintptr_t>(d + (int64_t)(RPP * p) * a.ldd * DB - 16 * jc) & 127)) : 0; };
    // 16 bytes of an LDS row that start `by` bytes behind this lane's piece
    auto bytes_from = [&](int row, int by) -> u32x4 {
        const u32x4 lo = slot(row, jc + by / 16);
        const int sh = by % 16;
        if (kSkew == 1 || sh == 0) return lo;
        const u32x4 hi = slot(row, jc + by / 16 + 1);
        auto five = [&](uint32_t x0, uint32_t x1, uint32_t x2, uint32_t x3, uint32_t x4) {
            return u32x4{__builtin_amdgcn_alignbyte(x1, x0, sh & 3), __builtin_amdgcn_alignbyte(x2, x1, sh & 3), __builtin_amdgcn_alignbyte(x3, x2, sh & 3),
                         __builtin_amdgcn_alignbyte(x4, x3, sh & 3)};
        };
        switch (sh >> 2) {
            case 0: return five(lo[0], lo[1], lo[2], lo[3], hi[0]);
            case 1: return five(lo[1], lo[2], lo[3], hi[0], hi[1]);
            case 2: return five(lo[2], lo[3], hi[0], hi[1], hi[2]);
            default: return five(lo[3], hi[0], hi[1], hi[2], hi[3]);
        }
    };
    // what lies before the first whole line of a row, in its first tile
    auto row_start = [&](int row, char* to, int sh) {
        const int left = min(sh / DB, jw) - Q * jc;
        if (left >= Q) store(slot(row, jc), to);
        else if (left > 0) store_first<DB>(to, slot(row, jc), left);
    };
    if (iw >= TI && jw >= TJ + JX * Q) {
        const char* const s = src + ((int64_t)(tj * TJ + Q * jr) * a.lds + ti * TI + pi * ES) * SB;
        u32x4 v[NB][Q];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int q = 0; q < Q; ++q)
                v[b][q] = load(s + (int64_t)(Q * NJ * b + q) * a.lds * SB);
        if constexpr (kSkew) {
            if (jr < JX) {
                u32x4 x[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) x[q] = load(s + (int64_t)(TJ + q) * a.lds * SB);
                put1(ES + pi * ES, x);
            }
        }
        put(ES + pi * ES, v);
        __syncthreads();
#pragma unroll
        for (int p = 0; p < TI / RPP; ++p) {
            const int sh = shift(p);
            char* const to = d + (int64_t)(RPP * p) * a.ldd * DB;
            if constexpr (kSkew) {
                store(bytes_from(ES + r0 + RPP * p, sh), to + sh);
                if (tj == 0) row_start(ES + r0 + RPP * p, to, sh);
            } else {
                store(slot(ES + r0 + RPP * p, jc), to);
            }
        }
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
                v[b][q] = load(s + (int64_t)j * a.lds * SB);
            }
        put(ES + il, v);
        if constexpr (kSkew) {
            if (jr < JX) {
                u32x4 x[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) x[q] = load(s + (int64_t)min(Q * (JC + jr) + q, jw - 1) * a.lds * SB);
                put1(ES + il, x);
            }
        }
    }
    __syncthreads();
    if constexpr (kSkew) {
#pragma unroll 1
        for (int p = 0; r0 + RPP * p < min(iw, TI); ++p) {
            const int sh = shift(p), row = ES + r0 + RPP * p;
            char* const to = d + (int64_t)(RPP * p) * a.ldd * DB;
            const int left = jw - Q * jc - sh / DB;
            if (left >= Q) store(bytes_from(row, sh), to + sh);
            else if (left > 0) store_first<DB>(to + sh, bytes_from(row, sh), left);
            if (tj == 0) row_start(row, to, sh);
        }
        return;
    }
    const int left = jw - Q * jc;
    if (left >= Q) {
#pragma unroll
        for (int p = 0; p < TI / RPP; ++p)
            if (r0 + RPP * p < iw)
                store(slot(ES + r0 + RPP * p, jc), d + (int64_t)(RPP * p) * a.ldd * DB);
    } else if (left > 0) {
#pragma unroll 1
        for (int p = 0; r0 + RPP * p < min(iw, TI); ++p) store_first<DB>(d + (int64_t)(RPP * p) * a.ldd * DB, slot(ES + r0 + RPP * p, jc), left);
    }
}

template <int kSrc, int kDst, int SB, int DB, int PI, int NB, int T, int kKeep, int kSkew = 0>
static int32_t launch_kept(TransposeArgs a, int lds_request, hipStream_t st) {
    constexpr int ES = 16 / SB, Q = 16 / DB, NJ = T / PI, TI = PI * ES, TJ = NJ * NB * Q, kLds = (TI + ES) * (TJ * DB + (kSkew ? 128 : 0));
    constexpr int kCap = 160 * 1024;  // all of a CU's LDS
    static_assert(kLds <= kCap, "the tile fits");
    auto kern = transpose_blocks<kSrc, kDst, SB, DB, PI, NB, T, kKeep, kSkew>;
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

// Which form of the destination's rows (kSkew), for tiles of 1 KiB of a row: 0 where their pitch is whole lines, or where the tiles more that the shift
// costs are worth more than the lines.  us without / with, operands not cached: fp16 into rows of whole pieces from four tiles to a row on,
// 4864 x 5992 28.0 / 23.1, 16000 x 16008 230 / 207, [1,3000,32,128] -> [1,32,128,3000] 10.7 / 10.1, [4,1672,32,128] 25.2 / 22.6, 14336 x 1640 21.9 / 21.6,
// 24704 x 1640 37.8 / 36.8, 22392 x 1992 40.3 / 37.9; three tiles to a row gain as often as they lose (21852 x 1288 25.7 / 26.3, 34908 x 1288 39.7 / 41.0,
// 38400 x 1288 43.7 / 42.2, 22004 x 1464 30.7 / 32.4), two as well (128 matrices 128 x 776 11.8 / 12.3, 128 x 904 14.1 / 13.4); f32 from 20 KiB and 48 MiB
// on, 4860 x 5992 50.3 / 47.5, 16000 x 16008 446 / 405, but 13361 x 3728 76.6 / 78.4, 3004 x 2996 15.7 / 16.3; fp16 into any rows of one matrix
// from 5888 elements on, 4861 x 5993 29.6 / 27.1, 16001 x 16011 254 / 216, 1033 x 14001 14.3 / 13.6, but 10001 x 4099 39.0 / 41.8, 4000 x 4499 20.8 / 21.8 and
// in batches [4,2001,32,128] 31.7 / 33.2; f32 into any rows 115.3 / 119.1 (10001 x 7003); f32 -> bf16 18.5 / 18.5 (5000 x 3000).
// Not 16-bit tiles, one to a CU, of which a second round has less than half a round's (1329 x 13256 18.2 / 18.8, 1691 x 11920 19.1 / 19.7, 8448 x 1640 16.1 / 16.4,
// 4216 x 4000 17.9 / 20.3).
static int skew_of(const TransposeArgs& a, int db, bool dst_lines) {
    constexpr int64_t Mi = 1 << 20;
    const int64_t row = (int64_t)a.nj * db;
    if (dst_lines || (db == 2 ? a.nj <= 3 * 512 : row < 20480) || (db == 4 && row * a.ni * a.batch < 48 * Mi)) return 0;
    const int64_t tiles = ((int64_t)a.ni + 127) / 128 * ((a.nj + 511) / 512) * a.batch, cus = 32 * a.xcds;
    if (db == 2 && tiles > cus && 2 * tiles < 3 * cus) return 0;
    int64_t all = reinterpret_cast<uintptr_t>(a.dst) | a.ldd * db;
    for (int m = 0; m < a.modes; ++m) all |= a.d_stride[m] * db;
    if (all % 16 == 0) return 1;
    return db == 2 && a.batch == 1 && a.nj >= 5888 ? 2 : 0;
}
template <int kSrc, int kDst, int SB, int DB>
static int32_t launch_skewed(const TransposeArgs& a, int skew, int keep, int lds_request, hipStream_t st) {
    if constexpr (DB == 2) {
        if (skew == 2)
            return keep == 1 ? launch_kept<kSrc, kDst, SB, DB, 16, 2, 512, 1, 2>(a, lds_request, st) : launch_kept<kSrc, kDst, SB, DB, 16, 2, 512, 0, 2>(a, lds_request, st);
    }
    return keep == 1 ? launch_kept<kSrc, kDst, SB, DB, 16, 2, 512, 1, 1>(a, lds_request, st) : launch_kept<kSrc, kDst, SB, DB, 16, 2, 512, 0, 1>(a, lds_request, st);
}

template <int kSrc, int kDst, int SB, int DB, int PI, int NB, int T>
static int32_t launch_blocks(const TransposeArgs& a, int keep, int lds_request, hipStream_t st) {
    if constexpr (SB <= 4 && DB <= 4) {
        if (keep == 1) return launch_kept<kSrc, kDst, SB, DB, PI, NB, T, 1>(a, lds_request, st);
    }
    if constexpr (SB <= 4 && DB == 1) {
        if (keep == 2) return launch_kept<kSrc, kDst, SB, DB, PI, NB, T, 2>(a, lds_request, st);
    }
    return launch_kept<kSrc, kDst, SB, DB, PI, NB, T, 0>(a, lds_request, st);
}

// The first of a list of tiles (its extents along i and j) that takes at most a quarter more than the tightest of them takes
// over an array's edges.
struct Tile {
    int i, j;
};
static int first_that_fits(const TransposeArgs& a, std::initializer_list<Tile> tiles) {
    auto padded = [&](const Tile& t) { return ((int64_t)a.ni + t.i - 1) / t.i * t.i * (((int64_t)a.nj + t.j - 1) / t.j * t.j); };
    int64_t tightest = padded(*tiles.begin());
    for (const Tile& t : tiles) tightest = std::min(tightest, padded(t));
    int n = 0;
    for (const Tile& t : tiles) {
        if (4 * padded(t) <= 5 * tightest) return n;
        ++n;
    }
    return 0;
}

// Which tile, and how the workgroups are spread.  Up to 2 Mi elements: small tiles, so that there are workgroups for every CU; up
// to 8 Mi: medium ones.  Beyond, rows that are whole 128-byte lines on both sides take tiles whose runs are whole lines,
// anything else the longest runs, whose ends are the smallest part of them.  In every class a matrix narrower than a tile
// (batches of small matrices, long strips) takes a tile that it fills.
//   Order: destination rows first where the source's contiguous extent is at least the destination's (writes are the side that
// needs locality on this part: 16384^2 f32 341 us, 353 source rows first), else bands of 64 tile columns with the source's
// index fastest, with whole lines from an extent of 4096 on (4096 x 32768 f32 196 us, 208 the other way; but bf16 -> f32
// 64 x 1048576 71 and 86).  Neighbouring tiles go to one XCD (`run`), so that lines two of them share meet in one L2 (f32
// 8192^2 102.8 -> 96.6 us, 16400 x 16392 ~420 -> 405), except where an even spread is worth more: few elements, and whole
// lines below 64 MiB (128 x 128 tiles, fp16 2048^2 5.2 -> 4.6, bf16 -> fp32 4096 x 1024 6.0 -> 5.2).
//   Measured with operands that are not cached, us, the kernels for whole 64 x 64 patches that this one replaced / one tile for
// every extent / this rule: fp16 32768 x [64, 64] 85 / 400 / 85; 16384 x [128, 64] 85 / 235 / 87; 1048576 x 128 93 / 148 / 89; 4096^2
// 15.8 / 14.8 / 12.6; fp32 2048^2 7.4 / 9.2 / 7.0; 16 x [512, 512] 7.2 / 8.6 / 7.0; 1048576 x 64 93 / 106 / 90; 100000 x [33, 33] 552 /
// 1051 / 206; 4096 x 32768 196 / 209 / 196; bytes 2048^2 4.4 / 4.7 / 4.0, 262144 x 256 26 / 28 / 28; 8-byte elements 256 x 262144
// 169 / 177 / 169, 8192 x [32, 32] 52 / 72 / 24; bf16 -> fp32 16384 x [64, 128] 138 / 216 / 135; fp8 -> bf16 64 x [1024, 1024] 34 / 40 / 36.
template <int kSrc, int kDst, int SB, int DB>
static int32_t launch_shape(TransposeArgs a, hipStream_t st) {
    constexpr int64_t Mi = 1 << 20;
    const int64_t n = (int64_t)a.ni * a.nj * a.batch, bytes = n * std::max(SB, DB);
    const bool src_lines = (a.lds * SB) % 128 == 0, dst_lines = (a.ldd * DB) % 128 == 0, lines = src_lines && dst_lines;
    const bool few = n <= 2 * Mi, huge = bytes >= 256 * Mi, narrow = std::min(a.ni, a.nj) <= 512;
    const bool medium = !few && lines && n <= 8 * Mi;
    a.run = few || (lines && bytes < 64 * Mi) ? 1 : 4;
    if (a.batch == 1 && a.ni < a.nj && (a.ni >= 4096 || !(few || lines))) a.band = 64;
    // Which accesses go without the non-temporal hint.  Lines of the source that two tiles share (a pitch that is no whole lines), or a
    // call of which the 256 MiB memory-side cache holds a good part: ordinary loads.  Bytes whose destination has such a pitch, from 16 Mi
    // elements on: ordinary stores instead.  us, hinted / loads / stores (/ both): f32 3000^2 18.3 / 17.0 / 19.0 /
    // 18.4, 10001 x 7003 134.6 / 118.8 / 146 / 125, 4096^2 24.3 / 20.4 / 24.2 / 28.6, but 16384 x 2048 47.7 / 51.2 / 51.1 / 56.0, 8192^2 94.8 / 101 / 102 / 109
    // and 2796 x 693 5.6 / 6.2 / 5.8 / 6.0; f32 -> bf16 4096^2 18.5 / 15.7 / 18.8 / 19.4, 5000 x 3000 19.1 / 16.1 / 18.6 / 18.0; fp16 10001 x 7003 75.3 /
    // 70.2 / 80.4 / 73.7; bytes 5000 x 7003 26.7 / 27.2 / 21.7 / 21.7, but 1968 x 6271 9.2 / 9.8 / 10.3 / 10.4; bf16 -> fp8 9001 x 7003 61.4 / 57.8 / 46.0 / 53.0.
    //   Only the destination's pitch ragged, the source's lines read once each: ordinary loads while the cache holds most of the source, up to
    // 300 MiB (f32 8192 x 8200 101.5 / 104.2 but cached 99.9 / 80.2, 5760 x 12408 121.5 / 123.3 but cached 120.5 / 105), hinted ones beyond (f32 9216 x 9000 126.6 / 135.0,
    // 16000 x 16010 445 / 471; f32 -> bf16 9216 x 9000 94.8 / 100.9, 14336 x 7000 114.9 / 121.4, 7168 x 14003 127.3 / 129.5; fp16 20480 x 10000
    // 156.3 / 165.3) and for few elements (up to 4 Mi, of 16-bit sources 8, over 45 sizes 0.96 of the time with loads, cached 1.02: f32 512 x 4792
    // 6.36 / 6.84, cached 5.32 / 5.19; f32 -> bf16 768 x 4128 7.02 / 7.40, 5.06 / 4.83; fp16 5760 x 963 6.88 / 7.11, 5.74 / 5.79).  Only the source's, bytes: loads (12408 x 5760 40.4 / 35.1 / 42.3, 10000 x 20480 99.4 / 87.4 / 99.9; bf16 -> fp8 7000 x 7168 33.1 /
    // 31.2 / 36.2).
    const int keep = few || (lines && DB == 1 && n <= 4 * Mi) ? 0
                     : lines                                  ? (n * (SB + DB) <= 160 * Mi ? 1 : 0)
                     : DB == 1                                ? (n < 16 * Mi ? 0 : dst_lines ? 1 : 2)
                                                              : (src_lines && (n * SB > 300 * Mi || n <= (SB == 2 ? 8 : 4) * Mi) ? 0 : 1);
    auto fit = [&](std::initializer_list<Tile> tiles) { return first_that_fits(a, tiles); };
#define MOYE_TILE(PI, NB, T, LDS) return launch_blocks<kSrc, kDst, SB, DB, PI, NB, T>(a, keep, LDS, st)
    if constexpr (SB == 2 && DB == 2) {
        if (few) switch (fit({{128, 64}, {64, 128}, {64, 64}})) {
            case 0: MOYE_TILE(16, 1, 128, 0);
            case 1: MOYE_TILE(8, 1, 128, 0);
            default: MOYE_TILE(8, 1, 64, 0);
        }
        if (n <= 8 * Mi) switch (fit({{128, 128}, {128, 64}, {64, 128}, {64, 64}})) {
            case 0: MOYE_TILE(16, 1, 256, 0);
            case 1: MOYE_TILE(16, 1, 128, 0);
            case 2: MOYE_TILE(8, 1, 128, 0);
            default: MOYE_TILE(8, 1, 64, 0);
        }
        if (!lines || (n <= 16 * Mi && !narrow)) switch (fit({{128, 512}, {128, 128}, {64, 64}})) {
            case 0:
                if (const int skew = skew_of(a, DB, dst_lines)) return launch_skewed<kSrc, kDst, SB, DB>(a, skew, keep, 0, st);
                MOYE_TILE(16, 2, 512, 0);
            case 1: MOYE_TILE(16, 1, 256, 0);
            default: MOYE_TILE(8, 1, 64, 0);
        }
        if (huge) switch (fit({{128, 256}, {128, 128}, {128, 64}})) {
            case 0: MOYE_TILE(16, 2, 256, 0);
            case 1: MOYE_TILE(16, 1, 256, 0);
            default: MOYE_TILE(16, 1, 128, 0);
        }
        if (!narrow && a.batch == 1) MOYE_TILE(8, 1, 256, 0);
        switch (fit({{256, 64}, {64, 128}, {64, 64}})) {
            case 0: MOYE_TILE(32, 1, 256, 0);
            case 1: MOYE_TILE(8, 1, 128, 0);
            default: MOYE_TILE(8, 1, 64, 0);
        }
    } else if constexpr (SB == 4 && DB == 4) {
        constexpr int kAlone = 96 * 1024;  // one workgroup per CU, where the arrays are far beyond the caches
        if (few) { if (fit({{32, 64}, {64, 64}}) == 0) MOYE_TILE(8, 1, 128, 0); else MOYE_TILE(16, 2, 128, 0); }
        if (medium) { if (fit({{128, 64}, {64, 64}}) == 0) MOYE_TILE(32, 2, 256, 0); else MOYE_TILE(16, 2, 128, 0); }
        if (!lines) switch (bytes >= 32 * Mi ? fit({{64, 256}, {128, 128}, {64, 64}}) : 3 + fit({{64, 128}, {64, 64}})) {
            case 0:
                if (const int skew = skew_of(a, DB, dst_lines)) return launch_skewed<kSrc, kDst, SB, DB>(a, skew, keep, kAlone, st);
                MOYE_TILE(16, 2, 512, kAlone);
            case 1: MOYE_TILE(32, 4, 256, 0);
            case 3: MOYE_TILE(16, 2, 256, 0);
            default: MOYE_TILE(16, 2, 128, 0);
        }
        if (a.ni <= 128) MOYE_TILE(32, 2, 256, 0);
        if (narrow) { if (fit({{64, 128}, {64, 64}}) == 0) MOYE_TILE(16, 2, 256, 0); else MOYE_TILE(16, 1, 256, 0); }
        if (bytes >= 600 * Mi) {  // (the tiles in plain order: 16384^2 341 us against 357)
            if (a.band == 0) a.run = 1;
            MOYE_TILE(16, 2, 512, kAlone);
        }
        if (a.band) MOYE_TILE(32, 4, 256, 0);
        MOYE_TILE(8, 1, 256, 0);
    } else if constexpr (SB == 1 && DB == 1) {
        if (n <= 6 * Mi || medium) switch (fit({{256, 64}, {128, 128}, {64, 256}})) {
            case 0: MOYE_TILE(16, 1, 64, 0);
            case 1: MOYE_TILE(8, 1, 64, 0);
            default: MOYE_TILE(4, 1, 64, 0);
        }
        if (!lines && n <= 8 * Mi) { if (fit({{256, 128}, {256, 64}}) == 0) MOYE_TILE(16, 1, 128, 0); else MOYE_TILE(16, 1, 64, 0); }
        switch (n > 64 * Mi                         ? 1 + fit({{128, 512}, {256, 128}, {256, 64}})
                : !lines                            ? fit({{256, 256}, {128, 512}, {256, 128}, {256, 64}})
                : a.batch == 1                      ? 4 + fit({{256, 256}, {256, 128}, {128, 256}, {256, 64}})
                                                    : 5 + fit({{256, 128}, {128, 256}, {256, 64}})) {
            case 0: case 4: MOYE_TILE(16, 1, 256, 0);
            case 1: MOYE_TILE(8, 1, 256, 0);
            case 2: case 5: MOYE_TILE(16, 1, 128, 0);
            case 6: MOYE_TILE(8, 1, 128, 0);
            default: MOYE_TILE(16, 1, 64, 0);
        }
    } else if constexpr (SB == 8 && DB == 8) {
        if (few) { if (fit({{32, 64}, {32, 32}}) == 0) MOYE_TILE(16, 4, 128, 0); else MOYE_TILE(16, 2, 128, 0); }
        if (medium) { if (fit({{64, 64}, {32, 32}}) == 0) MOYE_TILE(32, 4, 256, 0); else MOYE_TILE(16, 2, 128, 0); }
        if (!lines) switch (fit({{64, 128}, {64, 64}, {32, 32}})) {
            case 0: MOYE_TILE(32, 4, 512, bytes >= 24 * Mi ? 96 * 1024 : 0);
            case 1: MOYE_TILE(32, 4, 256, 0);
            default: MOYE_TILE(16, 2, 128, 0);
        }
        if (huge && a.nj > 128 && fit({{64, 128}, {64, 64}}) == 0) {  // (plain order from 1 GiB: 16384^2 699 us against 774, 8192^2 185 and 180)
            if (bytes >= 1024 * Mi || a.ni < a.nj) a.run = 1;
            a.band = 0;
            MOYE_TILE(32, 4, 512, 96 * 1024);
        }
        MOYE_TILE(32, 2, 512, 0);
    } else if constexpr (SB == 4 && DB == 2) {
        if (few) { if (fit({{32, 64}, {64, 64}}) == 0) MOYE_TILE(8, 1, 64, 0); else MOYE_TILE(16, 1, 128, 0); }
        if (medium) MOYE_TILE(16, 1, 128, 0);
        if (!lines) {
            const int t = fit({{64, 512}, {128, 128}, {64, 64}});
            if (t == 0) MOYE_TILE(16, 2, 512, 0);
            if (t == 1) MOYE_TILE(32, 1, 512, 0); else MOYE_TILE(16, 1, 128, 0);
        }
        if (narrow || a.batch > 1) switch (fit({{128, 128}, {64, 128}, {64, 64}})) {
            case 0: MOYE_TILE(32, 1, 512, 0);
            case 1: MOYE_TILE(16, 1, 256, 0);
            default: MOYE_TILE(16, 1, 128, 0);
        }
        if (n <= 16 * Mi) MOYE_TILE(32, 1, 256, 0);
        MOYE_TILE(16, 1, 512, 0);
    } else if constexpr (SB == 2 && DB == 4) {
        if (few) MOYE_TILE(8, 1, 128, 0);
        if (!lines) switch (fit({{128, 256}, {128, 128}, {64, 64}})) {
            case 0: MOYE_TILE(16, 2, 512, 0);
            case 1: MOYE_TILE(16, 2, 256, 0);
            default: MOYE_TILE(8, 1, 128, 0);
        }
        if (medium || std::min(a.ni, a.nj) <= 128 || (narrow && a.batch > 1)) {
            if (fit({{128, 64}, {64, 64}}) == 0) MOYE_TILE(16, 1, 256, 0); else MOYE_TILE(8, 1, 128, 0);
        }
        if (huge) MOYE_TILE(16, 2, 256, 0);
        MOYE_TILE(8, 1, 256, 0);
    } else if constexpr (SB == 4 && DB == 1) {
        if (few) MOYE_TILE(16, 1, 64, 0);
        if (medium) { if (fit({{128, 64}, {64, 64}}) == 0) MOYE_TILE(32, 1, 128, 0); else MOYE_TILE(16, 1, 64, 0); }
        switch (!lines && n <= 8 * Mi ? 1 + fit({{64, 256}, {64, 64}})
                : lines && huge       ? 3 + fit({{128, 128}, {64, 256}, {64, 64}})
                                      : 6 + fit({{64, 512}, {64, 256}, {128, 64}, {64, 64}})) {
            case 1: case 4: case 7: MOYE_TILE(16, 1, 256, 0);
            case 3: MOYE_TILE(32, 1, 256, 0);
            case 6: MOYE_TILE(16, 1, 512, 0);
            case 8: MOYE_TILE(32, 1, 128, 0);
            default: MOYE_TILE(16, 1, 64, 0);
        }
    } else if constexpr (SB == 2 && DB == 1) {
        if (few || medium) { if (fit({{64, 128}, {128, 64}}) == 0) MOYE_TILE(8, 1, 64, 0); else MOYE_TILE(16, 1, 64, 0); }
        switch (fit({{128, 256}, {128, 128}, {64, 256}, {128, 64}})) {
            case 0: MOYE_TILE(16, 1, 256, 0);
            case 1: MOYE_TILE(16, 1, 128, 0);
            case 2: MOYE_TILE(8, 1, 128, 0);
            default: MOYE_TILE(16, 1, 64, 0);
        }
    } else if constexpr (SB == 1 && DB == 2) {
        if (few) { if (fit({{128, 64}, {64, 128}}) == 0) MOYE_TILE(8, 1, 64, 0); else MOYE_TILE(4, 1, 64, 0); }
        switch (medium   ? 1 + fit({{128, 128}, {128, 64}})
                : !lines ? fit({{128, 256}, {128, 128}, {128, 64}})
                         : 3 + fit({{256, 128}, {256, 64}, {128, 64}})) {
            case 0: MOYE_TILE(8, 1, 256, 0);
            case 1: MOYE_TILE(8, 1, 128, 0);
            case 3: MOYE_TILE(16, 1, 256, 0);
            case 4: MOYE_TILE(16, 1, 128, 0);
            default: MOYE_TILE(8, 1, 64, 0);
        }
    } else if constexpr (SB == 1 && DB == 4) {
        if (few || medium) MOYE_TILE(4, 1, 64, 0);
        if (!lines) { if (fit({{128, 128}, {64, 64}}) == 0) MOYE_TILE(8, 1, 256, 0); else MOYE_TILE(4, 1, 64, 0); }
        if (fit({{128, 64}, {64, 64}}) == 0) MOYE_TILE(8, 1, 128, 0); else MOYE_TILE(4, 1, 64, 0);
    } else if constexpr (SB == 1) {
        static_assert(DB == 8, "every pair of sizes");
        MOYE_TILE(4, 1, 256, 0);
    } else if constexpr (SB == 8) {
        MOYE_TILE(16, DB == 4 ? 2 : 1, 256, 0);
    } else {
        static_assert(DB == 8, "every pair of sizes");
        MOYE_TILE(SB == 4 ? 16 : 8, SB == 4 ? 4 : 2, 256, 0);
    }
#undef MOYE_TILE
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

// Few elements, of one or two bytes, are a chain of latencies in a lane's block (16 loads and 256 bytes to turn for bytes), the
// longer one where destination rows end inside a piece; the general kernel has a wave for every 64 elements.  us, that one / this one:
// bytes 201 x 303 3.5 / 5.6, 700 x 500 4.9 / 5.8, 1001 x 700 6.9 / 6.8, 256 x 256 3.5 / 3.0; bf16 -> fp8 256 x 256 3.2 / 4.1, 700 x
// 500 4.5 / 5.5; fp16 128 x 128 2.5 / 2.2, 500 x 300 4.0 / 4.4, 700 x 500 4.9 / 4.4; fp8 -> fp32 201 x 303 3.4 / 5.4, 500 x 300 3.8 / 4.2; bf16 -> fp32 201 x 303
// 3.1 / 4.0, 128 x 128 3.0 / 2.4; fp32 201 x 303 3.6 / 3.5, 128 x 128 3.0 / 2.3.
bool transpose_pays(int32_t src_dt, int32_t dst_dt, const TransposeArgs& a) {
    const int sb = dtype_bytes(src_dt), db = dtype_bytes(dst_dt), lo = std::min(sb, db), hi = std::max(sb, db);
    const bool whole = a.nj % (16 / db) == 0;
    const int64_t n = (int64_t)a.ni * a.nj * a.batch;
    if (hi == 8 || lo == 4) return true;
    if (lo == 1 && hi <= 2) return n > (!whole ? 512 << 10 : hi == 2 ? 64 << 10 : 12 << 10);
    if (lo == 2 && hi == 2) return n > (whole ? 8 << 10 : 160 << 10);
    if (lo == 1) return whole || n > (160 << 10);
    return whole || n > (64 << 10);
}

int32_t transpose_run(int32_t src_dt, int32_t dst_dt, bool same_bits, bool linear_lds, int xcds, TransposeArgs a, hipStream_t st) {
    a.band = 0;  // (the tile's choice may set both)
    a.xcds = xcds;
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
