// copyto! on the device: layout-driven copy kernels for gfx950.
//
// Takes over the element loop of the reference's `copyto!`
// (src/algorithm/copy.jl:4-12,42-64 and :106-130): logical element i of src goes to logical
// element i of dst through both layouts.  Three kinds of kernel:
//   transpose_blocks (copy_transpose.hip)  the unit-stride mode differs between src and dst
//   copy_flat       both sides contiguous in the same order: 128-bit streaming copy
//   copy_generic, copy_groups    anything else: gather/scatter with optional conversion
#include <algorithm>

#include "copy_convert.hpp"
#include "copy_transpose.hpp"
#include "kernels.hpp"

namespace moye {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // one 128-bit access

// ------------------------------------------------------------------------------------------
// contiguous streaming copy, 16 bytes per lane per step
// ------------------------------------------------------------------------------------------
// One 16-byte piece per lane, one workgroup per 4 KiB, non-temporal on both sides, no loop: measured on 1 GiB
// 6.56 TB/s against 6.09 for workgroups that walk 16 KiB chunks with four pieces of a lane in flight (6.04-6.25 with two
// or four pieces per lane and no loop, 4.3 with eight; 6.2 without the non-temporal hints).
__global__ __launch_bounds__(256) void copy_flat_b128(const u32x4* __restrict__ src,
                                                      u32x4* __restrict__ dst, int64_t n16) {
    const int64_t i = flat_piece();
    if (i < n16) __builtin_nontemporal_store(__builtin_nontemporal_load(src + i), dst + i);
}

// The same for any length from 16 bytes on and any alignment: the last piece is moved back to end with the run (what two lanes then
// write twice is the same).  us, byte by byte / now: f16 3001 x 2003 10.3 / 5.3, bf16 14545 x 1766 56.6 / 18.2.
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
__global__ __launch_bounds__(256) void copy_flat_any(const char* __restrict__ src, char* __restrict__ dst, int64_t bytes) {
    const int64_t i = flat_piece() * 16;
    if (i >= bytes) return;
    const int64_t at = i + 16 <= bytes ? i : bytes - 16;
    const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(src + at));
    __builtin_nontemporal_store(w, reinterpret_cast<u32x4_any*>(dst + at));
}

__global__ __launch_bounds__(256) void copy_flat_bytes(const uint8_t* __restrict__ src,
                                                       uint8_t* __restrict__ dst, int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

// ------------------------------------------------------------------------------------------
// generic gather/scatter with conversion
// ------------------------------------------------------------------------------------------
struct FlatLayout {
    int32_t rank;
    int64_t shape[MOYE_MAX_RANK];
    int64_t stride[MOYE_MAX_RANK];
};

// colexicographic decomposition of a 0-based linear index (src/stride.jl:20-31)
__device__ __forceinline__ int64_t layout_offset(const FlatLayout& l, int64_t i) {
    int64_t off = 0;
#pragma unroll 1
    for (int m = 0; m < l.rank; ++m) {
        const int64_t s = l.shape[m];
        const int64_t q = i / s;
        off += (i - q * s) * l.stride[m];
        i = q;
    }
    return off;
}

// copyto_if! (src/algorithm/copy.jl:4-16): element i moves only where the mask's logical element i is nonzero
struct Mask {
    const uint8_t* ptr;  // null = every element moves
    FlatLayout l;
};
__device__ __forceinline__ bool masked_out(const Mask& m, int64_t i) { return m.ptr && !m.ptr[layout_offset(m.l, i)]; }

// layouts of one shape mode by mode, few enough pieces for 32-bit indices
static bool same_modes_32(const FlatLayout& a, const FlatLayout& b, int64_t n) {
    if (a.rank != b.rank || n >= ((int64_t)1 << 31)) return false;
    for (int m = 0; m < a.rank; ++m)
        if (a.shape[m] != b.shape[m] || a.shape[m] <= 0) return false;
    return true;
}

template <int kBytes>
__global__ __launch_bounds__(256) void copy_generic_bits(const char* __restrict__ src,
                                                         char* __restrict__ dst, FlatLayout ls,
                                                         FlatLayout ld, int64_t n, Mask mask) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        if (masked_out(mask, i)) continue;
        const char* s = src + layout_offset(ls, i) * kBytes;
        char* d = dst + layout_offset(ld, i) * kBytes;
        if constexpr (kBytes == 1) *reinterpret_cast<uint8_t*>(d) = *reinterpret_cast<const uint8_t*>(s);
        else if constexpr (kBytes == 2) *reinterpret_cast<uint16_t*>(d) = *reinterpret_cast<const uint16_t*>(s);
        else if constexpr (kBytes == 4) *reinterpret_cast<uint32_t*>(d) = *reinterpret_cast<const uint32_t*>(s);
        else if constexpr (kBytes == 8) *reinterpret_cast<uint64_t*>(d) = *reinterpret_cast<const uint64_t*>(s);
        else *reinterpret_cast<u32x4*>(d) = *reinterpret_cast<const u32x4*>(s);
    }
}

// The same for two layouts of one shape, mode by mode, and fewer than 2^31 pieces: the index is taken apart once, with
// 32-bit divisions, and the coordinates are weighed with both sides' strides (the general form divides 64-bit numbers
// twice per mode, which is most of its time: [16, 2048, 32, 128] -> [16, 32, 2048, 128] fp32 240 us against 172 this way).
// kStream: non-temporal accesses, for arrays far beyond the caches.
template <int kBytes, bool kStream>
__global__ __launch_bounds__(256) void copy_generic_bits_same(const char* __restrict__ src, char* __restrict__ dst, FlatLayout ls, FlatLayout ld,
                                                              uint32_t n) {
    typedef std::conditional_t<kBytes == 16, u32x4, std::conditional_t<kBytes == 8, uint64_t, std::conditional_t<kBytes == 4, uint32_t,
            std::conditional_t<kBytes == 2, uint16_t, uint8_t>>>> piece;
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        int64_t so = 0, dof = 0;
        uint32_t rest = i;
#pragma unroll 1
        for (int m = 0; m < ls.rank; ++m) {
            const uint32_t extent = (uint32_t)ls.shape[m], q = rest / extent, c = rest - q * extent;
            so += (int64_t)c * ls.stride[m];
            dof += (int64_t)c * ld.stride[m];
            rest = q;
        }
        const piece* s = reinterpret_cast<const piece*>(src + so * kBytes);
        piece* d = reinterpret_cast<piece*>(dst + dof * kBytes);
        if constexpr (kStream) __builtin_nontemporal_store(__builtin_nontemporal_load(s), d);
        else *d = *s;
    }
}

template <int kBytes>
static void launch_generic_bits_same(const char* s, char* d, const FlatLayout& ls, const FlatLayout& ld, int64_t n, hipStream_t st) {
    const dim3 g((unsigned)std::min<int64_t>((n + 255) / 256, (int64_t)1 << 22));
    if (n * kBytes >= ((int64_t)64 << 20)) copy_generic_bits_same<kBytes, true><<<g, 256, 0, st>>>(s, d, ls, ld, (uint32_t)n);
    else copy_generic_bits_same<kBytes, false><<<g, 256, 0, st>>>(s, d, ls, ld, (uint32_t)n);
}
template <int kSrc, int kDst>
__global__ __launch_bounds__(256) void copy_generic_cvt(const char* __restrict__ src,
                                                        char* __restrict__ dst, FlatLayout ls,
                                                        FlatLayout ld, int64_t n, int sb, int db, Mask mask) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        if (masked_out(mask, i)) continue;
        const double v = load_as_f64<kSrc>(src + layout_offset(ls, i) * sb);
        store_from<kDst>(dst + layout_offset(ld, i) * db, v, kSrc == MOYE_F64);
    }
}

// The same element loops, V elements per lane: for arrays whose first mode (once the modes are ordered by stride) is a
// run of unit stride and one length of at least V on every side -- pitched matrices, slices of larger arrays -- whatever its
// length, the pitches and the alignment.  The last group of a run is moved back to end with it: what two lanes then move
// twice is the same (under a mask too: both write the elements it names, and leave or write back the others) -- unless a
// conversion's source is its destination, where one lane may read what another has converted: launch_groups refuses that.
// The vectorisation the reference computes with max_common_vector
// (src/layout.jl:752-761) and leaves unused (src/algorithm/copy.jl:53-58), here also for converting copies (the wider
// side moves 16 bytes per lane) and for copyto_if! (the mask is read V bytes at a time; a group whose mask is all true
// goes out in one access, a mixed one element by element, so that elements whose mask is false are never written).
// Mode 0 of the layouts counts groups, the other modes elements.  Same conversion per
// element as copy_generic_cvt; kSrc == kDst moves bits.  us, element by element where V divided no run, pitch or address / now:
// copyto_if! f16 3001 x
// 2003 20.6 / 5.1, bf16 14545 x 1766 75.9 / 12.3; 3001 columns of 6002, 2003 rows, f32 -> bf16 25.4 / 8.0.  Aligned ones as before (window
// 8192^2 of 16384 columns f32 -> bf16 75.8 / 73.6).
template <int N> struct BytesOf;
template <> struct BytesOf<1> { typedef uint8_t type; };
template <> struct BytesOf<2> { typedef uint16_t type __attribute__((aligned(1))); };
template <> struct BytesOf<4> { typedef uint32_t type __attribute__((aligned(1))); };
template <> struct BytesOf<8> { typedef uint64_t type __attribute__((aligned(1))); };
template <> struct BytesOf<16> { typedef u32x4_any type; };
// kSame: the layouts (the mask's too) have one shape mode by mode and there are fewer than 2^31 groups: the index is taken
// apart once, with 32-bit divisions, for all of them (see copy_generic_bits_same).  `run`: elements in mode 0.
template <int kSrc, int kDst, int SB, int DB, int V, bool kSame = false>
__global__ __launch_bounds__(256) void copy_groups(const char* __restrict__ src, char* __restrict__ dst, FlatLayout ls, FlatLayout ld,
                                                   int64_t ngroups, int64_t run, Mask mask) {
    typedef typename BytesOf<V * SB>::type SrcWord;
    typedef typename BytesOf<V * DB>::type DstWord;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < ngroups; g += stride) {
        int64_t so = 0, dof = 0, mo = 0;
        if constexpr (kSame) {
            const uint32_t groups = (uint32_t)ls.shape[0];
            uint32_t rest = (uint32_t)g / groups;
            so = dof = mo = min((int64_t)((uint32_t)g - rest * groups) * V, run - V);
#pragma unroll 1
            for (int m = 1; m < ls.rank; ++m) {
                const uint32_t extent = (uint32_t)ls.shape[m], q = rest / extent, c = rest - q * extent;
                so += (int64_t)c * ls.stride[m];
                dof += (int64_t)c * ld.stride[m];
                if (mask.ptr) mo += (int64_t)c * mask.l.stride[m];
                rest = q;
            }
        } else {
            const int64_t groups = ls.shape[0], rest = g / groups, at = min((g - rest * groups) * V, run - V), first = rest * groups;  // (group 0 of the run)
            so = layout_offset(ls, first) + at;
            dof = layout_offset(ld, first) + at;
            if (mask.ptr) mo = layout_offset(mask.l, first) + at;
        }
        uint8_t keep[V];
        bool all = true, any = true;
        if (mask.ptr) {
            typedef typename BytesOf<V>::type MaskWord;
            const MaskWord mw = *reinterpret_cast<const MaskWord*>(mask.ptr + mo);
            __builtin_memcpy(keep, &mw, V);
            any = false;
#pragma unroll
            for (int e = 0; e < V; ++e) {
                all = all && keep[e];
                any = any || keep[e];
            }
            if (!any) continue;
        }
        const SrcWord in = *reinterpret_cast<const SrcWord*>(src + so * SB);
        char* const d = dst + dof * DB;
        DstWord out;
        if constexpr (kSrc == kDst) {
            static_assert(SB == DB, "bits");
            __builtin_memcpy(&out, &in, V * SB);
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e) {
                char e_in[SB], e_out[DB];
                __builtin_memcpy(e_in, reinterpret_cast<const char*>(&in) + e * SB, SB);
                store_from<kDst>(e_out, load_as_f64<kSrc>(e_in), kSrc == MOYE_F64);
                __builtin_memcpy(reinterpret_cast<char*>(&out) + e * DB, e_out, DB);
            }
        }
        if (all) {
            *reinterpret_cast<DstWord*>(d) = out;
        } else if constexpr (V >= 8) {
            // some of a group of eight or sixteen: the destination's own values fill the gaps and the group goes out in one
            // piece (the elements the mask leaves out are written back as they were read; nothing else writes them during a
            // copyto_if!).  Element by element, a random mask cost eight partial stores per lane: fp16 8192^2 3.07 TB/s
            // against 4.64.  Groups of four gain nothing from it (f32 -> f16 4.46 against 4.10 this way).
            DstWord old = *reinterpret_cast<const DstWord*>(d);
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (keep[e]) __builtin_memcpy(reinterpret_cast<char*>(&old) + e * DB, reinterpret_cast<const char*>(&out) + e * DB, DB);
            *reinterpret_cast<DstWord*>(d) = old;
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (keep[e]) __builtin_memcpy(d + e * DB, reinterpret_cast<const char*>(&out) + e * DB, DB);
        }
    }
}

// Converting copy between two dense, 16-byte aligned runs of elements of one width (fp16 <-> bf16): a lane converts the
// elements of one 16-byte piece; one workgroup per 256 pieces, no loop.  Element by element the same conversion as
// copy_generic_cvt.
template <int kSrc, int kDst, int SB, int DB>
__global__ __launch_bounds__(256) void copy_cvt_dense(const char* __restrict__ src, char* __restrict__ dst, int64_t nvec) {
    static_assert(SB == DB, "the widening and narrowing directions have kernels of their own");
    constexpr int E = 16 / SB;
    const u32x4* sv = reinterpret_cast<const u32x4*>(src);
    u32x4* dv = reinterpret_cast<u32x4*>(dst);
    const int64_t i = flat_piece();
    if (i >= nvec) return;
    const u32x4 in = __builtin_nontemporal_load(sv + i);
    u32x4 out;
#pragma unroll
    for (int k = 0; k < E; ++k) {
        char e_in[SB], e_out[DB];
        __builtin_memcpy(e_in, reinterpret_cast<const char*>(&in) + k * SB, SB);
        store_from<kDst>(e_out, load_as_f64<kSrc>(e_in), kSrc == MOYE_F64);
        __builtin_memcpy(reinterpret_cast<char*>(&out) + k * DB, e_out, DB);
    }
    __builtin_nontemporal_store(out, dv + i);
}

static FlatLayout flat_of(const moye_tensor& t) {
    FlatLayout f;
    f.rank = t.rank;
    for (int i = 0; i < MOYE_MAX_RANK; ++i) {
        f.shape[i] = i < t.rank ? t.shape[i] : 1;
        f.stride[i] = i < t.rank ? t.stride[i] : 0;
    }
    return f;
}

// Is the layout a dense run 0..size-1 visited in order (compact column-major after dropping
// size-1 modes)?
static bool is_contiguous(const moye_tensor& t) {
    int64_t expect = 1;
    for (int i = 0; i < t.rank; ++i) {
        if (t.shape[i] == 1) continue;
        if (t.stride[i] != expect) return false;
        expect *= t.shape[i];
    }
    return true;
}

// Are both one dense run in the same order: as written, or once the modes of both are ordered by stride (two row-major
// arrays of one shape: a copy may visit the elements in any order)?
static bool one_run_each(const moye_tensor& src, const moye_tensor& dst) {
    if (is_contiguous(src) && is_contiguous(dst)) return true;
    moye_tensor ts = src, td = dst;
    moye_tensor* both[2] = {&td, &ts};
    return order_modes_by_stride(both, 2) && is_contiguous(ts) && is_contiguous(td);
}

// The widening direction: a lane's 16-byte store holds EW = 16 / sizeof(dst) elements, which it reads as one access of
// EW * sizeof(src) bytes (8, 4 or 2), so that loads and stores of a wave are both contiguous; four of them in flight.
template <int NB> struct NarrowWord;
template <> struct NarrowWord<8> { typedef uint64_t type; };
template <> struct NarrowWord<4> { typedef uint32_t type; };
template <> struct NarrowWord<2> { typedef uint16_t type; };
template <int kSrc, int kDst, int SB, int DB>
__global__ __launch_bounds__(256) void copy_cvt_dense_widen(const char* __restrict__ src, char* __restrict__ dst, int64_t nvec) {
    constexpr int EW = 16 / DB, NB = EW * SB;
    typedef typename NarrowWord<NB>::type word;
    const word* sv = reinterpret_cast<const word*>(src);
    u32x4* dv = reinterpret_cast<u32x4*>(dst);
    auto convert = [](word in) {
        u32x4 out;
#pragma unroll
        for (int k = 0; k < EW; ++k) {
            char e_in[SB], e_out[DB];
            __builtin_memcpy(e_in, reinterpret_cast<const char*>(&in) + k * SB, SB);
            store_from<kDst>(e_out, load_as_f64<kSrc>(e_in), kSrc == MOYE_F64);
            __builtin_memcpy(reinterpret_cast<char*>(&out) + k * DB, e_out, DB);
        }
        return out;
    };
    // one piece per lane, one workgroup per 256 pieces, no loop (the form that is fastest for the plain copy)
    const int64_t i = flat_piece();
    if (i < nvec) __builtin_nontemporal_store(convert(__builtin_nontemporal_load(sv + i)), dv + i);
}

// The narrowing direction: a lane reads 16 bytes and stores the EN = 16 / sizeof(src) converted elements as one access of
// 2, 4 or 8 bytes; loads and stores of a wave are contiguous.
template <int kSrc, int kDst, int SB, int DB>
__global__ __launch_bounds__(256) void copy_cvt_dense_narrow(const char* __restrict__ src, char* __restrict__ dst, int64_t nvec) {
    constexpr int EN = 16 / SB, NB = EN * DB;
    typedef typename NarrowWord<NB>::type word;
    const u32x4* sv = reinterpret_cast<const u32x4*>(src);
    word* dv = reinterpret_cast<word*>(dst);
    auto convert = [](const u32x4& in) {
        word out;
#pragma unroll
        for (int k = 0; k < EN; ++k) {
            char e_in[SB], e_out[DB];
            __builtin_memcpy(e_in, reinterpret_cast<const char*>(&in) + k * SB, SB);
            store_from<kDst>(e_out, load_as_f64<kSrc>(e_in), kSrc == MOYE_F64);
            __builtin_memcpy(reinterpret_cast<char*>(&out) + k * DB, e_out, DB);
        }
        return out;
    };
    const int64_t i = flat_piece();
    if (i < nvec) __builtin_nontemporal_store(convert(__builtin_nontemporal_load(sv + i)), dv + i);
}

constexpr int float_bytes(int dt) { return dt == MOYE_F64 ? 8 : dt == MOYE_F32 ? 4 : dt == MOYE_F8E4M3 ? 1 : 2; }

// dense converting copy of the first n - n % E elements; returns how many elements it covered (0: not launched)
template <int kSrc, int kDst>
static int64_t launch_cvt_dense_pair(const char* s, char* d, int64_t n, hipStream_t st) {
    constexpr int SB = float_bytes(kSrc), DB = float_bytes(kDst), E = 16 / (SB < DB ? SB : DB);
    if constexpr (DB > SB) {
        constexpr int EW = 16 / DB;
        const int64_t nvec = n / EW;
        if (nvec == 0) return 0;
        copy_cvt_dense_widen<kSrc, kDst, SB, DB><<<flat_grid(nvec), 256, 0, st>>>(s, d, nvec);
        return nvec * EW;
    }
    if constexpr (SB > DB) {
        static_assert((16 / SB) * DB >= 2, "a lane's store is 2, 4 or 8 bytes");
        constexpr int EN = 16 / SB;
        const int64_t nvec = n / EN;
        if (nvec == 0) return 0;
        copy_cvt_dense_narrow<kSrc, kDst, SB, DB><<<flat_grid(nvec), 256, 0, st>>>(s, d, nvec);
        return nvec * EN;
    }
    if constexpr (SB == DB) {
        const int64_t nvec = n / E;
        if (nvec == 0) return 0;
        copy_cvt_dense<kSrc, kDst, SB, DB><<<flat_grid(nvec), 256, 0, st>>>(s, d, nvec);
        return nvec * E;
    }
    return 0;
}
template <int kSrc>
static int64_t launch_cvt_dense_dst(int32_t dd, const char* s, char* d, int64_t n, hipStream_t st) {
    switch (dd) {
        case MOYE_F32: if constexpr (kSrc != MOYE_F32) return launch_cvt_dense_pair<kSrc, MOYE_F32>(s, d, n, st); break;
        case MOYE_F16: if constexpr (kSrc != MOYE_F16) return launch_cvt_dense_pair<kSrc, MOYE_F16>(s, d, n, st); break;
        case MOYE_BF16: if constexpr (kSrc != MOYE_BF16) return launch_cvt_dense_pair<kSrc, MOYE_BF16>(s, d, n, st); break;
        case MOYE_F8E4M3: if constexpr (kSrc != MOYE_F8E4M3) return launch_cvt_dense_pair<kSrc, MOYE_F8E4M3>(s, d, n, st); break;
        case MOYE_F64: if constexpr (kSrc != MOYE_F64) return launch_cvt_dense_pair<kSrc, MOYE_F64>(s, d, n, st); break;
        default: break;
    }
    return 0;
}
static int64_t launch_cvt_dense(int32_t sd, int32_t dd, const char* s, char* d, int64_t n, hipStream_t st) {
    switch (sd) {
        case MOYE_F32: return launch_cvt_dense_dst<MOYE_F32>(dd, s, d, n, st);
        case MOYE_F16: return launch_cvt_dense_dst<MOYE_F16>(dd, s, d, n, st);
        case MOYE_BF16: return launch_cvt_dense_dst<MOYE_BF16>(dd, s, d, n, st);
        case MOYE_F8E4M3: return launch_cvt_dense_dst<MOYE_F8E4M3>(dd, s, d, n, st);
        case MOYE_F64: return launch_cvt_dense_dst<MOYE_F64>(dd, s, d, n, st);
        default: return 0;
    }
}

template <int kSrc>
static bool launch_cvt_dst(int32_t dd, dim3 g, hipStream_t st, const char* s, char* d, FlatLayout ls,
                           FlatLayout ld, int64_t n, int sb, int db, const Mask& mk) {
    switch (dd) {
        case MOYE_F32: copy_generic_cvt<kSrc, MOYE_F32><<<g, 256, 0, st>>>(s, d, ls, ld, n, sb, db, mk); return true;
        case MOYE_F16: copy_generic_cvt<kSrc, MOYE_F16><<<g, 256, 0, st>>>(s, d, ls, ld, n, sb, db, mk); return true;
        case MOYE_BF16: copy_generic_cvt<kSrc, MOYE_BF16><<<g, 256, 0, st>>>(s, d, ls, ld, n, sb, db, mk); return true;
        case MOYE_F8E4M3: copy_generic_cvt<kSrc, MOYE_F8E4M3><<<g, 256, 0, st>>>(s, d, ls, ld, n, sb, db, mk); return true;
        case MOYE_F64: copy_generic_cvt<kSrc, MOYE_F64><<<g, 256, 0, st>>>(s, d, ls, ld, n, sb, db, mk); return true;
        default: return false;
    }
}

// (the instance that takes the index apart once where the layouts, the mask's too, have one shape and the groups are few
// enough for 32-bit indices: 8192^2 inside a pitch of 16384, f32 -> f16 5.0 -> 5.4 TB/s, f16 -> f32 4.2 -> 5.4, f16 -> bf16 4.7 -> 6.7)
template <int kSrc, int kDst, int SB, int DB, int V>
static void run_groups(const char* s, char* d, const FlatLayout& ls, const FlatLayout& ld, int64_t ngroups, int64_t run, const Mask& mk, hipStream_t st) {
    if (same_modes_32(ls, ld, ngroups) && (!mk.ptr || same_modes_32(ls, mk.l, ngroups)))
        copy_groups<kSrc, kDst, SB, DB, V, true><<<strided_grid(ngroups), 256, 0, st>>>(s, d, ls, ld, ngroups, run, mk);
    else
        copy_groups<kSrc, kDst, SB, DB, V, false><<<strided_grid(ngroups), 256, 0, st>>>(s, d, ls, ld, ngroups, run, mk);
}
template <int kSrc, int kDst, int SB, int DB>
static void launch_groups_pair(const char* s, char* d, const FlatLayout& ls, const FlatLayout& ld, int64_t ngroups, int64_t run, const Mask& mk, hipStream_t st) {
    constexpr int V = 16 / (SB > DB ? SB : DB);
    static_assert(V >= 2, "groups of at least two elements");
    run_groups<kSrc, kDst, SB, DB, V>(s, d, ls, ld, ngroups, run, mk, st);
}
template <int kSrc, int SB>
static bool launch_groups_dst(int32_t dd, const char* s, char* d, const FlatLayout& ls, const FlatLayout& ld, int64_t ng, int64_t run, const Mask& mk, hipStream_t st) {
    switch (dd) {
        case MOYE_F32: launch_groups_pair<kSrc, MOYE_F32, SB, 4>(s, d, ls, ld, ng, run, mk, st); return true;
        case MOYE_F16: launch_groups_pair<kSrc, MOYE_F16, SB, 2>(s, d, ls, ld, ng, run, mk, st); return true;
        case MOYE_BF16: launch_groups_pair<kSrc, MOYE_BF16, SB, 2>(s, d, ls, ld, ng, run, mk, st); return true;
        case MOYE_F8E4M3: launch_groups_pair<kSrc, MOYE_F8E4M3, SB, 1>(s, d, ls, ld, ng, run, mk, st); return true;
        case MOYE_F64: launch_groups_pair<kSrc, MOYE_F64, SB, 8>(s, d, ls, ld, ng, run, mk, st); return true;
        default: return false;
    }
}
// Do the bytes between the first and the last element of two arrays overlap?
static bool share_memory(const moye_tensor& x, const moye_tensor& y) {
    const char *first[2], *last[2];
    const moye_tensor* both[2] = {&x, &y};
    for (int i = 0; i < 2; ++i) {
        int64_t lo = 0, hi = 0;
        for (int m = 0; m < both[i]->rank; ++m) {
            const int64_t span = (both[i]->shape[m] - 1) * both[i]->stride[m];
            (span < 0 ? lo : hi) += span;
        }
        first[i] = static_cast<const char*>(both[i]->ptr) + lo * dtype_bytes(both[i]->dtype);
        last[i] = static_cast<const char*>(both[i]->ptr) + (hi + 1) * dtype_bytes(both[i]->dtype);
    }
    return first[0] < last[1] && first[1] < last[0];
}

// Groups of V = 16 / (the wider element) elements along the first mode, when every layout of the call (the modes already
// ordered by stride) has it as a run of unit stride and one length of V and more.  `same_bits`: a copy of bits (with a mask:
// copyto_if!); `in_place`: a conversion whose two sides share memory, which takes groups only where they end with the run, so that
// every element has one lane.  Returns false, having launched nothing, when the call does not qualify.
static bool launch_groups(int32_t src_dt, int32_t dst_dt, const char* s, char* d, FlatLayout ls, FlatLayout ld, Mask mk, bool same_bits, bool in_place,
                          int64_t n, hipStream_t st) {
    const int sb = dtype_bytes(src_dt), db = dtype_bytes(dst_dt);
    const int V = 16 / std::max(sb, db);
    if (V < 2 || ls.rank < 1 || ld.rank != ls.rank) return false;
    const int64_t run = ls.shape[0];
    if (run < V || (in_place && run % V) || ld.shape[0] != run || ls.stride[0] != 1 || ld.stride[0] != 1) return false;
    if (mk.ptr && (mk.l.rank != ls.rank || mk.l.shape[0] != run || mk.l.stride[0] != 1)) return false;
    const int64_t groups = (run + V - 1) / V, ng = n / run * groups;
    ls.shape[0] = ld.shape[0] = mk.l.shape[0] = groups;
    if (same_bits) {
        switch (sb) {
            case 1: run_groups<MOYE_U8, MOYE_U8, 1, 1, 16>(s, d, ls, ld, ng, run, mk, st); return true;
            case 2: run_groups<MOYE_U16, MOYE_U16, 2, 2, 8>(s, d, ls, ld, ng, run, mk, st); return true;
            case 4: run_groups<MOYE_U32, MOYE_U32, 4, 4, 4>(s, d, ls, ld, ng, run, mk, st); return true;
            case 8: run_groups<MOYE_U64, MOYE_U64, 8, 8, 2>(s, d, ls, ld, ng, run, mk, st); return true;
            default: return false;
        }
    }
    switch (src_dt) {
        case MOYE_F32: return launch_groups_dst<MOYE_F32, 4>(dst_dt, s, d, ls, ld, ng, run, mk, st);
        case MOYE_F16: return launch_groups_dst<MOYE_F16, 2>(dst_dt, s, d, ls, ld, ng, run, mk, st);
        case MOYE_BF16: return launch_groups_dst<MOYE_BF16, 2>(dst_dt, s, d, ls, ld, ng, run, mk, st);
        case MOYE_F8E4M3: return launch_groups_dst<MOYE_F8E4M3, 1>(dst_dt, s, d, ls, ld, ng, run, mk, st);
        case MOYE_F64: return launch_groups_dst<MOYE_F64, 8>(dst_dt, s, d, ls, ld, ng, run, mk, st);
        default: return false;
    }
}

int32_t copy_dispatch(const moye_tiled_copy* tc, const moye_tensor* dst, const moye_tensor* src,
                      hipStream_t st) {
    return copy_if_dispatch(tc, dst, src, nullptr, st);
}

// `mask` null: copyto!; else copyto_if! with a mask array of one byte per logical element (nonzero = move)
int32_t copy_if_dispatch(const moye_tiled_copy* tc, const moye_tensor* dst, const moye_tensor* src,
                         const moye_tensor* mask, hipStream_t st) {
    if (int32_t e = check_tensor(dst, "dst")) return e;
    if (int32_t e = check_tensor(src, "src")) return e;
    int64_t n = tensor_size(*src);
    Mask mk{};
    if (mask) {
        if (int32_t e = check_tensor(mask, "mask")) return e;
        if (dtype_bytes(mask->dtype) != 1 || is_float_dtype(mask->dtype))
            return fail(MOYE_ERR_UNSUPPORTED, "copyto_if!: the mask holds one byte per element (Bool), not %s", dtype_name(mask->dtype));
        if (tensor_size(*mask) != n)
            return fail(MOYE_ERR_SHAPE, "copyto_if!: mask holds %lld elements, src %lld", (long long)tensor_size(*mask), (long long)n);
        mk.ptr = static_cast<const uint8_t*>(mask->ptr);
        mk.l = flat_of(*mask);
    }
    if (tensor_size(*dst) != n)
        return fail(MOYE_ERR_SHAPE, "copyto!: dst holds %lld elements, src %lld",
                    (long long)tensor_size(*dst), (long long)n);
    const int sb = dtype_bytes(src->dtype), db = dtype_bytes(dst->dtype);
    if (n == 0) return MOYE_OK;
    const bool same_bits = (src->dtype == dst->dtype) || (sb == db && !is_float_dtype(src->dtype) && !is_float_dtype(dst->dtype));
    if (!same_bits && !(is_float_dtype(src->dtype) && is_float_dtype(dst->dtype)))
        return fail(MOYE_ERR_UNSUPPORTED, "copyto!: no conversion %s -> %s", dtype_name(src->dtype),
                    dtype_name(dst->dtype));
    if (tc) {
        if (tc->op != MOYE_COPY_UNIVERSAL && tc->op != MOYE_COPY_LDS_TILED)
            return fail(MOYE_ERR_UNSUPPORTED, "copyto!: unknown copy op %d", tc->op);
        if (tc->vec_bits && (tc->vec_bits % 8 || tc->vec_bits > 128 || (tc->vec_bits & (tc->vec_bits - 1))))
            return fail(MOYE_ERR_ARG, "copyto!: vec_bits %d is not one of 8..128", tc->vec_bits);
        if (tc->vec_bits && tc->vec_bits % (8 * sb))
            return fail(MOYE_ERR_SHAPE, "copyto!: a %d-bit access does not hold whole %s values", tc->vec_bits,
                        dtype_name(src->dtype));
    }
    const char* s = static_cast<const char*>(src->ptr);
    char* d = static_cast<char*>(dst->ptr);

    // Arrays of one shape of rank three and more: modes of extent 1 go, and modes that are neighbours in memory on both
    // sides become one, whichever order the caller wrote them in (NCHW -> NHWC: H and W; [B,S,H,D] -> [B,H,D,S]: H and D), so that
    // what follows sees a matrix or a batch of matrices where there is one, with its longest rows (the tiler of the descriptor
    // speaks of the caller's modes: it is checked here, then dropped).  us, only modes written smallest stride first / any: f32 NCHW
    // -> NHWC 16 x 512 x 28 x 28 45.1 / 12.5, f16 NHWC -> NCHW 55 x 14 x 14 x 128 12.3 / 4.2, f16 [4,2000,32,128] -> [4,32,128,2000] 28.7 / 27.4.
    if (!mask && src->rank == dst->rank && src->rank > 2) {
        bool same = true;
        for (int m = 0; m < src->rank; ++m) same = same && src->shape[m] == dst->shape[m];
        int at[MOYE_MAX_RANK], left = 0;
        for (int m = 0; same && m < src->rank; ++m)
            if (src->shape[m] != 1) at[left++] = m;
        std::stable_sort(at, at + left, [&](int x, int y) { return dst->stride[x] != dst->stride[y] ? dst->stride[x] < dst->stride[y] : src->stride[x] < src->stride[y]; });
        moye_tensor cs = *src, cd = *dst;
        int r = 0;
        for (int q = 0; q < left; ++q) {
            const int m = at[q];
            if (r > 0 && src->stride[m] == cs.stride[r - 1] * cs.shape[r - 1] && dst->stride[m] == cd.stride[r - 1] * cd.shape[r - 1]) {
                cs.shape[r - 1] *= src->shape[m];
                cd.shape[r - 1] = cs.shape[r - 1];
            } else {
                cs.shape[r] = cd.shape[r] = src->shape[m];
                cs.stride[r] = src->stride[m];
                cd.stride[r] = dst->stride[m];
                ++r;
            }
        }
        if (same && r >= 1 && r < src->rank) {
            moye_tiled_copy plain{};
            if (tc) {
                if (tc->op == MOYE_COPY_LDS_TILED)
                    for (int m = 0; m < 2; ++m)
                        if (tc->tiler_mn[m] < 0 || (tc->tiler_mn[m] > 0 && src->shape[m] % tc->tiler_mn[m]))
                            return fail(MOYE_ERR_SHAPE, "copyto!: tiler extent %d does not divide mode %d of size %lld", tc->tiler_mn[m], m + 1,
                                        (long long)src->shape[m]);
                plain = *tc;
                plain.tiler_mn[0] = plain.tiler_mn[1] = 0;
            }
            cs.rank = cd.rank = r;
            return copy_if_dispatch(tc ? &plain : nullptr, &cd, &cs, nullptr, st);
        }
    }
    if (same_bits && !mask) {
        // (1) both sides one dense run in the same order
        if (one_run_each(*src, *dst)) {
            const int64_t bytes = n * sb;
            if (bytes % 16 == 0 && (reinterpret_cast<uintptr_t>(s) | reinterpret_cast<uintptr_t>(d)) % 16 == 0) {
                const int64_t n16 = bytes / 16;
                copy_flat_b128<<<flat_grid(n16), 256, 0, st>>>(reinterpret_cast<const u32x4*>(s), reinterpret_cast<u32x4*>(d), n16);
            } else if (bytes >= 16) {
                copy_flat_any<<<flat_grid((bytes + 15) / 16), 256, 0, st>>>(s, d, bytes);
            } else {
                const int blocks = (int)std::min<int64_t>((bytes + 255) / 256, 256 * 32);
                copy_flat_bytes<<<blocks, 256, 0, st>>>(reinterpret_cast<const uint8_t*>(s), reinterpret_cast<uint8_t*>(d), bytes);
            }
            MOYE_HIP_CHECK(hipGetLastError());
            return MOYE_OK;
        }
        // (2) the unit strides on different modes: a transpose, or a batch of them.
        // The tiler of the descriptor (tiler_MN of make_tiled_copy, src/atom/copy.jl:249-258; 32 x 32 in the reference's own
        // transpose kernel, test/host/copy_async.jl:51-76) must divide the array, as zipped_divide asserts; how the kernels
        // group elements into LDS tiles is their own business and changes no result.
        if (tc && tc->op == MOYE_COPY_LDS_TILED && src->rank >= 2) {
            for (int m = 0; m < 2; ++m)
                if (tc->tiler_mn[m] < 0 || (tc->tiler_mn[m] > 0 && src->shape[m] % tc->tiler_mn[m]))
                    return fail(MOYE_ERR_SHAPE, "copyto!: tiler extent %d does not divide mode %d of size %lld", tc->tiler_mn[m], m + 1,
                                (long long)src->shape[m]);
        }
        TransposeArgs ta;
        const bool lds_batch = tc && tc->op == MOYE_COPY_LDS_TILED && src->rank > 2;  // (a batch has no other kernel under that op)
        if (transpose_plan(*src, *dst, true, &ta) && (lds_batch || transpose_pays(src->dtype, dst->dtype, ta)))
            return transpose_run(src->dtype, dst->dtype, true, tc && (tc->flags & MOYE_GEMM_NO_LDS_SWIZZLE), device_shape().xcds, ta, st);
        // a pair the LDS-tiled op is meant for, but with too few elements along a side: the general kernel moves it
        const bool lds_pair = sb <= 8 && src->rank == 2 && dst->rank == 2 && src->shape[0] == dst->shape[0] && src->shape[1] == dst->shape[1] &&
                              ((src->stride[0] == 1 && dst->stride[1] == 1) || (src->stride[1] == 1 && dst->stride[0] == 1));
        if (tc && tc->op == MOYE_COPY_LDS_TILED && !lds_pair)
            return fail(MOYE_ERR_UNSUPPORTED,
                        "copyto!: the LDS-tiled copy takes rank-2 operands (or a batch of them) of 1- to 8-byte elements "
                        "with the unit stride on different modes");
    }

    // (2b) the same with a conversion on the way
    if (!same_bits && !mask && !(tc && tc->op == MOYE_COPY_LDS_TILED && (tc->tiler_mn[0] || tc->tiler_mn[1]))) {
        TransposeArgs ta;
        if (transpose_plan(*src, *dst, false, &ta) && transpose_pays(src->dtype, dst->dtype, ta))
            return transpose_run(src->dtype, dst->dtype, false, false, device_shape().xcds, ta, st);
    }

    // (3) generic
    FlatLayout ls = flat_of(*src), ld = flat_of(*dst);
    // same shape mode by mode: visit the coordinates along the destination's smallest strides first (then the source's)
    {
        FlatLayout* all[3] = {&ld, &ls, mask ? &mk.l : nullptr};
        order_modes_by_stride(all, mask ? 3 : 2);
    }
    if (same_bits && !mask) {
        // Vectorise when the layouts allow it, which the reference computes (max_common_vector,
        // src/layout.jl:752-761) and then leaves unused (src/algorithm/copy.jl:53-58): if logical
        // neighbours are memory neighbours on both sides in runs of v elements, and every other stride
        // and both pointers are multiples of v, both layouts are recast to elements of v * sizeof(T)
        // bytes (the upcast of src/layout.jl:945-975 on flattened modes) and moved 4..16 bytes at a time.
        const auto run = [](const FlatLayout& l) { return l.rank >= 1 && l.stride[0] == 1 ? l.shape[0] : 1; };
        int64_t v = std::min(run(ls), run(ld));
        // logical index i -> mode-0 coordinate i % shape[0] on each side: the runs must line up
        if (ls.shape[0] != ld.shape[0]) v = std::__gcd(std::__gcd(ls.shape[0], ld.shape[0]), v);
        int64_t width = 16 / sb;  // widest access in elements
        while (width > 1) {
            bool fits = v % width == 0 && reinterpret_cast<uintptr_t>(s) % (width * sb) == 0 &&
                        reinterpret_cast<uintptr_t>(d) % (width * sb) == 0;
            for (int m = 1; m < MOYE_MAX_RANK && fits; ++m)
                fits = (ls.shape[m] == 1 || ls.stride[m] % width == 0) && (ld.shape[m] == 1 || ld.stride[m] % width == 0);
            if (fits) break;
            width /= 2;
        }
        // (under 8 bytes at a time: runs in groups that need no alignment, where the layouts have runs)
        if (sb * width < 8 && launch_groups(src->dtype, dst->dtype, s, d, ls, ld, mk, true, false, n, st)) {
            MOYE_HIP_CHECK(hipGetLastError());
            return MOYE_OK;
        }
        if (width > 1 && sb * width <= 16) {
            for (FlatLayout* l : {&ls, &ld}) {
                l->shape[0] /= width;
                for (int m = 1; m < MOYE_MAX_RANK; ++m) l->stride[m] /= width;
            }
            const int64_t nv = n / width;
            if (same_modes_32(ls, ld, nv)) {
                switch (sb * width) {
                    case 2: launch_generic_bits_same<2>(s, d, ls, ld, nv, st); break;
                    case 4: launch_generic_bits_same<4>(s, d, ls, ld, nv, st); break;
                    case 8: launch_generic_bits_same<8>(s, d, ls, ld, nv, st); break;
                    default: launch_generic_bits_same<16>(s, d, ls, ld, nv, st); break;
                }
                MOYE_HIP_CHECK(hipGetLastError());
                return MOYE_OK;
            }
            const dim3 gv = strided_grid(nv);  // one piece per lane up to 16 GiB of 16-byte pieces
            switch (sb * width) {
                case 2: copy_generic_bits<2><<<gv, 256, 0, st>>>(s, d, ls, ld, nv, Mask{}); break;
                case 4: copy_generic_bits<4><<<gv, 256, 0, st>>>(s, d, ls, ld, nv, Mask{}); break;
                case 8: copy_generic_bits<8><<<gv, 256, 0, st>>>(s, d, ls, ld, nv, Mask{}); break;
                default: copy_generic_bits<16><<<gv, 256, 0, st>>>(s, d, ls, ld, nv, Mask{}); break;
            }
            MOYE_HIP_CHECK(hipGetLastError());
            return MOYE_OK;
        }
    }
    // (up to 64 MiB a run that does not end with a group: in groups below, which leave no rest for a second launch; f32 -> bf16 1301 x 1333 6.3 ->
    // 3.9 us)
    const int64_t per_lane = 16 / std::min(sb, db);
    const bool in_place = !same_bits && share_memory(*src, *dst);
    if (!same_bits && !mask && one_run_each(*src, *dst) && (n % per_lane == 0 || in_place || n * std::max(sb, db) > ((int64_t)64 << 20)) &&
        (reinterpret_cast<uintptr_t>(s) | reinterpret_cast<uintptr_t>(d)) % 16 == 0) {
        // both sides one aligned run: 16-byte accesses for all whole groups, the general kernel for what is left
        const int64_t done = launch_cvt_dense(src->dtype, dst->dtype, s, d, n, st);
        if (done > 0) {
            MOYE_HIP_CHECK(hipGetLastError());
            if (done == n) return MOYE_OK;
            s += done * sb;
            d += done * db;
            n -= done;
            for (FlatLayout* l : {&ls, &ld}) {
                l->rank = 1;
                for (int m = 0; m < MOYE_MAX_RANK; ++m) { l->shape[m] = 1; l->stride[m] = 0; }
                l->shape[0] = n;
                l->stride[0] = 1;
            }
        }
    }
    // converting copies between pitched arrays, and copyto_if!: groups of elements along the first mode where the layouts allow
    // (a plain copy of bits has had its turn above)
    if ((!same_bits || mask) && launch_groups(src->dtype, dst->dtype, s, d, ls, ld, mk, same_bits, in_place, n, st)) {
        MOYE_HIP_CHECK(hipGetLastError());
        return MOYE_OK;
    }
    const dim3 g((unsigned)std::min<int64_t>((n + 255) / 256, 256 * 64));
    bool ok = true;
    if (same_bits) {
        switch (sb) {
            case 1: copy_generic_bits<1><<<g, 256, 0, st>>>(s, d, ls, ld, n, mk); break;
            case 2: copy_generic_bits<2><<<g, 256, 0, st>>>(s, d, ls, ld, n, mk); break;
            case 4: copy_generic_bits<4><<<g, 256, 0, st>>>(s, d, ls, ld, n, mk); break;
            case 8: copy_generic_bits<8><<<g, 256, 0, st>>>(s, d, ls, ld, n, mk); break;
            case 16: copy_generic_bits<16><<<g, 256, 0, st>>>(s, d, ls, ld, n, mk); break;
            default: ok = false;
        }
    } else {
        switch (src->dtype) {
            case MOYE_F32: ok = launch_cvt_dst<MOYE_F32>(dst->dtype, g, st, s, d, ls, ld, n, sb, db, mk); break;
            case MOYE_F16: ok = launch_cvt_dst<MOYE_F16>(dst->dtype, g, st, s, d, ls, ld, n, sb, db, mk); break;
            case MOYE_BF16: ok = launch_cvt_dst<MOYE_BF16>(dst->dtype, g, st, s, d, ls, ld, n, sb, db, mk); break;
            case MOYE_F8E4M3: ok = launch_cvt_dst<MOYE_F8E4M3>(dst->dtype, g, st, s, d, ls, ld, n, sb, db, mk); break;
            case MOYE_F64: ok = launch_cvt_dst<MOYE_F64>(dst->dtype, g, st, s, d, ls, ld, n, sb, db, mk); break;
            default: ok = false;
        }
    }
    if (!ok) return fail(MOYE_ERR_UNSUPPORTED, "copyto!: no kernel for %s -> %s", dtype_name(src->dtype), dtype_name(dst->dtype));
    MOYE_HIP_CHECK(hipGetLastError());
    return MOYE_OK;
}

}  // namespace moye
