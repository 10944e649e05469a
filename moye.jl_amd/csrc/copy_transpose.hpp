// A transpose, or a batch of them, as copy_transpose.hip takes it.
#pragma once

#include "moye_common.hpp"

namespace moye {

struct TransposeArgs {
    const char* src;
    char* dst;
    int64_t lds, ldd;   // pitches in elements: of the source's rows (along j), of the destination's (along i)
    int32_t ni, nj;     // extents of the source's and of the destination's contiguous index
    int32_t tiles_i, tiles_j;
    int32_t band;       // 0: the tiles of a destination row one after the other; else bands of so many tile columns
    int32_t xcds, run;  // neighbouring tiles that go to one XCD
    int32_t linear;     // LDS rows as they come (for a study of bank conflicts)
    uint32_t batch;     // product of the extents of the modes that count matrices
    int32_t modes;
    uint32_t extent[MOYE_MAX_RANK];
    int64_t s_stride[MOYE_MAX_RANK], d_stride[MOYE_MAX_RANK];  // in elements
};

// Is this copy one (arrays of one shape, mode by mode, the unit strides on different modes of 32 and more elements)?
bool transpose_plan(const moye_tensor& src, const moye_tensor& dst, bool same_bits, TransposeArgs* a);
// Does it pay (against the general kernel, element by element)?
bool transpose_pays(int32_t src_dt, int32_t dst_dt, const TransposeArgs& a);
int32_t transpose_run(int32_t src_dt, int32_t dst_dt, bool same_bits, bool linear_lds, int xcds, TransposeArgs a, hipStream_t st);

}  // namespace moye
