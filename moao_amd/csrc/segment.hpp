// Y L = X over the columns of two to four whole leaves in one launch (see segment.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace moao {

constexpr int kSegGroups = 8;  // row groups per launch
constexpr int kSegment = 512;  // most columns

// Rows of X, in place: rows x nn at X (first column of the segment), leading dimension ld.
template <typename T>
struct SegRows {
    T* X;
    long ld;
    int rows;
    // FP32, optional: the split-BF16 planes of the result (gemm.hpp's Planes), column 0 at cp
    unsigned short* cp;
    long cpld, cpps;
};

// L: the segment's diagonal block of the factor (leading dimension lda, lower triangle), inv: the
// inverses of its leaves, kLeaf x kLeaf each; nn a multiple of kLeaf, kLeaf < nn <= kSegment.
// A no-op where *skip_if is set.
template <typename T>
int trsm_segment(const SegRows<T>* rows, int ngroups, const T* L, long lda, const T* inv, int nn,
                 const int* skip_if, hipStream_t s);

}  // namespace moao
