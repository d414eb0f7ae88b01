// Blocked history sums in FP64 (frm_blockhist.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace frm {

// Steps that share one pass over the settled history.  A block starts at a
// multiple N0 of it; its steps n = N0 + j take the slots before N0 from the
// block's far sums and the at most kHistBlock - 1 newer ones themselves.
constexpr int kHistBlock = 16;
// The same for sums kept in FP32.
constexpr int kMidBlock = 8;

// G[(t*kHistBlock + j)*ld + i] = sum_{s < N0} w[t*ldw + N0 + j - s - 1] Delta_s[i]
// for t < 2, j < kHistBlock and the ld nodes of the store (ld a multiple of
// 1024, N0 > 0 a multiple of kHistBlock).  Slots before `first` are left out:
// the caller's weights are zero there.  w is lag-indexed (w[0] for lag 1) and
// readable up to lag N0 + kHistBlock - 1, ldw >= N0 + kHistBlock - 1.
// An FP32 G rounds the FP64 sums once and has kMidBlock steps in kHistBlock's place.
// Returns nonzero on arguments outside these bounds or a failed launch.
int hist_far(hipStream_t st, const double* hist, int64_t ld, int first, int N0, const double* w,
             int ldw, double* G);
int hist_far(hipStream_t st, const float* hist, int64_t ld, int first, int N0, const double* w,
             int ldw, double* G);
int hist_far(hipStream_t st, const float* hist, int64_t ld, int first, int N0, const double* w,
             int ldw, float* G);

}  // namespace frm
