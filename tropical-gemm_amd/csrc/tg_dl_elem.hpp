// tg_dl_elem.hpp -- host interface of the element-load instantiations of
// tg_gemm_dl (32-bit types, any alignment), compiled in a file of their own
// (tg_dl_elem.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tg {

// Row-major problem, f32 or i32.  BT (argmax): dense B^T.
struct DlElemProblem {
    int sr;
    bool f32;
    const void *A, *B, *BT;
    void* C;
    int32_t* IDX;
    int64_t batch, M, N, K, sA, sB, sC;
};

// K slices per workgroup for `tiles` 64 x 64 tiles (1, 2 or 4).
int dl_elem_slices(int64_t tiles, int64_t K, bool argmax);

// cl: argmax chunk length, 8 or 16 (slices > 1: 8).
hipError_t dl_elem_launch(const DlElemProblem& p, int cl, int slices, hipStream_t st);

}  // namespace tg
