// tg_small.hpp -- host interface of the few-output kernel (tg_gemm_small.hpp),
// which is compiled in a file of its own (tg_small.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tg {

// Row-major problem of one dtype (0 f32, 1 f64, 2 i32, 3 i64).
struct SmallProblem {
    int sr, dtype;
    const void *A, *B;
    void* C;
    int32_t* IDX;
    int64_t batch, M, N, K, sA, sB, sC;
};

// Lanes down the rows and across the columns of a tile (4 x 4 outputs per
// lane), and waves per workgroup.
struct SmallForm {
    int lr, lc, waves;
};

// True when the kernel can run the problem; then `form` is the launch to use.
bool small_form(const SmallProblem& p, SmallForm* form);

hipError_t small_launch(const SmallProblem& p, const SmallForm& form, hipStream_t st);

}  // namespace tg
