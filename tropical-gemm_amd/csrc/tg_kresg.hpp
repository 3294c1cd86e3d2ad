// tg_kresg.hpp -- host interface of tg_gemm_kresg (i32 MaxPlus/MinPlus argmax
// at short K), which is compiled in a file of its own (tg_kresg.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tg {

// Row-major i32 problem with argmax; sr 0 (MaxPlus) or 1 (MinPlus).
struct KresgProblem {
    int sr;
    const int32_t *A, *B;
    int32_t *C, *IDX;
    int64_t batch, M, N, K, sA, sB, sC;
};

// True when the kernel can run these sizes.
bool kresg_fits(int64_t M, int64_t N, int64_t K);

// 16 x 64 wave tiles of one batch item.
int64_t kresg_wave_tiles(int64_t M, int64_t N);

hipError_t kresg_launch(const KresgProblem& p, int cus, hipStream_t st);

}  // namespace tg
