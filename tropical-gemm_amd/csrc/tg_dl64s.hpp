// tg_dl64s.hpp -- host interface of tg_gemm_dl64s (64-bit types on 64 x 64
// tiles), which is compiled in a file of its own (tg_dl64s.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tg {

// Row-major problem, f64 or i64.  BT (argmax): dense B^T; clsA / clsB (f64):
// operand classes per row of A and column of B (batch x M, batch x N).
struct Dl64sProblem {
    int sr;
    bool f64;
    const void *A, *B, *BT;
    void* C;
    int32_t* IDX;
    const uint32_t *clsA, *clsB;
    int64_t batch, M, N, K, sA, sB, sC;
};

// True when the kernel can run these sizes (32-bit lane offsets, 16-bit chunk
// slots, one launch).
bool dl64s_fits(int64_t M, int64_t N, int64_t K);

// 16-byte loads (otherwise element loads): K and N even, 16-byte aligned
// operands, even batch strides.
inline bool dl64s_vectors(int64_t N, int64_t K, int64_t sA, int64_t sB, const void* A, const void* B) {
    auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    return K % 2 == 0 && N % 2 == 0 && sA % 2 == 0 && sB % 2 == 0 && a16(A) && a16(B);
}

// K slices per workgroup for `tiles` 64 x 64 tiles.
int dl64s_slices(int64_t tiles, bool argmax);

hipError_t dl64s_launch(const Dl64sProblem& p, hipStream_t st);

}  // namespace tg
