// tg_elem_rows.hpp -- the k rows of B that the element loads read
// (tg_gemm_dl with ELEM, tg_gemm_dl64s with ELEM).
//
// A wave loads consecutive k rows of a k-tile through one pointer that steps
// from row to row.  In the last k-tile only `left` rows exist: a wave whose
// first row lies past them starts at the last one, and the pointer never steps
// past it, so every read stays inside B (the rows read twice are overwritten in
// LDS).  Plain C++, so that the rule can be replayed on the host: the results
// do not show a row read past the end.
#pragma once

#ifdef __HIPCC__
#define TG_HOST_DEVICE __host__ __device__
#else
#define TG_HOST_DEVICE
#endif

namespace tg {

// Row at which a wave whose first row is `row` starts.
TG_HOST_DEVICE constexpr int elem_first_row(int row, int left) {
    return row < left ? row : left - 1;
}

// Whether the pointer steps on after row `row` of the wave's rows.
TG_HOST_DEVICE constexpr bool elem_steps(int row, int left) { return row + 1 < left; }

}  // namespace tg
