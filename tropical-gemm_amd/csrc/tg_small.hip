// tg_small.hip -- launch rules and launches of tg_gemm_small.
#include "tg_gemm_small.hpp"

#include "../../include/tropical_gemm_hip.h"

namespace tg {
namespace {

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

int64_t small_tiles(const SmallProblem& p, int lr, int lc) {
    return ceil_div(p.M, 4 * lr) * ceil_div(p.N, 4 * lc);
}

// Tile and split of K.  Measured on MI355X over 140 shapes of every dtype,
// with and without argmax, against the best of all tiles and wave counts:
// 4% off it in the mean.  The largest tile that still makes about one
// workgroup per SIMD pair (loads shared by more products), less than 30% of
// it wasted at the edges; 32 x 32 only for short K, where its 128-byte output
// rows count (2001 x 2001 x 60 f32: 22 us against 36 for 16 x 16) and the
// k loop does not.
void choose_form(const SmallProblem& p, int kv, int max_waves, SmallForm* f) {
    if (p.N < 4) {
        *f = {4, 1, 1};
    } else {
        static constexpr int forms[4][3] = {{8, 8, 512}, {4, 4, 768}, {2, 4, 384}, {1, 4, 0}};
        double use[4], best = 0;
        for (int i = 0; i < 4; ++i) {
            use[i] = double(p.M) * double(p.N) /
                     (double(small_tiles(p, forms[i][0], forms[i][1])) * 16 * forms[i][0] * forms[i][1]);
            if (use[i] > best) best = use[i];
        }
        *f = {1, 4, 1};
        for (int i = p.K <= 128 ? 0 : 1; i < 4; ++i) {
            if (use[i] < 0.7 * best) continue;
            if (small_tiles(p, forms[i][0], forms[i][1]) * p.batch < forms[i][2]) continue;
            *f = {forms[i][0], forms[i][1], 1};
            break;
        }
    }
    // Waves of a workgroup: up to 2048 in all, each with at least one step;
    // beyond that up to four while a wave keeps eight steps (its waves then
    // share the tile's operand lines in L1: 900^3 f64 with argmax on 16 x 16
    // tiles 155 us with four waves, 214 with one).
    const int64_t tiles = small_tiles(p, f->lr, f->lc) * p.batch;
    const int64_t steps = ceil_div(p.K, int64_t(64 / (f->lr * f->lc)) * kv);
    int w = 1;
    while (w * 2 <= max_waves && w * 2 <= steps &&
           (tiles * w <= 1024 || (w < 4 && steps >= int64_t(8) * w)))
        w *= 2;
    f->waves = w;
}

template <int SR, typename T, bool ARGMAX, int LR, int LC, bool NCLAMP>
hipError_t launch(const SmallProblem& p, int waves, hipStream_t st) {
    using Cfg = SmallCfg<T, LR, LC>;
    const auto kernel = &tg_gemm_small<SR, T, ARGMAX, LR, LC, NCLAMP>;
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
        Cfg::lds_bytes(Cfg::MAX_WAVES, ARGMAX));
    if (attr != hipSuccess) return attr;
    const int tiles_m = int(ceil_div(p.M, Cfg::BM)), tiles_n = int(ceil_div(p.N, Cfg::BN));
    for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
        const int64_t nb = p.batch - z0 < 65535 ? p.batch - z0 : 65535;
        hipLaunchKernelGGL(kernel, dim3(unsigned(int64_t(tiles_m) * tiles_n), 1, unsigned(nb)),
                           dim3(64 * waves), Cfg::lds_bytes(waves, ARGMAX), st,
                           static_cast<const T*>(p.A) + z0 * p.sA,
                           static_cast<const T*>(p.B) + z0 * p.sB, static_cast<T*>(p.C) + z0 * p.sC,
                           ARGMAX ? p.IDX + z0 * p.sC : nullptr, p.M, p.N, p.K, p.sA, p.sB, p.sC,
                           tiles_m, tiles_n);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int SR, typename T, bool ARGMAX>
hipError_t launch_form(const SmallProblem& p, const SmallForm& f, hipStream_t st) {
    if (f.lc == 8) return launch<SR, T, ARGMAX, 8, 8, false>(p, f.waves, st);
    if (f.lc == 1) return launch<SR, T, ARGMAX, 4, 1, true>(p, f.waves, st);
    switch (f.lr) {
        case 4: return launch<SR, T, ARGMAX, 4, 4, false>(p, f.waves, st);
        case 2: return launch<SR, T, ARGMAX, 2, 4, false>(p, f.waves, st);
        default: return launch<SR, T, ARGMAX, 1, 4, false>(p, f.waves, st);
    }
}

template <int SR, typename T>
hipError_t launch_typed(const SmallProblem& p, const SmallForm& f, hipStream_t st) {
    return p.IDX != nullptr ? launch_form<SR, T, true>(p, f, st) : launch_form<SR, T, false>(p, f, st);
}

template <int SR>
hipError_t launch_sr(const SmallProblem& p, const SmallForm& f, hipStream_t st) {
    switch (p.dtype) {
        case TG_F32: return launch_typed<SR, float>(p, f, st);
        case TG_F64: return launch_typed<SR, double>(p, f, st);
        case TG_I32: return launch_typed<SR, int32_t>(p, f, st);
        default: return launch_typed<SR, int64_t>(p, f, st);
    }
}

}  // namespace

bool small_form(const SmallProblem& p, SmallForm* form) {
    const bool wide = p.dtype == TG_F64 || p.dtype == TG_I64;
    if (p.M <= 0 || p.N <= 0 || p.K <= 0 || p.batch <= 0) return false;
    // 32-bit element offsets inside a matrix, and K as the other kernels
    // with argmax bound it.
    constexpr int64_t kMaxElems = int64_t(1) << 31;
    if (p.M * p.K >= kMaxElems || p.K * p.N >= kMaxElems || p.K > int64_t(65535) * 32) return false;
    choose_form(p, wide ? 2 : 4, wide ? small_max_waves<double>() : small_max_waves<float>(), form);
    // The launch's thread count per dimension stays below 2^32.
    return small_tiles(p, form->lr, form->lc) < (int64_t(1) << 22);
}

hipError_t small_launch(const SmallProblem& p, const SmallForm& form, hipStream_t st) {
    switch (p.sr) {
        case TG_MAXPLUS: return launch_sr<SR_MAXPLUS>(p, form, st);
        case TG_MINPLUS: return launch_sr<SR_MINPLUS>(p, form, st);
        default: return launch_sr<SR_MAXMUL>(p, form, st);
    }
}

}  // namespace tg
