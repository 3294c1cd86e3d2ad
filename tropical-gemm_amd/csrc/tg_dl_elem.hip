// tg_dl_elem.hip -- launches of tg_gemm_dl with element loads.
#include "tg_dl_elem.hpp"

#include "../../include/tropical_gemm_hip.h"
#include "tg_gemm_dl.hpp"

namespace tg {
namespace {

template <int SR, typename T, bool ARGMAX, int CL, int HALVES>
hipError_t launch(const DlElemProblem& p, hipStream_t st) {
    using Cfg = DlCfg<4, 4>;
    const auto kernel = &tg_gemm_dl<SR, T, ARGMAX, 4, 4, CL, true, false, 0, HALVES, true>;
    constexpr int lds = HALVES * (ARGMAX ? Cfg::LDS_BYTES : Cfg::TILE_BYTES);
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    const int64_t tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    // Slices are whole k-tiles.
    const int64_t nkt = (p.K + Cfg::BK - 1) / Cfg::BK;
    const int64_t KS = HALVES > 1 ? (nkt + HALVES - 1) / HALVES * Cfg::BK : p.K;
    for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
        const int64_t nb = p.batch - z0 < 65535 ? p.batch - z0 : 65535;
        hipLaunchKernelGGL(kernel, dim3(unsigned(tiles_m * tiles_n), 1, unsigned(nb)),
                           dim3(TG_THREADS * HALVES), lds, st, static_cast<const T*>(p.A) + z0 * p.sA,
                           static_cast<const T*>(p.B) + z0 * p.sB,
                           ARGMAX ? static_cast<const T*>(p.BT) + z0 * p.K * p.N : nullptr,
                           static_cast<T*>(p.C) + z0 * p.sC, ARGMAX ? p.IDX + z0 * p.sC : nullptr,
                           p.M, p.N, p.K, p.sA, p.sB, p.sC, int(tiles_m), int(tiles_n), KS, int64_t(0));
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int SR, typename T>
hipError_t launch_typed(const DlElemProblem& p, int cl, int slices, hipStream_t st) {
    if (p.IDX != nullptr) {
        if (slices == 4) return launch<SR, T, true, 8, 4>(p, st);
        if (slices == 2) return launch<SR, T, true, 8, 2>(p, st);
        return cl == 8 ? launch<SR, T, true, 8, 1>(p, st) : launch<SR, T, true, 16, 1>(p, st);
    }
    if (slices == 4) return launch<SR, T, false, 32, 4>(p, st);
    if (slices == 2) return launch<SR, T, false, 32, 2>(p, st);
    return launch<SR, T, false, 32, 1>(p, st);
}

template <int SR>
hipError_t launch_sr(const DlElemProblem& p, int cl, int slices, hipStream_t st) {
    return p.f32 ? launch_typed<SR, float>(p, cl, slices, st)
                 : launch_typed<SR, int32_t>(p, cl, slices, st);
}

}  // namespace

// Measured on MI355X (us, f32, with 1 / 2 / 4 slices): argmax 1001^3 (256
// tiles) 111 / 78 / 76, 734 x 1071 x 3636 (204) 311 / 195 / 180, 1021^2 x 300
// 46 / 36 / 39, 544 x 2755 x 896 (396) 111 / 99 / 123, 1300^3 (441) 140 / 134 /
// 161, 1500^2 x 515 (576) 97 / 99 / 131; value-only 1001^3 81 / 48 / 45,
// 1300^3 109 / 94 / 107, 1700^3 (729) 206 / 189 / 210, 2001^2 x 1000 (1024) 159 /
// 149 / 175.
int dl_elem_slices(int64_t tiles, int64_t K, bool argmax) {
    if (K < 256 || K > (int64_t(1) << 19)) return 1;  // 16-bit slots hold chunks of 8
    if (argmax) return tiles <= 256 ? (K >= 1024 ? 4 : 2) : tiles <= 512 ? 2 : 1;
    return tiles <= 256 ? 4 : tiles <= 1024 ? 2 : 1;
}

hipError_t dl_elem_launch(const DlElemProblem& p, int cl, int slices, hipStream_t st) {
    switch (p.sr) {
        case TG_MAXPLUS: return launch_sr<SR_MAXPLUS>(p, cl, slices, st);
        case TG_MINPLUS: return launch_sr<SR_MINPLUS>(p, cl, slices, st);
        default: return launch_sr<SR_MAXMUL>(p, cl, slices, st);
    }
}

}  // namespace tg
