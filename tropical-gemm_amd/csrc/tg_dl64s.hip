// tg_dl64s.hip -- launches of tg_gemm_dl64s.
#include "tg_dl64s.hpp"

#include "../../include/tropical_gemm_hip.h"
#include "tg_gemm_dl64s.hpp"

namespace tg {
namespace {

template <int SR, typename T, bool ARGMAX, int HALVES, bool ELEM>
hipError_t launch(const Dl64sProblem& p, hipStream_t st) {
    using Cfg = Dl64sCfg;
    const auto kernel = &tg_gemm_dl64s<SR, T, ARGMAX, HALVES, ELEM>;
    constexpr int lds = HALVES * Cfg::LDS_BYTES;
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return attr;
    const int64_t tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
        const int64_t nb = p.batch - z0 < 65535 ? p.batch - z0 : 65535;
        hipLaunchKernelGGL(kernel, dim3(unsigned(tiles_m * tiles_n), 1, unsigned(nb)),
                           dim3(TG_THREADS * HALVES), lds, st, static_cast<const T*>(p.A) + z0 * p.sA,
                           static_cast<const T*>(p.B) + z0 * p.sB,
                           ARGMAX ? static_cast<const T*>(p.BT) + z0 * p.K * p.N : nullptr,
                           static_cast<T*>(p.C) + z0 * p.sC, ARGMAX ? p.IDX + z0 * p.sC : nullptr,
                           p.f64 ? p.clsA + z0 * p.M : nullptr, p.f64 ? p.clsB + z0 * p.N : nullptr,
                           p.M, p.N, p.K, p.sA, p.sB, p.sC, int(tiles_m), int(tiles_n));
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int SR, typename T, bool ELEM>
hipError_t launch_slices(const Dl64sProblem& p, hipStream_t st) {
    const int64_t tiles = ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch;
    if (p.IDX != nullptr) {
        if (dl64s_slices(tiles, true) == 3) return launch<SR, T, true, 3, ELEM>(p, st);
        return launch<SR, T, true, 1, ELEM>(p, st);
    }
    if (dl64s_slices(tiles, false) == 4) return launch<SR, T, false, 4, ELEM>(p, st);
    return launch<SR, T, false, 2, ELEM>(p, st);
}

template <int SR, typename T>
hipError_t launch_typed(const Dl64sProblem& p, hipStream_t st) {
    return dl64s_vectors(p.N, p.K, p.sA, p.sB, p.A, p.B) ? launch_slices<SR, T, false>(p, st)
                                                         : launch_slices<SR, T, true>(p, st);
}

}  // namespace

bool dl64s_fits(int64_t M, int64_t N, int64_t K) {
    return M > 0 && N >= 2 && K >= 2 && (K + Dl64sCfg::CL - 1) / Dl64sCfg::CL < 0xFFFF &&
           K < (int64_t(1) << 23) && N < (int64_t(1) << 27) &&
           ((M + 63) / 64) * ((N + 63) / 64) < (int64_t(1) << 22);
}

// As many slices as the registers allow while the tiles do not give every CU
// one; beyond that argmax workgroups (three per CU) overlap each other's
// epilogues, and value-only ones run two slices (measured in the kernel's header).
int dl64s_slices(int64_t tiles, bool argmax) {
    constexpr int64_t kCus = 256;
    if (argmax) return tiles <= kCus ? 3 : 1;
    return tiles <= kCus ? 4 : 2;
}

hipError_t dl64s_launch(const Dl64sProblem& p, hipStream_t st) {
    switch (p.sr) {
        case TG_MAXPLUS:
            return p.f64 ? launch_typed<SR_MAXPLUS, double>(p, st) : launch_typed<SR_MAXPLUS, int64_t>(p, st);
        case TG_MINPLUS:
            return p.f64 ? launch_typed<SR_MINPLUS, double>(p, st) : launch_typed<SR_MINPLUS, int64_t>(p, st);
        default:
            return p.f64 ? launch_typed<SR_MAXMUL, double>(p, st) : launch_typed<SR_MAXMUL, int64_t>(p, st);
    }
}

}  // namespace tg
