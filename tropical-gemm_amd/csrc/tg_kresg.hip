// tg_kresg.hip -- launches of tg_gemm_kresg.
#include "tg_kresg.hpp"

#include "tg_gemm_kresg.hpp"

namespace tg {
namespace {

template <int SR, int WAVES>
hipError_t launch(const KresgProblem& p, int cus, hipStream_t st) {
    using Cfg = KresgCfg<WAVES>;
    const auto kernel = &tg_gemm_kresg<SR, WAVES>;
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
        int(Cfg::lds_bytes(Cfg::K_MAX)));
    if (attr != hipSuccess) return attr;
    const int64_t tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    // The resident workgroups shared out over items and column tiles, and no
    // more per column tile than have a row tile for every wave.
    const int64_t slots = int64_t(cus) * (16 / WAVES);
    const int64_t rows = ((p.M + Cfg::ROWS - 1) / Cfg::ROWS + WAVES - 1) / WAVES;
    int64_t groups = slots / tiles_n / p.batch;
    groups = groups < 1 ? 1 : groups;
    groups = groups < rows ? groups : rows;
    for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
        const int64_t nb = p.batch - z0 < 65535 ? p.batch - z0 : 65535;
        hipLaunchKernelGGL(kernel, dim3(unsigned(groups * tiles_n), unsigned(nb)),
                           dim3(Cfg::THREADS), Cfg::lds_bytes(p.K), st, p.A + z0 * p.sA,
                           p.B + z0 * p.sB, p.C + z0 * p.sC, p.IDX + z0 * p.sC, p.M, p.N, p.K,
                           p.sA, p.sB, p.sC, int(tiles_n));
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int SR>
hipError_t launch_waves(const KresgProblem& p, int cus, hipStream_t st) {
    return p.K <= KresgCfg<8>::K_MAX ? launch<SR, 8>(p, cus, st) : launch<SR, 16>(p, cus, st);
}

}  // namespace

bool kresg_fits(int64_t M, int64_t N, int64_t K) {
    return M >= 16 && N >= 16 && N <= (int64_t(1) << 20) && K >= 4 && K <= KresgCfg<16>::K_MAX;
}

int64_t kresg_wave_tiles(int64_t M, int64_t N) { return ((M + 15) / 16) * ((N + 63) / 64); }

hipError_t kresg_launch(const KresgProblem& p, int cus, hipStream_t st) {
    return p.sr == SR_MAXPLUS ? launch_waves<SR_MAXPLUS>(p, cus, st)
                              : launch_waves<SR_MINPLUS>(p, cus, st);
}

}  // namespace tg
