// tg_capi.hip -- the C ABI declared in include/tropical_gemm_hip.h.
//
// Host side of the drop-in boundary: argument validation (done before any HIP
// call, so it is testable without a GPU), device selection, layout mapping,
// workspace handling and kernel dispatch.  Reference counterparts are cited
// per entry point in the header.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/tropical_gemm_hip.h"
#include "tg_backward.hpp"
#include "tg_dl64s.hpp"
#include "tg_dl_elem.hpp"
#include "tg_gemm_dl.hpp"
#include "tg_gemm_dl64.hpp"
#include "tg_gemm_kres.hpp"
#include "tg_gemm_kres8.hpp"
#include "tg_gemm_kresw.hpp"
#include "tg_gemm_shortk.hpp"
#include "tg_kernels.hpp"
#include "tg_kresg.hpp"
#include "tg_small.hpp"

namespace {

constexpr int kAbiVersion = 1;

thread_local std::string g_last_error = "";

int fail(int status, const std::string& msg) {
    g_last_error = msg;
    return status;
}

int hip_fail(hipError_t e, const char* what) {
    return fail(TG_ERR_DRIVER, std::string(what) + ": " + hipGetErrorString(e));
}

#define TG_HIP(expr)                                   \
    do {                                               \
        hipError_t _e = (expr);                        \
        if (_e != hipSuccess) return hip_fail(_e, #expr); \
    } while (0)

int elem_size(tg_dtype dt) {
    switch (dt) {
        case TG_F32:
        case TG_I32:
            return 4;
        case TG_F64:
        case TG_I64:
            return 8;
    }
    return 0;
}

const char* dtype_name(int dt) {
    switch (dt) {
        case TG_F32: return "f32";
        case TG_F64: return "f64";
        case TG_I32: return "i32";
        case TG_I64: return "i64";
    }
    return "?";
}

bool valid_semiring(int s) { return s == TG_MAXPLUS || s == TG_MINPLUS || s == TG_MAXMUL; }
bool valid_dtype(int d) { return d == TG_F32 || d == TG_F64 || d == TG_I32 || d == TG_I64; }
bool valid_layout(int l) { return l == TG_ROW_MAJOR || l == TG_COL_MAJOR; }

// Device handling: the ordinal is validated against the device count (the
// reference answers an out-of-range ordinal with DimensionMismatch,
// crates/tropical-gemm-cuda/src/lib.rs:81-87) and made current.
std::once_flag g_count_once;
int g_device_count = -1;
hipError_t g_count_err = hipSuccess;

int device_count_cached(int* out) {
    std::call_once(g_count_once, [] {
        int n = 0;
        g_count_err = hipGetDeviceCount(&n);
        g_device_count = (g_count_err == hipSuccess) ? n : 0;
    });
    if (g_count_err != hipSuccess && g_count_err != hipErrorNoDevice)
        return hip_fail(g_count_err, "hipGetDeviceCount");
    *out = g_device_count;
    return TG_OK;
}

int select_device(int device) {
    int n = 0;
    int rc = device_count_cached(&n);
    if (rc != TG_OK) return rc;
    if (n <= 0) return fail(TG_ERR_NO_DEVICE, "no HIP device available");
    if (device < 0 || device >= n)
        return fail(TG_ERR_DIMENSION_MISMATCH, "Device " + std::to_string(device) +
                                                   " not available (only " + std::to_string(n) +
                                                   " HIP device(s) found)");
    int cur = -1;
    TG_HIP(hipGetDevice(&cur));
    if (cur != device) TG_HIP(hipSetDevice(device));
    return TG_OK;
}

hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Optional event timing of the main GEMM kernels (tg_kernel_timing_*).
std::atomic<bool> g_timing{false};
std::mutex g_timing_mu;
std::vector<std::pair<hipEvent_t, hipEvent_t>> g_timing_events;

// Records an event pair around the launches made during its lifetime when
// timing is enabled; does nothing otherwise.
class KernelTimer {
  public:
    explicit KernelTimer(hipStream_t st) : st_(st) {
        if (!g_timing.load(std::memory_order_relaxed)) return;
        if (hipEventCreate(&e0_) != hipSuccess || hipEventCreate(&e1_) != hipSuccess ||
            hipEventRecord(e0_, st_) != hipSuccess) {
            release();
            return;
        }
        on_ = true;
    }
    ~KernelTimer() {
        if (!on_) return;
        if (hipEventRecord(e1_, st_) != hipSuccess) {
            release();
            return;
        }
        std::lock_guard<std::mutex> lk(g_timing_mu);
        g_timing_events.emplace_back(e0_, e1_);
    }
    KernelTimer(const KernelTimer&) = delete;
    KernelTimer& operator=(const KernelTimer&) = delete;

  private:
    void release() {
        if (e0_) (void)hipEventDestroy(e0_);
        if (e1_) (void)hipEventDestroy(e1_);
        e0_ = e1_ = nullptr;
        on_ = false;
    }
    hipStream_t st_;
    hipEvent_t e0_ = nullptr, e1_ = nullptr;
    bool on_ = false;
};

// ----------------------------------------------------------------------------
// Launch helpers
// ----------------------------------------------------------------------------

int launch_fill_zero(void* p, size_t bytes, hipStream_t st) {
    if (bytes == 0) return TG_OK;
    int64_t nvec = int64_t(bytes / 16);
    int64_t blocks = (nvec + 255) / 256;
    if (blocks < 1) blocks = 1;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(tg::tg_fill_zero, dim3(unsigned(blocks)), dim3(256), 0, st,
                       static_cast<unsigned char*>(p), int64_t(bytes));
    TG_HIP(hipGetLastError());
    return TG_OK;
}

template <typename T>
bool aligned16(const void* p) {
    return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

// B^T staging (BT[z][j][k] = B[z][k][j], nb batch items): 16-byte vectors when
// the shape, strides and pointers allow them, element by element otherwise.
// The callers have checked (K + 31) / 32 <= 65535.
template <typename T>
bool transpose_vectors(const T* B, const T* BT, int64_t K, int64_t N, int64_t sB, int64_t sBT) {
    constexpr int VW = tg::Vec16<T>::N;
    return K % VW == 0 && N % VW == 0 && sB % VW == 0 && sBT % VW == 0 && aligned16<T>(B) &&
           aligned16<T>(BT);
}

// cls (f64 only, and only where transpose_vectors holds): the column classes
// of B are ORed into cls[z*N + j] on the way (see tg_transpose_v).
template <typename T>
int launch_transpose(const T* B, T* BT, int64_t K, int64_t N, int64_t sB, int64_t sBT, int64_t nb,
                     hipStream_t st, uint32_t* cls = nullptr) {
    if (transpose_vectors<T>(B, BT, K, N, sB, sBT)) {
        dim3 grid(unsigned((N + 63) / 64), unsigned((K + 63) / 64), unsigned(nb));
        hipLaunchKernelGGL((tg::tg_transpose_v<T>), grid, dim3(256), 0, st, B, BT, K, N, sB, sBT,
                           cls);
    } else {
        if (cls != nullptr)
            return fail(TG_ERR_INVALID_ARGUMENT, "internal: column classes need the vector transpose");
        dim3 grid(unsigned((N + 31) / 32), unsigned((K + 31) / 32), unsigned(nb));
        hipLaunchKernelGGL((tg::tg_transpose<T>), grid, dim3(32, 8), 0, st, B, BT, K, N, sB, sBT);
    }
    TG_HIP(hipGetLastError());
    return TG_OK;
}

// Row-major problem description after the layout mapping.
struct Problem {
    const void* A;
    const void* B;
    void* C;
    int32_t* IDX;
    int64_t batch, M, N, K, sA, sB, sC;
};

size_t round_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Workspace layout: [B^T staging (argmax)][split-K value partials][split-K
// index partials (argmax)], each region 256-byte aligned.
struct WsLayout {
    size_t bt = 0, pv = 0, pi = 0, total = 0;
};

WsLayout ws_layout(tg_dtype dt, int64_t batch, int64_t M, int64_t N, int64_t K, bool argmax,
                   int splits) {
    WsLayout w;
    const size_t es = size_t(elem_size(dt));
    const size_t bt = argmax ? round_up(size_t(batch) * size_t(K) * size_t(N) * es, 256) : 0;
    const size_t part = splits > 1 ? round_up(size_t(splits) * size_t(batch) * size_t(M) * size_t(N) * es, 256) : 0;
    w.bt = 0;
    w.pv = bt;
    w.pi = bt + part;
    w.total = bt + part + (argmax ? part : 0);
    return w;
}

// Workspace of the f64 direct-to-LDS kernel: B^T (batch x K x N, argmax
// only), then the row classes of A (batch x M) and column classes of B
// (batch x N).
size_t dl64_ws_bytes(int64_t batch, int64_t M, int64_t N, int64_t K, bool argmax) {
    return (argmax ? round_up(size_t(batch) * size_t(K) * size_t(N) * 8, 256) : 0) +
           round_up(size_t(batch) * size_t(M + N) * 4, 256);
}

// Prepasses of the f64 direct-to-LDS kernels, into a workspace of
// dl64_ws_bytes: operand classes and, with argmax, B^T.
struct Dl64Ws {
    double* BT;
    uint32_t *clsA, *clsB;
};

int prepare_dl64(const Problem& p, void* ws, hipStream_t st, Dl64Ws* out) {
    if ((p.K + 31) / 32 > 65535 || (p.K + 255) / 256 > 65535)
        return fail(TG_ERR_DIMENSION_MISMATCH, "K too large for the staging grids");
    const double* A = static_cast<const double*>(p.A);
    const double* B = static_cast<const double*>(p.B);
    const bool argmax = p.IDX != nullptr;
    unsigned char* wsb = static_cast<unsigned char*>(ws);
    double* BT = argmax ? reinterpret_cast<double*>(wsb) : nullptr;
    const size_t bt_bytes = argmax ? round_up(size_t(p.batch) * size_t(p.K) * size_t(p.N) * 8, 256) : 0;
    uint32_t* cls = reinterpret_cast<uint32_t*>(wsb + bt_bytes);
    uint32_t* clsA = cls;
    uint32_t* clsB = cls + p.batch * p.M;
    // With argmax, the B^T transpose records the column classes when it runs
    // on 16-byte vectors (every batch chunk alike: sB and K*N are even).
    const bool cols_in_transpose =
        argmax && transpose_vectors<double>(B, BT, p.K, p.N, p.sB, p.K * p.N);
    hipLaunchKernelGGL(tg::tg_fill_zero, dim3(unsigned((p.batch * (p.M + p.N) * 4 / 16 + 255) / 256 + 1)),
                       dim3(256), 0, st, reinterpret_cast<unsigned char*>(cls), p.batch * (p.M + p.N) * 4);
    TG_HIP(hipGetLastError());
    {
        int64_t row_blocks = (p.batch * p.M + 3) / 4;
        if (row_blocks > 16384) row_blocks = 16384;
        int64_t col_blocks = cols_in_transpose ? 0 : ((p.N + 63) / 64) * ((p.K + 255) / 256) * p.batch;
        if (col_blocks > 16384) col_blocks = 16384;
        hipLaunchKernelGGL(tg::tg_class_prepass, dim3(unsigned(row_blocks + col_blocks)), dim3(256), 0,
                           st, A, p.M, p.K, p.sA, B, p.N, p.sB, p.batch, clsA,
                           cols_in_transpose ? nullptr : clsB, int(row_blocks));
        TG_HIP(hipGetLastError());
    }
    for (int64_t z0 = 0; argmax && z0 < p.batch; z0 += 65535) {
        const int64_t nb = (p.batch - z0 < 65535) ? p.batch - z0 : 65535;
        const int rc = launch_transpose<double>(B + z0 * p.sB, BT + z0 * p.K * p.N, p.K, p.N, p.sB,
                                                p.K * p.N, nb, st,
                                                cols_in_transpose ? clsB + z0 * p.N : nullptr);
        if (rc != TG_OK) return rc;
    }
    *out = Dl64Ws{BT, clsA, clsB};
    return TG_OK;
}

// f64, large problems (tg_gemm_dl64): the prepasses, then the GEMM.
// K % 32 == 0 and the rest of dl64_fits hold.
template <int SR>
int run_gemm_dl64(const Problem& p, void* ws, hipStream_t st) {
    using Cfg = tg::Dl64Cfg;
    const int64_t tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM;
    const int64_t tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    if (tiles_m * tiles_n > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "output too large for one launch");
    Dl64Ws w;
    const int rc = prepare_dl64(p, ws, st, &w);
    if (rc != TG_OK) return rc;
    const double* A = static_cast<const double*>(p.A);
    const double* B = static_cast<const double*>(p.B);
    const bool argmax = p.IDX != nullptr;
    double* const BT = w.BT;
    uint32_t *const clsA = w.clsA, *const clsB = w.clsB;
    KernelTimer timer(st);
    for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
        const int64_t nb = (p.batch - z0 < 65535) ? p.batch - z0 : 65535;
        const dim3 grid(unsigned(tiles_m * tiles_n), 1, unsigned(nb));
        double* Cz = static_cast<double*>(p.C) + z0 * p.sC;
        if (argmax)
            hipLaunchKernelGGL((tg::tg_gemm_dl64<SR, true>), grid, dim3(256), Cfg::LDS_BYTES, st,
                               A + z0 * p.sA, B + z0 * p.sB, BT + z0 * p.K * p.N, Cz,
                               p.IDX + z0 * p.sC, clsA + z0 * p.M, clsB + z0 * p.N, p.M, p.N, p.K,
                               p.sA, p.sB, p.sC, int(tiles_m), int(tiles_n));
        else
            hipLaunchKernelGGL((tg::tg_gemm_dl64<SR, false>), grid, dim3(256), Cfg::TILE_BYTES, st,
                               A + z0 * p.sA, B + z0 * p.sB, nullptr, Cz, nullptr, clsA + z0 * p.M,
                               clsB + z0 * p.N, p.M, p.N, p.K, p.sA, p.sB, p.sC, int(tiles_m),
                               int(tiles_n));
        TG_HIP(hipGetLastError());
    }
    return TG_OK;
}

// 64-bit problems on 64 x 64 tiles (tg_gemm_dl64s; tg::dl64s_fits holds): f64
// with its prepasses, i64 with B^T staging for argmax.
template <int SR, typename T>
int run_gemm_dl64s(const Problem& p, void* ws, hipStream_t st) {
    constexpr bool f64 = std::is_same<T, double>::value;
    Dl64Ws w{nullptr, nullptr, nullptr};
    T* BT = nullptr;
    if constexpr (f64) {
        const int rc = prepare_dl64(p, ws, st, &w);
        if (rc != TG_OK) return rc;
        BT = w.BT;
    } else if (p.IDX != nullptr) {
        if ((p.K + 31) / 32 > 65535)
            return fail(TG_ERR_DIMENSION_MISMATCH, "K too large for the transpose grid");
        BT = static_cast<T*>(ws);
        for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
            const int64_t nb = (p.batch - z0 < 65535) ? p.batch - z0 : 65535;
            const int rc = launch_transpose<T>(static_cast<const T*>(p.B) + z0 * p.sB,
                                               BT + z0 * p.K * p.N, p.K, p.N, p.sB, p.K * p.N, nb, st);
            if (rc != TG_OK) return rc;
        }
    }
    KernelTimer timer(st);
    TG_HIP(tg::dl64s_launch(tg::Dl64sProblem{SR, f64, p.A, p.B, BT, p.C, p.IDX, w.clsA, w.clsB,
                                             p.batch, p.M, p.N, p.K, p.sA, p.sB, p.sC},
                            st));
    return TG_OK;
}

// Split argmax on 64 x 64 tiles whose chunk holds an even number of
// fragments runs its K slices in one workgroup: the number of slices (four
// when each keeps at least 256 k, else two), or 0 when the split runs as
// separate launches into the workspace partials.
inline int wg_slices(bool slices_ok, bool argmax, int splits, int64_t K) {
    constexpr int BK = tg::TG_CHUNK;
    if (!slices_ok || !argmax || (splits != 2 && splits != 4) || K % (2 * BK) != 0) return 0;
    return (K % (4 * BK) == 0 && K / 4 >= 256) ? 4 : 2;
}

// Direct-to-LDS kernel for 32-bit types (partial edge tiles allowed, see
// tg::dl_fits).  splits > 1 (full tiles only) runs K in that many slices into
// the workspace partials, then merges them.
template <int SR, typename T, int TM, int TN, int CL>
int run_gemm_dl(const Problem& p, void* ws, int splits, hipStream_t st) {
    using Cfg = tg::DlCfg<TM, TN>;
    const int64_t tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM;  // the last ones may be partial
    const int64_t tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    if (tiles_m * tiles_n > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "output too large for one launch");
    const T* A = static_cast<const T*>(p.A);
    const T* B = static_cast<const T*>(p.B);
    T* C = static_cast<T*>(p.C);
    const bool argmax = p.IDX != nullptr;
    const WsLayout wl = ws_layout(std::is_same<T, float>::value ? TG_F32 : TG_I32, p.batch, p.M,
                                  p.N, p.K, argmax, splits);
    unsigned char* wsb = static_cast<unsigned char*>(ws);
    T* PV = splits > 1 ? reinterpret_cast<T*>(wsb + wl.pv) : nullptr;
    int32_t* PI = (splits > 1 && argmax) ? reinterpret_cast<int32_t*>(wsb + wl.pi) : nullptr;
    const int64_t MN = p.M * p.N;
    const int64_t sY = splits > 1 ? p.batch * MN : 0;
    const int64_t KS = p.K / splits;
    // Split-K problems are small: when all of B (every batch item) fits in
    // 4 MiB it stays in L2, and the resolve reads B's columns directly
    // (BDIRECT), with no B^T staged and one launch fewer.
    const bool bdirect = argmax && splits > 1 && TN == 4 && p.K % Cfg::BK == 0 &&
                         size_t(p.batch) * size_t(p.K) * size_t(p.N) * sizeof(T) <= (size_t(4) << 20);
    if (argmax && !bdirect) {  // B^T staging for the resolve, outside the timed GEMM launches
        if ((p.K + 31) / 32 > 65535)
            return fail(TG_ERR_DIMENSION_MISMATCH, "K too large for the transpose grid");
        for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
            const int64_t nb = (p.batch - z0 < 65535) ? p.batch - z0 : 65535;
            T* BT = reinterpret_cast<T*>(wsb + wl.bt) + z0 * p.K * p.N;
            const int rc = launch_transpose<T>(B + z0 * p.sB, BT, p.K, p.N, p.sB, p.K * p.N, nb, st);
            if (rc != TG_OK) return rc;
        }
    }
    // 128 x 128 value-only tiles take 64 KB of dynamic LDS: raise the
    // kernel's limit once (no stream work, so also fine under capture).
    // The value-only 8 x 8 tiles run the pipelined main loop (tg::pipe_fits).
    constexpr bool kPipe = TM == 8 && TN == 8;
    const bool pipe = kPipe && !argmax && tg::pipe_fits(p.N, p.K);
    if constexpr (Cfg::TILE_BYTES > 48 * 1024) {
        static const hipError_t attr = hipFuncSetAttribute(
            reinterpret_cast<const void*>(&tg::tg_gemm_dl<SR, T, false, TM, TN, CL>),
            hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::TILE_BYTES);
        TG_HIP(attr);
        if constexpr (kPipe) {
            static const hipError_t attr_pipe = hipFuncSetAttribute(
                reinterpret_cast<const void*>(&tg::tg_gemm_dl<SR, T, false, TM, TN, CL, false, false, 2>),
                hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::TILE_BYTES);
            TG_HIP(attr_pipe);
        }
    }
    // Split argmax on 64 x 64 tiles: the K slices of a tile run in one
    // workgroup, 256 threads per slice, and merge in LDS (no partials, no
    // merge launch).  Four slices (1024 threads, four waves per SIMD) when
    // each slice keeps at least 256 k, else two.
    constexpr bool kHalves = TM == 4 && TN == 4 && (Cfg::BK / CL) % 2 == 0;
    if (const int halves = wg_slices(kHalves, argmax, splits, p.K)) {
        if constexpr (kHalves) {
            const int64_t KSh = p.K / halves;
            static const hipError_t attr4 = hipFuncSetAttribute(
                reinterpret_cast<const void*>(&tg::tg_gemm_dl<SR, T, true, TM, TN, CL, false, false, 0, 4>),
                hipFuncAttributeMaxDynamicSharedMemorySize, 4 * Cfg::LDS_BYTES);
            static const hipError_t attr4d = hipFuncSetAttribute(
                reinterpret_cast<const void*>(&tg::tg_gemm_dl<SR, T, true, TM, TN, CL, false, true, 0, 4>),
                hipFuncAttributeMaxDynamicSharedMemorySize, 4 * Cfg::LDS_BYTES);
            TG_HIP(attr4);
            TG_HIP(attr4d);
            KernelTimer timer(st);
            for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
                const int64_t nb = (p.batch - z0 < 65535) ? p.batch - z0 : 65535;
                const T* Az = A + z0 * p.sA;
                const T* Bz = B + z0 * p.sB;
                T* Cz = C + z0 * p.sC;
                int32_t* Iz = p.IDX + z0 * p.sC;
                const T* BT = reinterpret_cast<const T*>(wsb + wl.bt) + z0 * p.K * p.N;
                dim3 grid(unsigned(tiles_m * tiles_n), 1, unsigned(nb));
                if (halves == 4) {
                    if (bdirect)
                        hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, true, TM, TN, CL, false, true, 0, 4>),
                                           grid, dim3(1024), 4 * Cfg::LDS_BYTES, st, Az, Bz, nullptr,
                                           Cz, Iz, p.M, p.N, p.K, p.sA, p.sB, p.sC, int(tiles_m),
                                           int(tiles_n), KSh, int64_t(0));
                    else
                        hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, true, TM, TN, CL, false, false, 0, 4>),
                                           grid, dim3(1024), 4 * Cfg::LDS_BYTES, st, Az, Bz, BT, Cz,
                                           Iz, p.M, p.N, p.K, p.sA, p.sB, p.sC, int(tiles_m),
                                           int(tiles_n), KSh, int64_t(0));
                } else if (bdirect) {
                    hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, true, TM, TN, CL, false, true, 0, 2>),
                                       grid, dim3(512), 2 * Cfg::LDS_BYTES, st, Az, Bz, nullptr, Cz,
                                       Iz, p.M, p.N, p.K, p.sA, p.sB, p.sC, int(tiles_m),
                                       int(tiles_n), KSh, int64_t(0));
                } else {
                    hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, true, TM, TN, CL, false, false, 0, 2>),
                                       grid, dim3(512), 2 * Cfg::LDS_BYTES, st, Az, Bz, BT, Cz, Iz,
                                       p.M, p.N, p.K, p.sA, p.sB, p.sC, int(tiles_m), int(tiles_n),
                                       KSh, int64_t(0));
                }
                TG_HIP(hipGetLastError());
            }
        }
        return TG_OK;
    }
    KernelTimer timer(st);
    for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
        const int64_t nb = (p.batch - z0 < 65535) ? p.batch - z0 : 65535;
        const T* Az = A + z0 * p.sA;
        const T* Bz = B + z0 * p.sB;
        // Split launches write dense partials (batch stride M*N).
        T* Cz = splits > 1 ? PV + z0 * MN : C + z0 * p.sC;
        int32_t* Iz = !argmax ? nullptr : splits > 1 ? PI + z0 * MN : p.IDX + z0 * p.sC;
        const int64_t sCk = splits > 1 ? MN : p.sC;
        dim3 grid(unsigned(tiles_m * tiles_n), unsigned(splits), unsigned(nb));
        const bool tailk = p.K % Cfg::BK != 0;  // the last k-tile is partial
        if (argmax) {
            const T* BT = reinterpret_cast<const T*>(wsb + wl.bt) + z0 * p.K * p.N;
            if constexpr (TM == 4 && TN == 4 && (Cfg::BK / CL) % 2 == 0) {
                if (bdirect) {
                    hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, true, TM, TN, CL, false, true>), grid,
                                       dim3(256), Cfg::LDS_BYTES, st, Az, Bz, nullptr, Cz, Iz, p.M,
                                       p.N, p.K, p.sA, p.sB, sCk, int(tiles_m), int(tiles_n), KS,
                                       sY);
                    TG_HIP(hipGetLastError());
                    continue;
                }
            }
            if constexpr (TM == 4 && (Cfg::BK / CL) % 2 == 0) {
                if (tailk) {
                    // 64 x 64 tiles only: the 64 x 128 kernel with the tail
                    // code would spill (the plan never picks it for a partial K).
                    if constexpr (TN == 4)
                        hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, true, TM, TN, CL, true>), grid,
                                           dim3(256), Cfg::LDS_BYTES, st, Az, Bz, BT, Cz, Iz, p.M,
                                           p.N, p.K, p.sA, p.sB, sCk, int(tiles_m), int(tiles_n),
                                           KS, sY);
                    else
                        return fail(TG_ERR_INVALID_ARGUMENT,
                                    "internal: 64x128 tiles need K % 32 == 0");
                } else
                    hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, true, TM, TN, CL>), grid, dim3(256),
                                       Cfg::LDS_BYTES, st, Az, Bz, BT, Cz, Iz, p.M, p.N, p.K,
                                       p.sA, p.sB, sCk, int(tiles_m), int(tiles_n), KS, sY);
            } else {
                return fail(TG_ERR_INVALID_ARGUMENT,
                            "internal: argmax tiles have 4 rows and an even chunk count per k-tile");
            }
        } else {
            if (tailk) {
                if constexpr (TM == 4 && TN == 4)
                    hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, false, TM, TN, CL, true>), grid,
                                       dim3(256), Cfg::TILE_BYTES, st, Az, Bz, nullptr, Cz,
                                       nullptr, p.M, p.N, p.K, p.sA, p.sB, sCk, int(tiles_m),
                                       int(tiles_n), KS, sY);
                else
                    return fail(TG_ERR_INVALID_ARGUMENT, "internal: wide tiles need K % 32 == 0");
            } else if (pipe) {
                if constexpr (kPipe)
                    hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, false, TM, TN, CL, false, false, 2>),
                                       grid, dim3(256), Cfg::TILE_BYTES, st, Az, Bz, nullptr, Cz,
                                       nullptr, p.M, p.N, p.K, p.sA, p.sB, sCk, int(tiles_m),
                                       int(tiles_n), KS, sY);
            } else
                hipLaunchKernelGGL((tg::tg_gemm_dl<SR, T, false, TM, TN, CL>), grid, dim3(256),
                                   Cfg::TILE_BYTES, st, Az, Bz, nullptr, Cz, nullptr, p.M, p.N,
                                   p.K, p.sA, p.sB, sCk, int(tiles_m), int(tiles_n), KS, sY);
        }
        TG_HIP(hipGetLastError());
    }
    if (splits > 1) {
        const int64_t nvec = p.batch * MN / 4;
        int64_t blocks = (nvec + 255) / 256;
        if (blocks > 8192) blocks = 8192;
        const T* BT = argmax && !bdirect ? reinterpret_cast<const T*>(wsb + wl.bt) : nullptr;
        if (argmax)
            hipLaunchKernelGGL((tg::tg_merge_splits<SR, T, true>), dim3(unsigned(blocks)), dim3(256), 0,
                               st, PV, PI, C, p.IDX, splits, MN, p.batch, sY, p.sC, A, B, BT, p.N,
                               p.K, p.sA, p.sB);
        else
            hipLaunchKernelGGL((tg::tg_merge_splits<SR, T, false>), dim3(unsigned(blocks)), dim3(256), 0,
                               st, PV, nullptr, C, nullptr, splits, MN, p.batch, sY, p.sC, A, B,
                               BT, p.N, p.K, p.sA, p.sB);
        TG_HIP(hipGetLastError());
    }
    return TG_OK;
}

// Direct-to-LDS kernel with element loads (32-bit types; N, K, strides and
// pointers of any alignment), 64 x 64 tiles, K in `slices` slices per
// workgroup.  With argmax the workspace holds B^T.
template <int SR, typename T>
int run_gemm_dl_elem(const Problem& p, int cl, int slices, void* ws, hipStream_t st) {
    const bool argmax = p.IDX != nullptr;
    if (((p.M + 63) / 64) * ((p.N + 63) / 64) > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "output too large for one launch");
    if (argmax && (p.K + 31) / 32 > 65535)
        return fail(TG_ERR_DIMENSION_MISMATCH, "K too large for the transpose grid");
    T* const BT = argmax ? static_cast<T*>(ws) : nullptr;
    const int64_t sBT = p.K * p.N;
    for (int64_t z0 = 0; argmax && z0 < p.batch; z0 += 65535) {
        const int64_t nb = (p.batch - z0 < 65535) ? p.batch - z0 : 65535;
        const int rc = launch_transpose<T>(static_cast<const T*>(p.B) + z0 * p.sB, BT + z0 * sBT, p.K,
                                           p.N, p.sB, sBT, nb, st);
        if (rc != TG_OK) return rc;
    }
    KernelTimer timer(st);
    TG_HIP(tg::dl_elem_launch(tg::DlElemProblem{SR, std::is_same<T, float>::value, p.A, p.B, BT, p.C,
                                                p.IDX, p.batch, p.M, p.N, p.K, p.sA, p.sB, p.sC},
                              cl, slices, st));
    return TG_OK;
}

// Compute units of the current device (cached per device).
int current_cu_count() {
    static std::mutex mu;
    static std::vector<int> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    std::lock_guard<std::mutex> lk(mu);
    if (int(cache.size()) <= dev) cache.resize(dev + 1, 0);
    if (cache[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            n = 256;
        cache[dev] = n;
    }
    return cache[dev];
}

// Workgroups of tg_gemm_kres<SR, T, KT> resident per CU (LDS and register
// limits), from the runtime's occupancy calculator; 2 if that fails.
template <int SR, typename T, int KT>
int kres_per_cu() {
    static const int n = [] {
        int b = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, tg::tg_gemm_kres<SR, T, KT>, 256, 0) !=
                hipSuccess ||
            b <= 0) {
            (void)hipGetLastError();
            b = 2;
        }
        return b;
    }();
    return n;
}

template <int SR, typename T, int KT>
void launch_kres(const Problem& p, int64_t tiles_m, int64_t tiles_n, hipStream_t st) {
    // Persistent grid: every resident workgroup slot, rounded down to a
    // multiple of the column-tile count (each workgroup owns one column tile).
    const int64_t total = p.batch * tiles_m * tiles_n;
    int64_t grid = int64_t(kres_per_cu<SR, T, KT>()) * current_cu_count();
    grid = (grid / tiles_n) * tiles_n;
    if (grid < tiles_n) grid = tiles_n;
    if (grid > total) grid = total;
    hipLaunchKernelGGL((tg::tg_gemm_kres<SR, T, KT>), dim3(unsigned(grid)), dim3(256), 0, st,
                       static_cast<const T*>(p.A), static_cast<const T*>(p.B), static_cast<T*>(p.C),
                       p.IDX, p.N, p.sA, p.sB, p.sC, int(tiles_m), int(tiles_n), p.batch);
}

// Workgroups of tg_gemm_kres8<SR, KT> resident per CU; 1 if the query fails.
template <int SR, int KT>
int kres8_per_cu() {
    static const int n = [] {
        int b = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, tg::tg_gemm_kres8<SR, KT>, 256, 0) !=
                hipSuccess ||
            b <= 0) {
            (void)hipGetLastError();
            b = 1;
        }
        return b;
    }();
    return n;
}

template <int SR, int KT>
void launch_kres8(const Problem& p, int64_t tiles_m, int64_t tiles_n, hipStream_t st) {
    const int64_t total = p.batch * tiles_m * tiles_n;
    int64_t grid = int64_t(kres8_per_cu<SR, KT>()) * current_cu_count();
    grid = (grid / tiles_n) * tiles_n;
    if (grid < tiles_n) grid = tiles_n;
    if (grid > total) grid = total;
    hipLaunchKernelGGL((tg::tg_gemm_kres8<SR, KT>), dim3(unsigned(grid)), dim3(256), 0, st,
                       static_cast<const int32_t*>(p.A), static_cast<const int32_t*>(p.B),
                       static_cast<int32_t*>(p.C), p.IDX, p.N, p.sA, p.sB, p.sC, int(tiles_m),
                       int(tiles_n), p.batch);
}

// K-resident argmax kernel with 64 x 128 tiles (i32 MaxPlus/MinPlus).
template <int SR>
int run_gemm_kres8(const Problem& p, hipStream_t st) {
    using Cfg = tg::Kres8Cfg;
    const int64_t tiles_m = p.M / Cfg::BM;
    const int64_t tiles_n = p.N / Cfg::BN;
    if (tiles_m > 0x7fffffffLL || tiles_n > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "output too large for one launch");
    KernelTimer timer(st);
    switch (p.K / Cfg::BK) {
        case 2: launch_kres8<SR, 2>(p, tiles_m, tiles_n, st); break;
        case 3: launch_kres8<SR, 3>(p, tiles_m, tiles_n, st); break;
        case 4: launch_kres8<SR, 4>(p, tiles_m, tiles_n, st); break;
        default: return fail(TG_ERR_INVALID_ARGUMENT, "K-resident kernel: unsupported K");
    }
    TG_HIP(hipGetLastError());
    return TG_OK;
}

// K-resident argmax kernel with wave-private 16-row tiles (i32
// MaxPlus/MinPlus, N a multiple of 128): one 1024-thread workgroup per CU,
// the CUs split evenly over the column tiles.
template <int SR, int KT>
int launch_kresw(const Problem& p, int64_t tiles_n, hipStream_t st) {
    constexpr size_t lds = tg::kresw_lds_bytes(KT);
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void*>(&tg::tg_gemm_kresw<SR, KT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    TG_HIP(attr);
    int64_t grid = (int64_t(current_cu_count()) / tiles_n) * tiles_n;
    if (grid < tiles_n) grid = tiles_n;
    // Fewer workgroups when the row tiles would not give each of a column
    // tile's workgroups one tile per wave.
    const int64_t per_col = (p.M / tg::KreswCfg::ROWS + tg::KreswCfg::WAVES - 1) / tg::KreswCfg::WAVES;
    if (grid > per_col * tiles_n) grid = per_col * tiles_n;
    hipLaunchKernelGGL((tg::tg_gemm_kresw<SR, KT>), dim3(unsigned(grid)), dim3(1024), lds, st,
                       static_cast<const int32_t*>(p.A), static_cast<const int32_t*>(p.B),
                       static_cast<int32_t*>(p.C), p.IDX, p.M, p.N, p.sA, p.sB, p.sC,
                       int(tiles_n), p.batch);
    return TG_OK;
}

int run_gemm_kresg(int sr, const Problem& p, hipStream_t st) {
    KernelTimer timer(st);
    TG_HIP(tg::kresg_launch(
        tg::KresgProblem{sr, static_cast<const int32_t*>(p.A), static_cast<const int32_t*>(p.B),
                         static_cast<int32_t*>(p.C), p.IDX, p.batch, p.M, p.N, p.K, p.sA, p.sB, p.sC},
        current_cu_count(), st));
    return TG_OK;
}

template <int SR>
int run_gemm_kresw(const Problem& p, hipStream_t st) {
    using Cfg = tg::KreswCfg;
    const int64_t tiles_n = p.N / Cfg::BN;
    KernelTimer timer(st);
    int rc = TG_OK;
    switch (p.K / Cfg::BK) {
        case 2: rc = launch_kresw<SR, 2>(p, tiles_n, st); break;
        case 3: rc = launch_kresw<SR, 3>(p, tiles_n, st); break;
        case 4: rc = launch_kresw<SR, 4>(p, tiles_n, st); break;
        default: return fail(TG_ERR_INVALID_ARGUMENT, "K-resident kernel: unsupported K");
    }
    if (rc != TG_OK) return rc;
    TG_HIP(hipGetLastError());
    return TG_OK;
}

// Short-K kernel: 32 x 256 (64-bit types: 16 x 256) tiles written as 1 KB
// row runs.
template <int SR, typename T>
int run_gemm_shortk(const Problem& p, hipStream_t st) {
    using Cfg = tg::ShortkCfg<T>;
    const int64_t tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM;
    const int64_t tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    if (tiles_m * tiles_n > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "output too large for one launch");
    const bool argmax = p.IDX != nullptr;
    KernelTimer timer(st);
    for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
        const int64_t nb = (p.batch - z0 < 65535) ? p.batch - z0 : 65535;
        const T* Az = static_cast<const T*>(p.A) + z0 * p.sA;
        const T* Bz = static_cast<const T*>(p.B) + z0 * p.sB;
        T* Cz = static_cast<T*>(p.C) + z0 * p.sC;
        dim3 grid(unsigned(tiles_m * tiles_n), 1, unsigned(nb));
        if (argmax)
            hipLaunchKernelGGL((tg::tg_gemm_shortk<SR, T, true>), grid, dim3(256), 0, st, Az, Bz,
                               Cz, p.IDX + z0 * p.sC, p.M, p.N, p.K, p.sA, p.sB, p.sC,
                               int(tiles_n));
        else
            hipLaunchKernelGGL((tg::tg_gemm_shortk<SR, T, false>), grid, dim3(256), 0, st, Az, Bz,
                               Cz, nullptr, p.M, p.N, p.K, p.sA, p.sB, p.sC, int(tiles_n));
        TG_HIP(hipGetLastError());
    }
    return TG_OK;
}

// K-resident argmax kernel for short K (32-bit types): no B^T staging.
template <int SR, typename T>
int run_gemm_kres(const Problem& p, hipStream_t st) {
    using Cfg = tg::KresCfg;
    const int64_t tiles_m = p.M / Cfg::BM;
    const int64_t tiles_n = p.N / Cfg::BN;
    if (tiles_m > 0x7fffffffLL || tiles_n > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "output too large for one launch");
    KernelTimer timer(st);
    switch (p.K / Cfg::BK) {
        case 2: launch_kres<SR, T, 2>(p, tiles_m, tiles_n, st); break;
        case 3: launch_kres<SR, T, 3>(p, tiles_m, tiles_n, st); break;
        case 4: launch_kres<SR, T, 4>(p, tiles_m, tiles_n, st); break;
        default: return fail(TG_ERR_INVALID_ARGUMENT, "K-resident kernel: unsupported K");
    }
    TG_HIP(hipGetLastError());
    return TG_OK;
}

// Argmax problems with K up to this run the generic tiles kernel in its exact
// mode (per-product index tracking, no resolve, no B^T staging): at short K
// the chunked kernels' resolve, which re-reads A and B^T windows per output,
// costs several times the main loop.
constexpr int64_t kExactMaxK = 32;
// Argmax problems with partial tiles (M, N or K) that the direct-to-LDS kernels
// can run take the generic kernel's exact mode up to this K: measured on
// MI355X (f32 MaxPlus, 4100^2 and 1000^2), exact 124 us against 153 at K = 64,
// 233 against 188 at K = 128.
constexpr int64_t kExactPartialMaxK = 96;
// Argmax problems that reach the generic tiles kernel (no direct-to-LDS or
// K-resident kernel takes them) run its exact mode up to this K: 4 VALU ops
// per product against the chunked mode's ~2 plus its resolve.  Crossovers
// measured on MI355X (MaxPlus, M = N = 4096): f32 near K = 480, f64 near
// K = 700, i64 near K = 4096 (its 64-bit compare costs as much as the add).
template <typename T>
constexpr int64_t exact_tiles_max_k() {
    return sizeof(T) == 4 ? 384 : std::is_same<T, int64_t>::value ? 2048 : 512;
}

// More than a round of tg_gemm_dl64s tiles by element loads on matrices narrower
// than 512.
bool narrow_elements(const Problem& p) {
    return (p.M < 512 || p.N < 512) && ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch > 256 &&
           !tg::dl64s_vectors(p.N, p.K, p.sA, p.sB, p.A, p.B);
}

// i64 argmax leaves the exact mode earlier where its chunked tiles run
// tg_gemm_dl64s, with the workspace for B^T (us on MI355X, chunked / exact).  The
// staging and the resolve weigh on short K, the more the fewer and the narrower
// the tiles are:
//   up to 256 tiles of 64 x 64, whose exact mode is one round of the chip: 1000^2 x
//     188 63 / 53, x 300 82 / 81, x 512 115 / 133, 256 x (64 x 64 x 512) 134 / 134;
//   up to 512, or narrow, 128 x (128 x 128 x 193) 114 / 110, x 257 140 / 143, 64 x
//     22528 x 193 115 / 107, x 257 138 / 139; 34 x 47910 x 161 145 / 137, x 225 183 / 185,
//     1220 x (64 x 64 x 161) 263 / 226, x 300 0.90 times;
//   beyond, wide: 1501^2 x 128 114 / 113, x 161 124 / 140; from 2048 tiles 3001^2 x 97
//     251 / 272 (2001 x 2003 x 97 127 / 124).
// MaxMul, whose 64-bit products the resolve computes once more (chunked / exact):
// 1500^2 x 193 186 / 165, x 301 249 / 252, 3001^2 x 225 563 / 563; narrower 128 x (128
// x 128 x 1025) 664 / 583, x 1500 834 / 869, 34 x 47910 x 1500 1296 / 1270 (by element loads 100 x
// 16383 x 2500 1485 / 1368 on the register-staged tiles); 1378 x 1379 x 400 244 /
// 232, 1000 x 1001 x 513 159 / 167.
template <int SR, typename T>
bool chunked_i64(const Problem& p, size_t ws_bytes) {
    if (!std::is_same<T, int64_t>::value || p.M < 32 || p.N < 32) return false;
    const int64_t tiles64 = ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch;
    const bool wide = p.M >= 512 && p.N >= 512;
    int64_t from = 513;
    if (SR == tg::SR_MAXMUL && narrow_elements(p)) return false;
    if (tiles64 > 256 && SR == tg::SR_MAXMUL) from = !wide ? 1501 : tiles64 <= 512 ? 513 : 301;
    else if (tiles64 > 512 && wide) from = tiles64 < 2048 ? 129 : 97;
    else if (tiles64 > 256) from = 257;
    if (p.K < from) return false;
    return ws_layout(TG_I64, p.batch, p.M, p.N, p.K, true, 1).total <= ws_bytes &&
           tg::dl64s_fits(p.M, p.N, p.K);
}

// Problems with K up to these run the short-K kernel (when N % 4 == 0 and B,
// C, IDX are 16-byte aligned).  Measured on MI355X (MaxPlus, against the
// kernels these problems took before): f32 65536 x 2048 x K, argmax K = 8
// 183 us against 251 (generic tiles, exact mode), K = 32 403 against 417,
// K = 48 567 against 554; value-only K = 8 104 against 143, K = 48 253
// against 336, K = 64 344 against 343 (direct-to-LDS); f64 8192^2 x K,
// argmax K = 8 163 against 236, K = 32 335 against 390; value-only K = 63
// 368 against 434.
constexpr int64_t kShortkArgmaxMaxK = 32;
constexpr int64_t kShortkValueMaxK = 63;

// The kernel a problem runs on.
enum class Path { SHORTK, KRESW, KRES8, KRES, KRESG, DL_88_32, DL_48_16, DL_48_VALUE, DL_44_8, DL_44_16, DL_44_32, DL_ELEM_8, DL_ELEM_16, DL_ELEM, DL64, DL64_VALUE, DL64S, DL64S_VALUE, DL64S_I64, DL64S_I64_VALUE, TILES_EXACT, TILES_CHUNKED, TILES };

struct Plan {
    Path path = Path::TILES;
    int splits = 1;
    int slices = 1;  // K slices per workgroup of the element-load paths
};

// True when the path reads the workspace: B^T staging for the resolve of the
// chunked argmax kernels, and split-K partials.
bool uses_workspace(const Plan& pl, bool argmax) {
    switch (pl.path) {
        case Path::SHORTK:
        case Path::KRESW:
        case Path::KRES8:
        case Path::KRES:
        case Path::KRESG:
        case Path::DL_ELEM:
        case Path::DL64S_I64_VALUE:
        case Path::TILES_EXACT:
        case Path::TILES: return false;
        case Path::TILES_CHUNKED:
        case Path::DL64:
        case Path::DL64_VALUE:
        case Path::DL64S:
        case Path::DL64S_VALUE:
        case Path::DL64S_I64: return true;
        default: return argmax || pl.splits > 1;
    }
}

// 64 x 128 tiles of a problem (tg_gemm_dl64).
int64_t dl64_tiles(const Problem& p) {
    return ((p.M + tg::Dl64Cfg::BM - 1) / tg::Dl64Cfg::BM) *
           ((p.N + tg::Dl64Cfg::BN - 1) / tg::Dl64Cfg::BN) * p.batch;
}

// True when tg_gemm_kresg is the kernel for an i32 MaxPlus/MinPlus argmax
// problem that the kernels for aligned sizes (kresw, kres8, kres) leave.
// Measured on MI355X (us, against the path it would take otherwise; in the key
// range, then with wide operands):
//   K <= 32, against the short-K kernel, which writes 256-column tiles: 100000
//     x 64 x 12 18 / 44, x 128 x 16 25 / 53, x 256 x 24 43 / 76, 30000 x 200 x
//     16 24 / 19, x 24 25 / 26; wide 262144 x 32 x 32 55 / 234, 50000 x 128 x
//     20 27 / 36.
//   K <= 160, against the generic exact mode and the direct-to-LDS kernels:
//     300 x 300 x 36 10 / 15, 20000 x 48 x 48 11 / 19, 4096^2 x 100 80 / 193,
//     200 x 20000 x 160 46 / 81; wide 20000 x 48 x 48 15 / 19, x 160 x 160 55 /
//     66, 262144 x 160 x 160 537 / 585.
//   beyond, 512 x 512 x 200 35 / 33, 20000 x 200 x 200 68 / 97, 4096 x 1024 x
//     240 43 / 85; wide 4096 x 1024 x 240 72 / 90, but 20000 x 200 x 240 133 /
//     105, whose wave tiles fill 1.2 rounds of the chip's 4096 waves: from
//     three quarters of the last round up.
//   Column groups that are not 16-byte aligned, from 4 M outputs up (which then
//     bound it), K >= 20: 524288 x 33 x 12 96 / 78, x 17 95 / 92, x 24 96 / 114.
bool takes_kresg(const Problem& p) {
    if (!tg::kresg_fits(p.M, p.N, p.K) || p.M < 32) return false;
    const int64_t tiles = tg::kresg_wave_tiles(p.M, p.N) * p.batch;
    if (tiles < 64) return false;
    if (p.N % 4 != 0 && p.K < 20 && double(p.batch) * double(p.M) * double(p.N) >= double(1 << 22))
        return false;
    if (p.K <= 32) return (p.N <= 64 && p.K >= 12) || (p.N <= 256 && p.K >= 20);
    if (p.K <= 160) return true;
    const int64_t rounds = (tiles + 4095) / 4096;
    return 4 * tiles >= 3 * 4096 * rounds;
}

// True when too much of a 32-bit product's 64 x 64 x 32 element-load tiles is
// padding for them, on more tiles than CUs (fewer make one round either way).
// us on MI355X, element loads / generic kernel, whose tiles are 128 x 64:
//   argmax: f32 500 x (65 x 65 x 97) 126 / 93, x 130 137 / 121, x 200 160 / 176,
//     1000000 x 2 x 130 784 / 713, 53 x (214 x 388 x 115) 81 / 75; i32, whose exact mode is the faster one, 100 x
//     (100 x 101 x 97) 43 / 38, x 130 47 / 48;
//   value-only: i32 500 x (65 x 65 x 65) 45 / 36, x 130 69 / 64, x 200 94 / 93, 1260 x (85 x 31 x 131) 85 / 75,
//     50000 x 50 x 65 26 / 24, x 130 38 / 40, 100 x 30000 x 97 31 / 27, 2001^2 x 97 33 / 31; f32 300000 x 5 x 65 72 / 62, x 200
//     146 / 155, 100000 x 33 x 65 29 / 32; four columns or fewer at any K: 1000000
//     x 2 x 515 1256 / 1121.
// A few rows are padding in the generic kernel too (3 x 100000 x 97 94 / 129).
bool elem_padded(const Problem& p, int64_t tiles64, bool i32) {
    if (p.M <= 16) return false;
    const bool argmax = p.IDX != nullptr;
    if (argmax && i32 && p.K < 128) return true;
    if (!argmax && p.N <= 4) return true;
    const double fill = double(p.batch) * double(p.M) * double(p.N) * double(p.K) /
                        (double(tiles64) * 4096 * double((p.K + 31) / 32 * 32));
    if (argmax) return (fill < 0.22 && p.K < 160) || (p.batch > 1 && tiles64 > 1024 && p.K < 128);
    if (p.K < 64) return i32 && fill < 0.3 && p.K < 56;
    if (i32 && tiles64 > 448 && p.K < 112 && p.K % 32 != 0) return true;
    return (p.K < 96 && fill < (i32 ? 0.7 : 0.3)) || (p.K < 200 && fill < (i32 ? 0.3 : 0.22));
}

// Chooses the kernel.  ws_bytes limits split K (the partials live in the
// workspace).
template <int SR, typename T>
Plan plan_typed(const Problem& p, size_t ws_bytes) {
    Plan pl;
    const bool argmax = p.IDX != nullptr;
    const bool exact = argmax && p.K <= kExactMaxK;
    const bool kresg = std::is_same<T, int32_t>::value && SR != tg::SR_MAXMUL && argmax && takes_kresg(p);
    if (kresg && p.K <= 32) {
        pl.path = Path::KRESG;
        return pl;
    }
    if (p.K <= (argmax ? kShortkArgmaxMaxK : kShortkValueMaxK) &&
        tg::shortk_fits(p.M, p.N, p.K, p.sB, p.sC, p.B, p.C, p.IDX)) {
        pl.path = Path::SHORTK;
        return pl;
    }
    if constexpr (sizeof(T) == 4) {
        if constexpr (std::is_same<T, int32_t>::value && SR != tg::SR_MAXMUL) {
            if (argmax && tg::kresw_fits(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
                pl.path = Path::KRESW;
                return pl;
            }
            if (argmax && tg::kres8_fits(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
                pl.path = Path::KRES8;
                return pl;
            }
        }
        if (argmax && tg::kres_fits(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
            pl.path = Path::KRES;
            return pl;
        }
        if (kresg) {
            pl.path = Path::KRESG;
            return pl;
        }
        // Partial tiles (M, N or K): short argmax problems take the generic
        // kernel's exact mode (no resolve); longer ones and value-only run
        // the direct-to-LDS kernels with clamped loads.
        const bool partial = !tg::dl_full_tiles<4, 4>(p.M, p.N, p.K);
        // Value-only with K below 64 and not a multiple of 32: most of the
        // direct-to-LDS kernel's padded last k-tile would be wasted work;
        // the generic kernel bounds its last tile instead.
        const bool short_tail = !argmax && p.K % 32 != 0 && p.K < 64;
        // The direct-to-LDS kernel with element loads (any N, K, strides and
        // pointers), from a quarter of the CUs' worth of tiles up.  Measured
        // on MI355X against the generic kernel (us): argmax 2001^3 f32 348 /
        // 750, i32 455 / 807, 701^3 54 / 301, 3001 x 1501 x 301 102 / 182,
        // 3001^2 x 100 104 / 121, x 65 91 / 86 (so up to K = 96 the exact mode
        // stays); value-only 2001^3 291 / 342, 2001^2 x 60 15.5 / 22.8.  Below
        // K = 48 most of a second k-tile would be padding.  More than a round of
        // tiles whose work is mostly padding (elem_padded).
        const int64_t tiles64 = ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch;
        const int slices = tg::dl_elem_slices(tiles64, p.K, argmax);
        auto take_elem = [&]() {
            if (tiles64 < 64 || !tg::dl_elem_fits<8>(p.M, p.N, p.K)) return false;
            // One launch holds less than 2^32 threads (256 per tile); the generic
            // kernel's tiles are twice as high.
            if (tiles64 / p.batch >= (int64_t(1) << 24)) return false;
            if (tiles64 > 256 && elem_padded(p, tiles64, std::is_same<T, int32_t>::value)) return false;
            if (!argmax) {
                if (p.K < 48) return false;
                pl.path = Path::DL_ELEM;
            } else {
                const tg_dtype dt = std::is_same<T, float>::value ? TG_F32 : TG_I32;
                if (p.K <= kExactPartialMaxK ||
                    ws_layout(dt, p.batch, p.M, p.N, p.K, true, 1).total > ws_bytes)
                    return false;
                pl.path = slices > 1 || p.K <= 512 ? Path::DL_ELEM_8 : Path::DL_ELEM_16;
            }
            pl.slices = slices;
            return true;
        };
        // Aligned problems of up to two tiles per CU whose K the kernels below
        // do not split: its K slices outweigh the element loads (1300^3 f32
        // argmax 134 / 137 us, 4000 x 300 x 2000 180 / 187, 1200 x 1300 x 700
        // 82 / 89; value-only 94 / 104, 135 / 158, 52 / 58; the shortest K only for f32
        // argmax, 1408^2 x 256 43 / 44, i32 51 / 49, value-only x 288 25 / 24).
        // (i32 argmax of batches neither: 36 x (128 x 320 x 1024) MaxMul 163 / 154).
        const bool f32_argmax = argmax && std::is_same<T, float>::value;
        const bool long_enough =
            tiles64 <= 256 || f32_argmax || (p.K >= 320 && !(argmax && p.batch > 1 && p.K >= 1024));
        if (slices > 1 && tiles64 <= 512 && (tiles64 > 256 || p.K % 64 != 0) && long_enough && take_elem())
            return pl;
        if (!exact && !short_tail && !(partial && argmax && p.K <= kExactPartialMaxK)) {
            // Direct-to-LDS kernels (value-only, or argmax beyond the exact
            // range).  Split K when the problem makes too few 64 x 64 tiles
            // and the workspace holds the partials (tg_gemm_workspace_size
            // includes them).
            const tg_dtype dt = std::is_same<T, float>::value ? TG_F32 : TG_I32;
            int splits = tg::dl_splits(p.M, p.N, p.K, p.batch);
            if (splits > 1 && ws_layout(dt, p.batch, p.M, p.N, p.K, argmax, splits).total > ws_bytes)
                splits = 1;
            const int64_t ks = p.K / splits;
            // Argmax chunk length.  The bookkeeping costs 2 VALU ops per output
            // per chunk (2K/CL); the resolve re-reads one chunk's A-row and
            // B^T-row segments per output from L2 and recomputes them, which
            // costs more than its ~4 ops per product suggest.  Measured on
            // MI355X (f32 MaxPlus, slices of 256 .. 4096 k): CL = 8 is fastest
            // up to 512 k per slice, CL = 16 above (CL = 32 is 4-18% slower
            // everywhere).
            const int cl = !argmax ? 32 : ks <= 512 ? 8 : 16;
            // 64 x 128 tiles for argmax problems big enough that the last
            // round of 768 resident workgroups is a small share of the work
            // (their main loop is the faster one); 64 x 64 tiles otherwise
            // (value-only runs four workgroups per CU, small problems get
            // twice the tiles).
            using W48 = tg::DlCfg<4, 8>;
            using W88 = tg::DlCfg<8, 8>;
            const bool wide = splits == 1 && argmax && cl == 16 && p.N % W48::BN == 0 &&
                              p.K % W48::BK == 0 &&
                              ((p.M + W48::BM - 1) / W48::BM) * (p.N / W48::BN) * p.batch >= 1536;
            // Value-only tile shape by how the tiles fill the resident slots
            // of the 256 CUs (128 x 128 tiles run two per CU, 512 slots;
            // 64 x 64 tiles four, 1024 slots).  128 x 128 tiles (8 x 8
            // outputs per thread) from two rounds up, or exactly one round
            // (2048 x 4096 x 1024: 241 against 267-279 us for 64 x 64; one
            // and a bit rounds, 3072^2 x 2048, take 855 against 593-628 us);
            // 64 x 128 tiles where 64 x 64 would make exactly one round
            // (2048^2 x 2048: 265-269 against 286-290 us; 5-8% at K = 1024 ..
            // 4096); 64 x 64 otherwise (0.75 or 1.25 rounds: 5-15% faster
            // than 64 x 128).
            constexpr int64_t kCus = 256;
            const int64_t t128 =
                ((p.M + W88::BM - 1) / W88::BM) * ((p.N + W88::BN - 1) / W88::BN) * p.batch;
            const int64_t t64 = ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch;
            const bool big = splits == 1 && !argmax && p.K % W88::BK == 0 &&
                             (t128 >= 4 * kCus || t128 == 2 * kCus);
            const bool mid = splits == 1 && !argmax && !big && t64 == 4 * kCus &&
                             p.N % W48::BN == 0 && p.K % W48::BK == 0;
            pl.splits = splits;
            if (wide && tg::dl_fits<16>(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
                pl.path = Path::DL_48_16;
                pl.splits = 1;
                return pl;
            }
            if (big && tg::dl_fits<32>(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
                pl.path = Path::DL_88_32;
                pl.splits = 1;
                return pl;
            }
            if (mid && tg::dl_fits<16>(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
                pl.path = Path::DL_48_VALUE;
                pl.splits = 1;
                return pl;
            }
            if (cl == 8 && tg::dl_fits<8>(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
                pl.path = Path::DL_44_8;
                return pl;
            }
            if (cl == 16 && tg::dl_fits<16>(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
                pl.path = Path::DL_44_16;
                return pl;
            }
            if (cl == 32 && tg::dl_fits<32>(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
                pl.path = Path::DL_44_32;
                return pl;
            }
            pl.splits = 1;
        }
        if (take_elem()) return pl;
    }
    if constexpr (std::is_same<T, double>::value) {
        // f64 from K = 256 with the workspace for the operand classes (and B^T
        // with argmax); below that the prepasses and their launches weigh on
        // the product.  64 x 128 tiles where they give every CU two (argmax
        // beyond the exact range, which they were measured against);
        // otherwise 64 x 64 tiles of any alignment from a quarter of the CUs
        // up (us on MI355X, against 64 x 128 tiles or the generic kernel):
        // argmax 1536^2 x 768 245 / 357, 1024^3 149 / 277, 2047 x 2049 x 1025
        // 518 / 1053, 3001^2 x 300 376 / 459, 3000 x 2000 x 256 221 / 250;
        // value-only 1536^2 x 768 200 / 263, 1024^3 111 / 203, 3001^2 x 300
        // 249 / 323.  Short K on few or narrow tiles stays on the generic kernel:
        // argmax (exact mode) 1000^2 x 300 70 / 63, x 384 77 / 78, 1500^2 x 256
        // 126 / 131, 1501^2 (element loads) x 256 150 / 140, x 257 142 / 142, 256 x
        // (64 x 64 x 512) 115 / 103, 128 x (128 x 128 x 449) 183 / 166; value-only 64 x
        // (128 x 128 x 257) 62 / 56, x 384 67 / 78, 512^2 x 256 35 / 42; in one to two
        // rounds of tiles 128 x (128 x 128 x 321) 96 / 83, x 513 128 / 127, 64 x 22528 x
        // 385 93 / 90, x 449 102 / 104, 1224 x 1225 x 300 76 / 71.
        const int64_t tiles = dl64_tiles(p);
        const int64_t tiles64 = ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch;
        if (p.K >= 256 && dl64_ws_bytes(p.batch, p.M, p.N, p.K, argmax) <= ws_bytes) {
            if (tiles >= 512 && (!argmax || p.K > exact_tiles_max_k<T>()) &&
                tg::dl64_fits(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX)) {
                pl.path = argmax ? Path::DL64 : Path::DL64_VALUE;
                return pl;
            }
            const int64_t narrow = p.M < p.N ? p.M : p.N;
            const bool enough =
                !argmax ? p.K >= 450 || (tiles64 <= 256 || tiles64 > 512 ? p.K >= 320 || narrow >= 512
                                                                         : p.K >= 350 && narrow >= 512)
                : p.K > exact_tiles_max_k<T>() ||
                      (narrow >= 256 &&
                       (tiles64 <= 512 ? p.K > 384
                                       : p.K > 256 || tg::dl64s_vectors(p.N, p.K, p.sA, p.sB, p.A, p.B)));
            if (enough && tiles64 >= 64 && tg::dl64s_fits(p.M, p.N, p.K)) {
                pl.path = argmax ? Path::DL64S : Path::DL64S_VALUE;
                return pl;
            }
        }
    }
    // i64: the chunked and the value-only tiles are tg_gemm_dl64s; the
    // register-staged kernel keeps sizes it does not fit and value-only short K
    // whose last k-tile is mostly padding (us, dl64s / tiles: one round of tiles
    // 1000^2 x 64 15 / 17, x 65 18.7 / 17.8, x 80 18 / 21, MaxMul x 81 30 / 29; more
    // 1500^2 x 100 53 / 50, x 128 57 / 61, 3000^2 x 129 183 / 173, x 161 213 / 213,
    // MaxMul 338 / 319, x 200 384 / 388).
    const bool i64_dl = std::is_same<T, int64_t>::value && tg::dl64s_fits(p.M, p.N, p.K) &&
                        !(argmax && SR == tg::SR_MAXMUL && narrow_elements(p));
    const int64_t tiles64 = ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch;
    if (!argmax)
        pl.path = i64_dl && (tiles64 <= 256 ? p.K >= 96 || (p.K >= 64 && p.K % 16 == 0)
                                            : p.K >= 192 || p.K == 128)
                      ? Path::DL64S_I64_VALUE
                      : Path::TILES;
    else if (exact || (p.K <= exact_tiles_max_k<T>() && !chunked_i64<SR, T>(p, ws_bytes)))
        pl.path = Path::TILES_EXACT;
    else
        pl.path = i64_dl ? Path::DL64S_I64 : Path::TILES_CHUNKED;
    return pl;
}

template <int SR, typename T>
int run_gemm_typed(const Problem& p, void* ws, size_t ws_bytes, hipStream_t st) {
    const Plan pl = plan_typed<SR, T>(p, ws_bytes);
    if (pl.path == Path::SHORTK) return run_gemm_shortk<SR, T>(p, st);
    if constexpr (std::is_same<T, double>::value) {
        if (pl.path == Path::DL64 || pl.path == Path::DL64_VALUE) return run_gemm_dl64<SR>(p, ws, st);
        if (pl.path == Path::DL64S || pl.path == Path::DL64S_VALUE)
            return run_gemm_dl64s<SR, double>(p, ws, st);
    }
    if constexpr (std::is_same<T, int64_t>::value) {
        if (pl.path == Path::DL64S_I64 || pl.path == Path::DL64S_I64_VALUE)
            return run_gemm_dl64s<SR, int64_t>(p, ws, st);
    }
    if constexpr (sizeof(T) == 4) {
        switch (pl.path) {
            case Path::KRESW:
                if constexpr (std::is_same<T, int32_t>::value && SR != tg::SR_MAXMUL)
                    return run_gemm_kresw<SR>(p, st);
                break;
            case Path::KRES8:
                if constexpr (std::is_same<T, int32_t>::value && SR != tg::SR_MAXMUL)
                    return run_gemm_kres8<SR>(p, st);
                break;
            case Path::KRES: return run_gemm_kres<SR, T>(p, st);
            case Path::KRESG:
                if constexpr (std::is_same<T, int32_t>::value && SR != tg::SR_MAXMUL)
                    return run_gemm_kresg(SR, p, st);
                break;
            case Path::DL_88_32: return run_gemm_dl<SR, T, 8, 8, 32>(p, ws, 1, st);
            case Path::DL_48_16: return run_gemm_dl<SR, T, 4, 8, 16>(p, ws, 1, st);
            case Path::DL_48_VALUE: return run_gemm_dl<SR, T, 4, 8, 16>(p, ws, 1, st);  // CL unused
            case Path::DL_44_8: return run_gemm_dl<SR, T, 4, 4, 8>(p, ws, pl.splits, st);
            case Path::DL_44_16: return run_gemm_dl<SR, T, 4, 4, 16>(p, ws, pl.splits, st);
            case Path::DL_44_32: return run_gemm_dl<SR, T, 4, 4, 32>(p, ws, pl.splits, st);
            case Path::DL_ELEM_8:
            case Path::DL_ELEM: return run_gemm_dl_elem<SR, T>(p, 8, pl.slices, ws, st);
            case Path::DL_ELEM_16: return run_gemm_dl_elem<SR, T>(p, 16, pl.slices, ws, st);
            default: break;
        }
    }
    using Cfg = tg::TileCfg<T>;
    const int64_t tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM;
    const int64_t tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    if (tiles_m * tiles_n > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "output too large for one launch");
    const T* A = static_cast<const T*>(p.A);
    const T* B = static_cast<const T*>(p.B);
    T* C = static_cast<T*>(p.C);
    constexpr int VW = 16 / int(sizeof(T));
    const bool vec = (p.K % VW == 0) && (p.N % VW == 0) && (p.sA % VW == 0) &&
                     (p.sB % VW == 0) && aligned16<T>(A) && aligned16<T>(B);
    const bool argmax = p.IDX != nullptr;

    for (int64_t z0 = 0; z0 < p.batch; z0 += 65535) {
        const int64_t nb = (p.batch - z0 < 65535) ? p.batch - z0 : 65535;
        const T* Az = A + z0 * p.sA;
        const T* Bz = B + z0 * p.sB;
        T* Cz = C + z0 * p.sC;
        int32_t* Iz = argmax ? p.IDX + z0 * p.sC : nullptr;
        dim3 grid(unsigned(tiles_m * tiles_n), 1, unsigned(nb));
        if (pl.path == Path::TILES_EXACT) {
            KernelTimer timer(st);
            if (vec)
                hipLaunchKernelGGL((tg::tg_gemm_tiles<SR, T, true, true, true>), grid, dim3(256), 0,
                                   st, Az, Bz, nullptr, Cz, Iz, p.M, p.N, p.K, p.sA, p.sB, p.sC,
                                   int(tiles_m), int(tiles_n));
            else
                hipLaunchKernelGGL((tg::tg_gemm_tiles<SR, T, true, false, true>), grid, dim3(256), 0,
                                   st, Az, Bz, nullptr, Cz, Iz, p.M, p.N, p.K, p.sA, p.sB, p.sC,
                                   int(tiles_m), int(tiles_n));
            TG_HIP(hipGetLastError());
        } else if (pl.path == Path::TILES_CHUNKED) {
            // B^T staging for the argmax epilogue (dense, batch stride K*N).
            T* BT = static_cast<T*>(ws);
            const int64_t sBT = p.K * p.N;
            if (p.K > 0) {
                if ((p.K + 31) / 32 > 65535)
                    return fail(TG_ERR_DIMENSION_MISMATCH, "K too large for the transpose grid");
                const int rc = launch_transpose<T>(Bz, BT, p.K, p.N, p.sB, sBT, nb, st);
                if (rc != TG_OK) return rc;
            }
            // 64-bit integers record 16-k chunks: their 128-byte windows halve
            // what the resolve reads (it misses L2), for one record per 64
            // instructions of products instead of 128.
            constexpr int CL = std::is_same<T, int64_t>::value ? 16 : tg::TG_CHUNK;
            KernelTimer timer(st);
            if (vec)
                hipLaunchKernelGGL((tg::tg_gemm_tiles<SR, T, true, true, false, CL>), grid, dim3(256),
                                   0, st, Az, Bz, BT, Cz, Iz, p.M, p.N, p.K, p.sA, p.sB, p.sC,
                                   int(tiles_m), int(tiles_n));
            else
                hipLaunchKernelGGL((tg::tg_gemm_tiles<SR, T, true, false, false, CL>), grid,
                                   dim3(256), 0, st, Az, Bz, BT, Cz, Iz, p.M, p.N, p.K, p.sA, p.sB,
                                   p.sC, int(tiles_m), int(tiles_n));
            TG_HIP(hipGetLastError());
        } else {
            KernelTimer timer(st);
            if (vec)
                hipLaunchKernelGGL((tg::tg_gemm_tiles<SR, T, false, true>), grid, dim3(256), 0, st,
                                   Az, Bz, nullptr, Cz, nullptr, p.M, p.N, p.K, p.sA, p.sB, p.sC,
                                   int(tiles_m), int(tiles_n));
            else
                hipLaunchKernelGGL((tg::tg_gemm_tiles<SR, T, false, false>), grid, dim3(256), 0,
                                   st, Az, Bz, nullptr, Cz, nullptr, p.M, p.N, p.K, p.sA, p.sB,
                                   p.sC, int(tiles_m), int(tiles_n));
            TG_HIP(hipGetLastError());
        }
    }
    return TG_OK;
}

template <int SR>
int run_gemm_sr(tg_dtype dt, const Problem& p, void* ws, size_t ws_bytes, hipStream_t st) {
    switch (dt) {
        case TG_F32: return run_gemm_typed<SR, float>(p, ws, ws_bytes, st);
        case TG_F64: return run_gemm_typed<SR, double>(p, ws, ws_bytes, st);
        case TG_I32: return run_gemm_typed<SR, int32_t>(p, ws, ws_bytes, st);
        case TG_I64: return run_gemm_typed<SR, int64_t>(p, ws, ws_bytes, st);
    }
    return fail(TG_ERR_INVALID_ARGUMENT, "bad dtype");
}

template <int SR>
Plan plan_sr(tg_dtype dt, const Problem& p, size_t ws_bytes) {
    switch (dt) {
        case TG_F32: return plan_typed<SR, float>(p, ws_bytes);
        case TG_F64: return plan_typed<SR, double>(p, ws_bytes);
        case TG_I32: return plan_typed<SR, int32_t>(p, ws_bytes);
        case TG_I64: return plan_typed<SR, int64_t>(p, ws_bytes);
    }
    return Plan{};
}

Plan plan_gemm(tg_semiring sr, tg_dtype dt, const Problem& p, size_t ws_bytes) {
    switch (sr) {
        case TG_MAXPLUS: return plan_sr<tg::SR_MAXPLUS>(dt, p, ws_bytes);
        case TG_MINPLUS: return plan_sr<tg::SR_MINPLUS>(dt, p, ws_bytes);
        case TG_MAXMUL: return plan_sr<tg::SR_MAXMUL>(dt, p, ws_bytes);
    }
    return Plan{};
}

const char* path_name(Path path) {
    switch (path) {
        case Path::SHORTK: return "shortk";
        case Path::KRESW: return "kresw";
        case Path::KRES8: return "kres8";
        case Path::KRES: return "kres";
        case Path::KRESG: return "kresg";
        case Path::DL_88_32: return "dl_8x8_cl32";
        case Path::DL_48_16: return "dl_4x8_cl16";
        case Path::DL_48_VALUE: return "dl_4x8";
        case Path::DL_44_8: return "dl_4x4_cl8";
        case Path::DL_44_16: return "dl_4x4_cl16";
        case Path::DL_44_32: return "dl_4x4_cl32";
        case Path::DL_ELEM_8: return "dl_elem_cl8";
        case Path::DL_ELEM_16: return "dl_elem_cl16";
        case Path::DL_ELEM: return "dl_elem";
        case Path::DL64: return "dl64_4x8_cl16";
        case Path::DL64_VALUE: return "dl64_4x8";
        case Path::DL64S:
        case Path::DL64S_I64: return "dl64s_4x4_cl16";
        case Path::DL64S_VALUE:
        case Path::DL64S_I64_VALUE: return "dl64s_4x4";
        case Path::TILES_EXACT: return "tiles_exact";
        case Path::TILES_CHUNKED: return "tiles_chunked";
        case Path::TILES: return "tiles";
    }
    return "?";
}

int run_gemm(tg_semiring sr, tg_dtype dt, const Problem& p, void* ws, size_t ws_bytes,
             hipStream_t st) {
    switch (sr) {
        case TG_MAXPLUS: return run_gemm_sr<tg::SR_MAXPLUS>(dt, p, ws, ws_bytes, st);
        case TG_MINPLUS: return run_gemm_sr<tg::SR_MINPLUS>(dt, p, ws, ws_bytes, st);
        case TG_MAXMUL: return run_gemm_sr<tg::SR_MAXMUL>(dt, p, ws, ws_bytes, st);
    }
    return fail(TG_ERR_INVALID_ARGUMENT, "bad semiring");
}

// B^T staging for argmax problems: K x N' elements per batch item, where N'
// is the kernel's N after the layout mapping (n for row-major calls, m for
// column-major ones, whose operands are swapped).  The size does not depend
// on the layout: K x max(m, n) covers both.  This is the minimum workspace.
size_t bt_bytes_for(tg_dtype dt, int64_t batch, int64_t m, int64_t n, int64_t k, bool with_argmax) {
    if (!with_argmax || batch <= 0 || m <= 0 || n <= 0 || k <= 0) return 0;
    const int64_t wide = m > n ? m : n;
    return round_up(size_t(batch) * size_t(k) * size_t(wide) * size_t(elem_size(dt)), 256);
}

// Full workspace: the minimum plus the split-K partials (values, and indices
// for argmax) of 32-bit problems that make too few tiles (tg::dl_splits,
// taken for both orientations: column-major calls swap m and n).  A
// workspace of at least the minimum runs the same products unsplit.
size_t workspace_bytes_for(tg_dtype dt, int64_t batch, int64_t m, int64_t n, int64_t k,
                           bool with_argmax) {
    if (batch <= 0 || m <= 0 || n <= 0 || k <= 0) return 0;
    size_t w = bt_bytes_for(dt, batch, m, n, k, with_argmax);
    if (dt == TG_F64)  // operand classes of the f64 direct-to-LDS kernel
        w += round_up(size_t(batch) * size_t(m + n) * 4, 256);
    if (elem_size(dt) == 4) {
        const int s1 = tg::dl_splits(m, n, k, batch), s2 = tg::dl_splits(n, m, k, batch);
        const int s = s1 > s2 ? s1 : s2;
        if (s > 1) {
            const size_t part = round_up(size_t(s) * size_t(batch) * size_t(m) * size_t(n) * 4, 256);
            w += part * (with_argmax ? 2 : 1);
        }
    }
    return w;
}

// Validation shared by the forward entry points.  Returns TG_OK or an error.
int validate_forward(int sr, int dt, int layout, const void* A, const void* B, const void* C,
                     int64_t batch, int64_t m, int64_t n, int64_t k, int64_t sa, int64_t sb,
                     int64_t sc, bool strided) {
    if (!valid_semiring(sr)) return fail(TG_ERR_INVALID_ARGUMENT, "unknown semiring " + std::to_string(sr));
    if (!valid_dtype(dt)) return fail(TG_ERR_INVALID_ARGUMENT, "unknown dtype " + std::to_string(dt));
    if (!valid_layout(layout)) return fail(TG_ERR_INVALID_ARGUMENT, "unknown layout " + std::to_string(layout));
    if (batch < 0 || m < 0 || n < 0 || k < 0)
        return fail(TG_ERR_DIMENSION_MISMATCH,
                    "negative dimension: batch=" + std::to_string(batch) + " m=" + std::to_string(m) +
                        " n=" + std::to_string(n) + " k=" + std::to_string(k));
    if (m > 0x7fffffffLL || n > 0x7fffffffLL || k > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "dimension exceeds 2^31-1 (argmax is int32)");
    const int64_t out = m * n;
    if (batch > 0 && out > 0) {
        if (C == nullptr) return fail(TG_ERR_INVALID_ARGUMENT, "C is NULL");
        if (k > 0 && (A == nullptr || B == nullptr))
            return fail(TG_ERR_INVALID_ARGUMENT, "A or B is NULL");
    }
    if (strided && batch > 1) {
        if (sc < out)
            return fail(TG_ERR_DIMENSION_MISMATCH,
                        "stride_c (" + std::to_string(sc) + ") < m*n (" + std::to_string(out) +
                            "): output matrices would overlap");
        if (sa < 0 || sb < 0) return fail(TG_ERR_DIMENSION_MISMATCH, "negative input stride");
    }
    return TG_OK;
}

// Layout mapping: a column-major product C = A (x) B is the row-major
// product C^T = B^T (x) A^T over the same buffers (kernels.rs:370-430).
Problem make_problem(tg_layout layout, const void* A, const void* B, void* C, int32_t* argmax,
                     int64_t batch, int64_t m, int64_t n, int64_t k, int64_t sa, int64_t sb,
                     int64_t sc, bool strided) {
    Problem p;
    if (layout == TG_ROW_MAJOR) {
        p = Problem{A, B, C, argmax, batch, m, n, k, sa, sb, sc};
    } else {
        p = Problem{B, A, C, argmax, batch, n, m, k, sb, sa, sc};
    }
    if (!strided) {
        p.sA = p.M * p.K;
        p.sB = p.K * p.N;
        p.sC = p.M * p.N;
    }
    return p;
}

// True when pl's workspace is a gain and not a need: without one the product
// runs on the generic tiles, which read none.  Callers that share one workspace
// (tg_gemm_noalloc) or would have to allocate it inside a capture use those.
// Value-only f64 that the 64 x 128 tiles can run needs it either way (operand
// classes).
bool workspace_optional(tg_semiring sr, tg_dtype dt, const Problem& p, const Plan& pl) {
    switch (pl.path) {
        case Path::DL_ELEM_8:
        case Path::DL64S:
        case Path::DL64S_I64: break;
        case Path::DL64S_VALUE:
            if (dl64_tiles(p) >= 256 &&
                tg::dl64_fits(p.M, p.N, p.K, p.sA, p.sB, p.sC, p.A, p.B, p.C, p.IDX))
                return false;
            break;
        default: return false;
    }
    return !uses_workspace(plan_gemm(sr, dt, p, 0), p.IDX != nullptr);
}

// Whether an optional workspace of this size pays when the call itself has to
// allocate and free it: about 8 us for a call that is waited for while the
// stream's pool keeps it between synchronisations (up to 2 MB), beyond that
// 25 us and 2.5 us per MB (MI355X), against what the path gains.  us, with the
// allocation / without a workspace: f32 argmax 1000 x 1001 x 97 (0.4 MB) 46 / 59,
// 16 x (64 x 1025 x 97) 78 / 60, 500 x (65 x 65 x 200) 206 / 189, 50000 x 50 x 384
// 303 / 187; i32, whose exact mode is the faster one, 64 x (33 x 65 x 97) 52 / 44,
// 30 x (129 x 131 x 255) 106 / 97; f64 argmax 1500^2 x 300 176 / 163, x 512 225 /
// 264, 128 x (128 x 128 x 512) 306 / 190, value-only 1000^2 x 257 63 / 55, 300 x
// 5000 x 384 104 / 97; i64 argmax 1500^2 x 188 170 / 161, x 300 216 / 245, 1000^3
// 231 / 267, 256 x (64 x 64 x 1000) 330 / 268.
bool allocation_pays(tg_semiring sr, tg_dtype dt, const Problem& p, size_t bytes) {
    constexpr size_t kMB = size_t(1) << 20;
    const int64_t narrow = p.M < p.N ? p.M : p.N;
    if (p.IDX == nullptr) return p.K >= (narrow >= 512 ? 300 : 400);
    if (bytes <= 2 * kMB) return dt != TG_I32 || p.K >= 128;
    const double products = double(p.batch) * double(p.M) * double(p.N) * double(p.K);
    if (dt == TG_F64) return narrow >= 256 && products >= 8e8;
    if (dt == TG_I64) return narrow >= 256 && (p.K >= 800 || (sr != TG_MAXMUL && products >= 5.5e8));
    return p.K >= (dt == TG_I32 ? 320 : 256) ? bytes <= 64 * kMB || narrow >= 128 : narrow >= 512;
}

// Bytes that tg_gemm allocates for the call: the full workspace, for the
// kernels that read it.  *optional: the product can run without.
size_t own_workspace(tg_semiring sr, tg_dtype dt, const Problem& p, bool* optional) {
    *optional = false;
    const bool argmax = p.IDX != nullptr;
    const size_t bytes = workspace_bytes_for(dt, p.batch, p.M, p.N, p.K, argmax);
    if (bytes == 0) return 0;
    const Plan pl = plan_gemm(sr, dt, p, bytes);
    if (!uses_workspace(pl, argmax)) return 0;
    *optional = workspace_optional(sr, dt, p, pl);
    return *optional && !allocation_pays(sr, dt, p, bytes) ? 0 : bytes;
}

int gemm_impl(int device, tg_semiring sr, tg_dtype dt, tg_layout layout, const void* A,
              const void* B, void* C, int32_t* argmax, int64_t batch, int64_t m, int64_t n,
              int64_t k, int64_t sa, int64_t sb, int64_t sc, bool strided, void* ws,
              size_t ws_bytes, bool ws_given, void* stream) {
    int rc = validate_forward(sr, dt, layout, A, B, C, batch, m, n, k, sa, sb, sc, strided);
    if (rc != TG_OK) return rc;
    const bool with_argmax = argmax != nullptr;
    const size_t need = bt_bytes_for(dt, batch, m, n, k, with_argmax);
    if (ws_given && need > 0) {
        if (ws == nullptr || ws_bytes < need)
            return fail(TG_ERR_INVALID_ARGUMENT, "workspace too small: need " + std::to_string(need) +
                                                     " bytes, got " + std::to_string(ws_bytes));
        if ((reinterpret_cast<uintptr_t>(ws) & 255u) != 0)
            return fail(TG_ERR_INVALID_ARGUMENT, "workspace must be 256-byte aligned");
    }
    // A workspace the split-K partials cannot use (none, or misaligned when
    // no B^T staging is needed) runs the product unsplit.
    if (ws_given && (ws == nullptr || (reinterpret_cast<uintptr_t>(ws) & 255u) != 0)) ws_bytes = 0;
    rc = select_device(device);
    if (rc != TG_OK) return rc;
    if (batch == 0 || m == 0 || n == 0) return TG_OK;
    hipStream_t st = as_stream(stream);

    Problem p = make_problem(layout, A, B, C, argmax, batch, m, n, k, sa, sb, sc, strided);

    // The kernels stage B^T (K x p.N per batch item) in the workspace.
    if (need > 0 && need < size_t(p.batch) * size_t(p.K) * size_t(p.N) * size_t(elem_size(dt)))
        return fail(TG_ERR_INVALID_ARGUMENT, "internal: workspace size below K x N");
    void* work = ws;
    bool own = false;
    if (!ws_given) {
        bool optional;
        ws_bytes = own_workspace(sr, dt, p, &optional);
        if (ws_bytes > 0 && optional) {
            // Under capture such a product runs without: no allocation nodes.
            hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
            if (hipStreamIsCapturing(st, &cap) != hipSuccess) (void)hipGetLastError();
            if (cap != hipStreamCaptureStatusNone) ws_bytes = 0;
        }
        if (ws_bytes > 0) {
            TG_HIP(hipMallocAsync(&work, ws_bytes, st));
            own = true;
        }
    }
    rc = run_gemm(sr, dt, p, work, ws_given || own ? ws_bytes : 0, st);
    if (own) {
        hipError_t e = hipFreeAsync(work, st);
        if (rc == TG_OK && e != hipSuccess) return hip_fail(e, "hipFreeAsync");
    }
    return rc;
}

tg::SmallProblem small_problem(tg_semiring sr, tg_dtype dt, const Problem& p) {
    return tg::SmallProblem{int(sr), int(dt), p.A, p.B, p.C, p.IDX, p.batch, p.M, p.N, p.K,
                            p.sA, p.sB, p.sC};
}

int64_t tiles64_of(const Problem& p) { return ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.batch; }

// True when the few-output kernel is the faster one for any number of outputs
// up to 64 columns wide at K <= 32.  The others write 256-column (short K, for
// aligned columns) or 64-column tiles, mostly padding there, but short K makes
// the outputs themselves the bound, which they write in longer runs.  us on
// MI355X, small / other:
//   aligned, argmax: f32 524288 x 64 x 2 114 / 60, x 8 160 / 128, x 12 170 / 190;
//     N <= 32 from K = 2; value-only from K = 3 beyond 32 columns (f64 524288 x 64
//     x 1 65 / 53), batches of few rows from 12 (f32 5000 x (48 x 48 x 8) 54 / 44, x
//     16 31 / 66);
//   any columns, argmax: beyond 32 never (524288 x 33 f32 x 32 182 / 125, f64 x 24
//     299 / 162); up to 16 f32 524288 x 3 x 2 48 / 30, x 12 47 / 54, f64 x 9 x 8
//     61 / 84; between, f32 x 21 x 24 99 / 96, x 32 107 / 115, f64 65536 x 30 x 12
//     15 / 18, x 17 x 17 22 / 20; value-only beyond 32 up to K = 16 (524288 x 50 f64
//     x 12 86 / 143, x 32 250 / 209).
bool small_takes_narrow(tg_dtype dt, const Plan& pl, const Problem& p) {
    const bool aligned = pl.path == Path::SHORTK, wide = dt == TG_F64 || dt == TG_I64;
    if (p.IDX == nullptr) {
        if (p.N <= 32) return true;
        return aligned ? p.K >= (p.batch > 1 && p.M < 64 ? 12 : 3) : p.K <= 16;
    }
    if (aligned) return p.K >= (p.N <= 32 ? 2 : 12);
    if (p.N <= 16) return p.K >= (wide ? 5 : 10);
    if (p.N <= 32) return wide ? p.K <= 16 : dt == TG_F32 && p.K >= 28;
    return false;
}

// True when a 32-bit product whose K the direct-to-LDS kernel splits over the
// whole chip (into launches, with a merge) is past the few-output kernel's K: a
// tile's waves there are at most 16.  us on MI355X, small / split, by K times
// the outputs of the split kernel's tiles: value-only f32 256^2 x 4096 (2.7e8)
// 19 / 29, x 8192 37 / 34, 512^2 x 1024 19 / 25, x 2048 (5.4e8) 33 / 27, 700^2 x 1024
// (5.1e8) 36 / 26, 128^2 x 32768 (5.4e8) 53 / 65, x 65536 99 / 82; argmax 256^2 x
// 8192 (5.4e8) 51 / 57, x 16384 96 / 82, i32 29 / 43 at 4096 (2.7e8), 75 / 66 at
// 8192.  One tile, value-only: 64^2 x 32768 52 / 67, x 65536 101 / 101, i32 98 /
// 84.  Up to 16 rows or columns that is mostly padding: 16 x 256 x 32768
// value-only 59 / 69, x 65536 115 / 88, 16^2 x 65536 argmax 72 / 113, x 262144 263 /
// 239.
bool split_outruns_small(const Plan& pl, const Problem& p) {
    const bool argmax = p.IDX != nullptr;
    const bool slices_ok = pl.path == Path::DL_44_8 || pl.path == Path::DL_44_16;
    if (pl.splits <= 1 || wg_slices(slices_ok, argmax, pl.splits, p.K) > 0) return false;
    const int64_t tiles64 = tiles64_of(p);
    if (tiles64 * pl.splits < 256) return false;
    if (p.M <= 16 || p.N <= 16) return p.K > (argmax ? 65536 : 32768);
    return (!argmax && p.K > 49152) ||
           double(p.K) * double(tiles64 * 4096) > (argmax ? 4.5e8 : 3.5e8);
}

// small_output_limit where the other kernel is the generic one or that of the
// 64-bit 64 x 64 tiles.  The generic tiles' time goes by their number, the few-output
// kernel's by the outputs, so full tiles and many items draw the line earlier, and
// K below 64 earliest (its first and last step weigh most).  us on MI355X, small /
// other:
//   32-bit: 42 x (452 x 92 x 52) f32 argmax 23 / 28, 2001^2 x 60 45 / 41; 47500 x 40 x
//     33 f32 argmax 29 / 22, x 64 1.10 times; i32 MaxMul 100 x 11000 x 33 18 / 16, 100 x
//     15000 x 64 26 / 24;
//   f64 argmax (the exact mode there has no window loads): 700^3 79 / 111, 1024^3
//     207 / 149, 256 x (64 x 64 x 300) 93 / 64, 1000^2 x 300 69 / 63, 300 x 5000 x 300
//     128 / 104, 256 x (65 x 65 x 300) 140 / 216, 475 x (41 x 41 x 33) 24 / 18, x 128 1.07
//     and x 200 1.00 times, 1784 x (41 x 41 x 128) 186 / 157;
//   f64 value-only: 700^3 54 / 78, 1024^3 147 / 111, 300 x 5000 x 300 80 / 70, 100 x
//     16384 x 257 75 / 61; below K = 192 100 x 15000 x 64 25 / 18, 1378 x 1379 x 128
//     38 / 35, 67 x (128 x 128 x 64) 19 / 17;
//   i64 argmax: 1536^2 x 768 340 / 365, 2047 x 2049 x 1025 780 / 803, 2048^3 1490 /
//     1160, in the exact mode's range 2048^2 x 80 83 / 95, 15000 x 40 x 33 17 / 14;
//     full tiles 1220 x (64 x 64 x 200) 286 / 270; MaxMul 100 x 15000 x 64 1.11 times,
//     full tiles 1220 x (64 x 64 x 161) 279 / 231, 100 x 50000 x 200 0.90 times;
//   i64 value-only: 2047 x 2049 x 1025 586 / 652, 3001^2 x 300 388 / 349, 732 x (64 x 64 x
//     400) 200 / 184, 128 x (128 x 128 x 129) 53 / 47, 463 x (64 x 64 x 64) 25 / 23.
int64_t small_limit_generic(tg_semiring sr, tg_dtype dt, const Plan& pl, const Problem& p) {
    constexpr int64_t k1 = int64_t(1) << 10;
    const bool argmax = p.IDX != nullptr;
    const int64_t tiles64 = tiles64_of(p);
    if (dt == TG_F32 || dt == TG_I32) {
        if (!argmax || p.K >= 96) return 2048 * k1;
        return dt == TG_F32 ? 1536 * k1 : p.K < 48 ? 1024 * k1 : 1280 * k1;
    }
    if (dt == TG_F64) {
        if (pl.path == Path::TILES_CHUNKED) return 2048 * k1;
        if (!argmax) return p.K < 192 ? 768 * k1 : tiles64 <= 700 ? 1280 * k1 : 1828 * tiles64;
        if (p.K < 64 || tiles64 <= 256) return 512 * k1;
        const int64_t limit = (p.K < 200 ? 1600 : 2048) * tiles64;
        return limit < 1920 * k1 ? limit : 1920 * k1;
    }
    if (!argmax) return p.K < 96 ? 1280 * k1 : p.batch > 1 || p.K < 256 ? 2048 * k1 : 4096 * k1;
    if (p.K < (sr == TG_MAXMUL ? 64 : 48)) return 512 * k1;
    const bool full = double(p.batch) * double(p.M) * double(p.N) > 0.9 * 4096 * double(tiles64);
    if (sr == TG_MAXMUL) {
        if (p.K < 112) return 1280 * k1;
        if (full) return 1792 * k1;
    }
    if (full && p.batch > 1 && p.K >= 128) return 4096 * k1;
    return pl.path == Path::TILES_EXACT ? 8192 * k1 : 4096 * k1;
}

// Outputs (batch x M x N) below which the few-output kernel (tg_gemm_small.hpp)
// is the faster one, by the path the problem would take otherwise.  Measured
// on MI355X over 290 shapes of every dtype, with and without argmax (small /
// other path, us; limits where the ratio nears 1):
//   short K (<= 32): the other kernels are bound by the output writes, which
//     leave in 1 KB runs there: f32 argmax 252 x 1672 x 18 8.6 / 8.7, 800 x
//     672 x 16 9.7 / 7.5; value-only 800 x 672 x 16 5.4 / 6.8, 368 x 4848 x 16
//     7.7 / 6.6.  Their 256-column tiles are mostly padding for narrow N:
//     262144 x 16 x 16 argmax 29 / 114.
//   direct-to-LDS and K-resident (32-bit, aligned): 768^3 f32 argmax 39 / 49,
//     1024^3 84 / 59; i32 5376 x 64 x 64 9.6 / 9.5.
//   direct-to-LDS with element loads (32-bit): f32 argmax 701^3 37 / 54, 734 x
//     1071 x 3636 232 / 180, 1001^3 102 / 76; value-only 701^3 27 / 29, 734 x
//     1071 x 3636 195 / 136 (i32 198 / 186); unsliced 1500^2 x 150 47 / 46.
//   any short K (i32): 10000 x 20 x 20 8.6 / 6.8, 5000 x 32 x 32 6.6 / 6.9,
//     5000 x 48 x 48 7.1 / 9.9, 10000 x 48 x 48 11.9 / 10.2, 5000 x 100 x 100
//     14 / 17, 10000 x 100 x 100 21 / 18, 5000 x 160 x 160 20.4 / 20.4, 5000 x
//     256 x 256 43 / 40.
//   K slices in one workgroup on most of the CUs: 256 x (48 x 48 x 512) argmax f32
//     53 / 46, i32 62 / 52, 64 x (48 x 48 x 512) 21 / 37, 700^2 x 1024 45 / 52.
int64_t small_output_limit(tg_semiring sr, tg_dtype dt, const Plan& pl, const Problem& p) {
    constexpr int64_t k1 = int64_t(1) << 10;
    const bool argmax = p.IDX != nullptr;
    const int64_t narrow = p.M < p.N ? p.M : p.N;
    if (pl.path == Path::KRESG)
        return p.K <= 32 ? 192 * k1 : p.K <= 48 ? 384 * k1 : p.K <= 160 ? 768 * k1 : 1280 * k1;
    if (p.K <= 32) {
        if (p.N <= 64 && small_takes_narrow(dt, pl, p)) return INT64_MAX;
        return !argmax ? 512 * k1 : dt == TG_F64 ? 128 * k1 : 256 * k1;
    }
    // Few rows of the short-K kernel's wide tiles, which it writes in 1 KB runs
    // (3 x 524288 x 33 value-only 43 / 28, 16 rows 40 / 30).
    if (pl.path == Path::SHORTK && p.N > 16) return 512 * k1;
    if (split_outruns_small(pl, p)) return 0;
    if (narrow <= 16) return INT64_MAX;  // tiles of the other kernels are mostly padding
    switch (pl.path) {
        case Path::SHORTK: return 512 * k1;
        case Path::KRESW:
        case Path::KRES8:
        case Path::KRES: return dt == TG_I32 ? 256 * k1 : 512 * k1;
        case Path::DL64:
        case Path::DL64_VALUE: return 2048 * k1;
        case Path::DL64S:
        case Path::DL64S_VALUE: return narrow <= 32 ? 2048 * k1 : 768 * k1;
        case Path::DL64S_I64:
        case Path::DL64S_I64_VALUE:
        case Path::TILES_EXACT:
        case Path::TILES_CHUNKED:
        case Path::TILES: break;
        case Path::DL_ELEM_8:
        case Path::DL_ELEM_16:
        case Path::DL_ELEM:
            if (narrow <= 32 || (argmax && p.K < 256)) return 2048 * k1;
            if (pl.slices == 1) return 1280 * k1;
            return argmax ? 640 * k1 : dt == TG_F32 ? 512 * k1 : 768 * k1;
        default:  // direct-to-LDS, 32-bit
            if (narrow <= 32) return 2048 * k1;
            return p.K < 256 ? 512 * k1 : pl.splits > 1 && tiles64_of(p) > 160 ? 448 * k1 : 640 * k1;
    }
    return small_limit_generic(sr, dt, pl, p);
}

// What tg_gemm_small runs: `form` is the few-output kernel's launch.
enum class Small { NONE, FEW, KRESG };

Small choose_small(tg_semiring sr, tg_dtype dt, const Problem& p, tg::SmallForm* form) {
    if (p.batch <= 0 || p.M <= 0 || p.N <= 0 || p.K <= 0) return Small::NONE;
    Plan pl = plan_gemm(sr, dt, p, workspace_bytes_for(dt, p.batch, p.M, p.N, p.K,
                                                       p.IDX != nullptr));
    // tg_gemm_kresw, one 16-wave workgroup per CU and one batch item after the
    // other, while an item's wave tiles do not give each of the chip's waves
    // more than one (us, kresw / kresg: 4096 x 1024 x 128 36 / 25, 32768 x 128 x
    // 64 22 / 14, 8 x (4096 x 128 x 128) 251 / 28; 16384 x 512 x 128 40 / 45).
    const bool few_wave_tiles = pl.path == Path::KRESW && takes_kresg(p) &&
                                tg::kresg_wave_tiles(p.M, p.N) <= 4096;
    if (few_wave_tiles) pl.path = Path::KRESG;
    // In floating point: batch * M * N of a caller's sizes may pass 2^63.
    if (double(p.batch) * double(p.M) * double(p.N) < double(small_output_limit(sr, dt, pl, p)) &&
        tg::small_form(small_problem(sr, dt, p), form))
        return Small::FEW;
    return few_wave_tiles ? Small::KRESG : Small::NONE;
}

// ----------------------------------------------------------------------------
// Workspace without allocation (tg_gemm_noalloc)
// ----------------------------------------------------------------------------

// The workspace of tg_gemm_noalloc: one fixed array in the code object's
// zero-initialised device data.  Each device that loads the library holds its
// own copy from the module's load until the process ends.  On the host the
// name `scratch` is only a stand-in, never a device address: host code uses
// the address hipGetSymbolAddress returns for the current device
// (scratch_address), in kernel arguments as everywhere else.
constexpr size_t kScratchBytes = TG_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kScratchMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchMaxDevices] = {};

// Device address of `scratch` on `device`, which must be the current device.
// Looked up once per device (tg_context_init, or the first tg_gemm_noalloc
// call on that device) and kept.
int scratch_address(int device, void** out) {
    if (device < 0 || device >= kScratchMaxDevices)
        return fail(TG_ERR_INVALID_ARGUMENT,
                    "tg_gemm_noalloc supports devices 0.." + std::to_string(kScratchMaxDevices - 1));
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device] == nullptr) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (ptr == nullptr) return fail(TG_ERR_DRIVER, "hipGetSymbolAddress(scratch) returned NULL");
        g_scratch_ptr[device] = ptr;
    }
    *out = g_scratch_ptr[device];
    return TG_OK;
}

// Plan of a tg_gemm_noalloc call, with kScratchBytes as the workspace, so
// split K is only chosen when its partials fit.  Every call shares the scratch,
// so a product that can run without it does (*ws_bytes is 0 then): such calls
// may overlap.
Plan scratch_plan(tg_semiring sr, tg_dtype dt, const Problem& p, size_t* ws_bytes) {
    *ws_bytes = kScratchBytes;
    const Plan pl = plan_gemm(sr, dt, p, kScratchBytes);
    if (!workspace_optional(sr, dt, p, pl)) return pl;
    *ws_bytes = 0;
    return plan_gemm(sr, dt, p, 0);
}

// Scratch bytes the planned path reads (0 when it reads none).  B^T staging
// alone may exceed the scratch.
size_t scratch_need(tg_dtype dt, const Problem& p, const Plan& pl) {
    const bool argmax = p.IDX != nullptr;
    if (!uses_workspace(pl, argmax)) return 0;
    // The f64 direct-to-LDS kernel's workspace: B^T (argmax) and the operand
    // classes of A's rows and B's columns (run_gemm_dl64).
    if (pl.path == Path::DL64 || pl.path == Path::DL64_VALUE || pl.path == Path::DL64S ||
        pl.path == Path::DL64S_VALUE)
        return dl64_ws_bytes(p.batch, p.M, p.N, p.K, argmax);
    return ws_layout(dt, p.batch, p.M, p.N, p.K, argmax, pl.splits).total;
}

// ----------------------------------------------------------------------------
// Backward
// ----------------------------------------------------------------------------

// Launch geometry of the deterministic backward kernels (tg_backward.hpp).
// Both kernels loop over their rows / column groups with a grid stride, so
// the grid is capped (kBwdMaxGrid workgroups) and no dimension of a launch
// grows with M, N or the batch.
constexpr int64_t kBwdMaxGrid = 16384;
constexpr size_t kBwdLdsBudget = 128 * 1024;  // bins of one grad_A row at most
constexpr size_t kBwdLdsLimit = 160 * 1024;   // the CU's LDS
// grad_B takes its keys in passes (8 columns per group) when the columns'
// bins do not fit eight at a time, a pass re-reads no more bytes than it
// writes (the group's M rows of index and dC against its keys' gradients)
// and there are at most kBwdMaxPasses of them.  Measured (bit-identical,
// f32 unless noted): 1024 x 4096 x 32768 770 -> 220 us, x 16384 227 -> 107,
// f64 1024 x 4096 x 16384 550 -> 206; 4096 x 1024 x 16384 (re-reads twice
// the writes) 93 -> 129 and 62 passes at K = 262144 1.05 -> 1.39 ms, hence
// the two limits.
constexpr int64_t kBwdMaxPasses = 16;

struct BwdGeometry {
    bool global = false;  // bins in the gradient itself (K too large for LDS)
    int waves = 1;        // waves per workgroup
    size_t lds = 0;       // dynamic LDS bytes per workgroup
    int64_t grid = 0;     // workgroups
    int64_t groups_n = 0; // grad_B: column groups per batch item
    int64_t groups = 0;   // grad_B: column groups in total
    int64_t kp = 0;       // grad_B: keys per pass (K: one pass)
};

// grad_A: one wave per row; a wave's LDS is its row's K bins plus its stage
// (tg::kRowStageElems elements).  Four waves per workgroup while that is at
// most 8 KB, two while at most 16 KB, else one (18 KB at K = 4096 f32: eight
// workgroups per CU); global bins beyond the LDS budget.
BwdGeometry bwd_rows_geometry(int64_t rows, int64_t K, size_t es) {
    BwdGeometry g;
    const size_t row_bytes = size_t(K) * es;
    const size_t stage_bytes = size_t(tg::kRowStageElems) * es;
    const size_t wave_bytes = row_bytes + stage_bytes;
    if (row_bytes > kBwdLdsBudget) {
        g.global = true;
        g.waves = 4;
    } else {
        g.waves = wave_bytes <= 8 * 1024 ? 4 : wave_bytes <= 16 * 1024 ? 2 : 1;
    }
    g.lds = size_t(g.waves) * (g.global ? stage_bytes : wave_bytes);
    const int64_t need = (rows + g.waves - 1) / g.waves;
    g.grid = need < kBwdMaxGrid ? need : kBwdMaxGrid;
    return g;
}

// grad_B: one wave per column, W <= 8 adjacent columns per workgroup: the
// most whose bins, the staged tiles of argmax and dC (tg::kBwdTileRows x W)
// and the waves' stages fit the CU's 160 KB (8 at K = 4096 f32: 154 KB).
// Longer columns over few rows keep 8 columns and take their keys in passes
// (kp: keys per pass, see kBwdMaxPasses); otherwise fewer columns, and
// global bins when not even one column's fit.
BwdGeometry bwd_cols_geometry(int64_t batch, int64_t M, int64_t N, int64_t K, size_t es) {
    BwdGeometry g;
    auto lds_for = [&](int64_t w, int64_t kp, bool global) {
        return (global ? 0 : size_t(w) * size_t(kp) * es) +
               size_t(tg::kBwdTileRows) * size_t(w + 1) * (4 + es) +
               size_t(w) * size_t(tg::kStageElems) * es;
    };
    g.kp = K;
    // Keys per pass with 8 columns: what the LDS holds, a multiple of 4.
    const size_t fixed8 = lds_for(8, 0, false);
    const int64_t kp8 = int64_t((kBwdLdsLimit - fixed8) / (8 * es)) & ~int64_t(3);
    const bool one_pass = lds_for(8, K, false) <= kBwdLdsLimit;
    const int64_t passes = kp8 > 0 ? (K + kp8 - 1) / kp8 : 0;
    if (!one_pass && kp8 > 0 && M * int64_t(4 + es) <= kp8 * int64_t(es) &&
        passes <= kBwdMaxPasses) {
        // Long columns, few rows: 8 columns in passes over the keys.
        g.kp = kp8;
        g.waves = 8;
        g.lds = lds_for(8, kp8, false);
    } else {
        int64_t w = size_t(K) * es > kBwdLdsBudget ? 0 : 8;
        while (w >= 1 && lds_for(w, K, false) > kBwdLdsLimit) --w;
        if (w < 1) {
            g.global = true;
            w = 8;
        }
        g.waves = int(w);
        g.lds = lds_for(w, K, g.global);
    }
    const int64_t w = g.waves;
    g.groups_n = (N + w - 1) / w;
    g.groups = batch * g.groups_n;
    g.grid = g.groups < kBwdMaxGrid ? g.groups : kBwdMaxGrid;
    return g;
}

// Raises a kernel's dynamic LDS limit once (needed above 64 KB).
template <typename K>
int allow_lds(K* kernel, size_t bytes) {
    if (bytes <= 64 * 1024) return TG_OK;
    TG_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes)));
    return TG_OK;
}

// A gradient with no contributions (the product has no rows or no columns):
// `batch` matrices of len elements, stride apart, all +0.  The scatter
// kernels would read their first (clamped) contribution at index -1.
template <typename T>
int zero_gradient(T* out, int64_t len, int64_t batch, int64_t stride, hipStream_t st) {
    const int64_t total = len * batch;
    if (total == 0) return TG_OK;
    if ((batch == 1 || stride == len) && (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
        // One contiguous run: 16-byte stores.
        const int64_t bytes = total * int64_t(sizeof(T));
        int64_t blocks = (bytes / 16 + 255) / 256;
        if (blocks > 8192) blocks = 8192;
        if (blocks < 1) blocks = 1;
        hipLaunchKernelGGL(tg::tg_fill_zero, dim3(unsigned(blocks)), dim3(256), 0, st,
                           reinterpret_cast<unsigned char*>(out), bytes);
        TG_HIP(hipGetLastError());
        return TG_OK;
    }
    int64_t bx = (len + 255) / 256;
    if (bx > 4096) bx = 4096;
    const int64_t by = batch < 65535 ? batch : 65535;
    hipLaunchKernelGGL((tg::tg_fill_zero_runs<T>), dim3(unsigned(bx), unsigned(by)), dim3(256), 0, st,
                       out, len, batch, stride);
    TG_HIP(hipGetLastError());
    return TG_OK;
}

template <typename T, bool MULT>
int run_backward_rows(const T* G, const int32_t* I, const T* O, T* GA, int64_t batch, int64_t M,
                      int64_t N, int64_t K, int64_t sC, int64_t sO, int64_t sA, hipStream_t st) {
    if (N == 0) return zero_gradient(GA, M * K, batch, sA, st);
    const BwdGeometry g = bwd_rows_geometry(batch * M, K, sizeof(T));
    if (g.grid == 0) return TG_OK;
    if (g.global) {
        hipLaunchKernelGGL((tg::tg_bwd_rows<T, MULT, true>), dim3(unsigned(g.grid)),
                           dim3(64 * g.waves), g.lds, st, G, I, O, GA, M, N, K, sC, sO, sA,
                           batch * M);
    } else {
        int rc = allow_lds(&tg::tg_bwd_rows<T, MULT, false>, g.lds);
        if (rc != TG_OK) return rc;
        hipLaunchKernelGGL((tg::tg_bwd_rows<T, MULT, false>), dim3(unsigned(g.grid)),
                           dim3(64 * g.waves), g.lds, st, G, I, O, GA, M, N, K, sC, sO, sA,
                           batch * M);
    }
    TG_HIP(hipGetLastError());
    return TG_OK;
}

template <typename T, bool MULT>
int run_backward_cols(const T* G, const int32_t* I, const T* O, T* GB, int64_t batch, int64_t M,
                      int64_t N, int64_t K, int64_t sC, int64_t sO, int64_t sB, hipStream_t st) {
    if (M == 0) return zero_gradient(GB, K * N, batch, sB, st);
    const BwdGeometry g = bwd_cols_geometry(batch, M, N, K, sizeof(T));
    if (g.grid == 0) return TG_OK;
    if (g.global) {
        // The bins are grad_B itself, zero-filled first in one coalesced
        // pass (1024 x 4096 x 65536 f32: 1.76 ms with each wave zeroing its
        // column, 0.48 ms this way).
        int rc = zero_gradient(GB, K * N, batch, sB, st);
        if (rc != TG_OK) return rc;
        rc = allow_lds(&tg::tg_bwd_cols<T, MULT, true>, g.lds);
        if (rc != TG_OK) return rc;
        hipLaunchKernelGGL((tg::tg_bwd_cols<T, MULT, true>), dim3(unsigned(g.grid)),
                           dim3(64 * g.waves), g.lds, st, G, I, O, GB, M, N, K, sC, sO, sB,
                           g.groups_n, g.groups, g.kp);
    } else {
        int rc = allow_lds(&tg::tg_bwd_cols<T, MULT, false>, g.lds);
        if (rc != TG_OK) return rc;
        hipLaunchKernelGGL((tg::tg_bwd_cols<T, MULT, false>), dim3(unsigned(g.grid)),
                           dim3(64 * g.waves), g.lds, st, G, I, O, GB, M, N, K, sC, sO, sB,
                           g.groups_n, g.groups, g.kp);
    }
    TG_HIP(hipGetLastError());
    return TG_OK;
}

// which: 0 = grad wrt the left operand (rows of C), 1 = wrt the right operand.
// Operates on the row-major problem.
template <typename T>
int run_backward_typed(int which, bool mult, const void* G, const int32_t* I, const void* O,
                       void* OUT, int64_t batch, int64_t M, int64_t N, int64_t K, int64_t sC,
                       int64_t sO, int64_t sOut, hipStream_t st) {
    const T* g = static_cast<const T*>(G);
    const T* o = static_cast<const T*>(O);
    T* out = static_cast<T*>(OUT);
    if (which == 0) {
        if (mult) return run_backward_rows<T, true>(g, I, o, out, batch, M, N, K, sC, sO, sOut, st);
        return run_backward_rows<T, false>(g, I, o, out, batch, M, N, K, sC, sO, sOut, st);
    }
    if (mult) return run_backward_cols<T, true>(g, I, o, out, batch, M, N, K, sC, sO, sOut, st);
    return run_backward_cols<T, false>(g, I, o, out, batch, M, N, K, sC, sO, sOut, st);
}

// Public-level backward: `want_a` selects grad wrt A (else B); `other` is B
// (for grad A) or A (for grad B) under the MaxMul rule, NULL otherwise.
int backward_impl(int device, tg_dtype dt, tg_layout layout, bool want_a, const void* grad_c,
                  const int32_t* argmax, const void* other, void* out, int64_t batch, int64_t m,
                  int64_t n, int64_t k, int64_t s_c, int64_t s_other, int64_t s_out, bool strided,
                  bool mult, void* stream) {
    if (!valid_dtype(dt)) return fail(TG_ERR_INVALID_ARGUMENT, "unknown dtype " + std::to_string(dt));
    if (dt != TG_F32 && dt != TG_F64)
        return fail(TG_ERR_UNSUPPORTED, std::string("backward is defined for f32/f64 only, got ") +
                                            dtype_name(dt));
    if (!valid_layout(layout)) return fail(TG_ERR_INVALID_ARGUMENT, "unknown layout " + std::to_string(layout));
    if (batch < 0 || m < 0 || n < 0 || k < 0) return fail(TG_ERR_DIMENSION_MISMATCH, "negative dimension");
    if (m > 0x7fffffffLL || n > 0x7fffffffLL || k > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "dimension exceeds 2^31-1");
    const int64_t out_elems = want_a ? m * k : k * n;
    if (batch > 0 && out_elems > 0 && out == nullptr)
        return fail(TG_ERR_INVALID_ARGUMENT, "gradient output is NULL");
    if (batch > 0 && m * n > 0 && (grad_c == nullptr || argmax == nullptr))
        return fail(TG_ERR_INVALID_ARGUMENT, "grad_c or argmax is NULL");
    if (mult && batch > 0 && m * n > 0 && k > 0 && other == nullptr)
        return fail(TG_ERR_INVALID_ARGUMENT, "MaxMul backward needs the other operand");
    if (strided && batch > 1) {
        if (s_out < out_elems)
            return fail(TG_ERR_DIMENSION_MISMATCH, "gradient stride smaller than one matrix");
        if (s_c < 0 || s_other < 0) return fail(TG_ERR_DIMENSION_MISMATCH, "negative stride");
    }
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    if (batch == 0 || out_elems == 0) return TG_OK;
    if (!strided) {
        s_c = m * n;
        s_other = want_a ? k * n : m * k;
        s_out = out_elems;
    }
    hipStream_t st = as_stream(stream);
    // Row-major problem C (M x N) = L (M x K) (x) R (K x N).  Column-major
    // data is the row-major transposed problem C^T = B^T (x) A^T, in which
    // A's gradient is the right operand's gradient and vice versa.
    int which;
    int64_t M, N;
    if (layout == TG_ROW_MAJOR) {
        which = want_a ? 0 : 1;
        M = m;
        N = n;
    } else {
        which = want_a ? 1 : 0;
        M = n;
        N = m;
    }
    if (dt == TG_F32)
        return run_backward_typed<float>(which, mult, grad_c, argmax, other, out, batch, M, N, k,
                                         s_c, s_other, s_out, st);
    return run_backward_typed<double>(which, mult, grad_c, argmax, other, out, batch, M, N, k, s_c,
                                      s_other, s_out, st);
}

}  // namespace

// ============================================================================
// Exported C ABI
// ============================================================================

extern "C" {

int tg_version(void) { return kAbiVersion; }

const char* tg_status_string(int status) {
    switch (status) {
        case TG_OK: return "success";
        case TG_ERR_DRIVER: return "HIP driver/runtime error";
        case TG_ERR_COMPILE: return "kernel compilation error";
        case TG_ERR_NO_DEVICE: return "no HIP device available";
        case TG_ERR_DIMENSION_MISMATCH: return "dimension mismatch";
        case TG_ERR_KERNEL_NOT_FOUND: return "kernel not found";
        case TG_ERR_INVALID_ARGUMENT: return "invalid argument";
        case TG_ERR_UNSUPPORTED: return "unsupported operation";
    }
    return "unknown status";
}

const char* tg_last_error(void) { return g_last_error.c_str(); }

int tg_device_count(int* count) {
    if (count == nullptr) return fail(TG_ERR_INVALID_ARGUMENT, "count is NULL");
    return device_count_cached(count);
}

int tg_context_init(int device) {
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    TG_HIP(hipFree(nullptr));  // forces runtime/context initialisation
    if (device < kScratchMaxDevices) {  // tg_gemm_noalloc's workspace address
        void* unused = nullptr;
        rc = scratch_address(device, &unused);
        if (rc != TG_OK) return rc;
    }
    return TG_OK;
}

int tg_device_name(int device, char* buf, size_t len) {
    if (buf == nullptr || len == 0) return fail(TG_ERR_INVALID_ARGUMENT, "buffer is NULL");
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    hipDeviceProp_t prop;
    TG_HIP(hipGetDeviceProperties(&prop, device));
    std::snprintf(buf, len, "HIP Device %d (%s, %s)", device, prop.name, prop.gcnArchName);
    return TG_OK;
}

int tg_malloc(int device, void** ptr, size_t bytes) {
    if (ptr == nullptr) return fail(TG_ERR_INVALID_ARGUMENT, "ptr is NULL");
    *ptr = nullptr;
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    if (bytes == 0) return TG_OK;
    TG_HIP(hipMalloc(ptr, bytes));
    return TG_OK;
}

int tg_free(int device, void* ptr) {
    if (ptr == nullptr) return TG_OK;
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    TG_HIP(hipFree(ptr));
    return TG_OK;
}

int tg_memcpy_htod(int device, void* dst, const void* src, size_t bytes) {
    if (bytes == 0) return TG_OK;
    if (dst == nullptr || src == nullptr) return fail(TG_ERR_INVALID_ARGUMENT, "NULL pointer");
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    TG_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return TG_OK;
}

int tg_memcpy_dtoh(int device, void* dst, const void* src, size_t bytes) {
    if (bytes == 0) return TG_OK;
    if (dst == nullptr || src == nullptr) return fail(TG_ERR_INVALID_ARGUMENT, "NULL pointer");
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    TG_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return TG_OK;
}

int tg_memcpy_dtod(int device, void* dst, const void* src, size_t bytes, void* stream) {
    if (bytes == 0) return TG_OK;
    if (dst == nullptr || src == nullptr) return fail(TG_ERR_INVALID_ARGUMENT, "NULL pointer");
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    TG_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, as_stream(stream)));
    return TG_OK;
}

int tg_memset_zero(int device, void* ptr, size_t bytes, void* stream) {
    if (bytes == 0) return TG_OK;
    if (ptr == nullptr) return fail(TG_ERR_INVALID_ARGUMENT, "ptr is NULL");
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    return launch_fill_zero(ptr, bytes, as_stream(stream));
}

int tg_synchronize(int device) {
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    TG_HIP(hipDeviceSynchronize());
    return TG_OK;
}

int tg_stream_synchronize(int device, void* stream) {
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    TG_HIP(hipStreamSynchronize(as_stream(stream)));
    return TG_OK;
}

int tg_kernel_timing_enable(int on) {
    g_timing.store(on != 0);
    return TG_OK;
}

int tg_kernel_timing_read(double* total_ms, int64_t* launches) {
    if (total_ms == nullptr || launches == nullptr)
        return fail(TG_ERR_INVALID_ARGUMENT, "total_ms or launches is NULL");
    std::vector<std::pair<hipEvent_t, hipEvent_t>> evs;
    {
        std::lock_guard<std::mutex> lk(g_timing_mu);
        evs.swap(g_timing_events);
    }
    double sum = 0.0;
    int rc = TG_OK;
    for (auto& e : evs) {
        float ms = 0.0f;
        hipError_t err = hipEventSynchronize(e.second);
        if (err == hipSuccess) err = hipEventElapsedTime(&ms, e.first, e.second);
        if (err != hipSuccess && rc == TG_OK) rc = hip_fail(err, "hipEventElapsedTime");
        sum += ms;
        (void)hipEventDestroy(e.first);
        (void)hipEventDestroy(e.second);
    }
    *total_ms = sum;
    *launches = int64_t(evs.size());
    return rc;
}

int tg_gemm(int device, tg_semiring semiring, tg_dtype dtype, tg_layout layout, const void* A,
            const void* B, void* C, int32_t* argmax, int64_t m, int64_t n, int64_t k,
            void* stream) {
    return gemm_impl(device, semiring, dtype, layout, A, B, C, argmax, 1, m, n, k, 0, 0, 0, false,
                     nullptr, 0, false, stream);
}

int tg_gemm_small(int device, tg_semiring semiring, tg_dtype dtype, tg_layout layout,
                  const void* A, const void* B, void* C, int32_t* argmax, int64_t batch, int64_t m,
                  int64_t n, int64_t k, int64_t stride_a, int64_t stride_b, int64_t stride_c,
                  void* stream, int* ran) {
    if (ran == nullptr) return fail(TG_ERR_INVALID_ARGUMENT, "ran is NULL");
    *ran = 0;
    int rc = validate_forward(semiring, dtype, layout, A, B, C, batch, m, n, k, stride_a, stride_b,
                              stride_c, true);
    if (rc != TG_OK) return rc;
    const Problem p = make_problem(layout, A, B, C, argmax, batch, m, n, k, stride_a, stride_b,
                                   stride_c, true);
    tg::SmallForm form;
    const Small kernel = choose_small(semiring, dtype, p, &form);
    if (kernel == Small::NONE) return TG_OK;
    rc = select_device(device);
    if (rc != TG_OK) return rc;
    hipStream_t st = as_stream(stream);
    if (kernel == Small::KRESG) {
        rc = run_gemm_kresg(semiring == TG_MAXPLUS ? tg::SR_MAXPLUS : tg::SR_MINPLUS, p, st);
        if (rc != TG_OK) return rc;
    } else {
        KernelTimer timer(st);
        TG_HIP(tg::small_launch(small_problem(semiring, dtype, p), form, st));
    }
    *ran = 1;
    return TG_OK;
}

const char* tg_gemm_small_plan(tg_semiring semiring, tg_dtype dtype, tg_layout layout,
                               const void* A, const void* B, const void* C, const int32_t* argmax,
                               int64_t batch, int64_t m, int64_t n, int64_t k, int64_t stride_a,
                               int64_t stride_b, int64_t stride_c) {
    static thread_local std::string name;
    const bool strided = stride_a != 0 || stride_b != 0 || stride_c != 0;
    if (validate_forward(semiring, dtype, layout, A, B, C, batch, m, n, k, stride_a, stride_b,
                         stride_c, strided) != TG_OK)
        return "invalid";
    const Problem p = make_problem(layout, A, B, const_cast<void*>(C), const_cast<int32_t*>(argmax),
                                   batch, m, n, k, stride_a, stride_b, stride_c, strided);
    tg::SmallForm f;
    switch (choose_small(semiring, dtype, p, &f)) {
        case Small::NONE: return "none";
        case Small::KRESG: return "kresg";
        case Small::FEW: break;
    }
    name = std::to_string(4 * f.lr) + "x" + std::to_string(4 * f.lc) + " waves " +
           std::to_string(f.waves);
    return name.c_str();
}

int tg_gemm_noalloc(int device, tg_semiring semiring, tg_dtype dtype, tg_layout layout,
                    const void* A, const void* B, void* C, int32_t* argmax, int64_t m, int64_t n,
                    int64_t k, void* stream) {
    int rc = validate_forward(semiring, dtype, layout, A, B, C, 1, m, n, k, 0, 0, 0, false);
    if (rc != TG_OK) return rc;
    const Problem p = make_problem(layout, A, B, C, argmax, 1, m, n, k, 0, 0, 0, false);
    // Host-only planning first, so an oversized problem is rejected before
    // any device work.
    const bool empty = m == 0 || n == 0;
    size_t ws_bytes = 0;
    const Plan pl = empty ? Plan{} : scratch_plan(semiring, dtype, p, &ws_bytes);
    const size_t need = empty ? 0 : scratch_need(dtype, p, pl);
    if (need > kScratchBytes)
        return fail(TG_ERR_INVALID_ARGUMENT,
                    "tg_gemm_noalloc: this problem needs " + std::to_string(need) +
                        " bytes of workspace, above the fixed " + std::to_string(kScratchBytes) +
                        "-byte scratch; use tg_gemm or tg_gemm_ws");
    rc = select_device(device);
    if (rc != TG_OK) return rc;
    if (empty) return TG_OK;
    void* ws = nullptr;
    rc = scratch_address(device, &ws);
    if (rc != TG_OK) return rc;
    return run_gemm(semiring, dtype, p, ws, ws_bytes, as_stream(stream));
}

size_t tg_gemm_noalloc_bytes(tg_semiring semiring, tg_dtype dtype, tg_layout layout,
                             const void* A, const void* B, const void* C, const int32_t* argmax,
                             int64_t m, int64_t n, int64_t k) {
    if (validate_forward(semiring, dtype, layout, A, B, C, 1, m, n, k, 0, 0, 0, false) != TG_OK)
        return ~size_t(0);
    if (m == 0 || n == 0) return 0;
    const Problem p = make_problem(layout, A, B, const_cast<void*>(C), const_cast<int32_t*>(argmax),
                                   1, m, n, k, 0, 0, 0, false);
    size_t ws_bytes = 0;
    const Plan pl = scratch_plan(semiring, dtype, p, &ws_bytes);
    return scratch_need(dtype, p, pl);
}

size_t tg_gemm_alloc_bytes(tg_semiring semiring, tg_dtype dtype, tg_layout layout, const void* A,
                           const void* B, const void* C, const int32_t* argmax, int64_t batch,
                           int64_t m, int64_t n, int64_t k, int64_t stride_a, int64_t stride_b,
                           int64_t stride_c) {
    const bool strided = stride_a != 0 || stride_b != 0 || stride_c != 0;
    if (validate_forward(semiring, dtype, layout, A, B, C, batch, m, n, k, stride_a, stride_b,
                         stride_c, strided) != TG_OK)
        return ~size_t(0);
    if (batch == 0 || m == 0 || n == 0) return 0;
    const Problem p = make_problem(layout, A, B, const_cast<void*>(C), const_cast<int32_t*>(argmax),
                                   batch, m, n, k, stride_a, stride_b, stride_c, strided);
    bool optional;
    return own_workspace(semiring, dtype, p, &optional);
}

size_t tg_gemm_workspace_size(tg_dtype dtype, int64_t batch, int64_t m, int64_t n, int64_t k,
                              int with_argmax) {
    if (!valid_dtype(dtype)) return 0;
    return workspace_bytes_for(dtype, batch, m, n, k, with_argmax != 0);
}

const char* tg_gemm_plan(tg_semiring semiring, tg_dtype dtype, tg_layout layout, const void* A,
                         const void* B, const void* C, const int32_t* argmax, int64_t batch,
                         int64_t m, int64_t n, int64_t k, int64_t stride_a, int64_t stride_b,
                         int64_t stride_c, size_t workspace_bytes) {
    static thread_local std::string name;
    const bool strided = stride_a != 0 || stride_b != 0 || stride_c != 0;
    if (validate_forward(semiring, dtype, layout, A, B, C, batch, m, n, k, stride_a, stride_b,
                         stride_c, strided) != TG_OK)
        return "invalid";
    if (batch == 0 || m == 0 || n == 0) return "none";
    const Problem p = make_problem(layout, A, B, const_cast<void*>(C), const_cast<int32_t*>(argmax),
                                   batch, m, n, k, stride_a, stride_b, stride_c, strided);
    const Plan pl = plan_gemm(semiring, dtype, p, workspace_bytes);
    name = path_name(pl.path);
    const bool slices_ok = pl.path == Path::DL_44_8 || pl.path == Path::DL_44_16;
    if (const int s = wg_slices(slices_ok, argmax != nullptr, pl.splits, p.K))
        name += " slices " + std::to_string(s);
    else if (pl.slices > 1)
        name += " slices " + std::to_string(pl.slices);
    else if (pl.splits > 1)
        name += " split " + std::to_string(pl.splits);
    return name.c_str();
}

const char* tg_backward_plan(tg_dtype dtype, tg_layout layout, int want_a, int64_t batch,
                             int64_t m, int64_t n, int64_t k) {
    static thread_local std::string name;
    if ((dtype != TG_F32 && dtype != TG_F64) || !valid_layout(layout) || batch < 0 || m < 0 ||
        n < 0 || k < 0)
        return "invalid";
    const size_t es = size_t(elem_size(dtype));
    // Row-major problem after the layout mapping (see backward_impl).
    const bool rows = (layout == TG_ROW_MAJOR) == (want_a != 0);
    const int64_t M = layout == TG_ROW_MAJOR ? m : n, N = layout == TG_ROW_MAJOR ? n : m;
    const BwdGeometry g = rows ? bwd_rows_geometry(batch * M, k, es)
                               : bwd_cols_geometry(batch, M, N, k, es);
    name = std::string(rows ? "rows" : "cols") + (g.global ? " global" : " lds") +
           " waves=" + std::to_string(g.waves) + " lds=" + std::to_string(g.lds) +
           " grid=" + std::to_string(g.grid);
    if (!rows && g.kp < k) name += " passes=" + std::to_string((k + g.kp - 1) / g.kp);
    return name.c_str();
}

int tg_gemm_ws(int device, tg_semiring semiring, tg_dtype dtype, tg_layout layout, const void* A,
               const void* B, void* C, int32_t* argmax, int64_t m, int64_t n, int64_t k,
               void* workspace, size_t workspace_bytes, void* stream) {
    return gemm_impl(device, semiring, dtype, layout, A, B, C, argmax, 1, m, n, k, 0, 0, 0, false,
                     workspace, workspace_bytes, true, stream);
}

int tg_gemm_strided_batched(int device, tg_semiring semiring, tg_dtype dtype, tg_layout layout,
                            const void* A, const void* B, void* C, int32_t* argmax, int64_t batch,
                            int64_t m, int64_t n, int64_t k, int64_t stride_a, int64_t stride_b,
                            int64_t stride_c, void* stream) {
    return gemm_impl(device, semiring, dtype, layout, A, B, C, argmax, batch, m, n, k, stride_a,
                     stride_b, stride_c, true, nullptr, 0, false, stream);
}

int tg_gemm_strided_batched_ws(int device, tg_semiring semiring, tg_dtype dtype, tg_layout layout,
                               const void* A, const void* B, void* C, int32_t* argmax,
                               int64_t batch, int64_t m, int64_t n, int64_t k, int64_t stride_a,
                               int64_t stride_b, int64_t stride_c, void* workspace,
                               size_t workspace_bytes, void* stream) {
    return gemm_impl(device, semiring, dtype, layout, A, B, C, argmax, batch, m, n, k, stride_a,
                     stride_b, stride_c, true, workspace, workspace_bytes, true, stream);
}

int tg_backward_a(int device, tg_dtype dtype, tg_layout layout, const void* grad_c,
                  const int32_t* argmax, void* grad_a, int64_t m, int64_t n, int64_t k,
                  void* stream) {
    return backward_impl(device, dtype, layout, true, grad_c, argmax, nullptr, grad_a, 1, m, n, k,
                         0, 0, 0, false, false, stream);
}

int tg_backward_b(int device, tg_dtype dtype, tg_layout layout, const void* grad_c,
                  const int32_t* argmax, void* grad_b, int64_t m, int64_t n, int64_t k,
                  void* stream) {
    return backward_impl(device, dtype, layout, false, grad_c, argmax, nullptr, grad_b, 1, m, n, k,
                         0, 0, 0, false, false, stream);
}

int tg_maxmul_backward_a(int device, tg_dtype dtype, tg_layout layout, const void* grad_c,
                         const int32_t* argmax, const void* B, void* grad_a, int64_t m, int64_t n,
                         int64_t k, void* stream) {
    return backward_impl(device, dtype, layout, true, grad_c, argmax, B, grad_a, 1, m, n, k, 0, 0,
                         0, false, true, stream);
}

int tg_maxmul_backward_b(int device, tg_dtype dtype, tg_layout layout, const void* grad_c,
                         const int32_t* argmax, const void* A, void* grad_b, int64_t m, int64_t n,
                         int64_t k, void* stream) {
    return backward_impl(device, dtype, layout, false, grad_c, argmax, A, grad_b, 1, m, n, k, 0, 0,
                         0, false, true, stream);
}

int tg_backward_a_strided_batched(int device, tg_dtype dtype, tg_layout layout,
                                  const void* grad_c, const int32_t* argmax, const void* other,
                                  void* grad_a, int64_t batch, int64_t m, int64_t n, int64_t k,
                                  int64_t stride_c, int64_t stride_other, int64_t stride_a,
                                  void* stream) {
    return backward_impl(device, dtype, layout, true, grad_c, argmax, other, grad_a, batch, m, n, k,
                         stride_c, stride_other, stride_a, true, other != nullptr, stream);
}

int tg_backward_b_strided_batched(int device, tg_dtype dtype, tg_layout layout,
                                  const void* grad_c, const int32_t* argmax, const void* other,
                                  void* grad_b, int64_t batch, int64_t m, int64_t n, int64_t k,
                                  int64_t stride_c, int64_t stride_other, int64_t stride_b,
                                  void* stream) {
    return backward_impl(device, dtype, layout, false, grad_c, argmax, other, grad_b, batch, m, n,
                         k, stride_c, stride_other, stride_b, true, other != nullptr, stream);
}

int tg_transpose(int device, tg_dtype dtype, const void* src, void* dst, int64_t batch,
                 int64_t rows, int64_t cols, void* stream) {
    if (!valid_dtype(dtype)) return fail(TG_ERR_INVALID_ARGUMENT, "unknown dtype " + std::to_string(dtype));
    if (batch < 0 || rows < 0 || cols < 0) return fail(TG_ERR_DIMENSION_MISMATCH, "negative dimension");
    if (rows > 0x7fffffffLL || cols > 0x7fffffffLL)
        return fail(TG_ERR_DIMENSION_MISMATCH, "dimension exceeds 2^31-1");
    if ((rows + 31) / 32 > 65535) return fail(TG_ERR_DIMENSION_MISMATCH, "rows too large for the transpose grid");
    const int64_t elems = rows * cols;
    if (batch > 0 && elems > 0 && (src == nullptr || dst == nullptr))
        return fail(TG_ERR_INVALID_ARGUMENT, "src or dst is NULL");
    int rc = select_device(device);
    if (rc != TG_OK) return rc;
    if (batch == 0 || elems == 0) return TG_OK;
    hipStream_t st = as_stream(stream);
    auto run = [&](auto tag) {
        using T = decltype(tag);
        const T* s = static_cast<const T*>(src);
        T* d = static_cast<T*>(dst);
        for (int64_t z0 = 0; z0 < batch; z0 += 65535) {
            const int64_t nb = (batch - z0 < 65535) ? batch - z0 : 65535;
            const int r = launch_transpose<T>(s + z0 * elems, d + z0 * elems, rows, cols, elems, elems,
                                              nb, st);
            if (r != TG_OK) return r;
        }
        return int(TG_OK);
    };
    switch (dtype) {
        case TG_F32: return run(float());
        case TG_F64: return run(double());
        case TG_I32: return run(int32_t());
        default: return run(int64_t());
    }
}

}  // extern "C"
