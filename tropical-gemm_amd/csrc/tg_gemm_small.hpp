// tg_gemm_small.hpp -- tropical GEMM for problems with few or narrow output
// tiles (gfx950).
//
// Same contract as tg_gemm_tiles (tg_kernels.hpp): any shape, alignment and
// dtype, with or without argmax, no workspace.
//
// Work split.  A wave's 64 lanes are LR x LC x LK: LR lanes down the rows, LC
// across the columns (4 x 4 outputs per lane, so tiles of 4 LR x 4 LC) and LK
// along k.  The W waves of a workgroup share one output tile and split K with
// it: wave w takes the k-steps w, w + W, ... of LK * KV consecutive k, lane
// lk of a wave the KV k (one 16-byte vector) at lk * KV of the step.  So every
// tile has W * LK partial results, which meet once in LDS at the end.  Operands
// come straight from global memory (L1 / L2) into registers, one step ahead
// of the products: no LDS staging and no barrier inside the k loop, so a
// problem of a few thousand outputs pays a load latency per step and one
// merge instead of a barrier per 32 k of one tile.
//
// Bound and measured (MI355X, kernel time through the C ABI, us; before is the
// kernel these sizes took): a handful of outputs is a launch and a chain of load
// latencies, f32 argmax 67 x 45 x 131 56.8 -> 6.1 (one 128 x 64 tile on one
// CU); a few rows against a large B stream B from HBM, 4 x 4096 x 4096
// 94.6 -> 17.4 (64 MB at 3.9 TB/s; B^T staging, 64-row tiles and a merge
// launch); in between the L1 operand reads (8 16-byte loads for 64 products of
// a lane), 300 x 300 x 4000 289 -> 33, 512^3 37 -> 16, f64 1024^3 271 -> 203.
// 8 x 4 outputs per lane would halve those reads but leave half the lanes'
// parallelism, which is what the sizes here lack.
//
// Argmax: the KV products of a step fold into the running value with max/min;
// the step's first k is recorded where the value strictly improved (the
// chunked argmax of tg_kernels.hpp with chunks of KV).  Partials merge by
// value and, between equal values, by the smaller k, which is the first k of
// the whole range; the thread that writes an output finds the k inside the
// recorded chunk by recomputing its KV products, and writes that product's
// bits.  k past K re-read k = K - 1 (a duplicate that can only tie).
//
// NaN: f32 chains propagate NaN (v_maximum3_f32); f64 products are tested in
// pairs (v_cmp_u_f64).  An output that met a NaN product in any partial is
// recomputed with the reference's serial rule (cpu_select).
#pragma once

#include "tg_kernels.hpp"
#include "tg_small.hpp"

namespace tg {

// Waves per workgroup, at most: 128 VGPRs hold a 32-bit lane (two operand sets
// of 32, 16 values, 16 records), a 64-bit one needs more.
template <typename T>
constexpr int small_max_waves() {
    return sizeof(T) == 4 ? 16 : 8;
}

template <typename T, int LR_, int LC_>
struct SmallCfg {
    static constexpr int LR = LR_, LC = LC_, LK = 64 / (LR_ * LC_);
    static constexpr int KV = Vec16<T>::N;          // k per lane and step
    static constexpr int STEP = LK * KV;            // k per wave and step
    static constexpr int BM = 4 * LR, BN = 4 * LC;  // output tile
    static constexpr int OUTS = BM * BN;
    static constexpr int MAX_WAVES = small_max_waves<T>();
    static constexpr int part_bytes(bool argmax) { return int(sizeof(T)) + (argmax ? 4 : 0); }
    static constexpr int lds_bytes(int waves, bool argmax) {
        return waves * LK * OUTS * part_bytes(argmax);
    }
};

// max / min of two f64 products or values as one instruction.  The
// compiler's maxnum canonicalizes loop-carried operands with another max; the
// operands here are add / multiply results or such maxima.  A NaN operand is
// dropped: the callers test the products.
template <int SR>
__device__ __forceinline__ double join_raw_f64(double x, double y) {
    double r;
    if constexpr (SR == SR_MINPLUS)
        asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    else
        asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}

// NCLAMP: N < 4, so a lane's four columns are clamped one by one; otherwise
// the four columns of a lane past the right edge shift left into the matrix
// (columns that another lane owns: computed twice, stored once).
// grid = (tiles_m * tiles_n, 1, batch), block = 64 * W, W <= MAX_WAVES,
// LDS = SmallCfg::lds_bytes(W, ARGMAX).  M * K and K * N below 2^31 elements
// (32-bit element offsets).
template <int SR, typename T, bool ARGMAX, int LR, int LC, bool NCLAMP>
__global__ __launch_bounds__(64 * small_max_waves<T>()) void tg_gemm_small(
    const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int32_t* __restrict__ IDX,
    int64_t M64, int64_t N64, int64_t K64, int64_t sA, int64_t sB, int64_t sC, int tiles_m,
    int tiles_n) {
    using Cfg = SmallCfg<T, LR, LC>;
    constexpr int LK = Cfg::LK, KV = Cfg::KV, STEP = Cfg::STEP, OUTS = Cfg::OUTS;
    constexpr bool F64 = std::is_same<T, double>::value;
    extern __shared__ __align__(16) unsigned char small_lds[];

    const int M = int(M64), N = int(N64), K = int(K64);
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int W = int(blockDim.x) >> 6;
    const int lc = lane % LC, lk = lane / LC % LK, lr = lane / (LC * LK);
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int row0 = tm * Cfg::BM, col0 = tn * Cfg::BN;
    const int64_t z = blockIdx.z;
    A += z * sA;
    B += z * sB;
    C += z * sC;
    if constexpr (ARGMAX) IDX += z * sC;

    // First column of the column group that starts at c0 (shifted into the
    // matrix), and column j of it.
    auto group_col = [&](int c0) { return NCLAMP ? c0 : (c0 < N - 4 ? c0 : N - 4); };
    auto lane_col = [&](int cg, int j) {
        if constexpr (NCLAMP) return cg + j < N ? cg + j : N - 1;
        return cg + j;
    };
    const int cg = group_col(col0 + lc * 4);
    uint32_t aoff[4];  // row starts, in elements
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = row0 + lr * 4 + i;
        aoff[i] = uint32_t(r < M ? r : M - 1) * uint32_t(K);
    }

    struct Step {
        T a[4][KV], b[KV][4];
    };
    // Operands of the step at k0 (this lane's k: k0 + lk * KV + q), all below K.
    auto load_full = [&](int k0, Step& s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const Vec16<T> v = *reinterpret_cast<const Vec16<T>*>(A + k0 + (aoff[i] + uint32_t(lk * KV)));
#pragma unroll
            for (int q = 0; q < KV; ++q) s.a[i][q] = v.v[q];
        }
#pragma unroll
        for (int q = 0; q < KV; ++q) {
            const T* row = B + int64_t(k0 + q) * N;
            const uint32_t off = uint32_t(lk * KV) * uint32_t(N);
            if constexpr (NCLAMP) {
#pragma unroll
                for (int j = 0; j < 4; ++j) s.b[q][j] = row[off + uint32_t(lane_col(cg, j))];
            } else {
#pragma unroll
                for (int j = 0; j < 4; j += KV) {
                    const Vec16<T> v = *reinterpret_cast<const Vec16<T>*>(row + (off + uint32_t(cg + j)));
#pragma unroll
                    for (int e = 0; e < KV; ++e) s.b[q][j + e] = v.v[e];
                }
            }
        }
    };
    // The last, partial step: k past K re-read K - 1.
    auto load_tail = [&](int k0, Step& s) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < KV; ++q) {
            const int kq = k0 + lk * KV + q;
            const int k = kq < K ? kq : K - 1;
#pragma unroll
            for (int i = 0; i < 4; ++i) s.a[i][q] = A[aoff[i] + uint32_t(k)];
#pragma unroll
            for (int j = 0; j < 4; ++j) s.b[q][j] = B[uint32_t(k) * uint32_t(N) + uint32_t(lane_col(cg, j))];
        }
    };

    // acc: running value; ch: first k of the last step that strictly improved
    // it (-1: the tropical zero was never beaten).
    T acc[4][4];
    int32_t ch[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc[i][j] = tzero<SR, T>();
            ch[i][j] = -1;
        }
    bool met_nan = false;
    auto join = [](T x, T y) {
        if constexpr (F64) return join_raw_f64<SR>(x, y);
        else return tjoin<SR, T>(x, y);
    };
    auto fold = [&](int k0, const Step& s) __attribute__((always_inline)) {
        const int32_t kl = k0 + lk * KV;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            T nv[4];
            bool better[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                T p[KV];
#pragma unroll
                for (int q = 0; q < KV; ++q) p[q] = tmul<SR, T>(s.a[i][q], s.b[q][j]);
                T v = acc[i][j];
#pragma unroll
                for (int q = 0; q < KV; q += 2) {
                    v = join(join(v, p[q]), p[q + 1]);
                    if constexpr (F64) met_nan |= __builtin_isunordered(p[q], p[q + 1]);
                }
                nv[j] = v;
                better[j] = tbetter<SR, T>(v, acc[i][j]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[i][j] = nv[j];
                if constexpr (ARGMAX) ch[i][j] = better[j] ? kl : ch[i][j];
            }
        }
    };

    const int nfull = K / STEP;
    if (wave < nfull) {
        Step cur, nxt;
        load_full(wave * STEP, cur);
        for (int s = wave; s < nfull; s += W) {
            const int sn = s + W < nfull ? s + W : s;
            load_full(sn * STEP, nxt);
            fold(s * STEP, cur);
            cur = nxt;
        }
    }
    if (nfull * STEP < K && nfull % W == wave) {
        Step s;
        load_tail(nfull * STEP, s);
        fold(nfull * STEP, s);
    }

    // ---- merge ----------------------------------------------------------------
    // Partial p = wave * LK + lk of output o at pv[p * OUTS + o] / pi[..]; a
    // record of -2 (f64 value-only: a NaN value) marks an output that met a
    // NaN product.
    const int parts = W * LK;
    T* const pv = reinterpret_cast<T*>(small_lds);
    int32_t* const pi = reinterpret_cast<int32_t*>(pv + parts * OUTS);
    {
        const int base = (wave * LK + lk) * OUTS + lr * 4 * Cfg::BN + lc * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                T v = acc[i][j];
                if constexpr (F64) {
                    if (met_nan) v = __builtin_nan("");
                }
                pv[base + i * Cfg::BN + j] = v;
                if constexpr (ARGMAX) pi[base + i * Cfg::BN + j] = tisnan(v) ? -2 : ch[i][j];
            }
    }
    __syncthreads();
    // Combines partials first, first + step, ... of output o.
    auto merge = [&](int o, int first, int step, int count, T& v, int32_t& c) {
        v = pv[first * OUTS + o];
        c = -1;
        bool nan = tisnan(v);
        if constexpr (ARGMAX) c = pi[first * OUTS + o];
        for (int p = first + step; p < count; p += step) {
            const T v1 = pv[p * OUTS + o];
            if constexpr (ARGMAX) {
                const int32_t c1 = pi[p * OUTS + o];
                const bool take = tbetter<SR, T>(v1, v) || (v1 == v && c1 < c);
                if (c == -2 || c1 == -2) {
                    c = -2;
                } else if (take) {
                    v = v1;
                    c = c1;
                }
            } else {
                nan |= tisnan(v1);
                v = join(v, v1);
            }
        }
        if constexpr (!ARGMAX && std::is_floating_point<T>::value) {
            if (nan) v = T(__builtin_nan(""));
        }
    };
    auto finish = [&](int o, T v, int32_t c) {
        const int r = row0 + o / Cfg::BN;
        const int c0 = col0 + (o % Cfg::BN) / 4 * 4;
        const int col = group_col(c0) + o % 4;
        if (r >= M || c0 >= N || col < c0 || col >= N) return;
        const T* a = A + uint32_t(r) * uint32_t(K);
        int32_t ix = 0;
        if (ARGMAX ? c == -2 : tisnan(v)) {
            cpu_select<SR, T>(a, 1, B + col, N, K, v, ix);
        } else if (ARGMAX && c >= 0) {
            // The first k of the recorded chunk that attains the value.
            T p[KV];
            int kk[KV];
#pragma unroll
            for (int q = 0; q < KV; ++q) {
                kk[q] = c + q < K ? c + q : K - 1;
                p[q] = tmul<SR, T>(a[kk[q]], B[uint32_t(kk[q]) * uint32_t(N) + uint32_t(col)]);
            }
            T w = p[KV - 1];
            ix = kk[KV - 1];
#pragma unroll
            for (int q = KV - 2; q >= 0; --q)
                if (p[q] == v) {
                    w = p[q];
                    ix = kk[q];
                }
            v = w;
        }
        C[int64_t(r) * N + col] = v;
        if constexpr (ARGMAX) IDX[int64_t(r) * N + col] = ix;
    };
    const int threads = W * 64;
    if (threads <= OUTS) {
        for (int o = tid; o < OUTS; o += threads) {
            T v;
            int32_t c;
            merge(o, 0, 1, parts, v, c);
            finish(o, v, c);
        }
    } else {
        // threads / OUTS threads per output: each combines its share of the
        // partials into the first of them (its own slot), then one the rest.
        const int o = tid % OUTS, g = tid / OUTS, groups = threads / OUTS;
        T v;
        int32_t c;
        merge(o, g, groups, parts, v, c);
        if (g > 0) {
            pv[g * OUTS + o] = v;
            if constexpr (ARGMAX) pi[g * OUTS + o] = c;
        }
        __syncthreads();
        if (g == 0) {
            pv[o] = v;
            if constexpr (ARGMAX) pi[o] = c;
            merge(o, 0, 1, groups, v, c);
            finish(o, v, c);
        }
    }
}

}  // namespace tg
