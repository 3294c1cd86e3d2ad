// tg_gemm_kresg.hpp -- K-resident argmax kernel for i32 MaxPlus/MinPlus at any
// short K, M and N (gfx950): Viterbi steps whose state count is not a multiple
// of the tiles of tg_gemm_kresw / tg_gemm_kres.
//
// Same scheme as tg_gemm_kresw (the column tile's B panel in LDS as f32 keys
// (a+b)*256 + (255-k) or + k, each wave on its own 16-row tiles, streaming A
// through wave-private LDS slots without barriers).  The edges cost no branch:
//   K   panel position p holds k = p; the last, partial quad and any past it
//       hold the row's last four k again (K - 4 ..), so every A load is a whole
//       16-byte one.  A product met twice changes no join and no strict
//       improvement;
//   N   likewise: the last, partial column quad is columns N - 4 ..;
//   M   the last row tile starts at M - 16: rows met twice are written twice
//       with the same values;
//   alignment  16-byte loads and stores at 4-byte alignment.
// Row tiles or panels outside the f32-key range (|x| >= 2^15) take the exact
// per-product rule over the same tiles.
// Bound: on ordinary K VALU issue, on the products of whole tiles (K to a
// multiple of 32, N of 64: 1.64 times those of 100 states, 1.13 instructions per
// ideal one of them), beside the LDS reads of the fragments (8 floats per 16
// products of a lane); at short K the writes of C and argmax.
// Measured on MI355X (us; before it: the generic kernel's exact mode,
// direct-to-LDS or short-K tiles): 262144 x 16 x 16 27 (130), x 32 x 32 27
// (234), x 48 x 48 45 (99), x 100 x 100 155 (364),
// x 160 x 160 286 (558), x 256 x 256 610 (999), 2001^2 x 100 29 (67);
// all by the exact rule (both operands wide): x 32 x 32 55 (234), x 100 x 100
// 241 (352), x 200 x 200 849 (954).
#pragma once

#include "tg_gemm_kresw.hpp"

namespace tg {

// WAVES per workgroup: 8, two workgroups per CU, while two B panels fit the LDS
// (K <= 160); 16, one workgroup per CU, beyond.  4 waves per SIMD either way
// (262144 x 160 x 160 286 us with 8 against 297 with 16, x 176 x 176 446 / 409;
// fewer waves per workgroup also share few row tiles out better: 20000 x 40 x
// 40 10.4 / 20.4).
template <int WAVES>
struct KresgCfg {
    static constexpr int K_MAX = WAVES == 8 ? 160 : 256;
    static constexpr int THREADS = 64 * WAVES;
    static constexpr int ROWS = 16, BK = 32, TM = 4, TN = 4, BN = 16 * TN;
    // An A slot: 4 rows of 32 k, then 4 words of padding, so that the four
    // row groups of a wave read from different banks.
    static constexpr int GROUP = 4 * BK + 4;
    static constexpr int SLOT = 4 * GROUP;
    static constexpr size_t lds_bytes(int64_t K) {
        return (size_t((K + BK - 1) / BK * BK) * BN + WAVES * 2 * SLOT) * 4 + 16;
    }
};

// grid = (G, batch, 1) with G a multiple of tiles_n, block = THREADS, dynamic
// LDS = lds_bytes(K).  M >= 16, N >= 4, 4 <= K <= K_MAX.
template <int SR, int WAVES>
__global__ __launch_bounds__(KresgCfg<WAVES>::THREADS, 4) void tg_gemm_kresg(
    const int32_t* __restrict__ A, const int32_t* __restrict__ B, int32_t* __restrict__ C,
    int32_t* __restrict__ IDX, int64_t M, int64_t N64, int64_t K64, int64_t sA, int64_t sB,
    int64_t sC, int tiles_n) {
    static_assert(SR == SR_MAXPLUS || SR == SR_MINPLUS, "keys need an additive semiring");
    using Cfg = KresgCfg<WAVES>;
    constexpr int BK = Cfg::BK, BN = Cfg::BN, TM = Cfg::TM, TN = Cfg::TN, ROWS = Cfg::ROWS;
    extern __shared__ __align__(16) unsigned char kg_lds[];
    const int K = int(K64), N = int(N64);
    const int KT = (K + BK - 1) / BK;
    float* const Bs = reinterpret_cast<float*>(kg_lds);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tx = lane & 15;
    const int ty = lane >> 4;  // rows ty*4 .. ty*4+3 of the wave's tile
    float* const As = Bs + KT * BK * BN + wave * 2 * Cfg::SLOT;
    int* const vote = reinterpret_cast<int*>(Bs + KT * BK * BN + WAVES * 2 * Cfg::SLOT);

    const int tn = int(blockIdx.x) % tiles_n;
    const int col0 = tn * BN;
    const int64_t stride = int64_t(int(gridDim.x) / tiles_n) * WAVES;
    const int64_t tiles = (M + ROWS - 1) / ROWS;
    const int64_t z = blockIdx.y;
    const int32_t* const Az = A + z * sA;
    const int32_t* const Bz = B + z * sB;
    int32_t* const Cz = C + z * sC;
    int32_t* const Iz = IDX + z * sC;

    auto small = [](int32_t x) { return uint32_t(x) + 32768u < 65536u; };  // |x| < 2^15
    auto row0 = [&](int64_t r) { return r * ROWS + ROWS <= M ? r * ROWS : M - ROWS; };

    // k tile t of row tile r: 16 rows x 32 positions = 128 quads; the lane
    // holds row lane >> 3 and that + 8, quad lane & 7.
    typedef int v4i_t __attribute__((ext_vector_type(4), aligned(4)));
    v4i_t pa[2];
    auto load_a = [&](int64_t r, int t) __attribute__((always_inline)) {
        const char* base = reinterpret_cast<const char*>(Az + row0(r) * K64);
        const int k = t * BK + (lane & 7) * 4;
        const uint32_t off = uint32_t((lane >> 3) * K + (k < K - 4 ? k : K - 4)) * 4;
        pa[0] = *reinterpret_cast<const v4i_t*>(base + off);
        pa[1] = *reinterpret_cast<const v4i_t*>(base + (off + uint32_t(8 * K) * 4));
    };
    auto pa_small = [&]() {
        bool ok = true;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) ok = ok && small(pa[u][e]);
        return __all(ok) != 0;
    };
    float* const a_in = As + (lane >> 5) * Cfg::GROUP + ((lane >> 3) & 3) * BK + (lane & 7) * 4;
    const float* const a_out = As + ty * Cfg::GROUP;
    auto store_a = [&](int s, auto conv) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
            *reinterpret_cast<float4*>(a_in + s * Cfg::SLOT + u * 2 * Cfg::GROUP) =
                make_float4(conv(pa[u][0]), conv(pa[u][1]), conv(pa[u][2]), conv(pa[u][3]));
    };
    // Columns tx*4 .. of row i of the lane's rows in row tile r.
    auto store_quad = [&](int64_t r, int i, v4i_t cv, v4i_t iv) __attribute__((always_inline)) {
        // From an opaque copy of the lane id: hoisted out of the tile loop the
        // addresses would stay live across the main loop.
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int col = col0 + (ln & 15) * 4;
        if (col >= N) return;
        const int64_t base = (row0(r) + i) * N64;
        const uint32_t off = uint32_t((ln >> 4) * 4 * N + (col < N - 4 ? col : N - 4)) * 4;
        __builtin_nontemporal_store(
            cv, reinterpret_cast<v4i_t*>(reinterpret_cast<char*>(Cz + base) + off));
        __builtin_nontemporal_store(
            iv, reinterpret_cast<v4i_t*>(reinterpret_cast<char*>(Iz + base) + off));
    };
    // The panel through conv(b, k); true if every b is in the key range.
    auto load_panel = [&](auto conv) {
        bool ok = true;
        for (int q = tid; q < KT * BK * BN; q += Cfg::THREADS) {
            const int p = q / BN;
            const int c = col0 + q % BN, c4 = c & ~3;
            const int p4 = p & ~3;
            const int k = (p4 < K - 4 ? p4 : K - 4) + (p & 3);
            const int col = c4 + 4 <= N ? c : c4 < N ? N - 4 + (c & 3) : 0;
            const int32_t b = Bz[k * N64 + col];
            ok = ok && small(b);
            Bs[q] = conv(b, k);
        }
        return ok;
    };
    auto bkey = [](int32_t b, int k) {
        return float(int32_t((uint32_t(b) << 8) + uint32_t(SR == SR_MINPLUS ? k : 255 - k)));
    };

    // Keys only if the panel and the waves' first rows are in range: rows that
    // are not usually come in numbers, and the exact rule is the faster on the
    // panel's own values.
    int64_t r = int64_t(int(blockIdx.x) / tiles_n) * WAVES + wave;
    if (r < tiles) load_a(r, 0);
    if (tid == 0) *vote = 1;
    __syncthreads();
    if (!load_panel(bkey) || (r < tiles && !pa_small())) *vote = 0;
    __syncthreads();
    const bool bkeys = *vote != 0;
    if (!bkeys) {  // the panel's own values, for the exact rule
        load_panel([](int32_t b, int) { return __int_as_float(b); });
        __syncthreads();
    }

    auto bvalue = [&](float f) { return bkeys ? int32_t(f) >> 8 : __float_as_int(f); };

#pragma unroll 1
    for (; r < tiles; r += stride) {
        bool loaded = true;  // pa holds the tile's first k tile
        if (bkeys) {
            bool fast = true;
            float key[TM][TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) key[i][j] = tzero<SR, float>();
#pragma unroll 1
            for (int t = 0; t < KT; ++t) {
                if (!pa_small()) {  // wave-uniform: the tile takes the exact rule
                    fast = false;
                    loaded = t == 0;
                    break;
                }
                store_a(t & 1, [](int32_t a) { return float(int32_t(uint32_t(a) << 8)); });
                if (t + 1 < KT) load_a(r, t + 1);
                else if (r + stride < tiles) load_a(r + stride, 0);
                const float* as = a_out + (t & 1) * Cfg::SLOT;
                const float* bs = Bs + t * BK * BN + tx * 4;
#pragma unroll
                for (int kk = 0; kk < BK; kk += 2) {
                    float a[TM][2], b[2][TN];
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        a[i][0] = as[i * BK + kk];
                        a[i][1] = as[i * BK + kk + 1];
                    }
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int j = 0; j < TN; ++j)
                            b[h][j] = bs[(kk + h) * BN + j];
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int j = 0; j < TN; ++j)
                            key[i][j] = tjoin<SR, float>(
                                tjoin<SR, float>(key[i][j], a[i][0] + b[0][j]),
                                a[i][1] + b[1][j]);
                    // One k pair's fragments at a time: hoisting more would
                    // take the registers of the fourth wave per SIMD.
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (fast) {
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    v4i_t cv, iv;
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        const int32_t ik = int32_t(key[i][j]);  // exact: an integer key
                        cv[j] = ik >> 8;
                        iv[j] = SR == SR_MINPLUS ? (ik & 255) : 255 - (ik & 255);
                    }
                    store_quad(r, i, cv, iv);
                }
                continue;
            }
        }
        // ---- exact rule -----------------------------------------------------
        // The reference's rule per output: from the tropical zero with index 0,
        // take (p, k) on every strict improvement, k ascending
        // (core/argmax.rs:24-33, core/kernel.rs:119-167).  Per quad of k the
        // join of its products, and on a strict improvement the quad; then the
        // first k of that quad that gives the value.
        int32_t val[TM][4], rec[TM][4];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                val[i][j] = tzero<SR, int32_t>();
                rec[i][j] = -1;
            }
        if (!loaded) load_a(r, 0);
        auto walk = [&](auto value) __attribute__((always_inline)) {
#pragma unroll 1
            for (int t = 0; t < KT; ++t) {
                store_a(t & 1, [](int32_t a) { return __int_as_float(a); });
                if (t + 1 < KT) load_a(r, t + 1);
                else if (r + stride < tiles) load_a(r + stride, 0);
                const float* as = a_out + (t & 1) * Cfg::SLOT;
                const float* bs = Bs + t * BK * BN + tx * 4;
                const int kend = K - t * BK < BK ? K - t * BK : BK;
#pragma unroll 2
                for (int kk = 0; kk < kend; kk += 4) {
                    int32_t a[TM][4], b[4][4];
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int h = 0; h < 4; ++h) a[i][h] = __float_as_int(as[i * BK + kk + h]);
#pragma unroll
                    for (int h = 0; h < 4; ++h)
#pragma unroll
                        for (int j = 0; j < 4; ++j) b[h][j] = value(bs[(kk + h) * BN + j]);
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int32_t was = val[i][j];
#pragma unroll
                            for (int h = 0; h < 4; ++h)
                                val[i][j] = tjoin<SR, int32_t>(
                                    val[i][j], tmul<SR, int32_t>(a[i][h], b[h][j]));
                            rec[i][j] = val[i][j] != was ? t * BK + kk : rec[i][j];
                        }
                }
            }
        };
        if (bkeys) walk([](float f) { return int32_t(f) >> 8; });
        else walk([](float f) { return __float_as_int(f); });
        const int32_t* const Ar = Az + (row0(r) + ty * 4) * K64;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            v4i_t cv, iv;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                cv[j] = val[i][j];
                const int p0 = rec[i][j];
                iv[j] = 0;
                if (p0 < 0) continue;  // no product beat the tropical zero
                const int k = p0 < K - 4 ? p0 : K - 4;
                const v4i_t a = *reinterpret_cast<const v4i_t*>(Ar + i * K + k);
#pragma unroll
                for (int h = 3; h >= 0; --h) {
                    const int32_t p =
                        tmul<SR, int32_t>(a[h], bvalue(Bs[(p0 + h) * BN + tx * 4 + j]));
                    iv[j] = p == cv[j] ? k + h : iv[j];
                }
            }
            store_quad(r, i, cv, iv);
        }
    }
}

}  // namespace tg
