// tg_gemm_dl64s.hpp -- direct-to-LDS tropical GEMM for 64-bit types on 64 x 64
// tiles (gfx950): f64 problems that make too few 64 x 128 tiles for
// tg_gemm_dl64, and i64.
//
// Same contract as tg_gemm_tiles (tg_kernels.hpp), with or without argmax, any
// shape.  The byte layout is that of tg_gemm_dl's 64 x 64 tiles with 8-byte
// elements (a 16-byte quad holds two k):
//   A tile  64 rows x 16 k, 128-byte rows; quad q of row r stored at quad
//           position q ^ ((r >> 2) & 7).
//   B tile  16 k x 64 columns, row-major (512 B per k-row).
// Two LDS buffers of 16 KB; 16 x 16 threads, thread (tx, ty) owns rows
// ty*4 + i and columns tx*4 + j (i, j < 4): 4 bytes of LDS per product.
//
// Why this tile: 16 outputs per thread and 32 KB of LDS per workgroup leave
// three (argmax) or four waves per SIMD resident.  64-bit chains want them: an
// i64 max is a compare and two selects that wait on it (the register-only i64
// mix issues 15.3 T tropical ops/s at two waves per SIMD and 18.2 T at eight),
// and the generic kernel's 68 KB of LDS allow two.  i64 4096^3 on MI355X:
// argmax 9.23 -> 8.15 ms, value-only 8.64 -> 7.72; 2048^3 argmax 2.05 (exact
// mode) -> 1.16.
//
// Slices (HALVES = 1 to 4): K is cut into that many slices of whole k-tiles,
// one 256-thread part of the workgroup each with its own LDS block; they merge
// in k order in LDS before one resolve, so a problem of few tiles still fills
// the chip without partials in memory (f64 1024^3, 256 tiles, prepasses
// included: argmax 187 us in one slice, 149 in three; value-only 157 in one, 111 in
// four; with more tiles than CUs one slice (value-only two) is faster: 2048^3
// argmax 739 against 828 in three).  The 64 x 128 tiles of tg_gemm_dl64 leave half
// the chip idle there (generic kernel before: 277 and 203 us).
//
// ELEM: operands of any alignment, two 4-byte lanes per element (16 load
// instructions per wave and k-tile instead of 4; f64 2048^3 argmax 770 against
// 739 us).  A last partial k-tile (any
// K) reads k = K - 1 and is overwritten in LDS with operands whose product is
// the tropical zero.
//
// Argmax: one chunk per k-tile (CL = 16), recorded and resolved as in
// tg_gemm_dl64; NaN for f64 by operand classes, as there (clsA / clsB).
#pragma once

#include "tg_elem_rows.hpp"
#include "tg_gemm_dl64.hpp"

namespace tg {

struct Dl64sCfg {
    static constexpr int TM = 4, TN = 4, BM = 64, BN = 64, BK = 16, CL = 16;
    static constexpr int A_BYTES = BM * BK * 8;  // 8 KB
    static constexpr int B_BYTES = BK * BN * 8;  // 8 KB
    static constexpr int LDS_BYTES = 2 * (A_BYTES + B_BYTES);  // per slice
    static constexpr int OUTS = BM * BN;
    // Epilogue (argmax), in the first slice's block.
    static constexpr int NB = 256;  // chunk buckets of the sort
    static constexpr int HIST_OFF = 0;
    static constexpr int CHS_OFF = HIST_OFF + NB * 4;
    static constexpr int LIST_OFF = CHS_OFF + OUTS * 2;
    static constexpr int MISC_OFF = LIST_OFF + OUTS * 2;  // scan scratch, one per slice
    static_assert(MISC_OFF + 64 <= LDS_BYTES, "epilogue arrays fit the LDS block");
};

// Records of four outputs (record4 with 64-bit compares).
template <int SR, typename T>
__device__ __forceinline__ void record4_64(int32_t& c0, int32_t& c1, int32_t& c2, int32_t& c3, T n0,
                                           T n1, T n2, T n3, T p0, T p1, T p2, T p3, int32_t cv) {
    if constexpr (std::is_same<T, double>::value) {
        record4_f64<SR>(c0, c1, c2, c3, n0, n1, n2, n3, p0, p1, p2, p3, cv);
    } else {
        const bool b0 = tbetter<SR, T>(n0, p0), b1 = tbetter<SR, T>(n1, p1);
        const bool b2 = tbetter<SR, T>(n2, p2), b3 = tbetter<SR, T>(n3, p3);
        c0 = b0 ? cv : c0;
        c1 = b1 ? cv : c1;
        c2 = b2 ? cv : c2;
        c3 = b3 ? cv : c3;
    }
}

// Waves per SIMD the kernel is built for: an argmax thread holds value, value
// before the chunk and record of 16 outputs (80 VGPRs) beside its fragments
// (32), 145-168 VGPRs as scheduled; held to 128 it spills (f64 1024^3 in four
// slices 154-183 us against 149 in three).
template <bool ARGMAX>
constexpr int dl64s_waves() {
    return ARGMAX ? 3 : 4;
}

// grid = (tiles_m * tiles_n, 1, batch), block = 256 * HALVES, LDS =
// HALVES * Dl64sCfg::LDS_BYTES.  BT (argmax): B^T, dense.  clsA / clsB (f64):
// operand classes of A's rows and B's columns, else unused.
template <int SR, typename T, bool ARGMAX, int HALVES, bool ELEM>
__global__ __launch_bounds__(TG_THREADS * HALVES) __attribute__((amdgpu_waves_per_eu(
    dl64s_waves<ARGMAX>()))) void tg_gemm_dl64s(
    const T* __restrict__ A, const T* __restrict__ B, const T* __restrict__ BT, T* __restrict__ C,
    int32_t* __restrict__ IDX, const uint32_t* __restrict__ clsA, const uint32_t* __restrict__ clsB,
    int64_t M, int64_t N, int64_t K, int64_t sA, int64_t sB, int64_t sC, int tiles_m, int tiles_n) {
    static_assert(sizeof(T) == 8, "64-bit types");
    using Cfg = Dl64sCfg;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, TM = Cfg::TM, TN = Cfg::TN, CL = Cfg::CL;
    constexpr bool F64 = std::is_same<T, double>::value;
    constexpr int NL = ELEM ? 8 : 2;       // load instructions of a wave per operand and k-tile
    constexpr int IB = ELEM ? 256 : 1024;  // bytes of one instruction
    extern __shared__ __align__(16) unsigned char dl64s_lds[];
    const int half = HALVES > 1 ? int(__builtin_amdgcn_readfirstlane(threadIdx.x >> 8)) : 0;
    unsigned char* const lds = dl64s_lds + half * Cfg::LDS_BYTES;
    T* const As0 = reinterpret_cast<T*>(lds);
    T* const Bs0 = reinterpret_cast<T*>(lds + 2 * Cfg::A_BYTES);

    const int tid = int(threadIdx.x) & (TG_THREADS - 1);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tx = tid & 15;
    const int ty = tid >> 4;
    int tm, tn;
    tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
    const int64_t row0 = int64_t(tm) * BM;
    const int64_t col0 = int64_t(tn) * BN;
    const int64_t z = blockIdx.z;
    A += z * sA;
    B += z * sB;
    C += z * sC;
    if constexpr (ARGMAX) {
        IDX += z * sC;
        BT += z * (N * K);
    }
    if constexpr (F64) {
        clsA += z * M;
        clsB += z * N;
    }
    auto trow = [&](int i) { return ty * 4 + i; };
    auto tcol = [&](int j) { return tx * 4 + j; };

    // Loads of k-tile t.  A: an instruction covers 8 rows (ELEM: 2) of 128
    // bytes, the lane's bytes in its row permuted by quads; B: 2 k rows (ELEM:
    // half a k row).  Addresses are wave-uniform bases plus per-lane byte
    // offsets (few registers: ELEM composes A's from the lane's byte and row).
    // Rows and columns past the edge read the last one (pairs of columns: the
    // last pair), k past K the last k (pair).
    constexpr int LPRA = ELEM ? 32 : 8;  // lanes per row of A
    constexpr int RPI = 64 / LPRA;       // rows of A per instruction
    const int abyte = (lane % LPRA) * (ELEM ? 4 : 16);
    const uint32_t rowK = uint32_t(lane / LPRA) * uint32_t(K) * 8;  // the lane's row in its instruction
    auto aswz = [&](int ins) { return abyte ^ ((ins * RPI >> 2 & 7) << 4); };  // ELEM
    uint32_t offA[ELEM ? 1 : NL];
    if constexpr (!ELEM) {
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const int r = (wave * NL + q) * RPI + lane / LPRA;
            const int64_t gr = row0 + r < M ? row0 + r : M - 1;
            offA[q] = uint32_t((gr - row0) * K * 8) + uint32_t(abyte ^ (((r >> 2) & 7) << 4));
        }
    }
    uint32_t offB[ELEM ? 2 : 1];
    if constexpr (ELEM) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int64_t gc = col0 + h * 32 + (lane >> 1);
            offB[h] = uint32_t(gc < N ? gc : N - 1) * 8 + uint32_t(lane & 1) * 4;
        }
    } else {
        const int64_t gc = col0 + (lane & 31) * 2;
        offB[0] = uint32_t(lane >> 5) * uint32_t(N) * 8 + uint32_t(gc < N ? gc : N - 2) * 8;
    }
    const uint32_t max_row = uint32_t(M - 1 - row0 < BM ? M - 1 - row0 : BM);  // last valid row of the tile
    auto issue_loads = [&](int64_t t, int buf, bool last) {
        unsigned char* adst = reinterpret_cast<unsigned char*>(As0 + buf * (BM * BK));
        unsigned char* bdst = reinterpret_cast<unsigned char*>(Bs0 + buf * (BK * BN));
        const unsigned char* ab = reinterpret_cast<const unsigned char*>(A + row0 * K + t * BK);
        const unsigned char* bb = reinterpret_cast<const unsigned char*>(B + t * BK * N);
        const int left = last ? int(K - t * BK) : BK;  // k in this tile
        // Row strides in bytes, opaque here: the row offsets are composed per
        // k-tile on the scalar unit instead of being held through the loop
        // (16 of them, which spilled).
        uint32_t k8 = uint32_t(K) * 8, n8 = uint32_t(N) * 8;
        if constexpr (ELEM) {
            asm volatile("" : "+s"(k8), "+s"(n8));
            bb += uint64_t(elem_first_row(wave * (BK / 4), left)) * n8;  // the wave's k rows of B
        }
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const int ins = wave * NL + q;
            if constexpr (ELEM) {
                const uint32_t r = uint32_t(ins * RPI);
                int byte = aswz(ins);
                if (last) {
                    const int max_byte = (left - 1) * 8 + (byte & 4);
                    byte = byte < max_byte ? byte : max_byte;
                }
                const unsigned char* row = ab + (r < max_row ? r : max_row) * k8;
                lds_load4(row + ((r < max_row ? rowK : 0u) + uint32_t(byte)), adst + ins * IB);
                lds_load4(bb + offB[q % 2], bdst + ins * IB);
                if (q % 2 == 1 && elem_steps(ins / 2, left)) bb += n8;
            } else {
                uint32_t oa = offA[q], ob = offB[0];
                if (last) {
                    const int byte = abyte ^ (((ins * RPI + lane / LPRA) >> 2 & 7) << 4);
                    const int max_byte = (left - 2) * 8;
                    oa += uint32_t((byte < max_byte ? byte : max_byte) - byte);
                }
                // K is even, so the two k rows are both inside it or both past.
                const int kr = ins * 2 < left ? ins * 2 : left - 2;
                lds_load16(ab + oa, adst + ins * IB);
                lds_load16(bb + uint64_t(kr) * uint64_t(N) * 8 + ob, bdst + ins * IB);
            }
        }
    };
    auto patch_tail = [&](int buf, int kv) {
        T* as = As0 + buf * (BM * BK);
        T* bs = Bs0 + buf * (BK * BN);
        const int nk = BK - kv;
        for (int e = tid; e < BM * nk; e += TG_THREADS) {
            const int r = e / nk, k = kv + e % nk;
            as[r * BK + (((k >> 1) ^ ((r >> 2) & 7)) << 1) + (k & 1)] = tzero<SR, T>();
        }
        for (int e = tid; e < nk * BN; e += TG_THREADS) bs[kv * BN + e] = T(0);
    };

    T acc[TM][TN], alt[TM][TN];
    int32_t ch[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            acc[i][j] = tzero<SR, T>();
            alt[i][j] = tzero<SR, T>();
            ch[i][j] = -1;
        }
    int swz_t = ty & 7;
    auto load_frag = [&](int buf, int kk, T (&a)[TM][2], T (&b)[2][TN]) {
        const T* as = As0 + buf * (BM * BK);
        const T* bs = Bs0 + buf * (BK * BN);
        const int q = (((kk >> 1) ^ swz_t) << 1);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const Vec16<T> v = *reinterpret_cast<const Vec16<T>*>(as + trow(i) * BK + q);
            a[i][0] = v.v[0];
            a[i][1] = v.v[1];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < TN; j += 2) {
                const Vec16<T> v = *reinterpret_cast<const Vec16<T>*>(bs + (kk + h) * BN + tcol(j));
                b[h][j] = v.v[0];
                b[h][j + 1] = v.v[1];
            }
    };
    // f64 as written instructions (see tg_gemm_dl64's join_f64).
    auto join = [](T x, T y) {
        if constexpr (F64) {
            T r;
            if constexpr (SR == SR_MINPLUS)
                asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
            else
                asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
            return r;
        } else {
            return tjoin<SR, T>(x, y);
        }
    };
    auto chunk = [&](int64_t t, int buf, const T (&from)[TM][TN], T (&to)[TM][TN]) {
#pragma unroll
        for (int kk = 0; kk < BK; kk += 2) {
            T a[TM][2], b[2][TN];
            load_frag(buf, kk, a, b);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const T p0 = tmul<SR, T>(a[i][0], b[0][j]);
                    const T p1 = tmul<SR, T>(a[i][1], b[1][j]);
                    const T st = kk == 0 ? from[i][j] : to[i][j];
                    to[i][j] = join(join(st, p0), p1);
                }
        }
        if constexpr (ARGMAX) {
            int32_t cv;
            asm volatile("v_mov_b32 %0, %1" : "=v"(cv) : "s"(int32_t(t)));
#pragma unroll
            for (int i = 0; i < TM; ++i)
                record4_64<SR, T>(ch[i][0], ch[i][1], ch[i][2], ch[i][3], to[i][0], to[i][1],
                                  to[i][2], to[i][3], from[i][0], from[i][1], from[i][2],
                                  from[i][3], cv);
        }
    };

    // Slice h covers k-tiles [t0, t1); every slice runs the same number of
    // rounds (and barriers), round s on its k-tile t0 + s in buffer s & 1;
    // rounds past the slice's end only hand the values on.
    const int nkt = int((K + BK - 1) / BK);
    const int per = (nkt + HALVES - 1) / HALVES;
    const int t0 = half * per;
    const int t1 = t0 + per < nkt ? t0 + per : nkt;
    const int kv = int(K - int64_t(nkt - 1) * BK);  // k in the last k-tile
    const int tail_round = kv < BK ? (nkt - 1) % per : -1;
    auto loads = [&](int t, int buf) __attribute__((always_inline)) {
        if (t == nkt - 1)
            issue_loads(t, buf, true);
        else
            issue_loads(t, buf, false);
    };
    auto round = [&](int s, int buf, const T (&from)[TM][TN], T (&to)[TM][TN])
                     __attribute__((always_inline)) {
        const int t = t0 + s;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (t + 1 < t1) loads(t + 1, buf ^ 1);
        if (s == tail_round) {
            if (t == nkt - 1) patch_tail(buf, kv);
            __syncthreads();
        }
        asm volatile("" : "+v"(swz_t));
        if (HALVES == 1 || t < t1) {
            chunk(t, buf, from, to);
        } else if constexpr (ARGMAX) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) to[i][j] = from[i][j];
        }
    };
    if (t0 < t1) loads(t0, 0);
    if constexpr (ARGMAX) {
        int s = 0;
        for (; s + 1 < per; s += 2) {
            round(s, 0, acc, alt);
            round(s + 1, 1, alt, acc);
        }
        if (s < per) {
            round(s, 0, acc, alt);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = alt[i][j];
        }
    } else {
        for (int s = 0; s < per; ++s) round(s, s & 1, acc, acc);
    }

    // ---- merge of the slices -----------------------------------------------------
    // In k order: a later slice replaces the running result only if strictly
    // better.  Values first (a slice's 32 KB hold exactly them), then the
    // records of the slice each output took.  Each 256-thread part merges, and
    // from here on owns, some rows of every thread's outputs: rows [er0, er0 +
    // ern), an extra one for the first part where they do not divide.
    constexpr int ER = (TM + HALVES - 1) / HALVES;
    const int er0 = HALVES == 3 ? (half == 0 ? 0 : half + 1) : half * ER;
    const int ern = HALVES == 3 && half > 0 ? 1 : ER;
    __syncthreads();  // every wave is done with the tile buffers
    if constexpr (HALVES > 1) {
        T* const mv = reinterpret_cast<T*>(lds);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) mv[(i * TN + j) * TG_THREADS + tid] = acc[i][j];
        __syncthreads();
        uint32_t took = 0;  // two bits per output: the slice its result came from
#pragma unroll
        for (int i = 0; i < ER; ++i) {
            if (i >= ern) break;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int o = ((er0 + i) * TN + j) * TG_THREADS + tid;
                T v = reinterpret_cast<const T*>(dl64s_lds)[o];
#pragma unroll
                for (int g = 1; g < HALVES; ++g) {
                    const T v1 = reinterpret_cast<const T*>(dl64s_lds + g * Cfg::LDS_BYTES)[o];
                    if (tbetter<SR, T>(v1, v)) {
                        v = v1;
                        took = (took & ~(3u << (2 * (i * TN + j)))) | (uint32_t(g) << (2 * (i * TN + j)));
                    }
                }
                acc[i][j] = v;
            }
        }
        if constexpr (ARGMAX) {
            __syncthreads();
            int32_t* const mi = reinterpret_cast<int32_t*>(lds);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) mi[(i * TN + j) * TG_THREADS + tid] = ch[i][j];
            __syncthreads();
#pragma unroll
            for (int i = 0; i < ER; ++i) {
                if (i >= ern) break;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const uint32_t g = (took >> (2 * (i * TN + j))) & 3u;
                    ch[i][j] = reinterpret_cast<const int32_t*>(
                        dl64s_lds + g * Cfg::LDS_BYTES)[((er0 + i) * TN + j) * TG_THREADS + tid];
                }
            }
            __syncthreads();  // the blocks are free again
        }
    }

    // ---- epilogue ------------------------------------------------------------------
    // f64 outputs whose row and column could meet in a NaN product: recomputed
    // after the stores with the serial rule.
    uint32_t redo = 0;
    auto erow = [&](int i) { return trow(er0 + i); };
    if constexpr (F64) {
        uint32_t cb[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int64_t gc = col0 + tcol(j);
            cb[j] = clsB[gc < N ? gc : N - 1];
        }
#pragma unroll
        for (int i = 0; i < ER; ++i) {
            if (i >= ern) break;
            const int64_t gr = row0 + erow(i);
            const uint32_t ra = clsA[gr < M ? gr : M - 1];
#pragma unroll
            for (int j = 0; j < TN; ++j)
                if (nan_danger<SR>(ra, cb[j])) {
                    redo |= 1u << (i * TN + j);
                    ch[i][j] = -2;
                }
        }
    }
    const bool vec_out = N % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15u) == 0 &&
                         (!ARGMAX || (reinterpret_cast<uintptr_t>(IDX) & 15u) == 0);
    auto store_row = [&](int i) {
        const int64_t gr = row0 + erow(i), gc = col0 + tcol(0);
        if (gr >= M || gc >= N) return;
        T* c = C + gr * N + gc;
        if (vec_out) {  // N a multiple of 4: whole groups only
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                Vec16<T> cv;
                cv.v[0] = acc[i][2 * h];
                cv.v[1] = acc[i][2 * h + 1];
                *reinterpret_cast<Vec16<T>*>(c + 2 * h) = cv;
            }
            if constexpr (ARGMAX) {
                Vec16<int32_t> iv;
#pragma unroll
                for (int e = 0; e < 4; ++e) iv.v[e] = ch[i][e];
                *reinterpret_cast<Vec16<int32_t>*>(IDX + gr * N + gc) = iv;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (gc + e >= N) continue;
                c[e] = acc[i][e];
                if constexpr (ARGMAX) IDX[gr * N + gc + e] = ch[i][e];
            }
        }
    };
    auto redo_outputs = [&]() {
#pragma unroll 1
        while (redo) {
            const int o = __builtin_ctz(redo);
            redo &= redo - 1;
            const int64_t gr = row0 + erow(o / TN), gc = col0 + tcol(o % TN);
            if (gr >= M || gc >= N) continue;
            T v;
            int32_t ix;
            if constexpr (ARGMAX)
                cpu_select<SR, T>(A + gr * K, 1, BT + gc * K, 1, K, v, ix);
            else
                cpu_select<SR, T>(A + gr * K, 1, B + gc, N, K, v, ix);
            C[gr * N + gc] = v;
            if constexpr (ARGMAX) IDX[gr * N + gc] = ix;
        }
    };
    if constexpr (!ARGMAX) {
#pragma unroll
        for (int i = 0; i < ER; ++i)
            if (i < ern) store_row(i);
        if constexpr (F64) redo_outputs();
    } else {
        // Exact first k inside each output's recorded chunk (as tg_gemm_dl): a
        // counting sort by chunk, then one output per thread at a time, every
        // slice's threads taking part.
        constexpr uint16_t NONE = 0xFFFF;
        uint32_t* hist = reinterpret_cast<uint32_t*>(dl64s_lds + Cfg::HIST_OFF);
        uint16_t* chs = reinterpret_cast<uint16_t*>(dl64s_lds + Cfg::CHS_OFF);
        uint16_t* list = reinterpret_cast<uint16_t*>(dl64s_lds + Cfg::LIST_OFF);
        int* misc = reinterpret_cast<int*>(lds + Cfg::MISC_OFF);
        int* const shared_total = reinterpret_cast<int*>(dl64s_lds + Cfg::MISC_OFF) + 8;
        int shift = 0;
        while (((nkt - 1) >> shift) >= Cfg::NB) ++shift;
        const int nb = ((nkt - 1) >> shift) + 1;
        const bool sorter = HALVES == 1 || half == 0;  // scans the buckets
        if (sorter && tid < Cfg::NB) hist[tid] = 0;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ER; ++i) {
            if (i >= ern) break;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                chs[erow(i) * BN + tcol(j)] = ch[i][j] < 0 ? NONE : uint16_t(ch[i][j]);
                if (ch[i][j] >= 0) atomicAdd(&hist[ch[i][j] >> shift], 1u);
            }
        }
        __syncthreads();
        const int cnt = sorter && tid < nb ? int(hist[tid]) : 0;
        int total = 0;
        const int start = block_exclusive_scan(cnt, misc, total, tid);
        if (sorter && tid < nb) hist[tid] = uint32_t(start);
        if (HALVES > 1 && threadIdx.x == 0) *shared_total = total;
        __syncthreads();
        if constexpr (HALVES > 1) total = *shared_total;
#pragma unroll
        for (int i = 0; i < ER; ++i) {
            if (i >= ern) break;
#pragma unroll
            for (int j = 0; j < TN; ++j)
                if (ch[i][j] >= 0)
                    list[atomicAdd(&hist[ch[i][j] >> shift], 1u)] = uint16_t(erow(i) * BN + tcol(j));
        }
        __syncthreads();
        constexpr int NW = CL / 2;  // 16-byte vectors per window
        for (int e = int(threadIdx.x); e < total; e += TG_THREADS * HALVES) {
            const int lid = int(list[e]);
            const int64_t c = int64_t(chs[lid]);
            const int64_t gr = row0 + lid / BN, gc = col0 + (lid & (BN - 1));
            const T* ap = A + (gr < M ? gr : M - 1) * K;
            const T* bp = BT + (gc < N ? gc : N - 1) * K;
            T p[CL];
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                // A pair past K shifts back into the row: its elements come
                // after their originals, or (a straddling pair's first one)
                // belong to the chunk before and cannot match.
                const int64_t k = c * CL + 2 * w < K - 2 ? c * CL + 2 * w : K - 2;
                const Vec16<T> av = *reinterpret_cast<const Vec16<T>*>(ap + k);
                const Vec16<T> bv = *reinterpret_cast<const Vec16<T>*>(bp + k);
                p[2 * w] = tmul<SR, T>(av.v[0], bv.v[0]);
                p[2 * w + 1] = tmul<SR, T>(av.v[1], bv.v[1]);
            }
            T mx = join(p[0], p[1]);
#pragma unroll
            for (int kk = 2; kk < CL; kk += 2) mx = join(join(mx, p[kk]), p[kk + 1]);
            uint32_t bits = 0;
#pragma unroll
            for (int kk = 0; kk < CL; ++kk) bits |= (p[kk] == mx) ? (1u << kk) : 0u;
            int f = bits ? int(__builtin_ctz(bits)) : 0;
            uint32_t neg = 0;
            if constexpr (F64) {
                if (mx == T(0)) {
#pragma unroll
                    for (int kk = 0; kk < CL; ++kk)
                        neg |= kk == f && __builtin_signbit(p[kk]) ? 32u : 0u;
                }
            }
            const int64_t past = c * CL + (f & ~1) - (K - 2);
            if (past > 0) f = f - int(past) > 0 ? f - int(past) : 0;
            chs[lid] = uint16_t(uint32_t(f) | neg);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ER; ++i) {
            if (i >= ern) break;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if (ch[i][j] == -2) {  // redone below
                    ch[i][j] = 0;
                } else if (ch[i][j] < 0) {  // the tropical zero was never beaten
                    acc[i][j] = tzero<SR, T>();
                    ch[i][j] = 0;
                } else {
                    const int r = chs[erow(i) * BN + tcol(j)];
                    ch[i][j] = ch[i][j] * CL + (r & 31);
                    if constexpr (F64) {
                        if (acc[i][j] == T(0)) acc[i][j] = (r & 32) ? -T(0) : T(0);
                    }
                }
            }
            store_row(i);
        }
        if constexpr (F64) redo_outputs();
    }
}

}  // namespace tg
