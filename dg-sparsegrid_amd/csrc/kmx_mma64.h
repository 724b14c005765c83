// kmx_mma64.h -- one FP64 output tile of a matrix product on the matrix cores
// (v_mfma_f64_16x16x4), shared by the batched GEMM and the real-space transform.
//
// A workgroup of four waves computes a TM x 64 tile of C = A B, k in chunks of KC
// staged in LDS in two buffers.  One 16x16x4 product is 64 cycles of a SIMD
// (gfx950's FP64 matrix rate is its vector rate), so what the matrix form buys is
// operand traffic: a wave's 2 x 2 output tiles read four operand values per lane
// and four products, 32 B / clock of LDS per CU against the 128 it has, where one
// FMA per entry read 8 LDS values per 16 FMAs and ran at 30 % of the rate.  The
// matrix pipe runs behind the wave, so everything else of a chunk is placed between
// its products: each step's operands are read one step ahead, the next chunk's LDS
// writes and the loads of two chunks later (a chunk is 1024 cycles of a lone wave,
// less than a load's way to HBM and back) follow a step each.
// TM = 64 (KC = 16) for square-ish products, waves on interleaved 16-row and
// 16-column tiles so that a 32 x 32 product still gives each wave one; TM = 16
// (KC = 32) for products of few rows.  16 x 16 tiles past the edge are skipped.
// Every entry sums its products in k order.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace kmx {

typedef double mma64_v4 __attribute__((ext_vector_type(4)));

template <int TM, int KC>
constexpr int mma64_lds() {  // doubles of LDS
    return 2 * KC * ((TM + 1) + 65);
}

// Where thread tid's u-th value of a chunk of R rows (or columns) x KC sits: along
// consecutive rows, or (ALONGK) along consecutive k.  WAVEK: one k per wave and load.
template <int R_, int KC_, bool ALONGK>
struct Mma64Map {
    static constexpr int R = R_, KC = KC_, N = R * KC / 256;
    static constexpr bool WAVEK = !ALONGK && R == 64;
    static __device__ __forceinline__ int row(int u) {
        const int e = int(threadIdx.x) + 256 * u;
        return ALONGK ? e / KC : e % R;
    }
    static __device__ __forceinline__ int k(int u) {
        if constexpr (WAVEK) return __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6) + 4 * u;
        const int e = int(threadIdx.x) + 256 * u;
        return ALONGK ? e % KC : e / R;
    }
};

// An operand is a class with its Map and load(k0, x): this thread's Map::N values of the
// chunk at k0, rows clamped to the last valid one and k to K - 1 (what a clamped
// row computes is never stored, and a clamped k's value is replaced by zero).
//
// Operands read through global-address-space pointers: a flat load would hold up the LDS
// reads of every step behind it.
typedef const __attribute__((address_space(1))) double* mma64_gptr;
__device__ __forceinline__ mma64_gptr mma64_global(const double* p) { return (mma64_gptr)p; }

// A plain matrix: value (row, k) at base + row rs + k cs.
template <class M>
struct Mma64Strided {
    using Map = M;
    mma64_gptr at[M::WAVEK ? 1 : M::N];  // the thread's rows at k = 0
    long long cs;
    int K;
    __device__ __forceinline__ Mma64Strided(const double* b, long long rs, long long c, int rows, int k) : cs(c), K(k) {
#pragma unroll
        for (int u = 0; u < (M::WAVEK ? 1 : M::N); ++u) at[u] = mma64_global(b) + min(M::row(u), rows - 1) * rs;
    }
    __device__ __forceinline__ void load(int k0, double (&x)[M::N]) {
#pragma unroll
        for (int u = 0; u < M::N; ++u) x[u] = at[M::WAVEK ? 0 : u][min(k0 + M::k(u), K - 1) * cs];
    }
};

// store(i, j, v) gets every entry of the tile inside m x n once; m, n > 0.
template <int TM, int KC, class LA, class LB, class FS>
__device__ __forceinline__ void mma64_tile(int m, int n, int K, LA& la, LB& lb, const FS& store,
                                           double* __restrict__ lds) {
    static_assert(TM == 64 || TM == 16, "tile rows");
    using MA = typename LA::Map;
    using MB = typename LB::Map;
    static_assert(MA::R == TM && MB::R == 64 && MA::KC == KC && MB::KC == KC, "operand maps");
    constexpr int PA = TM + 1, PB = 65, S = KC / 4;
    constexpr int RT = TM == 64 ? 2 : 1, CT = TM == 64 ? 2 : 1;
    double* As = lds;                // [2][KC][PA]
    double* Bs = lds + 2 * KC * PA;  // [2][KC][PB]
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const int r0 = TM == 64 ? 16 * (w & 1) : 0, c0 = TM == 64 ? 16 * (w >> 1) : 16 * w;
    double xa0[MA::N], xb0[MB::N], xa1[MA::N], xb1[MB::N];
    auto putA = [&](int ch, const double (&x)[MA::N]) {
        const int buf = ch & 1, left = K - ch * KC;
#pragma unroll
        for (int u = 0; u < MA::N; ++u) As[(buf * KC + MA::k(u)) * PA + MA::row(u)] = MA::k(u) < left ? x[u] : 0.0;
    };
    auto putB = [&](int ch, const double (&x)[MB::N]) {
        const int buf = ch & 1, left = K - ch * KC;
#pragma unroll
        for (int u = 0; u < MB::N; ++u) Bs[(buf * KC + MB::k(u)) * PB + MB::row(u)] = MB::k(u) < left ? x[u] : 0.0;
    };
    const int nch = (K + KC - 1) / KC;
    if (nch > 0) {
        la.load(0, xa0);
        lb.load(0, xb0);
        if (nch > 1) {
            la.load(KC, xa1);
            lb.load(KC, xb1);
        }
        putA(0, xa0);
        putB(0, xb0);
        if (nch > 1) {
            la.load(2 * KC, xa0);
            lb.load(2 * KC, xb0);
        }
    }
    __syncthreads();
    // The chunks, for a wave with two_r x two_c output tiles (on: any).  The accumulators
    // live inside one loop body without branches around the products: a copy of one
    // waits for the matrix pipe.
    auto run = [&](auto is_on, auto two_r, auto two_c) {
        constexpr bool ON = decltype(is_on)::value;
        constexpr int R = decltype(two_r)::value ? RT : 1, C = decltype(two_c)::value ? CT : 1;
        mma64_v4 acc[R][C];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < C; ++c) acc[r][c] = mma64_v4{0.0, 0.0, 0.0, 0.0};
        const double* as = As + lk * PA + r0 + li;
        const double* bs = Bs + lk * PB + c0 + li;
        double a[2][R], b[2][C];
        auto read = [&](int buf, int s, int slot) {
#pragma unroll
            for (int r = 0; r < R; ++r) a[slot][r] = as[(buf * KC + 4 * s) * PA + 32 * r];
#pragma unroll
            for (int c = 0; c < C; ++c) b[slot][c] = bs[(buf * KC + 4 * s) * PB + 32 * c];
        };
        auto mul = [&](int slot) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < C; ++c)
                    acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[slot][r], b[slot][c], acc[r][c], 0, 0, 0);
        };
        // chunk ch from buffer ch & 1; the other one, last read before this chunk's
        // opening barrier, takes chunk ch + 1 from xa / xb, which then take ch + 3
        // (past the last chunk: its last k again, stored as zeros and not read; without
        // branches the waits count the loads that may stay in flight)
        auto chunk = [&](int ch, int buf, double (&xa)[MA::N], double (&xb)[MB::N]) {
            if constexpr (ON) read(buf, 0, 0);
#pragma unroll
            for (int s = 0; s < S; ++s) {
                if constexpr (ON) {
                    if (s + 1 < S) read(buf, s + 1, (s + 1) & 1);
                    mul(s & 1);
                }
                if (s == 0) {
                    putA(ch + 1, xa);
                    la.load((ch + 3) * KC, xa);
                }
                if (s == 1) {
                    putB(ch + 1, xb);
                    lb.load((ch + 3) * KC, xb);
                }
            }
            __syncthreads();
        };
        int ch = 0;
        for (; ch + 2 <= nch; ch += 2) {
            chunk(ch, 0, xa1, xb1);
            chunk(ch + 1, 1, xa0, xb0);
        }
        if constexpr (ON) {
            if (ch < nch) {  // an odd last chunk, its steps of four k (the last one zero padded)
                const int ns = min(KC, K - ch * KC + 3) >> 2;
                for (int s = 0; s < ns; ++s) {
                    read(0, s, 0);
                    mul(0);
                }
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < C; ++c)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int i = r0 + 32 * r + (lane >> 4) + 4 * q, j = c0 + 32 * c + li;
                        if (i < m && j < n) store(i, j, acc[r][c][q]);
                    }
        }
    };
    const bool r1 = RT == 2 && r0 + 32 < m, c1 = CT == 2 && c0 + 32 < n;
    if (!(r0 < m && c0 < n)) run(std::false_type{}, std::false_type{}, std::false_type{});
    else if (r1 && c1) run(std::true_type{}, std::true_type{}, std::true_type{});
    else if (r1) run(std::true_type{}, std::true_type{}, std::false_type{});
    else if (c1) run(std::true_type{}, std::false_type{}, std::true_type{});
    else run(std::true_type{}, std::false_type{}, std::false_type{});
}

}  // namespace kmx
