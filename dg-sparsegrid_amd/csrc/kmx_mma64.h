// kmx_mma64.h -- one FP64 output tile of a matrix product on the matrix cores
// (v_mfma_f64_16x16x4), shared by the batched GEMM and the real-space transform.
//
// A workgroup of four waves computes a TM x 64 tile of C = A B, k in chunks of KC
// staged in LDS in two buffers: the next chunk's values are loaded into registers
// while the current one is multiplied.  One 16x16x4 product is 64 cycles of a SIMD
// (gfx950's FP64 matrix rate is its vector rate), so what the matrix form buys is
// operand traffic: a wave's 2 x 2 output tiles read four operand values per lane
// and four products, 32 B / clock of LDS per CU against the 128 it has, where one
// FMA per entry read 8 LDS values per 16 FMAs and ran at 30 % of the rate.
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

// fa(i, k): A's value at row i < m, fb(k, j): B's at column j < n; k < K.  store(i, j,
// v) gets every entry of the tile inside m x n once.
template <int TM, int KC, class FA, class FB, class FS>
__device__ __forceinline__ void mma64_tile(int m, int n, int K, const FA& fa, const FB& fb, const FS& store,
                                           double* __restrict__ lds) {
    static_assert(TM == 64 || TM == 16, "tile rows");
    constexpr int PA = TM + 1, PB = 65;
    constexpr int NA = TM * KC / 256, NBL = 64 * KC / 256;  // loads per thread and chunk
    constexpr int RT = TM == 64 ? 2 : 1, CT = TM == 64 ? 2 : 1;
    double* As = lds;                // [2][KC][PA]
    double* Bs = lds + 2 * KC * PA;  // [2][KC][PB]
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const int r0 = TM == 64 ? 16 * (w & 1) : 0, c0 = TM == 64 ? 16 * (w >> 1) : 16 * w;
    mma64_v4 acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[r][c] = mma64_v4{0.0, 0.0, 0.0, 0.0};
    double av[NA], bv[NBL];
    auto load = [&](int k0) {
#pragma unroll
        for (int u = 0; u < NA; ++u) {
            const int e = tid + 256 * u, i = e % TM, k = k0 + e / TM;
            av[u] = (i < m && k < K) ? fa(i, k) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < NBL; ++u) {
            const int e = tid + 256 * u, j = e % 64, k = k0 + e / 64;
            bv[u] = (j < n && k < K) ? fb(k, j) : 0.0;
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int u = 0; u < NA; ++u) {
            const int e = tid + 256 * u;
            As[(buf * KC + e / TM) * PA + e % TM] = av[u];
        }
#pragma unroll
        for (int u = 0; u < NBL; ++u) {
            const int e = tid + 256 * u;
            Bs[(buf * KC + e / 64) * PB + e % 64] = bv[u];
        }
    };
    const int nch = (K + KC - 1) / KC;
    if (nch > 0) {
        load(0);
        put(0);
    }
    __syncthreads();
    for (int ch = 0; ch < nch; ++ch) {
        const int buf = ch & 1;
        if (ch + 1 < nch) load((ch + 1) * KC);
        const int ns = min(KC, K - ch * KC + 3) >> 2;  // steps of four k (the last one zero padded)
        if (r0 < m && c0 < n) {
            const double* as = As + (buf * KC + lk) * PA + r0 + li;
            const double* bs = Bs + (buf * KC + lk) * PB + c0 + li;
            const bool r1 = RT == 2 && r0 + 32 < m, c1 = CT == 2 && c0 + 32 < n;
            auto steps = [&](auto two_r, auto two_c) {
                constexpr bool R1 = decltype(two_r)::value && RT == 2, C1 = decltype(two_c)::value && CT == 2;
                auto step = [&](int s) {
                    const double a0 = as[4 * s * PA], b0 = bs[4 * s * PB];
                    acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
                    if constexpr (C1) {
                        const double b1 = bs[4 * s * PB + 32];
                        acc[0][CT - 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][CT - 1], 0, 0, 0);
                        if constexpr (R1) {
                            const double a1 = as[4 * s * PA + 32];
                            acc[RT - 1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[RT - 1][0], 0, 0, 0);
                            acc[RT - 1][CT - 1] =
                                __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[RT - 1][CT - 1], 0, 0, 0);
                        }
                    } else if constexpr (R1) {
                        const double a1 = as[4 * s * PA + 32];
                        acc[RT - 1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[RT - 1][0], 0, 0, 0);
                    }
                };
                if (ns == KC / 4) {
#pragma unroll
                    for (int s = 0; s < KC / 4; ++s) step(s);
                } else {
                    for (int s = 0; s < ns; ++s) step(s);
                }
            };
            if (r1 && c1) steps(std::true_type{}, std::true_type{});
            else if (r1) steps(std::true_type{}, std::false_type{});
            else if (c1) steps(std::false_type{}, std::true_type{});
            else steps(std::false_type{}, std::false_type{});
        }
        // the other buffer was last read before this chunk's opening barrier
        if (ch + 1 < nch) put(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int i = r0 + 32 * r + (lane >> 4) + 4 * q, j = c0 + 32 * c + li;
                if (i < m && j < n) store(i, j, acc[r][c][q]);
            }
}

}  // namespace kmx
