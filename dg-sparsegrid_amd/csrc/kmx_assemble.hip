// kmx_assemble.hip -- the assembled operator of apply_A.m's build_A branch
// (apply_A.m:170-180 dense A, 150-155 and 246-248 the sparse triplets), on the
// device: for every connected pair (row element e, column element j) in the plan's
// pair order (rows in element order, a row's pairs in connectivity order), the
// deg^d x deg^d block sum_t scale_t krond(A_{t,1}(I_1, J_1), ..., A_{t,d}(I_d, J_d))
// (krond.m:7-17: dim 1 slowest), column-major -- the values A_s3 collects
// (view(:)), in its order.  Row / column of block entry (r, c) of pair (e, j):
// e * B + r and j * B + c (0-based, B = deg^d), as A_s2 / A_s1 hold them.
// Each entry multiplies its d factors left to right and adds the terms in order,
// without fused multiply-adds, as krond's successive kron products and
// apply_A.m's `A = A + view` do.
#include "kmx_internal.h"

#include <algorithm>
#include <cstring>

namespace kmx {
namespace {

// Bound by the blocks it writes (B^2 values a pair).  A workgroup takes one row
// element (or a slice of its pairs) and its threads keep fixed places inside every
// pair's block, so the digits of (r, c) -- divisions -- are worked out once per thread,
// not once per value written.  The block offsets of 128 pairs at a time and, up to
// 64 KB, the row's coefficient strips (every block (I_k, .) of every term) are staged
// in LDS; block J of a strip starts at J deg^2 and an entry's place inside a block is
// fixed.  With one entry a thread a value cost d T LDS reads, as many as the stores
// take: a thread's entries now share all but the column digits of dimensions 1 and 2
// (deg^2 of them, B^2 / deg^2 values apart: lanes still store runs), 2 deg + d - 2
// reads a term for deg^2 values.  3D lev 5 deg 3, 372 MB: 1.93 ms with the divisions
// per value, 0.132 with one entry a thread, 0.090 now, 4.1 TB/s (a fill of the same
// size: 6.2); 3D lev 4 deg 4 0.182 -> 0.087.  Small pairs share the workgroup.
constexpr int AS_THREADS = 256;
constexpr int AS_PAIRS = 128;

struct AsmArgs {
    KArgs<double> a;
    double* out;
    int B, slices, strip_off[KMX_MAX_DIM], strip_term;  // LDS offsets of (term 0, dim k); doubles per term
};

// A thread's C1 x C2 entries: all column digits of dimension 1 (C1 = deg) and of
// dimension 2 (C2 = deg), or one
template <int D, int C1, int C2, bool LDS>
__global__ void __launch_bounds__(AS_THREADS) k_assemble(AsmArgs g, int deg) {
    extern __shared__ __align__(16) double strip[];
    __shared__ int place[AS_PAIRS][D];
    const KArgs<double>& a = g.a;
    const int e = int(blockIdx.x) / g.slices, sl = int(blockIdx.x) - e * g.slices;
    const int tid = threadIdx.x, T = a.nterms, dd = deg * deg;
    const long long q0 = a.row_ptr ? a.row_ptr[e] : (long long)e * a.N;
    const int nq = int(a.row_ptr ? a.row_ptr[e + 1] - q0 : a.N);
    const int per = (nq + g.slices - 1) / g.slices;
    const int qa = sl * per, qb = min(nq, qa + per);
    if (qa >= qb) return;
    int ie[D];
#pragma unroll
    for (int k = 0; k < D; ++k) ie[k] = a.idx1d[(long long)e * D + k];
    if (LDS) {
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int k = 0; k < D; ++k) {
                const double* src = a.blk + a.off[t * D + k] + (long long)ie[k] * a.nb[k] * dd;
                double* dst = strip + t * g.strip_term + g.strip_off[k];
                for (int v = tid; v < a.nb[k] * dd; v += AS_THREADS) dst[v] = src[v];
            }
        __syncthreads();
    }
    const long long BB = (long long)g.B * g.B;
    constexpr int E = C1 * C2;
    const int s2 = g.B / (C2 == 1 ? 1 : C1 * C2);  // columns from one digit of dimension 2 to the next
    const long long BE = BB / E;  // threads of a pair
    const int G = BE < AS_THREADS ? AS_THREADS / int(BE) : 1;  // pairs at a time
    const int lane_q = BE < AS_THREADS ? tid / int(BE) : 0;
    for (int qc = qa; qc < qb; qc += AS_PAIRS) {  // the block offsets of the next pairs, in LDS
        const int nc = min(AS_PAIRS, qb - qc);
        if (qc > qa) __syncthreads();
        for (int v = tid; v < nc * D; v += AS_THREADS) {
            const int q = v / D, k = v - q * D;
            const int j = a.row_ptr ? a.cols[q0 + qc + q] : qc + q;
            place[q][k] = a.idx1d[(long long)j * D + k] * dd;
        }
        __syncthreads();
        if (lane_q >= G) continue;
        for (long long ent = tid - lane_q * BE; ent < BE; ent += AS_THREADS) {
            const int c = int(ent / g.B), r = int(ent - (long long)c * g.B);  // column-major inside the block
            int in[D];  // the entry's place inside block (I_k, J_k)
            int rr = r, cc = c;
#pragma unroll
            for (int k = D - 1; k >= 0; --k) {  // digits of r and c, dim 1 slowest
                const int r1 = rr / deg, c1 = cc / deg;
                in[k] = (rr - r1 * deg) * deg + cc - c1 * deg + (LDS ? g.strip_off[k] : 0);
                rr = r1;
                cc = c1;
            }
            double* out = g.out + (q0 + qc) * BB + ent;
#pragma unroll 2
            for (int q = lane_q; q < nc; q += G) {
                int at[D];
#pragma unroll
                for (int k = 0; k < D; ++k) at[k] = place[q][k] + in[k];
                double s[E];
#pragma unroll
                for (int x = 0; x < E; ++x) s[x] = 0.0;
                for (int t = 0; t < T; ++t) {
                    auto factor = [&](int k, int x) {
                        return LDS ? strip[t * g.strip_term + at[k] + x]
                                   : a.blk[a.off[t * D + k] + (long long)ie[k] * a.nb[k] * dd + at[k] + x];
                    };
                    double v[D], w[C2];
#pragma unroll
                    for (int k = 1; k < D; ++k)
                        if (k > 1 || C2 == 1) v[k] = factor(k, 0);
                    if constexpr (C2 > 1)
#pragma unroll
                        for (int y = 0; y < C2; ++y) w[y] = factor(1, y);
#pragma unroll
                    for (int x = 0; x < C1; ++x) {
                        const double u = factor(0, x);
#pragma unroll
                        for (int y = 0; y < C2; ++y) {
                            double p = u;
#pragma unroll
                            for (int k = 1; k < D; ++k) p = __dmul_rn(p, k == 1 && C2 > 1 ? w[y] : v[k]);
                            s[x * C2 + y] = __dadd_rn(s[x * C2 + y], a.scale[t] == 1.0 ? p : __dmul_rn(a.scale[t], p));
                        }
                    }
                }
#pragma unroll
                for (int x = 0; x < C1; ++x)
#pragma unroll
                    for (int y = 0; y < C2; ++y)
                        out[q * BB + (long long)(x * (g.B / C1) + y * s2) * g.B] = s[x * C2 + y];
            }
            if (BE < AS_THREADS) break;  // one entry per thread
        }
    }
}

template <int D, int C1, int C2, bool LDS>
hipError_t launch_as(const AsmArgs& g, int deg, size_t lds, unsigned grid, hipStream_t s) {
    hipLaunchKernelGGL((k_assemble<D, C1, C2, LDS>), dim3(grid), dim3(AS_THREADS), lds, s, g, deg);
    return hipGetLastError();
}

// In 1D a pair's block is a block of the strip, read once: the strips stay in global memory
// (lev 8 deg 4, all pairs, 2 terms: 46.9 us from LDS, 6.5 now; lev 9 deg 4, connected 14.4, 7.7)
template <int D>
hipError_t launch(const AsmArgs& g, int deg, size_t lds, unsigned grid, hipStream_t s) {
    constexpr bool LDS = D > 1;
    if (LDS && lds == 0) return launch_as<D, 1, 1, false>(g, deg, lds, grid, s);
    // both digits while a pair's threads fill a wave: shorter runs store in pieces
    const bool two = D > 1 && (long long)g.B * g.B >= 64ll * deg * deg;
    switch (deg) {
        case 2:
            return two ? launch_as<D, 2, D == 1 ? 1 : 2, LDS>(g, deg, lds, grid, s)
                       : launch_as<D, 2, 1, LDS>(g, deg, lds, grid, s);
        case 3:
            return two ? launch_as<D, 3, D == 1 ? 1 : 3, LDS>(g, deg, lds, grid, s)
                       : launch_as<D, 3, 1, LDS>(g, deg, lds, grid, s);
        case 4:
            return two ? launch_as<D, 4, D == 1 ? 1 : 4, LDS>(g, deg, lds, grid, s)
                       : launch_as<D, 4, 1, LDS>(g, deg, lds, grid, s);
        default: return launch_as<D, 1, 1, LDS>(g, deg, lds, grid, s);
    }
}

// The operator's diagonal, a workgroup per element: how often the element's row lists the
// element itself (once in a connectivity list) times sum_t scale_t prod_k of the diagonal
// blocks' diagonals.
struct DiagArgs {
    KArgs<double> a;
    double* out;
    int D, deg, B;
};
__global__ void __launch_bounds__(AS_THREADS) k_diagonal(DiagArgs g) {
    __shared__ int own;
    const KArgs<double>& a = g.a;
    const int e = blockIdx.x, tid = threadIdx.x, dd = g.deg * g.deg;
    if (tid == 0) own = a.row_ptr ? 0 : 1;
    __syncthreads();
    if (a.row_ptr) {
        int n = 0;
        for (long long q = a.row_ptr[e] + tid; q < a.row_ptr[e + 1]; q += AS_THREADS) n += a.cols[q] == e;
        if (n) atomicAdd(&own, n);
        __syncthreads();
    }
    for (int r = tid; r < g.B; r += AS_THREADS) {
        double s = 0.0;
        for (int t = 0; t < a.nterms; ++t) {
            double p = a.scale[t];
            int rr = r;
            for (int k = g.D - 1; k >= 0; --k) {  // digits of r, dim 1 slowest
                const int r1 = rr / g.deg, ab = (rr - r1 * g.deg) * (g.deg + 1), I = a.idx1d[(long long)e * g.D + k];
                p *= a.blk[a.off[t * g.D + k] + ((long long)I * a.nb[k] + I) * dd + ab];
                rr = r1;
            }
            s += p;
        }
        g.out[(long long)e * g.B + r] = own ? own * s : 0.0;
    }
}

// What the kernels here read of a plan
void operator_args(const kmx_plan* p, KArgs<double>& a) {
    a.blk = p->d_blk64;
    for (int i = 0; i < p->T * p->D; ++i) a.off[i] = p->off[i];
    for (int k = 0; k < p->D; ++k) a.nb[k] = p->nb[k];
    for (int t = 0; t < p->T; ++t) a.scale[t] = p->scale[t];
    a.idx1d = p->d_idx1d;
    a.row_ptr = p->all_pairs ? nullptr : p->d_row_ptr;
    a.cols = p->all_pairs ? nullptr : p->d_cols;
    a.N = p->N;
    a.nterms = p->T;
}

}  // namespace
}  // namespace kmx

using namespace kmx;

extern "C" int kmx_plan_diagonal(kmx_plan* p, double* d, void* stream) {
    if (!p || (p->N > 0 && !d)) {
        set_error("kmx_plan_diagonal: null argument");
        return KMX_E_ARG;
    }
    if (p->N == 0) return KMX_OK;
    DiagArgs g;
    std::memset(&g, 0, sizeof(g));
    operator_args(p, g.a);
    g.out = d;
    g.D = p->D;
    g.deg = p->deg;
    g.B = p->B;
    hipLaunchKernelGGL(k_diagonal, dim3(unsigned(p->N)), dim3(AS_THREADS), 0, reinterpret_cast<hipStream_t>(stream), g);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string("kmx_plan_diagonal: ") + hipGetErrorString(e));
        return KMX_E_HIP;
    }
    return KMX_OK;
}

extern "C" int kmx_plan_assemble(kmx_plan* p, double* blocks, void* stream) {
    if (!p || (p->P > 0 && !blocks)) {
        set_error("kmx_plan_assemble: null argument");
        return KMX_E_ARG;
    }
    if (p->N == 0 || p->P == 0) return KMX_OK;
    AsmArgs g;
    std::memset(&g, 0, sizeof(g));
    operator_args(p, g.a);
    int st = 0;
    for (int k = 0; k < p->D; ++k) {
        g.strip_off[k] = st;
        st += p->nb[k] * p->deg * p->deg;
    }
    g.strip_term = st;
    g.out = blocks;
    g.B = p->B;
    const size_t strips = size_t(st) * p->T * sizeof(double);
    const size_t lds = p->D > 1 && strips <= 64 * 1024 ? strips : 0;
    // Workgroups: about 2048, each of 16 pairs at least to pay for its strips.  Blocks of 256
    // values and more: two rounds of what the CUs hold (3D lev 5 deg 3, 3.5 thousand: 99 -> 90
    // us; 3D lev 4 deg 4, whose 37 KB of strips leave four a CU: 85 us with 2 thousand, 96 with
    // 4), of as few pairs as write twice the strips' values (6D lev 2 deg 2, 28 rows of 28
    // pairs: 133 -> 38 us).
    const long long per_row = p->P / p->N + 1, BB = (long long)p->B * p->B;
    long long want = 2048, least = 16;
    if (BB >= AS_THREADS) {
        want = 512 * std::min<long long>(8, 160 * 1024 / (long long)(lds + sizeof(int) * AS_PAIRS * p->D));
        least = std::min(16LL, 1 + 2LL * st * p->T / BB);
    }
    g.slices = int(std::max(1LL, std::min<long long>((want + p->N - 1) / p->N, per_row / least)));
    const unsigned grid = unsigned(p->N) * unsigned(g.slices);
    const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    hipError_t e = hipErrorInvalidValue;
    switch (p->D) {
        case 1: e = launch<1>(g, p->deg, lds, grid, s); break;
        case 2: e = launch<2>(g, p->deg, lds, grid, s); break;
        case 3: e = launch<3>(g, p->deg, lds, grid, s); break;
        case 4: e = launch<4>(g, p->deg, lds, grid, s); break;
        case 5: e = launch<5>(g, p->deg, lds, grid, s); break;
        case 6: e = launch<6>(g, p->deg, lds, grid, s); break;
    }
    if (e != hipSuccess) {
        set_error(std::string("kmx_plan_assemble: ") + hipGetErrorString(e));
        return KMX_E_HIP;
    }
    return KMX_OK;
}
