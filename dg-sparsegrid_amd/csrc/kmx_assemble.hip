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
// element (or a slice of its pairs) and its threads keep fixed places: thread t
// writes entries t, t + 256, ... of every pair's block, so the digits of (r, c) --
// divisions -- are worked out once per entry and thread, not once per value
// written (3D lev 5 deg 3, 372 MB: 1.93 ms with the divisions per value, 0.132 ms
// so: 2.8 TB/s).  For each entry it walks the pairs of its slice, a wave writing
// 512 contiguous bytes per pair (non-temporal stores: 0.150 ms).  The block offsets
// of 128 pairs at a time and, up to 64 KB, the row's coefficient strips (every block
// (I_k, .) of every term) are staged in LDS; block J of a strip starts at J deg^2 and
// the entry's place inside a block is fixed, so a value costs d T LDS reads, the
// products and one store.  Small blocks (B^2 < 256) share the workgroup: G =
// 256 / B^2 pairs at a time.
constexpr int AS_THREADS = 256;
constexpr int AS_PAIRS = 128;

struct AsmArgs {
    KArgs<double> a;
    double* out;
    int B, slices, strip_off[KMX_MAX_DIM], strip_term;  // LDS offsets of (term 0, dim k); doubles per term
};

template <int D, bool LDS>
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
    const int G = BB < AS_THREADS ? AS_THREADS / int(BB) : 1;  // pairs at a time
    const int lane_q = BB < AS_THREADS ? tid / int(BB) : 0;
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
        for (long long ent = tid - lane_q * BB; ent < BB; ent += AS_THREADS) {
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
                double s = 0.0;
                for (int t = 0; t < T; ++t) {
                    double p = 1.0;
#pragma unroll
                    for (int k = 0; k < D; ++k) {
                        const double v = LDS ? strip[t * g.strip_term + at[k]]
                                             : a.blk[a.off[t * D + k] + (long long)ie[k] * a.nb[k] * dd + at[k]];
                        p = k == 0 ? v : __dmul_rn(p, v);
                    }
                    s = __dadd_rn(s, a.scale[t] == 1.0 ? p : __dmul_rn(a.scale[t], p));
                }
                out[q * BB] = s;
            }
            if (BB < AS_THREADS) break;  // one entry per thread
        }
    }
}

template <int D>
hipError_t launch(const AsmArgs& g, int deg, size_t lds, unsigned grid, hipStream_t s) {
    if (lds > 0) {
        auto kern = k_assemble<D, true>;
        if (lds > 65536) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kern, dim3(grid), dim3(AS_THREADS), lds, s, g, deg);
    } else {
        hipLaunchKernelGGL((k_assemble<D, false>), dim3(grid), dim3(AS_THREADS), 0, s, g, deg);
    }
    return hipGetLastError();
}

}  // namespace
}  // namespace kmx

using namespace kmx;

extern "C" int kmx_plan_assemble(kmx_plan* p, double* blocks, void* stream) {
    if (!p || (p->P > 0 && !blocks)) {
        set_error("kmx_plan_assemble: null argument");
        return KMX_E_ARG;
    }
    if (p->N == 0 || p->P == 0) return KMX_OK;
    AsmArgs g;
    std::memset(&g, 0, sizeof(g));
    KArgs<double>& a = g.a;
    a.blk = p->d_blk64;
    for (int i = 0; i < p->T * p->D; ++i) a.off[i] = p->off[i];
    int st = 0;
    for (int k = 0; k < p->D; ++k) {
        a.nb[k] = p->nb[k];
        g.strip_off[k] = st;
        st += p->nb[k] * p->deg * p->deg;
    }
    g.strip_term = st;
    for (int t = 0; t < p->T; ++t) a.scale[t] = p->scale[t];
    a.idx1d = p->d_idx1d;
    a.row_ptr = p->all_pairs ? nullptr : p->d_row_ptr;
    a.cols = p->all_pairs ? nullptr : p->d_cols;
    a.N = p->N;
    a.nterms = p->T;
    g.out = blocks;
    g.B = p->B;
    // at least ~2048 workgroups (a few per CU), each with pairs enough to pay for its strips
    const long long per_row = p->P / p->N + 1;
    g.slices = int(std::max(1LL, std::min<long long>((2048 + p->N - 1) / p->N, per_row / 16)));
    const size_t strips = size_t(st) * p->T * sizeof(double);
    const size_t lds = strips <= 64 * 1024 ? strips : 0;
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
