// kmx_factor.hip -- the FP64 operator apply with its pair sum factored over index tuples.
//
// apply_A.m:100-237 sums, for every row element i and connected element j, the product
// A_{t,1}[I_1, J_1] x ... x A_{t,D}[I_D, J_D] applied to x_j: D block contractions per
// pair and term (kmx_kernels.h).  When the pair list is the tensor product of 1D
// connections over the element set -- all pairs trivially, connect_nD.m:63-106's lists
// by construction; checked exactly, row by row, when the plan is made -- the sum can be
// taken one group of dimensions at a time, with the connections as zero blocks of the 1D
// matrices.  Dimensions 1..K are the prefix, K+1..D the suffix:
//
//   W[(J_1..J_K), (I_K+1..I_D)] = sum over the elements j with that prefix of
//                                 (x)_{d>K} A_d[I_d, J_d] x_j
//   y_i                         = sum over prefixes of (x)_{d<=K} A_d[I_d, J_d] W[prefix, suffix(i)]
//
// for the prefixes and suffixes that occur in the element set (any set: no levels, no
// closure).  Both sums walk a tree of index tuples, so a node's partial sum is
// contracted once for all its children.  3D lev 7 deg 3 (1,903,000 pairs, 3 terms): 5.7
// million block contractions pair by pair, 1.6 million here; 6D lev 4: 1.5 million, 0.2.
//
// The split is made for lanes that agree: a wave's 64 lanes are 64 suffixes (k_factor_
// down) or 64 rows (k_factor_up) and walk the same list of nodes, so x_j and the node
// indices are wave-uniform (scalar loads, scalar FMA operands), nothing diverges, and the
// matrix blocks, stored [J][pair of entries][I], and W, [prefix][pair of values][suffix],
// are read along the lanes, 16 bytes each: a load of 8-byte values costs the address unit
// the same 16 cycles (k_factor_up 3D lev 7 deg 3: 36 us with 8-byte loads, 17 with 16).
// Pair by pair every lane gathers its own x_j and blocks, 64 cache lines per load.
// Prefixes with long lists are cut into virtual nodes of FAC_LIST contractions (their W's
// are summed like any others), the lists into waves' pieces, so the walks balance.
//
// Measured, us (down + up + sum; pair by pair before): 3D lev 7 deg 3 45 + 17 + 5 (135),
// 6D lev 4 deg 2 17 + 17 + 6 (68), 2D 2,145 adapted elements deg 4, 4 terms, transposed
// 62 + 67 + 6 (430).  3D and 6D are bound by the walks' instructions and latencies (4
// waves per SIMD, 3.2e8 and 1.0e8 FMAs; the FMAs alone take 8 and 3 us), 2D by the L2:
// the blocks of 368 column indices for 64 lanes are 3 MB per matrix.
//
// A value of y that is not finite is recomputed pair by pair, with its row: a masked
// block multiplies by zero what the pair list leaves out, which is not the same when x
// holds an infinity or a NaN.
//
// W and the partial sums of y live in workspaces of the plan, a stream's applies in one of up
// to four (the fifth stream takes the one longest unused, behind its last apply), and an
// apply under stream capture -- whose replays this cannot order -- runs pair by pair.
#include "kmx_kernels.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <stdexcept>
#include <type_traits>

using namespace kmx;

namespace kmx {
namespace {

constexpr int FAC_LIST = 24;   // contractions of a virtual node's list at most
constexpr int FAC_REC = 8;     // ints per walk record
constexpr int DOWN_WAVES = 4;  // waves of a workgroup of k_factor_down (each a piece of a list)
constexpr int FAC_PIECE = 12;  // contractions of a piece aimed at
constexpr int FAC_SLOTS = 4;   // workspaces of a plan (streams whose applies overlap) at most
constexpr double FAC_BYTES = 1024e6;  // ... and bytes of them together
constexpr int UP_WAVES = 4;    // waves of a workgroup of k_factor_up (each a range of nodes)

// Wave-uniform reads (x, the records) through the scalar cache: constant during a launch.
typedef const __attribute__((address_space(4))) double* fac_cx;
typedef const __attribute__((address_space(4))) int* fac_ci;

// Kernel arguments lie in host memory: only what every wave reads once stays there.  What a
// wave looks up by term or dimension is a table in device memory.
struct FacTab {
    long long off[KMX_MAX_TERMS * KMX_MAX_DIM];  // of the matrices in fac
    int nb[KMX_MAX_DIM];
    int cls_term[KMX_MAX_TERMS];  // terms, class by class of W
    int nup;                      // up: (class, term whose prefix matrices to use, does W hold the scales) triples
    int up_cls[KMX_MAX_TERMS], up_term[KMX_MAX_TERMS], up_scaled[KMX_MAX_TERMS];
};
typedef const __attribute__((address_space(4))) FacTab* fac_ct;

struct FacArgs {
    const double* x;
    double* W;      // [class][node][column group][pair][suffix][2], see FacShape
    double* part;   // [split][value][row], rows in suffix order
    const double* fac;  // the 1D matrices, [J][pair][I][2]
    const FacTab* tab;
    // down: records of the elements in tree order {element, flushes, J_K+1 .. J_D}
    const int* erec;
    const int* slot;    // one record per wave of a workgroup, see factor_slots
    const int* gidx;    // [suffix dim][suffix]: I_d
    // up: records of the virtual nodes {-, flushes, J_1 .. J_K}
    const int* vrec;
    const int* rgam;    // row (in suffix order) -> suffix
    const int* ridx;    // [prefix dim][row]: I_d
    const int* rowid;   // row -> element
    int G, NV, N, nwg, splits;
    double scale[KMX_MAX_TERMS];
};

__host__ __device__ constexpr int ipow(int a, int n) { return n == 0 ? 1 : a * ipow(a, n - 1); }
// the largest power of DEG dividing `cols` columns of `rows` values each with at most `most` values
constexpr int fit_cols(int deg, int cols, int rows, int most) {
    int c = cols;
    while (c > 1 && c * rows > most) c /= deg;
    return c;
}

template <int D, int DEG>
struct FacShape {
    static constexpr int K = D / 2;             // prefix dimensions
    static constexpr int S = D - K;             // suffix dimensions
    static constexpr int B = ipow(DEG, D);
    static constexpr int U = ipow(DEG, K);      // values of the prefix components
    static constexpr int V = ipow(DEG, S);      // ... of the suffix components
    static constexpr int C = fit_cols(DEG, U, V, 32 / S);   // prefix columns of a down wave
    static constexpr int CB = fit_cols(DEG, V, U, K == 1 ? 16 : 48 / K);  // suffix columns of an up wave
    static constexpr int BS = C * V, BU = CB * U;
    static constexpr int NC = U / C, NCB = V / CB;
    // W of a node: NCB column groups of BU values (prefix component, column in the group) in pairs
    static constexpr int BUP = (BU + 1) / 2, WN = NCB * BUP * 2;
};

// out[.., a, ..] += sum_b m[a][b] in[.., b, ..] along an index of stride ST of N values
template <int DEG, int N, int ST, class In>
__device__ __forceinline__ void contract_add(double (&out)[N], const double (&m)[DEG * DEG], const In& in) {
#pragma unroll
    for (int o = 0; o < N / (ST * DEG); ++o)
#pragma unroll
        for (int s = 0; s < ST; ++s)
#pragma unroll
            for (int b = 0; b < DEG; ++b) {
                const double v = in[o * ST * DEG + b * ST + s];
#pragma unroll
                for (int a = 0; a < DEG; ++a)
                    out[o * ST * DEG + a * ST + s] = __builtin_fma(m[a * DEG + b], v, out[o * ST * DEG + a * ST + s]);
            }
}

// The block of a matrix (`base`: [J][pair][I][2], the block's entries row by row in pairs)
// at column index J and this lane's row index I: 16 bytes per lane and load.
typedef double fac_d2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) fac_d2* fac_g2;
template <int DEG>
__device__ __forceinline__ void load_block(double (&m)[DEG * DEG], const double* base, int J, int nb, int I) {
    constexpr int P = (DEG * DEG + 1) / 2;
    const fac_g2 q = (fac_g2)base + (long long)J * P * nb;
#pragma unroll
    for (int e = 0; e < P; ++e) {
        const fac_d2 v = q[e * nb + I];
        m[2 * e] = v.x;
        if (2 * e + 1 < DEG * DEG) m[2 * e + 1] = v.y;
    }
}

// Blocks of a grid by chunks of consecutive items per XCD (workgroups go to the 8 XCDs in
// turn): what neighbours read meets in one L2.
__device__ __forceinline__ int xcd_item(int items) {
    const int per = (items + 7) / 8;
    const int b = int(blockIdx.x);
    const int it = (b & 7) * per + (b >> 3);
    return (b >> 3) < per && it < items ? it : -1;
}

// One wave: a piece of one virtual node's list in one class (elements ra .. of the class's
// term ti0 to element rb - 1 of its term ti1), 64 suffixes, C prefix columns; the pieces of
// a node lie in one workgroup and are added through LDS.
// t[l]: the sums below suffix dimension K + 1 + l; the element's block is contracted
// along dimension D into t[S - 1], and when the walk leaves a node of depth D - f its
// sum is contracted along that dimension into the level above.
// Four waves a SIMD, but three in 3D deg 4, whose 160 registers spilled at four (lev 7, 3
// terms: 223 us an apply then, 119 at three; lev 6, diffusion: 64, 40).
template <int D, int DEG>
__global__ void __launch_bounds__(DOWN_WAVES * 64, (D == 3 && DEG == 4 ? 3 : 4)) k_factor_down(FacArgs a) {
    using F = FacShape<D, DEG>;
    constexpr int K = F::K, S = F::S, BS = F::BS;
    static_assert(S >= 1 && S <= 3, "up to three suffix dimensions");
    constexpr int EC = BS < 8 ? BS : 8;  // values summed per pass
    __shared__ double red[DOWN_WAVES][EC][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int gb = (a.G + 63) / 64;
    // Workgroups go to the 8 XCDs in turn: each takes gb of the 8 gb units (a suffix block's
    // lists with j % 8 = i), neighbours in one L2, the longest lists first in all of them.
    const int cc = int(blockIdx.x) / 8 % F::NC, q = int(blockIdx.x) / (8 * F::NC);
    const int unit = int(blockIdx.x) % 8 * gb + q % gb, j = q / gb * 8 + unit % 8;
    if (j >= a.nwg) return;
    const int g0 = unit / 8 * 64;
    const fac_ct tab = (fac_ct)a.tab;
    const fac_ci sl = (fac_ci)a.slot + (long long)(j * DOWN_WAVES + w) * FAC_REC;
    const int out_node = sl[0], ti0 = sl[1], ti1 = sl[2], ra = sl[3], rb = sl[4], first = sl[5], last = sl[6];
    const int part = sl[7] & 255, nparts = (sl[7] >> 8) & 255, scaled = (sl[7] >> 16) & 1,
              shared = sl[7] >> 17;
    const bool ok = g0 + lane < a.G;
    const int g = ok ? g0 + lane : a.G - 1;
    int I[S];
#pragma unroll
    for (int l = 0; l < S; ++l) I[l] = a.gidx[l * a.G + g];
    double acc[BS];
    double t[S][BS];
#pragma unroll
    for (int e = 0; e < BS; ++e) acc[e] = t[0][e] = 0.0;
    for (int ti = ti0; ti <= ti1; ++ti) {
        const int tm = tab->cls_term[ti];
        const double sc = scaled ? a.scale[tm] : 1.0;
        const int r0 = ti == ti0 ? ra : first, r1 = ti == ti1 ? rb : last;
        const double* p[S];
        int nb[S];
#pragma unroll
        for (int l = 0; l < S; ++l) {
            p[l] = a.fac + tab->off[tm * D + K + l];
            nb[l] = tab->nb[K + l];
        }
#pragma unroll
        for (int l = 0; l < S; ++l)
            if (l > 0 || S == 1)
#pragma unroll
                for (int e = 0; e < BS; ++e) t[l][e] = 0.0;
        auto step = [&](auto FL, fac_ci rec) {
            constexpr int fl = decltype(FL)::value;  // levels to leave after this element
            double m[DEG * DEG], f[fl ? fl : 1][DEG * DEG];
            load_block<DEG>(m, p[S - 1], rec[2 + S - 1], nb[S - 1], I[S - 1]);
#pragma unroll
            for (int q = 0; q < fl; ++q) {
                const int l = S - 2 - q;
                load_block<DEG>(f[q], p[l], rec[2 + l], nb[l], I[l]);
            }
            const fac_cx xe = (fac_cx)a.x + (long long)rec[0] * F::B + cc * BS;
            contract_add<DEG, BS, 1>(t[S - 1], m, xe);
            if constexpr (fl == S - 1 && S > 1)
#pragma unroll
                for (int e = 0; e < DEG * DEG; ++e) f[fl - 1][e] *= sc;
            if constexpr (fl >= 1) {
                contract_add<DEG, BS, DEG>(t[S - 2], f[0], t[S - 1]);
#pragma unroll
                for (int e = 0; e < BS; ++e) t[S - 1][e] = 0.0;
            }
            if constexpr (fl >= 2) {
                contract_add<DEG, BS, DEG * DEG>(t[S - 3], f[1], t[S - 2]);
#pragma unroll
                for (int e = 0; e < BS; ++e) t[S - 2][e] = 0.0;
            }
        };
#pragma unroll 1
        for (int r = r0; r < r1; ++r) {
            const fac_ci rec = (fac_ci)a.erec + (long long)r * FAC_REC;
            const int fl = S == 1 ? 0 : r + 1 == r1 ? S - 1 : rec[1];
            if (S == 1 || fl == 0) step(std::integral_constant<int, 0>(), rec);
            else if (S == 2 || fl == 1) step(std::integral_constant<int, S >= 2 ? 1 : 0>(), rec);
            else step(std::integral_constant<int, S >= 3 ? 2 : 0>(), rec);
        }
        if constexpr (S == 1)
#pragma unroll
            for (int e = 0; e < BS; ++e) acc[e] = __builtin_fma(sc, t[0][e], acc[e]);
    }
    double(&sum)[BS] = S == 1 ? acc : t[0];
    if (shared) {  // uniform in the workgroup: some node lies in several waves
#pragma unroll
        for (int e0 = 0; e0 < BS; e0 += EC) {
            __syncthreads();
#pragma unroll
            for (int e = 0; e < EC; ++e)
                if (e0 + e < BS) red[w][e][lane] = sum[e0 + e];
            __syncthreads();
            if (part == 0)
                for (int q = 1; q < nparts; ++q)
#pragma unroll
                    for (int e = 0; e < EC; ++e)
                        if (e0 + e < BS) sum[e0 + e] += red[w + q][e][lane];
        }
    }
    if (part == 0 && nparts && ok) {
        constexpr int CB = F::CB, L = F::C * CB;  // values of a column group in this wave
        double* W = a.W + (long long)out_node * F::WN * a.G + 2 * g;
#pragma unroll
        for (int sc = 0; sc < F::NCB; ++sc) {
            auto value = [&](int i) { return sum[i / CB * F::V + sc * CB + i % CB]; };
#pragma unroll
            for (int i = 0; i < L; ++i) {
                if (L % 2 == 0) {  // whole pairs
                    if (i % 2 == 0)
                        *(fac_d2*)(W + (long long)(sc * F::BUP + (cc * L + i) / 2) * a.G * 2) = fac_d2{value(i), value(i + 1)};
                } else {
                    W[(long long)(sc * F::BUP + (cc * L + i) / 2) * a.G * 2 + (cc * L + i) % 2] = value(i);
                }
            }
        }
    }
}

// One workgroup: 64 rows, CB suffix columns, one split of the virtual nodes; its waves take
// consecutive ranges of the split and add their sums in wave order through LDS.
template <int D, int DEG>
__global__ void __launch_bounds__(UP_WAVES * 64, 2) k_factor_up(FacArgs a) {
    using F = FacShape<D, DEG>;
    constexpr int K = F::K, BU = F::BU, CB = F::CB, U = F::U, V = F::V;
    static_assert(K >= 1 && K <= 3, "up to three prefix dimensions");
    constexpr int EC = BU < 8 ? BU : 8;  // values summed per pass
    __shared__ double red[UP_WAVES][EC][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int rb = (a.N + 63) / 64;
    int bi = xcd_item(rb * F::NCB * a.splits);
    if (bi < 0) return;
    const int r0 = (bi % rb) * 64;
    bi /= rb;
    const int sc = bi % F::NCB, split = bi / F::NCB;
    const int r = min(r0 + lane, a.N - 1);
    const int g = a.rgam[r];
    int I[K];
#pragma unroll
    for (int d = 0; d < K; ++d) I[d] = a.ridx[d * a.N + r];
    const int parts = a.splits * UP_WAVES, pi = split * UP_WAVES + w;
    const int v0 = int((long long)a.NV * pi / parts), v1 = int((long long)a.NV * (pi + 1) / parts);
    double acc[BU];
    double u[K][BU];
#pragma unroll
    for (int e = 0; e < BU; ++e) acc[e] = u[0][e] = 0.0;
    const fac_ct tab = (fac_ct)a.tab;
    const int nup = tab->nup;
    for (int ui = 0; ui < nup && v0 < v1; ++ui) {
        const int tm = tab->up_term[ui], cls = tab->up_cls[ui];
        const double scl = tab->up_scaled[ui] ? 1.0 : a.scale[tm];
        const double* p[K];
        int nb[K];
#pragma unroll
        for (int d = 0; d < K; ++d) {
            p[d] = a.fac + tab->off[tm * D + d];
            nb[d] = tab->nb[d];
        }
        const fac_g2 W = (fac_g2)a.W + ((long long)cls * a.NV * F::NCB + sc) * F::BUP * a.G;
        struct In {
            double m[DEG * DEG], wv[BU];
        };
        auto fetch = [&](int v, fac_ci rec, In& x) {
            const fac_g2 Wv = W + (long long)v * F::NCB * F::BUP * a.G;
            load_block<DEG>(x.m, p[K - 1], rec[2 + K - 1], nb[K - 1], I[K - 1]);
#pragma unroll
            for (int e = 0; e < F::BUP; ++e) {
                const fac_d2 q = Wv[e * a.G + g];
                x.wv[2 * e] = q.x;
                if (2 * e + 1 < BU) x.wv[2 * e + 1] = q.y;
            }
        };
#pragma unroll
        for (int d = 0; d < K; ++d)
            if (d > 0 || K == 1)
#pragma unroll
                for (int e = 0; e < BU; ++e) u[d][e] = 0.0;
        fac_ci rec = (fac_ci)a.vrec + (long long)v0 * FAC_REC;
        In x;
        fetch(v0, rec, x);
#pragma unroll(K == 1 ? 2 : 1)
        for (int v = v0; v < v1; ++v) {
            // the next node's block and values during this one's contractions (the last one's again at the end)
            const int vn = min(v + 1, v1 - 1);
            const fac_ci recn = (fac_ci)a.vrec + (long long)vn * FAC_REC;
            In xn;
            fetch(vn, recn, xn);
            contract_add<DEG, BU, CB>(u[K - 1], x.m, x.wv);
            if constexpr (K >= 2) {
                const int fl = v + 1 == v1 ? K - 1 : rec[1];
                if (fl >= 1) {
                    constexpr int l = K - 2;
                    double f[DEG * DEG];
                    load_block<DEG>(f, p[l], rec[2 + l], nb[l], I[l]);
                    if (l == 0)
#pragma unroll
                        for (int e = 0; e < DEG * DEG; ++e) f[e] *= scl;
                    contract_add<DEG, BU, CB * DEG>(u[l], f, u[l + 1]);
#pragma unroll
                    for (int e = 0; e < BU; ++e) u[l + 1][e] = 0.0;
                }
                if constexpr (K >= 3) {
                    if (fl >= 2) {
                        constexpr int l = K - 3;
                        double f[DEG * DEG];
                        load_block<DEG>(f, p[l], rec[2 + l], nb[l], I[l]);
#pragma unroll
                        for (int e = 0; e < DEG * DEG; ++e) f[e] *= scl;
                        contract_add<DEG, BU, CB * DEG * DEG>(u[l], f, u[l + 1]);
#pragma unroll
                        for (int e = 0; e < BU; ++e) u[l + 1][e] = 0.0;
                    }
                }
            }
            x = xn;
            rec = recn;
        }
        if constexpr (K == 1)
#pragma unroll
            for (int e = 0; e < BU; ++e) acc[e] = __builtin_fma(scl, u[0][e], acc[e]);
    }
    const int nr = min(64, a.N - r0);
#pragma unroll
    for (int e0 = 0; e0 < BU; e0 += EC) {
        __syncthreads();
#pragma unroll
        for (int e = 0; e < EC; ++e)
            if (e0 + e < BU) red[w][e][lane] = K == 1 ? acc[e0 + e] : u[0][e0 + e];
        __syncthreads();
        for (int q = threadIdx.x; q < EC * 64; q += UP_WAVES * 64) {
            const int e = q >> 6, l = q & 63;
            if (e0 + e < BU && l < nr) {
                double s = red[0][e][l];
#pragma unroll
                for (int ww = 1; ww < UP_WAVES; ++ww) s += red[ww][e][l];
                const int val = (e0 + e) / CB * V + sc * CB + (e0 + e) % CB;
                a.part[((long long)split * F::B + val) * a.N + r0 + l] = s;
            }
        }
    }
}

// y from the splits' sums, 256 / B rows per workgroup; rows with a value that is not finite
// again, pair by pair.
template <int D, int DEG>
__global__ void __launch_bounds__(256) k_factor_sum(FacArgs a, KArgs<double> k) {
    using F = FacShape<D, DEG>;
    constexpr int R = 256 / F::B;
    static_assert(R >= 1, "blocks of at most 256 values");
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int bad[R];
    const int tid = threadIdx.x;
    if (tid < R) bad[tid] = 0;
    __syncthreads();
    __shared__ double sum[R * F::B];
    {  // rows along the lanes
        const int e = tid / R, rr = tid - e * R, r = int(blockIdx.x) * R + rr;
        if (e < F::B && r < a.N) {
            double s = 0.0;
#pragma unroll 4
            for (int q = 0; q < a.splits; ++q) s += a.part[((long long)q * F::B + e) * a.N + r];
            sum[rr * F::B + e] = s;
            if (!(__builtin_fabs(s) <= 1.7976931348623157e308)) bad[rr] = 1;
        }
    }
    __syncthreads();
    {  // a row's values along the lanes
        const int rr = tid / F::B, r = int(blockIdx.x) * R + rr;
        if (rr < R && r < a.N) k.y[(long long)a.rowid[r] * F::B + tid - rr * F::B] = sum[tid];
    }
    for (int q = 0; q < R; ++q) {
        if (!bad[q]) continue;  // uniform
        const int row = a.rowid[int(blockIdx.x) * R + q];
        if constexpr (F::B <= 32) apply_row<double, D, DEG, 256, 0, false>(k, k.x, k.y, row, smem);
        else if constexpr (DEG == 2 || DEG == 4) apply_row_split<double, D, DEG, 256, 0>(k, k.x, k.y, row, smem);
        __syncthreads();
    }
}

// [I][J][a][b] blocks of the matrices first, first + 1, ... (term by term) -> [J][pair][I][2],
// zero where the dimension's mask[I * nb + J] is 0 and in the half of an odd block's last pair.
// blockIdx.y: the matrix, z: forward or transposed.  One launch for all of them: a launch
// each was 130 us of a 6D plan's set-up.
struct LayoutArgs {
    const double* blk[2];
    double* out[2];
    long long src[KMX_MAX_TERMS * KMX_MAX_DIM], dst[KMX_MAX_TERMS * KMX_MAX_DIM];
    const unsigned char* mask;  // null: none
    long long mask_at[2][KMX_MAX_DIM];
    int nb[KMX_MAX_DIM];
    int D, dd, first;
};
__global__ void __launch_bounds__(256) k_factor_layout(LayoutArgs g) {
    const int m = g.first + int(blockIdx.y), d = m % g.D, o = int(blockIdx.z), dd = g.dd, nb = g.nb[d];
    const double* __restrict__ blk = g.blk[o] + g.src[m];
    double* __restrict__ out = g.out[o] + g.dst[m];
    const unsigned char* __restrict__ mask = g.mask ? g.mask + g.mask_at[o][d] : nullptr;
    const int pairs = (dd + 1) / 2;
    const long long n = (long long)nb * nb * pairs * 2;
    for (long long q = blockIdx.x * 256ll + threadIdx.x; q < n; q += (long long)gridDim.x * 256) {
        const int h = int(q & 1);
        long long r = q >> 1;
        const int I = int(r % nb);
        r /= nb;
        const int ab = int(r % pairs) * 2 + h, J = int(r / pairs);
        const long long at = (long long)I * nb + J;
        out[q] = ab < dd && (!mask || mask[at]) ? blk[at * dd + ab] : 0.0;
    }
}

struct Launch {
    void (*run)(const FacArgs&, const KArgs<double>&, hipStream_t);
    int K, NC, NCB, WN;
};

template <int D, int DEG>
void run_all(const FacArgs& a, const KArgs<double>& k, hipStream_t s) {
    using F = FacShape<D, DEG>;
    const int down = 8 * ((a.nwg + 7) / 8) * F::NC * ((a.G + 63) / 64), up = (a.N + 63) / 64 * F::NCB * a.splits;
    hipLaunchKernelGGL((k_factor_down<D, DEG>), dim3(unsigned(down)), dim3(DOWN_WAVES * 64), 0, s, a);
    hipLaunchKernelGGL((k_factor_up<D, DEG>), dim3(unsigned((up + 7) / 8 * 8)), dim3(UP_WAVES * 64), 0, s, a);
    constexpr int R = 256 / F::B;
    const size_t smem = size_t(4) * F::B * sizeof(double);
    hipLaunchKernelGGL((k_factor_sum<D, DEG>), dim3(unsigned((a.N + R - 1) / R)), dim3(256), smem, s, a, k);
}
template <int D, int DEG>
Launch shape() {
    using F = FacShape<D, DEG>;
    return Launch{&run_all<D, DEG>, F::K, F::NC, F::NCB, F::WN};
}
// Shapes whose rows the pair kernels can recompute (up to 32 values, or 64 split over
// lanes), except 2D deg 5: 25 values over 25-entry blocks leave too few waves (2,145
// elements, all pairs: 246 us against 251 pair by pair, smaller sets slower).
bool pick(int D, int deg, Launch& l) {
    switch (D * 16 + deg) {
        case 0x22: l = shape<2, 2>(); return true;
        case 0x23: l = shape<2, 3>(); return true;
        case 0x24: l = shape<2, 4>(); return true;
        case 0x32: l = shape<3, 2>(); return true;
        case 0x33: l = shape<3, 3>(); return true;
        case 0x34: l = shape<3, 4>(); return true;
        case 0x42: l = shape<4, 2>(); return true;
        case 0x52: l = shape<5, 2>(); return true;
        case 0x62: l = shape<6, 2>(); return true;
        default: return false;
    }
}

template <typename T>
T* fac_upload(const std::vector<T>& h) {
    T* d = nullptr;
    if (hipMalloc(&d, std::max<size_t>(1, h.size()) * sizeof(T)) != hipSuccess) throw std::bad_alloc();
    if (!h.empty() && hipMemcpy(d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess) {
        hipFree(d);
        throw std::runtime_error("hipMemcpy failed");
    }
    return d;
}

// Per dimension the 1D connections of a pair list that is their tensor product over the
// element set (every pair list row equals the product's row, as sets, without
// repetitions); false if it is not one.
bool product_masks(const kmx_plan* p, const std::vector<int>& idx, const std::vector<long long>& rp,
                   const std::vector<int>& cols, std::vector<std::vector<unsigned char>>& mask) {
    const int D = p->D, N = p->N;
    const size_t words = (size_t(N) + 63) / 64;
    double bits = double(N) * double(words) * 8.0;
    for (int d = 0; d < D; ++d) bits += double(p->nb[d]) * double(words) * 16.0;
    if (bits > 512e6) return false;
    typedef unsigned long long word;
    // the rows as bit sets: a word stays in a register while consecutive columns lie in it
    // (3D lev 7, 1,903,000 pairs: 0.9 of the check's 1.2 ms a column at a time, the plan 5.6 ms;
    // 5.3 with whole words.  Four threads took 0.4 once warm, but 3 to 4 ms in each of a
    // process's first plans.)
    std::vector<word> rows(size_t(N) * words, 0);
    for (int i = 0; i < N; ++i) {
        word* row = &rows[size_t(i) * words];
        const int* c = cols.data() + rp[size_t(i)];
        const int* const end = cols.data() + rp[size_t(i) + 1];
        while (c != end) {
            if (end - c >= 64 && *c % 64 == 0) {  // a whole word of consecutive columns
                int other = 0;
                for (int k = 0; k < 64; ++k) other |= c[k] ^ (*c + k);
                if (!other) {
                    row[unsigned(*c) / 64] = ~word(0);
                    c += 64;
                    continue;
                }
            }
            const unsigned at = unsigned(*c) / 64;
            word bits = 0;
            do bits |= word(1) << (unsigned(*c) % 64);
            while (++c != end && unsigned(*c) / 64 == at);
            row[at] |= bits;
        }
        long long held = 0;
        for (size_t k = 0; k < words; ++k) held += __builtin_popcountll(row[k]);
        if (held != rp[size_t(i) + 1] - rp[size_t(i)]) return false;  // a pair listed twice
    }
    // per dimension: (I, J) is connected where a row with index I holds an element with index
    // J; conn: per I the elements j whose J_d is connected to it
    std::vector<std::vector<word>> conn(static_cast<size_t>(D));
    mask.assign(size_t(D), {});
    for (int d = 0; d < D; ++d) {
        const int nb = p->nb[d];
        std::vector<unsigned char>& md = mask[size_t(d)];
        std::vector<word>& c = conn[size_t(d)];
        md.assign(size_t(nb) * nb, 0);
        c.assign(size_t(nb) * words, 0);
        std::vector<word> with(size_t(nb) * words, 0);  // per J the elements that have it
        for (int i = 0; i < N; ++i) {
            const size_t I = size_t(idx[size_t(i) * D + d]);
            with[I * words + size_t(i) / 64] |= word(1) << (i % 64);
            for (size_t k = 0; k < words; ++k) c[I * words + k] |= rows[size_t(i) * words + k];
        }
        for (int I = 0; I < nb; ++I) {
            word* set = &c[size_t(I) * words];
            for (int J = 0; J < nb; ++J) {
                const word* w = &with[size_t(J) * words];
                word any = 0;
                for (size_t k = 0; k < words; ++k) any |= set[k] & w[k];
                md[size_t(I) * nb + J] = any != 0;
            }
            for (int J = 0; J < nb; ++J)
                if (md[size_t(I) * nb + J])
                    for (size_t k = 0; k < words; ++k) set[k] |= with[size_t(J) * words + k];
        }
    }
    for (int i = 0; i < N; ++i)
        for (size_t k = 0; k < words; ++k) {
            word m = ~word(0);
            for (int d = 0; d < D; ++d) m &= conn[size_t(d)][size_t(idx[size_t(i) * D + d]) * words + k];
            if (k + 1 == words && N % 64) m &= (word(1) << (N % 64)) - 1;
            if (m != rows[size_t(i) * words + k]) return false;
        }
    return true;
}

}  // namespace
}  // namespace kmx

struct kmx_factor {
    Launch launch;
    int G = 0, NV = 0, splits = 1;
    bool masked = false;
    int* d_tables = nullptr;  // every index table
    size_t o_erec = 0, o_gidx = 0, o_vrec = 0, o_rgam = 0, o_ridx = 0, o_rowid = 0;
    unsigned char* d_mask = nullptr;
    size_t o_mask[2][KMX_MAX_DIM] = {};  // forward, transposed
    double* d_fac[2] = {nullptr, nullptr};
    double* d_ws = nullptr;  // W, the partial sums, the matrices of d_fac
    size_t w_elems = 0, mat = 0;  // values of W (of `room` classes), of one matrix set
    int room = 0;
    int ncls = 0, cls_ptr[KMX_MAX_TERMS + 1] = {};
    unsigned char cls_scaled[KMX_MAX_TERMS] = {};
    FacTab tab = {};
    FacTab* d_tab = nullptr;
    std::vector<int> vptr, list;  // first record and contractions of every virtual node
    int* d_slot = nullptr;
    int nwg = 0;
    // one apply at a time on a workspace; d_ws holds the first one
    struct Slot {
        double* ws = nullptr;
        hipStream_t last = nullptr;
        unsigned long long turn = 0;  // of its last apply (0: none yet)
    };
    std::mutex mu;
    Slot slot[FAC_SLOTS];
    unsigned long long turns = 0;
    hipEvent_t ev = nullptr;
};

// Classes of W.  Terms with bit-identical prefix matrices share one: their suffix sums add
// up, scaled, before the prefix contractions.  Terms alone in theirs share one, unscaled,
// where the suffix matrices are bit-identical: one W, several prefixes.
static void factor_classes(const kmx_plan* p, kmx_factor* f) {
    const int D = p->D, K = f->launch.K;
    auto same = [&](int t, int s, int d0, int d1) {
        for (int d = d0; d < d1; ++d) {
            const size_t n = size_t(p->n[d]) * p->n[d];
            if (std::memcmp(p->h_blk64.data() + p->off[t * D + d], p->h_blk64.data() + p->off[s * D + d],
                            n * sizeof(double)) != 0)
                return false;
        }
        return true;
    };
    std::vector<std::vector<int>> pre, cls;
    for (int t = 0; t < p->T; ++t) {
        auto c = std::find_if(pre.begin(), pre.end(), [&](const std::vector<int>& q) { return same(t, q[0], 0, K); });
        if (c != pre.end()) c->push_back(t);
        else pre.push_back({t});
    }
    f->tab.nup = 0;
    for (const auto& q : pre) {
        size_t c = cls.size();
        if (q.size() == 1)
            for (c = 0; c < cls.size(); ++c)
                if (cls[c].size() == 1 && same(q[0], cls[c][0], K, D)) break;
        if (c == cls.size()) cls.push_back(q);
        f->tab.up_cls[f->tab.nup] = int(c);
        f->tab.up_term[f->tab.nup++] = q[0];
    }
    f->ncls = int(cls.size());
    int n = 0;
    for (size_t c = 0; c < cls.size(); ++c) {
        f->cls_ptr[c] = n;
        f->cls_scaled[c] = cls[c].size() > 1;
        for (int t : cls[c]) f->tab.cls_term[n++] = t;
    }
    f->cls_ptr[cls.size()] = n;
    for (int u = 0; u < f->tab.nup; ++u) f->tab.up_scaled[u] = f->cls_scaled[f->tab.up_cls[u]];
}

// The waves of k_factor_down: every virtual node's list in every class cut into pieces of
// about FAC_PIECE contractions, at most DOWN_WAVES of them, packed into workgroups.
static void factor_slots(kmx_factor* f) {
    struct Node {
        int v, c, cost, np;
    };
    std::vector<Node> nodes;
    for (int c = 0; c < f->ncls; ++c)
        for (int v = 0; v < f->NV; ++v) {
            const int cost = f->list[size_t(v)] * (f->cls_ptr[c + 1] - f->cls_ptr[c]);
            const int seq = (f->vptr[size_t(v) + 1] - f->vptr[size_t(v)]) * (f->cls_ptr[c + 1] - f->cls_ptr[c]);
            nodes.push_back({v, c, cost, std::min({DOWN_WAVES, seq, (cost + FAC_PIECE - 1) / FAC_PIECE})});
        }
    // the longest pieces first
    std::stable_sort(nodes.begin(), nodes.end(), [](const Node& a, const Node& b) {
        return (a.cost + a.np - 1) / a.np > (b.cost + b.np - 1) / b.np;
    });
    std::vector<int> fill;                            // waves taken of every workgroup
    std::vector<int> open[DOWN_WAVES + 1];            // workgroups with this many waves free
    std::vector<int> slot;
    for (const Node& n : nodes) {
        int wg = -1;
        for (int r = n.np; r <= DOWN_WAVES && wg < 0; ++r)
            if (!open[r].empty()) {
                wg = open[r].front();
                open[r].erase(open[r].begin());
            }
        if (wg < 0) {
            wg = int(fill.size());
            fill.push_back(0);
            slot.resize(slot.size() + size_t(DOWN_WAVES) * FAC_REC, 0);
            for (int w = 0; w < DOWN_WAVES; ++w) slot[(size_t(wg) * DOWN_WAVES + w) * FAC_REC + 2] = -1;  // no terms
        }
        const int v0 = f->vptr[size_t(n.v)], len = f->vptr[size_t(n.v) + 1] - v0;
        const int t0 = f->cls_ptr[n.c], seq = len * (f->cls_ptr[n.c + 1] - t0);
        for (int q = 0; q < n.np; ++q) {
            const int a = int((long long)seq * q / n.np), b = int((long long)seq * (q + 1) / n.np) - 1;  // a <= b
            int* s = &slot[(size_t(wg) * DOWN_WAVES + fill[size_t(wg)] + q) * FAC_REC];
            s[0] = n.c * f->NV + n.v;
            s[1] = t0 + a / len;
            s[2] = t0 + b / len;
            s[3] = v0 + a % len;
            s[4] = v0 + b % len + 1;
            s[5] = v0;
            s[6] = v0 + len;
            s[7] = q | n.np << 8 | int(f->cls_scaled[n.c]) << 16;
        }
        fill[size_t(wg)] += n.np;
        if (fill[size_t(wg)] < DOWN_WAVES) open[DOWN_WAVES - fill[size_t(wg)]].push_back(wg);
    }
    f->nwg = int(fill.size());
    for (int wg = 0; wg < f->nwg; ++wg) {  // bit 17: the workgroup has a node in several waves
        int* s = &slot[size_t(wg) * DOWN_WAVES * FAC_REC];
        bool shared = false;
        for (int w = 0; w < DOWN_WAVES; ++w) shared = shared || (s[w * FAC_REC + 7] >> 8 & 255) > 1;
        for (int w = 0; w < DOWN_WAVES; ++w) s[w * FAC_REC + 7] |= int(shared) << 17;
    }
    int* d = fac_upload(slot);
    if (f->d_slot) hipFree(f->d_slot);
    f->d_slot = d;
    FacTab* t = fac_upload(std::vector<FacTab>(1, f->tab));
    if (f->d_tab) hipFree(f->d_tab);
    f->d_tab = t;
}

// Matrices [first, first + count) of the plan into the walks' layout.
static void factor_layout(const kmx_plan* p, kmx_factor* f, int first, int count, hipStream_t s) {
    LayoutArgs g;
    std::memset(&g, 0, sizeof(g));
    g.blk[0] = p->d_blk64;
    g.blk[1] = p->d_blkT64;
    for (int o = 0; o < 2; ++o) {
        g.out[o] = f->d_fac[o];
        for (int d = 0; d < p->D; ++d) g.mask_at[o][d] = (long long)f->o_mask[o][d];
    }
    g.mask = f->masked ? f->d_mask : nullptr;
    std::copy(p->off, p->off + p->T * p->D, g.src);
    std::copy(f->tab.off, f->tab.off + p->T * p->D, g.dst);
    std::copy(p->nb, p->nb + p->D, g.nb);
    g.D = p->D;
    g.dd = p->deg * p->deg;
    g.first = first;
    long long n = 0;
    for (int m = first; m < first + count; ++m)
        n = std::max(n, (long long)p->nb[m % p->D] * p->nb[m % p->D] * (g.dd + 1));
    hipLaunchKernelGGL(k_factor_layout, dim3(unsigned(std::min<long long>((n + 255) / 256, 8192)), unsigned(count),
                                             f->d_fac[1] ? 2u : 1u),
                       dim3(256), 0, s, g);
}

// The workspace for the classes that there are, with every matrix laid out in it: W of T
// classes would be three times as much on a 6D diffusion operator (42 -> 17 MB at lev 4).
static void factor_workspace(const kmx_plan* p, kmx_factor* f, hipStream_t s) {
    for (kmx_factor::Slot& t : f->slot) {  // (hipFree waits for what still runs on them)
        if (t.ws && t.ws != f->d_ws) hipFree(t.ws);
        t = kmx_factor::Slot();
    }
    if (f->d_ws) hipFree(f->d_ws);
    f->d_ws = f->d_fac[0] = f->d_fac[1] = nullptr;
    f->room = f->ncls;
    f->w_elems = size_t(f->ncls) * f->NV * f->launch.WN * size_t(f->G);
    const size_t ws = (f->w_elems + size_t(f->splits) * p->N * p->B + 31) / 32 * 32;
    if (hipMalloc(&f->d_ws, (ws + f->mat * (p->d_blkT64 ? 2 : 1)) * sizeof(double)) != hipSuccess) {
        f->d_ws = nullptr;
        throw std::bad_alloc();
    }
    f->slot[0].ws = f->d_ws;
    f->d_fac[0] = f->d_ws + ws;
    if (p->d_blkT64) f->d_fac[1] = f->d_fac[0] + f->mat;
    factor_layout(p, f, 0, p->T * p->D, s);
    if (hipStreamSynchronize(s) != hipSuccess || hipGetLastError() != hipSuccess)
        throw std::runtime_error("factor layout");
}

void kmx_factor_build(kmx_plan* p, const std::vector<int>& idx, const std::vector<long long>& rp,
                      const std::vector<int>& cols) {
    Launch L;
    const int D = p->D, N = p->N, T = p->T;
    if (!pick(D, p->deg, L) || N < 2) return;
    const double unit = double(p->B) * p->deg;
    const double pair_fma = double(p->P) * T * D * unit;
    const char* env = std::getenv("KMX_FACTOR_MIN_FMA");  // from this many of the pairs' FMAs on instead of the rule below
    if (env && pair_fma < std::atof(env)) return;
    const int K = L.K, S = D - K;
    // elements in tree order: by index tuple, dimension 1 slowest
    std::vector<int> order(static_cast<size_t>(N));
    std::iota(order.begin(), order.end(), 0);
    auto ix = [&](int e, int d) { return idx[size_t(e) * D + d]; };
    auto cmp_from = [&](int a, int b, int d0, int d1) {  // -1, 0, 1 over dims [d0, d1)
        for (int d = d0; d < d1; ++d)
            if (ix(a, d) != ix(b, d)) return ix(a, d) < ix(b, d) ? -1 : 1;
        return 0;
    };
    std::sort(order.begin(), order.end(), [&](int a, int b) { return cmp_from(a, b, 0, D) < 0; });
    for (int i = 0; i + 1 < N; ++i)
        if (cmp_from(order[size_t(i)], order[size_t(i) + 1], 0, D) == 0) return;  // an index tuple twice
    // virtual nodes: runs of one prefix, cut at FAC_LIST contractions (elements and flushes)
    std::vector<int> vptr, vcost, vfirst;
    long long contr = 0;
    for (int i = 0; i < N;) {
        vptr.push_back(i);
        int c = 0, j = i;
        while (j < N && cmp_from(order[size_t(i)], order[size_t(j)], 0, K) == 0 && (j == i || c < FAC_LIST)) {
            c += 1;
            if (j > i)
                for (int d = K; d + 1 < D; ++d)
                    if (cmp_from(order[size_t(j) - 1], order[size_t(j)], K, d + 1) != 0) ++c;
            ++j;
        }
        vcost.push_back(c + S - 1);
        contr += c + S - 1;
        i = j;
    }
    const int NV = int(vptr.size());
    vptr.push_back(N);
    // suffixes and rows in suffix order
    std::vector<int> rows(order);
    std::sort(rows.begin(), rows.end(), [&](int a, int b) {
        const int c = cmp_from(a, b, K, D);
        return c != 0 ? c < 0 : cmp_from(a, b, 0, K) < 0;
    });
    std::vector<int> rgam(static_cast<size_t>(N)), gfirst;
    for (int r = 0; r < N; ++r) {
        if (r == 0 || cmp_from(rows[size_t(r) - 1], rows[size_t(r)], K, D) != 0) gfirst.push_back(rows[size_t(r)]);
        rgam[size_t(r)] = int(gfirst.size()) - 1;
    }
    const int G = int(gfirst.size());
    // Where it is faster, by times measured over 2D lev 4-8 deg 2-4, 3D lev 3-7 deg 2-4, 4D to
    // 6D deg 2, level-limited and adapted sets: the three launches and their walks take 18 us
    // and 6e12 (2D) or 7e12 FMAs / s in whole waves, the pair kernels at best 4.7e12 or 1.1e13
    // (2D lev 7 deg 3 adapted: 26 against 22 us, lev 8: 44 against 139; 3D lev 6 deg 3: 29
    // against 27, lev 7: 66 against 135; 6D lev 4 deg 2: 41 against 77).  The pair kernels do
    // 5.5e12 in 2D deg 2 (lev 8, all pairs, 4 terms: 26.6 against 21.5 us; adapted, 2 terms:
    // 26.7 against 42.7) and 1.25e13 with 3 terms in 3D (lev 6 deg 3, all pairs: 27.6 against
    // 25.9; lev 7 deg 2, all pairs: 27.3 against 29.4).
    const double lanes = double((G + 63) / 64) * 64.0, rlanes = double((N + 63) / 64) * 64.0;
    const double fac_fma = T * (double(contr) * lanes + double(NV) * rlanes) * unit;
    // 3D deg 4, whose 16-entry blocks are cheaper here and whose pairs are split over four
    // lanes there: 19 us and 1e13 against 11 us and 1.2e13 (lev 5, 6 terms: 28 against 51; lev
    // 6, 3 terms: 41 / 80; lev 4 adapted, 6 terms: 25 / 35; lev 4, 6 terms: 23 / 20.5).
    const double pair_rate = D == 2 ? (p->deg == 2 ? 5.5e12 : 4.7e12) : D == 3 && T <= 3 ? 1.25e13 : 1.1e13;
    const bool slower = D == 3 && p->deg == 4
                            ? 19e-6 + fac_fma / 1e13 > 11e-6 + pair_fma / 1.2e13
                            : 18e-6 + fac_fma / (D == 2 ? 6e12 : 7e12) > pair_fma / pair_rate;
    if (!env && slower) return;
    const double w_elems = double(T) * NV * L.WN * double(G);
    if (w_elems * 8.0 > FAC_BYTES) return;
    auto f = new kmx_factor();
    f->launch = L;
    f->G = G;
    f->NV = NV;
    p->fac = f;
    try {
        std::vector<std::vector<unsigned char>> mask;
        if (!p->all_pairs) {
            if (!product_masks(p, idx, rp, cols, mask)) {
                kmx_factor_free(p);
                return;
            }
            for (const auto& m : mask)
                for (unsigned char c : m) f->masked = f->masked || !c;
        }
        std::vector<int> tab;
        auto add = [&](const std::vector<int>& h) {
            const size_t o = tab.size();
            tab.insert(tab.end(), h.begin(), h.end());
            while (tab.size() % 64) tab.push_back(0);
            return o;
        };
        std::vector<int> erec(size_t(N) * FAC_REC, 0), vrec(size_t(NV) * FAC_REC, 0), gidx(size_t(S) * G),
            ridx(size_t(K) * N);
        for (int v = 0; v < NV; ++v) {
            for (int i = vptr[size_t(v)]; i < vptr[size_t(v) + 1]; ++i) {
                int* r = &erec[size_t(i) * FAC_REC];
                r[0] = order[size_t(i)];
                int m = K;  // the first suffix dimension in which the next element of the node differs
                if (i + 1 < vptr[size_t(v) + 1])
                    while (ix(order[size_t(i)], m) == ix(order[size_t(i) + 1], m)) ++m;
                r[1] = D - 1 - m;
                for (int l = 0; l < S; ++l) r[2 + l] = ix(order[size_t(i)], K + l);
            }
            int* r = &vrec[size_t(v) * FAC_REC];
            const int e = order[size_t(vptr[size_t(v)])];
            int m = 0;
            if (v + 1 < NV) {
                const int n = order[size_t(vptr[size_t(v) + 1])];
                while (m < K && ix(e, m) == ix(n, m)) ++m;
            }
            r[1] = m < K ? K - 1 - m : 0;  // m = K: the same prefix goes on
            for (int d = 0; d < K; ++d) r[2 + d] = ix(e, d);
        }
        for (int l = 0; l < S; ++l)
            for (int g = 0; g < G; ++g) gidx[size_t(l) * G + g] = ix(gfirst[size_t(g)], K + l);
        for (int d = 0; d < K; ++d)
            for (int r = 0; r < N; ++r) ridx[size_t(d) * N + r] = ix(rows[size_t(r)], d);
        f->o_erec = add(erec);
        f->o_gidx = add(gidx);
        f->o_vrec = add(vrec);
        f->o_rgam = add(rgam);
        f->o_ridx = add(ridx);
        f->o_rowid = add(rows);
        f->d_tables = fac_upload(tab);
        if (f->masked) {
            std::vector<unsigned char> all;
            for (int o = 0; o < (p->d_blkT64 ? 2 : 1); ++o)
                for (int d = 0; d < D; ++d) {
                    const int nb = p->nb[d];
                    f->o_mask[o][d] = all.size();
                    for (int I = 0; I < nb; ++I)
                        for (int J = 0; J < nb; ++J)
                            all.push_back(mask[size_t(d)][o ? size_t(J) * nb + I : size_t(I) * nb + J]);
                }
            f->d_mask = fac_upload(all);
        }
        f->vptr = vptr;
        f->list = vcost;
        for (int d = 0; d < D; ++d) f->tab.nb[d] = p->nb[d];
        for (int t = 0; t < T; ++t)
            for (int d = 0; d < D; ++d) {
                f->tab.off[t * D + d] = (long long)f->mat;
                f->mat += size_t(p->nb[d]) * p->nb[d] * ((p->deg * p->deg + 1) / 2 * 2);
            }
        factor_classes(p, f);
        factor_slots(f);
        // splits of the node list until some 2048 waves run
        const long long wgs = (long long)((N + 63) / 64) * L.NCB;
        f->splits = int(std::max(1LL, std::min<long long>(512 / wgs, NV / (2 * UP_WAVES) + 1)));
        if (hipEventCreateWithFlags(&f->ev, hipEventDisableTiming) != hipSuccess) throw std::bad_alloc();
        factor_workspace(p, f, nullptr);
    } catch (const std::exception&) {  // no room: the plan runs pair by pair
        (void)hipGetLastError();
        kmx_factor_free(p);
    }
}

void kmx_factor_term_copied(kmx_plan* p, int term, int dim, hipStream_t s) {
    if (p->fac) factor_layout(p, p->fac, term * p->D + dim, 1, s);
}

void kmx_factor_term_updated(kmx_plan* p, hipStream_t s) {
    if (!p->fac) return;
    kmx_factor* f = p->fac;
    const FacTab tab = f->tab;
    try {
        factor_classes(p, f);
        if (std::memcmp(&tab, &f->tab, sizeof(tab)) == 0) return;
        factor_slots(f);
        if (f->ncls > f->room) factor_workspace(p, f, s);  // the matrix split a class
    } catch (const std::exception&) {  // no room: the plan runs pair by pair
        (void)hipGetLastError();
        kmx_factor_free(p);
    }
}

bool kmx_factor_ok(const kmx_plan* p, bool transpose) { return p->fac && p->fac->d_fac[transpose ? 1 : 0]; }

// A workspace for an apply on s: the stream's own last one, one that no stream has, or the one
// whose last apply is longest ago, behind that apply; null if that cannot be waited for.  So
// that applies on several streams overlap, as the pair kernels' do: 4D lev 5 deg 2, 8 terms,
// two streams in turn 39 us an apply with one workspace, 16.6 with one each (16.0 pair by
// pair); 3D lev 5 deg 4, 6 terms 39 and 17.8 (26.9).
static kmx_factor::Slot* factor_slot(const kmx_plan* p, kmx_factor* f, hipStream_t s) {
    kmx_factor::Slot* old = f->slot;
    const size_t bytes = (f->w_elems + size_t(f->splits) * p->N * p->B) * sizeof(double);
    for (int i = 0; i < FAC_SLOTS && double(bytes) * (i + 1) <= std::max(FAC_BYTES, double(bytes)); ++i) {
        kmx_factor::Slot& t = f->slot[i];
        if (t.ws && (!t.turn || t.last == s)) return &t;
        if (!t.ws) {
            // (another thread's capture must not see the allocation)
            hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
            const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
            const hipError_t e = hipMalloc(&t.ws, bytes);
            if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
            if (e == hipSuccess) return &t;
            t.ws = nullptr;
            (void)hipGetLastError();
            break;
        }
        if (t.turn < old->turn) old = &t;
    }
    // a last stream that records a graph now cannot be ordered against
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    const hipError_t q = hipStreamIsCapturing(old->last, &cap);
    (void)hipGetLastError();
    if (cap != hipStreamCaptureStatusNone || q == hipErrorStreamCaptureImplicit) return nullptr;
    if (hipEventRecord(f->ev, old->last) != hipSuccess || hipStreamWaitEvent(s, f->ev, 0) != hipSuccess) {
        (void)hipGetLastError();  // (a stream that is gone, or captures now)
        if (hipDeviceSynchronize() != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
    }
    return old;
}

// 1: launched; 0: this call runs pair by pair; negative: an error
int kmx_factor_apply(kmx_plan* p, bool transpose, const KArgs<double>& k, hipStream_t s) {
    kmx_factor* f = p->fac;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return 0;
    }
    FacArgs a;
    std::memset(&a, 0, sizeof(a));
    a.x = k.x;
    a.fac = f->d_fac[transpose ? 1 : 0];
    std::memcpy(a.scale, p->scale, sizeof(a.scale));
    a.tab = f->d_tab;
    a.erec = f->d_tables + f->o_erec;
    a.slot = f->d_slot;
    a.nwg = f->nwg;
    a.gidx = f->d_tables + f->o_gidx;
    a.vrec = f->d_tables + f->o_vrec;
    a.rgam = f->d_tables + f->o_rgam;
    a.ridx = f->d_tables + f->o_ridx;
    a.rowid = f->d_tables + f->o_rowid;
    a.G = f->G;
    a.NV = f->NV;
    a.N = p->N;
    a.splits = f->splits;
    std::lock_guard<std::mutex> lock(f->mu);
    kmx_factor::Slot* slot = factor_slot(p, f, s);
    if (!slot) return 0;
    a.W = slot->ws;
    a.part = slot->ws + f->w_elems;
    f->launch.run(a, k, s);
    slot->last = s;
    slot->turn = ++f->turns;
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error(std::string("factored apply launch: ") + hipGetErrorString(e));
        return KMX_E_HIP;
    }
    return 1;
}

void kmx_factor_free(kmx_plan* p) {
    kmx_factor* f = p->fac;
    if (!f) return;
    if (f->d_tables) hipFree(f->d_tables);
    if (f->d_slot) hipFree(f->d_slot);
    if (f->d_tab) hipFree(f->d_tab);
    if (f->d_mask) hipFree(f->d_mask);
    for (kmx_factor::Slot& t : f->slot)
        if (t.ws && t.ws != f->d_ws) hipFree(t.ws);
    if (f->d_ws) hipFree(f->d_ws);
    if (f->ev) hipEventDestroy(f->ev);
    delete f;
    p->fac = nullptr;
}
