// kmx_kron.hip -- the reference's standalone Kronecker building blocks on gfx950:
//   kmx_kronmult             Y = kron(A1..Ak) X   (kron_multd.m, Kronmult/kronmult{1..6}.m)
//   kmx_gemm_vbatched        variable-size batched GEMM (Kronmult/gemm_vbatched.m)
//   kmx_kronmult_batch_plan  the per-stage GEMM lists of Kronmult/kronmult{k}_batch.m
#include "kmx_internal.h"
#include "kmx_mma64.h"

#include <algorithm>
#include <cstdio>
#include <mutex>
#include <numeric>

namespace kmx {

// One mode product of the method-1 chain: contract dim `dim` (0 = slowest) of a
// column-major tensor whose dims have current extents ext[] (ext of dim k is
// ncol_k before its contraction and nrow_k after).  One thread per output entry:
// the form for factors whose mode alone is beyond k_mode_group's LDS tile.
struct ModeArgs {
    const double* in;
    double* out;
    const double* A;  // nrow x ncol
    int sr, sc;       // its strides along rows and columns
    long long inner;  // product of extents of dims faster than `dim`
    long long outer;  // product of extents of dims slower than `dim` times nvec
    int nrow, ncol;
};

__global__ void __launch_bounds__(256) k_mode_product(ModeArgs m) {
    const long long total = m.inner * m.nrow * m.outer;
    for (long long e = blockIdx.x * 256ll + threadIdx.x; e < total; e += (long long)gridDim.x * 256) {
        const long long s = e % m.inner;
        const long long r = e / m.inner;
        const int a = int(r % m.nrow);
        const long long o = r / m.nrow;
        const double* in = m.in + o * m.ncol * m.inner + s;
        double acc = 0.0;
        for (int b = 0; b < m.ncol; ++b) acc = __builtin_fma(m.A[(long long)b * m.sc + (long long)a * m.sr], in[b * m.inner], acc);
        m.out[e] = acc;
    }
}

// Several consecutive modes of the chain in one launch.  A workgroup holds, for OC
// values of the slower indices and IC of the faster ones, every value of the group's
// modes in LDS (two buffers) and contracts them last first; each tensor value is read
// and written in HBM once per group instead of once per mode.  A thread takes fibres
// along the mode: the inputs and the factor's columns (the same for every lane) come
// from LDS and up to 16 outputs accumulate in registers.  Factors of more than KG_FACTOR
// values together are read through the scalar cache instead, whose loads cannot be
// waited for one by one (the chain below: 17.0 us so, 16.1 us from LDS).
// Every output sums its products in column order with FMAs from zero, as the one-mode
// kernel does: the results are bit-identical however the chain is grouped.  LDS index
// i sits at i + i / 8: fibres of the fastest mode, ncol apart, spread over the banks.
// Four 8 x 8 factors on 128 vectors: 4 launches, 32 us of kernel time, now 1 of 16 us.
constexpr int KG_THREADS = 512;
constexpr int KG_TILE = 8448;   // values of a tile at most: 2 buffers x 9/8 x 8 bytes = 152 KB of the 160 KB
constexpr int KG_FACTOR = KMX_KRON_ROWMAJOR_VALUES;  // values of the factors kept in LDS
constexpr int KG_MIN_IC = 8;    // contiguous values per access at least when the modes are strided
struct GroupArgs {
    const double* in;
    double* out;
    const double* A[KMX_KRON_MAX_FACTORS];  // the group's factors, slowest first
    int nrow[KMX_KRON_MAX_FACTORS], ncol[KMX_KRON_MAX_FACTORS];
    long long inner;  // extent of the faster (already contracted) modes
    long long outer;  // extent of the slower modes times nvec
    int k, OC, IC, buf;  // buf: doubles of one LDS buffer
    int chunks;          // workgroups along inner
    int foff[KMX_KRON_MAX_FACTORS], nfac;  // the factors' places in LDS, their values (0: not kept there)
    unsigned rowmajor;                     // bit d: factor d is row-major (staged factors only)
};
__device__ __forceinline__ int kg_at(int i) { return i + (i >> 3); }
typedef const __attribute__((address_space(4))) double* kg_factor;  // read through the scalar cache

template <int NR, class P>
__device__ __forceinline__ void kg_fibre(P A, int nrow, int ncol, const double* __restrict__ src,
                                         double* __restrict__ dst, int ib, int ob, int inner) {
    double acc[NR];
#pragma unroll
    for (int a = 0; a < NR; ++a) acc[a] = 0.0;
#pragma unroll 4
    for (int b = 0; b < ncol; ++b) {
        const double x = src[kg_at(ib + b * inner)];
#pragma unroll
        for (int a = 0; a < NR; ++a) acc[a] = __builtin_fma(A[b * nrow + a], x, acc[a]);
    }
#pragma unroll
    for (int a = 0; a < NR; ++a) dst[kg_at(ob + a * inner)] = acc[a];
}

template <int NR, class P>
__device__ __forceinline__ void kg_mode(P A, int nrow, int ncol, int a0,
                                        const double* __restrict__ src, double* __restrict__ dst, int nf, int inner) {
    for (int f = threadIdx.x; f < nf; f += blockDim.x) {
        const int o = f / inner, s = f - o * inner;
        kg_fibre<NR>(A + a0, nrow, ncol, src, dst, o * ncol * inner + s, (o * nrow + a0) * inner + s, inner);
    }
}

// One mode of the tile: every fibre, 16 rows of the factor at a time.
template <class P>
__device__ __forceinline__ void kg_rows(P A, int nr, int nc, const double* __restrict__ src, double* __restrict__ dst,
                                        int nf, int fast) {
    for (int a0 = 0; a0 < nr; a0 += 16) {
        switch (min(16, nr - a0)) {
            case 1: kg_mode<1>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 2: kg_mode<2>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 3: kg_mode<3>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 4: kg_mode<4>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 5: kg_mode<5>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 6: kg_mode<6>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 7: kg_mode<7>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 8: kg_mode<8>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 9: kg_mode<9>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 10: kg_mode<10>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 11: kg_mode<11>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 12: kg_mode<12>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 13: kg_mode<13>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 14: kg_mode<14>(A, nr, nc, a0, src, dst, nf, fast); break;
            case 15: kg_mode<15>(A, nr, nc, a0, src, dst, nf, fast); break;
            default: kg_mode<16>(A, nr, nc, a0, src, dst, nf, fast); break;
        }
    }
}

__global__ void __launch_bounds__(KG_THREADS) k_mode_group(GroupArgs g) {
    extern __shared__ __align__(16) double kg_lds[];
    const long long wg = blockIdx.x;
    const long long ob = wg / g.chunks;
    const long long o0 = ob * g.OC, s0 = (wg - ob * g.chunks) * g.IC;
    const int oc = int(min((long long)g.OC, g.outer - o0)), ic = int(min((long long)g.IC, g.inner - s0));
    int pin = 1, pout = 1;
    for (int d = 0; d < g.k; ++d) {
        pin *= g.ncol[d];
        pout *= g.nrow[d];
    }
    double* src = kg_lds;
    double* dst = kg_lds + g.buf;
    double* fac = kg_lds + 2 * g.buf;
    const bool staged = g.nfac > 0;
    const int nt = blockDim.x;
    // the tile in: value p of the modes, s of the faster indices (IC = inner unless OC = 1),
    // eight loads of a thread in flight
    typedef const __attribute__((address_space(1))) double* gptr;
    const gptr in = (gptr)(g.in + o0 * pin * g.inner + s0);
    const int n_in = oc * pin * g.IC;
    for (int i0 = threadIdx.x; i0 < n_in; i0 += 8 * nt) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = min(i0 + u * nt, n_in - 1);
            const int p = g.IC == 1 ? i : i / g.IC, s = i - p * g.IC;
            v[u] = in[(long long)p * g.inner + min(s, ic - 1)];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i0 + u * nt < n_in) src[kg_at(i0 + u * nt)] = v[u];
    }
    if (staged)
        for (int d = 0; d < g.k; ++d) {
            const gptr A = (gptr)g.A[d];
            const int nr = g.nrow[d], nc = g.ncol[d];
            if (g.rowmajor >> d & 1)
                for (int i = threadIdx.x; i < nr * nc; i += nt) fac[g.foff[d] + i] = A[i % nr * nc + i / nr];
            else
                for (int i = threadIdx.x; i < nr * nc; i += nt) fac[g.foff[d] + i] = A[i];
        }
    __syncthreads();
    int fast = g.IC;  // extent of the faster indices inside the tile
    int slow = oc * pin;
    for (int d = g.k - 1; d >= 0; --d) {
        const int nr = g.nrow[d], nc = g.ncol[d];
        slow /= nc;
        const int nf = slow * fast;
        if (staged) kg_rows(fac + g.foff[d], nr, nc, src, dst, nf, fast);
        else kg_rows((kg_factor)g.A[d], nr, nc, src, dst, nf, fast);
        fast *= nr;
        __syncthreads();
        double* t = src;
        src = dst;
        dst = t;
    }
    __attribute__((address_space(1))) double* out =
        (__attribute__((address_space(1))) double*)(g.out + o0 * pout * g.inner + s0);
    const int n = oc * pout * g.IC;
    for (int i = threadIdx.x; i < n; i += nt) {
        const int p = g.IC == 1 ? i : i / g.IC, s = i - p * g.IC;
        if (s < ic) out[(long long)p * g.inner + s] = src[kg_at(i)];
    }
}

struct GemmDescDev {
    const double* A;
    const double* B;
    double* C;
    int m, n, k, lda, ldb, ldc;
};
// Descriptors that travel with the launch (kernel arguments are limited to 4 KB)
constexpr int GV_CHUNK = 80;
// Batches of up to this many GEMMs run in chunks; beyond, one launch over a device table
// (a launch of 80 small products is ~5 us, the table's set-up ~40 us)
constexpr int GV_MAX_CHUNKED = 8 * GV_CHUNK;
struct GemmChunk {
    GemmDescDev d[GV_CHUNK];
};
// The same in 18 bytes each: sizes below 2^16, leading dimensions the rows stored, matrices
// within 32 GB.  200 ragged products of 33..256 are one launch instead of three, each of
// which ended with 2.3 workgroups a CU: 82 -> 59 us a call; 100 of them 56 -> 38, 90 of
// 200..400 160 -> 140.  Up to GV_CHUNK products one launch does anyway.
constexpr int GV_PACK = 216;
struct GemmPack {
    const double* base;
    unsigned off[3][GV_PACK];  // of A, B, C from base, in doubles
    unsigned short mnk[3][GV_PACK];
};

// The batch's GEMMs in 64 x 64 tiles of C: workgroup (g, t) takes tiles t, t +
// gridDim.y, ... of GEMM g (row-tile fastest), on the FP64 matrix cores
// (kmx_mma64.h).  Every entry sums its k products in order with FMAs, then C = alpha
// sum + beta C (C not read when beta = 0), as the reference's gemm does entry by
// entry.  FP64: 200 ragged products of 33..256 in 58 us of kernel time (121 us with VALU
// FMAs, 84 in three launches), 2048^3 at 51 TFLOP/s (22), 80 x 256^3 at 37 (23).
constexpr int GV_T = 64;
template <bool TA, bool TB>
__device__ __forceinline__ void gemm_tiles(const GemmDescDev& d, double alpha, double beta, double* lds) {
    const GemmDescDev q = d;
    const int mt = (q.m + GV_T - 1) / GV_T, nt = (q.n + GV_T - 1) / GV_T;
    const long long tiles = (long long)mt * nt;
    for (long long tile = blockIdx.y; tile < tiles; tile += gridDim.y) {
        const int i0 = int(tile % mt) * GV_T, j0 = int(tile / mt) * GV_T;
        // loads run along each matrix's contiguous index: i or k of A, k or j of B
        const double* A = TA ? q.A + (long long)i0 * q.lda : q.A + i0;
        const double* B = TB ? q.B + j0 : q.B + (long long)j0 * q.ldb;
        double* C = q.C + (long long)j0 * q.ldc + i0;
        Mma64Strided<Mma64Map<64, 16, TA>> la(A, TA ? q.lda : 1, TA ? 1 : q.lda, q.m - i0, q.k);
        Mma64Strided<Mma64Map<64, 16, !TB>> lb(B, TB ? 1 : q.ldb, TB ? q.ldb : 1, q.n - j0, q.k);
        auto st = [&](int i, int j, double v) {
            double& c = C[(long long)j * q.ldc + i];
            c = (beta == 0.0 ? 0.0 : beta * c) + alpha * v;
        };
        mma64_tile<64, 16>(q.m - i0, q.n - j0, q.k, la, lb, st, lds);
        __syncthreads();  // a next tile's first chunk after this one's last reads
    }
}
template <bool TA, bool TB>
__global__ void __launch_bounds__(256, 2) k_gemm_chunk(GemmChunk c, double alpha, double beta) {
    __shared__ double lds[mma64_lds<64, 16>()];
    gemm_tiles<TA, TB>(c.d[blockIdx.x], alpha, beta, lds);
}
template <bool TA, bool TB>
__global__ void __launch_bounds__(256, 2) k_gemm_pack(GemmPack c, double alpha, double beta) {
    __shared__ double lds[mma64_lds<64, 16>()];
    const int g = blockIdx.x, m = c.mnk[0][g], n = c.mnk[1][g], k = c.mnk[2][g];
    const GemmDescDev d{c.base + c.off[0][g], c.base + c.off[1][g], const_cast<double*>(c.base) + c.off[2][g],
                        m, n, k, max(1, TA ? k : m), max(1, TB ? n : k), max(1, m)};
    gemm_tiles<TA, TB>(d, alpha, beta, lds);
}
template <bool TA, bool TB>
__global__ void __launch_bounds__(256, 2) k_gemm_vbatched(const GemmDescDev* __restrict__ d, double alpha, double beta) {
    __shared__ double lds[mma64_lds<64, 16>()];
    gemm_tiles<TA, TB>(d[blockIdx.x], alpha, beta, lds);
}

// ---- flops_kron{k} (Kronmult/flops_kron2.m:22-46, flops_kron3..6.m): cost of the
// better method for factors [l..k) and whether method 1 wins (ties -> method 1).
static double flops_best(const int* nr, const int* nc, int l, int k, int* method) {
    if (k - l == 1) {
        if (method) *method = 1;
        return 2.0 * nr[l] * nc[l];  // per vector (only used as a product term)
    }
    if (k - l == 2) {
        const double nrow1 = nr[l], ncol1 = nc[l], nrow2 = nr[l + 1], ncol2 = nc[l + 1];
        const double f1 = 2.0 * nrow2 * ncol2 * ncol1 + 2.0 * nrow2 * ncol1 * nrow1;
        const double f2 = 2.0 * ncol2 * ncol1 * nrow1 + 2.0 * nrow2 * ncol2 * nrow1;
        if (method) *method = (f1 <= f2) ? 1 : 2;
        return std::min(f1, f2);
    }
    double inner = flops_best(nr, nc, l + 1, k, nullptr);
    double prow = 1, pcol = 1;
    for (int i = l + 1; i < k; ++i) {
        prow *= nr[i];
        pcol *= nc[i];
    }
    const double f1 = inner * nc[l] + 2.0 * prow * nc[l] * nr[l];
    const double f2 = 2.0 * pcol * nc[l] * nr[l] + inner * nr[l];
    if (method) *method = (f1 <= f2) ? 1 : 2;
    return std::min(f1, f2);
}

struct Emitter {
    const int* nr;
    const int* nc;
    int K;  // number of factors
    std::vector<std::vector<kmx_gemm_desc>> stages;
    long long region = 0;  // elements per scratch region
    bool sizing = true;

    kmx_gemm_desc mk(int stage, char ta, char tb, int m, int n, int k, int lda, int ldb, int ldc, int bA,
                     long long oA, int bB, long long oB, int bC, long long oC) {
        kmx_gemm_desc g;
        g.stage = stage;
        g.transA = ta;
        g.transB = tb;
        g.m = m;
        g.n = n;
        g.k = k;
        g.lda = lda;
        g.ldb = ldb;
        g.ldc = ldc;
        g.alpha = 1.0;
        g.beta = 0.0;
        g.bufA = bA;
        g.offA = oA;
        g.bufB = bB;
        g.offB = oB;
        g.bufC = bC;
        g.offC = oC;
        return g;
    }
    void push(const kmx_gemm_desc& g) {
        if (!sizing) stages[g.stage - 1].push_back(g);
    }
    // factors [l..K), input (bin, oin), output (bout, oout), nvec vectors,
    // first stage index s0, scratch region depth.
    void emit(int l, int bin, long long oin, int bout, long long oout, long long nvec, int s0, int depth) {
        const int nrow1 = nr[l], ncol1 = nc[l];
        const long long tmpoff = (long long)depth * region;
        if (K - l == 1) {  // kronmult1_batch.m:45-61
            push(mk(s0, 'N', 'N', nrow1, int(nvec), ncol1, nrow1, ncol1, nrow1, KMX_BUF_FACTOR + l, 0, bin, oin,
                    bout, oout));
            return;
        }
        long long prow = 1, pcol = 1;
        for (int i = l + 1; i < K; ++i) {
            prow *= nr[i];
            pcol *= nc[i];
        }
        int method;
        flops_best(nr, nc, l, K, &method);
        const int nstage = K - l;
        if (method == 1) {
            // Ytmp = kronmult_{k-1}(A2..Ak, X): prow x (ncol1*nvec) in scratch
            const long long need = prow * ncol1 * nvec;
            if (sizing) region = std::max(region, need);
            emit(l + 1, bin, oin, KMX_BUF_W0, tmpoff, nvec * ncol1, s0, depth + 1);
            for (long long v = 0; v < nvec; ++v)  // kronmult2_batch.m:71-111, kronmult3_batch (method 1)
                push(mk(s0 + nstage - 1, 'N', 'T', int(prow), nrow1, ncol1, int(prow), nrow1, int(prow), KMX_BUF_W0,
                        tmpoff + v * prow * ncol1, KMX_BUF_FACTOR + l, 0, bout, oout + v * prow * nrow1));
        } else {
            // Ytmp(:, v) = X_v * A1^T : pcol x (nrow1*nvec); then kronmult_{k-1}(A2..Ak, Ytmp)
            const long long need = pcol * nrow1 * nvec;
            if (sizing) region = std::max(region, need);
            for (long long v = 0; v < nvec; ++v)
                push(mk(s0, 'N', 'T', int(pcol), nrow1, ncol1, int(pcol), nrow1, int(pcol), bin,
                        oin + v * pcol * ncol1, KMX_BUF_FACTOR + l, 0, KMX_BUF_W0, tmpoff + v * pcol * nrow1));
            emit(l + 1, KMX_BUF_W0, tmpoff, bout, oout, nvec * nrow1, s0 + 1, depth + 1);
        }
    }
};

}  // namespace kmx

using namespace kmx;

extern "C" int kmx_kronmult_batch_plan(int k, const int* nrow, const int* ncol, int nvec, kmx_gemm_desc* out,
                                       int capacity, int* count, int64_t* work_elems) {
    if (k < 1 || k > 6 || !nrow || !ncol || nvec < 1 || !count) {
        set_error("kmx_kronmult_batch_plan: bad arguments");
        return KMX_E_ARG;
    }
    for (int i = 0; i < k; ++i)
        if (nrow[i] < 1 || ncol[i] < 1) {
            set_error("kmx_kronmult_batch_plan: factor sizes must be positive");
            return KMX_E_SHAPE;
        }
    Emitter em{nrow, ncol, k, {}, 0, true};
    em.stages.assign(k, {});
    em.emit(0, KMX_BUF_X, 0, KMX_BUF_Y, 0, nvec, 1, 0);  // sizing pass
    em.sizing = false;
    em.emit(0, KMX_BUF_X, 0, KMX_BUF_Y, 0, nvec, 1, 0);
    int total = 0;
    for (auto& s : em.stages) total += int(s.size());
    *count = total;
    if (work_elems) *work_elems = em.region * k;
    if (out) {
        if (capacity < total) {
            set_error("kmx_kronmult_batch_plan: capacity too small");
            return KMX_E_ARG;
        }
        int o = 0;
        for (auto& s : em.stages)
            for (auto& g : s) out[o++] = g;
    }
    return KMX_OK;
}

namespace {

// Values of the largest intermediate of the method-1 chain (ext[i] = ncol_i until
// dim i is contracted, then nrow_i; nvec vectors).
long long chain_workspace(int k, const int* nrow, const int* ncol, int nvec) {
    std::vector<long long> e2(ncol, ncol + k);
    long long maxsz = 0;
    for (int d = k - 1; d >= 0; --d) {
        e2[d] = nrow[d];
        long long sz = nvec;
        for (int i = 0; i < k; ++i) sz *= e2[i];
        maxsz = std::max(maxsz, sz);
    }
    return maxsz;
}

// The chain's launches: modes [first, last] each, last modes first.  group: one
// k_mode_group launch; otherwise one mode through k_mode_product.
struct ChainStep {
    int first, last;
    bool group;
};

// As many modes as fit the LDS tile go into one launch: the trailing modes with every
// value of theirs contiguous, earlier ones with at least KG_MIN_IC contiguous values of
// the faster indices (all of them where there are fewer).
// A chain of several modes may be given Y on top of X (its first launch has read X
// before its last one writes): then every mode has a launch of its own.
std::vector<ChainStep> plan_chain(int k, const int* nrow, const int* ncol, int nvec, const double* X,
                                  const double* Y) {
    std::vector<ChainStep> steps;
    double nx = nvec, ny = nvec;
    for (int i = 0; i < k; ++i) {
        nx *= ncol[i];
        ny *= nrow[i];
    }
    const double gap = double(reinterpret_cast<intptr_t>(Y) - reinterpret_cast<intptr_t>(X));
    if (k > 1 && gap < 8.0 * nx && -gap < 8.0 * ny) {
        for (int d = k - 1; d >= 0; --d) steps.push_back(ChainStep{d, d, false});
        return steps;
    }
    double inner = 1.0;  // extent of the modes contracted so far
    for (int d = k - 1; d >= 0;) {
        const double ic = std::min<double>(inner, KG_MIN_IC);
        int e = d + 1;  // modes [e, d] fit
        double rows = 1.0;
        for (int q = d; q >= 0; --q) {  // largest extent of modes [q, d] during their contraction
            double cols = 1.0, r = 1.0, most = 0.0;
            for (int i = q; i <= d; ++i) cols *= ncol[i];
            most = cols;
            for (int i = d; i >= q; --i) {
                cols /= ncol[i];
                r *= nrow[i];
                most = std::max(most, cols * r);
            }
            if (most * ic > KG_TILE) break;
            e = q;
            rows = r;
        }
        if (e > d) {
            steps.push_back(ChainStep{d, d, false});
            inner *= nrow[d];
            --d;
        } else {
            steps.push_back(ChainStep{e, d, true});
            inner *= rows;
            d = e - 1;
        }
    }
    return steps;
}

// The mode products of kron(A1..Ak) X, last factor first (method 1), through the
// ping-pong buffers buf[0] / buf[1] (used only when the steps need them).  For k > 6
// this is also the order of kron_multd.m's recursion (kron_multd.m:64-86: Z = A_k X,
// then kron(A_1..A_{k-1}) on Z's transpose).  rowmajor: null, or per factor whether it is
// stored by rows (the factors have KG_FACTOR values at most then: groups keep them in LDS).
hipError_t launch_chain(const std::vector<ChainStep>& steps, int k, const int* nrow, const int* ncol,
                        const double* const* A, const unsigned char* rowmajor, const double* X, int nvec, double* Y,
                        double* const* buf, hipStream_t s) {
    std::vector<long long> ext(ncol, ncol + k);
    const double* cur = X;
    int ping = 0;
    for (const ChainStep& st : steps) {
        double* out = st.first == 0 ? Y : buf[ping];
        long long inner = 1, outer = nvec;
        for (int i = st.last + 1; i < k; ++i) inner *= ext[i];
        for (int i = 0; i < st.first; ++i) outer *= ext[i];
        if (!st.group) {
            ModeArgs m;
            m.in = cur;
            m.out = out;
            m.A = A[st.first];
            m.nrow = nrow[st.first];
            m.ncol = ncol[st.first];
            const bool rm = rowmajor && rowmajor[st.first];
            m.sr = rm ? m.ncol : 1;
            m.sc = rm ? 1 : m.nrow;
            m.inner = inner;
            m.outer = outer;
            const long long total = m.inner * m.nrow * m.outer;
            const int grid = int(std::min<long long>((total + 255) / 256, 65536));
            if (grid > 0) hipLaunchKernelGGL(k_mode_product, dim3(grid), dim3(256), 0, s, m);
        } else {
            GroupArgs g;
            g.in = cur;
            g.out = out;
            g.k = st.last - st.first + 1;
            g.rowmajor = 0;
            long long cols = 1, rows = 1;
            for (int i = 0; i < g.k; ++i) {
                g.rowmajor |= rowmajor && rowmajor[st.first + i] ? 1u << i : 0u;
                g.A[i] = A[st.first + i];
                g.nrow[i] = nrow[st.first + i];
                g.ncol[i] = ncol[st.first + i];
                cols *= g.ncol[i];
            }
            long long most = cols, c = cols;
            for (int i = g.k - 1; i >= 0; --i) {
                c /= g.ncol[i];
                rows *= g.nrow[i];
                most = std::max(most, c * rows);
            }
            g.inner = inner;
            g.outer = outer;
            // faster indices per tile: all of them if they fit, or else multiples of
            // KG_MIN_IC; slower ones until there are ~1024 workgroups, a wave of fibres each
            const long long fit = KG_TILE / most;
            long long ic = std::min(inner, fit);
            if (ic < inner && ic > KG_MIN_IC) ic -= ic % KG_MIN_IC;
            if (ic > 64 && ic < inner && inner * outer / ic < 512) ic = 64;
            long long oc = 1;
            if (ic == inner) {
                oc = std::max((outer + 1023) / 1024, 64 / std::max(1LL, cols * ic / std::max(1, g.ncol[g.k - 1])));
                oc = std::max(1LL, std::min({oc, outer, fit / ic}));
            }
            g.IC = int(ic);
            g.OC = int(oc);
            g.buf = int(most * ic * oc * 9 / 8 + 2);
            g.chunks = int((inner + ic - 1) / ic);
            const long long grid = (outer + oc - 1) / oc * g.chunks;
            g.nfac = 0;
            for (int i = 0; i < g.k; ++i) {
                g.foff[i] = g.nfac;
                g.nfac = int(std::min<long long>(KG_FACTOR + 1LL, g.nfac + (long long)g.nrow[i] * g.ncol[i]));
            }
            if (g.nfac > KG_FACTOR) g.nfac = 0;
            const size_t lds = (2 * size_t(g.buf) + size_t(g.nfac)) * sizeof(double);
            const int nt = most * ic * oc >= 2048 ? KG_THREADS : most * ic * oc >= 512 ? 256 : 64;
            if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
            if (lds > 65536) {
                const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_mode_group),
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
                if (e != hipSuccess) return e;
            }
            hipLaunchKernelGGL(k_mode_group, dim3(unsigned(grid)), dim3(nt), lds, s, g);
        }
        for (int i = st.first; i <= st.last; ++i) ext[i] = nrow[i];
        cur = out;
        ping ^= 1;
    }
    return hipGetLastError();
}

bool kron_args_ok(int k, const int* nrow, const int* ncol, const double* const* A, const double* X, int nvec,
                  const double* Y) {
    if (k < 1 || k > KMX_KRON_MAX_FACTORS || !nrow || !ncol || !A || !X || !Y || nvec < 0) return false;
    for (int i = 0; i < k; ++i)
        if (nrow[i] < 1 || ncol[i] < 1 || !A[i]) return false;
    return true;
}

// work: 2 chain_workspace() doubles of the caller's for the intermediates, or null
int kronmult(const char* who, int k, const int* nrow, const int* ncol, const double* const* A,
             const unsigned char* rowmajor, const double* X, int nvec, double* Y, double* work, void* stream) {
    if (!kron_args_ok(k, nrow, ncol, A, X, nvec, Y)) {
        set_error(std::string(who) + ": bad arguments");
        return KMX_E_ARG;
    }
    if (nvec == 0) return KMX_OK;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const std::vector<ChainStep> steps = plan_chain(k, nrow, ncol, nvec, X, Y);
    double* buf[2] = {nullptr, nullptr};
    if (steps.size() > 1 && work) {
        buf[0] = work;
        buf[1] = work + chain_workspace(k, nrow, ncol, nvec);
    } else if (steps.size() > 1) {  // intermediates between the launches
        const long long maxsz = chain_workspace(k, nrow, ncol, nvec);
        if (hipMalloc(&buf[0], sizeof(double) * maxsz) != hipSuccess ||
            (steps.size() > 2 && hipMalloc(&buf[1], sizeof(double) * maxsz) != hipSuccess)) {
            hipFree(buf[0]);
            set_error(std::string(who) + ": workspace allocation failed");
            return KMX_E_NOMEM;
        }
    }
    const hipError_t e = launch_chain(steps, k, nrow, ncol, A, rowmajor, X, nvec, Y, buf, s);
    if (buf[0] && !work) {
        hipStreamSynchronize(s);
        hipFree(buf[0]);
        if (buf[1]) hipFree(buf[1]);
    }
    if (e != hipSuccess) {
        set_error(std::string(who) + ": " + hipGetErrorString(e));
        return KMX_E_HIP;
    }
    return KMX_OK;
}

}  // namespace

extern "C" int kmx_kronmult(int k, const int* nrow, const int* ncol, const double* const* A, const double* X,
                            int nvec, double* Y, void* stream) {
    return kronmult("kmx_kronmult", k, nrow, ncol, A, nullptr, X, nvec, Y, nullptr, stream);
}

// ---- kmx_kronmult without allocation: the chain's two intermediates live in one
// file-scope device array (each GPU holds its own copy for the life of the
// process).  Its device address is looked up once per device, with that device
// current, and only that address reaches the kernels.
static __device__ __align__(256) double scratch[KMX_KRON_SCRATCH_ELEMS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch[kMaxDevices] = {};

double* scratch_for_current_device() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return nullptr;
        g_scratch[dev] = static_cast<double*>(ptr);
    }
    return g_scratch[dev];
}
}  // namespace

namespace {
int kronmult_noalloc(const char* who, int k, const int* nrow, const int* ncol, const double* const* A,
                     const unsigned char* rowmajor, const double* X, int nvec, double* Y, void* stream) {
    if (!kron_args_ok(k, nrow, ncol, A, X, nvec, Y)) {
        set_error(std::string(who) + ": bad arguments");
        return KMX_E_ARG;
    }
    if (nvec == 0) return KMX_OK;
    const long long maxsz = chain_workspace(k, nrow, ncol, nvec);
    const long long half = KMX_KRON_SCRATCH_ELEMS / 2;
    if (k > 1 && maxsz > half) {
        char msg[200];
        std::snprintf(msg, sizeof msg,
                      "%s: an intermediate of %lld values exceeds the scratch limit of %lld "
                      "(KMX_KRON_SCRATCH_ELEMS / 2); use kmx_kronmult",
                      who, maxsz, half);
        set_error(msg);
        return KMX_E_SHAPE;
    }
    double* base = scratch_for_current_device();
    if (!base) {
        set_error(std::string(who) + ": hipGetSymbolAddress of the scratch array failed");
        return KMX_E_HIP;
    }
    double* buf[2] = {base, base + half};
    const hipError_t e = launch_chain(plan_chain(k, nrow, ncol, nvec, X, Y), k, nrow, ncol, A, rowmajor, X, nvec, Y, buf,
                                      reinterpret_cast<hipStream_t>(stream));
    if (e != hipSuccess) {
        set_error(std::string(who) + ": " + hipGetErrorString(e));
        return KMX_E_HIP;
    }
    return KMX_OK;
}
}  // namespace

extern "C" int kmx_kronmult_noalloc(int k, const int* nrow, const int* ncol, const double* const* A,
                                    const double* X, int nvec, double* Y, void* stream) {
    return kronmult_noalloc("kmx_kronmult_noalloc", k, nrow, ncol, A, nullptr, X, nvec, Y, stream);
}

extern "C" int64_t kmx_kronmult_work(int k, const int* nrow, const int* ncol, int nvec) {
    if (k < 1 || k > KMX_KRON_MAX_FACTORS || !nrow || !ncol || nvec < 1) return 0;
    for (int i = 0; i < k; ++i)
        if (nrow[i] < 1 || ncol[i] < 1) return 0;
    return k == 1 ? 0 : 2 * chain_workspace(k, nrow, ncol, nvec);
}

extern "C" int kmx_kronmult_layout(int k, const int* nrow, const int* ncol, const double* const* A,
                                   const unsigned char* rowmajor, const double* X, int nvec, double* Y, int noalloc,
                                   double* work, void* stream) {
    if (rowmajor && kron_args_ok(k, nrow, ncol, A, X, nvec, Y)) {
        long long values = 0;
        bool any = false;
        for (int i = 0; i < k; ++i) {
            any = any || rowmajor[i];
            values += (long long)nrow[i] * ncol[i];
        }
        if (any && values > KG_FACTOR) {
            set_error("kmx_kronmult_layout: row-major factors of more than KMX_KRON_ROWMAJOR_VALUES values together");
            return KMX_E_SHAPE;
        }
    }
    return noalloc ? kronmult_noalloc("kmx_kronmult_layout", k, nrow, ncol, A, rowmajor, X, nvec, Y, stream)
                   : kronmult("kmx_kronmult_layout", k, nrow, ncol, A, rowmajor, X, nvec, Y, work, stream);
}

extern "C" int kmx_gemm_vbatched(char transA, char transB, const int* m, const int* n, const int* k, double alpha,
                                 const double* const* A, const int* lda, const double* const* B, const int* ldb,
                                 double beta, double* const* C, const int* ldc, int count, void* stream) {
    if (count < 0 || (count > 0 && (!m || !n || !k || !A || !lda || !B || !ldb || !C || !ldc))) {
        set_error("kmx_gemm_vbatched: bad arguments");
        return KMX_E_ARG;
    }
    auto tr = [](char c) { return c == 'T' || c == 't' || c == 'C' || c == 'c'; };
    auto valid = [](char c) { return c == 'N' || c == 'n' || c == 'T' || c == 't' || c == 'C' || c == 'c'; };
    if (!valid(transA) || !valid(transB)) {
        set_error("kmx_gemm_vbatched: trans must be N or T");
        return KMX_E_ARG;
    }
    if (count == 0) return KMX_OK;
    std::vector<GemmDescDev> h(count);
    for (int i = 0; i < count; ++i) {
        if (m[i] < 0 || n[i] < 0 || k[i] < 0) {
            set_error("kmx_gemm_vbatched: negative size");
            return KMX_E_SHAPE;
        }
        const int rowsA = tr(transA) ? k[i] : m[i];
        const int rowsB = tr(transB) ? n[i] : k[i];
        if (lda[i] < std::max(1, rowsA) || ldb[i] < std::max(1, rowsB) || ldc[i] < std::max(1, m[i])) {
            set_error("kmx_gemm_vbatched: leading dimension too small");  // gemm_vbatched.m:17-19 style
            return KMX_E_SHAPE;
        }
        h[i] = GemmDescDev{A[i], B[i], C[i], m[i], n[i], k[i], lda[i], ldb[i], ldc[i]};
    }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    // C tiles of the largest of GEMMs [i0, i1) (grid y; more loop)
    auto tiles_of = [&](int i0, int i1) {
        long long tiles = 1;
        for (int i = i0; i < i1; ++i)
            tiles = std::max(tiles, (long long)((h[i].m + 63) / 64) * ((h[i].n + 63) / 64));
        return unsigned(std::min<long long>(tiles, 65535));
    };
    const bool ta = tr(transA), tb = tr(transB);
    if (count <= GV_MAX_CHUNKED) {
        // Descriptors as kernel arguments, GV_PACK or GV_CHUNK a launch: no table to allocate, copy,
        // wait for and free (some 40 us a call whatever its size).  Longest k first: a
        // workgroup's time goes with k, so a launch holds workgroups of about one length.
        std::stable_sort(h.begin(), h.end(), [](const GemmDescDev& u, const GemmDescDev& v) { return u.k > v.k; });
        const double* lo = h[0].A;
        for (const GemmDescDev& d : h) lo = std::min({lo, d.A, d.B, static_cast<const double*>(d.C)});
        auto offset = [&](const double* q) {
            return (unsigned long long)(reinterpret_cast<uintptr_t>(q) - reinterpret_cast<uintptr_t>(lo));
        };
        auto packs = [&](const GemmDescDev& d) {
            for (const double* q : {d.A, d.B, static_cast<const double*>(d.C)})
                if (offset(q) >> 35 || offset(q) % 8) return false;
            return std::max({d.m, d.n, d.k}) < 65536 && d.lda == std::max(1, ta ? d.k : d.m) &&
                   d.ldb == std::max(1, tb ? d.n : d.k) && d.ldc == std::max(1, d.m);
        };
        const bool pack = count > GV_CHUNK && std::all_of(h.begin(), h.end(), packs);
        const int most = pack ? GV_PACK : GV_CHUNK, launches = (count + most - 1) / most;
        for (int l = 0; l < launches; ++l) {
            const int i0 = int((long long)count * l / launches), i1 = int((long long)count * (l + 1) / launches);
            if (pack) {
                GemmPack c;
                c.base = lo;
                for (int i = i0; i < i1; ++i) {
                    const GemmDescDev& d = h[i];
                    c.off[0][i - i0] = unsigned(offset(d.A) / 8);
                    c.off[1][i - i0] = unsigned(offset(d.B) / 8);
                    c.off[2][i - i0] = unsigned(offset(d.C) / 8);
                    c.mnk[0][i - i0] = (unsigned short)d.m;
                    c.mnk[1][i - i0] = (unsigned short)d.n;
                    c.mnk[2][i - i0] = (unsigned short)d.k;
                }
                auto* kern = ta ? (tb ? k_gemm_pack<true, true> : k_gemm_pack<true, false>)
                                : (tb ? k_gemm_pack<false, true> : k_gemm_pack<false, false>);
                hipLaunchKernelGGL(kern, dim3(unsigned(i1 - i0), tiles_of(i0, i1)), dim3(256), 0, s, c, alpha, beta);
                continue;
            }
            GemmChunk c;
            std::copy(h.begin() + i0, h.begin() + i1, c.d);
            const dim3 grid(unsigned(i1 - i0), tiles_of(i0, i1));
            auto* kern = ta ? (tb ? k_gemm_chunk<true, true> : k_gemm_chunk<true, false>)
                            : (tb ? k_gemm_chunk<false, true> : k_gemm_chunk<false, false>);
            hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, c, alpha, beta);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            set_error(std::string("kmx_gemm_vbatched: ") + hipGetErrorString(e));
            return KMX_E_HIP;
        }
        return KMX_OK;
    }
    GemmDescDev* d = nullptr;
    if (hipMalloc(&d, sizeof(GemmDescDev) * count) != hipSuccess) {
        set_error("kmx_gemm_vbatched: descriptor allocation failed");
        return KMX_E_NOMEM;
    }
    hipMemcpyAsync(d, h.data(), sizeof(GemmDescDev) * count, hipMemcpyHostToDevice, s);
    auto* kern = ta ? (tb ? k_gemm_vbatched<true, true> : k_gemm_vbatched<true, false>)
                    : (tb ? k_gemm_vbatched<false, true> : k_gemm_vbatched<false, false>);
    hipLaunchKernelGGL(kern, dim3(unsigned(count), tiles_of(0, count)), dim3(256), 0, s, d, alpha, beta);
    hipError_t e = hipGetLastError();
    hipStreamSynchronize(s);
    hipFree(d);
    if (e != hipSuccess) {
        set_error(std::string("kmx_gemm_vbatched: ") + hipGetErrorString(e));
        return KMX_E_HIP;
    }
    return KMX_OK;
}
