// kmx_realspace.hip -- wavelet space -> real space on gfx950
// (wavelet_to_realspace.m:1-79).
//
// The reference sums, over elements e, kron(Meval_1(:, J_1(e)), ..., Meval_d(:, J_d(e)))
// times the element's deg^d coefficients, where Meval_k(:, J) is the deg-column
// block of dimension k's evaluation matrix at the element's 1D index.  Here the
// sum runs dimension by dimension, last first, over the tree of index prefixes:
// with the elements sorted by (J_1, ..., J_d), a node of depth k is a distinct
// prefix (J_1, ..., J_k), and
//
//   Z_k[node (J_1..J_{k-1}); b_1..b_{k-1}; p_k, p_{k+1}..p_d] =
//       sum over its children J_k and b_k of Meval_k(p_k, (J_k, b_k)) Z_{k+1}[child; b_1..b_k; p_{k+1}..p_d]
//
// with Z_{d+1} the coefficients and Z_1 the result: d launches of products whose k
// index runs over a node's children, each value of Z written once.  (One Kronecker
// product per level tuple added into the output instead -- 84 tuples x 4 launches
// on a 3D lev 6 grid, each re-reading and adding all 192^3 points -- took 6.5 ms.)
// The products run on the FP64 matrix cores (kmx_mma64.h).  3D lev 6 deg 3 (192^3
// points): 0.106 ms with every child in every tile, the last stage's 2.7 GFLOP 71 us of
// it; 0.076 (44) since a tile of 64 points leaves out the children whose Meval block is
// zero on it.  Error against 64 bits 3.5e-16 (4.6e-16 by level tuples).  Same terms,
// summed in another order.
#include "kmx_internal.h"
#include "kmx_mma64.h"

#include <algorithm>
#include <cstring>
#include <map>
#include <numeric>
#include <stdexcept>
#include <vector>

namespace kmx {
namespace {

// One stage.  Nodes are consecutive; node q's children are cptr[q] .. cptr[q + 1] - 1
// with first Meval columns col[c]; nbeta = deg^(k - 1) values of (b_1..b_{k-1}).
struct StageArgs {
    const double* in;
    double* out;
    const double* A;   // Meval_k, M x (columns), column-major
    const int* cptr;
    const int* col;
    const int* row;    // last dimension: the child's element
    long long R;       // values of (p_{k+1}..p_d)
    int M, deg, nbeta, B;
    unsigned magic;    // 2^32 / deg + 1
    int items;         // node x beta (node alone in the last dimension)
    int mt, nt;        // tiles per item
    int xcd;           // 1: the row tiles of a column tile run on one XCD
    // Per node and tile of 64 points the children whose Meval block is not zero there
    // (null: every child everywhere): lptr[node * ptiles + tile], first columns, and the
    // child's place in its node's list (last dimension: its element).
    const int* lptr;
    const int* lcol;
    const int* lx;
    int ptiles;
    // A zero of Meval times an infinity or a NaN is a NaN everywhere: a stage that stores a
    // value that is not finite sets its own *flag to the call's number, and the next one,
    // which reads it as *before, takes every child (and stores such a value itself, so it
    // tells the one after).  No launch reads what it writes: the waves of a workgroup have
    // to agree on the list, or they pass different numbers of barriers.  (A replayed graph
    // finds its own number of a run before: the same sums, only more of them.)
    int* flag;
    const int* before;  // (last dimension: null, it looks at the coefficients themselves)
    int call;
};

// The children that a tile of a node's points sums over.
struct Children {
    const int* col;
    const int* x;  // (null: 0, 1, ...)
    int n;
};
__device__ __forceinline__ Children children(const StageArgs& a, int q, int tile, bool every, const int* x) {
    const int c0 = a.cptr[q];
    if (every) return Children{a.col + c0, x ? x + c0 : nullptr, a.cptr[q + 1] - c0};
    const int l0 = a.lptr[q * a.ptiles + tile];
    return Children{a.lcol + l0, a.lx + l0, a.lptr[q * a.ptiles + tile + 1] - l0};
}
__device__ __forceinline__ bool finite(double v) { return __builtin_fabs(v) <= 1.7976931348623157e308; }

// k / deg and k % deg of a position in a child list (k < 2^28; magic = 2^32 / deg + 1)
__device__ __forceinline__ void split_k(int k, const StageArgs& a, int& c, int& b) {
    c = a.deg == 1 ? k : int(__umulhi(unsigned(k), a.magic));
    b = k - c * a.deg;
}

// A list of k positions of a node, 64 at a time, one per lane (each lane works its
// own out once); the next 64 are fetched while these are used.  Chunks are read in
// order and never straddle a block of 64.
template <class F>
struct KList {
    const F f;
    const int K;
    int cur, nxt, blk;
    __device__ __forceinline__ KList(const F& fn, int k) : f(fn), K(k), blk(0) {
        const int l = int(threadIdx.x) & 63;
        cur = f(min(l, K - 1));
        nxt = f(min(64 + l, K - 1));
    }
    __device__ __forceinline__ void to(int k0) {
        if (k0 < K && k0 >> 6 != blk) {
            blk = k0 >> 6;
            cur = nxt;
            nxt = f(min(64 * (blk + 1) + (int(threadIdx.x) & 63), K - 1));
        }
    }
    __device__ __forceinline__ int at(int k) const { return __builtin_amdgcn_readlane(cur, k & 63); }
};

// Operand whose k-th line (64 consecutive values, one k per wave) starts at base +
// line(k) ld.
template <class M, class F>
struct LineOperand {
    using Map = M;
    static_assert(M::WAVEK, "one k per wave");
    KList<F> list;
    mma64_gptr at;  // the lane's value of line 0
    long long ld;
    __device__ __forceinline__ LineOperand(const F& line, const double* b, long long l, int rows, int K)
        : list(line, K), at(mma64_global(b) + min(int(threadIdx.x) & 63, rows - 1)), ld(l) {}
    __device__ __forceinline__ void load(int k0, double (&x)[M::N]) {
        list.to(k0);
#pragma unroll
        for (int u = 0; u < M::N; ++u) x[u] = at[list.at(min(k0 + M::k(u), list.K - 1)) * ld];
    }
};

// The coefficients of a node's elements: rows beta, value (beta, k) of element c(k).
template <class M>
struct CoefOperand {
    using Map = M;
    const StageArgs& a;
    const int* row;  // the children's elements
    int K, beta0, rows;
    __device__ __forceinline__ void load(int k0, double (&x)[M::N]) {
#pragma unroll
        for (int u = 0; u < M::N; ++u) {
            int c, b;
            split_k(min(k0 + M::k(u), K - 1), a, c, b);
            x[u] = mma64_global(a.in)[(long long)row[c] * a.B + (beta0 + min(M::row(u), rows - 1)) * a.deg + b];
        }
    }
};

// The last dimension: Z_d[node; beta; p] = sum_k f[element(k), beta, b(k)] Meval_d(p, k).
// Rows beta (few), columns p; a chunk of 32 k keeps enough loads in flight for the
// long child lists of the low prefixes.
__global__ void __launch_bounds__(256, 2) k_rs_last(StageArgs a) {
    __shared__ double lds[mma64_lds<16, 32>()];
    const int tiles = a.mt * a.nt;
    const int q = int(blockIdx.x) / tiles, t = int(blockIdx.x) - q * tiles;
    if (q >= a.items) return;
    const int i0 = 16 * (t % a.mt), j0 = 64 * (t / a.mt);
    bool every = !a.lptr;
    if (!every) {  // (or a coefficient of the node that is not finite)
        const int c0 = a.cptr[q];
        const unsigned B = unsigned(a.B), n = unsigned(a.cptr[q + 1] - c0) * B;
        int bad = 0;
        for (unsigned i = threadIdx.x; i < n; i += 256) {
            const unsigned c = i / B;
            bad |= !finite(a.in[(long long)a.row[c0 + c] * B + (i - c * B)]);
        }
        every = __syncthreads_or(bad);
    }
    const Children ch = children(a, q, t / a.mt, every, a.row);
    const int K = ch.n * a.deg;
    auto column = [&](int k) {
        int c, b;
        split_k(k, a, c, b);
        return ch.col[c] + b;
    };
    CoefOperand<Mma64Map<16, 32, false>> la{a, ch.x, K, i0, a.nbeta - i0};
    LineOperand<Mma64Map<64, 32, false>, decltype(column)> lb(column, a.A + j0, a.M, a.M - j0, K);
    double* out = a.out + (long long)q * a.nbeta * a.M;
    bool bad = false;
    auto st = [&](int i, int j, double v) {
        bad |= !finite(v);
        out[(long long)(i0 + i) * a.M + j0 + j] = v;
    };
    mma64_tile<16, 32>(a.nbeta - i0, a.M - j0, K, la, lb, st, lds);
    if (bad) *a.flag = a.call;
}

// Dimension k < d: Z_k[node; beta; p, r] = sum_k Meval_k(p, k) Z_{k+1}[child(k); beta, b(k); r].
// The column tiles of an item are dealt so that the workgroups of one column tile
// (its row tiles, which read the same values of Z_{k+1}) share an XCD's L2.
__global__ void __launch_bounds__(256, 2) k_rs_mode(StageArgs a) {
    __shared__ double lds[mma64_lds<64, 16>()];
    __shared__ int before;
    const int per = a.xcd ? a.mt * ((a.nt + 7) / 8) * 8 : a.mt * a.nt;
    const int item = int(blockIdx.x) / per, t = int(blockIdx.x) - item * per;
    if (item >= a.items) return;
    int rt, ct;
    if (a.xcd) {
        rt = (t / 8) % a.mt;
        ct = (t / 8) / a.mt * 8 + t % 8;
        if (ct >= a.nt) return;
    } else {
        rt = t % a.mt;
        ct = t / a.mt;
    }
    const int q = item / a.nbeta, beta = item - q * a.nbeta;
    const int i0 = 64 * rt;
    const long long j0 = 64LL * ct;
    const int c0 = a.cptr[q];
    bool every = !a.lptr;
    if (!every) {  // one read for the workgroup, whatever another stream's call writes meanwhile
        if (threadIdx.x == 0) before = *a.before;
        __syncthreads();
        every = before == a.call;
    }
    const Children ch = children(a, q, rt, every, nullptr);
    const int K = ch.n * a.deg;
    const int n = int(min(64LL, a.R - j0));
    auto column = [&](int k) {
        int c, b;
        split_k(k, a, c, b);
        return ch.col[c] + b;
    };
    // line of Z_{k+1}: child, beta, b; from the node's first child on, whose place is in 64
    // bits (children x deg^k stay below 2^31: a level's cells x deg^d do below 2^30)
    const double* in = a.in + ((long long)c0 * a.nbeta + beta) * a.deg * a.R + j0;
    auto line = [&](int k) {
        int c, b;
        split_k(k, a, c, b);
        return (ch.x ? ch.x[c] : c) * a.nbeta * a.deg + b;
    };
    using Map = Mma64Map<64, 16, false>;
    LineOperand<Map, decltype(column)> la(column, a.A + i0, a.M, a.M - i0, K);
    LineOperand<Map, decltype(line)> lb(line, in, a.R, n, K);
    double* out = a.out + (long long)item * a.M * a.R + j0;
    bool bad = false;
    auto st = [&](int i, int j, double v) {
        bad |= !finite(v);
        out[(long long)(i0 + i) * a.R + j] = v;
    };
    mma64_tile<64, 16>(a.M - i0, n, K, la, lb, st, lds);
    if (bad) *a.flag = a.call;
}

__global__ void __launch_bounds__(256) k_zero(double* y, long long n) {
    for (long long v = blockIdx.x * 256ll + threadIdx.x; v < n; v += (long long)gridDim.x * 256) y[v] = 0.0;
}

unsigned grid_for(long long n) { return unsigned(std::min<long long>((n + 255) / 256, 65536)); }

int level_of(int I0) {
    int l = 0;
    while ((1 << l) <= I0) ++l;
    return l;
}

}  // namespace
}  // namespace kmx

using namespace kmx;

struct kmx_realspace {
    int D = 0, deg = 0, N = 0, B = 0;
    int npts[KMX_MAX_DIM] = {0}, ncols[KMX_MAX_DIM] = {0};
    long long nout = 0;
    double* d_meval[KMX_MAX_DIM] = {nullptr};
    // stage k (contracting dimension k): its nodes (prefixes of length k), their
    // children (nodes of stage k + 1; elements in the last) and the children's columns
    struct Stage {
        int nodes = 0;
        size_t cptr = 0, col = 0;            // (places in d_tab)
        size_t lptr = 0, lcol = 0, lx = 0;   // of StageArgs
        bool lists = false;
    };
    Stage stage[KMX_MAX_DIM];
    // every index table in one allocation and copy (3D lev 5 deg 2: the plan 1.17 -> 1.01 ms)
    int* d_tab = nullptr;
    size_t row = 0;   // elements in prefix order
    size_t flag = 0;  // one per stage
    unsigned calls = 0;
    double* d_buf[2] = {nullptr, nullptr};  // Z_d, Z_{d-1}, ... in turn
};

static void free_rs(kmx_realspace* r) {
    for (auto& m : r->d_meval)
        if (m) hipFree(m);
    if (r->d_tab) hipFree(r->d_tab);
    for (auto& b : r->d_buf)
        if (b) hipFree(b);
}

// The lists of StageArgs for dimension k, where they leave out a tenth of the products or
// more: a wavelet of level l is zero on all but 2^(1-l) of its dimension, exactly, so a
// tile of 64 of 192 points meets 0.42 of 64 cells' blocks, of 3072 points 0.036 of 512's.
// Leaving a zero block out leaves every sum's bits as they are.
template <class Put>
static void build_lists(kmx_realspace* r, int k, const double* meval, const std::vector<int>& cptr,
                        const std::vector<int>& col, const std::vector<int>& order, const Put& put) {
    const int M = r->npts[k], deg = r->deg, tiles = (M + 63) / 64, blocks = r->ncols[k] / deg;
    if (tiles < 2 || col.empty()) return;
    std::vector<unsigned char> on(size_t(tiles) * blocks, 0);
    for (int b = 0; b < blocks; ++b)
        for (int t = 0; t < tiles; ++t) {
            // (all bits but the sign, a column's run at once: 67 MB of 1D lev 9 deg 4 in 4.7 ms,
            // 8.7 value by value)
            unsigned long long any = 0;
            for (int c = b * deg; c < (b + 1) * deg && !any; ++c) {
                const double* v = meval + size_t(c) * M;
                for (int i = 64 * t; i < std::min(M, 64 * t + 64); ++i) {
                    unsigned long long bits;
                    std::memcpy(&bits, v + i, sizeof bits);
                    any |= bits << 1;
                }
            }
            on[size_t(t) * blocks + b] = any != 0;
        }
    const int nodes = int(cptr.size()) - 1;
    if (double(col.size()) * tiles > 2e7) return;  // (160 MB of lists at most)
    std::vector<int> ptr, lcol, lx;
    for (int q = 0; q < nodes; ++q)
        for (int t = 0; t < tiles; ++t) {
            ptr.push_back(int(lcol.size()));
            for (int c = cptr[size_t(q)]; c < cptr[size_t(q) + 1]; ++c)
                if (on[size_t(t) * blocks + col[size_t(c)] / deg] ||
                    (c + 1 == cptr[size_t(q) + 1] && int(lcol.size()) == ptr.back())) {  // (no list is empty)
                    lcol.push_back(col[size_t(c)]);
                    lx.push_back(k + 1 == r->D ? order[size_t(c)] : c - cptr[size_t(q)]);
                }
        }
    ptr.push_back(int(lcol.size()));
    if (double(lcol.size()) > 0.9 * double(col.size()) * tiles) return;
    r->stage[k].lists = true;
    r->stage[k].lptr = put(ptr);
    r->stage[k].lcol = put(lcol);
    r->stage[k].lx = put(lx);
}

extern "C" int kmx_realspace_create(int ndim, int deg, int num_elem, const int* elem_idx1d, int index_base,
                                    const int* npts, const int* ncols, const double* const* meval,
                                    kmx_realspace** out) {
    if (!out || ndim < 1 || ndim > KMX_MAX_DIM || deg < 1 || deg > KMX_MAX_DEG || num_elem < 0 || !npts || !ncols ||
        !meval || (num_elem > 0 && !elem_idx1d) || (index_base != 0 && index_base != 1)) {
        set_error("kmx_realspace_create: bad arguments");
        return KMX_E_ARG;
    }
    *out = nullptr;
    auto* r = new kmx_realspace();
    try {
        r->D = ndim;
        r->deg = deg;
        r->N = num_elem;
        r->B = 1;
        r->nout = 1;
        for (int k = 0; k < ndim; ++k) {
            if (npts[k] < 1 || ncols[k] < deg || ncols[k] % deg || !meval[k])
                throw std::invalid_argument("Meval_d must be npts_d x (deg * cells), npts_d >= 1");
            r->B *= deg;
            r->npts[k] = npts[k];
            r->ncols[k] = ncols[k];
            r->nout *= npts[k];
            const size_t sz = size_t(npts[k]) * ncols[k];
            if (hipMalloc(&r->d_meval[k], sz * sizeof(double)) != hipSuccess) throw std::bad_alloc();
            if (hipMemcpy(r->d_meval[k], meval[k], sz * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
                throw std::runtime_error("hipMemcpy failed");
        }
        // element indices; and the limit on a level tuple's values, which the stages' 32-bit
        // places inside a node's list rely on
        std::map<std::vector<int>, long long> lev_cells;
        std::vector<int> idx(size_t(num_elem) * ndim);
        for (int e = 0; e < num_elem; ++e) {
            std::vector<int> lev(ndim);
            for (int k = 0; k < ndim; ++k) {
                const int I0 = elem_idx1d[size_t(e) * ndim + k] - index_base;
                if (I0 < 0 || (I0 + 1) * deg > ncols[k]) throw std::invalid_argument("elem_idx1d out of range");
                idx[size_t(e) * ndim + k] = I0;
                lev[k] = level_of(I0);
            }
            if (lev_cells.count(lev)) continue;
            long long ncell = 1;
            for (int k = 0; k < ndim; ++k) {
                const int c0 = lev[k] == 0 ? 0 : (1 << (lev[k] - 1));
                ncell *= std::min(lev[k] == 0 ? 1 : (1 << (lev[k] - 1)), ncols[k] / deg - c0);
            }
            if (ncell * r->B > (1LL << 30)) throw std::invalid_argument("level block too large");
            lev_cells[lev] = ncell;
        }
        // elements sorted by index tuple; the distinct prefixes of each length
        std::vector<int> order(static_cast<size_t>(num_elem));
        std::iota(order.begin(), order.end(), 0);
        auto ix = [&](int e, int k) { return idx[size_t(e) * ndim + k]; };
        std::sort(order.begin(), order.end(), [&](int a, int b) {
            for (int k = 0; k < ndim; ++k)
                if (ix(a, k) != ix(b, k)) return ix(a, k) < ix(b, k);
            return a < b;
        });
        // first position (in `order`) of every node of depth k: positions where one of
        // the indices 0..k-1 changes
        std::vector<std::vector<int>> first(size_t(ndim) + 1);
        for (int p = 0; p < num_elem; ++p) {
            int diff = p == 0 ? 0 : ndim;  // the first differing dimension
            for (int k = 0; p > 0 && k < ndim; ++k)
                if (ix(order[size_t(p)], k) != ix(order[size_t(p) - 1], k)) {
                    diff = k;
                    break;
                }
            if (p > 0 && diff == ndim) throw std::invalid_argument("two elements share one 1D index tuple");
            for (int k = diff + 1; k <= ndim; ++k) first[size_t(k)].push_back(p);
        }
        if (num_elem > 0) first[0].push_back(0);
        std::vector<int> tab;
        auto put = [&](const std::vector<int>& h) {
            const size_t at = tab.size();
            tab.insert(tab.end(), h.begin(), h.end());
            tab.resize((tab.size() + 31) / 32 * 32, 0);
            return at;
        };
        long long need[2] = {1, 1}, R = 1;
        for (int k = ndim - 1; k >= 0; --k) {
            const std::vector<int>& par = first[size_t(k)];
            const std::vector<int>& chl = first[size_t(k) + 1];
            std::vector<int> cptr, col(chl.size());
            size_t c = 0;
            for (size_t q = 0; q < par.size(); ++q) {
                cptr.push_back(int(c));
                const int end = q + 1 < par.size() ? par[q + 1] : num_elem;
                while (c < chl.size() && chl[c] < end) ++c;
            }
            cptr.push_back(int(c));
            for (size_t q = 0; q < chl.size(); ++q) col[q] = ix(order[size_t(chl[q])], k) * deg;
            r->stage[k].nodes = int(par.size());
            r->stage[k].cptr = put(cptr);
            r->stage[k].col = put(col);
            build_lists(r, k, meval[k], cptr, col, order, put);
            if (k > 0) {  // Z_{k+1} of the comment above (k from 1 there)
                R *= npts[k];
                long long nb = 1;
                for (int q = 0; q < k; ++q) nb *= deg;
                need[(ndim - 1 - k) & 1] = std::max(need[(ndim - 1 - k) & 1], (long long)par.size() * nb * R);
            }
        }
        r->row = put(order);
        r->flag = put(std::vector<int>(size_t(ndim), 0));
        if (hipMalloc(&r->d_tab, tab.size() * sizeof(int)) != hipSuccess) throw std::bad_alloc();
        if (hipMemcpy(r->d_tab, tab.data(), tab.size() * sizeof(int), hipMemcpyHostToDevice) != hipSuccess)
            throw std::runtime_error("hipMemcpy failed");
        for (int q = 0; q < 2; ++q)
            if (hipMalloc(&r->d_buf[q], size_t(need[q]) * sizeof(double)) != hipSuccess) throw std::bad_alloc();
        *out = r;
        return KMX_OK;
    } catch (const std::bad_alloc&) {
        set_error("kmx_realspace_create: device allocation failed");
        free_rs(r);
        delete r;
        return KMX_E_NOMEM;
    } catch (const std::exception& e) {
        set_error(std::string("kmx_realspace_create: ") + e.what());
        free_rs(r);
        delete r;
        return KMX_E_ARG;
    }
}

extern "C" int kmx_realspace_apply(kmx_realspace* r, const double* f_w, double* f_r, void* stream) {
    if (!r || !f_r || (r->N > 0 && !f_w)) {
        set_error("kmx_realspace_apply: bad arguments");
        return KMX_E_ARG;
    }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (r->N == 0) hipLaunchKernelGGL(k_zero, dim3(grid_for(r->nout)), dim3(256), 0, s, f_r, r->nout);
    const int D = r->D;
    const double* cur = f_w;
    long long R = 1;
    if (++r->calls == 0) r->calls = 1;  // never the flag's first value
    const int call = int(r->calls);
    for (int k = D - 1; k >= 0 && r->N > 0; --k) {
        StageArgs a;
        a.in = cur;
        a.out = k == 0 ? f_r : r->d_buf[(D - 1 - k) & 1];
        a.A = r->d_meval[k];
        const kmx_realspace::Stage& st = r->stage[k];
        a.cptr = r->d_tab + st.cptr;
        a.col = r->d_tab + st.col;
        a.row = r->d_tab + r->row;
        a.lptr = st.lists ? r->d_tab + st.lptr : nullptr;
        a.lcol = st.lists ? r->d_tab + st.lcol : nullptr;
        a.lx = st.lists ? r->d_tab + st.lx : nullptr;
        a.ptiles = (r->npts[k] + 63) / 64;
        a.flag = r->d_tab + r->flag + k;
        a.before = k + 1 < D ? a.flag + 1 : nullptr;
        a.call = call;
        a.R = R;
        a.M = r->npts[k];
        a.deg = r->deg;
        a.magic = unsigned((1ULL << 32) / unsigned(r->deg) + 1);
        a.B = r->B;
        a.nbeta = 1;
        for (int q = 0; q < k; ++q) a.nbeta *= r->deg;
        long long grid;
        if (k == D - 1) {
            a.items = r->stage[k].nodes;
            a.mt = (a.nbeta + 15) / 16;
            a.nt = (a.M + 63) / 64;
            a.xcd = 0;
            grid = (long long)a.items * a.mt * a.nt;
        } else {
            const long long items = (long long)r->stage[k].nodes * a.nbeta;
            a.items = int(std::min<long long>(items, 0x7fffffff));
            a.mt = (a.M + 63) / 64;
            const long long nt = (R + 63) / 64;
            if (nt >= (1LL << 30)) {
                set_error("kmx_realspace_apply: too many points");
                return KMX_E_UNSUPPORTED;
            }
            a.nt = int(nt);
            a.xcd = a.mt > 1 && a.nt >= 8 ? 1 : 0;
            grid = items * a.mt * (a.xcd ? (nt + 7) / 8 * 8 : nt);
        }
        if (grid >= (1LL << 31)) {
            set_error("kmx_realspace_apply: too many points");
            return KMX_E_UNSUPPORTED;
        }
        if (k == D - 1) hipLaunchKernelGGL(k_rs_last, dim3(unsigned(grid)), dim3(256), 0, s, a);
        else hipLaunchKernelGGL(k_rs_mode, dim3(unsigned(grid)), dim3(256), 0, s, a);
        R *= r->npts[k];
        cur = a.out;
    }
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        set_error(std::string("kmx_realspace_apply: ") + hipGetErrorString(err));
        return KMX_E_HIP;
    }
    return KMX_OK;
}

extern "C" int kmx_realspace_destroy(kmx_realspace* r) {
    if (!r) return KMX_OK;
    free_rs(r);
    delete r;
    return KMX_OK;
}
