// Batched solve: many independent problems in one persistent launch, one
// workgroup per problem running the whole restarted Halpern PDHG
// loop of reference src/solver.cu:121-169 on the device (evaluation cadence,
// KKT residuals, restarts with the PID primal weight, the BB inner solve,
// affine cones, termination).  The arithmetic follows the single-problem
// solver step for step (reference src/pdhg_core_op.cu); every vector lives in
// HBM in a per-problem slab and every reduction is a fixed-order workgroup
// reduction, so a problem's trajectory does not depend on the rest of the
// batch.  Scalars are held by every thread (each thread computes the same
// value from the same broadcast reductions), so the control flow is uniform.
// The once-per-iteration helpers are not inlined: each gets its own register
// allocation, which keeps the kernel at 248 VGPRs without spills, i.e. two
// waves per SIMD with 512 threads per problem (fully inlined at 256 threads
// it needed 294 registers and ran one problem per CU).
//
// What bounds it: with 256 problems or more running, the matrices and vectors
// of every problem stream through the memory-side cache in every pass, about
// 35 GB/s per compute unit; alone, the chain of dependent passes behind
// barriers.  So as many rows of R as fit stay in LDS for the whole launch, a
// mostly full A is stored dense (one copy without indices), the rest is read in
// 16-byte pieces with eight or more in flight per lane, and an inner body is
// two passes over the columns.  Measured on whole batches of 256 in FP64, start
// of this form against it: portfolios of 50 to 2000 assets 698 -> 352 ms,
// 2000-variable instances with rank 50 and power-law rows 740 -> 465 ms.
//
// Supported per problem: box bounds, rows [A; F], objective of type LP,
// diagonal Q, or dense low rank R'DR (k <= 256) plus a diagonal part, and
// affine cones (SOC / RSOC, exponential, power) on the rows.  Variable cones and off-diagonal sparse Q are handled by the
// single-problem solver only.
#pragma once

#include <cfloat>
#include <type_traits>

#include "dev_common.hpp"
#include "dev_cones.hpp"

namespace pdhcg {
namespace batch {

// Threads per problem: the launch picks 512 (two waves per SIMD at 248
// VGPRs) or 256 by timing (batch.hip); device loops stride by the template
// parameter BT, a compile-time constant.
constexpr int kBT = 512, kBTSmall = 256;
constexpr int kBW = kBT / kWave;  // waves of the largest workgroup (reduction slots)
constexpr int kStaticLds = 1024;  // bound on the kernel's static LDS (reductions)
constexpr int kMaxRank = 256;  // low-rank terms up to this rank (R x and D R x live in LDS)

enum QKind { kQNone = 0, kQDiag = 1, kQLowRank = 2 };

// Loop parameters shared by the batch (pdhg_parameters_t fields).
struct Params {
    int ef, iteration_limit, norm_inf, inner_limit, precond, stall_iters;
    double handover;  // FP32 phase: KKT error below which the FP64 kernel takes over
    double eps_opt, eps_feas, eps_inf, rho;
    double inner_tol0, inner_min_tol;
    double i_smooth, k_p, k_i, k_d, suff, nec, art;
};

// One problem: sizes, pool offsets and scaled-problem scalars.
struct Inst {
    int n, m, k, qkind, dkind, has_affine, ncones, cone0;
    int pn, pm;                    // n and m rounded up to 4: pitch of the slab's vectors and of R's rows
    int cone_lanes;                // lanes per short SOC/RSOC cone (4, 16, 64), 0: one thread
    int nlong;                     // SOC/RSOC cones above kMaxThreadCone slots: the last nlong cones
    int a_rp, a_ci, at_rp, at_ci;  // int-pool offsets of [A;F] and its transpose
    int a_dense;                   // 1: A is stored dense (m x pn row-major at a_v), no CSR and no transpose
    int a_nnz, a_chunk, at_chunk;  // entries of A; int-pool offsets of the products' chunk tables
    long long a_v, at_v;           // value-pool offsets of the matrix values
    long long vec;                 // slab offset of the problem's n- and m-vectors
    long long wvec;                // FP64 slab offset of its per-cone values
    long long rdense, dmat;        // value-pool offsets of R (k x pn row-major, zero padded) and D
    double cbr, ovr, obj_const, obj_norm, bound_norm, step, pw0, nonconvexity;
};

struct Cone {
    int type, start, vdim;
    double alpha;
};

// Per-problem results (the iterates stay in the slab).
struct Out {
    int status, iters, inner;
    double pobj, dobj, abs_pr, abs_du, rel_pr, rel_du, gap, rel_gap;
    double max_pray, max_dray, pray_lin_obj, dray_obj;
};

// Slab layout: n-vectors, then m-vectors (storage type of the kernel); the
// FP64 slab: per-cone values.  (The k-vectors live in LDS.)
enum NVec { vC, vLB, vUB, vVR, vQD, vDH, vX0, vX, vXP, vXR, vATY, vDS, vGR, vDIR, vQX, vDX, vMD, vMI, vLBF, vUBF,
            kNVec };
enum MVec { wG, wCL, wCU, wCLF, wCUF, wCR, wY0, wY, wYP, wYR, wAX, wDY, wPRES, wPSL, wAPR, wAMEM, wAFD, kMVec };
constexpr int kConeVals = 3;  // projection warm start, residual warm start, complementarity

__host__ __device__ inline int padded4(int n) { return (n + 3) & ~3; }
inline long long slab_size(int n, int m) {
    return (long long)kNVec * padded4(n) + (long long)kMVec * padded4(m);
}
inline long long wslab_size(int ncones) { return (long long)kConeVals * ncones; }

// Chunks of kChunk entries in which a product streams its matrix, at least one.
constexpr int kChunk = 4096;
__host__ __device__ inline int chunk_count(int nnz) {
    const int c = (nnz + kChunk - 1) / kChunk;
    return c > 0 ? c : 1;
}

__device__ inline int print_frequency(int it) {
    int step = 10;
    long long thr = 1000;
    while (it >= thr) {
        step *= 10;
        thr *= 10;
    }
    return step;
}

__device__ inline double clampd(double v, double lo, double hi) { return fmax(lo, fmin(v, hi)); }

// Workgroup-wide reductions; every thread receives the result (fixed order).
template <int BT> struct Red {
    double *lds;  // 2 * kBW doubles
    __device__ double sum(double v) const {
        v = wave_total(v);
        const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
        if (lane == 0) lds[w] = v;
        __syncthreads();
        double s = lds[0];
        for (int i = 1; i < BT / kWave; ++i) s += lds[i];
        __syncthreads();
        return s;
    }
    __device__ double max(double v) const {
        for (int off = kWave / 2; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, kWave));
        const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
        if (lane == 0) lds[w] = v;
        __syncthreads();
        double s = lds[0];
        for (int i = 1; i < BT / kWave; ++i) s = fmax(s, lds[i]);
        __syncthreads();
        return s;
    }
    // L2 or max norm of the values f(i), i < count
    template <class F> __device__ double norm(int count, bool inf, F f) const {
        double a = 0.0;
        for (int i = threadIdx.x; i < count; i += BT) {
            const double v = f(i);
            a = inf ? fmax(a, fabs(v)) : a + v * v;
        }
        return inf ? max(a) : sqrt(sum(a));
    }
    template <class F> __device__ double dot(int count, F f) const {
        double a = 0.0;
        for (int i = threadIdx.x; i < count; i += BT) a += f(i);
        return sum(a);
    }
};

// Two adjacent elements in global memory (aligned: every pitch is a multiple
// of four elements).  The address space is named because the pointers come
// from a structure in memory: the compiler would use flat accesses, which
// also wait for LDS.
template <class T> struct Pair {
    typedef T type __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(1))) type global;
    typedef __attribute__((address_space(1))) T scalar;
};
typedef const __attribute__((address_space(1))) int *GlobalInt;
template <class T> __device__ __forceinline__ typename Pair<T>::type load_pair(const T *p) {
    return *(const typename Pair<T>::global *)p;
}
template <class T> __device__ __forceinline__ void store_pair(T *p, T a, T b) {
    typename Pair<T>::type v = {a, b};
    *(typename Pair<T>::global *)p = v;
}

// Dynamic LDS: D R x and R x (kMaxRank doubles each), then elements of the
// storage type: the vector a product is taken of (when it fits), a chunk of a
// sparse product and the first rows of R (Ctx::stage_room, room).
extern __shared__ __align__(16) double batch_lds[];
__device__ __forceinline__ double *lds_u() { return batch_lds; }
__device__ __forceinline__ double *lds_rx() { return batch_lds + kMaxRank; }
template <class T> __device__ __forceinline__ T *lds_room() { return reinterpret_cast<T *>(batch_lds + 2 * kMaxRank); }
template <class T> __device__ __forceinline__ typename Pair<T>::type load_pair_lds(int i) {
    return *reinterpret_cast<const typename Pair<T>::type *>(lds_room<T>() + i);
}
template <class T> __device__ __forceinline__ void store_pair_lds(int i, T a, T b) {
    typename Pair<T>::type v = {a, b};
    *reinterpret_cast<typename Pair<T>::type *>(lds_room<T>() + i) = v;
}

// y = M x for a CSR matrix of `rows` rows and `nnz` entries.  With one
// workgroup per problem and two waves per SIMD there is little occupancy to
// hide memory latency, and a row per lane group is a chain of three dependent
// loads per few rows: 150 us for 1000 power-law rows of 20 entries on average,
// 25 us for 1300 rows of 24.  So the entries are streamed in chunks of kChunk
// whatever the rows: column and value of every entry of the next two chunks are
// in flight while this one's products, in LDS, are summed by row (chunk_row[c]:
// first row that starts in chunk c or later; a row that continues from the
// chunk before is added to).  Rows longer than 32 entries per lane of the
// chunk's groups take the whole wavefront.  x is copied to LDS first when it
// fits (prod_at: its room): a gather from the caches takes the address unit a
// cycle per lane, 4000 a chunk.  Measured in a batch of 256: 1000 power-law
// rows of 20 entries 150 -> 29 us, their transpose 36 -> 21 us.
template <class T, int BT>
__device__ __noinline__ void spmv(const int *rp_, const int *ci_, const T *v_, const int *chunk_row_, const T *x_,
                                  T *y_, int rows, int nnz, int cols, int prod_at) {
    const auto rp = (GlobalInt)rp_, ci = (GlobalInt)ci_, chunk_row = (GlobalInt)chunk_row_;
    const auto v = (const typename Pair<T>::scalar *)v_, x = (const typename Pair<T>::scalar *)x_;
    const auto y = (typename Pair<T>::scalar *)y_;
    constexpr int E = kChunk / BT, W = BT / kWave;
    T *prod = lds_room<T>() + prod_at;
    const T *xs = lds_room<T>();
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int chunks = chunk_count(nnz);
    struct Entries {
        int col[E];
        T val[E];
    } even, odd;
    auto fetch = [&](Entries &b, int c) {
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int e = c * kChunk + tid + q * BT;
            b.col[q] = e < nnz ? ci[e] : -1;
            b.val[q] = e < nnz ? v[e] : T(0);
        }
    };
    // sum of prod[i], i = from, from + step, ... < to, four loads in flight
    auto strided = [&](int from, int to, int step) {
        T acc[4] = {T(0), T(0), T(0), T(0)};
        for (int i = from; i < to; i += 4 * step) {
            T p[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) p[q] = prod[min(i + q * step, kChunk - 1)];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (i + q * step < to) acc[q] += p[q];
        }
        return (acc[0] + acc[1]) + (acc[2] + acc[3]);
    };
    int r0 = 0, r1 = chunk_row[1];
    auto process = [&](Entries &b, int c) {
        T g[E];
#pragma unroll
        for (int q = 0; q < E; ++q) {
            g[q] = T(0);
            if (b.col[q] >= 0) g[q] = prod_at ? xs[b.col[q]] : x[b.col[q]];
        }
#pragma unroll
        for (int q = 0; q < E; ++q)
            if (b.col[q] >= 0) prod[tid + q * BT] = b.val[q] * g[q];
        // lanes per row that starts here, and this group's first row
        const int count = r1 - r0;
        int lanes = kWave;
        while (lanes > 1 && lanes * count > BT) lanes >>= 1;
        const int per = BT / lanes, sub = tid & (lanes - 1), first = r0 + tid / lanes;
        int s = first < r1 ? rp[first] : 0, e = first < r1 ? rp[first + 1] : 0;
        const int next = chunk_row[min(c + 2, chunks)];
        const int cont_end = c > 0 ? rp[r0] : 0;  // end of the row before r0
        if (c + 2 < chunks) fetch(b, c + 2);
        __syncthreads();
        const int base = c * kChunk, top = min(base + kChunk, nnz);
        for (int k0 = r0; k0 < r1; k0 += per) {
            const int r = k0 + tid / lanes;
            if (k0 != r0) {
                s = r < r1 ? rp[r] : 0;
                e = r < r1 ? rp[r + 1] : 0;
            }
            const int end = min(e, top);
            const bool mine = r < r1 && end - s <= 32 * lanes;
            double t = mine ? (double)strided(s - base + sub, end - base, lanes) : 0.0;
            if (lanes >= 2) t += dpp_move<kDppXor1>(t);
            if (lanes >= 4) t += dpp_move<kDppXor2>(t);
            if (lanes >= 8) t += dpp_move<kDppHalfMirror>(t);
            if (lanes >= 16) t += dpp_move<kDppMirror>(t);
            if (lanes >= 32) t = fold16(t, t);
            if (lanes >= 64) t = fold32(t, t);
            if (mine && sub == 0) y[r] = (T)t;
            unsigned long long mask = __ballot(sub == 0 && r < r1 && !mine);
            for (; mask; mask &= mask - 1) {  // long rows: the whole wavefront
                const int src = __ffsll((long long)mask) - 1;
                const int row = __shfl(r, src, kWave), from = __shfl(s, src, kWave) - base;
                const double w = wave_total((double)strided(from + lane, __shfl(end, src, kWave) - base, kWave));
                if (lane == 0) y[row] = (T)w;
            }
        }
        if (cont_end > base && wave == W - 1) {
            const double t = wave_total((double)strided(lane, min(cont_end, top) - base, kWave));
            if (lane == 0) y[r0 - 1] = (T)((double)y[r0 - 1] + t);
        }
        r0 = r1;
        r1 = next;
        __syncthreads();
    };
    fetch(even, 0);
    if (chunks > 1) fetch(odd, 1);
    if (prod_at) {
        for (int p = tid; p < padded4(cols) / 2; p += BT) {
            const auto w = load_pair(x_ + 2 * p);
            store_pair_lds<T>(2 * p, w[0], w[1]);
        }
        __syncthreads();
    }
    for (int c = 0; c < chunks; c += 2) {
        process(even, c);
        if (c + 1 < chunks) process(odd, c + 1);
    }
}

// Everything one problem's loop needs, as device pointers.  T is the
// storage and product type of the iterates and matrix values (double, or
// float for the FP32 phase of the mixed batch); the k-vectors, per-cone
// values, D and every reduction and scalar stay FP64.
template <class T, int BT> struct Ctx {
    const Params *P;
    Inst I;
    const int *arp, *aci, *atrp, *atci, *ach, *atch;
    const T *av, *atv, *R;
    const double *D;
    T *V;       // n- and m-vectors of the slab
    double *W;  // per-cone values (FP64)
    const Cone *cones;
    Red<BT> red;
    // LDS: room for the vector of a product (at 0; 0: not staged), then a chunk
    // of a sparse product, then (offset `room`) the first `resident` rows of
    // R, which are loaded once per launch
    int stage_room, room, resident;
    __device__ T *nv(int which) const { return V + (long long)which * I.pn; }
    __device__ T *mv(int which) const { return V + (long long)kNVec * I.pn + (long long)which * I.pm; }
    __device__ double *cv(int which) const { return W + (long long)which * I.ncones; }
    // Products with A and A'.  A dense A (factor models: a few full rows) is
    // read once per product without indices, by the passes of a dense R.
    __device__ void A(const T *x, T *y) const {
        if (I.a_dense) dense_rows(x, y);
        else spmv<T, BT>(arp, aci, av, ach, x, y, I.m, I.a_nnz, I.n, stage_room);
    }
    __device__ void At(const T *y, T *x) const {
        if (I.a_dense) dense_columns(y, x);
        else spmv<T, BT>(atrp, atci, atv, atch, y, x, I.n, I.a_nnz, I.m, stage_room);
    }
    __device__ __noinline__ void dense_rows(const T *x, T *y) const {
        stage(x);
        __syncthreads();
        auto put = [&](int r, double v) { y[r] = (T)v; };
        if (stage_room) all_rows(av, I.m, 0, [&](int i) { return load_pair_lds<T>(i); }, put);
        else all_rows(av, I.m, 0, [&](int i) { return load_pair(x + i); }, put);
        __syncthreads();
    }
    __device__ __noinline__ void dense_columns(const T *y, T *x) const {
        for (int i = threadIdx.x; i < I.m; i += BT) lds_rx()[i] = (double)y[i];
        __syncthreads();
        for (int p = threadIdx.x; p < I.pn / 2; p += BT) {
            T v[2];
            columns(av, I.m, 0, lds_rx(), p, v);
            store_pair(x + 2 * p, v[0], v[1]);
        }
        __syncthreads();
    }

    // Sums of U rows of R times x over the wave; the lanes take pairs of
    // columns, four per row in flight, in four sums each (in FP32 a sum's length
    // is its error bound).  row(a, i), x(i): the pair at column i.
    template <int U, class Row, class Vec> __device__ __forceinline__ void row_sums(Row row, Vec x, double (&out)[U]) const {
        typedef typename Pair<T>::type P2;
        const int half = I.pn / 2, lane = threadIdx.x % kWave;
        T s[U][4];
#pragma unroll
        for (int a = 0; a < U; ++a) s[a][0] = s[a][1] = s[a][2] = s[a][3] = T(0);
        for (int p = lane; p < half; p += 4 * kWave) {
            P2 v[U][4], xv[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bool in = p + q * kWave < half;
                xv[q] = P2(T(0));
                if (in) xv[q] = x(2 * (p + q * kWave));
#pragma unroll
                for (int a = 0; a < U; ++a) {
                    v[a][q] = P2(T(0));
                    if (in) v[a][q] = row(a, 2 * (p + q * kWave));
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int a = 0; a < U; ++a) {
                    s[a][2 * (q & 1)] += v[a][q][0] * xv[q][0];
                    s[a][2 * (q & 1) + 1] += v[a][q][1] * xv[q][1];
                }
        }
#pragma unroll
        for (int a = 0; a < U; ++a)
            out[a] = wave_total(((double)s[a][0] + (double)s[a][1]) + ((double)s[a][2] + (double)s[a][3]));
    }
    // put(r, row r of M times x) in lane 0, for the rows [0, k) of a dense
    // k x pn M whose first `res` rows are the resident ones in LDS; x(i) as in
    // row_sums (staged x: written before a barrier).
    template <class Vec, class Put>
    __device__ __forceinline__ void all_rows(const T *M, int k, int res, Vec x, Put put) const {
        constexpr int W = BT / kWave;
        const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
        for (int r = res + wave; r < k; r += 2 * W) {
            const T *r0 = M + (long long)r * I.pn, *r1 = r0 + (long long)W * I.pn;
            if (r + W < k) {
                double v[2];
                row_sums<2>([&](int a, int i) { return load_pair((a ? r1 : r0) + i); }, x, v);
                if (lane == 0) {
                    put(r, v[0]);
                    put(r + W, v[1]);
                }
            } else {
                double v[1];
                row_sums<1>([&](int, int i) { return load_pair(r0 + i); }, x, v);
                if (lane == 0) put(r, v[0]);
            }
        }
        for (int r = wave; r < res; r += W) {
            const int r0 = room + r * I.pn;
            double v[1];
            row_sums<1>([&](int, int i) { return load_pair_lds<T>(r0 + i); }, x, v);
            if (lane == 0) put(r, v[0]);
        }
    }
    // u = D R x (in LDS); ends with a barrier.
    template <class Vec> __device__ __forceinline__ void low_rank_rows(Vec x) const {
        const int k = I.k;
        all_rows(R, k, resident, x, [&](int r, double v) {
            if (I.dkind == 2) lds_rx()[r] = v;
            else lds_u()[r] = I.dkind == 1 ? v * D[r] : v;
        });
        __syncthreads();
        if (I.dkind == 2) {  // the symmetric part of a dense D from its upper triangle (reference src/pdhg_core_op.cu:272-303)
            for (int i = threadIdx.x; i < k; i += BT) {
                double a = 0.0;
                for (int j = 0; j < k; ++j) {
                    const int lo = i < j ? i : j, hi = i < j ? j : i;
                    a += D[(long long)lo * k + hi] * lds_rx()[j];
                }
                lds_u()[i] = a;
            }
            __syncthreads();
        }
    }
    __device__ __forceinline__ void low_rank_u(const T *x) const {
        if (stage_room) low_rank_rows([&](int i) { return load_pair_lds<T>(i); });
        else low_rank_rows([&](int i) { return load_pair(x + i); });
    }
    // Columns 2 p and 2 p + 1 of R'u.
    __device__ __forceinline__ void low_rank_columns(int p, T (&out)[2]) const {
        columns(R, I.k, resident, lds_u(), p, out);
    }
    // Columns 2 p and 2 p + 1 of M'u for the M of all_rows and u in LDS, each in
    // four sums.  The first eight rows outside LDS are in flight while the
    // resident ones are added.
    __device__ __forceinline__ void columns(const T *M, int k, int resident, const double *u, int p, T (&out)[2]) const {
        typedef typename Pair<T>::type P2;
        constexpr int U = 8;
        const int pn = I.pn, lcol = room + 2 * p;
        const T *col = M + 2 * p;
        T s[4][2] = {};
        int r = resident;
        P2 g[U];
#pragma unroll
        for (int a = 0; a < U; ++a) {
            g[a] = P2(T(0));
            if (r + a < k) g[a] = load_pair(col + (long long)(r + a) * pn);
        }
        for (int j = 0; j < resident; j += 4) {
            P2 v[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                v[a] = P2(T(0));
                if (j + a < resident) v[a] = load_pair_lds<T>(lcol + (j + a) * pn);
            }
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const T uj = j + a < resident ? (T)u[j + a] : T(0);
                s[a][0] += v[a][0] * uj;
                s[a][1] += v[a][1] * uj;
            }
        }
        while (r < k) {
            P2 nx[U];
#pragma unroll
            for (int a = 0; a < U; ++a) {
                nx[a] = P2(T(0));
                if (r + U + a < k) nx[a] = load_pair(col + (long long)(r + U + a) * pn);
            }
#pragma unroll
            for (int a = 0; a < U; ++a) {
                const T uj = r + a < k ? (T)u[r + a] : T(0);
                s[a % 4][0] += g[a][0] * uj;
                s[a % 4][1] += g[a][1] * uj;
            }
#pragma unroll
            for (int a = 0; a < U; ++a) g[a] = nx[a];
            r += U;
        }
        out[0] = (s[0][0] + s[1][0]) + (s[2][0] + s[3][0]);
        out[1] = (s[0][1] + s[1][1]) + (s[2][1] + s[3][1]);
    }
    // Copies x into LDS (when the product's vector is staged); a barrier must follow.
    __device__ __forceinline__ void stage(const T *x) const {
        if (!stage_room) return;
        for (int p = threadIdx.x; p < I.pn / 2; p += BT) {
            const auto v = load_pair(x + 2 * p);
            store_pair_lds<T>(2 * p, v[0], v[1]);
        }
    }

    // qx = Q x (reference src/pdhg_core_op.cu:305-413): diagonal part plus R'DR x
    __device__ __noinline__ void obj_product(const T *x, T *qx) const {
        const int n = I.n;
        if (I.qkind == kQNone) return;
        const T *qd = nv(vQD);
        if (I.qkind == kQDiag) {
            for (int i = threadIdx.x; i < n; i += BT) qx[i] = qd[i] * x[i];
            __syncthreads();
            return;
        }
        stage(x);
        __syncthreads();
        low_rank_u(x);
        for (int p = threadIdx.x; p < I.pn / 2; p += BT) {
            T v[2];
            low_rank_columns(p, v);
            const auto q2 = load_pair(qd + 2 * p), x2 = load_pair(x + 2 * p);
            store_pair(qx + 2 * p, q2[0] * x2[0] + v[0], q2[1] * x2[1] + v[1]);
        }
        __syncthreads();
    }

    // Second-order cones among the first nshort, L lanes per cone.
    template <int L> __device__ void soc_groups(T *v, const T *d, double *warm, int nshort) const {
        const int lane = threadIdx.x % L;
        for (int c0 = 0; c0 < nshort; c0 += BT / L) {
            const int c = c0 + (int)threadIdx.x / L;
            Cone cn{CONE_EXPONENTIAL, 0, 0, 0.0};
            if (c < nshort) cn = cones[c];
            const bool live = cn.type == CONE_STANDARD_SOC || cn.type == CONE_ROTATED_SOC;
            const int s = cn.start, k = cn.vdim;
            const bool has = live && lane < k;
            double p = has ? (double)v[s + lane] : 0.0, e = has ? (double)d[s + lane] : 1.0;
            double a = live ? (double)v[s + k] : 0.0, b = live ? (double)v[s + k + 1] : 0.0;
            const double ea = live ? (double)d[s + k] : 1.0, eb = live ? (double)d[s + k + 1] : 1.0;
            soc_project_group<L>(live, p, e, lane, k, a, b, ea, eb, cn.type == CONE_ROTATED_SOC, warm + (live ? c : 0));
            if (has) v[s + lane] = (T)p;
            if (live && lane == 0) {
                v[s + k] = (T)a;
                v[s + k + 1] = (T)b;
            }
        }
    }

    // Projection of the m-vector v onto the affine cones, scaling affd
    // (reference src/cone_dispatch.cu:38-57 on the row space).  Second-order
    // cones take I.cone_lanes lanes each (soc_project_group): with one thread
    // per cone a portfolio's pass took about 30 us more, in the bisection of
    // its one cone of 12 to 52 slots (256 portfolios: 783 -> 698 ms).  With more cones than eight rounds of the workgroup's groups hold
    // (cone_lanes 0) a thread per cone is the faster form.
    __device__ __noinline__ void project_affine(T *v, double *warm) const {
        const T *d = mv(wAFD);
        const int nshort = I.ncones - I.nlong;
        if (I.cone_lanes == 4) soc_groups<4>(v, d, warm, nshort);
        else if (I.cone_lanes == 16) soc_groups<16>(v, d, warm, nshort);
        else if (I.cone_lanes == 64) soc_groups<64>(v, d, warm, nshort);
        for (int c = threadIdx.x; c < nshort; c += BT) {
            const Cone cn = cones[c];
            const int s = cn.start;
            if (cn.type == CONE_STANDARD_SOC || cn.type == CONE_ROTATED_SOC) {
                if (I.cone_lanes) continue;
                double pv[kMaxThreadCone + 2];
                for (int q = 0; q < cn.vdim + 2; ++q) pv[q] = v[s + q];
                if constexpr (std::is_same<T, double>::value) {
                    soc_project_block(pv, cn.vdim, d + s, cn.type == CONE_ROTATED_SOC, warm + c);
                } else {
                    double pd[kMaxThreadCone + 2];
                    for (int q = 0; q < cn.vdim + 2; ++q) pd[q] = d[s + q];
                    soc_project_block(pv, cn.vdim, pd, cn.type == CONE_ROTATED_SOC, warm + c);
                }
                for (int q = 0; q < cn.vdim + 2; ++q) v[s + q] = (T)pv[q];
            } else if (cn.type == CONE_EXPONENTIAL) {
                double o[3];
                exp_project_point(v[s], v[s + 1], v[s + 2], d[s], d[s + 1], d[s + 2], o);
                v[s] = (T)o[0];
                v[s + 1] = (T)o[1];
                v[s + 2] = (T)o[2];
            } else {
                double o[3];
                const double d0 = d[s], d1 = d[s + 1], d2 = d[s + 2];
                power_project_point(v[s] / d0, v[s + 1] / d1, v[s + 2] / d2, d0 * d0, d1 * d1, d2 * d2, cn.alpha, o);
                v[s] = (T)(o[0] * d0);
                v[s + 1] = (T)(o[1] * d1);
                v[s + 2] = (T)(o[2] * d2);
            }
        }
        __syncthreads();
        // long second-order cones: the whole workgroup on one cone at a time
        for (int c = nshort; c < I.ncones; ++c) {
            const Cone cn = cones[c];
            T *pv = v + cn.start;
            const T *pd = d + cn.start;
            auto P = [&](int m) { return (double)pv[m]; };
            auto E = [&](int m) { return (double)pd[m]; };
            auto Set = [&](int m, double val) { pv[m] = (T)val; };
            auto sum = [&](double x) { return red.sum(x); };
            if (cn.type == CONE_ROTATED_SOC) soc_project_coop<true>(P, E, Set, cn.vdim, warm + c, sum, false);
            else soc_project_coop<false>(P, E, Set, cn.vdim, warm + c, sum, false);
            __syncthreads();
        }
    }
};

// A problem that leaves the FP32 phase of the mixed batch before
// terminating (its iterates stopped improving at the FP32 rounding floor).
constexpr int kStalled = 100;
constexpr int kSatStall = 1;  // FP32 inner solves at the inner limit before the hand-over

// Loop state (identical in every thread).  best_err / best_iter track the
// KKT error of the FP32 phase (a problem whose error has not halved for
// max(1000, half its iterations) leaves that phase as kStalled), sat the
// FP32 inner solves in a row that reached the inner iteration limit, and
// eval_now asks for a KKT evaluation at the next pass.
struct State {
    int total, inner_count, inner_total, is_major, do_restart, reason, best_iter, sat, eval_now, pad;
    double best_err;
    double pw, pw_err_sum, pw_last_err, best_pw, best_gap;
    double fpe, init_fpe, last_trial_fpe, inner_tol, cached_inv_tau, tol_scale;
    double abs_pr, abs_du, rel_pr, rel_du, pobj, dobj, gap, rel_gap;
    double max_pray, max_dray, pray_lin_obj, dray_obj;
};

// Projected BB inner solve of the primal prox (reference
// src/pdhg_core_op.cu:495-669).  A thread owns the column pairs tid, tid + BT,
// ... of every vector throughout, so that a body is two passes: the gradient
// step with R'u and the curvature, and the step itself with its norm (and the
// new x_p staged).  Padding columns are zero in R and in every vector, with
// bounds 0, and stay zero.
template <class T, int BT> __device__ __noinline__ void bb_prox(const Ctx<T, BT> &C, State &S, double tau) {
    const Params &P = *C.P;
    const int n = C.I.n, half = C.I.pn / 2;
    T *x = C.nv(vX), *xp = C.nv(vXP), *xr = C.nv(vXR), *grad = C.nv(vGR), *dirn = C.nv(vDIR), *md = C.nv(vMD),
      *mi = C.nv(vMI);
    const T *c = C.nv(vC), *lb = C.nv(vLB), *ub = C.nv(vUB), *aty = C.nv(vATY), *dh = C.nv(vDH), *qd = C.nv(vQD);
    const double inv = 1.0 / tau;
    double a0 = 1.0 / inv;
    const bool pre = P.precond != 0;
    if (pre && S.cached_inv_tau != inv) {
        double sacc = 0.0;
        for (int p = threadIdx.x; p < half; p += BT)
            for (int i = 2 * p; i < 2 * p + 2 && i < n; ++i) {
                double mm = dh[i] + inv;
                if (mm <= 0.0) mm = 1.0;
                md[i] = mm;
                mi[i] = 1.0 / mm;
                sacc += fabs(mm);
            }
        const double sum = C.red.sum(sacc);
        S.cached_inv_tau = inv;
        S.tol_scale = n > 0 ? sqrt(sum / (double)n) : 1.0;
    }
    if (pre) a0 *= S.tol_scale * S.tol_scale;
    // The step from `from` (x or x_p) along -scale [M^-1] g for pair p; returns its term of |s|^2 or s'Ms.
    auto step = [&](int p, const T *from, double scale, double g0, double g1) {
        const auto f2 = load_pair(from + 2 * p), l2 = load_pair(lb + 2 * p), u2 = load_pair(ub + 2 * p);
        double w0 = 1.0, w1 = 1.0, m0 = 1.0, m1 = 1.0;
        if (pre) {
            const auto i2 = load_pair(mi + 2 * p), d2 = load_pair(md + 2 * p);
            w0 = i2[0];
            w1 = i2[1];
            m0 = d2[0];
            m1 = d2[1];
        }
        const T n0 = (T)clampd(f2[0] - scale * w0 * g0, l2[0], u2[0]);
        const T n1 = (T)clampd(f2[1] - scale * w1 * g1, l2[1], u2[1]);
        const T d0 = n0 - f2[0], d1 = n1 - f2[1];
        store_pair(xp + 2 * p, n0, n1);
        store_pair(dirn + 2 * p, d0, d1);
        if (C.stage_room) store_pair_lds<T>(2 * p, n0, n1);
        const double s0 = (double)d0 * (m0 * (double)d0), s1 = (double)d1 * (m1 * (double)d1);
        return s0 + (2 * p + 1 < n ? s1 : 0.0);
    };
    C.stage(x);
    __syncthreads();
    C.low_rank_u(x);
    double nacc = 0.0;
    for (int p = threadIdx.x; p < half; p += BT) {
        const auto c2 = load_pair(c + 2 * p), a2 = load_pair(aty + 2 * p), q2 = load_pair(qd + 2 * p),
                   x2 = load_pair(x + 2 * p);
        T v[2];
        C.low_rank_columns(p, v);
        const T qx0 = q2[0] * x2[0] + v[0], qx1 = q2[1] * x2[1] + v[1];
        const double g0 = (double)qx0 + (double)c2[0] - (double)a2[0], g1 = (double)qx1 + (double)c2[1] - (double)a2[1];
        store_pair(grad + 2 * p, (T)g0, (T)g1);
        nacc += step(p, x, a0, g0, g1);
    }
    int it = 1;
    while (it < P.inner_limit) {
        const double s2 = C.red.sum(nacc), nrm = sqrt(s2);
        if (nrm <= S.inner_tol) break;
        C.low_rank_u(xp);
        double tacc = 0.0;
        for (int p = threadIdx.x; p < half; p += BT) {
            const auto c2 = load_pair(c + 2 * p), a2 = load_pair(aty + 2 * p), q2 = load_pair(qd + 2 * p),
                       x2 = load_pair(x + 2 * p), p2 = load_pair(xp + 2 * p), g2 = load_pair(grad + 2 * p),
                       d2 = load_pair(dirn + 2 * p);
            T v[2];
            C.low_rank_columns(p, v);
            const T qx0 = q2[0] * p2[0] + v[0], qx1 = q2[1] * p2[1] + v[1];
            const double cur0 = (double)qx0 + (double)c2[0] - (double)a2[0] + inv * ((double)p2[0] - (double)x2[0]);
            const double cur1 = (double)qx1 + (double)c2[1] - (double)a2[1] + inv * ((double)p2[1] - (double)x2[1]);
            store_pair(grad + 2 * p, (T)cur0, (T)cur1);
            tacc += (double)d2[0] * (double)(T)(cur0 - (double)g2[0]);
            if (2 * p + 1 < n) tacc += (double)d2[1] * (double)(T)(cur1 - (double)g2[1]);
        }
        const double tmp = C.red.sum(tacc);
        const double alpha = pre ? s2 / tmp : (nrm * nrm) / tmp;
        nacc = 0.0;
        for (int p = threadIdx.x; p < half; p += BT) {
            const auto g2 = load_pair(grad + 2 * p);
            nacc += step(p, xp, alpha, (double)g2[0], (double)g2[1]);
        }
        it++;
    }
    for (int p = threadIdx.x; p < half; p += BT) {
        const auto p2 = load_pair(xp + 2 * p), x2 = load_pair(x + 2 * p);
        store_pair(xr + 2 * p, (T)(2.0 * (double)p2[0] - (double)x2[0]), (T)(2.0 * (double)p2[1] - (double)x2[1]));
    }
    __syncthreads();
    S.inner_total += it - 1;
    if (!std::is_same<T, double>::value) S.sat = (P.inner_limit > 1 && it >= P.inner_limit) ? S.sat + 1 : 0;
}

// One PDHG step (reference src/pdhg_core_op.cu:705-830).
template <class T, int BT> __device__ __noinline__ void pdhg_step(const Ctx<T, BT> &C, State &S) {
    const Inst &I = C.I;
    const int n = I.n, m = I.m;
    double tau = I.step / S.pw;
    if (I.nonconvexity < 0) {
        tau = fmax(tau, -1.01 * fmin(0.0, I.nonconvexity));
        tau /= 100;
    }
    const double sigma = I.step * S.pw;
    T *x = C.nv(vX), *xp = C.nv(vXP), *xr = C.nv(vXR), *aty = C.nv(vATY), *ds = C.nv(vDS);
    const T *c = C.nv(vC), *lb = C.nv(vLB), *ub = C.nv(vUB), *qd = C.nv(vQD);
    C.At(C.mv(wY), aty);
    const int tc = S.total;
    const bool store = S.is_major || ((tc + 2) % print_frequency(tc + 2)) == 0;
    if (I.qkind == kQNone) {
        for (int i = threadIdx.x; i < n; i += BT) {
            const double xi = x[i];
            const double t = xi - tau * (c[i] - aty[i]);
            const double pj = clampd(t, lb[i], ub[i]);
            xr[i] = 2.0 * pj - xi;
            if (store) {
                xp[i] = pj;
                ds[i] = (pj - t) / tau;
            }
        }
        __syncthreads();
    } else if (I.qkind == kQDiag) {
        for (int i = threadIdx.x; i < n; i += BT) {
            const double xi = x[i];
            const double t = (xi - tau * (c[i] - aty[i])) / (1.0 + tau * qd[i]);
            const double pj = clampd(t, lb[i], ub[i]);
            xr[i] = 2.0 * pj - xi;
            if (store) xp[i] = pj;
        }
        __syncthreads();
    } else {
        bb_prox(C, S, tau);
    }
    S.inner_total++;
    T *ax = C.mv(wAX), *y = C.mv(wY), *yp = C.mv(wYP), *yr = C.mv(wYR), *apr = C.mv(wAPR);
    const T *g = C.mv(wG), *cl = C.mv(wCL), *cu = C.mv(wCU);
    C.A(xr, ax);
    if (m == 0) return;
    if (I.has_affine) {  // reference src/pdhg_core_op.cu:809-829
        for (int i = threadIdx.x; i < m; i += BT) apr[i] = clampd(ax[i] + g[i] - y[i] / sigma, cl[i], cu[i]);
        __syncthreads();
        C.project_affine(apr, C.cv(0));
    }
    for (int i = threadIdx.x; i < m; i += BT) {
        const double cur = y[i];
        const double v = ax[i] + g[i];
        const double pj = I.has_affine ? apr[i] : clampd(v - cur / sigma, cl[i], cu[i]);
        const double nx = cur - sigma * v + sigma * pj;
        if (store) yp[i] = nx;
        yr[i] = 2.0 * nx - cur;
    }
    __syncthreads();
}

// reference src/pdhg_core_op.cu:832-845
template <class T, int BT> __device__ inline void halpern(const Ctx<T, BT> &C, const State &S) {
    const double rho = C.P->rho;
    const double wgt = (double)(S.inner_count + 1) / (S.inner_count + 2);
    T *x = C.nv(vX), *y = C.mv(wY);
    const T *xr = C.nv(vXR), *x0 = C.nv(vX0), *yr = C.mv(wYR), *y0 = C.mv(wY0);
    for (int i = threadIdx.x; i < C.I.n; i += BT) {
        const double r = rho * xr[i] + (1.0 - rho) * x[i];
        x[i] = wgt * r + (1.0 - wgt) * x0[i];
    }
    for (int i = threadIdx.x; i < C.I.m; i += BT) {
        const double r = rho * yr[i] + (1.0 - rho) * y[i];
        y[i] = wgt * r + (1.0 - wgt) * y0[i];
    }
    __syncthreads();
}

// reference src/pdhg_core_op.cu:973-1035
template <class T, int BT> __device__ __noinline__ void fixed_point_error(const Ctx<T, BT> &C, State &S) {
    const int n = C.I.n, m = C.I.m;
    T *dx = C.nv(vDX), *dy = C.mv(wDY), *aty = C.nv(vATY);
    const T *xr = C.nv(vXR), *x = C.nv(vX), *yr = C.mv(wYR), *y = C.mv(wY);
    for (int i = threadIdx.x; i < n; i += BT) dx[i] = xr[i] - x[i];
    for (int i = threadIdx.x; i < m; i += BT) dy[i] = yr[i] - y[i];
    __syncthreads();
    C.At(dy, aty);
    const double dn = sqrt(C.red.dot(m, [&](int i) { return dy[i] * dy[i]; }));
    const double pn = sqrt(C.red.dot(n, [&](int i) { return dx[i] * dx[i]; }));
    const double mov = pn * pn * S.pw + dn * dn / S.pw;
    const double cross = C.red.dot(n, [&](int i) { return aty[i] * dx[i]; });
    S.fpe = sqrt(mov + 2 * C.I.step * cross);
    if (C.I.qkind == kQLowRank)
        S.inner_tol = fmin(S.inner_tol, fmax(0.0005 * pn / C.I.step * S.pw, C.P->inner_min_tol));
}

// reference src/pdhg_core_op.cu:859-931
template <class T, int BT> __device__ __noinline__ void restart(const Ctx<T, BT> &C, State &S) {
    const Params &P = *C.P;
    const int n = C.I.n, m = C.I.m;
    T *x0 = C.nv(vX0), *x = C.nv(vX), *y0 = C.mv(wY0), *y = C.mv(wY);
    const T *xp = C.nv(vXP), *yp = C.mv(wYP);
    const double pd = sqrt(C.red.dot(n, [&](int i) { return (xp[i] - x0[i]) * (xp[i] - x0[i]); }));
    const double dd = sqrt(C.red.dot(m, [&](int i) { return (yp[i] - y0[i]) * (yp[i] - y0[i]); }));
    const double ratio = S.rel_du / S.rel_pr;
    if (pd > 1e-16 && dd > 1e-16 && pd < 1e12 && dd < 1e12 && ratio > 1e-8 && ratio < 1e8) {
        const double err = log(dd) - log(pd) - log(S.pw);
        S.pw_err_sum *= P.i_smooth;
        S.pw_err_sum += err;
        const double derr = err - S.pw_last_err;
        S.pw *= exp(P.k_p * err + P.k_i * S.pw_err_sum + P.k_d * derr);
        S.pw_last_err = err;
    } else {
        S.pw = S.best_pw;
        S.pw_err_sum = 0.0;
        S.pw_last_err = 0.0;
    }
    const double gapv = fabs(log10(S.rel_du / S.rel_pr));
    if (gapv < S.best_gap) {
        S.best_gap = gapv;
        S.best_pw = S.pw;
    }
    for (int i = threadIdx.x; i < n; i += BT) x0[i] = x[i] = xp[i];
    for (int i = threadIdx.x; i < m; i += BT) y0[i] = y[i] = yp[i];
    __syncthreads();
    S.inner_count = 0;
    S.last_trial_fpe = INFINITY;
}

// reference src/utils.cu:291-322
template <class T, int BT> __device__ inline bool should_restart(const Ctx<T, BT> &C, State &S) {
    const Params &P = *C.P;
    bool r = false;
    if (S.total == P.ef) r = true;
    else if (S.total > P.ef) {
        if (S.fpe <= P.suff * S.init_fpe) r = true;
        if (S.fpe <= P.nec * S.init_fpe && S.fpe > S.last_trial_fpe) r = true;
        if (S.inner_count >= P.art * S.total) r = true;
    }
    S.last_trial_fpe = S.fpe;
    return r;
}

// KKT residuals (reference src/pdhg_core_op.cu:1037-1294).
template <class T, int BT> __device__ __noinline__ void residual(const Ctx<T, BT> &C, State &S) {
    const Inst &I = C.I;
    const int n = I.n, m = I.m;
    const bool linf = C.P->norm_inf != 0;
    const double tau = I.step / S.pw;
    T *ax = C.mv(wAX), *aty = C.nv(vATY), *qx = C.nv(vQX), *ds = C.nv(vDS), *pres = C.mv(wPRES),
           *psl = C.mv(wPSL), *amem = C.mv(wAMEM);
    const T *xp = C.nv(vXP), *yp = C.mv(wYP), *g = C.mv(wG), *cl = C.mv(wCL), *cu = C.mv(wCU),
                 *clf = C.mv(wCLF), *cuf = C.mv(wCUF), *cr = C.mv(wCR), *c = C.nv(vC), *lb = C.nv(vLB),
                 *ub = C.nv(vUB), *vr = C.nv(vVR), *afd = C.mv(wAFD);
    C.A(xp, ax);
    C.At(yp, aty);
    C.obj_product(xp, qx);
    for (int i = threadIdx.x; i < m; i += BT) {
        const double v = ax[i] + g[i];
        const double pj = clampd(v, cl[i], cu[i]);
        pres[i] = (v - pj) * cr[i];
        psl[i] = fmax(yp[i], 0.0) * clf[i] + fmin(yp[i], 0.0) * cuf[i] - g[i] * yp[i];
    }
    const bool lp = I.qkind == kQNone;
    double dres_acc = 0.0;
    for (int j = threadIdx.x; j < n; j += BT) {
        double dres;
        if (lp) {
            dres = (c[j] - aty[j] - ds[j]) * vr[j];
        } else {
            const double gr = qx[j] + c[j] - aty[j];
            const double t = xp[j] - tau * gr;
            const double pj = fmax(lb[j], fmin(ub[j], t));
            const double dsj = (pj - t) / tau;
            dres = (gr - dsj) * vr[j];
            ds[j] = dsj;
        }
        dres_acc = linf ? fmax(dres_acc, fabs(dres)) : dres_acc + dres * dres;
    }
    __syncthreads();
    double abs_du = linf ? C.red.max(dres_acc) : sqrt(C.red.sum(dres_acc));
    double amem_norm = 0.0, acomp_norm = 0.0;
    if (I.has_affine) {  // reference src/pdhg_core_op.cu:1125-1129,114-201
        double *acomp = C.cv(2);
        for (int i = threadIdx.x; i < m; i += BT) {
            pres[i] = clampd(ax[i] + g[i], cl[i], cu[i]);
            amem[i] = 0.0;
        }
        __syncthreads();
        C.project_affine(pres, C.cv(1));
        for (int k = threadIdx.x; k < I.ncones; k += BT) {
            const Cone cn = C.cones[k];
            const int L = (cn.type == CONE_STANDARD_SOC || cn.type == CONE_ROTATED_SOC) ? cn.vdim + 2 : 3;
            double dotv = 0.0;
            for (int i = cn.start; i < cn.start + L; ++i) {
                amem[i] = -yp[i];
                dotv += yp[i] * (ax[i] + g[i]);
            }
            acomp[k] = fabs(dotv) / I.cbr;
        }
        __syncthreads();
        C.project_affine(amem, C.cv(1));
        for (int i = threadIdx.x; i < m; i += BT) {
            pres[i] = (ax[i] + g[i] - pres[i]) * cr[i];
            amem[i] *= afd[i];
        }
        __syncthreads();
        amem_norm = C.red.norm(m, linf, [&](int i) { return amem[i]; });
        acomp_norm = C.red.norm(I.ncones, linf, [&](int i) { return acomp[i]; });
    }
    S.abs_pr = C.red.norm(m, linf, [&](int i) { return pres[i]; }) / I.cbr;
    const double lin_pr = S.abs_pr;
    if (I.has_affine)
        abs_du = linf ? fmax(fmax(abs_du, amem_norm), acomp_norm)
                      : sqrt(abs_du * abs_du + amem_norm * amem_norm + acomp_norm * acomp_norm);
    S.abs_du = abs_du / I.ovr;
    const double half_xqx = lp ? 0.0 : 0.5 * C.red.dot(n, [&](int j) { return xp[j] * qx[j]; });
    S.pobj = (C.red.dot(n, [&](int j) { return c[j] * xp[j]; }) + half_xqx) / (I.cbr * I.ovr) + I.obj_const;
    const double base = C.red.dot(n, [&](int j) { return ds[j] * xp[j]; });
    const double sps = C.red.dot(m, [&](int i) { return psl[i]; });
    S.dobj = (base + sps - half_xqx) / (I.cbr * I.ovr) + I.obj_const;
    S.rel_pr = lin_pr / (1.0 + I.bound_norm);
    double den;
    if (lp) den = 1.0 + I.obj_norm;
    else {
        const double qn = C.red.norm(n, linf, [&](int j) { return qx[j] * vr[j]; });
        const double an = C.red.norm(n, linf, [&](int j) { return aty[j] * vr[j]; });
        den = 1.0 + fmax(I.obj_norm, fmax(qn / I.ovr, an / I.ovr));
    }
    S.rel_du = S.abs_du / den;
    S.gap = fabs(S.pobj - S.dobj);
    S.rel_gap = S.gap / (1.0 + fabs(S.pobj) + fabs(S.dobj));
}

// Infeasibility rays (reference src/pdhg_core_op.cu:1296-1429).
template <class T, int BT> __device__ __noinline__ void infeasibility(const Ctx<T, BT> &C, State &S) {
    const Inst &I = C.I;
    const int n = I.n, m = I.m;
    T *dx = C.nv(vDX), *dy = C.mv(wDY), *ax = C.mv(wAX), *aty = C.nv(vATY), *qx = C.nv(vQX);
    const T *lb = C.nv(vLB), *ub = C.nv(vUB), *cl = C.mv(wCL), *cu = C.mv(wCU), *c = C.nv(vC),
                 *clf = C.mv(wCLF), *cuf = C.mv(wCUF), *g = C.mv(wG), *lbf = C.nv(vLBF), *ubf = C.nv(vUBF),
                 *cr = C.mv(wCR), *vr = C.nv(vVR);
    for (int j = threadIdx.x; j < n; j += BT) {
        if (isfinite(lb[j])) dx[j] = fmax(dx[j], 0.0);
        if (isfinite(ub[j])) dx[j] = fmin(dx[j], 0.0);
    }
    for (int i = threadIdx.x; i < m; i += BT) {
        if (!isfinite(cl[i])) dy[i] = fmin(dy[i], 0.0);
        if (!isfinite(cu[i])) dy[i] = fmax(dy[i], 0.0);
    }
    __syncthreads();
    const double prn = C.red.norm(n, true, [&](int j) { return dx[j]; });
    if (prn > 0.0) {
        const double sc = 1.0 / prn;
        for (int j = threadIdx.x; j < n; j += BT) dx[j] *= sc;
        __syncthreads();
    }
    const double drn = C.red.norm(m, true, [&](int i) { return dy[i]; });
    C.A(dx, ax);
    C.At(dy, aty);
    S.pray_lin_obj = C.red.dot(n, [&](int j) { return c[j] * dx[j]; }) / (I.cbr * I.ovr);
    const double sps = C.red.dot(m, [&](int i) {
        return fmax(dy[i], 0.0) * clf[i] + fmin(dy[i], 0.0) * cuf[i] - g[i] * dy[i];
    });
    const double sds = C.red.dot(n, [&](int j) { return fmax(-aty[j], 0.0) * lbf[j] + fmin(-aty[j], 0.0) * ubf[j]; });
    S.dray_obj = (sps + sds) / (I.cbr * I.ovr);
    S.max_pray = C.red.norm(m, true, [&](int i) {
        const double pv = ax[i];
        return (fmax(0.0, -pv) * (double)isfinite(cl[i]) + fmax(0.0, pv) * (double)isfinite(cu[i])) * cr[i];
    });
    if (I.qkind != kQNone) {
        C.obj_product(dx, qx);
        const double qn = C.red.norm(n, true, [&](int j) { return qx[j]; });
        S.max_pray = fmax(S.max_pray, qn / I.ovr);
    }
    const double dsn = C.red.norm(n, true, [&](int j) {
        const double dv = -aty[j];
        return (fmax(0.0, dv) * (double)!isfinite(lb[j]) - fmin(0.0, dv) * (double)!isfinite(ub[j])) * vr[j];
    });
    S.max_dray = dsn;
    const double sc = fmax(drn, dsn);
    if (sc > 0.0) {
        S.max_dray /= sc;
        S.dray_obj /= sc;
    } else {
        S.max_dray = 0.0;
        S.dray_obj = 0.0;
    }
}

// reference src/utils.cu:219-289 (the batch applies no wall-clock limit)
template <class T, int BT> __device__ inline void check_termination(const Ctx<T, BT> &C, State &S) {
    const Params &P = *C.P;
    if (S.rel_du < P.eps_feas && S.rel_pr < P.eps_feas && S.rel_gap < P.eps_opt) {
        S.reason = TERMINATION_REASON_OPTIMAL;
        return;
    }
    if (C.I.has_affine) {
        if (S.total >= P.iteration_limit) S.reason = TERMINATION_REASON_ITERATION_LIMIT;
        return;
    }
    if (S.dray_obj > 0.0 && S.max_dray / S.dray_obj <= P.eps_inf) {
        S.reason = TERMINATION_REASON_PRIMAL_INFEASIBLE;
        return;
    }
    if (S.pray_lin_obj < 0.0 && S.max_pray / (-S.pray_lin_obj) <= P.eps_inf) {
        S.reason = TERMINATION_REASON_DUAL_INFEASIBLE;
        return;
    }
    if (S.total >= P.iteration_limit) S.reason = TERMINATION_REASON_ITERATION_LIMIT;
}

// The persistent launch: workgroup b advances problem b by up to `budget`
// passes of the main loop from its saved state (every loop is bounded), and
// a problem that has terminated leaves A'y and Q x of its final point in the
// slab for the reduced costs and returns at once on later launches.
//
// T = float is the FP32 phase of the mixed batch: iterates, matrix values and
// products in FP32 (vpool, slabs), D, the k-vectors and the cone values in
// FP64 (dpool, wslabs), and a problem whose KKT error stops improving leaves
// with kStalled; the host then widens the iterates into the FP64 slabs and
// the FP64 kernel re-evaluates every problem before it terminates.
template <class T, int BT>
__global__ void __launch_bounds__(BT) batch_solve_kernel(const Params *P, const Inst *insts, const int *ipool,
                                                          const T *vpool, const double *dpool, T *slabs,
                                                          double *wslabs, const Cone *cones, State *states, Out *out,
                                                          int budget, int lds_bytes) {
    __shared__ double lds[2 * kBW];
    State S = states[blockIdx.x];
    if (S.reason != TERMINATION_REASON_UNSPECIFIED) return;
    constexpr bool fp32 = !std::is_same<T, double>::value;
    Ctx<T, BT> C;
    C.P = P;
    C.I = insts[blockIdx.x];
    C.arp = ipool + C.I.a_rp;
    C.aci = ipool + C.I.a_ci;
    C.atrp = ipool + C.I.at_rp;
    C.atci = ipool + C.I.at_ci;
    C.ach = ipool + C.I.a_chunk;
    C.atch = ipool + C.I.at_chunk;
    C.av = vpool + C.I.a_v;
    C.atv = vpool + C.I.at_v;
    C.R = vpool + C.I.rdense;
    C.D = dpool + C.I.dmat;
    C.V = slabs + C.I.vec;
    C.W = wslabs + C.I.wvec;
    C.cones = cones + C.I.cone0;
    C.red.lds = lds;
    // products stage their vector when it takes at most half of what a chunk
    // leaves; as many rows of R stay as fit behind both
    const int left = (lds_bytes - 2 * kMaxRank * (int)sizeof(double)) / (int)sizeof(T) - kChunk;
    const int widest = max(C.I.pn, C.I.pm);
    C.stage_room = widest <= left / 2 ? widest : 0;
    C.room = C.stage_room + kChunk;
    C.resident = C.I.qkind == kQLowRank ? min(C.I.k, (left - C.stage_room) / max(C.I.pn, 1)) : 0;
    for (int e = 2 * (int)threadIdx.x; e < C.resident * C.I.pn; e += 2 * BT) {
        const auto v = load_pair(C.R + e);
        store_pair_lds<T>(C.room + e, v[0], v[1]);
    }
    __syncthreads();
    const int ef = P->ef;
    for (int pass = 0; pass < budget; ++pass) {
        if (!(S.total < P->iteration_limit)) {
            S.reason = TERMINATION_REASON_ITERATION_LIMIT;
            residual(C, S);
            break;
        }
        const int tc = S.total;
        if (S.is_major || tc == 0 || S.eval_now || tc % print_frequency(tc) == 0) {
            S.eval_now = 0;
            residual(C, S);
            if (!C.I.has_affine && S.is_major && tc < 3 * ef) infeasibility(C, S);
            check_termination(C, S);
            if (S.reason != TERMINATION_REASON_UNSPECIFIED) break;
            if (fp32) {  // near the tolerance or at the FP32 floor: hand the problem to the FP64 kernel
                const double err = fmax(S.rel_pr, fmax(S.rel_du, S.rel_gap));
                if (err < P->handover) {
                    S.reason = kStalled;
                    break;
                }
                if (err < 0.5 * S.best_err) {
                    S.best_err = err;
                    S.best_iter = tc;
                } else if (tc - S.best_iter >= max(P->stall_iters, tc / 2)) {
                    S.reason = kStalled;
                    break;
                }
            }
        }
        if (fp32 && S.sat >= kSatStall) {
            S.reason = kStalled;
            break;
        }
        if (S.is_major || tc == 0) {
            S.do_restart = should_restart(C, S);
            if (S.do_restart) restart(C, S);
        }
        S.is_major = ((tc + 1) % ef) == 0;
        pdhg_step(C, S);
        if (S.is_major || S.do_restart) {
            fixed_point_error(C, S);
            if (S.do_restart) {
                S.init_fpe = S.fpe;
                S.do_restart = 0;
            }
        }
        halpern(C, S);
        S.inner_count++;
        S.total++;
    }
    if (S.reason != TERMINATION_REASON_UNSPECIFIED && !fp32) {
        C.At(C.mv(wYP), C.nv(vATY));
        C.obj_product(C.nv(vXP), C.nv(vQX));
    }
    if (threadIdx.x == 0) {
        states[blockIdx.x] = S;
        Out o;
        o.status = S.reason;
        o.iters = S.total;
        o.inner = S.inner_total;
        o.pobj = S.pobj;
        o.dobj = S.dobj;
        o.abs_pr = S.abs_pr;
        o.abs_du = S.abs_du;
        o.rel_pr = S.rel_pr;
        o.rel_du = S.rel_du;
        o.gap = S.gap;
        o.rel_gap = S.rel_gap;
        o.max_pray = S.max_pray;
        o.max_dray = S.max_dray;
        o.pray_lin_obj = S.pray_lin_obj;
        o.dray_obj = S.dray_obj;
        out[blockIdx.x] = o;
    }
}

}  // namespace batch
}  // namespace pdhcg
