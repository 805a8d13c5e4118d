// The projected Barzilai-Borwein inner solve (reference pdhg_core_op.cu:495-669)
// as one launch per outer iteration, for problems that fit the chip: its first
// step, every loop body, the reflection and the Halpern update.
//
// Launched kernel by kernel, a body is six launches (five for a sparse Q) of
// 2-4 us each whatever the problem's size: 26 us per body at n = 60, 11-23 us
// with a 2000-variable sparse Q.  Here the columns are split over at most
// kInnerMaxGroups workgroups that stay resident, and a body costs two
// exchanges of a few values between them (1-3 us each).
//
// Exchange between workgroups.  A value crosses as two 64-bit words, each
// holding a 32-bit sequence number and one half of the double, stored and
// loaded with relaxed device-scope atomics.  A word is taken only when it
// carries the expected sequence number, so no fence, flag or ordering between
// different words is needed (a device-scope release writes back the XCD's L2:
// measured 17 us per barrier at 256 workgroups, against 3.2 us for an
// exchange).  Each kind of exchange alternates two buffers: a workgroup writes
// sequence number s + 2 only after it has read every workgroup's s + 1, and
// those were written after their writers' last read of s.
//
// Residency.  A workgroup waits for the others, so all of a grid's must be able
// to run at once.  Each fits a compute unit of its own, and only one does in
// places (512 threads are two waves per SIMD: 124 to 256 registers here leave
// room for no further waiting workgroup), so grids are safe beside each other
// while together they have at most one workgroup per unit of every XCD.
// Workgroups are dealt to the XCDs in turn: a grid of G takes up to
// ceil(G / 8) units of each.  Other kernels hold their units only for a time.
// InnerResidents keeps the count for the process: while all live resident grids
// fit the chip together they run side by side, else a launch first waits for
// the other solvers' streams, so that they run one after the other.  Large grids
// are launched cooperatively, which costs about 18 us per launch more: the
// runtime then refuses a grid that would not fit the empty chip.  Grids of other
// processes on the same GPU are in nobody's count.
//
// A wait that lasts kInnerWaitSeconds gives up: it notes the launch's number in
// DevScalars and clears inner_run, and every workgroup leaves.  All that changes
// the state after an inner solve is gated by inner_run (later inner solves, the
// dual step, the Halpern updates) and the inner solve itself writes no vector
// that it reads, so the state stays that before the launch, and the host, at its
// next read of the scalars, takes the loop back to there and goes on launch by
// launch (Solver::rewind_inner).
#pragma once

#include <algorithm>
#include <mutex>
#include <vector>

#include "dev_kernels.hpp"

namespace pdhcg {

constexpr int kInnerThreads = 512, kInnerWaves = kInnerThreads / kWave;
constexpr int kInnerCols = kInnerThreads;      // columns of a workgroup, one per thread
constexpr int kInnerColSets = kInnerCols / kWave;
constexpr int kInnerMaxGroups = 256;           // one workgroup per compute unit
constexpr int kInnerXcds = 8;
constexpr int kInnerPlainGroups = 8, kInnerSparseGroups = 16;
constexpr int kInnerAllGroups = 16;            // low rank: every workgroup sums all partial rows up to here
constexpr int kInnerMaxRank = 80;              // rows of R: ten per wave
constexpr int kInnerSparseVars = 8192;         // x_p of the sparse form is held in LDS (64 KB)
// Longer than other streams' kernels hold the chip as a rule; an exchange takes
// microseconds.
constexpr double kInnerWaitSeconds = 1.0;

typedef unsigned long long xword;

// The resident grids of this process: one entry per solver that has a resident
// form of several workgroups, from its set-up to its end.
class InnerResidents {
  public:
    struct Grid {
        int device = 0, units = 0;  // units: workgroups, rounded up to a multiple of the XCDs
        hipStream_t st = nullptr;
        hipEvent_t ev = nullptr;    // set while the grid is counted
        void enter() {
            HIP_OK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
            InnerResidents &all = instance();
            std::lock_guard<std::mutex> lock(all.mu_);
            all.live_.push_back(this);
        }
        // With the stream idle, or at least no resident launch in it.
        void leave() {
            if (!ev) return;
            InnerResidents &all = instance();
            std::lock_guard<std::mutex> lock(all.mu_);
            all.live_.erase(std::remove(all.live_.begin(), all.live_.end(), this), all.live_.end());
            (void)hipEventDestroy(ev);
            ev = nullptr;
        }
        Grid() = default;
        Grid(const Grid &) = delete;
        Grid &operator=(const Grid &) = delete;
        ~Grid() { leave(); }
    };
    static InnerResidents &instance() {
        static InnerResidents *all = new InnerResidents;  // solvers may outlive static objects
        return *all;
    }
    // Calls enqueue(), which launches g's grid, so that it runs only beside
    // grids that fit a chip of `units` compute units with it.  Beyond that it
    // waits on the device for all that the other solvers have enqueued (idle
    // ones are passed over); what they launch later waits for g in turn.
    template <class F> void launch(const Grid &g, int units, F enqueue) {
        std::lock_guard<std::mutex> lock(mu_);
        int total = 0;
        for (const Grid *o : live_)
            if (o->device == g.device) total += o->units;
        if (total > units)
            for (const Grid *o : live_) {
                if (o->device != g.device || o->st == g.st) continue;
                const hipError_t state = hipStreamQuery(o->st);
                if (state == hipSuccess) continue;
                if (state != hipErrorNotReady) HIP_OK(state);
                (void)hipGetLastError();  // the query's own "not ready"
                HIP_OK(hipEventRecord(o->ev, o->st));
                HIP_OK(hipStreamWaitEvent(g.st, o->ev, 0));
            }
        enqueue();
    }

  private:
    std::mutex mu_;
    std::vector<Grid *> live_;
};

// Device memory of the exchanges.
struct InnerExchange {
    xword *rows;     // [2][rows][groups] partial sums (low rank), or [2][n] x_p (sparse Q)
    xword *total;    // [2][rows] sums over the workgroups
    xword *scalar;   // [2][groups] partial sums (sparse Q: [2][groups * kInnerWaves])
    unsigned *seq;   // sequence numbers of the kinds of exchange, kept between launches
    long long wait;  // wall-clock ticks after which a wait gives up
};

// Arguments common to the forms.  The Halpern update goes to x_next, not to x:
// with an inner limit of 1 there is no exchange after the loads of x, and a
// workgroup that starts late still reads other workgroups' columns of x.
template <class X> struct InnerArgs {
    int n, limit, halpern;
    int launch;   // number of this inner solve
    int give_up;  // 1: the last workgroup gives up at its first wait (tests)
    double alpha0, inv_tau, tol, w, rho;
    const X *x;
    X *x_next, *xp, *xr;
    const X *x0, *c, *aty, *lb, *ub, *qdiag, *m_inv, *m_diag;
    InnerExchange ex;
    DevScalars *ds;
};

__device__ __forceinline__ void exchange_put(xword *slot, double v, unsigned seq) {
    const xword b = (xword)__double_as_longlong(v), t = (xword)seq << 32;
    __hip_atomic_store(slot, t | (b & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(slot + 1, t | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What a wait that gives up does: notes it for the host and the other
// workgroups (device memory), and for this workgroup (LDS, read after its next
// barrier, so that all its threads leave together).
struct InnerWait {
    long long ticks;  // negative: gives up at once
    int launch;
    DevScalars *ds;
    int *group_fail;
    __device__ bool others_gave_up() const {
        return __hip_atomic_load(&ds->inner_run, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
    }
    __device__ void give_up() const {
        __hip_atomic_store(&ds->inner_gave_up, launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&ds->inner_run, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *group_fail = 1;
    }
};
template <class X> __device__ __forceinline__ InnerWait inner_wait(const InnerArgs<X> &a, int *group_fail) {
    return InnerWait{a.give_up && blockIdx.x + 1 == gridDim.x ? -1LL : a.ex.wait, a.launch, a.ds, group_fail};
}

// Waits for U values with sequence number `seq`, those at first, first + step,
// ... below `count` (the others are 0), all loads in flight together (a load
// takes about 0.7 us).  The values are 0 after the time limit, or when another
// workgroup has given up.
template <int U>
__device__ __forceinline__ void exchange_get(const xword *slots, int first, int step, int count, unsigned seq,
                                             const InnerWait &w, double (&v)[U]) {
    xword a[U], b[U];
    long long start = 0;
    for (unsigned polls = 1;; ++polls) {
#pragma unroll
        for (int q = 0; q < U; ++q) {
            a[q] = b[q] = (xword)seq << 32;
            const int i = first + q * step;
            if (i < count) {
                a[q] = __hip_atomic_load(slots + (size_t)i * 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                b[q] = __hip_atomic_load(slots + (size_t)i * 2 + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        bool all = w.ticks >= 0;
#pragma unroll
        for (int q = 0; q < U; ++q) all = all && (unsigned)(a[q] >> 32) == seq && (unsigned)(b[q] >> 32) == seq;
        if (all) break;
        if (polls % 256 == 0 || w.ticks < 0) {
            const long long now = wall_clock64();
            if (start == 0) start = now;
            if (now - start > w.ticks || w.others_gave_up()) {
                w.give_up();
#pragma unroll
                for (int q = 0; q < U; ++q) a[q] = b[q] = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(8);
        }
    }
#pragma unroll
    for (int q = 0; q < U; ++q) v[q] = __longlong_as_double((long long)((b[q] << 32) | (a[q] & 0xffffffffull)));
}

// The flags before the first resident inner solve, and after one that gave up
// (whose bodies the launches that take its place count again).
__global__ void inner_reset_kernel(DevScalars *ds) {
    if (ds->inner_gave_up && ds->inner_counted == ds->inner_gave_up) ds->inner_total -= ds->bb_iter - 1;
    ds->inner_gave_up = 0;
    ds->inner_run = 1;
}

// A sequence number kept between launches: read before the workgroup's first
// barrier (an atomic load is not moved past it), since workgroup 0 stores the
// next launch's once it has every workgroup's first value.
__device__ __forceinline__ unsigned inner_seq(const unsigned *seq) {
    return __hip_atomic_load(seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Totals of NR <= 16 (a power of two) per-lane values over the wave, halving
// the values a lane carries with each exchange: lane l receives the total of
// value l / (64 / NR).  Fixed combination order.
template <int NR> __device__ __forceinline__ double wave_total_rows(double (&s)[NR], int lane) {
    if constexpr (NR == 1) {
        return wave_total(s[0]);
    } else {
        constexpr int h1 = NR / 2;
#pragma unroll
        for (int i = 0; i < h1; ++i) s[i] = fold32(s[i], s[i + h1]);
        constexpr int h2 = h1 > 1 ? h1 / 2 : 1;
#pragma unroll
        for (int i = 0; i < h2; ++i) s[i] = h1 > 1 ? fold16(s[i], s[i + h2]) : fold16(s[0], s[0]);
        constexpr int h3 = NR >= 8 ? NR / 8 : 1;
        const bool hi8 = (lane & 8) != 0, hi4 = (lane & 4) != 0;
        if constexpr (NR >= 8) {
#pragma unroll
            for (int i = 0; i < h3; ++i) {
                const double keep = hi8 ? s[i + h3] : s[i], give = hi8 ? s[i] : s[i + h3];
                s[i] = keep + dpp_move<kDppRor8>(give);
            }
        }
        double v = s[0];
        if constexpr (NR == 16) {
            const double keep = hi4 ? s[1] : s[0], give = hi4 ? s[0] : s[1];
            v = keep + dpp_move<kDppHalfMirror>(give);
        }
        v += dpp_move<kDppXor1>(v);
        v += dpp_move<kDppXor2>(v);
        if constexpr (NR <= 8) v += dpp_move<kDppHalfMirror>(v);
        if constexpr (NR <= 4) v += dpp_move<kDppMirror>(v);
        return v;
    }
}

// Sum of `count` <= 256 values over the wave, every lane receives it (fixed order).
__device__ __forceinline__ double exchange_sum(const xword *slots, int lane, int count, unsigned seq,
                                               const InnerWait &w) {
    double v[4];
    exchange_get<4>(slots, lane, kWave, count, seq, w, v);
    return wave_total((v[0] + v[1]) + (v[2] + v[3]));
}

// One column's part of the inner solve, in its owner thread's registers.
template <class X> struct InnerColumn {
    double x, lb, ub, mi, md, ec, qd;  // ec = c - A'y
    double c, aty;
    double xp, grad, dirn;
    bool live;
    __device__ void load(const InnerArgs<X> &a, long long i) {
        live = i < a.n;
        x = lb = ub = ec = qd = c = aty = xp = grad = dirn = 0.0;
        mi = md = 1.0;
        if (!live) return;
        x = (double)a.x[i];
        lb = (double)a.lb[i];
        ub = (double)a.ub[i];
        c = (double)a.c[i];
        aty = (double)a.aty[i];
        ec = c - aty;
        if (a.qdiag) qd = (double)a.qdiag[i];
        if (a.m_inv) {
            mi = (double)a.m_inv[i];
            md = (double)a.m_diag[i];
        }
    }
    // Steps along -scale grad from `from`; returns the step's term of |s|^2 or s'Ms.
    __device__ double step(double from, double scale, bool pre) {
        if (!live) return 0.0;
        double nx = pre ? from - scale * mi * grad : from - scale * grad;
        nx = fmax(lb, fmin(nx, ub));
        xp = (double)(X)nx;
        dirn = (double)(X)(xp - from);
        return pre ? dirn * (md * dirn) : dirn * dirn;
    }
    // First step from x (bb_init_kernel) for the product qx of x; returns the step's term.
    __device__ double first(double qx, double scale, bool pre) {
        grad = (double)(X)qx + c - aty;
        const double v = step(x, scale, pre);
        grad = (double)(X)grad;
        return v;
    }
    // Gradient at x_p (bb_gradient_kernel) for its product qx; returns the term of s'(g - g_old).
    __device__ double gradient(double qx, double inv_tau) {
        const double cur = (double)(X)qx + ec + inv_tau * (xp - x);
        const double dg = (double)(X)(cur - grad);
        grad = (double)(X)cur;
        return live ? dirn * dg : 0.0;
    }
    __device__ void finish(const InnerArgs<X> &a, long long i) const {
        if (!live) return;
        const double ref = 2.0 * xp - x;
        a.xp[i] = (X)xp;
        a.xr[i] = (X)ref;
        if (a.halpern) {
            const double refl = a.rho * ref + (1.0 - a.rho) * x;
            a.x_next[i] = (X)(a.w * refl + (1.0 - a.w) * (double)a.x0[i]);
        }
    }
};

// ---------------------------------------------------------------------------
// Q = R'DR (+ diagonal), R dense: n up to kInnerCols * kInnerMaxGroups, rank up
// to kInnerMaxRank.
//
// Workgroup g owns kInnerCols columns and keeps its slice of R in registers
// for the whole inner solve (at ranks 57 to 80 in FP64 160 of a thread's 256
// registers, of which 13 other values are spilled, in FP32 as well: 56 bytes of
// scratch per lane; no spills up to rank 56), so that R is read once per outer iteration instead of twice per body: wave w
// holds rows w, w + 8, ... and lane l of it columns l, l + 64, ...  R x is
// then a sum over a lane's eight columns and a butterfly over the wave, with
// no sum across waves; R'u is a sum over a thread's rows and, through LDS, the
// eight waves.  Measured at n = 100 000, rank 50 (R = 40 MB): see the figures
// at Solver::init_inner_form.
//
// Exchanges per body: the rows of R x_p together with the norm of the last
// step (the loop's stopping test), then the curvature s'(g - g_old).  With up
// to kInnerAllGroups workgroups each sums all partial rows itself; with
// more, workgroup j sums row j and publishes the total (the rows of all
// workgroups would be 53 MB of uncached reads at 256 workgroups and rank 50).
template <class V, class X, int RW>
__global__ void __launch_bounds__(kInnerThreads) inner_lowrank_kernel(InnerArgs<X> a, const V *R, int k,
                                                                       const double *ddiag, const double *ddense,
                                                                       int dkind) {
    constexpr int NR = RW <= 1 ? 1 : RW <= 2 ? 2 : RW <= 4 ? 4 : RW <= 8 ? 8 : 16;
    __shared__ double xs[kInnerCols], part[kInnerWaves * kInnerCols];
    __shared__ int group_fail, skip;
    __shared__ double dsum, us[kInnerMaxRank + 1], u2[kInnerMaxRank + 1], nw[kInnerWaves], dw[kInnerWaves];
    const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
    const int G = gridDim.x, g = blockIdx.x, rows = k + 1;
    const long long col0 = (long long)g * kInnerCols, i = col0 + t;
    const bool pre = a.m_inv != nullptr;
    unsigned seq_rows = inner_seq(a.ex.seq), seq_s = inner_seq(a.ex.seq + 1);
    DevScalars *ds = a.ds;
    const InnerWait wait = inner_wait(a, &group_fail);
    if (t == 0) {
        group_fail = 0;
        skip = G > 1 && wait.others_gave_up();
    }

    V r[RW][kInnerColSets];
    const long long padded = (long long)rx_chunks(a.n) * kRxWaveCols;
#pragma unroll
    for (int b = 0; b < RW; ++b)
#pragma unroll
        for (int q = 0; q < kInnerColSets; ++q) {
            const int j = wave + b * kInnerWaves;
            const long long cidx = col0 + lane + q * kWave;
            r[b][q] = (j < k && cidx < padded) ? R[rx_tile_index(j, cidx, k)] : V(0);
        }
    InnerColumn<X> col;
    col.load(a, i);

    // u = D R v for the v in xs, into us[0 .. k); the sum over the workgroups
    // of `extra` (thread 0 .. kInnerWaves - 1 terms in nw) into us[k].  Called
    // after a barrier that follows the writes of xs and nw; ends with one.
    // Returns false when a wait gave up.
    auto product = [&]() {
        double s[NR];
#pragma unroll
        for (int b = 0; b < NR; ++b) {
            s[b] = 0.0;
            if (b < RW)
#pragma unroll
                for (int q = 0; q < kInnerColSets; ++q) s[b] += (double)r[b < RW ? b : 0][q] * xs[lane + q * kWave];
        }
        const double tot = wave_total_rows<NR>(s, lane);
        const int j = wave + (lane / (kWave / NR)) * kInnerWaves;
        const bool lead = lane % (kWave / NR) == 0;
        double extra = 0.0;
        if (wave == k % kInnerWaves && lane == 0)
            for (int q = 0; q < kInnerWaves; ++q) extra += nw[q];
        if (G == 1) {
            if (lead && j < k) us[j] = dkind == 1 ? tot * ddiag[j] : tot;
            if (wave == k % kInnerWaves && lane == 0) us[k] = extra;
        } else {
            ++seq_rows;
            xword *P = a.ex.rows + (size_t)(seq_rows & 1) * rows * G * 2;
            if (lead && j < k) exchange_put(P + ((size_t)j * G + g) * 2, tot, seq_rows);
            if (wave == k % kInnerWaves && lane == 0) exchange_put(P + ((size_t)k * G + g) * 2, extra, seq_rows);
            if (G <= kInnerAllGroups) {
                // sixteen lanes (workgroups) per row, four rows per load; the
                // wave's rows are all in flight together
                constexpr int U = (RW + 1 + 3) / 4;
                const int o = lane % 16, row0 = wave + lane / 16 * kInnerWaves;
                double v[U];
                const bool in = o < G;
                exchange_get<U>(P + (size_t)o * 2, in ? row0 * G : rows * G, 4 * kInnerWaves * G, rows * G, seq_rows,
                                wait, v);
#pragma unroll
                for (int b = 0; b < U; ++b) {
                    const int row = row0 + b * 4 * kInnerWaves;
                    const double sum = row_total(v[b]);
                    if (o == 0 && row <= k) us[row] = (dkind == 1 && row < k) ? sum * ddiag[row] : sum;
                }
            } else {
                xword *T = a.ex.total + (size_t)(seq_rows & 1) * rows * 2;
                for (int row = g + wave * G; row <= k; row += kInnerWaves * G) {
                    const double v = exchange_sum(P + (size_t)row * G * 2, lane, G, seq_rows, wait);
                    if (lane == 0) exchange_put(T + (size_t)row * 2, (dkind == 1 && row < k) ? v * ddiag[row] : v, seq_rows);
                }
                if (t <= k) {
                    double v[1];
                    exchange_get<1>(T, t, 0, rows, seq_rows, wait, v);
                    us[t] = v[0];
                }
            }
        }
        __syncthreads();
        if (dkind == 2) {
            if (t < k) {
                double v = 0.0;
                for (int q = 0; q < k; ++q) {
                    const int lo = t < q ? t : q, hi = t < q ? q : t;
                    v += ddense[(size_t)lo * k + hi] * us[q];
                }
                u2[t] = v;
            }
            __syncthreads();
        }
        return group_fail == 0;
    };
    // R'u of the owner's column; ends after a barrier that frees `part` for
    // the next call's writers (they follow another product's barriers).
    auto transpose_product = [&]() {
        const double *u = dkind == 2 ? u2 : us;
        double p[kInnerColSets];
#pragma unroll
        for (int q = 0; q < kInnerColSets; ++q) p[q] = 0.0;
#pragma unroll
        for (int b = 0; b < RW; ++b) {
            const int j = wave + b * kInnerWaves;
            const double uj = j < k ? u[j] : 0.0;
#pragma unroll
            for (int q = 0; q < kInnerColSets; ++q) p[q] += (double)r[b][q] * uj;
        }
#pragma unroll
        for (int q = 0; q < kInnerColSets; ++q) part[wave * kInnerCols + lane + q * kWave] = p[q];
        __syncthreads();
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < kInnerWaves; ++q) v += part[q * kInnerCols + t];
        return v;
    };

    // first step from x
    xs[t] = col.x;
    if (t < kInnerWaves) nw[t] = 0.0;
    __syncthreads();
    if (skip || !product()) return;
    double qx = transpose_product();
    if (a.qdiag) qx = qx + col.qd * col.x;
    double nv = col.first(qx, pre ? a.alpha0 * (ds->tol_scale * ds->tol_scale) : a.alpha0, pre);
    int it = 1;
    while (it < a.limit) {
        xs[t] = col.xp;
        nv = wave_total(nv);
        if (lane == 0) nw[wave] = nv;
        __syncthreads();
        if (!product()) return;
        const double s2 = us[k], nrm = sqrt(s2);
        if (nrm <= a.tol) break;
        qx = transpose_product();
        if (a.qdiag) qx = qx + col.qd * col.xp;
        double curv = wave_total(col.gradient(qx, a.inv_tau));
        if (lane == 0) dw[wave] = curv;
        __syncthreads();
        curv = 0.0;
        for (int q = 0; q < kInnerWaves; ++q) curv += dw[q];
        if (G > 1) {
            ++seq_s;
            xword *P = a.ex.scalar + (size_t)(seq_s & 1) * G * 2;
            if (wave == 0) {
                if (lane == 0) exchange_put(P + (size_t)g * 2, curv, seq_s);
                curv = exchange_sum(P, lane, G, seq_s, wait);
                if (lane == 0) dsum = curv;
            }
            __syncthreads();
            curv = dsum;
        }
        const double alpha = pre ? s2 / curv : (nrm * nrm) / curv;
        nv = col.step(col.xp, alpha, pre);
        ++it;
    }
    col.finish(a, i);
    if (g == 0 && t == 0) {
        ds->bb_iter = it;
        ds->inner_total += it - 1;
        ds->inner_counted = a.launch;
        a.ex.seq[0] = seq_rows;
        a.ex.seq[1] = seq_s;
    }
}

// ---------------------------------------------------------------------------
// Q sparse (or only its diagonal): n up to kInnerSparseVars.
//
// Workgroup g owns `cols` (<= kInnerThreads) variables and their rows of Q, cut
// into tasks of at most kInnerTask entries (task_start: first entry of each
// task, row_task: first task of each row), at most one per thread, which keeps
// its entries in registers for the whole inner solve; the owner of a row adds
// its tasks in order.  (With a fixed number of threads per row the longest row
// decided: 3 us of a 7 us body at 41 entries per row on average.)  Every
// workgroup holds all of x_p in LDS, so the gathers of Q x_p hit LDS.  A Q with
// more tasks than threads would be reread in every body: 2000 to 4000 variables
// with 1000 tasks or more per workgroup measured 19 to 47 us per body, against
// 16 to 18 launch by launch, so those keep the launches.
//
// Exchanges per body: x_p, from which every workgroup forms the norm of the
// whole step itself (in the same order), then the curvature.  One wave per
// workgroup waits for that sum; with all eight of them polling, an exchange
// of 16 workgroups took 5.5 us instead of 1.5.
// Dynamic LDS: x_p (n doubles).
constexpr int kInnerTask = 16;

template <class V, class X, class Acc>
__global__ void __launch_bounds__(kInnerThreads) inner_sparse_kernel(InnerArgs<X> a, int cols, const int *row_task,
                                                                      const int *task_start, const int *ci,
                                                                      const V *val) {
    extern __shared__ double inner_lds[];
    __shared__ double sums[kInnerThreads], nw[kInnerWaves], dw[kInnerWaves], total;
    __shared__ int group_fail, skip;
    const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
    const int G = gridDim.x, g = blockIdx.x, n = a.n;
    const int row0 = g * cols, nrows = max(0, min(cols, n - row0));
    const bool pre = a.m_inv != nullptr;
    double *xs = inner_lds;
    unsigned seq_x = inner_seq(a.ex.seq), seq_s = inner_seq(a.ex.seq + 1);
    DevScalars *ds = a.ds;
    const InnerWait wait = inner_wait(a, &group_fail);
    if (t == 0) {
        group_fail = 0;
        skip = G > 1 && wait.others_gave_up();
    }
    InnerColumn<X> col;
    col.load(a, t < nrows ? (long long)row0 + t : (long long)n);

    const int task0 = val ? row_task[row0] : 0, tasks = val ? row_task[row0 + nrows] - task0 : 0;
    const int my0 = (val && t < nrows) ? row_task[row0 + t] - task0 : 0;
    const int my1 = (val && t < nrows) ? row_task[row0 + t + 1] - task0 : 0;
    int rc[kInnerTask];  // entry's column, -1: none
    V rv[kInnerTask];
    const int e0 = t < tasks ? task_start[task0 + t] : 0, e1 = t < tasks ? task_start[task0 + t + 1] : 0;
#pragma unroll
    for (int q = 0; q < kInnerTask; ++q) {
        rc[q] = e0 + q < e1 ? ci[e0 + q] : -1;
        rv[q] = e0 + q < e1 ? val[e0 + q] : V(0);
    }
    // Q v of the owner's variable for the v in xs (written before a barrier);
    // a barrier follows the last read of xs.
    auto product = [&](double own) {
        if (!val) {
            __syncthreads();
            return col.qd * own;
        }
        Acc x[kInnerTask], part = Acc(0), acc = Acc(0);
#pragma unroll
        for (int q = 0; q < kInnerTask; ++q) x[q] = (Acc)xs[rc[q] < 0 ? 0 : rc[q]];
#pragma unroll
        for (int q = 0; q < kInnerTask; ++q)
            if (rc[q] >= 0) part += (Acc)rv[q] * x[q];
        sums[t] = (double)part;
        __syncthreads();
        for (int q = my0; q < my1; ++q) acc += (Acc)sums[q];
        return (double)acc;
    };

    // Sum over the workgroups of a term per wave (given in its lane 0).
    auto all_sum = [&](double v) {
        if (G == 1) {
            if (lane == 0) dw[wave] = v;
            __syncthreads();
            double s = 0.0;
            for (int q = 0; q < kInnerWaves; ++q) s += dw[q];
            return s;
        }
        const int count = G * kInnerWaves;
        ++seq_s;
        xword *P = a.ex.scalar + (size_t)(seq_s & 1) * count * 2;
        if (lane == 0) exchange_put(P + (size_t)(g * kInnerWaves + wave) * 2, v, seq_s);
        if (wave == 0) {
            const double s = exchange_sum(P, lane, count, seq_s, wait);
            if (lane == 0) total = s;
        }
        __syncthreads();
        return total;
    };

    if (val)
        for (int i = t; i < n; i += kInnerThreads) xs[i] = (double)a.x[i];
    __syncthreads();
    if (skip) return;
    double nv = col.first(product(col.x), pre ? a.alpha0 * (ds->tol_scale * ds->tol_scale) : a.alpha0, pre);
    int it = 1;
    while (it < a.limit) {
        // x_p of every workgroup, and |s|^2 or s'Ms
        if (val && G > 1) {
            ++seq_x;
            xword *P = a.ex.rows + (size_t)(seq_x & 1) * n * 2;
            if (t < nrows) exchange_put(P + (size_t)(row0 + t) * 2, col.xp, seq_x);
            nv = 0.0;
            for (int i = t; i < n; i += 4 * kInnerThreads) {
                double v[4];
                exchange_get<4>(P, i, kInnerThreads, n, seq_x, wait, v);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int j = i + q * kInnerThreads;
                    if (j >= n) break;
                    const double s = (double)(X)(v[q] - xs[j]);
                    nv += pre ? s * ((double)a.m_diag[j] * s) : s * s;
                    xs[j] = v[q];
                }
            }
        } else if (val && t < nrows) {
            xs[t] = col.xp;
        }
        nv = wave_total(nv);
        if (lane == 0) nw[wave] = nv;
        __syncthreads();
        if (group_fail) return;
        double s2 = 0.0;
        for (int q = 0; q < kInnerWaves; ++q) s2 += nw[q];
        if (!val && G > 1) s2 = all_sum(nv);
        const double nrm = sqrt(s2);
        if (nrm <= a.tol) break;
        const double curv = all_sum(wave_total(col.gradient(product(col.xp), a.inv_tau)));
        const double alpha = pre ? s2 / curv : (nrm * nrm) / curv;
        nv = col.step(col.xp, alpha, pre);
        ++it;
    }
    col.finish(a, (long long)row0 + t);
    if (g == 0 && t == 0) {
        ds->bb_iter = it;
        ds->inner_total += it - 1;
        ds->inner_counted = a.launch;
        a.ex.seq[0] = seq_x;
        a.ex.seq[1] = seq_s;
    }
}

}  // namespace pdhcg
