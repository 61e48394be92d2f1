// Preconditioned CG with one launch per iteration.
//
// The library's order (z = D^-1 r; beta = rho / rho_prev; p = z + beta p;
// q = K p; alpha = rho / p.q; x += alpha p; r -= alpha q) has two grid-wide
// sums an iteration, r.z and p.q, so it takes two launches.  Here launch k
// applies the pending update of iteration k - 1 (x, r) while it stages the
// new direction for its own operator product, and beta is known before r is:
// every launch also sums q.z, q.D^-1 q, r.q and q.q of the vectors it holds,
// and with r' = r - alpha q
//     r'.z' = r.z - 2 alpha q.z + alpha^2 q.D^-1 q,
//     r'.r' = r.r - 2 alpha r.q + alpha^2 q.q.
// r.z and r.r on the right are sums over the actual vectors in every launch,
// so nothing accumulates; the one subtraction loses at most a factor
// 1 / kPcg1Keep: where a step shrinks either sum further than that, the launch
// only applies the update and sums r'.z' and r'.r' directly, and the next
// launch goes on from those (kPcg1Exact).  q = K p is always a product, never
// a recurrence.
//
// The vectors r, p, q, the state and the partial sums exist twice: a launch
// reads one set and writes the other (other workgroups read the old values on
// their halos), so launches alternate and a graph holds an even number.  x is
// read and written by the owner of a node only.
#pragma once
#include <type_traits>

#include "k_common.h"
#include "pcg1_schedule.h"

namespace tohip {

constexpr int kPcg1Vals = 8;          // sums of one launch (7 used), one row per workgroup
constexpr double kPcg1Keep = 1e-3;    // smallest r'.z' / r.z (r'.r' / r.r) formed by subtraction

struct Pcg1State {
    double rho_prev;  // r.z behind the current direction
    double rr, rr0;   // r.r of the last stopping test, of the start
    double tol;       // stopping threshold on ||r|| (< 0: set by the first test)
    double abstol, reltol;
    long long iter, maxiter;
    int pend;  // p and q hold an iteration whose update has not been applied
    int done, err, pad;
};

enum { kSumRZ, kSumPQ, kSumQZ, kSumQDQ, kSumRR, kSumRQ, kSumQQ };
enum { kPcg1Step, kPcg1Exact, kPcg1Stop };

struct Pcg1Plan {
    double alpha, beta;
    int mode;
};

// What a launch does, from the previous launch's state and sums; `o` is the
// state it leaves.  Every thread of every workgroup computes the same.
__device__ __forceinline__ Pcg1Plan pcg1_plan(const Pcg1State& s, const double (&v)[kPcg1Vals],
                                              Pcg1State& o) {
    o = s;
    double alpha = 0.0, rz = v[kSumRZ], rr = v[kSumRR];
    if (s.pend) {
        if (!(isfinite(rz) && isfinite(rr))) {
            o.err = kPcgErrNonFinite;
            o.done = 1;
            return {0.0, 0.0, kPcg1Stop};
        }
        const double pq = v[kSumPQ];
        if (!(pq > 0.0 && pq < INFINITY)) {
            o.err = kPcgErrIndefinite;
            o.done = 1;
            return {0.0, 0.0, kPcg1Stop};
        }
        alpha = rz / pq;
        o.iter = s.iter + 1;
        o.rho_prev = rz;
        const double rz1 = rz - 2.0 * alpha * v[kSumQZ] + alpha * alpha * v[kSumQDQ];
        const double rr1 = rr - 2.0 * alpha * v[kSumRQ] + alpha * alpha * v[kSumQQ];
        if (!(rz1 >= kPcg1Keep * rz && rr1 >= kPcg1Keep * rr)) {
            o.pend = 0;
            return {alpha, 0.0, kPcg1Exact};
        }
        rz = rz1;
        rr = rr1;
    }
    if (s.tol < 0.0) {
        o.tol = fmax(s.reltol * sqrt(rr), s.abstol);
        o.rr0 = rr;
    }
    o.rr = rr;
    // ||r|| <= tol; the root is taken only where the squares are near each other
    // (or tiny), for it is a good part of a small launch's serial chain
    const double t2 = o.tol * o.tol;
    const bool met = rr <= 2.0 * t2 || t2 < 1e-280 ? sqrt(rr) <= o.tol : false;
    int err = 0;
    if (!(isfinite(rr) && isfinite(rz)))
        err = kPcgErrNonFinite;
    else if (!(rz > 0.0) && rr > 0.0 && !met)
        err = kPcgErrPrecond;
    if (err != 0 || met || o.iter >= s.maxiter) {
        o.done = 1;
        o.err = err;
        return {alpha, 0.0, kPcg1Stop};
    }
    o.pend = 1;
    return {alpha, rz / o.rho_prev, kPcg1Step};
}

// The eight sums over the workgroup, returned to every thread: a reduce-scatter
// over the wave (lanes keep the half of the values that three of their lane
// bits select: 10 shuffles instead of 48), then the waves in order.
template <int NT>
__device__ __forceinline__ void block_sum8(double (&v)[kPcg1Vals], double (*red)[kPcg1Vals]) {
    const int lane = threadIdx.x & 63;
    auto halve = [&](auto half, int bit) {
        constexpr int h = decltype(half)::value;
        const bool up = (lane & bit) != 0;
#pragma unroll
        for (int j = 0; j < h; ++j) {
            const double keep = up ? v[j + h] : v[j], send = up ? v[j] : v[j + h];
            v[j] = keep + __shfl_xor(send, bit, 64);
        }
    };
    halve(std::integral_constant<int, 4>{}, 32);
    halve(std::integral_constant<int, 2>{}, 16);
    halve(std::integral_constant<int, 1>{}, 8);
    double t = v[0];
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
    __syncthreads();
    if ((lane & 7) == 0) red[threadIdx.x >> 6][lane >> 3] = t;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPcg1Vals; ++j) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) s += red[w][j];
        v[j] = s;
    }
}

// The workgroup's row of partial sums.
template <int NT = kThreads>
__device__ __forceinline__ void pcg1_store_sums(double (&sum)[kPcg1Vals],
                                                double (*red)[kPcg1Vals],
                                                double* __restrict__ part) {
    block_sum8<NT>(sum, red);
    if (threadIdx.x < kPcg1Vals) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) t += red[w][threadIdx.x];
        part[(size_t)blockIdx.x * kPcg1Vals + threadIdx.x] = t;
    }
}

// Sum of nb rows of the previous launch's partials, the same in every thread.
template <int NT>
__device__ __forceinline__ void pcg1_reduce(const double* __restrict__ part, int nb,
                                            double (&v)[kPcg1Vals], double (*red)[kPcg1Vals]) {
#pragma unroll
    for (int j = 0; j < kPcg1Vals; ++j) v[j] = 0.0;
    for (int i = threadIdx.x; i < nb; i += NT) {
        const double2* row = reinterpret_cast<const double2*>(part + (size_t)i * kPcg1Vals);
#pragma unroll
        for (int j = 0; j < kPcg1Vals / 2; ++j) {
            const double2 t = row[j];
            v[2 * j] += t.x;
            v[2 * j + 1] += t.y;
        }
    }
    block_sum8<NT>(v, red);
}

// One launch's operands: the set it reads, the set it writes.
struct Pcg1Args {
    double* x;
    const double *r, *p, *q, *dinv;
    double *rn, *pn, *qn;
    const Pcg1State* s;
    Pcg1State* sn;
    const double* part;
    double* partn;
    int nb;  // rows of part and partn: the grid of the start kernel and of every launch
};

// r = b - Ax (Ax may be null: x = 0), p = 0, nb rows of (r.z, r.r) into part.
hipError_t launch_pcg1_start(int64_t n, const double* b, const double* Ax, const double* dinv,
                             double* r, double* p, double* part, int nb, hipStream_t s);

// EnergyCriteria check on the current iterate (x, r = f - Ax): partial sums
// of x.r and f.x over kVecBlocks blocks into `partials`, then one block sets
// ec and, when converged or on a domain error, sc->done (before the next
// launch applies the pending update).  No-op once done.
hipError_t launch_energy_check(int64_t n, const double* x, const double* r, const double* f,
                               Pcg1State* sc, EnergyCrit* ec, double* partials, hipStream_t s);

// One iteration on the elasticity operator (k_pcg1.hip); a.nb = pcg1_blocks(g).
int pcg1_blocks(const Grid& g);
hipError_t launch_pcg1(const Grid& g, const ElemOp<double>& op, const uint8_t* fixmask,
                       const double* E, double meandiag, const Pcg1Args& a, hipStream_t s);

// y = K x on the assembled matrix, whose row pattern is the grid's (k_csr.hip).
hipError_t launch_csr_spmv(const Grid& g, const int64_t* rowptr, const double* vals,
                           const double* x, double* y, hipStream_t s);
// One PCG iteration on it: the vectors in place from the state st and the product's
// sums in part (csr_pcg1_blocks rows), then q = K p with the next sums; stn is the
// state left.
int csr_pcg1_blocks(const Grid& g);
hipError_t launch_csr_pcg1(const Grid& g, const int64_t* rowptr, const double* vals, double* x,
                           double* r, double* p, double* q, const double* dinv,
                           const Pcg1State* st, Pcg1State* stn, double* part, hipStream_t s);

// Launches the graph that sch names, as often as it says, and brings st[0] to *h; sch
// then has what comes next unless the solve is done.
inline hipError_t pcg1_replay(hipGraphExec_t graph, Pcg1Schedule& sch, const Pcg1State* st,
                              Pcg1State* h, hipStream_t s, int64_t* syncs, int64_t* graphs) {
    hipError_t e;
    for (int l = 0; l < sch.launches; ++l)
        if ((e = hipGraphLaunch(graph, s)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(h, st, sizeof(Pcg1State), hipMemcpyDeviceToHost, s)) != hipSuccess)
        return e;
    if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
    *syncs += 1;
    *graphs += sch.launches;
    if (!h->done) sch.next(h->iter, h->maxiter, h->rr, h->rr0, h->tol);
    return hipSuccess;
}

}  // namespace tohip
