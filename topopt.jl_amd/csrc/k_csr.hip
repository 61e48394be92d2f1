// Assembled stiffness matrix in CSR on the device: the comparator of the
// matrix-free operator, TopOpt.jl's CGAssemblySolver
// (src/FEA/solvers_api.jl:223-250; assemble!, src/TopOptProblems/
// assemble.jl:28-90, then Ferrite's apply!).
//
// Row 3n+d (node-major DOFs) holds, for every node m of the 3x3x3 block
// around n inside the grid (ascending node id) and every component e, the
// entry K[3n+d][3m+e] = sum over the cells containing n and m of
// rho_c Ke[(3a+d)][(3b+e)] (a, b the corner bit indices of n, m in c); the
// structural pattern is kept for prescribed rows and columns, whose entries
// are zero except the diagonal = mean |diag K| of the unconstrained matrix
// (apply!).  Each (node, neighbour) pair is assembled by one thread as a
// dim x dim block: no atomics, deterministic.
//
#include <algorithm>

#include "k_pcg1.h"

namespace tohip {

// The PCG operands of k_csr_spmv.
struct CsrPcgArgs {
    const double *r, *dinv;
    const Pcg1State* st;
    double* part;
};

// Valid neighbour offsets of node (i, j, k) in ascending node order; returns
// the count and, when o >= 0, the slot of offset o in *slot (-1 if invalid).
template <int DIM>
__device__ __forceinline__ int csr_neighbours(const Grid& g, int i, int j, int k, int o,
                                              int* slot) {
    int cnt = 0;
    if (slot) *slot = -1;
    for (int dz = (DIM == 3 ? -1 : 0); dz <= (DIM == 3 ? 1 : 0); ++dz)
        for (int dy = -1; dy <= 1; ++dy)
            for (int dx = -1; dx <= 1; ++dx) {
                const int oo = (dx + 1) + 3 * ((dy + 1) + 3 * (DIM == 3 ? dz + 1 : 0));
                const int mi = i + dx, mj = j + dy, mk = k + dz;
                const bool ok = mi >= 0 && mi < g.NX && mj >= 0 && mj < g.NY &&
                                (DIM == 2 || (mk >= 0 && mk < g.NZ));
                if (!ok) continue;
                if (slot && oo == o) *slot = cnt;
                ++cnt;
            }
    return cnt;
}

template <int DIM>
__global__ void k_csr_cols(Grid g, const int64_t* __restrict__ rowptr, int* __restrict__ cols) {
    for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n < g.nnodes;
         n += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(n % g.NX), j = (int)((n / g.NX) % g.NY);
        const int k = DIM == 3 ? (int)(n / ((int64_t)g.NX * g.NY)) : 0;
        int s = 0;
        for (int dz = (DIM == 3 ? -1 : 0); dz <= (DIM == 3 ? 1 : 0); ++dz)
            for (int dy = -1; dy <= 1; ++dy)
                for (int dx = -1; dx <= 1; ++dx) {
                    const int mi = i + dx, mj = j + dy, mk = k + dz;
                    if (mi < 0 || mi >= g.NX || mj < 0 || mj >= g.NY ||
                        (DIM == 3 && (mk < 0 || mk >= g.NZ)))
                        continue;
                    const int64_t m = mi + (int64_t)g.NX * (mj + (int64_t)g.NY * mk);
                    for (int d = 0; d < DIM; ++d)
                        for (int e = 0; e < DIM; ++e)
                            cols[rowptr[DIM * n + d] + DIM * s + e] = (int)(DIM * m + e);
                    ++s;
                }
    }
}

// Unconstrained diagonal of K (per DOF) and per-block partials of
// (sum |diag|, sum |diag| over prescribed DOFs, number of prescribed DOFs).
template <int DIM>
__global__ __launch_bounds__(kThreads) void k_csr_diag(Grid g, const double* __restrict__ Ke,
                                                       const double* __restrict__ E,
                                                       const uint8_t* __restrict__ fixmask,
                                                       double* __restrict__ diag,
                                                       double* __restrict__ partials) {
    __shared__ double red[kWaves];
    constexpr int ND = DIM << DIM;
    double acc = 0.0, accf = 0.0, nf = 0.0;
    for (int64_t n = blockIdx.x * (int64_t)kThreads + threadIdx.x; n < g.nnodes;
         n += (int64_t)gridDim.x * kThreads) {
        const int i = (int)(n % g.NX), j = (int)((n / g.NX) % g.NY);
        const int k = DIM == 3 ? (int)(n / ((int64_t)g.NX * g.NY)) : 0;
        double dv[DIM];
        for (int d = 0; d < DIM; ++d) dv[d] = 0.0;
        for (int cz = (DIM == 3 ? k - 1 : 0); cz <= (DIM == 3 ? k : 0); ++cz) {
            if (DIM == 3 && (cz < 0 || cz >= g.nz)) continue;
            for (int cy = j - 1; cy <= j; ++cy) {
                if (cy < 0 || cy >= g.ny) continue;
                for (int cx = i - 1; cx <= i; ++cx) {
                    if (cx < 0 || cx >= g.nx) continue;
                    const double ec = E[cx + (int64_t)g.nx * (cy + (int64_t)g.ny * cz)];
                    const int a = (i - cx) + 2 * (j - cy) + (DIM == 3 ? 4 * (k - cz) : 0);
                    for (int d = 0; d < DIM; ++d) dv[d] += ec * Ke[(DIM * a + d) * ND + DIM * a + d];
                }
            }
        }
        const uint8_t fm = fixmask[n];
        for (int d = 0; d < DIM; ++d) {
            diag[DIM * n + d] = dv[d];
            acc += fabs(dv[d]);
            if ((fm >> d) & 1) {
                accf += fabs(dv[d]);
                nf += 1.0;
            }
        }
    }
    const double s0 = block_sum_all(acc, red);
    const double s1 = block_sum_all(accf, red);
    const double s2 = block_sum_all(nf, red);
    if (threadIdx.x == 0) {
        partials[3 * (size_t)blockIdx.x] = s0;
        partials[3 * (size_t)blockIdx.x + 1] = s1;
        partials[3 * (size_t)blockIdx.x + 2] = s2;
    }
}

// apply!'s prescribed diagonal: mean |diag| of the unconstrained K; the safe
// value: mean |diag| of K after apply! (solvers_api.jl:232-239 runs after it).
__device__ __forceinline__ void csr_diag_values(const double* md, int64_t ndof, double& m_apply,
                                                double& m_safe) {
    m_apply = md[0] / (double)ndof;
    m_safe = (md[0] - md[1] + md[2] * m_apply) / (double)ndof;
}

// One thread per (node n, neighbour offset o): the dim x dim block K[n][m].
// mdiag_sum: the three sums of k_csr_diag (see csr_diag_values).
template <int DIM>
__global__ void k_csr_values(Grid g, const double* __restrict__ Ke, const double* __restrict__ E,
                             const uint8_t* __restrict__ fixmask,
                             const int64_t* __restrict__ rowptr,
                             const double* __restrict__ mdiag_sum, int safe,
                             double* __restrict__ vals) {
    constexpr int NO = DIM == 3 ? 27 : 9;
    constexpr int ND = DIM << DIM;
    double md, msafe;
    csr_diag_values(mdiag_sum, g.ndof, md, msafe);
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < g.nnodes * NO;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t n = t / NO;
        const int o = (int)(t % NO);
        const int dx = o % 3 - 1, dy = (o / 3) % 3 - 1, dz = DIM == 3 ? o / 9 - 1 : 0;
        const int i = (int)(n % g.NX), j = (int)((n / g.NX) % g.NY);
        const int k = DIM == 3 ? (int)(n / ((int64_t)g.NX * g.NY)) : 0;
        const int mi = i + dx, mj = j + dy, mk = k + dz;
        if (mi < 0 || mi >= g.NX || mj < 0 || mj >= g.NY || (DIM == 3 && (mk < 0 || mk >= g.NZ)))
            continue;
        int slot;
        csr_neighbours<DIM>(g, i, j, k, o, &slot);
        const int64_t m = mi + (int64_t)g.NX * (mj + (int64_t)g.NY * mk);
        double blk[DIM][DIM];
        for (int d = 0; d < DIM; ++d)
            for (int e = 0; e < DIM; ++e) blk[d][e] = 0.0;
        for (int cz = (DIM == 3 ? k - 1 : 0); cz <= (DIM == 3 ? k : 0); ++cz) {
            if (DIM == 3 && (cz < 0 || cz >= g.nz)) continue;
            for (int cy = j - 1; cy <= j; ++cy) {
                if (cy < 0 || cy >= g.ny) continue;
                for (int cx = i - 1; cx <= i; ++cx) {
                    if (cx < 0 || cx >= g.nx) continue;
                    const int bx = mi - cx, by = mj - cy, bz = DIM == 3 ? mk - cz : 0;
                    if (bx < 0 || bx > 1 || by < 0 || by > 1 || bz < 0 || bz > 1) continue;
                    const double ec = E[cx + (int64_t)g.nx * (cy + (int64_t)g.ny * cz)];
                    const int a = (i - cx) + 2 * (j - cy) + (DIM == 3 ? 4 * (k - cz) : 0);
                    const int b = bx + 2 * by + 4 * bz;
                    for (int d = 0; d < DIM; ++d)
                        for (int e = 0; e < DIM; ++e)
                            blk[d][e] += ec * Ke[(DIM * a + d) * ND + DIM * b + e];
                }
            }
        }
        const uint8_t fn = fixmask[n], fm = fixmask[m];
        for (int d = 0; d < DIM; ++d)
            for (int e = 0; e < DIM; ++e) {
                double v = blk[d][e];
                const bool diag = m == n && d == e;
                if (((fn >> d) & 1) || ((fm >> e) & 1)) v = diag ? md : 0.0;
                else if (safe && diag && v == 0.0) v = msafe;
                vals[rowptr[DIM * n + d] + DIM * slot + e] = v;
            }
    }
}

// dinv = 1 / diag(K after apply!) (jacobi), or 1 (identity preconditioner).
template <int DIM>
__global__ void k_csr_dinv(int64_t ndof, const double* __restrict__ diag,
                           const uint8_t* __restrict__ fixmask,
                           const double* __restrict__ mdiag_sum, int jacobi, int safe,
                           double* __restrict__ dinv) {
    double md, msafe;
    csr_diag_values(mdiag_sum, ndof, md, msafe);
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < ndof;
         i += (int64_t)gridDim.x * blockDim.x) {
        if (!jacobi) {
            dinv[i] = 1.0;
            continue;
        }
        const bool fixed = (fixmask[i / DIM] >> (i % DIM)) & 1;
        double d = fixed ? md : diag[i];
        if (safe && !fixed && d == 0.0) d = msafe;
        dinv[i] = 1.0 / d;
    }
}

// y = K x by nodes.  A group of 32 lanes (16 in 2D) takes four consecutive nodes:
// lane o holds neighbour offset o of each, so it loads x at that neighbour once
// for the node's D rows and its D x D block from them (D consecutive values a row,
// the rows of a node contiguous: coalesced).  The neighbour and the slot of its
// block follow from the grid, so the columns are not read: 8 bytes an entry
// instead of 12.  The 4 D row sums of a group come out of one reduce-scatter
// (lanes keep the half of the values that a lane bit selects) in place of a tree
// a row.
//
// PCG: x = p, with the sums of the one-launch iteration (k_pcg1.h) at the rows a
// lane owns; on a state without a pending update only (r.z, r.r).
// Bound by the matrix, 1.9 KB a node in 3D: at 60x20x20 (52 MB, in the last-level
// cache) an iteration with the vector kernel takes 19.8 us, against 32 for a
// direction, a product of 16 lanes a row over values and columns, and an update.
// Two nodes a group (5 waves per SIMD instead of 4): 21.1 us; row starts in closed
// form instead of the row pointers: 20.3.
constexpr int kCsrNodes = 4;  // nodes of one group
template <int DIM>
constexpr int csr_group = DIM == 3 ? 32 : 16;
template <int DIM, bool PCG>
__global__ __launch_bounds__(kThreads) void k_csr_spmv(Grid g, const int64_t* __restrict__ rowptr,
                                                       const double* __restrict__ vals,
                                                       const double* __restrict__ x,
                                                       double* __restrict__ y, CsrPcgArgs a) {
    constexpr int G = csr_group<DIM>, NV = DIM == 3 ? 16 : 8, DV = NV / kCsrNodes;
    __shared__ double red[kWaves][kPcg1Vals];
    double sum[kPcg1Vals] = {0, 0, 0, 0, 0, 0, 0, 0};
    const int lane = threadIdx.x & (G - 1);
    const int ox = lane % 3 - 1, oy = (lane / 3) % 3 - 1, oz = DIM == 3 ? lane / 9 - 1 : 0;
    const bool used = lane < (DIM == 3 ? 27 : 9);
    bool step = true;
    if (PCG) {
        if (a.st->done) return;
        step = a.st->pend != 0;
    }
    const int64_t per = kThreads / G * kCsrNodes;  // nodes a workgroup takes at a time
    for (int64_t n0 = blockIdx.x * per + threadIdx.x / G * kCsrNodes; n0 < g.nnodes;
         n0 += gridDim.x * per) {
        double t[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) t[v] = 0.0;
        if (!PCG || step) {
            double xv[kCsrNodes][DIM], kv[kCsrNodes][DIM][DIM];
            bool on[kCsrNodes];
#pragma unroll
            for (int q = 0; q < kCsrNodes; ++q) {
                const uint32_t n = (uint32_t)(n0 + q < g.nnodes ? n0 + q : n0);
                const int i = (int)(n % (uint32_t)g.NX), jk = (int)(n / (uint32_t)g.NX);
                const int j = DIM == 3 ? jk % g.NY : jk, k = DIM == 3 ? jk / g.NY : 0;
                const int x0 = i > 0 ? -1 : 0, y0 = j > 0 ? -1 : 0, z0 = DIM == 3 && k > 0 ? -1 : 0;
                const int cx = 1 - x0 + (i < g.NX - 1), cy = 1 - y0 + (j < g.NY - 1),
                          cz = DIM == 3 ? 1 - z0 + (k < g.NZ - 1) : 1;
                on[q] = used && n0 + q < g.nnodes && ox >= x0 && ox < x0 + cx && oy >= y0 &&
                        oy < y0 + cy && oz >= z0 && oz < z0 + cz;
                const int slot = on[q] ? (ox - x0) + cx * ((oy - y0) + cy * (oz - z0)) : 0;
                const uint32_t m = on[q] ? n + ox + g.NX * (oy + g.NY * oz) : n;
                const double* row = vals + rowptr[DIM * (int64_t)n] + DIM * slot;
                const int len = DIM * cx * cy * cz;
                ld_node<DIM>(x, m, xv[q]);
#pragma unroll
                for (int d = 0; d < DIM; ++d)
#pragma unroll
                    for (int e = 0; e < DIM; ++e) kv[q][d][e] = row[d * len + e];
            }
#pragma unroll
            for (int q = 0; q < kCsrNodes; ++q)
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    double s = 0.0;
#pragma unroll
                    for (int e = 0; e < DIM; ++e) s += kv[q][d][e] * xv[q][e];
                    t[q * DV + d] = on[q] ? s : 0.0;
                }
            // value v of the group ends up in lanes v G / NV ...
            auto halve = [&](auto half, int bit) {
                constexpr int h = decltype(half)::value;
                const bool up = (lane & bit) != 0;
#pragma unroll
                for (int v = 0; v < h; ++v) {
                    const double keep = up ? t[v + h] : t[v], send = up ? t[v] : t[v + h];
                    t[v] = keep + __shfl_xor(send, bit, 64);
                }
            };
            if constexpr (DIM == 3) halve(std::integral_constant<int, 8>{}, 16);
            halve(std::integral_constant<int, 4>{}, 8);
            halve(std::integral_constant<int, 2>{}, 4);
            halve(std::integral_constant<int, 1>{}, 2);
            t[0] += __shfl_xor(t[0], 1, 64);
        }
        const int v = lane >> 1, q = v / DV, d = v % DV;
        if ((lane & 1) == 0 && d < DIM && n0 + q < g.nnodes) {
            const int64_t i = DIM * (n0 + q) + d;
            if (PCG) {
                const double r = a.r[i], z = a.dinv[i] * r;
                sum[kSumRZ] += z * r;
                sum[kSumRR] += r * r;
                if (step) {
                    const double s = t[0];
                    y[i] = s;
                    sum[kSumPQ] += x[i] * s;
                    sum[kSumQZ] += z * s;
                    sum[kSumQDQ] += a.dinv[i] * s * s;
                    sum[kSumRQ] += r * s;
                    sum[kSumQQ] += s * s;
                }
            } else {
                y[i] = t[0];
            }
        }
    }
    if (PCG) pcg1_store_sums(sum, red, a.part);
}

// The vector part of an iteration, in place: x += alpha p, r -= alpha q,
// p = z + beta p (or the update alone, kPcg1Exact), from the product's sums.
__global__ __launch_bounds__(kThreads) void k_csr_vectors(int64_t n, double* __restrict__ x,
                                                          double* __restrict__ r,
                                                          double* __restrict__ p,
                                                          const double* __restrict__ q,
                                                          const double* __restrict__ dinv,
                                                          const Pcg1State* s, Pcg1State* sn,
                                                          const double* __restrict__ part,
                                                          int nb) {
    __shared__ double red[kWaves][kPcg1Vals];
    const int64_t i0 = blockIdx.x * (int64_t)kThreads + threadIdx.x;
    const int64_t stride = gridDim.x * (int64_t)kThreads;
    // the first element's loads are in flight while the sums are formed
    const int64_t ic = i0 < n ? i0 : 0;
    double cx = x[ic], cr = r[ic], cp = p[ic], cq = q[ic], cd = dinv[ic];
    const Pcg1State s0 = *s;
    if (s0.done) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *sn = s0;
        return;
    }
    double v[kPcg1Vals];
    pcg1_reduce<kThreads>(part, nb, v, red);
    Pcg1State s1;
    const Pcg1Plan plan = pcg1_plan(s0, v, s1);
    if (blockIdx.x == 0 && threadIdx.x == 0) *sn = s1;
    if (s1.err != 0 && s0.iter == s1.iter) return;
    const bool pend = s0.pend != 0;
    for (int64_t i = i0; i < n; i += stride) {
        if (i != i0) {
            cx = x[i];
            cr = r[i];
            cp = p[i];
            cq = q[i];
            cd = dinv[i];
        }
        if (pend) {
            x[i] = cx + plan.alpha * cp;
            cr = fma(-plan.alpha, cq, cr);
            if (plan.mode != kPcg1Stop) r[i] = cr;
        }
        if (plan.mode == kPcg1Step) p[i] = fma(plan.beta, cp, cd * cr);
    }
}

static unsigned csr_blocks(int64_t work, int per_block) {
    int64_t b = (work + per_block - 1) / per_block;
    if (b > kMaxPartials) b = kMaxPartials;
    if (b < 1) b = 1;
    return (unsigned)b;
}

hipError_t launch_csr_build(const Grid& g, const double* Ke, const double* E,
                            const uint8_t* fixmask, const int64_t* rowptr, int* cols, int safe,
                            double* vals, double* diag, double* partials, double* mdiag_sum,
                            bool pattern, hipStream_t s) {
    const unsigned nbn = csr_blocks(g.nnodes, kThreads);
    if (pattern) {
        if (g.dim == 3)
            hipLaunchKernelGGL((k_csr_cols<3>), dim3(nbn), dim3(kThreads), 0, s, g, rowptr, cols);
        else
            hipLaunchKernelGGL((k_csr_cols<2>), dim3(nbn), dim3(kThreads), 0, s, g, rowptr, cols);
    }
    if (g.dim == 3)
        hipLaunchKernelGGL((k_csr_diag<3>), dim3(nbn), dim3(kThreads), 0, s, g, Ke, E, fixmask,
                           diag, partials);
    else
        hipLaunchKernelGGL((k_csr_diag<2>), dim3(nbn), dim3(kThreads), 0, s, g, Ke, E, fixmask,
                           diag, partials);
    hipError_t e = launch_reduce(partials, (int)nbn, 3, mdiag_sum, s);
    if (e != hipSuccess) return e;
    const int no = g.dim == 3 ? 27 : 9;
    const unsigned nbv = csr_blocks(g.nnodes * no, kThreads);
    if (g.dim == 3)
        hipLaunchKernelGGL((k_csr_values<3>), dim3(nbv), dim3(kThreads), 0, s, g, Ke, E, fixmask,
                           rowptr, mdiag_sum, safe, vals);
    else
        hipLaunchKernelGGL((k_csr_values<2>), dim3(nbv), dim3(kThreads), 0, s, g, Ke, E, fixmask,
                           rowptr, mdiag_sum, safe, vals);
    return hipGetLastError();
}

hipError_t launch_csr_dinv(const Grid& g, const double* diag, const uint8_t* fixmask,
                           const double* mdiag_sum, int jacobi, int safe, double* dinv,
                           hipStream_t s) {
    const unsigned nb = csr_blocks(g.ndof, kThreads);
    if (g.dim == 3)
        hipLaunchKernelGGL((k_csr_dinv<3>), dim3(nb), dim3(kThreads), 0, s, g.ndof, diag, fixmask,
                           mdiag_sum, jacobi, safe, dinv);
    else
        hipLaunchKernelGGL((k_csr_dinv<2>), dim3(nb), dim3(kThreads), 0, s, g.ndof, diag, fixmask,
                           mdiag_sum, jacobi, safe, dinv);
    return hipGetLastError();
}

static unsigned csr_spmv_blocks(const Grid& g) {
    const int group = g.dim == 3 ? csr_group<3> : csr_group<2>;
    return std::min(csr_blocks(g.nnodes, kThreads / group * kCsrNodes), 2048u);
}
int csr_pcg1_blocks(const Grid& g) { return (int)csr_spmv_blocks(g); }

hipError_t launch_csr_spmv(const Grid& g, const int64_t* rowptr, const double* vals,
                           const double* x, double* y, hipStream_t s) {
    const dim3 grid(csr_spmv_blocks(g)), block(kThreads);
    const CsrPcgArgs a{};
    if (g.dim == 3)
        hipLaunchKernelGGL((k_csr_spmv<3, false>), grid, block, 0, s, g, rowptr, vals, x, y, a);
    else
        hipLaunchKernelGGL((k_csr_spmv<2, false>), grid, block, 0, s, g, rowptr, vals, x, y, a);
    return hipGetLastError();
}

hipError_t launch_csr_pcg1(const Grid& g, const int64_t* rowptr, const double* vals, double* x,
                           double* r, double* p, double* q, const double* dinv,
                           const Pcg1State* st, Pcg1State* stn, double* part, hipStream_t s) {
    const dim3 grid(csr_spmv_blocks(g)), block(kThreads);
    const unsigned nv = std::min(csr_blocks(g.ndof, kThreads), 1024u);
    hipLaunchKernelGGL(k_csr_vectors, dim3(nv), block, 0, s, g.ndof, x, r, p, q, dinv, st, stn,
                       part, (int)grid.x);
    const CsrPcgArgs a{r, dinv, stn, part};
    if (g.dim == 3)
        hipLaunchKernelGGL((k_csr_spmv<3, true>), grid, block, 0, s, g, rowptr, vals, p, q, a);
    else
        hipLaunchKernelGGL((k_csr_spmv<2, true>), grid, block, 0, s, g, rowptr, vals, p, q, a);
    return hipGetLastError();
}

}  // namespace tohip
