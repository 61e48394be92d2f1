// Heat conduction on the device: the scalar counterpart of the elasticity
// operator (TopOpt.jl src/TopOptProblems/matrices_and_vectors.jl:413-496 for
// the element conductivity matrix, src/FEA/matrix_free_operator.jl:66-105
// for the matrix-free product and its fixed-DOF rule).
//
// One DOF per node; K = sum_e rho_e Ke with one shared Ke (k * grad phi_a .
// grad phi_b integrated over the box cell).  Ke is a sum of Kronecker products
// of 1D stiffness and mass matrices, which the +-1 (Hadamard) basis of the
// corners diagonalises: Ke = H B H^T with B diagonal.
#include <algorithm>

#include "heat_internal.h"
#include "k_common.h"

namespace tohip {

// Ferrite corner index of the corner at offset (ox, oy, oz) of its cell.
__device__ __forceinline__ int heat_corner(int ox, int oy, int oz) {
    return (oy ? (ox ? 2 : 3) : (ox ? 1 : 0)) + 4 * oz;
}

// ---- the operator, alone and inside one-launch PCG ----
//
// A 256-thread workgroup owns a column of 15 x 15 output nodes and, in 3D, a
// chunk of node planes that it walks upwards; 2D is one plane.  Thread (ci, cj)
// stages node (ci, cj) of the column's 17 x 17 nodes (a one-node halo; threads
// 0..32 the far row and column too) and handles cell (ci, cj) of the 16 x 16
// cells.  Per plane: values to LDS with prescribed nodes zeroed; each thread
// transforms its cell's four nodes to the xy Hadamard basis; the layer's cells
// are the sum and difference with the transform of the plane below, scaled by
// E B; the part of the upper plane stays in registers, the lower plane's total
// is transformed back.  A node's four cell columns are summed as two x-pairs (a
// DPP row shift brings the left cell's value, a row of 16 lanes is a row of
// cells) and an LDS exchange between the rows: lower row first.  No atomics,
// the same bits every run.  About 50 FP64 operations and 7 LDS accesses a cell
// in place of 64 products and 27 bounds-tested loads a node.
//
// One launch is a whole PCG iteration.  Bound by latency on small grids, by the
// cache traffic of its vectors on larger ones: p, r, q, D^-1 in with the halo (1.3 x
// (zc + 2) / zc), x in and x, r, p, q out at the owner.  MI355X, one iteration:
// 128x96x80 22.4 us (direction, a 27-point gather of K p and update in three
// launches: 85 us; the 82 MB it must move take 17 us at the copy rate), 80x60 5.0 us
// (14 us).
constexpr int kHC = 16, kHO = kHC - 1, kHS = kHC + 1;

// Columns of 15 x 15 nodes and chunks of zc planes, about 768 workgroups when the
// grid has them.  Fewer planes a chunk fill the chip better but re-stage more (zc + 2
// planes each): a PCG iteration at 128x96x80 takes 23.8 us with 756 workgroups, 26.0
// with 1008.
struct HeatShape {
    int ncx, ncy, zc, nch, nwork;
};
static HeatShape heat_shape(const HeatGrid& g) {
    HeatShape s;
    s.ncx = (g.NX + kHO - 1) / kHO;
    s.ncy = (g.NY + kHO - 1) / kHO;
    const int64_t cols = (int64_t)s.ncx * s.ncy;
    const int64_t want = std::max<int64_t>(1, 768 / cols);
    s.zc = (int)std::max<int64_t>(std::min(2, g.NZ), (g.NZ + want - 1) / want);
    s.nch = (g.NZ + s.zc - 1) / s.zc;
    s.nwork = (int)(cols * s.nch);
    return s;
}
// Workgroups of the operator alone, and of a PCG iteration, where every workgroup
// sums every workgroup's row of partials: no more than run at once (three per CU), the
// rest of the work strided over.  MI355X, us an iteration with at most 512 / 768 / 1024
// / 4096 workgroups, and of three launches: 640x320 9.6 / 10.4 / 11.2 / 11.2 and 18.5,
// 1000x990 24 / 22 / 29 / 91 and 44, 2400x2400 144 / 134 / 162 / 199 and 198, 900x900x2
// 52 / 49 / 55 / 88 and 150.
constexpr int kHeatPcgBlocks = 768;
static int heat_op_blocks(const HeatShape& s, bool pcg) {
    return std::min(s.nwork, pcg ? kHeatPcgBlocks : kMaxPartials);
}
int heat_pcg_blocks(const HeatGrid& g) { return heat_op_blocks(heat_shape(g), true); }

// A staged node's operands.
struct HeatNode {
    double v, r, q, d;  // MODE 1: v = p; otherwise v = x
    uint8_t m;
};

// MODE 0: y = K x (prescribed nodes masked, their rows md x); MODE 1: one
// PCG iteration (k_pcg1.h); MODE 2: y = K_full x (no masking).
// LOOP: more work than workgroups.
template <int DIM, int MODE, typename Off, bool LOOP>
__global__ __launch_bounds__(kThreads) void k_heat_op(HeatGrid g, HeatModes B, HeatShape sh,
                                                      const double* __restrict__ xin,
                                                      const uint8_t* __restrict__ fixmask,
                                                      const double* __restrict__ E, double md,
                                                      double* __restrict__ y, Pcg1Args a) {
    __shared__ double pl[2][kHS * kHS];
    __shared__ double exch[kThreads];
    __shared__ double red[kWaves][kPcg1Vals];
    const int tid = threadIdx.x, ci = tid & (kHC - 1), cj = tid / kHC;
    // the second node of threads 0..32: the far column, then the far row
    const bool two = tid < 2 * kHC + 1;
    const int li2 = tid <= kHC ? kHC : tid - kHS, lj2 = tid <= kHC ? tid : kHC;
    Pcg1Plan plan{0.0, 0.0, kPcg1Step};
    bool pend = false, update = true;  // an update is pending; and may be applied

    // A node's (cell's) place: a base that is the same for the whole workgroup,
    // advanced by a plane a step, and an offset in bytes within the column's
    // plane that stays, so that an access costs no vector address arithmetic.
    int i0 = 0, j0 = 0;
    Off oa = 0, ob = 0, oe = 0;  // of the two nodes and the cell
    auto at64 = [](auto* p, int64_t base, Off o) -> auto& {
        using T = std::remove_pointer_t<decltype(p)>;
        using C = std::conditional_t<std::is_const<T>::value, const char, char>;
        return *reinterpret_cast<T*>(reinterpret_cast<C*>(p + base) + o);
    };
    bool ina = false, inb = false, ine = false;
    int64_t nbase = 0, ebase = 0;
    auto load = [&](Off o, int k) {
        const int nk = DIM == 3 ? min(max(k, 0), g.NZ - 1) : 0;
        const int64_t base = nbase + (int64_t)nk * g.NX * g.NY;
        HeatNode h;
        h.m = MODE == 2 ? 0 : at64(fixmask, base, o / 8);
        if (MODE == 1) {
            h.v = at64(a.p, base, o);
            h.r = at64(a.r, base, o);
            h.q = at64(a.q, base, o);
            h.d = at64(a.dinv, base, o);
        } else {
            h.v = at64(xin, base, o);
        }
        return h;
    };
    auto load_E = [&](int k) {  // the cell of this thread in layer k
        const int ck = DIM == 3 ? min(max(k, 0), g.nz - 1) : 0;
        const int64_t base = ebase + (int64_t)ck * g.nx * g.ny;
        return at64(E, base, oe);
    };
    double sum[kPcg1Vals] = {0, 0, 0, 0, 0, 0, 0, 0};
    int buf = 0;
    bool first = true;
    for (int w = blockIdx.x; w < sh.nwork; w += gridDim.x) {
        const int wr = xcd_remap(w, sh.nwork);
        const int ncol = sh.ncx * sh.ncy, col = wr % ncol, ch = wr / ncol;
        i0 = (col % sh.ncx) * kHO;
        j0 = (col / sh.ncx) * kHO;
        const int kb = DIM == 3 ? ch * sh.zc : 0, ke = DIM == 3 ? min(kb + sh.zc, g.NZ) : 1;
        const int gi = i0 - 1 + ci, gj = j0 - 1 + cj;
        const bool mine = ci >= 1 && cj >= 1 && gi < g.NX && gj < g.NY;
        {
            const int bi = max(i0 - 1, 0), bj = max(j0 - 1, 0);
            auto place = [&](int li, int lj, bool& in) {
                const int x = i0 - 1 + li, y = j0 - 1 + lj;
                const int cx = min(max(x, 0), g.NX - 1), cy = min(max(y, 0), g.NY - 1);
                in = x == cx && y == cy;
                return 8 * ((Off)(cx - bi) + (Off)g.NX * (Off)(cy - bj));
            };
            nbase = bi + (int64_t)g.NX * bj;
            ebase = bi + (int64_t)g.nx * bj;
            oa = place(ci, cj, ina);
            ob = place(two ? li2 : 0, two ? lj2 : 0, inb);
            ine = gi >= 0 && gi < g.nx && gj >= 0 && gj < g.ny;
            oe = ine ? 8 * ((Off)(gi - bi) + (Off)g.nx * (Off)(gj - bj)) : 0;
        }
        auto plane = [&](int k) { return nbase + (int64_t)(DIM == 3 ? k : 0) * g.NX * g.NY; };
        const int sb = DIM == 3 ? kb - 1 : 0, se = DIM == 3 ? ke : 0;  // staged planes
        HeatNode na = load(oa, sb), nb{};
        if (two) nb = load(ob, sb);
        double xa = 0.0;
        if (MODE == 1 && mine && sb >= kb) xa = at64(a.x, plane(sb), oa);
        double en = DIM == 3 ? 0.0 : load_E(0);
        if (MODE == 1 && first) {
            // the first plane's loads are in flight while the sums are formed
            first = false;
            const Pcg1State s0 = *a.s;
            if (s0.done) {
                if (blockIdx.x == 0 && tid == 0) *a.sn = s0;
                return;
            }
            double v[kPcg1Vals];
            pcg1_reduce<kThreads>(a.part, a.nb, v, red);
            Pcg1State s1;
            plan = pcg1_plan(s0, v, s1);
            if (blockIdx.x == 0 && tid == 0) *a.sn = s1;
            pend = s0.pend != 0;
            update = s1.err == 0 || s0.iter != s1.iter;
        }
        if (MODE == 1 && plan.mode != kPcg1Step) {
            // the pending update alone: x, and (exact) r with its two sums
            if (update) {
                for (int k = kb; k < ke; ++k) {
                    if (!mine) break;
                    const int64_t n = plane(k);
                    const double p = at64(a.p, n, oa);
                    if (pend) at64(a.x, n, oa) += plan.alpha * p;
                    if (plan.mode == kPcg1Exact) {
                        const double r = fma(-plan.alpha, at64(a.q, n, oa), at64(a.r, n, oa));
                        at64(a.rn, n, oa) = r;
                        at64(a.pn, n, oa) = p;
                        sum[kSumRZ] += at64(a.dinv, n, oa) * r * r;
                        sum[kSumRR] += r * r;
                    }
                }
            }
            if (LOOP) continue;
            break;
        }
        double fp[4] = {0, 0, 0, 0}, up[4] = {0, 0, 0, 0};
        double po = 0.0, ro = 0.0, dd = 0.0;  // own node of the plane below
        uint8_t mo = 0;
        for (int k = sb; k <= se; ++k) {
            // direction (or input) of this plane, then the next plane's loads
            // (what lies outside the mesh is put to 0 here, not where it is
            // loaded: a select there would wait for the whole prefetch)
            const bool kin = DIM == 2 || (k >= 0 && k < g.NZ);
            auto value = [&](HeatNode& h, bool in) {
                if (MODE == 1) {
                    // explicit FMAs: a halo copy and its owner get the same bits
                    h.r = fma(-plan.alpha, pend ? h.q : 0.0, h.r);
                    h.v = fma(plan.beta, h.v, h.d * h.r);
                }
                return (in && kin && !h.m) ? h.v : 0.0;
            };
            const double pold = na.v;
            const double va = value(na, ina);
            pl[buf][ci + kHS * cj] = va;
            if (two) pl[buf][li2 + kHS * lj2] = value(nb, inb);
            if (MODE == 1 && mine && k >= kb && k < ke) {
                const int64_t n = plane(k);
                if (pend) at64(a.x, n, oa) = xa + plan.alpha * pold;
                at64(a.rn, n, oa) = na.r;
                at64(a.pn, n, oa) = na.v;
            }
            const double ec = ine && (DIM == 2 || (k >= 1 && k <= g.nz)) ? en : 0.0;
            const HeatNode cur = na;
            if (k < se) {
                na = load(oa, k + 1);
                if (two) nb = load(ob, k + 1);
                if (MODE == 1 && mine && k + 1 >= kb && k + 1 < ke)
                    xa = at64(a.x, plane(k + 1), oa);
                en = load_E(k);
            }
            __syncthreads();
            double f[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) f[c] = pl[buf][ci + (c & 1) + kHS * (cj + (c >> 1))];
            buf ^= 1;
            hadamard_fwd<double, 2>(f);
            if (DIM == 2 || k > sb) {
                double lo[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    if (DIM == 3) {
                        const double z0 = ec * B.b[m] * (fp[m] + f[m]);
                        const double z1 = ec * B.b[m + 4] * (f[m] - fp[m]);
                        lo[m] = up[m] + (z0 - z1);
                        up[m] = z0 + z1;
                    } else {
                        lo[m] = ec * B.b[m] * f[m];
                    }
                }
                hadamard_inv<double, 2>(lo);
                const double y0 = row_shr1(lo[1]) + lo[0];
                exch[tid] = row_shr1(lo[3]) + lo[2];
                __syncthreads();
                const int ko = DIM == 3 ? k - 1 : 0;
                if (mine && ko >= kb && ko < ke) {
                    const double p = DIM == 3 ? po : cur.v, r = DIM == 3 ? ro : cur.r,
                                 d = DIM == 3 ? dd : cur.d;
                    double q = exch[tid - kHC] + y0;
                    if (MODE != 2 && (DIM == 3 ? mo : cur.m)) q = md * p;
                    if (MODE == 1) {
                        at64(a.qn, plane(ko), oa) = q;
                        const double z = d * r, dq = d * q;
                        sum[kSumRZ] += z * r;
                        sum[kSumPQ] += p * q;
                        sum[kSumQZ] += z * q;
                        sum[kSumQDQ] += dq * q;
                        sum[kSumRR] += r * r;
                        sum[kSumRQ] += r * q;
                        sum[kSumQQ] += q * q;
                    } else {
                        at64(y, plane(ko), oa) = q;
                    }
                }
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) fp[m] = f[m];
            po = cur.v;
            ro = cur.r;
            dd = cur.d;
            mo = cur.m;
        }
        if (!LOOP) break;
    }
    if (MODE == 1) {
        pcg1_store_sums(sum, red, a.partn);
    }
}

static unsigned heat_blocks(int64_t n) {
    int64_t b = (n + kThreads - 1) / kThreads;
    if (b > kMaxPartials) b = kMaxPartials;
    if (b < 1) b = 1;
    return (unsigned)b;
}

// The kernel's 32-bit offsets span the 17 rows of a column's plane.
template <int DIM, int MODE>
static hipError_t launch_heat_op(const HeatGrid& g, const HeatModes& B, const double* x,
                                 const uint8_t* fixmask, const double* E, double meandiag,
                                 double* y, const Pcg1Args& a, hipStream_t s) {
    const HeatShape sh = heat_shape(g);
    const dim3 grid(heat_op_blocks(sh, MODE == 1)), block(kThreads);
    const bool loop = sh.nwork > (int)grid.x;
    if ((int64_t)g.NX * kHS * 8 >= ((int64_t)1 << 32))
        hipLaunchKernelGGL((k_heat_op<DIM, MODE, uint64_t, true>), grid, block, 0, s, g, B, sh, x,
                           fixmask, E, meandiag, y, a);
    else if (loop)
        hipLaunchKernelGGL((k_heat_op<DIM, MODE, uint32_t, true>), grid, block, 0, s, g, B, sh, x,
                           fixmask, E, meandiag, y, a);
    else
        hipLaunchKernelGGL((k_heat_op<DIM, MODE, uint32_t, false>), grid, block, 0, s, g, B, sh, x,
                           fixmask, E, meandiag, y, a);
    return hipGetLastError();
}

hipError_t launch_heat_matvec(const HeatGrid& g, const HeatModes& B, const double* x,
                              const uint8_t* fixmask, const double* E, double meandiag, double* y,
                              int mode, hipStream_t s) {
    const Pcg1Args a{};
    if (g.dim == 3)
        return mode == 2 ? launch_heat_op<3, 2>(g, B, x, fixmask, E, meandiag, y, a, s)
                         : launch_heat_op<3, 0>(g, B, x, fixmask, E, meandiag, y, a, s);
    return mode == 2 ? launch_heat_op<2, 2>(g, B, x, fixmask, E, meandiag, y, a, s)
                     : launch_heat_op<2, 0>(g, B, x, fixmask, E, meandiag, y, a, s);
}

hipError_t launch_heat_pcg(const HeatGrid& g, const HeatModes& B, const uint8_t* fixmask,
                           const double* E, double meandiag, const Pcg1Args& a, hipStream_t s) {
    return g.dim == 3
               ? launch_heat_op<3, 1>(g, B, nullptr, fixmask, E, meandiag, nullptr, a, s)
               : launch_heat_op<2, 1>(g, B, nullptr, fixmask, E, meandiag, nullptr, a, s);
}

__global__ void k_heat_density(int64_t ncells, const double* __restrict__ x, double xmin,
                               Penalty pen, int pbi, double* __restrict__ E) {
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < ncells;
         c += (int64_t)gridDim.x * blockDim.x) {
        double r, dr;
        rho_drho(pen, x[c], xmin, pbi, r, dr);
        E[c] = r;
    }
}

hipError_t launch_heat_density(int64_t ncells, const double* x, double xmin, const Penalty& pen,
                               int pbi, double* E, hipStream_t s) {
    hipLaunchKernelGGL(k_heat_density, dim3(heat_blocks(ncells)), dim3(kThreads), 0, s, ncells, x,
                       xmin, pen, pbi, E);
    return hipGetLastError();
}

template <int DIM>
__global__ void k_heat_diag(HeatGrid g, HeatKe ke, const uint8_t* __restrict__ fixmask,
                            const double* __restrict__ E, double md, double* __restrict__ dinv) {
    constexpr int NC = DIM == 3 ? 8 : 4;
    for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n < g.nnodes;
         n += (int64_t)gridDim.x * blockDim.x) {
        if (fixmask[n]) {
            dinv[n] = 1.0 / md;
            continue;
        }
        const int i = (int)(n % g.NX), j = (int)((n / g.NX) % g.NY);
        const int k = DIM == 3 ? (int)(n / ((int64_t)g.NX * g.NY)) : 0;
        double d = 0.0;
        for (int cz = (DIM == 3 ? k - 1 : 0); cz <= (DIM == 3 ? k : 0); ++cz) {
            if (DIM == 3 && (cz < 0 || cz >= g.nz)) continue;
            for (int cy = j - 1; cy <= j; ++cy) {
                if (cy < 0 || cy >= g.ny) continue;
                for (int cx = i - 1; cx <= i; ++cx) {
                    if (cx < 0 || cx >= g.nx) continue;
                    const int a = heat_corner(i - cx, j - cy, DIM == 3 ? k - cz : 0);
                    d += E[cx + (int64_t)g.nx * (cy + (int64_t)g.ny * cz)] * ke.k[a * NC + a];
                }
            }
        }
        dinv[n] = 1.0 / d;
    }
}

hipError_t launch_heat_diag(const HeatGrid& g, const HeatKe& ke, const uint8_t* fixmask,
                            const double* E, double meandiag, double* dinv, hipStream_t s) {
    const dim3 grid(heat_blocks(g.nnodes)), block(kThreads);
    if (g.dim == 3)
        hipLaunchKernelGGL((k_heat_diag<3>), grid, block, 0, s, g, ke, fixmask, E, meandiag, dinv);
    else
        hipLaunchKernelGGL((k_heat_diag<2>), grid, block, 0, s, g, ke, fixmask, E, meandiag, dinv);
    return hipGetLastError();
}

__global__ void k_heat_rhs(int64_t n, const double* __restrict__ q, const double* __restrict__ lift,
                           const uint8_t* __restrict__ fixmask, const double* __restrict__ v,
                           double md, int use_v, double* __restrict__ b) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        if (fixmask[i])
            b[i] = use_v ? md * v[i] : 0.0;
        else
            b[i] = q[i] - (lift ? lift[i] : 0.0);
    }
}

hipError_t launch_heat_rhs(int64_t n, const double* q, const double* lift,
                           const uint8_t* fixmask, const double* v, double meandiag, int use_v,
                           double* b, hipStream_t s) {
    hipLaunchKernelGGL(k_heat_rhs, dim3(heat_blocks(n)), dim3(kThreads), 0, s, n, q, lift, fixmask,
                       v, meandiag, use_v, b);
    return hipGetLastError();
}

template <int DIM>
__global__ void k_heat_cell_products(HeatGrid g, HeatKe ke, const double* __restrict__ lam,
                                     const double* __restrict__ T, const double* __restrict__ x,
                                     double xmin, Penalty pen, int pbi, double sign,
                                     double* __restrict__ cell, double* __restrict__ grad) {
    constexpr int NC = DIM == 3 ? 8 : 4;
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < g.ncells;
         c += (int64_t)gridDim.x * blockDim.x) {
        const int cx = (int)(c % g.nx), cy = (int)((c / g.nx) % g.ny);
        const int cz = DIM == 3 ? (int)(c / ((int64_t)g.nx * g.ny)) : 0;
        double lv[NC], tv[NC];
#pragma unroll
        for (int b = 0; b < NC; ++b) {
            const int ox = (b & 1) ^ ((b >> 1) & 1), oy = (b >> 1) & 1, oz = b >> 2;
            const int64_t m = (cx + ox) + (int64_t)g.NX * ((cy + oy) + (int64_t)g.NY * (cz + oz));
            lv[b] = lam[m];
            tv[b] = T[m];
        }
        double s = 0.0;
#pragma unroll
        for (int a = 0; a < NC; ++a) {
            double t = 0.0;
#pragma unroll
            for (int b = 0; b < NC; ++b) t += ke.k[a * NC + b] * tv[b];
            s += lv[a] * t;
        }
        double r, dr;
        rho_drho(pen, x[c], xmin, pbi, r, dr);
        cell[c] = s;
        grad[c] = sign * dr * s;
    }
}

hipError_t launch_heat_cell_products(const HeatGrid& g, const HeatKe& ke, const double* lam,
                                     const double* T, const double* x, double xmin,
                                     const Penalty& pen, int pbi, double sign, double* cell,
                                     double* grad, hipStream_t s) {
    const dim3 grid(heat_blocks(g.ncells)), block(kThreads);
    if (g.dim == 3)
        hipLaunchKernelGGL((k_heat_cell_products<3>), grid, block, 0, s, g, ke, lam, T, x, xmin,
                           pen, pbi, sign, cell, grad);
    else
        hipLaunchKernelGGL((k_heat_cell_products<2>), grid, block, 0, s, g, ke, lam, T, x, xmin,
                           pen, pbi, sign, cell, grad);
    return hipGetLastError();
}

}  // namespace tohip
