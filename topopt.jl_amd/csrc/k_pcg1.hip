// One FP64 Jacobi-PCG iteration on K(E) in one launch (k_pcg1.h): the pending
// x and r update, the direction, q = K p and the sums of the next launch.
//
// A 256-thread workgroup owns a column of 15 x 15 output nodes and, in 3D, a
// chunk of node planes that it walks upwards; 2D is one plane.  Thread (ci, cj)
// stages node (ci, cj) of the column's 17 x 17 nodes (threads 0..32 the far
// column and row too) and handles cell (ci, cj) of the 16 x 16 cells.  Per
// plane:
//   * the update and the direction are formed in registers, the direction goes
//     to LDS with prescribed components zeroed (as bcmatrix does), the owner
//     writes x, r and p;
//   * each thread transforms its cell's four nodes to the xy Hadamard basis,
//     once for the layer below and the layer above;
//   * the layer's cells: sum and difference with the transform of the plane
//     below, the modal blocks of the element operator times E, and the lower
//     plane's total (with what the layer below left there) transformed back;
//   * a node's four cell columns are summed as two x-pairs (a DPP row shift
//     brings the left cell's value) and an LDS exchange between the rows.
// No atomics, no slot array; the same bits every run.
//
// Bound by latency below a few 100k nodes (an iteration's launch, loads, sums and
// one plane step are a chain), above by the loads of four vectors on the halo
// and 250 registers (two workgroups per CU).  MI355X, an iteration against the
// direction + update pair: 2D 160x40 5.2 us (12.2), 27x14x10 7.6 (12.0), 76x36x28
// 13.9 (23.1), 120x40x40 19.8 (33.7), 256x128x128 268 (307).
#include <algorithm>

#include "k_pcg1.h"

namespace tohip {

namespace {
constexpr int kPC = 16, kPO = kPC - 1, kPS = kPC + 1, kPP = kPS * kPS;
}

// Columns of 15 x 15 nodes and chunks of zc planes (zc + 2 are staged).  A
// workgroup per CU where that takes chunks of at most 5 planes, else two (256
// VGPRs: two run per CU).
// One iteration on MI355X, in the LOOP form (a straight body is 3-7 % faster),
// with 243 / 378 / 756 workgroups: 120x40x40 23.1 / 22.8 / 30.0 us; with 162 /
// 486 / 972: 256x128x128 408 / 272 / 297 us; with 180 / 270: 76x36x28 16.6 / 18.1.
struct Pcg1Shape {
    int ncx, ncy, zc, nch, nwork;
};
static Pcg1Shape pcg1_shape(const Grid& g) {
    Pcg1Shape s;
    s.ncx = (g.NX + kPO - 1) / kPO;
    s.ncy = (g.NY + kPO - 1) / kPO;
    const int64_t cols = (int64_t)s.ncx * s.ncy;
    auto planes = [&](int64_t target) {
        const int64_t want = std::max<int64_t>(1, target / cols);
        return (int)std::max<int64_t>(std::min(2, g.NZ), (g.NZ + want - 1) / want);
    };
    s.zc = planes(256);
    if (s.zc > 5) s.zc = planes(512);
    s.nch = (g.NZ + s.zc - 1) / s.zc;
    s.nwork = (int)(cols * s.nch);
    return s;
}

template <int D>
struct Pcg1Node {
    double p[D], r[D], q[D], d[D];
    uint8_t m;  // prescribed bits
};

// LOOP: more work than workgroups.  Without it the body is not in a loop, which
// costs it registers.
template <int DIM, bool CUBE, bool LOOP>
__global__ __launch_bounds__(kThreads, 2) void k_pcg1(Grid g, ElemOp<double> op, Pcg1Shape sh,
                                                   const uint8_t* __restrict__ fixmask,
                                                   const double* __restrict__ E, double md,
                                                   Pcg1Args a) {
    __shared__ double pl[2][DIM][kPP];
    __shared__ double exch[DIM][kThreads];
    __shared__ double red[kWaves][kPcg1Vals];
    const int tid = threadIdx.x, ci = tid & (kPC - 1), cj = tid / kPC;
    // the second node of threads 0..32: the far column, then the far row
    const bool two = tid < 2 * kPC + 1;
    const int li2 = tid <= kPC ? kPC : tid - kPS, lj2 = tid <= kPC ? tid : kPC;
    Pcg1Plan plan{0.0, 0.0, kPcg1Step};
    bool pend = false, update = true;  // an update is pending; and may be applied

    // A node's (cell's) place: a base that is the same for the whole workgroup,
    // advanced by a plane a step, and a node offset within the column's plane
    // (vectors are below 4 GiB, so byte offsets have 32 bits).
    int i0 = 0, j0 = 0;
    uint32_t oa = 0, ob = 0, oe = 0;
    bool ina = false, inb = false, ine = false;
    int64_t nbase = 0, ebase = 0;
    auto load = [&](uint32_t o, int k) {
        const int nk = DIM == 3 ? min(max(k, 0), g.NZ - 1) : 0;
        const int64_t base = nbase + (int64_t)nk * g.NX * g.NY;
        Pcg1Node<DIM> h;
        ld_node<DIM>(a.p + DIM * base, o, h.p);
        ld_node<DIM>(a.r + DIM * base, o, h.r);
        ld_node<DIM>(a.q + DIM * base, o, h.q);
        ld_node<DIM>(a.dinv + DIM * base, o, h.d);
        h.m = at(fixmask + base, o);
        return h;
    };
    // Prescribed bits (every bit outside the mesh) and modulus (0 outside) from
    // the loaded values, when they are used: a select at the load would wait
    // for it, and with it for the whole prefetch.
    auto bits = [&](const Pcg1Node<DIM>& h, bool in, int k) {
        return (in && (DIM == 2 || (k >= 0 && k < g.NZ))) ? (uint32_t)h.m : 0xffu;
    };
    auto load_E = [&](int k) {  // the cell of this thread in layer k
        const int ck = DIM == 3 ? min(max(k, 0), g.nz - 1) : 0;
        const int64_t base = ebase + (int64_t)ck * g.nx * g.ny;
        return at(E + base, oe);
    };
    double sum[kPcg1Vals] = {0, 0, 0, 0, 0, 0, 0, 0};
    int buf = 0;
    bool first = true;
    for (int w = blockIdx.x; w < sh.nwork; w += gridDim.x) {
        const int wr = xcd_remap(w, sh.nwork);
        const int ncol = sh.ncx * sh.ncy, col = wr % ncol, ch = wr / ncol;
        i0 = (col % sh.ncx) * kPO;
        j0 = (col / sh.ncx) * kPO;
        const int kb = DIM == 3 ? ch * sh.zc : 0, ke = DIM == 3 ? min(kb + sh.zc, g.NZ) : 1;
        const int gi = i0 - 1 + ci, gj = j0 - 1 + cj;
        const bool mine = ci >= 1 && cj >= 1 && gi < g.NX && gj < g.NY;
        {
            const int bi = max(i0 - 1, 0), bj = max(j0 - 1, 0);
            auto place = [&](int li, int lj, bool& in) {
                const int x = i0 - 1 + li, y = j0 - 1 + lj;
                const int cx = min(max(x, 0), g.NX - 1), cy = min(max(y, 0), g.NY - 1);
                in = x == cx && y == cy;
                return (uint32_t)(cx - bi) + (uint32_t)g.NX * (uint32_t)(cy - bj);
            };
            nbase = bi + (int64_t)g.NX * bj;
            ebase = bi + (int64_t)g.nx * bj;
            oa = place(ci, cj, ina);
            ob = place(two ? li2 : 0, two ? lj2 : 0, inb);
            ine = gi >= 0 && gi < g.nx && gj >= 0 && gj < g.ny;
            oe = ine ? (uint32_t)(gi - bi) + (uint32_t)g.nx * (uint32_t)(gj - bj) : 0u;
        }
        // node base of plane k
        auto plane = [&](int k) {
            return DIM * (nbase + (int64_t)(DIM == 3 ? k : 0) * g.NX * g.NY);
        };
        const int sb = DIM == 3 ? kb - 1 : 0, se = DIM == 3 ? ke : 0;  // staged planes
        Pcg1Node<DIM> na = load(oa, sb), nb{};
        if (two) nb = load(ob, sb);
        double xa[DIM] = {};
        if (mine && sb >= kb) ld_node<DIM>((const double*)a.x + plane(sb), oa, xa);
        double en = DIM == 3 ? 0.0 : load_E(0);
        if (first) {
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
        if (plan.mode != kPcg1Step) {
            // the pending update alone: x, and (exact) r with its two sums
            if (update && mine) {
                for (int k = kb; k < ke; ++k) {
                    const int64_t n = plane(k);
                    double p[DIM], x[DIM];
                    ld_node<DIM>(a.p + n, oa, p);
                    if (pend) {
                        ld_node<DIM>((const double*)a.x + n, oa, x);
#pragma unroll
                        for (int d = 0; d < DIM; ++d) x[d] += plan.alpha * p[d];
                        st_node<DIM>(a.x + n, oa, x);
                    }
                    if (plan.mode == kPcg1Exact) {
                        double r[DIM], q[DIM], dv[DIM];
                        ld_node<DIM>(a.r + n, oa, r);
                        ld_node<DIM>(a.q + n, oa, q);
                        ld_node<DIM>(a.dinv + n, oa, dv);
#pragma unroll
                        for (int d = 0; d < DIM; ++d) {
                            r[d] = fma(-plan.alpha, q[d], r[d]);
                            sum[kSumRZ] += dv[d] * r[d] * r[d];
                            sum[kSumRR] += r[d] * r[d];
                        }
                        st_node<DIM>(a.rn + n, oa, r);
                        st_node<DIM>(a.pn + n, oa, p);
                    }
                }
            }
            if (LOOP) continue;
            break;
        }
        double fp[DIM][4] = {}, up[DIM][4] = {};
        double po[DIM] = {}, ro[DIM] = {}, dd[DIM] = {};  // own node of the plane below
        uint32_t mo = 0;
        for (int k = sb; k <= se; ++k) {
            // the update and the direction of this plane, then the next plane's loads
            auto direction = [&](Pcg1Node<DIM>& h) {
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    // explicit FMAs: a halo copy and its owner get the same bits
                    h.r[d] = fma(-plan.alpha, pend ? h.q[d] : 0.0, h.r[d]);
                    h.p[d] = fma(plan.beta, h.p[d], h.d[d] * h.r[d]);
                }
            };
            double xc[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) xc[d] = xa[d] + plan.alpha * na.p[d];
            direction(na);
            const uint32_t mc = bits(na, ina, k);
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                pl[buf][d][ci + kPS * cj] = ((mc >> d) & 1) ? 0.0 : na.p[d];
            if (two) {
                direction(nb);
                const uint32_t m2 = bits(nb, inb, k);
#pragma unroll
                for (int d = 0; d < DIM; ++d)
                    pl[buf][d][li2 + kPS * lj2] = ((m2 >> d) & 1) ? 0.0 : nb.p[d];
            }
            const bool cell = ine && (DIM == 2 || (k >= 1 && k <= g.nz));  // layer k - 1
            const double ec = cell ? en : 0.0;
            double pc[DIM], rc[DIM], dc[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                pc[d] = na.p[d];
                rc[d] = na.r[d];
                dc[d] = na.d[d];
            }
            if (k < se) {
                na = load(oa, k + 1);
                if (two) nb = load(ob, k + 1);
                if (mine && k + 1 >= kb && k + 1 < ke)
                    ld_node<DIM>((const double*)a.x + plane(k + 1), oa, xa);
                en = load_E(k);
            }
            if (mine && k >= kb && k < ke) {
                if (pend) st_node<DIM>(a.x + plane(k), oa, xc);
                st_node<DIM>(a.rn + plane(k), oa, rc);
                st_node<DIM>(a.pn + plane(k), oa, pc);
            }
            __syncthreads();
            double f[DIM][4];
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    f[d][c] = pl[buf][d][ci + (c & 1) + kPS * (cj + (c >> 1))];
                hadamard_fwd<double, 2>(f[d]);
            }
            buf ^= 1;
            if (DIM == 2 || k > sb) {
                double lo[DIM][4];
                if constexpr (DIM == 3) {
                    double xm[3][8], z[3][8];
#pragma unroll
                    for (int d = 0; d < 3; ++d)
#pragma unroll
                        for (int m = 0; m < 4; ++m) {
                            xm[d][m] = fp[d][m] + f[d][m];
                            xm[d][m + 4] = f[d][m] - fp[d][m];
                        }
                    if constexpr (CUBE) {
                        double c[8];
#pragma unroll
                        for (int i = 0; i < 8; ++i) c[i] = op.cube[i] * ec;
                        modal_blocks_cube<double>(c, xm, z);
                    } else {
                        modal_blocks<double, 3, false>(op, xm, z);
#pragma unroll
                        for (int d = 0; d < 3; ++d)
#pragma unroll
                            for (int m = 0; m < 8; ++m) z[d][m] *= ec;
                    }
#pragma unroll
                    for (int d = 0; d < 3; ++d)
#pragma unroll
                        for (int m = 0; m < 4; ++m) {
                            lo[d][m] = up[d][m] + (z[d][m] - z[d][m + 4]);
                            up[d][m] = z[d][m] + z[d][m + 4];
                        }
                } else {
                    modal_blocks<double, 2, false>(op, f, lo);
#pragma unroll
                    for (int d = 0; d < 2; ++d)
#pragma unroll
                        for (int m = 0; m < 4; ++m) lo[d][m] *= ec;
                }
                double q[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    hadamard_inv<double, 2>(lo[d]);
                    q[d] = row_shr1(lo[d][1]) + lo[d][0];
                    exch[d][tid] = row_shr1(lo[d][3]) + lo[d][2];
                }
                __syncthreads();
                const int ko = DIM == 3 ? k - 1 : 0;
                if (mine && ko >= kb && ko < ke) {
                    const uint32_t m = DIM == 3 ? mo : mc;
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        const double p = DIM == 3 ? po[d] : pc[d], r = DIM == 3 ? ro[d] : rc[d],
                                     dv = DIM == 3 ? dd[d] : dc[d];
                        q[d] += exch[d][tid - kPC];
                        if ((m >> d) & 1) q[d] = md * p;
                        const double z = dv * r, dq = dv * q[d];
                        sum[kSumRZ] += z * r;
                        sum[kSumPQ] += p * q[d];
                        sum[kSumQZ] += z * q[d];
                        sum[kSumQDQ] += dq * q[d];
                        sum[kSumRR] += r * r;
                        sum[kSumRQ] += r * q[d];
                        sum[kSumQQ] += q[d] * q[d];
                    }
                    st_node<DIM>(a.qn + plane(ko), oa, q);
                }
            }
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
#pragma unroll
                for (int m = 0; m < 4; ++m) fp[d][m] = f[d][m];
                po[d] = pc[d];
                ro[d] = rc[d];
                dd[d] = dc[d];
            }
            mo = mc;
        }
        if (!LOOP) break;
    }
    pcg1_store_sums(sum, red, a.partn);
}

// 3D grids too small for the chunks to matter: one output plane a workgroup, 512
// threads, one group of 256 for the layer below the plane and one for the layer
// above, so that the three planes are loaded and the two layers computed at the
// same time instead of in turn.  27x14x10 box cells: 8.5 us an iteration against 13.2
// marching (whole solves).  164 VGPRs: one workgroup per CU, so a grid of more planes than CUs is
// left to the marching kernel (76x36x28: 26 against 15 us; 120x40x40: 47 against 22;
// bounded to two workgroups per CU it spills: 38 and 65).
static int pcg1_planes(const Grid& g) {
    const int64_t n = (int64_t)((g.NX + kPO - 1) / kPO) * ((g.NY + kPO - 1) / kPO) * g.NZ;
    return g.dim == 3 && n <= 256 ? (int)n : 0;
}

template <bool CUBE>
__global__ __launch_bounds__(2 * kThreads) void k_pcg1_plane(Grid g, ElemOp<double> op,
                                                             const uint8_t* __restrict__ fixmask,
                                                             const double* __restrict__ E,
                                                             double md, Pcg1Args a) {
    constexpr int NT = 2 * kThreads;
    __shared__ double pl[3][3][kPP];
    __shared__ double ex[3][3][NT];  // upper y1, lower y0, lower y1
    __shared__ double red[NT / 64][kPcg1Vals];
    const int tid = threadIdx.x, t = tid / kThreads, c2 = tid % kThreads;
    const int ci = c2 & (kPC - 1), cj = c2 / kPC;
    // this thread's nodes: (ci, cj) of the output plane (group 0) or the one below,
    // and one of the rest: (ci, cj) of the plane above (group 0), or one of the far
    // column and row of a plane (threads 0..98 of group 1)
    const int zm = t == 0 ? 1 : 0;  // staged planes 0, 1, 2: below, output, above
    int z2 = 2, li2 = ci, lj2 = cj;
    bool two = t == 0;
    if (t > 0) {
        const int e = tid - kThreads;
        two = e < (2 * kPC + 1) * 3;
        z2 = two ? e / (2 * kPC + 1) : 0;
        const int i = e - z2 * (2 * kPC + 1);
        li2 = i <= kPC ? kPC : i - kPS;
        lj2 = i <= kPC ? i : kPC;
    }
    Pcg1Plan plan{0.0, 0.0, kPcg1Step};
    bool pend = false, update = true;
    double sum[kPcg1Vals] = {0, 0, 0, 0, 0, 0, 0, 0};
    const int ncx = (g.NX + kPO - 1) / kPO, ncol = ncx * ((g.NY + kPO - 1) / kPO);
    const int wr = xcd_remap(blockIdx.x, gridDim.x), col = wr % ncol, kb = wr / ncol;
    const int i0 = (col % ncx) * kPO, j0 = (col / ncx) * kPO;
    auto load = [&](int li, int lj, int z, Pcg1Node<3>& h) {
        const int x = i0 - 1 + li, y = j0 - 1 + lj, k = kb - 1 + z;
        const int cx = min(max(x, 0), g.NX - 1), cy = min(max(y, 0), g.NY - 1),
                  ck = min(max(k, 0), g.NZ - 1);
        const uint32_t n = (uint32_t)cx + (uint32_t)g.NX * ((uint32_t)cy + (uint32_t)g.NY * ck);
        ld_node<3>(a.p, n, h.p);
        ld_node<3>(a.r, n, h.r);
        ld_node<3>(a.q, n, h.q);
        ld_node<3>(a.dinv, n, h.d);
        h.m = at(fixmask, n);
        return n;
    };
    auto bits = [&](const Pcg1Node<3>& h, int li, int lj, int z) {
        const int x = i0 - 1 + li, y = j0 - 1 + lj, k = kb - 1 + z;
        return (x >= 0 && x < g.NX && y >= 0 && y < g.NY && k >= 0 && k < g.NZ) ? (uint32_t)h.m
                                                                              : 0xffu;
    };
    Pcg1Node<3> na, nb;
    const uint32_t n = load(ci, cj, zm, na);
    if (two) load(li2, lj2, z2, nb);
    const int gi = i0 - 1 + ci, gj = j0 - 1 + cj;
    const bool mine = t == 0 && ci >= 1 && cj >= 1 && gi < g.NX && gj < g.NY;
    double xa[3] = {};
    if (mine) ld_node<3>((const double*)a.x, n, xa);
    double ec;  // modulus of the thread's cell
    bool cell;  // it is in the mesh
    {
        const int gz = kb - 1 + t;
        const int cx = min(max(gi, 0), g.nx - 1), cy = min(max(gj, 0), g.ny - 1),
                  ck = min(max(gz, 0), g.nz - 1);
        ec = at(E, (uint32_t)cx + (uint32_t)g.nx * ((uint32_t)cy + (uint32_t)g.ny * ck));
        cell = gi == cx && gj == cy && gz == ck;
    }
    {
        // the loads are in flight while the sums are formed
        const Pcg1State s0 = *a.s;
        if (s0.done) {
            if (blockIdx.x == 0 && tid == 0) *a.sn = s0;
            return;
        }
        double v[kPcg1Vals];
        pcg1_reduce<NT>(a.part, a.nb, v, red);
        Pcg1State s1;
        plan = pcg1_plan(s0, v, s1);
        if (blockIdx.x == 0 && tid == 0) *a.sn = s1;
        pend = s0.pend != 0;
        update = s1.err == 0 || s0.iter != s1.iter;
    }
    if (mine && pend && update) {
#pragma unroll
        for (int d = 0; d < 3; ++d) xa[d] += plan.alpha * na.p[d];
        st_node<3>(a.x, n, xa);
    }
    if (plan.mode != kPcg1Step) {
        // the pending update alone: x, and (exact) r with its two sums
        if (plan.mode == kPcg1Exact && mine) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                na.r[d] = fma(-plan.alpha, na.q[d], na.r[d]);
                sum[kSumRZ] += na.d[d] * na.r[d] * na.r[d];
                sum[kSumRR] += na.r[d] * na.r[d];
            }
            st_node<3>(a.rn, n, na.r);
            st_node<3>(a.pn, n, na.p);
        }
        pcg1_store_sums<NT>(sum, red, a.partn);
        return;
    }
    auto direction = [&](Pcg1Node<3>& h) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            // explicit FMAs: a halo copy and its owner get the same bits
            h.r[d] = fma(-plan.alpha, pend ? h.q[d] : 0.0, h.r[d]);
            h.p[d] = fma(plan.beta, h.p[d], h.d[d] * h.r[d]);
        }
    };
    if (!cell) ec = 0.0;
    direction(na);
    const uint32_t m1 = bits(na, ci, cj, zm);
#pragma unroll
    for (int d = 0; d < 3; ++d)
        pl[zm][d][ci + kPS * cj] = ((m1 >> d) & 1) ? 0.0 : na.p[d];
    if (two) {
        direction(nb);
        const uint32_t m2 = bits(nb, li2, lj2, z2);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            pl[z2][d][li2 + kPS * lj2] = ((m2 >> d) & 1) ? 0.0 : nb.p[d];
    }
    if (mine) {
        st_node<3>(a.rn, n, na.r);
        st_node<3>(a.pn, n, na.p);
    }
    __syncthreads();
    double xe[3][8], z[3][8];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
#pragma unroll
        for (int c = 0; c < 8; ++c)
            xe[d][c] = pl[t + (c >> 2)][d][ci + (c & 1) + kPS * (cj + ((c >> 1) & 1))];
        hadamard_fwd<double, 3>(xe[d]);
    }
    if constexpr (CUBE) {
        double c[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = op.cube[i] * ec;
        modal_blocks_cube<double>(c, xe, z);
    } else {
        modal_blocks<double, 3, false>(op, xe, z);
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int m = 0; m < 8; ++m) z[d][m] *= ec;
    }
    double q[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        hadamard_inv<double, 3>(z[d]);
        q[d] = row_shr1(z[d][5]) + z[d][4];  // the upper face, lower row
        ex[0][d][tid] = row_shr1(z[d][7]) + z[d][6];
        ex[1][d][tid] = row_shr1(z[d][1]) + z[d][0];
        ex[2][d][tid] = row_shr1(z[d][3]) + z[d][2];
    }
    __syncthreads();
    if (mine) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            q[d] = (ex[0][d][tid - kPC] + q[d]) +
                   (ex[2][d][tid + kThreads - kPC] + ex[1][d][tid + kThreads]);
            if ((m1 >> d) & 1) q[d] = md * na.p[d];
            const double zz = na.d[d] * na.r[d], dq = na.d[d] * q[d];
            sum[kSumRZ] += zz * na.r[d];
            sum[kSumPQ] += na.p[d] * q[d];
            sum[kSumQZ] += zz * q[d];
            sum[kSumQDQ] += dq * q[d];
            sum[kSumRR] += na.r[d] * na.r[d];
            sum[kSumRQ] += na.r[d] * q[d];
            sum[kSumQQ] += q[d] * q[d];
        }
        st_node<3>(a.qn, n, q);
    }
    pcg1_store_sums<NT>(sum, red, a.partn);
}

// Work beyond what the chip holds at once (three workgroups per CU in 2D, two in
// 3D, by the registers of the LOOP form) is strided over: every workgroup sums every
// workgroup's row of partials, so their number enters squared.  MI355X, us an
// iteration with at most 512 / 768 / 1024 / 4096 workgroups, and of the direction +
// update pair: 2D 640x320 11.1 / 11.9 / 13.1 / 13.0 and 17.0, 1000x990 30 / 31 / 37 /
// 97 and 41, 1500x1500 88 / 84 / 94 / 147 and 81, 2400x2400 213 / 227 / 254 / 274 and
// 236; 3D 900x900x2 167 / 186 / 174 / 215 and 180, 500x500x2 43 / 48 / 49 / 49 and 90.
static int pcg1_resident(const Grid& g) { return g.dim == 2 ? 768 : 512; }

int pcg1_blocks(const Grid& g) {
    const int n = pcg1_planes(g);
    return n ? n : std::min(pcg1_shape(g).nwork, pcg1_resident(g));
}

template <int DIM, bool CUBE>
static void launch_pcg1_march(const Grid& g, const ElemOp<double>& op, const uint8_t* fixmask,
                              const double* E, double md, const Pcg1Args& a, hipStream_t s) {
    const Pcg1Shape sh = pcg1_shape(g);
    const dim3 grid(pcg1_blocks(g)), block(kThreads);
    if (sh.nwork > (int)grid.x)
        hipLaunchKernelGGL((k_pcg1<DIM, CUBE, true>), grid, block, 0, s, g, op, sh, fixmask, E, md,
                           a);
    else
        hipLaunchKernelGGL((k_pcg1<DIM, CUBE, false>), grid, block, 0, s, g, op, sh, fixmask, E,
                           md, a);
}

hipError_t launch_pcg1(const Grid& g, const ElemOp<double>& op, const uint8_t* fixmask,
                       const double* E, double meandiag, const Pcg1Args& a, hipStream_t s) {
    if (const int n = pcg1_planes(g)) {
        if (op.is_cube)
            hipLaunchKernelGGL((k_pcg1_plane<true>), dim3(n), dim3(2 * kThreads), 0, s, g, op,
                               fixmask, E, meandiag, a);
        else
            hipLaunchKernelGGL((k_pcg1_plane<false>), dim3(n), dim3(2 * kThreads), 0, s, g, op,
                               fixmask, E, meandiag, a);
    } else if (g.dim == 2) {
        launch_pcg1_march<2, false>(g, op, fixmask, E, meandiag, a, s);
    } else if (op.is_cube) {
        launch_pcg1_march<3, true>(g, op, fixmask, E, meandiag, a, s);
    } else {
        launch_pcg1_march<3, false>(g, op, fixmask, E, meandiag, a, s);
    }
    return hipGetLastError();
}

}  // namespace tohip
