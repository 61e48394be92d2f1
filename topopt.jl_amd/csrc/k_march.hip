// The FP32 passes of the multigrid-preconditioned PCG over a 3D level, by marching
// columns as k_pcg1: a 256-thread workgroup walks up a column of 16 x 16 cells, the
// xy Hadamard transform of each node plane is formed once for the layers below and
// above it, and the corner sums leave the Hadamard basis once per node plane.
//
//   DIR   p = D r + beta p (D null: the unit), q = K p, partials of p.q: the
//         direction step of PCG iteration iter + 1 (k_matvec<PCG>)
//   POST  x' = x + P xc, z = x' + w D^-1 (b - K x'), partials of (b.z, b.b)
//   PRE   x = w D^-1 b, b_c = P^T (b - K x); UPD: on b - alpha q, the PCG update in
//         flight (MgFusedUpdate), with r and x stored by the owner
//
// PRE owns 14 x 14 nodes (an even origin) of the 15 x 15 whose residual it forms:
// that is all that its 7 x 7 coarse nodes reach.  The residual goes through LDS only.
// A plane's restriction follows the barrier of the next plane's staging.
//
// Bound by latency up to some 10^5 cells (a launch, loads, two barriers a plane), by
// registers above (118 to 149 a thread, 3 or 4 workgroups per CU): at 256x128x128 the
// passes move their vectors once at 2.7 to 3.4 TB/s.  DIR held to 5 workgroups per CU
// spills 22 registers: 152 against 86 us.
#include <algorithm>
#include <cstdlib>

#include "k_common.h"

namespace tohip {

namespace {
constexpr int kMC = 16, kMR = kMC - 1, kMS = kMC + 1;
constexpr int kMDir = 0, kMPost = 1, kMPre = 2;
}  // namespace

struct MarchShape {
    int ncx, ncy, zc, nch;
    int blocks() const { return ncx * ncy * nch; }
};
// Columns of 15 x 15 nodes (pre: 14 x 14) and chunks of zc planes (pre: even).
// Three workgroups per CU, which is what the post-smoothing's registers admit.  With
// 512 / 768 / 1024 / 1536 workgroups: post-smoothing 256x128x128 74 / 65 / 76 / 64
// us, a V-cycle 238 / 194 / 202 / 196, at 128x64x64 71 / 68 / 72 / 71.
static MarchShape march_shape(const Grid& g, bool pre) {
    constexpr int target = 768;
    const int step = pre ? kMR - 1 : kMR;
    MarchShape s;
    s.ncx = (g.NX + step - 1) / step;
    s.ncy = (g.NY + step - 1) / step;
    const int64_t cols = (int64_t)s.ncx * s.ncy;
    const int64_t want = std::max<int64_t>(1, target / cols);
    s.zc = std::max<int>(2, (int)((g.NZ + want - 1) / want));
    for (;; ++s.zc) {
        if (pre && s.zc % 2) ++s.zc;
        s.nch = (g.NZ + s.zc - 1) / s.zc;
        if (cols * s.nch <= kMaxPartials || s.zc >= g.NZ) return s;
    }
}

struct MarchArgs {
    const float* a;      // DIR: r; POST: x; PRE: b
    const float* dinv;
    const float* b;      // POST
    float* out;          // DIR: q; POST: z; PRE: x
    float *p0, *p1;      // DIR
    const float* xc;     // POST: the coarse correction (null: x is x' already)
    float* bc;           // PRE: the coarse right-hand side
    const uint8_t* cmask;
    Grid gc;
    float w;
    const float* wdev;
    double md;           // DIR: the diagonal at prescribed DOFs
    PcgScalars* sc;
    const double* partB;
    int nbB;
    double* part;
    MgFusedUpdate upd;
};

template <int MODE, bool CUBE, bool UPD>
__global__ __launch_bounds__(kThreads, MODE == kMPost ? 3 : 4) void k_march(Grid g, ElemOp<float> op, MarchShape sh,
                                                       const uint8_t* __restrict__ fixmask,
                                                       const float* __restrict__ E, MarchArgs a) {
    constexpr bool DIR = MODE == kMDir, POST = MODE == kMPost, PRE = MODE == kMPre;
    constexpr int OFF = PRE ? 2 : 1, OWN = PRE ? kMR - 1 : kMR;
    constexpr int NRES = kMR * kMR, HC = OWN / 2;  // PRE: residual nodes, coarse nodes a row
    __shared__ float pl[2][3][kMS * kMS];
    __shared__ float exch[3][kThreads];
    __shared__ float rl[PRE ? 3 : 1][PRE ? NRES : 1];
    __shared__ double red[kWaves];
    if (!DIR && a.sc && a.sc->done) return;
    float w = a.w;
    if (!DIR && a.wdev) w = *a.wdev;
    const int tid = threadIdx.x, ci = tid & (kMC - 1), cj = tid / kMC;
    // the second node of threads 0..32: the far column, then the far row
    const bool two = tid < 2 * kMC + 1;
    const int li2 = tid <= kMC ? kMC : tid - kMS, lj2 = tid <= kMC ? tid : kMC;

    float* pold = nullptr;
    float* pnew = nullptr;
    long long it = 0;
    if (DIR) {
        if (a.sc->done) return;
        it = a.sc->iter;
        pold = (it & 1) ? a.p1 : a.p0;
        pnew = (it & 1) ? a.p0 : a.p1;
    }
    const long long uk = UPD ? a.upd.sc->k_cur : 0;
    const float* up_ = UPD ? ((uk & 1) ? a.upd.p1 : a.upd.p0) : nullptr;

    const int ncol = sh.ncx * sh.ncy;
    const int wr = xcd_remap(blockIdx.x, gridDim.x), col = wr % ncol, ch = wr / ncol;
    const int i0 = (col % sh.ncx) * OWN, j0 = (col / sh.ncx) * OWN;
    const int kb = ch * sh.zc, ke = min(kb + sh.zc, g.NZ);
    const int gi = i0 - OFF + ci, gj = j0 - OFF + cj;
    const bool mine = ci >= OFF && cj >= OFF && gi < g.NX && gj < g.NY;
    const int bi = max(i0 - OFF, 0), bj = max(j0 - OFF, 0);
    const int64_t nbase = bi + (int64_t)g.NX * bj, ebase = bi + (int64_t)g.nx * bj;
    // coarse nodes of a fine node's xy interpolation, from the base (bi / 2, bj / 2)
    const bool prol = POST && a.xc;
    const int64_t cbase = POST ? (bi >> 1) + (int64_t)a.gc.NX * (bj >> 1) : 0;
    struct Corners {
        uint32_t o, dx, dy;
    };
    auto place = [&](int li, int lj, bool& in, Corners& cc) {
        const int x = i0 - OFF + li, y = j0 - OFF + lj;
        const int cx = min(max(x, 0), g.NX - 1), cy = min(max(y, 0), g.NY - 1);
        in = x == cx && y == cy;
        if (POST) {
            cc.o = (uint32_t)((cx >> 1) - (bi >> 1)) +
                   (uint32_t)a.gc.NX * (uint32_t)((cy >> 1) - (bj >> 1));
            cc.dx = cx & 1;
            cc.dy = (cy & 1) ? (uint32_t)a.gc.NX : 0u;
        }
        return (uint32_t)(cx - bi) + (uint32_t)g.NX * (uint32_t)(cy - bj);
    };
    bool ina, inb;
    Corners ca{0, 0, 0}, cb{0, 0, 0};
    const uint32_t oa = place(ci, cj, ina, ca);
    const uint32_t ob = place(two ? li2 : ci, two ? lj2 : cj, inb, cb);
    const bool ine = gi >= 0 && gi < g.nx && gj >= 0 && gj < g.ny;
    const uint32_t oe = ine ? (uint32_t)(gi - bi) + (uint32_t)g.nx * (uint32_t)(gj - bj) : 0u;
    auto node = [&](int k) { return nbase + (int64_t)k * g.NX * g.NY; };
    auto plane = [&](int k) { return 3 * node(k); };

    struct Node {
        float a[3], b[3], c[3];
        float cc[POST ? 4 : 1][3];  // coarse corners
        uint8_t m;
    };
    // the four coarse nodes around a fine node in coarse plane K (they repeat on even
    // coordinates: their mean is the interpolation in every case)
    auto corners = [&](const Corners& cc, int K, Node& h) {
        const int Kc = min(max(K, 0), a.gc.NZ - 1);
        const float* x = a.xc + 3 * (cbase + (int64_t)Kc * a.gc.NX * a.gc.NY);
#pragma unroll
        for (int c = 0; c < (POST ? 4 : 1); ++c)
            ld_node<3>(x, cc.o + (c & 1 ? cc.dx : 0u) + (c & 2 ? cc.dy : 0u), h.cc[c]);
    };
    auto load = [&](uint32_t o, const Corners& cc, int k, Node& h) {
        const int kc = min(max(k, 0), g.NZ - 1);
        const int64_t n = plane(kc);
        ld_node<3>(a.a + n, o, h.a);
        h.m = at(fixmask + node(kc), o);
        if (DIR) {
            if (a.dinv) {
                ld_node<3>(a.dinv + n, o, h.b);
            } else {
                h.b[0] = h.b[1] = h.b[2] = 1.f;
            }
            ld_node<3>((const float*)pold + n, o, h.c);
        }
        if (PRE) {
            ld_node<3>(a.dinv + n, o, h.b);
            if (UPD) ld_node<3>(a.upd.q + n, o, h.c);
        }
        if (POST && prol && (k & 1)) corners(cc, (k + 1) >> 1, h);
    };
    // the owner's further operands of plane k
    struct Own {
        float b[3], d[3];
    };
    auto load_own = [&](int k, Own& h) {
        const int64_t n = plane(min(max(k, 0), g.NZ - 1));
        if (POST) {
            ld_node<3>(a.b + n, oa, h.b);
            ld_node<3>(a.dinv + n, oa, h.d);
        }
        if (UPD) {
            ld_node<3>((const float*)a.upd.x + n, oa, h.b);
            ld_node<3>(up_ + n, oa, h.d);
        }
    };
    auto load_E = [&](int k) {  // the cell of this thread in layer k
        const int ck = min(max(k, 0), g.nz - 1);
        return at(E + ebase + (int64_t)ck * g.nx * g.ny, oe);
    };
    const int sb = kb - OFF, se = ke;  // staged planes
    Node na{}, nb{};
    Own oc{};
    load(oa, ca, sb, na);
    if (two) load(ob, cb, sb, nb);
    float en = 0.f;
    float cpa[3] = {}, cpb[3] = {};  // xy interpolation of the coarse plane at or below k
    auto mean4 = [](const float (&c)[POST ? 4 : 1][3], float (&v)[3]) {
#pragma unroll
        for (int d = 0; d < 3; ++d)
            v[d] = 0.25f * ((c[0][d] + c[POST ? 1 : 0][d]) + (c[POST ? 2 : 0][d] + c[POST ? 3 : 0][d]));
    };
    if (POST && prol) {
        // (sb odd, below: the plane that load() took is the next one)
        Node h{};
        corners(ca, sb >> 1, h);
        mean4(h.cc, cpa);
        if (two) {
            corners(cb, sb >> 1, h);
            mean4(h.cc, cpb);
        }
    }
    float beta = 0.f, ua = 0.f;
    double ualpha = 0.0, s1 = 0.0, s2 = 0.0;
    if (DIR) {
        // the first plane's loads are in flight
        const double rz = reduce_partials(a.partB, a.nbB, 2, 0, red);
        const double rr = reduce_partials(a.partB, a.nbB, 2, 1, red);
        const long long k = it + 1;
        const double tol_in = a.sc->tol;
        const double tol = tol_in < 0.0 ? fmax(a.sc->reltol * sqrt(rr), a.sc->abstol) : tol_in;
        int err;
        const bool stop = pcg_stop_test(a.sc, rz, rr, it, tol, err);
        const double rho_prev = a.sc->rho[(k - 1) & 1];
        if (blockIdx.x == 0 && tid == 0) {
            a.sc->rr = rr;
            if (tol_in < 0.0) {
                a.sc->tol = tol;
                a.sc->rr0 = rr;
            }
            if (stop) {
                a.sc->done = 1;
                if (err) a.sc->err = err;
            } else {
                a.sc->rho[k & 1] = rz;
                a.sc->rho_cur = rz;
                a.sc->k_cur = k;
            }
        }
        if (stop) return;
        beta = (float)(rz / rho_prev);
    }
    if (UPD) {
        const double pq = reduce_partials(a.upd.partA, a.upd.nbA, 1, 0, red);
        if (!(pq > 0.0 && pq < INFINITY)) {  // before x or r change
            if (blockIdx.x == 0 && tid == 0) {
                a.upd.sc->err = kPcgErrIndefinite;
                a.upd.sc->done = 1;
            }
            return;
        }
        ualpha = a.upd.sc->rho_cur / pq;
        ua = (float)ualpha;
    }

    // PRE: coarse node and component of this thread, and its sum over planes
    const int ro = tid / 3, rd = tid % 3, hi = ro % HC, hj = ro / HC;
    const int I = i0 / 2 + hi, J = j0 / 2 + hj;
    const bool coarse = PRE && tid < 3 * HC * HC && I < a.gc.NX && J < a.gc.NY;
    float acc = 0.f;
    auto put = [&](int K, float v) {
        const uint32_t N = (uint32_t)I + (uint32_t)a.gc.NX * ((uint32_t)J + (uint32_t)a.gc.NY * K);
        a.bc[3 * (size_t)N + rd] = ((a.cmask[N] >> rd) & 1) ? 0.f : v;
    };
    auto restrict_plane = [&](int k) {  // residual plane k in rl
        if (!coarse) return;
        float s = 0.f;
#pragma unroll
        for (int y = 0; y < 3; ++y)
#pragma unroll
            for (int x = 0; x < 3; ++x)
                s += (x == 1 ? 1.f : 0.5f) * (y == 1 ? 1.f : 0.5f) *
                     rl[PRE ? rd : 0][PRE ? (2 * hi + x) + kMR * (2 * hj + y) : 0];
        if (k & 1) {
            if (k > kb) put((k - 1) >> 1, acc + 0.5f * s);
            acc = 0.5f * s;
        } else {
            acc += s;
        }
    };

    float fp[3][4] = {}, up[3][4] = {};
    float vo[3] = {}, bo[3] = {};  // own node of the plane below
    uint32_t mo = 0xffu;
    int buf = 0;
    for (int k = sb; k <= se; ++k) {
        const bool kin = k >= 0 && k < g.NZ, own = mine && k >= kb && k < ke;
        float vc[3], bn[3] = {}, dn[3] = {}, xs[3] = {};
        // value of a node; PRE: and its right-hand side
        auto value = [&](const Node& h, float (&cp)[3], uint32_t m, float (&v)[3], float (&bv)[3]) {
            float cr[3] = {};
            if (POST && prol) {
                if (k & 1) {
                    float cn[3];
                    mean4(h.cc, cn);
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        cr[d] = 0.5f * (cp[d] + cn[d]);
                        cp[d] = cn[d];
                    }
                } else {
#pragma unroll
                    for (int d = 0; d < 3; ++d) cr[d] = cp[d];
                }
            }
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                // explicit FMAs: a halo copy and its owner get the same bits
                bv[d] = h.a[d];
                if (DIR) v[d] = __fmaf_rn(beta, h.c[d], h.b[d] * h.a[d]);
                if (POST) v[d] = h.a[d] + cr[d];
                if (PRE) {
                    if (UPD) bv[d] = __fmaf_rn(-ua, h.c[d], h.a[d]);
                    v[d] = w * h.b[d] * bv[d];
                }
                if (!DIR && ((m >> d) & 1)) v[d] = 0.f;
            }
        };
        const uint32_t mc = ina && kin ? (uint32_t)na.m : 0xffu;
        value(na, cpa, mc, vc, bn);
#pragma unroll
        for (int d = 0; d < 3; ++d)
            pl[buf][d][ci + kMS * cj] = DIR && ((mc >> d) & 1) ? 0.f : vc[d];
        if (two) {
            float v2[3], b2[3];
            const uint32_t m2 = inb && kin ? (uint32_t)nb.m : 0xffu;
            value(nb, cpb, m2, v2, b2);
#pragma unroll
            for (int d = 0; d < 3; ++d)
                pl[buf][d][li2 + kMS * lj2] = DIR && ((m2 >> d) & 1) ? 0.f : v2[d];
        }
        const float ec = ine && k >= 1 && k <= g.nz ? en : 0.f;  // layer k - 1
        if (UPD) {
#pragma unroll
            for (int d = 0; d < 3; ++d) xs[d] = __fmaf_rn(ua, oc.d[d], oc.b[d]);
        }
        if (k < se) {
            load(oa, ca, k + 1, na);
            if (two) load(ob, cb, k + 1, nb);
            en = load_E(k);
            if (UPD && mine && k + 1 >= kb && k + 1 < ke) load_own(k + 1, oc);
        }
        if (own) {
            if (DIR) st_node<3>(pnew + plane(k), oa, vc);
            if (PRE) st_node<3>(a.out + plane(k), oa, vc);
            if (UPD) {
                st_node<3>(a.upd.rnew + plane(k), oa, bn);
                st_node<3>(a.upd.x + plane(k), oa, xs);
            }
        }
        __syncthreads();
        if (PRE && k - 2 >= kb - 1) restrict_plane(k - 2);
        float f[3][4];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
#pragma unroll
            for (int c = 0; c < 4; ++c) f[d][c] = pl[buf][d][ci + (c & 1) + kMS * (cj + (c >> 1))];
            hadamard_fwd<float, 2>(f[d]);
        }
        buf ^= 1;
        if (k > sb) {
            float xm[3][8], z[3][8], lo[3][4];
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    xm[d][m] = fp[d][m] + f[d][m];
                    xm[d][m + 4] = f[d][m] - fp[d][m];
                }
            if constexpr (CUBE) {
                float c[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) c[i] = op.cube[i] * ec;
                modal_blocks_cube<float>(c, xm, z);
            } else {
                modal_blocks<float, 3, false>(op, xm, z);
#pragma unroll
                for (int d = 0; d < 3; ++d)
#pragma unroll
                    for (int m = 0; m < 8; ++m) z[d][m] *= ec;
            }
            float q[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    lo[d][m] = up[d][m] + (z[d][m] - z[d][m + 4]);
                    up[d][m] = z[d][m] + z[d][m + 4];
                }
                hadamard_inv<float, 2>(lo[d]);
                q[d] = row_shr1(lo[d][1]) + lo[d][0];
                exch[d][tid] = row_shr1(lo[d][3]) + lo[d][2];
            }
            __syncthreads();
            const int ko = k - 1;
            if (PRE ? (ko >= kb - 1 && ci >= 1 && cj >= 1) : (mine && ko >= kb)) {
                float o[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    q[d] += exch[d][tid - kMC];
                    const bool fx = (mo >> d) & 1;
                    if (DIR) {
                        o[d] = fx ? (float)a.md * vo[d] : q[d];
                        s1 += (double)vo[d] * (double)o[d];
                    }
                    if (POST) {
                        o[d] = fx ? 0.f : vo[d] + w * oc.d[d] * (oc.b[d] - q[d]);
                        s1 += (double)oc.b[d] * (double)o[d];
                        s2 += (double)oc.b[d] * (double)oc.b[d];
                    }
                    if (PRE)
                        rl[PRE ? d : 0][PRE ? (ci - 1) + kMR * (cj - 1) : 0] = fx ? 0.f : bo[d] - q[d];
                }
                if (!PRE) st_node<3>(a.out + plane(ko), oa, o);
            }
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
#pragma unroll
            for (int m = 0; m < 4; ++m) fp[d][m] = f[d][m];
            vo[d] = vc[d];
            if (PRE) bo[d] = bn[d];
        }
        mo = mc;
        if (POST && own) load_own(k, oc);  // used when plane k is finished, a step later
    }
    if (PRE) {
        __syncthreads();
        restrict_plane(ke - 1);
        // a last plane that is even has nothing above it
        if (coarse && ke == g.NZ) put((ke - 1) >> 1, acc);
        if (UPD && blockIdx.x == 0 && tid == 0) {
            a.upd.sc->iter = uk;
            a.upd.sc->alpha = ualpha;
        }
    }
    if (DIR) {
        const double s = block_sum_all(s1, red);
        if (tid == 0) a.part[blockIdx.x] = s;
    }
    if (POST && a.part) {
        const double t1 = block_sum_all(s1, red), t2 = block_sum_all(s2, red);
        if (tid == 0) {
            a.part[2 * (size_t)blockIdx.x] = t1;
            a.part[2 * (size_t)blockIdx.x + 1] = t2;
        }
    }
}

int march_blocks(const Grid& g) { return march_shape(g, false).blocks(); }

// The rule: 3D levels of 2^17 cells and more.  A V-cycle, its finest post-smoothing
// and the direction step against the tiles, MI355X, us: 120x40x40 (192,000 cells)
// 44.6 / 10.0 / 10.6 against 52.3 / 13.8 / 12.9; 76x36x28 (76,608) 45.0 / 8.7 / 9.1
// against 45.2 / 8.4 / 8.7; 128x64x64 68 / 14.4 / 14.5 against 90 / 26 / 23;
// 256x128x128 192 / 65 / 85 against 257 / 88 / 102 of marching columns without the
// shared transforms (whose update, 63, is now inside the pre-smoothing).
// TOHIP_MARCH_MINCELLS, read on every call, overrides the line for tests.
bool march_use(const Grid& g) {
    const char* e = getenv("TOHIP_MARCH_MINCELLS");
    const long long v = e ? atoll(e) : 0;
    return g.dim == 3 && g.ncells >= (v > 0 ? v : 1 << 17) && march_blocks(g) <= kMaxPartials;
}

template <int MODE, bool UPD>
static hipError_t launch_march(const Grid& g, const ElemOp<float>& op, const uint8_t* fixmask,
                               const float* E, const MarchArgs& a, hipStream_t s) {
    const MarchShape sh = march_shape(g, MODE == kMPre);
    if (g.dim != 3) return hipErrorInvalidValue;
    if (op.is_cube)
        hipLaunchKernelGGL((k_march<MODE, true, UPD>), dim3(sh.blocks()), dim3(kThreads), 0, s, g,
                           op, sh, fixmask, E, a);
    else
        hipLaunchKernelGGL((k_march<MODE, false, UPD>), dim3(sh.blocks()), dim3(kThreads), 0, s, g,
                           op, sh, fixmask, E, a);
    return hipGetLastError();
}

hipError_t launch_march_dir(const Grid& g, const ElemOp<float>& op, const float* r,
                            const float* dinv, float* p0, float* p1, float* q,
                            const uint8_t* fixmask, const float* E, double md, PcgScalars* sc,
                            const double* partB, int nbB, double* partA, hipStream_t s) {
    MarchArgs a{};
    a.a = r;
    a.dinv = dinv;
    a.out = q;
    a.p0 = p0;
    a.p1 = p1;
    a.md = md;
    a.sc = sc;
    a.partB = partB;
    a.nbB = nbB;
    a.part = partA;
    return launch_march<kMDir, false>(g, op, fixmask, E, a, s);
}

static bool halves(const Grid& g, const Grid& gc) {
    return gc.nx * 2 == g.nx && gc.ny * 2 == g.ny && gc.nz * 2 == g.nz;
}

hipError_t launch_march_post(const MgLevelView& L, float w, const float* b, const float* x,
                             const MgLevelView& C, const float* xc, float* z, const PcgScalars* sc,
                             double* part, hipStream_t s) {
    if (!halves(L.g, C.g)) return hipErrorInvalidValue;
    MarchArgs a{};
    a.a = x;
    a.dinv = L.dinv;
    a.b = b;
    a.out = z;
    a.xc = xc;
    a.gc = C.g;
    a.w = w;
    a.wdev = L.wdev;
    a.sc = const_cast<PcgScalars*>(sc);
    a.part = part;
    return launch_march<kMPost, false>(L.g, L.op, L.fixmask, L.E32, a, s);
}

hipError_t launch_march_pre(const MgLevelView& L, float w, const float* b, const MgLevelView& C,
                            float* xout, float* bc, const PcgScalars* sc, const MgFusedUpdate* upd,
                            hipStream_t s) {
    if (!halves(L.g, C.g) || (upd && (!upd->sc || upd->sc != sc))) return hipErrorInvalidValue;
    MarchArgs a{};
    a.a = b;
    a.dinv = L.dinv;
    a.out = xout;
    a.bc = bc;
    a.cmask = C.fixmask;
    a.gc = C.g;
    a.w = w;
    a.wdev = L.wdev;
    a.sc = const_cast<PcgScalars*>(sc);
    if (upd) a.upd = *upd;
    return upd ? launch_march<kMPre, true>(L.g, L.op, L.fixmask, L.E32, a, s)
               : launch_march<kMPre, false>(L.g, L.op, L.fixmask, L.E32, a, s);
}

}  // namespace tohip
