// BF16 implicit-GEMM 3D convolution on MFMA (FP32 accumulate) and the
// element-wise kernels of the learned warm-start network.
//
// Layout: activations are NDHWC (channel fastest), BF16, with a multiple of
// 8 channels.  Weights of a conv with T = kd*kh*kw taps are [Cout][T][Cin32]
// BF16 with Cin32 = Cin rounded up to 32 (zero padded).
//
// Forward (stride 1, zero padding): Y[p][co] = act(b[co] + sum_{tap, ci}
//   W[co][tap][ci] X[p + tap - pad][ci]) as a GEMM with M = output positions,
//   N = Cout, K = taps x channels.  One wave owns 16 positions x 16*NSUB
//   channels and issues v_mfma_f32_16x16x32_bf16; operand lanes follow the
//   instruction's layout: A[m = lane%16][k = 8*(lane/16) + 0..7],
//   B[k = 8*(lane/16) + 0..7][n = lane%16], D[m = 4*(lane/16) + 0..3][n = lane%16].
// Backward-data is the same kernel on dY with the tap-flipped, channel-
//   transposed weights Wt[ci][T-1-tap][co] and padding k-1-pad.
// Backward-weight: dW[co][tap][ci] = sum_p dY[p][co] X[p + tap - pad][ci], a
//   GEMM with K = positions, split over position ranges into FP32 partials
//   that a second kernel sums in a fixed order (deterministic).
#include <stdint.h>

#include <algorithm>
#include <cstdlib>

#include "k_common.h"
#include "nn_internal.h"

namespace tohip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }

// Round to nearest even (NaN kept quiet).
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return (uint16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ bf16x8 load8(const uint16_t* p) {
    return *reinterpret_cast<const bf16x8*>(p);
}

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }
// dA silu'(z) of the two bf16 values
__device__ __forceinline__ uint16_t silu_bwd(uint16_t dA, uint16_t zb) {
    const float z = bf2f(zb);
    const float sg = 1.0f / (1.0f + __expf(-z));
    return f2bf(bf2f(dA) * sg * (1.0f + z * (1.0f - sg)));
}

// ---------------------------------------------------------------- forward --
// The K dimension is walked in groups of 8 channels of one tap: group g is
// (tap = g / gpt, channels 8 (g % gpt) .. +7) with gpt = Cin / 8 groups per
// tap.  One 32-wide MFMA K-step takes 4 consecutive groups (one per 16-lane
// quarter of the wave), which may belong to different taps: a narrow input
// (8, 16, 48 channels) is packed across taps instead of padded to 32
// channels with zeros (the weights' zero padding past Cin is never read).
//
// Block = 4 waves on 16 output positions x 16*NSUB output channels.  The waves
// share the position tile and take every 4th K-step; the 4 partial accumulators are
// summed through LDS in wave order: for the coarse layers, where tiles of more
// positions cannot fill the chip, many blocks and a short load -> MFMA chain.
constexpr int kConvMaxTaps = 32;

template <int NSUB, bool BWD>
__global__ __launch_bounds__(256) void k_conv_fwd(ConvDesc c, const uint16_t* __restrict__ X,
                                                  const uint16_t* __restrict__ W,
                                                  const float* __restrict__ bias,
                                                  uint16_t* __restrict__ Y,
                                                  uint16_t* __restrict__ Z,
                                                  float* __restrict__ Yf) {
    __shared__ int4 taps[kConvMaxTaps];  // dz, dy, dx, element offset of the tap
    constexpr int KS = 4;
    __shared__ f4 red[KS - 1][NSUB][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 15, kq = lane >> 4;
    const int T = c.kd * c.kh * c.kw;
    if ((int)threadIdx.x < T) {
        const int t = threadIdx.x;
        const int dz = t / (c.kh * c.kw), dy = (t / c.kw) % c.kh, dx = t % c.kw;
        taps[t] = make_int4(dz, dy, dx, ((dz * c.H + dy) * c.W + dx) * c.Cin);
    }
    __syncthreads();
    const int64_t P = (int64_t)c.B * c.OD * c.OH * c.OW;
    const int64_t p0 = (int64_t)blockIdx.x * 16;
    const int co0 = blockIdx.y * 16 * NSUB;

    // this lane's A row: output position p0 + row
    const int64_t p = p0 + row;
    const bool pvalid = p < P;
    int ox = 0, oy = 0, oz = 0, bt = 0;
    if (pvalid) {
        int64_t t = p;
        ox = (int)(t % c.OW); t /= c.OW;
        oy = (int)(t % c.OH); t /= c.OH;
        oz = (int)(t % c.OD); bt = (int)(t / c.OD);
    }
    // element index of input voxel (oz - pd, oy - ph, ox - pw); a tap adds taps[].w
    const int64_t xbase =
        ((((int64_t)bt * c.D + oz - c.pd) * c.H + oy - c.ph) * c.W + ox - c.pw) * c.Cin;
    const int gpt = c.Cin / 8;
    const float inv_gpt = 1.0f / (float)gpt;
    const int S = (T * gpt + 3) / 4;  // K-steps
    int64_t wrow[NSUB];
#pragma unroll
    for (int j = 0; j < NSUB; ++j) {
        const int co = co0 + 16 * j + row;
        wrow[j] = co < c.Cout ? (int64_t)co * T * c.Cin32 : -1;
    }

    f4 acc[NSUB];
#pragma unroll
    for (int j = 0; j < NSUB; ++j) acc[j] = f4{0.f, 0.f, 0.f, 0.f};
    const bf16x8 zero = {};
    // U K-steps per iteration: all their loads are issued before the MFMAs,
    // so a wave keeps U gathers in flight (steps past S load zeros).
    constexpr int U = NSUB >= 4 ? 2 : 4;
    for (int s0 = wave; s0 < S; s0 += U * KS) {
        bf16x8 a[U], bv[U][NSUB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int g = 4 * (s0 + u * KS) + kq;
            // g / gpt, exact: (g + 0.5) / gpt is at least 0.5 / gpt from an integer
            const int tap = (int)(((float)g + 0.5f) * inv_gpt);
            const int ci = 8 * (g - tap * gpt);
            a[u] = zero;
            const bool tok = tap < T;
            if (tok) {
                const int4 td = taps[tap];
                const int iz = oz + td.x - c.pd, iy = oy + td.y - c.ph, ix = ox + td.z - c.pw;
                if (pvalid && iz >= 0 && iz < c.D && iy >= 0 && iy < c.H &&
                    ix >= 0 && ix < c.W)
                    a[u] = load8(X + xbase + td.w + ci);
            }
#pragma unroll
            for (int j = 0; j < NSUB; ++j)
                bv[u][j] = (tok && wrow[j] >= 0)
                               ? load8(W + wrow[j] + (int64_t)tap * c.Cin32 + ci)
                               : zero;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < NSUB; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], bv[u][j], acc[j], 0, 0, 0);
    }
    if (wave > 0)
#pragma unroll
        for (int j = 0; j < NSUB; ++j) red[wave - 1][j][lane] = acc[j];
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < KS - 1; ++w)
#pragma unroll
        for (int j = 0; j < NSUB; ++j) acc[j] += red[w][j][lane];
#pragma unroll
    for (int j = 0; j < NSUB; ++j) {
        const int co = co0 + 16 * j + row;
        if (co >= c.Cout) continue;
        const float bb = bias ? bias[co] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t pos = p0 + 4 * kq + i;
            if (pos >= P) continue;
            const float z = acc[j][i] + bb;
            const float y = c.act == 1 ? silu(z) : z;
            if (Yf) {
                if (co < c.out_cvalid) Yf[pos * c.out_cvalid + co] = y;
            } else {
                Y[pos * c.out_cstride + c.out_coff + co] =
                    BWD ? silu_bwd(f2bf(y), Z[pos * c.Cout + co]) : f2bf(y);
            }
            if (!BWD && Z) Z[pos * c.Cout + co] = f2bf(z);
        }
    }
}

// ---- forward from LDS tiles ----
// A workgroup stages its output tile's input places with their halo, 32 (16, 8)
// channels at a time, and reads every tap's operand from there; the kernel above
// gathers each of the K^3 taps from memory again.  An M tile is 8 x by 2 y
// positions of one z; the workgroup's 4 waves own MT each (8 x 4 x 2, 8 x 8 x 2 or
// 8 x 8 x 4 outputs) and all of NT x 16 output channels: per K-step of 32 MT LDS
// reads and NT weight loads (16 bytes a lane, the next step's in flight) for MT x NT
// MFMAs.  A K-step is one tap's 32 channels, two taps' 16 or four taps' 8.  Places
// are padded by 16 bytes (80, 48; 16 for 8 channels), which spreads 8 x 2 places
// over the banks and keeps the taps' offsets immediate.  Outputs of neighbouring
// lanes are paired into 4-byte stores.
template <int CK>
constexpr int kFwdPitch = CK == 8 ? 16 : CK * 2 + 16;  // bytes of a staged place

// BWD (act 2) is a form of its own: its epilogue as a branch cost a prediction 1-2 %.
template <int K, int NT, int MT, bool BWD>
__global__ __launch_bounds__(256) void k_conv_tile(ConvDesc c, int ntx, int nty, int ntz,
                                                   const uint16_t* __restrict__ X,
                                                   const uint16_t* __restrict__ W,
                                                   const float* __restrict__ bias,
                                                   uint16_t* __restrict__ Y,
                                                   uint16_t* __restrict__ Z,
                                                   float* __restrict__ Yf) {
    constexpr int BY = MT == 1 ? 4 : 8, BZ = MT == 4 ? 4 : 2, T = K * K * K;
    constexpr int HX = 8 + K - 1, HY = BY + K - 1, HZ = BZ + K - 1, NPL = HX * HY * HZ;
    __shared__ __align__(16) char lds[NPL * kFwdPitch<32>];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 15, kq = lane >> 4;
    int t = xcd_remap(blockIdx.x, gridDim.x);
    const int x0 = (t % ntx) * 8;
    t /= ntx;
    const int y0 = (t % nty) * BY;
    t /= nty;
    const int z0 = (t % ntz) * BZ, bt = t / ntz;
    const int co0 = blockIdx.y * 16 * NT;
    // the wave's M tiles: z and the first y pair
    const int wz = MT == 4 ? wave : wave & 1, wy = MT == 4 ? 0 : (wave >> 1) * 2 * MT;
    const int place0 = (wz * HY + wy + (row >> 3)) * HX + (row & 7);

    f4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = f4{0.f, 0.f, 0.f, 0.f};
    const uint16_t* wrow[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
        wrow[n] = W + (int64_t)min(co0 + 16 * n + row, c.Cout - 1) * T * c.Cin32;

    auto chunk = [&](auto ck, int c0) {
        constexpr int CK = decltype(ck)::value, G = CK / 8, P = kFwdPitch<CK>;
        constexpr int TS = 4 / G, S = (T + TS - 1) / TS;  // taps a K-step, K-steps
        // this lane's share of K-step s: tap TS s + kq / G, channels 8 (kq % G) ..
        const int lt = kq / G, lc = 8 * (kq % G);
        auto weights = [&](int tap, bf16x8 (&b)[NT]) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
                b[n] = load8(wrow[n] + min(tap, T - 1) * c.Cin32 + c0 + lc);
        };
        bf16x8 bn[CK == 32 ? K : 1][NT];
#pragma unroll
        for (int q = 0; q < (CK == 32 ? K : 1); ++q) weights(q + lt, bn[q]);
        __syncthreads();  // the previous chunk's reads
        for (int it = tid; it < NPL * G; it += 256) {
            const int pl = it / G, ch = c0 + 8 * (it % G);
            const int x = x0 - c.pw + pl % HX, y = y0 - c.ph + (pl / HX) % HY,
                      z = z0 - c.pd + pl / (HX * HY);
            uint4 v = make_uint4(0, 0, 0, 0);
            if (x >= 0 && x < c.W && y >= 0 && y < c.H && z >= 0 && z < c.D)
                v = *reinterpret_cast<const uint4*>(
                    X + ((((int64_t)bt * c.D + z) * c.H + y) * c.W + x) * c.Cin + ch);
            *reinterpret_cast<uint4*>(lds + pl * P + 16 * (it % G)) = v;
        }
        __syncthreads();
        const char* base = lds + place0 * P + 2 * lc;
        if constexpr (CK == 32) {
            // a K-step is a tap; a row of K taps at a time, the next row's weights in
            // flight (unrolled whole, every weight is loaded first: 256 registers)
#pragma unroll 1
            for (int r = 0; r < K * K; ++r) {
                bf16x8 bw[K][NT];
#pragma unroll
                for (int q = 0; q < K; ++q)
#pragma unroll
                    for (int n = 0; n < NT; ++n) bw[q][n] = bn[q][n];
                if (r + 1 < K * K)
#pragma unroll
                    for (int q = 0; q < K; ++q) weights((r + 1) * K + q, bn[q]);
                const char* at = base + ((r / K) * HY + r % K) * HX * P;
#pragma unroll
                for (int q = 0; q < K; ++q)
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        const bf16x8 av =
                            *reinterpret_cast<const bf16x8*>(at + (2 * m * HX + q) * P);
#pragma unroll
                        for (int n = 0; n < NT; ++n)
                            acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                av, bw[q][n], acc[m][n], 0, 0, 0);
                    }
            }
        } else {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                bf16x8 bw[NT];
#pragma unroll
                for (int n = 0; n < NT; ++n) bw[n] = bn[0][n];
                if (s + 1 < S) weights(TS * (s + 1) + lt, bn[0]);
                int off = 0;
#pragma unroll
                for (int q = 0; q < TS; ++q) {
                    const int tap = TS * s + q < T ? TS * s + q : 0;
                    const int o = P * (((tap / (K * K)) * HY + (tap / K) % K) * HX + tap % K);
                    off = q == 0 || lt >= q ? o : off;
                }
                const bool on = TS * s + lt < T;  // taps past the kernel: 0
                const bf16x8 zero = {};
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    bf16x8 av = *reinterpret_cast<const bf16x8*>(base + off + 2 * m * HX * P);
                    if (TS * s + TS > T && !on) av = zero;
#pragma unroll
                    for (int n = 0; n < NT; ++n)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bw[n], acc[m][n],
                                                                            0, 0, 0);
                }
            }
        }
    };
    int c0 = 0;
    for (; c0 + 32 <= c.Cin; c0 += 32) chunk(std::integral_constant<int, 32>{}, c0);
    if (c0 + 16 <= c.Cin) {
        chunk(std::integral_constant<int, 16>{}, c0);
        c0 += 16;
    }
    if (c0 < c.Cin) chunk(std::integral_constant<int, 8>{}, c0);

    // D[m = 4 kq + i][n = row]
    const int z = z0 + wz;
    if (z >= c.OD) return;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int y = y0 + wy + 2 * m + (kq >> 1);
        if (y >= c.OH) continue;
        const int64_t line = (((int64_t)bt * c.OD + z) * c.OH + y) * c.OW;
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int co = co0 + 16 * n + row;
            const float bb = bias && co < c.Cout ? bias[co] : 0.f;
            float zv[4], yv[4];
            uint16_t zb[4] = {};
            if (BWD)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int x = min(x0 + 4 * (kq & 1) + i, c.OW - 1);
                    zb[i] = Z[(line + x) * c.Cout + min(co, c.Cout - 1)];
                }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                zv[i] = acc[m][n][i] + bb;
                yv[i] = c.act == 1 ? silu(zv[i]) : zv[i];
                if (BWD) yv[i] = bf2f(silu_bwd(f2bf(yv[i]), zb[i]));
            }
            if (Yf)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int x = x0 + 4 * (kq & 1) + i;
                    if (x < c.OW && co < c.out_cvalid) Yf[(line + x) * c.out_cvalid + co] = yv[i];
                }
            // an even lane stores position i of both channels, its odd neighbour
            // position i + 1
            const bool odd = row & 1;
            auto store = [&](const float (&v)[4], uint16_t* out, int stride, int off) {
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const uint32_t own = f2bf(odd ? v[i + 1] : v[i]),
                                   send = f2bf(odd ? v[i] : v[i + 1]);
                    const uint32_t got = __builtin_amdgcn_update_dpp(0, (int)send, 0xB1, 0xf, 0xf,
                                                                     true);  // of lane ^ 1
                    const int x = x0 + 4 * (kq & 1) + i + (odd ? 1 : 0);
                    if (x < c.OW && co < c.Cout)
                        *reinterpret_cast<uint32_t*>(out + (line + x) * stride + off + (co & ~1)) =
                            odd ? got | own << 16 : own | got << 16;
                }
            };
            if (!Yf) store(yv, Y, c.out_cstride, c.out_coff);
            if (!BWD && Z) store(zv, Z, c.Cout, 0);
        }
    }
}

template <int K, int NT, int MT>
static hipError_t launch_conv_tile(const ConvDesc& c, const uint16_t* X, const uint16_t* W,
                                   const float* bias, uint16_t* Y, uint16_t* Z, float* Yf,
                                   hipStream_t s) {
    constexpr int BY = MT == 1 ? 4 : 8, BZ = MT == 4 ? 4 : 2;
    const int ntx = (c.OW + 7) / 8, nty = (c.OH + BY - 1) / BY, ntz = (c.OD + BZ - 1) / BZ;
    const dim3 grid((unsigned)(ntx * nty * ntz * c.B), (c.Cout + 16 * NT - 1) / (16 * NT));
    if (c.act == 2)
        hipLaunchKernelGGL((k_conv_tile<K, NT, MT, true>), grid, dim3(256), 0, s, c, ntx, nty, ntz,
                           X, W, bias, Y, Z, Yf);
    else
        hipLaunchKernelGGL((k_conv_tile<K, NT, MT, false>), grid, dim3(256), 0, s, c, ntx, nty, ntz,
                           X, W, bias, Y, Z, Yf);
    return hipGetLastError();
}

// The LDS-tile kernel with the largest tile that still gives a workgroup per CU;
// with the smallest, fewer output channels a workgroup until there are two per CU
// (all of an output's channels from one staging otherwise).  The split kernel (16
// positions a workgroup, the K-steps over its waves) below half a workgroup per CU,
// and for kernels and channel counts that the network has not.  MI355X, all forward
// and input-gradient convolutions of 12 training steps at 64x32x32, batch 8, and 6
// predictions at 120x40x40: 9.7 ms; with at least 256 / 512 / 1024 workgroups for the
// large tiles and all channels a workgroup 10.3 / 10.4 / 11.3; a workgroup per CU for
// the channels 10.0; never the split kernel 9.9; gathers from memory alone 15.6.
hipError_t launch_conv_fwd(const ConvDesc& c, const uint16_t* X, const uint16_t* W,
                           const float* bias, uint16_t* Y, uint16_t* Z, float* Yf,
                           hipStream_t s) {
    const int T = c.kd * c.kh * c.kw;
    if (T > kConvMaxTaps || c.Cin % 8 != 0 || c.Cin32 % 32 != 0 || c.Cin > c.Cin32)
        return hipErrorInvalidValue;
    const bool cube3 = c.kd == 3 && c.kh == 3 && c.kw == 3,
               cube2 = c.kd == 2 && c.kh == 2 && c.kw == 2;
    const int ct = (c.Cout + 15) / 16;
    int nt = ct % 4 == 0 ? 4 : ct % 3 == 0 ? 3 : ct % 2 == 0 ? 2 : 1;
    if (c.Cout % 8 == 0 && (cube3 || (cube2 && ct == 1)) &&
        (Yf || (c.out_cstride % 2 == 0 && c.out_coff % 2 == 0))) {
        auto blocks = [&](int by, int bz) {
            return (int64_t)c.B * ((c.OW + 7) / 8) * ((c.OH + by - 1) / by) *
                   ((c.OD + bz - 1) / bz) * (ct / nt);
        };
        int mt = blocks(8, 4) >= 256 ? 4 : blocks(8, 2) >= 256 ? 2 : 1;
        while (mt == 1 && nt > 1 && blocks(4, 2) < 512) nt = nt == 4 ? 2 : 1;
        if (mt == 1 && blocks(4, 2) < 128) mt = 0;
#define TOHIP_CT(K, N)                                                                         \
    (mt == 4   ? launch_conv_tile<K, N, 4>(c, X, W, bias, Y, Z, Yf, s)                         \
     : mt == 2 ? launch_conv_tile<K, N, 2>(c, X, W, bias, Y, Z, Yf, s)                         \
               : launch_conv_tile<K, N, 1>(c, X, W, bias, Y, Z, Yf, s))
        if (mt) {
            if (cube2) return TOHIP_CT(2, 1);
            return nt == 4 ? TOHIP_CT(3, 4) : nt == 3 ? TOHIP_CT(3, 3) : nt == 2 ? TOHIP_CT(3, 2)
                                                                                 : TOHIP_CT(3, 1);
        }
#undef TOHIP_CT
    }
    const int64_t P = (int64_t)c.B * c.OD * c.OH * c.OW;
    int nsub = c.Cout >= 64 ? 4 : c.Cout >= 32 ? 2 : 1;
    while (nsub > 1 && (P + 15) / 16 * ((c.Cout + 16 * nsub - 1) / (16 * nsub)) < 1024) nsub /= 2;
    const dim3 grid((unsigned)((P + 15) / 16), (unsigned)((c.Cout + 16 * nsub - 1) / (16 * nsub)));
#define TOHIP_CONV(NS)                                                                              \
    if (c.act == 2)                                                                                 \
        hipLaunchKernelGGL((k_conv_fwd<NS, true>), grid, dim3(256), 0, s, c, X, W, bias, Y, Z, Yf); \
    else                                                                                            \
        hipLaunchKernelGGL((k_conv_fwd<NS, false>), grid, dim3(256), 0, s, c, X, W, bias, Y, Z, Yf)
    if (nsub == 4) {
        TOHIP_CONV(4);
    } else if (nsub == 2) {
        TOHIP_CONV(2);
    } else {
        TOHIP_CONV(1);
    }
#undef TOHIP_CONV
    return hipGetLastError();
}

// ---------------------------------------------------------- weight grad --
// dW[co][tap][ci] = sum_p dY[p][co] X[p + tap - pad][ci] with the positions as the
// K dimension of the MFMA.  A lane's 8 consecutive k are the same place of 8
// separate spatial tiles ("subs"), so that in LDS, [place][16 channels][8 subs], an
// operand is one aligned 16-byte read for every tap's shift.  A K-step is 4
// consecutive y (the lane quarters) of the 8 subs.
//
// A workgroup takes 16 input channels, MC tiles of 16 output channels and every
// taps of units of 8 subs (8 x TY x TZ outputs each): it stages the inputs with
// their halo and the output gradients once (8 channels of 8 subs a thread,
// transposed in registers) and forms all K^3 taps from them.  A wave keeps one
// output tile's K^3 accumulators and walks x with a window of K inputs per (dz,
// dy) in registers: K^2 + 1 LDS reads for K^3 MFMAs.  Waves beyond the MC tiles
// take other (y, z) places; their sums are added through LDS in wave order.  The
// bias gradient is one more MFMA a step against ones.  Splits over the units are
// summed by k_conv_wgrad_sum in a fixed order.
//
// Bound by the staging (the halo is read 3 to 4 times from L2) and, per MFMA, by
// little else: MI355X, 64x32x32, batch 8, the weight and bias gradients of a step's
// 15 layers take 0.51 ms, against 2.34 ms for a wave per tap and 16 x 16 tile that
// gathered both operands again for every tap, with kernels of their own for the
// bias (140 TFLOP/s against 30).
constexpr int kWgTX = 8, kWgSubs = 8;

struct WgradShape {
    int ntx, nty, ntz, ntiles, nunits, ns, ct, it;
};

// 8 subs x 8 channels (one uint4 of 8 channels per sub) -> 8 channels x 8 subs.
__device__ __forceinline__ void transpose8(const uint4 (&r)[kWgSubs], uint4 (&o)[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        auto w = [&](int s) {
            return j == 0 ? r[s].x : j == 1 ? r[s].y : j == 2 ? r[s].z : r[s].w;
        };
        // bytes 0-1 (2-3) of both words: the even (odd) channel of two subs
        auto lo = [&](int s) { return __builtin_amdgcn_perm(w(s + 1), w(s), 0x05040100u); };
        auto hi = [&](int s) { return __builtin_amdgcn_perm(w(s + 1), w(s), 0x07060302u); };
        o[2 * j] = make_uint4(lo(0), lo(2), lo(4), lo(6));
        o[2 * j + 1] = make_uint4(hi(0), hi(2), hi(4), hi(6));
    }
}

template <int MC, int TY, int TZ, int K>
__global__ __launch_bounds__(256) void k_conv_wgrad(ConvDesc c, WgradShape sh,
                                                    const uint16_t* __restrict__ X,
                                                    const uint16_t* __restrict__ dY,
                                                    float* __restrict__ part,
                                                    float* __restrict__ bpart) {
    constexpr int HX = kWgTX + K - 1, HY = TY + K - 1, HZ = TZ + K - 1, T = K * K * K;
    constexpr int NX = HX * HY * HZ, NY = kWgTX * TY * TZ, PG = 4 / MC;
    static_assert((TY / 4) * TZ == PG, "a place group per wave");
    constexpr int kPl = 16 * kWgSubs;  // elements of a place: 16 channels x 8 subs
    extern __shared__ __align__(16) uint16_t wg_lds[];
    uint16_t* sx = wg_lds;            // [NX][16][8]
    uint16_t* sy = wg_lds + NX * kPl;  // [MC][NY][16][8]
    __shared__ int4 org[kWgSubs];     // first output of a sub and its batch (-1: none)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 15, kq = lane >> 4;
    const int m = wave % MC, pg = wave / MC, y0 = 4 * (pg % (TY / 4)), z0 = pg / (TY / 4);
    const int ci0 = blockIdx.z * 16, co0 = blockIdx.y * 16 * MC;

    f4 acc[T], accb = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    const uint32_t one2 = 0x3f803f80u;  // two BF16 ones
    const uint4 one4 = make_uint4(one2, one2, one2, one2);
    const bf16x8 ones = __builtin_bit_cast(bf16x8, one4);

    for (int u = blockIdx.x; u < sh.nunits; u += sh.ns) {
        __syncthreads();  // the previous unit's reads
        if (tid < kWgSubs) {
            int t = u * kWgSubs + tid;
            int4 o = make_int4(0, 0, 0, -1);
            if (t < sh.ntiles) {
                o.x = (t % sh.ntx) * kWgTX;
                t /= sh.ntx;
                o.y = (t % sh.nty) * TY;
                t /= sh.nty;
                o.z = (t % sh.ntz) * TZ;
                o.w = t / sh.ntz;
            }
            org[tid] = o;
        }
        __syncthreads();
        for (int it = tid; it < 2 * NX; it += 256) {
            const int pl = it >> 1, ch = ci0 + 8 * (it & 1);
            const int px = pl % HX - c.pw, py = (pl / HX) % HY - c.ph, pz = pl / (HX * HY) - c.pd;
            uint4 r[kWgSubs], o[8];
#pragma unroll
            for (int s = 0; s < kWgSubs; ++s) {
                const int4 g = org[s];
                const int x = g.x + px, y = g.y + py, z = g.z + pz;
                r[s] = make_uint4(0, 0, 0, 0);
                if (ch < c.Cin && g.w >= 0 && x >= 0 && x < c.W && y >= 0 && y < c.H && z >= 0 &&
                    z < c.D)
                    r[s] = *reinterpret_cast<const uint4*>(
                        X + ((((int64_t)g.w * c.D + z) * c.H + y) * c.W + x) * c.Cin + ch);
            }
            transpose8(r, o);
            uint4* d = reinterpret_cast<uint4*>(sx + pl * kPl + (it & 1) * 8 * kWgSubs);
#pragma unroll
            for (int j = 0; j < 8; ++j) d[j] = o[j];
        }
        for (int it = tid; it < 2 * MC * NY; it += 256) {
            const int q = it >> 1, pl = q % NY, ch = co0 + 16 * (q / NY) + 8 * (it & 1);
            const int px = pl % kWgTX, py = (pl / kWgTX) % TY, pz = pl / (kWgTX * TY);
            uint4 r[kWgSubs], o[8];
#pragma unroll
            for (int s = 0; s < kWgSubs; ++s) {
                const int4 g = org[s];
                const int x = g.x + px, y = g.y + py, z = g.z + pz;
                r[s] = make_uint4(0, 0, 0, 0);
                if (ch < c.Cout && g.w >= 0 && x < c.OW && y < c.OH && z < c.OD)
                    r[s] = *reinterpret_cast<const uint4*>(
                        dY + ((((int64_t)g.w * c.OD + z) * c.OH + y) * c.OW + x) * c.Cout + ch);
            }
            transpose8(r, o);
            uint4* d = reinterpret_cast<uint4*>(sy + q * kPl + (it & 1) * 8 * kWgSubs);
#pragma unroll
            for (int j = 0; j < 8; ++j) d[j] = o[j];
        }
        __syncthreads();
        const uint16_t* xr = sx + ((z0 * HY + y0 + kq) * HX) * kPl + row * kWgSubs;
        const uint16_t* yr = sy + ((m * TZ + z0) * TY + y0 + kq) * kWgTX * kPl + row * kWgSubs;
        bf16x8 win[K][K][K];  // [dz][dy][x mod K]
#pragma unroll
        for (int x = 0; x < HX; ++x) {
#pragma unroll
            for (int dz = 0; dz < K; ++dz)
#pragma unroll
                for (int dy = 0; dy < K; ++dy)
                    win[dz][dy][x % K] = load8(xr + ((dz * HY + dy) * HX + x) * kPl);
            if (x < K - 1) continue;
            const int xo = x - (K - 1);
            const bf16x8 av = load8(yr + xo * kPl);
            accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, ones, accb, 0, 0, 0);
#pragma unroll
            for (int t = 0; t < T; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    av, win[t / (K * K)][(t / K) % K][(xo + t % K) % K], acc[t], 0, 0, 0);
        }
    }
    if (PG > 1) {  // the place groups of an output tile, in order
        float4* red = reinterpret_cast<float4*>(wg_lds);
        for (int p = 1; p < PG; ++p) {
            __syncthreads();
            if (pg == p) {
#pragma unroll
                for (int t = 0; t < T; ++t)
                    red[(m * (T + 1) + t) * 64 + lane] =
                        make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
                red[(m * (T + 1) + T) * 64 + lane] =
                    make_float4(accb[0], accb[1], accb[2], accb[3]);
            }
            __syncthreads();
            if (pg == 0) {
#pragma unroll
                for (int t = 0; t <= T; ++t) {
                    const float4 v = red[(m * (T + 1) + t) * 64 + lane];
                    f4& d = t < T ? acc[t < T ? t : 0] : accb;
                    d += f4{v.x, v.y, v.z, v.w};
                }
            }
        }
        if (pg > 0) return;
    }
    // D[co = 4 kq + i][ci = row] of every tap
    const int tile = blockIdx.y * MC + m;
    if (tile >= sh.ct) return;
    float4* out = reinterpret_cast<float4*>(part) +
                  (((int64_t)blockIdx.x * sh.ct + tile) * sh.it + blockIdx.z) * T * 64 + lane;
#pragma unroll
    for (int t = 0; t < T; ++t)
        out[t * 64] = make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
    if (blockIdx.z == 0 && row == 0)
        reinterpret_cast<float4*>(bpart)[((int64_t)blockIdx.x * sh.ct + tile) * 4 + kq] =
            make_float4(accb[0], accb[1], accb[2], accb[3]);
}

// dW[co][tap][ci] and db[co] from the splits' partials.  Block (ct, it, tap): 64
// lanes as the MFMA leaves the 16 x 16 tile, times Q shares of the splits, added
// in order; the last ct blocks: the bias.  A share is a chain of round trips of 8
// loads: 16 shares from 64 splits on, 8.7 -> 6.1 us on average over the 15 layers at
// 64x32x32, batch 8 (line at 32: 6.3).
template <int Q>
__global__ __launch_bounds__(64 * Q) void k_conv_wgrad_sum(ConvDesc c, WgradShape sh, int T,
                                                        const float* __restrict__ part,
                                                        const float* __restrict__ bpart,
                                                        float* __restrict__ dW,
                                                        float* __restrict__ db) {
    __shared__ float4 red[Q][64];
    const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int nb = sh.ct * sh.it * T, chunk = (sh.ns + Q - 1) / Q;
    const int s0 = q * chunk, s1 = min(s0 + chunk, sh.ns);
    const bool bias = (int)blockIdx.x >= nb;
    const int tile = blockIdx.x - nb;
    const float4* p = bias ? reinterpret_cast<const float4*>(bpart) + tile * 4 + (lane & 3)
                           : reinterpret_cast<const float4*>(part) + (int64_t)blockIdx.x * 64 + lane;
    const int64_t stride = bias ? sh.ct * 4 : (int64_t)nb * 64;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    constexpr int U = 8;
    for (int s = s0; s < s1; s += U) {
        float4 v[U];
#pragma unroll
        for (int k = 0; k < U; ++k) v[k] = p[(int64_t)min(s + k, s1 - 1) * stride];
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (s + k < s1) {
                a.x += v[k].x;
                a.y += v[k].y;
                a.z += v[k].z;
                a.w += v[k].w;
            }
    }
    red[q][lane] = a;
    __syncthreads();
    if (q != 0) return;
    a = red[0][lane];
#pragma unroll
    for (int k = 1; k < Q; ++k) {
        const float4 v = red[k][lane];
        a.x += v.x;
        a.y += v.y;
        a.z += v.z;
        a.w += v.w;
    }
    const float e[4] = {a.x, a.y, a.z, a.w};
    if (bias) {
        if (lane < 4)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int co = tile * 16 + 4 * lane + i;
                if (co < c.Cout && db) db[co] = e[i];
            }
        return;
    }
    const int t = blockIdx.x % T, it = (blockIdx.x / T) % sh.it, ct = blockIdx.x / (T * sh.it);
    const int ci = it * 16 + (lane & 15);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int co = ct * 16 + 4 * (lane >> 4) + i;
        if (co < c.Cout && ci < c.Cin) dW[((int64_t)co * T + t) * c.Cin + ci] = e[i];
    }
}

// Output tiles a workgroup: 4 of 16 channels from Cout = 64 on, 2 from 32 on, else
// 1 with four place groups.  About 512 workgroups, at most one split a unit.
static int wgrad_mc(int Cout) { return Cout >= 64 ? 4 : Cout >= 32 ? 2 : 1; }
static WgradShape wgrad_shape(const ConvDesc& c) {
    const int mc = wgrad_mc(c.Cout);
    const int ty = mc == 1 ? 8 : 4, tz = mc == 4 ? 1 : 2;
    WgradShape s;
    s.ntx = (c.OW + kWgTX - 1) / kWgTX;
    s.nty = (c.OH + ty - 1) / ty;
    s.ntz = (c.OD + tz - 1) / tz;
    s.ntiles = s.ntx * s.nty * s.ntz * c.B;
    s.nunits = (s.ntiles + kWgSubs - 1) / kWgSubs;
    s.ct = (c.Cout + 15) / 16;
    s.it = (c.Cin + 15) / 16;
    const int per = (s.ct + mc - 1) / mc * s.it;
    s.ns = std::max(1, std::min(s.nunits, 512 / per));
    return s;
}
size_t conv_bwd_w_floats(const ConvDesc& c) {
    const WgradShape s = wgrad_shape(c);
    return (size_t)s.ns * s.ct * (size_t)(s.it * c.kd * c.kh * c.kw * 256 + 16);
}

template <int MC, int TY, int TZ, int K>
static hipError_t launch_wgrad(const ConvDesc& c, const WgradShape& sh, const uint16_t* X,
                               const uint16_t* dY, float* part, float* bpart, hipStream_t s) {
    constexpr int HX = kWgTX + K - 1, HY = TY + K - 1, HZ = TZ + K - 1, T = K * K * K;
    constexpr int stage = (HX * HY * HZ + MC * kWgTX * TY * TZ) * 256;
    constexpr int sums = MC < 4 ? MC * (T + 1) * 64 * 16 : 0;
    constexpr int lds = stage > sums ? stage : sums;
    static_assert(lds <= 159 * 1024, "LDS of a CU");
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(&k_conv_wgrad<MC, TY, TZ, K>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_conv_wgrad<MC, TY, TZ, K>), dim3(sh.ns, (sh.ct + MC - 1) / MC, sh.it),
                       dim3(256), lds, s, c, sh, X, dY, part, bpart);
    return hipGetLastError();
}

hipError_t launch_conv_bwd_w(const ConvDesc& c, const uint16_t* X, const uint16_t* dY,
                             float* part, float* dW, float* db, hipStream_t s) {
    const int k = c.kd, mc = wgrad_mc(c.Cout), T = k * k * k;
    if (c.kh != k || c.kw != k || k < 1 || k > 3 || c.Cin % 8 || c.Cout % 8 || 256 % c.Cout ||
        reinterpret_cast<uintptr_t>(X) % 16 || reinterpret_cast<uintptr_t>(dY) % 16)
        return hipErrorInvalidValue;
    const WgradShape sh = wgrad_shape(c);
    float* bpart = part + (size_t)sh.ns * sh.ct * sh.it * T * 256;
    hipError_t e;
#define TOHIP_WG(K)                                                                        \
    (mc == 4 ? launch_wgrad<4, 4, 1, K>(c, sh, X, dY, part, bpart, s)                      \
     : mc == 2 ? launch_wgrad<2, 4, 2, K>(c, sh, X, dY, part, bpart, s)                    \
               : launch_wgrad<1, 8, 2, K>(c, sh, X, dY, part, bpart, s))
    e = k == 3 ? TOHIP_WG(3) : k == 2 ? TOHIP_WG(2) : TOHIP_WG(1);
#undef TOHIP_WG
    if (e != hipSuccess) return e;
    const dim3 grid(sh.ct * sh.it * T + sh.ct);
    if (sh.ns >= 64)
        hipLaunchKernelGGL(k_conv_wgrad_sum<16>, grid, dim3(1024), 0, s, c, sh, T, part, bpart, dW,
                           db);
    else
        hipLaunchKernelGGL(k_conv_wgrad_sum<4>, grid, dim3(256), 0, s, c, sh, T, part, bpart, dW,
                           db);
    return hipGetLastError();
}

// --------------------------------------------------- weight conversions --
// Master FP32 [Cout][T][Cin] -> BF16 forward [Cout][T][Cin32] and
// backward-data Wt[Cin][T-1-tap][Cout32], every layer of the table in one launch
// (blockIdx.y): 15 launches of 4.5 us each took longer than the work.  Layers are below
// 2^31 weights (padded ones included).
__global__ void k_weights_to_bf16(ConvWeights t) {
    const ConvWeights::Layer l = t.layer[blockIdx.y];
    const int n = l.Cout * l.T * l.Cin32, nt = l.Cin * l.T * l.Cout32;
    const int step = gridDim.x * blockDim.x;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n || i < nt; i += step) {
        if (i < n) {
            const int r = i / l.Cin32, ci = i - r * l.Cin32;  // r = co T + tap
            l.wf[i] = f2bf(ci < l.Cin ? l.w[r * l.Cin + ci] : 0.f);
        }
        if (l.wt && i < nt) {
            const int r = i / l.Cout32, co = i - r * l.Cout32;
            const int ci = r / l.T, tap = l.T - 1 - (r - ci * l.T);
            l.wt[i] = f2bf(co < l.Cout ? l.w[(co * l.T + tap) * l.Cin + ci] : 0.f);
        }
    }
}

hipError_t launch_weights_to_bf16(const ConvWeights& t, hipStream_t s) {
    if (t.count < 1 || t.count > ConvWeights::kMax) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_weights_to_bf16, dim3(512, t.count), dim3(256), 0, s, t);
    return hipGetLastError();
}

// Samples idx[0..count) of the data set into the batch: sample b of dst_f / dst_u
// from sample idx[b], nf 16-byte words and nu floats each (blockIdx.y = b).
__global__ void k_nn_gather(NNBatch t, int64_t nf, const uint4* __restrict__ src_f,
                            uint4* __restrict__ dst_f, int64_t nu, const float* __restrict__ src_u,
                            float* __restrict__ dst_u) {
    const int64_t b = blockIdx.y, from = t.idx[blockIdx.y];
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nf || i < nu; i += step) {
        if (i < nf) dst_f[b * nf + i] = src_f[from * nf + i];
        if (i < nu) dst_u[b * nu + i] = src_u[from * nu + i];
    }
}

hipError_t launch_nn_gather(const NNBatch& t, int64_t nf, const void* src_f, void* dst_f, int64_t nu,
                            const float* src_u, float* dst_u, hipStream_t s) {
    if (t.count < 1 || t.count > NNBatch::kMax) return hipErrorInvalidValue;
    const int64_t n = nf > nu ? nf : nu, nb = (n + 255) / 256;
    hipLaunchKernelGGL(k_nn_gather, dim3((unsigned)(nb < 1024 ? nb : 1024), t.count), dim3(256), 0,
                       s, t, nf, (const uint4*)src_f, (uint4*)dst_f, nu, src_u, dst_u);
    return hipGetLastError();
}

// -------------------------------------------------------- element-wise --
// dZ = dA * silu'(z)
__global__ void k_silu_bwd(int64_t n, const uint16_t* __restrict__ dA,
                           const uint16_t* __restrict__ Z, uint16_t* __restrict__ dZ) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        dZ[i] = silu_bwd(dA[i], Z[i]);
    }
}

// 8 channels
union Bf8 {
    uint4 q;
    uint16_t v[8];
};

// Strided channel view helpers: tensor [P][cstride], view [coff, coff + C).
// 2x2x2 average pool: out (B, D/2, H/2, W/2, C) from in (B, D, H, W) view, 8
// channels (16 bytes) a thread; C, in_cs and in_co multiples of 8.
__global__ void k_avgpool_fwd(int B, int D, int H, int W, int C, const uint16_t* __restrict__ in,
                              int in_cs, int in_co, uint16_t* __restrict__ out) {
    const int C8 = C / 8;
    const int64_t n = (int64_t)B * (D / 2) * (H / 2) * (W / 2) * C8;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ch = 8 * (int)(i % C8);
        int64_t t = i / C8;
        const int64_t o = t * C + ch;
        const int x = (int)(t % (W / 2)); t /= (W / 2);
        const int y = (int)(t % (H / 2)); t /= (H / 2);
        const int z = (int)(t % (D / 2));
        const int b = (int)(t / (D / 2));
        Bf8 v[8], r;
#pragma unroll
        for (int c8 = 0; c8 < 8; ++c8) {
            const int zz = 2 * z + ((c8 >> 2) & 1), yy = 2 * y + ((c8 >> 1) & 1),
                      xx = 2 * x + (c8 & 1);
            v[c8].q = *reinterpret_cast<const uint4*>(
                in + ((((int64_t)b * D + zz) * H + yy) * W + xx) * in_cs + in_co + ch);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float s = 0.f;
#pragma unroll
            for (int c8 = 0; c8 < 8; ++c8) s += bf2f(v[c8].v[e]);
            r.v[e] = f2bf(0.125f * s);
        }
        *reinterpret_cast<uint4*>(out + o) = r.q;
    }
}

// Output gradient of a layer whose activation goes on as a skip connection and
// through the 2x2x2 average pool: dZ (B, D, H, W, C) = (skip view + d pool / 8)
// silu'(Z), 8 channels (16 bytes) a thread; C, cs and co multiples of 8.  One pass
// of 8.7 us for three (pool gradient added into the view 18.6, copy 7.6, SiLU 8.5 us
// on average over the levels, 64x32x32, batch 8).
__global__ void k_skip_bwd(int B, int D, int H, int W, int C, const uint16_t* __restrict__ dpool,
                           const uint16_t* __restrict__ dskip, int cs, int co,
                           const uint16_t* __restrict__ Z, uint16_t* __restrict__ dZ) {
    const int C8 = C / 8;
    const int64_t n = (int64_t)B * D * H * W * C8;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ch = 8 * (int)(i % C8);
        const int64_t o = i / C8;
        int64_t t = o;
        const int x = (int)(t % W); t /= W;
        const int y = (int)(t % H); t /= H;
        const int z = (int)(t % D);
        const int b = (int)(t / D);
        Bf8 p, k, a, r;
        p.q = *reinterpret_cast<const uint4*>(
            dpool + ((((int64_t)b * (D / 2) + z / 2) * (H / 2) + y / 2) * (W / 2) + x / 2) * C + ch);
        k.q = *reinterpret_cast<const uint4*>(dskip + o * cs + co + ch);
        a.q = *reinterpret_cast<const uint4*>(Z + o * C + ch);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            r.v[e] = silu_bwd(f2bf(bf2f(k.v[e]) + 0.125f * bf2f(p.v[e])), a.v[e]);
        *reinterpret_cast<uint4*>(dZ + o * C + ch) = r.q;
    }
}

// nearest 2x upsample of in (B, D, H, W, C) into the view [coff, coff+C) of
// out (B, 2D, 2H, 2W, out_cs)
__global__ void k_upsample_fwd(int B, int D, int H, int W, int C, const uint16_t* __restrict__ in,
                               uint16_t* __restrict__ out, int out_cs, int out_co) {
    const int64_t n = (int64_t)B * 8 * D * H * W * C;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ch = (int)(i % C);
        int64_t t = i / C;
        const int x = (int)(t % (2 * W)); t /= (2 * W);
        const int y = (int)(t % (2 * H)); t /= (2 * H);
        const int z = (int)(t % (2 * D));
        const int b = (int)(t / (2 * D));
        out[((((int64_t)b * 2 * D + z) * 2 * H + y) * 2 * W + x) * out_cs + out_co + ch] =
            in[((((int64_t)b * D + z / 2) * H + y / 2) * W + x / 2) * C + ch];
    }
}

// The same with 8 channels (16 bytes) per thread: C, out_cs and out_co are
// multiples of 8 and the tensors 16-byte aligned.
__global__ void k_upsample_fwd8(int B, int D, int H, int W, int C, const uint16_t* __restrict__ in,
                                uint16_t* __restrict__ out, int out_cs, int out_co) {
    const int C8 = C / 8;
    const int64_t n = (int64_t)B * 8 * D * H * W * C8;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ch = 8 * (int)(i % C8);
        int64_t t = i / C8;
        const int x = (int)(t % (2 * W)); t /= (2 * W);
        const int y = (int)(t % (2 * H)); t /= (2 * H);
        const int z = (int)(t % (2 * D));
        const int b = (int)(t / (2 * D));
        *reinterpret_cast<uint4*>(
            out + ((((int64_t)b * 2 * D + z) * 2 * H + y) * 2 * W + x) * out_cs + out_co + ch) =
            *reinterpret_cast<const uint4*>(
                in + ((((int64_t)b * D + z / 2) * H + y / 2) * W + x / 2) * C + ch);
    }
}

// dZ (B, D, H, W, C) = silu'(Z) times the sum of the 8 children in the view of
// d out, 8 channels (16 bytes) a thread; C, out_cs and out_co multiples of 8.
__global__ void k_upsample_bwd(int B, int D, int H, int W, int C,
                               const uint16_t* __restrict__ dout, int out_cs, int out_co,
                               const uint16_t* __restrict__ Z, uint16_t* __restrict__ dZ) {
    const int C8 = C / 8;
    const int64_t n = (int64_t)B * D * H * W * C8;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int ch = 8 * (int)(i % C8);
        int64_t t = i / C8;
        const int64_t o = t * C + ch;
        const int x = (int)(t % W); t /= W;
        const int y = (int)(t % H); t /= H;
        const int z = (int)(t % D);
        const int b = (int)(t / D);
        Bf8 v[8], a, r;
#pragma unroll
        for (int c8 = 0; c8 < 8; ++c8) {
            const int zz = 2 * z + ((c8 >> 2) & 1), yy = 2 * y + ((c8 >> 1) & 1),
                      xx = 2 * x + (c8 & 1);
            v[c8].q = *reinterpret_cast<const uint4*>(
                dout + ((((int64_t)b * 2 * D + zz) * 2 * H + yy) * 2 * W + xx) * out_cs + out_co +
                ch);
        }
        a.q = *reinterpret_cast<const uint4*>(Z + o);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float s = 0.f;
#pragma unroll
            for (int c8 = 0; c8 < 8; ++c8) s += bf2f(v[c8].v[e]);
            r.v[e] = silu_bwd(f2bf(s), a.v[e]);
        }
        *reinterpret_cast<uint4*>(dZ + o) = r.q;
    }
}

static inline unsigned ew_blocks(int64_t n) {
    int64_t b = (n + 255) / 256;
    if (b > 8192) b = 8192;
    if (b < 1) b = 1;
    return (unsigned)b;
}

hipError_t launch_silu_bwd(int64_t n, const uint16_t* dA, const uint16_t* Z, uint16_t* dZ,
                           hipStream_t s) {
    hipLaunchKernelGGL(k_silu_bwd, dim3(ew_blocks(n)), dim3(256), 0, s, n, dA, Z, dZ);
    return hipGetLastError();
}
hipError_t launch_avgpool_fwd(int B, int D, int H, int W, int C, const uint16_t* in, int in_cs,
                              int in_co, uint16_t* out, hipStream_t s) {
    const int64_t n = (int64_t)B * (D / 2) * (H / 2) * (W / 2) * (C / 8);
    hipLaunchKernelGGL(k_avgpool_fwd, dim3(ew_blocks(n)), dim3(256), 0, s, B, D, H, W, C, in, in_cs,
                       in_co, out);
    return hipGetLastError();
}
hipError_t launch_skip_bwd(int B, int D, int H, int W, int C, const uint16_t* dpool,
                           const uint16_t* dskip, int cs, int co, const uint16_t* Z, uint16_t* dZ,
                           hipStream_t s) {
    const int64_t n = (int64_t)B * D * H * W * (C / 8);
    hipLaunchKernelGGL(k_skip_bwd, dim3(ew_blocks(n)), dim3(256), 0, s, B, D, H, W, C, dpool, dskip,
                       cs, co, Z, dZ);
    return hipGetLastError();
}
hipError_t launch_upsample_fwd(int B, int D, int H, int W, int C, const uint16_t* in,
                               uint16_t* out, int out_cs, int out_co, hipStream_t s) {
    const int64_t n = (int64_t)B * 8 * D * H * W * C;
    if (C % 8 == 0 && out_cs % 8 == 0 && out_co % 8 == 0 && ((uintptr_t)in & 15) == 0 &&
        ((uintptr_t)out & 15) == 0)
        hipLaunchKernelGGL(k_upsample_fwd8, dim3(ew_blocks(n / 8)), dim3(256), 0, s, B, D, H, W, C,
                           in, out, out_cs, out_co);
    else
        hipLaunchKernelGGL(k_upsample_fwd, dim3(ew_blocks(n)), dim3(256), 0, s, B, D, H, W, C, in,
                           out, out_cs, out_co);
    return hipGetLastError();
}
hipError_t launch_upsample_bwd(int B, int D, int H, int W, int C, const uint16_t* dout,
                               int out_cs, int out_co, const uint16_t* Z, uint16_t* dZ,
                               hipStream_t s) {
    const int64_t n = (int64_t)B * D * H * W * (C / 8);
    hipLaunchKernelGGL(k_upsample_bwd, dim3(ew_blocks(n)), dim3(256), 0, s, B, D, H, W, C, dout,
                       out_cs, out_co, Z, dZ);
    return hipGetLastError();
}

}  // namespace tohip
