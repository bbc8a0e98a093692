// fl_fan_adj.h -- the fan adjoints' windowed form, shared by the
// single-problem kernels and the batched persistent kernels.
//
// A workgroup of W + 1 waves owns a tile of 8 x 8 pixels, one per lane.  W
// producer waves form the terms of W * VB consecutive views at a time; the
// last wave adds the previous batch's terms to the pixels' sums, views in
// list order and cells ascending, so the sum is the serial one bit for bit
// (a pixel's sum is one chain of float adds) while W times as many waves
// have work: 256 x 256 pixels alone are one wave per SIMD.
//
// A producer wave stages its view's footprint under the tile in LDS (a few
// dozen cells: their per-ray constants and sinogram values, each read from
// memory once per wave) and every lane evaluates the n cells from its own
// first one on, without branches: a cell beyond the pixel's shadow has a term
// of exactly 0, which leaves a sum that starts at +0 unchanged.  n, at most
// the plan's bound S, the tile's first cell and the shadow's half width are
// worked out for 64 views at a time, one view per lane.
//
// Bound: VALU issue (11 operations for a pixel's first cell, 18 per cell of
// the exact adjoint, 42 of the matched one) and the LDS reads behind them (24
// bytes per lane and cell): 512 x 512, exact, issues 0.24 instructions a SIMD and
// cycle with the LDS active for half the cycles.  Reading the cells from L1 instead took 32 clocks
// per cell and CU: the loads' 24 bytes x 64 lanes, twice that where unaligned.
#pragma once

#include <type_traits>

#include "fl_common.h"
#include "fl_fan.h"
#include "fl_geom.h"

// What the exact adjoint needs: fl_fan_exact_term.
struct FanExact {
    static constexpr bool matched = false;
    const float4* row;    // of the staged view
    const float* rowb;
    float xc, yc;
    __device__ FanExact(const FwdGeom&, const AdjGeom&, int, int, float x, float y) : row(nullptr), rowb(nullptr), xc(x), yc(y) {}
    __device__ void rows(const AdjGeom& g, unsigned off)
    {
        row = g.line_q + off;
        rowb = g.line_d;
    }
    __device__ void view(float, float, float) {}
    __device__ float term(float4 a, float b, float yv) const { return fl_fan_exact_term(a, b, xc, yc, yv); }
};

// What the matched adjoint needs: fl_fan_matched_term.
struct FanMatched {
    static constexpr bool matched = true;
    const float4* row;
    const float* rowb;
    int ix, iy;
    float fx, fy, nhx, nhy, x1, y1;
    __device__ FanMatched(const FwdGeom& f, const AdjGeom&, int ix_, int iy_, float, float)
        : row(nullptr), rowb(nullptr), ix(ix_), iy(iy_), fx((float)(ix_ - f.nx / 2)), fy((float)(iy_ - f.ny / 2)),
          nhx((float)(f.nx / 2)), nhy((float)(f.ny / 2)), x1(0.0f), y1(0.0f) {}
    __device__ void rows(const AdjGeom& g, unsigned off)
    {
        row = g.ray_q + off;
        rowb = g.ray_l + off;
    }
    __device__ void view(float c, float s, float SO)
    {
        x1 = c * (-SO);
        y1 = s * (-SO);
    }
    __device__ float term(float4 a, float b, float yv) const
    {
        return fl_fan_matched_term(a, b, fx - x1, (fx + 1.0f) - x1, fy - y1, (fy + 1.0f) - y1, x1, y1, nhx, nhy, ix, iy, yv);
    }
};

template <int S, int W, int VB>
struct FanTileLds {
    float4 cell[W][64];
    float2 cell2[W][64];
    float terms[2][W * VB][S][64];
};

// The tile with corner (ix0, iy0) of frame it; every thread of the workgroup
// (64 * (W + 1)) calls it.  Returns the pixel's scaled sum in the last wave.
template <class Kind, int S, int W, int VB, typename YT>
__device__ __forceinline__ float fl_fan_adj_tile(const YT* __restrict__ Y, const FwdGeom& f, const AdjGeom& g, int it,
                                                 int ix0, int iy0, FanTileLds<S, W, VB>& lds)
{
    constexpr int NV = W * VB;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int ix = ix0 + (lane & 7), iy = iy0 + (lane >> 3);
    const float xc = (float)ix + 0.5f - (float)(g.nx / 2);
    const float yc = (float)iy + 0.5f - (float)(g.ny / 2);
    const float xt = (float)(ix0 + 4 - g.nx / 2), yt = (float)(iy0 + 4 - g.ny / 2);   // the tile's centre
    const int nvf = g.Nv[it];
    const FanView* __restrict__ views = g.fan_views + (size_t)it * g.tmp_size;
    const int nph = (nvf + NV - 1) / NV;
    const unsigned nd = (unsigned)g.na;
    Kind kind(f, g, ix, iy, xc, yc);
    float acc = 0.0f;
    // The wave's views are its own 0, 1, ...: own view i is view i * W + w of
    // the frame's list.  fetch(i) sets up own view i and starts its loads, one
    // view ahead of its use.
    int a0s = 0, ns = 0;       // per lane: first cell and cell count of one of the wave's next 64 views
    float hs = 0.0f;           // and its shadow half width
    FanView v;                 // the fetched view, its A0, n and h, and this lane's cell of its footprint
    unsigned A0 = 0;
    int n = 0;
    float h = 0.0f;
    float4 ca = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float cb = 0.0f, cy = 0.0f;
    auto fetch = [&](int i) {
        if (i % 64 == 0) {
            const FanView u = views[min((i + lane) * W + w, nvf - 1)];
            // pixel centres lie within e of the tile's along and across the ray axis
            const float e = 3.5f * (fabsf(u.c) + fabsf(u.s));
            const float D = __builtin_fmaf(u.c, xt, __builtin_fmaf(u.s, yt, g.SO));
            const float yr = __builtin_fmaf(u.c, yt, -u.s * xt);
            const float rn = __builtin_amdgcn_rcpf(D - e), rf = __builtin_amdgcn_rcpf(D + e);
            const float tg = yr * __builtin_amdgcn_rcpf(D);
            // half width h(tan) = (|tan c + s| + |c - tan s|)/2 of a pixel's
            // shadow over D, at the tile's tan plus its change over the tile
            const float dt = e * (1.0f + fabsf(tg)) * rn;
            const float hc = fabsf(__builtin_fmaf(tg, u.c, u.s)) + fabsf(__builtin_fmaf(-tg, u.s, u.c));
            hs = fminf((hc + dt * (fabsf(u.c) + fabsf(u.s))) * g.fan_grow, g.fan_hmax);
            ns = min((int)(2.0f * hs * rn * g.fan_sdp + 0.101f) + 1, S);
            const float edge = yr - e - hs;
            a0s = (int)ceilf(__builtin_fmaf(edge * (edge > 0.0f ? rf : rn), g.fan_sdp, g.fan_klo - 0.01f));
            a0s = min(max(a0s, 0), g.na - S);
        }
        v = views[min(i * W + w, nvf - 1)];
        A0 = (unsigned)__builtin_amdgcn_readlane(a0s, i % 64);
        n = __builtin_amdgcn_readlane(ns, i % 64);
        h = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hs), i % 64));
        if (lane < g.fan_tile) {
            const unsigned id = min(A0 + (unsigned)lane, nd - 1);
            kind.rows(g, (unsigned)v.view * nd);
            ca = *fl_row_at(kind.row, id);
            cb = *fl_row_at(kind.rowb, id);
            cy = fl_load(fl_row_at(Y + (size_t)(unsigned)v.slot * nd, id), 0);
        }
    };
    if (w < W && nph > 0) fetch(0);
    for (int ph = 0; ph <= nph; ph++) {
        if (w < W) {
            if (ph < nph) {
#pragma unroll
                for (int b = 0; b < VB; b++) {
                    if (lane < g.fan_tile) {
                        lds.cell[w][lane] = ca;
                        lds.cell2[w][lane] = make_float2(cb, cy);
                    }
                    __builtin_amdgcn_wave_barrier();
                    // first cell of this pixel's shadow
                    const float D = __builtin_fmaf(v.c, xc, __builtin_fmaf(v.s, yc, g.SO));
                    const float yr = __builtin_fmaf(v.c, yc, __builtin_fmaf(-v.s, xc, -h));
                    int lo = (int)ceilf(__builtin_fmaf(yr * __builtin_amdgcn_rcpf(D), g.fan_sdp, g.fan_klo));
                    lo = min(max(lo, (int)A0), g.na - n) - (int)A0;
                    kind.view(v.cf, v.sf, g.SO);
                    const int m = n;
                    fetch(ph * VB + b + 1);
                    const float4* c1 = &lds.cell[w][lo];
                    const float2* c2 = &lds.cell2[w][lo];
                    float* t = &lds.terms[ph & 1][b * W + w][0][lane];
                    // m is the wave's: a scalar branch skips the cells no pixel needs
#pragma unroll
                    for (int k = 0; k < S; k++) {
                        float v1 = 0.0f;
                        if (k < 1 || k < m) v1 = kind.term(c1[k], c2[k].x, c2[k].y);
                        t[k * 64] = v1;
                    }
                    __builtin_amdgcn_wave_barrier();
                }
            }
        } else if (ph > 0) {
            const int nt = min(NV, nvf - (ph - 1) * NV) * S;
            const float* t = &lds.terms[(ph - 1) & 1][0][0][lane];
#pragma unroll 8
            for (int k = 0; k < nt; k++) acc = acc + t[k * 64];
        }
        __syncthreads();
    }
    return acc * g.scale;
}

// Producer waves, and the views each forms between two barriers: the most
// for which four workgroups (32 waves) and their terms fit a CU's LDS.
constexpr int FAN_W = 7;
constexpr int fl_fan_vb(int S) { return S <= 2 ? 4 : S <= 4 ? 2 : 1; }

// Whether the windowed form serves a plan, `tiles` of 8 x 8 pixels in its launch.
// It takes views by batches of FAN_W * fl_fan_vb(S), whole ones however few they
// are, and pays for the first batch's start; the general form takes a lane's
// views one by one, which is the shorter where tiles fill the chip by
// themselves and views are few.  512 x 512 (4096 tiles) and 1024 x 1024, us, general
// and windowed: exact, S = 2, 16 views 16 and 17, 41 and 58; 24 views 21 and 17, 58 and
// 59; S = 4, 8 views 13 and 14, 36 and 46; 12 views 17 and 14, 51 and 47; matched, S = 2,
// 8 views 18 and 23, 52 and 78; 16 views 34 and 22, 100 and 76; S = 4, 4 views 13 and 17,
// 34 and 57; 8 views 21 and 17, 65 and 60.  384 x 384 (2304 tiles), 960 cells: exact, 3
// views 7.4 and 9.0, 6 views 9.4 and 8.8; 256 x 256 (1024 tiles): within 7% from one view on.
// In a batch, 8 x 512 x 512: exact, S = 2, 8 views 76 and 172, 20 views 181 and 181.
inline bool fl_fan_windowed(const AdjGeom& g, bool matched, long long tiles)
{
    const int S = g.fan_cells;
    if (S == 0 || tiles < 2048) return S != 0;
    const int nv = g.tmp_size, per = FAN_W * fl_fan_vb(S), batches = (nv + per - 1) / per;
    const int few = matched ? (S <= 2 ? 2 + 8 * batches : S <= 3 ? 3 + 4 * batches : S <= 4 ? 1 + 5 * batches : 1 + 2 * batches)
                            : (S <= 2 ? 5 + 13 * batches : S <= 3 ? 6 + 6 * batches : S <= 4 ? 4 + 5 * batches : 3 + 2 * batches);
    return nv > (tiles < 4096 ? few / 2 : few);
}

// 512 x 512 pixels, 640 views x 491 cells (S = 2), exact: 0.64 -> 0.228 ms;
// 256 x 256, 360 x 512 (S = 4): 0.32 -> 0.059 ms (one lane per pixel and the
// reference's window before).  Three producer waves 0.28 and 0.072 ms,
// fifteen 0.35 and 0.069 ms; one barrier per view and wave 0.31 and 0.064 ms.
template <class Kind, typename YT, typename XT, int S>
__global__ __launch_bounds__(64 * (FAN_W + 1)) void k_adj_fan_w(const YT* __restrict__ Y, XT* __restrict__ X,
                                                               FwdGeom f, AdjGeom g)
{
    __shared__ FanTileLds<S, FAN_W, fl_fan_vb(S)> lds;
    const int it = blockIdx.z, ix0 = (int)blockIdx.x * 8, iy0 = (int)blockIdx.y * 8;
    const float v = fl_fan_adj_tile<Kind, S, FAN_W, fl_fan_vb(S)>(Y, f, g, it, ix0, iy0, lds);
    const int lane = threadIdx.x & 63, ix = ix0 + (lane & 7), iy = iy0 + (lane >> 3);
    if ((int)threadIdx.x >> 6 == FAN_W && ix < g.nx && iy < g.ny)
        fl_store(X, (size_t)it * g.nvox + (size_t)iy * g.nx + ix, v);
}

// Launches the windowed adjoint where it serves the plan (true).
template <class Kind, typename YT, typename XT>
static bool fl_launch_fan_adj_w(const YT* Y, XT* X, const FwdGeom& f, const AdjGeom& g, hipStream_t st)
{
    auto go = [&](auto s) {
        hipLaunchKernelGGL((k_adj_fan_w<Kind, YT, XT, decltype(s)::value>),
                           dim3((g.nx + 7) / 8, (g.ny + 7) / 8, g.nt), dim3(64 * (FAN_W + 1)), 0, st, Y, X, f, g);
        return true;
    };
    if (!fl_fan_windowed(g, Kind::matched, (long long)((g.nx + 7) / 8) * ((g.ny + 7) / 8) * g.nt)) return false;
    switch (g.fan_cells) {
    case 2: return go(std::integral_constant<int, 2>{});
    case 3: return go(std::integral_constant<int, 3>{});
    case 4: return go(std::integral_constant<int, 4>{});
    case 6: return go(std::integral_constant<int, 6>{});
    default: return false;
    }
}
