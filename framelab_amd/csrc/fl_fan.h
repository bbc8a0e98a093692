// fl_fan.h -- per-ray and per-pixel bodies of the 2D fan operators, shared by
// the single-problem kernels and the batched persistent kernels so both run
// exactly the same float arithmetic.
#pragma once

#include <type_traits>

#include "fl_chord.h"
#include "fl_common.h"
#include "fl_geom.h"
#include "fl_siddon.h"
#include "fl_walk.h"

// Element k of a row, by a 32-bit byte offset from the (wave-uniform) row.
template <typename T>
__device__ __forceinline__ const T* fl_row_at(const T* row, unsigned k)
{
    return (const T*)((const char*)row + k * (unsigned)sizeof(T));
}

// Rays a wave walks together: FAN_WA neighbouring cells of 64/FAN_WA
// neighbouring views, a compact patch of the image at every step whatever the
// view angle.  64 cells of one view spread over 64 rows of it where the rays
// run along x, a cache line each (1024 x 1024, 900 views x 1000 cells: 1.09 ms
// with 8 x 8, 1.26 with 16 x 4, 2.33 with 64 x 1, before the walk's tracking).
constexpr int FAN_WA = 8;

// Image sizes whose byte offsets fit 32 bits (the tracked walk's).
__host__ __device__ inline bool fl_fan_small(int nx, int ny) { return (size_t)nx * ny < ((size_t)1 << 30); }

// How a fan ray reads its image: by 64-bit indices (the walk without tracking),
// row by row, or a copy in bricks.
enum FanRead { FAN_LARGE, FAN_ROWS, FAN_BRICKS };

// Siddon ray sum of fan ray (view iv, cell id), scaled
// (Ax_fan_mf_cpu_siddon.cpp:32-91): called by every lane of a wave, live = the
// lane has a ray.
template <int READ, typename VT>
__device__ __forceinline__ float fl_fan_ray_sum(const VT* __restrict__ x, const FwdGeom& g, int iv, int id, bool live)
{
    const float c = g.cs[iv], s = g.sn[iv];
    const float x1 = c * (-g.SO), y1 = s * (-g.SO);
    const float yd = g.ydet[id];
    const float x2 = c * g.OD - s * yd;
    const float y2 = s * g.OD + c * yd;
    const float dx = x2 - x1, dy = y2 - y1;
    const float L = sqrtf(dx * dx + dy * dy);
    if constexpr (READ != FAN_LARGE) {
        using Layout = std::conditional_t<READ == FAN_BRICKS, FanBricks<sizeof(VT)>, FanImage<sizeof(VT)>>;
        WalkAxis ax, ay, az;
        walk_axis_init(ax, x1, dx, 1.0f, g.nx);
        walk_axis_init(ay, y1, dy, 1.0f, g.ny);
        walk_axis_init(az, 0.0f, 0.0f, 1.0f, 2);
        return walk_rays<false, true, false>(ax, ay, az, L, live, x, Layout(g.nx, g.ny)) * g.scale;
    } else {
        SidAxis ax, ay, az;
        sid_axis_init(ax, x1, dx, 1.0f, g.nx);
        sid_axis_init(ay, y1, dy, 1.0f, g.ny);
        sid_axis_init(az, 0.0f, 0.0f, 1.0f, 2);
        float acc = 0.0f;
        if (live)
            sid_walk<false>(ax, ay, az, L, true, [&](int j, float dal) { acc = acc + (dal * L) * fl_load(x, (size_t)j); });
        return acc * g.scale;
    }
}

// Gao column walk (Ax_fan_mf_cpu_new.cpp:28-119): per column of the ray's major
// axis the line's crossing of one pixel or two.
//
// A ray's columns are shared by the four lanes of a quad, GAO_D columns each at
// a time: their terms are formed without branches, so that their reads and
// roots are in flight together, and added in column order from the lanes in
// turn (a DPP add), as the serial walk adds them; a term that the reference
// skips is +0, which leaves a sum that starts at +0 unchanged.  A wave takes
// GAO_WA cells of 16 / GAO_WA views.
//
// Divisions by the column's span d are Markstein quotients of one reciprocal
// (fl_rcp_mid: a span is 0, which is not divided by, or 2^-22 .. 2); the root's
// argument lies in [1, 2], clear of the ranges that need scaling.
//
// 64 x 64, 60 views x 96 cells: 71 -> 9 us; 256 x 256, 256 x 256: 257 -> 36; 1024 x
// 1024, 900 x 1000: 3.04 -> 1.47 ms (90 waves' chains of 64 columns, each
// with a branch, a division pair, a root and a read behind one another).
constexpr int GAO_WA = 4;
constexpr int GAO_D = 4;

// v of lane Q of this lane's quad
template <int Q>
__device__ __forceinline__ float fl_quad(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), Q * 0x55, 0xf, 0xf, true));
}

// Sum of fan ray (view iv, cell id), scaled, in every lane of the ray's quad.
// Called by all lanes of a wave with a valid iv and id.
template <bool SMALL, typename VT>
__device__ __forceinline__ float fl_fan_gao_sum(const VT* __restrict__ x, const FwdGeom& g, int iv, int id)
{
    using Idx = std::conditional_t<SMALL, unsigned, size_t>;
    constexpr int D = GAO_D;
    const int nx = g.nx, ny = g.ny;
    const float c = g.cs[iv], s = g.sn[iv];
    const float x1 = c * (-g.SO), y1 = s * (-g.SO);
    const float yd = g.ydet[id];
    const float x2 = c * g.OD - s * yd;
    const float y2 = s * g.OD + c * yd;
    // u along the major axis, v along the other
    const bool xm = fl_absf(x1 - x2) > fl_absf(y1 - y2);
    const int nu = xm ? nx : ny, nv = xm ? ny : nx;
    const float u0 = xm ? x1 : y1, v0 = xm ? y1 : x1;
    const float slope = xm ? (y2 - y1) / (x2 - x1) : (x2 - x1) / (y2 - y1);
    const float nu2 = (float)(nu / 2), nv2 = (float)(nv / 2);
    const Idx su = xm ? 1 : nx, sv = xm ? nx : 1;
    const int quad = (int)threadIdx.x & 3;
    auto plane = [&](float u) { return v0 + slope * (u - u0) + nv2; };
    float acc = 0.0f;
    // the most columns any of the wave's rays has
    const int n = max(__builtin_amdgcn_ballot_w64(xm) ? nx : 0, __builtin_amdgcn_ballot_w64(!xm) ? ny : 0);
    for (int i0 = 0; i0 < n; i0 += 4 * D) {
        float t1[D], t2[D];
#pragma unroll
        for (int k = 0; k < D; k++) {
            const int iu = i0 + 4 * k + quad;
            const float u = (float)iu - nu2, pa = plane(u), pb = plane(u + 1.0f);
            const float va = fminf(pa, pb), vb = fmaxf(pa, pb);   // (the plane of the smaller v, by the slope's sign)
            const float fa = floorf(va), fb = floorf(vb);
            const int c1 = (int)fa, c2 = (int)fb;
            const bool one = c1 == c2, in = iu < nu;
            // the reference's y-major branch tests c2 == ny for c2 == nx
            const bool ok1 = in && (unsigned)c1 < (unsigned)nv && (one || c2 < nv || c2 == ny);
            const bool ok2 = in && !one && (unsigned)c2 < (unsigned)nv;
            const Idx col = (Idx)iu * su;
            const float xa = fl_load(x, ok1 ? col + (Idx)c1 * sv : (Idx)0), xb = fl_load(x, ok2 ? col + (Idx)c2 * sv : (Idx)0);
            const float d = vb - va, l = fl_sqrt_mid(d * d + 1.0f);
            const float r = fl_rcp_mid(d);
            const float wa = one ? l : sid_div(fb - va, d, r) * l, wb = sid_div(vb - fb, d, r) * l;
            t1[k] = ok1 ? wa * xa : 0.0f;
            t2[k] = ok2 ? wb * xb : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < D; k++) {
            acc = acc + fl_quad<0>(t1[k]);
            acc = acc + fl_quad<0>(t2[k]);
            acc = acc + fl_quad<1>(t1[k]);
            acc = acc + fl_quad<1>(t2[k]);
            acc = acc + fl_quad<2>(t1[k]);
            acc = acc + fl_quad<2>(t2[k]);
            acc = acc + fl_quad<3>(t1[k]);
            acc = acc + fl_quad<3>(t2[k]);
        }
    }
    return acc * g.scale;
}

// ---- pixel-driven adjoints, general form -----------------------------------
//
// Per pixel and view a loop over the cells of a window on the detector.  The
// plans whose geometry bounds a pixel's shadow to a few cells take the
// windowed form instead (fl_fan_adj.h), which shares the arithmetic of a cell.

// Exact adjoint: the term of one cell, the chord of its line a x + b y = d
// through the unit pixel at (xc, yc) (find_l.cpp:18-45) times the sinogram
// value (Atx_fan_mf_cpu_new.cpp:48-58: added only where the chord is
// positive, which is where the line passes within dmax = (|a| + |b|)/2).
// ln = (2a, 2b, 1/max(|a|,|b|), 1/(4|a||b|)), pd2 = 2d: the factors of two
// scale every intermediate exactly (t2 = 2t, num = 4(dmax - |t|), and num
// and den in the quotient num/den alike) and save the halvings.
__device__ __forceinline__ float fl_fan_exact_term(float4 ln, float pd2, float xc, float yc, float yv)
{
    const float a2 = fabsf(ln.x), b2 = fabsf(ln.y);
    const float t2 = fabsf(pd2 - ln.x * xc - ln.y * yc);
    const float num = __builtin_fmaf(-2.0f, t2, a2 + b2);
    // flat part of the chord: |t| <= ||a| - |b||/2
    const bool flat = __builtin_fmaf(-2.0f, t2, fabsf(a2 - b2)) >= 0.0f;
    // (dmax - |t|)/(|a||b|) by Markstein's correction of the tabulated
    // reciprocal (fl_div_r); where |a||b| is 0 or its reciprocal overflows,
    // |a| + |b| = ||a| - |b|| in float and the flat value is taken
    const float den = a2 * b2;
    const float q = num * ln.w;
    const float slope = __builtin_fmaf(__builtin_fmaf(-q, den, num), ln.w, q);
    const float l = flat ? ln.z : slope;
    return num > 0.0f ? l * yv : 0.0f;
}

// General exact adjoint of pixel (ix, iy) of frame it, scaled
// (Atx_fan_mf_cpu_new.cpp:35-62).
template <typename YT>
__device__ __forceinline__ float fl_fan_adj_pixel(const YT* __restrict__ Y, const AdjGeom& g, int it, int ix, int iy)
{
    const int nd = g.na, nd2 = nd / 2;
    const float SD = g.SO + g.OD;
    const float xc = (float)ix + 0.5f - (float)(g.nx / 2);
    const float yc = (float)iy + 0.5f - (float)(g.ny / 2);
    float acc = 0.0f;
    const int nvf = g.Nv[it];
    for (int j = 0; j < nvf; j++) {
        const int iv = g.id_Y[it * g.tmp_size + j];
        const YT* __restrict__ y = Y + (size_t)g.id_S[it * g.tmp_size + j] * nd;
        const float c = g.cphi[iv], s = g.sphi[iv];
        const float xr = c * xc + s * yc;
        const float yr = -s * xc + c * yc;
        const float t = SD / ((xr + g.SO) * g.dy_det);
        int hi = (int)floorf((yr + 1) * t - g.y_os + (float)nd2);
        int lo = (int)floorf((yr - 1) * t - g.y_os + (float)nd2);
        if (lo < 0) lo = 0;
        if (hi > nd - 1) hi = nd - 1;
        const float4* __restrict__ line = g.line_q + (size_t)iv * nd;
        for (int id = lo; id <= hi; id++)
            acc = acc + fl_fan_exact_term(line[id], g.line_d[id], xc, yc, fl_load(y, (size_t)id));
    }
    return acc * g.scale;
}

struct FlAxisIv {
    float in, out;   // entry / exit parameters of a voxel slab along one axis
};

// Entry/exit plane parameters of cell `cell` along one walk axis, the forward's
// quotients ((float)i*s - o)/d, both from rd = 1.0f / a.d (fl_div_r, bit-identical
// to the divisions).
__device__ __forceinline__ FlAxisIv fl_slab_r(const SidAxis& a, int cell, float rd)
{
    FlAxisIv r;
    if (!a.on) {
        r.in = -FL_INF;
        r.out = FL_INF;
        return r;
    }
    const float lo = fl_div_r((float)(cell - a.nh) * a.s - a.o, a.d, rd);
    const float hi = fl_div_r((float)(cell - a.nh + 1) * a.s - a.o, a.d, rd);
    r.in = a.st > 0 ? lo : hi;
    r.out = a.st > 0 ? hi : lo;
    return r;
}

// Matched adjoint: the term of one cell for a pixel whose x planes lie at xl,
// xl + 1 and y planes at yl, yl + 1 from the source (x1, y1): the Siddon
// segment of the ray inside the pixel, credited where the forward's midpoint
// rule maps it there, times the sinogram value.  r4 = (dx, dy, 1/dx, 1/dy) of
// the ray, 0 in place of the reciprocal of a zero component (the ray is
// parallel to that axis' planes), L its length.  Plane parameters are the
// forward's quotients (fl_div_r); every test is evaluated, without branches.
__device__ __forceinline__ float fl_fan_matched_term(float4 r4, float L, float xl, float xh, float yl, float yh,
                                                     float x1, float y1, float nhx, float nhy, int ix, int iy, float yv)
{
    auto quot = [](float num, float d, float r) {
        const float q = num * r;
        return __builtin_fmaf(__builtin_fmaf(-q, d, num), r, q);
    };
    const float ax = quot(xl, r4.x, r4.z), bx = quot(xh, r4.x, r4.z);
    const float ay = quot(yl, r4.y, r4.w), by = quot(yh, r4.y, r4.w);
    const bool onx = r4.x != 0.0f, ony = r4.y != 0.0f;
    const float inx = onx ? fminf(ax, bx) : -FL_INF, outx = onx ? fmaxf(ax, bx) : FL_INF;
    const float iny = ony ? fminf(ay, by) : -FL_INF, outy = ony ? fmaxf(ay, by) : FL_INF;
    const float ain = fmaxf(inx, iny), aout = fminf(outx, outy);
    const float m = (ain + aout) * 0.5f;
    const int tx = (int)floorf(x1 + m * r4.x + nhx), ty = (int)floorf(y1 + m * r4.y + nhy);
    const int hit = int(aout > ain) & int(tx == ix) & int(ty == iy);
    return hit ? ((aout - ain) * L) * yv : 0.0f;
}

// General matched (Siddon-transpose) adjoint of pixel (ix, iy) of frame it,
// scaled.
template <typename YT>
__device__ __forceinline__ float fl_fan_matched_pixel(const YT* __restrict__ Y, const FwdGeom& f, const AdjGeom& g,
                                                      int it, int ix, int iy)
{
    const int nd = f.na;
    const float SD = f.SO + f.OD;
    const float xc = (float)ix + 0.5f - (float)(f.nx / 2);
    const float yc = (float)iy + 0.5f - (float)(f.ny / 2);
    const float nhx = (float)(f.nx / 2), nhy = (float)(f.ny / 2);
    const float ya0 = f.ydet[0];
    float acc = 0.0f;
    const int nvf = g.Nv[it];
    for (int j = 0; j < nvf; j++) {
        const int iv = g.id_Y[it * g.tmp_size + j];
        const YT* __restrict__ y = Y + (size_t)g.id_S[it * g.tmp_size + j] * nd;
        const float c = f.cs[iv], s = f.sn[iv];
        const float xr = c * xc + s * yc, yr = -s * xc + c * yc;
        const float mag = SD / (xr + f.SO);
        int lo = (int)floorf(((yr - 1.0f) * mag - ya0) * f.inv_pa) - 1;
        int hi = (int)ceilf(((yr + 1.0f) * mag - ya0) * f.inv_pa) + 1;
        if (lo > hi) { int t = lo; lo = hi; hi = t; }
        if (lo < 0) lo = 0;
        if (hi > nd - 1) hi = nd - 1;
        const float x1 = c * (-f.SO), y1 = s * (-f.SO);
        const float xl = (float)(ix - f.nx / 2) - x1, xh = (float)(ix - f.nx / 2 + 1) - x1;
        const float yl = (float)(iy - f.ny / 2) - y1, yh = (float)(iy - f.ny / 2 + 1) - y1;
        const float4* __restrict__ ray = g.ray_q + (size_t)iv * nd;
        const float* __restrict__ len = g.ray_l + (size_t)iv * nd;
        for (int id = lo; id <= hi; id++)
            acc = acc + fl_fan_matched_term(ray[id], len[id], xl, xh, yl, yh, x1, y1, nhx, nhy, ix, iy,
                                            fl_load(y, (size_t)id));
    }
    return acc * f.scale;
}
