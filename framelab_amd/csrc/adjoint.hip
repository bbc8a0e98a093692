// adjoint.hip -- voxel-driven exact adjoints (backprojectors), atomic-free.
//
// Each thread owns one output pixel/voxel and gathers, view by view, the
// detector cells whose rays cross it, weighting each by the exact chord
// length.  No two threads write the same output, so there are no atomics
// and the result is deterministic.  The per-voxel summation order (views
// ascending, then detector rows, then columns) and the float arithmetic are
// those of the reference, so results are bit-identical to it:
//   fan:  matlab/mex/src/Atx_fan_mf_cpu_new.cpp:35-62
//   cone: matlab/mex/src/Atx_cone_mf_gpu_new.cu:41-84 (window from zr with
//         d=sqrt((1+dz^2)/2), ceil upper bounds, box sides (1,1,dz)).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "fl_chord.h"
#include "fl_common.h"
#include "fl_geom.h"
#include "fl_fan.h"
#include "fl_fan_adj.h"

// General form: one lane per pixel (fl_fan_adj_pixel).
template <typename YT, typename XT>
__global__ __launch_bounds__(256) void k_adj_fan(const YT* __restrict__ Y, XT* __restrict__ X, AdjGeom g)
{
    const int ix = blockIdx.x * 16 + threadIdx.x;
    const int iy = blockIdx.y * 16 + threadIdx.y;
    const int it = blockIdx.z;
    if (ix >= g.nx || iy >= g.ny) return;
    fl_store(X, (size_t)it * g.nvox + (size_t)iy * g.nx + ix, fl_fan_adj_pixel(Y, g, it, ix, iy));
}

// Cone, footprint-staged: per view the workgroup stages its detector
// footprint in LDS -- the rays' direction components, the six direction
// ratios find_l_3d divides out (each the IEEE quotient, computed once per
// workgroup instead of once per voxel), and the sinogram values.  Each voxel
// then evaluates, with the reference arithmetic and in the reference order,
// the chord of every cell in the intersection of the reference's window and
// the voxel's shadow on the detector (widened by 0.05 cells), or of the
// shadow alone where the plan has shown that the reference's window contains
// it (AdjGeom::win_ref clear).  Cells outside the shadow have exact-zero
// chords, and the reference adds l*y = +-0 for them, which leaves a sum that
// starts at +0 unchanged, so the result is bit-identical to the reference
// kernel.
namespace {
constexpr int FP_A = 48;      // footprint columns held in LDS
constexpr int FP_B = 64;      // footprint rows
static_assert(FP_A <= 64 && FP_B <= 64, "footprint columns / rows are staged by one wave each");

// A brick's staged footprint: per cell the slopes of z on the x and y faces
// (c/a, c/b), those of x and y on the z faces (a/c, b/c) and the sinogram
// value.  What the tables are formed from is double-buffered: written a view
// ahead.
template <int KZ>
struct ExactLds {
    static constexpr int CELLS = KZ == 8 ? 1152 : 1408;   // footprint cells (four workgroups' tables fit a CU)
    static constexpr int N = CELLS + FP_B;                // and a zero at each row's end
    float2 zs[N], xs[N];
    float y[N];
    float acc[KZ][256];   // the voxels' sums (a rolled loop over k indexes them)
    float a[2][FP_A], b[2][FP_A], ra[2][FP_A], rb[2][FP_A], sba[2][FP_A], sab[2][FP_A];
    float c[2][FP_B], rc[2][FP_B], ch[2][FP_B];   // (ch: a slice's half height signed by c)
    ShadowCols cols[2][64];
};
}  // namespace

// Exact cone adjoint, z-column form.  A workgroup is an 8 x 8 x (4*KZ)
// voxel brick; each thread owns KZ z-adjacent voxels of one (x, y) column,
// which share the view rotation, the detector-column window and the
// workgroup's per-view footprint tables in LDS.  Per voxel, the cells and
// the order of accumulation are those of the reference kernel
// (Atx_cone_mf_gpu_new.cu:58-86: views in order, rows outer, columns
// inner), restricted to the cells whose chord can be non-zero.
//
// What find_l_3d tests on a box's x and y faces splits into a test along the
// other of x and y, which depends on the detector column only, and one along
// z.  A thread works out the former once per view for its one to three
// columns: usually the ray enters the (x, y) square through one face and
// leaves through one, both known with the chord's x and y part.  A cell is
// then the heights zi, zo at which the ray crosses those faces: both inside
// the slice, the chord is known; one inside, the other end lies on a z face,
// if on the box; both beyond the same z face, there is none.  All of it is
// find_l_3d's arithmetic, operation by operation; what may differ is which
// faces it would find the ray to cross, and that only where a crossing lies
// within rounding of an edge.  There, and for a ray that crosses both z faces
// or runs parallel to x or y planes, the whole routine runs
// (fl_chord_box3_fast):
//   - heights: the coordinates of a crossing are off by a few u (u = 2^-24) of
//     the products that form them: in height by some 3u (|p2| + s), p2 the
//     box's height over the source and s the slope of z on the face, whichever
//     face names it; taken as 16u (|p2| + 1 + s);
//   - columns: a ray that misses the square by 16u (|p0| + |p1| + 1 + slope)
//     or more in x or y meets no face; one that does not, and has not exactly
//     one entry and one exit, takes the routine for all its cells, and so does
//     one within 1/4096 of an axis's direction.
// The waves' usual counts of columns, CA0 and one more, have a loop of their own;
// wider shadows take the routine throughout.
//
// Bound by VALU issue (some 300 instructions a voxel and view at 256^3: 1.8 rows
// of 2.3 columns at 26, and 22 more for each that some lane leaves through a z
// face), at 0.25 a SIMD and cycle: of the registers 62 scalar ones, the lane
// masks and the views' scalars, and 20 vector ones spill (84 bytes a lane).  256^3,
// 360 views x 512 x 384:
// 56.5 -> 48.4 ms; helix 180 x 156 x 132, 241 views x 301 x 217: 21.5 -> 8.5 ms
// (32 rows overflowed); 64^3, 60 views: 572 -> 299 us (before: every cell's six
// candidates, some 90 instructions).  Four waves per SIMD; three take 55.8 ms,
// five spill (69).
template <typename YT, typename XT, int KZ, int CA0>
__global__ __launch_bounds__(256, 4) void k_adj_cone_zc(const YT* __restrict__ Y, XT* __restrict__ X, AdjGeom g)
{
    constexpr int BZ = 4 * KZ;
    constexpr int NY = 2;   // values a thread loads a view ahead
    __shared__ __align__(16) ExactLds<KZ> t;
    const int bx = (g.nx + 7) / 8, by = (g.ny + 7) / 8, bz = (g.nz + BZ - 1) / BZ;
    const uint32_t nblk = (uint32_t)bx * by * bz;
    const uint32_t b = fl_xcd_remap(blockIdx.x, nblk);
    const int it = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ix0 = (int)(b % bx) * 8, iy0 = (int)((b / bx) % by) * 8, izb = (int)(b / ((uint32_t)bx * by)) * BZ;
    const int ix = ix0 + (tid & 7), iy = iy0 + ((tid >> 3) & 7), iz0 = izb + wv * KZ;
    const bool col = ix < g.nx && iy < g.ny;
    const int kn = min(KZ, g.nz - iz0);   // slices of this wave inside the volume

    const int na = g.na, nb = g.nb, na2 = na / 2, nb2 = nb / 2;
    const float SD = g.SO + g.OD;
    const float d = sqrtf((1 + g.dz * g.dz) / 2);
    const float yc = (float)iy + 0.5f - (float)(g.ny / 2);
    const float xc = (float)ix + 0.5f - (float)(g.nx / 2);
    const float hz = g.dz / 2;
    const ShadowMap ma = fl_shadow_map(g.ya0, g.inv_pa, 0.05f), mb = fl_shadow_map(g.zb0, g.inv_pb, 0.05f);
    const bool rows_ref = (g.win_ref & 2) != 0;
    // bounds the rays' slopes against their major axes
    const float tz = 1.5f * fmaxf(fabsf(g.zdet[0]), fabsf(g.zdet[nb - 1])) / SD;
#pragma unroll
    for (int k = 0; k < KZ; k++) t.acc[k][tid] = 0.0f;

    // 64 views at a time are set up one per lane: source and direction,
    // sinogram slot and the brick's footprint on the panel
    const int nvf = g.Nv[it];
    float uc = 0.0f, us = 0.0f, usz = 0.0f;
    int uslot = 0, ua = 0, uan = 0, ub = 0, ubn = 0;
    auto setup = [&](int i) {
        const int j = min(i + lane, nvf - 1);
        const int iv = g.id_Y[it * g.tmp_size + j];
        uslot = g.id_S[it * g.tmp_size + j];
        uc = g.cphi[iv];
        us = g.sphi[iv];
        usz = g.sdz[iv];
        // the brick, a hundredth of a voxel wider, and a tenth of a cell
        const float xm = (float)(ix0 + 4 - g.nx / 2), ym = (float)(iy0 + 4 - g.ny / 2);
        const float e = 4.01f * (fabsf(uc) + fabsf(us));
        const float D = uc * xm + us * ym + g.SO, yr = uc * ym - us * xm;
        const float rn = __builtin_amdgcn_rcpf(D - e) * SD, rf = __builtin_amdgcn_rcpf(D + e) * SD;
        const float zl = ((float)(izb - g.nz / 2) - 0.01f) * g.dz - usz;
        const float zh = ((float)(izb + BZ - g.nz / 2) + 0.01f) * g.dz - usz;
        const float yl = yr - e, yh = yr + e;
        const ShadowMap wa = fl_shadow_map(g.ya0, g.inv_pa, 0.15f), wb = fl_shadow_map(g.zb0, g.inv_pb, 0.15f);
        int a1, b1;
        fl_shadow_range(wa, yl * (yl > 0 ? rf : rn), yh * (yh > 0 ? rn : rf), na, ua, a1);
        fl_shadow_range(wb, zl * (zl > 0 ? rf : rn), zh * (zh > 0 ? rn : rf), nb, ub, b1);
        if (!(D - e > 0.01f)) {   // a brick that reaches past the source, outside the volume
            ua = ub = 0;
            a1 = na - 1;
            b1 = nb - 1;
        }
        uan = max(a1 - ua + 1, 0);
        ubn = max(b1 - ub + 1, 0);
    };
    struct View {
        float c, s, sz;
        int A0, nA, B0, nB;
        size_t off;
        bool any, fits;
    };
    auto lanef = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
    auto view = [&](int i) {
        const int l = i & 63;
        View v;
        v.c = lanef(uc, l);
        v.s = lanef(us, l);
        v.sz = lanef(usz, l);
        v.A0 = __builtin_amdgcn_readlane(ua, l);
        v.nA = __builtin_amdgcn_readlane(uan, l);
        v.B0 = __builtin_amdgcn_readlane(ub, l);
        v.nB = __builtin_amdgcn_readlane(ubn, l);
        v.off = (size_t)__builtin_amdgcn_readlane(uslot, l) * g.nd;
        v.any = v.nA > 0 && v.nB > 0;
        v.fits = v.nA <= FP_A && v.nB <= FP_B && v.nA * v.nB <= t.CELLS;
        return v;
    };
    // a view ahead: direction components and reciprocals of the columns (wave
    // 0) and rows (wave 1), the shadows of the thread columns (the same in all
    // four waves: the other two, in turn) and the cells' values
    float yv[NY];
    auto stage = [&](const View& v, int p) {
        if (!v.any) return;
        if (v.fits) {
            if (wv == 0 && lane < v.nA) {
                const float x1 = v.c * (-g.SO), y1 = v.s * (-g.SO), yd = g.ydet[v.A0 + lane];
                const float a = (v.c * g.OD - v.s * yd) - x1, bb = (v.s * g.OD + v.c * yd) - y1;
                const float ra = 1.0f / a, rb = 1.0f / bb;
                t.a[p][lane] = a;
                t.b[p][lane] = bb;
                t.ra[p][lane] = ra;
                t.rb[p][lane] = rb;
                t.sba[p][lane] = fl_div_r(bb, a, ra);
                t.sab[p][lane] = fl_div_r(a, bb, rb);
            }
            if (wv == 1 && lane < v.nB) {
                const float cc = (g.zdet[v.B0 + lane] + v.sz) - v.sz;
                t.c[p][lane] = cc;
                t.rc[p][lane] = 1.0f / cc;
                t.ch[p][lane] = cc > 0 ? hz : -hz;
            }
            const uint32_t mA = fl_small_div_m((uint32_t)v.nA);   // k * nA < 2^18 in these tables
            const YT* __restrict__ y = Y + v.off + (size_t)v.B0 * na + v.A0;
#pragma unroll
            for (int q = 0; q < NY; q++) {
                const int k = q * 256 + tid;
                if (k < v.nA * v.nB) {
                    const int kb = fl_small_div(k, mA), ka = k - __mul24(kb, v.nA);
                    yv[q] = fl_load(y, (size_t)((unsigned)kb * (unsigned)na + (unsigned)ka));
                }
            }
        }
        if (wv == 2 + p) {
            ShadowCols sc = fl_shadow_cols(v.c, v.s, g.SO, SD, xc, yc, ma, na);
            if (g.win_ref & 1) {
                const float xr = v.c * xc + v.s * yc, yr = -v.s * xc + v.c * yc;
                const float r = SD / ((xr + g.SO) * g.dy_det);
                sc.ahi = min(sc.ahi, (int)ceilf((yr + 1) * r - g.y_os + (float)na2));
                sc.alo = max(sc.alo, (int)floorf((yr - 1) * r - g.y_os + (float)na2));
            }
            t.cols[p][lane] = sc;
        }
    };
    View v{};
    int p = 0;   // the buffer of the staged view
    if (nvf > 0) {
        setup(0);
        v = view(0);
        stage(v, 0);
    }
    for (int i = 0; i < nvf; i++) {
        if (!v.any) {   // the brick is off the panel; the other buffer may be in use
            if (i + 1 < nvf) {
                if ((i + 1) % 64 == 0) setup(i + 1);
                v = view(i + 1);
                stage(v, p);
            }
            continue;
        }
        __syncthreads();
        if (v.fits) {
            // the ratios' IEEE quotients from the staged reciprocals
            const uint32_t mA = fl_small_div_m((uint32_t)v.nA);
            const int cells = v.nA * v.nB;
            if (tid < v.nB) t.y[__mul24(tid, v.nA + 1) + v.nA] = 0.0f;
            auto put = [&](int i, int ka, int kb, float yk) {
                const int k = i + kb;
                const float a = t.a[p][ka], bb = t.b[p][ka], cc = t.c[p][kb], rc = t.rc[p][kb];
                t.zs[k] = make_float2(fl_div_r(cc, a, t.ra[p][ka]), fl_div_r(cc, bb, t.rb[p][ka]));
                t.xs[k] = make_float2(fl_div_r(a, cc, rc), fl_div_r(bb, cc, rc));
                t.y[k] = yk;
            };
#pragma unroll
            for (int q = 0; q < NY; q++) {
                const int k = q * 256 + tid;
                if (k < cells) {
                    const int kb = fl_small_div(k, mA);
                    put(k, k - __mul24(kb, v.nA), kb, yv[q]);
                }
            }
            for (int k = NY * 256 + tid; k < cells; k += 256) {
                const int kb = fl_small_div(k, mA), ka = k - __mul24(kb, v.nA);
                put(k, ka, kb, fl_load(Y + v.off, (size_t)(v.B0 + kb) * na + (v.A0 + ka)));
            }
        }
        const View u = v;
        const int p0 = p;
        if (i + 1 < nvf) {
            if ((i + 1) % 64 == 0) setup(i + 1);
            v = view(i + 1);
        }
        __syncthreads();
        p ^= 1;
        if (i + 1 < nvf) stage(v, p);
        const ShadowCols sc = t.cols[p0][lane];
        const int alo = max(sc.alo, u.A0) - u.A0, ahi = min(sc.ahi, u.A0 + u.nA - 1) - u.A0;
        if (!col || alo > ahi) continue;
        const float x1 = u.c * (-g.SO), y1 = u.s * (-g.SO), z1 = u.sz;
        const float p0x = x1 - xc, p0y = y1 - yc;
        const float miss0 = 0.5f + 0x1p-20f * (fabsf(p0x) + fabsf(p0y) + 1.0f);
        float tr = 0.0f;
        if (rows_ref) tr = SD / (((u.c * xc + u.s * yc) + g.SO) * g.dz_det);
        // rows of the slice at zc
        auto rows = [&](float zc, int& blo, int& bhi) {
            const float zr = zc - u.sz;
            fl_shadow_rows(sc, zr, hz, mb, nb, blo, bhi);
            if (rows_ref) {
                bhi = min(bhi, (int)ceilf((zr + d) * tr + (float)nb2));
                blo = max(blo, (int)floorf((zr - d) * tr + (float)nb2));
            }
            blo = max(blo, u.B0) - u.B0;
            bhi = min(bhi, u.B0 + u.nB - 1) - u.B0;
        };
        auto height = [&](int k) { return ((float)(iz0 + k) + 0.5f - (float)(g.nz / 2)) * g.dz; };
        // find_l_3d's chord of staged cell (ka, kb) and the box at height zc
        auto chord = [&](int ka, int kb, float zc) {
            const float a = t.a[p0][ka], bb = t.b[p0][ka];
            if (a == 0 || bb == 0) {
                const float yd = g.ydet[u.A0 + ka];
                return fl_chord_box3(x1, y1, z1, u.c * g.OD - u.s * yd, u.s * g.OD + u.c * yd, g.zdet[u.B0 + kb] + u.sz, 1.0f,
                                     1.0f, g.dz, xc, yc, zc);
            }
            const float2 zs = t.zs[__mul24(kb, u.nA + 1) + ka], xs = t.xs[__mul24(kb, u.nA + 1) + ka];
            const float h[3] = {0.5f, 0.5f, hz}, pt[3] = {p0x, p0y, z1 - zc};
            FlRatiosS q;
            q.r.sba = t.sba[p0][ka]; q.r.sab = t.sab[p0][ka];
            q.r.sca = zs.x; q.r.scb = zs.y; q.r.sac = xs.x; q.r.sbc = xs.y;
            q.hs[0] = a > 0 ? 0.5f : -0.5f; q.hs[1] = bb > 0 ? 0.5f : -0.5f; q.hs[2] = t.ch[p0][kb];
            return fl_chord_box3_fast(pt, h, q, [&] { return fl_absf(a) > fl_absf(bb); });
        };
        if (!u.fits) {
            const YT* __restrict__ y = Y + u.off;
#pragma unroll 1
            for (int k = 0; k < kn; k++) {
                const float zc = height(k);
                float a = t.acc[k][tid];
                int blo, bhi;
                rows(zc, blo, bhi);
                for (int ib = blo + u.B0; ib <= bhi + u.B0; ib++) {
                    const float z2 = g.zdet[ib] + u.sz;
                    for (int ia = alo + u.A0; ia <= ahi + u.A0; ia++) {
                        const float yd = g.ydet[ia];
                        const float l = fl_chord_box3(x1, y1, z1, u.c * g.OD - u.s * yd, u.s * g.OD + u.c * yd, z2,
                                                      1.0f, 1.0f, g.dz, xc, yc, zc);
                        a = a + l * fl_load(y, (size_t)ib * na + ia);
                    }
                }
                t.acc[k][tid] = a;
            }
            continue;
        }
        auto ballot = [](bool which) { return __builtin_amdgcn_ballot_w64(which); };
        auto lanes = [](uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); };
        // the slices' cells, CA columns wide
        auto slices = [&](auto ca) {
            constexpr int CA = decltype(ca)::value;
            // per column: (x, y) of the ray's entry into and exit from the
            // square, the chord's share, and per end the slope of z on its face
            // (place in zs) and the face's distance from the source and half side;
            // ky, the value's place in its row, is that of the zero for a lane without
            // the column (the lane's last value again would make NaN of an
            // infinite sum: 0 * inf)
            float xi[CA], yi[CA], xo[CA], yo[CA], uv[CA], ni[CA], hi[CA], no[CA], ho[CA];
            int fi[CA], fo[CA], ky[CA];
            uint64_t hit[CA], full[CA];   // lanes whose ray crosses the square; that take the whole routine
            float ec = 0.0f;
#pragma unroll
            for (int c = 0; c < CA; c++) {
                const int ka = min(alo + c, ahi);
                const float sba = t.sba[p0][ka], sab = t.sab[p0][ka], a = t.a[p0][ka], bb = t.b[p0][ka];
                const float hx = a > 0 ? 0.5f : -0.5f, hy = bb > 0 ? 0.5f : -0.5f;
                const float mx = sba * (-p0x) + p0y, wx = sba * hx, my = sab * (-p0y) + p0x, wy = sab * hy;
                const float ex = mx - wx, xx = mx + wx, ey = my - wy, xy = my + wy;
                const bool bex = fl_absf(ex) <= 0.5f, bxx = fl_absf(xx) <= 0.5f;
                const bool bey = fl_absf(ey) <= 0.5f, bxy = fl_absf(xy) <= 0.5f;
                const float steep = fmaxf(fabsf(sba), fabsf(sab)), miss = miss0 + 0x1p-20f * steep;
                const bool off = (fminf(ex, xx) > miss || fmaxf(ex, xx) < -miss || fminf(ey, xy) > miss || fmaxf(ey, xy) < -miss) &&
                                 !(bex || bxx || bey || bxy);
                const bool all = !(steep < 4096.0f) || (!off && (bex == bey || bxx == bxy));
                const uint64_t have = ballot(alo + c <= ahi);
                full[c] = have & ballot(all);
                hit[c] = have & ballot(!off && !all);
                ec = fmaxf(ec, !off && !all ? steep : 0.0f);
                xi[c] = bex ? -hx : ey; yi[c] = bex ? ex : -hy;
                xo[c] = bxx ? hx : xy;  yo[c] = bxx ? xx : hy;
                const float du = xo[c] - xi[c], dv = yo[c] - yi[c];
                uv[c] = du * du + dv * dv;
                ni[c] = bex ? -p0x : -p0y; hi[c] = bex ? hx : hy;
                no[c] = bxx ? -p0x : -p0y; ho[c] = bxx ? hx : hy;
                ky[c] = alo + c <= ahi ? ka : u.nA;
                fi[c] = 2 * ka + (bex ? 0 : 1);
                fo[c] = 2 * ka + (bxx ? 0 : 1);
            }
            const float* zs = (const float*)t.zs;
#pragma unroll 1
            for (int k = 0; k < kn; k++) {
                const float zc = height(k), p2 = z1 - zc;
                const float eps = 0x1p-20f * (fabsf(p2) + 1.0f + tz * ec);
                float a = t.acc[k][tid];
                int blo, bhi;
                rows(zc, blo, bhi);
                for (int kb = blo; kb <= bhi; kb++) {
                    const int row = __mul24(kb, u.nA + 1);
                    float si[CA], so[CA], y[CA], l[CA];
#pragma unroll
                    for (int c = 0; c < CA; c++) {
                        si[c] = zs[2 * row + fi[c]];
                        so[c] = zs[2 * row + fo[c]];
                        y[c] = t.y[row + ky[c]];
                    }
                    uint64_t odd[CA], any = 0;
                    const float hzs = t.ch[p0][kb];
#pragma unroll
                    for (int c = 0; c < CA; c++) {
                        const float zi = (si[c] * ni[c] + p2) - si[c] * hi[c], zo = (so[c] * no[c] + p2) + so[c] * ho[c];
                        const float ai = fabsf(zi) - hz, ao = fabsf(zo) - hz, w = zo - zi;
                        const uint64_t in = ballot(ai <= 0.0f), out = ballot(ao <= 0.0f), cross = hit[c] & (in ^ out);
                        odd[c] = full[c] | hit[c] & (ballot(fabsf(ai) <= eps) | ballot(fabsf(ao) <= eps) | (~(in | out) & ballot(fabsf(w) > hz)));
                        float l2 = uv[c] + w * w;
                        uint64_t some = hit[c] & in & out;
                        if (cross) {   // one end on a z face
                            const bool low = lanes(in);
                            const float2 xs = t.xs[row + ky[c]];
                            const float hs = low ? hzs : -hzs;
                            const float pu = (xs.x * (-p2) + p0x) + xs.x * hs, pv = (xs.y * (-p2) + p0y) + xs.y * hs;
                            const float du = pu - (low ? xi[c] : xo[c]), dv = pv - (low ? yi[c] : yo[c]);
                            const float dw = hs - (low ? zi : zo);
                            l2 = lanes(cross) ? du * du + dv * dv + dw * dw : l2;
                            some |= cross & ballot(fabsf(pu) <= 0.5f) & ballot(fabsf(pv) <= 0.5f);
                        }
                        odd[c] |= some & ballot(l2 < 0x1p-96f);
                        any |= odd[c];
                        l[c] = lanes(some) ? fl_sqrt_mid(l2) : 0.0f;
                    }
                    if (any) {
#pragma unroll
                        for (int c = 0; c < CA; c++)
                            if (odd[c] != 0 && lanes(odd[c])) l[c] = chord(alo + c, kb, zc);
                    }
#pragma unroll
                    for (int c = 0; c < CA; c++) a += l[c] * y[c];
                }
                t.acc[k][tid] = a;
            }
        };
        auto most = [&](int n) { return __builtin_amdgcn_ballot_w64(alo + n <= ahi) == 0; };   // columns of a lane
        if (most(CA0)) slices(std::integral_constant<int, CA0>{});
        else if (most(CA0 + 1)) slices(std::integral_constant<int, CA0 + 1>{});
        else {
#pragma unroll 1
            for (int k = 0; k < kn; k++) {
                const float zc = height(k);
                float a = t.acc[k][tid];
                int blo, bhi;
                rows(zc, blo, bhi);
                for (int kb = blo; kb <= bhi; kb++)
                    for (int ka = alo; ka <= ahi; ka++) a = a + chord(ka, kb, zc) * t.y[__mul24(kb, u.nA + 1) + ka];
                t.acc[k][tid] = a;
            }
        }
    }
    if (col) {
#pragma unroll
        for (int k = 0; k < KZ; k++)
            if (iz0 + k < g.nz)
                fl_store(X, (size_t)it * g.nvox + ((size_t)(iz0 + k) * g.ny + iy) * g.nx + ix, t.acc[k][tid] * g.scale);
    }
}

// Per (view, cell) of a fan plan, the cell's line and its quotients that do
// not depend on the pixel (Atx_fan_mf_cpu_new.cpp:50-53, find_l.cpp:28-42).
__global__ __launch_bounds__(256) void k_fan_line_q(AdjGeom g, int nv, float4* __restrict__ out, float* __restrict__ pd)
{
    const size_t k = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= (size_t)nv * g.na) return;
    const int iv = (int)(k / g.na), id = (int)(k % g.na);
    const float c = g.cphi[iv], s = g.sphi[iv];
    const float sd = g.sdet[id], cd = g.cdet[id];
    const float Px = -(sd * c + cd * s);
    const float Py = cd * c - sd * s;
    const float a2 = fl_absf(Px), b2 = fl_absf(Py);
    const float hx = a2 / 2, hy = b2 / 2;
    out[k] = make_float4(2 * Px, 2 * Py, (hx < hy) ? 1.0f / b2 : 1.0f / a2, 0.25f * (1.0f / (a2 * b2)));
    if (iv == 0) pd[id] = 2 * (g.SO * sd);
}

// Per (view, cell) of a fan plan: the ray's (dx, dy, 1/dx, 1/dy), formed as
// the forward forms dx and dy, and its length.
__global__ __launch_bounds__(256) void k_fan_ray_q(FwdGeom f, int nv, float4* __restrict__ out, float* __restrict__ len)
{
    const size_t k = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= (size_t)nv * f.na) return;
    const int iv = (int)(k / f.na), id = (int)(k % f.na);
    const float c = f.cs[iv], s = f.sn[iv];
    const float x1 = c * (-f.SO), y1 = s * (-f.SO);
    const float yd = f.ydet[id];
    const float x2 = c * f.OD - s * yd;
    const float y2 = s * f.OD + c * yd;
    const float dx = x2 - x1, dy = y2 - y1;
    out[k] = make_float4(dx, dy, dx != 0.0f ? 1.0f / dx : 0.0f, dy != 0.0f ? 1.0f / dy : 0.0f);
    len[k] = sqrtf(dx * dx + dy * dy);
}

hipError_t fl_launch_fan_ray_q(const FwdGeom& f, int nv, float4* out, float* len, hipStream_t st)
{
    const size_t n = (size_t)nv * f.na;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fan_ray_q, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, f, nv, out, len);
    return hipGetLastError();
}

hipError_t fl_launch_fan_line_q(const AdjGeom& g, int nv, float4* out, float* pd, hipStream_t st)
{
    const size_t n = (size_t)nv * g.na;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fan_line_q, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, g, nv, out, pd);
    return hipGetLastError();
}

template <typename YT, typename XT>
static hipError_t launch_adj_fan_t(const void* Y, void* X, const FwdGeom& f, const AdjGeom& g, hipStream_t st)
{
    dim3 grid((g.nx + 15) / 16, (g.ny + 15) / 16, g.nt);
    if (grid.x == 0 || grid.y == 0 || grid.z == 0) return hipSuccess;
    const YT* y = (const YT*)Y;
    XT* x = (XT*)X;
    if (!fl_launch_fan_adj_w<FanExact>(y, x, f, g, st))
        hipLaunchKernelGGL((k_adj_fan<YT, XT>), grid, dim3(16, 16), 0, st, y, x, g);
    return hipGetLastError();
}

// Rows of the largest footprint of a brick of bz slices.
static double exact_rows(const AdjGeom& g, int bz)
{
    const double rc = 0.5 * sqrt((double)g.nx * g.nx + (double)g.ny * g.ny), SD = (double)g.SO + g.OD;
    const double near = std::max((double)g.SO - rc, 1.0), zmax = 0.5 * g.nz * g.dz + bz * g.dz;
    return (bz * g.dz * SD / near + zmax * (SD / near - SD / (near + 11.4))) * fabs((double)g.inv_pb) + 3.0;
}

template <typename YT, typename XT>
static hipError_t launch_adj_cone_t(const void* Y, void* X, const AdjGeom& g, hipStream_t st)
{
    const auto blocks = [&](int kz) { return (uint32_t)((g.nx + 7) / 8) * ((g.ny + 7) / 8) * ((g.nz + 4 * kz - 1) / (4 * kz)); };
    if (blocks(4) == 0 || g.nt == 0) return hipSuccess;
    auto launch = [&](auto kz, auto ca0) {
        constexpr int KZ = decltype(kz)::value, CA0 = decltype(ca0)::value;
        hipLaunchKernelGGL((k_adj_cone_zc<YT, XT, KZ, CA0>), dim3(blocks(KZ), g.nt), dim3(256), 0, st, (const YT*)Y, (XT*)X, g);
    };
    // Panels of under 0.9 cells a voxel (at the axis): lanes have one column or
    // two.  N^3 voxels, one and two columns against two and three, us: 128^3, 60
    // views, 0.33 cells 465 and 620, 0.66 604 and 695, 0.79 714 and 770, 0.99 891
    // and 870; 256^3, 30 views, 0.33 1293 and 1714, 0.79 2085 and 2224, 0.99 2784 and
    // 2721; 64^3, 60 views, 0.33 144 and 186, 0.99 232 and 232.  (In one kernel the
    // three forms cost the fine panels 1.3%.)
    const bool coarse = (g.SO + g.OD) / g.SO * fabsf(g.inv_pa) < 0.9f;
    auto go = [&](auto kz) {
        if (coarse) launch(kz, std::integral_constant<int, 1>{});
        else launch(kz, std::integral_constant<int, 2>{});
    };
    // Slices a thread: eight share a column's work best, but leave few bricks of
    // unequal cost.  N^3 voxels, 96 views, us (eight, four, two): 72^3 1486, 791,
    // 600; 80^3 1518, 805, 685; 96^3 1690, 1075, 1145; 128^3 2448, 2009, 2403;
    // 144^3 2944, 2862, 3333; 256^3, 360 views, ms: 48.4, 51.6, 64.8.  Rows that
    // overflow the tables cost more (helix 180 x 156 x 132: 25.0 ms against 8.5).
    if (blocks(8) * (size_t)g.nt >= 4096 && exact_rows(g, 32) <= FP_B) go(std::integral_constant<int, 8>{});
    else if (blocks(4) * (size_t)g.nt > 640) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 2>{});
    return hipGetLastError();
}

#define FL_DISPATCH_YX(FN, yt, xt, ...)                                                      \
    do {                                                                                     \
        if (yt == FL_F32 && xt == FL_F32) return FN<float, float>(__VA_ARGS__);               \
        if (yt == FL_BF16 && xt == FL_BF16) return FN<bf16_t, bf16_t>(__VA_ARGS__);           \
        if (yt == FL_F16 && xt == FL_F16) return FN<f16_t, f16_t>(__VA_ARGS__);               \
        if (yt == FL_BF16 && xt == FL_F32) return FN<bf16_t, float>(__VA_ARGS__);             \
        if (yt == FL_F16 && xt == FL_F32) return FN<f16_t, float>(__VA_ARGS__);               \
        if (yt == FL_F32 && xt == FL_BF16) return FN<float, bf16_t>(__VA_ARGS__);             \
        if (yt == FL_F32 && xt == FL_F16) return FN<float, f16_t>(__VA_ARGS__);               \
        return hipErrorInvalidValue;                                                         \
    } while (0)

hipError_t fl_launch_adj_fan(const void* Y, int yt, void* X, int xt, const FwdGeom& f, const AdjGeom& g,
                             hipStream_t st)
{
    FL_DISPATCH_YX(launch_adj_fan_t, yt, xt, Y, X, f, g, st);
}

hipError_t fl_launch_adj_cone(const void* Y, int yt, void* X, int xt, const AdjGeom& g, hipStream_t st)
{
    FL_DISPATCH_YX(launch_adj_cone_t, yt, xt, Y, X, g, st);
}
