// matched.hip -- voxel-driven transpose of the Siddon forward projector.
//
// For voxel v and a ray crossing it, the Siddon walk's segment inside v runs
// from the largest entry-plane parameter to the smallest exit-plane
// parameter of v's three face pairs; no other plane parameter of the ray
// lies strictly between them (each axis' parameters are monotone in the
// plane index), so that interval is exactly one element pair of the forward
// walk.  Computing the plane parameters with the forward's float formula
// ((float)i*s - o)/d therefore gives the forward's segment a_out - a_in bit for
// bit, |d| is the forward's too, and the forward's midpoint rule decides
// whether the walk credits v with it (segments shorter than the float
// resolution may have their rounded midpoint in a neighbouring voxel).  What
// differs is the rounding of a term: where the forward adds (segment |d|) x, the
// staged cone form adds segment (|d| y), fused with the sum; the fan and the
// cone's general loop round segment |d| first.  The result is the transpose of
// the FP32 forward to those roundings, so <Ax,y> = <x,A^T y> holds to
// summation rounding.  Gathers only: a voxel's sum belongs to one thread (view
// groups add theirs in a fixed order), no atomics, deterministic.
//
// No reference counterpart: the reference pairs its Siddon forward with the
// exact-chord adjoint, whose float chords differ from the forward's lengths
// by ~1e-5 relative.  This is the backward used for gradients.
#include "fl_capi_internal.h"
#include "fl_common.h"
#include "fl_geom.h"
#include "fl_siddon.h"
#include "fl_chord.h"
#include "fl_fan.h"
#include "fl_fan_adj.h"

// Per (ray, voxel) pair: the length (in parameter) of the Siddon segment of the
// ray inside the voxel, credited where the forward's midpoint rule maps it
// there, or 0.  in/out: entry and exit plane parameters, of x and y together
// and of z.
__device__ __forceinline__ float matched_length(float inxy, float outxy, float inz, float outz, const SidAxis& ax,
                                                const SidAxis& ay, const SidAxis& az, int ix, int iy, int iz, bool dz_one)
{
    const float ain = fmaxf(inxy, inz), aout = fminf(outxy, outz);
    const float m = (ain + aout) * 0.5f;
    // (every test evaluated: no short-circuit branches)
    const int hit = int(aout > ain) & int(sid_cell_xy(ax, m) == ix) & int(sid_cell_xy(ay, m) == iy) &
                    int(sid_cell_z(az, m, dz_one) == iz);
    return hit ? aout - ain : 0.0f;
}

namespace {
constexpr int MF_A = 48;     // footprint columns in LDS
constexpr int MF_B = 64;     // footprint rows
constexpr int MF_W = 2048;   // footprint cells, a column's padded to an odd count
static_assert(MF_A <= 64 && MF_B <= 64, "footprint columns / rows are staged by one wave each");

// What a group of four waves stages of a view: per footprint column the plane
// parameters of its brick's nine x and y planes, per row the entry and exit
// parameters of each slice's z planes, per cell ray length times sinogram value
// (column by column; zeros for a column that is none).  What the tables are
// formed from is double-buffered: written a view ahead.
template <int BZ>
struct MatchedLds {
    float ax[MF_A][9], ay[MF_A][9];
    float2 zio[MF_B][BZ];
    float w[MF_W], zero[MF_B];
    float dx[2][MF_A], dy[2][MF_A], rx[2][MF_A], ry[2][MF_A], dxy2[2][MF_A], tc[2][MF_A];
    float dz[2][MF_B], rz[2][MF_B], dz2[2][MF_B], tz[2][MF_B];
    ShadowCols cols[2][64];
};
}  // namespace

// 3D, footprint-staged, z-column form: a workgroup is a brick of 8 x 8 x 4 KZ
// voxels (KZ = 8, or 4 in small volumes), and each thread of a group of four
// waves owns KZ z-adjacent voxels of one (x, y) column.  Per view the group stages its footprint (MatchedLds;
// each plane parameter the forward's IEEE quotient, formed once per group);
// each voxel then visits the cells of its own shadow, two or three columns of a
// row at a time.
//
// The segment of a (ray, voxel) pair is the smallest of four differences of
// plane parameters: between the column's slab interval (kept in registers) and
// the slice's (read per row) both ways, and of either itself.  Where it is
// longer than tau the forward's midpoint rule credits the voxel (the argument
// in fl_walk.h: tau = 1.01 2^-23 (4 A + w/|d|), the largest over the axes), and
// where it is below -tau there is none; only what lies between takes the rule
// itself.  A z difference far larger than the segment cannot upset the rule
// along z, so the test is on the differences that involve z planes, and a
// column whose own interval is that short sends its rows there outright.
//
// The staged directions are 2^-e times the forward's, 2^e above every |d|
// (FwdGeom::seg_up): |d| times a value near the type's largest would overflow
// where the term does not.  Plane parameters, segments and tau are 2^e times
// the forward's for it, exactly, and the factors cancel in a midpoint's
// coordinates and in a term.
//
// VG groups share a brick's views between them and add their sums in group
// order.
//
// Bound by the waits between its two barriers a view and by VALU issue: some 120
// instructions a voxel and view at 256^3 (1.8 rows of 2.3 columns at 20, the
// rows' ranges 20, the column's slab 9, the rest the tables), issued at 0.21 a
// SIMD and cycle while 0.49 of the waves' cycles wait (helix 0.16 and 0.46,
// 128^3 0.18 and 0.47, 64^3 0.16 and 0.51).  Spills, of vector and scalar
// registers: 36 and 54 with eight slices (148 bytes a lane), 8 and 31 with four
// (36 bytes), 4 more where dz != 1.  256^3, 360 views x
// 512 x 384: 28.6 -> 21.4 ms; 128^3, 180 views: 2.13 -> 1.45 ms; 64^3, 60 views:
// 276 -> 81 us; helix 180 x 156 x 132, 241 views x 301 x 217: 15.3 -> 4.0 ms
// (before: four cell tests per pair, with a division where dz != 1, tables of
// 32 rows, four slices and one group throughout).  Four waves per SIMD; three
// (no spills) take 23.7 ms at 256^3.
template <typename YT, typename XT, int KZ, int VG, bool DZ1>
__global__ __launch_bounds__(256 * VG, 4) void k_adj_matched_cone(
    const YT* __restrict__ Y, XT* __restrict__ X, FwdGeom f, AdjGeom g)
{
    constexpr int BZ = 4 * KZ;
    constexpr int NY = 2;   // values a thread loads a view ahead
    __shared__ __align__(16) MatchedLds<BZ> s_lds[VG];

    const int bx = (f.nx + 7) / 8, by = (f.ny + 7) / 8, bz = (f.nz + BZ - 1) / BZ;
    const uint32_t nblk = (uint32_t)bx * by * bz;
    const uint32_t b = fl_xcd_remap(blockIdx.x, nblk);
    const int it = blockIdx.y;
    const int grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
    const int tid = threadIdx.x & 255, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    MatchedLds<BZ>& t = s_lds[grp];
    const int ix0 = (int)(b % bx) * 8, iy0 = (int)((b / bx) % by) * 8, iz0 = (int)(b / ((uint32_t)bx * by)) * BZ;
    const int lx = tid & 7, ly = (tid >> 3) & 7, lz0 = wv * KZ;
    const int ix = ix0 + lx, iy = iy0 + ly;
    const bool col = ix < f.nx && iy < f.ny;
    const int kn = min(KZ, f.nz - iz0 - lz0);   // slices of this wave inside the volume

    const int na = f.na, nb = f.nb;
    const float SD = f.SO + f.OD;
    const float xc = (float)ix + 0.5f - (float)(f.nx / 2);
    const float yc = (float)iy + 0.5f - (float)(f.ny / 2);
    const ShadowMap ma = fl_shadow_map(f.ya0, f.inv_pa, 0.05f), mb = fl_shadow_map(f.zb0, f.inv_pb, 0.05f);
    const float klo = mb.klo + 1.0f, khi = mb.khi;   // floor(k + 1) for ceil(k): the margin covers whole k
    const bool up = f.inv_pb > 0;
    const float z0 = (float)(iz0 + lz0 - f.nz / 2);
    // z planes one voxel apart: the z cell index needs no division (a
    // compile-time choice: a runtime flag lets the divide be speculated)
    constexpr bool dz_one = DZ1;
    // tau's constants (fl_walk.h): plane parameters reach at most A here
    const float rc = 0.5f * sqrtf((float)f.nx * f.nx + (float)f.ny * f.ny);
    const float A4 = 4.0f * 1.01f * (f.SO + rc + 1.0f) / SD * f.seg_up;
    const float wx = 1.5f * (float)f.nx + 3.0f, wy = 1.5f * (float)f.ny + 3.0f;
    const float wz = DZ1 ? 1.5f * (float)f.nz + 3.0f : f.dz0 * (2.5f * (float)f.nz + 5.0f);
    float acc[KZ];
#pragma unroll
    for (int k = 0; k < KZ; k++) acc[k] = 0.0f;
    if (tid < MF_B) t.zero[tid] = 0.0f;

    // The group's views are its own 0, 1, ...: own view i is view i * VG + grp
    // of the frame's list; 64 of them at a time are set up one per lane: source
    // and direction, sinogram slot and the brick's footprint on the panel.
    const int nvf = g.Nv[it], nown = (nvf - grp + VG - 1) / VG, ntrip = (nvf + VG - 1) / VG;
    float uc = 0.0f, us = 0.0f, usz = 0.0f;
    int uslot = 0, ua = 0, uan = 0, ub = 0, ubn = 0;   // first column and row and their counts
    auto setup = [&](int i) {
        const int j = min((i + lane) * VG + grp, nvf - 1);
        const int iv = g.id_Y[it * g.tmp_size + j];
        uslot = g.id_S[it * g.tmp_size + j];
        uc = f.cs[iv];
        us = f.sn[iv];
        usz = f.sdz[iv];
        // the brick, a hundredth of a voxel wider, and a tenth of a cell
        const float xm = (float)(ix0 + 4 - f.nx / 2), ym = (float)(iy0 + 4 - f.ny / 2);
        const float e = 4.01f * (fabsf(uc) + fabsf(us));
        const float D = uc * xm + us * ym + f.SO, yr = uc * ym - us * xm;
        const float rn = __builtin_amdgcn_rcpf(D - e) * SD, rf = __builtin_amdgcn_rcpf(D + e) * SD;
        const float zl = ((float)(iz0 - f.nz / 2) - 0.01f) * f.dz0 - usz;
        const float zh = ((float)(iz0 + BZ - f.nz / 2) + 0.01f) * f.dz0 - usz;
        const float yl = yr - e, yh = yr + e;
        const ShadowMap wa = fl_shadow_map(f.ya0, f.inv_pa, 0.15f), wb = fl_shadow_map(f.zb0, f.inv_pb, 0.15f);
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
        v.any = i < nown && v.nA > 0 && v.nB > 0;
        v.fits = v.nA <= MF_A && v.nB <= MF_B && v.nA * (v.nB | 1) <= MF_W;
        return v;
    };
    // a view ahead: direction components, their reciprocals and taus of the
    // columns (wave 0) and rows (wave 1), the shadows of the thread columns (the
    // same in all four waves: the other two, in turn) and the cells' values
    float yv[NY];
    auto stage = [&](const View& v, int p) {
        if (!v.any) return;
        if (v.fits) {
            if (wv == 0 && lane < v.nA) {
                const float x1 = v.c * (-f.SO), y1 = v.s * (-f.SO), yd = f.ydet[v.A0 + lane];
                const float dx = ((v.c * f.OD - v.s * yd) - x1) * f.seg_down, dy = ((v.s * f.OD + v.c * yd) - y1) * f.seg_down;
                const float rx = 1.0f / dx, ry = 1.0f / dy;
                t.dx[p][lane] = dx;
                t.dy[p][lane] = dy;
                t.rx[p][lane] = rx;
                t.ry[p][lane] = ry;
                t.dxy2[p][lane] = dx * dx + dy * dy;   // the first two terms of |d|^2, summed as the forward sums them
                t.tc[p][lane] = 1.01f * 0x1p-23f * (A4 + fmaxf(wx * fabsf(rx), wy * fabsf(ry)));
            }
            if (wv == 1 && lane < v.nB) {
                const float dz = ((f.zdet[v.B0 + lane] + v.sz) - v.sz) * f.seg_down;
                const float rz = 1.0f / dz;
                t.dz[p][lane] = dz;
                t.rz[p][lane] = rz;
                t.dz2[p][lane] = dz * dz;
                t.tz[p][lane] = 1.01f * 0x1p-23f * (wz * fabsf(rz));
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
        if (wv == 2 + p) t.cols[p][lane] = fl_shadow_cols(v.c, v.s, f.SO, SD, xc, yc, ma, na);
    };
    View v{};
    int p = 0;   // the buffer of the staged view
    if (nvf > 0) {
        setup(0);
        v = view(0);
        stage(v, 0);
    }
    for (int i = 0; i < ntrip; i++) {
        if (VG == 1 && !v.any) {   // the brick is off the panel; the other buffer may be in use
            if (i + 1 < ntrip) {
                if ((i + 1) % 64 == 0) setup(i + 1);
                v = view(i + 1);
                stage(v, p);
            }
            continue;
        }
        const bool staged = v.any && v.fits;
        const float x1 = v.c * (-f.SO), y1 = v.s * (-f.SO), z1 = v.sz;
        __syncthreads();
        if (staged) {
            // plane coordinate i -> ((float)i - o)/d, the forward's IEEE
            // quotient, from the staged reciprocal of d
            if ((tid & 15) < 9) {
                const int q = tid & 15;
                const float nx = (float)(ix0 + q - f.nx / 2) - x1, ny = (float)(iy0 + q - f.ny / 2) - y1;
                for (int ka = tid >> 4; ka < v.nA; ka += 16) {
                    t.ax[ka][q] = sid_div(nx, t.dx[p][ka], t.rx[p][ka]);
                    t.ay[ka][q] = sid_div(ny, t.dy[p][ka], t.ry[p][ka]);
                }
            }
            // per row and brick slice the parameters of the slice's two z
            // planes (the forward's quotients), ordered as entry and exit
            // along the ray (+-inf for a ray parallel to them)
            {
                const int q = tid % BZ;
                const float n0 = (float)(iz0 + q - f.nz / 2) * f.dz0 - z1, n1 = (float)(iz0 + q + 1 - f.nz / 2) * f.dz0 - z1;
                for (int kb = tid / BZ; kb < v.nB; kb += 256 / BZ) {
                    const float dz = t.dz[p][kb], rz = t.rz[p][kb];
                    const float lo = sid_div(n0, dz, rz), hi = sid_div(n1, dz, rz);
                    t.zio[kb][q] = dz != 0.0f ? make_float2(fminf(lo, hi), fmaxf(lo, hi)) : make_float2(-FL_INF, FL_INF);
                }
            }
            // |d| = sqrtf(dx*dx + dy*dy + dz*dz), the forward's ray length
            // (left-to-right sum, correctly rounded root), times the value
            const uint32_t mA = fl_small_div_m((uint32_t)v.nA);
            auto put = [&](int k, float yk) {
                const int kb = fl_small_div(k, mA), ka = k - __mul24(kb, v.nA);
                t.w[__mul24(ka, v.nB | 1) + kb] = fl_sqrt_nonneg(t.dxy2[p][ka] + t.dz2[p][kb]) * yk;
            };
            const int cells = v.nA * v.nB;
#pragma unroll
            for (int q = 0; q < NY; q++)
                if (q * 256 + tid < cells) put(q * 256 + tid, yv[q]);
            for (int k = NY * 256 + tid; k < cells; k += 256) {
                const int kb = fl_small_div(k, mA), ka = k - __mul24(kb, v.nA);
                put(k, fl_load(Y + v.off, (size_t)(v.B0 + kb) * na + (v.A0 + ka)));
            }
        }
        const View u = v;
        if (i + 1 < ntrip) {
            if ((i + 1) % 64 == 0) setup(i + 1);
            v = view(i + 1);
        }
        __syncthreads();
        const int p0 = p;
        p ^= 1;
        if (i + 1 < ntrip) stage(v, p);
        const ShadowCols sc = t.cols[p0][lane];
        if (!u.any || !col || sc.alo > sc.ahi) continue;
        // rows of slice k, from its edges' projections at the column's near and
        // far ends (e: the lower edge's, handed on to the next slice)
        const float rn = sc.rn * mb.inv_p, rf = sc.rf * mb.inv_p;
        struct Edge {
            float lo, hi;
        };
        auto edge = [&](int k) {
            const float e = (z0 + (float)k) * f.dz0 - u.sz;
            return Edge{fminf(e * rn, e * rf), fmaxf(e * rn, e * rf)};
        };
        const float kl = klo - (float)u.B0, kh = khi - (float)u.B0;
        auto rows = [&](Edge& e, int k, int& blo, int& bhi) {
            const Edge e1 = edge(k + 1);
            blo = max(sid_floor((up ? e.lo : e1.lo) + kl), 0);
            bhi = min(sid_floor((up ? e1.hi : e.hi) + kh), u.nB - 1);
            e = e1;
        };
        if (staged) {
            const int alo = max(sc.alo, u.A0) - u.A0, ahi = min(sc.ahi, u.A0 + u.nA - 1) - u.A0;
            const int wst = u.nB | 1;
            // CA columns from a on
            auto part = [&](auto ca, int a) {
                constexpr int CA = decltype(ca)::value;
                float ixy[CA], oxy[CA], dxy[CA], thc = 0.0f;
                const float* wp[CA];
#pragma unroll
                for (int c = 0; c < CA; c++) {
                    const int ka = min(a + c, ahi);
                    const float x0 = t.ax[ka][lx], x2 = t.ax[ka][lx + 1], y0 = t.ay[ka][ly], y2 = t.ay[ka][ly + 1];
                    const float tc = t.tc[p0][ka];
                    float inx = fminf(x0, x2), outx = fmaxf(x0, x2), iny = fminf(y0, y2), outy = fmaxf(y0, y2);
                    if (!(tc < FL_INF)) {   // parallel to an axis's planes: the rule decides
                        if (t.dx[p0][ka] == 0.0f) { inx = -FL_INF; outx = FL_INF; }
                        if (t.dy[p0][ka] == 0.0f) { iny = -FL_INF; outy = FL_INF; }
                    }
                    ixy[c] = fmaxf(inx, iny);
                    oxy[c] = fminf(outx, outy);
                    dxy[c] = oxy[c] - ixy[c];
                    wp[c] = &t.w[__mul24(ka, wst)];
                    if (a + c <= ahi && dxy[c] > 0.0f) {
                        thc = fmaxf(thc, dxy[c] > tc ? tc : FL_INF);
                    } else {   // misses the (x, y) column: nothing, whatever its values
                        ixy[c] = -1e30f;
                        oxy[c] = 1e30f;
                        dxy[c] = -1.0f;
                        wp[c] = t.zero;
                    }
                }
                Edge e = edge(0);
#pragma unroll
                for (int k = 0; k < KZ; k++) {
                    if (k >= kn) break;
                    int blo, bhi;
                    rows(e, k, blo, bhi);
                    for (int kb = blo; kb <= bhi; kb++) {
                        const float2 zio = t.zio[kb][lz0 + k];
                        const float th = thc + t.tz[p0][kb], dzz = zio.y - zio.x;
                        float w[CA], l[CA], near = dzz;
#pragma unroll
                        for (int c = 0; c < CA; c++) w[c] = wp[c][kb];
#pragma unroll
                        for (int c = 0; c < CA; c++) {
                            const float d1 = oxy[c] - zio.x, d2 = zio.y - ixy[c];
                            near = fminf(near, fminf(fabsf(d1), fabsf(d2)));
                            l[c] = __builtin_amdgcn_fmed3f(fminf(fminf(d1, d2), dxy[c]), 0.0f, dzz);
                        }
                        if (near <= th) {
                            SidAxis ax, ay, az;
                            sid_axis_init(az, z1, t.dz[p0][kb], f.dz0, f.nz);
#pragma unroll
                            for (int c = 0; c < CA; c++) {
                                if (dxy[c] <= 0.0f) continue;
                                const int ka = a + c;
                                sid_axis_init(ax, x1, t.dx[p0][ka], 1.0f, f.nx);
                                sid_axis_init(ay, y1, t.dy[p0][ka], 1.0f, f.ny);
                                l[c] = matched_length(ixy[c], oxy[c], zio.x, zio.y, ax, ay, az, ix, iy, iz0 + lz0 + k, dz_one);
                            }
                        }
#pragma unroll
                        for (int c = 0; c < CA; c++) acc[k] = __builtin_fmaf(l[c], w[c], acc[k]);
                    }
                }
            };
            // two columns or three, whichever the wave needs
            for (int a = alo; a <= ahi;) {
                if (__builtin_amdgcn_ballot_w64(a + 1 < ahi) == 0) {
                    part(std::integral_constant<int, 2>{}, a);
                    a += 2;
                } else {
                    part(std::integral_constant<int, 3>{}, a);
                    a += 3;
                }
            }
        } else {
            const YT* __restrict__ y = Y + u.off;
            Edge e = edge(0);
#pragma unroll
            for (int k = 0; k < KZ; k++) {
                if (k >= kn) break;
                const int iz = iz0 + lz0 + k;
                int blo, bhi;
                rows(e, k, blo, bhi);
                for (int ib = blo + u.B0; ib <= bhi + u.B0; ib++) {
                    const float dz = (f.zdet[ib] + u.sz) - z1;
                    SidAxis az;
                    sid_axis_init(az, z1, dz, f.dz0, f.nz);
                    const FlAxisIv sv = fl_slab_r(az, iz, 1.0f / dz);
                    for (int ia = max(sc.alo, u.A0); ia <= min(sc.ahi, u.A0 + u.nA - 1); ia++) {
                        const float yd = f.ydet[ia];
                        const float dx = (u.c * f.OD - u.s * yd) - x1, dy = (u.s * f.OD + u.c * yd) - y1;
                        SidAxis ax, ay;
                        sid_axis_init(ax, x1, dx, 1.0f, f.nx);
                        sid_axis_init(ay, y1, dy, 1.0f, f.ny);
                        const FlAxisIv sx = fl_slab_r(ax, ix, 1.0f / dx), sy = fl_slab_r(ay, iy, 1.0f / dy);
                        const float len = matched_length(fmaxf(sx.in, sy.in), fminf(sx.out, sy.out), sv.in, sv.out, ax, ay,
                                                         az, ix, iy, iz, dz_one);
                        const float Si = len * sqrtf(dx * dx + dy * dy + dz * dz);
                        if (Si != 0.0f) acc[k] = __builtin_fmaf(Si, fl_load(y, (size_t)ib * na + ia), acc[k]);
                    }
                }
            }
        }
    }
    if constexpr (VG > 1) {
        // the groups' sums, in group order
        __syncthreads();
        float* part = (float*)&s_lds[grp];
#pragma unroll
        for (int k = 0; k < KZ; k++) part[k * 256 + tid] = acc[k];
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int o = 1; o < VG; o++)
#pragma unroll
            for (int k = 0; k < KZ; k++) acc[k] = acc[k] + ((const float*)&s_lds[o])[k * 256 + tid];
    }
    if (col) {
#pragma unroll
        for (int k = 0; k < KZ; k++) {
            const int iz = iz0 + lz0 + k;
            if (iz < f.nz) fl_store(X, (size_t)it * f.nvox + ((size_t)iz * f.ny + iy) * f.nx + ix, acc[k] * f.scale);
        }
    }
}

// General form: one lane per pixel.
template <typename YT, typename XT>
__global__ __launch_bounds__(256) void k_adj_matched_fan(const YT* __restrict__ Y, XT* __restrict__ X,
                                                        FwdGeom f, AdjGeom g)
{
    const int ix = blockIdx.x * 16 + threadIdx.x;
    const int iy = blockIdx.y * 16 + threadIdx.y;
    const int it = blockIdx.z;
    if (ix >= f.nx || iy >= f.ny) return;
    fl_store(X, (size_t)it * f.nvox + (size_t)iy * f.nx + ix, fl_fan_matched_pixel(Y, f, g, it, ix, iy));
}

// Rows of the largest footprint of a brick of bz slices.
static double matched_rows(const FwdGeom& f, int bz)
{
    const double rc = 0.5 * sqrt((double)f.nx * f.nx + (double)f.ny * f.ny), SD = (double)f.SO + f.OD;
    const double near = std::max((double)f.SO - rc, 1.0), zmax = 0.5 * f.nz * f.dz0 + bz * f.dz0;
    return (bz * f.dz0 * SD / near + zmax * (SD / near - SD / (near + 11.4))) * fabs((double)f.inv_pb) + 3.0;
}

template <typename YT, typename XT>
static hipError_t launch_matched_t(const void* Y, void* X, const fl_plan_s* p, hipStream_t st)
{
    const FwdGeom& f = p->fg;
    if (p->cone) {
        const auto blocks = [&](int kz) { return (uint32_t)((f.nx + 7) / 8) * ((f.ny + 7) / 8) * ((f.nz + 4 * kz - 1) / (4 * kz)); };
        auto go = [&](auto kz, auto vg) {
            constexpr int KZ = decltype(kz)::value, VG = decltype(vg)::value;
            const dim3 grid(blocks(KZ), p->nt), block(256 * VG);
            if (f.dz0 == 1.0f)
                hipLaunchKernelGGL((k_adj_matched_cone<YT, XT, KZ, VG, true>), grid, block, 0, st, (const YT*)Y, (XT*)X, f, p->ag);
            else
                hipLaunchKernelGGL((k_adj_matched_cone<YT, XT, KZ, VG, false>), grid, block, 0, st, (const YT*)Y, (XT*)X, f, p->ag);
        };
        using I8 = std::integral_constant<int, 8>;
        using I4 = std::integral_constant<int, 4>;
        using I1 = std::integral_constant<int, 1>;
        // N^3 voxels, 96 views, us (eight slices a thread, four, four with the
        // views shared by four groups): 48^3 536, 319, 125; 80^3 585, 349, 245;
        // 96^3 614, 435, 473; 112^3 727, 689, 705; 120^3 743, 815, 921; 128^3
        // 759, 839, 961.  Four groups pay while a CU has at most two such
        // workgroups to run, eight slices once it has three or more.  A finely
        // sampled panel keeps to four slices (helix 180 x 156 x 132, rows 0.36
        // slices apart: 4.0 ms, 18.5 ms where the rows overflow the tables).
        if (blocks(4) * (size_t)p->nt <= 512) go(I4{}, I4{});
        else if (blocks(8) * (size_t)p->nt >= 768 && matched_rows(f, 32) <= MF_B) go(I8{}, I1{});
        else go(I4{}, I1{});
    } else {
        dim3 grid((f.nx + 15) / 16, (f.ny + 15) / 16, p->nt);
        if (!fl_launch_fan_adj_w<FanMatched>((const YT*)Y, (XT*)X, f, p->ag, st))
            hipLaunchKernelGGL((k_adj_matched_fan<YT, XT>), grid, dim3(16, 16), 0, st, (const YT*)Y, (XT*)X, f,
                               p->ag);
    }
    return hipGetLastError();
}

hipError_t fl_launch_adj_matched(const void* Y, int yt, void* X, int xt, const fl_plan_s* p, hipStream_t st)
{
    if (yt == FL_F32 && xt == FL_F32) return launch_matched_t<float, float>(Y, X, p, st);
    if (yt == FL_BF16 && xt == FL_BF16) return launch_matched_t<bf16_t, bf16_t>(Y, X, p, st);
    if (yt == FL_F16 && xt == FL_F16) return launch_matched_t<f16_t, f16_t>(Y, X, p, st);
    if (yt == FL_BF16 && xt == FL_F32) return launch_matched_t<bf16_t, float>(Y, X, p, st);
    if (yt == FL_F16 && xt == FL_F32) return launch_matched_t<f16_t, float>(Y, X, p, st);
    if (yt == FL_F32 && xt == FL_BF16) return launch_matched_t<float, bf16_t>(Y, X, p, st);
    if (yt == FL_F32 && xt == FL_F16) return launch_matched_t<float, f16_t>(Y, X, p, st);
    return hipErrorInvalidValue;
}
