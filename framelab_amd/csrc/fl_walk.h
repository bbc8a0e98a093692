// fl_walk.h -- the forward projectors' ray walk with tracked cells.
//
// What a step of the walk costs is not its operations but their kind: on
// gfx950 a wave's FP32 add, multiply and FMA, 32-bit integer add and AND, and
// move issue in 2 to 3 cycles of its SIMD (an FMA in over 4 if an operand is a
// scalar register), while compares, selects, min/max, shifts, conversions and
// three-operand integer forms take over 4 (measured, throughput of independent
// chains).  So the walk keeps no per-step index
// arithmetic and no selects: the lanes that cross a plane update that axis
// under the execution mask (walk_cross), and the rules that only matter at
// rounding distance are tested once per batch of steps.
//
// Between the entry parameter and the exit parameter (the smallest last-plane
// parameter of the active axes) the planes passed name the cell of every
// segment: per axis the one between the last plane passed and the next.  The
// reference's rule, floor(o + m d + n/2) of the rounded midpoint m, names the
// same cell unless rounding carries the midpoint over a plane, which a
// segment longer than
//   tau = 2u (4 A + s (2.5 n + 5)/|d|),  u = 2^-24, A the exit parameter,
// rules out on that axis: the planes' parameters are off by at most 2u A |d| +
// u |P| in coordinates (plane coordinate P rounded once, difference and
// quotient rounded), m by u A |d|, m d by u A |d|, the sum, the division by s
// and the addition of n/2 by u (|P| + s), u |P| and u s (n + 1), |P| <=
// s (n/2 + 1), and the midpoint lies half a segment from either plane (with
// s = 1 P is exact and nothing is divided: 1.5 n + 3 for 2.5 n + 5).  A
// segment longer than tau after the exit lies beyond the volume by the same
// argument.  Shorter segments, and those before the entry, take the rule
// itself, so every visited cell is the reference's.
#pragma once

#include "fl_common.h"
#include "fl_siddon.h"

// Steps per batch: the reads of one batch land behind the arithmetic of the
// next (cone 256^3, 360 views: 4, 5, 6 and 8 steps take 9.05, 8.93, 8.89 and
// 9.2 ms in FP32, 8.00, 8.00, 8.04 and 8.7 ms in BF16).
constexpr int WALK_D = 5;
// Cells a lane may read outside the volume: a tracked cell starts at most one
// cell outside, and a lane reads before each of a batch's crossings.
constexpr int WALK_OUTSIDE = WALK_D;

// A layout places the voxels of a frame: fx, fy, fz give a cell's byte offset
// field along an axis (of cells up to WALK_OUTSIDE outside, too), stepx .. its
// change over one cell, to be masked by mx .. (MASKED), place the byte offset
// to read at three fields, at the byte offset of a cell inside.

// Cone volumes: 4 x 4 x 4 bricks, brick counts along x and y rounded up to
// powers of two, and guard slices below and above.  A voxel's place is three
// disjoint bit fields, one per axis (two bits inside the brick, the brick
// index above), so stepping one cell along an axis is an add and an AND:
// field - mask carries through the gaps as +1, field - 1 borrows as -1.  A
// lane that overshoots the volume inside a batch reads a wrapped or guard
// voxel, whose value is never used.
template <unsigned E>
struct ConeBricks {
    static constexpr bool MASKED = true;
    static constexpr int GUARD = (WALK_OUTSIDE + 3) / 4 * 4;
    int lx, ly;            // log2 of the brick counts along x and y
    unsigned mx, my, mz;   // the fields
    __host__ __device__ ConeBricks(int nx, int ny)
    {
        lx = ly = 0;
        while ((4 << lx) < nx) lx++;
        while ((4 << ly) < ny) ly++;
        mx = (3u | ((1u << lx) - 1) << 6) * E;
        my = (12u | ((1u << ly) - 1) << (6 + lx)) * E;
        mz = ~(mx | my) & (0u - E);
    }
    // voxels per frame, guards and padding included
    __host__ __device__ size_t frame(int nz) const
    {
        return ((size_t)64 << (lx + ly)) * ((nz + 3) / 4 + 2 * GUARD / 4);
    }
    __device__ __forceinline__ unsigned fx(int t) const { return (((unsigned)t & 3u) | ((unsigned)t >> 2) << 6) * E & mx; }
    __device__ __forceinline__ unsigned fy(int t) const
    {
        return (((unsigned)t & 3u) << 2 | ((unsigned)t >> 2) << (6 + lx)) * E & my;
    }
    __device__ __forceinline__ unsigned fz(int t) const
    {
        const unsigned z = (unsigned)(t + GUARD);
        return ((z & 3u) << 4 | (z >> 2) << (6 + lx + ly)) * E;
    }
    __device__ __forceinline__ unsigned stepx(int st) const { return st > 0 ? 0u - mx : 0u - E; }
    __device__ __forceinline__ unsigned stepy(int st) const { return st > 0 ? 0u - my : 0u - E * 4; }
    __device__ __forceinline__ unsigned stepz(int st) const { return st > 0 ? 0u - mz : 0u - E * 16; }
    __device__ __forceinline__ unsigned place(unsigned x, unsigned y, unsigned z) const { return x | y | z; }
    __device__ __forceinline__ unsigned at(int tx, int ty, int tz) const { return fx(tx) | fy(ty) | fz(tz); }
};

// Fan images: row by row, as they come; an offset outside reads the last pixel.
template <unsigned E>
struct FanImage {
    static constexpr bool MASKED = false;
    unsigned row, last;
    static constexpr unsigned mx = ~0u, my = ~0u, mz = ~0u;
    __device__ FanImage(int nx, int ny) : row((unsigned)nx * E), last((unsigned)nx * (unsigned)ny * E - E) {}
    __device__ __forceinline__ unsigned fx(int t) const { return (unsigned)t * E; }
    __device__ __forceinline__ unsigned fy(int t) const { return (unsigned)t * row; }
    __device__ __forceinline__ unsigned fz(int) const { return 0u; }
    __device__ __forceinline__ unsigned stepx(int st) const { return (unsigned)st * E; }
    __device__ __forceinline__ unsigned stepy(int st) const { return (unsigned)st * row; }
    __device__ __forceinline__ unsigned stepz(int) const { return 0u; }
    __device__ __forceinline__ unsigned place(unsigned x, unsigned y, unsigned) const { return min(x + y, last); }
    __device__ __forceinline__ unsigned at(int tx, int ty, int) const { return fx(tx) + fy(ty); }
};

// Fan images in 4 x 4 bricks, brick counts along x rounded up to powers of two:
// as ConeBricks without z.  An offset outside reads the last pixel.
template <unsigned E>
struct FanBricks {
    static constexpr bool MASKED = true;
    int lx;
    unsigned mx, my, last;
    static constexpr unsigned mz = ~0u;
    __host__ __device__ FanBricks(int nx, int ny)
    {
        lx = 0;
        while ((4 << lx) < nx) lx++;
        mx = (3u | ((1u << lx) - 1) << 4) * E;
        my = ~mx & (0u - E);
        last = (unsigned)frame(ny) * E - E;
    }
    __host__ __device__ size_t frame(int ny) const { return ((size_t)16 << lx) * ((ny + 3) / 4); }
    __device__ __forceinline__ unsigned fx(int t) const { return (((unsigned)t & 3u) | ((unsigned)t >> 2) << 4) * E & mx; }
    __device__ __forceinline__ unsigned fy(int t) const
    {
        return (((unsigned)t & 3u) << 2 | ((unsigned)t >> 2) << (4 + lx)) * E & my;
    }
    __device__ __forceinline__ unsigned fz(int) const { return 0u; }
    __device__ __forceinline__ unsigned stepx(int st) const { return st > 0 ? 0u - mx : 0u - E; }
    __device__ __forceinline__ unsigned stepy(int st) const { return st > 0 ? 0u - my : 0u - E * 4; }
    __device__ __forceinline__ unsigned stepz(int) const { return 0u; }
    __device__ __forceinline__ unsigned place(unsigned x, unsigned y, unsigned) const { return min(x | y, last); }
    __device__ __forceinline__ unsigned at(int tx, int ty, int) const { return fx(tx) | fy(ty); }
};

// One axis of the walk: next plane (parameter a, coordinate index p), tracked
// cell (field f, as a byte offset, and its step), constants.
struct WalkAxis {
    SidAxis ax;
    float r;         // 1/d, correctly rounded
    float a, p, st;
    unsigned f, inc;
    __device__ __forceinline__ float alpha(int j) const
    {
        return sid_div((float)(ax.i0 + ax.st * j) * ax.s - ax.o, ax.d, r);
    }
};

__device__ __forceinline__ void walk_axis_init(WalkAxis& q, float o, float d, float s, int n)
{
    sid_axis_init(q.ax, o, d, s, n);
    q.r = q.ax.on ? 1.0f / d : 0.0f;
    q.st = (float)q.ax.st;
}

// If the axis's next plane is the one just reached (an), pass it: the plane
// after it (its parameter by the reference's quotient, sid_div) and the cell.
// Runs under the execution mask of the lanes concerned: one compare and cheap
// operations instead of as many selects.  `all` is the mask to restore; m the
// cell field's mask.
// OV: the register class of the origin, uniform over the wave (s) or not (v).
#define WALK_CROSS_ASM(SCALE, NUM, MASK, OV)                                                          \
    asm volatile("v_cmpx_eq_f32_e32 vcc, %0, %5\n\t"                                                  \
                 "v_add_f32_e32 %1, %6, %1\n\t"                                                       \
                 "v_add_u32_e32 %2, %7, %2\n\t" SCALE                                                 \
                 "v_subrev_f32_e32 %3, %8, " NUM "\n\t" MASK                                          \
                 "v_mul_f32_e32 %4, %3, %10\n\t"                                                      \
                 "v_fma_f32 %3, -%4, %9, %3\n\t"                                                      \
                 "v_fma_f32 %0, %3, %10, %4\n\t"                                                      \
                 "s_mov_b64 exec, %12"                                                                \
                 : "+v"(q.a), "+v"(q.p), "+v"(q.f), "=&v"(num), "=&v"(quo)                            \
                 : "v"(an), "v"(q.st), "v"(q.inc), OV(q.ax.o), "v"(q.ax.d), "v"(q.r), "s"(m), "s"(all), "s"(q.ax.s) \
                 : "vcc")
#define WALK_SCALE "v_mul_f32_e32 %3, %13, %1\n\t"
#define WALK_MASK "v_and_b32_e32 %2, %11, %2\n\t"
template <bool S1, bool UNIFORM, bool MASKED>
__device__ __forceinline__ void walk_cross(WalkAxis& q, float an, unsigned m, uint64_t all)
{
    float num, quo;
    if constexpr (UNIFORM && MASKED && S1) WALK_CROSS_ASM("", "%1", WALK_MASK, "s");
    else if constexpr (UNIFORM && MASKED) WALK_CROSS_ASM(WALK_SCALE, "%3", WALK_MASK, "s");
    else if constexpr (MASKED) {
        static_assert(S1, "a form in use");
        WALK_CROSS_ASM("", "%1", WALK_MASK, "v");
    } else {
        static_assert(S1 && !UNIFORM, "a form in use");
        WALK_CROSS_ASM("", "%1", "", "v");
    }
}
#undef WALK_SCALE
#undef WALK_MASK
#undef WALK_CROSS_ASM

// The planes around parameter t: c of them are below it, `prev` is the last of
// those (-inf: none) and `next` the first at or above it (+inf: none).
struct WalkAround {
    int c;
    float prev, next;
};
__device__ __forceinline__ WalkAround walk_around(const WalkAxis& q, float t, float rs)
{
    const int n = q.ax.n;
    const float est = ((q.ax.o + t * q.ax.d) * rs - (float)q.ax.i0) * q.st;
    int c = sid_floor(fminf(fmaxf(est, -1.0f), (float)n)) + 1;   // an estimate, 0 .. n + 1
    float prev = q.alpha(c - 1), next = q.alpha(c);
    while (c > 0 && prev >= t) {
        next = prev;
        prev = q.alpha(--c - 1);
    }
    while (c <= n && next < t) {
        prev = next;
        next = q.alpha(++c);
    }
    return WalkAround{c, c > 0 ? prev : -FL_INF, c <= n ? next : FL_INF};
}

// Walks a wave's rays and returns their sums, y = y + S*x in walk order.  NZ3:
// three axes (Z unused otherwise); DZ1: z planes one apart; UNIFORM: the rays
// share their source.  vol: the frame in layout `lay`; live: the lane has a
// ray.  Called by all lanes of a wave.
template <bool NZ3, bool DZ1, bool UNIFORM, typename VT, class Layout>
__device__ __forceinline__ float walk_rays(WalkAxis& X, WalkAxis& Y, WalkAxis& Z, float L, bool live,
                                           const VT* __restrict__ vol, const Layout& lay)
{
    constexpr int D = WALK_D;
    const SidAxis &ax = X.ax, &ay = Y.ax, &az = Z.ax;
    const float rs = DZ1 ? 1.0f : 1.0f / az.s;
    const float hx = (float)ax.nh, hy = (float)ay.nh, hz = (float)az.nh;
    auto cell = [&](float m, int& tx, int& ty, int& tz) {
        tx = sid_floor((ax.o + m * ax.d) + hx);
        ty = sid_floor((ay.o + m * ay.d) + hy);
        tz = 0;
        if (NZ3) {
            float c = az.o + m * az.d;
            if (!DZ1) c = sid_div(c, az.s, rs);
            tz = sid_floor(c + hz);
        }
        return sid_in(ax, tx) && sid_in(ay, ty) && (!NZ3 || sid_in(az, tz));
    };
    auto far = [&](int tx, int ty, int tz) { return sid_far(ax, tx) || sid_far(ay, ty) || (NZ3 && sid_far(az, tz)); };
    auto near = [&](int tx, int ty, int tz) { return sid_near(ax, tx) || sid_near(ay, ty) || (NZ3 && sid_near(az, tz)); };
    auto next = [&] { return NZ3 ? sid_min3(X.a, Y.a, Z.a) : sid_min(X.a, Y.a); };
    auto read = [&](unsigned off) { return fl_raw((const VT*)((const char*)vol + off)); };
    auto value = [&](decltype(read(0u)) r) { return fl_unraw((const VT*)nullptr, r); };
    float acc = 0.0f;

    // axes without planes: their cell is the same all along
    int tx0 = 0, ty0 = 0, tz0 = 0;
    if (!ax.on || !ay.on || (NZ3 && !az.on)) {
        (void)cell(0.5f, tx0, ty0, tz0);
        if ((!ax.on && !sid_in(ax, tx0)) || (!ay.on && !sid_in(ay, ty0)) || (NZ3 && !az.on && !sid_in(az, tz0)) ||
            (!ax.on && !ay.on && (!NZ3 || !az.on)))
            live = false;
    }
    float ae = -FL_INF, aexit = FL_INF, k = 0.0f;
    auto bounds = [&](const WalkAxis& q) {
        if (!q.ax.on) return;
        ae = fmaxf(ae, q.alpha(0));
        aexit = fminf(aexit, q.alpha(q.ax.n));
        const float w = q.ax.s == 1.0f ? 1.5f * (float)q.ax.n + 3.0f : q.ax.s * (2.5f * (float)q.ax.n + 5.0f);
        k = fmaxf(k, w * __builtin_amdgcn_rcpf(fabsf(q.ax.d)));
    };
    bounds(X);
    bounds(Y);
    if (NZ3) bounds(Z);
    const float tau = 1.01f * 0x1p-23f * (4.0f * fmaxf(aexit, 0.0f) + k);

    // Start: the entry, moved left while the preceding segment is not
    // provably before the volume (as sid_start).
    float cur = ae;
    const WalkAround none{0, -FL_INF, FL_INF};
    WalkAround wx = none, wy = none, wz = none;
    while (live) {
        if (ax.on) wx = walk_around(X, cur, 1.0f);
        if (ay.on) wy = walk_around(Y, cur, 1.0f);
        if (NZ3 && az.on) wz = walk_around(Z, cur, rs);
        const float pred = fmaxf(fmaxf(wx.prev, wy.prev), wz.prev);
        if (pred == -FL_INF) break;
        int tx, ty, tz;
        (void)cell((pred + cur) * 0.5f, tx, ty, tz);
        if (near(tx, ty, tz)) break;
        cur = pred;
    }
    // next planes, those at the start passed; an axis past its last plane has
    // none (sid_next_init)
    auto place = [&](WalkAxis& q, WalkAround& w) {
        while (w.c <= q.ax.n && w.next <= cur) w.next = q.alpha(++w.c);
        q.p = (float)(q.ax.i0 + q.ax.st * w.c);
        q.a = q.ax.on && w.c <= q.ax.n ? w.next : FL_INF;
    };
    place(X, wx);
    place(Y, wy);
    if (NZ3) place(Z, wz);
    else Z.a = FL_INF;

    // a step by the reference's rule; false once beyond the volume
    auto pass = [&](WalkAxis& q, float an) {
        SidNext n{q.a, q.p, q.st, q.r};
        sid_next_step<false>(n, q.ax, an);
        q.a = n.a;
        q.p = n.p;
    };
    auto exact_step = [&] {
        const float an = next();
        int tx, ty, tz;
        const bool in = cell((cur + an) * 0.5f, tx, ty, tz);
        if (in) acc = acc + ((an - cur) * L) * value(read(lay.at(tx, ty, tz)));
        const bool stop = !in && far(tx, ty, tz);
        pass(X, an);
        pass(Y, an);
        if (NZ3) pass(Z, an);
        cur = an;
        return !stop;
    };
    while (live && cur < ae) live = exact_step();   // rarely any: segments that rounding puts inside early

    // the tracked cell: the one the next plane closes
    auto track = [&](const WalkAxis& q, int t0) {
        if (!q.ax.on) return live ? t0 : 0;
        return q.ax.st > 0 ? (int)q.p - 1 + q.ax.nh : (int)q.p + q.ax.nh;
    };
    X.f = lay.fx(track(X, tx0));
    Y.f = lay.fy(track(Y, ty0));
    Z.f = NZ3 ? lay.fz(track(Z, tz0)) : 0u;
    X.inc = lay.stepx(ax.st);
    Y.inc = lay.stepy(ay.st);
    if (NZ3) Z.inc = lay.stepz(az.st);

    // run: still walking (without a plane ahead there is nothing to walk).  A
    // lane that has finished gets NaN plane parameters: it crosses nothing, and
    // whatever is computed from them is masked by run or ran.  (Lane masks, so
    // that the tests of a batch are scalar.)  Compiled with NaN semantics; the
    // mins are written out (sid_min), which cost as little as without.
    uint64_t run = __builtin_amdgcn_ballot_w64(live && next() < FL_INF);
    float nan;
    asm volatile("v_mov_b32_e32 %0, 0x7fc00000" : "=v"(nan));
    auto stop = [&](bool which) {
        X.a = which ? nan : X.a;
        Y.a = which ? nan : Y.a;
        if (NZ3) Z.a = which ? nan : Z.a;
    };
    stop(__builtin_amdgcn_inverse_ballot_w64(~run));
    struct Batch {
        float S[D];
        decltype(read(0u)) x[D];
        uint64_t ran;
    };
    const uint64_t all = __builtin_amdgcn_read_exec();
    auto issue = [&](Batch& t) {
        const float from = cur;
        float an[D], dmin = FL_INF, even = 0.0f;
#pragma unroll
        for (int u = 0; u < D; u++) {
            an[u] = next();
            const float dal = an[u] - cur;
            t.S[u] = dal * L;
            t.x[u] = read(lay.place(X.f, Y.f, Z.f));
            if (u % 2 == 1) dmin = sid_min3(dmin, even, dal);
            else if (u == D - 1) dmin = sid_min(dmin, dal);
            else even = dal;
            walk_cross<true, UNIFORM, Layout::MASKED>(X, an[u], lay.mx, all);
            walk_cross<true, UNIFORM, Layout::MASKED>(Y, an[u], lay.my, all);
            if constexpr (NZ3) walk_cross<DZ1, UNIFORM, Layout::MASKED>(Z, an[u], lay.mz, all);
            cur = an[u];
        }
        t.ran = run;
        const uint64_t outm = run & __builtin_amdgcn_ballot_w64(cur > aexit);
        const uint64_t tinym = run & __builtin_amdgcn_ballot_w64(dmin <= tau);
        if (outm) {
            // past the exit: terms outside read as 0 (S * 0 = +0).  A lane
            // whose last segment is long is done; one whose last segment is
            // short stays for the rule to tell, its cell moving no further.
            const bool out = __builtin_amdgcn_inverse_ballot_w64(outm);
#pragma unroll
            for (int u = 0; u < D; u++)
                if (out && an[u] > aexit) t.x[u] = 0;
            const bool fin = out && cur - an[D - 2] > tau;
            run &= ~__builtin_amdgcn_ballot_w64(fin);
            stop(fin);
            X.inc = out ? 0u : X.inc;
            Y.inc = out ? 0u : Y.inc;
            if (NZ3) Z.inc = out ? 0u : Z.inc;
        }
        if (__builtin_expect(tinym != 0, 0)) {
            const bool tiny = __builtin_amdgcn_inverse_ballot_w64(tinym);
            // segments too short for the planes to tell their cell: the rule,
            // which also ends a ray once it is beyond the volume
            float c0 = from;
            bool beyond = false;
#pragma unroll
            for (int u = 0; u < D; u++) {
                if (tiny && !(an[u] - c0 > tau)) {
                    int tx, ty, tz;
                    t.x[u] = 0;
                    if (cell((c0 + an[u]) * 0.5f, tx, ty, tz)) t.x[u] = read(lay.at(tx, ty, tz));
                    else if (far(tx, ty, tz)) beyond = true;
                }
                c0 = an[u];
            }
            run &= ~__builtin_amdgcn_ballot_w64(beyond);
            stop(beyond);
        }
    };
    auto commit = [&](const Batch& t) {
        if (__builtin_amdgcn_inverse_ballot_w64(t.ran)) {
#pragma unroll
            for (int u = 0; u < D; u++) acc = acc + t.S[u] * value(t.x[u]);
        }
    };
    Batch a, b;
    issue(a);
    for (;;) {
        if (!run) {
            commit(a);
            break;
        }
        issue(b);
        commit(a);
        if (!run) {
            commit(b);
            break;
        }
        issue(a);
        commit(b);
    }
    return acc;
}
