// capi.hip -- the C ABI of libframelab_hip.so: plans, drop-in entry points,
// error reporting.  Host code only; kernels live in siddon.hip / adjoint.hip.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "../../include/framelab_hip.h"
#include "fl_capi_internal.h"

// ------------------------------------------------------------ errors -----

static thread_local int tl_err = FL_OK;
static thread_local char tl_msg[512] = "";

int fl_fail(int code, const char* fmt, ...)
{
    tl_err = code;
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(tl_msg, sizeof tl_msg, fmt, ap);
    va_end(ap);
    return code;
}

int fl_ok()
{
    tl_err = FL_OK;
    tl_msg[0] = 0;
    return FL_OK;
}

int fl_hip_fail(hipError_t e, const char* what)
{
    return fl_fail(FL_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

extern "C" int fl_get_last_error(void) { return tl_err; }
extern "C" const char* fl_last_error_message(void) { return tl_msg; }
extern "C" const char* fl_error_string(int code)
{
    switch (code) {
    case FL_OK: return "ok";
    case FL_ERR_INVALID: return "invalid argument";
    case FL_ERR_HIP: return "HIP runtime error";
    case FL_ERR_ALLOC: return "device allocation failed";
    case FL_ERR_UNSUPPORTED: return "unsupported";
    default: return "unknown error";
    }
}
extern "C" int fl_version(void) { return 100; }

// ------------------------------------------------------------- plans -----

template <typename T>
static int upload(T** dst, const T* src, size_t n, const char* what)
{
    *dst = nullptr;
    if (n == 0) return FL_OK;
    hipError_t e = hipMalloc((void**)dst, n * sizeof(T));
    if (e != hipSuccess) return fl_fail(FL_ERR_ALLOC, "hipMalloc(%s, %zu bytes)", what, n * sizeof(T));
    e = hipMemcpy(*dst, src, n * sizeof(T), hipMemcpyHostToDevice);
    if (e != hipSuccess) return fl_hip_fail(e, what);
    return FL_OK;
}

static void plan_free_arrays(fl_plan_s* p)
{
    void* ptrs[] = {p->d_cs, p->d_sn, p->d_sdz, p->d_ydet, p->d_zdet, p->d_cphi, p->d_sphi,
                    p->d_cdet, p->d_sdet, p->d_slot_view, p->d_view_frame, p->d_idY, p->d_idS, p->d_Nv,
                    p->d_bricks,
                    p->d_fb_px, p->d_fb_py, p->d_fb_pd, p->d_cdet2, p->d_sdet2, p->d_line_q,
                    p->d_line_d, p->d_fan_views, p->d_ray_q, p->d_ray_l};
    for (void* q : ptrs)
        if (q) (void)hipFree(q);
    if (p->fwd_done) (void)hipEventDestroy(p->fwd_done);
}

// Forwards of one plan share its brick buffer, so each that uses it is ordered
// after the previous one, whatever streams they run on: wait for the event
// the previous forward recorded, record it again after this one (a fan
// forward that would wait takes no bricks: fl_bricks_busy).  A stream
// under graph capture is left alone (external events cannot enter a
// capture); the solvers that capture forwards order their private stream
// against the caller's, and a fan forward that anyone else captures takes no
// bricks (fl_forward_ordered).
static int fwd_order_begin(fl_plan_s* p, hipStream_t st, bool& order)
{
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess) cs = hipStreamCaptureStatusNone;
    order = p->fwd_done != nullptr && cs == hipStreamCaptureStatusNone;
    if (order && p->fwd_pending) {
        const hipError_t e = hipStreamWaitEvent(st, p->fwd_done, 0);
        if (e != hipSuccess) return fl_hip_fail(e, "forward ordering");
    }
    return FL_OK;
}

static int fwd_order_end(fl_plan_s* p, hipStream_t st, bool order)
{
    if (!order) return FL_OK;
    const hipError_t e = hipEventRecord(p->fwd_done, st);
    if (e != hipSuccess) return fl_hip_fail(e, "forward ordering");
    p->fwd_pending = true;
    p->fwd_stream = p->fwd_after = st;
    return FL_OK;
}

// Fan forwards on several streams need not wait for one another: the image as
// it is gives the same bits as its bricks.  (The query is made in relaxed
// capture mode, so that it is allowed while some other stream is captured.)
bool fl_bricks_busy(fl_plan_s* p, hipStream_t st)
{
    if (p->cone || !p->fwd_pending || st == p->fwd_stream || st == p->fwd_after) return false;
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    const bool busy = hipEventQuery(p->fwd_done) != hipSuccess;
    if (busy) (void)hipGetLastError();   // hipErrorNotReady
    if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
    return busy;
}

void fl_bricks_ordered(fl_plan_s* p, hipStream_t earlier, hipStream_t later)
{
    std::lock_guard<std::mutex> lk(p->fwd_mu);
    if (later != p->fwd_stream && (earlier == p->fwd_stream || earlier == p->fwd_after)) p->fwd_after = later;
}

// AdjGeom::win_ref for a cone plan: whether the reference's detector window
// (Atx_cone_mf_gpu_new.cu:64-73) can exclude a cell of a voxel's shadow
// window, per axis (bit 0 columns, bit 1 rows).  The rotated unit square of
// a voxel reaches ex = (|cos|+|sin|)/2 from its centre both along and across
// the ray axis, so at centre depth D = SO + xr its shadow's outer column
// edge is at most (|yr| + ex) SD / (D - ex) from the axis, the window's at
// (|yr| + 1) SD / D; the first is the smaller when ex (|yr| + 1) <= (1 - ex) D.
// For rows (half-height dz/2 against the window's d = sqrt((1+dz^2)/2)) the
// condition is ex (|zr| + d) <= (d - dz/2) D.  Both are checked at their
// worst voxel and view.  The two windows' index maps then differ by a
// constant (half a cell and y_os on the reference grid), which must leave
// 0.15 cells for the shadow's 0.05-cell margin and the rounding of both.
static int cone_ref_window_bits(const fl_geometry* g, double pa, double pb, const std::vector<float>& cphi,
                                const std::vector<float>& sphi, const std::vector<float>& sdz)
{
    double ex = 0.0;
    for (size_t v = 0; v < cphi.size(); v++) ex = fmax(ex, 0.5 * (fabs((double)cphi[v]) + fabs((double)sphi[v])));
    ex += 1e-6;
    const double SO = g->SO, SD = (double)g->SO + g->OD;
    const double rc = 0.5 * sqrt((double)(g->nx - 1) * (g->nx - 1) + (double)(g->ny - 1) * (g->ny - 1));
    const double dmin = SO - rc - 1.0;   // below every voxel centre's depth
    if (!(dmin > 0) || !(ex < 1)) return 3;
    int bits = 0;
    {
        const double geo = (1 - ex) * SO - ex - rc * sqrt((1 - ex) * (1 - ex) + ex * ex);
        const double slack = fabs(1.0 / pa - 1.0 / g->dy_det) * (rc + 1) * SD / dmin;
        const double off = -(double)g->y_det[0] / pa + g->y_os - (double)(g->na / 2);
        if (!(pa > 0 && g->dy_det > 0 && geo > 1e-3 * SO && fabs(off) + slack < 0.8)) bits |= 1;
    }
    {
        const double dz = g->dz, hz = dz / 2, d = sqrt((1 + dz * dz) / 2);
        const double zlo = (0.5 - g->nz / 2) * dz, zhi = (g->nz - 0.5 - g->nz / 2) * dz;
        double zmax = 0.0;
        for (float s : sdz) zmax = fmax(zmax, fmax(fabs(zlo - s), fabs(zhi - s)));
        const double geo = (d - hz) * dmin - ex * (zmax + d);
        const double slack = fabs(1.0 / pb - 1.0 / g->dz_det) * (zmax + d) * SD / dmin;
        const double off = -(double)g->z_det[0] / pb - (double)(g->nb / 2);
        if (!(pb > 0 && g->dz_det > 0 && geo > 1e-3 * SO && fabs(off) + slack < 0.8)) bits |= 2;
    }
    return bits;
}

// Cells a pixel's shadow can meet on a fan plan's detector, for the windowed
// adjoints (fl_fan_adj_tile); 0 where they must not be used.  The windowed
// form evaluates every cell of the shadow widened by `margin` cells, which
// holds every cell of non-zero chord or coefficient, and gives the reference's
// sum if the reference's window (Atx_fan_mf_cpu_new.cpp:41-47) holds them too.
// That needs: the shadow inside (|yr| + 1) SD / D (the condition of
// cone_ref_window_bits), whose index map floors on both sides, so that its
// constant offset may lie within (-1, 0) less the margins; detector cells
// on a uniform grid, angle tables that point at them to 0.02 cells, and the
// adjoint's view angles equal to the forward's (the matched adjoint's) to
// 0.01 cells; and a margin far above the rounding of a chord's distance test
// (some 3e-7 (SO + rc)).
static int fan_shadow_cells(const fl_geometry* g, double pa, double det_dev, const std::vector<float>& cphi,
                            const std::vector<float>& sphi, const std::vector<float>& cs,
                            const std::vector<float>& sn, const std::vector<float>& cdet,
                            const std::vector<float>& sdet, AdjGeom& out)
{
    const double margin = 0.05, SO = g->SO, SD = (double)g->SO + g->OD;
    double ex = 0.0;
    for (size_t v = 0; v < cphi.size(); v++) {
        const double c = cphi[v], s = sphi[v];
        if (!(fabs(c * c + s * s - 1.0) < 1e-5)) return 0;
        ex = fmax(ex, 0.5 * (fabs(c) + fabs(s)));
    }
    const double rc = 0.5 * sqrt((double)(g->nx - 1) * (g->nx - 1) + (double)(g->ny - 1) * (g->ny - 1));
    const double dmin = SO - rc - 0.01;   // below every pixel centre's depth
    if (!(pa > 0) || !(g->dy_det > 0) || !(det_dev <= FL_DET_DEV_MAX) || !(dmin > 4 * ex)) return 0;
    for (size_t v = 0; v < cphi.size(); v++)
        if (!(fmax(fabs(cphi[v] - cs[v]), fabs(sphi[v] - sn[v])) * 2 * (rc + 1) * SD / dmin < 0.01 * pa)) return 0;
    for (int a = 0; a < g->na; a++) {
        const double c = cdet[a], s = sdet[a];
        if (!(c > 0) || !(fabs(c * c + s * s - 1.0) < 1e-5) || !(fabs(SD * s / c - g->y_det[a]) < 0.02 * pa)) return 0;
    }
    const double geo = (1 - ex) * SO - ex - rc * sqrt((1 - ex) * (1 - ex) + ex * ex);
    const double slack = fabs(1.0 / pa - 1.0 / g->dy_det) * (rc + 1) * SD / dmin + margin + 0.05;
    const double off = -(double)g->y_det[0] / pa + g->y_os - (double)(g->na / 2);
    if (!(geo > 1e-3 * SO) || !(off + slack < 0) || !(slack - off < 1)) return 0;
    if (!((margin - 0.04) * 0.9 * pa * dmin / SD > 1e-6 * (SO + rc))) return 0;
    const double gr = 1.0 + ex / (dmin - ex);   // 1/(1 + dx/D) of a pixel's corner
    const double tg = rc / sqrt(SO * SO - rc * rc);
    const double hmax = sqrt(0.5 * (1.0 + tg * tg)) * gr * (1.0 + 1e-5);
    const double cells = 2.0 * hmax * SD / dmin / pa + 2 * margin + 1e-3;
    // the shadow of a tile's pixels: centres within e of the tile's (whose own
    // may lie that far beyond the image's corner)
    const double e = 3.5 * 2 * ex, dtile = dmin - 2 * e;
    if (!(dtile > e) || !(cells < 7)) return 0;
    const double tile = (2 * e * (1 + tg + e / dtile) + 2 * hmax) * SD / dtile / pa;
    int n = (int)floor(cells) + 1;
    n = n <= 2 ? 2 : n <= 4 ? n : n <= 6 ? 6 : 0;   // the instantiated counts
    out.fan_tile = (int)tile + 4 + n;
    out.fan_grow = (float)(0.5 * gr * (1.0 + 1e-5));
    out.fan_hmax = (float)hmax;
    out.fan_sdp = (float)(SD / pa);
    out.fan_klo = (float)(-(double)g->y_det[0] / pa - margin);
    return n <= g->na && out.fan_tile <= 64 ? n : 0;
}

extern "C" int fl_plan_create(fl_plan* out, const fl_geometry* g) { return fl_plan_create_with(out, g, true); }

int fl_plan_create_with(fl_plan* out, const fl_geometry* g, bool fan_bricks)
{
    if (!out || !g) return fl_fail(FL_ERR_INVALID, "null plan or geometry");
    *out = nullptr;
    const bool cone = g->nz > 0;
    if (g->nx <= 0 || g->ny <= 0 || g->nz < 0 || g->nt <= 0 || g->nv <= 0 || g->na <= 0 || g->nb <= 0)
        return fl_fail(FL_ERR_INVALID, "non-positive size (nx=%d ny=%d nz=%d nt=%d nv=%d na=%d nb=%d)",
                       g->nx, g->ny, g->nz, g->nt, g->nv, g->na, g->nb);
    if ((g->nx & 1) || (g->ny & 1) || (cone && (g->nz & 1)))
        return fl_fail(FL_ERR_INVALID, "volume sides must be even (plane index runs -n/2..n/2)");
    if (!cone && g->nb != 1) return fl_fail(FL_ERR_INVALID, "fan geometry needs nb == 1");
    if (!(g->SO > 0) || !(g->OD > 0) || !(g->scale > 0))
        return fl_fail(FL_ERR_INVALID, "SO, OD and scale must be positive");
    if (cone && !(g->dz > 0)) return fl_fail(FL_ERR_INVALID, "dz must be positive");
    if (!g->sd_phi || !g->y_det || (cone && (!g->z_det || !g->sd_z)))
        return fl_fail(FL_ERR_INVALID, "missing sd_phi / y_det / z_det / sd_z");
    if (g->tmp_size < 0) return fl_fail(FL_ERR_INVALID, "tmp_size < 0");
    const long long nvox = (long long)g->nx * g->ny * (cone ? g->nz : 1);
    const long long ndet = (long long)g->na * g->nb;
    if (nvox >= (1LL << 31)) return fl_fail(FL_ERR_INVALID, "volume exceeds 2^31 voxels per frame");

    // view -> frame, validated
    std::vector<int> view_frame(g->nv, 0);
    if (g->id_X) {
        for (int v = 0; v < g->nv; v++) {
            if (g->id_X[v] < 0 || g->id_X[v] >= g->nt)
                return fl_fail(FL_ERR_INVALID, "id_X[%d]=%d outside [0,nt)", v, g->id_X[v]);
            view_frame[v] = g->id_X[v];
        }
    } else if (g->nt != 1) {
        return fl_fail(FL_ERR_INVALID, "id_X required when nt > 1");
    }
    std::vector<int> slot_view(g->nv);
    for (int k = 0; k < g->nv; k++) {
        int v = g->slot_view ? g->slot_view[k] : k;
        if (v < 0 || v >= g->nv) return fl_fail(FL_ERR_INVALID, "slot_view[%d]=%d outside [0,nv)", k, v);
        slot_view[k] = v;
    }
    // frame -> views for the adjoint
    int tmp = g->tmp_size;
    std::vector<int> idY, Nv(g->nt);
    if (g->id_Y && g->Nv) {
        for (int it = 0; it < g->nt; it++) {
            Nv[it] = g->Nv[it];
            if (Nv[it] < 0 || Nv[it] > tmp) return fl_fail(FL_ERR_INVALID, "Nv[%d]=%d outside [0,tmp_size]", it, Nv[it]);
        }
        idY.assign(g->id_Y, g->id_Y + (size_t)tmp * g->nt);
        for (int it = 0; it < g->nt; it++)
            for (int j = 0; j < Nv[it]; j++) {
                int v = idY[(size_t)it * tmp + j];
                if (v < 0 || v >= g->nv) return fl_fail(FL_ERR_INVALID, "id_Y entry %d outside [0,nv)", v);
            }
    } else {
        // frame lists from view -> frame (views ascending within each
        // frame), the lists setPara builds (ConeBeamScanner/setPara.m:59-80)
        std::fill(Nv.begin(), Nv.end(), 0);
        for (int v = 0; v < g->nv; v++) Nv[view_frame[v]]++;
        tmp = 0;
        for (int it = 0; it < g->nt; it++) tmp = Nv[it] > tmp ? Nv[it] : tmp;
        idY.assign((size_t)tmp * g->nt, 0);
        std::vector<int> fill(g->nt, 0);
        for (int v = 0; v < g->nv; v++) {
            const int it = view_frame[v];
            idY[(size_t)it * tmp + fill[it]++] = v;
        }
    }
    if (idY.empty()) idY.push_back(0);
    // The adjoint reads the frame-list entry (it, j) from the slot the
    // forward writes its view to: the n-th listing of view v (frames in
    // order, then list order) reads the n-th slot holding v.  Without
    // slot_view, slot k holds view k.  (The reference GPU wrappers fill and
    // read their sinograms in this frame-list order,
    // Ax_cone_mf_gpu_new.cu:500-517, Atx_cone_mf_gpu_new.cu:140-150.)
    std::vector<int> idS(idY);
    bool slots_ok = true;
    if (g->slot_view) {
        std::vector<std::vector<int>> holders(g->nv);
        for (int k = 0; k < g->nv; k++) holders[slot_view[k]].push_back(k);
        std::vector<size_t> used(g->nv, 0);
        for (int it = 0; it < g->nt; it++)
            for (int j = 0; j < Nv[it]; j++) {
                const size_t e = (size_t)it * tmp + j;
                const int v = idY[e];
                if (used[v] < holders[v].size()) idS[e] = holders[v][used[v]++];
                else slots_ok = false;
            }
    }

    // forward trig: cosf/sinf of the single-precision angles, as the
    // reference's C++ forward evaluates (float)cos(sd_phi[iv])
    std::vector<float> cs(g->nv), sn(g->nv), cphi(g->nv), sphi(g->nv);
    for (int v = 0; v < g->nv; v++) {
        cs[v] = cosf(g->sd_phi[v]);
        sn[v] = sinf(g->sd_phi[v]);
        cphi[v] = g->cos_phi ? g->cos_phi[v] : (float)cos((double)g->sd_phi[v]);
        sphi[v] = g->sin_phi ? g->sin_phi[v] : (float)sin((double)g->sd_phi[v]);
    }
    std::vector<float> sdz(g->nv, 0.0f), zdet(cone ? g->nb : 1, 0.0f);
    if (cone) {
        for (int v = 0; v < g->nv; v++) sdz[v] = g->sd_z[v];
        for (int b = 0; b < g->nb; b++) zdet[b] = g->z_det[b];
    }
    std::vector<float> cdet(g->na, 0.0f), sdet(g->na, 0.0f);
    if (!cone) {
        for (int a = 0; a < g->na; a++) {
            if (g->cos_det && g->sin_det) {
                cdet[a] = g->cos_det[a];
                sdet[a] = g->sin_det[a];
            } else {
                double ang = atan2((double)g->y_det[a], (double)(g->SO + g->OD));
                float af = (float)ang;
                cdet[a] = (float)cos((double)af);
                sdet[a] = (float)sin((double)af);
            }
        }
    }

    fl_plan_s* p = new (std::nothrow) fl_plan_s();
    if (!p) return fl_fail(FL_ERR_ALLOC, "host allocation");
    (void)hipGetDevice(&p->device);
    p->cone = cone;
    p->nvox = nvox;
    p->ndet = ndet;
    p->nt = g->nt;
    p->nv = g->nv;
    p->h_sd_phi.assign(g->sd_phi, g->sd_phi + g->nv);
    p->slots_ok = slots_ok;
    int rc = FL_OK;
    if ((rc = upload(&p->d_cs, cs.data(), cs.size(), "cos table")) ||
        (rc = upload(&p->d_sn, sn.data(), sn.size(), "sin table")) ||
        (rc = upload(&p->d_sdz, sdz.data(), sdz.size(), "sd_z")) ||
        (rc = upload(&p->d_ydet, g->y_det, (size_t)g->na, "y_det")) ||
        (rc = upload(&p->d_zdet, zdet.data(), zdet.size(), "z_det")) ||
        (rc = upload(&p->d_cphi, cphi.data(), cphi.size(), "cos_phi")) ||
        (rc = upload(&p->d_sphi, sphi.data(), sphi.size(), "sin_phi")) ||
        (rc = upload(&p->d_cdet, cdet.data(), cdet.size(), "cos_det")) ||
        (rc = upload(&p->d_sdet, sdet.data(), sdet.size(), "sin_det")) ||
        (rc = upload(&p->d_slot_view, slot_view.data(), slot_view.size(), "slot_view")) ||
        (rc = upload(&p->d_view_frame, view_frame.data(), view_frame.size(), "id_X")) ||
        (rc = upload(&p->d_idY, idY.data(), idY.size(), "id_Y")) ||
        (rc = upload(&p->d_idS, idS.data(), idS.size(), "slot per frame-list entry")) ||
        (rc = upload(&p->d_Nv, Nv.data(), Nv.size(), "Nv"))) {
        plan_free_arrays(p);
        delete p;
        return rc;
    }
    if (!cone && g->cos_det2 && g->sin_det2 &&
        ((rc = upload(&p->d_cdet2, g->cos_det2, (size_t)g->na + 1, "cos_det2")) ||
         (rc = upload(&p->d_sdet2, g->sin_det2, (size_t)g->na + 1, "sin_det2")))) {
        plan_free_arrays(p);
        delete p;
        return rc;
    }
    p->h_ydet.assign(g->y_det, g->y_det + g->na);
    p->h_zdet = zdet;
    p->h_sdz = sdz;
    if (cone) {
        // the forward gathers from a bricked copy of its input (padded to
        // whole bricks of the largest layout; 4-byte elements cover every
        // storage type), in the tracked walk's layout if there is room
        const size_t tr = fl_cone_copy_bytes(g->nx, g->ny, g->nz, g->nt, true);
        if (tr) {
            p->fg.tracked = hipMalloc(&p->d_bricks, tr) == hipSuccess;
            if (!p->fg.tracked) (void)hipGetLastError();
        }
        if (!p->fg.tracked && hipMalloc(&p->d_bricks, fl_cone_copy_bytes(g->nx, g->ny, g->nz, g->nt, false)) != hipSuccess)
            rc = fl_fail(FL_ERR_ALLOC, "brick buffer");
        else if (hipEventCreateWithFlags(&p->fwd_done, hipEventDisableTiming) != hipSuccess)
            rc = fl_fail(FL_ERR_HIP, "forward ordering event");
    }
    // fan: likewise, if there is room, from 150 000 rays on.  A gather of 64
    // lanes touches 52 cache lines of a 1024 x 1024 image as it is, some 15 of
    // its 4 x 4 bricks, but the copy is a launch and an ordering event more
    // (8 us): 256 x 256, 256 views x 256 cells 40 us as it is, 48 from bricks;
    // 360 x 512 102 and 85; 384 x 384, 400 x 500 145 and 136; 1024 x 1024, 900 x
    // 1000 1176 and 925, 900 x 2000 1866 and 1313
    const size_t fb = !cone && fan_bricks && (size_t)g->nv * g->na >= 150000 ? fl_fan_brick_elems(g->nx, g->ny) : 0;
    if (!rc && fb) {
        p->fg.tracked = hipMalloc(&p->d_bricks, fb * (size_t)g->nt * 4) == hipSuccess;
        if (!p->fg.tracked) {
            p->d_bricks = nullptr;
            (void)hipGetLastError();
        } else if (hipEventCreateWithFlags(&p->fwd_done, hipEventDisableTiming) != hipSuccess) {
            rc = fl_fail(FL_ERR_HIP, "forward ordering event");
        }
    }
    if (rc) {
        plan_free_arrays(p);
        delete p;
        return rc;
    }

    FwdGeom& f = p->fg;
    f.cs = p->d_cs; f.sn = p->d_sn; f.sdz = p->d_sdz; f.ydet = p->d_ydet; f.zdet = p->d_zdet;
    f.slot_view = p->d_slot_view; f.view_frame = p->d_view_frame;
    f.SO = g->SO; f.OD = g->OD; f.scale = g->scale; f.dz0 = cone ? g->dz : 1.0f;
    f.nx = g->nx; f.ny = g->ny; f.nz = cone ? g->nz : 0; f.na = g->na; f.nb = g->nb;
    f.nslots = g->nv; f.nvox = (size_t)nvox; f.nframes = g->nt;
    f.bricks = p->d_bricks;
    // 16 x 16-ray workgroups of 8 x 8-ray waves gathering from 4 x 4 x 4
    // bricks: the fastest shape measured at 256^3 (fl_plan_autotune retimes)
    f.tile = cone ? 6 : 0;

    AdjGeom& a = p->ag;
    a.cphi = p->d_cphi; a.sphi = p->d_sphi; a.cdet = p->d_cdet; a.sdet = p->d_sdet;
    a.sdz = p->d_sdz; a.ydet = p->d_ydet; a.zdet = p->d_zdet; a.id_Y = p->d_idY; a.id_S = p->d_idS;
    a.Nv = p->d_Nv;
    a.SO = g->SO; a.OD = g->OD; a.scale = g->scale; a.dy_det = g->dy_det; a.y_os = g->y_os;
    a.dz_det = g->dz_det; a.dz = cone ? g->dz : 1.0f;
    a.nx = g->nx; a.ny = g->ny; a.nz = cone ? g->nz : 1; a.na = g->na; a.nb = g->nb; a.nt = g->nt;
    a.tmp_size = tmp; a.nvox = (size_t)nvox; a.nd = (size_t)ndet;
    // detector index maps (uniform pitch) used to bound voxel shadows
    {
        const double pa = g->na > 1 ? ((double)g->y_det[g->na - 1] - g->y_det[0]) / (g->na - 1) : (double)g->dy_det;
        const double pb = (cone && g->nb > 1) ? ((double)g->z_det[g->nb - 1] - g->z_det[0]) / (g->nb - 1)
                                              : (double)(cone ? g->dz_det : 1.0f);
        f.ya0 = a.ya0 = g->y_det[0];
        f.inv_pa = a.inv_pa = (float)(1.0 / pa);
        f.zb0 = a.zb0 = cone ? g->z_det[0] : 0.0f;
        f.inv_pb = a.inv_pb = (float)(1.0 / pb);
        // (a panel 2^40 voxels away has no precision left to lose)
        double y2 = 0.0, z2 = 0.0;
        for (int k = 0; k < g->na; k++) y2 = fmax(y2, (double)g->y_det[k] * g->y_det[k]);
        for (int k = 0; cone && k < g->nb; k++) z2 = fmax(z2, (double)g->z_det[k] * g->z_det[k]);
        const double SD = (double)g->SO + g->OD, len = sqrt(SD * SD + y2 + z2);
        const int e = len < 0x1p40 ? std::max(ilogb(len) + 1, 0) : 0;
        f.seg_up = ldexpf(1.0f, e);
        f.seg_down = ldexpf(1.0f, -e);
        // deviation from the uniform grids the window maps assume
        double dev = 0.0;
        for (int k = 0; k < g->na && pa != 0.0; k++)
            dev = fmax(dev, fabs(((double)g->y_det[k] - g->y_det[0]) / pa - k));
        for (int k = 0; cone && k < g->nb && pb != 0.0; k++)
            dev = fmax(dev, fabs(((double)g->z_det[k] - g->z_det[0]) / pb - k));
        p->det_dev = dev;
        a.win_ref = cone ? cone_ref_window_bits(g, pa, pb, cphi, sphi, sdz) : 3;
        const double rvol = 0.5 * sqrt((double)g->nx * g->nx + (double)g->ny * g->ny) + 1.0;
        if (!(pa != 0.0 && pb != 0.0) || !(g->SO > rvol)) {
            plan_free_arrays(p);
            delete p;
            return fl_fail(FL_ERR_INVALID, "source must lie outside the volume (SO=%g voxel units, volume "
                                           "radius %g) and detector pitches must be non-zero",
                           (double)g->SO, rvol);
        }
    }
    if (!cone) {
        std::vector<FanView> fv(idY.size(), FanView{1.0f, 0.0f, 1.0f, 0.0f, 0, 0});   // entries past Nv stay unread
        for (int it = 0; it < g->nt; it++)
            for (int j = 0; j < Nv[it]; j++) {
                const size_t k = (size_t)it * tmp + j;
                const int v = idY[k];
                fv[k] = FanView{cphi[v], sphi[v], cs[v], sn[v], v, idS[k]};
            }
        if ((rc = upload(&p->d_fan_views, fv.data(), fv.size(), "view list"))) {
            plan_free_arrays(p);
            delete p;
            return rc;
        }
        a.fan_views = p->d_fan_views;
        a.fan_cells = fan_shadow_cells(g, g->na > 1 ? ((double)g->y_det[g->na - 1] - g->y_det[0]) / (g->na - 1)
                                                    : (double)g->dy_det,
                                       p->det_dev, cphi, sphi, cs, sn, cdet, sdet, a);
        // the fan adjoint's lines and their quotients, built once on the device
        hipError_t e = hipMalloc((void**)&p->d_line_q, (size_t)g->nv * g->na * sizeof(float4));
        if (e == hipSuccess) e = hipMalloc((void**)&p->d_line_d, (size_t)g->na * sizeof(float));
        if (e == hipSuccess) e = hipMalloc((void**)&p->d_ray_q, (size_t)g->nv * g->na * sizeof(float4));
        if (e == hipSuccess) e = hipMalloc((void**)&p->d_ray_l, (size_t)g->nv * g->na * sizeof(float));
        if (e == hipSuccess) e = fl_launch_fan_line_q(p->ag, g->nv, p->d_line_q, p->d_line_d, nullptr);
        if (e == hipSuccess) e = fl_launch_fan_ray_q(p->fg, g->nv, p->d_ray_q, p->d_ray_l, nullptr);
        if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
        if (e != hipSuccess) {
            plan_free_arrays(p);
            delete p;
            return fl_hip_fail(e, "fan line quotients");
        }
        a.line_q = p->d_line_q;
        a.line_d = p->d_line_d;
        a.ray_q = p->d_ray_q;
        a.ray_l = p->d_ray_l;
    }
    if (cone && !(g->dy_det > 0 && g->dz_det > 0)) {
        plan_free_arrays(p);
        delete p;
        return fl_fail(FL_ERR_INVALID, "dy_det and dz_det must be positive");
    }
    if (!cone && !(g->dy_det > 0)) {
        plan_free_arrays(p);
        delete p;
        return fl_fail(FL_ERR_INVALID, "dy_det must be positive");
    }
    *out = p;
    return fl_ok();
}

// Frees a plan without touching this thread's error status (the drop-in
// entry points release their plans on every path, failed ones included).
static void plan_release(fl_plan_s* p)
{
    if (!p) return;
    fl_plan_release_workspace(p);
    fl_plan_release_f64(p);
    plan_free_arrays(p);
    delete p;
}

extern "C" int fl_plan_destroy(fl_plan p)
{
    plan_release(p);
    return fl_ok();
}

extern "C" int fl_plan_sizes(fl_plan p, long long* nvox, int* nt, long long* ndet, int* nv)
{
    if (!p) return fl_fail(FL_ERR_INVALID, "null plan");
    if (nvox) *nvox = p->nvox;
    if (nt) *nt = p->nt;
    if (ndet) *ndet = p->ndet;
    if (nv) *nv = p->nv;
    return fl_ok();
}

static bool dtype_ok(int t) { return t == FL_F32 || t == FL_BF16 || t == FL_F16; }

// Times every cone-forward ray-tile shape on this plan's geometry (zero
// volume, FP32; the traversal does not depend on the values) and keeps the
// fastest.  Fan plans have one shape.
extern "C" int fl_plan_autotune(fl_plan p, int* fwd_tile, float* fwd_ms)
{
    if (!p) return fl_fail(FL_ERR_INVALID, "null plan");
    if (!p->cone) {
        if (fwd_tile) *fwd_tile = 0;
        if (fwd_ms) *fwd_ms = 0.0f;
        return fl_ok();
    }
    const size_t nxb = (size_t)p->nvox * p->nt * sizeof(float), nyb = (size_t)p->ndet * p->nv * sizeof(float);
    float *x = nullptr, *y = nullptr;
    hipStream_t st = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    // the timed forwards use the plan's brick buffer: after any forward in
    // flight, and none may start meanwhile
    std::lock_guard<std::mutex> lk(p->fwd_mu);
    int rc = FL_OK;
    if (hipMalloc((void**)&x, nxb) != hipSuccess || hipMalloc((void**)&y, nyb) != hipSuccess)
        rc = fl_fail(FL_ERR_ALLOC, "autotune buffers (%zu + %zu bytes)", nxb, nyb);
    if (!rc && (hipStreamCreate(&st) != hipSuccess || hipEventCreate(&e0) != hipSuccess ||
                hipEventCreate(&e1) != hipSuccess))
        rc = fl_fail(FL_ERR_HIP, "autotune stream/events");
    if (!rc && p->fwd_pending && hipStreamWaitEvent(st, p->fwd_done, 0) != hipSuccess)
        rc = fl_fail(FL_ERR_HIP, "autotune ordering");
    int best = p->fg.tile;
    float best_ms = 1e30f;
    if (!rc) {
        hipError_t e = hipMemsetAsync(x, 0, nxb, st);
        FwdGeom g = p->fg;
        for (int t = 0; t < FL_FWD_NTILES && e == hipSuccess; t++) {
            g.tile = t;
            e = fl_launch_fwd_cone(x, FL_F32, y, FL_F32, g, st);
            if (e == hipSuccess) e = hipEventRecord(e0, st);
            if (e == hipSuccess) e = fl_launch_fwd_cone(x, FL_F32, y, FL_F32, g, st);
            if (e == hipSuccess) e = hipEventRecord(e1, st);
            if (e == hipSuccess) e = hipEventSynchronize(e1);
            float ms = 0.0f;
            if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
            if (e == hipSuccess && ms < best_ms) {
                best_ms = ms;
                best = t;
            }
        }
        if (e != hipSuccess) rc = fl_hip_fail(e, "autotune forward");
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (st) (void)hipStreamDestroy(st);
    if (x) (void)hipFree(x);
    if (y) (void)hipFree(y);
    if (rc) return rc;
    p->fg.tile = best;
    if (fwd_tile) *fwd_tile = best;
    if (fwd_ms) *fwd_ms = best_ms;
    return fl_ok();
}

// Selects a cone-forward ray-tile shape by index (0..FL_FWD_NTILES-1).
extern "C" int fl_plan_set_tile(fl_plan p, int tile)
{
    if (!p || tile < 0 || tile >= FL_FWD_NTILES) return fl_fail(FL_ERR_INVALID, "bad plan or tile %d", tile);
    std::lock_guard<std::mutex> lk(p->fwd_mu);
    p->fg.tile = tile;
    return fl_ok();
}

int fl_forward_ordered(fl_plan_s* p, const void* d_x, int xt, void* d_y, int yt, void* stream, bool owns_capture)
{
    if (!p || !d_x || !d_y) return fl_fail(FL_ERR_INVALID, "null plan or buffer");
    if (!dtype_ok(xt) || !dtype_ok(yt)) return fl_fail(FL_ERR_INVALID, "bad dtype");
    hipStream_t st = (hipStream_t)stream;
    auto launch = [&](const FwdGeom& g) {
        const hipError_t e = p->cone ? fl_launch_fwd_cone(d_x, xt, d_y, yt, g, st) : fl_launch_fwd_fan(d_x, xt, d_y, yt, g, st);
        if (e == hipErrorInvalidValue) return fl_fail(FL_ERR_UNSUPPORTED, "dtype combination %d/%d", xt, yt);
        return e == hipSuccess ? FL_OK : fl_hip_fail(e, "forward launch");
    };
    auto as_it_is = [&] {
        FwdGeom g = p->fg;
        g.tracked = false;
        const int rc = launch(g);
        return rc ? rc : fl_ok();
    };
    // a fan forward captured by someone else replays in no order with the
    // plan's other forwards: it reads its image as it is
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (!p->cone && p->d_bricks && !owns_capture && hipStreamIsCapturing(st, &cs) != hipSuccess) cs = hipStreamCaptureStatusActive;
    if (!p->d_bricks || cs != hipStreamCaptureStatusNone) return as_it_is();
    std::lock_guard<std::mutex> lk(p->fwd_mu);
    if (!owns_capture && fl_bricks_busy(p, st)) return as_it_is();
    bool order = false;
    int rc = fwd_order_begin(p, st, order);
    if (!rc) rc = launch(p->fg);
    if (!rc) rc = fwd_order_end(p, st, order);
    return rc ? rc : fl_ok();
}

extern "C" int fl_forward(fl_plan p, const void* d_x, int xt, void* d_y, int yt, void* stream)
{
    return fl_forward_ordered(p, d_x, xt, d_y, yt, stream, false);
}

extern "C" int fl_forward_gao_fan(fl_plan p, const void* d_x, int xt, void* d_y, int yt, void* stream)
{
    if (!p || !d_x || !d_y) return fl_fail(FL_ERR_INVALID, "null plan or buffer");
    if (p->cone) return fl_fail(FL_ERR_INVALID, "Gao column walk is the fan forward");
    hipError_t e = fl_launch_fwd_fan_gao(d_x, xt, d_y, yt, p->fg, (hipStream_t)stream);
    if (e == hipErrorInvalidValue) return fl_fail(FL_ERR_UNSUPPORTED, "dtype combination %d/%d", xt, yt);
    if (e != hipSuccess) return fl_hip_fail(e, "forward launch");
    return fl_ok();
}

// Strip lines of the finite-width fan forward per (view, cell, edge), with
// the reference's float trig (Ax_fan_mf_cpu_new_fb.cpp:38-47): edge
// u = y_det -+ dy_det/2, angle atan2f(u, SD), Px = -sinf(angle + phi),
// Py = cosf(angle + phi), Pd = SO*sinf(angle).
static int ensure_fb_tables(fl_plan_s* p)
{
    std::lock_guard<std::mutex> lk(p->fwd_mu);
    if (p->d_fb_px && p->d_fb_py && p->d_fb_pd) return FL_OK;
    const int nv = p->nv, nd = (int)p->ndet;
    const float SO = p->fg.SO, SD = p->fg.SO + p->fg.OD, dy = p->ag.dy_det;
    std::vector<float> px((size_t)nv * nd * 2), py((size_t)nv * nd * 2), pd((size_t)nd * 2);
    for (int id = 0; id < nd; id++)
        for (int e = 0; e < 2; e++) {
            const float u = e == 0 ? p->h_ydet[id] - dy / 2 : p->h_ydet[id] + dy / 2;
            const float ang = atan2f(u, SD);
            pd[(size_t)id * 2 + e] = SO * sinf(ang);
            for (int iv = 0; iv < nv; iv++) {
                const float a = ang + p->h_sd_phi[iv];
                px[((size_t)iv * nd + id) * 2 + e] = -sinf(a);
                py[((size_t)iv * nd + id) * 2 + e] = cosf(a);
            }
        }
    int rc;
    if ((rc = upload(&p->d_fb_px, px.data(), px.size(), "strip Px")) ||
        (rc = upload(&p->d_fb_py, py.data(), py.size(), "strip Py")) ||
        (rc = upload(&p->d_fb_pd, pd.data(), pd.size(), "strip Pd"))) {
        // leave no partial set behind: the next call builds all three again
        for (float** q : {&p->d_fb_px, &p->d_fb_py, &p->d_fb_pd}) {
            if (*q) (void)hipFree(*q);
            *q = nullptr;
        }
        return rc;
    }
    return FL_OK;
}

extern "C" int fl_forward_norm(fl_plan p, const float* d_y, float* d_yn, void* stream)
{
    if (!p || !d_y || !d_yn) return fl_fail(FL_ERR_INVALID, "null plan or buffer");
    if (!p->cone) return fl_fail(FL_ERR_INVALID, "the normalised sinogram is a cone output");
    hipError_t e = fl_launch_ynorm(d_y, d_yn, p->fg, (hipStream_t)stream);
    if (e != hipSuccess) return fl_hip_fail(e, "yNorm launch");
    return fl_ok();
}

extern "C" int fl_forward_fan_fb(fl_plan p, const float* d_x, float* d_y, void* stream)
{
    if (!p || !d_x || !d_y) return fl_fail(FL_ERR_INVALID, "null plan or buffer");
    if (p->cone) return fl_fail(FL_ERR_INVALID, "the finite-width beam is a fan projector");
    int rc = ensure_fb_tables(p);
    if (rc) return rc;
    hipError_t e = fl_launch_fwd_fan_fb(d_x, d_y, p, (hipStream_t)stream);
    if (e != hipSuccess) return fl_hip_fail(e, "finite-beam forward launch");
    return fl_ok();
}

extern "C" int fl_adjoint(fl_plan p, const void* d_y, int yt, void* d_x, int xt, int kind, void* stream)
{
    if (!p || !d_x || !d_y) return fl_fail(FL_ERR_INVALID, "null plan or buffer");
    if (!dtype_ok(xt) || !dtype_ok(yt)) return fl_fail(FL_ERR_INVALID, "bad dtype");
    if (!p->slots_ok)
        return fl_fail(FL_ERR_UNSUPPORTED, "a frame lists a view more often than the forward's output slots "
                                           "hold it (slot_view), so the adjoint has no slot to read");
    if (p->det_dev > FL_DET_DEV_MAX)
        return fl_fail(FL_ERR_UNSUPPORTED,
                       "detector coordinates stray %.3g cells from a uniform grid; the voxel-driven adjoints "
                       "need uniform spacing (the forward does not)", p->det_dev);
    hipStream_t st = (hipStream_t)stream;
    hipError_t e;
    if (kind == FL_ADJ_EXACT) {
        e = p->cone ? fl_launch_adj_cone(d_y, yt, d_x, xt, p->ag, st)
                    : fl_launch_adj_fan(d_y, yt, d_x, xt, p->fg, p->ag, st);
    } else if (kind == FL_ADJ_MATCHED) {
        e = fl_launch_adj_matched(d_y, yt, d_x, xt, p, st);
    } else if (kind == FL_ADJ_FAN_FB) {
        if (p->cone) return fl_fail(FL_ERR_INVALID, "the finite-width beam is a fan projector");
        if (!p->d_cdet2) return fl_fail(FL_ERR_INVALID, "plan has no cos_det2/sin_det2 edge tables");
        if (yt != FL_F32 || xt != FL_F32) return fl_fail(FL_ERR_UNSUPPORTED, "finite-width beam is FP32");
        e = fl_launch_adj_fan_fb((const float*)d_y, (float*)d_x, p, st);
    } else {
        return fl_fail(FL_ERR_INVALID, "unknown adjoint kind %d", kind);
    }
    if (e == hipErrorInvalidValue) return fl_fail(FL_ERR_UNSUPPORTED, "dtype combination %d/%d", yt, xt);
    if (e != hipSuccess) return fl_hip_fail(e, "adjoint launch");
    return fl_ok();
}

extern "C" int fl_siddon_trace(fl_plan p, int nrays, const int* rays, int cap, int* J, float* S, int* cnt)
{
    if (!p || nrays < 0 || cap < 0 || (nrays > 0 && (!rays || !J || !S || !cnt)))
        return fl_fail(FL_ERR_INVALID, "bad trace arguments");
    for (int k = 0; k < nrays; k++) {
        int v = rays[3 * k], a = rays[3 * k + 1], b = rays[3 * k + 2];
        if (v < 0 || v >= p->nv || a < 0 || a >= p->fg.na || b < 0 || b >= p->fg.nb)
            return fl_fail(FL_ERR_INVALID, "ray %d out of range", k);
    }
    if (nrays == 0) return fl_ok();
    std::vector<int> off(nrays), caps(nrays, cap);
    for (int k = 0; k < nrays; k++) off[k] = k * cap;
    int *d_rays = nullptr, *d_off = nullptr, *d_cap = nullptr, *d_J = nullptr, *d_cnt = nullptr;
    float* d_S = nullptr;
    int rc = FL_OK;
    size_t tot = (size_t)nrays * cap;
    hipError_t e;
    if ((rc = upload(&d_rays, rays, (size_t)nrays * 3, "rays")) || (rc = upload(&d_off, off.data(), off.size(), "off")) ||
        (rc = upload(&d_cap, caps.data(), caps.size(), "cap")))
        goto done;
    if ((e = hipMalloc((void**)&d_J, (tot ? tot : 1) * sizeof(int))) != hipSuccess ||
        (e = hipMalloc((void**)&d_S, (tot ? tot : 1) * sizeof(float))) != hipSuccess ||
        (e = hipMalloc((void**)&d_cnt, nrays * sizeof(int))) != hipSuccess) {
        rc = fl_fail(FL_ERR_ALLOC, "trace buffers");
        goto done;
    }
    e = fl_launch_trace(p->fg, p->cone ? 1 : 0, nrays, d_rays, d_off, d_cap, d_J, d_S, d_cnt, 0);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess && tot) e = hipMemcpy(J, d_J, tot * sizeof(int), hipMemcpyDeviceToHost);
    if (e == hipSuccess && tot) e = hipMemcpy(S, d_S, tot * sizeof(float), hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(cnt, d_cnt, nrays * sizeof(int), hipMemcpyDeviceToHost);
    if (e != hipSuccess) rc = fl_hip_fail(e, "trace");
done:
    for (void* q : {(void*)d_rays, (void*)d_off, (void*)d_cap, (void*)d_J, (void*)d_S, (void*)d_cnt})
        if (q) (void)hipFree(q);
    return rc ? rc : fl_ok();
}

// ------------------------------------------------ drop-in entry points ----
//
// Host pointers, synchronous, like the reference wrappers: allocate device
// buffers, copy in, run on the null stream, copy out, free.  Status through
// fl_get_last_error().

namespace {

struct DevBuf {
    void* p = nullptr;
    ~DevBuf()
    {
        if (p) (void)hipFree(p);
    }
    int alloc(size_t bytes, const char* what)
    {
        hipError_t e = hipMalloc(&p, bytes ? bytes : 4);
        return e == hipSuccess ? FL_OK : fl_fail(FL_ERR_ALLOC, "hipMalloc(%s, %zu bytes)", what, bytes);
    }
};

struct PlanGuard {
    fl_plan p = nullptr;
    ~PlanGuard() { plan_release(p); }
};

// Frame -> view lists to view -> frame and output slot order.
void frames_to_views(int nt, int nv, const int* id_Y, const int* Nv, int tmp, std::vector<int>& id_X,
                     std::vector<int>& slots)
{
    id_X.assign(nv, 0);
    slots.clear();
    for (int it = 0; it < nt; it++)
        for (int j = 0; j < Nv[it]; j++) {
            int v = id_Y[(size_t)it * tmp + j];
            if (v >= 0 && v < nv) id_X[v] = it;
            slots.push_back(v);
        }
}

int run_forward_host(const fl_geometry& g, const float* X, float* y, float* yNorm, bool gao, bool fb = false)
{
    PlanGuard pg;
    int rc = fl_plan_create_with(&pg.p, &g, !gao && !fb);
    if (rc) return rc;
    size_t nvox = (size_t)pg.p->nvox * g.nt, ny = (size_t)pg.p->ndet * g.nv;
    DevBuf dx, dy, dn;
    if ((rc = dx.alloc(nvox * 4, "X")) || (rc = dy.alloc(ny * 4, "y"))) return rc;
    hipError_t e = hipMemcpy(dx.p, X, nvox * 4, hipMemcpyHostToDevice);
    if (e != hipSuccess) return fl_hip_fail(e, "copy X");
    rc = fb    ? fl_forward_fan_fb(pg.p, (const float*)dx.p, (float*)dy.p, nullptr)
         : gao ? fl_forward_gao_fan(pg.p, dx.p, FL_F32, dy.p, FL_F32, nullptr)
               : fl_forward(pg.p, dx.p, FL_F32, dy.p, FL_F32, nullptr);
    if (rc) return rc;
    if (yNorm) {
        if ((rc = dn.alloc(ny * 4, "yNorm"))) return rc;
        e = fl_launch_ynorm((const float*)dy.p, (float*)dn.p, pg.p->fg, nullptr);
        if (e != hipSuccess) return fl_hip_fail(e, "yNorm");
    }
    e = hipMemcpy(y, dy.p, ny * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess && yNorm) e = hipMemcpy(yNorm, dn.p, ny * 4, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return fl_hip_fail(e, "copy y");
    return fl_ok();
}

int run_adjoint_host(const fl_geometry& g, const float* Y, float* X, int kind = FL_ADJ_EXACT)
{
    PlanGuard pg;
    int rc = fl_plan_create_with(&pg.p, &g, false);
    if (rc) return rc;
    size_t nvox = (size_t)pg.p->nvox * g.nt, ny = (size_t)pg.p->ndet * g.nv;
    DevBuf dx, dy;
    if ((rc = dx.alloc(nvox * 4, "X")) || (rc = dy.alloc(ny * 4, "y"))) return rc;
    hipError_t e = hipMemcpy(dy.p, Y, ny * 4, hipMemcpyHostToDevice);
    if (e != hipSuccess) return fl_hip_fail(e, "copy y");
    if ((rc = fl_adjoint(pg.p, dy.p, FL_F32, dx.p, FL_F32, kind, nullptr))) return rc;
    e = hipMemcpy(X, dx.p, nvox * 4, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return fl_hip_fail(e, "copy X");
    return fl_ok();
}

}  // namespace

extern "C" void Ax_fan_mf_gpu_siddon(float* X, float* y, float SO, float OD, float scale, int nx, int ny,
                                     int nv, float* sd_phi, int nd, float* y_det, int* id_X, int nt)
{
    fl_geometry g = {};
    g.nx = nx; g.ny = ny; g.nz = 0; g.nt = nt; g.nv = nv; g.na = nd; g.nb = 1;
    g.SO = SO; g.OD = OD; g.scale = scale; g.dy_det = 1.0f;
    g.sd_phi = sd_phi; g.y_det = y_det; g.id_X = id_X;
    run_forward_host(g, X, y, nullptr, false);
}

extern "C" void Ax_fan_mf_gpu_new(float* X, float* y, float SO, float OD, float scale, int nx, int ny,
                                  int nv, float* sd_phi, int nd, float* y_det, int* id_X, int nt)
{
    fl_geometry g = {};
    g.nx = nx; g.ny = ny; g.nz = 0; g.nt = nt; g.nv = nv; g.na = nd; g.nb = 1;
    g.SO = SO; g.OD = OD; g.scale = scale; g.dy_det = 1.0f;
    g.sd_phi = sd_phi; g.y_det = y_det; g.id_X = id_X;
    run_forward_host(g, X, y, nullptr, true);
}

extern "C" void Atx_fan_mf_gpu_new(float* x, float* Y, float SO, float OD, float scale, int nx, int ny,
                                   float* sd_phi, int nd, float* y_det, float dy_det, float y_os, int nt,
                                   int* id_Y, int* Nv, int tmp_size, int nv, float* cos_phi,
                                   float* sin_phi, float* cos_det, float* sin_det)
{
    fl_geometry g = {};
    g.nx = nx; g.ny = ny; g.nz = 0; g.nt = nt; g.nv = nv; g.na = nd; g.nb = 1;
    g.SO = SO; g.OD = OD; g.scale = scale; g.dy_det = dy_det; g.y_os = y_os;
    g.sd_phi = sd_phi; g.y_det = y_det; g.cos_phi = cos_phi; g.sin_phi = sin_phi;
    g.cos_det = cos_det; g.sin_det = sin_det; g.id_Y = id_Y; g.Nv = Nv; g.tmp_size = tmp_size;
    std::vector<int> idX, slots;
    if (id_Y && Nv) {
        frames_to_views(nt, nv, id_Y, Nv, tmp_size, idX, slots);
        g.id_X = idX.data();
    }
    run_adjoint_host(g, Y, x);
}

extern "C" void Ax_fan_mf_gpu_new_fb(float* X, float* y, float SO, float OD, float scale, int nx, int ny,
                                     int nv, float* sd_phi, int nd, float* y_det, int* id_X, int nt,
                                     float dy_det)
{
    fl_geometry g = {};
    g.nx = nx; g.ny = ny; g.nz = 0; g.nt = nt; g.nv = nv; g.na = nd; g.nb = 1;
    g.SO = SO; g.OD = OD; g.scale = scale; g.dy_det = dy_det;
    g.sd_phi = sd_phi; g.y_det = y_det; g.id_X = id_X;
    run_forward_host(g, X, y, nullptr, false, true);
}

extern "C" void Atx_fan_mf_gpu_new_fb(float* x, float* Y, float SO, float OD, float scale, int nx, int ny,
                                      float* sd_phi, int nd, float* y_det, float dy_det, int nt, int* id_Y,
                                      int* Nv, int tmp_size, int nv, float* cos_phi, float* sin_phi,
                                      float* cos_det, float* sin_det)
{
    fl_geometry g = {};
    g.nx = nx; g.ny = ny; g.nz = 0; g.nt = nt; g.nv = nv; g.na = nd; g.nb = 1;
    g.SO = SO; g.OD = OD; g.scale = scale; g.dy_det = dy_det;
    g.sd_phi = sd_phi; g.y_det = y_det; g.cos_phi = cos_phi; g.sin_phi = sin_phi;
    g.cos_det2 = cos_det; g.sin_det2 = sin_det; g.id_Y = id_Y; g.Nv = Nv; g.tmp_size = tmp_size;
    std::vector<int> idX, slots;
    if (id_Y && Nv) {
        frames_to_views(nt, nv, id_Y, Nv, tmp_size, idX, slots);
        g.id_X = idX.data();
    }
    run_adjoint_host(g, Y, x, FL_ADJ_FAN_FB);
}

static void cone_fwd_dropin(float* X, float* y, float* yNorm, float* sd_phi, float* sd_z, float* y_det,
                            float* z_det, int* id_Y, int* Nv, float SO, float OD, float scale, float dz,
                            int nx, int ny, int nz, int nt, int na, int nb, int nv, int tmp_size)
{
    fl_geometry g = {};
    g.nx = nx; g.ny = ny; g.nz = nz; g.nt = nt; g.nv = nv; g.na = na; g.nb = nb;
    g.SO = SO; g.OD = OD; g.scale = scale; g.dz = dz; g.dy_det = 1.0f; g.dz_det = 1.0f;
    g.sd_phi = sd_phi; g.sd_z = sd_z; g.y_det = y_det; g.z_det = z_det;
    std::vector<int> idX, slots;
    if (id_Y && Nv) {
        frames_to_views(nt, nv, id_Y, Nv, tmp_size, idX, slots);
        if ((int)slots.size() != nv) {
            fl_fail(FL_ERR_INVALID, "id_Y/Nv list %zu views, expected nv=%d", slots.size(), nv);
            return;
        }
        g.id_X = idX.data();
        g.slot_view = slots.data();
        g.id_Y = id_Y; g.Nv = Nv; g.tmp_size = tmp_size;
    }
    run_forward_host(g, X, y, yNorm, false);
}

extern "C" void Ax_cone_mf_gpu_siddon(float* X, float* y, float* sd_phi, float* sd_z, float* y_det,
                                      float* z_det, int* id_Y, int* Nv, float SO, float OD, float scale,
                                      float dz, int nx, int ny, int nz, int nt, int na, int nb, int nv,
                                      int tmp_size, int nv_block)
{
    (void)nv_block;  // views are not chunked: one launch covers all of them
    cone_fwd_dropin(X, y, nullptr, sd_phi, sd_z, y_det, z_det, id_Y, Nv, SO, OD, scale, dz, nx, ny, nz, nt,
                    na, nb, nv, tmp_size);
}

extern "C" void Ax_cone_mf_gpu_new(float* X, float* y, float* yNorm, float* sd_phi, float* sd_z,
                                   float* y_det, float* z_det, int* id_Y, int* Nv, float SO, float OD,
                                   float scale, float dz, int nx, int ny, int nz, int nt, int na, int nb,
                                   int nv, int tmp_size, int nv_block)
{
    (void)nv_block;
    cone_fwd_dropin(X, y, yNorm, sd_phi, sd_z, y_det, z_det, id_Y, Nv, SO, OD, scale, dz, nx, ny, nz, nt,
                    na, nb, nv, tmp_size);
}

extern "C" void Atx_cone_mf_gpu_new(float* X, float* y, float* cos_phi, float* sin_phi, float* sd_z,
                                    float* y_det, float* z_det, int* id_Y, int* Nv, float SO, float OD,
                                    float scale, float dy_det, float y_os, float dz_det, float dz, int nx,
                                    int ny, int nz, int nt, int na, int nb, int nv, int tmp_size,
                                    int nv_block)
{
    (void)nv_block;
    // the adjoint needs no angles beyond the cos/sin tables; sd_phi is only
    // a required plan field, so it is reconstructed from them
    std::vector<float> phi(nv > 0 ? nv : 1);
    for (int v = 0; v < nv; v++) phi[v] = (float)atan2((double)sin_phi[v], (double)cos_phi[v]);
    fl_geometry g = {};
    g.nx = nx; g.ny = ny; g.nz = nz; g.nt = nt; g.nv = nv; g.na = na; g.nb = nb;
    g.SO = SO; g.OD = OD; g.scale = scale; g.dz = dz; g.dy_det = dy_det; g.dz_det = dz_det; g.y_os = y_os;
    g.sd_phi = phi.data(); g.sd_z = sd_z; g.y_det = y_det; g.z_det = z_det;
    g.cos_phi = cos_phi; g.sin_phi = sin_phi; g.id_Y = id_Y; g.Nv = Nv; g.tmp_size = tmp_size;
    std::vector<int> idX, slots;
    if (id_Y && Nv) {
        // the reference wrapper reads y in frame-list order (slot id holds
        // the id-th listed view, Atx_cone_mf_gpu_new.cu:140-150), the order
        // the cone forward drop-ins write
        frames_to_views(nt, nv, id_Y, Nv, tmp_size, idX, slots);
        if ((int)slots.size() != nv) {
            fl_fail(FL_ERR_INVALID, "id_Y/Nv list %zu views, expected nv=%d", slots.size(), nv);
            return;
        }
        g.id_X = idX.data();
        g.slot_view = slots.data();
    }
    run_adjoint_host(g, y, X);
}
