// Geometric multigrid preconditioner (multigrid/*.f90 of the reference, with a zebra z-line smoother):
// hierarchy set-up and the preconditioner entry with its hipGraph replay.  The per-precision work is in
// ow3d_mg64.hip / ow3d_mg32.hip.
#include "ow3d_internal.hpp"

namespace ow3d_host {

namespace {
bool plane_coarsened(const Grid &f, const Grid &c) { return c.xc && c.yc && !c.zc && f.ny > 1; }   // MgLevel::ptab
}  // namespace

bool needs_b(const ow3d_tank *t, int k) {
    const int top = (int)t->levels.size() - 1;
    return !(k == top && top >= 1 && t->cfg.mg_precision == 0 && t->fused_rb && t->cfg.nu1 >= 1);
}
bool needs_r(const ow3d_tank *t, int k) {
    return k > t->bot_top && k > 0 && !plane_coarsened(t->levels[k], t->levels[k - 1]);
}

namespace {
constexpr size_t BOTTOM_DENSE = 512 << 10;
// One compute unit reads about 60-100 GB/s: an inverse of more than BOTTOM_DENSE bytes is read by all of them.
bool bottom_split(const ow3d_tank *t) {
    const size_t n = t->levels[0].n, p = t->cfg.mg_precision == 0 ? 8 : t->cfg.mg_precision == 2 ? 2 : 4;
    return n * n * p > BOTTOM_DENSE;
}
// Finest level of the group that the one-workgroup kernel takes (-1: none): levels below the finest with one column of a
// colour per thread and all vectors in the workgroup's LDS.  Measured per V cycle, one launch per step and one workgroup:
// 33^2 x 10 FP64 (17^2, 9^2, 5^2 and the dense level) 84 us and 13 launches more, 53 us; x-z 257 x 10 FP64 (six levels)
// 150 us and 27 launches more, 67 us; 97 x 161 x 9 FP32 (three levels, dense solve apart) 60 us and 8 launches more,
// 51 us.  Around a dense solve of its own a single level gains nothing (193 x 129 x 10 FP32: 321 us and 331 us the cycle).
int bottom_top(const ow3d_tank *t) {
    const size_t p = t->cfg.mg_precision == 0 ? 8 : 4;
    if (!t->fused_rb || t->cfg.nu1 < 1 || t->cfg.nu2 < 1) return -1;
    int top = -1;
    for (int k = 1; k < (int)t->levels.size() - 1 && k < MG_BOTTOM_MAX; k++) {
        const Grid &g = t->levels[k];
        if ((long)g.n > t->bot_lim || !has_records(g) || (g.ny > 1) != (t->levels[0].ny > 1) || !bottom_fits(g.nxg, g.nyg, g.ny > 1)) break;
        const int zh = g.nzg % 2 ? g.nzg : (g.nzg - 2) / 2 + 2, zc = t->levels[k - 1].nzg;   // the depths the kernel has steps for
        if (zc != g.nzg && zc != zh) break;
        if (bottom_layout<double>(t->levels, k, nullptr) * p > BOTTOM_LDS) break;
        top = k;
    }
    return top < 2 && bottom_split(t) ? -1 : top;
}
}  // namespace

void mg_choices(ow3d_tank *t) {
    if (const char *e = std::getenv("OW3D_MG_BOTTOM")) t->bot_lim = std::atol(e);
    if (const char *e = std::getenv("OW3D_MG_FUSED_RB")) t->fused_rb = e[0] != '0';
    t->bot_top = bottom_top(t);
    t->bot_split = bottom_split(t);
}

// Multigrid hierarchy of the tank (MGPreProcess.f90:6-460 with coarsening strategy 0), level operators in
// the precision the configuration asks for, and the levels handed to the one-workgroup kernel.
int mg_setup(ow3d_tank *t) {
    const ow3d_config &c = t->cfg;
    if (!mg_levels(t->g, c.mg_maxgrids, t->levels, err())) return -1;
    t->nlev = (int)t->levels.size();
    for (auto &L : t->levels)
        if (L.nzg < 3 || L.nzg > 14) { err() = "multigrid level depth outside 3..14"; return -1; }
    if (t->levels[0].n > 4096) { err() = "coarsest multigrid level too large for the dense solve"; return -1; }
    mg_choices(t);
    if (c.mg_precision == 0 ? mg_build64(t) : mg_build32(t)) return -1;
    return c.mg_precision == 0 ? mg_fill_bottom64(t) : mg_fill_bottom32(t);
}

// u = M^-1 r (device vectors, FP64 in / out), skipped once the solve's done flag is set.  When r is the
// handle's residual buffer the V cycle is replayed from a hipGraph captured on first use (one graph per
// handle; fixed buffers), unless a whole RK4 step is being captured (its graph then holds the V cycle).
int precond(ow3d_tank *t, const double *r, double *u, hipStream_t s) {
    const size_t n = t->g.n;
    if (t->cfg.precond != 3) {
        hipLaunchKernelGGL((k_convert<double, double>), dim3(grid_blocks(n)), dim3(256), 0, s, n, r, u, t->done());
        return 0;
    }
    if (t->use_graph && !t->capturing && r == t->w.p && s == t->s) {
        if (!t->pg_exec) {
            std::lock_guard<std::mutex> lk(capture_lock());
            hipGraph_t graph = nullptr;
            HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
            int rc = (t->cfg.mg_precision == 0 ? precond_body64(t, r, &t->mg_out, s, nullptr)
                                               : precond_body32(t, r, &t->mg_out, s, nullptr));
            hipError_t e = hipStreamEndCapture(s, &graph);
            if (rc) { if (graph) (void)hipGraphDestroy(graph); return -1; }
            HIPCHK(e);
            HIPCHK(hipGraphInstantiate(&t->pg_exec, graph, nullptr, nullptr, 0));
            (void)hipGraphDestroy(graph);
        }
        HIPCHK(hipGraphLaunch(t->pg_exec, s));
    } else {
        // inline (eager, or inside a captured step): the last sweep writes u itself
        const void *o = nullptr;
        if ((t->cfg.mg_precision == 0 ? precond_body64(t, r, &o, s, u) : precond_body32(t, r, &o, s, u))) return -1;
        if (!o) return 0;
        t->mg_out = o;
    }
    if (t->cfg.mg_precision == 0)
        hipLaunchKernelGGL((k_convert<double, double>), dim3(grid_blocks(n)), dim3(256), 0, s, n, (const double *)t->mg_out, u, t->done());
    else
        hipLaunchKernelGGL((k_convert<float, double>), dim3(grid_blocks(n)), dim3(256), 0, s, n, (const float *)t->mg_out, u, t->done());
    return 0;
}


}  // namespace ow3d_host
