// C ABI of libfcpt_hip.so (include/fcpt.h): context management, state
// transfer and one entry point per reference hydro-step function.  All device
// work of a context is enqueued on the context's own HIP stream (default
// priority); functions that hand a value back to the host synchronise it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "fcpt_device.hpp"
#include "fcpt_kernels.hpp"

using namespace fcpt;

// Iterations in one captured graph.  A graph's start and end cost the device
// 3 to 5 us beyond the kernels between them (32 x 64: 37.1 us per step with one
// iteration per graph, 33.1 with 4, 32.2 with 16; 251 x 757: 60.3, 57.6, 56.3).
// Capture and first use of the longer graph cost a context's first call of 8 steps
// 36 to 51 us more than those of a single iteration's (32 x 64: 292 and 256 us; 12
// steps 392 and 361, 16 and more no more), which its second call has back (195 and
// 234).
constexpr int kGraphSteps = 8;

// split storage: steps of fcpt_run_steps between two moves of the ring
// backgrounds unless the caller sets another interval
constexpr int kDefaultRebaseInterval = 1000;

struct fcpt_ctx {
    fcpt_disk_desc desc{};
    KParams P{};
    hipStream_t stream = nullptr;
    int device = 0;
    std::vector<void *> allocs;
    bool fused = true;  // fused step kernels (FCPT_PARAM_FUSED_STEP)
    DevScalars *s_dev = nullptr;
    DevScalars *s_host = nullptr;  // pinned mirror for read-back
    double *totals_ring = nullptr;
    double *totals_out = nullptr;
    double *totals_host = nullptr;
    double *force_part = nullptr;  // the disk force's partial sums per ring
    double *force_host = nullptr;  // its result (pinned, written by the kernel)
    hipGraphExec_t step_graph[2] = {nullptr, nullptr};  // of one iteration and of kGraphSteps
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::string err;
    // host copies of the per-ring metric (split storage derives its backgrounds from them)
    std::vector<double> Rinf, Rmed, Surf, InvRmed, InvDiffRmed, InvDiffRsup, InvDiffRsupRb;
    // split storage: host copies of the backgrounds last set from the host, and
    // a device ring array for re-expressing a field about a new background
    std::vector<double> hbg[FCPT_NUM_FIELDS];
    double *bg_tmp = nullptr;
    // the last step left derived fields to be formed (its lazy_derived), the scale
    // height among them (its h_lazy)
    bool derived_stale = false, h_stale = false;
    // the derived fields are those of the current E and Sigma (stored or
    // stale); false once a caller has set a field or stage of its own, which
    // the next step then reads as stored
    bool derived_own = true;
    // split storage: steps between background moves (FCPT_PARAM_REBASE_INTERVAL;
    // 0 = only on request) and steps since the last one
    int rebase_interval = 0;
    int steps_since_rebase = 0;
};

static void host_slots_join();
static void host_slots_leave();

// both graphs of a context or a batch, to be captured again
static hipError_t drop_graphs(hipGraphExec_t (&g)[2])
{
    hipError_t e = hipSuccess;
    for (hipGraphExec_t &x : g) {
        if (!x) continue;
        const hipError_t d = hipGraphExecDestroy(x);
        if (e == hipSuccess) e = d;
        x = nullptr;
    }
    return e;
}

namespace {

int fail(fcpt_ctx *c, int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    if (c) c->err = buf;
    return code;
}

#define HIP_TRY(ctx, expr)                                                            \
    do {                                                                              \
        hipError_t e_ = (expr);                                                       \
        if (e_ != hipSuccess)                                                         \
            return fail((ctx), FCPT_ERR_DEVICE, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

#define LAUNCH_CHECK(ctx)                                                             \
    do {                                                                              \
        hipError_t e_ = hipGetLastError();                                            \
        if (e_ != hipSuccess)                                                         \
            return fail((ctx), FCPT_ERR_DEVICE, "kernel launch: %s", hipGetErrorString(e_)); \
    } while (0)

#define CTX_CHECK(ctx)                                   \
    do {                                                 \
        if (!(ctx)) return FCPT_ERR_ARG;                 \
        hipError_t e_ = hipSetDevice((ctx)->device);     \
        if (e_ != hipSuccess)                            \
            return fail((ctx), FCPT_ERR_DEVICE, "hipSetDevice: %s", hipGetErrorString(e_)); \
    } while (0)

// When the fused step runs the kick walk, the derived fields are formed where
// the step needs them and left stale (KParams::lazy_derived) until
// sync_derived stores them (the same expressions on the stored E and Sigma).
// What is stale is the last step's doing, a batch's perhaps, and not a question
// of the parameters in force when the fields are read.
static bool lazy_applies(const fcpt_ctx *ctx) { return ctx->fused && kv_walk_applies(ctx->P); }
// Whether the next step has to read derived fields as the caller left them: it
// then runs the fused step's cell passes, which read them stored, in place of
// the walk (the fused step of an isothermal disk forms its pressure from Sigma
// anyway).  A final boundary call and the step after it, with the separate kernels
// and so: 512x1536 adiabatic 187 and 157 us, 1024x3072 553 and 481.
static bool reads_stored(const fcpt_ctx *ctx)
{
    return !ctx->derived_own && ctx->P.adiabatic && lazy_applies(ctx);
}
// the parameters of a step that forms its derived fields itself, or reads them
static KParams step_view(const fcpt_ctx *ctx, bool stored = false)
{
    KParams P = ctx->P;
    set_step_modes(P, ctx->fused && !stored);
    return P;
}
// after a whole iteration that ran with the parameters V
static void stepped(fcpt_ctx *ctx, const KParams &V)
{
    ctx->derived_stale = V.lazy_derived != 0;
    ctx->h_stale = V.h_lazy != 0;
    ctx->derived_own = true;
}
static int sync_derived(fcpt_ctx *ctx)
{
    if (!ctx->derived_stale) return FCPT_OK;
    KParams P = ctx->P;
    P.step_at = &ctx->s_dev->count_derived;  // rounded as the step would have
    launch_derived(P, ctx->stream);
    LAUNCH_CHECK(ctx);
    ctx->derived_stale = ctx->h_stale = false;
    return FCPT_OK;
}
// before an iteration with the parameters V: the stale fields it reads, stored
static int sync_for(fcpt_ctx *ctx, const KParams &V)
{
    return V.lazy_derived && (V.h_lazy || !ctx->h_stale) ? FCPT_OK : sync_derived(ctx);
}
// the fields sync_derived stores (an isothermal disk: the pressure alone)
static bool derived_field(int f)
{
    return f == FCPT_PRESSURE || f == FCPT_SOUNDSPEED || f == FCPT_SCALE_HEIGHT || f == FCPT_VISCOSITY ||
           f == FCPT_TEMPERATURE;
}
// entry points that read or expose the fields: the context, with the derived
// fields stored
#define CTX_SYNCED(ctx)                        \
    do {                                       \
        CTX_CHECK(ctx);                        \
        const int rc_sync_ = sync_derived(ctx); \
        if (rc_sync_) return rc_sync_;         \
    } while (0)

int dev_alloc_bytes(fcpt_ctx *c, void **p, size_t bytes)
{
    void *q = nullptr;
    hipError_t e = hipMalloc(&q, bytes + 256);
    if (e != hipSuccess)
        return fail(c, FCPT_ERR_DEVICE, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
    c->allocs.push_back(q);
    *p = q;
    return FCPT_OK;
}

template <typename T>
int dev_alloc(fcpt_ctx *c, T **p, size_t count)
{
    void *q = nullptr;
    const int rc = dev_alloc_bytes(c, &q, count * sizeof(T));
    *p = static_cast<T *>(q);
    return rc;
}

size_t field_rows(int field, int nr)
{
    return (field == FCPT_VRAD || field == FCPT_VRAD0 || field == FCPT_TAU_R_PHI) ? (size_t)nr + 1
                                                                                : (size_t)nr;
}

// log-mesh ring lookups with the reference's NDEBUG clamps
// (find_cell_id.cpp:218-224, 259-264, 107-215; damping.cpp:321-327, 377-383)
int rmed_id_log(const fcpt_disk_desc &d, double r)
{
    const double g = std::pow(d.rmax / d.rmin, 1.0 / ((double)d.nr - 2.0));
    const double opt = 3.0 / 2.0 / d.rmin * (1 - std::pow(g, 2.0)) / (1 - std::pow(g, 3.0));
    const double inv_log = 1.0 / std::log(g);
    int id = (int)std::floor(std::log(r * opt) * inv_log) + 1;
    if (id < 0) id = 0;
    if (id > d.nr - 1) id = d.nr - 1;
    return id;
}
int rinf_id_log(const fcpt_disk_desc &d, double r)
{
    const double g = std::pow(d.rmax / d.rmin, 1.0 / ((double)d.nr - 2.0));
    const double inv_log = 1.0 / std::log(g);
    int id = (int)std::floor(std::log(r / d.rmin) * inv_log) + 1;
    if (id < 0) id = 0;
    if (id > d.nr - 1) id = d.nr - 1;
    return id;
}
int clampi(int v, int hi) { return v < 0 ? 0 : (v > hi ? hi : v); }

// The radial profiles of the reference's profile initial condition, one
// function of R each, in the reference's operand order so that they round
// the same way (host libm, no contraction): Sigma (init.cpp:946-957 and the
// cutoffs :1047-1148; get_sigma, viscous_radial_speed.cpp:95-118), the
// pressure-supported smoothed v_phi (Theo.cpp:131-181), the viscosity of the
// viscous-speed estimate (get_nu2, viscous_radial_speed.cpp:38-93) and the
// numerical viscous radial speed (:120-195).
struct DiskProfile {
    const fcpt_disk_desc &d;
    const fcpt_ic_desc &ic;

    static double cut_out(double point, double width, double x) { return 1.0 / (1.0 + std::exp((x - point) / width)); }
    static double cut_in(double point, double width, double x) { return 1.0 / (1.0 + std::exp((point - x) / width)); }
    static double max_(double a, double b) { return (a < b) ? b : a; }
    static double min_(double a, double b) { return (b < a) ? b : a; }
    double floor_value() const { return d.sigma_floor * d.sigma0; }

    double cutoff(double R) const
    {
        double c = 1.0;
        if (ic.cutoff_outer) c *= cut_out(ic.cutoff_outer_point, ic.cutoff_outer_width, R);
        if (ic.cutoff_inner) c *= cut_in(ic.cutoff_inner_point, ic.cutoff_inner_width, R);
        return c;
    }
    // the grid's Sigma: power law, floor, then each cutoff with the floor again
    double sigma_cell(double R) const
    {
        double s = max_(d.sigma0 * std::pow(R, -ic.sigma_slope), floor_value());
        if (ic.cutoff_outer) s = max_(s * cut_out(ic.cutoff_outer_point, ic.cutoff_outer_width, R), floor_value());
        if (ic.cutoff_inner) s = max_(s * cut_in(ic.cutoff_inner_point, ic.cutoff_inner_width, R), floor_value());
        return s;
    }
    // the viscous-speed estimate's Sigma: both cutoffs, then the floor once
    double sigma_model(double R) const
    {
        double s = d.sigma0 * std::pow(R, -ic.sigma_slope);
        if (ic.cutoff_outer) s *= cut_out(ic.cutoff_outer_point, ic.cutoff_outer_width, R);
        if (ic.cutoff_inner) s *= cut_in(ic.cutoff_inner_point, ic.cutoff_inner_width, R);
        return max_(s, floor_value());
    }
    double energy(double R) const
    {
        return 1.0 / (d.gamma - 1.0) * d.sigma0 * std::pow(d.aspect_ratio, 2) *
               std::pow(R, -ic.sigma_slope - 1.0 + 2.0 * d.flaring_index) * d.G * d.hydro_center_mass;
    }
    double energy_floor(double sig) const { return d.t_min * sig / d.mu * d.R / (d.gamma - 1.0); }
    double vphi(double R) const
    {
        const double F = d.flaring_index;
        const double h = d.aspect_ratio * std::pow(R, F);
        const double he = h * d.thickness_smoothing;
        const double smoothing = (1.0 + (F + 1.0) * std::pow(he, 2)) / std::pow(std::sqrt(1 + std::pow(he, 2)), 3);
        const double pressure = (2.0 * F - 1.0 - ic.sigma_slope) * std::pow(h, 2);
        const double vk_2 = d.G * d.hydro_center_mass / R;
        return std::sqrt(vk_2 * (smoothing + pressure));
    }
    double nu(double R, double sig) const
    {
        const double v_k = std::sqrt(d.G * d.hydro_center_mass / R);
        const double h = d.aspect_ratio * std::pow(R, d.flaring_index);
        if (!d.adiabatic) return d.alpha * (h * v_k) * (h * R);
        const double g = d.gamma;
        double e = cutoff(R) * 1.0 / (g - 1.0) * sig * std::pow(h * v_k, 2);
        e = max_(e, d.t_min * sig / d.mu * d.R / (g - 1.0));
        e = min_(e, d.t_max * sig / d.mu * d.R / (g - 1.0));
        const double cs_adb = std::sqrt(g * (g - 1.0) * e / sig);
        const double cs_iso = std::sqrt((g - 1.0) * e / sig);
        return d.alpha * cs_adb * (cs_iso / (v_k / R));
    }
    double omega(double r) const { return vphi(r) / r; }
    double r2_omega(double r) const { return std::pow(r, 2) * omega(r); }
    // five-point derivative with the step 8e-4 r
    template <class Fn>
    static double derivative(double r, Fn f)
    {
        const double h = 8.0e-4 * r;
        const double t = -1.0 * f(r + 2.0 * h) + 8.0 * f(r + h) + -8.0 * f(r - h) + 1.0 * f(r - 2.0 * h);
        return t / (12.0 * h);
    }
    double torque_flux(double r) const  // nu Sigma r^3 d(omega)/dr
    {
        const double dw = derivative(r, [this](double x) { return omega(x); });
        const double sig = sigma_model(r);
        return nu(r, sig) * sig * std::pow(r, 3) * dw;
    }
    double vr_viscous(double r) const
    {
        const double num = 1.0 / r * derivative(r, [this](double x) { return torque_flux(x); });
        const double den = sigma_model(r) * derivative(r, [this](double x) { return r2_omega(x); });
        return num / den;
    }
};

}  // namespace

extern "C" {

const char *fcpt_last_error(const fcpt_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int fcpt_create(const fcpt_disk_desc *desc, fcpt_ctx **out)
{
    if (!desc || !out) return FCPT_ERR_ARG;
    *out = nullptr;
    if (desc->nr < 8 || desc->nr > 16384 || desc->nphi < 4 || desc->nphi > 262144 || !desc->radii)
        return FCPT_ERR_ARG;
    if (desc->precision != FCPT_PREC_FP64 && desc->precision != FCPT_PREC_SPLIT32) return FCPT_ERR_ARG;
    if (desc->integrator != FCPT_INTEGRATOR_EULER && desc->integrator != FCPT_INTEGRATOR_LEAPFROG)
        return FCPT_ERR_ARG;
    if (desc->potential_smoothing & ~(FCPT_SMOOTHING_NO_STAR | FCPT_SMOOTHING_PLANETLOC)) return FCPT_ERR_ARG;
    for (int i = 0; i + 1 < desc->nr + 2; ++i)
        if (!(desc->radii[i + 1] > desc->radii[i]) || !(desc->radii[i] > 0.0)) return FCPT_ERR_ARG;
    fcpt_ctx *c = new fcpt_ctx();
    host_slots_join();
    c->desc = *desc;
    c->desc.radii = nullptr;
    hipError_t e = hipGetDevice(&c->device);
    if (e != hipSuccess) {
        host_slots_leave();
        delete c;
        return FCPT_ERR_DEVICE;
    }
    const int nr = desc->nr, ns = desc->nphi;
    KParams &P = c->P;
    P.nr = nr;
    P.ns = ns;
    P.split = desc->precision == FCPT_PREC_SPLIT32 ? 1 : 0;
    P.split_rounding = P.split;  // stochastic rounding of the split deviations by default
    c->rebase_interval = P.split ? kDefaultRebaseInterval : 0;
    P.radial_tile = 0;
    P.radial_waves = 3;
    P.visc_tile = 0;
    P.kick_tile = 0;
    P.kv_tile = 0;
    P.lazy_derived = 0;
    P.split_emul = 0;
    P.kick = P.pad_ = 0;
    P.ealt = nullptr;
    // Interpret.cpp:230-231
    P.dphi = 2.0 * M_PI / (double)ns;
    P.invdphi = (double)ns / (2.0 * M_PI);
    P.rmin = desc->rmin;
    P.rmax = desc->rmax;
    P.adiabatic = desc->adiabatic;
    P.integrator = desc->integrator;
    P.artvisc = desc->artificial_viscosity;
    P.artvisc_dissipation = desc->artvisc_dissipation;
    P.heating_viscous = desc->heating_viscous;
    P.cooling_beta_enabled = desc->cooling_beta_enabled;
    P.cooling_beta_ref = desc->cooling_beta_ref;
    P.bc_inner = desc->bc_inner;
    P.bc_outer = desc->bc_outer;
    P.damping = desc->damping;
    P.G = desc->G;
    P.Rgas = desc->R;
    P.sigma_sb = desc->sigma_sb;
    P.c_light = desc->c_light;
    P.mstar = desc->hydro_center_mass;
    P.mu = desc->mu;
    P.gamma = desc->gamma;
    P.aspect_ratio = desc->aspect_ratio;
    P.flaring = desc->flaring_index;
    P.alpha = desc->alpha;
    P.thickness_smoothing = desc->thickness_smoothing;
    P.cfl = desc->cfl;
    P.cfl_max_var = desc->cfl_max_var;
    P.heating_cooling_cfl_limit = desc->heating_cooling_cfl_limit;
    P.sigma0 = desc->sigma0;
    P.sigma_floor = desc->sigma_floor;
    P.t_min = desc->t_min;
    P.t_max = desc->t_max;
    P.artvisc_factor = desc->artvisc_factor;
    P.heating_viscous_factor = desc->heating_viscous_factor;
    P.cooling_beta = desc->cooling_beta;
    P.cooling_beta_ramp_up = desc->cooling_beta_ramp_up;
    P.radial_viscosity_factor = desc->radial_viscosity_factor;
    P.damping_inner_limit = desc->damping_inner_limit;
    P.damping_outer_limit = desc->damping_outer_limit;
    P.damping_time_factor = desc->damping_time_factor;
    P.damping_time_radius_outer = desc->damping_time_radius_outer;
    P.omega_frame = desc->omega_frame;
    P.energy_per_t = P.Rgas / P.mu / (P.gamma - 1.0);
    P.const_ok = 1;
    for (double c : {P.Rgas, P.mu, P.gamma, P.gamma - 1.0, P.alpha, P.sigma_sb, P.c_light, P.G * P.mstar, P.radial_viscosity_factor, P.heating_viscous_factor})
        if (!(c >= 0x1p-40 && c <= 0x1p40)) P.const_ok = 0;
    if (!(desc->radii[0] >= 0x1p-20 && desc->radii[nr + 1] <= 0x1p20)) P.const_ok = 0;
    P.monitor_timestep = desc->monitor_timestep;
    int ids[4] = {desc->damp_inner_scalar, desc->damp_inner_vector, desc->damp_outer_scalar,
                  desc->damp_outer_vector};
    if (ids[0] < 0) ids[0] = clampi(rmed_id_log(*desc, desc->rmin * desc->damping_inner_limit), nr - 1);
    if (ids[1] < 0) ids[1] = clampi(rinf_id_log(*desc, desc->rmin * desc->damping_inner_limit), nr);
    if (ids[2] < 0)
        ids[2] = clampi(rmed_id_log(*desc, desc->rmax * desc->damping_outer_limit) + 1, nr - 1);
    if (ids[3] < 0)
        ids[3] = clampi(rinf_id_log(*desc, desc->rmax * desc->damping_outer_limit) + 1, nr);
    memcpy(P.damp_ids, ids, sizeof(ids));
    if (desc->damping && (ids[0] >= ids[2] || ids[1] >= ids[3])) {
        host_slots_leave();
        delete c;
        return FCPT_ERR_ARG;  // inner and outer damping zones overlap
    }

    // the zones as damping_single_inner / _outer test them (damping.cpp:311-427)
    for (int v = 0; v < 2; ++v) {
        // radius[0] and radius[size_radial - 1] of the scalar (Rmed) and vector (Rinf) grids
        auto rmed = [&](int i) {
            const double a = desc->radii[i], b = desc->radii[i + 1];
            double r = 2.0 / 3.0 * (std::pow(b, 3) - std::pow(a, 3));
            return r / (std::pow(b, 2) - std::pow(a, 2));
        };
        const double first = v ? desc->radii[0] : rmed(0), last = v ? desc->radii[nr] : rmed(nr - 1);
        const double lin = P.damping_inner_limit, lout = P.damping_outer_limit;
        P.zone_in[v] = P.damping && lin > 1.0 && first < P.rmin * lin ? ids[v] : -1;
        P.zone_out[v] = P.damping && lout < 1.0 && last > P.rmax * lout ? ids[2 + v] : INT32_MAX;
    }

    // per-ring metric arrays, init_radialarrays (init.cpp:188-225), in FP64 on the host
    const int n1 = nr + 2;
    std::vector<double> Rinf(n1, 0), Rsup(n1, 0), Rmed(n1, 0), Surf(n1, 0), InvSurf(n1, 0),
        InvRmed(n1, 0), InvRinf(n1, 0), InvDiffRmed(n1, 0), InvDiffRsup(n1, 0),
        InvDiffRsupRb(n1, 0), cosphi(ns), sinphi(ns);
    for (int i = 0; i < nr + 1; ++i) {
        Rinf[i] = desc->radii[i];
        Rsup[i] = desc->radii[i + 1];
        Rmed[i] = 2.0 / 3.0 * (std::pow(Rsup[i], 3) - std::pow(Rinf[i], 3));
        Rmed[i] = Rmed[i] / (std::pow(Rsup[i], 2) - std::pow(Rinf[i], 2));
        Surf[i] = M_PI * (std::pow(Rsup[i], 2) - std::pow(Rinf[i], 2)) / (double)ns;
        InvRmed[i] = 1.0 / Rmed[i];
        InvSurf[i] = 1.0 / Surf[i];
        InvDiffRsup[i] = 1.0 / (Rsup[i] - Rinf[i]);
        InvDiffRsupRb[i] = 1.0 / ((Rsup[i] - Rinf[i]) * Rmed[i]);
        InvRinf[i] = 1.0 / Rinf[i];
    }
    for (int i = 1; i < nr + 1; ++i) InvDiffRmed[i] = 1.0 / (Rmed[i] - Rmed[i - 1]);
    c->Rinf = Rinf;
    c->Rmed = Rmed;
    c->Surf = Surf;
    c->InvRmed = InvRmed;
    c->InvDiffRmed = InvDiffRmed;
    c->InvDiffRsup = InvDiffRsup;
    c->InvDiffRsupRb = InvDiffRsupRb;
    for (int j = 0; j < ns; ++j) {
        // cell centres, SideEuler.cpp:57-66
        cosphi[j] = std::cos(P.dphi * (double)j);
        sinphi[j] = std::sin(P.dphi * (double)j);
    }

    int rc = FCPT_OK;
    auto upload = [&](const double **dst, const std::vector<double> &src) -> int {
        double *d = nullptr;
        int r = dev_alloc(c, &d, src.size());
        if (r) return r;
        hipError_t e2 = hipMemcpy(d, src.data(), src.size() * sizeof(double), hipMemcpyHostToDevice);
        if (e2 != hipSuccess) return fail(c, FCPT_ERR_DEVICE, "hipMemcpy: %s", hipGetErrorString(e2));
        *dst = d;
        return FCPT_OK;
    };
    if ((rc = upload(&P.Rinf, Rinf)) || (rc = upload(&P.Rsup, Rsup)) || (rc = upload(&P.Rmed, Rmed)) ||
        (rc = upload(&P.Surf, Surf)) || (rc = upload(&P.InvSurf, InvSurf)) ||
        (rc = upload(&P.InvRmed, InvRmed)) || (rc = upload(&P.InvRinf, InvRinf)) ||
        (rc = upload(&P.InvDiffRmed, InvDiffRmed)) || (rc = upload(&P.InvDiffRsup, InvDiffRsup)) ||
        (rc = upload(&P.InvDiffRsupRb, InvDiffRsupRb)) || (rc = upload(&P.cosphi, cosphi)) ||
        (rc = upload(&P.sinphi, sinphi))) {
        fcpt_destroy(c);
        return rc;
    }
    const size_t ncell = (size_t)nr * ns;
    const size_t esz = element_size(P);
    for (int k = 0; k < FCPT_NUM_FIELDS && !rc; ++k)
        rc = dev_alloc_bytes(c, &P.f[k], field_rows(k, nr) * ns * field_element_size(P, k));
    if (!rc) rc = dev_alloc_bytes(c, &P.valt[0], field_rows(FCPT_VRAD, nr) * ns * esz);
    if (!rc) rc = dev_alloc_bytes(c, &P.valt[1], field_rows(FCPT_VAZI, nr) * ns * esz);
    if (!rc && P.adiabatic) rc = dev_alloc_bytes(c, &P.ealt, field_rows(FCPT_ENERGY, nr) * ns * esz);
    for (int k = 0; k < 4 && !rc; ++k) rc = dev_alloc_bytes(c, &P.mom[k], ncell * sizeof(double));  // FP64 in both modes
    if (!rc) rc = dev_alloc_bytes(c, &P.sig_c, ncell * sizeof(double));
    if (!rc) rc = dev_alloc_bytes(c, &P.en_c, ncell * sizeof(double));
    if (P.split) {
        for (int k = 0; k < FCPT_NUM_FIELDS && !rc; ++k) rc = dev_alloc(c, &P.bg[k], (size_t)nr + 2);
        for (int k = 0; k < 4 && !rc; ++k) rc = dev_alloc(c, &P.bgm[k], (size_t)nr + 2);
        if (!rc) rc = dev_alloc(c, &c->bg_tmp, (size_t)nr + 2);
        for (int k = 0; k < FCPT_NUM_FIELDS; ++k) c->hbg[k].assign((size_t)nr + 2, 0.0);
    }
    if (!rc) rc = dev_alloc(c, &P.iso_cs, (size_t)nr + 2);
    if (!rc) rc = dev_alloc(c, &P.iso_h, (size_t)nr + 2);
    if (!rc) rc = dev_alloc(c, &P.iso_nu, (size_t)nr + 2);
    if (!rc) rc = dev_alloc(c, &P.ring_tab, (size_t)kRingTabs * ((size_t)nr + 2));
    if (!rc) rc = dev_alloc(c, &P.sweep_tab, kSweepTabs * ((size_t)nr + 2));
    if (!rc) rc = dev_alloc(c, &P.cfl_tab, 8 * ((size_t)nr + 2));
    if (!rc) rc = dev_alloc(c, &P.damp_tab, 8 * ((size_t)nr + 2));
    if (!rc) rc = dev_alloc(c, &P.vmean, (size_t)nr + 1);
    if (!rc) rc = dev_alloc(c, &P.vuni, (size_t)nr + 1);
    if (!rc) rc = dev_alloc(c, &P.nshift, (size_t)nr + 1);
    if (!rc) rc = dev_alloc(c, &P.ring_min, (size_t)nr);
    if (!rc) rc = dev_alloc(c, &c->s_dev, 1);
    if (!rc) rc = dev_alloc(c, &c->totals_ring, 4 * (size_t)nr);
    if (!rc) rc = dev_alloc(c, &c->totals_out, 2);
    if (!rc) rc = dev_alloc(c, &c->force_part, (size_t)nr * 4 * kForceMaxBodies);
    if (rc) {
        fcpt_destroy(c);
        return rc;
    }
    P.s = c->s_dev;
    P.step_at = &c->s_dev->step_count;
    e = hipHostMalloc((void **)&c->s_host, sizeof(DevScalars), hipHostMallocDefault);
    if (e == hipSuccess) e = hipHostMalloc((void **)&c->totals_host, 2 * sizeof(double), hipHostMallocDefault);
    if (e == hipSuccess)
        e = hipHostMalloc((void **)&c->force_host, 4 * kForceMaxBodies * sizeof(double), hipHostMallocDefault);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        fcpt_destroy(c);
        return FCPT_ERR_DEVICE;
    }
    // zero every field (the reference's t_polargrid::set_size clears its arrays);
    // split storage: zero backgrounds and zero deviations
    for (int k = 0; k < FCPT_NUM_FIELDS; ++k)
        e = e == hipSuccess ? hipMemset(P.f[k], 0, field_rows(k, nr) * ns * field_element_size(P, k)) : e;
    for (int k = 0; P.split && k < FCPT_NUM_FIELDS; ++k)
        e = e == hipSuccess ? hipMemset(P.bg[k], 0, ((size_t)nr + 2) * sizeof(double)) : e;
    for (int k = 0; P.split && k < 4; ++k)
        e = e == hipSuccess ? hipMemset(P.bgm[k], 0, ((size_t)nr + 2) * sizeof(double)) : e;
    std::memset(c->s_host, 0, sizeof(DevScalars));
    c->s_host->count_next = 1;
    if (e == hipSuccess) e = hipMemcpy(c->s_dev, c->s_host, sizeof(DevScalars), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        launch_ring_tables(P, c->stream);
        if (!P.adiabatic) launch_iso_rings(P, c->stream);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    }
    if (e != hipSuccess) {
        fcpt_destroy(c);
        return FCPT_ERR_DEVICE;
    }
    *out = c;
    return FCPT_OK;
}

int fcpt_destroy(fcpt_ctx *ctx)
{
    if (!ctx) return FCPT_OK;
    hipSetDevice(ctx->device);
    if (ctx->stream) {
        hipStreamSynchronize(ctx->stream);
        hipStreamDestroy(ctx->stream);
    }
    drop_graphs(ctx->step_graph);
    if (ctx->ev0) hipEventDestroy(ctx->ev0);
    if (ctx->ev1) hipEventDestroy(ctx->ev1);
    for (void *p : ctx->allocs) hipFree(p);
    if (ctx->s_host) hipHostFree(ctx->s_host);
    if (ctx->totals_host) hipHostFree(ctx->totals_host);
    if (ctx->force_host) hipHostFree(ctx->force_host);
    host_slots_leave();
    delete ctx;
    return FCPT_OK;
}

int fcpt_synchronize(fcpt_ctx *ctx)
{
    CTX_CHECK(ctx);
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return FCPT_OK;
}

// read back the device scalars; flags a non-finite CFL result
static int read_scalars(fcpt_ctx *ctx)
{
    HIP_TRY(ctx, hipMemcpyAsync(ctx->s_host, ctx->s_dev, sizeof(DevScalars), hipMemcpyDeviceToHost,
                                ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return FCPT_OK;
}

// the non-finite-dt flag is reported once: a call that reports it clears it
// on the device, as do a new clock and a new state
static int clear_error_flags(fcpt_ctx *ctx)
{
    HIP_TRY(ctx, hipMemsetAsync(&ctx->s_dev->error_flags, 0, sizeof(int), ctx->stream));
    return FCPT_OK;
}
static bool take_nonfinite(fcpt_ctx *ctx)
{
    if (!(ctx->s_host->error_flags & 1)) return false;
    ctx->s_host->error_flags &= ~1;
    clear_error_flags(ctx);
    return true;
}

// split storage: the field's background becomes its ring means, the device
// holds (float)(value - background)
static int upload_split(fcpt_ctx *ctx, int field, const double *host)
{
    const int ns = ctx->P.ns;
    const size_t rows = field_rows(field, ctx->P.nr);
    std::vector<double> &bg = ctx->hbg[field];
    bg.assign((size_t)ctx->P.nr + 2, 0.0);
    std::vector<float> d(rows * ns);
    for (size_t i = 0; i < rows; ++i) {
        const double *row = host + i * ns;
        double sum = 0.0;
        for (int j = 0; j < ns; ++j) sum += row[j];
        bg[i] = sum / (double)ns;
        for (int j = 0; j < ns; ++j) d[i * ns + j] = (float)(row[j] - bg[i]);
    }
    HIP_TRY(ctx, hipMemcpyAsync(ctx->P.bg[field], bg.data(), bg.size() * sizeof(double),
                                hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipMemcpyAsync(ctx->P.f[field], d.data(), d.size() * sizeof(float),
                                hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return FCPT_OK;
}

// ---- fields to the host ----------------------------------------------------
// A copy into the caller's pageable arrays is bound by the host: its pages are
// touched for the first time (the kernel clears them) and written by one
// thread: 1.6 GB took 158 ms into touched pages and 233 into fresh ones, where the
// link takes 30.  So the bytes go through pinned slots, in pieces: the link fills
// a slot while kCopyThreads threads move earlier ones to the caller (and decode
// split storage's FP32 deviations there, so half the bytes cross the link): 37 ms
// into touched pages and 83 into fresh ones, and 21 for split storage instead of
// 292.  What fits the slots as a whole is decoded and written to
// them by one kernel, all fields at once: each transfer and its event cost
// tens of microseconds, more than the link's time below some MB (512 x
// 1536: 1.5 - 3.5 -> 0.9 - 1.5 ms, 32 x 64: 80 -> 21 us; slots filled in smaller
// pieces were slower than in one).
//
// The slots belong to the process: allocated by the first copy that needs them,
// as large as it asks, rounded up to a power of two (pinning 2, 4 and 48 MB costs
// 0.12 - 0.17, 0.3 and 0.5 ms), replaced by larger ones when one asks for more,
// lent to one copy at a time, and freed with the last context.  A copy that finds
// them lent to one whose disk's queue still runs goes without them, so that no
// disk's steps hold up another's copy (waiting for the own queue before taking the
// slots cost every copy behind queued steps 10 to 18 us); it waits for one that moves
// its bytes.  Copies up to 1 MB take a buffer each, as many as ever ran at once.  A
// copy that gets none goes without, as does the process's first of each kind that fits them: a
// process's first pinning and first use of it cost more than one copy gains (first
// copy of a 128x384 state 0.65 ms with them, 0.1 without; 512x1536 2.9 and 1.5).
constexpr size_t kSlotBytes = size_t(4) << 20;
constexpr int kSlots = 12, kCopyThreads = 8;
constexpr size_t kSmallBytes = size_t(1) << 20;  // copies up to this size take a buffer of their own
// One field that needs no decoding, above this size and up to kSmallBytes, is the
// runtime's to copy: 17 KB 10.8 us, 48 KB 12.3, 384 KB 25.9, 760 KB 41.1, where the
// kernel and the copy out of its buffer take 15.2, 16.0, 29.5, 45.3; 16 KB take
// 28.2 and 15.1, 1.5 MB 88.5 and 86.2, 3.1 MB 180 and 139.
constexpr size_t kDirectAbove = size_t(16) << 10;

struct HostSlots {
    std::mutex life;
    int users = 0;
    std::condition_variable freed;
    bool lent = false, queued = false;  // the slots; to a copy whose disk's queue still runs
    std::vector<char *> small;  // small buffers not in use
    size_t small_made = 0;
    char *slots = nullptr;
    size_t slots_bytes = 0;
    bool asked[2] = {false, false};  // by a copy for a small buffer, for the slots
};
static HostSlots &host_slots()
{
    static HostSlots *h = new HostSlots;  // outlives contexts that a program destroys at its end
    return *h;
}
static void host_slots_join()
{
    std::lock_guard<std::mutex> g(host_slots().life);
    ++host_slots().users;
}
static void host_slots_leave()
{
    HostSlots &h = host_slots();
    std::lock_guard<std::mutex> g(h.life);
    if (--h.users > 0) return;
    for (char *p : h.small) hipHostFree(p);
    h.small.clear();
    h.small_made = 0;
    if (h.slots) hipHostFree(h.slots);
    h.slots = nullptr;
}
// pinned memory, or null: the caller goes another way, and no later call reports it
static char *host_pin(size_t bytes)
{
    void *p = nullptr;
    if (hipHostMalloc(&p, bytes, hipHostMallocPortable) == hipSuccess) return static_cast<char *>(p);
    hipGetLastError();
    return nullptr;
}
// a small buffer for as long as this lives
struct SmallBuffer {
    char *p = nullptr;
    SmallBuffer()
    {
        HostSlots &h = host_slots();
        std::lock_guard<std::mutex> g(h.life);
        if (!h.small.empty()) {
            p = h.small.back();
            h.small.pop_back();
        } else if (!h.asked[0]) {
            h.asked[0] = true;
        } else {
            h.small.reserve(h.small_made + 1);  // room for its return
            p = host_pin(kSmallBytes);
            if (p) ++h.small_made;
        }
    }
    ~SmallBuffer()
    {
        if (!p) return;
        std::lock_guard<std::mutex> g(host_slots().life);
        host_slots().small.push_back(p);
    }
    SmallBuffer(const SmallBuffer &) = delete;
};
// the slots for as long as this lives, `bytes` or all of them, or null
struct SlotsLoan {
    char *p = nullptr;
    explicit SlotsLoan(size_t bytes);
    // the borrower's own queue has run
    void moving()
    {
        std::lock_guard<std::mutex> g(host_slots().life);
        host_slots().queued = false;
    }
    ~SlotsLoan()
    {
        if (!p) return;
        HostSlots &h = host_slots();
        std::lock_guard<std::mutex> g(h.life);
        h.lent = h.queued = false;
        h.freed.notify_all();
    }
    SlotsLoan(const SlotsLoan &) = delete;
};
SlotsLoan::SlotsLoan(size_t bytes)
{
    HostSlots &h = host_slots();
    std::unique_lock<std::mutex> g(h.life);
    h.freed.wait(g, [&] { return !h.lent || h.queued; });
    if (h.lent) return;
    size_t want = kSmallBytes;
    while (want < bytes && want < kSlotBytes * kSlots) want *= 2;
    want = std::min(want, kSlotBytes * kSlots);
    if (h.slots && h.slots_bytes < want) {
        hipHostFree(h.slots);
        h.slots = nullptr;
    }
    if (!h.slots) {
        if (!h.asked[1] && bytes <= kSlotBytes * kSlots) {
            h.asked[1] = true;
            return;
        }
        h.slots = host_pin(want);
        h.slots_bytes = want;
    }
    p = h.slots;
    h.lent = h.queued = p != nullptr;
}

struct HostCopy {
    int field;
    double *dst;
};
struct HostCopies {
    HostCopy c[4];
    size_t n = 0;
    void add(int field, double *dst) { c[n++] = HostCopy{field, dst}; }
    size_t size() const { return n; }
    const HostCopy &operator[](size_t k) const { return c[k]; }
    const HostCopy *begin() const { return c; }
    const HostCopy *end() const { return c + n; }
};

// one piece of a copy: n elements of fields[which] from element `first` on
struct CopyPiece {
    int which;
    size_t first, n;
};

// each field straight into the caller's pages
static int copy_pageable(fcpt_ctx *ctx, const HostCopies &fields)
{
    const KParams &P = ctx->P;
    hipError_t e = hipSuccess;
    for (const HostCopy &f : fields) {
        const size_t rows = field_rows(f.field, P.nr), ns = (size_t)P.ns;
        const bool decode = P.split && f.field != FCPT_POTENTIAL;
        std::vector<double> bg(decode ? rows : 0);
        std::vector<float> dev(decode ? rows * ns : 0);
        void *const to = decode ? (void *)dev.data() : (void *)f.dst;
        if (decode) e = hipMemcpyAsync(bg.data(), P.bg[f.field], rows * sizeof(double), hipMemcpyDeviceToHost, ctx->stream);
        if (e == hipSuccess)
            e = hipMemcpyAsync(to, P.f[f.field], rows * ns * field_element_size(P, f.field), hipMemcpyDeviceToHost, ctx->stream);
        const hipError_t se = hipStreamSynchronize(ctx->stream);  // nothing in flight into bg and dev below
        if (e == hipSuccess) e = se;
        HIP_TRY(ctx, e);
        for (size_t i = 0; decode && i < rows; ++i)
            for (size_t j = 0; j < ns; ++j) f.dst[i * ns + j] = bg[i] + (double)dev[i * ns + j];
    }
    return FCPT_OK;
}

static int copy_large(fcpt_ctx *ctx, const HostCopies &fields, SlotsLoan &loan)
{
    const KParams &P = ctx->P;
    char *const slots = loan.p;
    const size_t ns = (size_t)P.ns;
    std::vector<CopyPiece> pieces;
    std::vector<std::vector<double>> bg(fields.size());
    hipError_t err = hipSuccess;
    for (size_t k = 0; k < fields.size(); ++k) {
        const int f = fields[k].field;
        const size_t total = field_rows(f, P.nr) * ns, most = kSlotBytes / field_element_size(P, f);
        for (size_t a = 0; a < total; a += most) pieces.push_back({(int)k, a, std::min(most, total - a)});
        if (P.split && f != FCPT_POTENTIAL) {
            bg[k].resize(field_rows(f, P.nr));
            const hipError_t e = hipMemcpyAsync(bg[k].data(), P.bg[f], bg[k].size() * sizeof(double),
                                                hipMemcpyDeviceToHost, ctx->stream);
            if (err == hipSuccess) err = e;
        }
    }
    hipEvent_t ev[kSlots] = {};
    for (int k = 0; k < kSlots && err == hipSuccess; ++k) err = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    const hipError_t queue = hipStreamSynchronize(ctx->stream);  // the disk's own, and the backgrounds
    if (err == hipSuccess) err = queue;
    loan.moving();
    std::mutex m;
    std::condition_variable cv;
    size_t issued = 0, next = 0;
    std::vector<char> done(pieces.size(), 0);
    bool stop = err != hipSuccess;
    // moves piece c, whose transfer has been issued, out of its slot
    auto move_out = [&](size_t c) -> hipError_t {
        const hipError_t e = hipEventSynchronize(ev[c % kSlots]);
        if (e != hipSuccess) return e;
        const CopyPiece &p = pieces[c];
        const char *src = slots + (c % kSlots) * kSlotBytes;
        double *dst = fields[(size_t)p.which].dst + p.first;
        if (bg[(size_t)p.which].empty()) {
            std::memcpy(dst, src, p.n * sizeof(double));
            return hipSuccess;
        }
        const float *d = reinterpret_cast<const float *>(src);
        const double *b = bg[(size_t)p.which].data();
        for (size_t a = 0; a < p.n;) {
            const size_t row = (p.first + a) / ns, end = std::min(p.n, (row + 1) * ns - p.first);
            const double base = b[row];
            for (; a < end; ++a) dst[a] = base + (double)d[a];
        }
        return hipSuccess;
    };
    auto work = [&]() {
        hipError_t e = hipSetDevice(ctx->device);
        for (;;) {
            size_t c;
            {
                std::unique_lock<std::mutex> l(m);
                if (e != hipSuccess) {
                    err = e;
                    stop = true;
                    cv.notify_all();
                }
                cv.wait(l, [&] { return stop || next < issued || next >= pieces.size(); });
                if (stop || next >= pieces.size()) return;
                c = next++;
            }
            e = move_out(c);
            std::lock_guard<std::mutex> l(m);
            done[c] = 1;
            cv.notify_all();
        }
    };
    std::vector<std::thread> threads;
    if (!stop) {
        const size_t want = std::min<size_t>(kCopyThreads, pieces.size());
        try {
            threads.reserve(want);
            for (size_t t = 0; t < want; ++t) threads.emplace_back(work);
        } catch (...) {  // fewer threads than wanted; with none, this one moves the pieces
        }
    }
    for (size_t c = 0; c < pieces.size(); ++c) {
        {
            std::unique_lock<std::mutex> l(m);
            cv.wait(l, [&] { return stop || threads.empty() || c < kSlots || done[c - kSlots]; });
            if (stop) break;
        }
        const CopyPiece &p = pieces[c];
        const int f = fields[(size_t)p.which].field;
        const size_t esz = field_element_size(P, f);
        hipError_t e = hipMemcpyAsync(slots + (c % kSlots) * kSlotBytes, static_cast<const char *>(P.f[f]) + p.first * esz,
                                      p.n * esz, hipMemcpyDeviceToHost, ctx->stream);
        if (e == hipSuccess) e = hipEventRecord(ev[c % kSlots], ctx->stream);
        if (e == hipSuccess && threads.empty()) e = move_out(c);
        std::lock_guard<std::mutex> l(m);
        if (e != hipSuccess) {
            err = e;
            stop = true;
        } else {
            issued = c + 1;
        }
        cv.notify_all();
    }
    for (std::thread &t : threads) t.join();
    const hipError_t se = hipStreamSynchronize(ctx->stream);  // no transfer into a slot outlives the lease
    for (hipEvent_t e : ev)
        if (e) hipEventDestroy(e);
    HIP_TRY(ctx, err);
    HIP_TRY(ctx, se);
    return FCPT_OK;
}

// all fields by one kernel into the slots, then to the caller: by this thread
// below 1 MB, by several above
static int copy_export(fcpt_ctx *ctx, const HostCopies &fields, size_t total, char *out, SlotsLoan *loan)
{
    const KParams &P = ctx->P;
    ExportFields x{};
    size_t at = 0;
    for (const HostCopy &f : fields) {
        x.field[x.n] = f.field;
        x.rows[x.n] = (int)field_rows(f.field, P.nr);
        x.out[x.n] = reinterpret_cast<double *>(out) + at;
        at += (size_t)x.rows[x.n++] * (size_t)P.ns;
    }
    launch_export(P, ctx->stream, x);
    LAUNCH_CHECK(ctx);
    // strip t of T of every field
    auto strip = [&](size_t t, size_t T) {
        for (int k = 0; k < x.n; ++k) {
            const size_t n = (size_t)x.rows[k] * (size_t)P.ns, a = n * t / T, b = n * (t + 1) / T;
            std::memcpy(fields[(size_t)k].dst + a, x.out[k] + a, (b - a) * sizeof(double));
        }
    };
    const size_t T = std::max<size_t>(1, std::min<size_t>(kCopyThreads, total / kSmallBytes));
    std::mutex m;
    std::condition_variable cv;
    int go = 0;  // 1: the slots are filled, -1: they will not be
    std::vector<std::thread> threads;
    try {
        threads.reserve(T - 1);
        for (size_t t = 1; t < T; ++t)
            threads.emplace_back([&, t] {
                {
                    std::unique_lock<std::mutex> l(m);
                    cv.wait(l, [&] { return go != 0; });
                }
                if (go > 0) strip(t, T);
            });
    } catch (...) {  // this thread takes the strips that have no other
    }
    const hipError_t e = hipStreamSynchronize(ctx->stream);
    if (loan) loan->moving();
    {
        std::lock_guard<std::mutex> l(m);
        go = e == hipSuccess ? 1 : -1;
    }
    cv.notify_all();
    if (e == hipSuccess) {
        strip(0, T);
        for (size_t t = threads.size() + 1; t < T; ++t) strip(t, T);
    }
    for (std::thread &t : threads) t.join();
    HIP_TRY(ctx, e);
    return FCPT_OK;
}

// the fields to the caller's arrays in FP64 (split storage: background +
// deviation)
static int copy_to_host(fcpt_ctx *ctx, const HostCopies &fields)
{
    const KParams &P = ctx->P;
    size_t total = 0;
    for (const HostCopy &f : fields) total += field_rows(f.field, P.nr) * (size_t)P.ns * sizeof(double);
    try {
        const bool stored = !P.split || fields.c[0].field == FCPT_POTENTIAL;
        if (fields.n == 1 && stored && total > kDirectAbove && total <= kSmallBytes) return copy_pageable(ctx, fields);
        if (total <= kSmallBytes) {
            SmallBuffer b;
            if (b.p) return copy_export(ctx, fields, total, b.p, nullptr);
        } else {
            SlotsLoan loan(total);
            if (loan.p && total > kSlotBytes * kSlots) return copy_large(ctx, fields, loan);
            if (loan.p) return copy_export(ctx, fields, total, loan.p, &loan);
        }
        return copy_pageable(ctx, fields);
    } catch (const std::exception &e) {
        return fail(ctx, FCPT_ERR_DEVICE, "copy to the host: %s", e.what());
    }
}

int fcpt_upload_field(fcpt_ctx *ctx, int32_t field, const double *host)
{
    CTX_SYNCED(ctx);
    if (field < 0 || field >= FCPT_NUM_FIELDS || !host) return fail(ctx, FCPT_ERR_ARG, "bad field");
    if (field == FCPT_SIGMA || field == FCPT_ENERGY || derived_field(field)) ctx->derived_own = false;
    if (ctx->P.split && field != FCPT_POTENTIAL) return upload_split(ctx, field, host);
    const size_t n = field_rows(field, ctx->P.nr) * ctx->P.ns;
    HIP_TRY(ctx, hipMemcpyAsync(ctx->P.f[field], host, n * sizeof(double), hipMemcpyHostToDevice,
                                ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return FCPT_OK;
}

int fcpt_download_field(fcpt_ctx *ctx, int32_t field, double *host)
{
    CTX_CHECK(ctx);
    if (field < 0 || field >= FCPT_NUM_FIELDS || !host) return fail(ctx, FCPT_ERR_ARG, "bad field");
    if (derived_field(field))
        if (const int rc = sync_derived(ctx)) return rc;
    HostCopies one;
    one.add(field, host);
    return copy_to_host(ctx, one);
}

// split storage: re-express a field about a new host-given background
static int rebase_field(fcpt_ctx *ctx, int field, const std::vector<double> &newbg)
{
    const KParams &P = ctx->P;
    HIP_TRY(ctx, hipMemcpyAsync(ctx->bg_tmp, newbg.data(), ((size_t)P.nr + 2) * sizeof(double),
                                hipMemcpyHostToDevice, ctx->stream));
    launch_rebase(P, ctx->stream, P.f[field], P.bg[field], ctx->bg_tmp, (int)field_rows(field, P.nr));
    LAUNCH_CHECK(ctx);
    HIP_TRY(ctx, hipMemcpyAsync(P.bg[field], ctx->bg_tmp, ((size_t)P.nr + 2) * sizeof(double),
                                hipMemcpyDeviceToDevice, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    ctx->hbg[field] = newbg;
    return FCPT_OK;
}

// split storage: backgrounds of the derived fields and of the transport
// momenta, evaluated from the ring backgrounds of Sigma, v_r, v_phi and E with
// the expressions of the kernels that produce those fields (azimuthal
// differences vanish on a ring profile)
static int set_derived_backgrounds(fcpt_ctx *ctx)
{
    const KParams &P = ctx->P;
    const int nr = P.nr;
    const std::vector<double> &S = ctx->hbg[FCPT_SIGMA], &VR = ctx->hbg[FCPT_VRAD],
                              &VA = ctx->hbg[FCPT_VAZI], &E = ctx->hbg[FCPT_ENERGY];
    const size_t n1 = (size_t)nr + 2;
    std::vector<double> cs(n1, 0.0), H(n1, 0.0), Pr(n1, 0.0), nu(n1, 0.0), T(n1, 0.0), dv(n1, 0.0),
        trr(n1, 0.0), tpp(n1, 0.0), trp(n1, 0.0), mr0(n1, 0.0), mr1(n1, 0.0), ma(n1, 0.0);
    const double g = P.gamma;
    for (int i = 0; i < nr; ++i) {
        const double R = ctx->Rmed[i];
        const double omk = std::sqrt(P.G * P.mstar / (R * R * R));
        double c, h;
        if (P.adiabatic) {
            c = std::sqrt(g * (g - 1.0) * E[i] / S[i]);
            h = c / std::sqrt(g) / omk;
            Pr[i] = (g - 1.0) * E[i];
            T[i] = P.mu / P.Rgas * (g - 1.0) * E[i] / S[i];
        } else {
            c = P.aspect_ratio * std::pow(R, P.flaring) * std::sqrt(P.G * P.mstar / R);
            h = c / omk;
            Pr[i] = S[i] * (c * c);
            T[i] = P.mu / P.Rgas * Pr[i] / S[i];
        }
        cs[i] = c;
        H[i] = h;
        nu[i] = P.alpha * h * c;
        dv[i] = (VR[i + 1] * ctx->Rinf[i + 1] - VR[i] * ctx->Rinf[i]) * ctx->InvDiffRsupRb[i];
        trr[i] = 2.0 * nu[i] * S[i] * ((VR[i + 1] - VR[i]) * ctx->InvDiffRsup[i] - dv[i] / 3.0);
        tpp[i] = 2.0 * nu[i] * S[i] * (0.5 * (VR[i + 1] + VR[i]) * ctx->InvRmed[i] - dv[i] / 3.0);
        if (i >= 1)
            trp[i] = 0.5 * (nu[i] + nu[i - 1]) * 0.5 * (S[i] + S[i - 1]) * ctx->Rinf[i] *
                     (VA[i] * ctx->InvRmed[i] - VA[i - 1] * ctx->InvRmed[i - 1]) * ctx->InvDiffRmed[i];
        mr0[i] = S[i] * VR[i + 1];
        mr1[i] = S[i] * VR[i];
        ma[i] = S[i] * (VA[i] + R * P.omega_frame) * R;
    }
    if (!std::isfinite(cs[1]) || !std::isfinite(trp[1]))
        return fail(ctx, FCPT_ERR_ARG, "split storage needs a positive Sigma (and E) on every ring");
    const std::pair<int, const std::vector<double> *> derived[] = {
        {FCPT_SOUNDSPEED, &cs}, {FCPT_SCALE_HEIGHT, &H},  {FCPT_PRESSURE, &Pr},
        {FCPT_VISCOSITY, &nu},  {FCPT_TEMPERATURE, &T},   {FCPT_DIV_V, &dv},
        {FCPT_TAU_R_R, &trr},   {FCPT_TAU_PHI_PHI, &tpp}, {FCPT_TAU_R_PHI, &trp}};
    for (const auto &fd : derived) {
        const int rc = rebase_field(ctx, fd.first, *fd.second);
        if (rc) return rc;
    }
    const std::vector<double> *mom[4] = {&mr0, &mr1, &ma, &ma};
    for (int k = 0; k < 4; ++k)
        HIP_TRY(ctx, hipMemcpyAsync(P.bgm[k], mom[k]->data(), n1 * sizeof(double),
                                    hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return FCPT_OK;
}

// split storage: the backgrounds of the evolved fields move to their current
// ring means (each deviation re-expressed about the new background, rounded
// to nearest once) and the derived fields' and momenta's backgrounds follow
static int rebase_backgrounds(fcpt_ctx *ctx)
{
    const KParams &P = ctx->P;
    ctx->steps_since_rebase = 0;
    if (!P.split) return FCPT_OK;
    int rc = sync_derived(ctx);
    if (rc) return rc;
    const int state[4] = {FCPT_SIGMA, FCPT_VRAD, FCPT_VAZI, FCPT_ENERGY};
    for (int k = 0; k < (P.adiabatic ? 4 : 3); ++k) {
        const int f = state[k];
        const int rows = (int)field_rows(f, P.nr);
        std::vector<double> bg((size_t)P.nr + 2, 0.0);
        launch_split_ring_mean(P, ctx->stream, P.f[f], P.bg[f], rows, ctx->bg_tmp);
        LAUNCH_CHECK(ctx);
        HIP_TRY(ctx, hipMemcpyAsync(bg.data(), ctx->bg_tmp, (size_t)rows * sizeof(double),
                                    hipMemcpyDeviceToHost, ctx->stream));
        HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
        if ((rc = rebase_field(ctx, f, bg))) return rc;
    }
    return set_derived_backgrounds(ctx);
}

int fcpt_rebase_backgrounds(fcpt_ctx *ctx)
{
    CTX_CHECK(ctx);
    return rebase_backgrounds(ctx);
}

// copy_initial_values (damping.cpp:301-309): the damping references take the
// current fields (split storage: with their backgrounds)
static int copy_initial_values(fcpt_ctx *ctx)
{
    const KParams &P = ctx->P;
    const int pairs[4][2] = {{FCPT_SIGMA, FCPT_SIGMA0}, {FCPT_VRAD, FCPT_VRAD0},
                             {FCPT_VAZI, FCPT_VAZI0}, {FCPT_ENERGY, FCPT_ENERGY0}};
    for (const auto &pr : pairs) {
        const size_t bytes = field_rows(pr[0], P.nr) * P.ns * element_size(P);
        HIP_TRY(ctx, hipMemcpyAsync(P.f[pr[1]], P.f[pr[0]], bytes, hipMemcpyDeviceToDevice, ctx->stream));
        if (P.split) {
            ctx->hbg[pr[1]] = ctx->hbg[pr[0]];
            HIP_TRY(ctx, hipMemcpyAsync(P.bg[pr[1]], P.bg[pr[0]], ((size_t)P.nr + 2) * sizeof(double),
                                        hipMemcpyDeviceToDevice, ctx->stream));
        }
    }
    return FCPT_OK;
}

int fcpt_init_profiles(fcpt_ctx *ctx, const fcpt_ic_desc *ic)
{
    CTX_SYNCED(ctx);
    if (!ic) return fail(ctx, FCPT_ERR_ARG, "null initial-condition description");
    const KParams &P = ctx->P;
    const int nr = P.nr, ns = P.ns;
    const DiskProfile prof{ctx->desc, *ic};
    // ring profiles, O(nr) on the host
    std::vector<double> sig((size_t)nr + 2, 0.0), en((size_t)nr + 2, 0.0), vr((size_t)nr + 2, 0.0),
        vaz((size_t)nr + 2, 0.0), zero((size_t)nr + 2, 0.0);
    for (int i = 0; i < nr; ++i) {
        sig[i] = prof.sigma_cell(ctx->Rmed[i]);
        if (P.adiabatic) en[i] = DiskProfile::max_(prof.energy(ctx->Rmed[i]), prof.energy_floor(sig[i]));
    }
    // SigmaMed and SigmaInf (compute_azi_avg_Sigma, Theo.cpp:30-48): the ring
    // sum of nphi equal values, in order, divided by nphi
    std::vector<double> smed((size_t)nr, 0.0), sinf((size_t)nr, 0.0);
    for (int i = 0; i < nr; ++i) {
        double m = 0.0;
        for (int j = 0; j < ns; ++j) m += sig[i];
        smed[i] = m / (double)ns;
    }
    sinf[0] = smed[0];
    for (int i = 1; i < nr; ++i) {
        const double dr = ctx->Rmed[i] - ctx->Rmed[i - 1];
        sinf[i] = (smed[i - 1] * (ctx->Rmed[i] - ctx->Rinf[i]) + smed[i] * (ctx->Rinf[i] - ctx->Rmed[i - 1])) / dr;
    }
    for (int i = 0; i < nr; ++i) {
        const double r = ctx->Rmed[i], ri = ctx->Rinf[i];
        double v = prof.vphi(r);
        v -= P.omega_frame * r;
        vaz[i] = v;
        double u = ic->imposed_disk_drift * P.sigma0 / sinf[i] / ri;
        if (!ic->vradial_zero) u += prof.vr_viscous(ri);
        else u = 0.0;
        vr[i] = u;
    }
    // the rings on the device (one allocation per call, freed at the end)
    double *d_rings = nullptr;
    const size_t n1 = (size_t)nr + 2;
    HIP_TRY(ctx, hipMalloc(&d_rings, 5 * n1 * sizeof(double)));
    double *d_sig = d_rings, *d_en = d_rings + n1, *d_vr = d_rings + 2 * n1, *d_vaz = d_rings + 3 * n1,
           *d_zero = d_rings + 4 * n1;
    int rc = FCPT_OK;
    auto up = [&](double *dst, const std::vector<double> &src) {
        if (!rc && hipMemcpyAsync(dst, src.data(), n1 * sizeof(double), hipMemcpyHostToDevice, ctx->stream) != hipSuccess)
            rc = fail(ctx, FCPT_ERR_DEVICE, "ring profile upload");
    };
    up(d_sig, sig);
    up(d_en, en);
    up(d_vr, vr);
    up(d_vaz, vaz);
    up(d_zero, zero);
    // split storage: each field's background is its ring profile, so every
    // deviation is zero (the velocities' background is zero while init_euler
    // runs, then their profiles)
    auto fill = [&](int f, const std::vector<double> &ring, const double *d_ring, int rows) {
        const double *b = nullptr;
        if (P.split) {
            ctx->hbg[f] = ring;
            if (!rc && hipMemcpyAsync(P.bg[f], ring.data(), n1 * sizeof(double), hipMemcpyHostToDevice,
                                      ctx->stream) != hipSuccess)
                rc = fail(ctx, FCPT_ERR_DEVICE, "background upload");
            b = P.bg[f];
        }
        if (!rc) launch_fill_rows(P, ctx->stream, P.f[f], d_ring, b, rows);
    };
    fill(FCPT_SIGMA, sig, d_sig, nr);
    fill(FCPT_ENERGY, en, d_en, nr);
    // init_euler runs while the velocities are still zero (init.cpp:331-332)
    fill(FCPT_VRAD, zero, d_zero, nr + 1);
    fill(FCPT_VAZI, zero, d_zero, nr);
    if (!rc && P.split) rc = set_derived_backgrounds(ctx);
    if (!rc) {
        if (!P.adiabatic) {
            launch_iso_profile(P, ctx->stream);
            launch_recalc_viscosity(P, ctx->stream);
        } else {
            launch_derived(P, ctx->stream);
            launch_recalc_viscosity(P, ctx->stream);
            launch_stress(P, ctx->stream);
            launch_heatcool_cfl(P, ctx->stream);
        }
    }
    fill(FCPT_VRAD, vr, d_vr, nr + 1);
    fill(FCPT_VAZI, vaz, d_vaz, nr);
    if (!rc && P.split) rc = set_derived_backgrounds(ctx);
    if (!rc) rc = copy_initial_values(ctx);
    if (!rc) launch_boundaries(P, ctx->stream, 0, 0);
    if (!rc) rc = copy_initial_values(ctx);
    const hipError_t le = hipGetLastError();
    const hipError_t se = hipStreamSynchronize(ctx->stream);
    hipFree(d_rings);
    if (rc) return rc;
    if (le != hipSuccess) return fail(ctx, FCPT_ERR_DEVICE, "launch: %s", hipGetErrorString(le));
    if (se != hipSuccess) return fail(ctx, FCPT_ERR_DEVICE, "sync: %s", hipGetErrorString(se));
    ctx->derived_own = true;
    return FCPT_OK;
}

int fcpt_upload_reference(fcpt_ctx *ctx, const double *sigma0, const double *vrad0,
                          const double *vazi0, const double *energy0)
{
    int rc;
    if ((rc = fcpt_upload_field(ctx, FCPT_SIGMA0, sigma0))) return rc;
    if ((rc = fcpt_upload_field(ctx, FCPT_VRAD0, vrad0))) return rc;
    if ((rc = fcpt_upload_field(ctx, FCPT_VAZI0, vazi0))) return rc;
    if (energy0) return fcpt_upload_field(ctx, FCPT_ENERGY0, energy0);
    return FCPT_OK;
}

int fcpt_upload_state(fcpt_ctx *ctx, const double *sigma, const double *vrad, const double *vazi,
                      const double *energy)
{
    int rc;
    if ((rc = fcpt_upload_field(ctx, FCPT_SIGMA, sigma))) return rc;
    if ((rc = fcpt_upload_field(ctx, FCPT_VRAD, vrad))) return rc;
    if ((rc = fcpt_upload_field(ctx, FCPT_VAZI, vazi))) return rc;
    if (energy && (rc = fcpt_upload_field(ctx, FCPT_ENERGY, energy))) return rc;
    if (ctx->P.adiabatic && !energy) return fail(ctx, FCPT_ERR_ARG, "adiabatic disk needs energy");
    if (ctx->P.split && (rc = set_derived_backgrounds(ctx))) return rc;
    // init_euler recalculation (SourceEuler.cpp:264-284)
    const KParams &P = ctx->P;
    if (!P.adiabatic) {
        launch_iso_profile(P, ctx->stream);
        launch_recalc_viscosity(P, ctx->stream);
    } else {
        launch_derived(P, ctx->stream);
        // compute_heating_cooling_for_CFL (SourceEuler.cpp:1410-1450)
        launch_recalc_viscosity(P, ctx->stream);
        launch_stress(P, ctx->stream);
        launch_heatcool_cfl(P, ctx->stream);
    }
    LAUNCH_CHECK(ctx);
    ctx->derived_own = true;
    if ((rc = clear_error_flags(ctx))) return rc;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return FCPT_OK;
}

int fcpt_download_state(fcpt_ctx *ctx, double *sigma, double *vrad, double *vazi, double *energy)
{
    CTX_CHECK(ctx);
    HostCopies fields;
    double *const dst[4] = {sigma, vrad, vazi, energy};
    const int f[4] = {FCPT_SIGMA, FCPT_VRAD, FCPT_VAZI, FCPT_ENERGY};
    for (int k = 0; k < 4; ++k)
        if (dst[k]) fields.add(f[k], dst[k]);
    return fields.n == 0 ? FCPT_OK : copy_to_host(ctx, fields);
}

int fcpt_set_time(fcpt_ctx *ctx, double time, double last_dt, int32_t n_monitor)
{
    CTX_CHECK(ctx);
    launch_set_time(ctx->P, ctx->stream, time, last_dt, n_monitor);
    LAUNCH_CHECK(ctx);
    return clear_error_flags(ctx);
}

int fcpt_get_time(fcpt_ctx *ctx, double *time, double *last_dt, int32_t *n_monitor)
{
    CTX_CHECK(ctx);
    int rc = read_scalars(ctx);
    if (rc) return rc;
    if (time) *time = ctx->s_host->time;
    if (last_dt) *last_dt = ctx->s_host->last_dt;
    if (n_monitor) *n_monitor = ctx->s_host->n_monitor;
    return FCPT_OK;
}

// compute_smoothing (Force.cpp:145-159) per body, on the host with the
// reference's expressions (compute_smoothing_iso_planet :132-142, the body's
// r = hypot(x, y) as planet.cpp:159 keeps it); < 0 marks the default,
// ThicknessSmoothing times the scale height of the cell
static BodySmoothing body_smoothing(const fcpt_ctx *ctx, const fcpt_step_params &sp)
{
    BodySmoothing b{};
    const fcpt_disk_desc &d = ctx->desc;
    for (int k = 0; k < kMaxPlanets; ++k) {
        b.s[k] = -1.0;
        if (k >= sp.n_planets) continue;
        if ((d.potential_smoothing & FCPT_SMOOTHING_NO_STAR) && k == 0) {
            b.s[k] = 0;
        } else if (d.potential_smoothing & FCPT_SMOOTHING_PLANETLOC) {
            const double a = std::hypot(sp.planet[k].x, sp.planet[k].y);
            const double scale_height = d.aspect_ratio * std::pow(a, 1 + d.flaring_index);
            b.s[k] = d.thickness_smoothing * scale_height;
        }
    }
    return b;
}

int fcpt_set_step_params(fcpt_ctx *ctx, const fcpt_step_params *params)
{
    CTX_CHECK(ctx);
    if (!params || params->n_planets < 0 || params->n_planets > FCPT_MAX_PLANETS)
        return fail(ctx, FCPT_ERR_ARG, "bad step parameters");
    launch_set_params(ctx->P, ctx->stream, *params, body_smoothing(ctx, *params));
    LAUNCH_CHECK(ctx);
    return FCPT_OK;
}

static int cfl_common(fcpt_ctx *ctx, int mode, double *dt_out)
{
    CTX_SYNCED(ctx);
    launch_cfl(ctx->P, ctx->stream, mode);
    LAUNCH_CHECK(ctx);
    int rc = read_scalars(ctx);
    if (rc) return rc;
    if (take_nonfinite(ctx))
        return fail(ctx, FCPT_ERR_NONFINITE, "CFL time step is not finite and positive (%g)",
                    ctx->s_host->cfl_dt);
    if (dt_out) *dt_out = ctx->s_host->cfl_dt;
    return FCPT_OK;
}

int fcpt_condition_cfl(fcpt_ctx *ctx, double *dt_out) { return cfl_common(ctx, 0, dt_out); }
int fcpt_calculate_timestep(fcpt_ctx *ctx, double *dt_out) { return cfl_common(ctx, 1, dt_out); }

int fcpt_nbody_potential(fcpt_ctx *ctx)
{
    CTX_SYNCED(ctx);
    launch_potential(ctx->P, ctx->stream);
    LAUNCH_CHECK(ctx);
    return FCPT_OK;
}

#define DT_ENTRY(name, body)                         \
    int name(fcpt_ctx *ctx, double dt)               \
    {                                                \
        CTX_SYNCED(ctx);                             \
        launch_set_dt(ctx->P, ctx->stream, dt);      \
        body;                                        \
        LAUNCH_CHECK(ctx);                           \
        return FCPT_OK;                              \
    }

DT_ENTRY(fcpt_update_with_sourceterms, launch_sources(ctx->P, ctx->stream); ctx->derived_own = false)
DT_ENTRY(fcpt_artificial_viscosity, launch_artificial_viscosity(ctx->P, ctx->stream, 0); ctx->derived_own = false)
DT_ENTRY(fcpt_update_velocities_with_viscosity, launch_visc_update(ctx->P, ctx->stream))
DT_ENTRY(fcpt_transport, launch_transport(ctx->P, ctx->stream); ctx->derived_own = false)

int fcpt_recalculate_viscosity(fcpt_ctx *ctx)
{
    CTX_SYNCED(ctx);
    launch_recalc_viscosity(ctx->P, ctx->stream);
    LAUNCH_CHECK(ctx);
    return FCPT_OK;
}

int fcpt_viscous_stress_tensor(fcpt_ctx *ctx)
{
    CTX_SYNCED(ctx);
    launch_stress(ctx->P, ctx->stream);
    LAUNCH_CHECK(ctx);
    return FCPT_OK;
}

int fcpt_substep3(fcpt_ctx *ctx, double time, double dt)
{
    CTX_SYNCED(ctx);
    if (!ctx->P.adiabatic) return FCPT_OK;
    launch_set_clock(ctx->P, ctx->stream, time);
    launch_set_dt(ctx->P, ctx->stream, dt);
    launch_substep3(ctx->P, ctx->stream);
    ctx->derived_own = false;
    LAUNCH_CHECK(ctx);
    return FCPT_OK;
}

int fcpt_apply_boundary_condition(fcpt_ctx *ctx, double dt, int32_t final_call)
{
    CTX_SYNCED(ctx);
    launch_set_dt(ctx->P, ctx->stream, dt);
    launch_boundaries(ctx->P, ctx->stream, final_call, 0);
    // the damping changes E and Sigma of rings whose derived fields the step
    // reads; those of the ghost rings it does not
    if (final_call && ctx->P.damping) ctx->derived_own = false;
    LAUNCH_CHECK(ctx);
    return FCPT_OK;
}

int fcpt_recalculate_derived(fcpt_ctx *ctx)
{
    CTX_SYNCED(ctx);
    launch_derived(ctx->P, ctx->stream);
    ctx->derived_own = true;
    LAUNCH_CHECK(ctx);
    return FCPT_OK;
}

int fcpt_get_nshift(fcpt_ctx *ctx, int32_t *nshift)
{
    CTX_CHECK(ctx);
    if (!nshift) return fail(ctx, FCPT_ERR_ARG, "null output");
    HIP_TRY(ctx, hipMemcpyAsync(nshift, ctx->P.nshift, sizeof(int32_t) * ctx->P.nr,
                                hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    return FCPT_OK;
}

// the gas part of step_Euler (simulation.cpp:148-267); dt already in device memory
// The source part of a step (potential, sources, artificial viscosity,
// viscosity recalculation, viscous stress and update, SubStep3) with the dt
// and time in device memory.  The fused form runs the source terms, the
// artificial viscosity and the viscous stress + update as one pass each; each
// pass writes the velocities to the partner buffers, so the passes alternate
// between the two views of the state (P and its swapped view).  Returns the
// view that holds the velocities afterwards.  fold_mode >= 0 (fused only):
// the potential launch also folds the CFL minima of launch_cfl_cells.
static const KParams *enqueue_kick(const KParams &P, const KParams &Q, hipStream_t st, bool fused,
                                   bool pressure_first, int fold_mode = -1)
{
    if (P.lazy_derived) {
        // the potential pass and one walk, which forms the pressure itself
        launch_kick(P, st, fold_mode);
        return &Q;
    }
    if (fused) launch_potential_fold(P, st, fold_mode);
    else launch_potential(P, st);
    if (!fused) {
        if (pressure_first) launch_pressure(P, st);
        launch_sources(P, st);
        if (!launch_artificial_viscosity(P, st, 1)) launch_recalc_viscosity(P, st);
        launch_stress(P, st);
        launch_visc_update(P, st);
        if (P.adiabatic) launch_substep3(P, st);
        return &P;
    }
    const KParams *cur = &P, *other = &Q;
    auto flip = [&]() { std::swap(cur, other); };
    // the isothermal fused source pass forms the pressure from Sigma itself
    if (pressure_first && P.adiabatic) launch_pressure(P, st);
    launch_src_fused(*cur, st);
    flip();
    if (P.adiabatic) launch_src_energy(*cur, st);
    if (P.artvisc == FCPT_ARTVISC_TW || P.artvisc == FCPT_ARTVISC_SN) {
        launch_av_fused(*cur, st, 1);
        flip();
    } else {
        launch_artificial_viscosity(*cur, st, 1);  // temperature floor only
        launch_recalc_viscosity(*cur, st);
    }
    if (P.adiabatic) launch_visc_energy(*cur, st);
    else launch_visc_fused(*cur, st);
    flip();
    return cur;
}

// One gas step of step_Euler; the transport's velocity kernel writes the
// final velocities to the fields of view P and, in the fused step, applies
// the damping of the final boundary call that follows it.
static void enqueue_euler(const KParams &P, hipStream_t st, int count_monitor, bool fused, int fold_mode)
{
    const KParams Q = swapped_view(P);
    const KParams *cur = enqueue_kick(P, Q, st, fused, false, fused ? fold_mode : -1);
    if (fused) {
        // the transport's velocity kernel also runs the final boundary call
        // and the derived fields
        launch_transport_ghost(*cur, P, st, count_monitor ? 2 : 1);
    } else {
        launch_boundaries(*cur, st, 0, 0);
        launch_transport_to(*cur, P, st);
        launch_final_boundaries_derived(P, st, count_monitor ? 2 : 1);
    }
}

// One gas step of step_LeapFrog (simulation.cpp:276-459): kick with dt / 2,
// boundaries and transport over dt, kick with dt / 2 at the midstep time and
// bodies (compute_pressure first), final boundaries over dt, derived fields.
// The isothermal unfused path needs the pressure of the transported Sigma,
// as does the adiabatic one of the transported E.
static void enqueue_leapfrog(const KParams &P, hipStream_t st, int count_monitor, bool fused, int fold_mode)
{
    const KParams Q = swapped_view(P);
    if (P.lazy_derived) {
        // the walks take their half steps from KParams::kick, so the clock
        // needs no launches of its own
        KParams K = P;
        K.kick = 1;
        launch_kick(K, st, fold_mode);
        launch_transport_ghost(Q, P, st, 0);
        K.kick = 2;
        K.fold_in_kick = 0;
        launch_kick(K, st, -1);
        launch_final_leapfrog(P, st, count_monitor ? 2 : 1);
        return;
    }
    launch_leapfrog_phase(P, st, 0);
    const KParams *cur = enqueue_kick(P, Q, st, fused, false);
    launch_leapfrog_phase(P, st, 1);
    if (fused) {
        launch_transport_ghost(*cur, P, st, 0);
    } else {
        launch_boundaries(*cur, st, 0, 0);
        launch_transport_to(*cur, P, st);
    }
    launch_leapfrog_phase(P, st, 2);
    cur = enqueue_kick(P, Q, st, fused, true);
    if (cur != &P) {
        // an odd number of fused passes: the velocities go back to the fields
        launch_copy_velocities(*cur, st);
    }
    launch_leapfrog_phase(P, st, 3);
    launch_final_boundaries_derived(P, st, count_monitor ? 2 : 1);
}

static void enqueue_step(const KParams &P, hipStream_t st, int count_monitor, bool fused)
{
    if (P.integrator == FCPT_INTEGRATOR_LEAPFROG) enqueue_leapfrog(P, st, count_monitor, fused, -1);
    else enqueue_euler(P, st, count_monitor, fused, -1);
}

// one sim::run iteration: CalculateTimeStep with the monitor clip (mode 2),
// then the step; the fused Euler step folds the CFL minima inside its
// potential launch (one launch less)
// `report`: the step's clock goes to the pinned mirror as well
static void enqueue_iteration(const fcpt_ctx *ctx, KParams V, bool report = false)
{
    if (report) V.s_out = ctx->s_host;
    const bool leapfrog = V.integrator == FCPT_INTEGRATOR_LEAPFROG;
    if (V.lazy_derived || (ctx->fused && !leapfrog)) {
        if (V.cfl_pot) launch_cfl_potential(V, ctx->stream);
        else launch_cfl_cells(V, ctx->stream);
        V.fold_in_kick = fold_in_kick(V);
        const int fold_mode = V.cfl_pot ? kFoldDone : 2;
        if (leapfrog) enqueue_leapfrog(V, ctx->stream, 1, true, fold_mode);
        else enqueue_euler(V, ctx->stream, 1, true, fold_mode);
    } else {
        launch_cfl(V, ctx->stream, 2);
        enqueue_step(V, ctx->stream, 1, ctx->fused);
    }
}

int fcpt_step_euler(fcpt_ctx *ctx, double dt)
{
    CTX_SYNCED(ctx);
    launch_set_dt(ctx->P, ctx->stream, dt);
    const KParams V = step_view(ctx, reads_stored(ctx));
    enqueue_euler(V, ctx->stream, 0, ctx->fused, -1);
    LAUNCH_CHECK(ctx);
    stepped(ctx, V);
    return FCPT_OK;
}

int fcpt_step_leapfrog(fcpt_ctx *ctx, double dt)
{
    CTX_SYNCED(ctx);
    launch_set_dt(ctx->P, ctx->stream, dt);
    KParams V = ctx->P;
    V.integrator = FCPT_INTEGRATOR_LEAPFROG;  // the scheme, whatever the descriptor's own
    set_step_modes(V, ctx->fused && !reads_stored(ctx));
    enqueue_leapfrog(V, ctx->stream, 0, ctx->fused, -1);
    LAUNCH_CHECK(ctx);
    stepped(ctx, V);
    return FCPT_OK;
}

int fcpt_compute_pressure(fcpt_ctx *ctx)
{
    CTX_SYNCED(ctx);
    launch_pressure(ctx->P, ctx->stream);
    LAUNCH_CHECK(ctx);
    return FCPT_OK;
}

int fcpt_set_midstep_params(fcpt_ctx *ctx, const fcpt_step_params *params)
{
    CTX_CHECK(ctx);
    if (!params || params->n_planets < 0 || params->n_planets > FCPT_MAX_PLANETS)
        return fail(ctx, FCPT_ERR_ARG, "bad step parameters");
    launch_set_mid_params(ctx->P, ctx->stream, *params, body_smoothing(ctx, *params));
    LAUNCH_CHECK(ctx);
    return FCPT_OK;
}

int fcpt_run_step(fcpt_ctx *ctx, double *dt_out)
{
    CTX_CHECK(ctx);
    const KParams V = step_view(ctx, reads_stored(ctx));
    if (const int rc = sync_for(ctx, V)) return rc;
    enqueue_iteration(ctx, V, true);
    LAUNCH_CHECK(ctx);
    stepped(ctx, V);
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    if (take_nonfinite(ctx))
        return fail(ctx, FCPT_ERR_NONFINITE, "CFL time step is not finite and positive");
    if (dt_out) *dt_out = ctx->s_host->dt;
    return FCPT_OK;
}

// capture one iteration, or kGraphSteps of them (`many`), into a graph (each
// once per context)
static int ensure_step_graph(fcpt_ctx *ctx, bool many)
{
    hipGraphExec_t &exec = ctx->step_graph[many ? 1 : 0];
    if (exec) return FCPT_OK;
    hipGraph_t g = nullptr;
    HIP_TRY(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    for (int k = 0; k < (many ? kGraphSteps : 1); ++k) enqueue_iteration(ctx, step_view(ctx));
    hipError_t e = hipStreamEndCapture(ctx->stream, &g);
    if (e != hipSuccess) return fail(ctx, FCPT_ERR_DEVICE, "graph capture: %s", hipGetErrorString(e));
    e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    hipGraphDestroy(g);
    if (e != hipSuccess) {
        exec = nullptr;
        return fail(ctx, FCPT_ERR_DEVICE, "graph instantiate: %s", hipGetErrorString(e));
    }
    return FCPT_OK;
}

// split storage with a rebase interval: the steps before the next background move
static bool periodic_rebase(const fcpt_ctx *ctx) { return ctx->P.split && ctx->rebase_interval > 0; }

int fcpt_run_steps(fcpt_ctx *ctx, int32_t n_steps, int32_t use_graph)
{
    CTX_CHECK(ctx);
    if (n_steps < 0) return fail(ctx, FCPT_ERR_ARG, "negative step count");
    // calls of kGraphSteps or more replay that many per graph and launch the
    // rest one by one; shorter ones replay single iterations
    const bool many = n_steps >= kGraphSteps;
    if (use_graph) {
        int rc = ensure_step_graph(ctx, many);
        if (rc) return rc;
    }
    for (int left = n_steps; left > 0;) {
        int m = left;
        if (periodic_rebase(ctx)) m = std::min(m, ctx->rebase_interval - ctx->steps_since_rebase);
        const bool stored = reads_stored(ctx);
        if (stored) m = 1;  // one step, then as captured
        const KParams V = step_view(ctx, stored);
        if (const int rc = sync_for(ctx, V)) return rc;
        int k = 0;
        if (use_graph && !stored) {
            const int per = many ? kGraphSteps : 1;
            for (; k + per <= m; k += per) HIP_TRY(ctx, hipGraphLaunch(ctx->step_graph[many ? 1 : 0], ctx->stream));
        }
        for (; k < m; ++k) enqueue_iteration(ctx, V);
        LAUNCH_CHECK(ctx);
        left -= m;
        stepped(ctx, V);
        if (periodic_rebase(ctx) && (ctx->steps_since_rebase += m) >= ctx->rebase_interval) {
            const int rc = rebase_backgrounds(ctx);
            if (rc) return rc;
        }
    }
    return FCPT_OK;
}

static int ensure_events(fcpt_ctx *ctx)
{
    if (!ctx->ev0) HIP_TRY(ctx, hipEventCreate(&ctx->ev0));
    if (!ctx->ev1) HIP_TRY(ctx, hipEventCreate(&ctx->ev1));
    return FCPT_OK;
}

int fcpt_time_steps(fcpt_ctx *ctx, int32_t n_steps, int32_t use_graph, double *ms_total)
{
    CTX_CHECK(ctx);
    int rc = ensure_events(ctx);
    if (!rc && use_graph) rc = ensure_step_graph(ctx, n_steps >= kGraphSteps);
    if (rc) return rc;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    HIP_TRY(ctx, hipEventRecord(ctx->ev0, ctx->stream));
    rc = fcpt_run_steps(ctx, n_steps, use_graph);
    if (rc) return rc;
    HIP_TRY(ctx, hipEventRecord(ctx->ev1, ctx->stream));
    HIP_TRY(ctx, hipEventSynchronize(ctx->ev1));
    float ms = 0.f;
    HIP_TRY(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    rc = read_scalars(ctx);
    if (rc) return rc;
    if (take_nonfinite(ctx))
        return fail(ctx, FCPT_ERR_NONFINITE, "CFL time step became non-finite during the run");
    if (ms_total) *ms_total = (double)ms;
    return FCPT_OK;
}

int fcpt_time_kernel(fcpt_ctx *ctx, int32_t kernel, int32_t reps, double *ms_per_launch)
{
    CTX_SYNCED(ctx);
    if (reps <= 0) return fail(ctx, FCPT_ERR_ARG, "reps must be positive");
    int rc = ensure_events(ctx);
    if (rc) return rc;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    ForceBodies fb{};
    fb.n = 2;
    fb.flags = FCPT_FORCE_CORRECT_SELFGRAVITY;
    fb.x[1] = fb.r[1] = 1.0;
    fb.smooth_fixed[0] = fb.smooth_fixed[1] = -1.0;
    auto one = [&]() {
        switch (kernel) {
        case FCPT_KERNEL_DISK_FORCE:
            launch_disk_force(ctx->P, ctx->stream, fb, ctx->force_part, ctx->force_host);
            break;
        case FCPT_KERNEL_RADIAL_SWEEP:  // one kernel runs both sweeps
        case FCPT_KERNEL_AZIMUTHAL: launch_sweeps(ctx->P, ctx->stream); break;
        case FCPT_KERNEL_CFL: launch_cfl_cells(ctx->P, ctx->stream); break;
        case FCPT_KERNEL_STRESS: launch_stress(ctx->P, ctx->stream); break;
        case FCPT_KERNEL_POTENTIAL: launch_potential(ctx->P, ctx->stream); break;
        case FCPT_KERNEL_VISC_FUSED: launch_visc_fused(ctx->P, ctx->stream); break;
        default: break;
        }
    };
    if (kernel < 0 || kernel > FCPT_KERNEL_VISC_FUSED || kernel == 2)
        return fail(ctx, FCPT_ERR_ARG, "unknown kernel");
    one();  // warm-up
    HIP_TRY(ctx, hipEventRecord(ctx->ev0, ctx->stream));
    for (int k = 0; k < reps; ++k) one();
    HIP_TRY(ctx, hipEventRecord(ctx->ev1, ctx->stream));
    LAUNCH_CHECK(ctx);
    HIP_TRY(ctx, hipEventSynchronize(ctx->ev1));
    float ms = 0.f;
    HIP_TRY(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    if (ms_per_launch) *ms_per_launch = (double)ms / reps;
    return FCPT_OK;
}

int fcpt_time_copy(fcpt_ctx *ctx, int32_t reps, double *ms_per_launch, double *bytes_per_launch)
{
    CTX_CHECK(ctx);
    if (reps <= 0) return fail(ctx, FCPT_ERR_ARG, "reps must be positive");
    int rc = ensure_events(ctx);
    if (rc) return rc;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    launch_copy4(ctx->P, ctx->stream);
    HIP_TRY(ctx, hipEventRecord(ctx->ev0, ctx->stream));
    for (int k = 0; k < reps; ++k) launch_copy4(ctx->P, ctx->stream);
    HIP_TRY(ctx, hipEventRecord(ctx->ev1, ctx->stream));
    LAUNCH_CHECK(ctx);
    HIP_TRY(ctx, hipEventSynchronize(ctx->ev1));
    float ms = 0.f;
    HIP_TRY(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    if (ms_per_launch) *ms_per_launch = (double)ms / reps;
    if (bytes_per_launch)
        *bytes_per_launch = 2.0 * 4.0 * (double)((size_t)ctx->P.nr * ctx->P.ns * element_size(ctx->P) / 8 * 8);
    return FCPT_OK;
}

int fcpt_set_launch_param(fcpt_ctx *ctx, int32_t param, int32_t value)
{
    CTX_CHECK(ctx);
    if (param == FCPT_PARAM_RADIAL_TILE) {
        if (value < 0 || value > 64) return fail(ctx, FCPT_ERR_ARG, "radial tile must be 0 .. 64");
    } else if (param == FCPT_PARAM_RADIAL_WAVES) {
        if (value != 2 && value != 3) return fail(ctx, FCPT_ERR_ARG, "radial waves must be 2 or 3");
    } else if (param == FCPT_PARAM_FUSED_STEP) {
        if (value != 0 && value != 1) return fail(ctx, FCPT_ERR_ARG, "fused step must be 0 or 1");
    } else if (param == FCPT_PARAM_VISC_TILE) {
        if (value < 0 || value > 64) return fail(ctx, FCPT_ERR_ARG, "viscous tile must be 0 .. 64");
    } else if (param == FCPT_PARAM_KICK_TILE) {
        if (value < 0 || value > 64) return fail(ctx, FCPT_ERR_ARG, "kick tile must be 0 .. 64");
    } else if (param == FCPT_PARAM_SPLIT_ROUNDING) {
        if (value < 0 || value > 2) return fail(ctx, FCPT_ERR_ARG, "split rounding must be 0, 1 or 2");
    } else if (param == FCPT_PARAM_REBASE_INTERVAL) {
        if (value < 0) return fail(ctx, FCPT_ERR_ARG, "rebase interval must be 0 or positive");
        ctx->rebase_interval = ctx->P.split ? value : 0;
        ctx->steps_since_rebase = 0;
        return FCPT_OK;
    } else {
        return fail(ctx, FCPT_ERR_ARG, "unknown launch parameter");
    }
    // stale fields as the steps that left them would have stored them
    if (const int rc = sync_derived(ctx)) return rc;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    if (param == FCPT_PARAM_RADIAL_TILE) ctx->P.radial_tile = value;
    else if (param == FCPT_PARAM_RADIAL_WAVES) ctx->P.radial_waves = value;
    else if (param == FCPT_PARAM_VISC_TILE) ctx->P.visc_tile = value;
    else if (param == FCPT_PARAM_KICK_TILE) ctx->P.kick_tile = value;
    else if (param == FCPT_PARAM_SPLIT_ROUNDING) {
        const int mode = ctx->P.split ? value : 0;
        if (mode != ctx->P.split_rounding) ctx->derived_own = false;  // stored as the old mode rounds
        ctx->P.split_rounding = mode;
    }
    else ctx->fused = value != 0;
    HIP_TRY(ctx, drop_graphs(ctx->step_graph));
    return FCPT_OK;
}

// The kick walk's tile (the viscous walk's in a disk without artificial
// viscosity) by whole-step time: each candidate runs `reps` graph-replayed
// sim::run iterations from the same state, which is saved first (every field
// and the device scalars) and put back after each trial and at the end, so
// the context's state and clock come out as they went in.  Tiles 2 .. 32.
int fcpt_autotune_walks(fcpt_ctx *ctx, int32_t reps, int32_t *kick_tile, int32_t *visc_tile)
{
    CTX_SYNCED(ctx);
    if (reps <= 0) return fail(ctx, FCPT_ERR_ARG, "reps must be positive");
    int rc = ensure_events(ctx);
    if (rc) return rc;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    KParams &P = ctx->P;
    const int kick0 = resolve_kick_tile(P), visc0 = resolve_visc_tile(P);
    const bool kv = walks_tunable(P);
    if (!ctx->fused || P.integrator != FCPT_INTEGRATOR_EULER ||
        !(kv || (P.artvisc == FCPT_ARTVISC_NONE && visc0 > 1))) {
        if (kick_tile) *kick_tile = kick0;
        if (visc_tile) *visc_tile = visc0;
        return FCPT_OK;  // the walks do not run in this context's step
    }
    // the trials' steps neither move the split backgrounds (the saved
    // deviations go back about the same backgrounds) nor count toward the next move
    struct RebaseHold {
        fcpt_ctx *c;
        int interval, since;
        ~RebaseHold()
        {
            c->rebase_interval = interval;
            c->steps_since_rebase = since;
        }
    } hold{ctx, ctx->rebase_interval, ctx->steps_since_rebase};
    ctx->rebase_interval = 0;
    // the saved state: every field and the scalars
    size_t total = 0;
    std::vector<size_t> off(FCPT_NUM_FIELDS);
    for (int k = 0; k < FCPT_NUM_FIELDS; ++k) {
        off[k] = total;
        total += (field_rows(k, P.nr) * P.ns * field_element_size(P, k) + 255) / 256 * 256;
    }
    const bool own = ctx->derived_own;
    char *save = nullptr;
    HIP_TRY(ctx, hipMalloc((void **)&save, total));
    DevScalars s0;
    auto copy_fields = [&](bool to_save) -> hipError_t {
        for (int k = 0; k < FCPT_NUM_FIELDS; ++k) {
            const size_t bytes = field_rows(k, P.nr) * P.ns * field_element_size(P, k);
            hipError_t e = to_save ? hipMemcpyAsync(save + off[k], P.f[k], bytes, hipMemcpyDeviceToDevice, ctx->stream)
                                   : hipMemcpyAsync(P.f[k], save + off[k], bytes, hipMemcpyDeviceToDevice, ctx->stream);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    };
    auto restore = [&]() -> hipError_t {
        hipError_t e = copy_fields(false);
        if (e == hipSuccess) e = hipMemcpyAsync(ctx->s_dev, &s0, sizeof(DevScalars), hipMemcpyHostToDevice, ctx->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
        ctx->derived_stale = ctx->h_stale = false;
        ctx->derived_own = own;
        return e;
    };
    hipError_t e = copy_fields(true);
    if (e == hipSuccess) e = hipMemcpy(&s0, ctx->s_dev, sizeof(DevScalars), hipMemcpyDeviceToHost);
    auto trial = [&](double &ms_out) -> int {
        drop_graphs(ctx->step_graph);
        int r = fcpt_run_steps(ctx, 1, 1);  // capture + warm-up
        if (!r) r = fcpt_time_steps(ctx, reps, 1, &ms_out);
        const hipError_t er = restore();
        if (!r && er != hipSuccess) r = fail(ctx, FCPT_ERR_DEVICE, "state restore: %s", hipGetErrorString(er));
        return r;
    };
    const int cand[] = {2, 4, 8, 16, 32};
    int best_t = visc0;
    rc = e == hipSuccess ? FCPT_OK : fail(ctx, FCPT_ERR_DEVICE, "state save: %s", hipGetErrorString(e));
    double best = 1e300;
    for (int t : cand) {
        if (rc || t > P.nr) continue;
        if (kv) P.kick_tile = t;
        P.visc_tile = t;
        double ms = 0.0;
        if ((rc = trial(ms))) break;
        if (ms < best) {
            best = ms;
            best_t = t;
        }
    }
    if (kv) P.kick_tile = best_t;
    P.visc_tile = best_t;
    hipFree(save);
    drop_graphs(ctx->step_graph);
    if (rc) return rc;
    if (kick_tile) *kick_tile = resolve_kick_tile(P);
    if (visc_tile) *visc_tile = resolve_visc_tile(P);
    return FCPT_OK;
}

int fcpt_get_launch_param(fcpt_ctx *ctx, int32_t param, int32_t *value)
{
    if (!ctx || !value) return FCPT_ERR_ARG;
    const KParams &P = ctx->P;
    switch (param) {
    case FCPT_PARAM_RADIAL_TILE: *value = resolve_sweep_tile(P); break;
    case FCPT_PARAM_RADIAL_WAVES: *value = P.radial_waves; break;
    case FCPT_PARAM_FUSED_STEP: *value = ctx->fused ? 1 : 0; break;
    case FCPT_PARAM_VISC_TILE: *value = resolve_visc_tile(P); break;
    case FCPT_PARAM_KICK_TILE: *value = resolve_kick_tile(P); break;
    case FCPT_PARAM_SPLIT_ROUNDING: *value = P.split_rounding; break;
    case FCPT_PARAM_REBASE_INTERVAL: *value = ctx->rebase_interval; break;
    default: return fail(ctx, FCPT_ERR_ARG, "unknown launch parameter");
    }
    return FCPT_OK;
}

int fcpt_autotune(fcpt_ctx *ctx, int32_t reps, int32_t *radial_tile, int32_t *radial_waves)
{
    CTX_SYNCED(ctx);
    if (reps <= 0) return fail(ctx, FCPT_ERR_ARG, "reps must be positive");
    int rc = ensure_events(ctx);
    if (rc) return rc;
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    KParams &P = ctx->P;
    const int tiles[] = {1, 2, 4, 8, 16, 32};
    double best = 1e300;
    int best_t = resolve_sweep_tile(P);
    for (int t : tiles) {
        if (t > P.nr) continue;
        P.radial_tile = t;
        launch_sweeps(P, ctx->stream);  // warm-up
        HIP_TRY(ctx, hipEventRecord(ctx->ev0, ctx->stream));
        for (int k = 0; k < reps; ++k) launch_sweeps(P, ctx->stream);
        HIP_TRY(ctx, hipEventRecord(ctx->ev1, ctx->stream));
        LAUNCH_CHECK(ctx);
        HIP_TRY(ctx, hipEventSynchronize(ctx->ev1));
        float ms = 0.f;
        HIP_TRY(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        if (ms < best) {
            best = ms;
            best_t = t;
        }
    }
    P.radial_tile = best_t;
    HIP_TRY(ctx, drop_graphs(ctx->step_graph));
    if (radial_tile) *radial_tile = best_t;
    if (radial_waves) *radial_waves = P.radial_waves;
    return FCPT_OK;
}

int fcpt_disk_on_planet_accel(fcpt_ctx *ctx, const fcpt_force_body *bodies, int32_t n_bodies,
                              int32_t flags, double *accel_xy)
{
    CTX_CHECK(ctx);
    if (n_bodies < 0 || n_bodies > kForceMaxBodies || (n_bodies > 0 && (!bodies || !accel_xy)))
        return fail(ctx, FCPT_ERR_ARG, "1 .. %d bodies", kForceMaxBodies);
    if (flags & ~(FCPT_FORCE_NO_STAR_SMOOTHING | FCPT_FORCE_SMOOTHING_PLANETLOC |
                  FCPT_FORCE_CORRECT_SELFGRAVITY))
        return fail(ctx, FCPT_ERR_ARG, "unknown disk-force flags");
    if (n_bodies == 0) return FCPT_OK;
    ForceBodies B{};
    B.n = n_bodies;
    B.flags = flags;
    for (int k = 0; k < n_bodies; ++k) {
        B.x[k] = bodies[k].x;
        B.y[k] = bodies[k].y;
        B.r[k] = bodies[k].r;
        B.r_cubic[k] = bodies[k].r_cubic;
        // compute_smoothing (Force.cpp:145-159): fixed per body, or thickness x H(cell)
        if ((flags & FCPT_FORCE_NO_STAR_SMOOTHING) && k == 0)
            B.smooth_fixed[k] = 0.0;
        else if (flags & FCPT_FORCE_SMOOTHING_PLANETLOC)
            B.smooth_fixed[k] = ctx->desc.thickness_smoothing *
                                (ctx->desc.aspect_ratio * std::pow(bodies[k].r, 1 + ctx->desc.flaring_index));
        else
            B.smooth_fixed[k] = -1.0;
    }
    KParams P = ctx->P;
    P.h_lazy = ctx->h_stale;
    launch_disk_force(P, ctx->stream, B, ctx->force_part, ctx->force_host);
    LAUNCH_CHECK(ctx);
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    for (int k = 0; k < n_bodies; ++k) {
        const double *o = ctx->force_host + 4 * k;
        accel_xy[2 * k] = o[0] + o[2];      // inner + outer, Force.cpp:118-119
        accel_xy[2 * k + 1] = o[1] + o[3];
    }
    return FCPT_OK;
}

// ---- snapshots -------------------------------------------------------------

// the reference's grid names (data.cpp:13-250) of the fields this library holds
static const char *const kGridName[FCPT_NUM_FIELDS] = {
    "Sigma", "vrad", "vazi", "energy", "pressure", "soundspeed", "scale_height", "viscosity",
    "potential", "q_r", "q_phi", "div_v", "tau_r_r", "tau_r_phi", "tau_phi_phi", "Qplus",
    "Qminus", "Temperature", "dens0", "vrad0", "vazi0", "energy0"};

static std::string grid_path(const char *dir, int field)
{
    return std::string(dir) + "/" + kGridName[field] + ".dat";
}

static int write_file(fcpt_ctx *ctx, const std::string &path, const void *data, size_t bytes)
{
    FILE *f = std::fopen(path.c_str(), "wb");
    if (!f) return fail(ctx, FCPT_ERR_ARG, "cannot write %s", path.c_str());
    const size_t n = bytes ? std::fwrite(data, 1, bytes, f) : 0;
    const int closed = std::fclose(f);
    if (n != bytes || closed != 0) return fail(ctx, FCPT_ERR_ARG, "short write to %s", path.c_str());
    return FCPT_OK;
}

// a whole file of exactly `bytes` bytes; 1 if it does not exist
static int read_file(fcpt_ctx *ctx, const std::string &path, void *data, size_t bytes)
{
    FILE *f = std::fopen(path.c_str(), "rb");
    if (!f) return 1;
    std::fseek(f, 0, SEEK_END);
    const long size = std::ftell(f);
    std::fseek(f, 0, SEEK_SET);
    if (size < 0 || (size_t)size != bytes) {
        std::fclose(f);
        return fail(ctx, FCPT_ERR_ARG, "%s holds %ld bytes, expected %zu", path.c_str(), size, bytes);
    }
    const size_t n = std::fread(data, 1, bytes, f);
    std::fclose(f);
    if (n != bytes) return fail(ctx, FCPT_ERR_ARG, "short read from %s", path.c_str());
    return FCPT_OK;
}

static size_t grid_doubles(const fcpt_ctx *ctx, int field)
{
    return field_rows(field, ctx->P.nr) * (size_t)ctx->P.ns;
}

int fcpt_write_snapshot(fcpt_ctx *ctx, const char *dir, const fcpt_snapshot_info *info, uint32_t fields)
{
    CTX_SYNCED(ctx);
    if (!dir || !info) return fail(ctx, FCPT_ERR_ARG, "null snapshot directory or info");
    if (fields == 0) {
        fields = (1u << FCPT_SIGMA) | (1u << FCPT_VRAD) | (1u << FCPT_VAZI) | (1u << FCPT_ENERGY);
        if (ctx->P.adiabatic) fields |= (1u << FCPT_QPLUS) | (1u << FCPT_QMINUS);
    }
    if (fields >> FCPT_NUM_FIELDS) return fail(ctx, FCPT_ERR_ARG, "unknown field in the mask");
    std::vector<double> host;
    for (int f = 0; f < FCPT_NUM_FIELDS; ++f) {
        if (!(fields & (1u << f))) continue;
        host.resize(grid_doubles(ctx, f));
        int rc = fcpt_download_field(ctx, f, host.data());
        if (!rc) rc = write_file(ctx, grid_path(dir, f), host.data(), host.size() * sizeof(double));
        if (rc) return rc;
    }
    fcpt_snapshot_info m = *info;
    double t = 0.0, last_dt = 0.0;
    int32_t n_monitor = 0;
    int rc = fcpt_get_time(ctx, &t, &last_dt, &n_monitor);
    if (rc) return rc;
    m.time = t;
    m.last_dt = last_dt;
    m.n_monitor = (uint32_t)n_monitor;
    static_assert(sizeof(fcpt_snapshot_info) == 48, "misc.bin record");
    return write_file(ctx, std::string(dir) + "/misc.bin", &m, sizeof(m));
}

int fcpt_read_snapshot(fcpt_ctx *ctx, const char *dir, fcpt_snapshot_info *info)
{
    CTX_SYNCED(ctx);
    if (!dir) return fail(ctx, FCPT_ERR_ARG, "null snapshot directory");
    fcpt_snapshot_info m{};
    int rc = read_file(ctx, std::string(dir) + "/misc.bin", &m, sizeof(m));
    if (rc == 1) return fail(ctx, FCPT_ERR_ARG, "no misc.bin in %s", dir);
    if (rc) return rc;
    const bool adi = ctx->P.adiabatic != 0;
    std::vector<double> g[4];
    const int want[4] = {FCPT_SIGMA, FCPT_VRAD, FCPT_VAZI, FCPT_ENERGY};
    for (int k = 0; k < (adi ? 4 : 3); ++k) {
        g[k].resize(grid_doubles(ctx, want[k]));
        rc = read_file(ctx, grid_path(dir, want[k]), g[k].data(), g[k].size() * sizeof(double));
        if (rc == 1) return fail(ctx, FCPT_ERR_ARG, "no %s", grid_path(dir, want[k]).c_str());
        if (rc) return rc;
    }
    rc = fcpt_upload_state(ctx, g[0].data(), g[1].data(), g[2].data(), adi ? g[3].data() : nullptr);
    if (rc) return rc;
    if (adi) {
        // Qplus / Qminus make the restart bit for bit (restart.cpp:70-86);
        // without them the upload's heating/cooling estimate stays
        for (int f : {FCPT_QPLUS, FCPT_QMINUS}) {
            std::vector<double> q(grid_doubles(ctx, f));
            rc = read_file(ctx, grid_path(dir, f), q.data(), q.size() * sizeof(double));
            if (rc == 0) rc = fcpt_upload_field(ctx, f, q.data());
            else if (rc == 1) rc = FCPT_OK;
            if (rc) return rc;
        }
    }
    rc = fcpt_set_time(ctx, m.time, m.last_dt, (int32_t)m.n_monitor);
    if (rc) return rc;
    if (info) *info = m;
    return fcpt_synchronize(ctx);
}

int fcpt_read_snapshot_reference(fcpt_ctx *ctx, const char *dir)
{
    CTX_CHECK(ctx);
    if (!dir) return fail(ctx, FCPT_ERR_ARG, "null snapshot directory");
    const bool adi = ctx->P.adiabatic != 0;
    const int src[4] = {FCPT_SIGMA, FCPT_VRAD, FCPT_VAZI, FCPT_ENERGY};
    const int dst[4] = {FCPT_SIGMA0, FCPT_VRAD0, FCPT_VAZI0, FCPT_ENERGY0};
    for (int k = 0; k < (adi ? 4 : 3); ++k) {
        std::vector<double> g(grid_doubles(ctx, src[k]));
        int rc = read_file(ctx, grid_path(dir, src[k]), g.data(), g.size() * sizeof(double));
        if (rc == 1) return fail(ctx, FCPT_ERR_ARG, "no %s", grid_path(dir, src[k]).c_str());
        if (!rc) rc = fcpt_upload_field(ctx, dst[k], g.data());
        if (rc) return rc;
    }
    return FCPT_OK;
}

int fcpt_write_grid_files(fcpt_ctx *ctx, const char *outdir, const char *radial_spacing)
{
    CTX_CHECK(ctx);
    if (!outdir || !radial_spacing) return fail(ctx, FCPT_ERR_ARG, "null output directory or spacing");
    std::string text;
    char line[512];
    for (int i = 0; i <= ctx->P.nr; ++i) {
        std::snprintf(line, sizeof(line), "%.18g\n", ctx->Rinf[i]);
        text += line;
    }
    int rc = write_file(ctx, std::string(outdir) + "/used_rad.dat", text.data(), text.size());
    if (rc) return rc;
    text = "#RMIN\tRMAX\tPHIMIN\tPHIMAX          \tNRAD\tNAZ\tNGHRAD\tNGHAZ\tRadial_spacing\n";
    std::snprintf(line, sizeof(line), "%.16g\t%.16g\t%.16g\t%.16g\t%d\t%d\t%d\t%d\t%s\n", ctx->P.rmin,
                  ctx->P.rmax, 0.0, 2 * M_PI, ctx->P.nr, ctx->P.ns, 1, 1, radial_spacing);
    text += line;
    return write_file(ctx, std::string(outdir) + "/dimensions.dat", text.data(), text.size());
}

int fcpt_totals(fcpt_ctx *ctx, double radius, double *mass, double *angular_momentum)
{
    CTX_CHECK(ctx);
    launch_totals(ctx->P, ctx->stream, radius, ctx->totals_ring, ctx->totals_out);
    LAUNCH_CHECK(ctx);
    HIP_TRY(ctx, hipMemcpyAsync(ctx->totals_host, ctx->totals_out, 2 * sizeof(double),
                                hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    if (mass) *mass = ctx->totals_host[0];
    if (angular_momentum) *angular_momentum = ctx->totals_host[1];
    return FCPT_OK;
}

int fcpt_get_ring_geometry(fcpt_ctx *ctx, double *rmed, double *surf)
{
    if (!ctx) return FCPT_ERR_ARG;
    const size_t n = (size_t)ctx->P.nr;
    if (rmed) memcpy(rmed, ctx->Rmed.data(), n * sizeof(double));
    if (surf) memcpy(surf, ctx->Surf.data(), n * sizeof(double));
    return FCPT_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Totals that allocate nothing.  The ring geometry, the per-ring partial sums
// and the two results live in `scratch`, a file-scope device array: every GPU
// the library runs on holds its own copy until the process ends, at its own
// address, which is looked up once per device with hipGetSymbolAddress; host
// code uses only that address (the array's name is a host-side stand-in).
// Layout for nr rings: Rmed [0, nr), Surf [nr, 2 nr), ring partials
// [2 nr, 6 nr) (four per ring), results [6 nr, 6 nr + 2).  Every call writes
// each slot it later reads (the ring kernel writes all 4 nr partials, the
// fold both results), so nothing has to start at zero.  Calls on one GPU
// share the array: calls that overlap on one GPU race.
constexpr int kNoAllocMaxRings = FCPT_NOALLOC_MAX_RINGS;
static __device__ __align__(256) double scratch[6 * kNoAllocMaxRings + 2];

namespace {
constexpr int kNoAllocMaxDevices = 64;

std::mutex g_scratch_mu;
double *g_scratch_ptr[kNoAllocMaxDevices];
thread_local std::string g_noalloc_err;

int noalloc_fail(int code, const char *fmt, ...)
{
    char buf[256];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_noalloc_err = buf;
    return code;
}

// the current device's copy of `scratch`
int scratch_address(double **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return noalloc_fail(FCPT_ERR_DEVICE, "hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kNoAllocMaxDevices)
        return noalloc_fail(FCPT_ERR_DEVICE, "device %d beyond the %d devices served", dev, kNoAllocMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return noalloc_fail(FCPT_ERR_DEVICE, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        g_scratch_ptr[dev] = static_cast<double *>(p);
    }
    *out = g_scratch_ptr[dev];
    return FCPT_OK;
}
}  // namespace

extern "C" {

const char *fcpt_noalloc_last_error(void) { return g_noalloc_err.c_str(); }

int fcpt_totals_noalloc(int32_t nr, int32_t nphi, const double *rmed, const double *surf,
                        const double *sigma, const double *vazi, double omega_frame, double radius,
                        void *stream, double *mass, double *angular_momentum)
{
    g_noalloc_err.clear();
    if (!rmed || !surf || !sigma || !vazi || nr < 3 || nphi < 1)
        return noalloc_fail(FCPT_ERR_ARG, "null pointer or nr < 3 / nphi < 1");
    if (nr > kNoAllocMaxRings)
        return noalloc_fail(FCPT_ERR_ARG, "nr = %d exceeds the %d rings of the static scratch", nr,
                            kNoAllocMaxRings);
    double *s = nullptr;
    int rc = scratch_address(&s);
    if (rc) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    double *g_rmed = s, *g_surf = s + nr, *ring = s + 2 * (size_t)nr, *out = s + 6 * (size_t)nr;
    hipError_t e = hipMemcpyAsync(g_rmed, rmed, (size_t)nr * sizeof(double), hipMemcpyHostToDevice, st);
    if (e == hipSuccess)
        e = hipMemcpyAsync(g_surf, surf, (size_t)nr * sizeof(double), hipMemcpyHostToDevice, st);
    if (e != hipSuccess) return noalloc_fail(FCPT_ERR_DEVICE, "geometry upload: %s", hipGetErrorString(e));
    // only the fields k_totals_rings reads: sizes, Rmed, Surf, the frame, Sigma, v_phi
    KParams P{};
    P.nr = nr;
    P.ns = nphi;
    P.Rmed = g_rmed;
    P.Surf = g_surf;
    P.omega_frame = omega_frame;
    P.split = 0;
    P.f[FCPT_SIGMA] = const_cast<double *>(sigma);
    P.f[FCPT_VAZI] = const_cast<double *>(vazi);
    launch_totals(P, st, radius, ring, out);
    e = hipGetLastError();
    if (e != hipSuccess) return noalloc_fail(FCPT_ERR_DEVICE, "kernel launch: %s", hipGetErrorString(e));
    double res[2];
    e = hipMemcpyAsync(res, out, 2 * sizeof(double), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return noalloc_fail(FCPT_ERR_DEVICE, "result read-back: %s", hipGetErrorString(e));
    if (mass) *mass = res[0];
    if (angular_momentum) *angular_momentum = res[1];
    return FCPT_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Batches: many disks advanced by one launch per stage (plan_batch_step)

struct fcpt_batch {
    int device = 0;
    int split = 0;
    int radial_waves = 3;
    std::vector<fcpt_ctx *> disks;
    KParams *Ps = nullptr;  // device array: every disk's parameters, then their swapped views
    std::vector<BatchStageDev> stages;
    hipStream_t stream = nullptr;
    hipGraphExec_t graph[2] = {nullptr, nullptr};  // as a context's step_graph
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    hipEvent_t done = nullptr;  // end of the last batched run; every disk's stream waits for it
    std::string err;
    // the parameters the batched kernels see, and which members' radial tile
    // the batch chooses (left to the size rule by the disk)
    std::vector<KParams> host;
    std::vector<bool> auto_radial;
    std::vector<void *> plan_allocs;  // Ps and the stage tables of the current plan
};

namespace {
int bfail(fcpt_batch *b, int code, const char *msg)
{
    if (b) b->err = msg;
    return code;
}
#define BHIP(b, expr)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess) {                                                                \
            if (b) b->err = std::string(#expr) + ": " + hipGetErrorString(e_);                 \
            return FCPT_ERR_DEVICE;                                                            \
        }                                                                                      \
    } while (0)

void enqueue_batch_step(const fcpt_batch *b, hipStream_t st)
{
    for (const BatchStageDev &s : b->stages) launch_batch_stage(b->Ps, s, b->split, st);
}
}  // namespace

extern "C" {

const char *fcpt_batch_last_error(const fcpt_batch *b) { return b ? b->err.c_str() : "null batch"; }

// the device side of the batch's plan from b->host: every disk's parameters
// (disk d at d, its swapped view for the fused passes at n + d) and the work
// table of every stage; replaces the previous plan's arrays
static int upload_batch_plan(fcpt_batch *b)
{
    for (void *p : b->plan_allocs) hipFree(p);
    b->plan_allocs.clear();
    b->stages.clear();
    b->Ps = nullptr;
    auto alloc = [&](size_t bytes) -> void * {
        void *q = nullptr;
        if (hipMalloc(&q, bytes ? bytes : 16) != hipSuccess) return nullptr;
        b->plan_allocs.push_back(q);
        return q;
    };
    std::vector<KParams> views(b->host);
    for (const KParams &P : b->host) views.push_back(swapped_view(P));
    b->Ps = static_cast<KParams *>(alloc(views.size() * sizeof(KParams)));
    if (!b->Ps || hipMemcpy(b->Ps, views.data(), views.size() * sizeof(KParams), hipMemcpyHostToDevice) != hipSuccess)
        return bfail(b, FCPT_ERR_DEVICE, "batch parameters upload");
    for (const BatchStageHost &h : plan_batch_step(b->host)) {
        void *m = alloc(h.entries.size() * sizeof(BatchEntry));
        if (!m || hipMemcpy(m, h.entries.data(), h.entries.size() * sizeof(BatchEntry), hipMemcpyHostToDevice) !=
                      hipSuccess)
            return bfail(b, FCPT_ERR_DEVICE, "batch work table upload");
        b->stages.push_back(
            BatchStageDev{h.kind, h.arg, static_cast<const BatchEntry *>(m), (unsigned)h.entries.size()});
    }
    drop_graphs(b->graph);
    return FCPT_OK;
}

int fcpt_batch_create(fcpt_ctx *const *disks, int32_t n_disks, fcpt_batch **out)
{
    if (!disks || !out || n_disks <= 0) return FCPT_ERR_ARG;
    *out = nullptr;
    fcpt_batch *b = new fcpt_batch();
    b->device = disks[0] ? disks[0]->device : 0;
    b->split = disks[0] ? disks[0]->P.split : 0;
    std::vector<KParams> host;
    for (int k = 0; k < n_disks; ++k) {
        fcpt_ctx *c = disks[k];
        if (!c || c->device != b->device || c->P.split != b->split ||
            c->P.integrator != FCPT_INTEGRATOR_EULER) {
            delete b;
            return FCPT_ERR_ARG;  // one device, one storage mode, Euler disks
        }
        b->disks.push_back(c);
        // the fields the batched kernels read, stored
        if (c->derived_stale) {
            if (hipSetDevice(c->device) != hipSuccess || sync_derived(c) ||
                hipStreamSynchronize(c->stream) != hipSuccess) {
                delete b;
                return FCPT_ERR_DEVICE;
            }
        }
        KParams P = c->P;
        // the batch runs the fused step (its rounding points in split storage
        // are the disk's own, whatever tile the batch chooses below)
        set_step_modes(P, true);
        P.fold_in_kick = fold_in_kick(P);
        host.push_back(P);
    }
    // The walks' tiles of the members that leave them to the size rule,
    // chosen over the batch's wavefronts as the sweeps' tile below (results
    // do not depend on the tiles).
    resolve_kv_tiles(host);
    for (KParams &P : host)
        if (!kv_walk_applies(P)) P.visc_tile = resolve_visc_tile(P);
    // The sweeps' tile of the members that leave it to the size rule: all
    // members' blocks share one launch, so one tile by the batch's wavefronts
    // (the results do not depend on it).
    for (const KParams &P : host) b->auto_radial.push_back(P.radial_tile <= 0);
    const int sweep_tile = resolve_sweep_tile(host);
    for (KParams &P : host)
        if (P.radial_tile <= 0) P.radial_tile = sweep_tile;
    b->host = host;
    int rc = hipSetDevice(b->device) == hipSuccess ? FCPT_OK : FCPT_ERR_DEVICE;
    if (!rc) rc = upload_batch_plan(b);
    if (!rc && hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) rc = FCPT_ERR_DEVICE;
    if (!rc && hipEventCreateWithFlags(&b->done, hipEventDisableTiming) != hipSuccess) rc = FCPT_ERR_DEVICE;
    if (rc) {
        fcpt_batch_destroy(b);
        return rc;
    }
    *out = b;
    return FCPT_OK;
}

int fcpt_batch_destroy(fcpt_batch *b)
{
    if (!b) return FCPT_OK;
    hipSetDevice(b->device);
    if (b->stream) {
        hipStreamSynchronize(b->stream);
        hipStreamDestroy(b->stream);
    }
    drop_graphs(b->graph);
    if (b->ev0) hipEventDestroy(b->ev0);
    if (b->ev1) hipEventDestroy(b->ev1);
    if (b->done) hipEventDestroy(b->done);
    for (void *p : b->plan_allocs) hipFree(p);
    delete b;
    return FCPT_OK;
}

int fcpt_batch_set_radial_waves(fcpt_batch *b, int32_t waves)
{
    if (!b) return FCPT_ERR_ARG;
    if (waves != 2 && waves != 3) return bfail(b, FCPT_ERR_ARG, "radial waves must be 2 or 3");
    BHIP(b, hipSetDevice(b->device));
    BHIP(b, hipStreamSynchronize(b->stream));
    b->radial_waves = waves;
    BHIP(b, drop_graphs(b->graph));
    return FCPT_OK;
}

int fcpt_batch_synchronize(fcpt_batch *b)
{
    if (!b) return FCPT_ERR_ARG;
    BHIP(b, hipSetDevice(b->device));
    BHIP(b, hipStreamSynchronize(b->stream));
    return FCPT_OK;
}

static int ensure_batch_graph(fcpt_batch *b, bool many)
{
    hipGraphExec_t &exec = b->graph[many ? 1 : 0];
    if (exec) return FCPT_OK;
    hipGraph_t g = nullptr;
    BHIP(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    for (int k = 0; k < (many ? kGraphSteps : 1); ++k) enqueue_batch_step(b, b->stream);
    hipError_t e = hipStreamEndCapture(b->stream, &g);
    if (e != hipSuccess) return bfail(b, FCPT_ERR_DEVICE, hipGetErrorString(e));
    e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
    hipGraphDestroy(g);
    if (e != hipSuccess) {
        exec = nullptr;
        return bfail(b, FCPT_ERR_DEVICE, hipGetErrorString(e));
    }
    return FCPT_OK;
}

int fcpt_batch_run_steps(fcpt_batch *b, int32_t n_steps, int32_t use_graph)
{
    if (!b) return FCPT_ERR_ARG;
    if (n_steps < 0) return bfail(b, FCPT_ERR_ARG, "negative step count");
    BHIP(b, hipSetDevice(b->device));
    // the disks' own queued work (uploads, start-up calls) comes first
    for (fcpt_ctx *c : b->disks) BHIP(b, hipStreamSynchronize(c->stream));
    const bool many = n_steps >= kGraphSteps;
    if (use_graph) {
        const int rc = ensure_batch_graph(b, many);
        if (rc) return rc;
    }
    // the batched step after what has been queued on a disk's own stream since
    auto after = [b](fcpt_ctx *c) {
        const hipError_t e = hipEventRecord(b->done, c->stream);
        return e == hipSuccess ? hipStreamWaitEvent(b->stream, b->done, 0) : e;
    };
    // fields of its caller's own that a member's batched step would not read
    bool stored = false;
    for (size_t k = 0; k < b->disks.size(); ++k)
        stored = stored || (!b->disks[k]->derived_own && b->host[k].adiabatic && b->host[k].lazy_derived);
    if (n_steps > 0 && stored) {  // one iteration disk by disk
        for (fcpt_ctx *c : b->disks) {
            if (fcpt_run_steps(c, 1, 0)) return bfail(b, FCPT_ERR_DEVICE, c->err.c_str());
            BHIP(b, after(c));
        }
        --n_steps;
    }
    // what a member's own steps left stale and its batched step reads
    for (size_t k = 0; n_steps > 0 && k < b->disks.size(); ++k) {
        fcpt_ctx *c = b->disks[k];
        const bool stale = c->derived_stale;
        if (sync_for(c, b->host[k])) return bfail(b, FCPT_ERR_DEVICE, c->err.c_str());
        if (stale && !c->derived_stale) BHIP(b, after(c));
    }
    for (int left = n_steps; left > 0;) {
        // up to the next background move of a member in split storage
        int m = left;
        for (fcpt_ctx *c : b->disks)
            if (periodic_rebase(c)) m = std::min(m, c->rebase_interval - c->steps_since_rebase);
        int k = 0;
        if (use_graph) {
            const int per = many ? kGraphSteps : 1;
            for (; k + per <= m; k += per) BHIP(b, hipGraphLaunch(b->graph[many ? 1 : 0], b->stream));
        }
        for (; k < m; ++k) enqueue_batch_step(b, b->stream);
        BHIP(b, hipGetLastError());
        left -= m;
        // a disk call made after this one (a download, the totals) is ordered
        // after the batched steps on the disk's own stream
        BHIP(b, hipEventRecord(b->done, b->stream));
        for (fcpt_ctx *c : b->disks) BHIP(b, hipStreamWaitEvent(c->stream, b->done, 0));
        for (size_t k = 0; k < b->disks.size(); ++k) stepped(b->disks[k], b->host[k]);
        for (fcpt_ctx *c : b->disks) {
            if (!periodic_rebase(c) || (c->steps_since_rebase += m) < c->rebase_interval) continue;
            if (rebase_backgrounds(c)) return bfail(b, FCPT_ERR_DEVICE, c->err.c_str());
        }
    }
    return FCPT_OK;
}

int fcpt_batch_time_kernel(fcpt_batch *b, int32_t kernel, int32_t reps, double *ms_per_launch)
{
    if (!b) return FCPT_ERR_ARG;
    if (reps <= 0) return bfail(b, FCPT_ERR_ARG, "reps must be positive");
    int kinds[2] = {-1, -1};
    switch (kernel) {
    case FCPT_KERNEL_RADIAL_SWEEP:  // one kernel runs both sweeps
    case FCPT_KERNEL_AZIMUTHAL: kinds[0] = B_SWEEPS_ISO; kinds[1] = B_SWEEPS_ADI; break;
    case FCPT_KERNEL_CFL: kinds[0] = B_CFL_RINGS; kinds[1] = B_CFL_POT; break;  // some members' limits and
    case FCPT_KERNEL_POTENTIAL: kinds[0] = B_POTENTIAL; kinds[1] = B_CFL_POT; break;  // potential are one launch
    case FCPT_KERNEL_STRESS:
    case FCPT_KERNEL_VISC_FUSED:
        // the batched step runs the fused viscous pass, on views that differ
        // between disks; timed alone it could write the fields
        return bfail(b, FCPT_ERR_ARG, "the viscous kernels are not timed on a batch");
    default: return bfail(b, FCPT_ERR_ARG, "unknown kernel");
    }
    BHIP(b, hipSetDevice(b->device));
    if (!b->ev0) BHIP(b, hipEventCreate(&b->ev0));
    if (!b->ev1) BHIP(b, hipEventCreate(&b->ev1));
    auto one = [&]() {
        for (const BatchStageDev &s : b->stages) {
            if (s.kind != kinds[0] && s.kind != kinds[1]) continue;
            launch_batch_stage(b->Ps, s, b->split, b->stream);
        }
    };
    BHIP(b, hipStreamSynchronize(b->stream));
    one();
    BHIP(b, hipEventRecord(b->ev0, b->stream));
    for (int k = 0; k < reps; ++k) one();
    BHIP(b, hipEventRecord(b->ev1, b->stream));
    BHIP(b, hipGetLastError());
    BHIP(b, hipEventSynchronize(b->ev1));
    float ms = 0.f;
    BHIP(b, hipEventElapsedTime(&ms, b->ev0, b->ev1));
    if (ms_per_launch) *ms_per_launch = (double)ms / reps;
    return FCPT_OK;
}

// The batch's sweep tile (for the members that leave it to the size rule) by
// the sweeps' time: each candidate's plan is uploaded and the sweeps timed over
// `reps` launches, which write the transport's scratch arrays only, so the
// disks' state is untouched.
int fcpt_batch_autotune(fcpt_batch *b, int32_t reps, int32_t *radial_tile, int32_t *radial_waves)
{
    if (!b) return FCPT_ERR_ARG;
    if (reps <= 0) return bfail(b, FCPT_ERR_ARG, "reps must be positive");
    BHIP(b, hipSetDevice(b->device));
    BHIP(b, hipStreamSynchronize(b->stream));
    int cur_t = 0;
    for (size_t k = 0; k < b->host.size(); ++k)
        if (b->auto_radial[k]) cur_t = b->host[k].radial_tile;
    int best_t = cur_t;
    double best = 1e300;
    const int tiles[] = {4, 8, 16, 32};
    for (int t : tiles) {
        if (cur_t == 0) break;  // no member's tile is the batch's to choose
        for (size_t k = 0; k < b->host.size(); ++k)
            if (b->auto_radial[k]) b->host[k].radial_tile = t;
        int rc = upload_batch_plan(b);
        double ms = 0.0;
        if (!rc) rc = fcpt_batch_time_kernel(b, FCPT_KERNEL_RADIAL_SWEEP, reps, &ms);
        if (rc) return rc;
        if (ms < best) {
            best = ms;
            best_t = t;
        }
    }
    for (size_t k = 0; k < b->host.size(); ++k)
        if (b->auto_radial[k]) b->host[k].radial_tile = best_t;
    const int rc = upload_batch_plan(b);
    if (rc) return rc;
    if (radial_tile) *radial_tile = best_t;
    if (radial_waves) *radial_waves = b->radial_waves;
    return FCPT_OK;
}

int fcpt_batch_time_steps(fcpt_batch *b, int32_t n_steps, int32_t use_graph, double *ms_total)
{
    if (!b) return FCPT_ERR_ARG;
    BHIP(b, hipSetDevice(b->device));
    if (!b->ev0) BHIP(b, hipEventCreate(&b->ev0));
    if (!b->ev1) BHIP(b, hipEventCreate(&b->ev1));
    int rc = use_graph ? ensure_batch_graph(b, n_steps >= kGraphSteps) : FCPT_OK;  // outside the timed region
    if (!rc) rc = fcpt_batch_run_steps(b, 0, 0);  // waits for the disks' own queued work
    if (rc) return rc;
    BHIP(b, hipStreamSynchronize(b->stream));
    BHIP(b, hipEventRecord(b->ev0, b->stream));
    rc = fcpt_batch_run_steps(b, n_steps, use_graph);
    if (rc) return rc;
    BHIP(b, hipEventRecord(b->ev1, b->stream));
    BHIP(b, hipEventSynchronize(b->ev1));
    float ms = 0.f;
    BHIP(b, hipEventElapsedTime(&ms, b->ev0, b->ev1));
    for (fcpt_ctx *c : b->disks) {
        DevScalars sc;
        BHIP(b, hipMemcpy(&sc, c->s_dev, sizeof(DevScalars), hipMemcpyDeviceToHost));
        if (sc.error_flags & 1) {
            // reported once, like a disk's own calls report it
            BHIP(b, hipMemset(&c->s_dev->error_flags, 0, sizeof(int)));
            return bfail(b, FCPT_ERR_NONFINITE, "a disk's CFL time step became non-finite");
        }
    }
    if (ms_total) *ms_total = (double)ms;
    return FCPT_OK;
}

}  // extern "C"
