// Device-side data structures shared by the gfx950 kernels and the host glue.
//
// One disk = one KParams block passed by value to every kernel: grid sizes,
// physical scalars, pointers to the per-ring metric arrays and to every field
// in HBM (and, for split storage, to the per-ring backgrounds).  Quantities that change from step to step (dt, time, planets, the
// CFL minimum) live in a DevScalars block in device memory so that a captured
// graph of the step can be replayed without host involvement.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "../../include/fcpt.h"

namespace fcpt {

constexpr int kMaxPlanets = FCPT_MAX_PLANETS;
// a ring's values in KParams::ring_tab: the metric the walks read, and the
// ring-uniform products and quotients of their formulas
enum {
    TAB_RINF = 0, TAB_INV_RINF, TAB_RMED, TAB_INV_RMED, TAB_INV_DIFF_RMED, TAB_INV_DIFF_RSUP, TAB_INV_DIFF_RSUP_RB,
    TAB_SRC_INVDXTHETA, TAB_INV_DXTHETA, TAB_INV_OMEGA_K, TAB_OMEGA_K, TAB_VISC_AREA, TAB_RINF_SQ, TAB_RINF_OMEGA,
    TAB_TW_LSQ, TAB_RMED_SUM, TAB_RMED_SUM_RCP, TAB_RSUP_RINF, TAB_RMED_SQ_DIFF, TAB_RMED_SQ_DIFF_RCP,
    TAB_RMED_DIFF, TAB_E_LO, TAB_E_HI, TAB_SQRT_GAMMA, TAB_SQRT_GAMMA_RCP, TAB_C_LIGHT, TAB_C_LIGHT_RCP,
    TAB_G_GM1, TAB_MU_GM1, TAB_SIGMA_FLOOR10, TAB_BETA_INV, TAB_ARTVISC_SQ, kRingTabs
};

// KParams::split_emul: c_s, H, nu and the pressure; the source-term velocities
// and the viscous heating's stress tensor
enum { SPLIT_EMUL_DERIVED = 1, SPLIT_EMUL_STAGES = 2 };

struct DevPlanet {
    double x, y, mass, r_cubic;
    double smooth;  // fixed potential smoothing length, or < 0: ThicknessSmoothing * H of the cell
};

// per-body potential smoothing of one step, formed on the host (compute_smoothing)
struct BodySmoothing {
    double s[kMaxPlanets];
};

// Step-varying scalars, resident in device memory.
struct DevScalars {
    double dt;            // step size used by the current step's kernels
    double time;          // simulation time at the start of the step
    double last_dt;       // sim::last_dt (CFLmaxVar limiter)
    double cfl_dt;        // result of the last CFL reduction
    int n_monitor;
    int error_flags;      // bit 0: non-finite or non-positive dt
    int n_planets;
    unsigned step_count;  // CFL reductions so far: part of the split storage's rounding key
    double indirect_x, indirect_y;
    DevPlanet planet[kMaxPlanets];
    // LeapFrog: the full step's dt and start time while the kicks run with
    // dt / 2, the second kick's bodies (has_mid) and the first kick's, kept
    // while the second kick uses the slots above
    double dt_step, t_step;
    int has_mid, n_planets_mid, n_planets_first, pad2_;
    double indirect_mid_x, indirect_mid_y, indirect_first_x, indirect_first_y;
    DevPlanet planet_mid[kMaxPlanets];
    DevPlanet planet_first[kMaxPlanets];
    // last_dt and the next step_count as the last step left them: what a kick that folds
    // the CFL minima reads while one of its wavefronts writes last_dt and step_count
    double last_prev;
    unsigned count_next;
    unsigned count_derived;  // the step count at which the derived fields were last formed to be stored
};

// values per ring of KParams::sweep_tab
enum SweepTab { SW_RMED = 0, SW_INV_DIFF_RMED, SW_RINF, SW_INV_SURF, SW_WIDTH, SW_DXTHETA, SW_INV_DXTHETA, kSweepTabs = 8 };

struct KParams {
    int nr, ns;
    double dphi, invdphi;
    double rmin, rmax;
    // physics
    int adiabatic;
    int integrator;      // FCPT_INTEGRATOR_*
    int artvisc;
    int artvisc_dissipation;
    int heating_viscous;
    int cooling_beta_enabled;
    int cooling_beta_ref;
    int bc_inner, bc_outer;
    int damping;
    int damp_ids[4];
    int zone_in[2], zone_out[2];  // last ring of the inner and first of the outer damping
                                  // zone of the scalar [0] and vector [1] fields (none: -1, INT_MAX)
    double G, Rgas, sigma_sb, c_light, mstar, mu, gamma;
    double aspect_ratio, flaring, alpha, thickness_smoothing;
    double cfl, cfl_max_var, heating_cooling_cfl_limit;
    double sigma0, sigma_floor, t_min, t_max;
    double artvisc_factor, heating_viscous_factor;
    double cooling_beta, cooling_beta_ramp_up, radial_viscosity_factor;
    double damping_inner_limit, damping_outer_limit, damping_time_factor,
        damping_time_radius_outer;
    double omega_frame, monitor_timestep;
    // per-ring metric arrays (length nr + 2)
    const double *Rinf, *Rsup, *Rmed, *Surf, *InvSurf, *InvRmed, *InvRinf, *InvDiffRmed,
        *InvDiffRsup, *InvDiffRsupRb;
    // per-sector tables: cos / sin of dphi * j (cell-centre coordinates)
    const double *cosphi, *sinphi;
    // storage: 0 = FP64 fields; 1 = FP32 deviations from FP64 per-ring backgrounds
    int split;
    int split_rounding;  // split storage: 0 rounds deviations to nearest, 1 stochastically
    int radial_tile;     // rings per walk of the transport's sweeps (0: size-based choice)
    int radial_waves;    // FCPT_PARAM_RADIAL_WAVES as set (2 or 3); the sweeps have one register budget
    int visc_tile;       // rings per thread of the fused viscous pass (0: size-based choice)
    int kick_tile;       // rings per thread of the kick walk (0: size-based choice, 1: off)
    int kv_tile;         // batches: the kick walk's rings per thread, chosen over the batch
    // the fused step with the kick walk: the derived fields (the sound speed,
    // viscosity, temperature and pressure; the pressure of an isothermal
    // disk) are formed from E and Sigma where the step needs them instead of
    // stored, and the walk writes the updated E to its partner ealt; the host
    // stores the fields (k_derived) before anything else reads them
    int lazy_derived;
    // split storage: values the kick walk and the CFL round as if stored
    // (SPLIT_EMUL_*), in disks whose step keeps fewer values in FP64
    int split_emul;
    // the fused LeapFrog step's kick: 1 and 2 run over dt / 2, 2 from the midstep
    // time and with the midstep bodies; 0 elsewhere (the whole dt)
    int kick, pad_;
    // fields in HBM (indexed by fcpt_field): double, or float when split
    void *f[FCPT_NUM_FIELDS];
    // split storage: per-ring backgrounds of every field (nr + 2 values each;
    // null in FP64 mode); the potential's is rewritten by the potential kernel
    double *bg[FCPT_NUM_FIELDS];
    // what the transport's sweeps write and the end of the step reads, FP64 in
    // both storage modes (rounded once per step, on the final store)
    void *mom[4];        // radial momentum +/-, angular momentum +/-
    void *sig_c, *en_c;  // density and energy
    void *valt[2];       // partners of v_r and v_phi for the fused step kernels
    void *ealt;          // partner of E (adiabatic disks)
    double *bgm[4];      // backgrounds of the four momenta (split storage)
    double *iso_cs, *iso_h, *iso_nu;  // locally isothermal ring profiles of c_s, H, nu
    // kRingTabs values per ring, nr + 2 rings (k_ring_tables): one base pointer
    // and one run of memory per ring for the walks' scalar loads
    double *ring_tab;
    // the transport's ring constants, kSweepTabs per ring of one 64-byte line (k_ring_tables)
    double *sweep_tab;
    double *cfl_tab;     // per ring: radial, azimuthal, smaller and squared smaller cell size, each with its reciprocal
    double *damp_tab;     // per ring: the damping's squared ramp and time scale: scalar inner, outer, vector inner, outer
    double energy_per_t;  // R / mu / (gamma - 1): energy_at's factor, to rounding
    int const_ok;         // the physical constants lie in the range quot_in assumes
    double *vmean;       // per-ring mean azimuthal velocity
    double *vuni;        // per-ring uniform residual velocity (FARGO)
    int *nshift;         // per-ring integer shift
    double *ring_min;    // the smallest CFL limit of each ring (nr)
    DevScalars *s;
    int cfl_pot;         // the CFL limits and the potential run as one launch (set_step_modes)
    int h_lazy;          // and H is formed there, stored in the ghost rings only
    int fold_in_kick;    // the kick walk folds the ring minima of the CFL limits itself
    int pad1_;
    const unsigned *step_at;  // the count the rounding keys of this launch take
    DevScalars *s_out;  // pinned host mirror that the step's clock is written to, or null
};

}  // namespace fcpt
