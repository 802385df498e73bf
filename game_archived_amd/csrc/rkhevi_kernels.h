/*
 * rkhevi_kernels.h -- launchers of the device kernels (one namespace per
 * precision form of the step).
 */
#ifndef GAME_RKHEVI_KERNELS_H
#define GAME_RKHEVI_KERNELS_H

#include "rkhevi_dev.h"

/* horizontal operators and tendencies: work arrays double (FP64 form) or
   float (mixed form), register arithmetic FP64 in both */
namespace hor {
/* the pressure gradient of s (nl, l, old, their combination W.pgrad_comb for
   the implicit weight itw, and the condensates' term), and in every step but
   a first one the first substep's momentum tendency td and wind update
   (w_new = w_old + dt td at the edges), which read the carried W.pvt and
   W.vsq_grad.  The gas fractions come from W.gas_frac: s must be the state
   the last col::temperature(..., W.gas_frac, ...) was formed from */
void pgrad(const DevGrid &G, const DevState &s, const DevWork &W, int first, double itw, double *td,
           const double *w_old, double *w_new, double dt, hipStream_t st);
void pgrad(const DevGrid &G, const DevState &s, const DevWorkF &W, int first, double itw, float *td,
           const double *w_old, double *w_new, double dt, hipStream_t st);
/* mass flux, PV, TRSK flux, kinetic energy and its gradient */
void advection(const DevGrid &G, const double *wind, const double *rho_gas, const DevWork &W, hipStream_t st);
void advection(const DevGrid &G, const double *wind, const double *rho_gas, const DevWorkF &W, hipStream_t st);
/* the step's parts of it: mass flux, triangle vorticity and PV; kinetic energy */
void advection_pv(const DevGrid &G, const double *wind, const double *rho_gas, const DevWork &W, hipStream_t st);
void advection_pv(const DevGrid &G, const double *wind, const double *rho_gas, const DevWorkF &W, hipStream_t st);
void kinetic_energy(const DevGrid &G, const double *wind, const DevWork &W, hipStream_t st);
void kinetic_energy(const DevGrid &G, const double *wind, const DevWorkF &W, hipStream_t st);
/* and, from W.flux, W.pv and W.vsq: TRSK flux, kinetic-energy gradient and the
   tendency td = (1 - new_w) td_old + new_w (...) -- at the edges with the wind
   update; at the w points with the condensates' term of the densities rho
   (null: W.pgc_v as it is) */
void momentum_e(const DevGrid &G, const DevWork &W, double *td, const double *td_old, const double *w_old, double *w_new,
                double new_w, double dt, hipStream_t st);
void momentum_e(const DevGrid &G, const DevWorkF &W, float *td, const float *td_old, const double *w_old, double *w_new,
                double new_w, double dt, hipStream_t st);
void momentum_w(const DevGrid &G, const DevWork &W, double *td, const double *td_old, double new_w, const double *rho,
                hipStream_t st);
void momentum_w(const DevGrid &G, const DevWorkF &W, float *td, const float *td_old, double new_w, const double *rho,
                hipStream_t st);
void scalar_tend(const DevGrid &G, const DevState &s, const DevState &td, const DevWork &W, int rk, hipStream_t st);
void scalar_tend(const DevGrid &G, const DevState &s, const DevState &td, const DevWorkF &W, int rk, hipStream_t st);
void inner_product(const DevGrid &G, const double *a, const double *b, double *out, hipStream_t st);
void grad(const DevGrid &G, const double *f, double *out, hipStream_t st);
void curl_triangles(const DevGrid &G, const double *wind, double *out, hipStream_t st);
/* fills the slot-major tables of DevGrid from the others */
void tables(const DevGrid &G, unsigned *c_e, unsigned *c_n, unsigned *c_from, unsigned *e_ti, unsigned *e_tm, double *e_tw,
            unsigned *e_rc, double *e_rw, unsigned *t_e, hipStream_t st);
/* fills the grid constant G.vcw (n_oro x 6 x NSH doubles) */
void vcc_weights(const DevGrid &G, double *vcw, hipStream_t st);
void vorticity_flux(const DevGrid &G, const double *F, const double *pv, double *out, hipStream_t st);
}

/* column solvers, point physics and state arithmetic shared by both forms:
   FP64 arithmetic; the work arrays are double (FP64 form) or float (mixed) */
namespace col {
/* cpc (may be null): c_p of ice and of liquid water at the temperature, 2 x S;
   gf (may be null): gas density over total density, S */
void temperature(const DevGrid &G, const DevState &s, double *T, double *cpc, double *gf, hipStream_t st);
void temperature(const DevGrid &G, const DevState &s, float *T, float *cpc, double *gf, hipStream_t st);
void phase_trans(const DevGrid &G, const DevState &s, const double *T, const double *cpc, double *ptr, double *phr,
                 double dt, hipStream_t st);
void phase_trans(const DevGrid &G, const DevState &s, const float *T, const float *cpc, float *ptr, float *phr,
                 double dt, hipStream_t st);
/* moist (6 constituents, 4 condensates): temperature, c_p, gas fraction and
   phase transitions in one pass, the results of temperature + phase_trans */
void temperature_phase_trans(const DevGrid &G, const DevState &s, double *T, double *cpc, double *gf, double *ptr,
                             double *phr, double dt, hipStream_t st);
void temperature_phase_trans(const DevGrid &G, const DevState &s, float *T, float *cpc, double *gf, float *ptr,
                             float *phr, double dt, hipStream_t st);
/* snr: the new state as read before this substep writes it (at rk 0 the old
   state, which equals it by the step's entry condition) */
void ver_waves(const DevGrid &G, const DevState &so, const DevState &snr, const DevState &sn, const DevState &td,
               const StepConsts &K, int rk, hipStream_t st);
void ver_waves(const DevGrid &G, const DevState &so, const DevState &snr, const DevState &sn, const DevState &td,
               const float *td_wind, const StepConsts &K, int rk, hipStream_t st);
void gen_densities(const DevGrid &G, const DevState &so, const DevState &sn, const DevState &td, const double *T,
                   const double *cpc, double *sed_heat, const StepConsts &K, int rk, hipStream_t st);
void gen_densities(const DevGrid &G, const DevState &so, const DevState &sn, const DevState &td, const float *T,
                   const float *cpc, float *sed_heat, const StepConsts &K, int rk, hipStream_t st);
void linear_combine(const DevGrid &G, const DevState &a, const DevState &b, const DevState &o, double c0, double c1,
                    hipStream_t st);
/* G.idv[b] = (0.5 dt)/vol[b] */
void tracer_quotients(const DevGrid &G, double dt, hipStream_t st);
/* per-block compensated (sum, error) pairs of sum_i x[i]*y[i]*vol[i] (y may be
   null: sum_i x[i]*vol[i]) into partials[0 .. 2*INTEGRAL_BLOCKS) */
const int INTEGRAL_BLOCKS = 1024;
int integral_partials(i64 n, const double *x, const double *y, const double *vol, double *partials, hipStream_t st);
int integral_partials(i64 n, const double *x, const float *y, const double *vol, double *partials, hipStream_t st);
}

#endif
