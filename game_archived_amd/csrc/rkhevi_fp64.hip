/*
 * rkhevi_fp64.hip -- FP64 device kernels of GAME's RKHEVI step for gfx950.
 *
 * Each kernel evaluates one or more loops of the reference with the same
 * floating-point operations in the same order (this file is compiled with
 * -ffp-contract=off), so that the FP64 path reproduces the CPU reference to
 * the last bit wherever no transcendental function is involved.  Fusion only
 * ever recomputes a value with identical arithmetic; no reduction order is
 * changed.  All kernels are HBM-bandwidth bound gathers/stencils; there is no
 * dense contraction, hence no MFMA.
 */
#include <type_traits>

#include "rkhevi_dev.h"
#include "rkhevi_kernels.h"

#define GRID1(n) dim3((unsigned)(((n) + TPB - 1)/TPB))

/* ------------------------------------------------------------------ */
/* small device helpers restating reference functions                   */
/* ------------------------------------------------------------------ */

/* the constituent sum of derived_quantities.c:83-95 at element i of a row:
   rho is constituent 0's row, NC the constituent count, all loads first */
template <int NC>
__device__ __forceinline__ double density_total_at(const DevGrid &G, const double *rho, unsigned i)
{
    double v[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) v[k] = at(rho + (i64)k*G.s, i);
    double r = 0.0;
#pragma unroll
    for (int k = 0; k < NC; ++k) r += v[k];
    return r;
}

/* ------------------------------------------------------------------ */
/* kernels                                                              */
/* ------------------------------------------------------------------ */

/* derived_quantities.c:15-40 */
template <typename TO>
__global__ void __launch_bounds__(TPB) k_temperature(DevGrid G, DevState s, TO *T, TO *cpc, double *gf)
{
    i64 i = (i64)blockIdx.x*TPB + threadIdx.x;
    if (i >= G.s) return;
    /* the gas fraction of the box, as the pressure gradient forms it
       (manage_pressure_gradient.c:17-87) */
    if (gf) gf[i] = s.rho[(i64)G.n_cond*G.s + i]/density_total(G, s.rho, i);
    double t = (G.thbg[i] + s.tp[i])*(G.exbg[i] + s.ep[i]);
    if (G.moist)
        t = t/(1.0 + s.rho[(i64)(G.n_cond + 1)*G.s + i]/s.rho[(i64)G.n_cond*G.s + i]*(GC_M_D/GC_M_V - 1.0));
    T[i] = (TO)t;
    if (cpc) {
        /* dictionary.c:111-190: snow and cloud ice (even constituents) share
           the ice formula, rain and cloud water the liquid one */
        const double tt = (double)(TO)t;
        cpc[i] = (TO)c_p_ice(tt);
        cpc[G.s + i] = (TO)c_p_water(tt);
    }
}

/* what the momentum tendency and the wind update read and write beside the
   pressure gradient (vector_tendencies_expl.c:74-131, manage_rkhevi.c:67-75):
   the tendency td, the old and new wind, the substep's weight new_w of the
   new tendency.  friction_acc is zero with momentum diffusion and PBL off:
   x + 0.0 == x.  The old tendency has weight 1 - new_w = 0 in the first
   substep, where it is neither read nor added (its product with 0 is a zero,
   the identity of the sum); IEEE addition commutes, so adding it last changes
   no bit.  The kernels that form the last missing term take the update along:
   a kernel of its own read each term again (150 us per substep at res 7 x 26) */
template <typename TW>
struct Mom {
    TW *td;
    const TW *td_old;       /* the first substep's, read with weight 1 - new_w: td, or the tape's */
    const double *wind_old;
    double *wind_new;
    double new_w, dt;
};

/* derived_quantities.c:15-40 via gas fractions: gas over total density of one
   box of row l (NC constituents) */
template <int NC>
__device__ __forceinline__ double gas_fraction_at(const DevGrid &G, const double *rho, i64 row, unsigned h)
{
    constexpr int n_cond = NC == 6 ? 4 : 0;
    const double total = density_total_at<NC>(G, rho + row, h);
    return at(rho + n_cond*G.s + row, h)/total;
}

/* manage_pressure_gradient.c:17-87 at the interior w points (layers 1..L-1),
   fused with calc_pressure_grad_condensates_v; gf: the gas fractions of state
   s, formed with the reference's arithmetic by the temperature kernel.  TEND:
   with the first substep's tendency, for which the carried momentum advection
   is there (every step but a first one) */
template <typename TW, bool TEND>
__global__ void __launch_bounds__(TPB) k_pgrad_w(DevGrid G, DevState s, DevWorkT<TW> W, int first_step,
                                                 const double *gf, double cvw, Mom<TW> m, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned h = bk.x*TPB + threadIdx.x;
    if (h >= (unsigned)G.nsh) return;
    const int lev = (int)bk.y + 1;
    const i64 w = (i64)lev*G.vpl, lo = (i64)lev*G.nsh, up = lo - G.nsh;   /* rows of the level and of the layers around it */
    const double d_up = at(gf + up, h), d_lo = at(gf + lo, h);
    const double gm = at(G.gm + w, h);
    double pvt = 0.0, vg = 0.0;
    if (TEND) { pvt = (double)at(W.pvt + w, h); vg = (double)at(W.vsq_grad + w, h); }
    TW old_t = (TW)0;
    if (!first_step) old_t = (TW)(-(double)at(W.pgrad_nl + w, h) - (double)at(W.pgrad_l + w, h));
    const double tp_up = at(s.tp + up, h), tp_lo = at(s.tp + lo, h);
    double raw = (at(s.ep + up, h) - at(s.ep + lo, h))/at(G.nd + w, h);
    double p1_up = GC_C_D_P*(at(G.thbg + up, h) + tp_up), p1_lo = GC_C_D_P*(at(G.thbg + lo, h) + tp_lo);
    double nl = (0.5*(p1_up + p1_lo))*raw;
    double p2_up = GC_C_D_P*tp_up, p2_lo = GC_C_D_P*tp_lo;
    double ll = (0.5*(p2_up + p2_lo))*at(G.exbg_grad + w, h);
    nl = (0.5*(d_up + d_lo))*nl;
    ll = (0.5*(d_up + d_lo))*ll;
    if (first_step) old_t = (TW)(-nl - ll);
    /* the momentum tendency's combination of the stored values
       (vector_tendencies_expl.c), which the second substep reads */
    const TW comb = (TW)(-cvw*((double)(TW)nl + (double)(TW)ll));
    double c_up = d_up - 1.0, c_lo = d_lo - 1.0;
    const TW pgc = (TW)((0.5*(c_up + c_lo))*gm);
    put(W.pgrad_old + w, h, old_t);
    put(W.pgrad_nl + w, h, (TW)nl);
    put(W.pgrad_l + w, h, (TW)ll);
    put(W.pgrad_comb + w, h, comb);
    put(W.pgc_v + w, h, pgc);
    if (TEND) {
        const double tv = m.new_w*(
            (double)comb   /* -cvw*(nl + l) */
            + pvt
            - 0.5*vg
            + (double)pgc);
        put(m.td + w, h, (TW)tv);
    }
}

/* grad at the edges (gradient_operators.c:14-33 with the terrain term of
   averaging.c:113-133) for the successive layers l0, l0 + 1, ... of one
   edge, as manage_pressure_gradient.c:17-72 and the kinetic-energy gradient
   use it.  Over orography the two cells' values of layer l + 1 and their
   vertical gradients at the w level between layers l and l + 1, which layer
   l's terrain correction reads, are carried to layer l + 1 instead of loaded
   and formed again; each quotient is the one the layer-wise formula forms,
   so the results are identical.  The next layer's values are loaded before
   this layer's are combined.  A flat grid needs none of it and no registers
   for it.  The weights come from the cell-major copy ipwT: consecutive cells'
   weights are consecutive words, where ipw holds a cell's eight together (one
   64-byte line per lane). */
struct EdgeCarry { double ff, ft, gwf, gwt; };

template <bool FLAT, typename TF>
__device__ __forceinline__ double grad_edge_walk(const DevGrid &G, const TF *f, int l, int l0, unsigned e, unsigned fr,
                                                 unsigned to, EdgeCarry &c)
{
    const int nsh = G.nsh, L = G.L, lt = L - G.n_oro;
    const i64 vi = nsh + (i64)l*G.vpl;
    const TF *fl = f + (i64)l*nsh;
    if constexpr (FLAT) return ((double)at(fl, to) - (double)at(fl, fr))/at(G.nd + vi, e);
    if (l == l0) { c.ff = (double)at(fl, fr); c.ft = (double)at(fl, to); }
    /* layer l + 1 (the last layer reloads itself, unused) */
    const TF *fn = l + 1 < L ? fl + nsh : fl;
    const double nff = (double)at(fn, fr), nft = (double)at(fn, to);
    double g = (c.ft - c.ff)/at(G.nd + vi, e);
    if (l >= lt) {
        const double *w6 = G.ipwT + ((i64)l*8 + 6)*nsh, *w7 = w6 + nsh;
        /* the vertical gradient at level l of both cells
           (gradient_operators.c:35-54): carried unless layer l - 1 had no
           terrain term or lies in another chunk */
        if (l == l0 || l == lt) {
            const double *nw = G.nd + (i64)l*G.vpl;
            c.gwf = ((double)at(fl - nsh, fr) - c.ff)/at(nw, fr);
            c.gwt = ((double)at(fl - nsh, to) - c.ft)/at(nw, to);
        }
        double s = at(w6, fr)*c.gwf;
        s += at(w6, to)*c.gwt;
        if (l < L - 1) {
            /* at level l + 1 */
            const double *nw = G.nd + (i64)(l + 1)*G.vpl;
            const double gf1 = (c.ff - nff)/at(nw, fr);
            const double gt1 = (c.ft - nft)/at(nw, to);
            s += at(w7, fr)*gf1;
            s += at(w7, to)*gt1;
            c.gwf = gf1;
            c.gwt = gt1;
        }
        s = 0.5*s;
        g += -at(G.slope + vi, e)*s;
    }
    c.ff = nff;
    c.ft = nft;
    return g;
}

/* manage_pressure_gradient.c:17-72 at the edges: one thread per edge walks a
   chunk of layers, so the edge's table entries are read once.  TEND: with the
   first substep's tendency and wind update (as k_pgrad_w) */
template <bool FLAT, typename TW, bool TEND>
__global__ void __launch_bounds__(TPB) k_pgrad_e(DevGrid G, DevState s, DevWorkT<TW> W, int first_step,
                                                 const double *gf, double chw, double ohw, Mom<TW> m, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned e = bk.x*TPB + threadIdx.x;
    if (e >= (unsigned)G.nvh) return;
    const unsigned fr = G.from[e], to = G.to[e];
    int l0, l1;
    layer_chunk(G.L, bk.y, sp.run, l0, l1);
    EdgeCarry carry;
    for (int l = l0; l < l1; ++l) {
        const i64 vi = G.nsh + (i64)l*G.vpl, sl = (i64)l*G.nsh;
        TW old_t = 0;
        if (!first_step) old_t = (TW)(-(double)at(W.pgrad_nl + vi, e) - (double)at(W.pgrad_l + vi, e));
        double pvt = 0.0, vg = 0.0, wo = 0.0;
        if (TEND) {
            pvt = (double)at(W.pvt + vi, e);
            vg = (double)at(W.vsq_grad + vi, e);
            wo = at(m.wind_old + vi, e);
        }
        const double g = grad_edge_walk<FLAT, double>(G, s.ep, l, l0, e, fr, to, carry);
        const double tp_t = at(s.tp + sl, to), tp_f = at(s.tp + sl, fr);
        double p1_t = GC_C_D_P*(at(G.thbg + sl, to) + tp_t), p1_f = GC_C_D_P*(at(G.thbg + sl, fr) + tp_f);
        double nl = (0.5*(p1_t + p1_f))*g;
        double p2_t = GC_C_D_P*tp_t, p2_f = GC_C_D_P*tp_f;
        double ll = (0.5*(p2_t + p2_f))*at(G.exbg_grad + vi, e);
        const double d_t = at(gf + sl, to), d_f = at(gf + sl, fr);
        nl = (0.5*(d_t + d_f))*nl;
        ll = (0.5*(d_t + d_f))*ll;
        if (first_step) old_t = (TW)(-nl - ll);
        /* the momentum tendency's combination of the stored values
           (vector_tendencies_expl.c), which the second substep reads */
        const TW comb = (TW)(ohw*(double)old_t - chw*((double)(TW)nl + (double)(TW)ll));
        put(W.pgrad_old + vi, e, old_t);
        put(W.pgrad_nl + vi, e, (TW)nl);
        put(W.pgrad_l + vi, e, (TW)ll);
        put(W.pgrad_comb + vi, e, comb);
        if (TEND) {
            const double tv = m.new_w*(
                (double)comb   /* ohw*old - chw*(nl + l) */
                + pvt
                - 0.5*vg);
            put(m.td + vi, e, (TW)tv);
            put(m.wind_new + vi, e, wo + m.dt*tv);
        }
    }
}

/* vorticities.c:167-222, one thread per triangle and chunk of layers.
   The loads of the layer below are issued before the current layer is
   formed, and the wind and edge heights of the layers above and below (the
   two candidates of the terrain interpolation) are carried in registers, so
   no load waits on the sign test that selects between them. */
template <typename TW>
__global__ void __launch_bounds__(TPB) k_rel_vort_tri(DevGrid G, const double *w, TW *res, Span sp)
{
    const Blk bk = linear_block();
    const unsigned h = bk.x*TPB + threadIdx.x;
    if (h >= (unsigned)G.nt) return;
    const int L = G.L, lt = L - G.n_oro, nsh = G.nsh, vpl = G.vpl, nvh = G.nvh;
    const i64 dvpl = G.dvpl;
    unsigned vit[3];
    double sg[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const unsigned q = at(G.t_e + (i64)j*G.nt, h);
        vit[j] = q & 0x7fffffffu;
        sg[j] = q >> 31 ? -1.0 : 1.0;
    }
    struct Lay { double w[3], z[3], nd[3], dz, da; };
    auto load = [&](int l) {
        Lay x;
        const i64 vi = nsh + (i64)l*vpl, di = nvh + (i64)l*dvpl;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            x.w[j] = at(w + vi, vit[j]);
            x.z[j] = at(G.zv + vi, vit[j]);
            x.nd[j] = at(G.nd + vi, vit[j]);
        }
        x.dz = at(G.dzv + di, h);
        x.da = at(G.darea + di, h);
        return x;
    };
    int l0, l1;
    layer_chunk(L, bk.y, sp.run, l0, l1);
    if (l0 >= l1) return;
    double wp[3], zp[3];   /* layer l - 1 (layer 0, unused, at the top) */
    const i64 vp = nsh + (i64)(l0 > 0 ? l0 - 1 : 0)*vpl;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        wp[j] = at(w + vp, vit[j]);
        zp[j] = at(G.zv + vp, vit[j]);
    }
    Lay cur = load(l0);
    for (int l = l0; l < l1; ++l) {
        const Lay nxt = load(l + 1 < L ? l + 1 : l);
        double r = 0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double vel = cur.w[j], lrf = 1;
            if (l >= lt) {
                lrf = (G.radius + cur.dz)/(G.radius + cur.z[j]);
                const double delta_z = cur.dz - cur.z[j];
                /* the layer above where delta_z > 0 or at the lowest layer, else the layer below */
                const bool up = delta_z > 0 || l == L - 1;
                const double wg = up ? wp[j] : nxt.w[j], zg = up ? zp[j] : nxt.z[j];
                const double vg = (cur.w[j] - wg)/(cur.z[j] - zg);
                vel += delta_z*vg;
            }
            r += lrf*cur.nd[j]*sg[j]*vel;
        }
        put(res + (i64)l*G.nt, h, (TW)(r/cur.da));
#pragma unroll
        for (int j = 0; j < 3; ++j) { wp[j] = cur.w[j]; zp[j] = cur.z[j]; }
        cur = nxt;
    }
}

/* averaging.c:97-111 with averaging.c:14-39: the horizontal covariant
   component of edge e in layer l; its wind u and the w points wf and wt of
   level l at its cells are the caller's (it has loaded them) */
template <bool FLAT>
__device__ __forceinline__ double horizontal_covariant_t(const DevGrid &G, const double *w, int l, double u,
                                                         unsigned e, unsigned fr, unsigned to, double wf, double wt)
{
    const i64 vi = G.nsh + (i64)l*G.vpl;
    double r = u;
    if (!FLAT && l >= G.L - G.n_oro) {
        const double *w6 = G.ipwT + ((i64)l*8 + 6)*G.nsh, *w7 = w6 + G.nsh;
        const double *wn = w + (i64)(l + 1)*G.vpl;
        /* the lowest layer loads the surface terms and leaves them out */
        const double slope = at(G.slope + vi, e), a6 = at(w6, fr), b6 = at(w6, to), a7 = at(w7, fr), b7 = at(w7, to);
        const double nf = at(wn, fr), nt = at(wn, to);
        double c = a6*wf;
        c += b6*wt;
        if (l < G.L - 1) {
            c += a7*nf;
            c += b7*nt;
        }
        c = 0.5*c;
        r += slope*c;
    }
    return r;
}

/* calc_pot_vort = calc_rel_vort + add_f_to_rel_vort + division by the
   interpolated density (vorticities.c:18-165), and the mass flux density
   (scalar_times_vector of rho_gas and the wind, multiplications.c:35-117).
   One thread per edge walks a chunk of levels and writes the tangential
   element of each level and the rhombus element and mass flux of each layer,
   whose densities and wind the vorticity reads anyway (a kernel of its own
   took 92 us at res 7 x 26); the threads that have a cell of their number
   write the mass flux of its interior w points. */
template <bool FLAT, typename TW>
__global__ void __launch_bounds__(TPB) k_pot_vort(DevGrid G, const double *w, const double *rho, const TW *rvt,
                                                  TW *pv, TW *flux, Span sp)
{
    const Blk bk = FLAT ? linear_block() : xcd_block(sp);
    const unsigned e = bk.x*TPB + threadIdx.x;
    if (e >= (unsigned)G.nvh) return;
    const int nvh = G.nvh, nsh = G.nsh, L = G.L, vpl = G.vpl;
    const unsigned fr = G.from[e], to = G.to[e], fd = G.dfrom[e], td = G.dto[e];
    const double *nd = G.nd;
    unsigned dri[4];
    double drw[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) { dri[j] = at(G.e_rc + (i64)j*nvh, e); drw[j] = at(G.e_rw + (i64)j*nvh, e); }
    /* the edge's two cells are two of its rhombus cells: their densities come
       with the rhombus loads, and the layer above's are carried from the
       previous level, as are the covariant wind and normal distance of the
       edge in the layer above (each value is the one the reference's
       formula reads, so the arithmetic is unchanged) */
    int pf = 0, pt = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) { if (dri[j] == fr) pf = j; if (dri[j] == to) pt = j; }
    const double f_t = G.fvec[e], f_r = G.fvec[nvh + e];
    int l0, l1;
    layer_chunk(L + 1, bk.y, sp.run, l0, l1);
    if (l0 >= l1) return;
    const bool cell = e < (unsigned)nsh;
    auto cov = [&](int l, double u, double wf, double wt) {
        return horizontal_covariant_t<FLAT>(G, w, l, u, e, fr, to, wf, wt);
    };
    /* the tangential vorticity of level 1, which the top copies
       (vorticities.c:158-163); a first chunk that reaches level 1 has it */
    double rv1 = 0.0;
    if (l0 <= 1) {
        const i64 base = vpl;
        const double wf = at(w + base, fr), wt = at(w + base, to);
        const double c1 = cov(1, at(w + base + nsh, e), wf, wt), c0 = cov(0, at(w + nsh, e), at(w, fr), at(w, to));
        rv1 = 1/at(G.darea + G.dvpl, e)*(
            - at(nd + base + nsh, e)*c1
            + at(nd + base, fr)*wf
            + at(nd + nsh, e)*c0
            - at(nd + base, to)*wt);
    }
    /* layer l-1 at the edge: density of both cells, covariant wind, normal distance */
    double rf_m = 0.0, rt_m = 0.0, cv_m = 0.0, nd_m = 0.0;
    if (l0 >= 1) {
        const double *rm = rho + (i64)(l0 - 1)*nsh, *wm = w + (i64)(l0 - 1)*vpl;
        rf_m = at(rm, fr);
        rt_m = at(rm, to);
        cv_m = cov(l0 - 1, at(wm + nsh, e), FLAT ? 0.0 : at(wm, fr), FLAT ? 0.0 : at(wm, to));
        nd_m = at(nd + nsh + (i64)(l0 - 1)*vpl, e);
    }
    double rc_m = (cell && l0 >= 1) ? at(rho + (i64)(l0 - 1)*nsh, e) : 0.0;   /* the cell's density in the layer above */
    for (int l = l0; l < l1; ++l) {
        if (l == L) {
            /* the lowest level (vorticities.c:158-163 and the surface density extrapolation) */
            const double rv = 1/at(G.darea + (i64)l*G.dvpl, e)*nd_m*cv_m;
            const double *ra = rho + (i64)(l - 1)*nsh, *rb = ra - nsh;
            const double af = at(ra, fr), at_ = at(ra, to), bf = at(rb, fr), bt = at(rb, to);
            const double dv = 0.5*(af + at_)
                              + (0.5*(bf + bt) - 0.5*(af + at_))
                              /G.pv_sfc_dz1[e]*G.pv_sfc_dz2[e];
            put(pv + (i64)l*2*nvh, e, (TW)((rv + f_t)/dv));
            break;
        }
        /* loads of level l */
        const i64 base = (i64)l*vpl, db = nvh + (i64)l*G.dvpl;
        const double *rl = rho + (i64)l*nsh;
        double r4[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) r4[j] = at(rl, dri[j]);
        const double nd0 = at(nd + base + nsh, e), nd1 = at(nd + base, fr), nd3 = at(nd + base, to);
        const double w1 = at(w + base, fr), w3 = at(w + base, to);
        const double da_e = at(G.darea + (i64)l*G.dvpl, e), af = at(G.darea + db, fd), at_ = at(G.darea + db, td);
        const TW *rvl = rvt + (i64)l*G.nt;
        const double rvf = (double)at(rvl, fd), rvd = (double)at(rvl, td);
        const double u0 = at(w + base + nsh, e);
        double rc = 0.0, wc = 0.0;
        if (cell) { rc = at(rl, e); wc = at(w + base, e); }
        const double cv0 = cov(l, u0, w1, w3);
        const double rf = pf == 0 ? r4[0] : (pf == 1 ? r4[1] : (pf == 2 ? r4[2] : r4[3]));
        const double rt = pt == 0 ? r4[0] : (pt == 1 ? r4[1] : (pt == 2 ? r4[2] : r4[3]));
        /* tangential element at level l; the top copies level 1 (vorticities.c:158-163) */
        double rv;
        if (l <= 1) rv = rv1;
        else rv = 1/da_e*(- nd0*cv0 + nd1*w1 + nd_m*cv_m - nd3*w3);
        double dv;
        if (l == 0) {
            const double rf1 = at(rl + nsh, fr), rt1 = at(rl + nsh, to);
            dv = 0.5*(rf + rt) + (0.5*(rf + rt) - 0.5*(rf1 + rt1))/G.pv_top_dz1[e]*G.pv_top_dz2[e];
        } else dv = 0.25*(rf_m + rt_m + rf + rt);
        put(pv + (i64)l*2*nvh, e, (TW)((rv + f_t)/dv));
        /* rhombus element of layer l */
        const double rr = (af*rvf + at_*rvd)/(af + at_);
        double dr = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) dr += drw[j]*r4[j];
        put(pv + (i64)l*2*nvh + nvh, e, (TW)((rr + f_r)/dr));
        put(flux + base + nsh, e, (TW)((0.5*(rt + rf))*u0));
        if (cell) {
            if (l >= 1) put(flux + base, e, (TW)((0.5*(rc_m + rc))*wc));
            rc_m = rc;
        }
        rf_m = rf; rt_m = rt; cv_m = cv0; nd_m = nd0;
    }
}

/* vorticity_flux.c:16-187, horizontal part: one thread per edge and chunk of
   layers.  TEND: with the kinetic-energy gradient (gradient_operators.c:14-33)
   and the tendency and wind update of vector_tendencies_expl.c:74-131 and
   manage_rkhevi.c:67-75, whose other terms are there: the flux and the
   gradient are stored (the next step's first substep reads them) but not read
   back, and the terrain weights of both are loaded once. */
template <bool FLAT, typename TW, bool TEND>
/* at most two waves per SIMD: the register budget lets every gather of a
   layer issue in one batch (measured faster than four waves with the gathers
   issued in pairs) */
__global__ void __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_vorticity_flux_e(DevGrid G, const TW *F, const TW *pv, TW *out, DevWorkT<TW> W, Mom<TW> m, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned e = bk.x*TPB + threadIdx.x;
    if (e >= (unsigned)G.nvh) return;
    const int nsh = G.nsh, nvh = G.nvh;
    double tw[10];
    unsigned ti[10], tm[10];
#pragma unroll
    for (int j = 0; j < 10; ++j) {
        ti[j] = at(G.e_ti + (i64)j*nvh, e);
        tm[j] = at(G.e_tm + (i64)j*nvh, e);
        tw[j] = at(G.e_tw + (i64)j*nvh, e);
    }
    const unsigned fr = G.from[e], to = G.to[e];
    /* next to a pentagon a side has four terms: its fifth slot reads the
       first slot's (valid) entries and adds -0.0, the exact identity of IEEE
       addition, so every load of a layer issues without a branch */
    const bool pent_f = fr < GAME_N_PENT, pent_t = to < GAME_N_PENT;
    int l0, l1;
    layer_chunk(G.L, bk.y, sp.run, l0, l1);
    if (l0 >= l1) return;
    /* the w-point terms of layer l+1 are those of layer l+1's upper level:
       carried to the next layer instead of loaded again */
    double Ff = (double)at(F + (i64)l0*G.vpl, fr), Ft = (double)at(F + (i64)l0*G.vpl, to);
    double q0 = (double)at(pv + (i64)l0*2*nvh, e);
    const double old_w = TEND ? 1.0 - m.new_w : 0.0;
    EdgeCarry carry;
    for (int l = l0; l < l1; ++l) {
        const i64 vi = nsh + (i64)l*G.vpl;
        const TW *Fl = F + vi, *pl = pv + nvh + (i64)l*2*nvh;
        double Fv[10], pvv[10];
#pragma unroll
        for (int j = 0; j < 10; ++j) { Fv[j] = (double)at(Fl, ti[j]); pvv[j] = (double)at(pl, tm[j]); }
        const double pve = (double)at(pl, e);
        /* inner-product weights 6 and 7 of the two cells in layer l */
        const double *w6 = G.ipwT + ((i64)l*8 + 6)*nsh, *w7 = w6 + nsh;
        const double w6f = at(w6, fr), w6t = at(w6, to), w7f = at(w7, fr), w7t = at(w7, to);
        const double q1 = (double)at(pl + nvh, e);
        const double Ff1 = (double)at(F + (i64)(l + 1)*G.vpl, fr), Ft1 = (double)at(F + (i64)(l + 1)*G.vpl, to);
        double comb = 0.0, wo = 0.0, td_old = 0.0;
        if (TEND) {
            comb = (double)at(W.pgrad_comb + vi, e);
            wo = at(m.wind_old + vi, e);
            if (old_w != 0.0) td_old = (double)at(m.td_old + vi, e);
        }
        double o = 0;
#pragma unroll
        for (int j = 0; j < 10; ++j) {
            const bool pent = j < 5 ? pent_f : pent_t;
            /* slots 2 and 7 average with the edge's own PV, except next to a pentagon */
            double t = ((j == 2 || j == 7) && !pent) ? tw[j]*Fv[j]*0.5*(pvv[j] + pve) : tw[j]*Fv[j]*pvv[j];
            if ((j == 4 || j == 9) && pent) t = -0.0;
            o += t;
        }
        o -= 0.5*w6f*Ff*q0;
        o -= 0.5*w6t*Ft*q0;
        o -= 0.5*w7f*Ff1*q1;
        o -= 0.5*w7t*Ft1*q1;
        const TW pvt = (TW)o;
        if (TEND) {
            const TW vg = (TW)grad_edge_walk<FLAT, TW>(G, W.vsq, l, l0, e, fr, to, carry);
            double tv = m.new_w*(
                comb   /* ohw*old - chw*(nl + l) */
                + (double)pvt
                - 0.5*(double)vg);
            if (old_w != 0.0) tv = old_w*td_old + tv;
            put(W.vsq_grad + vi, e, vg);
            put(m.td + vi, e, (TW)tv);
            put(m.wind_new + vi, e, wo + m.dt*tv);
        }
        put(out + vi, e, pvt);
        Ff = Ff1; Ft = Ft1; q0 = q1;
    }
}

/* vorticity_flux.c:373-417, vertical part: one thread per cell and chunk of
   levels 0..L.  NC > 0: with the kinetic-energy gradient at the interior w
   points (gradient_operators.c:35-54), the condensates' pressure gradient of
   the densities rho (calc_pressure_grad_condensates_v; null: it is there) and
   the tendency (vector_tendencies_expl.c:74-131); NC is the number of
   constituents */
template <typename TW, int RUN, int NC>
__global__ void __launch_bounds__(TPB) k_vorticity_flux_w(DevGrid G, const TW *F, const TW *pv, TW *out, DevWorkT<TW> W,
                                                          Mom<TW> m, const double *rho, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned h = bk.x*TPB + threadIdx.x;
    if (h >= (unsigned)G.nsh) return;
    const int nsh = G.nsh, nvh = G.nvh;
    const int ne = h < GAME_N_PENT ? 5 : 6;
    /* a fixed six edges: a pentagon's sixth slot reads its first edge and
       adds -0.0, the exact identity of IEEE addition */
    unsigned adj[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) adj[j] = at(G.c_e + (i64)j*G.nsh, h);
    const int L = G.L, vpl = G.vpl;
    /* level l sums the terms of layers l - 1 and l; the flux and weights of
       layer l are carried to level l + 1 instead of loaded again */
    auto load_layer = [&](int l, double *Fx, double *Wx) {
        const TW *Fl = F + nsh + (i64)l*vpl;
        const double *wl = G.ipwT + (i64)l*8*nsh;
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            Fx[j] = (double)at(Fl, adj[j]);
            Wx[j] = at(wl + (i64)j*nsh, h);
        }
    };
    int l0, l1;
    layer_chunk(L + 1, bk.y, sp.run, l0, l1);
    if (l0 >= l1) return;
    double Fm[6], Wm[6];
    const int lm = l0 >= 1 ? l0 - 1 : 0;
    load_layer(lm, Fm, Wm);
    /* kinetic energy and gas fraction of the layer above, carried */
    double vs_m = 0.0, d_m = 0.0;
    const double old_w = NC > 0 ? 1.0 - m.new_w : 0.0;
    if constexpr (NC > 0) {
        vs_m = (double)at(W.vsq + (i64)lm*nsh, h);
        if (rho) d_m = gas_fraction_at<NC>(G, rho, (i64)lm*nsh, h);
    }
    /* a level's results: flux, and at interior levels the gradient, the
       condensates' term and the tendency */
    struct Out { double flux; TW vg, pgc, td; };
    auto level = [&](int l) {
        Out r;
        double Fc[6], Wc[6], q[6];
        const int lc = l <= L - 1 ? l : L - 1;
        load_layer(lc, Fc, Wc);
        const TW *pl = pv + (i64)l*2*nvh;
#pragma unroll
        for (int j = 0; j < 6; ++j) q[j] = (double)at(pl, adj[j]);
        double vs = 0.0, d = 0.0, comb = 0.0, td_old = 0.0, nd = 1.0, gm = 0.0, pgc = 0.0;
        const i64 row = (i64)l*vpl;
        if constexpr (NC > 0) {
            vs = (double)at(W.vsq + (i64)lc*nsh, h);
            comb = (double)at(W.pgrad_comb + row, h);
            nd = at(G.nd + row, h);
            if (old_w != 0.0) td_old = (double)at(m.td_old + row, h);
            if (rho) { gm = at(G.gm + row, h); d = gas_fraction_at<NC>(G, rho, (i64)lc*nsh, h); }
            else pgc = (double)at(W.pgc_v + row, h);
        }
        double vw = 0.5;
        if (l == 0 || l == L) vw = 1;
        double o = 0;
        if (l >= 1) {
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                double t = vw*Wm[j]*Fm[j]*q[j];
                if (j >= ne) t = -0.0;
                o += t;
            }
        }
        if (l <= L - 1) {
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                double t = vw*Wc[j]*Fc[j]*q[j];
                if (j >= ne) t = -0.0;
                o += t;
            }
        }
#pragma unroll
        for (int j = 0; j < 6; ++j) { Fm[j] = Fc[j]; Wm[j] = Wc[j]; }
        r.flux = o;
        if constexpr (NC > 0) {
            r.vg = (TW)((vs_m - vs)/nd);
            if (rho) {
                const double c_up = d_m - 1.0, c_lo = d - 1.0;
                pgc = (double)(TW)((0.5*(c_up + c_lo))*gm);
            }
            r.pgc = (TW)pgc;
            double tv = m.new_w*(
                comb   /* -cvw*(nl + l) */
                + (double)(TW)o
                - 0.5*(double)r.vg
                + pgc);
            if (old_w != 0.0) tv = old_w*td_old + tv;
            r.td = (TW)tv;
            vs_m = vs;
            d_m = d;
        }
        return r;
    };
    auto store = [&](int l, const Out &r) {
        const i64 row = (i64)l*vpl;
        put(out + row, h, (TW)r.flux);
        if constexpr (NC > 0) {
            const bool inner = l >= 1 && l <= L - 1;
            if (inner) {
                put(W.vsq_grad + row, h, r.vg);
                if (rho) put(W.pgc_v + row, h, r.pgc);
            }
            put(m.td + row, h, inner ? r.td : (TW)0.0);
        }
    };
    if constexpr (RUN > 0) {
        /* chunks of at most RUN levels: every level before any store, so no
           store orders a later level's loads (a step past the chunk repeats
           its last level) */
        Out o[RUN];
#pragma unroll
        for (int t = 0; t < RUN; ++t) o[t] = level(l0 + t < l1 ? l0 + t : l1 - 1);
#pragma unroll
        for (int t = 0; t < RUN; ++t)
            if (l0 + t < l1) store(l0 + t, o[t]);
    } else
        for (int l = l0; l < l1; ++l) store(l, level(l));
}

/* inner_product.c:13-43, one thread per box (107 us at res 7 x 26 with two
   layers per thread, which share the w points between them, 103 with one) */
template <typename TW>
__global__ void __launch_bounds__(TPB) k_inner_product(DevGrid G, const double *a, const double *b, TW *out, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned h = bk.x*TPB + threadIdx.x;
    if (h >= (unsigned)G.nsh) return;
    const int l = (int)bk.y, ne = h < GAME_N_PENT ? 5 : 6;
    /* a fixed six edges: a pentagon's sixth slot reads its first edge and
       adds -0.0, the exact identity of IEEE addition */
    unsigned adj[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) adj[j] = at(G.c_e + (i64)j*G.nsh, h);
    const double *w = G.ipwT + (i64)l*8*G.nsh;   /* weight j in row w + j*nsh */
    const i64 up = (i64)l*G.vpl, lo = up + G.vpl, vi = up + G.nsh;
    const double au = at(a + up, h), bu = at(b + up, h), al = at(a + lo, h), bl = at(b + lo, h);
    double o = 0;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        double t = at(w + j*(i64)G.nsh, h)*at(a + vi, adj[j])*at(b + vi, adj[j]);
        if (j >= ne) t = -0.0;
        o += t;
    }
    o += at(w + 6*(i64)G.nsh, h)*au*bu;
    o += at(w + 7*(i64)G.nsh, h)*al*bl;
    put(out + (i64)l*G.nsh, h, (TW)o);
}

/* grad (gradient_operators.c:56-74) of a scalar field: edges (one thread per
   edge and chunk of layers) */
template <bool FLAT, typename TW>
__global__ void __launch_bounds__(TPB) k_grad_e(DevGrid G, const TW *f, TW *out, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned e = bk.x*TPB + threadIdx.x;
    if (e >= (unsigned)G.nvh) return;
    const unsigned fr = G.from[e], to = G.to[e];
    int l0, l1;
    layer_chunk(G.L, bk.y, sp.run, l0, l1);
    EdgeCarry carry;
    for (int l = l0; l < l1; ++l)
        put(out + G.nsh + (i64)l*G.vpl, e, (TW)grad_edge_walk<FLAT, TW>(G, f, l, l0, e, fr, to, carry));
}

/* grad, interior w points (gradient_operators.c:35-54) */
template <typename TW>
__global__ void __launch_bounds__(TPB) k_grad_w(DevGrid G, const TW *f, TW *out, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned h = bk.x*TPB + threadIdx.x;
    if (h >= (unsigned)G.nsh) return;
    const int lev = (int)bk.y + 1;
    const TW *lo = f + (i64)lev*G.nsh;
    put(out + (i64)lev*G.vpl, h, (TW)(((double)at(lo - G.nsh, h) - (double)at(lo, h))/at(G.nd + (i64)lev*G.vpl, h)));
}

/* the slot-major tables of DevGrid, one thread per cell, edge and triangle of
   its number */
__global__ void __launch_bounds__(TPB) k_tables(DevGrid G, unsigned *c_e, unsigned *c_n, unsigned *c_from, unsigned *e_ti,
                                                unsigned *e_tm, double *e_tw, unsigned *e_rc, double *e_rw, unsigned *t_e)
{
    const int t = (int)(blockIdx.x*TPB + threadIdx.x);
    if (t < G.nsh) {
        const int ne = t < GAME_N_PENT ? 5 : 6;
        unsigned bits = 0;
        for (int j = 0; j < 6; ++j) {
            const int e = G.adj[6*t + (j < ne ? j : 0)], f = G.from[e];
            c_e[(i64)j*G.nsh + t] = (unsigned)e;
            c_n[(i64)j*G.nsh + t] = (unsigned)(j < ne ? (f == t ? G.to[e] : f) : t);
            if (j < ne && G.sgn[6*t + j] > 0) bits |= 1u << j;
        }
        c_from[t] = bits;
    }
    if (t < G.nvh) {
        for (int j = 0; j < 10; ++j) {
            const bool pent = (j < 5 ? G.from[t] : G.to[t]) < GAME_N_PENT;
            const i64 o = 10*(i64)t + (pent && (j == 4 || j == 9) ? j - 4 : j);
            e_ti[(i64)j*G.nvh + t] = (unsigned)G.ti[o];
            e_tm[(i64)j*G.nvh + t] = (unsigned)G.tmc[o];
            e_tw[(i64)j*G.nvh + t] = G.tw[10*(i64)t + j];
        }
        for (int j = 0; j < 4; ++j) {
            e_rc[(i64)j*G.nvh + t] = (unsigned)G.dri[4*(i64)t + j];
            e_rw[(i64)j*G.nvh + t] = G.drw[4*(i64)t + j];
        }
    }
    if (t < G.nt)
        for (int j = 0; j < 3; ++j)
            t_e[(i64)j*G.nt + t] = (unsigned)G.vit[3*t + j] | (G.vst[3*t + j] < 0 ? 0x80000000u : 0u);
}

/* the weights -0.5*ipw*slope of the corrections, cell-major per terrain level
   and edge slot (a pentagon's sixth slot holds its first edge's, unused):
   grid constants, formed once */
__global__ void __launch_bounds__(TPB) k_vcc_weights(DevGrid G, double *vcw)
{
    const i64 t = (i64)blockIdx.x*TPB + threadIdx.x;
    if (t >= (i64)G.n_oro*6*G.nsh) return;
    const int q = (int)(t/G.nsh), h = (int)(t - (i64)q*G.nsh), k = q/6, j = q - 6*k, l = G.L - G.n_oro + k;
    const int jj = j < (h < GAME_N_PENT ? 5 : 6) ? j : 0;
    vcw[t] = -0.5*G.ipwT[((i64)l*8 + jj)*G.nsh + h]*G.slope[G.nsh + (i64)l*G.vpl + G.adj[6*h + jj]];
}

/* Vertical contravariant corrections (averaging.c:41-95) of the three fields
   divv_h and divv_h_tracer need in the terrain-following levels L-n_oro..L-1:
   the wind (tracers, divergences.c:94-145), the gas mass flux and its
   rhotheta_v flux (divergences.c:41-59); the fluxes are formed on the fly
   exactly as scalar_times_vector_h forms them (multiplications.c:45-67).  MOIST:
   with the correction of the wind itself, which the tracers take */
template <bool MOIST>
__global__ void __launch_bounds__(TPB) k_vcc(DevGrid G, DevState s, double *vcc, Span sp)
{
    /* one thread per cell walks a chunk of the terrain levels.  The
       correction at level lev sums the cell's edge terms of layer lev - 1 and
       then of layer lev, starting from zero (from layer lev alone at the top
       terrain level): the running sum of layer lev - 1's terms is carried to
       the next level, so each layer's edge terms are formed once, and the sums
       are the reference's in the reference's order */
    const Blk bk = xcd_block(sp);
    const unsigned h = bk.x*TPB + threadIdx.x;
    if (h >= (unsigned)G.nsh) return;
    const int nsh = G.nsh, L = G.L, no = G.n_oro, top = L - no;
    const i64 n = (i64)no*nsh;
    const int ne = h < GAME_N_PENT ? 5 : 6;
    const double *rg = s.rho + (i64)G.n_cond*G.s;
    /* each edge as (edge, the cell across it): the means of the two cells
       are sums of two terms, which IEEE addition forms alike in either
       order, so the cell's own density and theta_v are loaded and divided
       once per layer */
    unsigned ej[6], nb[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) { ej[j] = at(G.c_e + (i64)j*nsh, h); nb[j] = at(G.c_n + (i64)j*nsh, h); }
    int c0, c1;
    layer_chunk(no, bk.y, sp.run, c0, c1);
    if (c0 >= c1) return;
    /* one layer's inputs: the cell's density and rhotheta_v, and per edge
       the wind, the neighbour's density and rhotheta_v and the weight
       -0.5*ipw*slope, a grid constant kept cell-major (coalesced, where the
       slope is a gather) */
    struct In { double rh, rt, u[6], rn[6], rtn[6], c[6]; };
    auto load = [&](int l) {
        In x;
        const i64 sl = (i64)l*nsh, vl = nsh + (i64)l*G.vpl, cl = (i64)(l - top)*6*nsh;
        x.rh = at(rg + sl, h); x.rt = at(s.rt + sl, h);
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            x.u[j] = at(s.wind + vl, ej[j]);
            x.rn[j] = at(rg + sl, nb[j]);
            x.rtn[j] = at(s.rt + sl, nb[j]);
            x.c[j] = at(G.vcw + cl + (i64)j*nsh, h);
        }
        return x;
    };
    /* the edge terms of a loaded layer added to (aw, a1, a2) and (pw, p1, p2) */
    auto add_layer = [&](const In &x, double &aw, double &a1, double &a2, double &pw, double &p1, double &p2) {
        const double rh = x.rh, th = x.rt/rh;
        double tw[6], t1[6], t2[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            const double u = x.u[j];
            const double rn = x.rn[j];
            const double f1 = (0.5*(rh + rn))*u;
            const double f2 = (0.5*(th + x.rtn[j]/rn))*f1;
            const double c = x.c[j];
            tw[j] = c*u;
            t1[j] = c*f1;
            t2[j] = c*f2;
        }
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            if (j < ne) {
                if (MOIST) { aw += tw[j]; pw += tw[j]; }
                a1 += t1[j]; a2 += t2[j];
                p1 += t1[j]; p2 += t2[j];
            }
        }
    };
    double pw = 0.0, p1 = 0.0, p2 = 0.0;
    /* the layer above the chunk (its terms start the first level's sum),
       then the chunk's layers, each loaded before the one before it is
       summed */
    const int k_first = c0 > 0 ? c0 - 1 : c0;
    In cur = load(top + k_first);
    for (int k = k_first; k < c1; ++k) {
        In nxt = cur;
        if (k + 1 < c1) nxt = load(top + k + 1);
        if (k < c0) {
            double dw = 0.0, d1 = 0.0, d2 = 0.0;
            add_layer(cur, pw, p1, p2, dw, d1, d2);
        } else {
            double rw = pw, r1 = p1, r2 = p2;
            pw = 0.0; p1 = 0.0; p2 = 0.0;
            add_layer(cur, rw, r1, r2, pw, p1, p2);
            double *row = vcc + (i64)k*nsh;
            if (MOIST) put(row, h, rw);
            put(row + n, h, r1);
            put(row + 2*n, h, r2);
        }
        cur = nxt;
    }
}

/* scalar_tendencies_expl.c:89-177 for every constituent (diffusion off): the
   centred gas mass flux and its rhotheta_v flux, the upstream tracer fluxes,
   their divergences (divergences.c:14-148) and the RK-weighted tendencies.
   One thread per box; the edge fluxes are formed on the fly from the
   reference's own formulas, so no flux array is written.  Bound by how many
   of its loads are in flight: with the tables slot-major a box of its own per
   thread costs 13 coalesced table loads, and its 122 registers keep four waves
   per SIMD with every neighbour load of a constituent in flight, where a
   thread walking two layers needs 207 (res 7 x 26 moist, us per launch, FP64
   and mixed: 393 and 366 with the tables read through the edges, 361 and 322
   with slot-major ones and two layers per thread, 323 and 294 with one) */
template <bool FLAT, typename TW, int NC>
__global__ void __launch_bounds__(TPB) k_scalar_tend(DevGrid G, DevState s, DevWorkT<TW> W, double *td_rho,
                                                     double *td_rt, int rk, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned h = bk.x*TPB + threadIdx.x;
    if (h >= (unsigned)G.nsh) return;
    /* NC: the number of constituents as a compile-time constant (1 dry, 6 moist),
       so the constituent loop unrolls and all neighbour loads can be in flight together */
    const int nsh = G.nsh, vpl = G.vpl, L = G.L, no = G.n_oro;
    constexpr int ncc = NC > 1 ? NC - 2 : 0;
    const i64 S = G.s, nvcc = (i64)no*nsh;
    const int ne = h < GAME_N_PENT ? 5 : 6;
    /* each edge as (edge, the cell across it, whether h is its from-cell);
       the centred fluxes are symmetric in the two cells and IEEE addition
       commutes, so they come out bit for bit as the reference forms them
       from from/to.  The neighbour loops run over a fixed six: a pentagon's
       sixth slot reads valid entries (its first edge, its own cell) and adds
       -0.0, the exact identity of IEEE addition, so no branch guards a load
       and the per-edge arrays stay in registers. */
    unsigned ej[6], nb[6];
    const unsigned from_bits = at(G.c_from, h);
#pragma unroll
    for (int j = 0; j < 6; ++j) { ej[j] = at(G.c_e + (i64)j*nsh, h); nb[j] = at(G.c_n + (i64)j*nsh, h); }
    const int l = (int)bk.y;
    double orho[NC], ort;
    {
        const i64 sl = (i64)l*nsh, vl = nsh + (i64)l*vpl;
        double a[6], u[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            a[j] = at(G.area + vl, ej[j]);
            u[j] = at(s.wind + vl, ej[j]);
        }
        /* which faces carry a terrain correction (divergences.c:41-59) */
        int has_u = 0, has_l = 0;
        if (!FLAT) {
            if (l == L - no - 1) has_l = 1;
            else if (l == L - 1) has_u = 1;
            else if (l > L - no - 1) { has_u = 1; has_l = 1; }
        }
        const double vol = at(G.vol + sl, h);
        const double area_u = has_u ? at(G.area + (i64)l*vpl, h) : 0.0;
        const double area_l = has_l ? at(G.area + (i64)(l + 1)*vpl, h) : 0.0;
        /* rows of the corrections at the box's upper and lower faces */
        const double *vcu = W.vcc + (i64)(l - (L - no))*nsh, *vcl = vcu + nsh;
        /* the new tendencies are kept in registers and stored after every
           load of the layer, so no store orders the loads */
        double out_rt = 0.0;
        /* moist: c_v_mass_weighted_air (derived_quantities.c:97-115), its
           condensates' terms added as their densities come by */
        double cv = 0.0, cp[2] = {0.0, 0.0}, rho_v = 0.0;
        if constexpr (NC == 6) {
            cp[0] = (double)at(W.cpc + sl, h);
            cp[1] = (double)at(W.cpc + S + sl, h);
            rho_v = at(s.rho + (i64)(NC - 1)*S + sl, h);
        }
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const double new_w = (rk == 1 && k != ncc) ? 0.5 : 1.0, old_w = 1.0 - new_w;
            const double *rl = s.rho + (i64)k*S + sl;
            const double rho_h = at(rl, h);
            double res;
            if (k == ncc) {
                const double *rtl = s.rt + sl;
                const double th_h = at(rtl, h)/rho_h;
                double c1 = 0.0, c2 = 0.0;
#pragma unroll
                for (int j = 0; j < 6; ++j) {
                    const double rho_nb = at(rl, nb[j]);
                    /* times the edge sign +-1: exact, so a sign flip */
                    const bool pos = (from_bits >> j) & 1u;
                    double f1 = (0.5*(rho_h + rho_nb))*u[j];
                    double f2 = (0.5*(th_h + at(rtl, nb[j])/rho_nb))*f1;
                    double t1 = (pos ? f1 : -f1)*a[j], t2 = (pos ? f2 : -f2)*a[j];
                    if (j >= ne) { t1 = -0.0; t2 = -0.0; }
                    c1 += t1;
                    c2 += t2;
                }
                double v1 = 0.0, v2 = 0.0;
                if (!FLAT) {
                    if (has_u && has_l) {
                        v1 = at(vcu + nvcc, h)*area_u - at(vcl + nvcc, h)*area_l;
                        v2 = at(vcu + 2*nvcc, h)*area_u - at(vcl + 2*nvcc, h)*area_l;
                    } else if (has_l) {
                        v1 = -at(vcl + nvcc, h)*area_l;
                        v2 = -at(vcl + 2*nvcc, h)*area_l;
                    } else if (has_u) {
                        v1 = at(vcu + nvcc, h)*area_u;
                        v2 = at(vcu + 2*nvcc, h)*area_u;
                    }
                }
                double div1 = 1.0/vol*(c1 + v1);
                double div2 = 1.0/vol*(c2 + v2);
                const double rg = rho_h;
                /* the gas weights are 1 and 0 in both substeps: the old
                   tendencies are neither read nor added (their product with 0
                   is a zero, the identity of the sum) */
                if constexpr (NC == 1) {
                    /* dry: every source term of the reference sum is a zero array */
                    res = new_w*(-div1);
                    out_rt = new_w*(-div2);
                } else {
                    /* the moist-air gas takes the vapour phase-transition rate
                       (scalar_tendencies_expl.c:94-99, 125-131, 174-176) */
                    double ptr_v = (double)at(W.ptr + (i64)k*S + sl, h);
                    const double th = th_h;
                    res = new_w*(-div1 + ptr_v);
                    cv += rg*GC_C_D_V;
                    cv += rho_v*GC_C_V_V;
                    double heat = (double)at(W.phr + sl, h) + (double)at(W.sed_heat + sl, h);
                    out_rt = new_w*(
                        -div2
                        + GC_C_D_V*rg/cv*heat/(GC_C_D_P*(at(G.exbg + sl, h) + at(s.ep + sl, h)))
                        + ptr_v*th);
                }
            } else {
                if (k < ncc) cv += rho_h*cp[k & 1];
                double c = 0.0;
#pragma unroll
                for (int j = 0; j < 6; ++j) {
                    /* upstream density: the from-cell for u >= 0 */
                    const bool is_from = (from_bits >> j) & 1u;
                    const double rho_nb = at(rl, nb[j]);
                    const double sv = ((u[j] >= 0.0) == is_from) ? rho_h : rho_nb;
                    const double f = sv*u[j];
                    double t = (is_from ? f : -f)*a[j];
                    if (j >= ne) t = -0.0;
                    c += t;
                }
                double v = 0.0;
                if (!FLAT) {
                    if (has_u && has_l) {
                        double cu = at(vcu, h), cl = at(vcl, h);
                        double du = (cu <= 0.0) ? at(rl - nsh, h) : rho_h;
                        double dl = (cl <= 0.0) ? rho_h : at(rl + nsh, h);
                        v = du*cu*area_u - dl*cl*area_l;
                    } else if (has_l) {
                        double cl = at(vcl, h);
                        double dl = (cl <= 0.0) ? rho_h : at(rl + nsh, h);
                        v = -dl*cl*area_l;
                    } else if (has_u) {
                        double cu = at(vcu, h);
                        double du = (cu <= 0.0) ? at(rl - nsh, h) : rho_h;
                        v = du*cu*area_u;
                    }
                }
                double div = 1.0/vol*(c + v);
                const int kp = (k == ncc + 1) ? k - 1 : k;
                /* the old tendency enters with weight 0.5 in the second
                   substep only (a uniform branch); IEEE addition commutes */
                res = new_w*(-div + (double)at(W.ptr + (i64)kp*S + sl, h));
                if (old_w != 0.0) res = old_w*at(td_rho + (i64)k*S + sl, h) + res;
            }
            orho[k] = res;
        }
        ort = out_rt;
    }
    const i64 sl = (i64)l*nsh;
#pragma unroll
    for (int k = 0; k < NC; ++k) put(td_rho + (i64)k*S + sl, h, orho[k]);
    put(td_rt + sl, h, ort);
}

/* three_band_solver_ver_waves (column_solvers.c:19-383), one column per lane.
   The coefficient rows are generated and eliminated in one downward sweep;
   the back substitution walks upwards and writes each layer as soon as both
   of its interface fluxes are known.  Quantities used in both sweeps are
   recomputed with identical arithmetic rather than stored. */
struct ColumnLayer {
    double re, rte, al, be, ga, tpe, epe;
};

__device__ __forceinline__ ColumnLayer column_layer(const DevGrid &G, const DevState &so, const DevState &sn,
                                                    const DevState &td, double dt, int rk, int i, int j)
{
    ColumnLayer c;
    i64 b = i + (i64)j*G.nsh, gi = (i64)G.n_cond*G.s;
    double vol = G.vol[b];
    double rho_o = so.rho[gi + b], rt_o = so.rt[b];
    c.re = rho_o + dt*td.rho[gi + b];
    c.rte = rt_o + dt*td.rt[b];
    if (rk == 0) {
        c.al = -rt_o/(rho_o*rho_o)/vol;
        c.be = 1.0/rho_o/vol;
        c.ga = GC_R_D/(GC_C_D_V*rt_o)*(G.exbg[b] + so.ep[b])/vol;
    } else {
        const double pdw = 0.5;
        double rho_n = sn.rho[gi + b], rt_n = sn.rt[b];
        double ao = -rt_o/(rho_o*rho_o);
        double bo = 1.0/rho_o;
        double go = GC_R_D/(GC_C_D_V*rt_o)*(G.exbg[b] + so.ep[b]);
        double an = -rt_n/(rho_n*rho_n);
        double bn = 1.0/rho_n;
        double gn = GC_R_D/(GC_C_D_V*rt_n)*(G.exbg[b] + sn.ep[b]);
        c.al = ((1.0 - pdw)*ao + pdw*an)/vol;
        c.be = ((1.0 - pdw)*bo + pdw*bn)/vol;
        c.ga = ((1.0 - pdw)*go + pdw*gn)/vol;
    }
    c.tpe = so.tp[b] + dt*vol*(c.al*td.rho[gi + b] + c.be*td.rt[b]);
    c.epe = so.ep[b] + dt*vol*c.ga*td.rt[b];
    return c;
}

/* interface values of the column at interface j (between layers j and j+1) */
__device__ __forceinline__ double theta_int_new(const DevGrid &G, const DevState &sn, int i, int j)
{
    i64 gi = (i64)G.n_cond*G.s, b = i + (i64)j*G.nsh, lo = b + G.nsh;
    return 0.5*(sn.rt[b]/sn.rho[gi + b] + sn.rt[lo]/sn.rho[gi + lo]);
}

__device__ __forceinline__ double rho_int_old(const DevGrid &G, const DevState &so, int i, int j)
{
    i64 gi = (i64)G.n_cond*G.s, b = i + (i64)j*G.nsh;
    return 0.5*(so.rho[gi + b] + so.rho[gi + b + G.nsh]);
}

template <int LT, typename TWIND>
__global__ void __launch_bounds__(128) k_ver_waves(DevGrid G, DevState so, DevState snr, DevState sn, DevState td,
                                                   const TWIND *td_wind, StepConsts K, int rk)
{
    int i = blockIdx.x*128 + threadIdx.x;
    if (i >= G.nsh) return;
    const int L = LT > 0 ? LT : G.L;
    const int nsh = G.nsh, vpl = G.vpl;
    const i64 gi = (i64)G.n_cond*G.s;
    const double dt = K.dt, iw = K.impl_weight;
    const double dt2 = dt*dt;
    const double *zs = G.zs, *exbg = G.exbg, *vol = G.vol, *area = G.area;
    double ep[(LT > 0 ? LT : GAME_MAX_LAYERS) - 1], x[(LT > 0 ? LT : GAME_MAX_LAYERS) - 1];

    /* downward sweep: build row j and eliminate it (column_solvers.c:141-189, 641-660) */
    ColumnLayer ca = column_layer(G, so, snr, td, dt, rk, i, 0);   /* layer j */
    ColumnLayer cb = column_layer(G, so, snr, td, dt, rk, i, 1);   /* layer j+1 */
    double tin = theta_int_new(G, snr, i, 0), rio = rho_int_old(G, so, i, 0);
    double c_prev = 0.0;
#pragma unroll
    for (int j = 0; j < L - 1; ++j) {
        i64 b = i + (i64)j*nsh, lo = b + nsh;
        i64 wi = i + (i64)(j + 1)*vpl;
        double w_old = so.wind[wi];
        double rie = 0.5*(ca.re + cb.re);
        double d = -(tin*tin)*(ca.ga + cb.ga)
                   + 0.5*(exbg[b] - exbg[lo])*(cb.al - ca.al + tin*(cb.be - ca.be))
                   - (zs[b] - zs[lo])/(iw*dt2*GC_C_D_P*rio)
                     *(2.0/area[wi] + dt*w_old*0.5*(-1.0/vol[b] + 1.0/vol[lo]));
        double r = -(w_old + dt*(double)td_wind[wi])*(zs[b] - zs[lo])/(iw*dt2*GC_C_D_P)
                   + tin*(ca.epe - cb.epe)/dt
                   + 0.5/dt*(ca.tpe + cb.tpe)*(exbg[b] - exbg[lo])
                   - (zs[b] - zs[lo])/(iw*dt2*GC_C_D_P)*w_old*rie/rio;
        double e = 0.0, c = 0.0, tin_n = 0.0, rio_n = 0.0;
        ColumnLayer cc = cb;
        if (j < L - 2) {
            i64 l2 = lo + nsh;
            tin_n = theta_int_new(G, snr, i, j + 1);
            rio_n = rho_int_old(G, so, i, j + 1);
            /* upper diagonal e[j] and lower diagonal c[j] (column_solvers.c:173-189) */
            c = tin_n*cb.ga*tin
                + 0.5*(exbg[lo] - exbg[l2])*(cb.al + cb.be*tin)
                - (zs[lo] - zs[l2])/(iw*dt*GC_C_D_P)*0.5*so.wind[i + (i64)(j + 2)*vpl]/(vol[lo]*rio_n);
            e = tin*cb.ga*tin_n
                - 0.5*(exbg[b] - exbg[lo])*(cb.al + cb.be*tin_n)
                + (zs[b] - zs[lo])/(iw*dt*GC_C_D_P)*0.5*w_old/(vol[lo]*rio);
            cc = column_layer(G, so, snr, td, dt, rk, i, j + 2);
        }
        if (j == 0) {
            if (L - 1 > 1) ep[0] = e/d;
            x[0] = r/d;
        } else {
            double den = d - ep[j - 1]*c_prev;
            if (j < L - 2) ep[j] = e/den;
            x[j] = (r - x[j - 1]*c_prev)/den;
        }
        c_prev = c;
        ca = cb; cb = cc;
        tin = tin_n; rio = rio_n;
    }
    /* back substitution (column_solvers.c:662-667) */
#pragma unroll
    for (int j = L - 3; j >= 0; --j) x[j] = x[j] - ep[j]*x[j + 1];
    /* Klemp (2008) damping of the solved fluxes (column_solvers.c:284-298) */
#pragma unroll
    for (int j = 0; j < L - 1; ++j) x[j] = x[j]/(1.0 + dt*G.damp[(i64)j*nsh + i]);
    /* new state, layer by layer, each layer read before it is written (column_solvers.c:300-370) */
    double tin_m = 0.0, rho_new_m = 0.0, rio_m = 0.0;
#pragma unroll
    for (int j = 0; j < L; ++j) {
        i64 b = i + (i64)j*nsh;
        ColumnLayer cl = column_layer(G, so, snr, td, dt, rk, i, j);
        double tin_j = (j < L - 1) ? theta_int_new(G, snr, i, j) : 0.0;
        double rio_j = (j < L - 1) ? rho_int_old(G, so, i, j) : 0.0;
        double v = vol[b];
        double rho_n, rt_n;
        if (j == 0) {
            rho_n = cl.re + dt*(x[j])/v;
            rt_n = cl.rte + dt*(tin_j*x[j])/v;
        } else if (j == L - 1) {
            rho_n = cl.re + dt*(-x[j - 1])/v;
            rt_n = cl.rte + dt*(-tin_m*x[j - 1])/v;
        } else {
            rho_n = cl.re + dt*(-x[j - 1] + x[j])/v;
            rt_n = cl.rte + dt*(-tin_m*x[j - 1] + tin_j*x[j])/v;
        }
        double rt_o = so.rt[b];
        sn.rho[gi + b] = rho_n;
        sn.rt[b] = rt_n;
        sn.tp[b] = rt_n/rho_n - G.thbg[b];
        sn.ep[b] = so.ep[b] + v*cl.ga*(rt_n - rt_o);
        if (j >= 1) {
            i64 wi = i + (i64)j*vpl;
            double din = 0.5*(rho_new_m + rho_n);
            sn.wind[wi] = (2.0*x[j - 1]/area[wi] - din*so.wind[wi])/rio_m;
        }
        tin_m = tin_j;
        rho_new_m = rho_n;
        rio_m = rio_j;
    }
}

/* the state of box (i, j) the solver reads, loaded in one batch: old state,
   tendencies, the state snr (the new state before this substep writes it),
   volume and background exner */
struct VwBox {
    double vol, exbg, rho_o, rt_o, ep_o, tp_o, trho, trt, rho_n, rt_n, ep_n;
};

/* box at element o of the rows jb*nsh (wave-uniform) of the S fields */
__device__ __forceinline__ VwBox vw_box(const DevGrid &G, const DevState &so, const DevState &snr,
                                        const DevState &td, i64 jb, unsigned o)
{
    const i64 gi = (i64)G.n_cond*G.s + jb;
    VwBox x;
    x.vol = at(G.vol + jb, o); x.exbg = at(G.exbg + jb, o);
    x.rho_o = at(so.rho + gi, o); x.rt_o = at(so.rt + jb, o); x.ep_o = at(so.ep + jb, o); x.tp_o = at(so.tp + jb, o);
    x.trho = at(td.rho + gi, o); x.trt = at(td.rt + jb, o);
    x.rho_n = at(snr.rho + gi, o); x.rt_n = at(snr.rt + jb, o); x.ep_n = at(snr.ep + jb, o);
    return x;
}

/* column_layer's arithmetic on loaded values */
__device__ __forceinline__ ColumnLayer vw_layer(const VwBox &x, double dt, int rk)
{
    ColumnLayer c;
    c.re = x.rho_o + dt*x.trho;
    c.rte = x.rt_o + dt*x.trt;
    if (rk == 0) {
        c.al = -x.rt_o/(x.rho_o*x.rho_o)/x.vol;
        c.be = 1.0/x.rho_o/x.vol;
        c.ga = GC_R_D/(GC_C_D_V*x.rt_o)*(x.exbg + x.ep_o)/x.vol;
    } else {
        const double pdw = 0.5;
        double ao = -x.rt_o/(x.rho_o*x.rho_o);
        double bo = 1.0/x.rho_o;
        double go = GC_R_D/(GC_C_D_V*x.rt_o)*(x.exbg + x.ep_o);
        double an = -x.rt_n/(x.rho_n*x.rho_n);
        double bn = 1.0/x.rho_n;
        double gn = GC_R_D/(GC_C_D_V*x.rt_n)*(x.exbg + x.ep_n);
        c.al = ((1.0 - pdw)*ao + pdw*an)/x.vol;
        c.be = ((1.0 - pdw)*bo + pdw*bn)/x.vol;
        c.ga = ((1.0 - pdw)*go + pdw*gn)/x.vol;
    }
    c.tpe = x.tp_o + dt*x.vol*(c.al*x.trho + c.be*x.trt);
    c.epe = x.ep_o + dt*x.vol*c.ga*x.trt;
    return c;
}

/* The same solve with NCOL columns per block and a group of NCOL lanes for
   every VR_PER boxes of them, in three phases:
     1. each group walks its boxes and builds their rows of the three-band
        system (row j couples interfaces j - 1, j, j + 1) into LDS, forming
        each box's linearisation (column_layer, nine divisions at rk 1) once;
     2. one lane per column eliminates and substitutes back in LDS, then every
        group damps its own rows' solution;
     3. each group forms the new state of its boxes.
   The kernel is bound by its loads and by the divisions (about 26 per box,
   half its time at res 7), so a box is linearised once: its explicit density,
   rhotheta_v and gamma wait for phase 3 in LDS, the interface theta and
   density in registers, and only what those do not hold (volume, old exner
   and rhotheta_v, area, old wind, background) is loaded again, during the
   elimination.  Four boxes per group keep three waves per SIMD (166
   registers; all of it in registers needs 206 and spills below that) and make
   a block 144 to 256 threads at any depth; the columns per block (64 up to 16
   layers, 32 up to 32, 16 beyond) keep its LDS under 56 KiB: three blocks per
   CU (46 KiB at 26 layers) or two (55 KiB at 16, 32 and 63).  A lane's loads take its column and the distance of its group from the
   wave's first row as one offset to rows that are the same for the wave.
   Against the kernels for 26 and 55 layers (runs of seven boxes, the state
   read and linearised again in phase 3) and the one for other depths, us per
   launch: res 7 x 26 206 -> 195, res 6 x 26 72 -> 65, res 4 x 26 23 -> 17,
   res 5 x 41 41 -> 33, res 6 x 55 141 -> 144.  Every quantity keeps the
   arithmetic of k_ver_waves, so the two agree bit for bit. */
#define VR_PER 4
__host__ __device__ constexpr int vr_ncol(int layers) { return layers <= 16 ? 64 : (layers <= 32 ? 32 : 16); }
static int vr_threads(int layers) { return (layers + VR_PER - 1)/VR_PER*vr_ncol(layers); }

template <int NCOL, typename TWIND>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) k_ver_waves_run(DevGrid G, DevState so, DevState snr, DevState sn,
                                                       DevState td, const TWIND *td_wind, StepConsts K, int rk)
{
    extern __shared__ double lds[];
    const int L = G.L, NI = L - 1, nsh = G.nsh, vpl = G.vpl;
    const double dt = K.dt, iw = K.impl_weight;
    const double dt2 = dt*dt;
    const int i0 = (int)xcd_x()*NCOL;
    if (i0 >= nsh) return;
    /* the row above the wave's first (uniform; the first itself at the top),
       and this lane's group's first row */
    const int jf = __builtin_amdgcn_readfirstlane((int)threadIdx.x/64)*(64/NCOL)*VR_PER, jw = jf > 0 ? jf - 1 : 0;
    const int j0 = (int)threadIdx.x/NCOL*VR_PER, col = (int)threadIdx.x%NCOL;
    const bool live = i0 + col < nsh;
    const int i = live ? i0 + col : nsh - 1;
    const i64 jb = (i64)jw*nsh, wb = (i64)jw*vpl, gi = (i64)G.n_cond*G.s + jb;
    /* offsets from row jw to row or level j >= jw of column i, clamped to the last */
    auto os = [&](int j) { return (unsigned)((j < L ? j : L - 1) - jw)*(unsigned)nsh + (unsigned)i; };
    auto ow = [&](int lev) { return (unsigned)((lev < L ? lev : L) - jw)*(unsigned)vpl + (unsigned)i; };
    double *cc = lds, *dd = lds + NI*NCOL, *ee = lds + 2*NI*NCOL, *rr = lds + 3*NI*NCOL;

    /* what phase 3 needs of the group's boxes (LDS) and, at index t + 1, of the
       interface below box j0 + t; index 0 and k_re0 are the box above the group */
    double k_re0, k_tin[VR_PER + 1], k_rio[VR_PER + 1];
    double *p_re = lds + 4*NI*NCOL, *p_rte = p_re + L*NCOL, *p_vga = p_rte + L*NCOL;
    /* phase 1: rows j0 .. j0 + VR_PER - 1 (column_solvers.c:141-189) */
    {
        VwBox A = vw_box(G, so, snr, td, jb, os(j0)), B = vw_box(G, so, snr, td, jb, os(j0 + 1));
        double za = at(G.zs + jb, os(j0)), zb = at(G.zs + jb, os(j0 + 1));
        /* the box above (the group's own first box at the top, unused) */
        const unsigned om = os(j0 > 0 ? j0 - 1 : 0);
        const double rho_om = at(so.rho + gi, om), trho_m = at(td.rho + gi, om);
        const double rt_nm = at(snr.rt + jb, om), rho_nm = at(snr.rho + gi, om);
        k_re0 = rho_om + dt*trho_m;
        ColumnLayer ca = vw_layer(A, dt, rk), cb = vw_layer(B, dt, rk);
        auto keep = [&](int j, const VwBox &x, const ColumnLayer &c) {
            if (j < L) { const int ix = j*NCOL + col; p_re[ix] = c.re; p_rte[ix] = c.rte; p_vga[ix] = x.vol*c.ga; }
        };
        keep(j0, A, ca);
        keep(j0 + 1, B, cb);
        double th_a = A.rt_n/A.rho_n, th_b = B.rt_n/B.rho_n;
        k_tin[0] = 0.5*(rt_nm/rho_nm + th_a);
        k_rio[0] = 0.5*(rho_om + A.rho_o);
#pragma unroll
        for (int t = 0; t < VR_PER; ++t) {
            const int j = j0 + t;
            const unsigned o2 = os(j + 2), wi = ow(j + 1);
            const VwBox C = vw_box(G, so, snr, td, jb, o2);
            const double zc = at(G.zs + jb, o2);
            const double w_old = at(so.wind + wb, wi), tdw = (double)at(td_wind + wb, wi), a_w = at(G.area + wb, wi);
            const double w_old2 = at(so.wind + wb, ow(j + 2 < L ? j + 2 : L - 1));   /* w at level j+2 (interface j+1) */
            const double th_c = C.rt_n/C.rho_n;
            const double tin = 0.5*(th_a + th_b), rio = 0.5*(A.rho_o + B.rho_o);
            const double rie = 0.5*(ca.re + cb.re);
            const double d = -(tin*tin)*(ca.ga + cb.ga)
                             + 0.5*(A.exbg - B.exbg)*(cb.al - ca.al + tin*(cb.be - ca.be))
                             - (za - zb)/(iw*dt2*GC_C_D_P*rio)
                               *(2.0/a_w + dt*w_old*0.5*(-1.0/A.vol + 1.0/B.vol));
            const double r = -(w_old + dt*tdw)*(za - zb)/(iw*dt2*GC_C_D_P)
                             + tin*(ca.epe - cb.epe)/dt
                             + 0.5/dt*(ca.tpe + cb.tpe)*(A.exbg - B.exbg)
                             - (za - zb)/(iw*dt2*GC_C_D_P)*w_old*rie/rio;
            double e = 0.0, c = 0.0;
            if (j < L - 2) {
                const double tin_n = 0.5*(th_b + th_c), rio_n = 0.5*(B.rho_o + C.rho_o);
                c = tin_n*cb.ga*tin
                    + 0.5*(B.exbg - C.exbg)*(cb.al + cb.be*tin)
                    - (zb - zc)/(iw*dt*GC_C_D_P)*0.5*w_old2/(B.vol*rio_n);
                e = tin*cb.ga*tin_n
                    - 0.5*(A.exbg - B.exbg)*(cb.al + cb.be*tin_n)
                    + (za - zb)/(iw*dt*GC_C_D_P)*0.5*w_old/(B.vol*rio);
            }
            if (j < NI) {
                const int idx = j*NCOL + col;
                cc[idx] = c; dd[idx] = d; ee[idx] = e; rr[idx] = r;
            }
            k_tin[t + 1] = tin; k_rio[t + 1] = rio;
            A = B; ca = cb; za = zb; th_a = th_b;
            B = C; cb = vw_layer(C, dt, rk); zb = zc; th_b = th_c;
            if (t + 2 < VR_PER) keep(j + 2, C, cb);
        }
    }
    /* what else phases 2 and 3 need, in flight during the elimination: these
       reads of the state come before the barriers, its writes after them */
    __builtin_amdgcn_sched_barrier(0);
    double k_vol[VR_PER + 1], k_epo[VR_PER], k_rto[VR_PER], k_aw[VR_PER], k_wo[VR_PER], k_thbg[VR_PER], k_damp[VR_PER];
    k_vol[0] = at(G.vol + jb, os(j0 > 0 ? j0 - 1 : 0));
#pragma unroll
    for (int t = 0; t < VR_PER; ++t) {
        const unsigned o = os(j0 + t), wi = ow(j0 + t);
        k_vol[t + 1] = at(G.vol + jb, o); k_epo[t] = at(so.ep + jb, o); k_rto[t] = at(so.rt + jb, o);
        k_aw[t] = at(G.area + wb, wi); k_wo[t] = at(so.wind + wb, wi);
        k_thbg[t] = at(G.thbg + jb, o);
        k_damp[t] = at(G.damp + jb, os(j0 + t < NI ? j0 + t : NI - 1));
    }
    __syncthreads();
    /* phase 2: Thomas algorithm (column_solvers.c:641-667), one lane per column */
    if ((int)threadIdx.x < NCOL && live) thomas_lds<NCOL>(cc, dd, ee, rr, NI, col);
    __syncthreads();
    /* Klemp (2008) damping of the solved fluxes (column_solvers.c:284-298) */
#pragma unroll
    for (int t = 0; t < VR_PER; ++t) {
        const int idx = (j0 + t)*NCOL + col;
        if (j0 + t < NI) rr[idx] = rr[idx]/(1.0 + dt*k_damp[t]);
    }
    __syncthreads();
    /* phase 3: the new state of boxes j0 .. j0 + VR_PER - 1 (column_solvers.c:300-370);
       every read of the state, which may be the one written, came before the barriers */
    double x_m = j0 >= 1 ? rr[(j0 - 1)*NCOL + col] : 0.0;
    const double x_mm = j0 >= 2 ? rr[(j0 - 2)*NCOL + col] : 0.0;
    /* the new density of the box above, with the arithmetic of its own group */
    double rho_prev = k_re0 + dt*(j0 == 1 ? x_m : -x_mm + x_m)/k_vol[0];
#pragma unroll
    for (int t = 0; t < VR_PER; ++t) {
        const int j = j0 + t;
        const double x_j = j < NI ? rr[j*NCOL + col] : 0.0;
        const double tin_m = k_tin[t], tin_j = k_tin[t + 1], v = k_vol[t + 1];
        const double sr = j == 0 ? x_j : (j == L - 1 ? -x_m : -x_m + x_j);
        const double st = j == 0 ? tin_j*x_j : (j == L - 1 ? -tin_m*x_m : -tin_m*x_m + tin_j*x_j);
        const int ix = (j < L ? j : L - 1)*NCOL + col;
        const double rho_n = p_re[ix] + dt*sr/v;
        const double rt_n = p_rte[ix] + dt*st/v;
        if (live && j < L) {
            const unsigned o = os(j);
            put(sn.rho + gi, o, rho_n);
            put(sn.rt + jb, o, rt_n);
            put(sn.tp + jb, o, rt_n/rho_n - k_thbg[t]);
            put(sn.ep + jb, o, k_epo[t] + p_vga[ix]*(rt_n - k_rto[t]));
            if (j >= 1) {
                const double din = 0.5*(rho_prev + rho_n);
                put(sn.wind + wb, ow(j), (2.0*x_m/k_aw[t] - din*k_wo[t])/k_rio[t]);
            }
        }
        x_m = x_j;
        rho_prev = rho_n;
    }
}

/* vertical fluxes of tracer k through interface jj of column i
   (column_solvers.c:414-465): fi with the old wind, fr with the new wind
   times the upstream density */
__device__ __forceinline__ void tracer_iface_flux(const DevGrid &G, const DevState &so, const DevState &sn,
                                                  const StepConsts &K, const double *rho_o, int k, int i, int jj,
                                                  double &fi, double &fr)
{
    const int nsh = G.nsh, vpl = G.vpl, ncc = G.n_cond;
    fi = so.wind[i + (i64)(jj + 1)*vpl];
    fr = sn.wind[i + (i64)(jj + 1)*vpl];
    if (k < ncc/4) { fi -= K.snow_v; fr -= K.snow_v; }
    else if (k < ncc/2) { fi -= K.rain_v; fr -= K.rain_v; }
    else if (k < ncc) { fi -= K.cloud_v; fr -= K.cloud_v; }
    double a = G.area[i + (i64)(jj + 1)*vpl];
    fi = a*fi;
    fr = a*fr;
    i64 b = i + (i64)jj*nsh;
    /* both candidates load before the sign is known: no load waits on another */
    const double d_lo = rho_o[b + nsh], d_up = rho_o[b];
    double doi = (fr >= 0.0) ? d_lo : d_up;
    fr = doi*fr;
}

/* three_band_solver_gen_densities (column_solvers.c:385-639): a block solves
   64 columns of one tracer, wave w the rows w*GD_PER .. of each, one column
   per lane, all of it in registers.
     1. every wave loads its rows at once and forms them (column_solvers.c:466-615).
        An interface has one nonzero off-diagonal, the upstream side of its
        flux: above a row that the row above depends on (e) the row's own lower
        entry c is 0.0, so the pivot d - (e/d)*c of the elimination
        (column_solvers.c:641-660) is d exactly and the quotients e/d of all
        rows are formed here, in parallel;
     2. the waves take turns downwards with x = (r - x*c)/d, the last row's x
        handed on in LDS, and upwards with x - (e/d)*x;
     3. each wave writes its clipped rows (column_solvers.c:616-637).
   What the rows' loads and the turns leave idle other blocks fill, so the
   columns in flight count: nine rows per wave take 148 registers and three
   waves at 26 layers (four blocks per CU), seven rows 120 registers and eight
   waves at 55 layers (two).  us per launch, against rows staged in LDS for one
   lane per system (five tracers per block at 26 layers, one otherwise) and
   here with 5, 7 and 9 rows:
     res 7 x 26   187 -> 229, 174, 168 (680 MB: 4.0 TB/s)
     res 5 x 26    19 -> 19.1, 15.3, 14.8
     res 5 x 41    47 -> 39.6, 30.6, 37.9
     res 6 x 55   139 -> 168, 102, 175 (360 MB: 3.5 TB/s)
   One lane per system with its column in LDS took 175, 33 and 166 us at
   res 7 x 26, 5 x 41 and 6 x 55: six waves per CU at 26 layers, two at 55. */
template <int GD_PER, int NT>
__global__ void __launch_bounds__(NT) k_gen_densities(DevGrid G, DevState so, DevState sn, DevState td, StepConsts K)
{
    __shared__ double hand[64], hand_ep[64];
    const int L = G.L, nsh = G.nsh, ncc = G.n_cond, vpl = G.vpl;
    /* the tracer is the fast block index: the blocks of one group of columns
       run side by side on one XCD and share the wind, area and volume columns in L2 */
    const unsigned ntr = (unsigned)G.n_const - 1, blk = xcd_x(), grp = blk/ntr;
    const int tr = (int)(blk - grp*ntr);
    const int k = tr < ncc ? tr : tr + 1;   /* skip the gas */
    const unsigned lane = threadIdx.x & 63u;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), nw = (int)(blockDim.x >> 6);
    /* lanes past the last column solve the last one again and write nothing */
    const bool mine = grp*64 + lane < (unsigned)nsh;
    const unsigned i = mine ? grp*64 + lane : (unsigned)nsh - 1;
    const double iw = 0.5, ew = 1.0 - iw, dt = K.dt;
    const double *rho_o = so.rho + (i64)k*G.s, *trho = td.rho + (i64)k*G.s;
    const bool cond = k < ncc;
    const double sv = k < ncc/4 ? K.snow_v : (k < ncc/2 ? K.rain_v : (cond ? K.cloud_v : 0.0));
    /* rows j0 .. j0 + GD_PER - 1 < L; rows past the last are loaded as the last
       and not used (every wave has at least one row) */
    const int j0 = w*GD_PER;
    double r[GD_PER], d[GD_PER], c[GD_PER], ep[GD_PER];
    {
        const int jm = j0 > 0 ? j0 - 1 : 0;
        const i64 wm = (i64)(jm + 1)*vpl;
        const double wo_m = at(so.wind + wm, i), wn_m = at(sn.wind + wm, i), a_m = at(G.area + wm, i);
        const double up_m = at(rho_o + (i64)jm*nsh, i), r_low = at(rho_o + (i64)(L - 1)*nsh, i);
        const double a_sfc = at(G.area + (i64)L*vpl, i);
        double rb = at(rho_o + (i64)j0*nsh, i), q = at(G.idv + (i64)j0*nsh, i);   /* q = iw*dt/vol, kept for the current dt */
        double wo[GD_PER], wn[GD_PER], a[GD_PER], dlo[GD_PER], qlo[GD_PER], v[GD_PER], tb[GD_PER];
#pragma unroll
        for (int t = 0; t < GD_PER; ++t) {
            const int j = j0 + t < L ? j0 + t : L - 1, jc = j < L - 1 ? j : L - 2;
            const i64 wi = (i64)(jc + 1)*vpl, b = (i64)j*nsh, lo = (i64)(jc + 1)*nsh;
            wo[t] = at(so.wind + wi, i); wn[t] = at(sn.wind + wi, i); a[t] = at(G.area + wi, i);
            dlo[t] = at(rho_o + lo, i); qlo[t] = at(G.idv + lo, i);
            v[t] = at(G.vol + b, i); tb[t] = at(trho + b, i);
        }
        /* the interface above the first row (column_solvers.c:414-465): fi with
           the old wind, fr with the new one times the upstream density; the
           top row has none: no fi, and an fr and a c of zero */
        double fi_m = -1.0, fr_m = 0.0, c_m = 0.0;
        if (j0 > 0) {
            const double fn = a_m*(wn_m - sv);
            fi_m = a_m*(wo_m - sv);
            fr_m = (fn >= 0.0 ? rb : up_m)*fn;
            c_m = fi_m >= 0.0 ? 0.0 : q*fi_m;
        }
#pragma unroll
        for (int t = 0; t < GD_PER; ++t) {
            const bool last = j0 + t >= L - 1;
            const double fn = a[t]*(wn[t] - sv);
            const double doi = fn >= 0.0 ? dlo[t] : rb;
            const double fi = last ? 0.0 : a[t]*(wo[t] - sv), fr = last ? -0.0 : doi*fn;
            double dj = 1.0, rj = rb + dt*tb[t];
            if (fi_m >= 0.0) dj += q*fi_m;
            if (fi < 0.0) dj -= q*fi;
            rj += ew*dt*(-fr_m + fr)/v[t];
            if (last && cond) {
                dj += iw*sv*dt*a_sfc/v[t];
                rj += -ew*sv*dt*r_low*a_sfc/v[t];
            }
            const bool up = fi >= 0.0;
            r[t] = rj;
            /* dj itself but for an infinite wind, whose NaN then goes on as in
               the elimination */
            d[t] = t > 0 ? dj - ep[t > 0 ? t - 1 : 0]*c_m : dj;
            c[t] = c_m;
            ep[t] = up && !last ? (-q)*fi/dj : 0.0;
            c_m = up ? 0.0 : qlo[t]*fi;
            fi_m = fi;
            fr_m = fr;
            rb = dlo[t];
            q = qlo[t];
        }
    }
    double x = 0.0;
    for (int s = 0; s < nw; ++s) {
        if (w == s) {
            if (s > 0) { x = hand[lane]; d[0] -= hand_ep[lane]*c[0]; }
#pragma unroll
            for (int t = 0; t < GD_PER; ++t)
                if (j0 + t < L) { x = (r[t] - x*c[t])/d[t]; r[t] = x; }
            if (s < nw - 1) { hand[lane] = x; hand_ep[lane] = ep[GD_PER - 1]; }
        }
        __syncthreads();
    }
    double *rho_n = sn.rho + (i64)k*G.s;
    for (int s = nw - 1; s >= 0; --s) {
        if (w == s) {
            if (s < nw - 1) x = hand[lane];
#pragma unroll
            for (int t = GD_PER - 1; t >= 0; --t)
                if (j0 + t < L) { x = j0 + t < L - 1 ? r[t] - ep[t]*x : r[t]; r[t] = x; }
            if (s > 0) hand[lane] = x;
        }
        if (s > 0) __syncthreads();
    }
    if (!mine) return;
#pragma unroll
    for (int t = 0; t < GD_PER; ++t)
        if (j0 + t < L) put(rho_n + (i64)(j0 + t)*nsh, i, r[t] < 0.0 ? 0.0 : r[t]);
}

/* The same tracer solve with one (column, tracer) per lane, the rows
   generated and eliminated in one downward sweep through registers (the
   layout k_ver_waves uses); selected with GAME_GPU_GD_STREAMING for
   measurement against the kernel above. */
template <int LT>
__global__ void __launch_bounds__(128) k_gen_densities_stream(DevGrid G, DevState so, DevState sn, DevState td,
                                                              StepConsts K)
{
    const unsigned ntr = (unsigned)G.n_const - 1, blk = xcd_x();
    const int tr = (int)(blk%ntr);
    const int ncc = G.n_cond;
    const int k = tr < ncc ? tr : tr + 1;
    const int i = (int)(blk/ntr)*128 + threadIdx.x;
    if (i >= G.nsh) return;
    const int L = LT > 0 ? LT : G.L;
    const int nsh = G.nsh;
    const double iw = 0.5, ew = 1.0 - iw, dt = K.dt;
    const double *vol = G.vol, *area = G.area;
    const double *rho_o = so.rho + (i64)k*G.s, *trho = td.rho + (i64)k*G.s;
    double vsink = 0.0;
    if (k < ncc/4) vsink = K.snow_v;
    else if (k < ncc/2) vsink = K.rain_v;
    else if (k < ncc) vsink = K.cloud_v;
    double ep[LT > 0 ? LT : GAME_MAX_LAYERS], x[LT > 0 ? LT : GAME_MAX_LAYERS];
    double fi_m = 0.0, fr_m = 0.0, c_prev = 0.0;
#pragma unroll
    for (int j = 0; j < L; ++j) {
        const i64 b = i + (i64)j*nsh;
        double fi = 0.0, fr = 0.0;
        if (j < L - 1) tracer_iface_flux(G, so, sn, K, rho_o, k, i, j, fi, fr);
        double d;
        if (j == 0) d = (fi >= 0.0) ? 1.0 : 1.0 - iw*dt/vol[b]*fi;
        else if (j == L - 1) {
            d = (fi_m >= 0.0) ? 1.0 + iw*dt/vol[b]*fi_m : 1.0;
            if (k < ncc) d += iw*vsink*dt*area[i + G.v - nsh]/vol[b];
        } else {
            d = 1.0;
            if (fi_m >= 0.0) d += iw*dt/vol[b]*fi_m;
            if (fi < 0.0) d -= iw*dt/vol[b]*fi;
        }
        double r = rho_o[b] + dt*trho[b];
        if (j == 0) r += ew*dt*fr/vol[b];
        else if (j == L - 1) {
            r += -ew*dt*fr_m/vol[b];
            if (k < ncc) r += -ew*vsink*dt*rho_o[i + G.s - nsh]*area[i + G.v - nsh]/vol[b];
        } else r += ew*dt*(-fr_m + fr)/vol[b];
        double c = 0.0, e = 0.0;
        if (j < L - 1) {
            if (fi >= 0.0) e = -iw*dt/vol[b]*fi;
            else c = iw*dt/vol[b + nsh]*fi;
        }
        if (j == 0) {
            ep[0] = e/d;
            x[0] = r/d;
        } else {
            const double den = d - ep[j - 1]*c_prev;
            if (j < L - 1) ep[j] = e/den;
            x[j] = (r - x[j - 1]*c_prev)/den;
        }
        c_prev = c;
        fi_m = fi;
        fr_m = fr;
    }
#pragma unroll
    for (int j = L - 2; j >= 0; --j) x[j] = x[j] - ep[j]*x[j + 1];
    double *rho_n = sn.rho + (i64)k*G.s;
#pragma unroll
    for (int j = 0; j < L; ++j) {
        double v = x[j];
        if (v < 0.0) v = 0.0;
        rho_n[i + (i64)j*nsh] = v;
    }
}

/* sediment heat of the condensates at rk 0 (column_solvers.c:414-465 and the
   sh updates of :500-611), a chunk of RUN boxes of a column per thread: the
   flux of each condensate through each interface is formed once, the
   contributions are added in the reference's constituent order, starting
   from 0, and every load of the chunk is issued before its first store */
template <typename TW, int NCC, int RUN>
__global__ void __launch_bounds__(TPB) k_sed_heat(DevGrid G, DevState so, DevState sn, const TW *T, const TW *cpc,
                                                  TW *sed_heat, StepConsts K, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned i = bk.x*TPB + threadIdx.x;
    if (i >= (unsigned)G.nsh) return;
    const int nsh = G.nsh, vpl = G.vpl, L = G.L;
    const i64 S = G.s;
    int l0, l1;
    layer_chunk(L, bk.y, RUN, l0, l1);
    if (l0 >= l1) return;
    /* box l0 - 1 + t, and the interface above box l0 + t; a step past the
       chunk or the column repeats the nearest row and is not used */
    double d[RUN + 2][NCC], c[RUN + 2][2], tt[RUN + 2], wn[RUN + 1], a[RUN + 1], v[RUN];
#pragma unroll
    for (int t = 0; t < RUN + 2; ++t) {
        const int j = l0 - 1 + t < 0 ? 0 : (l0 - 1 + t < L ? l0 - 1 + t : L - 1);
        const i64 b = (i64)j*nsh;
#pragma unroll
        for (int k = 0; k < NCC; ++k) d[t][k] = at(so.rho + k*S + b, i);
        c[t][0] = (double)at(cpc + b, i);
        c[t][1] = (double)at(cpc + S + b, i);
        tt[t] = (double)at(T + b, i);
    }
#pragma unroll
    for (int t = 0; t < RUN + 1; ++t) {
        const int j = l0 + t < L ? l0 + t : L;
        wn[t] = at(sn.wind + (i64)j*vpl, i);
        a[t] = at(G.area + (i64)j*vpl, i);
    }
#pragma unroll
    for (int t = 0; t < RUN; ++t) v[t] = at(G.vol + (i64)(l0 + t < L ? l0 + t : L - 1)*nsh, i);
    double sh[RUN];
#pragma unroll
    for (int t = 0; t < RUN; ++t) sh[t] = 0.0;
#pragma unroll
    for (int k = 0; k < NCC; ++k) {
        const double sv = k < NCC/4 ? K.snow_v : (k < NCC/2 ? K.rain_v : K.cloud_v);
        /* through the interface above box l0 + t (column_solvers.c:414-465) */
        auto flux = [&](int t) {
            double fr = a[t]*(wn[t] - sv);
            const bool lo = fr >= 0.0;
            const double doi = lo ? d[t + 1][k] : d[t][k], toi = lo ? tt[t + 1] : tt[t], cpi = lo ? c[t + 1][k & 1] : c[t][k & 1];
            fr = doi*fr;
            return cpi*toi*fr;
        };
        double f = flux(0);
#pragma unroll
        for (int t = 0; t < RUN; ++t) {
            const int j = l0 + t;
            const double fl = flux(t + 1);
            if (j == 0) sh[t] += fl/v[t];
            else if (j == L - 1) {
                sh[t] += -f/v[t];
                /* a[t + 1] is the surface's area */
                sh[t] += -sv*tt[t + 1]*c[t + 1][k & 1]*d[t + 1][k]*a[t + 1]/v[t];
            } else sh[t] += (-f + fl)/v[t];
            f = fl;
        }
    }
#pragma unroll
    for (int t = 0; t < RUN; ++t) if (l0 + t < l1) put(sed_heat + (i64)(l0 + t)*nsh, i, (TW)sh[t]);
}

/* The same sums with one thread per column walking down its layers: the flux
   through each interface is formed once (by the reference's arithmetic) and
   carried to the box below, and the upstream box's density, temperature and
   c_p are loaded once per box and kept for the next interface.  The helper's
   restrict-qualified pointers let the loads of later layers move ahead of the
   stores of earlier ones, as many layers of them as a turn of the loop has: UN,
   eight in the FP64 form and four in the mixed one, whose conversions take
   registers (us per launch with turns of 4, 8, 13 and, at 26 layers, of the
   whole column, which the compiler spreads over 64 registers, too few for the
   loads: res 7 x 26 FP64 83.4, 80.5, 82.0, 79.0 and mixed 67.5, 77.6, 88.0,
   86.2; res 7 x 24 78.1, 76.3, 74.8 and 62.9, 72.8, 74.6) */
template <typename TW, int NCC>
__device__ __forceinline__ void sed_heat_column(const DevGrid &G, const StepConsts &K, int i,
                                                const double *__restrict__ rho_o, const double *__restrict__ wind_n,
                                                const double *__restrict__ area, const double *__restrict__ vol,
                                                const TW *__restrict__ T, const TW *__restrict__ cpc,
                                                TW *__restrict__ sed_heat)
{
    constexpr int UN = sizeof(TW) == sizeof(double) ? 8 : 4;
    const int nsh = G.nsh, vpl = G.vpl, L = G.L;
    const i64 S = G.s;
    double vsink[NCC];
#pragma unroll
    for (int k = 0; k < NCC; ++k) vsink[k] = k < NCC/4 ? K.snow_v : (k < NCC/2 ? K.rain_v : K.cloud_v);
    /* values of the box above the current interface */
    double d_up[NCC], c_up[NCC], t_up = (double)T[i];
#pragma unroll
    for (int k = 0; k < NCC; ++k) { d_up[k] = rho_o[k*S + i]; c_up[k] = (double)cpc[(k & 1)*S + i]; }
    double fe_m[NCC];
#pragma unroll
    for (int k = 0; k < NCC; ++k) fe_m[k] = 0.0;
#pragma unroll UN
    for (int j = 0; j < L; ++j) {
        const i64 b = i + (i64)j*nsh;
        const double v = vol[b];
        double fe[NCC], d_lo[NCC], c_lo[NCC], t_lo = 0.0;
#pragma unroll
        for (int k = 0; k < NCC; ++k) { fe[k] = 0.0; d_lo[k] = 0.0; c_lo[k] = 0.0; }
        if (j <= L - 2) {
            /* interface j, below box j (column_solvers.c:414-465) */
            const double wn = wind_n[i + (i64)(j + 1)*vpl], a = area[i + (i64)(j + 1)*vpl];
            t_lo = (double)T[b + nsh];
#pragma unroll
            for (int k = 0; k < NCC; ++k) {
                d_lo[k] = rho_o[k*S + b + nsh];
                c_lo[k] = (double)cpc[(k & 1)*S + b + nsh];
                double fr = wn;
                fr -= vsink[k];
                fr = a*fr;
                const bool lo = fr >= 0.0;
                const double doi = lo ? d_lo[k] : d_up[k], toi = lo ? t_lo : t_up, cpi = lo ? c_lo[k] : c_up[k];
                fr = doi*fr;
                fe[k] = cpi*toi*fr;
            }
        }
        double sh = 0.0;
#pragma unroll
        for (int k = 0; k < NCC; ++k) {
            if (j == 0) sh += fe[k]/v;
            else if (j == L - 1) {
                const i64 sfc = i + G.v - nsh;
                sh += -fe_m[k]/v;
                /* the lowest box: t_up, d_up, c_up hold its values */
                sh += -vsink[k]*t_up*c_up[k]*d_up[k]*area[sfc]/v;
            } else sh += (-fe_m[k] + fe[k])/v;
            fe_m[k] = fe[k];
            d_up[k] = d_lo[k];
            c_up[k] = c_lo[k];
        }
        t_up = t_lo;
        sed_heat[b] = (TW)sh;
    }
}

template <typename TW, int NCC>
__global__ void __launch_bounds__(TPB) k_sed_heat_col(DevGrid G, DevState so, DevState sn, const TW *T, const TW *cpc,
                                                      TW *sed_heat, StepConsts K)
{
    const int i = (int)(xcd_x()*TPB + threadIdx.x);
    if (i >= G.nsh) return;
    sed_heat_column<TW, NCC>(G, K, i, so.rho, sn.wind, G.area, G.vol, T, cpc, sed_heat);
}

/* phase_trans.c:16-311 (surface phase transitions off), one thread per grid box */
__device__ __forceinline__ double sat_water(double t)
{   /* dictionary.c:287-333 */
    double tc = t - GC_T_0, r;
    if (tc > 100.0) tc = 100.0;
    if (tc > 0.0) r = exp(34.494 - 4924.99/(tc + 237.1))/pow(tc + 105.0, 1.57);
    else {
        if (tc < -50.0) tc = -50.0;
        r = 6.107799961
            + 4.436518521e-1*tc
            + 1.428945805e-2*(tc*tc)
            + 2.650648471e-4*pow(tc, 3.0)
            + 3.031240396e-6*pow(tc, 4.0)
            + 2.034080948e-8*pow(tc, 5.0)
            + 6.136820929e-11*pow(tc, 6.0);
        r = 100.0*r;
    }
    return r;
}

__device__ __forceinline__ double sat_ice(double t)
{   /* dictionary.c:361-385 */
    double tc = t - GC_T_0;
    if (tc < -80.0) tc = -80.0;
    if (tc > 0.0) tc = 0.0;
    double a = tc + 868.0;
    return exp(43.494 - 6545.8/(tc + 278.0))/(a*a);
}

__device__ __forceinline__ double dsat_water(double t)
{   /* dictionary.c:335-359 */
    double tc = t - GC_T_0;
    if (tc > 100.0) tc = 100.0;
    if (tc < 0.0) tc = 0.0;
    double a = tc + 237.1;
    return sat_water(t)*(4924.99/(a*a) - 1.57/(tc + 105.0));
}

__device__ __forceinline__ double dsat_ice(double t)
{   /* dictionary.c:387-412 */
    double tc = t - GC_T_0;
    if (tc < -80.0) tc = -80.0;
    if (tc > 0.0) tc = 0.0;
    double a = tc + 278.0;
    return sat_ice(t)*(6545.8/(a*a) - 2.0/(tc + 868.0));
}

__device__ __forceinline__ double enthalpy_evaporation(double t)
{   /* dictionary.c:222-258 */
    if (t < GC_T_0) {
        if (t < 30.0) t = 30.0;
        return (56579.0 - 42.212*t + exp(0.1149*(281.6 - t)))/GC_M_V;
    }
    if (t > GC_T_0 + 100.0) t = GC_T_0 + 100.0;
    return 3151378.0 - 2386.0*t;
}

__device__ __forceinline__ double enthalpy_sublimation(double t)
{   /* dictionary.c:260-285 */
    if (t < 30.0) t = 30.0;
    if (t > GC_T_0) t = GC_T_0;
    double q = t/123.75;
    return (46782.5 + 35.8925*t - 0.07414*(t*t) + 541.5*exp(-(q*q)))/GC_M_V;
}

__device__ __forceinline__ double phase_trans_heat(int dir, double t)
{   /* dictionary.c:192-220 */
    if (dir == 0) return enthalpy_evaporation(t);
    if (dir == 1) return enthalpy_sublimation(t);
    return enthalpy_sublimation(t) - enthalpy_evaporation(t);
}

/* the saturation adjustment of one grid box (phase_trans.c:16-311, surface
   phase transitions off) on loaded values: densities r[0..5] (snow, rain,
   cloud ice, cloud water, gas, vapour), temperature T and the condensates'
   c_p cp[0..3] as stored; rates out[0..4] and the heating rate */
__device__ __forceinline__ void phase_trans_point(const double *r, double T, const double *cp, double dt, double *out,
                                                  double &heat_out)
{
    const double rk0 = r[0], rk1 = r[1], rk2 = r[2], rk3 = r[3], rk4 = r[4], rk5 = r[5];
    const double mcwc = 0.2e-3;
    double wvp = rk5*GC_R_V*T;
    double dp = (rk4 - rk5)*GC_R_D*T;
    double ap = dp + wvp;
    const int warm = T >= GC_T_0;
    /* saturation pressure, enhancement factor, the phase's latent heat and the
       saturation pressure's derivative, over water or over ice: a branch, not
       a select, so a wave whose boxes are all above or all below freezing
       evaluates one set of exponentials */
    double sp, ef, pth, ds;
    if (warm) {
        sp = sat_water(T);
        ef = 1.00071*exp(0.000000045*ap);
        pth = phase_trans_heat(0, T);
        ds = dsat_water(T);
    } else {
        sp = sat_ice(T);
        ef = 0.99882*exp(0.00000008*ap);
        pth = phase_trans_heat(1, T);
        ds = dsat_ice(T);
    }
    sp = ef*sp;
    /* c_v_mass_weighted_air with the condensates' c_p (derived_quantities.c:97-115) */
    double cvm = 0.0;
    for (int k = 0; k < 4; ++k) cvm += r[k]*cp[k];
    cvm += rk4*GC_C_D_V;
    cvm += rk5*GC_C_V_V;
    double a = -GC_R_V*pth/cvm;
    double b = GC_R_V*T - GC_R_V*rk5*pth/cvm + ef*ds*pth/cvm;
    double cc = wvp - sp;
    double p = b/a, q = cc/a;
    /* the reference's pow(x, 0.5) (phase_trans.c:92-99): the square root,
       which IEEE rounds correctly (glibc's pow is within 0.52 ulp of it);
       the discriminant is never -0.0 or -inf, where the two differ */
    double dd = -0.5*p - sqrt(0.25*(p*p) - q);
    double r0, r1, r2, r3, r4, heat;
    if (sp >= wvp) {
        if (warm) {
            r2 = -rk2/dt;
            double ptd = fmin(rk3, dd);
            r4 = ptd/dt;
            r3 = rk2/dt - ptd/dt;
            heat = r2*phase_trans_heat(2, T) - ptd*phase_trans_heat(0, T)/dt;
        } else {
            r3 = -rk3/dt;
            double ptd = fmin(rk2, dd);
            r4 = ptd/dt;
            r2 = rk3/dt - ptd/dt;
            heat = -r3*phase_trans_heat(2, T) - ptd*phase_trans_heat(1, T)/dt;
        }
    } else {
        if (warm) {
            r2 = -rk2/dt;
            r4 = dd/dt;
            r3 = rk2/dt - dd/dt;
            heat = r2*phase_trans_heat(2, T) - dd*phase_trans_heat(0, T)/dt;
        } else {
            r3 = -rk3/dt;
            r4 = dd/dt;
            r2 = rk3/dt - dd/dt;
            heat = -r3*phase_trans_heat(2, T) - dd*phase_trans_heat(1, T)/dt;
        }
    }
    r0 = 0.0;
    r1 = 0.0;
    if (T < GC_T_0) {
        r0 = fmax(rk2 - mcwc*rk4, 0.0)/1000.0;
        r2 -= r0;
    } else if (T >= GC_T_0) {
        r1 = fmax(rk3 - mcwc*rk4, 0.0)/1000.0;
        r3 -= r1;
    }
    if (T >= GC_T_0 && rk0 > 0.0) {
        r0 = -rk0/dt;
        r1 -= r0;
        heat += r0*phase_trans_heat(2, T);
    }
    if (T < GC_T_0 && rk1 > 0.0) {
        r1 = -rk1/dt;
        r0 -= r1;
        heat += -r1*phase_trans_heat(2, T);
    }
    out[0] = r0; out[1] = r1; out[2] = r2; out[3] = r3; out[4] = r4;
    heat_out = heat;
}

template <typename TW>
__global__ void __launch_bounds__(TPB) k_phase_trans(DevGrid G, DevState s, const TW *temp, const TW *cpc, TW *ptr,
                                                     TW *phr, double dt)
{
    i64 i = (i64)blockIdx.x*TPB + threadIdx.x;
    if (i >= G.s) return;
    const i64 S = G.s;
    double r[6], cp[4], out[5], heat;
    for (int k = 0; k < 6; ++k) r[k] = s.rho[k*S + i];
    for (int k = 0; k < 4; ++k) cp[k] = (double)cpc[(k & 1)*S + i];
    phase_trans_point(r, (double)temp[i], cp, dt, out, heat);
    for (int k = 0; k < 5; ++k) ptr[k*S + i] = (TW)out[k];
    phr[i] = (TW)heat;
}

/* temperature_diagnostics, the condensates' c_p, the gas fraction and the
   saturation adjustment of a moist grid box in one pass: the adjustment
   takes the temperature and c_p as stored (rounded to TW), so its results
   are those of k_temperature followed by k_phase_trans */
template <typename TW>
__global__ void __launch_bounds__(TPB) k_temp_phase(DevGrid G, DevState s, TW *T, TW *cpc, double *gf, TW *ptr,
                                                    TW *phr, double dt)
{
    i64 i = (i64)blockIdx.x*TPB + threadIdx.x;
    if (i >= G.s) return;
    const i64 S = G.s;
    double r[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) r[k] = s.rho[k*S + i];
    const double thbg = G.thbg[i], tp = s.tp[i], exbg = G.exbg[i], ep = s.ep[i];
    /* density_total's left-to-right sum from 0 (derived_quantities.c:83-95)
       over the six densities already loaded */
    double rt = 0.0;
#pragma unroll
    for (int k = 0; k < 6; ++k) rt += r[k];
    gf[i] = r[4]/rt;
    double t = (thbg + tp)*(exbg + ep);
    t = t/(1.0 + r[5]/r[4]*(GC_M_D/GC_M_V - 1.0));
    T[i] = (TW)t;
    const double tt = (double)(TW)t;
    /* dictionary.c:111-190: snow and cloud ice share the ice formula, rain and
       cloud water the liquid one; each is evaluated once */
    const TW c_ice = (TW)c_p_ice(tt), c_liq = (TW)c_p_water(tt);
    double cp[4];
    for (int k = 0; k < 4; ++k) cp[k] = (double)((k & 1) == 0 ? c_ice : c_liq);
    cpc[i] = c_ice;
    cpc[S + i] = c_liq;
    double out[5], heat;
    phase_trans_point(r, tt, cp, dt, out, heat);
    for (int k = 0; k < 5; ++k) ptr[k*S + i] = (TW)out[k];
    phr[i] = (TW)heat;
}

/* linear_combine_two_states.c:14-43 */
__global__ void __launch_bounds__(TPB) k_lincomb_scalars(DevGrid G, DevState a, DevState b, DevState o, double c0,
                                                         double c1)
{
    i64 i = (i64)blockIdx.x*TPB + threadIdx.x;
    if (i >= G.s) return;
    for (int k = 0; k < G.n_const; ++k) o.rho[k*G.s + i] = c0*a.rho[k*G.s + i] + c1*b.rho[k*G.s + i];
    double rt = c0*a.rt[i] + c1*b.rt[i];
    o.rt[i] = rt;
    o.tp[i] = rt/o.rho[(i64)G.n_cond*G.s + i] - G.thbg[i];
    o.ep[i] = c0*a.ep[i] + c1*b.ep[i];
}

__global__ void __launch_bounds__(TPB) k_lincomb_vector(i64 n, const double *a, const double *b, double *o, double c0,
                                                        double c1)
{
    i64 i = (i64)blockIdx.x*TPB + threadIdx.x;
    if (i >= n) return;
    o[i] = c0*a[i] + c1*b[i];
}

/* merge of two compensated partial sums (s, c) += (s2, c2): the sum of the
   leading parts with its exact rounding error (Neumaier's two-sum), the
   compensations added */
__device__ __forceinline__ void neumaier_merge(double &s, double &c, double s2, double c2)
{
    const double t = s + s2;
    double err;
    if (fabs(s) >= fabs(s2)) err = (s - t) + s2;
    else err = (s2 - t) + s;
    s = t;
    c = (c + c2) + err;
}

/* per-block compensated partial sums of x*volume (write_output.c:1659-1668 with
   Neumaier summation).  Each lane sums a grid-strided subset; the 64 lanes of
   a wavefront are merged by butterfly shuffles (six steps of __shfl_xor, no
   LDS), the four wavefronts of the block through LDS; the host adds the
   block partials, also compensated. */
template <typename TY>
__global__ void __launch_bounds__(TPB) k_integral_partials(i64 n, const double *x, const TY *y, const double *vol,
                                                           double *partials)
{
    __shared__ double ss[TPB/64], sc[TPB/64];
    double s = 0.0, c = 0.0;
    for (i64 i = (i64)blockIdx.x*TPB + threadIdx.x; i < n; i += (i64)gridDim.x*TPB) {
        double v = x[i]*vol[i];
        if (y) v = x[i]*(double)y[i]*vol[i];
        neumaier_merge(s, c, v, 0.0);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double s2 = __shfl_xor(s, off, 64), c2 = __shfl_xor(c, off, 64);
        neumaier_merge(s, c, s2, c2);
    }
    const int wv = threadIdx.x/64, lane = threadIdx.x%64;
    if (lane == 0) { ss[wv] = s; sc[wv] = c; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double S = ss[0], Cc = sc[0];
        for (int k = 1; k < TPB/64; ++k) neumaier_merge(S, Cc, ss[k], sc[k]);
        partials[2*blockIdx.x] = S;
        partials[2*blockIdx.x + 1] = Cc;
    }
}

/* ------------------------------------------------------------------ */
/* host-side launchers                                                  */
/* ------------------------------------------------------------------ */
/* horizontal operators and tendencies; TW is the work-array type */
namespace hor {

#define FLAT_DISPATCH(NAME, KERNEL, GRIDDIM, ...)                                                 \
    do {                                                                                      \
        if (G.flat) LAUNCH(NAME, (KERNEL<true, TW>), GRIDDIM, dim3(TPB), st, __VA_ARGS__);    \
        else LAUNCH(NAME, (KERNEL<false, TW>), GRIDDIM, dim3(TPB), st, __VA_ARGS__);          \
    } while (0)

/* launches f for the longest chunk of n layers or levels in `chunks` chunks:
   1, 2 or 3 (the kernel holds a chunk's results until its last load), or 0
   for longer chunks, which store layer by layer */
template <class F>
static void run_dispatch(int n, int chunks, F f)
{
    const int run = (n + chunks - 1)/chunks;
    if (run == 1) f(std::integral_constant<int, 1>());
    else if (run == 2) f(std::integral_constant<int, 2>());
    else if (run == 3) f(std::integral_constant<int, 3>());
    else f(std::integral_constant<int, 0>());
}

template <typename TW>
static void pgrad_t(const DevGrid &G, const DevState &s, const DevWorkT<TW> &W, int first, double itw, const Mom<TW> &m,
                    hipStream_t st)
{
    /* the weights of the momentum tendency */
    const double chw = 0.5 + itw, ohw = 1.0 - chw, cvw = 1.0 - itw;
    const double *gf = W.gas_frac;
    const dim3 gw = grid_of(G.nsh, G.L - 1), ge = grid_of(G.nvh, G.split_grad), b(TPB);
    const Span sw = span_of(G.nsh, 1, 1), se = span_of(G.nvh, G.L, G.split_grad);
    if (first) {
        LAUNCH("k_pgrad_w", (k_pgrad_w<TW, false>), gw, b, st, G, s, W, first, gf, cvw, m, sw);
        if (G.flat) LAUNCH("k_pgrad_e", (k_pgrad_e<true, TW, false>), ge, b, st, G, s, W, first, gf, chw, ohw, m, se);
        else LAUNCH("k_pgrad_e", (k_pgrad_e<false, TW, false>), ge, b, st, G, s, W, first, gf, chw, ohw, m, se);
    } else {
        LAUNCH("k_pgrad_w", (k_pgrad_w<TW, true>), gw, b, st, G, s, W, first, gf, cvw, m, sw);
        if (G.flat) LAUNCH("k_pgrad_e", (k_pgrad_e<true, TW, true>), ge, b, st, G, s, W, first, gf, chw, ohw, m, se);
        else LAUNCH("k_pgrad_e", (k_pgrad_e<false, TW, true>), ge, b, st, G, s, W, first, gf, chw, ohw, m, se);
    }
}

template <typename TW>
static void vorticity_flux_t(const DevGrid &G, const TW *F, const TW *pv, TW *out, hipStream_t st)
{
    const DevWorkT<TW> W{};
    const Mom<TW> m{};
    LAUNCH("k_vorticity_flux_e", (k_vorticity_flux_e<true, TW, false>), grid_of(G.nvh, G.split_edge), dim3(TPB), st, G, F, pv,
           out, W, m, span_of(G.nvh, G.L, G.split_edge));
    run_dispatch(G.L + 1, G.split_cell_w, [&](auto r) {
        LAUNCH("k_vorticity_flux_w", (k_vorticity_flux_w<TW, decltype(r)::value, 0>), grid_of(G.nsh, G.split_cell_w),
               dim3(TPB), st, G, F, pv, out, W, m, (const double *)nullptr, span_of(G.nsh, G.L + 1, G.split_cell_w));
    });
}

template <typename TW>
static void momentum_e_t(const DevGrid &G, const DevWorkT<TW> &W, const Mom<TW> &m, hipStream_t st)
{
    const dim3 g = grid_of(G.nvh, G.split_edge), b(TPB);
    const Span sp = span_of(G.nvh, G.L, G.split_edge);
    const TW *F = W.flux, *pv = W.pv;
    if (G.flat) LAUNCH("k_vorticity_flux_e", (k_vorticity_flux_e<true, TW, true>), g, b, st, G, F, pv, W.pvt, W, m, sp);
    else LAUNCH("k_vorticity_flux_e", (k_vorticity_flux_e<false, TW, true>), g, b, st, G, F, pv, W.pvt, W, m, sp);
}

template <typename TW>
static void momentum_w_t(const DevGrid &G, const DevWorkT<TW> &W, const Mom<TW> &m, const double *rho, hipStream_t st)
{
    const dim3 g = grid_of(G.nsh, G.split_cell_w), b(TPB);
    const Span sp = span_of(G.nsh, G.L + 1, G.split_cell_w);
    const TW *F = W.flux, *pv = W.pv;
    run_dispatch(G.L + 1, G.split_cell_w, [&](auto r) {
        constexpr int RUN = decltype(r)::value;
        if (G.n_const == 6)
            LAUNCH("k_vorticity_flux_w", (k_vorticity_flux_w<TW, RUN, 6>), g, b, st, G, F, pv, W.pvt, W, m, rho, sp);
        else LAUNCH("k_vorticity_flux_w", (k_vorticity_flux_w<TW, RUN, 1>), g, b, st, G, F, pv, W.pvt, W, m, rho, sp);
    });
}

template <typename TW>
static void inner_product_t(const DevGrid &G, const double *a, const double *b, TW *out, hipStream_t st)
{
    LAUNCH("k_inner_product", k_inner_product<TW>, grid_of(G.nsh, G.L), dim3(TPB), st, G, a, b, out, span_of(G.nsh, 1, 1));
}

template <typename TW>
static void grad_t(const DevGrid &G, const TW *f, TW *out, hipStream_t st)
{
    FLAT_DISPATCH("k_grad_e", k_grad_e, grid_of(G.nvh, G.split_grad), G, f, out, span_of(G.nvh, G.L, G.split_grad));
    LAUNCH("k_grad_w", k_grad_w<TW>, grid_of(G.nsh, G.L - 1), dim3(TPB), st, G, f, out,
           span_of(G.nsh, 1, 1));
}

template <typename TW>
static void rel_vort_tri_t(const DevGrid &G, const double *wind, TW *out, hipStream_t st)
{
    LAUNCH("k_rel_vort_tri", k_rel_vort_tri<TW>, grid_of(G.nt, G.split_tri), dim3(TPB), st, G, wind, out,
           span_of(G.nt, G.L, G.split_tri));
}

template <typename TW>
static void advection_pv_t(const DevGrid &G, const double *wind, const double *rho_gas, const DevWorkT<TW> &W,
                           hipStream_t st)
{
    rel_vort_tri_t<TW>(G, wind, W.rvt, st);
    FLAT_DISPATCH("k_pot_vort", k_pot_vort, grid_of(G.nvh, G.split_edge), G, wind, rho_gas, (const TW *)W.rvt, W.pv, W.flux,
                  span_of(G.nvh, G.L + 1, G.split_edge));
}

template <typename TW>
static void advection_t(const DevGrid &G, const double *wind, const double *rho_gas, const DevWorkT<TW> &W,
                        hipStream_t st)
{
    advection_pv_t<TW>(G, wind, rho_gas, W, st);
    vorticity_flux_t<TW>(G, W.flux, W.pv, W.pvt, st);
    inner_product_t<TW>(G, wind, wind, W.vsq, st);
    grad_t<TW>(G, W.vsq, W.vsq_grad, st);
}

/* the precision of FP32 storage on an FP64 array (a probe of the mixed form) */
__global__ void __launch_bounds__(TPB) k_round_f32(double *x, i64 n)
{
    const i64 t = (i64)blockIdx.x*TPB + threadIdx.x;
    if (t < n) x[t] = (double)(float)x[t];
}

template <typename TW>
static void scalar_tend_t(const DevGrid &G, const DevState &s, const DevState &td, const DevWorkT<TW> &W, int rk,
                          hipStream_t st);

template <typename TW>
static void scalar_tend_probe(const DevGrid &G, const DevState &td, hipStream_t st)
{
    if (sizeof(TW) != sizeof(float) || !G.round_tendencies) return;
    if (G.round_tendencies & 1)
        LAUNCH("k_round_f32", k_round_f32, GRID1((i64)G.n_const*G.s), dim3(TPB), st, td.rho, (i64)G.n_const*G.s);
    if (G.round_tendencies & 2) LAUNCH("k_round_f32", k_round_f32, GRID1(G.s), dim3(TPB), st, td.rt, G.s);
}

template <typename TW>
static void scalar_tend_t(const DevGrid &G, const DevState &s, const DevState &td, const DevWorkT<TW> &W, int rk,
                          hipStream_t st)
{
    /* the chunks of terrain levels: set_layer_splits.  Bound by the gathers of
       six neighbours' densities and winds (107 MB that it cannot do without at
       res 6 x 26, 22 us at a copy's rate): each layer loaded before the one above
       it is summed, the weights -0.5*ipw*slope a grid constant (59 -> 43 us per
       launch), no load past the chunk's end and, for a dry model, no correction
       of the wind itself, which only the tracers take (43 -> 35) */
    if (!G.flat) {
        const dim3 g = grid_of(G.nsh, G.split_vcc);
        const Span sp = span_of(G.nsh, G.n_oro, G.split_vcc);
        if (G.n_const > 1) LAUNCH("k_vcc", k_vcc<true>, g, dim3(TPB), st, G, s, W.vcc, sp);
        else LAUNCH("k_vcc", k_vcc<false>, g, dim3(TPB), st, G, s, W.vcc, sp);
    }
    const dim3 g = grid_of(G.nsh, G.L), b(TPB);
    const Span sp = span_of(G.nsh, 1, 1);
    if (G.n_const == 6) {
        if (G.flat) LAUNCH("k_scalar_tend", (k_scalar_tend<true, TW, 6>), g, b, st, G, s, W, td.rho, td.rt, rk, sp);
        else LAUNCH("k_scalar_tend", (k_scalar_tend<false, TW, 6>), g, b, st, G, s, W, td.rho, td.rt, rk, sp);
    } else {
        if (G.flat) LAUNCH("k_scalar_tend", (k_scalar_tend<true, TW, 1>), g, b, st, G, s, W, td.rho, td.rt, rk, sp);
        else LAUNCH("k_scalar_tend", (k_scalar_tend<false, TW, 1>), g, b, st, G, s, W, td.rho, td.rt, rk, sp);
    }
    scalar_tend_probe<TW>(G, td, st);
}

/* the entry points of both forms */
#define BOTH_FORMS(T, WORK)                                                                                         \
    void pgrad(const DevGrid &G, const DevState &s, const WORK &W, int first, double itw, T *td, const double *w_old,   \
               double *w_new, double dt, hipStream_t st)                                                            \
    { pgrad_t<T>(G, s, W, first, itw, Mom<T>{td, td, w_old, w_new, 1.0, dt}, st); }                                     \
    void advection(const DevGrid &G, const double *wind, const double *rho_gas, const WORK &W, hipStream_t st)      \
    { advection_t<T>(G, wind, rho_gas, W, st); }                                                                    \
    void advection_pv(const DevGrid &G, const double *wind, const double *rho_gas, const WORK &W, hipStream_t st)   \
    { advection_pv_t<T>(G, wind, rho_gas, W, st); }                                                                 \
    void kinetic_energy(const DevGrid &G, const double *wind, const WORK &W, hipStream_t st)                        \
    { inner_product_t<T>(G, wind, wind, W.vsq, st); }                                                               \
    void momentum_e(const DevGrid &G, const WORK &W, T *td, const T *td_old, const double *w_old, double *w_new,    \
                    double new_w, double dt, hipStream_t st)                                                        \
    { momentum_e_t<T>(G, W, Mom<T>{td, td_old, w_old, w_new, new_w, dt}, st); }                                     \
    void momentum_w(const DevGrid &G, const WORK &W, T *td, const T *td_old, double new_w, const double *rho,       \
                    hipStream_t st)                                                                                 \
    { momentum_w_t<T>(G, W, Mom<T>{td, td_old, nullptr, nullptr, new_w, 0.0}, rho, st); }
BOTH_FORMS(double, DevWork)
BOTH_FORMS(float, DevWorkF)
#undef BOTH_FORMS
void scalar_tend(const DevGrid &G, const DevState &s, const DevState &td, const DevWork &W, int rk, hipStream_t st)
{ scalar_tend_t<double>(G, s, td, W, rk, st); }
void scalar_tend(const DevGrid &G, const DevState &s, const DevState &td, const DevWorkF &W, int rk, hipStream_t st)
{ scalar_tend_t<float>(G, s, td, W, rk, st); }

void inner_product(const DevGrid &G, const double *a, const double *b, double *out, hipStream_t st)
{ inner_product_t<double>(G, a, b, out, st); }

/* single operators (FP64), for the operator-level interface and its adjoints */
void grad(const DevGrid &G, const double *f, double *out, hipStream_t st) { grad_t<double>(G, f, out, st); }
void curl_triangles(const DevGrid &G, const double *wind, double *out, hipStream_t st)
{ rel_vort_tri_t<double>(G, wind, out, st); }

void tables(const DevGrid &G, unsigned *c_e, unsigned *c_n, unsigned *c_from, unsigned *e_ti, unsigned *e_tm, double *e_tw,
            unsigned *e_rc, double *e_rw, unsigned *t_e, hipStream_t st)
{
    const int n = G.nvh > G.nt ? G.nvh : G.nt;   /* more than nsh */
    LAUNCH("k_tables", k_tables, GRID1(n), dim3(TPB), st, G, c_e, c_n, c_from, e_ti, e_tm, e_tw, e_rc, e_rw, t_e);
}

void vcc_weights(const DevGrid &G, double *vcw, hipStream_t st)
{ LAUNCH("k_vcc_weights", k_vcc_weights, GRID1((i64)G.n_oro*6*G.nsh), dim3(TPB), st, G, vcw); }

void vorticity_flux(const DevGrid &G, const double *F, const double *pv, double *out, hipStream_t st)
{ vorticity_flux_t<double>(G, F, pv, out, st); }

}  // namespace hor

/* the column solvers and point physics, shared by both precision forms (the
   work arrays they read or write are double in the FP64 form, float in the
   mixed form) */
namespace col {

void temperature(const DevGrid &G, const DevState &s, double *T, double *cpc, double *gf, hipStream_t st)
{ LAUNCH("k_temperature", k_temperature<double>, GRID1(G.s), dim3(TPB), st, G, s, T, cpc, gf); }
void temperature(const DevGrid &G, const DevState &s, float *T, float *cpc, double *gf, hipStream_t st)
{ LAUNCH("k_temperature", k_temperature<float>, GRID1(G.s), dim3(TPB), st, G, s, T, cpc, gf); }

void phase_trans(const DevGrid &G, const DevState &s, const double *T, const double *cpc, double *ptr, double *phr,
                 double dt, hipStream_t st)
{ LAUNCH("k_phase_trans", k_phase_trans<double>, GRID1(G.s), dim3(TPB), st, G, s, T, cpc, ptr, phr, dt); }
void phase_trans(const DevGrid &G, const DevState &s, const float *T, const float *cpc, float *ptr, float *phr,
                 double dt, hipStream_t st)
{ LAUNCH("k_phase_trans", k_phase_trans<float>, GRID1(G.s), dim3(TPB), st, G, s, T, cpc, ptr, phr, dt); }
void temperature_phase_trans(const DevGrid &G, const DevState &s, double *T, double *cpc, double *gf, double *ptr,
                             double *phr, double dt, hipStream_t st)
{ LAUNCH("k_temp_phase", k_temp_phase<double>, GRID1(G.s), dim3(TPB), st, G, s, T, cpc, gf, ptr, phr, dt); }
void temperature_phase_trans(const DevGrid &G, const DevState &s, float *T, float *cpc, double *gf, float *ptr,
                             float *phr, double dt, hipStream_t st)
{ LAUNCH("k_temp_phase", k_temp_phase<float>, GRID1(G.s), dim3(TPB), st, G, s, T, cpc, gf, ptr, phr, dt); }

template <typename TWIND>
static void ver_waves_t(const DevGrid &G, const DevState &so, const DevState &snr, const DevState &sn,
                        const DevState &td, const TWIND *td_wind, const StepConsts &K, int rk, hipStream_t st)
{
    if (G.vw_streaming) {
        dim3 g((G.nsh + 127)/128), b(128);
        if (G.L == 26) LAUNCH("k_ver_waves", (k_ver_waves<26, TWIND>), g, b, st, G, so, snr, sn, td, td_wind, K, rk);
        else if (G.L == 55)
            LAUNCH("k_ver_waves", (k_ver_waves<55, TWIND>), g, b, st, G, so, snr, sn, td, td_wind, K, rk);
        else LAUNCH("k_ver_waves", (k_ver_waves<0, TWIND>), g, b, st, G, so, snr, sn, td, td_wind, K, rk);
        return;
    }
    const int ncol = vr_ncol(G.L);
    const dim3 g((unsigned)((G.nsh + ncol - 1)/ncol)), b((unsigned)vr_threads(G.L));
    /* four rows of the system and three values per box: 45 KiB at 26 layers, 55 KiB at 63 */
    const size_t lds = (size_t)(4*(G.L - 1) + 3*G.L)*ncol*sizeof(double);
    if (ncol == 64)
        LAUNCH_SHM("k_ver_waves", (k_ver_waves_run<64, TWIND>), g, b, lds, st, G, so, snr, sn, td, td_wind, K, rk);
    else if (ncol == 32)
        LAUNCH_SHM("k_ver_waves", (k_ver_waves_run<32, TWIND>), g, b, lds, st, G, so, snr, sn, td, td_wind, K, rk);
    else
        LAUNCH_SHM("k_ver_waves", (k_ver_waves_run<16, TWIND>), g, b, lds, st, G, so, snr, sn, td, td_wind, K, rk);
}

void ver_waves(const DevGrid &G, const DevState &so, const DevState &snr, const DevState &sn, const DevState &td,
               const StepConsts &K, int rk, hipStream_t st)
{ ver_waves_t<double>(G, so, snr, sn, td, td.wind, K, rk, st); }

void ver_waves(const DevGrid &G, const DevState &so, const DevState &snr, const DevState &sn, const DevState &td,
               const float *td_wind, const StepConsts &K, int rk, hipStream_t st)
{ ver_waves_t<float>(G, so, snr, sn, td, td_wind, K, rk, st); }

static void gen_densities_only(const DevGrid &G, const DevState &so, const DevState &sn, const DevState &td,
                               const StepConsts &K, hipStream_t st)
{
    if (G.gd_streaming) {
        const dim3 g((unsigned)(((G.nsh + 127)/128)*(G.n_const - 1))), b(128);
        if (G.L == 26) LAUNCH("k_gen_densities", k_gen_densities_stream<26>, g, b, st, G, so, sn, td, K);
        else if (G.L == 55) LAUNCH("k_gen_densities", k_gen_densities_stream<55>, g, b, st, G, so, sn, td, K);
        else LAUNCH("k_gen_densities", k_gen_densities_stream<0>, g, b, st, G, so, sn, td, K);
        return;
    }
    /* nine rows per wave up to 27 layers, seven beyond (k_gen_densities) */
    const int per = G.L <= 27 ? 9 : 7, nw = (G.L + per - 1)/per;
    const dim3 g((unsigned)(((G.nsh + 63)/64)*(G.n_const - 1))), b((unsigned)(64*nw));
    static_assert(64*((27 + 8)/9) <= 192 && 64*((GAME_MAX_LAYERS + 6)/7) <= 640, "the blocks' threads");
    if (per == 9) LAUNCH("k_gen_densities", (k_gen_densities<9, 192>), g, b, st, G, so, sn, td, K);
    else LAUNCH("k_gen_densities", (k_gen_densities<7, 640>), g, b, st, G, so, sn, td, K);
}

/* One thread per column loads each box once, from 256 blocks of columns on; a
   chunk of five layers loads 13 values per box, one of one layer 26, and smaller
   grids, which columns leave short of blocks, take chunks of five, or of two
   where five do.  us per launch, FP64 and mixed, in chunks of two and of five
   and by column:
     res 5 x 26    10.9  9.7    11.3  9.9    27 and more
     res 6 x 26                 24.8  22.5    45.5  34.4
     res 6 x 55    54.9  44.8   44.4  36.8
     res 7 x 12                 42.6  36.0    38.0  30.4
     res 7 x 24    95.9  78.0   83.3  66.6    76.3  62.9
     res 7 x 26   112.9  87.7   89.5  73.6    80.5  67.5
     res 7 x 41                 134   112     124   104
     res 7 x 55                 196   154     165   140 */
template <typename TW>
static void sed_heat_t(const DevGrid &G, const DevState &so, const DevState &sn, const TW *T, const TW *cpc, TW *sed_heat,
                       const StepConsts &K, hipStream_t st)
{
    const int bc = (G.nsh + TPB - 1)/TPB;
    const int run = G.sh_run ? G.sh_run : (bc >= 256 ? SH_COLUMN : (bc*G.L < 4096 ? 2 : 5));
    if (run == SH_COLUMN) {
        LAUNCH("k_sed_heat", (k_sed_heat_col<TW, 4>), grid_of(G.nsh, 1), dim3(TPB), st, G, so, sn, T, cpc, sed_heat, K);
        return;
    }
    const dim3 g = grid_of(G.nsh, (G.L + run - 1)/run), b(TPB);
    const Span sp = span_of(G.nsh, 1, 1);
    if (run == 1) LAUNCH("k_sed_heat", (k_sed_heat<TW, 4, 1>), g, b, st, G, so, sn, T, cpc, sed_heat, K, sp);
    else if (run == 2) LAUNCH("k_sed_heat", (k_sed_heat<TW, 4, 2>), g, b, st, G, so, sn, T, cpc, sed_heat, K, sp);
    else LAUNCH("k_sed_heat", (k_sed_heat<TW, 4, 5>), g, b, st, G, so, sn, T, cpc, sed_heat, K, sp);
}

void gen_densities(const DevGrid &G, const DevState &so, const DevState &sn, const DevState &td, const double *T,
                   const double *cpc, double *sed_heat, const StepConsts &K, int rk, hipStream_t st)
{
    if (rk == 0 && G.n_cond > 0) sed_heat_t(G, so, sn, T, cpc, sed_heat, K, st);
    gen_densities_only(G, so, sn, td, K, st);
}

void gen_densities(const DevGrid &G, const DevState &so, const DevState &sn, const DevState &td, const float *T,
                   const float *cpc, float *sed_heat, const StepConsts &K, int rk, hipStream_t st)
{
    if (rk == 0 && G.n_cond > 0) sed_heat_t(G, so, sn, T, cpc, sed_heat, K, st);
    gen_densities_only(G, so, sn, td, K, st);
}

__global__ void __launch_bounds__(TPB) k_tracer_quotients(DevGrid G, double dt)
{
    const i64 b = (i64)blockIdx.x*TPB + threadIdx.x;
    if (b >= G.s) return;
    const double iw = 0.5;   /* the tracer solver's implicit weight */
    G.idv[b] = iw*dt/G.vol[b];
}

void tracer_quotients(const DevGrid &G, double dt, hipStream_t st)
{ LAUNCH("k_tracer_quotients", k_tracer_quotients, GRID1(G.s), dim3(TPB), st, G, dt); }

void linear_combine(const DevGrid &G, const DevState &a, const DevState &b, const DevState &o, double c0, double c1,
                    hipStream_t st)
{
    LAUNCH("k_lincomb_scalars", k_lincomb_scalars, GRID1(G.s), dim3(TPB), st, G, a, b, o, c0, c1);
    LAUNCH("k_lincomb_vector", k_lincomb_vector, GRID1(G.v), dim3(TPB), st, G.v, (const double *)a.wind, (const double *)b.wind,
                       o.wind, c0, c1);
}

int integral_partials(i64 n, const double *x, const double *y, const double *vol, double *partials, hipStream_t st)
{
    LAUNCH("k_integral_partials", k_integral_partials<double>, dim3(INTEGRAL_BLOCKS), dim3(TPB), st, n, x, y, vol,
           partials);
    return INTEGRAL_BLOCKS;
}

int integral_partials(i64 n, const double *x, const float *y, const double *vol, double *partials, hipStream_t st)
{
    LAUNCH("k_integral_partials", k_integral_partials<float>, dim3(INTEGRAL_BLOCKS), dim3(TPB), st, n, x, y, vol,
           partials);
    return INTEGRAL_BLOCKS;
}

}  // namespace col
