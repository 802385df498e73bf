/*
 * rkhevi_adjoint.hip -- hand-written adjoints of the linear operators of the
 * RKHEVI step (FP64), for gfx950.
 *
 * Every adjoint is a gather: each thread owns one output element of the
 * adjoint and sums the contributions of the forward outputs that read it,
 * through reverse index tables built once on the host (no atomics, so the
 * result does not depend on scheduling).  Each coefficient is recomputed
 * exactly as the forward kernel forms it, terrain-following terms included,
 * so <A x, y> = <x, A^T y> holds to rounding.
 *
 *   operator (forward, reference)                    adjoint gather
 *   grad (gradient_operators.c:56-74)                 cell <- adjacent edges, own column
 *   divv_h (divergences.c:14-64)                      edge <- from/to cells
 *   curl on triangles (vorticities.c:167-222)         edge <- its two triangles, layers l-1..l+1
 *   rhombus density (vorticities.c:74-80)             cell <- rhombi that weight it (CSR)
 *   TRSK vorticity flux in F (vorticity_flux.c)       edge <- edges whose TRSK stencil holds it (CSR)
 *                                                     w point <- adjacent edges and own levels
 *   inner product in a (inner_product.c:13-43)        edge <- from/to cells, w <- own column
 *   three-band solve (column_solvers.c:641-667)       transposed three-band solve
 */
#include "rkhevi_dev.h"
#include "rkhevi_adjoint.h"

#define ATPB TPB

/* ------------------------------------------------------------------ */
/* grad^T: fbar(c, l) from gbar at the cell's edges and w points        */
/* ------------------------------------------------------------------ */
__global__ void __launch_bounds__(ATPB) k_grad_adj(DevGrid G, const double *gb, double *fb, double gs, int acc, Span sp)
{
    /* the input is gs*gb, formed as it is loaded; acc adds the result to fb */
    /* one thread per (cell, chunk of layers): layer l's edge cotangents feed
       the horizontal term of layer l and the terrain terms of the w points
       l (ipw slot 6) and l + 1 (slot 7); each w point's cotangent is formed
       once and carried to the next layer */
    const Blk bk = linear_block();
    const unsigned h = bk.x*ATPB + threadIdx.x;
    if (h >= (unsigned)G.nsh) return;
    const int nsh = G.nsh, vpl = G.vpl, L = G.L, top = G.flat ? L : L - G.n_oro;
    const int ne = h < GAME_N_PENT ? 5 : 6;
    unsigned ej[6];
    const unsigned from = at(G.c_from, h);
#pragma unroll
    for (int j = 0; j < 6; ++j) ej[j] = at(G.c_e + (i64)j*nsh, h);
    int l0, l1;
    layer_chunk(L, bk.y, sp.run, l0, l1);
    if (l0 >= l1) return;
    /* layer l: the horizontal sum and the two terrain sums */
    auto layer = [&](int l, double &hs, double &s6, double &s7) {
        double g[6], sl[6], nd[6];
        const i64 vi = nsh + (i64)l*vpl;
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            g[j] = gs*at(gb + vi, ej[j]);
            sl[j] = (l >= top) ? at(G.slope + vi, ej[j]) : 0.0;
            nd[j] = at(G.nd + vi, ej[j]);
        }
        hs = 0.0;
        /* g_e = (f_to - f_from)/d_e: the from-cell (sign +1) gets -1/d_e */
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            const double sg = j < ne ? ((from >> j) & 1u ? 1.0 : -1.0) : 0.0;
            hs += -sg*g[j]/nd[j];
        }
        s6 = 0.0; s7 = 0.0;
        if (l >= top) {
            const double *wl = G.ipwT + ((i64)l*8 + 6)*nsh;
            const double w6 = at(wl, h), w7 = at(wl + nsh, h);
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                if (j < ne) {
                    s6 += -sl[j]*0.5*w6*g[j];
                    s7 += -sl[j]*0.5*w7*g[j];
                }
            }
        }
    };
    /* the cotangent of the vertical gradient at w point lev over its normal distance */
    auto wcot = [&](int lev, double s6, double s7_above) {
        double r = gs*at(gb + (i64)lev*vpl, h) + s6 + s7_above;
        return r/at(G.nd + (i64)lev*vpl, h);
    };
    double hs, s6, s7, s7p = 0.0, unused_h, unused_s6;
    if (l0 >= 1) layer(l0 - 1, unused_h, unused_s6, s7p);
    layer(l0, hs, s6, s7);
    double wc = l0 >= 1 ? wcot(l0, s6, s7p) : 0.0;
    for (int l = l0; l < l1; ++l) {
        double hn = 0.0, s6n = 0.0, s7n = 0.0, wn = 0.0;
        if (l + 1 <= L - 1) {
            layer(l + 1, hn, s6n, s7n);
            wn = wcot(l + 1, s6n, s7);
        }
        const double v = hs + wn - wc;
        double *row = fb + (i64)l*nsh;
        put(row, h, acc ? at(row, h) + v : v);
        hs = hn; s7 = s7n; wc = wn;
    }
}

/* ------------------------------------------------------------------ */
/* divv_h and divv_h^T                                                   */
/* ------------------------------------------------------------------ */
/* divergences.c:14-64 with averaging.c:41-95, one thread per cell and chunk of
   layers.  The correction at terrain level lev sums the cell's edge terms of
   layer lev - 1 and then of layer lev, from zero (from layer lev alone at the
   top one): layer lev - 1's running sum is carried, so each layer's edges are
   read once (170 -> 63 us at res 6 x 26 over the mountain against forming
   both corrections of every box from ipw and slope) */
template <bool FLAT>
__global__ void __launch_bounds__(ATPB) k_divv(DevGrid G, const double *in, double *out, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned h = bk.x*ATPB + threadIdx.x;
    if (h >= (unsigned)G.nsh) return;
    const int nsh = G.nsh, vpl = G.vpl, L = G.L, top = FLAT ? L : L - G.n_oro;
    const int ne = h < GAME_N_PENT ? 5 : 6;
    /* a fixed six edges: a pentagon's sixth slot reads its first edge and adds
       -0.0, the exact identity of IEEE addition */
    unsigned ej[6];
    const unsigned from = at(G.c_from, h);
#pragma unroll
    for (int j = 0; j < 6; ++j) ej[j] = at(G.c_e + (i64)j*nsh, h);
    int l0, l1;
    layer_chunk(L, bk.y, sp.run, l0, l1);
    if (l0 >= l1) return;
    /* layer l's edges; its horizontal sum, and its terrain terms added to both
       the correction at level l (cu) and the start of that at level l + 1 (cn) */
    auto layer = [&](int l, double &cu, double &cn) {
        const i64 vi = nsh + (i64)l*vpl;
        double v[6], a[6], c[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            v[j] = at(in + vi, ej[j]);
            a[j] = at(G.area + vi, ej[j]);
            c[j] = 0.0;
            if (!FLAT && l >= top) c[j] = at(G.vcw + ((i64)(l - top)*6 + j)*nsh, h);
        }
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            const double t = ((from >> j) & 1u ? v[j] : -v[j])*a[j];
            s += j < ne ? t : -0.0;
        }
        if (!FLAT && l >= top) {
#pragma unroll
            for (int j = 0; j < 6; ++j)
                if (j < ne) {
                    const double t = c[j]*v[j];
                    cu += t;
                    cn += t;
                }
        }
        return s;
    };
    /* cu: the correction at the layer's upper level; cn: the next one's start */
    double cu = 0.0, cn = 0.0;
    if (!FLAT && l0 > top) { double unused = 0.0; layer(l0 - 1, unused, cu); }
    double s = layer(l0, cu, cn);
    for (int l = l0; l < l1; ++l) {
        double cl = cn, cnn = 0.0, sn = 0.0;
        if (l + 1 < L && (l + 1 < l1 || (!FLAT && l + 1 >= top))) sn = layer(l + 1, cl, cnn);
        double comp = s;
        if constexpr (!FLAT) {
            double comp_v = 0.0;
            if (l == top - 1) comp_v = -cl*at(G.area + (i64)(l + 1)*vpl, h);
            else if (l == L - 1) comp_v = cu*at(G.area + (i64)l*vpl, h);
            else if (l > top - 1) comp_v = cu*at(G.area + (i64)l*vpl, h) - cl*at(G.area + (i64)(l + 1)*vpl, h);
            comp = s + comp_v;
        }
        put(out + (i64)l*nsh, h, 1.0/at(G.vol + (i64)l*nsh, h)*comp);
        s = sn; cu = cl; cn = cnn;
    }
}

/* one thread per edge and chunk of layers; the cotangent of the vertical
   contravariant correction vcc(c, lev), lev in [L - n_oro, L - 1], enters layer
   lev with +area_w(lev) and layer lev - 1 with -area_w(lev)
   (divergences.c:41-59): formed once per level and carried, as is each cell's
   quotient by its volume */
__global__ void __launch_bounds__(ATPB) k_divv_adj(DevGrid G, AdjTables A, const double *db, double *Fb, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned t = bk.x*ATPB + threadIdx.x;
    const int nsh = G.nsh, vpl = G.vpl, L = G.L, top = G.flat ? L : L - G.n_oro;
    int l0, l1;
    layer_chunk(L, bk.y, sp.run, l0, l1);
    /* divv_h reads horizontal components only */
    if (t < (unsigned)nsh) {
        for (int l = l0; l < l1; ++l) put(Fb + (i64)l*vpl, t, 0.0);
        if (l0 < l1 && l1 == L) put(Fb + (i64)L*vpl, t, 0.0);
    }
    if (t >= (unsigned)G.nvh || l0 >= l1) return;
    const unsigned e = t, cell[2] = {(unsigned)G.from[e], (unsigned)G.to[e]};
    const unsigned slot[2] = {(unsigned)G.flat ? 0u : (unsigned)A.slot_from[e], (unsigned)G.flat ? 0u : (unsigned)A.slot_to[e]};
    double q[2], qm[2] = {0.0, 0.0}, vc[2] = {0.0, 0.0};   /* db/vol of this layer and the one above; vcc_cot at this layer's level */
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        q[p] = at(db + (i64)l0*nsh, cell[p])/at(G.vol + (i64)l0*nsh, cell[p]);
        if (l0 >= 1) qm[p] = at(db + (i64)(l0 - 1)*nsh, cell[p])/at(G.vol + (i64)(l0 - 1)*nsh, cell[p]);
    }
    auto cot = [&](int lev, int p, double lo, double up) {
        const double a = at(G.area + (i64)lev*vpl, cell[p]);
        return lo*a - up*a;
    };
    if (l0 >= top) {
#pragma unroll
        for (int p = 0; p < 2; ++p) vc[p] = cot(l0, p, q[p], qm[p]);
    }
    for (int l = l0; l < l1; ++l) {
        const i64 vi = nsh + (i64)l*vpl;
        const int ln = l + 1 < L ? l + 1 : l;
        double qn[2], vn[2] = {0.0, 0.0};
#pragma unroll
        for (int p = 0; p < 2; ++p) qn[p] = at(db + (i64)ln*nsh, cell[p])/at(G.vol + (i64)ln*nsh, cell[p]);
        double r = at(G.area + vi, e)*(q[0] - q[1]);
        if (l + 1 >= top && l + 1 <= L - 1) {
#pragma unroll
            for (int p = 0; p < 2; ++p) vn[p] = cot(l + 1, p, qn[p], q[p]);
        }
        if (l >= top) {
            const double *wl = G.vcw + (i64)(l - top)*6*nsh;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const double k = at(wl, slot[p]*(unsigned)nsh + cell[p]);
                double v = vc[p];
                if (l + 1 <= L - 1) v += vn[p];
                r += k*v;
            }
        }
        put(Fb + vi, e, r);
#pragma unroll
        for (int p = 0; p < 2; ++p) { q[p] = qn[p]; vc[p] = vn[p]; }
    }
}

/* ------------------------------------------------------------------ */
/* curl on triangles^T                                                  */
/* ------------------------------------------------------------------ */
/* one thread per (edge, chunk of layers) walking down the layers: the two
   triangles' contributions of layer l (to layer l itself and, in the terrain
   layers, to the layer its interpolation reads) are formed once and kept for
   the layers above and below; wind points at w levels get 0 (the forward
   reads none).  The sum for layer lp adds, per triangle, the terms of layers
   lp-1, lp, lp+1 in that order. */
struct CurlAdjTerm {
    double s[2], o[2];   /* base*self (to layer l) and base*other (to layer l -+ 1) */
    int d[2];            /* -1: the other term goes to l-1, +1: to l+1, 0: none */
};

__device__ __forceinline__ CurlAdjTerm curl_adj_term(const DevGrid &G, const double *zb, unsigned e, const unsigned *tri,
                                                     const double *sg, int l)
{
    const int nsh = G.nsh, vpl = G.vpl, L = G.L;
    const i64 vi = nsh + (i64)l*vpl;
    const i64 vu = l > 0 ? vi - vpl : vi, vd = l < L - 1 ? vi + vpl : vu;
    const double nd = at(G.nd + vi, e), zv = at(G.zv + vi, e), zu = at(G.zv + vu, e), zd = at(G.zv + vd, e);
    double z[2], da[2], dzv[2];
    const i64 di = G.nvh + (i64)l*G.dvpl;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        z[p] = at(zb + (i64)l*G.nt, tri[p]);
        da[p] = at(G.darea + di, tri[p]);
        dzv[p] = at(G.dzv + di, tri[p]);
    }
    CurlAdjTerm c;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        double lrf = 1.0, self = 1.0, other = 0.0;
        int d = 0;
        if (l >= L - G.n_oro) {
            lrf = (G.radius + dzv[p])/(G.radius + zv);
            const double dz = dzv[p] - zv;
            const bool up = dz > 0 || l == L - 1;
            const double qq = dz/(zv - (up ? zu : zd));
            self = 1.0 + qq;
            other = -qq;
            d = up ? -1 : 1;
        }
        const double base = z[p]*lrf*nd*sg[p]/da[p];
        c.s[p] = base*self;
        c.o[p] = base*other;
        c.d[p] = d;
    }
    return c;
}

__global__ void __launch_bounds__(ATPB) k_curl_adj(DevGrid G, AdjTables A, const double *zb, double *wb, int acc, Span sp)
{
    /* acc adds the edge cotangents to wb and leaves its w points; otherwise
       the w points are set to zero */
    const Blk bk = xcd_block(sp);
    const unsigned t = bk.x*ATPB + threadIdx.x;
    const int nsh = G.nsh, vpl = G.vpl, L = G.L;
    int l0, l1;
    layer_chunk(L, bk.y, sp.run, l0, l1);
    if (!acc && t < (unsigned)nsh) {
        for (int l = l0; l < l1; ++l) put(wb + (i64)l*vpl, t, 0.0);
        if (l0 < l1 && l1 == L) put(wb + (i64)L*vpl, t, 0.0);
    }
    if (t >= (unsigned)G.nvh || l0 >= l1) return;
    const unsigned e = t;
    unsigned tri[2];
    double sg[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        tri[p] = (unsigned)A.tri_of_edge[2*(i64)e + p];
        sg[p] = at(G.t_e + (i64)A.tri_slot[2*(i64)e + p]*G.nt, tri[p]) >> 31 ? -1.0 : 1.0;
    }
    CurlAdjTerm prev = {}, cur = curl_adj_term(G, zb, e, tri, sg, l0), nxt = {};
    if (l0 >= 1) prev = curl_adj_term(G, zb, e, tri, sg, l0 - 1);
    if (l0 + 1 <= L - 1) nxt = curl_adj_term(G, zb, e, tri, sg, l0 + 1);
    for (int lp = l0; lp < l1; ++lp) {
        double r = 0.0;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (lp >= 1 && prev.d[p] == 1) r += prev.o[p];
            r += cur.s[p];
            if (lp + 1 <= L - 1 && nxt.d[p] == -1) r += nxt.o[p];
        }
        double *row = wb + nsh + (i64)lp*vpl;
        put(row, e, acc ? at(row, e) + r : r);
        prev = cur;
        cur = nxt;
        if (lp + 2 <= L - 1 && lp + 1 < l1) nxt = curl_adj_term(G, zb, e, tri, sg, lp + 2);
    }
}

/* ------------------------------------------------------------------ */
/* rhombus density and its adjoint                                      */
/* ------------------------------------------------------------------ */
__global__ void __launch_bounds__(ATPB) k_rhombus(DevGrid G, const double *rho, double *out, Span sp)
{
    const Blk bk = xcd_block(sp);
    const unsigned e = bk.x*ATPB + threadIdx.x;
    if (e >= (unsigned)G.nvh) return;
    unsigned c[4];
    double w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) { c[j] = at(G.e_rc + (i64)j*G.nvh, e); w[j] = at(G.e_rw + (i64)j*G.nvh, e); }
    int l0, l1;
    layer_chunk(G.L, bk.y, sp.run, l0, l1);
    for (int l = l0; l < l1; ++l) {
        const double *row = rho + (i64)l*G.nsh;
        double dr = 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) dr += w[j]*at(row, c[j]);
        put(out + (i64)l*G.nvh, e, dr);
    }
}

__global__ void __launch_bounds__(ATPB) k_rhombus_adj(DevGrid G, AdjTables A, const double *db, double *rb, Span sp)
{
    /* one thread per (cell, chunk of layers): the cell's rhombus entries are
       loaded once, in ascending (edge, slot) order, padding weighted 0 */
    const Blk bk = xcd_block(sp);
    const unsigned c = bk.x*ATPB + threadIdx.x;
    if (c >= (unsigned)G.nsh) return;
    const int nsh = G.nsh, nvh = G.nvh;
    unsigned e[ADJ_RH_MAX];
    double w[ADJ_RH_MAX];
#pragma unroll
    for (int k = 0; k < ADJ_RH_MAX; ++k) { e[k] = (unsigned)at(A.rhp_e + (i64)k*nsh, c); w[k] = at(A.rhp_w + (i64)k*nsh, c); }
    int l0, l1;
    layer_chunk(G.L, bk.y, sp.run, l0, l1);
    for (int l = l0; l < l1; ++l) {
        const double *row = db + (i64)l*nvh;
        double r = 0.0;
#pragma unroll
        for (int k = 0; k < ADJ_RH_MAX; ++k) r += w[k]*at(row, e[k]);
        put(rb + (i64)l*nsh, c, r);
    }
}

/* ------------------------------------------------------------------ */
/* TRSK vorticity flux^T in the mass flux F (pv fixed)                   */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ double vflux_w_weight(const DevGrid &G, int lev)
{   /* vorticity_flux.c:373-417: half weights inside, full at top and surface */
    return (lev == 0 || lev == G.L) ? 1.0 : 0.5;
}

__global__ void __launch_bounds__(ATPB) k_vflux_adj_e(DevGrid G, AdjTables A, const double *pv, const double *ob,
                                                      double *Fb, Span sp)
{
    /* horizontal F of edge e' at layer l, one thread per (edge, chunk of
       layers): its TRSK reverse entries are loaded once */
    const Blk bk = xcd_block(sp);
    const unsigned ep = bk.x*ATPB + threadIdx.x;
    if (ep >= (unsigned)G.nvh) return;
    const int nsh = G.nsh, nvh = G.nvh, vpl = G.vpl;
    unsigned e[ADJ_TR_MAX], m[ADJ_TR_MAX];
    bool hf[ADJ_TR_MAX];
    double w[ADJ_TR_MAX];
#pragma unroll
    for (int k = 0; k < ADJ_TR_MAX; ++k) {
        e[k] = (unsigned)at(A.trp_e + (i64)k*nvh, ep);
        const int mm = at(A.trp_m + (i64)k*nvh, ep);
        hf[k] = mm < 0;
        m[k] = (unsigned)(mm < 0 ? -mm - 1 : mm);
        w[k] = at(A.trp_w + (i64)k*nvh, ep);
    }
    const unsigned cell[2] = {(unsigned)G.from[ep], (unsigned)G.to[ep]};
    const unsigned sc[2] = {(unsigned)A.slot_from[ep]*(unsigned)nsh + cell[0], (unsigned)A.slot_to[ep]*(unsigned)nsh + cell[1]};
    int l0, l1;
    layer_chunk(G.L, bk.y, sp.run, l0, l1);
    if (l0 >= l1) return;
    /* the vertical outputs of the edge's two cells and its own PV at level l, carried */
    double q0 = at(pv + (i64)l0*2*nvh, ep), o0[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) o0[p] = at(ob + (i64)l0*vpl, cell[p]);
    for (int l = l0; l < l1; ++l) {
        const double *pl = pv + nvh + (i64)l*2*nvh, *ol = ob + nsh + (i64)l*vpl;
        double pm[ADJ_TR_MAX], pe[ADJ_TR_MAX], oe[ADJ_TR_MAX];
#pragma unroll
        for (int k = 0; k < ADJ_TR_MAX; ++k) { pm[k] = at(pl, m[k]); pe[k] = at(pl, e[k]); oe[k] = at(ol, e[k]); }
        const double q1 = at(pl + nvh, ep);
        double wt[2], o1[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            wt[p] = at(G.ipwT + (i64)l*8*nsh, sc[p]);
            o1[p] = at(ob + (i64)(l + 1)*vpl, cell[p]);
        }
        double r = 0.0;
#pragma unroll
        for (int k = 0; k < ADJ_TR_MAX; ++k) {
            const double q = hf[k] ? 0.5*(pm[k] + pe[k]) : pm[k];
            r += w[k]*q*oe[k];
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            r += vflux_w_weight(G, l + 1)*wt[p]*q1*o1[p];
            r += vflux_w_weight(G, l)*wt[p]*q0*o0[p];
        }
        put(Fb + nsh + (i64)l*vpl, ep, r);
        q0 = q1; o0[0] = o1[0]; o0[1] = o1[1];
    }
}

__global__ void __launch_bounds__(ATPB) k_vflux_adj_w(DevGrid G, const double *pv, const double *ob, double *Fb, Span sp)
{
    /* vertical F of cell h at level l: the w terms of the cell's edges at
       layers l (ipw slot 6) and l - 1 (slot 7) (vorticity_flux.c:110-187);
       all loads first, layer indices clamped, out-of-range terms masked */
    const Blk bk = xcd_block(sp);
    const unsigned h = bk.x*ATPB + threadIdx.x;
    const int nsh = G.nsh, nvh = G.nvh, vpl = G.vpl, L = G.L;
    if (h >= (unsigned)nsh) return;
    const int l = (int)bk.y;
    const int ne = h < GAME_N_PENT ? 5 : 6;
    const int la = l <= L - 1 ? l : L - 1, lb = l >= 1 ? l - 1 : 0;
    const double w6 = at(G.ipwT + ((i64)la*8 + 6)*nsh, h), w7 = at(G.ipwT + ((i64)lb*8 + 7)*nsh, h);
    double q[6], oa[6], obb[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        const unsigned e = at(G.c_e + (i64)j*nsh, h);
        q[j] = at(pv + (i64)l*2*nvh, e);
        oa[j] = at(ob + nsh + (i64)la*vpl, e);
        obb[j] = at(ob + nsh + (i64)lb*vpl, e);
    }
    double r = 0.0;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        if (j >= ne) continue;
        if (l <= L - 1) r += -0.5*w6*q[j]*oa[j];
        if (l >= 1) r += -0.5*w7*q[j]*obb[j];
    }
    put(Fb + (i64)l*vpl, h, r);
}

/* ------------------------------------------------------------------ */
/* inner product^T in its first argument                                 */
/* ------------------------------------------------------------------ */
__global__ void __launch_bounds__(ATPB) k_ip_adj(DevGrid G, AdjTables A, const double *b, const double *ib,
                                                 double *ab, double scale, int acc)
{
    /* acc 1: ab += scale*result, 2: ab = scale*result, 0: ab = result.  One thread per edge and
       level, which does the cell of its number too */
    const Blk bk = linear_block();
    const unsigned t = bk.x*ATPB + threadIdx.x;
    const int nsh = G.nsh, L = G.L, l = (int)bk.y;
    const i64 row = (i64)l*G.vpl;
    if (t < (unsigned)G.nvh && l < L) {
        const unsigned fr = G.from[t], to = G.to[t];
        const unsigned sf = (unsigned)A.slot_from[t]*(unsigned)nsh + fr, st = (unsigned)A.slot_to[t]*(unsigned)nsh + to;
        const double *wl = G.ipwT + (i64)l*8*nsh, *il = ib + (i64)l*nsh;
        const double old = acc == 1 ? at(ab + row + nsh, t) : 0.0;
        const double r = at(b + row + nsh, t)*(at(wl, sf)*at(il, fr) + at(wl, st)*at(il, to));
        put(ab + row + nsh, t, acc ? old + scale*r : r);
    }
    if (t < (unsigned)nsh) {
        const double old = acc == 1 ? at(ab + row, t) : 0.0;
        double s = 0.0;
        if (l >= 1) s += at(G.ipwT + ((i64)(l - 1)*8 + 7)*nsh, t)*at(ib + (i64)(l - 1)*nsh, t);
        if (l <= L - 1) s += at(G.ipwT + ((i64)l*8 + 6)*nsh, t)*at(ib + (i64)l*nsh, t);
        const double r = at(b + row, t)*s;
        put(ab + row, t, acc ? old + scale*r : r);
    }
}

/* ------------------------------------------------------------------ */
/* batched three-band solve and its adjoint (element j of column k at    */
/* j*ncol + k, so lanes read consecutive words)                          */
/* ------------------------------------------------------------------ */
/* One column per lane with its quotients and solution in LDS (systems of TL_MIN
   to TL_ROWS rows): the rows of the next batch are loaded while the lane
   eliminates the current ones, so a wave has 32 row loads in flight where the
   walking kernel below waits for four at every row, and the quotients and the
   intermediate solution cost no traffic.  Each block is one wave of `lanes`
   columns, 64 up to 64 rows and 32 beyond, which keeps its LDS within 64 KiB.
   Bound by memory for many columns and by the recurrence's divisions for few
   (batches of 16 rows gain nothing, and staging a block's rows in LDS for one
   lane per column, 67 and 114 us at 163,842 columns, less).  us per solve and
   per adjoint, walking and here: 26 rows of 163,842 columns 183 together -> 39
   and 58 (4.3 and 5.3 TB/s), 55 rows of 10,243 columns 77 and 105 -> 17 and
   20.  Each value is formed as the walking kernel forms it.  The solve here reads
   all rows of a column before it writes one, the adjoint all rows of the bands
   and of xb, and of x each row before it writes that row of an output. */
#define TL_ROWS 128
#define TL_B 8
static int tl_lanes(int n) { return n <= 64 ? 64 : 32; }
/* the walking kernel for more rows, and for fewer than four, of which a batch
   of eight loads each several times (us per solve and adjoint of 1,000,003
   columns, walking and here: one row 17 and 21, 29 and 38; two 28 and 38, 43
   and 55; three 38 and 53, 44 and 58; four 54 and 83, 54 and 77); it keeps the
   quotients in a work array, which the reverse step (two rows or more) has not */
#define TL_MIN 4
static bool tl_walk(int n, const double *work) { return n > TL_ROWS || (n < TL_MIN && work); }
/* rows j0 .. j0 + TL_B - 1 of column k of the block (the arrays begin at the
   block's first column, so that any int is a valid column count: the 32-bit
   offset of at() takes the lane alone): lo[j - 1], d[j], up[j], r[j]; rows that
   the system does not have repeat its last, and a single row has no bands */
struct TlRows { double lo[TL_B], d[TL_B], up[TL_B], r[TL_B]; };
__device__ __forceinline__ TlRows tl_load(const double *lo, const double *d, const double *up, const double *r, int n,
                                          int ncol, int j0, unsigned k)
{
    TlRows x;
#pragma unroll
    for (int t = 0; t < TL_B; ++t) {
        const int j = j0 + t < n ? j0 + t : n - 1, jl = j > 0 ? j - 1 : 0, ju = j < n - 1 ? j : jl;
        x.lo[t] = n > 1 ? at(lo + (i64)jl*ncol, k) : 0.0;
        x.up[t] = n > 1 ? at(up + (i64)ju*ncol, k) : 0.0;
        x.d[t] = at(d + (i64)j*ncol, k);
        x.r[t] = at(r + (i64)j*ncol, k);
    }
    return x;
}

/* column_solvers.c:641-667 downwards; quotients and solution to this lane's
   LDS columns q and s (stride lanes) */
__device__ __forceinline__ void tl_down(const double *lo, const double *d, const double *up, const double *r, int n,
                                        int ncol, unsigned k, double *q, double *s, int lanes)
{
    TlRows cur = tl_load(lo, d, up, r, n, ncol, 0, k);
    double ep = 0.0, x = 0.0;
    for (int j0 = 0; j0 < n; j0 += TL_B) {
        const TlRows nxt = tl_load(lo, d, up, r, n, ncol, j0 + TL_B < n ? j0 + TL_B : j0, k);
#pragma unroll
        for (int t = 0; t < TL_B; ++t) {
            const int j = j0 + t;
            if (j < n) {
                if (j == 0) {
                    if (n > 1) ep = cur.up[t]/cur.d[t];
                    x = cur.r[t]/cur.d[t];
                } else {
                    const double den = cur.d[t] - ep*cur.lo[t];
                    x = (cur.r[t] - x*cur.lo[t])/den;
                    if (j < n - 1) ep = cur.up[t]/den;
                }
                q[j*lanes] = ep;
                s[j*lanes] = x;
            }
        }
        cur = nxt;
    }
}

__global__ void __launch_bounds__(64) k_thomas_lds(int n, int ncol, const double *c, const double *d, const double *e,
                                                   const double *r, double *x)
{
    extern __shared__ double lds[];
    const int lanes = (int)blockDim.x;
    const unsigned k = threadIdx.x;
    const i64 k0 = (i64)xcd_x()*lanes;
    if (k0 + k >= ncol) return;
    c += k0; d += k0; e += k0; r += k0; x += k0;
    double *q = lds + k, *s = q + n*lanes;
    tl_down(c, d, e, r, n, ncol, k, q, s, lanes);
    double xj = 0.0;
#pragma unroll 4
    for (int j = n - 1; j >= 0; --j) {
        xj = j == n - 1 ? s[j*lanes] : s[j*lanes] - q[j*lanes]*xj;
        put(x + (i64)j*ncol, k, xj);
    }
}

/* the transposed solve A^T rb = xb (sub-diagonal e, super-diagonal c) and the
   band cotangents -rb x^T */
__global__ void __launch_bounds__(64) k_thomas_adj_lds(int n, int ncol, const double *c, const double *d, const double *e,
                                                       const double *x, const double *xb, double *rb, double *cb,
                                                       double *db, double *eb)
{
    extern __shared__ double lds[];
    const int lanes = (int)blockDim.x;
    const unsigned k = threadIdx.x;
    const i64 k0 = (i64)xcd_x()*lanes;
    if (k0 + k >= ncol) return;
    c += k0; d += k0; e += k0; x += k0; xb += k0; rb += k0; cb += k0; db += k0; eb += k0;
    double *q = lds + k, *s = q + n*lanes;
    tl_down(e, d, c, xb, n, ncol, k, q, s, lanes);
    /* upwards, the solution's rows loaded TL_B ahead */
    auto load = [&](int j1, double *y) {
#pragma unroll
        for (int t = 0; t < TL_B; ++t) y[t] = at(x + (i64)(j1 - t > 0 ? j1 - t : 0)*ncol, k);
    };
    double cur[TL_B], nxt[TL_B], rj = 0.0, xj = 0.0;
    load(n - 1, cur);
    for (int j1 = n - 1; j1 >= 0; j1 -= TL_B) {
        load(j1 - TL_B > 0 ? j1 - TL_B : 0, nxt);
#pragma unroll
        for (int t = 0; t < TL_B; ++t) {
            const int j = j1 - t;
            if (j >= 0) {
                const double r1 = rj, x1 = xj;   /* row j + 1 */
                rj = j == n - 1 ? s[j*lanes] : s[j*lanes] - q[j*lanes]*rj;
                xj = cur[t];
                put(rb + (i64)j*ncol, k, rj);
                put(db + (i64)j*ncol, k, -rj*xj);
                if (j < n - 1) {
                    put(cb + (i64)j*ncol, k, -r1*xj);
                    put(eb + (i64)j*ncol, k, -rj*x1);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TL_B; ++t) cur[t] = nxt[t];
    }
}

/* one column per lane, for systems of more rows and of fewer than TL_MIN */
__global__ void __launch_bounds__(ATPB) k_thomas(int n, int ncol, const double *c, const double *d, const double *e,
                                                 const double *r, double *x, double *ep)
{
    const unsigned k = blockIdx.x*ATPB + threadIdx.x;
    if (k >= (unsigned)ncol) return;
    /* column_solvers.c:641-667 */
    double epj = (n > 1) ? e[k]/d[k] : 0.0, xj = r[k]/d[k];
    ep[k] = epj;
    x[k] = xj;
    for (int j = 1; j < n; ++j) {
        const i64 o = (i64)j*ncol + k, om = o - ncol;
        const double den = d[o] - epj*c[om];
        if (j < n - 1) epj = e[o]/den;
        xj = (r[o] - xj*c[om])/den;
        ep[o] = epj;
        x[o] = xj;
    }
    for (int j = n - 2; j >= 0; --j) {
        const i64 o = (i64)j*ncol + k;
        xj = x[o] - ep[o]*xj;
        x[o] = xj;
    }
}

/* A^T rbar = xbar (A^T has sub-diagonal e and super-diagonal c), then the
   coefficient cotangents -rbar x^T on the three bands */
__global__ void __launch_bounds__(ATPB) k_thomas_adj(int n, int ncol, const double *c, const double *d,
                                                     const double *e, const double *x, const double *xb,
                                                     double *rb, double *cb, double *db, double *eb, double *ep)
{
    const unsigned k = blockIdx.x*ATPB + threadIdx.x;
    if (k >= (unsigned)ncol) return;
    double epj = (n > 1) ? c[k]/d[k] : 0.0, yj = xb[k]/d[k];
    ep[k] = epj;
    rb[k] = yj;
    for (int j = 1; j < n; ++j) {
        const i64 o = (i64)j*ncol + k, om = o - ncol;
        const double den = d[o] - epj*e[om];
        if (j < n - 1) epj = c[o]/den;
        yj = (xb[o] - yj*e[om])/den;
        ep[o] = epj;
        rb[o] = yj;
    }
    for (int j = n - 2; j >= 0; --j) {
        const i64 o = (i64)j*ncol + k;
        yj = rb[o] - ep[o]*yj;
        rb[o] = yj;
    }
    for (int j = 0; j < n; ++j) {
        const i64 o = (i64)j*ncol + k;
        db[o] = -rb[o]*x[o];
        if (j < n - 1) {
            cb[o] = -rb[o + ncol]*x[o];
            eb[o] = -rb[o]*x[o + ncol];
        }
    }
}

/* ------------------------------------------------------------------ */
namespace adj {

/* the edge kernels also do the cells of their numbers, fewer than the edges (nvh = 3 nsh - 6) */
#define CELL_GRID grid_of(G.nsh, G.split_adj_c)
#define EDGE_GRID grid_of(G.nvh, G.split_adj_e)
#define CELL_SPAN span_of(G.nsh, G.L, G.split_adj_c)
#define EDGE_SPAN span_of(G.nvh, G.L, G.split_adj_e)

void grad_adjoint(const DevGrid &G, const AdjTables &, const double *gb, double *fb, hipStream_t st, double gs,
                  int acc)
{ LAUNCH("k_grad_adj", k_grad_adj, CELL_GRID, dim3(ATPB), st, G, gb, fb, gs, acc, CELL_SPAN); }

void divv_h(const DevGrid &G, const double *in, double *out, hipStream_t st)
{
    if (G.flat) LAUNCH("k_divv", k_divv<true>, CELL_GRID, dim3(ATPB), st, G, in, out, CELL_SPAN);
    else LAUNCH("k_divv", k_divv<false>, CELL_GRID, dim3(ATPB), st, G, in, out, CELL_SPAN);
}

void divv_h_adjoint(const DevGrid &G, const AdjTables &A, const double *db, double *Fb, hipStream_t st)
{ LAUNCH("k_divv_adj", k_divv_adj, EDGE_GRID, dim3(ATPB), st, G, A, db, Fb, EDGE_SPAN); }

void curl_triangles_adjoint(const DevGrid &G, const AdjTables &A, const double *zb, double *wb, hipStream_t st,
                            int acc)
{ LAUNCH("k_curl_adj", k_curl_adj, EDGE_GRID, dim3(ATPB), st, G, A, zb, wb, acc, EDGE_SPAN); }

void rhombus_density(const DevGrid &G, const double *rho, double *out, hipStream_t st)
{ LAUNCH("k_rhombus", k_rhombus, EDGE_GRID, dim3(ATPB), st, G, rho, out, EDGE_SPAN); }

void rhombus_density_adjoint(const DevGrid &G, const AdjTables &A, const double *db, double *rb, hipStream_t st)
{ LAUNCH("k_rhombus_adj", k_rhombus_adj, CELL_GRID, dim3(ATPB), st, G, A, db, rb, CELL_SPAN); }

void vorticity_flux_adjoint(const DevGrid &G, const AdjTables &A, const double *pv, const double *ob, double *Fb,
                            hipStream_t st)
{
    LAUNCH("k_vflux_adj_e", k_vflux_adj_e, EDGE_GRID, dim3(ATPB), st, G, A, pv, ob, Fb, EDGE_SPAN);
    LAUNCH("k_vflux_adj_w", k_vflux_adj_w, grid_of(G.nsh, G.L + 1), dim3(ATPB), st, G, pv, ob, Fb, span_of(G.nsh, 1, 1));
}

void inner_product_adjoint(const DevGrid &G, const AdjTables &A, const double *b, const double *ib, double *ab,
                           hipStream_t st, double scale, int acc)
{ LAUNCH("k_ip_adj", k_ip_adj, grid_of(G.nvh, G.L + 1), dim3(ATPB), st, G, A, b, ib, ab, scale, acc); }

void thomas(int n, int ncol, const double *c, const double *d, const double *e, const double *r, double *x,
            double *work, hipStream_t st)
{
    if (tl_walk(n, work)) {
        LAUNCH("k_thomas", k_thomas, dim3(((unsigned)ncol + ATPB - 1u)/ATPB), dim3(ATPB), st, n, ncol, c, d, e, r, x, work);
        return;
    }
    const int lanes = tl_lanes(n);
    const dim3 g(((unsigned)ncol + (unsigned)lanes - 1u)/(unsigned)lanes), b((unsigned)lanes);
    const size_t lds = (size_t)2*n*lanes*sizeof(double);
    LAUNCH_SHM("k_thomas", k_thomas_lds, g, b, lds, st, n, ncol, c, d, e, r, x);
}

void thomas_adjoint(int n, int ncol, const double *c, const double *d, const double *e, const double *x,
                    const double *xb, double *rb, double *cb, double *db, double *eb, double *work, hipStream_t st)
{
    if (tl_walk(n, work)) {
        LAUNCH("k_thomas_adj", k_thomas_adj, dim3(((unsigned)ncol + ATPB - 1u)/ATPB), dim3(ATPB), st, n, ncol, c, d, e, x, xb, rb, cb, db, eb, work);
        return;
    }
    const int lanes = tl_lanes(n);
    const dim3 g(((unsigned)ncol + (unsigned)lanes - 1u)/(unsigned)lanes), b((unsigned)lanes);
    const size_t lds = (size_t)2*n*lanes*sizeof(double);
    LAUNCH_SHM("k_thomas_adj", k_thomas_adj_lds, g, b, lds, st, n, ncol, c, d, e, x, xb, rb, cb, db, eb);
}

}  // namespace adj

/* ------------------------------------------------------------------ */
/* scratch of the allocation-free three-band solve                     */
/* ------------------------------------------------------------------ */
/* The elimination quotients of game_gpu_op_thomas_noalloc live here instead
   of in a caller's work buffer: THOMAS_SCRATCH_DOUBLES doubles (64 MiB) that
   every GPU the library runs on holds from module load to process end.  In
   host code `scratch` names a host-side stand-in, never the device memory:
   only the address hipGetSymbolAddress returns for the current device (kept
   per device below) may be passed to a kernel. */
static __device__ __align__(256) double scratch[THOMAS_SCRATCH_DOUBLES];

namespace {
const int SCRATCH_DEVICES = 64;
double *g_scratch_ptr[SCRATCH_DEVICES] = {nullptr};
}

namespace adj {

int thomas_scratch_resolve(char *err, size_t nerr)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        snprintf(err, nerr, "hipGetDevice failed: %s", hipGetErrorString(e));
        return -1;
    }
    if (dev < 0 || dev >= SCRATCH_DEVICES) {
        snprintf(err, nerr, "device %d is beyond the %d devices the solver scratch supports", dev, SCRATCH_DEVICES);
        return -1;
    }
    if (g_scratch_ptr[dev]) return 0;
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
        snprintf(err, nerr, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
        return -1;
    }
    g_scratch_ptr[dev] = (double *)p;
    return 0;
}

double *thomas_scratch(void)
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SCRATCH_DEVICES) return nullptr;
    return g_scratch_ptr[dev];
}

}  // namespace adj
