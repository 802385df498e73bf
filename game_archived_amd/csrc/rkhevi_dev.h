/*
 * rkhevi_dev.h -- device-side data of the RKHEVI step (shared by the HIP files).
 *
 * Fields keep the reference's element order (see include/game_rkhevi.h), so
 * one thread per (layer, horizontal index) with the horizontal index fastest
 * reads and writes whole cache lines; neighbour gathers go through the
 * reference's own index tables.
 */
#ifndef GAME_RKHEVI_DEV_H
#define GAME_RKHEVI_DEV_H

#include <hip/hip_runtime.h>

#define GAME_N_PENT 12
/* threads per block of the kernels with one thread per element of a row */
#define TPB 256
#define GAME_MAX_LAYERS 64
#define SH_COLUMN GAME_MAX_LAYERS

/* src/game_constants.h */
#define GC_T_0 273.15
#define GC_N_A (6.02214076e23)
#define GC_P_0 100000.0
#define GC_C_D_V 717.942189
#define GC_C_V_V 1396.475121
#define GC_C_D_P 1005.0
#define GC_M_D (GC_N_A*0.004810e-23)
#define GC_M_V (GC_N_A*0.002991e-23)
#define GC_R_D 287.057811
#define GC_R_V 461.524879

typedef long long i64;

/* grid tables and metrics (struct grid / dualgrid members) on the device */
struct DevGrid {
    int nsh, nvh, nt, vpl, dvpl, L, n_oro, n_const, n_cond, moist;
    int flat;   /* slope == 0 everywhere: every terrain-correction term is an exact zero */
    i64 s, v, curl;
    double radius, toa;
    const double *nd, *vol, *area, *zs, *zv, *phi, *gm, *slope, *thbg, *exbg, *exbg_grad;
    /* the inner-product weights in layer-major, slot-major order, so that
       lanes of consecutive cells read consecutive addresses:
       ipwT[(l*8 + j)*nsh + h] is weight j of cell h in layer l */
    const double *ipwT;
    /* terrain grids: -0.5*ipw*slope of every cell's edges in the terrain
       layers, vcw[(k*6 + j)*nsh + h] for layer L - n_oro + k and slot j (the
       weights of the vertical contravariant correction); null when flat */
    const double *vcw;
    const double *tw, *drw, *dnd, *dzv, *darea, *fvec;
    const int *from, *to, *adj, *sgn, *ti, *tmc, *dri, *dfrom, *dto, *vit, *vst;
    /* the tables the step's kernels read, slot-major, so that a wave's lanes
       read consecutive words (the reference keeps an item's slots together:
       a wave of edges touches 80 cache lines for one TRSK weight each):
       per cell the edges c_e[j*nsh + h] and the cells across them c_n, and
       the bits j where the edge's sign is positive (h is its from-cell),
       c_from; per edge the TRSK weights, edges and PV indices e_tw, e_ti, e_tm
       [j*nvh + e] and the rhombus cells and weights e_rc, e_rw; per triangle
       its edges t_e[j*nt + t], with the top bit set where the sign is
       negative.  A pentagon's sixth slot holds its first edge and its own
       cell; the fifth TRSK slot of a pentagon's side holds the side's first
       entries: valid indices whose terms the kernels leave out */
    const unsigned *c_e, *c_n, *c_from, *e_ti, *e_tm, *e_rc, *t_e;
    const double *e_tw, *e_rw;
    /* per-edge differences that calc_pot_vort forms for its density
       extrapolation to the top and the surface, read exactly as the
       reference's struct layout serves them (vorticities.c:48-71) */
    const double *pv_top_dz1, *pv_top_dz2, *pv_sfc_dz1, *pv_sfc_dz2;
    /* Klemp damping coefficient of every interior interface, (L-1)*NSH */
    const double *damp;
    /* (0.5 dt)/vol of every grid box for the dt of the last step (the tracer
       solver's implicit weight times dt over the volume); the runtime refills
       it when dt changes */
    double *idv;
    /* numbers of layer chunks (gridDim.y) of the kernels that walk a column:
       per cell the levels of the vertical TRSK flux, per edge (PV and TRSK
       flux; the gradients), per triangle, and of the terrain levels of the
       vertical corrections */
    int split_cell_w, split_edge, split_grad, split_tri, split_vcc;
    /* the same of the operator adjoints' kernels, per cell and per edge */
    int split_adj_c, split_adj_e;
    /* 1: tracer solver with one (column, tracer) per lane; 0: a column over the waves of a block */
    int gd_streaming;
    /* mixed form, a precision probe: bit 0 rounds the density tendencies,
       bit 1 the rhotheta_v tendency, to FP32 after the scalar tendencies
       (the precision of FP32 storage, not its bytes) */
    int round_tendencies;
    /* 1: sound-wave solver with one column per lane; 0: three phases over LDS */
    int vw_streaming;
    /* layers per thread of the sediment heat: 1, 2, 5 or SH_COLUMN, all; 0: by the grid's size */
    int sh_run;
    /* 1: temperature and phase transitions as two kernels instead of one */
    int unfused_phase;
};

struct DevState {
    double *rho, *rt, *tp, *ep, *wind;   /* rho, rhotheta_v, theta_v_pert, exner_pert, wind */
};

/* work arrays of the step; TW = double in the FP64 form, float in the mixed
   form (register arithmetic stays FP64 in both) */
template <typename TW>
struct DevWorkT {
    /* diagnostics */
    TW *flux, *rvt, *pv, *temp, *vsq;
    double *flux2, *flux_divv;   /* reference diagnostics the step leaves untouched */
    /* forcings */
    TW *pgrad_old, *pgrad_nl, *pgrad_l, *pgc_v, *vsq_grad, *pvt;
    /* the pressure-gradient part of the momentum tendency, formed with the
       gradient: ohw*old - chw*(nl + l) at edges, -cvw*(nl + l) at interior w
       points (vector_tendencies_expl.c's weights for the step's implicit weight) */
    TW *pgrad_comb;
    /* irreversible quantities */
    TW *ptr, *phr, *sed_heat;
    /* vertical contravariant corrections of wind, gas mass flux and rhotheta_v
       flux in the terrain-following levels, 3 x n_oro x NSH (unused when flat) */
    double *vcc;
    /* wind tendency (the FP64 form keeps it in the tendency state) */
    TW *td_wind;
    /* c_p of ice and of liquid water at the step's temperature, 2 x S
       (condensate k takes c_p k & 1): the temperature is fixed for the whole
       step, so each value is formed once */
    TW *cpc;
    /* gas density over total density of the step's old state, S (formed with
       the temperature; read by the pressure gradient at the first substep) */
    double *gas_frac;
};
typedef DevWorkT<double> DevWork;
typedef DevWorkT<float> DevWorkF;

struct StepConsts {
    double dt, impl_weight, damping_start, damping_max, snow_v, rain_v, cloud_v;
};

/* Workgroups are dispatched to the eight XCDs round-robin (workgroup i on
   XCD i % 8), each XCD with its own L2.  The gather kernels renumber their
   workgroups so that each XCD takes one contiguous range of the grid (x, the
   horizontal blocks, fastest; then y, the chunks of layers): the neighbour
   data a workgroup shares with the next one then sits in the same L2 instead
   of being fetched by several XCDs.  Giving each XCD an eighth of x in every
   chunk instead, so that the chunks share its tables, was slower (moist
   scalar transport 389 -> 445 us at res 7 x 26).  Span carries the layers per
   chunk and the reciprocal of gridDim.x: with divisions in the kernels (this
   one, and 64-bit ones in the layer split) a wave spent over 300 scalar
   instructions before its first load. */
#define N_XCD 8u
struct Span { int run; unsigned rcp; };
struct Blk { unsigned x, y; };
__device__ __forceinline__ unsigned xcd_linear(unsigned lin, unsigned T)
{
    const unsigned q = T/N_XCD, r = T%N_XCD, x = lin%N_XCD, k = lin/N_XCD;
    return (x < r) ? x*(q + 1) + k : r*(q + 1) + (x - r)*q + k;
}
/* (m % gx, m/gx) by the reciprocal of span_of: ceil(2^32/gx) is at most gx - 1
   parts of 2^32 too large, so for every 32-bit m the quotient is at most one
   too large.  2^32 itself, for one block per row (at most 256 columns or edges),
   has no 32 bits: rcp is 0 there and m the quotient */
__host__ __device__ __forceinline__ Blk block_at(unsigned m, unsigned gx, unsigned rcp)
{
    Blk b;
    b.y = rcp ? (unsigned)(((unsigned long long)m*rcp) >> 32) : m;
    b.x = m - b.y*gx;
    if ((int)b.x < 0) { --b.y; b.x += gx; }
    return b;
}
__device__ __forceinline__ Blk xcd_block(Span sp)
{
    return block_at(xcd_linear(blockIdx.y*gridDim.x + blockIdx.x, gridDim.x*gridDim.y), gridDim.x, sp.rcp);
}
/* the blocks as they are dispatched: for kernels that mostly stream, where eight
   ranges far apart cost more than neighbours in one L2 give (us per launch,
   renumbered and as dispatched: flat PV with the mass flux at res 7 x 26 270
   and 240, mixed 226 and 202; but kinetic energy at res 6 31 and 34, vertical
   corrections over the res 6 mountain 44 and 56, sound waves 198 and 228) */
__device__ __forceinline__ Blk linear_block() { return Blk{blockIdx.x, blockIdx.y}; }
/* the same renumbering of a one-dimensional grid */
__device__ __forceinline__ unsigned xcd_x() { return xcd_linear(blockIdx.x, gridDim.x); }
/* grid of n horizontal elements in `chunks` chunks, and its Span for `layers` layers or levels */
static dim3 grid_of(int n, int chunks) { return dim3((unsigned)((n + TPB - 1)/TPB), (unsigned)chunks); }
static Span span_of(int n, int layers, int chunks)
{
    const unsigned gx = (unsigned)((n + TPB - 1)/TPB);
    return Span{(layers + chunks - 1)/chunks, gx > 1 ? (unsigned)(((1ULL << 32) + gx - 1)/gx) : 0u};
}

/* layers [l0, l1) of a chunk when n layers are split into chunks of `run`;
   the last chunk may be shorter (or empty) */
__device__ __forceinline__ void layer_chunk(int n, unsigned chunk, int run, int &l0, int &l1)
{
    l0 = (int)chunk*run;
    l1 = l0 + run < n ? l0 + run : n;
}

/* element i of a row whose address is the same for the whole wave: the row's
   base stays in scalar registers and the lane adds a 32-bit byte offset, so a
   load costs one instruction and the offset is shared by every row read at
   the same index (a 64-bit element index takes an address pair per load).  The
   byte offset has 32 bits: i is below 2^29 for doubles, which a row of any
   grid that fits the memory is */
template <typename T>
__device__ __forceinline__ T at(const T *row, unsigned i)
{
    return *(const T *)((const char *)row + (size_t)(i*(unsigned)sizeof(T)));
}
template <typename T>
__device__ __forceinline__ void put(T *row, unsigned i, T v)
{
    *(T *)((char *)row + (size_t)(i*(unsigned)sizeof(T))) = v;
}

/* Thomas algorithm (column_solvers.c:641-667) on rows j*NCOL + col of LDS
   arrays c, d, e, r (n rows): the multipliers overwrite e, the solution r.
   The next row is read before the current one is written, so each step
   waits on its division chain only, not on an LDS round trip. */
template <int NCOL>
__device__ __forceinline__ void thomas_lds(const double *cc, const double *dd, double *ee, double *rr, int n, int col)
{
    double ep = 0.0, x;
    const double d0 = dd[col];
    if (n > 1) ep = ee[col]/d0;
    x = rr[col]/d0;
    ee[col] = ep; rr[col] = x;
    double cp = cc[col], dn = 0.0, en = 0.0, rn = 0.0;
    if (n > 1) { dn = dd[NCOL + col]; en = ee[NCOL + col]; rn = rr[NCOL + col]; }
#pragma unroll 4
    for (int j = 1; j < n; ++j) {
        const int o = j*NCOL + col, on = (j + 1 < n ? j + 1 : j)*NCOL + col;
        const double cpn = cc[o], dnn = dd[on], enn = ee[on], rnn = rr[on];
        const double den = dn - ep*cp;
        if (j < n - 1) ep = en/den;
        x = (rn - x*cp)/den;
        ee[o] = ep; rr[o] = x;
        cp = cpn; dn = dnn; en = enn; rn = rnn;
    }
    /* back substitution, upwards */
    double eb = 0.0, rb = 0.0;
    if (n > 1) { eb = ee[(n - 2)*NCOL + col]; rb = rr[(n - 2)*NCOL + col]; }
#pragma unroll 4
    for (int j = n - 2; j >= 0; --j) {
        const int o = j*NCOL + col, om = (j > 0 ? j - 1 : 0)*NCOL + col;
        const double ebn = ee[om], rbn = rr[om];
        x = rb - eb*x;
        rr[o] = x;
        eb = ebn; rb = rbn;
    }
}

__device__ __forceinline__ double density_total(const DevGrid &G, const double *rho, i64 i)
{   /* derived_quantities.c:83-95: left-to-right sum from 0 */
    double r = 0.0;
    for (int k = 0; k < G.n_const; ++k) r += rho[k*G.s + i];
    return r;
}

/* dictionary.c:111-190 */
__device__ __forceinline__ double c_p_ice(double t)
{
    if (t > GC_T_0) t = GC_T_0;
    if (t < 20.0) t = 20.0;
    double q = t/125.1;
    double r = -2.0572 + 0.14644*t + 0.06163*t*exp(-(q*q));
    return r/GC_M_V;
}

__device__ __forceinline__ double c_p_water(double t)
{
    double tc = t - GC_T_0, r;
    /* a branch, not a select: a wave whose boxes are all above or all below
       freezing evaluates one of the two polynomials */
    /* the reference's integer powers pow(x, 3.0) and pow(x, 4.0) as products
       (within about one ulp of glibc's pow, as the device's pow is) */
    if (tc >= 0.0) {
        if (tc > 35.0) tc = 35.0;
        double a = tc - 35.0;
        const double a2 = a*a;
        r = 0.9979 + 3.1e-6*(a*a) + 3.8e-9*(a2*a2);
    } else {
        if (tc < -37.0) tc = -37.0;
        const double t2 = tc*tc;
        r = 1.000938 - 2.7052e-3*tc - 2.3235e-5*(tc*tc) + 4.3778e-6*(t2*tc) + 2.7136e-7*(t2*t2);
    }
    return 4186.8*r;
}

/* per-kernel timing with HIP events on the launch stream (off unless enabled) */
struct KernelTimer {
    virtual void begin(const char *name, hipStream_t st) = 0;
    virtual void end(hipStream_t st) = 0;
};
extern KernelTimer *g_kernel_timer;

#define LAUNCH_SHM(NAME, KERNEL, GRID, BLOCK, SHM, STREAM, ...)                     \
    do {                                                                            \
        if (g_kernel_timer) g_kernel_timer->begin(NAME, STREAM);                    \
        hipLaunchKernelGGL(KERNEL, GRID, BLOCK, SHM, STREAM, __VA_ARGS__);          \
        if (g_kernel_timer) g_kernel_timer->end(STREAM);                            \
    } while (0)
#define LAUNCH(NAME, KERNEL, GRID, BLOCK, STREAM, ...) LAUNCH_SHM(NAME, KERNEL, GRID, BLOCK, 0, STREAM, __VA_ARGS__)

#endif
