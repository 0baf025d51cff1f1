// shyhip_conz.hip -- 3D scalar advection-diffusion (conz3d) on gfx950.
//
// Two kernels per substep:
//   k_conz_elem[_lds]  one work-item per element-layer of a precomputed work list
//                (workgroups of equal work whatever the depth): horizontal
//                advective fluxes (upwind rule, the itvd=2 TVD scheme with
//                precomputed upwind interpolation weights, or the itvd=1
//                scheme with node gradients) -> 3*fl per vertex, stored by
//                the vertex's position in its node's colour-order incidence
//                list.
//   k_conz_node  one workgroup per node tile (at most 256 nodes and 256
//                node-layers).  Phase 1, one work-item per node-layer: the
//                vertical diffusion/advection terms of the node column (they
//                depend on an element only through its bottom layer, so
//                three variants cover every element), then the incident
//                elements gathered in colour order -- the order in which
//                conz3d_omp accumulates them (concentration_omp.f90:243-290)
//                -- with the element terms of conz3d_element (:355-753), and
//                the boundary mass flux of conz3d_nodes; the column
//                coefficients go to LDS.  Phase 2, one work-item per node:
//                the implicit vertical solve (:757-886) and the write-back.
// Horizontal diffusion (rkpar > 0) is part of the element term; nudging,
// sinking and loads belong to launches of a single tracer (k_conz_node's EXT).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>

#include "shyhip_internal.h"

namespace shy {

// Up to kMaxTracers tracers are transported by one launch of each phase:
// they share every hydrodynamic load, the element flux coefficients and the
// node column matrix; each keeps its own arithmetic, identical to its
// transport alone.
constexpr int kMaxTracers = 2;

template <typename S>
struct ConzArgs {
    int nkn, nel, nlvdi, nlv, itvd, itvdv;
    int clip[kMaxTracers];
    double dt, az, ad, aa, rso, rsn;
    float difmol;
    const int *nen3v, *ilhv, *ilhkv, *iextb, *ibnd;
    const double *geo, *dis;
    const int *nkc_ptr, *nkc_el;
    const int4 *ek, *ep;             // elements' vertices and colour-order list positions (see Mesh)
    const int *slot_lev;
    const double *slot_aj4;
    int nslot;                       // 3 * nel
    const int *elem_iext;
    const int4 *tvd_up;              // upwind nodes, layers and weights of the ordered pairs (see Mesh)
    const double2 *tvd_w;
    const double *tvd_w2;
    const int *uoff, *uptr;          // node-layers of a workgroup's entries and places in them (see Mesh)
    const unsigned *uvert, *upair;
    const S *utn, *vtn, *uto, *vto, *uln, *vln;
    const S *hdkn, *hdko, *hden, *hdeo, *wln, *difv, *mflux;
    S *c[kMaxTracers];               // tracers (in/out)
    const S *cbound[kMaxTracers];    // source concentrations (may be null)
    S *hbuf;                         // element terms [l-1][list position][NT]
    int *err;
    // ensembles whose members run different numbers of substeps: member
    // istot (null: all run istot), node/element -> member, this substep and
    // the step as (double)(S)dt; members already past their last substep
    // are left alone
    const int *mem_istot, *node_mem, *elem_mem;
    int isact;
    double dtp;
    // element-layer work list and node tiles (see Mesh)
    const int *eitem, *ntile;
    int n_eitem;
    const int4 *nent;                // node tiles' entries, and the nodes' first places in their tiles
    const int *nplace;
    int clear_below;                 // also write the zeros below the bottom
    // the step's element-layer records (k_conz_prep)
    int *rec_code;
    uint2 *rec_pair;
    double *rec_f;
    S *rec_s;
    // the launch's single tracer's own terms (null: none): nudging factor
    // robs with target cobs and rate rtauv, sinking wsink * wsinkv, loads
    // rload * load (node arrays like the tracer; wsinkv on interfaces)
    float robs, wsink, rload;
    const S *cobs, *rtauv, *wsinkv;
    S *load;
    // horizontal diffusion (rkpar > 0): factor, element diffusivities
    // [l*nel + ie] and the weights [(3*(ii-1) + (iii-1))*nel + ie]
    float rkpar;
    const S *difhv, *wdif;
    // itvd = 1: the node-layer list, the element-order incidence lists and
    // the node gradients [((l-1)*NT + t)*2 + xy][nkn] (after hbuf's terms)
    const int *nitem, *inc_cnt, *inc_el, *nk_el;
    int n_nitem;
    S *grad;
};

template <typename S>
__device__ inline double cval(const ConzArgs<S> &a, int t, int l, int k) {
    const S v = a.c[t][(size_t)(l - 1) * a.nkn + k];
    if (a.clip[t] && v < (S)1.e-15) return 0.;
    return (double)v;
}

// ------------------------------------------------------------------ element phase
// One work-item per entry of the element-layer work list (Mesh::conz_eitem):
// chunks of kConzChunk consecutive elements, each chunk layer by layer with
// its elements ascending, so that a layer's loads are contiguous.  A
// workgroup takes kThreads consecutive entries, whatever the depth of the
// elements they come from, so every workgroup does the same work.
//
// Everything of an element-layer that depends on the flow only -- the flux
// coefficients f, the upwind case, and for TVD the two pairs of the flow
// direction with their Courant numbers -- holds for all the substeps of a
// step (the transports, velocities and the substep length do not change
// within it).  k_conz_prep computes it once per step into a record per list
// entry (columns indexed by the entry, so every load is contiguous);
// k_conz_elem then reads the record, gathers the tracers at the element's
// nodes and upwind points, and applies the upwind rule or the limiter.  The
// arithmetic is that of the element terms computed in one pass (the record
// holds the values, not approximations of them).
//
// What bounds both: the memory they move.  The record holds what the flow
// decides, 44 bytes (FP64) or 36 (FP32); an element's vertices, list
// positions, upwind nodes and weights come from the mesh's tables, which the
// layers of a chunk share in cache.  With all of it in the record, 144 bytes,
// it took 119 us a substep for the element terms and 132 us a step for the
// record on 300k nodes of 20 layers (FP64, T and S); now 92 and 56.

// v[i] for a run-time i in 0..2 without indexing a register array
template <typename T>
__device__ inline T sel3(const T (&v)[3], int i) {
    return i == 0 ? v[0] : (i == 1 ? v[1] : v[2]);
}

// A record's columns, each n_eitem long: the case word, the flux coefficients
// (RF_*, double), and in the tracers' precision (RS_*) the Courant numbers of
// the two pairs and, for itvd = 1 only, the pairs' edge vectors; where the
// element phase reads the node-layers from LDS, the two pairs' words of
// Mesh::conz_upair (rec_pair).
//
// With one or two vertices taking inflow one vertex, p, stands against the
// other two, a and b (ascending): the only one with inflow or the only one
// without.  The pairs are (p, a) and (p, b), upstream to downstream, or with
// two inflows (a, p) and (b, p); the terms of a and b are the flux
// coefficient times the pair's face value and p's the negative of their sum.
// The upwind rule has the same form with the upstream value for the face
// (except that with one inflow p's term is its own coefficient's), so the
// whole phase is a straight line.
// The case word: p - 1 (bits 0-1), two inflows (2), any flux (3), TVD pairs
// present (4), upwind points present (5, 6).
enum { RF_A = 0, RF_B, RF_P, RF_N };
enum { RS_ALFA = 0, RS_EDGE = 2, RS_N = 6 };
static inline size_t conz_rec_code_bytes(int n) { return ((size_t)n * sizeof(int) + 15) / 16 * 16; }

// the tracers' terms of one list position in hbuf
template <typename S, int NT>
struct alignas(NT * sizeof(S)) Terms {
    S t[NT];
};

// the place of the ordered pair (ic, id), 1-based, among an element's six
__device__ inline int tvd_pair(int ic, int id) { return 2 * (ic - 1) + ((id == (ic % 3) + 1) ? 0 : 1); }

template <typename S>
__global__ __launch_bounds__(kThreads) void k_conz_prep(ConzArgs<S> a) {
    using R = S;
    const int i = xcd_block() * kThreads + threadIdx.x;
    if (i >= a.n_eitem) return;
    const int n = a.n_eitem;
    const unsigned w = (unsigned)a.eitem[i];
    const int ie = (int)(w >> 5), l = (int)(w & 31u) + 1;
    const int nel = a.nel;
    const bool use_tvd = a.itvd > 0;
    double gb[3], gc[3];
#pragma unroll
    for (int ii = 0; ii < 3; ii++) {
        gb[ii] = a.geo[(size_t)ii * nel + ie];
        gc[ii] = a.geo[(size_t)(3 + ii) * nel + ie];
    }
    const size_t o = (size_t)(l - 1) * nel + ie;
    const S un = a.utn[o], uo = a.uto[o], vn = a.vtn[o], vo = a.vto[o];
    int iext = 1;
    S ul = 0, vl = 0;
    double dis3[3] = {0., 0., 0.}, ajr0 = 0.;
    if (use_tvd) {
        iext = a.elem_iext[ie];
        ul = a.uln[o];
        vl = a.vln[o];
#pragma unroll
        for (int ii = 0; ii < 3; ii++) dis3[ii] = a.dis[(size_t)ii * nel + ie];
        ajr0 = a.geo[(size_t)6 * nel + ie];
    }
    const double azt = 1. - a.az;
    const double us = a.az * (double)un + azt * (double)uo;
    const double vs = a.az * (double)vn + azt * (double)vo;
    int itot = 0, isum = 0;
    double f[3];
    for (int ii = 0; ii < 3; ii++) {
        f[ii] = us * gb[ii] + vs * gc[ii];
        if (f[ii] < 0.) { itot++; isum += ii + 1; }
    }
    const bool flux = itot >= 1 && itot <= 2;
    const int itot2 = itot - 1, itot1 = 2 - itot;
    const int ip = flux ? itot2 * (6 - isum) + itot1 * isum : 1;
    int code = (ip - 1) | (itot == 2 ? 4 : 0) | (flux ? 8 : 0);
    S alfa[2] = {0, 0};
    unsigned up[2] = {0, 0};
    if (use_tvd && iext == 0 && flux) {
        // TVD fluxes (tvd_fluxes, tvd_admin.f90:673-823): the two pairs
        // (ic, id) of the flow direction -- the vertices other than ip,
        // ascending -- and their Courant numbers and upwind points
        code |= 1 << 4;
        const R ajr = (R)(24. * ajr0);
        const double dte = a.mem_istot ? a.dtp / (double)a.mem_istot[a.elem_mem[ie]] : a.dt;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int ii = k == 0 ? (ip == 1 ? 2 : 1) : (ip == 3 ? 2 : 3);
            const int ic = itot2 * ii + itot1 * ip;
            const int id = itot2 * ip + itot1 * ii;
            const int iop = 6 - (id + ic);
            const int tet1 = 1 + iop % 3;
            R dx = (R)((double)ajr * sel3(gc, iop - 1));
            dx = (R)(-2 * (tet1 == id ? 1 : 0)) * dx + dx;
            R dy = (R)((double)ajr * sel3(gb, iop - 1));
            dy = (R)(-2 * (tet1 == ic ? 1 : 0)) * dy + dy;
            const R dis = (R)sel3(dis3, iop - 1);
            const R vel = (R)fabs((double)(ul * dx + vl * dy)) / dis;
            alfa[k] = (R)((dte * (double)vel) / (double)dis);
            if (a.itvd == 2) {
                const int pr = tvd_pair(ic, id);
                if (a.upair) up[k] = a.upair[(size_t)pr * n + i];
                else if (a.tvd_up[(size_t)pr * nel + ie].w >= l) code |= 1 << (5 + k);
            } else {
                // itvd = 1: the edge vector, for the gradient's projection
                a.rec_s[(size_t)(RS_EDGE + 2 * k) * n + i] = dx;
                a.rec_s[(size_t)(RS_EDGE + 2 * k + 1) * n + i] = dy;
            }
        }
    }
    a.rec_code[i] = code;
    if (a.upair) a.rec_pair[i] = make_uint2(up[0], up[1]);
    a.rec_f[(size_t)RF_A * n + i] = sel3(f, ip == 1 ? 1 : 0);
    a.rec_f[(size_t)RF_B * n + i] = sel3(f, ip == 3 ? 1 : 2);
    if (!(code & (4 | 16))) a.rec_f[(size_t)RF_P * n + i] = sel3(f, ip - 1);
    if (use_tvd) {
#pragma unroll
        for (int k = 0; k < 2; k++) a.rec_s[(size_t)(RS_ALFA + k) * n + i] = alfa[k];
    }
}

// ------------------------------------------------------------------ gradient TVD
// itvd = 1 (tvd_grad_3d, tvd_admin.f90:478-543, called before each substep's
// conz3d_omp, concentration.f90:744): each tracer's gradient at every
// node-layer, the mean of the gradients of the incident elements that have
// the layer, weighted by the element area ev(10), in the precision of the
// tracers.  k_tvd_grad_elem, one work-item per element-layer entry, writes
// the element's gradient times its area (the reference's ggx*area,
// ggy*area) into the element-term scratch, which k_conz_elem overwrites
// only afterwards; k_tvd_grad_node, one work-item per node-layer entry,
// adds the incident elements' products and areas in element order -- the
// order of the reference's element loop -- and divides.

// element-layer (ie, l) gradient product of tracer t, component xy, in hbuf
__device__ inline size_t egrad_at(int nel, int NT, int t, int xy, int l, int ie) {
    return ((size_t)((l - 1) * NT + t) * 2 + xy) * nel + ie;
}
__device__ inline size_t ngrad_at(int nkn, int NT, int t, int xy, int l, int k) {
    return ((size_t)((l - 1) * NT + t) * 2 + xy) * nkn + k;
}

template <typename S, int NT>
__global__ __launch_bounds__(kThreads) void k_tvd_grad_elem(ConzArgs<S> a) {
    using R = S;
    const int i = xcd_block() * kThreads + threadIdx.x;
    if (i >= a.n_eitem) return;
    const unsigned w = (unsigned)a.eitem[i];
    const int ie = (int)(w >> 5), l = (int)(w & 31u) + 1;
    if (a.mem_istot && a.isact > a.mem_istot[a.elem_mem[ie]]) return;
    const int nel = a.nel, nkn = a.nkn;
    int kn[3];
    R b[3], c[3];
#pragma unroll
    for (int ii = 0; ii < 3; ii++) {
        kn[ii] = a.nen3v[3 * ie + ii];
        b[ii] = (R)a.geo[(size_t)ii * nel + ie];
        c[ii] = (R)a.geo[(size_t)(3 + ii) * nel + ie];
    }
    const R area = (R)a.geo[(size_t)6 * nel + ie];
    S v[NT][3];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int ii = 0; ii < 3; ii++) {
            const S x = a.c[t][(size_t)(l - 1) * nkn + kn[ii]];
            v[t][ii] = (a.clip[t] && x < (S)1.e-15) ? (S)0 : x;
        }
    S *eg = a.hbuf;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        R ggx = 0, ggy = 0;
#pragma unroll
        for (int ii = 0; ii < 3; ii++) {
            ggx = ggx + (R)v[t][ii] * b[ii];
            ggy = ggy + (R)v[t][ii] * c[ii];
        }
        eg[egrad_at(nel, NT, t, 0, l, ie)] = ggx * area;
        eg[egrad_at(nel, NT, t, 1, l, ie)] = ggy * area;
    }
}

template <typename S, int NT>
__global__ __launch_bounds__(kThreads) void k_tvd_grad_node(ConzArgs<S> a) {
    using R = S;
    const int i = xcd_block() * kThreads + threadIdx.x;
    if (i >= a.n_nitem) return;
    const unsigned w = (unsigned)a.nitem[i];
    const int k = (int)(w >> 5), l = (int)(w & 31u) + 1;
    if (a.mem_istot && a.isact > a.mem_istot[a.node_mem[k]]) return;
    const int nel = a.nel, nkn = a.nkn;
    const S *eg = a.hbuf;
    // the first kIncWidth incident elements' data loaded at once (padding
    // slots hold element 0, a valid index), the rest one by one
    IncSlots inc;
    inc.load(a.inc_cnt, a.inc_el, nkn, k);
    int lv[kIncWidth];
    R ar[kIncWidth], gp[NT][2][kIncWidth];
#pragma unroll
    for (int s = 0; s < kIncWidth; s++) {
        const int ie = inc.pk[s] >> 2;
        lv[s] = a.ilhv[ie];
        ar[s] = (R)a.geo[(size_t)6 * nel + ie];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const bool has = lv[s] >= l;      // no product below the element's bottom
            gp[t][0][s] = has ? eg[egrad_at(nel, NT, t, 0, l, ie)] : (R)0;
            gp[t][1][s] = has ? eg[egrad_at(nel, NT, t, 1, l, ie)] : (R)0;
        }
    }
    R sx[NT], sy[NT], sa = 0;
#pragma unroll
    for (int t = 0; t < NT; t++) sx[t] = sy[t] = 0;
#pragma unroll
    for (int s = 0; s < kIncWidth; s++)
        if (s < inc.cnt && lv[s] >= l) {
            sa = sa + ar[s];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                sx[t] = sx[t] + gp[t][0][s];
                sy[t] = sy[t] + gp[t][1][s];
            }
        }
    const int q0 = a.nkc_ptr[k], q1 = a.nkc_ptr[k + 1];
    for (int q = q0 + kIncWidth; q < q1; q++) {
        const int ie = a.nk_el[q] >> 2;
        if (a.ilhv[ie] < l) continue;
        sa = sa + (R)a.geo[(size_t)6 * nel + ie];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            sx[t] = sx[t] + eg[egrad_at(nel, NT, t, 0, l, ie)];
            sy[t] = sy[t] + eg[egrad_at(nel, NT, t, 1, l, ie)];
        }
    }
#pragma unroll
    for (int t = 0; t < NT; t++) {
        a.grad[ngrad_at(nkn, NT, t, 0, l, k)] = sa > (R)0 ? sx[t] / sa : sx[t];
        a.grad[ngrad_at(nkn, NT, t, 1, l, k)] = sa > (R)0 ? sy[t] / sa : sy[t];
    }
}

// A pair's flux with the limited face value (tvd_fluxes): upstream conc,
// downstream cond, grad the limiter's upwind difference, flux coefficient f.
template <typename R>
__device__ inline double tvd_term(R conc, R cond, R grad, R alfa, double f) {
    const R rq = grad / (cond - conc) - (R)1;
    const R rf = (R)fabs((double)(conc - cond)) < (R)1.e-8 ? (R)-1 : rq;
    const double rfd = (double)rf;
    const R psi = (R)fmax(0., fmax(fmin(1., 2. * rfd), fmin(2., rfd)));
    const R conf = conc + (R)0.5 * psi * (cond - conc) * ((R)1 - alfa);
    return (double)(R)((double)conf * f);
}

// GRAD: itvd = 1 (the upstream node's gradient in place of the upwind point)
// HDIF: horizontal diffusion (rkpar > 0): the element's term
// rk3 hmed wdiff (concentration_omp.f90:560-570,727-735) is taken off the
// advective term before it is stored
template <typename S, int NT, bool GRAD, bool HDIF>
__global__ __launch_bounds__(kThreads) void k_conz_elem(ConzArgs<S> a) {
    using R = S;
    const int i = xcd_block() * kThreads + threadIdx.x;
    if (i >= a.n_eitem) return;
    const int n = a.n_eitem, nkn = a.nkn, nel = a.nel;
    const bool use_tvd = a.itvd > 0;
    const unsigned w = (unsigned)a.eitem[i];
    const int code = a.rec_code[i];
    const double f[2] = {a.rec_f[(size_t)RF_A * n + i], a.rec_f[(size_t)RF_B * n + i]};
    R alfa[2] = {0, 0};
    if (use_tvd)
#pragma unroll
        for (int k = 0; k < 2; k++) alfa[k] = a.rec_s[(size_t)(RS_ALFA + k) * n + i];
    const int ie = (int)(w >> 5), l = (int)(w & 31u) + 1;
    if (a.mem_istot && a.isact > a.mem_istot[a.elem_mem[ie]]) return;
    const int p = code & 3;
    const bool two = code & 4, flux = code & 8, tvd = code & 16;
    const int4 kp = a.ek[ie], ep = a.ep[ie];
    // vertices and list positions of p, a and b
    const int kn[3] = {p == 0 ? kp.x : (p == 1 ? kp.y : kp.z), p == 0 ? kp.y : kp.x, p == 2 ? kp.y : kp.z};
    const int so[3] = {p == 0 ? ep.x : (p == 1 ? ep.y : ep.z), p == 0 ? ep.y : ep.x, p == 2 ? ep.y : ep.z};
    const size_t lo = (size_t)(l - 1) * nkn;
    S cr[NT][3];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int q = 0; q < 3; q++) cr[t][q] = a.c[t][lo + kn[q]];
    // a pair's upwind point (nodes, weights; also where there is none or the
    // element takes the upwind rule: valid addresses, not used) or gradient
    S cu[2][NT][3] = {};
    double tw[2][3] = {};
    if (use_tvd) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            if (GRAD) {
                const int kc = two ? kn[k + 1] : kn[0];
                if (tvd)
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        tw[k][q] = (double)a.rec_s[(size_t)(RS_EDGE + 2 * k + q) * n + i];
#pragma unroll
                        for (int t = 0; t < NT; t++) cu[k][t][q] = a.grad[ngrad_at(nkn, NT, t, q, l, kc)];
                    }
            } else {
                const int v = k == 0 ? (p == 0 ? 1 : 0) : (p == 2 ? 1 : 2);
                const size_t po = (size_t)(two ? tvd_pair(v + 1, p + 1) : tvd_pair(p + 1, v + 1)) * nel + ie;
                const int4 up = a.tvd_up[po];
                const double2 w01 = a.tvd_w[po];
                tw[k][0] = w01.x; tw[k][1] = w01.y; tw[k][2] = a.tvd_w2[po];
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    cu[k][t][0] = a.c[t][lo + up.x];
                    cu[k][t][1] = a.c[t][lo + up.y];
                    cu[k][t][2] = a.c[t][lo + up.z];
                }
            }
        }
    }
    double fp = 0.;
    if (!two && !tvd) fp = a.rec_f[(size_t)RF_P * n + i];
    auto clip = [&](int t, S v) -> S { return (a.clip[t] && v < (S)1.e-15) ? (S)0 : v; };
    double fl[NT][3];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const R cp = clip(t, cr[t][0]);
        double u[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const R ci = clip(t, cr[t][k + 1]);
            const R conc = two ? ci : cp, cond = two ? cp : ci;
            u[k] = f[k] * (double)conc;
            if (use_tvd) {
                R grad;
                if (GRAD) {
                    // itvd = 1: grad = 2 (g(kc) . edge)
                    grad = (R)2. * (cu[k][t][0] * (R)tw[k][0] + cu[k][t][1] * (R)tw[k][1]);
                } else {
                    double zh = 0.;
#pragma unroll
                    for (int q = 0; q < 3; q++) zh = zh + (double)clip(t, cu[k][t][q]) * tw[k][q];
                    grad = cond - (((code >> (5 + k)) & 1) ? (R)zh : cond);
                }
                const double term = tvd_term(conc, cond, grad, alfa[k], f[k]);
                if (tvd) u[k] = term;
            }
        }
        fl[t][0] = two || tvd ? -(u[0] + u[1]) : fp * (double)cp;
        fl[t][1] = u[0];
        fl[t][2] = u[1];
        // no flux when no vertex or all take inflow
#pragma unroll
        for (int q = 0; q < 3; q++) fl[t][q] = flux ? fl[t][q] : 0.;
    }
    double hd[NT][3];
#pragma unroll
    for (int t = 0; t < NT; t++) hd[t][0] = hd[t][1] = hd[t][2] = 0.;
    if (HDIF) {
        // rk3 = 3 rkpar difhv in the tracers' precision, hmed the element
        // layer's thickness at this substep, wdiff(ii) = sum over iii of
        // wdifhv(iii, ii) c(iii), in the element's own order of the vertices
        const size_t o = (size_t)(l - 1) * nel + ie;
        double rso = a.rso;
        if (a.mem_istot) rso = (a.isact - 1) / (double)a.mem_istot[a.elem_mem[ie]];
        const double rk3 = (double)((R)3 * (R)a.rkpar * a.difhv[o]);
        const double hmed = rso * (double)a.hden[o] + (1. - rso) * (double)a.hdeo[o];
        double wv[3][3];
#pragma unroll
        for (int ii = 0; ii < 3; ii++)
#pragma unroll
            for (int q = 0; q < 3; q++) wv[ii][q] = (double)a.wdif[(size_t)(3 * ii + q) * nel + ie];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const double cv[3] = {(double)clip(t, cr[t][0]), (double)clip(t, cr[t][1]), (double)clip(t, cr[t][2])};
            const double cl[3] = {p == 0 ? cv[0] : cv[1], p == 0 ? cv[1] : (p == 1 ? cv[0] : cv[2]),
                                  p == 2 ? cv[0] : cv[2]};
            double h[3];
#pragma unroll
            for (int ii = 0; ii < 3; ii++) {
                double waux = 0.;
#pragma unroll
                for (int q = 0; q < 3; q++) waux = waux + wv[ii][q] * cl[q];
                h[ii] = rk3 * hmed * waux;
            }
            hd[t][0] = sel3(h, p);
            hd[t][1] = sel3(h, p == 0 ? 1 : 0);
            hd[t][2] = sel3(h, p == 2 ? 1 : 2);
        }
    }
    Terms<S, NT> *const hb = (Terms<S, NT> *)a.hbuf + (size_t)(l - 1) * a.nslot;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        Terms<S, NT> v;
#pragma unroll
        for (int t = 0; t < NT; t++) v.t[t] = (S)(HDIF ? 3. * fl[t][q] - hd[t][q] : 3. * fl[t][q]);
        hb[so[q]] = v;
    }
}

// The same for itvd = 2 without horizontal diffusion, over the node-layers of
// the workgroup's entries (Mesh::conz_uoff): each is read once into LDS, both
// tracers side by side, and an entry gathers there by 10-bit places.
//
// What bounds it: memory, at 3.7 TB/s of the 4.8 of a copy.  Gathering the
// tracers at three vertices and six upwind nodes from memory, 18 gathers of
// 8 bytes, kept the address path busy instead (1,250 cache accesses a
// wavefront against 670): 107 us a launch on 300k nodes of 20 layers (FP64, T
// and S) against 92, 15.1 against 12.4 on the 50k-node lagoon, FP32 on 285k
// nodes 42.6 against 33.  The lists hold 620 node-layers on average where
// the elements are numbered with locality; beyond kConzUniq the copies into
// LDS outgrow the gathers they save and k_conz_elem runs.
template <typename S, int NT>
__global__ __launch_bounds__(kThreads) void k_conz_elem_lds(ConzArgs<S> a) {
    using R = S;
    __shared__ Terms<S, NT> val[kConzUniq];
    const int wg = xcd_block();
    const int n = a.n_eitem, nel = a.nel;
    const int i0 = wg * kThreads + threadIdx.x;
    const int i = min(i0, n - 1);             // (the last workgroup's spare work-items read its last entry)
    // the workgroup's node-layers; kConzUniq of them at most
    const int u0 = a.uptr[wg], nu = a.uptr[wg + 1] - u0;
    constexpr int kPer = kConzUniq / kThreads;
    int uo[kPer];
#pragma unroll
    for (int q = 0; q < kPer; q++) {
        const int j = q * kThreads + threadIdx.x;
        uo[q] = j < nu ? a.uoff[u0 + j] : -1;
    }
    const unsigned w = (unsigned)a.eitem[i];
    const int code = a.rec_code[i];
    const unsigned uv = a.uvert[i];
    const uint2 rp = a.rec_pair[i];
    const unsigned up[2] = {rp.x, rp.y};
    const double f[2] = {a.rec_f[(size_t)RF_A * n + i], a.rec_f[(size_t)RF_B * n + i]};
    const R alfa[2] = {a.rec_s[(size_t)(RS_ALFA + 0) * n + i], a.rec_s[(size_t)(RS_ALFA + 1) * n + i]};
    Terms<S, NT> uc[kPer];
#pragma unroll
    for (int q = 0; q < kPer; q++)
#pragma unroll
        for (int t = 0; t < NT; t++) uc[q].t[t] = uo[q] >= 0 ? a.c[t][uo[q]] : (S)0;
    const int ie = (int)(w >> 5), l = (int)(w & 31u) + 1;
    const int p = code & 3;
    const bool two = code & 4, flux = code & 8, tvd = code & 16;
    const int4 ep = a.ep[ie];
    double tw[2][3];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int v = k == 0 ? (p == 0 ? 1 : 0) : (p == 2 ? 1 : 2);
        const size_t po = (size_t)(two ? tvd_pair(v + 1, p + 1) : tvd_pair(p + 1, v + 1)) * nel + ie;
        const double2 w01 = a.tvd_w[po];
        tw[k][0] = w01.x; tw[k][1] = w01.y; tw[k][2] = a.tvd_w2[po];
    }
    double fp = 0.;
    if (!two && !tvd) fp = a.rec_f[(size_t)RF_P * n + i];
    bool on = i0 < n;
    if (a.mem_istot && a.isact > a.mem_istot[a.elem_mem[ie]]) on = false;
    auto clip = [&](int t, S v) -> S { return (a.clip[t] && v < (S)1.e-15) ? (S)0 : v; };
#pragma unroll
    for (int q = 0; q < kPer; q++) {
        if (uo[q] < 0) continue;
        Terms<S, NT> v;
#pragma unroll
        for (int t = 0; t < NT; t++) v.t[t] = clip(t, uc[q].t[t]);
        val[q * kThreads + threadIdx.x] = v;
    }
    __syncthreads();
    if (!on) return;
    // list positions and values of p, a and b
    const int so[3] = {p == 0 ? ep.x : (p == 1 ? ep.y : ep.z), p == 0 ? ep.y : ep.x, p == 2 ? ep.y : ep.z};
    const int vp[3] = {10 * p, p == 0 ? 10 : 0, p == 2 ? 10 : 20};
    Terms<S, NT> cr[3], cu[2][3];
#pragma unroll
    for (int q = 0; q < 3; q++) {
        cr[q] = val[(uv >> vp[q]) & (kConzUniq - 1)];
#pragma unroll
        for (int k = 0; k < 2; k++) cu[k][q] = val[(up[k] >> (10 * q)) & (kConzUniq - 1)];
    }
    double fl[NT][3];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const R cp = cr[0].t[t];
        double u[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const R ci = cr[k + 1].t[t];
            const R conc = two ? ci : cp, cond = two ? cp : ci;
            double zh = 0.;
#pragma unroll
            for (int q = 0; q < 3; q++) zh = zh + (double)cu[k][q].t[t] * tw[k][q];
            const R grad = cond - ((up[k] >> 30) ? (R)zh : cond);
            const double term = tvd_term(conc, cond, grad, alfa[k], f[k]);
            u[k] = tvd ? term : f[k] * (double)conc;
        }
        fl[t][0] = two || tvd ? -(u[0] + u[1]) : fp * (double)cp;
        fl[t][1] = u[0];
        fl[t][2] = u[1];
    }
    Terms<S, NT> *const hb = (Terms<S, NT> *)a.hbuf + (size_t)(l - 1) * a.nslot;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        Terms<S, NT> v;
#pragma unroll
        for (int t = 0; t < NT; t++) v.t[t] = (S)(3. * (flux ? fl[t][q] : 0.));
        hb[so[q]] = v;
    }
}

// ------------------------------------------------------------------ node phase
// The limited face value of the vertical TVD flux (vertical_flux_ie,
// tvd_admin.f90:930-1016): centre conc, downstream cond, upstream conu,
// Courant number alfa.
__device__ inline double tvd_face(double conc, double cond, double conu, double alfa) {
    const double rq = (cond - conu) / (cond - conc) - 1.;
    const double rf = fabs(conc - cond) < (double)1.e-8f ? -1. : rq;
    const double psi = fmax(0., fmax(fmin(1., 2. * rf), fmin(2., rf)));
    return conc + 0.5 * psi * (cond - conc) * (1. - alfa);
}

// Node tiles (Mesh::conz_ntile, built at set-up): consecutive nodes, at most
// the node_tile setting (<= kNodeTileMax = the workgroup size) and at most
// kNodeItems node-layers, so that phase 1 is one pass of the workgroup
// whatever the depth of the tile's columns.
// EXT: the tracer's own terms (one tracer per launch): sinking in the
// vertical velocity, nudging in the explicit term (concentration_omp.f90:
// 479,697-701,727-735) and loads after the boundary flux (:816-834)
//
// What bounds it: the chain of a work-item -- its loads, about 20 FP64
// divisions, the column solve -- in one pass of 2,400 wavefronts, then the
// tracers' traffic on large basins.  Everything of a node-layer that only the
// mesh decides (its node and place in the tile, its list's start and length,
// which incident elements reach the layer, the next one and the one after)
// is one 16-byte table entry (Mesh::conz_nent), so the loads form two rounds:
// the entry, then all the rest.  Listing the tile's node-layers in the kernel
// instead (a ballot per layer, one work-item adding up 48 counts, three
// barriers), reading the list start and the elements' layers as data, and
// evaluating a limited face per sign of the vertical velocity took 26.5 us a
// launch on the 50k-node lagoon and 159 us on 300k nodes of 20 layers (T and
// S, FP64), against 21.5 and 115 us; 20.4 and 105 with an incident element's
// terms of both tracers in one load and selects in place of branches.
template <typename S, int NT, bool EXT>
__global__ __launch_bounds__(kThreads) void k_conz_node(ConzArgs<S> a) {
    using R = S;
    // phase-1 results by place in the tile (node after node, top down):
    // right-hand sides of NT tracers and the three diagonals of the column
    // matrix
    __shared__ double cnP[NT][kNodeItems], cdP[kNodeItems], cloP[kNodeItems], chiP[kNodeItems];
    const int nkn = a.nkn;
    const int tile = xcd_block();
    const int4 ent = a.nent[(size_t)tile * kNodeItems + threadIdx.x];
    const int k0 = a.ntile[tile], tn = a.ntile[tile + 1] - k0;
    const double ad = a.ad, aa = a.aa, adt = 1. - a.ad, aat = 1. - a.aa;
    const bool btvdv = a.itvdv > 0;

    // phase 1: one work-item per node-layer; members past their last substep
    // are left alone
    bool on = ent.x >= 0;
    const int k = on ? ent.w : 0;
    if (a.mem_istot && on && a.isact > a.mem_istot[a.node_mem[k]]) on = false;
    if (on) {
        const int l = (ent.x & 31) + 1, lmaxk = ((ent.x >> 5) & 31) + 1, it = (ent.x >> 10) & 255;
        double dt = a.dt, rso = a.rso, rsn = a.rsn;
        if (a.mem_istot) {
            const int ist = a.mem_istot[a.node_mem[k]];
            const double rstot = ist;
            rso = (a.isact - 1) / rstot;
            rsn = a.isact / rstot;
            dt = a.dtp / rstot;
        }
        const double rsot = 1. - rso, rsnt = 1. - rsn;
        // incident elements in colour order: list positions q0 .. q0+cnt-1
        const int q0 = ent.y;
        int cnt = ent.x >> 18;
        if (cnt == kNodeCntMax) cnt = a.nkc_ptr[k + 1] - q0;
        // The first kIncWidth positions are read unconditionally (clamped to
        // the list), contiguous for the node; the last two pairs only by
        // wavefronts that hold such a node; the rest one by one.
        double saj[kIncWidth];
        Terms<S, NT> shf[kIncWidth];
        const Terms<S, NT> *const hb = (const Terms<S, NT> *)a.hbuf + (size_t)(l - 1) * a.nslot;
        const bool any6 = __any(cnt > 6), any8 = __any(cnt > 8);
#pragma unroll
        for (int s = 0; s < kIncWidth; s++) {
            saj[s] = 0.; shf[s] = {};
            if (s < 6 || (s < 8 ? any6 : any8)) {
                const int q = min(q0 + s, a.nslot - 1);
                saj[s] = a.slot_aj4[q];
                shf[s] = hb[q];
            }
        }
        // node column around l (zero outside 1..lmaxk)
        double ckw[NT][5], hokw[5], hnkw[5];
#pragma unroll
        for (int j = 0; j < 5; j++) {
            const int x = l - 2 + j;
            hokw[j] = 0.; hnkw[j] = 0.;
#pragma unroll
            for (int t = 0; t < NT; t++) ckw[t][j] = 0.;
            if (x >= 1 && x <= lmaxk) {
#pragma unroll
                for (int t = 0; t < NT; t++) ckw[t][j] = cval(a, t, x, k);
                if (j >= 1 && j <= 3) {
                    const size_t o = (size_t)(x - 1) * nkn + k;
                    const double hn = (double)a.hdkn[o], ho = (double)a.hdko[o];
                    hokw[j] = rso * hn + rsot * ho;
                    hnkw[j] = rsn * hn + rsnt * ho;
                }
            }
        }
        const double rvptop = (double)(R)(a.difv[(size_t)(l - 1) * nkn + k] + (R)a.difmol);
        const double rvpbot = (double)(R)(a.difv[(size_t)l * nkn + k] + (R)a.difmol);
        double wtop = (l == 1) ? 0. : (double)a.wln[(size_t)(l - 1) * nkn + k];
        double wbot = (double)a.wln[(size_t)l * nkn + k];
        double hfn = 0.;            // hold * fnudge of the tracer (EXT, NT = 1)
        if (EXT) {
            // the vertical velocity less the sinking, in the tracers' precision
            if (a.wsinkv) {
                if (l > 1)
                    wtop = (double)(R)(a.wln[(size_t)(l - 1) * nkn + k] -
                                       (R)a.wsink * a.wsinkv[(size_t)(l - 1) * nkn + k]);
                wbot = (double)(R)(a.wln[(size_t)l * nkn + k] - (R)a.wsink * a.wsinkv[(size_t)l * nkn + k]);
            }
            if (a.cobs) {
                const size_t o = (size_t)(l - 1) * nkn + k;
                const double fn = (double)a.robs * (double)a.rtauv[o] * ((double)a.cobs[o] - 1. * ckw[0][2]);
                hfn = hokw[2] * fn;
            }
        }
        // element terms of the three column truncations: bottom layer l
        // (v = 0), l+1 (v = 1) or deeper (v = 2; nothing below l+2 is read).
        // The truncation enters only through the layers below l: the
        // diffusion and vertical flux across the bottom interface exist
        // for v >= 1, and the upstream value beyond the next layer for v = 2.
        // Each distinct term is computed once, with the arithmetic of the
        // truncated column (vertical_flux_ie: zero at the column's ends).
        // Without a layer below l its coefficients are zero; the explicit
        // part of the diffusion (adt) is left out when there is none.
        const double hom = hokw[1], hoc = hokw[2], hop = hokw[3];
        const double hnm = hnkw[1], hnc = hnkw[2], hnp = hnkw[3];
        const double pm = (l - 1 >= 1) ? 1. : 0.;
        const double hmntop = 2. * rvptop * pm / (hnm + hnc);
        const double hmnbot[2] = {0., 2. * rvpbot * 1. / (hnc + hnp)};
        double hmotop = 0., hmobot = 0.;
        if (adt != 0.) {
            hmotop = 2. * rvptop * pm / (hom + hoc);
            hmobot = 2. * rvpbot * 1. / (hoc + hop);
        }
        // matrix coefficients: [0] for v = 0, [1] for v >= 1 (the lower
        // diagonal does not depend on the truncation)
        double clcv[2], clpv[2], clm = 0.;
#pragma unroll
        for (int v = 0; v < 2; v++) {
            const double hmb = hmnbot[v];
            double clc = 0. + ad * (hmntop + hmb);
            clm = 0. - ad * hmntop;
            double clp = 0. - ad * hmb;
            double w = wtop;
            if (w >= 0.) clc += aa * w;
            else clm += aa * w;
            w = (v == 0) ? 0. : wbot;
            if (w > 0.) clp -= aa * w;
            else clc -= aa * w;
            clcv[v] = clc; clpv[v] = clp;
        }
        // Courant numbers of the two interfaces (tracer-independent)
        double alfa_t = 0., alfa_b = 0.;
        if (btvdv) {
            alfa_t = dt * fabs(wtop) / (0.5 * (hom + hoc));
            alfa_b = dt * fabs(wbot) / (0.5 * (hoc + hop));
        }
        // (one array per variant, indexed by the tracer only: a run-time
        // variant index would put the terms in scratch memory)
        double fd0[NT], fd1[NT], fw0[NT], fw1[NT], fw2[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const double c0 = ckw[t][0], c1 = ckw[t][1], c2 = ckw[t][2], c3 = ckw[t][3], c4 = ckw[t][4];
            fd0[t] = adt * ((c2 - 0.) * 0. - (c1 - c2) * hmotop);
            fd1[t] = adt * ((c2 - c3) * hmobot - (c1 - c2) * hmotop);
            // flux across the top interface (none at the surface): [0]
            // without a layer below l, [1] with one.  They differ only for a
            // rising flow, whose upstream value [0] is the downstream one: the
            // limiter is zero there and the face takes the centre's value.
            double vt[2];
            {
                const double w = wtop;
                const bool up = w > 0.;
                double face = up ? c2 : c1;
                if (btvdv) face = tvd_face(face, up ? c1 : c2, up ? c3 : (l - 2 >= 1 ? c0 : c2), alfa_t);
                vt[1] = l >= 2 ? w * face : 0.;
                vt[0] = l >= 2 && up ? w * c2 : vt[1];
            }
            // flux across the bottom interface (none for v = 0): [0] for
            // v = 1, [1] for v = 2, differing in the same way
            double vb[2];
            {
                const double w = wbot;
                const bool up = w > 0.;
                double face = up ? c3 : c2;
                if (btvdv) face = tvd_face(face, up ? c2 : c3, up ? c4 : (l - 1 >= 1 ? c1 : c3), alfa_b);
                vb[1] = w * face;
                vb[0] = up ? w * c3 : vb[1];
            }
            fw0[t] = aat * (vt[0] - 0.);
            fw1[t] = aat * (vt[1] - vb[0]);
            fw2[t] = aat * (vt[1] - vb[1]);
        }
        // incident elements in colour order (conz3d_element's scatter)
        double cn[NT], cd = 0., clo = 0., chi = 0.;
#pragma unroll
        for (int t = 0; t < NT; t++) cn[t] = 0.;
        // One element's terms (whether it has layer l, the next one, the one
        // after; 4 * area, horizontal terms of the tracers).  A position
        // without the layer (or beyond the list) adds zeros, to sums that are
        // never -0.: straight line instead of a branch per position.
        // (A macro rather than a lambda: the lambda's captures stayed in scratch
        // memory.)
#define CONZ_ADD(has_, deep_, deeper_, aj4_, hf_)                                                   \
    do {                                                                                           \
        const bool has = (has_), deep = (deep_), deeper = (deeper_); /* layer, v >= 1, v == 2 */    \
        const double aj4 = has ? (aj4_) : 0.;                                                       \
        const Terms<S, NT> hf = (hf_);                                                              \
        _Pragma("unroll") for (int t = 0; t < NT; t++) {                                           \
            const double fw = deeper ? fw2[t] : (deep ? fw1[t] : fw0[t]);                          \
            const double fd = deep ? fd1[t] : fd0[t];                                              \
            cn[t] += aj4 * (hoc * ckw[t][2] + dt * (hfn + (has ? (double)hf.t[t] : 0.) - fw - fd)); \
        }                                                                                          \
        clo += aj4 * dt * clm;                                                                     \
        chi += aj4 * dt * (deep ? clpv[1] : clpv[0]);                                              \
        cd += aj4 * dt * (deep ? clcv[1] : clcv[0]) + aj4 * (1. + dt * 0.) * hnc;                  \
    } while (0)
        const unsigned reach = (unsigned)ent.z;
#pragma unroll
        for (int s = 0; s < kIncWidth; s++)
            if (s < 6 || (s < 8 ? any6 : any8))
                CONZ_ADD((reach >> s) & 1u, (reach >> (kIncWidth + s)) & 1u, (reach >> (2 * kIncWidth + s)) & 1u, saj[s],
                         shf[s]);
        for (int q = q0 + kIncWidth; q < q0 + cnt; q++) {
            const int ilev = a.slot_lev[q];
            if (ilev >= l) CONZ_ADD(true, ilev > l, ilev > l + 1, a.slot_aj4[q], hb[q]);
        }
#undef CONZ_ADD
        // conz3d_nodes: boundary mass flux
        if (a.mflux) {
            const size_t o = (size_t)(l - 1) * nkn + k;
            const double qflux = (double)a.mflux[o];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                double cconz = a.cbound[t] ? (double)a.cbound[t][o] : 0.;
                if (qflux < 0. && a.ibnd[k] > 0) cconz = ckw[t][2];
                cn[t] += dt * (qflux * cconz);
            }
        }
        if (EXT && a.load) {
            // erosion, or deposition of at most what the node-layer holds
            const size_t o = (size_t)(l - 1) * nkn + k;
            double loading = (double)((R)a.rload * a.load[o]);
            if (loading < 0.) {
                double cload = 0.;
                if (cn[0] > 0.) {
                    cload = -dt * loading;
                    cload = cn[0] * (1. - exp(-cload / cn[0]));
                } else if (cn[0] < 0.) {
                    cn[0] = 0.;
                }
                if (cload > cn[0]) atomicCAS(a.err, 0, ERR_CONZ);
                loading = -cload / dt;
                if (a.rload > 0.f) a.load[o] = (S)(loading / (double)a.rload);
                cn[0] += dt * loading;
            } else if (loading > 0.) {
                cn[0] += dt * loading;
            }
        }
#pragma unroll
        for (int t = 0; t < NT; t++) cnP[t][it] = cn[t];
        cdP[it] = cd; cloP[it] = clo; chiP[it] = chi;
    }
    __syncthreads();

    // phase 2: the column solve of conz3d_nodes, one work-item per node; the
    // tracers share the column matrix and its elimination.  Layer l of a
    // node lies l - 1 places after its first one.
    const int kk = threadIdx.x, kn = k0 + kk;
    if (kk >= tn) return;
    if (a.mem_istot && a.isact > a.mem_istot[a.node_mem[kn]]) return;
    const int lmaxk = a.ilhkv[kn], p0 = a.nplace[kn];
    auto cn = [&](int t, int l0) -> double & { return cnP[t][p0 + l0]; };
    auto cd = [&](int l0) -> double & { return cdP[p0 + l0]; };
    auto clo = [&](int l0) -> double & { return cloP[p0 + l0]; };
    auto chi = [&](int l0) -> double & { return chiP[p0 + l0]; };
    bool bad = false;
    if ((aa == 0. && ad == 0.) || a.nlv == 1) {
        for (int l = 1; l <= lmaxk; l++)
            if (cd(l - 1) != 0.)
#pragma unroll
                for (int t = 0; t < NT; t++) cn(t, l - 1) = cn(t, l - 1) / cd(l - 1);
    } else {
        // the elimination's chain runs through registers (chip, cnp); LDS
        // supplies the coefficients and keeps the forward results for the
        // back substitution
        const double aux0 = 1. / cd(0);
        double chip = chi(0) * aux0, cnp[NT];
        chi(0) = chip;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            cnp[t] = cn(t, 0) * aux0;
            cn(t, 0) = cnp[t];
        }
        for (int l = 2; l <= lmaxk; l++) {
            const double cdl = cd(l - 1), clol = clo(l - 1), chil = chi(l - 1);
            double cnl[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) cnl[t] = cn(t, l - 1);
            if (cdl == 0.) bad = true;
            const double aux = 1. / (cdl - clol * chip);
            chip = chil * aux;
            chi(l - 1) = chip;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                cnp[t] = (cnl[t] - clol * cnp[t]) * aux;
                cn(t, l - 1) = cnp[t];
            }
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
            double nx = cnp[t];
            for (int l = lmaxk - 1; l >= 1; l--) {
                nx = cn(t, l - 1) - nx * chi(l - 1);
                cn(t, l - 1) = nx;
            }
        }
    }
    if (bad) { atomicCAS(a.err, 0, ERR_CONZ); return; }
#pragma unroll
    for (int t = 0; t < NT; t++) {
        for (int l = 1; l <= lmaxk; l++) a.c[t][(size_t)(l - 1) * nkn + kn] = (S)cn(t, l - 1);
        // zero below the bottom: once per step (nothing else writes there)
        if (a.clear_below)
            for (int l = lmaxk + 1; l <= a.nlvdi; l++) a.c[t][(size_t)(l - 1) * nkn + kn] = (S)0;
    }
}

template <typename S>
static ConzArgs<S> conz_args(Model &M, const TracerSet &ts, int istot, int isact, void *hbuf, void *rec);

template <typename S, int NT>
static int conz_t(Model &M, const TracerSet &ts, int istot, int isact, hipStream_t st, void *hbuf, void *rec,
                  bool prep) {
    if (!M.m.conz_eitem || !M.m.conz_ntile) return hip_check(M, hipErrorNotInitialized, "conz3d: no basin");
    if (!rec) return hip_check(M, hipErrorInvalidValue, "conz3d: no element-layer record buffer");
    ConzArgs<S> a = conz_args<S>(M, ts, istot, isact, hbuf, rec);
    a.clear_below = prep;          // a step's first substep, and every substep called by itself
    const int ge = (M.m.n_eitem + kThreads - 1) / kThreads;
    if (prep) {
        launch_timed(M, T_CONZ_PREP, k_conz_prep<S>, dim3(ge), dim3(kThreads), 0, st, a);
        HIPCHK(M, hipGetLastError());
    }
    if (M.p.rkpar > 0.f && !a.wdif) return hip_check(M, hipErrorNotInitialized, "conz3d: no diffusion weights");
    if (a.itvd == 1) {
        if (!M.m.conz_nitem) return hip_check(M, hipErrorNotInitialized, "conz3d: no node-layer list");
        if (!a.grad) return hip_check(M, hipErrorInvalidValue, "conz3d: no gradient buffer");
        const int gn = (M.m.n_nitem + kThreads - 1) / kThreads;
        launch_timed(M, T_TVD_GRAD, k_tvd_grad_elem<S, NT>, dim3(ge), dim3(kThreads), 0, st, a);
        launch_timed(M, T_TVD_GRAD, k_tvd_grad_node<S, NT>, dim3(gn), dim3(kThreads), 0, st, a);
        HIPCHK(M, hipGetLastError());
        if (a.wdif) launch_timed(M, T_CONZ_ELEM, k_conz_elem<S, NT, true, true>, dim3(ge), dim3(kThreads), 0, st, a);
        else launch_timed(M, T_CONZ_ELEM, k_conz_elem<S, NT, true, false>, dim3(ge), dim3(kThreads), 0, st, a);
    } else if (a.uoff) {
        launch_timed(M, T_CONZ_ELEM, k_conz_elem_lds<S, NT>, dim3(ge), dim3(kThreads), 0, st, a);
    } else {
        if (a.wdif) launch_timed(M, T_CONZ_ELEM, k_conz_elem<S, NT, false, true>, dim3(ge), dim3(kThreads), 0, st, a);
        else launch_timed(M, T_CONZ_ELEM, k_conz_elem<S, NT, false, false>, dim3(ge), dim3(kThreads), 0, st, a);
    }
    HIPCHK(M, hipGetLastError());
    if (a.cobs || a.wsinkv || a.load) {
        if (NT != 1) return hip_check(M, hipErrorInvalidValue, "conz3d: tracer terms need one tracer per launch");
        launch_timed(M, T_CONZ_NODE, k_conz_node<S, 1, true>, dim3(M.m.n_ntile), dim3(kThreads), 0, st, a);
    } else {
        launch_timed(M, T_CONZ_NODE, k_conz_node<S, NT, false>, dim3(M.m.n_ntile), dim3(kThreads), 0, st, a);
    }
    HIPCHK(M, hipGetLastError());
    return 0;
}

// The arguments of substep isact of istot (zeroed first, so that their
// bytes, padding included, identify the launch).
template <typename S>
static ConzArgs<S> conz_args(Model &M, const TracerSet &ts, int istot, int isact, void *hbuf, void *rec) {
    ConzArgs<S> a;
    std::memset(&a, 0, sizeof a);
    a.nkn = M.nkn; a.nel = M.nel; a.nlvdi = M.nlvdi; a.nlv = M.nlv;
    a.itvd = M.p.itvd; a.itvdv = M.p.itvdv;
    const double rstot = istot;
    a.rso = (isact - 1) / rstot;
    a.rsn = isact / rstot;
    a.dt = (double)(S)M.p.dt / rstot;
    a.az = M.p.azpar; a.ad = M.p.adpar; a.aa = M.p.aapar; a.difmol = M.p.difmol;
    a.nen3v = M.m.nen3v; a.ilhv = M.m.ilhv; a.ilhkv = M.m.ilhkv; a.iextb = M.m.iextb; a.ibnd = M.m.ibnd;
    a.geo = M.m.geo; a.dis = M.m.dis;
    a.nkc_ptr = M.m.nk_ptr; a.nkc_el = M.m.nkc_el;
    a.ek = (const int4 *)M.m.conz_ek; a.ep = (const int4 *)M.m.conz_ep;
    a.slot_lev = M.m.slot_lev; a.slot_aj4 = M.m.slot_aj4; a.nslot = 3 * M.nel;
    a.tvd_up = (const int4 *)M.m.tvd_up; a.tvd_w = (const double2 *)M.m.tvd_w;
    a.tvd_w2 = M.m.tvd_w ? M.m.tvd_w + 12 * (size_t)M.nel : nullptr;
    a.elem_iext = M.m.elem_iext;
    if (M.p.itvd == 2 && !(M.p.rkpar > 0.f) && M.m.conz_uoff) {
        a.uoff = M.m.conz_uoff; a.uptr = M.m.conz_uptr; a.uvert = M.m.conz_uvert; a.upair = M.m.conz_upair;
    }
    a.utn = (const S *)M.s.utn; a.vtn = (const S *)M.s.vtn; a.uto = (const S *)M.s.uto; a.vto = (const S *)M.s.vto;
    a.uln = (const S *)M.s.uln; a.vln = (const S *)M.s.vln;
    a.hdkn = (const S *)M.s.hdkn; a.hdko = (const S *)M.s.hdko; a.hden = (const S *)M.s.hden;
    a.hdeo = (const S *)M.s.hdeo; a.wln = (const S *)M.s.wln; a.difv = (const S *)M.s.difv;
    a.mflux = M.has_mflux ? (const S *)M.s.mflux : nullptr;
    for (int t = 0; t < ts.n && t < kMaxTracers; t++) {
        a.c[t] = (S *)M.s.tracer[ts.itr[t]];
        a.cbound[t] = (const S *)ts.cbound[t];
        a.clip[t] = ts.clip[t];
    }
    a.isact = isact;
    a.dtp = (double)(S)M.p.dt;
    if (M.mem_istot_on) {
        a.mem_istot = M.cur_mem_istot; a.node_mem = M.d_node_mem; a.elem_mem = M.d_elem_mem;
    }
    a.hbuf = (S *)hbuf;
    a.err = M.d_err;
    a.eitem = M.m.conz_eitem; a.n_eitem = M.m.n_eitem; a.ntile = M.m.conz_ntile;
    a.nent = (const int4 *)M.m.conz_nent; a.nplace = M.m.conz_nplace;
    if (ts.n == 1 && tracer_has_terms(M, ts.itr[0])) {
        const int t = ts.itr[0];
        if (M.tr_robs[t] != 0.f && M.s.cobs[t] && M.s.rtauv[t]) {
            a.robs = M.tr_robs[t];
            a.cobs = (const S *)M.s.cobs[t];
            a.rtauv = (const S *)M.s.rtauv[t];
        }
        if (M.tr_wsink[t] != 0.f && M.s.wsinkv[t]) {
            a.wsink = M.tr_wsink[t];
            a.wsinkv = (const S *)M.s.wsinkv[t];
        }
        if (M.tr_rload[t] != 0.f && M.s.load[t]) {
            a.rload = M.tr_rload[t];
            a.load = (S *)M.s.load[t];
        }
    }
    if (M.p.rkpar > 0.f) {
        a.rkpar = M.p.rkpar;
        a.difhv = (const S *)M.s.difhv;
        a.wdif = (const S *)M.m.wdif;
    }
    a.nitem = M.m.conz_nitem; a.n_nitem = M.m.n_nitem;
    a.inc_cnt = M.m.inc_cnt; a.inc_el = M.m.inc_el; a.nk_el = M.m.nk_el;
    // the node gradients follow the element terms in the same buffer
    a.grad = (M.p.itvd == 1 && hbuf) ? (S *)hbuf + conz_hbuf_terms(M, ts.n) : nullptr;
    if (rec) {
        a.rec_code = (int *)rec;
        a.rec_pair = (uint2 *)((char *)rec + conz_rec_code_bytes(M.m.n_eitem));
        a.rec_f = (double *)(a.rec_pair + M.m.n_eitem);
        a.rec_s = (S *)(a.rec_f + 3 * (size_t)M.m.n_eitem);
    }
    return a;
}

size_t conz_record_bytes(const Model &M) {
    const size_t n = M.m.n_eitem;
    return conz_rec_code_bytes(M.m.n_eitem) + n * sizeof(uint2) + RF_N * n * sizeof(double) + (size_t)RS_N * n * M.esize();
}

size_t conz_hbuf_terms(const Model &M, int ntr) { return (size_t)ntr * 3 * M.nlvdi * M.nel; }
size_t conz_hbuf_elems(const Model &M, int ntr) {
    return conz_hbuf_terms(M, ntr) + (size_t)ntr * 2 * M.nlvdi * M.nkn;
}

// uvtopr (transforms.f90:215-270) at the open-boundary nodes followed by
// bndo_setbc = bndo_impbc + bndo_adjbc (bndo.f90:620-890): impose the
// boundary value, and on outflow take the weighted mean of the inner
// neighbours.  One wavefront per open-boundary node, one lane per layer; a
// layer with no inner neighbour deep enough takes the final value of the
// layer above, resolved top-down after the lanes finish.  Each wavefront
// writes only its own column and reads only inner nodes.  The node's static
// data (open flag, bottom layer, incident elements in element order with
// their bottom layers and areas, the inner neighbours' bottom layers) comes
// from tables built at set-up, so a lane's loads depend on one another at
// most two deep.
constexpr int kBndoLanes = 64;
constexpr int kBndoNb = 6;          // inner neighbours of a node loaded at once

template <typename S>
struct BndoArgs {
    int nbndo, nkn, nel;
    const int *bk, *open, *lmax, *eptr, *el, *elev, *bptr, *bnb, *nblev;
    const double *eaj;
    const S *bnx, *bny, *bw, *uln, *vln;
    const int *iweg;
    S *cv[2];               // the tracers of the launch (grid row 0 and 1)
    const S *rbc[2];        // their boundary values (may be null)
    int *err;
    const int *mem_istot, *node_mem;
    int isact;
    // the outflow test's normal velocity scal per node and layer
    // ([i * nlvdi + l - 1]): computed and kept by the first substep of a
    // step (the velocities and the wet/dry mask hold for the whole step),
    // read by the others; null: computed by every call
    S *scal;
    int nlvdi;
};

template <typename S>
__global__ __launch_bounds__(kBndoLanes) void k_bndo(BndoArgs<S> a) {
    using R = S;
    __shared__ R val[kBndoLanes];
    __shared__ int status[kBndoLanes];
    const int i = blockIdx.x;
    if (i >= a.nbndo) return;
    // the node's static data in one round of loads
    const int open = a.open[i], k = a.bk[i], lmax = a.lmax[i];
    if (!open) return;
    if (a.mem_istot && a.isact > a.mem_istot[a.node_mem[k]]) return;
    S *const cv = a.cv[blockIdx.y];
    const S *const rbc = a.rbc[blockIdx.y];
    const int lane = threadIdx.x, l = lane + 1;
    const int nkn = a.nkn, nel = a.nel;
    const R flag = (R)-999.;
    status[lane] = 0;
    if (l <= lmax) {
        const size_t o = (size_t)(l - 1) * nkn + k;
        R cur = cv[o];
        if (rbc) {
            const R rb = rbc[o];
            if (rb != flag) cur = rb;
        }
        R scal;
        if (a.scal && a.isact > 1) {
            scal = a.scal[(size_t)i * a.nlvdi + l - 1];
        } else {
            R vv = 0, up = 0, vp = 0;
            for (int q = a.eptr[i]; q < a.eptr[i + 1]; q++) {
                const int ie = a.el[q];
                if (a.iweg[ie] != 0 || l > a.elev[q]) continue;
                const R aj = (R)a.eaj[q];
                vv = vv + aj;
                up = up + aj * a.uln[(size_t)(l - 1) * nel + ie];
                vp = vp + aj * a.vln[(size_t)(l - 1) * nel + ie];
            }
            R u = up, v = vp;
            if (vv > (R)0) { u = u / vv; v = v / vv; }
            scal = a.bnx[i] * u + a.bny[i] * v;
            if (a.scal && blockIdx.y == 0) a.scal[(size_t)i * a.nlvdi + l - 1] = scal;
        }
        const bool binside = scal <= (R)0 || cur == flag;
        R bc = 0, tw = 0;
        int ntbc = 0;
        if (binside) {
            // the first kBndoNb inner neighbours' entries loaded at once, then
            // their values, then added in list order; more one by one
            const int j0 = a.bptr[i], nj = a.bptr[i + 1] - j0;
            int nlev[kBndoNb], nbk[kBndoNb];
            R w[kBndoNb], cvn[kBndoNb];
#pragma unroll
            for (int s = 0; s < kBndoNb; s++) {
                nlev[s] = 0; nbk[s] = 0; w[s] = 0;
                if (s < nj) { nlev[s] = a.nblev[j0 + s]; nbk[s] = a.bnb[j0 + s]; w[s] = a.bw[j0 + s]; }
            }
#pragma unroll
            for (int s = 0; s < kBndoNb; s++) {
                cvn[s] = 0;
                if (s < nj && l <= nlev[s]) cvn[s] = cv[(size_t)(l - 1) * nkn + nbk[s]];
            }
#pragma unroll
            for (int s = 0; s < kBndoNb; s++)
                if (s < nj && l <= nlev[s]) {
                    ntbc++;
                    tw = tw + w[s];
                    bc = bc + w[s] * cvn[s];
                }
            for (int j = j0 + kBndoNb; j < j0 + nj; j++) {
                if (l <= a.nblev[j]) {
                    ntbc++;
                    tw = tw + a.bw[j];
                    bc = bc + a.bw[j] * cv[(size_t)(l - 1) * nkn + a.bnb[j]];
                }
            }
        } else {
            ntbc = a.bptr[i + 1] - a.bptr[i];
            tw = 1;
            bc = cur;
        }
        if (ntbc > 0) { val[lane] = bc / tw; status[lane] = 1; }
        else status[lane] = l > 1 ? 2 : 3;
    }
    __syncthreads();
    if (lane == 0) {
        for (int m = 1; m < lmax && m < kBndoLanes; m++)
            if (status[m] == 2) val[m] = val[m - 1];
        if (status[0] == 3) atomicCAS(a.err, 0, ERR_CONZ);
    }
    __syncthreads();
    if (l <= lmax && status[0] != 3) cv[(size_t)(l - 1) * nkn + k] = val[lane];
}

template <typename S>
static BndoArgs<S> bndo_args(Model &M, const TracerSet &ts, int isact, void *scal);

template <typename S>
static int bndo_t(Model &M, const TracerSet &ts, hipStream_t st, int isact, void *scal) {
    if (M.m.nbndo == 0) return 0;
    if (M.nlv > kBndoLanes) return hip_check(M, hipErrorInvalidValue, "bndo: more layers than lanes");
    const BndoArgs<S> a = bndo_args<S>(M, ts, isact, scal);
    hipLaunchKernelGGL(k_bndo<S>, dim3(M.m.nbndo, ts.n), dim3(kBndoLanes), 0, st, a);
    HIPCHK(M, hipGetLastError());
    return 0;
}

// (zeroed first, like conz_args)
template <typename S>
static BndoArgs<S> bndo_args(Model &M, const TracerSet &ts, int isact, void *scal) {
    BndoArgs<S> a;
    std::memset(&a, 0, sizeof a);
    a.nbndo = M.m.nbndo; a.nkn = M.nkn; a.nel = M.nel;
    a.bk = M.m.bndo_k; a.open = M.m.bndo_open; a.lmax = M.m.bndo_lmax; a.eptr = M.m.bndo_eptr; a.el = M.m.bndo_el;
    a.elev = M.m.bndo_elev; a.bptr = M.m.bndo_ptr; a.bnb = M.m.bndo_nb; a.nblev = M.m.bndo_nblev;
    a.eaj = M.m.bndo_eaj;
    a.bnx = (const S *)M.m.bndo_nx; a.bny = (const S *)M.m.bndo_ny; a.bw = (const S *)M.m.bndo_w;
    a.uln = (const S *)M.s.uln; a.vln = (const S *)M.s.vln;
    a.iweg = M.iweg_conz ? M.iweg_conz : M.s.iweg;
    for (int t = 0; t < 2; t++) {
        const int itr = ts.itr[t < ts.n ? t : 0];
        a.cv[t] = (S *)M.s.tracer[itr];
        a.rbc[t] = (const S *)M.s.tracer_bc[itr];
    }
    a.err = M.d_err;
    if (M.mem_istot_on) { a.mem_istot = M.cur_mem_istot; a.node_mem = M.d_node_mem; }
    a.isact = isact;
    a.scal = (S *)scal;
    a.nlvdi = M.nlvdi;
    return a;
}

int launch_bndo(Model &M, const TracerSet &ts, hipStream_t st, int isact, void *scal) {
    return M.prec == SHYHIP_FP64 ? bndo_t<double>(M, ts, st, isact, scal) : bndo_t<float>(M, ts, st, isact, scal);
}

int launch_bndo(Model &M, int itr, hipStream_t st, int isact) {
    TracerSet ts;
    ts.n = 1;
    ts.itr[0] = itr;
    return launch_bndo(M, ts, st, isact, nullptr);
}

int launch_conz3d(Model &M, const TracerSet &ts, int istot, int isact, hipStream_t st, void *hbuf, void *rec,
                  bool prep) {
    if (ts.n == 2)
        return M.prec == SHYHIP_FP64 ? conz_t<double, 2>(M, ts, istot, isact, st, hbuf, rec, prep)
                                     : conz_t<float, 2>(M, ts, istot, isact, st, hbuf, rec, prep);
    return M.prec == SHYHIP_FP64 ? conz_t<double, 1>(M, ts, istot, isact, st, hbuf, rec, prep)
                                 : conz_t<float, 1>(M, ts, istot, isact, st, hbuf, rec, prep);
}

void conz3d_key(Model &M, const TracerSet &ts, int istot, void *hbuf, void *rec, void *bscal, std::string &key) {
    key_add(key, istot);
    key_add(key, M.nl_tmpl);
    key_add(key, M.prec);
    key_add(key, ts.n);
    key_add(key, M.m.nbndo);
    key_add(key, M.m.n_ntile);
    if (M.prec == SHYHIP_FP64) {
        key_add(key, conz_args<double>(M, ts, istot, 1, hbuf, rec));
        key_add(key, bndo_args<double>(M, ts, 1, bscal));
    } else {
        key_add(key, conz_args<float>(M, ts, istot, 1, hbuf, rec));
        key_add(key, bndo_args<float>(M, ts, 1, bscal));
    }
}

int launch_conz3d(Model &M, int itr, int istot, int isact, int clip_small, hipStream_t st, void *hbuf, void *rec,
                  const void *cbound) {
    TracerSet ts;
    ts.n = 1;
    ts.itr[0] = itr;
    ts.clip[0] = clip_small;
    ts.cbound[0] = cbound;
    return launch_conz3d(M, ts, istot, isact, st, hbuf, rec, true);
}

// ------------------------------------------------------------------ stability
// scalar_stability (stability.f90:220-260): conzstab (concentration.f90:
// 1573-2097) for one second (one substep) with difmol = 0, no nudging and no
// sinking, then rindex = dt * (index / rstol) and istot = 1 + rindex.  One
// work-item per node-layer gathers its incident elements in element order --
// the order conzstab accumulates them -- with each element's advective term
// for this vertex (the larger of the last out- and in-flux seen over the
// element's vertices up to this one, as conzstab carries them), its explicit
// vertical diffusion and its share of the node volume; point sources add
// their inflow.  Horizontal diffusion (rkpar) is zero on the device path and
// adds nothing.  The node-layer ratios are non-negative, so their IEEE bit
// patterns order as unsigned integers; their maximum is taken across the
// wavefront and the workgroup first (exact in any order), and each workgroup
// then issues one atomic max per member it touches, none when the value
// already held is not smaller.

// maximum of v over the wavefront, in every lane
__device__ inline unsigned long long wave_max_u64(unsigned long long v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned lo = (unsigned)__shfl_xor((int)(unsigned)v, off);
        const unsigned hi = (unsigned)__shfl_xor((int)(unsigned)(v >> 32), off);
        const unsigned long long o = ((unsigned long long)hi << 32) | lo;
        v = o > v ? o : v;
    }
    return v;
}

// atomic max that skips the atomic when the value held is already at least v
// (a stale read is never larger than the value held, so skipping is exact)
__device__ inline void max_into(unsigned long long *p, unsigned long long v) {
    if (v == 0ull) return;
    const unsigned long long cur = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (v > cur) atomicMax(p, v);
}

// the ratio of one node-layer (l, k) as the bits of a non-negative double,
// 0 when it adds nothing.  The incident elements are taken in element order
// kStabBatch at a time: each batch's loads are issued together (the list
// entries, then every element's data and its vertices, then the vertices'
// vertical velocities), and the batch is then added in order.
//
// What bounds it: the gathers, so only what a term uses is read: the vertices
// before this one (the node's own velocities are loaded once), and the layer
// thicknesses only where the diffusion has an explicit part.  With all of
// them, three elements at a time and two wavefronts to a SIMD: 191 us on 300k
// nodes of 20 layers, 36.5 on 50k of 12 (FP64), 134 in FP32 on 285k of 10,
// against 137, 27 and 93.  Batches of one gain a little on 50k nodes and lose
// more on 300k and 3k of 6 layers (141, 26.5, 93; 15.8 against 13.5), batches
// of three lose everywhere (160, 31, 105; 13.7).
constexpr int kStabBatch = 2;

template <typename S>
__device__ inline unsigned long long stab_ratio(int l, int k, int nkn, int nel, int nlv, const int *ilhv,
                                                const int *nk_ptr, const int *nk_el, const int *nen3v,
                                                const double *geo, double az, double ad, double aa, const S *utn,
                                                const S *uto, const S *vtn, const S *vto, const S *wln,
                                                const S *difv, const S *hdeo, const S *hdkn, const S *hdko,
                                                const S *mflux, float rkpar, const S *difhv, const S *wdif,
                                                float robs, const S *rtauv, float wsink, const S *wsinkv) {
    const double azt = 1. - az, adt = 1. - ad, aat = 1. - aa;
    double chigh = 0., cn = 0., cdiag = 0., clow = 0.;
    double co = 0.;
    if (mflux) {
        const S q = mflux[(size_t)(l - 1) * nkn + k];
        if (q > (S)0) co = (double)q;
    }
    // the node's own data (the layer below exists for elements deeper than l)
    const double dtop = l > 1 ? (double)difv[(size_t)(l - 1) * nkn + k] : 0.;
    const double dbot = l < nlv ? (double)difv[(size_t)l * nkn + k] : 0.;
    const double hn = (double)hdkn[(size_t)(l - 1) * nkn + k], ho = (double)hdko[(size_t)(l - 1) * nkn + k];
    const double rtau = rtauv ? (double)rtauv[(size_t)(l - 1) * nkn + k] : 0.;
    // the vertical velocity at the top (at = l - 1) and bottom (at = l) of
    // node kk's layer, less the tracer's sinking in the tracers' precision
    auto wvel = [&](int at, int kk) {
        const size_t o = (size_t)at * nkn + kk;
        return wsinkv ? (double)(S)(wln[o] - (S)wsink * wsinkv[o]) : (double)wln[o];
    };
    const double wtk = l > 1 ? wvel(l - 1, k) : 0., wbk = l < nlv ? wvel(l, k) : 0.;
    const int p0 = nk_ptr[k], p1 = nk_ptr[k + 1];
    for (int pb = p0; pb < p1; pb += kStabBatch) {
        int ie[kStabBatch], iv[kStabBatch], ilev[kStabBatch], kj[kStabBatch][2];
        double aj4[kStabBatch], us[kStabBatch], vs[kStabBatch], hdv[kStabBatch], hdt[kStabBatch], hdb[kStabBatch];
        double gb[kStabBatch][3], gc[kStabBatch][3], wt[kStabBatch][2], wb[kStabBatch][2];
        double rk3[kStabBatch], wd[kStabBatch];
#pragma unroll
        for (int b = 0; b < kStabBatch; b++) {
            const int e = nk_el[min(pb + b, p1 - 1)];
            ie[b] = e >> 2;
            iv[b] = e & 3;
        }
#pragma unroll
        for (int b = 0; b < kStabBatch; b++) {
            const int el = ie[b];
            const size_t le = (size_t)(l - 1) * nel + el;
            ilev[b] = ilhv[el];
            aj4[b] = 4. * geo[(size_t)6 * nel + el];
            us[b] = az * (double)utn[le] + azt * (double)uto[le];
            vs[b] = az * (double)vtn[le] + azt * (double)vto[le];
            hdv[b] = hdt[b] = hdb[b] = 1.;
            if (adt != 0.) {
                hdv[b] = (double)hdeo[le];
                hdt[b] = l > 1 ? (double)hdeo[le - nel] : 0.;
                hdb[b] = l < nlv ? (double)hdeo[le + nel] : 0.;
            }
            rk3[b] = 0.;
            wd[b] = 0.;
            if (wdif) {
                // horizontal diffusion: 3 rkpar difhv in the tracers'
                // precision and the vertex's own weight wdifhv(ii, ii)
                rk3[b] = (double)((S)3 * (S)rkpar * difhv[le]);
                wd[b] = (double)wdif[(size_t)(4 * iv[b]) * nel + el];
            }
#pragma unroll
            for (int jj = 0; jj < 3; jj++) {
                gb[b][jj] = gc[b][jj] = 0.;
                if (jj <= iv[b]) {
                    gb[b][jj] = geo[(size_t)jj * nel + el];
                    gc[b][jj] = geo[(size_t)(3 + jj) * nel + el];
                }
                if (jj < 2) {
                    kj[b][jj] = k;
                    if (jj < iv[b]) kj[b][jj] = nen3v[3 * el + jj];
                }
            }
        }
        // (the vertices before this one; the node itself has its own)
#pragma unroll
        for (int b = 0; b < kStabBatch; b++)
#pragma unroll
            for (int jj = 0; jj < 2; jj++) {
                wt[b][jj] = wtk;
                wb[b][jj] = wbk;
                if (jj < iv[b]) {
                    if (l > 1) wt[b][jj] = wvel(l - 1, kj[b][jj]);
                    if (l < nlv) wb[b][jj] = wvel(l, kj[b][jj]);
                }
            }
#pragma unroll
        for (int b = 0; b < kStabBatch; b++) {
            if (pb + b >= p1 || l > ilev[b]) continue;
            const bool below = l < ilev[b];
            double coadv = 0., ciadv = 0., cadv = 0.;
#pragma unroll
            for (int jj = 0; jj < 3; jj++) {
                if (jj > iv[b]) break;
                const double f = us[b] * gb[b][jj] + vs[b] * gc[b][jj];
                double fwin = 0., fwout = 0.;
                const double w_t = jj < 2 ? wt[b][jj < 2 ? jj : 0] : wtk;
                const double w_b = below ? (jj < 2 ? wb[b][jj < 2 ? jj : 0] : wbk) : 0.;
                if (w_t > 0.) fwout = fwout + aat * w_t;
                else fwin = fwin - aat * w_t;
                if (w_b > 0.) fwin = fwin + aat * w_b;
                else fwout = fwout - aat * w_b;
                const double chadv = aj4[b] * 3. * f;
                const double cviadv = aj4[b] * fwin, cvoadv = aj4[b] * fwout;
                if (chadv < 0.) coadv = cvoadv - chadv;
                else ciadv = cviadv + chadv;
                cadv = coadv > ciadv ? coadv : ciadv;
            }
            chigh = chigh + cadv;
            if (adt != 0.) {
                double hmtop = 0., hmbot = 0.;
                if (l > 1) hmtop = 2. * dtop / (hdt[b] + hdv[b]);
                if (below) hmbot = 2. * dbot / (hdv[b] + hdb[b]);
                cn = cn + aj4[b] * (adt * (hmtop + hmbot));
            }
            clow = clow + aj4[b] * rk3[b] * ho * wd[b];
            if (rtauv) co = co + aj4[b] * ho * (double)robs * rtau;      // nudging
            cdiag = cdiag + aj4[b] * (ho < hn ? ho : hn);
        }
    }
    if (cdiag > 0.) {
        const double r = ((chigh + clow) + cn + co) / cdiag;
        if (r > 0.) return (unsigned long long)__double_as_longlong(r);
    }
    return 0ull;
}

// One work-item per entry of the node-layer list.
template <typename S>
__global__ void __launch_bounds__(kThreads) k_conz_stab(int nkn, int nel, int nlv, int n_nitem, const int *nitem,
                                                        const int *ilhv, const int *zbound, const int *nk_ptr,
                                                        const int *nk_el, const int *nen3v, const double *geo,
                                                        double az, double ad, double aa, const S *utn, const S *uto,
                                                        const S *vtn, const S *vto, const S *wln, const S *difv,
                                                        const S *hdeo, const S *hdkn, const S *hdko, const S *mflux,
                                                        float rkpar, const S *difhv, const S *wdif, float robs,
                                                        const S *rtauv, float wsink, const S *wsinkv,
                                                        const int *node_mem, unsigned long long *dmax) {
    const int i = xcd_block() * blockDim.x + threadIdx.x;
    unsigned long long val = 0ull;    // this node-layer's ratio as bits (0: none)
    int key = 0;                      // its member
    if (i < n_nitem) {
        const unsigned w = (unsigned)nitem[i];
        const int k = (int)(w >> 5), l = (int)(w & 31u) + 1;
        if (node_mem) key = node_mem[k];
        if (!zbound[k]) val = stab_ratio(l, k, nkn, nel, nlv, ilhv, nk_ptr, nk_el, nen3v, geo, az, ad, aa, utn, uto,
                                         vtn, vto, wln, difv, hdeo, hdkn, hdko, mflux, rkpar, difhv, wdif, robs,
                                         rtauv, wsink, wsinkv);
    }
    // the wavefront's maximum when its node-layers belong to one member
    // (always, for a single model); lanes of mixed waves go one by one
    __shared__ unsigned long long wval[kThreads / 64];
    __shared__ int wkey[kThreads / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int key0 = __shfl(key, 0);
    if (__all(key == key0)) {
        val = wave_max_u64(val);
        if (lane == 0) { wval[wv] = val; wkey[wv] = key0; }
    } else {
        max_into(dmax + key, val);
        if (lane == 0) { wval[wv] = 0ull; wkey[wv] = key0; }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        // one atomic per distinct member of the workgroup's waves
        for (int w = 0; w < kThreads / 64; w++) {
            if (wval[w] == 0ull) continue;
            unsigned long long m = wval[w];
            for (int q = w + 1; q < kThreads / 64; q++)
                if (wkey[q] == wkey[w] && wval[q] != 0ull) {
                    m = wval[q] > m ? wval[q] : m;
                    wval[q] = 0ull;
                }
            max_into(dmax + wkey[w], m);
        }
    }
}

// the index of each member rounded through a default real (the reference's
// shympi_max of a real), rindex = dt * index / rstol in the model's real,
// istot = 1 + rindex truncated.  w holds nmem maxima, then nmem istot and
// nmem rindex bits (as double); istot also goes to mem_istot (may be null);
// the maxima are cleared for the next call.  One work-item per member of one
// workgroup; the results also go to the host's pinned memory (host: nmem
// istot, nmem rindex), with the number of this report (hseq) behind them.
constexpr int kStabFinal = 256;

template <typename S>
__global__ __launch_bounds__(kStabFinal) void k_conz_stab_final(unsigned long long *w, int nmem, S dt, float rstol,
                                                                int *mem_istot, unsigned long long *host, int *hseq,
                                                                int seq) {
    for (int m = threadIdx.x; m < nmem; m += kStabFinal) {
        double stabind = __longlong_as_double((long long)w[m]);
        stabind = (double)(float)stabind;
        const S sindex = (S)(stabind / (double)rstol);
        const S ri = dt * sindex;
        const int ist = (int)((S)1 + ri);
        w[nmem + m] = (unsigned long long)(long long)ist;
        w[2 * nmem + m] = (unsigned long long)__double_as_longlong((double)ri);
        host[m] = (unsigned long long)(long long)ist;
        host[nmem + m] = (unsigned long long)__double_as_longlong((double)ri);
        if (mem_istot) mem_istot[m] = ist;
        w[m] = 0ull;
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(hseq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// per member (nmem = 1: the model): istot[m] and rindex[m] on the host
template <typename S>
static int stab_t(Model &M, float rstol, int *istot, double *rindex) {
    if (M.p.rkpar > 0.f && !M.m.wdif) return hip_check(M, hipErrorNotInitialized, "scalar_stability: no diffusion weights");
    // the nudging and sinking of the tracer being transported, if any
    const int t = M.terms_tracer;
    float robs = 0.f, wsink = 0.f;
    const void *rtauv = nullptr, *wsinkv = nullptr;
    if (t >= 0 && t < M.ntr) {
        if (M.tr_robs[t] != 0.f && M.s.cobs[t] && M.s.rtauv[t]) { robs = M.tr_robs[t]; rtauv = M.s.rtauv[t]; }
        if (M.tr_wsink[t] != 0.f && M.s.wsinkv[t]) { wsink = M.tr_wsink[t]; wsinkv = M.s.wsinkv[t]; }
    }
    const int nmem = M.nmem_dev > 1 ? M.nmem_dev : 1;
    unsigned long long *w = nmem > 1 ? M.d_mem_stab : (unsigned long long *)(M.d_err + 8);
    const int n = M.m.n_nitem;
    hipLaunchKernelGGL(k_conz_stab<S>, dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, M.stream, M.nkn,
                       M.nel, M.nlv, n, M.m.conz_nitem, M.m.ilhv, M.m.zbound, M.m.nk_ptr, M.m.nk_el, M.m.nen3v, M.m.geo,
                       (double)M.p.azpar, (double)M.p.adpar, (double)M.p.aapar, (const S *)M.s.utn,
                       (const S *)M.s.uto, (const S *)M.s.vtn, (const S *)M.s.vto, (const S *)M.s.wln,
                       (const S *)M.s.difv, (const S *)M.s.hdeo, (const S *)M.s.hdkn, (const S *)M.s.hdko,
                       M.has_mflux ? (const S *)M.s.mflux : (const S *)nullptr, M.p.rkpar,
                       (const S *)M.s.difhv, M.p.rkpar > 0.f ? (const S *)M.m.wdif : (const S *)nullptr,
                       robs, (const S *)rtauv, wsink, (const S *)wsinkv, nmem > 1 ? M.d_node_mem : nullptr, w);
    HIPCHK(M, hipGetLastError());
    unsigned long long *hbuf = nmem > 1 ? M.h_mem_stab : (unsigned long long *)(M.h_pinned + HP_STAB);
    const int seq = ++M.report_seq;
    hipLaunchKernelGGL(k_conz_stab_final<S>, dim3(1), dim3(kStabFinal), 0, M.stream, w, nmem, (S)M.p.dt, rstol,
                       nmem > 1 ? M.cur_mem_istot : nullptr, hbuf, M.h_pinned + HP_SEQ_STAB, seq);
    HIPCHK(M, hipGetLastError());
    if (wait_report(M, HP_SEQ_STAB, seq)) return 1;
    for (int m = 0; m < nmem; m++) {
        istot[m] = (int)(long long)hbuf[m];
        std::memcpy(&rindex[m], &hbuf[nmem + m], sizeof(double));
    }
    return 0;
}

int launch_scalar_stability(Model &M, float rstol, int *istot, double *rindex) {
    return M.prec == SHYHIP_FP64 ? stab_t<double>(M, rstol, istot, rindex) : stab_t<float>(M, rstol, istot, rindex);
}

}  // namespace shy
