// Discrete adjoint of the DG hydro step (gfx950, FP64): the reverse of the stage RHS with respect
// to the state, the per-node Manning n and the per-node depth DP, plus the gauge-misfit loss.
//
// The reference has no adjoint; this differentiates the operations of its explicit step as this
// library evaluates them (OCEAN/LAND/FLOW/INTERNAL_EDGE_HYDRO with the LLF flux
// src/numerical_flux.F:750-1022, RHS_DG_HYDRO src/rhs_dg_hydro.F:18-473, the SSP-RK update
// src/DG_hydro_timestep.F:238-290).  Non-smooth operations take the branch the forward values
// select: the LLF wave-speed bound differentiates through the largest of its six candidates, the
// Manning friction floor CF and the 0.9/DT friction cap pass no derivative when active, and
// Eirik's dry-ocean-edge fix differentiates |h|.  SLOPELIMITER5 is differentiated with its active
// set frozen (limiter_adj_kernel and the node passes after it).  WETDRY after the limiter is
// differentiated with its branches frozen too (wetdry_adj_element, run by the limiter kernel's
// adjoint variant on the limited values it forms again): the wet/dry flags at the start
// of each stage come from the forward run, a dry element's RHS is zero, and an edge with a dry
// side takes the reverse of the dry-side flux case the forward values select (dry_side_adj).
// Without the limiter WETDRY is differentiated only where it is the identity (every element wet
// and staying wet): the forward sweeps flag any element WETDRY changes, and the gradient call then
// fails.
//
// Kernel layout follows the forward's small-mesh stage kernel: four waves per 64 elements, gathers only.  The
// cotangent of an internal edge flux is the sum of what both neighbours' RHS cotangents ask of it;
// each element forms that sum from its own and its neighbour's cotangents and keeps the part of
// the flux derivative that belongs to its own trace, so no scatter or atomics are needed.
#include "dg_device.hpp"

namespace dg {

// Reverse of llf_flux: given fb = d(loss)/d(f0,f1,f2), returns the cotangents of
// (ze_in, ze_ex, qx_in, qx_ex, qy_in, qy_ex, hb_in, hb_ex) in bar[0..7].  NL: the nonlinear
// equations (NLEQ = 1, LEQ = 0) with the vanishing terms left out.
template <bool NL>
__device__ __forceinline__ void llf_flux_adj(const Phys& P, double zi, double ze, double xi, double xe,
                                             double yi, double ye, double hi, double he, double sfi,
                                             double sfe, double nx, double ny, double G,
                                             const double fb[3], double bar[8]) {
    // derivatives need not round like the forward step: let products and sums fuse
#pragma clang fp contract(fast)
    const double NLEQ = NL ? 1.0 : P.nleq, LEQ = NL ? 0.0 : P.leq, FG_L = NL ? 0.0 : P.fg_l;
    const double NLEQG = G * NLEQ;
    // ---- forward values needed by the reverse sweep
    const double j1 = ze - zi, j2 = xe - xi, j3 = ye - yi;
    const double side_z[2] = {zi, ze}, side_x[2] = {xi, xe}, side_y[2] = {yi, ye}, side_h[2] = {hi, he};
    const double side_s[2] = {sfi, sfe};
    double ht[2], fh[2], u[2], v[2], un[2], c[2], K[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        ht[s] = side_z[s] * NLEQ + side_h[s];
        fh[s] = NL ? 1.0 / ht[s] : 1.0 / (NLEQ * ht[s] + LEQ);
        u[s] = side_x[s] * fh[s];
        v[s] = side_y[s] * fh[s];
        un[s] = (u[s] * nx + v[s] * ny) * NLEQ;
        const double nxs = nx * side_s[s];
        K[s] = ny * ny + nxs * nxs;
        c[s] = sqrt(G * ht[s] * K[s]);
    }
    // largest wave-speed candidate, in the forward's comparison order
    const double cand[6] = {fabs(un[0] + c[0]), fabs(un[0]), fabs(un[0] - c[0]),
                            fabs(un[1] + c[1]), fabs(un[1]), fabs(un[1] - c[1])};
    int arg = 0;
    double em = cand[0];
#pragma unroll
    for (int q = 1; q < 6; q++)
        if (cand[q] > em) { em = cand[q]; arg = q; }
    // ---- reverse
    const double a1b = fb[0], a2b = fb[1], a3b = fb[2];
    double emb, j1b, j2b, j3b;
    if constexpr (NL) {
        emb = -0.5 * (j1 * fb[0] + j2 * fb[1] + j3 * fb[2]);
        j1b = -0.5 * em * fb[0];
        j2b = -0.5 * em * fb[1];
        j3b = -0.5 * em * fb[2];
    } else {
        const double nx2 = NLEQ + LEQ * nx * nx, ny2 = NLEQ + LEQ * ny * ny, nxy = nx * ny;
        emb = -0.5 * j1 * fb[0] - 0.5 * (j2 * nx2 + LEQ * j3 * nxy) * fb[1] -
              0.5 * (j3 * ny2 + LEQ * j2 * nxy) * fb[2];
        j1b = -0.5 * em * fb[0];
        j2b = -0.5 * em * (nx2 * fb[1] + LEQ * nxy * fb[2]);
        j3b = -0.5 * em * (LEQ * nxy * fb[1] + ny2 * fb[2]);
    }
    double unb[2] = {0.0, 0.0}, cb[2] = {0.0, 0.0};
    {
        const int s = arg / 3, q = arg % 3;
        const double val = q == 0 ? un[s] + c[s] : (q == 1 ? un[s] : un[s] - c[s]);
        const double sg = val > 0.0 ? 1.0 : (val < 0.0 ? -1.0 : 0.0);
        unb[s] += sg * emb;
        if (q == 0) cb[s] += sg * emb;
        else if (q == 2) cb[s] -= sg * emb;
    }
    // flux averages: a = 0.5*((f_in + f_ex).n)
    const double fx1b = 0.5 * nx * a1b, fy1b = 0.5 * ny * a1b;
    const double fx2b = 0.5 * nx * a2b, fy2b = 0.5 * ny * a2b;
    const double fx3b = 0.5 * nx * a3b, fy3b = 0.5 * ny * a3b;
    double zb[2], xb[2], yb[2], hbb[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const double z = side_z[s], x = side_x[s], y = side_y[s], h = side_h[s], sf = side_s[s];
        const double fnl = NL ? 1.0 : NLEQ + LEQ * h;
        const double fu = NLEQ * x, fv = NLEQ * y, fg = NLEQG * z;
        double zbar = 0.0, xbar = 0.0, ybar = 0.0, hbar = 0.0;
        // fy3 = hvv + gh2; fx3 = huv*sf; fy2 = huv; fx2 = (huu + gh2)*sf
        const double hvvb = fy3b;
        double gh2b = fy3b + sf * fx2b;
        const double huvb = sf * fx3b + fy2b;
        const double huub = sf * fx2b;
        // gh2 = fg*(0.5*z + h) + FG_L*z
        double fgb = (0.5 * z + h) * gh2b;
        zbar += (NL ? 0.5 * fg : 0.5 * fg + FG_L) * gh2b;
        hbar += fg * gh2b;
        // huu = fu*u, hvv = fv*v, huv = fu*v
        double fub = u[s] * huub + v[s] * huvb;
        double ub = fu * huub;
        const double fvb = v[s] * hvvb;
        double vb = fv * hvvb + fu * huvb;
        // un = (u*nx + v*ny)*NLEQ
        ub += nx * NLEQ * unb[s];
        vb += ny * NLEQ * unb[s];
        // c = sqrt(G*ht*K): dc/dht = G*K/(2c) = c/(2*ht), and fh = 1/ht for the nonlinear equations
        double htb;
        if constexpr (NL) htb = c[s] > 0.0 ? 0.5 * c[s] * fh[s] * cb[s] : 0.0;
        else htb = c[s] > 0.0 ? G * K[s] / (2.0 * c[s]) * cb[s] : 0.0;
        // u = x*fh, v = y*fh
        xbar += fh[s] * ub;
        ybar += fh[s] * vb;
        const double fhb = x * ub + y * vb;
        // fh = 1/(NLEQ*ht + LEQ)
        htb += -NLEQ * fh[s] * fh[s] * fhb;
        // fg = NLEQG*z, fu = NLEQ*x, fv = NLEQ*y
        zbar += NLEQG * fgb;
        xbar += NLEQ * fub;
        ybar += NLEQ * fvb;
        // fx1 = x*fnl*sf, fy1 = y*fnl
        xbar += fnl * sf * fx1b;
        ybar += fnl * fy1b;
        if constexpr (!NL) hbar += LEQ * (x * sf * fx1b + y * fy1b);
        // ht = z*NLEQ + h
        zbar += NLEQ * htb;
        hbar += htb;
        zb[s] = zbar; xb[s] = xbar; yb[s] = ybar; hbb[s] = hbar;
    }
    // jumps
    bar[0] = zb[0] - j1b;
    bar[1] = zb[1] + j1b;
    bar[2] = xb[0] - j2b;
    bar[3] = xb[1] + j2b;
    bar[4] = yb[0] - j3b;
    bar[5] = yb[1] + j3b;
    bar[6] = hbb[0];
    bar[7] = hbb[1];
}

// The part of llf_flux_adj that one side of an internal edge keeps: the cotangents of side `own`'s
// arguments (ze, qx, qy, hb) only.  Both elements of an edge run it for their own side, with the
// same canonical (in, ex) argument order, so no lane evaluates the other side's reverse.
template <bool NL>
__device__ __forceinline__ void llf_flux_adj_side(const Phys& P, double zi, double ze, double xi, double xe,
                                                  double yi, double ye, double hi, double he, double sfi,
                                                  double sfe, double nx, double ny, double G,
                                                  const double fb[3], int own, double& zbar,
                                                  double& xbar, double& ybar, double& hbar) {
#pragma clang fp contract(fast)
    const double NLEQ = NL ? 1.0 : P.nleq, LEQ = NL ? 0.0 : P.leq, FG_L = NL ? 0.0 : P.fg_l;
    const double NLEQG = G * NLEQ;
    const double j1 = ze - zi, j2 = xe - xi, j3 = ye - yi;
    // forward values of both sides (the wave-speed bound needs both)
    const double side_z[2] = {zi, ze}, side_x[2] = {xi, xe}, side_y[2] = {yi, ye}, side_h[2] = {hi, he};
    const double side_s[2] = {sfi, sfe};
    double fh[2], u[2], v[2], un[2], c[2], K[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const double ht = side_z[q] * NLEQ + side_h[q];
        fh[q] = NL ? 1.0 / ht : 1.0 / (NLEQ * ht + LEQ);
        u[q] = side_x[q] * fh[q];
        v[q] = side_y[q] * fh[q];
        un[q] = (u[q] * nx + v[q] * ny) * NLEQ;
        const double nxs = nx * side_s[q];
        K[q] = ny * ny + nxs * nxs;
        c[q] = sqrt(G * ht * K[q]);
    }
    const double cand[6] = {fabs(un[0] + c[0]), fabs(un[0]), fabs(un[0] - c[0]),
                            fabs(un[1] + c[1]), fabs(un[1]), fabs(un[1] - c[1])};
    int arg = 0;
    double em = cand[0];
#pragma unroll
    for (int q = 1; q < 6; q++)
        if (cand[q] > em) { em = cand[q]; arg = q; }
    double emb, j1b, j2b, j3b;
    if constexpr (NL) {
        emb = -0.5 * (j1 * fb[0] + j2 * fb[1] + j3 * fb[2]);
        j1b = -0.5 * em * fb[0];
        j2b = -0.5 * em * fb[1];
        j3b = -0.5 * em * fb[2];
    } else {
        const double nx2 = NLEQ + LEQ * nx * nx, ny2 = NLEQ + LEQ * ny * ny, nxy = nx * ny;
        emb = -0.5 * j1 * fb[0] - 0.5 * (j2 * nx2 + LEQ * j3 * nxy) * fb[1] -
              0.5 * (j3 * ny2 + LEQ * j2 * nxy) * fb[2];
        j1b = -0.5 * em * fb[0];
        j2b = -0.5 * em * (nx2 * fb[1] + LEQ * nxy * fb[2]);
        j3b = -0.5 * em * (LEQ * nxy * fb[1] + ny2 * fb[2]);
    }
    // this side's forward values
    const double z = own ? ze : zi, x = own ? xe : xi, y = own ? ye : yi, h = own ? he : hi;
    const double sf = own ? sfe : sfi;
    const double fhs = own ? fh[1] : fh[0], us = own ? u[1] : u[0], vs = own ? v[1] : v[0];
    const double cs = own ? c[1] : c[0], Ks = own ? K[1] : K[0];
    double unb = 0.0, cb = 0.0;
    if (arg / 3 == own) {
        const int q = arg % 3;
        const double uns = own ? un[1] : un[0];
        const double val = q == 0 ? uns + cs : (q == 1 ? uns : uns - cs);
        const double sg = val > 0.0 ? 1.0 : (val < 0.0 ? -1.0 : 0.0);
        unb = sg * emb;
        if (q == 0) cb = sg * emb;
        else if (q == 2) cb = -sg * emb;
    }
    const double fx1b = 0.5 * nx * fb[0], fy1b = 0.5 * ny * fb[0];
    const double fx2b = 0.5 * nx * fb[1], fy2b = 0.5 * ny * fb[1];
    const double fx3b = 0.5 * nx * fb[2], fy3b = 0.5 * ny * fb[2];
    const double fnl = NL ? 1.0 : NLEQ + LEQ * h;
    const double fu = NLEQ * x, fv = NLEQ * y, fg = NLEQG * z;
    double zb = 0.0, xb = 0.0, yb = 0.0, hb = 0.0;
    const double hvvb = fy3b;
    const double gh2b = fy3b + sf * fx2b;
    const double huvb = sf * fx3b + fy2b;
    const double huub = sf * fx2b;
    const double fgb = (0.5 * z + h) * gh2b;
    zb += (NL ? 0.5 * fg : 0.5 * fg + FG_L) * gh2b;
    hb += fg * gh2b;
    const double fub = us * huub + vs * huvb;
    double ub = fu * huub;
    const double fvb = vs * hvvb;
    double vb = fv * hvvb + fu * huvb;
    ub += nx * NLEQ * unb;
    vb += ny * NLEQ * unb;
    double htb;
    if constexpr (NL) htb = cs > 0.0 ? 0.5 * cs * fhs * cb : 0.0;
    else htb = cs > 0.0 ? G * Ks / (2.0 * cs) * cb : 0.0;
    xb += fhs * ub;
    yb += fhs * vb;
    const double fhb = x * ub + y * vb;
    htb += -NLEQ * fhs * fhs * fhb;
    zb += NLEQG * fgb;
    xb += NLEQ * fub;
    yb += NLEQ * fvb;
    xb += fnl * sf * fx1b;
    yb += fnl * fy1b;
    if constexpr (!NL) hb += LEQ * (x * sf * fx1b + y * fy1b);
    zb += NLEQ * htb;
    hb += htb;
    zbar = own ? zb + j1b : zb - j1b;
    xbar = own ? xb + j2b : xb - j2b;
    ybar = own ? yb + j3b : yb - j3b;
    hbar = hb;
}

// The P1 bathymetry modes from the vertex depths as the forward stage kernel stages them (no contraction).
__device__ __forceinline__ void hb_modes(double d0, double d1, double d2, double hb[3]) {
    const double c13 = 1.0 / 3.0, c16 = 1.0 / 6.0;
    hb[0] = c13 * (d0 + d1 + d2);
    hb[1] = -(c16 * (d0 + d1)) + c13 * d2;
    hb[2] = -(0.5 * d0) + 0.5 * d1;
}

// Reverse of an internal edge point where one side is dry (src/internal_edge_hydro.F:212-302),
// for this element's own side; i and x are the "in" and "ex" traces (elevation, discharges, bathymetry) as the
// forward forms them, so that the case is taken from the forward's mass flux; cin/cex are d(loss)/d(flux the
// "in"/"ex" side received).  Cases:
// 1 reflect into a dry "in" (both sides take the reflected flux's F0, "ex" its momentum: a function
// of the "ex" traces only), 2 zero-gravity momentum for a dry "in", 3 reflect into a dry "ex",
// 4 zero-gravity momentum for a dry "ex", 0 the plain flux.  Outputs this side's trace cotangents.
template <bool NL>
__device__ __forceinline__ int dry_side_case(const Phys& ph, int wd_in_el, int wd_ex_el, const double (&i)[4],
                                             const double (&x)[4], double sfi, double sfx, double nx, double ny) {
    double f0, f1, f2;
    llf<NL>(ph, i[0], x[0], i[1], x[1], i[2], x[2], i[3], x[3], sfi, sfx, nx, ny, ph.g, f0, f1, f2);
    if (!(fabs(f0) > 1.0e-8)) return 0;
    if (wd_in_el == 0) return f0 > 0.0 ? 1 : 2;
    if (wd_ex_el == 0) return f0 < 0.0 ? 3 : 4;
    return 0;
}

template <bool NL>
__device__ __forceinline__ void dry_side_adj(const Phys& ph, int cas, int role, const double (&i)[4], const double (&x)[4],
                                             double sfi, double sfx, double nx, double ny, const double (&cin)[3],
                                             const double (&cex)[3], double& zb, double& xb, double& yb, double& hbar) {
#pragma clang fp contract(fast)
    const double zi = i[0], xi = i[1], yi = i[2], hi = i[3], ze = x[0], xe = x[1], ye = x[2], he = x[3];
    zb = xb = yb = hbar = 0.0;
    if (cas == 0 || cas == 2 || cas == 4) {
        // the flux, and for cases 2 and 4 the zero-gravity momentum flux that replaces one side's
#pragma unroll 1
        for (int k = 0; k < (cas == 0 ? 1 : 2); k++) {
            double fb[3] = {cin[0] + cex[0], cin[1] + cex[1], cin[2] + cex[2]};
            if (cas != 0) {
                const bool in = (cas == 2) == (k == 1);
                fb[0] = k == 0 ? fb[0] : 0.0;
                fb[1] = in ? cin[1] : cex[1];
                fb[2] = in ? cin[2] : cex[2];
            }
            double z2, x2, y2, h2;
            llf_flux_adj_side<NL>(ph, zi, ze, xi, xe, yi, ye, hi, he, sfi, sfx, nx, ny, k == 0 ? ph.g : 0.0, fb, role, z2, x2,
                                  y2, h2);
            zb += z2; xb += x2; yb += y2; hbar += h2;
        }
        return;
    }
    // reflection: the flux is a function of one side's traces only (the "ex" side in case 1, the
    // "in" side in case 3); the other side keeps nothing
    const int src = cas == 1 ? 1 : 0;
    if (role != src) return;
    const double tx = -ny, ty = nx, den = nx * ty - ny * tx;
    const double sx = src ? xe : xi, sy = src ? ye : yi;
    const double qn = sx * nx + sy * ny, qt = sx * tx + sy * ty;
    const double mqx = (ty * -qn - ny * qt) / den, mqy = (-tx * -qn + nx * qt) / den;
    // d(mqx, mqy)/d(sx, sy)
    const double mxx = (-ty * nx - ny * tx) / den, mxy = (-ty * ny - ny * ty) / den;
    const double myx = (tx * nx + nx * tx) / den, myy = (tx * ny + nx * ty) / den;
    double bar[8];
    if (src) {
        const double fbr[3] = {cin[0] + cex[0], cex[1], cex[2]};
        llf_flux_adj<NL>(ph, ze, ze, mqx, xe, mqy, ye, he, he, sfx, sfx, nx, ny, ph.g, fbr, bar);
        zb = bar[0] + bar[1];
        hbar = bar[6] + bar[7];
        xb = bar[3] + mxx * bar[2] + myx * bar[4];
        yb = bar[5] + mxy * bar[2] + myy * bar[4];
    } else {
        const double fbr[3] = {cin[0] + cex[0], cin[1], cin[2]};
        llf_flux_adj<NL>(ph, zi, zi, xi, mqx, yi, mqy, hi, hi, sfi, sfi, nx, ny, ph.g, fbr, bar);
        zb = bar[0] + bar[1];
        hbar = bar[6] + bar[7];
        xb = bar[2] + mxx * bar[3] + myx * bar[5];
        yb = bar[4] + mxy * bar[3] + myy * bar[5];
    }
}

// Cotangent seed of the gauge misfit sum_g w (eta_g - d_g)^2 after a step.  ord lists the gauges grouped by element
// (ascending gauge index within a group, group u at ord[off[u]..off[u+1])), so gauges sharing an element add up
// in gauge order.
struct GaugeSeed {
    const int* __restrict__ idx;         // [ne] group of each element, or -1; nullptr: no seed
    const int* __restrict__ off;
    const int* __restrict__ ord;
    const double* __restrict__ phi;      // [ng][dof]
    const double* __restrict__ eta;      // the step's gauge elevations and data [ng]
    const double* __restrict__ data;
    double w;
};

template <int DOF>
__device__ __forceinline__ void add_gauge_seed(const GaugeSeed& s, int u, double (&t)[DOF]) {
    for (int j = s.off[u]; j < s.off[u + 1]; j++) {
        const int g = s.ord[j];
        const double r = 2.0 * s.w * (s.eta[g] - s.data[g]);
#pragma unroll
        for (int k = 0; k < DOF; k++) t[k] += r * s.phi[(size_t)g * DOF + k];
    }
}

struct AdjArgs {
    ElemData ed;
    Phys ph;
    Forcing fo;
    Met mt;                              // NWS=8 node forcing of the step (when met != 0)
    int met;
    const double* __restrict__ u;        // stage state U(IRK) [3][dof][ne]
    int irk;                             // stage index
    int nsrc;                            // later-stage cotangents entering this stage
    const double* src[KMAXRK];           // cotangent of U(I'+1), I' >= IRK
    double acoef[KMAXRK];                // ATVD(I',IRK)
    double bcoef[KMAXRK];                // BTVD(I',IRK) (times the scenario's DT in the kernel)
    double* __restrict__ out;            // cotangent of U(IRK)
    double* __restrict__ gdp;            // [3][ne] accumulated cotangent of the vertex depths
    double* __restrict__ gnbar;          // [ne] accumulated cotangent of the element mean Manning n
    const uint8_t* __restrict__ wd;      // WDFLG during the stage, or nullptr (every element wet)
    // block-local staging, as in the forward stage kernel: tile t stages its elements and its halo
    // hidx[t*nh..t*nh+nh) (-1 past the tile's last); snbl packs each side's local neighbour index
    // (10 bits each)
    const int* __restrict__ hidx;
    const int* __restrict__ snbl;
    int nh, ns;                          // halo entries per tile, staged elements per block (LDS row length)
    GaugeSeed seed;                      // of the step before (a step's first stage: out is that step's cotangent)
};

// The reverse of the LLF flux of an internal edge point for one side's own arguments: `o` the side's own traces
// (elevation, discharges, bathymetry), `n` the neighbour's, fs the flux cotangent with the sign of (neighbour - own),
// (mx, my) half the canonical normal with that sign.  The wave-speed bound is the first largest of the candidates
// in the canonical order ("in" side first, so `in` decides a tie between the sides); bo and bn, -1 for the "ex" side
// and NaN for the "in" side, make a NaN first candidate count on the "in" side only, as comparing one candidate
// after the other does.
template <bool NL>
__device__ __forceinline__ void llf_adj_own(const Phys& P, const double (&o)[4], const double (&n)[4], double so, double sn,
                                            double nx, double ny, double mx, double my, const double (&fs)[3], bool in,
                                            double bo, double bn, double (&bar)[4]) {
#pragma clang fp contract(fast)
    const double NLEQ = NL ? 1.0 : P.nleq, LEQ = NL ? 0.0 : P.leq, FG_L = NL ? 0.0 : P.fg_l;
    const double NLEQG = P.g * NLEQ;
    const double z = o[0], x = o[1], y = o[2], h = o[3];
    double un, c, K, fh, u, v, m, un_n, c_n, m_n;
    int q;                               // the own side's candidate: 0 un + c, 1 un, 2 un - c
    {
        const double ht = z * NLEQ + h;
        fh = NL ? 1.0 / ht : 1.0 / (NLEQ * ht + LEQ);
        u = x * fh;
        v = y * fh;
        un = (u * nx + v * ny) * NLEQ;
        const double nxs = nx * so;
        K = ny * ny + nxs * nxs;
        c = sqrt(P.g * ht * K);
        m = fmax(fabs(un + c), bo);
        q = 0;
        if (fabs(un) > m) { m = fabs(un); q = 1; }
        if (fabs(un - c) > m) { m = fabs(un - c); q = 2; }
    }
    {
        const double ht = n[0] * NLEQ + n[3];
        const double f = NL ? 1.0 / ht : 1.0 / (NLEQ * ht + LEQ);
        un_n = (n[1] * f * nx + n[2] * f * ny) * NLEQ;
        const double nxs = nx * sn;
        c_n = sqrt(P.g * ht * (ny * ny + nxs * nxs));
        m_n = fmax(fabs(un_n + c_n), bn);
        if (fabs(un_n) > m_n) m_n = fabs(un_n);
        if (fabs(un_n - c_n) > m_n) m_n = fabs(un_n - c_n);
    }
    const bool mine = in ? !(m_n > m) : m > m_n;
    const double em = mine ? m : m_n;
    const double j1 = n[0] - z, j2 = n[1] - x, j3 = n[2] - y;
    double emb, d1, d2, d3;              // cotangents of the bound and of the jumps (own minus neighbour)
    if constexpr (NL) {
        emb = -0.5 * (j1 * fs[0] + j2 * fs[1] + j3 * fs[2]);
        d1 = 0.5 * em * fs[0];
        d2 = 0.5 * em * fs[1];
        d3 = 0.5 * em * fs[2];
    } else {
        const double nx2 = NLEQ + LEQ * nx * nx, ny2 = NLEQ + LEQ * ny * ny, nxy = nx * ny;
        emb = -0.5 * j1 * fs[0] - 0.5 * (j2 * nx2 + LEQ * j3 * nxy) * fs[1] - 0.5 * (j3 * ny2 + LEQ * j2 * nxy) * fs[2];
        d1 = 0.5 * em * fs[0];
        d2 = 0.5 * em * (nx2 * fs[1] + LEQ * nxy * fs[2]);
        d3 = 0.5 * em * (LEQ * nxy * fs[1] + ny2 * fs[2]);
    }
    double unb = 0.0, cb = 0.0;
    if (mine) {
        const double val = q == 0 ? un + c : (q == 1 ? un : un - c);
        unb = val > 0.0 ? emb : (val < 0.0 ? -emb : 0.0);
        cb = q == 0 ? unb : (q == 2 ? -unb : 0.0);
    }
    const double fx1b = mx * fs[0], fy1b = my * fs[0];
    const double hvvb = my * fs[2];
    const double huub = so * (mx * fs[1]);
    const double gh2b = hvvb + huub;
    const double huvb = so * (mx * fs[2]) + my * fs[1];
    const double fnl = NL ? 1.0 : NLEQ + LEQ * h;
    const double fu = NLEQ * x, fv = NLEQ * y, fg = NLEQG * z;
    const double ub = fu * huub + nx * NLEQ * unb;
    const double vb = fv * hvvb + fu * huvb + ny * NLEQ * unb;
    double htb;
    if constexpr (NL) htb = c > 0.0 ? 0.5 * c * fh * cb : 0.0;
    else htb = c > 0.0 ? P.g * K / (2.0 * c) * cb : 0.0;
    htb += -NLEQ * fh * fh * (x * ub + y * vb);
    bar[0] = (NL ? 0.5 * fg : 0.5 * fg + FG_L) * gh2b + NLEQG * ((0.5 * z + h) * gh2b) + NLEQ * htb + d1;
    bar[1] = fh * ub + NLEQ * (u * huub + v * huvb) + fnl * so * fx1b + d2;
    bar[2] = fh * vb + NLEQ * (v * hvvb) + fnl * fy1b + d3;
    bar[3] = fg * gh2b + htb;
    if constexpr (!NL) bar[3] += LEQ * (x * so * fx1b + y * fy1b);
}

// Rows of the staged tile: state, bathymetry modes, scaled RHS cotangent of the modes, AREAS; and what a wave
// leaves for the sums: the cotangents of the modes, of the bathymetry modes and of Manning's n.
constexpr int ADJ_NT = 64;               // elements per block
constexpr int adj_stage_rows(int dof) { return 6 * dof + 4; }
constexpr int adj_sum_rows(int dof) { return 3 * dof + 4; }

// Reverse of one stage.  A block of four waves works on 64 elements, lane l of every wave on element l.  Wave c < 3
//   1. stages the state and the RHS cotangent of field c of the tile and its halo (wave 3: bathymetry, AREAS,
//      flags and the edge table),
//   2. reverses side slot c,
//   3. reverses its share of the area points (wave 3 without a side has more of them),
//   4. adds what the four waves have for field c and the later stages' cotangents (wave 3: the parameters).
// The time of this kernel was its serial chain: one lane per element took three sides and the area points one after
// the other with two waves per SIMD (p=1) or one (p=2: 504 registers), the sums read and written in LDS at every
// point.  49,800 p=1 elements: 27.2 us before, 15.8 us now; four p=2 storm basins of 99,000 elements with their
// flags 108.7 and 65 us.  Three waves per SIMD where the registers allow (168: a 40-step gradient of 59,600 p=2
// elements 5.69 ms with two, 5.43 ms with three; of four p=1 storms 6.14 and 5.75 ms); the p=2 form with flags would spill
// (85 us) and runs with two, like the forms with the hybrid friction factor.
// A step's first stage adds the misfit of the step before to the cotangent that it writes: as a launch of its own that
// took 4.3 us a step.
// The RHS cotangent is staged times M_INV, which leaves the plain basis values and derivatives as the
// transposed quadrature's tables: the edge cotangent is a trace like the state's, and the area points' ones
// are two sums per field.
// QF: quadratic bottom friction without the hybrid factor (NOLIBF=1), fixed at compile time.
// WD: the stage's wet/dry flags are read (a.wd) and dry elements and dry-side edge cases are
// reversed; without it every element is wet and that code is compiled out (it would otherwise
// raise the kernel's register use past what the all-wet runs need).
template <int P, bool SPH, bool NL, bool QF, bool WD>
__global__ void __launch_bounds__(4 * ADJ_NT) __attribute__((amdgpu_waves_per_eu(QF && !(P == 2 && WD) ? 3 : 2))) adj_stage_kernel(AdjArgs a) {
#pragma clang fp contract(fast)
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    constexpr int NAGP = (P == 1) ? 3 : 6;
    constexpr int NEGP = P + 2;
    constexpr int NC = P + 1;
    constexpr int NT = ADJ_NT, RL = 3 * DOF, SR = adj_sum_rows(DOF);
    // (lane-divergent index) edge basis at the points, and the basis functions along the edge as polynomials
    // in the points' coordinate
    __shared__ double tpe[3][NEGP][DOF], tpc[3][NC][DOF];
    extern __shared__ double stg[];        // the staged rows (ns entries each), then the flags; last the waves' sums
    const DevTables& T = tab<P>();
    const ElemData& E = a.ed;
    const Phys& ph = a.ph;
    const int ne = E.ne, ns = a.ns, nh = a.nh;
    const int c = __builtin_amdgcn_readfirstlane(threadIdx.x / NT), le = threadIdx.x % NT;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int e = tile * NT + le;
    const bool valid = e < ne;
    const int ec = valid ? e : ne - 1;     // lanes past the last element read element ne-1 and write nothing
    uint8_t* const stwd = reinterpret_cast<uint8_t*>(stg + (size_t)adj_stage_rows(DOF) * ns);
    const int* hx = a.hidx + (size_t)tile * nh;
    const int sid = E.sid ? (int)E.sid[ec] : 0;
    const Scen& sc = E.scen[sid];
    {
        // two staged elements at a time: the tile's and the first halo's, then the halo's rest
        auto load = [&](int g, double (&v)[2 * DOF]) {
            if (c < 3) {
#pragma unroll
                for (int k = 0; k < DOF; k++) v[k] = at(a.u + (size_t)(c * DOF + k) * ne, g);
#pragma unroll
                for (int k = 0; k < DOF; k++) v[DOF + k] = 0.0;
                const double dtdp = E.scen[E.sid ? (int)at(E.sid, g) : 0].dtdp;
                for (int j = 0; j < a.nsrc; j++) {
                    if (a.bcoef[j] == 0.0) continue;
                    const double b = a.bcoef[j] * dtdp;
                    const double* s = a.src[j];
#pragma unroll
                    for (int k = 0; k < DOF; k++) v[DOF + k] += b * at(s + (size_t)(c * DOF + k) * ne, g);
                }
            } else {
#pragma unroll
                for (int m = 0; m < 3; m++) v[m] = at(E.dpv + (size_t)m * ne, g);
                const double X0 = at(E.xv, g), X1 = at(E.xv + ne, g), X2 = at(E.xv + 2 * (size_t)ne, g);
                const double Y0 = at(E.yv, g), Y1 = at(E.yv + ne, g), Y2 = at(E.yv + 2 * (size_t)ne, g);
                v[3] = (X0 - X2) * (Y1 - Y2) + (X2 - X1) * (Y0 - Y2);
                if (WD) v[4] = __hiloint2double(0, at(a.wd, g));
            }
        };
        auto store = [&](int j, const double (&v)[2 * DOF]) {
            if (c < 3) {
#pragma unroll
                for (int k = 0; k < DOF; k++) stg[(c * DOF + k) * ns + j] = v[k];
#pragma unroll
                for (int k = 0; k < DOF; k++) stg[(RL + 3 + c * DOF + k) * ns + j] = T.m_inv[k] * v[DOF + k];
            } else {
                double hb[3];
                hb_modes(v[0], v[1], v[2], hb);
#pragma unroll
                for (int m = 0; m < 3; m++) stg[(RL + m) * ns + j] = hb[m];
                stg[(2 * RL + 3) * ns + j] = v[3];
                if (WD) stwd[j] = (uint8_t)__double2loint(v[4]);
            }
        };
        const int g0 = le < nh ? hx[le] : -1;
        double v[2 * DOF], v2[2 * DOF];
        load(ec, v);
        load(g0 < 0 ? 0 : g0, v2);
        store(le, v);
        if (g0 >= 0) store(NT + le, v2);
#pragma unroll 1
        for (int h = le + NT; h < nh; h += NT) {
            const int g = hx[h];
            if (g < 0) break;
            load(g, v);
            store(NT + h, v);
        }
        if (c == 3)
            for (int j = le; j < 3 * NEGP * DOF; j += NT) {
                const int l = j / (NEGP * DOF), g = (j / DOF) % NEGP, k = j % DOF;
                tpe[l][g][k] = T.phi_edge[l][g][k];
            }
        if (c == 3 && le < 3 * DOF) {
            const int l = le / DOF, k = le % DOF;
            const double lo = T.phi_edge[l][0][k], hi = T.phi_edge[l][NEGP - 1][k];   // at -1 and 1
            if (P == 1) {
                tpc[l][0][k] = T.phi_edge[l][1][k];                                   // at 0
            } else {
                // even part: at 1 and at the inner points
                const double a = 0.5 * (hi + lo), b = 0.5 * (T.phi_edge[l][1][k] + T.phi_edge[l][2][k]);
                const double c2 = (a - b) / (1.0 - T.xegp[1] * T.xegp[1]);
                tpc[l][NC - 1][k] = c2;
                tpc[l][0][k] = a - c2;
            }
            tpc[l][1][k] = 0.5 * (hi - lo);
        }
    }
    __syncthreads();
    const int wd = WD ? (valid ? stwd[le] : 0) : (valid ? 1 : 0);
    double ubar[3][DOF], hbb[3] = {0.0, 0.0, 0.0}, nbarb = 0.0;
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) ubar[f][k] = 0.0;
    // ---- side slot c
    if (c < 3) {
        const int bits = side_bits(at(E.sinfo, ec), c);
        const int L = bits & 3, role = (bits >> 2) & 1, kind = (bits >> 3) & 3, nled = (bits >> 5) & 3;
        const double nx = at(E.geo + (size_t)(3 * c) * ne, ec), ny = at(E.geo + (size_t)(3 * c + 1) * ne, ec);
        const double edfac = at(E.geo + (size_t)(3 * c + 2) * ne, ec);
        // cotangents of the own traces' polynomials
        double tb[3][NC], hc[2] = {0.0, 0.0};
#pragma unroll
        for (int f = 0; f < 3; f++)
#pragma unroll
            for (int m = 0; m < NC; m++) tb[f][m] = 0.0;
        auto add = [&](double zb, double xb, double yb, double hbar, double s) {
            double p = 1.0;
#pragma unroll
            for (int m = 0; m < NC; m++) {
                tb[0][m] += zb * p;
                tb[1][m] += xb * p;
                tb[2][m] += yb * p;
                if (m < 2) hc[m] += hbar * p;
                p = p * s;
            }
        };
        // the traces of the staged element j's RHS cotangent at an edge point
        auto cotangent = [&](int j, const double* ph_, double (&t)[3]) {
#pragma unroll
            for (int f = 0; f < 3; f++) {
                t[f] = stg[(RL + 3 + f * DOF) * ns + j];
#pragma unroll
                for (int k = 1; k < DOF; k++) t[f] += stg[(RL + 3 + f * DOF + k) * ns + j] * ph_[k];
            }
        };
        if (kind == SIDE_INTERNAL) {
            const int ln = (at(a.snbl, ec) >> (10 * c)) & 1023;
            const int wdn = WD ? stwd[ln] : 1;
            // (the forward adds no flux between dry elements)
            const double edfac_n = edfac * (stg[(2 * RL + 3) * ns + le] / stg[(2 * RL + 3) * ns + ln]);
            if (valid && (!WD || (wd != 0 && wdn != 0))) {
                const double mx = role ? -0.5 * nx : 0.5 * nx, my = role ? -0.5 * ny : 0.5 * ny;
                const double nan = __builtin_nan("");
                const double bo = role ? -1.0 : nan, bn = role ? nan : -1.0;
                // the traces along the edge as polynomials in the own points' coordinate (the neighbour's runs the
                // other way), formed once per side from the modes: at p=2 30 numbers stay instead of 78, and
                // the tables of the points are the same for every lane
                auto along = [&](int row, int j, int l, double sign, int n, double (&t)[NC]) {
#pragma unroll
                    for (int m = 0; m < NC; m++) t[m] = 0.0;
#pragma unroll
                    for (int k = 0; k < DOF; k++) {
                        if (k >= n) break;
                        const double v = stg[(row + k) * ns + j];
#pragma unroll
                        for (int m = 0; m < NC; m++)
                            if (n == DOF || m < 2) t[m] += v * tpc[l][m][k];
                    }
                    t[1] = sign * t[1];
                };
                double to[4][NC], tn[4][NC], fc[3][NC];
#pragma unroll
                for (int f = 0; f < 4; f++) {
                    along(f * DOF, le, L, 1.0, f < 3 ? DOF : 3, to[f]);
                    along(f * DOF, ln, nled, -1.0, f < 3 ? DOF : 3, tn[f]);
                }
#pragma unroll
                for (int f = 0; f < 3; f++) {
                    double co[NC], cn[NC];
                    along(RL + 3 + f * DOF, le, L, 1.0, DOF, co);
                    along(RL + 3 + f * DOF, ln, nled, -1.0, DOF, cn);
#pragma unroll
                    for (int m = 0; m < NC; m++) fc[f][m] = 2.0 * (edfac_n * cn[m] - edfac * co[m]);
                }
                auto point = [&](const double (&t)[NC], double s, int n) {
                    double v = t[n - 1];
#pragma unroll
                    for (int m = NC - 2; m >= 0; m--)
                        if (m < n - 1) v = v * s + t[m];
                    return v;
                };
#pragma unroll 1
                for (int q = 0; q < NEGP; q++) {
                    const double s = T.xegp[q], w = T.wegp[q];
                    const double o[4] = {point(to[0], s, NC), point(to[1], s, NC), point(to[2], s, NC), point(to[3], s, 2)};
                    const double n[4] = {point(tn[0], s, NC), point(tn[1], s, NC), point(tn[2], s, NC), point(tn[3], s, 2)};
                    const double fq[3] = {w * point(fc[0], s, NC), w * point(fc[1], s, NC), w * point(fc[2], s, NC)};
                    double so = 1.0, sn = 1.0;
                    if (SPH) {
                        const int I = role ? NEGP - 1 - q : q;
                        so = E.sfs[(size_t)(c * NEGP + I) * ne + ec];
                        sn = E.sfs[(size_t)((3 + c) * NEGP + I) * ne + ec];
                    }
                    double bar[4];
                    llf_adj_own<NL>(ph, o, n, so, sn, nx, ny, mx, my, fq, role == 0, bo, bn, bar);
                    add(bar[0], bar[1], bar[2], bar[3], s);
                }
            }
            if constexpr (WD)
                if (valid && (wd != 0) != (wdn != 0)) {
#pragma unroll 1
                    for (int q = 0; q < NEGP; q++) {
                        const int gi = role ? NEGP - 1 - q : q;
                        const double* po = tpe[L][q];
                        const double* pn = tpe[nled][NEGP - 1 - q];
                        const int jo = reread(le), jn = reread(ln);
                        double to[4], tn[4], co[3], cn[3];
                        edge_point<DOF>(stg, ns, role ? jn : jo, role ? pn : po, to);   // the "in" side's
                        edge_point<DOF>(stg, ns, role ? jo : jn, role ? po : pn, tn);   // the "ex" side's
                        double so = 1.0, sn = 1.0;
                        if (SPH) {
                            so = E.sfs[(size_t)(c * NEGP + gi) * ne + ec];
                            sn = E.sfs[(size_t)((3 + c) * NEGP + gi) * ne + ec];
                        }
                        // flux cotangents: the "in" element's RHS took -w_in*F, the "ex" element's +w_ex*F
                        cotangent(jo, po, co);
                        cotangent(jn, pn, cn);
                        const double w = 2.0 * T.wegp[q];
                        double cin[3], cex[3];
#pragma unroll
                        for (int f = 0; f < 3; f++) {
                            cin[f] = role ? -(w * edfac_n * cn[f]) : -(w * edfac * co[f]);
                            cex[f] = role ? w * edfac * co[f] : w * edfac_n * cn[f];
                        }
                        const double sfi = role ? sn : so, sfx = role ? so : sn;
                        const int cas = dry_side_case<NL>(ph, role ? wdn : wd, role ? wd : wdn, to, tn, sfi, sfx, nx, ny);
                        double zb, xb, yb, hbar;
                        dry_side_adj<NL>(ph, cas, role, to, tn, sfi, sfx, nx, ny, cin, cex, zb, xb, yb, hbar);
                        add(zb, xb, yb, hbar, T.xegp[q]);
                    }
                }
        } else if (wd != 0) {                            // the forward skips a dry element's boundary edges
            const double tx = -ny, ty = nx;
            const int nb = at(E.snbr + (size_t)c * ne, ec);
#pragma unroll 1
            for (int I = 0; I < NEGP; I++) {
                const double* pv = tpe[L][I];
                const int jo = reread(le);
                double t[4], co[3];
                edge_point<DOF>(stg, ns, jo, pv, t);
                cotangent(jo, pv, co);
                const double ze_in = t[0], qx_in = t[1], qy_in = t[2], hb_in = t[3];
                const double sf = SPH ? E.sfs[(size_t)(c * NEGP + I) * ne + ec] : 1.0;
                // flux cotangent: RHS(K) -= w_K*F with w_K = 2 M_INV(K)/AREAS*XLEN*PHI*WEGP
                const double wq = -2.0 * T.wegp[I] * edfac;
                const double fb[3] = {wq * co[0], wq * co[1], wq * co[2]};
                double bar[8];
                double zb = 0.0, xb = 0.0, yb = 0.0, hbar = 0.0;
                if (kind == SIDE_LAND) {
                    const double qn_int = qx_in * nx + qy_in * ny, qt_int = qx_in * tx + qy_in * ty;
                    const double qn_ext = -qn_int, qt_ext = qt_int;
                    const double den = 1.0 / (nx * ty - ny * tx);
                    const double qx_ex = (ty * qn_ext - ny * qt_ext) * den;
                    const double qy_ex = (-tx * qn_ext + nx * qt_ext) * den;
                    llf_flux_adj<NL>(ph, ze_in, ze_in, qx_in, qx_ex, qy_in, qy_ex, hb_in, hb_in, sf, sf, nx, ny, ph.g, fb, bar);
                    zb = bar[0] + bar[1];
                    hbar = bar[6] + bar[7];
                    // mirror: (qx_ex, qy_ex) from (qx_in, qy_in)
                    const double qnb = (ty * bar[3] - tx * bar[5]) * den;
                    const double qtb = (-ny * bar[3] + nx * bar[5]) * den;
                    const double qnib = -qnb, qtib = qtb;
                    xb = bar[2] + nx * qnib + tx * qtib;
                    yb = bar[4] + ny * qnib + ty * qtib;
                } else if (kind == SIDE_OCEAN) {
                    double ze_ex = 0.0;
                    const double xe = T.xegp[I];
                    // the constituents' endpoint terms EMO*RFF*COS(ARGJ-EFA) of this stage (tide_kernel)
                    for (int jj = 0; jj < a.fo.nbfr; jj++) {
                        const size_t o = ((size_t)nb * a.fo.nbfr + jj) * 2;
                        const double z1 = a.fo.tz[(size_t)a.irk * a.fo.tzn + o];
                        const double z2 = a.fo.tz[(size_t)a.irk * a.fo.tzn + o + 1];
                        ze_ex = ze_ex + (0.5 * (z1 + z2) + 0.5 * (z2 - z1) * xe);
                    }
                    const bool eirik = (ze_ex * ph.ifnlfa + hb_in) <= 0;
                    if (eirik) ze_ex = fabs(hb_in) + sc.h0;
                    llf_flux_adj<NL>(ph, ze_in, ze_ex, qx_in, qx_in, qy_in, qy_in, hb_in, hb_in, sf, sf, nx, ny, ph.g, fb, bar);
                    zb = bar[0];
                    xb = bar[2] + bar[3];
                    yb = bar[4] + bar[5];
                    hbar = bar[6] + bar[7];
                    if (eirik) hbar += (hb_in > 0.0 ? 1.0 : (hb_in < 0.0 ? -1.0 : 0.0)) * bar[1];
                } else {
                    // the step's specified normal flux at this point (flow_kernel)
                    const double qn_ext = a.fo.fz[(size_t)a.irk * a.fo.fzn + (size_t)nb * NEGP + I];
                    const double qt_ext = 0.0;
                    const double qx_ex = -(ty * qn_ext - ny * qt_ext) / (nx * ty - ny * tx);
                    const double qy_ex = -(-tx * qn_ext + nx * qt_ext) / (nx * ty - ny * tx);
                    llf_flux_adj<NL>(ph, ze_in, ze_in, qx_in, qx_ex, qy_in, qy_ex, hb_in, hb_in, sf, sf, nx, ny, ph.g, fb, bar);
                    zb = bar[0] + bar[1];
                    xb = bar[2];
                    yb = bar[4];
                    hbar = bar[6] + bar[7];
                }
                add(zb, xb, yb, hbar, T.xegp[I]);
            }
        }
#pragma unroll
        for (int k = 0; k < DOF; k++)
#pragma unroll
            for (int m = 0; m < NC; m++) {
                const double t = tpc[L][m][k];
#pragma unroll
                for (int f = 0; f < 3; f++) ubar[f][k] += tb[f][m] * t;
                if (k < 3 && m < 2) hbb[k] += hc[m] * t;
            }
    }

    // ---- volume quadrature (wet elements only, as in the forward): points [i0, i1) of this wave
    const int i0 = P == 1 || c == 3 ? 0 : 3 + c, i1 = c == 3 ? 3 : (P == 1 ? 0 : 4 + c);
    if (i0 < i1 && wd != 0) {
        double hb[3];
#pragma unroll
        for (int m = 0; m < 3; m++) hb[m] = stg[(RL + m) * ns + le];
        const bool quad = QF || ph.iflinbf == 0;
        const bool hybrid = !QF && ph.ifhybf == 1;
        const double drdx = at(E.geo + (size_t)9 * ne, ec), dsdx = at(E.geo + (size_t)10 * ne, ec);
        const double drdy = at(E.geo + (size_t)11 * ne, ec), dsdy = at(E.geo + (size_t)12 * ne, ec);
        const double depth_c = hb[0] + stg[le];
        const double fh_nl_c = NL ? 1.0 / depth_c : 1.0 / (ph.nleq * depth_c + ph.leq);
        const double cori = E.cori_el ? at(E.cori_el, ec) : sc.cori;
        const double nbar = ph.load_manning ? at(E.nbar, ec) : 0.0;
        double depth_cb = 0.0;
        // the bathymetry's gradient (its modes are linear, so it is the same at every point) and its cotangent
        double dpx[3], dpy[3], dhbx = 0.0, dhby = 0.0, dhbxb = 0.0, dhbyb = 0.0;
#pragma unroll
        for (int k = 1; k < 3; k++) {
            dpx[k] = T.drphi[0][k] * drdx + T.dsphi[0][k] * dsdx;
            dpy[k] = T.drphi[0][k] * drdy + T.dsphi[0][k] * dsdy;
            dhbx = dhbx + hb[k] * dpx[k];
            dhby = dhby + hb[k] * dpy[k];
        }
        // NWS=8: the stage's vertex wind stresses and the pressure-gradient sums, as the forward
        // forms them; the pressure term -g*SFAC*H*dP/dx depends on the state through H
        double mw[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, pdx = 0.0, pdy = 0.0;
        if (a.met) {
            const double4* st = a.mt.st + (size_t)a.irk * a.mt.np;
            const double drpsi[3] = {-1.0 / 2.0, 1.0 / 2.0, 0.0}, dspsi[3] = {-1.0 / 2.0, 0.0, 1.0 / 2.0};
#pragma unroll
            for (int v = 0; v < 3; v++) {
                const int n = at(E.nm + (size_t)v * ne, ec);
                const double4 s = st[n];
                if constexpr (!NL) {
                    mw[v] = s.x;
                    mw[3 + v] = s.y;
                }
                const double pr = s.z;
                pdx += pr * (drpsi[v] * drdx + dspsi[v] * dsdx);
                pdy += pr * (drpsi[v] * drdy + dspsi[v] * dsdy);
            }
        }
#pragma unroll 1
        for (int I = i0; I < i1; I++) {
            const double* pa = T.phi_area[I];
            // read where it is used: held over the points the modes would set the kernel's register count
            const int jo = reread(le);
            auto value = [&](int row) {
                double t = stg[row * ns + jo];
#pragma unroll
                for (int k = 1; k < DOF; k++) t += stg[(row + k) * ns + jo] * pa[k];
                return t;
            };
            const double ze = value(0), qx = value(DOF), qy = value(2 * DOF);
            const double hbq = trace1<3>(hb, pa);
            const double sfq = SPH ? at(E.sfacq + (size_t)I * ne, ec) : 1.0;
            const double depth = ze + hbq;
            const double f1 = NL ? 1.0 : ph.nleq + ph.leq * hbq;
            const double fu = NL ? qx : ph.nleq * qx, fv = NL ? qy : ph.nleq * qy;
            const double fg = ph.nleqg * ze;
            const double fh = NL ? 1.0 / depth : 1.0 / (ph.nleq * depth + ph.leq);
            const double u = qx * fh, v = qy * fh;
            double fric = sc.fric;
            bool fric_active = false;
            double pw = 0.0;
            if (ph.load_manning) {
                pw = crm::cr_pow_third(depth);
                fric = ph.g * (nbar * nbar) / pw;
                if (fric < sc.cf) fric = sc.cf;
                else fric_active = true;
            }
            double tau = fric, umag = 0.0, hyb = 1.0, hyb_in = 0.0;
            bool capped = false;
            if (quad) {
                umag = sqrt(u * u + v * v);
                tau = tau * umag * fh;
                if (hybrid) {
                    hyb_in = 1.0 + pow(ph.hbreak * fh_nl_c, ph.ftheta);
                    hyb = pow(hyb_in, ph.fgamma / ph.ftheta);
                    tau = tau * hyb;
                }
                const double cap = 0.9 * sc.dtdph;
                if (cap < tau) { tau = cap; capped = true; }
            }
            // cotangents of the quadrature-point fluxes and sources from RHS(K): XFAC = M_INV*WAGP*dphi/dx and
            // SRFAC = M_INV*WAGP*PHI, with WAGP = 2*(M_INV(1)*WAGP)
            const double wagp = 2.0 * T.mw[I][0];
            double dr[3] = {0.0, 0.0, 0.0}, ds[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 1; k < DOF; k++) {
                const double r = wagp * T.drphi[I][k], s = wagp * T.dsphi[I][k];
#pragma unroll
                for (int f = 0; f < 3; f++) {
                    const double l = stg[(RL + 3 + f * DOF + k) * ns + jo];
                    dr[f] += r * l;
                    ds[f] += s * l;
                }
            }
            const double fxb = drdx * dr[0] + dsdx * ds[0], fyb = drdy * dr[0] + dsdy * ds[0];
            const double gxb = drdx * dr[1] + dsdx * ds[1], gyb = drdy * dr[1] + dsdy * ds[1];
            const double hxb = drdx * dr[2] + dsdx * ds[2], hyb_ = drdy * dr[2] + dsdy * ds[2];
            const double sxb = wagp * value(RL + 3 + DOF), syb = wagp * value(RL + 3 + 2 * DOF);
            double zeb = 0.0, qxb = 0.0, qyb = 0.0, hbqb = 0.0, depthb = 0.0;
            // sx = -(tau*qx) + fg*dhbx*sfq + cori*qy ; sy = -(tau*qy) + fg*dhby - cori*qx
            double taub = -qx * sxb - qy * syb;
            double f1b_met = 0.0;
            if (a.met) {
                // sx += wsx/F1 - g*SFAC*H*pdx ; sy += wsy/F1 - g*H*pdy (F1 = 1 for the nonlinear equations)
                depthb += -ph.g * sfq * pdx * sxb - ph.g * pdy * syb;
                if constexpr (!NL) {
                    const double* ps = T.psi[I];
                    const double wsx = mw[0] * ps[0] + mw[1] * ps[1] + mw[2] * ps[2];
                    const double wsy = mw[3] * ps[0] + mw[4] * ps[1] + mw[5] * ps[2];
                    const double fw = 1.0 / f1;
                    f1b_met = -fw * fw * (wsx * sxb + wsy * syb);
                }
            }
            qxb += -tau * sxb - cori * syb;
            qyb += cori * sxb - tau * syb;
            double fgb = dhbx * sfq * sxb + dhby * syb;
            dhbxb += fg * sfq * sxb;
            dhbyb += fg * syb;
            // friction
            double fricb = 0.0, ub = 0.0, vb = 0.0, fhb = 0.0;
            if (quad) {
                if (!capped) {
                    // tau = fric*umag*fh*hyb
                    fricb += umag * fh * hyb * taub;
                    const double umagb = fric * fh * hyb * taub;
                    fhb += fric * umag * hyb * taub;
                    if (hybrid) {
                        const double hybb = fric * umag * fh * taub;
                        // hyb = (1 + (hbreak*fh_nl_c)^ftheta)^(fgamma/ftheta)
                        const double dh_in = (ph.fgamma / ph.ftheta) * pow(hyb_in, ph.fgamma / ph.ftheta - 1.0);
                        const double x = ph.hbreak * fh_nl_c;
                        const double dx_ = x > 0.0 ? ph.ftheta * pow(x, ph.ftheta - 1.0) : 0.0;
                        const double fhcb = hybb * dh_in * dx_ * ph.hbreak;
                        depth_cb += -ph.nleq * fh_nl_c * fh_nl_c * fhcb;
                    }
                    if (umag > 0.0) {
                        const double r = umagb / umag;
                        ub += u * r; vb += v * r;
                    }
                }
            } else {
                fricb += taub;
            }
            if (ph.load_manning && fric_active) {
                // fric = g*nbar^2/depth^(1/3): d/dnbar = 2*fric/nbar, d/ddepth = -fric/(3*depth)
                const double gp = ph.g / pw;
                nbarb += 2.0 * gp * nbar * fricb;
                depthb += -(1.0 / 3.0) * gp * (nbar * nbar) * (NL ? fh : 1.0 / depth) * fricb;
            }
            // hy = hvv + gh2 ; hx = huv*sfq ; gy = huv ; gx = (huu + gh2)*sfq ; fx = qx*f1*sfq ; fy = qy*f1
            const double hvvb = hyb_;
            const double gh2b = hyb_ + sfq * gxb;
            const double huvb = sfq * hxb + gyb;
            const double huub = sfq * gxb;
            fgb += (0.5 * ze + hbq) * gh2b;
            zeb += (0.5 * fg + ph.fg_l) * gh2b;
            hbqb += fg * gh2b;
            const double fub = u * huub + v * huvb;
            ub += fu * huub;
            const double fvb = v * hvvb;
            vb += fv * hvvb + fu * huvb;
            qxb += fh * ub; qyb += fh * vb;
            fhb += qx * ub + qy * vb;
            depthb += -ph.nleq * fh * fh * fhb;
            zeb += ph.nleqg * fgb;
            qxb += ph.nleq * fub;
            qyb += ph.nleq * fvb;
            qxb += f1 * sfq * fxb;
            qyb += f1 * fyb;
            const double f1b = qx * sfq * fxb + qy * fyb + f1b_met;
            hbqb += ph.leq * f1b;
            zeb += depthb;
            hbqb += depthb;
            // traces
#pragma unroll
            for (int k = 0; k < DOF; k++) {
                ubar[0][k] += zeb * pa[k];
                ubar[1][k] += qxb * pa[k];
                ubar[2][k] += qyb * pa[k];
            }
#pragma unroll
            for (int k = 0; k < 3; k++) hbb[k] += hbqb * pa[k];
        }
#pragma unroll
        for (int k = 1; k < 3; k++) hbb[k] += dhbxb * dpx[k] + dhbyb * dpy[k];
        // depth_c = hb[0] + U[0][0]
        hbb[0] += depth_cb;
        ubar[0][0] += depth_cb;
    }
    // ---- the waves' sums; the staged rows are no longer needed
    __syncthreads();
    {
        double* const x = stg + (size_t)c * SR * NT + le;
#pragma unroll
        for (int f = 0; f < 3; f++)
#pragma unroll
            for (int k = 0; k < DOF; k++) x[(f * DOF + k) * NT] = ubar[f][k];
#pragma unroll
        for (int k = 0; k < 3; k++) x[(RL + k) * NT] = hbb[k];
        x[(RL + 3) * NT] = nbarb;
    }
    __syncthreads();
    if (!valid) return;
    auto sum = [&](int r) {
        const double* x = stg + (size_t)r * NT + le;
        return x[0] + x[SR * NT] + x[2 * SR * NT] + x[3 * SR * NT];
    };
    if (c < 3) {
        // cotangent of U(IRK): this stage's RHS reverse plus later stages' ATVD terms
        double s[DOF];
#pragma unroll
        for (int k = 0; k < DOF; k++) s[k] = sum(c * DOF + k);
        for (int j = 0; j < a.nsrc; j++) {
            const double ac = a.acoef[j];
            if (ac == 0.0) continue;
#pragma unroll
            for (int k = 0; k < DOF; k++) s[k] += ac * at(a.src[j] + (size_t)(c * DOF + k) * ne, e);
        }
        if (c == 0 && a.seed.idx) {
            const int u = at(a.seed.idx, e);
            if (u >= 0) add_gauge_seed<DOF>(a.seed, u, s);
        }
#pragma unroll
        for (int k = 0; k < DOF; k++) at(a.out + (size_t)(c * DOF + k) * ne, e) = s[k];
    } else {
        // parameters: element-mean Manning n and the vertex depths through the P1 bathymetry modes
        const double c13 = 1.0 / 3.0, c16 = 1.0 / 6.0;
        const double b0 = sum(RL), b1 = sum(RL + 1), b2 = sum(RL + 2);
        if (a.gnbar) a.gnbar[e] += sum(RL + 3);
        if (a.gdp) {
            a.gdp[e] += c13 * b0 - c16 * b1 - 0.5 * b2;
            a.gdp[(size_t)ne + e] += c13 * b0 - c16 * b1 + 0.5 * b2;
            a.gdp[2 * (size_t)ne + e] += c13 * b0 + c13 * b1;
        }
    }
}

// ------------------------------------------------------------------------------------------
// WETDRY (src/wetdry.F:58-548) of element e reversed with its branches frozen: from the state it
// was applied to (U: the limited stage output's modes 1-3, formed by limit_wide_kernel's adjoint
// variant), the vertex depths D and the element's flag before it, the element retakes the
// forward's decisions operation by operation (no contraction, so that they are the forward's) --
// which vertices are dry, the branch, the vertices' depth order, the two fmax(H0, .) choices, the
// vertices dry after the redistribution and the check -- and applies the transpose of the linear
// map that branch is.  ub (in place): cotangent of WETDRY's output -> of its input; gdp += the
// cotangents of the vertex depths.
// ------------------------------------------------------------------------------------------
template <int P>
__device__ void wetdry_adj_element(const DevTables& T, const double (&U)[3][3], const double (&D)[3], int wdflg,
                                   double H0, int e, int ne, double* __restrict__ ub, double* __restrict__ gdp) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    const double ZERO = 1.0e-6, C13 = 1.0 / 3.0, C16 = 1.0 / 6.0;
    const double dpe_min = fmin(fmin(D[0], D[1]), D[2]);
    // the forward's vertex values, in its operation order
    int ndry = 0, ht_max_i = 0;
    double ht_max = ZERO, ze_node[3], ht_node[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double z = U[0][0];
#pragma unroll
        for (int k = 1; k < 3; k++) z = z + T.phi_corner[i][k] * U[0][k];
        ze_node[i] = z;
        ht_node[i] = D[i] + z;
        if (ht_node[i] > ht_max) { ht_max_i = i; ht_max = ht_node[i]; }
        if (ht_node[i] <= (H0 + ZERO)) ndry++;
    }
    if (ndry == 0 && wdflg == 1) return;                       // identity
    const double dp_avg = C13 * (D[0] + D[1] + D[2]);
    double G[3][DOF];                                           // output cotangent
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) G[f][k] = ub[(size_t)(f * DOF + k) * ne + e];
    double I[3][DOF];                                           // input cotangent
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) I[f][k] = 0.0;
    double Db[3] = {0.0, 0.0, 0.0};
    if (ndry == 0) {
        // the check alone: the element keeps its values, its momentum too when the highest
        // vertex is wet enough
        const bool keep = ze_node[ht_max_i] > (-dpe_min + H0);
#pragma unroll
        for (int k = 0; k < DOF; k++) {
            I[0][k] = G[0][k];
            I[1][k] = keep ? G[1][k] : 0.0;
            I[2][k] = keep ? G[2][k] : 0.0;
        }
    } else {
        const double ht_avg = U[0][0] + dp_avg;
        if (ndry == 3 || ht_avg <= (H0 + ZERO)) {
            // flat: ZE = (ht_avg - dp_avg | ZERO - dp_avg, -HB2, -HB3), momentum zero
            if (ht_avg < ZERO) {
#pragma unroll
                for (int i = 0; i < 3; i++) Db[i] -= C13 * G[0][0];
            } else {
                I[0][0] = G[0][0];
            }
            // -HB2 = C16*(D1+D2) - C13*D3, -HB3 = 0.5*D1 - 0.5*D2
            Db[0] += C16 * G[0][1] + 0.5 * G[0][2];
            Db[1] += C16 * G[0][1] - 0.5 * G[0][2];
            Db[2] += -C13 * G[0][1];
        } else {
            // redistribution, as the forward orders the vertices and takes its branches
            int l2h[3] = {0, 1, 2};
#pragma unroll
            for (int k1 = 0; k1 < 3; k1++)
#pragma unroll
                for (int k2 = k1; k2 < 3; k2++)
                    if (ht_node[l2h[k1]] > ht_node[l2h[k2]]) { const int t = l2h[k1]; l2h[k1] = l2h[k2]; l2h[k2] = t; }
            double dh[3];
            const bool b0 = H0 > ht_node[l2h[0]];
            dh[l2h[0]] = fmax(H0, ht_node[l2h[0]]) - ht_node[l2h[0]];
            const bool b1 = H0 > ht_node[l2h[1]] - 0.5 * dh[l2h[0]];
            dh[l2h[1]] = fmax(H0, ht_node[l2h[1]] - 0.5 * dh[l2h[0]]) - ht_node[l2h[1]];
            dh[l2h[2]] = -dh[l2h[0]] - dh[l2h[1]];
            double ht_hat[3];
            int nd = 0, dry[3];
            ht_max = 0;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                ht_hat[i] = ht_node[i] + dh[i];
                if (ht_hat[i] > ht_max) { ht_max_i = i; ht_max = ht_hat[i]; }
                dry[i] = ht_hat[i] <= (H0 + 1.0e-10);
                nd += dry[i];
            }
            double ze_hat[3];
#pragma unroll
            for (int i = 0; i < 3; i++) ze_hat[i] = ht_hat[i] - D[i];
            const bool keep = ze_hat[ht_max_i] > (-dpe_min + H0);
            // momentum: QX(1..3) from the vertex values qxh, qxh = qxn + qxs at wet vertices,
            // qxs = (sum of the dry vertices' qxn)/(3 - nd); zero when nd = 3 or the check fails
            if (keep && nd < 3) {
#pragma unroll
                for (int f = 1; f < 3; f++) {
                    double hb_[3];
#pragma unroll
                    for (int i = 0; i < 3; i++)
                        hb_[i] = C13 * G[f][0] + (i < 2 ? -C16 : C13) * G[f][1] + (i == 0 ? -0.5 : (i == 1 ? 0.5 : 0.0)) * G[f][2];
                    double sb = 0.0, nb_[3];
#pragma unroll
                    for (int i = 0; i < 3; i++) { nb_[i] = dry[i] ? 0.0 : hb_[i]; if (!dry[i]) sb += hb_[i]; }
                    const double w = sb / (3.0 - (double)nd);
#pragma unroll
                    for (int i = 0; i < 3; i++) if (dry[i]) nb_[i] += w;
                    // qxn_i = QX1 + PHI(i,2)*QX2 + PHI(i,3)*QX3
#pragma unroll
                    for (int i = 0; i < 3; i++) {
                        I[f][0] += nb_[i];
                        I[f][1] += T.phi_corner[i][1] * nb_[i];
                        I[f][2] += T.phi_corner[i][2] * nb_[i];
                    }
                }
            }
            // elevation: ZE1 kept; ZE(2..3) from ze_hat = ht_hat - D = ze_node + dh
            I[0][0] += G[0][0];
            double zb[3], dhb[3], htb[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int i = 0; i < 3; i++) {
                zb[i] = (i < 2 ? -C16 : C13) * G[0][1] + (i == 0 ? -0.5 : (i == 1 ? 0.5 : 0.0)) * G[0][2];
                dhb[i] = zb[i];
            }
            // dh(l2) = -dh(l0) - dh(l1)
            dhb[l2h[0]] -= dhb[l2h[2]];
            dhb[l2h[1]] -= dhb[l2h[2]];
            // dh(l1) = H0 - ht(l1), or (ht(l1) - 0.5*dh(l0)) - ht(l1) = -0.5*dh(l0)
            if (b1) htb[l2h[1]] -= dhb[l2h[1]];
            else dhb[l2h[0]] += -0.5 * dhb[l2h[1]];
            // dh(l0) = H0 - ht(l0), or zero
            if (b0) htb[l2h[0]] -= dhb[l2h[0]];
            // ht = D + ze_node
#pragma unroll
            for (int i = 0; i < 3; i++) {
                Db[i] += htb[i];
                zb[i] += htb[i];
                I[0][0] += zb[i];
                I[0][1] += T.phi_corner[i][1] * zb[i];
                I[0][2] += T.phi_corner[i][2] * zb[i];
            }
        }
    }
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) ub[(size_t)(f * DOF + k) * ne + e] = I[f][k];
    gdp[e] += Db[0];
    gdp[(size_t)ne + e] += Db[1];
    gdp[2 * (size_t)ne + e] += Db[2];
}

// Elevation at the gauges: eta_g = sum_K ZE(K, elem_g) * phi_K(gauge), written to out[g]; blockIdx.y counts states
// `stride` apart.
template <int P>
__global__ void gauge_kernel(int ng, int ne, const int* __restrict__ gel, const double* __restrict__ gphi,
                             const double* __restrict__ u0, size_t stride, double* __restrict__ out) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const int e = gel[g];
    const double* u = u0 + blockIdx.y * stride;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < DOF; k++) s = s + u[(size_t)k * ne + e] * gphi[(size_t)g * DOF + k];
    out[(size_t)blockIdx.y * ng + g] = s;
}

// The seed alone, one thread per gauge element: of the last step, whose cotangent no stage writes.
template <int P>
__global__ void __launch_bounds__(64) gauge_seed_kernel(int nu, int ne, GaugeSeed s, const int* __restrict__ gel,
                                                        double* __restrict__ lam) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= nu) return;
    const int e = gel[s.ord[s.off[u]]];
    double t[DOF];
#pragma unroll
    for (int k = 0; k < DOF; k++) t[k] = lam[(size_t)k * ne + e];
    add_gauge_seed<DOF>(s, u, t);
#pragma unroll
    for (int k = 0; k < DOF; k++) lam[(size_t)k * ne + e] = t[k];
}

// Group of each gauge element (the others hold -1).
__global__ void __launch_bounds__(64) gauge_index_kernel(int nu, const int* __restrict__ off, const int* __restrict__ ord,
                                                         const int* __restrict__ gel, int* __restrict__ idx) {
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u < nu) idx[gel[ord[off[u]]]] = u;
}

// ------------------------------------------------------------------------------------------
// Reverse of SLOPELIMITER5 (src/slopelimiter.F:3434-3676) with its active set frozen: the
// forward limiter of each element is re-run on the stage's pre-limiter state W to record which
// branch every clamp, every redistribution test and every min(redfac, redmax) took; given those,
// the limiter is linear in (the element's linear modes, the node bounds) and its transpose maps
// the cotangent of the limited modes (in ub, in place) to the cotangent of W's modes, plus the
// cotangents of the vertex bounds (nbc: a record of six doubles [field][min|max] per element and
// vertex, record 3e+v, so that a node reads each incident element's six values from one place).
// Modes >= 3 pass through.
// A wave per field of 64 elements: with the three fields in one thread the launch was a serial chain
// with three divisions by three and nine by a count of one to three for each (now div3, a product with 0.5 or
// nothing, the same values).  99,000 elements: 15.7 us before, 12.0 us now; 800,000 73 and 60 us.  (With a record per field the
// node pass took 127 us at 800,000 elements instead of 75.)
// ------------------------------------------------------------------------------------------
constexpr int LADJ_NT = 64;              // elements per block
template <int P>
__global__ void __launch_bounds__(3 * LADJ_NT) limiter_adj_kernel(int np, ElemData E, const double* __restrict__ W,
                                                          const double* __restrict__ mm, double* __restrict__ ub,
                                                          double* __restrict__ nbc) {
    // no contraction: the recorded branches must be those of the forward limiter, operation by
    // operation
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    const DevTables& T = tab<P>();
    const int ne = E.ne;
    // the block's bound-cotangent records, written out together: its elements hold one contiguous range of them
    __shared__ double rec[LADJ_NT * 18];
    const int iv = __builtin_amdgcn_readfirstlane(threadIdx.x / LADJ_NT), le = threadIdx.x % LADJ_NT;
    const int e0 = blockIdx.x * LADJ_NT;
    const bool valid = e0 + le < ne;
    const int e = valid ? e0 + le : ne - 1;     // lanes past the last element read element ne-1 and write nothing
    // x over the number of positive differences (one to three): exactly x and x*0.5 for one and two
    auto by_count = [](double x, int n) { return n == 3 ? div3(x) : (n == 2 ? x * 0.5 : x); };
    const double* mn = mm + (size_t)(2 * iv) * np;
    const double* mx = mn + np;
    const double* w = W + (size_t)(iv * DOF) * ne;
    double* const b = ub + (size_t)(iv * DOF) * ne;
    double vmin[3], vmax[3], wb[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const int n = at(E.nm + (size_t)c * ne, e);
        vmin[c] = at(mn, n);
        vmax[c] = at(mx, n);
        wb[c] = at(b + (size_t)c * ne, e);
    }
    const double c0 = at(w, e), w1 = at(w + ne, e), w2 = at(w + 2 * (size_t)ne, e);
    // forward, recording the branches
    int sel[3];
    double v[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        double t = c0;
        t = t + T.phi_corner[c][1] * w1;
        t = t + T.phi_corner[c][2] * w2;
        double x = t;
        sel[c] = 0;
        if (!(t <= vmax[c])) { x = vmax[c]; sel[c] = 1; }
        if (x < vmin[c]) { x = vmin[c]; sel[c] = 2; }
        v[c] = x;
    }
    double sgs[3];
    int divs[3][3];
    int pos = 0, usemax = 0;
#pragma unroll
    for (int ll = 0; ll < 3; ll++) {
        const double sumloc = div3(v[0] + v[1] + v[2]);
        double sumdif = (sumloc - c0) * 3.0;
        const double sg = copysign(1.0, sumdif);
        sgs[ll] = sg;
        double dif[3];
#pragma unroll
        for (int c = 0; c < 3; c++) dif[c] = (v[c] - c0) * sg;
        int kdp = (dif[0] > 0) + (dif[1] > 0) + (dif[2] > 0);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            divs[ll][k] = kdp;
            double redfac = 0.0;
            if (dif[k] > 0) { redfac = by_count(sumdif * sg, kdp); kdp = kdp - 1; pos |= 1 << (3 * ll + k); }
            const double redmax = (sg > 0) ? v[k] - vmin[k] : vmax[k] - v[k];
            if (!(redfac <= redmax)) { redfac = redmax; usemax |= 1 << (3 * ll + k); }
            sumdif = sumdif - redfac * sg;
            v[k] = v[k] - redfac * sg;
        }
    }
    // reverse: U1 = -(v0+v1)/6 + v2/3, U2 = (v1-v0)/2, U0 = c0
    const double u1b = wb[1], u2b = wb[2];
    double vb[3] = {-(1.0 / 6.0) * u1b - 0.5 * u2b, -(1.0 / 6.0) * u1b + 0.5 * u2b, (1.0 / 3.0) * u1b};
    double c0b = wb[0];
    double vminb[3] = {0.0, 0.0, 0.0}, vmaxb[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int ll = 2; ll >= 0; ll--) {
        const double sg = sgs[ll];
        double sb = 0.0;
#pragma unroll
        for (int k = 2; k >= 0; k--) {
            // v_k -= redfac*sg; sumdif -= redfac*sg
            const double rb = -sg * vb[k] - sg * sb;
            if (usemax & (1 << (3 * ll + k))) {
                // redfac = redmax = sg > 0 ? v_k - vmin_k : vmax_k - v_k
                if (sg > 0) { vb[k] += rb; vminb[k] -= rb; }
                else { vmaxb[k] += rb; vb[k] -= rb; }
            } else if (pos & (1 << (3 * ll + k))) {
                sb += by_count(rb * sg, divs[ll][k]);   // redfac = sumdif*sg/div
            }
        }
        // sumdif = ((v0+v1+v2)/3 - c0)*3
        vb[0] += sb; vb[1] += sb; vb[2] += sb;
        c0b += -3.0 * sb;
    }
    double w1b = 0.0, w2b = 0.0;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        if (sel[c] == 0) {
            c0b += vb[c];
            w1b += T.phi_corner[c][1] * vb[c];
            w2b += T.phi_corner[c][2] * vb[c];
        } else if (sel[c] == 1) {
            vmaxb[c] += vb[c];
        } else {
            vminb[c] += vb[c];
        }
    }
    if (valid) {
        at(b, e) = c0b;
        at(b + ne, e) = w1b;
        at(b + 2 * (size_t)ne, e) = w2b;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            rec[le * 18 + c * 6 + iv * 2] = vminb[c];
            rec[le * 18 + c * 6 + iv * 2 + 1] = vmaxb[c];
        }
    }
    __syncthreads();
    const int n = min(LADJ_NT, ne - e0) * 18;
    double* dst = nbc + (size_t)e0 * 18;
    for (int k = threadIdx.x; k < n; k += 3 * LADJ_NT) dst[k] = rec[k];
}

// Per node: the sums of the incident elements' vertex-bound cotangents, and the element whose
// cell mean attains each bound (the first in the node's element list on ties; -1 when the
// +-99999 starting bound stands).  gsum, arg: a record [field][min|max] of six per node.  The three
// fields go through the node's list together: every incident element's cell means and its bound
// cotangent record (nbc) are loaded in one pass, and each field's sums still run in list order.
template <int P>
__global__ void __launch_bounds__(256) limiter_adj_node_kernel(int np, int ne, const int* __restrict__ off,
                                                               const int* __restrict__ n2e,
                                                               const double* __restrict__ W,
                                                               const double* __restrict__ nbc,
                                                               double* __restrict__ gsum, int* __restrict__ arg) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= np) return;
    double lo[3], hi[3], slo[3], shi[3];
    int alo[3], ahi[3];
#pragma unroll
    for (int f = 0; f < 3; f++) {
        lo[f] = 99999.; hi[f] = -99999.; slo[f] = 0.0; shi[f] = 0.0;
        alo[f] = -1; ahi[f] = -1;
    }
    const int j1 = off[n + 1];
    for (int j = off[n]; j < j1; j++) {
        const int ent = n2e[j];
        const int e = ent >> 2, v = ent & 3;
        const double2* rec = reinterpret_cast<const double2*>(nbc + ((size_t)e * 3 + v) * 6);
        double c[3];
        double2 b[3];
#pragma unroll
        for (int f = 0; f < 3; f++) {
            c[f] = W[(size_t)(f * DOF) * ne + e];
            b[f] = rec[f];
        }
#pragma unroll
        for (int f = 0; f < 3; f++) {
            if (c[f] < lo[f]) { lo[f] = c[f]; alo[f] = e; }
            if (c[f] > hi[f]) { hi[f] = c[f]; ahi[f] = e; }
            slo[f] += b[f].x;
            shi[f] += b[f].y;
        }
    }
    double2* g = reinterpret_cast<double2*>(gsum + (size_t)n * 6);
    int2* a = reinterpret_cast<int2*>(arg + (size_t)n * 6);
#pragma unroll
    for (int f = 0; f < 3; f++) {
        g[f] = make_double2(slo[f], shi[f]);
        a[f] = make_int2(alo[f], ahi[f]);
    }
}

// Per element: the bound cotangents of the nodes where this element's cell mean is the bound.
template <int P>
__global__ void __launch_bounds__(256) limiter_adj_gather_kernel(int np, ElemData E, const double* __restrict__ gsum,
                                                                 const int* __restrict__ arg, double* __restrict__ ub) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    const int ne = E.ne;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne) return;
    // the node indices, then every node's bound owners and cotangent sums together (a sum that is
    // not this element's adds zero, which leaves the running sum as it is)
    int2 a[3][3];
    double2 g[3][3];
#pragma unroll
    for (int v = 0; v < 3; v++) {
        const int n = E.nm[(size_t)v * ne + e];
#pragma unroll
        for (int f = 0; f < 3; f++) {
            a[v][f] = reinterpret_cast<const int2*>(arg + (size_t)n * 6)[f];
            g[v][f] = reinterpret_cast<const double2*>(gsum + (size_t)n * 6)[f];
        }
    }
#pragma unroll
    for (int f = 0; f < 3; f++) {
        double add = 0.0;
#pragma unroll
        for (int v = 0; v < 3; v++) {
            add += a[v][f].x == e ? g[v][f].x : 0.0;
            add += a[v][f].y == e ? g[v][f].y : 0.0;
        }
        ub[(size_t)(f * DOF) * ne + e] += add;
    }
}

// Node gradients from the element accumulators: dJ/dDP(n) = sum over incident elements of the
// vertex-depth cotangent; dJ/dn(n) = sum of the element-mean cotangents / 3.
__global__ void __launch_bounds__(256) param_gather_kernel(int np, int ne, const int* __restrict__ off,
                                                           const int* __restrict__ lst,
                                                           const double* __restrict__ gdp,
                                                           const double* __restrict__ gnbar,
                                                           double* __restrict__ out_dp, double* __restrict__ out_n) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= np) return;
    double sdp = 0.0, sn = 0.0;
    for (int j = off[n]; j < off[n + 1]; j++) {
        const int ent = lst[j];
        const int e = ent >> 2, v = ent & 3;
        sdp += gdp[(size_t)v * ne + e];
        sn += gnbar[e];
    }
    out_dp[n] = sdp;
    out_n[n] = sn / 3.0;
}

}  // namespace dg
