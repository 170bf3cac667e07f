// Device-side data structures and the numerical flux of the DG hydro step (gfx950, FP64).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "dg_crmath.hpp"

namespace dg {

constexpr int KMAXDOF = 6;
constexpr int KMAXAGP = 6;
constexpr int KMAXEGP = 4;
constexpr int KMAXRK = 8;

// Per-slot side descriptor packed 7 bits per slot into one int32 per element:
//   bits 0-1 local edge L (edge L runs from vertex L+1 to L+2, mod 3)
//   bit  2   role: 0 = this element is NEDEL(1) ("in"), 1 = NEDEL(2) ("ex")
//   bits 3-4 kind: 0 internal, 1 elevation-specified (ocean), 2 no-normal-flow (land), 3 flux
//   bits 5-6 neighbour's local edge (internal edges)
// Slots are stored in the reference's accumulation order: boundary edges first (ocean, land,
// flux, each in its list order), then internal edges by global edge number.
enum SideKind { SIDE_INTERNAL = 0, SIDE_OCEAN = 1, SIDE_LAND = 2, SIDE_FLOW = 3 };

__host__ __device__ inline int side_bits(int info, int slot) { return (info >> (7 * slot)) & 127; }

// Reference-element tables in constant memory (filled from RefTables at init).
struct DevTables {
    double phi_area[KMAXAGP][KMAXDOF];
    double drphi[KMAXAGP][KMAXDOF];
    double dsphi[KMAXAGP][KMAXDOF];
    double mw[KMAXAGP][KMAXDOF];
    double srfac[KMAXAGP][KMAXDOF];
    double phi_edge[3][KMAXEGP][KMAXDOF];
    double edgeq[3][KMAXEGP][KMAXDOF];
    double phi_corner[3][KMAXDOF];
    double m_inv[KMAXDOF];
    double wegp[KMAXEGP];
    double xegp[KMAXEGP];
    double psi[KMAXAGP][3];   // linear nodal basis at the area points (wind stress interpolation)
};

// The p=1 area rule's values (RefTables' to the last bit, checked at set-up), as constants for unrolled code:
// basis values, M_INV*WAGP (the same at every point) and its products with the basis values.
struct P1Area {
    static constexpr double phi[3][3] = {{1.0, 1.0, 0.0}, {1.0, -0.5, 0x1.0000000000001p-1}, {1.0, -0.5, -0x1.0000000000001p-1}};
    static constexpr double mw[3] = {0x1.5555555555555p-2, 0x1.5555555555555p-1, 2.0};
    static constexpr double srfac[3][3] = {{0x1.5555555555555p-2, 0x1.5555555555555p-1, 0.0},
                                           {0x1.5555555555555p-2, -0x1.5555555555555p-2, 0x1.0000000000001p+0},
                                           {0x1.5555555555555p-2, -0x1.5555555555555p-2, -0x1.0000000000001p+0}};
};

// Physics switches and constants shared by every scenario of a batch
// (src/dgswem.F:131-170 derivations).
struct Phys {
    double g, nleq, leq, nleqg, fg_l;
    double hbreak, ftheta, fgamma;
    int ifnlfa, iflinbf, ifhybf, load_manning;
};

// Per-scenario scalars (one entry per ensemble member; one entry for a single run).
struct Scen {
    double dtdp;       // DTDP
    double dtdph;      // 1/DTDP (friction cap)
    double h0;         // H0
    double cf;         // CF
    double fric;       // uniform FRIC_EL (without Manning)
    double cori;       // uniform Coriolis (when cori_el == nullptr)
    double rain;       // rain source rate (rainfall = 1) or 0
    double pad;
};

// Element-major structure-of-arrays mesh data on the device.
struct ElemData {
    int ne;
    const uint16_t* __restrict__ sid;   // [ne] scenario of each element, nullptr for one scenario
    const Scen* __restrict__ scen;      // [nscen]
    const double* __restrict__ xv;      // [3][ne] vertex x
    const double* __restrict__ yv;      // [3][ne] vertex y
    const double* __restrict__ dpv;     // [3][ne] vertex depth DP
    const double* __restrict__ nbar;    // [ne] mean nodal Manning n, or nullptr
    const double* __restrict__ cori_el; // [ne] or nullptr
    const double* __restrict__ sfacq;   // [nagp][ne] spherical factor at area points, or nullptr
    const double* __restrict__ sfaced;  // [3][negp][ne] spherical factor at edge points, or nullptr
    const double* __restrict__ sfs;     // [2][3 slots][negp][ne] the same in slot order: [0] own side
                                        // at the edge's point I, [1] the internal neighbour's side
    const int* __restrict__ sinfo;      // [ne] packed side descriptors
    const int* __restrict__ snbr;       // [3][ne] neighbour element / boundary-list index per slot
    const int* __restrict__ nm;         // [3][ne] 0-based vertex nodes
    const double* __restrict__ geo;     // [13][ne] per slot s: rows 3s..3s+2 the side's unit normal
                                        // (NX, NY) and XLEN/AREAS; rows 9..12 DRDX, DSDX, DRDY, DSDY
};

// Boundary forcing.  Per-stage scalars come from host-built tables [scenario][row][constituent];
// the row of the current stage is (*step)*nrk + irk, with the step counter kept on the device so
// that a captured graph of several steps can be replayed.
struct Forcing {
    int nbfr, nffr, rows, nrk;
    const int* __restrict__ step;       // device counter of the tables' step at which a graph replay
                                        // starts, or nullptr (eager launches)
    int step_imm;                       // step within the replay, or within the tables
    const double* __restrict__ emo;     // [needs][nbfr][2]
    const double* __restrict__ efa;     // [needs][nbfr][2]
    const double* __restrict__ qnam;    // [nfeds][nffr][2]
    const double* __restrict__ qnph;    // [nfeds][nffr][2]
    const double* __restrict__ argj;    // [nstage][nbfr]
    const double* __restrict__ rff;     // [nstage][nbfr]
    const double* __restrict__ fargj;   // [nstage][nffr]
    const double* __restrict__ frff;    // [nstage][nffr]
    const double* __restrict__ ramp;    // [scenario][row] RAMPDG of each stage (meteorological forcing)
    // tidal elevation terms EMO*RFF*COS(ARGJ-EFA) of the current step, [stage][needs][nbfr][2]
    // (tzn = needs*nbfr*2 per stage), written by tide_kernel for a batch of steps
    const double* __restrict__ tz;
    int tzn;
    // specified normal flux Q_N_EXT at every flux-edge quadrature point of the current step,
    // [stage][nfeds][negp] (fzn = nfeds*negp per stage), written by flow_kernel
    const double* __restrict__ fz;
    int fzn;
    // non-periodic boundaries (NBFR = 0, NFFR = 0): the ramped end-node values of every stage row,
    // [scenario*rows + row][needs][2] (elevation; nbfr is 1) and [scenario*rows + row][nfeds][2]
    // (normal flux; nffr is 1), or nullptr
    const double* __restrict__ ets;
    const double* __restrict__ qts;
    int nfeds;
};

// Tidal potential (NTIP != 0): per-stage-row constituent terms and node data for tip_kernel, which
// writes TIP2 of every stage at the nodes for a batch of steps.
struct Tip {
    int np, ntif;
    const double* __restrict__ row;      // [scenario*rows + row][ntif][3]: ARGT, TPMUL, SALTMUL
    const int* __restrict__ na;          // [ntif]: 1 semidiurnal, 2 diurnal, else no term
    const double* __restrict__ slam;     // [np] longitude (rad)
    const double* __restrict__ ccsfea;   // [np] COS(SFEA)**2
    const double* __restrict__ s2sfea;   // [np] SIN(2*SFEA)
    const double* __restrict__ salt_amp; // [ntif][np], or nullptr (NTIP = 1: zero)
    const double* __restrict__ salt_pha; // [ntif][np] radians
    double* __restrict__ tip2;           // [step of the batch][stage][np]
};

// Step index within the current forcing tables.
__device__ __forceinline__ int table_step(const Forcing& f) { return (f.step ? *f.step : 0) + f.step_imm; }


// NWS=8 meteorological forcing at the nodes.  The node kernel evaluates the Holland profile once
// per step at TIME_A (the reference evaluates it at every stage with the same TIME_A) and forms
// WSX2 = RampMete*0.001293*Cd*Wx*|W|, WSY2 and PR2 = RampMete*P with each stage's ramp, in the
// reference's operation order.
struct Met {
    int np, rows;                        // rows: steps per scenario in the storm table
    const double* __restrict__ row;     // [scenario][rows][MET_ROW] storm scalars per step
    const uint16_t* __restrict__ nsid;  // [np] scenario of each node, nullptr for one scenario
    const double* __restrict__ xc;      // [np] longitude (deg)
    const double* __restrict__ yc;      // [np] latitude (deg)
    const double* __restrict__ cosy;    // [np] cos(latitude)
    const double* __restrict__ cor;     // [np] 2 omega sin(latitude)
    double4* __restrict__ st;           // [step of the batch][stage][np] WSX2, WSY2, PR2 of the stage, unused
};

// Block-local node bounds of the slope limiter.  Tile t (elements [t*nt, t*nt+nt)) stages the
// cell means of its own elements (rows 0..nt-1) and of its vertex halo -- the elements outside
// the tile that share a node with it, vhidx[t*nvh..t*nvh+nvh), -1 past its last (rows nt..) -- and forms
// the bounds of its nodes from their incident elements: node q's first eight as staged rows (times 8, the
// byte offset) qinc[(t*nql+q)*8..+8), fewer repeated (min and max are idempotent), and further ones in the extra entries
// xoff[t]..xoff[t+1) (xq: the node, xinc: eight rows).  elq packs each element's three tile-local node
// numbers (10 bits each).
struct LimTiles {
    const int* __restrict__ vhidx;
    const uint16_t* __restrict__ qinc;
    const int* __restrict__ xoff;
    const int* __restrict__ xq;
    const uint16_t* __restrict__ xinc;
    const int* __restrict__ elq;
    int nvh, nql;                       // halo entries and nodes per tile (the largest tile's)
    int nx;                             // extra entries of all tiles (none: xoff is not read)
};

// Local Lax-Friedrichs flux (src/numerical_flux.F:750-1022), operation order kept.
__device__ __forceinline__ void llf_flux(const Phys& P, double ze_in, double ze_ex, double qx_in,
                                         double qx_ex, double qy_in, double qy_ex, double hb_in,
                                         double hb_ex, double sf_in, double sf_ex, double nx,
                                         double ny, double G, double& f0, double& f1, double& f2) {
    const double NLEQ = P.nleq, LEQ = P.leq, FG_L = P.fg_l;
    const double NLEQG = G * NLEQ;
    const double j1 = ze_ex - ze_in, j2 = qx_ex - qx_in, j3 = qy_ex - qy_in;
    const double ht_in = ze_in * NLEQ + hb_in;
    double fnl = NLEQ + LEQ * hb_in;
    const double fx1_in = qx_in * fnl * sf_in, fy1_in = qy_in * fnl;
    double fu = NLEQ * qx_in, fv = NLEQ * qy_in, fg = NLEQG * ze_in;
    double fh = 1.0 / (NLEQ * ht_in + LEQ);
    const double u_in = qx_in * fh, v_in = qy_in * fh;
    double huu = fu * u_in, hvv = fv * v_in, huv = fu * v_in;
    double gh2 = fg * (0.5 * ze_in + hb_in) + FG_L * ze_in;
    const double fx2_in = (huu + gh2) * sf_in, fy2_in = huv;
    const double fx3_in = huv * sf_in, fy3_in = hvv + gh2;
    const double ht_ex = ze_ex * NLEQ + hb_ex;
    fnl = NLEQ + LEQ * hb_ex;
    const double fx1_ex = qx_ex * fnl * sf_ex, fy1_ex = qy_ex * fnl;
    fu = NLEQ * qx_ex; fv = NLEQ * qy_ex; fg = NLEQG * ze_ex;
    fh = 1.0 / (NLEQ * ht_ex + LEQ);
    const double u_ex = qx_ex * fh, v_ex = qy_ex * fh;
    huu = fu * u_ex; hvv = fv * v_ex; huv = fu * v_ex;
    gh2 = fg * (0.5 * ze_ex + hb_ex) + FG_L * ze_ex;
    const double fx2_ex = (huu + gh2) * sf_ex, fy2_ex = huv;
    const double fx3_ex = huv * sf_ex, fy3_ex = hvv + gh2;
    const double a1 = 0.5 * ((fx1_in + fx1_ex) * nx + (fy1_in + fy1_ex) * ny);
    const double a2 = 0.5 * ((fx2_in + fx2_ex) * nx + (fy2_in + fy2_ex) * ny);
    const double a3 = 0.5 * ((fx3_in + fx3_ex) * nx + (fy3_in + fy3_ex) * ny);
    const double un_in = (u_in * nx + v_in * ny) * NLEQ;
    double nxs = nx * sf_in;
    const double c_in = sqrt(G * ht_in * (ny * ny + nxs * nxs));
    const double un_ex = (u_ex * nx + v_ex * ny) * NLEQ;
    nxs = nx * sf_ex;
    const double c_ex = sqrt(G * ht_ex * (ny * ny + nxs * nxs));
    double em = fabs(un_in + c_in);
    em = fmax(em, fabs(un_in));
    em = fmax(em, fabs(un_in - c_in));
    em = fmax(em, fabs(un_ex + c_ex));
    em = fmax(em, fabs(un_ex));
    em = fmax(em, fabs(un_ex - c_ex));
    const double nx2 = NLEQ + LEQ * nx * nx, ny2 = NLEQ + LEQ * ny * ny, nxy = nx * ny;
    f0 = a1 - 0.5 * em * (j1);
    f1 = a2 - 0.5 * em * (j2 * nx2 + LEQ * j3 * nxy);
    f2 = a3 - 0.5 * em * (j3 * ny2 + LEQ * j2 * nxy);
}

// llf_flux for the nonlinear equations (NOLICAT != 0: NLEQ = 1, LEQ = 0) with those constants
// folded by hand: x*NLEQ = x, NLEQ + LEQ*h = 1 and y + LEQ*z = y hold exactly for finite operands,
// so the values equal llf_flux's bit for bit (up to the sign of an exact zero).
__device__ __forceinline__ void llf_flux_nl(double ze_in, double ze_ex, double qx_in, double qx_ex,
                                            double qy_in, double qy_ex, double hb_in, double hb_ex,
                                            double sf_in, double sf_ex, double nx, double ny, double G,
                                            double& f0, double& f1, double& f2) {
    const double j1 = ze_ex - ze_in, j2 = qx_ex - qx_in, j3 = qy_ex - qy_in;
    const double ht_in = ze_in + hb_in;
    const double fx1_in = qx_in * sf_in, fy1_in = qy_in;
    double fg = G * ze_in;
    double fh = 1.0 / ht_in;
    const double u_in = qx_in * fh, v_in = qy_in * fh;
    double huu = qx_in * u_in, hvv = qy_in * v_in, huv = qx_in * v_in;
    double gh2 = fg * (0.5 * ze_in + hb_in);
    const double fx2_in = (huu + gh2) * sf_in, fy2_in = huv;
    const double fx3_in = huv * sf_in, fy3_in = hvv + gh2;
    const double ht_ex = ze_ex + hb_ex;
    const double fx1_ex = qx_ex * sf_ex, fy1_ex = qy_ex;
    fg = G * ze_ex;
    fh = 1.0 / ht_ex;
    const double u_ex = qx_ex * fh, v_ex = qy_ex * fh;
    huu = qx_ex * u_ex; hvv = qy_ex * v_ex; huv = qx_ex * v_ex;
    gh2 = fg * (0.5 * ze_ex + hb_ex);
    const double fx2_ex = (huu + gh2) * sf_ex, fy2_ex = huv;
    const double fx3_ex = huv * sf_ex, fy3_ex = hvv + gh2;
    const double a1 = 0.5 * ((fx1_in + fx1_ex) * nx + (fy1_in + fy1_ex) * ny);
    const double a2 = 0.5 * ((fx2_in + fx2_ex) * nx + (fy2_in + fy2_ex) * ny);
    const double a3 = 0.5 * ((fx3_in + fx3_ex) * nx + (fy3_in + fy3_ex) * ny);
    const double un_in = u_in * nx + v_in * ny;
    double nxs = nx * sf_in;
    const double c_in = sqrt(G * ht_in * (ny * ny + nxs * nxs));
    const double un_ex = u_ex * nx + v_ex * ny;
    nxs = nx * sf_ex;
    const double c_ex = sqrt(G * ht_ex * (ny * ny + nxs * nxs));
    double em = fabs(un_in + c_in);
    em = fmax(em, fabs(un_in));
    em = fmax(em, fabs(un_in - c_in));
    em = fmax(em, fabs(un_ex + c_ex));
    em = fmax(em, fabs(un_ex));
    em = fmax(em, fabs(un_ex - c_ex));
    f0 = a1 - 0.5 * em * (j1);
    f1 = a2 - 0.5 * em * (j2);
    f2 = a3 - 0.5 * em * (j3);
}

// 1/x for x in [2^-500, 2^500], correctly rounded: the Newton steps and the final correction of the
// IEEE division without its scaling of extreme operands and its fix-up of zeros and infinities (7
// instructions instead of 11).
__device__ __forceinline__ double recip_mid(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
    r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
    return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}

// sqrt(x) for x in [2^-700, 2^700], correctly rounded: the Goldschmidt steps and two corrections of the
// IEEE square root without its scaling of small operands and its selection of zeros and infinities
// (10 instructions instead of 19).
__device__ __forceinline__ double sqrt_mid(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// High word of a depth, offset so that one unsigned comparison with DEPTH_SPAN tells whether it lies in
// [2^-500, 2^500), where recip_mid and sqrt_mid apply (negative values, zero and NaN lie outside).
constexpr uint32_t DEPTH_SPAN = 1000u << 20;
__device__ __forceinline__ uint32_t depth_key(double h) { return (uint32_t)__double2hiint(h) - ((1023u - 500u) << 20); }

// Twice llf_flux_nl's fluxes, the same bits, for depths ht in recip_mid's range and K = NY^2+(NX*SF)^2 such
// that G*ht*K is in sqrt_mid's.  Where the operations differ from llf_flux_nl's:
//   * multiplications by 0.5 are exact, so they move into the edge weight;
//   * 0.5*z is exact, so 0.5*z + h is one fused operation;
//   * c >= 0, so the largest of |un+c|, |un|, |un-c| is |un|+c (rounding is monotonic and symmetric).
__device__ __forceinline__ void llf_flux_nl2(double ze_in, double ze_ex, double qx_in, double qx_ex, double qy_in,
                                             double qy_ex, double hb_in, double hb_ex, double ht_in, double ht_ex,
                                             double sf_in, double sf_ex, double K_in, double K_ex, double nx, double ny,
                                             double G, double& f0, double& f1, double& f2) {
    const double j1 = ze_ex - ze_in, j2 = qx_ex - qx_in, j3 = qy_ex - qy_in;
    double fh = recip_mid(ht_in);
    const double u_in = qx_in * fh, v_in = qy_in * fh;
    double huu = qx_in * u_in, hvv = qy_in * v_in, huv = qx_in * v_in;
    double gh2 = G * ze_in * __builtin_fma(0.5, ze_in, hb_in);
    const double fx1_in = qx_in * sf_in, fx2_in = (huu + gh2) * sf_in, fy2_in = huv;
    const double fx3_in = huv * sf_in, fy3_in = hvv + gh2;
    fh = recip_mid(ht_ex);
    const double u_ex = qx_ex * fh, v_ex = qy_ex * fh;
    huu = qx_ex * u_ex; hvv = qy_ex * v_ex; huv = qx_ex * v_ex;
    gh2 = G * ze_ex * __builtin_fma(0.5, ze_ex, hb_ex);
    const double fx1_ex = qx_ex * sf_ex, fx2_ex = (huu + gh2) * sf_ex, fy2_ex = huv;
    const double fx3_ex = huv * sf_ex, fy3_ex = hvv + gh2;
    const double un_in = u_in * nx + v_in * ny, un_ex = u_ex * nx + v_ex * ny;
    const double em = fmax(fabs(un_in) + sqrt_mid(G * ht_in * K_in), fabs(un_ex) + sqrt_mid(G * ht_ex * K_ex));
    f0 = (fx1_in + fx1_ex) * nx + (qy_in + qy_ex) * ny - em * j1;
    f1 = (fx2_in + fx2_ex) * nx + (fy2_in + fy2_ex) * ny - em * j2;
    f2 = (fx3_in + fx3_ex) * nx + (fy3_in + fy3_ex) * ny - em * j3;
}

template <bool NL>
__device__ __forceinline__ void llf(const Phys& P, double ze_in, double ze_ex, double qx_in, double qx_ex,
                                    double qy_in, double qy_ex, double hb_in, double hb_ex, double sf_in,
                                    double sf_ex, double nx, double ny, double G, double& f0, double& f1,
                                    double& f2) {
    if constexpr (NL)
        llf_flux_nl(ze_in, ze_ex, qx_in, qx_ex, qy_in, qy_ex, hb_in, hb_ex, sf_in, sf_ex, nx, ny, G, f0, f1, f2);
    else
        llf_flux(P, ze_in, ze_ex, qx_in, qx_ex, qy_in, qy_ex, hb_in, hb_ex, sf_in, sf_ex, nx, ny, G, f0, f1, f2);
}

}  // namespace dg
