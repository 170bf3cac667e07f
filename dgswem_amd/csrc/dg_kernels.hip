// HIP kernels of the DG hydro step for gfx950 (MI355X), FP64.
//
// One time step = NRK stages; each stage is
//   stage_kernel     one thread per element: fluxes on its three edges (ocean / land / flux /
//                    internal, LLF), volume quadrature, SSP-RK update of the element's modes, and
//                    (when the slope limiter is off) the element's wet/dry correction.  Internal
//                    edge fluxes are evaluated by both neighbours with the same operands in the same
//                    order, so both see bit-identical values and no scatter or atomics are needed.
//                    Small meshes run stage_split_kernel, four waves per 64 elements, instead.
//   limit_wetdry     SLOPELIMITER5 on modes 2-3, then WETDRY: a wave per field of 64 elements, on large meshes
//                    (limit_wide) a wave for all three
// preceded once per batch of steps by tide_kernel (the tidal boundary terms of every stage) and, with
// NWS=8, met_kernel (the Holland profile at the nodes); plus modal2nodal (one thread per node) on output
// steps.
//
// Arithmetic follows the reference statement by statement (listed per kernel) and is compiled with
// -ffp-contract=off, so each product and sum is rounded as in dgswem_serial; the cosine of the
// tidal terms and Manning's DEPTH**(1/3) are correctly rounded (dg_crmath.hpp).
#include "dg_device.hpp"
#include "dg_setup.hpp"

namespace dg {

__constant__ DevTables c_tab1;   // p = 1
__constant__ DevTables c_tab2;   // p = 2

template <int P> __device__ __forceinline__ const DevTables& tab();
template <> __device__ __forceinline__ const DevTables& tab<1>() { return c_tab1; }
template <> __device__ __forceinline__ const DevTables& tab<2>() { return c_tab2; }

// Blocks are dispatched round-robin over the 8 XCDs; give each XCD a contiguous range of element
// tiles so that a tile's neighbours (close in the Hilbert order) sit in the same XCD's L2.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
    const int q = nb >> 3, r = nb & 7, x = b & 7;
    return x * q + min(x, r) + (b >> 3);
}

struct StageArgs {
    ElemData ed;
    Phys ph;
    Forcing fo;
    Met mt;
    const double* __restrict__ uin;      // U(IRK) [3][dof][ne]
    double* __restrict__ uout;           // U(IRK+1)
    const uint8_t* __restrict__ wd_in;   // WDFLG during the stage
    uint8_t* __restrict__ wd_out;        // WDFLG after WETDRY (fused variant)
    int nprev;                           // stages I < IRK entering the update
    const double* uprev[KMAXRK];
    double aprev[KMAXRK];                // ATVD(IRK,I), 0 = term absent
    const double* rprev[KMAXRK];
    double bprev[KMAXRK];                // BTVD(IRK,I) (times the scenario's DT in the kernel)
    double acur, bcur;                   // ATVD(IRK,IRK), BTVD(IRK,IRK)
    double* __restrict__ rout;           // RHS(IRK) kept for later stages, or nullptr
    int irk;                             // stage index
    // block-local staging: tile t (elements [t*NT, t*NT+NT)) stages its elements and its halo
    // hidx[t*nh..t*nh+nh) (-1 past the tile's last) in LDS; snbl packs each side's local neighbour
    // index (10 bits each)
    const int* __restrict__ hidx;
    const int* __restrict__ snbl;
    int nh, ns;                          // halo entries per tile, staged elements per block (LDS row length)
    int* __restrict__ wd_active;         // set to 1 when WETDRY changes an element, or nullptr
    const double* __restrict__ tip;      // TIP2 of this stage at the nodes (tidal potential), or nullptr
    double* __restrict__ cmout;          // copy of the output cell means [3][ne] for the limiter, or nullptr
    double* __restrict__ wout;           // copy of the output before the limiter (adjoint), or nullptr
    int mid;                             // G and the spherical factors allow llf_flux_nl2 (depths permitting)
};

// ------------------------------------------------------------------------------------------
// WETDRY for one element (src/wetdry.F:58-548, p=1 vertex logic; modes >= 4 zeroed).
// Updates ze/qx/qy in place and returns the new WDFLG.
// ------------------------------------------------------------------------------------------
template <int P>
__device__ __forceinline__ int wetdry_element(const DevTables& T, double (&U)[3][(P + 1) * (P + 2) / 2],
                                              const double dpn[3], const double hb[3], double dpe_min,
                                              int wdflg, double H0) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    const double ZERO = 1.0e-6, C13 = 1.0 / 3.0, C16 = 1.0 / 6.0;
    int ndry = 0, ht_max_i = 0;
    double ht_max = ZERO;
    double ze_node[3], ht_node[3], ze_hat[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double z = U[0][0];
#pragma unroll
        for (int k = 1; k < 3; k++) z = z + T.phi_corner[i][k] * U[0][k];
        ze_node[i] = z;
        ht_node[i] = dpn[i] + z;
        if (ht_node[i] > ht_max) { ht_max_i = i; ht_max = ht_node[i]; }
        if (ht_node[i] <= (H0 + ZERO)) ndry++;
    }
    const double dp_avg = C13 * (dpn[0] + dpn[1] + dpn[2]);
    int check = 0;
    if (ndry == 0) {
        if (wdflg == 1) return 1;
        ze_hat[0] = ze_node[0]; ze_hat[1] = ze_node[1]; ze_hat[2] = ze_node[2];
        check = 1;
    } else if (ndry == 3) {
        const double ht_avg = U[0][0] + dp_avg;
#pragma unroll
        for (int k = 0; k < DOF; k++) { U[0][k] = 0.0; U[1][k] = 0.0; U[2][k] = 0.0; }
        U[0][0] = ht_avg - dp_avg;
        if (ht_avg < ZERO) U[0][0] = ZERO - dp_avg;
        U[0][1] = -hb[1]; U[0][2] = -hb[2];
        return 0;
    } else {
        const double ht_avg = U[0][0] + dp_avg;
        if (ht_avg <= (H0 + ZERO)) {
#pragma unroll
            for (int k = 0; k < DOF; k++) { U[0][k] = 0.0; U[1][k] = 0.0; U[2][k] = 0.0; }
            U[0][0] = ht_avg - dp_avg;
            if (ht_avg < ZERO) U[0][0] = ZERO - dp_avg;
            U[0][1] = -hb[1]; U[0][2] = -hb[2];
            ze_hat[0] = ze_hat[1] = ze_hat[2] = U[0][0];
        } else {
            // order the vertices by depth (the reference's exchange sort)
            int l2h[3] = {0, 1, 2};
#pragma unroll
            for (int k1 = 0; k1 < 3; k1++)
#pragma unroll
                for (int k2 = k1; k2 < 3; k2++)
                    if (ht_node[l2h[k1]] > ht_node[l2h[k2]]) { const int t = l2h[k1]; l2h[k1] = l2h[k2]; l2h[k2] = t; }
            double dh[3];
            dh[l2h[0]] = fmax(H0, ht_node[l2h[0]]) - ht_node[l2h[0]];
            dh[l2h[1]] = fmax(H0, ht_node[l2h[1]] - 0.5 * dh[l2h[0]]) - ht_node[l2h[1]];
            dh[l2h[2]] = -dh[l2h[0]] - dh[l2h[1]];
            int nd = 0;
            double qxs = 0, qys = 0;
            ht_max = 0;
            double ht_hat[3], qxn[3], qyn[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                ht_hat[i] = ht_node[i] + dh[i];
                double a = U[1][0], b = U[2][0];
                if (ht_hat[i] > ht_max) { ht_max_i = i; ht_max = ht_hat[i]; }
#pragma unroll
                for (int k = 1; k < 3; k++) { a = a + T.phi_corner[i][k] * U[1][k]; b = b + T.phi_corner[i][k] * U[2][k]; }
                qxn[i] = a; qyn[i] = b;
                if (ht_hat[i] <= (H0 + 1.0e-10)) { nd++; qxs = qxs + a; qys = qys + b; }
            }
            if (nd == 3) {
#pragma unroll
                for (int k = 0; k < DOF; k++) { U[1][k] = 0.0; U[2][k] = 0.0; }
            } else {
                qxs = qxs / (3.0 - (double)nd);
                qys = qys / (3.0 - (double)nd);
                double qxh[3], qyh[3];
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    if (ht_hat[i] <= (H0 + 1.0e-10)) { qxh[i] = 0.0; qyh[i] = 0.0; }
                    else { qxh[i] = qxn[i] + qxs; qyh[i] = qyn[i] + qys; }
                }
                U[1][0] = C13 * (qxh[0] + qxh[1] + qxh[2]);
                U[1][1] = -(C16 * (qxh[0] + qxh[1])) + C13 * qxh[2];
                U[1][2] = -(0.5 * qxh[0]) + 0.5 * qxh[1];
                U[2][0] = C13 * (qyh[0] + qyh[1] + qyh[2]);
                U[2][1] = -(C16 * (qyh[0] + qyh[1])) + C13 * qyh[2];
                U[2][2] = -(0.5 * qyh[0]) + 0.5 * qyh[1];
            }
#pragma unroll
            for (int i = 0; i < 3; i++) ze_hat[i] = ht_hat[i] - dpn[i];
            U[0][1] = -(C16 * (ze_hat[0] + ze_hat[1])) + C13 * ze_hat[2];
            U[0][2] = -(0.5 * ze_hat[0]) + 0.5 * ze_hat[1];
        }
#pragma unroll
        for (int k = 3; k < DOF; k++) { U[0][k] = 0.0; U[1][k] = 0.0; U[2][k] = 0.0; }
        check = 1;
    }
    if (check) {
        if (ze_hat[ht_max_i] > (-dpe_min + H0)) return 1;
#pragma unroll
        for (int k = 0; k < DOF; k++) { U[1][k] = 0.0; U[2][k] = 0.0; }
        return 0;
    }
    return wdflg;
}

// True when WETDRY leaves the element as it is (every vertex wet and the element already wet: the
// identity branch of wetdry_element).
template <int P>
__device__ __forceinline__ bool wetdry_keeps(const DevTables& T, const double (&U)[3][(P + 1) * (P + 2) / 2],
                                             const double dpn[3], int wdflg, double H0) {
    if (wdflg != 1) return false;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double z = U[0][0];
#pragma unroll
        for (int k = 1; k < 3; k++) z = z + T.phi_corner[i][k] * U[0][k];
        if (dpn[i] + z <= (H0 + 1.0e-6)) return false;
    }
    return true;
}

// ------------------------------------------------------------------------------------------
// Element geometry, once per mesh (src/calc_normal.F:28-49, src/prep_DG.F:959-1163): per slot the
// side's unit normal in the reference's node order (the counter-clockwise order of the edge's
// NEDEL(1) element, so both elements of an internal edge form the same normal from the same two
// vertices) and XLEN/AREAS, and the Jacobian terms DRDX, DSDX, DRDY, DSDY.  The stage kernel
// reads them instead of forming them every stage; the expressions are the ones it would evaluate,
// so the values are the same bits.
// ------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) geom_kernel(int ne, const double* __restrict__ xv, const double* __restrict__ yv,
                                                   const int* __restrict__ sinfo, double* __restrict__ geo) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ne) return;
    const double X[3] = {xv[e], xv[(size_t)ne + e], xv[2 * (size_t)ne + e]};
    const double Y[3] = {yv[e], yv[(size_t)ne + e], yv[2 * (size_t)ne + e]};
    const double AREAS = (X[0] - X[2]) * (Y[1] - Y[2]) + (X[2] - X[1]) * (Y[0] - Y[2]);
    const int info = sinfo[e];
    for (int slot = 0; slot < 3; slot++) {
        const int bits = side_bits(info, slot);
        const int L = bits & 3, role = (bits >> 2) & 1;
        int va = (L + 1) % 3, vb = (L + 2) % 3;
        if (role) { const int t = va; va = vb; vb = t; }
        const double dy = Y[vb] - Y[va];
        const double dx = X[vb] - X[va];
        const double xlen = sqrt(dy * dy + dx * dx);
        geo[(size_t)(3 * slot) * ne + e] = dy / xlen;
        geo[(size_t)(3 * slot + 1) * ne + e] = -dx / xlen;
        geo[(size_t)(3 * slot + 2) * ne + e] = xlen / AREAS;
    }
    double AREA = (X[0] - X[2]) * (Y[1] - Y[2]) + (X[2] - X[1]) * (Y[0] - Y[2]);
    AREA = AREA * 0.5;
    geo[(size_t)9 * ne + e] = 1.0 / AREA * (Y[2] - Y[0]);
    geo[(size_t)10 * ne + e] = 1.0 / AREA * (Y[0] - Y[1]);
    geo[(size_t)11 * ne + e] = 1.0 / AREA * (X[0] - X[2]);
    geo[(size_t)12 * ne + e] = 1.0 / AREA * (X[1] - X[0]);
}

// XLEN of a side and AREAS (twice the element's area), formed from the vertex coordinates as the
// geometry kernel forms them: the boundary-edge terms need them apart.
__device__ __forceinline__ void side_xlen_areas(const ElemData& E, int ne, int e, int L, int role, double& xlen,
                                                double& AREAS) {
    const double X[3] = {E.xv[e], E.xv[(size_t)ne + e], E.xv[2 * (size_t)ne + e]};
    const double Y[3] = {E.yv[e], E.yv[(size_t)ne + e], E.yv[2 * (size_t)ne + e]};
    AREAS = (X[0] - X[2]) * (Y[1] - Y[2]) + (X[2] - X[1]) * (Y[0] - Y[2]);
    int va = (L + 1) % 3, vb = (L + 2) % 3;
    if (role) { const int t = va; va = vb; vb = t; }
    const double dy = Y[vb] - Y[va];
    const double dx = X[vb] - X[va];
    xlen = sqrt(dy * dy + dx * dx);
}

// ------------------------------------------------------------------------------------------
// Stage kernel.  Reference statements restated:
//   OCEAN_EDGE_HYDRO   src/ocean_edge_hydro.F:19-355
//   LAND_EDGE_HYDRO    src/land_edge_hydro.F:26-311
//   FLOW_EDGE_HYDRO    src/flow_edge_hydro.F:20-333
//   INTERNAL_EDGE_HYDRO + add_internal_flux  src/internal_edge_hydro.F:37-383
//   RHS_DG_HYDRO       src/rhs_dg_hydro.F:18-473
//   SSP-RK update      src/DG_hydro_timestep.F:238-290
//   element geometry   src/read_input.F:1408, src/prep_DG.F:959-1163, src/calc_normal.F:28-49
// ------------------------------------------------------------------------------------------
// Trace of the element's modes at a point with basis values ph[] (sum from zero, mode order).
template <int DOF>
__device__ __forceinline__ double trace(const double (&u)[DOF], const double* ph) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < DOF; k++) s = s + u[k] * ph[k];
    return s;
}

// The same sum where ph[0] == 1: 0 + u0*1 = u0 for every u0 but -0, so the sum starts at u0.
template <int DOF>
__device__ __forceinline__ double trace1(const double (&u)[DOF], const double* ph) {
    double s = u[0];
#pragma unroll
    for (int k = 1; k < DOF; k++) s = s + u[k] * ph[k];
    return s;
}

// Element i of a row, addressed as the row's (uniform) base plus a 32-bit byte offset: the form in which
// the base stays in scalar registers.  Batches hold fewer than 2^29 elements, so the offset fits.
template <typename T>
__device__ __forceinline__ T& at(T* row, int i) {
    return *reinterpret_cast<T*>(reinterpret_cast<char*>(const_cast<std::remove_const_t<T>*>(row)) + (uint32_t)i * (uint32_t)sizeof(T));
}

// The same value, opaque to the optimiser: what is addressed by it is read where it is used and not
// kept in registers over a loop.
__device__ __forceinline__ int reread(int j) {
    asm volatile("" : "+v"(j));
    return j;
}

// s + u*ph with ph an edge value of a p=1 mode: 0 or a power of two (checked at set-up), so the product is
// exact and one fused operation gives the two roundings' result.  At p=2 product and sum round apart.
template <int DOF>
__device__ __forceinline__ double edge_term(double s, double u, double ph) {
    return DOF == 3 ? __builtin_fma(u, ph, s) : s + u * ph;
}

// The staged element j's traces (elevation, the two discharges, bathymetry) at an edge point with
// basis values ph; PHI_EDGE of mode 1 is 1 (checked at set-up), so the sums start at mode 1.
template <int DOF>
__device__ __forceinline__ void edge_point(const double* stg, int ns, int j, const double* ph, double (&t)[4]) {
#pragma unroll
    for (int f = 0; f < 4; f++) {
        t[f] = stg[f * DOF * ns + j];
#pragma unroll
        for (int k = 1; k < (f < 3 ? DOF : 3); k++) t[f] = edge_term<DOF>(t[f], stg[(f * DOF + k) * ns + j], ph[k]);
    }
}

// The same at every point of an edge with the basis table tb, `rev`: the points in reverse.
template <int DOF, int NEGP>
__device__ __forceinline__ void edge_traces(const double* stg, int ns, int j, const double (*tb)[DOF], bool rev,
                                            double (&t)[4][NEGP]) {
    double V[3][DOF], hb[3];
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) V[f][k] = stg[(f * DOF + k) * ns + j];
#pragma unroll
    for (int m = 0; m < 3; m++) hb[m] = stg[(3 * DOF + m) * ns + j];
#pragma unroll
    for (int I = 0; I < NEGP; I++) {
        const double* ph = tb[rev ? NEGP - 1 - I : I];
#pragma unroll
        for (int f = 0; f < 3; f++) {
            t[f][I] = V[f][0];
#pragma unroll
            for (int k = 1; k < DOF; k++) t[f][I] = edge_term<DOF>(t[f][I], V[f][k], ph[k]);
        }
        t[3][I] = edge_term<DOF>(edge_term<DOF>(hb[0], hb[1], ph[1]), hb[2], ph[2]);
    }
}

// The tile's edge basis and edge quadrature tables in LDS: they are indexed by each lane's own local
// edge number, and read as divergent constant-memory loads they would put a memory latency into
// every point.
template <int DOF, int NEGP>
struct EdgeTables {
    double pe[3][NEGP][DOF], eq[3][NEGP][DOF];
};

template <int DOF, int NEGP>
__device__ __forceinline__ void load_edge_tables(const DevTables& T, EdgeTables<DOF, NEGP>& t, int tid, int nt) {
    for (int j = tid; j < 3 * NEGP * DOF; j += nt) {
        const int l = j / (NEGP * DOF), g = (j / DOF) % NEGP, k = j % DOF;
        t.pe[l][g][k] = T.phi_edge[l][g][k];
        t.eq[l][g][k] = T.edgeq[l][g][k];
    }
}

// One internal side (slot `slot`) of staged element `le`: its RHS terms, summed over the side's points
// (INTERNAL_EDGE_HYDRO + add_internal_flux).  acc is set.
template <int P, bool SPH, bool NL, int DRYU>
__device__ __forceinline__ void internal_side(const StageArgs& a, const EdgeTables<(P + 1) * (P + 2) / 2, P + 2>& tb,
                                              const double* stg, const uint8_t* stwd, int ne, int ec, int le, int slot,
                                              int bits, int sl, int wd, double nx, double ny, double edfac,
                                              double (&acc)[3][(P + 1) * (P + 2) / 2]) {
    constexpr int DOF = (P + 1) * (P + 2) / 2, NEGP = P + 2;
    const ElemData& E = a.ed;
    const Phys& ph = a.ph;
    const int ns = a.ns;
    const int L = bits & 3, role = (bits >> 2) & 1, nled = (bits >> 5) & 3;
    const int ln = (sl >> (10 * slot)) & 1023;
    const int wdn = stwd[ln];
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) acc[f][k] = 0.0;
    if (wd == 0 && wdn == 0) return;
    // the edge's "in" (NEDEL(1)) and "ex" (NEDEL(2)) elements as staged rows and their local edge numbers
    const int si0 = role ? ln : le, sx0 = role ? le : ln;
    const int Li = role ? nled : L, Lx = role ? L : nled;
    // the "in" side subtracts w*F and the "ex" side adds it; -(a*b) == (-a)*b exactly, so the sign
    // goes on the edge factor once and one update serves both roles
    const double edfs = role ? edfac : -edfac;
    // spherical factors of both sides at every point, loaded together
    double sfi[NEGP], sfx[NEGP];
#pragma unroll
    for (int I = 0; I < NEGP; I++) {
        sfi[I] = SPH ? at(E.sfs + ((size_t)((role ? 3 : 0) + slot) * NEGP + I) * ne, ec) : 1.0;
        sfx[I] = SPH ? at(E.sfs + ((size_t)((role ? 0 : 3) + slot) * NEGP + I) * ne, ec) : 1.0;
    }
    double F[3][NEGP];                   // twice the flux
    bool mid = NL && a.mid;
    {
        // the traces of one side after the other, so that only one side's modes are held
        double ti[4][NEGP], tx[4][NEGP];
        edge_traces<DOF, NEGP>(stg, ns, si0, tb.pe[Li], false, ti);
        edge_traces<DOF, NEGP>(stg, ns, sx0, tb.pe[Lx], true, tx);
        if constexpr (NL) {
            double Ki = 0.0, Kx = 0.0;
            uint32_t key = 0;
#pragma unroll
            for (int I = 0; I < NEGP; I++) {
                const double hi = ti[0][I] + ti[3][I], hx = tx[0][I] + tx[3][I];
                key = max(key, max(depth_key(hi), depth_key(hx)));
                if (SPH || I == 0) {
                    const double ni = nx * sfi[I], ne_ = nx * sfx[I];
                    Ki = ny * ny + ni * ni;
                    Kx = ny * ny + ne_ * ne_;
                }
                llf_flux_nl2(ti[0][I], tx[0][I], ti[1][I], tx[1][I], ti[2][I], tx[2][I], ti[3][I], tx[3][I], hi, hx,
                             sfi[I], sfx[I], Ki, Kx, nx, ny, ph.g, F[0][I], F[1][I], F[2][I]);
            }
            mid = mid && key < DEPTH_SPAN;
        } else {
#pragma unroll
            for (int I = 0; I < NEGP; I++) {
                llf<NL>(ph, ti[0][I], tx[0][I], ti[1][I], tx[1][I], ti[2][I], tx[2][I], ti[3][I], tx[3][I], sfi[I],
                        sfx[I], nx, ny, ph.g, F[0][I], F[1][I], F[2][I]);
#pragma unroll
                for (int f = 0; f < 3; f++) F[f][I] = 2.0 * F[f][I];
            }
            mid = true;
        }
    }
    if (!mid || wd == 0 || wdn == 0) {
        // a depth outside llf_flux_nl2's range, or one side dry (few lanes, at the shoreline;
        // src/internal_edge_hydro.F:212-302): 1 reflect into a dry "in" element, 2 zero-gravity flux for a
        // dry "in", 3 reflect into a dry "ex", 4 zero-gravity flux for a dry "ex"; only what this element's
        // side receives.  The traces are formed again from LDS: held over the fluxes above they would set
        // the kernel's register count.
        const int wd_in_el = role ? wdn : wd;
#pragma unroll DRYU
        for (int I = 0; I < NEGP; I++) {
            double f0 = 0.0, f1 = 0.0, f2 = 0.0;
            double si_ = 1.0, sx_ = 1.0;
#pragma unroll
            for (int j = 0; j < NEGP; j++)
                if (j == I) { f0 = 0.5 * F[0][j]; f1 = 0.5 * F[1][j]; f2 = 0.5 * F[2][j]; si_ = sfi[j]; sx_ = sfx[j]; }
            // the plain flux (where the range calls for it), then the dry-side case it selects
            int mode = 0;
#pragma unroll 1
            for (int pass = mid ? 1 : 0; pass < 2; pass++) {
                if (pass == 1) {
                    if ((wd != 0 && wdn != 0) || !(fabs(f0) > 1.0e-8)) break;
                    if (wd_in_el == 0) mode = (f0 > 0.0) ? 1 : (role ? 0 : 2);
                    else mode = (f0 < 0.0) ? 3 : (role ? 4 : 0);
                    if (mode == 0) break;
                }
                const double* pi_ = tb.pe[Li][I];
                const double* px_ = tb.pe[Lx][NEGP - 1 - I];
                const int si = reread(si0), sx = reread(sx0);
                // reflection: the wet side's own state against its mirror image
                const bool m1 = mode == 1, m3 = mode == 3;
                double ti[4], te[4];
                edge_point<DOF>(stg, ns, m1 ? sx : si, m1 ? px_ : pi_, ti);
                edge_point<DOF>(stg, ns, m3 ? si : sx, m3 ? pi_ : px_, te);
                const double sf_in = m1 ? sx_ : si_, sf_ex = m3 ? si_ : sx_;
                if (m1 || m3) {
                    const double tx = -ny, ty = nx;
                    const double qn = ti[1] * nx + ti[2] * ny, qt = ti[1] * tx + ti[2] * ty;
                    const double qnm = -qn, qtm = qt;
                    const double den = (nx * ty - ny * tx);
                    const double mqx = (ty * qnm - ny * qtm) / den;
                    const double mqy = (-tx * qnm + nx * qtm) / den;
                    ti[1] = m1 ? mqx : ti[1]; ti[2] = m1 ? mqy : ti[2];
                    te[1] = m1 ? te[1] : mqx; te[2] = m1 ? te[2] : mqy;
                }
                double r0, r1, r2;
                llf<NL>(ph, ti[0], te[0], ti[1], te[1], ti[2], te[2], ti[3], te[3], sf_in, sf_ex, nx, ny,
                        mode == 2 || mode == 4 ? 0.0 : ph.g, r0, r1, r2);
                // reflection: F0 and the wet side's momentum from the reflected flux, zero for the dry
                // side; zero gravity: the momentum alone
                const bool keep = m1 ? role != 0 : (m3 ? role == 0 : true);
                f0 = mode == 2 || mode == 4 ? f0 : r0;
                f1 = keep ? r1 : 0.0;
                f2 = keep ? r2 : 0.0;
            }
#pragma unroll
            for (int j = 0; j < NEGP; j++)
                if (j == I) { F[0][j] = 2.0 * f0; F[1][j] = 2.0 * f1; F[2][j] = 2.0 * f2; }
        }
    }
    const double edh = 0.5 * edfs;       // F is twice the flux
#pragma unroll
    for (int I = 0; I < NEGP; I++) {
        const double* eq = tb.eq[L][role ? NEGP - 1 - I : I];
#pragma unroll
        for (int k = 0; k < DOF; k++) {
            // the sums start from zero: 0 + x == x for every x but -0, so the first point's terms
            // start them
            const double ws = edh * eq[k];
#pragma unroll
            for (int f = 0; f < 3; f++) acc[f][k] = I == 0 ? ws * F[f][I] : acc[f][k] + ws * F[f][I];
        }
    }
}

// Number of an element's boundary sides: they are its first slots.
__device__ __forceinline__ int boundary_slots(int info) {
    return (((info >> 3) & 3) != SIDE_INTERNAL) + (((info >> 10) & 3) != SIDE_INTERNAL) + (((info >> 17) & 3) != SIDE_INTERNAL);
}

// The boundary sides (slots 0..nbd-1) of a wet element: their RHS terms accumulate point after point, as
// the reference's boundary routines do.  acc is set.
template <int P, bool SPH, bool NL>
__device__ __forceinline__ void boundary_sides(const StageArgs& a, const DevTables& T,
                                               const EdgeTables<(P + 1) * (P + 2) / 2, P + 2>& tb, const double* stg,
                                               int ne, int ec, int le, int info, int nbd, double h0,
                                               double (&acc)[3][(P + 1) * (P + 2) / 2]) {
    constexpr int DOF = (P + 1) * (P + 2) / 2, NEGP = P + 2;
    const ElemData& E = a.ed;
    const Phys& ph = a.ph;
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) acc[f][k] = 0.0;
#pragma unroll 1
    for (int s = 0; s < nbd; s++) {
        const int bits = side_bits(info, s);
        const int L = bits & 3, role = (bits >> 2) & 1, kind = (bits >> 3) & 3;
        const int nb = at(E.snbr + (size_t)s * ne, ec);
        const double nx = at(E.geo + (size_t)(3 * s) * ne, ec), ny = at(E.geo + (size_t)(3 * s + 1) * ne, ec);
        const double tx = -ny, ty = nx;
        double xlen, AREAS;
        side_xlen_areas(E, ne, ec, L, role, xlen, AREAS);
#pragma unroll 1
        for (int I = 0; I < NEGP; I++) {
            const double* pv = tb.pe[L][I];
            double t[4];
            edge_point<DOF>(stg, a.ns, reread(le), pv, t);
            const double ze_in = t[0], qx_in = t[1], qy_in = t[2], hb_in = t[3];
            const double sf = SPH ? at(E.sfs + ((size_t)s * NEGP + I) * ne, ec) : 1.0;
            // exterior values: a land side mirrors the normal flow, an ocean side takes the prescribed
            // elevation, a flux side the prescribed normal flow
            double ze_ex = ze_in, qx_ex = qx_in, qy_ex = qy_in;
            if (kind == SIDE_LAND) {
                const double qn_int = qx_in * nx + qy_in * ny, qt_int = qx_in * tx + qy_in * ty;
                const double qn_ext = -qn_int, qt_ext = qt_int;
                const double den = 1.0 / (nx * ty - ny * tx);
                qx_ex = (ty * qn_ext - ny * qt_ext) * den;
                qy_ex = (-tx * qn_ext + nx * qt_ext) * den;
            } else if (kind == SIDE_OCEAN) {
                ze_ex = 0.0;
                const double xe = T.xegp[I];
                // the constituents' endpoint terms EMO*RFF*COS(ARGJ-EFA) of this stage (tide_kernel)
                for (int jj = 0; jj < a.fo.nbfr; jj++) {
                    const size_t o = ((size_t)nb * a.fo.nbfr + jj) * 2;
                    const double z1 = a.fo.tz[(size_t)a.irk * a.fo.tzn + o];
                    const double z2 = a.fo.tz[(size_t)a.irk * a.fo.tzn + o + 1];
                    ze_ex = ze_ex + (0.5 * (z1 + z2) + 0.5 * (z2 - z1) * xe);
                }
                if ((ze_ex * ph.ifnlfa + hb_in) <= 0) ze_ex = fabs(hb_in) + h0;
            } else {
                // the specified normal flux at this point (flow_kernel); the reference forms the
                // exterior momentum after every constituent, so the last, full sum is what counts
                const double qn_ext = a.fo.fz[(size_t)a.irk * a.fo.fzn + (size_t)nb * NEGP + I];
                const double qt_ext = 0.0;
                qx_ex = -(ty * qn_ext - ny * qt_ext) / (nx * ty - ny * tx);
                qy_ex = -(-tx * qn_ext + nx * qt_ext) / (nx * ty - ny * tx);
            }
            double f0, f1, f2;
            llf<NL>(ph, ze_in, ze_ex, qx_in, qx_ex, qy_in, qy_ex, hb_in, hb_in, sf, sf, nx, ny, ph.g, f0, f1, f2);
#pragma unroll
            for (int k = 0; k < DOF; k++) {
                const double w = 2.0 * T.m_inv[k] / AREAS * xlen * pv[k] * T.wegp[I];
                acc[0][k] = acc[0][k] - w * f0;
                acc[1][k] = acc[1][k] - w * f1;
                acc[2][k] = acc[2][k] - w * f2;
            }
        }
    }
}

// What an element's area points share.
struct VolumeTerms {
    double drdx, dsdx, drdy, dsdy;       // Jacobian
    double dpx1, dpy1, dpx2, dpy2;       // gradients of the linear modes
    double dhbx, dhby;                   // gradient of the P1 bathymetry
    double mw[8];                        // MET: vertex wind stresses (x, then y), pressure gradient
    double tdx, tdy, tramp;              // tidal potential gradient and ramp
    double hybf;                         // hybrid friction factor
    double cori, nbar;                   // Coriolis, element-mean Manning n
    double cf, fric, dtdph;              // the scenario's CF, uniform friction and 1/DT
};

template <int P, bool MET, bool NL>
__device__ __forceinline__ void volume_terms(const StageArgs& a, const DevTables& T, int ne, int ec, int sid, int row,
                                             double ze1, const double hb[3], VolumeTerms& v) {
    const ElemData& E = a.ed;
    const Phys& ph = a.ph;
    const double drpsi[3] = {-1.0 / 2.0, 1.0 / 2.0, 0.0}, dspsi[3] = {-1.0 / 2.0, 0.0, 1.0 / 2.0};
    // wind stress at the element's vertices and the pressure gradient sums (MET)
    if (MET) {
        // nodal WSX2/WSY2/PR2 of this stage (src/met_forcing.F:507-509) and the QP-independent sums
        // PR2(Ni)*DPSIDX(i) of src/rhs_dg_hydro.F:117-122,366-372
        const double4* st = a.mt.st + (size_t)a.irk * a.mt.np;
        double pdx = 0.0, pdy = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const double4 s = st[at(E.nm + (size_t)i * ne, ec)];
            v.mw[i] = s.x;
            v.mw[3 + i] = s.y;
            const double pr = s.z;
            const double dpsidx = drpsi[i] * v.drdx + dspsi[i] * v.dsdx;
            const double dpsidy = drpsi[i] * v.drdy + dspsi[i] * v.dsdy;
            if (i == 0) { pdx = pr * dpsidx; pdy = pr * dpsidy; }
            else { pdx = pdx + pr * dpsidx; pdy = pdy + pr * dpsidy; }
        }
        v.mw[6] = pdx;
        v.mw[7] = pdy;
    }
    // tidal potential (src/rhs_dg_hydro.F:117-122,378-386): the sums DPSIDX(i)*TIP2(Ni) are the same
    // at every area point; RAMPDG multiplies them once more at each point
    v.tdx = 0.0; v.tdy = 0.0; v.tramp = 0.0;
    if (a.tip) {
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const double tv = a.tip[at(E.nm + (size_t)i * ne, ec)];
            const double dpsidx = drpsi[i] * v.drdx + dspsi[i] * v.dsdx;
            const double dpsidy = drpsi[i] * v.drdy + dspsi[i] * v.dsdy;
            if (i == 0) { v.tdx = dpsidx * tv; v.tdy = dpsidy * tv; }
            else { v.tdx = v.tdx + dpsidx * tv; v.tdy = v.tdy + dpsidy * tv; }
        }
        v.tramp = a.fo.ramp[(size_t)sid * a.fo.rows + row];
    }
    // hybrid friction factor (1 + (HBREAK/H_c)^FTHETA)^(FGAMMA/FTHETA) from the element-mean depth
    // (src/rhs_dg_hydro.F:306-309): the same at every area point, evaluated once and only when the
    // hybrid law is on
    v.hybf = 1.0;
    if (ph.ifhybf == 1) {
        const double depth_c = hb[0] + ze1;
        const double fh_nl_c = NL ? 1.0 / depth_c : 1.0 / (ph.nleq * depth_c + ph.leq);
        v.hybf = pow(1.0 + pow(ph.hbreak * fh_nl_c, ph.ftheta), ph.fgamma / ph.ftheta);
    }
    // gradients of the linear modes, whose reference derivatives are (0, 0), (0, 3/2), (1, 1/2) at every
    // area point (checked at set-up): products by 0, 1 and 1/2 are exact, so the fused sum rounds as the
    // separate one; with them the P1 bathymetry's gradient
    v.dpx1 = 1.5 * v.dsdx; v.dpy1 = 1.5 * v.dsdy;
    v.dpx2 = __builtin_fma(0.5, v.dsdx, v.drdx); v.dpy2 = __builtin_fma(0.5, v.dsdy, v.drdy);
    v.dhbx = hb[1] * v.dpx1 + hb[2] * v.dpx2;
    v.dhby = hb[1] * v.dpy1 + hb[2] * v.dpy2;
}

// Fluxes and sources of a wet element at area point I (RHS_DG_HYDRO): q = fx fy gx gy hx hy sx sy.
template <int P, bool MET, bool NL>
__device__ __forceinline__ void area_point(const StageArgs& a, const DevTables& T, int I,
                                           const VolumeTerms& v, double ze, double qx, double qy, double hbq, double sfq,
                                           int wd, double (&q)[8]) {
    const Phys& ph = a.ph;
    const double depth = ze + hbq;
    // with NL (NLEQ = 1, LEQ = 0) the constant factors fold exactly
    const double f1 = NL ? 1.0 : ph.nleq + ph.leq * hbq;
    const double fx = NL ? qx * sfq : qx * f1 * sfq, fy = NL ? qy : qy * f1;
    const double fu = NL ? qx : ph.nleq * qx, fv = NL ? qy : ph.nleq * qy;
    const double fg = ph.nleqg * ze * wd;
    const double fh = NL ? 1.0 / depth : 1.0 / (ph.nleq * depth + ph.leq);
    const double u = qx * fh, w = qy * fh;
    const double huu = fu * u, hvv = fv * w, huv = fu * w;
    const double gh2 = NL ? fg * (0.5 * ze + hbq) : fg * (0.5 * ze + hbq) + ph.fg_l * ze;
    double fric = v.fric;
    if (ph.load_manning) {
        // DEPTH**(1.D0/3.D0) (src/rhs_dg_hydro.F:302), correctly rounded
        fric = ph.g * (v.nbar * v.nbar) / crm::cr_pow_third(depth);
        if (fric < v.cf) fric = v.cf;
    }
    double tau = fric;
    if (ph.iflinbf == 0) {
        const double umag = sqrt(u * u + w * w);
        tau = tau * umag * fh;
        if (ph.ifhybf == 1) tau = tau * v.hybf;
        const double cap = 0.9 * v.dtdph;
        if (cap < tau) tau = cap;
    }
    double sx = -(tau * qx) + fg * v.dhbx * sfq + v.cori * qy;
    double sy = -(tau * qy) + fg * v.dhby - v.cori * qx;
    if (MET) {
        // wind stress and atmospheric pressure (src/rhs_dg_hydro.F:362-373)
        const double* ps = T.psi[I];
        const double wsx = v.mw[0] * ps[0] + v.mw[1] * ps[1] + v.mw[2] * ps[2];
        const double wsy = v.mw[3] * ps[0] + v.mw[4] * ps[1] + v.mw[5] * ps[2];
        const double fw = 1.0 / f1;
        sx = sx + (NL ? wsx : fw * wsx) - ph.g * sfq * depth * v.mw[6];
        sy = sy + (NL ? wsy : fw * wsy) - ph.g * depth * v.mw[7];
    }
    if (a.tip) {
        sx = sx + v.tramp * ph.g * depth * sfq * v.tdx;
        sy = sy + v.tramp * ph.g * depth * v.tdy;
    }
    q[0] = fx; q[1] = fy;
    q[2] = (huu + gh2) * sfq; q[3] = huv;
    q[4] = huv * sfq; q[5] = hvv + gh2;
    q[6] = sx; q[7] = sy;
}

// The staged element le's values at area point I (PHI_AREA of mode 1 is 1, checked at set-up, so the sums
// start at mode 1).  At p=1 the point's values are compile-time constants; mode 2's are powers of two, whose
// products are exact, so product and sum fuse without a change, and mode 3's is zero at the first point.
template <int P>
__device__ __forceinline__ void area_values(const DevTables& T, const double* stg, int ns, int le, int I, double (&t)[4]) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
#pragma unroll
    for (int f = 0; f < 4; f++) {
        t[f] = stg[f * DOF * ns + le];
        if constexpr (P == 1) {
            const double p1 = I == 0 ? P1Area::phi[0][1] : P1Area::phi[1][1];
            const double p2 = I == 1 ? P1Area::phi[1][2] : P1Area::phi[2][2];
            t[f] = __builtin_fma(stg[(f * DOF + 1) * ns + le], p1, t[f]);
            if (I > 0) t[f] = t[f] + stg[(f * DOF + 2) * ns + le] * p2;
        } else {
#pragma unroll
            for (int k = 1; k < (f < 3 ? DOF : 3); k++) t[f] = t[f] + stg[(f * DOF + k) * ns + le] * T.phi_area[I][k];
        }
    }
}

// One element's state and vertex depths.
template <int DOF>
__device__ __forceinline__ void load_entry(const double* __restrict__ u, const double* __restrict__ dpv, int ne, int g,
                                           double (&v)[3 * DOF + 3]) {
#pragma unroll
    for (int f = 0; f < 3 * DOF; f++) v[f] = at(u + (size_t)f * ne, g);
#pragma unroll
    for (int m = 0; m < 3; m++) v[3 * DOF + m] = at(dpv + (size_t)m * ne, g);
}

// Stages one element: its state v[0..3*DOF), the P1 bathymetry modes formed from its vertex depths
// v[3*DOF..], its wet/dry flag.
template <int DOF>
__device__ __forceinline__ void stage_entry(double* stg, uint8_t* stwd, int ns, int j, const double (&v)[3 * DOF + 3],
                                            uint8_t w) {
    const double c13 = 1.0 / 3.0, c16 = 1.0 / 6.0;
#pragma unroll
    for (int f = 0; f < 3 * DOF; f++) stg[f * ns + j] = v[f];
    const double d0 = v[3 * DOF], d1 = v[3 * DOF + 1], d2 = v[3 * DOF + 2];
    stg[(3 * DOF) * ns + j] = c13 * (d0 + d1 + d2);
    stg[(3 * DOF + 1) * ns + j] = -(c16 * (d0 + d1)) + c13 * d2;
    stg[(3 * DOF + 2) * ns + j] = -(0.5 * d0) + 0.5 * d1;
    stwd[j] = w;
}

// One lane per element.  What bounds it: FP64 instruction issue (2130 VALU instructions per element at p=1,
// a wave each 4 cycles; the reciprocals and inverse square roots of the fluxes 16) and the latency of three phases
// of loads (staging, quadrature, RK base), which the other waves on the SIMD have to cover.  So registers, which
// set how many waves there are, matter as much as instructions:
//   * the rare paths (dry sides, boundary sides) read the modes from LDS again at every point instead of holding
//     them, the side sums live in registers instead of LDS, and one side's traces are formed after the other's:
//     166 registers at p=1 (226 before), three waves per SIMD instead of two; 251 at p=2 (293 and accumulator
//     registers before), two instead of one;
//   * the spherical and the linearised p=1 variants would spill at three waves (16 storm basins of 438k elements 94 us
//     against 78 us per launch; linearised 796,320 elements 125 and 99 us, 118,933 31 and 26 us), so they keep two;
//   * loads go out early: a tile's halo indices lie at a fixed stride (no look-up first), the next side's geometry
//     is loaded while a side is evaluated, the quadrature's data before the sides and the RK base before the
//     quadrature (which stood still for two thirds of its time when its loads waited behind the RK base).
// Time per launch, 997,306 elements, p=1, limiter and wet/dry: 129 us before, 91 us with these and the shorter
// arithmetic of llf_flux_nl2 and cr_pow_third (33.2M VALU instructions instead of 44.1M); 298,579 elements, p=2:
// 121 us before, 86 us.
template <int P, int NT, bool SPH, bool WDFUSED, bool MET, bool NL>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(P == 1 && !SPH && NL ? 3 : 2))) stage_kernel(StageArgs a) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    constexpr int NAGP = (P == 1) ? 3 : 6;
    constexpr int NEGP = P + 2;
    __shared__ EdgeTables<DOF, NEGP> tb;
    // staged states: rows [field*DOF + mode] then the three bathymetry modes, ns entries each, then
    // the wet/dry flags (bytes)
    extern __shared__ double stg[];
    const DevTables& T = tab<P>();
    const ElemData& E = a.ed;
    const Phys& ph = a.ph;
    const int ne = E.ne;
    const int tid = threadIdx.x;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int e = tile * NT + tid;
    const int ns = a.ns;
    uint8_t* const stwd = reinterpret_cast<uint8_t*>(stg + (size_t)(3 * DOF + 3) * ns);
    load_edge_tables<DOF, NEGP>(T, tb, tid, NT);
    // per-element loads that do not depend on the staged data, issued before the staging loads so
    // that the latencies overlap (lanes past the last element read element ne-1 and exit after
    // the barrier)
    const int ec = e < ne ? e : ne - 1;
    // the first side's NX, NY, XLEN/AREAS; each further side's are loaded while the one before it is
    // evaluated
    double nx = at(E.geo, ec), ny = E.geo[(size_t)ne + ec], edfac = at(E.geo + (size_t)2 * ne, ec);
    const int info = at(E.sinfo, ec);
    const int sl = at(a.snbl, ec);
    {
        // this tile's elements and its halo: the first halo entry's index, then the tile's own loads, then
        // the halo's, before any is used (a halo past NT entries is staged after them)
        const int* hx = a.hidx + (size_t)tile * a.nh;
        const int nh = a.nh;
        const int g = tid < nh ? hx[tid] : -1;
        double v[3 * DOF + 3], v2[3 * DOF + 3];
        load_entry<DOF>(a.uin, E.dpv, ne, ec, v);
        const uint8_t w = at(a.wd_in, ec);
        const int gc = g < 0 ? 0 : g;
        load_entry<DOF>(a.uin, E.dpv, ne, gc, v2);
        const uint8_t w2 = at(a.wd_in, gc);
        stage_entry<DOF>(stg, stwd, ns, tid, v, w);
        if (g >= 0) stage_entry<DOF>(stg, stwd, ns, NT + tid, v2, w2);
#pragma unroll 1
        for (int h = tid + NT; h < nh; h += NT) {
            const int gh = hx[h];
            if (gh < 0) break;
            load_entry<DOF>(a.uin, E.dpv, ne, gh, v);
            stage_entry<DOF>(stg, stwd, ns, NT + h, v, at(a.wd_in, gh));
        }
    }
    __syncthreads();
    if (e >= ne) return;
    const int row = table_step(a.fo) * a.fo.nrk + a.irk;
    const int wd = stwd[tid];
    const int sid = E.sid ? (int)at(E.sid, e) : 0;

    // the Jacobian and Manning's n of the volume quadrature, loaded while the sides are evaluated
    const double jac0 = at(E.geo + (size_t)9 * ne, e), jac1 = at(E.geo + (size_t)10 * ne, e);
    const double jac2 = at(E.geo + (size_t)11 * ne, e), jac3 = at(E.geo + (size_t)12 * ne, e);
    const double nbar0 = ph.load_manning ? at(E.nbar, e) : 0.0;
    // ---- sides: the internal ones in slot order, then the boundary ones (a sum of the two, whose
    // order of evaluation does not matter): RHS = RHS(boundary edges) + slot sum
    double R[3][DOF];
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) R[f][k] = 0.0;
    const int nbd = boundary_slots(info);
#pragma unroll 1
    for (int slot = 0; slot < 3; slot++) {
        double nx1 = nx, ny1 = ny, ed1 = edfac;
        if (slot < 2) {
            nx1 = at(E.geo + (size_t)(3 * slot + 3) * ne, e);
            ny1 = at(E.geo + (size_t)(3 * slot + 4) * ne, e);
            ed1 = at(E.geo + (size_t)(3 * slot + 5) * ne, e);
        }
        if (slot >= nbd) {
            double acc[3][DOF];
            internal_side<P, SPH, NL, 1>(a, tb, stg, stwd, ne, e, tid, slot, side_bits(info, slot), sl, wd, nx, ny, edfac, acc);
#pragma unroll
            for (int f = 0; f < 3; f++)
#pragma unroll
                for (int k = 0; k < DOF; k++) R[f][k] = R[f][k] + acc[f][k];
        }
        nx = nx1; ny = ny1; edfac = ed1;
    }
    if (nbd != 0 && wd != 0) {
        double acc[3][DOF];
        boundary_sides<P, SPH, NL>(a, T, tb, stg, ne, e, tid, info, nbd, E.scen[sid].h0, acc);
#pragma unroll
        for (int f = 0; f < 3; f++)
#pragma unroll
            for (int k = 0; k < DOF; k++) R[f][k] = acc[f][k] + R[f][k];
    }

    // the scenario's scalars, then the first RK base state, loaded before the volume quadrature's arithmetic
    double dtdp, dtdph, cf, fric, rain;
    VolumeTerms v;
    if (E.sid) {
        const Scen& sc = E.scen[sid];
        dtdp = sc.dtdp; dtdph = sc.dtdph; cf = sc.cf; fric = sc.fric; rain = sc.rain; v.cori = sc.cori;
    } else {
        const Scen& sc = E.scen[0];
        dtdp = sc.dtdp; dtdph = sc.dtdph; cf = sc.cf; fric = sc.fric; rain = sc.rain; v.cori = sc.cori;
    }
    if (E.cori_el) v.cori = at(E.cori_el, e);
    double sfqv[NAGP];
#pragma unroll
    for (int I = 0; I < NAGP; I++) sfqv[I] = SPH ? at(E.sfacq + (size_t)I * ne, e) : 1.0;
    const bool pre0 = a.nprev > 0 && a.aprev[0] != 0.0;
    double B0[3][DOF];
    if (pre0) {
        const double* up = a.uprev[0];
#pragma unroll
        for (int f = 0; f < 3; f++)
#pragma unroll
            for (int k = 0; k < DOF; k++) B0[f][k] = at(up + (size_t)(f * DOF + k) * ne, e);
    }
    // ---- volume quadrature (RHS_DG_HYDRO)
    if (rain > 0.0) {
#pragma unroll 1
        for (int I = 0; I < NAGP; I++)
#pragma unroll
            for (int k = 0; k < DOF; k++) R[0][k] = R[0][k] + T.srfac[I][k] * rain;
    }
    if (wd != 0) {
        v.drdx = jac0; v.dsdx = jac1; v.drdy = jac2; v.dsdy = jac3; v.nbar = nbar0;
        v.dtdph = dtdph; v.cf = cf; v.fric = fric;
        {
            const double hb[3] = {stg[3 * DOF * ns + tid], stg[(3 * DOF + 1) * ns + tid], stg[(3 * DOF + 2) * ns + tid]};
            volume_terms<P, MET, NL>(a, T, ne, e, sid, row, stg[tid], hb, v);
        }
        // p=1: the three area points unrolled, with the quadrature's constants in the code and the factors
        // MW*DPSI formed once (the same at every point, checked at set-up); at p=2 the six points in a loop
        double xf1[3], yf1[3];
        if constexpr (P == 1) {
            xf1[1] = P1Area::mw[1] * v.dpx1; yf1[1] = P1Area::mw[1] * v.dpy1;
            xf1[2] = P1Area::mw[2] * v.dpx2; yf1[2] = P1Area::mw[2] * v.dpy2;
        }
#pragma unroll(P == 1 ? NAGP : 1)
        for (int I = 0; I < NAGP; I++) {
            double t[4], q[8];
            area_values<P>(T, stg, ns, tid, I, t);
            area_point<P, MET, NL>(a, T, I, v, t[0], t[1], t[2], t[3], sfqv[I], wd, q);
            const double sr0 = P == 1 ? P1Area::srfac[I][0] : T.srfac[I][0];
            R[1][0] = R[1][0] + sr0 * q[6];
            R[2][0] = R[2][0] + sr0 * q[7];
#pragma unroll
            for (int k = 1; k < DOF; k++) {
                double xf, yf, sr;
                if constexpr (P == 1) {
                    xf = xf1[k]; yf = yf1[k]; sr = P1Area::srfac[I][k];
                } else {
                    const double dpxk = k == 1 ? v.dpx1 : (k == 2 ? v.dpx2 : T.drphi[I][k] * v.drdx + T.dsphi[I][k] * v.dsdx);
                    const double dpyk = k == 1 ? v.dpy1 : (k == 2 ? v.dpy2 : T.drphi[I][k] * v.drdy + T.dsphi[I][k] * v.dsdy);
                    xf = T.mw[I][k] * dpxk; yf = T.mw[I][k] * dpyk; sr = T.srfac[I][k];
                }
                R[0][k] = R[0][k] + xf * q[0] + yf * q[1];
                R[1][k] = R[1][k] + xf * q[2] + yf * q[3];
                R[2][k] = R[2][k] + xf * q[4] + yf * q[5];
                if (P != 1 || I > 0 || k < 2) {     // p=1: SRFAC of mode 3 is zero at the first point
                    R[1][k] = R[1][k] + sr * q[6];
                    R[2][k] = R[2][k] + sr * q[7];
                }
            }
        }
    }
    // ---- SSP-RK update U(IRK+1) = sum_I ATVD(IRK,I) U(I) + BTVD(IRK,I) DT RHS(I)
    if (a.rout) {
#pragma unroll
        for (int f = 0; f < 3; f++)
#pragma unroll
            for (int k = 0; k < DOF; k++) at(a.rout + (size_t)(f * DOF + k) * ne, e) = R[f][k];
    }
    double W[3][DOF];
    const double bcur = a.bcur * dtdp;
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) W[f][k] = 0.0;
#pragma unroll 1
    for (int i = 0; i < a.nprev; i++) {
        const double ai = a.aprev[i], bi = a.bprev[i] * dtdp;
        if (i == 0 && pre0) {
#pragma unroll
            for (int f = 0; f < 3; f++)
#pragma unroll
                for (int k = 0; k < DOF; k++) W[f][k] = W[f][k] + ai * B0[f][k];
        } else if (ai != 0.0) {
            const double* up = a.uprev[i];
#pragma unroll
            for (int f = 0; f < 3; f++)
#pragma unroll
                for (int k = 0; k < DOF; k++) W[f][k] = W[f][k] + ai * at(up + (size_t)(f * DOF + k) * ne, e);
        }
        if (bi != 0.0) {
            const double* rp = a.rprev[i];
#pragma unroll
            for (int f = 0; f < 3; f++)
#pragma unroll
                for (int k = 0; k < DOF; k++) W[f][k] = W[f][k] + bi * at(rp + (size_t)(f * DOF + k) * ne, e);
        }
    }
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) W[f][k] = W[f][k] + a.acur * stg[(f * DOF + k) * ns + tid] + bcur * R[f][k];

    if (WDFUSED) {
        const double D[3] = {E.dpv[e], E.dpv[(size_t)ne + e], E.dpv[2 * (size_t)ne + e]};
        const double hb[3] = {stg[3 * DOF * ns + tid], stg[(3 * DOF + 1) * ns + tid], stg[(3 * DOF + 2) * ns + tid]};
        const double h0 = E.scen[sid].h0;
        const double dpe_min = fmin(fmin(D[0], D[1]), D[2]);
        if (a.wd_active && !wetdry_keeps<P>(T, W, D, wd, h0)) a.wd_active[0] = 1;
        const int nw = wetdry_element<P>(T, W, D, hb, dpe_min, wd, h0);
        at(a.wd_out, e) = (uint8_t)nw;
    }
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) at(a.uout + (size_t)(f * DOF + k) * ne, e) = W[f][k];
    if (a.wout) {
#pragma unroll
        for (int f = 0; f < 3; f++)
#pragma unroll
            for (int k = 0; k < DOF; k++) at(a.wout + (size_t)(f * DOF + k) * ne, e) = W[f][k];
    }
    if (a.cmout) {
#pragma unroll
        for (int f = 0; f < 3; f++) at(a.cmout + (size_t)f * ne, e) = W[f][0];
    }
}

// The same stage for meshes too small to fill the chip with one lane per element, where the time of a launch is
// the serial chain of its slowest wave: a block of four waves works on 64 elements, lane l of every wave on
// element l.  Wave c < 3
//   1. stages field c of the tile and its halo (wave 3: the flags and the edge tables),
//   2. evaluates side slot c if it is internal (wave 3: the boundary sides, one after the other),
//   3. evaluates the area points c, c+3,
//   4. sums field c's right-hand side in the reference's order from what the waves left in LDS, and updates
//      field c.
// Every value is formed by the operations of stage_kernel, so the results are the same bits.
constexpr int SPLIT_NT = 64;             // elements per block
constexpr int split_rows(int dof, int nagp) { return 4 * 3 * dof + 8 * nagp; }

template <int P, bool SPH, bool WDFUSED, bool MET>
__global__ void __launch_bounds__(4 * SPLIT_NT) __attribute__((amdgpu_waves_per_eu(2))) stage_split_kernel(StageArgs a) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    constexpr int NAGP = (P == 1) ? 3 : 6;
    constexpr int NEGP = P + 2;
    constexpr int NT = SPLIT_NT;
    __shared__ EdgeTables<DOF, NEGP> tb;
    // exchange between an element's lanes: the sums of the side slots and of the boundary sides
    // [wave*3*DOF + field*DOF + mode], then the area points' values [point*8 + quantity]; with WDFUSED last
    // the updated modes
    __shared__ double xch[split_rows(DOF, NAGP)][NT];
    extern __shared__ double stg[];      // as in stage_kernel
    const DevTables& T = tab<P>();
    const ElemData& E = a.ed;
    const Phys& ph = a.ph;
    const int ne = E.ne;
    const int c = __builtin_amdgcn_readfirstlane(threadIdx.x / NT), le = threadIdx.x % NT;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int e = tile * NT + le;
    const bool valid = e < ne;
    const int ns = a.ns, nh = a.nh;
    uint8_t* const stwd = reinterpret_cast<uint8_t*>(stg + (size_t)(3 * DOF + 3) * ns);
    double* const vol = &xch[4 * 3 * DOF][0];
    const int ec = valid ? e : ne - 1;   // lanes past the last element read element ne-1 and write nothing
    const int* hx = a.hidx + (size_t)tile * nh;
    const int g0 = le < nh ? hx[le] : -1;
    const int info = at(E.sinfo, ec);
    const int sl = at(a.snbl, ec);
    const int sid = E.sid ? (int)at(E.sid, ec) : 0;
    const int cs = c < 3 ? c : 0;
    const double nx = at(E.geo + (size_t)(3 * cs) * ne, ec), ny = at(E.geo + (size_t)(3 * cs + 1) * ne, ec);
    const double edfac = at(E.geo + (size_t)(3 * cs + 2) * ne, ec);
    if (c < 3) {
        const double c13 = 1.0 / 3.0, c16 = 1.0 / 6.0;
        auto load = [&](int g, double (&v)[DOF + 3]) {
#pragma unroll
            for (int k = 0; k < DOF; k++) v[k] = at(a.uin + (size_t)(c * DOF + k) * ne, g);
#pragma unroll
            for (int m = 0; m < 3; m++) v[DOF + m] = at(E.dpv + (size_t)m * ne, g);
        };
        auto store = [&](int j, const double (&v)[DOF + 3]) {
#pragma unroll
            for (int k = 0; k < DOF; k++) stg[(c * DOF + k) * ns + j] = v[k];
            const double d0 = v[DOF], d1 = v[DOF + 1], d2 = v[DOF + 2];
            stg[(3 * DOF + c) * ns + j] = c == 0 ? c13 * (d0 + d1 + d2)
                                                 : (c == 1 ? -(c16 * (d0 + d1)) + c13 * d2 : -(0.5 * d0) + 0.5 * d1);
        };
        double v[DOF + 3], v2[DOF + 3];
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
    } else {
        load_edge_tables<DOF, NEGP>(T, tb, le, NT);
        const uint8_t w = at(a.wd_in, ec), w2 = at(a.wd_in, g0 < 0 ? 0 : g0);
        stwd[le] = w;
        if (g0 >= 0) stwd[NT + le] = w2;
#pragma unroll 1
        for (int h = le + NT; h < nh; h += NT) {
            const int g = hx[h];
            if (g < 0) break;
            stwd[NT + h] = at(a.wd_in, g);
        }
    }
    // loads of the volume quadrature and the RK update, under way while the sides are evaluated
    const int row = table_step(a.fo) * a.fo.nrk + a.irk;
    constexpr int NP = NAGP / 3;           // area points per wave: c and, at p=2, c + 3
    VolumeTerms v;
    v.drdx = at(E.geo + (size_t)9 * ne, ec); v.dsdx = at(E.geo + (size_t)10 * ne, ec);
    v.drdy = at(E.geo + (size_t)11 * ne, ec); v.dsdy = at(E.geo + (size_t)12 * ne, ec);
    v.nbar = ph.load_manning ? at(E.nbar, ec) : 0.0;
    const Scen& sc = E.scen[sid];
    const double dtdp = sc.dtdp, rain = sc.rain, h0 = sc.h0;
    v.dtdph = sc.dtdph; v.cf = sc.cf; v.fric = sc.fric;
    v.cori = E.cori_el ? at(E.cori_el, ec) : sc.cori;
    double sfqv[NP];
#pragma unroll
    for (int j = 0; j < NP; j++) sfqv[j] = SPH ? at(E.sfacq + (size_t)(cs + 3 * j) * ne, ec) : 1.0;
    const bool pre0 = a.nprev > 0 && a.aprev[0] != 0.0;
    double B0[DOF];
    if (pre0) {
        const double* up = a.uprev[0];
#pragma unroll
        for (int k = 0; k < DOF; k++) B0[k] = at(up + (size_t)(cs * DOF + k) * ne, ec);
    }
    __syncthreads();
    const int wd = valid ? stwd[le] : 0;
    // ---- sides
    const int nbd = boundary_slots(info);
    {
        double acc[3][DOF];
        if (c < 3) {
            // a boundary slot is the boundary wave's; its place in the exchange is not read
            if (c >= nbd && valid)
                internal_side<P, SPH, true, NEGP>(a, tb, stg, stwd, ne, ec, le, c, side_bits(info, c), sl, wd, nx, ny,
                                                  edfac, acc);
        } else if (nbd != 0 && wd != 0) {
            boundary_sides<P, SPH, true>(a, T, tb, stg, ne, ec, le, info, nbd, h0, acc);
        } else {
#pragma unroll
            for (int f = 0; f < 3; f++)
#pragma unroll
                for (int k = 0; k < DOF; k++) acc[f][k] = 0.0;
        }
        if (c == 3 || (c >= nbd && valid)) {
#pragma unroll
            for (int f = 0; f < 3; f++)
#pragma unroll
                for (int k = 0; k < DOF; k++) xch[(c * 3 + f) * DOF + k][le] = acc[f][k];
        }
    }
    // ---- volume quadrature (RHS_DG_HYDRO) at this wave's area points
    {
        const double hb[3] = {stg[3 * DOF * ns + le], stg[(3 * DOF + 1) * ns + le], stg[(3 * DOF + 2) * ns + le]};
        volume_terms<P, MET, true>(a, T, ne, ec, sid, row, stg[le], hb, v);
    }
    if (c < 3 && wd != 0) {
#pragma unroll
        for (int j = 0; j < NP; j++) {
            double t[4], q[8];
            area_values<P>(T, stg, ns, le, c + 3 * j, t);
            area_point<P, MET, true>(a, T, c + 3 * j, v, t[0], t[1], t[2], t[3], sfqv[j], wd, q);
#pragma unroll
            for (int i = 0; i < 8; i++) vol[((c + 3 * j) * 8 + i) * NT + le] = q[i];
        }
    }
    __syncthreads();
    if (c == 3) {
        if (WDFUSED) { __syncthreads(); }
        return;
    }
    // ---- field c: add_internal_flux (RHS of the boundary edges + slot sum), then the volume terms, point after
    // point
    double R[DOF];
#pragma unroll
    for (int k = 0; k < DOF; k++) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++)
            if (i >= nbd) s = s + xch[(i * 3 + c) * DOF + k][le];
        R[k] = xch[(9 + c) * DOF + k][le] + s;
    }
    if (c == 0 && rain > 0.0) {
#pragma unroll 1
        for (int I = 0; I < NAGP; I++)
#pragma unroll
            for (int k = 0; k < DOF; k++) R[k] = R[k] + T.srfac[I][k] * rain;
    }
    if (wd != 0) {
#pragma unroll
        for (int I = 0; I < NAGP; I++) {
            const double fx = vol[(I * 8 + 2 * c) * NT + le], fy = vol[(I * 8 + 2 * c + 1) * NT + le];
            const double s = vol[(I * 8 + 5 + c) * NT + le];            // source of field c > 0
            if (c != 0) R[0] = R[0] + T.srfac[I][0] * s;
#pragma unroll
            for (int k = 1; k < DOF; k++) {
                const double dpxk = k == 1 ? v.dpx1 : (k == 2 ? v.dpx2 : T.drphi[I][k] * v.drdx + T.dsphi[I][k] * v.dsdx);
                const double dpyk = k == 1 ? v.dpy1 : (k == 2 ? v.dpy2 : T.drphi[I][k] * v.drdy + T.dsphi[I][k] * v.dsdy);
                R[k] = R[k] + (T.mw[I][k] * dpxk) * fx + (T.mw[I][k] * dpyk) * fy;
                if (c != 0) R[k] = R[k] + T.srfac[I][k] * s;
            }
        }
    }
    // ---- SSP-RK update U(IRK+1) = sum_I ATVD(IRK,I) U(I) + BTVD(IRK,I) DT RHS(I)
    if (a.rout && valid) {
#pragma unroll
        for (int k = 0; k < DOF; k++) at(a.rout + (size_t)(c * DOF + k) * ne, e) = R[k];
    }
    double W[DOF];
    const double bcur = a.bcur * dtdp;
#pragma unroll
    for (int k = 0; k < DOF; k++) W[k] = 0.0;
#pragma unroll 1
    for (int i = 0; i < a.nprev; i++) {
        const double ai = a.aprev[i], bi = a.bprev[i] * dtdp;
        if (i == 0 && pre0) {
#pragma unroll
            for (int k = 0; k < DOF; k++) W[k] = W[k] + ai * B0[k];
        } else if (ai != 0.0) {
            const double* up = a.uprev[i];
#pragma unroll
            for (int k = 0; k < DOF; k++) W[k] = W[k] + ai * at(up + (size_t)(c * DOF + k) * ne, ec);
        }
        if (bi != 0.0) {
            const double* rp = a.rprev[i];
#pragma unroll
            for (int k = 0; k < DOF; k++) W[k] = W[k] + bi * at(rp + (size_t)(c * DOF + k) * ne, ec);
        }
    }
#pragma unroll
    for (int k = 0; k < DOF; k++) W[k] = W[k] + a.acur * stg[(c * DOF + k) * ns + le] + bcur * R[k];
    if (WDFUSED) {
        // WETDRY needs all three fields: each wave takes the others' from LDS and keeps its own (the rows
        // are the boundary sums', of which wave c alone read field c's)
#pragma unroll
        for (int k = 0; k < DOF; k++) xch[(9 + c) * DOF + k][le] = W[k];
        __syncthreads();
        if (!valid) return;
        double A[3][DOF];
        const double hb[3] = {stg[3 * DOF * ns + le], stg[(3 * DOF + 1) * ns + le], stg[(3 * DOF + 2) * ns + le]};
#pragma unroll
        for (int f = 0; f < 3; f++)
#pragma unroll
            for (int k = 0; k < DOF; k++) A[f][k] = xch[(9 + f) * DOF + k][le];
        const double D[3] = {at(E.dpv, e), at(E.dpv + (size_t)ne, e), at(E.dpv + (size_t)2 * ne, e)};
        const double dpe_min = fmin(fmin(D[0], D[1]), D[2]);
        if (c == 0 && a.wd_active && !wetdry_keeps<P>(T, A, D, wd, h0)) a.wd_active[0] = 1;
        const int nw = wetdry_element<P>(T, A, D, hb, dpe_min, wd, h0);
        if (c == 0) at(a.wd_out, e) = (uint8_t)nw;
#pragma unroll
        for (int k = 0; k < DOF; k++) W[k] = c == 0 ? A[0][k] : (c == 1 ? A[1][k] : A[2][k]);
    }
    if (!valid) return;
#pragma unroll
    for (int k = 0; k < DOF; k++) at(a.uout + (size_t)(c * DOF + k) * ne, e) = W[k];
    if (a.wout) {
#pragma unroll
        for (int k = 0; k < DOF; k++) at(a.wout + (size_t)(c * DOF + k) * ne, e) = W[k];
    }
    if (a.cmout) at(a.cmout + (size_t)c * ne, e) = W[0];
}

// ------------------------------------------------------------------------------------------
// Tidal forcing of a batch of steps at the ocean boundary (src/ocean_edge_hydro.F:459-488): for
// every stage, ocean edge, constituent and end node the term EMO*RFF*COS(ARGJ - EFA) that the edge's
// elevation sums, with the cosine correctly rounded.  One thread per term, one block row per stage;
// the stage kernels read the stage's terms.  A few hundred terms a stage: the launch is bound by the
// latency of one cosine and takes as long for 64 steps as for one, so the boundary, potential and
// storm forcing is formed for several steps at a time (launch_forcing).  100 steps of 4,972 p=1
// elements 3.73 ms with a launch per step, 3.31 ms now; 30 of 59,600 p=2 elements under the
// potential 3.3 and 2.6 ms; 60 of 16 storms in graphs 15.9 and 14.8 ms.
// ------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) tide_kernel(Forcing fo, const uint16_t* __restrict__ osid,
                                                   double* __restrict__ tz) {
    const int o = blockIdx.x * blockDim.x + threadIdx.x;    // (edge*nbfr + jj)*2 + end
    if (o >= fo.tzn) return;
    const int irk = blockIdx.y;                             // stage, counted over the steps of the batch
    const size_t i = (size_t)irk * fo.tzn + o;
    const int jj = (o >> 1) % fo.nbfr, edge = (o >> 1) / fo.nbfr;
    const int sid = osid ? (int)osid[edge] : 0;
    const int row = table_step(fo) * fo.nrk + irk;
    if (fo.ets) {   // non-periodic: the stage's ramped end-node values (nbfr is 1)
        tz[i] = fo.ets[((size_t)sid * fo.rows + row) * fo.tzn + o];
        return;
    }
    const size_t t = ((size_t)sid * fo.rows + row) * fo.nbfr + jj;
    tz[i] = fo.emo[o] * fo.rff[t] * crm::cr_cos(fo.argj[t] - fo.efa[o]);
}

// ------------------------------------------------------------------------------------------
// Specified normal flux of a batch of steps (src/flow_edge_hydro.F:143-173): for every stage, flux edge
// and edge quadrature point Q_N_EXT = sum over constituents of QNAM_GP*RFF*COS(ARGJ - QNPH_GP),
// with the cosine correctly rounded.  For NFFR = 0 the one term has ARGJ = 0, RFF = RAMPDG and the
// end values of the time series (already ramped once, src/DG_hydro_timestep.F:188-195).
// ------------------------------------------------------------------------------------------
template <int P>
__global__ void __launch_bounds__(256) flow_kernel(Forcing fo, const uint16_t* __restrict__ fsid,
                                                   double* __restrict__ fz) {
    constexpr int NEGP = P + 2;
    const DevTables& T = tab<P>();
    const int o = blockIdx.x * blockDim.x + threadIdx.x;    // edge*NEGP + point
    if (o >= fo.fzn) return;
    const int irk = blockIdx.y;                             // stage, counted over the steps of the batch
    const size_t i = (size_t)irk * fo.fzn + o;
    const int edge = o / NEGP, I = o - edge * NEGP;
    const int sid = fsid ? (int)fsid[edge] : 0;
    const int row = table_step(fo) * fo.nrk + irk;
    const double xe = T.xegp[I];
    double qn = 0.0;
    for (int jj = 0; jj < fo.nffr; jj++) {
        const size_t t = ((size_t)sid * fo.rows + row) * fo.nffr + jj;
        const double argj = fo.fargj[t];
        const double rff = fo.frff[t];
        double q1, q2;
        if (fo.qts) {
            const size_t q = (((size_t)sid * fo.rows + row) * fo.nfeds + edge) * 2;
            q1 = fo.qts[q]; q2 = fo.qts[q + 1];
        } else {
            const size_t q = ((size_t)edge * fo.nffr + jj) * 2;
            q1 = fo.qnam[q]; q2 = fo.qnam[q + 1];
        }
        const size_t q = ((size_t)edge * fo.nffr + jj) * 2;
        const double p1 = fo.qnph[q], p2 = fo.qnph[q + 1];
        const double qnam_gp = 0.5 * (q1 + q2) + 0.5 * (q2 - q1) * xe;
        const double qnph_gp = 0.5 * (p1 + p2) + 0.5 * (p2 - p1) * xe;
        qn = qn + qnam_gp * rff * crm::cr_cos(argj - qnph_gp);
    }
    fz[i] = qn;
}

// ------------------------------------------------------------------------------------------
// TIDAL_POTENTIAL (src/tidal_potential.F:15-80) for every stage of a batch of steps: TIP2 at every
// node, with the cosines of the time-dependent arguments correctly rounded (COS(SFEA)**2 and
// SIN(2*SFEA) come from the host's libm).  Without self-attraction and load the second product is
// SALTMUL*0*COS: adding SALTMUL*0 gives the same sum without the cosine (half of the kernel's work).
// ------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) tip_kernel(Tip tp, Forcing fo) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= tp.np) return;
    const int irk = blockIdx.y;                             // stage, counted over the steps of the batch
    const int row = table_step(fo) * fo.nrk + irk;
    const double* r = tp.row + (size_t)row * tp.ntif * 3;
    double tip = 0.0;
    for (int j = 0; j < tp.ntif; j++) {
        const double argt = r[3 * j], tpmul = r[3 * j + 1], saltmul = r[3 * j + 2];
        const int na = tp.na[j];
        if (na != 1 && na != 2) continue;
        double salt = saltmul * 0.0;
        if (tp.salt_amp)
            salt = saltmul * tp.salt_amp[(size_t)j * tp.np + n] * crm::cr_cos(argt - tp.salt_pha[(size_t)j * tp.np + n]);
        if (na == 1) {
            const double argtp = argt + 2.0 * tp.slam[n];
            tip = tip + tpmul * tp.ccsfea[n] * crm::cr_cos(argtp) + salt;
        }
        if (na == 2) {
            const double argtp = argt + tp.slam[n];
            tip = tip + tpmul * tp.s2sfea[n] * crm::cr_cos(argtp) + salt;
        }
    }
    tp.tip2[(size_t)irk * tp.np + n] = tip;
}

// ------------------------------------------------------------------------------------------
// SLOPELIMITER5 part 1 (src/slopelimiter.F:3290-3404): node min/max of the updated cell means.
// nminmax layout [6][np]: zmin zmax qxmin qxmax qymin qymax.
// ------------------------------------------------------------------------------------------
template <int P>
__global__ void __launch_bounds__(256) node_minmax_kernel(int np, int ne, const int* __restrict__ off,
                                                          const int* __restrict__ n2e,
                                                          const double* __restrict__ u,
                                                          double* __restrict__ mm) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    const int n = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (n >= np) return;
    double zmin = 99999., zmax = -99999., xmin = 99999., xmax = -99999., ymin = 99999., ymax = -99999.;
    const int j1 = off[n + 1];
    // up to eight incidences per pass: all their indices, then all their cell means, are loaded
    // before any is used; past the node's last incidence the pass repeats that incidence (min and
    // max are exact and idempotent, so neither the order nor a repeat changes them)
    constexpr int B = 8;
    for (int j = off[n]; j < j1; j += B) {
        int ei[B];
#pragma unroll
        for (int q = 0; q < B; q++) ei[q] = n2e[min(j + q, j1 - 1)] >> 2;
        double z[B], x[B], y[B];
#pragma unroll
        for (int q = 0; q < B; q++) {
            z[q] = u[ei[q]];
            x[q] = u[(size_t)DOF * ne + ei[q]];
            y[q] = u[(size_t)2 * DOF * ne + ei[q]];
        }
#pragma unroll
        for (int q = 0; q < B; q++) {
            zmin = fmin(zmin, z[q]); xmin = fmin(xmin, x[q]); ymin = fmin(ymin, y[q]);
            zmax = fmax(zmax, z[q]); xmax = fmax(xmax, x[q]); ymax = fmax(ymax, y[q]);
        }
    }
    mm[n] = zmin; mm[(size_t)np + n] = zmax; mm[2 * (size_t)np + n] = xmin;
    mm[3 * (size_t)np + n] = xmax; mm[4 * (size_t)np + n] = ymin; mm[5 * (size_t)np + n] = ymax;
}

// ------------------------------------------------------------------------------------------
// SLOPELIMITER5 (src/slopelimiter.F:3290-3676) then WETDRY (src/wetdry.F).
// The node bounds of part 1 are formed per tile in LDS (LimTiles): the tile stages the updated cell
// means of its elements and of its vertex halo, each node of the tile takes the min/max over its
// incident elements, and each element then limits its modes 2-3 against the bounds of its nodes.
// With WETDRY the cell means come from the stage kernel's copy `cmean` [3][ne] (field stride
// cms = ne): WETDRY rewrites some cell means of u in place, which other tiles' halos must not see.
// Without it they are read from u itself (cms = DOF*ne), whose cell means the limiter keeps.
// ------------------------------------------------------------------------------------------
// limit_wetdry_kernel: three waves per 64 elements; wave c stages, bounds and limits field c, so its branches on c are
// uniform.  What bounds it on small meshes is the chain of loads before the first bound: a third of the work per lane
// keeps three times the loads under way, and lists at fixed strides need no look-up before them.  Tiles of 64 use four
// times the compute units of tiles of 256 there (7.4 against 9.0 us at 5k elements).  The modes past the third are
// touched only where WETDRY changes the element.
// Per launch, one lane per element and 256-element tiles before, now: 4,783 elements p=1 9.2 and 4.6 us, 99,015 elements
// p=2 16.3 and 12.0 us.
//
// limit_wide_kernel: a wave per tile, a lane for the three fields of an element.  On large meshes the chip is full
// either way, and what the three waves do three times (the lists, the addresses, the exchange before WETDRY) is time: 1103
// VALU instructions per element, 943 here, for the same bytes (174 per element at p=1).  lim_wide says from how many
// elements on it is the faster form.  Per launch, one lane per element and 256-element tiles before, three waves per
// tile, a wave per tile (us):
//   limiter and WETDRY  p=1  46.6, 52.6, 43.0 at 997,306 elements; 32.3, 31.4, 27.5 at 597,806; 22.0, 19.9, 19.5 at 298,563
//                       p=2  48.6, 39.2, 30.2 at 597,806; 26.7, 21.7, 19.9 at 298,579
//   WETDRY's reverse    p=2  29.9, 48.9, 24.5 at 792,120; 8.8, 9.2, 6.8 at 84,370; 7.2, 5.1, 4.7 at 4,783
//
// With WDADJ (the adjoint's reverse sweep; WETDRY false) the kernel writes nothing to u: each
// element's limited modes, formed exactly as the forward formed them, go to the
// frozen-branch WETDRY reverse of that element (wetdry_adj_element), which turns the cotangent ub
// of WETDRY's output into that of its input and adds the vertex-depth cotangents to gdp.
//
// The launches pass lim_lds() bytes of dynamic LDS.
constexpr int LIM_NT = 64;               // elements per tile
constexpr int lim_lds(int nvh, int nql) {
    return 8 * (3 * (LIM_NT + nvh) + 6 * nql > 9 * LIM_NT ? 3 * (LIM_NT + nvh) + 6 * nql : 9 * LIM_NT) + LIM_NT;
}

// x/3, correctly rounded: the rounded product with 1/3, its exact remainder and one correction (Markstein), in four
// instructions instead of eleven; the fix-up keeps infinities and zeros as a division has them.
__device__ __forceinline__ double div3(double x) {
    const double q = x * (1.0 / 3.0);
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-3.0, q, x), 1.0 / 3.0, q), 3.0, x);
}

// fmin and fmax as one instruction each: of the library's the compiler makes two where it cannot see that an operand
// (one read from memory) is no signalling NaN, which no arithmetic here produces.
__device__ __forceinline__ double min1(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double max1(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// SLOPELIMITER5 of one field of one element: mean c0, linear modes w1 and w2 (in place), its nodes' bounds.
// SIGNDIF is +-1, so products with it are exact: they become sign flips and fuse with the sums after them, and
// DIF > 0 is a comparison of the vertex value with the mean.
__device__ __forceinline__ void limit_field(const DevTables& T, double c0, double& w1, double& w2,
                                            const double (&vmin)[3], const double (&vmax)[3]) {
    double v[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        // the linear modes' corner values are powers of two or zero (checked at set-up): exact products fuse
        const double t = __builtin_fma(T.phi_corner[c][2], w2, __builtin_fma(T.phi_corner[c][1], w1, c0));
        v[c] = max1(min1(t, vmax[c]), vmin[c]);
    }
#pragma unroll
    for (int ll = 0; ll < 3; ll++) {
        const double sumloc = div3(v[0] + v[1] + v[2]);
        double sumdif = (sumloc - c0) * 3.0;
        const int sgn = __double2hiint(sumdif) & 0x80000000;
        const bool up = sgn == 0;
        const double signdif = __hiloint2double(0x3ff00000 | sgn, 0);
        bool d[3];
#pragma unroll
        for (int c = 0; c < 3; c++) d[c] = up ? v[c] > c0 : v[c] < c0;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            // REDFAC = (SUMDIF*SIGNDIF)/DIV with DIV the positive differences not yet passed: at most 3 - k.
            // x/1 and x/2 are x and x*0.5 exactly.
            const double a = __hiloint2double(__double2hiint(sumdif) ^ sgn, __double2loint(sumdif));
            double redfac = a;
            if (k < 2) redfac = (k == 0 ? d[1] || d[2] : d[2]) ? a * 0.5 : a;
            if (k == 0 && d[1] && d[2]) redfac = div3(a);
            redfac = d[k] ? redfac : 0.0;
            redfac = min1(redfac, up ? v[k] - vmin[k] : vmax[k] - v[k]);
            sumdif = __builtin_fma(-redfac, signdif, sumdif);
            v[k] = __builtin_fma(-redfac, signdif, v[k]);
        }
    }
    w1 = -(1.0 / 6.0 * (v[0] + v[1])) + 1.0 / 3.0 * v[2];
    w2 = -(0.5 * v[0]) + 0.5 * v[1];
}

template <int P>
__device__ void wetdry_adj_element(const DevTables& T, const double (&U)[3][3], const double (&D)[3], int wdflg,
                                   double H0, int e, int ne, double* __restrict__ ub, double* __restrict__ gdp);

// Minimum and maximum of the staged means at eight byte offsets.
__device__ __forceinline__ void minmax8(const char* cm, const uint4& r, double& lo, double& hi) {
    const uint32_t p[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const double a = *reinterpret_cast<const double*>(cm + (p[i] & 0xffffu));
        const double b = *reinterpret_cast<const double*>(cm + (p[i] >> 16));
        lo = min1(lo, min1(a, b));
        hi = max1(hi, max1(a, b));
    }
}

// WETDRY of an element that it changes, from its limited modes L (mean and linear modes of each field); the modes
// past the third are read here.
template <int P>
__device__ __forceinline__ void wetdry_limited(const DevTables& T, const double (&L)[3][3], const double (&D)[3], int wdi,
                                               double h0, double* __restrict__ u, int e, int ne,
                                               uint8_t* __restrict__ wd_out, int* __restrict__ wd_active) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    double U[3][DOF];
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < DOF; k++) U[f][k] = k < 3 ? L[f][k] : at(u + (size_t)(f * DOF + k) * ne, e);
    const double c13 = 1.0 / 3.0, c16 = 1.0 / 6.0;
    const double hb[3] = {c13 * (D[0] + D[1] + D[2]), -(c16 * (D[0] + D[1])) + c13 * D[2], -(0.5 * D[0]) + 0.5 * D[1]};
    const double dpe_min = fmin(fmin(D[0], D[1]), D[2]);
    if (wd_active) wd_active[0] = 1;
    at(wd_out, e) = (uint8_t)wetdry_element<P>(T, U, D, hb, dpe_min, wdi, h0);
#pragma unroll
    for (int f = 0; f < 3; f++) {
        // wetting and drying changes the cell mean only of some elements: written back when its bits changed
        if (__double_as_longlong(U[f][0]) != __double_as_longlong(L[f][0])) at(u + (size_t)(f * DOF) * ne, e) = U[f][0];
#pragma unroll
        for (int k = 1; k < DOF; k++) at(u + (size_t)(f * DOF + k) * ne, e) = U[f][k];
    }
}

template <int P, bool WETDRY>
__global__ void __launch_bounds__(3 * LIM_NT) __attribute__((amdgpu_waves_per_eu(4))) limit_wetdry_kernel(ElemData E, double* __restrict__ u,
                                                              const double* __restrict__ cmean, size_t cms,
                                                              LimTiles lt,
                                                              const uint8_t* __restrict__ wd_in,
                                                              uint8_t* __restrict__ wd_out,
                                                              int* __restrict__ wd_active) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    constexpr int NT = LIM_NT;
    const DevTables& T = tab<P>();
    const int ne = E.ne;
    const int c = __builtin_amdgcn_readfirstlane(threadIdx.x / NT), le = threadIdx.x - c * NT;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int e = tile * NT + le;
    const bool valid = e < ne;
    extern __shared__ double lds[];
    const int nsl = NT + lt.nvh, nql = lt.nql;
    double* const cm = lds + c * nsl;                       // field c's staged cell means
    double* const bnd = lds + 3 * nsl + 2 * c * nql;        // field c's node minima, maxima
    // the first halo entry's and node's indices and the element's own loads, then the staging (lanes past the last
    // element read element ne-1 and write nothing)
    const int ec = valid ? e : ne - 1;
    const int* vh = lt.vhidx + (size_t)tile * lt.nvh;
    const uint4* qi = reinterpret_cast<const uint4*>(lt.qinc) + (size_t)tile * nql;
    const int g = le < lt.nvh ? vh[le] : -1;
    uint4 rq = le < nql ? qi[le] : make_uint4(0, 0, 0, 0);
    const double* row = cmean + (size_t)c * cms;
    const double c0 = at(row, ec);
    double w1 = at(u + (size_t)(c * DOF + 1) * ne, ec), w2 = at(u + (size_t)(c * DOF + 2) * ne, ec);
    const int lq = at(lt.elq, ec);
    double D[3] = {0.0, 0.0, 0.0}, h0 = 0.0;
    int wdi = 0;
    if (WETDRY && c == 0) {
#pragma unroll
        for (int v = 0; v < 3; v++) D[v] = at(E.dpv + (size_t)v * ne, ec);
        const int sid = E.sid ? (int)at(E.sid, ec) : 0;
        h0 = E.scen[sid].h0;
        wdi = at(wd_in, ec);
    }
    const double m = at(row, g < 0 ? 0 : g);
    cm[le] = c0;
    if (g >= 0) cm[NT + le] = m;
#pragma unroll 1
    for (int h = le + NT; h < lt.nvh; h += NT) {
        const int gh = vh[h];
        if (gh < 0) break;
        cm[NT + h] = at(row, gh);
    }
    __syncthreads();
    // the bounds of the tile's nodes
    const char* const cmb = reinterpret_cast<const char*>(cm);
    for (int q = le; q < nql; q += NT) {
        if (q != le) rq = qi[q];
        double lo = 99999., hi = -99999.;
        minmax8(cmb, rq, lo, hi);
        bnd[q] = lo;
        bnd[nql + q] = hi;
    }
    if (lt.nx > 0) {
        // nodes with more than eight elements: one lane of each field goes through the tile's extra entries
        const int x0 = lt.xoff[tile], x1 = lt.xoff[tile + 1];
        if (x1 > x0) {
            __syncthreads();
            if (le == 0)
                for (int x = x0; x < x1; x++) {
                    const int q = lt.xq[x];
                    double lo = bnd[q], hi = bnd[nql + q];
                    minmax8(cmb, reinterpret_cast<const uint4*>(lt.xinc)[x], lo, hi);
                    bnd[q] = lo;
                    bnd[nql + q] = hi;
                }
        }
    }
    __syncthreads();
    {
        const int q[3] = {lq & 1023, (lq >> 10) & 1023, (lq >> 20) & 1023};
        double vmin[3], vmax[3];
#pragma unroll
        for (int i = 0; i < 3; i++) { vmin[i] = bnd[q[i]]; vmax[i] = bnd[nql + q[i]]; }
        limit_field(T, c0, w1, w2, vmin, vmax);
    }
    if (!WETDRY) {
        if (!valid) return;
        at(u + (size_t)(c * DOF + 1) * ne, e) = w1;
        at(u + (size_t)(c * DOF + 2) * ne, e) = w2;
        return;
    }
    // elements that WETDRY changes: the three lanes' values meet in LDS and the element's first lane goes on alone
    uint8_t* const keep = reinterpret_cast<uint8_t*>(lds + max(3 * nsl + 6 * nql, 9 * NT));
    bool mine = true;
    if (c == 0) {
        if (valid) {
            const double U[3][DOF] = {{c0, w1, w2}};
            mine = wetdry_keeps<P>(T, U, D, wdi, h0);
        }
        keep[le] = mine;
    }
    if (!__syncthreads_or(!mine)) {
        if (!valid) return;
        if (c == 0) at(wd_out, e) = 1;
        at(u + (size_t)(c * DOF + 1) * ne, e) = w1;
        at(u + (size_t)(c * DOF + 2) * ne, e) = w2;
        return;
    }
    mine = keep[le];
    double* const ex = lds;                                 // [field*3 + mode][NT]
    if (!mine) {
        ex[(c * 3) * NT + le] = c0;
        ex[(c * 3 + 1) * NT + le] = w1;
        ex[(c * 3 + 2) * NT + le] = w2;
    } else if (valid) {
        if (c == 0) at(wd_out, e) = 1;
        at(u + (size_t)(c * DOF + 1) * ne, e) = w1;
        at(u + (size_t)(c * DOF + 2) * ne, e) = w2;
    }
    __syncthreads();
    if (mine || c != 0) return;
    double U3[3][3];
#pragma unroll
    for (int f = 0; f < 3; f++)
#pragma unroll
        for (int k = 0; k < 3; k++) U3[f][k] = ex[(f * 3 + k) * NT + le];
    wetdry_limited<P>(T, U3, D, wdi, h0, u, e, ne, wd_out, wd_active);
}

template <int P, bool WETDRY, bool WDADJ>
__global__ void __launch_bounds__(LIM_NT) limit_wide_kernel(ElemData E, double* __restrict__ u, const double* __restrict__ cmean,
                                                            size_t cms, LimTiles lt, const uint8_t* __restrict__ wd_in,
                                                            uint8_t* __restrict__ wd_out, int* __restrict__ wd_active,
                                                            double* __restrict__ ub, double* __restrict__ gdp) {
    static_assert(!(WETDRY && WDADJ), "the WETDRY reverse starts from the limiter's output alone");
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    constexpr int NT = LIM_NT;
    const DevTables& T = tab<P>();
    const int ne = E.ne;
    const int le = threadIdx.x;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int e = tile * NT + le;
    const bool valid = e < ne;
    extern __shared__ double lds[];
    const int nsl = NT + lt.nvh, nql = lt.nql;
    double* const cm = lds;                                 // [field][nsl] staged cell means
    double* const bnd = lds + 3 * nsl;                      // [field][min, max][nql] node bounds
    const int ec = valid ? e : ne - 1;                      // lanes past the last element read element ne-1 and write nothing
    const int* vh = lt.vhidx + (size_t)tile * lt.nvh;
    const uint4* qi = reinterpret_cast<const uint4*>(lt.qinc) + (size_t)tile * nql;
    const int g = le < lt.nvh ? vh[le] : -1;
    uint4 rq = le < nql ? qi[le] : make_uint4(0, 0, 0, 0);
    double c0[3], w1[3], w2[3], m[3];
#pragma unroll
    for (int f = 0; f < 3; f++) {
        c0[f] = at(cmean + (size_t)f * cms, ec);
        w1[f] = at(u + (size_t)(f * DOF + 1) * ne, ec);
        w2[f] = at(u + (size_t)(f * DOF + 2) * ne, ec);
    }
    const int lq = at(lt.elq, ec);
    double D[3] = {0.0, 0.0, 0.0}, h0 = 0.0;
    int wdi = 0;
    if (WETDRY || WDADJ) {
#pragma unroll
        for (int v = 0; v < 3; v++) D[v] = at(E.dpv + (size_t)v * ne, ec);
        const int sid = E.sid ? (int)at(E.sid, ec) : 0;
        h0 = E.scen[sid].h0;
        wdi = at(wd_in, ec);
    }
#pragma unroll
    for (int f = 0; f < 3; f++) m[f] = at(cmean + (size_t)f * cms, g < 0 ? 0 : g);
#pragma unroll
    for (int f = 0; f < 3; f++) {
        cm[f * nsl + le] = c0[f];
        if (g >= 0) cm[f * nsl + NT + le] = m[f];
    }
#pragma unroll 1
    for (int h = le + NT; h < lt.nvh; h += NT) {
        const int gh = vh[h];
        if (gh < 0) break;
#pragma unroll
        for (int f = 0; f < 3; f++) cm[f * nsl + NT + h] = at(cmean + (size_t)f * cms, gh);
    }
    __syncthreads();
    const char* const cmb = reinterpret_cast<const char*>(cm);
    for (int q = le; q < nql; q += NT) {
        if (q != le) rq = qi[q];
#pragma unroll
        for (int f = 0; f < 3; f++) {
            double lo = 99999., hi = -99999.;
            minmax8(cmb + (size_t)8 * f * nsl, rq, lo, hi);
            bnd[2 * f * nql + q] = lo;
            bnd[(2 * f + 1) * nql + q] = hi;
        }
    }
    if (lt.nx > 0) {
        const int x0 = lt.xoff[tile], x1 = lt.xoff[tile + 1];
        if (x1 > x0) {
            // nodes with more than eight elements: a lane of each field goes through the tile's extra entries
            __syncthreads();
            if (le < 3)
                for (int x = x0; x < x1; x++) {
                    const int q = lt.xq[x];
                    double lo = bnd[2 * le * nql + q], hi = bnd[(2 * le + 1) * nql + q];
                    minmax8(cmb + (size_t)8 * le * nsl, reinterpret_cast<const uint4*>(lt.xinc)[x], lo, hi);
                    bnd[2 * le * nql + q] = lo;
                    bnd[(2 * le + 1) * nql + q] = hi;
                }
        }
    }
    __syncthreads();
    {
        const int q[3] = {lq & 1023, (lq >> 10) & 1023, (lq >> 20) & 1023};
#pragma unroll
        for (int f = 0; f < 3; f++) {
            double vmin[3], vmax[3];
#pragma unroll
            for (int i = 0; i < 3; i++) { vmin[i] = bnd[2 * f * nql + q[i]]; vmax[i] = bnd[(2 * f + 1) * nql + q[i]]; }
            limit_field(T, c0[f], w1[f], w2[f], vmin, vmax);
        }
    }
    if (!valid) return;
    if (WETDRY || WDADJ) {
        const double K[3][DOF] = {{c0[0], w1[0], w2[0]}};
        if (!wetdry_keeps<P>(T, K, D, wdi, h0)) {
            const double L[3][3] = {{c0[0], w1[0], w2[0]}, {c0[1], w1[1], w2[1]}, {c0[2], w1[2], w2[2]}};
            if constexpr (WDADJ) wetdry_adj_element<P>(T, L, D, wdi, h0, e, ne, ub, gdp);
            else wetdry_limited<P>(T, L, D, wdi, h0, u, e, ne, wd_out, wd_active);
            return;
        }
        if (WDADJ) return;
        at(wd_out, e) = 1;
    }
#pragma unroll
    for (int f = 0; f < 3; f++) {
        at(u + (size_t)(f * DOF + 1) * ne, e) = w1[f];
        at(u + (size_t)(f * DOF + 2) * ne, e) = w2[f];
    }
}

// ------------------------------------------------------------------------------------------
// modal2nodal (src/write_results.F:14-174) + NODECODE from the wet flags.  Each node's incident
// elements are summed in the order of its CSR row (the host's ELETAB order when the host gave it).
// With etamax set, ETAMAX is raised as the reference raises it: after every wet element's
// contribution to ETA2, so it also sees the partial sums (src/write_results.F:164).
// ------------------------------------------------------------------------------------------
// Bound by latency on small meshes: a node's row was walked one element at a time, each waiting for its loads.  1,600
// elements 9.9 us before, 5.5 us now with the groups below; one million 271 and 113 us.  64 nodes per block spread
// small meshes over more CUs.
constexpr int M2N_NT = 64;   // nodes per block

template <int P>
__global__ void __launch_bounds__(M2N_NT) modal2nodal_kernel(int np, ElemData E, const int* __restrict__ off,
                                                          const int* __restrict__ n2e,
                                                          const double* __restrict__ u,
                                                          const uint8_t* __restrict__ wd, double nleq,
                                                          double leq, double* __restrict__ out,
                                                          int* __restrict__ nodecode,
                                                          double* __restrict__ etamax) {
    constexpr int DOF = (P + 1) * (P + 2) / 2;
    // corner values in LDS: the corner differs from lane to lane
    __shared__ double pcn[3][DOF];
    if (threadIdx.x < 3 * DOF) pcn[threadIdx.x / DOF][threadIdx.x % DOF] = tab<P>().phi_corner[threadIdx.x / DOF][threadIdx.x % DOF];
    __syncthreads();
    const int ne = E.ne;
    const int n = xcd_tile(blockIdx.x, gridDim.x) * M2N_NT + threadIdx.x;
    if (n >= np) return;
    // the node's row in groups of up to B incidences whose loads are under way together (past the row's end the group
    // repeats its last incidence, which is then not summed); dry elements are skipped
    constexpr int B = P == 1 ? 6 : 4;
    const int j0 = off[n], j1 = off[n + 1];
    double asum = 0;
    int nc = 0;
    for (int j = j0; j < j1; j += B) {
        int ei[B];
        double ar[B];
        bool wet[B];
#pragma unroll
        for (int q = 0; q < B; q++) ei[q] = n2e[min(j + q, j1 - 1)] >> 2;
#pragma unroll
        for (int q = 0; q < B; q++) {
            wet[q] = j + q < j1 && at(wd, ei[q]) != 0;
            const double X0 = at(E.xv, ei[q]), X1 = at(E.xv + ne, ei[q]), X2 = at(E.xv + 2 * (size_t)ne, ei[q]);
            const double Y0 = at(E.yv, ei[q]), Y1 = at(E.yv + ne, ei[q]), Y2 = at(E.yv + 2 * (size_t)ne, ei[q]);
            ar[q] = (X0 - X2) * (Y1 - Y2) + (X2 - X1) * (Y0 - Y2);
        }
#pragma unroll
        for (int q = 0; q < B; q++)
            if (wet[q]) { nc = 1; asum = asum + 0.5 * ar[q]; }
    }
    double e2 = 0.0, u2 = 0.0, v2 = 0.0;
    double emax = etamax ? etamax[n] : 0.0;
    for (int j = j0; j < j1; j += B) {
        int ent[B];
        double z[B], x[B], y[B], h[B], ar[B];
        bool wet[B];
#pragma unroll
        for (int q = 0; q < B; q++) ent[q] = n2e[min(j + q, j1 - 1)];
#pragma unroll
        for (int q = 0; q < B; q++) {
            const int e = ent[q] >> 2, c = ent[q] & 3;
            wet[q] = j + q < j1 && at(wd, e) != 0;
            const double X0 = at(E.xv, e), X1 = at(E.xv + ne, e), X2 = at(E.xv + 2 * (size_t)ne, e);
            const double Y0 = at(E.yv, e), Y1 = at(E.yv + ne, e), Y2 = at(E.yv + 2 * (size_t)ne, e);
            ar[q] = (X0 - X2) * (Y1 - Y2) + (X2 - X1) * (Y0 - Y2);
            const double D0 = at(E.dpv, e), D1 = at(E.dpv + ne, e), D2 = at(E.dpv + 2 * (size_t)ne, e);
            const double hb[3] = {1.0 / 3.0 * (D0 + D1 + D2), -(1.0 / 6.0 * (D0 + D1)) + 1.0 / 3.0 * D2, -(0.5 * D0) + 0.5 * D1};
            double zd = at(u, e), xd = at(u + (size_t)DOF * ne, e), yd = at(u + (size_t)2 * DOF * ne, e), hd = hb[0];
#pragma unroll
            for (int kk = 1; kk < DOF; kk++) {
                const double pc = pcn[c][kk];
                zd = zd + pc * at(u + (size_t)kk * ne, e);
                xd = xd + pc * at(u + (size_t)(DOF + kk) * ne, e);
                yd = yd + pc * at(u + (size_t)(2 * DOF + kk) * ne, e);
                hd = hd + pc * (kk < 3 ? hb[kk] : 0.0);
            }
            z[q] = zd; x[q] = xd; y[q] = yd; h[q] = hd;
        }
#pragma unroll
        for (int q = 0; q < B; q++) {
            if (!wet[q]) continue;
            const double area = 0.50 * ar[q] / asum;
            const double depth = z[q] + h[q];
            const double fh = 1.0 / (nleq * depth + leq);
            e2 = e2 + area * z[q];
            if (emax < e2) emax = e2;
            u2 = u2 + area * x[q] * fh;
            v2 = v2 + area * y[q] * fh;
        }
    }
    out[n] = e2; out[(size_t)np + n] = u2; out[2 * (size_t)np + n] = v2;
    nodecode[n] = nc;
    if (etamax) etamax[n] = emax;
}

// ------------------------------------------------------------------------------------------
// NWS=8 node kernel: HollandGet's per-node profile (src/wind.F:2062-2131) and the wind speed and
// Garratt drag of MET_FORCING (src/met_forcing.F:488-500, src/wind.F:135-141), at TIME_A of every
// step of a batch.  The stresses and the pressure with each stage's ramp are formed here, one 32-byte record per
// node and stage: the stage kernels gather three records instead of fifteen values, and form nothing from
// them per element.  Stage of sixteen p=1 storm basins (440,000 elements) 76.4 us before, 74.1 us now.
// ------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) met_kernel(Met m, Forcing fo) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= m.np) return;
    const int s = blockIdx.y;                               // step of the batch
    const int sid = m.nsid ? (int)m.nsid[n] : 0;
    const double* r = m.row + ((size_t)sid * m.rows + table_step(fo) + s) * MET_ROW;
    const double re = 6378206.4;
    const double deg2rad = 3.141592653589793 / 180.0;
    const double lat = r[MR_LAT], lon = r[MR_LON], spd = r[MR_SPD], B = r[MR_B];
    const double dx = (m.xc[n] - lon) * deg2rad, dy = (m.yc[n] - lat) * deg2rad;
    const double theta = atan2(dy, dx);
    const double s1 = sin(dy / 2.0), s2 = sin(dx / 2.0);
    const double rad = re * (2.0 * asin(sqrt(s1 * s1 + r[MR_COSLAT] * m.cosy[n] * (s2 * s2))));
    const double cor = m.cor[n];
    const double rb = pow(r[MR_RMW] * 1000.0 / rad, B);
    const double press = (r[MR_CPRESS] + r[MR_DEFICIT] * exp(-rb)) / r[MR_RHOG];
    double vr = sqrt(rb * exp(1.0 - rb) * (spd * spd) + (rad * rad) * (cor * cor) / 4.0) - rad * cor / 2.0;
    const double tsx = (fabs(vr) / spd) * r[MR_TVX], tsy = (fabs(vr) / spd) * r[MR_TVY];
    vr = vr * r[MR_WMULT];
    double wx = -(vr * sin(theta)), wy = vr * cos(theta);
    wx = wx * r[MR_BLADJ]; wy = wy * r[MR_BLADJ];
    wx = wx * 0.88; wy = wy * 0.88;
    wx = wx + tsx; wy = wy + tsy;
    const double wmag = sqrt(wx * wx + wy * wy);
    double cd = 0.001 * (0.75 + 0.067 * wmag);
    if (cd > 0.0035) cd = 0.0035;
    const double* rp = fo.ramp + (size_t)sid * fo.rows + (size_t)(table_step(fo) + s) * fo.nrk;
    for (int irk = 0; irk < fo.nrk; irk++) {
        const double ramp = rp[irk];
        m.st[((size_t)s * fo.nrk + irk) * m.np + n] =
            make_double4(ramp * 0.001293 * cd * wx * wmag, ramp * 0.001293 * cd * wy * wmag, ramp * press, 0.0);
    }
}

// The state between the step's layout (soa: [field][mode][element]) and the host's (aos: [field][element][mode]), one
// value per thread in the host's order, so that the copy to or from the caller's arrays is a plain one; with `flags`
// WDFLG between bytes and the host's integers too.  Transposing on the host took longer than the copy: reading back
// 298,700 p=2 elements (43 MB) 14.4 ms before, 4.2 ms then, of which the kernel takes 0.03 ms (setting it 13.2 and 1.6 ms).
template <int DOF, bool OUT>
__global__ void __launch_bounds__(256) state_layout_kernel(int ne, double* __restrict__ soa, double* __restrict__ aos,
                                                           uint8_t* __restrict__ wd, int* __restrict__ flags) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, n = (size_t)ne * DOF;
    if (i >= 3 * n) return;
    if (flags && i < (size_t)ne) {
        if (OUT) flags[i] = wd[i];
        else wd[i] = flags[i] ? 1 : 0;
    }
    const int f = (int)(i / n);
    const size_t j = i - f * n, e = j / DOF, k = j - e * DOF;
    double* const s = soa + ((size_t)f * DOF + k) * ne + e;
    if (OUT) aos[i] = *s;
    else *s = aos[i];
}

// Rows of the forcing tables from one packed list of values: table t holds `w` values per scenario, taken from
// list position `off` on and `stride` apart in the table (whose rows are laid out for the longest call).
struct TableRows {
    int n;
    struct { double* dst; size_t off, w, stride; } t[9];
};

__device__ __forceinline__ void put_table_value(const TableRows& r, size_t i, double v) {
    for (int t = r.n - 1; t >= 0; t--)
        if (i >= r.t[t].off) {
            const size_t j = i - r.t[t].off, sc = j / r.t[t].w;
            r.t[t].dst[sc * r.t[t].stride + (j - sc * r.t[t].w)] = v;
            return;
        }
}

__global__ void __launch_bounds__(256) table_rows_kernel(TableRows r, const double* __restrict__ src, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) put_table_value(r, i, src[i]);
}

// The same with the values in the launch's arguments: nothing to copy and nothing to wait for, which is what a
// call of one step costs most (build_stage_tables).
constexpr int TABLE_ARGS = 448;   // with TableRows within the 4 KB that a launch's arguments may take
struct TableArgs { double v[TABLE_ARGS]; };

__global__ void __launch_bounds__(TABLE_ARGS) table_args_kernel(TableRows r, TableArgs a, size_t first, int n) {
    const int i = threadIdx.x;
    if (i < n) put_table_value(r, first + i, a.v[i]);
}

// Device step counter used by the forcing-table lookups of captured steps (a kernel, not a memset,
// so that the sequence can be captured into a HIP graph).
__global__ void step_counter_kernel(int* __restrict__ step, int set, int value) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *step = set ? value : *step + value;
}

// Water volume per element: 0.5*AREAS*(ze_1 + hb_1), reduced per block.
template <int P>
__global__ void __launch_bounds__(256) mass_kernel(ElemData E, const double* __restrict__ u,
                                                   double* __restrict__ partial) {
    __shared__ double sh[256];
    const int ne = E.ne;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    double m = 0.0;
    if (e < ne) {
        const double X0 = E.xv[e], X1 = E.xv[(size_t)ne + e], X2 = E.xv[2 * (size_t)ne + e];
        const double Y0 = E.yv[e], Y1 = E.yv[(size_t)ne + e], Y2 = E.yv[2 * (size_t)ne + e];
        const double D0 = E.dpv[e], D1 = E.dpv[(size_t)ne + e], D2 = E.dpv[2 * (size_t)ne + e];
        const double areas = (X0 - X2) * (Y1 - Y2) + (X2 - X1) * (Y0 - Y2);
        m = 0.5 * areas * (u[e] + 1.0 / 3.0 * (D0 + D1 + D2));
    }
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

// out = ((0 + v[0]) + v[1]) + ... + v[n-1], the left-to-right order of a host loop.
__global__ void __launch_bounds__(64) sum_in_order_kernel(const double* __restrict__ v, int n,
                                                          double* __restrict__ out) {
    if (threadIdx.x != 0) return;
    double s = 0.0;
    for (int i = 0; i < n; i++) s += v[i];
    *out = s;
}

}  // namespace dg
