// Device kernels of the lattice update.
//
// One time step (the reference's src/main.F90:290-329) is
//   1. step_kernel      : pull-stream + moments + equilibrium + regularization + Vreman tau +
//                         relaxation + inflow-turbulence df + body-force df + solid swap, one
//                         pass over the interior, reading buffer P(n-1) and writing P(n);
//   2. boundary_kernel  : the non-periodic ghost passes of boundarycond on the buffer just
//                         written (closed i, j, k faces; edges and corners; inflow/outflow), where
//                         the step kernel does not perform them itself.
// The buffers hold post-collision populations (the reference's f1 after postcoll/solids) in
// the interior and the reference's persistent ghost layers.  The reference's post-streaming
// state f1 = drift(P(n)) is formed on the fly by the next step, and by StateOut when the
// caller asks for it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <type_traits>

#include "codec.h"
#include "fields.h"
#include "lattice.h"
#include "layout.h"
#include "impl.h"

namespace lbm {

template <typename R>
struct StepArgs {
    Layout lay;
    const void* src;       // buffer holding P(n-1) (or the uploaded state when stream == 0)
    void* dst;             // buffer receiving P(n)
    int stream;            // 1: pull-stream from src; 0: collide the state in place
    R fac0;                // 1 - 1/tau0 when Vreman is off (tau0 = 3*kinevisc + 0.5)
    R kinevisc, vconst, eps, tiny;
    const R* ablvisc;      // [nz]
    const R* ext_rho;      // moments to use instead of the computed ones (first step after
    const R* ext_u;        //   an equilibrium initialisation, src/main.F90:214,243,299);
    const R* ext_v;        //   cell layout, nullptr otherwise
    const R* ext_w;
    const uint32_t* solid; // one bit per interior cell in rows along the contiguous axis,
                           //   solid_wpr words per row; nullptr: no solids
    int solid_wpr;
    int ip;                // inflow-turbulence slice (reference: 10)
    const R* tu;           // turbulence slice (ny*nz, j fastest) for this step; nullptr: off
    const R* tv;
    const R* tw;
    R ampl;
    R* avg;                // six cell planes: sums of u, v, w, u^2, v^2, w^2 of the streamed
                           //   input (the moments after the previous step); nullptr: off
    const R* Fx;           // external forcing (cell layout); nullptr: off
    const R* Fy;
    const R* Fz;
    int flo[3], fhi[3];    // cells (i, j, k; inclusive) whose force is read (the others have none)
    const R* theta;        // potential temperature (cell layout) of the buoyancy forcing; nullptr: off
    R btheta0, bscale;     // its reference temperature and g * time^2 / length
    R* tau_out;            // cell layout; nullptr: tau not stored
    int fold_dir;          // closed axis whose face pass this kernel performs (-1: none)
    int fold_opt_lo, fold_opt_hi;
    // inflow/outflow planes of i written by the cells at i = 1 and i = nx (0: separate pass; 2: but for
    // the rows along the walls of j and k, both closed, whose ghosts the face passes read first)
    int inflow_fold;
    const R* shear;        // uvel_shear(nz)
    R utime, cosd, sind, rho0;
    int heavy_first;       // bit 0 / bit 1: cells 1 and n of ax1 / ax2 are dispatched first
    int halo_dir;          // axis whose ghost planes are halos filled by lbm_halo_unpack (-1: none)
    int xcd_groups;        // 1: the blocks of one row group run on one XCD (step_kernel)
    // split step along the halo axis (step_kernel): 0 every cell; 1 the part_edge cells next to
    // each halo plane (the launch covers 2 * part_edge along part_axis); 2 the others (the launch
    // covers n - 2 * part_edge).  part_axis: 1 the halo axis is ax1, 2 it is ax2.
    int part, part_axis, part_edge;
    int store_end;         // last column stored in a row (Layout::row_store_end)
};

// Signed sum  sx*a + sy*b + sz*c  for compile-time signs in {-1,0,1}: adds only.  With no term the
// result is -0, the additive identity, so that a sum it starts folds away.
template <typename R>
__host__ __device__ __forceinline__ R sdot(int sx, int sy, int sz, R a, R b, R c) {
    R s = -R(0);
    bool first = true;
    if (sx != 0) { s = sx > 0 ? a : -a; first = false; }
    if (sy != 0) { s = first ? (sy > 0 ? b : -b) : (sy > 0 ? s + b : s - b); first = false; }
    if (sz != 0) { s = first ? (sz > 0 ? c : -c) : (sz > 0 ? s + c : s - c); }
    return s;
}

// Reciprocal: the hardware's (1 ulp) in FP32 device code, the IEEE quotient otherwise.  Used for
// 1/rho, 1/tau and the Vreman ratio, where the FP32 quotient's correction sequence costs about
// ten instructions per use in an issue-bound kernel.
template <typename R>
__host__ __device__ __forceinline__ R recip(R x) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (std::is_same<R, float>::value) return __builtin_amdgcn_rcpf(x);
#endif
    return R(1) / x;
}

// Square root: the hardware's in FP32 device code (the Vreman ratio is a normal number wherever it
// is used), the IEEE root otherwise.  The adjoint uses it; the forward collision keeps the IEEE
// root (a one-ulp change of the eddy viscosity moves the realization of a turbulent run).
template <typename R>
__host__ __device__ __forceinline__ R sqrt_r(R x) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (std::is_same<R, float>::value) return __builtin_amdgcn_sqrtf(x);
#endif
    using std::sqrt;   // the tangent type brings its own sqrt
    return sqrt(x);
}

// Hermite equilibrium of direction l (src/m_postcoll_kernel.F90:136-183 in closed form):
//   feq = w rho (1 - 1.5 u.u + cu (3 + 4.5 cu [+ 4.5 (cu^2 - u.u)]))   with cu = c.u
// The bracket is the reference's full H3:A3 contraction, 4.5 rho cu (cu^2 - u.u), applied for
// l > 0 when the third order is on.
template <int Q, bool ORDER3, typename R>
__device__ __forceinline__ R feq_dir(int l, R rho, R ux, R uy, R uz, R usq) {
    using Lt = Lattice<Q>;
    const R cu = sdot<R>(Lt::cx(l), Lt::cy(l), Lt::cz(l), ux, uy, uz);
    R poly = R(3) + R(4.5) * cu;
    if (ORDER3 && l > 0) poly += R(4.5) * (cu * cu - usq);
    return (weight<Q, R>(l) * rho) * ((R(1) - R(1.5) * usq) + cu * poly);
}

// Reflected direction for a wall normal to axis d: normal component negated, tangential
// components multiplied by opt (-1 no-slip, +1 free-slip).
template <int Q>
__host__ __device__ constexpr int mirror(int l, int d, int opt) {
    using Lt = Lattice<Q>;
    return Lt::find(d == 0 ? -Lt::cx(l) : opt * Lt::cx(l), d == 1 ? -Lt::cy(l) : opt * Lt::cy(l),
                    d == 2 ? -Lt::cz(l) : opt * Lt::cz(l));
}

// The per-cell part of a step: moments, collision, turbulence and body-force increments, solid
// swap.  rv holds the streamed populations of cell (i,j,k) (storage coordinates ca,cb,cc, device
// cell offset oc); dev receives the departures S*(f_l - w_l) of its post-collision populations
// (S = C::kDepScale), tau the Vreman relaxation time.
//
// Directions come in opposite pairs (l, l+1) for odd l (src/mod_D3Q27setup.F90:31,43).  Every
// quantity the collision forms per direction is even or odd in c, so each pair is evaluated
// once: moments accumulate from D_l +- D_l+1 and the outputs are (even) +- (odd), with
//   feq_l - w_l = w (rho*base - 1 + 4.5 rho cu^2) + w rho cu (3 [+ 4.5 (cu^2 - u.u)])
//   (src/m_postcoll_kernel.F90:136-183 in closed form; base = 1 - 1.5 u.u; the bracket is the
//   reference's full H3:A3 contraction, applied for l > 0 when the third order is on)
// and the regularized non-equilibrium (src/m_postcoll_kernel.F90:189-244)
//   fneq_l = 4.5 w [ (cAc - T/3) + (cu (3 cAc - T) - 2 c.g) ],  T = tr a2,  g = a2 u.
// Working on departures needs no decode/encode arithmetic for the shifted 16-bit formats and
// forms rho = 1 + sum D/S, j = sum c D/S without the cancellation of sum f.
// Per-cell inputs of the collision besides the populations: the ABL viscosity of the layer and the
// word of the row's solid mask holding the cell's bit.  For 16-bit storage the step kernel reads
// them ahead of the population loads, so that their latency overlaps those loads' instead of
// stalling the collision where they are used (measured on MI355X, D3Q27 reg+Vreman 384x192x128:
// FP16 214 -> 198 us, BF16 215 -> 196 us per step kernel; FP32 352 -> 358 us, so 4- and 8-byte
// storage read them where they are used).  The external force stays where it is used: read ahead,
// its three registers would be held through every collision, forced or not (they cost the D3Q19
// BGK kernel its fifth wave per SIMD).
template <typename R>
struct CellAux {
    R abl;
    uint32_t sword;
};
template <bool VRE, typename R>
__host__ __device__ __forceinline__ CellAux<R> cell_aux(const StepArgs<R>& a, int k, int ca, int cb, int cc) {
    const Layout& L = a.lay;
    CellAux<R> x{R(0), 0u};
    if (VRE) x.abl = a.ablvisc[k - 1];
    if (a.solid != nullptr) x.sword = a.solid[((cc - 1) * L.n(L.ax1) + (cb - 1)) * a.solid_wpr + ((ca - 1) >> 5)];
    return x;
}

// AUX: the per-cell inputs come from aux (read ahead by the caller); otherwise they are read here
// where they are used.  sums: add the cell to the averaging sums if those are on (false in a lane
// that repeats another's cell).
template <int Q, class C, bool BGK3, bool HRR, bool VRE, bool AUX = false>
__host__ __device__ __forceinline__ void collide_cell(const StepArgs<typename C::real>& a, const typename C::raw (&rv)[Q],
                                                      const CellAux<typename C::real>& aux, int i, int j, int k, int ca,
                                                      int cb, int cc, int oc, bool sums, typename C::real (&dev)[Q],
                                                      typename C::real& tau_out) {
    using R = typename C::real;
    using Lt = Lattice<Q>;
    const Layout& L = a.lay;
    constexpr int NP = (Q - 1) / 2;
    constexpr R S = C::kDepScale;
    constexpr R invS = R(1) / S;

    R D[Q];
#pragma unroll
    for (int l = 0; l < Q; ++l) D[l] = C::template dep<Q>(rv[l], l);
    // accumulators start at -0, the additive identity the compiler may fold (0 + x is not x for
    // x = -0)
    const R z0 = -R(0);
    R jx = z0, jy = z0, jz = z0;
    R pxy = z0, pxz = z0, pyz = z0;
    // pair sums by the axes c spans (a face axis, an edge plane, the corners): the density and
    // the diagonal second moments are sums of these (a corner counts in all three diagonals, an
    // edge plane in two)
    R sfx = z0, sfy = z0, sfz = z0, sexy = z0, sexz = z0, seyz = z0, scn = z0;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int l = 2 * p + 1;
        const int cx = Lt::cx(l), cy = Lt::cy(l), cz = Lt::cz(l);
        const int n2 = Lt::norm2(l);
        const R sp = D[l] + D[l + 1];
        const R dp = D[l] - D[l + 1];
        if (n2 == 1) (cx != 0 ? sfx : cy != 0 ? sfy : sfz) += sp;
        else if (n2 == 2) (cz == 0 ? sexy : cy == 0 ? sexz : seyz) += sp;
        else scn += sp;
        if (cx > 0) jx += dp; else if (cx < 0) jx -= dp;
        if (cy > 0) jy += dp; else if (cy < 0) jy -= dp;
        if (cz > 0) jz += dp; else if (cz < 0) jz -= dp;
        if (HRR || VRE) {
            if (cx * cy > 0) pxy += sp; else if (cx * cy < 0) pxy -= sp;
            if (cx * cz > 0) pxz += sp; else if (cx * cz < 0) pxz -= sp;
            if (cy * cz > 0) pyz += sp; else if (cy * cz < 0) pyz -= sp;
        }
    }
    R dr = D[0] + (((sfx + sfy) + sfz) + ((sexy + sexz) + seyz) + scn);
    const R pxx = sfx + sexy + sexz + scn, pyy = sfy + sexy + seyz + scn, pzz = sfz + sexz + seyz + scn;
    dr *= invS;
    R rh = R(1) + dr;
    const R invrho = recip(rh);
    R ux = (jx * invS) * invrho, uy = (jy * invS) * invrho, uz = (jz * invS) * invrho;
    if (a.avg != nullptr && sums) {
        // time averaging of the moments after the previous step (src/m_averaging_full_kernel.F90:33-39)
        // (the six sums are read before any is written: one memory round trip instead of six)
        R* p = a.avg + oc;
        const size_t P = (size_t)L.cplane;
        const R s0 = p[0], s1 = p[P], s2 = p[2 * P], s3 = p[3 * P], s4 = p[4 * P], s5 = p[5 * P];
        p[0] = s0 + ux;
        p[P] = s1 + uy;
        p[2 * P] = s2 + uz;
        p[3 * P] = s3 + ux * ux;
        p[4 * P] = s4 + uy * uy;
        p[5 * P] = s5 + uz * uz;
    }
    if (a.ext_rho) { rh = a.ext_rho[oc]; ux = a.ext_u[oc]; uy = a.ext_v[oc]; uz = a.ext_w[oc]; }
    const R usq = ux * ux + uy * uy + uz * uz;
    const R base = R(1) - R(1.5) * usq;
    const R rb1 = rh * base - R(1);      // rho*base - 1
    const R r45 = R(4.5) * rh;

    // Non-equilibrium second-order tensor a2 = sum_l H2_l (f_l - feq_l)
    //   = Pi' - rho u u - (sum_l (f_l - w_l)) I/3   (Pi' = sum_l c c (f_l - w_l)),
    // exact for D3Q19/D3Q27 because sum_l c c feq_l = rho u u + rho I/3.  For the regularized
    // populations the same tensor is the Vreman alpha (src/m_postcoll_kernel.F90:255-268), since
    // sum_l w_l H2_l H2_l : a2 * 4.5 = a2 on these lattices.
    R axx = 0, ayy = 0, azz = 0, axy = 0, axz = 0, ayz = 0;
    if (HRR || VRE) {
        const R third = R(1) / R(3);
        const R rux = rh * ux, ruy = rh * uy, ruz = rh * uz;
        axx = pxx * invS - rux * ux - dr * third;
        ayy = pyy * invS - ruy * uy - dr * third;
        azz = pzz * invS - ruz * uz - dr * third;
        axy = pxy * invS - rux * uy;
        axz = pxz * invS - rux * uz;
        ayz = pyz * invS - ruy * uz;
    }

    R fac = a.fac0;
    R tau = 0;
    if (VRE) {
        // Vreman (2004) eddy viscosity as src/m_postcoll_kernel.F90:270-304 forms it.
        R amag = axx * axx + ayy * ayy + azz * azz + R(2) * (axy * axy + axz * axz + ayz * ayz);
        amag = amag > a.tiny ? amag : a.tiny;
        const R b11 = a.eps + (axx * axx + axy * axy + axz * axz);
        const R b22 = a.eps + (axy * axy + ayy * ayy + ayz * ayz);
        const R b33 = a.eps + (axz * axz + ayz * ayz + azz * azz);
        const R b12 = a.eps + (axx * axy + axy * ayy + axz * ayz);
        const R b13 = a.eps + (axx * axz + axy * ayz + axz * azz);
        const R b23 = a.eps + (axy * axz + ayy * ayz + ayz * azz);
        const R bb = b11 * b22 - b12 * b12 + b11 * b33 - b13 * b13 + b22 * b33 - b23 * b23;
        const R t = bb * recip(amag);
        using std::sqrt;   // the tangent type brings its own sqrt
        const R eddy = t > a.eps ? a.vconst * sqrt(t) : R(0);
        tau = R(3) * (a.kinevisc + eddy + (AUX ? aux.abl : a.ablvisc[k - 1])) + R(0.5);
        fac = R(1) - recip(tau);
    }

    const R T = axx + ayy + azz;
    const R gx = axx * ux + axy * uy + axz * uz;
    const R gy = axy * ux + ayy * uy + ayz * uz;
    const R gz = axz * ux + ayz * uy + azz * uz;

    {   // rest population
        const R wS = weight<Q, R>(0) * S;
        const R e = wS * rb1;
        const R ne = HRR ? -(R(1.5) * wS) * T : D[0] - e;
        dev[0] = e + fac * ne;
    }
    // Factors shared by every direction of a weight class (|c|^2 = 1, 2, 3; directions 1, 7, 19
    // are the first of each class), hoisted out of the pair loop:
    //   even part  ev = kE0 + kE2 cu^2 + kF cAc
    //   odd part   od = kO cu pol + kF (cu (3 cAc - T) + c.(-2 g))
    //                 = cu (kA + kB cu^2 + kC cAc) + kF c.(-2 g)      (regularized)
    // with kE2 = wS*4.5rho, kO = wS*rho, kF = fac*4.5wS, kE0 = wS(rho base - 1) - kF T/3,
    // pol = 3 - 4.5 u.u + 4.5 cu^2 (third order) or 3, so kA = kO (3 - 4.5 u.u) - kF T or
    // 3 kO - kF T, kB = 4.5 kO or 0, kC = 3 kF.
    constexpr int NC = Q == 27 ? 3 : 2;
    R kE0[NC + 1], kE2[NC + 1], kO[NC + 1], kF[NC + 1], kA[NC + 1], kB[NC + 1], kC[NC + 1];
    const R T3 = T * (R(1) / R(3));
    const R P0 = R(3) - R(4.5) * usq;
#pragma unroll
    for (int n = 1; n <= NC; ++n) {
        const R wS = weight<Q, R>(n == 1 ? 1 : n == 2 ? 7 : 19) * S;
        kE2[n] = wS * r45;
        kO[n] = wS * rh;
        kF[n] = fac * (R(4.5) * wS);
        kE0[n] = HRR ? wS * rb1 - kF[n] * T3 : wS * rb1;
        kA[n] = (BGK3 ? kO[n] * P0 : R(3) * kO[n]) - kF[n] * T;
        kB[n] = R(4.5) * kO[n];
        kC[n] = R(3) * kF[n];
    }
    const R a2xy = R(2) * axy, a2xz = R(2) * axz, a2yz = R(2) * ayz;
    const R gmx = R(-2) * gx, gmy = R(-2) * gy, gmz = R(-2) * gz;
    // c.A.c by the axes c spans: one axis a_dd; two axes (a_dd + a_ee) +- 2 a_de; three axes
    // T + sxy 2a_xy + sxz 2a_xz + syz 2a_yz, whose signs multiply to +1, so with sxy fixed the
    // other two are (s, s) or (s, -s): T +- 2a_xy +- (2a_xz +- 2a_yz)
    const R exy = axx + ayy, exz = axx + azz, eyz = ayy + azz;
    const R tpp = T + a2xy, tmm = T - a2xy, up = a2xz + a2yz, um = a2xz - a2yz;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int l = 2 * p + 1;
        const int cx = Lt::cx(l), cy = Lt::cy(l), cz = Lt::cz(l);
        const int n2 = Lt::norm2(l);
        const R cu = sdot<R>(cx, cy, cz, ux, uy, uz);
        const R cu2 = cu * cu;
        if (HRR) {
            R cac;
            if (n2 == 1) cac = cx != 0 ? axx : cy != 0 ? ayy : azz;
            else if (n2 == 2) cac = cz == 0 ? (cx * cy > 0 ? exy + a2xy : exy - a2xy)
                                  : cy == 0 ? (cx * cz > 0 ? exz + a2xz : exz - a2xz)
                                            : (cy * cz > 0 ? eyz + a2yz : eyz - a2yz);
            else cac = cx * cy > 0 ? (cx * cz > 0 ? tpp + up : tpp - up) : (cx * cz > 0 ? tmm + um : tmm - um);
            const R ev = kE0[n2] + kE2[n2] * cu2 + kF[n2] * cac;
            const R in = BGK3 ? kA[n2] + kB[n2] * cu2 + kC[n2] * cac : kA[n2] + kC[n2] * cac;
            const R od = cu * in + kF[n2] * sdot<R>(cx, cy, cz, gmx, gmy, gmz);
            dev[l] = ev + od;
            dev[l + 1] = ev - od;
        } else {
            const R pol = BGK3 ? P0 + R(4.5) * cu2 : R(3);
            const R cp = cu * pol;
            const R e = kE0[n2] + kE2[n2] * cu2;   // S (E - w)
            const R o = kO[n2] * cp;               // S O
            dev[l] = (e + o) + fac * (D[l] - (e + o));
            dev[l + 1] = (e - o) + fac * (D[l + 1] - (e - o));
        }
    }

    // Equilibrium increments feq(rho, v) - feq(rho, u) for the inflow-turbulence forcing on
    // slice ip (src/m_inflow_turbulence_forcing.F90:57-128, added after the collision as
    // src/m_inflow_turbulence_apply.F90:21-26; third order when ibgk = 3) and for the external
    // body force (Kupershtokh exact difference with the 2nd-order equilibrium and du = -F/rho,
    // src/m_forcings_apply_kernel.F90:142-271; a cell with rho <= 0 is skipped).
    auto add_feq_diff = [&](R vx, R vy, R vz, auto order3) {
        constexpr bool O3 = decltype(order3)::value;
        const R vsq = vx * vx + vy * vy + vz * vz;
        const R vrb1 = rh * (R(1) - R(1.5) * vsq) - R(1);
        dev[0] = dev[0] + weight<Q, R>(0) * S * (vrb1 - rb1);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int l = 2 * p + 1;
            const R wS = weight<Q, R>(l) * S;
            const R cv = sdot<R>(Lt::cx(l), Lt::cy(l), Lt::cz(l), vx, vy, vz);
            const R cu = sdot<R>(Lt::cx(l), Lt::cy(l), Lt::cz(l), ux, uy, uz);
            R pv = R(3), pu = R(3);
            if (O3) { pv += R(4.5) * (cv * cv - vsq); pu += R(4.5) * (cu * cu - usq); }
            const R de = wS * ((vrb1 + r45 * cv * cv) - (rb1 + r45 * cu * cu));
            const R dodd = wS * (rh * (cv * pv) - rh * (cu * pu));
            dev[l] = dev[l] + (de + dodd);
            dev[l + 1] = dev[l + 1] + (de - dodd);
        }
    };
    if (a.tu != nullptr && i == a.ip) {
        const int sl = (k - 1) * L.ny + (j - 1);
        add_feq_diff(ux + a.ampl * a.tu[sl], uy + a.ampl * a.tv[sl], uz + a.ampl * a.tw[sl],
                     std::integral_constant<bool, BGK3>());
    }
    // force box: every interior cell for the caller's field, the deposit box for turbines (which the
    // tangent storage never has; the test is compiled out there, where it trips the register allocator)
    bool in_fbox = true;
    if constexpr (sizeof(R) <= 8)
        in_fbox = i >= a.flo[0] && i <= a.fhi[0] && j >= a.flo[1] && j <= a.fhi[1] && k >= a.flo[2] && k <= a.fhi[2];
    // One increment for both producers (a second inlined copy of add_feq_diff costs the unforced
    // kernels registers: D3Q19 BGK FP16 71 -> 101 VGPRs).
    if ((a.Fx != nullptr || a.theta != nullptr) && rh > R(0)) {
        R Fx = 0, Fy = 0, Fz = 0;
        bool forced = false;
        if (a.Fx != nullptr && in_fbox) {
            Fx = a.Fx[oc];
            Fy = a.Fy[oc];
            Fz = a.Fz[oc];
            forced = true;
        }
        if (a.theta != nullptr) {
            // buoyancy added to the forcing of every interior cell (src/m_buoyancy_forcing_kernel.F90:37,
            // the reference's operation order): F_z - scaling * (theta - theta0) / theta0
            Fz = Fz - (a.bscale * (a.theta[oc] - a.btheta0)) / a.btheta0;
            forced = true;
        }
        if (forced) {
            const R ir = recip(rh);
            add_feq_diff(ux - Fx * ir, uy - Fy * ir, uz - Fz * ir, std::integral_constant<bool, false>());
        }
    }

    // Solid cells: swap the opposite pairs (2,3),(4,5),... (src/m_solids.F90:19-32).
    if (a.solid != nullptr) {
        // rows of bits along the contiguous axis
        const uint32_t word = AUX ? aux.sword : a.solid[((cc - 1) * L.n(L.ax1) + (cb - 1)) * a.solid_wpr + ((ca - 1) >> 5)];
        if ((word >> ((ca - 1) & 31)) & 1u) {
#pragma unroll
            for (int l = 1; l + 1 < Q; l += 2) {
                const R t = dev[l];
                dev[l] = dev[l + 1];
                dev[l + 1] = t;
            }
        }
    }
    tau_out = tau;
}
template <int Q, class C, bool BGK3, bool HRR, bool VRE>
__host__ __device__ __forceinline__ void collide_cell(const StepArgs<typename C::real>& a, const typename C::raw (&rv)[Q], int i,
                                                      int j, int k, int ca, int cb, int cc, int oc,
                                                      typename C::real (&dev)[Q], typename C::real& tau_out) {
    collide_cell<Q, C, BGK3, HRR, VRE, false>(a, rv, CellAux<typename C::real>{}, i, j, k, ca, cb, cc, oc, true, dev, tau_out);
}

// Directions by run-time values, from packed constants (scalar shifts and masks).
template <int Q>
struct Outgoing {
    // populations with c_d > 0 (side 1) or < 0 (side 0), in lattice order, five bits each
    static constexpr int count = Q == 27 ? 9 : 5;
    static constexpr unsigned long long pack(int d, int side) {
        unsigned long long p = 0;
        int n = 0;
        for (int l = 0; l < Q; ++l)
            if (Lattice<Q>::c(l, d) == (side ? 1 : -1)) p |= (unsigned long long)l << (5 * n++);
        return p;
    }
    __device__ static __forceinline__ int pop(int d, int side, int q) {
        constexpr unsigned long long k[6] = {pack(0, 0), pack(0, 1), pack(1, 0), pack(1, 1), pack(2, 0), pack(2, 1)};
        const unsigned long long p = d == 0 ? (side ? k[1] : k[0]) : d == 1 ? (side ? k[3] : k[2]) : (side ? k[5] : k[4]);
        return (int)((p >> (5 * q)) & 31ull);
    }
};
template <int Q>
struct Direction {
    // the direction with velocity (x, y, z), 31 if the lattice has none
    static constexpr unsigned long long pack(int part) {
        unsigned long long p = 0;
        for (int e = 0; e < 9; ++e) {
            const int l = Lattice<Q>::find(part - 1, e / 3 - 1, e % 3 - 1);
            p |= (unsigned long long)(l < 0 ? 31 : l) << (5 * e);
        }
        return p;
    }
    __device__ static __forceinline__ int find(int x, int y, int z) {
        constexpr unsigned long long k[3] = {pack(0), pack(1), pack(2)};
        const unsigned long long p = x < 0 ? k[0] : x == 0 ? k[1] : k[2];
        return (int)((p >> (5 * (3 * (y + 1) + z + 1))) & 31ull);
    }
};

// Inflow ghost value (src/m_boundary_i_inflow_kernel.F90:61-74) from population l of cell (1, j, k):
// f_l - 2 w_l rho0 (c_x u cos(udir) + c_y u sin(udir)) / cs^2.
// The ghost takes it for c_x <= 0 and that of the opposite direction otherwise (:89-104).  Not
// contracted: the step kernel's unrolled directions and boundary_kernel's run-time ones round alike.
template <int Q, typename R>
__host__ __device__ __forceinline__ R inflow_ghost_value(R f, int l, R uu, R cosd, R sind, R rho0) {
#pragma clang fp contract(off)
    using Lt = Lattice<Q>;
    const R cs2 = R(1) / R(3);
    const R wl = weight<Q, R>(l);
    const R cxl = R(Lt::cx(l)), cyl = R(Lt::cy(l));
    return f - R(2) * wl * rho0 * (cxl * uu * cosd + cyl * uu * sind) / cs2;
}

// The boundary passes performed by the step kernel for its cell (i, j, k) (offset oc in f1, post-collision
// departures dev), when at most one axis D is closed (the other axes periodic, halo, or i carrying the
// inflow/outflow planes).
//
// Closed face (src/m_boundary_{i,j,k}_closed_kernel.F90): for ghost cell G of the face and outgoing l
// the reference sets
//   f1(m, G) = f2(l, G)                 (m = l reflected: normal negated, tangential * opt)
//   f1(l, G) = f1(l, G - c_l tangentially, on the wall plane).
// The cell x above G does the first; the second is pushed by the cell G - c_l that computed
// the value (periodic tangential axes wrapped), or, when G - c_l is a stored ghost of the
// inflow axis, copied from that ghost (still holding its value from before this step).
//
// Inflow/outflow (src/m_boundary_i_inflow_kernel.F90): the ghost row (j, k) of i is written by the cell
// with i = 1 (inflow ghost i = 0) or i = nx (outflow ghost i = nx+1, a copy of the cell) from the
// values it has just stored.  The face pass reads this ghost's value from before the step
// (f1(l, G - c_l) on the wall plane): those copies are made before the ghost is rewritten.
//
// All of a cell's loads are issued before the first of its ghost stores: one memory round trip where a
// copy at a time took up to twelve, each of them behind the stores before it, which was the whole time
// of a small grid.  (Issued before the cell's own 27 stores instead, they cost 20 registers.)
// Measured on MI355X, D3Q27 inflow and one closed axis, per step: FP32 60x14x5 11.6 -> 6.6 us,
// 384x200x128 416 -> 408 us, 384x192x128 351.5 -> 349.7 us; FP16 400x200x100 181 -> 178 us.
template <int Q, class C, int D, int SIDE>
__device__ __forceinline__ void fold_face(const StepArgs<typename C::real>& a, int i, int j, int k, int oc, bool at_end,
                                          const typename C::real (&dev)[Q]) {
    using raw = typename C::raw;
    using Lt = Lattice<Q>;
    constexpr int NO = Outgoing<Q>::count;
    constexpr unsigned long long out = Outgoing<Q>::pack(D, SIDE);
    constexpr int T0 = D == 0 ? 1 : 0, T1 = D == 2 ? 1 : 2;   // the axes along the face
    const Layout& L = a.lay;
    const int x[3] = {i, j, k};
    const int n[3] = {L.nx, L.ny, L.nz};
    const int per[3] = {L.per_i, L.per_j, L.per_k};
    const int st[3] = {L.si, L.sj, L.sk};
    const raw* __restrict__ f2 = static_cast<const raw*>(a.src);
    raw* __restrict__ f1 = static_cast<raw*>(a.dst);
    const int og = oc + (SIDE ? st[D] : -st[D]);
    raw above[NO], old[3];
#pragma unroll
    for (int q = 0; q < NO; ++q) above[q] = f2[(size_t)((out >> (5 * q)) & 31) * L.plane + og];
    // the inflow ghost's populations that leave the fluid through the face, by their movement along
    // the third axis
    const int ci = i == 1 ? 1 : -1;
    const bool copy_end = D > 0 && at_end;
    if (copy_end) {
#pragma unroll
        for (int o = 0; o < 3; ++o) {
            const int l = D == 1 ? Direction<Q>::find(ci, SIDE ? 1 : -1, o - 1) : Direction<Q>::find(ci, o - 1, SIDE ? 1 : -1);
            if (l < Q) old[o] = f1[(size_t)l * L.plane + oc - ci * st[0]];
        }
    }
    // a step c along each axis of the face: offset, and whether it stays in the face's range
    int off[2][3];
    bool ok[2][3];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int d = t ? T1 : T0;
        const int wrapd = per[d] ? n[d] * st[d] : 0;
        off[t][0] = -st[d] + (x[d] == 1 ? wrapd : 0);
        off[t][1] = 0;
        off[t][2] = st[d] - (x[d] == n[d] ? wrapd : 0);
        ok[t][0] = per[d] || x[d] > 1;
        ok[t][1] = true;
        ok[t][2] = per[d] || x[d] < n[d];
    }
#pragma unroll
    for (int l = 1; l < Q; ++l) {
        if (Lt::c(l, D) != (SIDE ? 1 : -1)) continue;
        const int c0 = Lt::c(l, T0) + 1, c1 = Lt::c(l, T1) + 1;
        if (ok[0][c0] && ok[1][c1])
            f1[(size_t)l * L.plane + (og + off[0][c0] + off[1][c1])] = C::template enc_dep<Q>(dev[l], l);
    }
    const int opt = SIDE ? a.fold_opt_hi : a.fold_opt_lo;
#pragma unroll
    for (int q = 0; q < NO; ++q) {
        const int l = (int)((out >> (5 * q)) & 31);
        f1[(size_t)(opt < 0 ? mirror<Q>(l, D, -1) : mirror<Q>(l, D, +1)) * L.plane + og] = above[q];
    }
    if (copy_end) {
        constexpr int t = T0 == 0 ? 1 : 0;   // the third axis
#pragma unroll
        for (int o = 0; o < 3; ++o) {
            const int l = D == 1 ? Direction<Q>::find(ci, SIDE ? 1 : -1, o - 1) : Direction<Q>::find(ci, o - 1, SIDE ? 1 : -1);
            if (l < Q && ok[t][o]) f1[(size_t)l * L.plane + (og + off[t][o])] = old[o];   // not ok: a halo ghost
        }
    }
    if (a.halo_dir < 0 && (a.inflow_fold || per[0])) return;
    // G - c_l beyond the face's range in a halo domain, or next to inflow planes of a separate pass.
    // On a halo plane only: the neighbour's value of this step, pushed by that halo's unpack.  On
    // the inflow axis only: copied above when the inflow planes are folded too, else here.  On both
    // (the inflow ghost of a halo plane): the value that ghost holds now, the neighbour's inflow
    // ghost from before this step.
#pragma unroll
    for (int l = 1; l < Q; ++l) {
        if (Lt::c(l, D) != (SIDE ? 1 : -1)) continue;
        int s[3] = {i, j, k};
        bool from_inflow = false, from_halo = false;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int d = t ? T1 : T0;
            s[d] = x[d] - Lt::c(l, d);
            if (per[d]) s[d] = Layout::wrap(s[d], n[d], 1);
            else if (s[d] < 1 || s[d] > n[d]) {
                if (d == a.halo_dir) from_halo = true;
                else from_inflow = true;
            }
        }
        if (from_inflow && (from_halo || !a.inflow_fold))
            f1[(size_t)l * L.plane + og] = f1[(size_t)l * L.plane + L.cell(s[0], s[1], s[2])];
    }
}

template <int Q, class C>
__device__ __forceinline__ void fold_boundaries(const StepArgs<typename C::real>& a, int i, int j, int k, int oc,
                                                const typename C::real (&dev)[Q]) {
    using R = typename C::real;
    using raw = typename C::raw;
    using Lt = Lattice<Q>;
    const Layout& L = a.lay;
    raw* __restrict__ f1 = static_cast<raw*>(a.dst);
    const bool at_end = a.inflow_fold && (i == 1 || i == L.nx) &&
                        (a.inflow_fold == 1 || (j > 1 && j < L.ny && k > 1 && k < L.nz));
    if (a.fold_dir == 0) {
        if (i == 1) fold_face<Q, C, 0, 0>(a, i, j, k, oc, false, dev);
        if (i == L.nx) fold_face<Q, C, 0, 1>(a, i, j, k, oc, false, dev);
    } else if (a.fold_dir == 1) {
        if (j == 1) fold_face<Q, C, 1, 0>(a, i, j, k, oc, at_end, dev);
        if (j == L.ny) fold_face<Q, C, 1, 1>(a, i, j, k, oc, at_end, dev);
    } else if (a.fold_dir == 2) {
        if (k == 1) fold_face<Q, C, 2, 0>(a, i, j, k, oc, at_end, dev);
        if (k == L.nz) fold_face<Q, C, 2, 1>(a, i, j, k, oc, at_end, dev);
    }
    if (!at_end) return;
    const int og = oc + (i == 1 ? -L.si : L.si);
    if (i == 1) {
        R fg[Q];
#pragma unroll
        for (int l = 0; l < Q; ++l) fg[l] = C::template decode<Q>(C::template enc_dep<Q>(dev[l], l), l);
        const R uu = a.utime * a.shear[k - 1];
#pragma unroll
        for (int l = 0; l < Q; ++l) fg[l] = inflow_ghost_value<Q, R>(fg[l], l, uu, a.cosd, a.sind, a.rho0);
#pragma unroll
        for (int l = 0; l < Q; ++l)
            f1[(size_t)l * L.plane + og] = C::template encode<Q>(Lt::cx(l) <= 0 ? fg[l] : fg[Lt::opposite(l)], l);
    } else {
#pragma unroll
        for (int l = 0; l < Q; ++l) f1[(size_t)l * L.plane + og] = C::template enc_dep<Q>(dev[l], l);
    }
}

#if defined(__HIP_DEVICE_COMPILE__)
// Raw buffer access of 2- or 4-byte values: base (scalar), byte offset voff (vector), byte offset
// soff (scalar), bounds nbytes.  The descriptor word 3 is the gfx9-family raw-buffer format.
template <typename raw>
__device__ __forceinline__ raw buffer_load(const void* base, int nbytes, uint32_t voff, uint32_t soff) {
    __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, nbytes, 0x00020000);
    if constexpr (sizeof(raw) == 2) return __builtin_bit_cast(raw, __builtin_amdgcn_raw_buffer_load_b16(r, (int)voff, (int)soff, 0));
    else return __builtin_bit_cast(raw, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
}
// NT: the non-temporal cache policy (aux bit 1), as the pointer path's non-temporal stores.
template <typename raw, bool NT>
__device__ __forceinline__ void buffer_store(void* base, int nbytes, uint32_t voff, uint32_t soff, raw v) {
    __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(base, 0, nbytes, 0x00020000);
    if constexpr (sizeof(raw) == 2)
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), r, (int)voff, (int)soff, NT ? 2 : 0);
    else
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, (int)voff, (int)soff, NT ? 2 : 0);
}
#endif

// One cell of the step at storage coordinates (cs, cb, cc) (1-based along ax0, ax1, ax2):
// gather the streamed populations, collide, store, and the folded face pass.  Columns cs past the
// row's last cell, up to store_end, store that cell's populations (Layout::row_store_end).
// VAR bit 0: non-temporal stores, bit 1: non-temporal loads (measured slower; kept for tuning),
// bit 3: the buffer is below 4 GiB (32-bit offsets from one base), bit 4: row-blocked buffers of
// any size addressed per slab of the slowest axis (one scalar base per source slab, 32-bit offsets
// within it; needs AXS >= 0 and a slab below 4 GiB).
// AXS >= 0: the contiguous storage axis is AXS (known at compile time, the other two in
// make_layout's order), so i, j, k map to (ca, cb, cc) without run-time selects, and the caller's
// wave-uniform cb, cc keep the row's offsets, wraps and checks in scalar registers.
template <int Q, class C, bool BGK3, bool HRR, bool VRE, int VAR, int AXS = -1>
__device__ __forceinline__ void step_cell(const StepArgs<typename C::real>& a, int cs, int cb, int cc) {
    using R = typename C::real;
    using raw = typename C::raw;
    using Lt = Lattice<Q>;
    const Layout& L = a.lay;
    if (cs > a.store_end || cb > L.n(L.ax1) || cc > L.n(L.ax2)) return;
    const int n0 = L.n(L.ax0);
    const int ca = cs < n0 ? cs : n0;
    int i, j, k;
    constexpr int A1 = AXS == 0 ? 1 : 0, A2 = AXS == 2 ? 1 : 2;
    if constexpr (AXS < 0) {
        L.ijk(ca, cb, cc, i, j, k);
    } else {
        i = AXS == 0 ? ca : A1 == 0 ? cb : cc;
        j = AXS == 1 ? ca : A1 == 1 ? cb : cc;
        k = AXS == 2 ? ca : A1 == 2 ? cb : cc;
    }

    // Source offsets: population l comes from (i - cx, j - cy, k - cz), periodic directions
    // folded onto the interior.  Index d = c + 1.
    // The cell's own offset is formed once; the neighbours' by adding the uniform stride, and
    // for a periodic axis at its first/last cell by the uniform wrap distance (no per-offset
    // multiplies).
    const int s = a.stream;
    // the contiguous axis has unit stride in both buffer arrangements (make_layout)
    const int oc0 = AXS < 0 ? L.cell(i, j, k)
                            : L.base + ca + cb * (A1 == 0 ? L.si : A1 == 1 ? L.sj : L.sk) +
                                  cc * (A2 == 0 ? L.si : A2 == 1 ? L.sj : L.sk);
    int ox[3], oy[3], oz[3];
    auto offsets = [&](int x, int n, int per, int st, int (&o)[3]) {
        // o[d]: offset change of the source x - s*(d-1) along this axis
        const int wrapd = per ? n * st : 0;
        const int lo = (per && x == n) ? -wrapd : 0;   // x + 1 wraps to 1
        const int hi = (per && x == 1) ? wrapd : 0;    // x - 1 wraps to n
        o[0] = s * (st + lo);                          // source x + 1 (c = -1)
        o[1] = 0;
        o[2] = -s * (st - hi);                         // source x - 1 (c = +1)
    };
    offsets(i, L.nx, L.per_i, L.si, ox);
    offsets(j, L.ny, L.per_j, L.sj, oy);
    offsets(k, L.nz, L.per_k, L.sk, oz);
    // slab form (VAR bit 4): offsets stay relative, the cell's own offset is split into its slab's
    // start and its offset within the slab
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr bool SLAB = (VAR & 16) != 0 && AXS >= 0 && (sizeof(raw) == 2 || sizeof(raw) == 4);
#else
    constexpr bool SLAB = false;
#endif
    if constexpr (!SLAB) {
        ox[0] += oc0;
        ox[1] += oc0;
        ox[2] += oc0;
    }
    // per-cell arrays, and (16-bit storage) the collision's per-cell inputs read ahead of the
    // populations
    const int occ = AXS < 0 ? L.cidx(i, j, k)
                            : L.base + ca + cb * (A1 == 0 ? L.ci : A1 == 1 ? L.cj : L.ck) +
                                  cc * (A2 == 0 ? L.ci : A2 == 1 ? L.cj : L.ck);
    constexpr bool AUX = sizeof(raw) == 2;
    CellAux<R> aux{};
    if constexpr (AUX) aux = cell_aux<VRE>(a, k, ca, cb, cc);
    // Plane bases are uniform (scalar registers); the per-lane part is a 32-bit byte offset
    // within a plane (planes are below 4 GiB), so loads and stores take the scalar-base form
    // without 64-bit address arithmetic per population.
    // With VAR bit 3 the whole buffer is below 4 GiB: one scalar base and 32-bit offsets that
    // include the plane (two scalar registers instead of one pair per plane).
    const char* __restrict__ srcb = static_cast<const char*>(a.src);
    const size_t pbytes = (size_t)L.plane * sizeof(raw);
    const uint32_t pb32 = (uint32_t)pbytes;
    raw rv[Q];
    // 2- and 4-byte storage in a buffer below 4 GiB: raw buffer loads/stores, the plane offset in
    // the scalar offset operand, so an access costs no vector address arithmetic at all.
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr bool BUF = (VAR & 8) != 0 && (sizeof(raw) == 2 || sizeof(raw) == 4);
#else
    constexpr bool BUF = false;
#endif
    // descriptor byte count: an unsigned 32-bit field (the variant runs only below 4 GiB)
    const size_t tbytes = (size_t)L.total * sizeof(raw);
    const int nbytes = (int)(uint32_t)(tbytes < 0xffffffffull ? tbytes : 0xffffffffull);
    // slab form: the element offset of the cell within its slab of the slowest axis and the slab's
    // start; a source's slab start moves by the ax2 offset (wrap included), its offset within the
    // slab by the ax0 and ax1 offsets
    const int s2 = A2 == 0 ? L.si : A2 == 1 ? L.sj : L.sk;
    const int (&d0)[3] = AXS == 0 ? ox : AXS == 1 ? oy : oz;
    const int (&d1)[3] = A1 == 0 ? ox : A1 == 1 ? oy : oz;
    const int (&d2)[3] = A2 == 0 ? ox : A2 == 1 ? oy : oz;
    const int w0 = SLAB ? oc0 - cc * s2 : 0;      // cell offset within its slab
    const size_t slab0 = SLAB ? (size_t)cc * (size_t)s2 : 0;
    const int sbytes = (int)(((uint32_t)s2 + (uint32_t)line_elems(sizeof(raw))) * (uint32_t)sizeof(raw));
#pragma unroll
    for (int l = 0; l < Q; ++l) {
        if constexpr (SLAB) {
#if defined(__HIP_DEVICE_COMPILE__)
            const int c0 = Lt::c(l, AXS), c1 = Lt::c(l, A1), c2 = Lt::c(l, A2);
            const char* sb = srcb + (size_t)((long long)slab0 + d2[c2 + 1]) * sizeof(raw);
            rv[l] = buffer_load<raw>(sb, sbytes, (uint32_t)(w0 + d0[c0 + 1] + d1[c1 + 1]) * (uint32_t)sizeof(raw),
                                     (uint32_t)l * pb32);
#endif
            continue;
        }
        const uint32_t offe = (uint32_t)(oz[Lt::cz(l) + 1] + oy[Lt::cy(l) + 1] + ox[Lt::cx(l) + 1]);
        const uint32_t off = offe * (uint32_t)sizeof(raw);
        if constexpr (BUF) {
#if defined(__HIP_DEVICE_COMPILE__)
            rv[l] = buffer_load<raw>(srcb, nbytes, off, (uint32_t)l * pb32);
#endif
            continue;
        }
        const raw* p;
        if constexpr ((VAR & 8) != 0) p = reinterpret_cast<const raw*>(srcb + (off + (uint32_t)l * pb32));
        else p = reinterpret_cast<const raw*>(srcb + (size_t)l * pbytes + (size_t)offe * sizeof(raw));
        if constexpr ((VAR & 2) != 0) rv[l] = __builtin_nontemporal_load(p);
        else rv[l] = *p;
    }

    R out[Q];
    R tau = 0;
    const int oc = oc0 + (cs - ca);   // unit stride along ax0
    collide_cell<Q, C, BGK3, HRR, VRE, AUX>(a, rv, aux, i, j, k, ca, cb, cc, occ, cs == ca, out, tau);

    char* __restrict__ dstb = static_cast<char*>(a.dst);
    const uint32_t ob = (uint32_t)oc * (uint32_t)sizeof(raw);
#pragma unroll
    for (int l = 0; l < Q; ++l) {
        if constexpr (SLAB) {
#if defined(__HIP_DEVICE_COMPILE__)
            buffer_store<raw, (VAR & 1) != 0>(dstb + slab0 * sizeof(raw), sbytes, (uint32_t)(w0 + (cs - ca)) * (uint32_t)sizeof(raw),
                                              (uint32_t)l * pb32, C::template enc_dep<Q>(out[l], l));
#endif
            continue;
        }
        if constexpr (BUF) {
#if defined(__HIP_DEVICE_COMPILE__)
            buffer_store<raw, (VAR & 1) != 0>(dstb, nbytes, ob, (uint32_t)l * pb32, C::template enc_dep<Q>(out[l], l));
#endif
            continue;
        }
        raw* p;
        if constexpr ((VAR & 8) != 0) p = reinterpret_cast<raw*>(dstb + (ob + (uint32_t)l * pb32));
        else p = reinterpret_cast<raw*>(dstb + (size_t)l * pbytes + (size_t)(uint32_t)oc * sizeof(raw));
        if constexpr ((VAR & 1) != 0) __builtin_nontemporal_store(C::template enc_dep<Q>(out[l], l), p);
        else *p = C::template enc_dep<Q>(out[l], l);
    }
    if (cs != ca) return;
    if (VRE && a.tau_out != nullptr) a.tau_out[occ] = tau;
    if (a.fold_dir >= 0 || a.inflow_fold) fold_boundaries<Q, C>(a, i, j, k, oc0, out);
}

// Threads run along the storage axes: x along the contiguous axis ax0, y along ax1, z along ax2.
// heavy_first bit 0 (ax1) / bit 1 (ax2): that axis's cells are taken in the order 1, n, 2, 3, ..,
// n-1, so that the rows and planes of a folded face or of the folded inflow/outflow planes, which
// carry extra stores, are dispatched first (blocks start in x, y, z order) instead of forming the
// launch's tail.
__device__ __forceinline__ int heavy_order(int x, int n) { return x == 0 ? 1 : x == 1 ? n : x; }

// With xcd_groups (several blocks along ax0 per row group), the blocks of one row group run on one
// XCD: workgroups are dispatched to the 8 XCDs in turn, so hardware block b (x fastest) works on
// row group ((b / 8) / gx) * 8 + b % 8, segment (b / 8) % gx.  The segments of a row group share the
// cache lines at their edges (the +-1 shift along ax0), which another XCD's L2 would fetch again;
// consecutive row groups still go to different XCDs.  Blocks past the last full set of 8 row
// groups keep their own position.
// AXS >= 0: step_cell's compile-time contiguous axis; the row coordinate is then taken as wave-uniform
// (block_x is a multiple of 64, so each wave lies in one row).
template <int Q, class C, bool BGK3, bool HRR, bool VRE, int VAR, int AXS = -1>
__global__ void __launch_bounds__(sizeof(typename C::raw) >= 8 ? 256 : 1024, sizeof(typename C::raw) >= 8 ? 3 : 1) step_kernel(const StepArgs<typename C::real> a) {
    int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
    // (compiled out for the 16-byte tangent storage, which keeps the plain order: the order code
    // there makes the compiler's register allocator fail)
    if (sizeof(typename C::raw) <= 8 && a.xcd_groups) {
        const int gx = gridDim.x, gy = gridDim.y;
        const int b = bx + gx * (by + gy * bz);
        const int rows = gy * gridDim.z;
        if (b < 8 * gx * (rows / 8)) {
            const int slot = b >> 3;
            const int r = (slot / gx) * 8 + (b & 7);
            bx = slot % gx;
            by = r % gy;
            bz = r / gy;
        }
    }
    int y = by * blockDim.y + threadIdx.y;
    if constexpr (AXS >= 0) y = __builtin_amdgcn_readfirstlane(y);
    if (a.part) {
        // launch coordinate along the halo axis -> the part's cell (part_row)
        const int n = a.lay.n(a.part_axis == 1 ? a.lay.ax1 : a.lay.ax2);
        const int m = part_row(a.part_axis == 1 ? y : bz, a.part, n, a.part_edge);
        if (a.part_axis == 1) y = m;
        else bz = m;
    }
    const int n1 = a.lay.n(a.lay.ax1);
    const int cb = (a.heavy_first & 1) && y < n1 ? heavy_order(y, n1) : y + 1;
    const int cc = (a.heavy_first & 2) ? heavy_order(bz, a.lay.n(a.lay.ax2)) : bz + 1;
    step_cell<Q, C, BGK3, HRR, VRE, VAR, AXS>(a, bx * blockDim.x + threadIdx.x + 1, cb, cc);
}

// ------------------------------------------------------------------------------------------
// Boundary kernel (non-periodic ghost layers).
// ------------------------------------------------------------------------------------------
template <typename R>
struct BoundaryArgs {
    Layout lay;
    void* f1;
    const void* f2;
    int face[3];               // the axis has closed faces (all of them are this launch's)
    int opt_lo[3], opt_hi[3];
    int face_blocks[3];        // blocks of 256 threads: sides x populations x the face's area
    int ta[3];                 // the face's axis that is stored first
    int inflow;                // i has inflow/outflow planes
    int inflow_blocks;         // their blocks; 0: not this launch's
    int inflow_rim;            // only their rows along the walls of j and k
    const R* shear;            // uvel_shear(nz)
    R utime, cosd, sind, rho0;
    EdgeList edges;
};
template <int Q, class C>
__device__ __forceinline__ typename C::real ld(const Layout& L, const void* f, int l, int off) {
    return C::template decode<Q>(static_cast<const typename C::raw*>(f)[(size_t)l * (size_t)L.plane + (size_t)off], l);
}
template <int Q, class C>
__device__ __forceinline__ void st(const Layout& L, void* f, int l, int off, typename C::real v) {
    static_cast<typename C::raw*>(f)[(size_t)l * (size_t)L.plane + (size_t)off] = C::template encode<Q>(v, l);
}
// boundarycond's passes over the ghost layers of the non-periodic axes (src/m_boundarycond.F90:166-365)
// in one launch: closed faces (src/m_boundary_{i,j,k}_closed_kernel.F90), edges and corners
// (src/m_boundary_{j_k,i_j,i_k}_edges.F90, src/m_boundary_closed_corners.F90) and the inflow/outflow
// planes of i (src/m_boundary_i_inflow_kernel.F90:61-111).  f1 is the buffer the step just wrote, f2
// the other one.  For l pointing out of the fluid at ghost G the reference sets
//   f1(m, G) = f2(l, G)       m = l reflected at the wall,
//   f1(l, G) = f1(l, S)       S = G - c_l on the wall plane (faces: moved along the face only),
// face after face in the order i, j, k, then edges and corners, then inflow/outflow.
//
// The passes are latency: a few thousand threads each, one after the other, each thread with all the
// loads and stores of its ghost cell (with i contiguous every one of them in a line of its own).
// Here every written value has a thread of its own, and one launch takes the place of up to seven.
// That needs no value to be read after another thread may have replaced it:
//   * S in the interior: no pass writes it;
//   * S on the ghost plane of a closed axis E that comes before the face's: the passes leave there
//     f2(l', S), l' = l reflected at E, which is read instead;
//   * S on a plane that comes later (E > D, the inflow planes, an edge), or the copy that the first
//     periodic pass made of such a cell (S beyond a periodic axis too): the value from before this
//     call, which the thread that replaces it passes on first;
//   * S on an inflow plane and a closed axis at once: no pass writes it.
// Measured on MI355X, FP32, per step: closed box 101x61x45 (three closed axes) 38.4 us in four launches
// -> 7.9 us; duct 250x98x70 (inflow, two closed axes) 52.1 us in four launches -> 25.5 us (a kernel trace, which
// runs launches apart).  The inflow planes were most of the duct's: with i contiguous, four lines for every value.
// Where the step kernel's end cells write them but for the rows along the walls (inflow_fold = 2), the launch
// takes 11.6 us and the step kernel 78 instead of 66 us in the trace; untraced a step takes 84 us instead of 90.
template <int Q, class C>
__global__ void __launch_bounds__(256) boundary_kernel(const BoundaryArgs<typename C::real> a) {
    using R = typename C::real;
    using raw = typename C::raw;
    const Layout& L = a.lay;
    raw* __restrict__ f1 = static_cast<raw*>(a.f1);
    const raw* __restrict__ f2 = static_cast<const raw*>(a.f2);
    const int n[3] = {L.nx, L.ny, L.nz};
    const int per[3] = {L.per_i, L.per_j, L.per_k};
    auto at = [&](int l, const int (&x)[3]) { return (size_t)l * (size_t)L.plane + (size_t)L.cell(x[0], x[1], x[2]); };
    // the axis' coordinate x moved by c: the periodic image, or false beyond another axis' range
    auto inside = [&](int d, int& x, bool& wrapped) {
        if (x >= 1 && x <= n[d]) return true;
        if (!per[d]) return false;
        x = Layout::wrap(x, n[d], 1);
        wrapped = true;
        return true;
    };
    // Passes the value of slot (l, x), x on the ghost plane of axis E, on to the face of axis A whose
    // pass reads it: A's wall plane holds x and l leaves the fluid there.  late: this slot's own pass
    // comes after A's; otherwise only the copy beyond a periodic axis is passed on.
    auto pass_on = [&](int l, const int (&x)[3], int E, int A, bool late) {
        const int cA = Lattice<Q>::c(l, A);
        if (!(a.face[A] && cA != 0 && x[A] == (cA < 0 ? 1 : n[A]))) return;
        const int T = 3 - E - A;
        int g[3];
        g[A] = x[A] + cA;
        g[E] = x[E] + Lattice<Q>::c(l, E);
        g[T] = x[T] + Lattice<Q>::c(l, T);
        bool wrapped = false;
        if (!inside(T, g[T], wrapped) || !(late || wrapped)) return;
        f1[at(l, g)] = f1[at(l, x)];
    };

    int b = blockIdx.x;
    // ---- closed faces: (along the face, population of the side)
#pragma unroll 1
    for (int D = 0; D < 3; ++D) {
        if (b >= a.face_blocks[D]) {
            b -= a.face_blocks[D];
            continue;
        }
        const int T0 = a.ta[D], T1 = 3 - D - T0;
        const int area = n[T0] * n[T1];
        const int per_pop = (area + 255) / 256;
        const int sq = b / per_pop;                       // side, population: the same for a block
        const int e = (b - sq * per_pop) * 256 + threadIdx.x;
        if (e >= area) return;
        const int side = sq >= Outgoing<Q>::count;
        const int l = Outgoing<Q>::pop(D, side, sq - side * Outgoing<Q>::count);
        const int opt = side ? a.opt_hi[D] : a.opt_lo[D];
        int c[3], g[3], s[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) c[d] = Lattice<Q>::c(l, d);
        g[D] = side ? n[D] + 1 : 0;
        g[T1] = e / n[T0] + 1;
        g[T0] = e - (g[T1] - 1) * n[T0] + 1;
        // the value that streams along the wall
        s[D] = side ? n[D] : 1;
        bool wrapped = false, mine = true;
        int E = -1, out = 0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int T = q ? T1 : T0;
            s[T] = g[T] - c[T];
            if (!inside(T, s[T], wrapped)) {
                ++out;
                if (!(a.inflow && T == 0)) E = T;
            }
        }
        raw along;
        if (out == 0 || (out == 2 && a.inflow)) along = f1[at(l, s)];
        else if (out == 1 && E >= 0 && E < D && !wrapped) {
            const int o = s[E] < 1 ? a.opt_lo[E] : a.opt_hi[E];
            int r[3] = {o * c[0], o * c[1], o * c[2]};
            r[E] = -c[E];
            along = f2[at(Direction<Q>::find(r[0], r[1], r[2]), s)];
        } else {
            mine = false;                                  // passed on by the slot's own thread
        }
        int r[3] = {opt * c[0], opt * c[1], opt * c[2]};
        r[D] = -c[D];
        const int m = Direction<Q>::find(r[0], r[1], r[2]);
        pass_on(m, g, D, T0, D > T0);
        pass_on(m, g, D, T1, D > T1);
        f1[at(m, g)] = f2[at(l, g)];
        if (mine) f1[at(l, g)] = along;
        return;
    }
    // ---- inflow/outflow planes: (along the plane, population)
    if (b < a.inflow_blocks) {
        const int T0 = a.ta[0], T1 = 3 - T0;
        const int area = a.inflow_rim ? inflow_rim_cells(n[T0], n[T1]) : n[T0] * n[T1];
        const int per_pop = (area + 255) / 256;
        const int l = b / per_pop;
        const int e = (b - l * per_pop) * 256 + threadIdx.x;
        if (e >= area) return;
        int x[3];
        if (a.inflow_rim) {
            inflow_rim_cell(e, n[T0], n[T1], x[T0], x[T1]);
        } else {
            x[T1] = e / n[T0] + 1;
            x[T0] = e - (x[T1] - 1) * n[T0] + 1;
        }
        const int cx = Lattice<Q>::cx(l);
        const int src = cx <= 0 ? l : Lattice<Q>::opposite(l);
        x[0] = 1;
        R v = C::template decode<Q>(f1[at(src, x)], src);
        v = inflow_ghost_value<Q, R>(v, src, a.utime * a.shear[x[2] - 1], a.cosd, a.sind, a.rho0);
        x[0] = n[0];
        const raw keep = f1[at(l, x)];
        x[0] = 0;
        if (cx > 0) {
            pass_on(l, x, 0, 1, true);
            pass_on(l, x, 0, 2, true);
        }
        f1[at(l, x)] = C::template encode<Q>(v, l);
        x[0] = n[0] + 1;
        if (cx < 0) {
            pass_on(l, x, 0, 1, true);
            pass_on(l, x, 0, 2, true);
        }
        f1[at(l, x)] = keep;
        return;
    }
    b -= a.inflow_blocks;
    // ---- edges and corners: (along the edge, velocity along it)
    const int t = b * 256 + threadIdx.x;
    int q = 0, k = t;
    while (q < a.edges.n && k >= 3 * a.edges.len[q]) k -= 3 * a.edges.len[q++];
    if (q >= a.edges.n) return;
    const EdgeList& e = a.edges;
    int g[3] = {e.g[q][0], e.g[q][1], e.g[q][2]}, c[3] = {e.out[q][0], e.out[q][1], e.out[q][2]}, s[3];
    const int T = e.t[q];
    if (e.kind[q] == 0) {
        g[T] = k % e.len[q] + 1;
        c[T] = k / e.len[q] - 1;
    } else if (k > 0) {
        return;
    }
    const int l = Direction<Q>::find(c[0], c[1], c[2]);
    if (l >= Q) return;
#pragma unroll
    for (int d = 0; d < 3; ++d) s[d] = e.out[q][d] != 0 ? g[d] - c[d] : g[d];
    const raw along = f1[at(l, s)];
    const int m = Direction<Q>::find(e.mir[q][0] * c[0], e.mir[q][1] * c[1], e.mir[q][2] * c[2]);
    if (m < Q) {
        // the face at the end of the edge reads what the edge held
        const int cT = Lattice<Q>::c(m, T);
        if (e.kind[q] == 0 && a.face[T] && cT != 0 && g[T] == (cT < 0 ? 1 : n[T])) {
            int x[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) x[d] = g[d] + Lattice<Q>::c(m, d);
            f1[at(m, x)] = f1[at(m, g)];
        }
        f1[at(m, g)] = f2[at(l, g)];
    }
    f1[at(l, g)] = along;
}

// The ghosts that a step needs its output buffer to hold beforehand, copied from src to dst: dst then
// receives the step as if it had received the one before the last (the adjoint's recompute writes each
// step into a snapshot slot of its own instead of ping-ponging two buffers).  With at most one closed axis
// D a step rewrites every ghost that anything reads but two kinds, both at an inflow plane of i next to a
// closed D (j or k), which is where the kernel copies: the edges (D = 0, n + 1), which no pass writes, and the
// wall planes (D = 1, n), whose values from before the step the face pass reads.  (Populations that
// move along a closed face are neither written nor read in its ghosts.)  One thread per value, along the
// periodic axis T.  Copying the whole shell, a thread per ghost cell, took 11.4 us of a D3Q19 FP32 step
// of 192x96x96 cells; this takes 4.8 us.
template <int Q, class C>
__global__ void __launch_bounds__(256) ghost_keep_kernel(Layout L, const void* src, void* dst, int D) {
    using raw = typename C::raw;
    const int T = 3 - D;
    const unsigned nt = (unsigned)L.n(T), e = blockIdx.x * 256 + threadIdx.x;
    const unsigned q = e / nt;
    if (q >= 8u * Q) return;
    const unsigned l = q / 8;
    const int n = L.n(D), w = (int)(q & 3);
    int x[3];
    x[0] = (q & 4) ? L.nx + 1 : 0;
    x[D] = w == 0 ? 0 : w == 1 ? 1 : w == 2 ? n : n + 1;
    x[T] = (int)(e - q * nt) + 1;
    const size_t o = (size_t)l * (size_t)L.plane + (size_t)L.cell(x[0], x[1], x[2]);
    static_cast<raw*>(dst)[o] = static_cast<const raw*>(src)[o];
}

// ------------------------------------------------------------------------------------------
// Halo planes of j for a domain tiled along j (src/m_mpi_pack_jplane.F90,
// src/m_mpi_unpack_jplane.F90, exchanged in src/m_mpi_halo_exchange_j.F90:55-120).  A halo holds
// only the populations that cross the plane: pack side 0 sends plane j = 1's populations with
// c_y = -1 (to the neighbour below), side 1 plane j = ny's with c_y = +1; unpack side 0 fills
// ghost j = 0 with c_y = +1 populations, side 1 ghost j = ny+1 with c_y = -1.  Buffer order
// [q][k = 0..nz+1][i = 0..nx+1], q counting those populations in lattice order (both sides: side
// 0's halo, then side 1's); values in the storage encoding.
// ------------------------------------------------------------------------------------------
template <int Q>
__host__ __device__ constexpr int halo_count() { return Q == 27 ? 9 : 5; }

// the q-th population with c_y = cy
template <int Q>
__device__ __forceinline__ int halo_pop(int q, int cy) {
    int n = 0;
#pragma unroll
    for (int l = 0; l < Q; ++l)
        if (Lattice<Q>::cy(l) == cy) {
            if (n == q) return l;
            ++n;
        }
    return -1;
}

// One thread per buffer element e = ((h * count + q) * (nz+2) + k) * (nx+2) + i over the nside
// sides side0 .. side0 + nside - 1 (h = side - side0); with both sides the buffer holds side 0's
// halo and then side 1's.
struct HaloIdx {
    int i, k, q, h;
};
template <int Q>
__device__ __forceinline__ bool halo_index(const Layout& L, int nside, HaloIdx& x) {
    const unsigned e = blockIdx.x * blockDim.x + threadIdx.x;
    const unsigned ni = L.nx + 2, nk = L.nz + 2;
    if (e >= (unsigned)nside * halo_count<Q>() * nk * ni) return false;
    x.i = e % ni;
    const unsigned r = e / ni;
    x.k = r % nk;
    const unsigned qh = r / nk;
    x.q = qh % halo_count<Q>();
    x.h = qh / halo_count<Q>();
    return true;
}

template <int Q, class C>
__global__ void __launch_bounds__(256) halo_pack_kernel(Layout L, const void* f, int side0, int nside, void* buf) {
    using raw = typename C::raw;
    HaloIdx x;
    if (!halo_index<Q>(L, nside, x)) return;
    const int side = side0 + x.h;
    const int l = halo_pop<Q>(x.q, side ? 1 : -1);
    const int j = side ? L.ny : 1;
    static_cast<raw*>(buf)[blockIdx.x * blockDim.x + threadIdx.x] =
        static_cast<const raw*>(f)[(size_t)l * L.plane + L.cell(x.i, j, x.k)];
}

// Unpack, and the closed-face pass's copies whose source lies on this halo plane: for ghost G of
// the face of fold_dir and population l pointing out of the fluid, f(l, G) = f(l, G - c_l) on the
// wall plane (src/m_boundary_k_closed_kernel.F90:39-41); when G - c_l is on the halo plane it is
// the neighbour's value of this step, which only the halo brings.  Sources on a ghost of another
// non-periodic axis (the inflow ghost of the halo plane) are left to the step kernel, which reads
// them before this unpack replaces them.
template <int Q, class C>
__global__ void __launch_bounds__(256) halo_unpack_kernel(Layout L, void* f, int side0, int nside, const void* buf,
                                                          int fold_dir) {
    using raw = typename C::raw;
    using Lt = Lattice<Q>;
    HaloIdx hx;
    if (!halo_index<Q>(L, nside, hx)) return;
    const int i = hx.i, k = hx.k;
    const int side = side0 + hx.h;
    const int cy = side ? -1 : 1;
    const int l = halo_pop<Q>(hx.q, cy);
    const int j = side ? L.ny + 1 : 0;
    raw* __restrict__ p = static_cast<raw*>(f);
    const raw v = static_cast<const raw*>(buf)[blockIdx.x * blockDim.x + threadIdx.x];
    p[(size_t)l * L.plane + L.cell(i, j, k)] = v;
    const int D = fold_dir;
    if (D != 0 && D != 2) return;
    const int x[3] = {i, j, k};
    const int n[3] = {L.nx, L.ny, L.nz};
    const int O = 2 - D;   // the face's tangential axis other than j
    if (x[O] < 1 || x[O] > n[O]) return;
    const int cD = Lt::c(l, D);
    const int side_d = x[D] == 1 && cD < 0 ? 0 : x[D] == n[D] && cD > 0 ? 1 : -1;
    if (side_d < 0) return;
    int t[3];
    t[1] = j + cy;
    t[D] = side_d ? n[D] + 1 : 0;
    t[O] = x[O] + Lt::c(l, O);
    const int perO = O == 0 ? L.per_i : L.per_k;
    if (perO) t[O] = Layout::wrap(t[O], n[O], 1);
    else if (t[O] < 1 || t[O] > n[O]) return;
    p[(size_t)l * L.plane + L.cell(t[0], t[1], t[2])] = v;
}

// ------------------------------------------------------------------------------------------
// Ensembles: many domains of one lattice, storage and collision model advanced by one launch of
// a kernel per step.  Every domain's rows are cut into segments of 64 bytes, and the
// segments of each (ax0, ax1) plane into tiles of blockDim.x cells; the tiles of all members form one
// list that the blocks of the grid walk with stride gridDim.x (by default a block for each).  Whole segments matter: tiles of
// consecutive cells, which the first form cut regardless of rows, left lines of rows that are no
// multiple of 64 cells to two waves, whose separate partial stores memory read and wrote twice.
// Measured on MI355X, D3Q19 per step: 16 members of about 112x84x70 cells (10.8 M) FP32 560 -> 319 us,
// FP64 880 -> 641 us, FP16 388 -> 242 us; 64 of about 28x21x17 (0.61 M) FP32 59 -> 46 us; 16 members of 96-160x64-96x64-96 (14.2 M), most rows aligned before, 402 ->
// 386 us.
//
// A step is one plain launch, with the step number and the buffers' parity as arguments.  Captured in
// graphs of 16 steps, which had to read them from a device clock, the steps were further apart than
// launches queued on a stream: 64 small members FP32 46.3 -> 42.9 us per step, FP16 44.4 -> 39.9 us, 16
// ordinary ones FP16 242 -> 232 us, FP32 and FP64 as before.  Each member's closed face and inflow/outflow planes are folded into the
// step (at most one closed axis per member).
// ------------------------------------------------------------------------------------------
template <typename R>
struct MemberTab {
    StepArgs<R> a;          // src, dst, tu, tv, tw are set per step
    void* buf[2];
    int cur0;               // buffer holding the current state when the table was made
    int nrturb, slice;      // turbulence slices of ny*nz reals; nrturb = 0: off
    const R* turb[3];       // slice 0 of uu, vv, ww
    int seg_row, tiles_plane;   // segments per row; tiles per (ax0, ax1) plane
    int start;              // the member's first tile
};

// Cells of a segment.
template <typename raw>
constexpr int kSegment = 64 / (int)sizeof(raw);

// it: the step; s: steps done since the table was made; vals: the step's (uvel_time(it), cos(udir),
// sin(udir)) per member; owner: the member of each tile.
template <int Q, class C, bool BGK3, bool HRR, bool VRE>
__global__ void __launch_bounds__(1024) step_kernel_batch(const MemberTab<typename C::real>* __restrict__ tab,
                                                          const int* __restrict__ owner, int total, int it, int s,
                                                          const typename C::real* __restrict__ vals) {
    using R = typename C::real;
    constexpr unsigned W = kSegment<typename C::raw>;
    for (int t = blockIdx.x; t < total; t += gridDim.x) {
        const int m = owner[t];
        const MemberTab<R>& M = tab[m];
        StepArgs<R> a = M.a;
        const int p = (M.cur0 + s) & 1;
        a.src = M.buf[p];
        a.dst = M.buf[p ^ 1];
        if (a.inflow_fold) {
            const R* v = vals + (size_t)m * 3;
            a.utime = v[0];
            a.cosd = v[1];
            a.sind = v[2];
        }
        if (M.nrturb > 0) {
            int lit = it % M.nrturb;             // src/m_inflow_turbulence_forcing.F90:45-46
            if (lit == 0) lit = M.nrturb;
            const size_t off = (size_t)lit * M.slice;
            a.tu = M.turb[0] + off;
            a.tv = M.turb[1] + off;
            a.tw = M.turb[2] + off;
        }
        const int local = t - M.start;
        const int cc = local / M.tiles_plane;
        const unsigned e = (unsigned)(local - cc * M.tiles_plane) * blockDim.x + threadIdx.x;
        const unsigned u = e / W;
        const unsigned cb = u / (unsigned)M.seg_row;
        step_cell<Q, C, BGK3, HRR, VRE, 1>(a, (int)((u - cb * (unsigned)M.seg_row) * W + e % W) + 1, (int)cb + 1, cc + 1);
    }
}

// ------------------------------------------------------------------------------------------
// State transfer between the reference's layout f(nl,0:nx+1,0:ny+1,0:nz+1) and the device buffers
// (H = float or double, the caller's REAL kind): what the tiled kernels of fields.h do with a cell.
// ------------------------------------------------------------------------------------------
template <int Q, class C>
struct StateIn {
    void* a;
    void* b;   // nullptr: one buffer only
    template <typename H>
    __device__ void operator()(const Layout& L, int i, int j, int k, const H (&f)[Q]) const {
        const int oc = L.cell(i, j, k);
#pragma unroll
        for (int l = 0; l < Q; ++l) {
            const typename C::real v = (typename C::real)f[l];
            st<Q, C>(L, a, l, oc, v);
            if (b) st<Q, C>(L, b, l, oc, v);
        }
    }
};

// The reference's f1 (post-streaming state including ghosts):
//   interior: stream_interior ? cur(l, x - c) : cur(l, x)
//   ghosts  : ghost_raw ? gsrc(l, x) as stored : gsrc(l, x with periodic axes wrapped)
template <int Q, class C>
struct StateOut {
    const void* cur;
    const void* gsrc;
    int stream_interior, ghost_raw;
    __device__ void cell(const Layout& L, int i, int j, int k, typename C::real (&f)[Q]) const {
        using Lt = Lattice<Q>;
        const bool interior = interior_cell(L, i, j, k);
#pragma unroll
        for (int l = 0; l < Q; ++l) {
            if (interior) {
                const int s = stream_interior;
                f[l] = ld<Q, C>(L, cur, l, L.cell_w(i - s * Lt::cx(l), j - s * Lt::cy(l), k - s * Lt::cz(l)));
            } else {
                f[l] = ld<Q, C>(L, gsrc, l, ghost_raw ? L.cell(i, j, k) : L.cell_w(i, j, k));
            }
        }
    }
    template <typename H>
    __device__ void operator()(const Layout& L, int i, int j, int k, H (&o)[Q]) const {
        typename C::real f[Q];
        cell(L, i, j, k, f);
#pragma unroll
        for (int l = 0; l < Q; ++l) o[l] = (H)f[l];
    }
};

// Its moments rho, u, v, w (src/m_macrovars_kernel.F90:41-49, all cells including ghosts).  *unstable
// becomes non-zero if one of them is not finite or a density is not positive
// (src/m_diag.F90:169-173): every cell that sees it writes the same value.
template <int Q, class C>
struct MomentsOut {
    StateOut<Q, C> state;
    int* unstable;
    template <typename H>
    __device__ void operator()(const Layout& L, int i, int j, int k, H (&o)[4]) const {
        using R = typename C::real;
        using Lt = Lattice<Q>;
        R f[Q];
        state.cell(L, i, j, k, f);
        R tr = 0, tu = 0, tv = 0, tw = 0;
#pragma unroll
        for (int l = 0; l < Q; ++l) {
            tr += f[l];
            if (Lt::cx(l) > 0) tu += f[l]; else if (Lt::cx(l) < 0) tu -= f[l];
            if (Lt::cy(l) > 0) tv += f[l]; else if (Lt::cy(l) < 0) tv -= f[l];
            if (Lt::cz(l) > 0) tw += f[l]; else if (Lt::cz(l) < 0) tw -= f[l];
        }
        const R inv = R(1) / tr;
        o[0] = (H)tr;
        o[1] = (H)(tu * inv);
        o[2] = (H)(tv * inv);
        o[3] = (H)(tw * inv);
        if (!(isfinite(o[0]) && isfinite(o[1]) && isfinite(o[2]) && isfinite(o[3]) && o[0] > H(0))) *unstable = 1;
    }
};

// Equilibrium initialisation (src/m_fequil3_kernel.F90 then src/m_fillghosts.F90): every cell,
// ghosts included, gets feq of its clamped interior cell, whose moments v holds.  The moments are
// also kept in the device cell layout for the first collision.
template <int Q, class C, bool BGK3>
struct EquilibriumIn {
    void* dst;
    typename C::real *mr, *mu, *mv, *mw;
    template <typename H>
    __device__ void operator()(const Layout& L, int i, int j, int k, const H (&v)[4]) const {
        using R = typename C::real;
        const R r = (R)v[0], ux = (R)v[1], uy = (R)v[2], uz = (R)v[3];
        const R usq = ux * ux + uy * uy + uz * uz;
        const int oc = L.cell(i, j, k);
#pragma unroll
        for (int l = 0; l < Q; ++l)
            st<Q, C>(L, dst, l, oc, feq_dir<Q, BGK3, R>(l, r, ux, uy, uz, usq));
        if (interior_cell(L, i, j, k)) {
            const int ox = L.cidx(i, j, k);
            mr[ox] = r; mu[ox] = ux; mv[ox] = uy; mw[ox] = uz;
        }
    }
};

// Adds the moments of the current state (streamed when stream_interior) to the averaging sums.
template <int Q, class C>
__global__ void average_kernel(Layout L, const void* cur, int stream_interior, typename C::real* avg) {
    using R = typename C::real;
    using Lt = Lattice<Q>;
    const int ca = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int cb = blockIdx.y + 1;
    const int cc = blockIdx.z + 1;
    if (ca > L.n(L.ax0)) return;
    int i, j, k;
    L.ijk(ca, cb, cc, i, j, k);
    const int s = stream_interior;
    R dr = 0, jx = 0, jy = 0, jz = 0;
#pragma unroll
    for (int l = 0; l < Q; ++l) {
        const R d = C::template dep<Q>(static_cast<const typename C::raw*>(cur)[(size_t)l * L.plane +
                                           L.cell_w(i - s * Lt::cx(l), j - s * Lt::cy(l), k - s * Lt::cz(l))], l) /
                    C::kDepScale;
        dr += d;
        jx += R(Lt::cx(l)) * d;
        jy += R(Lt::cy(l)) * d;
        jz += R(Lt::cz(l)) * d;
    }
    const R inv = R(1) / (R(1) + dr);
    const R ux = jx * inv, uy = jy * inv, uz = jz * inv;
    R* p = avg + L.cidx(i, j, k);
    const size_t P = (size_t)L.cplane;
    p[0] += ux;
    p[P] += uy;
    p[2 * P] += uz;
    p[3 * P] += ux * ux;
    p[4 * P] += uy * uy;
    p[5 * P] += uz * uz;
}

// Global mass and momentum of the state (interior cells) in FP64, with the smallest cell density
// and the number of non-finite populations (the instability test of src/m_diag.F90:169-173):
// per-block partial results partial[kTotalsSlots*block + {0..5}] = (mass, mx, my, mz, min rho,
// non-finite count), finished on the host.  Every block writes all of its slots.
template <int Q, class C>
__global__ void __launch_bounds__(256) totals_kernel(Layout L, const void* cur, int stream_interior, double* partial) {
    using Lt = Lattice<Q>;
    __shared__ double sh[kTotalsSlots][256];
    const long long ncell = (long long)L.nx * L.ny * L.nz;
    double m = 0, mx = 0, my = 0, mz = 0, rmin = INFINITY, bad = 0;
    const int s = stream_interior;
    // in storage order: along i, with j contiguous, a wave reads 64 rows at a time, and the rows' pitch decided its time
    // (D3Q19 FP32 200x120x80 277 us with 5 lines, 379 with 4, 72 in storage order; 384x192x128 1950 -> 170)
    const int n0 = L.n(L.ax0), n1 = L.n(L.ax1);
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell; c += (long long)gridDim.x * blockDim.x) {
        int i, j, k;
        L.ijk((int)(c % n0) + 1, (int)((c / n0) % n1) + 1, (int)(c / ((long long)n0 * n1)) + 1, i, j, k);
        double r = 0;
#pragma unroll
        for (int l = 0; l < Q; ++l) {
            const double f = (double)ld<Q, C>(L, cur, l, L.cell_w(i - s * Lt::cx(l), j - s * Lt::cy(l), k - s * Lt::cz(l)));
            if (!isfinite(f)) bad += 1;
            r += f;
            mx += Lt::cx(l) * f;
            my += Lt::cy(l) * f;
            mz += Lt::cz(l) * f;
        }
        m += r;
        rmin = r < rmin ? r : rmin;
    }
    const int t = threadIdx.x;
    sh[0][t] = m; sh[1][t] = mx; sh[2][t] = my; sh[3][t] = mz; sh[4][t] = rmin; sh[5][t] = bad;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if (t < w) {
            for (int q = 0; q < 4; ++q) sh[q][t] += sh[q][t + w];
            sh[4][t] = sh[4][t + w] < sh[4][t] ? sh[4][t + w] : sh[4][t];
            sh[5][t] += sh[5][t + w];
        }
        __syncthreads();
    }
    if (t == 0)
        for (int q = 0; q < kTotalsSlots; ++q) partial[kTotalsSlots * blockIdx.x + q] = sh[q][0];
}

}  // namespace lbm
