// Reverse mode (adjoint) of the DEM step for contact model 2, with bonds and
// walls, on a recorded forward pass, for every simulation of a context.  The
// reference has no counterpart.
//
// The forward pass records, per step, the state the step reads (positions,
// velocities, angular velocities, the tangential displacements, the walls,
// and each bond's inputs) and the contact rows after the interaction pass,
// which hold exactly the contacts that produced a force.  The reverse pass
// then runs the steps backwards with that contact list frozen and every
// branch (normal-force clamp, stick or slip, wall friction, bond breakage)
// taken as the forward took it, and propagates cotangents:
//
//   integrate (TY3)     x' = x + v dt + (2/3) a dt^2 - (1/6) a0 dt^2
//                       v' = v + (3/2) a dt - (1/2) a0 dt,  a = F/m + g
//   contactLinear       F, T and the new tangential displacement of each
//                       contact, as functions of both particles' state, the
//                       stored displacement and (k_n, k_t, gamma_n, gamma_t,
//                       mu_s, mu_d)
//   contactLinear_wall  F, T of each wall contact and the force it puts on
//                       the wall (k_n, gamma_wn, gamma_wt, mu_wd), as
//                       functions of the particle's and the wall's state
//   bondsLinear         the bond's force and torque and its new
//                       displacements and rotations (k_n, k_t, gamma_n,
//                       gamma_t)
//   integrateWalls      p' = p + u dt + (2/3) a dt^2 - (1/6) a0 dt^2,
//                       u' = u + (3/2) a dt - (1/2) a0 dt, with
//                       a = (sum of wall forces - sigma0 Lx Ly) / m for a
//                       stress-controlled wall (wmode 1) and a = 0 for a
//                       velocity-controlled one (wmode 2)
//
// Lengths are differentiated as exact roots (the forward rounds them to
// FP32, which is locally constant and has no useful derivative).  Sums
// that span particles (parameter cotangents, the walls' position and
// velocity cotangents) are formed per workgroup and then per simulation in
// a fixed order, so gradients are reproducible bit for bit.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "adjoint.hpp"
#include "dem_math.hpp"
#include "dem_scalar.hpp"

namespace sphx {

namespace {

// The parameter table is read-only for every kernel: read through the
// constant address space (scalar loads that stores do not invalidate).
typedef const __attribute__((address_space(4))) DevParams CParams;

constexpr double PI = 3.14159265358979;  // src/constants.h:14

__device__ __forceinline__ d3 zero3() { return mk3(0.0, 0.0, 0.0); }

// Cotangents of the parameters, in the order of AdjParam: one work-item's
// running sums (indexed by constants only: registers).
struct PGrad {
    double s[ADJ_NPARAM];
    __device__ __forceinline__ void add(int k, double x) { s[k] += x; }
    __device__ __forceinline__ void add(bool own, int k, double x) { s[k] += own ? x : 0.0; }
};

// Reverse of contactLinear (src/contactmodels.cuh:244-411, kappa = 0,
// E <= 0.001) for one contact of particle a with partner b.  Inputs are the
// forward inputs; gF, gT are the cotangents of a's force and torque and gdt
// that of the new tangential displacement.  The outputs are what falls on
// one of the two: with `own` on a (gx, gv, gw, the stored displacement's
// cotangent gdt0, and the parameters added to gp), else on b (gx, gv, gw).
__device__ __forceinline__ void adj_contact_linear(CParams& p, bool own, d3 va, d3 wa, d3 vb,
                                                   d3 wb, double ra, double rb, d3 x, d3 dt0,
                                                   d3 gF, d3 gT, d3 gdt, d3& gx, d3& gv, d3& gw,
                                                   d3& gdt0, PGrad& gp) {
    // forward (same expressions and FP32 lengths, so the same branches)
    const double len = length(x);
    const double delta = len - (ra + rb);
    const d3 n = x / len;
    const d3 vl = va - vb;
    const double ca = ra + delta / 2.0, cb = rb + delta / 2.0;
    const d3 na = cross(n, wa), nb = cross(n, wb);
    const d3 vel = vl + ca * na + cb * nb;
    const double vel_n = -dot(vl, n);
    const double nv = dot(n, vel);
    const d3 vel_t = vel - n * nv;
    const double vtl = length(vel_t);
    const double nd0 = dot(n, dt0);
    const d3 dtp = dt0 - n * nd0;
    const double dtpl = length(dtp);
    const double cn_raw = -p.k_n * delta + p.gamma_n * vel_n;
    const double cn = fmax(0.0, cn_raw);
    // kappa = 0: the capillary term is a signed zero and |f_n - f_c| = |f_n|.
    const double L = length(cn * n);
    const bool active = dtpl > 0.0 || vtl > 0.0;
    d3 dtmp = zero3(), f_raw = zero3(), t = zero3(), f_t = zero3();
    double frl = 0.0, limit = 0.0;
    bool slip = false;
    if (active) {
        dtmp = dtp + vel_t * p.dt;
        f_raw = -p.k_t * dtmp + -p.gamma_t * vel_t;
        frl = length(f_raw);
        limit = p.mu_s * L;
        slip = frl > limit;
        if (slip) {
            t = f_raw / frl;
            f_t = limit * t;
        } else {
            f_t = f_raw;
        }
    }
    // reverse
    d3 gn = zero3();
    double gdelta = 0.0;
    d3 gft = gF, gfn = gF;
    const double cu = -(ra + delta * 0.5);
    const d3 u = cu * n;
    gft += cross(gT, u);
    const d3 gu = cross(f_t, gT);
    gn += cu * gu;
    gdelta += -0.5 * dot(n, gu);
    d3 gdtp = zero3(), gvel_t = zero3();
    double gL = 0.0;
    if (active) {
        d3 gdtmp = zero3(), gfraw = zero3();
        if (slip) {
            // dt_new = -1/k_t (mu_d L t + gamma_t vel_t), f_t = mu_s L t
            const d3 A = p.mu_d * L * t + p.gamma_t * vel_t;
            const d3 gA = gdt * (-1.0 / p.k_t);
            gp.add(own, ADJ_KT, dot(gdt, A) / (p.k_t * p.k_t));
            gp.add(own, ADJ_MUD, L * dot(t, gA));
            gL += p.mu_d * dot(t, gA);
            d3 gt = (p.mu_d * L) * gA;
            gp.add(own, ADJ_GT, dot(vel_t, gA));
            gvel_t += p.gamma_t * gA;
            const double glim = dot(t, gft);
            gt += limit * gft;
            gp.add(own, ADJ_MUS, L * glim);
            gL += p.mu_s * glim;
            gfraw = (gt - t * dot(t, gt)) / frl;
        } else {
            gdtmp = gdt;
            gfraw = gft;
        }
        // f_raw = -k_t dtmp - gamma_t vel_t, dtmp = dtp + vel_t dt
        gdtmp += -p.k_t * gfraw;
        gp.add(own, ADJ_KT, -dot(dtmp, gfraw));
        gp.add(own, ADJ_GT, -dot(vel_t, gfraw));
        gvel_t += -p.gamma_t * gfraw;
        gdtp += gdtmp;
        gvel_t += p.dt * gdtmp;
    } else {
        gdtp += gdt;
    }
    if (L > 0.0) gfn += (gL / L) * (cn * n);
    const double gcn = dot(n, gfn);
    gn += cn * gfn;
    double gvel_n = 0.0;
    if (cn_raw > 0.0) {
        gp.add(own, ADJ_KN, -delta * gcn);
        gdelta += -p.k_n * gcn;
        gp.add(own, ADJ_GN, vel_n * gcn);
        gvel_n = p.gamma_n * gcn;
    }
    // dtp = dt0 - n (n . dt0)
    gdt0 = gdtp - n * dot(n, gdtp);
    gn += -(nd0 * gdtp + dot(n, gdtp) * dt0);
    // vel_t = vel - n (n . vel)
    const d3 gvel = gvel_t - n * dot(n, gvel_t);
    gn += -(nv * gvel_t + dot(n, gvel_t) * vel);
    // vel_n = -(vl . n)
    d3 gvl = -gvel_n * n;
    gn += -gvel_n * vl;
    // vel = vl + ca (n x wa) + cb (n x wb)
    gvl += gvel;
    gdelta += 0.5 * dot(gvel, na) + 0.5 * dot(gvel, nb);
    const d3 gna = ca * gvel, gnb = cb * gvel;
    gn += cross(wa, gna) + cross(wb, gnb);
    gw = cross(own ? gna : gnb, n);
    gv = own ? gvl : -gvl;
    // n = x / |x|, delta = |x| - (ra + rb)
    const d3 gxa = (gn - n * dot(n, gn)) / len + n * gdelta;
    gx = own ? gxa : -gxa;
}

// Reverse of contactLinear_wall (src/contactmodels.cuh:10-117) for one wall
// with normal n at distance delta from the particle (delta = e . x + const,
// with the wall position entering const), moving at speed wv, whose return
// value dot(f_n, n) (the force on the wall) has cotangent gret.  Adds to the
// particle's cotangents; returns the cotangents of delta and of wv.
__device__ void adj_contact_wall(CParams& p, d3 va, d3 wa, double ra, d3 n, double delta,
                                 double wv, d3 gF, d3 gT, double gret, d3& gva, d3& gwa,
                                 double& gdelta, double& gwv, PGrad& gp) {
    const d3 vl = va;
    const double c = ra + delta / 2.0;
    const d3 nw = cross(n, wa);
    const d3 vel = vl + c * nw + wv;
    const double vel_n = dot(vl, n);
    const double nv = dot(n, vel);
    const d3 vel_t = vel - n * nv;
    const double vtl = length(vel_t);
    const double cn_raw = -p.k_n * delta - p.gamma_wn * vel_n;
    const double cn = fmax(0.0, cn_raw);
    const d3 f_n = cn * n;
    const double fnl = length(f_n);
    d3 f_t = zero3();
    bool fric = vtl > 0.0 && p.gamma_wt > 0.0, stick = false;
    double limit = 0.0;
    if (fric) {
        const d3 f_t_visc = p.gamma_wt * vel_t;
        limit = p.mu_wd * fnl;
        stick = length(f_t_visc) < limit;
        f_t = stick ? -1.0 * f_t_visc : -limit * vel_t / vtl;
    }
    d3 gft = gF, gfn = gF + gret * n;
    gdelta = 0.0;
    const double cu = -(ra + delta * 0.5);
    gft += cross(gT, cu * n);
    gdelta += -0.5 * dot(n, cross(f_t, gT));
    d3 gvel_t = zero3();
    if (fric) {
        if (stick) {
            gvel_t += -p.gamma_wt * gft;
            gp.add(ADJ_GWT, -dot(vel_t, gft));
        } else {
            const d3 s = vel_t / vtl;
            const double glim = -dot(s, gft);
            const d3 gs = -limit * gft;
            gvel_t += (gs - s * dot(s, gs)) / vtl;
            gp.add(ADJ_MUWD, fnl * glim);
            if (fnl > 0.0) gfn += (p.mu_wd * glim / fnl) * f_n;
        }
    }
    const double gcn = dot(n, gfn);
    double gvel_n = 0.0;
    if (cn_raw > 0.0) {
        gp.add(ADJ_KN, -delta * gcn);
        gdelta += -p.k_n * gcn;
        gp.add(ADJ_GWN, -vel_n * gcn);
        gvel_n = -p.gamma_wn * gcn;
    }
    const d3 gvel = gvel_t - n * dot(n, gvel_t);
    d3 gvl = gvel_n * n + gvel;
    gdelta += 0.5 * dot(gvel, nw);
    gwa += cross(c * gvel, n);
    gva += gvl;
    // vel = vl + c (n x w) + wv: the wall speed is added to every component.
    gwv = gvel.x + gvel.y + gvel.z;
}

constexpr int ALPP = 4;               // work-items per particle
constexpr int ASPL = NC / ALPP;       // contact slots per work-item
static_assert(ADJ_PPB * ALPP == 256, "four work-items per particle");

// Orders the wavefront's LDS accesses around it.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Force and torque cotangents of one particle (reverse of TY3 for the
// accelerations the step computes from them): from the cotangents of its
// new position, velocity and angular velocity and of the new accelerations
// (which also feed the next step as acc0).
__device__ __forceinline__ void force_cotangents(CParams& p, double r, double fv,
                                                 double4 Lx, double4 Lv, double4 Lw, double4 La,
                                                 double4 Laa, d3& gF, d3& gT) {
    const double dt = p.dt;
    const double m = 4.0 / 3.0 * PI * r * r * r * p.rho;
    const double I = 2.0 / 5.0 * m * r * r;
    d3 ga = mk3(La.x + (2.0 / 3.0) * dt * dt * Lx.x + 1.5 * dt * Lv.x,
                La.y + (2.0 / 3.0) * dt * dt * Lx.y + 1.5 * dt * Lv.y,
                La.z + (2.0 / 3.0) * dt * dt * Lx.z + 1.5 * dt * Lv.z);
    d3 gaa = mk3(Laa.x + 1.5 * dt * Lw.x, Laa.y + 1.5 * dt * Lw.y, Laa.z + 1.5 * dt * Lw.z);
    // fixvel modes (src/integration.cuh): the masked components do not
    // depend on the force.
    if (fv > 0.0001 && fv < 10.0) {
        ga.x = 0.0;
        ga.y = 0.0;
        gaa = zero3();
    }
    if (fv >= 10.0) {
        ga.y = 0.0;
        gaa.x = 0.0;
        gaa.z = 0.0;
    }
    if (fv < -0.0001) {
        ga = zero3();
        gaa = zero3();
    }
    gF = mk3(ga.x / m, ga.y / m, ga.z / m);
    gT = mk3(gaa.x / I, gaa.y / I, gaa.z / I);
}

__device__ __forceinline__ d3 image_shift(CParams& p, uint32_t wrd) {
    const uint32_t cx = (wrd >> CW_SHIFT_X) & 3u, cy = (wrd >> CW_SHIFT_Y) & 3u;
    return mk3(cx == 1u ? 0.0 + p.L[0] : cx == 2u ? 0.0 - p.L[0] : 0.0,
               cy == 1u ? 0.0 + p.L[1] : cy == 2u ? 0.0 - p.L[1] : 0.0, 0.0);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Reverse of one whole step, ALPP work-items per particle, in the step's
// sorted order (partner gathers then stay near each other in the recorded
// state).  Every particle's input cotangent is gathered by its own group,
// with no atomics:
//  1. integrate (TY3): from the cotangents of the step's outputs (Lout,
//     La/Laa out) the force and torque cotangents and the integrate part
//     of the input cotangents; the acceleration cotangents of the step's
//     inputs go to La/Laa in;
//  2. contacts.  A contact a -> b of the row the step left gives two
//     evaluations: its own (a's contactLinear: a's part, the parameters, and
//     the stored displacement's cotangent, handed to the step before where
//     that slot held the same partner then), and its mirror (b's
//     contactLinear against a, found in b's row: the part that falls on a,
//     with b's force cotangents recomputed from b's Lout).  The wavefront's
//     evaluations are numbered, all own ones first, then the mirrors, each
//     particle's in slot order, and taken one per lane; each particle's lanes
//     then add its contributions in that order (lane 0 x, lane 1 v, lane 2
//     w), so that a particle's sums do not depend on its neighbours in the
//     wavefront.  Contact rows are symmetric unless a row overflowed; a
//     contact whose partner does not list it is counted in `asym` (the host
//     then refuses the result);
//  3. walls, on work-item 0, including the cotangent of each wall force
//     the particle puts on a list wall (from the wall's equation of
//     motion) and the cotangents of the walls' position and velocity;
//  4. the group's sums are written to Lin; the workgroup's partial sums of
//     the parameter and wall cotangents to part.
// Bound by the latency of its load chain (order, row, partner and its row,
// displacements) at two wavefronts per SIMD (202 VGPRs; three spill 59 and
// took 102 us where two take 76).  Each work-item walking its own slots, both
// evaluations of each one after the other, took 91 us a step on 1e5
// particles and 25 on 2,000; this takes 76 and 17.
__global__ __launch_bounds__(256) void k_adj_step(AdjStep st, AdjState g) {
    constexpr int G = 64 / ALPP;  // particles per wavefront
    struct Work {
        double con[9][64];
        uint16_t tab[G * NC];
    };
    __shared__ Work s_work[4];
    __shared__ uint32_t s_row[4][G][NC];
    __shared__ double4 s_state[4][3][G];
    __shared__ double s_force[4][6][G];
    __shared__ uint32_t s_orig[4][G];
    __shared__ uint2 s_prev[4][G];
    __shared__ __align__(16) uint8_t s_zc[4][G];
    __shared__ double red[ADJ_NPART][4];
    touch_lines<sizeof(AdjStep) + sizeof(AdjState)>((cvoid*)__builtin_amdgcn_kernarg_segment_ptr());
    const uint32_t sim = st.nsim == 1u ? 0u : st.chunk_sim[blockIdx.x / (256 / ADJ_PPB)];
    touch_lines<sizeof(DevParams)>((cvoid*)(st.ptab + sim));
    CParams& p = *(CParams*)(st.ptab + sim);
    const uint32_t lane = threadIdx.x % 64, wv = threadIdx.x / 64;
    const uint32_t q = threadIdx.x % ALPP, gw = lane / ALPP;
    const uint32_t ia = blockIdx.x * ADJ_PPB + threadIdx.x / ALPP;
    const bool in = ia - p.base < p.np;
    const double dt = p.dt;
    // The workgroup's sums so far, when the steps accumulate.
    double* const part = g.part + (size_t)threadIdx.x * gridDim.x + blockIdx.x;
    const double before = st.accumulate && threadIdx.x < ADJ_NPART ? *part : 0.0;
    PGrad gp;
#pragma unroll
    for (int k = 0; k < ADJ_NPARAM; ++k) gp.s[k] = 0.0;
    uint32_t a = 0, occ = 0;
    d3 acc = zero3();
    if (in) {
        a = st.perm[ia];
        // This work-item's row words (slots ASPL q, ...).
        uint32_t word[ASPL];
        const uint4* row = reinterpret_cast<const uint4*>(st.rows + (size_t)ia * NC + ASPL * q);
#pragma unroll
        for (int h = 0; h < ASPL / 4; ++h) {
            const uint4 u = row[h];
            word[4 * h] = u.x;
            word[4 * h + 1] = u.y;
            word[4 * h + 2] = u.z;
            word[4 * h + 3] = u.w;
        }
        const uint2 prev = st.prev[ia];
        const double4 xa4 = st.x[ia], va4 = st.v[ia], wa4 = st.w[ia];
        // 1. integrate
        const double4 Lx = g.Lout[0][a], Lv = g.Lout[1][a], Lw = g.Lout[2][a];
        const double4 La = g.La_out[a], Laa = g.Laa_out[a];
        d3 gF, gT;
        force_cotangents(p, xa4.w, va4.w, Lx, Lv, Lw, La, Laa, gF, gT);
        // x' = x + ..., v' = v + ..., w' = w + ...
        if (q == 0) acc = mk3(Lx.x, Lx.y, Lx.z);
        if (q == 1) acc = mk3(Lx.x * dt + Lv.x, Lx.y * dt + Lv.y, Lx.z * dt + Lv.z);
        if (q == 2) acc = mk3(Lw.x, Lw.y, Lw.z);
        if (q == 3) {
            const double c0 = st.first ? 0.0 : 1.0;  // acc0 is zero on a run's first step
            g.La_in[a] = make_double4(c0 * (-(dt * dt / 6.0) * Lx.x - 0.5 * dt * Lv.x),
                                      c0 * (-(dt * dt / 6.0) * Lx.y - 0.5 * dt * Lv.y),
                                      c0 * (-(dt * dt / 6.0) * Lx.z - 0.5 * dt * Lv.z), 0.0);
            g.Laa_in[a] = make_double4(c0 * -0.5 * dt * Lw.x, c0 * -0.5 * dt * Lw.y,
                                       c0 * -0.5 * dt * Lw.z, 0.0);
        }
        if (q == 0) {
            s_state[wv][0][gw] = make_double4(xa4.x, xa4.y, xa4.z, xa4.w);
            s_orig[wv][gw] = a;
            s_prev[wv][gw] = prev;
        }
        if (q == 1) s_state[wv][1][gw] = make_double4(va4.x, va4.y, va4.z, va4.w);
        if (q == 2) s_state[wv][2][gw] = make_double4(wa4.x, wa4.y, wa4.z, 0.0);
        if (q == 3) {
            s_force[wv][0][gw] = gF.x;
            s_force[wv][1][gw] = gF.y;
            s_force[wv][2][gw] = gF.z;
            s_force[wv][3][gw] = gT.x;
            s_force[wv][4][gw] = gT.y;
            s_force[wv][5][gw] = gT.z;
        }
#pragma unroll
        for (int j = 0; j < ASPL; ++j) {
            const uint32_t slot = ASPL * q + j;
            const bool o = (word[j] & CW_IDX_MASK) != EMPTY;
            s_row[wv][gw][slot] = word[j];
            occ |= o ? 1u << slot : 0u;
            // A slot that has lost its partner: no cotangent reaches the
            // displacement it held.
            if (!o && ((prev.x >> slot) & 1u))
                g.Ldt_out[(size_t)a * NC + slot] = make_double4(0.0, 0.0, 0.0, 0.0);
        }
    }
#pragma unroll
    for (int m = 1; m < ALPP; m <<= 1) occ |= (uint32_t)__shfl_xor((int)occ, m, 64);
    const uint32_t zg = __popc(occ);
    if (q == 0) s_zc[wv][gw] = (uint8_t)zg;
    wave_sync();
    // The group's first contact number and the wavefront's contact count
    // (byte sums of the counts, each at most NC).
    uint32_t first = 0, total = 0;
    {
        const uint32_t* zw = reinterpret_cast<const uint32_t*>(s_zc[wv]);
#pragma unroll
        for (int i = 0; i < G / 4; ++i) {
            const uint32_t w = zw[i];
            const int below_w = (int)gw - 4 * i;
            const uint32_t m = below_w <= 0 ? 0u
                               : below_w >= 4 ? 0xffffffffu
                                              : (1u << (8 * below_w)) - 1u;
            first += ((w & m) * 0x01010101u) >> 24;
            total += (w * 0x01010101u) >> 24;
        }
    }
#pragma unroll
    for (int j = 0; j < ASPL; ++j) {
        const uint32_t slot = ASPL * q + j;
        if ((occ >> slot) & 1u)
            s_work[wv].tab[first + __popc(occ & ((1u << slot) - 1u))] =
                (uint16_t)((gw << 5) | slot);
    }
    wave_sync();
    // 2. contacts
    for (uint32_t r0 = 0; r0 < 2 * total; r0 += 64) {
        const uint32_t it = r0 + lane;
        d3 gx = zero3(), g1v = zero3(), g1w = zero3();
        if (it < 2 * total) {
            const bool own = it < total;
            const uint32_t e = s_work[wv].tab[own ? it : it - total];
            const uint32_t h = e >> 5, ih = ia - gw + h;
            uint32_t slot = e & 31u, word = s_row[wv][h][slot];
            const uint32_t bs = word & CW_IDX_MASK;
            const double4 xb4 = st.x[bs], vb4 = st.v[bs], wb4 = st.w[bs];
            uint32_t o1 = s_orig[wv][h], i1 = ih;  // whose contact it is
            d3 gF, gT;
            if (own) {
                gF = mk3(s_force[wv][0][h], s_force[wv][1][h], s_force[wv][2][h]);
                gT = mk3(s_force[wv][3][h], s_force[wv][4][h], s_force[wv][5][h]);
            } else {
                // The contact's mirror in b's row.  Every word is read (no
                // branch between the loads, which would make each wait for
                // the one before) and the first match kept.
                const uint32_t b = st.perm[bs];
                const uint4* brow = reinterpret_cast<const uint4*>(st.rows + (size_t)bs * NC);
                slot = NC;
#pragma unroll
                for (int k = NC / 4 - 1; k >= 0; --k) {
                    const uint4 u = brow[k];
                    if ((u.w & CW_IDX_MASK) == ih) { slot = 4 * k + 3; word = u.w; }
                    if ((u.z & CW_IDX_MASK) == ih) { slot = 4 * k + 2; word = u.z; }
                    if ((u.y & CW_IDX_MASK) == ih) { slot = 4 * k + 1; word = u.y; }
                    if ((u.x & CW_IDX_MASK) == ih) { slot = 4 * k; word = u.x; }
                }
                o1 = b;
                i1 = bs;
                force_cotangents(p, xb4.w, vb4.w, g.Lout[0][b], g.Lout[1][b], g.Lout[2][b],
                                 g.La_out[b], g.Laa_out[b], gF, gT);
            }
            if (slot == NC) {
                atomicAdd(g.asym, 1u);
            } else {
                const d3 dt0 = xyz(st.dt0[(size_t)i1 * NC + slot]);
                const size_t mp = (size_t)o1 * NC + slot;
                const d3 gdt = st.last ? zero3() : xyz(g.Ldt_in[mp]);
                const double4 xh4 = s_state[wv][0][h], vh4 = s_state[wv][1][h],
                              wh4 = s_state[wv][2][h];
                // The contact's particle (1) and its partner (2).
                const double4 x1 = own ? xh4 : xb4, x2 = own ? xb4 : xh4;
                const double4 v1 = own ? vh4 : vb4, v2 = own ? vb4 : vh4;
                const double4 w1 = own ? wh4 : wb4, w2 = own ? wb4 : wh4;
                const d3 dm = image_shift(p, word);
                const d3 x12 = mk3(x1.x - x2.x + dm.x, x1.y - x2.y + dm.y, x1.z - x2.z + dm.z);
                d3 gdt0;
                adj_contact_linear(p, own, xyz(v1), xyz(w1), xyz(v2), xyz(w2), x1.w, x2.w, x12,
                                   dt0, gF, gT, gdt, gx, g1v, g1w, gdt0, gp);
                const uint2 prev = s_prev[wv][h];
                if (own && ((prev.x >> slot) & 1u))
                    g.Ldt_out[mp] = ((prev.y >> slot) & 1u)
                                        ? make_double4(gdt0.x, gdt0.y, gdt0.z, 0.0)
                                        : make_double4(0.0, 0.0, 0.0, 0.0);
            }
        }
        s_work[wv].con[0][lane] = gx.x;
        s_work[wv].con[1][lane] = gx.y;
        s_work[wv].con[2][lane] = gx.z;
        s_work[wv].con[3][lane] = g1v.x;
        s_work[wv].con[4][lane] = g1v.y;
        s_work[wv].con[5][lane] = g1v.z;
        s_work[wv].con[6][lane] = g1w.x;
        s_work[wv].con[7][lane] = g1w.y;
        s_work[wv].con[8][lane] = g1w.z;
        wave_sync();
        if (q < 3) {
#pragma unroll
            for (int part = 0; part < 2; ++part) {
                const uint32_t f = first + (part ? total : 0u);
                const uint32_t lo = f > r0 ? f : r0;
                const uint32_t hi = f + zg < r0 + 64 ? f + zg : r0 + 64;
                for (uint32_t c = lo; c < hi; ++c) {
                    acc.x += s_work[wv].con[3 * q][c - r0];
                    acc.y += s_work[wv].con[3 * q + 1][c - r0];
                    acc.z += s_work[wv].con[3 * q + 2][c - r0];
                }
            }
        }
        wave_sync();
    }
    // 3. walls, as in the forward pass (src/contactsearch.cuh:602-701):
    // top (wall 0, or the implicit wall at L_z), bottom, then the side
    // walls by boundary mode; walls beyond nw are the implicit ones.
    if (lane < 2 * MAXWALLS) red[ADJ_NPARAM + lane][wv] = 0.0;
    bool any_wall = false;
    d3 gxw = zero3(), gvw = zero3(), gww = zero3();
    {
        const double4 xa4 = s_state[wv][0][gw];
        // Side s: top, bottom, then x high and low, y high and low.  The
        // contact distance changes with the position along e.
#pragma unroll 1
        for (int s = 0; s < 6; ++s) {
            if ((s == 2 || s == 3) && p.periodic != 0) continue;
            if ((s == 4 || s == 5) && p.periodic != 0 && p.periodic != 2) continue;
            const int w = s == 0 ? 0 : s == 1 ? -1 : s - 1;  // its list wall
            const bool listed = w >= 0 && (uint32_t)w < p.nw;
            const double side = (s == 1 || s == 3 || s == 5) ? 1.0 : -1.0;
            const d3 e = s < 2 ? mk3(0.0, 0.0, side)
                               : s < 4 ? mk3(side, 0.0, 0.0) : mk3(0.0, side, 0.0);
            d3 wn = e;
            double wpos = s == 0 ? p.L[2] : s == 1 ? p.origo[2] : s == 2 ? p.L[0]
                          : s == 4 ? p.L[1] : 0.0;
            double wvel = 0.0;
            if (listed) {
                const auto* nx = (const __attribute__((address_space(4))) double*)(
                    st.wall_nx + p.wall_base + w);
                const auto* mv = (const __attribute__((address_space(4))) double*)(
                    st.wall_mvfd + p.wall_base + w);
                wn = mk3(nx[0], nx[1], nx[2]);
                wpos = nx[3];
                wvel = mv[1];
            }
            const double xc = s < 2 ? xa4.z : s < 4 ? xa4.x : xa4.y;
            const double dw = side < 0.0 ? wpos - (xc + xa4.w) : xc - xa4.w - wpos;
            const bool touch = in && q == 0 && dw < 0.0;
            if (__ballot(touch) == 0ull) continue;
            any_wall = true;
            double gdel = 0.0, gwv = 0.0;
            if (touch) {
                const d3 va = xyz(s_state[wv][1][gw]), wa = xyz(s_state[wv][2][gw]);
                const d3 gF = mk3(s_force[wv][0][gw], s_force[wv][1][gw], s_force[wv][2][gw]);
                const d3 gT = mk3(s_force[wv][3][gw], s_force[wv][4][gw], s_force[wv][5][gw]);
                // The force sum's cotangent; the wall's position moves dw
                // against `side`.
                const double gS = listed ? g.wall[(p.wall_base + w) * ADJ_WALL + 3] : 0.0;
                adj_contact_wall(p, va, wa, xa4.w, wn, dw, wvel, gF, gT, gS, gvw, gww, gdel, gwv,
                                 gp);
                gxw += gdel * e;
            }
            if (listed) {
                const double vp = wave_sum(-side * gdel), vu = wave_sum(gwv);
                if (lane == 0) {
                    red[ADJ_NPARAM + 2 * w][wv] = vp;
                    red[ADJ_NPARAM + 2 * w + 1][wv] = vu;
                }
            }
        }
    }
    if (any_wall) {
        // Lane 0's parts to the lanes that hold the sums.
        const int src = (int)(lane - q);
        const d3 v1 = mk3(__shfl(gvw.x, src, 64), __shfl(gvw.y, src, 64), __shfl(gvw.z, src, 64));
        const d3 w1 = mk3(__shfl(gww.x, src, 64), __shfl(gww.y, src, 64), __shfl(gww.z, src, 64));
        acc += q == 0 ? gxw : q == 1 ? v1 : w1;
    }
    // 4. the particle's input cotangents
    double4* const lin = q == 0 ? +g.Lin[0] : q == 1 ? +g.Lin[1] : +g.Lin[2];
    if (in && q < 3) lin[a] = make_double4(acc.x, acc.y, acc.z, 0.0);
    // Partial sums of the workgroup: wavefront butterflies, then the four
    // wavefronts in order (a fixed order: reproducible bit for bit).  The
    // walls' quantities are zero in a wavefront that touches none.
#pragma unroll
    for (int k = 0; k < ADJ_GWN; ++k) {
        const double v = wave_sum(gp.s[k]);
        if (lane == 0) red[k][wv] = v;
    }
    if (any_wall) {
#pragma unroll
        for (int k = ADJ_GWN; k < ADJ_NPARAM; ++k) {
            const double v = wave_sum(gp.s[k]);
            if (lane == 0) red[k][wv] = v;
        }
    } else if (lane >= ADJ_GWN && lane < ADJ_NPARAM) {
        red[lane][wv] = 0.0;
    }
    __syncthreads();
    if (threadIdx.x < ADJ_NPART) {
        const int k = threadIdx.x;
        *part = before + (red[k][0] + red[k][1] + red[k][2] + red[k][3]);
    }
}

// Reverse of bondsLinear (src/cohesion.cuh:8-233) for the bonds that applied
// forces in the step, from the recorded inputs: the cotangents of the
// particles' forces and torques (recomputed from their output cotangents)
// and of the bond's new displacements and rotations.  Writes the
// cotangents of both particles' x, v, w to bcontrib, of the displacements
// and rotations it read to Lb_in, and its parameter cotangents to bpart.
// A bond that applied no force (broken, or broken in this step) leaves its
// displacements and rotations as they were: their cotangents pass through.
__global__ __launch_bounds__(256) void k_adj_bonds(AdjStep st, AdjState g) {
    const uint32_t b = blockIdx.x * 256 + threadIdx.x;
    if (b >= st.nbond) return;
    CParams& p = *(CParams*)(st.ptab + st.bond_sim[b]);
    const uint4 idx = st.bond_idx[b];
    double4* co = g.bcontrib + (size_t)6 * b;
    double* bp = g.bpart + (size_t)ADJ_NBPARAM * b;
    const double4 z4 = make_double4(0.0, 0.0, 0.0, 0.0);
    const double4 Ld = st.last ? z4 : g.Lb_out[2 * b], Lo = st.last ? z4 : g.Lb_out[2 * b + 1];
    if (!idx.z) {
        g.Lb_in[2 * b] = Ld;
        g.Lb_in[2 * b + 1] = Lo;
        for (int k = 0; k < 6; ++k) co[k] = z4;
        for (int k = 0; k < ADJ_NBPARAM; ++k) bp[k] = 0.0;
        return;
    }
    const uint32_t bi = idx.x, bj = idx.y;
    const double4* in = st.bond_in + (size_t)8 * b;
    const double4 x_i = in[0], x_j = in[1], v_i4 = in[2], v_j4 = in[3];
    const d3 w_i = xyz(in[4]), w_j = xyz(in[5]);
    const double4 d0 = in[6], o0 = in[7];
    const d3 v_i = xyz(v_i4), v_j = xyz(v_j4);
    const double dt = p.dt;
    // cotangents of the bond's force on i and torque t_j (force_i += f,
    // force_j -= f, torque_i -= t_j, torque_j += t_j)
    d3 gFi, gTi, gFj, gTj;
    force_cotangents(p, x_i.w, v_i4.w, g.Lout[0][bi], g.Lout[1][bi], g.Lout[2][bi],
                     g.La_out[bi], g.Laa_out[bi], gFi, gTi);
    force_cotangents(p, x_j.w, v_j4.w, g.Lout[0][bj], g.Lout[1][bj], g.Lout[2][bj],
                     g.La_out[bj], g.Laa_out[bj], gFj, gTj);
    const d3 gf = gFi - gFj, gtj = gTj - gTi;
    // forward
    const double R_bar = p.lambda_bar * fmin(x_i.w, x_j.w);
    const double A = PI * R_bar * R_bar;
    const double I = 0.25 * PI * R_bar * R_bar * R_bar * R_bar;
    const double J = I * 2.0;
    const d3 x = mk3(x_i.x - x_j.x, x_i.y - x_j.y, x_i.z - x_j.z);
    const double len = length(x);
    const double sep = len - (x_i.w + x_j.w);
    const double overlap = fmin(0.0, sep);
    const d3 n = x / len;
    const d3 dt0 = xyz(d0), om0 = xyz(o0);
    const double nd0 = dot(n, dt0);
    const d3 dt0p = dt0 - n * nd0;
    const double ci = x_i.w + overlap / 2.0, cj = x_j.w + overlap / 2.0;
    const d3 ni = cross(n, w_i), nj = cross(n, w_j);
    const d3 dd = ((v_i - v_j) + ci * ni + cj * nj) * dt;
    const double ddn = -dot(dd, n);
    const double dn = d0.w + ddn;
    const double ndd = dot(n, dd);
    const d3 ddt = dd - n * ndd;
    const d3 dtv = dt0p + ddt;
    // Stiffness per unit area (the bond option replaces k_n, k_t here; its
    // own cotangent is not formed, and then k_n, k_t get none from bonds).
    const bool ref_k = !(p.bond_k > 0.0);
    const double kn = ref_k ? p.k_n : p.bond_k / A;
    const double kt = ref_k ? p.k_t : p.bond_k / A;
    const double cfn = kn * A * dn + p.gamma_n * ddn / dt;
    const double no0 = dot(n, om0);
    const d3 dom = (w_j - w_i) * dt;
    const double ndo = dot(n, dom);
    const double don = -ndo;
    const double omn = o0.w + don;
    const d3 omt = (om0 - n * no0) + (dom - n * ndo);
    // reverse
    const d3 gdtv = xyz(Ld), gomt_o = xyz(Lo);
    double gdn = Ld.w, gomn = Lo.w;
    d3 gn = zero3();
    // t_j = t_n + t_t; t_n = k_t J omn n; t_t = -k_n I omt
    const d3 gomt = gomt_o + (-kn * I) * gtj;
    bp[0] = -I * dot(omt, gtj);                       // k_n
    const double ngt = dot(n, gtj);
    gomn += kt * J * ngt;
    bp[1] = J * omn * ngt;                            // k_t
    gn += (kt * J * omn) * gtj;
    // omt = om0 - n (n . om0) + dom - n (n . dom); omn = o0.w - n . dom
    d3 gom0 = gomt - n * dot(n, gomt);
    gn += -(no0 * gomt + dot(n, gomt) * om0);
    d3 gdom = gomt - n * dot(n, gomt);
    gn += -(ndo * gomt + dot(n, gomt) * dom);
    const double gom0n = gomn;
    gdom += -gomn * n;
    gn += -gomn * dom;
    d3 gwi = -dt * gdom, gwj = dt * gdom;
    // f = f_n + f_t; f_n = cfn n; f_t = -k_t A dtv - gamma_t ddt / dt
    const double gcfn = dot(n, gf);
    gn += cfn * gf;
    gdn += kn * A * gcfn;
    bp[0] += A * dn * gcfn;
    double gddn = p.gamma_n / dt * gcfn;
    bp[2] = ddn / dt * gcfn;                          // gamma_n
    const d3 gdtv_tot = gdtv + (-kt * A) * gf;
    bp[1] += -A * dot(dtv, gf);
    if (!ref_k) bp[0] = bp[1] = 0.0;
    d3 gddt = (-p.gamma_t / dt) * gf;
    bp[3] = -dot(ddt, gf) / dt;                       // gamma_t
    // dtv = dt0p + ddt; dn = d0.w + ddn
    const d3 gdt0p = gdtv_tot;
    gddt += gdtv_tot;
    const double gd0n = gdn;
    gddn += gdn;
    // ddt = dd - n (n . dd); ddn = -(dd . n)
    d3 gdd = gddt - n * dot(n, gddt);
    gn += -(ndd * gddt + dot(n, gddt) * dd);
    gdd += -gddn * n;
    gn += -gddn * dd;
    // dd = ((v_i - v_j) + ci (n x w_i) + cj (n x w_j)) dt
    const d3 gw = dt * gdd;
    const d3 gvi = gw, gvj = -gw;
    gn += cross(w_i, ci * gw) + cross(w_j, cj * gw);
    gwi += cross(ci * gw, n);
    gwj += cross(cj * gw, n);
    const double gov = 0.5 * (dot(gw, ni) + dot(gw, nj));
    // dt0p = dt0 - n (n . dt0)
    const d3 gdt0 = gdt0p - n * dot(n, gdt0p);
    gn += -(nd0 * gdt0p + dot(n, gdt0p) * dt0);
    // overlap = fmin(0, len - R); n = x / len
    const double glen = sep < 0.0 ? gov : 0.0;
    const d3 gx = (gn - n * dot(n, gn)) / len + n * glen;
    g.Lb_in[2 * b] = make_double4(gdt0.x, gdt0.y, gdt0.z, gd0n);
    g.Lb_in[2 * b + 1] = make_double4(gom0.x, gom0.y, gom0.z, gom0n);
    co[0] = make_double4(gx.x, gx.y, gx.z, 0.0);
    co[1] = make_double4(gvi.x, gvi.y, gvi.z, 0.0);
    co[2] = make_double4(gwi.x, gwi.y, gwi.z, 0.0);
    co[3] = make_double4(-gx.x, -gx.y, -gx.z, 0.0);
    co[4] = make_double4(gvj.x, gvj.y, gvj.z, 0.0);
    co[5] = make_double4(gwj.x, gwj.y, gwj.z, 0.0);
}

// Adds each particle's share of its bonds' cotangents to its input
// cotangents, in ascending bond id over the bonds the forward gather
// visited (the particle's own CSR list, or the whole list for particle nb0
// after a broken bond was retargeted onto it).
__global__ __launch_bounds__(256) void k_adj_bond_gather(AdjStep st, AdjState g) {
    CParams& p = *(CParams*)(st.ptab + st.chunk_sim[blockIdx.x]);
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i - p.base >= p.np) return;
    const bool full = (i - p.base == p.nb0) && st.bond_full[p.sim] != 0u;
    const uint32_t b0 = full ? p.bond_base : st.badj_off[i];
    const uint32_t b1 = full ? p.bond_base + p.nb0 : st.badj_off[i + 1];
    if (b0 == b1) return;
    double4 gx = g.Lin[0][i], gv = g.Lin[1][i], gw = g.Lin[2][i];
    for (uint32_t k = b0; k < b1; ++k) {
        const uint32_t b = full ? k : st.badj[k];
        const uint4 idx = st.bond_idx[b];
        if (!idx.z) continue;
        const double4* co = g.bcontrib + (size_t)6 * b;
        for (int side = 0; side < 2; ++side) {
            if ((side == 0 ? idx.x : idx.y) != i) continue;
            const double4 cx = co[3 * side], cv = co[3 * side + 1], cw = co[3 * side + 2];
            gx.x += cx.x; gx.y += cx.y; gx.z += cx.z;
            gv.x += cv.x; gv.y += cv.y; gv.z += cv.z;
            gw.x += cw.x; gw.y += cw.y; gw.z += cw.z;
        }
    }
    g.Lin[0][i] = gx;
    g.Lin[1][i] = gv;
    g.Lin[2][i] = gw;
}

// Per simulation (one workgroup each): the step's parameter cotangents
// (particle workgroups, then bonds) added to the running sums, and the
// reverse of integrateWalls (src/integration.cuh:344-450) for the walls:
// from the cotangents of the position, velocity and acceleration the step
// left (P, U, A) and of the wall contacts' position and velocity (cp, cu),
// those of the position, velocity and acceleration the step started from;
// then the force sum's cotangent for the step before (the wall's
// acceleration there is (sum + N) / m for wmode 1, zero for wmode 2, and
// wall w integrates wall 0's sum unless each wall has its own).
//
// Each sum has a fixed order: 256 strided shares, then a halving tree over
// them.  Latency is all that bounds this kernel, so every quantity's shares
// are summed at once (four groups of 256 work-items, each group every fourth
// quantity), then one wavefront per quantity runs its tree by shuffles.
// Quantity after quantity with a barrier per tree level, and partials read at
// a stride of all quantities, took 44.6 us on 1e5 particles (1,564 partials)
// and 17.9 on 2,000; this takes 8.0 and 4.4.
constexpr int RED_Q = ADJ_NPART + ADJ_NBPARAM;  // quantities: partials, bonds
constexpr int RED_WG = 1024;
__global__ __launch_bounds__(RED_WG) void k_adj_reduce(AdjStep st, AdjState g) {
    __shared__ double share[RED_Q][256];
    __shared__ double tot[RED_Q];
    __shared__ double wsum[MAXWALLS];
    touch_lines<sizeof(AdjStep) + sizeof(AdjState)>((cvoid*)__builtin_amdgcn_kernarg_segment_ptr());
    touch_lines<sizeof(DevParams)>((cvoid*)(st.ptab + blockIdx.x));
    CParams& p = *(CParams*)(st.ptab + blockIdx.x);
    const uint32_t wb0 = p.base / ADJ_PPB, nwb = p.npad / ADJ_PPB;
    const uint32_t nwg = st.ntot / ADJ_PPB;
    const uint32_t grp = threadIdx.x / 256, t = threadIdx.x % 256;
    const bool bonds = st.nbond && p.nb0;
    // What the results are added to, requested before the sums.
    double* gp = g.gparam + (size_t)p.sim * ADJ_NPARAM;
    double* W = g.wall + (size_t)p.wall_base * ADJ_WALL;
    double old = 0.0, P = 0.0, U = 0.0, mass = 1.0;
    if (threadIdx.x < ADJ_NPARAM) old = gp[threadIdx.x];
    const uint32_t w = threadIdx.x;
    if (w < p.nw) {
        P = W[w * ADJ_WALL];
        U = W[w * ADJ_WALL + 1];
        mass = st.wall_mvfd[p.wall_base + w].x;
    }
    constexpr int QPG = (ADJ_NPART + 3) / 4;  // quantities per group
    double s[QPG];
#pragma unroll
    for (int j = 0; j < QPG; ++j) s[j] = 0.0;
    for (uint32_t k = t; k < nwb; k += 256) {
#pragma unroll
        for (int j = 0; j < QPG; ++j) {
            const int q = (int)grp + 4 * j;
            if (q < ADJ_NPART) s[j] += g.part[(size_t)q * nwg + wb0 + k];
        }
    }
#pragma unroll
    for (int j = 0; j < QPG; ++j) {
        const int q = (int)grp + 4 * j;
        if (q < ADJ_NPART) share[q][t] = s[j];
    }
    static_assert(ADJ_NBPARAM == 4, "one bond quantity per group");
    if (bonds) {
        double b = 0.0;
        const double* v = g.bpart + (size_t)p.bond_base * ADJ_NBPARAM + grp;
        for (uint32_t k = t; k < p.nb0; k += 256) b += v[(size_t)k * ADJ_NBPARAM];
        share[ADJ_NPART + grp][t] = b;
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    for (int q = (int)wave; q < (bonds ? RED_Q : ADJ_NPART); q += RED_WG / 64) {
        double v = (share[q][lane] + share[q][lane + 128]) +
                   (share[q][lane + 64] + share[q][lane + 192]);
#pragma unroll
        for (unsigned h = 32; h > 0; h >>= 1) v += __shfl_down(v, h, 64);
        if (lane == 0) tot[q] = v;
    }
    __syncthreads();
    if (threadIdx.x < ADJ_NPARAM) {
        const double b = threadIdx.x < ADJ_NBPARAM && bonds ? tot[ADJ_NPART + threadIdx.x] : 0.0;
        gp[threadIdx.x] = old + (tot[threadIdx.x] + b);
    }
    // Work-item w: wall w.
    const double dt = p.dt;
    if (w < p.nw) {
        const double cp = tot[ADJ_NPARAM + 2 * w], cu = tot[ADJ_NPARAM + 2 * w + 1];
        double* sw = W + w * ADJ_WALL;
        if (p.wmode[w] == 0) {
            sw[0] = P + cp;
            sw[1] = U + cu;
        } else {
            const double s0 = P + cp, s1 = dt * P + U + cu;
            const double A = st.first ? 0.0 : -(dt * dt / 6.0) * P - 0.5 * dt * U;
            sw[0] = s0;
            sw[1] = s1;
            sw[2] = A;
            if (p.wmode[w] == 1)
                wsum[w] = (A + (2.0 / 3.0) * dt * dt * s0 + 1.5 * dt * s1) / mass;
        }
    }
    __syncthreads();
    // The force sums' cotangents: of wall w's own sum, or all of wall 0's.
    if (w < p.nw) {
        double f = 0.0;
        for (uint32_t k = 0; k < p.nw; ++k)
            if (p.wmode[k] == 1 && (p.wall_sums ? k : 0u) == w) f += wsum[k];
        W[w * ADJ_WALL + 3] = f;
    }
}

// Host rows <-> batch arrays.
__device__ __forceinline__ bool host_row(const AdjStep& st, uint32_t i, uint32_t& h) {
    CParams& p = *(CParams*)(st.ptab + st.chunk_sim[i / 256]);
    const uint32_t local = i - p.base;
    h = p.hbase + local;
    return local < p.np;
}

__global__ __launch_bounds__(256) void k_adj_expand(double4* dst, const double* src, AdjStep st) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= st.ntot) return;
    uint32_t h;
    dst[i] = host_row(st, i, h) ? make_double4(src[3 * h], src[3 * h + 1], src[3 * h + 2], 0.0)
                                : make_double4(0.0, 0.0, 0.0, 0.0);
}

__global__ __launch_bounds__(256) void k_adj_pack(double* dst, const double4* src, AdjStep st) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    uint32_t h;
    if (i >= st.ntot || !host_row(st, i, h)) return;
    const double4 v = src[i];
    dst[3 * h] = v.x;
    dst[3 * h + 1] = v.y;
    dst[3 * h + 2] = v.z;
}

// dst[i].xyz += the host row of particle i (a loss term on an intermediate
// state).
__global__ __launch_bounds__(256) void k_adj_accumulate(double4* dst, const double* src,
                                                        AdjStep st) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    uint32_t h;
    if (i >= st.ntot || !host_row(st, i, h)) return;
    double4 v = dst[i];
    v.x += src[3 * h];
    v.y += src[3 * h + 1];
    v.z += src[3 * h + 2];
    dst[i] = v;
}

}  // namespace

hipError_t launch_adj_accumulate(double4* dst, const double* src, const AdjStep& st,
                                 hipStream_t s) {
    hipLaunchKernelGGL(k_adj_accumulate, dim3((st.ntot + 255) / 256), dim3(256), 0, s, dst, src,
                       st);
    return hipGetLastError();
}

hipError_t launch_adj_expand(double4* dst, const double* src, const AdjStep& st, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_expand, dim3((st.ntot + 255) / 256), dim3(256), 0, s, dst, src, st);
    return hipGetLastError();
}

hipError_t launch_adj_pack(double* dst, const double4* src, const AdjStep& st, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_pack, dim3((st.ntot + 255) / 256), dim3(256), 0, s, dst, src, st);
    return hipGetLastError();
}

hipError_t launch_adj_reduce(const AdjStep& st, const AdjState& g, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_reduce, dim3(st.nsim), dim3(RED_WG), 0, s, st, g);
    return hipGetLastError();
}

hipError_t launch_adj_step(const AdjStep& st, const AdjState& g, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_step, dim3(st.ntot / ADJ_PPB), dim3(256), 0, s, st, g);
    if (st.nbond) {
        hipLaunchKernelGGL(k_adj_bonds, dim3((st.nbond + 255) / 256), dim3(256), 0, s, st, g);
        hipLaunchKernelGGL(k_adj_bond_gather, dim3(st.ntot / 256), dim3(256), 0, s, st, g);
    }
    if (!st.accumulate) return launch_adj_reduce(st, g, s);
    return hipGetLastError();
}

}  // namespace sphx
