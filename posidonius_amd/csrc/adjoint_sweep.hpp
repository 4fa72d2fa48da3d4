// adjoint_sweep.hpp -- the reverse sweep in two parts, for ensembles that leave
// most of the chip idle.
//
// The reverse of a step is linear in the cotangents and everything else in it
// follows from the tape: only the chain of small products below is serial.
// prepare_step, one wavefront per set of systems, step and part of the step,
// writes the coefficients of every product of a stretch of steps;
// sweep_stretch walks the stretch backwards and only multiplies.  In place of
// 40 us a step (one wavefront a SIMD at most, 11,000 vector instructions in
// one chain) the preparation, spread over the chip, takes 4.8 us and the sweep
// 6.5 us, bound by the latency of its 20 exchanges through LDS; both at once 7.4
// us (1,024 systems of four bodies).  An ensemble that fills the chip is bound by
// its instructions, not by their chain, and would be by the coefficients'
// traffic (3 KB a body and step each way): there adjoint_segment_kernel, which
// keeps nothing, is the faster one.
//
// Coefficients of a step, planes of two doubles per body, body fastest:
//   each kick (the second one first), for every component i of the cotangents
//   of the pair's acceleration, of dL_p/dt and of dL_h/dt (i = 0..8):
//     (U, P)[i], (H, R)[i]   the components of the cotangents of the relative
//       velocity, the body's spin angular momentum, the host's, (h/2 times) and
//       of the relative position (h times)
//     the parameters' gradients (h times) that depend on i: dissipation factor
//       and fluid Love number of the host and of the body, both Love numbers
//   each Kepler drift (the second one first): its transposed Jacobian, by
//       columns of (Q, P); Jacobi: with the interaction's indirect term
//   gravity: with every body of the chain, V = sqrt(3 G / d^5) d and w = G / d^3,
//       the pair's Hessian being V V^T - w 1
#pragma once

#include "adjoint_kernels.hpp"

#pragma clang fp contract(on)   // see adjoint_kernels.hpp

namespace posdev {

constexpr int CF_KICK = 69;      // planes of a kick: 54 of the matrix, 15 of the parameters
constexpr int CF_DRIFT = 18;     // planes of a Kepler drift
constexpr int CF_K2 = 0, CF_K1 = CF_KICK, CF_D2 = 2 * CF_KICK, CF_D1 = CF_D2 + CF_DRIFT, CF_GRAV = CF_D1 + CF_DRIFT;
__host__ __device__ constexpr int coefficient_planes(int max_n) { return CF_GRAV + 2 * max_n; }

struct Coefficients {
    double2 *base;     // [steps][planes][n_bodies]
    int planes, n_bodies;
    __device__ __forceinline__ double2 *at(int step, int plane, int body) const {
        return base + ((size_t)step * planes + plane) * (size_t)n_bodies + body;
    }
};

struct PrepareLds {
    double m[WAVE], I[WAVE], R[WAVE], sg[WAVE], k2[WAVE], kf[WAVE], eta[WAVE];
    double wv[3][WAVE], wL[3][WAVE];
    double xb[9][WAVE];
};

// The coefficients of one kick: the columns of the pair's vector-Jacobian
// product (a host's are zero but for its own wind torque).  KIND: the three
// columns of the acceleration's cotangent, of dL_p/dt's or of dL_h/dt's, each of
// which needs its part of the product only.
template <int KIND>
__device__ __forceinline__ void write_kick_columns(const Coefficients &Cf, int t, int plane, const AdjLane &A,
                                                   const KickPoint &K, double h) {
    const double hh = 0.5 * h;
    const double im = 1. / A.m, sI = hh / A.I, sIh = hh / A.Ih;
    const size_t nb = Cf.n_bodies;
#pragma unroll 1
    for (int i = 0; i < 3; ++i) {
        const V3 e{i == 0 ? 1. : 0., i == 1 ? 1. : 0., i == 2 ? 1. : 0.};
        const V3 z{0., 0., 0.};
        posadj::PairIn Ib{z, z, z, z};
        posadj::PairParBar Pb{0., 0., 0., 0., 0., 0.};
        if (A.orbiting()) {
            // the force on the body and its acceleration enter as F / m + g
            const posadj::PairOut ob{KIND == 0 ? im * e : z, KIND == 0 ? e : z, KIND == 1 ? e : z, KIND == 2 ? e : z};
            posadj::pair_vjp_of<KIND == 0, KIND == 1, KIND == 2>(K.C, K.P, K.in, ob, Ib, Pb);
        }
        if (KIND == 1 && A.wind) Ib.Wp += wind_vjp(A, K.in.Wp, e);
        const V3 U = hh * Ib.u, P = sI * Ib.Wp, H = sIh * Ib.Wh, R = h * Ib.r;
        double2 *o = Cf.at(t, plane + 6 * (3 * KIND + i), A.body);
        o[0] = double2{U.x, P.x}; o[nb] = double2{U.y, P.y}; o[2 * nb] = double2{U.z, P.z};
        o[3 * nb] = double2{H.x, R.x}; o[4 * nb] = double2{H.y, R.y}; o[5 * nb] = double2{H.z, R.z};
        const double2 ph{h * Pb.sh, h * Pb.kfh}, pp{h * Pb.sp, h * Pb.kfp};
        if (KIND == 0) {
            double2 *q = Cf.at(t, plane + 54 + 3 * i, A.body);
            q[0] = ph; q[nb] = pp; q[2 * nb] = double2{h * Pb.k2h, h * Pb.k2p};
        } else {
            *Cf.at(t, plane + 63 + 2 * i + (KIND == 1 ? 1 : 0), A.body) = KIND == 1 ? pp : ph;
        }
    }
}
__device__ inline void write_kick(const Coefficients &Cf, int t, int plane, const AdjLane &A, const KickPoint &K,
                                  double h) {
    write_kick_columns<0>(Cf, t, plane, A, K, h);
    write_kick_columns<1>(Cf, t, plane, A, K, h);
    write_kick_columns<2>(Cf, t, plane, A, K, h);
}

// The coefficients of one Kepler drift; N: the interaction's indirect term at Q,
// which the drift's initial position also enters.
__device__ inline void write_drift(const Coefficients &Cf, int t, int plane, const AdjLane &A, double mu, double dt,
                                   double X, V3 Q, V3 P, const double g[6], const Indirect &N) {
#pragma unroll 1
    for (int i = 0; i < 6; ++i) {
        const V3 e{i % 3 == 0 ? 1. : 0., i % 3 == 1 ? 1. : 0., i % 3 == 2 ? 1. : 0.};
        const V3 z{0., 0., 0.};
        V3 q = z, p = z;
        if (A.orbiting()) {
            posadj::kepler_vjp_g(mu, dt, X, Q, P, i < 3 ? e : z, i < 3 ? z : e, q, p, g);
            q += N.r3 * p - (N.r5 * posadj::dot(Q, p)) * Q;
        }
        double2 *o = Cf.at(t, plane + 3 * i, A.body);
        const size_t nb = Cf.n_bodies;
        o[0] = double2{q.x, p.x}; o[nb] = double2{q.y, p.y}; o[2 * nb] = double2{q.z, p.z};
    }
}

// The coefficients of the step at `row` of the tape, into step t of the
// workspace: the first kick's, or all others; slots: the chain positions the
// sweep's kernel reads.
template <bool ALT, bool EVO>
__device__ inline void prepare_step(const TapeRef &T, PrepareLds &L, AdjLane &A, const Coefficients &Cf, int row, int t,
                                    int slots, bool first_kick) {
    const StepTape S = step_tape(T, A, row);
    step_radii<EVO>(T, L, A, row);
    const double h = 0.5 * A.dt;
    if (first_kick) {
        wsync();
        if (EVO && A.evolving) A.Ih = L.I[A.hl()];
        const KickPoint K1 = kick_point(L, A, S.x0, S.v0, S.L0, S.v1, S.L1);
        if (A.valid) write_kick(Cf, t, CF_K1, A, K1, h);
        return;
    }
    const bool jacobi = ALT && A.jacobi, whds = ALT && A.whds;
    const DriftPoint D = jacobi ? drift_point_jacobi<EVO>(L, A, S)
                       : whds ? drift_point<EVO, true>(L, A, S)
                              : drift_point<EVO, false>(L, A, S);
    // gravity: the pairs of the interaction, by the other body's chain position
    if (A.valid) put3(L, 0, A.lane, D.xg);
    wsync();
    const int first = A.host == 0 ? 1 : 0;
    for (int c = 0; A.valid && c < slots; ++c) {
        const int j = c == 0 ? A.host : (c - 1 < A.host ? c - 1 : c);
        double2 a{0., 0.}, b{0., 0.};
        const bool pair = c < A.n && j != A.k &&
                          (jacobi ? !((A.is_host && j == first) || (j == A.host && A.k == first))
                                  : A.orbiting() && j != A.host);
        if (pair) {
            const V3 d = D.xg - get3(L, 0, A.gbase + j);
            const double id = 1. / sqrt(posadj::dot(d, d));
            const double w = posadj::G_K2 * id * id * id;
            const V3 V = (sqrt(3. * w) * id) * d;
            a = double2{V.x, V.y};
            b = double2{V.z, w};
        }
        *Cf.at(t, CF_GRAV + 2 * c, A.body) = a;
        *Cf.at(t, CF_GRAV + 2 * c + 1, A.body) = b;
    }
    wsync();
    const double mu = posadj::G_K2 * (jacobi ? A.eta_le : whds ? A.mh + A.m : A.mh);
    const Indirect none{0., 0.};
    if (A.valid) {
        write_drift(Cf, t, CF_D2, A, mu, h, S.X2, D.Q2, D.P1pp, D.g2, jacobi ? indirect_term(A, D.Q2) : none);
        write_drift(Cf, t, CF_D1, A, mu, h, S.X1, D.Q0, D.P0, D.g1, none);
    }
    const KickPoint K2 = kick_point(L, A, S.x2, D.v2p, S.L1, S.v2, S.L2);
    if (A.valid) write_kick(Cf, t, CF_K2, A, K2, h);
}

// ---------------------------------------------------------------------------
// The sweep: four lanes per body, three of them each holding one component of
// the cotangents, so that a product's rows and its operands sit in
// neighbouring lanes and a wavefront's registers hold the coefficients of half a step
// in use and of half a step on their way.  NM slots per system, in chain order
// (host first, then index order).
// ---------------------------------------------------------------------------
struct SweepLds {
    double v[5][WAVE];
    double m[WAVE / 4];        // mass, and with the chain's up to the body: 1 / eta_lt
    double inv_lt[WAVE / 4];
};

struct KickRow {
    double2 up[9], hr[9];      // (U, P) and (H, R) of this lane's component
    double2 pa[3], pb[3];      // this lane's two parameters, by the acceleration's cotangent and one of the torques'
};
struct DriftRow {
    double2 d[6];              // (Q, P) of this lane's component
};

struct SweepLane {
    int lane, c, slot, g0;     // component (3: none), chain position, first lane of the system
    bool live, orb, spin;      // holds a component of a body; of an orbiting one; spins integrated
    int body;
    double m, rm, mM, dt, h;   // mass, m / m_host (0 for the host), m / M
    double ifv, fv, cw, cj, dtf, whds;   // heliocentric and WHDS transforms (see adjoint_step)
    double ile, ilt;           // Jacobi: m / eta_le, 1 / eta_lt
    double lx, lv, lL, wv, wL;
    double p0, p1;             // gradients of this lane's parameters
};

// The sweep's stop of the midpoint equation (see ADJ_FIXED_POINT_TOL).  The last
// pass's products also give the position and parameter parts, so it stops where
// the pass changes mu by no more than its rounding: one evaluation fewer than a
// stop at 1e-10 with those parts formed after it, at the same accuracy.
constexpr int SWEEP_BITS = 50;

// High word of the largest of a body's components (lane 3 holds 0): the exponent
// and 20 bits, in the order of the magnitudes.
__device__ __forceinline__ int quad_magnitude(double x) {
    int a = __double2hiint(x) & 0x7fffffff;
    a = max(a, __builtin_amdgcn_mov_dpp(a, 0xB1, 0xf, 0xf, true));    // lanes 1 0 3 2
    return max(a, __builtin_amdgcn_mov_dpp(a, 0x4E, 0xf, 0xf, true)); // lanes 2 3 0 1
}
// |a - b| at most 2^-SWEEP_BITS |a| (or zero)
__device__ __forceinline__ bool quad_settled(double a, double b) {
    const int d = quad_magnitude(a - b);
    return d == 0 || d + (SWEEP_BITS << 20) <= quad_magnitude(a);
}

__device__ __forceinline__ V3 lds3(const double *row, int lane0) { return V3{row[lane0], row[lane0 + 1], row[lane0 + 2]}; }
template <int NM>
__device__ __forceinline__ double slot_sum(const double *row, const SweepLane &A) {
    double s = 0.;
#pragma unroll
    for (int j = 0; j < NM; ++j) s += row[A.g0 + 4 * j + A.c];
    return s;
}

__device__ __forceinline__ KickRow load_kick(const Coefficients &Cf, const SweepLane &A, int t, int plane) {
    KickRow K;
    const double2 z{0., 0.};
    if (A.live) {
        const double2 *o = Cf.at(t, plane + A.c, A.body);
        const size_t nb = Cf.n_bodies;
#pragma unroll
        for (int i = 0; i < 9; ++i) { K.up[i] = o[(6 * i) * nb]; K.hr[i] = o[(6 * i + 3) * nb]; }
#pragma unroll
        for (int i = 0; i < 3; ++i) K.pa[i] = o[(54 + 3 * i) * nb];
        const double2 *q = Cf.at(t, plane + 63 + (A.c == 1 ? 1 : 0), A.body);
#pragma unroll
        for (int i = 0; i < 3; ++i) K.pb[i] = q[(2 * i) * nb];
    } else {
#pragma unroll
        for (int i = 0; i < 9; ++i) { K.up[i] = z; K.hr[i] = z; }
#pragma unroll
        for (int i = 0; i < 3; ++i) { K.pa[i] = z; K.pb[i] = z; }
    }
    return K;
}
__device__ __forceinline__ DriftRow load_drift(const Coefficients &Cf, const SweepLane &A, int t, int plane) {
    DriftRow D;
    if (A.live) {
        const double2 *o = Cf.at(t, plane + A.c, A.body);
#pragma unroll
        for (int i = 0; i < 6; ++i) D.d[i] = o[(3 * i) * (size_t)Cf.n_bodies];
    } else {
#pragma unroll
        for (int i = 0; i < 6; ++i) D.d[i] = double2{0., 0.};
    }
    return D;
}
template <int NM> struct GravityRow {
    double2 a[NM], b[NM];
};
template <int NM>
__device__ __forceinline__ GravityRow<NM> load_gravity(const Coefficients &Cf, const SweepLane &A, int t) {
    GravityRow<NM> G;
    if (A.live) {
        const double2 *o = Cf.at(t, CF_GRAV, A.body);
        const size_t nb = Cf.n_bodies;
#pragma unroll
        for (int j = 0; j < NM; ++j) { G.a[j] = o[(2 * j) * nb]; G.b[j] = o[(2 * j + 1) * nb]; }
    } else {
#pragma unroll
        for (int j = 0; j < NM; ++j) { G.a[j] = double2{0., 0.}; G.b[j] = double2{0., 0.}; }
    }
    return G;
}

// Adjoint of one kick (see kick_adjoint).
template <int NM>
__device__ __forceinline__ void sweep_kick(SweepLds &S, SweepLane &A, const KickRow &K, unsigned long long group) {
    const bool host = A.slot == 0;
    const int own = A.lane & ~3;
    double mv = A.lv + A.wv, mL = A.spin ? A.lL + A.wL : 0.;
    double nv, nL, gL, gx, in[9];
    for (int pass = 1;; ++pass) {
        S.v[0][A.lane] = mv; S.v[1][A.lane] = mL;
        wsync();
        const V3 ov = lds3(S.v[0], own), oL = lds3(S.v[1], own), hv = lds3(S.v[0], A.g0), hL = lds3(S.v[1], A.g0);
        in[0] = ov.x - A.rm * hv.x; in[1] = ov.y - A.rm * hv.y; in[2] = ov.z - A.rm * hv.z;
        in[3] = oL.x; in[4] = oL.y; in[5] = oL.z;
        in[6] = hL.x; in[7] = hL.y; in[8] = hL.z;
        double u = 0., p = 0., q = 0., r = 0.;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            u += K.up[i].x * in[i]; p += K.up[i].y * in[i];
            q += K.hr[i].x * in[i]; r += K.hr[i].y * in[i];
        }
        S.v[2][A.lane] = u; S.v[3][A.lane] = q; S.v[4][A.lane] = r;
        wsync();
        double gv = u;
        gL = p; gx = r;
        if (host) {   // its own rows are zero but for the wind torque's in p
            gv = -slot_sum<NM>(S.v[2], A);
            gL = p + slot_sum<NM>(S.v[3], A);
            gx = -slot_sum<NM>(S.v[4], A);
        }
        nv = A.lv + gv;
        nL = A.spin ? A.lL + gL : 0.;
        const bool conv = quad_settled(nv, mv) && quad_settled(nL, mL);
        const unsigned long long all = __ballot(conv);
        if (pass >= ADJ_MAX_PASSES || __all((all & group) == group)) break;
        // a system that is done repeats the pass as it was
        if ((all & group) != group) { mv = nv; mL = nL; }
    }
    A.wv = nv - A.lv;
    A.wL = A.spin ? nL - A.lL : 0.;
    A.lv = 2. * nv - A.lv;
    A.lL = A.spin ? 2. * nL - A.lL : A.lL + 2. * gL;
    A.lx += gx;
    double s0 = 0., s1 = 0.;
    const double side = A.c == 2 ? 0. : 1.;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double t = side * (A.c == 1 ? in[3 + i] : in[6 + i]);
        s0 += K.pa[i].x * in[i] + K.pb[i].x * t;
        s1 += K.pa[i].y * in[i] + K.pb[i].y * t;
    }
    A.p0 += s0;
    A.p1 += s1;
}

// (Q, P) components of a drift's transposed Jacobian applied to the body's (q, p)
__device__ __forceinline__ void sweep_drift(SweepLds &S, const SweepLane &A, const DriftRow &D, double q, double p,
                                            double &Q, double &P) {
    S.v[0][A.lane] = q; S.v[1][A.lane] = p;
    wsync();
    const V3 a = lds3(S.v[0], A.lane & ~3), b = lds3(S.v[1], A.lane & ~3);
    Q = D.d[0].x * a.x + D.d[1].x * a.y + D.d[2].x * a.z + D.d[3].x * b.x + D.d[4].x * b.y + D.d[5].x * b.z;
    P = D.d[0].y * a.x + D.d[1].y * a.y + D.d[2].y * a.z + D.d[3].y * b.x + D.d[4].y * b.y + D.d[5].y * b.z;
    wsync();
}

// Cotangent of a body's position from the accelerations' cotangents a
// (universe.rs:198-303): sum_j (V V^T - w) (m_j a - m a_j).
template <int NM>
__device__ __forceinline__ double sweep_gravity(SweepLds &S, const SweepLane &A, const GravityRow<NM> &G, double a) {
    S.v[2][A.lane] = a;
    wsync();
    const V3 o = lds3(S.v[2], A.lane & ~3);
    double x = 0.;
#pragma unroll
    for (int j = 0; j < NM; ++j) {
        const double mj = S.m[(A.g0 >> 2) + j];
        const V3 b = lds3(S.v[2], A.g0 + 4 * j);
        const V3 s{mj * o.x - A.m * b.x, mj * o.y - A.m * b.y, mj * o.z - A.m * b.z};
        const double t = G.a[j].x * s.x + G.a[j].y * s.y + G.b[j].x * s.z;
        const double V = A.c == 0 ? G.a[j].x : (A.c == 1 ? G.a[j].y : G.b[j].x);
        const double sc = A.c == 0 ? s.x : (A.c == 1 ? s.y : s.z);
        x += V * t - G.b[j].y * sc;
    }
    wsync();
    return x;
}

// The drifts and the interaction of one step in heliocentric or WHDS
// coordinates (see adjoint_step).  The forces of gravity on the orbiting bodies
// cancel in their sum, so the jumps share one sum of position cotangents.
template <int NM>
__device__ __forceinline__ void sweep_middle(SweepLds &S, SweepLane &A, const DriftRow &D2, const DriftRow &D1,
                                             const GravityRow<NM> &G) {
    S.v[0][A.lane] = A.lx; S.v[1][A.lane] = A.lv;
    wsync();
    const double xt = slot_sum<NM>(S.v[0], A), vt = slot_sum<NM>(S.v[1], A);
    const double lvh = S.v[1][A.g0 + A.c];
    wsync();
    double Q, P;
    sweep_drift(S, A, D2, A.orb ? A.lx - A.mM * xt : 0., A.orb ? A.ifv * A.lv - A.cw * lvh : 0., Q, P);
    S.v[0][A.lane] = Q;
    wsync();
    const double SQ = slot_sum<NM>(S.v[0], A);
    P += A.cj * (SQ - A.whds * Q);
    const double xg = sweep_gravity<NM>(S, A, G, A.dtf * P);
    if (A.orb) Q += xg;
    P += A.cj * (SQ - A.whds * Q);
    double Q0, P0;
    sweep_drift(S, A, D1, Q, P, Q0, P0);
    const double v1 = A.fv * P0;
    S.v[0][A.lane] = Q0; S.v[1][A.lane] = v1;
    wsync();
    const double SX = slot_sum<NM>(S.v[0], A), SV = slot_sum<NM>(S.v[1], A);
    A.lx = (A.orb ? Q0 : A.live ? -SX : 0.) + A.mM * xt;
    A.lv = (A.orb ? v1 : 0.) + A.mM * (vt + A.dt * xt - SV);
    wsync();
}

// The same in Jacobi coordinates (see adjoint_step_jacobi).
template <int NM>
__device__ __forceinline__ void sweep_middle_jacobi(SweepLds &S, SweepLane &A, const DriftRow &D2, const DriftRow &D1,
                                                    const GravityRow<NM> &G) {
    auto upto = [&](const double *row) {
        double s = 0.;
#pragma unroll
        for (int j = 0; j < NM; ++j) s += j <= A.slot ? row[A.g0 + 4 * j + A.c] : 0.;
        return s;
    };
    auto after = [&](const double *row) {
        double s = 0.;
#pragma unroll
        for (int j = 1; j < NM; ++j) s += j > A.slot ? S.inv_lt[(A.g0 >> 2) + j] * row[A.g0 + 4 * j + A.c] : 0.;
        return s;
    };
    S.v[0][A.lane] = A.lx; S.v[1][A.lane] = A.lv;
    wsync();
    const double xt = slot_sum<NM>(S.v[0], A), vt = slot_sum<NM>(S.v[1], A);
    const double q = A.orb ? A.lx - A.ile * upto(S.v[0]) : 0., p = A.orb ? A.lv - A.ile * upto(S.v[1]) : 0.;
    wsync();
    double Q, P;
    sweep_drift(S, A, D2, q, p, Q, P);
    S.v[0][A.lane] = A.dt * P;
    wsync();
    const double acc = A.dt * P - A.m * after(S.v[0]);
    const double xg = sweep_gravity<NM>(S, A, G, acc);
    S.v[0][A.lane] = xg;
    wsync();
    if (A.orb) Q += xg - A.ile * upto(S.v[0]);
    wsync();
    double Q0, P0;
    sweep_drift(S, A, D1, Q, P, Q0, P0);
    S.v[0][A.lane] = Q0; S.v[1][A.lane] = P0;
    wsync();
    A.lx = Q0 - A.m * after(S.v[0]) + A.mM * xt;
    A.lv = P0 - A.m * after(S.v[1]) + A.mM * (vt + A.dt * xt);
    wsync();
}

// What a stretch hands to the one before it in time: the midpoint solve's last
// correction and the sums of the lane's parameters, three components each.  The
// stretches' length then leaves no trace in the result.
enum { CARRY_WV = 0, CARRY_WL = 3, CARRY_P0 = 6, CARRY_P1 = 9, CARRY_ROWS = 12 };

// Lane state of the systems of one wavefront: systems first.., NM slots each;
// first: no stretch was swept before.
template <int NM>
__device__ __forceinline__ void sweep_load(const AdjArgs &Ar, SweepLds &S, SweepLane &A, int &sys, bool &jacobi, bool first) {
    const DevEnsemble &E = Ar.E;
    const int lane = threadIdx.x;
    const int quad = lane >> 2;
    const int nb = E.n_bodies;
    A.lane = lane;
    A.c = lane & 3;
    A.slot = quad % NM;
    A.g0 = (quad - A.slot) * 4;
    sys = blockIdx.x * (16 / NM) + quad / NM;
    const bool in = sys < E.n_systems;
    if (!in) sys = E.n_systems - 1;
    const int b0 = E.body_offset[sys];
    const int n = E.body_offset[sys + 1] - b0, host = E.host[sys];
    auto body = [&](int slot) { return b0 + (slot == 0 ? host : (slot - 1 < host ? slot - 1 : slot)); };
    const bool valid = in && A.slot < n;
    A.live = valid && A.c < 3;
    A.orb = A.live && A.slot > 0;
    A.body = valid ? body(A.slot) : b0;
    const uint32_t eff = E.effects[sys];
    A.spin = eff & (POS_EFFECT_TIDES | POS_EFFECT_ROTATIONAL_FLATTENING | POS_EFFECT_GENERAL_RELATIVITY | POS_EFFECT_EVOLUTION);
    jacobi = E.coord[sys] == POS_COORD_JACOBI;
    const bool whds = E.coord[sys] == POS_COORD_WHDS;
    const double mh = E.mass[b0 + host];
    double M = 0., eta = 0.;
    for (int j = 0; j < n; ++j) {
        const double m = E.mass[body(j)];
        M += m;
        if (j <= A.slot) eta += m;
    }
    A.m = A.live ? E.mass[A.body] : 0.;
    A.dt = E.dt[sys];
    A.h = 0.5 * A.dt;
    A.rm = A.orb ? A.m / mh : 0.;
    A.mM = A.m / M;
    const double f = (mh + A.m) / mh, w = A.m / (mh + A.m);
    A.fv = A.orb && whds ? f : 1.;
    A.ifv = 1. / A.fv;
    A.cw = whds ? w : A.m / mh;
    A.cj = A.orb ? A.h * A.cw : 0.;
    A.dtf = A.orb ? A.dt * A.fv : 0.;
    A.whds = whds ? 1. : 0.;
    A.ile = A.orb ? A.m / eta : 0.;
    if (A.c == 0) {
        S.m[quad] = A.m;
        S.inv_lt[quad] = A.orb ? 1. / (eta - A.m) : 0.;
    }
    A.lx = A.live ? Ar.lx[A.c * nb + A.body] : 0.;
    A.lv = A.live ? Ar.lv[A.c * nb + A.body] : 0.;
    A.lL = A.live ? Ar.lL[A.c * nb + A.body] : 0.;
    auto carried = [&](int row) { return A.live && !first ? Ar.carry[(size_t)(row + A.c) * nb + A.body] : 0.; };
    A.wv = carried(CARRY_WV);
    A.wL = carried(CARRY_WL);
    A.p0 = carried(CARRY_P0);
    A.p1 = carried(CARRY_P1);
    wsync();
}

// The cotangents, the parameters' gradients so far (a host's are the sums over
// its pairs) and what the next stretch goes on from.
template <int NM>
__device__ __forceinline__ void sweep_store(const AdjArgs &Ar, SweepLds &S, const SweepLane &A) {
    const int nb = Ar.E.n_bodies;
    S.v[0][A.lane] = A.p0; S.v[1][A.lane] = A.p1;
    wsync();
    const double s0 = slot_sum<NM>(S.v[0], A), s1 = slot_sum<NM>(S.v[1], A);
    if (!A.live) return;
    Ar.lx[A.c * nb + A.body] = A.lx;
    Ar.lv[A.c * nb + A.body] = A.lv;
    Ar.lL[A.c * nb + A.body] = A.lL;
    auto carry = [&](int row, double x) { Ar.carry[(size_t)(row + A.c) * nb + A.body] = x; };
    carry(CARRY_WV, A.wv);
    carry(CARRY_WL, A.wL);
    carry(CARRY_P0, A.p0);
    carry(CARRY_P1, A.p1);
    if (A.c == 0 && !A.orb) { Ar.gs[A.body] = s0; Ar.gkf[A.body] = s1; }
    if (A.c == 1 && A.orb) { Ar.gs[A.body] = A.p0; Ar.gkf[A.body] = A.p1; }
    if (A.c == 2) Ar.gk2[A.body] = A.orb ? A.p1 : s0;
}

// Steps [row0, row0 + len) of a segment and where their coefficients are, as the
// workspace's steps 0 .. len - 1.
struct Stretch {
    TapeRef T;
    long long seg_start;
    int row0, len;
    bool first;           // the first to be swept
    Coefficients Cf;
};

// The reverse of a stretch, last step first.
template <int NM, bool ALT>
__device__ inline void sweep_stretch(const AdjArgs &Ar, SweepLds &S, const Stretch &W) {
    const Coefficients &Cf = W.Cf;
    const int len = W.len;
    SweepLane A;
    int sys;
    bool jacobi;
    sweep_load<NM>(Ar, S, A, sys, jacobi, W.first);
    const long long done = Ar.steps_done[sys] - W.seg_start - W.row0;   // steps of the stretch the system took
    const unsigned long long group = (NM == 16 ? ~0ull : ((1ull << (4 * NM % 64)) - 1) << A.g0);
    // Each part's coefficients are asked for a part or more before their use:
    // while a kick runs, those of the drifts and of the step's other kick (at 16
    // slots the other kick's follow only once the first one's are spent, or the
    // registers spill), and then the next step's.
    constexpr bool EARLY = NM < 16;
    KickRow K2 = load_kick(Cf, A, len - 1, CF_K2), K1;
    for (int t = len - 1; t >= 0; --t) {
        if (EARLY) K1 = load_kick(Cf, A, t, CF_K1);
        const DriftRow D2 = load_drift(Cf, A, t, CF_D2), D1 = load_drift(Cf, A, t, CF_D1);
        const GravityRow<NM> G = load_gravity<NM>(Cf, A, t);
        // uniform within the system, not the wavefront: the others keep calling
        // wsync(), which is correct only because the workgroup is one wavefront
        const bool on = t < done;
        if (on) sweep_kick<NM>(S, A, K2, group);
        if (EARLY) K2 = load_kick(Cf, A, t > 0 ? t - 1 : 0, CF_K2);
        else K1 = load_kick(Cf, A, t, CF_K1);
        if (on) {
            if (ALT && jacobi) sweep_middle_jacobi<NM>(S, A, D2, D1, G);
            else sweep_middle<NM>(S, A, D2, D1, G);
        }
        if (!EARLY) K2 = load_kick(Cf, A, t > 0 ? t - 1 : 0, CF_K2);
        if (on) sweep_kick<NM>(S, A, K1, group);
    }
    sweep_store<NM>(Ar, S, A);
}

}  // namespace posdev

#pragma clang fp contract(off)
