// whfast_fixed.hpp -- the step of the fixed effect set (VAR_FAST): systems with
// exactly tides + flattening + Kidder GR with spins, in any coordinates, run by teams of one, two or four
// wavefronts.
//
// Most of a step is the evaluation of those effects inside the two
// implicit-midpoint solves, a long serial instruction stream.  A team of M
// wavefronts holds the same bodies (lane i <-> the same body in each) and
// splits the families of pair terms:
//   M = 1: everything in one wavefront;
//   M = 2: wave 0 tides and flattening, wave 1 the GR terms;
//   M = 4: tides | spin-orbit GR | flattening | 1PN and 2PN GR.
// Wave 0 owns positions and velocities (their updates and the whole drift:
// transforms, Kepler, gravity), wave 1 owns the spin angular momenta (wave 0
// does when alone).  The wavefronts meet at workgroup barriers, two per effects
// evaluation: after the pair terms are published, and after the new
// velocities and spins are.  Between them each owner sums the host reactions
// its update needs, so the sums need no barrier of their own.
//
// Every sum keeps the reference's order and every value its rounding (see
// whfast_step.hpp), so the results do not depend on M.  Pair terms that
// depend only on positions and constants are evaluated once per drift and
// serve the two solves at those positions: the second kick of a step and the
// first kick of the next.
#pragma once

#include "whfast_step.hpp"

namespace posdev {

// ---- LDS of one team --------------------------------------------------------
// What only a team of several wavefronts needs.  Each array is written by one
// wavefront per phase and read by others after a barrier.
struct TeamRows {
    double v[3][WAVE];          // velocities of the current evaluation, written by wave 0
    double x[3][WAVE];          // positions, written by wave 0 after a drift
    double so[3][WAVE];         // spins of the evaluation before a solve, written by their owner
    double ex[15][WAVE];        // an orbiting body's own accelerations and torques for their owner
    double cv[4][WAVE + 1];     // convergence sums of a solve; column WAVE holds +0
    unsigned long long live, snap;   // lanes whose system takes the next step / records a snapshot before it
};
struct NoRows {};
enum { EX_TORQUE_T = 0, EX_TORQUE_R = 3, EX_ACC_R = 6, EX_GR = 9, EX_GR_SO = 12 };

// Mass-only constants of a body.  A wavefront alone keeps them in LDS (its
// registers are full), the wavefronts of a larger team in registers.  The
// host's own entries of the first four, which no pair uses, hold constants of
// the system there: 1 / m_h, the total mass and its reciprocal, and 1 / the
// mass the reverse Jacobi recurrence leaves for the host.
enum {
    K_F = 0,          // Kidder mass factor of the pair with the host (general_relativity.rs:91)
    K_M_OVER_HM = 1,  // m / m_h
    K_MFM = 2,        // (m_h - m) / (m_h + m) (m_h + m) (general_relativity.rs:326-330)
    K_MR = 3,         // m_h m / (m_h + m)
    K_FM_HOST = 4,    // 2 + 3/2 m / m_h
    K_FM_BODY = 5,    // 2 + 3/2 m_h / m
    K_COUNT = 6,
    K_INV_HM = K_F, K_TOTAL = K_M_OVER_HM, K_INV_TOTAL = K_MFM, K_INV_LEFT = K_MR
};

// A lane's body.  The lanes of a group follow the chain of the reference's
// recurrences: lane 0 holds the host, the others follow in body order.  The
// host is thus at a known lane (Lane::host is 0 here), an ordered sum over the
// orbiting bodies runs over lanes 1 to n-1, and only what runs over all bodies
// in body order has to ask where the host stands among them.  A wavefront
// keeps what its role uses; the rest is never loaded.
struct FixedLane : Lane {
    bool orb, host_lane;
    int idx, hidx;              // body index of this lane and of the host within the system
    int nmax;                   // largest body count of this wavefront's systems (uniform)
    bool pairs;                 // it holds systems of two bodies (uniform)
    bool hosts_first;           // every host is its system's body 0 (uniform)
    double near2, far2;         // screen of the pair checks: see fixed_gravity
    double I, inv_I;            // moment of inertia and its reciprocal
    double mu;                  // Jacobi: Kepler mass of this body's drift
    double jeta;                // Jacobi: mass of the chain up to this body
    bool jfirst;                // Jacobi: the first body after the host
    double kc[K_COUNT], ksys[4]; // teams of several wavefronts: the constants above
    double s[3];                // teams of several wavefronts: spin of the last evaluation
};

template <int M, bool JACOBI>
struct FixedLds {
    struct SoloRows { double k[K_COUNT][WAVE]; };
    struct ChainRows {
        // Jacobi chain, masses only (whfast.rs:889-933, 1034-1080), of body j:
        // 1 / the mass before it, and the same in the reverse recurrence, whose
        // masses are found by subtraction
        double ei[WAVE], rei[WAVE];
    };
    double m[WAVE + 1];   // entry WAVE is +0, the mass of the zero column
    double R[WAVE], I[WAVE], k2f[WAVE];
    double s[3][WAVE];    // spins of the current evaluation
    // contributions to the host inside the solves, exchange rows in the
    // drift; column WAVE holds +0 in every row
    double xb[NX][WAVE + 1];
    std::conditional_t<(M > 1), TeamRows, SoloRows> team;
    std::conditional_t<JACOBI, ChainRows, NoRows> chain;

    // A snapshot is recorded by wave 0 while the other wavefronts already write
    // their contributions: it exchanges through rows that only wave 0 writes.
    static constexpr __device__ int hist_x_row(int q) { return C_TF + q; }
    static constexpr __device__ int hist_v_row(int q) { return C_TN + q; }
    // Velocities of the current evaluation.  Alone, the wavefront has read
    // them when it writes the contributions that share their rows.
    __device__ __forceinline__ double &vel(int q, int lane) {
        if constexpr (M == 1) return xb[C_RF + q][lane];
        else return team.v[q][lane];
    }
    __device__ __forceinline__ double konst(const FixedLane &B, int i) const {
        if constexpr (M == 1) return team.k[i][B.lane];
        else return B.kc[i];
    }
    __device__ __forceinline__ double of_system(const FixedLane &B, int i) const {
        if constexpr (M == 1) return team.k[i][B.hl()];
        else return B.ksys[i];
    }
    __device__ __forceinline__ double sigma_of(const DevEnsemble &E, int, int body) const { return E.sigma[body]; }
    __device__ __forceinline__ double k2_of(const DevEnsemble &E, int, int body) const { return E.k2[body]; }
};
// alone, a team's LDS must leave eight of them on a CU
static_assert(sizeof(FixedLds<1, true>) <= 20480, "eight single-wavefront teams per CU");

// Hides a uniform value from the optimiser, so that a loop over the two halves
// of a step is not turned back into two copies of its body.
__device__ __forceinline__ void opaque(int &uniform) { asm volatile("" : "+s"(uniform)); }

// Orders a team's LDS accesses.  Global accesses need no order: no wavefront
// reads what another writes.
template <int M>
__device__ __forceinline__ void team_sync() {
    if constexpr (M == 1) {
        wsync();
    } else {
        team_barrier();
    }
}

// What wavefront ROLE of a team of M does.
template <int M, int ROLE>
struct Role {
    static constexpr bool OWN_V = ROLE == 0;
    static constexpr bool OWN_L = M == 1 || ROLE == 1;
    static constexpr bool TIDES = ROLE == 0;
    static constexpr bool FLAT = M == 4 ? ROLE == 2 : ROLE == 0;
    static constexpr bool ORBIT = M == 4 ? ROLE == 3 : OWN_L;   // 1PN and 2PN
    static constexpr bool SPIN_ORBIT = OWN_L;
};

// Pair terms of an orbiting body with its host that depend only on positions
// and constants; a wavefront fills and keeps those of its families.  Each is
// the rounded value of the reference's expression; a quotient by a kept divisor
// uses its correctly rounded reciprocal (divr), which is exact.
struct FixedGeo {
    double px[3];            // heliocentric position
    Rcp Rd;                  // distance and its reciprocal
    Rcp Rp8;                 // distance^8 and its reciprocal
    double d5;               // distance^5
    double os, op;           // tidal orthogonal components (constant_time_lag.rs:206-264)
    double od, pd, id;       // os / d, op / d, 1 / d
    double conservative;     // conservative radial tidal component (266-307)
    double term1, term2;     // the two dissipative radial terms without their velocity factor
    double m3d5, c15;        // -3 / d^5 and 15 / d^7 (oblate_spheroid.rs:51-60)
    double mgc, mg_d;        // -(G m_h + G m) / (d^2 c^2) and (G m_h + G m) / d
    double c1pn, o1pn;       // 1PN: 2 (2 + f) mg / d and (mg / (d^2 c^2)) 2 (2 - f)
    double c2pn;             // 2PN: 3/4 (12 + 29 f) (mg^2 / d^2)
    double n3[3];            // unit vector of the separation
    // scalar products of the separation with the host's and the body's spins
    // of the previous evaluation (tides/common.rs:143-170,
    // rotational_flattening/common.rs:93-120)
    double rs_star, rs_planet;
};

// Lane of the body of index j of this group.
__device__ __forceinline__ int lane_of_body(const FixedLane &B, int j) {
    return B.gbase + (j == B.hidx ? 0 : j < B.hidx ? j + 1 : j);
}

// ---- ordered sums over the bodies of a group --------------------------------
// Column of chain slot c (>= 1) of a batch: the zero column past the last body.
__device__ __forceinline__ int fold_column(const Lane &B, int c) { return c < B.n ? B.gbase + c : WAVE; }

// Lane q of a group (q < 3) does component q; in a system of two bodies lane 0
// also does component 2.
template <class F>
__device__ __forceinline__ void by_component(const FixedLane &B, F f) {
    if (B.k < 3) f(B.k);
    if (B.pairs && B.n == 2 && B.k == 0) f(2);
}

// T vectors of sums over the orbiting bodies in body order, of the terms in
// rows [0, 3T) of the exchange area, each starting from init (NEG: the terms
// are subtracted).  A skipped slot adds or subtracts +0, which changes no
// value: a sum that starts at +0 is never -0, and -0 - +0 is -0.  DIRECT: every
// lane forms every sum itself, one LDS round trip; otherwise lanes 0-2 form
// one component each and hand it out through rows [12, 12 + 3T), fewer
// instructions for two round trips.  Teams of several wavefronts take the
// first (they run where the chip is not full and latency is all), single
// wavefronts the second.
//
// The loops run to the wavefront's largest system, a uniform bound: a lane
// past its own last body adds the zero column, which costs less than masking
// it out.
template <int T, bool NEG, bool DIRECT, class Lds>
__device__ __forceinline__ void group_sums(Lds &lds, const FixedLane &B, const double (&init)[T][3], double (&out)[T][3]) {
    if constexpr (DIRECT) {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int q = 0; q < 3; ++q) out[t][q] = init[t][q];
        for (int c0 = 1; c0 < B.nmax; c0 += FOLD_BATCH) {
            double a[T][3][FOLD_BATCH];
#pragma unroll
            for (int u = 0; u < FOLD_BATCH; ++u) {
                const int l = fold_column(B, c0 + u);
#pragma unroll
                for (int t = 0; t < T; ++t)
#pragma unroll
                    for (int q = 0; q < 3; ++q) a[t][q][u] = lds.xb[3 * t + q][l];
            }
#pragma unroll
            for (int u = 0; u < FOLD_BATCH; ++u)
#pragma unroll
                for (int t = 0; t < T; ++t)
#pragma unroll
                    for (int q = 0; q < 3; ++q) out[t][q] = NEG ? out[t][q] - a[t][q][u] : out[t][q] + a[t][q][u];
        }
    } else {
        by_component(B, [&](int q) {
            double acc[T];
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t] = q == 0 ? init[t][0] : q == 1 ? init[t][1] : init[t][2];
            const double(*row)[WAVE + 1] = &lds.xb[q];
            for (int c0 = 1; c0 < B.nmax; c0 += FOLD_BATCH) {
                double a[T][FOLD_BATCH];
#pragma unroll
                for (int u = 0; u < FOLD_BATCH; ++u) {
                    const int l = fold_column(B, c0 + u);
#pragma unroll
                    for (int t = 0; t < T; ++t) a[t][u] = row[3 * t][l];
                }
#pragma unroll
                for (int u = 0; u < FOLD_BATCH; ++u)
#pragma unroll
                    for (int t = 0; t < T; ++t) acc[t] = NEG ? acc[t] - a[t][u] : acc[t] + a[t][u];
            }
#pragma unroll
            for (int t = 0; t < T; ++t) lds.xb[12 + 3 * t + q][B.gbase] = acc[t];
        });
        wsync();
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int q = 0; q < 3; ++q) out[t][q] = lds.xb[12 + 3 * t + q][B.gbase];
        wsync();
    }
}

// Host reactions: lane q of a group (q < 3; both lanes of a two-body system
// share the components) sums component q of the contributions over the bodies
// in body order and leaves the host's additional acceleration
// (tides/common.rs:312-345, rotational_flattening/common.rs:203-237,
// general_relativity.rs:236-238, 295-297, 453-455) in row C_TF and its spin
// derivative (tides/common.rs:223-261, rotational_flattening/common.rs:165-201,
// general_relativity.rs:312-315) in row C_TN of the host's column, which is
// never an input.  One address per body serves every row of a component;
// spreading the 24 rows over the lanes instead took 1,450 cycles per
// evaluation of a four-body system, most of them index arithmetic.
template <bool FORCES, bool TORQUES, class Lds>
__device__ __forceinline__ void host_reactions(Lds &lds, const FixedLane &B) {
    constexpr int N = (FORCES ? 5 : 0) + (TORQUES ? 3 : 0), T0 = FORCES ? 5 : 0;
    const int hl = B.hl();
    by_component(B, [&](int q) {
        double(*row)[WAVE + 1] = &lds.xb[q];
        double sum[N];
#pragma unroll
        for (int i = 0; i < N; ++i) sum[i] = 0.;
        for (int c0 = 1; c0 < B.nmax; c0 += FOLD_BATCH) {
            double a[N][FOLD_BATCH];
#pragma unroll
            for (int u = 0; u < FOLD_BATCH; ++u) {
                const int l = fold_column(B, c0 + u);
                if constexpr (FORCES) {
                    a[0][u] = row[C_TF][l]; a[1][u] = row[C_RF][l];
                    a[2][u] = row[C_G1][l]; a[3][u] = row[C_G2][l]; a[4][u] = row[C_G3][l];
                }
                if constexpr (TORQUES) { a[T0][u] = row[C_TN][l]; a[T0 + 1][u] = row[C_RN][l]; a[T0 + 2][u] = row[C_GL][l]; }
            }
#pragma unroll
            for (int u = 0; u < FOLD_BATCH; ++u)
#pragma unroll
                for (int i = 0; i < N; ++i) sum[i] = sum[i] + a[i][u];
        }
        if constexpr (FORCES) {
            const double inv_hm = lds.of_system(B, K_INV_HM);
            double a = 0. + -1.0 * inv_hm * sum[0];
            a = a + -1.0 * inv_hm * sum[1];
            double g = -1.0 * sum[2];
            g = g + -1.0 * sum[3];
            g = g + -1.0 * sum[4];
            row[C_TF][hl] = a + g;
        }
        if constexpr (TORQUES) row[C_TN][hl] = (sum[T0] + sum[T0 + 1]) + sum[T0 + 2];
    });
}

// a / b < DBL_EPS_2 for a, b >= 0 (or NaN): DBL_EPS_2 is a power of two and
// its predecessor is closer than half an ulp of the quotient can reach, so the
// rounded quotient is below it exactly when a < b DBL_EPS_2, barring underflow
// of the product, where the quotient decides.
__device__ __forceinline__ bool below_eps2(double a, double b) {
    const double limit = b * DBL_EPS_2;
    if (!(limit >= 1e-290)) return a / b < DBL_EPS_2;
    return a < limit;
}

// whfast.rs:424-451 for this lane's group: four sums over the bodies in body
// order, which every lane of the team forms itself.
template <class Rows>
__device__ __forceinline__ bool solve_converged(const Rows &cv, const FixedLane &B) {
    double sum[4] = {0., 0., 0., 0.};
    auto add = [&](auto lane_of) {
        for (int j0 = 0; j0 < B.nmax; j0 += FOLD_BATCH) {
            double a[4][FOLD_BATCH];
#pragma unroll
            for (int u = 0; u < FOLD_BATCH; ++u) {
                const int l = j0 + u < B.n ? lane_of(j0 + u) : WAVE;
#pragma unroll
                for (int i = 0; i < 4; ++i) a[i][u] = cv[i][l];
            }
#pragma unroll
            for (int u = 0; u < FOLD_BATCH; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) sum[i] = sum[i] + a[i][u];
        }
    };
    if (B.hosts_first) add([&](int j) { return B.gbase + j; });
    else add([&](int j) { return lane_of_body(B, j); });
    return below_eps2(sum[0], sum[1]) && below_eps2(sum[2], sum[3]);
}

// ===========================================================================
// Pair terms
// ===========================================================================
// Orbiting lanes only.  Every lane's position and the spins of the previous
// evaluation are visible.
template <int M, int ROLE, class Lds>
__device__ __forceinline__ void fixed_geometry(const DevEnsemble &E, Lds &lds, const FixedLane &B, FixedGeo &g) {
    using W = Role<M, ROLE>;
    const int lane = B.lane, hl = B.hl();
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        if constexpr (M == 1) g.px[q] = B.x[q] - lds.xb[q][hl];
        else g.px[q] = (W::OWN_V ? B.x[q] : lds.team.x[q][lane]) - lds.team.x[q][hl];
    }
    const double d = sqrt(p2(g.px[0]) + p2(g.px[1]) + p2(g.px[2]));
    g.Rd = rcp(d);
    const double m = B.m, hm = lds.m[hl];
    if constexpr (W::TIDES || W::FLAT) {
        const double(*so)[WAVE];
        if constexpr (M == 1) so = lds.s;
        else so = lds.team.so;
        g.rs_star = g.px[0] * so[0][hl] + g.px[1] * so[1][hl] + g.px[2] * so[2][hl];
        g.rs_planet = g.px[0] * so[0][lane] + g.px[1] * so[1][lane] + g.px[2] * so[2][lane];
        const Rcp Rd7 = rcp(p7(d));
        if constexpr (W::TIDES) {
            const double hR = lds.R[hl], R = lds.R[lane];
            const int hb = B.body - B.idx + B.hidx;
            const double sigma_host = E.sigma[hb], sigma_pair = E.sigma[B.body];
            const double hm2 = hm * hm;
            const double pm2 = m * m;
            g.Rp8 = rcp(p8(d));
            g.os = divr(4.5 * p2(m) * p10(hR) * sigma_host, Rd7);
            g.op = divr(4.5 * p2(hm) * p10(R) * sigma_pair, Rd7);
            g.conservative = divr(-3.0 * K2, Rd7) * (pm2 * p5(hR) * E.k2[hb] + hm2 * p5(R) * E.k2[B.body]);
            g.term1 = pm2 * p10(hR) * sigma_host;
            g.term2 = hm2 * p10(R) * sigma_pair;
            g.od = divr(g.os, g.Rd);
            g.pd = divr(g.op, g.Rd);
            g.id = divr(1.0, g.Rd);
        }
        if constexpr (W::FLAT) {
            g.d5 = p5(d);
            g.m3d5 = -3. / g.d5;
            g.c15 = divr(15., Rd7);
        }
    }
    if constexpr (W::ORBIT) {
        const double hmg = hm * K2, pmg = m * K2;
        const double f = lds.konst(B, K_F);
        const double mg = hmg + pmg;
        const double distance_2 = p2(d);
        const Rcp Rdc = rcp(distance_2 * SPEED_OF_LIGHT_2);
        g.mgc = divr(-mg, Rdc);
        g.mg_d = divr(mg, g.Rd);
        g.c1pn = divr(2.0 * (2.0 + f) * mg, g.Rd);
        g.o1pn = divr(mg, Rdc) * 2.0 * (2.0 - f);
        g.c2pn = 3.0 / 4.0 * (12.0 + 29.0 * f) * (p2(mg) / distance_2);
    }
    if constexpr (W::SPIN_ORBIT) {
#pragma unroll
        for (int q = 0; q < 3; ++q) g.n3[q] = divr(g.px[q], g.Rd);
    }
}

// Tides: force and torques (constant_time_lag.rs:171-332, tides/common.rs:223-261).
template <class Lds>
__device__ __forceinline__ void pair_tides(Lds &lds, const FixedLane &B, const FixedGeo &g, const double pv[3], double vr,
                                           const double hs[3], const double s[3], double a[3], double torque[3]) {
    const int lane = B.lane;
    const double *px = g.px;
    const double d = g.Rd.b;
    const double factor1 = divr(-13.5 * vr, g.Rp8);
    const double diss_pm = factor1 * g.term2;
    const double dissipative = diss_pm + factor1 * g.term1;
    const double radial = g.conservative + dissipative;
    const double factor3 = radial + divr((g.os + g.op) * vr, g.Rd);
    const double F0 = divr(factor3 * px[0], g.Rd) + g.od * (hs[1] * px[2] - hs[2] * px[1] - pv[0])
                    + g.pd * (s[1] * px[2] - s[2] * px[1] - pv[0]);
    const double F1 = divr(factor3 * px[1], g.Rd) + g.od * (hs[2] * px[0] - hs[0] * px[2] - pv[1])
                    + g.pd * (s[2] * px[0] - s[0] * px[2] - pv[1]);
    const double F2 = divr(factor3 * px[2], g.Rd) + g.od * (hs[0] * px[1] - hs[1] * px[0] - pv[2])
                    + g.pd * (s[0] * px[1] - s[1] * px[0] - pv[2]);
    put3(lds, C_TF, lane, F0, F1, F2);
    a[0] = 0. + B.inv_m * F0;
    a[1] = 0. + B.inv_m * F1;
    a[2] = 0. + B.inv_m * F2;
    const double cx = px[1] * pv[2] - px[2] * pv[1];
    const double cy = px[2] * pv[0] - px[0] * pv[2];
    const double cz = px[0] * pv[1] - px[1] * pv[0];
    put3(lds, C_TN, lane,
         -1.0 * (g.os * (d * hs[0] - divr(g.rs_star * px[0], g.Rd) - g.id * cx)),
         -1.0 * (g.os * (d * hs[1] - divr(g.rs_star * px[1], g.Rd) - g.id * cy)),
         -1.0 * (g.os * (d * hs[2] - divr(g.rs_star * px[2], g.Rd) - g.id * cz)));
    torque[0] = -1.0 * (g.op * (d * s[0] - divr(g.rs_planet * px[0], g.Rd) - g.id * cx));
    torque[1] = -1.0 * (g.op * (d * s[1] - divr(g.rs_planet * px[1], g.Rd) - g.id * cy));
    torque[2] = -1.0 * (g.op * (d * s[2] - divr(g.rs_planet * px[2], g.Rd) - g.id * cz));
}

// Flattening: force and torques (oblate_spheroid.rs:21-97,
// rotational_flattening/common.rs:165-201); a is inv_m F.
template <class Lds>
__device__ __forceinline__ void pair_flattening(Lds &lds, const FixedLane &B, const FixedGeo &g, const double hs[3],
                                                const double s[3], double a[3], double torque[3]) {
    const int lane = B.lane, hl = B.hl();
    const double *px = g.px;
    const double m = B.m, hm = lds.m[hl];
    const double hs2 = p2(hs[0]) + p2(hs[1]) + p2(hs[2]), s2 = p2(s[0]) + p2(s[1]) + p2(s[2]);
    constexpr Rcp R6{6., 1. / 6.};
    const double fs = divr(m * lds.k2f[hl] * hs2 * p5(lds.R[hl]), R6);
    const double ofs = -6. * fs * g.rs_star / (hs2 * g.d5);
    const double fp = divr(hm * lds.k2f[lane] * s2 * p5(lds.R[lane]), R6);
    const double ofp = -6. * fp * g.rs_planet / (s2 * g.d5);
    const double radial = g.m3d5 * (fp + fs) + g.c15 * (fs * g.rs_star * g.rs_star / hs2 + fp * g.rs_planet * g.rs_planet / s2);
    const double F0 = radial * px[0] + ofp * s[0] + ofs * hs[0];
    const double F1 = radial * px[1] + ofp * s[1] + ofs * hs[1];
    const double F2 = radial * px[2] + ofp * s[2] + ofs * hs[2];
    put3(lds, C_RF, lane, F0, F1, F2);
    a[0] = B.inv_m * F0;
    a[1] = B.inv_m * F1;
    a[2] = B.inv_m * F2;
    put3(lds, C_RN, lane,
         -1.0 * (ofs * (px[1] * hs[2] - px[2] * hs[1])),
         -1.0 * (ofs * (px[2] * hs[0] - px[0] * hs[2])),
         -1.0 * (ofs * (px[0] * hs[1] - px[1] * hs[0])));
    torque[0] = -1.0 * (ofp * (px[1] * s[2] - px[2] * s[1]));
    torque[1] = -1.0 * (ofp * (px[2] * s[0] - px[0] * s[2]));
    torque[2] = -1.0 * (ofp * (px[0] * s[1] - px[1] * s[0]));
}

// Kidder 1995 first and second order (general_relativity.rs:177-298); gr is
// their sum.
template <class Lds>
__device__ __forceinline__ void pair_gr_orbit(Lds &lds, const FixedLane &B, const FixedGeo &g, const double pv[3], double vr,
                                              double gr[3]) {
    const int lane = B.lane;
    const double *px = g.px;
    const double nv2 = p2(pv[0]) + p2(pv[1]) + p2(pv[2]);
    const double nv = sqrt(nv2);
    const double f = lds.konst(B, K_F), m_over_hm = lds.konst(B, K_M_OVER_HM);
    const Rcp Rnv = rcp(nv);
    {   // 1PN
        const double radial_velocity_2 = p2(vr);
        const double radial = g.mgc * ((1.0 + 3.0 * f) * nv2 - g.c1pn - 1.5 * f * radial_velocity_2);
        const double orthogonal = g.o1pn * vr * nv;
#pragma unroll
        for (int q = 0; q < 3; ++q) gr[q] = divr(radial * px[q], g.Rd) + divr(orthogonal * pv[q], Rnv);
        put3(lds, C_G1, lane, m_over_hm * gr[0], m_over_hm * gr[1], m_over_hm * gr[2]);
    }
    {   // 2PN
        const double nv4 = p2(nv2);
        const double vr2 = p2(vr);
        const double vr4 = p2(vr2);
        const double f2 = p2(f);
        const double radial = g.mgc
            * (g.c2pn
               + f * (3.0 - 4.0 * f) * nv4
               + 15.0 / 8.0 * f * (1.0 - 3.0 * f) * vr4
               - 3.0 / 2.0 * f * (3.0 - 4.0 * f) * vr2 * nv2
               - 0.5 * f * (13.0 - 4.0 * f) * g.mg_d * nv2
               - (2.0 + 25.0 * f + 2.0 * f2) * g.mg_d * vr2);
        const double orthogonal = g.mgc * (-0.5) * vr
            * (f * (15.0 + 4.0 * f) * nv2
               - (4.0 + 41.0 * f + 8.0 * f2) * g.mg_d
               - 3.0 * f * (3.0 + 2.0 * f) * vr2);
        double a[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            a[q] = divr(radial * px[q], g.Rd) + orthogonal * pv[q];
            gr[q] = gr[q] + a[q];
        }
        put3(lds, C_G2, lane, m_over_hm * a[0], m_over_hm * a[1], m_over_hm * a[2]);
    }
}

// Kidder 1995 spin-orbit terms (general_relativity.rs:300-456): acceleration a,
// this body's spin derivative gL.
template <class Lds>
__device__ __forceinline__ void pair_gr_spin(Lds &lds, const FixedLane &B, const FixedGeo &g, const double pv[3], double vr,
                                             const double hs[3], const double s[3], double a[3], double gL[3]) {
    const int lane = B.lane, hl = B.hl();
    const double *px = g.px, *n3 = g.n3;
    const Rcp Rhm{lds.m[hl], lds.of_system(B, K_INV_HM)};
    const Rcp Rm{B.m, B.inv_m};
    const double hI = lds.I[hl], I = lds.I[lane];
    const double m_over_hm = lds.konst(B, K_M_OVER_HM), mfM = lds.konst(B, K_MFM), mr = lds.konst(B, K_MR);
    const double fm_body = lds.konst(B, K_FM_BODY);
    const double Ls[3] = {hI * hs[0], hI * hs[1], hI * hs[2]};
    const double Lp[3] = {I * s[0], I * s[1], I * s[2]};
    const double factor_a = G / SPEED_OF_LIGHT_2;
    {
        double msf[3], e7[3], e3s[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            msf[q] = mfM * (divr(Lp[q], Rm) - divr(Ls[q], Rhm));
            e7[q] = 7. * (Ls[q] + Lp[q]) + 3. * msf[q];
            e3s[q] = 3. * (Ls[q] + Lp[q]) + msf[q];
        }
        const double e10 = 6. * n3[0] * ((n3[1] * pv[2] - n3[2] * pv[1]) * (2. * (Ls[0] + Lp[0]) + msf[0]));
        const double e11 = 6. * n3[1] * ((n3[2] * pv[0] - n3[0] * pv[2]) * (2. * (Ls[1] + Lp[1]) + msf[1]));
        const double e12 = 6. * n3[2] * ((n3[0] * pv[1] - n3[1] * pv[0]) * (2. * (Ls[2] + Lp[2]) + msf[2]));
        a[0] = factor_a * (e10 - (pv[1] * e7[2] - pv[2] * e7[1]) + 3. * vr * (n3[1] * e3s[2] - n3[2] * e3s[1]));
        a[1] = factor_a * (e11 - (pv[2] * e7[0] - pv[0] * e7[2]) + 3. * vr * (n3[2] * e3s[0] - n3[0] * e3s[2]));
        a[2] = factor_a * (e12 - (pv[0] * e7[1] - pv[1] * e7[0]) + 3. * vr * (n3[0] * e3s[1] - n3[1] * e3s[0]));
    }
    put3(lds, C_G3, lane, m_over_hm * a[0], m_over_hm * a[1], m_over_hm * a[2]);
    const double Lo[3] = {mr * (px[1] * pv[2] - px[2] * pv[1]), mr * (px[2] * pv[0] - px[0] * pv[2]),
                          mr * (px[0] * pv[1] - px[1] * pv[0])};
    const double sh = n3[0] * Ls[0] + n3[1] * Ls[1] + n3[2] * Ls[2];
    gL[0] = factor_a * (fm_body * (Lo[1] * Lp[2] - Lo[2] * Lp[1]) - (Ls[1] * Lp[2] - Ls[2] * Lp[1]) + 3. * sh * (n3[1] * Lp[2] - n3[2] * Lp[1]));
    gL[1] = factor_a * (fm_body * (Lo[2] * Lp[0] - Lo[0] * Lp[2]) - (Ls[2] * Lp[0] - Ls[0] * Lp[2]) + 3. * sh * (n3[2] * Lp[0] - n3[0] * Lp[2]));
    gL[2] = factor_a * (fm_body * (Lo[0] * Lp[1] - Lo[1] * Lp[0]) - (Ls[0] * Lp[1] - Ls[1] * Lp[0]) + 3. * sh * (n3[0] * Lp[1] - n3[1] * Lp[0]));
}

// The host's spin derivative from this body (general_relativity.rs:300-456).
template <class Lds>
__device__ __forceinline__ void pair_gr_host(Lds &lds, const FixedLane &B, const FixedGeo &g, const double pv[3],
                                             const double hs[3], const double s[3]) {
    const int lane = B.lane, hl = B.hl();
    const double *px = g.px, *n3 = g.n3;
    const double hI = lds.I[hl], I = lds.I[lane];
    const double mr = lds.konst(B, K_MR), fm_host = lds.konst(B, K_FM_HOST);
    const double Ls[3] = {hI * hs[0], hI * hs[1], hI * hs[2]};
    const double Lp[3] = {I * s[0], I * s[1], I * s[2]};
    const double factor_a = G / SPEED_OF_LIGHT_2;
    const double Lo[3] = {mr * (px[1] * pv[2] - px[2] * pv[1]), mr * (px[2] * pv[0] - px[0] * pv[2]),
                          mr * (px[0] * pv[1] - px[1] * pv[0])};
    const double sp = n3[0] * Lp[0] + n3[1] * Lp[1] + n3[2] * Lp[2];
    put3(lds, C_GL, lane,
             factor_a * (fm_host * (Lo[1] * Ls[2] - Lo[2] * Ls[1]) - (Lp[1] * Ls[2] - Lp[2] * Ls[1]) + 3. * sp * (n3[1] * Ls[2] - n3[2] * Ls[1])),
             factor_a * (fm_host * (Lo[2] * Ls[0] - Lo[0] * Ls[2]) - (Lp[2] * Ls[0] - Lp[0] * Ls[2]) + 3. * sp * (n3[2] * Ls[0] - n3[0] * Ls[2])),
             factor_a * (fm_host * (Lo[0] * Ls[1] - Lo[1] * Ls[0]) - (Lp[0] * Ls[1] - Lp[1] * Ls[0]) + 3. * sp * (n3[0] * Ls[1] - n3[1] * Ls[0])));
}

__device__ __forceinline__ void put_rows(double (*rows)[WAVE], int lane, const double a[3]) {
#pragma unroll
    for (int q = 0; q < 3; ++q) rows[q][lane] = a[q];
}

// spin = L / I of this body (particles/common.rs:3-14), published; unchanged
// when I is 0, which is raised as a status at the end of the kick.
template <int M, class Lds>
__device__ __forceinline__ void publish_spin(Lds &lds, FixedLane &B) {
    const Rcp RI{M == 1 ? lds.I[B.lane] : B.I, B.inv_I};
    if constexpr (M == 1) {
        if (RI.b == 0.) return;
#pragma unroll
        for (int q = 0; q < 3; ++q) lds.s[q][B.lane] = divr(B.L[q], RI);
    } else {
        if (RI.b != 0.) {
#pragma unroll
            for (int q = 0; q < 3; ++q) B.s[q] = divr(B.L[q], RI);
        }
        put_rows(lds.s, B.lane, B.s);
    }
}
template <class Lds>
__device__ __forceinline__ void publish_velocity(Lds &lds, const FixedLane &B) {
#pragma unroll
    for (int q = 0; q < 3; ++q) lds.vel(q, B.lane) = B.v[q];
}

// ===========================================================================
// The implicit-midpoint solve (whfast.rs:322-466).  On entry the velocities
// and spins of the first evaluation are published and visible to the team.
// act: this lane's system takes the step; uniform over a group and alike in
// every wavefront.  All wavefronts of a team pass the same barriers: the loop
// ends when no group iterates any more, which each decides from the same sums.
// ===========================================================================
template <int M, int ROLE, class Lds>
__device__ __forceinline__ void fixed_kick(Lds &lds, FixedLane &B, FixedGeo &g, bool act) {
    using W = Role<M, ROLE>;
    const double h = 0.5 * B.dt;
    const int lane = B.lane, hl = B.hl();
    double v_orig[3], dv[3], L_orig[3], dL[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        dv[q] = dL[q] = 0.;
        if (W::OWN_V) v_orig[q] = B.v[q];
        if (W::OWN_L) L_orig[q] = B.L[q];
    }
    bool run = act, converged = false;
    for (int it = 0;; ++it) {
        double a_add[3] = {0., 0., 0.}, dLdt[3] = {0., 0., 0.};
        if (run && B.orb) {
            double pv[3], hs[3], s[3], vr = 0.;
            if (W::TIDES || W::ORBIT || W::SPIN_ORBIT) {
#pragma unroll
                for (int q = 0; q < 3; ++q) pv[q] = (W::OWN_V ? B.v[q] : lds.vel(q, lane)) - lds.vel(q, hl);
            }
            if (W::TIDES || W::ORBIT || W::SPIN_ORBIT) {
                vr = divr(g.px[0] * pv[0] + g.px[1] * pv[1] + g.px[2] * pv[2], g.Rd);
            }
            if (W::TIDES || W::FLAT || W::SPIN_ORBIT) {
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    hs[q] = lds.s[q][hl];
                    s[q] = W::OWN_L && M > 1 ? B.s[q] : lds.s[q][lane];
                }
            }
            double t[3], r[3], a[3], tr[3], rr[3];
            if constexpr (W::TIDES) pair_tides(lds, B, g, pv, vr, hs, s, t, tr);
            if constexpr (W::FLAT) pair_flattening(lds, B, g, hs, s, r, rr);
            if constexpr (W::SPIN_ORBIT) pair_gr_host(lds, B, g, pv, hs, s);
            if constexpr (W::ORBIT) pair_gr_orbit(lds, B, g, pv, vr, a);
            if constexpr (W::SPIN_ORBIT) {
                double so[3];
                pair_gr_spin(lds, B, g, pv, vr, hs, s, so, dLdt);
                if constexpr (M == 4) put_rows(&lds.team.ex[EX_GR_SO], lane, so);
                else {
#pragma unroll
                    for (int q = 0; q < 3; ++q) a[q] = a[q] + so[q];
                }
            }
            if constexpr (M == 1) {
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    a_add[q] = (t[q] + r[q]) + a[q];
                    dLdt[q] = (tr[q] + rr[q]) + dLdt[q];
                }
            } else if constexpr (M == 2) {
                if constexpr (W::OWN_V) {
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        a_add[q] = t[q] + r[q];
                        lds.team.ex[EX_TORQUE_T + q][lane] = tr[q] + rr[q];
                    }
                } else {
                    put_rows(&lds.team.ex[EX_GR], lane, a);
                }
            } else {
                if constexpr (W::TIDES) {
                    put_rows(&lds.team.ex[EX_TORQUE_T], lane, tr);
#pragma unroll
                    for (int q = 0; q < 3; ++q) a_add[q] = t[q];
                }
                if constexpr (W::FLAT) { put_rows(&lds.team.ex[EX_ACC_R], lane, r); put_rows(&lds.team.ex[EX_TORQUE_R], lane, rr); }
                if constexpr (W::ORBIT) put_rows(&lds.team.ex[EX_GR], lane, a);
            }
            if constexpr (W::TIDES || W::FLAT) {   // for the next evaluation, whose spins are refreshed before it reads them
                g.rs_star = g.px[0] * hs[0] + g.px[1] * hs[1] + g.px[2] * hs[2];
                g.rs_planet = g.px[0] * s[0] + g.px[1] * s[1] + g.px[2] * s[2];
            }
        }
        team_sync<M>();
        double got[3];   // this body's acceleration or spin derivative, with the other wavefronts' parts
        if constexpr (W::OWN_V) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                if constexpr (M == 1) got[q] = a_add[q];
                else if constexpr (M == 2) got[q] = a_add[q] + lds.team.ex[EX_GR + q][lane];
                else got[q] = (a_add[q] + lds.team.ex[EX_ACC_R + q][lane]) + (lds.team.ex[EX_GR + q][lane] + lds.team.ex[EX_GR_SO + q][lane]);
            }
        } else if constexpr (W::OWN_L) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                if constexpr (M == 2) got[q] = lds.team.ex[EX_TORQUE_T + q][lane] + dLdt[q];
                else got[q] = (lds.team.ex[EX_TORQUE_T + q][lane] + lds.team.ex[EX_TORQUE_R + q][lane]) + dLdt[q];
            }
        }
        if (run) {
            if constexpr (W::OWN_V || W::OWN_L) host_reactions<W::OWN_V, W::OWN_L>(lds, B);
        }
        if constexpr (W::OWN_V || W::OWN_L) wsync();
        const bool check = it >= MIDPOINT_MIN_ITER - 1;
        if (run) {
            if constexpr (W::OWN_V) {
                double pdv = 0., fv2 = 0.;   // |change of the final velocity|^2, |final velocity|^2
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const double ah = lds.xb[C_TF + q][lane];
                    const double a = B.host_lane ? ah : got[q];
                    const double v_prev = v_orig[q] + dv[q];   // it >= 2 where it is used
                    dv[q] = h * a - B.ev[q];
                    const double vf = v_orig[q] + dv[q];
                    pdv = pdv + p2(vf - v_prev);
                    fv2 = fv2 + p2(vf);
                    B.v[q] = 0.5 * (v_orig[q] + vf);
                }
                if (check) {
                    if constexpr (M == 1) { lds.xb[0][lane] = pdv; lds.xb[1][lane] = fv2; }
                    else { lds.team.cv[0][lane] = pdv; lds.team.cv[1][lane] = fv2; }
                } else publish_velocity(lds, B);
            }
            if constexpr (W::OWN_L) {
                double pdL = 0., fL2 = 0.;
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const double ah = lds.xb[C_TN + q][lane];
                    const double a = B.host_lane ? ah : M == 1 ? dLdt[q] : got[q];
                    const double L_prev = L_orig[q] + dL[q];
                    dL[q] = h * (a + 0.) - B.eL[q];   // + 0.: no wind (universe.rs:603-614)
                    const double Lf = L_orig[q] + dL[q];
                    pdL = pdL + p2(Lf - L_prev);
                    fL2 = fL2 + p2(Lf);
                    B.L[q] = 0.5 * (L_orig[q] + Lf);
                }
                if (check) {
                    if constexpr (M == 1) { lds.xb[2][lane] = pdL; lds.xb[3][lane] = fL2; }
                    else { lds.team.cv[2][lane] = pdL; lds.team.cv[3][lane] = fL2; }
                } else publish_spin<M>(lds, B);
            }
        }
        team_sync<M>();
        if (!check) continue;
        if (run) {
            if constexpr (M == 1) converged = solve_converged(lds.xb, B);
            else converged = solve_converged(lds.team.cv, B);
            if (converged || it == MIDPOINT_MAX_ITER - 1) run = false;
        }
        if (!__any(run)) break;
        if constexpr (M == 1) wsync();
        if (run) {
            if constexpr (W::OWN_V) publish_velocity(lds, B);
            if constexpr (W::OWN_L) publish_spin<M>(lds, B);
        }
        team_sync<M>();
    }
    if (act) {
        if (W::OWN_V && !converged) B.status |= POS_STATUS_MIDPOINT_NOT_CONVERGED;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            if constexpr (W::OWN_V) {
                B.v[q] = v_orig[q] + dv[q];
                B.ev[q] = (B.v[q] - v_orig[q]) - dv[q];
            }
            if constexpr (W::OWN_L) {
                B.L[q] = L_orig[q] + dL[q];
                B.eL[q] = (B.L[q] - L_orig[q]) - dL[q];
            }
        }
    }
}

// ===========================================================================
// The drift (wave 0 alone): transforms, Kepler, jump, gravity
// ===========================================================================
// universe.rs:198-303 with every position in rows 0-2; leaves the acceleration
// in acc.  The pairs of a batch are independent, so their square roots and
// divisions overlap; they are added in body order.  The checks of a pair
// (Roche, collision, ejection) fire rarely: a pair no farther apart than near2
// (the largest squared distance one of this body's pairs fires at) or farther
// than far2 (the host's ejection limit) raises a flag, and then all are
// evaluated as the reference does.
template <bool JACOBI, int BATCH, class Lds>
__device__ __forceinline__ void fixed_gravity(const DevEnsemble &E, Lds &lds, FixedLane &B, double acc[3]) {
    acc[0] = acc[1] = acc[2] = 0.;
    bool flagged = false;
    auto separation = [&](int l, double &dx, double &dy, double &dz) {
        dx = B.x[0] - lds.xb[0][l];
        dy = B.x[1] - lds.xb[1][l];
        dz = B.x[2] - lds.xb[2][l];
        return dx * dx + dy * dy + dz * dz;
    };
    // heliocentric splittings leave out every pair with the host, Jacobi the
    // one of the host and the first body after it
    for (int j0 = JACOBI ? 0 : 1; j0 < B.nmax; j0 += BATCH) {
        double t[BATCH][3];
        bool use[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; ++u) {
            const int j = j0 + u;   // Jacobi: body index, else place in the chain
            const int l = j < B.n ? (JACOBI ? lane_of_body(B, j) : B.gbase + j) : B.lane;
            const bool pair = l != B.lane;
            double dx, dy, dz;
            const double distance_2 = separation(l, dx, dy, dz);
            flagged = flagged || (pair && (distance_2 <= B.near2 || distance_2 > B.far2));
            use[u] = JACOBI ? pair && l - B.gbase + B.k != 1 : pair && B.k != 0;
            const double distance = sqrt(distance_2);
            const double prefact = -G / (distance * distance * distance) * lds.m[l];
            t[u][0] = prefact * dx; t[u][1] = prefact * dy; t[u][2] = prefact * dz;
        }
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
            if (use[u]) {
#pragma unroll
                for (int q = 0; q < 3; ++q) acc[q] = acc[q] + t[u][q];
            }
    }
    if (!JACOBI && !B.hosts_first) {   // a body before the host makes the checks of their pair
        double dx, dy, dz;
        if (B.idx < B.hidx) flagged = flagged || separation(B.gbase, dx, dy, dz) <= B.near2;
    }
    if (!__any(flagged)) return;
    const double Ri = lds.R[B.lane];
    for (int j = B.idx + 1; flagged && j < B.n; ++j) {
        const int l = lane_of_body(B, j);
        double dx, dy, dz;
        const double distance_2 = separation(l, dx, dy, dz);
        const double rr = E.roche[(size_t)B.body * POS_MAX_BODIES + j];
        if (distance_2 <= rr * rr) B.status |= POS_STATUS_ROCHE;
        if (distance_2 <= p2(Ri + lds.R[l])) B.status |= POS_STATUS_COLLISION;
        if (B.host_lane && distance_2 > MAX_DISTANCE_2) B.status |= POS_STATUS_EJECTION;
    }
}

// Democratic heliocentric and WHDS drift (whfast.rs:495-625, 973-1155).  Each body
// forms its own term of every sum (a quotient by a mass included) before the
// terms are exchanged, so a sum is only its additions.
template <bool DIRECT, bool REC, bool WHDS, class Lds>
__device__ __forceinline__ void drift_heliocentric(const DevEnsemble &E, Lds &lds, FixedLane &B, double acc[3], const TapeRef &T,
                                                   int row) {
    const int lane = B.lane, hl = B.hl();
    const double half_dt = 0.5 * B.dt;
    const Rcp Rm0{lds.m[hl], lds.of_system(B, K_INV_HM)};
    const Rcp Rmt{lds.of_system(B, K_TOTAL), lds.of_system(B, K_INV_TOTAL)};
    // WHDS: the mass of the pair with the host, the velocities' factor (whfast.rs:973-1023)
    const Rcp Rpair = rcp(WHDS ? Rm0.b + B.m : 1.);
    const double factor = WHDS ? divr(Rpair.b, Rm0) : 1.;
    // centre of mass, the host first
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        lds.xb[q][lane] = B.x[q] * B.m;
        lds.xb[3 + q][lane] = B.v[q] * B.m;
        lds.xb[6 + q][lane] = B.x[q];
    }
    wsync();
    {
        double init[2][3], com[2][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) { init[0][q] = 0. + lds.xb[q][hl]; init[1][q] = 0. + lds.xb[3 + q][hl]; }
        group_sums<2, false, DIRECT>(lds, B, init, com);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            B.comx[q] = divr(com[0][q], Rmt);
            B.comv[q] = divr(com[1][q], Rmt);
            B.ax[q] = B.x[q] - lds.xb[6 + q][hl];
            B.av[q] = B.v[q] - B.comv[q];
            if constexpr (WHDS) B.av[q] = B.av[q] * factor;
        }
        wsync();
    }
    auto drift = [&](int field) {
        if (B.orb) kepler_individual_step(B, WHDS ? mg_of(lds, hl) + mg_of(lds, lane) : mg_of(lds, hl), half_dt);
#pragma unroll
        for (int q = 0; q < 3; ++q) B.comx[q] = B.comx[q] + half_dt * B.comv[q];
        if (REC) *T.at(row, field, B.body) = B.orb ? B.kx : 0.;
    };
    auto jump = [&] {
        const double zero[1][3] = {{0., 0., 0.}};
        double p[1][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) lds.xb[q][lane] = WHDS ? divr(B.m * B.av[q], Rpair) : B.m * B.av[q];
        wsync();
        group_sums<1, false, DIRECT>(lds, B, zero, p);
        wsync();
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            if constexpr (WHDS) B.ax[q] = B.ax[q] + half_dt * (p[0][q] - divr(B.m * B.av[q], Rpair));
            else B.ax[q] = B.ax[q] + divr(half_dt * p[0][q], Rm0);
        }
    };
    drift(TP_XK1);
    jump();
    {   // positions for the gravity
        const double init[1][3] = {{B.comx[0], B.comx[1], B.comx[2]}};
        double h[1][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) lds.xb[q][lane] = divr(B.ax[q] * B.m, Rmt);
        wsync();
        group_sums<1, true, DIRECT>(lds, B, init, h);
        wsync();
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            B.x[q] = B.host_lane ? h[0][q] : B.ax[q] + h[0][q];
            lds.xb[q][lane] = B.x[q];
        }
        wsync();
    }
    fixed_gravity<false, DIRECT ? 4 : 2>(E, lds, B, acc);
    wsync();
#pragma unroll
    for (int q = 0; q < 3; ++q) B.av[q] = B.av[q] + (WHDS ? divr(B.dt * Rpair.b * acc[q], Rm0) : B.dt * acc[q]);
    jump();
    drift(TP_XK2);
    {
        const double init[2][3] = {{B.comx[0], B.comx[1], B.comx[2]}, {B.comv[0], B.comv[1], B.comv[2]}};
        double h[2][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            lds.xb[q][lane] = divr(B.ax[q] * B.m, Rmt);
            lds.xb[3 + q][lane] = B.av[q] * (WHDS ? divr(B.m, Rpair) : lds.konst(B, K_M_OVER_HM));
        }
        wsync();
        group_sums<2, true, DIRECT>(lds, B, init, h);
        wsync();
        const Rcp Rfactor = rcp(factor);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            B.x[q] = B.host_lane ? h[0][q] : B.ax[q] + h[0][q];
            B.v[q] = B.host_lane ? h[1][q] : (WHDS ? divr(B.av[q], Rfactor) : B.av[q]) + B.comv[q];
        }
    }
}

// Jacobi drift (whfast.rs:495-625, 881-1080): prefix recurrences along the
// chain, formed by every lane; their mass ratios are the launch's constants.
template <bool DIRECT, bool REC, class Lds>
__device__ __forceinline__ void drift_jacobi(const DevEnsemble &E, Lds &lds, FixedLane &B, double acc[3], const TapeRef &T,
                                             int row) {
    const int lane = B.lane, hl = B.hl();
    const double half_dt = 0.5 * B.dt;
    const Rcp Rmt{lds.of_system(B, K_TOTAL), lds.of_system(B, K_INV_TOTAL)};
    // T vectors of rows [0, 3T): own value relative to the bodies before it in
    // the chain, and the last running sums
    auto forward = [&](auto &own, auto &sum) {
        constexpr int N = sizeof(own) / sizeof(double);
        double eta = lds.m[hl];
#pragma unroll
        for (int q = 0; q < N; ++q) { sum[q] = eta * lds.xb[q][hl]; own[q] = 0.; }
        for (int j = 1; j < B.n; ++j) {
            const int l = B.gbase + j;
            const double mj = lds.m[l], ei = lds.chain.ei[l];
            eta = eta + mj;
            const double pme = eta * ei;
#pragma unroll
            for (int q = 0; q < N; ++q) {
                const double a = lds.xb[q][l] - sum[q] * ei;
                if (j == B.k) own[q] = a;
                sum[q] = sum[q] * pme + mj * a;
            }
        }
    };
    // the reverse recurrence of rows [0, 3T) from the centre of mass: own value
    auto reverse = [&](auto &own, const auto &com) {
        constexpr int N = sizeof(own) / sizeof(double);
        double sum[N], eta = Rmt.b;
#pragma unroll
        for (int q = 0; q < N; ++q) { sum[q] = eta * com[q]; own[q] = 0.; }
        for (int j = B.n - 1; j >= 1; --j) {
            const int l = B.gbase + j;
            const double mj = lds.m[l], ei = lds.chain.rei[l];
#pragma unroll
            for (int q = 0; q < N; ++q) {
                const double aj = lds.xb[q][l];
                sum[q] = (sum[q] - mj * aj) * ei;
                const double a = aj + sum[q];
                if (j == B.k) own[q] = a;
            }
            eta = eta - mj;
#pragma unroll
            for (int q = 0; q < N; ++q) sum[q] = sum[q] * eta;
        }
        const double inv_left = lds.of_system(B, K_INV_LEFT);
#pragma unroll
        for (int q = 0; q < N; ++q)
            if (B.host_lane) own[q] = sum[q] * inv_left;
    };
    auto drift = [&](int field) {
        if (B.orb) kepler_individual_step(B, B.mu, half_dt);
#pragma unroll
        for (int q = 0; q < 3; ++q) B.comx[q] = B.comx[q] + half_dt * B.comv[q];
        if (REC) *T.at(row, field, B.body) = B.orb ? B.kx : 0.;
    };
#pragma unroll
    for (int q = 0; q < 3; ++q) { lds.xb[q][lane] = B.x[q]; lds.xb[3 + q][lane] = B.v[q]; }
    wsync();
    {
        double own[6], sum[6];
        forward(own, sum);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            if (B.orb) { B.ax[q] = own[q]; B.av[q] = own[3 + q]; }
            B.comx[q] = sum[q] * Rmt.r;
            B.comv[q] = sum[3 + q] * Rmt.r;
        }
        wsync();
    }
    drift(TP_XK1);
    {   // positions for the gravity
        double own[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) lds.xb[q][lane] = B.ax[q];
        wsync();
        reverse(own, B.comx);
        wsync();
#pragma unroll
        for (int q = 0; q < 3; ++q) { B.x[q] = own[q]; lds.xb[q][lane] = own[q]; }
        wsync();
    }
    fixed_gravity<true, DIRECT ? 4 : 2>(E, lds, B, acc);
    wsync();
    {   // interaction: the gravity in the chain's coordinates and the indirect term
        double own[3], sum[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) lds.xb[q][lane] = acc[q];
        wsync();
        forward(own, sum);
        wsync();
        if (B.orb) {
#pragma unroll
            for (int q = 0; q < 3; ++q) B.av[q] = B.av[q] + B.dt * own[q];
            if (!B.jfirst) {
                const double rj2i = 1. / (p2(B.ax[0]) + p2(B.ax[1]) + p2(B.ax[2]) + 1e-12);
                const double rji = sqrt(rj2i);
                const double rj3im = rji * rj2i * G * B.jeta;
                const double prefac = B.dt * rj3im;
#pragma unroll
                for (int q = 0; q < 3; ++q) B.av[q] = B.av[q] + prefac * B.ax[q];
            }
        }
    }
    drift(TP_XK2);
    {
        double own[6];
        const double com[6] = {B.comx[0], B.comx[1], B.comx[2], B.comv[0], B.comv[1], B.comv[2]};
#pragma unroll
        for (int q = 0; q < 3; ++q) { lds.xb[q][lane] = B.ax[q]; lds.xb[3 + q][lane] = B.av[q]; }
        wsync();
        reverse(own, com);
        wsync();
#pragma unroll
        for (int q = 0; q < 3; ++q) { B.x[q] = own[q]; B.v[q] = own[3 + q]; }
    }
}

// ===========================================================================
// Load, store, the steps of a launch
// ===========================================================================
// The lane's body and its constants; wave 0 fills the shared constants and the
// published positions and velocities, the owner of the spins the spins of the
// last evaluation.  Ends without a barrier.
template <int M, int ROLE, int V>
__device__ __forceinline__ void fixed_load(const DevEnsemble &E, FixedLds<M, (V & VAR_JACOBI) != 0> &lds, FixedLane &B, int wave) {
    using W = Role<M, ROLE>;
    constexpr bool JACOBI = (V & VAR_JACOBI) != 0;
    const int lane = threadIdx.x & (WAVE - 1);
    const LaneGroup lg = lane_group(E, wave, lane);
    const int s = lg.sys;
    B.lane = lane;
    B.gbase = lg.gbase;
    B.k = lg.k;
    B.sys = s;
    const int b0 = E.body_offset[s];
    B.n = lg.gvalid ? E.body_offset[s + 1] - b0 : 0;
    const bool valid = lg.gvalid && lg.k < B.n;
    B.host = 0;
    B.hidx = E.host[s];
    B.idx = !valid || lg.k == 0 ? B.hidx : lg.k <= B.hidx ? lg.k - 1 : lg.k;
    B.body = b0 + B.idx;
    B.host_lane = valid && lg.k == 0;
    B.orb = valid && lg.k != 0;
    B.nmax = 2;
    while (__any(B.n > B.nmax)) ++B.nmax;
    B.pairs = __any(B.n == 2);
    B.hosts_first = !__any(valid && B.hidx != 0);
    B.coord = JACOBI ? POS_COORD_JACOBI : (V & VAR_WHDS) ? POS_COORD_WHDS : POS_COORD_DEMOCRATIC_HELIOCENTRIC;
    B.flags = (valid ? F_VALID : 0u) | (B.host_lane ? F_HOST : 0u) | F_TIDES | F_RF | F_GR | F_SPIN |
              (B.orb ? (F_TIDES_ROLE | F_RF_ROLE | F_GR_ROLE) : 0u);
    const int b = B.body, nb = E.n_bodies;
    B.dt = E.dt[s];
    B.m = E.mass[b];
    B.inv_m = 1. / B.m;
    const double hm = E.mass[b0 + B.hidx];
    const Rcp Rhm = rcp(hm);
    B.I = E.inertia[b];
    B.inv_I = 1. / B.I;
    double k[K_COUNT] = {0., 0., 0., 0., 0., 0.}, ksys[4];
    if (B.orb) {
        const double m = B.m, hmg = hm * K2, pmg = m * K2;
        const Rcp Rm{m, B.inv_m}, RM = rcp(hm + m);
        k[K_F] = hmg * pmg / p2(hmg + pmg);
        k[K_M_OVER_HM] = divr(m, Rhm);
        k[K_MFM] = divr(hm - m, RM) * RM.b;
        k[K_MR] = divr(hm * m, RM);
        k[K_FM_HOST] = 2. + divr(3. / 2. * m, Rhm);
        k[K_FM_BODY] = 2. + divr(3. / 2. * hm, Rm);
    }
    if constexpr (W::OWN_V) {
        B.hist_period = E.hist_period[s];
        B.time_limit = E.time_limit[s];
        // the pair checks of this body are those with the bodies after it
        B.near2 = -1.;
        B.far2 = B.host_lane ? MAX_DISTANCE_2 : __builtin_inf();
        for (int j = B.idx + 1; valid && j < B.n; ++j) {
            const double rr = E.roche[(size_t)b * POS_MAX_BODIES + j];
            B.near2 = fmax(B.near2, fmax(rr * rr, p2(E.radius[b] + E.radius[b0 + j])));
        }
        B.t = E.t[s];
        B.last_hist = E.last_hist[s];
        B.iteration = E.iteration[s];
        B.status = E.status[s];
        if (!valid) B.status |= POS_STATUS_COMPLETED;   // idle lanes never iterate
        B.tw = E.timestep_warning[s];
        B.seen_status = B.status;
        B.seen_tw = B.tw;
        B.hcount = E.hist ? E.hist_count[s] : 0;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            B.x[q] = E.x[q * nb + b];
            B.v[q] = E.v[q * nb + b];
            B.ev[q] = E.err_v[q * nb + b];
            B.ax[q] = B.av[q] = B.comx[q] = B.comv[q] = 0.;
            lds.vel(q, lane) = B.v[q];
            if constexpr (M == 1) lds.xb[q][lane] = B.x[q];
            else lds.team.x[q][lane] = B.x[q];
        }
        lds.m[lane] = valid ? B.m : 0.;
        lds.R[lane] = E.radius[b];
        lds.I[lane] = E.inertia[b];
        lds.k2f[lane] = E.k2f[b];
        if (lane < NX) lds.xb[lane][WAVE] = 0.;   // the zero column
        if (lane == 0) lds.m[WAVE] = 0.;
        if constexpr (M > 1) {
            if (lane < 4) lds.team.cv[lane][WAVE] = 0.;
        }
        // masses along the chain, the host first then the others in index
        // order: their total, this body's Kepler mass and, in Jacobi
        // coordinates, the recurrences' ratios
        double total = hm, mass_g = hm * K2;
        B.mu = mass_g;
        B.jeta = hm;
        B.jfirst = true;
        bool first = true;
        for (int j = 0; j < B.n; ++j) {
            if (j == B.hidx) continue;
            const double mj = E.mass[b0 + j];
            const double ei = 1. / total;
            total = total + mj;
            mass_g = mass_g + mj * K2;
            if constexpr (JACOBI) {
                if (j == B.idx) {
                    B.mu = mass_g;
                    B.jeta = total;
                    B.jfirst = first;
                    lds.chain.ei[lane] = ei;
                }
            }
            first = false;
        }
        B.com_m = total;
        ksys[K_INV_HM] = Rhm.r;
        ksys[K_TOTAL] = total;
        ksys[K_INV_TOTAL] = 1. / total;
        ksys[K_INV_LEFT] = 0.;
        if constexpr (JACOBI) {
            double eta = total;
            for (int j = B.n - 1; j >= 0; --j) {
                if (j == B.hidx) continue;
                const double mj = E.mass[b0 + j];
                const double ei = 1. / eta;
                eta = eta - mj;
                if (j == B.idx) lds.chain.rei[lane] = ei;
            }
            ksys[K_INV_LEFT] = 1. / eta;
        }
    } else {
        ksys[K_INV_HM] = Rhm.r;
        ksys[K_TOTAL] = ksys[K_INV_TOTAL] = ksys[K_INV_LEFT] = 0.;
    }
    if constexpr (M == 1) {
#pragma unroll
        for (int i = 0; i < K_COUNT; ++i) lds.team.k[i][lane] = i < 4 && B.host_lane ? ksys[i] : k[i];
    } else {
#pragma unroll
        for (int i = 0; i < K_COUNT; ++i) B.kc[i] = k[i];
#pragma unroll
        for (int i = 0; i < 4; ++i) B.ksys[i] = ksys[i];
    }
    if constexpr (W::OWN_L) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            B.L[q] = E.L[q * nb + b];
            B.eL[q] = E.err_L[q * nb + b];
            if constexpr (M == 1) {
                lds.s[q][lane] = E.spin[q * nb + b];
            } else {
                B.s[q] = E.spin[q * nb + b];
                lds.team.so[q][lane] = B.s[q];
            }
        }
    }
}

template <int M, int ROLE, class Lds>
__device__ __forceinline__ void fixed_store(const DevEnsemble &E, const Lds &lds, const FixedLane &B) {
    using W = Role<M, ROLE>;
    if (!B.valid()) return;
    // The indices pass through an empty asm so that the field addresses are
    // formed here again rather than kept across the step loop.
    int b = B.body, s = B.sys;
    asm volatile("" : "+v"(b), "+v"(s));
    const int nb = E.n_bodies;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        if constexpr (W::OWN_V) {
            E.x[q * nb + b] = B.x[q];
            E.v[q * nb + b] = B.v[q];
            E.err_v[q * nb + b] = B.ev[q];
        }
        if constexpr (W::OWN_L) {
            E.L[q * nb + b] = B.L[q];
            E.spin[q * nb + b] = M == 1 ? lds.s[q][B.lane] : B.s[q];
            E.err_L[q * nb + b] = B.eL[q];
        }
    }
    if (W::OWN_V && B.k == 0) {
        E.t[s] = B.t;
        E.last_hist[s] = B.last_hist;
        E.iteration[s] = B.iteration;
        E.status[s] = B.status;
        E.timestep_warning[s] = B.tw;
        if (E.hist) E.hist_count[s] = B.hcount;
    }
}

// The steps of one launch for the systems of wave `wave`, wavefront ROLE of the
// team.  With REC each step also writes its tape row.
template <int M, int ROLE, bool REC, int V>
__device__ __forceinline__ void fixed_run(const DevEnsemble &E, FixedLds<M, (V & VAR_JACOBI) != 0> &lds, int wave, int n_steps, const TapeRef &T) {
    using W = Role<M, ROLE>;
    constexpr bool JACOBI = (V & VAR_JACOBI) != 0;
    constexpr uint32_t STOPPED = POS_STATUS_COMPLETED | POS_STATUS_FATAL;
    FixedLane B;
    FixedGeo g{};
    fixed_load<M, ROLE, V>(E, lds, B, wave);
    const int lane = B.lane;
    bool act = false, snap = false;
    double s_last[3];
    // What a step's first evaluation needs: velocities, spins (L / I at the
    // start of the step; whether the system takes the step is known to their
    // owner only after the barrier, a stopped system keeps those of its last
    // evaluation), and which systems go on and record a snapshot
    // (whfast.rs:239-256).  `snap` takes no branch: with `&&` the compiler saved
    // B.sys inside the branch, for the lanes of systems that go on alone, and
    // fixed_store then wrote a stopped system's time over another's (build.py's
    // partial_spills).
    auto publish = [&](bool velocities) {
        if constexpr (W::OWN_V) {
            act = !(B.status & STOPPED);
            snap = act & ((B.last_hist < 0.) | (B.last_hist + B.hist_period <= B.t));
            if constexpr (M > 1) {
                const unsigned long long live = __ballot(act), taken = __ballot(snap);
                if (lane == 0) { lds.team.live = live; lds.team.snap = taken; }
            }
            if (velocities && act) publish_velocity(lds, B);
        }
        if constexpr (M == 1) {
            if (act) publish_spin<M>(lds, B);
        } else if constexpr (W::OWN_L) {
#pragma unroll
            for (int q = 0; q < 3; ++q) s_last[q] = B.s[q];
            publish_spin<M>(lds, B);
        }
    };
    if constexpr (M == 1) {   // the geometry reads the last spins before the new ones are published
        wsync();
        if (B.orb) fixed_geometry<M, ROLE>(E, lds, B, g);
        wsync();
        publish(false);
        wsync();
    } else {
        publish(false);
        team_sync<M>();
        if (B.orb) fixed_geometry<M, ROLE>(E, lds, B, g);
    }
    // One pass per kick, one copy of the kick in the code: the first of a step is
    // followed by the drift, the second ends the step (star + 2 planets, 4,096
    // systems: 863 us per 64 steps against 890 with two copies).
    for (int pass = 0, step = 0;; ++pass) {
        int second = pass & 1;
        opaque(second);
        if (second == 0) {
            if (step == n_steps) break;
            if (step > 0) {
                publish(true);
                team_sync<M>();
            }
            if constexpr (!W::OWN_V) {
                act = (lds.team.live >> lane) & 1ull;
                snap = (lds.team.snap >> lane) & 1ull;
            }
            if constexpr (W::OWN_L && M > 1) {
#pragma unroll
                for (int q = 0; q < 3; ++q) B.s[q] = act ? B.s[q] : s_last[q];
            }
            if (!__any(act)) break;   // alike in every wavefront
            if ((W::TIDES || W::FLAT) && __any(snap)) {
                // a snapshot refreshes the spins before the step, so the first
                // evaluation's scalar products are taken with the refreshed ones
                if (snap) {
                    const int hl = B.hl();
                    if (B.orb) {
                        g.rs_star = g.px[0] * lds.s[0][hl] + g.px[1] * lds.s[1][hl] + g.px[2] * lds.s[2][hl];
                        g.rs_planet = g.px[0] * lds.s[0][lane] + g.px[1] * lds.s[1][lane] + g.px[2] * lds.s[2][lane];
                    }
                    if constexpr (W::OWN_V) {
                        if (E.hist) write_history_record<false>(E, lds, B);
                        B.last_hist = B.last_hist < 0. ? 0. : B.last_hist + B.hist_period;
                    }
                }
            }
            if (REC && act) {
                if (W::OWN_V) { tape_put3(T, step, TP_X, B.body, B.x); tape_put3(T, step, TP_V, B.body, B.v); }
                if (W::OWN_L) tape_put3(T, step, TP_L, B.body, B.L);
            }
        }
        fixed_kick<M, ROLE>(lds, B, g, act);
        if (second == 0) {
            if (REC && act) {
                if (W::OWN_V) {
                    tape_put3(T, step, TP_V1, B.body, B.v);
                    *T.at(step, TP_R, B.body) = lds.R[lane];
                    *T.at(step, TP_I, B.body) = lds.I[lane];
                }
                if (W::OWN_L) tape_put3(T, step, TP_L1, B.body, B.L);
            }
            if constexpr (W::OWN_L && M > 1) {
                // for the second kick: the spins just used (its scalar products
                // are taken with them) and those of its first evaluation
                if (act) {
                    put_rows(lds.team.so, lane, B.s);
                    publish_spin<M>(lds, B);
                }
            }
            if constexpr (W::OWN_V) {
                if (act) {
                    if (lds.I[lane] == 0.) B.status |= POS_STATUS_ZERO_INERTIA;   // particles/common.rs:5-7
                    double acc[3];
                    wsync();
                    if constexpr (JACOBI) drift_jacobi<(M > 1), REC>(E, lds, B, acc, T, step);
                    else drift_heliocentric<(M > 1), REC, (V & VAR_WHDS) != 0>(E, lds, B, acc, T, step);
                    // the state's gravitational acceleration, stored here rather than held through the second kick
                    const int nb = E.n_bodies;
#pragma unroll
                    for (int q = 0; q < 3; ++q) E.acc[q * nb + B.body] = acc[q];
                    wsync();
                    publish_velocity(lds, B);
                    if constexpr (M == 1) put3(lds, 0, lane, B.x[0], B.x[1], B.x[2]);
                    else put_rows(lds.team.x, lane, B.x);
                }
            }
            team_sync<M>();
            if (act && B.orb) fixed_geometry<M, ROLE>(E, lds, B, g);
            if constexpr (M == 1) {
                wsync();
                if (act) publish_spin<M>(lds, B);
                wsync();
            }
        } else {
            if (act) {
                if constexpr (REC) {
                    if (W::OWN_V) { tape_put3(T, step + 1, TP_X, B.body, B.x); tape_put3(T, step + 1, TP_V, B.body, B.v); }
                    if (W::OWN_L) tape_put3(T, step + 1, TP_L, B.body, B.L);
                }
                if constexpr (W::OWN_V) {
                    B.t = B.t + B.dt;
                    B.iteration += 1;
                    if constexpr (M == 1) wsync();
                    merge_status(lds, B);
                    if (B.t + B.dt > B.time_limit) B.status |= POS_STATUS_COMPLETED;
                }
            }
            ++step;
        }
    }
    fixed_store<M, ROLE>(E, lds, B);
}

}  // namespace posdev
