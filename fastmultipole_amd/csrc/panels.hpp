// Device functions of the constant-strength panel kernels, shared by the
// nearfield (p2p.hip) and the Gauss-Seidel influence matrices (fgs.hip).
#pragma once
#include "fmmhip_internal.hpp"

namespace fmmhip {

static constexpr double PANEL_INV4PI = 1.0 / (4.0 * 3.141592653589793);

// ================================================================ panels
// Constant-strength planar panels, nearfield: induced() of test/panels.jl
// (rotate_to_panel :78-93, source_dipole_preliminaries :95-133, Panel{Source}
// :139-216, Panel{Dipole} :224-315) for every (target, panel) pair, FP64 in both
// precision forms. The per-panel frame and edge geometry is computed once per panel
// and evaluation (k_panel_records) or when a panel is staged into LDS.
//
// The reference sums, over the edges, one log and two arctangents of quotients. The logs stay one per edge, as
// log((r+ - d)/(r+ + d)) = -2 atanh(d / r+) (edge_log). The arctangents of all edges sum to the signed solid angle of
// the panel. It is formed from the edges' angles in the form of Wilton et al. (1984), whose terms are smooth away from the
// edges, as the argument of a product of complex numbers: one arctangent per panel. (Two triangles' solid angles, van
// Oosterom and Strackee 1983, take fewer operations but cancel at targets near the diagonal, where the centroid of a
// quadrilateral lies.) Divisions and square roots are refined hardware estimates. A pair of a quadrilateral's
// potential and gradient takes about 300 FP64 operations instead of 8 arctangents, 20 divisions and 4 logs.

static constexpr int PANEL_TILE = 64;   // panels per LDS tile

template <int NV> struct PanelStage {
    double c[3], ex[3], ey[3], ez[3];   // centroid, panel frame (R' rows)
    double vx[NV], vy[NV];              // vertices in the panel frame
    double tx[NV], ty[NV], ds[NV];      // unit tangent and length of edge k -> k + 1
    double strength;
    double strength2;   // a source-dipole panel's dipole strength
    // an odd number of doubles: lanes on consecutive panels of a tile read different LDS banks
    double pad[(14 + 5 * NV) % 2 == 0 ? 1 : 2];
};
static_assert(sizeof(PanelStage<3>) == 8 * panel_record_doubles(3) && sizeof(PanelStage<4>) == 8 * panel_record_doubles(4),
              "the request server's estimate counts these records");

// panel j of the sorted arrays (rows after radius: NSTR strengths, v1, v2, ...) into a stage
template <int NV, int NSTR = 1>
__device__ inline void stage_panel(const double* __restrict__ px, const double* __restrict__ py, const double* __restrict__ pz,
                                   const double* __restrict__ rows, int64_t n, int64_t j, PanelStage<NV>& P) {
    double v[NV][3];
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int a = 0; a < 3; ++a) v[k][a] = rows[(int64_t)(NSTR + 3 * k + a) * n + j];
    P.c[0] = px[j]; P.c[1] = py[j]; P.c[2] = pz[j];
    P.strength = rows[j];
    P.strength2 = NSTR > 1 ? rows[n + j] : 0.0;
    // unit normal from the first three vertices (get_normal, src/compatibility.jl:65-72)
    const double a0 = v[1][0] - v[0][0], a1 = v[1][1] - v[0][1], a2 = v[1][2] - v[0][2];
    const double b0 = v[2][0] - v[0][0], b1 = v[2][1] - v[0][1], b2 = v[2][2] - v[0][2];
    double nz[3] = {a1 * b2 - a2 * b1, a2 * b0 - a0 * b2, a0 * b1 - a1 * b0};
    const double nzn = sqrt(nz[0] * nz[0] + nz[1] * nz[1] + nz[2] * nz[2]);
    double nx[3] = {b0, b1, b2};
    const double nxn = sqrt(b0 * b0 + b1 * b1 + b2 * b2);
#pragma unroll
    for (int a = 0; a < 3; ++a) { nz[a] /= nzn; nx[a] /= nxn; }
    const double ny[3] = {nz[1] * nx[2] - nz[2] * nx[1], nz[2] * nx[0] - nz[0] * nx[2], nz[0] * nx[1] - nz[1] * nx[0]};
#pragma unroll
    for (int a = 0; a < 3; ++a) { P.ex[a] = nx[a]; P.ey[a] = ny[a]; P.ez[a] = nz[a]; }
    double vx[NV], vy[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double d0 = v[k][0] - P.c[0], d1 = v[k][1] - P.c[1], d2 = v[k][2] - P.c[2];
        vx[k] = nx[0] * d0 + nx[1] * d1 + nx[2] * d2;
        vy[k] = ny[0] * d0 + ny[1] * d1 + ny[2] * d2;
        P.vx[k] = vx[k];
        P.vy[k] = vy[k];
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double dx = vx[(k + 1) % NV] - vx[k], dy = vy[(k + 1) % NV] - vy[k];
        const double d = sqrt(dx * dx + dy * dy);
        P.ds[k] = d;
        P.tx[k] = d == 0.0 ? 0.0 : dx / d;   // a vertex given twice: an edge that adds nothing
        P.ty[k] = d == 0.0 ? 0.0 : dy / d;
    }
}

// 1/x of a normal number (two Newton steps on the hardware estimate)
__device__ inline double panel_rcp(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y = fma(fma(-x, y, 1.0), y, y);
    return fma(fma(-x, y, 1.0), y, y);
}
// a / b, correctly rounded but for the last bit
__device__ inline double panel_div(double a, double b) {
    const double y = panel_rcp(b), q = a * y;
    return fma(fma(-b, q, a), y, q);
}
// sqrt(x) of x > 0, correctly rounded but for the last bit
__device__ inline double panel_sqrt(double x) {
    double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    y = fma(y * e, fma(e, 0.375, 0.5), y);
    const double r = x * y;
    return fma(fma(-r, r, x), 0.5 * y, r);
}

// log((rp - d) / (rp + d)), d >= 0: 2 atanh(s) - e ln 2 with the ratio's power of two e split off so that
// |s| <= 3 - 2 sqrt(2), then the series of atanh to s^21 (the next term is below 2^-56 of the sum). Without a power of
// two s = -d / rp, so a far panel's small logarithm keeps its relative accuracy; a wavefront whose pairs are all far
// (d <= 0.17 rp) skips the split. For a target on the edge rp - d rounds to zero or a few ulps below it (the distances and
// the length are rounded apart): either takes the reference's eps() for zero, so the logarithm is large and bounded.
__device__ inline double edge_log(double rp, double d) {
    const double EPS = 2.220446049250313e-16;   // the reference's eps() perturbation
    double a = -d, b = rp, shift = 0.0;
    if (__builtin_amdgcn_ballot_w64(d > 0.17 * rp)) {
        double num = rp - d;
        if (num <= 0.0) num = EPS;
        const double den = rp + d;
        int e = __builtin_amdgcn_frexp_exp(den) - __builtin_amdgcn_frexp_exp(num);
        double m = __builtin_amdgcn_ldexp(num, e);
        if (m > 1.4142135623730951 * den) { e -= 1; m *= 0.5; }
        if (m < 0.7071067811865476 * den) { e += 1; m *= 2.0; }
        if (e != 0) {
            a = m - den;
            b = m + den;
            shift = (double)e;
        }
    }
    const double s = panel_div(a, b), z = s * s;
    double p = 1.0 / 21.0;
    p = fma(p, z, 1.0 / 19.0);
    p = fma(p, z, 1.0 / 17.0);
    p = fma(p, z, 1.0 / 15.0);
    p = fma(p, z, 1.0 / 13.0);
    p = fma(p, z, 1.0 / 11.0);
    p = fma(p, z, 1.0 / 9.0);
    p = fma(p, z, 1.0 / 7.0);
    p = fma(p, z, 1.0 / 5.0);
    p = fma(p, z, 1.0 / 3.0);
    const double t = 2.0 * s;
    return fma(-shift, 0.6931471805599453, fma(t * z, p, t));
}

// one (target, panel) pair: the source's terms of strength st and / or the dipole's of strength std; accumulates
// [phi, velocity slot (3), Hessian slot (9)] into a
template <int NV, bool SOURCE, bool DIPOLE, bool PS, bool GS, bool HS>
__device__ inline void panel_terms(const PanelStage<NV>& P, double tx, double ty, double tz, double* a, double st, double std) {
    const double EPS = 2.220446049250313e-16;   // the reference's eps() perturbation
    const double d0 = tx - P.c[0], d1 = ty - P.c[1], d2 = tz - P.c[2];
    const double tRx = P.ex[0] * d0 + P.ex[1] * d1 + P.ex[2] * d2;
    const double tRy = P.ey[0] * d0 + P.ey[1] * d1 + P.ey[2] * d2;
    double dz = P.ez[0] * d0 + P.ez[1] * d1 + P.ez[2] * d2;
    if (dz == 0.0) dz = EPS;
    const double dz2 = dz * dz;
    double rxs[NV + 1], rys[NV + 1], rs[NV + 1];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        rxs[i] = tRx - P.vx[i];
        rys[i] = tRy - P.vy[i];
        // 1e-290: a target at a vertex whose dz^2 underflows
        rs[i] = panel_sqrt(fmax(fma(rxs[i], rxs[i], fma(rys[i], rys[i], dz2)), 1e-290));
    }
    rxs[NV] = rxs[0];
    rys[NV] = rys[0];
    rs[NV] = rs[0];
    constexpr bool ANGLE = PS || (SOURCE && GS), DOTS = (DIPOLE && GS) || HS;
    double dot[NV];   // R_i . R_(i + 1)
    if (DOTS) {
#pragma unroll
        for (int i = 0; i < NV; ++i) dot[i] = fma(rxs[i], rxs[i + 1], fma(rys[i], rys[i + 1], dz2));
    }
    // The solid angle: edge k adds atan(p l1 / (h + |z| r1)) - atan(p l0 / (h + |z| r0)), p the target's signed distance
    // from the edge's line in the plane, l0 and l1 the edge's ends along it, h = p^2 + z^2. An edge's angle lies in
    // (-pi, pi); two of one sign whose product's imaginary part has the other sign sum past pi. Lengths are taken in
    // units of the power of two above the distance R to the farthest vertex: |p|, |l|, |z| <= R, so an edge's number is at
    // most 8 and the product of all of them in range whatever the edges' lengths are.
    double angle = 0.0;
    if (ANGLE) {
        const double az = fabs(dz);
        int far = __double2hiint(rs[0]);   // distances are positive: their high words are in the order of the distances
#pragma unroll
        for (int k = 1; k < NV; ++k) far = max(far, __double2hiint(rs[k]));
        const int e0 = 2 * (1022 - (far >> 20));
        double re = 0.0, im = 0.0;
        int turns = 0;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const double p = rys[k] * P.tx[k] - rxs[k] * P.ty[k];
            const double l0 = -fma(rxs[k], P.tx[k], rys[k] * P.ty[k]), l1 = l0 + P.ds[k];
            const double h = fma(p, p, dz2);
            const double a0 = __builtin_amdgcn_ldexp(fma(az, rs[k], h), e0), a1 = __builtin_amdgcn_ldexp(fma(az, rs[k + 1], h), e0);
            const double ps = __builtin_amdgcn_ldexp(p, e0), b0 = ps * l0, b1 = ps * l1;
            const double er = fma(a1, a0, b1 * b0), ei = fma(b1, a0, -(a1 * b0));
            if (k == 0) { re = er; im = ei; continue; }
            const double nim = fma(re, ei, im * er);
            // a zero imaginary part with a negative real part is +pi here and in atan2
            if (im >= 0.0 && ei > 0.0 && nim < 0.0) ++turns;
            if (im < 0.0 && ei < 0.0 && nim >= 0.0) --turns;
            re = fma(re, er, -(im * ei));
            im = nim + 0.0;
        }
        const double beta = atan2(im, re) + turns * 6.283185307179586;
        angle = dz > 0.0 ? -beta : beta;   // the reference's sign
    }
    auto add = [&](bool dipole, double pot, double u0, double u1, double u2, const double* h, double s4) {
        if (PS) a[0] += pot * s4;
        if (GS) {   // velocity = (+-) s/(4 pi) R u, R = [ex ey ez] as columns
            const double sv = dipole ? s4 : -s4;
#pragma unroll
            for (int c = 0; c < 3; ++c) a[1 + c] += sv * (P.ex[c] * u0 + P.ey[c] * u1 + P.ez[c] * u2);
        }
        if (HS) {   // -s/(4 pi) R h R'
            const double H[3][3] = {{h[0], h[1], h[2]}, {h[1], h[3], h[4]}, {h[2], h[4], h[5]}};
            const double* E[3] = {P.ex, P.ey, P.ez};
            double RH[3][3];
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int k = 0; k < 3; ++k) RH[r][k] = E[0][r] * H[0][k] + E[1][r] * H[1][k] + E[2][r] * H[2][k];
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) a[4 + 3 * r + c] += -s4 * (RH[r][0] * E[0][c] + RH[r][1] * E[1][c] + RH[r][2] * E[2][c]);
        }
    };
    if (SOURCE) {
        double pot = dz * angle, u0 = 0.0, u1 = 0.0;
        double h[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};   // xx, xy, xz, yy, yz, zz
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const double r_plus = rs[i] + rs[i + 1], ds = P.ds[i];
            if (PS || GS) {
                const double log_term = edge_log(r_plus, ds);
                if (PS) pot = fma(rxs[i] * P.ty[i] - rys[i] * P.tx[i], log_term, pot);
                if (GS) { u0 = fma(P.ty[i], log_term, u0); u1 = fma(-P.tx[i], log_term, u1); }
            }
            if (HS) {
                const double dx = P.tx[i] * ds, dy = P.ty[i] * ds;
                const double r_times = rs[i] * rs[i + 1], rho = r_times + dot[i];
                const double lambda = rxs[i] * rys[i + 1] - rxs[i + 1] * rys[i];
                const double v1 = panel_rcp(r_plus * r_plus - ds * ds), i0 = panel_rcp(rs[i]), i1 = panel_rcp(rs[i + 1]);
                const double val2 = rxs[i] * i0 + rxs[i + 1] * i1;
                const double val3 = rys[i] * i0 + rys[i + 1] * i1;
                const double val4 = panel_div(r_plus, r_times * rho);
                h[0] += 2 * dy * v1 * val2;
                h[1] += -2 * dx * v1 * val2;
                h[2] += dz * dy * val4;
                h[3] += -2 * dx * v1 * val3;
                h[4] += -dz * dx * val4;
                h[5] += lambda * val4;
            }
        }
        add(false, pot, u0, u1, angle, h, st * PANEL_INV4PI);
    }
    if (DIPOLE) {
        double u0 = 0.0, u1 = 0.0, u2 = 0.0;
        double h[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            if (!GS && !HS) break;
            const double r_plus = rs[i] + rs[i + 1], dx = P.tx[i] * P.ds[i], dy = P.ty[i] * P.ds[i];
            const double r_times = rs[i] * rs[i + 1], rho = r_times + dot[i];
            const double lambda = rxs[i] * rys[i + 1] - rxs[i + 1] * rys[i];
            if (GS) {
                const double val4 = panel_div(r_plus, r_times * rho);
                u0 += dz * dy * val4;
                u1 += -dz * dx * val4;
                u2 += lambda * val4;
            }
            if (HS) {
                const double rp2 = r_plus * r_plus;
                const double val1 = panel_div(r_times * rp2 + rho * rs[i + 1] * rs[i + 1], rho * rs[i] * r_plus);
                const double val2 = panel_div(r_times * rp2 + rho * rs[i] * rs[i], rho * rs[i + 1] * r_plus);
                const double val3 = panel_div(r_plus, rho * r_times * r_times);
                h[0] += dz * dy * val3 * (rxs[i] * val1 + rxs[i + 1] * val2);
                h[1] += dz * dy * val3 * (rys[i] * val1 + rys[i + 1] * val2);
                h[3] += -dz * dx * val3 * (rys[i] * val1 + rys[i + 1] * val2);
                const double val6 = dz * (panel_div(rp2, rho) + panel_div(rs[i] * rs[i] - r_times + rs[i + 1] * rs[i + 1], r_times));
                h[5] += lambda * val3 * val6;
                const double val8 = val3 * (r_times - dz * val6);
                h[2] += -dy * val8;
                h[4] += dx * val8;
            }
        }
        add(true, -angle, u0, u1, u2, h, std * PANEL_INV4PI);
    }
}

// one (target, panel) pair of a source (DIPOLE false) or dipole panel of strength st
template <int NV, bool DIPOLE, bool PS, bool GS, bool HS>
__device__ inline void panel_pair(const PanelStage<NV>& P, double tx, double ty, double tz, double* a, double st) {
    panel_terms<NV, !DIPOLE, DIPOLE, PS, GS, HS>(P, tx, ty, tz, a, st, st);
}

// one (target, panel) pair of a panel kind: MODE 0 a source panel, 1 a dipole panel, 2 a source-dipole panel
// (the source's closed form with the first strength and the dipole's with the second, test/panels.jl:323-429, from one
// set of distances, dot products and solid angle)
template <int NV, int MODE, bool PS, bool GS, bool HS>
__device__ inline void panel_pair_kind(const PanelStage<NV>& P, double tx, double ty, double tz, double* a) {
    panel_terms<NV, MODE != 1, MODE != 0, PS, GS, HS>(P, tx, ty, tz, a, P.strength, MODE == 1 ? P.strength : P.strength2);
}

}  // namespace fmmhip
