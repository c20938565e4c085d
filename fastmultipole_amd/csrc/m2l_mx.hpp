// Register-resident M2L on the matrix cores (v_mfma_f64_4x4x4_4b_f64, gfx950).
//
// multipole_to_local! (src/translate.jl:519-550 fixed order, :555-1412 error-controlled) as rotate,
// translate along z, Lamb-Helmholtz transform, rotate back, for BP interactions of one target box at once
// per wavefront. The wavefront's 16 matrix columns are the potentials of the BP interactions ("slots"):
// NP = 2 with the Lamb-Helmholtz potential (phi, chi), NP = 1 without, so BP = 16 / NP. Real and imaginary
// parts are two registers of the same lane.
//
// Register layout. A degree-n coefficient vector (rows m = 0..n, one column per potential) is split by
// the parity of m: the even part E holds m = 8e + 2q in register e of the lanes of quad q = lane / 16, the
// odd part O holds m = 8o + 2q + 1, column = lane % 16. A register is a group of four rows of one parity: the
// K-block in which the 4x4x4 MFMA takes its B operand (lane l supplies B(l / 16, l % 16): four blocks of four
// columns, every block with the same A), and the layout of the four rows that it returns. Products therefore
// chain with no data movement, and since a given m sits in the same lane and register index for every degree, the
// z-translation L_j^m += F(j + k) M_k^m is a lane-local multiply-add.
//
// Rotations. The y-rotation of degree n is the factorised form of the reference's Wigner matrices
// (update_Ts!, src/rotate.jl:260-441, with the zeta / eta magnitudes of :625-1004):
//   U = g_in(m') X,  S_E(v) = A(0, v) U_0 / 2 + sum_{m' even > 0} A(m', v) U_m',  S_O(v) = sum_{m' odd} A(m', v) U_m'
//   n + v even:  R_e = cos Re S_E + sigma sin Im S_O           (real),
//                R_o = sigma sin Re S_E - cos Im S_O           (imaginary)
//   n + v odd:   R_e = cos Im S_E - sigma sin Re S_O           (imaginary),
//                R_o = -(cos Re S_O + sigma sin Im S_E)        (real),    cos, sin of v beta
//   out_m = 4 g_out(m) sum_v w_v A(m, v) R_(parity of m)(v),  w_0 = 1/2, else 1
// with A the degree-n pi/2 table (symmetric; A(0, v) = 0 for n + v odd). So for every v one of the two sums is needed
// per real or imaginary part, not both: with real and imaginary parts in registers of their own and the v of one
// parity in a register, the products that are not needed are not formed, and the combination is two multiplies and
// two multiply-adds in the lane. (Components in neighbouring columns, sums over m' and v in 16x16x4 products and the
// combination masked per element over DPP exchanges took 31,000 instructions per 4 interactions at order 20.) The
// number of 4x4x4 products of a degree is 2 (KE + KO)^2 for 16 complex columns, each at a quarter of a 16x16x4's 64
// cycles, and their FP64 units are those of the vector ALU: the two do not overlap (measured: a product and a
// multiply-add take the sum of their times), so both counts matter.
//
// z-translation, streamed by degree. The reference forms L_n^m = sum_{k=m}^{P} F(n + k) M_k^m with
// F(j) = j! / t^(j+1) after the whole rotated multipole exists. Here degree k of the multipole is
// rotated, added to L_k (which then holds the degree-k part translate_multipole_to_local_z_n! and
// translate_multipole_to_local_z_m01_n! compute for the error tests), the order tests of degree k run,
// and only if the interaction's order is not settled below k is M_k added to the other degrees L_j.
// F(j) follows the reference's product chain F(j) = F(j - 1) ((j) / t) from F(0) = 1 / t, so every
// factor is the same double the reference uses. The terms of each L_n^m are added in the reference's
// order (ascending k); multiply-adds are fused.
//
// The tests of the error-controlled methods (RotatedCoefficients*, PowerPotential / PowerGradient,
// absolute or relative) use the reference's formulas and running products; the sums over m of the
// power tests are taken as lane reductions, so a test value can differ from the reference's in the last
// bits and an order decision sitting on the tolerance can flip.
//
// The engine is written against a backend B (per-lane value types, cross-lane moves, the MFMA) so the
// same source runs on the GPU (backend in m2l_mx_gpu.hpp) and lane by lane on the CPU (the emulation
// used by the tests), with the same tables and scratch in the same order. It is plain C++ apart from the backend.
#pragma once
#include <cstdint>
#include <type_traits>

#if defined(__HIPCC__)
#define MX_FN __device__ __forceinline__
#else
#define MX_FN inline
#endif

namespace fmmhip {
namespace mx {

constexpr int mnh(int p) { return p < 0 ? 0 : ((p + 1) * (p + 2)) >> 1; }
constexpr int KE(int n) { return (n / 2 + 4) / 4; }          // registers of the even part of degree n
constexpr int KO(int n) { return ((n + 1) / 2 + 3) / 4; }    // registers of the odd part
constexpr int LOFF(int n) { return n <= 0 ? 0 : LOFF(n - 1) + KE(n - 1) + KO(n - 1); }   // degree n in L
constexpr int NLREG(int cap) { return LOFF(cap + 1); }
template <int n>
struct LO {   // LOFF(n) as a constant (register arrays need compile-time indices)
    static constexpr int v = LOFF(n);
};
constexpr int AST(int n) { return (n + 2) & ~1; }            // row length of degree n in the dense pi/2 tables (host_dense_A)
constexpr int ABASE(int n) { return (n * (n + 1) * (2 * n + 1)) / 6 + ((n + 1) / 2) * ((n + 1) / 2); }
// zero-padded pi/2 table: degree n as (KE + KO)^2 blocks of 4x4 at PBASE(n), rows and columns by parity (E groups, then O).
// Rows and columns past the degree are zero in every product, so no row of a rotation needs a mask.
constexpr int PBASE(int n) { return n <= 0 ? 0 : PBASE(n - 1) + 16 * (KE(n - 1) + KO(n - 1)) * (KE(n - 1) + KO(n - 1)); }
constexpr int PLEN(int cap) { return PBASE(cap + 1); }
constexpr int imin(int a, int b) { return a < b ? a : b; }
constexpr int imax(int a, int b) { return a > b ? a : b; }

template <int I0, int I1, class F>
MX_FN void sfor(F&& f) {
    if constexpr (I0 < I1) {
        f(std::integral_constant<int, I0>());
        sfor<I0 + 1, I1>(f);
    }
}

// Shared tables (LDS on the GPU), for degrees 0..CAP; per (n, m) tables are indexed mnh(n - 1) + m.
struct Tabs {
    double* A;     // zero-padded pi/2 tables
    double* zin;   // zeta input scale (multipole rotation)
    double* zoh;   // half the zeta output scale
    double* ein;   // eta input scale (local rotation)
    double* eoh;   // half the eta output scale
    double* Mt;    // multipole power normalisation
    double* Lt;    // local power normalisation
    double* tf;    // per degree n: 1/(n-1)!, (n+1)!
    double* i0;    // per degree n: 1 / Mt(n, 0), 1 / Lt(n, 0)
};

// per-wavefront scratch
struct Wave {
    double* eim;   // BP x (CAP + 1) x 2: 8 e^{i m alpha} of each slot (the 8 is the rotation's 4 and g_out's halves)
    double* cs;    // BP x (CAP + 1) x 2: w_v cos / sin (v beta) of each slot
    double* acc;   // mnh(CAP) x NC: the target box's local expansion, summed over the wave's interactions
    double* F;     // BP x (2 CAP + 1): z-translation factors j! / t^(j+1) of each slot
};

// Where they lie: the tables, then each wavefront's scratch. Rows past a degree are read unmasked (they are multiplied by
// zero): past a degree's row of an (n, m) table into the next degree or the next table, past a slot's phases into the
// next slot's, and past the last slot's eim into cs, past its cs into F. Every double so read is written before.
template <int CAP>
constexpr int shared_doubles() {
    return PLEN(CAP) + 6 * mnh(CAP) + 4 * (CAP + 1);
}
template <int CAP>
MX_FN Tabs tabs(double* lds) {
    constexpr int H = mnh(CAP);
    double* t = lds + PLEN(CAP);
    return {lds, t, t + H, t + 2 * H, t + 3 * H, t + 4 * H, t + 5 * H, t + 6 * H, t + 6 * H + 2 * (CAP + 1)};
}
template <int CAP, bool LH>
constexpr int wave_doubles() {
    return (LH ? 4 : 2) * mnh(CAP) + 4 * (LH ? 8 : 16) * (CAP + 1) + (LH ? 8 : 16) * (2 * CAP + 1);
}
template <int CAP, bool LH>
MX_FN Wave wave(double* w) {
    constexpr int A = (LH ? 4 : 2) * mnh(CAP), E = 2 * (LH ? 8 : 16) * (CAP + 1);
    return {w + A, w + A + E, w, w + A + 2 * E};
}
// entry t of degree n's blocks in the padded table, from the dense tables
template <class D>
MX_FN double padded(const D* Ad, int n, int t) {
    const int ke = KE(n), nb = ke + KO(n);
    const int rq = t / (16 * nb), kq = (t >> 4) % nb, i = (t >> 2) & 3, q = t & 3;
    const int row = (rq < ke ? 8 * rq : 8 * (rq - ke) + 1) + 2 * i, col = (kq < ke ? 8 * kq : 8 * (kq - ke) + 1) + 2 * q;
    return row <= n && col <= n ? Ad[ABASE(n) + row * AST(n) + col] : 0.0;
}

// BP consecutive entries b0 .. b0 + nb - 1 of the target box's part of the M2L list, taken in the
// order perm gives (list indices; null: list order)
struct Batch {
    const int32_t* m2l_s;   // source branch per list entry
    const int32_t* perm;    // processing order of the list entries, or null
    int b0, nb;
    int32_t* orders;        // expansion order per list entry (written)
};

// the target box and the method (uniform over the wavefront)
struct Box {
    double tc[3], tbox[3];
    double r_l;     // target radius
    double limit;   // 4 pi eps (eps scaled by max_influence for the relative methods)
    int P;          // expansion order (fixed) or order cap (error-controlled), <= CAP
    int kind;       // 0 fixed order, 1 rotated coefficients (gradient), 2 power potential, 3 power gradient
    int BE;         // the order settles at the passing degree (1) or one below (0)
};

// ERR: error-controlled orders (Box::kind 1 to 3), else the fixed order P (kind 0)
template <class B, int CAP, bool LH, bool ERR>
struct Engine {
    using V = typename B::V;
    using I = typename B::I;
    using M = typename B::M;
    using PV = typename B::PV;
    static constexpr int NP = LH ? 2 : 1;    // potentials
    static constexpr int NC = 2 * NP;        // real components per coefficient
    static constexpr int BP = 16 / NP;
    static constexpr int NL = NLREG(CAP);    // registers of the local expansion, per real or imaginary part
    static constexpr int NS = CAP + 1;   // slot-table entries
    static constexpr int NF = 2 * CAP + 1;   // translation factors per slot
    static constexpr int NX = KE(CAP) + KO(CAP);   // registers of one degree
    static constexpr double SQ3 = 1.7320508075688772;

    // src/error.jl:5-10
    MX_FN static V md1(V dx, double rm, double rp) {
        const V right = dx + rp, left = dx + rm;
        const M same = right * left >= 0.0;
        const V mn = B::sel(B::fabs(right) <= B::fabs(left), right, left);
        return B::sel(same, mn, V(0.0));
    }

    // list index of slot `slot` of the batch (of its first slot for an empty one)
    MX_FN static I entry(const Batch& Bt, I slot, M ok) {
        const I k = B::seli(ok, slot, I(0)) + Bt.b0;
        return Bt.perm ? B::gldi(Bt.perm, k, M(true)) : k;
    }

    // translation vector target centre - source centre of source branch js (benign values for empty slots)
    MX_FN static void geometry(const Box& X, I js, M ok, const double* sbr, int br_stride, int sc_off, V& dx, V& dy, V& dz) {
        const I base = js * br_stride + sc_off;
        const V sx = B::gld(sbr, base, ok), sy = B::gld(sbr, base + 1, ok), sz = B::gld(sbr, base + 2, ok);
        dx = B::sel(ok, X.tc[0] - sx, V(0.0));
        dy = B::sel(ok, X.tc[1] - sy, V(0.0));
        dz = B::sel(ok, X.tc[2] - sz, V(1.0));
    }

    // cos / sin of the azimuth and polar angle of (x, y, z) from the Cartesian components
    // (cartesian_to_spherical, src/rotate.jl:5-21, up to rounding); returns r
    MX_FN static V angles(V x, V y, V z, V& cp, V& sp, V& cb, V& sb) {
        const V x2y2 = x * x + y * y;
        const V r = B::sqrt(x2y2 + z * z);
        const M has = x2y2 > 0.0;
        const V rho = B::sqrt(x2y2);
        const V rs = B::sel(has, rho, V(1.0)), rr = B::sel(r > 0.0, r, V(1.0));
        cp = B::sel(has, x / rs, V(1.0));
        sp = B::sel(has, y / rs, V(0.0));
        cb = B::sel(has, z / rr, B::sel(z < 0.0, V(-1.0), V(1.0)));
        sb = B::sel(has, rho / rr, V(0.0));
        return r;
    }

    // Per-slot tables in the wave's LDS: e^{i m alpha} and (cos, sin)(m beta), m = 0..CAP, and the
    // z-translation factors F(j) = j! / t^(j+1), j = 0..2 CAP. Lane l serves slot l / (64 / BP) and
    // entries l % (64 / BP) + h (64 / BP): it forms its first entry by repeated multiplication and each
    // later one by continuing the same recurrence (update_eimphis!, src/rotate.jl:25-36; the
    // angle-addition recurrence of update_Ts!, :380-435; the factor chain of
    // translate_multipole_to_local_z!, src/translate.jl:181-232), so every entry is the double the
    // reference's chain produces.
    MX_FN static void slot_tables(const Box& X, const Wave& W, const Batch& Bt, const double* sbr, int br_stride, int sc_off) {
        constexpr int LPS = 64 / BP;
        B::wsync();   // the previous batch's reads of the tables are done
        const I l = B::lane();
        const I sT = l / LPS, kT = l % LPS;
        const M vT = sT < Bt.nb;
        V dx, dy, dz;
        geometry(X, B::gldi(Bt.m2l_s, entry(Bt, sT, vT), vT), vT, sbr, br_stride, sc_off, dx, dy, dz);
        V cp, sp, cb, sb;
        const V r = angles(dx, dy, dz, cp, sp, cb, sb);
        const V ot = 1.0 / r;
        // an empty slot's phases are zero: its multipole and its local expansion are then zero in every degree
        V er = B::sel(vT, V(8.0), V(0.0)), ei = 0.0, c = 1.0, s = 0.0, f = ot;
        auto step = [&](M st, int x) {
            const V t = er;
            const V ner = er * cp - ei * sp;
            const V nei = t * sp + ei * cp;
            const V cn = cb * c - sb * s;
            const V sn = sb * c + cb * s;
            er = B::sel(st, ner, er);
            ei = B::sel(st, nei, ei);
            c = B::sel(st, cn, c);
            s = B::sel(st, sn, s);
            (void)x;
        };
        // F's own chain: F(x) = F(x - 1) (x / t)
        for (int j = 0; j < LPS - 1; ++j) {
            const M st = kT > j;
            step(st, j);
            f = B::sel(st, f * ((double)(j + 1) * ot), f);
        }
        sfor<0, (2 * CAP + LPS) / LPS>([&](auto HH) {
            constexpr int h = decltype(HH)::value;
            if constexpr (h > 0) {
                for (int j = 0; j < LPS; ++j) {
                    if (h * LPS - LPS + j < CAP) step(M(true), j);
                    f = f * (B::tod(kT + (h * LPS - LPS + j + 1)) * ot);
                }
            }
            const I k = kT + h * LPS;
            const M okk = k <= CAP, okf = k <= 2 * CAP;
            const I idx = B::seli(okk, (sT * NS + k) * 2, I(0));
            B::lds_st(W.eim, idx, er, okk);
            B::lds_st(W.eim, idx + 1, ei, okk);
            if constexpr (h == 0) B::lds_st(W.cs, idx, B::sel(kT == 0, V(0.5), c), okk);
            else B::lds_st(W.cs, idx, c, okk);
            B::lds_st(W.cs, idx + 1, s, okk);
            B::lds_st(W.F, B::seli(okf, sT * NF + k, I(0)), f, okf);
        });
        B::wsync();
    }

    // One rotation of degree n (compile-time) of the coefficient vector u (input scale applied, row 0 halved): out as in
    // the header, without the factor 4 w (in the slot tables). sigma = +1 multipole (zeta), -1 local (eta). Rows m > n of u
    // may hold any finite value (the padded table's columns are zero there); rows m > n of the result are zero.
    template <int n>
    MX_FN static void rotate(const Tabs& T, const Wave& W, const double* gout, double sigma, I c, I q, I s,
                             const V (&uEr)[imax(KE(n), 1)], const V (&uEi)[imax(KE(n), 1)], const V (&uOr)[imax(KO(n), 1)],
                             const V (&uOi)[imax(KO(n), 1)], V (&oEr)[imax(KE(n), 1)], V (&oEi)[imax(KE(n), 1)],
                             V (&oOr)[imax(KO(n), 1)], V (&oOi)[imax(KO(n), 1)]) {
        constexpr int ke = KE(n), ko = KO(n);
        const I q2 = q * 2, i2 = (c & 3) * 2;
        // A block of rows 8 r + pr + 2 (lane % 4) and columns 8 k + pk + 2 (lane / 16)
        auto blk = [&](auto R, auto PR, auto KK, auto PK) {
            constexpr int rq = decltype(R)::value + (decltype(PR)::value ? ke : 0);
            constexpr int kq = decltype(KK)::value + (decltype(PK)::value ? ke : 0);
            return B::lds(T.A, i2 * 2 + q + (PBASE(n) + (rq * (ke + ko) + kq) * 16));
        };
        using C0 = std::integral_constant<int, 0>;
        using C1 = std::integral_constant<int, 1>;
        const I sb = s * (NS * 2);
        sfor<0, ke>([&](auto AA) { oEr[decltype(AA)::value] = V(0.0); oEi[decltype(AA)::value] = V(0.0); });
        sfor<0, imax(ko, 1)>([&](auto AA) { oOr[decltype(AA)::value] = V(0.0); oOi[decltype(AA)::value] = V(0.0); });
        auto add = [](const V& a, const V& b, V& d) { d = B::mfma4(a, b, d); };
        // the v of one register (parity par): first products, combination, second products
        auto half = [&](auto par, auto VI) {
            constexpr int pv = decltype(par)::value, vi = decltype(VI)::value, v0 = 8 * vi + pv;
            constexpr bool even = ((n + pv) & 1) == 0;   // n + v even
            V se = V(0.0), so = V(0.0);   // the needed parts of S_E and S_O
            sfor<0, ke>([&](auto EE) { add(blk(VI, par, EE, C0()), even ? uEr[decltype(EE)::value] : uEi[decltype(EE)::value], se); });
            sfor<0, ko>([&](auto OO) { add(blk(VI, par, OO, C1()), even ? uOi[decltype(OO)::value] : uOr[decltype(OO)::value], so); });
            const I vr = q2 + v0;
            const I ci = sb + vr * 2;
            const V cv = B::lds(W.cs, ci), sv = B::lds(W.cs, ci + 1) * sigma;
            V re, ro;
            if constexpr (even) {
                re = B::fma(sv, so, cv * se);
                ro = B::fma(-cv, so, sv * se);
            } else {
                re = B::fma(-sv, so, cv * se);
                ro = -B::fma(cv, so, sv * se);
            }
            sfor<0, ke>([&](auto AA) {
                constexpr int a = decltype(AA)::value;
                add(blk(AA, C0(), VI, par), re, even ? oEr[a] : oEi[a]);
            });
            sfor<0, ko>([&](auto AA) {
                constexpr int a = decltype(AA)::value;
                add(blk(AA, C1(), VI, par), ro, even ? oOi[a] : oOr[a]);
            });
        };
        sfor<0, ke>([&](auto VI) { half(C0(), VI); });
        sfor<0, ko>([&](auto VI) { half(C1(), VI); });
        auto out = [&](auto par, auto RI, V& xr, V& xi) {
            constexpr int m0 = 8 * decltype(RI)::value + decltype(par)::value;
            const V g = B::lds(gout, q2 + (m0 + mnh(n - 1)));
            xr = g * xr;
            xi = g * xi;
        };
        sfor<0, ke>([&](auto EE) { out(C0(), EE, oEr[decltype(EE)::value], oEi[decltype(EE)::value]); });
        sfor<0, ko>([&](auto OO) { out(C1(), OO, oOr[decltype(OO)::value], oOi[decltype(OO)::value]); });
    }

    // the source coefficients of degree n for this lane's rows (E registers, then O); rows m > n are row n's
    template <int n>
    MX_FN static void fetch(const PV& src, I q, I pot, V (&xr)[NX], V (&xi)[NX]) {
        auto one = [&](auto par, auto RI, V& r, V& i) {
            constexpr int m0 = 8 * decltype(RI)::value + decltype(par)::value;
            const I at = (q * 2) * 4 + pot * 2;
            constexpr int k0 = (m0 + mnh(n - 1)) * 4;
            if constexpr (m0 + 6 > n) {
                const I last = B::mini(q * 2 + m0, n) * 4 + pot * 2;
                r = B::gldp(src, last + mnh(n - 1) * 4);
                i = B::gldp(src, last + (mnh(n - 1) * 4 + 1));
            } else {
                r = B::gldp(src, at + k0);
                i = B::gldp(src, at + (k0 + 1));
            }
        };
        sfor<0, KE(n)>([&](auto EE) { one(std::integral_constant<int, 0>(), EE, xr[decltype(EE)::value], xi[decltype(EE)::value]); });
        sfor<0, KO(n)>([&](auto OO) {
            one(std::integral_constant<int, 1>(), OO, xr[KE(n) + decltype(OO)::value], xi[KE(n) + decltype(OO)::value]);
        });
    }

    // phi's and chi's value of a column, in both of the slot's columns
    MX_FN static V phi_of(V x) {
        if constexpr (LH) return B::template qbcast<2, 0>(x);
        else return x;
    }
    MX_FN static V chi_of(V x) { return B::template qbcast<2, 1>(x); }

    // One batch of interactions of one target box: their local expansions are added to W.acc and their
    // orders written to Bt.orders. pmax / ok collect the largest order and whether every tolerance was met.
    MX_FN static void batch(const Tabs& T, const Wave& W, const Box& X, const Batch& Bt, const double* sbr, int br_stride,
                            int sc_off, const double* sex, int64_t HE4, int& pmax, int& okflag) {
        slot_tables(X, W, Bt, sbr, br_stride, sc_off);
        const I l0 = B::lane();
        const I c0 = l0 & 15, q0 = l0 >> 4;
        const I s0 = LH ? (c0 >> 1) & 7 : c0, pot0 = LH ? c0 & 1 : I(0);
        const M valid = s0 < Bt.nb;
        const int P = X.P;
        constexpr bool err = ERR;

        // an empty slot reads the batch's first interaction; its phases are zero (slot_tables)
        const I li = entry(Bt, s0, valid);
        const I js = B::gldi(Bt.m2l_s, li, M(true));
        V dx, dy, dz;
        geometry(X, js, valid, sbr, br_stride, sc_off, dx, dy, dz);
        const V r = B::sqrt(dx * dx + dy * dy + dz * dz);
        const PV src = B::ptr(sex, js, HE4);
        const M chi_lane = pot0 == 1;
        V r_mp = V(1.0), rmi = V(1.0);
        if (err) {
            const V d0 = md1(dx, -X.tbox[0], X.tbox[0]), d1 = md1(dy, -X.tbox[1], X.tbox[1]), d2 = md1(dz, -X.tbox[2], X.tbox[2]);
            r_mp = B::sqrt(d0 * d0 + d1 * d1 + d2 * d2);
            rmi = 1.0 / r_mp;
        }

        V Lr[NL], Li[NL];
        sfor<0, NL>([&](auto II) { Lr[decltype(II)::value] = V(0.0); Li[decltype(II)::value] = V(0.0); });
        // degree k's source coefficients are loaded during degree k - 1 (their HBM latency hidden)
        V xnr[NX], xni[NX];
        fetch<0>(src, q0, pot0, xnr, xni);
        M active = valid;
        M succ = valid && !err;
        I Pl = I(P);
        V rmi_np2 = rmi * rmi * rmi;  // r_mp^-(n+2) at the test of degree n
        double rl_nm1 = 1.0;          // r_l^(n-1)
        V mp_pow = V(0.0);            // multipole power (phi) of the previous degree
        bool running = true;
        int kdone = -1;

        sfor<0, CAP + 1>([&](auto KK) {
            constexpr int k = decltype(KK)::value;
            if (!running || k > P) return;
            B::sched_fence();   // keep each degree's instructions together (limits register pressure)
            kdone = k;
            constexpr int ke = KE(k), ko = KO(k), ke1 = imax(ke, 1), ko1 = imax(ko, 1);
            // lane indices made opaque per degree: their derived addresses and masks are recomputed here
            // instead of being hoisted (one register each for the whole kernel)
            const I c = B::opaque(c0) & 15, q = B::opaque(q0) & 3;
            const I s = LH ? c >> 1 : c, pot = LH ? c & 1 : I(0);
            const I fb = s * NF, sb2 = s * (NS * 2), q2 = q * 2;
            // ---- degree k of the source multipoles: power terms, z-rotation, input scale
            V uEr[ke1], uEi[ke1], uOr[ko1], uOi[ko1], MEr[ke1], MEi[ke1], MOr[ko1], MOi[ko1];
            V xcr[NX], xci[NX];
            sfor<0, ke + ko>([&](auto II) {
                xcr[decltype(II)::value] = xnr[decltype(II)::value];
                xci[decltype(II)::value] = xni[decltype(II)::value];
            });
            if constexpr (k + 1 <= CAP) {
                if (k + 1 <= P) fetch<k + 1>(src, q, pot, xnr, xni);
            }
            V pw_t = V(0.0);
            const bool power = err && X.kind >= 2;
            auto load = [&](auto par, auto RI, V& ur, V& ui) {
                constexpr int pr = decltype(par)::value, ri = decltype(RI)::value, m0 = 8 * ri + pr;
                const I mi = q2 + m0;
                const V xr = xcr[(pr ? ke : 0) + ri], xi = xci[(pr ? ke : 0) + ri];
                if (power) {
                    V nt = B::lds(T.Mt, mi + mnh(k - 1));
                    if constexpr (m0 + 6 > k) nt = B::sel(q2 + m0 <= k, nt, V(0.0));
                    pw_t = B::fma(B::fma(xr, xr, xi * xi) * nt, nt, pw_t);
                }
                const I ei = sb2 + mi * 2;
                const V er = B::lds(W.eim, ei), eimg = B::lds(W.eim, ei + 1);
                const V g = B::lds(T.zin, mi + mnh(k - 1));
                ur = g * B::fma(xr, er, -(xi * eimg));
                ui = g * B::fma(xi, er, xr * eimg);
                if constexpr (m0 == 0) ur = ur * B::sel(q == 0, V(0.5), V(1.0));   // half of row 0 (ui's multiplies A(0, v) = 0)
            };
            sfor<0, ke>([&](auto EE) { load(std::integral_constant<int, 0>(), EE, uEr[decltype(EE)::value], uEi[decltype(EE)::value]); });
            sfor<0, ko>([&](auto OO) { load(std::integral_constant<int, 1>(), OO, uOr[decltype(OO)::value], uOi[decltype(OO)::value]); });
            if constexpr (ko == 0) { uOr[0] = V(0.0); uOi[0] = V(0.0); }
            V pw_phi = V(0.0), pw_chi = V(0.0);
            if (power) {
                const V t = B::sqrt(B::quadsum(pw_t));
                pw_phi = phi_of(t);
                if constexpr (LH) pw_chi = chi_of(t);
            }
            // ---- y-rotation of degree k (rotate_multipole_y!, zeta magnitudes)
            rotate<k>(T, W, T.zoh, 1.0, c, q, s, uEr, uEi, uOr, uOi, MEr, MEi, MOr, MOi);
            // ---- L_k += F(2k) M_k
            {
                V fac = B::lds(W.F, fb + 2 * k);
                if (err) fac = B::sel(active, fac, V(0.0));
                sfor<0, ke>([&](auto EE) {
                    constexpr int e = decltype(EE)::value;
                    Lr[LO<k>::v + e] = B::fma(fac, MEr[e], Lr[LO<k>::v + e]);
                    Li[LO<k>::v + e] = B::fma(fac, MEi[e], Li[LO<k>::v + e]);
                });
                sfor<0, ko>([&](auto OO) {
                    constexpr int o = decltype(OO)::value;
                    Lr[LO<k>::v + ke + o] = B::fma(fac, MOr[o], Lr[LO<k>::v + ke + o]);
                    Li[LO<k>::v + ke + o] = B::fma(fac, MOi[o], Li[LO<k>::v + ke + o]);
                });
            }
            // ---- order tests of degree k. Uniform factors are formed once per degree from reciprocal
            // tables (reordered products: test values agree with the reference's to a few ulps), and the
            // local part is skipped when no active interaction's multipole part is within the tolerance
            // (the reference evaluates it only then).
            if (err) {
                M pass = M(false);
                if constexpr (k >= 1) {
                    constexpr double ik = 1.0 / k, ik1 = 1.0 / (k + 1);
                    const double nm1_f_inv = T.tf[2 * k], np1_f = T.tf[2 * k + 1];
                    V eps_mp, eps_l = V(0.0);
                    if (X.kind == 1) {
                        // rotated coefficients (src/translate.jl:555-826): m = 0, 1 of the rotated multipole and
                        // of the degree-k local (translate_multipole_to_local_z_m01_n!, :302-362)
                        const V e0 = B::bperm(MEr[0], c), e1r = B::bperm(MOr[0], c), e1i = B::bperm(MOi[0], c);
                        const V n1 = B::sqrt(e1r * e1r + e1i * e1i);
                        eps_mp = phi_of(n1 + B::fabs(e0)) * np1_f * rmi_np2;
                        if constexpr (LH) eps_mp = eps_mp + chi_of(n1) * np1_f * rmi_np2 * r_mp;
                        if (B::any(active && (eps_mp <= X.limit))) {
                            const V l0 = B::bperm(Lr[LO<k>::v], c), l1r = B::bperm(Lr[LO<k>::v + ke], c),
                                    l1i = B::bperm(Li[LO<k>::v + ke], c);
                            const V p0 = phi_of(l0);
                            V p1r = phi_of(l1r), p1i = phi_of(l1i);
                            const double cl = rl_nm1 * nm1_f_inv;
                            if constexpr (LH) {
                                const V d1r = chi_of(l1r), d1i = chi_of(l1i);
                                const V ton = r * ik;
                                p1r = p1r - ton * d1i;
                                p1i = p1i + ton * d1r;
                                eps_l = (B::fabs(p1r) + B::fabs(p1i) + B::fabs(p0)) * cl + B::sqrt(d1r * d1r + d1i * d1i) * (cl * X.r_l);
                            } else {
                                eps_l = (B::fabs(p1r) + B::fabs(p1i) + B::fabs(p0)) * cl;
                            }
                        }
                    } else {
                        // powers (src/translate.jl:831-1412): multipole power of degree k (or k - 1), local
                        // power of the degree-k local (local_power, :455-502)
                        const double iM0 = T.i0[2 * (k - 1)], iM1 = T.i0[2 * k], iN = T.i0[2 * k + 1];
                        if (X.kind == 3) {
                            eps_mp = mp_pow * (SQ3 * np1_f * iM0);
                            if (LH) eps_mp = eps_mp + pw_chi * (SQ3 * (double)k * np1_f * iM1);
                            eps_mp = eps_mp * rmi_np2;
                        } else {
                            eps_mp = pw_phi * (SQ3 * np1_f * iM0 * ik1);
                            if (LH) eps_mp = eps_mp + pw_chi * (SQ3 * (double)k * np1_f * iM1 * ik1);
                            eps_mp = eps_mp * rmi_np2 * r_mp;
                        }
                        if (B::any(active && (eps_mp <= X.limit))) {
                            const V qd = B::tod(q2);
                            const V rk = B::sel(chi_lane, V(0.0), r * ik), rk1 = B::sel(chi_lane, r * ik1, V(0.0));
                            V lsum = V(0.0);
                            auto term = [&](auto par, auto RI) {
                                constexpr int pr = decltype(par)::value, ri = decltype(RI)::value, m0 = 8 * ri + pr;
                                constexpr int at = LO<k>::v + (pr ? ke : 0) + ri;
                                const I m = q2 + m0;
                                V vr = Lr[at], vi = Li[at];
                                if constexpr (LH) {
                                    // phi lanes: phi + i (r m / k) chi; chi lanes: chi_m - r / (k + 1) chi_(m + 1), the odd
                                    // register of the same lane for even m; for odd m the even part's next entry, one quad up
                                    // (or register ri + 1 of quad 0)
                                    const V rm = rk * (qd + (double)m0);
                                    V nr, ni;
                                    if constexpr (pr == 0) {
                                        nr = ri < ko ? Lr[LO<k>::v + ke + imin(ri, ko1 - 1)] : V(0.0);
                                        ni = ri < ko ? Li[LO<k>::v + ke + imin(ri, ko1 - 1)] : V(0.0);
                                    } else {
                                        const V hr = ri + 1 < ke ? Lr[LO<k>::v + imin(ri + 1, ke - 1)] : V(0.0);
                                        const V hi = ri + 1 < ke ? Li[LO<k>::v + imin(ri + 1, ke - 1)] : V(0.0);
                                        const I up = ((q + 1) & 3) * 16 + c;
                                        nr = B::bperm(B::sel(q == 0, hr, Lr[LO<k>::v + ri]), up);
                                        ni = B::bperm(B::sel(q == 0, hi, Li[LO<k>::v + ri]), up);
                                    }
                                    if constexpr (m0 + 7 > k) {
                                        const M has = m + 1 <= k;
                                        nr = B::sel(has, nr, V(0.0));
                                        ni = B::sel(has, ni, V(0.0));
                                    }
                                    const V yr = B::perm1(vr), yi = B::perm1(vi);
                                    vr = B::fma(-rk1, nr, B::fma(-rm, yi, vr));
                                    vi = B::fma(-rk1, ni, B::fma(rm, yr, vi));
                                }
                                const V t2 = B::fma(vr, vr, vi * vi);
                                if constexpr (m0 + 6 <= k) {
                                    const V nt = B::lds(T.Lt, m + mnh(k - 1));
                                    lsum = B::fma(t2 * nt, nt, lsum);
                                } else {
                                    const M ok = m <= k;
                                    const V nt = B::sel(ok, B::lds(T.Lt, B::mini(m, k) + mnh(k - 1)), V(0.0));
                                    lsum = B::fma(t2 * nt, nt, lsum);
                                }
                            };
                            sfor<0, ke>([&](auto EE) { term(std::integral_constant<int, 0>(), EE); });
                            sfor<0, ko>([&](auto OO) { term(std::integral_constant<int, 1>(), OO); });
                            const V tl = B::sqrt(B::quadsum(lsum));
                            const double cl = SQ3 * rl_nm1 * nm1_f_inv * iN;
                            eps_l = phi_of(tl) * (X.kind == 3 ? cl : cl * X.r_l * ik);
                            if constexpr (LH) eps_l = eps_l + chi_of(tl) * (cl * X.r_l);
                        }
                    }
                    pass = (eps_mp <= X.limit) && (eps_mp + eps_l * 2.0 <= X.limit);
                }
                const M newly = active && pass;
                Pl = B::seli(newly, I(k - 1 + X.BE), Pl);
                succ = succ || newly;
                const M addk = active && (!pass || X.BE != 0);
                active = active && !pass;
                sfor<0, ke>([&](auto EE) {
                    constexpr int e = decltype(EE)::value;
                    MEr[e] = B::sel(addk, MEr[e], V(0.0));
                    MEi[e] = B::sel(addk, MEi[e], V(0.0));
                });
                sfor<0, ko>([&](auto OO) {
                    constexpr int o = decltype(OO)::value;
                    MOr[o] = B::sel(addk, MOr[o], V(0.0));
                    MOi[o] = B::sel(addk, MOi[o], V(0.0));
                });
            }
            // ---- M_k into the other degrees: L_j += F(j + k) M_k
            sfor<0, CAP + 1>([&](auto JJ) {
                constexpr int j = decltype(JJ)::value;
                if constexpr (j != k) {
                    const V fac = B::lds(W.F, fb + (k + j));
                    sfor<0, imin(KE(j), ke)>([&](auto EE) {
                        constexpr int e = decltype(EE)::value;
                        Lr[LO<j>::v + e] = B::fma(fac, MEr[e], Lr[LO<j>::v + e]);
                        Li[LO<j>::v + e] = B::fma(fac, MEi[e], Li[LO<j>::v + e]);
                    });
                    sfor<0, imin(KO(j), ko)>([&](auto OO) {
                        constexpr int o = decltype(OO)::value;
                        Lr[LO<j>::v + KE(j) + o] = B::fma(fac, MOr[o], Lr[LO<j>::v + KE(j) + o]);
                        Li[LO<j>::v + KE(j) + o] = B::fma(fac, MOi[o], Li[LO<j>::v + KE(j) + o]);
                    });
                }
            });
            // ---- running products for the next degree
            if constexpr (k >= 1) {
                rmi_np2 = rmi_np2 * rmi;
                rl_nm1 = rl_nm1 * X.r_l;
            }
            mp_pow = pw_phi;
            running = !err || B::any(active);
        });

        // ---- Lamb-Helmholtz transform of the translated locals (transform_lh_local!, src/translate.jl:98-142)
        if constexpr (LH) {
            const V rphi = B::sel(chi_lane, V(0.0), r);
            sfor<0, CAP + 1>([&](auto NN) {
                constexpr int n = decltype(NN)::value;
                if (n > kdone) return;
                constexpr int ke = KE(n), ko = KO(n);
                const I q = B::opaque(q0);
                // phi += i (r m / n) chi on the phi lanes; chi -= r / (n + 1) chi_(n+1) on the chi lanes below
                // the interaction's order. Per-lane coefficients, zero where a term does not apply (x + 0 y = x).
                const V r_n = rphi * (1.0 / (n > 0 ? n : 1)), qd = B::tod(q * 2);
                const V bco = B::sel(chi_lane && (Pl > n), r * (-1.0 / (n + 1)), V(0.0));
                auto lh = [&](auto par, auto RI) {
                    constexpr int pr = decltype(par)::value, ri = decltype(RI)::value;
                    constexpr int at = LOFF(n) + (pr ? ke : 0) + ri;
                    constexpr int nn = imin(n + 1, CAP);
                    constexpr int at1 = LOFF(nn) + (pr ? KE(nn) : 0) + ri;
                    V xr = Lr[at], xi = Li[at];
                    if constexpr (n > 0) {
                        const V rm = r_n * (qd + (double)(8 * ri + pr));
                        const V yr = B::perm1(xr), yi = B::perm1(xi);
                        xr = B::fma(-rm, yi, xr);
                        xi = B::fma(rm, yr, xi);
                    }
                    if constexpr (n < CAP) {
                        xr = B::fma(bco, Lr[at1], xr);
                        xi = B::fma(bco, Li[at1], xi);
                    }
                    Lr[at] = xr;
                    Li[at] = xi;
                };
                sfor<0, ke>([&](auto EE) { lh(std::integral_constant<int, 0>(), EE); });
                sfor<0, ko>([&](auto OO) { lh(std::integral_constant<int, 1>(), OO); });
            });
        }

        // ---- back rotation (rotate_local_y!, eta magnitudes), back z-rotation, sum over slots
        sfor<0, CAP + 1>([&](auto NN) {
            constexpr int n = decltype(NN)::value;
            if (n > kdone) return;
            B::sched_fence();
            constexpr int ke = KE(n), ko = KO(n), ke1 = imax(ke, 1), ko1 = imax(ko, 1);
            const I c = B::opaque(c0) & 15, q = B::opaque(q0) & 3;
            const I s = LH ? c >> 1 : c, pot = LH ? c & 1 : I(0);
            const I sb2 = s * (NS * 2), q2 = q * 2;
            const M on = Pl >= n;
            V uEr[ke1], uEi[ke1], uOr[ko1], uOi[ko1], oEr[ke1], oEi[ke1], oOr[ko1], oOi[ko1];
            auto scale = [&](auto par, auto RI, V& ur, V& ui) {
                constexpr int pr = decltype(par)::value, ri = decltype(RI)::value, m0 = 8 * ri + pr;
                constexpr int at = LO<n>::v + (pr ? ke : 0) + ri;
                V g = B::lds(T.ein, q2 + (m0 + mnh(n - 1)));
                if (err) g = B::sel(on, g, V(0.0));
                ur = g * Lr[at];
                ui = g * Li[at];
                if constexpr (m0 == 0) ur = ur * B::sel(q == 0, V(0.5), V(1.0));
            };
            sfor<0, ke>([&](auto EE) { scale(std::integral_constant<int, 0>(), EE, uEr[decltype(EE)::value], uEi[decltype(EE)::value]); });
            sfor<0, ko>([&](auto OO) { scale(std::integral_constant<int, 1>(), OO, uOr[decltype(OO)::value], uOi[decltype(OO)::value]); });
            if constexpr (ko == 0) { uOr[0] = V(0.0); uOi[0] = V(0.0); }
            rotate<n>(T, W, T.eoh, -1.0, c, q, s, uEr, uEi, uOr, uOi, oEr, oEi, oOr, oOi);
            auto store = [&](auto par, auto RI, const V& xr, const V& xi) {
                constexpr int m0 = 8 * decltype(RI)::value + decltype(par)::value;
                const I m = q2 + m0;
                const I ei = sb2 + m * 2;
                const V er = B::lds(W.eim, ei), eimg = B::lds(W.eim, ei + 1);
                // back_rotate_z! (src/rotate.jl:584-616)
                const V zr = B::template slotsum<NP>(B::fma(xr, er, xi * eimg));
                const V zi = B::template slotsum<NP>(B::fma(xi, er, -(xr * eimg)));
                const M w = (c < NP) && (m0 + 6 <= n ? M(true) : (m <= n));
                const I at = B::seli(w, m * NC + pot * 2, I(0)) + mnh(n - 1) * NC;
                B::lds_add(W.acc, at, zr, w);
                B::lds_add(W.acc, at + 1, zi, w);
            };
            sfor<0, ke>([&](auto EE) { store(std::integral_constant<int, 0>(), EE, oEr[decltype(EE)::value], oEi[decltype(EE)::value]); });
            sfor<0, ko>([&](auto OO) { store(std::integral_constant<int, 1>(), OO, oOr[decltype(OO)::value], oOi[decltype(OO)::value]); });
        });
        B::wsync();

        // ---- orders and flags
        const M wr = valid && (q0 == 0) && (pot0 == 0);
        B::sti(Bt.orders, B::seli(wr, li, I(0)), Pl, wr);
        const int mx = B::maxi(Pl, valid);
        if (mx > pmax) pmax = mx;
        if (!B::all(succ || !valid)) okflag = 0;
    }
};

}  // namespace mx
}  // namespace fmmhip
