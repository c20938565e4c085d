// Lane-by-lane CPU emulation of the matrix-core M2L engine (fastmultipole_amd/csrc/m2l_mx.hpp).
// Test infrastructure: the engine's source is compiled here with a backend whose per-lane values are
// arrays of 64 doubles, whose cross-lane moves are permutations of those arrays, and whose MFMA is
// v_mfma_f64_4x4x4_4b_f64's product with its lane layout (four blocks; lane l supplies A(l % 4, l / 16) and
// B(l / 16, l % 4) of block (l % 16) / 4 and holds its D(l / 16, l % 4)). The tables and the wavefront's
// scratch lie in one array in the order of the GPU's LDS, NaN where nothing has been written, so a read of
// anything but a written double shows. tests/test_m2l_mx_emul.py compares the result with the
// oracle's multipole_to_local.
#include <array>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <limits>
#include <vector>

#include "../fastmultipole_amd/csrc/m2l_mx.hpp"
#include "../fastmultipole_amd/csrc/tables_host.hpp"

namespace {

constexpr int W = 64;

struct CpuB {
    struct M {
        std::array<bool, W> v;
        M() { v.fill(false); }
        M(bool b) { v.fill(b); }
    };
    struct I {
        std::array<int64_t, W> v;
        I() { v.fill(0); }
        I(int64_t x) { v.fill(x); }
    };
    struct V {
        std::array<double, W> v;
        V() { v.fill(0.0); }
        V(double x) { v.fill(x); }
    };
    struct PV {
        std::array<const double*, W> v;
    };

    static I lane() {
        I r;
        for (int i = 0; i < W; ++i) r.v[i] = i;
        return r;
    }
    static V sel(const M& m, const V& a, const V& b) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = m.v[i] ? a.v[i] : b.v[i];
        return r;
    }
    static I seli(const M& m, const I& a, const I& b) {
        I r;
        for (int i = 0; i < W; ++i) r.v[i] = m.v[i] ? a.v[i] : b.v[i];
        return r;
    }
    static I opaque(const I& a) { return a; }
    static void sched_fence() {}
    static I mini(const I& a, int b) {
        I r;
        for (int i = 0; i < W; ++i) r.v[i] = a.v[i] < b ? a.v[i] : b;
        return r;
    }
    static V fabs(const V& a) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = std::fabs(a.v[i]);
        return r;
    }
    static V sqrt(const V& a) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = std::sqrt(a.v[i]);
        return r;
    }
    static V fma(const V& a, const V& b, const V& c) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = std::fma(a.v[i], b.v[i], c.v[i]);
        return r;
    }
    static V tod(const I& a) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = (double)a.v[i];
        return r;
    }
    static V from(const V& a, int (*src)(int)) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = a.v[src(i)];
        return r;
    }
    static V perm1(const V& a) { return from(a, [](int i) { return i ^ 1; }); }
    static V bperm(const V& a, const I& src) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = a.v[src.v[i] & 63];
        return r;
    }
    static V quadsum(const V& a) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = (a.v[i] + a.v[i ^ 16]) + (a.v[i ^ 32] + a.v[i ^ 48]);
        return r;
    }
    template <int NC>
    static V slotsum(const V& a) {
        V r;
        for (int i = 0; i < W; ++i) {
            const int row = i & ~15, c = i & 15;
            double s = 0.0;
            for (int j = c % NC; j < 16; j += NC) s += a.v[row + j];
            r.v[i] = s;
        }
        return r;
    }
    template <int NC, int j>
    static V qbcast(const V& a) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = a.v[(i & ~(NC - 1)) + j];
        return r;
    }
    static V mfma4(const V& a, const V& b, const V& d) {
        V r;
        for (int l = 0; l < W; ++l) {
            const int i = l / 16, blk = (l % 16) / 4;   // D(i, j) of block blk: A of the block's lanes with l % 4 = i
            double s = d.v[l];
            for (int k = 0; k < 4; ++k) s = std::fma(a.v[16 * k + 4 * blk + i], b.v[16 * k + l % 16], s);
            r.v[l] = s;
        }
        return r;
    }
    static bool any(const M& m) {
        for (int i = 0; i < W; ++i)
            if (m.v[i]) return true;
        return false;
    }
    static bool all(const M& m) {
        for (int i = 0; i < W; ++i)
            if (!m.v[i]) return false;
        return true;
    }
    static int maxi(const I& a, const M& m) {
        int64_t r = INT32_MIN;
        for (int i = 0; i < W; ++i)
            if (m.v[i] && a.v[i] > r) r = a.v[i];
        return (int)r;
    }
    static V gld(const double* p, const I& idx, const M& ok) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = ok.v[i] ? p[idx.v[i]] : 0.0;
        return r;
    }
    static I gldi(const int32_t* p, const I& idx, const M& ok) {
        I r;
        for (int i = 0; i < W; ++i) r.v[i] = ok.v[i] ? p[idx.v[i]] : 0;
        return r;
    }
    static PV ptr(const double* base, const I& js, int64_t stride) {
        PV r;
        for (int i = 0; i < W; ++i) r.v[i] = base + js.v[i] * stride;
        return r;
    }
    static V gldp(const PV& p, const I& idx) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = p.v[i][idx.v[i]];
        return r;
    }
    static V lds(const double* p, const I& idx) {
        V r;
        for (int i = 0; i < W; ++i) r.v[i] = p[idx.v[i]];
        return r;
    }
    static void lds_st(double* p, const I& idx, const V& x, const M& ok) {
        for (int i = 0; i < W; ++i)
            if (ok.v[i]) p[idx.v[i]] = x.v[i];
    }
    static void lds_add(double* p, const I& idx, const V& x, const M& ok) {
        for (int i = 0; i < W; ++i)
            if (ok.v[i]) p[idx.v[i]] += x.v[i];
    }
    static void sti(int32_t* p, const I& idx, const I& x, const M& ok) {
        for (int i = 0; i < W; ++i)
            if (ok.v[i]) p[idx.v[i]] = (int32_t)x.v[i];
    }
    static void wsync() {}
};

// ---- element-wise operators of the emulated lane types
#define MX_BIN(T, R, op)                                                                     \
    inline R operator op(const T& a, const T& b) {                                           \
        R r;                                                                                 \
        for (int i = 0; i < W; ++i) r.v[i] = a.v[i] op b.v[i];                               \
        return r;                                                                            \
    }
#define MX_BIN_S(T, S, R, op)                                                                \
    inline R operator op(const T& a, S b) {                                                  \
        R r;                                                                                 \
        for (int i = 0; i < W; ++i) r.v[i] = a.v[i] op b;                                    \
        return r;                                                                            \
    }                                                                                        \
    inline R operator op(S a, const T& b) {                                                  \
        R r;                                                                                 \
        for (int i = 0; i < W; ++i) r.v[i] = a op b.v[i];                                    \
        return r;                                                                            \
    }
using V = CpuB::V;
using I = CpuB::I;
using M = CpuB::M;
MX_BIN(V, V, +) MX_BIN(V, V, -) MX_BIN(V, V, *) MX_BIN(V, V, /)
MX_BIN_S(V, double, V, +) MX_BIN_S(V, double, V, -) MX_BIN_S(V, double, V, *) MX_BIN_S(V, double, V, /)
MX_BIN(V, M, <) MX_BIN(V, M, <=) MX_BIN(V, M, >) MX_BIN(V, M, >=)
MX_BIN_S(V, double, M, <) MX_BIN_S(V, double, M, <=) MX_BIN_S(V, double, M, >) MX_BIN_S(V, double, M, >=)
MX_BIN(I, I, +) MX_BIN(I, I, -) MX_BIN(I, I, *) MX_BIN(I, I, /) MX_BIN(I, I, %) MX_BIN(I, I, &)
MX_BIN_S(I, int, I, +) MX_BIN_S(I, int, I, -) MX_BIN_S(I, int, I, *) MX_BIN_S(I, int, I, /) MX_BIN_S(I, int, I, %)
MX_BIN_S(I, int, I, &) MX_BIN_S(I, int, I, >>)
MX_BIN(I, M, <) MX_BIN(I, M, <=) MX_BIN(I, M, >) MX_BIN(I, M, >=) MX_BIN(I, M, ==) MX_BIN(I, M, !=)
MX_BIN_S(I, int, M, <) MX_BIN_S(I, int, M, <=) MX_BIN_S(I, int, M, >) MX_BIN_S(I, int, M, >=) MX_BIN_S(I, int, M, ==)
MX_BIN_S(I, int, M, !=)
MX_BIN(M, M, &&) MX_BIN(M, M, ||) MX_BIN(M, M, !=) MX_BIN(M, M, ==)
inline V operator-(const V& a) {
    V r;
    for (int i = 0; i < W; ++i) r.v[i] = -a.v[i];
    return r;
}
inline M operator!(const M& a) {
    M r;
    for (int i = 0; i < W; ++i) r.v[i] = !a.v[i];
    return r;
}
inline M operator&&(const M& a, bool b) { return a && M(b); }
inline M operator||(const M& a, bool b) { return a || M(b); }

template <int CAP>
void fill_tables(const fmmhip::mx::Tabs& T) {
    using namespace fmmhip::tabh;
    std::vector<double> Hs, z, e, Mt, Lt;
    host_Hs(Hs, CAP);
    host_mags(z, e, CAP);
    host_power_norms(Mt, Lt, CAP);
    const std::vector<double> A = host_dense_A(Hs, CAP), tf = host_test_factorials(CAP);
    for (int n = 0, i = 0, at = 0; n <= CAP; ++n) {
        const int len = fmmhip::mx::PBASE(n + 1) - fmmhip::mx::PBASE(n);
        for (int t = 0; t < len; ++t) T.A[at + t] = fmmhip::mx::padded(A.data(), n, t);
        at += len;
        for (int m = 0; m <= n; ++m, ++i) {
            const int b = len_Ts(n - 1);
            T.zin[i] = z[b + m];
            T.zoh[i] = 0.5 * z[b + m * (n + 1)];
            T.ein[i] = e[b + m];
            T.eoh[i] = 0.5 * e[b + m * (n + 1)];
            T.Mt[i] = Mt[i];
            T.Lt[i] = Lt[i];
        }
        T.tf[2 * n] = tf[2 * n];
        T.tf[2 * n + 1] = tf[2 * n + 1];
        T.i0[2 * n] = 1.0 / Mt[nh(n - 1)];
        T.i0[2 * n + 1] = 1.0 / Lt[nh(n - 1)];
    }
}

template <int CAP, bool LH, bool ERR>
int run(int P, int kind, int relative, double eps, int BE, const double* tg, int nsrc, const double* sg,
        const double* sex, int64_t he4, const int32_t* perm, double* out, int32_t* orders, int* pmax, int* ok) {
    using E = fmmhip::mx::Engine<CpuB, CAP, LH, ERR>;
    // the GPU's LDS of a workgroup of one wavefront, and as much again of what another wavefront has not written yet
    constexpr int shared = fmmhip::mx::shared_doubles<CAP>(), wave = fmmhip::mx::wave_doubles<CAP, LH>();
    std::vector<double> lds(shared + 2 * wave, std::numeric_limits<double>::quiet_NaN());
    const fmmhip::mx::Tabs T = fmmhip::mx::tabs<CAP>(lds.data());
    fill_tables<CAP>(T);
    const fmmhip::mx::Wave Wv = fmmhip::mx::wave<CAP, LH>(lds.data() + shared);
    double* acc = Wv.acc;
    for (int i = 0; i < E::NC * fmmhip::mx::mnh(CAP); ++i) acc[i] = 0.0;
    fmmhip::mx::Box X;
    for (int d = 0; d < 3; ++d) { X.tc[d] = tg[3 + d]; X.tbox[d] = tg[11 + d]; }
    X.r_l = tg[7];
    const double e2 = relative ? tg[14] * eps : eps;
    X.limit = e2 * 4 * 3.141592653589793;
    X.P = P; X.kind = kind; X.BE = BE;
    // source centres as the branch array (stride 15, source centre at offset 0)
    std::vector<int32_t> ms(nsrc);
    for (int i = 0; i < nsrc; ++i) ms[i] = i;
    int pm = 0, okf = 1;
    for (int b0 = 0; b0 < nsrc; b0 += E::BP)
        E::batch(T, Wv, X, fmmhip::mx::Batch{ms.data(), perm, b0, std::min(E::BP, nsrc - b0), orders}, sg, 15, 0, sex, he4,
                 pm, okf);
    const int H = fmmhip::mx::mnh(P);
    for (int i = 0; i < H; ++i)
        for (int c = 0; c < 4; ++c) out[4 * i + c] = c < E::NC ? acc[i * E::NC + c] : 0.0;
    *pmax = pm;
    *ok = okf;
    return 0;
}

}  // namespace

// perm: processing order of the list (null: list order)
extern "C" int mx_emul_m2l(int LH, int cap, int P, int kind, int relative, double eps, int BE, const double* tgeom,
                           int nsrc, const double* sgeoms, const double* sexp, int64_t he4, const int32_t* perm, double* out,
                           int32_t* orders, int* pmax, int* ok) {
    constexpr int K = MX_CAP;   // one order cap per library (compiled side by side)
    if (cap != K) return -1;
#define MX_RUN(L, E) run<K, L, E>(P, kind, relative, eps, BE, tgeom, nsrc, sgeoms, sexp, he4, perm, out, orders, pmax, ok)
    return kind ? (LH ? MX_RUN(true, true) : MX_RUN(false, true)) : (LH ? MX_RUN(true, false) : MX_RUN(false, false));
#undef MX_RUN
}
