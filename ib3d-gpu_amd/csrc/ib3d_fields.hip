// ib3d_fields.hip -- momentum predictor, boundary conditions, projection
// corrections and the steady-state check (subNavierStokes.f90:622-1122,
// subBoundaryConditions.f90:137-217, subPcorVcor.f90:2-142).
//
// The reference iterates gathered fluid lists; each fluid cell's update is
// independent of the others, so these kernels walk the padded grid in
// Fortran order (coalesced, i fastest) and test the int8 tag instead.
// Arithmetic is written operand for operand like the reference (built with
// -ffp-contract=off, correctly rounded division), so results are bitwise.
// The predictor takes its index-only sub-expressions from per-axis tables
// computed on the host in the same operations, and divides field values
// through correctly rounded reciprocals (dv below), which is also exact.
#include "ib3d_internal.h"

#include <type_traits>

namespace ib3d {

struct Tabs {
    const double *t[6];
    int tn[6];
};

enum { UU = 0, VV = 1, WW = 2, UV = 3, VU = 4, WU = 5 };


// Per-axis momentum tables, quantity-major with n+3 entries per quantity.
// Each entry is a sub-expression of the momentum formula that depends on
// one grid index only, evaluated once on the host in the same IEEE
// operations as the formula (so reading it changes no bit), together with
// the correctly rounded reciprocal of every denominator that divides a
// field value.  "S" quantities serve the velocity component staggered along
// the axis (u along x), "C" the two components across it.
enum MomQ {
    M_AS,        // d(i+1) / (d(i) + d(i+1)): face interpolation weight
    M_CS,        // 2 / (d(i) + d(i+1)): second-difference weight
    M_D1, M_RD1, // d(i+1) and 1/d(i+1)
    M_D0, M_RD0, // d(i) and 1/d(i)
    M_KS1, M_RKS1, M_KS2, M_RKS2,  // face table: t5*d(i+1), (2 t11)*d(i), reciprocals
    M_US,        // 7 upwind factors at den = d(i+1), r = d(i)/d(i+1)
    M_CC = M_US + 7,               // 2 / (0.5 ((d(i)+d(i+1)) + (d(i)+d(i-1))))
    M_H1, M_RH1, // h1 = 0.5 (d(i) + d(i+1)) and 1/h1
    M_H0, M_RH0, // h0 = 0.5 (d(i) + d(i-1)) and 1/h0
    M_KC1, M_RKC1, M_KC2, M_RKC2,  // centre table: t5*h1, (2 t11)*h0, reciprocals
    M_UC,        // 7 upwind factors at den = h1, r = h0/h1
    M_NQ = M_UC + 7
};

typedef __attribute__((address_space(4))) double CDouble;

struct MomTabs {
    const double *m[3];    // quantity-major tables (x axis: lanes read consecutive entries)
    int mn[3];
    const double *rec[3];  // y, z axes: one kMomRec-double record per index (see below)
};

// y and z records: the M_NQ quantities, then the face (staggered) and the
// centre (across) convection coefficients of that axis.  A wave shares one
// j and one k, so a record arrives through a few wide scalar loads.
static constexpr int kMomRec = 64, kRecS = M_NQ, kRecC = M_NQ + 12;
static_assert(kRecC + 12 <= kMomRec, "momentum record overflow");

// a / b, correctly rounded, from y = RN(1/b) and two FMA corrections of
// a*y.  The first brings the quotient within one ulp; by Markstein's
// theorem (y within half an ulp of 1/b, quotient within one ulp) the
// remainder a - b*q is then exact and the second correction rounds
// correctly.  The host enables this only when every denominator lies in
// [2^-64, 2^64].
//   kDivide   the division instruction
//   kChecked  numerators outside [2^-900, 2^900] (zeros, NaN and infinities
//             among them) use the division instruction, so no intermediate
//             leaves the normal range and signed zeros come out as from a / b
//   kCheckedAlone  the same, its steps not shared with the forms below: the
//             compiler then fits k_momentum_rows into 96 registers (with kChecked it
//             spills 56 bytes, 798 us at 256x192x192 instead of 652); k_momentum is
//             10% slower with it
//   kPlain    the caller knows that a is zero or in that range and b > 0
//   kPlainNeg the same, b < 0
// The remainder of a zero is +0 and its quotient's sign that of a*y: the
// correction adds -(b*q - a) * y for b > 0 and (a - b*q) * y for b < 0, both -0
// there, so the zero keeps its sign.
enum Quot { kDivide, kChecked, kCheckedAlone, kPlain, kPlainNeg };
template <Quot Q>
__device__ __forceinline__ double dv(double a, double b, double y) {
    if (Q == kDivide) return a / b;
    if (Q == kChecked || Q == kCheckedAlone) {
        const double m = fabs(a);
        if (!(m >= 0x1p-900 && m <= 0x1p900)) return a / b;
        if (Q == kCheckedAlone) {
            const double q = fma(fma(-b, a * y, a), y, a * y);
            return fma(fma(-b, q, a), y, q);
        }
    }
    double q = a * y;
    if (Q == kPlain) {
        q = fma(-fma(b, q, -a), y, q);
        return fma(-fma(b, q, -a), y, q);
    }
    q = fma(fma(-b, q, a), y, q);
    return fma(fma(-b, q, a), y, q);
}

// Whether a velocity is zero or of a magnitude in [2^-200, 2^200].  Of such
// velocities (multiples of 2^-252) and of weights that are zero or in
// [2^-64, 2^64], every numerator of the predictor is zero or in [2^-900,
// 2^900]: a difference is a multiple of 2^-252; an interpolated velocity adds a
// product of at least 2^-316, a multiple of 2^-368, and halves: a multiple of
// 2^-369; a stencil sum is a multiple of 2^-316; so a convection numerator is
// zero or at least 2^-685, and below 2^470.
__device__ __forceinline__ bool plain_velocity(double x) {
    const double m = fabs(x);
    return m == 0.0 || (m >= 0x1p-200 && m <= 0x1p200);
}

// 3rd-order Kawamura-Kuwahara convection term (subNavierStokes.f90:812-831);
// dA = t5*dA', dB = (2 t11)*dB' come from the axis table with their reciprocals
// (coefficient c of the stencil: tc(c))
template <Quot Q, class TCOEF>
__device__ __forceinline__ double kk3(TCOEF tc, double vel, double f2, double f1, double f0, double fm1, double fm2,
                                      double dA, double rA, double dB, double rB) {
#define TC(c) tc(c)
    const double sa = (((TC(0) * f2 + TC(1) * f1) + TC(2) * f0) + TC(3) * fm1) + TC(4) * fm2;
    const double sk = (((TC(6) * f2 + TC(7) * f1) + TC(8) * f0) + TC(9) * fm1) + TC(10) * fm2;
#undef TC
    return dv<Q == kPlain ? kPlainNeg : Q>(vel * sa, dA, rA) + dv<Q>(fabs(vel) * sk, dB, rB);
}

// non-uniform 1st-order upwind term (subNavierStokes.f90:847-866), al = 1;
// g[0..6*n] = -1/(r(r+1)), 1-1/r, r/(r+1), 2/(r(r+1)), 2/r, 2/(r+1), 1/(2 den)
template <Quot Q, class PT>
__device__ __forceinline__ double up1(PT g, int n, double vel, double den, double rden, double fm,
                                      double f0, double fp) {
    const double t1 = ((g[0] * fm - g[n] * f0) + g[2 * n] * fp);
    const double t2 = (g[3 * n] * fm - g[4 * n] * f0) + g[5 * n] * fp;
    return dv<Q>(vel, den, rden) * t1 - (fabs(vel) * g[6 * n]) * t2;
}

// Where the predictor reads u, v, w at offset (a, b, d) from its cell, and
// how it addresses the other arrays of the padded grid (at<a, b, d>(base):
// the element at that offset).
// GlobalFields: straight from the padded fields in HBM, 64-bit indices.
struct GlobalFields {
    const double *__restrict__ u, *__restrict__ v, *__restrict__ w;
    int64_t c, sx, sxy;
    template <int a, int b, int d> __device__ __forceinline__ double U() const { return u[c + a + b * sx + d * sxy]; }
    template <int a, int b, int d> __device__ __forceinline__ double V() const { return v[c + a + b * sx + d * sxy]; }
    template <int a, int b, int d> __device__ __forceinline__ double W() const { return w[c + a + b * sx + d * sxy]; }
    template <int a, int b, int d, class T> __device__ __forceinline__ T &at(T *base) const {
        return base[c + a + b * sx + d * sxy];
    }
    __device__ __forceinline__ void split() const {}
};

// GlobalFields32: the same values through 32-bit byte offsets from the uniform
// array bases, one offset register per address instead of a 64-bit pair (fewer
// registers, one more wave per SIMD).  For grids whose FP64 fields span less than
// 4 GiB.
struct GlobalFields32 {
    const double *__restrict__ u, *__restrict__ v, *__restrict__ w;
    uint32_t c, sx, sxy;  // element offsets; c * 8 < 2^32
    template <int a, int b, int d, int S> __device__ __forceinline__ uint32_t off() const {
        return (c + (uint32_t)a + (uint32_t)b * sx + (uint32_t)d * sxy) * (uint32_t)S;
    }
    template <int a, int b, int d> __device__ __forceinline__ double U() const { return at<a, b, d>(u); }
    template <int a, int b, int d> __device__ __forceinline__ double V() const { return at<a, b, d>(v); }
    template <int a, int b, int d> __device__ __forceinline__ double W() const { return at<a, b, d>(w); }
    template <int a, int b, int d, class T> __device__ __forceinline__ T &at(T *base) const {
        typedef std::conditional_t<std::is_const_v<T>, const char, char> B;
        return *reinterpret_cast<T *>(reinterpret_cast<B *>(base) + off<a, b, d, (int)sizeof(T)>());
    }
    __device__ __forceinline__ void split() const {}
};

// TiledFields: planes k-1, k and k+1 from LDS tiles (row stride kTileS; v and w
// one and two tiles after u), the cell's own column at k-2 and k+2 from
// registers.
static constexpr int kMomTX = 64, kMomTY = 8;
static constexpr int kTileS = kMomTX + 4, kTileR = kMomTY + 4, kTile = kTileR * kTileS;
struct TiledFields {
    const double *below, *here, *above;   // LDS, at the cell
    double m2[3], p2[3];
    int64_t c, sx, sxy;
    template <int f, int a, int b, int d> __device__ __forceinline__ double value() const {
        static_assert((d >= -1 && d <= 1) || (a == 0 && b == 0), "off the tiles");
        if constexpr (d == -2) return m2[f];
        else if constexpr (d == 2) return p2[f];
        else return (d < 0 ? below : d > 0 ? above : here)[f * kTile + a + b * kTileS];
    }
    template <int a, int b, int d> __device__ __forceinline__ double U() const { return value<0, a, b, d>(); }
    template <int a, int b, int d> __device__ __forceinline__ double V() const { return value<1, a, b, d>(); }
    template <int a, int b, int d> __device__ __forceinline__ double W() const { return value<2, a, b, d>(); }
    template <int a, int b, int d, class T> __device__ __forceinline__ T &at(T *base) const {
        return base[c + a + b * sx + d * sxy];
    }
    // the three components are scheduled one after the other: their values
    // come from LDS, so loading them late costs little, and keeping the
    // components apart keeps the register count down
    __device__ __forceinline__ void split() const { __builtin_amdgcn_sched_barrier(0); }
};

// The x-axis tables of a cell's column: quantity q of MomTabs (not the upwind
// factors), coefficient c of the face and the centre convection table, and the
// upwind factors (read near walls and bodies only) as a strided run.
// GlobalColumns: each from its global table.
struct GlobalColumns {
    const double *__restrict__ m, *__restrict__ tf, *__restrict__ tc;   // at the column
    int mn, nf, nc;
    __device__ __forceinline__ double q(int k) const { return m[k * mn]; }
    __device__ __forceinline__ double face(int c) const { return tf[c * nf]; }
    __device__ __forceinline__ double cent(int c) const { return tc[c * nc]; }
    __device__ __forceinline__ const double *up(int k) const { return m + k * mn; }
};
__device__ __forceinline__ GlobalColumns columns(const Tabs &T, const MomTabs &M, int i) {
    return {M.m[0] + i, T.t[UU] + i, T.t[UV] + i, M.mn[0], T.tn[UU], T.tn[UV]};
}
// LdsColumns: a copy of a tile's columns in LDS, [quantity][column].
static constexpr int kColQ = 19, kColFace = kColQ, kColCent = kColQ + 10, kColN = kColQ + 20;
// row of quantity q in that copy, and the quantity of row r
__host__ __device__ constexpr int col_row(int q) { return q < M_US ? q : q == M_CC ? M_US : q - M_H1 + M_US + 1; }
__host__ __device__ constexpr int col_quantity(int r) { return r < M_US ? r : r == M_US ? M_CC : r - M_US - 1 + M_H1; }
static_assert(col_row(M_RKC2) == kColQ - 1 && col_quantity(kColQ - 1) == M_RKC2, "x-axis quantities kept in LDS");
struct LdsColumns {
    const double *t;                 // LDS, at the column
    const double *__restrict__ m;    // the global table, at the column
    int mn;
    __device__ __forceinline__ double q(int k) const { return t[col_row(k) * 64]; }
    __device__ __forceinline__ double face(int c) const { return t[(kColFace + (c < 5 ? c : c - 1)) * 64]; }
    __device__ __forceinline__ double cent(int c) const { return t[(kColCent + (c < 5 ? c : c - 1)) * 64]; }
    __device__ __forceinline__ const double *up(int k) const { return m + k * mn; }
};

// One fluid cell of the explicit predictor (subNavierStokes.f90:622-1122).
// The Kawamura-Kuwahara stencil applies away from the walls and from
// intercepted cells, the upwind stencil elsewhere.  F supplies the velocity
// values (GlobalFields or TiledFields: the same values, so the same bits), X the
// x-axis tables.
// INNER: the caller has found that the cell is fluid, that the Kawamura-Kuwahara
// stencil applies to every component and that the pressure differences pd are
// plain too, so the code has no branch.
template <Quot Q, bool INNER, class F, class XT>
__device__ __forceinline__ void momentum_cell(
    const F &A, const XT &X, const double (&pd)[3], int i, int j, int k, const double *__restrict__ p, const int8_t *__restrict__ cell,
    double *__restrict__ ut, double *__restrict__ vt, double *__restrict__ wt, double *__restrict__ ru,
    double *__restrict__ rv, double *__restrict__ rw, const MomTabs &M, int nx, int ny, int nz, double rev,
    double deltat) {
    if (!INNER && A.template at<0, 0, 0>(cell) != 0) return;
    constexpr Quot QP = INNER ? Q : Q == kPlain ? kChecked : Q;   // of the pressure differences
#define U(a, b, d) A.template U<a, b, d>()
#define V(a, b, d) A.template V<a, b, d>()
#define W(a, b, d) A.template W<a, b, d>()
#define P(a, b, d) A.template at<a, b, d>(p)
#define CL(a, b, d) A.template at<a, b, d>(cell)
#define AT(f) A.template at<0, 0, 0>(f)
    // the y and z records go through the constant address space: the kernel
    // never writes them, so uniform reads of them stay scalar loads even after
    // the stores of an earlier cell in the same thread
    const CDouble *ry = (const CDouble *)(M.rec[1] + (int64_t)j * kMomRec);
    const CDouble *rz = (const CDouble *)(M.rec[2] + (int64_t)k * kMomRec);
    const auto xface = [&](int c) { return X.face(c); };
    const auto xcent = [&](int c) { return X.cent(c); };
    const auto yface = [&](int c) { return ry[kRecS + c]; };
    const auto ycent = [&](int c) { return ry[kRecC + c]; };
    const auto zface = [&](int c) { return rz[kRecS + c]; };
    const auto zcent = [&](int c) { return rz[kRecC + c]; };
#define MX(k) X.q(k)
#define MY(q) ry[q]
#define MZ(q) rz[q]
    // each component's differences and pressure gradient are formed inside
    // its own block, so that none of them stays live across another
    // component
    const bool no_ib = INNER || (CL(1, 0, 0) != 2 && CL(-1, 0, 0) != 2 && CL(0, 1, 0) != 2 && CL(0, -1, 0) != 2 &&
                                 CL(0, 0, 1) != 2 && CL(0, 0, -1) != 2);
    const int mx = X.mn, my = 1, mz = 1;

    // U momentum (subNavierStokes.f90:792-897)
    {
        const double u22 = U(-1, 0, 0) - U(0, 0, 0), u4 = U(0, 0, 0) - U(1, 0, 0);
        const double u6 = U(0, -1, 0) - U(0, 0, 0), u8 = U(0, 0, 0) - U(0, 1, 0);
        const double u10 = U(0, 0, -1) - U(0, 0, 0), u12 = U(0, 0, 0) - U(0, 0, 1);
        const double dpdx = dv<QP>(INNER ? pd[0] : P(0, 0, 0) - P(1, 0, 0), MX(M_H1), MX(M_RH1));
        const double ax = MX(M_AS);
        const double vu_e = V(1, 0, 0) + ax * (V(0, 0, 0) - V(1, 0, 0));
        const double vu_w = V(1, -1, 0) + ax * (V(0, -1, 0) - V(1, -1, 0));
        const double v_in_um = 0.5 * (vu_e + vu_w);
        const double wu_n = W(1, 0, 0) + ax * (W(0, 0, 0) - W(1, 0, 0));
        const double wu_s = W(1, 0, -1) + ax * (W(0, 0, -1) - W(1, 0, -1));
        const double w_in_um = 0.5 * (wu_n + wu_s);
        double a, b, d;
        if (INNER || (i != 2 && i < nx && j != 2 && j < ny + 1 && k != 2 && k < nz + 1 && no_ib)) {
            const double uc = U(0, 0, 0);
            a = kk3<Q>(xface, uc, U(2, 0, 0), U(1, 0, 0), uc, U(-1, 0, 0), U(-2, 0, 0), MX(M_KS1), MX(M_RKS1),
                          MX(M_KS2), MX(M_RKS2));
            b = kk3<Q>(ycent, v_in_um, U(0, 2, 0), U(0, 1, 0), uc, U(0, -1, 0), U(0, -2, 0), MY(M_KC1),
                          MY(M_RKC1), MY(M_KC2), MY(M_RKC2));
            d = kk3<Q>(zcent, w_in_um, U(0, 0, 2), U(0, 0, 1), uc, U(0, 0, -1), U(0, 0, -2), MZ(M_KC1),
                          MZ(M_RKC1), MZ(M_KC2), MZ(M_RKC2));
        } else {
            a = up1<Q>(X.up(M_US), mx, U(0, 0, 0), MX(M_D1), MX(M_RD1), U(-1, 0, 0), U(0, 0, 0), U(1, 0, 0));
            b = up1<Q>(&MY(M_UC), my, v_in_um, MY(M_H1), MY(M_RH1), U(0, -1, 0), U(0, 0, 0), U(0, 1, 0));
            d = up1<Q>(&MZ(M_UC), mz, w_in_um, MZ(M_H1), MZ(M_RH1), U(0, 0, -1), U(0, 0, 0), U(0, 0, 1));
        }
        const double d2x = MX(M_CS) * (dv<Q>(-u4, MX(M_D1), MX(M_RD1)) + dv<Q>(u22, MX(M_D0), MX(M_RD0)));
        const double d2y = MY(M_CC) * (dv<Q>(-u8, MY(M_H1), MY(M_RH1)) + dv<Q>(u6, MY(M_H0), MY(M_RH0)));
        const double d2z = MZ(M_CC) * (dv<Q>(-u12, MZ(M_H1), MZ(M_RH1)) + dv<Q>(u10, MZ(M_H0), MZ(M_RH0)));
        const double xtt2 = rev * ((d2x + d2y) + d2z);
        const double res = ((-a - b) - d) + xtt2;
        AT(ut) = U(0, 0, 0) + deltat * (res + dpdx);
        AT(ru) = res;
    }
    A.split();
    // V momentum (subNavierStokes.f90:901-1006)
    {
        const double v4 = V(-1, 0, 0) - V(0, 0, 0), v6 = V(0, 0, 0) - V(1, 0, 0);
        const double v8 = V(0, -1, 0) - V(0, 0, 0), v10 = V(0, 0, 0) - V(0, 1, 0);
        const double v12 = V(0, 0, -1) - V(0, 0, 0), v14 = V(0, 0, 0) - V(0, 0, 1);
        const double dpdy = dv<QP>(INNER ? pd[1] : P(0, 0, 0) - P(0, 1, 0), MY(M_H1), MY(M_RH1));
        const double ay = MY(M_AS);
        const double uv_e = U(0, 1, 0) + ay * (U(0, 0, 0) - U(0, 1, 0));
        const double uv_w = U(-1, 1, 0) + ay * (U(-1, 0, 0) - U(-1, 1, 0));
        const double u_in_vm = 0.5 * (uv_e + uv_w);
        const double wv_n = W(0, 1, 0) + ay * (W(0, 0, 0) - W(0, 1, 0));
        const double wv_s = W(0, 1, -1) + ay * (W(0, 0, -1) - W(0, 1, -1));
        const double w_in_vm = 0.5 * (wv_n + wv_s);
        double a, b, d;
        if (INNER || (i != 2 && i < nx + 1 && j != 2 && j < ny && k != 2 && k < nz + 1 && no_ib)) {
            const double vc = V(0, 0, 0);
            a = kk3<Q>(xcent, u_in_vm, V(2, 0, 0), V(1, 0, 0), vc, V(-1, 0, 0), V(-2, 0, 0), MX(M_KC1),
                          MX(M_RKC1), MX(M_KC2), MX(M_RKC2));
            b = kk3<Q>(yface, vc, V(0, 2, 0), V(0, 1, 0), vc, V(0, -1, 0), V(0, -2, 0), MY(M_KS1), MY(M_RKS1),
                          MY(M_KS2), MY(M_RKS2));
            d = kk3<Q>(zcent, w_in_vm, V(0, 0, 2), V(0, 0, 1), vc, V(0, 0, -1), V(0, 0, -2), MZ(M_KC1),
                          MZ(M_RKC1), MZ(M_KC2), MZ(M_RKC2));
        } else {
            a = up1<Q>(X.up(M_UC), mx, u_in_vm, MX(M_H1), MX(M_RH1), V(-1, 0, 0), V(0, 0, 0), V(1, 0, 0));
            b = up1<Q>(&MY(M_US), my, V(0, 0, 0), MY(M_D1), MY(M_RD1), V(0, -1, 0), V(0, 0, 0), V(0, 1, 0));
            d = up1<Q>(&MZ(M_UC), mz, w_in_vm, MZ(M_H1), MZ(M_RH1), V(0, 0, -1), V(0, 0, 0), V(0, 0, 1));
        }
        const double d2x = MX(M_CC) * (dv<Q>(-v6, MX(M_H1), MX(M_RH1)) + dv<Q>(v4, MX(M_H0), MX(M_RH0)));
        const double d2y = MY(M_CS) * (dv<Q>(-v10, MY(M_D1), MY(M_RD1)) + dv<Q>(v8, MY(M_D0), MY(M_RD0)));
        const double d2z = MZ(M_CC) * (dv<Q>(-v14, MZ(M_H1), MZ(M_RH1)) + dv<Q>(v12, MZ(M_H0), MZ(M_RH0)));
        const double ytt2 = rev * ((d2x + d2y) + d2z);
        const double res = ((-a - b) - d) + ytt2;
        AT(vt) = V(0, 0, 0) + deltat * (res + dpdy);
        AT(rv) = res;
    }
    A.split();
    // W momentum (subNavierStokes.f90:1010-1116)
    {
        const double w6 = W(-1, 0, 0) - W(0, 0, 0), w8 = W(0, 0, 0) - W(1, 0, 0);
        const double w10 = W(0, -1, 0) - W(0, 0, 0), w12 = W(0, 0, 0) - W(0, 1, 0);
        const double w14 = W(0, 0, -1) - W(0, 0, 0), w16 = W(0, 0, 0) - W(0, 0, 1);
        const double dpdz = dv<QP>(INNER ? pd[2] : P(0, 0, 0) - P(0, 0, 1), MZ(M_H1), MZ(M_RH1));
        const double az = MZ(M_AS);
        const double uw_e = U(0, 0, 1) + az * (U(0, 0, 0) - U(0, 0, 1));
        const double uw_w = U(-1, 0, 1) + az * (U(-1, 0, 0) - U(-1, 0, 1));
        const double u_in_wm = 0.5 * (uw_e + uw_w);
        const double vw_n = V(0, 0, 1) + az * (V(0, 0, 0) - V(0, 0, 1));
        const double vw_s = V(0, -1, 1) + az * (V(0, -1, 0) - V(0, -1, 1));
        const double v_in_wm = 0.5 * (vw_n + vw_s);
        double a, b, d;
        if (INNER || (i != 2 && i < nx + 1 && j != 2 && j < ny + 1 && k != 2 && k < nz && no_ib)) {
            const double wc = W(0, 0, 0);
            a = kk3<Q>(xcent, u_in_wm, W(2, 0, 0), W(1, 0, 0), wc, W(-1, 0, 0), W(-2, 0, 0), MX(M_KC1),
                          MX(M_RKC1), MX(M_KC2), MX(M_RKC2));
            b = kk3<Q>(ycent, v_in_wm, W(0, 2, 0), W(0, 1, 0), wc, W(0, -1, 0), W(0, -2, 0), MY(M_KC1),
                          MY(M_RKC1), MY(M_KC2), MY(M_RKC2));
            d = kk3<Q>(zface, wc, W(0, 0, 2), W(0, 0, 1), wc, W(0, 0, -1), W(0, 0, -2), MZ(M_KS1), MZ(M_RKS1),
                          MZ(M_KS2), MZ(M_RKS2));
        } else {
            a = up1<Q>(X.up(M_UC), mx, u_in_wm, MX(M_H1), MX(M_RH1), W(-1, 0, 0), W(0, 0, 0), W(1, 0, 0));
            b = up1<Q>(&MY(M_UC), my, v_in_wm, MY(M_H1), MY(M_RH1), W(0, -1, 0), W(0, 0, 0), W(0, 1, 0));
            d = up1<Q>(&MZ(M_US), mz, W(0, 0, 0), MZ(M_D1), MZ(M_RD1), W(0, 0, -1), W(0, 0, 0), W(0, 0, 1));
        }
        const double d2x = MX(M_CC) * (dv<Q>(-w8, MX(M_H1), MX(M_RH1)) + dv<Q>(w6, MX(M_H0), MX(M_RH0)));
        const double d2y = MY(M_CC) * (dv<Q>(-w12, MY(M_H1), MY(M_RH1)) + dv<Q>(w10, MY(M_H0), MY(M_RH0)));
        const double d2z = MZ(M_CS) * (dv<Q>(-w16, MZ(M_D1), MZ(M_RD1)) + dv<Q>(w14, MZ(M_D0), MZ(M_RD0)));
        const double ztt2 = rev * ((d2x + d2y) + d2z);
        const double res = ((-a - b) - d) + ztt2;
        AT(wt) = W(0, 0, 0) + deltat * (res + dpdz);
        AT(rw) = res;
    }
#undef U
#undef V
#undef W
#undef P
#undef CL
#undef AT
#undef MX
#undef MY
#undef MZ
}

// Interior columns i in [3, nx-1], where the stencil choice depends on j, k
// and the tags only: a wave takes rows of 64 columns of one j and k, so their
// table entries come through scalar loads and the wall tests are scalar
// branches.  All rows (left == nullptr: one per wave), or the *n_left that
// k_momentum_lds has listed there.  The first `edge` workgroups take the wall
// columns i = 2, nx, nx+1 of every row, kept out of the interior waves so that
// those run one stencil branch.
static constexpr int kRestBlocks = 1024;   // for the listed rows (3072 of its 4096 waves run at once)
template <bool FAST>
__global__ void __launch_bounds__(256)
k_momentum(const double *__restrict__ u, const double *__restrict__ v, const double *__restrict__ w,
           const double *__restrict__ p, const int8_t *__restrict__ cell, double *__restrict__ ut,
           double *__restrict__ vt, double *__restrict__ wt, double *__restrict__ ru, double *__restrict__ rv,
           double *__restrict__ rw, const int *__restrict__ left, const int *__restrict__ n_left, Tabs T, MomTabs M,
           int nx, int ny, int nz, int edge, int tiles, double rev, double deltat) {
    const int64_t sx = nx + 2, sxy = sx * (ny + 2);
    const auto compute = [&](int i, int j, int k) {
        const GlobalFields A{u, v, w, (i - 1) + sx * (j - 1) + sxy * (k - 1), sx, sxy};
        momentum_cell<FAST ? kChecked : kDivide, false>(A, columns(T, M, i), {}, i, j, k, p, cell, ut, vt, wt, ru, rv,
                                                        rw, M, nx, ny, nz, rev, deltat);
    };
    if ((int)blockIdx.x < edge) {
        const int t = (int)blockIdx.x * 256 + (int)threadIdx.x;
        if (t >= 3 * ny * nz) return;
        const int s = t % 3, r = t / 3;
        if (s == 1 && nx < 3) return;   // i = nx is then column 2 again
        compute(s == 0 ? 2 : nx + s - 1, r % ny + 2, r / ny + 2);
        return;
    }
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(((int)blockIdx.x - edge) * 4 + (int)threadIdx.x / 64);
    const int waves = ((int)gridDim.x - edge) * 4, rows = left ? *n_left : tiles * ny * nz;
    for (int q = wave; q < rows; q += waves) {
        const int r = left ? left[q] : q;
        const int i = r % tiles * 64 + lane + 3;
        if (i <= nx - 1) compute(i, r / tiles % ny + 2, r / tiles / ny + 2);
    }
}

// The interior columns of a large grid, one wave per row, on their own: with the
// code for the wall columns beside them (k_momentum) the kernel needs 166 registers,
// three waves per SIMD.  With 32-bit offsets and the fast divisions this fits 96,
// five waves (the other forms need more and keep the compiler's choice).  A call
// at 256x192x192 652 us, by k_momentum alone 707.
template <bool FAST, bool OFF32>
__global__ void __launch_bounds__(256, (FAST && OFF32) ? 5 : 1)
k_momentum_rows(const double *__restrict__ u, const double *__restrict__ v, const double *__restrict__ w,
                const double *__restrict__ p, const int8_t *__restrict__ cell, double *__restrict__ ut,
                double *__restrict__ vt, double *__restrict__ wt, double *__restrict__ ru, double *__restrict__ rv,
                double *__restrict__ rw, Tabs T, MomTabs M, int nx, int ny, int nz, double rev, double deltat) {
    const int64_t sx = nx + 2, sxy = sx * (ny + 2);
    const int i = (int)blockIdx.x * 64 + (int)threadIdx.x + 3;
    const int j = __builtin_amdgcn_readfirstlane((int)(blockIdx.y * 4 + threadIdx.y)) + 2, k = (int)blockIdx.z + 2;
    if (j > ny + 1 || i > nx - 1) return;
    const int64_t c = (i - 1) + sx * (j - 1) + sxy * (k - 1);
    using Index = std::conditional_t<OFF32, uint32_t, int64_t>;
    const std::conditional_t<OFF32, GlobalFields32, GlobalFields> A{u, v, w, (Index)c, (Index)sx, (Index)sxy};
    momentum_cell<FAST ? kCheckedAlone : kDivide, false>(A, columns(T, M, i), {}, i, j, k, p, cell, ut, vt, wt, ru, rv,
                                                         rw, M, nx, ny, nz, rev, deltat);
}

// The same interior columns, a 64 x 8 tile of (i, j) marching through tz planes.
// Planes k-1, k, k+1 of u, v, w over the tile and a two-cell ring (the corners
// the cross terms reach included) and the x-axis tables of its columns lie in
// LDS.  What plane k+2 adds is loaded before plane k is computed and stored after
// it.
//
// Only rows (64 columns of one j and k) without a branch are computed: away from
// the walls, no cell of the workgroup's tile and ring in three planes other than
// fluid, every velocity staged so far and every pressure difference plain (the
// host has found the tables fit for it).  The others are listed in `left` for
// k_momentum.  With the general cell in this kernel the compiler spilled.
//
// Bounded by FP64 issue (486 of 692 vector instructions per row; 220 us of issue at
// 256 x 192 x 192) and latency at four waves per SIMD: 338 us there, 1.75 ms at
// 512 x 320 x 320 (3.55 before), and 66 and 405 us for the rows it leaves.  Reading
// every stencil value and table through the vector cache, 108 eight-byte loads per
// row that it serves at 16 clocks each, took 640 us; the tiles with a tested quotient
// each, and the general cell beside it, 410.
__global__ void __launch_bounds__(kMomTX * kMomTY, 4)
k_momentum_lds(const double *__restrict__ u, const double *__restrict__ v, const double *__restrict__ w,
               const double *__restrict__ p, const int8_t *__restrict__ cell, double *__restrict__ ut,
               double *__restrict__ vt, double *__restrict__ wt, double *__restrict__ ru, double *__restrict__ rv,
               double *__restrict__ rw, int *__restrict__ left, int *__restrict__ n_left, int *__restrict__ n_next, Tabs T,
               MomTabs M, int nx, int ny, int nz, int tz, double rev, double deltat) {
    __shared__ double tile[3][3 * kTile];
    __shared__ double xtab[kColN * kMomTX];
    __shared__ int odd;        // a velocity that is not plain has been staged
    __shared__ int solid[4];   // slot (plane - kb + 1) & 3: a cell that is not fluid lies in its tile or ring
    const auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
    const int tx = (int)threadIdx.x, ty = (int)threadIdx.y, tid = ty * kMomTX + tx;
    const int i0 = 3 + (int)blockIdx.x * kMomTX, j0 = 2 + (int)blockIdx.y * kMomTY;
    const int i = i0 + tx;
    const int j = __builtin_amdgcn_readfirstlane(j0 + ty);
    const int kb = 2 + (int)blockIdx.z * tz, ke = min(kb + tz, nz + 2);
    const int64_t sx = nx + 2, sxy = sx * (ny + 2);
    const bool mine_in = i <= nx + 2 && j <= ny + 2;   // (i, j) inside the padded grid
    const bool compute = i <= nx - 1 && j <= ny + 1;
    const int64_t col = (int64_t)(i - 1) + sx * (j - 1);
    if (tid == 0) odd = solid[0] = solid[1] = solid[2] = solid[3] = 0;
    for (int r = tid; r < kColN * kMomTX; r += kMomTX * kMomTY) {
        const int q = r / kMomTX, ic = i0 + r % kMomTX;
        const int f = q - kColFace, e = q - kColCent;
        double x = 0.0;
        if (q < kColFace) {
            if (ic < M.mn[0]) x = M.m[0][col_quantity(q) * M.mn[0] + ic];
        } else if (e < 0) {
            if (ic < T.tn[UU]) x = T.t[UU][(f < 5 ? f : f + 1) * T.tn[UU] + ic];
        } else {
            if (ic < T.tn[UV]) x = T.t[UV][(e < 5 ? e : e + 1) * T.tn[UV] + ic];
        }
        xtab[r] = x;
    }
    // ring cells of a tile: rows j0..j0+TY-1 at x offsets -2, -1, 64, 65 (4 TY
    // cells), rows -2, -1, TY, TY+1 over the 64 columns (256 cells), and the
    // corners (64, -1) and (-1, TY) that V(1,-1,0) and U(-1,1,0) reach.  A
    // thread has at most two of the three fields' ring cells: where each lies in
    // a tile (-1: none) and in a plane (-1: outside the padded grid).
    constexpr int nside = 4 * kMomTY, nrow = 4 * kMomTX, nring = nside + nrow + 2;
    static_assert(3 * nring <= 2 * kMomTX * kMomTY, "two ring cells per thread");
    int rt[2], rp[2];
    const double *rf[2];
#pragma unroll
    for (int n = 0; n < 2; n++) {
        const int r = tid + n * kMomTX * kMomTY;
        const int f = r / nring, e = r - f * nring;
        rf[n] = f == 0 ? u : (f == 1 ? v : w);
        int ox, oy;
        if (e < nside) {
            const int s4 = e & 3;
            ox = s4 < 2 ? s4 - 2 : kMomTX + s4 - 2;
            oy = e >> 2;
        } else if (e < nside + nrow) {
            const int e2 = e - nside, s4 = e2 / kMomTX;
            ox = e2 - s4 * kMomTX;
            oy = s4 < 2 ? s4 - 2 : kMomTY + s4 - 2;
        } else if (e == nside + nrow) {
            ox = kMomTX;
            oy = -1;
        } else {
            ox = -1;
            oy = kMomTY;
        }
        const int gi = i0 + ox, gj = j0 + oy;
        const bool in = gi >= 1 && gi <= nx + 2 && gj >= 1 && gj <= ny + 2;
        rt[n] = r < 3 * nring ? f * kTile + (oy + 2) * kTileS + ox + 2 : -1;
        rp[n] = in && r < 3 * nring ? (gi - 1) + (int)sx * (gj - 1) : -1;
    }
    const int at = (ty + 2) * kTileS + tx + 2;
    const double *const own[3] = {u, v, w};
    bool strange = false;
    // a value of plane kk (0 outside the padded grid)
    auto load_own = [&](int f, int kk) {
        return mine_in && kk >= 1 && kk <= nz + 2 ? own[f][col + sxy * (kk - 1)] : 0.0;
    };
    auto load_ring = [&](int n, int kk) { return rp[n] >= 0 && kk <= nz + 2 ? rf[n][rp[n] + sxy * (kk - 1)] : 0.0; };
    // pressure at (i + a, j + b, kk) of a computed cell
    auto load_p = [&](int a, int b, int kk) {
        return compute && kk <= nz + 2 ? p[col + a + sx * b + sxy * (kk - 1)] : 0.0;
    };
    // whether one of my cells (my column, and my first ring cell: every cell of
    // the ring is somebody's first) of plane kk is not fluid
    auto tag_own = [&](int kk) { return mine_in && kk >= 1 && kk <= nz + 2 ? cell[col + sxy * (kk - 1)] : (int8_t)0; };
    auto tag_ring = [&](int kk) { return rp[0] >= 0 && kk >= 1 && kk <= nz + 2 ? cell[rp[0] + sxy * (kk - 1)] : (int8_t)0; };
    auto note = [&](double x) {
        strange |= !plain_velocity(x);
    };
    double m2[3], p2[3];
#pragma unroll
    for (int f = 0; f < 3; f++) {
        m2[f] = load_own(f, kb - 2);
        note(m2[f]);
#pragma unroll
        for (int d = -1; d <= 1; d++) {
            const double x = load_own(f, kb + d);
            note(x);
            tile[d + 1][f * kTile + at] = x;
        }
        p2[f] = load_own(f, kb + 2);
        note(p2[f]);
    }
#pragma unroll
    for (int n = 0; n < 2; n++)
#pragma unroll
        for (int d = -1; d <= 1; d++)
            if (rt[n] >= 0) {
                const double x = load_ring(n, kb + d);
                note(x);
                tile[d + 1][rt[n]] = x;
            }
    __syncthreads();   // (odd = 0 before anyone sets it)
    if (strange) odd = 1;
#pragma unroll
    for (int d = -1; d <= 1; d++)
        if (tag_own(kb + d) | tag_ring(kb + d)) solid[d + 1] = 1;
    __syncthreads();
    double *below = tile[0], *here = tile[1], *above = tile[2];
    const double p0 = load_p(0, 0, kb);
    double pc = load_p(0, 0, kb + 1);
    double pd[3] = {p0 - load_p(1, 0, kb), p0 - load_p(0, 1, kb), p0 - pc};
    uint64_t skipped = 0;   // my wave's rows, by plane (tz <= 64)
#pragma unroll 1
    for (int k = kb; k < ke; k++) {
        const int n = k - kb;
        const double g0 = load_ring(0, k + 2), g1 = load_ring(1, k + 2);
        double n2[3];
#pragma unroll
        for (int f = 0; f < 3; f++) n2[f] = load_own(f, k + 3);
        const double px = load_p(1, 0, k + 1), py = load_p(0, 1, k + 1), pz = load_p(0, 0, k + 2);
        const int8_t t0 = tag_own(k + 2), t1 = tag_ring(k + 2);
        if (compute) {
            const LdsColumns X{xtab + tx, M.m[0] + i, M.mn[0]};
            const TiledFields A{below + at, here + at, above + at, {m2[0], m2[1], m2[2]}, {p2[0], p2[1], p2[2]},
                                col + sxy * (k - 1), sx, sxy};
            const bool inner = j > 2 && j < ny && k > 2 && k < nz && uniform(odd) == 0 &&
                               uniform(solid[n & 3] | solid[(n + 1) & 3] | solid[(n + 2) & 3]) == 0 &&
                               __ballot(!(plain_velocity(pd[0]) && plain_velocity(pd[1]) && plain_velocity(pd[2]))) == 0;
            if (inner)
                momentum_cell<kPlain, true>(A, X, pd, i, j, k, p, cell, ut, vt, wt, ru, rv, rw, M, nx, ny, nz, rev,
                                            deltat);
            if (!inner) skipped |= (uint64_t)1 << n;
        }
#pragma unroll
        for (int f = 0; f < 3; f++) {
            m2[f] = below[f * kTile + at];
            note(n2[f]);
        }
        note(g0);
        note(g1);
        pd[0] = pc - px;
        pd[1] = pc - py;
        pd[2] = pc - pz;
        pc = pz;
        __syncthreads();   // plane k - 1 has been read
#pragma unroll
        for (int f = 0; f < 3; f++) below[f * kTile + at] = p2[f];
        if (rt[0] >= 0) below[rt[0]] = g0;
        if (rt[1] >= 0) below[rt[1]] = g1;
        if (strange) odd = 1;
        if (tid == 0) solid[n & 3] = 0;   // (plane k - 1's; plane k + 3 takes it)
        if (t0 | t1) solid[(n + 3) & 3] = 1;
        __syncthreads();
#pragma unroll
        for (int f = 0; f < 3; f++) p2[f] = n2[f];
        double *t = below;
        below = here;
        here = above;
        above = t;
    }
    // list what was skipped, one addition to the count per workgroup; the next
    // call's count is cleared here
    __shared__ int count[kMomTY], first;
    // lane 0's mask for the whole wave: lanes past the last column have none of
    // their own, but each lane lists the plane of its number
    skipped = (uint64_t)(uint32_t)uniform((int)(uint32_t)(skipped >> 32)) << 32 |
              (uint32_t)uniform((int)(uint32_t)skipped);
    if (tx == 0) count[ty] = __popcll(skipped);
    __syncthreads();
    int before = 0, all = 0;
    for (int q = 0; q < kMomTY; q++) {
        if (q < ty) before += count[q];
        all += count[q];
    }
    if (tid == 0 && all) first = atomicAdd(n_left, all);
    if (tid == 0 && blockIdx.x + blockIdx.y + blockIdx.z == 0) *n_next = 0;
    __syncthreads();
    if (skipped >> tx & 1)
        left[first + before + __popcll(skipped & (((uint64_t)1 << tx) - 1))] =
            ((kb + tx - 2) * ny + (j - 2)) * (int)gridDim.x + (int)blockIdx.x;
}

// subBoundaryConditions.f90:141-156: inlet u = 1, reflected v and w; outlet
// zero gradient
__global__ void k_bc_x(double *ut, double *vt, double *wt, int nx, int ny, int nz) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x + 2;
    const int k = blockIdx.y + 2;
    if (j > ny + 1) return;
    const int64_t sx = nx + 2;
    const int64_t r = sx * ((j - 1) + (int64_t)(ny + 2) * (k - 1));  // index of (1,j,k)
    ut[r] = 1.0;
    vt[r] = -vt[r + 1];
    wt[r] = -wt[r + 1];
    ut[r + nx] = ut[r + nx - 1];
    vt[r + nx + 1] = vt[r + nx];
    wt[r + nx + 1] = wt[r + nx];
}

// subBoundaryConditions.f90:161-174: free slip at the y walls
__global__ void k_bc_y(double *ut, double *vt, double *wt, int nx, int ny, int nz) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 2;
    const int k = blockIdx.y + 2;
    if (i > nx + 1) return;
    const int64_t sx = nx + 2, sxy = sx * (ny + 2);
    const int64_t b = (i - 1) + sxy * (k - 1);  // (i,1,k)
    const int64_t t = b + sx * (ny + 1);        // (i,ny+2,k)
    ut[b] = ut[b + sx];
    wt[b] = wt[b + sx];
    vt[b] = 0.0;
    ut[t] = ut[t - sx];
    wt[t] = wt[t - sx];
    vt[t - sx] = 0.0;
}

// subBoundaryConditions.f90:179-192: free slip at the z walls
__global__ void k_bc_z(double *ut, double *vt, double *wt, int nx, int ny, int nz) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 2;
    const int j = blockIdx.y + 2;
    if (i > nx + 1) return;
    const int64_t sx = nx + 2, sxy = sx * (ny + 2);
    const int64_t b = (i - 1) + sx * (j - 1);  // (i,j,1)
    const int64_t t = b + sxy * (nz + 1);      // (i,j,nz+2)
    ut[b] = ut[b + sxy];
    vt[b] = vt[b + sxy];
    wt[b] = 0.0;
    ut[t] = ut[t - sxy];
    vt[t] = vt[t - sxy];
    wt[t - sxy] = 0.0;
}

// subBoundaryConditions.f90:207-215
__global__ void k_solid_bc(const int *list, int64_t n, double *ut, double *vt, double *wt, double *p, int nx,
                           int ny, double wu, double wv, double ww) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int i = list[q], j = list[n + q], k = list[2 * n + q];
    const int64_t c = (i - 1) + (int64_t)(nx + 2) * ((j - 1) + (int64_t)(ny + 2) * (k - 1));
    ut[c] = wu;   // 0 in the reference (a body at rest); the body's velocity when it moves
    vt[c] = wv;
    wt[c] = ww;
    p[c] = 0.0;
}

__device__ __forceinline__ double pc_at(const double *p0, const double *p1, int64_t H, int sy, int ii, int jj,
                                        int kk) {
    const int64_t f = ((int64_t)jj + (int64_t)sy * kk) * H + (ii >> 1);
    return ((ii + jj + kk) & 1) ? p1[f] : p0[f];
}

// subPcorVcor.f90:113-118 and 132-140, fused: p += pc and the velocity
// correction on the east/north/top faces of each fluid cell
__global__ void __launch_bounds__(256)
k_correct(double *__restrict__ p, double *__restrict__ ut, double *__restrict__ vt, double *__restrict__ wt,
          const double *__restrict__ pc0, const double *__restrict__ pc1, const int8_t *__restrict__ cell,
          const double *__restrict__ dxa, const double *__restrict__ dya, const double *__restrict__ dza, int nx,
          int ny, int nz, int64_t H, double dt, int do_p, int do_v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 2;
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 2;
    const int k = blockIdx.z + 2;
    if (i > nx + 1 || j > ny + 1) return;
    const int sy = ny + 2;
    const int64_t c = (i - 1) + (int64_t)(nx + 2) * ((j - 1) + (int64_t)sy * (k - 1));
    if (cell[c] != 0) return;
    const int ii = i - 1, jj = j - 1, kk = k - 1;
    const double pcc = pc_at(pc0, pc1, H, sy, ii, jj, kk);
    if (do_p) p[c] = p[c] + pcc;
    if (do_v) {
        ut[c] = ut[c] - (dt / (0.5 * (dxa[i + 1] + dxa[i]))) * (pc_at(pc0, pc1, H, sy, ii + 1, jj, kk) - pcc);
        vt[c] = vt[c] - (dt / (0.5 * (dya[j + 1] + dya[j]))) * (pc_at(pc0, pc1, H, sy, ii, jj + 1, kk) - pcc);
        wt[c] = wt[c] - (dt / (0.5 * (dza[k + 1] + dza[k]))) * (pc_at(pc0, pc1, H, sy, ii, jj, kk + 1) - pcc);
    }
}

// subPcorVcor.f90:45-77: derrStdSt = max |ut-u|/dt over fluid cells, then
// u = ut over the whole padded grid
__global__ void __launch_bounds__(256)
k_steady_copy(double *__restrict__ u, double *__restrict__ v, double *__restrict__ w, const double *__restrict__ ut,
              const double *__restrict__ vt, const double *__restrict__ wt, const int8_t *__restrict__ cell, int nx,
              int ny, int nz, double dt, double *partial) {
    const int P = (nx + 2) * (ny + 2) * (nz + 2);  // < 2^31
    const int c = (int)blockIdx.x * (int)blockDim.x + (int)threadIdx.x;
    double m = 0.0;
    if (c < P) {
        const double a = ut[c], b = vt[c], d = wt[c];
        if (cell[c] == 0) {
            const int row = c / (nx + 2);
            const int ii = c - row * (nx + 2);
            const int kk = row / (ny + 2);
            const int jj = row - kk * (ny + 2);
            if (ii >= 1 && ii <= nx && jj >= 1 && jj <= ny && kk >= 1 && kk <= nz) {
                const double du = fabs(a - u[c]) / dt, dv = fabs(b - v[c]) / dt, dw = fabs(d - w[c]) / dt;
                m = fmax(fmax(du, dv), dw);
                if (du != du || dv != dv || dw != dw) m = __builtin_nan("");
            }
        }
        u[c] = a;
        v[c] = b;
        w[c] = d;
    }
    block_max_partial(m, partial);
}

// ------------------------------------------------------------------ host
static Tabs tabs(const Ctx &c) {
    Tabs T;
    for (int s = 0; s < 6; s++) {
        T.t[s] = c.tab[s];
        T.tn[s] = (int)c.tn[s];
    }
    return T;
}

// The momentum formula's index-only sub-expressions per axis, evaluated in
// the formula's own operations (host IEEE double, no contraction), and the
// reciprocals of the denominators that divide field values.  The fast
// division is enabled only if every such denominator lies in [2^-64, 2^64].
static int build_mom_tables(Ctx &c) {
    const std::vector<double> *dl[3] = {&c.hdx, &c.hdy, &c.hdz};
    const int64_t nn[3] = {c.nx, c.ny, c.nz};
    bool fast = true, plain = true;   // plain: see plain_velocity
    auto in_range = [](double d) {
        const double m = std::fabs(d);
        return m >= 0x1p-64 && m <= 0x1p64;
    };
    auto weight = [&](double d) { return d == 0.0 || in_range(d); };
    for (int a = 0; a < 3; a++) {
        const int64_t n = nn[a], tn = n + 3, ftn = c.tn[a];
        const std::vector<double> &d = *dl[a], &face = c.htab[a], &cent = c.htab[3 + a];
        std::vector<double> h(M_NQ * tn, 0.0);
        auto put = [&](int q, int64_t i, double x) { h[q * tn + i] = x; };
        auto upwind = [&](int q, int64_t i, double den, double r) {
            put(q, i, -1.0 / (r * (r + 1.0)));
            put(q + 1, i, 1.0 - 1.0 / r);
            put(q + 2, i, r / (r + 1.0));
            put(q + 3, i, 2.0 / (r * (r + 1.0)));
            put(q + 4, i, 2.0 / r);
            put(q + 5, i, 2.0 / (r + 1.0));
            put(q + 6, i, 1.0 / (2.0 * den));
        };
        for (int64_t i = 2; i <= n + 1; i++) {
            const double d0 = d[i], d1 = d[i + 1], dm = d[i - 1];
            const double h1 = 0.5 * (d0 + d1), h0 = 0.5 * (d0 + dm);
            put(M_AS, i, d1 / (d0 + d1));
            put(M_CS, i, 2.0 / (d0 + d1));
            put(M_D1, i, d1);
            put(M_RD1, i, 1.0 / d1);
            put(M_D0, i, d0);
            put(M_RD0, i, 1.0 / d0);
            upwind(M_US, i, d1, d0 / d1);
            put(M_CC, i, 2.0 / (0.5 * ((d0 + d1) + (d0 + dm))));
            put(M_H1, i, h1);
            put(M_RH1, i, 1.0 / h1);
            put(M_H0, i, h0);
            put(M_RH0, i, 1.0 / h0);
            upwind(M_UC, i, h1, h0 / h1);
            fast = fast && in_range(d0) && in_range(d1) && in_range(h0) && in_range(h1);
            plain = plain && d0 > 0.0 && d1 > 0.0 && h0 > 0.0 && h1 > 0.0 && in_range(d1 / (d0 + d1));
            if (i >= 3 && i <= n) {   // where the Kawamura-Kuwahara stencil can apply
                const double ks1 = face[5 * ftn + i] * d1, ks2 = (2.0 * face[11 * ftn + i]) * d0;
                const double kc1 = cent[5 * ftn + i] * h1, kc2 = (2.0 * cent[11 * ftn + i]) * h0;
                put(M_KS1, i, ks1);
                put(M_RKS1, i, 1.0 / ks1);
                put(M_KS2, i, ks2);
                put(M_RKS2, i, 1.0 / ks2);
                put(M_KC1, i, kc1);
                put(M_RKC1, i, 1.0 / kc1);
                put(M_KC2, i, kc2);
                put(M_RKC2, i, 1.0 / kc2);
                // the staggered component uses the face table for i <= n-1 only
                fast = fast && in_range(kc1) && in_range(kc2) && (i == n || (in_range(ks1) && in_range(ks2)));
                plain = plain && kc1 < 0.0 && kc2 > 0.0 && (i == n || (ks1 < 0.0 && ks2 > 0.0));
                for (int q = 0; q < 11; q++)
                    plain = plain && (q == 5 || ((weight(cent[q * ftn + i])) && (i == n || weight(face[q * ftn + i]))));
            }
        }
        // y and z: the same quantities and this axis's two convection tables, per index
        std::vector<double> r(a ? kMomRec * tn : 0, 0.0);
        for (int64_t i = 0; a && i < tn; i++) {
            for (int q = 0; q < M_NQ; q++) r[i * kMomRec + q] = h[q * tn + i];
            for (int q = 0; q < 12 && i < ftn; q++) {
                r[i * kMomRec + kRecS + q] = face[q * ftn + i];
                r[i * kMomRec + kRecC + q] = cent[q * ftn + i];
            }
        }
        if (c.mtn[a] != tn) {
            if (c.mtab[a]) IB3D_CHECK(hipFree(c.mtab[a]));
            if (c.mrec[a]) IB3D_CHECK(hipFree(c.mrec[a]));
            c.mtab[a] = c.mrec[a] = nullptr;
            c.mtn[a] = 0;
            IB3D_CHECK(hipMalloc((void **)&c.mtab[a], h.size() * sizeof(double)));
            if (a) IB3D_CHECK(hipMalloc((void **)&c.mrec[a], r.size() * sizeof(double)));
            c.mtn[a] = tn;
        }
        IB3D_CHECK(h2d(c.mtab[a], h.data(), h.size() * sizeof(double)));
        if (a) IB3D_CHECK(h2d(c.mrec[a], r.data(), r.size() * sizeof(double)));
    }
    const int64_t rows = ((c.nx + 63) / 64) * c.ny * c.nz;
    if (c.mom_rows < rows) {
        if (c.mom_left) IB3D_CHECK(hipFree(c.mom_left));
        c.mom_left = nullptr;
        c.mom_rows = 0;
        IB3D_CHECK(hipMalloc((void **)&c.mom_left, (rows + 2) * sizeof(int)));
        c.mom_counts = false;
        c.mom_rows = rows;
    }
    c.mom_fast = fast;
    c.mom_plain = fast && plain;
    c.mom_ready = true;
    return 0;
}

// the interior predictor: 0 by size, 1..3 from LDS tiles, 4 straight from HBM
static int g_mom_lds = 0;
// From this many cells on the tiles pay for their second launch (a call and
// its synchronisation, direct / tiles, us: 128x96x64 78 / 84, 160x80x80 106 / 98,
// 190x128x100 193 / 150, 256x192x192 754 / 433).
static constexpr int64_t kMomTilesFrom = 1000000;
// From this many cells on the interior rows straight from HBM pay for a launch of
// their own, k_momentum_rows (in k_momentum / apart, us: 128x64x64 42 / 52,
// 128x88x88 73 / 77, 128x96x96 82 / 87, 160x100x96 125 / 122, 190x128x100 164 / 156,
// 256x192x192 707 / 652).
static constexpr int64_t kMomRowsFrom = 1500000;
int set_momentum_tiles(int on) {
    IB3D_REQUIRE(on >= 0 && on <= 4, "set_momentum_tiles: variant must be 0..4");
    g_mom_lds = on;
    return 0;
}

// planes per workgroup of k_momentum_lds: two workgroups run on each of the 256
// compute units, and a workgroup spends about three planes' time on its start,
// so take the count that makes (rounds of 512 workgroups) x (planes + 3) least
static int momentum_planes(int64_t columns, int nz) {
    int best = 1;
    int64_t least = -1;
    for (int chunks = (nz + 63) / 64; chunks <= nz; chunks++) {   // (64: the mask of skipped planes)
        const int tz = (nz + chunks - 1) / chunks;
        const int64_t rounds = (columns * ((nz + tz - 1) / tz) + 511) / 512, cost = rounds * (tz + 3);
        if (least < 0 || cost < least) {
            least = cost;
            best = tz;
        }
    }
    return best;
}

int ns_momentum(Ctx &c, double rev, double deltat) {
    IB3D_REQUIRE(c.coeff_ready, "nsMomentum: non_uni_coeff has not run");
    IB3D_REQUIRE(c.lists_ready, "nsMomentum: cellCount has not run");
    if (!c.mom_ready && build_mom_tables(c)) return -1;
    MomTabs M;
    for (int a = 0; a < 3; a++) {
        M.m[a] = c.mtab[a];
        M.mn[a] = (int)c.mtn[a];
        M.rec[a] = c.mrec[a];
    }
    const Tabs T = tabs(c);
    const int nx = (int)c.nx, ny = (int)c.ny, nz = (int)c.nz;
    const int nxi = std::max(0, nx - 3);   // interior columns 3..nx-1
    const unsigned tnx = nblocks(nxi, kMomTX), tny = nblocks(ny, kMomTY);
    const int tz = momentum_planes((int64_t)tnx * tny, nz);
    const bool use_tiles = nxi > 0 && c.mom_plain && g_mom_lds != 4 &&
                           (g_mom_lds || (int64_t)nx * ny * nz >= kMomTilesFrom);
    const bool apart = nxi > 0 && !use_tiles && (int64_t)nx * ny * nz >= kMomRowsFrom;
    const bool off32 = c.P * (int64_t)sizeof(double) < ((int64_t)1 << 32);
    if (use_tiles && !c.mom_counts) {
        IB3D_CHECK(dzero(c.mom_left, 2 * sizeof(int)));
        c.mom_turn = 0;
    }
    auto launch = [&](auto fast) {
        constexpr bool F = decltype(fast)::value;
        const int turn = c.mom_turn;
        if (use_tiles) {
            c.mom_turn = 1 - turn;
            c.mom_counts = false;   // until the launches are known to have gone out
            hipLaunchKernelGGL(k_momentum_lds, dim3(tnx, tny, (unsigned)nblocks(nz, tz)), dim3(kMomTX, kMomTY, 1), 0,
                               c.stream, c.u, c.v, c.w, c.p, c.tag, c.ut, c.vt, c.wt, c.resi_u, c.resi_v, c.resi_w,
                               c.mom_left + 2, c.mom_left + turn, c.mom_left + 1 - turn, T, M, nx, ny, nz, tz, rev, deltat);
        }
        if (apart)
            hipLaunchKernelGGL((off32 ? k_momentum_rows<F, true> : k_momentum_rows<F, false>),
                               dim3(tnx, nblocks(ny, 4), (unsigned)nz), dim3(64, 4, 1), 0, c.stream, c.u, c.v, c.w, c.p,
                               c.tag, c.ut, c.vt, c.wt, c.resi_u, c.resi_v, c.resi_w, T, M, nx, ny, nz, rev, deltat);
        const int rows = apart ? 0 : (int)((int64_t)tnx * ny * nz), row_blocks = (rows + 3) / 4;
        const int edge = nblocks((int64_t)3 * ny * nz, 256);
        hipLaunchKernelGGL(k_momentum<F>, dim3(edge + (use_tiles ? std::min(kRestBlocks, row_blocks) : row_blocks)),
                           dim3(256), 0, c.stream, c.u, c.v, c.w, c.p, c.tag, c.ut, c.vt, c.wt, c.resi_u, c.resi_v,
                           c.resi_w, use_tiles ? c.mom_left + 2 : nullptr, c.mom_left + turn, T, M, nx, ny, nz, edge, (int)tnx, rev, deltat);
    };
    if (c.mom_fast)
        launch(std::true_type{});
    else
        launch(std::false_type{});
    IB3D_CHECK(hipGetLastError());
    if (use_tiles) c.mom_counts = true;
    return 0;
}

int velocity_bc(Ctx &c) {
    const int nx = (int)c.nx, ny = (int)c.ny, nz = (int)c.nz;
    hipLaunchKernelGGL(k_bc_x, dim3(nblocks(ny, 64), nz), dim3(64), 0, c.stream, c.ut, c.vt, c.wt, nx, ny, nz);
    hipLaunchKernelGGL(k_bc_y, dim3(nblocks(nx, 64), nz), dim3(64), 0, c.stream, c.ut, c.vt, c.wt, nx, ny, nz);
    hipLaunchKernelGGL(k_bc_z, dim3(nblocks(nx, 64), ny), dim3(64), 0, c.stream, c.ut, c.vt, c.wt, nx, ny, nz);
    IB3D_CHECK(hipGetLastError());
    return 0;
}

int solid_bc(Ctx &c) {
    IB3D_REQUIRE(c.lists_ready, "solidCellBC: cellCount has not run");
    if (c.solidCount == 0) return 0;
    hipLaunchKernelGGL(k_solid_bc, dim3(nblocks(c.solidCount, 256)), dim3(256), 0, c.stream, c.solidList,
                       c.solidCount, c.ut, c.vt, c.wt, c.p, (int)c.nx, (int)c.ny, c.wall_vel[0], c.wall_vel[1],
                       c.wall_vel[2]);
    IB3D_CHECK(hipGetLastError());
    return 0;
}

int correct(Ctx &c, double dt, int do_p, int do_v) {
    dim3 blk(64, 4, 1), grd(nblocks(c.nx, 64), nblocks(c.ny, 4), (unsigned)c.nz);
    hipLaunchKernelGGL(k_correct, grd, blk, 0, c.stream, c.p, c.ut, c.vt, c.wt, c.pc[0], c.pc[1], c.tag, c.dx, c.dy,
                       c.dz, (int)c.nx, (int)c.ny, (int)c.nz, c.H, dt, do_p, do_v);
    IB3D_CHECK(hipGetLastError());
    return 0;
}

// derr_std == nullptr: the result is left to arrive in c.hscal[3] at the
// caller's next synchronisation (one fewer host round trip per step)
int steady_copy(Ctx &c, double dt, double *derr_std) {
    const unsigned nb = nblocks(c.P, 256);
    if (ensure_partial(nb)) return -1;
    hipLaunchKernelGGL(k_steady_copy, dim3(nb), dim3(256), 0, c.stream, c.u, c.v, c.w, c.ut, c.vt,
                       c.wt, c.tag, (int)c.nx, (int)c.ny, (int)c.nz, dt, c.partial);
    launch_max_partials(c.partial, (int64_t)nb, c.scalars + 3);
    IB3D_CHECK(hipGetLastError());
    IB3D_CHECK(hipMemcpyAsync(c.hscal + 3, c.scalars + 3, sizeof(double), hipMemcpyDeviceToHost, c.stream));
    if (!derr_std) return 0;
    IB3D_CHECK(hipStreamSynchronize(c.stream));
    *derr_std = c.hscal[3];
    return 0;
}

}  // namespace ib3d
