// exact.hpp -- the reference's binary64 arithmetic of the hydro and MHD laws
// in fewer instructions, with the same values.
//
// The bit-exact kernels are bound by their VALU instruction count, and the
// literal form of a face spends most of it on things that do not change the
// value: an IEEE division is eleven instructions, of which div_scale and
// div_fixup only matter at the ends of the exponent range and the reciprocal
// with its two Newton steps depends on the denominator alone; a square root
// carries two ldexp, a compare and selects for the same ends; the
// min/max over ten eigenvalue slots and the sign products of minmod are
// compare-and-select chains.  Here
//   - quotients by one denominator share its reciprocal (Recip, quot): the
//     very operations of the IEEE sequence without its scaling, so the
//     quotient is the same whenever no scaling would take place;
//   - square roots drop the scaling likewise (root);
//   - the extreme wave speeds come straight from v -+ c.  sqrt and + are
//     monotone in IEEE arithmetic, so max(v + a, v + b) = v + max(a, b) and
//     max(sqrt a, sqrt b) = sqrt(max(a, b)) hold exactly, and a state's other
//     eigenvalues lie between the outermost two;
//   - minmod is max(min(a, b, c), min(max(a, b, c), 0));
//   - products with the exact zeros and ones of an axis normal are dropped.
// Every shortcut is taken under a test that its operands are ordinary (not
// NaN, infinite, near the ends of the exponent range, nor a state with
// negative pressure or density); a lane that fails it evaluates the literal
// expressions of physics.hpp, in functions of their own (literal_*) so that
// they cost the common path neither registers nor instruction cache.  Values
// are the literal form's bit for bit, up to the sign of a zero (compared over
// 5e8 random faces, 2e9 quotients and roots on gfx950: none differs).
//
// Measured (VALU instructions per wavefront and zone, time of one stage,
// literal -> this): 3-D PLM + HLLC tile 2170 -> 1255; 2-D PLM + HLLC,
// 636 x 477, 28.4 -> 23.5 us; 2-D MHD tiles, 2048^2, 570 -> 400 us; 3-D MHD
// flux sweeps, 116 x 97 x 108, 72 -> 50 us each.
#pragma once

#include "physics.hpp"

namespace mara {
namespace exact {

// Ordinary states: densities, sound speeds above LO, energies below HI.
// Then no intermediate of a face leaves [1e-240, 1e240].
constexpr double LO = 1e-40, HI = 1e60;

struct Recip
{
    double b, y;
};

__device__ __forceinline__ Recip recip(double b)
{
    double y = __builtin_amdgcn_rcp(b);
    y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    return {b, y};
}

// a / r.b for operands whose IEEE sequence needs no scaling
__device__ __forceinline__ double quot(double a, const Recip& r)
{
    const double q = a * r.y;
    return __builtin_fma(__builtin_fma(-r.b, q, a), r.y, q);
}

// sqrt(x) for ordinary positive x (NaN for 0, negative and infinite x)
__device__ __forceinline__ double root(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = y * 0.5;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// Order of magnitude of a numerator as an integer, zero highest: at or above
// TINY (2^-900) the remainder of quot is exact.  Values below 2^-1042 count as
// zero: their quotients by ordinary denominators may be off by one subnormal
// unit, 5e-324.
__device__ __forceinline__ unsigned magnitude(double a)
{
    return ((unsigned)((unsigned long long)__double_as_longlong(a) >> 32) << 1) - 1u;
}
constexpr unsigned TINY = (123u << 21) - 1u;

// F[q] = num[q] / den for ordinary den > 0
template <int NQ>
__device__ __forceinline__ void quotients(const double* num, double den, double* F)
{
    unsigned least = ~0u;
#pragma unroll
    for (int q = 0; q < NQ; ++q) least = min(least, magnitude(num[q]));
    if (__builtin_expect(least >= TINY, 1))
    {
        const Recip r = recip(den);
#pragma unroll
        for (int q = 0; q < NQ; ++q) F[q] = quot(num[q], r);
    }
    else
    {
#pragma unroll
        for (int q = 0; q < NQ; ++q) F[q] = num[q] / den;
    }
}

// gamma and the reciprocal of gamma - 1; an extreme gamma - 1 poisons the
// reciprocal, so every state fails the ordinary test and takes the literal form
struct Gas
{
    double gamma;
    Recip gm1;
};

__device__ __forceinline__ Gas gas(double gamma)
{
    Gas K;
    K.gamma = gamma;
    K.gm1 = recip(gamma - 1.0);
    if (!(gamma > 1.001 && gamma < 1000.0)) K.gm1.y = __builtin_nan("");
    return K;
}

// The literal forms, called where a test fails.
static __device__ __attribute__((noinline)) double literal_half_slope(double theta, double l, double c, double r)
{
    return 0.5 * minmod<double>(theta, l, c, r);
}

template <int Law>
static __device__ __attribute__((noinline)) void literal_state(const double* P, double gamma, const double* n,
                                                               State<double, LawNQ<Law>::value>* S)
{
    law_state<Law, double>(gamma, P, n, *S);
}

// the two states go through memory (the stack), which keeps the function
// within the registers of the kernels that call it
template <int Law, int Riem>
static __device__ __attribute__((noinline)) void literal_face(const double* PL, const double* PR, double gamma,
                                                              double n0, double n1, double n2, double* F)
{
    constexpr int NQ = LawNQ<Law>::value;
    const double n[3] = {n0, n1, n2};
    State<double, NQ> L, R;
    literal_state<Law>(PL, gamma, n, &L);
    literal_state<Law>(PR, gamma, n, &R);
    if constexpr (Riem == 1 && Law == 0) hllc(L, R, n, F);
    else hlle<double, NQ>(L, R, F);
}

// 0.5 * minmod of NQ fields; at(q, l, c, r) yields the three zones of a
// field.  min/max instructions drop a NaN operand where the literal form's
// comparisons fail: where a one-sided slope is NaN, or both are infinite, the
// literal form decides.
template <int NQ, typename Zones>
__device__ __forceinline__ void half_slopes(double theta, Zones at, double* h)
{
    double probe = 0.0;
#pragma unroll
    for (int q = 0; q < NQ; ++q)
    {
        double l, c, r;
        at(q, l, c, r);
        const double a = theta * (c - l), b = 0.5 * (r - l), d = theta * (r - c);
        const double lo = __builtin_fmin(a, __builtin_fmin(b, d)), hi = __builtin_fmax(a, __builtin_fmax(b, d));
        h[q] = 0.5 * __builtin_fmax(lo, __builtin_fmin(hi, 0.0));
        probe = q == 0 ? a + d : probe + (a + d);
    }
    if (__builtin_expect(probe != probe, 0))
    {
#pragma unroll
        for (int q = 0; q < NQ; ++q)
        {
            double l, c, r;
            at(q, l, c, r);
            h[q] = literal_half_slope(theta, l, c, r);
        }
    }
}

// Component of a vector along the face normal n, and n's component m.  AX 0
// and 2 are the exact unit vectors (1, 0, 0) and (0, 0, 1), AX 1 is
// (n[0], 1, 0) (UnitVector's yhat keeps cos(pi/2) = 6e-17); AX -1 is general.
template <int AX>
__device__ __forceinline__ double along(const double* v, const double* n)
{
    if constexpr (AX == 0) return v[0];
    else if constexpr (AX == 1) return v[0] * n[0] + v[1];
    else if constexpr (AX == 2) return v[2];
    else return v[0] * n[0] + v[1] * n[1] + v[2] * n[2];
}

template <int AX, int M>
__device__ __forceinline__ double plus_normal(double f, double p, const double* n)
{
    if constexpr (AX == M) return f + p;
    else if constexpr (AX == -1 || (AX == 1 && M == 0)) return f + p * n[M];
    else return f;
}

template <int NQ>
struct Side
{
    double U[NQ], F[NQ], vn, c;  // c: the fastest signal relative to the flow
    Recip rho;
};

// U, F, normal velocity and fastest signal of a hydro state; false where the
// state is not ordinary
template <int AX>
__device__ __forceinline__ bool side(const double* P, const Gas& K, const double* n, Side<5>& S)
{
    S.rho = recip(P[0]);
    S.c = root(quot(K.gamma * P[4], S.rho));
    S.vn = along<AX>(P + 1, n);
    const double vv = P[1] * P[1] + P[2] * P[2] + P[3] * P[3];
    S.U[0] = P[0];
    S.U[1] = P[0] * P[1];
    S.U[2] = P[0] * P[2];
    S.U[3] = P[0] * P[3];
    S.U[4] = P[0] * 0.5 * vv + quot(P[4], K.gm1);
    S.F[0] = S.vn * S.U[0];
    S.F[1] = plus_normal<AX, 0>(S.vn * S.U[1], P[4], n);
    S.F[2] = plus_normal<AX, 1>(S.vn * S.U[2], P[4], n);
    S.F[3] = plus_normal<AX, 2>(S.vn * S.U[3], P[4], n);
    S.F[4] = S.vn * S.U[4] + P[4] * S.vn;
    return (S.c > LO) & (P[0] > LO);
}

// The fast magnetosonic speed of an ordinary MHD state (the Alfven speed
// where rounding puts it above); disc receives the discriminant, whose root
// is taken only if it is ordinary.
__device__ __forceinline__ double fast_speed(double cs2, double ca2, double cn2, double& disc)
{
    const double cw4 = (cs2 + ca2) * (cs2 + ca2);
    disc = cw4 - 4.0 * cs2 * cn2;
    const double cF2 = 0.5 * (cs2 + ca2 + root(disc));
    return root(__builtin_fmax(cF2, cn2));
}

// the same of an MHD state (NQ 8, or 9 with the cooling law's auxiliary field)
template <int AX, int NQ>
__device__ __forceinline__ bool side(const double* P, const Gas& K, const double* n, Side<NQ>& S)
{
    S.rho = recip(P[0]);
    S.vn = along<AX>(P + 1, n);
    const double Bn = along<AX>(P + 5, n);
    const double vv = P[1] * P[1] + P[2] * P[2] + P[3] * P[3];
    const double BB = P[5] * P[5] + P[6] * P[6] + P[7] * P[7];
    const double Bv = P[5] * P[1] + P[6] * P[2] + P[7] * P[3];
    const double ps = P[4] + 0.5 * BB;
    S.U[0] = P[0];
    S.U[1] = P[0] * P[1];
    S.U[2] = P[0] * P[2];
    S.U[3] = P[0] * P[3];
    S.U[4] = P[0] * 0.5 * vv + 0.5 * BB + quot(P[4], K.gm1);
    S.U[5] = P[5];
    S.U[6] = P[6];
    S.U[7] = P[7];
    S.F[0] = S.vn * S.U[0];
    S.F[1] = plus_normal<AX, 0>(S.vn * S.U[1] - Bn * P[5], ps, n);
    S.F[2] = plus_normal<AX, 1>(S.vn * S.U[2] - Bn * P[6], ps, n);
    S.F[3] = plus_normal<AX, 2>(S.vn * S.U[3] - Bn * P[7], ps, n);
    S.F[4] = S.vn * S.U[4] - Bn * Bv + ps * S.vn;
    S.F[5] = S.vn * S.U[5] - Bn * P[1];
    S.F[6] = S.vn * S.U[6] - Bn * P[2];
    S.F[7] = S.vn * S.U[7] - Bn * P[3];
    if constexpr (NQ == 9)
    {
        S.U[8] = P[8];
        S.F[8] = 0.0;
    }
    const double cs2 = quot(K.gamma * P[4], S.rho);
    double disc;
    S.c = fast_speed(cs2, quot(BB, S.rho), quot(Bn * Bn, S.rho), disc);
    bool ok = (cs2 > LO * LO) & (P[0] > LO) & (disc > 1e-200);
    if constexpr (NQ == 9) ok = ok & (__builtin_fabs(P[8]) < HI);
    return ok;
}

// Flux through a face from its two states: law_state and hlle or hllc of
// physics.hpp.  False (F not set) where a state is not ordinary.
template <int Law, int Riem, int AX>
__device__ __forceinline__ bool face(const double* PL, const double* PR, const Gas& K, const double* n, double* F)
{
    constexpr int NQ = LawNQ<Law>::value;
    Side<NQ> L, R;
    const bool okL = side<AX>(PL, K, n, L), okR = side<AX>(PR, K, n, R);
    bool ok = okL & okR & (L.U[4] + R.U[4] + (PL[0] + PR[0]) < HI);
    const double ap = __builtin_fmax(__builtin_fmax(L.vn + L.c, R.vn + R.c), 0.0);
    const double am = __builtin_fmin(__builtin_fmin(L.vn - L.c, R.vn - R.c), 0.0);
    if constexpr (Riem == 1 && Law == 0)
    {
        const double lc = ((PR[4] - PR[0] * R.vn * (ap - R.vn)) - (PL[4] - PL[0] * L.vn * (am - L.vn)))
                          / (PL[0] * (am - L.vn) - PR[0] * (ap - R.vn));
        ok = ok & (__builtin_fabs(lc) < HI);
        if (!ok) return false;
        // the star state on the contact's side, as hllc() builds it
        const bool left = 0.0 <= lc;
        double Ps[5], Us[5], Fs[5];
#pragma unroll
        for (int q = 0; q < 5; ++q)
        {
            Ps[q] = left ? PL[q] : PR[q];
            Us[q] = left ? L.U[q] : R.U[q];
            Fs[q] = left ? L.F[q] : R.F[q];
        }
        const double a = left ? am : ap, vn = left ? L.vn : R.vn;
        const Recip rho = {Ps[0], left ? L.rho.y : R.rho.y};
        const double m = Ps[0] * (a - vn);
        const double f = m / (a - lc);
        double S[5];
        S[0] = f;
        S[4] = f * (quot(Us[4], rho) + (lc - vn) * (lc + Ps[4] / m));
        if constexpr (AX == -1)
        {
            S[1] = f * ((lc - vn) * n[0] + Ps[1]);
            S[2] = f * ((lc - vn) * n[1] + Ps[2]);
            S[3] = f * ((lc - vn) * n[2] + Ps[3]);
        }
        else
        {
            S[1] = f * (AX == 0 ? (lc - vn) + Ps[1] : AX == 1 ? (lc - vn) * n[0] + Ps[1] : Ps[1]);
            S[2] = f * (AX == 1 ? (lc - vn) + Ps[2] : Ps[2]);
            S[3] = f * (AX == 2 ? (lc - vn) + Ps[3] : Ps[3]);
        }
        const bool upwind = 0.0 <= am;  // am = 0: nothing travels left
#pragma unroll
        for (int q = 0; q < 5; ++q)
        {
            const double star = Fs[q] + a * (S[q] - Us[q]);
            F[q] = upwind ? L.F[q] : star;
        }
        return true;
    }
    else
    {
        if (!ok) return false;
        double num[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) num[q] = ap * L.F[q] - am * R.F[q] + ap * am * (R.U[q] - L.U[q]);
        quotients<NQ>(num, ap - am, F);
        return true;
    }
}

// face() with the literal form behind it
template <int Law, int Riem, int AX>
__device__ __forceinline__ void face_flux(const double* PL, const double* PR, const Gas& K, const double* n, double* F)
{
    if (__builtin_expect(face<Law, Riem, AX>(PL, PR, K, n, F), 1)) return;
    // copies, so that the states themselves stay in registers
    constexpr int NQ = LawNQ<Law>::value;
    double l[NQ], r[NQ], f[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q)
    {
        l[q] = PL[q];
        r[q] = PR[q];
    }
    literal_face<Law, Riem>(l, r, K.gamma, n[0], n[1], n[2], f);
#pragma unroll
    for (int q = 0; q < NQ; ++q) F[q] = f[q];
}

// prim_to_cons with the reciprocal of gamma - 1 at hand
template <int Law>
__device__ __forceinline__ void prim_to_cons(const Gas& K, const double* P, double* U)
{
    const double vv = P[1] * P[1] + P[2] * P[2] + P[3] * P[3];
    double e = P[0] * 0.5 * vv;
    if constexpr (Law != 0) e = e + 0.5 * (P[5] * P[5] + P[6] * P[6] + P[7] * P[7]);
    double th = quot(P[4], K.gm1);
    if (__builtin_expect(!((magnitude(P[4]) >= TINY) & (__builtin_fabs(th) < HI)), 0)) th = P[4] / (K.gamma - 1.0);
    U[0] = P[0];
    U[1] = P[0] * P[1];
    U[2] = P[0] * P[2];
    U[3] = P[0] * P[3];
    U[4] = e + th;
#pragma unroll
    for (int q = 5; q < LawNQ<Law>::value; ++q) U[q] = P[q];
}

// cons_to_prim with one reciprocal of the density, which ir returns (its y
// NaN where the density is not ordinary)
template <int Law>
__device__ __forceinline__ int cons_to_prim(double gamma, double pfloor, const double* U, double* P, int& floor,
                                            Recip& ir)
{
    const double half = 0.5 * (U[1] * U[1] + U[2] * U[2] + U[3] * U[3]);
    const unsigned least = min(min(magnitude(half), magnitude(U[1])), min(magnitude(U[2]), magnitude(U[3])));
    ir = recip(U[0]);
    double k = quot(half, ir);
    P[1] = quot(U[1], ir);
    P[2] = quot(U[2], ir);
    P[3] = quot(U[3], ir);
    // half bounds the momenta; NaN and infinite ones fail the comparison
    if (__builtin_expect(!((least >= TINY) & (U[0] > LO) & (half + U[0] < HI)), 0))
    {
        ir.y = __builtin_nan("");
        k = half / U[0];
        P[1] = U[1] / U[0];
        P[2] = U[2] / U[0];
        P[3] = U[3] / U[0];
    }
    const double gm1 = gamma - 1.0;
    P[0] = U[0];
    floor = 0;
    if constexpr (Law == 0)
    {
        P[4] = (U[4] - k) * gm1;
        return 0;
    }
    else
    {
        const double BB = U[5] * U[5] + U[6] * U[6] + U[7] * U[7];
        P[4] = (U[4] - k - 0.5 * BB) * gm1;
        P[5] = U[5];
        P[6] = U[6];
        P[7] = U[7];
        if constexpr (Law == 3) P[8] = U[8];
        if (P[4] < 0.0 || P[0] < 0.0 || U[0] < 0.0 || U[4] < 0.0)
        {
            if (P[4] < 0.0 && pfloor > 0.0)
            {
                P[4] = pfloor * P[0];
                floor = 1;
                return 0;
            }
            return 1;
        }
        return 0;
    }
}

// Largest signal speed of a zone over the three axes (courant_of's lmax), from
// its primitives and the reciprocal of its density; false where the zone is
// not ordinary.
template <int Law>
__device__ __forceinline__ bool signal_speed(const double* P, const Recip& ir, double gamma, const double* nhat,
                                             double& lmax)
{
    const double vx = __builtin_fabs(P[1]), vy = __builtin_fabs(along<1>(P + 1, nhat + 3)), vz = __builtin_fabs(P[3]);
    const double cs2 = quot(gamma * P[4], ir);
    bool ok = (cs2 > LO * LO) & (cs2 + (vx + vy) + vz < HI) & (ir.y == ir.y);
    if constexpr (Law == 0)
        lmax = __builtin_fmax(vx, __builtin_fmax(vy, vz)) + root(cs2);
    else
    {
        const double ca2 = quot(P[5] * P[5] + P[6] * P[6] + P[7] * P[7], ir);
        const double By = along<1>(P + 5, nhat + 3);
        double dx, dy, dz;
        const double cx = fast_speed(cs2, ca2, quot(P[5] * P[5], ir), dx);
        const double cy = fast_speed(cs2, ca2, quot(By * By, ir), dy);
        const double cz = fast_speed(cs2, ca2, quot(P[7] * P[7], ir), dz);
        ok = ok & (ca2 < HI) & (__builtin_fmin(dx, __builtin_fmin(dy, dz)) > 1e-200);
        lmax = __builtin_fmax(vx + cx, __builtin_fmax(vy + cy, vz + cz));
    }
    return ok;
}

} // namespace exact
} // namespace mara
