// shockx_kernels.h -- gfx950 device code for the SHOCK RHS / RK-stage path (FP64 form).
//
// Layout: ghost-padded SoA, linear index i*ng1*ng2 + j*ng2 + k (k fastest), the reference's
// own layout (src/Functions.c:56-103), so host arrays cross the C ABI without a transpose.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace shx {

// Physical and scheme constants shared by every kernel (kernel-argument struct).
struct Consts {
    double gamma, upsilon, psi, gam_heat, suth, eps;
    double gm1_ups;   // (gamma - 1) / Upsilon
    double igm1;      // 1 / (gamma - 1)
    double mach;      // reference Mach number (post-processing)
    double zd_mid[10], zd_int[10], zd_der[11];
    int mms;
};

// Pointer to a device array (hipMalloc'd, so in the global address space).  Element accesses
// cast to that address space, so the compiler emits global loads and stores even where the
// pointer itself was read from memory (the per-case records of the batched kernels); a plain
// pointer read from memory is generic and gets flat instructions, which share the LDS wait
// counter and serialise against the LDS traffic of the sweeps.  Host code assigns plain pointers.
template <class T>
struct gptr {
    T *p;
    gptr() = default;
    __host__ __device__ gptr(T *q) : p(q) {}
    template <class U>
    __host__ __device__ gptr(const gptr<U> &o) : p(o.p) {}
    __device__ __forceinline__ T &operator[](const long i) const
    {
        return *(T *)&((__attribute__((address_space(1))) T *)p)[i];
    }
    __host__ __device__ explicit operator bool() const { return p != nullptr; }
};
using gdp = gptr<double>;
using gcdp = gptr<const double>;

struct Fields5 { gdp f[5]; };
struct CFields5 { gcdp f[5]; };
struct Fields10 { gdp f[10]; };
struct CFields10 { gcdp f[10]; };
struct CFields12 { gcdp f[12]; };
struct Fields12 { gdp f[12]; };

struct Geom {
    int ng[3];        // padded extents
    int n[3];         // interior counts (n[2] = 1 in 2D)
    int lo[3];        // padded index of the first interior node (g, or 0 for the 2D z axis)
    long st[3];       // strides; the contiguous axis is padded to a multiple of 16 doubles
    int per[3];       // 1 where the direction is periodic (ghosts wrap), 0 where face writers fill them
    int dims, g;
    long ntot;        // logical padded nodes ng0*ng1*ng2
    long nalloc;      // doubles allocated per field (with the row padding)
};

// linear index of the t-th logical padded node (t in [0, ntot)); ijk receives its indices
__device__ __forceinline__ long padded_node(const Geom &gm, const long t, int ijk[3])
{
    ijk[2] = (int)(t % gm.ng[2]);
    const long r = t / gm.ng[2];
    ijk[1] = (int)(r % gm.ng[1]);
    ijk[0] = (int)(r / gm.ng[1]);
    return (long)ijk[0] * gm.st[0] + (long)ijk[1] * gm.st[1] + (long)ijk[2] * gm.st[2];
}

// ---------------------------------------------------------------------------------------
// Reciprocal from the hardware estimate (v_rcp_f64) refined by two Newton steps: within an ulp
// of 1/x for the normal, finite arguments the flux kernels pass, at a fraction of the cost of
// the IEEE-exact division sequence.
__device__ __forceinline__ double frcp(const double x)
{
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}

// Averaged interface state and the scalars the eigenvector entries share.
struct Eig {
    double nx, ny, nz, u, v, w, rho, cs;
    double gm1, q2, hm, gc, ics, irho, un, gs, h0;
};

__device__ __forceinline__ Eig make_eig(double nx, double ny, double nz, double u, double v, double w,
                                        double rho, double cs, double gamma)
{
    Eig e;
    e.nx = nx; e.ny = ny; e.nz = nz; e.u = u; e.v = v; e.w = w; e.rho = rho; e.cs = cs;
    e.gm1 = gamma - 1.0;
    e.q2 = u * u + v * v + w * w;
    const double ic = frcp(cs);
    const double M = sqrt(e.q2) * ic;
    e.hm = 1.0 - 0.5 * e.gm1 * (M * M);
    e.gc = e.gm1 * (ic * ic);
    e.ics = ic * 0.70710678118654752440;
    e.irho = frcp(rho);
    e.un = u * nx + v * ny + w * nz;
    e.gs = e.gm1 * ic;
    e.h0 = e.q2 / 2. + cs * cs * frcp(e.gm1);
    return e;
}

// Row C of the left eigenvector matrix (src/WENO.c:1208-1236).
template <int C>
__device__ __forceinline__ void left_row(const Eig &e, double L[5])
{
    constexpr double is2 = 0.70710678118654752440;
    if constexpr (C == 0) {
        L[0] = e.nx * e.hm - e.irho * (e.v * e.nz - e.w * e.ny);
        L[1] = e.gc * e.u * e.nx; L[2] = e.gc * e.v * e.nx + e.nz * e.irho;
        L[3] = e.gc * e.w * e.nx - e.ny * e.irho; L[4] = -e.gc * e.nx;
    } else if constexpr (C == 1) {
        L[0] = e.ny * e.hm - e.irho * (e.w * e.nx - e.u * e.nz);
        L[1] = e.gc * e.u * e.ny - e.nz * e.irho; L[2] = e.gc * e.v * e.ny;
        L[3] = e.gc * e.w * e.ny + e.nx * e.irho; L[4] = -e.gc * e.ny;
    } else if constexpr (C == 2) {
        L[0] = e.nz * e.hm - e.irho * (e.u * e.ny - e.v * e.nx);
        L[1] = e.gc * e.u * e.nz + e.ny * e.irho; L[2] = e.gc * e.v * e.nz - e.nx * e.irho;
        L[3] = e.gc * e.w * e.nz; L[4] = -e.gc * e.nz;
    } else if constexpr (C == 3) {
        L[0] = e.ics * (e.gm1 * e.q2 / 2. - e.cs * e.un);
        L[1] = (-e.gs * e.u + e.nx) * is2; L[2] = (-e.gs * e.v + e.ny) * is2;
        L[3] = (-e.gs * e.w + e.nz) * is2; L[4] = e.gm1 * e.ics;
    } else {
        L[0] = e.ics * (e.gm1 * e.q2 / 2. + e.cs * e.un);
        L[1] = (-e.gs * e.u - e.nx) * is2; L[2] = (-e.gs * e.v - e.ny) * is2;
        L[3] = (-e.gs * e.w - e.nz) * is2; L[4] = e.gm1 * e.ics;
    }
}

// Row M of the right eigenvector matrix (src/WENO.c:1176-1204): R[M][0..4].
template <int M>
__device__ __forceinline__ void right_row(const Eig &e, double R[5])
{
    if constexpr (M == 0) {
        R[0] = e.nx; R[1] = e.ny; R[2] = e.nz; R[3] = e.ics; R[4] = e.ics;
    } else if constexpr (M == 1) {
        R[0] = e.u * e.nx; R[1] = e.u * e.ny - e.rho * e.nz; R[2] = e.u * e.nz + e.rho * e.ny;
        R[3] = e.ics * (e.u + e.nx * e.cs); R[4] = e.ics * (e.u - e.nx * e.cs);
    } else if constexpr (M == 2) {
        R[0] = e.v * e.nx + e.rho * e.nz; R[1] = e.v * e.ny; R[2] = e.v * e.nz - e.rho * e.nx;
        R[3] = e.ics * (e.v + e.ny * e.cs); R[4] = e.ics * (e.v - e.ny * e.cs);
    } else if constexpr (M == 3) {
        R[0] = e.w * e.nx - e.rho * e.ny; R[1] = e.w * e.ny + e.rho * e.nx; R[2] = e.w * e.nz;
        R[3] = e.ics * (e.w + e.nz * e.cs); R[4] = e.ics * (e.w - e.nz * e.cs);
    } else {
        R[0] = e.q2 / 2. * e.nx + e.rho * (e.v * e.nz - e.w * e.ny);
        R[1] = e.q2 / 2. * e.ny + e.rho * (e.w * e.nx - e.u * e.nz);
        R[2] = e.q2 / 2. * e.nz + e.rho * (e.u * e.ny - e.v * e.nx);
        R[3] = e.ics * (e.h0 + e.cs * e.un); R[4] = e.ics * (e.h0 - e.cs * e.un);
    }
}

// ---- axis-aligned normals (diagonal metric) -----------------------------------------------------
// With n = s e_AX (s = +-1) the eigenvector rows above lose most entries.  eps3(a, b, c) is the
// Levi-Civita symbol; the rows below are the general ones with the zero components dropped, so
// they produce the same values.
__host__ __device__ constexpr int eps3(int a, int b, int c)
{
    return (a == b || b == c || a == c) ? 0 : (((a + 1) % 3 == b) ? 1 : -1);
}
// L[C][q] can be non-zero
__host__ __device__ constexpr bool lnz(int C, int AX, int q)
{
    return (C == AX || C >= 3) ? true : (q == 0 || q == 1 + (3 - C - AX));
}
// R[M][C] can be non-zero
__host__ __device__ constexpr bool rnz(int M, int AX, int C)
{
    return (C >= 3 || M == 4) ? true
         : (M == 0 ? C == AX : (C == AX || eps3(M - 1, C, AX) != 0));
}

template <int C, int AX>
__device__ __forceinline__ void left_row_ax(const Eig &e, const double s, double L[5])
{
    constexpr double is2 = 0.70710678118654752440;
    const double uu[3] = {e.u, e.v, e.w};
    if constexpr (C == AX) {
        L[0] = s * e.hm;
        L[1] = e.gc * e.u * s; L[2] = e.gc * e.v * s; L[3] = e.gc * e.w * s; L[4] = -e.gc * s;
    } else if constexpr (C < 3) {
        constexpr int T = 3 - C - AX;
        constexpr double sg = (double)eps3(C, AX, T);
        L[0] = sg * s * (e.irho * uu[T]);
        L[1 + T] = -sg * s * e.irho;
    } else {
        constexpr double pm = (C == 3) ? 1.0 : -1.0;
        L[0] = e.ics * (e.gm1 * e.q2 / 2. - pm * e.cs * e.un);
#pragma unroll
        for (int q = 0; q < 3; q++) L[1 + q] = (q == AX) ? (-e.gs * uu[q] + pm * s) * is2 : (-e.gs * uu[q]) * is2;
        L[4] = e.gm1 * e.ics;
    }
}

template <int M, int AX>
__device__ __forceinline__ void right_row_ax(const Eig &e, const double s, double R[5])
{
    const double uu[3] = {e.u, e.v, e.w};
    if constexpr (M == 0) {
        R[AX] = s; R[3] = e.ics; R[4] = e.ics;
    } else if constexpr (M < 4) {
        constexpr int q = M - 1;
#pragma unroll
        for (int C = 0; C < 3; C++) {
            if (C == AX) R[C] = uu[q] * s;
            else if (eps3(q, C, AX) != 0) R[C] = -(double)eps3(q, C, AX) * (e.rho * s);
        }
        R[3] = (q == AX) ? e.ics * (uu[q] + s * e.cs) : e.ics * uu[q];
        R[4] = (q == AX) ? e.ics * (uu[q] - s * e.cs) : e.ics * uu[q];
    } else {
#pragma unroll
        for (int C = 0; C < 3; C++) {
            if (C == AX) R[C] = e.q2 / 2. * s;
            else R[C] = e.rho * ((double)eps3(C, 3 - C - AX, AX) * uu[3 - C - AX] * s);
        }
        R[3] = e.ics * (e.h0 + e.cs * e.un);
        R[4] = e.ics * (e.h0 - e.cs * e.un);
    }
}

// ---- characteristic projection without the eigenvector entries ------------------------------------
// The left and right eigenvectors above applied to a vector g = (g0, gm, g4) of differences through
// S = gm - g0 u (momentum less the mean velocity's share) and t = g4 - u.S - |u|^2/2 g0 (the pressure
// difference over gamma - 1):
//   L_0..2 . g = n_c E + (n x S)-component / rho,  E = g0 - (gamma-1)/c^2 t
//   L_3,4 . g  = ((gamma-1)/c t +- n.S) / sqrt(2)
// which is 23 operations for the five projections (11 with a diagonal metric) instead of 25 (19), and
// needs no entry of L in registers.  char_project leaves out constant factors of a field, which the
// assembly puts back: the deviation Phi is homogeneous of degree one in its inputs, so only epsilon
// has to follow (times the factor's inverse squared).  Left out: 1/sqrt(2) of the acoustic fields;
// with a diagonal metric also the normal's sign and the shear fields' 1/rho, against which the right
// eigenvectors' rho cancels.
struct CharBasis {
    double u[3];          // mean velocity
    double n[3], rn[3];   // mean unit normal, over rho (general metric)
    double s;             // diagonal metric: the normal's component along the axis (+-1; 0 between
                          // nodes of opposite sign)
    double q2h, ic, gic, gic2;   // |u|^2 / 2, 1/c, (gamma-1)/c, (gamma-1)/c^2
};
template <int AX>
__device__ __forceinline__ void char_basis(CharBasis &c, const double rho, const double cs, const double gamma)
{
    c.q2h = 0.5 * (c.u[0] * c.u[0] + c.u[1] * c.u[1] + c.u[2] * c.u[2]);
    c.ic = frcp(cs);
    c.gic = (gamma - 1.0) * c.ic;
    c.gic2 = c.gic * c.ic;
    if constexpr (AX < 0) {
        const double ir = frcp(rho);
#pragma unroll
        for (int q = 0; q < 3; q++) c.rn[q] = c.n[q] * ir;
    }
}
// o: fields 0, 1, 2 (diagonal metric: entropy, then the shear fields of the axes after AX), acoustic +, -
template <int AX>
__device__ __forceinline__ void char_project(const CharBasis &c, const double g[5], double o[5])
{
    double S[3];
#pragma unroll
    for (int q = 0; q < 3; q++) S[q] = fma(-c.u[q], g[0], g[1 + q]);
    const double t = fma(-c.u[2], S[2], fma(-c.u[1], S[1], fma(-c.u[0], S[0], fma(-c.q2h, g[0], g[4]))));
    const double E = fma(-c.gic2, t, g[0]);
    const double Xc = c.gic * t;
    if constexpr (AX < 0) {
        o[0] = fma(c.n[0], E, fma(c.rn[2], S[1], -(c.rn[1] * S[2])));
        o[1] = fma(c.n[1], E, fma(c.rn[0], S[2], -(c.rn[2] * S[0])));
        o[2] = fma(c.n[2], E, fma(c.rn[1], S[0], -(c.rn[0] * S[1])));
        const double sn = fma(c.n[2], S[2], fma(c.n[1], S[1], c.n[0] * S[0]));
        o[3] = Xc + sn;
        o[4] = Xc - sn;
    } else {
        o[0] = E;
        o[1] = S[(AX + 1) % 3];
        o[2] = S[(AX + 2) % 3];
        o[3] = fma(c.s, S[AX], Xc);
        o[4] = fma(-c.s, S[AX], Xc);
    }
}
// R . Phi from the fields' deviations psi (six times Phi, as w5_pair returns them); c2g = c^2/(gamma-1)
template <int AX>
__device__ __forceinline__ void char_assemble(const CharBasis &c, const double rho, const double c2g,
                                              const double psi[5], double out[5])
{
    const double P = (c.ic * (1. / 12.)) * (psi[3] + psi[4]);
    if constexpr (AX < 0) {
        const double D = (1. / 12.) * (psi[3] - psi[4]);
        const double r6 = rho * (1. / 6.);
        const double M0 = fma(1. / 6., fma(c.n[2], psi[2], fma(c.n[1], psi[1], c.n[0] * psi[0])), P);
        double W[3];
        W[0] = r6 * fma(c.n[1], psi[2], -(c.n[2] * psi[1]));
        W[1] = r6 * fma(c.n[2], psi[0], -(c.n[0] * psi[2]));
        W[2] = r6 * fma(c.n[0], psi[1], -(c.n[1] * psi[0]));
#pragma unroll
        for (int q = 0; q < 3; q++) W[q] = fma(c.n[q], D, W[q]);
        out[0] = M0;
#pragma unroll
        for (int q = 0; q < 3; q++) out[1 + q] = fma(c.u[q], M0, W[q]);
        out[4] = fma(c.q2h, M0, fma(c2g, P, fma(c.u[2], W[2], fma(c.u[1], W[1], c.u[0] * W[0]))));
    } else {
        constexpr int T1 = (AX + 1) % 3, T2 = (AX + 2) % 3;
        const double s6 = (c.s * c.s) * (1. / 6.);
        const double D = (c.s * (1. / 12.)) * (psi[3] - psi[4]);
        const double W1 = s6 * psi[1], W2 = s6 * psi[2];
        const double M0 = fma(s6, psi[0], P);
        out[0] = M0;
        out[1 + AX] = fma(c.u[AX], M0, D);
        out[1 + T1] = fma(c.u[T1], M0, W1);
        out[1 + T2] = fma(c.u[T2], M0, W2);
        out[4] = fma(c.q2h, M0, fma(c2g, P, fma(c.u[AX], D, fma(c.u[T1], W1, c.u[T2] * W2))));
    }
}

// 2^-floor(log2 x) of a positive normal x
__device__ __forceinline__ double inv_pow2(const double x)
{
    const int hi = (int)(__double_as_longlong(x) >> 32);
    return __longlong_as_double((long long)(0x7FE00000 - (hi & 0x7FF00000)) << 32);
}
// N / D from the hardware's reciprocal (24 bits) and one third-order step
__device__ __forceinline__ double quotient(const double N, const double D)
{
    const double r = __builtin_amdgcn_rcp(D);
    const double e = fma(-D, r, 1.0);
    const double y = N * r;
    return fma(y, fma(e, e, e), y);
}
// N[1] / D[1] - N[0] / D[0] with one reciprocal
__device__ __forceinline__ double pair_quotient(const double N[2], const double D[2])
{
    return quotient(fma(N[1], D[0], -(N[0] * D[1])), D[0] * D[1]);
}

// Six times the Jiang-Shu WENO5 deviation of a field (Phi_Function_W5, src/WENO.c:118-204, of the minus
// side less the plus side), from the four split differences of each side.  With IS_k the indicators
// over three, q_k = IS_k + eps and a = q1 q2, b = q0 q1, c = q0 q2:
//   3 Phi = N / D - (second difference) / 4,  D = a^2 + 3 b^2 + 6 c^2,  N = a^2 (d0-2d1+d2) + 3/2 b^2 (d1-2d2+d3)
// and the two sides share one reciprocal.  The indicators of both sides are scaled by the power of two
// that brings the largest to [1, 2) (exact; the weights are ratios), and the scaled epsilon is held at
// f = 2^-150: the smallest product, of a side without differences (D = 10 f^4) and a side with one
// indicator (9 f^2), is then 2^-894, still normal.  The other side's largest differences bound what
// that floor can change: where it replaces all indicators of a side, that side's differences are below
// 2^-75 of the other's, less than the rounding of their sum.
__device__ __forceinline__ double w5_pair(const double eps, const double p[4], const double m[4])
{
    double I[2][3], g1[2], g2[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const double *d = h ? m : p;
        const double t0 = d[0] - d[1], t1 = fma(-3., d[1], d[0]);
        const double t2 = d[1] - d[2], t3 = d[1] + d[2];
        const double t4 = d[2] - d[3], t5 = fma(3., d[2], -d[3]);
        I[h][0] = fma(13. / 3. * t0, t0, t1 * t1);
        I[h][1] = fma(13. / 3. * t2, t2, t3 * t3);
        I[h][2] = fma(13. / 3. * t4, t4, t5 * t5);
        g1[h] = t0 - t2;
        g2[h] = t2 - t4;
    }
    const double mx = fmax(fmax(fmax(I[0][0], I[0][1]), fmax(I[0][2], I[1][0])), fmax(fmax(I[1][1], I[1][2]), eps));
    const double sc = inv_pow2(mx);
    const double fl = fmax(eps * sc, 0x1p-150);
    double N[2], D[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const double q0 = fma(I[h][0], sc, fl), q1 = fma(I[h][1], sc, fl), q2 = fma(I[h][2], sc, fl);
        const double a = q1 * q2, b = q0 * q1, c = q0 * q2;
        const double A = a * a, B = 1.5 * b * b;
        D[h] = fma(6. * c, c, fma(2., B, A));
        N[h] = fma(B, g2[h], A * g1[h]);
    }
    return fma(0.25, g2[0] - g2[1], pair_quotient(N, D));
}

// ---- FP32 forms for the mixed-precision sweeps ------------------------------------------------
// Smoothness indicators scaled by a common power of two so that the largest lies in [1/2, 1), each
// clamped from below at 2^lo and squared; the weights are ratios, so the scale drops out.  Inputs are
// FP32 node-to-node differences.  epsilon is dropped: FP32 cannot hold the reference's
// 10 sqrt(DBL_MIN), and the clamp gives the ideal weights where all indicators vanish, which is what an
// epsilon far below every indicator does.
template <int N>
__device__ __forceinline__ void scaled_sq_f(float s[N], const int lo)
{
    float mx = s[0];
#pragma unroll
    for (int i = 1; i < N; i++) mx = fmaxf(mx, s[i]);
    const int ex = __builtin_amdgcn_frexp_expf(mx);
    const float floor_ = __builtin_amdgcn_ldexpf(1.0f, lo);
#pragma unroll
    for (int i = 0; i < N; i++) {
        const float t = fmaxf(__builtin_amdgcn_ldexpf(s[i], -ex), floor_);
        s[i] = t * t;
    }
}

__device__ __forceinline__ float phi_w5_f(const float d0, const float d1, const float d2, const float d3)
{
    const float t0 = d0 - d1, t1 = d0 - 3.f * d1;
    const float t2 = d1 - d2, t3 = d1 + d2;
    const float t4 = d2 - d3, t5 = 3.f * d2 - d3;
    float q[3] = {13.f * t0 * t0 + 3.f * t1 * t1, 13.f * t2 * t2 + 3.f * t3 * t3, 13.f * t4 * t4 + 3.f * t5 * t5};
    scaled_sq_f<3>(q, -30);
    const float P0 = q[1] * q[2], P2 = 3.f * (q[0] * q[1]);
    const float r = __builtin_amdgcn_rcpf(P0 + 6.f * (q[0] * q[2]) + P2);
    const float w0 = P0 * r, w2 = P2 * r;
    const float q1 = d0 - 2.f * d1 + d2;
    const float qq2 = d1 - 2.f * d2 + d3;
    return (1.f / 3.f) * w0 * q1 + (1.f / 6.f) * (w2 - 0.5f) * qq2;
}

// The Balsara-Shu indicators rewritten as sums of squares of difference combinations (the
// LDL^T factorisation of each quadratic form in the four first differences of its sub-stencil,
// exact rationals): every term is non-negative, so FP32 keeps them to ~1e-6 relative where the
// point-value form loses 1e-4 to cancellation on smooth data.
__device__ __forceinline__ float phi_w9_f(const float *d)
{
    const float y00 = d[0] + (-163185.f / 45316.f) * d[1] + (100839.f / 22658.f) * d[2] + (-86329.f / 45316.f) * d[3];
    const float y01 = d[1] + (-41089198.f / 14249315.f) * d[2] + (1813059.f / 838195.f) * d[3];
    const float y02 = d[2] + (-350813921.f / 232768856.f) * d[3];
    const float y03 = d[3];
    const float is0 = 22658.f * y00 * y00 + (299235615.f / 90632.f) * y01 * y01 + (39105167808.f / 14249315.f) * y02 * y02 + (116566909305.f / 29096107.f) * y03 * y03;
    const float y10 = d[1] + (-47055.f / 13816.f) * d[2] + (26079.f / 6908.f) * d[3] + (-18079.f / 13816.f) * d[4];
    const float y11 = d[2] + (-12448558.f / 5880675.f) * d[3] + (5686883.f / 5880675.f) * d[4];
    const float y12 = d[3] + (-146761231.f / 232768856.f) * d[4];
    const float y13 = d[4];
    const float is1 = 6908.f * y10 * y10 + (123494175.f / 27632.f) * y11 * y11 + (13035055936.f / 1960225.f) * y12 * y12 + (116566909305.f / 29096107.f) * y13 * y13;
    const float y20 = d[2] + (-37185.f / 13816.f) * d[3] + (15369.f / 6908.f) * d[4] + (-8209.f / 13816.f) * d[5];
    const float y21 = d[3] + (-1032654.f / 838195.f) * d[4] + (5686883.f / 14249315.f) * d[5];
    const float y22 = d[4] + (-20636113.f / 51089708.f) * d[5];
    const float y23 = d[5];
    const float is2 = 6908.f * y20 * y20 + (299235615.f / 27632.f) * y21 * y21 + (8583070944.f / 838195.f) * y22 * y22 + (233133818610.f / 217131259.f) * y23 * y23;
    const float y30 = d[3] + (-94935.f / 45316.f) * d[4] + (35109.f / 22658.f) * d[5] + (-18079.f / 45316.f) * d[6];
    const float y31 = d[4] + (-106728718.f / 110863235.f) * d[5] + (30822003.f / 110863235.f) * d[6];
    const float y32 = d[5] + (-1745642471.f / 4217089556.f) * d[6];
    const float y33 = d[6];
    const float is3 = 22658.f * y30 * y30 + (2328127935.f / 90632.f) * y31 * y31 + (101210149344.f / 15837605.f) * y32 * y32 + (233133818610.f / 1054272389.f) * y33 * y33;
    const float y40 = d[4] + (-433665.f / 215836.f) * d[5] + (162579.f / 107918.f) * d[6] + (-86329.f / 215836.f) * d[7];
    const float y41 = d[5] + (-945305518.f / 890329635.f) * d[6] + (290071763.f / 890329635.f) * d[7];
    const float y42 = d[6] + (-8384962321.f / 17843974736.f) * d[7];
    const float y43 = d[7];
    const float is4 = 107918.f * y40 * y40 + (18696922335.f / 431672.f) * y41 * y41 + (999262585216.f / 296776545.f) * y42 * y42 + (16652415615.f / 318642406.f) * y43 * y43;
    // weights d_k / q_k with the indicators scaled by the largest and clamped at 2^-60 of it, so
    // every q_k >= 2^-120 and the sum stays finite (products of four q, as in the FP64 form,
    // would need a clamp near 2^-15 in FP32, which distorts weights that still matter)
    float q[5] = {is0, is1, is2, is3, is4};
    scaled_sq_f<5>(q, -60);
    const float A0 = (1.f / 126.f) * __builtin_amdgcn_rcpf(q[0]), A1 = (10.f / 63.f) * __builtin_amdgcn_rcpf(q[1]);
    const float A2 = (10.f / 21.f) * __builtin_amdgcn_rcpf(q[2]), A3 = (20.f / 63.f) * __builtin_amdgcn_rcpf(q[3]);
    const float A4 = (5.f / 126.f) * __builtin_amdgcn_rcpf(q[4]);
    const float ia = __builtin_amdgcn_rcpf(A0 + A1 + A2 + A3 + A4);
    const float w0 = A0 * ia, w2 = A2 * ia, w3 = A3 * ia, w4 = A4 * ia;
    const float q1 = d[0] - 4.f * d[1] + 6.f * d[2] - 4.f * d[3] + d[4];
    const float q2 = d[1] - 4.f * d[2] + 6.f * d[3] - 4.f * d[4] + d[5];
    const float q3 = d[2] - 4.f * d[3] + 6.f * d[4] - 4.f * d[5] + d[6];
    const float q4 = d[3] - 4.f * d[4] + 6.f * d[5] - 4.f * d[6] + d[7];
    return (1.f / 5.f) * w0 * q1 + (1.f / 20.f) * w2 * q2 + (1.f / 60.f) * w3 * (3.f * q2 - 2.f * q3)
         + (1.f / 60.f) * w4 * (3.f * q2 - 2.f * q3 + 3.f * q4) - (1.f / 840.f) * (39.f * q2 - 14.f * q3 + 3.f * q4);
}

// Balsara-Shu indicator of one five-point sub-stencil from its four differences, as the sum of squares
// of the LDL^T factorisation of its quadratic form (exact rationals, as in phi_w9_f): the same number
// as the reference's form in point values (src/WENO.c:11-116), without its cancellation between terms
// of the size of the squared values, in 14 operations instead of 20.  K: sub-stencil 0, 1 or 2; 3 and 4
// are 1 and 0 mirrored.
template <int K>
__device__ __forceinline__ double w9_is(const double a, const double b, const double c, const double d)
{
    if constexpr (K == 0) {
        const double y0 = fma(-86329. / 45316., d, fma(100839. / 22658., c, fma(-163185. / 45316., b, a)));
        const double y1 = fma(1813059. / 838195., d, fma(-41089198. / 14249315., c, b));
        const double y2 = fma(-350813921. / 232768856., d, c);
        return fma(22658. * y0, y0, fma(299235615. / 90632. * y1, y1,
               fma(39105167808. / 14249315. * y2, y2, (116566909305. / 29096107. * d) * d)));
    } else if constexpr (K == 1) {
        const double y0 = fma(-18079. / 13816., d, fma(26079. / 6908., c, fma(-47055. / 13816., b, a)));
        const double y1 = fma(5686883. / 5880675., d, fma(-12448558. / 5880675., c, b));
        const double y2 = fma(-146761231. / 232768856., d, c);
        return fma(6908. * y0, y0, fma(123494175. / 27632. * y1, y1,
               fma(13035055936. / 1960225. * y2, y2, (116566909305. / 29096107. * d) * d)));
    } else {
        const double y0 = fma(-8209. / 13816., d, fma(15369. / 6908., c, fma(-37185. / 13816., b, a)));
        const double y1 = fma(5686883. / 14249315., d, fma(-1032654. / 838195., c, b));
        const double y2 = fma(-20636113. / 51089708., d, c);
        return fma(6908. * y0, y0, fma(299235615. / 27632. * y1, y1,
               fma(8583070944. / 838195. * y2, y2, (233133818610. / 217131259. * d) * d)));
    }
}

// Six times the WENO9 deviation of a field (Phi_Function_W9, src/WENO.c:11-116, of the minus side less
// the plus side, as w5_pair) from the eight split differences of each side.  Each side's indicators are
// scaled by the power of two that brings the largest to [1, 2) and epsilon is held at f = 2^-160 there.
// Beside a jump the smooth sub-stencils' indicators are the small ones, and they carry the weights: what
// the floor hides is differences below 2^-80 of the largest, which are not seen beside its rounding.
// With s_k = (IS_k + eps)^2 the sums D = sum_k 126 d_k prod_{j != k} s_j are at least f^6 = 2^-960, still
// normal; a product that falls below belongs to a weight under 2^-55.  The product of both sides' would not
// be, so each has its reciprocal (seven instructions; scaling both for one took eighteen).
__device__ __forceinline__ double w9_pair(const double eps, const double p[8], const double m[8])
{
    double Q[2], T[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const double *d = h ? m : p;
        double s[5] = {w9_is<0>(d[0], d[1], d[2], d[3]), w9_is<1>(d[1], d[2], d[3], d[4]),
                       w9_is<2>(d[2], d[3], d[4], d[5]), w9_is<1>(d[6], d[5], d[4], d[3]),
                       w9_is<0>(d[7], d[6], d[5], d[4])};
        const double mx = fmax(fmax(fmax(s[0], s[1]), fmax(s[2], s[3])), fmax(s[4], eps));
        const double sc = inv_pow2(mx);
        const double fl = fmax(eps * sc, 0x1p-160);
#pragma unroll
        for (int k = 0; k < 5; k++) {
            const double q = fma(s[k], sc, fl);
            s[k] = q * q;
        }
        const double p01 = s[0] * s[1], p012 = p01 * s[2], s34 = s[3] * s[4], s234 = s[2] * s34;
        const double P0 = s[1] * s234, P1 = s[0] * s234, P2 = p01 * s34, P3 = p012 * s[4], P4 = p012 * s[3];
        const double D = fma(5., P4, fma(40., P3, fma(60., P2, fma(20., P1, P0))));
        double v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = fma(6., d[k + 2], fma(-4., d[k + 1] + d[k + 3], d[k] + d[k + 4]));
        const double r = fma(3., v[1], -2. * v[2]);
        Q[h] = quotient(fma(0.25 * P4, fma(3., v[3], r), fma(2. * P3, r, fma(9. * P2, v[1], (0.6 * P0) * v[0]))), D);
        T[h] = fma(39., v[1], fma(-14., v[2], 3. * v[3]));
    }
    return fma(1. / 280., T[0] - T[1], Q[1] - Q[0]);
}

__device__ __forceinline__ double pressure(const Consts &k, double rho, double u, double v, double w, double e)
{
    return fabs(rho * (k.gamma - 1) / k.upsilon * (e - 0.5 * ((u * u) + (v * v) + (w * w))));
}

// p = |rho (gamma-1)/Upsilon (e - |u|^2/2)| with the constant ratio folded (CalcValues,
// src/Functions.c:2445-2459)
__device__ __forceinline__ double pressure_fast(const Consts &k, double rho, double u, double v, double w, double e)
{
    return fabs(rho * k.gm1_ups * (e - 0.5 * ((u * u) + (v * v) + (w * w))));
}

}  // namespace shx
