// Device helpers shared by the pGM HIP kernels (gfx950): the box and its minimum image, the Gaussian-damped
// Ewald pair kernels G_n, cardinal B-splines, sub-wavefront reductions.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pgmhip {

constexpr double kPi = 3.14159265358979323846;
constexpr double kSqrtPi = 1.7724538509055160273;
constexpr double kTwoOverSqrtPi = 1.1283791670955125739;

// Reduced triclinic box (rows a = (ax,0,0), b = (bx,by,0), c = (cx,cy,cz)) and its inverse
// recip[k][a] = (H^-1)_{k a}: the fractional coordinate a of r is sum_k r_k recip[k][a].
template<class T>
struct BoxT {
    T ax, bx, by, cx, cy, cz;
    T iax, iby, icz;   // 1/ax, 1/by, 1/cz
    T recip[3][3];
};

// Minimum image in a reduced triclinic box: c first, then b, then a (core/pgm_math.h:153-160).  rint of a
// product instead of round of a quotient: they differ only at half-box ties, far outside any pair cutoff.
template<class T>
__device__ __forceinline__ void minImage(T& x, T& y, T& z, const BoxT<T>& b) {
    T k = rint(z*b.icz);
    x -= k*b.cx;
    y -= k*b.cy;
    z -= k*b.cz;
    k = rint(y*b.iby);
    x -= k*b.bx;
    y -= k*b.by;
    k = rint(x*b.iax);
    x -= k*b.ax;
}

// The gfx950 dispatcher deals workgroups to its 8 XCDs round-robin (workgroup b runs on XCD b % 8), and each
// XCD has an L2 of its own.  This renumbering gives XCD x a contiguous range of logical blocks, so the kernels
// over spatially sorted atoms gather their partners from one slab of the system per L2 instead of from all of
// it.  A bijection of [0, gridDim.x) for any grid size.  reverse: each XCD walks its range from the end (the
// part of the data that the pass before, walking forward, touched last comes first).
__device__ __forceinline__ int xcdBlock(int b, int nb, bool reverse) {
    constexpr int kXcd = 8;
    const int per = nb/kXcd, rem = nb%kXcd, x = b%kXcd, local = b/kXcd;
    const int l = reverse ? (x < rem ? per : per-1)-local : local;
    return x < rem ? x*(per+1)+l : rem*(per+1)+(x-rem)*per+l;
}
__device__ __forceinline__ int xcdBlock(bool reverse = false) {
    return xcdBlock((int) blockIdx.x, (int) gridDim.x, reverse);
}

// Precision traits of the pair kernels: series length below a r = 1 and the damping cut beyond which the
// erfc(a r) part is dropped (the reference's GPU constants, openmm/platforms/common/src/CommonPGMKernels.cpp:351-352).
template<class T>
struct PairPrec;
template<>
struct PairPrec<float> {
    static constexpr int kSeries = 12;
    static constexpr float kDampCut = 4.5f;
};
template<>
struct PairPrec<double> {
    static constexpr int kSeries = 15;
    static constexpr double kDampCut = 6.0;
};

__device__ __forceinline__ float erfT(float x) { return erff(x); }
__device__ __forceinline__ double erfT(double x) { return erf(x); }
__device__ __forceinline__ float expT(float x) { return __expf(x); }
__device__ __forceinline__ double expT(double x) { return exp(x); }
__device__ __forceinline__ float rsqrtT(float x) { return __frsqrt_rn(x); }
__device__ __forceinline__ double rsqrtT(double x) { return rsqrt(x); }

// exp(x^2) erfc(x) for 0 <= x <= 4.5 in FP32 (the range of the pair kernels): t Q(t) with t = 1/(1 + x/2) and
// Q a degree-8 polynomial fitted to exp(x^2) erfc(x)/t on that range (minimax relative error by iteratively
// reweighted least squares, pgm-md_amd/csrc/erfcx_fit.py; 1.6e-8 for the fit, below 3e-7 evaluated in FP32).
// erfc(x) is this times exp(-x^2), the factor the kernels' Gaussian term needs too, so that a kernel evaluation
// takes one exp per width instead of two.  v_rcp instead of a division.
__device__ __forceinline__ float erfcxFast(float x) {
    const float t = __builtin_amdgcn_rcpf(fmaf(0.5f, x, 1.0f));
    float p = -4.658861831e-02f;
    p = fmaf(t, p, 2.203130424e-01f);
    p = fmaf(t, p, -3.455681503e-01f);
    p = fmaf(t, p, 1.038070619e-01f);
    p = fmaf(t, p, 1.041026637e-01f);
    p = fmaf(t, p, 1.415342391e-01f);
    p = fmaf(t, p, 2.605046332e-01f);
    p = fmaf(t, p, 2.796235681e-01f);
    p = fmaf(t, p, 2.822715342e-01f);
    return t*p;
}

// erfc(x) for 0 <= x <= 4.5 in FP32: erfcxFast(x) exp(-x^2); relative error below 2.5e-6 in FP32 (the rounding
// of x^2 in the exponent dominates near x = 4.5).
__device__ __forceinline__ float erfcFast(float x) { return erfcxFast(x)*__expf(-x*x); }

// A polynomial in FP64, C::at(k) its coefficients from the highest degree down.  Each comes from scalar registers, tied
// to the accumulator so that it is set right before its step: left to itself the compiler keeps the coefficients in
// vector registers through the pair loops and copies each into the accumulator first (the passes at 200 registers, two
// wavefronts per SIMD, two vector instructions per step).
template<int N, class C>
__device__ __forceinline__ double hornerD(double x) {
    double p = C::at(0);
#pragma unroll
    for (int k = 1; k < N; k++) {
        double c = C::at(k);
        asm("" : "+s"(c) : "v"(p));
        p = fma(p, x, c);
    }
    return p;
}

// 1/(m! (2m+2k+1)) and its sign in the series below.
constexpr double erfSeriesCoef(int m, int k) {
    double f = (m & 1) ? -1.0 : 1.0;
    for (int i = 2; i <= m; i++)
        f /= i;
    return f/(2*m+2*k+1);
}

template<int K>
struct ErfSeriesD {
    __device__ static constexpr double at(int k) { return erfSeriesCoef(PairPrec<double>::kSeries-1-k, K); }
};

// B_n of erf(a r)/r, n < NMAX, by the series in s = (a r)^2 (valid for s < 1; no cancellation at short
// range): B_n = (2a/sqrt(pi)) (2a^2)^n sum_m (-s)^m / (m! (2m+2n+1)) (core/pgm_math.h:31-49, docs/spec.md Sec. 4).
template<class T, int NMAX, int K = 0>
__device__ __forceinline__ void erfSeries(T a, T s, T* B, T scale = T(1)) {
    constexpr int NS = PairPrec<T>::kSeries;
    if constexpr (K == 0)
        scale = T(kTwoOverSqrtPi)*a;
    if constexpr (sizeof(T) == sizeof(double))
        B[K] = scale*hornerD<NS, ErfSeriesD<K>>(s);
    else {
        T acc = T(erfSeriesCoef(NS-1, K));
#pragma unroll
        for (int m = NS-2; m >= 0; m--)
            acc = fma(acc, s, T(erfSeriesCoef(m, K)));
        B[K] = scale*acc;
    }
    if constexpr (K+1 < NMAX)
        erfSeries<T, NMAX, K+1>(a, s, B, scale*(T(2)*a*a));
}

// FP64 building blocks of the pair kernels, without library calls, divisions or square roots (one of the library's erfc,
// exp, sqrt or divide is 20 to 100 instructions with range branches, and a pair needs seven of them).
// 1/sqrt(v), v > 0: v_rsq_f64 and one third-order step, within 1 ulp.
__device__ __forceinline__ double rsqD(double v) {
    const double y = __builtin_amdgcn_rsq(v), e = fma(-v*y, y, 1.0);
    return fma(y*e, fma(0.375, e, 0.5), y);
}
// 1/v: v_rcp_f64 and one third-order step.
__device__ __forceinline__ double rcpD(double v) {
    const double y = __builtin_amdgcn_rcp(v), e = fma(-v, y, 1.0);
    return fma(y, fma(e, e, e), y);
}
struct ExpD {
    __device__ static constexpr double at(int k) {
        constexpr double c[12] = {
            2.51003765231722297e-08, 2.76137965905202207e-07, 2.75572684786510166e-06, 2.48015364068864706e-05,
            1.98412698630417918e-04, 1.38888889058726541e-03, 8.33333333333006500e-03, 4.16666666666513641e-02,
            1.66666666666666685e-01, 0.5, 1.0, 1.0,
        };
        return c[k];
    }
};
// exp(-(s + lo)), s >= 0, |lo| << 1: 2^n e^r, |r| <= ln 2 / 2, the Taylor terms to r^2 exact and a degree-8 polynomial
// (interpolation at Chebyshev nodes, 3.4e-17; erfcx_fit.py) for the rest.
__device__ __forceinline__ double expNegD(double s, double lo) {
    const double k = rint(s*-1.44269504088896339);
    const double r = fma(k, -2.31904681384629956e-17, fma(k, -6.93147180559945286e-01, -s)-lo);
    const double p = hornerD<12, ExpD>(r);
    return __builtin_amdgcn_ldexp(p, (int) k);
}
// v^-1/2 and exp(-s) in the pair type.
__device__ __forceinline__ float rsqT(float v) { return __frsqrt_rn(v); }
__device__ __forceinline__ double rsqT(double v) { return rsqD(v); }
__device__ __forceinline__ float expNegT(float s) { return __expf(-s); }
__device__ __forceinline__ double expNegT(double s) { return expNegD(s, 0.0); }
struct ErfcxD {
    __device__ static constexpr double at(int k) {
        constexpr double c[25] = {
            -1.13943375763050212e-09, -3.46738851456642846e-11, 1.13616654610778355e-08, 6.46203952133591332e-09,
            -5.36892735908146752e-08, -7.41995606534354225e-08, 1.39210995565696456e-07, 4.54263266929759196e-07,
            -6.74541909340868799e-09, -1.96813742087781588e-06, -2.33199485288660954e-06, 6.75738056042995359e-06,
            1.82443088002155857e-05, -1.95333384577758414e-05, -1.12604824560452857e-04, 5.83080587353616042e-05,
            7.02693723353389125e-04, -4.39208300105815538e-04, -4.81878552320537737e-03, 8.39304430476217091e-03,
            2.83615501319947304e-02, -1.71251145246119035e-01, 4.53914116648096055e-01, -8.04651849439148137e-01,
            1.05403182030571796e+00,
        };
        return c[k];
    }
};
// exp(x^2) erfc(x) for x >= 0: P(u)/(x + K), u = (x - K)/(x + K), K = 2.5, the Chebyshev expansion of
// (x + K) exp(x^2) erfc(x) in u to degree 24 (erfcx_fit.py; remainder 3.3e-17; the mapping of Shepherd and Laframboise,
// Math. Comp. 36, 249, 1981), 4.5e-16 evaluated in FP64.
__device__ __forceinline__ double erfcxD(double x) {
    const double t = rcpD(x+2.5), u = (x-2.5)*t;
    return hornerD<25, ErfcxD>(u)*t;
}

// B_n of erfc(c r)/r (SIGN = 1) or erf(c r)/r (-1) by the upward recursion, from s = (c r)^2 with its rounding error lo,
// 1/r and 1/r^2: for erfc all terms are positive (core/pgm_math.h:63-71), for erf s >= 1.
template<int SIGN, int NMAX>
__device__ __forceinline__ void gaussKernelsD(double c, double s, double lo, double r, double rinv, double ir2,
                                              double* B) {
    const double e = expNegD(s, lo), erfcV = erfcxD(c*r)*e;
    const double g = kTwoOverSqrtPi*c*e, twoC2 = 2.0*c*c;
    B[0] = (SIGN > 0 ? erfcV : 1.0-erfcV)*rinv;
    double scale = SIGN;
#pragma unroll
    for (int k = 1; k < NMAX; k++) {
        B[k] = fma(double(2*k-1), B[k-1], scale*g)*ir2;
        scale *= twoC2;
    }
}

// B_n of erf(a r)/r and erfc(a r)/r in FP32: 1/r from v_rsq, erfc(x) from erfcxFast(x) and the exp(-x^2) of the
// Gaussian term, no divisions.
template<int NMAX>
__device__ __forceinline__ void erfKernelsF(float a, float r, float rinv, float* B) {
    const float x = a*r, s = x*x;
    if (s < 1.0f) {
        erfSeries<float, NMAX>(a, s, B);
        return;
    }
    const float e = __expf(-s);
    const float g = float(kTwoOverSqrtPi)*a*e;
    const float ir2 = rinv*rinv;
    B[0] = (1.0f-erfcxFast(x)*e)*rinv;
    float scale = 1.0f;
    const float twoA2 = 2.0f*a*a;
#pragma unroll
    for (int k = 1; k < NMAX; k++) {
        B[k] = (float(2*k-1)*B[k-1]-scale*g)*ir2;
        scale *= twoA2;
    }
}

template<int NMAX>
__device__ __forceinline__ void erfcKernelsF(float a, float r, float rinv, float* B) {
    const float x = a*r;
    const float e = __expf(-x*x);   // shared by erfc(x) and the Gaussian term
    const float g = float(kTwoOverSqrtPi)*a*e;
    const float ir2 = rinv*rinv;
    B[0] = erfcxFast(x)*e*rinv;
    float scale = 1.0f;
    const float twoA2 = 2.0f*a*a;
#pragma unroll
    for (int k = 1; k < NMAX; k++) {
        B[k] = (float(2*k-1)*B[k-1]+scale*g)*ir2;
        scale *= twoA2;
    }
}

// G_n for FP32 from r^2 and rg_i + rg_j (a = (rg_i + rg_j)^-1/2): the branches of pairKernelsD below.
template<int NMAX>
__device__ __forceinline__ void pairKernelsF(float rgSum, float beta, float r2, float* G) {
    const float a = __builtin_amdgcn_rsqf(rgSum);
    const float rinv = __builtin_amdgcn_rsqf(r2);
    const float r = r2*rinv;
    float B[NMAX];
    if (a*r < 1.0f) {
        erfSeries<float, NMAX>(a, (a*r)*(a*r), G);
        erfKernelsF<NMAX>(beta, r, rinv, B);
    }
    else {
        erfcKernelsF<NMAX>(beta, r, rinv, G);
        if (a*r < PairPrec<float>::kDampCut)
            erfcKernelsF<NMAX>(a, r, rinv, B);
        else {
#pragma unroll
            for (int k = 0; k < NMAX; k++)
                B[k] = 0.0f;
        }
    }
#pragma unroll
    for (int k = 0; k < NMAX; k++)
        G[k] -= B[k];
}

// G_n = B_n[erf(a r)/r] - B_n[erf(beta r)/r] for n < NMAX in FP64, a = rgSum^-1/2: the series difference for a r < 1,
// the erfc form Bc(beta) - Bc(a) beyond (core/pgm_math.h:78-92), the Bc(a) part dropped beyond a r > kDampCut.  The
// exponents (c r)^2 carry their rounding error along, so that exp(-(c r)^2) is good to an ulp at every distance.
// Against the library's functions the setup pass over 88 million pairs took 1,403 us instead of 1,552, when it also
// stored 32 bytes of kernels per pair.
template<int NMAX>
__device__ __forceinline__ void pairKernelsD(double rgSum, double beta, double r2In, double* G) {
    const double r2 = fmax(r2In, 1e-280);   // coincident atoms: r = 0 in the series
    const double a = rsqD(rgSum), rinv = rsqD(r2), r = r2*rinv;
    double ir2 = rinv*rinv;
    ir2 = fma(ir2, fma(-r2, ir2, 1.0), ir2);
    const double b2 = beta*beta, b2Lo = fma(beta, beta, -b2);
    const double sb = b2*r2, sbLo = fma(b2, r2, -sb)+b2Lo*r2;
    double B[NMAX];
    if (a*r < 1.0) {
        erfSeries<double, NMAX>(a, (a*r)*(a*r), G);
        if (sb < 1.0)
            erfSeries<double, NMAX>(beta, sb, B);
        else
            gaussKernelsD<-1, NMAX>(beta, sb, sbLo, r, rinv, ir2, B);
    }
    else {
        gaussKernelsD<1, NMAX>(beta, sb, sbLo, r, rinv, ir2, G);
        if (a*r < PairPrec<double>::kDampCut) {
            const double a2 = a*a, sa = r2*a2;
            gaussKernelsD<1, NMAX>(a, sa, fma(-sa, rgSum, r2)*a2, r, rinv, ir2, B);
        }
        else {
#pragma unroll
            for (int k = 0; k < NMAX; k++)
                B[k] = 0;
        }
    }
#pragma unroll
    for (int k = 0; k < NMAX; k++)
        G[k] -= B[k];
}

// GVDW, the Gaussian-density van der Waals (core/gvdw_kernel.h): G(y) = F(y)/y^6 and H(y) = G'(y)/y with
// F = A^2 + g^2/2, A = erf y - (2y/sqrt(pi))(1 + 2y^2/3) e^{-y^2}, g = (4y^3/(3 sqrt(pi))) e^{-y^2}.  Below
// y = 0.6 the Taylor series of G in y^2 (coefficients c_k of G/C0, C0 = 8/(9 pi): exact rationals, from the
// series of erf and exp), above it the closed form.
template<class T>
__device__ __forceinline__ void gvdwG(T y, T& G, T& H) {
    constexpr double c[15] = {1.0, -2.0, 58.0/25, -188.0/105, 2222.0/2205, -1532.0/3465, 64244.0/405405,
                              -162056.0/3378375, 1587734.0/126351225, -211108.0/72747675,
                              11902564.0/19860115275.0, -611992.0/5465775315.0, 755028172.0/39529267903125.0,
                              -213335384.0/71152682225625.0, 15291334888.0/35078272337233125.0};
    const T c0 = T(8.0/(9.0*kPi)), s = y*y;
    if (y < T(0.6)) {
        T g = T(c[14]), h = T(28.0*c[14]);
#pragma unroll
        for (int k = 13; k >= 0; k--) {
            g = g*s+T(c[k]);
            if (k > 0)
                h = h*s+T(2.0*k*c[k]);
        }
        G = c0*g;
        H = c0*h;
        return;
    }
    const T e = expT(-s), isp = T(1.0/kSqrtPi);
    const T A = erfT(y)-T(2)*isp*y*(T(1)+T(2.0/3.0)*s)*e, g = T(4.0/3.0)*isp*s*y*e;
    const T dA = T(8.0/3.0)*isp*s*s*e, dg = T(4)*isp*s*(T(1)-T(2.0/3.0)*s)*e;
    const T F = A*A+T(0.5)*g*g, dF = T(2)*A*dA+g*dg, y6 = s*s*s;
    G = F/y6;
    H = (dF/y6-T(6)*F/(y6*y))/y;
}

// One GVDW pair: U = A exp(-B y^2) (Gaussian) or A exp(-B y) (Slater) - C6 b^6 G(y), y = b r; returns U and
// dEdR = -(1/r) dU/dr (the force on i is dEdR (r_i - r_j)); the Slater force at r = 0 is 0
// (core/gvdw_kernel.h:58-77).
template<class T>
__device__ __forceinline__ T gvdwPair(T r, T bij, T A, T C6, T B, bool slater, T& dEdR) {
    const T y = bij*r, b2 = bij*bij, b6 = b2*b2*b2;
    T erep, drep;
    if (!slater) {
        erep = A*expT(-B*y*y);
        drep = T(-2)*B*b2*erep;
    }
    else {
        erep = A*expT(-B*y);
        drep = r > T(0) ? -B*bij*erep/r : T(0);
    }
    T G, H;
    gvdwG<T>(y, G, H);
    dEdR = C6*b6*b2*H-drep;
    return erep-C6*b6*G;
}

// Cardinal B-spline weights of order P at fraction fr on the grid points (base - j), j = 0..P-1
// (core/pgm_core.cpp:131-152): th[j] = M_P(fr + j), dth[j] = M_P'(fr + j), d2th[j] = M_P''(fr + j).
template<class T, int P>
__device__ __forceinline__ void bsplines(T fr, T* th, T* dth, T* d2th) {
    T m[P+1];   // m[j] = M_k(fr + j), rebuilt for k = 1..P
    T m1[P+1], m2[P+1];
#pragma unroll
    for (int j = 0; j <= P; j++)
        m[j] = m1[j] = m2[j] = T(0);
    m[0] = T(1);
#pragma unroll
    for (int k = 2; k <= P; k++) {
        if (k == P-1) {
#pragma unroll
            for (int j = 0; j <= P; j++)
                m2[j] = m[j];   // M_{P-2}
        }
        if (k == P) {
#pragma unroll
            for (int j = 0; j <= P; j++)
                m1[j] = m[j];   // M_{P-1}
        }
        T nxt[P+1];
        const T inv = T(1)/T(k-1);
#pragma unroll
        for (int j = 0; j <= P; j++) {
            const T hi = (j < k-1 ? m[j] : T(0));
            const T lo = (j >= 1 && j-1 < k-1 ? m[j-1] : T(0));
            nxt[j] = (j < k ? ((fr+T(j))*hi+(T(k)-fr-T(j))*lo)*inv : T(0));
        }
#pragma unroll
        for (int j = 0; j <= P; j++)
            m[j] = nxt[j];
    }
#pragma unroll
    for (int j = 0; j < P; j++) {
        th[j] = m[j];
        const T a1 = (j < P-1 ? m1[j] : T(0)), b1 = (j >= 1 ? m1[j-1] : T(0));
        dth[j] = a1-b1;
        const T a2 = (j < P-2 ? m2[j] : T(0)), b2 = (j >= 1 && j-1 < P-2 ? m2[j-1] : T(0)),
                c2 = (j >= 2 && j-2 < P-2 ? m2[j-2] : T(0));
        d2th[j] = a2-T(2)*b2+c2;
    }
}

// Sum over the L lanes of a sub-wavefront group (L a power of two dividing 64).
template<int L, class V>
__device__ __forceinline__ V groupSum(V v) {
#pragma unroll
    for (int o = L/2; o > 0; o >>= 1)
        v += __shfl_xor(v, o, L);
    return v;
}

// slot = atomicAdd(&count[key], 1) for every lane with valid set, with one atomic per distinct key in the
// wavefront: spatially sorted atoms share a key across most of a wavefront, and atomics on one address
// serialize.  Every lane of the wavefront calls it (valid = false where there is no item); the slots within a
// key follow lane order, and those of different wavefronts the order of their atomics.
__device__ __forceinline__ int waveSlot(int* count, int key, bool valid) {
    const int lane = threadIdx.x & 63;
    unsigned long long pending = __ballot(valid);
    int slot = 0;
    while (pending != 0ull) {
        const int leader = __ffsll((unsigned long long) pending)-1;
        const int lk = __shfl(key, leader, 64);
        const unsigned long long same = __ballot(valid && key == lk) & pending;
        int base = 0;
        if (lane == leader)
            base = atomicAdd(&count[lk], __popcll(same));
        base = __shfl(base, leader, 64);
        if ((same >> lane) & 1ull)
            slot = base+__popcll(same & ((1ull << lane)-1ull));
        pending &= ~same;
    }
    return slot;
}

// Block-wide sum of a double (blockDim.x a multiple of 64, <= 1024); the result is valid in thread 0.
__device__ __forceinline__ double blockSum(double v, double* smem) {
    v = groupSum<64>(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0)
        smem[w] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0)
        for (int k = 0; k < (int) (blockDim.x >> 6); k++)
            r += smem[k];
    __syncthreads();
    return r;
}

__device__ __forceinline__ double groupMax64(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ double blockMax(double v, double* smem) {
    v = groupMax64(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0)
        smem[w] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0)
        for (int k = 0; k < (int) (blockDim.x >> 6); k++)
            r = fmax(r, smem[k]);
    __syncthreads();
    return r;
}

// Vector types of the two precisions: xyz + charge (positions) or xyz + 0 (dipoles), 16 or 32 bytes.
template<class T>
struct Vec4;
template<>
struct Vec4<float> {
    typedef float4 type;
};
template<>
struct Vec4<double> {
    typedef double4 type;
};
template<class T>
struct Vec2;
template<>
struct Vec2<float> {
    typedef float2 type;
};
template<>
struct Vec2<double> {
    typedef double2 type;
};

}   // namespace pgmhip
