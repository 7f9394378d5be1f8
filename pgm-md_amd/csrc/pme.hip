// Smooth PME of charges and dipoles (Essmann 1995; dipoles as Sagui 2004) for pGM on gfx950.
//
//   bin/place  atoms binned into grid bricks once per evaluation, their base points and fractions stored in brick
//              order (core/pgm_core.cpp:123-153 convention: M_p(fr + j) on grid point base - j);
//   spread     one workgroup per brick accumulates q theta theta theta + e . grad(theta theta theta) into a 64-bit
//              fixed-point LDS tile (brick + order-1 halo) with LDS atomics, then adds the tile to the grid
//              (core/pgm_core.cpp:191-207; replaces the reference's 64-bit fixed-point global atomics);
//   transform  in-house mixed-radix Stockham FFTs in LDS: z (two real lines per complex transform), y, then x fused
//              with the influence function, the energy and the k-space strain (core/pgm_core.cpp:213-237), and back;
//   gather     E = -grad phi at the atoms, from LDS tiles of the bricks; at the end of an evaluation also the
//              reciprocal forces -[q grad phi + (grad grad phi) . d] (core/pgm_core.cpp:241-264, 453-487);
//   x-planes   small and many grids: spread + z + y, and y + z + gather, one x-plane per workgroup in LDS.
#include "kernels.hpp"
#include "pairfield.hpp"

#include <type_traits>

#include <algorithm>
#include <stdexcept>
#include <string>

namespace pgmhip {

// The stages of a transform of length K.  Narrow: radix 4 while it divides, then 2, 3, 5, 7.  Wide: the factorisation
// into radices 2..10 with the fewest stages (every stage is a pass of the lines through LDS and a barrier), of those
// the one whose largest radix is smallest, and in it first the radix with the fewest factors of two (the first stage
// writes with a stride of its radix, and an odd stride of 8- or 16-byte elements touches every bank).
FftPlan makePlan(int K, bool wide) {
    if (K >= 4096)
        throw std::runtime_error("pgm_hip: PME grid dimension "+std::to_string(K)+" above 4095");
    int best[12], nbest = 0;
    int m = K;
    for (int r : {4, 2, 3, 5, 7})
        while (m%r == 0 && nbest < 12) {
            best[nbest++] = r;
            m /= r;
        }
    if (m != 1)
        throw std::runtime_error("pgm_hip: PME grid dimension "+std::to_string(K)+
                                 " must factor into 2, 3, 5 and 7");
    if (wide && K > 1) {
        int cur[12], bestMax = 0;
        nbest = 0;
        auto search = [&](auto&& self, int rest, int most, int n) -> void {
            if (rest == 1) {
                if (nbest == 0 || n < nbest || (n == nbest && cur[0] < bestMax)) {
                    std::copy(cur, cur+n, best);
                    nbest = n;
                    bestMax = cur[0];
                }
                return;
            }
            if (nbest > 0 && n+1 > nbest)
                return;
            for (int r = std::min(most, rest); r >= 2; r--)   // non-increasing radices: each multiset once
                if (rest%r == 0) {
                    cur[n] = r;
                    self(self, rest/r, r, n+1);
                }
        };
        search(search, K, 10, 0);
        std::stable_sort(best, best+nbest, [](int x, int y) { return (x & -x) < (y & -y); });
    }
    FftPlan p{};
    if (nbest > (int) (sizeof(p.stage)/sizeof(p.stage[0])))
        throw std::runtime_error("pgm_hip: PME grid dimension has too many factors");
    p.nstage = nbest;
    int ns = 1;
    for (int st = 0; st < nbest; st++) {
        p.stage[st].radix = best[st];
        p.stage[st].byM = fastDiv(K/best[st]);
        p.stage[st].byNs = fastDiv(ns);
        ns *= best[st];
    }
    return p;
}

namespace {

constexpr int kBlock = 256;
constexpr int kPlaneList = 2048;      // atoms listed at a time by the x-plane spread and gather

template<class T2>
__device__ __forceinline__ T2 cmul(T2 a, T2 b) {
    T2 r;
    r.x = a.x*b.x-a.y*b.y;
    r.y = a.x*b.y+a.y*b.x;
    return r;
}

template<class T2>
__device__ __forceinline__ T2 cadd(T2 a, T2 b) {
    T2 r;
    r.x = a.x+b.x;
    r.y = a.y+b.y;
    return r;
}

template<class T2>
__device__ __forceinline__ T2 csub(T2 a, T2 b) {
    T2 r;
    r.x = a.x-b.x;
    r.y = a.y-b.y;
    return r;
}

template<class T2>
__device__ __forceinline__ T2 conjIf(T2 a, bool c) {
    if (c)
        a.y = -a.y;
    return a;
}

// -i a (forward) or +i a (inverse)
template<class T2>
__device__ __forceinline__ T2 rotQuarter(T2 a, bool inverse) {
    T2 r;
    if (inverse) {
        r.x = -a.y;
        r.y = a.x;
    }
    else {
        r.x = a.y;
        r.y = -a.x;
    }
    return r;
}

// cos(2 pi k/R) and sin(2 pi k/R) for R = 5 or 7 and 0 < k < R (cos(2 pi/5) = (sqrt 5 - 1)/4, and so on).
__host__ __device__ constexpr double cosTwoPi(int R, int k) {
    const int q = k <= R/2 ? k : R-k;
    return R == 5 ? (q == 1 ? 0.30901699437494742410 : -0.80901699437494742410)
                  : (q == 1 ? 0.62348980185873353053 : q == 2 ? -0.22252093395631440429 : -0.90096886790241912624);
}
__host__ __device__ constexpr double sinTwoPi(int R, int k) {
    const int q = k <= R/2 ? k : R-k;
    const double s = R == 5 ? (q == 1 ? 0.95105651629515357212 : 0.58778525229247312917)
                            : (q == 1   ? 0.78183148246802980871
                               : q == 2 ? 0.97492791218182360702
                                        : 0.43388373911755812048);
    return k <= R/2 ? s : -s;
}

// e^{-/+ 2 pi i k/N} (forward/inverse) times a, for compile-time constants cos and sin of 2 pi k/N.
template<class T2, class T>
__device__ __forceinline__ T2 rotate(T2 a, T c, T sn, bool inverse) {
    const T s = inverse ? sn : -sn;
    T2 r;
    r.x = a.x*c-a.y*s;
    r.y = a.x*s+a.y*c;
    return r;
}

// The R-point transform of v[0..R) in registers, natural order.  R is a compile-time constant, so the values stay in
// registers: with a runtime radix the array was indexed at run time and lived in per-lane scratch memory.  2, 3, 4
// directly; 5 and 7 in closed form; 6, 8 and 10 as two transforms of the even and odd values, 9 as three of three.
template<int R, class T>
__device__ __forceinline__ void dft(typename Vec2<T>::type* v, bool inverse) {
    typedef typename Vec2<T>::type T2;
    if constexpr (R == 2) {
        const T2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    }
    else if constexpr (R == 3) {
        const T c = T(-0.5), sn = (inverse ? T(0.86602540378443864676) : T(-0.86602540378443864676));
        const T2 sum = cadd(v[1], v[2]), d = csub(v[1], v[2]);
        T2 t, u;
        t.x = v[0].x+c*sum.x;
        t.y = v[0].y+c*sum.y;
        u.x = -sn*d.y;
        u.y = sn*d.x;
        v[0] = cadd(v[0], sum);
        v[1] = cadd(t, u);
        v[2] = csub(t, u);
    }
    else if constexpr (R == 4) {
        const T2 s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
        const T2 s13 = cadd(v[1], v[3]), d13 = rotQuarter(csub(v[1], v[3]), inverse);
        v[0] = cadd(s02, s13);
        v[1] = cadd(d02, d13);
        v[2] = csub(s02, s13);
        v[3] = csub(d02, d13);
    }
    else if constexpr (R == 5 || R == 7) {
        // with a_r = v_r + v_{R-r}, b_r = v_r - v_{R-r} (r = 1..h, h = (R-1)/2), X_s = v_0 + sum a_r cos(2 pi rs/R)
        // -/+ i sum b_r sin(2 pi rs/R) and X_{R-s} the other sign (forward/inverse); the cosines and sines fold to
        // constants
        constexpr int h = (R-1)/2;
        T2 a[h+1], b[h+1];
        const T2 v0 = v[0];
        T2 x0 = v0;
#pragma unroll
        for (int r = 1; r <= h; r++) {
            a[r] = cadd(v[r], v[R-r]);
            b[r] = csub(v[r], v[R-r]);
            x0 = cadd(x0, a[r]);
        }
        v[0] = x0;
#pragma unroll
        for (int s = 1; s <= h; s++) {
            T2 A = v0, B;
            B.x = B.y = T(0);
#pragma unroll
            for (int r = 1; r <= h; r++) {
                const T c = T(cosTwoPi(R, (r*s)%R)), sn = T(sinTwoPi(R, (r*s)%R));
                A.x += c*a[r].x;
                A.y += c*a[r].y;
                B.x += sn*b[r].x;
                B.y += sn*b[r].y;
            }
            const T2 rb = rotQuarter(B, inverse);
            v[s] = cadd(A, rb);
            v[R-s] = csub(A, rb);
        }
    }
    else if constexpr (R == 9) {
        // cos and sin of 2 pi k/9, k = 1, 2, 4
        constexpr double c1 = 0.76604444311897803520, s1 = 0.64278760968653932632;
        constexpr double c2 = 0.17364817766693034885, s2 = 0.98480775301220805937;
        constexpr double c4 = -0.93969262078590838405, s4 = 0.34202014332566873304;
        T2 y[3][3];
#pragma unroll
        for (int n = 0; n < 3; n++) {
            T2 t[3] = {v[n], v[n+3], v[n+6]};
            dft<3, T>(t, inverse);
#pragma unroll
            for (int k = 0; k < 3; k++)
                y[k][n] = t[k];
        }
        y[1][1] = rotate(y[1][1], T(c1), T(s1), inverse);
        y[1][2] = rotate(y[1][2], T(c2), T(s2), inverse);
        y[2][1] = rotate(y[2][1], T(c2), T(s2), inverse);
        y[2][2] = rotate(y[2][2], T(c4), T(s4), inverse);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            dft<3, T>(y[k], inverse);
#pragma unroll
            for (int q = 0; q < 3; q++)
                v[k+3*q] = y[k][q];
        }
    }
    else {
        static_assert(R == 6 || R == 8 || R == 10, "radices 2..10");
        constexpr int H = R/2;
        // cos and sin of 2 pi k/R, 0 < k < R/2
        constexpr double c[5] = {1.0, R == 6 ? 0.5 : R == 8 ? 0.70710678118654752440 : 0.80901699437494742410,
                                 R == 6 ? -0.5 : R == 8 ? 0.0 : 0.30901699437494742410,
                                 R == 8 ? -0.70710678118654752440 : -0.30901699437494742410, -0.80901699437494742410};
        constexpr double sn[5] = {0.0,
                                  R == 6 ? 0.86602540378443864676 : R == 8 ? 0.70710678118654752440
                                                                           : 0.58778525229247312917,
                                  R == 6 ? 0.86602540378443864676 : R == 8 ? 1.0 : 0.95105651629515357212,
                                  R == 8 ? 0.70710678118654752440 : 0.95105651629515357212, 0.58778525229247312917};
        T2 e[H], o[H];
#pragma unroll
        for (int k = 0; k < H; k++) {
            e[k] = v[2*k];
            o[k] = v[2*k+1];
        }
        dft<H, T>(e, inverse);
        dft<H, T>(o, inverse);
#pragma unroll
        for (int k = 0; k < H; k++) {
            const T2 w = k == 0 ? o[0] : (R == 8 && k == 2) ? rotQuarter(o[2], inverse)
                                                           : rotate(o[k], T(c[k]), T(sn[k]), inverse);
            v[k] = cadd(e[k], w);
            v[k+H] = csub(e[k], w);
        }
    }
}

// One radix-R stage of a Stockham FFT over nlines lines of length K in LDS (line l at buf[l*K]): butterfly j of
// line l takes in[j + r*m], r < R (m = K/R), each times w^(r*kk*span) (kk = j mod Ns, span = K/(Ns*R); all 1 in the
// first stage), and writes out[(j div Ns)*Ns*R + kk + s*Ns], s < R.
template<int R, class T>
__device__ __forceinline__ void fftStage(const typename Vec2<T>::type* src, typename Vec2<T>::type* dst,
                                         const typename Vec2<T>::type* tw, int K, int Ns, FastDiv byM, FastDiv byNs,
                                         int nlines, bool inverse) {
    typedef typename Vec2<T>::type T2;
    const int m = K/R, span = K/(Ns*R);
    for (int idx = threadIdx.x; idx < nlines*m; idx += blockDim.x) {
        const int l = byM.div(idx), j = idx-l*m;
        const T2* in = src+l*K+j;
        T2 v[R];
#pragma unroll
        for (int r = 0; r < R; r++)
            v[r] = in[r*m];
        int at = l*K+j*R;
        if (Ns > 1) {
            const int jq = byNs.div(j), kk = j-jq*Ns;
#pragma unroll
            for (int r = 1; r < R; r++)
                v[r] = cmul(v[r], conjIf(tw[r*kk*span], inverse));
            at = l*K+jq*Ns*R+kk;
        }
        dft<R, T>(v, inverse);
        T2* out = dst+at;
#pragma unroll
        for (int r = 0; r < R; r++)
            out[r*Ns] = v[r];
    }
}

// Mixed-radix Stockham FFT of nlines lines of length K held in LDS (line l at buf[l*K]); tw[j] =
// e^{-2 pi i j/K} and the plan in LDS too.  Returns the buffer that holds the result (natural order).  WIDE: the
// radices above 5 besides 7 are compiled in (they are most of the code, which a launch of few blocks fetches anew).
template<class T, bool WIDE>
__device__ __forceinline__ typename Vec2<T>::type* ldsFft(typename Vec2<T>::type* src, typename Vec2<T>::type* dst,
                                                          const typename Vec2<T>::type* tw, const FftPlan* p, int K,
                                                          int nlines, bool inverse) {
    typedef typename Vec2<T>::type T2;
    int Ns = 1;
    const int nstage = __builtin_amdgcn_readfirstlane(p->nstage);
    for (int st = 0; st < nstage; st++) {
        const int R = __builtin_amdgcn_readfirstlane(p->stage[st].radix);
        FastDiv byM, byNs;
        byM.magic = __builtin_amdgcn_readfirstlane(p->stage[st].byM.magic);
        byNs.magic = __builtin_amdgcn_readfirstlane(p->stage[st].byNs.magic);
        auto stage = [&](auto r) { fftStage<r(), T>(src, dst, tw, K, Ns, byM, byNs, nlines, inverse); };
        if constexpr (WIDE) {
            switch (R) {
            case 6:
                stage(std::integral_constant<int, 6>{});
                break;
            case 8:
                stage(std::integral_constant<int, 8>{});
                break;
            case 9:
                stage(std::integral_constant<int, 9>{});
                break;
            case 10:
                stage(std::integral_constant<int, 10>{});
                break;
            default:
                break;
            }
        }
        switch (R) {
        case 2:
            stage(std::integral_constant<int, 2>{});
            break;
        case 3:
            stage(std::integral_constant<int, 3>{});
            break;
        case 4:
            stage(std::integral_constant<int, 4>{});
            break;
        case 5:
            stage(std::integral_constant<int, 5>{});
            break;
        case 7:
            stage(std::integral_constant<int, 7>{});
            break;
        default:
            break;
        }
        __syncthreads();
        T2* t = src;
        src = dst;
        dst = t;
        Ns *= R;
    }
    return src;
}

// for i in [0, count) over the block: store(i, load(i)), U loads in flight per thread before the first store.
template<int U, class V, class Load, class Store>
__device__ __forceinline__ void blockCopy(int count, Load load, Store store) {
    for (int i0 = threadIdx.x; i0 < count; i0 += U*blockDim.x) {
        V v[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i0+u*(int) blockDim.x < count)
                v[u] = load(i0+u*(int) blockDim.x);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i0+u*(int) blockDim.x < count)
                store(i0+u*(int) blockDim.x, v[u]);
    }
}

// ---------------------------------------------------------------------------------------- binning

template<class T>
__device__ __forceinline__ void fracGrid(const double4& p, const BoxT<double>& box, const PmeGrid& g, int base[3],
                                         T fr[3]) {
#pragma unroll
    for (int a = 0; a < 3; a++) {
        double t = p.x*box.recip[0][a]+p.y*box.recip[1][a]+p.z*box.recip[2][a];
        t -= floor(t);
        const double w = g.K[a]*t;
        int b = (int) floor(w);
        fr[a] = (T) (w-b);
        if (b >= g.K[a])
            b -= g.K[a];
        base[a] = b;
    }
}

// The grid and box of a system: the single one, or from the batch table.
template<bool BATCH>
__device__ __forceinline__ const PmeSys* sysEntry(const PmeSel& ps, int sys) {
    return BATCH ? ps.table+sys : nullptr;
}

template<class T, bool BATCH>
__global__ void kPmeBin(int n, const double4* posD, PmeSel ps, int* brickOf, int* slot, int* brickCount) {
    const int s = blockIdx.x*blockDim.x+threadIdx.x;
    const bool valid = s < n;   // no early return: the whole wavefront takes part in waveSlot
    int b = 0;
    if (valid) {
        const PmeSys* se = sysEntry<BATCH>(ps, BATCH ? ps.sysOf[s] : 0);
        const PmeGrid& g = BATCH ? se->g : ps.g;
        const BoxT<double>& box = BATCH ? se->box : ps.box;
        int base[3];
        T fr[3];
        fracGrid<T>(posD[s], box, g, base, fr);
        b = ((base[0]/g.brick)*g.nb[1]+base[1]/g.brick)*g.nb[2]+base[2]/g.brick+(BATCH ? se->brickOff : 0);
        brickOf[s] = b;
    }
    const int k = waveSlot(brickCount, b, valid);
    if (valid)
        slot[s] = k;
}

template<class T, bool BATCH>
__global__ void kPmePlace(int n, const double4* posD, PmeSel ps, const int* brickOf, const int* slot,
                          const int* brickStart, PmeAtom<T>* atoms) {
    const int s = blockIdx.x*blockDim.x+threadIdx.x;
    if (s >= n)
        return;
    const PmeSys* se = sysEntry<BATCH>(ps, BATCH ? ps.sysOf[s] : 0);
    const PmeGrid& g = BATCH ? se->g : ps.g;
    const BoxT<double>& box = BATCH ? se->box : ps.box;
    PmeAtom<T> a;
    fracGrid<T>(posD[s], box, g, a.base, a.fr);
    a.s = s;
    a.fr[3] = T(0);
    atoms[brickStart[brickOf[s]]+slot[s]] = a;
}

// The weights of one dimension at the row j (a run-time index) by selection.  The values pass through an empty asm
// first: without it the compiler turns the selection back into an array indexed at run time, in scratch memory.
__device__ __forceinline__ void opaque(float& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void opaque(double& v) { asm volatile("" : "+v"(v)); }
template<class T, int P>
__device__ __forceinline__ T pick(const T* v, int j) {
    T r = v[0];
#pragma unroll
    for (int k = 1; k < P; k++) {
        T c = v[k];
        opaque(c);
        r = j == k ? c : r;
    }
    return r;
}

// ---------------------------------------------------------------------------------------- spreading

// The P contributions A t3 + C u3 of one grid row into the fixed-point tile (row[-j3]; FP64: the second words
// wordStride on).
template<class T, int P, bool FAST>
__device__ __forceinline__ void spreadRow(unsigned long long* row, int wordStride, T A, T C, const T* t3,
                                          const T* u3) {
#pragma unroll
    for (int j3 = 0; j3 < P; j3++) {
        const T v = A*t3[j3]+C*u3[j3];
        long long hi, lo;
        if (FAST)
            toFixedFast<T>(v, hi, lo);
        else
            toFixed<T>(v, hi, lo);
        atomicAdd(row-j3, (unsigned long long) hi);
        if (GridFixed<T>::words == 2)
            atomicAdd(row+wordStride-j3, (unsigned long long) lo);
    }
}

// The same onto a periodic row of K2 points, from point z downwards.
template<class T, int P, bool FAST>
__device__ __forceinline__ void spreadRow(unsigned long long* row, int wordStride, int z, int K2, T A, T C,
                                          const T* t3, const T* u3) {
#pragma unroll
    for (int j3 = 0; j3 < P; j3++) {
        const T v = A*t3[j3]+C*u3[j3];
        long long hi, lo;
        if (FAST)
            toFixedFast<T>(v, hi, lo);
        else
            toFixed<T>(v, hi, lo);
        const int at = z-j3+(z < j3 ? K2 : 0);
        atomicAdd(row+at, (unsigned long long) hi);
        if (GridFixed<T>::words == 2)
            atomicAdd(row+wordStride+at, (unsigned long long) lo);
    }
}

// TAN: instead of the charges and dipoles, the change of their grid density when every atom moves by g_s and its
// dipole changes by d'_s: the density q theta(r - r_s) + d . grad_s theta moves to first order by
// (q g + d') . grad_s theta + g^T (grad_s grad_s theta) d, i.e. a dipole q g + d' and a symmetric second moment
// (g d^T + d g^T)/2 on the second spline derivatives.
//
// The charge and dipole grids (not TAN) accumulate in 64-bit fixed point, GridFixed<T>::scale units per grid
// unit, in the LDS tile and in the global grid: integer additions commute, so the grid, and everything after
// it, is the same bit for bit whatever the order of the atomics (the reference's 2^32 fixed-point grid,
// core/cuda/pgm_cuda.cu:52,67-69,804-843).  Each contribution is rounded to the fixed-point unit once.  TAN
// grids, whose scale follows the caller's cotangent, accumulate in FP64 in the tile and in T in the grid.
//
// G lanes per atom, each taking the rows j1 = lane, lane + G, ... of P x P points.  Every lane evaluates the atom's
// splines from its record (about 250 instructions).  Bound by the flush: with it taken out the pass takes 40% of its
// time at 112^3 and half at 216^3, with the LDS additions taken out 65%.
template<class T, int P, bool TAN, bool BATCH, int G>
__global__ void __launch_bounds__(kBlock) kSpread(PmeSel ps, const int* __restrict__ brickStart,
                                                  const PmeAtom<T>* __restrict__ atoms,
                                                  const typename Vec4<T>::type* __restrict__ dip,
                                                  const typename Vec4<T>::type* __restrict__ posq, int withQ,
                                                  T* __restrict__ gridAll, long long* __restrict__ fixedAll,
                                                  CgSkip skip,
                                                  const typename Vec4<T>::type* __restrict__ dipDot,
                                                  const typename Vec4<T>::type* __restrict__ disp) {
    typedef typename Vec4<T>::type T4;
    // The TAN tile accumulates in FP64 for both precisions: ds_add_f64 is several times faster than ds_add_f32
    // on gfx950, and the FP64 sums lose nothing.
    constexpr int W = GridFixed<T>::words;
    extern __shared__ __align__(16) unsigned char smemRaw[];
    double* tile = reinterpret_cast<double*>(smemRaw);
    unsigned long long* tileI = reinterpret_cast<unsigned long long*>(smemRaw);   // W words per point, apart
    if (skip())
        return;
    const int bid = blockIdx.x;
    const PmeSys* se = sysEntry<BATCH>(ps, BATCH ? ps.brickSys[bid] : 0);
    const PmeGrid& g = BATCH ? se->g : ps.g;
    const BoxT<double>& box = BATCH ? se->box : ps.box;
    T* __restrict__ grid = TAN ? gridAll+(BATCH ? se->gridOff : 0) : nullptr;
    long long* __restrict__ gridI = TAN ? nullptr : fixedAll+(BATCH ? se->gridOff : 0);
    const int lb = bid-(BATCH ? se->brickOff : 0);
    const int b2 = lb%g.nb[2], b1 = (lb/g.nb[2])%g.nb[1], b0 = lb/(g.nb[2]*g.nb[1]);
    const int E = g.brick+P-1, E3 = E*E*E;
    const int lo0 = b0*g.brick-(P-1), lo1 = b1*g.brick-(P-1), lo2 = b2*g.brick-(P-1);
    for (int i = threadIdx.x; i < (TAN ? 1 : W)*E3; i += blockDim.x)
        tileI[i] = 0ull;
    __syncthreads();
    T rc[3][3];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int a = 0; a < 3; a++)
            rc[k][a] = (T) (g.K[a]*box.recip[k][a]);
    const int first = brickStart[bid], count = brickStart[bid+1]-first;
    for (int it = threadIdx.x; it < count*G; it += blockDim.x) {
        const int k = first+it/G, lane = it%G;
        if (lane >= P)
            continue;
        const PmeAtom<T> a = atoms[k];
        const T4 d = dip[a.s];
        const T q = (withQ || TAN) ? posq[a.s].w : T(0);
        T e[3], D[3], S[3][3];
#pragma unroll
        for (int c = 0; c < 3; c++)
            e[c] = d.x*rc[0][c]+d.y*rc[1][c]+d.z*rc[2][c];
        if (TAN) {
            const T4 dd = dipDot[a.s], gs = disp[a.s];
            T ga[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                ga[c] = gs.x*rc[0][c]+gs.y*rc[1][c]+gs.z*rc[2][c];
                D[c] = q*ga[c]+dd.x*rc[0][c]+dd.y*rc[1][c]+dd.z*rc[2][c];
            }
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int b = 0; b < 3; b++)
                    S[c][b] = T(0.5)*(ga[c]*e[b]+ga[b]*e[c]);
        }
        T t1s[P], u1s[P], v1s[P], t2s[P], u2s[P], v2s[P], t3[P], u3[P], v3[P];
        bsplines<T, P>(a.fr[0], t1s, u1s, v1s);
        bsplines<T, P>(a.fr[1], t2s, u2s, v2s);
        bsplines<T, P>(a.fr[2], t3, u3, v3);
        // one test, the same for the whole wavefront, admits every contribution to the conversion of a few
        // instructions; anything beyond its range, or not finite, takes the general one
        const bool fast = !TAN && __all(fixedFits<T>(q, e, a.fr));
        const int l1b = a.base[1]-lo1, l2b = a.base[2]-lo2;
        for (int j1 = lane; j1 < P; j1 += G) {
            const T t1 = pick<T, P>(t1s, j1), u1 = pick<T, P>(u1s, j1), v1 = TAN ? pick<T, P>(v1s, j1) : T(0);
            const int l0 = a.base[0]-j1-lo0;
#pragma unroll
            for (int j2 = 0; j2 < P; j2++) {
                const T t2 = t2s[j2], u2 = u2s[j2];
                T A, C, V = 0;
                if (TAN) {
                    const T v2 = v2s[j2];
                    A = D[0]*u1*t2+D[1]*t1*u2+S[0][0]*v1*t2+S[1][1]*t1*v2+T(2)*S[0][1]*u1*u2;
                    C = D[2]*t1*t2+T(2)*(S[0][2]*u1*t2+S[1][2]*t1*u2);
                    V = S[2][2]*t1*t2;
                }
                else {
                    A = (q*t1+e[0]*u1)*t2+e[1]*t1*u2;
                    C = e[2]*t1*t2;
                }
                const int r0 = (l0*E+(l1b-j2))*E+l2b;
                if (TAN) {
#pragma unroll
                    for (int j3 = 0; j3 < P; j3++)
                        atomicAdd(tile+r0-j3, (double) (A*t3[j3]+C*u3[j3]+V*v3[j3]));
                }
                else if (fast)
                    spreadRow<T, P, true>(tileI+r0, E3, A, C, t3, u3);
                else
                    spreadRow<T, P, false>(tileI+r0, E3, A, C, t3, u3);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < E3; i += blockDim.x) {
        if (TAN ? tile[i] == 0.0 : (tileI[i] == 0ull && (W == 1 || tileI[E3+i] == 0ull)))
            continue;
        const int x2 = i%E, x1 = (i/E)%E, x0 = i/(E*E);
        int g0 = lo0+x0, g1 = lo1+x1, g2 = lo2+x2;
        g0 += (g0 < 0 ? g.K[0] : 0);
        g0 -= (g0 >= g.K[0] ? g.K[0] : 0);
        g1 += (g1 < 0 ? g.K[1] : 0);
        g1 -= (g1 >= g.K[1] ? g.K[1] : 0);
        g2 += (g2 < 0 ? g.K[2] : 0);
        g2 -= (g2 >= g.K[2] ? g.K[2] : 0);
        const size_t at = ((size_t) g0*g.K[1]+g1)*g.K[2]+g2;
        if (TAN)
            unsafeAtomicAdd(grid+at, (T) tile[i]);
        else {
            atomicAdd(reinterpret_cast<unsigned long long*>(gridI+at), tileI[i]);
            if (W == 2)
                atomicAdd(reinterpret_cast<unsigned long long*>(gridI+ps.fixedStride+at), tileI[E3+i]);
        }
    }
}

// ---------------------------------------------------------------------------------------- transforms

// The twiddles and the plan of the transform along axis into LDS (plan: kPlanInts ints), no barrier.
template<class T>
__device__ __forceinline__ void loadTransform(typename Vec2<T>::type* tw, FftPlan* plan,
                                              const typename Vec2<T>::type* __restrict__ twAll, const FftGroup& grp,
                                              int axis) {
    const int K = grp.g.K[axis], off = grp.twOff+(axis > 0 ? grp.g.K[0] : 0)+(axis > 1 ? grp.g.K[1] : 0);
    for (int i = threadIdx.x; i < K; i += blockDim.x)
        tw[i] = twAll[off+i];
    if (threadIdx.x < kPlanInts)
        reinterpret_cast<int*>(plan)[threadIdx.x] = reinterpret_cast<const int*>(&grp.plan[axis])[threadIdx.x];
}

// The group (grid shape) of this block.
__device__ __forceinline__ const FftGroup& groupOf(const FftGroup* groups, const int* blockGroup) {
    return groups[blockGroup ? blockGroup[blockIdx.x] : 0];
}

// z: two real lines per complex FFT, unpacked into their half spectra.
// Forward: from the fixed-point grid when fixedAll is set (each word zeroed once read: the grid is clean for
// the next spread), else from the real grid.
template<class T, bool INVERSE, bool WIDE>
__global__ void __launch_bounds__(kBlock) kFftZ(const FftGroup* __restrict__ groups,
                                                const int* __restrict__ blockGroup,
                                                T* __restrict__ realAll, typename Vec2<T>::type* __restrict__ cplxAll,
                                                const typename Vec2<T>::type* __restrict__ twAll, CgSkip skip,
                                                long long* __restrict__ fixedAll, size_t fixedStride) {
    typedef typename Vec2<T>::type T2;
    extern __shared__ __align__(16) unsigned char smemRaw[];
    if (skip())
        return;
    const FftGroup& grp = groupOf(groups, blockGroup);
    const PmeGrid& g = grp.g;
    const int ngrid = grp.ngrid, pairsPerBlock = grp.pz, blk = (int) blockIdx.x-grp.blk0[0];
    T* __restrict__ real = realAll+grp.realOff;
    T2* __restrict__ cplx = cplxAll+grp.cplxOff;
    const FastDiv byK2 = grp.byK2, byKh = grp.byKh;
    const int K = g.K[2], Kh = g.K3h, nlines = ngrid*g.K[0]*g.K[1];
    FftPlan* plan = reinterpret_cast<FftPlan*>(smemRaw);
    T2* tw = reinterpret_cast<T2*>(plan+1);
    T2* b0 = tw+K;
    T2* b1 = b0+pairsPerBlock*K;
    loadTransform<T>(tw, plan, twAll, grp, 2);
    const int pair0 = blk*pairsPerBlock;
    const int npairs = min(pairsPerBlock, (nlines+1)/2-pair0);
    auto store = [&](int i, const T2& z) { b0[i] = z; };
    if (!INVERSE && fixedAll) {
        long long* fixed = fixedAll+grp.realOff;
        auto load = [&](int i) {
            const int l = byK2.div(i), k = i-l*K;
            const int la = 2*(pair0+l), lb = la+1;
            T2 z;
            z.x = fromFixed<T>(fixed+(size_t) la*K+k, fixedStride);
            z.y = (lb < nlines ? fromFixed<T>(fixed+(size_t) lb*K+k, fixedStride) : T(0));
            return z;
        };
        blockCopy<4, T2>(npairs*K, load, store);
        __syncthreads();   // every word read
        const int nwords = min(2*npairs, nlines-2*pair0)*K;   // the block's rows are contiguous
        for (int i = threadIdx.x; i < nwords; i += blockDim.x) {
            fixed[(size_t) 2*pair0*K+i] = 0;
            if (GridFixed<T>::words == 2)
                fixed[fixedStride+(size_t) 2*pair0*K+i] = 0;
        }
    }
    else if (!INVERSE) {
        auto load = [&](int i) {
            const int l = byK2.div(i), k = i-l*K;
            const int la = 2*(pair0+l), lb = la+1;
            T2 z;
            z.x = real[(size_t) la*K+k];
            z.y = (lb < nlines ? real[(size_t) lb*K+k] : T(0));
            return z;
        };
        blockCopy<4, T2>(npairs*K, load, store);
    }
    else {
        auto load = [&](int i) {
            const int l = byK2.div(i), k = i-l*K;
            const int la = 2*(pair0+l), lb = la+1;
            const bool lower = k < Kh;
            const int kk = lower ? k : K-k;
            T2 X = cplx[(size_t) la*Kh+kk];
            T2 Y;
            Y.x = Y.y = T(0);
            if (lb < nlines)
                Y = cplx[(size_t) lb*Kh+kk];
            if (kk == 0 || 2*kk == K) {
                X.y = T(0);
                Y.y = T(0);
            }
            T2 z;
            if (lower) {
                z.x = X.x-Y.y;
                z.y = X.y+Y.x;
            }
            else {
                z.x = X.x+Y.y;
                z.y = Y.x-X.y;
            }
            return z;
        };
        blockCopy<4, T2>(npairs*K, load, store);
    }
    __syncthreads();
    T2* res = ldsFft<T, WIDE>(b0, b1, tw, plan, K, npairs, INVERSE);
    if (!INVERSE) {
        for (int i = threadIdx.x; i < npairs*Kh; i += blockDim.x) {
            const int l = byKh.div(i), k = i-l*Kh;
            const int la = 2*(pair0+l), lb = la+1;
            const T2 Z = res[l*K+k], Zc = res[l*K+(k == 0 ? 0 : K-k)];
            T2 X, Y;
            X.x = T(0.5)*(Z.x+Zc.x);
            X.y = T(0.5)*(Z.y-Zc.y);
            Y.x = T(0.5)*(Z.y+Zc.y);
            Y.y = T(-0.5)*(Z.x-Zc.x);
            cplx[(size_t) la*Kh+k] = X;
            if (lb < nlines)
                cplx[(size_t) lb*Kh+k] = Y;
        }
    }
    else {
        for (int i = threadIdx.x; i < npairs*K; i += blockDim.x) {
            const int l = byK2.div(i), k = i-l*K;
            const int la = 2*(pair0+l), lb = la+1;
            const T2 z = res[i];
            real[(size_t) la*K+k] = z.x;
            if (lb < nlines)
                real[(size_t) lb*K+k] = z.y;
        }
    }
}

// y: lines of K2 for fixed (x, z), a tile of consecutive z per block.
template<class T, bool INVERSE, bool WIDE>
__global__ void __launch_bounds__(kBlock) kFftY(const FftGroup* __restrict__ groups,
                                                const int* __restrict__ blockGroup,
                                                typename Vec2<T>::type* __restrict__ cplxAll,
                                                const typename Vec2<T>::type* __restrict__ twAll, CgSkip skip) {
    typedef typename Vec2<T>::type T2;
    extern __shared__ __align__(16) unsigned char smemRaw[];
    if (skip())
        return;
    const FftGroup& grp = groupOf(groups, blockGroup);
    const PmeGrid& g = grp.g;
    const int zt = grp.zy, blk = (int) blockIdx.x-grp.blk0[1];
    const FastDiv byZ = grp.byZy;
    T2* __restrict__ cplx = cplxAll+grp.cplxOff;
    const int K = g.K[1], Kh = g.K3h;
    const int ntile = (Kh+zt-1)/zt;
    const int x = blk/ntile, z0 = (blk%ntile)*zt;
    const int nl = min(zt, Kh-z0);
    FftPlan* plan = reinterpret_cast<FftPlan*>(smemRaw);
    T2* tw = reinterpret_cast<T2*>(plan+1);
    T2* b0 = tw+K;
    T2* b1 = b0+zt*K;
    loadTransform<T>(tw, plan, twAll, grp, 1);
    // (the tile indexed by its full width: a last tile may be narrower)
    T2* __restrict__ row = cplx+(size_t) x*K*Kh+z0;
    blockCopy<4, T2>(zt*K,
                     [&](int i) {
                         const int y = byZ.div(i), l = i-y*zt;
                         return l < nl ? row[(size_t) y*Kh+l] : T2{};
                     },
                     [&](int i, const T2& v) {
                         const int y = byZ.div(i), l = i-y*zt;
                         b0[l*K+y] = v;
                     });
    __syncthreads();
    T2* res = ldsFft<T, WIDE>(b0, b1, tw, plan, K, nl, INVERSE);
    for (int i = threadIdx.x; i < zt*K; i += blockDim.x) {
        const int y = byZ.div(i), l = i-y*zt;
        if (l < nl)
            row[(size_t) y*Kh+l] = res[l*K+y];
    }
}

// The z and y transforms of one x-plane in LDS.  Forward: bufA holds the plane's real rows two per complex line
// (npairs lines of K2); their z spectra are unpacked transposed (a line of K1 per z), y transformed and written to
// cplx.  Inverse: the other way round; returns the buffer that holds the real rows two per complex line.
template<class T>
struct PlaneLds {   // two plans, the twiddles of y and z, two plane buffers
    typedef typename Vec2<T>::type T2;
    FftPlan* plan;
    T2 *twY, *twZ, *bufA, *bufB;
    __device__ __forceinline__ PlaneLds(unsigned char* smem, const PmeGrid& g) {
        plan = reinterpret_cast<FftPlan*>(smem);
        twY = reinterpret_cast<T2*>(plan+2);
        twZ = twY+g.K[1];
        bufA = twZ+g.K[2];
        bufB = bufA+max(((g.K[1]+1)/2)*g.K[2], g.K3h*g.K[1]);
    }
    __device__ __forceinline__ void load(const T2* __restrict__ twAll, const FftGroup& grp) {
        loadTransform<T>(twY, plan, twAll, grp, 1);
        loadTransform<T>(twZ, plan+1, twAll, grp, 2);
    }
};

template<class T, bool WIDE>
__device__ __forceinline__ void planeForward(const PmeGrid& g, const FftGroup& grp, const PlaneLds<T>& m,
                                             typename Vec2<T>::type* __restrict__ cplx) {
    typedef typename Vec2<T>::type T2;
    const int K1 = g.K[1], K2 = g.K[2], Kh = g.K3h, npairs = (K1+1)/2;
    T2 *bufA = m.bufA, *bufB = m.bufB;
    T2* res = ldsFft<T, WIDE>(bufA, bufB, m.twZ, m.plan+1, K2, npairs, false);
    T2* other = (res == bufA ? bufB : bufA);
    for (int i = threadIdx.x; i < npairs*Kh; i += blockDim.x) {
        const int l = grp.byKh.div(i), k = i-l*Kh;
        const T2 Z = res[l*K2+k], Zc = res[l*K2+(k == 0 ? 0 : K2-k)];
        T2 X, Y;
        X.x = T(0.5)*(Z.x+Zc.x);
        X.y = T(0.5)*(Z.y-Zc.y);
        Y.x = T(0.5)*(Z.y+Zc.y);
        Y.y = T(-0.5)*(Z.x-Zc.x);
        other[k*K1+2*l] = X;
        if (2*l+1 < K1)
            other[k*K1+2*l+1] = Y;
    }
    __syncthreads();
    T2* res2 = ldsFft<T, WIDE>(other, res, m.twY, m.plan, K1, Kh, false);
    for (int i = threadIdx.x; i < K1*Kh; i += blockDim.x) {
        const int y = grp.byKh.div(i), z = i-y*Kh;
        cplx[i] = res2[z*K1+y];
    }
}

template<class T, bool WIDE>
__device__ __forceinline__ typename Vec2<T>::type* planeInverse(const PmeGrid& g, const FftGroup& grp,
                                                                const typename Vec2<T>::type* __restrict__ cplx,
                                                                const PlaneLds<T>& m) {
    typedef typename Vec2<T>::type T2;
    const int K1 = g.K[1], K2 = g.K[2], Kh = g.K3h, npairs = (K1+1)/2;
    T2 *bufA = m.bufA, *bufB = m.bufB;
    blockCopy<4, T2>(K1*Kh, [&](int i) { return cplx[i]; },
                     [&](int i, const T2& v) {
                         const int y = grp.byKh.div(i), z = i-y*Kh;
                         bufA[z*K1+y] = v;
                     });
    __syncthreads();
    T2* res = ldsFft<T, WIDE>(bufA, bufB, m.twY, m.plan, K1, Kh, true);
    T2* other = (res == bufA ? bufB : bufA);
    for (int i = threadIdx.x; i < npairs*K2; i += blockDim.x) {
        const int l = grp.byK2.div(i), k = i-l*K2;
        const int ya = 2*l, yb = ya+1;
        const bool lower = k < Kh;
        const int kk = lower ? k : K2-k;
        T2 X = res[kk*K1+ya];
        T2 Y;
        Y.x = Y.y = T(0);
        if (yb < K1)
            Y = res[kk*K1+yb];
        if (kk == 0 || 2*kk == K2) {
            X.y = T(0);
            Y.y = T(0);
        }
        T2 z;
        if (lower) {
            z.x = X.x-Y.y;
            z.y = X.y+Y.x;
        }
        else {
            z.x = X.x+Y.y;
            z.y = Y.x-X.y;
        }
        other[l*K2+k] = z;
    }
    __syncthreads();
    return ldsFft<T, WIDE>(other, res, m.twZ, m.plan+1, K2, npairs, true);
}

// z and y of one x-plane per block (many small grids): forward, the plane's real rows two per complex transform
// along z (as kFftZ), their half spectra unpacked transposed (a line of K1 per z), then the y transforms; inverse
// the other way round.  The plane goes through global memory once each way instead of twice.
template<class T, bool INVERSE, bool WIDE>
__global__ void __launch_bounds__(kPlaneThreads) kFftZY(const FftGroup* __restrict__ groups,
                                                        const int* __restrict__ blockGroup,
                                                        T* __restrict__ realAll,
                                                        typename Vec2<T>::type* __restrict__ cplxAll,
                                                        const typename Vec2<T>::type* __restrict__ twAll,
                                                        CgSkip skip, long long* __restrict__ fixedAll,
                                                        size_t fixedStride) {
    typedef typename Vec2<T>::type T2;
    extern __shared__ __align__(16) unsigned char smemRaw[];
    if (skip())
        return;
    const FftGroup& grp = groupOf(groups, blockGroup);
    const PmeGrid& g = grp.g;
    const int K1 = g.K[1], K2 = g.K[2], Kh = g.K3h;
    const int plane = (int) blockIdx.x-grp.blk0[3];   // grid * K0 + x
    T* __restrict__ real = realAll+grp.realOff+(size_t) plane*K1*K2;
    T2* __restrict__ cplx = cplxAll+grp.cplxOff+(size_t) plane*K1*Kh;
    const int npairs = (K1+1)/2;
    PlaneLds<T> m(smemRaw, g);
    m.load(twAll, grp);
    if (!INVERSE) {
        long long* fixed = fixedAll ? fixedAll+grp.realOff+(size_t) plane*K1*K2 : nullptr;
        for (int i = threadIdx.x; i < npairs*K2; i += blockDim.x) {
            const int l = grp.byK2.div(i), k = i-l*K2;
            const int ya = 2*l, yb = ya+1;
            T2 z;
            if (fixed) {
                z.x = takeFixed<T>(fixed+(size_t) ya*K2+k, fixedStride);
                z.y = (yb < K1 ? takeFixed<T>(fixed+(size_t) yb*K2+k, fixedStride) : T(0));
            }
            else {
                z.x = real[(size_t) ya*K2+k];
                z.y = (yb < K1 ? real[(size_t) yb*K2+k] : T(0));
            }
            m.bufA[i] = z;
        }
        __syncthreads();
        planeForward<T, WIDE>(g, grp, m, cplx);
    }
    else {
        const T2* res = planeInverse<T, WIDE>(g, grp, cplx, m);
        for (int i = threadIdx.x; i < npairs*K2; i += blockDim.x) {
            const int l = grp.byK2.div(i), k = i-l*K2;
            const int ya = 2*l, yb = ya+1;
            const T2 z = res[i];
            real[(size_t) ya*K2+k] = z.x;
            if (yb < K1)
                real[(size_t) yb*K2+k] = z.y;
        }
    }
}

// ---------------------------------------------------------------------------------------- x-plane passes
//
// Many small grids, or one small one: a block owns an x-plane of a grid, and the spreading and the gathering happen
// where the plane's transforms do, in its LDS.  Forward (kPlaneSpread): the plane's points accumulate the rows of
// the atoms that reach it, in the same 64-bit fixed point as kSpread's tiles (the sums are integers, so the grid
// is the same bit for bit), then the z and y transforms run on it: no grid of fixed-point words in memory, no
// global atomics on it, no clearing.  Inverse (kPlaneGather): the plane's potential is gathered from LDS as it
// leaves the z transform, each atom's share of the field from this plane written to its own place (out, P per atom,
// summed by the reader): no grid of potentials in memory, no gather of 36 unaligned rows per atom.  A solve is three
// launches (with kFftXConv) instead of seven.  Measured at 64 snapshots (2,735 planes, 207,831 atoms): spread + z + y
// 128 -> 91 us, y + z + gather 90 -> 77 us per pass.  Bound by LDS latency and barriers: few wavefronts per plane.
//
// The atoms that reach plane x have x base points x..x+P-1 (mod K0): a run of slabs of bricks, contiguous in brick
// order, and a second run where the range wraps.  planeAtoms walks the two runs in chunks: the chunk's atoms that
// do reach the plane are listed in LDS (with their row j1 = base - x), then work(atom in brick order, j1) runs with
// every lane busy, one lane per atom and its P rows of P points.
template<class T, int P, class Work>
__device__ __forceinline__ void planeAtoms(const PmeGrid& g, int brickOff, int x, const int* __restrict__ brickStart,
                                           const PmeAtom<T>* __restrict__ atoms, int* list, int* counter, Work work) {
    constexpr int cap = kPlaneList;
    const int K0 = g.K[0], nb12 = g.nb[1]*g.nb[2];
    for (int wrap = 0; wrap < 2; wrap++) {
        const int lo = wrap ? 0 : x, hi = wrap ? x+P-1-K0 : min(x+P-1, K0-1);
        if (hi < lo)
            continue;   // block-uniform
        const int first = brickStart[brickOff+(lo/g.brick)*nb12];
        const int last = brickStart[brickOff+min(hi/g.brick+1, g.nb[0])*nb12];
        for (int c0 = first; c0 < last; c0 += cap) {
            const int c1 = min(c0+cap, last);
            __syncthreads();   // the list of the chunk before is used up
            if (threadIdx.x == 0)
                *counter = 0;
            __syncthreads();
            for (int k0 = c0; k0 < c1; k0 += blockDim.x) {
                const int k = k0+(int) threadIdx.x;
                bool in = false;
                int j1 = 0;
                if (k < c1) {
                    const int b = atoms[k].base[0];
                    j1 = b-x+(wrap ? K0 : 0);
                    in = (wrap ? b < x : b >= x) && j1 < P;
                }
                const unsigned long long m = __ballot(in);
                const int lane = threadIdx.x & 63;
                int at = 0;
                if (lane == 0 && m != 0ull)
                    at = atomicAdd(counter, __popcll(m));
                at = __shfl(at, 0, 64)+__popcll(m & ((1ull << lane)-1ull));
                if (in)
                    list[at] = (k-c0)*8+j1;
            }
            __syncthreads();
            const int items = *counter;
            for (int it = threadIdx.x; it < items; it += blockDim.x) {
                const int e = list[it];
                work(c0+(e >> 3), e & 7);
            }
        }
    }
    __syncthreads();
}

// The grid of a plane block: its group, the plane of the stacked grids, its system.
template<bool BATCH>
__device__ __forceinline__ const PmeSys* planeSystem(const PmeSel& ps, const FftGroup& grp, int grid) {
    return BATCH ? ps.table+ps.groupSys[grp.boxOff+grid] : nullptr;
}

// PAIR: the first planes blocks are that; the others run the rows of the CG field pass, which need nothing of it.  Few
// planes leave most CUs idle, and the field pass of a small system takes less than a plane: a CG product of 8,600 atoms
// 59 -> 49 us, of 12,000 62 -> 51, of 24,000 91 -> 78.
template<class T, int P, bool BATCH, bool WIDE, bool PAIR>
__global__ void __launch_bounds__(kPlaneThreads) kPlaneSpread(const FftGroup* __restrict__ groups,
                                                              const int* __restrict__ blockGroup, PmeSel ps,
                                                              const int* __restrict__ brickStart,
                                                              const PmeAtom<T>* __restrict__ atoms,
                                                              const typename Vec4<T>::type* __restrict__ posq,
                                                              PlaneSolves<T> solves,
                                                              typename Vec2<T>::type* __restrict__ cplxAll,
                                                              const typename Vec2<T>::type* __restrict__ twAll,
                                                              CgSkip skip, PairFieldArgs<T> pair, int planes,
                                                              int pairSh) {
    typedef typename Vec4<T>::type T4;
    typedef typename Vec2<T>::type T2;
    constexpr int W = GridFixed<T>::words;
    extern __shared__ __align__(16) unsigned char smemRaw[];
    __shared__ __align__(16) int list[kPlaneList+4];   // and its counter: whole 16 bytes before the dynamic LDS
    if (skip())
        return;
    if constexpr (PAIR) {
        if ((int) blockIdx.x >= planes) {
            const int gid = xcdBlock((int) blockIdx.x-planes, (int) gridDim.x-planes, pair.reverse)*blockDim.x+threadIdx.x;
            if constexpr (sizeof(T) == sizeof(float)) {
                if (pair.otf) {
                    pairFieldRowOtf<4, BATCH>(gid, pairSh, pair);
                    return;
                }
            }
            pairFieldRow<T, 4, BATCH>(gid, pairSh, pair);
            return;
        }
    }
    const FftGroup& grp = groupOf(groups, blockGroup);
    const PmeGrid& g = grp.g;
    const int K0 = g.K[0], K1 = g.K[1], K2 = g.K[2], Kh = g.K3h, KK = K1*K2;
    const int plane = (int) blockIdx.x-grp.blk0[3], gi = plane/K0, x = plane-gi*K0;
    const PmeSys* se = planeSystem<BATCH>(ps, grp, gi);
    const BoxT<double>& box = BATCH ? se->box : ps.box;
    const int solve = blockIdx.y;
    const T4* __restrict__ dip = solves.dip[solve];
    const bool withQ = solves.withQ[solve] != 0;
    T2* __restrict__ cplx = cplxAll+solve*solves.cplxStride+grp.cplxOff+(size_t) plane*K1*Kh;
    const int npairs = (K1+1)/2;
    PlaneLds<T> m(smemRaw, g);
    m.load(twAll, grp);
    // the fixed-point plane lies over bufB: read into bufA before the transforms use it
    unsigned long long* tile = reinterpret_cast<unsigned long long*>(m.bufB);
    for (int i = threadIdx.x; i < W*KK; i += blockDim.x)
        tile[i] = 0ull;
    T rc[3][3];
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int a = 0; a < 3; a++)
            rc[k][a] = (T) (g.K[a]*box.recip[k][a]);
    planeAtoms<T, P>(g, BATCH ? se->brickOff : 0, x, brickStart, atoms, list, list+kPlaneList, [&](int k, int j1) {
        const PmeAtom<T> a = atoms[k];
        const T4 d = dip[a.s];
        const T q = withQ ? posq[a.s].w : T(0);
        T t1s[P], u1s[P], t2[P], u2[P], t3[P], u3[P], w[P];
        bsplines<T, P>(a.fr[0], t1s, u1s, w);
        bsplines<T, P>(a.fr[1], t2, u2, w);
        bsplines<T, P>(a.fr[2], t3, u3, w);
        const T t1 = pick<T, P>(t1s, j1), u1 = pick<T, P>(u1s, j1);
        const int y0 = a.base[1], z = a.base[2];
        T e[3];
#pragma unroll
        for (int c = 0; c < 3; c++)
            e[c] = d.x*rc[0][c]+d.y*rc[1][c]+d.z*rc[2][c];
        const bool fast = __all(fixedFits<T>(q, e, a.fr));   // (as kSpread)
#pragma unroll
        for (int j2 = 0; j2 < P; j2++) {
            const T A = (q*t1+e[0]*u1)*t2[j2]+e[1]*t1*u2[j2];
            const T C = e[2]*t1*t2[j2];
            unsigned long long* row = tile+(y0-j2+(y0 < j2 ? K1 : 0))*K2;
            if (fast)
                spreadRow<T, P, true>(row, KK, z, K2, A, C, t3, u3);
            else
                spreadRow<T, P, false>(row, KK, z, K2, A, C, t3, u3);
        }
    });
    const long long* words = reinterpret_cast<const long long*>(tile);
    for (int i = threadIdx.x; i < npairs*K2; i += blockDim.x) {
        const int l = grp.byK2.div(i), k = i-l*K2, ya = 2*l;
        T2 z;
        z.x = fromFixed<T>(words+ya*K2+k, KK);
        z.y = (ya+1 < K1 ? fromFixed<T>(words+(ya+1)*K2+k, KK) : T(0));
        m.bufA[i] = z;
    }
    __syncthreads();
    planeForward<T, WIDE>(g, grp, m, cplx);
}

// The plane's share of E = -grad phi at the atoms that reach it: out[(s P + j1) 3 + c], s the sorted atom.
template<class T, int P, bool BATCH, bool WIDE>
__global__ void __launch_bounds__(kPlaneThreads) kPlaneGather(const FftGroup* __restrict__ groups,
                                                              const int* __restrict__ blockGroup, PmeSel ps,
                                                              const int* __restrict__ brickStart,
                                                              const PmeAtom<T>* __restrict__ atoms, PlaneSolves<T> solves,
                                                              typename Vec2<T>::type* __restrict__ cplxAll,
                                                              const typename Vec2<T>::type* __restrict__ twAll,
                                                              CgSkip skip) {
    typedef typename Vec2<T>::type T2;
    extern __shared__ __align__(16) unsigned char smemRaw[];
    __shared__ __align__(16) int list[kPlaneList+4];   // and its counter: whole 16 bytes before the dynamic LDS
    if (skip())
        return;
    const FftGroup& grp = groupOf(groups, blockGroup);
    const PmeGrid& g = grp.g;
    const int K0 = g.K[0], K1 = g.K[1], K2 = g.K[2], Kh = g.K3h;
    const int plane = (int) blockIdx.x-grp.blk0[3], gi = plane/K0, x = plane-gi*K0;
    const PmeSys* se = planeSystem<BATCH>(ps, grp, gi);
    const BoxT<double>& box = BATCH ? se->box : ps.box;
    const int solve = blockIdx.y;
    double* __restrict__ out = solves.out[solve];
    const T2* __restrict__ cplx = cplxAll+solve*solves.cplxStride+grp.cplxOff+(size_t) plane*K1*Kh;
    PlaneLds<T> m(smemRaw, g);
    m.load(twAll, grp);
    // row y of the plane: the real (y even) or imaginary (y odd) parts of pair y/2
    const T* phi = reinterpret_cast<const T*>(planeInverse<T, WIDE>(g, grp, cplx, m));
    double rk[3][3];
#pragma unroll
    for (int kk = 0; kk < 3; kk++)
#pragma unroll
        for (int a = 0; a < 3; a++)
            rk[kk][a] = g.K[a]*box.recip[kk][a];
    planeAtoms<T, P>(g, BATCH ? se->brickOff : 0, x, brickStart, atoms, list, list+kPlaneList, [&](int k, int j1) {
        const PmeAtom<T> a = atoms[k];
        const int s = a.s, B1 = a.base[1], B2 = a.base[2];
        T t1s[P], u1s[P], t2[P], u2[P], t3[P], u3[P], w[P];
        bsplines<T, P>(a.fr[0], t1s, u1s, w);
        bsplines<T, P>(a.fr[1], t2, u2, w);
        bsplines<T, P>(a.fr[2], t3, u3, w);
        const T t1 = pick<T, P>(t1s, j1), u1 = pick<T, P>(u1s, j1);
        int z[P];
#pragma unroll
        for (int j = 0; j < P; j++)
            z[j] = 2*(B2-j+(B2 < j ? K2 : 0));
        double f[3] = {0, 0, 0};
#pragma unroll
        for (int j2 = 0; j2 < P; j2++) {
            const int y = B1-j2+(B1 < j2 ? K1 : 0);
            const T* row = phi+2*((y >> 1)*K2)+(y & 1);
            T st = 0, su = 0;
#pragma unroll
            for (int j3 = 0; j3 < P; j3++) {
                const T ph = row[z[j3]];
                st += t3[j3]*ph;
                su += u3[j3]*ph;
            }
            f[0] += (double) (u1*t2[j2]*st);
            f[1] += (double) (t1*u2[j2]*st);
            f[2] += (double) (t1*t2[j2]*su);
        }
        double* o3 = out+((size_t) s*P+j1)*3;
#pragma unroll
        for (int kk = 0; kk < 3; kk++)
            o3[kk] = -(rk[kk][0]*f[0]+rk[kk][1]*f[1]+rk[kk][2]*f[2]);
    });
}

// x: forward, influence function (energy, strain), back; a tile of consecutive z for fixed y per block.
template<class T, bool WIDE>
__global__ void __launch_bounds__(kBlock) kFftXConv(const FftGroup* __restrict__ groups,
                                                    const int* __restrict__ blockGroup,
                                                    typename Vec2<T>::type* __restrict__ cplxAll,
                                                    const T* __restrict__ inflAll,
                                                    const typename Vec2<T>::type* __restrict__ twAll,
                                                    BoxT<double> boxOne, const BoxT<double>* boxes, double beta,
                                                    int energy, int strain, double* __restrict__ partials,
                                                    CgSkip skip, size_t cplxStride) {
    typedef typename Vec2<T>::type T2;
    extern __shared__ __align__(16) unsigned char smemRaw[];
    __shared__ double red[kBlock/64][10];
    if (skip())
        return;
    const FftGroup& grp = groupOf(groups, blockGroup);
    const PmeGrid& g = grp.g;
    const int zt = grp.zx, blk = (int) blockIdx.x-grp.blk0[2];
    const int K = g.K[0], K2 = g.K[1], K3 = g.K[2], Kh = g.K3h;
    const int ntile = (Kh+zt-1)/zt;
    // stacked grids of one shape: block -> (grid, y, z tile)
    const int gi = grp.ngrid > 1 ? blk/(K2*ntile) : 0, lb = blk-gi*(K2*ntile);
    const size_t goff = (size_t) grp.cplxOff+(size_t) gi*K*K2*Kh;
    // (blockIdx.y: the solve, where several are transformed at once)
    typename Vec2<T>::type* __restrict__ cplx = cplxAll+blockIdx.y*cplxStride+goff;
    const T* __restrict__ infl = inflAll+goff;
    const BoxT<double>& box = boxes ? boxes[grp.boxOff+gi] : boxOne;
    const int y = lb/ntile, z0 = (lb%ntile)*zt;
    const int nl = min(zt, Kh-z0);
    const FastDiv byZ = grp.byZx;
    FftPlan* plan = reinterpret_cast<FftPlan*>(smemRaw);
    T2* tw = reinterpret_cast<T2*>(plan+1);
    T2* b0 = tw+K;
    T2* b1 = b0+zt*K;
    loadTransform<T>(tw, plan, twAll, grp, 0);
    // (the tile indexed by its full width: a last tile may be narrower)
    const size_t plane = (size_t) K2*Kh;
    const size_t row = (size_t) y*Kh+z0;
    blockCopy<4, T2>(zt*K,
                     [&](int i) {
                         const int xx = byZ.div(i), l = i-xx*zt;
                         return l < nl ? cplx[xx*plane+row+l] : T2{};
                     },
                     [&](int i, const T2& v) {
                         const int xx = byZ.div(i), l = i-xx*zt;
                         b0[l*K+xx] = v;
                     });
    __syncthreads();
    T2* res = ldsFft<T, WIDE>(b0, b1, tw, plan, K, nl, false);
    T2* other = (res == b0 ? b1 : b0);
    double acc[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const double fac = kPi*kPi/(beta*beta);
    auto convolve = [&](int i, const T& G) {
        const int m1 = byZ.div(i), l = i-m1*zt, m3 = z0+l;
        if (l >= nl)
            return;
        T2 F = res[l*K+m1];
        if (energy) {
            const double w = (m3 == 0 || (K3%2 == 0 && m3 == K3/2)) ? 1.0 : 2.0;
            const double em = 0.5*w*(double) G*((double) F.x*F.x+(double) F.y*F.y);
            acc[0] += em;
            if (strain && G != T(0)) {
                const int f1 = (m1 <= K/2 ? m1 : m1-K), f2 = (y <= K2/2 ? y : y-K2);
                double mv[3];
#pragma unroll
                for (int k = 0; k < 3; k++)
                    mv[k] = f1*box.recip[k][0]+f2*box.recip[k][1]+m3*box.recip[k][2];
                const double c2 = 2.0*(fac+1.0/(mv[0]*mv[0]+mv[1]*mv[1]+mv[2]*mv[2]));
#pragma unroll
                for (int a = 0; a < 3; a++)
#pragma unroll
                    for (int b = 0; b < 3; b++)
                        acc[1+3*a+b] += em*((a == b ? -1.0 : 0.0)+c2*mv[a]*mv[b]);
            }
        }
        F.x *= G;
        F.y *= G;
        res[l*K+m1] = F;
    };
    blockCopy<4, T>(zt*K,
                    [&](int i) {
                        const int m1 = byZ.div(i), l = i-m1*zt;
                        return l < nl ? infl[m1*plane+row+l] : T(0);
                    },
                    convolve);
    __syncthreads();
    T2* res2 = ldsFft<T, WIDE>(res, other, tw, plan, K, nl, true);
    for (int i = threadIdx.x; i < zt*K; i += blockDim.x) {
        const int xx = byZ.div(i), l = i-xx*zt;
        if (l < nl)
            cplx[xx*plane+row+l] = res2[l*K+xx];
    }
    if (energy) {
        const int nq = strain ? 10 : 1;
        for (int q = 0; q < nq; q++) {
            const double v = groupSum<64>(acc[q]);
            if ((threadIdx.x & 63) == 0)
                red[threadIdx.x >> 6][q] = v;
        }
        __syncthreads();
        if (threadIdx.x < 10) {
            double v = 0;
            if (threadIdx.x < nq)
                for (int w = 0; w < kBlock/64; w++)
                    v += red[w][threadIdx.x];
            partials[((size_t) grp.partOff+blk)*10+threadIdx.x] = v;
        }
    }
}

// ---------------------------------------------------------------------------------------- gathering

// What a gather evaluates: the field -grad phi; the field and the reciprocal forces of dipoles dip and charges posq.w
// (an evaluation's end); the potential and the field (adjoint, energy cotangent only); those and their tangents when
// every atom moves by g_s and the grid changes by phiDot: phi' = g . grad phi + phiDot, E' = -(grad grad phi) g -
// grad phiDot.
enum { kGatherField = 0, kGatherForce = 1, kGatherPot = 2, kGatherTan = 3 };

// One workgroup per brick: the brick's potential with its halo is loaded into LDS in whole rows, and G lanes per atom
// gather from there, lane g the rows j1 = g, g + G, ... of P x P points.  Gathered from memory, an atom's 36 rows of
// 6 points touch some 40 lines, 2.4 cycles each of the CU's address path; the tile's rows are read once for all of
// the brick's atoms.  Sums in FP64, the G lanes' in a fixed order.  Per solve, alone, FP32: 999,000 atoms on 216^3 250 -> 96 us,
// 96,000 on 72^3 24 -> 16 us, 98,000 on 112^3 26 -> 19 us.
// Field and force per sorted atom; potential and tangents as out: phi[n], E[3n] at offsets 0 and n, phi'[n], E'[3n] at
// offsets 5n and 6n.
template<class T, int P, int MODE, bool BATCH, int G>
__global__ void __launch_bounds__(kBlock) kGather(PmeSel ps, int n, const int* __restrict__ brickStart,
                                                  const PmeAtom<T>* __restrict__ atoms,
                                                  const T* __restrict__ phiAll, const T* __restrict__ phiDotAll,
                                                  const typename Vec4<T>::type* __restrict__ dip,
                                                  const typename Vec4<T>::type* __restrict__ posq,
                                                  const typename Vec4<T>::type* __restrict__ disp,
                                                  double* __restrict__ field, double* __restrict__ force,
                                                  CgSkip skip) {
    typedef typename Vec4<T>::type T4;
    constexpr bool POT = MODE >= kGatherPot, HESS = MODE == kGatherForce || MODE == kGatherTan, TAN = MODE == kGatherTan;
    extern __shared__ __align__(16) unsigned char smemRaw[];
    T* tile = reinterpret_cast<T*>(smemRaw);
    if (skip())
        return;
    const int bid = blockIdx.x;
    const int first = brickStart[bid], count = brickStart[bid+1]-first;
    if (count == 0)   // block-uniform
        return;
    const PmeSys* se = sysEntry<BATCH>(ps, BATCH ? ps.brickSys[bid] : 0);
    const PmeGrid& g = BATCH ? se->g : ps.g;
    const BoxT<double>& box = BATCH ? se->box : ps.box;
    const T* __restrict__ phi = phiAll+(BATCH ? se->gridOff : 0);
    const T* __restrict__ phiDot = TAN ? phiDotAll+(BATCH ? se->gridOff : 0) : nullptr;
    const int lb = bid-(BATCH ? se->brickOff : 0);
    const int b2 = lb%g.nb[2], b1 = (lb/g.nb[2])%g.nb[1], b0 = lb/(g.nb[2]*g.nb[1]);
    const int E = g.brick+P-1, E3 = E*E*E;
    const int lo0 = b0*g.brick-(P-1), lo1 = b1*g.brick-(P-1), lo2 = b2*g.brick-(P-1);
    const FastDiv byE = ps.byTile;
    auto at = [&](int i) {
        const int xy = byE.div(i), x0 = byE.div(xy), x1 = xy-x0*E, x2 = i-xy*E;
        int g0 = lo0+x0, g1 = lo1+x1, g2 = lo2+x2;
        g0 += (g0 < 0 ? g.K[0] : 0);
        g0 -= (g0 >= g.K[0] ? g.K[0] : 0);
        g1 += (g1 < 0 ? g.K[1] : 0);
        g1 -= (g1 >= g.K[1] ? g.K[1] : 0);
        g2 += (g2 < 0 ? g.K[2] : 0);
        g2 -= (g2 >= g.K[2] ? g.K[2] : 0);
        return ((size_t) g0*g.K[1]+g1)*g.K[2]+g2;
    };
    blockCopy<8, T>(E3, [&](int i) { return phi[at(i)]; }, [&](int i, T v) { tile[i] = v; });
    if (TAN)
        blockCopy<8, T>(E3, [&](int i) { return phiDot[at(i)]; }, [&](int i, T v) { tile[E3+i] = v; });
    __syncthreads();
    double rk[3][3];
#pragma unroll
    for (int kk = 0; kk < 3; kk++)
#pragma unroll
        for (int a = 0; a < 3; a++)
            rk[kk][a] = g.K[a]*box.recip[kk][a];
    const int items = (count*G+63) & ~63;   // whole wavefronts: the lanes' sums are exchanged
    for (int it = threadIdx.x; it < items; it += blockDim.x) {
        const int k = it/G, lane = it%G;
        const bool valid = k < count;
        const PmeAtom<T> a = atoms[first+(valid ? k : 0)];
        T t1s[P], u1s[P], v1s[P], t2[P], u2[P], v2[P], t3[P], u3[P], v3[P];
        bsplines<T, P>(a.fr[0], t1s, u1s, v1s);
        bsplines<T, P>(a.fr[1], t2, u2, v2);
        bsplines<T, P>(a.fr[2], t3, u3, v3);
        // pot, f[3], h[6] of phi; pot', f'[3] of phiDot
        double acc[14] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        const int l1b = a.base[1]-lo1, l2b = a.base[2]-lo2;
        for (int j1 = lane; j1 < P; j1 += G) {
            const T t1 = pick<T, P>(t1s, j1), u1 = pick<T, P>(u1s, j1), v1 = HESS ? pick<T, P>(v1s, j1) : T(0);
            const T* plane = tile+((a.base[0]-j1-lo0)*E+l1b)*E+l2b;
#pragma unroll
            for (int j2 = 0; j2 < P; j2++) {
                const T* row = plane-j2*E;
                T st = 0, su = 0, sv = 0, dt = 0, du = 0;
#pragma unroll
                for (int j3 = 0; j3 < P; j3++) {
                    const T ph = row[-j3];
                    st += t3[j3]*ph;
                    su += u3[j3]*ph;
                    if (HESS)
                        sv += v3[j3]*ph;
                    if (TAN) {
                        const T pd = row[E3-j3];
                        dt += t3[j3]*pd;
                        du += u3[j3]*pd;
                    }
                }
                if (POT)
                    acc[0] += (double) (t1*t2[j2]*st);
                acc[1] += (double) (u1*t2[j2]*st);
                acc[2] += (double) (t1*u2[j2]*st);
                acc[3] += (double) (t1*t2[j2]*su);
                if (HESS) {
                    acc[4] += (double) (v1*t2[j2]*st);   // 00
                    acc[5] += (double) (t1*v2[j2]*st);   // 11
                    acc[6] += (double) (t1*t2[j2]*sv);   // 22
                    acc[7] += (double) (u1*u2[j2]*st);   // 01
                    acc[8] += (double) (u1*t2[j2]*su);   // 02
                    acc[9] += (double) (t1*u2[j2]*su);   // 12
                }
                if (TAN) {
                    acc[10] += (double) (t1*t2[j2]*dt);
                    acc[11] += (double) (u1*t2[j2]*dt);
                    acc[12] += (double) (t1*u2[j2]*dt);
                    acc[13] += (double) (t1*t2[j2]*du);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < 14; c++)
            if (c == 0 ? POT : c < 4 ? true : c < 10 ? HESS : TAN)
                acc[c] = groupSum<G>(acc[c]);
        if (!valid || lane != 0)
            continue;
        const int s = a.s;
        double* eOut = POT ? field+n : field;
        if (POT)
            field[s] = acc[0];
#pragma unroll
        for (int kk = 0; kk < 3; kk++)
            eOut[3*(size_t) s+kk] = -(rk[kk][0]*acc[1]+rk[kk][1]*acc[2]+rk[kk][2]*acc[3]);
        if (HESS) {
            const double H[3][3] = {{acc[4], acc[7], acc[8]}, {acc[7], acc[5], acc[9]}, {acc[8], acc[9], acc[6]}};
            const T4 d = TAN ? disp[s] : dip[s];
            double e[3], c[3];
#pragma unroll
            for (int b = 0; b < 3; b++)
                e[b] = rk[0][b]*d.x+rk[1][b]*d.y+rk[2][b]*d.z;
            const double q = TAN ? 0.0 : (double) posq[s].w;
#pragma unroll
            for (int b = 0; b < 3; b++)
                c[b] = (TAN ? acc[11+b] : q*acc[1+b])+e[0]*H[b][0]+e[1]*H[b][1]+e[2]*H[b][2];
            double* o = TAN ? field+6*(size_t) n : force;
#pragma unroll
            for (int kk = 0; kk < 3; kk++)
                o[3*(size_t) s+kk] = -(rk[kk][0]*c[0]+rk[kk][1]*c[1]+rk[kk][2]*c[2]);
            if (TAN)
                field[5*(size_t) n+s] = e[0]*acc[1]+e[1]*acc[2]+e[2]*acc[3]+acc[10];
        }
    }
}

// ---------------------------------------------------------------------------------------- setup

template<class T>
__global__ void kInfluence(PmeGrid g, const double* bmod, BoxT<double> box, double beta, double volume, T* infl) {
    const int K1 = g.K[0], K2 = g.K[1], Kh = g.K3h;
    const size_t total = (size_t) K1*K2*Kh;
    const size_t idx = (size_t) blockIdx.x*blockDim.x+threadIdx.x;
    if (idx >= total)
        return;
    const int m3 = idx%Kh, m2 = (idx/Kh)%K2, m1 = idx/((size_t) Kh*K2);
    const int f1 = (m1 <= K1/2 ? m1 : m1-K1), f2 = (m2 <= K2/2 ? m2 : m2-K2);
    double val = 0;
    if (f1 != 0 || f2 != 0 || m3 != 0) {
        double mv[3];
        for (int k = 0; k < 3; k++)
            mv[k] = f1*box.recip[k][0]+f2*box.recip[k][1]+m3*box.recip[k][2];
        const double m2s = mv[0]*mv[0]+mv[1]*mv[1]+mv[2]*mv[2];
        const double b = bmod[m1]*bmod[K1+m2]*bmod[K1+K2+m3];
        val = exp(-kPi*kPi/(beta*beta)*m2s)/(kPi*volume*m2s)/b;
    }
    infl[idx] = (T) val;
}

template<class T>
__global__ void kTwiddles(PmeGrid g, typename Vec2<T>::type* tw) {
    const int i = blockIdx.x*blockDim.x+threadIdx.x;
    const int total = g.K[0]+g.K[1]+g.K[2];
    if (i >= total)
        return;
    const int a = (i < g.K[0] ? 0 : (i < g.K[0]+g.K[1] ? 1 : 2));
    const int j = i-(a == 0 ? 0 : (a == 1 ? g.K[0] : g.K[0]+g.K[1]));
    double sn, cs;
    sincospi(-2.0*j/g.K[a], &sn, &cs);
    typename Vec2<T>::type v;
    v.x = (T) cs;
    v.y = (T) sn;
    tw[i] = v;
}

template<class T>
__global__ void kZero(T* p, size_t count, CgSkip skip) {
    if (skip())
        return;
    for (size_t i = (size_t) blockIdx.x*blockDim.x+threadIdx.x; i < count; i += (size_t) gridDim.x*blockDim.x)
        p[i] = T(0);
}

inline int nblk(long long threads, int bs) { return (int) ((threads+bs-1)/bs); }

template<class T>
int linesPerBlock(int K, long long lines, int ldsBytes) {
    // LDS: twiddles + two line buffers within ldsBytes; and enough blocks to fill 256 CUs twice over.  More
    // lines per block keep more of the 256 threads busy in each radix stage.
    const int elems = (int) (ldsBytes/sizeof(typename Vec2<T>::type));
    const int byLds = std::max(1, std::min(64, (elems-K)/(2*K)));
    const int byFill = (int) std::max(1LL, lines/512);
    return std::min(byLds, byFill);
}

// The y and x passes tile a row of K3h half-spectrum lines and read each tile as runs of consecutive z: up to
// 64 KB of LDS (less the x pass's static reduction buffer) gives runs of whole 128-byte lines where the grid
// allows (16 complex floats or 8 complex doubles at K = 216, against 6 and 3 within 24 KB), and the tiles are
// balanced over the row, with no short tail tile.
template<class T>
int tileLines(int K, int Kh, long long lines) {
    const int L = linesPerBlock<T>(K, lines, 64*1024-512);
    const int ntile = (Kh+L-1)/L;
    return (Kh+ntile-1)/ntile;
}

}   // namespace

// Runs fn with the PME order and the batch flag as compile-time constants.
template<class Fn>
void dispatchOrder(int order, bool batch, Fn fn) {
    auto withBatch = [&](auto P) {
        if (batch)
            fn(P, std::true_type{});
        else
            fn(P, std::false_type{});
    };
    switch (order) {
    case 4:
        withBatch(std::integral_constant<int, 4>{});
        break;
    case 5:
        withBatch(std::integral_constant<int, 5>{});
        break;
    case 6:
        withBatch(std::integral_constant<int, 6>{});
        break;
    case 7:
        withBatch(std::integral_constant<int, 7>{});
        break;
    case 8:
        withBatch(std::integral_constant<int, 8>{});
        break;
    default:
        throw std::runtime_error("pgm_hip: PME order must be 4..8");
    }
}

template<class T>
void launchPmeBin(hipStream_t st, int n, const double4* posD, PmeSel ps, int* brickOf, int* slot, int* brickCount) {
    if (ps.table)
        kPmeBin<T, true><<<nblk(n, 256), 256, 0, st>>>(n, posD, ps, brickOf, slot, brickCount);
    else
        kPmeBin<T, false><<<nblk(n, 256), 256, 0, st>>>(n, posD, ps, brickOf, slot, brickCount);
}

template<class T>
void launchPmePlace(hipStream_t st, int n, const double4* posD, PmeSel ps, const int* brickOf, const int* slot,
                    const int* brickStart, PmeAtom<T>* atoms) {
    if (ps.table)
        kPmePlace<T, true><<<nblk(n, 256), 256, 0, st>>>(n, posD, ps, brickOf, slot, brickStart, atoms);
    else
        kPmePlace<T, false><<<nblk(n, 256), 256, 0, st>>>(n, posD, ps, brickOf, slot, brickStart, atoms);
}

// ... and the lanes per atom of the passes over bricks.
template<class Fn>
void dispatchBricks(const PmeSel& ps, Fn fn) {
    dispatchOrder(ps.order, ps.table != nullptr, [&](auto P, auto B) {
        if (ps.atomLanes == 2)
            fn(P, B, std::integral_constant<int, 2>{});
        else
            fn(P, B, std::integral_constant<int, 4>{});
    });
}

template<class T>
void launchSpread(hipStream_t st, PmeSel ps, const int* brickStart, const PmeAtom<T>* atoms,
                  const typename Vec4<T>::type* dip, const typename Vec4<T>::type* posq, int withQ, T* grid,
                  long long* fixed, CgSkip skip, const typename Vec4<T>::type* dipDot,
                  const typename Vec4<T>::type* disp) {
    const int E = ps.brick+ps.order-1;
    const size_t lds = (size_t) E*E*E*sizeof(double)*(dipDot ? 1 : GridFixed<T>::words);
    dispatchBricks(ps, [&](auto P, auto B, auto G) {
        if (dipDot)
            kSpread<T, P(), true, B(), G()><<<ps.nbrick, kBlock, lds, st>>>(ps, brickStart, atoms, dip, posq, withQ, grid,
                                                                           nullptr, skip, dipDot, disp);
        else
            kSpread<T, P(), false, B(), G()><<<ps.nbrick, kBlock, lds, st>>>(ps, brickStart, atoms, dip, posq, withQ,
                                                                            nullptr, fixed, skip, dip, dip);
    });
}

template<class T>
void fftGroupShape(FftGroup& G, bool wide, int blocks[4], size_t lds[5]) {
    typedef typename Vec2<T>::type T2;
    const PmeGrid& g = G.g;
    const int ngrid = G.ngrid;
    const int nlines = ngrid*g.K[0]*g.K[1];
    // z: pairs of real lines; y: the stacked grids are one grid of ngrid K0 x-planes; x: lines of K0
    G.pz = linesPerBlock<T>(g.K[2], (nlines+1)/2, 24*1024);   // contiguous lines: small tiles, more blocks
    blocks[0] = nblk((nlines+1)/2, G.pz);
    lds[0] = sizeof(FftPlan)+(size_t) (g.K[2]+2*G.pz*g.K[2])*sizeof(T2);
    G.zy = tileLines<T>(g.K[1], g.K3h, (long long) ngrid*g.K[0]*g.K3h);
    blocks[1] = ngrid*g.K[0]*((g.K3h+G.zy-1)/G.zy);
    lds[1] = sizeof(FftPlan)+(size_t) (g.K[1]+2*G.zy*g.K[1])*sizeof(T2);
    G.zx = tileLines<T>(g.K[0], g.K3h, (long long) ngrid*g.K[1]*g.K3h);
    blocks[2] = ngrid*g.K[1]*((g.K3h+G.zx-1)/G.zx);
    lds[2] = sizeof(FftPlan)+(size_t) (g.K[0]+2*G.zx*g.K[0])*sizeof(T2);
    // fused z+y: one block per x-plane; plans and twiddles of y and z and two plane buffers
    const int S = std::max(((g.K[1]+1)/2)*g.K[2], g.K3h*g.K[1]);
    blocks[3] = ngrid*g.K[0];
    lds[3] = 2*sizeof(FftPlan)+(size_t) (g.K[1]+g.K[2]+2*S)*sizeof(T2);
    // the x-plane spread: one plane buffer and, over the other, the fixed-point words
    lds[4] = 2*sizeof(FftPlan)+(size_t) (g.K[1]+g.K[2]+S)*sizeof(T2)+
             std::max((size_t) S*sizeof(T2), (size_t) g.K[1]*g.K[2]*GridFixed<T>::words*sizeof(long long));
    G.byK2 = fastDiv(g.K[2]);
    G.byKh = fastDiv(g.K3h);
    G.byZy = fastDiv(G.zy);
    G.byZx = fastDiv(G.zx);
    for (int a = 0; a < 3; a++)
        G.plan[a] = makePlan(g.K[a], wide);
}

template<class T>
void launchPmeConvolve(hipStream_t st, const FftLaunch& L, T* real, typename Vec2<T>::type* cplx, const T* influence,
                       const typename Vec2<T>::type* tw, BoxT<double> box, const BoxT<double>* boxes, double beta,
                       int energy, int strain, double* partials, CgSkip skip, long long* fixed,
                       size_t fixedStride, int stages, int nsolve, size_t cplxStride) {
    const FftGroup* G = L.groups;
    auto go = [&](auto W) {
        constexpr bool wide = W();
        if (stages & kFftForward) {
            if (L.zyFused)
                kFftZY<T, false, wide><<<L.blocks[3], L.planeThreads, L.lds[3], st>>>(G, L.blockGroup[3], real, cplx, tw,
                                                                                     skip, fixed, fixedStride);
            else {
                kFftZ<T, false, wide><<<L.blocks[0], kBlock, L.lds[0], st>>>(G, L.blockGroup[0], real, cplx, tw, skip,
                                                                            fixed, fixedStride);
                kFftY<T, false, wide><<<L.blocks[1], kBlock, L.lds[1], st>>>(G, L.blockGroup[1], cplx, tw, skip);
            }
        }
        kFftXConv<T, wide><<<dim3(L.blocks[2], nsolve), kBlock, L.lds[2], st>>>(G, L.blockGroup[2], cplx, influence, tw,
                                                                               box, boxes, beta, energy, strain,
                                                                               partials, skip, cplxStride);
        if (stages & kFftInverse) {
            if (L.zyFused)
                kFftZY<T, true, wide><<<L.blocks[3], L.planeThreads, L.lds[3], st>>>(G, L.blockGroup[3], real, cplx, tw,
                                                                                    skip, nullptr, 0);
            else {
                kFftY<T, true, wide><<<L.blocks[1], kBlock, L.lds[1], st>>>(G, L.blockGroup[1], cplx, tw, skip);
                kFftZ<T, true, wide><<<L.blocks[0], kBlock, L.lds[0], st>>>(G, L.blockGroup[0], real, cplx, tw, skip,
                                                                           nullptr, 0);
            }
        }
    };
    L.wide ? go(std::true_type{}) : go(std::false_type{});
}

template<class T>
void launchPlaneSpread(hipStream_t st, const FftLaunch& L, PmeSel ps, const int* brickStart, const PmeAtom<T>* atoms,
                       const typename Vec4<T>::type* posq, const PlaneSolves<T>& solves,
                       typename Vec2<T>::type* cplx, const typename Vec2<T>::type* tw, CgSkip skip,
                       const PairFieldArgs<T>* pair, int pairLanes) {
    const int planes = L.blocks[3];
    dispatchOrder(ps.order, ps.table != nullptr, [&](auto P, auto B) {
        auto go = [&](auto W, auto F) {
            const int sh = pairLanes == 16 ? 4 : pairLanes == 32 ? 5 : 6;
            const int extra = F() ? (int) ((((long long) pair->n << sh)+L.planeThreads-1)/L.planeThreads) : 0;
            kPlaneSpread<T, P(), B(), W(), F()><<<dim3(planes+extra, solves.n), L.planeThreads, L.lds[4], st>>>(
                L.groups, L.blockGroup[3], ps, brickStart, atoms, posq, solves, cplx, tw, skip,
                F() ? *pair : PairFieldArgs<T>{}, planes, sh);
        };
        if constexpr (!B()) {
            if (pair) {
                go(std::false_type{}, std::true_type{});
                return;
            }
        }
        L.wide ? go(std::true_type{}, std::false_type{}) : go(std::false_type{}, std::false_type{});
    });
}

template<class T>
void launchPlaneGather(hipStream_t st, const FftLaunch& L, PmeSel ps, const int* brickStart, const PmeAtom<T>* atoms,
                       const PlaneSolves<T>& solves, typename Vec2<T>::type* cplx,
                       const typename Vec2<T>::type* tw, CgSkip skip) {
    dispatchOrder(ps.order, ps.table != nullptr, [&](auto P, auto B) {
        auto go = [&](auto W) {
            kPlaneGather<T, P(), B(), W()><<<dim3(L.blocks[3], solves.n), L.planeThreads, L.lds[3], st>>>(
                L.groups, L.blockGroup[3], ps, brickStart, atoms, solves, cplx, tw, skip);
        };
        L.wide ? go(std::true_type{}) : go(std::false_type{});
    });
}

template<class T>
int convolveBlocksPerGrid(PmeGrid g, int ngrid) {
    const int zx = tileLines<T>(g.K[0], g.K3h, (long long) ngrid*g.K[1]*g.K3h);
    return g.K[1]*((g.K3h+zx-1)/zx);
}

template<class T>
size_t gatherLds(const PmeSel& ps, int grids) {
    const int E = ps.brick+ps.order-1;
    return (size_t) E*E*E*sizeof(T)*grids;
}

template<class T>
void launchGatherTangent(hipStream_t st, PmeSel ps, int n, const int* brickStart, const PmeAtom<T>* atoms,
                         const T* phi, const T* phiDot, const typename Vec4<T>::type* disp, double* out) {
    ps.byTile = fastDiv(ps.brick+ps.order-1);
    dispatchBricks(ps, [&](auto P, auto B, auto G) {
        if (phiDot)
            kGather<T, P(), kGatherTan, B(), G()><<<ps.nbrick, kBlock, gatherLds<T>(ps, 2), st>>>(
                ps, n, brickStart, atoms, phi, phiDot, disp, nullptr, disp, out, nullptr, CgSkip{});
        else
            kGather<T, P(), kGatherPot, B(), G()><<<ps.nbrick, kBlock, gatherLds<T>(ps, 1), st>>>(
                ps, n, brickStart, atoms, phi, nullptr, nullptr, nullptr, nullptr, out, nullptr, CgSkip{});
    });
}

template<class T>
void launchGather(hipStream_t st, PmeSel ps, const int* brickStart, const PmeAtom<T>* atoms, const T* phi,
                  const typename Vec4<T>::type* dip, const typename Vec4<T>::type* posq, int final_, double* field,
                  double* force, CgSkip skip) {
    ps.byTile = fastDiv(ps.brick+ps.order-1);
    dispatchBricks(ps, [&](auto P, auto B, auto G) {
        if (final_)
            kGather<T, P(), kGatherForce, B(), G()><<<ps.nbrick, kBlock, gatherLds<T>(ps, 1), st>>>(
                ps, 0, brickStart, atoms, phi, nullptr, dip, posq, nullptr, field, force, skip);
        else
            kGather<T, P(), kGatherField, B(), G()><<<ps.nbrick, kBlock, gatherLds<T>(ps, 1), st>>>(
                ps, 0, brickStart, atoms, phi, nullptr, dip, posq, nullptr, field, force, skip);
    });
}

template<class T>
void launchInfluence(hipStream_t st, PmeGrid g, const double* bmod, BoxT<double> box, double beta, double volume,
                     T* influence) {
    const size_t total = (size_t) g.K[0]*g.K[1]*g.K3h;
    kInfluence<T><<<nblk((long long) total, 256), 256, 0, st>>>(g, bmod, box, beta, volume, influence);
}

template<class T>
void launchTwiddles(hipStream_t st, PmeGrid g, typename Vec2<T>::type* tw) {
    kTwiddles<T><<<nblk(g.K[0]+g.K[1]+g.K[2], 256), 256, 0, st>>>(g, tw);
}

template<class T>
void launchZero(hipStream_t st, T* p, size_t count, CgSkip skip) {
    const int blocks = (int) std::min<size_t>(2048, (count+255)/256);
    kZero<T><<<std::max(1, blocks), 256, 0, st>>>(p, count, skip);
}

#define PGM_INSTANTIATE_PME(T)                                                                                          \
    template void launchPmeBin<T>(hipStream_t, int, const double4*, PmeSel, int*, int*, int*);                         \
    template void launchPmePlace<T>(hipStream_t, int, const double4*, PmeSel, const int*, const int*, const int*,      \
                                    PmeAtom<T>*);                                                                      \
    template void launchSpread<T>(hipStream_t, PmeSel, const int*, const PmeAtom<T>*,                                  \
                                  const Vec4<T>::type*, const Vec4<T>::type*, int, T*, long long*, CgSkip,             \
                                  const Vec4<T>::type*, const Vec4<T>::type*);                                         \
    template void launchGatherTangent<T>(hipStream_t, PmeSel, int, const int*, const PmeAtom<T>*, const T*,            \
                                         const T*, const Vec4<T>::type*, double*);                                     \
    template void fftGroupShape<T>(FftGroup&, bool, int*, size_t*);                                                       \
    template void launchPmeConvolve<T>(hipStream_t, const FftLaunch&, T*, Vec2<T>::type*, const T*,                    \
                                       const Vec2<T>::type*, BoxT<double>, const BoxT<double>*, double, int, int,     \
                                       double*, CgSkip, long long*, size_t, int, int, size_t);                    \
    template void launchPlaneSpread<T>(hipStream_t, const FftLaunch&, PmeSel, const int*, const PmeAtom<T>*,           \
                                       const Vec4<T>::type*, const PlaneSolves<T>&, Vec2<T>::type*,         \
                                       const Vec2<T>::type*, CgSkip, const PairFieldArgs<T>*, int);                   \
    template void launchPlaneGather<T>(hipStream_t, const FftLaunch&, PmeSel, const int*, const PmeAtom<T>*,           \
                                       const PlaneSolves<T>&, Vec2<T>::type*, const Vec2<T>::type*,         \
                                       CgSkip);                                                                        \
    template void launchGather<T>(hipStream_t, PmeSel, const int*, const PmeAtom<T>*, const T*,                        \
                                  const Vec4<T>::type*, const Vec4<T>::type*, int, double*, double*, CgSkip);          \
    template void launchInfluence<T>(hipStream_t, PmeGrid, const double*, BoxT<double>, double, double, T*);           \
    template void launchTwiddles<T>(hipStream_t, PmeGrid, Vec2<T>::type*);                                             \
    template void launchZero<T>(hipStream_t, T*, size_t, CgSkip);                                                     \
    template int convolveBlocksPerGrid<T>(PmeGrid, int);
PGM_INSTANTIATE_PME(float)
PGM_INSTANTIATE_PME(double)
template void launchZero<int>(hipStream_t, int*, size_t, CgSkip);
template void launchZero<unsigned>(hipStream_t, unsigned*, size_t, CgSkip);
template void launchZero<long long>(hipStream_t, long long*, size_t, CgSkip);

}   // namespace pgmhip
