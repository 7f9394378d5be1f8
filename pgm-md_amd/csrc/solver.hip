// Induced-dipole solver and the per-atom stages around it, FP64 vectors in the sorted order:
//   guess       mu4 / mu3 / last-solution predictor from the history (global order) or alpha b
//               (core/pgm_core.cpp:307-328; initialGuess, core/cuda/pgm_cuda.cu:1318-1335);
//   CG          Jacobi-preconditioned CG with the flexible Polak-Ribiere beta, err = max|alpha r| / mean|alpha b|
//               (core/pgm_core.cpp:330-385).  Every sum is written as per-block partials and added up again,
//               identically, by every block of the consuming kernel, and the residual goes through an atomic maximum:
//               deterministic;
//   post        peek, history push, total dipoles (core/pgm_core.cpp:386-397, 413-416);
//   final       total field, self/polarization sums, covalent chain rule, forces out
//               (core/pgm_core.cpp:488-534).
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace pgmhip {

namespace {

constexpr int kCgBlock = 256;

inline int nblk(long long threads, int bs) { return (int) ((threads+bs-1)/bs); }

// Sums of the partials regions r[0..N) of nb entries each, computed redundantly by every block; valid in all threads.
// One pass over the regions and one barrier.
template<int N>
__device__ __forceinline__ void reduceRegions(const double* partials, const int (&r)[N], int nb, double (*smem)[N],
                                              double (&out)[N]) {
    double v[N];
#pragma unroll
    for (int q = 0; q < N; q++)
        v[q] = 0;
    for (int k = threadIdx.x; k < nb; k += kCgBlock)
#pragma unroll
        for (int q = 0; q < N; q++)
            v[q] += partials[r[q]*kCgMaxBlocks+k];
#pragma unroll
    for (int q = 0; q < N; q++) {
        v[q] = groupSum<64>(v[q]);
        if ((threadIdx.x & 63) == 0)
            smem[threadIdx.x >> 6][q] = v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; q++) {
        out[q] = 0;
#pragma unroll
        for (int w = 0; w < kCgBlock/64; w++)
            out[q] += smem[w][q];
    }
}

// The block's sums of v into its entries of the regions r, and the maximum of mx into word (integer atomics on the
// bits of a non-negative double).
template<int N>
__device__ __forceinline__ void writePartials(double (&v)[N], const int (&r)[N], double* partials, double (*smem)[N+1],
                                              double mx, double* word) {
#pragma unroll
    for (int q = 0; q < N; q++)
        v[q] = groupSum<64>(v[q]);
    if (word)
        mx = groupMax64(mx);
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int q = 0; q < N; q++)
            smem[threadIdx.x >> 6][q] = v[q];
        smem[threadIdx.x >> 6][N] = mx;
    }
    __syncthreads();
    if (threadIdx.x < N) {
        double t = 0;
        for (int w = 0; w < kCgBlock/64; w++)
            t += smem[w][threadIdx.x];
        partials[r[threadIdx.x]*kCgMaxBlocks+blockIdx.x] = t;
    }
    if (threadIdx.x == N && word) {
        double t = 0;
        for (int w = 0; w < kCgBlock/64; w++)
            t = fmax(t, smem[w][N]);
        atomicMax(reinterpret_cast<unsigned long long*>(word), (unsigned long long) __double_as_longlong(t));
    }
}

template<class T>
__device__ __forceinline__ typename Vec4<T>::type pairVector(const double* v, T w) {
    typename Vec4<T>::type o;
    o.x = (T) v[0];
    o.y = (T) v[1];
    o.z = (T) v[2];
    o.w = w;
    return o;
}

template<class T>
__global__ void kGuess(int n, const int* order, const int* gidx, const double* hist, size_t stride, GuessCoef gc,
                       const double* alpha, CgRhs rhs, double cself, double* bOut, double* x,
                       typename Vec4<T>::type* xT, const T* rgw) {
    const int s = blockIdx.x*blockDim.x+threadIdx.x;
    if (s >= n)
        return;
    const double a = alpha[s];
    double v[3] = {0, 0, 0};
    if (gc.nc == 0) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double b = rhsOf(rhs, cself, s, c);
            if (bOut)
                bOut[3*s+c] = b;
            v[c] = a*b;
        }
    }
    else {
        const double* h = hist+3*(size_t) gidx[order[s]];
        for (int q = 0; q < gc.nc; q++)
#pragma unroll
            for (int c = 0; c < 3; c++)
                v[c] += gc.c[q]*h[gc.slot[q]*stride+c];
#pragma unroll
        for (int c = 0; c < 3; c++)
            v[c] = (a > 0 ? v[c] : 0.0);
    }
#pragma unroll
    for (int c = 0; c < 3; c++)
        x[3*s+c] = v[c];
    xT[s] = pairVector<T>(v, rgw ? rgw[s] : T(0));
}

__global__ void kCombineB(int n, const double* ed, RecField er, const double* perm, double cself, double* b) {
    const int k = blockIdx.x*blockDim.x+threadIdx.x;
    if (k < 3*n)
        b[k] = ed[k]+recField(er, k/3, k%3)+cself*perm[k];
}

// The pair vector type of a 3-vector per atom, w = rgw[s] (the radius parameter, read by the FP32 field pass
// that evaluates its kernels on the fly) or 0.
template<class T>
__global__ void kToVec4(int n, const double* v, typename Vec4<T>::type* out, const T* rgw) {
    const int s = blockIdx.x*blockDim.x+threadIdx.x;
    if (s < n)
        out[s] = pairVector<T>(v+3*s, rgw ? rgw[s] : T(0));
}

// An iteration of the solve is launch-bound on small systems (each launch costs ~6 us of the stream, a kernel of 1,536
// atoms runs 3-5 us) and a pass over 24-byte rows on large ones, so it takes two kernels: kCgAp with every sum the
// step needs (p.Ap, z.Ap, Ap.f Ap: beta follows from those, z' = z - step f Ap), and kCgStep, which moves x, r and p at
// once and evaluates z = f r where it is used.  The residual goes through one atomic maximum, which every later kernel
// compares for itself.  Against four kernels per iteration, a separate convergence flag and the final stage in ten
// launches: 1,536 atoms 522 -> 467 us per step, 8,550 557 -> 496, 24,000 685 -> 605, 999,000 10.2 -> 9.95 ms.
// r = b - A x (polarizable rows); partials of sum |alpha b| and max |alpha r|.  Jacobi (not pc.pre): z = p =
// alpha/(1 - alpha cj) r and the partials of r.z; with the short-range preconditioner kPrecond<true> does that.
template<class T>
__global__ void __launch_bounds__(kCgBlock) kCgInit(int n, const double* alpha, CgRhs rhs, const double* x,
                                                    const double* td, RecField tr, double cself, double* r,
                                                    double* p, typename Vec4<T>::type* pT, double* partials,
                                                    Precond pc, const T* rgw) {
    __shared__ double smem[40];
    double nrm = 0, rz = 0, mx = 0;
    for (int s = blockIdx.x*blockDim.x+threadIdx.x; s < n; s += gridDim.x*blockDim.x) {
        const double a = alpha[s];
        const double f = a/(1.0-a*pc.cj);
        double pv[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int k = 3*s+c;
            const double b = rhsOf(rhs, cself, s, c);
            const double ax = (a > 0 ? x[k]/a-(td[k]+recField(tr, s, c)+cself*x[k]) : 0.0);
            const double rv = (a > 0 ? b-ax : 0.0);
            const double zv = f*rv;
            r[k] = rv;
            nrm += fabs(a*b);
            mx = fmax(mx, fabs(a*rv));   // the tolerance is on |alpha r| with every preconditioner
            if (!pc.pre) {
                p[k] = zv;
                rz += rv*zv;
            }
            pv[c] = zv;
        }
        if (!pc.pre)
            pT[s] = pairVector<T>(pv, rgw ? rgw[s] : T(0));
    }
    nrm = blockSum(nrm, smem);
    rz = blockSum(rz, smem);
    mx = blockMax(mx, smem);
    if (threadIdx.x == 0) {
        partials[kPNorm*kCgMaxBlocks+blockIdx.x] = nrm;
        if (!pc.pre)
            partials[kPRz0*kCgMaxBlocks+blockIdx.x] = rz;
        partials[kPMax*kCgMaxBlocks+blockIdx.x] = mx;
    }
}

// The norm and the first residual into cg.
__global__ void __launch_bounds__(kCgBlock) kCgInitCheck(int n, int nb, const double* partials, double* cg) {
    __shared__ double smem[40];
    double nrm = 0, mx = 0;
    for (int k = threadIdx.x; k < nb; k += blockDim.x) {
        nrm += partials[kPNorm*kCgMaxBlocks+k];
        mx = fmax(mx, partials[kPMax*kCgMaxBlocks+k]);
    }
    nrm = blockSum(nrm, smem);
    mx = blockMax(mx, smem);
    if (threadIdx.x == 0) {
        cg[0] = nrm/(3.0*n)+1e-300;
        cg[1] = mx;
    }
}

// Ap of iteration it and its partial sums; clears the iteration's residual word, also where the solve has converged
// (the iterations after it are then skipped as well).
__global__ void __launch_bounds__(kCgBlock) kCgAp(int n, int it, const double* alpha, const double* p, const double* r,
                                                  const double* td, RecField tr, double cself, double* ap,
                                                  double* partials, double* cg, CgSkip skip, Precond pc) {
    __shared__ double smem[kCgBlock/64][4];
    if (blockIdx.x == 0 && threadIdx.x == 0)
        cg[2+it] = 0.0;
    double v[3] = {0, 0, 0};   // p.Ap, z.Ap, Ap.f Ap
    auto row = [&](int s, double* q) {
        const double a = alpha[s], f = a/(1.0-a*pc.cj);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int k = 3*s+c;
            const double pk = p[k];
            q[c] = (a > 0 ? pk/a-(td[k]+recField(tr, s, c)+cself*pk) : 0.0);
            v[0] += pk*q[c];
            if (!pc.pre) {
                v[1] += f*r[k]*q[c];
                v[2] += f*q[c]*q[c];
            }
        }
    };
    // the first row before the residual is looked at: its loads and the residual's are then one round trip, not two (with
    // kCgStep alike 1,536 atoms 434 -> 408 us per step of 4 iterations)
    int s = blockIdx.x*blockDim.x+threadIdx.x;
    double q[3] = {0, 0, 0};
    if (s < n)
        row(s, q);
    asm volatile("" : "+v"(v[0]), "+v"(v[1]));
    if (skip())
        return;
    while (s < n) {
#pragma unroll
        for (int c = 0; c < 3; c++)
            ap[3*s+c] = q[c];
        s += gridDim.x*blockDim.x;
        if (s < n)
            row(s, q);
    }
    const int reg[3] = {kPpAp, kPzAp, kPfAA};
    writePartials<3>(v, reg, partials, smem, 0.0, nullptr);
}

// x += step p, r' = r - step Ap, z' = f r', p' = z' + beta p: the partials of r'.z' and max |alpha r'|.
template<class T>
__global__ void __launch_bounds__(kCgBlock) kCgStep(int n, int it, const double* alpha, const double* ap, double* x,
                                                    double* r, double* p, typename Vec4<T>::type* pT,
                                                    double* partials, double* cg, CgSkip skip, Precond pc,
                                                    const T* rgw) {
    __shared__ double smem[kCgBlock/64][4];
    __shared__ double smem2[kCgBlock/64][2];
    // the first row's operands before the residual and the partial sums are looked at (as kCgAp)
    struct Row {
        double a, x[3], r[3], p[3], ap[3];
    } w{};
    auto load = [&](int s) {
        w.a = alpha[s];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            w.x[c] = x[3*s+c];
            w.r[c] = r[3*s+c];
            w.p[c] = p[3*s+c];
            w.ap[c] = ap[3*s+c];
        }
    };
    int s = blockIdx.x*blockDim.x+threadIdx.x;
    if (s < n)
        load(s);
    asm volatile("" : "+v"(w.a));
#pragma unroll
    for (int c = 0; c < 3; c++)
        asm volatile("" : "+v"(w.x[c]), "+v"(w.r[c]), "+v"(w.p[c]), "+v"(w.ap[c]));
    if (skip())
        return;
    const int reg[4] = {kPpAp, kPzAp, kPfAA, (it & 1) ? kPRz1 : kPRz0};
    double sum[4];
    reduceRegions<4>(partials, reg, gridDim.x, smem, sum);
    const double rz = sum[3], step = rz/fmax(sum[0], 1e-300);
    const double bc = -step*(sum[1]-step*sum[2])/fmax(rz, 1e-300);
    double v[1] = {0}, mx = 0;
    while (s < n) {
        const double f = w.a/(1.0-w.a*pc.cj);
        double d[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int k = 3*s+c;
            x[k] = w.x[c]+step*w.p[c];
            const double rn = w.r[c]-step*w.ap[c];
            const double zn = f*rn;
            r[k] = rn;
            d[c] = zn+bc*w.p[c];
            p[k] = d[c];
            mx = fmax(mx, fabs(w.a*rn));
            v[0] += rn*zn;
        }
        pT[s] = pairVector<T>(d, rgw ? rgw[s] : T(0));
        s += gridDim.x*blockDim.x;
        if (s < n)
            load(s);
    }
    const int out[1] = {(it & 1) ? kPRz0 : kPRz1};
    writePartials<1>(v, out, partials, smem2, mx, cg+2+it);
}

// With the short-range preconditioner: x += step p, r' = r - step Ap and max |alpha r'| (kPrecond<false> does the rest).
__global__ void __launch_bounds__(kCgBlock) kCgUpdate(int n, int it, const double* alpha, const double* p,
                                                      const double* ap, double* x, double* r, double* partials,
                                                      double* cg, CgSkip skip) {
    __shared__ double smem[kCgBlock/64][2];
    __shared__ double red[40];
    if (skip())
        return;
    const int reg[2] = {kPpAp, (it & 1) ? kPRz1 : kPRz0};
    double sum[2];
    reduceRegions<2>(partials, reg, gridDim.x, smem, sum);
    const double step = sum[1]/fmax(sum[0], 1e-300);
    double mx = 0;
    for (int k = blockIdx.x*blockDim.x+threadIdx.x; k < 3*n; k += gridDim.x*blockDim.x) {
        x[k] += step*p[k];
        const double rn = r[k]-step*ap[k];
        mx = fmax(mx, fabs(alpha[k/3]*rn));
        r[k] = rn;
    }
    mx = blockMax(mx, red);
    if (threadIdx.x == 0)
        atomicMax(reinterpret_cast<unsigned long long*>(cg+2+it), (unsigned long long) __double_as_longlong(mx));
}

// The short-range preconditioner, z_s = alpha_s (r_s + sum_j T_sj alpha_j r_j), T_sj u = -u G1 + (u.x) x G2 over
// the atom's short list (partners with alpha_j > 0; *over: z_s = alpha_s r_s everywhere), FP64 sums of the
// pair terms from the stored kernels and the positions of the pair type (core/cuda/pgm_cuda.cu:1533-1570).
// INIT (after kCgInit): p = z and its pair-type copy, partials of r.z; else (after kCgUpdate of iteration it):
// partials of -step z.Ap (= z.(r' - r)) and r.z.  One thread per atom, the CG kernels' grid.
template<class T, bool INIT, bool BATCH>
__global__ void __launch_bounds__(kCgBlock) kPrecond(int n, int it, const double* alpha, const double* r,
                                                     const double* ap, const typename Vec4<T>::type* pos,
                                                     BoxSel<T> bs, const int* srCount, const int* srJ,
                                                     const typename Vec2<T>::type* srG, const int* over, double* z,
                                                     double* p, typename Vec4<T>::type* pT, double* partials,
                                                     CgSkip skip, const T* rgw) {
    typedef typename Vec4<T>::type T4;
    typedef typename Vec2<T>::type T2;
    __shared__ double smem[40];
    __shared__ double red[kCgBlock/64][2];
    if (!INIT && skip())
        return;
    double step = 0;
    if (!INIT) {
        const int reg[2] = {kPpAp, (it & 1) ? kPRz1 : kPRz0};
        double sum[2];
        reduceRegions<2>(partials, reg, gridDim.x, red, sum);
        step = sum[1]/fmax(sum[0], 1e-300);
    }
    const bool useT = (*over == 0);
    double rz = 0, bnum = 0;
    for (int s = blockIdx.x*blockDim.x+threadIdx.x; s < n; s += gridDim.x*blockDim.x) {
        const double a = alpha[s];
        double e[3] = {0, 0, 0};
        if (useT && a > 0) {
            const BoxT<T> box = selectBox<BATCH>(bs, s);
            const T4 pi = pos[s];
            const int cnt = srCount[s];
            for (int q = 0; q < cnt; q++) {
                const int v = srJ[(size_t) s*kPreCap+q], j = entryAtom(v, bs.ext);
                const double aj = alpha[j];
                if (aj == 0)
                    continue;
                const T2 g = srG[(size_t) s*kPreCap+q];
                const T4 pj = pos[j];
                T x = pi.x-pj.x, y = pi.y-pj.y, zz = pi.z-pj.z;
                pairImage(x, y, zz, box, v, bs.ext);
                const double xd[3] = {(double) x, (double) y, (double) zz};
                const double u[3] = {aj*r[3*j], aj*r[3*j+1], aj*r[3*j+2]};
                const double ux = u[0]*xd[0]+u[1]*xd[1]+u[2]*xd[2];
#pragma unroll
                for (int c = 0; c < 3; c++)
                    e[c] += -u[c]*(double) g.x+ux*xd[c]*(double) g.y;
            }
        }
        double zv[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int k = 3*s+c;
            zv[c] = a*(r[k]+e[c]);
            z[k] = zv[c];
            rz += r[k]*zv[c];
            if (INIT)
                p[k] = zv[c];
            else
                bnum -= step*zv[c]*ap[k];
        }
        if (INIT) {
            T4 o;
            o.x = (T) zv[0];
            o.y = (T) zv[1];
            o.z = (T) zv[2];
            o.w = rgw ? rgw[s] : T(0);
            pT[s] = o;
        }
    }
    rz = blockSum(rz, smem);
    if (!INIT)
        bnum = blockSum(bnum, smem);
    if (threadIdx.x == 0) {
        if (INIT)
            partials[kPRz0*kCgMaxBlocks+blockIdx.x] = rz;
        else {
            partials[kPBnum*kCgMaxBlocks+blockIdx.x] = bnum;
            partials[((it & 1) ? kPRz0 : kPRz1)*kCgMaxBlocks+blockIdx.x] = rz;
        }
    }
}

template<class T>
__global__ void __launch_bounds__(kCgBlock) kCgDirection(int n, int it, const double* z, double* p,
                                                         typename Vec4<T>::type* pT, const double* partials,
                                                         CgSkip skip, const T* rgw) {
    __shared__ double smem[kCgBlock/64][2];
    if (skip())
        return;
    const int reg[2] = {kPBnum, (it & 1) ? kPRz1 : kPRz0};
    double sum[2];
    reduceRegions<2>(partials, reg, gridDim.x, smem, sum);
    const double bc = sum[0]/fmax(sum[1], 1e-300);
    for (int s = blockIdx.x*blockDim.x+threadIdx.x; s < n; s += gridDim.x*blockDim.x) {
        double v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int k = 3*s+c;
            v[c] = z[k]+bc*p[k];
            p[k] = v[c];
        }
        pT[s] = pairVector<T>(v, rgw ? rgw[s] : T(0));
    }
}

template<class T>
__global__ void kPost(int n, double peek, const double* alpha, const double* r, double* x, const double* perm,
                      const int* order, const int* gidx, double* hist, double* d, const double* rgS,
                      typename Vec4<T>::type* dT) {
    const int s = blockIdx.x*blockDim.x+threadIdx.x;
    if (s >= n)
        return;
    const double a = alpha[s];
    double v[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const int k = 3*s+c;
        double xv = x[k];
        if (peek != 0)
            xv += peek*a*r[k];
        x[k] = xv;
        if (hist)
            hist[3*(size_t) gidx[order[s]]+c] = xv;
        v[c] = perm[k]+xv;
        d[k] = v[c];
    }
    typename Vec4<T>::type o;
    o.x = (T) v[0];
    o.y = (T) v[1];
    o.z = (T) v[2];
    o.w = (T) rgS[s];   // the radius parameter rides along for the pair passes' partner gathers
    dT[s] = o;
}

// Adds the chain-rule terms of covalent entry m: dE/dr_partner = c (g - (g.u) u)/|v|, g = -E_atom: t on the atom, -t on
// the partner, strain t (x) v (core/pgm_core.cpp:512-529).
__device__ __forceinline__ void covalentTerm(int m, const FinalArgs& a, const BoxT<double>& box, double t[3],
                                             double v[3]) {
    const int i = a.covAtomOf[m], j = a.covPartner[m];
    double x = a.pos[3*j]-a.pos[3*i], y = a.pos[3*j+1]-a.pos[3*i+1], z = a.pos[3*j+2]-a.pos[3*i+2];
    minImage(x, y, z, box);
    const double len = sqrt(x*x+y*y+z*z);
    const double u[3] = {x/len, y/len, z/len};
    const int si = a.rank[i];
    double g[3];
#pragma unroll
    for (int k = 0; k < 3; k++)
        g[k] = -(a.ed[3*si+k]+a.er[3*si+k]+a.cself*a.d[3*si+k]);
    const double gu = g[0]*u[0]+g[1]*u[1]+g[2]*u[2];
    const double c = a.covStrength[m]/len;
#pragma unroll
    for (int k = 0; k < 3; k++)
        t[k] = c*(g[k]-gu*u[k]);
    v[0] = x;
    v[1] = y;
    v[2] = z;
}

// Everything after the last field and force passes in one launch (launch-bound up to some 10^4 atoms, then the pass over
// its ~250 bytes per atom): the entry fields are re-evaluated at a covalent partner instead of stored and read back.
// One thread per atom i (caller's order; sorted index s): the force with the chain-rule terms of the covalent entries it
// carries (+t) and of those it is the partner of (-t), and its rows of the sums.
template<bool STRAIN, bool BATCH>
__global__ void __launch_bounds__(kFinalChunk) kFinal(FinalArgs a) {
    constexpr int NW = STRAIN ? kFinalWide : kFinalNarrow;
    __shared__ double smem[kFinalChunk/64][NW];
    const int lo = a.chunkStart[blockIdx.x], hi = a.chunkStart[blockIdx.x+1];
    const int i = lo+(int) threadIdx.x;
    double acc[NW];
#pragma unroll
    for (int q = 0; q < NW; q++)
        acc[q] = 0;
    if (i < hi) {
        const BoxT<double> box = selectBox<BATCH>(a.box, i);
        const int s = a.rank[i];
        double dv[3], er[3], f[3], t[3], v[3];
        const double al = a.alpha[s];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            dv[k] = a.d[3*s+k];
            er[k] = a.er[3*s+k];
            f[k] = 0;
            acc[1] += dv[k]*dv[k];
            if (al > 0)
                acc[2] += a.mu[3*s+k]*a.mu[3*s+k]/(2.0*al);
        }
        if (a.gvdw)
            acc[3] = a.gvdw[s];
        if (STRAIN) {
            const double* row = a.pairRows+10*(size_t) s;
            acc[0] = row[0];
#pragma unroll
            for (int q = 0; q < 9; q++) {
                acc[4+q] = row[1+q];
                acc[13+q] = er[q/3]*dv[q%3];
            }
        }
        else
            acc[0] = a.pairRows[s];
        for (int m = a.covStart[i]; m < a.covStart[i+1]; m++) {
            covalentTerm(m, a, box, t, v);
#pragma unroll
            for (int k = 0; k < 3; k++) {
                f[k] += t[k];
                if (STRAIN)
#pragma unroll
                    for (int b = 0; b < 3; b++)
                        acc[22+3*k+b] += t[k]*v[b];
            }
        }
        for (int e = a.revStart[i]; e < a.revStart[i+1]; e++) {
            covalentTerm(a.revEntry[e], a, box, t, v);
#pragma unroll
            for (int k = 0; k < 3; k++)
                f[k] -= t[k];
        }
        const bool add = !a.shortOf.cg || a.shortOf();
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const double w = a.ke*(a.fpair[3*s+k]+a.frec[3*s+k]+f[k]);
            if (a.fAssign)
                a.fAssign[3*i+k] = w;
            if (a.fOut && add)
                a.fOut[3*i+k] += w;
            if (a.fixedOut && add)
                atomicAdd(reinterpret_cast<unsigned long long*>(a.fixedOut+i+(size_t) k*a.stride),
                          (unsigned long long) llrint(w*a.fixedScale));
            if (a.posKeep)
                a.posKeep[3*i+k] = a.pos[3*i+k];
        }
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < NW; q++) {
        const double v = groupSum<64>(acc[q]);
        if (lane == 0)
            smem[w][q] = v;
    }
    __syncthreads();
    if (threadIdx.x < NW) {
        double v = 0;
        for (int k = 0; k < kFinalChunk/64; k++)
            v += smem[k][threadIdx.x];
        a.chunkSums[(size_t) blockIdx.x*NW+threadIdx.x] = v;
    }
}

// One block per system: the chunks' columns and the x pass's (energy, strain) columns into its result slots.
constexpr int kSumBlock = 512;

template<bool STRAIN>
__global__ void __launch_bounds__(kSumBlock) kFinalSums(const double* chunkSums, const int* sysChunk,
                                                        const double* recRows, const int* recStart,
                                                        const int* sysRec, double* res, int resStride) {
    constexpr int NW = STRAIN ? kFinalWide : kFinalNarrow, NR = STRAIN ? 10 : 1;
    __shared__ double smem[kSumBlock/64][NW+NR];
    const int y = blockIdx.x, r = sysRec[y];
    double acc[NW+NR];
#pragma unroll
    for (int q = 0; q < NW+NR; q++)
        acc[q] = 0;
    for (int k = sysChunk[y]+(int) threadIdx.x; k < sysChunk[y+1]; k += kSumBlock)
#pragma unroll
        for (int q = 0; q < NW; q++)
            acc[q] += chunkSums[(size_t) k*NW+q];
    for (int k = recStart[r]+(int) threadIdx.x; k < recStart[r+1]; k += kSumBlock)
#pragma unroll
        for (int q = 0; q < NR; q++)
            acc[NW+q] += recRows[(size_t) k*10+q];
#pragma unroll
    for (int q = 0; q < NW+NR; q++) {
        const double v = groupSum<64>(acc[q]);
        if ((threadIdx.x & 63) == 0)
            smem[threadIdx.x >> 6][q] = v;
    }
    __syncthreads();
    const int q = threadIdx.x;
    if (q >= NW+NR)
        return;
    double v = 0;
    for (int w = 0; w < kSumBlock/64; w++)
        v += smem[w][q];
    const int slot = q >= NW ? kResRec+q-NW : q == 0 ? kResPair : q < 3 ? kResComb+q-1 : q == 3 ? kResGvdw
                     : q < 13 ? kResPair+1+q-4 : q < 22 ? kResComb+2+q-13 : kResCov+q-22;
    res[(size_t) y*resStride+slot] = v;
}

// The operands of a field evaluation of given charges q and dipoles d (caller's order): the sorted charges into
// the positions' w (FP64 and, when set, the pair type), the sorted dipoles as FP64 3-vectors and as the pair type
// with w = the radius parameter.
template<class T>
__global__ void kFieldOperands(int n, const int* order, const double* q, const double* d, const T* rgw,
                               double4* posD, typename Vec4<T>::type* posT, double* dS, typename Vec4<T>::type* dT) {
    const int s = blockIdx.x*blockDim.x+threadIdx.x;
    if (s >= n)
        return;
    const int i = order[s];
    posD[s].w = q[i];
    if (posT)
        posT[s].w = (T) q[i];
    typename Vec4<T>::type o;
    o.x = (T) d[3*i];
    o.y = (T) d[3*i+1];
    o.z = (T) d[3*i+2];
    o.w = rgw[s];
    dT[s] = o;
    for (int c = 0; c < 3; c++)
        dS[3*s+c] = d[3*i+c];
}

__global__ void kUnsort3(int n, const int* rank, const double* v, double* out) {
    const int k = blockIdx.x*blockDim.x+threadIdx.x;
    if (k >= 3*n)
        return;
    const int i = k/3, c = k-3*i;
    out[k] = v[3*rank[i]+c];
}

}   // namespace

int cgBlocks(int n) { return std::max(1, std::min(kCgMaxBlocks, nblk(n, kCgBlock))); }

template<class T>
void launchGuess(hipStream_t st, int n, const int* order, const int* gidx, const double* hist, size_t slotStride,
                 GuessCoef gc, const double* alpha, CgRhs rhs, double cself, double* bOut, double* x,
                 typename Vec4<T>::type* xT, const T* rgw) {
    kGuess<T><<<nblk(n, 256), 256, 0, st>>>(n, order, gidx, hist, slotStride, gc, alpha, rhs, cself, bOut, x, xT, rgw);
}

void launchCombineB(hipStream_t st, int n, const double* ed, RecField er, const double* perm, double cself,
                    double* b) {
    kCombineB<<<nblk(3LL*n, 256), 256, 0, st>>>(n, ed, er, perm, cself, b);
}

template<class T>
void launchToVec4(hipStream_t st, int n, const double* v, typename Vec4<T>::type* out, const T* rgw) {
    kToVec4<T><<<nblk(n, 256), 256, 0, st>>>(n, v, out, rgw);
}

template<class T>
void launchCgInit(hipStream_t st, int n, const double* alpha, CgRhs rhs, const double* x, const double* td,
                  RecField tr, double cself, double* r, double* p,
                  typename Vec4<T>::type* pT, double* partials, double* cg, Precond pc, const T* rgw) {
    const int nb = cgBlocks(n);
    kCgInit<T><<<nb, kCgBlock, 0, st>>>(n, alpha, rhs, x, td, tr, cself, r, p, pT, partials, pc, rgw);
    kCgInitCheck<<<1, kCgBlock, 0, st>>>(n, nb, partials, cg);
}

void launchCgAp(hipStream_t st, int n, int it, const double* alpha, const double* p, const double* r, const double* td,
                RecField tr, double cself, double* ap, double* partials, double* cg, CgSkip skip, Precond pc) {
    kCgAp<<<cgBlocks(n), kCgBlock, 0, st>>>(n, it, alpha, p, r, td, tr, cself, ap, partials, cg, skip, pc);
}

template<class T>
void launchCgStep(hipStream_t st, int n, int it, const double* alpha, const double* ap, double* x, double* r,
                  double* p, typename Vec4<T>::type* pT, double* partials, double* cg, CgSkip skip, Precond pc,
                  const T* rgw) {
    kCgStep<T><<<cgBlocks(n), kCgBlock, 0, st>>>(n, it, alpha, ap, x, r, p, pT, partials, cg, skip, pc, rgw);
}

void launchCgUpdate(hipStream_t st, int n, int it, const double* alpha, const double* p, const double* ap, double* x,
                    double* r, double* partials, double* cg, CgSkip skip) {
    kCgUpdate<<<cgBlocks(n), kCgBlock, 0, st>>>(n, it, alpha, p, ap, x, r, partials, cg, skip);
}

template<class T>
void launchPrecond(hipStream_t st, int n, int it, bool init, const double* alpha, const double* r, const double* ap,
                   const typename Vec4<T>::type* pos, BoxSel<T> box, const int* srCount, const int* srJ,
                   const typename Vec2<T>::type* srG, const int* over, double* z, double* p,
                   typename Vec4<T>::type* pT, double* partials, CgSkip skip, const T* rgw) {
    const int nb = cgBlocks(n);
    auto go = [&](auto I, auto B) {
        kPrecond<T, I(), B()><<<nb, kCgBlock, 0, st>>>(n, it, alpha, r, ap, pos, box, srCount, srJ, srG, over, z, p,
                                                       pT, partials, skip, rgw);
    };
    const bool b = box.table != nullptr;
    if (init)
        b ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
    else
        b ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
}

template<class T>
void launchCgDirection(hipStream_t st, int n, int it, const double* z, double* p, typename Vec4<T>::type* pT,
                       double* partials, CgSkip skip, const T* rgw) {
    kCgDirection<T><<<cgBlocks(n), kCgBlock, 0, st>>>(n, it, z, p, pT, partials, skip, rgw);
}

template<class T>
void launchPost(hipStream_t st, int n, double peek, const double* alpha, const double* r, double* x, const double* perm,
                const int* order, const int* gidx, double* hist, double* d, const double* rgS,
                typename Vec4<T>::type* dT) {
    kPost<T><<<nblk(n, 256), 256, 0, st>>>(n, peek, alpha, r, x, perm, order, gidx, hist, d, rgS, dT);
}

void launchFinal(hipStream_t st, const FinalArgs& a, int nchunks, bool strain) {
    auto go = [&](auto S, auto B) { kFinal<S(), B()><<<nchunks, kFinalChunk, 0, st>>>(a); };
    const bool b = a.box.table != nullptr;
    if (strain)
        b ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
    else
        b ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
}

void launchFinalSums(hipStream_t st, const double* chunkSums, bool strain, const int* sysChunk, int nsys,
                     const double* recRows, const int* recStart, const int* sysRec, double* res, int resStride) {
    if (strain)
        kFinalSums<true><<<nsys, kSumBlock, 0, st>>>(chunkSums, sysChunk, recRows, recStart, sysRec, res, resStride);
    else
        kFinalSums<false><<<nsys, kSumBlock, 0, st>>>(chunkSums, sysChunk, recRows, recStart, sysRec, res, resStride);
}

template<class T>
void launchFieldOperands(hipStream_t st, int n, const int* order, const double* q, const double* d, const T* rgw,
                         double4* posD, typename Vec4<T>::type* posT, double* dS, typename Vec4<T>::type* dT) {
    kFieldOperands<T><<<nblk(n, 256), 256, 0, st>>>(n, order, q, d, rgw, posD, posT, dS, dT);
}

void launchUnsort3(hipStream_t st, int n, const int* rank, const double* v, double* out) {
    kUnsort3<<<nblk(3LL*n, 256), 256, 0, st>>>(n, rank, v, out);
}

#define PGM_INSTANTIATE_SOLVER(T)                                                                                     \
    template void launchFieldOperands<T>(hipStream_t, int, const int*, const double*, const double*, const T*,      \
                                         double4*, Vec4<T>::type*, double*, Vec4<T>::type*);                          \
    template void launchGuess<T>(hipStream_t, int, const int*, const int*, const double*, size_t, GuessCoef,         \
                                 const double*, CgRhs, double, double*, double*, Vec4<T>::type*, const T*);          \
    template void launchToVec4<T>(hipStream_t, int, const double*, Vec4<T>::type*, const T*);                       \
    template void launchCgInit<T>(hipStream_t, int, const double*, CgRhs, const double*, const double*, RecField,    \
                                  double, double*, double*, Vec4<T>::type*, double*, double*, Precond,               \
                                  const T*);                                                                \
    template void launchCgStep<T>(hipStream_t, int, int, const double*, const double*, double*, double*, double*,    \
                                  Vec4<T>::type*, double*, double*, CgSkip, Precond, const T*);             \
    template void launchPrecond<T>(hipStream_t, int, int, bool, const double*, const double*, const double*,         \
                                   const Vec4<T>::type*, BoxSel<T>, const int*, const int*, const Vec2<T>::type*,     \
                                   const int*, double*, double*, Vec4<T>::type*, double*, CgSkip, const T*);         \
    template void launchCgDirection<T>(hipStream_t, int, int, const double*, double*, Vec4<T>::type*, double*,       \
                                       CgSkip, const T*);                                                             \
    template void launchPost<T>(hipStream_t, int, double, const double*, const double*, double*, const double*,     \
                                const int*, const int*, double*, double*, const double*, Vec4<T>::type*);
PGM_INSTANTIATE_SOLVER(float)
PGM_INSTANTIATE_SOLVER(double)

}   // namespace pgmhip
