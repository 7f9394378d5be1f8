// The rows of the CG field pass: the pair pass's own kernels and the x-plane spread that carries the rows of a small
// system in its idle blocks.
#pragma once

#include "device.hpp"
#include "kernels.hpp"

namespace pgmhip {

template<class T>
__device__ __forceinline__ void fieldTerm(const typename Vec4<T>::type& pi, const typename Vec4<T>::type& pj,
                                          const typename Vec4<T>::type& d, const typename Vec2<T>::type& g,
                                          const BoxT<T>& box, int v, int ext, double& ex, double& ey,
                                          double& ez) {
    T x = pi.x-pj.x, y = pi.y-pj.y, z = pi.z-pj.z;
    pairImage(x, y, z, box, v, ext);
    const T c2 = (d.x*x+d.y*y+d.z*z)*g.y;
    ex += (double) (c2*x-d.x*g.x);
    ey += (double) (c2*y-d.y*g.x);
    ez += (double) (c2*z-d.z*g.x);
}

// A buffer resource over n float4 records (the gfx9 raw-buffer data word): a gather then addresses a record with
// one 32-bit offset, the same for the position and the dipole of a partner, instead of two 64-bit addresses.  An
// offset past the records reads zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t float4Records(const float4* p, int n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float4*>(p), (short) 0, n*(int) sizeof(float4), 0x00020000);
}
__device__ __forceinline__ float4 loadRecord(__amdgpu_buffer_rsrc_t r, int offset) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, offset, 0, 0));
}

// v summed over the L lanes of a group (L a power of two, known or not when compiling).
__device__ __forceinline__ double lanesSum(double v, int L) {
    for (int o = L/2; o > 0; o >>= 1)
        v += __shfl_xor(v, o, 64);
    return v;
}

// The dipole field at atom gid/2^SH from its list with the stored G1, G2: thread gid of a pass of 2^SH lanes per atom.
template<class T, int U, bool BATCH>
__device__ __forceinline__ void pairFieldRow(int gid, int sh, const PairFieldArgs<T>& a) {
    typedef typename Vec4<T>::type T4;
    typedef typename Vec2<T>::type T2;
    const int L = 1 << sh, s = gid >> sh, lane = gid & (L-1);
    if (s >= a.n)
        return;
    const T4* __restrict__ pos = a.pos;
    const T4* __restrict__ dip = a.dip;
    const int* __restrict__ pj = a.pj;
    const T2* __restrict__ g12 = a.g12;
    const BoxSel<T>& bs = a.bs;
    double* __restrict__ field = a.field;
    const BoxT<T> box = selectBox<BATCH>(bs, s);
    const T4 pi = pos[s];
    const int start = a.candStart[s], cnt = a.nb[s];
    double ex = 0, ey = 0, ez = 0;
    int k = lane;
    for (; k+(U-1)*L < cnt; k += U*L) {
        int v[U];
        T2 g[U];
        T4 pjv[U], d[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            v[u] = pj[start+k+u*L];
            g[u] = g12[start+k+u*L];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int j = entryAtom(v[u], bs.ext);
            pjv[u] = pos[j];
            d[u] = dip[j];
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            fieldTerm<T>(pi, pjv[u], d[u], g[u], box, v[u], bs.ext, ex, ey, ez);
    }
    for (; k < cnt; k += L) {
        const int v = pj[start+k], j = entryAtom(v, bs.ext);
        fieldTerm<T>(pi, pos[j], dip[j], g12[start+k], box, v, bs.ext, ex, ey, ez);
    }
    ex = lanesSum(ex, L);
    ey = lanesSum(ey, L);
    ez = lanesSum(ez, L);
    if (lane == 0) {
        field[3*s] = ex;
        field[3*s+1] = ey;
        field[3*s+2] = ez;
    }
}

// The FP32 field pass with the kernels evaluated on the fly (no stored kernels read): per entry the partner's
// index, position and dipole (w = its radius parameter rg_j; rg_i rides in the atom's own dipole w), G1 and G2
// from r^2 and rg_i + rg_j (pairKernelsF, as the setup pass evaluates them).
template<int U, bool BATCH>
__device__ __forceinline__ void pairFieldRowOtf(int gid, int sh, const PairFieldArgs<float>& a) {
    const int L = 1 << sh, s = gid >> sh, lane = gid & (L-1);
    if (s >= a.n)
        return;
    const int n = a.n;
    const float4* __restrict__ pos = a.pos;
    const float4* __restrict__ dip = a.dip;
    const int* __restrict__ pj = a.pj;
    const BoxSel<float>& bs = a.bs;
    double* __restrict__ field = a.field;
    const BoxT<float> box = selectBox<BATCH>(bs, s);
    const float4 pi = pos[s];
    const float rgi = dip[s].w;
    const __amdgpu_buffer_rsrc_t posR = float4Records(pos, n), dipR = float4Records(dip, n);
    const int start = a.candStart[s], cnt = a.nb[s];
    // the U entries of a step summed in FP32 (the matrix-vector product is FP32), the steps in FP64
    double ex = 0, ey = 0, ez = 0;
    auto term = [&](const float4& pjv, const float4& d, int v, float& fx, float& fy, float& fz) {
        float x = pi.x-pjv.x, y = pi.y-pjv.y, z = pi.z-pjv.z;
        pairImage(x, y, z, box, v, bs.ext);
        float G[3];
        pairKernelsF<3>(rgi+d.w, a.beta, x*x+y*y+z*z, G);
        const float c2 = (d.x*x+d.y*y+d.z*z)*G[2];
        fx = fmaf(c2, x, fmaf(-d.x, G[1], fx));
        fy = fmaf(c2, y, fmaf(-d.y, G[1], fy));
        fz = fmaf(c2, z, fmaf(-d.z, G[1], fz));
    };
    int k = lane;
    for (; k+(U-1)*L < cnt; k += U*L) {
        int v[U];
        float4 pjv[U], d[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            v[u] = pj[start+k+u*L];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int o = entryAtom(v[u], bs.ext)*(int) sizeof(float4);
            pjv[u] = loadRecord(posR, o);
            d[u] = loadRecord(dipR, o);
        }
        float fx = -0.0f, fy = -0.0f, fz = -0.0f;   // -0: adding it is exact for every x, so it folds away
#pragma unroll
        for (int u = 0; u < U; u++)
            term(pjv[u], d[u], v[u], fx, fy, fz);
        ex += (double) fx;
        ey += (double) fy;
        ez += (double) fz;
    }
    for (; k < cnt; k += L) {
        const int v = pj[start+k], o = entryAtom(v, bs.ext)*(int) sizeof(float4);
        float fx = -0.0f, fy = -0.0f, fz = -0.0f;   // -0: adding it is exact for every x, so it folds away
        term(loadRecord(posR, o), loadRecord(dipR, o), v, fx, fy, fz);
        ex += (double) fx;
        ey += (double) fy;
        ez += (double) fz;
    }
    ex = lanesSum(ex, L);
    ey = lanesSum(ey, L);
    ez = lanesSum(ez, L);
    if (lane == 0) {
        field[3*s] = ex;
        field[3*s+1] = ey;
        field[3*s+2] = ez;
    }
}

}   // namespace pgmhip
