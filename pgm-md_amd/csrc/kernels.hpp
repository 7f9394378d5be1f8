// Host-side launchers of the pGM HIP kernels (one translation unit per subsystem) and the plain-data
// structures they share with the engine.
#pragma once

#include <hip/hip_runtime.h>

#include "device.hpp"

namespace pgmhip {

// -------------------------------------------------------------------------------------------- CG state
//
// The CG's device-resident scalars: cg[0] = mean |alpha b| + 1e-300, cg[1+it] = max |alpha r| before iteration it (it =
// 0..maxIter; 0 until known).  Iterations are enqueued ahead: every kernel of iteration it returns at once when the
// solve has converged before it, cg[1+it]/cg[0] <= tol, and a skipped iteration leaves the next one's word zero, which
// says the same.  The words are maxima of non-negative values, so they are gathered by integer atomics on their bits,
// in any order (no kernel of its own reduces them and writes a flag).
struct CgSkip {
    const double* cg;   // nullptr: never
    int it;
    double tol;
    __device__ __forceinline__ bool operator()() const { return cg && !(cg[1+it]/cg[0] > tol); }
};

// Partial sums of the CG kernels: regions of kCgMaxBlocks doubles.
constexpr int kCgMaxBlocks = 1024;
enum { kPNorm = 0, kPRz0 = 1, kPRz1 = 2, kPpAp = 3, kPBnum = 4, kPMax = 5, kPzAp = 6, kPfAA = 7, kPRegions = 8 };

// -------------------------------------------------------------------------------------------- systems

// The box of an atom.  A batch packs several independent periodic systems into one set of arrays: the atoms
// of a system are contiguous, with the same index range in the caller's and in the sorted order, so one
// system index per atom index serves both orders.  table == nullptr: a single system with box.
// ext != 0: the pair list is the caller's (pgm_set_candidates), whose entries carry their periodic images;
// positions are then used as given, not wrapped into the box.
template<class T>
struct BoxSel {
    BoxT<T> box;
    const BoxT<T>* table;
    const int* sysOf;
    int ext;
};

template<bool BATCH, class T>
__device__ __forceinline__ BoxT<T> selectBox(const BoxSel<T>& b, int idx) {
    if (BATCH)
        return b.table[b.sysOf[idx]];
    return b.box;
}

// An entry of a caller's pair list: partner j in the low kExtIndexBits bits, the image t (|t_k| <= 7 box
// vectors) in the 12 above, code = (t0 + 8) | (t1 + 8) << 4 | (t2 + 8) << 8, for x = r_i - r_j + t.box
// (core/cuda/pgm_cuda.cu:2699-2713 packs the shifts alike).  Entries of the engine's own list are plain j.
constexpr int kExtIndexBits = 20;
constexpr unsigned kExtIndexMask = (1u << kExtIndexBits)-1u;

__host__ __device__ __forceinline__ int extEntry(int j, int t0, int t1, int t2) {
    return (int) ((unsigned) j | ((unsigned) (t0+8) | (unsigned) (t1+8) << 4 | (unsigned) (t2+8) << 8)
                                     << kExtIndexBits);
}

__device__ __forceinline__ int entryAtom(int v, int ext) {
    return ext ? (int) ((unsigned) v & kExtIndexMask) : v;
}

// x = r_i - r_j of a list entry v: the minimum image, or, in a caller's list, plus the entry's image.
template<class T>
__device__ __forceinline__ void pairImage(T& x, T& y, T& z, const BoxT<T>& b, int v, int ext) {
    if (ext) {
        const unsigned c = (unsigned) v >> kExtIndexBits;
        const T t0 = T((int) (c & 15u)-8), t1 = T((int) ((c >> 4) & 15u)-8), t2 = T((int) ((c >> 8) & 15u)-8);
        x += t0*b.ax+t1*b.bx+t2*b.cx;
        y += t1*b.by+t2*b.cy;
        z += t2*b.cz;
    }
    else
        minImage(x, y, z, b);
}

// -------------------------------------------------------------------------------------------- pair list

struct CellGrid {
    int nc[3];     // fractional cells per box dimension
    int ncell;
    int off[3][5];   // distinct neighbour-cell offsets per dimension
    int noff[3];
};

// Cell of every atom (fractional cells of the wrapped position), the per-cell counts and each atom's slot.
void launchCellAssign(hipStream_t st, int n, const double* pos, BoxT<double> box, CellGrid g, int* cellOf, int* slot,
                      int* cellCount, int* subOf);
// Exclusive scan of m ints into out[0..m] (out[m] = total); scratch: >= 1024 ints.
// Exclusive scan of m ints into out[0..m] (out[m] = the total).  Above 4,096 elements it runs over tiles, with
// scratch of scanScratchInts(m) ints (null: one block, slower on long arrays).
int scanScratchInts(int m);
void launchScan(hipStream_t st, const int* in, int* out, int m, int* scratch);
// Sorted order: atoms grouped by cell, inside a cell by (2x2x2 sub-cell, original index).
// base: added to the atom indices written (the system's first atom in a batch).
void launchCellScatter(hipStream_t st, int n, const int* cellOf, const int* slot, const int* cellStart, int* order,
                       int base);
void launchCellSort(hipStream_t st, int ncell, const int* cellStart, const int* subOf, int* order);
void launchRank(hipStream_t st, int n, const int* order, int* rank, int* sortedCell, const int* cellOf, int base);
// Full candidate lists (both directions) of the sorted atoms within rl: counts, then the lists.
void launchCandCount(hipStream_t st, int n, const double4* posS, const int* sortedCell, const int* cellStart,
                     CellGrid g, BoxT<double> box, double rl2, int* count);
void launchCandFill(hipStream_t st, int n, const double4* posS, const int* sortedCell, const int* cellStart,
                    CellGrid g, BoxT<double> box, double rl2, const int* candStart, int* cand, int base);
// Largest squared displacement (minimum image) since the list build, as float bits in *maxBits.
void launchMaxDisplacement(hipStream_t st, int n, const double* pos, const double* posBuild, BoxSel<double> box,
                           unsigned* maxBits);

// -------------------------------------------------------------------------------------------- per atom

// Sorted positions wrapped into the box (xyz, w = charge) in FP64 and, for the mixed path, FP32.
void launchGatherPositions(hipStream_t st, int n, const int* order, const double* pos, const double* qS,
                           BoxSel<double> box, double4* posD, float4* posF);
void launchPermute(hipStream_t st, int n, const int* order, const double* in, double* out);
// The same atoms under new caller indices (newOf: old -> new): order, rank and the build positions renamed.
void launchRename(hipStream_t st, int n, const int* newOf, const int* order, const int* rank, const double* build,
                  int* order2, int* rank2, double* build2);
void launchToFloat(hipStream_t st, int n, const double* in, float* out);
// Caller-order float4 (xyz, w ignored) or float xyz positions to FP64 xyz.
void launchF4ToDouble(hipStream_t st, int n, const float4* posq, double* out);
// *differs = 1 when the count doubles of a and b are not all equal (*differs cleared by the caller).
void launchDiffers(hipStream_t st, long long count, const double* a, const double* b, int* differs);
// Permanent dipoles of the sorted atoms from the covalent CSR (caller's order, positions in FP64).
void launchPermDipoles(hipStream_t st, int n, const int* order, const double* pos, const int* covStart,
                       const int* covPartner, const double* covStrength, BoxSel<double> box, double* perm);

// The per-evaluation preparation of the sorted atoms in one pass: the wrapped positions with charges (FP64
// and, when posF is set, FP32 with the FP32 radius parameters rgF), the permanent dipoles (FP64 and as the
// pair/PME vector type permT, w = the radius parameter), and the clearing of the counters and sums the kernels
// after it accumulate into (zeroI: nZeroI ints, zeroD: nZeroD doubles, maxBits: the next list check's maximum).
struct PrepArgs {
    int n;
    const int* order;
    const double* pos;   // caller's order, FP64 xyz
    const double* qS;    // sorted charges
    const double* rgS;   // sorted radius parameters
    const int* covStart;
    const int* covPartner;
    const double* covStrength;
    BoxSel<double> box;
    double4* posD;
    float4* posF;
    float* rgF;
    double* perm;
    void* permT;
    int* zeroI;
    int nZeroI;
    double* zeroD;
    int nZeroD;
    unsigned* maxBits;
    const double* gvIn;   // GVDW (sqrt A, sqrt C6, b) per atom, caller's order (nullptr: none)
    void* gvOut;          // ... as the pair vector type, sorted order
};
template<class T>
void launchPrepAtoms(hipStream_t st, const PrepArgs& a);

// -------------------------------------------------------------------------------------------- pair passes

// Short-range pairs per atom kept for the CG preconditioner (core/cuda/pgm_cuda.cu:162).
constexpr int kPreCap = 48;

// Lanes per atom of the pair passes: 16, 32 or 64 (picked per engine by the autotuner, 16 by default).
constexpr int kPairLaneChoices[3] = {16, 32, 64};

// Per evaluation: every atom's candidates compacted in place to the pairs within rc (pj: partner; nb: pairs
// per atom), in the atom's candidate segment.
template<class T>
void launchPairCompact(hipStream_t st, int n, const typename Vec4<T>::type* pos, const int* candStart,
                       const int* cand, int* nb, int* pj, BoxSel<T> box, T rc2, int lanes);
// Per evaluation, over the compacted pairs: the kernels (g12: G1, G2, null in FP32: not stored; g03: G0,
// G3, FP64 only), the direct field of
// the charges and dipoles dip and, when dual is given, of the dipoles dual alone (the first CG product).
template<class T>
void launchPairSetup(hipStream_t st, int n, const typename Vec4<T>::type* pos, const T* rg,
                     const typename Vec4<T>::type* dip, const typename Vec4<T>::type* dual, const int* candStart,
                     const int* nb, const int* pj, typename Vec2<T>::type* g12, typename Vec2<T>::type* g03,
                     BoxSel<T> box, T beta, double* field, double* fieldDual, int lanes);
// launchPairCompact + launchPairSetup in one pass (compacted pairs buffered in LDS per atom); the pairs with
// r^2 < rg_i + rgMax (rgMax: the largest rg, or any value: it orders the segment, nothing else) come last in it.
template<class T>
void launchPairCompactSetup(hipStream_t st, int n, const typename Vec4<T>::type* pos, const T* rg,
                            const typename Vec4<T>::type* dip, const typename Vec4<T>::type* dual,
                            const int* candStart, const int* cand, int* nb, int* pj, typename Vec2<T>::type* g12,
                            typename Vec2<T>::type* g03, BoxSel<T> box, T rc2, T beta, T rgMax, double* field,
                            double* fieldDual, int lanes);
// The dipole part of a CG matrix-vector product from the stored G1, G2 or, otf (FP32 only), with the kernels
// evaluated on the fly from the positions and the radius parameters in the dipoles' w.  reverse (here and in
// launchPairFinal): the atoms in the opposite block order (the same results; the engine alternates the
// direction from one pass over the list to the next, so that a pass starts on what the one before touched last).
template<class T>
struct PairFieldArgs {
    int n;
    const typename Vec4<T>::type* pos;
    const typename Vec4<T>::type* dip;
    const int* candStart;
    const int* nb;
    const int* pj;
    const typename Vec2<T>::type* g12;
    BoxSel<T> bs;
    double* field;
    bool otf;
    T beta;
    bool reverse;
};
template<class T>
void launchPairField(hipStream_t st, const PairFieldArgs<T>& args, int lanes, CgSkip skip);
// The CG preconditioner's short-range list: per atom, its compacted pairs within the radius (srJ partner, srG its
// G1, G2; at most kPreCap, counted in srCount); *over set when an atom has more (cleared by the caller).
template<class T>
void launchShortList(hipStream_t st, int n, const typename Vec4<T>::type* pos, const int* candStart, const int* nb,
                     const int* pj, const T* rg, T beta, BoxSel<T> box, T rpre2, int* srCount, int* srJ,
                     typename Vec2<T>::type* srG, int* over);
// The GVDW pair term of the final pass (core/gvdw_kernel.h, combination rule; gv == nullptr: none).
template<class T>
struct GvdwArgs {
    const typename Vec4<T>::type* gv;   // per sorted atom (sqrt A, sqrt C6, b, 0)
    T rvdw2;
    int slater;                         // repulsion: 0 Gaussian, 1 Slater
    T invKe;                            // forces and strain in units of ke, as the electrostatics
    double* energy;                     // per sorted atom: half of its pairs' GVDW energy [kJ/mol]
};

// Energy, forces, field and (strain set) strain of the pairs at the total dipoles (w: the radius parameters), from
// the stored kernels in FP64; per atom (sorted order) perAtom[n][10] = energy, strain
// 0..8 with strain, else perAtom[n] = energy (each pair's half).
template<class T>
void launchPairFinal(hipStream_t st, int n, const typename Vec4<T>::type* pos, const typename Vec4<T>::type* dip,
                     const T* rg, T beta, const int* candStart, const int* nb, const int* pj,
                     const typename Vec2<T>::type* g12, const typename Vec2<T>::type* g03, BoxSel<T> box,
                     double* force, double* field, double* perAtom, bool strain, const GvdwArgs<T>& gvdw,
                     int lanes, bool reverse = false);
// After launchPairFinal with GVDW: the GVDW terms of the skipped pairs (per atom CSR of partners in the caller's
// order, both directions) subtracted from the atoms' forces, GVDW energies and (strain) strain rows.
template<class T>
void launchGvdwSkip(hipStream_t st, int n, const int* order, const int* rank, const typename Vec4<T>::type* pos,
                    const T* rg, const int* skipStart, const int* skipPartner, BoxSel<T> box, T rc2, bool strain,
                    const GvdwArgs<T>& gvdw, double* force, double* perAtom);

// Parameter derivatives of the pair energy at fixed dipoles and, with dipDot (and disp) given, their tangents
// along the displacement disp and the dipole change dipDot, sorted order, each atom from its own visits of its
// pairs.  out (FP64): phi[n], E[3n], dU/dR[n], then with tangents phi'[n], E'[3n], (dU/dR)'[n].
template<class T>
void launchPairTangent(hipStream_t st, int n, const typename Vec4<T>::type* pos, const T* rg, T beta,
                       const typename Vec4<T>::type* dip, const typename Vec4<T>::type* dipDot,
                       const typename Vec4<T>::type* disp, const int* candStart, const int* nb, const int* pj,
                       const typename Vec2<T>::type* g12, const typename Vec2<T>::type* g03, BoxSel<T> box,
                       double* out);

// -------------------------------------------------------------------------------------------- PME

// a / d for 0 <= a < 2^20 and 1 <= d < 2^12 by one multiply: floor(a * ceil(2^32 / d) / 2^32) is exact there
// (the rounding of the reciprocal contributes a * (ceil - 2^32/d) / 2^32 < a * d / 2^32 < 1/d).  Replaces the
// ~20-instruction integer divisions of the FFT index arithmetic.  magic 0: d = 1.
struct FastDiv {
    unsigned magic;
    __host__ __device__ __forceinline__ int div(int a) const {
        return magic ? (int) (((unsigned long long) (unsigned) a*magic) >> 32) : a;
    }
};
inline FastDiv fastDiv(int d) {
    return FastDiv{d == 1 ? 0u : (unsigned) (((1ull << 32)+(unsigned long long) d-1)/(unsigned long long) d)};
}

// Stages of a mixed-radix FFT; for each the divisions by m = K/R and by Ns = R_0...R_{s-1}.
struct FftPlan {
    struct Stage {
        int radix;
        FastDiv byM, byNs;
    };
    int nstage;
    int pad;
    Stage stage[10];
};
constexpr int kPlanInts = sizeof(FftPlan)/sizeof(int);
// wide: radices 2..10 (the fewest stages), else 2, 3, 4, 5, 7.  Throws for a length with other prime factors.
FftPlan makePlan(int K, bool wide = false);

struct PmeGrid {
    int K[3];
    int K3h;
    int order;
    int brick;     // edge of the spreading bricks in grid points
    int nb[3];     // bricks per dimension
    int nbrick;
};

// One system's PME grid in a batch: its grid, box, the offset of its real grid and its first global brick.
struct PmeSys {
    PmeGrid g;
    BoxT<double> box;
    long long gridOff;
    int brickOff;
    int pad;
};
// The grid of an atom or a brick: one system (g, box), or per system from a table (batch).
struct PmeSel {
    PmeGrid g;
    BoxT<double> box;
    const PmeSys* table;    // batch: per system; nullptr: a single system
    const int* sysOf;       // batch: system of every (sorted) atom index
    const int* brickSys;    // batch: system of every global brick
    const int* groupSys;    // batch: system of every stacked grid, group after group
    int nbrick;             // bricks of all systems
    int order;
    int brick;
    FastDiv byTile;         // (the gather's) division by its tile's edge
    int atomLanes;          // lanes per atom of the spread and the gather over bricks: 2 (full bricks) or 4
    size_t fixedStride;     // FP64 fixed-point grids: the second words' offset (the stacked real grids' size)
};

// An atom of the PME passes, in brick order: its base grid point, its (sorted) index and its fractions of a grid
// cell, from which a pass evaluates the spline weights it needs (bsplines).  32 or 48 bytes in place of a table of 9 P
// weights per atom (216 or 432 bytes at order 6), whose lines were what the spread and the gather waited for.
template<class T>
struct __align__(16) PmeAtom {
    int base[3];
    int s;
    T fr[4];   // (the last unused)
};
// Binning of the sorted atoms into spreading bricks, and their records in brick order.
template<class T>
void launchPmeBin(hipStream_t st, int n, const double4* posD, PmeSel ps, int* brickOf, int* slot, int* brickCount);
template<class T>
void launchPmePlace(hipStream_t st, int n, const double4* posD, PmeSel ps, const int* brickOf, const int* slot,
                    const int* brickStart, PmeAtom<T>* atoms);
// Spread charges (withQ) and dipoles of the sorted atoms onto the fixed-point grids fixed (GridFixed<T>::words
// words per point, the second words of all points after the first words of all points; zeroed by the caller;
// order-independent) or, with dipDot, the change of that density for displacements disp and dipole changes dipDot
// onto the real grids grid (zeroed by the caller).
template<class T>
void launchSpread(hipStream_t st, PmeSel ps, const int* brickStart, const PmeAtom<T>* atoms,
                  const typename Vec4<T>::type* dip, const typename Vec4<T>::type* posq, int withQ, T* grid,
                  long long* fixed, CgSkip skip, const typename Vec4<T>::type* dipDot = nullptr,
                  const typename Vec4<T>::type* disp = nullptr);
// The PME charge and dipole grids in 64-bit fixed point.  FP32: one word per point, 2^32 units per grid unit, the
// reference's scale (core/cuda/pgm_cuda.cu:52), for |grid values| < 2^31.  FP64: two words per point, the value
// split into hi = rint(v 2^24) and lo = rint((v - hi 2^-24) 2^56): each contribution is rounded at 2^-57 (below
// FP64's own rounding of values of order one), and the sum reads back exactly for |grid values| < 2^29.  The two
// words are accumulated apart (the lo words of up to 2^22 contributions cannot overflow) and combined once.
template<class T>
struct GridFixed;
template<>
struct GridFixed<float> {
    static constexpr int words = 1;
    static constexpr double scale = 4294967296.0, inv = 1.0/4294967296.0;
};
template<>
struct GridFixed<double> {
    static constexpr int words = 2;
    static constexpr double scale = 16777216.0, inv = 1.0/16777216.0;           // hi: 2^24
    static constexpr double loScale = 72057594037927936.0, loInv = 1.0/72057594037927936.0;   // lo: 2^56
};
template<class T>
__device__ __forceinline__ void toFixed(T v, long long& hi, long long& lo) {
    hi = __double2ll_rn((double) v*GridFixed<T>::scale);
    if constexpr (GridFixed<T>::words == 2)
        lo = __double2ll_rn(fma(-(double) hi, GridFixed<T>::inv, (double) v)*GridFixed<T>::loScale);
    else
        lo = 0;
}
// toFixed for |v| < fixedLimit<T>() without the 64-bit conversions (about ten FP64 instructions each): adding
// 1.5 2^k puts the last place of the sum at the fixed-point unit, so the sum's bits less the constant's are the
// value rounded to nearest even, the same integer as toFixed gives.  FP32: k = 20 (unit 2^-32); FP64: k = 28 for
// the first word (2^-24), the exact remainder with k = -4 for the second (2^-56).
template<class T>
__host__ __device__ constexpr T fixedLimit() {
    return sizeof(T) == sizeof(float) ? T(1 << 18) : T(1 << 26);
}
// Whether every contribution of an atom with charge q, dipole e (per grid unit) and grid fractions fr (0..1) may take
// toFixedFast: the splines and their first derivatives are at most 1.  One sum over all they are made of, which anything
// that is not finite fails.
template<class T>
__device__ __forceinline__ bool fixedFits(T q, const T* e, const T* fr) {
    return fabs(q)+fabs(e[0])+fabs(e[1])+fabs(e[2])+(fr[0]+fr[1]+fr[2]) < fixedLimit<T>();
}
template<class T>
__device__ __forceinline__ void toFixedFast(T v, long long& hi, long long& lo) {
    if constexpr (GridFixed<T>::words == 2) {
        constexpr double m1 = 402653184.0, m2 = 0.09375;
        const double d = v+m1;
        hi = __double_as_longlong(d)-__double_as_longlong(m1);
        const double e = (v-(d-m1))+m2;
        lo = __double_as_longlong(e)-__double_as_longlong(m2);
    }
    else {
        constexpr double m = 1572864.0;
        hi = __double_as_longlong((double) v+m)-__double_as_longlong(m);
        lo = 0;
    }
}
// The value of a point whose words are at p[0] and (FP64) p[stride].
template<class T>
__device__ __forceinline__ T fromFixed(const long long* p, size_t stride) {
    if constexpr (GridFixed<T>::words == 2)
        return (T) ((double) p[0]*GridFixed<T>::inv+(double) p[stride]*GridFixed<T>::loInv);
    else
        return (T) ((double) p[0]*GridFixed<T>::inv);
}
// The same, leaving the words zero for the next spread (the forward z transform reads every point once).
template<class T>
__device__ __forceinline__ T takeFixed(long long* p, size_t stride) {
    const T v = fromFixed<T>(p, stride);
    p[0] = 0;
    if constexpr (GridFixed<T>::words == 2)
        p[stride] = 0;
    return v;
}

// One grid shape's share of a merged transform launch: every shape of a batch goes through each stage (z, y,
// x + convolution, y, z) in one launch.
struct FftGroup {
    PmeGrid g;
    int ngrid;                   // stacked grids of this shape
    long long realOff, cplxOff;  // first element of its real grids / complex grids and influence functions
    int twOff;                   // its twiddles
    int partOff;                 // first row of its x-pass partial sums
    int boxOff;                  // its first system's box in the batch box table
    int pz, zy, zx;              // lines per block of the z, y and x stages
    int blk0[4];                 // its first block in the z, y, x and fused z+y launches
    FastDiv byK2, byKh, byZy, byZx;
    FftPlan plan[3];             // the transforms along x, y and z
};
constexpr int kPlaneThreads = 1024;   // most threads of a block of the x-plane passes
struct FftLaunch {
    const FftGroup* groups;      // device table
    int ngroups;
    const int* blockGroup[4];   // the group of every block of the four launches (nullptr: one group)
    int blocks[4];               // z, y, x and fused z+y launch sizes
    size_t lds[5];               // dynamic LDS of those stages and the x-plane spread (the largest shape's)
    int wide;                    // the plans' radices (makePlan)
    int zyFused;                 // z and y in one pass per x-plane (many small grids), else apart
    int plane;                   // spread and gather in the x-plane passes too (kPlaneSpread, kPlaneGather)
    int planeThreads;            // threads per block of the x-plane passes (kPlaneThreads, or fewer for many planes)
};
// The shape of group g's stages (lines per block) and its blocks per stage, as the transforms use them.
template<class T>
void fftGroupShape(FftGroup& G, bool wide, int blocks[4], size_t lds[5]);
// The z and y transforms a convolution includes beside its x pass.
enum { kFftForward = 1, kFftInverse = 2 };
// Forward transforms, influence function (energy and strain partials when asked), inverse transforms of all
// grids of all groups; real: the stacked real grids, cplx/influence/tw: the stacked complex arrays.  boxes: per
// stacked grid (nullptr: box for all).  partials: [.][10] (energy, strain 0..8) per x block, the blocks of a
// group's grid k being rows partOff + [k, k+1) x blocks per grid.  fixed: the forward transforms read the
// fixed-point grids (as the spread left them) instead of real, and leave them zero; the inverse transforms
// write real.
template<class T>
void launchPmeConvolve(hipStream_t st, const FftLaunch& L, T* real, typename Vec2<T>::type* cplx, const T* influence,
                       const typename Vec2<T>::type* tw, BoxT<double> box, const BoxT<double>* boxes, double beta,
                       int energy, int strain, double* partials, CgSkip skip, long long* fixed,
                       size_t fixedStride, int stages = kFftForward | kFftInverse, int nsolve = 1,
                       size_t cplxStride = 0);
// The solves an x-plane launch runs at once: dipoles (and charges), and where each solve's field goes: P shares per
// sorted atom, one per x-plane it reaches, out[(s P + j) 3 + c] (summed by the readers, RecField).  cplxStride:
// elements between the solves' complex grids.
template<class T>
struct PlaneSolves {
    int n;
    const typename Vec4<T>::type* dip[2];
    int withQ[2];
    double* out[2];
    size_t cplxStride;
};
// The density of the solves spread into the x-planes and transformed in z and y into cplx; their potentials transformed
// back and gathered (launchPmeConvolve with stages = 0 in between).
// pair (may be null; one system, L.planeThreads = kPlaneThreads and not L.wide): the rows of launchPairField with that
// many lanes in further blocks of the launch.
template<class T>
void launchPlaneSpread(hipStream_t st, const FftLaunch& L, PmeSel ps, const int* brickStart, const PmeAtom<T>* atoms,
                       const typename Vec4<T>::type* posq, const PlaneSolves<T>& solves,
                       typename Vec2<T>::type* cplx, const typename Vec2<T>::type* tw, CgSkip skip,
                       const PairFieldArgs<T>* pair = nullptr, int pairLanes = 0);
template<class T>
void launchPlaneGather(hipStream_t st, const FftLaunch& L, PmeSel ps, const int* brickStart, const PmeAtom<T>* atoms,
                       const PlaneSolves<T>& solves, typename Vec2<T>::type* cplx,
                       const typename Vec2<T>::type* tw, CgSkip skip);
// Blocks of the x pass per grid (the rows of its energy partials) when ngrid grids of shape g are stacked.
template<class T>
int convolveBlocksPerGrid(PmeGrid g, int ngrid);
// Field -grad phi (sorted order) and, when final, the reciprocal forces.
template<class T>
void launchGather(hipStream_t st, PmeSel ps, const int* brickStart, const PmeAtom<T>* atoms, const T* phi,
                  const typename Vec4<T>::type* dip, const typename Vec4<T>::type* posq, int final_, double* field,
                  double* force, CgSkip skip);
// Potential and field of the convolved grid phi at the atoms and, with phiDot, their tangents for atoms displaced
// by disp: out (sorted order) phi[n], E[3n] at offsets 0 and n, phi'[n], E'[3n] at offsets 5n and 6n.
template<class T>
void launchGatherTangent(hipStream_t st, PmeSel ps, int n, const int* brickStart, const PmeAtom<T>* atoms,
                         const T* phi, const T* phiDot, const typename Vec4<T>::type* disp, double* out);
template<class T>
void launchInfluence(hipStream_t st, PmeGrid g, const double* bmod, BoxT<double> box, double beta, double volume,
                     T* influence);
template<class T>
void launchTwiddles(hipStream_t st, PmeGrid g, typename Vec2<T>::type* tw);
template<class T>
void launchZero(hipStream_t st, T* p, size_t count, CgSkip skip);

// -------------------------------------------------------------------------------------------- solver

struct GuessCoef {
    int nc;          // 0: x = alpha b
    int slot[4];
    double c[4];
};

// The reciprocal field of a solve: parts 3-vectors per sorted atom to be summed (the x-plane gather writes one per
// plane an atom reaches, kGather the sum).
struct RecField {
    const double* p;
    int parts;
};
__device__ __forceinline__ double recField(const RecField& f, int s, int c) {
    const double* v = f.p+(size_t) s*f.parts*3+c;
    double sum = v[0];
    for (int j = 1; j < f.parts; j++)
        sum += v[3*j];
    return sum;
}

// b = field_dir + field_rec + cself * perm.
void launchCombineB(hipStream_t st, int n, const double* ed, RecField er, const double* perm, double cself,
                    double* b);
template<class T>
void launchToVec4(hipStream_t st, int n, const double* v, typename Vec4<T>::type* out, const T* rgw = nullptr);
int cgBlocks(int n);
// The CG's preconditioner: Jacobi z = alpha/(1 - alpha cj) r (cj = 0, or the self coefficient), or, with a short
// list (pre), the short-range z = alpha (r + T_s alpha r), computed by launchPrecond after launchCgInit and after
// each launchCgUpdate.
struct Precond {
    bool pre;
    double cj;
};
// The right-hand side of a solve: b, or, b null, the field of the charges and permanent dipoles, ed + er + cself perm.
struct CgRhs {
    const double* b;
    const double* ed;
    RecField er;
    const double* perm;
};
__device__ __forceinline__ double rhsOf(const CgRhs& q, double cself, int s, int c) {
    const int k = 3*s+c;
    return q.b ? q.b[k] : q.ed[k]+recField(q.er, s, c)+cself*q.perm[k];
}
// The initial guess, also as the pair vector type (w = rgw): the predictor over the history, or, gc.nc == 0, alpha b
// (b then written to bOut when it is not null: a solve without a history needs b before its first product).
template<class T>
void launchGuess(hipStream_t st, int n, const int* order, const int* gidx, const double* hist, size_t slotStride,
                 GuessCoef gc, const double* alpha, CgRhs rhs, double cself, double* bOut, double* x,
                 typename Vec4<T>::type* xT, const T* rgw = nullptr);
template<class T>
void launchCgInit(hipStream_t st, int n, const double* alpha, CgRhs rhs, const double* x, const double* td,
                  RecField tr, double cself, double* r, double* p,
                  typename Vec4<T>::type* pT, double* partials, double* cg, Precond pc,
                  const T* rgw = nullptr);
// An iteration (Jacobi): the product A p with the sums p.Ap, z.Ap and Ap.f Ap (f the preconditioner's diagonal), then
// everything else in one pass: with step = r.z/p.Ap and z' = z - step f Ap, the Polak-Ribiere numerator z'.(r' - r) is
// -step (z.Ap - step Ap.f Ap), so the direction's coefficient is known before r' is written.
void launchCgAp(hipStream_t st, int n, int it, const double* alpha, const double* p, const double* r, const double* td,
                RecField tr, double cself, double* ap, double* partials, double* cg, CgSkip skip, Precond pc);
template<class T>
void launchCgStep(hipStream_t st, int n, int it, const double* alpha, const double* ap, double* x, double* r,
                  double* p, typename Vec4<T>::type* pT, double* partials, double* cg, CgSkip skip, Precond pc,
                  const T* rgw = nullptr);
// ... and with the short-range preconditioner: launchCgAp, launchCgUpdate, launchPrecond, launchCgDirection.
void launchCgUpdate(hipStream_t st, int n, int it, const double* alpha, const double* p, const double* ap, double* x,
                    double* r, double* partials, double* cg, CgSkip skip);
// z = alpha (r + sum_j T_ij alpha_j r_j) over the short list (partners with alpha_j > 0; M = D when *over), its
// sums into the CG partials: init (after launchCgInit): p = z, r.z; else (after launchCgUpdate of iteration it):
// -step z.Ap and the new r.z (core/cuda/pgm_cuda.cu:1526-1588).
template<class T>
void launchPrecond(hipStream_t st, int n, int it, bool init, const double* alpha, const double* r, const double* ap,
                   const typename Vec4<T>::type* pos, BoxSel<T> box, const int* srCount, const int* srJ,
                   const typename Vec2<T>::type* srG, const int* over, double* z, double* p,
                   typename Vec4<T>::type* pT, double* partials, CgSkip skip, const T* rgw = nullptr);
template<class T>
void launchCgDirection(hipStream_t st, int n, int it, const double* z, double* p, typename Vec4<T>::type* pT,
                       double* partials, CgSkip skip, const T* rgw = nullptr);
// x += peek alpha r; history push (global order, hist may be NULL); total dipoles d = perm + x, also as the pair
// vector type dT with w = the radius parameter rgS of the (sorted) atom.
template<class T>
void launchPost(hipStream_t st, int n, double peek, const double* alpha, const double* r, double* x, const double* perm,
                const int* order, const int* gidx, double* hist, double* d, const double* rgS,
                typename Vec4<T>::type* dT);
// The end of an evaluation in one pass over chunks of atoms (each inside one system): the total field ed + er + cself d
// at the atoms and their covalent neighbours, the covalent chain rule, the forces out (caller's order, added; where
// skip says that a solve enqueued ahead fell short, none), the positions kept, and per chunk the sums of the sorted
// atoms' rows: with strain all of kFinalWide columns, else the kFinalNarrow first ones, which are the pair energy,
// |d|^2, mu^2/(2 alpha) and the GVDW energy; then the pair strain, E_rec (x) d and the covalent strain, 9 each.
constexpr int kFinalNarrow = 4, kFinalWide = 31, kFinalChunk = 256;
// The result slots of one system's evaluation (device, read back once).
enum {
    kResPair = 0,      // energy, strain[9] (pair, already halved)
    kResRec = 10,      // energy, strain[9] (k-space)
    kResComb = 20,     // |d|^2, polarization, E_rec (x) d [9]
    kResCov = 31,      // covalent strain [9]
    kResGvdw = 40,     // GVDW energy
    kResCount = 41,
};
struct FinalArgs {
    int n;
    const int* rank;
    const double* pos;
    const int *covStart, *covPartner;
    const double* covStrength;
    const int *revStart, *revEntry, *covAtomOf;
    const double *d, *mu, *alpha, *ed, *er;   // sorted
    const double *fpair, *frec;               // sorted pair and reciprocal forces
    const double* pairRows;                   // sorted: [n] energy, or with strain [n][10] energy, strain
    const double* gvdw;                       // sorted GVDW energies (nullptr: none)
    double cself, ke;
    BoxSel<double> box;
    double* fAssign;                          // forces assigned, 3n (may be null)
    double* fOut;                             // forces added (each may be null)
    long long* fixedOut;
    int stride;
    double fixedScale;
    CgSkip shortOf;                           // the forces are added only if this says converged (or is unset)
    double* posKeep;                          // pos copied here (may be null)
    const int* chunkStart;
    double* chunkSums;                        // [chunks][kFinalNarrow or kFinalWide]
};
void launchFinal(hipStream_t st, const FinalArgs& a, int nchunks, bool strain);
// The result slots of every system from the chunks' sums and the x pass's partials (recRows: [.][10] energy, strain).
void launchFinalSums(hipStream_t st, const double* chunkSums, bool strain, const int* sysChunk, int nsys,
                     const double* recRows, const int* recStart, const int* sysRec, double* res, int resStride);
// In the caller's order: out[i] = v[rank[i]] (3-vectors).
// The operands of a field evaluation of given charges q and dipoles d (caller's order) into the sorted arrays:
// posD.w and, when set, posT.w = q; dS, dT = d (dT.w = rgw).
template<class T>
void launchFieldOperands(hipStream_t st, int n, const int* order, const double* q, const double* d, const T* rgw,
                         double4* posD, typename Vec4<T>::type* posT, double* dS, typename Vec4<T>::type* dT);
void launchUnsort3(hipStream_t st, int n, const int* rank, const double* v, double* out);

// -------------------------------------------------------------------------------------------- parameter gradients

// In the sorted order: out[s] = v[order[s]] (3-vectors).
void launchSort3(hipStream_t st, int n, const int* order, const double* v, double* out);
// Change of the sorted permanent dipoles when the atoms move by disp (caller's order, FP64 xyz).
void launchPermTangent(hipStream_t st, int n, const int* order, const double* pos, const double* disp,
                       const int* covStart, const int* covPartner, const double* covStrength, BoxSel<double> box,
                       double* pdot);
// b = -(E'_pair + E'_rec + cself p') on polarizable rows (pair / PME tangent outputs, E' at offset 6n).
void launchAdjointRhs(hipStream_t st, int n, const double* alpha, const double* pairOut, const double* pmeOut,
                      const double* pdot, double cself, double* b);
// d' = p' - lambda (lambda may be null), FP64 and the pass vector type.
template<class T>
void launchDipoleTangent(hipStream_t st, int n, const double* pdot, const double* lambda, double* ddot,
                         typename Vec4<T>::type* ddotT);

struct ParamAtomArgs {
    int n;
    const int* order;
    const double *q, *alpha, *mu, *lambda, *d, *ddot;   // sorted; lambda, ddot null without a force cotangent
    const double *pairOut, *pmeOut;                     // pair / PME tangent-pass outputs
    double ke, wE, cself;
    double qSelf;                                       // 2 beta / sqrt(pi)
    double qBackground;                                 // pi Q / (V beta^2) (single system)
    const double* qBackSys;                             // batch: pi Q / (V beta^2) per system
    const double* wESys;                                // batch: dL/dE per system
    const int* sysOf;                                   // batch: system of every atom index
    double *gq, *galpha, *gR;                           // caller's order (each may be null)
    double *etot, *etotDot;                             // sorted total field and its tangent
};
// Per-atom charge, polarizability and radius gradients; total field (and tangent) for the covalent terms.
void launchParamAtoms(hipStream_t st, const ParamAtomArgs& a);
// Covalent-strength gradients per entry, written at the entry's input index.
void launchParamCov(hipStream_t st, int ncov, const int* covAtomOf, const int* covPartner, const int* inputOf,
                    const int* rank, const double* pos, const double* disp, const double* etot,
                    const double* etotDot, BoxSel<double> box, double ke, double wE, const double* wESys,
                    double* gc);

}   // namespace pgmhip
