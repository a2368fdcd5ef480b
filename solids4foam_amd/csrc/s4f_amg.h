// s4f_amg.h -- aggregation multigrid V-cycle used as the PCG preconditioner
// (the device counterpart of running OpenFOAM's PCG with `preconditioner GAMG`).
//
// Hierarchy: plain (piecewise-constant) aggregation of strongly connected
// cells, Galerkin coarse operators A_c = P^T A P, built once per matrix on the
// host.  Cycle: V(1,1) with damped Jacobi smoothing (omega = kMgOmega) and an
// exact solve on the coarsest level (explicit inverse of each instance's
// block, <= kCoarseBlock rows), so the cycle is a fixed symmetric positive
// definite operator and CG stays CG.  A batch of meshes is one block-diagonal
// matrix: aggregates never cross instances, every level keeps each
// instance's rows contiguous, and each row looks up its instance's control
// block (converged instances and components are skipped).
//
// Launch shape per level (level 0: 3 components, SoA, stride = the row
// count, converged components skipped; coarser levels: rows of four):
//   restriction: b_c[I] = sum_{i in I} r[i] (members gathered, no atomics)
//         and the pre-smoothed value x_c = w D_c^-1 b_c in the same pass
//   down: r = b - A x (on level 0 the neighbours' x = w D^-1 b is recomputed
//         from their b and 1/diag)
//   up:   prolongation x += e[agg] fused into the post-smoothing sweep,
//         formed from the down sweep's residual and q = offdiag(A) P (no
//         matrix pass; only the coarser correction is gathered)
// Level 0 is the solver mesh's own sliced-ELL matrix; coarser levels have
// their own sliced-ELL arrays.  Every row's arithmetic runs in a fixed order
// that depends only on its own instance, so results do not depend on which
// other instances share a launch.
#pragma once

#include "s4f_kernels.h"

namespace s4f {

constexpr int kCoarseBlock = 1024;  // rows per instance on the coarsest level (explicit inverse)
constexpr int kMgChunk = 8;         // slots per unconditional load group of the wide (Galerkin / G) rows
// smoothed hierarchy: relative size below which first-coarse-level entries
// are lumped into the diagonal (|a_IJ| < f sqrt(|a_II a_JJ|)).  Off: lumping
// keeps row sums but can make the coarse operator indefinite (it did on a
// 384-tetrahedron mesh at f = 0.04), and the cycle must stay SPD.
constexpr double kMgSmoothedFilter = 0.0;
constexpr double kMgCoarseScaleDefault = 1.8;  // coarse-correction scale when the caller gives 0
// Jacobi damping of the smoothing sweeps: near the best smoothing factor of
// damped Jacobi for 7-point-like operators in 3-D (6/7) and below 1, where
// the sweep converges on every level's diagonally dominant M-matrix, so the
// cycle stays symmetric positive definite
constexpr double kMgOmega = 0.9;

// device view of one coarse level
struct MgLevel {
    int n;             // rows
    int nSlices;
    const int* sliceStart;
    const int* sliceWidth;
    const int* col;    // >= 0 neighbour row, kPad empty
    const float* a32;  // off-diagonal magnitude (entry = -a)
    const double* a64;
    const float* diag32;
    const double* diag64;
    const float* invD32;
    const double* invD64;
    const int* agg;    // row -> row of the next coarser level (nullptr on the coarsest)
    const int* memOff; // (coarse side) row -> first member of the finer level
    const int* mem;    // members (rows of the finer level)
    const float* memW32;   // member weights (smoothed prolongation; nullptr: all 1)
    const double* memW64;
    const int* rStart;     // the weighted member lists as sliced ELL (smoothed prolongation only)
    const int* rWidth;
    const int* rMem;
    const float* rW32;
    const double* rW64;
    const int* rowInst;  // row -> instance
    const int* blkRow0;  // coarsest level, per instance: first row of its block
    const int* blkN;     //   rows of its block
    const int* invOff;   //   offset of its explicit inverse (blkN^2 entries, row-major)
    const int* pass;     // per instance: passes through this level unchanged (no smoothing, no scaling)
    const int* qCol;     // q = offdiag(A) P in the level's slots (< 0: empty; nullptr on the coarsest)
    const float* q32;
    const double* q64;
    const int* qWidth;   // per slice: filled q slots
};

template <typename T> struct MgSel;
template <> struct MgSel<double> {
    __device__ static const double* q(const MgLevel& L) { return L.q64; }
    __device__ static const double* memW(const MgLevel& L) { return L.memW64; }
    __device__ static const double* rW(const MgLevel& L) { return L.rW64; }
    __device__ static const double* a(const MgLevel& L) { return L.a64; }
    __device__ static const double* d(const MgLevel& L) { return L.diag64; }
    __device__ static const double* iD(const MgLevel& L) { return L.invD64; }
};
template <> struct MgSel<float> {
    __device__ static const float* q(const MgLevel& L) { return L.q32; }
    __device__ static const float* memW(const MgLevel& L) { return L.memW32; }
    __device__ static const float* rW(const MgLevel& L) { return L.rW32; }
    __device__ static const float* a(const MgLevel& L) { return L.a32; }
    __device__ static const float* d(const MgLevel& L) { return L.diag32; }
    __device__ static const float* iD(const MgLevel& L) { return L.invD32; }
};

__device__ __forceinline__ bool mgSkip(const Ctl* c) { return c->outerDone || c->innerDone; }

// Coarse-level vectors are rows of four (three components and a zero pad):
// one 16-byte (FP32) or 32-byte (FP64) load per neighbour instead of three
// component gathers; the fine level's residual r0, which the restriction
// gathers, is rows of three.  The PCG's vectors stay component-major.
template <typename T> struct Row4Sel;
template <> struct Row4Sel<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct Row4Sel<double> { typedef double type __attribute__((ext_vector_type(4))); };
template <typename T> using Row4 = typename Row4Sel<T>::type;

// The fine level's residual is stored without the pad: it is as large as the
// PCG's vectors, and written and read once per cell besides the gathers.
// First weighted restriction with rows of four -> three: 45 -> 37 us (128^3 cells,
// FP32), 23.0 -> 21.5 (566,475, FP64); V-cycle at 200^3 0.763 -> 0.725 ms
// (component-major with one wavefront per slice: 0.732).
template <typename T>
struct Row3 {
    T v[3];
    __device__ __forceinline__ T operator[](int j) const { return v[j]; }
};

template <typename T>
__device__ __forceinline__ Row4<T> row4(T a, T b, T c) {
    Row4<T> v;
    v[0] = a; v[1] = b; v[2] = c; v[3] = (T)0;
    return v;
}

// ---------------------------------------------------------------------------
// level 0 (the mesh's own matrix, BlockMap iteration)
// ---------------------------------------------------------------------------

// Level-0 rows with all three components active and a compile-time slot
// count W: every load is issued unconditionally (invalid slots gather the
// row's own cell with a zero coefficient) so a wave's gathers overlap.
template <typename T, int W>
__device__ __forceinline__ void mg0DownRowAll(const DevMesh& m, int P, int e0, int lane, int C, const T* __restrict__ b,
                                              Row3<T>* __restrict__ r, T w) {
    const T* __restrict__ A = MatSel<T>::a(m);
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    int nb[W];
    T a[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const int e = e0 + k * kSlice + lane;
        nb[k] = ldS(m.col + e);
        a[k] = ldS(A + e);
    }
    const T iD = invD[P], dP = MatSel<T>::diag(m)[P];
    T bP[3], xP[3], y[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        bP[j] = b[(size_t)j * C + P];
        xP[j] = w * iD * bP[j];
        y[j] = dP * xP[j];
    }
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const bool v = nb[k] >= 0;
        const int c = v ? nb[k] : P;
        const T av = v ? a[k] : (T)0;
        const T wi = w * invD[c];
#pragma unroll
        for (int j = 0; j < 3; ++j) y[j] -= av * (wi * b[(size_t)j * C + c]);
    }
    r[P] = Row3<T>{{bP[0] - y[0], bP[1] - y[1], bP[2] - y[2]}};
}

// level-0 prolongation + post-smoothing of one row (all three components,
// compile-time slot count W, every load unconditional: an empty slot reads
// the row's own coarse row with a zero weight)
template <typename T, int W>
__device__ __forceinline__ void mg0UpRowAll(const DevMesh& m, const int* __restrict__ qCol, const T* __restrict__ q,
                                            int P, int e0, int lane, int C, const T* __restrict__ b,
                                            const Row3<T>* __restrict__ r0, const int* __restrict__ agg,
                                            const Row4<T>* __restrict__ e, T* __restrict__ z, T w, T w1, T al,
                                            double* acc) {
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    int J[W];
    T qv[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const int en = e0 + k * kSlice + lane;
        J[k] = ldS(qCol + en);
        qv[k] = ldS(q + en);
    }
    const int IP = agg[P];
    const T wi = w * invD[P];
    T s[3] = {(T)0, (T)0, (T)0};
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const bool v = J[k] >= 0;
        const Row4<T> ek = e[v ? J[k] : IP];
        const T c = v ? qv[k] : (T)0;
#pragma unroll
        for (int j = 0; j < 3; ++j) s[j] += c * ek[j];
    }
    const Row4<T> eP = e[IP];
    const Row3<T> rP = r0[P];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const size_t i = (size_t)j * C + P;
        const T bv = b[i];
        const T zv = wi * (bv + rP[j]) + al * (w1 * eP[j] + wi * s[j]);
        stS(z + i, zv);
        acc[j] += (double)zv * (double)bv;
    }
}

// pre-smoothing from zero and the residual for the restriction:
// x = w D^-1 b (not stored: k_mg0_up works from b and r), r = b - A x
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mg0_down(const DevMesh m, const BlockMap bm, const T* __restrict__ b,
                                                     Row3<T>* __restrict__ r, double omega,
                                                     const Ctl* __restrict__ ctl) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int inst = tl.inst;
    const Ctl* c = ctl + inst;
    if (mgSkip(c)) return;
    const int C = m.nCells;
    const T* __restrict__ A = MatSel<T>::a(m);
    const T* __restrict__ dg = MatSel<T>::diag(m);
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const bool act[3] = {c->active[0] != 0, c->active[1] != 0, c->active[2] != 0};
    const bool all = act[0] && act[1] && act[2];
    const T w = (T)omega;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        if (P >= tl.cEnd) continue;
        const int width = m.width(s);
        const int e0 = m.entry0(s);
        if (all && width == 6) {
            mg0DownRowAll<T, 6>(m, P, e0, lane, C, b, r, w);
            continue;
        }
        if (all && width == 4) {
            mg0DownRowAll<T, 4>(m, P, e0, lane, C, b, r, w);
            continue;
        }
        // some components, or another slot count: as in k_spmvp
        const T iD = invD[P], dP = dg[P];
        T bP[3] = {}, y[3] = {};
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if (!act[j]) continue;
            bP[j] = b[(size_t)j * C + P];
            y[j] = rounded(dP * (w * iD * bP[j]));
        }
        for (int k0 = 0; k0 < width; k0 += kRowChunk) {
            int n[kRowChunk];
            T av[kRowChunk], iDn[kRowChunk];
#pragma unroll
            for (int u = 0; u < kRowChunk; ++u) {
                const int e = e0 + (k0 + u < width ? k0 + u : k0) * kSlice + lane;
                const int ne = ldS(m.col + e);
                const T ae = ldS(A + e);
                const bool v = k0 + u < width && ne >= 0;
                n[u] = v ? ne : P;
                av[u] = v ? ae : (T)0;
            }
#pragma unroll
            for (int u = 0; u < kRowChunk; ++u) iDn[u] = invD[n[u]];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                if (!act[j]) continue;
                T bn[kRowChunk];
#pragma unroll
                for (int u = 0; u < kRowChunk; ++u) bn[u] = b[(size_t)j * C + n[u]];
#pragma unroll
                for (int u = 0; u < kRowChunk; ++u) y[j] = fmaT(-av[u], w * iDn[u] * bn[u], y[j]);
            }
        }
        T rP[3];  // a converged component's residual is not read
#pragma unroll
        for (int j = 0; j < 3; ++j) rP[j] = act[j] ? bP[j] - y[j] : (T)0;
        r[P] = Row3<T>{{rP[0], rP[1], rP[2]}};
    }
}

// Prolongation + post-smoothing on level 0.  With x = w D^-1 b the
// pre-smoothed value and r0 = b - A x from k_mg0_down, the corrected
// xf = x + alpha P e and its Jacobi sweep z = xf + w D^-1 (b - A xf) are
//   z = w D^-1 (b + r0) + alpha ((1 - w) e[agg] + w D^-1 sum_J q_J e_J)
// with q = offdiag(A) P grouped per coarse row J (host-built in the fine
// matrix's slots): no fine-matrix pass and no neighbour b, 1/diag or agg
// gathers.  e == nullptr: no coarse correction.  Partial z.b per block (b is
// the PCG residual: z.b = rho of the preconditioned residual).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mg0_up(const DevMesh m, const BlockMap bm, const T* __restrict__ b,
                                                   const Row3<T>* __restrict__ r0, const int* __restrict__ agg,
                                                   const int* __restrict__ qCol, const T* __restrict__ q,
                                                   const Row4<T>* __restrict__ e, T* __restrict__ z, double omega,
                                                   double alpha, const Ctl* __restrict__ ctl,
                                                   double* __restrict__ part) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int inst = tl.inst;
    const Ctl* c = ctl + inst;
    if (mgSkip(c)) return;
    const int C = m.nCells;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const bool act[3] = {c->active[0] != 0, c->active[1] != 0, c->active[2] != 0};
    const bool all = act[0] && act[1] && act[2] && e != nullptr;
    const T w = (T)omega, w1 = (T)(1.0 - omega), al = (T)alpha;
    double acc[3] = {0, 0, 0};
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        if (P >= tl.cEnd) continue;
        const int width = m.width(s);
        const int e0 = m.entry0(s);
        if (all && width == 6) {
            mg0UpRowAll<T, 6>(m, qCol, q, P, e0, lane, C, b, r0, agg, e, z, w, w1, al, acc);
            continue;
        }
        if (all && width == 4) {
            mg0UpRowAll<T, 4>(m, qCol, q, P, e0, lane, C, b, r0, agg, e, z, w, w1, al, acc);
            continue;
        }
        const T wi = w * invD[P];
        T s3[3] = {(T)0, (T)0, (T)0};
        Row4<T> eP = {};
        if (e) {
            eP = e[agg[P]];
            for (int k = 0; k < width; ++k) {
                const int en = e0 + k * kSlice + lane;
                const int J = qCol[en];
                if (J >= 0) {
                    const Row4<T> ek = e[J];
                    const T cq = q[en];
#pragma unroll
                    for (int j = 0; j < 3; ++j) s3[j] += cq * ek[j];
                }
            }
        }
        const Row3<T> rP = r0[P];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if (!act[j]) continue;
            const size_t i = (size_t)j * C + P;
            const T bv = b[i];
            const T zv = e ? wi * (bv + rP[j]) + al * (w1 * eP[j] + wi * s3[j]) : wi * (bv + rP[j]);
            z[i] = zv;
            acc[j] += (double)zv * (double)bv;
        }
    }
    storeBlockPartials<3, 0>(acc, part, kOffRho, lb, bm.nBlocks);
}

// Prolongation + post-smoothing on level 0 of a smoothed hierarchy (the first
// prolongation P = (I - wp D^-1 A) P_aggregation).  The corrected
// xf = x + alpha P e and its Jacobi sweep reduce as in k_mg0_up to
//   z = w D^-1 (b + r0) + alpha w D^-1 sum_J G_J e_J,   G = (D / w) P - A P,
// with G host-built per row in its own sliced-ELL slots (an empty slot
// repeats the row's first column with a zero weight, so every load is
// unconditional and in bounds).  Partial z.b per block.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mg0_up_g(const DevMesh m, const BlockMap bm, const T* __restrict__ b,
                                                     const Row3<T>* __restrict__ r0, const int* __restrict__ gStart,
                                                     const int* __restrict__ gWidth, const int* __restrict__ gCol,
                                                     const T* __restrict__ g, const Row4<T>* __restrict__ e,
                                                     T* __restrict__ z, double omega, double alpha,
                                                     const Ctl* __restrict__ ctl, double* __restrict__ part) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int inst = tl.inst;
    const Ctl* c = ctl + inst;
    if (mgSkip(c)) return;
    const int C = m.nCells;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const bool act[3] = {c->active[0] != 0, c->active[1] != 0, c->active[2] != 0};
    const T w = (T)omega, al = (T)alpha;
    double acc[3] = {0, 0, 0};
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        if (P >= tl.cEnd) continue;
        const int e0 = gStart[s];
        const int width = gWidth[s];
        T sum[3] = {(T)0, (T)0, (T)0};
        for (int k0 = 0; k0 < width; k0 += kMgChunk) {
            int J[kMgChunk];
            T cw[kMgChunk];
#pragma unroll
            for (int u = 0; u < kMgChunk; ++u) {
                const int k = k0 + u < width ? k0 + u : width - 1;
                const int en = e0 + k * kSlice + lane;
                J[u] = ldS(gCol + en);
                cw[u] = k0 + u < width ? ldS(g + en) : (T)0;
            }
#pragma unroll
            for (int u = 0; u < kMgChunk; ++u) {
                const Row4<T> ev = e[J[u]];
#pragma unroll
                for (int j = 0; j < 3; ++j) sum[j] += cw[u] * ev[j];
            }
        }
        const T wi = w * invD[P];
        const Row3<T> rP = r0[P];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if (!act[j]) continue;
            const size_t i = (size_t)j * C + P;
            const T bv = b[i];
            const T zv = wi * (bv + rP[j]) + al * (wi * sum[j]);
            stS(z + i, zv);
            acc[j] += (double)zv * (double)bv;
        }
    }
    storeBlockPartials<3, 0>(acc, part, kOffRho, lb, bm.nBlocks);
}

// ---------------------------------------------------------------------------
// coarse levels (grid-stride over the slices of one level, in the XCD-aware
// order of the level-0 kernels: each XCD a contiguous range of rows, so gathers
// of neighbouring rows and of a restriction's fine members stay in its L2)
//
// A coarse level has few rows of many slots (Galerkin stencils; 27 to 60), so
// a wavefront per slice left most of the chip idle while each walked its slots
// in dependent groups of loads.  A slice's slots are dealt over the workgroup's
// four wavefronts (slot k to wavefront k mod 4, whatever the slice's width:
// the order of a row's sum depends on the row alone) and the four sums added in
// wavefront order.
// Measured, one wavefront per slice -> four: weighted restriction 18.3 -> 6.6 us
// (262,144 fine cells, FP32), 42 -> 24 us (566,475, FP64), 54 -> 45 us (2.1
// million, FP32: bound by its gathers); down sweep 8 -> 4.6 us (262,144).  List
// restriction with one lane per row -> eight: 13.8 -> 4.6 us (262,144), 19.6 ->
// 5.2 us (566,475, FP64), 5.8 -> 3.2 us (20,250 tetrahedra).
// ---------------------------------------------------------------------------

// the instance's PCG runs (rowInst: nullptr where all rows are instance 0's;
// -1: padding row)
__device__ __forceinline__ bool mgLive(const MgLevel& L, int row, bool on, const Ctl* ctl, int& inst) {
    inst = L.rowInst ? (on ? L.rowInst[row] : -1) : 0;
    return on && inst >= 0 && !mgSkip(ctl + inst);
}

// sum += sum over slots k = wave, wave + 4, ... of coef_k x[idx_k], kMgChunk
// slots' loads in flight at a time, all unconditional.  A slot past the width
// reads the group's first one again, and where there is nothing to add row 0 is
// read and dropped: that row belongs to the launch's first instance, so its
// value must not enter even with a zero coefficient (zero times infinity or NaN
// is NaN).  V-cycle with a row of the instance's own gathered in its place ->
// row 0 dropped: 194 -> 191 us (128^3 cells, FP32, smoothed), 53.8 -> 53.0
// (64^3), 120.9 -> 117.7 (83^3, FP64).
template <typename T, typename Row>
__device__ __forceinline__ void slotSum(const int* __restrict__ idx, const T* __restrict__ coef, int width, int wave,
                                        int lane, const Row* __restrict__ x, T* sum) {
    constexpr int kWaves = kBlock / 64;
    for (int k0 = wave; k0 < width; k0 += kWaves * kMgChunk) {
        int J[kMgChunk];
        T c[kMgChunk];
#pragma unroll
        for (int u = 0; u < kMgChunk; ++u) {
            const int k = k0 + kWaves * u;
            const int o = (k < width ? k : k0) * kSlice;
            J[u] = at32(idx + o, lane * 4u);
            c[u] = at32(coef + o, lane * (unsigned)sizeof(T));
        }
#pragma unroll
        for (int u = 0; u < kMgChunk; ++u) {
            const bool v = k0 + kWaves * u < width && J[u] >= 0;
            const Row xv = x[v ? J[u] : 0];
#pragma unroll
            for (int j = 0; j < 3; ++j) sum[j] += c[u] * (v ? xv[j] : (T)0);
        }
    }
}

// the four wavefronts' sums of a slice, in wavefront 0 (a barrier: all threads)
template <typename T>
__device__ __forceinline__ void sumWaves(T (*sh)[3][kSlice], int wave, int lane, T* sum) {
    if (wave > 0) {
#pragma unroll
        for (int j = 0; j < 3; ++j) sh[wave - 1][j][lane] = sum[j];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int q = 0; q < kBlock / 64 - 1; ++q)
#pragma unroll
            for (int j = 0; j < 3; ++j) sum[j] += sh[q][j][lane];
    }
}

// value of the lane at distance 1, 2 (within a quad) and 4 (once a quad's
// lanes hold equal values) of a group of eight
template <int CTRL>
__device__ __forceinline__ float dppOf(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dppOf(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
template <typename T>
__device__ __forceinline__ T sumOf8(T v) {
    v += dppOf<0xB1>(v);   // quad_perm 1 0 3 2
    v += dppOf<0x4E>(v);   // quad_perm 2 3 0 1
    return v + dppOf<0x141>(v);  // row_half_mirror
}

// restriction: bc[I] = sum over members i of I of r[i] (r of the finer level;
// each member weighted when the prolongation into I is smoothed), and the
// coarse pre-smoothed value xc[I] = w D^-1 bc[I] (the coarse level's smoothing
// from zero, formed once here instead of at every use).  Eight lanes per row:
// a row's member list is read in one coalesced load, and levels of a few
// thousand rows still fill the chip.
template <typename T, typename Row>
__global__ __launch_bounds__(kBlock) void k_mg_restrict(const MgLevel Lc, const Row* __restrict__ r,
                                                        Row4<T>* __restrict__ bc, Row4<T>* __restrict__ xc,
                                                        double omega, const Ctl* __restrict__ ctl) {
    constexpr int kRows = kBlock / 8;
    const T* __restrict__ iDg = MgSel<T>::iD(Lc);
    const T* __restrict__ mw = MgSel<T>::memW(Lc);
    const T w = (T)omega;
    const int sub = threadIdx.x & 7;
    for (int I = logicalBlock(gridDim.x) * kRows + (threadIdx.x >> 3); I < Lc.n; I += gridDim.x * kRows) {
        const int k0 = Lc.memOff[I], k1 = Lc.memOff[I + 1];
        const T wi = w * iDg[I];
        int inst;
        if (!mgLive(Lc, I, true, ctl, inst)) continue;  // the eight lanes alike
        T s[3] = {(T)0, (T)0, (T)0};
        // loads unconditional (past the end: the last member again, weight zero)
        for (int kb = k0; kb < k1; kb += 32) {
            int mi[4];
            T wv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = kb + 8 * u + sub;
                const int kc = k < k1 ? k : k1 - 1;
                mi[u] = Lc.mem[kc];
                wv[u] = k < k1 ? (mw ? mw[kc] : (T)1) : (T)0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const Row v = r[mi[u]];
#pragma unroll
                for (int j = 0; j < 3; ++j) s[j] += wv[u] * v[j];
            }
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) s[j] = sumOf8(s[j]);
        // all three components stored: a converged component's coarse
        // values are never read for an active one
        if (sub == 0) bc[I] = row4(s[0], s[1], s[2]);
        if (sub == 1) xc[I] = row4(wi * s[0], wi * s[1], wi * s[2]);
    }
}

// restriction into the first coarse level of a smoothed hierarchy: bc = P^T r0
// with the weighted member lists in the coarse level's sliced-ELL slots (each
// slot one coalesced load of members and weights; members in ascending
// fine-row order), and xc = w D^-1 bc
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mg_restrict_w(const MgLevel Lc, const Row3<T>* __restrict__ r0,
                                                          Row4<T>* __restrict__ bc, Row4<T>* __restrict__ xc,
                                                          double omega, const Ctl* __restrict__ ctl) {
    __shared__ T sh[kBlock / 64 - 1][3][kSlice];
    const T* __restrict__ iDg = MgSel<T>::iD(Lc);
    const T w = (T)omega;
    const int wave = waveOf(), lane = threadIdx.x & 63;
    for (int s = logicalBlock(gridDim.x); s < Lc.nSlices; s += gridDim.x) {
        const int I = s * kSlice + lane;
        const int e0 = Lc.rStart[s];
        const int width = Lc.rWidth[s];
        int inst;
        const bool live = mgLive(Lc, I, I < Lc.n, ctl, inst);
        T sum[3] = {(T)0, (T)0, (T)0};
        if (live) slotSum(Lc.rMem + e0, MgSel<T>::rW(Lc) + e0, width, wave, lane, r0, sum);
        sumWaves<T>(sh, wave, lane, sum);
        if (live && wave == 0) {
            const T wi = w * iDg[I];
            bc[I] = row4(sum[0], sum[1], sum[2]);
            xc[I] = row4(wi * sum[0], wi * sum[1], wi * sum[2]);
        }
        __syncthreads();  // the next slice's sums take the same LDS
    }
}

// down on a coarse level: r = b - A x with x = w D^-1 b from the restriction
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mg_down(const MgLevel L, const Row4<T>* __restrict__ b,
                                                    const Row4<T>* __restrict__ x, Row4<T>* __restrict__ r,
                                                    const Ctl* __restrict__ ctl) {
    __shared__ T sh[kBlock / 64 - 1][3][kSlice];
    const T* __restrict__ dg = MgSel<T>::d(L);
    const int wave = waveOf(), lane = threadIdx.x & 63;
    for (int s = logicalBlock(gridDim.x); s < L.nSlices; s += gridDim.x) {
        const int P = s * kSlice + lane;
        const int e0 = L.sliceStart[s];
        const int width = L.sliceWidth[s];
        int inst;
        const bool live = mgLive(L, P, P < L.n, ctl, inst);
        const bool pass = live && L.pass[inst];  // already coarsest for this instance: hand b down unchanged
        const bool last = live && wave == 0;
        Row4<T> bP = {}, xP = {};
        T d = (T)0;
        if (last) {
            bP = b[P];
            xP = x[P];
            d = dg[P];
        }
        T sum[3] = {(T)0, (T)0, (T)0};
        if (live && !pass) slotSum(L.col + e0, MgSel<T>::a(L) + e0, width, wave, lane, x, sum);
        sumWaves<T>(sh, wave, lane, sum);
        if (last)
            r[P] = pass ? bP
                        : row4(bP[0] - (d * xP[0] - sum[0]), bP[1] - (d * xP[1] - sum[1]), bP[2] - (d * xP[2] - sum[2]));
        __syncthreads();
    }
}

// up on a coarse level: the corrected xf = x + alpha e[agg] and its Jacobi
// sweep out = xf + w D^-1 (b - A xf), formed as on level 0 from the down
// sweep's residual r = b - A x and q = offdiag(A) P:
//   out = x + w D^-1 r + alpha ((1 - w) e[agg] + w D^-1 sum_J q_J e_J)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mg_up(const MgLevel L, const Row4<T>* __restrict__ x,
                                                  const Row4<T>* __restrict__ r, const Row4<T>* __restrict__ e,
                                                  Row4<T>* __restrict__ out, double omega, double alpha,
                                                  const Ctl* __restrict__ ctl) {
    __shared__ T sh[kBlock / 64 - 1][3][kSlice];
    const T* __restrict__ iDg = MgSel<T>::iD(L);
    const T w = (T)omega, w1 = (T)(1.0 - omega), al = (T)alpha;
    const int wave = waveOf(), lane = threadIdx.x & 63;
    for (int s = logicalBlock(gridDim.x); s < L.nSlices; s += gridDim.x) {
        const int P = s * kSlice + lane;
        const int e0 = L.sliceStart[s];
        const int width = L.qWidth[s];
        int inst;
        const bool live = mgLive(L, P, P < L.n, ctl, inst);
        const bool pass = live && L.pass[inst];  // already coarsest: the coarser solution unchanged
        const bool last = live && wave == 0;
        Row4<T> xv = {}, rv = {}, eP = {};
        T iD = (T)0;
        if (last) {
            eP = e[L.agg[P]];
            xv = x[P];
            rv = r[P];
            iD = iDg[P];
        }
        T sum[3] = {(T)0, (T)0, (T)0};
        if (live && !pass) slotSum(L.qCol + e0, MgSel<T>::q(L) + e0, width, wave, lane, e, sum);
        sumWaves<T>(sh, wave, lane, sum);
        if (last) {
            const T wi = w * iD;
            out[P] = pass ? eP
                          : row4(xv[0] + wi * rv[0] + al * (w1 * eP[0] + wi * sum[0]),
                                 xv[1] + wi * rv[1] + al * (w1 * eP[1] + wi * sum[1]),
                                 xv[2] + wi * rv[2] + al * (w1 * eP[2] + wi * sum[2]));
        }
        __syncthreads();
    }
}

// coarsest level: x = A^-1 b with the explicit (symmetric) inverse of the
// row's instance block, one wavefront per row (each lane's terms in column
// order, then the wavefront reduction)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mg_dense(const MgLevel L, const T* __restrict__ Ainv,
                                                     const Row4<T>* __restrict__ b, Row4<T>* __restrict__ x,
                                                     const Ctl* __restrict__ ctl) {
    const int row = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    int inst;
    if (!mgLive(L, row, row < L.n, ctl, inst)) return;
    const int r0 = L.blkRow0[inst], nb = L.blkN[inst];
    double acc[3] = {0, 0, 0};
    const T* __restrict__ a = Ainv + (size_t)L.invOff[inst] + (size_t)(row - r0) * nb;
#pragma unroll 4
    for (int k = lane; k < nb; k += 64) {
        const double v = (double)a[k];
        const Row4<T> bk = b[r0 + k];
#pragma unroll
        for (int j = 0; j < 3; ++j) acc[j] += v * (double)bk[j];
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) acc[j] = waveReduce<false>(acc[j]);
    if (lane == 0) x[row] = row4((T)acc[0], (T)acc[1], (T)acc[2]);
}

// ---------------------------------------------------------------------------
// packing of per-mesh hierarchies into one block-diagonal hierarchy (server)
// ---------------------------------------------------------------------------

// int segment: mode 0 dst = src + add; 1 dst = src >= 0 ? src + add : src;
// 2 dst = add + k; 3 dst = add
struct SegInt {
    const int* src;
    int* dst;
    int n, add, mode, pad;
};
// 32-bit word copy segment
struct SegWords {
    const unsigned* src;
    unsigned* dst;
    long long n;
};

__global__ __launch_bounds__(kBlock) void k_seg_int(const SegInt* __restrict__ segs) {
    const SegInt g = segs[blockIdx.y];
    for (int k = blockIdx.x * kBlock + threadIdx.x; k < g.n; k += gridDim.x * kBlock) {
        int v;
        if (g.mode == 0) v = g.src[k] + g.add;
        else if (g.mode == 1) { v = g.src[k]; if (v >= 0) v += g.add; }
        else if (g.mode == 2) v = g.add + k;
        else v = g.add;
        g.dst[k] = v;
    }
}

__global__ __launch_bounds__(kBlock) void k_seg_words(const SegWords* __restrict__ segs) {
    const SegWords g = segs[blockIdx.y];
    for (long long k = (long long)blockIdx.x * kBlock + threadIdx.x; k < g.n; k += (long long)gridDim.x * kBlock)
        g.dst[k] = g.src[k];
}

}  // namespace s4f
