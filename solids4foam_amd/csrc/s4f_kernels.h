// s4f_kernels.h -- HIP kernels of the segregated small-strain solid solver.
//
// All kernels walk the sliced-ELL cell->face lists: wave w of a workgroup
// owns one 64-row slice at a time, lane l owns one cell, and each slot of the
// slice is one coalesced load per array.  Face contributions are gathered
// per cell in OpenFOAM's face order, so no atomics touch field data and the
// summation order is fixed (run-to-run bitwise deterministic).  Reductions
// are per workgroup (wave shuffles + LDS) into a partial array; the next kernel
// of a merged launch sequence (Chain), or else a one-block-per-instance finalize
// kernel, then reduces the instance's partials in fixed order and updates the
// control block (kernel boundaries order the writes of every XCD before they
// are read).
//
// Kernel <-> reference map (paths relative to the solids4foam tree):
//   k_residual   linGeomTotalDispSolid.C:141-149: fvc::div(sigma) [Gauss linear]
//                + momentumStabilisation.C:210-217 (RhieChow) + the normalisation
//                of OpenFOAM lduMatrix::solver::normFactor for the PCG initial residual
//   k_spmvp      OpenFOAM PCG search-direction update p = z + beta p fused with
//                lduMatrix::Amul (3 right-hand sides sharing M)
//   k_update     OpenFOAM PCG solution/residual update + diagonal preconditioner
//   fin* / k_fin  the scalar parts of PCG::solve / normFactor / solidModel::converged
//   k_grad       solidTractionFvPatchVectorField.C:398-463 / fixedDisplacement
//                boundary values, leastSquares grad(D) (mechanicalModel.C:571-582),
//                gaussGrad boundary correction, linearElastic::correct on
//                boundary faces (linearElastic.C:318-339), solidTraction
//                updateCoeffs (:321-395 + linGeomTotalDispSolid.C:235-271) and
//                solidModel::converged (solidModelTemplates.C:26-188)
#pragma once

#include "s4f_device.h"

namespace s4f {

// One workgroup tile: its instance, slices [s0, s1), the end of the
// instance's cells, and the instance's tiles and cell count (32 bytes, one
// scalar load)
struct alignas(32) Tile {
    int inst, s0, s1, cEnd, blk0, nBlk, nCell, pad;
};

struct BlockMap {
    const Tile* tile;  // each logical block's tile
    // one instance (spb > 0): tiles of spb slices from slice 0, computed
    // instead of loaded (a load less in front of every kernel's own loads)
    int spb, nSlices, nCells;
    const int* iBlk0;  // per instance: first logical block
    const int* iNBlk;  // per instance: number of blocks
    const int* iNCell; // per instance: number of cells
    const int* finInst;// instance finalized by finalize-kernel workgroup i (nullptr: i itself)
    const int* iB0;    // per instance: first boundary face
    const int* iNB;    // per instance: number of boundary faces
    int nBlocks;
    __device__ __forceinline__ Tile at(int lb) const {
        if (spb == 0) return tile[lb];
        const int s0 = lb * spb;
        return Tile{0, s0, s0 + spb < nSlices ? s0 + spb : nSlices, nCells, 0, nBlocks, nCells, 0};
    }
};

// Workgroups are dispatched round-robin over the 8 XCDs (hardware block b runs
// on XCD b % 8).  Give XCD x a contiguous run of logical blocks so that
// neighbouring cells (and their gathers) stay in one XCD's L2.
__device__ __forceinline__ int logicalBlock(int nb) {
    const int b = blockIdx.x;
    const int x = b & 7, q = nb >> 3, r = nb & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// NaN-propagating maximum (fmax would drop a NaN and hide a diverged solve)
__device__ __forceinline__ double nanMax(double a, double b) { return (b > a || b != b) ? b : a; }

// v of the lane a row rotation away (a row: 16 lanes)
template <int ROR>
__device__ __forceinline__ double rowRor(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x120 + ROR, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x120 + ROR, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// x + y (or their maximum) of the two halves (32) or the two rows of each half
// (16): with values a and b, lanes of the lower half (even row) get a's result,
// those of the upper half (odd row) b's
template <bool MAX>
__device__ __forceinline__ double redOp(double x, double y) { return MAX ? nanMax(x, y) : x + y; }
template <bool MAX>
__device__ __forceinline__ double halves(double a, double b) {
    const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return redOp<MAX>(__hiloint2double(h[0], l[0]), __hiloint2double(h[1], l[1]));
}
template <bool MAX>
__device__ __forceinline__ double rows(double a, double b) {
    const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return redOp<MAX>(__hiloint2double(h[0], l[0]), __hiloint2double(h[1], l[1]));
}
template <bool MAX>
__device__ __forceinline__ double inRow(double v) {
    v = redOp<MAX>(v, rowRor<8>(v));
    v = redOp<MAX>(v, rowRor<4>(v));
    v = redOp<MAX>(v, rowRor<2>(v));
    return redOp<MAX>(v, rowRor<1>(v));
}

// Butterfly over the wavefront (distances 32, 16, 8, 4, 2, 1): every lane gets
// the result.  The first two steps swap half-wavefronts and rows in registers,
// the others rotate within a row: once lanes at the larger distances hold
// equal values, a rotation by d gives the value of the lane at distance d.
template <bool MAX>
__device__ __forceinline__ double waveReduce(double v) {
    v = halves<MAX>(v, v);
    return inRow<MAX>(rows<MAX>(v, v));
}

// The same tree for N values at once, each step halving the values a lane
// carries (21 additions for 12 values instead of 72): value i of the
// wavefront goes to out[4 i + w].  The reductions were 8 of 20 KB of the
// merged residual's code, and a kernel of a few workgroups mostly waits for
// its instructions.
template <int N, bool MAX>
__device__ __forceinline__ void waveReduceTo(const double* v, double* out, int w) {
    constexpr int M = (N + 1) / 2, K = (M + 1) / 2;
    double r[M], q[K];
#pragma unroll
    for (int i = 0; i < M; ++i) r[i] = halves<MAX>(v[i], v[i + M < N ? i + M : i]);
#pragma unroll
    for (int i = 0; i < K; ++i) q[i] = inRow<MAX>(rows<MAX>(r[i], r[i + K < M ? i + K : i]));
    const int lane = threadIdx.x & 63;
    if ((lane & 15) == 0) {
        const int upper = lane >> 5, odd = (lane >> 4) & 1;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const int ir = odd && i + K < M ? i + K : i;
            const int iv = upper && ir + M < N ? ir + M : ir;
            out[4 * iv + w] = q[i];
        }
    }
}
// values [0, NMAX) by maximum, the rest by sum
template <int N, int NMAX>
__device__ __forceinline__ void waveReduceAll(const double* v, double* out, int w) {
    if constexpr (NMAX > 0) waveReduceTo<NMAX, true>(v, out, w);
    waveReduceTo<N - NMAX, false>(v + NMAX, out + 4 * NMAX, w);
}
// value i over the workgroup's wavefronts, from out[4 i + w]
template <int NMAX>
__device__ __forceinline__ double overWaves(const double* out, int i) {
    double r = out[4 * i];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) r = i < NMAX ? nanMax(r, out[4 * i + w]) : r + out[4 * i + w];
    return r;
}

constexpr int kFinBlock = 256;
constexpr int kFinWideTiles = 4096;

// Block partials are stored value-major: value i of logical block lb sits at
// part[i * nb + lb] (nb = the launch's logical block count), so a finalize
// reads each value's partials as one contiguous run instead of one 128-byte
// row per block.
//
// Fixed-order reduction of the instance's partials (one workgroup per
// instance); the first NMAX values by maximum, the others by sum.  Result in
// out[0..NV) (shared), valid for every thread after the call.
template <int NV, int NMAX>
__device__ void finReduce(const double* __restrict__ part, int nb, int blk0, int nblk, double* out) {
    double v[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = 0.0;
    for (int b = threadIdx.x; b < nblk; b += kFinBlock) {
        const double* col = part + blk0 + b;
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = i < NMAX ? nanMax(v[i], col[(size_t)i * nb]) : v[i] + col[(size_t)i * nb];
    }
    __shared__ double sh[4 * NV];
    waveReduceAll<NV, NMAX>(v, sh, threadIdx.x >> 6);
    __syncthreads();
    if (threadIdx.x < NV) out[threadIdx.x] = overWaves<NMAX>(sh, threadIdx.x);
    __syncthreads();
}

// block-level reduction of NV per-thread values (the first NMAX by maximum);
// threads 0..NV-1 store them at part[(off + i) * nb + lb]
template <int NV, int NMAX>
__device__ __forceinline__ void storeBlockPartials(const double* acc, double* part, int off, int lb, int nb) {
    __shared__ double sh[4 * NV];
    waveReduceAll<NV, NMAX>(acc, sh, threadIdx.x >> 6);
    __syncthreads();
    if (threadIdx.x < NV) part[(size_t)(off + threadIdx.x) * nb + lb] = overWaves<NMAX>(sh, threadIdx.x);
}

// ---------------------------------------------------------------------------
// The control block's path through the launch sequence.
//
// Every reducing kernel leaves block partials; the scalars they give (alpha,
// beta, residual norms, convergence) are needed by the next kernel only.  Up
// to kMergeTiles tiles per instance that kernel's workgroups each reduce the
// partials themselves (same order, same bits in every workgroup), apply the
// scalar step to a copy of the control block in LDS, and the instance's first
// workgroup writes it to the next control block of the chain: no launch
// between two kernels of the PCG.  Above that a one-workgroup finalize kernel
// (k_fin) does it in place.  Measured at 5,000 cells (20 tiles), FP64 diagonal
// PCG: 20.2 us per iteration with finalize kernels, 11.3 us merged.
// ---------------------------------------------------------------------------
struct Stage {
    const Ctl* in;  // control blocks left by the previous kernel of the chain
    Ctl* out;       // where the resolved ones go
    double* hist;   // per-outer-iteration history (may be null)
};

// points of the launch sequence at which scalars are resolved
enum Point {
    kPtGrad = 0,    // before the gradient step: PCG convergence; may the outer step run?
    kPtRes = 1,     // before the residual: solidModel::converged, next outer iteration
    kPtInner = 2,   // before the first PCG iteration of a pass: PCG start (normFactor, initial residual)
    kPtAgain = 3,   // before a further one: the previous iteration's convergence
    kPtSpmv = 4,    // before the matrix product of a multigrid PCG: beta
    kPtUpdate = 5,  // before the solution update: alpha
    kPtSettle = 6   // PCG convergence only (the tile map is about to change, or the host reads the state)
};

static_assert(sizeof(Ctl) % 8 == 0 && sizeof(Ctl) / 8 <= 64, "control block copied by one wavefront");

// The scalar steps run on lanes 0..2 of a workgroup's first wavefront, one per
// component (j), on the LDS copy of the control block; what concerns the
// instance as a whole follows on lane 0.

// Each reads what it needs of the control block before it writes to it (val(i):
// value i of the reduced partials): one round of LDS reads, where reads between
// the writes waited for one another (1.1 us of every kernel's passage, now 0.5).

// PCG::solve start: normFactor (lduMatrix::solver::normFactor), normalised
// initial residual, convergence check before the first iteration, z.r; returns
// whether any component iterates
template <typename V>
__device__ __forceinline__ bool finResidual(Ctl* c, const V& val, int j) {
    const double v0 = val(j), v1 = val(3 + j), v2 = val(6 + j), rho = val(9 + j);
    const bool solved = (c->solveMask >> j) & 1;  // fvMatrix::solveSegregated valid components
    const int maxIter = c->pcgMaxIter;
    const double tol = c->pcgTol;
    const double nf = v1 + v2 + 1e-20;
    const double ir = solved ? v0 / nf : 0.0;
    c->normFactor[j] = nf;
    c->initRes[j] = ir;
    c->finalRes[j] = ir;
    c->rho[j] = rho;
    c->nIter[j] = 0;
    c->alpha[j] = 0.0;
    c->beta[j] = 0.0;
    // iterate unless already converged (finalRes = initRes < tolerance)
    const int act = solved && (maxIter > 0) && !(ir < tol);
    c->active[j] = act;
    const bool any = __ballot(act) != 0;
    const double ir1 = __shfl(ir, 1), ir2 = __shfl(ir, 2);
    if (j == 0) {
        c->initResMag = sqrt(ir * ir + ir1 * ir1 + ir2 * ir2);
        c->innerDone = !any;
        c->firstInner = 1;
        c->pIt = 0;
        c->pending = kPendNone;
    }
    return any;
}

// PCG convergence per component (tolerance, relTol, maxIter) and beta; returns
// whether any component iterates on
template <typename V>
__device__ __forceinline__ bool finUpdate(Ctl* c, const V& val, int j) {
    const int did = c->active[j], n = c->nIter[j] + 1, maxIter = c->pcgMaxIter, pcMode = c->pcMode, it = c->pIt;
    const double nf = c->normFactor[j], tol = c->pcgTol, rel = c->pcgRelTol, ir = c->initRes[j], rho = c->rho[j];
    const long long total = c->innerTotal;
    const double v0 = val(j), v1 = val(3 + j);
    int act = did;
    if (act) {
        const double fr = v1 / nf;
        c->nIter[j] = n;
        c->finalRes[j] = fr;
        const bool conv = fr < tol || (rel > 1e-20 && fr < rel * ir);
        act = !conv && n < maxIter;
        if (pcMode == 0) {  // diagonal preconditioner: z.r came with the update
            c->beta[j] = v0 / rho;
            c->rho[j] = v0;
        }
        c->active[j] = act;
    }
    const bool any = __ballot(act) != 0;
    const int count = __popcll(__ballot(did));
    if (j == 0) {
        c->innerTotal = total + count;
        c->innerDone = !any;
        c->firstInner = 0;
        c->pIt = it + 1;
        c->pending = kPendNone;
    }
    return any;
}

// alpha = rho / p.q, with PCG's singularity test |p.q|/normFactor < VSMALL
template <typename V>
__device__ __forceinline__ void finSpmv(Ctl* c, const V& val, int j) {
    int act = c->active[j];
    const double nf = c->normFactor[j], rho = c->rho[j], v = val(j);
    double al = 0.0;
    if (act) {
        if (fabs(v) / nf < kVSmall) {
            act = 0;
            c->active[j] = 0;
        } else {
            al = rho / v;
        }
    }
    c->alpha[j] = al;
    const bool any = __ballot(act) != 0;
    if (j == 0) {
        if (!any) c->innerDone = 1;
        c->pending = any ? kPendUpd : kPendNone;
    }
}

// rho' = z.r of a V-cycle-preconditioned PCG: beta = rho'/rho (first
// iteration: no beta), rho = rho'
template <typename V>
__device__ __forceinline__ void finRho(Ctl* c, const V& val, int j) {
    const int act = c->active[j], first = c->firstInner;
    const double rho = c->rho[j], v = val(j);
    if (act) {
        c->beta[j] = first ? 0.0 : v / rho;
        c->rho[j] = v;
    }
    if (j == 0) c->pending = kPendSpmv;
}

// solidModel::converged (total-displacement form) and the mean field for the
// next normFactor
template <typename V>
__device__ __forceinline__ void finGrad(Ctl* c, const V& val, double nc, int inst, double* hist, int j) {
    const double v0 = val(0), v1 = val(1), v2 = val(2), vs = val(3 + j);
    const double ir = c->initResMag, solTol = c->solTol, altTol = c->altTol;
    const int i = c->iCorr, n0 = c->nIter[0], n1 = c->nIter[1], n2 = c->nIter[2], nCorr = c->nCorr, cap = c->histCap;
    const int dpar = c->dpar;
    const long long total = c->pcgTotal;
    c->xbar[j] = vs / nc;
    if (j != 0) return;
    c->dpar = dpar ^ 1;  // k_grad wrote D' into the other buffer
    const double dmax = sqrt(v2);  // the partials are squares: sqrt is monotonic
    double denom = sqrt(v1);
    if (denom < kSmall) denom = dmax < kSmall ? kSmall : dmax;
    const double rvf = sqrt(v0) / denom;
    c->rvf = rvf;
    const int n01 = n0 > n1 ? n0 : n1;
    c->pcgTotal = total + (n01 > n2 ? n01 : n2);
    const bool conv = i > 1 && ((ir < solTol && rvf < solTol) || rvf < altTol || ir < altTol);
    if (hist && i < cap) {
        double* h = hist + (size_t)inst * 3 * cap;
        h[i] = ir;
        h[cap + i] = rvf;
        h[2 * cap + i] = (double)(n0 + n1 + n2);
    }
    int done = 1;
    if (!isfinite(ir) || !isfinite(rvf)) c->diverged = 1;
    else if (conv) c->converged = 1;
    else if (i + 1 < nCorr) done = 0;
    if (done) {
        c->outerDone = 1;
        c->nOuter = i + 1;
    } else {
        c->iCorr = i + 1;
    }
    c->pending = done ? kPendNone : kPendRes;
}

// the PCG has finished: mixed precision's stall test (an |initRes| with no new
// minimum 1 % below the last one within the window stops the instance here),
// then the outer step may run
struct InnerEnd {
    int outerDone, hold, window, iCorr, bestIt;
    double res, best;
    __device__ __forceinline__ void read(const Ctl* c) {
        outerDone = c->outerDone; hold = c->hold; window = c->stallWindow; iCorr = c->iCorr; bestIt = c->bestIt;
        res = c->initResMag; best = c->bestRes;
    }
    __device__ __forceinline__ void run(Ctl* c, int innerDone, int pending) const {
        if (outerDone || !innerDone || pending != kPendNone || hold) return;
        if (window > 0 && iCorr >= 2) {
            if (res < 0.99 * best) {
                c->bestRes = res;
                c->bestIt = iCorr;
            } else if (iCorr - bestIt >= window) {
                c->stalled = 1;
                c->hold = 1;
                return;
            }
        }
        c->pending = kPendGrad;
    }
};

// what a point of the launch sequence reduces: the pending step, its partials
template <int POINT> struct PointOf;
template <> struct PointOf<kPtGrad> { enum { pend = kPendUpd, off = kOffUpd, nv = 6, nmax = 0 }; };
template <> struct PointOf<kPtRes> { enum { pend = kPendGrad, off = kOffGrad, nv = 6, nmax = 3 }; };
template <> struct PointOf<kPtInner> { enum { pend = kPendRes, off = kOffRes, nv = 12, nmax = 0 }; };
template <> struct PointOf<kPtAgain> { enum { pend = kPendUpd, off = kOffUpd, nv = 6, nmax = 0 }; };
template <> struct PointOf<kPtSpmv> { enum { pend = kPendRho, off = kOffRho, nv = 3, nmax = 0 }; };
template <> struct PointOf<kPtUpdate> { enum { pend = kPendSpmv, off = kOffSpmv, nv = 3, nmax = 0 }; };
template <> struct PointOf<kPtSettle> { enum { pend = kPendUpd, off = kOffUpd, nv = 6, nmax = 0 }; };

// A kernel's passage through its point, in three parts so that its own loads
// can be in flight meanwhile:
//   load()    the control block's words and this thread's first partial row
//   reduce()  the control block in LDS and the reduced partials (one barrier)
//   finish()  the scalar step, the instance's first workgroup stores the
//             result (one barrier)
template <int POINT>
struct StageRun {
    typedef PointOf<POINT> Pt;
    long long word;
    double v[Pt::nv];
    __device__ __forceinline__ void load(const Ctl* in, const double* __restrict__ part, int nb, int blk0, int nblk) {
        constexpr int n = (int)(sizeof(Ctl) / 8);
        word = (int)threadIdx.x < n ? reinterpret_cast<const long long*>(in)[threadIdx.x] : 0;
        const double* col = part + (size_t)Pt::off * nb + blk0 + threadIdx.x;
#pragma unroll
        for (int i = 0; i < Pt::nv; ++i) v[i] = (int)threadIdx.x < nblk ? col[(size_t)i * nb] : 0.0;
    }
    // owed: false if the caller knows that finish() will not use the partials
    __device__ __forceinline__ void reduce(Ctl* sh, double* tot, const double* __restrict__ part, int nb, int blk0,
                                           int nblk, bool owed = true) {
        constexpr int n = (int)(sizeof(Ctl) / 8);
        if ((int)threadIdx.x < n) reinterpret_cast<long long*>(sh)[threadIdx.x] = word;
        if (!owed) {
            __syncthreads();
            return;
        }
        const double* col = part + (size_t)Pt::off * nb + blk0;
        for (int b = threadIdx.x + kFinBlock; b < nblk; b += kFinBlock)
#pragma unroll
            for (int i = 0; i < Pt::nv; ++i) {
                const double x = col[(size_t)i * nb + b];
                v[i] = i < Pt::nmax ? nanMax(v[i], x) : v[i] + x;
            }
        const int w = waveOf();
        if (w == 0 || nblk > 64) waveReduceAll<Pt::nv, Pt::nmax>(v, tot, w);
        else if ((int)(threadIdx.x & 63) < Pt::nv) tot[4 * (threadIdx.x & 63) + w] = 0.0;  // no rows here
        __syncthreads();
    }
    // tot[4 i + w]: wavefront w's share of value i
    __device__ __forceinline__ void finish(Ctl* sh, const double* tot, const Tile& tl, double* hist, bool first,
                                           Ctl* out) {
        if (threadIdx.x < 3) {
            const int j = threadIdx.x;
            int pend = sh->pending, innerDone = sh->innerDone;
            const int outerDone = sh->outerDone, pcMode = sh->pcMode;
            InnerEnd end;
            if constexpr (POINT == kPtGrad) end.read(sh);
            if (pend == Pt::pend) {
                auto val = [&](int i) { return overWaves<Pt::nmax>(tot, i); };
                if constexpr (POINT == kPtRes) {
                    finGrad(sh, val, (double)tl.nCell, tl.inst, first ? hist : nullptr, j);
                } else if constexpr (POINT == kPtInner) {
                    innerDone = !finResidual(sh, val, j);
                    pend = kPendNone;
                } else if constexpr (POINT == kPtSpmv) {
                    finRho(sh, val, j);
                } else if constexpr (POINT == kPtUpdate) {
                    finSpmv(sh, val, j);
                } else {
                    innerDone = !finUpdate(sh, val, j);
                    pend = kPendNone;
                }
            } else if (POINT == kPtRes && pend == kPendStart) {
                if (j == 0) sh->pending = kPendRes;
            }
            if (j == 0) {
                if constexpr (POINT == kPtGrad) end.run(sh, innerDone, pend);
                if ((POINT == kPtInner || POINT == kPtAgain) && !outerDone && !innerDone && pend == kPendNone)
                    sh->pending = pcMode ? kPendRho : kPendSpmv;
            }
        }
        __syncthreads();
        if (out && first) {
            constexpr int n = (int)(sizeof(Ctl) / 8);
            if ((int)threadIdx.x < n)
                reinterpret_cast<long long*>(out)[threadIdx.x] = reinterpret_cast<const long long*>(sh)[threadIdx.x];
        }
    }
};

__device__ __forceinline__ int pendingOf(const Ctl* c) { return __builtin_amdgcn_readfirstlane(c->pending); }

// linearElastic: sigma = 2 mu dev(symm G) + K tr(symm G) I   (xx xy xz yy yz zz)
__device__ __forceinline__ void hooke(const double* G, double mu, double K, double* s) {
    const double e0 = G[0], e1 = 0.5 * (G[1] + G[3]), e2 = 0.5 * (G[2] + G[6]);
    const double e3 = G[4], e4 = 0.5 * (G[5] + G[7]), e5 = G[8];
    const double tr = e0 + e3 + e5;
    const double sh = K * tr;
    const double t3 = tr / 3.0;
    s[0] = 2.0 * mu * (e0 - t3) + sh;
    s[1] = 2.0 * mu * e1;
    s[2] = 2.0 * mu * e2;
    s[3] = 2.0 * mu * (e3 - t3) + sh;
    s[4] = 2.0 * mu * e4;
    s[5] = 2.0 * mu * (e5 - t3) + sh;
}

__device__ __forceinline__ double cellMu(const DevMesh& m, int c) { return m.mu ? m.mu[c] : m.mu0; }
__device__ __forceinline__ double cellK(const DevMesh& m, int c) { return m.K ? m.K[c] : m.K0; }
__device__ __forceinline__ double cellImpK(const DevMesh& m, int c) { return m.impK ? m.impK[c] : m.impK0; }

__device__ __forceinline__ double fmaT(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmaT(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// v, rounded here: no later addition contracts with the product that formed it
template <typename T>
__device__ __forceinline__ T rounded(T v) {
    asm("" : "+v"(v));
    return v;
}

// a.b, rounded as the compiler contracts a0 b0 + a1 b1 + a2 b2
__device__ __forceinline__ double dot3(double a0, double b0, double a1, double b1, double a2, double b2) {
    return fmaT(a2, b2, fmaT(a0, b0, a1 * b1));
}

// A group of loads ends here: the scheduler would otherwise put each next to its
// first use to save registers, and they would wait for one another.
__device__ __forceinline__ void loadedHere(double& a, double& b, double& c, double& d, double& e, double& f, double* g,
                                           double* h, double* i) {
    asm volatile(""
                 : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e), "+v"(f), "+v"(g[0]), "+v"(g[1]), "+v"(g[2]),
                   "+v"(g[3]), "+v"(g[4]), "+v"(g[5]), "+v"(g[6]), "+v"(g[7]), "+v"(g[8]), "+v"(h[0]), "+v"(h[1]),
                   "+v"(h[2]), "+v"(i[0]), "+v"(i[1]), "+v"(i[2]));
}

__device__ __forceinline__ void loadedHere(double* x) {
    asm volatile(""
                 : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]), "+v"(x[6]), "+v"(x[7]),
                   "+v"(x[8]), "+v"(x[9]), "+v"(x[10]), "+v"(x[11]), "+v"(x[12]), "+v"(x[13]), "+v"(x[14]),
                   "+v"(x[15]), "+v"(x[16]), "+v"(x[17]), "+v"(x[18]), "+v"(x[19]), "+v"(x[20]), "+v"(x[21]),
                   "+v"(x[22]), "+v"(x[23]));
}
__device__ __forceinline__ void loadedHere(double (*a)[3], double (*b)[3], double (*c)[3], double* s) {
    asm volatile(""
                 : "+v"(a[0][0]), "+v"(a[0][1]), "+v"(a[0][2]), "+v"(a[1][0]), "+v"(a[1][1]), "+v"(a[1][2]),
                   "+v"(b[0][0]), "+v"(b[0][1]), "+v"(b[0][2]), "+v"(b[1][0]), "+v"(b[1][1]), "+v"(b[1][2]),
                   "+v"(c[0][0]), "+v"(c[0][1]), "+v"(c[0][2]), "+v"(c[1][0]), "+v"(c[1][1]), "+v"(c[1][2]),
                   "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(s[4]), "+v"(s[5]), "+v"(s[6]), "+v"(s[7]),
                   "+v"(s[8]));
}

template <typename T> struct MatSel;
template <> struct MatSel<double> {
    __device__ static const double* a(const DevMesh& m) { return m.eA; }
    __device__ static const double* diag(const DevMesh& m) { return m.diag; }
    __device__ static const double* invDiag(const DevMesh& m) { return m.invDiag; }
};
template <> struct MatSel<float> {
    __device__ static const float* a(const DevMesh& m) { return m.eA32; }
    __device__ static const float* diag(const DevMesh& m) { return m.diag32; }
    __device__ static const float* invDiag(const DevMesh& m) { return m.invDiag32; }
};

// Internal-face slots of a k_residual row of any slot count (launches without a
// single one of 6 or 4; the others take k_residual_u), branch-free: a boundary or empty slot gathers the row's own cell and has
// zero area, Rhie-Chow and matrix coefficients, so it adds exactly zero.
// Rows list internal faces before boundary faces, so running the boundary
// slots afterwards keeps the summation order of the slot loop.
__device__ __forceinline__ void residualInternal(const DevMesh& m, int P, int e0, int W, int lane, int C,
                                                  const double* __restrict__ D, const double* __restrict__ G,
                                                  const double* DP, const double* GP, const double* CP,
                                                  const double* sP, double sf, double* div, double* rc,
                                                  double* off, double& asum, bool& hasB) {
    const size_t E = m.nEntries;
#pragma unroll 1
    for (int k = 0; k < W; ++k) {
        const int e = e0 + k * kSlice + lane;
        const int n = ldS(m.col + e);
        const bool v = n >= 0;
        hasB |= (!v && n != kPad);
        const int c = v ? n : P;
        const double S0r = ldS(m.eS + e), S1r = ldS(m.eS + E + e), S2r = ldS(m.eS + 2 * E + e);
        const double w = ldS(m.eW + e), cfr = ldS(m.eC + e), ar = ldS(m.eA + e);
        const double S0 = v ? S0r : 0.0, S1 = v ? S1r : 0.0, S2 = v ? S2r : 0.0;
        const double cf = v ? cfr : 0.0, a = v ? ar : 0.0;
        double GN[9], sN[6], DN[3], d[3];
#pragma unroll
        for (int q = 0; q < 9; ++q) GN[q] = G[(size_t)q * C + c];
#pragma unroll
        for (int q = 0; q < 3; ++q) { DN[q] = D[(size_t)q * C + c]; d[q] = m.cC[(size_t)q * C + c] - CP[q]; }
        hooke(GN, cellMu(m, c) * sf, cellK(m, c) * sf, sN);
        double sfc[6];
#pragma unroll
        for (int q = 0; q < 6; ++q) sfc[q] = w * (sP[q] - sN[q]) + sN[q];
        div[0] += S0 * sfc[0] + S1 * sfc[1] + S2 * sfc[2];
        div[1] += S0 * sfc[1] + S1 * sfc[3] + S2 * sfc[4];
        div[2] += S0 * sfc[2] + S1 * sfc[4] + S2 * sfc[5];
        double Gf[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) Gf[q] = w * (GP[q] - GN[q]) + GN[q];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double dG = d[0] * Gf[j] + d[1] * Gf[3 + j] + d[2] * Gf[6 + j];
            rc[j] += cf * ((DN[j] - DP[j]) - dG);
        }
        asum += a;
#pragma unroll
        for (int j = 0; j < 3; ++j) off[j] += a * DN[j];
    }
}

// ---------------------------------------------------------------------------
// k_residual: R = div(sigma) + RhieChow (integrated), r = R, and per-workgroup
// partials of sum|R|, the two normFactor sums and z.r (finResidual).
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void k_residual(const DevMesh m, const BlockMap bm, const double* __restrict__ D0,
                                                     const double* __restrict__ D1, const double* __restrict__ G, const double* __restrict__ sigb,
                                                     T* __restrict__ r, const Ctl* __restrict__ ctlAll,
                                                     double* __restrict__ part) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int inst = tl.inst;
    const Ctl* ctl = ctlAll + inst;
    if (ctl->pending != kPendRes) return;
    const double* __restrict__ D = ctl->dpar ? D1 : D0;
    const int C = m.nCells;
    const double xb0 = ctl->xbar[0], xb1 = ctl->xbar[1], xb2 = ctl->xbar[2];
    // a cold start's first residual sees the zero initial stress field (the
    // constructor computes grad(D) but no sigma, linGeomTotalDispSolid.C:64-84)
    const double sf = (ctl->sigma0 && ctl->iCorr == 0) ? 0.0 : 1.0;
    double acc[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) acc[i] = 0.0;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        const int width = m.width(s);
        const int e0 = m.entry0(s);
        if (P >= tl.cEnd) continue;
        double DP[3], GP[9], CP[3], sP[6];
#pragma unroll
        for (int k = 0; k < 3; ++k) { DP[k] = D[(size_t)k * C + P]; CP[k] = m.cC[(size_t)k * C + P]; }
#pragma unroll
        for (int k = 0; k < 9; ++k) GP[k] = G[(size_t)k * C + P];
        const double muP = cellMu(m, P) * sf, KP = cellK(m, P) * sf;
        hooke(GP, muP, KP, sP);
        double div[3] = {0, 0, 0}, rc[3] = {0, 0, 0}, off[3] = {0, 0, 0}, asum = 0.0;
        bool hasB = false;
        residualInternal(m, P, e0, width, lane, C, D, G, DP, GP, CP, sP, sf, div, rc, off, asum, hasB);
        for (int k = 0; hasB && k < width; ++k) {
            const int e = e0 + k * kSlice + lane;
            const int n = m.col[e];
            if (n < 0 && n != kPad) {
                const int b = -1 - n;
                const size_t E = m.nEntries;
                const double S0 = m.eS[e], S1 = m.eS[E + e], S2 = m.eS[2 * E + e];
                double sb[6];
#pragma unroll
                for (int q = 0; q < 6; ++q) sb[q] = sigb[(size_t)q * m.nBoundary + b];
                div[0] += S0 * sb[0] + S1 * sb[1] + S2 * sb[2];
                div[1] += S0 * sb[1] + S1 * sb[3] + S2 * sb[4];
                div[2] += S0 * sb[2] + S1 * sb[4] + S2 * sb[5];
            }
        }
        const double dg = m.diag[P];
        const double rowsum = dg - asum;
        const double xb[3] = {xb0, xb1, xb2};
        // body force and the inertia terms (rho g V + source - diag D)
        double src[3] = {0.0, 0.0, 0.0};
        if (m.fext) {
#pragma unroll
            for (int j = 0; j < 3; ++j) src[j] = m.fext[(size_t)j * C + P] - (m.iner ? m.iner[P] * DP[j] : 0.0);
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double R = (div[j] + rc[j]) + src[j];
            const double MD = dg * DP[j] - off[j];
            const double t = rowsum * xb[j];
            acc[j] += fabs(R);
            acc[3 + j] += fabs(MD - t);
            acc[6 + j] += fabs((MD + R) - t);
            const T rT = (T)R;
            stS(r + (size_t)j * C + P, rT);
            const T z = invD[P] * rT;
            acc[9 + j] += (double)z * (double)rT;
        }
    }
    storeBlockPartials<12, 0>(acc, part, kOffRes, lb, bm.nBlocks);
}

// Slots of a row whose loads are in flight together where the row's slot count
// is not compiled in.  One component of a 7-point matrix, 272,640 rows, FP64:
// 13.0 us slot by slot, 10.4 six at a time; two of three components active, FP32,
// 128^3 cells: 66 -> 51 us (and 53 -> 33 for the V-cycle's first residual).
constexpr int kRowChunk = 6;

// Row of the fused direction update + SpMV with all three components active
// and a compile-time slot count W: every load of the row is issued without a
// branch (invalid slots gather the row's own cell and contribute zero), so
// the wave keeps all of its gathers in flight at once.
template <typename T, int W, bool MG>
__device__ __forceinline__ void spmvpRowAll(const DevMesh& m, int P, int e0, int lane, int C, const T* __restrict__ r,
                                            const T* __restrict__ pOld, const T* __restrict__ zArr,
                                            T* __restrict__ pNew, T* __restrict__ q, int first, const T* be,
                                            double* acc) {
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
    auto dir = [&](int j, int c, T iDc) -> T {
        const size_t i = (size_t)j * C + c;
        const T z = MG ? zArr[i] : iDc * r[i];
        const T d = z + be[j] * pOld[i];
        return first ? z : d;
    };
    const T iDP = MG ? (T)0 : invD[P];
    T pP[3], y[3];
    const T dP = MatSel<T>::diag(m)[P];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        pP[j] = dir(j, P, iDP);
        y[j] = dP * pP[j];
    }
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const bool v = nb[k] >= 0;
        const int c = v ? nb[k] : P;
        const T av = v ? a[k] : (T)0;
        const T iDc = MG ? (T)0 : invD[c];
#pragma unroll
        for (int j = 0; j < 3; ++j) y[j] -= av * dir(j, c, iDc);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const size_t i = (size_t)j * C + P;
        stS(pNew + i, pP[j]);
        stS(q + i, y[j]);
        acc[j] += (double)pP[j] * (double)y[j];
    }
}

// ---------------------------------------------------------------------------
// k_spmvp: p = z + beta p (z = D^-1 r, or the multigrid output when MG),
// q = M p for the three components; partial p.q per component.  With
// reduce = 0 it is a plain q = M p (s4f_spmv3).
// ---------------------------------------------------------------------------
template <typename T, bool MG>
__global__ __launch_bounds__(kBlock, 5) void k_spmvp(const DevMesh m, const BlockMap bm, const T* __restrict__ r,
                                                  T* pA, T* pB, T* __restrict__ q, const Ctl* __restrict__ ctlAll,
                                                  double* __restrict__ part, int reduce,
                                                  const T* __restrict__ zArr) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int inst = tl.inst;
    const Ctl* ctl = ctlAll + inst;
    if (reduce && ctl->pending != kPendSpmv) return;
    // the two direction buffers alternate with the PCG iteration
    const bool odd = reduce && (ctl->pIt & 1);
    const T* __restrict__ pOld = odd ? pB : pA;
    T* __restrict__ pNew = odd ? pA : pB;
    const int C = m.nCells;
    const T* __restrict__ A = MatSel<T>::a(m);
    const T* __restrict__ dg = MatSel<T>::diag(m);
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const int first = reduce ? ctl->firstInner : 0;
    const bool act[3] = {reduce ? ctl->active[0] != 0 : true, reduce ? ctl->active[1] != 0 : true,
                         reduce ? ctl->active[2] != 0 : true};
    const bool all = reduce && act[0] && act[1] && act[2];
    const T be[3] = {reduce ? (T)ctl->beta[0] : (T)0, reduce ? (T)ctl->beta[1] : (T)0, reduce ? (T)ctl->beta[2] : (T)0};
    double acc[3] = {0, 0, 0};
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        const int width = m.width(s);
        const int e0 = m.entry0(s);
        if (P >= tl.cEnd) continue;
        if (all && width == 6) {
            spmvpRowAll<T, 6, MG>(m, P, e0, lane, C, r, pOld, zArr, pNew, q, first, be, acc);
            continue;
        }
        if (all && width == 4) {
            spmvpRowAll<T, 4, MG>(m, P, e0, lane, C, r, pOld, zArr, pNew, q, first, be, acc);
            continue;
        }
        // some components, or another slot count: kRowChunk slots' loads in
        // flight at a time (a slot past the row or empty reads the row's own
        // cell with a zero coefficient), the active components only
        auto dir = [&](int j, T z0, T iD, T o) -> T {
            if (!reduce) return o;
            const T z = MG ? z0 : iD * z0;
            return first ? z : z + be[j] * o;
        };
        const T* __restrict__ src = MG ? zArr : r;
        const bool diagZ = !MG && reduce;
        T pP[3] = {}, y[3] = {};
        const T d = dg[P], iDP = diagZ ? invD[P] : (T)0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if (!act[j]) continue;
            const size_t i = (size_t)j * C + P;
            pP[j] = dir(j, reduce ? src[i] : (T)0, iDP, pOld[i]);
            y[j] = rounded(d * pP[j]);
        }
        for (int k0 = 0; k0 < width; k0 += kRowChunk) {
            int c[kRowChunk];
            T av[kRowChunk], iD[kRowChunk];
#pragma unroll
            for (int u = 0; u < kRowChunk; ++u) {
                const int e = e0 + (k0 + u < width ? k0 + u : k0) * kSlice + lane;
                const int n = ldS(m.col + e);
                const T ae = ldS(A + e);
                const bool v = k0 + u < width && n >= 0;
                c[u] = v ? n : P;
                av[u] = v ? ae : (T)0;
            }
            if (diagZ) {
#pragma unroll
                for (int u = 0; u < kRowChunk; ++u) iD[u] = invD[c[u]];
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                if (!act[j]) continue;
                T z[kRowChunk], o[kRowChunk];
#pragma unroll
                for (int u = 0; u < kRowChunk; ++u) {
                    const size_t i = (size_t)j * C + c[u];
                    z[u] = reduce ? src[i] : (T)0;
                    o[u] = pOld[i];
                }
                if (!reduce) {  // a caller's vector: zero times its own infinity would be NaN
#pragma unroll
                    for (int u = 0; u < kRowChunk; ++u) o[u] = c[u] == P ? (T)0 : o[u];
                }
#pragma unroll
                for (int u = 0; u < kRowChunk; ++u) y[j] = fmaT(-av[u], dir(j, z[u], iD[u], o[u]), y[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if (!act[j]) continue;
            const size_t i = (size_t)j * C + P;
            if (reduce) pNew[i] = pP[j];
            q[i] = y[j];
            acc[j] += (double)pP[j] * (double)y[j];
        }
    }
    if (!reduce) return;
    storeBlockPartials<3, 0>(acc, part, kOffSpmv, lb, bm.nBlocks);
}

// ---------------------------------------------------------------------------
// k_update: x += alpha p, r -= alpha q, z = r/diag; partials z.r and sum|r|
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void k_update(const DevMesh m, const BlockMap bm, T* __restrict__ x,
                                                   const T* __restrict__ pA, const T* __restrict__ pB,
                                                   T* __restrict__ r, const T* __restrict__ q,
                                                   const Ctl* __restrict__ ctlAll, double* __restrict__ part) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int inst = tl.inst;
    const Ctl* ctl = ctlAll + inst;
    if (ctl->pending != kPendUpd) return;
    // the direction k_spmvp wrote
    const T* __restrict__ p = (ctl->pIt & 1) ? pA : pB;
    const int C = m.nCells;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const T al[3] = {(T)ctl->alpha[0], (T)ctl->alpha[1], (T)ctl->alpha[2]};
    const bool act[3] = {ctl->active[0] != 0, ctl->active[1] != 0, ctl->active[2] != 0};
    const int first = ctl->firstInner;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        if (P >= tl.cEnd) continue;
        const T iD = invD[P];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const size_t i = (size_t)j * C + P;
            if (!act[j]) {
                if (first) x[i] = (T)0;
                continue;
            }
            const T xv = first ? (T)0 : x[i];
            x[i] = xv + al[j] * p[i];
            const T rv = r[i] - al[j] * q[i];
            r[i] = rv;
            const T z = iD * rv;
            acc[j] += (double)z * (double)rv;
            acc[3 + j] += fabs((double)rv);
        }
    }
    storeBlockPartials<6, 0>(acc, part, kOffUpd, lb, bm.nBlocks);
}

// Internal-face slots of the least-squares gradient sum with compile-time
// slot count W, branch-free (boundary and empty slots gather the row's own
// cell with zero weight); boundary slots follow in the general loop, in slot
// order, as rows list internal faces first.
template <typename T, int W, bool HASX>
__device__ __forceinline__ void gradInternalW(const DevMesh& m, int P, int e0, int lane, int C,
                                              const double* __restrict__ D, const T* __restrict__ x,
                                              double ra, const double* DnP, const double* CP, double* A,
                                              bool& hasB) {
    // every column first, then two faces' gathers in flight at a time (128^3
    // cells: 175 us with a column's and its gathers' latency per face, 163 now;
    // 94 for each array moved once)
    const int* __restrict__ col = m.col + e0;
    int nb[W];
#pragma unroll
    for (int k = 0; k < W; ++k) nb[k] = at32s(col + k * kSlice, lane * 4u);
#pragma unroll
    for (int k0 = 0; k0 < W; k0 += 2) {
        double cN[2][3], dN[2][3], xN[2][3];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int c = nb[k0 + u] >= 0 ? nb[k0 + u] : P;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                cN[u][q] = at32(m.cC + (size_t)q * C, c * 8u);
                dN[u][q] = at32(D + (size_t)q * C, c * 8u);
                xN[u][q] = HASX ? (double)at32(x + (size_t)q * C, c * (unsigned)sizeof(T)) : 0.0;
            }
        }
        loadedHere(cN, dN, xN, A);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const bool v = nb[k0 + u] >= 0;
            hasB |= !v && nb[k0 + u] != kPad;
            double d[3], dv[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                d[q] = cN[u][q] - CP[q];
                dv[q] = (HASX ? fmaT(ra, xN[u][q], dN[u][q]) : dN[u][q]) - DnP[q];
            }
            const double rr = v ? 1.0 / dot3(d[0], d[0], d[1], d[1], d[2], d[2]) : 0.0;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double di = rounded(d[i] * rr);
#pragma unroll
                for (int j = 0; j < 3; ++j) A[3 * i + j] = fmaT(di, dv[j], A[3 * i + j]);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// The gradient step of an outer iteration, in three launches:
//   k_grad_bnd_pre   boundary faces: D' = D + x at the face cell, boundary
//                    values D_b (solidTraction evaluate / fixedDisplacement /
//                    solidSymmetry) and the snGrad used by the residual
//   k_grad           cells: least-squares grad(D') with the boundary values,
//                    D' stored, partials of the outer convergence test
//   k_grad_bnd_post  boundary faces: boundary gradient and stress, the next
//                    traction snGrad
// mode 0: outer iteration; mode 1: initialisation (x = 0, G_old = 0, g = 0,
// no convergence test); mode 2: gradient from given D_b/snb (no boundary
// update: k_grad_bnd_pre is not launched, k_grad_bnd_post leaves g).
// The face kernels run one workgroup row (blockIdx.y) per instance over that
// instance's boundary faces; empty faces carry no value and are skipped.
// Merged launch sequences run the three as one kernel (k_grad_m).
// ---------------------------------------------------------------------------
// boundary fields of the fused gradient step
struct BndBufs {
    double *g, *snb, *Gb, *sigb;
};

__device__ __forceinline__ int faceInst(const BlockMap& bm) {
    return bm.finInst ? bm.finInst[blockIdx.y] : (int)blockIdx.y;
}

// Aitken factor update of relaxField (solidModel.C:876-892) at one cell or
// boundary face: r = D_prev - D*, alpha = a0 on the first outer iteration,
// else clip(alpha (r_prev . (r_prev - r)) / (|r_prev - r|^2 + SMALL), 0, 2);
// returns alpha and stores it with r (the next r_prev)
__device__ __forceinline__ double aitkenFactor(const double* r, double* alpha, double* res, size_t i, size_t n,
                                               bool first, double a0) {
    double al = a0;
    if (!first) {
        const double rp[3] = {res[i], res[n + i], res[2 * n + i]};
        const double d[3] = {rp[0] - r[0], rp[1] - r[1], rp[2] - r[2]};
        al = alpha[i] * (rp[0] * d[0] + rp[1] * d[1] + rp[2] * d[2]) / ((d[0] * d[0] + d[1] * d[1] + d[2] * d[2]) + kSmall);
        al = al > 2.0 ? 2.0 : (al < 0.0 ? 0.0 : al);
    }
    alpha[i] = al;
    res[i] = r[0];
    res[n + i] = r[1];
    res[2 * n + i] = r[2];
    return al;
}

// relaxField, Aitken (solidModel.C:842-897), on the cells: D' = D* - alpha
// (D_prev - D*) with D* = D + x the solved field, into the buffer receiving D'
template <typename T>
__global__ __launch_bounds__(kBlock) void k_aitken(const DevMesh m, const BlockMap bm, double* __restrict__ D0,
                                                   const T* __restrict__ x, double* __restrict__ D1,
                                                   double* __restrict__ alpha, double* __restrict__ res,
                                                   const Ctl* __restrict__ ctlAll) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int inst = tl.inst;
    const Ctl* ctl = ctlAll + inst;
    if (ctl->pending != kPendGrad) return;
    if (ctl->firstInner) x = nullptr;
    const double* D = ctl->dpar ? D1 : D0;
    double* Dn = ctl->dpar ? D0 : D1;
    const bool first = ctl->iCorr == 0;
    const double a0 = ctl->relaxD;
    const int C = m.nCells;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        if (P >= tl.cEnd) continue;
        double Ds[3], r[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double DP = D[(size_t)k * C + P];
            Ds[k] = DP + (x ? (double)x[(size_t)k * C + P] : 0.0);
            r[k] = DP - Ds[k];
        }
        const double al = aitkenFactor(r, alpha, res, P, C, first, a0);
#pragma unroll
        for (int k = 0; k < 3; ++k) Dn[(size_t)k * C + P] = Ds[k] - al * r[k];
    }
}

// Settings of an instance's boundary update, the same for all of its faces.
struct BndStep {
    int mode;
    bool aitken, relax, first;
    double ra, a0;
};
__device__ __forceinline__ BndStep bndStep(const Ctl* ctl, int mode) {
    BndStep u;
    u.mode = mode;
    u.aitken = mode == 0 && ctl->relaxAitken;
    u.relax = mode == 0 && !u.aitken && ctl->relaxD != 1.0;
    u.ra = u.relax ? ctl->relaxD : 1.0;
    u.first = ctl->iCorr == 0;
    u.a0 = ctl->relaxD;
    return u;
}

// What a boundary face's update reads, loaded at once whatever the face's type
// uses of it: loads behind the type's branches cost a latency each (one face
// per thread took 2.3 us before and 2.1 us after the gradient, of 16).
struct FaceIn {
    int type;
    double n[3], kv[3], dl, val[3], g[3], Db[3];
    __device__ __forceinline__ void fixed(const DevMesh& m, int b) {
        const size_t B = m.nBoundary;
        type = at32(m.bType, b * 4u);
        dl = at32(m.bDelta, b * 8u);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            n[q] = at32(m.bN + q * B, b * 8u);
            kv[q] = at32(m.bKv + q * B, b * 8u);
            val[q] = at32(m.bVal + q * B, b * 8u);
        }
    }
    __device__ __forceinline__ void fields(const DevMesh& m, int b, const double* gArr, const double* DbArr) {
        const size_t B = m.nBoundary;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            g[q] = at32(gArr + q * B, b * 8u);
            Db[q] = at32(DbArr + q * B, b * 8u);
        }
    }
};

// Boundary value Dbv and snGrad sn of face b (type != empty) of a cell with
// updated displacement DuP (the solve's D + x), relaxed displacement DnP and
// previous gradient Gold
__device__ __forceinline__ void bndPreFace(const DevMesh& m, const BndStep& u, int b, const FaceIn& f,
                                           const double* DuP, const double* DnP, const double* Gold, double* alphaB,
                                           double* resB, double* Dbv, double* sn) {
    const int mode = u.mode, B = m.nBoundary, type = f.type;
    const bool aitken = u.aitken, relax = u.relax, first = u.first;
    const double ra = u.ra;
    const double k0 = f.kv[0], k1 = f.kv[1], k2 = f.kv[2];
    const double dl = f.dl;
    const bool trac = type == 1;
    const bool sym = type == 3;
    const bool zs = type == 4;
    // solidSymmetry (first order, normal patch delta so no k correction):
    // value D_P - n (n.D_P) after the solve (relaxed like every boundary
    // value), snGrad -n (n.D_P) deltaCoeffs from the relaxed cell value
    const double nb0 = f.n[0], nb1 = f.n[1], nb2 = f.n[2];
    const double nDu = nb0 * DuP[0] + nb1 * DuP[1] + nb2 * DuP[2];
    const double nDn = nb0 * DnP[0] + nb1 * DnP[1] + nb2 * DnP[2];
    const double nbv[3] = {nb0, nb1, nb2};
    double kGv[3], gvv[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        kGv[j] = k0 * Gold[j] + k1 * Gold[3 + j] + k2 * Gold[6 + j];
        gvv[j] = (mode == 1 || !(trac || zs)) ? 0.0 : f.g[j];
    }
    // fixedDisplacementZeroShear (direction-mixed, valueFraction nn, first
    // order): n (n.Dbar) + (I - nn).(D_P + k.G_P + g/deltaCoeffs), the value
    // from the solved cell value, the snGrad from the relaxed one
    double zu[3] = {0, 0, 0}, zn[3] = {0, 0, 0};
    if (zs) {
        double gu[3], gn[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            gu[j] = DuP[j] + kGv[j] + gvv[j] / dl;
            gn[j] = DnP[j] + kGv[j] + gvv[j] / dl;
        }
        const double nD = nb0 * f.val[0] + nb1 * f.val[1] + nb2 * f.val[2];
        const double ngu = nb0 * gu[0] + nb1 * gu[1] + nb2 * gu[2];
        const double ngn = nb0 * gn[0] + nb1 * gn[1] + nb2 * gn[2];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            zu[j] = nbv[j] * nD + (gu[j] - nbv[j] * ngu);
            zn[j] = nbv[j] * nD + (gn[j] - nbv[j] * ngn);
        }
    }
    // correctBoundaryConditions after the solve, then relaxField on the
    // patch values (fixed values stay); the snGrads follow the relaxed cell
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const double kG = kGv[j];
        if (zs) {
            Dbv[j] = zu[j];
            sn[j] = (zn[j] - (DnP[j] + kG)) * dl;
        } else if (sym) {
            Dbv[j] = DuP[j] - nbv[j] * nDu;
            sn[j] = -nbv[j] * nDn * dl;
        } else if (trac) {
            Dbv[j] = DuP[j] + kG + gvv[j] / dl;
            sn[j] = gvv[j];
        } else {
            Dbv[j] = f.val[j];
            sn[j] = (Dbv[j] - (DnP[j] + kG)) * dl;
        }
    }
    if (type != 0 && (relax || aitken)) {
        const double Dbp[3] = {f.Db[0], f.Db[1], f.Db[2]};
        if (aitken) {
            const double r[3] = {Dbp[0] - Dbv[0], Dbp[1] - Dbv[1], Dbp[2] - Dbv[2]};
            const double al = aitkenFactor(r, alphaB, resB, b, B, first, u.a0);
#pragma unroll
            for (int j = 0; j < 3; ++j) Dbv[j] -= al * r[j];
        } else {
#pragma unroll
            for (int j = 0; j < 3; ++j) Dbv[j] = Dbp[j] + ra * (Dbv[j] - Dbp[j]);
        }
    }
}

// Boundary gradient and stress of face b from the cell gradient Gn and the
// face's snGrad, and the next traction snGrad
__device__ __forceinline__ void bndPostFace(const DevMesh& m, int mode, bool zeroStress, int b, int type, int P,
                                            const double* Gn, const double* nv, const double* val, const double* snv,
                                            double* __restrict__ Gb, double* __restrict__ sigb,
                                            double* __restrict__ g) {
    const int B = m.nBoundary;
    const double pres = at32(m.bPres, b * 8u);
    double Gbv[9], sb[6];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const double nG = nv[0] * Gn[j] + nv[1] * Gn[3 + j] + nv[2] * Gn[6 + j];
        const double sn = snv[j];
#pragma unroll
        for (int i = 0; i < 3; ++i) Gbv[3 * i + j] = Gn[3 * i + j] + nv[i] * (sn - nG);
    }
    hooke(Gbv, cellMu(m, P), cellK(m, P), sb);
    if (zeroStress) {  // cold start: the stress field is still zero
#pragma unroll
        for (int q = 0; q < 6; ++q) sb[q] = 0.0;
    }
    if (Gb) {
#pragma unroll
        for (int q = 0; q < 9; ++q) Gb[(size_t)q * B + b] = Gbv[q];
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) sigb[(size_t)q * B + b] = sb[q];
    if (mode != 2 && (type == 1 || type == 4)) {
        // fixedDisplacementZeroShear: the traction snGrad for zero
        // traction and pressure (its shear-free refGrad)
        const bool zs = type == 4;
        const double ik = cellImpK(m, P);
        const double Tt[9] = {sb[0] - ik * Gbv[0], sb[1] - ik * Gbv[1], sb[2] - ik * Gbv[2],
                              sb[1] - ik * Gbv[3], sb[3] - ik * Gbv[4], sb[4] - ik * Gbv[5],
                              sb[2] - ik * Gbv[6], sb[4] - ik * Gbv[7], sb[5] - ik * Gbv[8]};
        const double rik = 1.0 / ik;
        const double pr = zs ? 0.0 : pres;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double nT = nv[0] * Tt[j] + nv[1] * Tt[3 + j] + nv[2] * Tt[6 + j];
            g[(size_t)j * B + b] = (zs ? -nT : (val[j] - nv[j] * pr) - nT) * rik;
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_grad_bnd_pre(const DevMesh m, const BlockMap bm,
                                                         const double* __restrict__ D0, const T* __restrict__ x,
                                                         const double* __restrict__ D1, const double* __restrict__ G,
                                                         double* __restrict__ Db, const double* __restrict__ g,
                                                         double* __restrict__ snb, const Ctl* __restrict__ ctlAll,
                                                         double* __restrict__ alphaB, double* __restrict__ resB,
                                                         int mode) {
    const int inst = faceInst(bm);
    const Ctl* ctl = ctlAll + inst;
    if (mode == 0 && ctl->pending != kPendGrad) return;
    if (mode == 0 && ctl->firstInner) x = nullptr;  // no PCG iteration ran: the update is zero
    const double* __restrict__ D = ctl->dpar ? D1 : D0;
    // Aitken: the relaxed cell values are in the buffer receiving D' (k_aitken)
    const BndStep u = bndStep(ctl, mode);
    const double* __restrict__ Dr = ctl->dpar ? D0 : D1;
    const int C = m.nCells, B = m.nBoundary;
    const int b0 = bm.iB0[inst], b1 = b0 + bm.iNB[inst];
    for (int b = b0 + blockIdx.x * kBlock + threadIdx.x; b < b1; b += gridDim.x * kBlock) {
        FaceIn f;
        f.fixed(m, b);
        f.fields(m, b, g, Db);
        const int P = m.bCell[b];
        if (f.type == 2) continue;
        // DuP: the solve's update D + x; DnP: after the fixed field
        // under-relaxation D_prev + a (DuP - D_prev) (a = 1: the same)
        double DuP[3], DnP[3], Gold[9];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double DP = D[(size_t)k * C + P];
            const double xv = x ? (double)x[(size_t)k * C + P] : 0.0;
            DuP[k] = DP + xv;
            DnP[k] = u.aitken ? Dr[(size_t)k * C + P] : DP + u.ra * xv;
        }
#pragma unroll
        for (int q = 0; q < 9; ++q) Gold[q] = (mode == 1) ? 0.0 : G[(size_t)q * C + P];
        double Dbv[3], sn[3];
        bndPreFace(m, u, b, f, DuP, DnP, Gold, alphaB, resB, Dbv, sn);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            Db[(size_t)j * B + b] = Dbv[j];
            snb[(size_t)j * B + b] = sn[j];
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_grad(const DevMesh m, const BlockMap bm, double* __restrict__ D0,
                                                 const T* __restrict__ x, double* __restrict__ D1,
                                                 double* __restrict__ G, const double* __restrict__ Db,
                                                 const double* __restrict__ DI, const double* __restrict__ Dold,
                                                 const Ctl* __restrict__ ctlAll, double* __restrict__ part, int mode) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int inst = tl.inst;
    const Ctl* ctl = ctlAll + inst;
    if (mode == 0 && ctl->pending != kPendGrad) return;
    if (mode == 0 && ctl->firstInner) x = nullptr;  // no PCG iteration ran: the update is zero
    // current field and the buffer receiving D' (per-instance ping-pong)
    const double* __restrict__ D = ctl->dpar ? D1 : D0;
    double* Dn = (mode == 0) ? (ctl->dpar ? D0 : D1) : nullptr;
    // D' = D + a x (fixed relaxation, a = 1 without), or the Aitken-relaxed
    // field k_aitken already stored in Dn
    const bool aitken = mode == 0 && ctl->relaxAitken;
    const bool relax = mode == 0 && !aitken && ctl->relaxD != 1.0;
    const double ra = relax ? ctl->relaxD : 1.0;  // x scaled by exactly 1.0 without relaxation
    const double* Dg = aitken ? Dn : D;
    const T* xg = aitken ? nullptr : x;
    const int C = m.nCells, B = m.nBoundary;
    double acc[6] = {0, 0, 0, 0, 0, 0};  // max|D'-D|^2, max|D'-Dold|^2, max|D'|^2, sum D'
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        const int width = m.width(s);
        const int e0 = m.entry0(s);
        if (P >= tl.cEnd) continue;
        double DP[3], DnP[3], CP[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            DP[k] = D[(size_t)k * C + P];
            const double xv = xg ? (double)xg[(size_t)k * C + P] : 0.0;
            DnP[k] = aitken ? Dg[(size_t)k * C + P] : DP[k] + ra * xv;
            CP[k] = m.cC[(size_t)k * C + P];
        }
        double A[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) A[q] = 0.0;
        bool hasB = false;
        int kInt = width;  // internal slots left to the general loop below
        // a slice holding bi-material interface faces: every slot goes
        // through the general loop, which gives each side's sub-mesh the
        // interface displacement as a boundary value
        const bool ifs = m.sliceIf && m.sliceIf[s];
        if (ifs) {
            hasB = true;
        } else if (width == 6) {
            if (xg) gradInternalW<T, 6, true>(m, P, e0, lane, C, Dg, xg, ra, DnP, CP, A, hasB);
            else gradInternalW<T, 6, false>(m, P, e0, lane, C, Dg, xg, ra, DnP, CP, A, hasB);
            kInt = 0;
        } else if (width == 4) {
            if (xg) gradInternalW<T, 4, true>(m, P, e0, lane, C, Dg, xg, ra, DnP, CP, A, hasB);
            else gradInternalW<T, 4, false>(m, P, e0, lane, C, Dg, xg, ra, DnP, CP, A, hasB);
            kInt = 0;
        } else {
            hasB = true;
        }
        for (int k = 0; hasB && k < width; ++k) {
            const int e = e0 + k * kSlice + lane;
            const int n = m.col[e];
            if (n >= 0) {
                if (k >= kInt) continue;  // already summed by the fixed-width pass
                if (ifs && m.eIf[e] >= 0) {
                    const int si = m.eIf[e], nI2 = 2 * m.nIf;
                    const double lv[3] = {m.ifLs[si], m.ifLs[(size_t)nI2 + si], m.ifLs[2 * (size_t)nI2 + si]};
                    double dv[3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) dv[q] = DI[(size_t)q * m.nIf + (si >> 1)] - DnP[q];
#pragma unroll
                    for (int i = 0; i < 3; ++i)
#pragma unroll
                        for (int j = 0; j < 3; ++j) A[3 * i + j] += lv[i] * dv[j];
                    continue;
                }
                double d[3], dv[3];
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    d[q] = m.cC[(size_t)q * C + n] - CP[q];
                    const double DN =
                        xg ? Dg[(size_t)q * C + n] + ra * (double)xg[(size_t)q * C + n] : Dg[(size_t)q * C + n];
                    dv[q] = DN - DnP[q];
                }
                const double rr = 1.0 / (d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const double di = d[i] * rr;
#pragma unroll
                    for (int j = 0; j < 3; ++j) A[3 * i + j] += di * dv[j];
                }
            } else if (n != kPad) {
                const int b = -1 - n;
                const double lv[3] = {m.bLs[b], m.bLs[(size_t)B + b], m.bLs[2 * (size_t)B + b]};
                double Dbv[3];
#pragma unroll
                for (int q = 0; q < 3; ++q) Dbv[q] = Db[(size_t)q * B + b];
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) A[3 * i + j] += lv[i] * (Dbv[j] - DnP[j]);
            }
        }
        const double M0 = m.minv[P], M1 = m.minv[(size_t)C + P], M2 = m.minv[2 * (size_t)C + P];
        const double M3 = m.minv[3 * (size_t)C + P], M4 = m.minv[4 * (size_t)C + P], M5 = m.minv[5 * (size_t)C + P];
        double Gn[9];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            Gn[j] = M0 * A[j] + M1 * A[3 + j] + M2 * A[6 + j];
            Gn[3 + j] = M1 * A[j] + M3 * A[3 + j] + M4 * A[6 + j];
            Gn[6 + j] = M2 * A[j] + M4 * A[3 + j] + M5 * A[6 + j];
        }
#pragma unroll
        for (int q = 0; q < 9; ++q) stS(G + (size_t)q * C + P, Gn[q]);
        if (Dn && !aitken) {
#pragma unroll
            for (int q = 0; q < 3; ++q) stS(Dn + (size_t)q * C + P, DnP[q]);
        }
        if (mode != 2) {
            double dx2 = 0.0, dold2 = 0.0, dn2 = 0.0;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const double a = DnP[q] - DP[q];
                const double o = Dold ? DnP[q] - Dold[(size_t)q * C + P] : DnP[q];
                dx2 += a * a;
                dold2 += o * o;
                dn2 += DnP[q] * DnP[q];
                acc[3 + q] += DnP[q];
            }
            acc[0] = nanMax(acc[0], dx2);
            acc[1] = nanMax(acc[1], dold2);
            acc[2] = nanMax(acc[2], dn2);
        }
    }
    if (mode == 2) return;
    storeBlockPartials<6, 3>(acc, part, kOffGrad, lb, bm.nBlocks);
}

// ---------------------------------------------------------------------------
// Sub-meshes of a multi-law case (one law per cellZone): the internal faces
// between zones are boundary faces of the sub-mesh on either side, holding
// an interface displacement D_I that is iterated to traction balance.
// k_iface_pre  solidSubMeshes::interpolateDtoSubMeshD (solidSubMeshes.C:
//              1550-1950), side a the owner, b the neighbour, n from a to b:
//                D_I += wab n.(sigma_b - sigma_a) + wa (D_a - Dprev_a) + wb (D_b - Dprev_b)
//              da = 1/deltaCoeffs_a, db = 1/deltaCoeffs_b, K = impK,
//              wab = da db/(db Ka + da Kb), wa = db Ka/(db Ka + da Kb), wb = 1 - wa;
//              sigma_a, sigma_b the sub-meshes' boundary stresses from the
//              previous correct().  Seen from sub-mesh b the normal, weights
//              and sides swap and the update is the same, so one D_I serves
//              both.  Modes 0/1 as k_grad (D = the current field, the new one
//              D + a x or the Aitken-relaxed one); mode 3: after the loop
//              (mechanicalModel::interpolate, mechanicalModel.C:851-852),
//              D the final field and Dprev the one its last iteration began
//              from.
// k_iface_post the sub-meshes' boundary gradient at the face,
//              G_P + n_s ((D_I - D_P) deltaCoeffs - n_s.G_P) (fvc::grad's
//              boundary value corrected by solidSubMeshes::
//              correctBoundarySnGrad, solidSubMeshes.C:1952-2031, whose k
//              vanishes for the normal patch delta), n_s = +n on side a, -n
//              on side b, and the side's Hooke's law (mechanicalModel.C:
//              477-498).  A cold start's first stress is zero, like the
//              cell stress.
// One instance (sub-meshes are solved alone).
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void k_iface_pre(const DevMesh m, const double* __restrict__ D0,
                                                      const T* __restrict__ x, const double* __restrict__ D1,
                                                      double* __restrict__ DI, const double* __restrict__ sigI,
                                                      const Ctl* __restrict__ ctl, int mode) {
    if (mode == 0 && ctl->pending != kPendGrad) return;
    if (mode != 0 || ctl->firstInner) x = nullptr;
    const bool post = mode == 3;
    const double* __restrict__ Dcur = ctl->dpar ? D1 : D0;
    const double* __restrict__ Doth = ctl->dpar ? D0 : D1;
    // the old field and the new one: (D, D + a x or the Aitken-relaxed one),
    // after the loop (Dprev, D)
    const bool aitken = mode == 0 && ctl->relaxAitken;
    const double ra = (mode == 0 && !aitken && ctl->relaxD != 1.0) ? ctl->relaxD : 1.0;
    const double* __restrict__ Dp = post ? Doth : Dcur;
    const int C = m.nCells, nI = m.nIf, nI2 = 2 * m.nIf;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < nI; i += gridDim.x * kBlock) {
        const int a = m.ifCell[2 * i], b = m.ifCell[2 * i + 1];
        const double n[3] = {m.ifN[i], m.ifN[(size_t)nI + i], m.ifN[2 * (size_t)nI + i]};
        const double da = 1.0 / m.ifDc[2 * i], db = 1.0 / m.ifDc[2 * i + 1];
        const double Ka = cellImpK(m, a), Kb = cellImpK(m, b);
        const double wab = da * db / (db * Ka + da * Kb);
        const double wa = db * Ka / (db * Ka + da * Kb), wb = 1.0 - wa;
        double sa[6], sb[6];
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            sa[q] = sigI[(size_t)q * nI2 + 2 * i];
            sb[q] = sigI[(size_t)q * nI2 + 2 * i + 1];
        }
        const double ta[3] = {sa[0] * n[0] + sa[1] * n[1] + sa[2] * n[2], sa[1] * n[0] + sa[3] * n[1] + sa[4] * n[2],
                              sa[2] * n[0] + sa[4] * n[1] + sa[5] * n[2]};
        const double tb[3] = {sb[0] * n[0] + sb[1] * n[1] + sb[2] * n[2], sb[1] * n[0] + sb[3] * n[1] + sb[4] * n[2],
                              sb[2] * n[0] + sb[4] * n[1] + sb[5] * n[2]};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const double pa = Dp[(size_t)q * C + a], pb = Dp[(size_t)q * C + b];
            double na, nb;
            if (post) {
                na = Dcur[(size_t)q * C + a];
                nb = Dcur[(size_t)q * C + b];
            } else if (aitken) {
                na = Doth[(size_t)q * C + a];
                nb = Doth[(size_t)q * C + b];
            } else {
                na = pa + (x ? ra * (double)x[(size_t)q * C + a] : 0.0);
                nb = pb + (x ? ra * (double)x[(size_t)q * C + b] : 0.0);
            }
            DI[(size_t)q * nI + i] += wab * (tb[q] - ta[q]) + wa * (na - pa) + wb * (nb - pb);
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_iface_post(const DevMesh m, const double* __restrict__ D0,
                                                       const double* __restrict__ D1, const double* __restrict__ G,
                                                       const double* __restrict__ DI, double* __restrict__ sigI,
                                                       const Ctl* __restrict__ ctl, int mode) {
    if (mode == 0 && ctl->pending != kPendGrad) return;
    // the gradient's cell values: k_grad left D' in the buffer the flip at
    // the end of the step makes current (mode 0), else the current field
    const double* __restrict__ D = (mode == 0) == (ctl->dpar != 0) ? D0 : D1;
    const bool zero = mode == 1 && ctl->sigma0;
    const int C = m.nCells, nI = m.nIf, nI2 = 2 * m.nIf;
    for (int k = blockIdx.x * kBlock + threadIdx.x; k < nI2; k += gridDim.x * kBlock) {
        const int i = k >> 1, side = k & 1;
        const int P = m.ifCell[k];
        const double sg = side ? -1.0 : 1.0;
        const double n[3] = {sg * m.ifN[i], sg * m.ifN[(size_t)nI + i], sg * m.ifN[2 * (size_t)nI + i]};
        double GI[9], sI[6];
        if (zero) {
#pragma unroll
            for (int q = 0; q < 6; ++q) sI[q] = 0.0;
        } else {
            double GP[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) GP[q] = G[(size_t)q * C + P];
            const double dc = m.ifDc[k];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const double nG = n[0] * GP[j] + n[1] * GP[3 + j] + n[2] * GP[6 + j];
                const double sn = (DI[(size_t)j * nI + i] - D[(size_t)j * C + P]) * dc;
#pragma unroll
                for (int r = 0; r < 3; ++r) GI[3 * r + j] = GP[3 * r + j] + n[r] * (sn - nG);
            }
            hooke(GI, cellMu(m, P), cellK(m, P), sI);
        }
#pragma unroll
        for (int q = 0; q < 6; ++q) sigI[(size_t)q * nI2 + k] = sI[q];
    }
}

__global__ __launch_bounds__(kBlock) void k_grad_bnd_post(const DevMesh m, const BlockMap bm,
                                                          const double* __restrict__ G,
                                                          const double* __restrict__ snb, double* __restrict__ Gb,
                                                          double* __restrict__ sigb, double* __restrict__ g,
                                                          const Ctl* __restrict__ ctlAll, int mode) {
    const int inst = faceInst(bm);
    const Ctl* ctl = ctlAll + inst;
    if (mode == 0 && ctl->pending != kPendGrad) return;
    const int C = m.nCells;
    const int b0 = bm.iB0[inst], b1 = b0 + bm.iNB[inst];
    for (int b = b0 + blockIdx.x * kBlock + threadIdx.x; b < b1; b += gridDim.x * kBlock) {
        const int type = m.bType[b];
        const int P = m.bCell[b];
        const size_t B = m.nBoundary;
        double Gn[9], nv[3], val[3], sn[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            nv[q] = at32(m.bN + q * B, b * 8u);
            val[q] = at32(m.bVal + q * B, b * 8u);
            sn[q] = at32(snb + q * B, b * 8u);
        }
        if (type == 2) continue;
#pragma unroll
        for (int q = 0; q < 9; ++q) Gn[q] = G[(size_t)q * C + P];
        bndPostFace(m, mode, mode == 1 && ctl->sigma0, b, type, P, Gn, nv, val, sn, Gb, sigb, g);
    }
}

// sigma = Hooke(G) for output (xx xy xz yy yz zz, SoA)
__global__ __launch_bounds__(kBlock) void k_sigma(const DevMesh m, const double* __restrict__ G,
                                                  double* __restrict__ sig, int c0, int n) {
    const int C = m.nCells;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const int P = c0 + i;
        double GP[9], s[6];
#pragma unroll
        for (int q = 0; q < 9; ++q) GP[q] = G[(size_t)q * C + P];
        hooke(GP, cellMu(m, P), cellK(m, P), s);
#pragma unroll
        for (int q = 0; q < 6; ++q) sig[(size_t)q * C + P] = s[q];
    }
}

// solidModel::writeFields (solidModel.C:1936-1962): epsilon = symm(gradD)
// (xx xy xz yy yz zz, SoA), epsilonEq = sqrt(2/3 |dev epsilon|^2),
// sigmaEq = sqrt(3/2 |dev sigma|^2) with sigma from Hooke's law
__global__ __launch_bounds__(kBlock) void k_strain_fields(const DevMesh m, const double* __restrict__ G,
                                                          double* __restrict__ eps, double* __restrict__ epsEq,
                                                          double* __restrict__ sigEq) {
    const int C = m.nCells;
    for (int P = blockIdx.x * kBlock + threadIdx.x; P < C; P += gridDim.x * kBlock) {
        double GP[9], s[6];
#pragma unroll
        for (int q = 0; q < 9; ++q) GP[q] = G[(size_t)q * C + P];
        const double e[6] = {GP[0], 0.5 * (GP[1] + GP[3]), 0.5 * (GP[2] + GP[6]), GP[4], 0.5 * (GP[5] + GP[7]), GP[8]};
        if (eps) {
#pragma unroll
            for (int q = 0; q < 6; ++q) eps[(size_t)q * C + P] = e[q];
        }
        // |dev t|^2 of a symmetric tensor (xx xy xz yy yz zz)
        auto magDev2 = [](const double* t) {
            const double tr3 = (t[0] + t[3] + t[5]) / 3.0;
            const double a = t[0] - tr3, b = t[3] - tr3, c = t[5] - tr3;
            return a * a + b * b + c * c + 2.0 * (t[1] * t[1] + t[2] * t[2] + t[4] * t[4]);
        };
        if (epsEq) epsEq[P] = sqrt((2.0 / 3.0) * magDev2(e));
        if (sigEq) {
            hooke(GP, cellMu(m, P), cellK(m, P), s);
            sigEq[P] = sqrt(1.5 * magDev2(s));
        }
    }
}

// mechanicalModel::interpolate -> enhancedVolPointInterpolation with the
// gradient (mechanicalModel.C:829-845, enhancedVolPointInterpolate.C:350-420):
// point value = sum_c w (D_c + (x_p - C_c).gradD_c) / sum_c w over the
// point's cells (ascending cell order), w = 1/|x_p - C_c|
__global__ __launch_bounds__(kBlock) void k_point_interpolate(const DevMesh m, const double* __restrict__ D,
                                                              const double* __restrict__ G, int nPoints,
                                                              const double* __restrict__ pts,
                                                              const int* __restrict__ pcOff,
                                                              const int* __restrict__ pcCell,
                                                              double* __restrict__ pD) {
    const int C = m.nCells;
    for (int p = blockIdx.x * kBlock + threadIdx.x; p < nPoints; p += gridDim.x * kBlock) {
        const double x[3] = {pts[3 * (size_t)p], pts[3 * (size_t)p + 1], pts[3 * (size_t)p + 2]};
        const int k0 = pcOff[p], k1 = pcOff[p + 1];
        // material zones: each sub-mesh interpolates from its own cells and
        // the point takes the mean over the materials around it
        // (mapSubMeshPointFields, solidSubMeshesTemplates.C:271-336), the
        // materials in the order of their first cell in the list
        int nz = 1;
        if (m.zone) {
            nz = 0;
            for (int k = k0; k < k1; ++k) {
                bool first = true;
                for (int k2 = k0; k2 < k; ++k2) first &= m.zone[pcCell[k2]] != m.zone[pcCell[k]];
                nz += first ? 1 : 0;
            }
        }
        double res[3] = {0, 0, 0};
        for (int kz = k0; kz < (m.zone ? k1 : k0 + 1); ++kz) {
            if (m.zone) {
                bool first = true;
                for (int k2 = k0; k2 < kz; ++k2) first &= m.zone[pcCell[k2]] != m.zone[pcCell[kz]];
                if (!first) continue;
            }
            const int z = (m.zone && kz < k1) ? m.zone[pcCell[kz]] : 0;
            double acc[3] = {0, 0, 0}, sw = 0.0;
            for (int k = k0; k < k1; ++k) {
                const int c = pcCell[k];
                if (m.zone && m.zone[c] != z) continue;
                double d[3];
#pragma unroll
                for (int q = 0; q < 3; ++q) d[q] = x[q] - m.cC[(size_t)q * C + c];
                const double w = 1.0 / sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const double dG = d[0] * G[(size_t)j * C + c] + d[1] * G[(size_t)(3 + j) * C + c] +
                                      d[2] * G[(size_t)(6 + j) * C + c];
                    acc[j] += w * (D[(size_t)j * C + c] + dG);
                }
                sw += w;
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const double v = sw > 1e-300 ? acc[j] / sw : acc[j];
                res[j] = nz == 1 ? v : res[j] + v / nz;
            }
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) pD[3 * (size_t)p + j] = res[j];
    }
}

// von Mises equivalent stress sqrt(3/2 |dev sigma|^2) (solidModel.C:1957-1961)
__global__ __launch_bounds__(kBlock) void k_sigma_eq(const double* __restrict__ sig, double* __restrict__ eq, int n) {
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const double xx = sig[i], xy = sig[(size_t)n + i], xz = sig[2 * (size_t)n + i];
        const double yy = sig[3 * (size_t)n + i], yz = sig[4 * (size_t)n + i], zz = sig[5 * (size_t)n + i];
        const double t3 = (xx + yy + zz) / 3.0;
        const double a = xx - t3, b = yy - t3, c = zz - t3;
        eq[i] = sqrt(1.5 * (a * a + b * b + c * c + 2.0 * (xy * xy + xz * xz + yz * yz)));
    }
}

// serving: (re)initialise one instance's state ranges; cold start zeroes the
// displacement, warm start keeps the resident field of buffer `dpar` and makes
// it the old-time field
__global__ __launch_bounds__(kBlock) void k_slot_init(double* __restrict__ D0, double* __restrict__ D1,
                                                      double* __restrict__ Dold, double* __restrict__ G,
                                                      double* __restrict__ g, int C, int B, int c0, int n, int b0,
                                                      int nb, int warm, int dpar) {
    double* D = dpar ? D1 : D0;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const int P = c0 + i;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const size_t k = (size_t)q * C + P;
            if (!warm) D[k] = 0.0;
            Dold[k] = D[k];
        }
#pragma unroll
        for (int q = 0; q < 9; ++q) G[(size_t)q * C + P] = 0.0;
    }
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < nb; i += gridDim.x * kBlock)
#pragma unroll
        for (int q = 0; q < 3; ++q) g[(size_t)q * B + b0 + i] = 0.0;
}

// PCG start from a given right-hand side b (for the standalone PCG entry):
// r = b, p = z = b/diag; normalised initial residual with the supplied normFactor
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pcg_start(const DevMesh m, const BlockMap bm, const double* __restrict__ b,
                                                      T* __restrict__ r, T* __restrict__ p, Ctl* __restrict__ ctlAll,
                                                      double* __restrict__ part) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int C = m.nCells;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    double acc[6] = {0, 0, 0, 0, 0, 0};
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        if (P >= tl.cEnd) continue;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const size_t i = (size_t)j * C + P;
            const T rT = (T)b[i];
            r[i] = rT;
            const T z = invD[P] * rT;
            p[i] = z;
            acc[j] += fabs(b[i]);
            acc[3 + j] += (double)z * (double)rT;
        }
    }
    storeBlockPartials<6, 0>(acc, part, kOffRho, lb, bm.nBlocks);
}

// lduMatrix::solver start for one component (component 0) of a caller's LDU
// matrix: r = source - A psi, and the partials of sum|r| and of OpenFOAM's
// normFactor, sum |A psi - rowSum avg(psi)| + |source - rowSum avg(psi)|,
// laid out as finResidual reads them (components 1 and 2 zero)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_ldu_start(const DevMesh m, const BlockMap bm, const double* __restrict__ psi,
                                                      const double* __restrict__ src, double avg, T* __restrict__ r,
                                                      double* __restrict__ part) {
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    const int C = m.nCells;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    double acc[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) acc[i] = 0.0;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = tl.s0 + wave; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        const int width = m.width(s);
        const int e0 = m.entry0(s);
        if (P >= tl.cEnd) continue;
        const double dg = m.diag[P];
        double Ap = dg * psi[P], asum = 0.0;
        for (int k = 0; k < width; ++k) {
            const int e = e0 + k * kSlice + lane;
            const int n = m.col[e];
            if (n >= 0) {
                const double a = m.eA[e];
                Ap -= a * psi[n];
                asum += a;
            }
        }
        const double t = (dg - asum) * avg;
        const double rv = src[P] - Ap;
        const T rT = (T)rv;
        r[P] = rT;
        r[(size_t)C + P] = (T)0;
        r[2 * (size_t)C + P] = (T)0;
        acc[0] += fabs(rv);
        acc[3] += fabs(Ap - t);
        acc[6] += fabs(src[P] - t);
        acc[9] += (double)(invD[P] * rT) * (double)rT;
    }
    storeBlockPartials<12, 0>(acc, part, kOffRes, lb, bm.nBlocks);
}

// ===========================================================================
// finalize kernels: one workgroup per instance (grid = number of instances)
// ===========================================================================

// the scalar step of one point of the launch sequence, from st.in to st.out
// (the same array when the launch sequence is not merged).  A pass finds many
// points with nothing owed (an outer step's while the PCG goes on): their
// partials are not reduced.  Solves with and without that test, per outer
// iteration: 128^3 cells FP32 1,655 -> 1,606 us, FP64 2,500 -> 2,455;
// 83^3 FP64 690 -> 676.
template <int POINT>
__global__ __launch_bounds__(kFinBlock) void k_fin(const BlockMap bm, const Stage st, const double* __restrict__ part) {
    const int inst = bm.finInst ? bm.finInst[blockIdx.x] : (int)blockIdx.x;
    __shared__ Ctl sh;
    __shared__ double tot[4 * PointOf<POINT>::nv];
    const Tile tl{inst, 0, 0, 0, bm.iBlk0[inst], bm.iNBlk[inst], bm.iNCell[inst], 0};
    const bool owed = pendingOf(st.in + inst) == PointOf<POINT>::pend;
    StageRun<POINT> run;
    run.load(st.in + inst, part, bm.nBlocks, tl.blk0, tl.nBlk);
    run.reduce(&sh, tot, part, bm.nBlocks, tl.blk0, tl.nBlk, owed);
    run.finish(&sh, tot, tl, st.hist, true, st.out + inst);
}

// The same on four times the threads, for launches of more than kFinWideTiles
// tiles: an instance of more has its rows split into four runs, each reduced as
// k_fin does and the four added in order (one of fewer keeps k_fin's order, and
// its bits, in the first).  Measured for 12, 6 and 3 values, k_fin -> wide: 8,192
// tiles (128^3 cells) 20.6 -> 18.6, 16.0 -> 11.9 (points before the outer step
// 12.8 -> 8.8), 10.4 -> 5.6 us, then bound by what one CU reads from beyond its
// L2; 2,213 tiles 6.4 -> 6.9, 5.5 -> 7.5, 4.8 -> 5.4.
template <int POINT>
__global__ __launch_bounds__(4 * kFinBlock) void k_fin_wide(const BlockMap bm, const Stage st,
                                                            const double* __restrict__ part) {
    typedef PointOf<POINT> Pt;
    const int inst = bm.finInst ? bm.finInst[blockIdx.x] : (int)blockIdx.x;
    __shared__ Ctl sh;
    __shared__ double run4[4][4 * Pt::nv], tot[4 * Pt::nv];
    const Tile tl{inst, 0, 0, 0, bm.iBlk0[inst], bm.iNBlk[inst], bm.iNCell[inst], 0};
    constexpr int nw = (int)(sizeof(Ctl) / 8);
    if ((int)threadIdx.x < nw)
        reinterpret_cast<long long*>(&sh)[threadIdx.x] = reinterpret_cast<const long long*>(st.in + inst)[threadIdx.x];
    const int g = threadIdx.x / kFinBlock, t = threadIdx.x % kFinBlock, nb = bm.nBlocks;
    const int len = tl.nBlk > kFinWideTiles ? (tl.nBlk + 3) / 4 : tl.nBlk;
    const bool owed = pendingOf(st.in + inst) == Pt::pend;
    const int b1 = tl.nBlk < (g + 1) * len ? tl.nBlk : (g + 1) * len;
    const double* col = part + (size_t)Pt::off * nb + tl.blk0;
    constexpr int kRows = 24 / Pt::nv;  // rows whose loads are in flight together
    double v[Pt::nv];
#pragma unroll
    for (int i = 0; i < Pt::nv; ++i) v[i] = 0.0;
    for (int b = g * len + t; b < b1; b += kRows * kFinBlock) {
        double x[24];
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
            for (int i = 0; i < Pt::nv; ++i) {
                const int row = b + r * kFinBlock;
                x[r * Pt::nv + i] = col[(size_t)i * nb + (row < b1 ? row : b)];
            }
        loadedHere(x);
        if (!owed) break;
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
            for (int i = 0; i < Pt::nv; ++i) {
                const double xv = b + r * kFinBlock < b1 ? x[r * Pt::nv + i] : 0.0;
                v[i] = i < Pt::nmax ? nanMax(v[i], xv) : v[i] + xv;
            }
    }
    waveReduceAll<Pt::nv, Pt::nmax>(v, run4[g], (t >> 6));
    __syncthreads();
    if (threadIdx.x < Pt::nv) {
        const int i = threadIdx.x;
        double s = overWaves<Pt::nmax>(run4[0], i);
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            const double x = overWaves<Pt::nmax>(run4[q], i);
            s = i < Pt::nmax ? nanMax(s, x) : s + x;
        }
        tot[4 * i] = s;
#pragma unroll
        for (int q = 1; q < 4; ++q) tot[4 * i + q] = 0.0;
    }
    __syncthreads();
    StageRun<POINT> run;
    run.finish(&sh, tot, tl, st.hist, true, st.out + inst);
}

// mean field of the initial gradient step (the first normFactor's xbar)
__global__ __launch_bounds__(kFinBlock) void k_fin_init(const BlockMap bm, Ctl* __restrict__ ctlAll,
                                                        const double* __restrict__ part) {
    const int inst = bm.finInst ? bm.finInst[blockIdx.x] : (int)blockIdx.x;
    __shared__ double tot[6];
    finReduce<6, 3>(part + (size_t)kOffGrad * bm.nBlocks, bm.nBlocks, bm.iBlk0[inst], bm.iNBlk[inst], tot);
    if (threadIdx.x == 0)
        for (int j = 0; j < 3; ++j) ctlAll[inst].xbar[j] = tot[3 + j] / (double)bm.iNCell[inst];
}

// n rows of K components from component-major storage (K arrays `stride` apart)
template <int K>
__global__ __launch_bounds__(kBlock) void k_to_rows(const double* __restrict__ src, size_t stride, int n,
                                                    double* __restrict__ out) {
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n * K; i += gridDim.x * kBlock)
        out[i] = src[(size_t)(i % K) * stride + i / K];
}

// a symmetric LDU matrix into the sliced-ELL entries of its faces (-upper) ...
__global__ __launch_bounds__(kBlock) void k_ldu_faces(int nFaces, const double* __restrict__ upper,
                                                      const int* __restrict__ own, const int* __restrict__ nei,
                                                      double* __restrict__ a64, float* __restrict__ a32) {
    for (int f = blockIdx.x * kBlock + threadIdx.x; f < nFaces; f += gridDim.x * kBlock) {
        const double a = -upper[f];
        a64[own[f]] = a;
        a64[nei[f]] = a;
        if (a32) {
            a32[own[f]] = (float)a;
            a32[nei[f]] = (float)a;
        }
    }
}
// ... and its diagonal's inverse and FP32 copies
__global__ __launch_bounds__(kBlock) void k_ldu_diag(int n, const double* __restrict__ d, double* __restrict__ inv,
                                                     float* __restrict__ d32, float* __restrict__ inv32) {
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        inv[i] = 1.0 / d[i];
        const float v = (float)d[i];
        d32[i] = v;
        inv32[i] = 1.0f / v;
    }
}

// stops the instances at the end of their current PCG solve (mixed
// precision's fallback)
__global__ void k_ctl_hold(Ctl* __restrict__ c, int n, int hold) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        c[i].hold = hold;
        c[i].stallWindow = 0;
        c[i].stalled = 0;
    }
}

// PCG start from a caller-supplied right-hand side (normFactor given)
__global__ __launch_bounds__(kFinBlock) void k_fin_pcg_start(const BlockMap bm, Ctl* __restrict__ ctlAll,
                                                             const double* __restrict__ part) {
    const int inst = bm.finInst ? bm.finInst[blockIdx.x] : (int)blockIdx.x;
    Ctl* ctl = ctlAll + inst;
    __shared__ double tot[6];
    finReduce<6, 0>(part + (size_t)kOffRho * bm.nBlocks, bm.nBlocks, bm.iBlk0[inst], bm.iNBlk[inst], tot);
    if (threadIdx.x == 0) {
        int any = 0;
        for (int j = 0; j < 3; ++j) {
            const bool solved = (ctl->solveMask >> j) & 1;
            ctl->initRes[j] = solved ? tot[j] / ctl->normFactor[j] : 0.0;
            ctl->finalRes[j] = ctl->initRes[j];
            ctl->rho[j] = tot[3 + j];
            ctl->nIter[j] = 0;
            const int act = solved && (ctl->pcgMaxIter > 0) && !(ctl->initRes[j] < ctl->pcgTol);
            ctl->active[j] = act;
            any |= act;
        }
        ctl->innerDone = !any;
        ctl->firstInner = 1;
    }
}

// control block set from a host value passed by argument (no host->device copy)
__global__ void k_ctl_set(Ctl* __restrict__ c, const Ctl v) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *c = v;
}

// p[0..n) = v (a kernel rather than a memset node, so callers may capture it)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_fill(T* __restrict__ p, size_t n, T v) {
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) p[i] = v;
}

// b = (double)a, exact
__global__ __launch_bounds__(kBlock) void k_widen(const float* __restrict__ a, double* __restrict__ b, size_t n) {
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock)
        b[i] = (double)a[i];
}

// plain streaming copy: the measured streaming ceiling and the known-size
// reference of the traffic counters.  One 32-byte load and store per thread
// over a grid covering the whole array (no grid-stride loop): of the copy
// forms measured on MI355X (grid-stride with one or four loads in flight per
// thread, 4-32 workgroups per CU, plain or non-temporal) this one streams
// fastest.  n is in 32-byte units.
typedef double dbl4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(kBlock) void k_copy(const dbl4* __restrict__ a, dbl4* __restrict__ b, size_t n) {
    const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) b[i] = a[i];
}

}  // namespace s4f
