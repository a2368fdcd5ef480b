// s4f_merged.h -- kernels for one slot count (6: hexahedra, 4: tetrahedra, 2-D
// quadrilaterals): those of merged launch sequences (Chain; meshes and batch
// members of up to kMergeTiles tiles), and k_residual_u, which larger meshes run
// too, between finalize kernels.
//
// Merged kernels move little data; their time is the launch and the chain of
// dependent loads behind it (data another XCD has just written comes from
// beyond the L2, about 0.7 us a step).  So each
//   * resolves its predecessor's scalars itself (StageRun) instead of waiting
//     for a finalize launch,
//   * issues loads that do not depend on those scalars first and reduces the
//     scalars while they are in flight.
// The arithmetic and its order are those of the kernels in s4f_kernels.h and
// s4f_amg.h, so results do not depend on which form a launch sequence takes.
#pragma once

#include "s4f_amg.h"

namespace s4f {

// y = d x - sum_k a_k x_k in slot order, rounded as the kernels for tiles of
// any kind round it: their unrolled rows (all three components active)
// contract d x with the first term's subtraction, their loops over the slots
// each term's product with its subtraction.  A capped PCG amplifies a last-bit
// difference, so both forms are spelled out here.
template <typename T, int W>
__device__ __forceinline__ T rowProduct(bool all, T d, T x, const T* a, const T* xn) {
    T y = all ? fmaT(d, x, -rounded(a[0] * xn[0])) : fmaT(-a[0], xn[0], rounded(d * x));
#pragma unroll
    for (int k = 1; k < W; ++k) y = fmaT(-a[k], xn[k], y);
    return y;
}

// hooke() with its contractions spelled out (mu2 = 2 mu)
__device__ __forceinline__ void hookeF(const double* G, double mu2, double K, double* s) {
    const double e0 = G[0], e3 = G[4], e5 = G[8];
    const double tr = e0 + e3 + e5;
    const double sh = tr * K, t3 = tr / 3.0;
    s[0] = fmaT(e0 - t3, mu2, sh);
    s[1] = rounded(((G[1] + G[3]) * 0.5) * mu2);
    s[2] = rounded(((G[2] + G[6]) * 0.5) * mu2);
    s[3] = fmaT(e3 - t3, mu2, sh);
    s[4] = rounded(((G[5] + G[7]) * 0.5) * mu2);
    s[5] = fmaT(e5 - t3, mu2, sh);
}

// One face's contribution to its row cell's residual sums (residualInternal),
// with every contraction as the compiler chooses it there: how many slots a
// kernel unrolls would otherwise decide the last bits.
__device__ __forceinline__ void faceTerms(double w, double S0, double S1, double S2, double cf, double a, double mu2,
                                          double K, const double* sP, const double* GP, const double* DP,
                                          const double* CP, const double* GN, const double* DN, const double* CN,
                                          double* sum) {
    const double tr = GN[0] + GN[4] + GN[8];
    const double sh = tr * K, t3 = tr / 3.0;
    const double e1 = (GN[1] + GN[3]) * 0.5, e2 = (GN[2] + GN[6]) * 0.5, e4 = (GN[5] + GN[7]) * 0.5;
    const double n0 = fmaT(GN[0] - t3, mu2, sh), n3 = fmaT(GN[4] - t3, mu2, sh), n5 = fmaT(GN[8] - t3, mu2, sh);
    const double f0 = fmaT(w, sP[0] - n0, n0), f3 = fmaT(w, sP[3] - n3, n3), f5 = fmaT(w, sP[5] - n5, n5);
    const double f1 = fmaT(w, fmaT(-e1, mu2, sP[1]), e1 * mu2);
    const double f2 = fmaT(w, fmaT(-e2, mu2, sP[2]), e2 * mu2);
    const double f4 = fmaT(w, fmaT(-e4, mu2, sP[4]), e4 * mu2);
    sum[0] += fmaT(S2, f2, fmaT(S1, f1, S0 * f0));
    sum[1] += dot3(S0, f1, S1, f3, S2, f4);
    sum[2] += dot3(S0, f2, S1, f4, S2, f5);
    double Gf[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) Gf[q] = fmaT(w, GP[q] - GN[q], GN[q]);
    const double d0 = CN[0] - CP[0], d1 = CN[1] - CP[1], d2 = CN[2] - CP[2];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        sum[3 + j] = fmaT(cf, (DN[j] - DP[j]) - dot3(d0, Gf[j], d1, Gf[3 + j], d2, Gf[6 + j]), sum[3 + j]);
        sum[6 + j] = fmaT(a, DN[j], sum[6 + j]);
    }
    sum[9] += a;
}

// the row slots of slice s, column and matrix coefficient
template <typename T, int W>
struct RowSlots {
    int nb[W];
    T a[W];
    __device__ __forceinline__ void load(const DevMesh& m, int e0, int lane) {
        const int* __restrict__ col = m.col + e0;
        const T* __restrict__ A = MatSel<T>::a(m) + e0;
#pragma unroll
        for (int k = 0; k < W; ++k) {
            nb[k] = at32(col + k * kSlice, lane * 4u);
            a[k] = at32(A + k * kSlice, lane * (unsigned)sizeof(T));
        }
    }
};

// k_update: x += alpha p, r -= alpha q, z = r/diag
template <typename T>
__global__ __launch_bounds__(kBlock) void k_update_m(const DevMesh m, const BlockMap bm, T* __restrict__ x,
                                                     const T* __restrict__ pA, const T* __restrict__ pB,
                                                     T* __restrict__ r, const T* __restrict__ q, const Stage st,
                                                     double* __restrict__ part) {
    constexpr int kPt = kPtUpdate;
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    __shared__ Ctl sh;
    __shared__ double tot[4 * PointOf<kPt>::nv];
    StageRun<kPt> run;
    run.load(st.in + tl.inst, part, bm.nBlocks, tl.blk0, tl.nBlk);
    const int C = m.nCells;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const int wave = waveOf(), lane = threadIdx.x & 63;
    int s = tl.s0 + wave;
    T xv[3], rv[3], qv[3], av[3], bv[3], iD = (T)0;
    auto fetch = [&](int s) {
        const unsigned o = lane * (unsigned)sizeof(T);
        const size_t c0 = (size_t)s * kSlice;
        iD = at32(invD + c0, o);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const size_t i = (size_t)j * C + c0;
            xv[j] = at32(x + i, o);
            rv[j] = at32(r + i, o);
            qv[j] = at32(q + i, o);
            av[j] = at32(pA + i, o);
            bv[j] = at32(pB + i, o);
        }
    };
    bool have = s < tl.s1 && s * kSlice + lane < tl.cEnd;
    if (have) fetch(s);
    run.reduce(&sh, tot, part, bm.nBlocks, tl.blk0, tl.nBlk);
    run.finish(&sh, tot, tl, st.hist, lb == tl.blk0, st.out + tl.inst);
    if (pendingOf(&sh) != kPendUpd) return;
    const bool odd = sh.pIt & 1;
    const T al[3] = {(T)sh.alpha[0], (T)sh.alpha[1], (T)sh.alpha[2]};
    const bool act[3] = {sh.active[0] != 0, sh.active[1] != 0, sh.active[2] != 0};
    const int first = sh.firstInner;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        if (P >= tl.cEnd) continue;
        if (!have) fetch(s);
        have = false;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const size_t i = (size_t)j * C + (size_t)s * kSlice;
            const unsigned o = lane * (unsigned)sizeof(T);
            if (!act[j]) {
                if (first) put32(x + i, o, (T)0);
                continue;
            }
            const T x0 = first ? (T)0 : xv[j];
            put32(x + i, o, (T)(x0 + al[j] * (odd ? av[j] : bv[j])));
            const T r1 = rv[j] - al[j] * qv[j];
            put32(r + i, o, r1);
            const T z = iD * r1;
            acc[j] += (double)z * (double)r1;
            acc[3 + j] += fabs((double)r1);
        }
    }
    storeBlockPartials<6, 0>(acc, part, kOffUpd, lb, bm.nBlocks);
}

// k_spmvp: p = z + beta p, q = M p.  The gathers need only the iteration's
// parity, known once the control block is there: they are in flight while the
// scalars are formed.
template <typename T, bool MG, bool AGAIN, int W>
__global__ __launch_bounds__(kBlock) void k_spmvp_m(const DevMesh m, const BlockMap bm, const T* __restrict__ r, T* pA,
                                                    T* pB, T* __restrict__ q, const Stage st,
                                                    double* __restrict__ part, const T* __restrict__ zArr) {
    constexpr int kPt = MG ? kPtSpmv : AGAIN ? kPtAgain : kPtInner;
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    __shared__ Ctl sh;
    __shared__ double tot[4 * PointOf<kPt>::nv];
    StageRun<kPt> run;
    run.load(st.in + tl.inst, part, bm.nBlocks, tl.blk0, tl.nBlk);
    const int C = m.nCells;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const T* __restrict__ dg = MatSel<T>::diag(m);
    const T* __restrict__ src = MG ? zArr : r;  // z, or r with z = r/diag
    const int wave = waveOf(), lane = threadIdx.x & 63;
    int s = tl.s0 + wave;
    RowSlots<T, W> row;
    T dP = (T)0, iDP = (T)0, zP[3] = {}, zN[W][3], iDN[W], oP[3], oN[W][3];
    const T* __restrict__ pOld = pA;
    constexpr unsigned kT = sizeof(T);
    auto fetch1 = [&](int s) {  // first-level loads
        const size_t c0 = (size_t)s * kSlice;
        row.load(m, m.entry0(s), lane);
        dP = at32(dg + c0, lane * kT);
        iDP = MG ? (T)0 : at32(invD + c0, lane * kT);
#pragma unroll
        for (int j = 0; j < 3; ++j) zP[j] = at32(src + (size_t)j * C + c0, lane * kT);
    };
    auto fetch2 = [&](int s) {  // gathers
        const int P = s * kSlice + lane;
#pragma unroll
        for (int j = 0; j < 3; ++j) oP[j] = at32(pOld + (size_t)j * C, P * kT);
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const bool v = row.nb[k] >= 0;
            const unsigned o = (v ? row.nb[k] : P) * kT;
            row.a[k] = v ? row.a[k] : (T)0;
            iDN[k] = MG ? (T)0 : at32(invD, o);
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                zN[k][j] = at32(src + (size_t)j * C, o);
                oN[k][j] = at32(pOld + (size_t)j * C, o);
            }
        }
    };
    bool have = s < tl.s1 && s * kSlice + lane < tl.cEnd;
    if (have) fetch1(s);
    run.reduce(&sh, tot, part, bm.nBlocks, tl.blk0, tl.nBlk);
    // the parity after this point's scalar step
    const int pend0 = pendingOf(&sh);
    int it = __builtin_amdgcn_readfirstlane(sh.pIt);
    if (!MG && pend0 == PointOf<kPt>::pend) it = AGAIN ? it + 1 : 0;
    const bool odd = it & 1;
    pOld = odd ? pB : pA;
    T* __restrict__ pNew = odd ? pA : pB;
    if (have) fetch2(s);
    run.finish(&sh, tot, tl, st.hist, lb == tl.blk0, st.out + tl.inst);
    if (pendingOf(&sh) != kPendSpmv) return;
    const int first = sh.firstInner;
    const bool act[3] = {sh.active[0] != 0, sh.active[1] != 0, sh.active[2] != 0};
    const bool all = __builtin_amdgcn_readfirstlane(act[0] && act[1] && act[2]);
    const T be[3] = {(T)sh.beta[0], (T)sh.beta[1], (T)sh.beta[2]};
    auto dir = [&](int j, T z0, T iD, T o) -> T {
        const T z = MG ? z0 : iD * z0;
        const T d = z + be[j] * o;
        return first ? z : d;
    };
    double acc[3] = {0, 0, 0};
    for (; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        if (P >= tl.cEnd) continue;
        if (!have) {
            fetch1(s);
            fetch2(s);
        }
        have = false;
        T pP[3], y[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            T pN[W];
            pP[j] = dir(j, zP[j], iDP, oP[j]);
#pragma unroll
            for (int k = 0; k < W; ++k) pN[k] = dir(j, zN[k][j], iDN[k], oN[k][j]);
            y[j] = rowProduct<T, W>(all, dP, pP[j], row.a, pN);
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            if (!act[j]) continue;
            const size_t i = (size_t)j * C + (size_t)s * kSlice;
            put32(pNew + i, lane * kT, pP[j]);
            put32(q + i, lane * kT, y[j]);
            acc[j] += (double)pP[j] * (double)y[j];
        }
    }
    storeBlockPartials<3, 0>(acc, part, kOffSpmv, lb, bm.nBlocks);
}
// k_mg0_down: r = b - A x with x = w D^-1 b; no load depends on the scalars
template <typename T, bool AGAIN, int W>
__global__ __launch_bounds__(kBlock) void k_mg0_down_m(const DevMesh m, const BlockMap bm, const T* __restrict__ b,
                                                       Row3<T>* __restrict__ r, double omega, const Stage st,
                                                       const double* __restrict__ part) {
    constexpr int kPt = AGAIN ? kPtAgain : kPtInner;
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    __shared__ Ctl sh;
    __shared__ double tot[4 * PointOf<kPt>::nv];
    StageRun<kPt> run;
    run.load(st.in + tl.inst, part, bm.nBlocks, tl.blk0, tl.nBlk);
    const int C = m.nCells;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const T* __restrict__ dg = MatSel<T>::diag(m);
    const T w = (T)omega;
    const int wave = waveOf(), lane = threadIdx.x & 63;
    int s = tl.s0 + wave;
    RowSlots<T, W> row;
    T iDP = (T)0, dP = (T)0, bP[3] = {}, bN[W][3], iDN[W];
    constexpr unsigned kT = sizeof(T);
    auto fetch = [&](int s) {
        const int P = s * kSlice + lane;
        row.load(m, m.entry0(s), lane);
        iDP = at32(invD, P * kT);
        dP = at32(dg, P * kT);
#pragma unroll
        for (int j = 0; j < 3; ++j) bP[j] = at32(b + (size_t)j * C, P * kT);
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const bool v = row.nb[k] >= 0;
            const unsigned o = (v ? row.nb[k] : P) * kT;
            row.a[k] = v ? row.a[k] : (T)0;
            iDN[k] = at32(invD, o);
#pragma unroll
            for (int j = 0; j < 3; ++j) bN[k][j] = at32(b + (size_t)j * C, o);
        }
    };
    bool have = s < tl.s1 && s * kSlice + lane < tl.cEnd;
    if (have) fetch(s);
    run.reduce(&sh, tot, part, bm.nBlocks, tl.blk0, tl.nBlk);
    run.finish(&sh, tot, tl, st.hist, lb == tl.blk0, st.out + tl.inst);
    if (mgSkip(&sh)) return;
    const bool act[3] = {sh.active[0] != 0, sh.active[1] != 0, sh.active[2] != 0};
    const bool all = __builtin_amdgcn_readfirstlane(act[0] && act[1] && act[2]);
    for (; s < tl.s1; s += kBlock / 64) {
        const int P = s * kSlice + lane;
        if (P >= tl.cEnd) continue;
        if (!have) fetch(s);
        have = false;
        T y[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            T xn[W];
#pragma unroll
            for (int k = 0; k < W; ++k) xn[k] = w * iDN[k] * bN[k][j];
            y[j] = rowProduct<T, W>(all, dP, w * iDP * bP[j], row.a, xn);
        }
        r[P] = Row3<T>{{(T)(bP[0] - y[0]), (T)(bP[1] - y[1]), (T)(bP[2] - y[2])}};  // a converged component's is not read
    }
}
// The residual of meshes of one slot count, in merged launch sequences
// (MERGED) and with finalize kernels: one slice per wavefront,
// the slots in a loop.  A wavefront's time is its instructions (one about every
// 2.5 ns) plus a load latency per slot, so
//   * the slots are not unrolled (unrolled, 512 cells took 16.1 us, as a loop 11.2),
//   * the loop's registers are kept to what one slot needs: the sums over the
//     workgroup's cells (SliceAcc) are no part of it,
//   * boundary slots are visited only where the wavefront has any (a bit per slot).

// A thread's sums over its cells: its first (mostly only) slice's live in
// registers from that slice's end on, earlier slices' of larger tiles in LDS.
template <int N>
struct SliceAcc {
    double (*lds)[kBlock];
    bool first = true;
    __device__ __forceinline__ void get(double* v) const {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = first ? 0.0 : lds[i][threadIdx.x];
    }
    __device__ __forceinline__ void put(const double* v) {
#pragma unroll
        for (int i = 0; i < N; ++i) lds[i][threadIdx.x] = v[i];
        first = false;
    }
};

// k_residual.  MU: moduli per cell (a branch in the row would let the loads of
// all slots drift together).  Not MERGED (more cells than the L2s hold): a
// slot's loads are issued together and the face data streams past the L2;
// 128^3 cells (FP32 PCG): 277 us before (k_residual), 335 with the loads as the
// compiler schedules them, 270 now, against 169 for each array read once: the
// neighbour planes' gradients are fetched again from beyond the 4 MB L2s.  Two
// slots at a time: 287.  MERGED the compiler's schedule is better (512 cells:
// 10.4 us, 12.4 with the loads together; before 11.2).
template <typename T, int W, bool MU, bool MERGED>
__global__ __launch_bounds__(kBlock, 3) void k_residual_u(
    const DevMesh m, const BlockMap bm, const double* __restrict__ D0, const double* __restrict__ D1,
    const double* __restrict__ G, const double* __restrict__ sigb, T* __restrict__ r, const Stage st,
    double* __restrict__ part) {
    constexpr int kPt = kPtRes;
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    __shared__ Ctl sh;
    __shared__ double tot[4 * PointOf<kPt>::nv];
    __shared__ double accL[12][kBlock];
    const int C = m.nCells, B = m.nBoundary;
    const size_t E = m.nEntries;
    const T* __restrict__ invD = MatSel<T>::invDiag(m);
    const int wave = waveOf(), lane = threadIdx.x & 63;
    int s = tl.s0 + wave;
    int e0 = s < tl.s1 ? m.entry0(s) : 0;
    int nb = kPad;  // column of the slot at hand
    // face data read once: past the gathered rows in the L2 where those do not fit
    auto stream = [&](const double* p) { return MERGED ? at32(p, lane * 8u) : at32s(p, lane * 8u); };
    auto col = [&](int e0, int k) {
        const int* p = m.col + e0 + k * kSlice;
        return MERGED ? at32(p, lane * 4u) : at32s(p, lane * 4u);
    };
    const Ctl* c;
    if constexpr (MERGED) {
        StageRun<kPt> run;
        run.load(st.in + tl.inst, part, bm.nBlocks, tl.blk0, tl.nBlk);
        if (s < tl.s1) nb = col(e0, 0);
        run.reduce(&sh, tot, part, bm.nBlocks, tl.blk0, tl.nBlk);
        run.finish(&sh, tot, tl, st.hist, lb == tl.blk0, st.out + tl.inst);
        c = &sh;
    } else {
        c = st.in + tl.inst;
        if (s < tl.s1) nb = col(e0, 0);
    }
    if (pendingOf(c) != kPendRes) return;
    const double* __restrict__ D = __builtin_amdgcn_readfirstlane(c->dpar) ? D1 : D0;
    const double xb[3] = {c->xbar[0], c->xbar[1], c->xbar[2]};
    // a cold start's first residual sees the zero initial stress field
    const double sf = (c->sigma0 && c->iCorr == 0) ? 0.0 : 1.0;
    SliceAcc<12> sa{accL};
    double acc[12];
    sa.get(acc);
    while (s < tl.s1) {
        const int P = s * kSlice + lane;
        const bool on = P < tl.cEnd;
        const unsigned l8 = lane * 8u, p8 = (on ? P : tl.cEnd - 1) * 8u;  // no cell: any row, its sums dropped
        double DP[3], GP[9], CP[3], sP[6];
#pragma unroll
        for (int k = 0; k < 3; ++k) { DP[k] = at32(D + (size_t)k * C, p8); CP[k] = at32(m.cC + (size_t)k * C, p8); }
#pragma unroll
        for (int k = 0; k < 9; ++k) GP[k] = at32(G + (size_t)k * C, p8);
        loadsAbove();
        hookeF(GP, 2.0 * ((MU ? at32(m.mu, p8) : m.mu0) * sf), (MU ? at32(m.K, p8) : m.K0) * sf, sP);
        double sum[10] = {};  // div sigma, Rhie-Chow, off-diagonal product, coefficient sum
        unsigned bs = 0;      // slots in which the wavefront has boundary faces
#pragma unroll 1
        for (int k = 0; k < W; ++k) {
            const int nx = k + 1 < W ? col(e0, k + 1) : kPad;
            const size_t e = (size_t)e0 + k * kSlice;
            const bool v = nb >= 0;
            bs |= __any(!v && nb != kPad) ? 1u << k : 0u;
            const unsigned c8 = v ? nb * 8u : p8;
            double S0r = stream(m.eS + e), S1r = stream(m.eS + E + e), S2r = stream(m.eS + 2 * E + e);
            double w = stream(m.eW + e), cfr = stream(m.eC + e), ar = stream(m.eA + e);
            double GN[9], DN[3], CN[3];
#pragma unroll
            for (int q = 0; q < 9; ++q) GN[q] = at32(G + (size_t)q * C, c8);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                DN[q] = at32(D + (size_t)q * C, c8);
                CN[q] = at32(m.cC + (size_t)q * C, c8);
            }
            const double muN = MU ? at32(m.mu, c8) : m.mu0, KNr = MU ? at32(m.K, c8) : m.K0;
            if (!MERGED) loadedHere(S0r, S1r, S2r, w, cfr, ar, GN, DN, CN);
            const double S0 = v ? S0r : 0.0, S1 = v ? S1r : 0.0, S2 = v ? S2r : 0.0;
            const double cf = v ? cfr : 0.0, a = v ? ar : 0.0;
            const double mu2 = 2.0 * (muN * sf), KN = KNr * sf;
            faceTerms(w, S0, S1, S2, cf, a, mu2, KN, sP, GP, DP, CP, GN, DN, CN, sum);
            nb = nx;
        }
        for (; bs; bs &= bs - 1) {
            const int k = __builtin_ctz(bs);
            const size_t e = (size_t)e0 + k * kSlice;
            const int n = col(e0, k);
            if (n >= 0 || n == kPad) continue;
            const unsigned b8 = (-1 - n) * 8u;
            double S[3], sb[6];
#pragma unroll
            for (int q = 0; q < 3; ++q) S[q] = at32(m.eS + (size_t)q * E + e, l8);
#pragma unroll
            for (int q = 0; q < 6; ++q) sb[q] = at32(sigb + (size_t)q * B, b8);
            sum[0] += dot3(S[0], sb[0], S[1], sb[1], S[2], sb[2]);
            sum[1] += dot3(S[0], sb[1], S[1], sb[3], S[2], sb[4]);
            sum[2] += dot3(S[0], sb[2], S[1], sb[4], S[2], sb[5]);
        }
        const double dg = at32(m.diag, p8);
        const T iDP = at32(invD, p8 / (unsigned)(8 / sizeof(T)));
        const double rowsum = dg - sum[9];
        double src[3] = {0.0, 0.0, 0.0};
        if (m.fext && on) {
#pragma unroll
            for (int j = 0; j < 3; ++j) src[j] = m.fext[(size_t)j * C + P] - (m.iner ? m.iner[P] * DP[j] : 0.0);
        }
        sa.get(acc);
        if (on) {
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const double R = (sum[j] + sum[3 + j]) + src[j];
                const double MD = fmaT(dg, DP[j], -sum[6 + j]);
                acc[j] += fabs(R);
                acc[3 + j] += fabs(fmaT(-rowsum, xb[j], MD));
                acc[6 + j] += fabs(fmaT(-rowsum, xb[j], MD + R));
                const T rT = (T)R;
                put32(r + (size_t)j * C, P * (unsigned)sizeof(T), rT);
                const T z = iDP * rT;
                acc[9 + j] += (double)z * (double)rT;
            }
        }
        s += kBlock / 64;
        if (s >= tl.s1) break;
        sa.put(acc);
        e0 = m.entry0(s);
        nb = col(e0, 0);
    }
    storeBlockPartials<12, 0>(acc, part, kOffRes, lb, bm.nBlocks);
}

// The gradient step in one launch (no Aitken relaxation, no sub-meshes): the
// tile's boundary faces go into a queue in LDS, its threads update them one
// face each (k_grad_bnd_pre), the cells form their gradients (k_grad), and the
// threads return to the faces (k_grad_bnd_post).  Workgroup barriers order the
// three through the workgroup's own global stores.  Two slots' gathers in
// flight at a time (three, with the cell's own values loaded over the first
// face update, measured the same up to 64,000 cells and worse above; face
// loads issued before the scalars are known slowed the launches that find
// nothing to do).  Of 16 us at 512 cells the faces took 5.6 (queue, update,
// return); with a ballot per slot for the queue and a face's loads at once it
// is 14.7, and 10 + 6 + 4 us in three launches.  24 boxes: 41 -> 38 us.  The
// update in the cells' own lanes, without queue or barriers, took 19.4 and 45.
template <typename T, int W>
__global__ __launch_bounds__(kBlock, 4) void k_grad_m(
    const DevMesh m, const BlockMap bm, double* __restrict__ D0, const T* __restrict__ x, double* __restrict__ D1,
    double* G, double* Db, const double* __restrict__ Dold, const Stage st, double* __restrict__ part,
    const BndBufs bb) {
    constexpr int U = 2;
    constexpr int kPt = kPtGrad;
    constexpr int kWaves = kBlock / 64;
    const int lb = logicalBlock(bm.nBlocks);
    const Tile tl = bm.at(lb);
    __shared__ Ctl sh;
    __shared__ double tot[4 * PointOf<kPt>::nv];
    __shared__ int qCount[kWaves], qFace[kBlock * W], qCell[kBlock * W];
    StageRun<kPt> run;
    run.load(st.in + tl.inst, part, bm.nBlocks, tl.blk0, tl.nBlk);
    const int C = m.nCells, B = m.nBoundary;
    const int wave = waveOf(), lane = threadIdx.x & 63;
    int nb[W];
    auto cols = [&](int s) {
#pragma unroll
        for (int k = 0; k < W; ++k) nb[k] = kPad;
        if (s < tl.s1 && s * kSlice + lane < tl.cEnd) {
            const int* __restrict__ col = m.col + m.entry0(s);
#pragma unroll
            for (int k = 0; k < W; ++k) nb[k] = at32(col + k * kSlice, lane * 4u);
        }
    };
    cols(tl.s0 + wave);
    run.reduce(&sh, tot, part, bm.nBlocks, tl.blk0, tl.nBlk);
    run.finish(&sh, tot, tl, st.hist, lb == tl.blk0, st.out + tl.inst);
    if (pendingOf(&sh) != kPendGrad) return;
    const bool dpar = __builtin_amdgcn_readfirstlane(sh.dpar) != 0;
    const double* __restrict__ D = dpar ? D1 : D0;
    double* __restrict__ Dn = dpar ? D0 : D1;
    const bool hasX = __builtin_amdgcn_readfirstlane(sh.firstInner) == 0;  // else no PCG iteration ran: the update is zero
    const BndStep u = bndStep(&sh, 0);
    const double ra = u.ra;
    double acc[6] = {0, 0, 0, 0, 0, 0};  // max|D'-D|^2, max|D'-Dold|^2, max|D'|^2, sum D'
    for (int sb = tl.s0; sb < tl.s1; sb += kWaves) {
        const int s = sb + wave;
        const int P = s * kSlice + lane;
        const bool on = s < tl.s1 && P < tl.cEnd;
        const unsigned p8 = P * 8u, pT = P * (unsigned)sizeof(T);
        if (sb != tl.s0) {
            __syncthreads();  // the queue is reused
            cols(s);
        }
        // a wavefront's boundary faces, in its own part of the queue
        int n = 0;
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const bool isB = nb[k] < 0 && nb[k] != kPad;
            const unsigned long long mask = __ballot(isB);
            if (isB) {
                const int at = wave * (kSlice * W) + n + __popcll(mask & ((1ull << lane) - 1));
                qFace[at] = -1 - nb[k];
                qCell[at] = P;
            }
            n += __popcll(mask);
        }
        if (lane == 0) qCount[wave] = n;
        __syncthreads();
        // its parts end to end
        const int q0 = qCount[0], q1 = q0 + qCount[1], q2 = q1 + qCount[2], nq = q2 + qCount[3];
        auto place = [&](int i) {
            const int w = (i >= q0) + (i >= q1) + (i >= q2);
            return w * (kSlice * W) + i - (w == 0 ? 0 : w == 1 ? q0 : w == 2 ? q1 : q2);
        };
        double DP[3], DnP[3], CP[3], Mi[6];
        for (int i = threadIdx.x; i < nq; i += kBlock) {
            const int at = place(i), b = qFace[at], Pf = qCell[at];
            FaceIn f;
            f.fixed(m, b);
            f.fields(m, b, bb.g, Db);
            double Du[3], Dr[3], Gold[9], Dbn[3], sn[3];
#pragma unroll
            for (int q = 0; q < 9; ++q) Gold[q] = at32(G + (size_t)q * C, Pf * 8u);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double d0 = at32(D + (size_t)k * C, Pf * 8u);
                const double xv = hasX ? (double)at32(x + (size_t)k * C, Pf * (unsigned)sizeof(T)) : 0.0;
                Du[k] = d0 + xv;
                Dr[k] = fmaT(ra, xv, d0);
            }
            bndPreFace(m, u, b, f, Du, Dr, Gold, nullptr, nullptr, Dbn, sn);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                put32(Db + (size_t)q * B, b * 8u, Dbn[q]);
                put32(bb.snb + (size_t)q * B, b * 8u, sn[q]);
            }
        }
        __syncthreads();
        if (on) {
            double A[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) A[q] = 0.0;
            bool hasB = false;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                DP[k] = at32(D + (size_t)k * C, p8);
                const double xv = hasX ? (double)at32(x + (size_t)k * C, pT) : 0.0;
                DnP[k] = fmaT(ra, xv, DP[k]);
                CP[k] = at32(m.cC + (size_t)k * C, p8);
            }
#pragma unroll
            for (int q = 0; q < 6; ++q) Mi[q] = at32(m.minv + (size_t)q * C, p8);
            const int* __restrict__ colS = m.col + m.entry0(s);
#pragma unroll 1
            for (int k0 = 0; k0 < W; k0 += U) {
                int n[U];
                double cN[U][3], dN[U][3];
                T xN[U][3];
#pragma unroll
                for (int u = 0; u < U; ++u) n[u] = at32(colS + (k0 + u) * kSlice, lane * 4u);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int c = n[u] >= 0 ? n[u] : P;
                    const unsigned c8 = c * 8u, cT = c * (unsigned)sizeof(T);
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        cN[u][q] = at32(m.cC + (size_t)q * C, c8);
                        xN[u][q] = at32(x + (size_t)q * C, cT);
                        dN[u][q] = at32(D + (size_t)q * C, c8);
                    }
                }
                loadsAbove();
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool v = n[u] >= 0;
                    hasB |= !v && n[u] != kPad;
                    double d[3], dv[3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        d[q] = cN[u][q] - CP[q];
                        dv[q] = fmaT(ra, hasX ? (double)xN[u][q] : 0.0, dN[u][q]) - DnP[q];
                    }
                    const double dd = dot3(d[0], d[0], d[1], d[1], d[2], d[2]);
                    const double rr = v ? 1.0 / dd : 0.0;
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        const double di = rounded(d[i] * rr);
#pragma unroll
                        for (int j = 0; j < 3; ++j) A[3 * i + j] = fmaT(di, dv[j], A[3 * i + j]);
                    }
                }
            }
            if (__any(hasB)) {
#pragma unroll 1
                for (int k0 = 0; k0 < W; k0 += W / 2) {
                    bool v[W / 2];
                    double lv[W / 2][3], dv[W / 2][3];
#pragma unroll
                    for (int u = 0; u < W / 2; ++u) {
                        const int n = at32(colS + (k0 + u) * kSlice, lane * 4u);
                        v[u] = n < 0 && n != kPad;
                        const unsigned b8 = v[u] ? (-1 - n) * 8u : 0u;
#pragma unroll
                        for (int q = 0; q < 3; ++q) {
                            lv[u][q] = at32(m.bLs + (size_t)q * B, b8);
                            dv[u][q] = at32(Db + (size_t)q * B, b8) - DnP[q];
                        }
                    }
#pragma unroll
                    for (int u = 0; u < W / 2; ++u) {
                        if (!v[u]) continue;
#pragma unroll
                        for (int i = 0; i < 3; ++i)
#pragma unroll
                            for (int j = 0; j < 3; ++j) A[3 * i + j] = fmaT(lv[u][i], dv[u][j], A[3 * i + j]);
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                put32(G + (size_t)j * C, p8, dot3(Mi[0], A[j], Mi[1], A[3 + j], Mi[2], A[6 + j]));
                put32(G + (size_t)(3 + j) * C, p8, dot3(Mi[1], A[j], Mi[3], A[3 + j], Mi[4], A[6 + j]));
                put32(G + (size_t)(6 + j) * C, p8, dot3(Mi[2], A[j], Mi[4], A[3 + j], Mi[5], A[6 + j]));
            }
            double a[3], o[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                put32(Dn + (size_t)q * C, p8, DnP[q]);
                a[q] = DnP[q] - DP[q];
                o[q] = Dold ? DnP[q] - at32(Dold + (size_t)q * C, p8) : DnP[q];
                acc[3 + q] += DnP[q];
            }
            acc[0] = nanMax(acc[0], dot3(a[0], a[0], a[1], a[1], a[2], a[2]));
            acc[1] = nanMax(acc[1], dot3(o[0], o[0], o[1], o[1], o[2], o[2]));
            acc[2] = nanMax(acc[2], dot3(DnP[0], DnP[0], DnP[1], DnP[1], DnP[2], DnP[2]));
        }
        __syncthreads();
        for (int i = threadIdx.x; i < nq; i += kBlock) {
            const int at = place(i), b = qFace[at], Pf = qCell[at];
            const int type = at32(m.bType, b * 4u);
            double Gn[9], n[3], val[3], sn[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                n[q] = at32(m.bN + (size_t)q * B, b * 8u);
                val[q] = at32(m.bVal + (size_t)q * B, b * 8u);
                sn[q] = at32(bb.snb + (size_t)q * B, b * 8u);
            }
#pragma unroll
            for (int q = 0; q < 9; ++q) Gn[q] = at32(G + (size_t)q * C, Pf * 8u);
            bndPostFace(m, 0, false, b, type, Pf, Gn, n, val, sn, bb.Gb, bb.sigb, bb.g);
        }
    }
    storeBlockPartials<6, 3>(acc, part, kOffGrad, lb, bm.nBlocks);
}
}  // namespace s4f
