// kernels_modify.h -- rank-k update/downdate of the resident supernodal LL'
// factor (CHOLMOD's cholmod_updown, CHOLMOD/Modify/cholmod_updown.c:74):
//   Lnew Lnew' = L L' + C C' (update) or L L' - C C' (downdate),
// C's rows in the factor's order, at most UD_RANK columns per pass.
//
// Each column j on the paths of C's columns is modified by the recurrence of
// Modify/t_cholmod_updown_numkr.c on its LDL' form:
//   pivot (:294-324): d = l_jj^2; per rank r whose path holds j, in order:
//     a = alpha_r +- w_r(j)^2 / d;  d *= a;  alpha_r = a;
//     gamma_r = -+ w_r(j) / d;      d /= alpha_r (old)
//   rows i below j (:363-372): l = l_ij / l_jj (old);
//     per rank: w_r(i) -= w_r(j) l;  l -= gamma_r w_r(i)
//   then l_jj = sqrt(d), l_ij = l * l_jj.
// A 64-column block of a supernode is one workgroup (k_updown_block), a wave per
// rank.  The rows below the block take the block's 64 columns of pivot data in a
// second launch (k_updown_rows), a lane per row.  The modified
// blocks' inverses (the solve sweeps use them) are formed once at the end, all
// blocks in parallel (k_updown_inv).  Every operation is
// written out and contraction is off, so the result does not depend on the
// block a column falls in or on the launch that takes its rows; a column that
// no path reaches is not touched (its LDL' round trip would not be exact).
#pragma once
#include <hip/hip_runtime.h>
#include "mxc_kernels.h"

namespace mxc {

constexpr int UD_RANK = 8;                 // columns of C per pass (Common->maxrank)
constexpr int UD_PAR = 2 + 2 * UD_RANK;    // per column: old pivot, new pivot, then w_r(j) and gamma_r

// One 64-column block [c0, c0 + nb) of a supernode s on the paths.
struct UdBlock {
    long long lx;            // W offset of supernode s (Lpx[s])
    long long winv;          // W offset of this block's inverse (ld nb)
    int nsrow, nscol;
    int k1, psi;             // first column, first row index position in Ls
    int c0, nb;
    int start[UD_RANK];      // per rank: first column of s on its path, or INT_MAX
    int slot;                // pivot-data slot of this block in its launch
    int pad;
};

// Rows [r0, min(r0 + 64, nsrow)) of the supernode of block blk, below the block.
struct UdRows {
    int blk;
    int r0;
};

// C's entries: W[row * UD_RANK + rank] = value (the host keeps the last of
// repeated entries of a column).
template <typename T>
__global__ __launch_bounds__(256) void k_updown_scatter(const long long *__restrict__ idx,
                                                        const double *__restrict__ val, long long nz,
                                                        T *__restrict__ Wc) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nz) Wc[idx[k]] = (T)val[k];
}

// The diagonal block, a wave per rank (rank r = wave r), lanes = the block's
// rows.  The recurrence at (column c, rank r) needs (c, r-1) for the pivot and
// for the rows' l, and (c-1, r) for w_r and alpha_r, so at step k wave r takes
// column k - r: the ranks' divisions, one after the other in a single wave, run
// side by side, and a block takes nb + 7 steps of one pivot each instead of
// 8 nb.  d and the rows' l pass from wave to wave in LDS, one barrier a step; w
// and alpha stay in the rank's registers.  The division of the rows by the old
// pivots before the chain and the product with the new ones after it are done
// for the whole block at once.  What bounds it: the two dependent divisions of
// a step (a 64-column block with 8 ranks, 48^3: 81 us with one wave, 29 us so).
constexpr int UD_THREADS = 64 * UD_RANK;

template <typename T>
__global__ __launch_bounds__(UD_THREADS) void k_updown_block(const UdBlock *__restrict__ blocks,
                                                             T *__restrict__ W, T *__restrict__ Wc,
                                                             T *__restrict__ alpha, T *__restrict__ par, int update,
                                                             double dbound, int *__restrict__ flag) {
#pragma clang fp contract(off)
    __shared__ T S[NB][DS];                // the diagonal block by columns: S[c][i] = L(i, c), then l
    __shared__ T Dj[NB];                   // a column's pivot d on its way through the ranks
    __shared__ T Lold[NB];
    const UdBlock b = blocks[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63, nb = b.nb;
    const int r = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long long base = b.lx + (long long)b.c0 * b.nsrow + b.c0;   // element (c0, c0)
    const int il = min(lane, nb - 1);
    {
        T v[NB / UD_RANK];                 // every load in flight, then the LDS stores
#pragma unroll
        for (int q = 0; q < NB / UD_RANK; q++)
            v[q] = W[base + (long long)min(r + UD_RANK * q, nb - 1) * b.nsrow + il];
#pragma unroll
        for (int q = 0; q < NB / UD_RANK; q++) S[r + UD_RANK * q][lane] = v[q];
    }
    const long long g = (long long)(b.k1 + b.c0 + il) * UD_RANK;
    T w = Wc[g + r];
    const int last = b.c0 + nb - 1;
    int first = INT_MAX;                   // columns before every path are left alone
#pragma unroll
    for (int q = 0; q < UD_RANK; q++) first = min(first, b.start[q]);
    const int start = blocks[blockIdx.x].start[r];
    const bool own = start <= last;        // rank r passes here
    T al = own ? alpha[r] : (T)1;
    T *ps = par + (long long)b.slot * NB * UD_PAR;
    __syncthreads();
    if (r == 0 && lane < nb) {
        const T lo = S[lane][lane];
        Lold[lane] = lo;
        Dj[lane] = lo * lo;
    }
    __syncthreads();
    for (int c = r; c < nb; c += UD_RANK)
        if (b.c0 + c >= first && lane > c) S[c][lane] = S[c][lane] / Lold[c];
    __syncthreads();

    const int cfirst = max(first - b.c0, 0);
    for (int k = cfirst; k < nb + UD_RANK - 1; k++) {
        const int c = k - r;
        if (c >= cfirst && c < nb && b.c0 + c >= start) {
            T dj = Dj[c];
            T l = S[c][lane];
            const T wr = lane_bcast(w, c), a0 = al;
            T t = wr * wr;
            t = t / dj;
            const T a = update ? a0 + t : a0 - t;
            dj = dj * a;
            al = a;
            const T gm = update ? (-wr) / dj : wr / dj;
            dj = dj / a0;
            const T wn = w - wr * l;
            l = l - gm * wn;
            if (lane > c) {
                w = wn;
                S[c][lane] = l;
            } else if (lane == c) {
                Dj[c] = dj;
                ps[c * UD_PAR + 2 + r] = wr;
                ps[c * UD_PAR + 2 + UD_RANK + r] = gm;
            }
        }
        __syncthreads();
    }
    // the new pivots, column by lane
    if (r == 0 && lane < nb && b.c0 + lane >= first) {
        T dj = Dj[lane];
        if (dbound > 0 && !(dj != dj)) {
            const T bnd = (T)dbound;
            if (dj >= (T)0 ? dj < bnd : dj > -bnd) {
                dj = dj >= (T)0 ? bnd : -bnd;
                atomicAdd(flag + 1, 1);
            }
        }
        if (!(dj > (T)0)) atomicMin(flag, b.k1 + b.c0 + lane);
        const T lnew = sqrt(dj);
        Dj[lane] = lnew;
        ps[lane * UD_PAR] = Lold[lane];
        ps[lane * UD_PAR + 1] = lnew;
    }
    __syncthreads();
    for (int c = r; c < nb; c += UD_RANK)
        if (b.c0 + c >= first && lane >= c && lane < nb)
            W[base + (long long)c * b.nsrow + lane] = lane > c ? S[c][lane] * Dj[c] : Dj[c];
    if (own && lane == 0) alpha[r] = al;
}

// The new inverses of the modified diagonal blocks (the solve sweeps use
// them), all at once after the last pass: a workgroup per block; lane c forms
// column c of inv(L) by forward substitution, row after row,
//   x_i = (delta_ic - sum_{c <= k < i} L_ik x_k) / L_ii,
// with four partial sums.
template <typename T>
__global__ __launch_bounds__(64) void k_updown_inv(const DiagTask *__restrict__ tasks, T *__restrict__ W) {
    __shared__ T S[NB][DS];
    __shared__ T X[NB][DS];
    __shared__ T rd[NB];
    const DiagTask t = tasks[blockIdx.x];
    const int lane = threadIdx.x, nb = t.nb;
    {
        T v[NB];
#pragma unroll
        for (int c = 0; c < NB; c++) v[c] = (lane < nb && c <= lane) ? W[t.off + (long long)c * t.ld + lane] : (T)0;
#pragma unroll
        for (int c = 0; c < NB; c++) S[lane][c] = v[c];
    }
    if (lane < nb) rd[lane] = (T)1 / W[t.off + (long long)lane * t.ld + lane];
    __syncthreads();
    for (int i = 0; i < nb; i++) {
        T s0 = (T)0, s1 = (T)0, s2 = (T)0, s3 = (T)0;
        int k = lane;
        for (; k + 3 < i; k += 4) {
            s0 += S[i][k] * X[k][lane];
            s1 += S[i][k + 1] * X[k + 1][lane];
            s2 += S[i][k + 2] * X[k + 2][lane];
            s3 += S[i][k + 3] * X[k + 3][lane];
        }
        for (; k < i; k++) s0 += S[i][k] * X[k][lane];
        const T v = ((i == lane ? (T)1 : (T)0) - ((s0 + s1) + (s2 + s3))) * rd[i];
        X[i][lane] = lane <= i ? v : (T)0;
    }
    __syncthreads();
    for (int c = 0; c < nb; c++)
        if (lane < nb) W[t.winv + lane + (long long)c * nb] = X[lane][c];
}

// 64 rows below a block, a lane per row and a wave per rank, in the block
// kernel's order: at step k wave r takes column k - r, the rows' l pass from wave
// to wave in LDS.  A wave alone (all ranks of a column in turn, every operation
// waiting for the one before) took 37 us per launch, and 22 us with the columns
// and ranks in anti-diagonal order, and 13 us so; with a few thousand rows at most below a
// block, the eight waves per 64 rows still leave CUs free.
template <typename T>
__global__ __launch_bounds__(UD_THREADS) void k_updown_rows(const UdBlock *__restrict__ blocks,
                                                            const UdRows *__restrict__ rows, T *__restrict__ W,
                                                            const int *__restrict__ Ls, T *__restrict__ Wc,
                                                            const T *__restrict__ par) {
#pragma clang fp contract(off)
    __shared__ T X[NB][DS];                // X[c][row]
    __shared__ T Pw[UD_RANK][NB], Pg[UD_RANK][NB];
    const UdRows rr = rows[blockIdx.x];
    const UdBlock b = blocks[rr.blk];
    const T *ps = par + (long long)b.slot * NB * UD_PAR;
    const int tid = threadIdx.x, lane = tid & 63, nb = b.nb;
    const int r = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ii = rr.r0 + lane;
    const bool on = ii < b.nsrow;
    const int ir = min(ii, b.nsrow - 1);
    T *col = W + b.lx + (long long)b.c0 * b.nsrow + ir;
    int first = INT_MAX;                   // columns before every path are left alone
#pragma unroll
    for (int q = 0; q < UD_RANK; q++) first = min(first, b.start[q]);
    const int cfirst = max(first - b.c0, 0);
    const int start = blocks[rr.blk].start[r];
    constexpr int PER = NB / UD_RANK;
    T lnew[PER];
    T w;
    {
        // every load in flight, unconditional (a predicated one is a branch)
        T v[PER], lo[PER];
        const int pl = min(lane, nb - 1) * UD_PAR;
        const T pw = ps[pl + 2 + r], pg = ps[pl + 2 + UD_RANK + r];
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int c = min(r + UD_RANK * q, nb - 1);
            v[q] = col[(long long)c * b.nsrow];
            lo[q] = ps[c * UD_PAR];
            lnew[q] = ps[c * UD_PAR + 1];
        }
        const long long g = (long long)(ir < b.nscol ? b.k1 + ir : Ls[b.psi + ir]) * UD_RANK;
        w = Wc[g + r];
        Pw[r][lane] = pw;
        Pg[r][lane] = pg;
#pragma unroll
        for (int q = 0; q < PER; q++) X[r + UD_RANK * q][lane] = v[q] / lo[q];
    }
    __syncthreads();
    for (int k = cfirst; k < nb + UD_RANK - 1; k++) {
        const int c = k - r;
        if (c >= cfirst && c < nb && b.c0 + c >= start) {
            const T l = X[c][lane];
            w = w - Pw[r][c] * l;
            X[c][lane] = l - Pg[r][c] * w;
        }
        __syncthreads();
    }
    if (!on) return;
#pragma unroll
    for (int q = 0; q < PER; q++) {
        const int c = r + UD_RANK * q;
        if (c >= cfirst && c < nb) col[(long long)c * b.nsrow] = X[c][lane] * lnew[q];
    }
    if (start <= b.c0 + nb - 1) {
        const long long g = (long long)(ii < b.nscol ? b.k1 + ii : Ls[b.psi + ii]) * UD_RANK;
        Wc[g + r] = w;
    }
}

}  // namespace mxc
