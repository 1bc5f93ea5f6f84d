// kernels_factor.h -- device code of the numeric factorization (included once,
// by mxc_device.hip).
//
// Replaces, in one device-resident pass over a level schedule of the
// supernodal elimination tree:
//   * zero + scatter of A into the supernodes  (t_cholmod_super_numeric_worker.c:360-520)
//   * descendant SYRK/GEMM + relative-map scatter-subtract
//       (worker :769-930; GPU: t_cholmod_gpu.c:381-617, kernelAddUpdate
//        cholmod_gpu_kernels.cu:43-54)
//   * diagonal POTRF and panel TRSM (worker :1023-1027, :1175-1181;
//       GPU: t_cholmod_gpu.c:784-1135, :1151-1393)
#pragma once
#include "mxc_kernels.h"

namespace mxc {

// Row stride of a 64x64 diagonal block and its inverse in LDS: rows start on 16
// bytes (16-byte reads of a lane's row), and 16 rows 4 banks apart fill the 64
// banks.
constexpr int PS = NB + 2;

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct MfmaOp;
// Accumulator layout of the 16x16x4 MFMAs: lane l, register v holds
// D[row(l, v)][l % 16].  FP64 interleaves rows by 4 (row = l/16 + 4v); FP32
// keeps each lane's 4 rows contiguous (row = 4(l/16) + v).
template <> struct MfmaOp<double> {
    typedef f64x4 acc_t;
    static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <> struct MfmaOp<float> {
    typedef f32x4 acc_t;
    static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

__device__ __forceinline__ void atomic_sub(double *p, double v) { unsafeAtomicAdd(p, -v); }
__device__ __forceinline__ void atomic_sub(float *p, float v) { unsafeAtomicAdd(p, -v); }

// ---------------------------------------------------------------------------
// Assembly of A into L: Lx = 0; Lx[pos[p]] = Ax[p]; diagonal += beta.
// pos folds the fill-reducing permutation, so the values of tril(A) go in in
// their original order (no host-side P A P').
// ---------------------------------------------------------------------------
template <typename T>
__global__ void k_fill(T *__restrict__ p, long long n, T v) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

template <typename T>
__global__ void k_scatter_a(const double *__restrict__ Ax, const long long *__restrict__ pos,
                            long long nnz, T *__restrict__ W) {
    long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    long long stride = (long long)gridDim.x * blockDim.x;
    for (; p < nnz; p += stride) W[pos[p]] = (T)Ax[p];
}

// beta is read from device memory so that a captured factorization graph
// serves every beta
template <typename T>
__global__ void k_add_diag(const long long *__restrict__ dpos, long long n,
                           const double *__restrict__ beta, T *__restrict__ W,
                           double *__restrict__ adiag) {
    const double b = *beta;
    long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    T v = W[dpos[k]];
    if (b != 0.0) {
        v += (T)b;
        W[dpos[k]] = v;
    }
    adiag[k] = (double)v;           // assembled diagonal, for the pivot-ratio test
}

__global__ void k_set_int(int *p, int v) { *p = v; }

// Min / max of the diagonal of L (rcond diagnostic): each block writes
// (min, max, has_nan) of its share to out[3*blockIdx.x ...].
template <typename T>
__global__ void k_diag_minmax(const T *__restrict__ W, const long long *__restrict__ dpos, long long n,
                              double *__restrict__ out) {
    __shared__ double smin[256], smax[256];
    __shared__ int snan;
    if (threadIdx.x == 0) snan = 0;
    __syncthreads();
    double lo = INFINITY, hi = -INFINITY;
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (long long)gridDim.x * blockDim.x) {
        const double v = (double)W[dpos[k]];
        if (isnan(v)) snan = 1;
        lo = fmin(lo, v);
        hi = fmax(hi, v);
    }
    smin[threadIdx.x] = lo;
    smax[threadIdx.x] = hi;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            smin[threadIdx.x] = fmin(smin[threadIdx.x], smin[threadIdx.x + w]);
            smax[threadIdx.x] = fmax(smax[threadIdx.x], smax[threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[3 * blockIdx.x] = smin[0];
        out[3 * blockIdx.x + 1] = smax[0];
        out[3 * blockIdx.x + 2] = snan;
    }
}

// ---------------------------------------------------------------------------
// Dense TS x TS update tile on MFMA (see UpdDesc).  TS = 32: one wave owns the
// tile; TS = 64 / 128: four waves, each owning a (TS/2) x (TS/2) quarter, as
// (TS/32)^2 ... i.e. 2x2 or 4x4 blocks of 16x16 MFMA.  The larger tiles do more
// MFMA work per staged byte, which hides the global-load latency of the next
// K chunk (prefetched into registers while the current chunk computes from
// the other LDS buffer).  The MFMA is fed X (C-column side) as its A operand
// and Y (C-row side) as its B operand, so 16 consecutive lanes hold 16
// consecutive C rows: stores into the column-major target are contiguous runs.
// ---------------------------------------------------------------------------
// Workgroup b of a launch is dispatched to XCD b % 8.  Tiles are dealt to
// the XCDs in chunks of 8 consecutive list entries instead (round robin over
// chunks), so the tiles of a chunk, which share an operand strip, run on one
// XCD and share its L2, while the chunks still spread evenly over the XCDs.
// The tail that does not fill a round of 8 chunks keeps its own order.
__device__ __forceinline__ int xcd_tile(int b, int g) {
    constexpr int C = 8;
    const int full = g / (8 * C) * (8 * C);
    if (b >= full) return b;
    const int x = b & 7, k = b >> 3;
    return (x + 8 * (k / C)) * C + (k % C);
}

// Split-FP16 form of the FP32 factor (see k_tile_h): the scale exponent of
// global row g, s_g = 13 - floor(log2 sqrt(a_gg)), and the packed pair
// (hi | lo << 16) of a value v of that row, hi = fp16(v 2^s), lo = fp16(v 2^s - hi).
__device__ __forceinline__ int row_scale_exp(const double *__restrict__ adiag, int g) {
    const double a = adiag[g];
    if (!(a > 0.0) || !(a < 1e300)) return 0;
    return min(max(13 - ilogb(sqrt(a)), -100), 100);
}

__device__ __forceinline__ unsigned split_pack(float v, int e) {
    const float sv = v * ldexpf(1.0f, e);
    const _Float16 hi = (_Float16)sv;
    const _Float16 lo = (_Float16)(sv - (float)hi);
    return (unsigned)__builtin_bit_cast(unsigned short, hi) |
           ((unsigned)__builtin_bit_cast(unsigned short, lo) << 16);
}

// FP64 redo of the diagonal blocks of a low-precision factor whose pivot ratio
// signals breakdown (a pivot at or below rho * a_jj).  cnt: [0] blocks queued
// since the last k_potrf_redo64 launch, [1] blocks refactored in FP64 in this
// factorization, [2] redo workgroups finished (queue clearing).  The rest
// finds A's own entries of a block: the full CSR of A in the original order,
// its values (refreshed every factorization), Perm, the inverse permutation
// and beta.
struct Redo {
    int *cnt;
    DiagTask *list;
    const long long *rowptr;
    const int *col;
    const double *vals;
    const long long *perm;
    const int *pinv;
    const double *beta;
};

__device__ __forceinline__ void redo_push(const Redo &rd, const DiagTask &t) {
    const int k = atomicAdd(rd.cnt, 1);
    rd.list[k] = t;
}

// Refactor diagonal block t in FP64 with the nt threads tid < nt of the
// caller (sync() is their barrier), in place of its low-precision result:
//   1. A64 = the block as assembled in W (A's values in T minus the descendant
//      and earlier-step updates accumulated in T), in FP64, with A's own
//      entries swapped for their FP64 values (+ beta on the diagonal):
//      A64 = W + (A - fl_T(A)).  Column Perm[col0 + c] of A's CSR holds, among
//      its neighbours, the rows whose permuted index falls in the block;
//   2. right-looking Cholesky of A64 in FP64 (a pivot <= 0 is reported as the
//      failing column, as CHOLMOD reports it), L written to W in T;
//   3. inv(L) in place, last column first (column j from the columns right
//      of it: X_ij = -X_jj sum_{k=j+1..i} X_ik L_kj), written to W in T.
// A: NB x (NB + 1) doubles, tmp: NB doubles, sbad: one int (all in LDS).
template <typename T, typename Sync>
__device__ __forceinline__ void redo_block64(const DiagTask &t, T *__restrict__ W, double *A, double *tmp,
                                             int *sbad, int tid, int nt, const Redo &rd,
                                             int *__restrict__ fail, Sync sync) {
    constexpr int LD = NB + 1;
    const int nb = t.nb;
    for (int q = tid; q < nb * nb; q += nt) {
        const int i = q % nb, c = q / nb;
        A[i * LD + c] = (c <= i) ? (double)W[t.off + i + (long long)c * t.ld] : 0.0;
    }
    if (tid == 0) *sbad = -1;
    sync();
    const double b = *rd.beta;
    const int per = nt >= 4 * nb ? 4 : 1;           // threads per column (distinct rows each)
    for (int c = tid / per; c < nb; c += nt / per) {
        const long long o = rd.perm[t.col0 + c];
        for (long long q = rd.rowptr[o] + (tid % per); q < rd.rowptr[o + 1]; q += per) {
            const int i = rd.pinv[rd.col[q]] - t.col0;
            if (i < c || i >= nb) continue;
            const double a = rd.vals[q];
            T a_t = (T)a;                           // what the assembly stored (k_scatter_a, k_add_diag)
            double a64 = a;
            if (i == c && b != 0.0) {
                a_t += (T)b;
                a64 += b;
            }
            A[i * LD + c] += a64 - (double)a_t;
        }
    }
    sync();
    for (int j = 0; j < nb; j++) {
        double d = A[j * LD + j];
        if (!(d > 0.0)) {
            if (tid == 0 && *sbad < 0) *sbad = j;
            d = 1.0;
        }
        const double r = 1.0 / sqrt(d);
        sync();                                     // every thread has read the pivot
        if (tid == 0) A[j * LD + j] = d * r;
        for (int i = j + 1 + tid; i < nb; i += nt) A[i * LD + j] *= r;
        sync();
        const int m = nb - j - 1;
        for (int q = tid; q < m * m; q += nt) {
            const int i = j + 1 + q % m, c = j + 1 + q / m;
            if (c <= i) A[i * LD + c] -= A[i * LD + j] * A[c * LD + j];
        }
        sync();
    }
    for (int q = tid; q < nb * nb; q += nt) {
        const int i = q % nb, c = q / nb;
        if (c <= i) W[t.off + i + (long long)c * t.ld] = (T)A[i * LD + c];
    }
    sync();
    for (int j = nb - 1; j >= 0; j--) {
        if (tid == 0) A[j * LD + j] = 1.0 / A[j * LD + j];
        for (int i = j + 1 + tid; i < nb; i += nt) tmp[i] = A[i * LD + j];
        sync();
        const double xjj = -A[j * LD + j];
        for (int i = j + 1 + tid; i < nb; i += nt) {
            double acc = 0.0;
            for (int k = j + 1; k <= i; k++) acc += A[i * LD + k] * tmp[k];
            A[i * LD + j] = xjj * acc;
        }
        sync();
    }
    for (int q = tid; q < nb * nb; q += nt) {
        const int i = q % nb, c = q / nb;
        W[t.winv + i + (long long)c * nb] = (c <= i) ? (T)A[i * LD + c] : (T)0;
    }
    if (tid == 0) {
        if (*sbad >= 0) atomicMin(fail, t.col0 + *sbad);
        atomicAdd(rd.cnt + 1, 1);
    }
}

// Where potrf_core keeps block (i, j), i >= j, of the inverse, in elements from
// its block S.  FP64: off-diagonal blocks take the place of S's unused blocks
// (j, i), diagonal ones stand side by side in 16 rows below S: 42 KB, so that
// three workgroups of a trailing kernel with tails share a CU instead of two
// (64^3 diffusion factor 14.99 -> 14.75 ms, 80^3 27-point 52.7 -> 52.0 ms).
// FP32, whose FP64 redo needs the 33 KB anyway: a square of its own below S
// (its addresses are cheaper: 41^3 factor 2.75 ms, 2.80 ms in FP64's places).
template <typename T>
__device__ __forceinline__ int inv_at(int i, int j) {
    if (std::is_same<T, float>::value) return (NB + 16 * i) * PS + 16 * j;
    return i == j ? NB * PS + 16 * i : 16 * j * PS + 16 * i;
}

// LDS of potrf_block, in bytes: the block and its inverse, and with `redo` at
// least the FP64 redo's block.
template <typename T>
constexpr size_t potrf_lds(bool redo) {
    const size_t own = sizeof(T) * (std::is_same<T, float>::value ? 2 * NB : NB + 16) * PS;
    const size_t r64 = redo ? sizeof(double) * NB * (NB + 1) : 0;
    return own > r64 ? own : r64;
}

template <typename T, bool SAFE, bool LOADED = false>
__device__ __forceinline__ void potrf_block(const DiagTask &t, T *__restrict__ W, T *S, int *sfail,
                                            int *__restrict__ fail, const double *__restrict__ adiag,
                                            double rho, const Redo &rd, double *tmp);

// Arguments of the diagonal-block tail of a trailing launch (PD): after its
// epilogue, the workgroup of tile (0, 0) of a block with pd >= 0 has the final
// values of the next step's diagonal block and factors it (potrf_block).
//
// With a folded TRSM (UpdDesc::fold) the tail publishes the factored block:
// ready[pd] is set once its L and inverse are in W (a device-scope release
// of every wave after its stores), and the tiles of column 0 below it wait for
// that flag (device-scope acquire) before applying the inverse.  Producer
// tiles come first in the launch (the first nfirst workgroups map to tiles
// 0 .. nfirst-1, which hold them) and never wait, and workgroups start in
// index order, so every wait ends; a wait is still bounded (FOLD_SPIN polls),
// past which it raises *abort and the host reports a device error.
struct PdArgs {
    const DiagTask *diags;
    int *fail;
    double rho;
    Redo rd;
    int *ready;        // per diagonal task: 1 once a folding tail has published it
    int *abort;        // set by a wait that gave up
    int nfirst;        // producer tiles at the head of the launch (no XCD remap)
};

constexpr int FOLD_SPIN = 1 << 22;

// The tail itself: potrf_block in the tile's LDS buffer.
// LOADED: the tile's epilogue has put the block into S (tail_entry); else it is
// read back from W.
template <typename T, bool LOADED>
__device__ __forceinline__ void pd_tail(const PdArgs &pda, int pd, T *__restrict__ W, unsigned char *smem,
                                        const double *__restrict__ adiag, bool publish) {
    __shared__ int sfail[2];
    __syncthreads();                        // the tile's stores and LDS reads are done
    T *S = reinterpret_cast<T *>(smem);
    if (pda.rho > 0) {
        __shared__ double tmp[NB];
        potrf_block<T, true, LOADED>(pda.diags[pd], W, S, sfail, pda.fail, adiag, pda.rho, pda.rd, tmp);
    } else {
        potrf_block<T, false, LOADED>(pda.diags[pd], W, S, sfail, pda.fail, adiag, pda.rho, pda.rd, nullptr);
    }
    if (publish) {
        // every wave waits for its own stores of L and the inverse: the release of the
        // flag's store orders those of thread 0's wave only
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __syncthreads();
        if (threadIdx.x == 0) __hip_atomic_store(pda.ready + pd, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Entry (i, j) of the block that a tail factors (nb columns, extended by the
// identity), a its value in the trailing tile.
template <typename T>
__device__ __forceinline__ T tail_entry(int i, int j, int nb, T a) {
    return i < nb && j < nb ? (j <= i ? a : (T)0) : (i == j ? (T)1 : (T)0);
}

// Wait (whole workgroup) until *flag != 0 or the wait gives up.
__device__ __forceinline__ void fold_wait(const int *flag, int *abort) {
    if ((threadIdx.x & 63) == 0) {
        for (int it = 1; __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0; it++) {
            __builtin_amdgcn_s_sleep(1);
            if ((it & 63) == 0 &&
                (it >= FOLD_SPIN || __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
                __hip_atomic_store(abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");   // the inverse's loads come after the flag
    __syncthreads();
}

// One tile of a launch: virtual workgroup bx of g (k_tile: the workgroup
// itself; k_tile_grid: each of its workgroups takes bx, bx + grid, ...).
template <typename T, int MODE, int TS, bool PD, bool FOLD>
__device__ __forceinline__ void tile_work(const UpdDesc *__restrict__ descs, const Tile *__restrict__ tiles,
                                          T *__restrict__ W, const int *__restrict__ Ls, unsigned *__restrict__ Lh,
                                          const double *__restrict__ adiag, const PdArgs &pda, const int bx,
                                          const int g) {
    typedef typename MfmaOp<T>::acc_t acc_t;
    constexpr int NT = TS <= 32 ? 64 : 256;     // threads (tiles of 16 and 32: one wave)
    constexpr int WB = TS <= 32 ? TS : TS / 2;  // edge of a wave's block of C
    constexpr int MB = WB / 16;                 // 16x16 MFMA blocks per wave edge
    constexpr int KG = NT / TS;                 // k rows staged per pass
    constexpr int PER = (BK * TS) / NT;         // elements of X (and of Y) each thread stages
    static_assert(!PD || (MODE == MODE_TRAIL && TS >= 64), "diagonal tails: trailing tiles of 64 or 128");
    // one LDS buffer: the staged X / Y chunks, reused by the diagonal-block tail.
    // Tiles of 32 and 64 stage into a single buffer: the extra barrier per
    // chunk costs less than the resident tiles that half the LDS adds (64³ FP64
    // update kernel 28.1 -> 30.2 TFLOP/s); a 128 tile is register-bound at two
    // waves per SIMD either way and keeps two buffers.
    constexpr int NBUF = TS == 128 ? 2 : 1;
    constexpr size_t XY_BYTES = sizeof(T) * NBUF * BK * (TS + LDS_PAD);
    constexpr size_t PD_BYTES = PD ? potrf_lds<T>(std::is_same<T, float>::value) : 0;
    // folded TRSM (FP64, 64-wide trailing tiles): the updated block and the
    // next diagonal block's inverse, both k-major like the staged chunks
    // (a variant of its own: its buffers, 69 KB, leave room for two workgroups per
    // CU, the tail's 42 KB for three)
    constexpr bool CAN_FOLD = FOLD;
    static_assert(!FOLD || (PD && TS == NB && std::is_same<T, double>::value), "folded TRSM: FP64 tails");
    constexpr size_t FOLD_HALF = sizeof(T) * NB * (TS + LDS_PAD);
    constexpr size_t FOLD_BYTES = CAN_FOLD ? 2 * FOLD_HALF : 0;
    constexpr size_t SMEM0 = 2 * XY_BYTES > PD_BYTES ? 2 * XY_BYTES : PD_BYTES;
    constexpr size_t SMEM = SMEM0 > FOLD_BYTES ? SMEM0 : FOLD_BYTES;
    __shared__ __attribute__((aligned(16))) unsigned char smem[SMEM];
    T (*Xs)[BK][TS + LDS_PAD] = reinterpret_cast<T (*)[BK][TS + LDS_PAD]>(smem);
    T (*Ys)[BK][TS + LDS_PAD] = reinterpret_cast<T (*)[BK][TS + LDS_PAD]>(smem + XY_BYTES);
    __shared__ int relr[TS];
    __shared__ int relc[TS];

    const int nf = FOLD ? pda.nfirst : 0;
    const Tile tl = tiles[bx < nf ? bx : nf + xcd_tile(bx - nf, g - nf)];
    const UpdDesc d = descs[tl.desc];
    const int i0 = tl.ti * TS, j0 = tl.tj * TS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = TS <= 32 ? 0 : (wave & 1), wc = TS <= 32 ? 0 : (wave >> 1);
    const bool tail = PD && d.pd >= 0 && tl.ti == 0 && tl.tj == 0;   // factors the next diagonal block
    if (tail) __builtin_amdgcn_s_setprio(3);    // on the critical path: ahead of the CU's other tiles

    // thread t stages row r = t % TS of chunk rows k = t/TS + KG*q, q < PER.  The
    // loads are unconditional (rows and k clamped into the block, a predicated
    // load is a branch each): rows past the block's edge give entries of C that
    // are not stored, and columns past K are staged as zeros.  k is the same for
    // a whole wave in the four-wave tiles.
    const T *__restrict__ Xp = W + d.x_off;
    const T *__restrict__ Yp = W + d.y_off;
    const int r = tid % TS;
    const int kq = TS >= 64 ? __builtin_amdgcn_readfirstlane(tid / TS) : tid / TS;
    const unsigned yo = (unsigned)min(i0 + r, d.M - 1) * (unsigned)sizeof(T);
    const unsigned xo = (unsigned)min(j0 + r, d.N - 1) * (unsigned)sizeof(T);
    auto at = [](const T *p, unsigned o) {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + o);
    };
    T ry[PER], rx[PER];
    auto fetch = [&](int k0) {
        if (k0 + BK <= d.K) {
#pragma unroll
            for (int q = 0; q < PER; q++) {
                ry[q] = at(Yp + (long long)(k0 + kq + KG * q) * d.ldy, yo);
                rx[q] = at(Xp + (long long)(k0 + kq + KG * q) * d.ldx, xo);
            }
        } else {
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int gk = min(k0 + kq + KG * q, d.K - 1);
                const bool kin = k0 + kq + KG * q < d.K;
                const T y = at(Yp + (long long)gk * d.ldy, yo), x = at(Xp + (long long)gk * d.ldx, xo);
                ry[q] = kin ? y : (T)0;
                rx[q] = kin ? x : (T)0;
            }
        }
    };
    fetch(0);                                   // in flight during the search below

    if (MODE == MODE_SCATTER) {
        for (int e = tid; e < 2 * TS; e += NT) {
            if (e < TS) {
                int i = i0 + e;
                int r = -1;
                if (i < d.M) {
                    int g = Ls[d.ls_off + i];
                    if (g < d.base + d.t_nscol) {
                        r = g - d.base;
                    } else {
                        int lo = d.t_psi + d.t_nscol, hi = d.t_psi + d.t_nsrow - 1;
                        while (lo < hi) {
                            int mid = (lo + hi) >> 1;
                            if (Ls[mid] < g) lo = mid + 1; else hi = mid;
                        }
                        r = lo - d.t_psi;
                    }
                }
                relr[e] = r;
            } else {
                int j = j0 + e - TS;
                relc[e - TS] = (j < d.N) ? (Ls[d.ls_off + j] - d.base) : -1;
            }
        }
    }

    acc_t acc[MB][MB];
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
        for (int b = 0; b < MB; b++) acc[a][b] = acc_t{0, 0, 0, 0};

    // trailing tiles: the entries of C, loaded together and unconditionally, clamped
    // into the block (a predicated read-modify-write each waited for its own round
    // trip).  A launch with tails waits for its diagonal tile, so there the loads go
    // under the last chunk's products; elsewhere, and in tiles of 128, a row of MFMA
    // blocks at a time in the epilogue, which leaves the registers for another
    // resident tile (80^3 27-point FP64 pass 56.1 ms, 58.4 ms with all ahead).  FP32
    // factor 28.9 -> 27.4 ms at 80^3 27-point, 2.95 -> 2.74 ms at 41^3; FP64
    // 15.06 -> 14.94 ms at 64^3.
    constexpr int OM = MODE != MODE_TRAIL ? 0 : PD && MB <= 2 ? MB : 1;
    T old[OM > 0 ? OM : 1][MB][4];
    auto load_c = [&](int m, int o) {
#pragma unroll
        for (int n = 0; n < MB; n++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                old[o][n][v] = W[d.c_off + (long long)min(j0 + wc * WB + m * 16 + MfmaOp<T>::row(lane, v), d.N - 1) * d.ldc +
                                 min(i0 + wr * WB + n * 16 + (lane & 15), d.M - 1)];
    };

    int buf = 0;
    for (int k0 = 0; k0 < d.K; k0 += BK) {
        if (NBUF == 1 && k0 > 0) __syncthreads();   // the previous chunk's reads are done
#pragma unroll
        for (int q = 0; q < PER; q++) {
            Ys[buf][kq + KG * q][r] = ry[q];
            Xs[buf][kq + KG * q][r] = rx[q];
        }
        __syncthreads();
        if (k0 + BK < d.K) {
            fetch(k0 + BK);                     // next chunk in flight during the MFMAs
        } else if constexpr (OM > 1) {
#pragma unroll
            for (int m = 0; m < OM; m++) load_c(m, m);
        }
        // operands one step ahead: their LDS latency passes under the MFMAs
        // (with the unconditional loads, one 64-wide FP64 launch over 6000 x 5600,
        // K = 384: 55.5 -> 60.5 TFLOP/s; a chunk alone on its CU 2,190 -> 1,920
        // cycles, of which the MFMAs take 1,024)
        T xa[2][MB], yb[2][MB];
        auto operands = [&](int kk, T (&x)[MB], T (&y)[MB]) {
#pragma unroll
            for (int m = 0; m < MB; m++) x[m] = Xs[buf][kk + (lane >> 4)][wc * WB + m * 16 + (lane & 15)];
#pragma unroll
            for (int n = 0; n < MB; n++) y[n] = Ys[buf][kk + (lane >> 4)][wr * WB + n * 16 + (lane & 15)];
        };
        operands(0, xa[0], yb[0]);
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            const int c = (kk >> 2) & 1;
            if (kk + 4 < BK) operands(kk + 4, xa[c ^ 1], yb[c ^ 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < MB; m++)
#pragma unroll
                for (int n = 0; n < MB; n++) acc[m][n] = MfmaOp<T>::mma(xa[c][m], yb[c][n], acc[m][n]);
        }
        if constexpr (NBUF == 2) buf ^= 1;
    }
    if (MODE == MODE_STORE) __syncthreads();   // in-place TRSM: every read of the panel is done
    const bool fold = CAN_FOLD && d.fold && d.pd >= 0 && tl.tj == 0 && tl.ti >= 1;
    T (*Af)[TS + LDS_PAD] = reinterpret_cast<T (*)[TS + LDS_PAD]>(smem);               // Af[k][i]
    T (*If)[TS + LDS_PAD] = reinterpret_cast<T (*)[TS + LDS_PAD]>(smem + FOLD_HALF);   // If[k][j]
    // the tail's block goes to LDS as well as to W
    constexpr bool TAIL_LDS = PD && TS == NB;
    T *S = reinterpret_cast<T *>(smem);
    const int tail_nb = TAIL_LDS && tail ? pda.diags[d.pd].nb : 0;
    if ((CAN_FOLD && fold) || (TAIL_LDS && tail)) __syncthreads();   // every wave is done with the staged chunks

    // FP32 TRSM with Lh: the panel is also stored in split-FP16 form, each row
    // scaled by its own exponent, for the update and trailing tiles that read it
    int exs[MB];
#pragma unroll
    for (int n = 0; n < MB; n++) exs[n] = 0;
    if (MODE == MODE_STORE && std::is_same<T, float>::value && Lh) {
#pragma unroll
        for (int n = 0; n < MB; n++) {
            const int i = i0 + wr * WB + n * 16 + (lane & 15);
            if (i < d.M) exs[n] = row_scale_exp(adiag, Ls[d.ls_off + i]);
        }
    }

    // epilogue: acc[m][n][v] = C(i, j), i = i0 + WB*wr + 16n + lane%16,
    //                                   j = j0 + WB*wc + 16m + row(lane, v)
#pragma unroll
    for (int m = 0; m < MB; m++) {
        if constexpr (OM == 1) load_c(m, 0);
#pragma unroll
        for (int n = 0; n < MB; n++) {
            const int il = wr * WB + n * 16 + (lane & 15);
            const int i = i0 + il;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int jl = wc * WB + m * 16 + MfmaOp<T>::row(lane, v);
                const int j = j0 + jl;
                const T c = acc[m][n][v];
                if (TAIL_LDS && tail) S[il * PS + jl] = tail_entry(il, jl, tail_nb, old[OM > 1 ? m : 0][n][v] - c);
                if (i >= d.M || j >= d.N) continue;
                if (MODE == MODE_SCATTER) {
                    if (i < j) continue;
                    atomic_sub(W + d.c_off + (long long)relc[jl] * d.ldc + relr[il], c);
                } else if (MODE == MODE_TRAIL) {
                    if (i < j) continue;
                    const T a = old[OM > 1 ? m : 0][n][v] - c;
                    if (CAN_FOLD && fold) Af[jl][il] = a;        // the next TRSM's input, kept here
                    else W[d.c_off + (long long)j * d.ldc + i] = a;
                } else {
                    W[d.c_off + (long long)j * d.ldc + i] = c;
                    if (std::is_same<T, float>::value && Lh)
                        Lh[d.c_off + (long long)j * d.ldc + i] = split_pack((float)c, exs[n]);
                }
            }
        }
    }
    if constexpr (CAN_FOLD) {
        if (fold) {
            // the next step's TRSM of these rows: L(i, j) = sum_k A(i, k) inv(j, k),
            // with the MFMA sequence of the TRSM tile (k ascending)
            const DiagTask dt = pda.diags[d.pd];
            fold_wait(pda.ready + d.pd, pda.abort);
            for (int e = tid; e < NB * NB; e += NT) If[e / NB][e % NB] = W[dt.winv + e];
            __syncthreads();
            acc_t a2[MB][MB];
#pragma unroll
            for (int a = 0; a < MB; a++)
#pragma unroll
                for (int b = 0; b < MB; b++) a2[a][b] = acc_t{0, 0, 0, 0};
#pragma unroll 4
            for (int kk = 0; kk < NB; kk += 4) {
                T xa[MB], yb[MB];
#pragma unroll
                for (int m = 0; m < MB; m++) xa[m] = If[kk + (lane >> 4)][wc * WB + m * 16 + (lane & 15)];
#pragma unroll
                for (int n = 0; n < MB; n++) yb[n] = Af[kk + (lane >> 4)][wr * WB + n * 16 + (lane & 15)];
#pragma unroll
                for (int m = 0; m < MB; m++)
#pragma unroll
                    for (int n = 0; n < MB; n++) a2[m][n] = MfmaOp<T>::mma(xa[m], yb[n], a2[m][n]);
            }
#pragma unroll
            for (int m = 0; m < MB; m++) {
#pragma unroll
                for (int n = 0; n < MB; n++) {
                    const int i = i0 + wr * WB + n * 16 + (lane & 15);
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const int j = wc * WB + m * 16 + MfmaOp<T>::row(lane, v);
                        if (i < d.M) W[d.c_off + (long long)j * d.ldc + i] = a2[m][n][v];
                    }
                }
            }
        }
    }
    if constexpr (PD) {
        if (tail) pd_tail<T, TAIL_LDS>(pda, d.pd, W, smem, adiag, d.fold != 0);
    }
}

template <typename T, int MODE, int TS, bool PD = false, bool FOLD = false>
__global__ __launch_bounds__(TS <= 32 ? 64 : 256, TS == 128 ? 2 : 1) void k_tile(const UpdDesc *__restrict__ descs,
                                                              const Tile *__restrict__ tiles,
                                                              T *__restrict__ W,
                                                              const int *__restrict__ Ls,
                                                              unsigned *__restrict__ Lh,
                                                              const double *__restrict__ adiag,
                                                              PdArgs pda = PdArgs{}) {
    tile_work<T, MODE, TS, PD, FOLD>(descs, tiles, W, Ls, Lh, adiag, pda, (int)blockIdx.x, (int)gridDim.x);
}

// The tiles of a launch on a grid of at most a few workgroups per CU (a
// multiple of 8, so a workgroup's tiles keep its XCD): the second-stream
// trailing update under MXC_OPT_T2_GRID, which leaves room on every CU for
// the main stream's launches.
template <typename T, int MODE, int TS>
__global__ __launch_bounds__(256, 1) void k_tile_grid(const UpdDesc *__restrict__ descs,
                                                      const Tile *__restrict__ tiles, T *__restrict__ W,
                                                      const int *__restrict__ Ls, const double *__restrict__ adiag,
                                                      int ntiles) {
    static_assert(TS >= 64, "four-wave tiles");
    for (int b = (int)blockIdx.x; b < ntiles; b += (int)gridDim.x) {
        tile_work<T, MODE, TS, false, false>(descs, tiles, W, Ls, nullptr, adiag, PdArgs{}, b, ntiles);
        __syncthreads();                   // the next tile restages the LDS buffers
    }
}

// ---------------------------------------------------------------------------
// FP32 factor, split-FP16 products (update and trailing blocks).  An FP32
// value v of L in global row g is scaled by 2^s_g, s_g = 13 - floor(log2
// sqrt(a_gg)) with a_gg the assembled diagonal of A (|L_gk| <= sqrt(a_gg), so
// the scaled values stay below 2^14), and split into hi = fp16(v 2^s) and
// lo = fp16(v 2^s - hi).  The TRSM that finalizes a value writes the pair
// once into Lh (same layout as L), so the tiles here stage the halves as they
// are.  C = Y X' accumulates hi*hi + hi*lo + lo*hi in FP32 on the 16x16x32
// FP16 MFMA (lo*lo lies below FP32 rounding relative to the row norms) and is
// unscaled by 2^-(s_i + s_j) in the epilogue, which is the one of k_tile.
// One LDS buffer of hi / lo rows, k contiguous, row stride 40 halves (the
// 16-byte reads of a 16-row group fall in distinct banks); the next chunk is
// prefetched into registers.
// ---------------------------------------------------------------------------
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

template <int MODE, int TS, bool PD = false>
__global__ __launch_bounds__(256, 2) void k_tile_h(const UpdDesc *__restrict__ descs,
                                                                  const Tile *__restrict__ tiles,
                                                                  float *__restrict__ W,
                                                                  const unsigned *__restrict__ Lh,
                                                                  const int *__restrict__ Ls,
                                                                  const double *__restrict__ adiag,
                                                                  PdArgs pda = PdArgs{}) {
    static_assert(TS == 64 || TS == 128, "split-FP16 tiles are 64 or 128 wide");
    constexpr int NT = 256;              // 2 x 2 waves
    constexpr int WB = TS / 2;           // edge of a wave's block of C
    constexpr int MB = WB / 16;
    constexpr int BKH = 32;              // K per chunk: one MFMA depth
    constexpr int RS = BKH + 8;          // LDS row stride (halves)
    constexpr int KG = NT / TS;          // staging threads per row
    constexpr int PER = BKH / KG;        // consecutive k per staging thread
    static_assert(!PD || (MODE == MODE_TRAIL && TS >= 64), "diagonal tails: trailing tiles of 64 or 128");
    // one LDS buffer: the staged halves, reused by the diagonal-block tail
    constexpr size_t H_BYTES = 4 * sizeof(_Float16) * TS * RS;
    constexpr size_t PD_BYTES = PD ? potrf_lds<float>(true) : 0;
    __shared__ __attribute__((aligned(16))) unsigned char smem[H_BYTES > PD_BYTES ? H_BYTES : PD_BYTES];
    _Float16 *Xh = reinterpret_cast<_Float16 *>(smem);
    _Float16 *Xl = Xh + TS * RS;
    _Float16 *Yh = Xl + TS * RS;
    _Float16 *Yl = Yh + TS * RS;
    __shared__ int relr[TS], relc[TS];
    __shared__ int exr[TS], exc[TS];     // scale exponents of the Y rows (i) and X rows (j)

    const Tile tl = tiles[xcd_tile((int)blockIdx.x, (int)gridDim.x)];
    const UpdDesc d = descs[tl.desc];
    const int i0 = tl.ti * TS, j0 = tl.tj * TS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = wave & 1, wc = wave >> 1;
    const bool tail = PD && d.pd >= 0 && tl.ti == 0 && tl.tj == 0;   // as in tile_work
    if (tail) __builtin_amdgcn_s_setprio(3);

    for (int e = tid; e < 2 * TS; e += NT) {
        if (e < TS) {
            const int i = i0 + e;
            int r = -1, ex = 0;
            if (i < d.M) {
                const int g = Ls[d.ls_off + i];
                ex = row_scale_exp(adiag, g);
                if (MODE == MODE_SCATTER) {
                    if (g < d.base + d.t_nscol) {
                        r = g - d.base;
                    } else {
                        int lo = d.t_psi + d.t_nscol, hi = d.t_psi + d.t_nsrow - 1;
                        while (lo < hi) {
                            int mid = (lo + hi) >> 1;
                            if (Ls[mid] < g) lo = mid + 1; else hi = mid;
                        }
                        r = lo - d.t_psi;
                    }
                }
            }
            relr[e] = r;
            exr[e] = ex;
        } else {
            const int j = j0 + e - TS;
            int c = -1, ex = 0;
            if (j < d.N) {
                const int g = Ls[d.ls_off + j];
                ex = row_scale_exp(adiag, g);
                c = g - d.base;
            }
            relc[e - TS] = c;
            exc[e - TS] = ex;
        }
    }
    __syncthreads();

    // staging: thread t holds row r = t % TS, k in [kq * PER, kq * PER + PER) of a chunk
    // (unconditional loads, rows and k clamped; columns past K staged as zeros)
    const int r = tid % TS, kq = __builtin_amdgcn_readfirstlane(tid / TS);
    const int yr = min(i0 + r, d.M - 1), xr = min(j0 + r, d.N - 1);
    const unsigned *Yp = Lh + d.y_off, *Xp = Lh + d.x_off;
    unsigned ry[PER], rx[PER];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int gk = min(k0 + kq * PER + q, d.K - 1);
            ry[q] = Yp[(long long)gk * d.ldy + yr];
            rx[q] = Xp[(long long)gk * d.ldx + xr];
        }
    };
    auto half_of = [](unsigned u) { return __builtin_bit_cast(_Float16, (unsigned short)(u & 0xffffu)); };
    auto stage = [&](int k0) {
        if (k0 + BKH > d.K) {
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const bool kin = k0 + kq * PER + q < d.K;
                ry[q] = kin ? ry[q] : 0u;
                rx[q] = kin ? rx[q] : 0u;
            }
        }
#pragma unroll
        for (int h = 0; h < PER; h += 8) {
            half8_t yh, yl, xh, xl;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                yh[q] = half_of(ry[h + q]);
                yl[q] = half_of(ry[h + q] >> 16);
                xh[q] = half_of(rx[h + q]);
                xl[q] = half_of(rx[h + q] >> 16);
            }
            const int o = r * RS + kq * PER + h;
            *reinterpret_cast<half8_t *>(&Yh[o]) = yh;
            *reinterpret_cast<half8_t *>(&Yl[o]) = yl;
            *reinterpret_cast<half8_t *>(&Xh[o]) = xh;
            *reinterpret_cast<half8_t *>(&Xl[o]) = xl;
        }
    };

    f32x4 acc[MB][MB];
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
        for (int b = 0; b < MB; b++) acc[a][b] = f32x4{0, 0, 0, 0};

    // the entries of C, as in tile_work
    constexpr int OM = MODE != MODE_TRAIL ? 0 : PD && MB <= 2 ? MB : 1;
    float old[OM > 0 ? OM : 1][MB][4];
    auto load_c = [&](int m, int o) {
#pragma unroll
        for (int n = 0; n < MB; n++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                old[o][n][v] = W[d.c_off + (long long)min(j0 + wc * WB + m * 16 + 4 * (lane >> 4) + v, d.N - 1) * d.ldc +
                                 min(i0 + wr * WB + n * 16 + (lane & 15), d.M - 1)];
    };

    fetch(0);
    const int ko = 8 * (lane >> 4);
    for (int k0 = 0; k0 < d.K; k0 += BKH) {
        __syncthreads();                         // the previous chunk's reads are done
        stage(k0);
        __syncthreads();
        if (k0 + BKH < d.K) {
            fetch(k0 + BKH);                     // next chunk in flight during the MFMAs
        } else if constexpr (OM > 1) {
#pragma unroll
            for (int m = 0; m < OM; m++) load_c(m, m);
        }
        half8_t xh[MB], xl[MB], yh[MB], yl[MB];
#pragma unroll
        for (int m = 0; m < MB; m++) {
            const int o = (wc * WB + m * 16 + (lane & 15)) * RS + ko;
            xh[m] = *reinterpret_cast<const half8_t *>(&Xh[o]);
            xl[m] = *reinterpret_cast<const half8_t *>(&Xl[o]);
        }
#pragma unroll
        for (int n = 0; n < MB; n++) {
            const int o = (wr * WB + n * 16 + (lane & 15)) * RS + ko;
            yh[n] = *reinterpret_cast<const half8_t *>(&Yh[o]);
            yl[n] = *reinterpret_cast<const half8_t *>(&Yl[o]);
        }
#pragma unroll
        for (int m = 0; m < MB; m++)
#pragma unroll
            for (int n = 0; n < MB; n++) {
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[m], yh[n], acc[m][n], 0, 0, 0);
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[m], yl[n], acc[m][n], 0, 0, 0);
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[m], yh[n], acc[m][n], 0, 0, 0);
            }
    }

    // epilogue: acc[m][n][v] = C(i, j) 2^(s_i + s_j), i = i0 + WB*wr + 16n + lane%16,
    //                                               j = j0 + WB*wc + 16m + 4 (lane/16) + v
    constexpr bool TAIL_LDS = PD && TS == NB;
    float *S = reinterpret_cast<float *>(smem);
    const int tail_nb = TAIL_LDS && tail ? pda.diags[d.pd].nb : 0;
    if (TAIL_LDS && tail) __syncthreads();       // every wave is done with the staged chunks
#pragma unroll
    for (int m = 0; m < MB; m++) {
        if constexpr (OM == 1) load_c(m, 0);
#pragma unroll
        for (int n = 0; n < MB; n++) {
            const int il = wr * WB + n * 16 + (lane & 15);
            const int i = i0 + il;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int jl = wc * WB + m * 16 + 4 * (lane >> 4) + v;
                const int j = j0 + jl;
                const float c = ldexpf(acc[m][n][v], -(exr[il] + exc[jl]));
                if (TAIL_LDS && tail) S[il * PS + jl] = tail_entry(il, jl, tail_nb, old[OM > 1 ? m : 0][n][v] - c);
                if (i >= d.M || j >= d.N || i < j) continue;
                if (MODE == MODE_SCATTER)
                    atomic_sub(W + d.c_off + (long long)relc[jl] * d.ldc + relr[il], c);
                else
                    W[d.c_off + (long long)j * d.ldc + i] = old[OM > 1 ? m : 0][n][v] - c;
            }
        }
    }
    if constexpr (PD) {
        if (tail) pd_tail<float, TAIL_LDS>(pda, d.pd, W, smem, adiag, false);
    }
}

// Diagonal block Cholesky + triangular inverse of a 64x64 block (a block
// narrower than 64 is extended by the identity), one 256-thread workgroup,
// over 16-column panels p = 0..3 (panel_elim, potrf_core):
//   wave 0: rows of panel p, one per lane: POTRF of D_pp and the rows below it
//           in one elimination (no separate panel TRSM)
//   wave 1: D_pp again with the 16 identity rows below it: their elimination
//           leaves inv(D_pp)' (no separate inverse)
//   waves 2, 3, beside them: panel p-1's other updates (MFMA) and the sums
//           T_pj = sum_k L_pk X_kj of the inverse's block row p
//   then, all waves: the update of block column p+1 by panel p (MFMA) and
//           X_pj = -X_pp T_pj; wave 1 stores L_pp, which both had to read
// Two barriers per panel.  The lower factor is written back in place (the
// strict upper triangle is left alone, as dpotrf leaves it) and inv(L) (zero
// above the diagonal) goes to the block's inverse slot (ld nb).  A
// non-positive pivot at column j records col0 + j in *fail (atomic min).
// ---------------------------------------------------------------------------

// 1/sqrt(x) for x > 0: the hardware estimate y0 (relative error below 2^-23)
// refined once to third order, y = y0 (1 + e/2 + 3e^2/8) with e = 1 - x y0^2
// below 2^-22: the remaining term 5e^3/16 is below 2^-67, and the chain is four
// dependent operations where two Newton steps take six (every pivot waits for it).
__device__ __forceinline__ double rsqrt_nr(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    const double ye = y * e;
    return fma(ye, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ float rsqrt_nr(float x) {
    float y = __builtin_amdgcn_rsqf(x);
    const float e = fmaf(-x * y, y, 1.0f);
    return fmaf(0.5f * y, e, y);
}

// LDS stores of one lane visible to the other lanes of its wave
__device__ __forceinline__ void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// value of v in lane k (k wave-uniform), through a scalar register
__device__ __forceinline__ double lane_bcast(double v, int k) {
    int lo = __builtin_amdgcn_readlane(__double2loint(v), k);
    int hi = __builtin_amdgcn_readlane(__double2hiint(v), k);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ float lane_bcast(float v, int k) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}

// acc += X * Y' for 16x16 blocks X at S[rx..][cx..], Y at S[ry..][cy..] (row-major, stride PS)
template <typename T>
__device__ __forceinline__ void mma_nt16(const T *S, int rx, int cx, const T *S2, int ry, int cy,
                                         typename MfmaOp<T>::acc_t &acc, int lane) {
#pragma unroll
    for (int kk = 0; kk < 16; kk += 4) {
        const T a = S[(rx + (lane & 15)) * PS + cx + kk + (lane >> 4)];
        const T b = S2[(ry + (lane & 15)) * PS + cy + kk + (lane >> 4)];
        acc = MfmaOp<T>::mma(a, b, acc);
    }
}

// acc += X * Y for 16x16 blocks X at S[rx..][cx..], Y at S2[ry..][cy..]
template <typename T>
__device__ __forceinline__ void mma_nn16(const T *S, int rx, int cx, const T *S2, int ry, int cy,
                                         typename MfmaOp<T>::acc_t &acc, int lane) {
#pragma unroll
    for (int kk = 0; kk < 16; kk += 4) {
        const T a = S[(rx + (lane & 15)) * PS + cx + kk + (lane >> 4)];
        const T b = S2[(ry + kk + (lane >> 4)) * PS + cy + (lane & 15)];
        acc = MfmaOp<T>::mma(a, b, acc);
    }
}

// C at S[r0..][c0..] (op) acc, where acc holds D[row(lane,v)][lane%16] = C(m, n) with
// m indexing the MFMA A side (rows) and n the B side (columns)
template <typename T>
__device__ __forceinline__ void store16(T *S, int r0, int c0, const typename MfmaOp<T>::acc_t &acc,
                                        int lane, T alpha, bool accumulate) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
        T *q = S + (r0 + MfmaOp<T>::row(lane, v)) * PS + c0 + (lane & 15);
        *q = accumulate ? *q + alpha * acc[v] : alpha * acc[v];
    }
}

// Elimination of a 16-column panel by one wave, a row per lane: lanes 0..15 hold
// the rows of the diagonal block (their entries above the diagonal are not
// used), the other lanes rows below it.  On return a[] holds the rows of L:
// the diagonal block's factor in lanes 0..15 (zero or unused above the
// diagonal) and A L^-T in the others; an identity row e_q becomes column q of
// the inverse of the diagonal block.  Each pivot costs one reciprocal square
// root (no divide on the serial path): L_jj = d_jj r_j and L_ij = a_ij r_j
// with r_j = 1/sqrt(d_jj).  Returns the first non-positive pivot among the
// panel's nreal real columns (16 if none), wave-uniform.  SAFE: *brk is set
// when a pivot falls to its floor or below (floor_l, lane j holds column j's:
// rho * a_jj, a_jj the assembled diagonal of A): the block's result is then not
// used (redo_block64 refactors it).
//
// A non-positive pivot is replaced by 1, so that the values after it stay
// finite.  The test would lie on the chain from pivot to pivot, so the columns
// are eliminated without it first (REPLACE false: NaN from that pivot on), and
// once more with it, from the entries entry(c) of the lane's row again, if a
// pivot was not positive.
template <typename T, bool SAFE, bool REPLACE>
__device__ __forceinline__ void panel_pivots(T (&a)[16], T floor_l, int lane, unsigned &badm, unsigned &lowm) {
    badm = lowm = 0;                // bit j: pivot j is not positive / at or below its floor
    T djj = lane_bcast(a[0], 0);
#pragma unroll
    for (int j = 0; j < 16; j++) {
        badm |= (unsigned)__ballot(!(djj > (T)0)) & (1u << j);
        if (SAFE) lowm |= (unsigned)__ballot(djj <= lane_bcast(floor_l, j)) & (1u << j);
        if (REPLACE && !(djj > (T)0)) {
            djj = (T)1;
            if (lane == j) a[j] = (T)1;
        }
        const T l = a[j] * rsqrt_nr(djj);
        a[j] = l;
        if (j + 1 < 16) {
            // the next pivot first: its reciprocal square root then runs beside
            // the updates of the columns after it
            a[j + 1] -= l * lane_bcast(l, j + 1);
            djj = lane_bcast(a[j + 1], j + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        T bl[16];
#pragma unroll
        for (int c = j + 2; c < 16; c++) bl[c] = lane_bcast(l, c);
#pragma unroll
        for (int c = j + 2; c < 16; c++) a[c] -= l * bl[c];
    }
}

template <typename T, bool SAFE, typename Entry>
__device__ __forceinline__ int panel_elim(T (&a)[16], Entry entry, int nreal, T floor_l, int lane, bool *brk) {
    const unsigned realm = nreal >= 16 ? 0xffffu : (1u << nreal) - 1;
    unsigned badm, lowm;
#pragma unroll
    for (int c = 0; c < 16; c++) a[c] = entry(c);
    panel_pivots<T, SAFE, false>(a, floor_l, lane, badm, lowm);
    if (__builtin_expect((badm & realm) != 0, 0)) {
        // (one load at a time, from addresses that the compiler takes for others than
        // the first ones: it would keep those in registers throughout, 98 instead of
        // 55 in k_potrf_small)
        int o = 0;
        asm volatile("" : "+v"(o));
#pragma unroll
        for (int c = 0; c < 16; c++) {
            a[c] = entry(c + o);
            __builtin_amdgcn_sched_barrier(0);
        }
        panel_pivots<T, SAFE, true>(a, floor_l, lane, badm, lowm);
    }
    if (SAFE && (lowm & realm)) *brk = true;
    badm &= realm;
    return badm ? __builtin_ctz(badm) : 16;
}

// Factor and invert the diagonal block of nb columns held in LDS (256
// threads).  S: the block, NB x PS row-major, its lower triangle (extended by
// the identity past nb) on entry and L on return.  Its inverse: the lower
// triangle's 16x16 blocks at inv_at, in the same LDS.  sfail[0] receives the
// first failing column (-1 on entry), sfail[1] the breakdown flag (0 on entry).
// The inverse's four diagonal blocks hold the identity on entry (potrf_init).
// The caller synchronizes before; the block and its inverse are complete (and
// visible) on return.  Between two barriers no entry of LDS that one wave reads
// or writes is written by another.
template <typename T>
__device__ __forceinline__ void potrf_init(T *S, int *sfail) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int e = tid + 256 * q, i = e >> 4, c = e & 15;
        S[inv_at<T>(i >> 4, i >> 4) + (i & 15) * PS + c] = (i & 15) == c ? (T)1 : (T)0;
    }
    if (tid == 0) {
        sfail[0] = -1;
        sfail[1] = 0;
    }
}

template <typename T, bool SAFE>
__device__ __forceinline__ void potrf_core(T *S, int *sfail, int nb, const double *__restrict__ adiag,
                                           int col0, double rho) {
    typedef typename MfmaOp<T>::acc_t acc_t;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int np = (nb + 15) >> 4;          // 16-column panels that hold real columns
    // S(i, j) -= L(i, k) L(j, k)'
    auto update = [&](int i, int j, int k) {
        acc_t acc = acc_t{0, 0, 0, 0};
        // C(m = row in block j, n = row in block i)
        mma_nt16<T>(S, 16 * j, 16 * k, S, 16 * i, 16 * k, acc, lane);
#pragma unroll
        for (int v = 0; v < 4; v++) S[(16 * i + (lane & 15)) * PS + 16 * j + MfmaOp<T>::row(lane, v)] -= acc[v];
    };
    // X(p, j) = -X(p, p) T(p, j), T(p, j) held in the place of X(p, j)
    auto inv_row = [&](int p, int j) {
        acc_t acc = acc_t{0, 0, 0, 0};
        mma_nn16<T>(S + inv_at<T>(p, p), 0, 0, S + inv_at<T>(p, j), 0, 0, acc, lane);
        wave_sync_lds();                    // the wave's reads of T, before its stores
        store16<T>(S + inv_at<T>(p, j), 0, 0, acc, lane, (T)-1, false);
    };
    for (int p = 0; p < np; p++) {
        const int R = 16 * p;
        if (p > 0) {
            // block column p by panel p-1, and the inverse's block row p-1
            if (wave < np - p) update(p + wave, p, p - 1);
            if (wave == 3)
                for (int j = 0; j < p - 1; j++) inv_row(p - 1, j);
            __syncthreads();
        }
        T a[16];
        if (wave < 2) {
            // wave 0: row R + lane (past the last row: that row again, not stored);
            // wave 1: the diagonal block's rows, then the inverse's identity rows
            const bool row = R + lane < NB;
            const T *ar = (wave == 0 || lane < 16) ? S + min(R + lane, NB - 1) * PS + R
                                                   : S + inv_at<T>(p, p) + (lane & 15) * PS;
            auto entry = [&](int c) { return ar[c]; };
            T floor_l = 0;
            if (SAFE && lane < 16 && R + lane < nb) floor_l = (T)(rho * adiag[col0 + R + lane]);
            bool brk = false;
            const int badj = panel_elim<T, SAFE>(a, entry, nb - R, floor_l, lane, &brk);
            if (wave == 0) {
                if (lane == 0 && badj < 16 && sfail[0] < 0) sfail[0] = R + badj;
                if (SAFE && lane == 0 && brk) sfail[1] = 1;
                if (lane >= 16 && row) {
#pragma unroll
                    for (int c = 0; c < 16; c++) S[(R + lane) * PS + R + c] = a[c];
                }
            } else if (lane >= 16 && lane < 32) {
                // lane 16 + q: column q of the inverse
#pragma unroll
                for (int c = 0; c < 16; c++) S[inv_at<T>(p, p) + c * PS + lane - 16] = a[c];
            }
        } else {
            // waves 2, 3: panel p-1's updates right of block column p, then T(p, j)
            int q = 0;
            for (int i = p + 1; p > 0 && i < np; i++)
                for (int j = p + 1; j <= i; j++)
                    if ((q++ & 1) == wave - 2) update(i, j, p - 1);
            for (int j = 0; j < p; j++) {
                if ((q++ & 1) != wave - 2) continue;
                acc_t acc = acc_t{0, 0, 0, 0};
                for (int k = j; k < p; k++) mma_nn16<T>(S, R, 16 * k, S + inv_at<T>(k, j), 0, 0, acc, lane);
                store16<T>(S + inv_at<T>(p, j), 0, 0, acc, lane, (T)1, false);
            }
        }
        __syncthreads();
        // L(p, p), now that waves 0 and 1 have both read A(p, p); nothing before the
        // last barrier reads it (wave 1 has it as wave 0 does, and less to do next)
        if (wave == 1 && lane < 16) {
#pragma unroll
            for (int c = 0; c < 16; c++) S[(R + lane) * PS + R + c] = a[c];
        }
    }
    if (wave < np - 1) inv_row(np - 1, wave);
    __syncthreads();
}

// SAFE (rho > 0, low-precision factor): a pivot d_jj <= rho * a_jj (a_jj the
// assembled diagonal of A) signals breakdown of the block.  Its low-precision
// result is dropped and the same workgroup refactors the block in FP64 in
// place (redo_block64, in the LDS of the block and its inverse), before anything
// reads it.  Without SAFE a pivot <= 0 is reported as the failing column.
//
// potrf_block: the whole workgroup (256 threads) factors diagonal block t in
// LDS (S: potrf_lds<T>(SAFE) bytes, potrf_core's layout;
// sfail: two shared ints, the first failing column and the breakdown flag;
// tmp: NB shared doubles for the redo) and writes L_tt and the inverse back
// to W.
template <typename T, bool SAFE, bool LOADED>
__device__ __forceinline__ void potrf_block(const DiagTask &t, T *__restrict__ W, T *S, int *sfail,
                                            int *__restrict__ fail, const double *__restrict__ adiag,
                                            double rho, const Redo &rd, double *tmp) {
    const int tid = threadIdx.x;
    const int nb = t.nb;
    const int i = tid & (NB - 1), c0 = tid >> 6;
    if constexpr (!LOADED) {
        // all 16 loads of a thread in flight at once (unconditional, from inside the
        // block: a predicated load is a branch each), then the LDS stores
        T v[16];
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int c = c0 + 4 * q;
            v[q] = W[t.off + min(i, nb - 1) + (long long)min(c, nb - 1) * t.ld];
        }
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int c = c0 + 4 * q;
            S[i * PS + c] = (i < nb && c < nb) ? (c <= i ? v[q] : (T)0) : (i == c ? (T)1 : (T)0);
        }
    }
    potrf_init(S, sfail);
    __syncthreads();
    potrf_core<T, SAFE>(S, sfail, nb, adiag, t.col0, rho);
    if (SAFE && sfail[1]) {
        // breakdown: the block again from W, in FP64, in the same LDS
        redo_block64<T>(t, W, reinterpret_cast<double *>(S), tmp, sfail, tid, 256, rd, fail,
                        [] { __syncthreads(); });
        return;
    }
    if (tid == 0 && sfail[0] >= 0) atomicMin(fail, t.col0 + sfail[0]);
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int c = c0 + 4 * q;
        if (i < nb && c < nb) {
            if (c <= i) W[t.off + i + (long long)c * t.ld] = S[i * PS + c];
            W[t.winv + i + (long long)c * nb] =
                c <= i ? S[std::is_same<T, float>::value ? (NB + i) * PS + c
                                                         : inv_at<T>(i >> 4, c >> 4) + (i & 15) * PS + (c & 15)]
                       : (T)0;
        }
    }
}

template <typename T, bool SAFE>
__global__ __launch_bounds__(256) void k_potrf_diag(const DiagTask *__restrict__ tasks,
                                                    T *__restrict__ W, int *__restrict__ fail,
                                                    const double *__restrict__ adiag, double rho, Redo rd) {
    __shared__ __attribute__((aligned(16))) T SX[potrf_lds<T>(SAFE) / sizeof(T)];   // the block and its inverse
    __shared__ int sfail[2];
    __shared__ double tmp[SAFE ? NB : 1];
    potrf_block<T, SAFE>(tasks[blockIdx.x], W, SX, sfail, fail, adiag, rho, rd, tmp);
}

// Diagonal blocks of at most 16 columns (the many tiny supernodes of the
// lower etree levels): one wave per block, four blocks per workgroup, the
// block and its inverse from one elimination (panel_elim).
template <typename T, bool SAFE>
__global__ __launch_bounds__(256) void k_potrf_small(const DiagTask *__restrict__ tasks, int ntask,
                                                     T *__restrict__ W, int *__restrict__ fail,
                                                     const double *__restrict__ adiag, double rho, Redo rd) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ti = blockIdx.x * 4 + w;
    if (ti >= ntask) return;
    const DiagTask t = tasks[ti];
    const int nb = t.nb;
    // lanes 0..15: the block's rows (extended by the identity), lanes 16..31: identity rows
    T a[16];
    auto entry = [&](int c) {
        // (loads from inside the block, unconditional: a predicated load is a branch each)
        const T v = W[t.off + min(lane, nb - 1) + (long long)min(c, nb - 1) * t.ld];
        return (lane < nb && c <= lane) ? v : ((lane < 32 && (lane & 15) == c) ? (T)1 : (T)0);
    };
    T floor_l = 0;
    if (SAFE && lane < nb) floor_l = (T)(rho * adiag[t.col0 + lane]);
    bool brk = false;
    const int badj = panel_elim<T, SAFE>(a, entry, nb, floor_l, lane, &brk);
    if (SAFE && brk) {
        // breakdown: leave the assembled block in W for the FP64 redo
        if (lane == 0) redo_push(rd, t);
        return;
    }
    if (lane == 0 && badj < nb) atomicMin(fail, t.col0 + badj);
    // L by rows; lane 16 + q holds column q of the inverse
#pragma unroll
    for (int c = 0; c < 16; c++) {
        if (lane < nb && c <= lane) W[t.off + lane + (long long)c * t.ld] = a[c];
        if (lane >= 16 && lane - 16 < nb && c < nb) W[t.winv + c + (long long)(lane - 16) * nb] = a[c];
    }
}

// Diagonal blocks of at most TINY_DIAG columns (the bottom levels of a forest:
// mostly one to five columns): one lane factors and inverts a whole block, with
// panel_elim's arithmetic: pivot d_jj (when SAFE, a pivot at or below
// rho a_jj sends the block to the FP64 redo queue), a non-positive pivot
// reported and replaced by 1, r_j = 1/sqrt(d_jj), L_jj = d_jj r_j,
// L_ij = a_ij r_j, the inverse by forward substitution with r_j.
constexpr int TINY_DIAG = 6;

template <typename T, bool SAFE>
__global__ __launch_bounds__(256) void k_potrf_tiny(const DiagTask *__restrict__ tasks, int ntask,
                                                    T *__restrict__ W, int *__restrict__ fail,
                                                    const double *__restrict__ adiag, double rho, Redo rd) {
    const int ti = blockIdx.x * blockDim.x + threadIdx.x;
    if (ti >= ntask) return;
    const DiagTask t = tasks[ti];
    const int nb = t.nb;
    T a[TINY_DIAG][TINY_DIAG], x[TINY_DIAG][TINY_DIAG], rinv[TINY_DIAG];
#pragma unroll
    for (int i = 0; i < TINY_DIAG; i++)
#pragma unroll
        for (int c = 0; c <= i; c++)
            a[i][c] = i < nb ? W[t.off + i + (long long)c * t.ld] : (i == c ? (T)1 : (T)0);
    bool low_any = false;
    int badj = TINY_DIAG;
#pragma unroll
    for (int j = 0; j < TINY_DIAG; j++) {
        const bool real = j < nb;
        T djj = a[j][j];
        if (SAFE) low_any = low_any || (real && djj <= (T)(rho * adiag[t.col0 + j]));
        const bool bad = !(djj > (T)0);
        badj = (bad && real && badj == TINY_DIAG) ? j : badj;
        djj = bad ? (T)1 : djj;
        const T rj = rsqrt_nr(djj);
        rinv[j] = rj;
        a[j][j] = djj * rj;
#pragma unroll
        for (int i = j + 1; i < TINY_DIAG; i++) a[i][j] *= rj;
#pragma unroll
        for (int c = j + 1; c < TINY_DIAG; c++)
#pragma unroll
            for (int i = c; i < TINY_DIAG; i++) a[i][c] -= a[i][j] * a[c][j];
    }
    if (SAFE && low_any) {
        redo_push(rd, t);            // breakdown: the FP64 redo refactors the assembled block
        return;
    }
    if (badj < nb) atomicMin(fail, t.col0 + badj);
#pragma unroll
    for (int c = 0; c < TINY_DIAG; c++)
#pragma unroll
        for (int i = c; i < TINY_DIAG; i++) {
            T sacc = (i == c) ? (T)1 : (T)0;
#pragma unroll
            for (int k = c; k < i; k++) sacc -= a[i][k] * x[k][c];
            x[i][c] = sacc * rinv[i];
        }
#pragma unroll
    for (int c = 0; c < TINY_DIAG; c++)
#pragma unroll
        for (int i = 0; i < TINY_DIAG; i++)
            if (i < nb && c < nb) {
                if (c <= i) W[t.off + i + (long long)c * t.ld] = a[i][c];
                W[t.winv + i + (long long)c * nb] = (c <= i) ? x[i][c] : (T)0;
            }
}

// The FP64 redo of the blocks that the one-wave and one-lane POTRF kernels
// (k_potrf_small, k_potrf_tiny) queued on breakdown: launched after each such
// launch, so a queued block is final before the next launch reads it.  A
// workgroup takes queued blocks in turn (redo_block64); the last one to
// finish clears the queue for the next launch.  With nothing queued each
// workgroup only reads the counter.
constexpr int REDO_WG = 4;

template <typename T>
__global__ __launch_bounds__(256) void k_potrf_redo64(Redo rd, T *__restrict__ W, int *__restrict__ fail) {
    __shared__ double A[NB * (NB + 1)];
    __shared__ double tmp[NB];
    __shared__ int sbad;
    const int tid = threadIdx.x;
    const int cnt = rd.cnt[0];
    for (int e = blockIdx.x; e < cnt; e += gridDim.x) {
        redo_block64<T>(rd.list[e], W, A, tmp, &sbad, tid, (int)blockDim.x, rd, fail, [] { __syncthreads(); });
        __syncthreads();
    }
    __syncthreads();
    if (tid == 0) {
        __threadfence();
        if (atomicAdd(rd.cnt + 2, 1) == (int)gridDim.x - 1) {     // the last workgroup: clear the queue
            rd.cnt[0] = 0;
            rd.cnt[2] = 0;
        }
    }
}

// Panel TRSM of a tiny supernode (K <= TINY_DIAG columns, at most
// TINY_TRSM_ROWS rows below): one lane forms L2 = S2 inv(L11)' row by row, in
// place, as MODE_STORE does for a tile (C[i, j] = sum_k Y[i, k] X[j, k] with X
// the inverse at x_off + j + k ldx), and for a split-FP16 factor also writes
// the value's hi/lo pair scaled by its row's exponent.
constexpr int TINY_TRSM_ROWS = 16;

template <typename T>
__global__ __launch_bounds__(256) void k_trsm_tiny(const UpdDesc *__restrict__ descs,
                                                   const Tile *__restrict__ tiles, int ntile,
                                                   T *__restrict__ W, const int *__restrict__ Ls,
                                                   unsigned *__restrict__ Lh, const double *__restrict__ adiag) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ntile) return;
    const UpdDesc d = descs[tiles[e].desc];
    T inv[TINY_DIAG][TINY_DIAG];
#pragma unroll
    for (int j = 0; j < TINY_DIAG; j++)
#pragma unroll
        for (int k = 0; k < TINY_DIAG; k++)
            inv[j][k] = (j < d.N && k < d.K) ? W[d.x_off + j + (long long)k * d.ldx] : (T)0;
    for (int i = 0; i < d.M; i++) {
        T y[TINY_DIAG];
#pragma unroll
        for (int k = 0; k < TINY_DIAG; k++) y[k] = k < d.K ? W[d.y_off + i + (long long)k * d.ldy] : (T)0;
        const int ex = Lh ? row_scale_exp(adiag, Ls[d.ls_off + i]) : 0;
#pragma unroll
        for (int j = 0; j < TINY_DIAG; j++) {
            if (j >= d.N) break;
            T c = 0;
#pragma unroll
            for (int k = 0; k < TINY_DIAG; k++) c += y[k] * inv[j][k];
            const long long q = d.c_off + (long long)j * d.ldc + i;
            W[q] = c;
            if (std::is_same<T, float>::value && Lh) Lh[q] = split_pack((float)c, ex);
        }
    }
}


// ---------------------------------------------------------------------------
// Small supernodes of one etree level, fused: a supernode of at most
// SMALL_COLS columns and SMALL_NROW rows has one 64-column step, so its whole
// numeric factorization (t_cholmod_super_numeric_worker.c:537-1190: the
// descendant updates by dsyrk/dgemm scattered through the relative map, then
// dpotrf of the diagonal block and dtrsm of the rows below) is done by one
// workgroup, the supernode held in LDS from its assembly to its last store.
// The workgroups walk the level's tasks on a grid sized to the device (a
// persistent grid: task b, then b + gridDim.x, ...).  This replaces the
// level's descendant-update launch, its POTRF launch and its TRSM launch for
// these supernodes by one launch.
//
// Per descendant pair (the UpdDesc of the update launch, MODE_SCATTER
// semantics), wave w taking pairs w, w + 4, ...: C = Y X' by 16x16x4 FP64
// MFMAs straight from W (row blocks of 16 rows of Y against the N <= 16 rows
// of X), then S[rel(i)][rel(j)] -= C(i, j) for i >= j by LDS atomics, rel the
// block rows' positions among the supernode's rows.  Factorization, by wave 0:
// right-looking over the nscol columns with lane r owning row r of the panel,
// panel_elim's pivot arithmetic (r_j = 1/sqrt(d_jj), L_jj = d_jj r_j,
// L_rj = a_rj r_j, a non-positive pivot reported and replaced by 1) applied
// to the rows below the diagonal block as well, which makes the TRSM part of
// the same pass.  Column c of the diagonal block's inverse is formed by lane c.
// ---------------------------------------------------------------------------
constexpr int SMALL_COLS = 16;
constexpr int SMALL_NROW = 64;

__global__ __launch_bounds__(256) void k_small_level(const SmallTask *__restrict__ tasks, int ntask,
                                                     const UpdDesc *__restrict__ descs, double *__restrict__ W,
                                                     const int *__restrict__ Ls, int *__restrict__ fail) {
    constexpr int SD = SMALL_COLS + 1;
    __shared__ double S[SMALL_NROW * SD];
    __shared__ int rows[SMALL_NROW];
    __shared__ int rel[4][SMALL_NROW];
    __shared__ double rpiv[SMALL_COLS];        // r_j = 1/sqrt(d_jj) of each column
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int jl = lane & 15, kq = lane >> 4;
    int *rl = rel[w];
    for (int ti = blockIdx.x; ti < ntask; ti += gridDim.x) {
        const SmallTask t = tasks[ti];
        const int nsrow = t.nsrow, nscol = t.nscol;
        // the assembled block (thread e: row e % 64 of columns e / 64, e / 64 + 4, ...) and its rows
#pragma unroll
        for (int q = 0; q < SMALL_NROW * SMALL_COLS / 256; q++) {
            const int r = lane, c = w + 4 * q;
            S[r * SD + c] = (r < nsrow && c < nscol) ? W[t.lx + r + (long long)c * nsrow] : 0.0;
        }
        if (w == 0) rows[lane] = lane < nsrow ? Ls[t.psi + lane] : INT_MAX;
        __syncthreads();

#pragma unroll 1
        for (int p = t.u0 + w; p < t.u0 + t.nu; p += 4) {
            const UpdDesc u = descs[p];
            if (lane < u.M) {
                const int g = Ls[u.ls_off + lane];
                int r;
                if (g < t.k1 + nscol) {
                    r = g - t.k1;
                } else {
                    int lo = nscol, hi = nsrow - 1;
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        if (rows[mid] < g) lo = mid + 1; else hi = mid;
                    }
                    r = lo;
                }
                rl[lane] = r;
            }
            const int nblk = (u.M + 15) >> 4;
            f64x4 acc[4];
#pragma unroll
            for (int n = 0; n < 4; n++) acc[n] = f64x4{0, 0, 0, 0};
            // 8 columns of the descendant per pass: all 10 loads of a lane in
            // flight at once (32-bit offsets from the pair's base), then the
            // MFMAs in ascending k
            const double *xb = W + u.x_off, *yb0 = W + u.y_off;
#pragma unroll 1
            for (int k0 = 0; k0 < u.K; k0 += 8) {
                double xa[2], yb[2][4];
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const int k = k0 + 4 * c + kq;
                    const bool kin = k < u.K;
                    xa[c] = (kin && jl < u.N) ? xb[jl + k * u.ldx] : 0.0;
#pragma unroll
                    for (int n = 0; n < 4; n++)
                        yb[c][n] = (kin && 16 * n + jl < u.M) ? yb0[16 * n + jl + k * u.ldy] : 0.0;
                }
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    if (k0 + 4 * c >= u.K) break;
#pragma unroll
                    for (int n = 0; n < 4; n++)
                        if (n < nblk) acc[n] = MfmaOp<double>::mma(xa[c], yb[c][n], acc[n]);
                }
            }
            wave_sync_lds();                 // rel[] of every lane of the wave
            // acc[n][v] = C(i, j), i = 16 n + lane % 16, j = row(lane, v)
#pragma unroll
            for (int n = 0; n < 4; n++) {
                const int i = 16 * n + jl;
                if (n >= nblk || i >= u.M) continue;
                const int ri = rl[i];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int j = MfmaOp<double>::row(lane, v);
                    if (j < u.N && j <= i)
                        __hip_atomic_fetch_add(&S[ri * SD + rl[j]], -acc[n][v], __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                }
            }
            wave_sync_lds();                 // the map's reads, before the next pair's map
        }
        __syncthreads();

        if (w == 0) {
            // the panel, right-looking, lane r owning row r
            double a[SMALL_COLS];
#pragma unroll
            for (int c = 0; c < SMALL_COLS; c++) a[c] = c < nscol ? S[lane * SD + c] : 0.0;
            int badj = SMALL_COLS;
#pragma unroll
            for (int j = 0; j < SMALL_COLS; j++) {
                if (j >= nscol) continue;
                double djj = lane_bcast(a[j], j);
                const bool bad = !(djj > 0.0);
                badj = (bad && badj == SMALL_COLS) ? j : badj;
                djj = bad ? 1.0 : djj;
                const double rj = rsqrt_nr(djj);
                if (lane == j) rpiv[j] = rj;
                const double l = (lane > j) ? a[j] * rj : ((lane == j) ? djj * rj : 0.0);
                a[j] = l;
#pragma unroll
                for (int c = j + 1; c < SMALL_COLS; c++)
                    if (c < nscol) a[c] -= l * lane_bcast(l, c);
            }
            if (lane == 0 && badj < nscol) atomicMin(fail, t.k1 + badj);
            if (lane < nsrow) {
#pragma unroll
                for (int c = 0; c < SMALL_COLS; c++)
                    if (c < nscol && c <= lane) W[t.lx + lane + (long long)c * nsrow] = a[c];
            }
            // the inverse of the diagonal block: lane c forms column c
            if (lane < nscol) {
#pragma unroll
                for (int c = 0; c < SMALL_COLS; c++) S[lane * SD + c] = a[c];
            }
            wave_sync_lds();
            // x overwrites the partial sums in place: x_k = sm_k r_k once sm_k is final
            double x[SMALL_COLS];
#pragma unroll
            for (int i = 0; i < SMALL_COLS; i++) x[i] = (i == lane) ? 1.0 : 0.0;
#pragma unroll
            for (int k = 0; k < SMALL_COLS; k++) {
                if (k >= nscol) break;
                x[k] = x[k] * rpiv[k];
#pragma unroll
                for (int i = k + 1; i < SMALL_COLS; i++)
                    if (i < nscol) x[i] -= S[i * SD + k] * x[k];
            }
            if (lane < nscol) {
#pragma unroll
                for (int i = 0; i < SMALL_COLS; i++)
                    if (i < nscol) W[t.winv + i + (long long)lane * nscol] = (i >= lane) ? x[i] : 0.0;
            }
        }
        __syncthreads();                     // this task's LDS reads, before the next task's stores
    }
}

}  // namespace mxc
