// kb_blk_impl.h -- blocked batched Cholesky family, one workgroup per matrix (four
// waves, two for large batches of smaller orders), for orders above the
// register-resident range.
//
// Left-looking blocked algorithm with panel width NBK = 32, the same POTRF ->
// TRSM(R,L,T) -> SYRK(L,N,-1,+1) arithmetic the reference runs as a recursion
// of separate launches (src/batch_triangular/Xpotrf_batch_drivers.cuh:91-131),
// here inside one kernel.  Per panel (blk_potrf below):
//   - wave 0 reads the 32x32 diagonal block as three 16x16 tiles, subtracts
//     the products of the finished columns on the matrix cores, factors it in
//     registers (4-column panels on DPP rows, rank-4 updates on the matrix
//     cores) and leaves the inverses of the two 16x16 diagonal tiles in LDS;
//   - meanwhile the other waves read the 16-row tiles below and subtract the same
//     products, then solve them against the inverses (with a correction step
//     where a diagonal tile is ill-conditioned), all in registers: every
//     element of A is read once and every element of L written once, and the
//     only other traffic is re-reading finished columns of L;
//   - right-hand sides (POSV) are further row tiles of the panel: the forward
//     sweep L Y = B is the panel solve Y^T = B^T L^-T.
// What bounds it: for small batches the serial chain of a panel (the loads'
// latency, the 32 pivots, two barriers); with the four or eight workgroups of a CU
// that hide it, memory (finished columns are read again once per panel: the
// non-uniform DPOSV of orders 8..256 moves 13.1 GB in 2.82 ms, a copy's rate).
// Against the right-looking form it replaces (trailing matrix read and written once
// per 64 columns, rows solved by substitution one per thread), kernel times: DPOTRF
// n = 200 x 2,000 721 -> 339 us, n = 256 x 4,096 1.82 -> 0.92 ms, n = 128 x 8,000 0.86 ->
// 0.37 ms; SPOTRF n = 200 x 4,000 966 -> 397 us; the workgroup phase of the non-uniform
// DPOSV of orders 8..256 x 20,000 4.69 -> 2.82 ms.
// The solve (POSV/POTRS) runs blocked forward and backward sweeps over up to
// 64 right-hand sides per pass (so L is streamed once per sweep for up to 64
// right-hand sides): the diagonal blocks by DPP-row substitutions, the
// off-diagonal block products on the matrix cores.
#pragma once
#include "kb_device.h"
#include "kb_launch.h"
#include "kb_reg_impl.h"
#include "kb_rg_impl.h"
#include "kb_tile_impl.h"

constexpr int KB_BLK_NBK = 32;
constexpr int KB_BLK_WG = 256;
constexpr int KB_LL_LD = 17;    // pitch of a staged 16 x 16 tile
// 16-row tiles a wave holds at once (C and the running sums: FP64 16 VGPRs each
// per tile), kernel times: FP64 2 against 3, n = 128 x 8,000 373 against 363 us, n =
// 128 x 1,000 64.4 against 65.6; FP32 4 against 2, n = 200 x 4,000 397 against 431 us.
template <typename T> constexpr int ll_g();
template <> constexpr int ll_g<double>() { return 2; }
template <> constexpr int ll_g<float>() { return 4; }

// The factorization's blocks and the solve's staging are never live together.
// CB: the widest pass of the solve, in blocks of 16 right-hand sides.
template <typename T, int CB = 4>
struct BlkSmem {
    union {
        struct {
            T sY[16 * CB * (KB_BLK_NBK + 1)];     // the solve's staging of a block of the solution
            T sD[KB_BLK_NBK * (KB_BLK_NBK + 1)];  // the diagonal block
        };
        struct {
            T fD[KB_BLK_NBK * (KB_BLK_NBK + 1)];  // the factored diagonal block
            T fW[2][16 * KB_LL_LD];               // the inverses of its diagonal 16 x 16 tiles
            T tpan[4][16][4];                     // panel transposes of the diagonal-block factorization
        };
    };
    T sInv[KB_BLK_NBK];
    int flag;
    int grow;   // KB_GROW_* bits
};

// B(i, c) of a right-hand-side block: side_left -> column c, else row c.
template <typename T>
KB_DEV T& rhs_at(T* B, int ldb, int side_left, int i, int c)
{
    return side_left ? B[i + (long)c * ldb] : B[c + (long)i * ldb];
}

// The diagonal block L(k0.., k0..) of the factor in two steps, so the solve
// can issue the loads of the next block before working on the current one:
// blk_diag_fetch reads this thread's elements (e = tid + 256 m) into
// registers, blk_diag_put writes them to LDS with the inverse diagonal.
template <int W> constexpr int blk_dpt() { return KB_BLK_NBK * KB_BLK_NBK / W; }   // elements per thread of W

template <typename T, int W>
KB_DEV void blk_diag_fetch(T (&v)[blk_dpt<W>()], const T* L, int lda, int k0, int kb)
{
    constexpr int NBK = KB_BLK_NBK;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // lane-dependent values formed per call, not kept live across
#pragma unroll
    for (int m = 0; m < blk_dpt<W>(); ++m) {
        const int e = tid + W * m;
        const int r = e % NBK, c = e / NBK;
        const bool in = r < kb && c <= r;
        const T x = gld(L + (in ? (k0 + r) + (long)(k0 + c) * lda : 0));
        v[m] = in ? x : T(0);
    }
}

template <typename T, int CB, int W>
KB_DEV void blk_diag_put(const T (&v)[blk_dpt<W>()], int kb, BlkSmem<T, CB>& S, int unit = 0)
{
    constexpr int NBK = KB_BLK_NBK;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
#pragma unroll
    for (int m = 0; m < blk_dpt<W>(); ++m) {
        const int e = tid + W * m;
        const int r = e % NBK, c = e / NBK;
        S.sD[r * (NBK + 1) + c] = v[m];
        if (r == c) S.sInv[r] = (r < kb && !unit) ? T(1) / v[m] : T(1);
    }
    __syncthreads();
}

// Row of a 16x16 matrix-core accumulator held in register q by lanes 16g..16g+15
// (the column is the lane's position in its row of 16): FP64 interleaves the
// rows, FP32 blocks them.
template <typename T>
KB_DEV int blk_drow(int q, int g)
{
    return (sizeof(T) == 8) ? 4 * q + g : 4 * g + q;
}

// Substitution with the staged diagonal block (sD, sInv) for the NS groups of
// W / 16 right-hand sides of a pass: DPP row (wave, lg) of the workgroup takes
// right-hand sides c = W / 16 s + 4 wave + lg, lane li of the row holds block rows
// li and 16 + li, and y(j) comes from lane j by DPP; the NS independent
// substitutions are interleaved and share the LDS reads of L.
// FWD: L_D y = b, else L_D^T x = y; the result also goes to sY (right-hand
// side major) for the off-diagonal update that follows.  b is read as sc * b.
template <typename T, int NS, bool FWD, int CB, int W>
KB_DEV void blk_diag_subst(T* B, int ldb, int side_left, int k0, int kb, int c0, int rc, BlkSmem<T, CB>& S, T* sY,
                           T sc = T(1))
{
    constexpr int NBK = KB_BLK_NBK;
    int tid = threadIdx.x;
    // opaque to the optimizer, so the lane-dependent offsets below are formed
    // here and not hoisted out of the caller's loops (where they would stay
    // live through the factorization)
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, lg = lane >> 4;
    T y[NS][2], iv[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) iv[h] = S.sInv[16 * h + li];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int c = W / 16 * s + 4 * wave + lg;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = 16 * h + li;
            const bool in = c < rc && r < kb;
            // unconditional load from a clamped address, then a select: every load of the
            // block is in flight at once (a load under a branch waits before the join)
            const T v = gld(rhs_elem(B, ldb, side_left, in ? k0 + r : 0, in ? c0 + c : 0));
            y[s][h] = in ? sc * v : T(0);
        }
    }
#pragma unroll
    for (int jj = 0; jj < NBK; ++jj) {
        const int j = FWD ? jj : NBK - 1 - jj;
        const T ij = S.sInv[j];
        T t[NS];     // lane j: y(j) / L(j, j), read through DPP (lane j is not updated at step j)
#pragma unroll
        for (int s = 0; s < NS; ++s) t[s] = y[s][j >> 4] * ij;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = 16 * h + li;
            if (FWD ? (16 * h + 15 > j) : (16 * h < j)) {
                const T l = FWD ? ((r > j) ? S.sD[r * (NBK + 1) + j] : T(0))
                                : ((r < j) ? S.sD[j * (NBK + 1) + r] : T(0));
#pragma unroll
                for (int s = 0; s < NS; ++s) fnmac_rowk<T>(y[s][h], t[s], l, j);
            }
        }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int c = W / 16 * s + 4 * wave + lg;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = 16 * h + li;
            const T v = y[s][h] * iv[h];
            if (c < rc && r < kb) {
                gst(rhs_elem(B, ldb, side_left, k0 + r, c0 + c), v);
                sY[c * (NBK + 1) + r] = v;
            }
        }
    }
}

// all rc right-hand sides of a pass of up to 16 CB (ncb blocks of 16)
template <typename T, bool FWD, int CB, int W>
KB_DEV void blk_diag_subst_n(int ncb, T* B, int ldb, int side_left, int k0, int kb, int c0, int rc, BlkSmem<T, CB>& S, T* sY,
                             T sc = T(1))
{
    constexpr int MX = 16 * CB / (W / 16);   // groups of a full pass
    static_assert(MX == 2 || MX == 4, "one case per group count");
    const int ns = W == 256 ? ncb : (rc + W / 16 - 1) / (W / 16);
    if (MX == 2 || ns <= 2) {
        if (ns == 1) blk_diag_subst<T, 1, FWD, CB, W>(B, ldb, side_left, k0, kb, c0, rc, S, sY, sc);
        else blk_diag_subst<T, 2, FWD, CB, W>(B, ldb, side_left, k0, kb, c0, rc, S, sY, sc);
        return;
    }
    if constexpr (MX > 2) {
        if (ns == 3) blk_diag_subst<T, 3, FWD, CB, W>(B, ldb, side_left, k0, kb, c0, rc, S, sY, sc);
        else blk_diag_subst<T, 4, FWD, CB, W>(B, ldb, side_left, k0, kb, c0, rc, S, sY, sc);
    }
}

// B(r, c) := sc B(r, c) - sum_k Lk(r, k) Y(k, c) for the rows r in [r_lo, r_hi), k < kb and
// the pass's right-hand sides, on the matrix cores.  Lk(r, k) = L(r, k0 + k)
// (TRANS false: the block column below the diagonal block, forward sweep) or
// L(k0 + k, r) (TRANS true: the block row left of it, backward sweep); Y is
// staged in sY (right-hand side major).  Each wave takes 16-row blocks: the
// L fragment (eight K steps of 4) and the B blocks of the NCB column blocks of
// 16 right-hand sides are loaded together, then NCB independent MFMA chains.
template <typename T, bool TRANS, int NCB, int W>
KB_DEV void blk_update_rows(const T* L, int lda, T* B, int ldb, int side_left, int k0, int kb, int r_lo,
                            int r_hi, int c0, int rc, const T* sY, T sc = T(1))
{
    constexpr int NBK = KB_BLK_NBK;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // lane-dependent offsets stay local (as in blk_diag_subst)
    const int wave = tid >> 6, lane = tid & 63;
    const int li = lane & 15, lg = lane >> 4;
    for (int r0 = r_lo + 16 * wave; r0 < r_hi; r0 += W / 4) {
        T a[NBK / 4];
#pragma unroll
        for (int q = 0; q < NBK / 4; ++q) {
            const int kk = 4 * q + lg;
            const int row = r0 + li;
            const bool ain = row < r_hi && kk < kb;
            const long off = TRANS ? (k0 + kk) + (long)row * lda : row + (long)(k0 + kk) * lda;
            const T av = gld(L + (ain ? off : 0));
            a[q] = ain ? av : T(0);
        }
        T bv[NCB][4];
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
            const int cc = 16 * cb + li;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = r0 + blk_drow<T>(q, lg);
                const bool in = row < r_hi && cc < rc;
                const T v = gld(rhs_elem(B, ldb, side_left, in ? row : 0, in ? c0 + cc : c0));
                bv[cb][q] = in ? v : T(0);
            }
        }
        typename TileV<T>::v4 acc[NCB];
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) acc[cb] = typename TileV<T>::v4{T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int q = 0; q < NBK / 4; ++q) {
            const int kk = 4 * q + lg;
#pragma unroll
            for (int cb = 0; cb < NCB; ++cb) {
                const int cc = 16 * cb + li;
                const T b = (kk < kb && cc < rc) ? sY[cc * (NBK + 1) + kk] : T(0);
                acc[cb] = mfma16x16x4(a[q], b, acc[cb]);
            }
        }
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
            const int cc = 16 * cb + li;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = r0 + blk_drow<T>(q, lg);
                if (row < r_hi && cc < rc) gst(rhs_elem(B, ldb, side_left, row, c0 + cc), sc * bv[cb][q] - acc[cb][q]);
            }
        }
    }
}

template <typename T, bool TRANS, int CB, int W>
KB_DEV void blk_update_rows_n(int ncb, const T* L, int lda, T* B, int ldb, int side_left, int k0, int kb, int r_lo,
                              int r_hi, int c0, int rc, const T* sY, T sc = T(1))
{
    if (CB == 2 || ncb <= 2) {
        if (ncb == 1) blk_update_rows<T, TRANS, 1, W>(L, lda, B, ldb, side_left, k0, kb, r_lo, r_hi, c0, rc, sY, sc);
        else blk_update_rows<T, TRANS, 2, W>(L, lda, B, ldb, side_left, k0, kb, r_lo, r_hi, c0, rc, sY, sc);
        return;
    }
    if constexpr (CB > 2) {
        if (ncb == 3) blk_update_rows<T, TRANS, 3, W>(L, lda, B, ldb, side_left, k0, kb, r_lo, r_hi, c0, rc, sY, sc);
        else blk_update_rows<T, TRANS, 4, W>(L, lda, B, ldb, side_left, k0, kb, r_lo, r_hi, c0, rc, sY, sc);
    }
}

// One block step of the forward sweep L Y = B: substitution with the
// diagonal block staged in sD / sInv, then the rows below updated with the
// block column of L (all right-hand sides, in passes of up to 16 CB: a
// narrower pass needs fewer registers, a wider one streams L fewer times).
// sc scales the right-hand sides as they are first read (the first step).
template <typename T, int CB, int W>
KB_DEV void blk_fwd_step(const T* L, int lda, int n, int k0, int kb, T* B, int ldb, int side_left, int nrhs,
                         BlkSmem<T, CB>& S, T sc = T(1))
{
    constexpr int RC = 16 * CB;
    T* sY = S.sY;   // RC x (NBK + 1) staging of the block's solution
    for (int c0 = 0; c0 < nrhs; c0 += RC) {
        const int rc = min(RC, nrhs - c0);
        const int ncb = (rc + 15) / 16;
        blk_diag_subst_n<T, true, CB, W>(ncb, B, ldb, side_left, k0, kb, c0, rc, S, sY, sc);
        __syncthreads();
        blk_update_rows_n<T, false, CB, W>(ncb, L, lda, B, ldb, side_left, k0, kb, k0 + kb, n, c0, rc, sY, sc);
        __syncthreads();
    }
}

// Forward sweep L Y = alpha B over 32-row blocks (right-looking), the next
// diagonal block fetched while the current one is used; unit: the diagonal
// of L is taken as 1 (not read).
template <typename T, int CB = 4, int W = KB_BLK_WG>
KB_DEV void blk_solve_fwd(const T* L, int lda, int n, T* B, int ldb, int side_left, int nrhs, BlkSmem<T, CB>& S,
                          T alpha = T(1), int unit = 0)
{
    constexpr int NBK = KB_BLK_NBK;
    T dnext[blk_dpt<W>()];
    blk_diag_fetch<T, W>(dnext, L, lda, 0, min(NBK, n));
    for (int k0 = 0; k0 < n; k0 += NBK) {
        const int kb = min(NBK, n - k0);
        blk_diag_put<T, CB, W>(dnext, kb, S, unit);
        if (k0 + NBK < n) blk_diag_fetch<T, W>(dnext, L, lda, k0 + NBK, min(NBK, n - k0 - NBK));
        blk_fwd_step<T, CB, W>(L, lda, n, k0, kb, B, ldb, side_left, nrhs, S, k0 == 0 ? alpha : T(1));
    }
}

// Backward sweep L^T X = alpha Y over 32-row blocks (right-looking: after
// each block's substitution the rows above it are updated); unit as above.
template <typename T, int CB = 4, int W = KB_BLK_WG>
KB_DEV void blk_solve_bwd(const T* L, int lda, int n, T* B, int ldb, int side_left, int nrhs, BlkSmem<T, CB>& S,
                          T alpha = T(1), int unit = 0)
{
    constexpr int NBK = KB_BLK_NBK, RC = 16 * CB;
    T* sY = S.sY;
    T dnext[blk_dpt<W>()];
    const int nblk = (n + NBK - 1) / NBK;
    blk_diag_fetch<T, W>(dnext, L, lda, (nblk - 1) * NBK, n - (nblk - 1) * NBK);
    for (int bk = nblk - 1; bk >= 0; --bk) {
        const int k0 = bk * NBK;
        const int kb = min(NBK, n - k0);
        blk_diag_put<T, CB, W>(dnext, kb, S, unit);
        if (bk > 0) blk_diag_fetch<T, W>(dnext, L, lda, k0 - NBK, NBK);
        const T sc = bk == nblk - 1 ? alpha : T(1);
        for (int c0 = 0; c0 < nrhs; c0 += RC) {
            const int rc = min(RC, nrhs - c0);
            const int ncb = (rc + 15) / 16;
            blk_diag_subst_n<T, false, CB, W>(ncb, B, ldb, side_left, k0, kb, c0, rc, S, sY, sc);
            __syncthreads();
            blk_update_rows_n<T, true, CB, W>(ncb, L, lda, B, ldb, side_left, k0, kb, 0, k0, c0, rc, sY, sc);
            __syncthreads();
        }
    }
}

// Solve (L L^T) X = B for nrhs vectors stored by rhs_at(); L lower in A.
template <typename T, int CB = 4, int W = KB_BLK_WG>
KB_DEV void blk_solve(const T* L, int lda, int n, T* B, int ldb, int side_left, int nrhs, BlkSmem<T, CB>& S)
{
    blk_solve_fwd<T, CB, W>(L, lda, n, B, ldb, side_left, nrhs, S);
    blk_solve_bwd<T, CB, W>(L, lda, n, B, ldb, side_left, nrhs, S);
}

// ---------------------------------------------------------------------------
// factorization
// ---------------------------------------------------------------------------
// A 16-row tile of the panel: element (row i of the tile, column k) at
// p + i * rs + k * cs.  Rows of A: (rs, cs) = (1, lda); right-hand sides
// (row i is right-hand side i): (1, ldb) for side right, (ldb, 1) for left.
template <typename T>
struct LlTile {
    T* p;
    long rs, cs;
    int rows;   // valid rows (1..16)
};

// Columns between a lane's accumulator elements e and e + 1 of a tile.
template <typename T> constexpr int ll_step(int e) { return sizeof(T) == 8 ? 4 : (e & 3) == 3 ? 13 : 1; }

// K steps of 4 columns whose loads go out together (a second set is in flight
// while they are multiplied).
constexpr int KB_LL_U = 1;
constexpr int KB_LL_KC = 64;   // columns whose products are summed before they are taken from C

// A diagonal tile L counts as ill-conditioned when four columns of W = L^-1 give a
// row of |W| |L| (unchanged by a scaling of A's rows and columns) more than this;
// its row sums stay below 16 otherwise.  B B^T + n I of order 200 has sums of 1.6,
// Q diag(s) Q^T of condition 1e4 up to 10, a Gaussian kernel matrix at the limit of
// FP64 1e6: without the correction POTRF's error there is 1,000 times
// substitution's, or a pivot comes out negative.  (Not with a NaN in |W| |L|: an
// infinity on A's diagonal leaves a zero column in W, and c - L x would be NaN.)
// Forming the measure is in wave 0's serial part: DPOTRF n = 200, one matrix, 87.7
// -> 88.7 us, SPOTRF 66.9 -> 68.3 us, batches that fill the chip as before.
constexpr int KB_LL_GROW = 4;
// The same for the mixed routine's FP32 sweeps, whose result a refinement corrects:
// row sums below 128 cost no more than the rounding of a substitution over 65 or
// more rows, and random matrices of condition 1e4 (2,000 systems of order
// 128..512: 5.55 ms, with a limit of 4 5.70) stay without the correction.
constexpr int KB_LL_GROW_SWEEP = 32;
constexpr int KB_GROW_NOW = 1;   // the factored panel has a tile above KB_LL_GROW
constexpr int KB_GROW_ANY = 2;   // a panel so far has one above KB_LL_GROW_SWEEP

// c[j] := C_j - L_j L_P^T in transposed form for NT tiles: register r of column
// block q holds, in lane (i, g), row i and panel column 16 q + blk_drow(r, g).
// Lp: the panel's rows of L (row k0, column 0), kb of them valid; rows and
// columns beyond the valid ones repeat the last (their results are never
// used).  The products of 64 columns at a time are summed by themselves and
// then taken from C: added to C one by one they would each be rounded at its
// size, and a sum over all the columns at the size of the whole sum.
template <typename T, int NT>
KB_DEV void ll_update(const T* Lp, int lda, int kb, int k0, const LlTile<T>* t, int li, int lg,
                      typename TileV<T>::v4 (&c)[NT][2])
{
    typedef typename TileV<T>::v4 v4;
    // formed here, not kept live (or as induction variables) across panels
    asm volatile("" : "+v"(li), "+v"(lg));
    asm volatile("" : "+s"(k0));
    constexpr int U = KB_LL_U;
    const T* pb[NT];
    const T* pa[2];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const T* p = t[j].p + (long)min(li, t[j].rows - 1) * t[j].rs;
        pb[j] = p + lg * t[j].cs;
        // a running pointer (opaque each step), so the column addresses are not
        // all formed at once; it stops at the last valid column
        p += (k0 + min(blk_drow<T>(0, lg), kb - 1)) * t[j].cs;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            c[j][e >> 2][e & 3] = gld(p);
            if (16 * ((e + 1) >> 2) + blk_drow<T>((e + 1) & 3, lg) < kb) p += ll_step<T>(e) * t[j].cs;
            asm volatile("" : "+v"(p));
        }
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) pa[q] = Lp + min(16 * q + li, kb - 1) + (long)lg * lda;
    T a[U][2], b[U][NT], an[U][2], bn[U][NT];
    auto fetch = [&](T (&xa)[U][2], T (&xb)[U][NT]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                xa[u][q] = gld(pa[q]);
                pa[q] += 4 * (long)lda;
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                xb[u][j] = gld(pb[j]);
                pb[j] += 4 * t[j].cs;
            }
        }
    };
    v4 acc[NT][2];
    auto mult = [&](const T (&xa)[U][2], const T (&xb)[U][NT]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[j][q] = mfma16x16x4(xa[u][q], xb[u][j], acc[j][q]);
    };
    if (k0 > 0) fetch(a, b);
    for (int kc = 0; kc < k0; kc += KB_LL_KC) {
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j][0] = acc[j][1] = v4{T(0), T(0), T(0), T(0)};
        // k0 and KB_LL_KC are multiples of 32, so the steps come in pairs of U
        const int ke = min(kc + KB_LL_KC, k0);
        for (int k = kc; k < ke; k += 8 * U) {
            fetch(an, bn);
            mult(a, b);
            __builtin_amdgcn_sched_barrier(0);
            if (k + 8 * U < k0) fetch(a, b);
            mult(an, bn);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int q = 0; q < 2; ++q) c[j][q] -= acc[j][q];
    }
}

// x + W c for the inverse W of a 16 x 16 triangle
template <typename T>
KB_DEV typename TileV<T>::v4 ll_apply(const T* W, int li, int lg, const typename TileV<T>::v4& c,
                                      typename TileV<T>::v4 x = {T(0), T(0), T(0), T(0)})
{
#pragma unroll
    for (int s = 0; s < 4; ++s) x = mfma16x16x4(W[li * KB_LL_LD + blk_drow<T>(s, lg)], c[s], x);
    return x;
}

// c - L x for the 16 x 16 triangle L (zero above its diagonal) at L, pitch LD
template <typename T, int LD>
KB_DEV typename TileV<T>::v4 ll_resid(const T* L, int li, int lg, const typename TileV<T>::v4& x,
                                      typename TileV<T>::v4 c)
{
#pragma unroll
    for (int s = 0; s < 4; ++s) c = mfma16x16x4(-L[li * LD + blk_drow<T>(s, lg)], x[s], c);
    return c;
}

// One updated tile solved against the factored diagonal block and stored:
// X1^T = L11^-1 C1^T, X2^T = L22^-1 (C2^T - L21 X1^T).  A 16 x 16 accumulator is
// itself the second operand of the next product (register s of lane group g
// holds row kmap(s, g)), so nothing leaves the registers.
// The product W c with an inverse W errs by eps |L| |W| |L| |x|, a substitution by
// eps |L| |x|: where |W| |L| is large (COR, see KB_LL_GROW) one correction
// x += W (c - L x) brings the error back to the substitution's.
template <typename T, int CB, bool COR>
KB_DEV void ll_solve(const LlTile<T>& t, int kb, int k0, int li, int lg, const BlkSmem<T, CB>& S,
                     typename TileV<T>::v4 (&c)[2])
{
    constexpr int LD = KB_BLK_NBK + 1;
    typename TileV<T>::v4 x[2];
    if (kb < KB_BLK_NBK) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (16 * (e >> 2) + blk_drow<T>(e & 3, lg) >= kb) c[e >> 2][e & 3] = T(0);
    }
    x[0] = ll_apply<T>(S.fW[0], li, lg, c[0]);
    if (COR) x[0] = ll_apply<T>(S.fW[0], li, lg, ll_resid<T, LD>(S.fD, li, lg, x[0], c[0]), x[0]);
#pragma unroll
    for (int s = 0; s < 4; ++s) c[1] = mfma16x16x4(-S.fD[(16 + li) * LD + blk_drow<T>(s, lg)], x[0][s], c[1]);
    x[1] = ll_apply<T>(S.fW[1], li, lg, c[1]);
    if (COR)
        x[1] = ll_apply<T>(S.fW[1], li, lg, ll_resid<T, LD>(S.fD + 16 * LD + 16, li, lg, x[1], c[1]), x[1]);
    T* p = t.p + (long)li * t.rs + (k0 + blk_drow<T>(0, lg)) * t.cs;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        if (li < t.rows && 16 * (e >> 2) + blk_drow<T>(e & 3, lg) < kb) gst(p, x[e >> 2][e & 3]);
        p += ll_step<T>(e) * t.cs;
        asm volatile("" : "+v"(p));
    }
}

template <typename T, int NT, int CB, bool COR>
KB_DEV void ll_solve_n(const LlTile<T>* t, int kb, int k0, int li, int lg, const BlkSmem<T, CB>& S,
                       typename TileV<T>::v4 (&c)[NT][2])
{
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        ll_solve<T, CB, COR>(t[j], kb, k0, li, lg, S, c[j]);
        __builtin_amdgcn_sched_barrier(0);   // one tile's products at a time (registers)
    }
}

// One wave's NT tiles of a panel: update, wait for the diagonal block (first:
// every wave of the workgroup passes exactly one barrier here, in ll_diag's
// branch or in one of these), solve.  Returns S.flag.
template <typename T, int NT, int CB>
KB_DEV int ll_group(bool first, const T* Lp, int lda, int kb, int k0, const LlTile<T>* t, int li, int lg,
                    const BlkSmem<T, CB>& S)
{
    typename TileV<T>::v4 c[NT > 0 ? NT : 1][2];
    if constexpr (NT > 0) ll_update<T, NT>(Lp, lda, kb, k0, t, li, lg, c);
    if (first) __syncthreads();
    const int f = uniform(S.flag), grow = uniform(S.grow);   // (one wait for both)
    if (first && f) return f;
    if constexpr (NT > 0) {
        // formed here, not kept live (or as induction variables) across panels
        asm volatile("" : "+v"(li), "+v"(lg));
        asm volatile("" : "+s"(k0));
        if (grow & KB_GROW_NOW) ll_solve_n<T, NT, CB, true>(t, kb, k0, li, lg, S, c);
        else ll_solve_n<T, NT, CB, false>(t, kb, k0, li, lg, S, c);
    }
    return 0;
}

// Wave 0's part of a panel: the diagonal block (k0, kb) updated with the k0
// finished columns, factored and written to memory, its tile (1, 0) and the
// inverses of its two diagonal tiles to LDS.  S.flag: 0 or k0 + the failing
// column (1-based).  This is the serial part the other waves wait for, so its
// products run three to a pair of loads with the next 16 columns' loads in
// flight (with four loads to three products and none in flight, the update
// took 28,000 instead of 10,000 cycles a panel at n = 200 in FP32, and SPOTRF
// n = 200 x 4,000 0.57 instead of 0.40 ms).
template <typename T, int CB>
KB_DEV void ll_diag(T* A, int lda, int k0, int kb, BlkSmem<T, CB>& S, int lane, T* W)
{
    typedef typename TileV<T>::v4 v4;
    constexpr int LD = KB_BLK_NBK + 1;
    asm volatile("" : "+v"(lane));
    asm volatile("" : "+s"(k0));
    const int i = lane & 15, g = lane >> 4;
    T* D = A + k0 + (long)k0 * lda;
    // tiles (0,0), (1,0), (1,1) in ll_update's layout: lane (i, g) register r is
    // row i, column blk_drow(r, g)
    v4 c[3];
#pragma unroll
    for (int I = 0; I < 2; ++I)
#pragma unroll
        for (int J = 0; J <= I; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * I + i, col = 16 * J + blk_drow<T>(r, g);
                c[tix(I, J)][r] = gld(D + ((row < kb && col <= row) ? row + (long)col * lda : 0));
            }
    const T* p[2];
#pragma unroll
    for (int I = 0; I < 2; ++I) p[I] = A + k0 + min(16 * I + i, kb - 1) + (long)g * lda;
    if (k0 > 0) {
        constexpr int CH = 16, ST = CH / 4;
        T x[ST][2], xn[ST][2];
        auto fetch = [&](T (&y)[ST][2]) {
#pragma unroll
            for (int u = 0; u < ST; ++u)
#pragma unroll
                for (int I = 0; I < 2; ++I) {
                    y[u][I] = gld(p[I]);
                    p[I] += 4 * (long)lda;
                }
        };
        v4 acc[3];
        auto mult = [&](const T (&y)[ST][2]) {
#pragma unroll
            for (int u = 0; u < ST; ++u) {
                acc[0] = mfma16x16x4(y[u][0], y[u][0], acc[0]);
                acc[1] = mfma16x16x4(y[u][0], y[u][1], acc[1]);
                acc[2] = mfma16x16x4(y[u][1], y[u][1], acc[2]);
            }
        };
        fetch(x);
        for (int kc = 0; kc < k0; kc += KB_LL_KC) {   // sums of KB_LL_KC columns, as in ll_update
            acc[0] = acc[1] = acc[2] = v4{T(0), T(0), T(0), T(0)};
            const int ke = min(kc + KB_LL_KC, k0);
            for (int k = kc; k < ke; k += 2 * CH) {   // k0 is a multiple of 32
                fetch(xn);
                mult(x);
                __builtin_amdgcn_sched_barrier(0);
                if (k + 2 * CH < k0) fetch(x);
                mult(xn);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) c[q] -= acc[q];
        }
    }
    // rows and columns at or beyond kb, and the upper triangle, read as the identity
#pragma unroll
    for (int I = 0; I < 2; ++I)
#pragma unroll
        for (int J = 0; J <= I; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * I + i, col = 16 * J + blk_drow<T>(r, g);
                const T v = (row < kb && col <= row) ? c[tix(I, J)][r] : (row == col) ? T(1) : T(0);
                c[tix(I, J)][r] = v;
                if (sizeof(T) == 8) S.fD[row * LD + col] = v;
            }
    if constexpr (sizeof(T) == 8) {   // (the FP32 accumulators are in the factorization's layout)
        wave_lds_sync();
#pragma unroll
        for (int I = 0; I < 2; ++I)
#pragma unroll
            for (int J = 0; J <= I; ++J)
#pragma unroll
                for (int r = 0; r < 4; ++r) c[tix(I, J)][r] = S.fD[(16 * I + i) * LD + 16 * J + 4 * g + r];
    }
    T invd[2] = {T(1), T(1)};
    const int info = tile_potrf<T, 2>(c, invd, kb, S.tpan, lane);
#pragma unroll
    for (int I = 0; I < 2; ++I)
#pragma unroll
        for (int J = 0; J <= I; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * I + i, col = 16 * J + 4 * g + r;
                if (row < kb && col <= row) gst(D + row + (long)col * lda, c[tix(I, J)][r]);
                S.fD[row * LD + col] = (col <= row) ? c[tix(I, J)][r] : T(0);
            }
    // the row sums of the diagonal tiles' |L|
    T* rs = &S.tpan[0][0][0];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        T v = T(0);
#pragma unroll
        for (int r = 0; r < 4; ++r) v += (4 * g + r <= i) ? kb_abs<T>(c[tix(b, b)][r]) : T(0);
        rs[16 * b + i] = sum_rows4<T>(v);
    }
    if (g == 0) {
        S.sInv[i] = invd[0];
        S.sInv[16 + i] = invd[1];
    }
    if (lane == 0) S.flag = info ? k0 + info : 0;
    wave_lds_sync();
    // the inverses of both diagonal tiles: DPP row g takes columns 4g..4g+3 of
    // each, lane i of the row holds their row i
    T y[2][4], lsum[2][4];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int s = 0; s < 4; ++s) lsum[b][s] = rs[16 * b + 4 * g + s];
#pragma unroll
    for (int s = 0; s < 4; ++s) y[0][s] = y[1][s] = (i == 4 * g + s) ? T(1) : T(0);
#pragma unroll
    for (int j = 0; j < 15; ++j) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const T ij = S.sInv[16 * b + j];
            const T l = (i > j) ? S.fD[(16 * b + i) * LD + 16 * b + j] : T(0);
#pragma unroll
            for (int s = 0; s < 4; ++s) fnmac_rowk<T>(y[b][s], y[b][s] * ij, l, j);
        }
    }
    T m[2];   // this lane's four columns' part of a row of |W| |L| (its sum)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        m[b] = T(0);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const T v = y[b][s] * S.sInv[16 * b + i];
            S.fW[b][i * KB_LL_LD + 4 * g + s] = v;
            if (W && 16 * b < kb) gst(W + 16L * (k0 + 16 * b) + 16 * i + 4 * g + s, v);
            m[b] += kb_abs<T>(v) * lsum[b][s];
        }
    }
    int grow = k0 > 0 ? S.grow & KB_GROW_ANY : 0;
    const T mm = m[0] > m[1] ? m[0] : m[1], ms = m[0] + m[1];
    if (__any(mm > T(KB_LL_GROW)) && !__any(ms != ms)) {
        grow |= KB_GROW_NOW;
        if (__any(mm > T(KB_LL_GROW_SWEEP))) grow |= KB_GROW_ANY;
    }
    if (lane == 0) S.grow = grow;
}

// In-place lower Cholesky of an n x n matrix by the whole workgroup.
// Returns LAPACK info (identical in every thread).  With B given (POSV), the
// forward sweep L Y = B runs inside the factorization, the right-hand sides
// being further row tiles of every panel; a factorization that fails at panel k
// leaves B forward-solved in the rows of the panels before k and as it was in
// the others.  Wt, if given, receives the inverses of the factor's 16 x 16
// diagonal tiles (row-major, identity beyond n); S.grow then says whether
// products with them need the correction (KB_GROW_ANY).
template <typename T, int CB = 4, int W = KB_BLK_WG>
KB_DEV int blk_potrf(T* A, int lda, int n, BlkSmem<T, CB>& S, T* B = nullptr, int ldb = 0, int side_left = 0,
                     int nrhs = 0, T* Wt = nullptr)
{
    constexpr int NBK = KB_BLK_NBK, G = ll_g<T>(), NW = W / 64;
    static_assert(G <= 4, "one case per tile count below");
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // lane-dependent values formed per call, not kept live across
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int li = lane & 15, lg = lane >> 4;
    const int nrt = B ? (max(nrhs, 0) + 15) >> 4 : 0;   // (non-uniform counts come unchecked from the device)
    for (int k0 = 0; k0 < n; k0 += NBK) {
        const int kb = min(NBK, n - k0);
        const int nt = max((n - k0 - NBK + 15) >> 4, 0);   // row tiles below the diagonal block
        const int rest = nt + nrt;
        auto tile = [&](int q) {   // tile q of the panel: rows of A, then right-hand sides
            LlTile<T> t;
            if (q < nt) {
                const int r0 = k0 + NBK + 16 * q;
                t.p = A + r0;
                t.rs = 1;
                t.cs = lda;
                t.rows = min(16, n - r0);
            } else {
                const int c0 = 16 * (q - nt);
                t.rs = side_left ? ldb : 1;
                t.cs = side_left ? 1 : ldb;
                t.p = B + c0 * t.rs;
                t.rows = min(16, nrhs - c0);
            }
            return t;
        };
        // rounds of up to G tiles per wave; in the first, wave 0 factors the
        // diagonal block instead, and nothing is solved before that is done
        for (int base = 0, nw = NW - 1; base < rest || nw == NW - 1; nw = NW) {
            const int round = min(rest - base, nw * G);
            const int per = (round + nw - 1) / nw;
            const int q0 = base + (wave - NW + nw) * per;
            const int cnt = (q0 < base) ? 0 : max(min(per, base + round - q0), 0);
            const bool diag = nw == NW - 1;
            LlTile<T> t[G];
#pragma unroll
            for (int j = 0; j < G; ++j) t[j] = tile(max(min(q0 + j, rest - 1), 0));
            int f;
            if (diag && wave == 0) {
                ll_diag<T, CB>(A, lda, k0, kb, S, lane, Wt);
                f = ll_group<T, 0, CB>(diag, A + k0, lda, kb, k0, t, li, lg, S);
            } else if (G >= 4 && cnt == 4) {
                f = ll_group<T, G >= 4 ? 4 : 1, CB>(diag, A + k0, lda, kb, k0, t, li, lg, S);
            } else if (G >= 3 && cnt == 3) {
                f = ll_group<T, G >= 3 ? 3 : 1, CB>(diag, A + k0, lda, kb, k0, t, li, lg, S);
            } else if (cnt == 2) {
                f = ll_group<T, 2, CB>(diag, A + k0, lda, kb, k0, t, li, lg, S);
            } else if (cnt == 1) {
                f = ll_group<T, 1, CB>(diag, A + k0, lda, kb, k0, t, li, lg, S);
            } else {
                f = ll_group<T, 0, CB>(diag, A + k0, lda, kb, k0, t, li, lg, S);
            }
            if (f) return f;
            base += round;
        }
        __syncthreads();
    }
    return 0;
}

// CB = 2: passes of 32 right-hand sides, few enough registers for four
// waves per SIMD (FP32 POTRF: five, SPOTRF n = 256 x 1,100 177 us, with four 231);
// CB = 4: passes of 64 (L streamed half as often), three.
template <typename T, int MODE, int CB> constexpr int blk_wpe()
{
    return CB != 2 ? 2 : sizeof(T) == 4 && MODE == KB_MODE_POTRF ? 5 : 4;
}

template <typename T, int MODE, int CB, int W>
__global__ void __launch_bounds__(W) __attribute__((amdgpu_waves_per_eu(blk_wpe<T, MODE, CB>())))
k_blk_chol(int n, int nrhs, int side_left, BatchArg<T> A, BatchArg<T> B, int* info, int batch)
{
    __shared__ BlkSmem<T, CB> S;
    for (long mat = blockIdx.x; mat < batch; mat += gridDim.x) {
        T* Ap = uniform(A.get(mat));
        const int lda = uniform(A.ldim(mat));
        int inf = 0;
        if constexpr (MODE == KB_MODE_POTRF) {
            inf = blk_potrf<T, CB, W>(Ap, lda, n, S);
            if (threadIdx.x == 0 && info) info[mat] = inf;
        } else if constexpr (MODE == KB_MODE_POSV) {
            T* Bp = uniform(B.get(mat));
            const int ldb = uniform(B.ldim(mat));
            inf = blk_potrf<T, CB, W>(Ap, lda, n, S, Bp, ldb, side_left, nrhs);
            if (threadIdx.x == 0 && info) info[mat] = inf;
            if (inf == 0) blk_solve_bwd<T, CB, W>(Ap, lda, n, Bp, ldb, side_left, nrhs, S);
        } else {
            blk_solve<T, CB, W>(Ap, lda, n, uniform(B.get(mat)), uniform(B.ldim(mat)), side_left, nrhs, S);
        }
        __syncthreads();
    }
}

// Passes of 32 right-hand sides when the count allows (POTRF: none), else 64.
constexpr int KB_BLK_NARROW = 32;
// Matrices the 256-thread kernel holds at once (256 CUs; registers allow four,
// five or six workgroups).
template <typename T, int MODE> constexpr int blk_held()
{
    if (MODE == KB_MODE_POTRS) return 256 * (sizeof(T) == 8 ? 5 : 6);
    return 256 * (sizeof(T) == 4 && MODE == KB_MODE_POTRF ? 5 : 4);
}

// Two waves per matrix instead of four where a panel has too few row tiles to
// keep three waves busy while the first factors the diagonal block: twice the
// matrices per CU then hide its chain.  Only for batches that the four-wave form
// does not hold at once, and up to the order and right-hand sides where the four
// waves' updates win again (POTRS beyond 2,048 matrices: earlier, the factors in
// flight, read twice, no longer fit the caches).  256 -> 128 threads, us: DPOTRF n = 80 x
// 4,000 152 -> 101, n = 200 x 1,300 to 4,000 0.95 to 1.04 of the time; SPOTRF n = 128 x
// 1,100 53 -> 57, x 1,300 79 -> 59; SPOSV n = 128 x 2,100, 8 right-hand sides 185 ->
// 151; DPOTRS n = 192 x 4,000, 8 right-hand sides 434 -> 394, n = 130, 16 right-hand
// sides, x 1,700 0.98 of the time, x 2,100 156 -> 184; SPOTRS n = 100 x 1,300, 17
// right-hand sides 77 -> 85, x 1,700 0.93 of the time.
template <typename T, int MODE>
static bool blk_two_waves(int n, int nrhs, int batch)
{
    int nmax = 224;
    if (MODE != KB_MODE_POTRF && nrhs > 4) nmax = nrhs <= 16 ? 192 : 128;
    if (MODE == KB_MODE_POTRS && nrhs > 8 && batch > 2048) nmax = nrhs <= 24 ? 128 : 96;
    return n <= nmax && batch > blk_held<T, MODE>();
}

// FP64 POTRS: dynamic LDS that leaves four of five workgroups to a CU, where the
// fifth saves no round or is one of many: it only pushes the factors, read twice,
// out of the caches (n = 200 x 1,300, 32 right-hand sides 385 us, with four 363).
template <typename T, int MODE>
static int blk_pad_lds(int nrhs, int batch)
{
    const bool pad = sizeof(T) == 8 && MODE == KB_MODE_POTRS && nrhs > 8 &&
                     (batch > 2 * 1280 || (batch + 1023) / 1024 == (batch + 1279) / 1280);
    return pad ? 16384 : 0;
}

template <typename T, int MODE>
static void launch_blk_mode(int n, int nrhs, int side_left, BatchArg<T> a, BatchArg<T> b, int* info, int batch,
                            int grid, hipStream_t s)
{
    const bool narrow = MODE == KB_MODE_POTRF || nrhs <= KB_BLK_NARROW;
    if (narrow && blk_two_waves<T, MODE>(n, nrhs, batch))
        // (a CU holds eight, in FP32 POTRS fourteen: n = 128 x 2,100, 8 right-hand
        // sides 1.04 of the four waves' time with 2,048 workgroups, 0.90 with more)
        hipLaunchKernelGGL((k_blk_chol<T, MODE, 2, 128>),
                           dim3(sizeof(T) == 4 && MODE == KB_MODE_POTRS ? min(batch, 4096) : grid), dim3(128), 0, s, n,
                           nrhs, side_left, a, b, info, batch);
    else if (narrow)
        hipLaunchKernelGGL((k_blk_chol<T, MODE, 2, KB_BLK_WG>), dim3(grid), dim3(KB_BLK_WG),
                           (blk_pad_lds<T, MODE>(nrhs, batch)), s, n, nrhs, side_left, a, b, info, batch);
    else
        hipLaunchKernelGGL((k_blk_chol<T, MODE, 4, KB_BLK_WG>), dim3(grid), dim3(KB_BLK_WG), 0, s, n, nrhs, side_left, a,
                           b, info, batch);
}

// Batched lower TRSM for orders above the register range: one sweep of the
// blocked solve, FWD: L X = alpha B, else L^T X = alpha B, for the nrhs
// vectors of B (side_left: columns, else rows, i.e. X op(L) = alpha B as
// op(L)^T X^T = alpha B^T).
template <typename T, bool FWD, int CB>
__global__ void __launch_bounds__(KB_BLK_WG) __attribute__((amdgpu_waves_per_eu(CB == 2 ? 4 : 2)))
k_blk_trsm(int n0, int nrhs0, int side_left, int unit, T alpha, BatchArg<T> A, BatchArg<T> B, int batch,
           const int* vm, const int* vn)
{
    __shared__ BlkSmem<T, CB> S;
    for (long mat = blockIdx.x; mat < batch; mat += gridDim.x) {
        int n = n0, nrhs = nrhs0;
        if (vm) {   // non-uniform: this matrix's order and right-hand-side count
            n = side_left ? vm[mat] : vn[mat];
            nrhs = side_left ? vn[mat] : vm[mat];
            if (n <= 0 || nrhs <= 0) continue;
        }
        if (alpha == T(0)) {
            // B := 0 without reading it (BLAS semantics for alpha = 0)
            T* Bp = B.get(mat);
            const int ldb = B.ldim(mat);
            for (long e = threadIdx.x; e < (long)n * nrhs; e += KB_BLK_WG)
                gst(rhs_elem(Bp, ldb, side_left, (int)(e % n), (int)(e / n)), T(0));
            continue;
        }
        if constexpr (FWD)
            blk_solve_fwd<T, CB>(A.get(mat), A.ldim(mat), n, B.get(mat), B.ldim(mat), side_left, nrhs, S, alpha, unit);
        else
            blk_solve_bwd<T, CB>(A.get(mat), A.ldim(mat), n, B.get(mat), B.ldim(mat), side_left, nrhs, S, alpha, unit);
        __syncthreads();
    }
}

template <typename T>
static int launch_blk_trsm(int fwd, int side_left, int unit, int n, int nrhs, T alpha, kb_mat_t A, kb_mat_t B,
                           const int* vm, const int* vn, int batch, hipStream_t s)
{
    const int grid = batch < 2048 ? batch : 2048;
    BatchArg<T> a = to_arg<T>(A), b = to_arg<T>(B);
    const bool narrow = nrhs <= KB_BLK_NARROW;
    if (fwd && narrow)
        hipLaunchKernelGGL((k_blk_trsm<T, true, 2>), dim3(grid), dim3(KB_BLK_WG), 0, s, n, nrhs, side_left, unit,
                           alpha, a, b, batch, vm, vn);
    else if (fwd)
        hipLaunchKernelGGL((k_blk_trsm<T, true, 4>), dim3(grid), dim3(KB_BLK_WG), 0, s, n, nrhs, side_left, unit,
                           alpha, a, b, batch, vm, vn);
    else if (narrow)
        hipLaunchKernelGGL((k_blk_trsm<T, false, 2>), dim3(grid), dim3(KB_BLK_WG), 0, s, n, nrhs, side_left, unit,
                           alpha, a, b, batch, vm, vn);
    else
        hipLaunchKernelGGL((k_blk_trsm<T, false, 4>), dim3(grid), dim3(KB_BLK_WG), 0, s, n, nrhs, side_left, unit,
                           alpha, a, b, batch, vm, vn);
    return (int)hipGetLastError();
}

template <typename T>
static int launch_blk(int mode, int n, int nrhs, int side_left, kb_mat_t A, kb_mat_t B, int* info,
                      int batch, hipStream_t s)
{
    const int grid = batch < 2048 ? batch : 2048;
    BatchArg<T> a = to_arg<T>(A), b = to_arg<T>(B);
    if (mode == KB_MODE_POTRF)
        launch_blk_mode<T, KB_MODE_POTRF>(n, nrhs, side_left, a, b, info, batch, grid, s);
    else if (mode == KB_MODE_POSV)
        launch_blk_mode<T, KB_MODE_POSV>(n, nrhs, side_left, a, b, info, batch, grid, s);
    else
        launch_blk_mode<T, KB_MODE_POTRS>(n, nrhs, side_left, a, b, info, batch, grid, s);
    return (int)hipGetLastError();
}
