// kb_sposv_big.h -- mixed-precision POSV (LAPACK dsposv restated) for the
// orders above the register range of a non-uniform batch: one 256-thread
// workgroup per matrix, persistent over the size-sorted queue.
//
// Per matrix (dsposv, SRC/dsposv.f): B and the lower triangle of A are
// converted to FP32 with the range checks of DLAG2S / DLAT2S (ITER = -2); the
// FP32 copy is factored by the blocked workgroup routine (ITER = -3 on a
// non-positive pivot); x0 = solve32(b); then, at most 30 times, r = b - A x in
// FP64 on the matrix cores (the first one also forms ||A||inf, CTE = ||A||inf
// eps sqrt(n)), stop when every right-hand side has ||r||inf <= ||x||inf CTE
// (ITER = the number of corrections), else r to FP32 (overflow: ITER = -2),
// solve32, x += d.  Every failure ends in the FP64 path (X := B, A := L,
// solve; A then holds L).  The FP32 factor, the inverses of its 16 x 16
// diagonal tiles and the FP32 right-hand sides live in a workspace slot owned
// by the workgroup (sb_slot_floats); orders or right-hand-side counts beyond
// the slot (or the limits below) take the FP64 path directly with ITER = -1,
// dsposv's "full precision for implementation reasons".
//
// Who does what: a wave owns 16 right-hand sides through both sweeps and the
// update of X (no barrier, nothing shared but L); the residual's 32-row blocks
// go round the waves, each with all right-hand sides, operands straight from
// memory.  The FP32 right-hand sides are packed by 16 x 16 tiles in the
// matrix-core layout: lane (c, g) holds rows 4g..4g+3 of right-hand side c, so
// a tile is one 16-byte access per lane, and a product's result is the next
// product's operand.  On 2,000 systems of order 128..512 with 64 right-hand
// sides: 5.6 ms, where sweeps shared by the waves (two barriers per 32 rows, the
// right-hand sides updated in memory at each) and a residual staging X in LDS
// took 13.7 ms.
#pragma once
#include "kb_blk_impl.h"

constexpr int KB_SB_MAX_N = 1024;      // orders served by the mixed path
constexpr int KB_SB_MAX_RHS = 64;      // right-hand sides served by the mixed path
constexpr double KB_SB_FLT_MAX = 3.4028234663852886e38;
constexpr int KB_SB_ITERMAX = 30;

struct SbSmem {
    union {
        BlkSmem<float> f;                  // FP32 factorization
        BlkSmem<double> d;                 // FP64 path
    };
    unsigned long long rn[KB_SB_MAX_RHS];  // max |r| per right-hand side (bits of a non-negative double)
    unsigned long long xn[KB_SB_MAX_RHS];  // max |x| per right-hand side
    double red[KB_BLK_WG / 64];
};

KB_DEV unsigned long long sb_bits(double x) { return __builtin_bit_cast(unsigned long long, __builtin_fabs(x)); }
KB_DEV double sb_val(unsigned long long b) { return __builtin_bit_cast(double, b); }

// Workgroup-wide maximum (NaN wins).
KB_DEV double sb_block_max(double v, SbSmem& S)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = (o > v || o != o) ? o : v;
    }
    if (lane == 0) S.red[wave] = v;
    __syncthreads();
    double m = S.red[0];
#pragma unroll
    for (int w = 1; w < KB_BLK_WG / 64; ++w) {
        const double o = S.red[w];
        m = (o > m || o != o) ? o : m;
    }
    __syncthreads();
    return m;
}

// floats of a slot: the factor (ld n), its diagonal tiles' inverses, the packed
// right-hand sides
constexpr long sb_pad16(long x) { return (x + 15) & ~15L; }
constexpr long sb_slot_floats(long max_n, long max_nrhs)
{
    return (sb_pad16(max_n * max_n) + sb_pad16(max_n) * 16 + sb_pad16(max_n) * sb_pad16(max_nrhs) + 63) & ~63L;
}

// 16-byte loads from addresses aligned to the element only
KB_DEV kb_f4 gld4u(const float* p)
{
    typedef float v __attribute__((ext_vector_type(4), aligned(4)));
    return *(const __attribute__((address_space(1))) v*)p;
}
typedef double kb_d2 __attribute__((ext_vector_type(2)));
KB_DEV kb_d2 gld2u(const double* p)
{
    typedef double v __attribute__((ext_vector_type(2), aligned(8)));
    return *(const __attribute__((address_space(1))) v*)p;
}

// A32 := FP32 copy of the lower triangle of A (ld n), SB_U columns at a time;
// big is set when an entry exceeds FP32 range.
constexpr int SB_U = 16;

KB_DEV void sb_convert(const double* A, int lda, int n, float* A32, bool& big)
{
    for (int j0 = 0; j0 < n; j0 += SB_U) {
        for (int i = (j0 & ~63) + threadIdx.x; i < n; i += KB_BLK_WG) {
            double v[SB_U];
#pragma unroll
            for (int u = 0; u < SB_U; ++u) {
                const int j = min(j0 + u, n - 1);
                v[u] = gld_opaque(A + max(i, j) + (long)j * lda);
            }
#pragma unroll
            for (int u = 0; u < SB_U; ++u) {
                if (j0 + u <= i) {
                    big = big || __builtin_fabs(v[u]) > KB_SB_FLT_MAX;
                    gst(A32 + i + (long)(j0 + u) * n, (float)v[u]);
                }
            }
        }
    }
}

// One wave: z := FP32 copy of right-hand sides 16 cb .. 16 cb + 15 (packed,
// zero beyond n and nrhs); big as above.
KB_DEV void sb_pack(const double* B, int ldb, int side_left, int n, int nrhs, int cb, float* z, bool& big, int lane)
{
    const int li = lane & 15, lg = lane >> 4;
    const int c = 16 * cb + li;
    for (int t0 = 0; 16 * t0 < n; t0 += 2) {
        double v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int row = 16 * (t0 + (e >> 2)) + 4 * lg + (e & 3);
            const bool in = row < n && c < nrhs;
            const double x = gld_opaque(rhs_elem(const_cast<double*>(B), ldb, side_left, in ? row : 0, in ? c : 0));
            v[e] = in ? x : 0.0;
            big = big || __builtin_fabs(v[e]) > KB_SB_FLT_MAX;
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
            if (16 * (t0 + t) < n)
                gst((kb_f4*)(z + (t0 + t) * 256L + 4 * lane),
                    kb_f4{(float)v[4 * t], (float)v[4 * t + 1], (float)v[4 * t + 2], (float)v[4 * t + 3]});
    }
}

constexpr int SB_R = 4;    // 16-row tiles of a sweep's block
constexpr int SB_KT = 4;   // tiles whose products are summed before they are taken from the right-hand side

// rows at or beyond n of a packed tile are zero
KB_DEV kb_f4 sb_clip(kb_f4 v, int row0, int n)
{
#pragma unroll
    for (int s = 0; s < 4; ++s) v[s] = (row0 + s < n) ? v[s] : 0.0f;
    return v;
}

// x + W (c - L x) for a diagonal tile: l and w are this lane's four elements of
// the operands L and W (or their transposes), as in the sweeps.
KB_DEV kb_f4 sb_correct(const float (&l)[4], const float (&w)[4], const kb_f4& c, kb_f4 x)
{
    kb_f4 r = c;
#pragma unroll
    for (int s = 0; s < 4; ++s) r = mfma16x16x4(-l[s], x[s], r);
#pragma unroll
    for (int s = 0; s < 4; ++s) x = mfma16x16x4(w[s], r[s], x);
    return x;
}

// One wave: z := L^-1 z for 16 packed right-hand sides, left-looking by blocks
// of SB_R tiles; W: the inverses of the diagonal tiles (16 x 16, row-major).
// Sums of SB_KT tiles, as in ll_update.  COR: the products with the inverses get
// the correction of ll_solve (both sweeps); without it, a kernel matrix of
// condition 5e12 took up to 19 refinement steps for 7, or none of 30 converged.
template <bool COR>
KB_DEV void sb_fwd(const float* L, int n, const float* W, float* z, int lane)
{
    // formed here, not kept live across the phases of a matrix
    asm volatile("" : "+v"(lane));
    asm volatile("" : "+s"(n), "+s"(L), "+s"(W));
    const int li = lane & 15, lg = lane >> 4;
    const int nt = (n + 15) >> 4;
    float* zl = z + 4 * lane;
    for (int I = 0; I < nt; I += SB_R) {
        const int nr = min(SB_R, nt - I);
        kb_f4 c[SB_R], w[SB_R];
        const float* p[SB_R];
        float ld[SB_R][SB_R][4];   // the block's own tiles below the diagonal
#pragma unroll
        for (int r = 0; r < SB_R; ++r) {
            const int t = min(I + r, nt - 1);
            c[r] = gld((const kb_f4*)(zl + t * 256L));
            w[r] = gld((const kb_f4*)(W + t * 256L + 16 * li + 4 * lg));
            p[r] = L + min(16 * (I + r) + li, n - 1) + 4L * lg * n;
#pragma unroll
            for (int q = 0; q < r; ++q) {
                const float* pd = p[r] + 16L * min(I + q, nt - 1) * n;
#pragma unroll
                for (int s = 0; s < 4; ++s) ld[r][q][s] = gld(pd + (long)min(s, max(n - 1 - 16 * min(I + q, nt - 1) - 4 * lg, 0)) * n);
            }
        }
        float a[2][SB_R][4];
        kb_f4 y[2];
        auto fetch = [&](int x, int J) {
            y[x] = gld((const kb_f4*)(zl + J * 256L));
#pragma unroll
            for (int r = 0; r < SB_R; ++r)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    a[x][r][s] = gld(p[r]);
                    p[r] += (s == 3) ? 13L * n : (long)n;
                }
        };
        kb_f4 acc[SB_R];
        auto mult = [&](int x) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int r = 0; r < SB_R; ++r) acc[r] = mfma16x16x4(a[x][r][s], y[x][s], acc[r]);
        };
        static_assert(SB_R == SB_KT && SB_KT % 2 == 0, "a block's sums are whole, its tiles come in pairs");
        if (I > 0) fetch(0, 0);
        for (int J0 = 0; J0 < I; J0 += SB_KT) {
#pragma unroll
            for (int r = 0; r < SB_R; ++r) acc[r] = kb_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int J = J0; J < J0 + SB_KT; J += 2) {
                fetch(1, J + 1);
                mult(0);
                __builtin_amdgcn_sched_barrier(0);
                if (J + 2 < I) fetch(0, J + 2);
                mult(1);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int r = 0; r < SB_R; ++r) c[r] -= acc[r];
        }
        kb_f4 x[SB_R];
#pragma unroll
        for (int r = 0; r < SB_R; ++r) {
            if (r < nr) {
#pragma unroll
                for (int q = 0; q < r; ++q)
#pragma unroll
                    for (int s = 0; s < 4; ++s) c[r] = mfma16x16x4(-ld[r][q][s], x[q][s], c[r]);
                x[r] = kb_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int s = 0; s < 4; ++s) x[r] = mfma16x16x4(w[r][s], c[r][s], x[r]);
                if (COR) {
                    const int c0 = 16 * (I + r), row = c0 + li;
                    float l[4], wr[4];
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const int col = c0 + 4 * lg + s;
                        const bool in = row < n && col <= row;
                        const float v = gld_opaque(L + (in ? row + (long)col * n : 0));
                        l[s] = in ? v : 0.0f;
                        wr[s] = w[r][s];
                    }
                    x[r] = sb_correct(l, wr, c[r], x[r]);
                }
                x[r] = sb_clip(x[r], 16 * (I + r) + 4 * lg, n);
                gst((kb_f4*)(zl + (I + r) * 256L), x[r]);
            }
        }
    }
}

// One wave: z := L^-T z, then X := (first ? 0 : X) + z for right-hand sides
// 16 cb .. 16 cb + 15; returns the bits of max |x| over this lane's right-hand
// side.
template <bool COR>
KB_DEV unsigned long long sb_bwd(const float* L, int n, const float* W, float* z, int lane, double* X, int ldx,
                                 int side_left, int nrhs, int cb, bool first)
{
    asm volatile("" : "+v"(lane));
    asm volatile("" : "+s"(n), "+s"(L), "+s"(W), "+s"(X), "+s"(ldx));
    const int li = lane & 15, lg = lane >> 4;
    const int nt = (n + 15) >> 4;
    const bool col = 16 * cb + li < nrhs;
    const long rs = side_left ? 1 : ldx;
    double* Xc = X + (col ? 16 * cb + li : 0) * (side_left ? (long)ldx : 1L);
    float* zl = z + 4 * lane;
    unsigned long long xmax = 0;
    for (int I = (nt - 1) / SB_R * SB_R; I >= 0; I -= SB_R) {
        const int nr = min(SB_R, nt - I);
        kb_f4 c[SB_R];
        const float* p[SB_R];
        kb_f4 ld[SB_R][SB_R];   // the block's own tiles below the diagonal, transposed
        float w[SB_R][4];
#pragma unroll
        for (int r = 0; r < SB_R; ++r) {
            const int t = min(I + r, nt - 1);
            c[r] = gld((const kb_f4*)(zl + t * 256L));
#pragma unroll
            for (int s = 0; s < 4; ++s) w[r][s] = gld(W + t * 256L + 16 * (4 * lg + s) + li);
            p[r] = L + (long)min(16 * (I + r) + li, n - 1) * n + 4 * lg;
#pragma unroll
            for (int q = r + 1; q < SB_R; ++q) ld[r][q] = sb_clip(gld4u(p[r] + 16 * min(I + q, nt - 1)), 16 * (I + q) + 4 * lg, n);
        }
        kb_f4 a[2][SB_R], y[2];
        auto fetch = [&](int x, int J) {
            y[x] = gld((const kb_f4*)(zl + J * 256L));
#pragma unroll
            for (int r = 0; r < SB_R; ++r) {
                a[x][r] = gld4u(p[r] + 16 * J);
                if (J == nt - 1) a[x][r] = sb_clip(a[x][r], 16 * J + 4 * lg, n);
            }
        };
        kb_f4 acc[SB_R];
        auto mult = [&](int x) {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int r = 0; r < SB_R; ++r) acc[r] = mfma16x16x4(a[x][r][s], y[x][s], acc[r]);
        };
        const int lo = I + SB_R;
        if (nt > lo) fetch(0, nt - 1);
        for (int J = nt - 1; J >= lo;) {
#pragma unroll
            for (int r = 0; r < SB_R; ++r) acc[r] = kb_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int u = 0; u < SB_KT; ++u) {
                if (J >= lo) {
                    if (J > lo) fetch((u + 1) & 1, J - 1);
                    mult(u & 1);
                    __builtin_amdgcn_sched_barrier(0);
                    --J;
                }
            }
#pragma unroll
            for (int r = 0; r < SB_R; ++r) c[r] -= acc[r];
        }
        kb_f4 x[SB_R];
#pragma unroll
        for (int r = SB_R - 1; r >= 0; --r) {
            if (r < nr) {
                const int row0 = 16 * (I + r) + 4 * lg;
                double xo[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) xo[s] = first ? 0.0 : gld_opaque(Xc + min(row0 + s, n - 1) * rs);
#pragma unroll
                for (int q = SB_R - 1; q > r; --q)
                    if (q < nr) {
#pragma unroll
                        for (int s = 0; s < 4; ++s) c[r] = mfma16x16x4(-ld[r][q][s], x[q][s], c[r]);
                    }
                x[r] = kb_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int s = 0; s < 4; ++s) x[r] = mfma16x16x4(w[r][s], c[r][s], x[r]);
                if (COR) {
                    const int col = 16 * (I + r) + li;
                    float l[4];
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const bool in = row0 + s < n && col <= row0 + s;
                        const float v = gld_opaque(L + (in ? row0 + s + (long)col * n : 0));
                        l[s] = in ? v : 0.0f;
                    }
                    x[r] = sb_correct(l, w[r], c[r], x[r]);
                }
                x[r] = sb_clip(x[r], row0, n);
                gst((kb_f4*)(zl + (I + r) * 256L), x[r]);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    if (col && row0 + s < n) {
                        const double v = xo[s] + (double)x[r][s];
                        gst(Xc + (row0 + s) * rs, v);
                        const unsigned long long bits = sb_bits(v);
                        xmax = bits > xmax ? bits : xmax;
                    }
                }
            }
        }
    }
    return xmax;
}

// max over the four lanes of a wave that share li
KB_DEV unsigned long long sb_lane_max(unsigned long long v)
{
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
        const unsigned long long o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    return v;
}

// R = B - A X for the symmetric A (lower triangle stored), its FP32 copy packed
// in Z, S.rn[c] := max_i |r(i, c)|; ovf set when an |r| exceeds FP32 range.
// NORM: also returns this lane's largest row sum of |A| (valid on lanes
// 0..15).  Wave w takes the 32-row blocks w, w + 4, ... with all right-hand
// sides: 16x16x4 FP64 products over k, K step s of tile J being columns
// 16 J + 4 g + s (g the lane group), so both triangles read whole lines: left
// of the diagonal 16 rows of a column at a time, right of it (by symmetry) 16
// consecutive rows of 16 columns as 16-byte pairs.  Half a tile's operands are
// in flight during the other half's products.
template <int K> struct SbKind { static constexpr int value = K; };

template <int NCB, bool NORM>
KB_DEV double sb_residual(const double* A, int lda, int n, const double* B, int ldb, const double* X, int ldx,
                          int side_left, int nrhs, float* Z, SbSmem& S, bool& ovf)
{
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    asm volatile("" : "+s"(n), "+s"(A), "+s"(lda), "+s"(X), "+s"(ldx));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int li = lane & 15, lg = lane >> 4;
    const int nt = (n + 15) >> 4, full = n >> 4;   // tiles; tiles with 16 rows
    const long xr = side_left ? 1 : ldx;           // X: step between rows
    const double* xp[NCB];
    unsigned long long rmax[NCB];
    double amax = 0.0;
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
        xp[cb] = X + min(16 * cb + li, nrhs - 1) * (side_left ? (long)ldx : 1L);
        rmax[cb] = 0;
    }
    for (int I = 2 * wave; I < nt; I += 2 * (KB_BLK_WG / 64)) {
        kb_d4 acc[2][NCB];
        double asum[2] = {0.0, 0.0};
        int row[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            row[r] = min(16 * (I + r) + li, n - 1);
#pragma unroll
            for (int cb = 0; cb < NCB; ++cb) acc[r][cb] = kb_d4{0.0, 0.0, 0.0, 0.0};
        }
        double a[2][2][2], x[2][2][NCB];   // [buffer][K step of the half][row tile / column block]
        // half h of tile J: columns k, k + 1 with k = 16 J + 4 lg + 2 h; KIND 0:
        // left of the diagonal, 1: right of it, 2: any (the tiles on the
        // diagonal and the last columns, element by element)
        auto fetch = [&](auto kind, int q, int J, int h) {
            constexpr int KIND = decltype(kind)::value;
            const int k = 16 * J + 4 * lg + 2 * h;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const long kk = (KIND == 2) ? min(k + s, n - 1) : k + s;
#pragma unroll
                for (int cb = 0; cb < NCB; ++cb) {
                    const double v = gld(xp[cb] + kk * xr);
                    x[q][s][cb] = (KIND != 2 || k + s < n) ? v : 0.0;
                }
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    if (KIND == 0) a[q][s][r] = gld(A + row[r] + kk * lda);
                    if (KIND == 2) {
                        const double v = gld(A + max((long)row[r], kk) + min((long)row[r], kk) * lda);
                        a[q][s][r] = (k + s < n) ? v : 0.0;
                    }
                }
            }
            if (KIND == 1) {
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const kb_d2 v = gld2u(A + k + (long)row[r] * lda);
                    a[q][0][r] = v[0];
                    a[q][1][r] = v[1];
                }
            }
        };
        auto mult = [&](int q) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    if (NORM) asum[r] += __builtin_fabs(a[q][s][r]);
#pragma unroll
                    for (int cb = 0; cb < NCB; ++cb) acc[r][cb] = mfma16x16x4(a[q][s][r], x[q][s][cb], acc[r][cb]);
                }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto tiles = [&](auto kind, int J0, int J1) {
            if (J0 >= J1) return;
            fetch(kind, 0, J0, 0);
            for (int J = J0; J < J1; ++J) {
                fetch(kind, 1, J, 1);
                mult(0);
                if (J + 1 < J1) fetch(kind, 0, J + 1, 0);
                mult(1);
            }
        };
        tiles(SbKind<0>(), 0, I);
        tiles(SbKind<2>(), I, min(I + 2, nt));
        tiles(SbKind<1>(), I + 2, full);
        if (full > I + 1 && full < nt) tiles(SbKind<2>(), full, nt);
        if (NORM) {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                double t = asum[r];
                t += __shfl_xor(t, 16, 64);
                t += __shfl_xor(t, 32, 64);
                amax = (t > amax || t != t) ? t : amax;   // (a row past n repeats row n - 1)
            }
        }
        // lane (li, lg) register q: row 4 q + lg of the tile, right-hand side li
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if (I + r >= nt) break;
#pragma unroll
            for (int cb = 0; cb < NCB; ++cb) {
                const int col = 16 * cb + li;
                double bv[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int ro = 16 * (I + r) + 4 * q + lg;
                    const bool in = ro < n && col < nrhs;
                    bv[q] = gld_opaque(rhs_elem(const_cast<double*>(B), ldb, side_left, in ? ro : 0, in ? col : 0));
                }
                float* zt = Z + ((long)cb * nt + I + r) * 256;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int ro = 16 * (I + r) + 4 * q + lg;
                    double v = bv[q] - acc[r][cb][q];
                    v = (ro < n && col < nrhs) ? v : 0.0;
                    ovf = ovf || __builtin_fabs(v) > KB_SB_FLT_MAX;
                    const unsigned long long bits = sb_bits(v);
                    rmax[cb] = bits > rmax[cb] ? bits : rmax[cb];
                    gst(zt + 4 * (li + 16 * q) + lg, (float)v);
                }
            }
        }
    }
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
        const unsigned long long m = sb_lane_max(rmax[cb]);
        if (lg == 0 && 16 * cb + li < nrhs) atomicMax(&S.rn[16 * cb + li], m);
    }
    return amax;
}

template <bool NORM>
KB_DEV double sb_residual_n(int ncb, const double* A, int lda, int n, const double* B, int ldb, const double* X,
                            int ldx, int side_left, int nrhs, float* Z, SbSmem& S, bool& ovf)
{
    if (ncb == 1) return sb_residual<1, NORM>(A, lda, n, B, ldb, X, ldx, side_left, nrhs, Z, S, ovf);
    if (ncb == 2) return sb_residual<2, NORM>(A, lda, n, B, ldb, X, ldx, side_left, nrhs, Z, S, ovf);
    if (ncb == 3) return sb_residual<3, NORM>(A, lda, n, B, ldb, X, ldx, side_left, nrhs, Z, S, ovf);
    return sb_residual<4, NORM>(A, lda, n, B, ldb, X, ldx, side_left, nrhs, Z, S, ovf);
}

// One matrix of the mixed path (all threads of the workgroup).  Returns
// (info, iter) through the pointers (written by thread 0).
KB_DEV void sb_sposv_one(long mat, int n, int nrhs, int side_left, double* Ap, int lda, const double* Bp, int ldb,
                         double* Xp, int ldx, float* slot, int* info, int* iter, SbSmem& S)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nt = (n + 15) >> 4, ncb = (nrhs + 15) >> 4;
    static_assert(KB_SB_MAX_RHS <= 16 * (KB_BLK_WG / 64), "a wave for every 16 right-hand sides");
    float* A32 = slot;
    float* W = A32 + sb_pad16((long)n * n);
    float* Z = W + 256L * nt;
    float* z = Z + (long)wave * nt * 256;   // this wave's right-hand sides
    // FP32 range of B and of A
    bool big = false;
    if (wave < ncb) sb_pack(Bp, ldb, side_left, n, nrhs, wave, z, big, lane);
    sb_convert(Ap, lda, n, A32, big);
    double cte = 0.0;
    int iters = 0, cor = 0;
    bool ok = !__syncthreads_or(big);
    if (!ok) {
        iters = -2;
    } else {
        const int f32 = blk_potrf<float>(A32, n, n, S.f, nullptr, 0, 0, 0, W);
        cor = uniform(S.f.grow) & KB_GROW_ANY;
        if (f32 != 0) {
            ok = false;
            iters = -3;
        }
    }
    for (int it = 0; ok; ++it) {
        // x += (L32 L32^T)^-1 r  (r = b at it = 0)
        if (threadIdx.x < KB_SB_MAX_RHS) S.rn[threadIdx.x] = 0ull;
        if (wave < ncb) {
            unsigned long long m;
            if (cor) {
                sb_fwd<true>(A32, n, W, z, lane);
                m = sb_bwd<true>(A32, n, W, z, lane, Xp, ldx, side_left, nrhs, wave, it == 0);
            } else {
                sb_fwd<false>(A32, n, W, z, lane);
                m = sb_bwd<false>(A32, n, W, z, lane, Xp, ldx, side_left, nrhs, wave, it == 0);
            }
            m = sb_lane_max(m);
            if (lane < 16) S.xn[16 * wave + lane] = m;
        }
        __syncthreads();
        // r = b - A x, its FP32 copy in Z
        bool ovf = false;
        if (it == 0) {
            double anrm = sb_residual_n<true>(ncb, Ap, lda, n, Bp, ldb, Xp, ldx, side_left, nrhs, Z, S, ovf);
            anrm = sb_block_max(anrm, S);
            cte = anrm * 1.1102230246251565e-16 * __builtin_sqrt((double)n);
        } else {
            sb_residual_n<false>(ncb, Ap, lda, n, Bp, ldb, Xp, ldx, side_left, nrhs, Z, S, ovf);
        }
        const bool rovf = __syncthreads_or(ovf);
        bool conv = true;
        for (int c = 0; c < nrhs; ++c) conv = conv && (sb_val(S.rn[c]) <= sb_val(S.xn[c]) * cte);
        if (conv) {
            iters = it;
            break;
        }
        if (rovf || it == KB_SB_ITERMAX) {
            ok = false;
            iters = rovf ? -2 : -(KB_SB_ITERMAX + 1);
        }
        __syncthreads();
    }
    int inf = 0;
    if (!ok) {
        // FP64: X := B, A := L, solve
        __syncthreads();
        copy_rhs<double>(Bp, ldb, Xp, ldx, side_left, n, nrhs, threadIdx.x, KB_BLK_WG);
        __syncthreads();
        inf = blk_potrf<double>(Ap, lda, n, S.d, Xp, ldx, side_left, nrhs);
        if (inf == 0) blk_solve_bwd<double>(Ap, lda, n, Xp, ldx, side_left, nrhs, S.d);
    }
    if (threadIdx.x == 0) {
        if (info) info[mat] = inf;
        if (iter) iter[mat] = iters;
    }
}
