// trench-gguf_amd/csrc/chol.cuh - the LDLQ factor: U upper with U^T U = A^-1 for a symmetric positive definite A
// (tools/ldlq.py:34-68 of the reference, which factors A, inverts it and factors the inverse in numpy or torch).
//
// Route: A = V V^T with V upper (Cholesky from the last column to the first), then U = V^-1. The factor with a positive
// diagonal is unique, so this is the reference's U, without the explicit inverse: 2/3 n^3 operations instead of 4/3 n^3,
// and an error that grows with the condition of V (the square root of A's).
//
// Everything works in place on the upper triangle of one row-major n x n matrix (n a multiple of 256) in blocks of 128:
//   for block k from the last to the first:
//     k_chol_panel:  V[i][k] = A[i][k] W_k^T for the blocks i above (W_k = V_kk^-1, which has replaced V_kk)
//     k_chol_update: A[i][j] -= V[i][k] V[j][k]^T for i <= j < k; its first workgroup takes the block (k-1, k-1) and goes
//                    on to factor it and invert the factor (chol_diag), beside the others' products, so that the serial
//                    part of a step costs nothing while the rest of the matrix is large
//   then U from the diagonal blocks' inverses by doubling: of neighbouring inverted runs of s blocks, U11 and U22, with
//   V12 between them, U12 = -U11 (V12 U22) (k_tri_mul1, k_tri_mul2; the product in brackets goes, transposed, to the
//   unused lower triangle), s = 1, 2, 4, ...; k_upper_rows clears the lower triangle at the end.
//
// All products run on the f64 matrix cores. 7168 columns take 7.3 ms, where potrf, potri and potrf of rocSOLVER between
// permutation and triangle kernels took 67.6 ms (26 ms of it in their serial 128-column kernels): 56 steps of 48 to 164 us
// (a step's floor is the serial part, 30 us for the block's factor and inverse and 11 us for its update; at the start its
// products, 6.5e9 flops, and 400 MB of A read and written), their panels 0.6 ms, the doubling 2.5 ms (49 to 57 TFLOP/s in
// the two largest steps, 67% of the flops), building and clearing the matrix 0.2 ms. Against a 64-bit factor worked out on
// the CPU the error is 0.87 to 0.95 of what it was from 512 to 7168 columns (1.51e-14 against 1.59e-14 at 7168): the sums
// over a step's 128 columns, and over each 64 in the doubling, are formed on their own before they meet the total.
#pragma once
#include "ldlq.cuh"

#define CH_NB 128
#define CH_AS 18              // LDS row of an [x][k] panel: 18 doubles (a wave's 16 x 4 operand reads in distinct banks)

typedef double ch_d2 __attribute__((ext_vector_type(2), aligned(8)));   // (the matrix is 8-byte aligned)

// the wave's number in its workgroup, as a scalar (branches and addresses that depend on it stay scalar)
DEV int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// The product of a TM x TN output tile over K (a multiple of 16): acc += A B, four waves as WR x 4/WR, k in chunks of 16
// through two LDS buffers (one barrier a chunk). An operand is stored [x][k] (k contiguous) or, with AK / BK, [k][x].
template <int TM, int TN, int WR, bool AK, bool BK> struct ChTile {
    static constexpr int WC = 4 / WR, MI = TM / (16 * WR), NJ = TN / (16 * WC);
    static constexpr int ASZ = AK ? 16 * (TM + 16) : TM * CH_AS, BSZ = BK ? 16 * (TN + 16) : TN * CH_AS;
    static constexpr int LDS = 2 * (ASZ + BSZ);            // doubles
    static constexpr int AL = TM / 32, BL = TN / 32;       // 16-byte loads a thread and chunk
    template <int T, bool KX> static DEV void load(const double *p, int64_t ld, int k0, ch_d2 *v) {
#pragma unroll
        for (int j = 0; j < T / 32; ++j) {
            const int idx = (int)threadIdx.x + 256 * j;
            v[j] = KX ? *(const ch_d2 *)(p + (int64_t)(k0 + idx / (T / 2)) * ld + 2 * (idx % (T / 2)))
                      : *(const ch_d2 *)(p + (int64_t)(idx / 8) * ld + k0 + 2 * (idx % 8));
        }
    }
    template <int T, bool KX> static DEV void stash(double *s, const ch_d2 *v) {
#pragma unroll
        for (int j = 0; j < T / 32; ++j) {
            const int idx = (int)threadIdx.x + 256 * j;
            double *d = KX ? s + (idx / (T / 2)) * (T + 16) + 2 * (idx % (T / 2)) : s + (idx / 8) * CH_AS + 2 * (idx % 8);
            d[0] = v[j].x;
            d[1] = v[j].y;
        }
    }
    // the wave's rows / columns of the tile
    static DEV int row0() { return wave_id() / WC * (16 * MI); }
    static DEV int col0() { return wave_id() % WC * (16 * NJ); }
    template <class F> static DEV void loop(const double *A, int64_t lda, const double *B, int64_t ldb, int K,
                                            double *lds, F &&step) {
        double *As = lds, *Bs = lds + 2 * ASZ;
        ch_d2 av[AL], bv[BL];
        load<TM, AK>(A, lda, 0, av);
        load<TN, BK>(B, ldb, 0, bv);
        stash<TM, AK>(As, av);
        stash<TN, BK>(Bs, bv);
        __syncthreads();
        int buf = 0;
        for (int k0 = 0; k0 < K; k0 += 16) {
            const bool more = k0 + 16 < K;
            if (more) {
                load<TM, AK>(A, lda, k0 + 16, av);
                load<TN, BK>(B, ldb, k0 + 16, bv);
            }
            step(As + buf * ASZ, Bs + buf * BSZ);
            if (more) {
                stash<TM, AK>(As + (buf ^ 1) * ASZ, av);
                stash<TN, BK>(Bs + (buf ^ 1) * BSZ, bv);
            }
            __syncthreads();
            buf ^= 1;
        }
    }
    // operand elements of k-step ks for the 16 rows / columns at x0
    static DEV double fa(const double *s, int x0, int ks) {
        const int x = x0 + (lane_id() & 15), k = ks + (lane_id() >> 4);
        return AK ? s[k * (TM + 16) + x] : s[x * CH_AS + k];
    }
    static DEV double fb(const double *s, int x0, int ks) {
        const int x = x0 + (lane_id() & 15), k = ks + (lane_id() >> 4);
        return BK ? s[k * (TN + 16) + x] : s[x * CH_AS + k];
    }
    // acc += A B, or acc -= A B, k in one ascending chain; with SUM > 0 every SUM values of k are summed on their own
    template <bool NEG, int SUM = 0> static DEV void product(const double *A, int64_t lda, const double *B, int64_t ldb, int K,
                                                double *lds, ldlq_d4 (&acc)[MI][NJ]) {
        const int r0 = row0(), c0 = col0();
        ldlq_d4 part[MI][NJ];
        if (SUM) zero(part);
        ldlq_d4 (&to)[MI][NJ] = SUM ? part : acc;
        int run = 0;
        loop(A, lda, B, ldb, K, lds, [&](const double *as, const double *bs) {
#pragma unroll
            for (int ks = 0; ks < 16; ks += 4) {
                double a[MI], b[NJ];
#pragma unroll
                for (int i = 0; i < MI; ++i) a[i] = NEG ? -fa(as, r0 + 16 * i, ks) : fa(as, r0 + 16 * i, ks);
#pragma unroll
                for (int j = 0; j < NJ; ++j) b[j] = fb(bs, c0 + 16 * j, ks);
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
                        to[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], to[i][j], 0, 0, 0);
            }
            if (SUM && (run += 16) == SUM) {
                run = 0;
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) acc[i][j] += part[i][j];
                zero(part);
            }
        });
        if (SUM) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] += part[i][j];
        }
    }
    static DEV void zero(ldlq_d4 (&acc)[MI][NJ]) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = ldlq_d4{0.0, 0.0, 0.0, 0.0};
    }
    // f(row, column, value) for the wave's outputs (element e of lane l: row 4e + l/16, column l%16)
    template <class F> static DEV void each(ldlq_d4 (&acc)[MI][NJ], F &&f) {
        const int l = lane_id();
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    double v = acc[i][j][e];
                    f(row0() + 16 * i + 4 * e + (l >> 4), col0() + 16 * j + (l & 15), v);
                    acc[i][j][e] = v;
                }
    }
};

// ------------------------------------------------------------------ a diagonal block: its factor's inverse
// A 128 x 128 block, read backwards (row I of M is row 127 - I of the block), is M = L L^T with L lower, and the block's
// W = V_kk^-1 is L^-1 read backwards. M lies in LDS as its 36 lower blocks of 16 x 16 (rows 17 doubles apart: 78,336
// bytes, two workgroups a CU).
#define CHD_ROW 17
#define CHD_BLK (16 * CHD_ROW)
#define CHD_LDS (36 * CHD_BLK)
DEV double *chd_blk(double *M, int bi, int bj) { return M + (bi * (bi + 1) / 2 + bj) * CHD_BLK; }
DEV double *chd_at(double *M, int I, int J) { return chd_blk(M, I >> 4, J >> 4) + (I & 15) * CHD_ROW + (J & 15); }

// One doubling step of L^-1 over runs of S blocks: T = L21 L11^-1, a block row a wave (so that every wave has the same
// number of products), in L21's place, then -L22^-1 T, a block column a wave.
template <int S> DEV void chd_double(double *M) {
    const int w = wave_id(), l = lane_id(), x = l & 15, y = l >> 4;
    const int base = 2 * S * (w / S), ii = w % S;
    ldlq_d4 T[S];
#pragma unroll
    for (int j = 0; j < S; ++j) T[j] = ldlq_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < S; ++k)
#pragma unroll
        for (int ks = 0; ks < 16; ks += 4) {
            const double a = chd_blk(M, base + S + ii, base + k)[x * CHD_ROW + ks + y];
#pragma unroll
            for (int j = 0; j <= k; ++j)
                T[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, chd_blk(M, base + k, base + j)[(ks + y) * CHD_ROW + x],
                                                            T[j], 0, 0, 0);
        }
    // (a wave replaces only the block row that it alone has read)
#pragma unroll
    for (int j = 0; j < S; ++j) {
        double *o = chd_blk(M, base + S + ii, base + j);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[(4 * e + y) * CHD_ROW + x] = T[j][e];
    }
    __syncthreads();
    ldlq_d4 X[S];
#pragma unroll
    for (int i = 0; i < S; ++i) X[i] = ldlq_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < S; ++k)
#pragma unroll
        for (int ks = 0; ks < 16; ks += 4) {
            const double b = chd_blk(M, base + S + k, base + ii)[(ks + y) * CHD_ROW + x];
#pragma unroll
            for (int i = k; i < S; ++i)
                X[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(-chd_blk(M, base + S + i, base + S + k)[x * CHD_ROW + ks + y], b,
                                                            X[i], 0, 0, 0);
        }
    // (and only the block column that it alone has read)
#pragma unroll
    for (int i = 0; i < S; ++i) {
        double *o = chd_blk(M, base + S + i, base + ii);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[(4 * e + y) * CHD_ROW + x] = X[i][e];
    }
    __syncthreads();
}

// A block column of 16: a lane holds a row's 16 values, lanes 0..15 the diagonal block's rows; a column's pivot and the
// pivot rows' values come by readlane. The next pivot's reciprocal square root (the hardware's estimate, error e below
// 2^-23, and one third-order step: it leaves 5/16 e^3, under a rounding) is worked out between the updates of the columns
// after it, so that neither waits for the other: sched_barrier keeps the compiler from putting them back in turn (212
// clocks a column before, 200 after: what is left is the issue of two readlanes and a multiply-add for each value).
DEV void chd_column(double (&a)[16]) {
    double d = readlane_f64(a[0], 0), y = __builtin_amdgcn_rsq(d), e = fma(-(d * y), y, 1.0);
    double r = fma(y * e, fma(0.375, e, 0.5), y);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        a[j] *= r;
        if (j == 15) break;
        auto upd = [&](int k) { a[k] = fma(-a[j], readlane_f64(a[j], k), a[k]); };
        // the columns left after j + 1, in five parts beside the steps of the reciprocal square root
        const int n = 14 - j;
        auto part = [&](int q) {
#pragma unroll
            for (int k = 0; k < 14; ++k)
                if (k < n && k >= n * q / 5 && k < n * (q + 1) / 5) upd(j + 2 + k);
            __builtin_amdgcn_sched_barrier(0);
        };
        upd(j + 1);
        __builtin_amdgcn_sched_barrier(0);
        d = readlane_f64(a[j + 1], j + 1);
        y = __builtin_amdgcn_rsq(d);
        part(0);
        const double h = d * y;
        part(1);
        e = fma(-h, y, 1.0);
        part(2);
        const double ye = y * e, c = fma(0.375, e, 0.5);
        part(3);
        r = fma(ye, c, y);
        part(4);
    }
}

// M (in LDS, complete after the caller's writes) -> L^-1 -> W at D (leading dimension n). A pivot that is not positive and
// finite, or whose reciprocal is not finite, sets *info.
DEV void chol_diag(double *M, double *D, int64_t n, int *info) {
    const int w = wave_id(), l = lane_id(), x = l & 15, y = l >> 4;
    __syncthreads();
#pragma unroll 1
    for (int p = 0; p < 8; ++p) {
        // factor block column p: lanes 16..63 of waves 0..2 hold three blocks below the diagonal block (which each wave
        // factors for itself); the last sixteen lanes of wave 2, which no block needs, hold the unit matrix's rows instead,
        // which become the transposed inverse of the diagonal block's factor. It takes the block's place (nothing reads
        // the factor itself)
        const int pb = l < 16 ? p : p + 3 * w + y;
        const bool live = w < 3 && l >= 16 && pb < 8, unit = w == 2 && y == 3;
        double *src = chd_blk(M, pb < 8 ? pb : p, p);
        double a[16];
        if (w < 3) {
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                a[c] = src[x * CHD_ROW + c];
                if (unit) a[c] = c == x ? 1.0 : 0.0;
            }
        }
        __syncthreads();
        if (w < 3) {
            chd_column(a);
            if (live) {
#pragma unroll
                for (int c = 0; c < 16; ++c) src[x * CHD_ROW + c] = a[c];
            }
            if (unit) {
                double r = a[0];                         // 1 / the square root of pivot x
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    src[c * CHD_ROW + x] = a[c];
                    r = c == x ? a[c] : r;
                }
                if (!(r > 0.0 && r < 0x1p511)) *info = 1;
            }
        }
        __syncthreads();
        // the lower blocks right of it less the column's products: block t of them is in row r, where r(r+1)/2 <= t; each
        // wave takes every fourth, four of them together (two where that is all it has left)
        const int m = 7 - p, nt = m * (m + 1) / 2;
        auto blocks = [&](int t0, auto nu) {
            constexpr int NU = decltype(nu)::value;
            const double *pf[NU], *pg[NU];
            double *o[NU], f[NU][4], g[NU][4], v[NU][4];
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int t = t0 + 4 * u < nt ? t0 + 4 * u : t0;
                const int r = (t >= 1) + (t >= 3) + (t >= 6) + (t >= 10) + (t >= 15) + (t >= 21);
                const int bi = p + 1 + r, bj = p + 1 + t - r * (r + 1) / 2;
                pf[u] = chd_blk(M, bi, p) + x * CHD_ROW + y;
                pg[u] = chd_blk(M, bj, p) + x * CHD_ROW + y;
                o[u] = chd_blk(M, bi, bj) + y * CHD_ROW + x;
            }
#pragma unroll
            for (int u = 0; u < NU; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    f[u][e] = pf[u][4 * e];
                    g[u][e] = pg[u][4 * e];
                }
#pragma unroll
            for (int u = 0; u < NU; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[u][e] = o[u][4 * e * CHD_ROW];
            ldlq_d4 s[NU];
#pragma unroll
            for (int u = 0; u < NU; ++u) s[u] = ldlq_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int u = 0; u < NU; ++u) s[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(f[u][e], g[u][e], s[u], 0, 0, 0);
#pragma unroll
            for (int u = 0; u < NU; ++u)
                if (t0 + 4 * u < nt) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[u][4 * e * CHD_ROW] = v[u][e] - s[u][e];
                }
        };
        int t = w;
        for (; t + 8 < nt; t += 16) blocks(t, IntC<4>());
        if (t < nt) blocks(t, IntC<2>());
        __syncthreads();
    }
    chd_double<1>(M);
    chd_double<2>(M);
    chd_double<4>(M);
    // block (R, C) of W is block (7 - R, 7 - C) of L^-1 read backwards
#pragma unroll 4
    for (int t = 0; t < 16; ++t) {
        const int R = 2 * w + (t >> 3), C = t & 7;
        const double *b = chd_blk(M, 7 - R, R <= C ? 7 - C : 0) + 15 * CHD_ROW + 15;
        double *o = D + (int64_t)(16 * R) * n + 16 * C + x;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = 4 * e + y;
            const double v = b[-r * CHD_ROW - x];
            o[(int64_t)r * n] = R < C || (R == C && r <= x) ? v : 0.0;
        }
    }
}

// the last diagonal block (no update before it); one workgroup
__global__ __launch_bounds__(256) void k_chol_last(double *__restrict__ A, int64_t n, int *__restrict__ info) {
    __shared__ double M[CHD_LDS];
    double *D = A + (n - CH_NB) * n + n - CH_NB;
    const int w = wave_id(), x = lane_id() & 15, y = lane_id() >> 4;
    for (int R = 2 * w; R < 2 * w + 2; ++R) {            // (a row of eight blocks' reads at a time)
        double v[8][4];
#pragma unroll
        for (int C = 0; C < 8; ++C)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[C][e] = D[(int64_t)(16 * R + 4 * e + y) * n + 16 * C + x];
#pragma unroll
        for (int C = 0; C < 8; ++C)
            if (R <= C) {
#pragma unroll
                for (int e = 0; e < 4; ++e) chd_blk(M, 7 - R, 7 - C)[(15 - 4 * e - y) * CHD_ROW + 15 - x] = v[C][e];
            }
    }
    chol_diag(M, D, n, info);
}

// V[i][k] = A[i][k] W_k^T, in place; 32 rows a workgroup, grid 4k
__global__ __launch_bounds__(256) void k_chol_panel(double *__restrict__ A, int64_t n, int64_t k) {
    using G = ChTile<32, CH_NB, 1, false, false>;
    __shared__ __align__(16) double lds[G::LDS];
    double *P = A + (int64_t)blockIdx.x * 32 * n + k * CH_NB;
    const double *W = A + k * CH_NB * n + k * CH_NB;
    ldlq_d4 acc[G::MI][G::NJ];
    G::zero(acc);
    G::product<false>(P, n, W, n, CH_NB, lds, acc);             // (its last barrier: every read of P is done)
    G::each(acc, [&](int r, int c, double v) { P[(int64_t)r * n + c] = v; });
}

// A[i][j] -= V[i][k] V[j][k]^T for the blocks i <= j < k; workgroup 0 takes the block (k-1, k-1), which it also factors, and
// the rest of the grid (k(k+1)/2 - 1 rounded up to a multiple of 8) the other tiles, numbered column by column and dealt to
// the 8 XCDs in contiguous runs.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_chol_update(double *__restrict__ A,
                                                                                            int64_t n, int64_t k,
                                                                                            int *__restrict__ info) {
    using G = ChTile<CH_NB, CH_NB, 2, false, false>;
    __shared__ __align__(16) double lds[G::LDS > CHD_LDS ? G::LDS : CHD_LDS];
    if (blockIdx.x == 0) {
        const int w = wave_id(), l = lane_id();
        double *D = A + (k - 1) * CH_NB * n + (k - 1) * CH_NB;
        const double *P = A + (k - 1) * CH_NB * n + k * CH_NB;
        // the upper triangle's 36 blocks of 16 x 16: waves 0 and 3 the ten of a diagonal quarter, 1 and 2 half of the
        // quarter between them
        const bool tri = w == 0 || w == 3;
        const int r0 = w == 3 ? 64 : 0, c0 = w == 0 ? 0 : w == 2 ? 96 : 64;
        ldlq_d4 acc[4][4];
        auto at = [&](int i, int j, int e) {
            return (int64_t)(r0 + 16 * i + 4 * e + (l >> 4)) * n + c0 + 16 * j + (l & 15);
        };
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.0;
        G::loop(P, n, P, n, CH_NB, lds, [&](const double *as, const double *bs) {
#pragma unroll
            for (int ks = 0; ks < 16; ks += 4) {
                double a[4], b[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) a[i] = G::fa(as, r0 + 16 * i, ks);
                if (tri) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) b[j] = G::fb(bs, c0 + 16 * j, ks);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int j = i; j < 4; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
                } else {
#pragma unroll
                    for (int j = 0; j < 2; ++j) b[j] = G::fb(bs, c0 + 16 * j, ks);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
                }
            }
        });
        // (a row of blocks read at once, the lower halves too: a branch a value would wait for each read in turn)
        const int64_t nj = tri ? 4 : 2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            double d[4][4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) d[j][e] = D[at(i, j < nj ? j : 0, e)];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (j >= nj || (tri && j < i)) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = r0 + 16 * i + 4 * e + (l >> 4), c = c0 + 16 * j + (l & 15);
                    if (r <= c) *chd_at(lds, 127 - r, 127 - c) = d[j][e] - acc[i][j][e];
                }
            }
        }
        chol_diag(lds, D, n, info);
        return;
    }
    const int64_t nt = k * (k + 1) / 2 - 1, nper = (nt + 7) / 8, b = (int64_t)blockIdx.x - 1;
    const int64_t t = (b % 8) * nper + b / 8;
    if (b / 8 >= nper || t >= nt) return;
    int64_t j = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while (j * (j + 1) / 2 > t) --j;
    while ((j + 1) * (j + 2) / 2 <= t) ++j;
    const int64_t i = t - j * (j + 1) / 2;
    double *C = A + i * CH_NB * n + j * CH_NB;
    ldlq_d4 acc[G::MI][G::NJ];
    G::zero(acc);
    G::product<false>(A + i * CH_NB * n + k * CH_NB, n, A + j * CH_NB * n + k * CH_NB, n, CH_NB, lds, acc);
    // (the products are summed on their own first: one rounding at A's magnitude a step instead of 128.) A quarter of the
    // tile is read before the quarter before it is stored
    const int l = lane_id();
    double *Cw = C + (int64_t)(G::row0() + (l >> 4)) * n + G::col0() + (l & 15);
    double c[2][4][G::NJ];
    auto read = [&](int a, double (&v)[4][G::NJ]) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int q = 0; q < G::NJ; ++q) v[e][q] = Cw[(int64_t)(16 * a + 4 * e) * n + 16 * q];
    };
    read(0, c[0]);
#pragma unroll
    for (int a = 0; a < G::MI; ++a) {
        if (a + 1 < G::MI) read(a + 1, c[(a + 1) & 1]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int q = 0; q < G::NJ; ++q) Cw[(int64_t)(16 * a + 4 * e) * n + 16 * q] = c[a & 1][e][q] - acc[a][q][e];
    }
}

// One doubling step over runs of s blocks: pair q joins the blocks [2sq, 2sq + s) and [2sq + s, min(2sq + 2s, nb)).
// k_tri_mul1: (V12 U22)^T to the lower triangle, at the transposed place; k_tri_mul2: U12 = -U11 (V12 U22). Tiles of
// CHT x CHT; a tile's k stops where the triangular operand's zeros begin. Grid (tiles of the longest run squared, pairs);
// tiles with the longest k first.
#define CHT 64
struct TriTile { int64_t r0, c0; int rt, ct, nr, nc; bool in; };   // the pair's rows and columns, the tile
DEV TriTile tri_tile(int64_t n, int64_t s, bool mul1) {
    constexpr int PB = CH_NB / CHT;
    const int64_t nb = n / CH_NB, q = blockIdx.y;
    TriTile t;
    t.r0 = 2 * s * q * CH_NB;
    t.c0 = t.r0 + s * CH_NB;
    t.nr = (int)s * PB;
    const int64_t left = nb - (2 * q + 1) * s;
    t.nc = (int)(left < s ? left : s) * PB;
    const int u = (int)blockIdx.x;
    if (mul1) {                 // k: the columns up to the tile's: the last columns first, rows fastest
        t.rt = u % t.nr;
        t.ct = t.nc - 1 - u / t.nr;
        t.in = t.ct >= 0;
    } else {                    // k: the rows from the tile's on: the first rows first, columns fastest
        t.ct = u % t.nc;
        t.rt = u / t.nc;
        t.in = t.rt < t.nr;
    }
    return t;
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_tri_mul1(double *__restrict__ A, int64_t n, int64_t s) {
    using G = ChTile<CHT, CHT, 2, true, false>;
    __shared__ __align__(16) double lds[G::LDS];
    const TriTile t = tri_tile(n, s, true);
    if (!t.in) return;
    // out[c][r] = sum over k <= c of U22[k][c] V12[r][k]
    ldlq_d4 acc[G::MI][G::NJ];
    G::zero(acc);
    G::product<false, CHT>(A + t.c0 * n + t.c0 + t.ct * CHT, n, A + (t.r0 + t.rt * CHT) * n + t.c0, n, (t.ct + 1) * CHT, lds, acc);
    double *o = A + (t.c0 + t.ct * CHT) * n + t.r0 + t.rt * CHT;
    G::each(acc, [&](int r, int c, double v) { o[(int64_t)r * n + c] = v; });
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_tri_mul2(double *__restrict__ A, int64_t n, int64_t s) {
    using G = ChTile<CHT, CHT, 2, false, false>;
    __shared__ __align__(16) double lds[G::LDS];
    const TriTile t = tri_tile(n, s, false);
    if (!t.in) return;
    // out[r][c] = - sum over k >= r of U11[r][k] T[k][c], T stored transposed
    ldlq_d4 acc[G::MI][G::NJ];
    G::zero(acc);
    const int64_t k0 = t.r0 + t.rt * CHT;
    G::product<true, CHT>(A + k0 * n + k0, n, A + (t.c0 + t.ct * CHT) * n + k0, n, (t.nr - t.rt) * CHT, lds, acc);
    double *o = A + k0 * n + t.c0 + t.ct * CHT;
    G::each(acc, [&](int r, int c, double v) { o[(int64_t)r * n + c] = v; });
}

// Zero the strict lower triangle and add up the squares of the rest, a row a workgroup: the trace of U^T U, by which the
// caller sees whether A was so ill-conditioned that the reference's route has to be asked (gpuq_prepare_hessian_dev). The
// rows' sums go to CH_SUMS sums, in any order: the rule that reads them leaves more room than that makes. 56 us at 7168
// columns, and 48 without the squares.
#define CH_SUMS 64
__global__ __launch_bounds__(256) void k_upper_rows(double *__restrict__ A, int64_t n, double *__restrict__ sums) {
    __shared__ double part[4];
    const int64_t i = blockIdx.x;
    double *row = A + i * n, s = 0.0;
    for (int64_t j = threadIdx.x; j < i; j += 256) row[j] = 0.0;
#pragma unroll 4
    for (int64_t j = (i & ~255ll) + threadIdx.x; j < n; j += 256) {
        const double v = row[j];
        s = fma(v, j < i ? 0.0 : v, s);
    }
    for (int d = 32; d; d >>= 1) s += __shfl_xor(s, d);
    if (lane_id() == 0) part[wave_id()] = s;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(sums + i % CH_SUMS, part[0] + part[1] + part[2] + part[3]);
}

// X = U^T U read backwards (row i of R is row n-1-i of X), the 128-blocks of its upper triangle; grid nb(nb+1)/2. The first
// workgroup clears what the factorization adds to (nz <= 256 doubles)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_utu_reversed(const double *__restrict__ U,
                                                                                             int64_t n,
                                                                                             double *__restrict__ R,
                                                                                             double *__restrict__ z, int nz) {
    using G = ChTile<CH_NB, CH_NB, 2, true, true>;
    __shared__ __align__(16) double lds[G::LDS];
    const int64_t t = blockIdx.x;
    if (t == 0 && (int)threadIdx.x < nz) z[threadIdx.x] = 0.0;
    int64_t p = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while (p * (p + 1) / 2 > t) --p;
    while ((p + 1) * (p + 2) / 2 <= t) ++p;
    const int64_t q = t - p * (p + 1) / 2;               // blocks q <= p of X: its lower triangle, R's upper one
    ldlq_d4 acc[G::MI][G::NJ];
    G::zero(acc);
    G::template product<false>(U + p * CH_NB, n, U + q * CH_NB, n, (int)(q + 1) * CH_NB, lds, acc);
    double *o = R + (n - 1 - p * CH_NB) * n + n - 1 - q * CH_NB;
    G::each(acc, [&](int r, int c, double v) { o[-(int64_t)r * n - c] = v; });
}
