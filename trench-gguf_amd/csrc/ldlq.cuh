// trench-gguf_amd/csrc/ldlq.cuh - the LDLQ error-feedback loop on the device (tools/ldlq.py:71-107, 391-431).
//
// For column block k (256 permuted columns, c0 = 256k) of nmat matrices of ne1 rows:
//   1. the quantizer runs on the strided view of block k of every row (frame.cuh) and writes each row's block
//      into its output slot;
//   2. k_ldlq_solve / k_ldlq_solve16: E = blk - to_float(block bytes) in f32, then Es = E U_BB^-1 by forward substitution in f64:
//      Es[j] = (E[j] - sum_{i<j} Es[i] U[c0+i][c0+j]) / U[c0+j][c0+j], each sum a fused multiply-add chain over i in
//      ascending order (the part over earlier 32-column chunks on the matrix cores);
//   3. k_ldlq_update, an f64 GEMM on the matrix cores: W[r][c] -= (float)(sum_{i<256} Es[r][i] U[c0+i][c]) for the
//      later columns c, each output a fused multiply-add chain over i in ascending order from 0.0.
// The reference leaves the order of those sums to LAPACK / BLAS (numpy's LU solve, torch's solve_triangular and
// GEMM); this library fixes it as above, and its CPU oracle computes the same chains, so the bytes are reproducible
// on any hardware. v_mfma_f64_16x16x4f64 accumulates its four products into each output as four IEEE fused
// multiply-adds in k order (checked bit for bit on gfx950 against a sequential fma chain, subnormal results
// included), so a chain of them over k = 0, 4, ..., 252 is exactly the ascending fma chain; its output layout is
// lane l, element e -> row 4e + l/16, column l%16.
#pragma once
#include "frame.cuh"
#include "dequant.cuh"

#ifndef LDLQ_BK
#define LDLQ_BK 16            // k-chunk of the update GEMM
#endif

typedef double ldlq_d4 __attribute__((ext_vector_type(4)));

// The solve of many rows (fewer go to k_ldlq_solve16, which ends sooner but fills a CU with 16 rows):
// one wave = 64 rows of one matrix (blockIdx.y); the block's 256 columns in chunks of 32. Chunk c:
//   E = blk - to_float(bytes) (f32, then f64), one lane a row, into LDS;
//   E -= Es[:, 0 .. 32c) U[0 .. 32c, chunk] on the f64 matrix cores (each output an fma chain over ascending k,
//   started from E: the serial loop's order), with Es read back (k-major) from the earlier chunks' stores;
//   the 32 x 32 triangle by forward substitution, one lane a row, U's diagonal block broadcast from LDS.
template <int TYPE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_ldlq_solve(const float *__restrict__ W, const uint8_t *__restrict__ q,
                                                   int64_t q_stride, int64_t q_off, const double *__restrict__ U,
                                                   int64_t u_stride, int64_t ne1, int64_t ne0, int64_t c0,
                                                   double *__restrict__ Es, const uint64_t *__restrict__ grid) {
    __shared__ double T[64][33];            // the chunk's 64 rows x 32 columns (33: a row per lane hits distinct banks)
    __shared__ double Ud[32][32];           // U's diagonal block of the chunk
    const int64_t m = blockIdx.y;
    const int lane = lane_id();
    const int64_t row0 = (int64_t)blockIdx.x * 64, row = row0 + lane;
    const bool live = row < ne1;
    const int64_t r = m * ne1 + (live ? row : ne1 - 1);
    const int64_t R = (int64_t)gridDim.y * ne1;            // Es rows (k-major: Es[k * R + r])
    const double *Um = U + m * u_stride;
    const float *wrow = W + r * ne0 + c0;
    const uint8_t *qb = q + r * q_stride + q_off;
    // MFMA operand rows of this lane (rows past the matrix read row ne1 - 1: their results are not stored)
    int64_t arow[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int64_t rr = row0 + 16 * t + lane % 16;
        arow[t] = m * ne1 + (rr < ne1 ? rr : ne1 - 1);
    }
    for (int c = 0; c < 8; ++c) {
        const int64_t cc = c0 + 32 * c;                     // the chunk's first column
        {
            float y[32];
            dq_chunk<TYPE>(qb, c, y, grid);
            const float4 *wp = (const float4 *)(wrow + 32 * c);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const float4 v = wp[t];
                T[lane][4 * t + 0] = (double)(v.x - y[4 * t + 0]);
                T[lane][4 * t + 1] = (double)(v.y - y[4 * t + 1]);
                T[lane][4 * t + 2] = (double)(v.z - y[4 * t + 2]);
                T[lane][4 * t + 3] = (double)(v.w - y[4 * t + 3]);
            }
        }
        {
            const double *up = Um + (cc + lane / 32) * ne0 + cc + lane % 32;
#pragma unroll
            for (int i = 0; i < 16; ++i, up += 2 * ne0) Ud[lane / 32 + 2 * i][lane % 32] = *up;
        }
        wave_sync();
        if (c > 0) {
            ldlq_d4 acc[4][2];
#pragma unroll
            for (int ti = 0; ti < 4; ++ti)
#pragma unroll
                for (int tj = 0; tj < 2; ++tj)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[ti][tj][e] = T[16 * ti + 4 * e + lane / 16][16 * tj + lane % 16];
            // k in steps of 16: the operands of four MFMA k-steps are read together, so one memory latency covers
            // four steps (the MFMAs still run in ascending k)
            for (int k0 = 0; k0 < 32 * c; k0 += 16) {
                double a[4][4], b[4][2];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int k = k0 + 4 * s + lane / 16;
#pragma unroll
                    for (int ti = 0; ti < 4; ++ti) a[s][ti] = -Es[k * R + arow[ti]];
#pragma unroll
                    for (int tj = 0; tj < 2; ++tj) b[s][tj] = Um[(c0 + k) * ne0 + cc + 16 * tj + lane % 16];
                }
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int ti = 0; ti < 4; ++ti)
#pragma unroll
                        for (int tj = 0; tj < 2; ++tj)
                            acc[ti][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s][ti], b[s][tj], acc[ti][tj], 0, 0, 0);
            }
#pragma unroll
            for (int ti = 0; ti < 4; ++ti)
#pragma unroll
                for (int tj = 0; tj < 2; ++tj)
#pragma unroll
                    for (int e = 0; e < 4; ++e) T[16 * ti + 4 * e + lane / 16][16 * tj + lane % 16] = acc[ti][tj][e];
            wave_sync();
        }
        double x[32];
#pragma unroll
        for (int t = 0; t < 32; ++t) x[t] = T[lane][t];
        // (branch-free, the results stored after: a store inside would split the unrolled rows into blocks whose
        // reordering keeps many of U's values live at once)
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            x[i] = x[i] / Ud[i][i];
#pragma unroll
            for (int t = i + 1; t < 32; ++t) x[t] = fma(-x[i], Ud[i][t], x[t]);
        }
        if (live) {
            double *ep = Es + (int64_t)(32 * c) * R + r;
#pragma unroll
            for (int i = 0; i < 32; ++i, ep += R) *ep = x[i];
        }
        // this chunk's Es (stored by other lanes) is read back as MFMA operands by the later chunks
        __threadfence_block();
        wave_sync();
    }
}

// A workgroup of 5 waves owns 16 rows of one matrix (blockIdx.y); E and then Es of the block's 256 columns lie in LDS,
// column by column. E = blk - to_float(bytes) (f32, then f64) comes from 128 threads, one a row and 32-column chunk. The
// 16 x 16 MFMA tiles of E, 16 of them, are dealt to four waves in turn and stay in their accumulators. Chunk c:
//   the two waves that hold its tiles put them into LDS;
//   the fifth wave solves the 32 x 32 triangle by forward substitution: four lanes a row, each with every fourth column,
//   the row's next Es passed to the four by DPP, U's diagonal block in LDS;
//   the four multiply the chunk's Es with U's rows (read while the triangle was solved) into their later tiles, each output
//   an fma chain over ascending k, started from E: the serial loop's order.
// The chain of 256 columns bounds it, so a row is spread over lanes and a matrix over workgroups: 4096 rows (IQ2_S) take
// 25 us, and 135 with k_ldlq_solve, on 64 of the 1024 SIMDs. One workgroup fits a CU (its fifth wave would be the fourth on
// one of the SIMDs, whose registers hold three), so a GPU-full of rows, 16 a CU, takes another 25 us.
//
// x / d, d from U's diagonal: with r = 1 / d correctly rounded (worked out beside the chain), q0 = x r, q1 = q0 + (x - d q0)
// r and q2 = q1 + (x - d q1) r, each residual one fma: q1 lies within an ulp of x / d, so q2 is the correctly rounded
// quotient (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", 1990, theorem 8.7
// of the Handbook of Floating-Point Arithmetic), where no step leaves the normal range: both operands within 2^-500 and
// 2^500, or x is a zero (q0 is the quotient). A chunk with any other operand is solved over with divisions.
#define LDLQ_SR 16            // rows a workgroup
#define LDLQ_TROW 17          // LDS column stride (the tiles' transposed writes spread over the banks)
#define LDLQ_UROW 34
// the value of lane S of each four
template <int S> DEV double quad_bcast(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    constexpr int ctl = S * 0x55;                           // quad_perm [S, S, S, S]
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)b, ctl, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), ctl, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// What column I of the forward substitution reads: lane s of a row's four holds columns 4q + s in x[q]; ud: U's rows,
// column 4q + s at s * 8 + q; dr: the diagonal and its reciprocal
struct LdlqRow {
    double u[8], d, r;
    template <int I> DEV void load(const double (*ud)[LDLQ_UROW], const double (*dr)[2], int s) {
#pragma unroll
        for (int q = I / 4; q < 8; ++q) u[q] = ud[I][s * 8 + q];
        d = dr[I][0];
        r = dr[I][1];
    }
};
// the range of the operands: the high word of the largest magnitude, the least exponent (a zero's counts as 0)
struct LdlqRange {
    int hi, lo;
    DEV void see(double v) {
        hi = imax(hi, (int)((unsigned long long)__double_as_longlong(v) >> 32) & 0x7fffffff);
        lo = imin(lo, __builtin_amdgcn_frexp_exp(v));
    }
    DEV bool mid() const { return hi < (1023 + 500) << 20 && lo > -500; }
};
// Columns I .. 31, each row's results to T. Rows of U are read two columns ahead, and no further, and a column's results
// are worked out in it (the empty asm: left free, the compiler moves the reads up and the later columns' products down, and
// keeps what lies between in scratch). DIV divides.
template <int I, bool DIV> DEV void ldlq_columns(double (&x)[8], const LdlqRow &c0, const LdlqRow &c1,
                                                 const double (*ud)[LDLQ_UROW], const double (*dr)[2], int s,
                                                 double *out, LdlqRange &rg) {
    constexpr int Q = I / 4, S = I % 4;
    LdlqRow c2;
    if constexpr (I < 30) c2.load<I + 2>(ud, dr, s);
    const double v = quad_bcast<S>(x[Q]), d = c0.d;
    double xi;
    if (DIV) {
        xi = v / d;
    } else {
        const double r = c0.r, q0 = v * r, q1 = fma(fma(-d, q0, v), r, q0);
        xi = __builtin_copysign(fma(fma(-d, q1, v), r, q1), q0);         // (a zero's sign is q0's)
        rg.see(v);
    }
    out[I * LDLQ_TROW] = xi;                                // (the four lanes write the same value)
#pragma unroll
    for (int q = Q; q < 8; ++q) x[q] = fma(-xi, c0.u[q], x[q]);          // (columns up to I are not read again)
#pragma unroll
    for (int q = Q; q < 8; ++q) asm volatile("" : "+v"(x[q]));
    asm volatile("" : "+v"(rg.hi), "+v"(rg.lo) :: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (I < 31) ldlq_columns<I + 1, DIV>(x, c1, c2, ud, dr, s, out, rg);
}
// one chunk's triangle, x to be overwritten; false: an operand was out of the short division's range
template <bool DIV> DEV bool ldlq_triangle(double (&x)[8], const double (*ud)[LDLQ_UROW], const double (*dr)[2], int s,
                                           double *out) {
    LdlqRange rg{0, 0};
    if (!DIV) {
        const double d = dr[lane_id() & 31][0];
        rg.see(d);
        rg.lo = d == 0.0 ? -1000 : rg.lo;
    }
    LdlqRow c0, c1;
    c0.load<0>(ud, dr, s);
    c1.load<1>(ud, dr, s);
    ldlq_columns<0, DIV>(x, c0, c1, ud, dr, s, out, rg);
    return DIV || rg.mid();
}

template <int TYPE>
__global__ __launch_bounds__(320) __attribute__((amdgpu_waves_per_eu(3))) void k_ldlq_solve16(
    const float *__restrict__ W, const uint8_t *__restrict__ q, int64_t q_stride, int64_t q_off,
    const double *__restrict__ U, int64_t u_stride, int64_t ne1, int64_t ne0, int64_t c0, double *__restrict__ Es,
    const uint64_t *__restrict__ grid) {
    __shared__ double T[QK][LDLQ_TROW];                     // E, then Es: [column][row]
    __shared__ __align__(16) double Ud[2][32][LDLQ_UROW];                // U's diagonal block of the chunk, of the next one
    __shared__ __align__(16) double Dr[2][32][2];           // and its diagonal, with the reciprocals
    const int64_t m = blockIdx.y, row0 = (int64_t)blockIdx.x * LDLQ_SR;
    const int tid = threadIdx.x, lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t R = (int64_t)gridDim.y * ne1;             // Es rows (k-major: Es[k * R + r])
    const double *Ub = U + m * u_stride + c0 * ne0 + c0;    // the block's diagonal square
    double du[4], dd = 1.0;
    auto load_diag = [&](int c) {
        const double *p = Ub + (int64_t)(32 * c) * ne0 + 32 * c;
#pragma unroll
        for (int j = 0; j < 4; ++j) du[j] = p[(int64_t)((tid >> 5) + 8 * j) * ne0 + (tid & 31)];
        if (tid < 32) dd = p[(int64_t)tid * ne0 + tid];
    };
    auto stash_diag = [&](int c) {
        const int t = tid & 31;
#pragma unroll
        for (int j = 0; j < 4; ++j) Ud[c & 1][(tid >> 5) + 8 * j][(t & 3) * 8 + (t >> 2)] = du[j];
        if (tid < 32) {
            Dr[c & 1][tid][0] = dd;
            Dr[c & 1][tid][1] = 1.0 / dd;
        }
    };
    if (wave < 4) load_diag(0);
    if (tid < 128) {
        const int r = tid & 15, c = tid >> 4;
        // (rows past the matrix read row ne1 - 1: their results are not stored)
        const int64_t gr = m * ne1 + (row0 + r < ne1 ? row0 + r : ne1 - 1);
        const float4 *wp = (const float4 *)(W + gr * ne0 + c0 + 32 * c);
        float y[32];
        dq_chunk<TYPE>(q + gr * q_stride + q_off, c, y, grid);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float4 v = wp[t];
            T[32 * c + 4 * t + 0][r] = (double)(v.x - y[4 * t + 0]);
            T[32 * c + 4 * t + 1][r] = (double)(v.y - y[4 * t + 1]);
            T[32 * c + 4 * t + 2][r] = (double)(v.z - y[4 * t + 2]);
            T[32 * c + 4 * t + 3][r] = (double)(v.w - y[4 * t + 3]);
        }
    }
    if (wave < 4) stash_diag(0);
    __syncthreads();
    const int lx = lane & 15, ly = lane >> 4;
    if (wave == 4) {                                        // the triangles
        const int r = lane >> 2, s = lane & 3;
#pragma unroll 1
        for (int c = 0; c < 8; ++c) {
            __syncthreads();
            double x[8], x0[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = x0[i] = T[32 * c + 4 * i + s][r];
            const bool ok = ldlq_triangle<false>(x, Ud[c & 1], Dr[c & 1], s, &T[32 * c][r]);
            if (__ballot(!ok)) ldlq_triangle<true>(x0, Ud[c & 1], Dr[c & 1], s, &T[32 * c][r]);
            __syncthreads();
        }
        return;
    }
    ldlq_d4 acc[4];                                         // tiles wave, wave + 4, wave + 8, wave + 12
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[u][e] = T[16 * (wave + 4 * u) + lx][4 * e + ly];
    // chunks 2h and 2h + 1: of the wave's tiles, number h is in one of them, and those after it are still to come
    auto half = [&](auto hc) {
        constexpr int h = decltype(hc)::value;
#pragma unroll 1
        for (int c = 2 * h; c < 2 * h + 2; ++c) {
            const bool own = (wave >> 1) == (c & 1), mine = (wave >> 1) > (c & 1);   // tile h is in the chunk / after it
            if (c > 0 && own) {
#pragma unroll
                for (int e = 0; e < 4; ++e) T[16 * (wave + 4 * h) + lx][4 * e + ly] = acc[h][e];
            }
            __syncthreads();
            // the triangle is solved meanwhile
            const double *Uc = Ub + (int64_t)(32 * c + ly) * ne0 + 16 * wave + lx;
            double b[4][8];
            if (mine)
#pragma unroll
                for (int k = 0; k < 8; ++k) b[h][k] = Uc[(int64_t)(4 * k) * ne0 + 64 * h];
#pragma unroll
            for (int u = h + 1; u < 4; ++u)
#pragma unroll
                for (int k = 0; k < 8; ++k) b[u][k] = Uc[(int64_t)(4 * k) * ne0 + 64 * u];
            if (c < 7) {
                load_diag(c + 1);
                stash_diag(c + 1);                          // (the other buffer: last read before the last barrier)
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int k = 32 * c + (tid >> 4) + 16 * j, r = tid & 15;
                if (row0 + r < ne1) Es[k * R + m * ne1 + row0 + r] = T[k][r];
            }
            double a[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) a[k] = -T[32 * c + 4 * k + ly][lx];
            if (mine)                                       // (the next chunk's tiles first: the triangle waits for them)
#pragma unroll
                for (int k = 0; k < 8; ++k) acc[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k], b[h][k], acc[h], 0, 0, 0);
#pragma unroll
            for (int k = 0; k < 8; ++k)
#pragma unroll
                for (int u = h + 1; u < 4; ++u)
                    acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k], b[u][k], acc[u], 0, 0, 0);
        }
    };
    half(std::integral_constant<int, 0>{});
    half(std::integral_constant<int, 1>{});
    half(std::integral_constant<int, 2>{});
    half(std::integral_constant<int, 3>{});
}

// W[m][row][c] -= (float)(sum_i Es[c0+i][m*ne1+row] U_m[c0+i][c]) for c in [cb, ce) (later columns than block
// c0's: cb >= c0 + 256). Es is k-major (Es[k][row], k < 256). A workgroup of 4 waves owns a TT x TT tile, 128
// or 64 a side (each wave a quarter: 4 x 4 or 2 x 2 MFMA tiles of 16 x 16; launch_update chooses); k runs in chunks of 16 staged in LDS, k-major, two buffers (one barrier
// a chunk). A loader thread moves k row t/16, elements t%16 + 16j: 16 lanes read 128 contiguous bytes and write 16
// consecutive LDS doubles; LDS rows are TT + 16 doubles apart (128 B mod 256), so the MFMA operand reads (4 k
// rows x 16 consecutive doubles a wave) and the loader's writes fall in distinct banks.
//
// Tiles are numbered matrix by matrix, and within a matrix in groups of LDLQ_GM row tiles, rows fastest, so that the
// workgroups running together share LDLQ_GM Es panels and as many U panels. The 1-D grid (padded to a multiple of
// 8) is dealt to the 8 XCDs round-robin, so workgroup i takes tile (i % 8) * nper + i / 8: each XCD works through one
// contiguous range of tiles and its L2 holds the panels they share (128 x 256 doubles each, 256 KB; half that for TT 64).
#define LDLQ_GM 8
DEV bool ldlq_tile(int64_t ntr, int64_t ntc, int64_t nmat, int64_t &m, int64_t &tr, int64_t &tc) {
    const int64_t nt = ntr * ntc * nmat, nper = (nt + 7) / 8;
    const int64_t t = (int64_t)(blockIdx.x % 8) * nper + blockIdx.x / 8;
    if (t >= nt) return false;
    const int64_t per = ntr * ntc, u = t % per;
    m = t / per;
    const int64_t gsz = LDLQ_GM * ntc, g = u / gsz, r0 = g * LDLQ_GM;
    const int64_t gm = ntr - r0 < LDLQ_GM ? ntr - r0 : LDLQ_GM;   // rows of this group
    const int64_t v = u % gsz;
    tr = r0 + v % gm;
    tc = v / gm;
    return true;
}
template <int TT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_ldlq_update(
    float *__restrict__ W, const double *__restrict__ Es, const double *__restrict__ U, int64_t u_stride, int64_t nmat,
    int64_t ne1, int64_t ne0, int64_t c0, int64_t cb, int64_t ce) {
    __shared__ __align__(16) double As[2][LDLQ_BK][TT + 16];
    __shared__ __align__(16) double Bs[2][LDLQ_BK][TT + 16];
    int64_t m, tr, tc;
    if (!ldlq_tile((ne1 + TT - 1) / TT, (ce - cb + TT - 1) / TT, nmat, m, tr, tc)) return;
    const int64_t R = nmat * ne1;
    const int64_t row0 = tr * TT;
    const int64_t col0 = cb + tc * TT;
    const double *Um = U + m * u_stride;
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
    constexpr int NT = TT / 32, NL = TT / 16;                  // 16 x 16 tiles a side of the wave's sub-tile; loads
    const int wr0 = (wave >> 1) * (TT / 2), wc0 = (wave & 1) * (TT / 2);
    ldlq_d4 acc[NT][NT];
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[a][b] = ldlq_d4{0.0, 0.0, 0.0, 0.0};
    static_assert(LDLQ_BK * 16 == 256 && (TT == 128 || TT == 64), "loader: 16 k rows x 16 lanes, NL a thread");
    const int lk = tid >> 4, le = tid & 15;
    const double *abase = Es + m * ne1 + row0 + le;          // + k * R + 16 j
    const double *bbase = Um + col0 + le;                     // + (c0 + k) * ne0 + 16 j
    double av[NL], bv[NL];
    // a tile inside the matrix (the usual case) loads unguarded: no per-element branches
    const bool full = row0 + TT <= ne1 && col0 + TT <= ce;
    auto load = [&](int k0) {
        const double *ap = abase + (int64_t)(k0 + lk) * R;
        const double *bp = bbase + (c0 + k0 + lk) * ne0;
        if (full) {
#pragma unroll
            for (int j = 0; j < NL; ++j) av[j] = ap[16 * j];
#pragma unroll
            for (int j = 0; j < NL; ++j) bv[j] = bp[16 * j];
        } else {
#pragma unroll
            for (int j = 0; j < NL; ++j) av[j] = row0 + le + 16 * j < ne1 ? ap[16 * j] : 0.0;
#pragma unroll
            for (int j = 0; j < NL; ++j) bv[j] = col0 + le + 16 * j < ce ? bp[16 * j] : 0.0;
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int j = 0; j < NL; ++j) As[buf][lk][le + 16 * j] = av[j];
#pragma unroll
        for (int j = 0; j < NL; ++j) Bs[buf][lk][le + 16 * j] = bv[j];
    };
    float wv[NT][4][NT];                      // the wave's W values (full tiles: read during the last chunk)
    auto read_w = [&](int i0, int i1) {
#pragma unroll
        for (int i = i0; i < i1; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float *wr = W + (m * ne1 + row0 + wr0 + 16 * i + 4 * e + lane / 16) * ne0 + col0 + wc0 + lane % 16;
#pragma unroll
                for (int j = 0; j < NT; ++j) wv[i][e][j] = wr[16 * j];
            }
    };
    auto chunk = [&](int buf) {             // this wave's MFMAs over the staged k-chunk
#pragma unroll
        for (int ks = 0; ks < LDLQ_BK; ks += 4) {
            const int kk = ks + lane / 16;
            double a[NT], b[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                a[t] = As[buf][kk][wr0 + 16 * t + lane % 16];
                b[t] = Bs[buf][kk][wc0 + 16 * t + lane % 16];
            }
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };
    load(0);
    stash(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 + LDLQ_BK < QK; k0 += LDLQ_BK) {
        load(k0 + LDLQ_BK);                 // the next chunk's global reads overlap this chunk's MFMAs
        chunk(buf);
        stash(buf ^ 1);                     // (the other buffer was last read before the previous barrier)
        __syncthreads();
        buf ^= 1;
    }
    if (full) read_w(0, 1);                 // half the epilogue's reads overlap the last chunk's MFMAs (all of
    chunk(buf);                             // them would not fit in the registers beside the accumulators)
    if (full) read_w(1, NT);
    // epilogue: every W value of the wave's sub-tile is read before the first store (a store between the reads
    // would make each read wait for the one before it); a full tile runs unguarded, so the stores need no
    // per-element branches (and their waits no conservative counts)
    if (full) {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float *wr = W + (m * ne1 + row0 + wr0 + 16 * i + 4 * e + lane / 16) * ne0 + col0 + wc0 + lane % 16;
#pragma unroll
                for (int j = 0; j < NT; ++j) wr[16 * j] = wv[i][e][j] - (float)acc[i][j][e];
            }
        return;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t row = row0 + wr0 + 16 * i + 4 * e + lane / 16;
            const float *wr = W + (m * ne1 + (row < ne1 ? row : 0)) * ne0;
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int64_t col = col0 + wc0 + 16 * j + lane % 16;
                wv[i][e][j] = row < ne1 && col < ce ? wr[col] : 0.f;
            }
        }
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t row = row0 + wr0 + 16 * i + 4 * e + lane / 16;
            if (row >= ne1) continue;
            float *wr = W + (m * ne1 + row) * ne0;
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int64_t col = col0 + wc0 + 16 * j + lane % 16;
                if (col < ce) wr[col] = wv[i][e][j] - (float)acc[i][j][e];
            }
        }
}

// ------------------------------------------------------------------ the 'schur' importance of a block's columns
// tools/ldlq.py:90-93 (and 424-426): qw = diag((U_BB^T U_BB)^-1) of each 256-column diagonal block U_BB, which the
// reference leaves to LAPACK (np.linalg.inv) or torch. Here the order is fixed: (U_BB^T U_BB)^-1 = X X^T with
// X = U_BB^-1, so qw[i] is the squared norm of X's row i. The row comes from X U_BB = I by substitution along it:
//   x_t = ((t == i ? 1 : 0) - acc_t) / U[t][t] for t = i .. 255, acc_t = sum_{s=i}^{t-1} x_s U[s][t],
// each acc_t an fma chain over s ascending from 0.0 (kept as running sums: after x_s, acc_j = fma(x_s, U[s][j], acc_j)
// for the later columns), and qw[i] = (float)(sum_t x_t^2), an fma chain over t ascending from 0.0.
// One wave a row (grid: 256 rows x the blocks): lane L keeps acc for the block's columns L, L+64, L+128, L+192; row
// t + 1 of U is read while row t is used. Columns at or before t are updated too (their sums are no longer read).
// The result goes to nrep rows of w, ne0 apart (matrices that share U).
DEV double readlane_f64(double v, int lane) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__global__ __launch_bounds__(64) void k_schur_weights(const double *__restrict__ U, int64_t ne0, float *__restrict__ w,
                                                      int64_t nrep) {
    const int64_t c0 = (int64_t)blockIdx.y * QK;
    const int i = (int)blockIdx.x, lane = lane_id();
    const double *ub = U + c0 * ne0 + c0;          // U_BB[s][t] = ub[s * ne0 + t]
    double acc[4] = {0.0, 0.0, 0.0, 0.0}, u[4], un[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) u[q] = ub[(int64_t)i * ne0 + 64 * q + lane];
    double ws = 0.0;
    for (int t = i; t < QK; ++t) {
        const int tn = t + 1 < QK ? t + 1 : t;
#pragma unroll
        for (int q = 0; q < 4; ++q) un[q] = ub[(int64_t)tn * ne0 + 64 * q + lane];
        const int qt = t >> 6, lt = t & 63;        // column t: lane lt, slot qt
        const double at = readlane_f64(qt == 0 ? acc[0] : qt == 1 ? acc[1] : qt == 2 ? acc[2] : acc[3], lt);
        const double dt = readlane_f64(qt == 0 ? u[0] : qt == 1 ? u[1] : qt == 2 ? u[2] : u[3], lt);
        const double x = ((t == i ? 1.0 : 0.0) - at) / dt;
        ws = fma(x, x, ws);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            acc[q] = fma(x, u[q], acc[q]);
            u[q] = un[q];
        }
    }
    if (lane == 0)
        for (int64_t r = 0; r < nrep; ++r) w[r * ne0 + c0 + i] = (float)ws;
}
