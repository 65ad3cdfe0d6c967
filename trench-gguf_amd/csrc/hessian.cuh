// trench-gguf_amd/csrc/hessian.cuh - the LDLQ Hessian preparation on the device (tools/ldlq.py:34-68 of the
// reference): Hp = Hn[perm][:, perm] with zero-energy columns replaced by unit rows, Hn = H / max(n, 1), plus a ridge
// on the diagonal; U = the upper Cholesky factor of Hp^-1 (chol.cuh). These kernels build Hp and the sums it comes from.
#pragma once
#include "ldlq.cuh"

// d[i] = H[i][i] / nd
__global__ __launch_bounds__(256) void k_hess_diag(const double *__restrict__ H, int64_t ne0, double nd,
                                                   double *__restrict__ d) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < ne0) d[i] = H[i * ne0 + i] / nd;
}

// Hp[i][j] = Hn[perm[i]][perm[j]] (a dead column's row and column zero, its diagonal 1), plus ridge on the diagonal, for
// the 128-blocks of the upper triangle (all that the factorization reads); with REV Hp read backwards, from the same
// entries of H; grid (ceil(ne0 / 256), ne0). The first workgroup clears what the factorization adds to (nz <= 256 doubles)
template <bool REV>
__global__ __launch_bounds__(256) void k_hess_perm(const double *__restrict__ H, int64_t ne0, double nd,
                                                   const int64_t *__restrict__ perm, const uint8_t *__restrict__ dead,
                                                   double ridge, double *__restrict__ Hp, double *__restrict__ z, int nz) {
    const int64_t i = blockIdx.y, j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i == 0 && blockIdx.x == 0 && (int)threadIdx.x < nz) z[threadIdx.x] = 0.0;
    if (j >= ne0 || j / 128 < i / 128) return;
    const int64_t pi = perm[REV ? ne0 - 1 - j : i], pj = perm[REV ? ne0 - 1 - i : j];
    double v = dead[pi] || dead[pj] ? (pi == pj ? 1.0 : 0.0) : H[pi * ne0 + pj] / nd;
    if (i == j) v += ridge;
    Hp[i * ne0 + j] = v;
}

// A[i][i] += r
__global__ __launch_bounds__(256) void k_diag_add(double *__restrict__ A, int64_t ne0, double r) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < ne0) A[i * ne0 + i] += r;
}

// Wp[row][c] = W[row][perm[c]] for rows [0, rows); grid (ceil(ne0 / 256), <= 65535), rows strided by gridDim.y
__global__ __launch_bounds__(256) void k_gather_cols(const float *__restrict__ W, float *__restrict__ Wp,
                                                     const int64_t *__restrict__ perm, int64_t rows, int64_t ne0) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= ne0) return;
    const int64_t pc = perm[c];
    for (int64_t r = blockIdx.y; r < rows; r += gridDim.y) Wp[r * ne0 + c] = W[r * ne0 + pc];
}

// H += X^T X (tools/hessian_from_dump.py:73-79 of the reference: the Hessian sum over activation rows), X [nrows][ne0]
// f32 row-major, H [ne0][ne0] f64; every product exact in f64 and each output an fma chain over the rows in order on
// the f64 matrix cores. A workgroup of 4 waves owns a 128 x 128 tile of the lower triangle and writes its values to
// the mirrored place too (the tiles beside the diagonal blocks; those hold both halves themselves); rows run in chunks
// of 16 staged in LDS as f64 (two buffers, one barrier a chunk). The matrix cores bound it: a chunk's floats are read
// before the last chunk's products and become f64 only after them, on their way into LDS (converted where they are
// read, each chunk would wait for its loads). The 1-D grid holds the triangle's tiles alone and each XCD gets one range
// of them (dealt row by row of a square grid the XCDs' shares differ by 28%), in groups of XTX_GM row tiles, rows
// fastest, whose panels its L2 shares. 4096 rows of 7168 columns: 5.71 -> 3.89 ms with these and without the mirroring
// pass (0.17 ms of it), 54 TFLOP/s of the 73 that a large f64 product reaches (the 1596 tiles are 6.2 for each CU, so
// the last round leaves a tenth of the time idle; 128 x 64 tiles, 12.5 a CU, took 3.96 ms).
#define XTX_BK 16
#define XTX_LDS_ROW 144
#define XTX_GM 8
#define XTX_MROW 17           // LDS row of the mirrored values: a column's 16 rows, spread over the banks
typedef float xtx_f4 __attribute__((ext_vector_type(4), aligned(4)));   // (X is 4-byte aligned)
// the tiles above row tile r
DEV int64_t xtx_before(int64_t r) { return r * (r + 1) / 2; }

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_xtx(
    const float *__restrict__ X, int64_t nrows, int64_t ne0, double *__restrict__ H) {
    __shared__ __align__(16) double As[2][XTX_BK][XTX_LDS_ROW];
    __shared__ __align__(16) double Bs[2][XTX_BK][XTX_LDS_ROW];
    const int64_t nr = ne0 / 128, nt = xtx_before(nr), nper = (nt + 7) / 8;
    const int64_t t = (int64_t)(blockIdx.x % 8) * nper + blockIdx.x / 8;
    if ((int64_t)(blockIdx.x / 8) >= nper || t >= nt) return;   // (uniform)
    int64_t g0 = 0;                                       // the group's first row tile
    while (g0 + XTX_GM < nr && xtx_before(g0 + XTX_GM) <= t) g0 += XTX_GM;
    const int64_t gm = nr - g0 < XTX_GM ? nr - g0 : XTX_GM, u = t - xtx_before(g0), sq = g0 * gm;
    int64_t tr, tc;
    if (u < sq) {                                         // columns that every row of the group has
        tr = g0 + u % gm;
        tc = u / gm;
    } else {                                              // the group's triangle, row by row
        const int64_t v = u - sq;
        int64_t r = 0;
        while (xtx_before(r + 1) <= v) ++r;
        tr = g0 + r;
        tc = g0 + (v - xtx_before(r));
    }
    const int64_t row0 = tr * 128, col0 = tc * 128;
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
    const int wr0 = (wave >> 1) * 64, wc0 = (wave & 1) * 64;
    ldlq_d4 acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = ldlq_d4{0.0, 0.0, 0.0, 0.0};
    const int lk = tid >> 4, le = (tid & 15) * 4;          // loader: chunk row lk, elements le + 64 j .. + 3
    const float *ap = X + row0 + le, *bp = X + col0 + le;
    xtx_f4 av[2], bv[2];
    auto load = [&](int64_t k0) {                          // (rows past the end read the last one: stash clears them)
        const int64_t k = k0 + lk < nrows ? k0 + lk : nrows - 1;
#pragma unroll
        for (int j = 0; j < 2; ++j) av[j] = *(const xtx_f4 *)(ap + k * ne0 + 64 * j);
#pragma unroll
        for (int j = 0; j < 2; ++j) bv[j] = *(const xtx_f4 *)(bp + k * ne0 + 64 * j);
    };
    auto stash = [&](int buf, int64_t k0) {
        const bool in = k0 + lk < nrows;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) As[buf][lk][le + 64 * j + e] = in ? (double)av[j][e] : 0.0;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) Bs[buf][lk][le + 64 * j + e] = in ? (double)bv[j][e] : 0.0;
    };
    load(0);
    stash(0, 0);
    __syncthreads();
    int buf = 0;
    for (int64_t k0 = 0; k0 < nrows; k0 += XTX_BK) {
        const bool more = k0 + XTX_BK < nrows;
        if (more) load(k0 + XTX_BK);
#pragma unroll
        for (int ks = 0; ks < XTX_BK; ks += 4) {
            const int kk = ks + lane / 16;
            double a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[buf][kk][wr0 + 16 * i + lane % 16];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[buf][kk][wc0 + 16 * j + lane % 16];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);                 // (the conversions, which wait for the loads, stay here)
        if (more) stash(buf ^ 1, k0 + XTX_BK);
        __syncthreads();
        buf ^= 1;
    }
    // output element e of lane l: row 4e + l/16, column l%16 of its 16 x 16 tile. A row of four tiles is read before the row
    // before it is stored (read between the stores, each tile would wait for the stores before it). The mirrored values go
    // through the wave's part of LDS, so that 16 lanes store a contiguous run there too: stored from where they are, in runs of
    // four lanes, they cost a call of 16 rows and 512 columns 15.6 us instead of 10.1 (a second pass over H took 12.0)
    const bool mirror = tr != tc;
    double *Hw = H + (row0 + wr0 + lane / 16) * ne0 + col0 + wc0 + lane % 16;
    double *Hm = H + (col0 + wc0 + lane / 16) * ne0 + row0 + wr0 + lane % 16;
    double *S = &As[0][0][0] + wave * (64 * XTX_MROW);    // (the loop's last barrier: nothing reads the panels any more)
    static_assert(4 * 64 * XTX_MROW <= 2 * XTX_BK * XTX_LDS_ROW, "the four waves' mirrored rows of tiles");
    double h[2][4][4];
    auto read = [&](int i, double (&v)[4][4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[j][e] = Hw[(int64_t)(16 * i + 4 * e) * ne0 + 16 * j];
    };
    read(0, h[0]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i < 3) read(i + 1, h[(i + 1) & 1]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double v = h[i & 1][j][e] + acc[i][j][e];
                Hw[(int64_t)(16 * i + 4 * e) * ne0 + 16 * j] = v;
                if (mirror) S[(16 * j + lane % 16) * XTX_MROW + 4 * e + lane / 16] = v;
            }
        if (mirror) {
            wave_sync();
#pragma unroll
            for (int c = 0; c < 16; ++c)
                Hm[(int64_t)(4 * c) * ne0 + 16 * i] = S[(4 * c + lane / 16) * XTX_MROW + lane % 16];
            wave_sync();
        }
    }
}
