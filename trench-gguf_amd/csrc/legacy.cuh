// trench-gguf_amd/csrc/legacy.cuh - Q4_0, Q5_0, Q5_1 and F16: the types llama-quantize writes for rows that are not
// whole 256-weight super-blocks (tools/requant_experts.py:180-192, tensor_type_fallback). The reference hands them to
// ggml on the CPU (tools/requant_experts.py:732-747: ggml_quantize_chunk); here they are quantized on the device with
// ggml's rules:
//  - without an imatrix, quantize_row_q4_0_ref / q5_0_ref / q5_1_ref: one scale from the block's extreme value(s),
//    levels by C's float-to-integer conversion;
//  - with one, quantize_row_q4_0_impl / q5_0_impl / q5_1_impl: weights qw * sqrt(sigma2 + x^2) with sigma2 the mean
//    of x^2 over the WHOLE ROW (not a super-block), then make_qx_quants (nmax 8 / 16, rmse_type 1) or
//    make_qkx3_quants (nmax 31, rmin -0.9, rdelta 0.05, 36 steps), the searches the k-quants use
//    (gpuq/gpuq.hip:1427-1466, 1510-1587 restate them);
//  - F16: ggml_fp32_to_fp16_row, each value rounded as GGML_FP32_TO_FP16 (f2h), any row length.
// One lane a 32-weight block (blocks: Q4_0 d qs[16], 18 bytes; Q5_0 d qh[4] qs[16], 22; Q5_1 d m qh[4] qs[16], 24).
#pragma once
#include <float.h>
#include "kquants.cuh"

// C's conversion of a float to an 8-bit integer as ggml's x86 builds perform it: truncation to a 32-bit integer
// (cvttss2si, whose result for NaN or a value out of range is INT_MIN), then the low byte. Finite levels in these
// rules are in range; the invalid case arises only from non-finite or extreme scales.
DEV int trunc_i32_x86(float v) { return (v >= -2147483648.f && v < 2147483648.f) ? (int)v : (int)0x80000000u; }
DEV int trunc_i8(float v) { return (int)(int8_t)(trunc_i32_x86(v) & 0xff); }
DEV uint32_t trunc_u8(float v) { return (uint32_t)trunc_i32_x86(v) & 0xffu; }

// the 16 bytes of low nibbles and the 32 fifth bits of 5-bit levels lv[0..31] (value j in byte j % 16, low nibble
// for j < 16), ggml's Q5 layout
DEV void q5_pack(const uint32_t (&lv)[32], uint8_t *img, int qh_off, int qs_off) {
    uint32_t qh = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        qh |= ((lv[j] & 0x10u) >> 4) << j;
        qh |= ((lv[j + 16] & 0x10u) >> 4) << (j + 16);
    }
    img_or32(img, qh_off, qh);
#pragma unroll
    for (int j = 0; j < 16; j += 2) {
        const uint32_t b0 = (lv[j] & 0x0Fu) | ((lv[j + 16] & 0x0Fu) << 4);
        const uint32_t b1 = (lv[j + 1] & 0x0Fu) | ((lv[j + 17] & 0x0Fu) << 4);
        img_or16(img, qs_off + j, b0 | (b1 << 8));
    }
}

// Q4_0 (NMAX 8) and Q5_0 (NMAX 16): symmetric levels around d = max / -NMAX
template <int NMAX> struct KQ0 {
    static constexpr int BS = 32, G = 1, N = 32, BB = NMAX == 8 ? 18 : 22, TAB = 0;
    static constexpr bool ROWSIG = true;
    static DEV void stage(const QParams &, uint8_t *) {}
    static DEV void quant_rs(const float (&x)[N], const float *qwp, float sigma2, int, uint8_t *img, int boff,
                             uint8_t *, const QParams &) {
        uint32_t lv[32];
        float d;
        if (!qwp) {         // quantize_row_q{4,5}_0_ref
            float amax = 0.0f, mx = 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                if (amax < fabsf(x[j])) {
                    amax = fabsf(x[j]);
                    mx = x[j];
                }
            }
            d = mx / -(float)NMAX;
            const float id = d ? 1.0f / d : 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                const int l = trunc_i8(x[j] * id + (NMAX + 0.5f));
                lv[j] = (uint32_t)imin(2 * NMAX - 1, l) & 0xffu;      // MIN(15 / 31, (int8_t)...) into a uint8_t
            }
        } else {            // quantize_row_q{4,5}_0_impl: make_qx_quants(32, NMAX, x, L, 1, weight)
            float qv[N], w[N];
            load_qw<N>(qwp, qv);
#pragma unroll
            for (int j = 0; j < N; ++j) w[j] = qv[j] * sqrtf(sigma2 + x[j] * x[j]);
            Lv<N> L;
            d = sym_levels<N>(NMAX, x, L, w);
#pragma unroll
            for (int j = 0; j < 32; ++j) lv[j] = L.get(j);
        }
        img_or16(img, boff, f2h(d));
        if (NMAX == 8) {
#pragma unroll
            for (int j = 0; j < 16; j += 2) {   // qs[j] = xi0, then |= xi1 << 4 (a byte: a level of 255 fills it)
                const uint32_t b0 = (lv[j] | (lv[j + 16] << 4)) & 0xffu;
                const uint32_t b1 = (lv[j + 1] | (lv[j + 17] << 4)) & 0xffu;
                img_or16(img, boff + 2 + j, b0 | (b1 << 8));
            }
        } else {
            q5_pack(lv, img, boff + 2, boff + 6);
        }
    }
};
using KQ40 = KQ0<8>;
using KQ50 = KQ0<16>;

// Q5_1: affine levels 0..31, x ~ d * l + m
struct KQ51 {
    static constexpr int BS = 32, G = 1, N = 32, BB = 24, TAB = 0;
    static constexpr bool ROWSIG = true;
    static DEV void stage(const QParams &, uint8_t *) {}
    static DEV void quant_rs(const float (&x)[N], const float *qwp, float sigma2, int, uint8_t *img, int boff,
                             uint8_t *, const QParams &) {
        uint32_t lv[32];
        float d, m;
        if (!qwp) {         // quantize_row_q5_1_ref
            float mn = FLT_MAX, mx = -FLT_MAX;
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                if (x[j] < mn) mn = x[j];
                if (x[j] > mx) mx = x[j];
            }
            d = (mx - mn) / 31;
            m = mn;
            const float id = d ? 1.0f / d : 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) lv[j] = trunc_u8((x[j] - mn) * id + 0.5f);
        } else {            // quantize_row_q5_1_impl: make_qkx3_quants(32, 31, ...), m = -the_min
            float qv[N], w[N];
            load_qw<N>(qwp, qv);
#pragma unroll
            for (int j = 0; j < N; ++j) w[j] = qv[j] * sqrtf(sigma2 + x[j] * x[j]);
            Lv<N> L;
            float the_min;
            d = affine_levels<true, N>(31, x, w, L, the_min, -0.9f, 0.05f, 36, false);
            m = -the_min;
#pragma unroll
            for (int j = 0; j < 32; ++j) lv[j] = L.get(j);
        }
        img_or16(img, boff, f2h(d));
        img_or16(img, boff + 2, f2h(m));
        q5_pack(lv, img, boff + 4, boff + 8);
    }
};

// one source value, decoded as the quantize kernels' loads decode it (SrcLoad)
template <int SRC> DEV float src_value(const uint8_t *raw, int64_t i) {
    if (SRC == T_F32) return ((const float *)raw)[i];
    if (SRC == T_F16) return h2f(((const uint16_t *)raw)[i]);
    if (SRC == T_BF16) return ffrom((uint32_t)((const uint16_t *)raw)[i] << 16);
    if (SRC == T_Q8_0) {
        const uint8_t *blk = raw + (i / 32) * 34;
        const float d = h2f(((const uint16_t *)blk)[0]);
        return (float)(int8_t)blk[2 + i % 32] * d;
    }
    const uint8_t *blk = raw + (i / 32) * 17;          // MXFP4: e2m1 codes {0, 1, 2, 3, 4, 6, 8, 12} and sign
    const int j = (int)(i % 32);
    const uint32_t q = ld_u8(blk + 1 + (j % 16));
    const int c = (int)(j < 16 ? (q & 0x0f) : (q >> 4)), m = c & 7;
    const int v = m < 4 ? m : m < 6 ? 2 * m - 4 : 4 * m - 16;
    return (float)(c & 8 ? -v : v) * e8m0_half(ld_u8(blk));
}

// F16 output: value i of n, one a thread
template <int SRC> __global__ void k_to_f16(const uint8_t *raw, uint16_t *dst, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = f2h(src_value<SRC>(raw, i));
}

// The Q4_0 / Q5_0 / Q5_1 imatrix rules' sigma2 of each row: the sum of x^2 over the row in index order (ggml's
// serial loop: a multiply and an add a value) over the row length. One lane a row, 32 values a step: for short rows and
// for many (launch_rows).
template <int SRC> __global__ void k_rowsig(const uint8_t *raw, float *sig, int64_t rows, int64_t n_per_row) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    float s = 0.f;
    for (int64_t c = 0; c < n_per_row; c += 32) {
        float v[32];
        SrcLoad<SRC, 32>::load(raw, r * n_per_row + c, v);
#pragma unroll
        for (int j = 0; j < 32; ++j) s += v[j] * v[j];
    }
    sig[r] = s / (float)n_per_row;
}

// The same sums, RSW_ROWS rows a workgroup: waves 1..3 read 12 blocks of 32 values of every row, contiguous runs, and put
// their squares into LDS while the first 16 lanes of wave 0, a row each, add up those of the round before (two buffers, one
// barrier a round). The chain of additions bounds it (2048 rows of 7200 BF16 values: 32 us, 10 clocks a value); with a lane a row
// every 32 values wait for their loads besides (109 us).
#define RSW_ROWS 16
#define RSW_UNITS 12
#define RSW_US 36             // LDS floats a block (the blocks' writes in distinct banks)
#define RSW_RS (RSW_UNITS * RSW_US + 4)
template <int SRC> __global__ __launch_bounds__(256) void k_rowsig_wg(const uint8_t *raw, float *sig, int64_t rows,
                                                                      int64_t n_per_row) {
    __shared__ __align__(16) float sq[2][RSW_ROWS][RSW_RS];
    const int64_t r0 = (int64_t)blockIdx.x * RSW_ROWS, nu = n_per_row / 32, rounds = (nu + RSW_UNITS - 1) / RSW_UNITS;
    const int p = (int)threadIdx.x - 64, pr = p / RSW_UNITS, pu = p % RSW_UNITS;
    auto stage = [&](int64_t t) {
        const int64_t u = t * RSW_UNITS + pu;
        if (p < 0 || t >= rounds || u >= nu || r0 + pr >= rows) return;
        float v[32];
        SrcLoad<SRC, 32>::load(raw, (r0 + pr) * n_per_row + u * 32, v);
        float4 *o = (float4 *)&sq[t & 1][pr][pu * RSW_US];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            o[j] = make_float4(v[4 * j] * v[4 * j], v[4 * j + 1] * v[4 * j + 1], v[4 * j + 2] * v[4 * j + 2],
                               v[4 * j + 3] * v[4 * j + 3]);
    };
    const bool sums = threadIdx.x < RSW_ROWS && r0 + threadIdx.x < rows;
    float s = 0.f;
    stage(0);
    __syncthreads();
    for (int64_t t = 0; t < rounds; ++t) {
        stage(t + 1);
        if (sums) {
            const int n = (int)(nu - t * RSW_UNITS < RSW_UNITS ? nu - t * RSW_UNITS : RSW_UNITS);
            const float *q = sq[t & 1][threadIdx.x];
            float4 a[8], b[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) a[j] = ((const float4 *)q)[j];
            for (int u = 0; u < n; ++u) {
                q += u + 1 < n ? RSW_US : 0;                // (the next block's squares are read meanwhile)
#pragma unroll
                for (int j = 0; j < 8; ++j) b[j] = ((const float4 *)q)[j];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    s += a[j].x;
                    s += a[j].y;
                    s += a[j].z;
                    s += a[j].w;
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) a[j] = b[j];
            }
        }
        __syncthreads();
    }
    if (sums) sig[r0 + threadIdx.x] = s / (float)n_per_row;
}
