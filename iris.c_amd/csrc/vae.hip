/*
 * vae.hip - the VAE decoder's HBM-bound kernels for gfx950, NHWC layout.
 *
 * The decoder (iris_vae_decode, iris_vae.c:835-998) keeps activations
 * channels-last on the device: one pixel's channels are contiguous, so a
 * 3x3 convolution is an implicit GEMM with pixels as rows (iris_hip_conv3x3,
 * gemm.hip) and every kernel here streams whole 16- or 32-byte channel
 * chunks. Replaced reference pieces:
 *   - GroupNorm (iris_group_norm, iris_kernels.c:542-582) + swish
 *     (swish_inplace, iris_vae.c:195): a statistics pass that writes per-block
 *     float64 channel sums, a per-group finalize, and an apply pass that folds
 *     gamma, beta, mean and 1/std into one scale and shift per channel and
 *     writes the bf16 conv input;
 *   - denormalize + unpatchify + post_quant_conv (iris_vae.c:860-897): one
 *     kernel from the NCHW latent to the conv_in input;
 *   - the mid-block attention's softmax and V transpose (iris_vae.c:260-357);
 *   - conv_out 128 -> 3 with its GroupNorm and swish and the [-1,1] -> uint8
 *     conversion (iris_vae.c:968-994): one kernel on f32 MFMA.
 */
#include "iris_internal.h"

#include <mutex>

namespace {

constexpr int NT = 256;
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void load8(const float *p, float v[8]) {
    const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void load8(const uint16_t *p, float v[8]) {
    const uint4 a = *(const uint4 *)p;
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        v[2 * j] = __uint_as_float(w[j] << 16);
        v[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
}
__device__ __forceinline__ uint4 pack8(const float v[8]) {
    uint4 o;
    o.x = (uint32_t)f2bf_hw(v[0]) | ((uint32_t)f2bf_hw(v[1]) << 16);
    o.y = (uint32_t)f2bf_hw(v[2]) | ((uint32_t)f2bf_hw(v[3]) << 16);
    o.z = (uint32_t)f2bf_hw(v[4]) | ((uint32_t)f2bf_hw(v[5]) << 16);
    o.w = (uint32_t)f2bf_hw(v[6]) | ((uint32_t)f2bf_hw(v[7]) << 16);
    return o;
}

/* Per-block group sums of x and x^2 over pixels [b*ppb, (b+1)*ppb):
 * part[(b * G + g) * 2 + {0, 1}], float64. Thread t reads channel chunk
 * t % (C/8) of every (256 / (C/8))-th pixel; the block then sums the threads
 * of each chunk, then the channels of each group, in a fixed order, so the
 * result does not depend on timing. */
template <typename T>
__global__ __launch_bounds__(NT) void gn_stats_kernel(const T *x, int pixels, int C, int G, int ppb, double *part) {
    __shared__ double ls[NT][8], lq[NT][8];
    __shared__ double cs[512], cq[512];
    const int cpr = C >> 3, tid = threadIdx.x, ci = tid % cpr, rows = NT / cpr;
    const int p0 = blockIdx.x * ppb, p1 = min(pixels, p0 + ppb);
    double s[8], q[8];
#pragma unroll
    for (int j = 0; j < 8; j++) s[j] = q[j] = 0.0;
#pragma unroll 4
    for (int p = p0 + tid / cpr; p < p1; p += rows) {
        float v[8];
        load8(x + (size_t)p * C + ci * 8, v);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            s[j] += (double)v[j];
            q[j] += (double)v[j] * (double)v[j];
        }
    }
#pragma unroll
    for (int j = 0; j < 8; j++) {
        ls[tid][j] = s[j];
        lq[tid][j] = q[j];
    }
    __syncthreads();
    for (int c = tid; c < C; c += NT) {
        double a = 0.0, b = 0.0;
        for (int r = 0; r < rows; r++) {
            a += ls[r * cpr + (c >> 3)][c & 7];
            b += lq[r * cpr + (c >> 3)][c & 7];
        }
        cs[c] = a;
        cq[c] = b;
    }
    __syncthreads();
    const int cpg = C / G;
    for (int g = tid; g < G; g += NT) {
        double a = 0.0, b = 0.0;
        for (int c = g * cpg; c < (g + 1) * cpg; c++) {
            a += cs[c];
            b += cq[c];
        }
        part[((size_t)blockIdx.x * G + g) * 2] = a;
        part[((size_t)blockIdx.x * G + g) * 2 + 1] = b;
    }
}

/* One block per group: mean and variance of the group from the per-block
 * partial sums (float64, fixed order), then per channel y = x * a + b with
 * a = gamma / sqrt(var + eps), b = beta - mean * a; ab[c] = a, ab[C + c] = b. */
__global__ __launch_bounds__(NT) void gn_finalize_kernel(const double *part, int nblk, int C, int G,
                                                         const float *gamma, const float *beta, float eps,
                                                         double count, float *ab) {
    __shared__ double rs[NT], rq[NT];
    const int g = blockIdx.x, cpg = C / G, tid = threadIdx.x;
    double s = 0.0, q = 0.0;
    for (int e = tid; e < nblk; e += NT) {
        s += part[((size_t)e * G + g) * 2];
        q += part[((size_t)e * G + g) * 2 + 1];
    }
    rs[tid] = s;
    rq[tid] = q;
    __syncthreads();
    for (int h = NT / 2; h > 0; h >>= 1) {
        if (tid < h) {
            rs[tid] += rs[tid + h];
            rq[tid] += rq[tid + h];
        }
        __syncthreads();
    }
    const double mean = rs[0] / count;
    double var = rq[0] / count - mean * mean;
    if (var < 0.0) var = 0.0;
    const float inv = 1.0f / sqrtf((float)var + eps);
    for (int t = tid; t < cpg; t += NT) {
        const int c = g * cpg + t;
        const float a = inv * gamma[c];
        ab[c] = a;
        ab[C + c] = beta[c] - (float)mean * a;
    }
}

/* y = act(x * ab[c] + ab[C + c]) in bf16, act = swish or identity; raw (if
 * not NULL) receives x itself in bf16 (the input of a 1x1 skip convolution).
 * HBM-bound once its arithmetic is short: the channel of a chunk by a mask (a
 * 64-bit remainder for channel counts that are no power of two), the hardware
 * reciprocal and bf16 conversion on values rounded to bf16 next. 1024 x 1024 x
 * 128 bf16: 129 -> 102 us (5.3 TB/s); f32 in 152-164 (4.9-5.3 TB/s); four
 * 16-byte loads in flight per thread gave nothing more. Error of the swish
 * against float64 after the rounding, 4 M normal values: 1.676549679e-3 with
 * the reciprocal and with an IEEE division (35 and 26 of them not the nearest
 * bf16), which would cost the 1024 x 1024 decode 0.8 %. */
template <typename T>
__global__ __launch_bounds__(NT) void gn_apply_kernel(const T *x, const float *ab, int C, size_t n8, int swish,
                                                      uint16_t *y, uint16_t *raw) {
    const int cpr = C >> 3;
    const bool pow2 = (cpr & (cpr - 1)) == 0;
    for (size_t i = (size_t)blockIdx.x * NT + threadIdx.x; i < n8; i += (size_t)gridDim.x * NT) {
        const int c0 = (pow2 ? (int)i & (cpr - 1) : (int)(i % cpr)) * 8;
        float v[8];
        load8(x + i * 8, v);
        if (raw) *(uint4 *)(raw + i * 8) = pack8(v);
        const float4 a0 = *(const float4 *)(ab + c0), a1 = *(const float4 *)(ab + c0 + 4);
        const float4 b0 = *(const float4 *)(ab + C + c0), b1 = *(const float4 *)(ab + C + c0 + 4);
        const float a[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
        const float b[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float t = v[j] * a[j] + b[j];
            v[j] = swish ? silu_fast(t) : t;
        }
        *(uint4 *)(y + i * 8) = pack8(v);
    }
}

/* Latent [4z][h][w] (NCHW, f32) -> conv_in input [2h][2w][64] bf16:
 * per latent channel x * sc + sh (Flux: sc = sqrt(var + eps), sh = mean) or
 * x / sc + sh (Z-Image: sc = scaling factor, sh = shift); unpatchify 2x2
 * (channel c * 4 + 2 * (oy & 1) + (ox & 1) at (oy / 2, ox / 2) becomes
 * channel c at (oy, ox)); then the 1x1 post_quant_conv when pqw is not NULL;
 * channels z..63 are zero (conv_in's weights are padded to match). A block
 * takes 32 pixels, their z values in LDS, and a thread 8 channels of one
 * pixel: a thread for all 64 of a pixel left most CUs idle. 64 x 64 latent 42 -> 10 us. */
constexpr int FR_PIX = NT / 8;
__global__ __launch_bounds__(NT) void vae_front_kernel(const float *lat, int z, int h, int w, const float *sc,
                                                       const float *sh, int divide, const float *pqw,
                                                       const float *pqb, uint16_t *out) {
    __shared__ float wsh[32 * 33], vs[FR_PIX][33];   /* rows one word apart in the banks */
    if (pqw)
        for (int i = threadIdx.x; i < z * z; i += NT) wsh[i / z * 33 + i % z] = pqw[i];
    const int W2 = 2 * w, npix = 4 * h * w, p0 = blockIdx.x * FR_PIX;
    for (int i = threadIdx.x; i < FR_PIX * z; i += NT) {
        const int q = i % FR_PIX, c = i / FR_PIX, p = p0 + q;
        if (p >= npix) continue;
        const int oy = p / W2, ox = p % W2, ic = c * 4 + (oy & 1) * 2 + (ox & 1);
        const float x = lat[((size_t)ic * h + (oy >> 1)) * w + (ox >> 1)];
        vs[q][c] = divide ? x / sc[ic] + sh[ic] : x * sc[ic] + sh[ic];
    }
    __syncthreads();
    const int q = threadIdx.x >> 3, j0 = (threadIdx.x & 7) * 8;
    if (p0 + q >= npix) return;
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        o[j] = 0.0f;
        if (j0 + j >= z) continue;
        if (pqw) {
            float a = pqb ? pqb[j0 + j] : 0.0f;
            for (int c = 0; c < z; c++) a += wsh[(j0 + j) * 33 + c] * vs[q][c];
            o[j] = a;
        } else {
            o[j] = vs[q][j0 + j];
        }
    }
    *(uint4 *)(out + (size_t)(p0 + q) * 64 + j0) = pack8(o);
}

/* Encoder input: image [3][H][W] f32 (NCHW) -> bf16 [H][W][64], channels
 * 3..63 zero (conv_in's weights are padded to match). */
__global__ __launch_bounds__(NT) void vae_img_in_kernel(const float *img, int npix, uint16_t *out) {
    /* 8 threads a pixel, one 16-byte chunk each: whole lines per store */
    const int p = blockIdx.x * (NT / 8) + (threadIdx.x >> 3), k = threadIdx.x & 7;
    if (p >= npix) return;
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = 0.0f;
    if (k == 0) {
        o[0] = img[p];
        o[1] = img[(size_t)npix + p];
        o[2] = img[2 * (size_t)npix + p];
    }
    *(uint4 *)(out + (size_t)p * 64 + k * 8) = pack8(o);
}

/* Encoder output (iris_vae.c:440-482): moments [h][w][2z] f32 (NHWC) ->
 * optional 1x1 quant_conv (qw [2z][2z]) -> the mean (first z channels) ->
 * patchify 2x2 (channel c at (y, x) becomes channel c * 4 + 2 (y & 1) + (x & 1)
 * at (y / 2, x / 2)) -> per latent channel (x - sh) * sc (Z-Image: scaling,
 * shift; Flux: 1 / sqrt(var + eps), mean) -> latent [4z][h/2][w/2] f32.
 * A block takes EO_PIX pixels and every (pixel, channel) a thread; the
 * pixels' moments and the mean rows of qw sit in LDS (LDS false: too many
 * channels for it, read from memory). One thread per pixel left 240 CUs idle
 * at 64 x 64 moments. 277 -> 8 us. */
constexpr int EO_PIX = 16;
template <bool LDS>
__global__ __launch_bounds__(NT) void vae_enc_out_kernel(const float *mom, int z, int h, int w, const float *qw,
                                                         const float *qb, const float *sc, const float *sh,
                                                         float *lat) {
    extern __shared__ float esh[];
    const int z2 = 2 * z, p0 = blockIdx.x * EO_PIX, np = min(EO_PIX, h * w - p0), lh = h / 2, lw = w / 2;
    const int mstr = LDS ? z2 + 1 : z2;   /* rows one word apart in the banks */
    float *const ws = esh + EO_PIX * (z2 + 1);
    if constexpr (LDS) {
        for (int i = threadIdx.x; i < np * z2; i += NT) esh[i / z2 * mstr + i % z2] = mom[(size_t)p0 * z2 + i];
        if (qw)
            for (int i = threadIdx.x; i < z * z2; i += NT) ws[i] = qw[i];
        __syncthreads();
    }
    for (int i = threadIdx.x; i < EO_PIX * z; i += NT) {
        const int q = i % EO_PIX, c = i / EO_PIX;
        const int y = (p0 + q) / w, x = (p0 + q) % w;
        if (q >= np || (y >> 1) >= lh || (x >> 1) >= lw) continue;
        auto m = [&](int k) { return LDS ? esh[q * mstr + k] : mom[(size_t)(p0 + q) * z2 + k]; };
        float v;
        if (qw) {
            v = qb ? qb[c] : 0.0f;
            for (int k = 0; k < z2; k++) v += (LDS ? ws[c * z2 + k] : qw[(size_t)c * z2 + k]) * m(k);
        } else {
            v = m(c);
        }
        const int lc = c * 4 + (y & 1) * 2 + (x & 1);
        lat[((size_t)lc * lh + (y >> 1)) * lw + (x >> 1)] = (v - sh[lc]) * sc[lc];
    }
}

/* Row softmax from f32 scores to bf16 probabilities, one block per row:
 * pass 1 keeps a running (max, sum of exp) per thread and merges them,
 * pass 2 writes exp(x - max) / sum; columns cols..cols_pad-1 get zero. */
__global__ __launch_bounds__(NT) void softmax_bf16_kernel(const float *s, int ld_s, int cols, uint16_t *p, int ld_p,
                                                          int cols_pad) {
    __shared__ float rm[NT / IRIS_WAVE], rl[NT / IRIS_WAVE];
    const float *row = s + (size_t)blockIdx.x * ld_s;
    uint16_t *prow = p + (size_t)blockIdx.x * ld_p;
    float m = -INFINITY, l = 0.0f;
    for (int c = threadIdx.x * 4; c < cols; c += NT * 4) {
        const float4 x = *(const float4 *)(row + c);
        const float mx = fmaxf(fmaxf(x.x, x.y), fmaxf(x.z, x.w));
        const float nm = fmaxf(m, mx);
        l = l * __expf(m - nm) + __expf(x.x - nm) + __expf(x.y - nm) + __expf(x.z - nm) + __expf(x.w - nm);
        m = nm;
    }
    /* merge (m, l) pairs: wave, then block */
    for (int o = 32; o > 0; o >>= 1) {
        const float om = __shfl_xor(m, o), ol = __shfl_xor(l, o);
        const float nm = fmaxf(m, om);
        l = (m == -INFINITY ? 0.0f : l * __expf(m - nm)) + (om == -INFINITY ? 0.0f : ol * __expf(om - nm));
        m = nm;
    }
    const int wv = threadIdx.x / IRIS_WAVE;
    if ((threadIdx.x & (IRIS_WAVE - 1)) == 0) {
        rm[wv] = m;
        rl[wv] = l;
    }
    __syncthreads();
    float M = rm[0];
    for (int i = 1; i < NT / IRIS_WAVE; i++) M = fmaxf(M, rm[i]);
    float Lsum = 0.0f;
    for (int i = 0; i < NT / IRIS_WAVE; i++) Lsum += rm[i] == -INFINITY ? 0.0f : rl[i] * __expf(rm[i] - M);
    const float inv = 1.0f / Lsum;
    for (int c = threadIdx.x * 4; c < cols_pad; c += NT * 4) {
        uint2 o = make_uint2(0u, 0u);
        if (c < cols) {
            const float4 x = *(const float4 *)(row + c);
            o.x = (uint32_t)f2bf(__expf(x.x - M) * inv) | ((uint32_t)f2bf(__expf(x.y - M) * inv) << 16);
            o.y = (uint32_t)f2bf(__expf(x.z - M) * inv) | ((uint32_t)f2bf(__expf(x.w - M) * inv) << 16);
        }
        *(uint2 *)(prow + c) = o;
    }
}

/* dst[c][r] = src[r][c] for r < rows, 0 for rows <= r < rows_pad; 64x64
 * tiles through LDS (stride 65 keeps the transposed reads conflict-free). */
__global__ __launch_bounds__(NT) void transpose_bf16_kernel(const uint16_t *src, int ld_src, int rows, int cols,
                                                            uint16_t *dst, int ld_dst) {
    __shared__ uint16_t t[64][65];
    const int r0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
    for (int i = threadIdx.x; i < 64 * 64; i += NT) {
        const int r = i / 64, c = i % 64;
        t[r][c] = r0 + r < rows && c0 + c < cols ? src[(size_t)(r0 + r) * ld_src + c0 + c] : (uint16_t)0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * 64; i += NT) {
        const int c = i / 64, r = i % 64;
        if (c0 + c < cols) dst[(size_t)(c0 + c) * ld_dst + r0 + r] = t[r][c];
    }
}

/* conv_out (3x3, cin -> 3, zero padding) and the image conversion:
 * v = conv + bias; u8 = (uint8)(clamp(((v + 1) * 0.5) * 255, 0, 255) + 0.5) in
 * the reference's order of operations; f32 (if not NULL) receives v as
 * [3][H][W]. A pixel's 27 products over its channels (9 taps x 3 outputs) are
 * one row of a matrix product, formed once where the pixel is read, and an
 * output sums the nine of its neighbours' rows: f32 MFMA (the weights are
 * f32), K = cin, the 27 columns in two 16-row tiles. A block takes 30 x 16
 * outputs: with their halo 32 x 18 pixels, 36 groups of 16 for 4 waves, whose
 * rows of 27 (odd: consecutive pixels in different banks) fit in LDS beside
 * the weights twice per CU. A lane holds 8 consecutive channels of its pixel
 * per 32-channel step, the next 128 channels loading while the products of
 * this 128 run. NORM: x is f32 and swish(x * ab[c] + ab[cin + c]) is taken on
 * the way in, without a bf16 pass through memory. Blocks take tiles in order
 * within an XCD's band, so a halo's second reading finds its L2.
 * Bound by its products (64 f32 MFMAs per 16 pixels, halo 1.2 times) with the
 * activation beside them: 1024 x 1024 x 128 in 187 us from f32, which replaces
 * an apply pass of about 155 and a kernel of one thread per output over
 * LDS-staged tiles of 356; from bf16 about 180. */
constexpr int CO_X = 30, CO_Y = 16, CO_W = CO_X + 2, CO_P = CO_W * (CO_Y + 2), CO_N = 27, CO_KC = 128;
constexpr int CO_GW = CO_P / 16 / (NT / IRIS_WAVE);   /* groups of 16 pixels per wave */
static_assert(CO_GW * 16 * (NT / IRIS_WAVE) == CO_P, "whole groups for every wave");

template <typename T, bool NORM>
__global__ __launch_bounds__(NT, 2) void conv_out_kernel(const T *x, const float *ab, int H, int W, int cin,
                                                         const float *wt, const float *bias, uint8_t *rgb, float *f32,
                                                         int tx, int tiles, int per_xcd) {
    extern __shared__ __attribute__((aligned(16))) float cosm[];
    const int nch = (cin + CO_KC - 1) / CO_KC, tid = threadIdx.x, lane = tid & 63, q = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float *rows = cosm, *wl = cosm + CO_P * CO_N, *abl = wl + nch * 32 * CO_KC;
    /* wl[step][tile][half][lane][4]: channels 32 step + 8 (lane / 16) + 4 half.., column 16 tile + lane % 16
     * (columns past the 27th stay unset: their rows of the product are not stored) */
#pragma unroll 5
    for (int i = tid; i < 9 * nch * CO_KC; i += NT) {
        const int tap = i / (nch * CO_KC), c = i % (nch * CO_KC);
        const float4 w4 = ((const float4 *)wt)[(size_t)tap * cin + (c < cin ? c : 0)];
        const float w[3] = {w4.x, w4.y, w4.z};
#pragma unroll
        for (int o = 0; o < 3; o++) {
            const int col = 3 * tap + o, ln = ((c >> 3) & 3) * 16 + (col & 15);
            wl[((c >> 5) << 10) + ((col >> 4) << 9) + (((c >> 2) & 1) << 8) + ln * 4 + (c & 3)] = c < cin ? w[o] : 0.0f;
        }
    }
    if (NORM)
        for (int i = tid; i < 2 * nch * CO_KC; i += NT) {
            const int c = i % (nch * CO_KC);
            abl[i] = c < cin ? ab[i < nch * CO_KC ? c : cin + c] : 0.0f;
        }
    const int items = CO_GW * nch;
    for (int k = blockIdx.x >> 3; k < per_xcd; k += gridDim.x >> 3) {
        const int L = (blockIdx.x & 7) * per_xcd + k;
        if (L >= tiles) break;
        const int x0 = L % tx * CO_X, y0 = L / tx * CO_Y;
        float raw[32];
        auto inside = [&](int it) {
            const int g = wave * CO_GW + it / nch, gy = y0 + (g >> 1) - 1, gx = x0 + (g & 1) * 16 + n - 1;
            return (unsigned)gy < (unsigned)H && (unsigned)gx < (unsigned)W ? gy * W + gx : -1;
        };
        auto load = [&](int it) {
            const int p = inside(it), c0 = it % nch * CO_KC + q * 8;
            const T *src = x + (size_t)(p < 0 ? 0 : p) * cin;
#pragma unroll
            for (int s = 0; s < 4; s++) load8(src + (c0 + 32 * s < cin ? c0 + 32 * s : 0), raw + 8 * s);
        };
        load(0);
        __syncthreads();   /* wl and abl are there; the last tile's rows are read */
        f32x4 acc[2];
#pragma unroll 1
        for (int it = 0; it < items; it++) {
            const int ch = it % nch, c0 = ch * CO_KC + q * 8;
            const bool in = inside(it) >= 0;
            float v[32];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const uint32_t keep = in && c0 + 32 * s < cin ? ~0u : 0u;
                float a[8], b[8];
                if (NORM) {
                    load8(abl + c0 + 32 * s, a);
                    load8(abl + nch * CO_KC + c0 + 32 * s, b);
                }
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float t = raw[8 * s + j];
                    v[8 * s + j] = __uint_as_float(__float_as_uint(NORM ? silu_fast(t * a[j] + b[j]) : t) & keep);
                }
            }
            if (it + 1 < items) load(it + 1);
            if (ch == 0) acc[0] = acc[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const float *w = wl + ((ch * 4 + s) << 10) + lane * 4;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const f32x4 w0 = *(const f32x4 *)(w + 256 * h), w1 = *(const f32x4 *)(w + 512 + 256 * h);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(w0[e], v[8 * s + 4 * h + e], acc[0], 0, 0, 0);
                        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[e], v[8 * s + 4 * h + e], acc[1], 0, 0, 0);
                    }
                }
            }
            if (ch == nch - 1) {
                float *o = rows + ((wave * CO_GW + it / nch) * 16 + n) * CO_N + 4 * q;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    o[r] = acc[0][r];
                    if (16 + 4 * q + r < CO_N) o[16 + r] = acc[1][r];
                }
            }
        }
        __syncthreads();
        for (int i = tid; i < CO_X * CO_Y; i += NT) {
            const int px = i % CO_X, py = i / CO_X, xx = x0 + px, yy = y0 + py;
            if (xx >= W || yy >= H) continue;
            float o[3] = {bias[0], bias[1], bias[2]};
#pragma unroll
            for (int tap = 0; tap < 9; tap++) {
                const float *r = rows + ((py + tap / 3) * CO_W + px + tap % 3) * CO_N + 3 * tap;
                o[0] += r[0];
                o[1] += r[1];
                o[2] += r[2];
            }
            const int p = yy * W + xx;
#pragma unroll
            for (int ch = 0; ch < 3; ch++) {
                if (f32) f32[(size_t)ch * H * W + p] = o[ch];
                float val = (o[ch] + 1.0f) * 0.5f;
                val = val * 255.0f;
                if (val < 0) val = 0;
                if (val > 255) val = 255;
                rgb[(size_t)p * 3 + ch] = (uint8_t)(val + 0.5f);
            }
        }
    }
}

template <typename T, bool NORM>
int launch_conv_out(const T *x, const float *ab, int H, int W, int cin, const float *wt, const float *bias,
                    uint8_t *rgb, float *f32) {
    const int tx = (W + CO_X - 1) / CO_X, tiles = tx * ((H + CO_Y - 1) / CO_Y), per_xcd = (tiles + 7) / 8;
    const int nch = (cin + CO_KC - 1) / CO_KC, round = (2 * iris_cu_count() + 7) / 8;
    constexpr size_t most = sizeof(float) * (CO_P * CO_N + 2 * CO_KC * (32 + 2));   /* cin <= 256 */
    const size_t smem = sizeof(float) * (CO_P * CO_N + nch * CO_KC * (32 + 2));
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    std::call_once(once, [] {
        attr = hipFuncSetAttribute((const void *)conv_out_kernel<T, NORM>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)most);
    });
    if (iris_check(attr, "conv_out smem attribute")) return -1;
    IRIS_LAUNCH((conv_out_kernel<T, NORM>), dim3(8 * (per_xcd < round ? per_xcd : round)), dim3(NT), smem,
                iris_stream(), x, ab, H, W, cin, wt, bias, rgb, f32, tx, tiles, per_xcd);
    return iris_launch_check("conv_out_kernel");
}

unsigned blocks_for(size_t n) {
    const size_t b = (n + NT - 1) / NT;
    return (unsigned)(b < 65536 ? b : 65536);
}

}  // namespace

extern "C" int iris_hip_gn_stats(const void *x, int is_bf16, int pixels, int C, int groups, double *part, int nblk) {
    if (!x || !part || pixels <= 0 || nblk <= 0) return iris_set_error("gn_stats: bad arguments");
    if (C < 64 || C > 512 || (C & (C - 1))) return iris_set_error("gn_stats: C=%d (a power of two in 64..512)", C);
    if (groups <= 0 || C % groups) return iris_set_error("gn_stats: %d groups of %d channels", groups, C);
    if ((uintptr_t)x & 15) return iris_set_error("gn_stats: x must be 16-byte aligned");
    const int ppb = (pixels + nblk - 1) / nblk;
    const int used = (pixels + ppb - 1) / ppb;
    if (is_bf16)
        IRIS_LAUNCH(gn_stats_kernel<uint16_t>, dim3(used), dim3(NT), 0, iris_stream(), (const uint16_t *)x,
                           pixels, C, groups, ppb, part);
    else
        IRIS_LAUNCH(gn_stats_kernel<float>, dim3(used), dim3(NT), 0, iris_stream(), (const float *)x, pixels,
                           C, groups, ppb, part);
    if (iris_launch_check("gn_stats_kernel")) return -1;
    return used;
}

extern "C" int iris_hip_gn_finalize(const double *part, int nblk, int pixels, int C, int groups, const float *gamma,
                                    const float *beta, float eps, float *ab) {
    if (!part || !gamma || !beta || !ab || nblk <= 0 || groups <= 0 || C % groups)
        return iris_set_error("gn_finalize: bad arguments");
    const double count = (double)pixels * (C / groups);
    IRIS_LAUNCH(gn_finalize_kernel, dim3(groups), dim3(NT), 0, iris_stream(), part, nblk, C, groups, gamma,
                       beta, eps, count, ab);
    return iris_launch_check("gn_finalize_kernel");
}

extern "C" int iris_hip_gn_apply(const void *x, int is_bf16, const float *ab, int pixels, int C, int swish,
                                 uint16_t *y, uint16_t *raw) {
    if (!x || !ab || !y || pixels <= 0 || C % 8 || ((uintptr_t)x & 15) || ((uintptr_t)y & 15) ||
        ((uintptr_t)raw & 15) || ((uintptr_t)ab & 15))
        return iris_set_error("gn_apply: bad arguments");
    const size_t n8 = (size_t)pixels * C / 8;
    if (is_bf16)
        IRIS_LAUNCH(gn_apply_kernel<uint16_t>, dim3(blocks_for(n8)), dim3(NT), 0, iris_stream(),
                           (const uint16_t *)x, ab, C, n8, swish, y, raw);
    else
        IRIS_LAUNCH(gn_apply_kernel<float>, dim3(blocks_for(n8)), dim3(NT), 0, iris_stream(), (const float *)x,
                           ab, C, n8, swish, y, raw);
    return iris_launch_check("gn_apply_kernel");
}

extern "C" int iris_hip_vae_front(uint16_t *out, const float *lat, int z, int h, int w, const float *sc,
                                  const float *sh, int divide, const float *pqw, const float *pqb) {
    if (!out || !lat || !sc || !sh || z <= 0 || z > 32 || h <= 0 || w <= 0 || ((uintptr_t)out & 15))
        return iris_set_error("vae_front: bad arguments (z=%d, %dx%d)", z, h, w);
    const int npix = 4 * h * w;
    IRIS_LAUNCH(vae_front_kernel, dim3((npix + FR_PIX - 1) / FR_PIX), dim3(NT), 0, iris_stream(), lat, z, h, w, sc, sh,
                       divide, pqw, pqb, out);
    return iris_launch_check("vae_front_kernel");
}

extern "C" int iris_hip_softmax_bf16(uint16_t *p, int ld_p, int cols_pad, const float *s, int ld_s, int rows,
                                     int cols) {
    if (!p || !s || rows <= 0 || cols <= 0 || cols % 4 || ld_s % 4 || ld_p % 4 || cols_pad % 4 || cols_pad < cols ||
        ld_s < cols || ld_p < cols_pad || ((uintptr_t)s & 15) || ((uintptr_t)p & 7))
        return iris_set_error("softmax_bf16: bad shape (rows %d cols %d pad %d ld %d/%d)", rows, cols, cols_pad, ld_s,
                              ld_p);
    IRIS_LAUNCH(softmax_bf16_kernel, dim3(rows), dim3(NT), 0, iris_stream(), s, ld_s, cols, p, ld_p, cols_pad);
    return iris_launch_check("softmax_bf16_kernel");
}

extern "C" int iris_hip_transpose_bf16(uint16_t *dst, int ld_dst, int rows_pad, const uint16_t *src, int ld_src,
                                       int rows, int cols) {
    if (!dst || !src || rows <= 0 || cols <= 0 || rows_pad < rows || rows_pad % 64 || ld_dst < rows_pad ||
        ld_src < cols)
        return iris_set_error("transpose_bf16: bad shape");
    IRIS_LAUNCH(transpose_bf16_kernel, dim3(rows_pad / 64, (cols + 63) / 64), dim3(NT), 0, iris_stream(), src,
                       ld_src, rows, cols, dst, ld_dst);
    return iris_launch_check("transpose_bf16_kernel");
}

static bool conv_out_ok(const uint8_t *rgb, const void *x, int H, int W, int cin, const float *wt, const float *bias) {
    return rgb && x && wt && bias && H > 0 && W > 0 && H <= 32768 && W <= 32768 && cin > 0 && cin <= 256 &&
           cin % 8 == 0 && !((uintptr_t)x & 15) && !((uintptr_t)wt & 15);
}

extern "C" int iris_hip_vae_conv_out(uint8_t *rgb, float *f32, const uint16_t *g, int H, int W, int cin,
                                     const float *wt, const float *bias) {
    if (!conv_out_ok(rgb, g, H, W, cin, wt, bias)) return iris_set_error("vae_conv_out: bad arguments");
    return launch_conv_out<uint16_t, false>(g, NULL, H, W, cin, wt, bias, rgb, f32);
}

extern "C" int iris_hip_vae_conv_out_norm(uint8_t *rgb, float *f32, const float *x, const float *ab, int H, int W,
                                          int cin, const float *wt, const float *bias) {
    if (!ab || !conv_out_ok(rgb, x, H, W, cin, wt, bias)) return iris_set_error("vae_conv_out_norm: bad arguments");
    return launch_conv_out<float, true>(x, ab, H, W, cin, wt, bias, rgb, f32);
}

extern "C" int iris_hip_vae_img_in(uint16_t *out, const float *img, int H, int W) {
    if (!out || !img || H <= 0 || W <= 0 || ((uintptr_t)out & 15)) return iris_set_error("vae_img_in: bad arguments");
    const int npix = H * W;
    IRIS_LAUNCH(vae_img_in_kernel, dim3((npix + NT / 8 - 1) / (NT / 8)), dim3(NT), 0, iris_stream(), img, npix, out);
    return iris_launch_check("vae_img_in_kernel");
}

extern "C" int iris_hip_vae_enc_out(float *lat, const float *mom, int z, int h, int w, const float *qw,
                                    const float *qb, const float *sc, const float *sh) {
    if (!lat || !mom || !sc || !sh || z <= 0 || h < 2 || w < 2) return iris_set_error("vae_enc_out: bad arguments");
    const size_t smem = ((size_t)EO_PIX * (2 * z + 1) + (qw ? (size_t)2 * z * z : 0)) * sizeof(float);
    const dim3 grid((h * w + EO_PIX - 1) / EO_PIX);
    if (smem <= 64 * 1024)
        IRIS_LAUNCH(vae_enc_out_kernel<true>, grid, dim3(NT), smem, iris_stream(), mom, z, h, w, qw, qb, sc, sh, lat);
    else
        IRIS_LAUNCH(vae_enc_out_kernel<false>, grid, dim3(NT), 0, iris_stream(), mom, z, h, w, qw, qb, sc, sh, lat);
    return iris_launch_check("vae_enc_out_kernel");
}
