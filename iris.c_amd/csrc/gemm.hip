/*
 * gemm.hip - bf16 x bf16 -> f32 MFMA GEMM for gfx950 with fused epilogues.
 *
 * Replaces the reference's linears (LINEAR_BF16_OR_F32 -> iris_linear ->
 * cblas_sgemm, iris_transformer_flux.c:121-131, iris_kernels.c:220-290) and the
 * elementwise passes that follow them (gated_add :136-143, iris_silu_mul
 * iris_kernels.c:626-638, the split/concat copies :3833-3840, :3897-3902).
 * The same kernel body also runs the VAE's implicit-GEMM 3x3 convolutions
 * (iris_vae.c:203-251) and the row softmax of its bottleneck attention in the
 * epilogues of two passes over the score product (iris_vae.c:320-335).
 *
 * out = A[M,K] . W[N,K]^T. Block tile 256x256x64 with 512 threads = 8 waves in
 * a 4x2 arrangement; each wave owns 64x128 as 4x8 v_mfma_f32_16x16x32_bf16
 * tiles (narrower block tiles: 256x224 for plain GEMMs whose last round of
 * 256-wide tiles would be part-empty, 256x128 for convolutions of at most
 * 128 output channels or few tiles). The 16x16x32 form does the same work per
 * LDS byte as 32x32x16 and, with the chip at its power limit on random data,
 * sustains about 10 % more MFMA throughput. Products of few rows run on
 * gemm_ring_kernel and most stride-1 convolutions on conv3x3_patch_kernel,
 * both below.
 *
 * Waves w and w+4 share a SIMD. The two groups (waves 0..3, waves 4..7) run
 * ping-pong: separated by block barriers, one group reads a whole 64-wide K
 * step of operand fragments from LDS and issues loads while the other runs
 * that step's 64 MFMAs, so every SIMD always has a wave issuing MFMAs and no
 * MFMA waits behind a load that is waiting for the address unit.
 *
 * A and W stream through two 64 KiB LDS stages filled by LDS-DMA
 * (buffer_load ... lds): global data goes straight into LDS, with no staging
 * registers and no ds_write. Each row of a stage is a full 128-byte line of
 * the operand, so every request to HBM fetches whole lines. The stages are
 * separate __shared__ objects, which lets the compiler wait only for the DMA
 * of the stage it reads. LDS serves a 16-byte-per-lane read 16 lanes at a
 * time over 64 banks: a group reads rows r..r+15 at one logical 16-byte chunk,
 * and XOR with (row / 2) mod 8 puts those rows on 16 distinct (row parity,
 * chunk) bank groups.
 *
 * Loads use buffer resources whose range ends at the operand's last valid row,
 * so rows past M (or N) read as zero without predicates. Blocks are mapped
 * XCD-major: block b runs on XCD b % 8 and takes a contiguous range of tiles,
 * ordered in groups of 8 M-tiles, so concurrently running blocks of one XCD
 * share A and W panels in that XCD's L2.
 */
#include "iris_internal.h"

#include <algorithm>
#include <mutex>
#include <string.h>

namespace {

constexpr int BM = 256, BN = 256, BK = 64, NT = 512;
constexpr int WAVES_M = 4, WAVES_N = 2, TW_M = BM / WAVES_M;
constexpr int FM = TW_M / 16;
constexpr int TILE_ELEMS = BM * BK;                 /* A tile = W tile = 16384 bf16 */
constexpr int DMA_ROWS = 8;                         /* rows of one 64-lane x 16-byte LDS-DMA load */
constexpr int GROUP_M = 8;
constexpr int MAXP = 4;

struct GemmParams {
    iris_gemm_problem_t p[MAXP];
    int tiles_m[MAXP], tiles_n[MAXP], tile_start[MAXP + 1];
    int nprob, total, per_xcd;
    /* split-K: problem i with chunks[i] > 1 has tiles_m[i] * tiles_n[i] *
     * chunks[i] blocks; block t of it works on K chunk t / (tiles_m * tiles_n)
     * (kchunk[i] elements) and writes its f32 partial product to
     * ws[i] + chunk * ws_stride[i] (M x N, row stride N) */
    int chunks[MAXP], kchunk[MAXP];
    float *ws[MAXP];
    long long ws_stride[MAXP];
    /* two-phase launch: blocks [0, phase_blocks) take tiles [0, phase_tiles)
     * (phase_blocks = 8 ceil(phase_tiles / 8), XCD-major over that range),
     * the blocks after them tiles [phase_tiles, total) (XCD-major, per_xcd
     * each), so the tiles of the first phase are dispatched before any of the
     * second's. 0: one phase. */
    int phase_tiles, phase_blocks;
    /* implicit 3x3 convolution (one problem, CONV kernels only): A is the bf16
     * NHWC input of (conv_h >> up) x (conv_w >> up) pixels, 2^cin_bshift bytes
     * per pixel; output row m is pixel (m / conv_w, m % conv_w) and K index
     * tap * cin + c reads channel c of the pixel at offset
     * (tap / 3 - 1, tap % 3 - 1) */
    int conv_h, conv_w, conv_up, conv_cpt_shift, conv_cin_bshift;
    unsigned conv_in_bytes;
    /* GroupNorm statistics of a convolution's output (CONV kernels, no
     * split-K): per row tile and group, sum and sum of squares in f64 */
    double *gn_part;
    int gn_groups;
    /* row softmax of scaled products (MODES 4, 5; one problem): s = sm_scale
     * * acc in log2 units, columns past N excluded. MODE 4: per row and tile,
     * (max s, sum 2^(s - max)) into sm_stat[row * tiles_n + tile column];
     * MODE 5: bf16 2^(s - sm_row[row].x) * sm_row[row].y into out, and zeros
     * in columns N .. sm_pad - 1 */
    float sm_scale;
    float2 *sm_stat;
    const float2 *sm_row;
    int sm_pad;
};

__device__ __forceinline__ int swz(int row, int chunk) {   /* element offset in a tile */
    return row * BK + ((chunk ^ ((row >> 1) & 7)) << 3);
}

/* s_waitcnt immediate: vmcnt in bits 3:0 and 15:14, expcnt 6:4 (no wait),
 * lgkmcnt 11:8 */
constexpr int waitcnt_imm(int vm, int lgkm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | (lgkm << 8); }

typedef __attribute__((address_space(3))) void lds_void;

/* element offset of (row, col) in a staged output half of OC columns: rows
 * padded by 16 bytes, or for 256 columns (a full 64 KiB stage) with the
 * 16-byte chunk index XORed with row % 16 */
template <int OC> __device__ __forceinline__ int opos(int row, int col) {
    if constexpr (OC == 256) return row * 256 + ((((col >> 3) ^ (row & 15)) << 3) | (col & 7));
    else return row * (OC + 8) + col;
}

/* bf16 epilogue of a whole tile through LDS (the caller has checked that the
 * tile is in range and the output rows 16-byte aligned). Group g (rows
 * GR g .. GR g + GR - 1, GR = 128 for 256-row tiles) stages its rows in
 * stage g. SWIGLU: accumulator
 * columns are 32-row gate / up groups, OC = half the tile width. */
template <int OC, bool SWIGLU, int FM_, int FNT_>
__device__ __forceinline__ void stage_out(const f32x4 (&acc)[FM_][FNT_], uint16_t *lds0, uint16_t *lds1,
                                          const iris_gemm_problem_t &pr, const float *vec, int m0, int oc0, int wm,
                                          int wn, int twn) {
    static_assert(128 * (OC == 256 ? 256 : OC + 8) * 2 <= 2 * TILE_ELEMS * 2, "a staged half fits one stage");
    constexpr int CPR = OC / 8; /* 16-byte chunks per row */
    constexpr int GR = 32 * FM_; /* rows of a wave group: 2 waves of 16 FM_ rows */
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const int grp = (tid >> 6) >> 2;
    uint16_t *const st = grp ? lds1 : lds0;
    const int hrow = (wm & 1) * (16 * FM_) + lr;
    __syncthreads(); /* every wave is done with the K loop's stages */
    if constexpr (SWIGLU) {
#pragma unroll
        for (int g = 0; g < FNT_ / 4; g++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int col = ((wn * twn + g * 64) >> 1) + h * 16 + lg * 4;
#pragma unroll
                for (int mi = 0; mi < FM_; mi++) {
                    const f32x4 gt = acc[mi][4 * g + h], up = acc[mi][4 * g + 2 + h];
                    uint16_t y[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) y[r] = f2bf_hw(silu_fast(gt[r]) * up[r]);
                    *(uint2 *)(st + opos<OC>(hrow + mi * 16, col)) =
                        make_uint2((uint32_t)y[0] | ((uint32_t)y[1] << 16), (uint32_t)y[2] | ((uint32_t)y[3] << 16));
                }
            }
    } else {
#pragma unroll
        for (int ni = 0; ni < FNT_; ni++) {
            const int col = wn * twn + ni * 16 + lg * 4;
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (vec) {
                const float4 t = *(const float4 *)(vec + oc0 + col);
                v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
            }
#pragma unroll
            for (int mi = 0; mi < FM_; mi++) {
                const f32x4 x = acc[mi][ni];
                *(uint2 *)(st + opos<OC>(hrow + mi * 16, col)) =
                    make_uint2((uint32_t)f2bf_hw(x[0] + v[0]) | ((uint32_t)f2bf_hw(x[1] + v[1]) << 16),
                               (uint32_t)f2bf_hw(x[2] + v[2]) | ((uint32_t)f2bf_hw(x[3] + v[3]) << 16));
            }
        }
    }
    __syncthreads();
    uint16_t *const out = (uint16_t *)pr.out + (size_t)(m0 + GR * grp) * pr.ldo + oc0;
    const int gt = tid & 255;
#pragma unroll
    for (int i = 0; i < GR * CPR / 256; i++) {
        const int c = gt + 256 * i, row = c / CPR, ch = c - row * CPR;
        *(uint4 *)(out + (size_t)row * pr.ldo + ch * 8) = *(const uint4 *)(st + opos<OC>(row, ch * 8));
    }
}

/* The epilogues of MODES 4 and 5 (the products of one query block against
 * the keys of one 256-wide tile): per-row statistics of the tile (STATS), or
 * the probabilities. Lane l holds row lr of each 16x16 tile at columns
 * lg*4 .. lg*4+3; a row's 256 columns are spread over the 4 lanes lr + 16j of
 * a wave and the 2 waves across N. */
template <bool STATS, int FNT_>
__device__ __forceinline__ void softmax_epilogue(f32x4 (&acc)[FM][FNT_], const GemmParams &P,
                                                 const iris_gemm_problem_t &pr, int m0, int n0, int tn, int wm, int wn,
                                                 uint16_t *lds0, uint16_t *lds1) {
    constexpr int TWN_ = FNT_ * 16, BNT_ = TWN_ * WAVES_N;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const int M = pr.M, N = pr.N;
    const int rowb = m0 + wm * TW_M + lr, colb = n0 + wn * TWN_ + lg * 4;
    /* scaled scores in place; columns past N hold -inf (2^-inf = 0) */
#pragma unroll
    for (int mi = 0; mi < FM; mi++)
#pragma unroll
        for (int ni = 0; ni < FNT_; ni++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                acc[mi][ni][r] = colb + ni * 16 + r < N ? acc[mi][ni][r] * P.sm_scale : -INFINITY;
    if constexpr (STATS) {
        /* the tile's row max, then its row sum of 2^(s - max): lane, the
         * row's 4 lanes (xor 16, 32), the 2 waves across N (in LDS) */
        __shared__ float red[2][WAVES_N][BM];
#pragma unroll
        for (int mi = 0; mi < FM; mi++) {
            float m = -INFINITY;
#pragma unroll
            for (int ni = 0; ni < FNT_; ni++)
                m = fmaxf(m, fmaxf(fmaxf(acc[mi][ni][0], acc[mi][ni][1]), fmaxf(acc[mi][ni][2], acc[mi][ni][3])));
            m = fmaxf(m, __shfl_xor(m, 16, 64));
            m = fmaxf(m, __shfl_xor(m, 32, 64));
            if (lg == 0) red[0][wn][wm * TW_M + mi * 16 + lr] = m;
        }
        __syncthreads();
#pragma unroll
        for (int mi = 0; mi < FM; mi++) {
            const int rr = wm * TW_M + mi * 16 + lr;
            const float mt = fmaxf(red[0][0][rr], red[0][1][rr]);
            float l = 0.0f;
#pragma unroll
            for (int ni = 0; ni < FNT_; ni++)
#pragma unroll
                for (int r = 0; r < 4; r++) l += __builtin_amdgcn_exp2f(acc[mi][ni][r] - mt);
            l += __shfl_xor(l, 16, 64);
            l += __shfl_xor(l, 32, 64);
            if (lg == 0) red[1][wn][rr] = l;
        }
        __syncthreads();
        if (tid < BM && m0 + tid < M)
            P.sm_stat[(size_t)(m0 + tid) * P.tiles_n[0] + tn] =
                make_float2(fmaxf(red[0][0][tid], red[0][1][tid]), red[1][0][tid] + red[1][1][tid]);
        return;
    } else {
#pragma unroll
        for (int mi = 0; mi < FM; mi++) {
            const int row = rowb + mi * 16;
            const float2 rs = row < M ? P.sm_row[row] : make_float2(0.0f, 0.0f);
#pragma unroll
            for (int ni = 0; ni < FNT_; ni++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[mi][ni][r] = __builtin_amdgcn_exp2f(acc[mi][ni][r] - rs.x) * rs.y;
        }
        const int ldo = pr.ldo;
        if (m0 + BM <= M && n0 + BNT_ <= N && (ldo & 7) == 0 && ((uintptr_t)pr.out & 15) == 0) {
            stage_out<BNT_, false, FM, FNT_>(acc, lds0, lds1, pr, nullptr, m0, n0, wm, wn, TWN_);
            return;
        }
        /* edge tiles element by element, zeros in the padding columns */
#pragma unroll
        for (int mi = 0; mi < FM; mi++) {
            const int row = rowb + mi * 16;
            if (row >= M) continue;
#pragma unroll
            for (int ni = 0; ni < FNT_; ni++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int col = colb + ni * 16 + r;
                    if (col < P.sm_pad)
                        ((uint16_t *)pr.out)[(size_t)row * ldo + col] = col < N ? f2bf_hw(acc[mi][ni][r]) : (uint16_t)0;
                }
        }
    }
}

/* MODE 0: GEMM; 1: 3x3 convolution, stride 1, input optionally read through
 * a nearest 2x upsample; 2: 3x3 convolution, stride 2, right/bottom padding;
 * 3: GEMM with a second K segment (A2, W2) after the first; 4, 5: GEMMs
 * whose epilogue is a row softmax pass (softmax_epilogue: row statistics,
 * probabilities). The modes are
 * separate kernels: the load-issue phase has no cycles to spare for the
 * address arithmetic of the modes it does not run. */
template <int MODE, int BNT = BN, int BMT = BM>
__global__ __launch_bounds__(NT) void gemm_bf16_kernel(const GemmParams P) {
    constexpr bool CONV = MODE == 1 || MODE == 2, SEG2 = MODE == 3, SMX = MODE == 4 || MODE == 5;
    /* BNT: block tile width, 256, or (MODE 0, no SwiGLU) 224 = 2 waves x 7
     * MFMA tiles, for launches whose 256-wide tiles leave the last wave of
     * blocks part-empty, or (convolutions) 128 = 2 waves x 4 MFMA tiles for
     * outputs of at most 128 channels, which a 256-wide tile would compute
     * half empty */
    static_assert(BNT == BN || (BNT == 224 && MODE == 0) || (BNT == 128 && (MODE == 1 || MODE == 2)),
                  "narrow tiles are for plain GEMMs and convolutions");
    /* BMT: block tile height, 256, or 128 (plain GEMMs on few rows: twice
     * the tiles of a 256-row tile; wave tile 32 x 128) */
    static_assert(BMT == BM || (BMT == 128 && MODE == 0 && BNT == BN), "128-row tiles are for plain GEMMs");
    constexpr int TWN = BNT / WAVES_N, FNT = TWN / 16, W_DMA = BNT / DMA_ROWS / 4;
    constexpr int TWM = BMT / WAVES_M, FMT = TWM / 16, A_DMA = BMT / DMA_ROWS / 4;
    /* two stages, each an A tile then a W tile; separate objects so the
     * compiler tracks the LDS-DMA writes of one stage apart from reads of
     * the other */
    __shared__ __attribute__((aligned(16))) uint16_t lds0[2 * TILE_ELEMS];
    __shared__ __attribute__((aligned(16))) uint16_t lds1[2 * TILE_ELEMS];
    const int b = blockIdx.x;
    int L;
    if (b < P.phase_blocks) {
        L = (b & 7) * (P.phase_blocks >> 3) + (b >> 3);
        if (L >= P.phase_tiles) return;
    } else {
        const int b2 = b - P.phase_blocks;
        L = P.phase_tiles + (b2 & 7) * P.per_xcd + (b2 >> 3);
        if (L >= P.total) return;
    }
    int pi = 0;
#pragma unroll
    for (int i = 1; i < MAXP; i++)
        if (i < P.nprob && L >= P.tile_start[i]) pi = i;
    iris_gemm_problem_t pr = P.p[pi];
    int t = L - P.tile_start[pi];
    int kt0 = 0;   /* first K step of this block's chunk (split-K convolution) */
    if (P.chunks[pi] > 1) {
        const int per = P.tiles_m[pi] * P.tiles_n[pi];
        const int chunk = t / per;
        const int k0 = chunk * P.kchunk[pi];
        t -= chunk * per;
        if (CONV) kt0 = k0 / BK;
        else pr.A += k0;
        pr.W += k0;
        pr.K = min(P.kchunk[pi], pr.K - k0);
        pr.out = P.ws[pi] + chunk * P.ws_stride[pi];
        pr.ldo = pr.N;
        pr.vec = nullptr;
        pr.epi = IRIS_EPI_F32;
    }
    const int tmc = P.tiles_m[pi], tnc = P.tiles_n[pi];
    const int group = t / (GROUP_M * tnc);
    const int first_m = group * GROUP_M;
    const int gsz = min(tmc - first_m, GROUP_M);
    const int tm = first_m + (t % (GROUP_M * tnc)) % gsz;
    const int tn = (t % (GROUP_M * tnc)) / gsz;
    const int m0 = tm * BMT, n0 = tn * BNT;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    /* waves w and w + 4 share SIMD w: group 0 (waves 0..3) and group 1
     * (waves 4..7) alternate between an LDS phase and an MFMA phase */
    const int grp = wave >> 2, gw = wave & 3;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int lr = lane & 15, lg = lane >> 4;

    /* LDS-DMA: load j of an operand covers tile rows 8j..8j+7 and writes
     * 1 KiB at byte j*1024 of the operand's tile, lane l at + 16l, i.e. row
     * 8j + l/8, stored chunk l%8; the lane fetches global chunk
     * (l%8) ^ ((row >> 1) & 7), which depends on j only through its parity.
     * Group 0 loads the A tiles and group 1 the W tiles; wave gw of a group
     * issues A loads j = 8gw..8gw+7 and W loads j = W_DMA gw .. + W_DMA-1
     * (W_DMA = 7 for 224-wide tiles, where the parity of j is that of
     * gw + i). */
    const uint16_t *a_base = pr.A + (size_t)m0 * pr.lda;
    const uint16_t *w_base = pr.W + (size_t)n0 * pr.ldw;
    const int a_rows = min(BMT, pr.M - m0), w_rows = min(BNT, pr.N - n0);
    const __amdgpu_buffer_rsrc_t a_rsrc =
        CONV ? __builtin_amdgcn_make_buffer_rsrc((void *)pr.A, (short)0, (int)P.conv_in_bytes, 0x00020000)
             : __builtin_amdgcn_make_buffer_rsrc((void *)a_base, (short)0, a_rows * pr.lda * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)w_base, (short)0, w_rows * pr.ldw * 2, 0x00020000);
    const int drow = lane >> 3, dch = lane & 7;
    int a_voff[2], w_voff[2], a_chunk[2];
#pragma unroll
    for (int par = 0; par < 2; par++) {
        const int c = dch ^ ((4 * par + (drow >> 1)) & 7);
        const int row = gw * A_DMA * DMA_ROWS + drow;
        a_voff[par] = (row * pr.lda + c * 8) * 2;
        /* W: load i of wave gw is tile load j = W_DMA gw + i */
        const int cw = dch ^ ((4 * ((par + (W_DMA & 1) * gw) & 1) + (drow >> 1)) & 7);
        w_voff[par] = ((gw * W_DMA * DMA_ROWS + drow) * pr.ldw + cw * 8) * 2;
        a_chunk[par] = c * 16;
    }
    const int a_step = DMA_ROWS * pr.lda * 2, w_step = DMA_ROWS * pr.ldw * 2;
    /* second segment (MODE 3): the same lane layout over A2 / W2; a lane's
     * offset there is its first-segment offset + row * (ld2 - ld) * 2, formed
     * at each load from scalars chosen by the K step, so the two segments
     * share one load sequence and no registers are held for the second */
    const int nk1 = pr.K / BK;
    const int dma_row = gw * A_DMA * DMA_ROWS + drow;
    __amdgpu_buffer_rsrc_t a2_rsrc = a_rsrc, w2_rsrc = w_rsrc;
    if (SEG2) {
        a2_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(pr.A2 + (size_t)m0 * pr.lda2), (short)0,
                                                    a_rows * pr.lda2 * 2, 0x00020000);
        w2_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(pr.W2 + (size_t)n0 * pr.ldw2), (short)0,
                                                    w_rows * pr.ldw2 * 2, 0x00020000);
    }
    /* convolution: the output pixel of each row this lane loads, y << 16 | x;
     * rows past M get y = 0x4000, outside every image */
    uint32_t pix[A_DMA];
    if (CONV) {
#pragma unroll
        for (int i = 0; i < A_DMA; i++) {
            const int m = m0 + gw * A_DMA * DMA_ROWS + i * DMA_ROWS + drow;
            pix[i] = m < pr.M ? ((uint32_t)(m / P.conv_w) << 16) | (uint32_t)(m % P.conv_w) : 0x40000000u;
        }
    }
    auto dma_a = [&](uint16_t *stage, int kt) {
        if (CONV) {
            /* K step kt covers channels 64 * (kt mod cin/64) .. +63 of tap kt / (cin/64);
             * taps outside the image (zero padding) get an offset past the end of the
             * buffer, which reads as zero */
            const int kg = kt + kt0;
            const int tap = kg >> P.conv_cpt_shift;
            const int soff = (kg & ((1 << P.conv_cpt_shift) - 1)) * (BK * 2);
            const int ty = tap / 3;
            const int dy = ty - 1, dx = tap - 3 * ty - 1;
            /* MODE 1: input pixel ((y + dy) >> up, (x + dx) >> up); MODE 2 (stride 2,
             * zero padding on the right and bottom only): input pixel
             * (2y + dy + 1, 2x + dx + 1) of a (2 conv_h) x (2 conv_w) image */
            const int up = MODE == 1 ? P.conv_up : 0;
            const int hin = MODE == 2 ? 2 * P.conv_h : P.conv_h, win = MODE == 2 ? 2 * P.conv_w : P.conv_w;
            constexpr int mul = MODE == 2 ? 2 : 1, off = MODE == 2 ? 1 : 0;
#pragma unroll
            for (int i = 0; i < A_DMA; i++) {
                const int yy = (int)(pix[i] >> 16) * mul + dy + off, xx = (int)(pix[i] & 0xffffu) * mul + dx + off;
                const bool ok = (unsigned)yy < (unsigned)hin && (unsigned)xx < (unsigned)win;
                const int src = ((((yy >> up) * (win >> up)) + (xx >> up)) << P.conv_cin_bshift) + a_chunk[i & 1];
                __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_void *)(stage + (gw * A_DMA + i) * 512), 16,
                                                         ok ? src : (int)0x80000000u, soff, 0, 0);
            }
        } else if (SEG2) {
            const bool s2 = kt >= nk1;
            const __amdgpu_buffer_rsrc_t r = s2 ? a2_rsrc : a_rsrc;
            const int extra = s2 ? dma_row * ((pr.lda2 - pr.lda) * 2) : 0;
            const int step = s2 ? DMA_ROWS * pr.lda2 * 2 : a_step, ks = (s2 ? kt - nk1 : kt) * BK * 2;
#pragma unroll
            for (int i = 0; i < A_DMA; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)(stage + (gw * A_DMA + i) * 512), 16,
                                                         a_voff[i & 1] + extra + i * step, ks, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < A_DMA; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_void *)(stage + (gw * A_DMA + i) * 512),
                                                         16, a_voff[i & 1] + i * a_step, kt * BK * 2, 0, 0);
        }
    };
    auto dma_w = [&](uint16_t *stage, int kt) {
        if (SEG2) {
            const bool s2 = kt >= nk1;
            const __amdgpu_buffer_rsrc_t r = s2 ? w2_rsrc : w_rsrc;
            const int extra = s2 ? dma_row * ((pr.ldw2 - pr.ldw) * 2) : 0;
            const int step = s2 ? DMA_ROWS * pr.ldw2 * 2 : w_step, ks = (s2 ? kt - nk1 : kt) * BK * 2;
#pragma unroll
            for (int i = 0; i < W_DMA; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r,
                                                         (lds_void *)(stage + TILE_ELEMS + (gw * W_DMA + i) * 512),
                                                         16, w_voff[i & 1] + extra + i * step, ks, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < W_DMA; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc,
                                                         (lds_void *)(stage + TILE_ELEMS + (gw * W_DMA + i) * 512),
                                                         16, w_voff[i & 1] + i * w_step, kt * BK * 2, 0, 0);
        }
    };

    f32x4 acc[FMT][FNT];
#pragma unroll
    for (int i = 0; i < FMT; i++)
#pragma unroll
        for (int j = 0; j < FNT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0.0f;

    const int nk = (pr.K + (SEG2 ? pr.K2 : 0)) / BK;
    /* fragments of one K-step: two 32-wide slices */
    bf16x8 a[2][FMT], w[2][FNT];
    auto frags = [&](const uint16_t *stage) {
        const uint16_t *As = stage;
        const uint16_t *Ws = stage + TILE_ELEMS;
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            const int ch = kk * 4 + lg;
#pragma unroll
            for (int mi = 0; mi < FMT; mi++) a[kk][mi] = *(const bf16x8 *)(As + swz(wm * TWM + mi * 16 + lr, ch));
#pragma unroll
            for (int ni = 0; ni < FNT; ni++) w[kk][ni] = *(const bf16x8 *)(Ws + swz(wn * TWN + ni * 16 + lr, ch));
        }
    };
    auto mfmas = [&](int kk) {
#pragma unroll
            for (int mi = 0; mi < FMT; mi++)
#pragma unroll
                for (int ni = 0; ni < FNT; ni++)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[kk][ni], a[kk][mi], acc[mi][ni], 0, 0, 0);
    };
/* explicit waits and barriers stay where they are written */
#define WAIT(vm, lgkm)                                              \
    do {                                                            \
        __builtin_amdgcn_sched_barrier(0);                          \
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(vm, lgkm));          \
        __builtin_amdgcn_sched_barrier(0);                          \
    } while (0)
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    /* Barrier-separated phases; group 0 runs L(t), C(t) in phases 2t, 2t+1,
     * group 1 runs L(t), C(t) in phases 2t+1, 2t+2. L(t) reads tile t (stage
     * t&1) into registers, C(t) runs its MFMAs, so on every SIMD one wave
     * issues MFMAs while the other reads LDS. Loads are issued only in L
     * phases (a load waiting for the address unit holds up the instructions
     * behind it) and each group issues half of every tile:
     *  - group 0 issues A of tile t+1 in L(t): stage (t+1)&1 last held tile
     *    t-1, read by both groups before phase 2t; it waits for the loads at
     *    the end of C(t), before phase 2t+2 where tile t+1 is first read;
     *  - group 1 issues W of tile t+2 in L(t), into the stage it has just
     *    read. Two waves of the group read each W row, so the loads wait for
     *    a barrier in the middle of phase 2t+1 that every wave of the group
     *    reaches only after its reads of tile t have returned (group 0 read
     *    tile t in phase 2t and meets this barrier between the two halves of
     *    C(t)). Group 1 waits for the loads in L(t+1), before phase 2t+4.
     * Every wait is for all of a wave's loads: completions of LDS-DMA loads
     * are not ordered, so a partial count does not mean the oldest loads are
     * done. Past the last tile the loads repeat tile nk-1 into a stage
     * nothing reads again. */
    auto step0 = [&](uint16_t *cur, uint16_t *nxt, int kt) {
        frags(cur);
        dma_a(nxt, min(kt + 1, nk - 1));
        /* spread the loads over the fragment reads */
#pragma unroll
        for (int i = 0; i < A_DMA; i++) {
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        WAIT(63, 0);
        barrier();
        mfmas(0);
        barrier();   /* group 1's reads of tile kt are done */
        mfmas(1);
        WAIT(0, 0);
        barrier();
    };
    auto step1 = [&](uint16_t *cur, int kt) {
        frags(cur);
        WAIT(0, 0);
        barrier();   /* every wave of the group has read tile kt */
        dma_w(cur, min(kt + 2, nk - 1));
        barrier();
        mfmas(0);
        mfmas(1);
        if (kt + 1 < nk) barrier();
    };

    if (grp) {
        dma_w(lds0, 0);
        WAIT(0, 0);
        barrier();
        dma_w(lds1, min(1, nk - 1));
        barrier();
        int kt = 0;
        for (; kt + 1 < nk; kt += 2) {
            step1(lds0, kt);
            step1(lds1, kt + 1);
        }
        if (kt < nk) step1(lds0, kt);
    } else {
        dma_a(lds0, 0);
        WAIT(0, 0);
        barrier();
        int kt = 0;
        for (; kt + 1 < nk; kt += 2) {
            step0(lds0, lds1, kt);
            step0(lds1, lds0, kt + 1);
        }
        if (kt < nk) step0(lds0, lds1, kt);
    }
    WAIT(0, 0);   /* no DMA outstanding at exit */
#undef WAIT
    if constexpr (SMX) {
        softmax_epilogue<MODE == 4, FNT>(acc, P, pr, m0, n0, tn, wm, wn, lds0, lds1);
        return;
    }

    /* ---- epilogue: W is the MFMAs' first operand, so lane l holds row lr of
     *      each 16x16 tile at the 4 consecutive columns lg*4 .. lg*4+3 ---- */
    const int M = pr.M, N = pr.N, ldo = pr.ldo;
    const float *vec = pr.vec;
    const int rowb = m0 + wm * TWM + lr;
    const int colb = n0 + wn * TWN + lg * 4;
    /* whole tile in range and 4-wide accesses aligned: one 8- or 16-byte
     * access per lane and 16x16 tile */
    const bool aligned = (ldo & 3) == 0 && ((uintptr_t)pr.out & 15) == 0 && ((uintptr_t)vec & 15) == 0;
    const bool full = m0 + BMT <= M && n0 + BNT <= N && aligned;
    /* GroupNorm statistics of a convolution's output: each lane sums the
     * values it writes per 4-channel chunk (one group: groups are multiples
     * of 4 channels), then the tile's sums per group are formed in a fixed
     * order below (the direct stores: the tile's values stay in registers) */
    const bool gn = CONV && P.gn_part != nullptr;
    float gs1[FNT], gs2[FNT];
#pragma unroll
    for (int ni = 0; ni < FNT; ni++) gs1[ni] = gs2[ni] = 0.0f;
    auto gn_add = [&](int ni, float y) {
        gs1[ni] += y;
        gs2[ni] += y * y;
    };
    /* Whole tiles of bf16 output (plain or SwiGLU) go out through LDS: each
     * group writes its 128 rows into one of the stages, now free, and then
     * stores them as 16-byte chunks of whole rows, so one store instruction
     * covers full 128-byte lines instead of 32-byte pieces of 16 rows (the
     * direct stores left the waves stalled on issue). */
    bool staged = false;
    if (full && (ldo & 7) == 0 && (pr.epi == IRIS_EPI_BF16 || (BNT == BN && pr.epi == IRIS_EPI_SWIGLU))) {
        if (gn) {   /* a convolution's bf16 tile: the sums of the values before rounding */
#pragma unroll
            for (int ni = 0; ni < FNT; ni++) {
                const float4 t = vec ? *(const float4 *)(vec + colb + ni * 16) : make_float4(0, 0, 0, 0);
#pragma unroll
                for (int mi = 0; mi < FMT; mi++) {
                    gn_add(ni, acc[mi][ni][0] + t.x);
                    gn_add(ni, acc[mi][ni][1] + t.y);
                    gn_add(ni, acc[mi][ni][2] + t.z);
                    gn_add(ni, acc[mi][ni][3] + t.w);
                }
            }
        }
        if (pr.epi == IRIS_EPI_SWIGLU) stage_out<BNT / 2, true, FMT, FNT>(acc, lds0, lds1, pr, vec, m0, n0 >> 1, wm, wn, TWN);
        else stage_out<BNT, false, FMT, FNT>(acc, lds0, lds1, pr, vec, m0, n0, wm, wn, TWN);
        if (!gn) return;
        staged = true;
    }
    if (!staged) switch (pr.epi) {
    case IRIS_EPI_F32:
    case IRIS_EPI_BF16:
    case IRIS_EPI_GATED_ADD:
    case IRIS_EPI_ADD: {
        const float vdef = pr.epi == IRIS_EPI_GATED_ADD ? 1.0f : 0.0f;
#pragma unroll
        for (int ni = 0; ni < FNT; ni++) {
            const int col = colb + ni * 16;
            /* a lane's 4 columns are all in range or (N % 4 == 0 aside) all out */
            const bool cols4 = full || (aligned && col + 3 < N);
            float v[4];
            if (cols4 && vec) {
                const float4 t = *(const float4 *)(vec + col);
                v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] = vec && col + r < N ? vec[col + r] : vdef;
            }
#pragma unroll
            for (int mi = 0; mi < FMT; mi++) {
                const int row = rowb + mi * 16;
                const f32x4 x = acc[mi][ni];
                const size_t o = (size_t)row * ldo + col;
                if (full || (cols4 && row < M)) {
                    float4 y;
                    if (pr.epi == IRIS_EPI_F32) {
                        y = make_float4(x[0] + v[0], x[1] + v[1], x[2] + v[2], x[3] + v[3]);
                        *(float4 *)((float *)pr.out + o) = y;
                    } else if (pr.epi == IRIS_EPI_BF16) {
                        y = make_float4(x[0] + v[0], x[1] + v[1], x[2] + v[2], x[3] + v[3]);
                        uint2 p;
                        p.x = (uint32_t)f2bf_hw(y.x) | ((uint32_t)f2bf_hw(y.y) << 16);
                        p.y = (uint32_t)f2bf_hw(y.z) | ((uint32_t)f2bf_hw(y.w) << 16);
                        *(uint2 *)((uint16_t *)pr.out + o) = p;
                    } else if (pr.epi == IRIS_EPI_GATED_ADD) {
                        float4 *dst = (float4 *)((float *)pr.out + o);
                        y = *dst;
                        y.x += v[0] * x[0]; y.y += v[1] * x[1]; y.z += v[2] * x[2]; y.w += v[3] * x[3];
                        *dst = y;
                    } else {
                        float4 *dst = (float4 *)((float *)pr.out + o);
                        y = *dst;
                        y.x += x[0] + v[0]; y.y += x[1] + v[1]; y.z += x[2] + v[2]; y.w += x[3] + v[3];
                        *dst = y;
                    }
                    if (gn) {
                        gn_add(ni, y.x);
                        gn_add(ni, y.y);
                        gn_add(ni, y.z);
                        gn_add(ni, y.w);
                    }
                } else if (row < M) {
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        if (col + r >= N) continue;
                        float *const f = (float *)pr.out + o + r;
                        float y = x[r] + v[r];
                        if (pr.epi == IRIS_EPI_F32) *f = y;
                        else if (pr.epi == IRIS_EPI_BF16) ((uint16_t *)pr.out)[o + r] = f2bf_hw(y);
                        else if (pr.epi == IRIS_EPI_GATED_ADD) *f = y = *f + v[r] * x[r];
                        else *f = y = *f + (x[r] + v[r]);
                        if (gn) gn_add(ni, y);
                    }
                }
            }
        }
        break;
    }
    case IRIS_EPI_SWIGLU:
        if constexpr (BNT == BN) {
            /* each 64 columns of the wave are one interleaved group: tiles 4g,
             * 4g+1 = 32 gate rows, tiles 4g+2, 4g+3 = the matching 32 up rows;
             * output columns = group * 32 + h * 16 + lg * 4 + (0..3) */
#pragma unroll
            for (int g = 0; g < FNT / 4; g++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int col = ((n0 + wn * TWN + g * 64) >> 1) + h * 16 + lg * 4;
#pragma unroll
                    for (int mi = 0; mi < FMT; mi++) {
                        const int row = rowb + mi * 16;
                        const f32x4 gt = acc[mi][4 * g + h], up = acc[mi][4 * g + 2 + h];
                        uint16_t y[4];
#pragma unroll
                        for (int r = 0; r < 4; r++) y[r] = f2bf_hw(silu_fast(gt[r]) * up[r]);
                        uint16_t *dst = (uint16_t *)pr.out + (size_t)row * ldo + col;
                        if (full) {
                            *(uint2 *)dst = make_uint2((uint32_t)y[0] | ((uint32_t)y[1] << 16),
                                                       (uint32_t)y[2] | ((uint32_t)y[3] << 16));
                        } else if (row < M) {
#pragma unroll
                            for (int r = 0; r < 4; r++)
                                if (col + r < (N >> 1)) dst[r] = y[r];
                        }
                    }
                }
        }
        break;
    case IRIS_EPI_F32_T: {
#pragma unroll
        for (int ni = 0; ni < FNT; ni++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int col = colb + ni * 16 + r;
                if (col >= N) continue;
                const float v = vec ? vec[col] : 0.0f;
#pragma unroll
                for (int mi = 0; mi < FMT; mi++) {
                    const int row = rowb + mi * 16;
                    if (row < M) ((float *)pr.out)[(size_t)col * ldo + row] = acc[mi][ni][r] + v;
                }
            }
        break;
    }
    default:
        break;
    }
    if constexpr (CONV) {
        if (gn) {
            /* per wave, the 16 lanes of a row hold one 4-channel chunk's 16
             * rows of each of the wave's 4 row blocks: the chunk's sums over
             * the wave's 64 rows, then over the tile's 4 waves in M and the
             * group's chunks in order, in f64 */
            __shared__ float gnl[WAVES_M * WAVES_N * FNT * 4 * 2];
#pragma unroll
            for (int ni = 0; ni < FNT; ni++) {
                const float s = row16_sum(gs1[ni]), q = row16_sum(gs2[ni]);
                if (lr == 0) {
                    float *d = gnl + (((wm * WAVES_N + wn) * FNT + ni) * 4 + lg) * 2;
                    d[0] = s;
                    d[1] = q;
                }
            }
            __syncthreads();
            const int G = P.gn_groups, cpg = N / G, t = threadIdx.x;
            if (t < BNT / cpg && n0 + t * cpg < N) {
                double s = 0.0, q = 0.0;
                for (int c = t * cpg; c < (t + 1) * cpg; c += 4) {
                    const int w = c % TWN;
                    for (int wm_ = 0; wm_ < WAVES_M; wm_++) {
                        const float *d = gnl + (((wm_ * WAVES_N + c / TWN) * FNT + w / 16) * 4 + (w % 16) / 4) * 2;
                        s += (double)d[0];
                        q += (double)d[1];
                    }
                }
                double *dst = P.gn_part + ((size_t)(m0 / BMT) * G + n0 / cpg + t) * 2;
                dst[0] = s;
                dst[1] = q;
            }
        }
    }
}

/* Products on few rows: block tiles of 32 FM x 32 FN over a ring of NS LDS
 * stages, 8 waves: waves 0..3 compute (2x2, wave tile 16 FM x 16 FN), waves
 * 4..7 only load, one of each on a SIMD. The K step of a small tile is bound
 * by issue, not by its products: a wave that issues an LDS-DMA load waits for
 * the address unit (16 clocks per 1 KiB load), so where the computing waves
 * also load, a step takes the sum of its load issue, products and fragment
 * reads; with waves of their own the loads cost the products nothing, and
 * NS - 1 steps are in flight (96 or 120 KiB per CU) against the latency of
 * weights that come from HBM.
 *
 * One barrier per K step. A computing wave runs step t's first 32-wide half
 * on fragments read during step t-1 while it reads the second half's, meets
 * the barrier when its reads of tile t are done, then reads tile t+1's first
 * half while the second half's products run. A loading wave meets step t's
 * barrier when its loads of tile t+1 are done (loads of a wave complete in
 * order: the count of the younger ones is enough), then issues tile t+NS into
 * the stage of tile t. Past the last tile it repeats tile nk-1 into stages
 * nothing reads again. Every output element gets the additions of the kernel
 * above in its order. */
template <int FM_, int FN_, int NS>
__global__ __launch_bounds__(512) void gemm_ring_kernel(const GemmParams P) {
    constexpr int BMR = 32 * FM_, BNR = 32 * FN_, TM = 16 * FM_, TN = 16 * FN_;
    constexpr int A_DMA = BMR / DMA_ROWS / 4, W_DMA = BNR / DMA_ROWS / 4, LD = A_DMA + W_DMA;
    constexpr int A_ELEMS = BMR * BK, ST_ELEMS = (BMR + BNR) * BK;
    static_assert(NS >= 3 && (NS - 1) * LD < 64, "ring depth");
    extern __shared__ __attribute__((aligned(16))) uint16_t ring[];
    const int L = (blockIdx.x & 7) * P.per_xcd + (blockIdx.x >> 3);
    if (L >= P.total) return;
    int pi = 0;
#pragma unroll
    for (int i = 1; i < MAXP; i++)
        if (i < P.nprob && L >= P.tile_start[i]) pi = i;
    iris_gemm_problem_t pr = P.p[pi];
    int t = L - P.tile_start[pi];
    if (P.chunks[pi] > 1) {
        const int per = P.tiles_m[pi] * P.tiles_n[pi];
        const int chunk = __builtin_amdgcn_readfirstlane(t / per), k0 = chunk * P.kchunk[pi];
        t -= chunk * per;
        pr.A += k0;
        pr.W += k0;
        pr.K = min(P.kchunk[pi], pr.K - k0);
        pr.out = P.ws[pi] + chunk * P.ws_stride[pi];
        pr.ldo = pr.N;
        pr.vec = nullptr;
        pr.epi = IRIS_EPI_F32;
    }
    const int tmc = P.tiles_m[pi], tnc = P.tiles_n[pi];
    /* scalar registers for what the buffer resources are made of */
    const int first_m = __builtin_amdgcn_readfirstlane(t / (GROUP_M * tnc)) * GROUP_M;
    const int gsz = min(tmc - first_m, GROUP_M), tg = t - first_m * tnc;
    const int tn = __builtin_amdgcn_readfirstlane(tg / gsz);
    const int m0 = (first_m + tg - tn * gsz) * BMR, n0 = tn * BNR;

    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = (wave >> 1) & 1, wn = wave & 1;
    const int nk = pr.K / BK;
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wave >= 4) {
        const int lw = wave & 3;
        const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(pr.A + (size_t)m0 * pr.lda), (short)0, min(BMR, pr.M - m0) * pr.lda * 2, 0x00020000);
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(pr.W + (size_t)n0 * pr.ldw), (short)0, min(BNR, pr.N - n0) * pr.ldw * 2, 0x00020000);
        /* load j of an operand covers tile rows 8j .. 8j+7; loading wave w
         * issues loads j = DMA w .. + DMA - 1; lane l fetches row 8j + l/8,
         * chunk (l%8) ^ ((row >> 1) & 7) */
        const int drow = lane >> 3, dch = lane & 7;
        int a_voff[2], w_voff[2];
#pragma unroll
        for (int par = 0; par < 2; par++) {
            const int ca = dch ^ ((4 * ((par + (A_DMA & 1) * lw) & 1) + (drow >> 1)) & 7);
            const int cw = dch ^ ((4 * ((par + (W_DMA & 1) * lw) & 1) + (drow >> 1)) & 7);
            a_voff[par] = ((lw * A_DMA * DMA_ROWS + drow) * pr.lda + ca * 8) * 2;
            w_voff[par] = ((lw * W_DMA * DMA_ROWS + drow) * pr.ldw + cw * 8) * 2;
        }
        const int a_step = DMA_ROWS * pr.lda * 2, w_step = DMA_ROWS * pr.ldw * 2;
        auto dma = [&](int stage, int kt) {
            const int soff = kt * BK * 2;
            uint16_t *const st = ring + stage * ST_ELEMS;
#pragma unroll
            for (int i = 0; i < W_DMA; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (lds_void *)(st + A_ELEMS + (lw * W_DMA + i) * 512),
                                                         16, w_voff[i & 1] + i * w_step, soff, 0, 0);
#pragma unroll
            for (int i = 0; i < A_DMA; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_void *)(st + (lw * A_DMA + i) * 512), 16,
                                                         a_voff[i & 1] + i * a_step, soff, 0, 0);
        };
        for (int i = 0; i < NS; i++) dma(i, min(i, nk - 1));
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(waitcnt_imm((NS - 1) * LD, 15));
        barrier();
        for (int kt = 0, st = 0; kt < nk; kt++) {
            __builtin_amdgcn_s_waitcnt(waitcnt_imm((NS - 2) * LD, 15));
            barrier();
            dma(st, min(kt + NS, nk - 1));
            st = st == NS - 1 ? 0 : st + 1;
        }
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));   /* no DMA outstanding at exit */
        return;
    }

    f32x4 acc[FM_][FN_];
#pragma unroll
    for (int i = 0; i < FM_; i++)
#pragma unroll
        for (int j = 0; j < FN_; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0.0f;
    bf16x8 a0[FM_], w0[FN_], a1[FM_], w1[FN_];
    /* rows 16 apart keep their swizzle: one base per half */
    const int ab0 = swz(wm * TM + lr, lg), wb0 = A_ELEMS + swz(wn * TN + lr, lg);
    const int ab1 = swz(wm * TM + lr, 4 + lg), wb1 = A_ELEMS + swz(wn * TN + lr, 4 + lg);
    auto frags = [&](int st, int ab, int wb, bf16x8 (&a)[FM_], bf16x8 (&w)[FN_]) {
#pragma unroll
        for (int mi = 0; mi < FM_; mi++) a[mi] = *(const bf16x8 *)(ring + st + ab + mi * 16 * BK);
#pragma unroll
        for (int ni = 0; ni < FN_; ni++) w[ni] = *(const bf16x8 *)(ring + st + wb + ni * 16 * BK);
    };
    auto mfmas = [&](const bf16x8 (&a)[FM_], const bf16x8 (&w)[FN_]) {
#pragma unroll
        for (int mi = 0; mi < FM_; mi++)
#pragma unroll
            for (int ni = 0; ni < FN_; ni++)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[ni], a[mi], acc[mi][ni], 0, 0, 0);
    };
    /* a fragment read between products, whose operands are in registers */
    auto interleave = [&]() {
#pragma unroll
        for (int i = 0; i < FM_ + FN_; i++) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
    };
    barrier();   /* tile 0 */
    frags(0, ab0, wb0, a0, w0);
    for (int kt = 0, st = 0; kt < nk; kt++) {
        frags(st, ab1, wb1, a1, w1);
        mfmas(a0, w0);
        interleave();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
        barrier();   /* tile kt + 1 is there, tile kt is read */
        st = st == (NS - 1) * ST_ELEMS ? 0 : st + ST_ELEMS;
        frags(st, ab0, wb0, a0, w0);
        mfmas(a1, w1);
        interleave();
        __builtin_amdgcn_sched_barrier(0);
    }

    /* lane l holds row lr of each 16x16 tile at the 4 columns lg*4 .. lg*4+3 */
    const int M = pr.M, N = pr.N, ldo = pr.ldo;
    const float *vec = pr.vec;
    const bool aligned = (ldo & 3) == 0 && ((uintptr_t)pr.out & 15) == 0 && ((uintptr_t)vec & 15) == 0;
    if (pr.epi == IRIS_EPI_SWIGLU) {
        /* 64 columns of the wave are 32 gate rows, then the matching 32 up rows */
#pragma unroll
        for (int g = 0; g < FN_ / 4; g++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int col = ((n0 + wn * TN + g * 64) >> 1) + h * 16 + lg * 4;
                if (col >= (N >> 1)) continue;   /* N % 64 == 0: all four columns or none */
#pragma unroll
                for (int mi = 0; mi < FM_; mi++) {
                    const int row = m0 + wm * TM + mi * 16 + lr;
                    if (row >= M) continue;
                    const f32x4 gt = acc[mi][4 * g + h], up = acc[mi][4 * g + 2 + h];
                    uint16_t y[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) y[r] = f2bf_hw(silu_fast(gt[r]) * up[r]);
                    uint16_t *dst = (uint16_t *)pr.out + (size_t)row * ldo + col;
                    if (aligned) {
                        *(uint2 *)dst = make_uint2((uint32_t)y[0] | ((uint32_t)y[1] << 16),
                                                   (uint32_t)y[2] | ((uint32_t)y[3] << 16));
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; r++) dst[r] = y[r];
                    }
                }
            }
        return;
    }
#pragma unroll
    for (int ni = 0; ni < FN_; ni++) {
        const int col = n0 + wn * TN + ni * 16 + lg * 4;
        const bool cols4 = aligned && col + 3 < N;
        const float vdef = pr.epi == IRIS_EPI_GATED_ADD ? 1.0f : 0.0f;
        float v[4];
        if (cols4 && vec) {
            const float4 q = *(const float4 *)(vec + col);
            v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = vec && col + r < N ? vec[col + r] : vdef;
        }
#pragma unroll
        for (int mi = 0; mi < FM_; mi++) {
            const int row = m0 + wm * TM + mi * 16 + lr;
            if (row >= M) continue;
            const f32x4 x = acc[mi][ni];
            const size_t o = (size_t)row * ldo + col;
            if (cols4 && pr.epi != IRIS_EPI_F32_T) {
                if (pr.epi == IRIS_EPI_BF16) {
                    *(uint2 *)((uint16_t *)pr.out + o) =
                        make_uint2((uint32_t)f2bf_hw(x[0] + v[0]) | ((uint32_t)f2bf_hw(x[1] + v[1]) << 16),
                                   (uint32_t)f2bf_hw(x[2] + v[2]) | ((uint32_t)f2bf_hw(x[3] + v[3]) << 16));
                } else {
                    float4 *dst = (float4 *)((float *)pr.out + o);
                    float4 y = make_float4(x[0] + v[0], x[1] + v[1], x[2] + v[2], x[3] + v[3]);
                    if (pr.epi == IRIS_EPI_GATED_ADD) {
                        y = *dst;
                        y.x += v[0] * x[0]; y.y += v[1] * x[1]; y.z += v[2] * x[2]; y.w += v[3] * x[3];
                    } else if (pr.epi == IRIS_EPI_ADD) {
                        const float4 q = *dst;
                        y.x = q.x + y.x; y.y = q.y + y.y; y.z = q.z + y.z; y.w = q.w + y.w;
                    }
                    *dst = y;
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (col + r >= N) continue;
                    float *const f = (float *)pr.out + (pr.epi == IRIS_EPI_F32_T ? (size_t)(col + r) * ldo + row : o + r);
                    const float y = x[r] + v[r];
                    if (pr.epi == IRIS_EPI_BF16) ((uint16_t *)pr.out)[o + r] = f2bf_hw(y);
                    else if (pr.epi == IRIS_EPI_GATED_ADD) *f += v[r] * x[r];
                    else if (pr.epi == IRIS_EPI_ADD) *f += y;
                    else *f = y;
                }
            }
        }
    }
}

/* the tile shapes of gemm_ring_kernel: 6 stages of 24 KiB, 4 of 32 KiB */
enum { RING_NONE, RING_64, RING_128 };
constexpr int RING_BM[] = {0, 64, 128}, RING_BN = 128;

template <int FM_, int FN_, int NS> int launch_ring(const dim3 &grid, const GemmParams &P) {
    constexpr size_t smem = (size_t)NS * 32 * (FM_ + FN_) * BK * 2;
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    std::call_once(once, [] {
        attr = hipFuncSetAttribute((const void *)gemm_ring_kernel<FM_, FN_, NS>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    });
    if (iris_check(attr, "gemm_ring smem attribute")) return -1;
    IRIS_LAUNCH((gemm_ring_kernel<FM_, FN_, NS>), grid, dim3(512), smem, iris_stream(), P);
    return 0;
}

/* Split-K partials of up to MAXP problems, reduced in one launch: each
 * output element is the sum of its problem's partials in chunk order
 * (deterministic), then that problem's epilogue. A thread takes VW = vw[i]
 * consecutive output elements of a row (4 where the partial rows, the output
 * and the bias allow 16-byte accesses, else 1); each element gets the same
 * additions either way. */
struct ReduceParams {
    iris_gemm_problem_t p[MAXP];
    const float *ws[MAXP];
    long long stride[MAXP];
    int chunks[MAXP], vw[MAXP];
    long long start[MAXP + 1];   /* first work item of each problem; start[n] = all */
    int n;
};

__global__ void splitk_reduce_kernel(const ReduceParams R) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= R.start[R.n]) return;
    int pi = 0;
#pragma unroll
    for (int j = 1; j < MAXP; j++)
        if (j < R.n && i >= R.start[j]) pi = j;
    const iris_gemm_problem_t p = R.p[pi];
    const float *ws = R.ws[pi];
    const long long stride = R.stride[pi];
    const int splits = R.chunks[pi];
    const int nout = p.epi == IRIS_EPI_SWIGLU ? p.N / 2 : p.N;
    if (R.vw[pi] == 4) {
        const long long e = (i - R.start[pi]) * 4;
        const int m = (int)(e / nout), c = (int)(e % nout);
        if (p.epi == IRIS_EPI_SWIGLU) {
            /* W rows interleaved in 32-row gate / up groups; c % 4 == 0 keeps
             * the four columns in one group */
            const int gc = (c >> 5) * 64 + (c & 31);
            float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f), u = g;
            for (int k = 0; k < splits; k++) {
                const float *row = ws + k * stride + (size_t)m * p.N;
                const float4 a = ld_stream((const float4 *)(row + gc)), b = ld_stream((const float4 *)(row + gc + 32));
                g.x += a.x; g.y += a.y; g.z += a.z; g.w += a.w;
                u.x += b.x; u.y += b.y; u.z += b.z; u.w += b.w;
            }
            *(uint2 *)((uint16_t *)p.out + (size_t)m * p.ldo + c) =
                make_uint2((uint32_t)f2bf_hw(silu_fast(g.x) * u.x) | ((uint32_t)f2bf_hw(silu_fast(g.y) * u.y) << 16),
                           (uint32_t)f2bf_hw(silu_fast(g.z) * u.z) | ((uint32_t)f2bf_hw(silu_fast(g.w) * u.w) << 16));
            return;
        }
        float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int k = 0; k < splits; k++) {
            const float4 a = ld_stream((const float4 *)(ws + k * stride + (size_t)m * p.N + c));
            s.x += a.x; s.y += a.y; s.z += a.z; s.w += a.w;
        }
        const float vd = p.epi == IRIS_EPI_GATED_ADD ? 1.0f : 0.0f;
        const float4 v = p.vec ? *(const float4 *)(p.vec + c) : make_float4(vd, vd, vd, vd);
        const size_t o = (size_t)m * p.ldo + c;
        switch (p.epi) {
        case IRIS_EPI_F32:
            *(float4 *)((float *)p.out + o) = make_float4(s.x + v.x, s.y + v.y, s.z + v.z, s.w + v.w);
            break;
        case IRIS_EPI_BF16:
            *(uint2 *)((uint16_t *)p.out + o) =
                make_uint2((uint32_t)f2bf_hw(s.x + v.x) | ((uint32_t)f2bf_hw(s.y + v.y) << 16),
                           (uint32_t)f2bf_hw(s.z + v.z) | ((uint32_t)f2bf_hw(s.w + v.w) << 16));
            break;
        case IRIS_EPI_GATED_ADD: {
            float4 *dst = (float4 *)((float *)p.out + o);
            float4 y = *dst;
            y.x += v.x * s.x; y.y += v.y * s.y; y.z += v.z * s.z; y.w += v.w * s.w;
            *dst = y;
            break;
        }
        case IRIS_EPI_ADD: {
            float4 *dst = (float4 *)((float *)p.out + o);
            float4 y = *dst;
            y.x += s.x + v.x; y.y += s.y + v.y; y.z += s.z + v.z; y.w += s.w + v.w;
            *dst = y;
            break;
        }
        default: break;
        }
        return;
    }
    const long long e = i - R.start[pi];
    const int m = (int)(e / nout), c = (int)(e % nout);
    if (p.epi == IRIS_EPI_SWIGLU) {
        const int gc = (c >> 5) * 64 + (c & 31);
        float g = 0.0f, u = 0.0f;
        for (int k = 0; k < splits; k++) {
            g += ws[k * stride + (size_t)m * p.N + gc];
            u += ws[k * stride + (size_t)m * p.N + gc + 32];
        }
        ((uint16_t *)p.out)[(size_t)m * p.ldo + c] = f2bf_hw(silu_fast(g) * u);
        return;
    }
    float s = 0.0f;
    for (int k = 0; k < splits; k++) s += ws[k * stride + (size_t)m * p.N + c];
    switch (p.epi) {
    case IRIS_EPI_F32: ((float *)p.out)[(size_t)m * p.ldo + c] = s + (p.vec ? p.vec[c] : 0.0f); break;
    case IRIS_EPI_BF16: ((uint16_t *)p.out)[(size_t)m * p.ldo + c] = f2bf_hw(s + (p.vec ? p.vec[c] : 0.0f)); break;
    case IRIS_EPI_GATED_ADD: ((float *)p.out)[(size_t)m * p.ldo + c] += (p.vec ? p.vec[c] : 1.0f) * s; break;
    case IRIS_EPI_F32_T: ((float *)p.out)[(size_t)c * p.ldo + m] = s + (p.vec ? p.vec[c] : 0.0f); break;
    case IRIS_EPI_ADD: ((float *)p.out)[(size_t)m * p.ldo + c] += s + (p.vec ? p.vec[c] : 0.0f); break;
    default: break;
    }
}

/* the reduce launch over the split problems of a launch (n of them) */
int launch_reduce(const iris_gemm_problem_t *ps, float *const *ws, const long long *stride, const int *chunks, int n) {
    ReduceParams R;
    memset(&R, 0, sizeof(R));
    R.n = n;
    long long items = 0;
    for (int i = 0; i < n; i++) {
        const iris_gemm_problem_t &p = ps[i];
        R.p[i] = p;
        R.ws[i] = ws[i];
        R.stride[i] = stride[i];
        R.chunks[i] = chunks[i];
        const int nout = p.epi == IRIS_EPI_SWIGLU ? p.N / 2 : p.N;
        const int ob = p.epi == IRIS_EPI_BF16 || p.epi == IRIS_EPI_SWIGLU ? 8 : 16;
        const bool v4 = p.epi != IRIS_EPI_F32_T && nout % 4 == 0 && p.N % 4 == 0 && p.ldo % 4 == 0 &&
                        ((uintptr_t)p.out % ob) == 0 && ((uintptr_t)p.vec % 16) == 0 && ((uintptr_t)ws[i] % 16) == 0;
        R.vw[i] = v4 ? 4 : 1;
        R.start[i] = items;
        items += (long long)p.M * nout / R.vw[i];
    }
    for (int i = n; i <= MAXP; i++) R.start[i] = items;
    if (items == 0) return 0;
    IRIS_LAUNCH(splitk_reduce_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, iris_stream(), R);
    return iris_launch_check("splitk_reduce_kernel");
}

int check_problem(const iris_gemm_problem_t &p) {
    if (p.K <= 0 || p.K % BK) return iris_set_error("gemm: K=%d must be a positive multiple of %d", p.K, BK);
    if (p.lda % 8 || p.ldw % 8 || p.lda < p.K || p.ldw < p.K)
        return iris_set_error("gemm: lda=%d ldw=%d must be multiples of 8 and >= K=%d", p.lda, p.ldw, p.K);
    if (((uintptr_t)p.A | (uintptr_t)p.W) & 15) return iris_set_error("gemm: A/W must be 16-byte aligned");
    if (!p.A || !p.W || !p.out) return iris_set_error("gemm: null operand");
    if (p.epi == IRIS_EPI_SWIGLU && (p.N % 64)) return iris_set_error("gemm: SwiGLU needs N %% 64 == 0");
    if (p.epi < 0 || p.epi > IRIS_EPI_ADD) return iris_set_error("gemm: epilogue %d", p.epi);
    if (p.K2 < 0 || p.K2 % BK) return iris_set_error("gemm: K2=%d must be a multiple of %d", p.K2, BK);
    if (p.K2 > 0) {
        if (!p.A2 || !p.W2 || (((uintptr_t)p.A2 | (uintptr_t)p.W2) & 15))
            return iris_set_error("gemm: second segment operands null or not 16-byte aligned");
        if (p.lda2 % 8 || p.ldw2 % 8 || p.lda2 < p.K2 || p.ldw2 < p.K2)
            return iris_set_error("gemm: lda2=%d ldw2=%d must be multiples of 8 and >= K2=%d", p.lda2, p.ldw2, p.K2);
        if ((long long)BM * p.lda2 * 2 >= (1LL << 31) || (long long)BN * p.ldw2 * 2 >= (1LL << 31))
            return iris_set_error("gemm: second segment leading dimension too large");
    }
    const int ldo_need = p.epi == IRIS_EPI_SWIGLU ? p.N / 2 : p.epi == IRIS_EPI_F32_T ? p.M : p.N;
    if (p.ldo < ldo_need) return iris_set_error("gemm: ldo=%d < %d", p.ldo, ldo_need);
    /* 32-bit buffer offsets: one tile's rows must span < 2 GiB */
    if ((long long)BM * p.lda * 2 >= (1LL << 31) || (long long)BN * p.ldw * 2 >= (1LL << 31))
        return iris_set_error("gemm: leading dimension too large");
    return 0;
}

}  // namespace

namespace {

/* the row passes of iris_hip_gemm_fill_tail; done: the reduce launch took them */
struct RowTail {
    const iris_row_tail_t *t;
    bool done;
};

/* whether one row pass over the partials of these split problems (nr of n in
 * the launch) is what t asks for: whole rows of at most 4096 columns in 16-byte
 * chunks, in the order of the rows it updates */
bool tail_fits(const iris_gemm_problem_t *ps, float *const *ws, int nr, int n, const iris_row_tail_t &t) {
    const bool sand = t.x != nullptr;
    if (nr != n || (sand && n != 1) || (!sand && !t.norm)) return false;
    const int N = ps[0].N;
    const float *const x = sand ? t.x : t.norm->x;
    const int ldx = sand ? N : t.norm->ldx;
    long long rows = 0;
    for (int i = 0; i < n; i++) {
        const iris_gemm_problem_t &p = ps[i];
        if (p.N != N || ((uintptr_t)ws[i] & 15) || ((uintptr_t)p.vec & 15)) return false;
        if (sand ? p.epi != IRIS_EPI_F32 || p.vec : p.epi != IRIS_EPI_GATED_ADD || p.ldo != ldx ||
                                                         (const float *)p.out != x + rows * ldx)
            return false;
        rows += p.M;
    }
    /* a block per row: fewer rows than half the CUs leave the sums of many
     * chunks to too few of them (37 rows: text encode 2802 us with the separate
     * passes, 2934 in one) */
    if (rows * 2 < iris_cu_count()) return false;
    if (N % 4 || N > 4096 || ldx % 4 || ldx < N || ((uintptr_t)x & 15)) return false;
    if (sand && (((uintptr_t)t.w | (uintptr_t)t.gate) & 15)) return false;
    if (!t.norm) return true;
    const iris_norm_args_t &a = *t.norm;
    return a.x == x && a.ldx == ldx && a.cols == N && a.rows == rows &&
           (sand ? a.mode == IRIS_NORM_RMS : a.mode == IRIS_NORM_RMS || a.mode == IRIS_NORM_LN_MOD);
}

int launch_tail(const iris_gemm_problem_t *ps, float *const *ws, const long long *stride, const int *chunks, int n,
                const iris_row_tail_t &t) {
    iris_reduce_rows_t R;
    memset(&R, 0, sizeof(R));
    int rows = 0;
    for (int i = 0; i < n; i++) {
        R.ws[i] = ws[i];
        R.vec[i] = t.x ? t.gate : ps[i].vec;
        R.stride[i] = stride[i];
        R.chunks[i] = chunks[i];
        R.start[i] = rows;
        rows += ps[i].M;
    }
    R.n = n;
    R.cols = ps[0].N;
    R.x = t.x ? t.x : (float *)ps[0].out;
    R.ldx = t.x ? ps[0].N : ps[0].ldo;
    if (t.x) {
        R.w = t.w;
        R.eps = t.eps;
    }
    if (t.norm) {
        R.has_norm = 1;
        R.norm = *t.norm;
    }
    return iris_reduce_rows(&R, rows);
}

/* One launch of up to MAXP problems. want[i] > 1 (want may be NULL) splits
 * problem i over K into that many chunks of whole K steps: its f32 partials
 * go to the workspace (after those of the split problems before it) and one
 * reduce launch after the GEMM sums them and applies the epilogues. Tiles
 * are 256 wide, or 224 wide (plain GEMM, no SwiGLU output written by the
 * tiles) when that needs fewer rounds of tile widths: with one block per CU
 * a launch takes ceil(blocks / CUs) rounds, each as long as one tile's width.
 * The tile width does not change any output element's accumulation order.
 * phase1 > 0: the tiles of the first phase1 problems are dispatched before
 * those of the others (a launch whose last problems fill a part-empty last
 * round); bnt > 0 forces the tile width. bmt = 128: 128 x 256 tiles (no
 * second K segment). */
int launch_gemm(const iris_gemm_problem_t *probs, int n, const int *want, float *ws, size_t ws_bytes,
                int phase1 = 0, int force_bnt = 0, int bmt = BM, int ring = RING_NONE, RowTail *tail = nullptr) {
    if (!probs || n < 1 || n > MAXP) return iris_set_error("gemm: %d problems (1..%d)", n, MAXP);
    if (ring) bmt = RING_BM[ring];
    GemmParams P;
    memset(&P, 0, sizeof(P));
    P.nprob = n;
    bool seg2 = false, swiglu_tiles = false, split = false;
    size_t ws_used = 0;
    for (int i = 0; i < n; i++) {
        const iris_gemm_problem_t &p = probs[i];
        P.p[i] = p;
        P.chunks[i] = 1;
        if (p.M <= 0 || p.N <= 0) continue;
        if (check_problem(p)) return -1;
        if (bmt != BM && p.K2) return iris_set_error("gemm: tiles of %d rows take no second K segment", bmt);
        P.tiles_m[i] = (p.M + bmt - 1) / bmt;
        if (want && want[i] > 1) {
            const int nk = p.K / BK;
            const int kchunk = (nk + want[i] - 1) / want[i] * BK;
            const int chunks = (p.K + kchunk - 1) / kchunk;
            /* K of one step leaves one chunk: that is the plain product */
            if (chunks > 1) {
                if (p.K2) return iris_set_error("gemm_splitk: no second K segment");
                P.chunks[i] = chunks;
                P.kchunk[i] = kchunk;
                P.ws_stride[i] = (long long)p.M * p.N;
                P.ws[i] = ws + ws_used / sizeof(float);
                ws_used += (size_t)chunks * P.ws_stride[i] * sizeof(float);
                split = true;
            }
        }
        seg2 = seg2 || p.K2 > 0;
        swiglu_tiles = swiglu_tiles || (p.epi == IRIS_EPI_SWIGLU && P.chunks[i] == 1);
    }
    if (split && (!ws || ((uintptr_t)ws & 15) || ws_used > ws_bytes))
        return iris_set_error("gemm_splitk: workspace of %zu bytes for %zu bytes of f32 partials", ws_bytes, ws_used);
    long long t256 = 0, t224 = 0;
    for (int i = 0; i < n; i++) {
        if (!P.tiles_m[i]) continue;
        t256 += (long long)P.tiles_m[i] * ((probs[i].N + 255) / 256) * P.chunks[i];
        t224 += (long long)P.tiles_m[i] * ((probs[i].N + 223) / 224) * P.chunks[i];
    }
    if (t256 == 0) return 0;
    int bnt = BN;
    const int cus = iris_cu_count();
    if (ring) {
        bnt = RING_BN;
    } else if (bmt != BM) {
        bnt = BN;
    } else if (force_bnt == 224 && !seg2 && !swiglu_tiles) {
        bnt = 224;
    } else if (!force_bnt && !seg2 && !swiglu_tiles && cus > 0) {
        const long long w256 = (t256 + cus - 1) / cus * BN, w224 = (t224 + cus - 1) / cus * 224;
        if (w224 * 100 < w256 * 97) bnt = 224;
    }
    int total = 0;
    for (int i = 0; i < n; i++) {
        P.tile_start[i] = total;
        if (!P.tiles_m[i]) continue;
        P.tiles_n[i] = (probs[i].N + bnt - 1) / bnt;
        total += P.tiles_m[i] * P.tiles_n[i] * P.chunks[i];
    }
    for (int i = n; i <= MAXP; i++) P.tile_start[i] = total;
    P.total = total;
    if (phase1 > 0 && phase1 < n) {
        P.phase_tiles = P.tile_start[phase1];
        P.phase_blocks = (P.phase_tiles + 7) / 8 * 8;
    }
    P.per_xcd = (total - P.phase_tiles + 7) / 8;
    const dim3 grid(P.phase_blocks + 8 * P.per_xcd);
    if (ring) {
        if (ring == RING_64 ? launch_ring<2, 4, 6>(grid, P) : launch_ring<4, 4, 4>(grid, P)) return -1;
    } else if (bmt != BM)
        IRIS_LAUNCH((gemm_bf16_kernel<0, 256, 128>), grid, dim3(NT), 0, iris_stream(), P);
    else if (bnt == 224)
        IRIS_LAUNCH((gemm_bf16_kernel<0, 224>), grid, dim3(NT), 0, iris_stream(), P);
    else if (seg2)
        IRIS_LAUNCH(gemm_bf16_kernel<3>, grid, dim3(NT), 0, iris_stream(), P);
    else
        IRIS_LAUNCH(gemm_bf16_kernel<0>, grid, dim3(NT), 0, iris_stream(), P);
    if (iris_launch_check("gemm_bf16_kernel")) return -1;
    if (!split) return 0;
    iris_gemm_problem_t rp[MAXP];
    float *rws[MAXP];
    long long rstride[MAXP];
    int rchunks[MAXP], nr = 0;
    for (int i = 0; i < n; i++)
        if (P.chunks[i] > 1) {
            rp[nr] = probs[i];
            rws[nr] = P.ws[i];
            rstride[nr] = P.ws_stride[i];
            rchunks[nr++] = P.chunks[i];
        }
    if (tail && tail_fits(rp, rws, nr, n, *tail->t)) {
        tail->done = true;
        return launch_tail(rp, rws, rstride, rchunks, nr, *tail->t);
    }
    return launch_reduce(rp, rws, rstride, rchunks, nr);
}

}  // namespace

/* A launch whose 256-row tiles fill at most half of the CUs runs on 128-row
 * tiles (twice the tiles, one round; the same additions per element): on the
 * products measured (512-1536 rows) they took 0.71-0.79 of the time. */
extern "C" int iris_hip_gemm(const iris_gemm_problem_t *probs, int n) {
    if (!probs || n < 1 || n > MAXP) return iris_set_error("gemm: %d problems (1..%d)", n, MAXP);
    const int cus = iris_cu_count();
    long long tiles = 0;
    bool seg2 = false;
    for (int i = 0; i < n; i++) {
        if (probs[i].M <= 0 || probs[i].N <= 0) continue;
        tiles += (long long)((probs[i].M + BM - 1) / BM) * ((probs[i].N + BN - 1) / BN);
        seg2 = seg2 || probs[i].K2 > 0;
    }
    const bool half = tiles > 0 && !seg2 && cus > 0 && 2 * tiles <= cus;
    return launch_gemm(probs, n, nullptr, nullptr, 0, 0, 0, half ? 128 : BM);
}

/* Split-K partials without a caller workspace: a file-scope device array of
 * IRIS_NOALLOC_SCRATCH_BYTES, held by each GPU the library runs on until the
 * process ends. Host code never passes the array's name to a kernel (on the
 * host it is a stand-in, not a device address): its device address is looked
 * up once per device with hipGetSymbolAddress and kept per device. Every
 * call on a GPU shares that GPU's array, so calls that overlap on one GPU
 * (different streams, threads) race. Each chunk's partial overwrites its
 * whole M x N region, so nothing is cleared between calls. */
__device__ __align__(256) float scratch[IRIS_NOALLOC_SCRATCH_BYTES / sizeof(float)];

namespace {
constexpr int MAX_DEVICES = 64;
void *g_scratch_ptr[MAX_DEVICES];
std::mutex g_scratch_mutex;

float *scratch_ptr() {
    int dev = -1;
    if (iris_check(hipGetDevice(&dev), "noalloc: hipGetDevice")) return nullptr;
    if (dev < 0 || dev >= MAX_DEVICES) {
        iris_set_error("noalloc: device %d outside 0..%d", dev, MAX_DEVICES - 1);
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        if (iris_check(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "noalloc: hipGetSymbolAddress")) return nullptr;
        g_scratch_ptr[dev] = ptr;
    }
    return (float *)g_scratch_ptr[dev];
}
}  // namespace

extern "C" int iris_hip_gemm_splitk_noalloc(const iris_gemm_problem_t *p, int splits) {
    if (!p) return iris_set_error("gemm_splitk_noalloc: null problem");
    if (splits <= 1) return iris_hip_gemm(p, 1);
    if (p->M <= 0 || p->N <= 0) return 0;
    if (check_problem(*p)) return -1;
    const int nk = p->K / BK;
    const int kchunk = (nk + splits - 1) / splits * BK;
    const size_t chunks = (size_t)((p->K + kchunk - 1) / kchunk);
    /* one chunk is the plain product, which needs no scratch */
    if (chunks <= 1) return iris_hip_gemm(p, 1);
    const size_t need = chunks * (size_t)p->M * (size_t)p->N * sizeof(float);
    if (need > IRIS_NOALLOC_SCRATCH_BYTES)
        return iris_set_error("gemm_splitk_noalloc: %zu chunks x %d x %d f32 partials need %zu bytes, the scratch "
                              "holds %zu", chunks, p->M, p->N, need, (size_t)IRIS_NOALLOC_SCRATCH_BYTES);
    float *ws = scratch_ptr();
    if (!ws) return -1;
    return iris_hip_gemm_splitk(p, splits, ws, IRIS_NOALLOC_SCRATCH_BYTES);
}

extern "C" int iris_hip_gemm_splitk(const iris_gemm_problem_t *p, int splits, float *ws, size_t ws_bytes) {
    if (!p) return iris_set_error("gemm_splitk: null problem");
    return launch_gemm(p, 1, &splits, ws, ws_bytes);
}

namespace {

/* the problem restricted to output rows [r0, M) (rows = true) or output
 * columns [c0, N) */
iris_gemm_problem_t sub_problem(const iris_gemm_problem_t &p, bool rows, int from) {
    iris_gemm_problem_t q = p;
    const size_t es = (p.epi == IRIS_EPI_BF16 || p.epi == IRIS_EPI_SWIGLU) ? 2 : 4;
    if (rows) {
        q.A = p.A + (size_t)from * p.lda;
        q.out = (char *)p.out + es * (p.epi == IRIS_EPI_F32_T ? (size_t)from : (size_t)from * p.ldo);
        q.M = p.M - from;
    } else {
        q.W = p.W + (size_t)from * p.ldw;
        if (p.vec) q.vec = p.vec + from;
        const size_t col = p.epi == IRIS_EPI_SWIGLU ? (size_t)from / 2 : (size_t)from;
        q.out = (char *)p.out + es * (p.epi == IRIS_EPI_F32_T ? col * p.ldo : col);
        q.N = p.N - from;
    }
    return q;
}

/* A product whose 256-wide tiles fill one or more whole rounds of blocks on
 * the CUs and then a part-empty last round: the whole rounds run as they
 * are, and the leftover tiles -- taken as whole tile rows (or columns) at
 * the end of the output -- are split over K across the CUs the whole rounds
 * free, in the same launch, with one reduce launch after it. Taken when a
 * cost estimate in units of one round (the split pieces' share of a round,
 * plus the reduce pass's traffic at 4.5 TB/s and its launch) beats the plain
 * launch at either tile width by 8 %. Returns the number of chunks (0: not
 * taken) and the two problems. */
int tail_plan(const iris_gemm_problem_t &p, size_t ws_bytes, iris_gemm_problem_t parts[2]) {
    const int cus = iris_cu_count();
    if (cus <= 0 || p.K2 || p.M <= 0 || p.N <= 0) return 0;
    const int tm = (p.M + BM - 1) / BM, tn = (p.N + BN - 1) / BN, nk = p.K / BK;
    const long long T = (long long)tm * tn, full = T / cus, tail = T - full * cus;
    if (full < 1 || tail == 0 || nk < 8) return 0;
    const int kr = (int)((tail + tn - 1) / tn), kc = (int)((tail + tm - 1) / tm);
    const bool rows_ok = kr < tm, cols_ok = kc < tn && !(p.epi == IRIS_EPI_SWIGLU && (p.N % 64));
    if (!rows_ok && !cols_ok) return 0;
    const bool rows = rows_ok && (!cols_ok || (long long)kr * tn <= (long long)kc * tm);
    const int from = rows ? (tm - kr) * BM : (tn - kc) * BN;
    const long long tail_tiles = rows ? (long long)kr * tn : (long long)kc * tm;
    const size_t part_bytes = rows ? (size_t)(p.M - from) * p.N * 4 : (size_t)p.M * (p.N - from) * 4;
    int pieces = (int)std::min<long long>(cus / tail_tiles, nk / 4);
    while (pieces > 1 && (size_t)pieces * part_bytes > ws_bytes) pieces--;
    if (pieces < 2) return 0;
    /* estimates in units of one round of 256-wide tiles over the whole K */
    const double round_us = 2.0 * BM * BN * (double)p.K / 5.1e12 * 1e6;
    const bool rmw = p.epi == IRIS_EPI_GATED_ADD || p.epi == IRIS_EPI_ADD;
    const double out_bytes = part_bytes / 4.0 * ((p.epi == IRIS_EPI_BF16 || p.epi == IRIS_EPI_SWIGLU) ? 2 : 4) *
                             (rmw ? 2 : 1);
    const double reduce_us = ((double)pieces * part_bytes + out_bytes) / 4.5e12 * 1e6 + 6.0;
    const double split_cost = (double)full + 1.0 / pieces + reduce_us / round_us;
    double plain = (double)full + 1.0;
    if (p.epi != IRIS_EPI_SWIGLU) {
        const long long t224 = (long long)tm * ((p.N + 223) / 224);
        plain = std::min(plain, (double)((t224 + cus - 1) / cus) * 224.0 / 256.0);
    }
    if (split_cost > 0.92 * plain) return 0;
    parts[0] = p;
    if (rows) parts[0].M = from;
    else parts[0].N = from;
    parts[1] = sub_problem(p, rows, from);
    return pieces;
}

}  // namespace

namespace {

/* The faster plan of gemm_ring_kernel for these problems: at most 128 rows
 * each, in up to one round of blocks, or one problem whose 128 x 128 tiles
 * fill most of a round unsplit; K of 2048 and more (32 steps). Elsewhere its
 * tiles load more bytes per product than the larger ones and lose (measured,
 * cold weights, us, two-stage kernel's plan / this kernel unsplit: 512 x 2560
 * x 4096 32.7 / 40.8, 384 x 2560 x 9728 42.3 / 98.3; 768 x 18432 x 3072 69 /
 * 122). The estimate (us): K steps per block times a step of the tile, plus
 * launch, prologue and epilogue, plus the reduce pass; not less than the
 * weights' read at the device's copy rate. It and the two-stage kernel's are
 * each fitted as a whole to their own kernel's times (a reduce pass is 3.5 in
 * this one and 6 in that one) and know nothing of the row pass that may take
 * the reduce's place. Measured, cold weights, us between events (two-stage
 * plan -> this kernel): 37 rows, N x K 6144 x 2560 22.8 -> 19.0, 2560 x 4096
 * 23.2 -> 19.3, 19456 x 2560 SwiGLU 36.6 -> 28.1, 2560 x 9728 30.3 -> 24.0;
 * 96 rows, 3840 x 3840 26.0 -> 20.6; 128 rows, 2560 x 9728 34.4 -> 30.3; 512
 * x 6144 x 2560 (192 tiles, no reduce pass) 42.2 -> 33.1, 385 rows 41.3 ->
 * 25.7. Nowhere in 84 shapes of 8 to 128 rows is the choice slower than the
 * two-stage plan by more than the runs differ. It leaves gains: K below 2048
 * keeps the two-stage plan, whose chunk count does not depend on the number of
 * rows, though this kernel is faster there too (128 x 3840 x 1024 21.8 / 11.2,
 * 37 x 3840 x 1536 19.3 / 17.3); 65 x 19456 x 2560 38.1 / 31.9 and 37 x 20480
 * x 3840 46.2 / 37.3 fall to the estimate's 3 % margin and floor; one problem
 * of 257 to 384 rows by N 6144 (144 tiles) is below the line of 60 % of a
 * round, 34.9 / 27.7 at 300. */
struct RingPlan {
    int ring, splits;
    double us;
};

RingPlan ring_plan(const iris_gemm_problem_t *probs, int n, int cus, size_t ws_bytes) {
    RingPlan best = {RING_NONE, 1, 1e30};
    long long tiles[3] = {0, 0, 0};
    double per = 0, out = 0, wbytes = 0;
    int min_nk = 1 << 30, max_nk = 0, max_m = 0;
    for (int i = 0; i < n; i++) {
        const iris_gemm_problem_t &p = probs[i];
        if (p.M <= 0 || p.N <= 0) continue;
        for (int r = RING_64; r <= RING_128; r++)
            tiles[r] += (long long)((p.M + RING_BM[r] - 1) / RING_BM[r]) * ((p.N + RING_BN - 1) / RING_BN);
        per += (double)p.M * p.N * 4;
        out += (double)p.M * p.N * (p.epi == IRIS_EPI_GATED_ADD || p.epi == IRIS_EPI_ADD ? 8 : 4);
        wbytes += (double)p.N * p.K * 2;
        min_nk = std::min(min_nk, p.K / BK);
        max_nk = std::max(max_nk, p.K / BK);
        max_m = std::max(max_m, p.M);
    }
    for (int r = RING_64; r <= RING_128 && min_nk >= 32; r++) {
        if (tiles[r] > cus) continue;
        if (max_m > 128 && (n > 1 || r != RING_128 || tiles[r] * 10 < cus * 6LL)) continue;
        const int most = max_m > 128 ? 1 : (int)std::min<long long>(cus / tiles[r], min_nk / 4);
        for (int s = 1; s <= std::max(1, most) && (s == 1 || s * per <= (double)ws_bytes); s++) {
            const double steps = (max_nk + s - 1) / s;
            double us = r == RING_64 ? steps * 0.40 + 9.0 : steps * 0.56 + 9.5;
            us = std::max(us, wbytes / 5.1e6 + 6.0);
            if (s > 1) us += (s * per + out) / 4.5e6 + 3.5;
            if (us < best.us) best = {r, s, us};
        }
    }
    return best;
}

}  // namespace

namespace {

int fill_impl(const iris_gemm_problem_t *probs, int n, float *ws, size_t ws_bytes, RowTail *tail) {
    if (!probs || n < 1 || n > MAXP) return iris_set_error("gemm_fill: %d problems (1..%d)", n, MAXP);
    const int cus = iris_cu_count();
    long long tiles = 0, tiles128 = 0;
    size_t per = 0, out_bytes = 0;
    int min_nk = 1 << 30, max_nk = 0;
    bool seg2 = false;
    for (int i = 0; i < n; i++) {
        const iris_gemm_problem_t &p = probs[i];
        if (p.M <= 0 || p.N <= 0) continue;
        tiles += (long long)((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
        tiles128 += (long long)((p.M + 127) / 128) * ((p.N + BN - 1) / BN);
        per += (size_t)p.M * (size_t)p.N * sizeof(float);
        const bool rmw = p.epi == IRIS_EPI_GATED_ADD || p.epi == IRIS_EPI_ADD;
        const size_t es = p.epi == IRIS_EPI_BF16 ? 2 : p.epi == IRIS_EPI_SWIGLU ? 1 : rmw ? 8 : 4;
        out_bytes += (size_t)p.M * (size_t)p.N * es;
        min_nk = std::min(min_nk, p.K / BK);
        max_nk = std::max(max_nk, p.K / BK);
        seg2 = seg2 || p.K2 > 0;
    }
    /* Tiles filling at most half of the CUs and a long K: split K into up to
     * CUs / tiles chunks of at least 4 K steps, as many as the workspace
     * holds, on 256 x 256 tiles, or on 128 x 256 tiles where those still fit
     * one round (twice the tiles, so fewer chunks: less reduce traffic and
     * shorter f32 partial epilogues) and an estimate of the launch and its
     * reduce is lower. The estimate (us): K steps per block times the step
     * time of the tile shape with the chip partly idle, plus a tile's
     * prologue and partial store, plus the reduce pass's traffic at 4.5 TB/s
     * and its launch; measured over the encoder, caption, embedder and
     * 512x512 products, it picks the faster shape in each. */
    if (tiles > 0 && !seg2 && cus > 0 && ws && 2 * tiles <= cus && min_nk >= 8) {
        auto fit = [&](long long s) {
            s = std::max(1LL, std::min<long long>(s, min_nk / 4));
            while (s > 1 && (size_t)s * per > ws_bytes) s--;
            return (int)s;
        };
        auto est = [&](bool half, int s) {
            const double step = half ? 0.9 : 1.3, fixed = half ? 8.0 : 14.0;
            const double red = s > 1 ? ((double)s * per + out_bytes) / 4.5e6 + 6.0 : 0.0;
            return (double)max_nk / s * step + fixed + red;
        };
        const int s256 = fit(cus / tiles);
        const int s128 = tiles128 <= cus ? fit(cus / tiles128) : 0;
        int want[MAXP];
        const RingPlan r = ring_plan(probs, n, cus, ws_bytes);
        if (r.ring && r.us < 0.97 * std::min(est(false, s256), s128 > 0 ? est(true, s128) : 1e30)) {
            for (int i = 0; i < n; i++) want[i] = r.splits;
            return launch_gemm(probs, n, r.splits > 1 ? want : nullptr, ws, ws_bytes, 0, 0, BM, r.ring, tail);
        }
        if (s128 > 0 && est(true, s128) < est(false, s256)) {
            for (int i = 0; i < n; i++) want[i] = s128;
            return launch_gemm(probs, n, s128 > 1 ? want : nullptr, ws, ws_bytes, 0, 0, 128, RING_NONE, tail);
        }
        if (s256 > 1) {
            for (int i = 0; i < n; i++) want[i] = s256;
            return launch_gemm(probs, n, want, ws, ws_bytes, 0, 0, BM, RING_NONE, tail);
        }
    }
    if (n == 1 && ws && !((uintptr_t)ws & 15)) {
        iris_gemm_problem_t parts[2];
        const int pieces = tail_plan(probs[0], ws_bytes, parts);
        if (pieces > 1) {
            if (check_problem(probs[0])) return -1;
            const int want[2] = {1, pieces};
            return launch_gemm(parts, 2, want, ws, ws_bytes, 1, BN);
        }
    }
    return launch_gemm(probs, n, nullptr, nullptr, 0);
}

}  // namespace

extern "C" int iris_hip_gemm_fill_n(const iris_gemm_problem_t *probs, int n, float *ws, size_t ws_bytes) {
    return fill_impl(probs, n, ws, ws_bytes, nullptr);
}

extern "C" int iris_hip_gemm_fill_tail(const iris_gemm_problem_t *probs, int n, float *ws, size_t ws_bytes,
                                       const iris_row_tail_t *tail) {
    if (!probs || !tail || (tail->x && (n != 1 || probs->epi != IRIS_EPI_F32 || probs->vec || probs->ldo != probs->N ||
                                        !tail->w)))
        return iris_set_error("gemm_fill_tail: a gated residual follows one F32 product of contiguous rows");
    RowTail t = {tail, false};
    if (fill_impl(probs, n, ws, ws_bytes, &t)) return -1;
    if (t.done) return 0;
    if (tail->x && iris_hip_rms_gated_add(tail->x, (const float *)probs->out, tail->w, tail->gate, probs->M, probs->N,
                                          tail->eps, 0))
        return -1;
    return tail->norm ? iris_hip_rownorm(tail->norm) : 0;
}

extern "C" int iris_hip_gemm_ring(const iris_gemm_problem_t *probs, int n, int rows, int splits, float *ws,
                                  size_t ws_bytes) {
    if (rows != 64 && rows != 128) return iris_set_error("gemm_ring: tiles of %d rows (64 or 128)", rows);
    int want[MAXP];
    for (int i = 0; i < MAXP; i++) want[i] = splits;
    return launch_gemm(probs, n, splits > 1 ? want : nullptr, ws, ws_bytes, 0, 0, BM, rows == 64 ? RING_64 : RING_128);
}

extern "C" int iris_hip_gemm_fill(const iris_gemm_problem_t *p, float *ws, size_t ws_bytes) {
    if (!p) return iris_set_error("gemm_fill: null problem");
    return iris_hip_gemm_fill_n(p, 1, ws, ws_bytes);
}

namespace {

/* per row, one wave: the tiles' (max, sum) pairs merged into (max, 1 / sum);
 * lane j takes tiles j, j + 64, ..., then the wave's butterfly (a fixed
 * order) */
__global__ __launch_bounds__(256) void softmax_rows_kernel(const float2 *stat, int tiles, int rows,
                                                           float2 *row_out) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= rows) return;
    const float2 *s = stat + (size_t)r * tiles;
    float m = -INFINITY;
    for (int t = lane; t < tiles; t += 64) m = fmaxf(m, s[t].x);
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    float l = 0.0f;
    for (int t = lane; t < tiles; t += 64) l += s[t].y * __builtin_amdgcn_exp2f(s[t].x - m);
    for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
    if (lane == 0) row_out[r] = make_float2(m, 1.0f / l);
}

}  // namespace

extern "C" int iris_hip_softmax_scores(const uint16_t *q, int ld_q, const uint16_t *k, int ld_k, int M, int N, int d,
                                       float scale, uint16_t *p, int ld_p, int pad_n, float *stat, float *row) {
    if (!q || !k || !p || !stat || !row || M <= 0 || N <= 0)
        return iris_set_error("softmax_scores: null buffer or empty shape (%d x %d)", M, N);
    const int tiles_n = (N + BN - 1) / BN;
    if (pad_n < N || pad_n > tiles_n * BN || ld_p < pad_n)
        return iris_set_error("softmax_scores: pad %d for %d columns (ld %d)", pad_n, N, ld_p);
    if (((uintptr_t)stat | (uintptr_t)row) & 7) return iris_set_error("softmax_scores: statistics not 8-byte aligned");
    if ((long long)M * tiles_n >= (1LL << 31)) return iris_set_error("softmax_scores: too many rows");
    GemmParams P;
    memset(&P, 0, sizeof(P));
    iris_gemm_problem_t &pr = P.p[0];
    pr.A = q; pr.lda = ld_q; pr.W = k; pr.ldw = ld_k; pr.out = p; pr.ldo = ld_p;
    pr.M = M; pr.N = N; pr.K = d; pr.epi = IRIS_EPI_BF16;
    if (check_problem(pr)) return -1;
    P.nprob = 1;
    P.chunks[0] = 1;
    P.tiles_m[0] = (M + BM - 1) / BM;
    P.tiles_n[0] = tiles_n;
    P.total = P.tiles_m[0] * tiles_n;
    for (int i = 1; i <= MAXP; i++) P.tile_start[i] = P.total;
    P.per_xcd = (P.total + 7) / 8;
    P.sm_scale = scale * 1.44269504088896341f;   /* log2(e): scores in log2 units */
    P.sm_stat = (float2 *)stat;
    P.sm_pad = pad_n;
    const dim3 grid(8 * P.per_xcd);
    IRIS_LAUNCH(gemm_bf16_kernel<4>, grid, dim3(NT), 0, iris_stream(), P);
    if (iris_launch_check("gemm_bf16_kernel<4> (row statistics)")) return -1;
    IRIS_LAUNCH(softmax_rows_kernel, dim3((M + 3) / 4), dim3(256), 0, iris_stream(), (const float2 *)stat, tiles_n, M,
                (float2 *)row);
    if (iris_launch_check("softmax_rows_kernel")) return -1;
    P.sm_row = (const float2 *)row;
    IRIS_LAUNCH(gemm_bf16_kernel<5>, grid, dim3(NT), 0, iris_stream(), P);
    return iris_launch_check("gemm_bf16_kernel<5> (probabilities)");
}

namespace {

/* checks a convolution and fills what its kernels need for tiles of bnt
 * output channels (bnt 0: 128 for at most 128 channels -- the decoder's
 * full-resolution convolutions -- else 256; the same additions per element) */
int conv_params(const iris_conv3x3_t *c, int bnt, GemmParams &P) {
    if (!c || !c->in || !c->wt || !c->out) return iris_set_error("conv3x3: null operand");
    if (c->cin < 64 || c->cin > 8192 || (c->cin & (c->cin - 1)))
        return iris_set_error("conv3x3: cin=%d must be a power of two in 64..8192", c->cin);
    if (c->up < 0 || c->up > 2) return iris_set_error("conv3x3: up=%d (0, 1 or 2)", c->up);
    if (c->H <= 0 || c->W <= 0 || c->H > 8000 || c->W > 8000 || (c->up == 1 && ((c->H | c->W) & 1)))
        return iris_set_error("conv3x3: output %dx%d", c->H, c->W);
    if (c->epi != IRIS_EPI_F32 && c->epi != IRIS_EPI_BF16 && c->epi != IRIS_EPI_ADD)
        return iris_set_error("conv3x3: epilogue %d (F32, BF16 or ADD)", c->epi);
    const size_t in_pix = c->up == 1 ? (size_t)(c->H / 2) * (c->W / 2)
                          : c->up == 2 ? (size_t)(2 * c->H) * (2 * c->W) : (size_t)c->H * c->W;
    const size_t in_bytes = in_pix * (size_t)c->cin * 2;
    if (in_bytes >= (1ull << 31)) return iris_set_error("conv3x3: input of %zu bytes (< 2 GiB)", in_bytes);
    if ((long long)c->H * c->W >= (1LL << 31)) return iris_set_error("conv3x3: too many pixels");
    iris_gemm_problem_t p;
    memset(&p, 0, sizeof(p));
    p.A = c->in;
    p.W = c->wt;
    p.out = c->out;
    p.vec = c->bias;
    p.M = c->H * c->W;
    p.N = c->cout;
    p.K = 9 * c->cin;
    p.lda = p.ldw = p.K;
    p.ldo = c->ldo;
    p.epi = c->epi;
    memset(&P, 0, sizeof(P));
    P.p[0] = p;
    if (p.N <= 0) return 0;
    if (check_problem(p)) return -1;
    P.nprob = 1;
    if (!bnt) bnt = p.N <= 128 ? 128 : BN;
    P.tiles_m[0] = (p.M + BM - 1) / BM;
    P.tiles_n[0] = (p.N + bnt - 1) / bnt;
    P.conv_h = c->H;
    P.conv_w = c->W;
    P.conv_up = c->up;
    P.conv_cpt_shift = __builtin_ctz((unsigned)c->cin) - 6;
    P.conv_cin_bshift = __builtin_ctz((unsigned)c->cin) + 1;
    P.conv_in_bytes = (unsigned)in_bytes;
    if (c->gn_part) {
        const int G = c->gn_groups, cpg = G > 0 && p.N % G == 0 ? p.N / G : 0;
        if (cpg == 0 || cpg % 4 || bnt % cpg || c->splits > 1 || ((uintptr_t)c->gn_part & 7))
            return iris_set_error("conv3x3: GroupNorm statistics need groups of a multiple of 4 channels dividing the "
                                  "%d-wide tile, no split-K and an 8-byte aligned buffer (cout %d, groups %d, splits %d)",
                                  bnt, p.N, G, c->splits);
        P.gn_part = c->gn_part;
        P.gn_groups = G;
    }
    return 0;
}

/* Output channels per tile of iris_hip_conv3x3, for arguments conv_params
 * takes: 128 also where 256 leave half the CUs without a tile (a GroupNorm's
 * group must stay within one): 128 x 128 pixels out, stride 2, 256 -> 256 (64
 * tiles of 256) 62 -> 42 us; 64 x 64, 512 -> 512 split by 4 (128) 39 -> 30. */
int conv_width(const iris_conv3x3_t *c) {
    const long long tiles = ((long long)c->H * c->W + BM - 1) / BM * (c->cout <= 128 ? 1 : (c->cout + BN - 1) / BN);
    const bool few = 2 * tiles * (c->splits > 1 ? c->splits : 1) <= iris_cu_count();
    return c->cout <= 128 || (few && (!c->gn_part || 128 % (c->cout / c->gn_groups) == 0)) ? 128 : BN;
}

}  // namespace

extern "C" int iris_hip_conv3x3(const iris_conv3x3_t *c) {
    GemmParams P;
    if (conv_params(c, 0, P)) return -1;
    const iris_gemm_problem_t &p = P.p[0];
    if (p.N <= 0) return 0;
    const int bnt = conv_width(c);
    if (conv_params(c, bnt, P)) return -1;
    int chunks = 1;
    long long stride = 0;
    P.chunks[0] = 1;
    if (c->splits > 1) {
        const int nk = p.K / BK;
        P.kchunk[0] = (nk + c->splits - 1) / c->splits * BK;
        chunks = (p.K + P.kchunk[0] - 1) / P.kchunk[0];
        stride = (long long)p.M * p.N;
        if (!c->ws || ((uintptr_t)c->ws & 15) || (size_t)chunks * stride * sizeof(float) > c->ws_bytes)
            return iris_set_error("conv3x3: split-K workspace of %zu bytes for %d x %d x %d f32", c->ws_bytes, chunks,
                                  p.M, p.N);
    }
    P.total = P.tiles_m[0] * P.tiles_n[0] * chunks;
    for (int i = 1; i <= MAXP; i++) P.tile_start[i] = P.total;
    P.per_xcd = (P.total + 7) / 8;
    if (chunks > 1) {
        P.chunks[0] = chunks;
        P.ws[0] = c->ws;
        P.ws_stride[0] = stride;
    }
    if (c->up == 2 && bnt == 128)
        IRIS_LAUNCH((gemm_bf16_kernel<2, 128>), dim3(8 * P.per_xcd), dim3(NT), 0, iris_stream(), P);
    else if (c->up == 2)
        IRIS_LAUNCH(gemm_bf16_kernel<2>, dim3(8 * P.per_xcd), dim3(NT), 0, iris_stream(), P);
    else if (bnt == 128)
        IRIS_LAUNCH((gemm_bf16_kernel<1, 128>), dim3(8 * P.per_xcd), dim3(NT), 0, iris_stream(), P);
    else
        IRIS_LAUNCH(gemm_bf16_kernel<1>, dim3(8 * P.per_xcd), dim3(NT), 0, iris_stream(), P);
    if (iris_launch_check("gemm_bf16_kernel<conv>")) return -1;
    if (chunks == 1) return 0;
    float *rws = c->ws;
    return launch_reduce(&p, &rws, &stride, &chunks, 1);
}

namespace {

/* 3x3 convolution, stride 1 (UP: the input read through a nearest 2x
 * upsample), one 16 x 16 pixel tile x 128 output channels per block. The
 * implicit GEMM above loads an input pixel from L2 once per tap: 48 KiB per
 * 64-wide K step of a 256 x 128 tile, more than a CU gets in the time of the
 * step's products. Here the tile's pixels and their halo (18 x 18, or 10 x 10
 * before the upsample) are staged once per 64 channels and all nine taps read
 * their fragments from that patch; only the weights (16 KiB per step) stream:
 * 185 KiB per 64 channels (192 with the loads past the patch's end) instead of
 * 432. The tile then leaves through LDS, the residual of IRIS_EPI_ADD in
 * flight while it is staged. Measured against the implicit GEMM, us: 1024 x
 * 1024, 128 -> 128 with the residual 498 -> 367 (f32 stream in and out: 210 of
 * it), bf16 out 342 -> 311, 256 -> 128 619 -> 497; 512 x 512, 512 -> 256 467
 * -> 429 (1.44 PFLOP/s); 256 x 256 x 512 upsampled 219 -> 196 (1.58); 128 x
 * 128, 512 -> 512 80.5 -> 53.8. The direct stores of the accumulators took 614
 * where it takes 367: 64-byte pieces, behind a load each.
 *
 * 8 waves as in gemm_ring_kernel: waves 0..3 compute (2x2, wave tile 8 pixel
 * rows x TN / 2 channels), waves 4..7 load, one barrier per K step (a tap of a
 * 64-channel chunk; taps within chunks). Weights go through 4 stages. The
 * patch has two buffers: chunk c+1's is loaded in the first AL steps of chunk
 * c, and it is complete when step 8 of chunk c waits for the weights of the
 * next step, which each step issues after its patch loads (loads of a wave
 * complete in order).
 *
 * LDS patch pixel (r, c) is row r PW + c of 128 bytes, its 16-byte chunk k
 * stored at k ^ ((c / 2) mod 8): PW is even, so 16 neighbouring columns of a
 * row lie in 16 distinct bank groups, and the swizzle depends on the lane
 * only: every fragment is one of six lane addresses plus a constant. */
struct ConvParams {
    const uint16_t *in, *wt;
    void *out;
    const float *bias;
    int H, W, cin, cout, ldo, epi;
    int tx, tn, tiles, total, per_xcd;   /* tile columns, 128-channel tiles, blocks of a split, of all */
    int cps;                             /* 64-channel chunks per split of K */
    float *ws;                           /* f32 partials of the splits, ws_stride apart; NULL: one split */
    long long ws_stride;
    unsigned in_bytes;
    double *gn_part;
    int gn_groups;
    uint16_t *bf16_out;   /* IRIS_EPI_ADD: the sum leaves here in bf16, out stays */
};

template <bool UP, int TN>
__global__ __launch_bounds__(512) void conv3x3_patch_kernel(const ConvParams P) {
    constexpr int PW = UP ? 10 : 18, NPX = PW * PW, SLOTS = (NPX + 7) / 8, AL = (SLOTS + 7) / 8;
    constexpr int A_BYTES = SLOTS * 1024, W_BYTES = TN * BK * 2, NSW = 4, FM_ = 8, FN_ = TN / 32, WL = TN / 32;
    extern __shared__ __attribute__((aligned(16))) char sm[];
    __shared__ float gnl[2048 / TN][TN / 4][2];
    const int L = (blockIdx.x & 7) * P.per_xcd + (blockIdx.x >> 3);
    if (L >= P.total) return;
    /* scalar registers for what the buffer resources and addresses are made of */
    const int split = __builtin_amdgcn_readfirstlane(L / P.tiles), Ls = L - split * P.tiles;
    const int tile = __builtin_amdgcn_readfirstlane(Ls / P.tn), ty = __builtin_amdgcn_readfirstlane(tile / P.tx);
    const int n0 = (Ls - tile * P.tn) * TN, y0 = ty * 16, x0 = (tile - ty * P.tx) * 16;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = split * P.cps, chunks = min(P.cps, P.cin / BK - c0);   /* this block's 64-channel chunks */
    char *const wring = sm + 2 * A_BYTES;
    const bool gn = P.gn_part != nullptr;
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wave >= 4) {
        const int lw = wave & 3, drow = lane >> 3, dch = lane & 7;
        const __amdgpu_buffer_rsrc_t a_rsrc =
            __builtin_amdgcn_make_buffer_rsrc((void *)P.in, (short)0, (int)P.in_bytes, 0x00020000);
        const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(P.wt + (size_t)n0 * 9 * P.cin), (short)0, min(TN, P.cout - n0) * 9 * P.cin * 2, 0x00020000);
        /* patch slot j holds patch pixels 8j .. 8j+7; this wave's are
         * 8s + 2 lw + i of step s (the last slot again past the end). Pixels
         * outside the image, and past the patch, read as zero: an offset past
         * the end of the buffer */
        const int hin = UP ? P.H / 2 : P.H, win = UP ? P.W / 2 : P.W;
        const int py0 = (UP ? y0 / 2 : y0) - 1, px0 = (UP ? x0 / 2 : x0) - 1;
        int a_off[12];   /* 2 AL of them */
#pragma unroll
        for (int i = 0; i < 2 * AL; i++) {
            const int px = min((i >> 1) * 8 + lw * 2 + (i & 1), SLOTS - 1) * 8 + drow;
            const int r = px / PW, c = px - r * PW, gy = py0 + r, gx = px0 + c;
            const bool ok = px < NPX && (unsigned)gy < (unsigned)hin && (unsigned)gx < (unsigned)win;
            a_off[i] = ok ? (gy * win + gx) * P.cin * 2 + ((dch ^ ((c >> 1) & 7)) << 4) : (int)0x80000000u;
        }
        int w_off[2];
#pragma unroll
        for (int par = 0; par < 2; par++)
            w_off[par] = (lw * (TN / 4) + drow) * 9 * P.cin * 2 + ((dch ^ ((4 * par + (drow >> 1)) & 7)) << 4);
        const int w_step = 8 * 9 * P.cin * 2;
        auto dma_a = [&](int chunk, int i) {
            const int slot = min((i >> 1) * 8 + lw * 2 + (i & 1), SLOTS - 1);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                a_rsrc, (lds_void *)(sm + (chunk & 1) * A_BYTES + slot * 1024), 16, a_off[i],
                (c0 + min(chunk, chunks - 1)) * (BK * 2), 0, 0);
        };
        auto dma_w = [&](int stage, int chunk, int tap) {
            const int soff = (tap * P.cin + (c0 + chunk) * BK) * 2;
#pragma unroll
            for (int i = 0; i < WL; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (lds_void *)(wring + stage * W_BYTES + (lw * WL + i) * 1024),
                                                         16, w_off[i & 1] + i * w_step, soff, 0, 0);
        };
#pragma unroll
        for (int i = 0; i < 2 * AL; i++) dma_a(0, i);
#pragma unroll
        for (int g = 0; g < NSW; g++) dma_w(g, 0, g);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(waitcnt_imm((NSW - 1) * WL, 15));
        barrier();
        /* Step s waits for the weights of the next step: issued 3 steps ago,
         * before the loads of the last two. After the barrier it issues its
         * patch loads, then the weights of step g + 4 (past the last step,
         * the last chunk's again). A macro: the wait is an immediate. */
#define CONV_STEP(s)                                                                                               \
    do {                                                                                                           \
        __builtin_amdgcn_s_waitcnt(                                                                                \
            waitcnt_imm(2 * WL + (((s) + 8) % 9 < AL ? 2 : 0) + (((s) + 7) % 9 < AL ? 2 : 0), 15));                     \
        barrier();                                                                                                 \
        if ((s) < AL) {                                                                                            \
            dma_a(chunk + 1, (s) < AL ? 2 * (s) : 0);                                                              \
            dma_a(chunk + 1, (s) < AL ? 2 * (s) + 1 : 0);                                                          \
        }                                                                                                          \
        dma_w(st, min(chunk + ((s) + NSW) / 9, chunks - 1), ((s) + NSW) % 9);                                      \
        st = (st + 1) & (NSW - 1);                                                                                 \
    } while (0)
        for (int chunk = 0, st = 0; chunk < chunks; chunk++) {
            CONV_STEP(0); CONV_STEP(1); CONV_STEP(2);
            CONV_STEP(3); CONV_STEP(4); CONV_STEP(5);
            CONV_STEP(6); CONV_STEP(7); CONV_STEP(8);
        }
#undef CONV_STEP
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));   /* no DMA outstanding past here */
    }
    const int wm = (wave >> 1) & 1, wn = wave & 1;
    f32x4 acc[FM_][FN_];
    if (wave < 4) {
#pragma unroll
    for (int i = 0; i < FM_; i++)
#pragma unroll
        for (int j = 0; j < FN_; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0.0f;
    /* lane addresses of the patch per tap column and half, of the weights per half */
    int ab[3][2], wb[2];
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
#pragma unroll
        for (int dx = 0; dx < 3; dx++) {
            const int c = UP ? ((lr + dx - 1) >> 1) + 1 : lr + dx;
            ab[dx][kk] = (wm * (UP ? 4 : 8) * PW + c) * 128 + (((kk * 4 + lg) ^ ((c >> 1) & 7)) << 4);
        }
        wb[kk] = swz(wn * (TN / 2) + lr, kk * 4 + lg) * 2;
    }
    bf16x8 a0[FM_], w0[FN_], a1[FM_], w1[FN_];
    auto frags = [&](int buf, int st, int s, int kk, bf16x8 (&a)[FM_], bf16x8 (&w)[FN_]) {
        const char *const pa = sm + buf * A_BYTES + ab[s % 3][kk], *const pw = wring + st * W_BYTES + wb[kk];
#pragma unroll
        for (int ni = 0; ni < FN_; ni++) w[ni] = *(const bf16x8 *)(pw + ni * 16 * BK * 2);
#pragma unroll
        for (int mi = 0; mi < FM_; mi++) {
            const int r = UP ? ((mi + s / 3 - 1) >> 1) + 1 : mi + s / 3;
            a[mi] = *(const bf16x8 *)(pa + r * PW * 128);
        }
    };
    auto mfmas = [&](const bf16x8 (&a)[FM_], const bf16x8 (&w)[FN_]) {
#pragma unroll
        for (int mi = 0; mi < FM_; mi++)
#pragma unroll
            for (int ni = 0; ni < FN_; ni++)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[ni], a[mi], acc[mi][ni], 0, 0, 0);
    };
    auto interleave = [&]() {
#pragma unroll
        for (int i = 0; i < FM_ + FN_; i++) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, FM_ * FN_ / (FM_ + FN_), 0);
        }
    };
    barrier();   /* chunk 0's patch, step 0's weights */
    frags(0, 0, 0, 0, a0, w0);
    for (int chunk = 0, st = 0; chunk < chunks; chunk++) {
#pragma unroll
        for (int s = 0; s < 9; s++) {
            frags(chunk & 1, st, s, 1, a1, w1);
            mfmas(a0, w0);
            interleave();
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
            barrier();
            st = (st + 1) & (NSW - 1);
            frags(s == 8 ? (chunk + 1) & 1 : chunk & 1, st, (s + 1) % 9, 0, a0, w0);
            mfmas(a1, w1);
            interleave();
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    }

    /* The tile leaves through LDS (free now), as f32 rows of TN channels and
     * 16 bytes: all eight waves store it, TN / 4 lanes a whole pixel row, and the
     * residual is in flight meanwhile. Thread t has the 4 channels 4 c4
     * of pixels pr0 + OPX i. Pixels outside the image take an address inside
     * it and are not stored. */
    constexpr int OSTR = TN + 4, OPX = 2048 / TN, ONI = 256 / OPX;
    static_assert(256 * OSTR * 4 <= 2 * A_BYTES + NSW * W_BYTES || UP, "the f32 tile fits the rings");
    float *const ot = (float *)sm;
    const int c4 = tid & (TN / 4 - 1), pr0 = tid / (TN / 4), px = pr0 & 15, py = pr0 >> 4, col = n0 + c4 * 4;
    const bool part = P.ws != nullptr;   /* a split's partial sums: plain f32 rows of cout channels */
    void *const out = part ? (void *)(P.ws + split * P.ws_stride) : P.out;
    const bool to_bf16 = !part && (P.epi == IRIS_EPI_BF16 || P.bf16_out);
    uint16_t *const out16 = P.bf16_out ? P.bf16_out : (uint16_t *)out;
    const int epi = part ? IRIS_EPI_F32 : P.epi, ldo = part ? P.cout : P.ldo;
    const float *const bias = part ? nullptr : P.bias;
    size_t off[ONI];
    float4 res[ONI];
#pragma unroll
    for (int i = 0; i < ONI; i++) {
        off[i] = ((size_t)min(y0 + i * (OPX / 16) + py, P.H - 1) * P.W + min(x0 + px, P.W - 1)) * ldo + col;
        if (epi == IRIS_EPI_ADD) res[i] = *(const float4 *)((const float *)out + off[i]);
    }
    __syncthreads();   /* every read and every load of the rings is done */
    if (wave < 4) {
#pragma unroll
        for (int mi = 0; mi < FM_; mi++)
#pragma unroll
            for (int ni = 0; ni < FN_; ni++)
                *(f32x4 *)(ot + ((wm * 8 + mi) * 16 + lr) * OSTR + wn * (TN / 2) + ni * 16 + lg * 4) = acc[mi][ni];
    }
    __syncthreads();
    const float4 v = bias ? *(const float4 *)(bias + col) : make_float4(0, 0, 0, 0);
    float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int i = 0; i < ONI; i++) {
        const bool on = y0 + i * (OPX / 16) + py < P.H && x0 + px < P.W;
        const float4 q = *(const float4 *)(ot + (i * OPX + pr0) * OSTR + c4 * 4);
        float4 r = make_float4(q.x + v.x, q.y + v.y, q.z + v.z, q.w + v.w);
        if (epi == IRIS_EPI_ADD) {
            r.x += res[i].x; r.y += res[i].y; r.z += res[i].z; r.w += res[i].w;
        }
        if (on) {
            if (to_bf16)
                *(uint2 *)(out16 + off[i]) =
                    make_uint2((uint32_t)f2bf_hw(r.x) | ((uint32_t)f2bf_hw(r.y) << 16),
                               (uint32_t)f2bf_hw(r.z) | ((uint32_t)f2bf_hw(r.w) << 16));
            else
                *(float4 *)((float *)out + off[i]) = r;
            s1 += (r.x + r.y) + (r.z + r.w);
            s2 += (r.x * r.x + r.y * r.y) + (r.z * r.z + r.w * r.w);
        }
    }
    if (gn) {
        /* per thread the sums of 4 channels over its pixels, then the OPX
         * threads of the channels and the group's chunks in order, in f64 */
        gnl[pr0][c4][0] = s1;
        gnl[pr0][c4][1] = s2;
        __syncthreads();
        const int cpg = P.cout / P.gn_groups;
        if (tid < TN / cpg) {
            double s = 0.0, q = 0.0;
            for (int c = tid * cpg / 4; c < (tid + 1) * cpg / 4; c++)
                for (int m = 0; m < OPX; m++) {
                    s += (double)gnl[m][c][0];
                    q += (double)gnl[m][c][1];
                }
            double *dst = P.gn_part + ((size_t)tile * P.gn_groups + n0 / cpg + tid) * 2;
            dst[0] = s;
            dst[1] = q;
        }
    }
}

template <bool UP, int TN> int launch_patch(const ConvParams &P) {
    constexpr int PW = UP ? 10 : 18;
    /* the rings, or the f32 tile of the epilogue */
    constexpr size_t ring = 2 * ((PW * PW + 7) / 8) * 1024 + 4 * TN * BK * 2, ot = 256 * (TN + 4) * 4;
    constexpr size_t smem = ring > ot ? ring : ot;
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    std::call_once(once, [] {
        attr = hipFuncSetAttribute((const void *)conv3x3_patch_kernel<UP, TN>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)smem);
    });
    if (iris_check(attr, "conv3x3 smem attribute")) return -1;
    IRIS_LAUNCH((conv3x3_patch_kernel<UP, TN>), dim3(8 * P.per_xcd), dim3(512), smem, iris_stream(), P);
    return iris_launch_check("conv3x3_patch_kernel");
}

int launch_patch_of(int up, int tn, const ConvParams &P) {
    if (up) return tn == 64 ? launch_patch<true, 64>(P) : launch_patch<true, 128>(P);
    return tn == 64 ? launch_patch<false, 64>(P) : launch_patch<false, 128>(P);
}

}  // namespace

/* bf16_out (or NULL): the residual's sum in bf16 there, the f32 stream not
 * written back (bound by bytes: 512 x 512 x 256 saves 134 MB and a pass of
 * 400 MB; the 512 x 512 encode 1923 -> 1854 us, the 1024 x 1024 decode 11456
 * -> 11347 with it in the blocks before a resampling) */
static int conv_tiled(const iris_conv3x3_t *c, int *gn_blocks, uint16_t *bf16_out) {
    if (gn_blocks) *gn_blocks = 0;
    auto convert = [&]() {
        return bf16_out ? iris_hip_f32_to_bf16(bf16_out, (const float *)c->out, (size_t)c->H * c->W * c->cout) : 0;
    };
    auto other = [&]() {
        if (gn_blocks && c && c->gn_part) *gn_blocks = (c->H * c->W + 255) / 256;
        return iris_hip_conv3x3(c) ? -1 : convert();
    };
    if (!c || (c->up != 0 && c->up != 1) || c->H <= 0 || c->W <= 0 || c->cout <= 0 || c->splits > 1) return other();
    const int cus = iris_cu_count();
    const long long ty = (c->H + 15) / 16, tx = (c->W + 15) / 16, tiles = ty * tx * (c->cout / 128);
    const double area = (double)c->H * c->W;
    /* a GroupNorm group wider than a tile, or no whole number of channels, is the other kernel's to take or refuse */
    const int G = c->gn_part ? c->gn_groups : 0;
    const bool wide = c->gn_part && (G <= 0 || c->cout % G || 128 % (c->cout / G));
    if (c->cout % 128 || wide || c->ldo % 4 || (((uintptr_t)c->out | (uintptr_t)c->bias) & 15) || tiles >= (1LL << 28))
        return other();
    GemmParams chk;
    if (conv_params(c, 128, chk)) return -1;
    const int chunks = c->cin / BK;
    /* Past one round the kernel with the shorter rounds: tiles of 16 x 16
     * pixels come in other numbers than row tiles of 256, overshoot the image,
     * and have half the channels. The estimate (us) is a full round's time by
     * the 64-channel chunks and the last round's by its fill, fitted to 88
     * convolutions of 128 to 512 channels and sides of 17 to 1024 pixels, most
     * within 8 %; 7 more for the other kernel, whose output the pass after it
     * finds less of in L2 (144 x 144 x 512: apply pass 13 -> 17 us), so that
     * near ties stay here. Measured, this kernel / the other, bf16 out, 512 ->
     * 512: 144 x 144 94 / 93, 176 x 176 105 / 112, 180 x 180 (576 tiles / 254)
     * 145 / 114, 192 x 192 148 / 187, upsampled 180 x 180 138 / 115, 90 x 166
     * (264 tiles / 236 of 128 channels) 93 / 67, 17 x 640 94 / 62; 360 x 360,
     * 512 -> 256 248 / 225. With the choice instead of this kernel throughout:
     * 720 x 720 decode 6367 -> 6157 us, encode 3607 -> 3522, 1328 x 720 decode
     * 11229 -> 11059.
     * Within a round a tile's overshoot only uses idle CUs, and a lone chunk
     * (the layer in front of the decoder, f32 out) is bound by its stores in
     * both: 144 x 144 x 64 -> 512 28.1 / 28.7, 224 x 224 52.6 / 54.4, 180 x
     * 180 39.7 / 32.4. */
    if (tiles > cus && chunks > 1) {
        const int width = conv_width(c);
        const long long rows = ((long long)c->H * c->W + BM - 1) / BM * ((c->cout + width - 1) / width);
        const double epi = c->epi == IRIS_EPI_ADD ? 11.0 : c->epi == IRIS_EPI_F32 ? 5.0 : 0.0;
        const auto rounds = [&](long long n, double last, int power) {
            const double r = (double)((n + cus - 1) / cus), fill = (n - (r - 1) * cus) / cus;
            return r + last * (power == 3 ? fill * fill * fill : fill);
        };
        const double tiled = (10.0 + 5.0 * chunks) * (c->up ? 0.94 : 1.0) * (rounds(tiles, 0.2, 1) - 0.12);
        const double gemm = (width == 128 ? 10.0 + 7.0 * chunks + epi / 2 : 16.0 + 12.0 * chunks + epi) *
                            (rounds(rows, 0.26, 3) - 0.22) +
                            7.0 + (bf16_out ? 6.0 * area * c->cout / 4.5e6 + 3.5 : 0.0);   /* the conversion pass */
        if (gemm < tiled) return other();
    }
    const bool can = c->ws && !((uintptr_t)c->ws & 15);
    /* Few tiles: half their channels each where twice as many still have a CU
     * (a GroupNorm's group must stay within a tile), and a split over the
     * input channels, by an estimate (us): 0.5 per K step of 128 channels, 0.3
     * of 64, 8 per block, the partials written and read at 2.2 TB/s with one
     * launch more, and a statistics pass where the sums were asked for.
     * Measured, 128 channels / 64 / 64 split by 4: 64 x 64, 512 -> 512 (64
     * tiles of 128) 44.4 / 30.8 / 42.7; 96 x 96, 256 -> 256 (72) 26.4 / 18.6 /
     * 41.9; 64 x 128, 512 -> 512 (128) 46.5 / 38.0 / 73.5; 32 x 32, 512 -> 512
     * (16) 40.3 / 26.3 / 25.2; past a CU per tile 64 lose: 128 x 128, 512 ->
     * 512 (256) 59.3 / 70.8. */
    const bool can64 = !G || 64 % (c->cout / G) == 0;
    int splits = 1, tn = 128;
    double best = 1e30;
    for (int n = 128; n >= (can64 ? 64 : 128); n /= 2)
        for (int s = 1; s <= 8 && s <= chunks; s *= 2) {
            const double part = 4.0 * area * c->cout;
            if ((s > 1 || n < 128) && tiles * (128 / n) * s > cus) break;
            if (s > 1 && (!can || s * part > (double)c->ws_bytes)) break;
            const double us = 9.0 * ((chunks + s - 1) / s) * (n == 128 ? 0.5 : 0.3) + 8.0 +
                              (s > 1 ? (s + 1) * part / 2.2e6 + 3.5 + (c->gn_part ? 3.5 : 0.0) : 0.0);
            if (us < best) { best = us; splits = s; tn = n; }
        }
    ConvParams P;
    memset(&P, 0, sizeof(P));
    P.in = c->in; P.wt = c->wt; P.out = c->out; P.bias = c->bias;
    P.H = c->H; P.W = c->W; P.cin = c->cin; P.cout = c->cout; P.ldo = c->ldo; P.epi = c->epi;
    P.tx = (int)tx; P.tn = c->cout / tn; P.tiles = (int)(ty * tx * P.tn);
    P.cps = (chunks + splits - 1) / splits;
    P.total = P.tiles * splits; P.per_xcd = (P.total + 7) / 8;
    P.in_bytes = chk.conv_in_bytes;
    if (splits == 1) {
        P.gn_part = c->gn_part; P.gn_groups = c->gn_groups;
        if (gn_blocks && c->gn_part) *gn_blocks = (int)(ty * tx);
        P.bf16_out = bf16_out;
        return launch_patch_of(c->up, tn, P);
    }
    P.ws = c->ws;
    P.ws_stride = (long long)c->H * c->W * c->cout;
    if (launch_patch_of(c->up, tn, P)) return -1;
    return launch_reduce(&chk.p[0], &P.ws, &P.ws_stride, &splits, 1) ? -1 : convert();
}

extern "C" int iris_hip_conv3x3_tiled(const iris_conv3x3_t *c, int *gn_blocks) {
    return conv_tiled(c, gn_blocks, nullptr);
}

extern "C" int iris_hip_conv3x3_add_bf16(const iris_conv3x3_t *c, uint16_t *out) {
    if (!c || !out || c->epi != IRIS_EPI_ADD || c->ldo != c->cout || c->gn_part || ((uintptr_t)out & 7))
        return iris_set_error("conv3x3_add_bf16: bad arguments (a packed residual, no sums)");
    return conv_tiled(c, nullptr, out);
}
