/* q8_tile.hip: Y = X W^T for long prompts (more than 64 tokens) on the matrix cores.
 *
 * The sums are q8_gemm.hip's, bit for bit (a block's 32 columns in three bf16 limb MFMAs, the block
 * scale applied after them, the ranges of each K split in order, the splits' sums in split order),
 * so a token's output does not depend on which kernel computed it. What differs is the tile. The
 * streaming kernel of q8_gemm.hip gives a workgroup 64 tokens and a K split: for 512 tokens it reads
 * and converts the weights eight times, splits x into limbs once a row tile (48 times at 12288
 * rows), reads 12 KiB of limbs from LDS for 12 MFMAs, and writes and re-reads ks partials. Here:
 *
 *   ximage_k    x (or its RMS norm) as three bf16 limbs, once a product, in the order the tiles' LDS
 *               stages hold them: [pair of blocks][token tile][block][limb][lane] of 16 bytes;
 *   gemm_tile   a workgroup owns up to 128 tokens x 256 rows and all of K. The limbs of a pair of
 *               blocks go from the image straight into LDS (buffer loads to LDS, NB - 1 pairs ahead),
 *               the weights from HBM into registers by the wave that owns the rows; each is converted
 *               once for all the tile's tokens, and each limb read feeds every row tile of the wave.
 *               The splits' sums are added in registers: no partials, no second launch; the
 *               residual or the pair's SwiGLU is applied in the store.
 *
 * 12288 x 4096 at 512 tokens: 295 us as eight 64-token products, 160 us here (320 TFLOP/s of the
 * product, 960 of issued MFMA work, where a large bf16 library product reaches 1385 on this card:
 * both run at the clock the power limit leaves, 2.07 GHz measured under this kernel against 2.45 on
 * a quarter of the compute units). */
#include <hip/hip_runtime.h>

#include <stdio.h>
#include <stdlib.h>

#include "q8_device.h"

#include "q8_bf16.h"

template <int V>
struct tile_c {
    static constexpr int value = V;
};

/* ---------------------------------------------------------------- the limb image */

/* The limbs of token tile blockIdx.y's blocks [16 blockIdx.x, +16), one block a wave; lane L holds
 * token L & 15 and the columns KCOL(L >> 4) .. +7 of the block. What lies past t or past the last
 * block is zero. nw != NULL: of the RMS norm, nw[k] * (x[k] * s), s from the sum of x^2 in rmsnorm_k's
 * order (a thread's columns, the wave, the waves), a wave a token: every
 * workgroup of the tile sums its 16 tokens again, from the L2, which costs less than a launch of
 * its own (4.9 us at 512 tokens of 4096 columns, and its x written and read again). */
#define XIMG_BLOCKS 16
__global__ __launch_bounds__(64 * XIMG_BLOCKS) void ximage_k(const float *__restrict__ x, long xs, long t, long cols, const float *__restrict__ nw,
                                                            float eps, uint4 *__restrict__ img)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nb = (int)(cols / Q8_BLOCK), np = (nb + 1) / 2;
    __shared__ float scale[16];
    if (nw) {
        const long tok = 16 * (long)blockIdx.y + wave;
        const float *xr = x + (tok < t ? tok : t - 1) * xs;
        /* the lane's part of each of rmsnorm_k's waves */
        auto sum = [&](auto wc) {
            constexpr int W = decltype(wc)::value;
            float a[W];
#pragma unroll
            for (int q = 0; q < W; q++)
                a[q] = 0.0f;
            for (long k = 4 * (long)lane; k < cols; k += 256 * W) {
                float4 v[W];
#pragma unroll
                for (int q = 0; q < W; q++)
                    v[q] = *(const float4 *)(xr + (k + 256 * q < cols ? k + 256 * q : k));
#pragma unroll
                for (int q = 0; q < W; q++)
                    if (k + 256 * q < cols)
                        a[q] = q8_norm_add(v[q], a[q]);
            }
#pragma unroll
            for (int q = 0; q < W; q++)
                a[q] = q8_wave_sum_dpp(a[q]);
            if (lane == 0)
                scale[wave] = 1.0f / sqrtf(eps + q8_norm_fold<W>(a) / (float)cols);
        };
        if (cols <= 1024)
            sum(tile_c<4>{});
        else if (cols <= 2048)
            sum(tile_c<8>{});
        else
            sum(tile_c<16>{});
        __syncthreads();
    }
    const int b = (int)blockIdx.x * XIMG_BLOCKS + wave;
    if (b >= 2 * np)
        return;
    const long tok = 16 * (long)blockIdx.y + (lane & 15);
    const bool in = tok < t && b < nb;
    const long k0 = (long)(b < nb ? b : nb - 1) * Q8_BLOCK + kcol(lane >> 4);
    const float *px = x + (tok < t ? tok : t - 1) * xs + k0;
    float4 a = *(const float4 *)px, c = *(const float4 *)(px + 4);
    if (nw) {
        const float s = scale[lane & 15];
        const float4 g = *(const float4 *)(nw + k0), e = *(const float4 *)(nw + k0 + 4);
        a = make_float4(g.x * (a.x * s), g.y * (a.y * s), g.z * (a.z * s), g.w * (a.w * s));
        c = make_float4(e.x * (c.x * s), e.y * (c.y * s), e.z * (c.z * s), e.w * (c.w * s));
    }
    const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    uint4 h, m, o;
    xsplit8(in ? a : z, in ? c : z, h, m, o);
    uint4 *d = img + (((long)(b >> 1) * gridDim.y + blockIdx.y) * 2 + (b & 1)) * 192 + lane;
    d[0] = h;
    d[64] = m;
    d[128] = o;
}

/* ---------------------------------------------------------------- the product */

struct tile_args {
    int n;                        /* products (the pair: 2 matrices, one output) */
    const uint8_t *w[Q8_ROUND_MAX];
    float *y[Q8_ROUND_MAX];
    int rtn[Q8_ROUND_MAX];        /* 16-row tiles of each product */
    int spl[Q8_ROUND_MAX];        /* pairs of blocks a K split */
    int start[Q8_ROUND_MAX + 1];  /* first workgroup row tile of each product; start[n] = their count */
    const float *res;
    const void *img;
    int img_bytes, groups;        /* token groups of MT token tiles */
    long cols, t;
};

typedef __attribute__((address_space(3))) void tile_lds;

/* A workgroup of NW waves, MT token tiles x NW * RT row tiles (of each of the NP = 2 matrices of the
 * pair), all of K in steps of one pair of blocks.
 *
 * A step is 2 MT units, each one token tile against the wave's TR = NP * RT row tiles for one block:
 * 3 TR MFMAs, with the next unit's three limb reads, the previous unit's 4 TR scale FMAs and a share
 * of the step's other work (the loads of a later pair, the int8 to bf16 conversion of the next block)
 * between them. In program order the waves waited for each unit's limbs and results in turn, and all
 * of a step's loads issued at its start while no MFMA ran: 214 us at 12288 x 4096, 512 tokens, 167
 * with the units interleaved. (Loads to LDS by global_load_lds instead of the buffer form count in
 * lgkmcnt, which makes every limb read wait for all of them: 181 us.)
 *
 * Pair c's limbs and weights are issued in step c - NB + 1: first the SI loads of the stage, then the
 * 2 TR of the weights. At the start of step c a wave waits until at most VN = (NB - 2) (SI + 2 TR) +
 * 2 TR loads are outstanding, which leaves only loads issued after its part of stage c, and the
 * barrier then covers every wave's part; stage c + NB - 1 overwrites the buffer of step c - 1, whose
 * reads every wave has used before that barrier. Loads past the last pair repeat the last pair.
 *
 * 8 waves, two a SIMD, each hiding the other's waits: 4 waves with twice the row tiles measured
 * slower (246 against 214 us), and so did 6 (unequal SIMDs: a pair at 512 tokens 299 us with 33 %
 * fewer idle workgroup slots against 305). */
template <int MT, int RT, int NW, int NP, int NB>
__global__ __launch_bounds__(64 * NW) void gemm_tile(tile_args a)
{
    constexpr int TR = NP * RT;
    constexpr int SN = MT * 384;    /* 16-byte words of a stage */
    constexpr int SI = MT * 6 / NW; /* its 1 KiB loads a wave */
    static_assert(MT * 6 % NW == 0 && NB >= 3 && NB <= 4, "a stage divides among the waves");
    /* separate arrays, so that the reads of one do not wait for the loads of another */
    __shared__ uint4 s0[SN], s1[SN], s2[SN], s3[NB > 3 ? SN : 1];
    uint4 *bufs[NB];
    bufs[0] = s0;
    bufs[1] = s1;
    bufs[2] = s2;
    if constexpr (NB > 3)
        bufs[3] = s3;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nb = (int)(a.cols / Q8_BLOCK), np = (nb + 1) / 2;
    const int n = lane & 15, kq = lane >> 4;
    /* workgroups b, b + 8, ... share an XCD: the token groups of a row tile sit there next to each
     * other and read its weights from one L2 */
    const int seq = (int)blockIdx.x >> 3, group = seq % a.groups;
    const int wt = ((int)blockIdx.x & 7) + 8 * (seq / a.groups);
    if (wt >= a.start[NP == 2 ? 1 : a.n])
        return;
    int p = 0;
    if constexpr (NP == 1) {
#pragma unroll
        for (int k = 1; k < Q8_ROUND_MAX; k++)
            if (k < a.n && wt >= a.start[k])
                p = k;
    }
    const int rtn = a.rtn[p], spl = a.spl[p];
    const int rt0 = ((wt - a.start[p]) * NW + wave) * RT, tt0 = group * MT, ttn = (int)((a.t + 15) / 16);

    /* a row tile past the last one reads the last and stores nothing */
    const uint8_t *wq[TR], *wd[TR];
#pragma unroll
    for (int k = 0; k < TR; k++) {
        const int rt = rt0 + k % RT < rtn ? rt0 + k % RT : rtn - 1;
        wq[k] = a.w[NP == 2 ? k / RT : p] + (size_t)rt * 17 * (size_t)a.cols;
        wd[k] = wq[k] + 16 * (size_t)a.cols;
    }
    const unsigned woff = (unsigned)(n * a.cols + 16 * kq), doff = (unsigned)(2 * n * nb);
    const __amdgpu_buffer_rsrc_t irs = __builtin_amdgcn_make_buffer_rsrc((void *)a.img, 0, a.img_bytes, 0x00027000);
    const unsigned istep = (unsigned)ttn * 6144, ioff = (unsigned)tt0 * 6144 + (unsigned)(wave * SI) * 1024;
    /* load i of the wave's share of pair c's stage. Token tiles past the last one read the next pair's
     * tiles, or zeros past the image's end: tokens that are not stored, and no token's sums see another's */
    auto stage1 = [&](uint4 *buf, int c, int i) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(irs, (tile_lds *)(buf + (wave * SI + i) * 64), 16, lane * 16, (int)((unsigned)c * istep + ioff + i * 1024),
                                                 0, 0);
    };
    /* a row tile's weights of pair c, 16 bytes a lane, and its row's two scales as one load (2-byte
     * aligned where the row has an odd count of blocks; its last pair reads the two blocks before
     * the row's end, never past it) */
    struct __attribute__((packed, aligned(2))) u32u {
        uint32_t v;
    };
    struct wset {
        uint4 q[TR];
        uint32_t d[TR];
    };
    auto wload1 = [&](wset &S, int c, int k) __attribute__((always_inline)) {
        S.q[k] = *(const uint4 *)(wq[k] + (woff + 64u * (unsigned)c));
        S.d[k] = ((const u32u *)(wd[k] + (doff + (unsigned)(4 * c < 2 * nb - 4 ? 4 * c : 2 * nb - 4))))->v;
    };
    /* block h of pair c as MFMA operands: lanes 0-31 hold block 2c, 32-63 block 2c + 1 (q8_bf16.h).
     * The block past an odd count needs no mask: its limbs are zero and its weights finite, and its
     * scale becomes 0 (the row's last scale is the high half of that load) */
    struct ops {
        bf16x8 wb[TR];
        float d[TR];
    };
    const int odd = nb & 1;
    auto conv1 = [&](ops &O, const wset &S, int k, int h, int c) __attribute__((always_inline)) {
        const auto s02 = __builtin_amdgcn_permlane32_swap(S.q[k].x, S.q[k].z, false, false);
        const auto s13 = __builtin_amdgcn_permlane32_swap(S.q[k].y, S.q[k].w, false, false);
        O.wb[k] = q8_bf16(s02[h], s13[h]);
        const uint32_t dd = S.d[k] >> (odd && c == np - 1 ? 16 : 0);
        float d = q8_half((uint16_t)(h ? dd >> 16 : dd));
        asm("" : "+v"(d)); /* converted once here, not in each of its FMAs */
        O.d[k] = d;
    };
    auto lread = [&](uint4 (&xa)[3], const uint4 *buf, int m, int h) __attribute__((always_inline)) {
#pragma unroll
        for (int l = 0; l < 3; l++)
            xa[l] = buf[((m * 2 + h) * 3 + l) * 64 + lane];
    };

    f32x4 acc[TR][MT], tot[TR][MT]; /* the split being summed; the splits before it */
#pragma unroll
    for (int k = 0; k < TR; k++)
#pragma unroll
        for (int m = 0; m < MT; m++)
            acc[k][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int left = spl; /* pairs to the end of the split */
    bool first = true;
    auto fold = [&]() __attribute__((always_inline)) {
        if (--left == 0) {
#pragma unroll
            for (int k = 0; k < TR; k++)
#pragma unroll
                for (int m = 0; m < MT; m++) {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        tot[k][m][j] = first ? acc[k][m][j] : tot[k][m][j] + acc[k][m][j];
                    acc[k][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                }
            first = false;
            left = spl;
        }
    };
    ops O[2];
    wset W[NB];
    /* step c: limbs in bufs[I % NB], weights in W[I % NB], block 0's operands in O[I & 1]; during block
     * 0 block 1's are made, during block 1 the next pair's block 0's */
    auto step = [&](auto Ic, int c) __attribute__((always_inline)) {
        constexpr int I = decltype(Ic)::value, U = 2 * MT;
        constexpr int LP = (SI + TR + U - 3) / (U - 2); /* of the SI + TR groups of loads a unit */
        constexpr int EV = MT / (TR + 1) < 1 ? 1 : MT / (TR + 1);
        const int cn = c + NB - 1 < np ? c + NB - 1 : np - 1, c1 = c + 1 < np ? c + 1 : np - 1;
        ops O1;
        uint4 xa[2][3];
        f32x4 pv[2][TR];
        lread(xa[0], bufs[I % NB], 0, 0);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int h = u / MT, m = u % MT;
            if (u + 1 < U)
                lread(xa[(u + 1) & 1], bufs[I % NB], (u + 1) % MT, (u + 1) / MT);
#pragma unroll
            for (int k = u * LP; k < (u + 1) * LP; k++) {
                if (k < SI)
                    stage1(bufs[(I + NB - 1) % NB], cn, k);
                else if (k < SI + TR)
                    wload1(W[(I + NB - 1) % NB], cn, k - SI);
            }
            const ops &OC = h ? O1 : O[I & 1];
            f32x4(&r)[TR] = pv[u & 1];
            const f32x4(&q)[TR] = pv[(u + 1) & 1];
#pragma unroll
            for (int l = 0; l < 3; l++)
#pragma unroll
                for (int k = 0; k < TR; k++)
                    r[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xa[u & 1][l]), OC.wb[k],
                                                                   l ? r[k] : f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            if (u > 0) {
                const ops &OP = (u - 1) / MT ? O1 : O[I & 1];
#pragma unroll
                for (int k = 0; k < TR; k++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        acc[k][(u - 1) % MT][j] = __builtin_fmaf(q[k][j], OP.d[k], acc[k][(u - 1) % MT][j]);
            }
#pragma unroll
            for (int k = 0; k < TR; k++)
                if (m == (1 + k * EV < MT ? 1 + k * EV : MT - 1)) {
                    if (h == 0)
                        conv1(O1, W[I % NB], k, 1, c);
                    else
                        conv1(O[(I + 1) & 1], W[(I + 1) % NB], k, 0, c1);
                }
            /* the order within the unit: the limb reads, the loads, then two VALU between MFMAs */
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
#pragma unroll
            for (int i = 0; i < 3 * TR; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int k = 0; k < TR; k++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[k][MT - 1][j] = __builtin_fmaf(pv[1][k][j], O1.d[k], acc[k][MT - 1][j]);
        fold();
    };
    /* pairs 0 .. NB - 2 in flight, each its stage and then its weights, as the steps issue them */
    auto fetch = [&](uint4 *buf, wset &S, int c) __attribute__((always_inline)) {
        c = c < np ? c : np - 1;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < SI; k++)
            stage1(buf, c, k);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < TR; k++)
            wload1(S, c, k);
        __builtin_amdgcn_sched_barrier(0);
    };
    fetch(bufs[0], W[0], 0);
    fetch(bufs[1], W[1], 1);
    if constexpr (NB > 3)
        fetch(bufs[2], W[2], 2);
#pragma unroll
    for (int k = 0; k < TR; k++)
        conv1(O[0], W[0], k, 0, 0);
    constexpr int VN = (NB - 2) * (SI + 2 * TR) + 2 * TR;
    static_assert(VN < 64, "vmcnt");
#define STEP(I)                                                                                                        \
    {                                                                                                                  \
        __builtin_amdgcn_sched_barrier(0);                                                                             \
        __builtin_amdgcn_s_waitcnt(0x0f70 | (VN & 15) | (VN >> 4 << 14)); /* vmcnt(VN) */                              \
        __builtin_amdgcn_s_barrier();                                                                                  \
        __builtin_amdgcn_sched_barrier(0);                                                                             \
        step(tile_c<I>{}, c + (I));                                                                                    \
        if (c + (I) + 1 >= np)                                                                                         \
            break;                                                                                                     \
    }
    if constexpr (NB == 3)
        for (int c = 0;; c += 6) {
            STEP(0) STEP(1) STEP(2) STEP(3) STEP(4) STEP(5)
        }
    else
        for (int c = 0;; c += 4) {
            STEP(0) STEP(1) STEP(2) STEP(3)
        }
#undef STEP
    const bool tail = left != spl; /* the last split is shorter: its sums are still in acc */
    float *y = a.y[p];
    const long rows = 16L * rtn;
#pragma unroll
    for (int r = 0; r < RT; r++) {
        if (rt0 + r >= rtn)
            continue;
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float v[NP];
#pragma unroll
                for (int k = 0; k < NP; k++) {
                    const float s = acc[k * RT + r][m][j], b = tot[k * RT + r][m][j];
                    v[k] = !tail ? b : first ? s : b + s;
                }
                const long tok = 16L * (tt0 + m) + 4 * kq + j, i = tok * rows + (rt0 + r) * 16 + n;
                if (tok < a.t) {
                    const float o = NP == 2 ? q8_swiglu(v[0], v[NP - 1]) : v[0];
                    y[i] = NP == 1 && a.res ? a.res[i] + o : o;
                }
            }
    }
}

/* ---------------------------------------------------------------- launchers */

/* The instantiated tiles, as X(MT, RT, NW, NP, NB, least, us0, us1). For a product (NP 1) 256 rows x
 * 128 tokens, 256 x 64, 128 x 64, 64 x 64; for the fused pair 128 rows of both x 128 tokens, 128 x 64,
 * 64 x 64. The large tile does the most work a limb read and a converted weight; the small ones fill
 * the device where there are few tiles. A step (one pair of blocks) of a round of workgroups takes us0
 * + us1 f us, f the share of the compute units that hold one (the clock falls as they fill), and a
 * product at least `least` us a step. Measured, 1-6 rounds, f from 1/8 to 1, K = 2048 to 12288:
 * 256 x 128 2.04 at f <= 1/2, 2.63 at 3/4, 3.1 at 1; 256 x 64 1.25, 1.39, 1.67; 128 x 64 0.77, 0.86,
 * 0.98; 64 x 64 (two workgroups a unit) 0.67-0.74 up to 256 workgroups, 1.14 at 512, 1.75 at 768;
 * the pair 2.02, 2.42, 2.68; 1.47-1.58 at 3/4, 1.62 at 1; 1.7 at 384, 2.85 at 768, 5.45 at 1536. */
#define TILE_CFGS(X)                                                                                                   \
    X(8, 2, 8, 1, 3, 0.0, 1.70, 1.30)                                                                                  \
    X(4, 2, 8, 1, 4, 0.0, 1.10, 0.45)                                                                                  \
    X(4, 1, 8, 1, 4, 0.0, 0.70, 0.25)                                                                                  \
    X(4, 1, 4, 1, 3, 0.67, 0.57, 0.0)                                                                                  \
    X(8, 1, 8, 2, 3, 0.0, 1.75, 0.90)                                                                                  \
    X(4, 1, 8, 2, 4, 0.0, 1.30, 0.30)                                                                                  \
    X(4, 1, 4, 2, 3, 1.00, 0.93, 0.0)

struct tile_cfg {
    int mt, rt, nw, np, nb;
    float least, us0, us1;
};
#define CFG(M, R, N, P, B, L, U0, U1) {M, R, N, P, B, L##f, U0##f, U1##f},
static const tile_cfg TILES[] = {TILE_CFGS(CFG)};
#undef CFG

/* workgroup row tiles of a round's products under a configuration */
static long tile_rows(const tile_cfg &k, int n, const long *rows)
{
    long sum = 0;
    for (int i = 0; i < (k.np == 2 ? 1 : n); i++)
        sum += (rows[i] + 16L * k.nw * k.rt - 1) / (16L * k.nw * k.rt);
    return sum;
}

static int tile_cus()
{
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) {
            fprintf(stderr, "q8_tile: the device's compute units are not known\n");
            abort();
        }
    }
    return cus;
}

/* The configuration for n products (pair: the fused two) of t tokens with the least modelled time */
static const tile_cfg *tile_plan(int n, const long *rows, long cols, long t, bool pair, float *us)
{
    const tile_cfg *best = nullptr;
    for (const tile_cfg &k : TILES) {
        if (k.np != (pair ? 2 : 1))
            continue;
        const long groups = ((t + 15) / 16 + k.mt - 1) / k.mt, wgs = tile_rows(k, n, rows) * groups;
        const long rounds = (wgs + tile_cus() - 1) / tile_cus();
        const float step = (float)rounds * (k.us0 + k.us1 * (float)wgs / (float)(rounds * tile_cus()));
        const float cost = (float)((cols / Q8_BLOCK + 1) / 2) * (step > k.least ? step : k.least);
        if (!best || cost < *us) {
            best = &k;
            *us = cost;
        }
    }
    return best;
}

long q8_ximage_bytes(long t, long cols) { return (t + 15) / 16 * ((cols / Q8_BLOCK + 1) / 2) * 6144; }

bool q8_tile_takes(int n, const long *rows, long cols, long t, bool pair)
{
    /* a row of one block has no two scales to load at once */
    if (t <= 64 || cols < 2 * Q8_BLOCK || n < 1 || n > Q8_ROUND_MAX || (pair && (n != 2 || rows[0] != rows[1])))
        return false;
    /* Against the 64-token launches: measured 35, 34, 20, 21 and 14 us a launch at 12288 x 4096, 4096 x
     * 12288, 4096 x 4096, 2048 x 6144 and 2048 x 2048 (13 us and 0.44 a million weights;
     * less below 1024 rows, a few workgroups and their sums: 8 us); the image takes 3.5 us, and
     * 0.2 a MiB of it from there (10.5 us at 36 MiB). Few rows leave most of the device idle here,
     * where the 64-token launches split K over it: 4096 x 12288 at 128 tokens 66 against 117 us. */
    float us = 0.0f;
    if (!tile_plan(n, rows, cols, t, pair, &us))
        return false;
    float weights = 0.0f, all = 0.0f;
    for (int i = 0; i < n; i++) {
        weights += (float)rows[i] * (float)cols;
        all += (float)rows[i];
    }
    const float mib = (float)q8_ximage_bytes(t, cols) / 1048576.0f;
    return us + 3.5f + 0.2f * mib < (float)((t + 63) / 64) * (8.0f + (all < 1024.0f ? all / 1024.0f : 1.0f) * 5.0f + 0.44e-6f * weights);
}

void q8_launch_ximage(q8_stream_t stream, const float *x, long x_stride, long t, long cols, const float *nw, float eps, void *img)
{
    const int np = (int)((cols / Q8_BLOCK + 1) / 2);
    ximage_k<<<dim3((unsigned)((2 * np + XIMG_BLOCKS - 1) / XIMG_BLOCKS), (unsigned)((t + 15) / 16)), dim3(64 * XIMG_BLOCKS), 0, (hipStream_t)stream>>>(
        x, x_stride, t, cols, nw, eps, (uint4 *)img);
}

void q8_launch_tile(q8_stream_t stream, int n, const void *const *w, const long *rows, long cols, long t, const void *img, float *const *y, const float *res,
                    float *pair_y, q8_gemm_opts o)
{
    hipStream_t s = (hipStream_t)stream;
    float us = 0.0f;
    const tile_cfg *k = tile_plan(n, rows, cols, t, pair_y != nullptr, &us);
    tile_args a{};
    a.n = n;
    for (int i = 0; i < n; i++) {
        int ks, cps;
        q8_gemm_split(rows[i], cols, o, &ks, &cps);
        a.w[i] = (const uint8_t *)w[i];
        a.y[i] = pair_y ? pair_y : y[i];
        a.rtn[i] = (int)(rows[i] / 16);
        a.spl[i] = Q8_SPLIT_PAIRS * cps;
        a.start[i + 1] = a.start[i] + (int)tile_rows(*k, 1, rows + i);
    }
    a.res = res;
    a.img = img;
    a.img_bytes = (int)q8_ximage_bytes(t, cols);
    a.groups = (int)(((t + 15) / 16 + k->mt - 1) / k->mt);
    a.cols = cols;
    a.t = t;
    const long tiles = tile_rows(*k, n, rows);
    const unsigned grid = (unsigned)((tiles + 7) / 8 * 8 * a.groups);
    bool done = false;
#define GO(M, R, N, P, B, L, U0, U1)                                                                                          \
    if (!done && k->mt == M && k->rt == R && k->nw == N && k->np == P) {                                               \
        Q8_LAUNCH(q8_time_name("gemm_tile", 5, M, R, N, P, B), (gemm_tile<M, R, N, P, B>), dim3(grid), dim3(64 * N), s, a); \
        done = true;                                                                                                   \
    }
    TILE_CFGS(GO)
#undef GO
    if (!done) {
        fprintf(stderr, "q8_tile: no kernel for the plan\n");
        abort();
    }
}
