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
    /* this wave's block, loaded before the norm's sum so that the two memory round trips overlap
     * (traced at 64 tokens of 4096 columns on a norm 8.2 against 9.4 us) */
    const int b = (int)blockIdx.x * XIMG_BLOCKS + wave;
    const long tok = 16 * (long)blockIdx.y + (lane & 15);
    const bool in = tok < t && b < nb;
    const long k0 = (long)(b < nb ? b : nb - 1) * Q8_BLOCK + kcol(lane >> 4);
    const float *px = x + (tok < t ? tok : t - 1) * xs + k0;
    float4 a = *(const float4 *)px, c = *(const float4 *)(px + 4), g{}, e{};
    if (nw) {
        g = *(const float4 *)(nw + k0);
        e = *(const float4 *)(nw + k0 + 4);
        __builtin_amdgcn_sched_barrier(0);
        const long row = 16 * (long)blockIdx.y + wave;
        const float *xr = x + (row < t ? row : t - 1) * xs;
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
    if (b >= 2 * np)
        return;
    if (nw) {
        const float s = scale[lane & 15];
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

/* A barrier that no memory access moves across in the compiler, and that waits for none: the callers
 * say what has to be there (__syncthreads would also wait for the loads in flight) */
__device__ __forceinline__ void tile_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
}

/* A workgroup of NW waves, MT token tiles x NW * RT row tiles (of each of the NP = 2 matrices of the
 * pair), all of K in steps of one pair of blocks. KG == 2: two such sets of waves on the same tile, one
 * taking the even K splits and one the odd, each with its own stages; the second hands each split's
 * sums to the first through LDS, which adds them in split order.
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
 * slower (246 against 214 us), and 6 no faster (unequal SIMDs). */
template <int MT, int RT, int NW, int NP, int NB, int KG>
__global__ __launch_bounds__(64 * NW * KG) void gemm_tile(tile_args a)
{
    constexpr int TR = NP * RT;
    constexpr int WB = NB == 2 ? 3 : NB; /* weight sets: pair c's weights are issued in step c - WB + 1 */
    constexpr int SN = MT * 384;    /* 16-byte words of a stage */
    constexpr int SI = (MT * 6 + NW - 1) / NW; /* its 1 KiB loads a wave */
    static_assert(NB >= 2 && NB <= 4 && (KG == 1 || KG == 2), "the buffers and groups the steps are written for");
    /* separate arrays, so that the reads of one do not wait for the loads of another; each K group has
     * its half */
    __shared__ uint4 s0[KG * SN], s1[KG * SN], s2[NB > 2 ? KG * SN : 1], s3[NB > 3 ? KG * SN : 1];
    __shared__ f32x4 ex[KG > 1 ? TR * MT * NW * 64 : 1]; /* group 1's split on its way to group 0 */
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int kg = KG > 1 ? wid / NW : 0, wave = KG > 1 ? wid % NW : wid;
    uint4 *bufs[NB];
    bufs[0] = s0 + kg * SN;
    bufs[1] = s1 + kg * SN;
    if constexpr (NB > 2)
        bufs[2] = s2 + kg * SN;
    if constexpr (NB > 3)
        bufs[3] = s3 + kg * SN;
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
    const unsigned istep = (unsigned)ttn * 6144, ioff = (unsigned)tt0 * 6144;
    /* load i of the wave's share of pair c's stage. Token tiles past the last one read the next pair's
     * tiles, or zeros past the image's end: tokens that are not stored, and no token's sums see another's */
    auto stage1 = [&](uint4 *buf, int c, int i) __attribute__((always_inline)) {
        int u = wave * SI + i; /* where the stage does not divide, the last loads repeat its last KiB */
        if constexpr (MT * 6 % NW != 0)
            u = u < MT * 6 ? u : MT * 6 - 1;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(irs, (tile_lds *)(buf + u * 64), 16, lane * 16, (int)((unsigned)c * istep + ioff + u * 1024), 0, 0);
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
    /* block h of pair c as MFMA operands, in pieces of a few VALU instructions that spread over the
     * units (all of a row tile's at once kept both waves of a SIMD on the VALU at the same time):
     * piece 0 the row's scale, and for block 0 the pair's halves traded in place, lanes 0-31 hold block
     * 2c and 32-63 block 2c + 1 (q8_bf16.h); pieces 1 to 4 two values a lane each. The block past
     * an odd count needs no mask: its limbs are zero and its weights finite, and its scale becomes 0
     * (the row's last scale is the high half of that load) */
    struct ops {
        uint32_t wb[TR][4];
        float d[TR];
    };
    constexpr int CP = 5;
    const int odd = nb & 1;
    auto conv1 = [&](ops &O, wset &S, int k, int h, int c, int piece) __attribute__((always_inline)) {
        if (piece == 0) {
            if (h == 0) {
                const auto s02 = __builtin_amdgcn_permlane32_swap(S.q[k].x, S.q[k].z, false, false);
                const auto s13 = __builtin_amdgcn_permlane32_swap(S.q[k].y, S.q[k].w, false, false);
                S.q[k] = make_uint4(s02[0], s13[0], s02[1], s13[1]);
            }
            const uint32_t dd = S.d[k] >> (odd && c == np - 1 ? 16 : 0);
            float d = q8_half((uint16_t)(h ? dd >> 16 : dd));
            asm("" : "+v"(d)); /* converted once here, not in each of its FMAs */
            O.d[k] = d;
        } else {
            const int i = piece - 1;
            const uint32_t v = h ? (i < 2 ? S.q[k].z : S.q[k].w) : (i < 2 ? S.q[k].x : S.q[k].y);
            O.wb[k][i] = pack_hi((float)(int8_t)(v >> (16 * (i & 1))), (float)(int8_t)(v >> (16 * (i & 1) + 8)));
        }
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
    /* Steps: KG == 1, the pairs in order; KG == 2, group g's splits g, g + 2, ... in order, both groups in
     * step, so a step is at pair c of the group, r pairs into its split. pos[k]: where step + k is */
    struct place {
        int c, r;
    };
    auto next = [&](place q) __attribute__((always_inline)) {
        const bool end = q.r + 1 == spl;
        return place{q.c + 1 + (KG > 1 && end ? spl : 0), end ? 0 : q.r + 1};
    };
    place pos[4];
    pos[0] = place{kg * spl, 0};
#pragma unroll
    for (int k = 1; k < 4; k++)
        pos[k] = next(pos[k - 1]);
    const int splits = (np + spl - 1) / spl;
    const int steps = KG == 1 ? np : splits % 2 ? splits / 2 * spl + np - (splits - 1) * spl : splits / 2 * spl;
    auto clamp = [&](int c) __attribute__((always_inline)) { return c < np ? c : np - 1; };
    bool first = true, pend = false; /* pend: group 1 has put a split into ex */
    auto put_ex = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < TR; k++)
#pragma unroll
            for (int m = 0; m < MT; m++)
                ex[((k * MT + m) * NW + wave) * 64 + lane] = acc[k][m];
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xc07f); /* lgkmcnt(0): in LDS before the next barrier */
    };
    auto add_ex = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < TR; k++)
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const f32x4 v = ex[((k * MT + m) * NW + wave) * 64 + lane];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    tot[k][m][j] += v[j];
            }
    };
    /* the end of a split: its sums join the splits' before it. Group 1's go through ex, which group 0
     * reads in the next step (two steps at least before the next write: a split has two pairs or more) */
    auto fold = [&]() __attribute__((always_inline)) {
        if (pos[0].r + 1 == spl) {
            if (KG > 1 && kg) {
                put_ex();
            } else {
#pragma unroll
                for (int k = 0; k < TR; k++)
#pragma unroll
                    for (int m = 0; m < MT; m++)
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            tot[k][m][j] = first ? acc[k][m][j] : tot[k][m][j] + acc[k][m][j];
                first = false;
                pend = KG > 1 && pos[0].c + spl < np; /* group 1 ends a whole split in this step too */
            }
#pragma unroll
            for (int k = 0; k < TR; k++)
#pragma unroll
                for (int m = 0; m < MT; m++)
                    acc[k][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    };
    ops O[2];
    wset W[WB];
    /* a step: limbs in bufs[I % NB], weights in W[I % WB], block 0's operands in O[I & 1]; during block
     * 0 block 1's are made, during block 1 the next pair's block 0's */
    auto step = [&](auto Ic) __attribute__((always_inline)) {
        constexpr int I = decltype(Ic)::value, U = 2 * MT;
        constexpr int LP = (SI + TR + U - 3) / (U - 2); /* of the SI + TR groups of loads a unit */
        constexpr int LW = (SI + LP - 1) / LP;          /* the first unit that loads weights */
        static_assert(LW + (TR + LP - 1) / LP <= U, "every load of a step is issued in one of its units");
        constexpr int PU = (CP * TR + MT - 1) / MT;                  /* conversion pieces a unit */
        constexpr int VU = (4 * TR + 3 * PU + 3 * TR - 1) / (3 * TR); /* VALU instructions an MFMA */
        const int c = pos[0].c, c1 = clamp(pos[1].c), cn = clamp(pos[NB - 1].c), cw = clamp(pos[WB - 1].c);
        ops O1;
        uint4 xa[2][3];
        f32x4 pv[2][TR];
        lread(xa[0], bufs[I % NB], 0, 0);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int h = u / MT, m = u % MT;
            if (u + 1 < U)
                lread(xa[(u + 1) & 1], bufs[I % NB], (u + 1) % MT, (u + 1) / MT);
            /* in units apart, as no unit's loads move into another (the sched_barrier at its end): the
             * VN of the next wait counts weights after the last load of the stage */
            if (u < LW) {
#pragma unroll
                for (int k = u * LP; k < (u + 1) * LP && k < SI; k++)
                    stage1(bufs[(I + NB - 1) % NB], cn, k);
            } else {
#pragma unroll
                for (int k = (u - LW) * LP; k < (u - LW + 1) * LP && k < TR; k++)
                    wload1(W[(I + WB - 1) % WB], cw, k);
            }
            const ops &OC = h ? O1 : O[I & 1];
            f32x4(&r)[TR] = pv[u & 1];
            const f32x4(&q)[TR] = pv[(u + 1) & 1];
#pragma unroll
            for (int l = 0; l < 3; l++)
#pragma unroll
                for (int k = 0; k < TR; k++)
                    r[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xa[u & 1][l]), __builtin_bit_cast(bf16x8, OC.wb[k]),
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
            for (int k = m * PU; k < (m + 1) * PU && k < CP * TR; k++) {
                if (h == 0)
                    conv1(O1, W[I % WB], k / CP, 1, c, k % CP);
                else
                    conv1(O[(I + 1) & 1], W[(I + 1) % WB], k / CP, 0, c1, k % CP);
            }
            /* the order within the unit: the limb reads, the loads, then the VALU work between MFMAs */
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
#pragma unroll
            for (int i = 0; i < 3 * TR; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, VU, 0);
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
    /* the stages of the first NB - 1 pairs and the weights of WB - 1 in flight, each pair's stage and then
     * its weights, as the steps issue them (NB == 2: a pair's weights come a step before its stage) */
    auto fetch = [&](int k) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        if (k < NB - 1)
#pragma unroll
            for (int i = 0; i < SI; i++)
                stage1(bufs[k], clamp(pos[k].c), i);
        __builtin_amdgcn_sched_barrier(0);
        const int q = NB == 2 ? k + 1 : k;
#pragma unroll
        for (int i = 0; i < TR; i++)
            wload1(W[q], clamp(pos[q].c), i);
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (NB == 2)
#pragma unroll
        for (int i = 0; i < TR; i++)
            wload1(W[0], clamp(pos[0].c), i);
#pragma unroll
    for (int k = 0; k < NB - 1; k++)
        fetch(k);
#pragma unroll
    for (int k = 0; k < CP * TR; k++)
        conv1(O[0], W[0], k / CP, 0, clamp(pos[0].c), k % CP);
    constexpr int VN = (NB - 2) * (SI + 2 * TR) + 2 * TR;
    static_assert(VN < 64, "vmcnt");
    int done = 0;
#define STEP(I)                                                                                                        \
    {                                                                                                                  \
        __builtin_amdgcn_sched_barrier(0);                                                                             \
        __builtin_amdgcn_s_waitcnt(0x0f70 | (VN & 15) | (VN >> 4 << 14)); /* vmcnt(VN) */                              \
        tile_barrier();                                                                                                \
        if (KG > 1 && pend) {                                                                                          \
            add_ex();                                                                                                  \
            pend = false;                                                                                              \
        }                                                                                                              \
        if (KG == 1 || pos[0].c < np) /* group 1's last split may be shorter, or missing */                            \
            step(tile_c<I>{});                                                                                         \
        pos[0] = pos[1];                                                                                               \
        pos[1] = pos[2];                                                                                               \
        pos[2] = pos[3];                                                                                               \
        pos[3] = next(pos[3]);                                                                                         \
        if (++done >= steps)                                                                                           \
            break;                                                                                                     \
    }
    if constexpr (NB < 4)
        for (;;) {
            STEP(0) STEP(1) STEP(2) STEP(3) STEP(4) STEP(5)
        }
    else
        for (;;) {
            STEP(0) STEP(1) STEP(2) STEP(3)
        }
#undef STEP
    if constexpr (KG > 1) {
        /* the last of group 1's splits: in ex since the last step, or, shorter than the others, still in
         * its acc */
        const bool rest = splits % 2 == 0 && np % spl != 0;
        tile_barrier();
        if (rest && kg)
            put_ex();
        tile_barrier();
        if (kg)
            return;
        if (pend || rest)
            add_ex();
    }
    const bool tail = steps % spl != 0; /* the last split is shorter: its sums are still in acc */
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

/* The instantiated tiles, as X(MT, RT, NW, NP, NB, KG, ur, us, us2, uf, uh). For a product (NP 1) 256 rows x
 * 128 tokens, 256 x 64, 128 x 64, 64 x 64, 64 x 48 and 64 x 32; for the fused pair 128 rows of both x 128
 * tokens, 128 x 64, 64 x 64 and 64 x 32. The large tile does the most work a limb read and a converted
 * weight; the small ones fill the device where there are few tiles, with two K groups, so that a compute
 * unit still holds 8 (for 64 x 64 4) waves of two row tiles each: one row tile a wave reads 1 KiB of limbs
 * an MFMA, all that LDS gives. 4096 x 12288 at 512 tokens 157 us against 170 for 128 x 64 with one row tile
 * on 8 waves and no K groups; 2048 x 6144 at 203 tokens 55 us against 68 for 64 x 64.
 *
 * The costs, in us: a round of workgroups ur, and a step (one pair of blocks; of both groups' one each) us
 * + uf f, f the workgroups a compute unit of the fullest XCD (the clock falls as they fill). One workgroup
 * a unit, but where us2 is given, two of which take us2 a step. Token groups share a row tile's weights
 * in their XCD's L2, and one group alone loads them from HBM: with g groups all of it times 1 + uh f / g^2
 * (f up to 1; with us2 from 1/2 to 2, as f - 1/2). Fitted to 14488 random calls of 5 to 700
 * tokens, 64 to 24576 rows and 64 to 14336 columns, each timed on most of its configurations: 80 % of the
 * times within 7 % (64 x 32: 10 %). */
#define TILE_CFGS(X)                                                                                                   \
    X(8, 2, 8, 1, 3, 1, 3.48, 1.92, 0, 0.16, 0.12)                                                                           \
    X(4, 2, 8, 1, 4, 1, 2.07, 1.22, 0, 0.09, 0.16)                                                                           \
    X(4, 2, 4, 1, 2, 2, 1.39, 1.42, 0, 0.04, 0.18)                                                                           \
    X(4, 2, 2, 1, 2, 2, 2.00, 1.05, 0, 0.03, 0.08)                                                                           \
    X(3, 2, 2, 1, 2, 2, 1.54, 0.91, 0, 0.03, 0.10)                                                                           \
    X(2, 2, 2, 1, 2, 2, 0.59, 0.78, 1.15, 0.03, 0.40)                                                                        \
    X(8, 1, 8, 2, 3, 1, 3.02, 1.87, 0, 0.29, 0.00)                                                                           \
    X(4, 1, 8, 2, 4, 1, 1.96, 1.18, 0, 0.19, 0.16)                                                                           \
    X(4, 1, 4, 2, 2, 2, 1.04, 1.42, 0, 0.08, 0.15)                                                                           \
    X(2, 1, 4, 2, 2, 2, 0.11, 1.09, 1.91, 0.07, 0.40)

struct tile_cfg {
    int mt, rt, nw, np, nb, kg;
    float ur, us, us2, uf, uh;
};
#define CFG(M, R, N, P, B, G, UR, US, US2, UF, UH) {M, R, N, P, B, G, (float)UR, (float)US, (float)US2, (float)UF, (float)UH},
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
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 8) {
            fprintf(stderr, "q8_tile: the device's compute units are not known\n");
            abort();
        }
        return n;
    }();
    return cus;
}

/* The configuration for n products (pair: the fused two) of t tokens with the least modelled time */
static const tile_cfg *tile_plan(int n, const long *rows, long cols, long t, bool pair, q8_gemm_opts o, float *us)
{
    const tile_cfg *best = nullptr;
    const long pairs = (cols / Q8_BLOCK + 1) / 2;
    long half = 0; /* steps with two K groups: the most of any product */
    for (int i = 0; i < n; i++) {
        int ks, cps;
        q8_gemm_split(rows[i], cols, o, &ks, &cps);
        const long spl = (long)Q8_SPLIT_PAIRS * cps, splits = (pairs + spl - 1) / spl;
        const long k = splits % 2 ? splits / 2 * spl + pairs - (splits - 1) * spl : splits / 2 * spl;
        half = k > half ? k : half;
    }
    for (const tile_cfg &k : TILES) {
        if (k.np != (pair ? 2 : 1))
            continue;
        /* the kernel gives an XCD every eighth row tile with all its token groups: the fullest one sets the
         * rounds. 5232 x 4352 at 148 tokens on 82 row tiles of 3 groups puts 33 workgroups on 32 units,
         * 87 us where 64 x 32 tiles take 49 */
        const long groups = ((t + 15) / 16 + k.mt - 1) / k.mt, per = (tile_rows(k, n, rows) + 7) / 8 * groups, units = tile_cus() / 8;
        const long rounds = (per + units - 1) / units;
        const float f = (float)per / (float)units;
        const float step = (k.us2 > 0.0f ? (float)(rounds % 2) * k.us + (float)(rounds / 2) * k.us2 : (float)rounds * k.us) + k.uf * f;
        const float fill = k.us2 > 0.0f ? (f < 0.5f ? 0.0f : f < 2.0f ? f - 0.5f : 1.5f) : f < 1.0f ? f : 1.0f;
        const float cost = ((float)rounds * k.ur + (float)(k.kg == 2 ? half : pairs) * step) * (1.0f + k.uh * fill / (float)(groups * groups));
        if (!best || cost < *us) {
            best = &k;
            *us = cost;
        }
    }
    return best;
}

long q8_ximage_bytes(long t, long cols) { return (t + 15) / 16 * ((cols / Q8_BLOCK + 1) / 2) * 6144; }

bool q8_tile_takes(int n, const long *rows, long cols, long t, bool pair, bool norm, q8_gemm_opts o)
{
    /* up to 64 tokens only rounds on a norm, from three token tiles: the image takes the norm's launch in, and
     * a round's many small splits leave the most partials to sum (the 9B DeltaNet quartet at 64
     * tokens: norm, product and sums 59 us, image and tiles 42). Single products and the pair gain
     * nothing (12288 x 4096 at 64 tokens 42 + 3.5 against 35, the pair 61 + 3.5 against 63) */
    if ((t <= 64 && (t <= 32 || n < 2 || pair || !norm)) || n < 1 || n > Q8_ROUND_MAX || (pair && (n != 2 || rows[0] != rows[1])))
        return false;
    /* a row of one block has no two scales to load at once */
    if (cols < 2 * Q8_BLOCK)
        return false;
    float us = 0.0f;
    if (!tile_plan(n, rows, cols, t, pair, o, &us))
        return false;
    /* and the image's launch, its bytes, the norm in it and the stores, as fitted with TILE_CFGS, against the
     * 64-token launches (q8_gemm_us). Above 64 tokens 8 % ahead, for the error of the two: of 8311 random
     * calls there 8 took more than 1.03 of the launches' time (few rows leave most of the device idle
     * here, where the launches split K over it: 1024 x 3072 at 91 tokens 28 against 22.6 us; below 512 rows
     * 20 %, 256 x 1504 at 94 tokens 17.2 against 15.7 and priced 9 % below). Up to 64
     * tokens the streams' errors weigh more, large matrices' above all (13568 + 1696 + 32 rows of 3136
     * columns at 53 tokens 54.5 against 50.9 us, priced 5 % below): 20 % ahead above 36 million weights and
     * 3 % below, and no lead where 40 % of the launches' time is their partials and sums, which the tiles
     * do without (the 9B DeltaNet quartet at 64 tokens 55.9 against 58.9 us) */
    long outs = 0;
    for (int i = 0; i < (pair ? 1 : n); i++)
        outs += rows[i] * t;
    us += 5.25f + 0.656f * (float)q8_ximage_bytes(t, cols) / 1048576.0f + 1.1e-6f * (float)outs;
    if (norm)
        us += 1.44f + 0.00081f * (float)cols;
    float sums = 0.0f, weights = 0.0f;
    for (int i = 0; i < n; i++)
        weights += (float)rows[i] * (float)cols;
    const float launches = q8_gemm_us(n, rows, cols, t, norm, o, &sums);
    const float lead = t > 64 ? (weights < 512.0f * (float)cols ? 1.2f : 1.08f) : sums >= 0.4f * launches ? 1.0f : weights > 36e6f ? 1.2f : 1.03f;
    return lead * us < launches;
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
    const tile_cfg *k = tile_plan(n, rows, cols, t, pair_y != nullptr, o, &us);
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
#define GO(M, R, N, P, B, G, UR, US, US2, UF, UH)                                                                              \
    if (!done && k->mt == M && k->rt == R && k->nw == N && k->np == P && k->kg == G) {                                 \
        Q8_LAUNCH(q8_time_name("gemm_tile", 6, M, R, N, P, B, G), (gemm_tile<M, R, N, P, B, G>), dim3(grid), dim3(64 * N * G), s, a); \
        done = true;                                                                                                   \
    }
    TILE_CFGS(GO)
#undef GO
    if (!done) {
        fprintf(stderr, "q8_tile: no kernel for the plan\n");
        abort();
    }
}
