/* q8_gemv.h: the body of the decode kernels (q8_kernels.hip, q8_gemv_any.hip). */
#ifndef Q8_GEMV_H
#define Q8_GEMV_H

#include <hip/hip_runtime.h>

#include "q8_device.h"

/* the least power of two >= n, 1 <= n <= 64 (q8_pow2ceil at run time) */
__host__ __device__ inline int q8_pow2_from(int n)
{
    int p = 1;
    while (p < n)
        p *= 2;
    return p;
}

/* The waves of a decode workgroup for any cols: one a started 1024 columns. One a whole 1024, with the
 * tail's units given to the threads once more, only where that is a whole number of waves a SIMD (4, 8,
 * 12) and the threads hold the tail for 16 rows and matrices (every shape of it: the rule must not
 * depend on rows, tokens or the pair, so that a product has the same bits in all of them). There one
 * wave more loads the SIMDs unevenly and takes the instance of the next 4 waves: the pair 12288 x 4128
 * at 3 tokens 1.55 times, the product 12288 x 8224 1.16 times the tail's time. Everywhere else the
 * wave is the faster by 5 to 35 %, as it adds no second pass over x: the pair 12288 x 5280 at 3 tokens
 * 65 us with the tail, 51 with the wave. */
__host__ __device__ inline int q8_any_waves(long cols)
{
    const int whole = (int)(cols / 1024), tail = (int)(cols % 1024 / 16);
    if (tail == 0)
        return whole;
    return whole > 0 && whole % 4 == 0 && q8_pow2_from(tail) <= 4 * whole ? whole : whole + 1;
}

/* The most rows (a round's together, both matrices' of the pair) at which the decode kernels of 5 to 8
 * waves take an epilogue in at mt tokens. Each workgroup does the norm's arithmetic again, and at 4
 * tokens an epilogue takes them past 128 registers, which leaves one workgroup a compute unit where
 * there were two; apart it costs a launch, whatever the rows. Apart against fused, us: the norm on
 * 8192 columns at 4 tokens at 4096, 8192 and 20480 rows 15.0 / 14.0, 24.0 / 25.8 and 49.8 / 60.7, at
 * 3 tokens 42.9 / 45.8 at 20480; a round on the norm of 25632 rows at 2 tokens 50.1 / 53.5; the pair on 8192 columns (pair8k: 8 waves of whole 1024s) at 4 tokens
 * 42.4 / 43.2 at 2 x 8192 rows, 92 / 101 at 2 x 20480; the residual on 5120 columns at 4 tokens 0.97
 * and 0.84 of fused at 4096 and 20480 rows. */
inline long q8_epi_rows(int mt, bool pair8k) { return mt == 1 ? 1L << 40 : mt <= 3 || pair8k ? 16384 : 4096; }

/* The decode kernel for cols % 1024 == 0: a workgroup of NW waves owns RW rows and all of K;
 * wave w takes the K-slice [w*1024*S, (w+1)*1024*S), S steps of 64 16-column units (lane l:
 * units l + 64 s). Every load of a lane is issued before any arithmetic, x first and then the
 * weights row by row (loads retire in order, so row r's arithmetic waits for rows 0..r only), so
 * the whole matrix is in flight in the first round trip: the layer matrices are latency-bound
 * otherwise. Per unit: 16 exact int8->f32 converts shared by the MT tokens, a 16-step fma chain
 * per token, then acc = fma(s, d, acc) with the unit's block scale. The lanes' partials are summed
 * by q8_wave_sum_dpp, the NW waves' in LDS in wave order: the same order every run. */
/* EPI: 0 none; 1 the RMS norm of x first (e.nw, e.eps); 2 y = e.res + the product (q8_epi). y and
 * e.res may be the same array: each element is read and then written by the one thread that owns it. */
/* ANY: cols any multiple of 32, S = 1, the waves the launch gave (at most NW; q8_any_waves). With a
 * wave a started 1024 columns, a lane past the row's last unit loads unit 0 and counts as zero, x (after
 * its product with the norm's weight: 0 times an infinite weight would be NaN) and scale (0 times an
 * infinite scale would be, too). With a wave a whole 1024 columns, the
 * tail's units go to the workgroup's threads once more, a row and a unit each (every row and matrix
 * has TP neighbouring lanes, TP the power of two from its units up), and are added after the waves'
 * sums: 129 blocks would otherwise take a fifth wave for two units. */
template <int MT, int RW, int S, int NW, int PAIR, int EPI, int ANY = 0>
__device__ __forceinline__ void gemv_body(const uint8_t *__restrict__ w0, const uint8_t *__restrict__ w1, long rows, long cols, const float *__restrict__ x,
                                          long x_stride, float *y, long r0, q8_epi e)
{
    constexpr int P = PAIR + 1;
    static_assert(!ANY || S == 1, "one unit a lane");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nw = ANY ? (int)(blockDim.x >> 6) : NW; /* waves of the workgroup */
    const int units = ANY ? (int)(cols / 16) : 0, tail = ANY ? units - 64 * nw : 0; /* > 0: the tail's units */
    const bool live = !ANY || (int)threadIdx.x < units;
    const long u0 = live ? (long)wave * 64 * S + lane : 0;

    float4 xv[MT][S][4];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int s = 0; s < S; s++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                xv[m][s][c] = *(const float4 *)(x + m * x_stride + 16 * (u0 + 64 * s) + 4 * c);
    /* the residual of the output this thread stores (thread k < RW*MT stores row k / MT, token
     * k % MT; the others load one of those too, so the load is unconditional), issued with x so
     * that it is not a memory latency at the kernel's end */
    float rv = 0.0f;
    if constexpr (EPI == 2) {
        static_assert(64 * (ANY ? 1 : NW) >= RW * MT, "the residual epilogue stores from threads < RW * MT");
        const int k = (int)threadIdx.x % (RW * MT);
        rv = e.res[(long)(k % MT) * rows + r0 + k / MT];
    }
    /* the norm's weights, the lane's columns, issued with x before the matrix */
    float4 nv[S][4];
    if constexpr (EPI == 1) {
#pragma unroll
        for (int s = 0; s < S; s++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                nv[s][c] = *(const float4 *)(e.nw + 16 * (u0 + 64 * s) + 4 * c);
        /* keep them there: left to itself the scheduler issues them after the matrix, and the
         * products of x and the norm weights, which every fma needs, then wait for all of it */
        __builtin_amdgcn_sched_barrier(0);
    }
    uint4 q[RW][P][S];
    uint16_t dh[RW][P][S];
#pragma unroll
    for (int r = 0; r < RW; r++)
#pragma unroll
        for (int p = 0; p < P; p++) {
            const uint8_t *w = p ? w1 : w0;
            const uint8_t *wq = w + q8s_row_q(r0 + r, cols);
            const uint16_t *wd = (const uint16_t *)(w + q8s_row_d(r0 + r, cols));
#pragma unroll
            for (int s = 0; s < S; s++) {
                q[r][p][s] = *(const uint4 *)(wq + 16 * (u0 + 64 * s));
                dh[r][p][s] = wd[(u0 + 64 * s) >> 1];
            }
        }
    /* every load issued before any arithmetic: left to itself the scheduler sinks the last rows'
     * loads past the first rows' arithmetic, and past the wait for x, so they start a memory round
     * trip late (4096x12288 at one token 10.85 against 11.0 us, at three 13.3 against 13.5). Not
     * for 16 rows at two tokens, where the scheduler's own order measured faster (4096x12288: 11.4
     * against 11.6 us) */
    if constexpr (!(MT == 2 && RW == 16))
        __builtin_amdgcn_sched_barrier(0);
    /* the tail's unit of this thread: row tr, matrix tm, unit 64 nw + tj; loaded with the rest */
    const int tp = ANY && tail > 0 ? q8_pow2_from(tail) : 1;
    const int tk = (int)threadIdx.x / tp, tj = (int)threadIdx.x % tp;
    const bool tlive = ANY && tail > 0 && tk < RW * P && tj < tail;
    const int tr = tlive ? tk / P : 0, tu = tlive ? 64 * nw + tj : 0;
    uint4 tq;
    uint16_t td;
    if constexpr (ANY) {
        if (tail > 0) {
            const uint8_t *w = PAIR && tlive && tk % P ? w1 : w0;
            tq = *(const uint4 *)(w + q8s_row_q(r0 + tr, cols) + 16 * tu);
            td = ((const uint16_t *)(w + q8s_row_d(r0 + tr, cols)))[tu >> 1];
        }
    }
    auto live4 = [&](float4 v) { return make_float4(live ? v.x : 0.0f, live ? v.y : 0.0f, live ? v.z : 0.0f, live ? v.w : 0.0f); };
    if constexpr (ANY && EPI != 1) {
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                xv[m][0][c] = live4(xv[m][0][c]);
    }

    /* the norm: x <- nw * x at once, and per token the sum of x^2 (the lane's, then the wave's,
     * left in LDS for the final reduction, whose barrier covers it); s = 1 / sqrt(eps + sum / cols)
     * multiplies the outputs at the end, W (nw * x) s = W (nw * (x s)): no barrier before the
     * arithmetic starts, and x and nw are dead once multiplied */
    float ss[MT];
    if constexpr (EPI == 1) {
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float a = 0.0f;
#pragma unroll
            for (int s = 0; s < S; s++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const float4 v = xv[m][s][c], g = nv[s][c];
                    a = __builtin_fmaf(v.x, v.x, a);
                    a = __builtin_fmaf(v.y, v.y, a);
                    a = __builtin_fmaf(v.z, v.z, a);
                    a = __builtin_fmaf(v.w, v.w, a);
                    xv[m][s][c] = live4(make_float4(g.x * v.x, g.y * v.y, g.z * v.z, g.w * v.w));
                }
            ss[m] = q8_wave_sum_dpp(live ? a : 0.0f);
        }
    }
    /* the wave's RW*P*MT sums over its lanes (q8_wave_sums, padded to a power of two), each
     * written to LDS once; then the NW waves' in wave order. CH: in chunks of up to 8 rows, each
     * chunk's sums run while later rows' loads still arrive. The two forms give the same bits; the
     * compiler allocates their registers differently, and each was measured where it is used:
     * chunks for the pair at 2 tokens (20.0 against 21.2 us on 12288x4096) and for 16 rows at 3
     * tokens (119 registers, where one block of sums spills: 13.7 against 14.4 us at 8 rows on
     * 4096x12288); one block everywhere else (the pair at 1 token 18.0 against 18.5 us, 16 rows at
     * 2 and 4 tokens 11.7 / 14.5 against 12.5 / 15.6). */
    constexpr bool CH = (PAIR && MT == 2) || (MT == 3 && RW == 16);
    constexpr int RC = CH && RW > 8 ? 8 : RW, VC = RC * P * MT, VP = q8_pow2ceil(VC);
    __shared__ float red[NW][RW * P * MT];
    __shared__ float nsum[EPI == 1 ? NW : 1][MT];
    if constexpr (EPI == 1) {
        if (lane == 0)
#pragma unroll
            for (int m = 0; m < MT; m++)
                nsum[wave][m] = ss[m];
    }
    /* row r's sum of token m of matrix p over the lane's columns */
    auto row_sum = [&](int r, int p, int m) {
        float acc = 0.0f;
#pragma unroll
        for (int s = 0; s < S; s++) {
            const uint32_t qw[4] = {q[r][p][s].x, q[r][p][s].y, q[r][p][s].z, q[r][p][s].w};
            const float xs[16] = {xv[m][s][0].x, xv[m][s][0].y, xv[m][s][0].z, xv[m][s][0].w, xv[m][s][1].x, xv[m][s][1].y,
                                  xv[m][s][1].z, xv[m][s][1].w, xv[m][s][2].x, xv[m][s][2].y, xv[m][s][2].z, xv[m][s][2].w,
                                  xv[m][s][3].x, xv[m][s][3].y, xv[m][s][3].z, xv[m][s][3].w};
            float sum = 0.0f;
#pragma unroll
            for (int j = 0; j < 16; j++)
                sum = __builtin_fmaf(q8_s8(qw[j >> 2], j & 3), xs[j], sum);
            acc = __builtin_fmaf(sum, q8_half(live ? dh[r][p][s] : (uint16_t)0), acc);
        }
        return acc;
    };
    /* a block of VC sums (rows [ch*RC, +RC)) over the lanes, into LDS */
    auto lane_sums = [&](float (&vals)[VP], int ch) {
#pragma unroll
        for (int i = VC; i < VP; i++)
            vals[i] = 0.0f;
        q8_wave_sums<VP>(vals, lane);
        if (q8_wave_sums_owner<VP>(lane)) {
#pragma unroll
            for (int k = 0; k < (VP >> q8_wave_sums_steps<VP>()); k++) {
                const int g = q8_wave_sums_index<VP>(lane, k);
                if (g < VC)
                    red[wave][ch * VC + g] = vals[k];
            }
        }
    };
    if constexpr (CH) {
#pragma unroll
        for (int ch = 0; ch < RW / RC; ch++) {
            float vals[VP];
#pragma unroll
            for (int rr = 0; rr < RC; rr++)
#pragma unroll
                for (int p = 0; p < P; p++)
#pragma unroll
                    for (int m = 0; m < MT; m++)
                        vals[(rr * P + p) * MT + m] = row_sum(ch * RC + rr, p, m);
            lane_sums(vals, ch);
        }
    } else {
        float acc[RW][P][MT];
#pragma unroll
        for (int r = 0; r < RW; r++)
#pragma unroll
            for (int p = 0; p < P; p++)
#pragma unroll
                for (int m = 0; m < MT; m++)
                    acc[r][p][m] = row_sum(r, p, m);
        float vals[VP];
#pragma unroll
        for (int r = 0; r < RW; r++)
#pragma unroll
            for (int p = 0; p < P; p++)
#pragma unroll
                for (int m = 0; m < MT; m++)
                    vals[(r * P + p) * MT + m] = acc[r][p][m];
        lane_sums(vals, 0);
    }
    __shared__ float tred[ANY ? RW * P * MT : 1];
    __shared__ float tsum[ANY && EPI == 1 ? MT : 1];
    if constexpr (ANY) {
        if (tail > 0) {
            const uint32_t qw[4] = {tq.x, tq.y, tq.z, tq.w};
            const float d = q8_half(tlive ? td : (uint16_t)0);
#pragma unroll
            for (int m = 0; m < MT; m++) {
                float sum = 0.0f, sq = 0.0f;
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    float4 v = *(const float4 *)(x + m * x_stride + 16 * tu + 4 * c);
                    if constexpr (EPI == 1) {
                        const float4 g = *(const float4 *)(e.nw + 16 * tu + 4 * c);
                        sq = __builtin_fmaf(v.x, v.x, sq);
                        sq = __builtin_fmaf(v.y, v.y, sq);
                        sq = __builtin_fmaf(v.z, v.z, sq);
                        sq = __builtin_fmaf(v.w, v.w, sq);
                        v = make_float4(g.x * v.x, g.y * v.y, g.z * v.z, g.w * v.w);
                    }
                    v = make_float4(tlive ? v.x : 0.0f, tlive ? v.y : 0.0f, tlive ? v.z : 0.0f, tlive ? v.w : 0.0f);
                    sum = __builtin_fmaf(q8_s8(qw[c], 0), v.x, sum);
                    sum = __builtin_fmaf(q8_s8(qw[c], 1), v.y, sum);
                    sum = __builtin_fmaf(q8_s8(qw[c], 2), v.z, sum);
                    sum = __builtin_fmaf(q8_s8(qw[c], 3), v.w, sum);
                }
                float acc = sum * d;
                if constexpr (EPI == 1)
                    sq = tlive ? sq : 0.0f;
                for (int off = tp >> 1; off >= 1; off >>= 1) {
                    acc += __shfl_xor(acc, off, 64);
                    if constexpr (EPI == 1)
                        sq += __shfl_xor(sq, off, 64);
                }
                if (tj == 0 && tk < RW * P)
                    tred[tk * MT + m] = acc;
                if constexpr (EPI == 1)
                    if (threadIdx.x == 0)
                        tsum[m] = sq;
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < RW * MT) {
        const int r = threadIdx.x / MT, m = threadIdx.x % MT;
        float v[P];
#pragma unroll
        for (int p = 0; p < P; p++) {
            v[p] = red[0][(r * P + p) * MT + m];
#pragma unroll
            for (int k = 1; k < NW; k++)
                if (k < nw)
                    v[p] += red[k][(r * P + p) * MT + m];
            if constexpr (ANY)
                if (tail > 0)
                    v[p] += tred[(r * P + p) * MT + m];
        }
        if constexpr (EPI == 1) {
            /* the token's sum of x^2 over the waves, in wave order */
            float tot = nsum[0][m];
#pragma unroll
            for (int k = 1; k < NW; k++)
                if (k < nw)
                    tot += nsum[k][m];
            if constexpr (ANY)
                if (tail > 0)
                    tot += tsum[m];
            const float sc = 1.0f / sqrtf(e.eps + tot / (float)cols);
#pragma unroll
            for (int p = 0; p < P; p++)
                v[p] *= sc;
        }
        const long i = m * rows + r0 + r;
        const float o = PAIR ? q8_swiglu(v[0], v[P - 1]) : v[0];
        y[i] = EPI == 2 ? rv + o : o;
    }
}

#endif
