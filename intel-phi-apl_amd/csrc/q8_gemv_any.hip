/* q8_gemv_any.hip: the decode kernels (t = 1..4) for any cols, a multiple of 32 up to 16384: matrices
 * whose K is no multiple of 1024, and the epilogues at the multiples that q8_kernels.hip has no fused
 * instance for. The body is the same (q8_gemv.h) on one wave a started 1024 columns, the last wave's lanes
 * past the row counting as zero, or on 4, 8 or 12 whole ones and a tail (q8_any_waves).
 *
 * HBM-bound like the others: every load of a workgroup's rows is issued before any arithmetic, where
 * the loop over K (gemv_s, for more than 16384 columns now) keeps 4 rows' loads of one 1024-column
 * step in flight. The pair 11008 x 4128 (4 waves and a tail) at 3
 * tokens 35.1 -> 25.2 us (3.84 TB/s of weights); one-token pair 5424 x 4256 16.9 -> 10.5; a layer of
 * 1536 columns with its epilogues, which ran apart at such sizes, at 2 tokens 41.8 -> 17.4 us. With
 * a fifth wave for the two units that 4128 columns have past 4096 the pair took 39.7 us, slower than
 * the loop: five waves load the SIMDs unevenly and spend a fifth of the arithmetic on dead lanes. */
#include <hip/hip_runtime.h>

#include "q8_gemv.h"

/* any cols up to 1024 NC, with or without an epilogue */
template <int MT, int RW, int NC, int PAIR, int EPI>
__global__ __launch_bounds__(64 * NC) void gemv_any(const uint8_t *__restrict__ w0, const uint8_t *__restrict__ w1, long rows, long cols,
                                                    const float *__restrict__ x, long x_stride, float *y, q8_epi e)
{
    gemv_body<MT, RW, 1, NC, PAIR, EPI, 1>(w0, w1, rows, cols, x, x_stride, y, (long)blockIdx.x * RW, e);
}

/* a round at any cols up to 1024 NC (EPI 1: on the RMS norm of x) */
template <int MT, int RW, int NC, int EPI>
__global__ __launch_bounds__(64 * NC) void gemv_round_any(q8_round r, long cols, const float *__restrict__ x, long x_stride, q8_epi e)
{
    int p = 0;
#pragma unroll
    for (int k = 1; k < Q8_ROUND_MAX; k++)
        if (k < r.n && (long)blockIdx.x >= r.start[k])
            p = k;
    gemv_body<MT, RW, 1, NC, 0, EPI, 1>((const uint8_t *)r.w[p], nullptr, r.rows[p], cols, x, x_stride, r.y[p], ((long)blockIdx.x - r.start[p]) * RW, e);
}

/* The instances hold up to NC waves (4, 8, 12, 16), as the registers a lane may take fall with the
 * waves a workgroup may have: 8 rows a workgroup (for the pair at one token 4), as gemv_choose picks
 * for a multiple of 1024, fewer for small matrices; 4 at 13 to 16 waves where 8 spill. The norm's
 * weights take more registers: its instances stop at 8 waves. */
template <int MT, int RW, int NC, int PAIR, int EPI>
static void any_go(hipStream_t s, int nw, const void *w0, const void *w1, long rows, long cols, const float *x, long xs, float *y, const q8_epi &e)
{
    Q8_LAUNCH(q8_time_name("gemv_any", 5, MT, RW, NC, PAIR, EPI), (gemv_any<MT, RW, NC, PAIR, EPI>), dim3((unsigned)(rows / RW)), dim3(64 * nw), s,
              (const uint8_t *)w0, (const uint8_t *)w1, rows, cols, x, xs, y, e);
}
template <int MT, int NC, int PAIR, int EPI>
static void any_rw(hipStream_t s, int rw, int nw, const void *w0, const void *w1, long rows, long cols, const float *x, long xs, float *y, const q8_epi &e)
{
    if constexpr (NC < 16 || MT * (PAIR + 1) <= 2)
        if (rw == 8)
            return any_go<MT, 8, NC, PAIR, EPI>(s, nw, w0, w1, rows, cols, x, xs, y, e);
    if (rw >= 4)
        any_go<MT, 4, NC, PAIR, EPI>(s, nw, w0, w1, rows, cols, x, xs, y, e);
    else
        any_go<MT, 2, NC, PAIR, EPI>(s, nw, w0, w1, rows, cols, x, xs, y, e);
}
template <int MT, int PAIR, int EPI>
static bool any_try(hipStream_t s, const void *w0, const void *w1, long rows, long cols, const float *x, long xs, float *y, const q8_epi &e)
{
    const int nw = q8_any_waves(cols);
    /* the pair at 5 to 8 waves from two tokens: 151 to 176 registers at 8 rows leave one workgroup a
     * compute unit (12288 x 5120 at 3 tokens 45.2 us, 41.1 at 4 rows; four waves and nine or more are 5
     * to 15 % slower so). Not on the norm at 2 tokens (no gain) and at 4 (10 % slower) */
    const bool mid = nw > 4 && nw <= 8;
    int rw = PAIR && (MT == 1 || (mid && (EPI != 1 || MT == 3))) ? 4 : 8;
    while (rw > 2 && rows / rw * nw < (PAIR ? 4096 : 1024))
        rw /= 2;
    if (cols > 16384 || (EPI == 1 && nw > 8) || (mid && EPI && !e.fuse && (EPI == 1 || MT == 4) && (PAIR + 1) * rows > q8_epi_rows(MT, false)))
        return false;
    if (nw <= 4)
        any_rw<MT, 4, PAIR, EPI>(s, rw, nw, w0, w1, rows, cols, x, xs, y, e);
    else if (nw <= 8)
        any_rw<MT, 8, PAIR, EPI>(s, rw, nw, w0, w1, rows, cols, x, xs, y, e);
    if constexpr (EPI != 1) {
        if (nw > 8 && nw <= 12)
            any_rw<MT, 12, PAIR, EPI>(s, rw, nw, w0, w1, rows, cols, x, xs, y, e);
        else if (nw > 12)
            any_rw<MT, 16, PAIR, EPI>(s, rw, nw, w0, w1, rows, cols, x, xs, y, e);
    }
    return true;
}
template <int MT>
static bool any_t(hipStream_t s, const void *w0, const void *w1, long rows, long cols, const float *x, long xs, float *y, const q8_epi &e)
{
    if (w1)
        return e.nw ? any_try<MT, 1, 1>(s, w0, w1, rows, cols, x, xs, y, e) : any_try<MT, 1, 0>(s, w0, w1, rows, cols, x, xs, y, e);
    if (e.nw)
        return any_try<MT, 0, 1>(s, w0, w1, rows, cols, x, xs, y, e);
    return e.res ? any_try<MT, 0, 2>(s, w0, w1, rows, cols, x, xs, y, e) : any_try<MT, 0, 0>(s, w0, w1, rows, cols, x, xs, y, e);
}

bool q8_launch_gemv_any(q8_stream_t stream, const void *w0, const void *w1, long rows, long cols, const float *x, long x_stride, long t, float *y, q8_epi e)
{
    hipStream_t s = (hipStream_t)stream;
    switch (t) {
    case 1: return any_t<1>(s, w0, w1, rows, cols, x, x_stride, y, e);
    case 2: return any_t<2>(s, w0, w1, rows, cols, x, x_stride, y, e);
    case 3: return any_t<3>(s, w0, w1, rows, cols, x, x_stride, y, e);
    default: return any_t<4>(s, w0, w1, rows, cols, x, x_stride, y, e);
    }
}

template <int MT, int EPI>
static bool round_try(hipStream_t s, const q8_round &r, long cols, const float *x, long xs, const q8_epi &e)
{
    const int nw = q8_any_waves(cols);
#define ANY(N)                                                                                                         \
    Q8_LAUNCH(q8_time_name("gemv_round_any", 4, MT, Q8_ROUND_RW, N, EPI), (gemv_round_any<MT, Q8_ROUND_RW, N, EPI>), dim3((unsigned)r.start[r.n]), \
              dim3(64 * nw), s, r, cols, x, xs, e)
    if (cols > 16384 || nw > (EPI == 1 ? 8 : MT > 2 ? 12 : 16) || (EPI == 1 && !e.fuse && nw > 4 && r.start[r.n] * Q8_ROUND_RW > q8_epi_rows(MT, false)))
        return false;
    if (nw <= 4)
        ANY(4);
    else if (nw <= 8)
        ANY(8);
    if constexpr (EPI != 1) {
        if (nw > 8 && nw <= 12)
            ANY(12);
        if constexpr (MT <= 2)
            if (nw > 12)
                ANY(16);
    }
#undef ANY
    return true;
}
template <int MT>
static bool round_t(hipStream_t s, const q8_round &r, long cols, const float *x, long xs, const q8_epi &e)
{
    return e.nw ? round_try<MT, 1>(s, r, cols, x, xs, e) : round_try<MT, 0>(s, r, cols, x, xs, e);
}

bool q8_launch_round_any(q8_stream_t stream, const q8_round &r, long cols, const float *x, long x_stride, long t, q8_epi e)
{
    hipStream_t s = (hipStream_t)stream;
    switch (t) {
    case 1: return round_t<1>(s, r, cols, x, x_stride, e);
    case 2: return round_t<2>(s, r, cols, x, x_stride, e);
    case 3: return round_t<3>(s, r, cols, x, x_stride, e);
    default: return round_t<4>(s, r, cols, x, x_stride, e);
    }
}
