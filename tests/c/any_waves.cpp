/* The decode kernels' waves for every number of columns: "cols waves tail_units tail_lanes" lines. */
#include <stdio.h>

#include "q8_gemv.h"

int main()
{
    for (long cols = 32; cols <= 16384; cols += 32) {
        const int nw = q8_any_waves(cols), tail = (int)(cols / 16) - 64 * nw;
        printf("%ld %d %d %d\n", cols, nw, tail > 0 ? tail : 0, tail > 0 ? q8_pow2_from(tail) : 0);
    }
    return 0;
}
