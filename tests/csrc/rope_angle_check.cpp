// The rotary table entry (lk_rope_angle_straight, host build) against the host library's
// fp64 cosine and sine rounded to fp32, the oracle's formula: argv = first
// position, end position, stride.  Prints the number compared and of entries
// whose bits differ.
#include "../../lfm2-ampere_amd/csrc/lk_common.h"
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

int main(int argc, char ** argv) {
    if (argc != 4) return 2;
    static const float F[32] = { LK_ROPE_FREQ_INIT };
    long n = 0, bad = 0;
    const long end = atol(argv[2]), step = atol(argv[3]);
    for (long pos = atol(argv[1]); pos < end; pos += step)
        for (int i = 0; i < 32; ++i, ++n) {
            float c, s;
            lk_rope_angle_straight((int) pos, F[i], c, s);
            const float a = (float) (int) pos * F[i];
            if (c != (float) cos((double) a) || s != (float) sin((double) a)) ++bad;
        }
    printf("%ld %ld\n", n, bad);
    return 0;
}
