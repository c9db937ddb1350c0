/* Checks the two quotients of the traversal step (woxel_amd/csrc/lane.hpp) against IEEE
 * division, with the hardware reciprocal taken as the correctly rounded one and as one ulp
 * to either side of it. The sizes are those of every slot: 1..15 voxels, 8 and 128 times the
 * distance of a tile, 4096 for a missing node.
 *
 *  fast step     floor(fma(floor(p), y, y / 2)) is floor(p / size) for 2^-64 <= |p| <= 2^20:
 *                every integer f = floor(p) next to a multiple of the size (all integers for
 *                sizes below 16), p the least, a middle and the largest float with that floor.
 *  general step  fma(fma(-size, y, 1), y, y) is RN(1 / size).
 * Prints "tests N mismatches M", exits 1 if M > 0.
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static float ulps(float y, int k) {
    uint32_t u;
    memcpy(&u, &y, 4);
    u += (uint32_t)k;
    memcpy(&y, &u, 4);
    return y;
}

static long tests, bad;

static void check(float size, int f) {
    const float ff = (float)f, last = nextafterf(ff + 1.0f, -INFINITY);
    const float ps[3] = {ff, 0.5f * (ff + last), last};
    for (int k = -1; k <= 1; ++k) {
        const float y = ulps(1.0f / size, k), got = floorf(fmaf(ff, y, 0.5f * y));
        for (int i = 0; i < 3; ++i) {
            const float p = ps[i];
            if (floorf(p) != ff || fabsf(p) < 0x1p-64f || fabsf(p) > 0x1p20f) continue;
            ++tests;
            if (floorf(p / size) != got && bad++ < 5) printf("size %g p %a: %g, not %g\n", size, p, got, floorf(p / size));
        }
    }
}

static void sweep(float size) {
    const int s = (int)size, top = 1 << 20;
    for (int k = -1; k <= 1; ++k) {
        const float y0 = ulps(1.0f / size, k), y = fmaf(fmaf(-size, y0, 1.0f), y0, y0);
        ++tests;
        if (y != 1.0f / size && bad++ < 5) printf("reciprocal of %g: %a\n", size, y);
    }
    if (s < 16) {
        for (int f = -top; f <= top; ++f) check(size, f);
    } else {
        for (int m = -(top / s) * s; m <= top; m += s)
            for (int f = m - 3; f <= m + 3; ++f)
                if (f >= -top && f <= top) check(size, f);
    }
}

int main(void) {
    for (int d = 1; d <= 15; ++d) sweep((float)d), sweep((float)(8 * d));
    for (int d = 1; d <= 255; ++d) sweep((float)(128 * d));
    sweep(4096.0f);
    printf("tests %ld mismatches %ld\n", tests, bad);
    return bad ? 1 : 0;
}
