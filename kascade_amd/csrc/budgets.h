// Index budgets of the prefill kernels.  Plain arithmetic, the same on the host and on the device.
#pragma once
#include <math.h>

namespace kascade {

// max(128, floor(pct tile_start / 100)) rounded up to 128: the entries a tile at tile_start takes under rolling budgets.
__host__ __device__ inline int rolling_budget(float pct, int tile_start) {
    // The floor without a division, which every unit's first list entry would wait for (517 tokens
    // 9.80 -> 9.68 us).  x is exact, and where it is no multiple of 100 it lies a relative 2^-44 or more off
    // the next one: the quotient's rounding does not reach it, so this is the floor of the rounded quotient too.
    // Percentages are not bounded by the calls: 10^9 entries are more than any list holds and fit an int.
    const double x = fmin((double)pct * (double)tile_start, 1e11);
    int fl = (int)(x * 0.01);
    fl += (double)(fl + 1) * 100.0 <= x;
    fl -= (double)fl * 100.0 > x;
    return fl > 128 ? (fl + 127) & ~127 : 128;
}

// Index-row width the host gives a prompt of L keys: min(128 ceil(min(max(128, floor(pct L / 100)), L) / 128), L).
__host__ __device__ inline int topk_width_of(float pct, int L) {
    long long k = (long long)floor((double)pct * (double)L / 100.0);
    if (k < 128) k = 128;
    if (k > L) k = L;
    k = ((k + 127) / 128) * 128;
    return (int)(k > L ? L : k);
}

}  // namespace kascade
