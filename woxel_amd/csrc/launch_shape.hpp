// How many rays a wave takes and which kernels a ray list goes to: host rules of the ray
// count and the GPU's compute units alone, in plain C++ so that a CPU test can sweep them.
#pragma once

#include <cstdint>

namespace wxk {

// How many rays a wave of the one-lane-per-ray shapes takes, as a power of two: 64, or fewer
// in launches too small to fill the GPU, whose time is that of their longest waves. A wave
// alone on its SIMD pays 50 clocks for a region of a step even to skip it, with 6 to 8 more
// for each instruction inside and 129 or more for a load, and it enters a region when one of
// its rays needs it, so fewer rays mean shorter steps and fewer of them; up to 4 waves per
// SIMD (16 per compute unit) hardly slow each other. 8 rays (4x2 pixels) were slower than 4
// and 16 at most sizes. Measured on 256 compute units, 64 rays against this rule: 64x36
// pixels of the ball 50.4 -> 41.4 us, of an isosurface 77.1 -> 63.9, 160x90 pixels of 1000
// spheres 112 -> 106, 448x252 164 -> 156; 500 scattered rays 50.5 -> 43.0, 8000 66.5 -> 60.9,
// 128000 75.2 -> 77.0; panoramas of 8192 and 131072 rays 85.5 -> 74.2 and 129 -> 117.
// `fast`: the grid's bound allows the fast step (kFastBound). Beyond it rays sit on cell
// borders, lane by lane alike, until the step cap: 64 Ki in waves of 16 took 645 us, in waves
// of 64 470.
inline uint32_t rays_per_wave_log2(uint64_t rays, uint32_t cus, bool fast) {
    if (!fast) return 6u;
    uint32_t lg = 0;
    while (lg < 6u && (rays >> lg) > 16u * cus) ++lg;
    return lg == 3u ? 4u : lg;
}

// A ray list of the one-lane shape: rays per wave, and whether the sets of 64 rays that
// scatter are left to the refilling kernel (k_persist1), which is when there are at least two
// sets for every wave the GPU holds: at 1 Mi rays scattered ones took 286 us against 346 in
// one kernel, a panorama 243 against 234; at half that scattered ones 251 against 193. Both
// kernels ask the same sets of 64 whether they scatter, so a split list has 64 rays a wave.
struct ListShape {
    uint32_t lg;
    bool split;
};
// k_persist1 refills the fast step alone; without it a scattered list of 1 Mi rays took 2109 us
// split, 1835 in one kernel (16 Mi 22.9 and 24.7 ms).
inline ListShape list_shape(uint64_t rays, uint32_t cus, bool fast) {
    ListShape s;
    s.split = fast && (rays + 63u) / 64u >= 2u * cus * 32u;
    s.lg = s.split ? 6u : rays_per_wave_log2(rays, cus, fast);
    return s;
}

}  // namespace wxk
