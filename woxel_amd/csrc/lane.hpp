// Per-lane HDDA + grid-SDF traversal shared by the traversal and render kernels.
//
// The per-ray arithmetic restates hdda_ray (src/shaders/raycast.comp.wgsl:84-126)
// operation for operation, in FP32 with contraction off (-ffp-contract=off) and
// IEEE division and square root, so results are bit-identical to the scalar
// oracle. The lookups restate get_vdb_leaf_from_{leaf,nothing,node5,node4,node3}
// (raycast.comp.wgsl:360-494) over one 2-byte entry per node slot (a child's rank, or
// the step size of a tile) and one 4-bit slot per voxel (0 = active, else SDF), so every
// tree level costs a single gather and next to no decoding.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/woxel_hip.h"
#include "device_arena.hpp"
#include "launch_shape.hpp"

namespace wxk {

constexpr uint32_t kMaxSteps = 1000u;  // HDDA_MAX_RAY_STEPS (raycast.comp.wgsl:82)
constexpr uint32_t kRun = 0xFFu;       // lane state: still stepping

struct GridDev {
    const int4 *root;     // n5 x {kx, ky, kz, index}
    const void *n5;       // n5 x 32768 slot entries (below)
    const void *n4;       // n4 x 4096 slot entries
    const uint32_t *leaf; // n3 x 64 words
    const uint32_t *base; // compact entries: base[i] + kWalk = index of node-4 i's rank-0 leaf,
                          // base[-1 - k] + kWalk = index of node-5 k's rank-0 node-4
    uint32_t n5count;
    float bound;
    uint32_t form;        // kOneRoot, kTable or kIndexed
    int32_t kx, ky, kz;   // the key of root[0]
};
static_assert(sizeof(GridDev) == 64, "GridDev layout");

// Slot entries of the device node pools, in child-offset order (x major, z minor), made
// on the device from the 16-byte records of the layout (k_expand). An entry of 2 bytes is
// either kWalk | rank -- the child to walk into, counted from the node's base (children of
// a node are consecutive, at most 32768 in a node-5 and 4096 in a node-4) -- or the size of
// a step out of the slot, its SDF distance times its 128 (node-5) or 8 (node-4) voxels, as
// the upper half of the float, which holds every distance up to 255; +0.0 is an active
// tile. Against the records (8 or 16 slots in 16 bytes: child and walk bits, first child,
// packed distances) an entry needs no bit tests, popcount or distance extraction. A
// node-5 takes the same 64 KiB, a node-4 8 KiB instead of 4, and the records stay beside them
// for wx_grid_save (the 2000-sphere grid: 167 MiB with, 134 before entries); entries of 4
// bytes with whole child indices (measured first) took twice that and lost on the 4096^3
// sphere set what the shorter lookup gained: L2 requests per frame 13.4 M (records), 23.9 M (4 bytes).
// Forms of a grid, from its node counts and records (wx_grid_create):
//   kOneRoot  compact entries, one node-5 of base 0 with a key of 20 bits, every pool within
//             32-bit byte offsets;
//   kTable    compact entries, any root table, 64-bit addresses;
//   kIndexed  4-byte entries (kWalk32 | child index, or the size as a float) for a layout
//             whose children are not consecutive, which no builder here makes.
constexpr uint32_t kOneRoot = 0u, kTable = 1u, kIndexed = 2u;
constexpr uint32_t kWalk = 0x8000u, kWalk32 = 0x80000000u;

// Root tables of up to kRootLds entries are scanned from LDS by the kernels that
// trace one grid (a copy made at workgroup start); a grid with one node-5 needs no
// table at all (GridDev::kx), a larger table is scanned through the L1 cache.
constexpr uint32_t kRootLds = 16u;
// Stages the root table of g in s_root when it has 2..kRootLds entries; returns
// whether it did (the lookups then scan s_root, else g.root). Every lane of the
// workgroup calls it; n5count is uniform, and so is the barrier that publishes the copy.
__device__ __forceinline__ bool stage_root(const GridDev &g, int4 *s_root) {
    if (g.n5count <= 1u || g.n5count > kRootLds) return false;
    for (uint32_t i = threadIdx.x; i < g.n5count; i += blockDim.x) s_root[i] = g.root[i];
    __syncthreads();
    return true;
}

__device__ __forceinline__ float smin(float a, float b) { return b < a ? b : a; }
__device__ __forceinline__ float smax(float a, float b) { return a < b ? b : a; }

// f32 -> i32: truncate, saturate, NaN -> 0. This is exactly the rule of the
// hardware conversion, so it is one instruction (a C++ cast of an out-of-range
// value would be undefined and lets the compiler assume anything).
__device__ __forceinline__ int32_t f2i(float x) {
    int32_t r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// f2i(floorf(x)) in one instruction: equal on every input but the NaNs.
__device__ __forceinline__ int32_t f2i_floor(float x) {
    int32_t r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// One ray in flight. The lookup cache of the reference (VdbLeaf.parents) is kept
// as the last looked-up voxel and the last entries read at node-5 and node-4: a cached
// node is the one containing that voxel, and an entry that is not a walk ended the
// lookup, so its level is looked up again. The ray origin is not kept: camera rays start
// at the (uniform) eye, explicit rays re-read it at the end, shadow rays keep it in LDS.
// The axis mask of the last step is kept as the nudge each axis received (+-4e-4 on the
// stepped axes, a zero on the others).
struct RayLane {
    float dx, dy, dz, ix, iy, iz, px, py, pz;
    float ax, ay, az;     // last nudge per axis
    uint32_t qx, qy, qz;  // last looked-up voxel, biased (voxel_bits)
    uint32_t e5, e4;      // last node-5 / node-4 entry, as 4 bytes (an entry of 2 bytes in the upper half)
    uint32_t b5, b4;      // base of the last node-5 (not in kOneRoot, where it is 0) / node-4 looked up
    int32_t i5;           // node-5 index of the last root lookup, -1: none (not in kOneRoot)
    uint32_t c5, c4;      // node-5 (with root misses) / node-4 lookups | those that walked on << 15
    uint32_t miss, n3;    // root misses; leaf lookups
    float fx, fy, fz;       // floor of the position last looked up
    float size;             // step size found there, 0: a hit
    uint32_t state;       // kRun or the final state
    uint32_t s01, s23;    // record words (lane_finish): steps[k] = lookups resolved at num_parents k,
    uint32_t lk;          // s01 = steps0 | steps1 << 16, s23 = steps2 | steps3 << 16; L5 | L4 << 10
};

// The hit record's lookup word L5 | L4 << 10 | L3 << 20 (every leaf lookup ends the chain: L3 = steps3).
__device__ __forceinline__ uint32_t lookup_word(const RayLane &r) { return r.lk | (r.s23 >> 16) << 20; }

// Iterations done: every iteration ends its lookup chain at exactly one level.
__device__ __forceinline__ uint32_t lane_iterations(const RayLane &r) {
    return (r.s01 & 0xFFFFu) + (r.s01 >> 16) + (r.s23 & 0xFFFFu) + (r.s23 >> 16);
}

__device__ __forceinline__ uint32_t lane_state(const RayLane &r) { return r.state; }
__device__ __forceinline__ void set_state(RayLane &r, uint32_t st) { r.state = st; }

// The T at byte `off` of node or leaf `idx`, of 2^kShift bytes each, in a pool. The narrow
// form is a 32-bit offset that the load itself adds to the uniform base.
template <typename T, bool kNarrow, int kShift>
__device__ __forceinline__ T pool_at(const void *pool, uint32_t idx, uint32_t off) {
    const char *base = static_cast<const char *>(pool);
    if (kNarrow) return *reinterpret_cast<const T *>(base + ((idx << kShift) | off));
    return *reinterpret_cast<const T *>(base + (((uint64_t)idx << kShift) | off));
}

// Workgroup -> image tile under XCD-aware dispatch. The hardware hands workgroup b
// to XCD b % 8; with `band` the tiles are renumbered so that each XCD takes one
// contiguous band of the nb row-major tiles and its own L2 holds that band's nodes
// (otherwise neighbouring tiles land on different XCDs). A bijection on [0, nb).
constexpr uint32_t kXcds = 8u;
__device__ __forceinline__ void tile_of_block(bool band, uint32_t &bx, uint32_t &by) {
    bx = blockIdx.x, by = blockIdx.y;
    if (!band) return;
    const uint32_t nb = gridDim.x * gridDim.y, b = by * gridDim.x + bx;
    const uint32_t q = nb / kXcds, r = nb % kXcds, x = b % kXcds, k = b / kXcds;
    const uint32_t t = x < r ? x * (q + 1u) + k : r * (q + 1u) + (x - r) * q + k;
    bx = t % gridDim.x, by = t / gridDim.x;
}

// A lane takes up a ray that lane_start left running: nothing looked up or counted yet.
__device__ __forceinline__ void lane_resume(RayLane &r, float px, float py, float pz, float dx, float dy, float dz,
                                            float ix, float iy, float iz) {
    r.px = px, r.py = py, r.pz = pz;
    r.dx = dx, r.dy = dy, r.dz = dz;
    r.ix = ix, r.iy = iy, r.iz = iz;
    r.ax = 0.0f, r.ay = 0.0f, r.az = 0.0f;
    r.s01 = 0, r.s23 = 0, r.lk = 0, r.state = kRun;
    r.c5 = 0, r.c4 = 0, r.miss = 0, r.n3 = 0, r.qx = 0, r.qy = 0, r.qz = 0;
    r.e5 = 0, r.e4 = 0, r.b5 = 0, r.b4 = 0, r.i5 = -1;  // nothing cached
}

// Entry clip (extension of the reference's bound test, identical in the oracle):
// a ray starting outside [-bound, bound]^3 starts at its slab entry point,
// clamped into the box; a ray missing the box ends OOB with no lookups.
__device__ __forceinline__ void lane_start(RayLane &r, float ox, float oy, float oz, float dx, float dy, float dz,
                                           float B, bool clip) {
    // canonicalized: quiet a signalling NaN so that a max over |p| ignores it like the
    // comparisons of the bound test and of the clip below do (every other value passes unchanged)
    ox = __builtin_canonicalizef(ox), oy = __builtin_canonicalizef(oy), oz = __builtin_canonicalizef(oz);
    lane_resume(r, ox, oy, oz, dx, dy, dz, 1.0f / dx, 1.0f / dy, 1.0f / dz);  // :88
    if (clip && (B < fabsf(ox) || B < fabsf(oy) || B < fabsf(oz))) {
        float tn = -__builtin_inff(), tf = __builtin_inff();
        float a = (-B - ox) * r.ix, b = (B - ox) * r.ix;
        tn = smax(tn, smin(a, b));
        tf = smin(tf, smax(a, b));
        a = (-B - oy) * r.iy, b = (B - oy) * r.iy;
        tn = smax(tn, smin(a, b));
        tf = smin(tf, smax(a, b));
        a = (-B - oz) * r.iz, b = (B - oz) * r.iz;
        tn = smax(tn, smin(a, b));
        tf = smin(tf, smax(a, b));
        if (!(tn <= tf) || tf < 0.0f) {
            set_state(r, WX_OOB);
            return;
        }
        r.px = smin(smax(ox + tn * dx, -B), B);
        r.py = smin(smax(oy + tn * dy, -B), B);
        r.pz = smin(smax(oz + tn * dz, -B), B);
    }
}

// The fast step is taken by waves whose running rays all satisfy, per axis:
//  * the direction is finite and its reciprocal too, or the direction is +0 and the
//    start p is >= 0 or <= -2^-9;
//  * the start is not -0 and at most 2^21 in magnitude;
// and whose largest direction component is at least 2^-60, on a grid with bound <=
// kFastBound. Then nothing in the step is a NaN and the shortcuts below give the
// reference's values:
//  * t = (1/d) * (size * max(0, s) - m) is finite on the largest axis, so the least t is
//    finite and the advance t * d too. On an axis with d = +0 it is inf * c with c > 0:
//    c = size - m, and m reaches size only by rounding, for p in [-2^-10, 0) (size <
//    2^15); p never changes on that axis, as its t is never the least.
//  * t <= both others exactly when t equals their minimum; a minimum of zeros of either
//    sign may pick another zero than the reference's comparisons, which only the sign of a
//    zero p can show -- and p is never -0, since a sum is -0 only if both terms are.
//  * with p never -0, adding 0 instead of -0 on the axes not stepped changes nothing.
//  * floor(p / size) of the rounded IEEE quotient equals the floor of the true one unless
//    the quotient underflows: size is an integer, so p differs from a multiple k size by at
//    least one ulp of p, more than half an ulp of k carries. And the true one is
//    floor((floor(p) + 1/2) / size): that argument lies at least 1/(2 size) from every
//    integer, so a reciprocal good to one ulp decides it for |p| <= 2^20 (error below
//    0.2 / size). k size is an exact float, so p - k size in one fma rounds as the
//    reference's product and difference do.
// An underflowing quotient (p in (-2^-64, 0)) is looked at separately. A step moves no axis
// by more than its size (< 2^15), so |p| stays below 2^21 + 2^15 and the voxel is exact in
// the mantissa of floor(p) + 1.5 * 2^23 (voxel_bits).
constexpr float kFastBound = 0x1p20f;

// The steps a wave can take, each where the one before does not serve; all give the same
// records. kClean: direction, reciprocal and start are finite, whatever the bound. Then every t
// is a product of finite numbers, an infinite position ends at the bound test, and nothing in
// the step is a NaN: one conversion floors, and t equals the minimum exactly when it is <= both
// others. It and the general step take the quotient in three operations where IEEE division
// takes eleven each: 1 Mi rays with a -0 start in every wave 755 -> 645 us, a 1080p frame of a
// grid of one node-5 and bound 2^21 4854 -> 3100.
constexpr int kGeneral = 0, kClean = 1, kFast = 2;

__device__ __forceinline__ bool axis_fast(float d, float inv, float p) {
    constexpr float kInf = __builtin_inff();
    const bool dir = (fabsf(d) < kInf && fabsf(inv) < kInf) ||
                     (__float_as_uint(d) == 0u && (p >= 0.0f || p <= -0x1p-9f));
    return dir && fabsf(p) <= 0x1p21f && __float_as_uint(p) != 0x80000000u;
}

__device__ __forceinline__ bool lane_fast(const RayLane &r) {
    return axis_fast(r.dx, r.ix, r.px) && axis_fast(r.dy, r.iy, r.py) && axis_fast(r.dz, r.iz, r.pz) &&
           fmaxf(fmaxf(fabsf(r.dx), fabsf(r.dy)), fabsf(r.dz)) >= 0x1p-60f;
}

__device__ __forceinline__ bool lane_clean(const RayLane &r) {
    constexpr float kInf = __builtin_inff();
    return fabsf(r.dx) < kInf && fabsf(r.dy) < kInf && fabsf(r.dz) < kInf && fabsf(r.ix) < kInf && fabsf(r.iy) < kInf &&
           fabsf(r.iz) < kInf && fabsf(r.px) < kInf && fabsf(r.py) < kInf && fabsf(r.pz) < kInf;
}

// A voxel coordinate as the lookups use it: x + kVoxelBias (mod 2^32). The low 22 bits are
// the coordinate's, differences are the coordinate's, and for |x| < 2^22 it is the bit
// pattern of the float x + 1.5 * 2^23: one add instead of a conversion.
constexpr uint32_t kVoxelBias = 0x4B400000u;
__device__ __forceinline__ uint32_t voxel_bits(float floored) { return __float_as_uint(floored + 12582912.0f); }

// The root lookup (get_vdb_leaf_from_nothing, :398-413) in a table: index of the first
// root entry with the key of voxel (x, y, z), or -1. No lane leaves a scan by itself: the
// masks that takes had come to cost more than the entries it saves, and a scan in memory
// waited for every entry. Two steps of this file ago, last, and now: 1080p of 2000 spheres
// over 9 node-5s 517, 482, 424 us, 16.8 M scattered rays over 8 7147, 3889, 3100; 1080p over 64
// 47.9, 57.6, 40.1 ms. The LDS scan unrolled takes 66 to 82 VGPRs instead of 52; from memory
// one entry at a time 53.8 ms for the last, two 44.3, four and a pair apart for tables of two
// (8 requests over 2 node-5s: 3.03 ms, in fours 4.42).
__device__ __forceinline__ int32_t root_find(const GridDev &g, uint32_t x, uint32_t y, uint32_t z,
                                             const int4 *s_root, bool root_lds) {
    const int32_t kx = (int32_t)(x - kVoxelBias) >> 12, ky = (int32_t)(y - kVoxelBias) >> 12,
                  kz = (int32_t)(z - kVoxelBias) >> 12;
    if (g.n5count == 1u) return kx == g.kx && ky == g.ky && kz == g.kz ? 0 : -1;
    int32_t found = -1;
    if (root_lds) {  // from the last entry to the first, so that the first of equal keys stands
#pragma clang loop unroll(disable)
        for (uint32_t k = g.n5count; k-- > 0u;) {
            const int4 e = s_root[k];
            found = ((e.x ^ kx) | (e.y ^ ky) | (e.z ^ kz)) == 0 ? e.w : found;
        }
    } else {  // a few entries at a time, read as constants: scalar loads where the grid is uniform
        using Entry = int32_t __attribute__((ext_vector_type(4)));
        const auto *root = (const __attribute__((address_space(4))) Entry *)(uintptr_t)g.root;
        auto pick = [&](uint32_t k) {
            const Entry e = root[k < g.n5count ? k : g.n5count - 1u];
            found = (found < 0) & (((e.x ^ kx) | (e.y ^ ky) | (e.z ^ kz)) == 0) ? e.w : found;
        };
        if (g.n5count <= 2u) {
            if (g.n5count) pick(0u), pick(1u);
            return found;
        }
#pragma clang loop unroll(disable)
        for (uint32_t k = 0; k < g.n5count; k += 4u) {
            pick(k), pick(k + 1u), pick(k + 2u), pick(k + 3u);
            if (__ballot(found < 0) == 0ull) break;  // the wave's lanes all have theirs
        }
    }
    return found;
}

// a's bits where the mask is set, b's elsewhere (in C the compiler masks both operands first);
// acc | (a ^ b) and acc | (~a & b).
__device__ __forceinline__ uint32_t bits_of(uint32_t mask, uint32_t a, uint32_t b) {
    return (uint32_t)__builtin_amdgcn_bitop3_b32((int)mask, (int)a, (int)b, 0xCA);
}
__device__ __forceinline__ uint32_t or_xor(uint32_t acc, uint32_t a, uint32_t b) {
    return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)acc, 0xBE);
}
__device__ __forceinline__ uint32_t or_andn(uint32_t acc, uint32_t a, uint32_t b) {
    return (uint32_t)__builtin_amdgcn_bitop3_b32((int)acc, (int)a, (int)b, 0xF2);
}

// a && b as the compiler cannot see through it: a flag in a scalar mask, not branches threaded
// past the code that follows.
__device__ __forceinline__ bool opaque_and(bool a, bool b) {
    uint64_t m = __builtin_amdgcn_ballot_w64(a) & __builtin_amdgcn_ballot_w64(b);
    asm volatile("" : "+s"(m));
    return __builtin_amdgcn_inverse_ballot_w64(m);
}

// The lookup of one iteration (raycast.comp.wgsl:344-494): the step size at voxel (x, y, z).
// Each level is one region of the lanes that need it, and no region nests in another: a
// wave alone on its SIMD pays about 25 ns for a divergent region, six VALU instructions.
// Large frames are bound by VALU issue first (VALUBusy 81 % on the 1080p sphere frame, its tail
// included), so the regions are written for their instruction count: offsets by bit-field
// inserts of shifted coordinates, whose unwanted bits the last insert drops, and an entry's walk
// mark left in an index and taken off its base instead.
template <uint32_t kForm>
__device__ __forceinline__ float lane_lookup(const GridDev &g, RayLane &r, uint32_t x, uint32_t y, uint32_t z,
                                             const int4 *s_root, bool root_lds) {
    // get_vdb_leaf_from_leaf (:360-396): the lookup starts at the deepest cached node that
    // still contains the voxel; a level whose entry was no walk is looked up again
    const uint32_t diff = or_xor(or_xor(x ^ r.qx, y, r.qy), z, r.qz);
    r.qx = x, r.qy = y, r.qz = z;
    if (or_andn(diff, r.e5, kWalk32) >= 128u) {  // get_vdb_leaf_from_nothing / _node5 (:398-444)
        bool miss;
        uint32_t raw = 0;
        if (kForm == kOneRoot) {  // every slot lies inside the node, so a miss may read one too
            const uint32_t kx = kVoxelBias + ((uint32_t)g.kx << 12), ky = kVoxelBias + ((uint32_t)g.ky << 12),
                           kz = kVoxelBias + ((uint32_t)g.kz << 12);
            const uint32_t off = bits_of(0x3Eu, z >> 6, bits_of(0x7C0u, y >> 1, x << 4)) & 0xFFFEu;
            raw = pool_at<uint16_t, true, 16>(g.n5, 0u, off);
            miss = or_xor(or_xor(x ^ kx, y, ky), z, kz) >= 4096u;
        } else {
            const uint32_t slot = (x & 0xF80u) << 3 | (y & 0xF80u) >> 2 | (z & 0xF80u) >> 7;
            if (diff >= 4096u || r.i5 < 0) {
                r.i5 = root_find(g, x, y, z, s_root, root_lds);
                if (kForm == kTable && r.i5 >= 0) r.b5 = g.base[-1 - (int64_t)r.i5];
            }
            miss = r.i5 < 0;
            if (!miss)
                raw = kForm == kTable ? pool_at<uint16_t, false, 16>(g.n5, (uint32_t)r.i5, slot * 2u)
                                      : pool_at<uint32_t, false, 17>(g.n5, (uint32_t)r.i5, slot * 4u);
        }
        constexpr int kUp = kForm == kIndexed ? 0 : 16;
        if (miss) raw = __float_as_uint(4096.0f) >> kUp;  // distance 1 at depth 0 (:412)
        r.c5 += kForm == kIndexed ? (raw >> 31 << 15) + 1u : (raw & kWalk) + 1u;
        r.miss += miss ? 1u : 0u;
        r.e5 = raw << kUp;
    }
    const bool in4 = (int32_t)r.e5 < 0;
    const uint32_t y2 = y << 2, z2 = z << 2;
    if (in4 & (or_andn(diff, r.e4, kWalk32) >= 8u)) {  // get_vdb_leaf_from_node4 (:446-475)
        if (kForm == kOneRoot) {
            const uint32_t off = bits_of(0x1Eu, z >> 2, bits_of(0x1E0u, y2, x << 6));
            const char *n4 = static_cast<const char *>(g.n4) - ((size_t)kWalk << 13);
            const uint32_t raw = pool_at<uint16_t, true, 0>(n4, 0u, bits_of(0x1FFEu, off, r.e5 >> 3));
            r.b4 = pool_at<uint32_t, true, 0>(g.base - kWalk, 0u, r.e5 >> 14);
            r.c4 += (raw & kWalk) + 1u;
            r.e4 = raw << 16;
        } else {
            const uint32_t off = (x & 0x78u) << 6 | (y & 0x78u) << 2 | ((z >> 2) & 0x1Eu);
            if (kForm == kTable) {
                const uint32_t i4 = (r.e5 >> 16) + r.b5;
                r.e4 = (uint32_t)pool_at<uint16_t, false, 13>(g.n4, i4, off) << 16;
                r.b4 = g.base[i4];
            } else {
                r.e4 = pool_at<uint32_t, false, 14>(g.n4, r.e5 & ~kWalk32, off * 2u);
            }
            r.c4 += (r.e4 >> 31 << 15) + 1u;
        }
    }
    float size = __uint_as_float(in4 ? r.e4 : r.e5);
    if (in4 & ((int32_t)r.e4 < 0)) {  // get_vdb_leaf_from_node3 (:477-494)
        // word (off >> 3) of 64 per leaf holds 8 4-bit slots, off = x<<6 | y<<3 | z
        const uint32_t leaf = kForm == kIndexed ? r.e4 & ~kWalk32 : r.b4 + (r.e4 >> 16);
        const uint32_t w = pool_at<uint32_t, kForm == kOneRoot, 8>(g.leaf, leaf, bits_of(0x1Cu, y2, x << 5) & 0xFCu);
        r.n3 += 1u;
        size = (float)__builtin_amdgcn_ubfe(w, z2, 4u);  // the shift takes 5 bits: (z & 7) * 4
    }
    return size;
}

// First half of an iteration of the hdda_ray loop (raycast.comp.wgsl:92-103): looks the
// position up; false when the ray ends there, at a hit or out of bounds.
//  kStep  kFast when every running ray of the wave is fast (lane_fast) and the bound allows
//         it, kClean when every one is clean (lane_clean), else kGeneral
//  kForm  the grid's form (GridDev::form; kTable serves kOneRoot too)
template <int kStep, uint32_t kForm>
__device__ __forceinline__ bool lane_look(const GridDev &g, RayLane &r, const int4 *s_root, bool root_lds) {
    r.fx = floorf(r.px), r.fy = floorf(r.py), r.fz = floorf(r.pz);
    if (kStep == kFast)
        r.size = lane_lookup<kForm>(g, r, voxel_bits(r.fx), voxel_bits(r.fy), voxel_bits(r.fz), s_root, root_lds);
    else if (kStep == kClean)
        r.size = lane_lookup<kForm>(g, r, (uint32_t)f2i_floor(r.px) + kVoxelBias, (uint32_t)f2i_floor(r.py) + kVoxelBias,
                                    (uint32_t)f2i_floor(r.pz) + kVoxelBias, s_root, root_lds);
    else
        r.size = lane_lookup<kForm>(g, r, (uint32_t)f2i(r.fx) + kVoxelBias, (uint32_t)f2i(r.fy) + kVoxelBias,
                                    (uint32_t)f2i(r.fz) + kVoxelBias, s_root, root_lds);
    // :96-98 hit (distance 0), then :101-103 any(bound < |p|) (NaN components compare
    // false either way)
    const bool run = opaque_and(!(g.bound < fmaxf(fmaxf(fabsf(r.px), fabsf(r.py)), fabsf(r.pz))), r.size != 0.0f);
    // a negative quotient that underflows has floor -0, not -1
    if (kStep == kFast && fminf(fminf(fabsf(r.px), fabsf(r.py)), fabsf(r.pz)) < 0x1p-64f) {
        if (fabsf(r.px) < 0x1p-64f && r.px / r.size == 0.0f) r.fx = 0.0f;
        if (fabsf(r.py) < 0x1p-64f && r.py / r.size == 0.0f) r.fy = 0.0f;
        if (fabsf(r.pz) < 0x1p-64f && r.pz / r.size == 0.0f) r.fz = 0.0f;
    }
    return run;
}

// p / size rounded to nearest (Markstein), for size = d 2^k with d < 256, y = RN(1/size) and
// 2^-64 <= |p| <= 2^100: no intermediate leaves the range of normal numbers.
__device__ __forceinline__ float quotient(float p, float size, float y) {
    const float q0 = p * y;
    return __builtin_fmaf(__builtin_fmaf(-q0, size, p), y, q0);
}

// Second half (:105-122): the step out of the slot that lane_look found.
template <int kStep>
__device__ __forceinline__ void lane_advance(RayLane &r) {
    constexpr bool fast = kStep == kFast;
    const float size = r.size;
    // modulo_vec3f (:78-80): m = p - size * floor(p / size)
    float mx, my, mz, tm;
    bool bx, by, bz;
    if (fast) {
        const float y1 = __builtin_amdgcn_rcpf(size), yh = 0.5f * y1;
        mx = __builtin_fmaf(-size, floorf(__builtin_fmaf(r.fx, y1, yh)), r.px);
        my = __builtin_fmaf(-size, floorf(__builtin_fmaf(r.fy, y1, yh)), r.py);
        mz = __builtin_fmaf(-size, floorf(__builtin_fmaf(r.fz, y1, yh)), r.pz);
    } else {
        // the IEEE quotient, with y = RN(1/size) from v_rcp_f32 (one ulp) and one Newton step;
        // |p| <= 2^100 as the bound is
        const float y0 = __builtin_amdgcn_rcpf(size), y = __builtin_fmaf(__builtin_fmaf(-size, y0, 1.0f), y0, y0);
        float qx = quotient(r.px, size, y), qy = quotient(r.py, size, y), qz = quotient(r.pz, size, y);
        if (!(fminf(fminf(fabsf(r.px), fabsf(r.py)), fabsf(r.pz)) >= 0x1p-64f))
            qx = r.px / size, qy = r.py / size, qz = r.pz / size;
        mx = r.px - size * floorf(qx);
        my = r.py - size * floorf(qy);
        mz = r.pz - size * floorf(qz);
    }
    const bool nx = r.dx < 0.0f, ny = r.dy < 0.0f, nz = r.dz < 0.0f;  // sign11 (:70-76)
    // :114; size * max(0, sign) is size or 0, exact in the fma (whose negated operand would
    // flip the sign of a NaN)
    const float gx = nx ? 0.0f : 1.0f, gy = ny ? 0.0f : 1.0f, gz = nz ? 0.0f : 1.0f;
    const float tx = r.ix * (fast ? __builtin_fmaf(size, gx, -mx) : size * gx - mx);
    const float ty = r.iy * (fast ? __builtin_fmaf(size, gy, -my) : size * gy - my);
    const float tz = r.iz * (fast ? __builtin_fmaf(size, gz, -mz) : size * gz - mz);
    if (kStep != kGeneral) {  // :116, :118-120
        tm = fast ? fminf(fminf(tx, ty), tz) : smin(smin(tx, ty), tz);
        bx = tx == tm, by = ty == tm, bz = tz == tm;
    } else {
        tm = smin(smin(tx, ty), tz);
        bx = (tx <= ty) & (tx <= tz);
        by = (ty <= tz) & (ty <= tx);
        bz = (tz <= tx) & (tz <= ty);
    }
    // :122, p + (4e-4 * step) * f32(mask): the product is 4e-4 * step or a zero with the
    // sign of step
    const float sx = nx ? -4e-4f : 4e-4f, sy = ny ? -4e-4f : 4e-4f, sz = nz ? -4e-4f : 4e-4f;
    r.ax = bx ? sx : (fast ? 0.0f : 0.0f * sx);
    r.ay = by ? sy : (fast ? 0.0f : 0.0f * sy);
    r.az = bz ? sz : (fast ? 0.0f : 0.0f * sz);
    r.px = (r.px + tm * r.dx) + r.ax;
    r.py = (r.py + tm * r.dy) + r.ay;
    r.pz = (r.pz + tm * r.dz) + r.az;
}

// The state and the record words of a lane whose ray ended, or met the step cap.
__device__ __forceinline__ void lane_finish(RayLane &r, bool capped) {
    const uint32_t l5 = (r.c5 & 0x7FFFu) - r.miss, n4 = r.c4 & 0x7FFFu;
    r.s01 = r.miss | (l5 - (r.c5 >> 15)) << 16;
    r.s23 = (n4 - (r.c4 >> 15)) | r.n3 << 16;
    r.lk = l5 | n4 << 10;
    r.state = capped ? WX_MAXSTEPS : (r.size == 0.0f ? WX_HIT : WX_OOB);
}

// The rays of a wave whose lanes start together, to their end: the trip count, and with it
// the step cap, is a scalar. The loop starts with the second half of an iteration, so that
// leaving it is the only region between a lookup and the step after it; whether a ray left
// it at its end or at the cap is asked again behind it, not carried through it (three scalar
// instructions a step: 3837x2157 noise frame 467 -> 461 us, 1080p spheres 287 -> 284).
template <int kStep, uint32_t kForm>
__device__ __forceinline__ void lane_loop(const GridDev &g, RayLane &r, const int4 *s_root, bool root_lds) {
    if (lane_state(r) != kRun) return;
    if (lane_look<kStep, kForm>(g, r, s_root, root_lds)) {
        uint32_t looks = 1;
        do {
            lane_advance<kStep>(r);
            if (!lane_look<kStep, kForm>(g, r, s_root, root_lds)) break;
        } while (++looks < kMaxSteps);
    }
    const bool run = !(g.bound < fmaxf(fmaxf(fabsf(r.px), fabsf(r.py)), fabsf(r.pz))) & (r.size != 0.0f);
    if (run) lane_advance<kStep>(r);
    lane_finish(r, run);
}

// Runs the rays of a wave whose lanes all started together (the one-lane-per-ray
// shapes) to their end. The choices that hold for the whole wave (fast rays, the grid's
// form) are made once here, so the loop carries no branch on them.
__device__ __forceinline__ void lane_run(const GridDev &g, RayLane &r, const int4 *s_root = nullptr,
                                         bool root_lds = false) {
    const bool fast = g.bound <= kFastBound && __ballot(lane_state(r) == kRun && !lane_fast(r)) == 0ull;
    if (fast && g.form == kOneRoot) return lane_loop<kFast, kOneRoot>(g, r, s_root, root_lds);
    if (fast && g.form == kTable) return lane_loop<kFast, kTable>(g, r, s_root, root_lds);
    if (fast) return lane_loop<kFast, kIndexed>(g, r, s_root, root_lds);
    const bool clean = __ballot(lane_state(r) == kRun && !lane_clean(r)) == 0ull;
    if (clean && g.form == kOneRoot) lane_loop<kClean, kOneRoot>(g, r, s_root, root_lds);
    else if (clean && g.form != kIndexed) lane_loop<kClean, kTable>(g, r, s_root, root_lds);
    else if (g.form != kIndexed) lane_loop<kGeneral, kTable>(g, r, s_root, root_lds);
    else lane_loop<kGeneral, kIndexed>(g, r, s_root, root_lds);
}

// cp_main (raycast.comp.wgsl:62-63): dir = normalize(p.x*u + p.y*mv + wp), p = pixel + offset,
// with the camera words u, mv, wp (ComputeState bytes 144..191).
__device__ __forceinline__ void camera_ray(const float *u, const float *mv, const float *wp, float off, uint32_t px,
                                           uint32_t py, float &dx, float &dy, float &dz) {
    const float fx = (float)px + off, fy = (float)py + off;
    const float vx = (fx * u[0] + fy * mv[0]) + wp[0];
    const float vy = (fx * u[1] + fy * mv[1]) + wp[1];
    const float vz = (fx * u[2] + fy * mv[2]) + wp[2];
    const float len = sqrtf((vx * vx + vy * vy) + vz * vz);
    dx = vx / len, dy = vy / len, dz = vz / len;
}

}  // namespace wxk

// A device-resident grid (the opaque wx_grid of the C ABI): the layout's four pools as
// given (root table, node-5 and node-4 records, leaf words), the slot entries and bases made
// of the records, and the addresses the kernels take.
struct wx_grid {
    wxk::GridDev dev;
    wx::DeviceArena arena;  // holds every pool below
    void *mem[4] = {nullptr, nullptr, nullptr, nullptr};
    void *entries[3] = {nullptr, nullptr, nullptr};  // node-5, node-4, bases
    uint64_t bytes = 0;
    int device = 0;
    uint32_t n5 = 0, n4 = 0, n3 = 0;  // node counts of the layout
};
