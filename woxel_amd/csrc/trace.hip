// HDDA + grid-SDF traversal kernels for gfx950, and the device-side C ABI.
//
// The per-lane traversal (RayLane, lane_look, lane_advance) lives in lane.hpp. The launch shapes
// (wx_tune.persistent) share it:
//  * k_simple_*: one lane per ray, 8x8-pixel wave tiles (the reference's dispatch
//    shape); camera tiles dealt round-robin over the XCDs, or in one band per XCD
//    (wx_tune.xcd_split = 2: better L2 locality, worse balance -- measured slower);
//  * k_persist1, k_persist_batch: wave64 workers that refill. Once `refill` lanes of a wave
//    have finished, the idle lanes take new slots: of the wave's fixed share of the one
//    request (also for the scattered sets of a long ray list in the one-lane shape), or of
//    chunks of a batch's work queue (per-XCD regions, with stealing; shadow rays continue
//    in the lane of their primary; one kernel per grid form for a batch on one grid). Every
//    wave exits once its slots are used up and its lanes are idle; every ray ends within 1000
//    steps, so the grid always drains.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "lane.hpp"
#include "request.hpp"
#include "wx_internal.hpp"

using wx::set_error;

namespace {

using namespace wxk;

constexpr uint32_t kRegions = 8u;      // queue regions (one per XCD)
constexpr uint32_t kMaxGridsLds = 64u; // grid table entries staged in LDS
constexpr uint32_t kMaxReqsLds = 1024u;

// ---------------------------------------------------------------- simple shape

// Shadow continuation of a finished primary in the same lane (WX_TRACE_SHADOW).
__device__ __forceinline__ void finish_with_shadow(const GridDev &g, const ReqDev &q, RayLane &r, uint32_t pix,
                                                   const int4 *s_root = nullptr, bool root_lds = false) {
    if (lane_state(r) != WX_HIT) {
        write_no_ray(q.shadow + pix);
        return;
    }
    float ox, oy, oz;
    shadow_origin(r, ox, oy, oz);
    start_shadow(r, q, g.bound, ox, oy, oz);
    lane_run(g, r, s_root, root_lds);
    lane_write(r, ox, oy, oz, q.shadow + pix);
}

// 128-lane workgroups of two wave tiles (8x8 pixels at 64 rays per wave: 16x8 pixels): a
// finished workgroup frees its slots for the next one sooner than a 16x16 one (measured
// faster). lg: rays_per_wave_log2.
template <bool kShadow>
__global__ __launch_bounds__(128) void k_simple_camera(GridDev g, ReqDev q, uint32_t lg, uint32_t band) {
    __shared__ int4 s_root_buf[kRootLds];
    const bool root_lds = stage_root(g, s_root_buf);
    uint32_t bx, by;
    tile_of_block(band != 0u, bx, by);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t lw = (lg + 1u) >> 1, px = ((bx * 2u + wave) << lw) + (lane & ((1u << lw) - 1u));
    const uint32_t py = (by << (lg >> 1)) + (lane >> lw);
    if (lane >> lg || px >= q.w || py >= q.h) return;
    float dx, dy, dz;
    camera_dir(q, px, py, dx, dy, dz);
    RayLane r;
    lane_start(r, q.ex, q.ey, q.ez, dx, dy, dz, g.bound, (q.flags & WX_TRACE_CLIP) != 0u);
    lane_run(g, r, s_root_buf, root_lds);
    const uint32_t pix = py * q.w + px;
    lane_write(r, q.ex, q.ey, q.ez, q.out + pix);
    if (kShadow) finish_with_shadow(g, q, r, pix, s_root_buf, root_lds);
}

// Whether a wave's rays (lanes with `in`, direction (x, y, z)) go the same way: at least
// half of them within about 25 degrees of the first. A scan line, a panorama or a light's
// rays do; of rays that have nothing to do with each other one in twenty does. Every lane
// of the wave calls it.
__device__ __forceinline__ bool rays_together(bool in, float x, float y, float z) {
    auto lead = [](float v) { return __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(v))); };
    const float x0 = lead(x), y0 = lead(y), z0 = lead(z);
    const float c = x * x0 + y * y0 + z * z0;
    const bool near = c > 0.0f && c * c > 0.81f * (x * x + y * y + z * z) * (x0 * x0 + y0 * y0 + z0 * z0);
    return 2u * (uint32_t)__popcll(__ballot(in && near)) >= (uint32_t)__popcll(__ballot(in));
}

// split: only the waves whose rays go together trace theirs, k_persist1 the others'.
template <bool kShadow>
__global__ __launch_bounds__(128) void k_simple_rays(GridDev g, ReqDev q, uint32_t lg, uint32_t split) {
    __shared__ int4 s_root_buf[kRootLds];
    const bool root_lds = stage_root(g, s_root_buf);
    const uint32_t lane = threadIdx.x & 63u, i = ((blockIdx.x * 2u + (threadIdx.x >> 6)) << lg) + lane;
    const float *p = reinterpret_cast<const float *>(q.rays + std::min(i, q.w - 1u));
    const float dx = p[3], dy = p[4], dz = p[5];
    if (split && !rays_together(i < q.w, dx, dy, dz)) return;
    if (lane >> lg || i >= q.w) return;
    RayLane r;
    lane_start(r, p[0], p[1], p[2], dx, dy, dz, g.bound, (q.flags & WX_TRACE_CLIP) != 0u);
    lane_run(g, r, s_root_buf, root_lds);
    lane_write(r, p[0], p[1], p[2], q.out + i);
    if (kShadow) finish_with_shadow(g, q, r, i, s_root_buf, root_lds);
}

// Any batch, one lane per slot: slot s of the launch is request r's slot
// s - begin[r]; a primary hit with WX_TRACE_SHADOW continues as the shadow ray.
struct BatchArgs {
    const GridDev *grids;
    const ReqDev *reqs;
    const uint32_t *begin;
    uint32_t n_grids, n_reqs, total, lg;
};
// The same with the tables among the kernel's arguments, which take 4 KiB at most: a request
// takes 132 bytes and a grid 64, so twice as many requests as grids, 24 on 12, fill them.
// Such a batch needs no copy before the launch: 24 requests of 64x48 on 4 grids 119 us a call
// and 25, by copy, 131; 24 on 12 grids 153 and on 13 167.
constexpr uint32_t kInlineGrids = 12u, kInlineReqs = 24u;
struct BatchInline {
    ReqDev reqs[kInlineReqs];
    GridDev grids[kInlineGrids];
    uint32_t begin[kInlineReqs + 1u];
    uint32_t n_reqs, total, lg;
};
static_assert(sizeof(BatchInline) <= 3968, "kernel arguments");

template <typename Tables>
__global__ __launch_bounds__(128) void k_simple_batch(Tables a) {
    const uint32_t lane = threadIdx.x & 63u, slot = ((blockIdx.x * 2u + (threadIdx.x >> 6)) << a.lg) + lane;
    if (lane >> a.lg || slot >= a.total) return;
    // so the 64 slots of a wave belong to one request: find it once per wave
    const uint32_t wslot = (uint32_t)__builtin_amdgcn_readfirstlane((int)(slot & ~63u));
    uint32_t lo = 0, hi = a.n_reqs;  // slot -> request: binary search over the prefix
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (a.begin[mid] <= wslot) lo = mid;
        else hi = mid;
    }
    lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
    const ReqDev &q = a.reqs[lo];
    const GridDev g = a.grids[q.grid];
    const uint32_t s = slot - a.begin[lo];
    float ox, oy, oz, dx, dy, dz;
    uint32_t pix;
    if (q.kind == WX_REQ_CAMERA) {
        uint32_t px, py;
        if (!camera_pixel(q, s, px, py)) return;
        pix = py * q.w + px;
        ox = q.ex, oy = q.ey, oz = q.ez;
        camera_dir(q, px, py, dx, dy, dz);
    } else {
        if (s >= q.w) return;
        pix = s;
        const float *p = reinterpret_cast<const float *>(q.rays + s);
        ox = p[0], oy = p[1], oz = p[2], dx = p[3], dy = p[4], dz = p[5];
    }
    RayLane r;
    lane_start(r, ox, oy, oz, dx, dy, dz, g.bound, (q.flags & WX_TRACE_CLIP) != 0u);
    lane_run(g, r);
    lane_write(r, ox, oy, oz, q.out + pix);
    if (q.flags & WX_TRACE_SHADOW) finish_with_shadow(g, q, r, pix);
}

// ---------------------------------------------------------------- persistent shape

struct PersistArgs {
    const GridDev *grids;  // n_grids
    const ReqDev *reqs;    // n_reqs
    const uint32_t *begin; // n_reqs + 1 slot prefix (camera: 64 slots per 8x8 tile; rays: one per ray)
    uint32_t *ctr;         // kRegions counters, 16 words apart
    uint32_t n_grids, n_reqs, total, regions;
    uint32_t refill, chunk;
    uint32_t pad[2];
};

__global__ __launch_bounds__(256) void k_zero(uint32_t *p, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += 256u) p[i] = 0u;
}

// Work queue of one persistent wave: chunks of `chunk` slots from the wave's
// queue region (regions are per XCD; a drained region passes the wave on to the
// next one). All values are wave-uniform.
struct WaveQueue {
    uint32_t region, probed, cur, end, regsize;

    __device__ __forceinline__ void init(const PersistArgs &a) {
        regsize = ((a.total + a.regions * 64u - 1u) / (a.regions * 64u)) * 64u;
        region = blockIdx.x % a.regions;  // workgroups are dispatched round-robin over the XCDs
        probed = 0;
        cur = end = 0;
    }
    __device__ __forceinline__ bool drained(const PersistArgs &a) const { return cur == end && probed >= a.regions; }
    // Take the next chunk once the current one is used up.
    __device__ __forceinline__ void fetch(const PersistArgs &a, uint32_t lane) {
        if (cur != end || probed >= a.regions) return;
        for (;;) {
            const uint32_t rs = region * regsize;
            uint32_t got = 0;
            if (lane == 0) got = atomicAdd(&a.ctr[region * 16u], a.chunk);
            got = __builtin_amdgcn_readfirstlane(got);
            const uint32_t re = std::min(rs + regsize, a.total);
            if (got < regsize && rs + got < re) {
                cur = rs + got;
                end = std::min(cur + a.chunk, re);
                return;
            }
            if (++probed >= a.regions) return;
            region = (region + 1u) % a.regions;
        }
    }
};

// Rays of one wave that are started and wait for a lane, in LDS: the wave starts 64 at a
// time on full lanes (direction, reciprocals, entry clip: as many instructions as two
// steps), and idle lanes take from here.
struct ReadyRays {
    float w[12][64];  // position, direction, reciprocal direction, origin
    uint32_t pix[64];
};

// The ray of slot s of a request; false when the slot has none (outside the image).
template <uint32_t KIND>
__device__ __forceinline__ bool slot_ray(const ReqDev &q, uint32_t s, uint32_t &pix, float *o, float *d) {
    if (KIND == WX_REQ_CAMERA) {
        uint32_t px, py;
        if (!camera_pixel(q, s, px, py)) return false;
        pix = py * q.w + px;
        o[0] = q.ex, o[1] = q.ey, o[2] = q.ez;
        camera_dir(q, px, py, d[0], d[1], d[2]);
        return true;
    }
    if (s >= q.w) return false;
    pix = s;
    const float *p = reinterpret_cast<const float *>(q.rays + s);
    o[0] = p[0], o[1] = p[1], o[2] = p[2], d[0] = p[3], d[1] = p[4], d[2] = p[5];
    return true;
}

// One request (camera or ray list), no shadow rays, by n waves that each take every n-th
// set of 64 slots and refill: once `refill` lanes are idle, their records are written
// together and they take new rays. No counters in memory; rays that are not fast
// (lane_fast) wait until the wave's others are done, so that the loop holds the fast step
// of one grid form alone (64 VGPRs, eight waves per SIMD; 103 with the general step beside
// it; the table form spills two to five there, at 72 and seven waves 16.8 M rays on eight
// node-5s take 4022 us instead of 2944). A grid whose bound rules the fast step out goes to the
// one-lane shapes instead (16.8 M rays at bound 2^21: 24.7 ms, here 39.6). With `split` the wave leaves out the sets whose rays go
// together: those lose by refilling, which breaks up their lookups, and by a fixed share per
// wave (16.8 M panorama rays: 2.05 ms one lane per ray, 2.56 refilled, 3.05 in fixed shares
// without refilling), while scattered rays gain, as one lane per ray leaves nine lanes in ten
// idle (16.8 M: 4.22 ms one lane per ray, 1.97 here).
template <uint32_t KIND, uint32_t kForm>
__global__ __launch_bounds__(256, 8) void k_persist1(GridDev g, ReqDev q, uint32_t total, uint32_t refill,
                                                   uint32_t split) {
    __shared__ int4 s_root_buf[kRootLds];
    __shared__ ReadyRays s_ready[4];
    __shared__ float s_org[3][256];
    __shared__ uint32_t s_pix[256], s_start[256];
    const bool root_lds = stage_root(g, s_root_buf);
    const uint32_t lane = threadIdx.x & 63u;
    ReadyRays &ready = s_ready[threadIdx.x >> 6];
    const uint64_t lt = (1ull << lane) - 1ull;
    const bool clip = (q.flags & WX_TRACE_CLIP) != 0u;
    const uint64_t stride = (uint64_t)gridDim.x * 256u, end = total;
    const uint64_t first =
        (uint64_t)blockIdx.x * 256u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x & ~63u));
    uint64_t next = first;
    bool running = false, pending = false, capped = false, slow = false;
    uint32_t n_ready = 0, trip = 0, oldest = 0;
    RayLane r;
    for (;;) {
        if (pending && !running) {  // records of the rays that ended since the last refill
            lane_finish(r, capped);
            lane_write(r, s_org[0][threadIdx.x], s_org[1][threadIdx.x], s_org[2][threadIdx.x], q.out + s_pix[threadIdx.x]);
            pending = false;
        }
        uint32_t n_idle = (uint32_t)__popcll(__ballot(!running));
        while (n_idle) {
            while (!n_ready && next < end) {  // start the next 64 slots; rays that miss the box end here
                const uint32_t s = (uint32_t)next + lane;
                next += stride;
                RayLane f;
                f.state = WX_OOB;
                uint32_t fp = 0;
                float o[3], d[3] = {0.0f, 0.0f, 0.0f};
                const bool in = s < end && slot_ray<KIND>(q, s, fp, o, d);
                if (KIND == WX_REQ_RAYS && split && rays_together(in, d[0], d[1], d[2])) continue;
                if (in) {
                    lane_start(f, o[0], o[1], o[2], d[0], d[1], d[2], g.bound, clip);
                    if (lane_state(f) != kRun) {
                        lane_write(f, o[0], o[1], o[2], q.out + fp);
                    } else if (!lane_fast(f)) {
                        slow = true;
                        f.state = WX_OOB;
                    }
                }
                const uint64_t m = __ballot(lane_state(f) == kRun);
                if (lane_state(f) == kRun) {
                    const uint32_t k = (uint32_t)__popcll(m & lt);
                    ready.w[0][k] = f.px, ready.w[1][k] = f.py, ready.w[2][k] = f.pz;
                    ready.w[3][k] = f.dx, ready.w[4][k] = f.dy, ready.w[5][k] = f.dz;
                    ready.w[6][k] = f.ix, ready.w[7][k] = f.iy, ready.w[8][k] = f.iz;
                    ready.w[9][k] = o[0], ready.w[10][k] = o[1], ready.w[11][k] = o[2];
                    ready.pix[k] = fp;
                }
                n_ready = (uint32_t)__popcll(m);
                // the wave's own LDS accesses stay in order; this keeps the compiler to it
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
            if (!n_ready) break;
            const uint32_t take = std::min(n_idle, n_ready);
            const uint32_t rank = (uint32_t)__popcll(__ballot(!running) & lt);
            if (!running && rank < take) {
                const uint32_t k = n_ready - 1u - rank;
                lane_resume(r, ready.w[0][k], ready.w[1][k], ready.w[2][k], ready.w[3][k], ready.w[4][k],
                            ready.w[5][k], ready.w[6][k], ready.w[7][k], ready.w[8][k]);
                for (uint32_t c = 0; c < 3u; ++c) s_org[c][threadIdx.x] = ready.w[9u + c][k];
                s_pix[threadIdx.x] = ready.pix[k];
                s_start[threadIdx.x] = trip;
                capped = false;
                running = pending = true;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            n_ready -= take;
            n_idle -= take;
        }
        if (!__any(running)) break;  // every slot is started and no fast ray is left
        // no running ray started before trip `oldest`, so none meets the step cap before
        // trip oldest + kMaxSteps
        if (trip - oldest > kMaxSteps / 2u) {
            uint32_t m = running ? trip - s_start[threadIdx.x] : 0u;
            for (int d = 1; d < 64; d <<= 1) m = std::max(m, (uint32_t)__shfl_xor((int)m, d));
            oldest = trip - (uint32_t)__builtin_amdgcn_readfirstlane((int)m);
        }
        const uint32_t keep = n_idle ? 0u : 64u - refill;  // idle lanes: there are no more slots
        do {
            ++trip;
            if (running) {
                running = lane_look<kFast, kForm>(g, r, s_root_buf, root_lds);
                if (running) lane_advance<kFast>(r);
            }
            if (trip - oldest >= kMaxSteps && running && trip - s_start[threadIdx.x] == kMaxSteps)
                capped = true, running = false;
        } while ((uint32_t)__popcll(__ballot(running)) > keep);
    }
    if (!__any(slow)) return;
    for (next = first; next < end; next += stride) {  // the rays that were left out, set by set
        const uint32_t s = (uint32_t)next + lane;
        uint32_t pix;
        float o[3], d[3] = {0.0f, 0.0f, 0.0f};
        const bool in = s < end && slot_ray<KIND>(q, s, pix, o, d);
        if (KIND == WX_REQ_RAYS && split && rays_together(in, d[0], d[1], d[2])) continue;
        if (!in) continue;
        lane_start(r, o[0], o[1], o[2], d[0], d[1], d[2], g.bound, clip);
        if (lane_state(r) != kRun || lane_fast(r)) continue;
        lane_loop<kGeneral, kForm == kIndexed ? kIndexed : kTable>(g, r, s_root_buf, root_lds);
        lane_write(r, o[0], o[1], o[2], q.out + pix);
    }
}

// Any batch: many requests and grids, shadow rays continued in the lane of
// their primary. Ray origins live in LDS (one per lane); the 128-byte request record is read
// when a ray starts or ends. kForm is the form of the batch's only grid, whose descriptor is
// then an argument, or kMixed: lanes trace different grids, keep theirs as an index and
// read its descriptor from LDS on each step. The general step alone: lanes here are at
// different depths and enter every region of a step, so the fast step gained less than the
// registers of both lost (112, four waves per SIMD; 96 with one, five for one grid). Measured
// against both steps and per-lane descriptors for one grid: a shadowed 1080p request
// 2800 -> 2440 us, 12 of 640x360 1445 -> 1330 (16 waves per CU), on eight node-5s 3340 -> 2890.
constexpr uint32_t kMixed = 3u;
template <uint32_t kForm>
__global__ __launch_bounds__(256, kForm == kMixed ? 4 : 5) void k_persist_batch(PersistArgs a, GridDev one) {
    constexpr bool mixed = kForm == kMixed;
    __shared__ GridDev s_grid[mixed ? kMaxGridsLds : 1u];
    __shared__ uint32_t s_begin[kMaxReqsLds + 1];
    __shared__ float s_org[3][256];
    if (mixed)
        for (uint32_t i = threadIdx.x; i < a.n_grids; i += 256u) s_grid[i] = a.grids[i];
    for (uint32_t i = threadIdx.x; i <= a.n_reqs; i += 256u) s_begin[i] = a.begin[i];
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t lt = (1ull << lane) - 1ull;
    WaveQueue wq;
    wq.init(a);
    bool alive = false, shadow = false;
    uint32_t req = 0, gi = 0, pix = 0, it = 0;
    RayLane r;
    r.state = 0;
    for (;;) {
        const uint64_t idle = __ballot(!alive);
        const uint32_t nidle = (uint32_t)__popcll(idle);
        if (nidle >= a.refill) {
            wq.fetch(a, lane);
            const uint32_t avail = wq.end - wq.cur;
            const uint32_t rank = (uint32_t)__popcll(idle & lt);
            if (!alive && rank < avail) {
                const uint32_t slot = wq.cur + rank;
                uint32_t lo = 0, hi = a.n_reqs;  // slot -> request: binary search over the prefix
                while (hi - lo > 1u) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (s_begin[mid] <= slot) lo = mid;
                    else hi = mid;
                }
                const ReqDev &q = a.reqs[lo];
                const uint32_t s = slot - s_begin[lo];
                bool ok;
                float ox, oy, oz, dx, dy, dz;
                if (q.kind == WX_REQ_CAMERA) {
                    uint32_t px, py;
                    ok = camera_pixel(q, s, px, py);
                    pix = py * q.w + px;
                    ox = q.ex, oy = q.ey, oz = q.ez;
                    if (ok) camera_dir(q, px, py, dx, dy, dz);
                } else {
                    ok = s < q.w;
                    pix = s;
                    if (ok) {
                        const float *p = reinterpret_cast<const float *>(q.rays + s);
                        ox = p[0], oy = p[1], oz = p[2], dx = p[3], dy = p[4], dz = p[5];
                    }
                }
                if (ok) {
                    gi = q.grid;
                    lane_start(r, ox, oy, oz, dx, dy, dz, mixed ? s_grid[gi].bound : one.bound, (q.flags & WX_TRACE_CLIP) != 0u);
                    s_org[0][threadIdx.x] = ox, s_org[1][threadIdx.x] = oy, s_org[2][threadIdx.x] = oz;
                    req = lo;
                    it = 0;
                    shadow = false;
                    alive = true;
                }
            }
            wq.cur += std::min(avail, nidle);
        }
        if (!__any(alive)) {
            if (wq.drained(a)) break;
            continue;
        }
        if (alive) {
            const GridDev &g = mixed ? s_grid[gi] : one;
            if (lane_state(r) == kRun) {
                ++it;
                auto step = [&](auto look, auto advance) {
                    const bool on = look(g, r, nullptr, false);
                    if (on) advance(r);
                    if (!on || it == kMaxSteps) lane_finish(r, on);
                };
                if constexpr (!mixed) step(lane_look<kGeneral, kForm>, lane_advance<kGeneral>);
                else if (g.form == kIndexed) step(lane_look<kGeneral, kIndexed>, lane_advance<kGeneral>);
                else step(lane_look<kGeneral, kTable>, lane_advance<kGeneral>);
            }
            if (lane_state(r) != kRun) {
                const ReqDev &q = a.reqs[req];
                const float ox = s_org[0][threadIdx.x], oy = s_org[1][threadIdx.x], oz = s_org[2][threadIdx.x];
                lane_write(r, ox, oy, oz, (shadow ? q.shadow : q.out) + pix);
                alive = false;
                if (!shadow && (q.flags & WX_TRACE_SHADOW)) {
                    if (lane_state(r) == WX_HIT) {
                        float sx, sy, sz;
                        shadow_origin(r, sx, sy, sz);
                        start_shadow(r, q, g.bound, sx, sy, sz);
                        s_org[0][threadIdx.x] = sx, s_org[1][threadIdx.x] = sy, s_org[2][threadIdx.x] = sz;
                        it = 0;
                        shadow = true;
                        alive = true;
                        if (lane_state(r) != kRun) {  // the shadow ray missed the bound box
                            lane_write(r, sx, sy, sz, q.shadow + pix);
                            alive = false;
                        }
                    } else {
                        write_no_ray(q.shadow + pix);
                    }
                }
            }
        }
    }
}

template <uint32_t KIND>
void launch_persist1(uint32_t blocks, hipStream_t stream, const GridDev &g, const ReqDev &q, uint32_t total,
                     uint32_t refill, uint32_t split) {
    const dim3 n(blocks), t(256);
    if (g.form == kOneRoot) hipLaunchKernelGGL((k_persist1<KIND, kOneRoot>), n, t, 0, stream, g, q, total, refill, split);
    else if (g.form == kTable) hipLaunchKernelGGL((k_persist1<KIND, kTable>), n, t, 0, stream, g, q, total, refill, split);
    else hipLaunchKernelGGL((k_persist1<KIND, kIndexed>), n, t, 0, stream, g, q, total, refill, split);
}

int hip_fail(hipError_t e, const char *what) {
    return set_error(WX_ERR_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

// ---------------------------------------------------------------- per-stream scratch

// Device scratch for one stream: queue counters + the batch tables, and a pinned
// host staging buffer for the tables. Launches on one stream are ordered, so a
// stream's scratch is never used by two launches at once (callers that share a
// stream between threads serialise their calls on it, as for any stream).
struct StreamScratch {
    void *dev = nullptr;
    size_t dev_cap = 0;
    void *host = nullptr;
    size_t host_cap = 0;
    hipEvent_t copied = nullptr;  // the last table upload from `host` is done
    bool pending = false;
};

std::mutex g_scratch_mu;
std::map<std::pair<int, void *>, StreamScratch> g_scratch;

int scratch_for(hipStream_t s, size_t dev_bytes, size_t host_bytes, StreamScratch **out) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    StreamScratch &S = g_scratch[{dev, (void *)s}];
    if (S.pending) {
        hipError_t e = hipEventSynchronize(S.copied);
        if (e != hipSuccess) return hip_fail(e, "scratch: event sync");
        S.pending = false;
    }
    if (S.dev_cap < dev_bytes) {
        if (S.dev) {
            hipError_t e = hipStreamSynchronize(s);
            if (e != hipSuccess) return hip_fail(e, "scratch: stream sync");
            (void)hipFree(S.dev);
        }
        size_t cap = std::max<size_t>(dev_bytes, 64u << 10);
        hipError_t e = hipMalloc(&S.dev, cap);
        if (e != hipSuccess) {
            S.dev = nullptr;
            S.dev_cap = 0;
            return set_error(WX_ERR_BUDGET, std::string("scratch: hipMalloc: ") + hipGetErrorString(e));
        }
        S.dev_cap = cap;
    }
    if (S.host_cap < host_bytes) {
        if (S.host) (void)hipHostFree(S.host);
        size_t cap = std::max<size_t>(host_bytes, 64u << 10);
        hipError_t e = hipHostMalloc(&S.host, cap, hipHostMallocDefault);
        if (e != hipSuccess) {
            S.host = nullptr;
            S.host_cap = 0;
            return set_error(WX_ERR_BUDGET, std::string("scratch: hipHostMalloc: ") + hipGetErrorString(e));
        }
        S.host_cap = cap;
    }
    if (!S.copied) {
        hipError_t e = hipEventCreateWithFlags(&S.copied, hipEventDisableTiming);
        if (e != hipSuccess) return hip_fail(e, "scratch: event");
    }
    *out = &S;
    return WX_OK;
}

}  // namespace

// Frees the scratch of a stream about to be destroyed (its work is waited for).
void wx::drop_stream_scratch(void *stream) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    for (auto it = g_scratch.begin(); it != g_scratch.end();) {
        if (it->first.second != stream) {
            ++it;
            continue;
        }
        StreamScratch &S = it->second;
        (void)hipStreamSynchronize(static_cast<hipStream_t>(stream));
        if (S.dev) (void)hipFree(S.dev);
        if (S.host) (void)hipHostFree(S.host);
        if (S.copied) (void)hipEventDestroy(S.copied);
        it = g_scratch.erase(it);
    }
}

namespace {

// ---------------------------------------------------------------- tuning

std::mutex g_tune_mu;
std::map<int, wx_tune> g_tune;

wx_tune default_tune() {
    wx_tune t;
    t.persistent = 0;
    t.refill = 16;
    t.chunk = 256;
    t.waves_per_cu = 16;
    t.xcd_split = 1;
    return t;
}

wx_tune current_tune() {
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune.find(dev);
    return it == g_tune.end() ? default_tune() : it->second;
}

bool tune_ok(const wx_tune &t) {
    return t.persistent <= 3 && t.refill >= 1 && t.refill <= 64 && t.chunk >= 64 && t.chunk % 64 == 0 && t.chunk <= (1u << 20) &&
           t.waves_per_cu >= 1 && t.waves_per_cu <= 32 && t.xcd_split <= 2;
}

}  // namespace

// CUs of the current device, queried once per device; no lock and no allocation, as the
// allocation-free launches ask too.
int wx::cu_count() {
    static std::atomic<int> cus[16];
    int dev = 0, n = 0;
    (void)hipGetDevice(&dev);
    std::atomic<int> *const known = dev >= 0 && dev < 16 ? &cus[dev] : nullptr;
    if (known && (n = known->load(std::memory_order_relaxed)) > 0) return n;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    if (known) known->store(n, std::memory_order_relaxed);
    return n;
}

namespace {

// Host request -> device request; checks everything the kernel indexes with.
int make_req(const wx_request &in, uint32_t n_grids, ReqDev &q, uint32_t &slots) {
    std::memset(&q, 0, sizeof q);
    if (in.grid >= n_grids) return set_error(WX_ERR_INVALID, "request: grid index out of range");
    if (in.kind != WX_REQ_CAMERA && in.kind != WX_REQ_RAYS) return set_error(WX_ERR_INVALID, "request: bad kind");
    if (in.flags & ~(WX_TRACE_CLIP | WX_TRACE_SHADOW)) return set_error(WX_ERR_INVALID, "request: unknown flags");
    if (!in.out && in.width && in.height) return set_error(WX_ERR_INVALID, "request: NULL output buffer");
    if ((in.flags & WX_TRACE_SHADOW) && !in.shadow_out && in.width && in.height)
        return set_error(WX_ERR_INVALID, "request: SHADOW without a shadow output buffer");
    q.kind = in.kind;
    q.grid = in.grid;
    q.flags = in.flags;
    q.out = in.out;
    q.shadow = in.shadow_out;
    q.lx = in.light[0], q.ly = in.light[1], q.lz = in.light[2];
    if (in.kind == WX_REQ_CAMERA) {
        if (in.width > 65536u || in.height > 65536u) return set_error(WX_ERR_INVALID, "request: image too large");
        q.w = in.width;
        q.h = in.height;
        q.tiles_x = (in.width + 7u) / 8u;
        const uint64_t tiles = (uint64_t)q.tiles_x * ((in.height + 7u) / 8u);
        if (tiles * 64u > 0x7FFFFFFFull) return set_error(WX_ERR_INVALID, "request: image too large");
        slots = (uint32_t)(tiles * 64u);
        q.off = in.pixel_offset;
        q.ex = in.camera.eye[0], q.ey = in.camera.eye[1], q.ez = in.camera.eye[2];
        q.ux = in.camera.u[0], q.uy = in.camera.u[1], q.uz = in.camera.u[2];
        q.mx = in.camera.mv[0], q.my = in.camera.mv[1], q.mz = in.camera.mv[2];
        q.wx = in.camera.wp[0], q.wy = in.camera.wp[1], q.wz = in.camera.wp[2];
        if (!in.width || !in.height) slots = 0;
    } else {
        if (!in.rays && in.width) return set_error(WX_ERR_INVALID, "request: NULL ray buffer");
        if (in.width > 0x7FFFFFC0u) return set_error(WX_ERR_INVALID, "request: too many rays");
        q.w = in.width;
        q.h = 1;
        q.rays = in.rays;
        slots = (in.width + 63u) & ~63u;
    }
    return WX_OK;
}

// Table layout of a batched launch in its scratch memory: queue counters, then the
// grid table, the request table and the slot prefix, packed.
constexpr size_t kOffCtr = 0, kOffGrids = 1024;
constexpr size_t off_reqs(uint32_t n_grids) { return kOffGrids + sizeof(GridDev) * n_grids; }
constexpr size_t off_begin(uint32_t n_grids, uint32_t n_reqs) { return off_reqs(n_grids) + sizeof(ReqDev) * n_reqs; }
constexpr size_t table_bytes(uint32_t n_grids, uint32_t n_reqs) {
    return off_begin(n_grids, n_reqs) + 4u * (n_reqs + 1u);
}

// Allocation-free launches (wx_trace_batch_static) keep the same tables in a
// file-scope device array, one copy per GPU, sized for the largest batch a launch
// takes. Host code reaches it through the address hipGetSymbolAddress returns on
// each device, never through the array's name.
constexpr size_t kStaticBytes = (table_bytes(kMaxGridsLds, kMaxReqsLds) + 255u) & ~size_t(255);
__device__ __align__(256) unsigned char scratch[kStaticBytes];

constexpr int kMaxStaticDevices = 16;
std::mutex g_static_mu;
void *g_static_dev[kMaxStaticDevices];  // scratch's address on each device (nullptr until first use)
// Host staging of the tables, one area per device. The tables are copied with
// hipMemcpyAsync from this pageable memory, which the runtime has consumed when
// the call returns, so the next call on the device may overwrite it.
alignas(256) unsigned char g_static_host[kMaxStaticDevices][kStaticBytes];

// The current device's static scratch (device address, host staging).
int static_scratch(char **dev_out, char **host_out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return set_error(WX_ERR_DEVICE, std::string("static scratch: ") + hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxStaticDevices)
        return set_error(WX_ERR_UNSUPPORTED, "static scratch: device ordinal beyond 15");
    std::lock_guard<std::mutex> lk(g_static_mu);
    if (!g_static_dev[dev]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return set_error(WX_ERR_DEVICE, std::string("static scratch: hipGetSymbolAddress: ") + hipGetErrorString(e));
        g_static_dev[dev] = ptr;
    }
    *dev_out = static_cast<char *>(g_static_dev[dev]);
    *host_out = reinterpret_cast<char *>(g_static_host[dev]);
    return WX_OK;
}

// Where a launch's tables and counters live: per-stream scratch that grows on
// demand (wx_trace_batch) or the device's static scratch (wx_trace_batch_static).
struct Staging {
    bool is_static = false;
    char *host = nullptr;  // static: host staging area; tables are built in place
    char *dev = nullptr;   // static: device scratch
};

// Copies the grid table and the request/prefix tables (already at their packed
// offsets in `host`) to the device scratch `dev` and returns their device addresses.
int copy_tables(wx_grid *const *grids, uint32_t n_grids, uint32_t n_reqs, char *host, char *dev, hipStream_t stream,
                const GridDev **g_out, const ReqDev **q_out, const uint32_t **b_out) {
    for (uint32_t i = 0; i < n_grids; ++i)
        std::memcpy(host + kOffGrids + sizeof(GridDev) * i, &grids[i]->dev, sizeof(GridDev));
    const size_t bytes = table_bytes(n_grids, n_reqs);
    hipError_t e = hipMemcpyAsync(dev + kOffGrids, host + kOffGrids, bytes - kOffGrids, hipMemcpyHostToDevice, stream);
    if (e != hipSuccess) return hip_fail(e, "batch: table upload");
    *g_out = reinterpret_cast<const GridDev *>(dev + kOffGrids);
    *q_out = reinterpret_cast<const ReqDev *>(dev + off_reqs(n_grids));
    *b_out = reinterpret_cast<const uint32_t *>(dev + off_begin(n_grids, n_reqs));
    return WX_OK;
}

// Upload the grid/request/prefix tables of a batch into the stream's scratch
// (after the counter block) and return their device addresses.
int upload_tables(wx_grid *const *grids, uint32_t n_grids, const ReqDev *q, const uint32_t *begin, uint32_t n_reqs,
                  hipStream_t stream, StreamScratch **S_out, const GridDev **g_out, const ReqDev **q_out,
                  const uint32_t **b_out) {
    const size_t bytes = table_bytes(n_grids, n_reqs);
    StreamScratch *S = nullptr;
    int rc = scratch_for(stream, bytes, bytes, &S);
    if (rc) return rc;
    char *h = static_cast<char *>(S->host);
    std::memcpy(h + off_reqs(n_grids), q, sizeof(ReqDev) * n_reqs);
    std::memcpy(h + off_begin(n_grids, n_reqs), begin, 4u * (n_reqs + 1u));
    rc = copy_tables(grids, n_grids, n_reqs, h, static_cast<char *>(S->dev), stream, g_out, q_out, b_out);
    if (rc) return rc;
    if (hipEventRecord(S->copied, stream) != hipSuccess) return set_error(WX_ERR_DEVICE, "batch: event record");
    S->pending = true;
    *S_out = S;
    return WX_OK;
}

// A batch, validated and launched in the shape `t` selects. may_split: a long ray list may
// go to two kernels. With a static
// staging the tables are built directly in the device's host staging area and no
// memory is allocated.
int launch_batch(wx_grid *const *grids, uint32_t n_grids, const wx_request *reqs, uint32_t n_reqs,
                 const wx_tune &t, hipStream_t stream, const Staging &stg = Staging(), bool may_split = true) {
    if (!tune_ok(t)) return set_error(WX_ERR_INVALID, "tune: out of range");
    std::vector<ReqDev> qv;
    std::vector<uint32_t> bv;
    ReqDev *q;
    uint32_t *begin;
    if (stg.is_static) {
        if (n_grids > kMaxGridsLds || n_reqs > kMaxReqsLds)
            return set_error(WX_ERR_INVALID, "batch: at most 64 grids and 1024 requests per allocation-free call");
        q = reinterpret_cast<ReqDev *>(stg.host + off_reqs(n_grids));
        begin = reinterpret_cast<uint32_t *>(stg.host + off_begin(n_grids, n_reqs));
    } else {
        qv.resize(n_reqs);
        bv.resize(n_reqs + 1u);
        q = qv.data();
        begin = bv.data();
    }
    uint64_t total = 0;
    for (uint32_t i = 0; i < n_reqs; ++i) {
        uint32_t slots = 0;
        int rc = make_req(reqs[i], n_grids, q[i], slots);
        if (rc) return rc;
        begin[i] = (uint32_t)total;
        total += slots;
        if (total > 0x7FFFFFFFull) return set_error(WX_ERR_INVALID, "batch: more than 2^31 ray slots");
    }
    begin[n_reqs] = (uint32_t)total;
    if (total == 0) return WX_OK;
    for (uint32_t i = 0; i < n_grids; ++i)
        if (!grids[i]) return set_error(WX_ERR_INVALID, "batch: NULL grid");
    const bool one = n_reqs == 1u && n_grids == 1u;
    const bool single = one && !(q[0].flags & WX_TRACE_SHADOW);
    if (!one && (n_grids > kMaxGridsLds || n_reqs > kMaxReqsLds))
        return set_error(WX_ERR_INVALID, "batch: at most 64 grids and 1024 requests per launch");
    // device tables of a multi-request launch
    auto tables = [&](const GridDev **g_out, const ReqDev **q_out, const uint32_t **b_out, uint32_t **ctr) -> int {
        if (stg.is_static) {
            *ctr = reinterpret_cast<uint32_t *>(stg.dev + kOffCtr);
            return copy_tables(grids, n_grids, n_reqs, stg.host, stg.dev, stream, g_out, q_out, b_out);
        }
        StreamScratch *S = nullptr;
        int rc = upload_tables(grids, n_grids, q, begin, n_reqs, stream, &S, g_out, q_out, b_out);
        if (rc) return rc;
        *ctr = reinterpret_cast<uint32_t *>(S->dev);
        return WX_OK;
    };
    hipError_t e;
    const uint32_t cus = (uint32_t)wx::cu_count();
    bool fast = true;  // every grid's bound allows the fast step
    for (uint32_t i = 0; i < n_grids; ++i) fast = fast && grids[i]->dev.bound <= kFastBound;
    if (t.persistent != 1u || (single && !fast)) {  // the one-lane shape
        if (one) {
            const bool sh = (q[0].flags & WX_TRACE_SHADOW) != 0u;
            if (q[0].kind == WX_REQ_CAMERA) {
                const uint32_t lg = rays_per_wave_log2(total, cus, fast), lw = 1u + ((lg + 1u) >> 1), lh = lg >> 1;
                dim3 grid((q[0].w + (1u << lw) - 1u) >> lw, (q[0].h + (1u << lh) - 1u) >> lh, 1);
                const uint32_t band = t.xcd_split == 2u ? 1u : 0u;  // XCD-banded tile order
                if (sh) hipLaunchKernelGGL(k_simple_camera<true>, grid, dim3(128), 0, stream, grids[0]->dev, q[0], lg, band);
                else hipLaunchKernelGGL(k_simple_camera<false>, grid, dim3(128), 0, stream, grids[0]->dev, q[0], lg, band);
            } else {
                // split: the sets of 64 rays that scatter go to k_persist1, the others stay
                const ListShape list = list_shape(q[0].w, cus, fast);
                const uint32_t lg = list.lg, split = list.split && may_split && !sh ? 1u : 0u;
                dim3 grid((q[0].w + (2u << lg) - 1u) >> (lg + 1u));
                if (sh) hipLaunchKernelGGL(k_simple_rays<true>, grid, dim3(128), 0, stream, grids[0]->dev, q[0], lg, 0u);
                else hipLaunchKernelGGL(k_simple_rays<false>, grid, dim3(128), 0, stream, grids[0]->dev, q[0], lg, split);
                if (split) {
                    const uint32_t sets = (q[0].w + 63u) / 64u, most = cus * 32u;
                    const uint32_t per_wave = (sets + most - 1u) / most;
                    launch_persist1<WX_REQ_RAYS>((sets + 4u * per_wave - 1u) / (4u * per_wave), stream, grids[0]->dev, q[0],
                                                 q[0].w, 24u, 1u);
                }
            }
        } else {
            const uint32_t lg = rays_per_wave_log2(total, cus, fast);
            const dim3 grid((uint32_t)((total + (2u << lg) - 1u) >> (lg + 1u)));
            if (n_reqs <= kInlineReqs && n_grids <= kInlineGrids) {
                BatchInline b;
                std::memcpy(b.reqs, q, sizeof(ReqDev) * n_reqs);
                std::memcpy(b.begin, begin, 4u * (n_reqs + 1u));
                for (uint32_t i = 0; i < n_grids; ++i) b.grids[i] = grids[i]->dev;
                b.n_reqs = n_reqs;
                b.total = (uint32_t)total;
                b.lg = lg;
                hipLaunchKernelGGL(k_simple_batch<BatchInline>, grid, dim3(128), 0, stream, b);
            } else {
                BatchArgs b;
                std::memset(&b, 0, sizeof b);
                uint32_t *ctr = nullptr;
                int rc = tables(&b.grids, &b.reqs, &b.begin, &ctr);
                if (rc) return rc;
                b.n_grids = n_grids;
                b.n_reqs = n_reqs;
                b.total = (uint32_t)total;
                b.lg = lg;
                hipLaunchKernelGGL(k_simple_batch<BatchArgs>, grid, dim3(128), 0, stream, b);
            }
        }
        e = hipGetLastError();
        if (e != hipSuccess) return hip_fail(e, "batch: launch");
        return WX_OK;
    }
    if (single) {
        // as many waves as asked for at most, each with the same number of sets of 64 slots
        const uint64_t sets = total / 64u, most = (uint64_t)cus * t.waves_per_cu;
        const uint64_t per_wave = (sets + most - 1u) / most;
        const uint32_t blocks = (uint32_t)(((sets + per_wave - 1u) / per_wave + 3u) / 4u);
        if (q[0].kind == WX_REQ_CAMERA)
            launch_persist1<WX_REQ_CAMERA>(blocks, stream, grids[0]->dev, q[0], (uint32_t)total, t.refill, 0u);
        else
            launch_persist1<WX_REQ_RAYS>(blocks, stream, grids[0]->dev, q[0], q[0].w, t.refill, 0u);
    } else {
        PersistArgs a;
        std::memset(&a, 0, sizeof a);
        a.n_grids = n_grids;
        a.n_reqs = n_reqs;
        a.total = (uint32_t)total;
        a.regions = t.xcd_split ? kRegions : 1u;
        a.refill = t.refill;
        a.chunk = t.chunk;
        int rc = tables(&a.grids, &a.reqs, &a.begin, &a.ctr);
        if (rc) return rc;
        // the queue counters start at zero: a fill kernel (no memset node, so the launch
        // sequence stays valid inside a captured graph)
        hipLaunchKernelGGL(k_zero, dim3(1), dim3(256), 0, stream, a.ctr, 16u * kRegions);
        const uint32_t blocks = std::max<uint32_t>(1u, cus * t.waves_per_cu / 4u);
        const dim3 n(blocks), th(256);
        const GridDev &g = grids[0]->dev;
        if (n_grids != 1u) hipLaunchKernelGGL(k_persist_batch<kMixed>, n, th, 0, stream, a, g);
        else if (g.form == kOneRoot) hipLaunchKernelGGL(k_persist_batch<kOneRoot>, n, th, 0, stream, a, g);
        else if (g.form == kTable) hipLaunchKernelGGL(k_persist_batch<kTable>, n, th, 0, stream, a, g);
        else hipLaunchKernelGGL(k_persist_batch<kIndexed>, n, th, 0, stream, a, g);
    }
    e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "batch: launch");
    return WX_OK;
}

// Slot entries of the node pools (lane.hpp) from the layout's records: one record per
// lane, its 8 (node-5) or 16 (node-4) slots written as 16-byte words. base[node],
// which is kWalk less than the node's first child, is taken off the child indices of compact
// (2-byte) entries; base NULL makes 4-byte entries. Bound
// by the entries written.
template <int kSlots>
__global__ __launch_bounds__(256) void k_expand(const uint4 *rec, uint64_t n, const uint32_t *base, int base_step,
                                                uint4 *out) {
    constexpr uint32_t kBits = 64u / kSlots, kMask = (1u << kBits) - 1u, kNodeRecs = kSlots == 8 ? 4096u : 256u;
    constexpr float kVoxels = kSlots == 8 ? 128.0f : 8.0f;
    for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) {
        const uint4 q = rec[i];
        const uint64_t dist = (uint64_t)q.w << 32 | q.z;
        const uint32_t off = base ? base[(int64_t)(i / kNodeRecs) * base_step] : 0u;
        uint32_t e[kSlots];
#pragma unroll
        for (uint32_t b = 0; b < (uint32_t)kSlots; ++b) {
            const uint32_t size = __float_as_uint((float)(uint32_t)((dist >> (b * kBits)) & kMask) * kVoxels);
            const uint32_t child = q.y - off + (uint32_t)__builtin_popcount(q.x & ((1u << b) - 1u));
            const bool walk = (q.x >> (kSlots + b)) & 1u;
            e[b] = base ? (walk ? child : size >> 16) : (walk ? kWalk32 | child : size);  // base holds kWalk off
        }
        if (base) {
#pragma unroll
            for (uint32_t b = 0; b < (uint32_t)kSlots / 8u; ++b)
                out[i * (kSlots / 8u) + b] =
                    make_uint4(e[8u * b] | e[8u * b + 1u] << 16, e[8u * b + 2u] | e[8u * b + 3u] << 16,
                               e[8u * b + 4u] | e[8u * b + 5u] << 16, e[8u * b + 6u] | e[8u * b + 7u] << 16);
        } else {
#pragma unroll
            for (uint32_t b = 0; b < (uint32_t)kSlots / 4u; ++b)
                out[i * (kSlots / 4u) + b] = make_uint4(e[4u * b], e[4u * b + 1u], e[4u * b + 2u], e[4u * b + 3u]);
        }
    }
}

// Every index the kernels derive from a descriptor stays inside its pool: root
// entries name a node-5 below n5; a record that can be walked into has its walk
// bits inside its child bits, and its first child plus its child count is at most
// the child pool's size (the child of slot b is first + popcount(kids below b)).
// Records are checked in parallel on the host; returns the first bad one. base receives
// the entries' bases (GridDev::base: n5 in reverse, then n4) -- the least child index a
// node's records walk into, less kWalk -- and compact whether every rank from there fits its entry.
int check_desc(const wx_grid_desc *d, const char *who, std::vector<uint32_t> &base, bool &compact) {
    base.assign((size_t)d->n5 + d->n4, 0u - kWalk);
    compact = true;
    for (uint32_t k = 0; k < d->n5; ++k) {
        const int32_t idx = d->root[4u * k + 3u];
        if (idx < 0 || (uint32_t)idx >= d->n5)
            return set_error(WX_ERR_INVALID, std::string(who) + ": root entry " + std::to_string(k) +
                                                 " names node-5 " + std::to_string(idx) + " of " +
                                                 std::to_string(d->n5));
    }
    struct Level {
        const uint32_t *rec;
        uint64_t n;
        uint32_t kid_bits, child_pool;
        const char *name;
    };
    const Level lv[2] = {{d->n5_records, (uint64_t)d->n5 * 4096u, 8u, d->n4, "node-5"},
                         {d->n4_records, (uint64_t)d->n4 * 256u, 16u, d->n3, "node-4"}};
    for (const Level &L : lv) {
        if (!L.n) continue;
        const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
        const uint64_t parts = std::min<uint64_t>(std::min<unsigned>(hw, 16u), (L.n + 65535u) / 65536u);
        const uint64_t node_recs = L.kid_bits == 8u ? 4096u : 256u, nodes = L.n / node_recs;
        std::vector<uint64_t> bad(parts, ~0ull), irregular(parts, 0u);
        auto scan = [&](uint64_t p) {
            const uint32_t km = (1u << L.kid_bits) - 1u;
            for (uint64_t node = nodes * p / parts; node < nodes * (p + 1u) / parts; ++node) {
                uint64_t least = ~0ull, end = 0;
                for (uint64_t i = node * node_recs; i < (node + 1u) * node_recs; ++i) {
                    const uint32_t w = L.rec[4u * i], first = L.rec[4u * i + 1u];
                    const uint32_t kids = w & km, walk = (w >> L.kid_bits) & km;
                    if (!walk) continue;
                    const uint64_t last = (uint64_t)first + (uint64_t)__builtin_popcount(kids);
                    if ((walk & ~kids) || last > L.child_pool) {
                        bad[p] = i;
                        return;
                    }
                    least = std::min<uint64_t>(least, first);
                    end = std::max(end, last);
                }
                if (least == ~0ull) continue;
                base[L.kid_bits == 8u ? d->n5 - 1u - node : d->n5 + node] = (uint32_t)least - kWalk;
                if (end - least > node_recs * L.kid_bits) irregular[p] = 1u;
            }
        };
        if (parts <= 1u) {
            scan(0);
        } else {
            std::vector<std::thread> th;
            for (uint64_t p = 0; p < parts; ++p) th.emplace_back(scan, p);
            for (auto &t : th) t.join();
        }
        for (uint64_t b : bad)
            if (b != ~0ull)
                return set_error(WX_ERR_INVALID, std::string(who) + ": " + L.name + " record " +
                                                     std::to_string(b) + " walks into a child outside the pool");
        for (uint64_t b : irregular) compact = compact && !b;
    }
    return WX_OK;
}

int trace_one(wx_grid *g, const wx_request &in, uint32_t flags, hipStream_t stream) {
    wx_grid *gs[1] = {g};
    wx_tune t = current_tune();
    if (flags & WX_TRACE_SIMPLE) t.persistent = 0;
    return launch_batch(gs, 1, &in, 1, t, stream, Staging(), !(flags & WX_TRACE_SIMPLE));
}

}  // namespace

namespace wx {

// Checks the descriptor, allocates the grid's four pools and copies the root table,
// the node records and, when d->leaves is set, the leaf words from the host; with
// d->leaves NULL the leaf pool is left for the caller to fill. `who` prefixes errors.
int grid_new(const wx_grid_desc *d, const char *who, wx_grid **out) {
    const std::string w(who);
    if ((d->n5 && !d->root) || (d->n5 && !d->n5_records) || (d->n4 && !d->n4_records))
        return set_error(WX_ERR_INVALID, w + ": NULL pool with a non-zero count");
    // the general step's quotient (lane.hpp) needs |p| <= 2^100 after the bound test
    if (!(d->bound > 0.0f) || !(d->bound <= 0x1p100f))
        return set_error(WX_ERR_INVALID, w + ": bound must be in (0, 2^100]");
    // at most 4 GiB of records per node level
    if (d->n5 > (1u << 16) || d->n4 > (1u << 20))
        return set_error(WX_ERR_UNSUPPORTED, w + ": more than 65536 node-5 or 2^20 node-4 nodes");
    std::vector<uint32_t> base;
    bool compact = true;
    try {  // base takes 4 bytes per node
        if (int rc = check_desc(d, who, base, compact)) return rc;
    } catch (const std::bad_alloc &) {
        return set_error(WX_ERR_BUDGET, w + ": host allocation failed");
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return set_error(WX_ERR_DEVICE, w + ": no HIP device");
    wx_grid *g = new (std::nothrow) wx_grid();
    if (!g) return set_error(WX_ERR_BUDGET, w + ": host allocation failed");
    (void)hipGetDevice(&g->device);
    const size_t sz[4] = {(size_t)d->n5 * 16u, (size_t)d->n5 * 4096u * 16u, (size_t)d->n4 * 256u * 16u,
                          (size_t)d->n3 * 64u * 4u};
    const void *src[4] = {d->root, d->n5_records, d->n4_records, d->leaves};
    const uint64_t nrec[3] = {(uint64_t)d->n5 * 4096u, (uint64_t)d->n4 * 256u, base.size()};
    const uint64_t rec_bytes[3] = {compact ? 16u : 32u, compact ? 32u : 64u, 4u};
    size_t n[7], all = 0;
    for (int k = 0; k < 7; ++k) {
        n[k] = std::max<size_t>(k < 4 ? sz[k] : nrec[k - 4] * rec_bytes[k - 4], 16u);
        g->bytes += n[k];
        all += wx::DeviceArena::piece(n[k]);
    }
    hipError_t e = g->arena.allocate(all);
    if (e != hipSuccess) {
        wx_grid_destroy(g);
        return set_error(e == hipErrorOutOfMemory ? WX_ERR_BUDGET : WX_ERR_DEVICE,
                         w + ": hipMalloc: " + hipGetErrorString(e));
    }
    for (int k = 0; k < 7; ++k) (k < 4 ? g->mem[k] : g->entries[k - 4]) = g->arena.take<void>(n[k]);
    for (int k = 0; k < 4; ++k) {
        if (!sz[k] || !src[k]) continue;
        e = hipMemcpy(g->mem[k], src[k], sz[k], hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            wx_grid_destroy(g);
            return hip_fail(e, (w + ": hipMemcpy").c_str());
        }
    }
    // the slot entries, made on the default stream after the copies and waited for, so the
    // grid is complete for work on any stream
    const uint32_t *dbase = static_cast<const uint32_t *>(g->entries[2]) + d->n5;
    if (!base.empty()) e = hipMemcpy(g->entries[2], base.data(), base.size() * 4u, hipMemcpyHostToDevice);
    for (int k = 0; k < 2 && e == hipSuccess; ++k) {
        if (!nrec[k]) continue;
        const uint4 *rec = static_cast<const uint4 *>(g->mem[1 + k]);
        uint4 *out = static_cast<uint4 *>(g->entries[k]);
        const dim3 blocks((uint32_t)std::min<uint64_t>((nrec[k] + 255u) / 256u, 8192u));
        if (k == 0)
            hipLaunchKernelGGL(k_expand<8>, blocks, dim3(256), 0, nullptr, rec, nrec[k], compact ? dbase - 1 : nullptr, -1,
                               out);
        else
            hipLaunchKernelGGL(k_expand<16>, blocks, dim3(256), 0, nullptr, rec, nrec[k], compact ? dbase : nullptr, 1, out);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    if (e != hipSuccess) {
        wx_grid_destroy(g);
        return hip_fail(e, (w + ": slot entries").c_str());
    }
    g->dev.root = static_cast<const int4 *>(g->mem[0]);
    g->dev.n5 = g->entries[0];
    g->dev.n4 = g->entries[1];
    g->dev.leaf = static_cast<const uint32_t *>(g->mem[3]);
    g->dev.base = dbase;
    g->dev.n5count = d->n5;
    g->dev.bound = d->bound;
    g->n5 = d->n5;
    g->n4 = d->n4;
    g->n3 = d->n3;
    if (d->n5) g->dev.kx = d->root[0], g->dev.ky = d->root[1], g->dev.kz = d->root[2];
    // WX_WIDE_LEAVES=1 takes the 64-bit pool addressing at any size (to test it on small grids)
    const char *wide = std::getenv("WX_WIDE_LEAVES");
    const bool narrow = d->n3 <= (1u << 24) && !(wide && wide[0] == '1');
    // a key that 20 bits hold is one that a voxel coordinate mod 2^32 decides (lane_lookup)
    auto key_fits = [](int32_t k) { return k >= -(1 << 19) && k < (1 << 19); };
    const bool one_root = d->n5 == 1u && base[0] == 0u - kWalk && key_fits(g->dev.kx) && key_fits(g->dev.ky) &&
                          key_fits(g->dev.kz);
    g->dev.form = !compact ? kIndexed : (one_root && narrow ? kOneRoot : kTable);
    *out = g;
    return WX_OK;
}

void *grid_pool(wx_grid *g, int k) { return g->mem[k]; }

}  // namespace wx

extern "C" {

int wx_device_count(int *count) {
    if (!count) return set_error(WX_ERR_INVALID, "wx_device_count: NULL argument");
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    *count = (e == hipSuccess) ? n : 0;
    return WX_OK;
}

int wx_grid_create(const wx_grid_desc *d, wx_grid **out) {
    if (!d || !out) return set_error(WX_ERR_INVALID, "wx_grid_create: NULL argument");
    if (d->n3 && !d->leaves) return set_error(WX_ERR_INVALID, "wx_grid_create: NULL pool with a non-zero count");
    return wx::grid_new(d, "wx_grid_create", out);
}

int wx_vdb_grid_create(const wx_vdb *v, float bound, wx_grid **out) {
    if (!v || !out) return set_error(WX_ERR_INVALID, "wx_vdb_grid_create: NULL argument");
    const wx::HostVdb &t = v->tree;
    if (!t.finalized()) return set_error(WX_ERR_STATE, "wx_vdb_grid_create: tree not finalized");
    wx_grid_desc d;
    d.n5 = t.n5();
    d.n4 = t.n4();
    d.n3 = t.n3();
    d.bound = bound;
    d.root = t.root_table().data();
    d.n5_records = reinterpret_cast<const uint32_t *>(t.n5_records().data());
    d.n4_records = reinterpret_cast<const uint32_t *>(t.n4_records().data());
    d.leaves = nullptr;
    // leaf words a device replay left on this device are copied there; otherwise
    // they come from the host copy (fetched first if it is not on the host yet)
    int cur = 0;
    if (hipGetDevice(&cur) != hipSuccess) return set_error(WX_ERR_DEVICE, "wx_vdb_grid_create: no HIP device");
    const wx::DeviceWords *dw = t.device_words();
    const bool on_device = dw && dw->device() == cur;
    if (!on_device) {
        std::string err;
        if (!t.host_words(err)) return set_error(WX_ERR_DEVICE, "wx_vdb_grid_create: " + err);
        d.leaves = t.leaf_slots();
    }
    wx_grid *g = nullptr;
    if (int rc = wx::grid_new(&d, "wx_vdb_grid_create", &g)) return rc;
    if (on_device && d.n3) {
        // waited for, so the grid is complete for work on any stream when this returns
        hipError_t e = hipMemcpyAsync(g->mem[3], dw->data(), (size_t)d.n3 * 256u, hipMemcpyDeviceToDevice, nullptr);
        if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
        if (e != hipSuccess) {
            wx_grid_destroy(g);
            return hip_fail(e, "wx_vdb_grid_create: device copy of the leaf words");
        }
    }
    *out = g;
    return WX_OK;
}

int wx_grid_destroy(wx_grid *g) {
    if (!g) return WX_OK;
    delete g;
    return WX_OK;
}

int wx_grid_bytes(const wx_grid *g, uint64_t *out) {
    if (!g || !out) return set_error(WX_ERR_INVALID, "wx_grid_bytes: NULL argument");
    *out = g->bytes;
    return WX_OK;
}

int wx_trace_camera(wx_grid *g, const wx_camera *cam, uint32_t w, uint32_t h, float pixel_offset, uint32_t flags,
                    wx_hit *out, wx_stream stream) {
    if (!g || !cam || !out) return set_error(WX_ERR_INVALID, "wx_trace_camera: NULL argument");
    if (flags & ~(WX_TRACE_CLIP | WX_TRACE_SIMPLE)) return set_error(WX_ERR_INVALID, "wx_trace_camera: bad flags");
    wx_request r;
    std::memset(&r, 0, sizeof r);
    r.kind = WX_REQ_CAMERA;
    r.width = w;
    r.height = h;
    r.flags = flags & WX_TRACE_CLIP;
    r.pixel_offset = pixel_offset;
    r.camera = *cam;
    r.out = out;
    return trace_one(g, r, flags, (hipStream_t)stream);
}

int wx_trace_rays(wx_grid *g, const wx_ray *rays, uint32_t n, uint32_t flags, wx_hit *out, wx_stream stream) {
    if (!g || ((!rays || !out) && n)) return set_error(WX_ERR_INVALID, "wx_trace_rays: NULL argument");
    if (flags & ~(WX_TRACE_CLIP | WX_TRACE_SIMPLE)) return set_error(WX_ERR_INVALID, "wx_trace_rays: bad flags");
    wx_request r;
    std::memset(&r, 0, sizeof r);
    r.kind = WX_REQ_RAYS;
    r.width = n;
    r.height = 1;
    r.flags = flags & WX_TRACE_CLIP;
    r.rays = rays;
    r.out = out;
    return trace_one(g, r, flags, (hipStream_t)stream);
}

int wx_tune_get(wx_tune *out) {
    if (!out) return set_error(WX_ERR_INVALID, "wx_tune_get: NULL argument");
    *out = current_tune();
    return WX_OK;
}

int wx_tune_set(const wx_tune *t) {
    if (!t || !tune_ok(*t)) return set_error(WX_ERR_INVALID, "wx_tune_set: out of range");
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tune[dev] = *t;
    return WX_OK;
}

int wx_trace_batch(wx_grid *const *grids, uint32_t n_grids, const wx_request *reqs, uint32_t n_reqs,
                   const wx_tune *tune, wx_stream stream) {
    if ((!grids && n_grids) || (!reqs && n_reqs)) return set_error(WX_ERR_INVALID, "wx_trace_batch: NULL argument");
    if (n_reqs == 0) return WX_OK;
    if (n_grids == 0) return set_error(WX_ERR_INVALID, "wx_trace_batch: no grids");
    return launch_batch(grids, n_grids, reqs, n_reqs, tune ? *tune : current_tune(), (hipStream_t)stream);
}

int wx_trace_batch_static(wx_grid *const *grids, uint32_t n_grids, const wx_request *reqs, uint32_t n_reqs,
                          const wx_tune *tune, wx_stream stream) {
    if ((!grids && n_grids) || (!reqs && n_reqs))
        return set_error(WX_ERR_INVALID, "wx_trace_batch_static: NULL argument");
    if (n_reqs == 0) return WX_OK;
    if (n_grids == 0) return set_error(WX_ERR_INVALID, "wx_trace_batch_static: no grids");
    if (n_grids > kMaxGridsLds || n_reqs > kMaxReqsLds)
        return set_error(WX_ERR_INVALID, "wx_trace_batch_static: at most 64 grids and 1024 requests per call");
    Staging stg;
    stg.is_static = true;
    if (int rc = static_scratch(&stg.dev, &stg.host)) return rc;
    return launch_batch(grids, n_grids, reqs, n_reqs, tune ? *tune : current_tune(), (hipStream_t)stream, stg);
}

int wx_autotune(wx_grid *const *grids, uint32_t n_grids, const wx_request *reqs, uint32_t n_reqs, wx_stream stream,
                wx_tune *best, float *best_ms) {
    if (!grids || !reqs || !n_grids || !n_reqs) return set_error(WX_ERR_INVALID, "wx_autotune: empty batch");
    hipStream_t s = (hipStream_t)stream;
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return set_error(WX_ERR_DEVICE, "wx_autotune: event create");
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return set_error(WX_ERR_DEVICE, "wx_autotune: event create");
    }
    const uint32_t refills[] = {1, 8, 16, 24, 32, 48};
    const uint32_t chunks[] = {64, 128, 256, 512};
    const uint32_t waves[] = {8, 12, 16, 24, 32};
    wx_tune bt = default_tune();
    float bms = 1e30f;
    int rc = WX_OK;
    auto time_it = [&](const wx_tune &t, float &ms) -> int {
        int r = launch_batch(grids, n_grids, reqs, n_reqs, t, s);  // warm
        if (r) return r;
        float acc = 0.f;
        for (int rep = 0; rep < 3; ++rep) {
            if (hipEventRecord(e0, s) != hipSuccess) return set_error(WX_ERR_DEVICE, "wx_autotune: event record");
            r = launch_batch(grids, n_grids, reqs, n_reqs, t, s);
            if (r) return r;
            if (hipEventRecord(e1, s) != hipSuccess) return set_error(WX_ERR_DEVICE, "wx_autotune: event record");
            if (hipEventSynchronize(e1) != hipSuccess) return set_error(WX_ERR_DEVICE, "wx_autotune: sync");
            float m = 0.f;
            if (hipEventElapsedTime(&m, e0, e1) != hipSuccess) return set_error(WX_ERR_DEVICE, "wx_autotune: event time");
            acc += m;
        }
        ms = acc / 3.f;
        return WX_OK;
    };
    // the one-lane-per-ray shape, then a coordinate search over the persistent shape: waves,
    // refill and, where there is a work queue (not for one request without shadow rays), chunk
    // and XCD split
    const bool queue = n_reqs > 1u || n_grids > 1u || (reqs[0].flags & WX_TRACE_SHADOW);
    {
        wx_tune c = default_tune();
        c.persistent = 0;
        float ms;
        rc = time_it(c, ms);
        if (rc == WX_OK && ms < bms) bms = ms, bt = c;
    }
    wx_tune t = default_tune();
    t.persistent = 1;
    wx_tune pbest = t;
    float pms = 1e30f;
    for (int pass = 0; pass < 2 && rc == WX_OK; ++pass) {
        for (uint32_t w : waves) {
            wx_tune c = t;
            c.waves_per_cu = w;
            float ms;
            if ((rc = time_it(c, ms))) break;
            if (ms < pms) pms = ms, pbest = c;
        }
        t = pbest;
        for (uint32_t rf : refills) {
            wx_tune c = t;
            c.refill = rf;
            float ms;
            if ((rc = time_it(c, ms))) break;
            if (ms < pms) pms = ms, pbest = c;
        }
        t = pbest;
        for (uint32_t ch : chunks) {
            if (!queue) break;
            wx_tune c = t;
            c.chunk = ch;
            float ms;
            if ((rc = time_it(c, ms))) break;
            if (ms < pms) pms = ms, pbest = c;
        }
        t = pbest;
        for (uint32_t x = 0; x <= 1 && queue; ++x) {
            wx_tune c = t;
            c.xcd_split = x;
            float ms;
            if ((rc = time_it(c, ms))) break;
            if (ms < pms) pms = ms, pbest = c;
        }
        t = pbest;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    if (pms < bms) bms = pms, bt = pbest;
    wx_tune_set(&bt);
    if (best) *best = bt;
    if (best_ms) *best_ms = bms;
    return WX_OK;
}

}  // extern "C"
