// vp_render.hip — the render path on gfx950.
//
// One persistent megakernel traces camera paths; each 64-lane wavefront
// claims new paths with one atomic per wave (ballot + popcount rank) once
// enough of its lanes are idle, so lanes stay busy across uneven path
// lengths.  Per bounce a lane
//   1. takes the argmin of closed-form per-primitive free flights over the
//      primitives containing its origin and, in one walk of the
//      BVH, over every primitive the ray enters (no hit buffer: each
//      primitive's uniform is a counter hash, so the minimum can be taken in
//      any order and the walk prunes boxes beyond the running minimum); at
//      bounce 0 the same walk integrates the analytic direct term;
//   2. rebuilds the active set at the scatter point from the primitives the
//      argmin walk entered, applying the reference's per-primitive exit
//      tests;
//   3. evaluates albedo, samples the HG phase, and runs NEE (balance-MIS of
//      phase and environment sampling, or product RIS) with shadow rays whose
//      optical depth is accumulated in fixed point;
//   4. applies Russian roulette and the throughput guards.
// The argmin and shadow walks and the work on the active sets are done by the
// 64 lanes of a wavefront together, for all its paths.
// Each path adds its radiance to its pixel's exact fixed-point sums; a second
// kernel divides them, so the image does not depend on which lane ran which
// path or on what else shared the launch.
//
// Reference (kfernandez31/cuda-volprim): device/entry/raygen.cuh:21-243,
// device/entry/path_stages.cuh:25-226, device/core/sampling.cuh:257-583,
// device/entry/anyhit.cuh:53-86, device/kernels/normalize_accumulator.cu:16-35.
// The megakernel holds a whole path per lane at 4 waves per SIMD (128 VGPRs);
// a wavefront's queues and ray tables take the 10 KiB of LDS that 16 waves
// leave each other of a CU's 160 KiB.
#include "vp_device.h"

namespace vp {
namespace {

struct PathState {
    f3 o, d, beta, L;
    Pcg32 rng;
    uint64_t key;
    uint32_t bounce, job, na, cur, pix, sl;
    float ts_set;  // minimum free flight over the active set (timed kernel, bounces > 0)
};

// Minimum waves per SIMD the register allocator targets for the megakernel.
#ifndef VP_RENDER_WAVES_PER_EU
#define VP_RENDER_WAVES_PER_EU 4
#endif

// How many free flights of an argmin walk wait to be inverted together (see
// argmin_walk_shared).
constexpr uint32_t kFlightMin = 16;

// The path key and bounce of lane l's draws.
__device__ __forceinline__ uint64_t draw_key(const MegaQueue& q, uint32_t l) {
    return (static_cast<uint64_t>(q.draw(l)[1]) << 32) | q.draw(l)[0];
}
__device__ __forceinline__ uint32_t draw_bounce(const MegaQueue& q, uint32_t l) { return q.draw(l)[2] & 0x7fffffffu; }

// The rounds of argmin walks, from nn items on, over the stack and leaf queue
// of stack and the rays of rays (those of wavefront rays_of of the workgroup).
// The rays' own wavefront (kOwn) keeps their ends: a ray is walked up to the
// bound of its minimum, a direct one whole until its depth reaches the limit,
// and with kMeasure every ray whole, its entries counted.
template <bool kOwn, bool kMeasure>
__device__ __forceinline__ void argmin_rounds(const WaveScene& ws, uint32_t* lds, const MegaQueue& stack,
                                              const MegaQueue& rays, uint32_t rays_of, uint64_t lim,
                                              uint32_t* __restrict__ slab, uint32_t cap, uint32_t nn,
                                              uint32_t& rounds) {
    const uint32_t lane = __lane_id();
    const MegaQueue q = rays_with_stack(rays, stack);
    auto set_tmax = [&]() {
        q.tmax[2 * lane] = kMeasure || q.acc[2 * lane] < lim ? kTMax : __uint_as_float(q.bound(lane));
    };
    // the first thread of the rays' wavefront, for the owners' candidate buffers
    const uint32_t gbase = blockIdx.x * blockDim.x + rays_of * 64u;
    const uint32_t bs = mega_slab_stride(cap);
    uint32_t nl = 0, nf = 0;
    if (kOwn) {
        set_tmax();
        wave_sync();
    }
    static_assert(kLeafItems >= 64u + kFlightMin + 64 + 4, "room for a step's leaves and the flights");
    while (true) {
        if (nl < 64u && nn != 0u) {
            if (nn >= kHelpMin && (rounds & (kHelpEvery - 1u)) == 0u) give_items(lds, q, rays_of, ws.one, true, nn);
            walk_nodes<true>(q, ws, nn, nl, kLeafItems - nf);
            ++rounds;
            continue;
        }
        if (nl != 0u) {
            // 64 leaves (or the last ones): their crossings (entry, exit and
            // whole-chord depth from one transform).  On a direct ray the
            // depth joins the ray's sum; a leaf entered before the running
            // minimum is a rebuild candidate (beyond it nothing can change,
            // t >= entry > minimum) and its free flight is sampled, which
            // ends inside the chord when the sampled depth is at most the
            // chord's.
            const uint32_t n = nl < 64u ? nl : 64u;
            nl -= n;
            ++rounds;
            bool keep = false;
            uint32_t ray = 0, prim = 0;
            if (lane < n) {
                ray = q.leaf_ray[nl + lane];
                prim = q.leaf[nl + lane];
                const uint32_t own = ray >> 1;
                const f3 ro = lds_load3(q.ro + 3 * own), rd = lds_load3(q.rd + 3 * ray);
                const Crossing x = crossing(load_wave_leaf(q, ws, own, prim), ro, rd);
                if (x.t0 >= 0.0f) {
                    if (kMeasure) atomicAdd(&q.hits(own), 1u);
                    const uint32_t meta = q.draw(own)[2];
                    if ((meta >> 31) != 0u && x.tau > 0.0f) atomicAdd(&q.acc[ray], tau_fixed(x.tau));
                    if (x.t0 <= __uint_as_float(q.bound(own))) {
                        const uint32_t pos = atomicAdd(&q.nc(own), 1u);
                        if (pos < cap) {
                            uint32_t* mine = slab + static_cast<size_t>(gbase + own) * kMegaSlabBuffers * bs;
                            mine[2 * bs + pos] = prim;
                            mine[3 * bs + pos] = __float_as_uint(x.t0);
                            mine[4 * bs + pos] = __float_as_uint(x.t1);
                        }
                        const float tau = free_flight_tau(prim_uniform(draw_key(q, own), meta & 0x7fffffffu, 1u, prim));
                        keep = tau <= x.tau;
                        if (keep) atomicMin(&q.bound(own), __float_as_uint(x.t1));
                    }
                }
            }
            const unsigned long long km = __builtin_amdgcn_ballot_w64(keep);
            wave_sync();
            // the flights to invert wait at the end of the leaf queue (the
            // slots of the leaves just taken are free)
            if (keep) {
                const uint32_t at = kLeafItems - 1u - nf - lanes_below(km);
                q.leaf[at] = prim;
                q.leaf_ray[at] = static_cast<uint8_t>(ray);
            }
            nf += static_cast<uint32_t>(__popcll(km));
            wave_sync();
            if (kOwn) set_tmax();
            wave_sync();
        }
        if (nf >= kFlightMin || (nl == 0u && nf != 0u)) {
            // invert the waiting flights into distances
            for (uint32_t f = lane; f < nf; f += 64u) {
                const uint32_t ray = q.leaf_ray[kLeafItems - 1u - f], prim = q.leaf[kLeafItems - 1u - f];
                const uint32_t own = ray >> 1;
                const f3 ro = lds_load3(q.ro + 3 * own), rd = lds_load3(q.rd + 3 * ray);
                const PrimRecord pr = load_prim(ws.jobs[q.job[own]].scene.prims, prim);
                const float tau = free_flight_tau(prim_uniform(draw_key(q, own), draw_bounce(q, own), 1u, prim));
                const float t = entered_flight(pr, ro, rd, crossing(pr, ro, rd), tau);
                const uint32_t tb = t == 0.0f ? 0u : __float_as_uint(t);
                atomicMin(&q.ts(own), tb);
                atomicMin(&q.bound(own), tb);
            }
            nf = 0;
            wave_sync();
            if (kOwn) set_tmax();
            wave_sync();
        }
        if (nl == 0u && nn == 0u) break;
    }
    if (kOwn)
        while (help_load(q.help + 1) != 0u) {
            set_tmax();
            __builtin_amdgcn_s_sleep(4);
        }
}

// Argmin free flight over the entered primitives (sampling.cuh:372-412) with
// the wave-shared leaf queue.  All 64 lanes of the wavefront call it: a lane
// with a path (alive) walks its own ray, and the origin-set members and queued
// leaves of all rays are shared out among all lanes, so a wavefront with few
// paths left still evaluates them 64 at a time.
// Each ray's running minimum is an LDS atomic minimum over float bits (all
// candidates are >= 0), so the result does not depend on which lane handles
// which leaf.  Candidates for the rebuild are recorded while t_entry is at
// most the running minimum at the time, which covers every primitive entered
// before the final one; their order is fixed by the sort in the rebuild.  At
// bounce 0 (direct) the walk also sums the direct term's optical depth into
// dacc, and runs over the whole ray until that sum reaches dlimit (the
// tau = 88 saturation or the direct term's roulette level, where T becomes
// 0); from there on it prunes at the running minimum like any other ray.
// ts_origin is the minimum over the origin set; the result keeps it unless a
// walk candidate is strictly smaller.
// Flights waiting to be inverted are taken up once there are kFlightMin of
// them (few leaves have one, and the inversion's erf and erfinv cost as much
// as the leaf round), or at the end of a run of leaves.  A flight ends inside
// its chord, so until then its exit bounds the minimum (bound, which the walk
// prunes by): without that bound, waiting for 16 flights cost the 10^6 cloud
// 12 % and the 192x128 cloud 18 % against waiting for 4; with it, nothing.
// hits receives the ray's entries (kMeasure).
template <bool kMeasure>
__device__ __forceinline__ void argmin_walk_shared(bool alive, const WaveScene& ws, uint32_t job, f3 o, f3 d, uint64_t key,
                                                   uint32_t b, bool direct, const uint32_t* act, uint32_t na_path,
                                                   float* act_exit, float ts_set, uint32_t* __restrict__ slab,
                                                   uint32_t cap, const MegaQueue& q, float& ts, uint32_t& nc,
                                                   uint64_t dlimit, uint64_t& dacc, uint32_t& rounds,
                                                   uint32_t* lds, uint32_t& hits) {
    const uint32_t lane = __lane_id();
    const uint32_t na = direct ? na_path : 0u;
    lds_store3(q.ro + 3 * lane, o);
    lds_store3(q.rd + 3 * (2 * lane), d);
    lds_store3(q.inv + 3 * (2 * lane), safe_inv(d));
    q.draw(lane)[0] = static_cast<uint32_t>(key);
    q.draw(lane)[1] = static_cast<uint32_t>(key >> 32);
    q.draw(lane)[2] = b | (direct ? 0x80000000u : 0u);
    q.job[lane] = job;
    q.acc[2 * lane] = 0ull;
    q.ts(lane) = __float_as_uint(direct ? kTMax : ts_set);
    q.nc(lane) = 0u;
    if (kMeasure) q.hits(lane) = 0u;
    // The origin set (sampling.cuh:356-370) of a path at bounce 0; from then
    // on the last vertex's pass over the set has evaluated it (vertex_members)
    // and ts_set is its minimum.  The wavefront's (member, lane) pairs are
    // numbered through a prefix sum of the set sizes and shared out over the
    // lanes.  Per member: its exit (kept in the owner's slab for the rebuild),
    // its free flight into the owner's running minimum, and its chord into the
    // owner's direct-term optical depth; minima and fixed-point sums do not
    // depend on which lane adds what.  (Active sets of the megakernel are
    // contiguous.)
    if (__builtin_amdgcn_ballot_w64(na != 0u) != 0ull) {
        const uint32_t** set_of = reinterpret_cast<const uint32_t**>(q.scratch);  // [64]
        float** exit_of = reinterpret_cast<float**>(q.scratch) + 64;               // [64]
        uint32_t* pre_of = q.scratch + 4 * 64;                                    // [64]
        static_assert(kScratch >= 5 * 64, "the origin-set tables must fit in the queue");
        uint32_t total;
        pre_of[lane] = wave_prefix(na, total);
        set_of[lane] = act;
        exit_of[lane] = act_exit;
        wave_sync();
        for (uint32_t g = lane; g < total; g += 64u) {
            const uint32_t ol = prefix_owner(pre_of, g), k = g - pre_of[ol];
            const uint32_t i = set_of[ol][k];
            const PrimRecord pr = load_prim(ws.jobs[q.job[ol]].scene.prims, i);
            const f3 ro = lds_load3(q.ro + 3 * ol), rd = lds_load3(q.rd + 3 * (2 * ol));
            const InsideChord x = inside_chord(pr, ro, rd);
            exit_of[ol][k] = x.t1;
            const float tau = free_flight_tau(prim_uniform(draw_key(q, ol), draw_bounce(q, ol), 0u, i));
            if (tau <= x.tau) {
                const float t = origin_flight(pr, ro, rd, x, tau);
                atomicMin(&q.ts(ol), t == 0.0f ? 0u : __float_as_uint(t));
            }
            if (x.tau > 0.0f) atomicAdd(&q.acc[2 * ol], tau_fixed(x.tau));
        }
    }
    wave_sync();
    const float ts_origin = __uint_as_float(q.ts(lane));
    q.bound(lane) = q.ts(lane);
    uint32_t nn = 0;
    const unsigned long long am = __builtin_amdgcn_ballot_w64(alive);
    if (alive) q.list[lanes_below(am)] = static_cast<uint8_t>(2 * lane);
    wave_sync();
    push_rays(q, ws, q.list, static_cast<uint32_t>(__popcll(am)), nn);
    // a direct ray is walked until its depth reaches the limit
    argmin_rounds<true, kMeasure>(ws, lds, q, q, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), direct ? dlimit : 0ull, slab,
                        cap, nn, rounds);
    const float wmin = __uint_as_float(q.ts(lane));
    ts = wmin < ts_origin ? wmin : ts_origin;
    nc = q.nc(lane);
    dacc = q.acc[2 * lane];
    if (kMeasure) hits = q.hits(lane);
    wave_sync();
}

// A wavefront without paths works for the others of its workgroup until none
// of them has any.
template <bool kMeasure>
__device__ __forceinline__ void help_walks(uint32_t* lds, const JobDesc* jobs, uint32_t* __restrict__ slab,
                                           uint32_t cap) {
    const uint32_t lane = __lane_id();
    const MegaQueue q = mega_queue(lds);
    uint32_t* const active = mega_queue_of(lds, 0u).help + 2;
    if (lane == 0u)
        (void)__hip_atomic_fetch_sub(active, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (true) {
        if (lane == 0u)
            __hip_atomic_store(q.help, kHelpWait, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        uint32_t given;
        while (((given = help_load(q.help)) & kHelpWork) == 0u) {
            if (help_load(active) == 0u) return;
            __builtin_amdgcn_s_sleep(8);
        }
        const uint32_t rays_of = (given >> 8) & 0xffu, n = given >> 16;
        const MegaQueue rq = mega_queue_of(lds, rays_of);
        WaveScene ws = wave_scene(jobs[rq.job[q.node_ray[0] >> 1]].scene, true, jobs);
        ws.one = ws.one && (given & 4u) != 0u;
        uint32_t rounds = 0;
        if ((given & 8u) != 0u)
            argmin_rounds<false, kMeasure>(ws, lds, q, rq, rays_of, 0ull, slab, cap, n, rounds);
        else
            shadow_rounds<false>(ws, lds, q, rq, rays_of, 0u, 0ull, 0ull, n, rounds);
        // the candidates as well as the sums and minima are there first
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if (lane == 0u)
            (void)__hip_atomic_fetch_sub(rq.help + 1, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

// ---- the vertex stage of the timed kernel, all lanes of a wavefront together ----
//
// Slab buffers of a path at a vertex (kMegaSlabBuffers of bs words each): its
// active set in buffer cur, the members' exits along the ray in the other set
// buffer, cur ^ 1, and the ray's candidates in 2 (index), 3 and 4 (entry and
// exit).  The rebuild compacts the members and candidates that contain the
// vertex in place (buffers cur and 2) and merges them into buffer cur ^ 1,
// which becomes the active set; the pass over its members then writes their
// albedo terms over buffers 2 to 5 and their exits along the next ray into the
// old set's buffer.

// Words of the slab before lane own's buffers (gbase: the wavefront's first thread).
__device__ __forceinline__ uint32_t* slab_of(uint32_t* slab, uint32_t gbase, uint32_t own, uint32_t bs) {
    return slab + static_cast<size_t>(gbase + own) * kMegaSlabBuffers * bs;
}

// Kept candidates of a wavefront that the merge below holds in LDS; more than
// these are read from the slab.
constexpr uint32_t kCandItems = 512;

// The active sets at the scatter points (sampling.cuh:422-458) of the lanes
// with a vertex (part): a member stays while ts <= its exit; an entered
// candidate joins if its entry <= ts <= its exit; the set keeps ascending
// stored index, and the first cap of it are kept.  Both steps run over the
// wavefront's flattened items (members, then candidates, of every lane), 64
// at a time: first the tests, compacting what is kept within each path's
// buffers, then each kept item's position in the merged set, which is the
// number of kept members and candidates below it: a member's rank or a binary
// search among the members (ascending), plus a scan of the candidates (in the
// order the walk found them; 64 items scan at a time, so also thousands of
// candidates are ranked sooner than one lane sorts them: 64x64 image of 3000
// overlapping Gaussians, capacity 3000, 5.8 ms against 151).  A per-lane loop over its own lists waited on a
// load per entry and ran as long as the wavefront's longest list: 7 to 13 % of
// the dense scenes' and 11 % of a preview's time.
__device__ __forceinline__ uint32_t rebuild_shared(bool part, uint32_t na, uint32_t nc, uint32_t cur, float ts,
                                                   uint32_t* __restrict__ slab, uint32_t cap, const MegaQueue& q,
                                                   uint32_t& overflow) {
    const uint32_t lane = __lane_id();
    const uint32_t gbase = blockIdx.x * blockDim.x + (threadIdx.x & ~63u);
    const uint32_t bs = mega_slab_stride(cap);
    // tables in the queue's space, 64 words each
    uint32_t* pre_of = q.scratch;
    uint32_t* na_of = pre_of + 64;        // members of the list being flattened | set buffer << 31
    uint32_t* kept_of = pre_of + 128;     // [2][64] kept members, kept candidates
    float* ts_of = reinterpret_cast<float*>(pre_of + 256);
    uint32_t* cand = pre_of + 320;        // [kCandItems + 3] kept candidates
    static_assert(kScratch >= 5 * 64 + kCandItems + 3, "the rebuild's tables must fit in the queue");
    uint32_t total, total_c = 0;
    pre_of[lane] = wave_prefix(part ? na + nc : 0u, total);
    na_of[lane] = na | (cur << 31);
    kept_of[lane] = 0u;
    kept_of[64 + lane] = 0u;
    ts_of[lane] = ts;
    wave_sync();
    for (uint32_t base = 0; base < total; base += 64u) {
        const uint32_t g = base + lane;
        const uint32_t own = prefix_owner(pre_of, g), p0 = pre_of[own], k = g - p0;
        const uint32_t meta = na_of[own], n = meta & 0x7fffffffu, set = (meta >> 31) * bs;
        uint32_t* mine = slab_of(slab, gbase, own, bs);
        const bool member = k < n;
        const uint32_t kc = k - n;
        bool keep = false;
        uint32_t id = 0;
        if (g < total) {
            const float t = ts_of[own];
            id = mine[member ? set + k : 2u * bs + kc];
            const float t1 = __uint_as_float(mine[member ? bs - set + k : 4u * bs + kc]);
            const float t0 = member ? 0.0f : __uint_as_float(mine[3u * bs + kc]);
            keep = t0 >= 0.0f && (member || t0 <= t) && t <= t1;
        }
        const unsigned long long km = __builtin_amdgcn_ballot_w64(keep && member);
        const unsigned long long kc_m = __builtin_amdgcn_ballot_w64(keep && !member);
        // the lanes of this round with the same owner start at p0 - base
        const unsigned long long seg = p0 > base ? ~0ull << (p0 - base) : ~0ull;
        if (keep) {
            uint32_t* kept = kept_of + (member ? own : 64u + own);
            const uint32_t pos = *kept + lanes_below((member ? km : kc_m) & seg);
            atomicAdd(kept, 1u);
            mine[(member ? set : 2u * bs) + pos] = id;
            const uint32_t at = total_c + lanes_below(kc_m);
            if (!member && at < kCandItems) cand[at] = id;
        }
        total_c += static_cast<uint32_t>(__popcll(kc_m));
        wave_sync();
    }
    bool serial = false;
    if (total != 0u) {
        // items were met path by path, so the kept candidates lie in LDS path
        // by path, from c_of[path]
        const bool in_lds = total_c <= kCandItems;
        uint32_t* c_of = reinterpret_cast<uint32_t*>(ts_of);
        uint32_t total_m;
        wave_sync();
        pre_of[lane] = wave_prefix(kept_of[lane], total_m);
        c_of[lane] = wave_prefix(kept_of[64 + lane], total_c);
        wave_sync();
        // kept candidates of path own below id
        auto below = [&](uint32_t own, uint32_t id) {
            const uint32_t nk = kept_of[64 + own];
            uint32_t n = 0;
            auto count = [&](uint32_t j, uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3) {
                n += (v0 < id ? 1u : 0u) + (j + 1u < nk && v1 < id ? 1u : 0u) + (j + 2u < nk && v2 < id ? 1u : 0u) +
                     (j + 3u < nk && v3 < id ? 1u : 0u);
            };
            if (in_lds) {
                const uint32_t* c = cand + c_of[own];
                for (uint32_t j = 0; j < nk; j += 4u) count(j, c[j], c[j + 1u], c[j + 2u], c[j + 3u]);
            } else {
                const uint32_t* c = slab_of(slab, gbase, own, bs) + 2u * bs;
                for (uint32_t j = 0; j < nk; j += 4u) {
                    const uint4 v = *reinterpret_cast<const uint4*>(c + j);
                    count(j, v.x, v.y, v.z, v.w);
                }
            }
            return n;
        };
        for (uint32_t g = lane; g < total_m; g += 64u) {
            const uint32_t own = prefix_owner(pre_of, g), k = g - pre_of[own];
            const uint32_t set = (na_of[own] >> 31) * bs;
            uint32_t* mine = slab_of(slab, gbase, own, bs);
            const uint32_t id = mine[set + k];
            const uint32_t pos = k + below(own, id);
            if (pos < cap) mine[bs - set + pos] = id;
        }
        for (uint32_t g = lane; g < total_c; g += 64u) {
            const uint32_t own = prefix_owner(c_of, g);
            const uint32_t set = (na_of[own] >> 31) * bs, nm = kept_of[own];
            uint32_t* mine = slab_of(slab, gbase, own, bs);
            const uint32_t id = in_lds ? cand[g] : mine[2u * bs + g - c_of[own]];
            uint32_t lo = 0, hi = nm;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (mine[set + mid] < id) lo = mid + 1u;
                else hi = mid;
            }
            // a candidate that is also a member (an origin the rounding puts
            // outside a member's bound can enter it again) was counted twice
            if (lo < nm && mine[set + lo] == id) serial = true;
            const uint32_t pos = lo + below(own, id);
            if (pos < cap) mine[bs - set + pos] = id;
        }
    }
    wave_sync();
    const uint32_t mm = kept_of[lane], mc = kept_of[64 + lane];
    uint32_t nn = mm + mc;
    if (__builtin_amdgcn_ballot_w64(serial) != 0ull) {
        // each lane sorts its kept candidates and merges them with its kept
        // members, an index that is in both once
        wave_sync();
        uint32_t* mine = slab_of(slab, gbase, lane, bs);
        const uint32_t* set = mine + cur * bs;
        uint32_t* out = mine + (cur ^ 1u) * bs;
        uint32_t* own_cand = mine + 2u * bs;
        for (uint32_t i = 1; i < mc; ++i) {
            const uint32_t v = own_cand[i];
            uint32_t j = i;
            for (; j > 0 && own_cand[j - 1] > v; --j) own_cand[j] = own_cand[j - 1];
            own_cand[j] = v;
        }
        nn = 0;
        for (uint32_t i = 0, j = 0; i < mm || j < mc; ++nn) {
            const uint32_t a = i < mm ? set[i] : 0xffffffffu, c = j < mc ? own_cand[j] : 0xffffffffu;
            const uint32_t v = a < c ? a : c;
            if (a == v) ++i;
            if (c == v) ++j;
            if (nn < cap) out[nn] = v;
        }
    }
    wave_sync();
    if (nn > cap) {
        overflow += nn - cap;
        nn = cap;
    }
    return nn;
}

// One pass over the members of the wavefront's new active sets (nn members in
// buffer cur of the lanes with a vertex), flattened over the lanes: a
// member's record and its frame's origin serve its albedo term
// (evaluate_albedo, sampling.cuh:257-283), the chords of both shadow rays
// (has_a, has_b) and the next ray's exit and free flight (sampling.cuh:356-370
// at bounce b1), which were three passes with a load of the record each, the
// albedo's a loop per lane (11 to 22 % of the dense scenes' time).
// The albedo terms {albedo w, w} go to the owner's slab, to be summed in set
// order; the shadow rays' fixed-point depths stay in q.acc; ts_next receives
// the minimum free flight of the next ray over the set, kTMax if none.
// da, db and wo are the two shadow rays' and the next ray's directions from x.
__device__ __forceinline__ f3 vertex_members(uint32_t nn, uint32_t cur, bool has_a, bool has_b, const WaveScene& ws,
                                             f3 x, f3 da, f3 db, f3 wo, uint64_t key, uint32_t b1,
                                             uint32_t* __restrict__ slab, uint32_t cap, const MegaQueue& q,
                                             float& ts_next) {
    const uint32_t lane = __lane_id();
    const uint32_t gbase = blockIdx.x * blockDim.x + (threadIdx.x & ~63u);
    const uint32_t bs = mega_slab_stride(cap);
    // tables in the queue's space
    unsigned long long* key_of = reinterpret_cast<unsigned long long*>(q.scratch);  // [64]
    uint32_t* pre_of = q.scratch + 2 * 64;                           // [64]
    uint32_t* meta_of = pre_of + 64;                                 // [64] set buffer | has_a << 1 | has_b << 2
    uint32_t* ts_of = meta_of + 64;                                  // [64]
    uint32_t* b_of = ts_of + 64;                                     // [64]
    float* wo_of = reinterpret_cast<float*>(b_of + 64);              // [64 * 3]
    constexpr uint32_t kFlightItems = 256;
    uint32_t* flight = q.scratch + 9 * 64;                           // [kFlightItems] primitives
    uint8_t* flight_of = q.node_ray;                                 // [kFlightItems] their lanes
    static_assert(kScratch >= 9 * 64 + kFlightItems && kNodeQ >= kFlightItems,
                  "the member pass's tables must fit in the queue");
    uint32_t total;
    pre_of[lane] = wave_prefix(nn, total);
    meta_of[lane] = cur | (has_a ? 2u : 0u) | (has_b ? 4u : 0u);
    lds_store3(q.ro + 3 * lane, x);
    lds_store3(q.rd + 3 * (2 * lane), da);
    lds_store3(q.rd + 3 * (2 * lane + 1), db);
    q.acc[2 * lane] = 0ull;
    q.acc[2 * lane + 1] = 0ull;
    lds_store3(wo_of + 3 * lane, wo);
    key_of[lane] = key;
    ts_of[lane] = __float_as_uint(kTMax);
    b_of[lane] = b1;
    wave_sync();
    uint32_t nf = 0;  // flights waiting
    for (uint32_t base = 0; base < total; base += 64u) {
        const uint32_t g = base + lane;
        bool flies = false;
        uint32_t own = 0, i = 0;
        if (g < total) {
            own = prefix_owner(pre_of, g);
            const uint32_t k = g - pre_of[own];
            const uint32_t meta = meta_of[own], set = (meta & 1u) * bs;
            uint32_t* mine = slab_of(slab, gbase, own, bs);
            i = mine[set + k];
            const PrimRecord pr = load_wave_prim(q, ws, own, i);
            const f3 ro = lds_load3(q.ro + 3 * own);
            const f3 p = to_local_pos(pr, ro);
            const float pp = length2(p);
            const float ex = expf_(-0.5f * pp);
            const float wgt = pr.mass * (ex * pr.dnf);  // mass * prim_pdf
            *reinterpret_cast<float4*>(mine + 2u * bs + 4u * k) =
                make_float4(pr.ar * wgt, pr.ag * wgt, pr.ab * wgt, wgt);
            if ((meta & 2u) != 0u) {
                const float ta = inside_chord_from(pr, p, pp, lds_load3(q.rd + 3 * (2 * own)), ex).tau;
                if (ta > 0.0f) atomicAdd(&q.acc[2 * own], tau_fixed(ta));
            }
            if ((meta & 4u) != 0u) {
                const float tb = inside_chord_from(pr, p, pp, lds_load3(q.rd + 3 * (2 * own + 1)), ex).tau;
                if (tb > 0.0f) atomicAdd(&q.acc[2 * own + 1], tau_fixed(tb));
            }
            const InsideChord c = inside_chord_from(pr, p, pp, lds_load3(wo_of + 3 * own), ex);
            mine[bs - set + k] = __float_as_uint(c.t1);
            flies = free_flight_tau(prim_uniform(key_of[own], b_of[own], 0u, i)) <= c.tau;
        }
        // the few flights that end inside their chords wait until there are
        // enough to invert together (the inversion's erf, erfinv and exp took
        // as long as half a round for one or two lanes in most rounds)
        const unsigned long long fm = __builtin_amdgcn_ballot_w64(flies);
        if (flies) {
            flight[nf + lanes_below(fm)] = i;
            flight_of[nf + lanes_below(fm)] = static_cast<uint8_t>(own);
        }
        nf += static_cast<uint32_t>(__popcll(fm));
        wave_sync();
        if (nf + 64u > kFlightItems || base + 64u >= total) {
            for (uint32_t f = lane; f < nf; f += 64u) {
                const uint32_t fo = flight_of[f], fi = flight[f];
                const PrimRecord pr = load_wave_leaf(q, ws, fo, fi);
                const f3 ro = lds_load3(q.ro + 3 * fo), rw = lds_load3(wo_of + 3 * fo);
                const float tau = free_flight_tau(prim_uniform(key_of[fo], b_of[fo], 0u, fi));
                const float t = origin_flight(pr, ro, rw, inside_chord(pr, ro, rw), tau);
                atomicMin(&ts_of[fo], t == 0.0f ? 0u : __float_as_uint(t));
            }
            nf = 0;
            wave_sync();
        }
    }
    wave_sync();
    ts_next = __uint_as_float(ts_of[lane]);
    // the owner's terms in set order, read four at a time
    const float4* terms = reinterpret_cast<const float4*>(slab_of(slab, gbase, lane, bs) + 2u * bs);
    f3 aa = mk(0.0f);
    float aw = 0.0f;
    for (uint32_t k = 0; k < nn; k += 4u) {
        float4 t[4];
#pragma unroll
        for (uint32_t q = 0; q < 4u; ++q) t[q] = terms[k + q];  // (entries past nn lie in the slab and are not used)
#pragma unroll
        for (uint32_t q = 0; q < 4u; ++q) {
            if (k + q < nn) {
                aa = aa + f3{t[q].x, t[q].y, t[q].z};
                aw += t[q].w;
            }
        }
    }
    wave_sync();
    return aw <= 0.0f ? mk(0.0f) : aa * rcpf(aw);
}

// launch_desc[0] = number of job slices, launch_desc[1] = end of the
// launch's path range, launch_desc[2] = its start; read from device memory so
// one captured graph serves every step of a job mix.  A wavefront claims new
// paths once at least regen_min of its lanes are idle (or none is busy), with
// one fetch-and-add on the counter of a part of the launch's range (its XCD's
// part first): part start + counter.  A counter may run past its part (later
// claims there get nothing), and each launch has its own counters and range,
// so launches that run at once (the server starts a launch over the paths a
// longer job table adds while the earlier ones drain) hand out every path
// exactly once, without the retries a compare-and-swap on one shared counter
// costs when paths are short.
//
// How many of a wavefront's lanes hold a path: enough that a bounce's walks
// take about rounds_target rounds (node steps and leaf rounds), which its fixed
// part (set-up, rebuild, sampling, the walks' ends) is small against, and not
// more, since what a wavefront holds it has to finish by itself: a path of the
// 10^6 cloud takes about 40 rounds a bounce and one of the scattering scene 5.
// A wavefront starts on first_paths paths and claims at most claim_step at a
// time, so it sees what its paths cost before it takes more (neighbouring
// paths cost alike: with 64 paths to a wavefront, or a small launch's paths
// handed out at once, the longest wavefront of the torus ran 3.1 times and of
// the 192x128 cloud 9 times the mean).  At least 4 paths, target 128, 192 and
// 256 rounds, scattering 27.3, 26.4, 25.9 ms, torus 19.9, 20.2, 20.6, 10^6 cloud
// 202, 199, 197; 64 lanes always: 25.9, 41.3, 243.
// A wavefront that may hold 64 paths, in a scene of at most 4096 primitives
// (6 levels), claims claim_cheap at a time: where paths end after a bounce or
// two, 8 a claim are all it ever holds (1 Gaussian at 1024x1024x16 12.4 -> 7.6
// ms, 10 at 1024x1024x8 6.5 -> 2.7, 97 at 1024x1024x8 18.3 -> 13.5; 8.7, 3.7
// and 26.6 with one path per lane and no limits).  In larger scenes the cheap
// paths are those beside the object and the next ones may cost hundreds of
// times as much: 10^6 cloud 1024x1024x4 856 -> 904 ms, a far view of it 20 -> 49.
// hand_out: first_paths | claim_step << 8 | claim_cheap << 16 | regen_min << 24
// (one scalar register, where four were spilled to a vector register's lanes).
// The argmin and shadow walks are run by all 64 lanes of a wavefront together,
// so lanes without a path work on
// the rays of those that have one: a wavefront with two paths left evaluates
// their members and leaves 64 at a time and shares out their walks.  The
// counting build does not (kShared): it walks each ray by its own lane.
constexpr uint32_t kPathsMin = 4;
template <bool kCount, bool kMeasure>
__global__ void __launch_bounds__(kCount ? 256 : 1024)
    __attribute__((amdgpu_waves_per_eu(VP_RENDER_WAVES_PER_EU)))
k_render(const JobDesc* __restrict__ jobs, const uint64_t* __restrict__ job_begin,
         const uint64_t* __restrict__ launch_desc, unsigned long long* __restrict__ path_counter,
         uint32_t* __restrict__ slab, uint32_t cap, uint32_t hand_out, uint32_t rounds_target,
         unsigned long long* __restrict__ counters) {
    constexpr bool kShared = !kCount;
    extern __shared__ __align__(16) uint32_t s_leafq[];  // a queue of kMegaBytes to a wavefront
    const uint32_t first_paths = hand_out & 0xffu;
    const uint32_t njobs = static_cast<uint32_t>(launch_desc[0]);
    const uint64_t total_paths = launch_desc[1];
    const uint64_t path_lo = launch_desc[2];
    const uint32_t gl = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    // the lane's two active-set buffers, contiguous (lanes read and append
    // to their own sets at different times, so each set stays in few lines)
    constexpr uint32_t stride = 1;
    // buffers 0 and 1: active sets (ping-pong); buffer 2: primitives the
    // argmin walk entered before the running minimum (rebuild candidates)
    const uint32_t bs = mega_slab_stride(cap);
    uint32_t* my = slab + static_cast<size_t>(gl) * kMegaSlabBuffers * bs;  // entry k of buffer b at my[b * bs + k]
    const LeafQueue lq = mega_leaf_queue(s_leafq);
    const MegaQueue q = mega_queue(s_leafq);  // the same LDS, used by the wave-wide walks
    if constexpr (kShared) {
        help_begin(s_leafq);
        __syncthreads();
    }
    PathState st{};
    bool alive = false;
    bool exhausted = false;  // every part of the path range is used up (the same in all lanes)
    Ev<kCount> ev;
    ev.reset();
    uint32_t overflow = 0;
    uint32_t max_hits = 0, max_overlap = 0;  // of the lane's paths (kMeasure)
    // The launch's paths in kClaimParts parts.  The first paths of part k are
    // handed out without a counter: the wavefronts of the workgroups with
    // blockIdx % kClaimParts = k start on first_paths paths each (workgroups are
    // dealt out to the XCDs in turn), a workgroup's wavefronts on paths far
    // apart, since neighbouring ones cost alike (192x128x2 cloud 11.9 -> 10.3
    // ms, others the same), so a launch with no more
    // paths than that needs no atomics (each wavefront's 8 on the way out took
    // 430 us of a 4096-path launch).  The rest of part k is claimed through
    // path_counter[k * kClaimStride]; a wavefront starts with the part of the
    // XCD it runs on (the XCC_ID hardware register, bits 3:0), so each XCD's
    // waves trace a narrower band of the image and its L2 holds more of what
    // they read.  Which lane traces which path changes no result.
    // parts_done: the parts this wavefront has found used up.
    const uint32_t xcd = __builtin_amdgcn_s_getreg((3u << 11) | (0u << 6) | 20u) % kClaimParts;
    const uint64_t part = (total_paths - path_lo + kClaimParts - 1u) / kClaimParts;
    const uint32_t waves_per_block = blockDim.x / 64u;
    // paths of part k handed out at the start
    auto part_static = [&](uint32_t k) -> uint64_t {
        return static_cast<uint64_t>((gridDim.x + kClaimParts - 1u - k) / kClaimParts) * waves_per_block * first_paths;
    };
    uint32_t parts_done = 0;
    bool first = true;
    // paths this wavefront may hold, and the smoothed rounds of one per bounce
    uint32_t limit = kShared ? first_paths : 64u, work = 0;

    while (true) {
        // ---- claim new paths for idle lanes: one atomic per wavefront and part tried ----
        const unsigned long long idle = __builtin_amdgcn_ballot_w64(!alive);
        const uint32_t busy = 64u - static_cast<uint32_t>(__popcll(idle));
        const uint32_t lanes = limit < 64u ? limit : 64u;
        uint32_t room = lanes > busy ? lanes - busy : 0u;
        const uint32_t regen_min = hand_out >> 24;
        const uint32_t claim_min = regen_min < (limit + 1u) / 2u ? regen_min : (limit + 1u) / 2u;
        if (!exhausted && room != 0u && (room >= claim_min || busy == 0u)) {
            const uint32_t most = (limit > 64u ? hand_out >> 16 : hand_out >> 8) & 0xffu;
            if (kShared && room > most) room = most;
            const uint32_t leader = static_cast<uint32_t>(__builtin_ctzll(idle));
            unsigned long long base = 0;
            uint32_t got = 0;
            if (first) {
                const uint32_t k = blockIdx.x % kClaimParts;
                const uint64_t lo_k = path_lo + k * part;
                const uint64_t hi_k = lo_k + part < total_paths ? lo_k + part : total_paths;
                const uint32_t blocks_k = (gridDim.x + kClaimParts - 1u - k) / kClaimParts;
                base = lo_k + (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * blocks_k +
                               blockIdx.x / kClaimParts) * first_paths;
                if (base < hi_k) got = hi_k - base < first_paths ? static_cast<uint32_t>(hi_k - base) : first_paths;
                first = false;
            }
            if (got == 0u) {
                const uint32_t leader = static_cast<uint32_t>(__builtin_ctzll(idle));
                if (lane == leader) {
                    for (uint32_t t = 0; t < kClaimParts; ++t) {
                        const uint32_t k = (xcd + t) % kClaimParts;
                        if ((parts_done >> k) & 1u) continue;
                        const uint64_t lo_k = path_lo + k * part + part_static(k);
                        const uint64_t end_k = path_lo + (k + 1u) * part;
                        const uint64_t hi_k = end_k < total_paths ? end_k : total_paths;
                        if (lo_k < hi_k) {
                            const unsigned long long c =
                                __hip_atomic_fetch_add(path_counter + k * kClaimStride,
                                                       static_cast<unsigned long long>(room), __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT);
                            const uint64_t b = lo_k + c;
                            if (b < hi_k) {
                                base = b;
                                got = hi_k - b < room ? static_cast<uint32_t>(hi_k - b) : room;
                                break;
                            }
                        }
                        parts_done |= 1u << k;
                    }
                }
                base = __shfl(base, leader);
                got = __builtin_amdgcn_readfirstlane(__shfl(got, leader));
                parts_done = __builtin_amdgcn_readfirstlane(__shfl(parts_done, leader));
            }
            // every part used up: this wavefront claims no more
            if (got == 0u) exhausted = true;
            const uint32_t rank = lanes_below(idle);
            if (!alive && rank < got) {
                const uint64_t p = base + rank;
                // ---- path setup (raygen.cuh:72-113) ----
                const uint32_t j = find_job(job_begin, njobs, p);
                const JobDesc& J = jobs[j];
                if (path_begin(J, p - J.path_begin, st.o, st.d, st.rng, st.key, st.pix, st.sl)) {
                    st.beta = mk(1.0f);
                    st.L = mk(0.0f);
                    st.bounce = 0;
                    st.job = j;
                    st.cur = 0;
                    // origin-inside set (sampling.cuh:322-341) by point query
                    uint32_t na = 0, ov = 0, visits = 0, tests = 0;
                    const SceneView sc = J.scene;
                    const f3 o = st.o;
                    walk_point(sc, o, visits, [&](uint32_t prim) {
                        ++tests;
                        if (point_inside(load_prim(sc.prims, prim), o)) {
                            // counters updated without a branch keep them in registers
                            const bool fits = na < cap;
                            if (fits) my[na * stride] = prim;
                            na += fits ? 1u : 0u;
                            overflow += fits ? 0u : 1u;
                            ++ov;
                        }
                    });
                    st.na = na;
                    ev.add(kCntNodeVisits, visits);
                    ev.add(kCntVisitsPoint, visits);
                    ev.add(kCntContain, tests);
                    ev.add(kCntPaths);
                    if constexpr (kMeasure) max_overlap = ov > max_overlap ? ov : max_overlap;
                    alive = true;
                }
            }
        }
        if (__builtin_amdgcn_ballot_w64(alive) == 0) {
            if (exhausted) break;
            continue;
        }
        if constexpr (!kShared)
            if (!alive) continue;

        // ---- one bounce (raygen.cuh:115-208) ----
        const JobDesc& J = jobs[st.job];
        const SceneView sc = J.scene;
        const f3 o = st.o, d = st.d;
        const uint32_t b = st.bounce;
        uint32_t* act = my + (st.cur * bs) * stride;
        uint32_t* nxt = my + ((st.cur ^ 1u) * bs) * stride;
        const uint32_t na = st.na;
        bool finish = false;

        // At bounce 0 the analytic direct term needs the transmittance of the
        // camera ray itself, so it is integrated during the argmin (the walk
        // then runs over the whole ray instead of stopping at the running
        // minimum): the same chords, summed in the same fixed point as a
        // shadow ray's.  The counting build keeps the separate shadow walk, so
        // its counts are per-ray work.
        const bool direct = kShared && alive && b == 0;

        float ts = kTMax;
        // the origin-set members' exits, kept for the rebuild
        float* act_exit = kShared ? reinterpret_cast<float*>(nxt) : reinterpret_cast<float*>(my + 5 * bs * stride);
        ev.add(kCntArgActive, na);
        ev.add(kCntTrace);
        // argmin over the origin set (sampling.cuh:356-370) and over entered
        // primitives (sampling.cuh:372-412) in one walk; primitives entered
        // before the running minimum are kept as rebuild candidates (every
        // primitive entered before the final minimum is among them, because
        // the walk only prunes beyond the running one)
        uint32_t* cnd = my + 2 * bs * stride;
        uint32_t nc = 0;
        // the analytic direct term's factor and its roulette (a no-op unless
        // J.shadow_rr > 0): the walk that integrates its depth needs only the
        // depth where the term becomes 0; both are formed again after the
        // walk (the same values), so they hold no registers during it
        auto direct_rr = [&](f3& kd) {
            kd = st.beta * env_lookup(env_view(J.env), d);
            return shadow_rr(max3(kd), J.shadow_rr, st.key, 0u, 2u);
        };
        uint64_t dwalk = 0;
        WaveScene ws{};
        uint32_t rounds = 0;
        const uint32_t nalive = static_cast<uint32_t>(__popcll(__builtin_amdgcn_ballot_w64(alive)));
        if constexpr (kShared) {
            ws = wave_scene(sc, alive, jobs);
            uint64_t dlimit = kTauLimitFixed;
            if (direct) {
                f3 kd;
                dlimit = direct_rr(kd).limit();
            }
            uint32_t hits = 0;
            argmin_walk_shared<kMeasure>(alive, ws, st.job, o, d, st.key, b, direct, act, na, act_exit, st.ts_set, slab,
                                         cap, q, ts, nc, dlimit, dwalk, rounds, s_leafq, hits);
            if constexpr (kMeasure) max_hits = alive && hits > max_hits ? hits : max_hits;
        } else {
            for (uint32_t k = 0; k < na; ++k) {
                const uint32_t i = act[k * stride];
                const PrimRecord pr = load_prim(sc.prims, i);
                const InsideChord x = inside_chord(pr, o, d);
                act_exit[k * stride] = x.t1;
                const float tau = free_flight_tau(prim_uniform(st.key, b, 0u, i));
                if (tau <= x.tau) ts = minf(ts, origin_flight(pr, o, d, x, tau));
            }
            const f3 inv = safe_inv(d);
            const bool prune = !kMeasure;
            float tmax = prune ? ts : kTMax;
            uint32_t hits = 0, visits = 0, leaves = 0, accept = 0;
            walk_ray_q(sc, o, inv, tmax, visits, lq, [&](uint32_t prim) -> bool {
                const PrimRecord pr = load_prim(sc.prims, prim);
                ++leaves;
                const Crossing x = crossing(pr, o, d);
                if (x.t0 < 0.0f) return true;
                ++hits;
                // beyond the running minimum nothing below can change
                // (t >= entry > ts)
                if (x.t0 > ts) return true;
                if (nc < cap) {
                    cnd[nc * stride] = prim;
                    my[(3 * bs + nc) * stride] = __float_as_uint(x.t0);
                    my[(4 * bs + nc) * stride] = __float_as_uint(x.t1);
                }
                ++nc;
                const float tau = free_flight_tau(prim_uniform(st.key, b, 1u, prim));
                if (tau <= x.tau) {
                    ++accept;
                    const float t = entered_flight(pr, o, d, x, tau);
                    if (t < ts) {
                        ts = t;
                        if (prune) tmax = ts;
                    }
                }
                return true;
            });
            ev.add(kCntArgHit, hits);
            ev.add(kCntArgAccept, accept);
            ev.add(kCntNodeVisits, visits);
            ev.add(kCntLeafTests, leaves);
            if constexpr (kMeasure) max_hits = hits > max_hits ? hits : max_hits;
        }

        const EnvView env = env_view(J.env);
        // analytic direct term at bounce 0 (raygen.cuh:148-160)
        if (alive && b == 0) {
            ev.add(kCntShadowRays);
            f3 kd;
            const ShadowRr drr = direct_rr(kd);
            uint64_t a;
            if constexpr (kCount) a = shadow_depth(sc, o, d, act, na, stride, lq, ev, drr.limit());
            else a = dwalk;
            const float T = shadow_rr_T(a, drr, depth_T(a));
            st.L = st.L + kd * T;
        }

        // The vertex of a path that scatters: its active set, the next
        // direction and the NEE shadow rays (rays a and b of MIS, or ray a of
        // RIS; a limit of 0 is no ray), whose depths are summed below.
        const bool vertex = alive && ts < kTMax;
        if (alive && !vertex) finish = true;  // escape: with NEE + analytic direct nothing more is added
        f3 x = mk(0.0f), wo = mk(0.0f), da = mk(0.0f), db = mk(0.0f), ka = mk(0.0f), kb = mk(0.0f);
        uint32_t nn = 0;
        uint64_t lim_a = 0, lim_b = 0;
        bool has_a = false, has_b = false;
        // the sampled directions' densities (MIS); pdf_a is RIS's weight sum
        // and ka its candidate's radiance until the albedo is known
        float pdf_a = 0.0f, pdf_b = 0.0f;
        const f3 luma = f3{kLumR, kLumG, kLumB};
        // the shadow rays' roulettes (a no-op unless J.shadow_rr > 0) are
        // drawn before and again after the walks (the same values), so they
        // hold no registers during them
        auto nee_rr = [&](f3 k, uint32_t ray) { return shadow_rr(max3(k), J.shadow_rr, st.key, b, ray); };
        // rebuild the active set at the scatter point (sampling.cuh:422-458):
        // from the candidates of the argmin walk, or, if they were more than
        // fit (and in the counting build), by a point query
        const bool listed = kShared && nc <= cap;
        if constexpr (kShared)
            nn = rebuild_shared(vertex && listed, na, nc, st.cur, ts, slab, cap, q, overflow);
        if (vertex) {
            x = o + ts * d;
            if (!listed) {
                uint32_t ia = 0, visits = 0, rb_a = 0, rb_h = 0;
                // (the timed kernel's exits are in nxt: its set is built in
                // buffer 5 and copied)
                uint32_t* out = kShared ? my + 5 * bs * stride : nxt;
                nn = 0;
                auto push = [&](uint32_t v) {
                    const bool fits = nn < cap;
                    if (fits) out[nn * stride] = v;
                    nn += fits ? 1u : 0u;
                    overflow += fits ? 0u : 1u;
                };
                // old member ia stays while the vertex is before its exit (kept
                // from the argmin's origin loop)
                auto keep_member = [&]() {
                    ++rb_a;
                    const bool k = ts <= act_exit[ia * stride];
                    ++ia;
                    return k;
                };
                auto drain_below = [&](uint32_t c) {
                    while (ia < na) {
                        const uint32_t a = act[ia * stride];
                        if (a >= c) break;
                        if (keep_member()) push(a);
                    }
                };
                // a candidate: an old member kept while the vertex is inside
                // it, else an entered primitive kept if the vertex lies on its
                // chord (entry and exit as the argmin recorded them, or
                // computed here for the point query)
                auto visit = [&](uint32_t c, bool stored, float tj, float te) {
                    bool keep = false;
                    if (ia < na && act[ia * stride] == c) keep = keep_member();
                    if (!keep) {
                        ++rb_h;
                        if (!stored) {
                            const Crossing cx = crossing(load_prim(sc.prims, c), o, d);
                            tj = cx.t0;
                            te = cx.t1;
                        }
                        keep = tj >= 0.0f && tj <= ts && ts <= te;
                    }
                    if (keep) push(c);
                };
                if (!kShared && !kMeasure && nc <= cap) {
                    // candidates from the argmin walk, in ascending index order
                    float* ctj = reinterpret_cast<float*>(my + 3 * bs * stride);
                    float* cte = reinterpret_cast<float*>(my + 4 * bs * stride);
                    for (uint32_t i = 1; i < nc; ++i) {
                        const uint32_t v = cnd[i * stride];
                        const float vt = ctj[i * stride], ve = cte[i * stride];
                        uint32_t j = i;
                        while (j > 0 && cnd[(j - 1) * stride] > v) {
                            cnd[j * stride] = cnd[(j - 1) * stride];
                            ctj[j * stride] = ctj[(j - 1) * stride];
                            cte[j * stride] = cte[(j - 1) * stride];
                            --j;
                        }
                        cnd[j * stride] = v;
                        ctj[j * stride] = vt;
                        cte[j * stride] = ve;
                    }
                    for (uint32_t k = 0; k < nc; ++k) {
                        const uint32_t c = cnd[k * stride];
                        drain_below(c);
                        visit(c, true, ctj[k * stride], cte[k * stride]);
                    }
                } else {
                    // one BVH point query at the vertex
                    walk_point_q(sc, x, visits, lq, [&](uint32_t c) {
                        drain_below(c);
                        visit(c, false, 0.0f, 0.0f);
                    });
                }
                while (ia < na) {
                    const uint32_t a = act[ia * stride];
                    if (keep_member()) push(a);
                }
                if constexpr (kShared)
                    for (uint32_t k = 0; k < nn; ++k) nxt[k * stride] = out[k * stride];
                ev.add(kCntNodeVisits, visits);
                ev.add(kCntVisitsPoint, visits);
                ev.add(kCntRbActive, rb_a);
                ev.add(kCntRbHit, rb_h);
            }
            st.cur ^= 1u;
            st.na = nn;
            act = nxt;
            if constexpr (kMeasure) {
                uint32_t ovl = 0, v2 = 0;
                walk_point(sc, x, v2, [&](uint32_t c) { ovl += point_inside(load_prim(sc.prims, c), x) ? 1u : 0u; });
                max_overlap = ovl > max_overlap ? ovl : max_overlap;
            }

            // the next direction, then NEE's (accumulate_nee_direct,
            // path_stages.cuh:148-226): RIS picks one environment candidate,
            // MIS draws one direction from the phase function and one from
            // the environment
            float phase_pdf;
            wo = phase_sample(J.hg, d, st.rng, &phase_pdf);
            ev.add(kCntScatter);
            if (J.use_ris) {
                for (uint32_t c = 0; c < J.ris_candidates; ++c) {
                    float cpdf;
                    const f3 cwo = env_sample(env, st.rng, &cpdf);
                    if (cpdf <= 0.0f) continue;
                    const f3 envc = env_lookup(env, cwo);
                    const float lumc = dot(envc, luma);
                    const float wgt = phase_eval(J.hg, d, cwo) * lumc * rcpf(cpdf);
                    if (!(wgt > 0.0f)) continue;
                    pdf_a += wgt;
                    if (next_uniform(st.rng) * pdf_a < wgt) {
                        da = cwo;
                        ka = envc;
                    }
                }
                has_a = pdf_a > 0.0f && dot(ka, luma) > 0.0f;
            } else {
                da = phase_sample(J.hg, d, st.rng, &pdf_a);
                db = env_sample(env, st.rng, &pdf_b);
                has_a = has_b = true;
            }
        }

        // evaluate_albedo (sampling.cuh:257-283)
        f3 albedo;
        if constexpr (kShared) {
            albedo = vertex_members(nn, st.cur, has_a, has_b, ws, x, da, db, wo, st.key, b + 1u, slab, cap, q,
                                    st.ts_set);
        } else {
            f3 aa = mk(0.0f);
            float aw = 0.0f;
            for (uint32_t k = 0; k < nn; ++k) {
                const PrimRecord pr = load_prim(sc.prims, act[k * stride]);
                const float wgt = pr.mass * prim_pdf(pr, x);
                aa = aa + f3{pr.ar, pr.ag, pr.ab} * wgt;
                aw += wgt;
            }
            ev.add(kCntAlb, nn);
            albedo = aw <= 0.0f ? mk(0.0f) : aa * rcpf(aw);
        }
        if (vertex) {
            // the factors the shadow rays' transmittances multiply; base is
            // also the next bounce's throughput (raygen.cuh:189), set here so
            // the albedo holds no registers during the shadow walks
            const f3 base = st.beta * albedo;
            st.beta = base;
            if (J.use_ris) {
                if (has_a) {
                    ev.add(kCntShadowRays);
                    const float Wr = pdf_a * rcpf(static_cast<float>(J.ris_candidates));
                    ka = (base * (ka * rcpf(dot(ka, luma)))) * Wr;
                }
            } else {
                if constexpr (kShared) {
                    da = lds_load3(q.rd + 3 * (2 * lane));
                    db = lds_load3(q.rd + 3 * (2 * lane + 1));
                }
                const float pb_a = env_pdf(env, da);
                const float sa = pdf_a + pb_a;
                const float wa = sa > 0.0f ? pdf_a / sa : 0.0f;
                const f3 enva = env_lookup(env, da);
                const float ph_b = phase_eval(J.hg, d, db);
                const float sb = pdf_b + ph_b;
                const float wb = sb > 0.0f ? pdf_b / sb : 0.0f;
                const f3 envb = env_lookup(env, db);
                ev.add(kCntShadowRays, 2);
                ka = (base * enva) * wa;
                kb = (((base * envb) * wb) * ph_b) * rcpf(pdf_b);
            }
            if (has_a) lim_a = nee_rr(ka, 0u).limit();
            if (has_b) lim_b = nee_rr(kb, 1u).limit();
        }

        // the shadow rays' depths (the counting build walks them one by one,
        // so its counts are per-ray work)
        uint64_t acc_a = 0, acc_b = 0;
        if constexpr (kShared) {
            shadow_walks(ws, s_leafq, q, lim_a, lim_b, acc_a, acc_b, rounds);
            // the bounce's rounds per path, smoothed over bounces, in sixteenths
            work = (3u * work + 16u * rounds / nalive) / 4u;
            limit = 16u * rounds_target / (work + 1u);
            const uint32_t all = ws.leaf_base <= w4_level_base(5u) ? 65u : 64u;
            limit = limit < kPathsMin ? kPathsMin : (limit < 64u ? limit : all);
        } else {
            if (has_a) acc_a = shadow_depth(sc, x, da, act, nn, stride, lq, ev, lim_a);
            if (has_b) acc_b = shadow_depth(sc, x, db, act, nn, stride, lq, ev, lim_b);
        }

        if (vertex) {
            if (has_a) st.L = st.L + ka * shadow_rr_T(acc_a, nee_rr(ka, 0u), depth_T(acc_a));
            if (has_b) st.L = st.L + kb * shadow_rr_T(acc_b, nee_rr(kb, 1u), depth_T(acc_b));

            // russian_roulette (path_stages.cuh:25-37) and guards (raygen.cuh:191-204)
            if (b >= J.rr_depth) {
                const float ps = minf(J.rr_max_survival, max3(st.beta));
                if (next_uniform(st.rng) > ps || ps <= 0.0f) finish = true;
                else st.beta = st.beta * rcpf(ps);
            }
            if (!finish && max3(st.beta) < kMinThroughput) finish = true;
            if (!finish && !isfinitef_(sum3(st.beta))) finish = true;
            if (!finish) {
                st.o = x;
                st.d = wo;
                st.bounce = b + 1;
                if (st.bounce >= J.max_depth) finish = true;
            }
        }

        if (finish) {
            path_finish(J, st.pix, st.sl, st.L);
            alive = false;
            ev.flush(counters);
        }
    }
    if (overflow) atomicAdd(&counters[kCntActiveOverflow], static_cast<unsigned long long>(overflow));
    if constexpr (kMeasure) {
        // The maxima once per wavefront, and only where they raise the counter:
        // an atomic of every lane and bounce on one line bounded the renders of
        // short paths (512x512x8: one Gaussian 2.23 -> 1.31 ms, 4096 at
        // max_depth 1 8.8 -> 8.4).
        auto raise = [&](CounterSlot k, uint32_t v) {
            for (int off = 32; off > 0; off >>= 1) {
                const uint32_t u = __shfl_xor(v, off);
                v = u > v ? u : v;
            }
            if (lane == 0u && v > __hip_atomic_load(&counters[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicMax(&counters[k], static_cast<unsigned long long>(v));
        };
        raise(kCntMaxHits, max_hits);
        raise(kCntMaxOverlap, max_overlap);
    }
    if constexpr (kShared) help_walks<kMeasure>(s_leafq, jobs, slab, cap);
}

// Adaptive sampling, after a batch (the slice of J): the batch's samples of
// pixel i, in sample order, are folded into its Welford mean and M2 as the
// reference's raygen does per sample (raygen.cuh:214-233: n_inv =
// 1/(prev + s + 1), delta1 = x - mean, mean += delta1 n_inv, M2 += delta1
// (x - mean)), and the convergence test the reference runs at the start of
// the next batch (raygen.cuh:53-69: n >= min samples and max over channels
// of sqrt(M2/(n-1)) / max(mean, 1e-6) below the threshold) sets bit 31 of
// the state, so the next batch skips the pixel.  A converged pixel traced
// nothing in this batch and keeps its state.
__device__ __forceinline__ void fold_pixel(const JobDesc& J, uint32_t i) {
    const uint32_t st = J.adapt_state[i];
    if ((st >> 31) != 0u) return;
    const size_t npix = static_cast<size_t>(J.width) * J.height;
    float4 m = J.mean[i], m2 = J.adapt_m2[i];
    float mean[3] = {m.x, m.y, m.z}, M2[3] = {m2.x, m2.y, m2.z};
    for (uint32_t k = 0; k < J.s_count; ++k) {
        const float4 v = J.samples[k * npix + i];
        const float x[3] = {v.x, v.y, v.z};
        const float n_inv = 1.0f / static_cast<float>(st + k + 1u);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float d1 = x[c] - mean[c];
            mean[c] = mean[c] + d1 * n_inv;
            M2[c] = M2[c] + d1 * (x[c] - mean[c]);
        }
    }
    const uint32_t n = st + J.s_count;
    bool conv = false;
    if (n >= J.adapt_min) {
        const float r = 1.0f / static_cast<float>(n - 1u);
        float err = 0.0f;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float e = sqrtf_(M2[c] * r) / maxf(mean[c], 1e-6f);
            err = c == 0 ? e : maxf(err, e);
        }
        conv = err < J.adapt_threshold;
    }
    J.mean[i] = make_float4(mean[0], mean[1], mean[2], 1.0f);
    J.adapt_m2[i] = make_float4(M2[0], M2[1], M2[2], 0.0f);
    J.adapt_state[i] = n | (conv ? 0x80000000u : 0u);
}

// The mean of every pixel of job-table entry J from its accumulator
// (raygen.cuh:214-238 keeps a running mean; here the sums are exact and the
// division happens once).  Alpha is 1, as the reference writes it.  Under
// adaptive sampling the batch is folded instead.
__device__ __forceinline__ void resolve_pixel(const JobDesc& J, uint32_t i) {
    if (J.adapt_state != nullptr) {
        fold_pixel(J, i);
        return;
    }
    const unsigned long long* a = J.accum + static_cast<size_t>(i) * kAccumWords;
    const uint64_t n = a[3];
    J.mean[i] = make_float4(accum_mean(a[0], a[4], n), accum_mean(a[1], a[5], n), accum_mean(a[2], a[6], n), 1.0f);
}

// Resolve every entry of the launch's job table: blockIdx.y picks the entry;
// blocks beyond the table's length or the entry's pixels exit.  Entries that
// are slices of one job (the same accumulator) write the same values.
__global__ void k_resolve_all(const JobDesc* __restrict__ jobs, const uint64_t* __restrict__ launch_desc) {
    const uint32_t j = blockIdx.y;
    if (j >= static_cast<uint32_t>(launch_desc[0])) return;
    const JobDesc& J = jobs[j];
    const uint32_t npix = J.width * J.height;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < npix; i += gridDim.x * blockDim.x) resolve_pixel(J, i);
}

__global__ void k_resolve_job(const JobDesc* __restrict__ jobs, uint32_t j) {
    const JobDesc& J = jobs[j];
    const uint32_t npix = J.width * J.height;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < npix; i += gridDim.x * blockDim.x) resolve_pixel(J, i);
}

__global__ void k_fill_u64(unsigned long long* p, uint32_t n, unsigned long long v) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void k_fill_u32(uint32_t* p, uint32_t n, uint32_t v) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Start of a step.  The tables are read straight from pinned memory: one
// launch instead of three copies and three fills, which with the image's
// copies and the allocations took 100 of the 160 us of the smallest renders.
__global__ void __launch_bounds__(256) k_begin(const uint32_t* __restrict__ jobs_from, uint32_t* __restrict__ jobs, uint32_t job_words,
                        const uint64_t* __restrict__ begin_from, uint64_t* __restrict__ job_begin, uint32_t njobs,
                        const uint64_t* __restrict__ desc_from, uint64_t* __restrict__ desc,
                        unsigned long long* __restrict__ path_counter, unsigned long long* __restrict__ counters,
                        uint32_t n_counters, uint4* __restrict__ accum, size_t accum_n) {
    const size_t t = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x;
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (size_t i = t; i < job_words; i += stride) jobs[i] = jobs_from[i];
    for (size_t i = t; i < njobs; i += stride) job_begin[i] = begin_from[i];
    if (t < 3) desc[t] = desc_from[t];
    for (size_t i = t; i < kClaimWords; i += stride) path_counter[i] = 0ull;
    if (t < n_counters) counters[t] = 0ull;
    for (size_t i = t; i < accum_n; i += stride) accum[i] = make_uint4(0u, 0u, 0u, 0u);
}

__global__ void __launch_bounds__(256) k_copy_parts(CopyParts c) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
#pragma unroll
    for (uint32_t k = 0; k < kCopyParts; ++k)
        for (uint32_t i = t; i < c.words[k]; i += stride) c.dst[k][i] = c.src[k][i];
}

// normalize_accumulator_kernel (device/kernels/normalize_accumulator.cu:16-35)
__global__ void k_normalize(float4* __restrict__ out, const float4* __restrict__ in, size_t n, float scale) {
    for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const float4 v = in[i];
        out[i] = make_float4(v.x * scale, v.y * scale, v.z * scale, v.w * scale);
    }
}

// Transmittance along fixed rays, origin set = every primitive containing the
// origin (the bounce-0 scan), no capacity limit.
__global__ void k_transmittance_rays(SceneView sc, const float* __restrict__ rays, uint32_t m, float* __restrict__ T) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= m) return;
    const f3 o = f3{rays[6 * r], rays[6 * r + 1], rays[6 * r + 2]};
    const f3 d = f3{rays[6 * r + 3], rays[6 * r + 4], rays[6 * r + 5]};
    uint64_t acc = 0;
    bool full = false;
    uint32_t visits = 0;
    walk_point(sc, o, visits, [&](uint32_t prim) {
        const PrimRecord pr = load_prim(sc.prims, prim);
        if (full || !point_inside(pr, o)) return;
        if (tau_add(acc, inside_chord(pr, o, d).tau)) full = true;
    });
    if (!full) {
        const f3 inv = safe_inv(d);
        const float tmax = kTMax;
        walk_ray(sc, o, inv, tmax, visits, [&](uint32_t prim) -> bool {
            const Crossing x = crossing(load_prim(sc.prims, prim), o, d);
            if (x.t0 < 0.0f) return true;
            if (tau_add(acc, x.tau)) {
                full = true;
                return false;
            }
            return true;
        });
    }
    T[r] = full ? 0.0f : tau_to_T(acc);
}

// Entry list of each ray (collect_hits, sampling.cuh:287-305) sorted by (t, index).
__global__ void k_overlaps(SceneView sc, const float* __restrict__ rays, uint32_t m, uint32_t cap,
                           uint32_t* __restrict__ counts, float* __restrict__ tout, uint32_t* __restrict__ iout) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= m) return;
    const f3 o = f3{rays[6 * r], rays[6 * r + 1], rays[6 * r + 2]};
    const f3 d = f3{rays[6 * r + 3], rays[6 * r + 4], rays[6 * r + 5]};
    float* tr = tout + static_cast<size_t>(r) * cap;
    uint32_t* ir = iout + static_cast<size_t>(r) * cap;
    uint32_t c = 0, visits = 0;
    const f3 inv = safe_inv(d);
    const float tmax = kTMax;
    walk_ray(sc, o, inv, tmax, visits, [&](uint32_t prim) -> bool {
        const float tj = entry_t(load_prim(sc.prims, prim), o, d);
        if (tj < 0.0f) return true;
        if (c < cap) {
            uint32_t k = c;
            while (k > 0 && (tr[k - 1] > tj || (tr[k - 1] == tj && ir[k - 1] > prim))) {
                tr[k] = tr[k - 1];
                ir[k] = ir[k - 1];
                --k;
            }
            tr[k] = tj;
            ir[k] = prim;
        }
        ++c;
        return true;
    });
    counts[r] = c;
}

__global__ void k_math(int fn, const float* __restrict__ x, const float* __restrict__ y, uint32_t n,
                       float* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float a = x[i], b = y[i];
    float r;
    switch (fn) {
        case 0: r = expf_(a); break;
        case 1: r = logf_(a); break;
        case 2: r = sinf_(a); break;
        case 3: r = cosf_(a); break;
        case 4: r = atan2f_(a, b); break;
        case 5: r = acosf_(a); break;
        case 6: r = erff_(a); break;
        case 7: r = erfcf_(a); break;
        case 8: r = erfinvf_(a); break;
        case 9: r = erf_diff_(a, b); break;
        case 10: r = sqrtf_(a); break;
        case 11: r = a / b; break;
        case 12: r = chord_poly_(a); break;
        case 13: r = rcpf(a); break;
        default: r = __builtin_nanf("");
    }
    out[i] = r;
}

// The records as vp_scene_export gives them: the reference's fields in its
// order, the inverse-CDF factor M dnf sqrt(pi/2) in word 11.
__global__ void k_export_records(const PrimRecord* __restrict__ in, uint32_t n, float4* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if ((i >> 2) >= n) return;
    float4 v = reinterpret_cast<const float4*>(in)[i];
    if ((i & 3u) == 2u) v.w *= kRootHalfPi;
    out[i] = v;
}

__global__ void k_prim(int fn, const PrimRecord* __restrict__ rec, const float* __restrict__ args, uint32_t m,
                       float* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    PrimRecord p = *rec;
    p.md = p.mass * p.dnf;  // (the exported record has the inverse-CDF factor there)
    const float* a = args + 9 * i;
    const f3 o = f3{a[0], a[1], a[2]}, d = f3{a[3], a[4], a[5]};
    float r;
    switch (fn) {
        case 0: r = inv_cdf(p, o, d, a[8]); break;
        case 1: r = inv_cdf_span(p, o, d, a[6], a[8]); break;
        case 2: r = optical_depth(p, o, d, a[6], a[7]); break;
        case 3: r = exit_from_inside(p, o, d); break;
        case 4: r = crossing(p, o, d).t0; break;
        case 5: {
            const Crossing x = crossing(p, o, d);
            r = x.t0 >= 0.0f ? x.t1 : -1.0f;
        } break;
        case 6: r = point_inside(p, o) ? 1.0f : 0.0f; break;
        case 7: r = prim_pdf(p, o); break;
        case 8: r = crossing(p, o, d).tau; break;
        case 9: r = entered_flight(p, o, d, crossing(p, o, d), a[8]); break;
        case 10: r = inside_chord(p, o, d).tau; break;
        case 11: r = origin_flight(p, o, d, inside_chord(p, o, d), a[8]); break;
        default: r = __builtin_nanf("");
    }
    out[i] = r;
}

using RenderKernel = void (*)(const JobDesc*, const uint64_t*, const uint64_t*, unsigned long long*, uint32_t*,
                              uint32_t, uint32_t, uint32_t, unsigned long long*);
RenderKernel render_kernel(int count_events, int measure) {
    if (count_events) return measure ? k_render<true, true> : k_render<true, false>;
    return measure ? k_render<false, true> : k_render<false, false>;
}

inline uint32_t cdiv(uint64_t a, uint32_t b) { return static_cast<uint32_t>((a + b - 1) / b); }

}  // namespace
}  // namespace vp

using namespace vp;

// One persistent render launch over a job table (device pointers): the
// kernel claims the paths from launch_desc[2] below launch_desc[1], in
// kClaimParts parts with one counter each (counter[0 .. kClaimWords), zero at
// the start).
hipError_t vp_launch_render(const RenderLaunch& L, const JobDesc* jobs, const uint64_t* job_begin,
                            const uint64_t* launch_desc, unsigned long long* counter, uint32_t* slab,
                            unsigned long long* counters, hipStream_t s) {
    const size_t lds = mega_queue_bytes(L.block);
    const auto k = render_kernel(L.count_events, L.measure);
    hipLaunchKernelGGL(k, dim3(L.grid), dim3(L.block), lds, s, jobs, job_begin, launch_desc, counter, slab,
                       L.active_cap, L.first_paths | L.claim_step << 8 | L.claim_cheap << 16 | L.regen_min << 24,
                       L.rounds_target, counters);
    return hipGetLastError();
}

// One step of the persistent renderer over the job table in ctx->jobs_dev:
// trace every path of every job slice, resolve the means.  The table, its job
// count and path total (ctx->launch_desc) and the zeroed path counters are
// vp_launch_begin's.
hipError_t vp_launch_step(vp_context* ctx, const RenderLaunch& L, uint32_t max_jobs, uint32_t max_npix,
                          hipStream_t s) {
    const hipError_t e = vp_launch_render(L, ctx->jobs_dev, ctx->job_begin_dev, ctx->launch_desc, ctx->path_counter,
                                          ctx->slab, ctx->counters, s);
    if (e != hipSuccess) return e;
    return vp_launch_resolve(ctx, max_jobs, max_npix, s);
}

hipError_t vp_launch_resolve(vp_context* ctx, uint32_t max_jobs, uint32_t max_npix, hipStream_t s) {
    const uint32_t gx = std::max<uint32_t>(1u, std::min<uint32_t>(cdiv(max_npix, 256), 512u));
    hipLaunchKernelGGL(k_resolve_all, dim3(gx, max_jobs), dim3(256), 0, s, ctx->jobs_dev, ctx->launch_desc);
    return hipGetLastError();
}

hipError_t vp_launch_resolve_job(const JobDesc* jobs, uint32_t j, uint32_t npix, hipStream_t s) {
    const uint32_t gx = std::max<uint32_t>(1u, std::min<uint32_t>(cdiv(npix, 256), 1024u));
    hipLaunchKernelGGL(k_resolve_job, dim3(gx), dim3(256), 0, s, jobs, j);
    return hipGetLastError();
}

hipError_t vp_launch_begin(vp_context* ctx, uint32_t max_jobs, bool first, unsigned long long* accum,
                           size_t accum_words, hipStream_t s) {
    const uint32_t job_words = static_cast<uint32_t>(sizeof(JobDesc) / sizeof(uint32_t)) * max_jobs;
    const size_t accum_n = first ? accum_words / 2 : 0;  // kAccumWords is even
    const size_t most = std::max<size_t>(std::max<size_t>(job_words, kClaimWords), accum_n / 4);
    const uint32_t grid = static_cast<uint32_t>(std::min<size_t>((most + 255) / 256, 2048u));
    hipLaunchKernelGGL(k_begin, dim3(grid), dim3(256), 0, s, reinterpret_cast<const uint32_t*>(ctx->jobs_pinned),
                       reinterpret_cast<uint32_t*>(ctx->jobs_dev), job_words, ctx->begin_pinned, ctx->job_begin_dev,
                       max_jobs, ctx->desc_pinned, ctx->launch_desc, ctx->path_counter, ctx->counters,
                       first ? static_cast<uint32_t>(kNumCounters) : 0u, reinterpret_cast<uint4*>(accum), accum_n);
    return hipGetLastError();
}
hipError_t vp_launch_copy_parts(const CopyParts& c, hipStream_t s) {
    uint32_t most = 1;
    for (uint32_t w : c.words) most = std::max(most, w);
    hipLaunchKernelGGL(k_copy_parts, dim3(std::min<uint32_t>(cdiv(most, 256), 256u)), dim3(256), 0, s, c);
    return hipGetLastError();
}

hipError_t vp_launch_fill_u64(unsigned long long* p, uint32_t n, unsigned long long v, hipStream_t s) {
    hipLaunchKernelGGL(k_fill_u64, dim3(cdiv(n, 64)), dim3(64), 0, s, p, n, v);
    return hipGetLastError();
}
hipError_t vp_launch_fill_u32(uint32_t* p, uint32_t n, uint32_t v, hipStream_t s) {
    hipLaunchKernelGGL(k_fill_u32, dim3(cdiv(n, 256)), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

int vp_render_occupancy(uint32_t block, uint32_t, int count_events, int* blocks_per_cu) {
    int nb = 0;
    hipError_t e;
    const size_t lds = mega_queue_bytes(block);
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &nb, reinterpret_cast<const void*>(render_kernel(count_events, 0)), block, lds);
    *blocks_per_cu = nb > 0 ? nb : 1;
    return e == hipSuccess ? 0 : -1;
}

hipError_t vp_launch_normalize(float4* out, const float4* in, size_t n, float scale, hipStream_t s) {
    const uint32_t grid = std::min<uint32_t>(cdiv(n, 256), 1024u);
    hipLaunchKernelGGL(k_normalize, dim3(grid ? grid : 1), dim3(256), 0, s, out, in, n, scale);
    return hipGetLastError();
}

hipError_t vp_launch_transmittance(SceneView sc, const float* rays, uint32_t m, float* T, hipStream_t s) {
    hipLaunchKernelGGL(k_transmittance_rays, dim3(cdiv(m, 128)), dim3(128), 0, s, sc, rays, m, T);
    return hipGetLastError();
}

hipError_t vp_launch_overlaps(SceneView sc, const float* rays, uint32_t m, uint32_t cap, uint32_t* counts, float* t,
                              uint32_t* idx, hipStream_t s) {
    hipLaunchKernelGGL(k_overlaps, dim3(cdiv(m, 128)), dim3(128), 0, s, sc, rays, m, cap, counts, t, idx);
    return hipGetLastError();
}

hipError_t vp_launch_math(int fn, const float* x, const float* y, uint32_t n, float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_math, dim3(cdiv(n, 256)), dim3(256), 0, s, fn, x, y, n, out);
    return hipGetLastError();
}

hipError_t vp_launch_export_records(const PrimRecord* prims, uint32_t n, float4* out, hipStream_t s) {
    hipLaunchKernelGGL(k_export_records, dim3(cdiv(uint64_t(4) * n, 256)), dim3(256), 0, s, prims, n, out);
    return hipGetLastError();
}

hipError_t vp_launch_prim(int fn, const PrimRecord* rec, const float* args, uint32_t m, float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_prim, dim3(cdiv(m, 256)), dim3(256), 0, s, fn, rec, args, m, out);
    return hipGetLastError();
}
