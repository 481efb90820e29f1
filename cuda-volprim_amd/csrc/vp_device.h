// vp_device.h — device building blocks shared by the render kernels:
// record loads, the stackless walks of single lanes (plain and with a leaf
// queue in LDS), the wave-wide walks of the megakernel (a node stack in LDS) and
// the help between wavefronts, fixed-point optical depth, event counters and
// the job lookup.  Included by vp_render.hip (megakernel, test kernels) and
// vp_wavefront.hip (wavefront pipeline).
#pragma once

#include "vp_internal.h"

namespace vp {
namespace {

constexpr float kTauInvScale = 1.0f / 1099511627776.0f;

__device__ __forceinline__ f3 safe_inv(f3 d) {
    const float x = fabsf_(d.x) < 1e-20f ? copysignf_(1e-20f, d.x) : d.x;
    const float y = fabsf_(d.y) < 1e-20f ? copysignf_(1e-20f, d.y) : d.y;
    const float z = fabsf_(d.z) < 1e-20f ? copysignf_(1e-20f, d.z) : d.z;
    return f3{rcpf(x), rcpf(y), rcpf(z)};
}

// Scene arrays are reached through pointers stored in device memory (the job
// table), which the compiler can only treat as generic; they always point to
// global memory, and saying so turns flat loads into global loads (which do
// not wait on the LDS counter).
// (The host pass of the compiler only parses these device functions; the
// qualifier is applied in the device pass.)
#if defined(__HIP_DEVICE_COMPILE__)
#define VP_GLOBAL_AS __attribute__((address_space(1)))
#else
#define VP_GLOBAL_AS
#endif
template <typename T>
__device__ __forceinline__ const VP_GLOBAL_AS T* as_global(const T* p) {
    return (const VP_GLOBAL_AS T*)(p);
}

__device__ __forceinline__ PrimRecord load_prim(const PrimRecord* prims, uint32_t i) {
    const auto* p = as_global(reinterpret_cast<const float4*>(prims + i));
    const float4 a = p[0], b = p[1], c = p[2], d = p[3];
    PrimRecord r;
    r.cx = a.x; r.cy = a.y; r.cz = a.z; r.qw = a.w;
    r.qx = b.x; r.qy = b.y; r.qz = b.z; r.rsx = b.w;
    r.rsy = c.x; r.rsz = c.y; r.dnf = c.z; r.md = c.w;
    r.ar = d.x; r.ag = d.y; r.ab = d.z; r.mass = d.w;
    return r;
}

// The 48 bytes of record i that crossing() reads (albedo and mass are left at
// 0), loaded here: left alone, the compiler moves the load of what is used
// last to its use, behind the wait for the others.
template <typename Index>
__device__ __forceinline__ PrimRecord load_leaf(const PrimRecord* prims, Index i) {
    const auto* p = reinterpret_cast<const VP_GLOBAL_AS float4*>(
        reinterpret_cast<const VP_GLOBAL_AS char*>(as_global(prims)) + i * static_cast<Index>(sizeof(PrimRecord)));
    float4 a = p[0], b = p[1], c = p[2];
    asm volatile("" : "+v"(a.x), "+v"(a.y), "+v"(a.z), "+v"(a.w), "+v"(b.x), "+v"(b.y), "+v"(b.z), "+v"(b.w),
                      "+v"(c.x), "+v"(c.y), "+v"(c.z), "+v"(c.w));
    PrimRecord r{};
    r.cx = a.x; r.cy = a.y; r.cz = a.z; r.qw = a.w;
    r.qx = b.x; r.qy = b.y; r.qz = b.z; r.rsx = b.w;
    r.rsy = c.x; r.rsz = c.y; r.dnf = c.z; r.md = c.w;
    return r;
}

// number of set bits of m below the calling lane
__device__ __forceinline__ uint32_t lanes_below(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
}

// Hand-off point for data exchanged between lanes of one wavefront through
// LDS (queues, compaction, per-ray tables, steal slots): the wavefront-scope
// release/acquire pair keeps the compiler from moving LDS accesses across it
// (a lane's reads of entries other lanes write, and the reverse), and the
// wave barrier keeps the active lanes converged there.  The hardware already
// executes a wavefront's LDS operations in order.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Exclusive prefix sum over the wavefront's 64 lanes of v (every lane active),
// from one ballot per bit in use; total receives the sum.
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v, uint32_t& total) {
    uint32_t pre = 0;
    total = 0;
    for (uint32_t bit = 0; __builtin_amdgcn_ballot_w64((v >> bit) != 0u) != 0ull; ++bit) {
        const unsigned long long bm = __builtin_amdgcn_ballot_w64(((v >> bit) & 1u) != 0u);
        pre += lanes_below(bm) << bit;
        total += static_cast<uint32_t>(__popcll(bm)) << bit;
    }
    return pre;
}
// The lane that item g of a wavefront's flattened lists belongs to: the last
// one whose prefix (pre[64], ascending) is at most g.
__device__ __forceinline__ uint32_t prefix_owner(const uint32_t* pre, uint32_t g) {
    uint32_t lo = 0;
#pragma unroll
    for (uint32_t s = 32u; s > 0u; s >>= 1)
        if (pre[lo + s] <= g) lo += s;
    return lo;
}

// ---- walk-tree traversal (tree layout and Walk4 in vp_walk.h) ----

// Children of node n that the ray crosses within [0, tmax], as a 4-bit mask.
// Slab distances are fma(bound, 1/d, -o/d).  Which boxes a walk enters only
// decides what is visited (leaf boxes are conservative and the test is
// monotone in the box), never a result.
__device__ __forceinline__ bool slab_hit(float lx, float ly, float lz, float hx, float hy, float hz, f3 inv, f3 oi,
                                         float tmax) {
    const float tx0 = fmaf_(lx, inv.x, -oi.x), tx1 = fmaf_(hx, inv.x, -oi.x);
    const float ty0 = fmaf_(ly, inv.y, -oi.y), ty1 = fmaf_(hy, inv.y, -oi.y);
    const float tz0 = fmaf_(lz, inv.z, -oi.z), tz1 = fmaf_(hz, inv.z, -oi.z);
    const float tnear = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fmaxf(fminf(tz0, tz1), 0.0f));
    const float tfar = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fminf(fmaxf(tz0, tz1), tmax));
    return tnear <= tfar;
}
__device__ __forceinline__ uint32_t w4_ray_mask(const float4* w4, uint32_t n, f3 inv, f3 oi, float tmax) {
    const auto* r = as_global(w4) + static_cast<size_t>(kW4RecordF4) * n;
    const float4 lx = r[0], ly = r[1], lz = r[2], hx = r[3], hy = r[4], hz = r[5];
    return (slab_hit(lx.x, ly.x, lz.x, hx.x, hy.x, hz.x, inv, oi, tmax) ? 1u : 0u) |
           (slab_hit(lx.y, ly.y, lz.y, hx.y, hy.y, hz.y, inv, oi, tmax) ? 2u : 0u) |
           (slab_hit(lx.z, ly.z, lz.z, hx.z, hy.z, hz.z, inv, oi, tmax) ? 4u : 0u) |
           (slab_hit(lx.w, ly.w, lz.w, hx.w, hy.w, hz.w, inv, oi, tmax) ? 8u : 0u);
}

// The same mask with the near and far bound of each axis picked by the sign
// of the direction component, through the load address: since t is monotone
// in the bound, the near distance is exactly min(t(min), t(max)) and needs
// no min/max per axis.  A third fewer instructions per node, but six 64-bit
// addresses: faster where registers are spare (the wavefront walk kernels,
// +5 % on the scattering workload; the megakernel at 4 waves per SIMD),
// slower where they are not (the megakernel at 6 waves per SIMD: -20 %).
__device__ __forceinline__ uint32_t w4_ray_mask_nf(const float4* w4, uint32_t n, f3 inv, f3 oi, float tmax) {
    // byte offsets of the near bounds (min.x at 0, min.y 16, min.z 32,
    // max.x 48, max.y 64, max.z 80)
    const uint32_t fx = (__float_as_uint(inv.x) >> 31) * 48u;
    const uint32_t fy = (__float_as_uint(inv.y) >> 31) * 48u;
    const uint32_t fz = (__float_as_uint(inv.z) >> 31) * 48u;
    const auto* rec = reinterpret_cast<const VP_GLOBAL_AS char*>(as_global(w4) + static_cast<size_t>(kW4RecordF4) * n);
    const float4 nx = *reinterpret_cast<const VP_GLOBAL_AS float4*>(rec + fx);
    const float4 ny = *reinterpret_cast<const VP_GLOBAL_AS float4*>(rec + 16u + fy);
    const float4 nz = *reinterpret_cast<const VP_GLOBAL_AS float4*>(rec + 32u + fz);
    const float4 gx = *reinterpret_cast<const VP_GLOBAL_AS float4*>(rec + 48u - fx);
    const float4 gy = *reinterpret_cast<const VP_GLOBAL_AS float4*>(rec + 64u - fy);
    const float4 gz = *reinterpret_cast<const VP_GLOBAL_AS float4*>(rec + 80u - fz);
    auto hit = [&](float ax, float ay, float az, float bx, float by, float bz) {
        const float tn = fmaxf(fmaxf(fmaf_(ax, inv.x, -oi.x), fmaf_(ay, inv.y, -oi.y)),
                               fmaxf(fmaf_(az, inv.z, -oi.z), 0.0f));
        // (the clamp to tmax also rejects the +inf boxes of empty children
        // for a direction with all components positive)
        const float tf = fminf(fminf(fmaf_(bx, inv.x, -oi.x), fmaf_(by, inv.y, -oi.y)),
                               fminf(fmaf_(bz, inv.z, -oi.z), tmax));
        return tn <= tf;
    };
    return (hit(nx.x, ny.x, nz.x, gx.x, gy.x, gz.x) ? 1u : 0u) | (hit(nx.y, ny.y, nz.y, gx.y, gy.y, gz.y) ? 2u : 0u) |
           (hit(nx.z, ny.z, nz.z, gx.z, gy.z, gz.z) ? 4u : 0u) | (hit(nx.w, ny.w, nz.w, gx.w, gy.w, gz.w) ? 8u : 0u);
}

// ---- the same tests on 16-bit records (layout in vp_walk.h) ----
// The low and high binary16 of word w as float (exact).  As an FMA operand
// the conversion folds into v_fma_mix_f32, so a slab distance costs one
// instruction, as on 32-bit records, for half the bytes per node.
__device__ __forceinline__ float h16lo(uint32_t w) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w)));
}
__device__ __forceinline__ float h16hi(uint32_t w) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w >> 16)));
}
// record n of a 16-bit tree (kW4hRecordB = 4 float4)
__device__ __forceinline__ const VP_GLOBAL_AS uint4* w4h_record(const float4* w4, uint32_t n) {
    return reinterpret_cast<const VP_GLOBAL_AS uint4*>(as_global(w4) + 4u * static_cast<size_t>(n));
}
__device__ __forceinline__ uint32_t w4h_ray_mask(const float4* w4, uint32_t n, f3 inv, f3 oi, float tmax) {
    const auto* r = w4h_record(w4, n);
    // a = min.x (children 0,1 | 2,3), min.y; b = min.z, max.x; c = max.y, max.z
    const uint4 a = r[0], b = r[1], c = r[2];
    return (slab_hit(h16lo(a.x), h16lo(a.z), h16lo(b.x), h16lo(b.z), h16lo(c.x), h16lo(c.z), inv, oi, tmax) ? 1u
                                                                                                             : 0u) |
           (slab_hit(h16hi(a.x), h16hi(a.z), h16hi(b.x), h16hi(b.z), h16hi(c.x), h16hi(c.z), inv, oi, tmax) ? 2u
                                                                                                             : 0u) |
           (slab_hit(h16lo(a.y), h16lo(a.w), h16lo(b.y), h16lo(b.w), h16lo(c.y), h16lo(c.w), inv, oi, tmax) ? 4u
                                                                                                             : 0u) |
           (slab_hit(h16hi(a.y), h16hi(a.w), h16hi(b.y), h16hi(b.w), h16hi(c.y), h16hi(c.w), inv, oi, tmax) ? 8u
                                                                                                             : 0u);
}
// near/far form: the bounds of one axis and side are 8 bytes (min.x at 0,
// min.y 8, min.z 16, max.x 24, max.y 32, max.z 40)
__device__ __forceinline__ uint32_t w4h_ray_mask_nf(const float4* w4, uint32_t n, f3 inv, f3 oi, float tmax) {
    const uint32_t fx = (__float_as_uint(inv.x) >> 31) * 24u;
    const uint32_t fy = (__float_as_uint(inv.y) >> 31) * 24u;
    const uint32_t fz = (__float_as_uint(inv.z) >> 31) * 24u;
    const auto* rec = reinterpret_cast<const VP_GLOBAL_AS char*>(w4h_record(w4, n));
    const uint2 nx = *reinterpret_cast<const VP_GLOBAL_AS uint2*>(rec + fx);
    const uint2 ny = *reinterpret_cast<const VP_GLOBAL_AS uint2*>(rec + 8u + fy);
    const uint2 nz = *reinterpret_cast<const VP_GLOBAL_AS uint2*>(rec + 16u + fz);
    const uint2 gx = *reinterpret_cast<const VP_GLOBAL_AS uint2*>(rec + 24u - fx);
    const uint2 gy = *reinterpret_cast<const VP_GLOBAL_AS uint2*>(rec + 32u - fy);
    const uint2 gz = *reinterpret_cast<const VP_GLOBAL_AS uint2*>(rec + 40u - fz);
    auto hit = [&](float ax, float ay, float az, float bx, float by, float bz) {
        const float tn = fmaxf(fmaxf(fmaf_(ax, inv.x, -oi.x), fmaf_(ay, inv.y, -oi.y)),
                               fmaxf(fmaf_(az, inv.z, -oi.z), 0.0f));
        const float tf = fminf(fminf(fmaf_(bx, inv.x, -oi.x), fmaf_(by, inv.y, -oi.y)),
                               fminf(fmaf_(bz, inv.z, -oi.z), tmax));
        return tn <= tf;
    };
    return (hit(h16lo(nx.x), h16lo(ny.x), h16lo(nz.x), h16lo(gx.x), h16lo(gy.x), h16lo(gz.x)) ? 1u : 0u) |
           (hit(h16hi(nx.x), h16hi(ny.x), h16hi(nz.x), h16hi(gx.x), h16hi(gy.x), h16hi(gz.x)) ? 2u : 0u) |
           (hit(h16lo(nx.y), h16lo(ny.y), h16lo(nz.y), h16lo(gx.y), h16lo(gy.y), h16lo(gz.y)) ? 4u : 0u) |
           (hit(h16hi(nx.y), h16hi(ny.y), h16hi(nz.y), h16hi(gx.y), h16hi(gy.y), h16hi(gz.y)) ? 8u : 0u);
}

// The ray tests on either record form (half = the scene's w4_half).
__device__ __forceinline__ uint32_t ray_mask(const float4* w4, uint32_t half, uint32_t n, f3 inv, f3 oi,
                                             float tmax) {
    return half ? w4h_ray_mask(w4, n, inv, oi, tmax) : w4_ray_mask(w4, n, inv, oi, tmax);
}
__device__ __forceinline__ uint32_t ray_mask_nf(const float4* w4, uint32_t half, uint32_t n, f3 inv, f3 oi,
                                                float tmax) {
    return half ? w4h_ray_mask_nf(w4, n, inv, oi, tmax) : w4_ray_mask_nf(w4, n, inv, oi, tmax);
}

// The megakernel's node test: the near and far form on whole 16-byte words,
// the sides picked by selects after the load, since a load costs the L1 a
// cycle per lane whatever its size (three for a 16-bit record, where the form
// above makes six).  n: the node's index, 32 bits wide where the tree lies
// within 2^32 bytes (the address is then a scalar and an offset), else 64.
// hits(c, v): whether child c is crossed.
template <typename Index, typename Hits>
__device__ __forceinline__ void mega_ray_hits(const float4* w4, uint32_t half, Index n, f3 inv, f3 oi, float tmax,
                                              float (&tn4)[4], Hits&& hits) {
    const bool sx = inv.x < 0.0f, sy = inv.y < 0.0f, sz = inv.z < 0.0f;
    auto hit = [&](int c, float ax, float ay, float az, float bx, float by, float bz) {
        const float tn = fmaxf(fmaxf(fmaf_(ax, inv.x, -oi.x), fmaf_(ay, inv.y, -oi.y)),
                               fmaxf(fmaf_(az, inv.z, -oi.z), 0.0f));
        const float tf = fminf(fminf(fmaf_(bx, inv.x, -oi.x), fmaf_(by, inv.y, -oi.y)),
                               fminf(fmaf_(bz, inv.z, -oi.z), tmax));
        tn4[c] = tn <= tf ? tn : kTMax;
        hits(c, tn <= tf);
    };
    if (half) {
        const auto* r = reinterpret_cast<const VP_GLOBAL_AS uint4*>(
            reinterpret_cast<const VP_GLOBAL_AS char*>(as_global(w4)) + n * static_cast<Index>(kW4hRecordB));
        // a = min.x (children 0,1 | 2,3), min.y; b = min.z, max.x; c = max.y, max.z
        const uint4 a = r[0], b = r[1], c = r[2];
        auto pair = [&](int c, uint32_t lx, uint32_t ly, uint32_t lz, uint32_t hx, uint32_t hy, uint32_t hz) {
            const uint32_t ax = sx ? hx : lx, ay = sy ? hy : ly, az = sz ? hz : lz;
            const uint32_t bx = sx ? lx : hx, by = sy ? ly : hy, bz = sz ? lz : hz;
            hit(c, h16lo(ax), h16lo(ay), h16lo(az), h16lo(bx), h16lo(by), h16lo(bz));
            hit(c + 1, h16hi(ax), h16hi(ay), h16hi(az), h16hi(bx), h16hi(by), h16hi(bz));
        };
        pair(0, a.x, a.z, b.x, b.z, c.x, c.z);
        pair(2, a.y, a.w, b.y, b.w, c.y, c.w);
        return;
    }
    const auto* r = reinterpret_cast<const VP_GLOBAL_AS float4*>(
        reinterpret_cast<const VP_GLOBAL_AS char*>(as_global(w4)) + n * static_cast<Index>(16u * kW4RecordF4));
    const float4 lx = r[0], ly = r[1], lz = r[2], hx = r[3], hy = r[4], hz = r[5];
    auto one = [&](int c, float l0, float l1, float l2, float h0, float h1, float h2) {
        hit(c, sx ? h0 : l0, sy ? h1 : l1, sz ? h2 : l2, sx ? l0 : h0, sy ? l1 : h1, sz ? l2 : h2);
    };
    one(0, lx.x, ly.x, lz.x, hx.x, hy.x, hz.x);
    one(1, lx.y, ly.y, lz.y, hx.y, hy.y, hz.y);
    one(2, lx.z, ly.z, lz.z, hx.z, hy.z, hz.z);
    one(3, lx.w, ly.w, lz.w, hx.w, hy.w, hz.w);
}

// children of node n whose box contains x
__device__ __forceinline__ uint32_t point_mask(const float4* w4, uint32_t half, uint32_t n, f3 x) {
    auto in = [&](float l0, float l1, float l2, float h0, float h1, float h2) {
        return x.x >= l0 && x.x <= h0 && x.y >= l1 && x.y <= h1 && x.z >= l2 && x.z <= h2;
    };
    if (half) {
        const auto* r = w4h_record(w4, n);
        const uint4 a = r[0], b = r[1], c = r[2];
        return (in(h16lo(a.x), h16lo(a.z), h16lo(b.x), h16lo(b.z), h16lo(c.x), h16lo(c.z)) ? 1u : 0u) |
               (in(h16hi(a.x), h16hi(a.z), h16hi(b.x), h16hi(b.z), h16hi(c.x), h16hi(c.z)) ? 2u : 0u) |
               (in(h16lo(a.y), h16lo(a.w), h16lo(b.y), h16lo(b.w), h16lo(c.y), h16lo(c.w)) ? 4u : 0u) |
               (in(h16hi(a.y), h16hi(a.w), h16hi(b.y), h16hi(b.w), h16hi(c.y), h16hi(c.w)) ? 8u : 0u);
    }
    const auto* r = as_global(w4) + static_cast<size_t>(kW4RecordF4) * n;
    const float4 lx = r[0], ly = r[1], lz = r[2], hx = r[3], hy = r[4], hz = r[5];
    return (in(lx.x, ly.x, lz.x, hx.x, hy.x, hz.x) ? 1u : 0u) | (in(lx.y, ly.y, lz.y, hx.y, hy.y, hz.y) ? 2u : 0u) |
           (in(lx.z, ly.z, lz.z, hx.z, hy.z, hz.z) ? 4u : 0u) | (in(lx.w, ly.w, lz.w, hx.w, hy.w, hz.w) ? 8u : 0u);
}

// Walk over [0, tmax]; leaf(prim) returns false to stop.  tmax may be
// lowered by the caller between leaves.
template <typename Leaf>
__device__ __forceinline__ void walk_ray(const SceneView& s, f3 o, f3 inv, const float& tmax, uint32_t& visits,
                                         Leaf&& leaf) {
    const f3 oi = o * inv;
    Walk4 w = walk4_begin();
    while (w.n != kWalkEnd) {
        ++visits;
        const uint32_t m = ray_mask(s.w4, s.w4_half, w.n, inv, oi, tmax);
        uint32_t first;
        for (uint32_t lm = walk4_advance(w, s.w4_levels, m, first); lm != 0u; lm &= lm - 1u)
            if (!leaf(first + static_cast<uint32_t>(__builtin_ctz(lm)))) return;
    }
}

// Walk visiting every leaf whose box contains x, in ascending stored-primitive
// order.
template <typename Leaf>
__device__ __forceinline__ void walk_point(const SceneView& s, f3 x, uint32_t& visits, Leaf&& leaf) {
    Walk4 w = walk4_begin();
    while (w.n != kWalkEnd) {
        ++visits;
        const uint32_t m = point_mask(s.w4, s.w4_half, w.n, x);
        uint32_t first;
        for (uint32_t lm = walk4_advance(w, s.w4_levels, m, first); lm != 0u; lm &= lm - 1u)
            leaf(first + static_cast<uint32_t>(__builtin_ctz(lm)));
    }
}

// Leaf queue depth per lane.  The walks below postpone leaves into a per-lane
// LDS queue (row `thread` of a [blockDim][kLeafQ + 1] array: the odd row
// length puts the 64 lanes' entries k in distinct banks) and keep walking
// until every lane of the wavefront has a full queue or has finished; then all
// lanes process their queued leaves together.  Node steps stay convergent and
// the expensive leaf work runs with most lanes active (the "while-while"
// scheme of Aila and Laine 2009, with speculative postponing).
#ifndef VP_LEAF_Q
#define VP_LEAF_Q 16
#endif
constexpr uint32_t kLeafQ = VP_LEAF_Q;
constexpr uint32_t kLeafRow = kLeafQ + 1;

// Wave-shared leaf queue of the wavefront pipeline.  The LDS of a wavefront
// holds either its threads' queue rows or one queue for the whole wavefront
// (in different kernels): node phases append crossed leaves with their owner
// lane, and in the leaf phase every active lane takes the next entry, whichever
// lane's ray it belongs to.  Leaf work then runs at full width however
// unevenly the lanes' walks found leaves.  Per-ray results are combined with
// LDS atomics whose outcome does not depend on order (fixed-point sums, and
// minima).
#ifndef VP_WAVE_Q
#define VP_WAVE_Q 224
#endif
constexpr uint32_t kWaveQ = VP_WAVE_Q;
// A node phase of the shared-queue walks ends early, to share out the queued
// leaves, once the queue holds kWaveQ / 4 entries and fewer than
// VP_SHARED_STEP_MIN lanes still step.
#ifndef VP_SHARED_STEP_MIN
#define VP_SHARED_STEP_MIN VP_WALK_MIN
#endif
// (the queue fill, as a fraction 1 / VP_SHARED_END_DIV, from which that rule applies)
#ifndef VP_SHARED_END_DIV
#define VP_SHARED_END_DIV 4u
#endif
// A lane walks one ray; queued leaves belong to the lane of their ray.
struct WaveQueue {
    uint32_t* prim;                // [kWaveQ] queued leaf
    uint8_t* owner;                // [kWaveQ] the lane each leaf belongs to
    float* ro;                     // [64 * 3] ray origin of each lane
    const PrimRecord** prims;      // [64] primitive array of each lane's scene (lanes of one
                                   //      wavefront may run jobs over different scenes)
    float* rd;                     // [64 * 3] ray directions
    unsigned long long* acc;       // [64] fixed-point optical depth of each ray (shadow walks), or
    unsigned long long* key;       // [64] path key of each lane (argmin walks, as the rest)
    uint32_t* ts;                  // [64] running minimum of each lane's argmin, as float bits
    uint32_t* nc;                  // [64] candidates recorded for each lane's argmin
    uint32_t* meta;                // [64] bounce
    uint32_t* slot;                // [64] pool slot of each lane's path
};
constexpr uint32_t kWaveQueueBytes = kWaveQ * 5 + 64 * (12 + 8 + 12 + 8 + 4 * 4);
static_assert(kWaveQ % 8 == 0, "queue arrays keep the per-lane arrays 8-byte aligned");
// LDS bytes per wavefront: the larger of the two uses, in 16-byte units
constexpr uint32_t kWaveBytes =
    ((64 * kLeafRow * 4 > kWaveQueueBytes ? 64 * kLeafRow * 4 : kWaveQueueBytes) + 15) / 16 * 16;

// the calling wavefront's queue
__device__ __forceinline__ WaveQueue wave_queue(uint32_t* lds) {
    uint8_t* base = reinterpret_cast<uint8_t*>(lds) + (threadIdx.x >> 6) * kWaveBytes;
    WaveQueue q;
    q.prim = reinterpret_cast<uint32_t*>(base);
    q.owner = base + 4 * kWaveQ;
    q.ro = reinterpret_cast<float*>(base + 5 * kWaveQ);
    q.prims = reinterpret_cast<const PrimRecord**>(q.ro + 64 * 3);
    q.rd = reinterpret_cast<float*>(q.prims + 64);
    q.acc = q.key = reinterpret_cast<unsigned long long*>(q.rd + 64 * 3);
    q.ts = reinterpret_cast<uint32_t*>(q.key + 64);
    q.nc = q.ts + 64;
    q.meta = q.nc + 64;
    q.slot = q.meta + 64;
    return q;
}

__device__ __forceinline__ f3 lds_load3(const float* p) { return f3{p[0], p[1], p[2]}; }
__device__ __forceinline__ void lds_store3(float* p, f3 v) {
    p[0] = v.x;
    p[1] = v.y;
    p[2] = v.z;
}

// Node phase of the per-lane ray walk: a lane steps while its leaf queue has
// room for a step (up to four leaves) and its walk has nodes left.  With
// VP_WALK_MIN > 0 the loop runs for the whole wavefront, which leaves it early
// once fewer than VP_WALK_MIN lanes are stepping and some lane's queue is
// full, so full lanes do not wait for the last few; the stepping lanes resume
// after the leaf phase.  A node phase that starts with every queue empty can
// only end early after some lane has queued leaves, so walks always progress.
// Every query consumes leaves order-independently, so this changes only the
// schedule.
#ifndef VP_WALK_MIN
#define VP_WALK_MIN 8
#endif

// room in a lane's queue for one more node step
__device__ __forceinline__ bool queue_room(uint32_t cnt) { return cnt + 4u <= kLeafQ; }
// true while this lane (VP_WALK_MIN == 0) or the wavefront stays in the node
// phase (room: the lane's queue has room for its next step)
__device__ __forceinline__ bool node_phase(bool step, bool room) {
#if VP_WALK_MIN > 0
    const unsigned long long sm = __builtin_amdgcn_ballot_w64(step);
    if (sm == 0) return false;
    return __popcll(sm) >= VP_WALK_MIN || __builtin_amdgcn_ballot_w64(!room) == 0;
#else
    (void)room;
    return step;
#endif
}

struct LeafQueue {
    uint32_t* row;  // &lds[thread][0]
    __device__ __forceinline__ uint32_t& at(uint32_t k) const { return row[k]; }
};

// the calling thread's queue in a dynamic LDS array of leaf_queue_bytes(blockDim.x)
__device__ __forceinline__ LeafQueue leaf_queue(uint32_t* lds) {
    return LeafQueue{lds + (threadIdx.x >> 6) * (kWaveBytes / 4) + (threadIdx.x & 63u) * kLeafRow};
}
inline size_t leaf_queue_bytes(uint32_t block) { return static_cast<size_t>(kWaveBytes) * ((block + 63) / 64); }

// Appends the leaves of mask lm (over first .. first + 3) to a lane's queue at
// cnt, which has room for four.  Slot cnt + (set bits of lm below k) is
// written for every k, set or not, and a later set bit overwrites it, so the
// step has no branches; the writes stay below cnt + 4.
__device__ __forceinline__ void queue_leaves(const LeafQueue& q, uint32_t& cnt, uint32_t lm, uint32_t first) {
    for (uint32_t k = 0; k < 4u; ++k) q.at(cnt + static_cast<uint32_t>(__popc(lm & ((1u << k) - 1u)))) = first + k;
    cnt += static_cast<uint32_t>(__popc(lm));
}

// The ray walk of the counting build, a lane per ray: the boxes of all levels
// are tested and the crossed leaves queued, as in the wave-wide walks
// (walk_nodes).  Their order differs, and with it where the argmin's bound
// stands when a node is met, and the camera ray's direct term is a walk of its
// own here: the timed kernel makes 0.95 of the node visits and 0.94 of the leaf
// tests counted here in the 4096-Gaussian scattering scene, 0.89 and 0.79 on
// the torus, 0.97 and 0.94 in the cloud of 200000, 1.04 and 0.83 in that of
// 10^6.
template <typename Leaf>
__device__ __forceinline__ void walk_ray_q(const SceneView& s, f3 o, f3 inv, const float& tmax, uint32_t& visits,
                                           const LeafQueue& q, Leaf&& leaf) {
    const f3 oi = o * inv;
    Walk4 w = walk4_begin();
    while (true) {
        uint32_t cnt = 0;
        while (true) {
            const bool room = queue_room(cnt);
            const bool step = w.n != kWalkEnd && room;
            if (!node_phase(step, room)) break;
            if (!step) continue;
            ++visits;
            const uint32_t m = ray_mask(s.w4, s.w4_half, w.n, inv, oi, tmax);
            uint32_t first;
            const uint32_t lm = walk4_advance(w, s.w4_levels, m, first);
            if (lm != 0u) queue_leaves(q, cnt, lm, first);
        }
        for (uint32_t k = 0; k < cnt; ++k)
            if (!leaf(q.at(k))) return;
        if (w.n == kWalkEnd) return;
    }
}

template <typename Leaf>
__device__ __forceinline__ void walk_point_q(const SceneView& s, f3 x, uint32_t& visits, const LeafQueue& q,
                                             Leaf&& leaf) {
    Walk4 w = walk4_begin();
    while (true) {
        uint32_t cnt = 0;
        while (w.n != kWalkEnd && queue_room(cnt)) {
            ++visits;
            const uint32_t m = point_mask(s.w4, s.w4_half, w.n, x);
            uint32_t first;
            const uint32_t lm = walk4_advance(w, s.w4_levels, m, first);
            if (lm != 0u) queue_leaves(q, cnt, lm, first);
        }
        for (uint32_t k = 0; k < cnt; ++k) leaf(q.at(k));
        if (w.n == kWalkEnd) return;
    }
}

// Appends the leaves of the calling lanes' crossed leaf blocks (bm: a mask
// over the blocks first .. first + 3 of a walk of leaf blocks,
// walk4_block_levels; block c holds the stored primitives kLeafBlock c ..
// kLeafBlock (c + 1) - 1, records past the scene's last primitive being zero
// records, which the leaf tests reject) to the wave queue at count, in lane
// order, as far as they fit in kWaveQ.  Returns false for a lane whose leaves
// did not fit: its node step is to be repeated after the leaf phase.  The
// lanes that fit form a prefix in lane order, so the queue has no gaps; count
// advances by the leaves written and stays a multiple of 4, so each group of
// four leaves is one 16-byte LDS write of ids and one 4-byte write of owners.
// Every lane of the wavefront that is active here must call it.
__device__ __forceinline__ bool wave_push_blocks(const WaveQueue& wq, uint32_t& count, uint32_t bm, uint32_t first,
                                                 uint32_t owner) {
    static_assert(kWaveQ % 4 == 0, "blocks are queued four leaves at a time");
    const uint32_t nb = static_cast<uint32_t>(__popc(bm));  // 0 .. 4 blocks
    const unsigned long long b0 = __builtin_amdgcn_ballot_w64((nb & 1u) != 0u);
    const unsigned long long b1 = __builtin_amdgcn_ballot_w64((nb & 2u) != 0u);
    const unsigned long long b2 = __builtin_amdgcn_ballot_w64((nb & 4u) != 0u);
    if ((b0 | b1 | b2) == 0ull) return true;  // no blocks this step
    const uint32_t pos = count + kLeafBlock * (lanes_below(b0) + 2u * lanes_below(b1) + 4u * lanes_below(b2));
    const bool fits = nb == 0u || pos + kLeafBlock * nb <= kWaveQ;
    const unsigned long long f = __builtin_amdgcn_ballot_w64(fits);
    if (fits && nb != 0u) {
        uint32_t p = pos;
        for (uint32_t b = bm; b != 0u; b &= b - 1u) {
            const uint32_t l0 = kLeafBlock * (first + static_cast<uint32_t>(__builtin_ctz(b)));
#pragma unroll
            for (uint32_t k = 0; k < kLeafBlock; k += 4u, p += 4u) {
                *reinterpret_cast<uint4*>(wq.prim + p) = make_uint4(l0 + k, l0 + k + 1u, l0 + k + 2u, l0 + k + 3u);
                *reinterpret_cast<uint32_t*>(wq.owner + p) = owner * 0x01010101u;
            }
        }
    }
    count += kLeafBlock * static_cast<uint32_t>(__popcll(b0 & f) + 2 * __popcll(b1 & f) + 4 * __popcll(b2 & f));
    return fits;
}

// Add one chord to the fixed-point optical depth; true once the total
// reaches 88 (exp(-88) underflows), which is order independent because every
// term is non-negative.
__device__ __forceinline__ bool tau_add(uint64_t& acc, float od) {
    const float c = od > 0.0f ? od : 0.0f;
    if (c >= kMaxTau) return true;
    acc += static_cast<uint64_t>(c * kTauScaleF);
    return acc >= kTauLimitFixed;
}

__device__ __forceinline__ float tau_to_T(uint64_t acc) {
    const float tau = static_cast<float>(acc) * kTauInvScale;
    return tau >= kMaxTau ? 0.0f : expf_(-tau);
}
// Transmittance of a fixed-point depth (0 once saturated).
__device__ __forceinline__ float depth_T(uint64_t acc) { return acc >= kTauLimitFixed ? 0.0f : tau_to_T(acc); }

struct EvCount {
    uint32_t v[kNumCounters];
};

template <bool kCount>
struct Ev {
    EvCount c;
    __device__ __forceinline__ void reset() {
        if constexpr (kCount)
            for (int i = 0; i < kNumCounters; ++i) c.v[i] = 0;
    }
    __device__ __forceinline__ void add(int slot, uint32_t n = 1) {
        if constexpr (kCount) c.v[slot] += n;
    }
    __device__ __forceinline__ void flush(unsigned long long* g) {
        if constexpr (kCount) {
            for (int i = kCntPaths; i < kNumCounters; ++i)
                if (c.v[i]) atomicAdd(&g[i], static_cast<unsigned long long>(c.v[i]));
            reset();
        }
    }
};

// compute_transmittance_to_env (sampling.cuh:548-583) with the fused
// any-hit integration (anyhit.cuh:53-66), as a fixed-point optical depth: the
// walk stops once the sum reaches limit (at most the tau = 88 saturation,
// which it returns as kTauLimitFixed).
template <bool kCount>
__device__ uint64_t shadow_depth(const SceneView& s, f3 o, f3 d, const uint32_t* act, uint32_t na, uint32_t stride,
                                 const LeafQueue& lq, Ev<kCount>& ev, uint64_t limit) {
    uint64_t acc = 0;
    if (acc >= limit) return acc;
    for (uint32_t k = 0; k < na; ++k) {
        const PrimRecord pr = load_prim(s.prims, act[k * stride]);
        const InsideChord x = inside_chord(pr, o, d);
        ev.add(kCntShActive);
        if (x.tau > 0.0f) {
            if (tau_add(acc, x.tau)) return kTauLimitFixed;
            if (acc >= limit) return acc;
        }
    }
    const f3 inv = safe_inv(d);
    const float tmax = kTMax;
    uint32_t visits = 0, leaves = 0, sh = 0;
    walk_ray_q(s, o, inv, tmax, visits, lq, [&](uint32_t prim) -> bool {
        const PrimRecord pr = load_prim(s.prims, prim);
        ++leaves;
        const Crossing x = crossing(pr, o, d);
        if (x.t0 < 0.0f) return true;
        ++sh;
        if (tau_add(acc, x.tau)) {
            acc = kTauLimitFixed;
            return false;
        }
        return acc < limit;
    });
    ev.add(kCntNodeVisits, visits);
    ev.add(kCntVisitsShadow, visits);
    ev.add(kCntLeafTests, leaves);
    ev.add(kCntShHit, sh);
    return acc;
}

// one chord in fixed point, as tau_add adds it; a chord of tau >= 88 alone
// adds the saturation limit
__device__ __forceinline__ unsigned long long tau_fixed(float od) {
    const float c = od > 0.0f ? od : 0.0f;
    return c >= kMaxTau ? kTauLimitFixed : static_cast<unsigned long long>(c * kTauScaleF);
}

// ---- wave-wide walks of the megakernel ----
//
// The rays of a wavefront are walked together by its 64 lanes from one stack
// of (node, ray) items in LDS: every lane takes an item from the top, tests
// its node's four children against its ray, and appends the crossed ones; the
// crossed children of a last-level node are leaves and go to a leaf queue,
// from which 64 at a time are evaluated.  Which lane tests which node is of no
// account: all results are fixed-point sums and minima.  Node steps and leaf
// tests then run at full width however few rays are left and however uneven
// their walks are, and no lane holds a walk in registers.  (With a walk per
// lane, the argmin's node steps ran at 19 to 28 % of the lanes, and a walk's
// nodes were a serial chain.)
// The walks are bound by VALU issue and the L1's data return, which takes a
// cycle per lane of each load whatever its size: with six 8-byte loads a node
// it was busy 91 % of the scattering workload's time (VALU 85 %); whole 16-byte
// words, one scene's pointers in scalar registers and the ray's end in one
// word took 10 % off it, 14 % off the torus and 23 % off the 10^6 cloud.
// Measured and not taken: four lanes to a node (16 nodes a step, a record read
// as 64 contiguous bytes: 38 ms against 27), a leaf's record read by four lanes
// and transposed by lane swaps (+3 to +7 %: 60 more VALU a round), two leaves
// per lane and round (0).
// Node k of the implicit 4-ary tree has the children 4k + 1 .. 4k + 4 in heap
// order; a node is on the last level from index w4_level_base(levels - 1) on.
constexpr uint32_t kNodeQ = 648;      // stack items
constexpr uint32_t kLeafItems = 240;  // leaf queue items
// Items of the stack held back from wide steps: one item at a time adds at
// most 3 per level, so a walk always finishes.
constexpr uint32_t kNodeReserve = 3 * kW4MaxLevels + 3;
static_assert(kNodeQ > kNodeReserve + 3 * 64 + 64 && kLeafItems >= 64 + 4, "room for a step of every lane");

// The rays are numbered 2 l and 2 l + 1 for lane l: its two shadow rays, or
// for the argmin ray 2 l alone, with the argmin's state in the other's place.
struct MegaQueue {
    uint32_t* node;          // [kNodeQ] stack: nodes still to be tested
    uint32_t* leaf;          // [kLeafItems] stored primitives still to be tested
    uint8_t* node_ray;       // [kNodeQ] their rays
    uint8_t* leaf_ray;       // [kLeafItems]
    float* ro;               // [64 * 3] ray origin of each lane
    float* rd;               // [128 * 3] ray directions
    float* inv;              // [128 * 3] their reciprocals (safe_inv)
    unsigned long long* acc;   // [128] fixed-point optical depth of each ray
    float* tmax;             // [128] the rays' ends; negative once a ray is done
    uint32_t* job;           // [64] job-table entry of each lane's path
    uint8_t* list;           // [128] the rays still to be walked
    uint32_t* scratch;       // [kScratch] words over node and leaf, free outside the walks
    uint32_t* help;          // [4] see help_walks

    // argmin state of lane l
    __device__ __forceinline__ uint32_t& ts(uint32_t l) const {  // running minimum, float bits
        return reinterpret_cast<uint32_t*>(acc + 2 * l + 1)[0];
    }
    __device__ __forceinline__ uint32_t& bound(uint32_t l) const {  // an upper bound of the final minimum, float bits
        return reinterpret_cast<uint32_t*>(tmax)[2 * l + 1];
    }
    __device__ __forceinline__ uint32_t& nc(uint32_t l) const {  // candidates recorded
        return reinterpret_cast<uint32_t*>(acc + 2 * l + 1)[1];
    }
    __device__ __forceinline__ uint32_t& hits(uint32_t l) const {  // entries counted (measuring build)
        return reinterpret_cast<uint32_t*>(inv + 3 * (2 * l + 1))[0];
    }
    __device__ __forceinline__ uint32_t* draw(uint32_t l) const {  // [3] path key (2 words), bounce | direct << 31
        return reinterpret_cast<uint32_t*>(rd + 3 * (2 * l + 1));
    }
};
constexpr uint32_t kScratch = kNodeQ + kLeafItems;
constexpr uint32_t kMegaQueueBytes = 5 * (kNodeQ + kLeafItems) + 64 * 12 + 128 * 24 + 128 * 8 + 128 * 4 + 64 * 4 + 128 + 16;
static_assert((5 * (kNodeQ + kLeafItems)) % 8 == 0, "the 8-byte arrays stay aligned");
constexpr uint32_t kMegaBytes =
    ((64 * kLeafRow * 4 > kMegaQueueBytes ? 64 * kLeafRow * 4 : kMegaQueueBytes) + 15) / 16 * 16;
static_assert(64 * kLeafRow * 4 <= kMegaQueueBytes - 16, "the point-query queue leaves the help words alone");
static_assert(16 * kMegaBytes <= 160 * 1024, "16 wavefronts to a CU");
inline size_t mega_queue_bytes(uint32_t block) { return static_cast<size_t>(kMegaBytes) * ((block + 63) / 64); }

// the queue of wavefront `wave` of the workgroup
__device__ __forceinline__ MegaQueue mega_queue_of(uint32_t* lds, uint32_t wave) {
    uint8_t* base = reinterpret_cast<uint8_t*>(lds) + wave * kMegaBytes;
    MegaQueue q;
    q.scratch = q.node = reinterpret_cast<uint32_t*>(base);
    q.leaf = q.node + kNodeQ;
    q.node_ray = reinterpret_cast<uint8_t*>(q.leaf + kLeafItems);
    q.leaf_ray = q.node_ray + kNodeQ;
    q.ro = reinterpret_cast<float*>(q.leaf_ray + kLeafItems);
    q.rd = q.ro + 64 * 3;
    q.inv = q.rd + 128 * 3;
    q.acc = reinterpret_cast<unsigned long long*>(q.inv + 128 * 3);
    q.tmax = reinterpret_cast<float*>(q.acc + 128);
    q.job = reinterpret_cast<uint32_t*>(q.tmax + 128);
    q.list = reinterpret_cast<uint8_t*>(q.job + 64);
    q.help = reinterpret_cast<uint32_t*>(q.list + 128);
    return q;
}
// the calling wavefront's queue
__device__ __forceinline__ MegaQueue mega_queue(uint32_t* lds) { return mega_queue_of(lds, threadIdx.x >> 6); }
// the calling thread's point-query queue over the same LDS
__device__ __forceinline__ LeafQueue mega_leaf_queue(uint32_t* lds) {
    return LeafQueue{lds + (threadIdx.x >> 6) * (kMegaBytes / 4) + (threadIdx.x & 63u) * kLeafRow};
}

// The scene of a wavefront's paths.  Lanes may run jobs over different scenes
// (batches, the server); when all paths of the wavefront share one (one, as
// nearly always) its pointers are held in scalar registers and records are
// read through 32-bit offsets from them, else each item's scene is looked up
// through its lane's job.  A scene too large for the offsets takes the second
// way as well.
struct WaveScene {
    bool one;
    const PrimRecord* prims;
    const float4* w4;
    uint32_t half, leaf_base;
    const JobDesc* jobs;
};
template <typename T>
__device__ __forceinline__ const T* read_lane_ptr(const T* p, uint32_t l) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(l)));
    const uint32_t hi =
        static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v >> 32), static_cast<int>(l)));
    return reinterpret_cast<const T*>((static_cast<uint64_t>(hi) << 32) | lo);
}
// on: the lanes with a path (at least one)
__device__ __forceinline__ WaveScene wave_scene(const SceneView& sc, bool on, const JobDesc* jobs) {
    const uint32_t lead = static_cast<uint32_t>(__builtin_ctzll(__builtin_amdgcn_ballot_w64(on)));
    WaveScene ws;
    ws.prims = read_lane_ptr(sc.prims, lead);
    ws.w4 = read_lane_ptr(sc.w4, lead);
    const uint32_t tree = static_cast<uint32_t>(
        __builtin_amdgcn_readlane(static_cast<int>(sc.w4_levels | (sc.w4_half << 8)), static_cast<int>(lead)));
    const uint32_t levels = tree & 0xffu;
    ws.half = tree >> 8;
    ws.leaf_base = w4_level_base(levels - 1u);
    ws.jobs = jobs;
    // records of 64 bytes (primitives) and at most 128 (nodes) within 2^32
    ws.one = levels <= 13u && __builtin_amdgcn_ballot_w64(on && (sc.prims != ws.prims || sc.w4 != ws.w4)) == 0ull;
    return ws;
}
// Record `prim` of the scene of lane own's path: what crossing() needs, or all
// of it.
__device__ __forceinline__ PrimRecord load_wave_leaf(const MegaQueue& q, const WaveScene& ws, uint32_t own,
                                                     uint32_t prim) {
    if (ws.one) return load_leaf(ws.prims, prim);
    return load_leaf(ws.jobs[q.job[own]].scene.prims, static_cast<size_t>(prim));
}
__device__ __forceinline__ PrimRecord load_wave_prim(const MegaQueue& q, const WaveScene& ws, uint32_t own,
                                                     uint32_t prim) {
    if (ws.one) {
        const auto* p = reinterpret_cast<const VP_GLOBAL_AS char*>(as_global(ws.prims)) +
                        prim * static_cast<uint32_t>(sizeof(PrimRecord));
        return load_prim((const PrimRecord*)p, 0u);
    }
    return load_prim(ws.jobs[q.job[own]].scene.prims, prim);
}

// Exclusive prefix sum over the wavefront of v <= 7 (every lane active).
__device__ __forceinline__ uint32_t wave_prefix3(uint32_t v, uint32_t& total) {
    const unsigned long long b0 = __builtin_amdgcn_ballot_w64((v & 1u) != 0u);
    const unsigned long long b1 = __builtin_amdgcn_ballot_w64((v & 2u) != 0u);
    const unsigned long long b2 = __builtin_amdgcn_ballot_w64((v & 4u) != 0u);
    total = static_cast<uint32_t>(__popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2));
    return lanes_below(b0) + 2u * lanes_below(b1) + 4u * lanes_below(b2);
}

// One node step of the wavefront: the top items of the stack (nn of them in
// all, at least one), as many as the lanes and the room left allow, are
// replaced by their crossed children, and crossed leaves are appended to the
// leaf queue (nl items, leaf_cap at most).  A ray is tested over [0, its
// tmax], and not at all once that is negative.
// The order of the children on the stack: for the argmin, nearest first and
// lane by lane, so a few rays at a time reach their nearest leaves and the
// bounds they prune by; for shadow rays, first children of all lanes first, so
// the step's rays descend together and one that reaches its limit leaves few
// items behind.  (Lane by lane in index order for both, an argmin flight kept
// waiting: 10^6 cloud 310 ms, torus 49, scattering 26.9; nearest first: 281,
// 42.6, 27.0; first children first for the shadow rays as well: 266, 41.7,
// 26.7; for both: 258, 46, 25.0.)
// The crossing tests of all lanes are one scalar mask per child (every lane
// tests, so no branch turns them into vectors), and a child's mask gives its
// lanes' places by a bit count: against a 4-bit mask per lane with its own
// prefix sums and bit scans, 190 -> 130 VALU a step, scattering 23.7 -> 22.9 ms,
// 10^6 cloud 169.5 -> 163.5, adaptive 18.0 -> 17.4.
template <bool kNearFirst>
__device__ __forceinline__ void walk_nodes(const MegaQueue& q, const WaveScene& ws, uint32_t& nn, uint32_t& nl,
                                           uint32_t leaf_cap) {
    const uint32_t lane = __lane_id();
    const uint32_t room = nn + kNodeReserve + 3u < kNodeQ ? (kNodeQ - kNodeReserve - nn) / 3u : 1u;
    uint32_t n = nn < 64u ? nn : 64u;
    n = n < room ? n : room;
    nn -= n;
    // every lane tests, so the tests' lane masks are scalars: one without an
    // item, or whose ray is done, takes an item's box over an empty interval
    const uint32_t item = nn + (lane < n ? lane : 0u);
    const uint32_t node = q.node[item], ray = q.node_ray[item];
    const float end = q.tmax[ray], tmax = lane < n ? end : -1.0f;
    const f3 inv = lds_load3(q.inv + 3 * ray), oi = lds_load3(q.ro + 3 * (ray >> 1)) * inv;
    uint32_t base = ws.leaf_base;
    float tn[4];
    unsigned long long h[4];  // the lanes that cross child c
    if (ws.one) {
        mega_ray_hits(ws.w4, ws.half, node, inv, oi, tmax, tn, [&](int c, bool v) { h[c] = __builtin_amdgcn_ballot_w64(v); });
    } else {
        const SceneView& sc = ws.jobs[q.job[ray >> 1]].scene;
        uint32_t m = 0;
        mega_ray_hits(sc.w4, sc.w4_half, static_cast<size_t>(node), inv, oi, tmax, tn,
                      [&](int c, bool v) { m |= v ? 1u << c : 0u; });
        for (int c = 0; c < 4; ++c) h[c] = __builtin_amdgcn_ballot_w64(((m >> c) & 1u) != 0u);
        base = w4_level_base(sc.w4_levels - 1u);
    }
    const bool last = node >= base;
    const unsigned long long last_mask = __builtin_amdgcn_ballot_w64(last);
    uint32_t child = last ? 4u * (node - base) : 4u * node + 1u;
    wave_sync();
    // leaves, child by child
    unsigned long long back = 0ull;  // last-level nodes whose leaves do not fit go back
    const uint32_t total = static_cast<uint32_t>(__popcll(h[0] & last_mask) + __popcll(h[1] & last_mask) +
                                                 __popcll(h[2] & last_mask) + __popcll(h[3] & last_mask));
    if (total != 0u) {
        if (nl + total > leaf_cap) {
            // the lanes whose leaves fit come first
            uint32_t c = 0, all;
            for (int k = 0; k < 4; ++k) c += __builtin_amdgcn_inverse_ballot_w64(h[k] & last_mask) ? 1u : 0u;
            const bool over = c != 0u && nl + wave_prefix3(c, all) + c > leaf_cap;
            back = __builtin_amdgcn_ballot_w64(over);
            if (over) child = node;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const unsigned long long m = h[c] & last_mask & ~back;
            if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                const uint32_t at = nl + lanes_below(m);
                q.leaf[at] = child + c;
                q.leaf_ray[at] = static_cast<uint8_t>(ray);
            }
            nl += static_cast<uint32_t>(__popcll(m));
        }
    }
    if constexpr (kNearFirst) {
        uint32_t push = __builtin_amdgcn_inverse_ballot_w64((h[0] & ~last_mask) | back) ? 1u : 0u;
        for (int c = 1; c < 4; ++c) push |= __builtin_amdgcn_inverse_ballot_w64(h[c] & ~last_mask) ? 1u << c : 0u;
        if (__builtin_amdgcn_ballot_w64(push != 0u) != 0ull) {
            // the nearest child on top, its sibling below it, then the others
            // (children c ^ s, c descending)
            const float a = fminf(tn[0], tn[1]), b = fminf(tn[2], tn[3]);
            uint32_t s = b < a ? (tn[3] < tn[2] ? 3u : 2u) : (tn[1] < tn[0] ? 1u : 0u);
            if (last) s = 0u;
            push = (s & 1u) != 0u ? ((push & 5u) << 1) | ((push >> 1) & 5u) : push;
            push = (s & 2u) != 0u ? ((push & 3u) << 2) | (push >> 2) : push;
            const uint32_t c = static_cast<uint32_t>(__popc(push));
            uint32_t all;
            uint32_t at = nn + wave_prefix3(c, all) + c;
            for (uint32_t b = push; b != 0u; b &= b - 1u) {
                --at;
                q.node[at] = child + (static_cast<uint32_t>(__builtin_ctz(b)) ^ s);
                q.node_ray[at] = static_cast<uint8_t>(ray);
            }
            nn += all;
        }
    } else {
        // every lane's first child on top, below them the second ones, and so
        // on: the next step goes on with all the rays of this one
#pragma unroll
        for (int c = 3; c >= 0; --c) {
            const unsigned long long m = (h[c] & ~last_mask) | (c == 0 ? back : 0ull);
            if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                const uint32_t at = nn + lanes_below(m);
                q.node[at] = child + c;
                q.node_ray[at] = static_cast<uint8_t>(ray);
            }
            nn += static_cast<uint32_t>(__popcll(m));
        }
    }
    wave_sync();
}

// Pushes the rays list[0 .. k) (k <= 64) onto the stack.  Up to four rays start
// at the third level of a tree of 3 to 7 levels (17 to 16384 primitives)
// instead of its root, a lane per node: the top of the tree is a chain of
// steps with little in them, two of the six or seven that such a walk takes
// (64x64x2 scattering 1.92 -> 1.77 ms, 157x83x3 of 97 Gaussians 0.58 -> 0.54).
// In deeper trees the top is less of the chain, and in larger images a walk that
// prunes or saturates loses by opening all of it at once (512x512 torus +2 %,
// 192x128x2 cloud of 200000 and 10^6 cloud +4 %).  With against without, at 64x64x2:
// scattering of 100, 1000, 4096 (4 to 6 levels) 0.88, 0.87, 0.89, of 8000 and
// 16384 (7) 0.91 and 0.92, and it would be 0.94, 0.97 and 0.96 for 30000, 65536 (8)
// and 150000 (9); at 96x96x1 torus and cloud of 10000 (7) 0.89 and 0.91, and 0.93
// to 0.95 for 40000 and 100000 (8 and 9).
__device__ __forceinline__ void push_rays(const MegaQueue& q, const WaveScene& ws, const uint8_t* list, uint32_t k,
                                          uint32_t& nn) {
    const uint32_t lane = __lane_id();
    const bool third = ws.one && ws.leaf_base >= w4_level_base(2u) && ws.leaf_base <= w4_level_base(6u) && k <= 4u;
    const uint32_t s = third ? 4u : 0u;  // log2 of the items per ray
    if (lane < k << s) {
        q.node[nn + lane] = third ? w4_level_base(2u) + (lane & 15u) : 0u;
        q.node_ray[nn + lane] = list[lane >> s];
    }
    nn += k << s;
    wave_sync();
}

// Help between the wavefronts of a workgroup.  A wavefront that has finished
// its own paths waits for stack items of another's walk: one with enough of
// them hands over the bottom half of its stack (the largest subtrees), and the
// helper walks them with its own stack and leaf queue over the giver's rays,
// into their sums and minima.  The giver waits for its helpers at the end of
// its walk, so its rays stay in place, and a helper leaves once no wavefront of
// the workgroup has paths, so every wait ends.  Sums are fixed point and minima
// exact: who adds what changes no result.
// The end of a launch is a few long paths (at most max_depth bounces, each with
// up to thousands of items in a dense cloud) on a nearly idle device: in the
// 192x128x2 cloud the longest wavefront ran 4.4 times the mean.  No help, help
// with the shadow walks among 4 wavefronts, among 16, with the argmin walks as
// well, first paths spread over the workgroups: that cloud 16.7, 13.5, 12.0,
// 12.0, 10.3 ms; torus 18.6, 18.6, 18.5, 16.9, 16.9; adaptive scattering 19.8,
// 18.6, 18.0, 18.2, 18.0.
// help[0]: kHelpWait of a wavefront that waits, kHelpNone, or what it was given
// (kHelpWork | one scene << 2 | argmin << 3 | wavefront whose rays they are << 8 |
// items << 16);
// help[1]: the helpers at work on a wavefront's rays; help[2] of wavefront 0:
// the wavefronts with paths.
constexpr uint32_t kHelpNone = 0u, kHelpWait = 1u, kHelpWork = 2u;
// Items that a wavefront gives away half of, and how often it looks (in rounds,
// a power of two): 48 items and every round are the same but for the 64x64
// preview (-1 %) and the wider scenes (+0.5 %).
constexpr uint32_t kHelpMin = 96, kHelpEvery = 2;
__device__ __forceinline__ uint32_t help_load(uint32_t* p) {
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
}
// Before the workgroup's barrier.
__device__ __forceinline__ void help_begin(uint32_t* lds) {
    const MegaQueue q = mega_queue(lds);
    if ((threadIdx.x & 63u) == 0u) {
        q.help[0] = kHelpNone;
        q.help[1] = 0u;
        q.help[2] = blockDim.x >> 6;
    }
}
// Gives items of the stack q (nn) to waiting wavefronts; the rays are those of
// wavefront rays_of.
__device__ __forceinline__ void give_items(uint32_t* lds, const MegaQueue& q, uint32_t rays_of, bool one, bool argmin,
                                           uint32_t& nn) {
    const uint32_t lane = __lane_id(), waves = blockDim.x >> 6;
    const uint32_t see = lane < waves ? __hip_atomic_load(mega_queue_of(lds, lane).help, __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_WORKGROUP)
                                      : kHelpNone;
    unsigned long long idle = __builtin_amdgcn_ballot_w64(see == kHelpWait);
    while (idle != 0ull && nn >= kHelpMin) {
        const MegaQueue h = mega_queue_of(lds, static_cast<uint32_t>(__builtin_ctzll(idle)));
        idle &= idle - 1ull;
        uint32_t won = 0;
        if (lane == 0u) {
            uint32_t expect = kHelpWait;
            won = __hip_atomic_compare_exchange_strong(h.help, &expect, kHelpNone, __ATOMIC_ACQUIRE, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_WORKGROUP)
                      ? 1u
                      : 0u;
            if (won != 0u)
                (void)__hip_atomic_fetch_add(mega_queue_of(lds, rays_of).help + 1, 1u, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        if (__builtin_amdgcn_readfirstlane(won) == 0u) continue;
        const uint32_t k = nn / 2u < 64u ? nn / 2u : 64u;
        uint32_t top = 0, top_ray = 0;
        if (lane < k) {
            h.node[lane] = q.node[lane];
            h.node_ray[lane] = q.node_ray[lane];
            top = q.node[nn - k + lane];
            top_ray = q.node_ray[nn - k + lane];
        }
        wave_sync();
        if (lane < k) {
            q.node[lane] = top;
            q.node_ray[lane] = static_cast<uint8_t>(top_ray);
        }
        nn -= k;
        wave_sync();
        if (lane == 0u)
            __hip_atomic_store(h.help, kHelpWork | (one ? 4u : 0u) | (argmin ? 8u : 0u) | rays_of << 8 | k << 16, __ATOMIC_RELEASE,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

// The rays of rq with the stack and the leaf queue of q.
__device__ __forceinline__ MegaQueue rays_with_stack(const MegaQueue& rq, const MegaQueue& q) {
    MegaQueue w = rq;
    w.node = q.node;
    w.leaf = q.leaf;
    w.node_ray = q.node_ray;
    w.leaf_ray = q.leaf_ray;
    return w;
}

// The rounds of shadow walks, over the stack and leaf queue of q and the rays
// of rq (those of wavefront rays_of).  The rays' own wavefront (kOwn) pushes
// its nr listed rays and ends the ones that have reached their limits.
template <bool kOwn>
__device__ __forceinline__ void shadow_rounds(const WaveScene& ws, uint32_t* lds, const MegaQueue& q,
                                              const MegaQueue& rq, uint32_t rays_of, uint32_t nr, uint64_t lim_a,
                                              uint64_t lim_b, uint32_t nn, uint32_t& rounds) {
    const uint32_t lane = __lane_id();
    const MegaQueue w = rays_with_stack(rq, q);
    uint32_t next = 0, nl = 0;
    auto end_rays = [&]() {
        if (w.acc[2 * lane] >= lim_a) w.tmax[2 * lane] = -1.0f;
        if (w.acc[2 * lane + 1] >= lim_b) w.tmax[2 * lane + 1] = -1.0f;
    };
    while (true) {
        if (kOwn && nn < 64u && next < nr) {
            // the next rays, up to an item per lane
            const uint32_t k = nr - next < 64u - nn ? nr - next : 64u - nn;
            push_rays(w, ws, w.list + next, k, nn);
            next += k;
        }
        if (nl < 64u && nn != 0u) {
            if (nn >= kHelpMin && (rounds & (kHelpEvery - 1u)) == 0u) give_items(lds, w, rays_of, ws.one, false, nn);
            walk_nodes<false>(w, ws, nn, nl, kLeafItems);
            ++rounds;
            continue;
        }
        if (nl == 0u) break;
        // 64 leaves (or the last ones): each one's crossing (entry test and
        // whole-chord depth from one transform) goes into its ray's sum
        const uint32_t n = nl < 64u ? nl : 64u;
        nl -= n;
        ++rounds;
        if (lane < n) {
            const uint32_t ray = w.leaf_ray[nl + lane], own = ray >> 1, prim = w.leaf[nl + lane];
            const f3 ro = lds_load3(w.ro + 3 * own), rd = lds_load3(w.rd + 3 * ray);
            if (w.tmax[ray] >= 0.0f) {
                const Crossing x = crossing(load_wave_leaf(w, ws, own, prim), ro, rd);
                if (x.tau > 0.0f) atomicAdd(&w.acc[ray], tau_fixed(x.tau));
            }
        }
        wave_sync();
        if (kOwn) end_rays();
        wave_sync();
    }
    if (kOwn)
        while (help_load(w.help + 1) != 0u) {
            end_rays();
            __builtin_amdgcn_s_sleep(4);
        }
}

// The shadow rays of a wavefront's lanes, up to two each (the MIS rays a and
// b, or the one of RIS).  All 64 lanes of the wavefront call it.  q.ro, q.job,
// q.rd and q.acc hold the rays' origins, jobs, directions and the depths of
// their origin sets.  Each ray's chords are summed in fixed point in LDS (a
// ray is saturated once its sum reaches the tau = 88 limit, in whatever order
// the chords arrive), so the depths equal those of shadow_depth() bit for
// bit.
// Each ray's walk may stop once its depth reaches its limit (lim_a, lim_b:
// the tau = 88 saturation, or a shadow-roulette threshold); a limit of 0 is a
// ray that is not walked.  acc_a and acc_b receive the fixed-point depths;
// rounds counts the node steps and leaf rounds.
__device__ __forceinline__ void shadow_walks(const WaveScene& ws, uint32_t* lds, const MegaQueue& q, uint64_t lim_a,
                                             uint64_t lim_b, uint64_t& acc_a, uint64_t& acc_b, uint32_t& rounds) {
    const uint32_t lane = __lane_id();
    lds_store3(q.inv + 3 * (2 * lane), safe_inv(lds_load3(q.rd + 3 * (2 * lane))));
    lds_store3(q.inv + 3 * (2 * lane + 1), safe_inv(lds_load3(q.rd + 3 * (2 * lane + 1))));
    // the rays to walk: every ray a, then every ray b, that is not done already
    const bool walk_a = q.acc[2 * lane] < lim_a, walk_b = q.acc[2 * lane + 1] < lim_b;
    q.tmax[2 * lane] = walk_a ? kTMax : -1.0f;
    q.tmax[2 * lane + 1] = walk_b ? kTMax : -1.0f;
    const unsigned long long pa = __builtin_amdgcn_ballot_w64(walk_a);
    const unsigned long long pb = __builtin_amdgcn_ballot_w64(walk_b);
    const uint32_t npa = static_cast<uint32_t>(__popcll(pa));
    const uint32_t nr = npa + static_cast<uint32_t>(__popcll(pb));
    if (walk_a) q.list[lanes_below(pa)] = static_cast<uint8_t>(2 * lane);
    if (walk_b) q.list[npa + lanes_below(pb)] = static_cast<uint8_t>(2 * lane + 1);
    wave_sync();
    shadow_rounds<true>(ws, lds, q, q, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nr, lim_a, lim_b, 0u, rounds);
    acc_a = q.acc[2 * lane];
    acc_b = q.acc[2 * lane + 1];
    wave_sync();
}

__device__ __forceinline__ EnvView env_view(const EnvDev& e) {
    EnvView v;
    v.tex = e.tex;
    v.alias = e.has_table ? e.alias : nullptr;
    v.joint = e.joint;
    v.w = e.w;
    v.h = e.h;
    v.total = e.total;
    return v;
}

__device__ __forceinline__ uint32_t find_job(const uint64_t* begin, uint32_t njobs, uint64_t p) {
    uint32_t lo = 0, hi = njobs;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (begin[mid] <= p) lo = mid;
        else hi = mid;
    }
    return lo;
}


// finalize_sample (path_stages.cuh:52-62): optional luminance clamp,
// non-finite radiance to zero.
__device__ __forceinline__ float4 finalize_radiance(const JobDesc& J, f3 L) {
    if (J.firefly_clamp > 0.0f) {
        const float lum = dot(L, f3{kLumR, kLumG, kLumB});
        if (lum > J.firefly_clamp) L = L * (J.firefly_clamp * rcpf(lum));
    }
    if (!isfinitef_(sum3(L))) L = mk(0.0f);
    return make_float4(L.x, L.y, L.z, 1.0f);
}

// Path setup (raygen.cuh:72-113) for path q of job J's current slice: pixel
// and sample from the 8x8-tile numbering, RNG stream, counter-hash key and
// jittered camera ray; pix receives the pixel index (y * width + x) and sl the
// sample's index within the slice.  False for the padding paths of partial
// tiles and for the paths of pixels that adaptive sampling has stopped.
__device__ __forceinline__ bool path_begin(const JobDesc& J, uint64_t q, f3& o, f3& d, Pcg32& rng, uint64_t& key,
                                           uint32_t& pix_out, uint32_t& sl_out) {
    // the slice's samples of one pixel are consecutive paths, so a
    // wavefront's lanes start on few pixels (nearly the same camera rays)
    const uint32_t r = static_cast<uint32_t>(q / J.s_count);
    const uint32_t sl = static_cast<uint32_t>(q - static_cast<uint64_t>(r) * J.s_count);
    // 8x8 tiles, in bands of kTileBand tile rows, column by column within a
    // band, so the paths in flight on one XCD (a run of consecutive path
    // indices) cover a compact patch of the image
    constexpr uint32_t kTileBand = 16;
    const uint32_t tile = r >> 6, w = r & 63u;
    const uint32_t tiles_y = (J.height + 7u) / 8u;
    const uint32_t band = tile / (kTileBand * J.tiles_x), c = tile - band * (kTileBand * J.tiles_x);
    const uint32_t rows = tiles_y - band * kTileBand < kTileBand ? tiles_y - band * kTileBand : kTileBand;
    const uint32_t px = (c / rows) * 8u + (w & 7u);
    const uint32_t py = (band * kTileBand + c % rows) * 8u + (w >> 3);
    if (px >= J.width || py >= J.height) return false;
    const uint32_t sample = J.s_begin + sl;
    const uint64_t pix = static_cast<uint64_t>(py) * J.width + px;
    // adaptive sampling: a converged pixel traces nothing more
    // (raygen.cuh:53-69); its paths end like padding
    if (J.adapt_state != nullptr && (J.adapt_state[pix] >> 31) != 0u) return false;
    const uint64_t seq = hash64(pix * J.spp + sample);
    rng = pcg_init(J.seed, seq);
    key = path_key(J.seed, seq);
    float jx, jy;
    if (J.filter_stddev > 0.0f) {
        gaussian_jitter(rng, J.filter_stddev, &jx, &jy);
    } else {
        jx = next_uniform(rng) - 0.5f;
        jy = next_uniform(rng) - 0.5f;
    }
    camera_ray(J.cam, px, py, jx, jy, &o, &d);
    pix_out = static_cast<uint32_t>(pix);
    sl_out = sl;
    return true;
}

// A finished path (raygen.cuh:214-238): its radiance is added to its pixel's
// exact fixed-point sums (fire-and-forget atomics: integer adds commute, so
// the total does not depend on which path finishes first), written to its
// per-sample slot if the caller asked for per-sample output, and counted
// against its job-table entry if the entry is tracked (the server).  The
// count follows the completion of the sums' atomics, so a host that sees the
// entry complete and then copies the sums reads finished ones.
__device__ __forceinline__ void path_finish(const JobDesc& J, uint32_t pix, uint32_t sl, f3 L) {
    const float4 v = finalize_radiance(J, L);
    unsigned long long* a = J.accum + static_cast<size_t>(pix) * kAccumWords;
    const float c[3] = {v.x, v.y, v.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const uint64_t q = radiance_fixed(c[k]);
        __hip_atomic_fetch_add(a + k, static_cast<unsigned long long>(q & 0xffffffffull), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        if ((q >> 32) != 0ull)
            __hip_atomic_fetch_add(a + 4 + k, static_cast<unsigned long long>(q >> 32), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    }
    __hip_atomic_fetch_add(a + 3, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (J.samples != nullptr) J.samples[static_cast<size_t>(sl) * (static_cast<size_t>(J.width) * J.height) + pix] = v;
    if (J.done != nullptr) {
        // The sums are agent-scope atomics, which the device performs where
        // every compute unit sees them; the count only has to follow their
        // completion, so the wave waits for all its outstanding memory
        // operations (s_waitcnt with every counter at 0) before adding it.
        // An agent-scope release fence would also write back the XCD's
        // whole L2 for every finished path.  Entries with per-sample output
        // are not counted (the server asks for none).
        __builtin_amdgcn_s_waitcnt(0);
        __hip_atomic_fetch_add(J.done, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}


}  // namespace
}  // namespace vp
