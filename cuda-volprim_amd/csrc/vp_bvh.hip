// vp_bvh.hip — GPU construction of the scene: primitive records, Morton
// codes, a stable LDS radix sort, the depth of the Karras (2012) binary radix
// tree over them, and the walk tree over the stored order (vp_walk.h).  The
// radix tree orders the leaves as the sort does, and no walk uses its inner
// nodes, so their boxes are not built.
//
// Replaces the reference's Morton sort (src/thesis/host/app/renderer.cpp:90-121,
// include/thesis/host/utils/math.h:103-160) and its OptiX GAS/IAS build
// (renderer.cpp:123-173, include/thesis/host/optix/gas.h:47-79).  Morton codes
// are bit-exact with the reference's morton3D on primitive centres; ties are
// broken by input index (a stable sort), which the reference leaves to
// std::sort.
#include "vp_internal.h"

namespace vp {
namespace {

constexpr uint32_t kSortBlock = 256;
constexpr uint32_t kSortItems = 8;
constexpr uint32_t kSortTile = kSortBlock * kSortItems;

__device__ __forceinline__ uint32_t expand_bits(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

// Records, centres and conservative leaf boxes (conservative_box).
__global__ void k_setup(const vp_primitive* in, uint32_t n, PrimRecord* rec, float* centers, float* box) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const vp_primitive p = in[i];
    const f3 c = f3{p.center[0], p.center[1], p.center[2]};
    const f3 s = f3{p.scale[0], p.scale[1], p.scale[2]};
    const PrimRecord r = make_prim(c, p.quat_wxyz[0], p.quat_wxyz[1], p.quat_wxyz[2], p.quat_wxyz[3], s,
                                   f3{p.albedo[0], p.albedo[1], p.albedo[2]}, p.mass);
    rec[i] = r;
    centers[3 * i + 0] = c.x;
    centers[3 * i + 1] = c.y;
    centers[3 * i + 2] = c.z;
    conservative_box(r, p.scale, box + 6 * i, box + 6 * i + 3);
}

// Centre bounds: per-block partial min/max, then one block folds them.
__global__ void k_bounds_partial(const float* centers, uint32_t n, float* partial) {
    __shared__ float smin[3][256], smax[3][256];
    const uint32_t t = threadIdx.x;
    float mn[3] = {3.402823466e38f, 3.402823466e38f, 3.402823466e38f};
    float mx[3] = {-3.402823466e38f, -3.402823466e38f, -3.402823466e38f};
    for (uint32_t i = blockIdx.x * blockDim.x + t; i < n; i += gridDim.x * blockDim.x)
        for (int k = 0; k < 3; ++k) {
            const float c = centers[3 * i + k];
            mn[k] = minf(mn[k], c);
            mx[k] = maxf(mx[k], c);
        }
    for (int k = 0; k < 3; ++k) {
        smin[k][t] = mn[k];
        smax[k][t] = mx[k];
    }
    __syncthreads();
    for (uint32_t s = 128; s > 0; s >>= 1) {
        if (t < s)
            for (int k = 0; k < 3; ++k) {
                smin[k][t] = minf(smin[k][t], smin[k][t + s]);
                smax[k][t] = maxf(smax[k][t], smax[k][t + s]);
            }
        __syncthreads();
    }
    if (t == 0)
        for (int k = 0; k < 3; ++k) {
            partial[6 * blockIdx.x + k] = smin[k][0];
            partial[6 * blockIdx.x + 3 + k] = smax[k][0];
        }
}

// One wavefront folds the partial bounds, a lane every 64th of them (a single
// lane over all took 181 us for 250000 primitives, this 7).
__global__ void __launch_bounds__(64) k_bounds_final(const float* partial, uint32_t nb, float* bounds) {
    float mn[3] = {3.402823466e38f, 3.402823466e38f, 3.402823466e38f};
    float mx[3] = {-3.402823466e38f, -3.402823466e38f, -3.402823466e38f};
    for (uint32_t b = threadIdx.x; b < nb; b += 64u)
        for (int k = 0; k < 3; ++k) {
            mn[k] = minf(mn[k], partial[6 * b + k]);
            mx[k] = maxf(mx[k], partial[6 * b + 3 + k]);
        }
    for (int off = 32; off > 0; off >>= 1)
        for (int k = 0; k < 3; ++k) {
            mn[k] = minf(mn[k], __shfl_xor(mn[k], off));
            mx[k] = maxf(mx[k], __shfl_xor(mx[k], off));
        }
    if (threadIdx.x != 0) return;
    for (int k = 0; k < 3; ++k) {
        bounds[k] = mn[k];
        bounds[3 + k] = 1.0f / maxf(mx[k] + (-mn[k]), 1e-30f);  // inverse extent
    }
}

// morton3D of the reference (host/utils/math.h:117-131).
__global__ void k_morton(const float* centers, uint32_t n, const float* bounds, uint32_t* codes, uint32_t* idx) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t q[3];
    for (int k = 0; k < 3; ++k) {
        const float nrm = (centers[3 * i + k] + (-bounds[k])) * bounds[3 + k];
        q[k] = static_cast<uint32_t>(clampf(nrm, 0.0f, 1.0f) * 1023.0f);
    }
    codes[i] = (expand_bits(q[2]) << 2) | (expand_bits(q[1]) << 1) | expand_bits(q[0]);
    idx[i] = i;
}

// ---- stable LSD radix sort, 8-bit digits ---------------------------------
// A block owns a tile of 2048 keys; item r of thread t is key base + r*256 + t,
// so processing rounds in order and lanes by id visits keys in index order.
__global__ void __launch_bounds__(kSortBlock) k_hist(const uint32_t* keys, uint32_t n, uint32_t shift, uint32_t* hist,
                                                     uint32_t nblocks) {
    __shared__ uint32_t h[256];
    const uint32_t t = threadIdx.x;
    h[t] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * kSortTile;
    for (uint32_t r = 0; r < kSortItems; ++r) {
        const uint32_t i = base + r * kSortBlock + t;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[t * nblocks + blockIdx.x] = h[t];
}

// Exclusive scan of hist (digit-major, block-minor; count is a multiple of
// 256) in one 1024-thread block, 8192 entries a round, eight consecutive ones
// a thread (each thread scanning one long run of its own, read with a stride
// of its length, took 49 us for 250000 keys, this 6).
__global__ void __launch_bounds__(1024) k_scan(uint32_t* hist, uint32_t count) {
    __shared__ uint32_t wave_sum[16];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    uint32_t carry = 0;
    for (uint32_t base = 0; base < count; base += 8192u) {
        const uint32_t i = base + 8u * t;
        uint4* at = reinterpret_cast<uint4*>(hist + i);
        uint4 a = make_uint4(0u, 0u, 0u, 0u), b = a;
        if (i < count) {
            a = at[0];
            b = at[1];
        }
        const uint32_t s = a.x + a.y + a.z + a.w + b.x + b.y + b.z + b.w;
        uint32_t incl = s;
        for (uint32_t off = 1; off < 64u; off <<= 1) {
            const uint32_t u = __shfl_up(incl, off);
            if (lane >= off) incl += u;
        }
        if (lane == 63u) wave_sum[wave] = incl;
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (uint32_t w = 0; w < 16u; ++w) {
            before += w < wave ? wave_sum[w] : 0u;
            all += wave_sum[w];
        }
        if (i < count) {
            uint4 o;
            o.x = carry + before + incl - s;
            o.y = o.x + a.x;
            o.z = o.y + a.y;
            o.w = o.z + a.z;
            at[0] = o;
            o.x = o.w + a.w;
            o.y = o.x + b.x;
            o.z = o.y + b.y;
            o.w = o.z + b.z;
            at[1] = o;
        }
        carry += all;
        __syncthreads();
    }
}

__global__ void __launch_bounds__(kSortBlock) k_scatter(const uint32_t* keys, const uint32_t* vals, uint32_t n,
                                                        uint32_t shift, const uint32_t* offsets, uint32_t nblocks,
                                                        uint32_t* keys_out, uint32_t* vals_out) {
    __shared__ uint32_t s_base[256];
    __shared__ uint32_t s_wave[kSortBlock / 64][256];
    const uint32_t t = threadIdx.x;
    const uint32_t wave = t >> 6;
    const uint32_t lane = t & 63u;
    s_base[t] = offsets[t * nblocks + blockIdx.x];
    for (uint32_t w = 0; w < kSortBlock / 64; ++w) s_wave[w][t] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * kSortTile;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (uint32_t r = 0; r < kSortItems; ++r) {
        const uint32_t i = base + r * kSortBlock + t;
        const bool valid = i < n;
        const uint32_t key = valid ? keys[i] : 0u;
        const uint32_t val = valid ? vals[i] : 0u;
        const uint32_t digit = (key >> shift) & 255u;
        unsigned long long m = __ballot(valid);
        for (uint32_t b = 0; b < 8; ++b) {
            const bool bit = (digit >> b) & 1u;
            const unsigned long long bal = __ballot(bit);
            m &= bit ? bal : ~bal;
        }
        const uint32_t rank = __popcll(m & lt);
        const uint32_t cnt = __popcll(m);
        if (valid && rank == 0) s_wave[wave][digit] = cnt;
        __syncthreads();
        if (valid) {
            uint32_t pre = s_base[digit];
            for (uint32_t w = 0; w < wave; ++w) pre += s_wave[w][digit];
            keys_out[pre + rank] = key;
            vals_out[pre + rank] = val;
        }
        __syncthreads();
        uint32_t add = 0;
        for (uint32_t w = 0; w < kSortBlock / 64; ++w) {
            add += s_wave[w][t];
            s_wave[w][t] = 0;
        }
        s_base[t] += add;
        __syncthreads();
    }
}

// ---- Karras 2012 radix tree ---------------------------------------------
// Keys are (code << 32 | index), unique, so delta = clz64(k_i ^ k_j).
__device__ __forceinline__ int delta(const uint32_t* codes, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    const unsigned long long a = (static_cast<unsigned long long>(codes[i]) << 32) | static_cast<uint32_t>(i);
    const unsigned long long b = (static_cast<unsigned long long>(codes[j]) << 32) | static_cast<uint32_t>(j);
    return __clzll(a ^ b);
}

// Parents of the radix tree's nodes: inner node i is i, leaf k is n - 1 + k.
__global__ void k_karras(const uint32_t* codes, int n, int* parent) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    if (i == 0) parent[0] = -1;
    const int d = (delta(codes, n, i, i + 1) - delta(codes, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(codes, n, i, i - d);
    int lmax = 2;
    while (delta(codes, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(codes, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta(codes, n, i, j);
    int s = 0;
    for (int div = 2;; div <<= 1) {
        const int t = (l + div - 1) / div;
        if (delta(codes, n, i, i + (s + t) * d) > dnode) s += t;
        if (t == 1) break;
    }
    const int gamma = i + s * d + (d < 0 ? -1 : 0);
    const int lo = min(i, j), hi = max(i, j);
    parent[lo == gamma ? n - 1 + gamma : gamma] = i;
    parent[hi == gamma + 1 ? n - 1 + gamma + 1 : gamma + 1] = i;
}

// The tree's depth: the longest way from a leaf to the root (one atomic per
// wavefront).
__global__ void k_depth(int n, const int* parent, uint32_t* max_depth) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t depth = 0;
    if (k < n)
        for (int u = parent[n - 1 + k]; u >= 0; u = parent[u]) ++depth;
    for (int off = 32; off > 0; off >>= 1) depth = max(depth, static_cast<uint32_t>(__shfl_xor(depth, off)));
    if ((threadIdx.x & 63u) == 0u) atomicMax(max_depth, depth);
}

// Records and leaf boxes in stored order.
__global__ void k_gather(const uint32_t* order, uint32_t n, const PrimRecord* rec, const float* box, PrimRecord* rec_out,
                         float* box_out) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t i = order[k];
    rec_out[k] = rec[i];
    for (int q = 0; q < 6; ++q) box_out[6 * k + q] = box[6 * i + q];
}

// ---- walk tree (implicit 4-ary, see vp_walk.h) ----

__device__ __forceinline__ void w4_store(float4* w4, uint32_t idx, const float lo[3][4], const float hi[3][4]) {
    float4* r = w4 + static_cast<size_t>(kW4RecordF4) * idx;
    for (int a = 0; a < 3; ++a) {
        r[a] = make_float4(lo[a][0], lo[a][1], lo[a][2], lo[a][3]);
        r[3 + a] = make_float4(hi[a][0], hi[a][1], hi[a][2], hi[a][3]);
    }
    r[6] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    r[7] = r[6];
}

// Last level: node k holds the leaves 4k .. 4k + 3.
__global__ void k_w4_bottom(const float* box, uint32_t n, uint32_t levels, float4* w4) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (1u << (2u * (levels - 1u)))) return;
    float lo[3][4], hi[3][4];
    for (uint32_t c = 0; c < 4; ++c) {
        const uint32_t j = 4u * k + c;
        for (int a = 0; a < 3; ++a) {
            lo[a][c] = j < n ? box[6 * static_cast<size_t>(j) + a] : INFINITY;
            hi[a][c] = j < n ? box[6 * static_cast<size_t>(j) + 3 + a] : INFINITY;
        }
    }
    w4_store(w4, w4_level_base(levels - 1u) + k, lo, hi);
}

// Level l above the last: the box of child c of node k is the union of the
// children of node 4k + c of level l + 1 (empty children are skipped).
__global__ void k_w4_level(uint32_t l, float4* w4) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (1u << (2u * l))) return;
    float lo[3][4], hi[3][4];
    for (uint32_t c = 0; c < 4; ++c) {
        const float4* r = w4 + static_cast<size_t>(kW4RecordF4) * (w4_level_base(l + 1u) + 4u * k + c);
        const float4 mnx = r[0];
        const float4 full = make_float4(mnx.x < INFINITY ? 1.0f : 0.0f, mnx.y < INFINITY ? 1.0f : 0.0f,
                                        mnx.z < INFINITY ? 1.0f : 0.0f, mnx.w < INFINITY ? 1.0f : 0.0f);
        const bool any = full.x + full.y + full.z + full.w > 0.0f;
        for (int a = 0; a < 3; ++a) {
            const float4 mn = r[a], mx = r[3 + a];
            lo[a][c] = fminf(fminf(mn.x, mn.y), fminf(mn.z, mn.w));
            float h = -INFINITY;
            if (full.x > 0.0f) h = fmaxf(h, mx.x);
            if (full.y > 0.0f) h = fmaxf(h, mx.y);
            if (full.z > 0.0f) h = fmaxf(h, mx.z);
            if (full.w > 0.0f) h = fmaxf(h, mx.w);
            hi[a][c] = any ? h : INFINITY;
        }
    }
    w4_store(w4, w4_level_base(l) + k, lo, hi);
}

// 16-bit records from the 32-bit ones (one thread per record): min bounds
// rounded toward -inf, max bounds toward +inf, packed in the byte order of
// vp_walk.h.  For the last level's records (index >= leaf_base) it also sums
// the surfaces ex ey + ey ez + ez ex of the non-empty leaf boxes, of both
// forms, into sums[0] (32-bit) and sums[1] (16-bit).
__global__ void k_w4_half(const float4* w4, uint32_t records, uint32_t leaf_base, uint4* out, double* sums) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    double s32 = 0.0, s16 = 0.0;
    if (k < records) {
        const float4* r = w4 + static_cast<size_t>(kW4RecordF4) * k;
        float b[6][4];
        uint32_t words[12];
        for (int g = 0; g < 6; ++g) {
            const float4 v = r[g];
            b[g][0] = v.x;
            b[g][1] = v.y;
            b[g][2] = v.z;
            b[g][3] = v.w;
            for (int c = 0; c < 4; c += 2) {
                const uint32_t h0 = g < 3 ? f16_down(b[g][c]) : f16_up(b[g][c]);
                const uint32_t h1 = g < 3 ? f16_down(b[g][c + 1]) : f16_up(b[g][c + 1]);
                words[2 * g + c / 2] = h0 | (h1 << 16);
            }
        }
        uint4* o = out + 4 * static_cast<size_t>(k);
        o[0] = make_uint4(words[0], words[1], words[2], words[3]);
        o[1] = make_uint4(words[4], words[5], words[6], words[7]);
        o[2] = make_uint4(words[8], words[9], words[10], words[11]);
        o[3] = make_uint4(0u, 0u, 0u, 0u);
        if (k >= leaf_base) {
            for (int c = 0; c < 4; ++c) {
                if (!(b[0][c] < INFINITY)) continue;
                double e32[3], e16[3];
                for (int a = 0; a < 3; ++a) {
                    e32[a] = static_cast<double>(b[3 + a][c]) - b[a][c];
                    e16[a] = static_cast<double>(f16_value(f16_up(b[3 + a][c]))) - f16_value(f16_down(b[a][c]));
                }
                s32 += e32[0] * e32[1] + e32[1] * e32[2] + e32[2] * e32[0];
                s16 += e16[0] * e16[1] + e16[1] * e16[2] + e16[2] * e16[0];
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        s32 += __shfl_xor(s32, off);
        s16 += __shfl_xor(s16, off);
    }
    if ((threadIdx.x & 63u) == 0u && s16 != 0.0) {
        atomicAdd(sums, s32);
        atomicAdd(sums + 1, s16);
    }
}

inline uint32_t cdiv(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// Parts of one allocation, each 256-byte aligned; with base null it only
// adds up the bytes.
struct Arena {
    char* base = nullptr;
    size_t used = 0;
    template <typename T>
    T* take(size_t count) {
        T* p = reinterpret_cast<T*>(base + used);
        used += (count * sizeof(T) + 255) / 256 * 256;
        return p;
    }
};

// Device temporaries of a scene build: of the order,
struct OrderTemps {
    vp_primitive* in;
    PrimRecord* rec;                // input order
    float *centers, *box, *partial, *bounds;
    uint32_t *codes, *idx, *codes2, *idx2, *hist, *depth;
    int* parent;
    OrderTemps(Arena& a, uint32_t n, uint32_t nb_sort, uint32_t nbounds) {
        in = a.take<vp_primitive>(n);
        rec = a.take<PrimRecord>(n);
        centers = a.take<float>(3 * static_cast<size_t>(n));
        box = a.take<float>(6 * static_cast<size_t>(n));
        partial = a.take<float>(6 * nbounds);
        bounds = a.take<float>(6);
        codes = a.take<uint32_t>(n);
        idx = a.take<uint32_t>(n);
        codes2 = a.take<uint32_t>(n);
        idx2 = a.take<uint32_t>(n);
        hist = a.take<uint32_t>(256 * static_cast<size_t>(nb_sort));
        depth = a.take<uint32_t>(1);
        parent = a.take<int>(2 * static_cast<size_t>(n));
    }
};
// between the order and the tree,
struct BoxTemps {
    float* sorted_box;
    double* sums;
    BoxTemps(Arena& a, uint32_t n) {
        sorted_box = a.take<float>(6 * static_cast<size_t>(n));
        sums = a.take<double>(2);
    }
};
// and of the tree.
struct TreeTemps {
    float4* w4;                     // 32-bit records
    uint4* w4_half;
    TreeTemps() = default;
    TreeTemps(Arena& a, size_t records) {
        w4 = a.take<float4>(kW4RecordF4 * records);
        w4_half = a.take<uint4>(kW4hRecordB / sizeof(uint4) * records);
    }
};

struct DevMem {
    void* p = nullptr;
    DevMem() = default;
    DevMem(const DevMem&) = delete;
    DevMem& operator=(const DevMem&) = delete;
    ~DevMem() {
        if (p) (void)hipFree(p);
    }
};

vp_status scene_malloc(vp_context* ctx, void** p, size_t bytes) {
    if (vp_device_malloc(ctx, p, bytes) == hipSuccess) return VP_OK;
    *p = nullptr;
    (void)hipGetLastError();
    vp_set_error("cannot allocate " + std::to_string(bytes) + " bytes of device memory");
    return VP_ERR_OOM;
}

}  // namespace
}  // namespace vp

// The build of scene sc (see vp_build_scene).  Its temporaries are one block
// of scratch, or (staged) one of each stage's own, the order's released before
// the tree's are taken: 2 more allocations and a wait, but 276 bytes a
// primitive, then 104 and 192 a node, at once, scene included, against 276
// and 320.
static vp_status build_scene(vp_context* ctx, const vp_primitive* host_prims, uint32_t n, uint32_t flags, vp_scene* sc,
                             bool staged) {
    using namespace vp;
    hipStream_t s = ctx->stream;
    const uint32_t nb_sort = cdiv(n, kSortTile);
    const uint32_t nbounds = min(cdiv(n, 256u), 1024u);
    const uint32_t levels = w4_levels(n);
    const size_t records = w4_records(levels);
    Arena order_need, box_need, tree_need;
    OrderTemps(order_need, n, nb_sort, nbounds);
    BoxTemps(box_need, n);
    TreeTemps(tree_need, records);
    ScratchLease boxes, first;
    DevMem w4_32, w4_16;  // of the staged form
    vp_status st = vp_lease_scratch(ctx, staged ? order_need.used : order_need.used + box_need.used + tree_need.used,
                                    s, first);
    if (st == VP_OK && staged) st = vp_lease_scratch(ctx, box_need.used, s, boxes);
    if (st != VP_OK) return st;
    Arena arena, box_arena;
    arena.base = static_cast<char*>(first.p);
    box_arena.base = static_cast<char*>(boxes.p);
    const OrderTemps T(arena, n, nb_sort, nbounds);
    const BoxTemps B(staged ? box_arena : arena, n);
    // the records are padded to a multiple of the leaf block with zero records
    // (zero inverse scales: no ray enters them), so a walk may hand every slot
    // of a leaf block to the leaf tests
    const size_t n_slots = (static_cast<size_t>(n) + kLeafBlock - 1u) / kLeafBlock * kLeafBlock;
    for (int pass = 0; pass < 2; ++pass) {
        Arena a;
        a.base = static_cast<char*>(sc->mem);
        sc->prims = a.take<PrimRecord>(n_slots);
        sc->order = a.take<uint32_t>(n);
        sc->morton = a.take<uint32_t>(n);
        if (pass == 0 && (st = scene_malloc(ctx, &sc->mem, a.used)) != VP_OK) return st;
    }
    if (n_slots > n) VP_HIP_TRY(hipMemsetAsync(sc->prims + n, 0, sizeof(PrimRecord) * (n_slots - n), s));
    bool valid = false;
    st = vp_copy_in(ctx, T.in, host_prims, sizeof(vp_primitive), n, vp_primitives_valid, &valid, s);
    if (st != VP_OK || !valid) return st != VP_OK ? st : VP_ERR_INVALID;
    VP_HIP_TRY(hipMemsetAsync(T.depth, 0, sizeof(uint32_t), s));
    VP_HIP_TRY(hipMemsetAsync(B.sums, 0, 2 * sizeof(double), s));

    const uint32_t g = cdiv(n, 256u);
    hipLaunchKernelGGL(k_setup, dim3(g), dim3(256), 0, s, T.in, n, T.rec, T.centers, T.box);
    hipLaunchKernelGGL(k_bounds_partial, dim3(nbounds), dim3(256), 0, s, T.centers, n, T.partial);
    hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(64), 0, s, T.partial, nbounds, T.bounds);
    hipLaunchKernelGGL(k_morton, dim3(g), dim3(256), 0, s, T.centers, n, T.bounds, T.codes, T.idx);
    VP_HIP_TRY(hipGetLastError());
    VP_HIP_TRY(hipMemcpyAsync(sc->morton, T.codes, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, s));

    uint32_t depth = 0;
    std::vector<uint32_t> host_order;
    const bool host_tree = (flags & (VP_SCENE_BVH_SAH | VP_SCENE_BVH_MEDIAN)) != 0u;
    if (host_tree) {
        vp_host_tree_order(host_prims, n, (flags & VP_SCENE_BVH_MEDIAN) != 0u, host_order, sc->depth);
        VP_HIP_TRY(hipMemcpyAsync(sc->order, host_order.data(), sizeof(uint32_t) * n, hipMemcpyHostToDevice, s));
    } else {
        uint32_t *kin = T.codes, *vin = T.idx, *kout = T.codes2, *vout = T.idx2;
        for (uint32_t shift = 0; shift < 32; shift += 8) {
            hipLaunchKernelGGL(k_hist, dim3(nb_sort), dim3(kSortBlock), 0, s, kin, n, shift, T.hist, nb_sort);
            hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, s, T.hist, 256 * nb_sort);
            hipLaunchKernelGGL(k_scatter, dim3(nb_sort), dim3(kSortBlock), 0, s, kin, vin, n, shift, T.hist, nb_sort,
                               kout, vout);
            std::swap(kin, kout);
            std::swap(vin, vout);
        }
        // after 4 passes the sorted data is back in kin/vin
        VP_HIP_TRY(hipMemcpyAsync(sc->order, vin, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, s));
        if (n > 1) {
            hipLaunchKernelGGL(k_karras, dim3(cdiv(n - 1, 256u)), dim3(256), 0, s, kin, (int)n, T.parent);
            hipLaunchKernelGGL(k_depth, dim3(g), dim3(256), 0, s, (int)n, T.parent, T.depth);
        }
        VP_HIP_TRY(hipGetLastError());
    }
    hipLaunchKernelGGL(k_gather, dim3(g), dim3(256), 0, s, sc->order, n, T.rec, T.box, sc->prims, B.sorted_box);
    TreeTemps R = staged ? TreeTemps{} : TreeTemps(arena, records);
    if (staged) {
        const HostCopy out{&depth, T.depth, sizeof(depth)};
        if ((st = vp_copy_out(ctx, &out, 1, s)) != VP_OK) return st;
        first.release();
        st = scene_malloc(ctx, &w4_32.p, sizeof(float4) * kW4RecordF4 * records);
        if (st == VP_OK && !(flags & VP_SCENE_WALK_F32))
            st = scene_malloc(ctx, &w4_16.p, static_cast<size_t>(kW4hRecordB) * records);
        if (st != VP_OK) return st;
        R.w4 = static_cast<float4*>(w4_32.p);
        R.w4_half = static_cast<uint4*>(w4_16.p);
    }

    // the walk tree in 32-bit records, bottom up
    const uint32_t bottom = 1u << (2u * (levels - 1u));
    hipLaunchKernelGGL(k_w4_bottom, dim3(cdiv(bottom, 256u)), dim3(256), 0, s, B.sorted_box, n, levels, R.w4);
    for (uint32_t l = levels - 1u; l-- > 0;)
        hipLaunchKernelGGL(k_w4_level, dim3(cdiv(1u << (2u * l), 256u)), dim3(256), 0, s, l, R.w4);
    sc->w4_levels = levels;
    // the 16-bit records, kept when forced or when the leaf boxes' summed
    // surface grows by at most 1/16 (more leaf tests and node visits, against
    // half the bytes per node visit)
    double sums[2] = {0.0, 0.0};
    if (!(flags & VP_SCENE_WALK_F32)) {
        hipLaunchKernelGGL(k_w4_half, dim3(cdiv(static_cast<uint32_t>(records), 256u)), dim3(256), 0, s, R.w4,
                           static_cast<uint32_t>(records), w4_level_base(levels - 1u), R.w4_half, B.sums);
    }
    VP_HIP_TRY(hipGetLastError());
    const HostCopy outs[2] = {{sums, B.sums, sizeof(sums)}, {&depth, T.depth, sizeof(depth)}};
    st = vp_copy_out(ctx, outs, staged ? 1 : 2, s);
    if (st != VP_OK) return st;
    if (!host_tree) sc->depth = depth;
    sc->w4_growth = sums[0] > 0.0 ? sums[1] / sums[0] - 1.0 : 0.0;
    const bool half = !(flags & VP_SCENE_WALK_F32) && ((flags & VP_SCENE_WALK_F16) || sc->w4_growth <= 1.0 / 16.0);
    sc->w4_half = half ? 1u : 0u;
    if (staged) {
        DevMem& kept = half ? w4_16 : w4_32;
        sc->w4 = static_cast<float4*>(kept.p);
        kept.p = nullptr;
    } else {
        const size_t w4_bytes = (half ? static_cast<size_t>(kW4hRecordB) : sizeof(float4) * kW4RecordF4) * records;
        void* w4 = nullptr;
        if ((st = scene_malloc(ctx, &w4, w4_bytes)) != VP_OK) return st;
        sc->w4 = static_cast<float4*>(w4);
        VP_HIP_TRY(hipMemcpyAsync(w4, half ? static_cast<const void*>(R.w4_half) : R.w4, w4_bytes,
                                  hipMemcpyDeviceToDevice, s));
    }
    VP_HIP_TRY(hipStreamSynchronize(s));
    first.done = boxes.done = true;
    return VP_OK;
}

// Builds scene sc (whose n is set): records, Morton codes and stored order,
// the order from the radix sort or, with VP_SCENE_BVH_SAH / _MEDIAN in flags,
// from the host tree, and the walk tree over it.  Temporaries are scratch;
// the scene owns two allocations.  Returns VP_ERR_INVALID without a message
// where a primitive is not valid.
vp_status vp_build_scene(vp_context* ctx, const vp_primitive* host_prims, uint32_t n, uint32_t flags, vp_scene* sc) {
    const vp_status st = build_scene(ctx, host_prims, n, flags, sc, false);
    if (st != VP_ERR_OOM) return st;
    if (sc->mem) (void)hipFree(sc->mem);
    sc->mem = nullptr;
    return build_scene(ctx, host_prims, n, flags, sc, true);
}
