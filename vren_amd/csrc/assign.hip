// assign.hip -- assign_lights (clustered_shading.cpp:473-690, assign_lights.comp:77-241,
// clustered_shading.glsl:58-110).
//
// Reference: one wave32 per unique cluster (indirect dispatch), a DFS over the 32-ary BVH with a per-level
// ballot stack, run twice (COUNT then WRITE) around a fixed 2^17-entry Blelloch scan of the counts; lists come
// out in traversal order with reversed lanes inside each leaf block.
// Here: persistent kernels over the clusters of every frame (their number is read on the device; it never returns
// to the host). COUNT takes them in chunks of up to 64 whose AABBs are computed one cluster per lane, runs two
// traversals per wave, one per 32-lane half (the BVH's fan-out), each from its own LDS stack, and keeps lists of at most
// VREN_LIST_SLOT (192) lights, sorted by rank, in per-cluster slots; LISTS turns the counts into offsets, copies the
// kept lists and traverses again only for longer ones, with the whole wave testing two BVH blocks per step, one bit per
// hit light in an LDS bitmask, emitted in ascending light index (the canonical order) by a popcount prefix over the
// bitmask words.
// The cluster AABB and both tests are restated operation for operation (including the inverted y range of
// the two-corner AABB); padding leaves and invalid nodes (empty AABB) never match.
#include "chain.hpp"
#include "scan_device.hpp"

namespace {

constexpr uint32_t kStack = 384; // per-wave stack entries (levels are nondecreasing on the stack: <= 64 per level)
// per-half entries of the counting pass: the stack holds blocks of inner nodes (a half pops one and pushes at most 32, so
// at most 31 entries of each level above the deepest inner one and 32 of that, 31 * 2 + 32 = 94 for 2^20 lights), the
// leaf list blocks of leaves, which are tested when it has no room for 32 more or no inner block is left
constexpr uint32_t kStackHalf = 96;
// (128 entries and 64 take the same time)
constexpr uint32_t kLeafList = 128;
// leaf blocks per half and step, whose loads overlap: a 1920x1080 frame with 4096 lights takes 77.0 us with 2, 76.7 with 4 and
// 81.9 with 8, the stage calls of a 1366x769 frame 66.1, 66.7 and 79.7 (eight blocks' nodes and positions do not fit the
// registers of eight waves per SIMD)
constexpr int kLeafUnroll = 4;
constexpr uint32_t kLevelShift = 28;
constexpr uint32_t kAddrMask = (1u << kLevelShift) - 1u;

struct Box {
    float mn[3], mx[3];
};

__device__ Box cluster_aabb(const FrameDev& fd, uint32_t key)
{
    uint32_t ci = key & 0xFFu, cj = (key >> 8) & 0xFFu, ck;
    float near_k, far_k;
    if (fd.key_mode == VREN_KEYS_SLICED) {
        ck = (key >> 16) & 0xFFu;
        float S = (float)fd.depth_slices;
        near_k = fd.near_plane * vren_expf((float)ck / S * fd.log_fn);
        far_k = fd.near_plane * vren_expf((float)(ck + 1) / S * fd.log_fn);
    } else {
        ck = (key >> 16) & 0x3FFu;
        near_k = fd.near_plane * vren_powi(fd.slice_a, ck);
        far_k = near_k * fd.slice_a;
    }
    const float fSx = (float)fd.Sx, fSy = (float)fd.Sy;
    const float x0 = (float)ci / fSx, y0 = (float)cj / fSy;
    const float x1 = (float)(ci + 1) / fSx, y1 = (float)(cj + 1) / fSy;
    Box b;
    if (fd.aabb_mode == VREN_CLUSTER_AABB_TIGHT) {
        for (int a = 0; a < 3; a++) {
            b.mn[a] = VREN_F32_INF;
            b.mx[a] = -VREN_F32_INF;
        }
        for (int corner = 0; corner < 4; corner++) {
            float cx = (corner & 1) ? x1 : x0, cy = (corner & 2) ? y1 : y0;
            float v[4] = {cx * 2.0f - 1.0f, (1.0f - cy) * 2.0f - 1.0f, 0.0f, 1.0f};
            float r[4];
            vren_mat4_mul_vec4(fd.inv_proj, v, r);
            float p[3] = {r[0] / r[3], r[1] / r[3], r[2] / r[3]};
            float d[3];
            vren_normalize3(p, d);
            for (int plane = 0; plane < 2; plane++) {
                float zp = plane ? far_k : near_k;
                float sc = zp / d[2];
                for (int a = 0; a < 3; a++) {
                    float q = sc * d[a];
                    b.mn[a] = tmin(b.mn[a], q);
                    b.mx[a] = tmax(b.mx[a], q);
                }
            }
        }
        return b;
    }
    float vmin[4] = {x0, 1.0f - y0, 0.0f, 1.0f};
    vmin[0] = vmin[0] * 2.0f - 1.0f;
    vmin[1] = vmin[1] * 2.0f - 1.0f;
    float vmax[4] = {x1, 1.0f - y1, 0.0f, 1.0f};
    vmax[0] = vmax[0] * 2.0f - 1.0f;
    vmax[1] = vmax[1] * 2.0f - 1.0f;
    float rmin[4], rmax[4];
    vren_mat4_mul_vec4(fd.inv_proj, vmin, rmin);
    vren_mat4_mul_vec4(fd.inv_proj, vmax, rmax);
    float pmin[3] = {rmin[0] / rmin[3], rmin[1] / rmin[3], rmin[2] / rmin[3]};
    float pmax[3] = {rmax[0] / rmax[3], rmax[1] / rmax[3], rmax[2] / rmax[3]};
    float d1[3], d2[3];
    vren_normalize3(pmin, d1);
    vren_normalize3(pmax, d2);
    const float s1 = near_k / d1[2], s2 = far_k / d2[2];
    for (int a = 0; a < 3; a++) {
        b.mn[a] = s1 * d1[a];
        b.mx[a] = s2 * d2[a];
    }
    return b;
}

__device__ __forceinline__ float gmin(float x, float y) { return y < x ? y : x; }
__device__ __forceinline__ float gmax(float x, float y) { return x < y ? y : x; }

// test_aabb_aabb (assign_lights.comp:84-94), cluster first
__device__ __forceinline__ bool test_aabb_aabb(const Box& c, const float4& lo, const float4& hi)
{
    return c.mx[0] >= lo.x && c.mn[0] <= hi.x && c.mx[1] >= lo.y && c.mn[1] <= hi.y && c.mx[2] >= lo.z &&
           c.mn[2] <= hi.z;
}

// assign_lights.comp:97-102 with r = (max.x - min.x) / 2 (assign_lights.comp:214)
__device__ __forceinline__ bool test_leaf(const Box& c, const float4& o, float leaf_min_x, float leaf_max_x)
{
    const float r = (leaf_max_x - leaf_min_x) / 2.0f;
    float d[3];
    const float oo[3] = {o.x, o.y, o.z};
    for (int a = 0; a < 3; a++) {
        float p = gmax(c.mn[a], gmin(oo[a], c.mx[a]));
        d[a] = p - oo[a];
    }
    return vren_sqrtf(vren_dot3(d, d)) < r;
}

// The same test against a leaf record (position, limit): the limit is the smallest squared distance whose square root
// is not below the light's radius (leaf_limit, lights_device.hpp), 0 for a record without a light, so sqrt(d2) < r is
// d2 < limit exactly, without the square root and the node. The clamp as plain minimum and maximum: a NaN position
// gives a NaN distance either way, and leaf_box takes the boxes with a NaN lower corner out.
__device__ __forceinline__ bool test_leaf_record(const Box& c, vf4 o)
{
    float d[3];
    const float oo[3] = {o.x, o.y, o.z};
    for (int a = 0; a < 3; a++) d[a] = fmaxf(c.mn[a], fminf(oo[a], c.mx[a])) - oo[a];
    return vren_dot3(d, d) < o.w;
}

// a cluster box for the traversal: one with a NaN in its lower corner, which no node and no leaf meets, becomes one
// that meets none by its numbers
__device__ __forceinline__ Box leaf_box(Box c)
{
    const bool nan = !(c.mn[0] == c.mn[0] && c.mn[1] == c.mn[1] && c.mn[2] == c.mn[2]);
    for (int a = 0; a < 3; a++) {
        c.mn[a] = nan ? VREN_F32_INF : c.mn[a];
        c.mx[a] = nan ? -VREN_F32_INF : c.mx[a];
    }
    return c;
}

// Traverse the BVH for one cluster with the whole wave, setting one bit per hit light in the wave's LDS bitmask (and
// the word's bit in the summary, one bit per bitmask word).
__device__ void traverse(const FrameDev& fd, const Box& box, uint32_t* stack, uint32_t* bitmask,
                             uint32_t* summary)
{
    const uint32_t lane = lane_id();
    const uint32_t sub = lane & 31u;
    const uint32_t leaf_level = fd.bvh_levels - 1;
    const vren_bvh_node* bvh = fd.bvh;
    // level 0 = the root's children (assign_lights.comp:108-119): the first child of the root
    const uint32_t root_first = __float_as_uint(reinterpret_cast<const float4*>(&bvh[fd.bvh_root])[0].w);
    uint32_t sp = 0;
    if (root_first == VREN_BVH_INVALID_NODE) return;
    if (lane == 0) stack[0] = root_first; // level 0
    sp = 1;
    __builtin_amdgcn_wave_barrier();
    while (sp > 0) {
        uint32_t e0, e1 = 0xFFFFFFFFu;
        if (sp >= 2) {
            e0 = stack[sp - 2];
            e1 = stack[sp - 1];
            sp -= 2;
        } else {
            e0 = stack[sp - 1];
            sp -= 1;
        }
        const uint32_t e = lane < 32 ? e0 : e1;
        // entries always address a whole 32-node block inside the BVH; anything else is ignored
        const bool active = e != 0xFFFFFFFFu && (e >> kLevelShift) <= leaf_level &&
                            (e & kAddrMask) + 32u <= fd.bvh_length;
        bool leaf_hit = false, push = false;
        uint32_t child = 0, level = 0, li = 0xFFFFFFFFu;
        if (active) {
            level = e >> kLevelShift;
            const uint32_t addr = (e & kAddrMask) + sub;
            if (level == leaf_level) {
                if (addr < fd.L) {
                    li = *((guint*)fd.codes + 2 * (uint64_t)addr + 1);
                    if (fd.leaf_rec) {
                        leaf_hit = test_leaf_record(box, *((gvf4*)fd.leaf_rec + addr));
                    } else {
                        const vf4 lo = *((gvf4*)&bvh[addr]), hi = *((gvf4*)&bvh[addr] + 1);
                        if (__float_as_uint(lo.w) == VREN_BVH_LEAF_NODE && li < fd.L) {
                            const vf4 v = *((gvf4*)fd.view_pos + li);
                            leaf_hit = test_leaf(box, make_float4(v.x, v.y, v.z, 0.f), lo.x, hi.x);
                        }
                    }
                }
                if (leaf_hit) {
                    atomicOr(&bitmask[li >> 5], 1u << (li & 31u));
                    atomicOr(&summary[li >> 10], 1u << ((li >> 5) & 31u));
                }
            } else {
                const vf4 lo = *((gvf4*)&bvh[addr]), hi = *((gvf4*)&bvh[addr] + 1);
                const uint32_t next = __float_as_uint(lo.w);
                push = next < VREN_BVH_INVALID_NODE &&
                       test_aabb_aabb(box, make_float4(lo.x, lo.y, lo.z, 0.f), make_float4(hi.x, hi.y, hi.z, 0.f));
                child = next | ((level + 1) << kLevelShift);
            }
        }
        const uint64_t pm = ballot(push);
        if (pm) {
            const uint32_t r = mbcnt(pm);
            if (push && sp + r < kStack) stack[sp + r] = child;
            sp += (uint32_t)__popcll(pm);
            if (sp > kStack) sp = kStack; // unreachable by the level bound; never write past the stack
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Two traversals of one frame's BVH at once, one per 32-lane half of the wave (lanes 0-31 and 32-63, each with its own
// cluster box, stack and lists; a half with live = false does nothing). Inner blocks are popped one per half and step, each
// child tested by a lane of the half; the blocks of leaves that they reach wait in the half's leaf list and are tested
// kLeafUnroll at a time, so that the two kinds of test do not share a step (a step issued both before: 96 instructions,
// now about 60 and 30 a block) and the leaves' loads overlap. Counts the hit lights of each half (returned to every
// lane of the half) and keeps the first VREN_LIST_SLOT of them in `list` (traversal order): the leaf's place with
// COMPACT (leaf records; the caller looks the light index up), else the light index.
template <bool COMPACT>
__device__ __forceinline__ uint32_t traverse_halves(const FrameDev& fd, const Box& box, bool live, uint32_t* stack,
                                                    uint32_t* leaves, uint32_t* list)
{
    const uint32_t leaf_level = fd.bvh_levels - 1, length = fd.bvh_length;
    const vren_bvh_node* bvh = fd.bvh;
    const uint32_t lane = lane_id();
    const uint32_t sub = lane & 31u;
    const uint64_t half = lane < 32 ? 0x00000000FFFFFFFFull : 0xFFFFFFFF00000000ull;
    // leaf blocks end by this (at least 32): the groups of 32 that hold a light (records), or the nodes
    const uint32_t leaf_end = COMPACT ? (fd.L + 31u) & ~31u : length;
    // level 0 = the root's children (assign_lights.comp:108-119), the 32 nodes ahead of the root in a chain's own BVH (its
    // root is valid: there is a light); a caller's BVH says where they are
    uint32_t sp = 0, m = 0; // the half's stack and leaf-list entries
    const uint32_t root_first = COMPACT ? fd.bvh_root - 32u : *((guint*)&bvh[fd.bvh_root] + 3);
    if (live && root_first != VREN_BVH_INVALID_NODE) {
        if (leaf_level == 0) {
            if (root_first <= leaf_end - 32u) {
                if (sub == 0) leaves[0] = root_first;
                m = 1;
            }
        } else {
            if (sub == 0) stack[0] = root_first;
            sp = 1;
        }
    }
    uint32_t hits = 0;
    __builtin_amdgcn_wave_barrier();
    for (;;) {
        // inner blocks, while both leaf lists have room
        while (ballot(sp > 0) && !ballot(m + 32u > kLeafList)) {
            uint32_t e = 0xFFFFFFFFu;
            if (sp > 0) {
                e = stack[sp - 1];
                sp -= 1;
            }
            const uint32_t level = e >> kLevelShift, addr = (e & kAddrMask) + sub;
            bool push = false;
            uint32_t next = 0;
            // entries always address a whole 32-node block of inner nodes in the BVH; anything else is ignored
            if (e != 0xFFFFFFFFu && level < leaf_level && (e & kAddrMask) + 32u <= length) {
                const vf4 lo = load_at<vf4>(bvh, 2 * addr), hi = load_at<vf4>(bvh, 2 * addr + 1);
                next = __float_as_uint(lo.w);
                push = next < VREN_BVH_INVALID_NODE &&
                       test_aabb_aabb(box, make_float4(lo.x, lo.y, lo.z, 0.f), make_float4(hi.x, hi.y, hi.z, 0.f));
            }
            const bool to_leaves = level + 1u == leaf_level; // uniform in the half
            push = push && (!to_leaves || next <= leaf_end - 32u);
            const uint64_t pm = ballot(push) & half;
            const uint32_t r = mbcnt(pm), n = (uint32_t)__popcll(pm);
            if (push) {
                if (to_leaves) leaves[m + r] = next; // m + 32 <= kLeafList
                else if (sp + r < kStackHalf) stack[sp + r] = next | ((level + 1u) << kLevelShift);
            }
            if (to_leaves) m += n;
            else sp = min(sp + n, kStackHalf); // the level bound keeps it below kStackHalf
            __builtin_amdgcn_wave_barrier();
        }
        // leaf blocks
        for (uint32_t k = 0; ballot(k < m); k += kLeafUnroll) {
            uint32_t addr[kLeafUnroll];
            bool on[kLeafUnroll], hit[kLeafUnroll];
#pragma unroll
            for (int u = 0; u < kLeafUnroll; u++) {
                on[u] = k + u < m;
                addr[u] = (on[u] ? leaves[k + u] : 0u) + sub;
            }
            if constexpr (COMPACT) {
                vf4 rec[kLeafUnroll];
#pragma unroll
                for (int u = 0; u < kLeafUnroll; u++) rec[u] = on[u] ? load_at<vf4>(fd.leaf_rec, addr[u]) : vf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < kLeafUnroll; u++) hit[u] = test_leaf_record(box, rec[u]); // limit 0: never
            } else {
                // the blocks' nodes and light indices together, then their positions together (entry 0 of each array in
                // place of what there is not): two loads' latency a step (a 1366x769 frame with 1000 lights 17.5 -> 16.2 us)
                vf4 lo[kLeafUnroll], pos[kLeafUnroll];
                float hi_x[kLeafUnroll];
                uint32_t li[kLeafUnroll];
#pragma unroll
                for (int u = 0; u < kLeafUnroll; u++) {
                    on[u] = on[u] && addr[u] < fd.L;
                    const uint32_t at = on[u] ? addr[u] : 0u;
                    lo[u] = load_at<vf4>(bvh, 2 * at);
                    hi_x[u] = load_at<float>(bvh, 8 * at + 4);
                    li[u] = load_at<uint32_t>(fd.codes, 2 * at + 1);
                }
#pragma unroll
                for (int u = 0; u < kLeafUnroll; u++) {
                    on[u] = on[u] && __float_as_uint(lo[u].w) == VREN_BVH_LEAF_NODE && li[u] < fd.L;
                    pos[u] = load_at<vf4>(fd.view_pos, on[u] ? li[u] : 0u);
                }
#pragma unroll
                for (int u = 0; u < kLeafUnroll; u++) {
                    addr[u] = li[u]; // what the list keeps
                    hit[u] = on[u] && test_leaf(box, make_float4(pos[u].x, pos[u].y, pos[u].z, 0.f), lo[u].x, hi_x[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < kLeafUnroll; u++) {
                const uint64_t all = ballot(hit[u]);
                if (all == 0) continue; // uniform
                const uint64_t hm = all & half;
                const uint32_t pos = hits + mbcnt(hm);
                if (hit[u] && pos < VREN_LIST_SLOT) list[pos] = addr[u];
                hits += (uint32_t)__popcll(hm);
            }
        }
        m = 0;
        if (!ballot(sp > 0)) break;
        __builtin_amdgcn_wave_barrier();
    }
    return hits;
}

// Clusters per chunk: about four chunks per wave, strided over the whole range, so that every wave samples every
// part of the frames (the costly clusters, those covering many lights, sit together in the image), at most 64
// (one per lane).
__device__ __forceinline__ uint32_t chunk_size(uint32_t total, uint32_t waves)
{
    // 32-bit arithmetic: total <= 64 frames x 2^20 clusters and waves < 2^20, so nothing here wraps
    return max(1u, min(VREN_WAVE, (total + 4u * waves - 1u) / (4u * waves)));
}

// Clusters of every frame of the table are counted as one flattened range, in chunks of at most 64 consecutive
// clusters per wave: lane i takes cluster i of the chunk, finds its frame among 64 frames at a time (their
// device-side cluster counts, one per lane, prefix-summed) and runs pre(fd, c) (the cluster AABB), so work that is
// uniform per cluster is done for a whole chunk at once. Then the whole wave runs fn(fd, k, two, cA, cB) for clusters
// k and, with `two`, k + 1 of the chunk, cA and cB their frame-local indices; the two are of one frame, so that its record
// is uniform and read with scalar loads.
template <typename Pre, typename Fn>
__device__ __forceinline__ void for_each_cluster_pair(const FrameDev* __restrict__ frames, uint32_t F, uint32_t gw,
                                                        uint32_t stride, Pre pre, Fn fn)
{
    const uint32_t lane = lane_id();
    for (uint32_t f0 = 0; f0 < F; f0 += VREN_WAVE) {
        const uint32_t fi = f0 + lane;
        uint32_t nf = 0;
        if (fi < F) {
            const FrameDev& d = frames[fi];
            if (d.L != 0 && d.cluster_count != nullptr) nf = min(*d.cluster_count, d.key_cap);
        }
        const uint32_t incl = wave_inclusive_sum(nf);
        const uint32_t excl = incl - nf;
        const uint32_t total = __builtin_amdgcn_readlane(incl, VREN_WAVE - 1);
        const uint32_t cs = chunk_size(total, stride);
        const uint32_t chunks = (total + cs - 1u) / cs;
        // the chunks in eight contiguous blocks, one per XCD (workgroup b runs on XCD b mod 8), each block strided
        // over that XCD's waves: an L2 then holds the BVHs of an eighth of the frames (a grid that is not a
        // multiple of 8 workgroups keeps the plain stride)
        uint32_t first = gw, end = chunks, step = stride;
        if (gridDim.x % 8u == 0u) {
            const uint32_t xcd = blockIdx.x % 8u, wpb = blockDim.x / VREN_WAVE;
            first = (uint32_t)((uint64_t)chunks * xcd / 8u) + (blockIdx.x / 8u) * wpb + gw % wpb;
            end = (uint32_t)((uint64_t)chunks * (xcd + 1u) / 8u);
            step = stride / 8u;
        }
        for (uint32_t chunk = first; chunk < end; chunk += step) {
            const uint32_t c0 = chunk * cs;
            const uint32_t c = c0 + lane;
            uint32_t pos = 0;
#pragma unroll
            for (uint32_t step = VREN_WAVE / 2; step >= 1; step >>= 1)
                if (shfl(incl, (int)(pos + step - 1)) <= c) pos += step;
            const uint32_t fl = min(pos, VREN_WAVE - 1);
            const uint32_t base = shfl(excl, (int)fl);
            if (lane < cs && c < total) pre(frames[f0 + fl], c - base);
            const uint32_t local = c - base;
            const uint32_t n = min(total - c0, cs);
            for (uint32_t k = 0; k < n;) {
                const uint32_t k1 = min(k + 1, n - 1), f = __builtin_amdgcn_readlane(fl, k);
                const bool two = k1 != k && (uint32_t)__builtin_amdgcn_readlane(fl, k1) == f;
                fn(frames[f0 + f], k, two, __builtin_amdgcn_readlane(local, k), __builtin_amdgcn_readlane(local, k1));
                k += two ? 2u : 1u;
            }
        }
    }
}


// Emits the lights set in a wave's bitmask in ascending index to dst[0 .. cap), clearing the bitmask and its summary.
// Only the words the summary marks are read: lane l of a
// step takes summary word s0 + l (bitmask words 32 (s0 + l) ..), counts its lights, and writes them after the
// lights of the lanes before it, so a cluster's list costs its hit words, not the L / 32 words of the mask.
__device__ __forceinline__ void emit_bitmask(uint32_t* bitmask, uint32_t* summary, uint32_t summary_words, uint32_t* dst,
                                             uint32_t cap)
{
    const uint32_t lane = lane_id();
    uint32_t out = 0;
    for (uint32_t s0 = 0; s0 < summary_words; s0 += VREN_WAVE) {
        const uint32_t si = s0 + lane;
        const uint32_t sw = si < summary_words ? summary[si] : 0u;
        if (sw) summary[si] = 0u;
        uint32_t cnt = 0;
        for (uint32_t m = sw; m; m &= m - 1u) cnt += (uint32_t)__popc(bitmask[si * 32u + __builtin_ctz(m)]);
        const uint32_t incl = wave_inclusive_sum(cnt);
        uint32_t pos = out + incl - cnt;
        for (uint32_t m = sw; m; m &= m - 1u) {
            const uint32_t wi = si * 32u + (uint32_t)__builtin_ctz(m);
            uint32_t bits = bitmask[wi];
            bitmask[wi] = 0u;
            while (bits) {
                const uint32_t b = (uint32_t)__builtin_ctz(bits);
                bits &= bits - 1u;
                if (pos < cap) dst[pos] = wi * 32u + b;
                pos++;
            }
        }
        out += __builtin_amdgcn_readlane(incl, VREN_WAVE - 1);
    }
}

// COUNT (assign_lights.comp, count pass): two clusters per wave at a time (one per half, traverse_halves), each
// counting its hit lights and keeping the first VREN_LIST_SLOT of them in the half's LDS list; a list of at most
// VREN_LIST_SLOT lights is sorted (the rank of each index among the list) into the cluster's slot, so the writing
// pass copies it instead of traversing again.
template <bool COMPACT>
__device__ __forceinline__ void assign_count_body(const FrameDev* __restrict__ frames, uint32_t F, uint32_t* s_mem)
{
    const uint32_t wpb = blockDim.x / VREN_WAVE;
    const uint32_t wave = wave_id();
    const uint32_t lane = lane_id();
    const uint32_t hb = lane < 32 ? 0u : 1u; // half of the wave
    constexpr uint32_t kHalf = kStackHalf + kLeafList + VREN_LIST_SLOT;
    uint32_t* stack = s_mem + (wave * 2 + hb) * kHalf;
    uint32_t* leaves = stack + kStackHalf;
    uint32_t* list = leaves + kLeafList;
    Box* boxes = reinterpret_cast<Box*>(s_mem + wpb * 2 * kHalf) + wave * VREN_WAVE;
    const uint32_t gw = blockIdx.x * wpb + wave;
    // the chunk's cluster AABBs wait in LDS (one per lane) while the wave traverses two at a time
    for_each_cluster_pair(
        frames, F, gw, gridDim.x * wpb,
        [&](const FrameDev& fdl, uint32_t c) { boxes[lane] = leaf_box(cluster_aabb(fdl, fdl.keys[c])); },
        [&](const FrameDev& fd, uint32_t k, bool two, uint32_t cA, uint32_t cB) {
            // half 0: cluster k of the chunk, half 1: cluster k + 1
            __builtin_amdgcn_wave_barrier();
            const bool live = hb == 0 || two;
            const uint32_t c = hb ? cB : cA;
            const Box box = boxes[live ? k + hb : k];
            const uint32_t h = traverse_halves<COMPACT>(fd, box, live, stack, leaves, list);
            __builtin_amdgcn_wave_barrier();
            const bool keep = live && fd.list_slots && c < fd.slot_cap && h <= VREN_LIST_SLOT;
            if constexpr (COMPACT) {
                if (keep)
                    for (uint32_t q = lane & 31u; q < h; q += 32u) list[q] = load_at<uint32_t>(fd.codes, 2 * list[q] + 1);
                __builtin_amdgcn_wave_barrier();
            }
            if (keep) {
                // ascending light index: each entry's rank among the (distinct) entries of the half's list, entries q
                // and q + 32 on a lane at once, four entries of the list per read (padded with one that ranks above all)
                const uint32_t sub = lane & 31u;
                if (sub < 4u && h + sub < VREN_LIST_SLOT) list[h + sub] = 0xFFFFFFFFu;
                __builtin_amdgcn_wave_barrier();
                for (uint32_t q = sub; q < h; q += 64u) {
                    const bool two = q + 32u < h;
                    const uint32_t l0 = list[q], l1 = two ? list[q + 32u] : 0u;
                    uint32_t r0 = 0, r1 = 0;
                    for (uint32_t j = 0; j < h; j += 4u) {
                        const uint4 x = *reinterpret_cast<const uint4*>(list + j);
                        r0 += (x.x < l0 ? 1u : 0u) + (x.y < l0 ? 1u : 0u) + (x.z < l0 ? 1u : 0u) + (x.w < l0 ? 1u : 0u);
                        r1 += (x.x < l1 ? 1u : 0u) + (x.y < l1 ? 1u : 0u) + (x.z < l1 ? 1u : 0u) + (x.w < l1 ? 1u : 0u);
                    }
                    uint32_t* slot = fd.list_slots + (size_t)c * VREN_LIST_SLOT;
                    slot[r0] = l0;
                    if (two) slot[r1] = l1;
                }
            }
            if (live && (lane & 31u) == 0) fd.counts[c] = h;
            __builtin_amdgcn_wave_barrier();
        });
}

// [begin, end) of the index-buffer entries of a tile's light lists, for shade: the tile's clusters are the consecutive
// indices [c0, c0 + u) (clusters kernel) and their lists are consecutive in the index buffer, so the range runs from the
// first cluster's offset to the end of the last list (both clamped to the capacities like the per-pixel lists).
struct TileRanges {
    const uint2* tile_cl;
    uint2* tile_range; // null: no ranges
};

// LISTS: offsets, light lists and tile ranges in one launch. A frame's clusters are cut into `parts` runs, one workgroup
// each, which sums the counts before its run itself (a frame holds a few thousand clusters; a launch of its own for
// their prefix sum took longer) and takes its run 256 clusters at a time: their offsets by a block scan, then their
// lists, which are consecutive in the index buffer, as one range of entries spread over the threads, each finding its
// cluster among the 256 prefixes and copying it from the slot that the counting pass kept.
// A list that has no slot or is longer than one is traversed again (bitmask, emitted in ascending light index) by a
// wave with room for a bitmask, `masks` of a workgroup. The clusters that meet many lights sit together in the image, so
// a run has a `team` of workgroups for them: the first also writes the run's offsets, copies and ranges, the helpers
// traverse their share of the long lists, and leave at once where there are none. One workgroup a run made frames of
// long lists slower than a pass of their own had been; with teams (us, counting, offsets and lists, then | in one pass each |
// one workgroup | team): 1920x1080 with 4096 lights of six times the radius 200 | 209 | 115, 3840x2160 with 65536 of twice
// the radius 508 | 517 | 372, 8192x8192 with 110 k clusters 327 | 438 | 225; a frame without long lists takes what it took
// (640x360 42.6 a frame, 3840x2160 with 65536 lights 563), since a helper leaves as soon as it sees that it has no share.
// 64 frames of 1080p with 4096 lights took 6 + 54 us in two launches, the copies one cluster per wave and step with a
// load's latency each, and take 24; one frame 5 + 4.8, now 6.7; a 3840x2160 frame with 65536 lights 12 + 15, now 16.
constexpr uint32_t kListThreads = 256;
constexpr int kListUnroll = 4; // entries per thread and step (2 is within 1 %)

__device__ __forceinline__ uint32_t list_sum(uint32_t v, uint32_t* s_wave)
{
    const uint32_t w = wave_sum(v);
    if (lane_id() == 0) s_wave[wave_id()] = w;
    __syncthreads();
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t i = 0; i < kListThreads / VREN_WAVE; i++) sum += s_wave[i];
    __syncthreads();
    return sum;
}

__device__ __forceinline__ void assign_lists_body(const FrameDev& fd, uint32_t part, uint32_t parts, uint32_t helper,
                                                  uint32_t team, uint32_t mask_words, uint32_t masks,
                                                  const TileRanges ranges, uint32_t* s_mem)
{
    __shared__ uint32_t s_pre[kListThreads + 1]; // list starts of the 256 clusters, relative to the first one's
    __shared__ uint32_t s_wave[kListThreads / VREN_WAVE];
    __shared__ uint64_t s_long[kListThreads / VREN_WAVE];
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    const uint32_t n = (fd.L == 0 || fd.cluster_count == nullptr) ? 0u : min(*fd.cluster_count, fd.key_cap);
    const uint32_t run_len = (n + parts - 1) / parts;
    const uint32_t begin = min(part * run_len, n), end = min(begin + run_len, n);
    const bool last = part == parts - 1 && helper == 0;
    const auto kept = [&](uint32_t c, uint32_t cnt) {
        return fd.list_slots != nullptr && c < fd.slot_cap && cnt <= VREN_LIST_SLOT;
    };
    if (helper) {
        if (run_len <= helper * masks) return; // the waves before these take every list of a run
        bool any = false;
        for (uint32_t c = begin + tid; c < end; c += kListThreads) any = any || !kept(c, load_at<uint32_t>(fd.counts, c));
        if (!__syncthreads_or(any)) return; // the whole workgroup
    }
    uint32_t sum = 0;
    const uint32_t quads = (reinterpret_cast<uintptr_t>(fd.counts) & 15) == 0 ? begin / 4 : 0u;
#pragma unroll 8
    for (uint32_t i = tid; i < quads; i += kListThreads) {
        const vu4 x = load_at<vu4>(fd.counts, i);
        sum += (x.x + x.y) + (x.z + x.w);
    }
    for (uint32_t i = quads * 4 + tid; i < begin; i += kListThreads) sum += load_at<uint32_t>(fd.counts, i);
    uint32_t run = list_sum(sum, s_wave);

    // first clusters ascend over the frame's tiles, so 256 of them, one per thread, bracket each sub-run's tiles
    const uint32_t tiles = ranges.tile_range && helper == 0 ? fd.Sx * fd.Sy : 0u;
    const uint2* tile_cl = ranges.tile_cl + fd.tile_base;
    const uint32_t step = (tiles + kListThreads - 1) / kListThreads;
    uint32_t sample = 0xFFFFFFFFu;
    if (tiles) {
        if (tid * step < tiles) sample = tile_cl[tid * step].x;
        if (last) // a tile without clusters below the capacity (of a frame without lights, every tile) has an empty range
            for (uint32_t t = tid; t < tiles; t += kListThreads)
                if (!(tile_cl[t].x < n && tile_cl[t].y > 0)) ranges.tile_range[fd.tile_base + t] = make_uint2(0u, 0u);
    }

    bool cleared = false; // this wave's bitmask (which emit_bitmask leaves clear)
    for (uint32_t c0 = begin; c0 < end; c0 += kListThreads) {
        const uint32_t m = min(kListThreads, end - c0), c = c0 + tid;
        const uint32_t cnt = tid < m ? load_at<uint32_t>(fd.counts, c) : 0u;
        uint32_t total;
        const uint32_t ex = block_exclusive_sum<kListThreads>(cnt, s_wave, &total);
        if (tid < m && helper == 0) fd.offsets[c] = run + ex;
        const uint64_t longs = ballot(tid < m && !kept(c, cnt));
        if (lane == 0) s_long[wave] = longs;
        s_pre[tid] = ex;
        if (tid == 0) s_pre[kListThreads] = total;
        __syncthreads();
        const uint32_t copied = helper == 0 ? total : 0u;
        for (uint32_t q0 = 0; q0 < copied; q0 += kListThreads * kListUnroll) { // entries whose searches and loads overlap
            uint32_t at[kListUnroll];
#pragma unroll
            for (int u = 0; u < kListUnroll; u++) at[u] = 0;
#pragma unroll
            for (uint32_t s = kListThreads / 2; s >= 1; s >>= 1)
#pragma unroll
                for (int u = 0; u < kListUnroll; u++) // the last cluster whose list starts at or before the entry
                    if (s_pre[at[u] + s] <= q0 + u * kListThreads + tid) at[u] += s;
            uint32_t li[kListUnroll];
            bool on[kListUnroll];
#pragma unroll
            for (int u = 0; u < kListUnroll; u++) {
                const uint32_t q = q0 + u * kListThreads + tid, i = at[u];
                on[u] = q < total && (uint64_t)run + q < fd.index_cap && !((s_long[i / VREN_WAVE] >> (i % VREN_WAVE)) & 1ull);
                li[u] = on[u] ? fd.list_slots[(size_t)(c0 + i) * VREN_LIST_SLOT + (q - s_pre[i])] : 0u;
            }
#pragma unroll
            for (int u = 0; u < kListUnroll; u++)
                if (on[u]) fd.indices[run + q0 + u * kListThreads + tid] = li[u];
        }
        if (tiles) {
            // tiles [t0, t1): from the last sample below c0 to the first one past the sub-run
            const uint32_t below = list_sum(sample < c0 ? 1u : 0u, s_wave), upto = list_sum(sample < c0 + m ? 1u : 0u, s_wave);
            const uint32_t t0 = below ? (below - 1) * step : 0u, t1 = min(upto * step, tiles);
            for (uint32_t t = t0 + tid; t < t1; t += kListThreads) {
                const uint2 cl = tile_cl[t];
                if (!(cl.y > 0 && cl.x >= c0 && cl.x < c0 + m)) continue;
                const uint32_t stop = (uint32_t)min<uint64_t>((uint64_t)cl.x + cl.y, n), in = min(stop - c0, m);
                uint64_t e = (uint64_t)run + s_pre[in];
                for (uint32_t k = c0 + in; k < stop; k++) e += fd.counts[k]; // clusters past the sub-run
                const uint32_t a = min(run + s_pre[cl.x - c0], fd.index_cap);
                ranges.tile_range[fd.tile_base + t] = make_uint2(a, e > fd.index_cap ? fd.index_cap : (uint32_t)e);
            }
        }
        if (wave < masks) {
            const uint32_t summary_words = (mask_words + 31) / 32;
            uint32_t* stack = s_mem + wave * (kStack + mask_words + summary_words);
            uint32_t* bitmask = stack + kStack;
            uint32_t* summary = bitmask + mask_words;
            uint32_t seen = 0; // long lists of the sub-run so far
            for (uint32_t w = 0; w < kListThreads / VREN_WAVE; w++) {
                for (uint64_t rem = s_long[w]; rem; rem &= rem - 1, seen++) {
                    if (seen % (masks * team) != helper * masks + wave) continue;
                    const uint32_t i = w * VREN_WAVE + (uint32_t)__builtin_ctzll(rem);
                    if (s_pre[i + 1] == s_pre[i]) continue; // an empty list past the slots
                    if (!cleared) {
                        cleared = true;
                        for (uint32_t k = lane; k < mask_words; k += VREN_WAVE) bitmask[k] = 0u;
                        for (uint32_t k = lane; k < summary_words; k += VREN_WAVE) summary[k] = 0u;
                        __builtin_amdgcn_wave_barrier();
                    }
                    const uint32_t out = run + s_pre[i];
                    const Box box = leaf_box(cluster_aabb(fd, fd.keys[c0 + i]));
                    traverse(fd, box, stack, bitmask, summary);
                    __builtin_amdgcn_wave_barrier();
                    // emit set bits in ascending light index, clearing the mask as we go
                    emit_bitmask(bitmask, summary, ((fd.L + 31) / 32 + 31) / 32, fd.indices + out,
                                 out < fd.index_cap ? fd.index_cap - out : 0u);
                    __builtin_amdgcn_wave_barrier();
                }
            }
        }
        run += total;
        __syncthreads(); // s_pre, s_long are rewritten
    }
    if (last && tid == 0) {
        *fd.assigned_total = run;
        if (run > fd.index_cap) atomic_or_agent(fd.flags, VREN_FLAG_INDEX_CAPACITY);
    }
}

// clear: the cluster stage's tickets and statuses, which nothing reads after it, left zero for the chain's next run
__global__ __launch_bounds__(256, 8) void assign_count_kernel(const FrameDev* __restrict__ frames, uint32_t F,
                                                             uint32_t* __restrict__ clear, uint32_t clear_words)
{
    extern __shared__ uint32_t s_mem[];
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < clear_words; i += gridDim.x * 256) clear[i] = 0u;
    assign_count_body<true>(frames, F, s_mem);
}
__global__ __launch_bounds__(256, 8) void assign_count_one_kernel(const FrameDev one)
{
    extern __shared__ uint32_t s_mem[];
    assign_count_body<false>(inline_frame(), 1, s_mem);
}
// grid: the first workgroups of all runs, then the helpers
__global__ __launch_bounds__(kListThreads) void assign_lists_kernel(const FrameDev* __restrict__ frames, uint32_t runs,
                                                                    uint32_t parts, uint32_t team, uint32_t mask_words,
                                                                    uint32_t masks, const TileRanges ranges)
{
    extern __shared__ uint32_t s_mem[];
    const uint32_t helper = blockIdx.x / runs, r = blockIdx.x - helper * runs;
    assign_lists_body(frames[r / parts], r % parts, parts, helper, team, mask_words, masks, ranges, s_mem);
}
__global__ __launch_bounds__(kListThreads) void assign_lists_one_kernel(const FrameDev one, uint32_t parts, uint32_t team,
                                                                        uint32_t mask_words, uint32_t masks)
{
    extern __shared__ uint32_t s_mem[];
    assign_lists_body(*inline_frame(), blockIdx.x % parts, parts, blockIdx.x / parts, team, mask_words, masks,
                      TileRanges{nullptr, nullptr}, s_mem);
}

__global__ void empty_lists_kernel(uint32_t* counts, uint32_t* offsets, uint32_t n, uint32_t* total)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) counts[i] = offsets[i] = 0u;
    if (blockIdx.x == 0 && threadIdx.x == 0) *total = 0u;
}

// enough resident waves per CU (32 by default, the chain shape's choice otherwise) to hide the dependent node loads
// of the traversals
uint32_t persistent_blocks(vren_ctx* ctx, uint32_t wpb, uint32_t waves_per_cu)
{
    const uint32_t wpc = waves_per_cu ? waves_per_cu : 32u;
    return (uint32_t)ctx->num_cus * (wpc / wpb > 0 ? wpc / wpb : 1u);
}

} // namespace

int launch_assign(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w,
                  const FrameDev* one)
{
    if (w.max_L == 0) { // no lists; the next run finds cleared words
        const int st = one ? VREN_OK : launch_chain_init(ctx, s, w);
        chain_mark(w, s, !one);
        chain_mark(w, s, false);
        chain_mark(w, s, false);
        return st;
    }
    // per wave that traverses long lists: a stack, the bitmask and its summary
    const uint32_t mask_words = (w.max_L + 31) / 32;
    const size_t per_mask = (size_t)(kStack + mask_words + (mask_words + 31) / 32) * 4;
    if (per_mask > 150 * 1024) return vren_fail(ctx, VREN_EINVAL, "assign_lights: too many lights for the LDS bitmask");
    const uint32_t masks = (uint32_t)std::min<size_t>(kListThreads / VREN_WAVE, 150 * 1024 / per_mask);
    // per wave, two stacks, leaf lists and hit lists (one per half) and the chunk's boxes
    constexpr size_t count_per_wave = (size_t)2 * (kStackHalf + kLeafList + VREN_LIST_SLOT) * 4 + VREN_WAVE * sizeof(float) * 6;
    static_assert(count_per_wave * 4 <= 160 * 1024 / 8, "assign_count: 8 workgroups of 4 waves must fit a CU's LDS");
    const uint32_t count_blocks = persistent_blocks(ctx, 4, w.assign_wpc);
    // list runs per frame: 2048 over a batch, at most 512 and at least 8 a frame (a 3840x2160 frame with 65536 lights 567 us;
    // 574 with half as many runs, 572 with twice; smaller frames and batches within the spread)
    const uint32_t parts = std::max<uint32_t>(8, std::min<uint32_t>(512, 2048 / F));
    // and up to 4096 workgroups, four a run at most, for the long lists (64 frames of 1920x1080 with 4096 lights of four
    // times the radius: lists 735 us with one a run, 445 with two; short lists take the same with both)
    const uint32_t runs = F * parts, team = std::max<uint32_t>(1, std::min<uint32_t>(4, 4096 / runs));
    if (one) {
        assign_count_one_kernel<<<count_blocks, 4 * VREN_WAVE, count_per_wave * 4, s>>>(*one);
        VREN_LAUNCH_CHECK(ctx);
        assign_lists_one_kernel<<<runs * team, kListThreads, per_mask * masks, s>>>(*one, parts, team, mask_words, masks);
        VREN_LAUNCH_CHECK(ctx);
        return VREN_OK;
    }
    assign_count_kernel<<<count_blocks, 4 * VREN_WAVE, count_per_wave * 4, s>>>(
        d_frames, F, w.tickets, (uint32_t)(chain_work_clear_bytes(w.total_tiles) / 4));
    VREN_LAUNCH_CHECK(ctx);
    chain_mark(w, s);
    chain_mark(w, s, false); // the offsets are written with the lists
    assign_lists_kernel<<<runs * team, kListThreads, per_mask * masks, s>>>(d_frames, runs, parts, team, mask_words, masks,
                                                                            TileRanges{w.tile_cl, w.tile_range});
    VREN_LAUNCH_CHECK(ctx);
    chain_mark(w, s);
    return VREN_OK;
}

extern "C" VREN_EXPORT int vren_assign_lights(vren_ctx* ctx, vren_stream_t stream, uint32_t width, uint32_t height,
                                              const vren_camera* camera, const vren_cluster_cfg* cfg,
                                              const uint32_t* cluster_keys, const uint32_t* cluster_count,
                                              uint32_t key_capacity, const vren_bvh_node* bvh, uint32_t light_count,
                                              const uint32_t* light_codes, const float* view_positions,
                                              uint32_t* light_counts, uint32_t* light_offsets, uint32_t* light_indices,
                                              uint32_t index_capacity, uint32_t* assigned_total)
{
    if (!ctx) return VREN_EINVAL;
    int st = vren_validate_camera(ctx, camera);
    if (!st) st = vren_validate_cfg(ctx, cfg);
    if (st) return st;
    if (width == 0 || height == 0 || width > 8192 || height > 8192)
        return vren_fail(ctx, VREN_EINVAL, "assign_lights: screen must be in [1, 8192]^2");
    if (!cluster_keys || !cluster_count || !light_counts || !light_offsets || !assigned_total || key_capacity == 0)
        return vren_fail(ctx, VREN_EINVAL, "assign_lights: null buffer or zero key capacity");
    if (light_count > 0 && (!bvh || !light_codes || !view_positions || !light_indices || index_capacity == 0))
        return vren_fail(ctx, VREN_EINVAL, "assign_lights: null light buffer or zero index capacity");
    if (light_count > (1u << 20)) return vren_fail(ctx, VREN_EINVAL, "assign_lights: at most 2^20 lights");
    if (ctx->device < 0) return vren_fail(ctx, VREN_EINVAL, "assign_lights: context has no device");
    hipStream_t s = (hipStream_t)stream;
    FrameDev f;
    memset(&f, 0, sizeof(f));
    vren_frame_setup(&f, width, height, camera, cfg);
    f.keys = const_cast<uint32_t*>(cluster_keys);
    f.cluster_count = const_cast<uint32_t*>(cluster_count);
    f.key_cap = key_capacity;
    f.bvh = const_cast<vren_bvh_node*>(bvh);
    f.L = light_count;
    f.codes = const_cast<uint32_t*>(light_codes);
    f.view_pos = const_cast<float*>(view_positions);
    f.bvh_padded = vren_calc_bvh_padded_leaf_count(light_count);
    f.bvh_root = vren_calc_bvh_root_index(light_count);
    f.bvh_levels = vren_calc_bvh_level_count(light_count);
    f.bvh_length = vren_calc_bvh_buffer_length(light_count);
    f.counts = light_counts;
    f.offsets = light_offsets;
    f.indices = light_indices;
    f.index_cap = index_capacity;
    f.assigned_total = assigned_total;
    f.flags = ctx->d_flags;
    if (light_count == 0) {
        // no lights: every list is empty
        empty_lists_kernel<<<std::min<uint32_t>(256, (key_capacity + 255) / 256), 256, 0, s>>>(light_counts, light_offsets,
                                                                                            key_capacity, assigned_total);
        VREN_LAUNCH_CHECK(ctx);
        return VREN_OK;
    }
    // list slots for the first clusters, as a batch has them (without them every list is traversed a second time)
    f.list_slots = ctx->list_slots;
    f.slot_cap = ctx->list_slots ? std::min<uint32_t>(key_capacity, VREN_SLOT_CLUSTERS) : 0u;
    ChainWork w;
    memset(&w, 0, sizeof(w));
    w.max_L = light_count;
    return launch_assign(ctx, s, nullptr, 1, w, &f);
}
