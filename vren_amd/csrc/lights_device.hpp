// lights_device.hpp -- device code of the light stage that more than one kernel uses: the AABB of view-space positions,
// BVH nodes and leaf records, and the body that sorts one chunk of lights (and builds the BVH of a frame of one chunk).
#pragma once

#include "chain.hpp"
#include "radix_device.hpp"
#include "scan_device.hpp"

namespace {

constexpr int kLT = 1024;            // threads of a chunk's workgroup
constexpr int kLWaves = kLT / VREN_WAVE;
constexpr int kLKPT = 4;             // lights per thread of a full chunk
constexpr uint32_t kLChunk = VREN_LIGHT_CHUNK;
static_assert(kLChunk == kLT * kLKPT, "a chunk is what one workgroup sorts");
// every third bit of the result holds one of the low 10 bits of q
__device__ __forceinline__ uint32_t spread3(uint32_t q)
{
    q = (q | (q << 16)) & 0x030000FFu;
    q = (q | (q << 8)) & 0x0300F00Fu;
    q = (q | (q << 4)) & 0x030C30C3u;
    return (q | (q << 2)) & 0x09249249u;
}

// bits <= 10 per axis: x at bit 3 i, y at 3 i + 1, z at 3 i + 2 (what lies above an axis' bits is dropped)
__device__ __forceinline__ uint32_t morton_interleave(uint32_t qx, uint32_t qy, uint32_t qz, uint32_t bits)
{
    const uint32_t m = (1u << bits) - 1u;
    return spread3(qx & m) | (spread3(qy & m) << 1) | (spread3(qz & m) << 2);
}

// floats as integers of the same order (-0 below +0), so that min and max of any number of them are integer minima
__device__ __forceinline__ uint32_t ordered_bits(float x)
{
    const uint32_t u = __float_as_uint(x);
    return u ^ ((u >> 31) ? 0xFFFFFFFFu : 0x80000000u);
}
__device__ __forceinline__ float from_ordered(uint32_t o) { return __uint_as_float(o ^ ((o >> 31) ? 0x80000000u : 0xFFFFFFFFu)); }

// The AABB of view-space positions as six minima: ordered_bits of the three lower corners, and the complements of
// the three upper ones'. A NaN coordinate widens neither corner. Start: the reduce identities +-1e35.
struct BoxKeys {
    uint32_t k[6];
};
__device__ __forceinline__ BoxKeys empty_box()
{
    BoxKeys b;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        b.k[a] = ordered_bits(1e35f);
        b.k[3 + a] = ~ordered_bits(-1e35f);
    }
    return b;
}
__device__ __forceinline__ void add_to_box(BoxKeys& b, const float r[3])
{
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const uint32_t o = ordered_bits(r[a]);
        const bool num = r[a] == r[a];
        b.k[a] = min(b.k[a], num ? o : 0xFFFFFFFFu);
        b.k[3 + a] = min(b.k[3 + a], num ? ~o : 0xFFFFFFFFu);
    }
}

// minimum over each row of 16 lanes, in every lane of the row
__device__ __forceinline__ uint32_t row_min(uint32_t v)
{
    v = min(v, dpp0<0xB1, 0xF>(v));    // quad_perm [1,0,3,2]
    v = min(v, dpp0<0x4E, 0xF>(v));    // quad_perm [2,3,0,1]
    v = min(v, dpp0<0x141, 0xF>(v));   // row_half_mirror
    return min(v, dpp0<0x140, 0xF>(v)); // row_mirror
}

// The box of a whole workgroup of kLWaves waves, in every thread: the waves' minima meet in LDS, and every wave reads
// them all and reduces them by rows of 16 lanes (one barrier). s_red: 6 * 16 words.
__device__ __forceinline__ void block_box(BoxKeys& b, uint32_t* s_red)
{
    static_assert(kLWaves == 16, "a row of lanes holds one minimum per wave");
    const uint32_t lane = lane_id(), wave = wave_id();
#pragma unroll
    for (int a = 0; a < 6; a++) {
        const uint32_t m = wave_min_u32(b.k[a]);
        if (lane == 0) s_red[a * kLWaves + wave] = m;
    }
    __syncthreads();
    const uint32_t p = row_min(s_red[lane]), q = row_min(s_red[64 + (lane & 31)]);
    b.k[0] = __builtin_amdgcn_readlane(p, 0);
    b.k[1] = __builtin_amdgcn_readlane(p, 16);
    b.k[2] = __builtin_amdgcn_readlane(p, 32);
    b.k[3] = __builtin_amdgcn_readlane(p, 48);
    b.k[4] = __builtin_amdgcn_readlane(q, 0);
    b.k[5] = __builtin_amdgcn_readlane(q, 16);
}

// 32-lane AABB of the half-wave's leaves or nodes, in its last lane (31 or 63). Lanes without a box pass the empty
// one (min = +inf, max = -inf). The hardware's minimum and maximum order -0 below +0, so any order gives the same bits.
// Written out because the compiler puts a canonicalising maximum between every move and minimum (90 instructions for
// these 30): four steps within the rows of 16 lanes, then lane 15 of each even row into the odd row after it. Steps of one
// value are six instructions apart, which covers the two wait states from a write to a DPP read.
#define VREN_BOX_STEP(ctrl)                                                                                            \
    "v_min_f32_dpp %0, %0, %0 " ctrl " bank_mask:0xf\n\t"                                                             \
    "v_min_f32_dpp %1, %1, %1 " ctrl " bank_mask:0xf\n\t"                                                             \
    "v_min_f32_dpp %2, %2, %2 " ctrl " bank_mask:0xf\n\t"                                                             \
    "v_max_f32_dpp %3, %3, %3 " ctrl " bank_mask:0xf\n\t"                                                             \
    "v_max_f32_dpp %4, %4, %4 " ctrl " bank_mask:0xf\n\t"                                                             \
    "v_max_f32_dpp %5, %5, %5 " ctrl " bank_mask:0xf\n\t"
__device__ __forceinline__ void half_wave_box(float (&mn)[3], float (&mx)[3])
{
    asm("s_nop 1\n\t"
        VREN_BOX_STEP("quad_perm:[1,0,3,2] row_mask:0xf")
        VREN_BOX_STEP("quad_perm:[2,3,0,1] row_mask:0xf")
        VREN_BOX_STEP("row_half_mirror row_mask:0xf")
        VREN_BOX_STEP("row_mirror row_mask:0xf")
        VREN_BOX_STEP("row_bcast:15 row_mask:0xa")
        : "+v"(mn[0]), "+v"(mn[1]), "+v"(mn[2]), "+v"(mx[0]), "+v"(mx[1]), "+v"(mx[2]));
}

// f2u_sat(floor(t)): the hardware's conversion truncates, takes negative numbers and NaN to 0 and saturates
__device__ __forceinline__ uint32_t floor_u32_sat(float t)
{
    uint32_t q;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(q) : "v"(t));
    return q;
}

__device__ __forceinline__ void store_node(vren_bvh_node* n, const float (&mn)[3], const float (&mx)[3], uint32_t next)
{
    float4* q = reinterpret_cast<float4*>(n);
    q[0] = make_float4(mn[0], mn[1], mn[2], __uint_as_float(next));
    q[1] = make_float4(mx[0], mx[1], mx[2], 0.0f);
}

__device__ __forceinline__ void store_invalid(vren_bvh_node* n)
{
    const float inf[3] = {VREN_F32_INF, VREN_F32_INF, VREN_F32_INF};
    const float ninf[3] = {-VREN_F32_INF, -VREN_F32_INF, -VREN_F32_INF};
    store_node(n, inf, ninf, VREN_BVH_INVALID_NODE);
}

// The smallest squared distance (a non-negative float) whose square root is not below r, so that sqrt(d2) < r is
// d2 < limit for every float d2; 0, which nothing is below, for a radius that is not positive. A correctly rounded
// square root reaches r from the square of the midpoint m between r and the float below it on (m * m has an odd bit
// past a float's, so none rounds to even there), and with u the distance of the two, m * m = r * r - r * u + u * u / 4,
// of which the first two are exact in double and a multiple of u * u, as every float there is: the limit is the first
// float above r * r - r * u. (Checked against the square root for radii of every magnitude.)
__device__ __forceinline__ float leaf_limit(float r)
{
    const double u = (double)(r - __uint_as_float(__float_as_uint(r) - 1u));
    const double d = (double)r * (double)r - (double)r * u;
    const float t = (float)d;
    const float up = __uint_as_float(__float_as_uint(t) + 1u);
    const float limit = (double)t > d ? t : up;
    return r > 0.0f ? (r < VREN_F32_INF ? limit : r) : 0.0f;
}

// the leaf record of a leaf box (clustered.hpp): the radius as the traversal takes it from the box
// (assign_lights.comp:214)
__device__ __forceinline__ float4 leaf_record(float x, float y, float z, float min_x, float max_x)
{
    return make_float4(x, y, z, leaf_limit((max_x - min_x) / 2.0f));
}

// the frame and the chunk of a flattened chunk number
__device__ __forceinline__ const FrameDev& frame_of_chunk(const FrameDev* __restrict__ frames, uint32_t F, uint32_t c,
                                                          uint32_t* chunk)
{
    const uint32_t f = F > 1 ? find_frame_wave(frames, F, c, [](const FrameDev& d) { return d.light_chunk_base; }) : 0u;
    *chunk = c - frames[f].light_chunk_base;
    return frames[f];
}

// One chunk: its lights' Morton codes, sorted stably with the light indices by an LSD radix sort on BITS-bit digits
// (8 by default; 4 is a chain-shape choice), as few keys per thread as the chunk needs, so that a small frame's keys are
// spread over all the waves (block_sort). Blocks at and past `chunks` write the frame's padding leaves (single-frame calls).
// A frame of one chunk then builds its BVH from the sorted lights: leaves, the first parent level over half-waves, the
// rest from LDS. 4096 lights and their BVH took 34 us in three launches (21.7 + 6 + 6.8) and take one of 21 us
// (256 lights: 21 -> 7 us), bound by the vector issue of its one CU; 65 536 lights took 292 us in one workgroup that
// sorted in global memory and take 36 us (bounds 6, chunks 12.5, merge 17).
template <int BITS>
__device__ __forceinline__ void lights_body(const FrameDev* __restrict__ frames, uint32_t F, uint32_t chunks)
{
    __shared__ uint2 s_pair[kLChunk];              // (code, light index)
    __shared__ float4 s_light[kLChunk];            // view position, radius (frames of one chunk)
    __shared__ BlockSortLds<BITS, kLWaves> s_sort;
    __shared__ uint32_t s_red[6 * kLWaves];
    __shared__ float s_node[kLChunk / 32][6];      // the first parent level, then the second one
    __shared__ float s_node2[kLChunk / 1024][6];

    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    if (blockIdx.x >= chunks) {
        const FrameDev& fd = frames[0];
        const uint32_t i = (blockIdx.x - chunks) * kLT + tid, padded = fd.bvh_padded;
        if (i < ((fd.L + 31u) & ~31u) || i >= padded) return;
        store_invalid(&fd.bvh[i]);
        if ((i & 31u) == 0) store_invalid(&fd.bvh[padded + i / 32]);
        return;
    }
    uint32_t chunk;
    const FrameDev& fd = frame_of_chunk(frames, F, blockIdx.x, &chunk);
    const uint32_t L = fd.L, first = chunk * kLChunk;
    const bool whole = L <= kLChunk; // the frame is this chunk
    const uint32_t n = min(kLChunk, L - first);
    const uint32_t kpt = (n + kLT - 1) / kLT;
    const uint32_t wbase = wave * kpt * VREN_WAVE;

    // view positions and the frame's box (reduce_vec4 min/max of clustered_shading.cpp:137-191)
    float r[kLKPT][3];
    BoxKeys box = empty_box();
#pragma unroll
    for (int j = 0; j < kLKPT; j++) {
        const uint32_t i = wbase + j * VREN_WAVE + lane;
        if (j < (int)kpt && i < n) {
            float q[4];
            if (whole) {
                const vf4 p = *((gvf4*)fd.light_pos + i);
                const float radius = *((gfloat*)fd.lights + 4 * i + 3);
                const float v[4] = {p.x, p.y, p.z, 1.0f};
                vren_mat4_mul_vec4(fd.view, v, q);
                reinterpret_cast<float4*>(fd.view_pos)[i] = make_float4(q[0], q[1], q[2], q[3]);
                s_light[i] = make_float4(q[0], q[1], q[2], radius);
                add_to_box(box, q);
            } else {
                const vf4 p = *((gvf4*)fd.view_pos + first + i);
                q[0] = p.x;
                q[1] = p.y;
                q[2] = p.z;
            }
#pragma unroll
            for (int a = 0; a < 3; a++) r[j][a] = q[a];
        }
    }
    float lo[3], hi[3];
    if (fd.morton_aabb_mode == VREN_MORTON_GIVEN_AABB) {
        for (int a = 0; a < 3; a++) {
            lo[a] = fd.morton_min[a];
            hi[a] = fd.morton_max[a];
        }
    } else {
        if (whole) {
            block_box(box, s_red);
        } else {
            const uint32_t n_chunks = (L + kLChunk - 1) / kLChunk;
            for (uint32_t c = lane; c < n_chunks; c += VREN_WAVE)
#pragma unroll
                for (int a = 0; a < 6; a++) box.k[a] = min(box.k[a], *((guint*)fd.chunk_box + c * 6 + a));
#pragma unroll
            for (int a = 0; a < 6; a++) box.k[a] = wave_min_u32(box.k[a]);
        }
        for (int a = 0; a < 3; a++) {
            lo[a] = from_ordered(box.k[a]);
            hi[a] = from_ordered(~box.k[3 + a]);
        }
    }

    // Morton codes (discretize_point_light_positions.comp:26-43), paired with the light index
    const uint32_t bits = fd.morton_bits, total_bits = 3 * bits;
    const float scale = (float)(1u << bits);
    // The quotients (r - lo) / (hi - lo) by one correctly rounded reciprocal per axis and two fused steps (vmath.h), if every
    // light of the wave is inside the box on every axis, as all are in the lights' own box; a given box takes the
    // division where one is not.
    float ext[3], rec[3];
    bool inside = true;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        ext[a] = hi[a] - lo[a];
        rec[a] = 1.0f / ext[a];
        inside = inside && vren_unit_quotient_extent(ext[a]);
    }
#pragma unroll
    for (int j = 0; j < kLKPT; j++)
        if (j < (int)kpt && wbase + j * VREN_WAVE + lane < n)
#pragma unroll
            for (int a = 0; a < 3; a++) {
                r[j][a] = r[j][a] - lo[a];
                inside = inside && __builtin_fabsf(r[j][a]) <= ext[a];
            }
    const bool fused = ballot(!inside) == 0;
    uint2 e[kLKPT];
#pragma unroll
    for (int j = 0; j < kLKPT; j++) {
        const uint32_t i = wbase + j * VREN_WAVE + lane;
        e[j] = make_uint2(0u, 0u);
        if (j < (int)kpt && i < n) {
            uint32_t q[3];
#pragma unroll
            for (int a = 0; a < 3; a++) {
                float t;
                if (fused) t = vren_unit_quotient(r[j][a], ext[a], rec[a]); // uniform
                else t = r[j][a] / ext[a];
                q[a] = floor_u32_sat(t * scale);
            }
            e[j] = make_uint2(morton_interleave(q[0], q[1], q[2], bits), first + i);
        }
    }

    // the stable sort by code (ties keep light-index order)
    block_sort<BITS, kLKPT, kLWaves>(e, kpt, n, 0, total_bits, s_pair, s_sort, [](const uint2& x) { return x.x; });
    uint2* out = reinterpret_cast<uint2*>(whole ? fd.codes : fd.codes_tmp) + first;
    if (!whole) {
        for (uint32_t i = tid; i < n; i += kLT) out[i] = s_pair[i];
        return;
    }

    // leaves (init_light_array_bvh.comp:42-65) in light-holding groups of 32, and their parents
    const uint32_t padded = fd.bvh_padded;
    const uint32_t groups = (n + 31) / 32;
#pragma unroll
    for (int k = 0; k < kLKPT; k++) {
        const uint32_t i = k * kLT + tid;
        if (i >= groups * 32) break; // whole half-waves leave together; the others' lanes do not read them
        float mn[3] = {VREN_F32_INF, VREN_F32_INF, VREN_F32_INF};
        float mx[3] = {-VREN_F32_INF, -VREN_F32_INF, -VREN_F32_INF};
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < n) {
            const uint2 pr = s_pair[i];
            v = s_light[pr.y];
            out[i] = pr;
            mn[0] = v.x - v.w;
            mn[1] = v.y - v.w;
            mn[2] = v.z - v.w;
            mx[0] = v.x + v.w;
            mx[1] = v.y + v.w;
            mx[2] = v.z + v.w;
        }
        if (fd.leaf_rec)
            reinterpret_cast<float4*>(fd.leaf_rec)[i] = i < n ? leaf_record(v.x, v.y, v.z, mn[0], mx[0])
                                                               : make_float4(0.f, 0.f, 0.f, 0.f);
        store_node(&fd.bvh[i], mn, mx, i < n ? VREN_BVH_LEAF_NODE : VREN_BVH_INVALID_NODE);
        half_wave_box(mn, mx);
        if ((lane & 31) == 31) {
            const uint32_t g = i / 32;
            store_node(&fd.bvh[padded + g], mn, mx, g * 32);
            for (int a = 0; a < 3; a++) {
                s_node[g][a] = mn[a];
                s_node[g][3 + a] = mx[a];
            }
        }
    }
    if (padded < 1024) return; // 32 leaves: the first parent is the root
    __syncthreads();
    // second parent level: padded / 1024 nodes, the first n2 of them over first-level nodes that hold lights
    const uint32_t level1 = padded, level2 = level1 + padded / 32, size2 = padded / 1024;
    const uint32_t n2 = (groups + 31) / 32;
    if (tid < n2 * 32) {
        float mn[3] = {VREN_F32_INF, VREN_F32_INF, VREN_F32_INF};
        float mx[3] = {-VREN_F32_INF, -VREN_F32_INF, -VREN_F32_INF};
        if (tid < groups) {
            for (int a = 0; a < 3; a++) {
                mn[a] = s_node[tid][a];
                mx[a] = s_node[tid][3 + a];
            }
        }
        half_wave_box(mn, mx);
        if ((lane & 31) == 31) {
            const uint32_t g = tid / 32;
            store_node(&fd.bvh[level2 + g], mn, mx, level1 + g * 32);
            for (int a = 0; a < 3; a++) {
                s_node2[g][a] = mn[a];
                s_node2[g][3 + a] = mx[a];
            }
        }
    }
    if (tid >= n2 && tid < size2) store_invalid(&fd.bvh[level2 + tid]);
    if (size2 == 1) return; // 1024 leaves: that was the root
    __syncthreads();
    if (tid < 32) { // the root over the 32 second-level nodes of 32768 leaves
        float mn[3] = {VREN_F32_INF, VREN_F32_INF, VREN_F32_INF};
        float mx[3] = {-VREN_F32_INF, -VREN_F32_INF, -VREN_F32_INF};
        if (tid < n2) {
            for (int a = 0; a < 3; a++) {
                mn[a] = s_node2[tid][a];
                mx[a] = s_node2[tid][3 + a];
            }
        }
        half_wave_box(mn, mx);
        if (tid == 31) store_node(&fd.bvh[level2 + 32], mn, mx, level2);
    }
}

} // namespace
