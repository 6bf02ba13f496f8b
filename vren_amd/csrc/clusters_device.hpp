// clusters_device.hpp -- device code of the cluster stage that more than one kernel uses: a pixel's cluster key and the body
// that finds the unique keys of a group of tiles.
#pragma once

#include "chain.hpp"
#include "scan_device.hpp"

namespace {

// The dominant axis of a normal: the reference picks the smallest t_i = sign(n_i) / n_i (first index on ties;
// a zero component gives NaN and is never picked), clustered_shading.glsl:7-43. The components are f16 values
// converted exactly, so distinct magnitudes differ by at least 2^-11 relative and their float reciprocals keep
// the reverse order: the smallest t_i is the largest |n_i| (first index on ties), found without dividing.
// Returns the axis, or 3 when no component qualifies (the reference then keeps t = 1e35 and axis 0).
__device__ __forceinline__ uint32_t dominant_axis(const float n[3])
{
    uint32_t axis = 3;
    float best = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < 3; i++) {
        const float a = fabsf(n[i]);
        if (a > best) {
            best = a;
            axis = i;
        }
    }
    return axis;
}

// 1 / a, correctly rounded, for a > 0 an f16 value widened to float: v_rcp_f32 (within 1 ulp) and one FMA Newton
// step. A divisor with an 11-bit significand keeps 1 / a at least 2^-36 (relative) away from every rounding
// boundary of float, far beyond the step's ~2^-46 error; the CPU tests check every finite f16 divisor against
// every reciprocal within 1 ulp. a = +inf gives +0, as the division does (the Newton step would give NaN).
__device__ __forceinline__ float rcp_f16_exact(float a)
{
    const float y = __builtin_amdgcn_rcpf(a);
    const float r = __builtin_fmaf(y, __builtin_fmaf(-a, y, 1.0f), y);
    return a < __builtin_inff() ? r : 0.0f;
}

__device__ __forceinline__ uint32_t discretize_normal(const float n[3])
{
    // clustered_shading.glsl:7-43
    if (n[0] == 0.0f && n[1] == 0.0f && n[2] == 0.0f) return 0xFFFFFFFFu;
    const uint32_t ax = dominant_axis(n);
    float min_t = 1e35f;
    uint32_t axis = 0, face_idx = 0;
    if (ax < 3) {
        axis = ax;
        // sign(n) / n = 1 / |n|, |n[ax]| > 0 being the largest magnitude (finite or +inf)
        min_t = rcp_f16_exact(fabsf(n[ax]));
        face_idx = (n[ax] > 0.0f ? 1u : 0u) * 3u + ax;
    }
    float p[3] = {n[0] * min_t, n[1] * min_t, n[2] * min_t};
    float u = p[(axis + 1) % 3];
    float v = p[(axis + 2) % 3];
    uint32_t du = vren_third_index(u);
    uint32_t dv = vren_third_index(v);
    return (face_idx * 9u + du * 3u + dv) & 0x3Fu;
}

__device__ __forceinline__ uint32_t face_of_normal(const float n[3])
{
    if (n[0] == 0.0f && n[1] == 0.0f && n[2] == 0.0f) return 7u;
    const uint32_t ax = dominant_axis(n);
    return ax < 3 ? (n[ax] > 0.0f ? 1u : 0u) * 3u + ax : 0u;
}

// f16 -> f32 on the conversion unit. A key depends on a NaN component only through comparisons and through
// f2u_sat(floor(NaN)) = 0, never on its payload, so the conversion's NaN payload need not be the oracle's.
__device__ __forceinline__ float key_h2f(uint32_t h)
{
    const uint16_t b = (uint16_t)h;
    _Float16 x;
    __builtin_memcpy(&x, &b, 2);
    return (float)x;
}

// the conversion as the hardware does it: a negative value and a NaN give 0
__device__ __forceinline__ uint32_t cvt_u32(float x)
{
    uint32_t r;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// The code of a normal (the face alone in sliced mode) without branches: right where the function returns true, for a zero
// normal (the background of a cleared G-buffer) and wherever the largest magnitude is positive and finite; not for
// infinities and for zeros with NaNs. The maximum drops NaNs, and no NaN equals it. The cell of u in [-1, 1] is
// the truncation of 1.5 (u + 1), the reference's (u + 1) / 2 * 3 with its exact halving folded in.
__device__ __forceinline__ bool normal_code(bool sliced, uint2 nb, uint32_t* code)
{
    const float n0 = key_h2f(nb.x & 0xFFFFu), n1 = key_h2f(nb.x >> 16), n2 = key_h2f(nb.y & 0xFFFFu);
    const bool zero = ((nb.x & 0x7FFF7FFFu) | (nb.y & 0x7FFFu)) == 0u;
    const float m = fmaxf(fmaxf(fabsf(n0), fabsf(n1)), fabsf(n2));
    const bool x = fabsf(n0) == m, y = fabsf(n1) == m;
    float d = y ? n1 : n2;
    d = x ? n0 : d;
    if (sliced) {
        *code = zero ? 7u : (x ? 0u : (y ? 1u : 2u)) + (d > 0.0f ? 3u : 0u);
    } else {
        const float rcp = __builtin_amdgcn_rcpf(m), t = __builtin_fmaf(rcp, __builtin_fmaf(-m, rcp, 1.0f), rcp);
        float u = y ? n2 : n0, v = y ? n0 : n1;
        u = x ? n1 : u;
        v = x ? n2 : v;
        const uint32_t du = cvt_u32((u * t + 1.0f) * 1.5f), dv = cvt_u32((v * t + 1.0f) * 1.5f);
        *code = zero ? 0x3Fu : (x ? 0u : (y ? 9u : 18u)) + (d > 0.0f ? 27u : 0u) + (du * 3u + dv);
    }
    return zero || __builtin_amdgcn_classf(m, 0x100); // a positive normal number
}

// The depth slice of a view depth z by the reference's formula (find_unique_clusters.comp:58-62): log mode
// f2u_sat(floor(log(z / near) / log_a)) before the 10-bit mask, sliced mode the same over [near, far] in
// depth_slices steps, clamped to the last slice. A non-positive or NaN z gives 0 (log of a non-positive ratio is
// NaN or -inf, which f2u_sat maps to 0).
__device__ __forceinline__ uint32_t slice_exact(const FrameDev& fd, float z)
{
    if (fd.key_mode == VREN_KEYS_SLICED) {
        uint32_t k = vren_f2u_sat(vren_floorf(vren_logf(z / fd.near_plane) / fd.log_fn * (float)fd.depth_slices));
        return k >= fd.depth_slices ? fd.depth_slices - 1 : k;
    }
    return vren_f2u_sat(vren_floorf(vren_logf(z / fd.near_plane) / fd.log_a));
}

// A pixel's view depth (find_unique_clusters.comp:48-56) as the numerator r[0] and the denominator r[1] of the division
// that gives it.
__device__ __forceinline__ void pixel_view_zw(const FrameDev& fd, uint32_t gx, uint32_t gy, float depth, float r[2])
{
    if (fd.proj_zw_xy_zero) {
        // the z and w rows of inverse(P) have zero x and y coefficients: ((0 x + 0 y) + m2 depth) + m3 reduces to
        // m2 depth + m3 exactly (a zero result may only change sign, and z = 0 gives the same slice either way)
        r[0] = fd.inv_proj[2 * 4 + 2] * depth + fd.inv_proj[3 * 4 + 2];
        r[1] = fd.inv_proj[2 * 4 + 3] * depth + fd.inv_proj[3 * 4 + 3];
    } else {
        float v[4] = {(float)gx / (float)fd.W, (float)gy / (float)fd.H, depth, 1.0f};
        v[1] = 1.0f - v[1];
        v[0] = v[0] * 2.0f - 1.0f;
        v[1] = v[1] * 2.0f - 1.0f;
        float o[4];
        vren_mat4_mul_vec4(fd.inv_proj, v, o);
        r[0] = o[2];
        r[1] = o[3];
    }
}

// The slice of nearly every pixel without a division, a logarithm's polynomial or a table: the floor of
// log2(z) slice_c1 + slice_c0 with the hardware's reciprocal and logarithm, certain where that value is farther from a
// whole number than the two formulas can lie apart and z is not far outside the planes (FrameDev's slice_*). What is not
// certain (a few pixels in ten thousand, and any depth whose z is not a positive number) takes slice_exact.
// Values below 0.5 are in slice 0, with everything in front of the near plane. With the branch-free normal code and the rows'
// wide loads the cluster stage of 64 1920x1080 frames went from 580 us (an IEEE division, a search in a table of
// thresholds in LDS and a branch per case of the normal) to 516, 16 frames with sliced keys from 218 to 139 (their
// background, at the end of the last slice, took the formula), a 1366x769 frame from 23 and 8 for its table to 17.
// What is left is mostly memory: 2.1 GB for the 64 frames, 452 us at the rate of a large copy.
__device__ __forceinline__ bool slice_estimate(const FrameDev& fd, const float zw[2], uint32_t* k)
{
    const float lg = __builtin_amdgcn_logf(zw[0] * __builtin_amdgcn_rcpf(zw[1]));
    const float e = __builtin_amdgcn_fmed3f(__builtin_fmaf(lg, fd.slice_c1, fd.slice_c0), 0.5f, fd.slice_max);
    *k = (uint32_t)e;
    return fabsf(lg) <= fd.slice_reach && fabsf(__builtin_amdgcn_fractf(e) - 0.5f) < fd.slice_safe;
}

// the high half of a cluster key, from its slice and normal (find_unique_clusters.comp:58-65); the low half are the
// tile's ids
__device__ __forceinline__ uint32_t key_high(const FrameDev& fd, uint32_t k, uint32_t code)
{
    return fd.key_mode == VREN_KEYS_SLICED ? (k & 0xFFu) | (code << 8) : (k & 0x3FFu) | (code << 10);
}

constexpr uint32_t kClusterWaves = 8;   // waves per workgroup, one 32x32 tile per wave (16 measured slower)

// 16 bytes at a 4-byte boundary: one load or store, whatever the row's alignment
typedef float vf4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t vu4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef const __attribute__((address_space(1))) vf4_a4 gvf4_a4;
typedef const __attribute__((address_space(1))) vu4_a4 gvu4_a4;

// the reference's REPEAT sampler: (x mod W, y mod H)
__device__ __forceinline__ void wrap_pixel(const FrameDev& fd, uint32_t& x, uint32_t& y)
{
    if (x >= fd.W) x %= fd.W;
    if (y >= fd.H) y %= fd.H;
}

// The depths and normals of lane `lane` of N / 4 of a tile's four 8-row groups, from group j0 on (pixels i = 4 j + q, stored
// at [4 (j - j0) + q]): pixel (x0 + q, tj * 32 + 8 j + lane / 8). A tile inside the frame (uniform across the wave) takes
// one 16-byte depth load and two 16-byte normal loads per row; other tiles load per pixel, wrapped. Every load is issued
// before any is used.
template <int N>
__device__ __forceinline__ void load_tile(const FrameDev& fd, uint32_t ti, uint32_t tj, uint32_t lane, uint32_t j0,
                                          float dep[N], uint2 nrm[N])
{
    const uint32_t x0 = ti * 32 + (lane & 7) * 4;
    if ((ti + 1) * 32 <= fd.W && (tj + 1) * 32 <= fd.H) {
#pragma unroll
        for (int jj = 0; jj < N / 4; jj++) {
            const uint64_t p0 = (uint64_t)(tj * 32 + (j0 + jj) * 8 + (lane >> 3)) * fd.W + x0;
            const vf4_a4 d4 = *(gvf4_a4*)(fd.depth + p0);
            const vu4_a4 n01 = *(gvu4_a4*)(fd.normals + 4 * p0);
            const vu4_a4 n23 = *(gvu4_a4*)(fd.normals + 4 * p0 + 8);
            dep[4 * jj + 0] = d4.x;
            dep[4 * jj + 1] = d4.y;
            dep[4 * jj + 2] = d4.z;
            dep[4 * jj + 3] = d4.w;
            nrm[4 * jj + 0] = make_uint2(n01.x, n01.y);
            nrm[4 * jj + 1] = make_uint2(n01.z, n01.w);
            nrm[4 * jj + 2] = make_uint2(n23.x, n23.y);
            nrm[4 * jj + 3] = make_uint2(n23.z, n23.w);
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; i++) {
            uint32_t x = x0 + (i & 3), y = tj * 32 + (j0 + (i >> 2)) * 8 + (lane >> 3);
            wrap_pixel(fd, x, y);
            const uint64_t p = (uint64_t)y * fd.W + x;
            dep[i] = *(gfloat*)(fd.depth + p);
            const vu2 n = *(gvu2*)(fd.normals + 4 * p);
            nrm[i] = make_uint2(n.x, n.y);
        }
    }
}

// Tiles are flattened over every frame of the table (tile_base, a multiple of VREN_TILE_GROUP). A workgroup takes
// ONE ticket for a group of kClusterWaves consecutive tiles of one frame, one per wave -- a ticket on a single
// counter costs ~11 ns of serialised atomic throughput, so one per tile would cap the kernel at ~90 M tiles/s.
// The group's unique counts are summed in LDS and chained to the frame's previous groups by one decoupled
// look-back per workgroup (per tile, the walk's round trips of ~1.4 us covered 64 tiles each and could not keep up
// with the tiles finishing). The walk waits only on groups of lower tickets, whose workgroups are already running,
// so every wait ends. Lane l owns the pixels (4 (l % 8) + q, 8 j + l / 8), q, j = 0..3, of its tile.
// DEEP: a tile's loads are all in flight at once (48 registers of them); otherwise its two halves are loaded one after
// the other, which keeps the register peak of a wave below 64 (eight waves per SIMD).
template <bool DEEP>
__device__ __forceinline__ void clusters_body(const FrameDev* __restrict__ frames,
                                              const uint32_t* __restrict__ tile_frame, uint32_t total_tiles,
                                              uint64_t* tile_status, uint32_t* ticket, uint2* __restrict__ tile_cl)
{
    static_assert(kClusterWaves == VREN_TILE_GROUP, "one workgroup per tile group");
    __shared__ uint32_t s_unique[kClusterWaves][1024];
    __shared__ uint32_t s_u[kClusterWaves];
    __shared__ uint32_t s_t, s_prefix;
    const uint32_t lane = lane_id();
    const uint32_t wave = wave_id();
    if (threadIdx.x == 0) s_t = atomic_add_agent(ticket, 1u);
    __syncthreads();
    const uint32_t g0 = s_t * kClusterWaves;
    if (g0 >= total_tiles) return; // the whole workgroup
    // a workgroup's tiles are one group of its frame (frame tile ranges start at multiples of VREN_TILE_GROUP)
    const FrameDev& fd = frames[frame_of_tile(tile_frame, g0)];
    uint32_t* uq = s_unique[wave];
    const uint32_t g = g0 + wave;
    const uint32_t t0 = g0 - fd.tile_base; // the group's first tile in its frame
    const uint32_t t = t0 + wave;
    const uint32_t tiles = fd.Sx * fd.Sy;
    const bool live = g < total_tiles && t < tiles; // not past the table nor on a frame's padding
    const uint32_t ti = t % fd.Sx, tj = t / fd.Sx;
    const uint32_t x0 = ti * 32 + (lane & 7) * 4;
    uint32_t key[16];
    uint32_t u = 0;
    if (live) {
        constexpr int N = DEEP ? 16 : 8;
        const bool sliced = fd.key_mode == VREN_KEYS_SLICED;
        uint32_t pend = 0u;
#pragma unroll
        for (uint32_t h = 0; h < 16 / N; h++) {
            float dep[N];
            uint2 nrm[N];
            load_tile<N>(fd, ti, tj, lane, h * (N / 4), dep, nrm);
#pragma unroll
            for (int r = 0; r < N; r++) {
                const int i = N * h + r;
                float zw[2];
                uint32_t k, code;
                pixel_view_zw(fd, x0 + (i & 3), tj * 32 + (i >> 2) * 8 + (lane >> 3), dep[r], zw);
                const bool slice_ok = slice_estimate(fd, zw, &k), code_ok = normal_code(sliced, nrm[r], &code);
                key[i] = key_high(fd, k, code);
                pend |= slice_ok && code_ok ? 0u : 1u << i;
                // a pixel's key and flag are finished before the next pixel's: their temporaries together would not fit
                asm volatile("" : "+v"(key[i]), "+v"(pend));
            }
            // the second half's loads stay after the first half's keys (the register peak of one half)
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
        }
        // the other pixels by the reference's formulas, one of each lane at a time, read again
        while (ballot(pend != 0u)) {
            if (pend) {
                const uint32_t i = (uint32_t)__builtin_ctz(pend);
                const uint32_t x = x0 + (i & 3), y = tj * 32 + (i >> 2) * 8 + (lane >> 3);
                uint32_t wx = x, wy = y;
                wrap_pixel(fd, wx, wy);
                const uint64_t p = (uint64_t)wy * fd.W + wx;
                float zw[2];
                pixel_view_zw(fd, x, y, *((gfloat*)fd.depth + p), zw);
                const vu2 nb = *(gvu2*)(fd.normals + 4 * p);
                const float n[3] = {key_h2f(nb.x & 0xFFFFu), key_h2f(nb.x >> 16), key_h2f(nb.y & 0xFFFFu)};
                const uint32_t code = sliced ? face_of_normal(n) : discretize_normal(n) & 0x3Fu;
                const uint32_t exact = key_high(fd, slice_exact(fd, zw[0] / zw[1]), code);
#pragma unroll
                for (uint32_t q = 0; q < 16; q++) key[q] = q == i ? exact : key[q];
                pend &= pend - 1u;
            }
        }
        // the tile's unique keys in ascending order, by repeated wave minima (one round per distinct key). Every
        // key of the tile has the tile's ids in its low 16 bits, so the keys compare by their high halves; a
        // pixel whose key has been emitted takes 0x10000 + the key's index in the list, above every high half
        // still pending, and keeps it as its index (no search afterwards)
        const uint32_t low = (ti & 0xFFu) | ((tj & 0xFFu) << 8);
        for (;;) {
            uint32_t mine = key[0];
#pragma unroll
            for (int q = 1; q < 16; q++) mine = min(mine, key[q]);
            const uint32_t m = wave_min_u32(mine);
            if (m > 0xFFFFu) break; // every key emitted (wave-uniform)
            if (lane == 0) uq[u] = (m << 16) | low;
#pragma unroll
            for (int q = 0; q < 16; q++) key[q] = key[q] == m ? 0x10000u + u : key[q];
            u++;
        }
        __builtin_amdgcn_wave_barrier();
    }
    // the group's aggregate is published as soon as its tiles' unique counts are known, before this group's own
    // walk, so that the next groups' walks can sum it without waiting for the walk
    if (lane == 0) s_u[wave] = u;
    __syncthreads();
    if (wave == 0) {
        const uint32_t agg = wave_sum(lane < kClusterWaves ? s_u[lane] : 0u);
        if (lane == 0) wave_lookback_publish(tile_status + fd.tile_base / VREN_TILE_GROUP, t0 / VREN_TILE_GROUP, agg);
    }
    // decoupled look-back over the frame's tile groups (row-major order), one walk per workgroup: a round trip of
    // the walk covers 64 groups = 512 tiles
    if (wave == 0) {
        const uint32_t agg = wave_sum(lane < kClusterWaves ? s_u[lane] : 0u);
        const uint32_t prefix = wave_lookback_walk(tile_status + fd.tile_base / VREN_TILE_GROUP, t0 / VREN_TILE_GROUP, agg);
        if (lane == 0) s_prefix = prefix;
    }
    __syncthreads();
    if (!live) return;
    uint32_t prefix = s_prefix;
    for (uint32_t w = 0; w < wave; w++) prefix += s_u[w];
    if (lane == 0) tile_cl[g] = make_uint2(prefix, u);
    for (uint32_t i = lane; i < u; i += VREN_WAVE) {
        const uint32_t idx = prefix + i;
        if (idx < fd.key_cap) fd.keys[idx] = uq[i];
    }
    if (lane == 0 && t == tiles - 1) {
        const uint32_t total = prefix + u;
        *fd.cluster_count = total;
        if (total > fd.key_cap) atomic_or_agent(fd.flags, VREN_FLAG_KEY_CAPACITY);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t y = tj * 32 + j * 8 + (lane >> 3);
        if (y >= fd.H) continue;
        uint32_t ref[4];
#pragma unroll
        for (int q = 0; q < 4; q++) ref[q] = (prefix - 0x10000u) + key[4 * j + q]; // key = 0x10000 + index
        uint32_t* row = fd.refs + (uint64_t)y * fd.W;
        if (x0 + 3 < fd.W) {
            *reinterpret_cast<vu4_a4*>(row + x0) = vu4_a4{ref[0], ref[1], ref[2], ref[3]};
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (x0 + q < fd.W) row[x0 + q] = ref[q];
        }
    }
}

} // namespace
