// lights.hip -- construct_point_light_bvh (clustered_shading.cpp:60-346) and build_bvh (build_bvh.cpp:38-99).
//
// Reference: 8 recorded steps and ~10 dispatches per frame (view transform, two vec4 reduce trees, a copy,
// Morton codes, a 65 536-bucket atomic bucket sort with a fixed 2^16 scan, leaf init, then one dispatch per BVH
// level). Here a frame's lights are cut into chunks of 4096, one workgroup each:
//   lights_kernel        view transform, AABB (order-independent min/max), Morton codes and a stable LSD radix sort of
//                        (code, light index) in LDS. A frame of one chunk also builds its whole BVH there, from the
//                        sorted lights in LDS, so it takes one launch; a chunk of a larger frame leaves its sorted
//                        run in global memory.
// and for the frames of more than one chunk:
//   lights_bounds_kernel (ahead) view transform and the AABB of each chunk;
//   lights_merge_kernel  each light's rank in the frame: its place in its own run plus the number of lights that sort
//                        before it in every other run (binary searches), which is the stable order;
//   bvh_leaf_kernel      every leaf: leaf AABB = view position -+ radius, and the first parent level straight from
//                        registers (32-lane min/max over half-waves);
//   bvh_upper_kernel     one workgroup per frame for the remaining (<= 32^k / 32) parent levels.
// A batch of frames runs the same launches with the chunks (or leaf ranges) of every frame side by side.
#include "lights_device.hpp"

namespace {

constexpr uint32_t kMergeThreads = 256;
constexpr uint32_t kMergeParts = kLChunk / kMergeThreads; // merge workgroups per chunk

// Frames of more than one chunk: the chunk's view positions (point_light_position_to_view_space.comp:26-32) and box.
__global__ __launch_bounds__(kLT) void lights_bounds_kernel(const FrameDev* __restrict__ frames, uint32_t F)
{
    __shared__ uint32_t s_red[6 * kLWaves];
    uint32_t chunk;
    const FrameDev& fd = frame_of_chunk(frames, F, blockIdx.x, &chunk);
    if (fd.L <= kLChunk) return; // the whole workgroup
    const uint32_t first = chunk * kLChunk;
    BoxKeys box = empty_box();
#pragma unroll
    for (int j = 0; j < kLKPT; j++) {
        const uint32_t i = first + j * kLT + threadIdx.x;
        if (i < fd.L) {
            const float4 p = reinterpret_cast<const float4*>(fd.light_pos)[i];
            const float v[4] = {p.x, p.y, p.z, 1.0f};
            float r[4];
            vren_mat4_mul_vec4(fd.view, v, r);
            reinterpret_cast<float4*>(fd.view_pos)[i] = make_float4(r[0], r[1], r[2], r[3]);
            add_to_box(box, r);
        }
    }
    block_box(box, s_red);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int a = 0; a < 6; a++) fd.chunk_box[chunk * 6 + a] = box.k[a];
    }
}

template <int BITS>
__global__ __launch_bounds__(kLT) void lights_kernel(const FrameDev* __restrict__ frames, uint32_t F, uint32_t chunks)
{
    lights_body<BITS>(frames, F, chunks);
}
__global__ __launch_bounds__(kLT) void lights_one_kernel(const FrameDev one) { lights_body<8>(inline_frame(), 1, 1); }

// Frames of more than one chunk: codes[rank] for every light of the chunks' sorted runs. A light's rank is its place in
// its run plus, for every other run, the number of its lights that sort before it: codes up to and including the
// light's in the runs before its own (their light indices are lower), codes below it in the runs after. A workgroup
// takes kMergeThreads neighbouring lights of a run, whose bounds fall into a short range of every other run: one wave
// finds the range from every 64th code of the run (one load and two ballots) and stages it in LDS, kMergeRuns runs at
// a time, and each thread searches the staged codes. A range that is longer than the stage (a run that lies inside the
// workgroup's range of codes, as when light indices follow their places) is searched in global memory. 65 536 lights
// took 34 us with every search in global memory (26 dependent loads that miss the L2 of their XCD) and take 17 us.
constexpr uint32_t kMergeRuns = 16;   // runs staged at a time (8 take the same time)
// codes staged per run, two workgroups' worth (a 3840x2160 frame with 65536 lights 580 us with 256, 567 with 512, 568 with 1024)
constexpr uint32_t kMergeStage = 512;
constexpr uint32_t kMergeWaves = kMergeThreads / VREN_WAVE;

// the number of codes below `bound` among codes[0 .. len), ascending, len <= 2 * top (a power of 2)
template <typename Get>
__device__ __forceinline__ uint32_t count_below(Get code, uint32_t len, uint32_t bound, uint32_t top)
{
    uint32_t pos = 0;
    // the halving steps reach 2 top - 1, the last one 2 top
    for (uint32_t step = top; step >= 1; step >>= 1)
        if (pos + step <= len && code(pos + step - 1u) < bound) pos += step;
    if (pos < len && code(pos) < bound) pos++;
    return pos;
}

__global__ __launch_bounds__(kMergeThreads) void lights_merge_kernel(const FrameDev* __restrict__ frames, uint32_t F)
{
    __shared__ uint32_t s_code[kMergeRuns][kMergeStage];
    __shared__ uint32_t s_first[kMergeRuns], s_len[kMergeRuns]; // the staged range of each run; 0xFFFFFFFF: not staged
    uint32_t chunk;
    const FrameDev& fd = frame_of_chunk(frames, F, blockIdx.x / kMergeParts, &chunk);
    const uint32_t L = fd.L;
    const uint32_t p0 = (blockIdx.x % kMergeParts) * kMergeThreads;
    const uint32_t own_len = min(kLChunk, L - chunk * kLChunk);
    if (L <= kLChunk || p0 >= own_len) return; // the whole workgroup
    const uint32_t lane = lane_id(), wave = wave_id();
    gvu2* runs = (gvu2*)fd.codes_tmp;
    const uint32_t p = p0 + threadIdx.x;
    const vu2 mine = runs[chunk * kLChunk + min(p, own_len - 1u)];
    // the lowest and the highest code of the workgroup's lights
    const uint32_t low = runs[chunk * kLChunk + p0].x;
    const uint32_t high = runs[chunk * kLChunk + min(p0 + kMergeThreads, own_len) - 1u].x;
    const uint32_t n_chunks = (L + kLChunk - 1) / kLChunk;
    uint32_t rank = p;
    for (uint32_t c0 = 0; c0 < n_chunks; c0 += kMergeRuns) {
        __syncthreads(); // the previous stage's readers are done
        uint32_t first[kMergeRuns / kMergeWaves], len[kMergeRuns / kMergeWaves];
#pragma unroll
        for (uint32_t k = 0; k < kMergeRuns / kMergeWaves; k++) {
            const uint32_t c = c0 + k * kMergeWaves + wave;
            const uint32_t n = c < n_chunks ? min(kLChunk, L - c * kLChunk) : 0u;
            static_assert(kLChunk == VREN_WAVE * VREN_WAVE, "one sample per lane");
            const uint32_t sample = lane * VREN_WAVE < n ? runs[c * kLChunk + lane * VREN_WAVE].x : 0xFFFFFFFFu;
            // every bound of the workgroup is in [low, high + 1]: of the codes in front of the first range are all
            // below it, and of the codes past the last sample below high + 1 at most the rest of its 64
            const uint32_t m1 = (uint32_t)__popcll(ballot(sample < low)), m2 = (uint32_t)__popcll(ballot(sample < high + 1u));
            first[k] = m1 ? (m1 - 1u) * VREN_WAVE : 0u;
            len[k] = min(n, m2 * VREN_WAVE) - min(first[k], min(n, m2 * VREN_WAVE));
        }
#pragma unroll
        for (uint32_t k = 0; k < kMergeRuns / kMergeWaves; k++) {
            const uint32_t u = k * kMergeWaves + wave, c = c0 + u;
            if (len[k] <= kMergeStage)
                for (uint32_t i = lane; i < len[k]; i += VREN_WAVE) s_code[u][i] = runs[c * kLChunk + first[k] + i].x;
            if (lane == 0) {
                s_first[u] = first[k];
                s_len[u] = len[k] <= kMergeStage ? len[k] : 0xFFFFFFFFu;
            }
        }
        __syncthreads();
        const uint32_t m = min(kMergeRuns, n_chunks - c0);
#pragma unroll 8
        for (uint32_t u = 0; u < m; u++) {
            const uint32_t c = c0 + u;
            if (c == chunk) continue; // uniform
            const uint32_t bound = mine.x + (c < chunk ? 1u : 0u); // codes have at most 30 bits
            const uint32_t n = s_len[u];
            if (n != 0xFFFFFFFFu) {
                const uint32_t* codes = s_code[u];
                rank += s_first[u] + count_below([&](uint32_t i) { return codes[i]; }, n, bound, kMergeStage / 2);
            } else {
                rank += count_below([&](uint32_t i) { return (uint32_t)runs[c * kLChunk + i].x; },
                                    min(kLChunk, L - c * kLChunk), bound, kLChunk / 2);
            }
        }
    }
    if (p < own_len) reinterpret_cast<uint2*>(fd.codes)[rank] = make_uint2(mine.x, mine.y);
}

// leaves (init_light_array_bvh.comp:42-65) + the first parent level (build_bvh.comp:32-55). `span` selects the
// 32-leaf groups written: every group, only those holding a light (the groups past the last light are all INVALID
// leaves under an INVALID parent, which depend on the light count alone: a batch writes them once, with
// kLeavesPadding, when it is created), or only those padding groups.
__global__ __launch_bounds__(256) void bvh_leaf_kernel(const FrameDev* __restrict__ frames, uint32_t F, bool from_lights,
                                                       uint32_t span)
{
    const uint32_t g = blockIdx.x * 256 + threadIdx.x;
    // the live span's grid covers each frame's light-holding groups only (numbered by live_leaf_base)
    const bool live_grid = span == kLeavesLive;
    const uint32_t f = live_grid ? find_frame(frames, F, blockIdx.x * 256, [](const FrameDev& d) { return d.live_leaf_base; })
                                 : find_frame(frames, F, blockIdx.x * 256, [](const FrameDev& d) { return d.leaf_base; });
    const FrameDev& fd = frames[f];
    const uint32_t i = g - (live_grid ? fd.live_leaf_base : fd.leaf_base);
    const uint32_t padded = fd.bvh_padded;
    if (i >= padded) return; // whole half-waves leave together (padded is a multiple of 32)
    const uint32_t live_end = (fd.L + 31u) & ~31u; // first 32-leaf group without a light
    if (span == kLeavesLive && i >= live_end) return;
    if (span == kLeavesPadding) {
        if (i < live_end) return;
        store_invalid(&fd.bvh[i]);
        if ((lane_id() & 31) == 0) store_invalid(&fd.bvh[padded + i / 32]);
        return;
    }
    float mn[3], mx[3];
    bool valid;
    if (from_lights) {
        valid = i < fd.L;
        if (valid) {
            uint32_t li = reinterpret_cast<const uint2*>(fd.codes)[i].y;
            float4 vp = reinterpret_cast<const float4*>(fd.view_pos)[li];
            float r = reinterpret_cast<const float4*>(fd.lights)[li].w;
            mn[0] = vp.x - r;
            mn[1] = vp.y - r;
            mn[2] = vp.z - r;
            mx[0] = vp.x + r;
            mx[1] = vp.y + r;
            mx[2] = vp.z + r;
            if (fd.leaf_rec) reinterpret_cast<float4*>(fd.leaf_rec)[i] = leaf_record(vp.x, vp.y, vp.z, mn[0], mx[0]);
        } else {
            if (fd.leaf_rec && i < live_end) reinterpret_cast<float4*>(fd.leaf_rec)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            mn[0] = mn[1] = mn[2] = VREN_F32_INF;
            mx[0] = mx[1] = mx[2] = -VREN_F32_INF;
        }
        store_node(&fd.bvh[i], mn, mx, valid ? VREN_BVH_LEAF_NODE : VREN_BVH_INVALID_NODE);
    } else {
        const vren_bvh_node& n = fd.bvh[i];
        valid = n.next != VREN_BVH_INVALID_NODE;
        for (int a = 0; a < 3; a++) {
            mn[a] = valid ? n.min[a] : VREN_F32_INF;
            mx[a] = valid ? n.max[a] : -VREN_F32_INF;
        }
    }
    const uint64_t vm = ballot(valid);
    const uint32_t half = (lane_id() >> 5) << 5;
    const bool any = ((vm >> half) & 0xFFFFFFFFull) != 0ull;
    half_wave_box(mn, mx);
    if ((lane_id() & 31) == 31) {
        uint32_t gi = i / 32;
        store_node(&fd.bvh[padded + gi], mn, mx, any ? gi * 32 : VREN_BVH_INVALID_NODE);
    }
}

// Remaining parent levels, one workgroup per frame. from_lights: only the first ceil(L / 32) nodes of the first
// parent level hold lights (the rest are INVALID), so only they and their ancestors are read; the padding parents are
// INVALID without reading their children (65 536 lights in 2^20 padded leaves: 94 -> 6.6 us). Frames of one chunk
// have their whole BVH from lights_kernel.
__global__ __launch_bounds__(1024) void bvh_upper_kernel(const FrameDev* __restrict__ frames, bool from_lights)
{
    const FrameDev& fd = frames[blockIdx.x];
    if (from_lights && fd.L <= kLChunk) return;
    const uint32_t padded = fd.bvh_padded;
    uint32_t src = padded, size = padded / 32;
    uint32_t live = from_lights ? (fd.L + 31) / 32 : size; // nodes of the level that may be valid
    const uint32_t tid = threadIdx.x;
    while (size > 1) {
        const uint32_t dst = src + size, parents = size / 32, live_parents = (live + 31) / 32;
        // one half-wave per parent
        for (uint32_t base = 0; base < live_parents * 32; base += 1024) {
            const uint32_t c = base + tid;
            const bool in = c < live_parents * 32; // whole half-waves
            float mn[3] = {VREN_F32_INF, VREN_F32_INF, VREN_F32_INF};
            float mx[3] = {-VREN_F32_INF, -VREN_F32_INF, -VREN_F32_INF};
            bool valid = false;
            if (c < live) {
                const float4* q = reinterpret_cast<const float4*>(&fd.bvh[src + c]);
                float4 lo = q[0], hi = q[1];
                valid = __float_as_uint(lo.w) != VREN_BVH_INVALID_NODE;
                if (valid) {
                    mn[0] = lo.x;
                    mn[1] = lo.y;
                    mn[2] = lo.z;
                    mx[0] = hi.x;
                    mx[1] = hi.y;
                    mx[2] = hi.z;
                }
            }
            const uint64_t vm = ballot(valid);
            const uint32_t half = (lane_id() >> 5) << 5;
            const bool any = ((vm >> half) & 0xFFFFFFFFull) != 0ull;
            half_wave_box(mn, mx);
            if (in && (lane_id() & 31) == 31)
                store_node(&fd.bvh[dst + c / 32], mn, mx, any ? src + (c & ~31u) : VREN_BVH_INVALID_NODE);
        }
        for (uint32_t p = live_parents + tid; p < parents; p += 1024) store_invalid(&fd.bvh[dst + p]);
        __syncthreads();
        src = dst;
        size = parents;
        live = live_parents;
    }
}

} // namespace

int launch_light_bounds(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w)
{
    if (w.max_L <= kLChunk) return VREN_OK;
    lights_bounds_kernel<<<w.light_chunks, kLT, 0, s>>>(d_frames, F);
    VREN_LAUNCH_CHECK(ctx);
    return VREN_OK;
}

int launch_light_merge(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w)
{
    if (w.max_L <= kLChunk) return VREN_OK;
    lights_merge_kernel<<<w.light_chunks * kMergeParts, kMergeThreads, 0, s>>>(d_frames, F);
    VREN_LAUNCH_CHECK(ctx);
    return VREN_OK;
}

int launch_lights(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w,
                  const FrameDev* one)
{
    const uint32_t chunks = w.light_chunks;
    if (one) { // one chunk; the workgroups past the first write the padding leaves
        const bool padding = one->bvh_padded > ((one->L + 31u) & ~31u);
        lights_one_kernel<<<1 + (padding ? (one->bvh_padded + kLT - 1) / kLT : 0u), kLT, 0, s>>>(*one);
        VREN_LAUNCH_CHECK(ctx);
    } else if (chunks) {
        int st = launch_light_bounds(ctx, s, d_frames, F, w);
        if (st) return st;
        if (w.light_bits == 4) lights_kernel<4><<<chunks, kLT, 0, s>>>(d_frames, F, chunks);
        else lights_kernel<8><<<chunks, kLT, 0, s>>>(d_frames, F, chunks);
        VREN_LAUNCH_CHECK(ctx);
        st = launch_light_merge(ctx, s, d_frames, F, w);
        if (st) return st;
    }
    chain_mark(w, s, chunks || one);
    return VREN_OK;
}

// total_leaf_slots: the grid in leaf slots, the frames' live slots (live_leaf_base numbering) for kLeavesLive; none
// when no frame has more than one chunk of lights (lights_kernel has built their BVHs)
int launch_bvh(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, uint32_t total_leaf_slots,
               bool leaves_from_lights, const ChainWork* w, uint32_t span)
{
    if (total_leaf_slots) {
        bvh_leaf_kernel<<<total_leaf_slots / 256, 256, 0, s>>>(d_frames, F, leaves_from_lights, span);
        VREN_LAUNCH_CHECK(ctx);
    }
    if (span == kLeavesPadding) return VREN_OK;
    if (w) chain_mark(*w, s, total_leaf_slots);
    if (total_leaf_slots) {
        bvh_upper_kernel<<<F, 1024, 0, s>>>(d_frames, leaves_from_lights);
        VREN_LAUNCH_CHECK(ctx);
    }
    if (w) chain_mark(*w, s, total_leaf_slots);
    return VREN_OK;
}

static bool is_pow32(uint32_t n)
{
    if (n < 32) return false;
    while (n > 1) {
        if (n % 32) return false;
        n /= 32;
    }
    return true;
}

extern "C" {

VREN_EXPORT int vren_build_bvh(vren_ctx* ctx, vren_stream_t stream, vren_bvh_node* nodes, uint32_t padded_leaf_count)
{
    if (!ctx) return VREN_EINVAL;
    if (!nodes || !is_pow32(padded_leaf_count))
        return vren_fail(ctx, VREN_EINVAL, "build_bvh: leaf count must be a power of 32 and >= 32 (build_bvh.cpp:45)");
    if (ctx->device < 0) return vren_fail(ctx, VREN_EINVAL, "build_bvh: context has no device");
    hipStream_t s = (hipStream_t)stream;
    FrameDev f;
    memset(&f, 0, sizeof(f));
    f.bvh = nodes;
    f.bvh_padded = padded_leaf_count;
    FrameDev* slot = vren_next_frame_slot(ctx);
    int st = vren_upload_frames(ctx, s, slot, &f, 1);
    if (st) return st;
    uint32_t slots = (padded_leaf_count + VREN_LEAF_ALIGN - 1) / VREN_LEAF_ALIGN * VREN_LEAF_ALIGN;
    return launch_bvh(ctx, s, slot, 1, slots, false, nullptr, kLeavesAll);
}

VREN_EXPORT int vren_construct_point_light_bvh(vren_ctx* ctx, vren_stream_t stream, const float* light_positions,
                                               const float* point_lights, uint32_t light_count,
                                               const vren_camera* camera, const vren_cluster_cfg* cfg,
                                               float* view_positions, uint32_t* light_codes, vren_bvh_node* bvh)
{
    if (!ctx) return VREN_EINVAL;
    int st = vren_validate_camera(ctx, camera);
    if (!st) st = vren_validate_cfg(ctx, cfg);
    if (st) return st;
    if (light_count == 0) return VREN_OK; // the reference skips the stage without lights (clustered_shading.cpp:957)
    if (!light_positions || !point_lights || !view_positions || !light_codes || !bvh)
        return vren_fail(ctx, VREN_EINVAL, "construct_point_light_bvh: null buffer");
    if (light_count > (1u << 20))
        return vren_fail(ctx, VREN_EINVAL, "construct_point_light_bvh: at most 2^20 lights (config.hpp:18)");
    if (ctx->device < 0) return vren_fail(ctx, VREN_EINVAL, "construct_point_light_bvh: context has no device");
    hipStream_t s = (hipStream_t)stream;
    FrameDev f;
    memset(&f, 0, sizeof(f));
    vren_frame_setup(&f, 32, 32, camera, cfg);
    f.light_pos = light_positions;
    f.lights = point_lights;
    f.L = light_count;
    f.view_pos = view_positions;
    f.codes = light_codes;
    f.bvh = bvh;
    f.bvh_padded = vren_calc_bvh_padded_leaf_count(light_count);
    f.bvh_root = vren_calc_bvh_root_index(light_count);
    f.bvh_levels = vren_calc_bvh_level_count(light_count);
    f.bvh_length = vren_calc_bvh_buffer_length(light_count);
    const uint32_t chunks = (light_count + kLChunk - 1) / kLChunk;
    if (chunks > 1) {
        const size_t runs = (size_t)light_count * 8;
        st = vren_ensure_scratch(ctx, runs + (size_t)chunks * VREN_CHUNK_BOX_BYTES, s);
        if (st) return st;
        f.codes_tmp = static_cast<uint32_t*>(ctx->scratch);
        f.chunk_box = reinterpret_cast<uint32_t*>(static_cast<char*>(ctx->scratch) + runs);
    }
    ChainWork w;
    memset(&w, 0, sizeof(w));
    w.max_L = light_count;
    w.light_chunks = chunks;
    if (chunks == 1) return launch_lights(ctx, s, nullptr, 1, w, &f);
    FrameDev* slot = vren_next_frame_slot(ctx);
    st = vren_upload_frames(ctx, s, slot, &f, 1);
    if (!st) st = launch_lights(ctx, s, slot, 1, w);
    if (st) return st;
    uint32_t slots = (f.bvh_padded + VREN_LEAF_ALIGN - 1) / VREN_LEAF_ALIGN * VREN_LEAF_ALIGN;
    return launch_bvh(ctx, s, slot, 1, slots, true, nullptr, kLeavesAll);
}

} // extern "C"
