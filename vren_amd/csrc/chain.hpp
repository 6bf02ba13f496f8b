// chain.hpp -- internal launchers of the clustered-shading chain, shared by the per-stage entry points (one
// frame) and the batched chain (many frames in one launch per stage).
#pragma once

#include "clustered.hpp"

int vren_validate_cfg(vren_ctx* ctx, const vren_cluster_cfg* cfg);
int vren_validate_camera(vren_ctx* ctx, const vren_camera* cam);
int vren_upload_frames(vren_ctx* ctx, hipStream_t s, FrameDev* dst, const FrameDev* src, uint32_t n);
int vren_validate_material_set(vren_ctx* ctx, const vren_material_set* m, const char* what);
void vren_frame_set_materials(FrameDev* f, const vren_material_set* m);
FrameDev* vren_next_frame_slot(vren_ctx* ctx);

#define VREN_LEAF_ALIGN 256u
// lights that one workgroup sorts (lights.hip); a frame of at most this many has its BVH from that workgroup
#define VREN_LIGHT_CHUNK 4096u
#define VREN_CHUNK_BOX_BYTES 24u
// a frame's 32x32 tiles start at a multiple of this in the flattened tile numbering of a table (the clusters kernel
// chains its look-back over groups of this many tiles, one workgroup each); tiles of the padding do nothing
#define VREN_TILE_GROUP 8u

// look-back statuses and ticket counter of one chain launch, and the per-tile tables between its stages
struct ChainWork {
    uint64_t* tile_status; // cluster compaction: one word per group of VREN_TILE_GROUP tiles of every frame
    uint32_t* tickets;     // [0] cluster tile groups
    uint2* tile_cl;        // per 32x32 tile: (first cluster index, cluster count), written by the clusters kernel
    uint2* tile_range;     // per 32x32 tile: [begin, end) of the index-buffer entries of its clusters' light lists
    const uint32_t* tile_frame; // frame of every flattened 32x32 tile (null for a one-frame table)
    uint32_t total_tiles;
    uint32_t max_L;
    uint32_t light_chunks;  // chunks of VREN_LIGHT_CHUNK lights over the table's frames (light_chunk_base numbering)
    uint32_t fresh;         // a single-frame shade call whose output holds nothing: zeros for background pixels
    uint32_t any_materials; // some frame of the table takes the material path (shade picks its kernel by it)
    // launch shape (vren_chain_shape; 0 = the default): shade strips per workgroup, persistent assignment waves
    // per CU, digit width of the light sort
    uint32_t shade_ppt = 0;
    uint32_t assign_wpc = 0;
    uint32_t light_bits = 0;
    uint32_t light_concurrent = 0; // batched runs: the light BVH on a second stream beside the cluster stage
    // optional per-stage timing: an event is recorded after every stage of the chain that launches something
    hipEvent_t* events = nullptr;
    int* n_events = nullptr;    // stages so far
    uint32_t* launched = nullptr; // one bit per stage
};

// the end of the chain's next stage; one that launches nothing in this run has no event and no time. A failed record
// surfaces at the checked synchronisation on the last event (vren_batch_run_profiled).
inline void chain_mark(const ChainWork& w, hipStream_t s, bool launched = true)
{
    if (!w.events) return;
    const int i = (*w.n_events)++;
    if (!launched) return;
    *w.launched |= 1u << i;
    vren_teardown(hipEventRecord(w.events[i], s));
}

// stages of one chain launch, in order (chain_mark follows each)
#define VREN_CHAIN_KERNELS 9

// workspace: 256 bytes of tickets, the look-back statuses, the per-tile cluster spans and list ranges. The tickets and
// statuses (the first chain_work_clear_bytes) are zero between runs of a chain: the light-count kernel, which follows
// their last use, clears them.
inline size_t chain_work_clear_bytes(uint32_t total_tiles)
{
    return 256 + ((size_t)total_tiles + VREN_TILE_GROUP - 1) / VREN_TILE_GROUP * sizeof(uint64_t);
}
inline size_t chain_work_bytes(uint32_t total_tiles)
{
    return chain_work_clear_bytes(total_tiles) + (size_t)total_tiles * 16;
}
void chain_work_bind(ChainWork* w, void* mem, uint32_t total_tiles);

// Stage launchers. d_frames is a device table of F FrameDev records; `one`, when given, is the host record of a
// single-frame call instead, passed to the kernels by value (F = 1): the call needs no upload ahead of them.
int launch_chain_init(vren_ctx* ctx, hipStream_t s, const ChainWork& w);
int launch_lights(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w,
                  const FrameDev* one = nullptr);
// the two parts of launch_lights around the chunks' sort, for frames of more than one chunk; launch_lights, but not these,
// marks the stage
int launch_light_bounds(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w);
int launch_light_merge(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w);
// the chunks' sort and the cluster stage in one launch (front.hip), where front_fits
bool front_fits(const vren_ctx* ctx, const ChainWork& w);
int launch_front(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w);
// which 32-leaf groups the leaf kernel writes: all, those holding a light, or the all-padding ones
enum : uint32_t { kLeavesAll = 0, kLeavesLive = 1, kLeavesPadding = 2 };
int launch_bvh(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, uint32_t total_leaf_slots,
               bool leaves_from_lights, const ChainWork* w, uint32_t span);
int launch_clusters(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w,
                    const FrameDev* one = nullptr);
int launch_assign(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w,
                  const FrameDev* one = nullptr);
int launch_shade(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w,
                 const FrameDev* one = nullptr);

// device: the record that a kernel was passed by value as its first argument, where it lies: its fields are then read
// with scalar loads from the kernel's argument segment
__device__ __forceinline__ const FrameDev* inline_frame()
{
    return (const FrameDev*)(const void*)__builtin_amdgcn_kernarg_segment_ptr();
}

// device: frame of a flattened 32x32 tile: one load from the tile -> frame table (uniform across the workgroup)
__device__ __forceinline__ uint32_t frame_of_tile(const uint32_t* tile_frame, uint32_t g)
{
    return tile_frame ? tile_frame[g] : 0u;
}

// device: frame of a flattened index, given a per-frame base field (bases ascending)
template <typename Get>
__device__ __forceinline__ uint32_t find_frame(const FrameDev* frames, uint32_t F, uint32_t g, Get base)
{
    uint32_t lo = 0, hi = F;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) / 2;
        if (base(frames[mid]) <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

// device: the same search done by one whole wave at once (every lane calls it with the same g): lane i reads frame
// c + i's base, and a ballot gives the last frame whose base is <= g. One round of loads instead of log2(F)
// dependent ones.
template <typename Get>
__device__ __forceinline__ uint32_t find_frame_wave(const FrameDev* frames, uint32_t F, uint32_t g, Get base)
{
    const uint32_t lane = lane_id();
    uint32_t f = 0;
    for (uint32_t c = 0; c < F; c += VREN_WAVE) {
        const uint32_t i = c + lane;
        const uint64_t m = ballot(i < F && base(frames[i]) <= g);
        if (m == 0ull) break;
        f = c + 63u - (uint32_t)__builtin_clzll(m);
        if (m != ~0ull) break;
    }
    return f;
}
