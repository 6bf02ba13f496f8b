// clusters.hip -- find_unique_cluster_list (clustered_shading.cpp:363-448, find_unique_clusters.comp:46-121).
//
// One wave per 32x32 tile (tiles flattened over every frame of a batch); each lane derives the 32-bit cluster keys
// of 16 pixels (depth slice from the D32 depth, cube-face normal code from the RGBA16F normal). The reference
// sorts the tile's 1024 keys with a 55-step LDS bitonic network and 20 barriers; here the wave extracts the tile's
// unique keys in ascending order by repeated wave64 minima (one round per distinct key -- a tile of a real scene
// holds a handful), and the unique counts of a group of 8 tiles are chained to the previous groups of the same frame
// by a decoupled look-back. This replaces the reference's atomicAdd allocation (whose order across tiles is nondeterministic,
// find_unique_clusters.comp:100-103) by the canonical row-major tile order, and needs no separate scan dispatch.
// Each pixel keeps the index of its key in the tile's list from the round that emitted the key and stores the
// frame-wide cluster index.
//
// Defined behaviour where the reference has none: pixels of partial tiles sample (x mod W, y mod H) like its
// REPEAT sampler (gbuffer.cpp:28-34) and do not store a reference; a view depth below near gives slice 0; keys
// past the key capacity are not stored and raise the capacity flag.
#include "clusters_device.hpp"

namespace {

__global__ void chain_init_kernel(uint32_t* clear, uint32_t clear_words)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < clear_words; i += gridDim.x * blockDim.x) clear[i] = 0u;
}

template <bool DEEP>
__global__ __launch_bounds__(kClusterWaves * 64, DEEP ? 2 : 8) void clusters_kernel(
    const FrameDev* __restrict__ frames, const uint32_t* __restrict__ tile_frame, uint32_t total_tiles,
    uint64_t* tile_status, uint32_t* ticket, uint2* __restrict__ tile_cl)
{
    clusters_body<DEEP>(frames, tile_frame, total_tiles, tile_status, ticket, tile_cl);
}
template <bool DEEP>
__global__ __launch_bounds__(kClusterWaves * 64, DEEP ? 2 : 8) void clusters_one_kernel(const FrameDev one,
                                                                                       uint32_t total_tiles,
                                                                                       uint64_t* tile_status,
                                                                                       uint32_t* ticket,
                                                                                       uint2* __restrict__ tile_cl)
{
    clusters_body<DEEP>(inline_frame(), nullptr, total_tiles, tile_status, ticket, tile_cl);
}

} // namespace

void chain_work_bind(ChainWork* w, void* mem, uint32_t total_tiles)
{
    w->tickets = static_cast<uint32_t*>(mem);
    w->tile_status = reinterpret_cast<uint64_t*>(static_cast<char*>(mem) + 256);
    w->tile_cl = reinterpret_cast<uint2*>(static_cast<char*>(mem) + chain_work_clear_bytes(total_tiles));
    w->tile_range = w->tile_cl + total_tiles;
    w->total_tiles = total_tiles;
}

// the words that a run finds zero (tickets and statuses) are cleared here only where the previous run may not have
// left them so
int launch_chain_init(vren_ctx* ctx, hipStream_t s, const ChainWork& w)
{
    const uint32_t words = (uint32_t)(chain_work_clear_bytes(w.total_tiles) / 4);
    chain_init_kernel<<<std::max<uint32_t>(1, std::min<uint32_t>(256, (words + 255) / 256)), 256, 0, s>>>(w.tickets, words);
    VREN_LAUNCH_CHECK(ctx);
    return VREN_OK;
}

int launch_clusters(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w,
                    const FrameDev* one)
{
    const uint32_t blocks = (w.total_tiles + kClusterWaves - 1) / kClusterWaves;
    // one workgroup per CU at most: two waves per SIMD, which have the registers to load a whole tile at once
    const bool deep = blocks <= (uint32_t)ctx->num_cus;
    if (one) {
        const int st = launch_chain_init(ctx, s, w);
        if (st) return st;
        const auto kernel = deep ? clusters_one_kernel<true> : clusters_one_kernel<false>;
        kernel<<<blocks, kClusterWaves * 64, 0, s>>>(*one, w.total_tiles, w.tile_status, w.tickets + 0, w.tile_cl);
    } else {
        const auto kernel = deep ? clusters_kernel<true> : clusters_kernel<false>;
        kernel<<<blocks, kClusterWaves * 64, 0, s>>>(d_frames, F > 1 ? w.tile_frame : nullptr, w.total_tiles, w.tile_status,
                                                     w.tickets + 0, w.tile_cl);
    }
    VREN_LAUNCH_CHECK(ctx);
    chain_mark(w, s);
    return VREN_OK;
}

extern "C" VREN_EXPORT int vren_find_unique_cluster_list(vren_ctx* ctx, vren_stream_t stream, uint32_t width,
                                                         uint32_t height, const vren_camera* camera,
                                                         const vren_cluster_cfg* cfg, const float* depth,
                                                         const uint16_t* normals, uint32_t* cluster_keys,
                                                         uint32_t key_capacity, uint32_t* cluster_count,
                                                         uint32_t* cluster_refs)
{
    if (!ctx) return VREN_EINVAL;
    int st = vren_validate_camera(ctx, camera);
    if (!st) st = vren_validate_cfg(ctx, cfg);
    if (st) return st;
    if (width == 0 || height == 0 || width > 8192 || height > 8192)
        return vren_fail(ctx, VREN_EINVAL, "find_unique_cluster_list: screen must be in [1, 8192]^2 (8-bit tile ids)");
    if (!depth || !normals || !cluster_keys || !cluster_count || !cluster_refs || key_capacity == 0)
        return vren_fail(ctx, VREN_EINVAL, "find_unique_cluster_list: null buffer or zero key capacity");
    if (ctx->device < 0) return vren_fail(ctx, VREN_EINVAL, "find_unique_cluster_list: context has no device");
    hipStream_t s = (hipStream_t)stream;
    FrameDev f;
    memset(&f, 0, sizeof(f));
    vren_frame_setup(&f, width, height, camera, cfg);
    f.depth = depth;
    f.normals = normals;
    f.keys = cluster_keys;
    f.key_cap = key_capacity;
    f.cluster_count = cluster_count;
    f.refs = cluster_refs;
    f.flags = ctx->d_flags;
    ChainWork w;
    memset(&w, 0, sizeof(w));
    uint32_t tiles = f.Sx * f.Sy;
    st = vren_ensure_scratch(ctx, chain_work_bytes(tiles), s);
    if (st) return st;
    chain_work_bind(&w, ctx->scratch, tiles);
    return launch_clusters(ctx, s, nullptr, 1, w, &f);
}
