// front.hip -- the chain's two independent first stages in one launch, for tables that leave the chip mostly idle: the
// workgroups of the light stage (a chunk of lights each) and those of the cluster stage (eight tiles each) side by side.
// One after the other, a frame waits for one CU to sort its lights while the others have nothing to do: 21 us for 4096.
// Together the stages of a 1920x1080 frame take 22.9 us (44 one after the other), now bound by the lights, and those
// of a 640x360 frame with 256 lights 13.1 (25).
#include "clusters_device.hpp"
#include "lights_device.hpp"

namespace {

// Workgroups of lights first (the longest-running ones). A workgroup of the cluster stage uses its first eight waves:
// the others end at once, and a barrier waits for the waves that are left.
template <int BITS>
__global__ __launch_bounds__(kLT) void front_kernel(const FrameDev* __restrict__ frames, uint32_t F, uint32_t chunks,
                                                    const uint32_t* __restrict__ tile_frame, uint32_t total_tiles,
                                                    uint64_t* tile_status, uint32_t* ticket,
                                                    uint2* __restrict__ tile_cl)
{
    if (blockIdx.x < chunks) {
        lights_body<BITS>(frames, F, chunks);
    } else {
        if (threadIdx.x >= kClusterWaves * VREN_WAVE) return;
        clusters_body<true>(frames, tile_frame, total_tiles, tile_status, ticket, tile_cl);
    }
}

} // namespace

// One workgroup per CU at most: above that the cluster stage fills the chip by itself, with four of its workgroups on a
// CU where the light stage's LDS leaves room for one.
bool front_fits(const vren_ctx* ctx, const ChainWork& w)
{
    const uint32_t groups = (w.total_tiles + kClusterWaves - 1) / kClusterWaves;
    return w.light_chunks > 0 && groups + w.light_chunks <= (uint32_t)ctx->num_cus;
}

int launch_front(vren_ctx* ctx, hipStream_t s, const FrameDev* d_frames, uint32_t F, const ChainWork& w)
{
    const uint32_t grid = w.light_chunks + (w.total_tiles + kClusterWaves - 1) / kClusterWaves;
    const uint32_t* tf = F > 1 ? w.tile_frame : nullptr;
    if (w.light_bits == 4)
        front_kernel<4><<<grid, kLT, 0, s>>>(d_frames, F, w.light_chunks, tf, w.total_tiles, w.tile_status, w.tickets + 0,
                                             w.tile_cl);
    else
        front_kernel<8><<<grid, kLT, 0, s>>>(d_frames, F, w.light_chunks, tf, w.total_tiles, w.tile_status, w.tickets + 0,
                                             w.tile_cl);
    VREN_LAUNCH_CHECK(ctx);
    return VREN_OK;
}
