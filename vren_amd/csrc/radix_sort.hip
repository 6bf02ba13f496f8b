// radix_sort.hip -- radix_sort (radix_sort.hpp:9-53, radix_sort.cpp:149-338) as a onesweep LSD sort for gfx950.
//
// The reference runs, per 4-bit digit, six dispatches (fill, local count, 16-block reduce, global offset,
// 16-block down-sweep, reorder) over N/1024 workgroups, i.e. 8 passes x 3 reads/writes of the keys and ~48
// dispatches, and its reorder assumes a 32-wide subgroup (radix_sort_reorder.comp:15-17). Here:
//   1. one histogram kernel reads the keys once and counts every pass's digit (LDS atomics, one set of counts per
//      workgroup, which a second kernel adds up and scans);
//   2. one kernel per pass: tiles taken from a ticket counter are ranked stably in LDS with wave64 ballot
//      matching, each tile's per-digit counts are chained across tiles by a per-digit decoupled look-back, and
//      the tile is scattered through an LDS staging buffer so global writes go out in per-digit runs.
// Per pass each key (and value) is read once and written once. Digit width, keys per thread and waves per
// workgroup are template parameters chosen by the autotuner (autotune.hip).
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "radix_device.hpp"
#include "radix_sort.hpp"
#include "scan_device.hpp"

namespace {

// predecessor states read per round trip of the onesweep look-back (2^26 keys in 15360-key tiles: 4 689 us, 8 695, 16 744)
constexpr int kLookback = 4;

// status word of (tile, digit): [31:30] state, [29:0] count
#define RS_AGG (1u << 30)
#define RS_INCL (2u << 30)
#define RS_MASK ((1u << 30) - 1u)

// one workgroup of 1024 threads per CU at most, so that there are few counts to add up afterwards
constexpr uint32_t kHistThreads = 1024;

// PAIRS: the keys are the first words of interleaved (key, value) pairs (key i at keys[2 i]).
// Every workgroup stores its own counts, pass by pass (parts[(pass * gridDim.x + blockIdx.x) * RADIX + digit]), and
// workgroup 0 clears the passes' tile tickets.
template <int BITS, bool PAIRS>
__global__ __launch_bounds__(kHistThreads) void rs_hist_kernel(const uint32_t* __restrict__ keys, uint64_t n,
                                                               uint32_t begin_bit, uint32_t end_bit, uint32_t passes,
                                                               uint32_t* __restrict__ parts,
                                                               uint32_t* __restrict__ clear, uint64_t clear_words,
                                                               uint32_t* __restrict__ counters)
{
    if (blockIdx.x == 0 && threadIdx.x < passes) counters[threadIdx.x] = 0u;
    constexpr uint32_t KPV = PAIRS ? 2 : 4; // keys per 16-byte load
    constexpr int RADIX = 1 << BITS;
    __shared__ uint32_t s_h[8 * RADIX];
    for (uint32_t i = threadIdx.x; i < passes * RADIX; i += kHistThreads) s_h[i] = 0u;
    // clear the first pass's look-back statuses while we are here
    for (uint64_t i = (uint64_t)blockIdx.x * kHistThreads + threadIdx.x; i < clear_words;
         i += (uint64_t)gridDim.x * kHistThreads)
        clear[i] = 0u;
    __syncthreads();
    // the pass loop runs outside the keys held in registers, so its shift, width and bounds (wave-uniform) are
    // computed once per batch of keys rather than once per key
    auto count_keys = [&](const uint32_t* k, int m) {
        for (uint32_t p = 0; p < passes; p++) {
            const uint32_t sh = begin_bit + p * BITS;
            const uint32_t w = min((uint32_t)BITS, end_bit - sh);
            uint32_t* h = s_h + p * RADIX;
            for (int u = 0; u < m; u++) atomicAdd(&h[__builtin_amdgcn_ubfe(k[u], sh, w)], 1u);
        }
    };
    const bool aligned = (reinterpret_cast<uintptr_t>(keys) & 15) == 0;
    const uint64_t n4 = aligned ? n / KPV : 0;
    const uint4* k4 = reinterpret_cast<const uint4*>(keys);
    const uint64_t stride = (uint64_t)gridDim.x * kHistThreads;
    uint64_t i = (uint64_t)blockIdx.x * kHistThreads + threadIdx.x;
    // eight 128-bit loads in flight per thread before the LDS counting
    constexpr int U = 8;
    for (; i + (U - 1) * stride < n4; i += U * stride) {
        uint4 q[U];
#pragma unroll
        for (int u = 0; u < U; u++) q[u] = ntload4(k4 + i + u * stride);
        uint32_t k[U * KPV];
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (PAIRS) {
                k[2 * u] = q[u].x;
                k[2 * u + 1] = q[u].z;
            } else {
                k[4 * u] = q[u].x;
                k[4 * u + 1] = q[u].y;
                k[4 * u + 2] = q[u].z;
                k[4 * u + 3] = q[u].w;
            }
        }
        for (uint32_t p = 0; p < passes; p++) {
            const uint32_t sh = begin_bit + p * BITS;
            const uint32_t w = min((uint32_t)BITS, end_bit - sh);
            uint32_t* h = s_h + p * RADIX;
#pragma unroll
            for (int u = 0; u < U * (int)KPV; u++) atomicAdd(&h[__builtin_amdgcn_ubfe(k[u], sh, w)], 1u);
        }
    }
    for (; i < n4; i += stride) {
        const uint4 q = k4[i];
        const uint32_t k[4] = {q.x, PAIRS ? q.z : q.y, q.z, q.w};
        count_keys(k, (int)KPV);
    }
    for (uint64_t j = n4 * KPV + (uint64_t)blockIdx.x * kHistThreads + threadIdx.x; j < n; j += stride) {
        const uint32_t k = keys[PAIRS ? 2 * j : j];
        count_keys(&k, 1);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < passes * RADIX; i += kHistThreads)
        parts[(i / RADIX * gridDim.x + blockIdx.x) * RADIX + i % RADIX] = s_h[i];
}

// The digits' first output positions of pass blockIdx.x: the n_parts workgroups' counts added up and scanned. The counts
// were written by other XCDs, so a thread asks for many of them at once. Parts that are added up here, in place of
// atomics on one histogram that a launch of its own cleared: 2^20 pairs 78 -> 73 us.
template <int BITS>
__global__ __launch_bounds__(1024) void rs_hexscan_kernel(const uint32_t* __restrict__ parts, uint32_t n_parts,
                                                          uint32_t* __restrict__ hist)
{
    constexpr uint32_t RADIX = 1u << BITS, GROUPS = 1024 / RADIX, U = 16;
    __shared__ uint32_t s_sum[1024];
    __shared__ uint32_t s_wave[16];
    const uint32_t digit = threadIdx.x % RADIX, group = threadIdx.x / RADIX;
    const uint32_t* src = parts + (uint64_t)blockIdx.x * n_parts * RADIX + digit;
    uint32_t sum = 0;
    for (uint32_t b = group; b < n_parts; b += U * GROUPS) {
        uint32_t c[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) c[u] = src[(uint64_t)min(b + u * GROUPS, n_parts - 1u) * RADIX];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) sum += b + u * GROUPS < n_parts ? c[u] : 0u;
    }
    s_sum[threadIdx.x] = sum;
    __syncthreads();
    if (threadIdx.x < RADIX) {
        for (uint32_t g = 1; g < GROUPS; g++) sum += s_sum[g * RADIX + threadIdx.x];
    } else {
        sum = 0;
    }
    uint32_t total;
    const uint32_t ex = block_exclusive_sum<1024>(sum, s_wave, &total);
    if (threadIdx.x < RADIX) hist[blockIdx.x * RADIX + threadIdx.x] = ex;
}

// Reduce-then-scan form, pass part 1: the digit counts of every tile (tiles as in the scatter pass), written
// digit-major (count of digit d in tile t at d * tiles + t) so that one exclusive scan of the whole array gives
// every (digit, tile) its first output position. Per-wave LDS counters keep the atomics uncontended.
template <int BITS, int KPT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void rs_upsweep_kernel(const uint32_t* __restrict__ keys, uint64_t n,
                                                                uint32_t shift, uint32_t width,
                                                                uint32_t* __restrict__ tile_hist, uint32_t tiles)
{
    constexpr int THREADS = WAVES * 64;
    constexpr int RADIX = 1 << BITS;
    constexpr int TILE = THREADS * KPT;
    __shared__ uint32_t s_h[WAVES * RADIX];
    const uint32_t tid = threadIdx.x, wave = tid / VREN_WAVE;
    for (uint32_t i = tid; i < (uint32_t)(WAVES * RADIX); i += THREADS) s_h[i] = 0u;
    __syncthreads();
    const uint32_t tile = blockIdx.x;
    const uint64_t tile_start = (uint64_t)tile * TILE;
    const uint32_t tile_count = (uint32_t)min<uint64_t>((uint64_t)TILE, n - tile_start);
    const uint32_t mask = (1u << width) - 1u;
    uint32_t* h = s_h + wave * RADIX;
    const uint32_t* src = keys + tile_start;
    if ((reinterpret_cast<uintptr_t>(src) & 15) == 0) {
        const uint32_t n4 = tile_count / 4;
        for (uint32_t i = tid; i < n4; i += THREADS) {
            const uint4 q = ntload4(reinterpret_cast<const uint4*>(src) + i);
            atomicAdd(&h[(q.x >> shift) & mask], 1u);
            atomicAdd(&h[(q.y >> shift) & mask], 1u);
            atomicAdd(&h[(q.z >> shift) & mask], 1u);
            atomicAdd(&h[(q.w >> shift) & mask], 1u);
        }
        for (uint32_t i = n4 * 4 + tid; i < tile_count; i += THREADS) atomicAdd(&h[(src[i] >> shift) & mask], 1u);
    } else {
        for (uint32_t i = tid; i < tile_count; i += THREADS) atomicAdd(&h[(src[i] >> shift) & mask], 1u);
    }
    __syncthreads();
    for (uint32_t d = tid; d < (uint32_t)RADIX; d += THREADS) {
        uint32_t c = 0;
#pragma unroll
        for (int w = 0; w < WAVES; w++) c += s_h[w * RADIX + d];
        tile_hist[(uint64_t)d * tiles + tile] = c;
    }
}

// keys and values are staged through LDS one after the other when staging both at once would leave room for
// fewer than two workgroups per CU
template <int KPT, int WAVES, bool VALS>
constexpr bool rs_sequential_staging()
{
    return VALS && 2 * WAVES * 64 * KPT * 4 > 80 * 1024;
}

// the element at a byte offset of 32 bits, which a store takes beside its scalar base
__device__ __forceinline__ uint32_t& at32(uint32_t* p, uint32_t bytes)
{
    return *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(p) + bytes);
}

// tiles of 15360 keys leave room for a second workgroup on the CU, in LDS (79 KB) and, held to 64, in registers: one
// ranks while the other waits for its loads, its look-back or its stores (2^26 keys in 15360-key tiles 947 -> 682 us; one
// workgroup in 23552-key tiles 851 -> 775). With values that needs them read late, when the keys have left, and their
// stores' shorter runs take back part of it: see vren_radix_default_tile. Measured and not kept: counters of 16 bits,
// for tiles of 17408 keys (2^26 pairs 1175 -> 1398 us); workgroups that take one tile after the other and load the next
// tile's keys during this one's stores (1077 -> 1304: the CUs fall into step).
constexpr bool rs_two_per_cu(int kpt, int waves) { return kpt == 15 && waves == 16; }

// RTS = false: onesweep (tiles from a ticket counter, per-digit decoupled look-back, digit_base = the digit's
// first output position). RTS = true: reduce-then-scan scatter pass (tile = workgroup id; digit_base = the scanned
// digit-major tile counts of rs_upsweep_kernel), no tickets and no waiting.
// IN_PAIRS: keys_in holds interleaved (key, value) pairs and vals_in is unused. OUT_PAIRS: the pass writes
// interleaved pairs to keys_out and vals_out is unused. Both need VALS.
// Bucket starts written by a final pass over interleaved pairs (OUT_PAIRS and BSTARTS): bucket(k) = (k >> shift) &
// mask. The staged keys of a tile are sorted by the whole bucket (the pass digit is the bucket's top bits and the
// earlier pass left each digit run sorted by the rest), so a staged key whose staged predecessor has the same pass
// digit has that key as its predecessor in the output too, and writes offsets[c] = its position for the buckets c in
// (bucket(predecessor), bucket(key)]. The first key of each tile's digit run and the buckets past the last key are
// left to bucket_run_starts_kernel, which reads them from the output.
struct BucketStarts {
    uint32_t* offsets;
    uint32_t shift, mask;
};

// The histogram workgroups' counts of one pass (rs_hist_kernel), n of them; n = 0: the pass reads scanned
// digit bases. Up to kPartsMaxKeys keys, each tile sums and scans the few parts itself, beside its
// key loads, which saves the launch that adds them up and, with it, the clearing one that there was (2^16 pairs: 45.3
// -> 38.9 us); tile 0 leaves the bases for whoever reads them after the pass. Above, the sum would take each tile longer
// than the launch takes all of them.
struct HistParts {
    const uint32_t* counts;
    uint32_t n;
};
constexpr uint64_t kPartsMaxKeys = 1ull << 19;
constexpr uint32_t kPartsMaxBlocks = 16;
// the tiles that take them: those of few keys per thread, whose registers have room
constexpr bool takes_parts(int kpt) { return kpt <= 8; }

// the scratch has room for them at every size, so that a scratch sized for more keys is always enough for fewer
uint32_t parts_room(uint64_t n)
{
    return (uint32_t)std::min<uint64_t>(kPartsMaxBlocks, ceil_div_u64(std::max<uint64_t>(n, 1), 4096));
}

template <int BITS, int KPT, int WAVES, bool VALS, bool RTS = false, bool IN_PAIRS = false, bool OUT_PAIRS = false,
          bool BSTARTS = false>
__global__ __launch_bounds__(WAVES * 64, rs_two_per_cu(KPT, WAVES) && !IN_PAIRS && !OUT_PAIRS ? 8 : 1) void rs_onesweep_kernel(const uint32_t* __restrict__ keys_in,
                                                                 const uint32_t* __restrict__ vals_in,
                                                                 uint32_t* __restrict__ keys_out,
                                                                 uint32_t* __restrict__ vals_out, uint64_t n,
                                                                 uint32_t shift, uint32_t width,
                                                                 uint32_t* __restrict__ digit_base,
                                                                 uint32_t* status, uint32_t* counter,
                                                                 uint32_t* __restrict__ clear_next,
                                                                 const BucketStarts bs, const HistParts parts)
{
    constexpr int THREADS = WAVES * 64;
    constexpr int RADIX = 1 << BITS;
    constexpr int TILE = THREADS * KPT;
    constexpr bool SEQ = rs_sequential_staging<KPT, WAVES, VALS>();
    constexpr bool LATE = VALS && !IN_PAIRS && !OUT_PAIRS && rs_two_per_cu(KPT, WAVES);
    static_assert(THREADS >= RADIX, "one thread per digit");
    static_assert(VALS || !(IN_PAIRS || OUT_PAIRS), "interleaved pairs carry values");
    static_assert(OUT_PAIRS || !BSTARTS, "bucket starts come from a pass that writes pairs");
    __shared__ uint32_t s_keys[TILE];
    __shared__ uint32_t s_vals[(VALS && !SEQ) ? TILE : 1];
    __shared__ uint32_t s_whist[WAVES * RADIX];
    __shared__ uint32_t s_goff[RADIX];
    constexpr uint32_t DIGIT_WAVES = (RADIX + VREN_WAVE - 1) / VREN_WAVE;
    __shared__ uint32_t s_scan[2 * DIGIT_WAVES];
    __shared__ uint32_t s_ticket;

    uint32_t tid = threadIdx.x;
    uint32_t lane = lane_id();
    const uint32_t wave = wave_id();
    uint32_t* const row = s_whist + wave * RADIX; // the wave's own counters: no other wave writes them while it ranks
    if (!RTS && tid == 0) s_ticket = atomic_add_agent(counter, 1u);
    for (uint32_t i = lane; i < (uint32_t)RADIX; i += VREN_WAVE) row[i] = 0u;
    if (RTS) __builtin_amdgcn_wave_barrier();
    else __syncthreads();
    const uint32_t tile = RTS ? blockIdx.x : __builtin_amdgcn_readfirstlane(s_ticket);
    const uint64_t tile_start = (uint64_t)tile * TILE;
    const uint32_t tile_count = (uint32_t)min<uint64_t>((uint64_t)TILE, n - tile_start);
    const bool full = tile_count == (uint32_t)TILE;
    if (!RTS && clear_next) {
        for (uint32_t i = tid; i < (uint32_t)RADIX; i += THREADS) clear_next[(uint64_t)tile * RADIX + i] = 0u;
    }

    // warp-striped load; positions past the end of a partial tile hold 0xFFFFFFFF, whose digit is the largest, so
    // they rank after every real key of the tile and the real keys keep the staged positions [0, tile_count)
    const uint32_t wbase = wave * KPT * VREN_WAVE;
    const uint32_t* kin = keys_in + tile_start + wbase + lane;
    const uint32_t* vin = vals_in + tile_start + wbase + lane;
    uint32_t key[KPT], val[VALS ? KPT : 1];
    if (IN_PAIRS) {
        const vu2* pin = reinterpret_cast<const vu2*>(keys_in) + tile_start + wbase + lane;
        if (full) {
#pragma unroll
            for (int j = 0; j < KPT; j++) {
                const vu2 q = __builtin_nontemporal_load(pin + j * VREN_WAVE);
                key[j] = q.x;
                val[j] = q.y;
            }
        } else {
#pragma unroll
            for (int j = 0; j < KPT; j++) {
                const uint32_t i = wbase + j * VREN_WAVE + lane;
                const vu2 q = reinterpret_cast<const vu2*>(keys_in)[tile_start + min(i, tile_count - 1u)];
                key[j] = i < tile_count ? q.x : 0xFFFFFFFFu;
                val[j] = q.y;
            }
        }
    } else if (full) {
#pragma unroll
        for (int j = 0; j < KPT; j++) key[j] = __builtin_nontemporal_load(kin + j * VREN_WAVE);
    } else {
#pragma unroll
        for (int j = 0; j < KPT; j++) {
            const uint32_t i = wbase + j * VREN_WAVE + lane;
            const uint32_t k = keys_in[tile_start + min(i, tile_count - 1u)];
            key[j] = i < tile_count ? k : 0xFFFFFFFFu;
        }
    }
    const auto load_vals = [&]() {
        if (full) {
#pragma unroll
            for (int j = 0; j < KPT; j++) val[j] = __builtin_nontemporal_load(vin + j * VREN_WAVE);
        } else {
#pragma unroll
            for (int j = 0; j < KPT; j++)
                val[j] = vals_in[tile_start + min(wbase + j * VREN_WAVE + lane, tile_count - 1u)];
        }
    };
    uint32_t digit[KPT], local[KPT];
    // the histogram's parts of this thread's digit are requested with the keys and summed after the ranking
    constexpr bool PARTS = !RTS && takes_parts(KPT);
    uint32_t part[PARTS ? kPartsMaxBlocks : 1];
    if constexpr (PARTS) {
#pragma unroll
        for (uint32_t b = 0; b < kPartsMaxBlocks; b++)
            part[b] = tid < (uint32_t)RADIX && b < parts.n ? parts.counts[b * RADIX + tid] : 0u;
    }
#pragma unroll
    for (int j = 0; j < KPT; j++) digit[j] = __builtin_amdgcn_ubfe(key[j], shift, width);
    rank_wave_keys<BITS, KPT>(digit, row, local);
    // the values are read after the ranking: their loads overlap the counts, the look-back and the key stores
    if (VALS && !IN_PAIRS && !LATE) load_vals();
    __syncthreads();
    // per digit: tile count, then the exclusive prefix across waves offset by the digit's tile-local start, so a
    // key's staged position is s_whist[wave][d] + local. The waves of the digits do it, each 64 of them.
    uint32_t dcount = 0, dstart = 0, base = 0;
    if (wave < DIGIT_WAVES) {
        if (tid < (uint32_t)RADIX) {
#pragma unroll
            for (int w = 0; w < WAVES; w++) dcount += s_whist[w * RADIX + tid];
            // onesweep: the tile's per-digit counts (the padding of a partial tile included: only the last tile has
            // padding, and no tile looks back at the last one) are published before they are scanned
            if (!RTS) st_agent_u32(status + (uint64_t)tile * RADIX + tid, (tile == 0 ? RS_INCL : RS_AGG) | dcount);
        }
        dstart = wave_inclusive_sum(dcount);
        if (lane == VREN_WAVE - 1) s_scan[wave] = dstart;
        if constexpr (PARTS) {
            if (parts.n) {
                uint32_t c = 0;
#pragma unroll
                for (uint32_t b = 0; b < kPartsMaxBlocks; b++) c += part[b];
                base = wave_inclusive_sum(c);
                if (lane == VREN_WAVE - 1) s_scan[DIGIT_WAVES + wave] = base;
                base -= c;
            }
        }
    }
    __syncthreads();
    if (wave < DIGIT_WAVES && tid < (uint32_t)RADIX) {
        dstart -= dcount;
        for (uint32_t w = 0; w < wave; w++) dstart += s_scan[w];
        if constexpr (PARTS) {
            if (parts.n) {
                for (uint32_t w = 0; w < wave; w++) base += s_scan[DIGIT_WAVES + w];
                if (tile == 0) digit_base[tid] = base;
            }
        }
        uint32_t run = dstart;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            const uint32_t c = s_whist[w * RADIX + tid];
            s_whist[w * RADIX + tid] = run;
            run += c;
        }
    }
    __syncthreads();
    // the waves that hold the digits look back while the others already scatter
    if (tid < (uint32_t)RADIX) {
        uint32_t prefix = 0;
        if (!RTS && tile != 0) {
            // windowed decoupled look-back on this digit: the states of the kLookback nearest unread predecessors
            // are loaded at once and their counts summed up to the first inclusive one; an unpublished state is
            // waited for and the walk resumes there (tile 0 is always inclusive, so the walk ends at or before it)
            int64_t t = (int64_t)tile - 1;
            for (;;) {
                uint32_t st[kLookback];
#pragma unroll
                for (int i = 0; i < kLookback; i++)
                    st[i] = t - i >= 0 ? ld_agent_u32(status + (uint64_t)(t - i) * RADIX + tid) : RS_INCL;
                int i = 0;
                bool done = false;
                for (; i < kLookback; i++) {
                    if ((st[i] & ~RS_MASK) == 0u) break;
                    prefix += st[i] & RS_MASK;
                    if (st[i] & RS_INCL) {
                        done = true;
                        break;
                    }
                }
                if (done) break;
                t -= i;
                if (i < kLookback) __builtin_amdgcn_s_sleep(1);
            }
            st_agent_u32(status + (uint64_t)tile * RADIX + tid, RS_INCL | (prefix + dcount));
        }
        // global destination of staged position i = s_goff[digit] + i: RTS from the scanned digit-major tile
        // counts, onesweep from the pass histogram's exclusive scan (rs_hexscan_kernel) plus the look-back prefix
        if (RTS) s_goff[tid] = digit_base[(uint64_t)tid * ((n + TILE - 1) / TILE) + tile] - dstart;
        else s_goff[tid] = (PARTS && parts.n ? base : digit_base[tid]) + prefix - dstart;
    }
    // scatter into LDS in tile-local sorted order (every staged position is < TILE, padding included)
    uint32_t sh = shift;
    asm volatile("" : "+s"(sh)); // the digits again from the keys: kept since the ranking, they would take a register a key
#pragma unroll
    for (int j = 0; j < KPT; j++) {
        local[j] += row[__builtin_amdgcn_ubfe(key[j], sh, width)];
        s_keys[local[j]] = key[j];
        if (VALS && !SEQ) s_vals[local[j]] = val[j];
    }
    __syncthreads();
    // staged position i = tid + j * THREADS goes to s_goff[digit] + i (< n: the digit's count over the tiles up to
    // this one never exceeds its count in the pass histogram). A full tile reads all its staged keys before the
    // first store, so the LDS reads overlap.
    if constexpr (OUT_PAIRS) {
        // keys and values of staged position i leave together as one 8-byte pair (positions past the end of a
        // partial tile hold padding and are not stored)
        uint32_t k[KPT], o[KPT], v[KPT];
#pragma unroll
        for (int j = 0; j < KPT; j++) {
            k[j] = s_keys[tid + j * THREADS];
            o[j] = s_goff[__builtin_amdgcn_ubfe(k[j], shift, width)] + tid + j * THREADS;
        }
        if constexpr (BSTARTS) {
            // the staged predecessor, read before the staging is reused for values
#pragma unroll
            for (int j = 0; j < KPT; j++) {
                const uint32_t i = tid + j * THREADS;
                if (i == 0 || !(full || i < tile_count)) continue;
                const uint32_t kp = s_keys[i - 1];
                if (__builtin_amdgcn_ubfe(kp, shift, width) != __builtin_amdgcn_ubfe(k[j], shift, width)) continue;
                const uint32_t b1 = (k[j] >> bs.shift) & bs.mask;
                for (uint32_t c = ((kp >> bs.shift) & bs.mask) + 1u; c <= b1; c++) bs.offsets[c] = o[j];
            }
        }
        if (SEQ) {
            __syncthreads();
#pragma unroll
            for (int j = 0; j < KPT; j++) s_keys[local[j]] = val[j];
            __syncthreads();
#pragma unroll
            for (int j = 0; j < KPT; j++) v[j] = s_keys[tid + j * THREADS];
        } else {
#pragma unroll
            for (int j = 0; j < KPT; j++) v[j] = s_vals[tid + j * THREADS];
        }
        vu2* pout = reinterpret_cast<vu2*>(keys_out);
#pragma unroll
        for (int j = 0; j < KPT; j++)
            if (full || tid + j * THREADS < tile_count) pout[o[j]] = vu2{k[j], v[j]};
        return;
    }
    uint32_t o[KPT]; // in bytes: n < 2^30
    if (full) {
        uint32_t k[KPT];
#pragma unroll
        for (int j = 0; j < KPT; j++) k[j] = s_keys[tid + j * THREADS];
#pragma unroll
        for (int j = 0; j < KPT; j++) o[j] = (s_goff[__builtin_amdgcn_ubfe(k[j], shift, width)] + tid + j * THREADS) * 4u;
        if (VALS && !SEQ) {
            uint32_t v[KPT];
#pragma unroll
            for (int j = 0; j < KPT; j++) v[j] = s_vals[tid + j * THREADS];
#pragma unroll
            for (int j = 0; j < KPT; j++) {
                at32(keys_out, o[j]) = k[j];
                at32(vals_out, o[j]) = v[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < KPT; j++) at32(keys_out, o[j]) = k[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < KPT; j++) {
            const uint32_t i = tid + j * THREADS;
            o[j] = 0u;
            if (i < tile_count) {
                const uint32_t k = s_keys[i];
                o[j] = (s_goff[__builtin_amdgcn_ubfe(k, shift, width)] + i) * 4u;
                at32(keys_out, o[j]) = k;
                if (VALS && !SEQ) at32(vals_out, o[j]) = s_vals[i];
            }
        }
    }
    if (LATE) load_vals(); // the key stores are on their way, and most registers free
    if (SEQ) {
        // the values through the same staging buffer, to the destinations kept from the keys
        __syncthreads();
#pragma unroll
        for (int j = 0; j < KPT; j++) s_keys[local[j]] = val[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < KPT; j++) {
            const uint32_t i = tid + j * THREADS;
            if (full || i < tile_count) at32(vals_out, o[j]) = s_keys[i];
        }
    }
}

// words of one histogram part: every pass's digits (at most four passes of 256, six of 64 or eight of 16)
constexpr uint32_t kPartWords = 1024;

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct Layout {
    size_t tmp_keys, tmp_vals, hist, counters, status_a, status_b, parts, total;
};

Layout layout_for(uint64_t n, bool vals, uint32_t min_tile, uint32_t max_radix)
{
    Layout l;
    uint64_t tiles = ceil_div_u64(std::max<uint64_t>(n, 1), min_tile);
    size_t off = 0;
    l.tmp_keys = off;
    off += align256(n * 4);
    l.tmp_vals = off;
    off += vals ? align256(n * 4) : 0;
    l.hist = off;
    off += align256(8 * 256 * 4);
    l.counters = off;
    off += 256;
    l.status_a = off;
    off += align256(tiles * max_radix * 4);
    l.status_b = off;
    off += align256(tiles * max_radix * 4);
    l.parts = off;
    off += (size_t)parts_room(n) * kPartWords * 4;
    l.total = off;
    return l;
}

// smallest tile among the instantiated configurations (4 waves x 8 keys per thread)
constexpr uint32_t kMinTile = 4 * 64 * 8;

// reduce-then-scan LSD sort: per pass, tile digit counts -> one exclusive scan -> scatter (the tile-count array
// and the scan workspace reuse the onesweep status regions of the scratch)
template <int BITS, int KPT, int WAVES>
int run_sort_rts(vren_ctx* ctx, hipStream_t s, uint32_t* keys, uint32_t* vals, uint64_t n, uint32_t begin_bit,
                 uint32_t end_bit, char* scratch, const Layout& L)
{
    constexpr int RADIX = 1 << BITS;
    constexpr int TILE = WAVES * 64 * KPT;
    const uint32_t passes = (end_bit - begin_bit + BITS - 1) / BITS;
    const uint32_t tiles = (uint32_t)ceil_div_u64(n, TILE);
    uint32_t* tile_hist = reinterpret_cast<uint32_t*>(scratch + L.status_a);
    void* scan_work = scratch + L.status_b;
    uint32_t* tk = reinterpret_cast<uint32_t*>(scratch + L.tmp_keys);
    uint32_t* tv = vals ? reinterpret_cast<uint32_t*>(scratch + L.tmp_vals) : nullptr;
    uint32_t *ksrc = keys, *vsrc = vals, *kdst = tk, *vdst = tv;
    for (uint32_t p = 0; p < passes; p++) {
        uint32_t shift = begin_bit + p * BITS;
        uint32_t width = std::min<uint32_t>(BITS, end_bit - shift);
        rs_upsweep_kernel<BITS, KPT, WAVES><<<tiles, WAVES * 64, 0, s>>>(ksrc, n, shift, width, tile_hist, tiles);
        VREN_LAUNCH_CHECK(ctx);
        int st = vren_scan_with_work(ctx, s, tile_hist, tile_hist, (uint64_t)RADIX * tiles, 1, scan_work);
        if (st) return st;
        if (vals) {
            rs_onesweep_kernel<BITS, KPT, WAVES, true, true><<<tiles, WAVES * 64, 0, s>>>(
                ksrc, vsrc, kdst, vdst, n, shift, width, tile_hist, nullptr, nullptr, nullptr, BucketStarts{}, HistParts{});
        } else {
            rs_onesweep_kernel<BITS, KPT, WAVES, false, true><<<tiles, WAVES * 64, 0, s>>>(
                ksrc, nullptr, kdst, nullptr, n, shift, width, tile_hist, nullptr, nullptr, nullptr, BucketStarts{},
                HistParts{});
        }
        VREN_LAUNCH_CHECK(ctx);
        std::swap(ksrc, kdst);
        std::swap(vsrc, vdst);
    }
    if (ksrc != keys) {
        VREN_HIP(ctx, hipMemcpyAsync(keys, ksrc, n * 4, hipMemcpyDeviceToDevice, s));
        if (vals) VREN_HIP(ctx, hipMemcpyAsync(vals, vsrc, n * 4, hipMemcpyDeviceToDevice, s));
    }
    return VREN_OK;
}

// The digit counts of every pass, ready for the passes: parts that the tiles sum (few keys), or scanned digit bases in
// `hist`; the look-back statuses of the first pass and the tickets are cleared too.
template <int BITS, int KPT, bool PAIRS>
int run_hist(vren_ctx* ctx, hipStream_t s, const uint32_t* keys, uint64_t n, uint32_t begin_bit, uint32_t end_bit,
             uint32_t passes, uint64_t tiles, char* scratch, const Layout& L, HistParts* parts)
{
    constexpr uint32_t RADIX = 1u << BITS;
    uint32_t* hist = reinterpret_cast<uint32_t*>(scratch + L.hist);
    uint32_t* counters = reinterpret_cast<uint32_t*>(scratch + L.counters);
    uint32_t* status = reinterpret_cast<uint32_t*>(scratch + L.status_a);
    // up to kPartsMaxKeys keys the scratch holds the parts in a place of their own, above in the first pass's output,
    // which is longer (n / 16384 parts of 4 KB at most) and not written before they are added up
    const bool few = n <= kPartsMaxKeys;
    const uint32_t blocks = few ? parts_room(n) : (uint32_t)std::min<uint64_t>((uint64_t)ctx->num_cus, n / 16384);
    uint32_t* counts = reinterpret_cast<uint32_t*>(scratch + (few ? L.parts : L.tmp_keys));
    rs_hist_kernel<BITS, PAIRS><<<blocks, kHistThreads, 0, s>>>(keys, n, begin_bit, end_bit, passes, counts, status,
                                                                tiles * RADIX, counters);
    VREN_LAUNCH_CHECK(ctx);
    if (few && takes_parts(KPT)) {
        *parts = HistParts{counts, blocks};
        return VREN_OK;
    }
    rs_hexscan_kernel<BITS><<<passes, 1024, 0, s>>>(counts, blocks, hist);
    VREN_LAUNCH_CHECK(ctx);
    *parts = HistParts{nullptr, 0};
    return VREN_OK;
}

// the counts of pass p
inline HistParts pass_parts(const HistParts& parts, uint32_t p, uint32_t radix)
{
    return HistParts{parts.n ? parts.counts + p * parts.n * radix : nullptr, parts.n};
}

template <int BITS, int KPT, int WAVES>
int run_sort(vren_ctx* ctx, hipStream_t s, uint32_t* keys, uint32_t* vals, uint64_t n, uint32_t begin_bit,
             uint32_t end_bit, char* scratch, const Layout& L)
{
    constexpr int RADIX = 1 << BITS;
    constexpr int TILE = WAVES * 64 * KPT;
    const uint32_t passes = (end_bit - begin_bit + BITS - 1) / BITS;
    const uint64_t tiles = ceil_div_u64(n, TILE);
    uint32_t* hist = reinterpret_cast<uint32_t*>(scratch + L.hist);
    uint32_t* counters = reinterpret_cast<uint32_t*>(scratch + L.counters);
    uint32_t* st[2] = {reinterpret_cast<uint32_t*>(scratch + L.status_a),
                       reinterpret_cast<uint32_t*>(scratch + L.status_b)};
    uint32_t* tk = reinterpret_cast<uint32_t*>(scratch + L.tmp_keys);
    uint32_t* tv = vals ? reinterpret_cast<uint32_t*>(scratch + L.tmp_vals) : nullptr;

    HistParts parts;
    const int err = run_hist<BITS, KPT, false>(ctx, s, keys, n, begin_bit, end_bit, passes, tiles, scratch, L, &parts);
    if (err) return err;
    uint32_t *ksrc = keys, *vsrc = vals, *kdst = tk, *vdst = tv;
    for (uint32_t p = 0; p < passes; p++) {
        uint32_t shift = begin_bit + p * BITS;
        uint32_t width = std::min<uint32_t>(BITS, end_bit - shift);
        uint32_t* clear_next = p + 1 < passes ? st[(p + 1) & 1] : nullptr;
        if (vals) {
            rs_onesweep_kernel<BITS, KPT, WAVES, true><<<(uint32_t)tiles, WAVES * 64, 0, s>>>(
                ksrc, vsrc, kdst, vdst, n, shift, width, hist + p * RADIX, st[p & 1], counters + p, clear_next,
                BucketStarts{}, pass_parts(parts, p, RADIX));
        } else {
            rs_onesweep_kernel<BITS, KPT, WAVES, false><<<(uint32_t)tiles, WAVES * 64, 0, s>>>(
                ksrc, nullptr, kdst, nullptr, n, shift, width, hist + p * RADIX, st[p & 1], counters + p, clear_next,
                BucketStarts{}, pass_parts(parts, p, RADIX));
        }
        VREN_LAUNCH_CHECK(ctx);
        std::swap(ksrc, kdst);
        std::swap(vsrc, vdst);
    }
    if (ksrc != keys) {
        VREN_HIP(ctx, hipMemcpyAsync(keys, ksrc, n * 4, hipMemcpyDeviceToDevice, s));
        if (vals) VREN_HIP(ctx, hipMemcpyAsync(vals, vsrc, n * 4, hipMemcpyDeviceToDevice, s));
    }
    return VREN_OK;
}

// The bucket starts that the final pass leaves out: the first key of every tile's digit run (its output predecessor
// belongs to another tile or digit) and the buckets past the last key. Run (t, d) starts at digit_base[d] plus the
// inclusive count of digit d over tiles < t, which the pass's look-back states hold; one thread per (tile, digit).
__global__ __launch_bounds__(256) void bucket_run_starts_kernel(const uint32_t* __restrict__ pairs, uint64_t n,
                                                                const uint32_t* __restrict__ status,
                                                                const uint32_t* __restrict__ digit_base, uint32_t tiles,
                                                                uint32_t radix, const BucketStarts bs,
                                                                uint32_t n_buckets)
{
    const uint64_t g = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (g >= (uint64_t)tiles * radix) return;
    const uint32_t t = (uint32_t)(g / radix), d = (uint32_t)(g - (uint64_t)t * radix);
    const uint32_t before = t == 0 ? 0u : status[(uint64_t)(t - 1) * radix + d] & RS_MASK;
    const uint32_t upto = status[(uint64_t)t * radix + d] & RS_MASK;
    if (upto > before) {
        const uint64_t q = (uint64_t)digit_base[d] + before;
        if (q < n) { // a run of real keys (the last tile's padding counts but is not in the output)
            const uint32_t bq = (pairs[2 * q] >> bs.shift) & bs.mask;
            const uint32_t first = q == 0 ? 0u : ((pairs[2 * q - 2] >> bs.shift) & bs.mask) + 1u;
            for (uint32_t c = first; c <= bq; c++) bs.offsets[c] = (uint32_t)q;
        }
    }
    if (g == 0) {
        const uint32_t bl = (pairs[2 * (n - 1)] >> bs.shift) & bs.mask;
        for (uint32_t c = bl + 1u; c < n_buckets; c++) bs.offsets[c] = (uint32_t)n;
    }
}

// The bucket starts of sorted pairs by binary search, one thread per bucket: for fewer pairs than buckets, where the
// passes would write most starts one after the other in the gaps between neighbouring keys (1000 pairs into 65536
// buckets: 66 -> 9.7 us, 20000: 45 -> 24).
__global__ __launch_bounds__(256) void bucket_search_kernel(const uint32_t* __restrict__ pairs, uint32_t n,
                                                            const BucketStarts bs, uint32_t n_buckets)
{
    const uint32_t b = blockIdx.x * 256 + threadIdx.x;
    if (b >= n_buckets) return;
    uint32_t lo = 0, hi = n; // the first position whose bucket is at least b
    while (lo < hi) {
        const uint32_t mid = (lo + hi) / 2;
        if (((pairs[2 * (uint64_t)mid] >> bs.shift) & bs.mask) < b) lo = mid + 1;
        else hi = mid;
    }
    bs.offsets[b] = lo;
}

// stable sort of interleaved (key, value) pairs on bits [begin_bit, end_bit), at most two digit passes: the first
// pass reads the pairs and the last one writes them (a single pass does both); between two passes the keys and
// values sit split in the scratch. Per pair: 8 B histogram read + 16 B per pass. With bucket_offsets, the final
// pass and bucket_run_starts_kernel also write the start of every bucket (k >> begin_bit) & (n_buckets - 1).
template <int BITS, int KPT, int WAVES>
int run_sort_pairs(vren_ctx* ctx, hipStream_t s, const uint32_t* in, uint32_t* out, uint64_t n, uint32_t begin_bit,
                   uint32_t end_bit, char* scratch, const Layout& L, uint32_t* bucket_offsets, uint32_t n_buckets)
{
    constexpr int RADIX = 1 << BITS;
    constexpr int TILE = WAVES * 64 * KPT;
    const uint32_t passes = (end_bit - begin_bit + BITS - 1) / BITS;
    if (passes > 2) return vren_fail(ctx, VREN_EINVAL, "radix_sort: interleaved pairs take at most %d bits", 2 * BITS);
    const uint64_t tiles = ceil_div_u64(n, TILE);
    uint32_t* hist = reinterpret_cast<uint32_t*>(scratch + L.hist);
    uint32_t* counters = reinterpret_cast<uint32_t*>(scratch + L.counters);
    uint32_t* st[2] = {reinterpret_cast<uint32_t*>(scratch + L.status_a),
                       reinterpret_cast<uint32_t*>(scratch + L.status_b)};
    uint32_t* tk = reinterpret_cast<uint32_t*>(scratch + L.tmp_keys);
    uint32_t* tv = reinterpret_cast<uint32_t*>(scratch + L.tmp_vals);

    HistParts parts;
    const int err = run_hist<BITS, KPT, true>(ctx, s, in, n, begin_bit, end_bit, passes, tiles, scratch, L, &parts);
    if (err) return err;
    const HistParts parts1 = pass_parts(parts, 1, RADIX);
    const BucketStarts bs{bucket_offsets, begin_bit, n_buckets ? n_buckets - 1u : 0u};
    if (passes == 1) {
        if (bucket_offsets)
            rs_onesweep_kernel<BITS, KPT, WAVES, true, false, true, true, true><<<(uint32_t)tiles, WAVES * 64, 0, s>>>(
                in, nullptr, out, nullptr, n, begin_bit, end_bit - begin_bit, hist, st[0], counters, nullptr, bs, parts);
        else
            rs_onesweep_kernel<BITS, KPT, WAVES, true, false, true, true><<<(uint32_t)tiles, WAVES * 64, 0, s>>>(
                in, nullptr, out, nullptr, n, begin_bit, end_bit - begin_bit, hist, st[0], counters, nullptr, bs, parts);
        VREN_LAUNCH_CHECK(ctx);
    } else {
        const uint32_t shift1 = begin_bit + BITS;
        rs_onesweep_kernel<BITS, KPT, WAVES, true, false, true, false><<<(uint32_t)tiles, WAVES * 64, 0, s>>>(
            in, nullptr, tk, tv, n, begin_bit, BITS, hist, st[0], counters, st[1], BucketStarts{}, parts);
        VREN_LAUNCH_CHECK(ctx);
        if (bucket_offsets)
            rs_onesweep_kernel<BITS, KPT, WAVES, true, false, false, true, true><<<(uint32_t)tiles, WAVES * 64, 0, s>>>(
                tk, tv, out, nullptr, n, shift1, end_bit - shift1, hist + RADIX, st[1], counters + 1, nullptr, bs, parts1);
        else
            rs_onesweep_kernel<BITS, KPT, WAVES, true, false, false, true><<<(uint32_t)tiles, WAVES * 64, 0, s>>>(
                tk, tv, out, nullptr, n, shift1, end_bit - shift1, hist + RADIX, st[1], counters + 1, nullptr, bs, parts1);
        VREN_LAUNCH_CHECK(ctx);
    }
    if (bucket_offsets) {
        const uint64_t threads = tiles * RADIX;
        bucket_run_starts_kernel<<<(uint32_t)ceil_div_u64(threads, 256), 256, 0, s>>>(
            out, n, st[(passes - 1) & 1], hist + (uint64_t)(passes - 1) * RADIX, (uint32_t)tiles, RADIX, bs, n_buckets);
        VREN_LAUNCH_CHECK(ctx);
    }
    return VREN_OK;
}

// ---- a few thousand keys: one workgroup, one launch ----------------------------------------------------------------
// Every pass in LDS (block_sort). Up to kRadixOneWorkgroupMax keys the launches of the multi-tile sort, each with its own loads
// and its own wait for the previous one, take longer than one CU takes to rank the keys: 4096 pairs on 32 bits 64.7 us
// (29.2 with its best configuration) -> 13.7, 8192 pairs 66.1 (30.4) -> 21.7.
constexpr int kBlockSortThreads = 1024, kBlockSortWaves = kBlockSortThreads / VREN_WAVE;

template <int KPT, bool VALS>
__global__ __launch_bounds__(kBlockSortThreads) void rs_block_kernel(uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                                     uint32_t n, uint32_t begin_bit, uint32_t end_bit)
{
    typedef std::conditional_t<VALS, uint2, uint32_t> E;
    __shared__ E s_elem[KPT * kBlockSortThreads];
    __shared__ BlockSortLds<8, kBlockSortWaves> s_sort;
    const uint32_t kpt = (n + kBlockSortThreads - 1) / kBlockSortThreads;
    const uint32_t first = wave_id() * kpt * VREN_WAVE + lane_id();
    E e[KPT];
#pragma unroll
    for (int j = 0; j < KPT; j++) {
        const uint32_t i = first + j * VREN_WAVE;
        e[j] = E{};
        if (j < (int)kpt && i < n) {
            if constexpr (VALS) e[j] = make_uint2(keys[i], vals[i]);
            else e[j] = keys[i];
        }
    }
    block_sort<8, KPT, kBlockSortWaves>(e, kpt, n, begin_bit, end_bit, s_elem, s_sort, [](const E& x) {
        if constexpr (VALS) return x.x;
        else return x;
    });
    for (uint32_t i = threadIdx.x; i < n; i += kBlockSortThreads) {
        if constexpr (VALS) {
            keys[i] = s_elem[i].x;
            vals[i] = s_elem[i].y;
        } else {
            keys[i] = s_elem[i];
        }
    }
}

// the same for interleaved pairs, with the bucket starts: position i writes the starts of the buckets after its
// predecessor's up to its own, the last position also those after it
template <int KPT>
__global__ __launch_bounds__(kBlockSortThreads) void rs_block_pairs_kernel(const uint2* __restrict__ in, uint2* __restrict__ out,
                                                                           uint32_t n, uint32_t begin_bit, uint32_t end_bit,
                                                                           const BucketStarts bs, uint32_t n_buckets)
{
    __shared__ uint2 s_elem[KPT * kBlockSortThreads];
    __shared__ BlockSortLds<8, kBlockSortWaves> s_sort;
    const uint32_t kpt = (n + kBlockSortThreads - 1) / kBlockSortThreads;
    const uint32_t first = wave_id() * kpt * VREN_WAVE + lane_id();
    uint2 e[KPT];
#pragma unroll
    for (int j = 0; j < KPT; j++) {
        const uint32_t i = first + j * VREN_WAVE;
        e[j] = j < (int)kpt && i < n ? in[i] : make_uint2(0u, 0u);
    }
    block_sort<8, KPT, kBlockSortWaves>(e, kpt, n, begin_bit, end_bit, s_elem, s_sort, [](const uint2& x) { return x.x; });
    for (uint32_t i = threadIdx.x; i < n; i += kBlockSortThreads) out[i] = s_elem[i];
    if (!bs.offsets) return;
    const auto bucket = [&](uint32_t i) { return (s_elem[i].x >> bs.shift) & bs.mask; };
    for (uint32_t i = threadIdx.x; i <= n; i += kBlockSortThreads) {
        const uint32_t from = i == 0 ? 0u : bucket(i - 1) + 1u, to = i == n ? n_buckets : bucket(i) + 1u;
        for (uint32_t c = from; c < to; c++) bs.offsets[c] = i;
    }
}

int run_sort_one_workgroup(vren_ctx* ctx, hipStream_t s, uint32_t* keys, uint32_t* vals, uint64_t n, uint32_t begin_bit,
                           uint32_t end_bit, char* scratch, const Layout& L)
{
    if (n > kRadixOneWorkgroupMax) {
        switch (vren_radix_default_tile(n, ctx->num_cus, vals != nullptr, false)) {
        case kRadixTile4096: return run_sort<8, 8, 8>(ctx, s, keys, vals, n, begin_bit, end_bit, scratch, L);
        case kRadixTile8192: return run_sort<8, 8, 16>(ctx, s, keys, vals, n, begin_bit, end_bit, scratch, L);
        case kRadixTile15360: return run_sort<8, 15, 16>(ctx, s, keys, vals, n, begin_bit, end_bit, scratch, L);
        default: return run_sort<8, 23, 16>(ctx, s, keys, vals, n, begin_bit, end_bit, scratch, L);
        }
    }
    const uint32_t m = (uint32_t)n;
    if (vals) {
        if (m <= 2048) rs_block_kernel<2, true><<<1, kBlockSortThreads, 0, s>>>(keys, vals, m, begin_bit, end_bit);
        else rs_block_kernel<8, true><<<1, kBlockSortThreads, 0, s>>>(keys, vals, m, begin_bit, end_bit);
    } else {
        if (m <= 2048) rs_block_kernel<2, false><<<1, kBlockSortThreads, 0, s>>>(keys, vals, m, begin_bit, end_bit);
        else rs_block_kernel<8, false><<<1, kBlockSortThreads, 0, s>>>(keys, vals, m, begin_bit, end_bit);
    }
    VREN_LAUNCH_CHECK(ctx);
    return VREN_OK;
}

typedef int (*sort_fn)(vren_ctx*, hipStream_t, uint32_t*, uint32_t*, uint64_t, uint32_t, uint32_t, char*, const Layout&);

struct SortConfig {
    int bits, kpt, waves;
    sort_fn fn;
    int algorithm; // RadixAlgorithm
};

#define RS_CFG(B, K, W) {B, K, W, &run_sort<B, K, W>, kRadixOnesweep}
#define RS_CFG_RTS(B, K, W) {B, K, W, &run_sort_rts<B, K, W>, kRadixReduceThenScan}
const SortConfig kConfigs[] = {
    RS_CFG(8, 8, 4),  RS_CFG(8, 15, 4), RS_CFG(8, 23, 4), RS_CFG(8, 8, 8),  RS_CFG(8, 15, 8),
    RS_CFG(8, 23, 8), RS_CFG(8, 8, 16), RS_CFG(8, 15, 16), RS_CFG(8, 23, 16), RS_CFG(6, 8, 4),  RS_CFG(6, 15, 4), RS_CFG(6, 23, 4),
    RS_CFG(6, 8, 8),  RS_CFG(6, 15, 8), RS_CFG(6, 23, 8), RS_CFG(6, 8, 16), RS_CFG(4, 8, 4),
    RS_CFG(4, 15, 4), RS_CFG(4, 23, 4), RS_CFG(4, 8, 8),  RS_CFG(4, 15, 8), RS_CFG(4, 23, 8),
    RS_CFG(4, 8, 16),
    RS_CFG_RTS(8, 15, 8), RS_CFG_RTS(8, 23, 8), RS_CFG_RTS(8, 8, 16), RS_CFG_RTS(8, 15, 16), RS_CFG_RTS(8, 23, 4),
    {8, 8, 16, &run_sort_one_workgroup, kRadixOneWorkgroup},
};

} // namespace

// Untuned sorts of up to kRadixOneWorkgroupMax keys take one workgroup. Above, they use 8-bit digits and the smallest tile that still gives no CU more than one tile per pass: a pass then
// takes one tile's time, which is what its size makes it, and above that the largest tile, whose digit runs are the
// longest stores. The smallest one stops at half the CUs, since the look-back over more tiles costs what the tile saves.
// 2^16 pairs on 32 bits: 38.9 us in 4096-key tiles, 45.6 in 8192, 83.5 in 23552; 2^20: 79.5, 76.6, 101; 3 M: 142, 125,
// 115 and 103 in 15360; 4.2 M: 173, 147, 123 and 148.
//
// Above one 23552-key tile per CU: keys alone in 15360-key tiles, two workgroups to a CU (2^24 keys 224 us, in 23552-key
// tiles 241; 2^26 682, 775); with values up to 20 M too (2^23 pairs 183, 192; 2^24 279, 288), above in 23552-key tiles,
// whose digit runs fill more of a cache line in each of the two stores (25 M pairs 428, 423; 2^26 1175, 1072). Interleaved
// pairs need more registers than two workgroups have.
RadixTile vren_radix_default_tile(uint64_t n, int num_cus, bool vals, bool interleaved)
{
    const uint64_t cus = (uint64_t)num_cus;
    if (n <= 4096 * cus / 2) return kRadixTile4096;
    if (n <= 8192 * cus) return kRadixTile8192;
    if (n <= 15360 * cus) return kRadixTile15360;
    if (n <= 23552 * cus || interleaved || (vals && n > 5u << 22)) return kRadixTile23552;
    return kRadixTile15360;
}

int vren_radix_config_count() { return (int)(sizeof(kConfigs) / sizeof(kConfigs[0])); }

void vren_radix_config_info(int i, int* bits, int* kpt, int* waves, int* algorithm)
{
    *bits = kConfigs[i].bits;
    *kpt = kConfigs[i].kpt;
    *waves = kConfigs[i].waves;
    if (algorithm) *algorithm = kConfigs[i].algorithm;
}

int vren_radix_sort_with_config(vren_ctx* ctx, hipStream_t s, int cfg, uint32_t* keys, uint32_t* vals, uint64_t n,
                                uint32_t begin_bit, uint32_t end_bit, void* scratch, size_t scratch_bytes)
{
    Layout L = layout_for(n, vals != nullptr, kMinTile, 256);
    if (scratch_bytes < L.total)
        return vren_fail(ctx, VREN_EINVAL, "radix_sort: scratch of %zu bytes, %zu required", scratch_bytes, L.total);
    if (begin_bit >= end_bit) return VREN_OK;
    return kConfigs[cfg].fn(ctx, s, keys, vals, n, begin_bit, end_bit, static_cast<char*>(scratch), L);
}

int vren_radix_sort_pairs_interleaved(vren_ctx* ctx, hipStream_t s, const uint32_t* in_pairs, uint32_t* out_pairs,
                                      uint64_t n, uint32_t begin_bit, uint32_t end_bit, void* scratch,
                                      size_t scratch_bytes, uint32_t* bucket_offsets, uint32_t n_buckets)
{
    Layout L = layout_for(n, true, kMinTile, 256);
    if (scratch_bytes < L.total)
        return vren_fail(ctx, VREN_EINVAL, "radix_sort: scratch of %zu bytes, %zu required", scratch_bytes, L.total);
    if (n == 0) return VREN_OK;
    if (begin_bit >= end_bit) {
        if (bucket_offsets) return vren_fail(ctx, VREN_EINVAL, "radix_sort: bucket starts need a bit range");
        VREN_HIP(ctx, hipMemcpyAsync(out_pairs, in_pairs, n * 8, hipMemcpyDeviceToDevice, s));
        return VREN_OK;
    }
    // fewer pairs than buckets: the starts by search, after a sort without them
    const bool search = bucket_offsets && n < n_buckets;
    uint32_t* starts = search ? nullptr : bucket_offsets;
    const BucketStarts bs{bucket_offsets, begin_bit, n_buckets ? n_buckets - 1u : 0u};
    int st = VREN_OK;
    if (n <= kRadixOneWorkgroupMax) {
        const uint2* in = reinterpret_cast<const uint2*>(in_pairs);
        uint2* out = reinterpret_cast<uint2*>(out_pairs);
        const BucketStarts own{starts, bs.shift, bs.mask};
        if (n <= 2048)
            rs_block_pairs_kernel<2><<<1, kBlockSortThreads, 0, s>>>(in, out, (uint32_t)n, begin_bit, end_bit, own, n_buckets);
        else
            rs_block_pairs_kernel<8><<<1, kBlockSortThreads, 0, s>>>(in, out, (uint32_t)n, begin_bit, end_bit, own, n_buckets);
        VREN_LAUNCH_CHECK(ctx);
    } else {
        const auto sort = [&](auto run) {
            return run(ctx, s, in_pairs, out_pairs, n, begin_bit, end_bit, static_cast<char*>(scratch), L, starts, n_buckets);
        };
        switch (vren_radix_default_tile(n, ctx->num_cus, true, true)) {
        case kRadixTile4096: st = sort(run_sort_pairs<8, 8, 8>); break;
        case kRadixTile8192: st = sort(run_sort_pairs<8, 8, 16>); break;
        case kRadixTile15360: st = sort(run_sort_pairs<8, 15, 16>); break;
        default: st = sort(run_sort_pairs<8, 23, 16>);
        }
    }
    if (st || !search) return st;
    bucket_search_kernel<<<(n_buckets + 255) / 256, 256, 0, s>>>(out_pairs, (uint32_t)n, bs, n_buckets);
    VREN_LAUNCH_CHECK(ctx);
    return VREN_OK;
}

extern "C" {

VREN_EXPORT size_t vren_radix_sort_scratch_bytes(uint64_t n, int with_values)
{
    return layout_for(n, with_values != 0, kMinTile, 256).total;
}

VREN_EXPORT int vren_radix_sort(vren_ctx* ctx, vren_stream_t stream, uint32_t* keys, uint32_t* vals, uint64_t n,
                                uint32_t begin_bit, uint32_t end_bit, void* scratch, size_t scratch_bytes)
{
    if (!ctx) return VREN_EINVAL;
    if (!keys || n == 0 || !scratch) return vren_fail(ctx, VREN_EINVAL, "radix_sort: null buffer or n == 0");
    if (n >= (1ull << 30)) return vren_fail(ctx, VREN_EINVAL, "radix_sort: n must be below 2^30");
    if (begin_bit > end_bit || end_bit > 32) return vren_fail(ctx, VREN_EINVAL, "radix_sort: bad bit range");
    if (scratch_bytes < vren_radix_sort_scratch_bytes(n, vals != nullptr))
        return vren_fail(ctx, VREN_EINVAL, "radix_sort: scratch of %zu bytes, %zu required", scratch_bytes,
                         vren_radix_sort_scratch_bytes(n, vals != nullptr));
    if (ctx->device < 0) return vren_fail(ctx, VREN_EINVAL, "radix_sort: context has no device");
    int cfg = vren_radix_pick_config(ctx, (hipStream_t)stream, n, vals != nullptr, end_bit - begin_bit);
    return vren_radix_sort_with_config(ctx, (hipStream_t)stream, cfg, keys, vals, n, begin_bit, end_bit, scratch,
                                       scratch_bytes);
}

} // extern "C"
