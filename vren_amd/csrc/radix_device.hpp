// radix_device.hpp -- the stable tile ranking of the onesweep radix sort, and the stable sort of one workgroup's elements
// in LDS that the light stage and the sorts of a few thousand keys share.
//
// Keys are held warp-striped: key j of lane l of wave w sits at tile position (w * KPT + j) * 64 + l, so the
// order (w, j, l) is the input order and ranking in that order is stable. A key's digit peers inside the wave
// come from BITS ballots (wave64 match), its rank among them from mbcnt, and the wave's running per-digit
// count lives in LDS (one row of RADIX counters per wave). After ranking, per-digit counts are turned into
// exclusive prefixes across waves, giving every key its tile-local position:
//   digit_start[d] + wave_prefix[w][d] + local[j].
#pragma once

#include "common.hpp"

// One digit bit of the wave match: bc = the lane's bit b broadcast to a word (v_bfe_i32), VCC = its ballot, and
// per 32-lane half peers &= ~(ballot ^ bc) in one v_bitop3_b32 (truth table over S0 = 0xF0, S1 = 0xCC,
// S2 = 0xAA: 0xF0 & ~(0xCC ^ 0xAA) = 0x90). A VALU write of VCC needs two wait states before a VALU reads it as
// an operand (s_nop 1).
template <int B>
__device__ __forceinline__ void match_bit(uint32_t d, uint32_t& lo, uint32_t& hi)
{
    uint32_t bc;
    asm("v_bfe_i32 %2, %3, %4, 1\n\t"
        "v_cmp_ne_u32_e32 vcc, 0, %2\n\t"
        "s_nop 1\n\t"
        "v_bitop3_b32 %0, %0, vcc_lo, %2 bitop3:0x90\n\t"
        "v_bitop3_b32 %1, %1, vcc_hi, %2 bitop3:0x90"
        : "+v"(lo), "+v"(hi), "=&v"(bc)
        : "v"(d), "i"(B)
        : "vcc");
}

// Bit 0 of a match that starts from every lane: peers = ~(ballot ^ bc) (truth table ~(0xCC ^ 0xAA) = 0x99, S0
// unused).
__device__ __forceinline__ void match_bit0_all(uint32_t d, uint32_t& lo, uint32_t& hi)
{
    uint32_t bc;
    asm("v_bfe_i32 %2, %3, 0, 1\n\t"
        "v_cmp_ne_u32_e32 vcc, 0, %2\n\t"
        "s_nop 1\n\t"
        "v_bitop3_b32 %0, %2, vcc_lo, %2 bitop3:0x99\n\t"
        "v_bitop3_b32 %1, %2, vcc_hi, %2 bitop3:0x99"
        : "=&v"(lo), "=&v"(hi), "=&v"(bc)
        : "v"(d)
        : "vcc");
}

template <int B, int BITS>
__device__ __forceinline__ void match_bits(uint32_t d, uint32_t& lo, uint32_t& hi)
{
    if constexpr (B < BITS) {
        match_bit<B>(d, lo, hi);
        match_bits<B + 1, BITS>(d, lo, hi);
    }
}

// Lanes of the wave holding the same BITS-bit digit as this lane, four VALU operations per digit bit.
// ALL = true: every lane of the wave takes part (lo:hi are outputs only); ALL = false: only the lanes set in lo:hi
// on entry.
template <int BITS, bool ALL = false>
__device__ __forceinline__ void match_digit(uint32_t d, uint32_t& lo, uint32_t& hi)
{
    if constexpr (ALL) {
        match_bit0_all(d, lo, hi);
        match_bits<1, BITS>(d, lo, hi);
    } else {
        match_bits<0, BITS>(d, lo, hi);
    }
}

// s_wave_row: the wave's RADIX counters, zero before the call. Writes local[j] = rank of key j among the same-digit keys
// of this wave that precede it. Every lane takes part: a caller padding a partial tile gives its padding the largest
// digit, so that the padding ranks after every real key of the tile, which keep the positions from 0.
template <int BITS, int KPT>
__device__ __forceinline__ void rank_wave_keys(const uint32_t (&digit)[KPT], uint32_t* s_wave_row, uint32_t (&local)[KPT])
{
    const uint32_t lane = lane_id();
#pragma unroll
    for (int j = 0; j < KPT; j++) {
        const uint32_t d = digit[j];
        uint32_t lo, hi;
        const uint32_t before = s_wave_row[d];
        match_digit<BITS, true>(d, lo, hi);
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
        const uint64_t peers = ((uint64_t)hi << 32) | lo;
        // the highest peer lane publishes the new running count
        if ((peers >> lane) == 1ull) s_wave_row[d] = before + rank + 1u;
        local[j] = before + rank;
        __builtin_amdgcn_wave_barrier();
    }
}

// LDS of block_sort: per-wave digit rows and the digit counts of every 64 digits
template <int BITS, int WAVES>
struct BlockSortLds {
    uint32_t row[WAVES << BITS];
    uint32_t digits[4];
};

// Stable LSD sort of the n elements that a workgroup of WAVES waves holds, on key bits [begin_bit, end_bit) in BITS-bit
// digits, one pass at least; s_elem[0 .. n) holds them in order afterwards (every thread may read it at once). Elements
// are warp-striped, kpt <= KPT per thread (uniform): e[j] of lane l of wave w is element (w kpt + j) 64 + l. They stay in
// registers within a pass and go through s_elem between passes. Three barriers per pass: each wave ranks its elements
// in its own row of digit counters, which it clears itself; one thread per digit turns the rows into wave prefixes;
// what lies in the groups of 64 digits before a digit's is added by the readers.
template <int BITS, int KPT, int WAVES, typename E, typename Key>
__device__ __forceinline__ void block_sort(E (&e)[KPT], uint32_t kpt, uint32_t n, uint32_t begin_bit, uint32_t end_bit,
                                           E* s_elem, BlockSortLds<BITS, WAVES>& lds, Key key)
{
    constexpr uint32_t RADIX = 1u << BITS;
    static_assert(BITS <= 8 && WAVES * VREN_WAVE >= (int)RADIX, "one thread per digit");
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    const uint32_t wbase = wave * kpt * VREN_WAVE;
    uint32_t* row = lds.row + wave * RADIX;
    uint32_t shift = begin_bit;
    for (;;) {
        const uint32_t width = min((uint32_t)BITS, end_bit - shift);
        for (uint32_t i = lane; i < RADIX; i += VREN_WAVE) row[i] = 0u;
        __builtin_amdgcn_wave_barrier();
        uint32_t digit[KPT], local[KPT];
#pragma unroll
        for (int j = 0; j < KPT; j++) {
            digit[j] = __builtin_amdgcn_ubfe(key(e[j]), shift, width);
            local[j] = 0u;
            if (j < (int)kpt) {
                const bool valid = wbase + j * VREN_WAVE + lane < n;
                const uint64_t vm = ballot(valid);
                uint32_t lo = (uint32_t)vm, hi = (uint32_t)(vm >> 32);
                const uint32_t before = valid ? row[digit[j]] : 0u;
                match_digit<BITS>(digit[j], lo, hi);
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
                const uint64_t peers = ((uint64_t)hi << 32) | lo;
                if (valid && (peers >> lane) == 1ull) row[digit[j]] = before + rank + 1u; // the highest peer lane
                local[j] = before + rank;
                __builtin_amdgcn_wave_barrier();
            }
        }
        __syncthreads();
        if (tid < ((RADIX + 63u) & ~63u)) { // whole waves
            uint32_t c[WAVES], sum = 0;
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                c[w] = tid < RADIX ? lds.row[w * RADIX + tid] : 0u;
                sum += c[w];
            }
            const uint32_t incl = wave_inclusive_sum(sum);
            if (lane == VREN_WAVE - 1) lds.digits[wave] = incl;
            uint32_t run = incl - sum;
            if (tid < RADIX) {
#pragma unroll
                for (int w = 0; w < WAVES; w++) {
                    lds.row[w * RADIX + tid] = run;
                    run += c[w];
                }
            }
        }
        __syncthreads();
        uint32_t d1 = 0, d2 = 0, d3 = 0; // elements in the digit groups before groups 1, 2, 3
        if (RADIX > 64) {
            d1 = lds.digits[0];
            d2 = d1 + lds.digits[1];
            d3 = d2 + lds.digits[2];
        }
#pragma unroll
        for (int j = 0; j < KPT; j++) {
            if (j < (int)kpt && wbase + j * VREN_WAVE + lane < n) {
                const uint32_t d = digit[j], g = d >> 6;
                const uint32_t before = g == 0 ? 0u : (g == 1 ? d1 : (g == 2 ? d2 : d3));
                s_elem[before + row[d] + local[j]] = e[j];
            }
        }
        __syncthreads();
        shift += BITS;
        if (shift >= end_bit) return;
#pragma unroll
        for (int j = 0; j < KPT; j++)
            if (j < (int)kpt && wbase + j * VREN_WAVE + lane < n) e[j] = s_elem[wbase + j * VREN_WAVE + lane];
    }
}
