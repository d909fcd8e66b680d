// Texts of a few thousand symbols: a sort whose time is not launches and round trips.
//
// The sorts and scans of a large partition are 15 to 20 launches and three round trips however few suffixes it has. A short text is
// ranked by counting instead: the rank of a suffix is the number of smaller ones, and with the whole text (or all ranks) in the LDS
// of every workgroup each suffix is compared with all others. n^2 comparisons by 256 CUs take less time than one round trip up
// to the length below. Generation 0 compares four symbols, generation t the ranks of the generation before at x and x + h,
// so every rank, active set and group is that of the prefix doubling of large texts.
//   short_first_kernel   generation 0
//   short_rest_kernel    all later ones, in one workgroup, if no group is long (nearly every text)
//   short_next_kernel    one later generation, over the whole device, otherwise
// A suffix leaves for its place in the output in the generation that finds it alone.
// 4096 Zipf tokens, no copies among them: 39 us a sort, 158 the long way; with copies 76 and 447.
#pragma once

#include "device_utils.hpp"
#include "doubling.hpp"

namespace csa {

constexpr int SHORT_BLOCK = 1024;
constexpr u32 SHORT_MAX = 8192;  // the keys of a text take 64 KB of LDS (us a sort of that length, and the long way: tokens 103 and 427, runs 336 and 776,
                                 // bytes 174 and 314, four letters 171 and 391)
constexpr u32 SHORT_X = 16;      // suffixes of a workgroup, each compared with the others by ...
constexpr u32 SHORT_SLICES = SHORT_BLOCK / SHORT_X; // ... so many threads
constexpr u32 SHORT_GROUP = 256; // members of the longest group that one workgroup takes to the end (each looks at all others)
constexpr u32 SHORT_TIED = 0x80000000u; // of a rank: others have it too ...
constexpr u32 SHORT_RANK_BITS = 13, SHORT_RANK = (1u << SHORT_RANK_BITS) - 1; // ... and how many of them are earlier in the text, above the rank
static_assert(SHORT_MAX <= 1u << SHORT_RANK_BITS, "a rank and a place in a group take 26 bits");
constexpr u32 SHORT_GENERATIONS = 16;   // 4, 8, ... symbols: more than SHORT_MAX after 12, one more with keys of three words
constexpr u32 SHORT_LONG = 2 * SHORT_GENERATIONS; // counter: not zero if a group of generation 1 is longer than that
constexpr u32 SHORT_COUNTERS = SHORT_LONG + 1;

struct ShortArgs {
    const u16* text;
    u32 n;
    u64 index_base;
    u8* out;            // 5-byte entries
    const u32* rank_in; // [n] by text position, with SHORT_TIED
    u32* rank_out;
    u32* counters;      // [SHORT_COUNTERS], zeroed: [2 g] suffixes that are still tied when generation g begins, [2 g + 1] their groups
    u32 generation;     // the one that is run
    u32 hops[SHORT_GENERATIONS]; // of generation g: it compares the ranks of x + hops[g]; 0 behind the last
};

__device__ __forceinline__ void short_emit(const ShortArgs& a, u32 place, u32 x)
{
    const u64 v = a.index_base + x;
#pragma unroll
    for (int b = 0; b < 5; ++b)
        a.out[5ull * place + b] = (u8)(v >> (8 * b));
}

// Sums over the slices of every suffix of the workgroup (the lanes of equal threadIdx.x % SHORT_X), and what follows for it:
// its rank, or its place if it is alone. `less`, `equal` (itself not included), `before`: of the equal ones, those earlier in the text.
__device__ __forceinline__ void short_settle(const ShortArgs& a, u32 x, bool there, u32 base, u32 less, u32 equal, u32 before, u32 (*sums)[3])
{
    const u32 t = threadIdx.x, lane = t & 63u, mine = t % SHORT_X;
#pragma unroll
    for (int o = SHORT_X; o < 64; o <<= 1) {
        less += __shfl_xor(less, o);
        equal += __shfl_xor(equal, o);
        before += __shfl_xor(before, o);
    }
    if (lane < SHORT_X) {
        atomicAdd(&sums[mine][0], less);
        atomicAdd(&sums[mine][1], equal);
        atomicAdd(&sums[mine][2], before);
    }
    __syncthreads();
    if (t >= 64)
        return;
    bool tied = false, head = false;
    if (t < SHORT_X && there) {
        const u32 rank = base + sums[t][0];
        tied = sums[t][1] != 0;
        head = tied && sums[t][2] == 0;
        a.rank_out[x] = rank | (tied ? SHORT_TIED | sums[t][2] << SHORT_RANK_BITS : 0u);
        if (!tied)
            short_emit(a, rank, x);
        if (head && a.generation == 0 && sums[t][1] + 1 > SHORT_GROUP)
            a.counters[SHORT_LONG] = 1u;
    }
    const u64 all = __ballot(tied), heads = __ballot(head);
    if (t == 0 && all) {
        atomicAdd(&a.counters[2 * (a.generation + 1)], (u32)__popcll(all));
        atomicAdd(&a.counters[2 * (a.generation + 1) + 1], (u32)__popcll(heads));
    }
}

__global__ __launch_bounds__(SHORT_BLOCK) void short_first_kernel(ShortArgs a)
{
    __shared__ u64 s_key[SHORT_MAX];
    __shared__ u32 s_sums[SHORT_X][3];
    const u32 t = threadIdx.x;
    if (t < SHORT_X * 3)
        s_sums[t / 3][t % 3] = 0;
    for (u32 y = t; y < a.n; y += SHORT_BLOCK)
        s_key[y] = load_kgram(a.text, a.n, y, 0);
    __syncthreads();
    const u32 x = blockIdx.x * SHORT_X + t % SHORT_X;
    const bool there = x < a.n;
    u32 less = 0, equal = 0, before = 0;
    if (there) {
        const u64 key = s_key[x];
        // suffixes that run off the text inside the key tie with nobody, and come before those with the same padded key, shortest first
        const bool whole = x + 4 < a.n;
        const u32 wholes = a.n > 4 ? a.n - 4 : 0u;
#pragma unroll 4
        for (u32 y = t / SHORT_X; y < wholes; y += SHORT_SLICES) {
            const u64 v = s_key[y];
            const u32 same = v == key && whole && y != x ? 1u : 0u;
            less += v < key ? 1u : 0u;
            equal += same;
            before += y < x ? same : 0u;
        }
        if (t / SHORT_X == 0)
            for (u32 y = wholes; y < a.n; ++y) {
                const u64 v = s_key[y];
                less += v < key || (v == key && (whole || y > x)) ? 1u : 0u;
            }
    }
    short_settle(a, x, there, 0, less, equal, before, s_sums);
}

// One generation. The groups are the suffixes of one rank; nobody in them runs off the text.
__global__ __launch_bounds__(SHORT_BLOCK) void short_next_kernel(ShortArgs a)
{
    __shared__ u16 s_rank[SHORT_MAX];
    __shared__ u32 s_sums[SHORT_X][3];
    if (a.counters[2 * a.generation] == 0)
        return;
    const u32 t = threadIdx.x, x = blockIdx.x * SHORT_X + t % SHORT_X;
    const u32 own = x < a.n ? a.rank_in[x] : 0u;
    const bool there = (own & SHORT_TIED) != 0;
    if (t < SHORT_X && x < a.n && !there)
        a.rank_out[x] = own;
    if (__ballot(there) == 0) // (every wave holds the same suffixes)
        return;
    if (t < SHORT_X * 3)
        s_sums[t / 3][t % 3] = 0;
    for (u32 y = t; y < a.n; y += SHORT_BLOCK)
        s_rank[y] = (u16)(a.rank_in[y] & SHORT_RANK);
    __syncthreads();
    const u32 hop = a.hops[a.generation], rank = own & SHORT_RANK;
    u32 less = 0, equal = 0, before = 0;
    if (there && x + hop < a.n) {
        const u32 next = s_rank[x + hop];
#pragma unroll 4
        for (u32 y = t / SHORT_X; y < a.n - hop; y += SHORT_SLICES) {
            const u32 in = s_rank[y] == rank ? 1u : 0u, v = s_rank[y + hop];
            const u32 same = v == next && y != x ? in : 0u;
            less += v < next ? in : 0u;
            equal += same;
            before += y < x ? same : 0u;
        }
    }
    short_settle(a, x, there, rank, less, equal, before, s_sums);
}

// All generations from a.generation on, unless a group is longer than SHORT_GROUP. The members of a group stand side by side, at the places
// that are theirs in the end: a thread owns every SHORT_BLOCK-th place and compares who stands there with the others of the group.
__global__ __launch_bounds__(SHORT_BLOCK) void short_rest_kernel(ShortArgs a)
{
    constexpr int ITEMS = SHORT_MAX / SHORT_BLOCK;
    constexpr u16 NOBODY = 0xFFFFu;
    __shared__ u16 s_rank[SHORT_MAX];
    __shared__ u16 s_member[SHORT_MAX];
    __shared__ u16 s_next[SHORT_MAX]; // the rank that is compared
    __shared__ u16 s_end[SHORT_MAX];  // of the group that stands here
    __shared__ u32 s_tied[2];
    const u32 t = threadIdx.x;
    if (a.counters[2 * a.generation] == 0 || a.counters[SHORT_LONG] != 0)
        return;
    for (u32 y = t; y < a.n; y += SHORT_BLOCK) {
        s_member[y] = NOBODY;
        s_end[y] = 0;
    }
    __syncthreads();
    for (u32 y = t; y < a.n; y += SHORT_BLOCK) {
        const u32 v = a.rank_in[y], rank = v & SHORT_RANK, before = (v >> SHORT_RANK_BITS) & SHORT_RANK;
        s_rank[y] = (u16)rank;
        if ((v & SHORT_TIED) && rank + before < a.n)
            s_member[rank + before] = (u16)y;
    }
    __syncthreads();
    // ends of the groups: the place behind a member whose right neighbour is of another group, or nobody
    for (u32 j = t; j < a.n; j += SHORT_BLOCK) {
        const u32 x = s_member[j];
        if (x == NOBODY)
            continue;
        u32 end = j + 1;
        while (end < a.n && s_member[end] != NOBODY && s_rank[s_member[end]] == s_rank[x])
            ++end;
        s_end[j] = (u16)end;
    }
    for (u32 g = a.generation; g < SHORT_GENERATIONS - 1 && a.hops[g] != 0; ++g) {
        const u32 hop = a.hops[g];
        u32 x[ITEMS], to[ITEMS], end[ITEMS]; // who stands at the thread's places; the new place and end of group
        __syncthreads();
        if (t < 2)
            s_tied[t] = 0;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const u32 j = k * SHORT_BLOCK + t;
            x[k] = j < a.n ? s_member[j] : (u32)NOBODY;
            to[k] = end[k] = 0;
            if (x[k] != NOBODY && x[k] + hop < a.n) // (nobody who is tied runs off the text)
                s_next[j] = s_rank[x[k] + hop];
        }
        __syncthreads();
        u32 tied = 0, heads = 0;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            if (x[k] == NOBODY)
                continue;
            const u32 j = k * SHORT_BLOCK + t, first = s_rank[x[k]], last = s_end[j], mine = s_next[j];
            u32 less = 0, equal = 0, before = 0;
            for (u32 i = first; i < last; ++i) {
                const u32 v = s_next[i];
                less += v < mine ? 1u : 0u;
                equal += v == mine ? 1u : 0u;
                before += v == mine && i < j ? 1u : 0u;
            }
            to[k] = first + less + before;
            end[k] = first + less + equal;
            tied += equal > 1 ? 1u : 0u;
            heads += equal > 1 && before == 0 ? 1u : 0u;
            if (equal == 1)
                short_emit(a, to[k], x[k]);
            x[k] |= (first + less) << 16; // the new rank
            end[k] |= equal > 1 ? 0u : 0x10000u;
        }
        const u32 all_tied = wave_reduce_sum(tied), all_heads = wave_reduce_sum(heads);
        if ((t & 63u) == 0 && all_tied) {
            atomicAdd(&s_tied[0], all_tied);
            atomicAdd(&s_tied[1], all_heads);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const u32 j = k * SHORT_BLOCK + t;
            if (x[k] != NOBODY)
                s_member[j] = NOBODY;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            if (x[k] == NOBODY)
                continue;
            const u32 who = x[k] & 0xFFFFu;
            s_rank[who] = (u16)(x[k] >> 16);
            if (!(end[k] & 0x10000u)) {
                s_member[to[k]] = (u16)who;
                s_end[to[k]] = (u16)end[k];
            }
        }
        const u32 left = s_tied[0];
        if (t < 2)
            a.counters[2 * (g + 1) + t] = s_tied[t];
        if (left == 0)
            break;
    }
}

} // namespace csa
