// The end of a sort whose list is runs and periods: groups whose members stand in it at equal distances in the text.
//
// The suffixes of a run of one token (or of a stretch of period d) that are tied on ctx symbols are x, x + d, x + 2 d, ..., up to a last
// one. Where that one and the one before it differ, L symbols on, every member differs from the next: x and x + d agree on
// all symbols up to there, so the closer to the end, the shorter the tie, and all comparisons come out the same way. The group in
// order is the group by text position, forwards or backwards, and when the doubling would have let each member go follows from L. The
// doubling itself needs log2(length) generations for it, each of which retires no more suffixes than it looks ahead: 2^26 symbols,
// 10.5 M of them in a run and a stretch of period 7, spent 18 generations of
// 0.37 ms on a list that hardly got shorter (the whole sort 11.5 ms; 6.3 with 0.06 ms here).
// Since the last member + d is not in the group, L < ctx + d (or the text ends before that): one short comparison per group.
// A list with any other group in it goes on by doubling.
#pragma once

#include "copies.hpp"

namespace csa {

constexpr u32 CHAIN_STEP_MAX = 1024; // longest period (the comparison is one thread's)
constexpr u32 CHAIN_TALLIES = 4;     // of each context: members, groups, members of groups longer than limit_lo, than limit_hi

struct ChainArgs {
    const u16* text;
    u32 n;
    u32 ctx; // symbols that the members of a group are tied on
    const u32* sufs; // the active list, its groups and where they start in it and in the suffix array
    const u32* gids;
    const u32* gstart;
    const u32* gprim;
    u32 m, groups;
    u32* sa32;
    u32* backwards; // [groups]: the order of the group is that of the list reversed
    u32 limit_lo, limit_hi;
    u32 contexts[SETTLE_CONTEXTS]; // of the doubling, rising; [0] = ctx
    u32 num_contexts;
    u32* tallies; // [SETTLE_CONTEXTS][CHAIN_TALLIES], zeroed
    u32* failed;  // zeroed
    u32* err;
};

__global__ __launch_bounds__(256) void chain_groups_kernel(ChainArgs a)
{
    __shared__ u32 s_tally[SETTLE_CONTEXTS * CHAIN_TALLIES];
    const u32 t = threadIdx.x;
    for (u32 i = t; i < SETTLE_CONTEXTS * CHAIN_TALLIES; i += 256)
        s_tally[i] = 0;
    __syncthreads();
    const u32 g = blockIdx.x * 256 + t;
    if (g < a.groups) {
        const u32 from = a.gstart[g], to = a.gstart[g + 1];
        bool chain = false;
        if (to > a.m || from >= to || to - from < 2) {
            atomicExch(a.err, DEV_ERR_SMALLSORT_TABLES);
        } else {
            const u32 size = to - from, x0 = a.sufs[from], x1 = a.sufs[from + 1], xl = a.sufs[to - 1];
            const u32 d = x1 > x0 ? x1 - x0 : x0 - x1, last = x0 > xl ? x0 : xl, first = x0 > xl ? xl : x0;
            chain = d != 0 && d <= a.ctx && d <= CHAIN_STEP_MAX && (u64)first + (u64)d * (size - 1) == last && (x1 > x0) == (xl > x0);
            Agreement end = {0u, false, false};
            chain = chain && differ_within(a.text, a.n, last - d, last, a.ctx, a.ctx + d + 1, end);
            if (chain) {
                a.backwards[g] = end.larger == (x1 > x0) ? 0u : 1u;
                for (u32 c = 0; c < a.num_contexts; ++c) {
                    // pair j counts from the end: it agrees on L + j d symbols, its later member must not run off the text inside the context
                    const u64 ctx = a.contexts[c];
                    u64 j = ctx > end.length ? (ctx - end.length + d - 1) / d : 0;
                    if (last + ctx >= a.n) {
                        const u64 inside = (last + ctx - a.n) / d + 1;
                        j = inside > j ? inside : j;
                    }
                    if (j >= size - 1)
                        break;
                    const u32 members = size - (u32)j;
                    atomicAdd(&s_tally[c * CHAIN_TALLIES + 0], members);
                    atomicAdd(&s_tally[c * CHAIN_TALLIES + 1], 1u);
                    if (members > a.limit_lo)
                        atomicAdd(&s_tally[c * CHAIN_TALLIES + 2], members);
                    if (members > a.limit_hi)
                        atomicAdd(&s_tally[c * CHAIN_TALLIES + 3], members);
                }
            }
        }
        if (!chain)
            *a.failed = 1u;
    }
    __syncthreads();
    for (u32 i = t; i < SETTLE_CONTEXTS * CHAIN_TALLIES; i += 256)
        if (s_tally[i])
            atomicAdd(&a.tallies[i], s_tally[i]);
}

// The members to their places. Bounded by reading the list (8 bytes a member) and writing the places in it.
__global__ __launch_bounds__(256) void chain_place_kernel(ChainArgs a)
{
    const u64 e = (u64)blockIdx.x * 256 + threadIdx.x;
    if (e >= a.m || *a.failed)
        return;
    const u32 g = a.gids[e];
    if (g >= a.groups) {
        atomicExch(a.err, DEV_ERR_SMALLSORT_TABLES);
        return;
    }
    const u32 from = a.gstart[g], to = a.gstart[g + 1], x = a.sufs[e];
    if (e < from || e >= to) {
        atomicExch(a.err, DEV_ERR_SMALLSORT_TABLES);
        return;
    }
    const u32 j = (u32)e - from;
    // all of the group at the distance of its first two, and they do not wrap around (its ends were looked at)
    if (x != a.sufs[from] + j * (a.sufs[from + 1] - a.sufs[from])) {
        *a.failed = 1u; // (what has been written are places of this list's members: each is written again when it retires)
        return;
    }
    const u64 place = (u64)a.gprim[g] + (a.backwards[g] ? to - 1 - from - j : j);
    if (place >= a.n) {
        atomicExch(a.err, DEV_ERR_RERANK_RANGE);
        return;
    }
    a.sa32[place] = x;
}

} // namespace csa
