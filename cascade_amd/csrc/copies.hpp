// The end of a sort whose groups are short: ties that come from copied passages are settled by where the copies end, all generations
// at once and without ranks.
//
// Two suffixes that are tied on ctx symbols and belong to copies of one passage stay tied for as long as the copies agree, and so do the
// suffixes after them: what a position of the copy differs by, and where, is the same for all positions before it. Prefix doubling finds
// that out in log2(length) generations, each of which gathers a rank (a line of 128 bytes) for every suffix that is still tied, and
// needs the ranks of all n suffixes by text position in the first place. Here every member y of a group is compared with one of them, the
// group's root (its member that comes first in the text), and the comparison is made once for a whole passage:
//   anchors   text positions that are multiples of A (a power of two, A <= ctx); an anchor that is a member of a group, and not its root,
//             has a record of that root;
//   links     anchor i is linked to i + 1 if the root of i + 1 is that of i, A symbols on: both pairs belong to the same two copies;
//   ends      an anchor that is not linked compares the text behind its ctx symbols with its root's, until they differ (how far on,
//             and which way) or an anchor further on shows the same two copies again (then its record is open: it says how far they
//             agree at least);
//   spread    a linked anchor gets what the end of its chain of links says (a search for a zero bit, with two levels of summaries
//             above the bits), so that a look at one anchor's record is all that is left to a member.
// A group is put in order by how its members agree with the root: those smaller than the root by rising agreement, the root, those larger by
// falling agreement; members that agree with the root for equally long are told apart by their next symbol, and by a comparison
// of their own past that. The agreement of neighbours gives the generation in which the doubling would have told them apart, and
// with it the sizes of its lists.
// Every comparison has a limit; a group that runs into it, or is longer than SETTLE_MAX, raises a flag, and the sort goes on by doubling from
// where it was. All that has changed by then is the order inside the groups of tiles that were settled: a tile with a comparison that came
// to nothing writes none of its groups. (Comparisons that did and places in the list where they did not are no order together:
// with y before x by the text, x before z and z before y by their places, all three would go to one place.)
#pragma once

#include "device_utils.hpp"
#include "packed_text.hpp"

namespace csa {

// Small tiles, whose waves wait for few others at the barriers, as far as the SETTLE_MAX places behind a tile, which it reads as well, allow (ms of 108 M members of
// 4e8 letters / of 2^28 tokens' copies: 512 x 4 members 5.12 / 0.42, 256 x 4 4.81 / 0.39, 256 x 3 4.56 / 0.35, 128 x 8 5.54 / 0.44). Groups of up to
// SETTLE_MAX_WORDS take the largest block, which settles the longest of them (10^8 letters: 256 x 4 1.18, 512 x 4 0.95, 1024 x 2 0.67).
constexpr int SETTLE_BLOCK = 256, SETTLE_ITEMS = 3;
constexpr int SETTLE_WORDS_BLOCK = 1024, SETTLE_WORDS_ITEMS = 2;
constexpr int SETTLE_MAX = 256; // longest group ...
// ... and of lists that are tied on two words of written text, where one phrase may come a thousand times (5 * 10^7 symbols: 434 times on 24
// letters, the next longest group has 55 members).
constexpr int SETTLE_MAX_WORDS = 2048;
constexpr u32 SETTLE_CONTEXTS = 40;  // contexts of the doubling from here on
constexpr u32 SETTLE_SLOTS = 16;     // copies of the counters, so that the workgroups' additions do not queue on one address
// A record: root << 32 | agreement past the anchor << 1 | the member is the larger one; with OPEN the agreement is that long at least.
constexpr u64 NO_RECORD = ~0ull, OPEN = 1ull << 63; // (positions are below 2^31)
#ifndef CSA_SETTLE_ENDS
#define CSA_SETTLE_ENDS 16
#endif
constexpr u32 SETTLE_ENDS = CSA_SETTLE_ENDS; // anchors that an end looks ahead
#ifndef CSA_SETTLE_STEPS
#define CSA_SETTLE_STEPS 32
#endif
// Steps (records, and stretches between anchors) of a member's comparison with its root, and of its comparisons with the members of its
// key past the first two of each, together. Texts with copies take 13 at most (4e8 letters, a fifth of them copies), and groups of 250
// members, a hundred of which go on alike, one or two a comparison. Passages whose anchors say little take as many as they are long: ms a
// sort with 256 steps for every comparison, with these limits, and doubled: 12437 symbols, 125 steps, 1.97, 0.63, 0.52; 2.9 M symbols, 187
// steps, 4.0, 1.3, 1.1; a group of 250, 20 steps a comparison, 174304 symbols, 8.5, 2.0, 1.1, and worse the longer the passage.
constexpr u32 SETTLE_STEPS = CSA_SETTLE_STEPS;
constexpr int LINK_TILE = 64 * 64;           // anchors of a workgroup of the link kernel: one word of the first summary

struct SettleArgs {
    const u16* text;
    u32 n;
    u32 ctx;      // symbols that the members of a group are tied on
    u32 log2_gap; // anchors are 1 << log2_gap <= ctx symbols apart
    u32 anchors;  // n >> log2_gap, and one more
    const u32* sufs; // the active list, its groups and where they start in it and in the suffix array
    const u32* gids;
    const u32* gstart;
    const u32* gprim;
    u32 m, groups;
    u32 most;     // members of a group: SETTLE_MAX or SETTLE_MAX_WORDS
    const u32* stream; // null, or the codes of the symbols (packed_text.hpp), the bits of one, and of as many as 64 bits hold
    u32 sym_bits, word_bits;
    u64* records; // [anchors + 1], NO_RECORD
    unsigned long long* links[3]; // bits of the anchors, of the words of links[0] that are all ones, of those of links[1]
    u32 words[3];
    u32* sa32;
    u32 contexts[SETTLE_CONTEXTS]; // of the doubling, rising; [0] = ctx
    u32 num_contexts;
    // [SETTLE_SLOTS][2 * (SETTLE_CONTEXTS + 1)], zeroed: of the members, the number of contexts on which each is tied (with either neighbour);
    // of the places where groups of the doubling's lists start, +1 at the first context that has the group and -1 behind the last
    u32* tallies;
    u32* failed;
    u32* err;
};

struct Agreement {
    u32 length; // symbols
    bool larger; // the suffix further on in the text is the larger one
    bool found;
};

// Symbols [from, to) of suffixes r < y, tied on all before: how far they agree, whether that is short of `to`, and if so which
// is larger. The shorter one, y, is smaller if it is a prefix of the other. Reads eight symbols of each at a time where the text has them.
__device__ __forceinline__ bool differ_within(const u16* __restrict__ text, u32 n, u32 r, u32 y, u32 from, u32 to, Agreement& out)
{
    u64 off = from;
    while (off < to) {
        if ((u64)y + off + 8 <= n) {
            u64 a[2], b[2];
            __builtin_memcpy(a, text + (u64)r + off, 16);
            __builtin_memcpy(b, text + (u64)y + off, 16);
            const u64 d0 = a[0] ^ b[0], d1 = a[1] ^ b[1];
            if ((d0 | d1) == 0) {
                off += 8;
                continue;
            }
            off += d0 ? (u32)__builtin_ctzll(d0) / 16u : 4u + (u32)__builtin_ctzll(d1) / 16u;
            break;
        }
        if ((u64)y + off >= n || text[(u64)r + off] != text[(u64)y + off])
            break;
        ++off;
    }
    if (off >= to)
        return false;
    out.length = (u32)off;
    out.larger = (u64)y + off < n && text[(u64)y + off] > text[(u64)r + off];
    out.found = true;
    return true;
}

// The same from the stream, where there is one: as many symbols at a time as 64 bits hold, 32 of four letters, and an eighth of the memory.
__device__ __forceinline__ bool differ_within_stream(const SettleArgs& a, u32 r, u32 y, u32 from, u32 to, Agreement& out)
{
    const u32 syms = a.word_bits / a.sym_bits, room = a.n - y; // (y < n; zeros follow the text)
    u64 off = from;
    bool larger = false;
    for (; off < to && off < room; off += syms) {
        const u64 of_r = packed_window(a.stream, (r + off) * a.sym_bits, a.word_bits), of_y = packed_window(a.stream, (y + off) * a.sym_bits, a.word_bits);
        if (of_r != of_y) {
            off += ((u32)__builtin_clzll(of_r ^ of_y) - (64u - a.word_bits)) / a.sym_bits;
            larger = of_y > of_r;
            break;
        }
    }
    if (off >= room) {
        off = room;
        larger = false;
    }
    if (off >= to)
        return false;
    out.length = (u32)off;
    out.larger = larger;
    out.found = true;
    return true;
}

template <bool STREAM> __device__ __forceinline__ bool differ_within(const SettleArgs& a, u32 r, u32 y, u32 from, u32 to, Agreement& out)
{
    if constexpr (STREAM)
        return differ_within_stream(a, r, y, from, to, out);
    else
        return differ_within(a.text, a.n, r, y, from, to, out);
}

// The first anchor at or after i that is not linked to the next (the last anchor never is).
__device__ __forceinline__ u32 chain_end(const SettleArgs& a, u32 i)
{
    u64 open = ~a.links[0][i / 64] >> (i & 63u);
    if (open)
        return i + (u32)__builtin_ctzll(open);
    u32 w[3] = {i / 64 + 1, 0, 0}; // the word of each level that is looked at next
    // up: until a level has a zero bit at or after the place
    int level = 0;
    while (level < 2) {
        if (w[level] >= a.words[level])
            return a.anchors - 1;
        ++level;
        const u32 at = w[level - 1];
        w[level] = at / 64;
        open = w[level] < a.words[level] ? ~a.links[level][w[level]] >> (at & 63u) : ~0ull;
        if (open) {
            w[level - 1] = at + (u32)__builtin_ctzll(open);
            break;
        }
        ++w[level];
        if (level == 2) {
            while (w[2] < a.words[2] && a.links[2][w[2]] == ~0ull)
                ++w[2];
            if (w[2] >= a.words[2])
                return a.anchors - 1;
            w[1] = w[2] * 64 + (u32)__builtin_ctzll(~a.links[2][w[2]]);
        }
    }
    // down: w[level - 1] is a word of the level below that has a zero bit
    for (int l = level - 1; l >= 0; --l) {
        if (w[l] >= a.words[l])
            return a.anchors - 1;
        const u32 bit = w[l] * 64 + (u32)__builtin_ctzll(~a.links[l][w[l]]);
        if (l == 0)
            return bit;
        w[l - 1] = bit;
    }
    return a.anchors - 1;
}

__device__ __forceinline__ u32 root_of(u64 record) { return (u32)(record >> 32) & 0x7FFFFFFFu; }
__device__ __forceinline__ u32 length_of(u64 record) { return (u32)record >> 1; }

// The last anchor up to which suffix y is known to agree with whoever shares its group (at y or after it: ctx >= gap).
__device__ __forceinline__ u32 first_anchor(const SettleArgs& a, u32 y)
{
    const u64 reach = (u64)y + a.ctx;
    return (u32)((reach < a.n ? reach : (u64)a.n) >> a.log2_gap);
}

// How far suffixes r < y agree, which are tied on their first `tied` >= ctx symbols; takes its steps from steps_left.
template <bool STREAM>
__device__ __forceinline__ Agreement agreement(const SettleArgs& a, u32 r, u32 y, u32 tied, u32& steps_left)
{
    Agreement out = {tied, false, false};
    u64 off = tied;
    const u32 gap = 1u << a.log2_gap;
    while (steps_left > 0) {
        --steps_left;
        const u64 reach = (u64)y + off;
        const u32 i = (u32)((reach < a.n ? reach : (u64)a.n) >> a.log2_gap); // the last anchor up to which they are known to agree
        u32 shift = (i << a.log2_gap) - y;                                  // (tied >= ctx >= gap: it lies at y or after it)
        u64 of_y = a.records[i];
        if (of_y != NO_RECORD && root_of(of_y) == r + shift) {
            out.length = shift + length_of(of_y);
            if (!(of_y & OPEN)) {
                out.larger = (of_y & 1u) != 0;
                out.found = true;
                return out;
            }
            off = out.length; // (two anchors past this one at least)
            continue;
        }
        // A third copy, further to the front: y agrees with it that far from this anchor on; does r, from its own next anchor on? (r and y must be
        // known to agree up to there; else from the anchor before.)
        const u32 d = (0u - (r + shift)) & (gap - 1u);
        if (shift + d > off) {
            of_y = shift >= gap ? a.records[i - 1] : NO_RECORD;
            shift -= gap;
        }
        if (of_y != NO_RECORD) {
            const u64 of_r = a.records[(r + shift + d) >> a.log2_gap];
            if (of_r != NO_RECORD && root_of(of_r) == root_of(of_y) + d) {
                const u32 y_len = length_of(of_y), r_len = d + length_of(of_r);
                if (y_len < r_len && !(of_y & OPEN)) {
                    out.length = shift + y_len;
                    out.larger = (of_y & 1u) != 0;
                    out.found = true;
                    return out;
                }
                if (r_len < y_len && !(of_r & OPEN)) {
                    out.length = shift + r_len;
                    out.larger = (of_r & 1u) == 0;
                    out.found = true;
                    return out;
                }
                const u64 both = (u64)shift + (y_len < r_len ? y_len : r_len);
                off = both > off ? both : off;
            }
        }
        if (differ_within<STREAM>(a, r, y, (u32)off, (u32)off + gap, out))
            return out;
        off += gap;
    }
    return out;
}

// The records of the anchors among the members of groups: their roots.
__global__ __launch_bounds__(256) void copy_roots_kernel(SettleArgs a)
{
    const u64 e = (u64)blockIdx.x * 256 + threadIdx.x;
    if (e >= a.m)
        return;
    const u32 x = a.sufs[e];
    if (x & ((1u << a.log2_gap) - 1u))
        return;
    const u32 g = a.gids[e];
    if (g >= a.groups || x >= a.n) {
        atomicExch(a.err, DEV_ERR_SMALLSORT_TABLES);
        return;
    }
    const u32 from = a.gstart[g], to = a.gstart[g + 1];
    if (to - from > a.most || to > a.m) {
        *a.failed = 1u;
        return;
    }
    u32 root = x;
    for (u32 i = from; i < to; ++i) {
        const u32 y = a.sufs[i];
        root = y < root ? y : root;
    }
    if (root != x)
        a.records[x >> a.log2_gap] = (u64)root << 32;
}

// links[0], links[1] and the ends. Bounded by reading the records once; the anchors that are not linked are few.
template <bool STREAM>
__global__ __launch_bounds__(1024) void copy_links_kernel(SettleArgs a)
{
    __shared__ unsigned long long s_word[LINK_TILE / 64];
    const u32 t = threadIdx.x, gap = 1u << a.log2_gap;
    const u32 first = blockIdx.x * LINK_TILE;
    if (*a.failed) // (set by the kernel before, if at all)
        return;
    for (u32 k = 0; k < LINK_TILE; k += 1024) {
        const u32 i = first + k + t;
        // (an end only ever changes the lower half of a record, so the roots can be read meanwhile)
        const u64 record = i < a.anchors ? a.records[i] : NO_RECORD; // (records[anchors] is there, and NO_RECORD)
        const u32 root = root_of(record);
        const bool copied = record != NO_RECORD, linked = copied && a.records[i + 1] != NO_RECORD && root_of(a.records[i + 1]) == root + gap;
        const u64 b = __ballot(linked);
        if ((t & 63u) == 0) {
            s_word[(k + t) / 64] = b;
            if (i / 64 < a.words[0])
                a.links[0][i / 64] = b;
        }
        if (copied && !linked) {
            const u32 y = i << a.log2_gap;
            Agreement out = {0u, false, false};
            u32 from = a.ctx, known = SETTLE_ENDS << a.log2_gap;
            for (u32 skip = 2; skip <= SETTLE_ENDS; ++skip) {
                const u32 to = skip << a.log2_gap;
                if (from < to) {
                    if (differ_within<STREAM>(a, root, y, from, to, out))
                        break;
                    from = to;
                }
                if (i + skip < a.anchors && a.records[i + skip] != NO_RECORD && root_of(a.records[i + skip]) == root + to) {
                    known = to;
                    break;
                }
            }
            if (out.found)
                reinterpret_cast<u32*>(a.records)[2ull * i] = out.length << 1 | (out.larger ? 1u : 0u);
            else {
                reinterpret_cast<u32*>(a.records)[2ull * i] = (known > a.ctx ? known : a.ctx) << 1;
                reinterpret_cast<u32*>(a.records)[2ull * i + 1] = root | 0x80000000u;
            }
        }
    }
    __syncthreads();
    if (t < 64) {
        const u64 b = __ballot(s_word[t] == ~0ull);
        if (t == 0)
            a.links[1][blockIdx.x] = b;
    }
}

__global__ __launch_bounds__(256) void copy_links_top_kernel(SettleArgs a)
{
    const u32 w = blockIdx.x * 256 + threadIdx.x;
    const u64 b = __ballot(w < a.words[1] && a.links[1][w] == ~0ull);
    if ((threadIdx.x & 63u) == 0 && w / 64 < a.words[2])
        a.links[2][w / 64] = b;
}

// The linked anchors' records: what the ends of their chains say. (The records of ends are not changed here.)
__global__ __launch_bounds__(256) void copy_spread_kernel(SettleArgs a)
{
    const u32 i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.anchors || *a.failed || !((a.links[0][i / 64] >> (i & 63u)) & 1ull))
        return;
    const u32 end = chain_end(a, i);
    const u64 record = a.records[end];
    const u32 length = length_of(record) + ((end - i) << a.log2_gap);
    reinterpret_cast<u32*>(a.records)[2ull * i] = length << 1 | ((u32)record & 1u);
    if (record & OPEN)
        reinterpret_cast<u32*>(a.records)[2ull * i + 1] |= 0x80000000u;
}

// The members of every group in order, to their places in the suffix array, and the tallies. A tile settles the groups that start in it.
// What bounds it is the random read of a member: its anchor's record. (1e9 Zipf tokens with 6 % of their documents copied, 55.7 M members
// tied on 8 symbols: 1.5 ms here, 1.1 for the records, where the update of 1e9 ranks took 10.5 and ten generations 9.8.)
template <int BLOCK, int PER, int MAXG, bool STREAM>
__global__ __launch_bounds__(BLOCK) void settle_groups_kernel(SettleArgs a)
{
    constexpr int TILE = BLOCK * PER, SPAN = TILE + MAXG, ITEMS = (SPAN + BLOCK - 1) / BLOCK;
    constexpr u32 TALLIES = 2 * (SETTLE_CONTEXTS + 1), COPIES = 4;
    __shared__ u64 s_key[SPAN];
    // Of groups that may be long, the word of nine to twelve symbols after those in the key: members that are told from their root in the same way are told apart
    // by it as a rule. (10^8 letters, 1.8 ms of the kernel in one tile with a
    // group of a thousand, when all such pairs were compared by the text or by four symbols more; 1.0 with the word.)
    constexpr bool MORE = MAXG > SETTLE_MAX;
    static_assert(STREAM || !MORE, "the words are those of the stream");
    __shared__ u64 s_more[MORE ? SPAN : 1];
    __shared__ u32 s_suf[SPAN];
    __shared__ u32 s_tally[TALLIES * COPIES];
    __shared__ u16 s_queue[SPAN];
    __shared__ u32 s_queued;
    __shared__ u32 s_over;   // a tile before has given up
    __shared__ u32 s_lost[2]; // some member of the tile could not be compared with its root; two members with each other
    const u32 t = threadIdx.x;
    for (u32 i = t; i < TALLIES * COPIES; i += BLOCK)
        s_tally[i] = 0;
    if (t == 0) {
        // (An atomic load: a plain one of this address comes from the scalar cache, where a word that other tiles write stays as it was for the whole kernel. 3 * 10^7
        // letters of passages and their copies, 27.3 -> 20.3 ms: every tile did all of its work. 4 * 10^8 letters that are settled: 17.5 -> 17.6.
        // The load stays in front of the others: a build that looked at the flag just before the barrier put some 90 of 4 * 10^8 suffixes in wrong places in every sort,
        // other ones each time, for no reason that was found in the source or in the assembly.)
        s_over = dev_failed(a.failed) ? 1u : 0u;
        s_lost[0] = s_lost[1] = s_queued = 0;
    }
    const u64 t0 = (u64)blockIdx.x * TILE;
    u32 x[ITEMS], place[ITEMS];
    int from[ITEMS], to[ITEMS]; // the group, by places of the span; to = 0: nothing to do
    u32 prim[ITEMS];
    u64 key[ITEMS] = {}, more[MORE ? ITEMS : 1] = {};
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const u32 j = k * BLOCK + t;
        const u64 e = t0 + j;
        x[k] = 0;
        from[k] = to[k] = 0;
        prim[k] = 0;
        if (e >= a.m || j >= (u32)SPAN)
            continue;
        x[k] = a.sufs[e];
        s_suf[j] = x[k];
        const u32 g = a.gids[e];
        if (g >= a.groups) {
            atomicExch(a.err, DEV_ERR_SMALLSORT_TABLES);
            continue;
        }
        const u32 gs = a.gstart[g], ge = a.gstart[g + 1];
        if (gs < t0 || gs >= t0 + TILE)
            continue; // another tile's
        if (gs > e || ge <= e || ge > a.m || ge - gs > (u32)MAXG) {
            __hip_atomic_store(a.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            continue;
        }
        from[k] = (int)(gs - t0);
        to[k] = (int)(ge - t0);
        prim[k] = a.gprim[g];
        if (prim[k] >= a.n || prim[k] + (ge - gs) > a.n) {
            atomicExch(a.err, DEV_ERR_RERANK_RANGE);
            to[k] = 0;
        }
    }
    __syncthreads();
    if (s_over)
        return;
    // A member's key: which side of the root it is on, how far it agrees with it (the closer the longer), the symbol after that (0: none).
    // 2 + 31 + 17 bits.
    constexpr u64 ROOT = 1ull << 48, LARGER = 2ull << 48, FAR = 0x7FFFFFFFull;
    auto agreement_of = [](u64 w) -> u32 { // of a member with its root
        const u32 v = (u32)(w >> 17) & (u32)FAR;
        return (w >> 48) == 0 ? v : (w >> 48) == 1 ? (u32)FAR : (u32)FAR - v;
    };
    volatile u32* const lost = s_lost;
    auto put_key = [&](u32 j, u32 y, bool alone, const Agreement& w) { // (alone: one of a pair has nobody else to be told from)
        const u64 next = (u64)y + w.length;
        const u64 symbol = alone || next >= a.n ? 0u : (STREAM ? packed_window(a.stream, next * a.sym_bits, a.sym_bits) : (u64)a.text[next]) + 1u;
        s_key[j] = w.larger ? LARGER | ((FAR - w.length) << 17) | symbol : ((u64)w.length << 17) | symbol;
        if constexpr (MORE)
            s_more[j] = symbol && next + 1 < a.n ? packed_window(a.stream, (next + 1) * a.sym_bits, a.word_bits) : 0u;
    };
    // Most members' first record tells. Those whose does not are queued, and take their steps side by side: a wave would wait for the one
    // lane in each item that takes the most. (4e8 letters, 108 M members, every member at its item: 6.57 ms; queued
    // 5.92; and what the records leave open read from the stream of codes, 100 MB that stay in the cache, instead of the text: 5.12.)
    u32 root[ITEMS];
    u64 first[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        root[k] = x[k];
        first[k] = NO_RECORD;
        if (to[k] == 0)
            continue;
        for (int i = from[k]; i < to[k]; ++i)
            root[k] = s_suf[i] < root[k] ? s_suf[i] : root[k];
        if (root[k] != x[k])
            first[k] = a.records[first_anchor(a, x[k])];
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        if (to[k] == 0)
            continue;
        const u32 j = k * BLOCK + t, shift = (first_anchor(a, x[k]) << a.log2_gap) - x[k];
        if (root[k] == x[k]) {
            s_key[j] = ROOT;
            if constexpr (MORE)
                s_more[j] = 0;
        } else if (first[k] != NO_RECORD && root_of(first[k]) == root[k] + shift && !(first[k] & OPEN)) {
            put_key(j, x[k], to[k] - from[k] == 2, Agreement{shift + length_of(first[k]), (first[k] & 1u) != 0, true});
        } else {
            s_queue[atomicAdd(&s_queued, 1u)] = (u16)j;
            s_key[j] = (u64)root[k] << 1 | (to[k] - from[k] == 2 ? 1u : 0u);
        }
    }
    __syncthreads();
    for (u32 q = t; q < s_queued && !lost[0]; q += BLOCK) { // (a tile that has lost a member writes nothing)
        const u32 j = s_queue[q], y = s_suf[j];
        u32 steps_left = SETTLE_STEPS;
        const Agreement w = agreement<STREAM>(a, (u32)(s_key[j] >> 1), y, a.ctx, steps_left);
        if (!w.found)
            lost[0] = 1u;
        else
            put_key(j, y, (s_key[j] & 1u) != 0, w);
    }
    __syncthreads();
    if (s_lost[0]) {
        if (t == 0)
            __hip_atomic_store(a.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k)
        if (to[k] != 0) {
            key[k] = s_key[k * BLOCK + t];
            if constexpr (MORE)
                more[k] = s_more[k * BLOCK + t];
        }
    // does suffix y go before suffix z of the same key: their agreement from the symbol after the one that tells them from their root
    // (more_left: steps that comparisons may take past their first two)
    auto further = [&](u32 y, u32 z, u64 w, u32& more_left) -> Agreement {
        const u32 r = y < z ? y : z, o = y < z ? z : y;
        u32 steps_left = more_left + 2u, tied = agreement_of(w) + 1u;
        if constexpr (MORE) // (they share the word behind it, too, and where that is inside the text its symbols)
            tied += (u64)o + tied + a.word_bits / a.sym_bits <= a.n ? a.word_bits / a.sym_bits : 0u;
        const Agreement v = agreement<STREAM>(a, r, o, tied, steps_left);
        more_left = steps_left < more_left ? steps_left : more_left;
        return v;
    };
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        place[k] = (u32)(k * BLOCK) + t;
        if (to[k] == 0)
            continue;
        const int j = k * BLOCK + (int)t;
        u32 before = 0, more_left = SETTLE_STEPS;
        for (int i = from[k]; i < to[k]; ++i) {
            const u64 w = s_key[i];
            bool smaller = w < key[k], same = w == key[k];
            if constexpr (MORE)
                if (same) {
                    smaller = s_more[i] < more[k];
                    same = s_more[i] == more[k];
                }
            if (smaller) {
                ++before;
            } else if (same && i != j) {
                if (lost[1])
                    break;
                const u32 y = s_suf[i];
                const Agreement v = further(x[k], y, w, more_left);
                if (!v.found)
                    lost[1] = 1u;
                before += (y < x[k]) == v.larger ? 1u : 0u;
            }
        }
        place[k] = (u32)from[k] + before;
    }
    __syncthreads();
    if (s_lost[1]) { // (the same for all threads: nobody sets it past the barrier)
        if (t == 0)
            __hip_atomic_store(a.failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k)
        if (to[k] != 0) {
            s_suf[place[k]] = x[k];
            s_key[place[k]] = key[k];
            if constexpr (MORE)
                s_more[place[k]] = more[k];
        }
    __syncthreads();
    // the thread's places from here on: who stands there now, and on how many contexts it is tied with its neighbours
    auto contexts_of = [&](int right) -> u32 { // of places right - 1 and right of one group
        const u64 v = s_key[right - 1], w = s_key[right];
        const u32 y = s_suf[right - 1], z = s_suf[right];
        const u32 of_v = agreement_of(v), of_w = agreement_of(w);
        u32 agree = of_v < of_w ? of_v : of_w;
        const u64 differ = MORE && v == w ? s_more[MORE ? right - 1 : 0] ^ s_more[MORE ? right : 0] : 0u;
        if (differ) {
            agree = of_w + 1u + ((u32)__builtin_clzll(differ) - (64u - a.word_bits)) / a.sym_bits;
        } else if (v == w) {
            u32 more_left = SETTLE_STEPS; // (enough: the two have been compared before)
            agree = further(y, z, w, more_left).length;
        }
        const u32 room = a.n - 1u - (y > z ? y : z); // (whoever runs off the text within a context is tied with nobody on it)
        agree = agree < room ? agree : room;
        u32 c = 0;
        while (c < a.num_contexts && agree >= a.contexts[c])
            ++c;
        return c;
    };
    u32* const mine = s_tally + TALLIES * (t & (COPIES - 1));
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        if (to[k] == 0)
            continue;
        const int j = k * BLOCK + (int)t;
        const u32 left = j > from[k] ? contexts_of(j) : 0u, right = j + 1 < to[k] ? contexts_of(j + 1) : 0u;
        atomicAdd(&mine[left > right ? left : right], 1u);
        if (right > left) {
            atomicAdd(&mine[SETTLE_CONTEXTS + 1 + left], 1u);
            atomicAdd(&mine[SETTLE_CONTEXTS + 1 + right], 0xFFFFFFFFu);
        }
        a.sa32[prim[k] + (u32)(j - from[k])] = s_suf[j];
    }
    __syncthreads();
    for (u32 i = t; i < TALLIES; i += BLOCK) {
        u32 v = 0;
#pragma unroll
        for (u32 c = 0; c < COPIES; ++c)
            v += s_tally[c * TALLIES + i];
        if (v)
            atomicAdd(&a.tallies[(u64)(blockIdx.x % SETTLE_SLOTS) * TALLIES + i], v);
    }
}

} // namespace csa
