// Texts over 17 to 128 symbols (written text): the first sort on 64 bits of the code stream, and on 64 more where those tie.
//
// A symbol takes b = 5 to 7 bits of the stream (packed_text.hpp has codes of a power of two), a word is the L = 64 / b symbols that fit 64 bits: twelve letters.
// Written text takes about two bits a letter to tell apart, so eight letters leave nine suffixes in ten tied, twelve six in ten and 24 the
// copies. After the passes over the first words, resolve_words_kernel reads the second word of every suffix that shares its first (a line of the
// stream), puts runs of up to WORDS_MAX suffixes in order inside its tile and counts, from the words, on how many of the doubling's contexts neighbours
// tie; longer runs are collected and radix sorted by the second word. What is left are copies as a rule, and settled as such (copies.hpp). The generations that
// this stands for used to gather a rank for every tied suffix: 10^8 symbols of text 15.2 -> 9.6 ms. (Words of 56 bits take a pass less: independent letters 4 to 11 % faster, but such
// a text then has more than three members to a group left, which are not settled: 15.2 ms.)
#pragma once

#include "coded_keys.hpp"
#include "copies.hpp"
#include "device_utils.hpp"
#include "doubling.hpp"
#include "packed_text.hpp"

namespace csa {

constexpr u32 WORD_LEVELS = 4; // contexts that a list is counted on, the two words among them

struct WordLevels {
    u32 count;
    u32 in_first;               // of them, those inside the first word
    u32 context[WORD_LEVELS];   // symbols, rising
    u32 drop[WORD_LEVELS];      // bits of a word (the first one; the second for contexts past it) behind the context
};

// ---- the stream, and the digit counts of the passes over its words ----

constexpr int WORD_BLOCK = 256;
constexpr u32 WORD_SPAN = 256;      // words of a workgroup's stretch

// stream[wd], wd < words: bits 32 wd .. of the codes of all symbols, `bits` each, zero past the text. Sets the counts of windows to zero.
__global__ __launch_bounds__(WORD_BLOCK) void encode_words_kernel(const u16* __restrict__ text, u32 n, SymbolCodes codes, u32* __restrict__ stream, u64 words, u32* __restrict__ windows, u32 bins)
{
    constexpr u32 MAX_SYMS = WORD_SPAN * 32 / 5 + 8;
    __shared__ u64 s_text[(MAX_SYMS + 6) / 4 + 2];
    __shared__ SymbolCodes s_codes;
    const u32 t = threadIdx.x, b = codes.bits;
    for (u64 i = (u64)blockIdx.x * WORD_BLOCK + t; i < bins; i += (u64)gridDim.x * WORD_BLOCK)
        windows[i] = 0;
    for (u32 i = t; i < sizeof(SymbolCodes) / 4; i += WORD_BLOCK)
        reinterpret_cast<u32*>(&s_codes)[i] = reinterpret_cast<const u32*>(&codes)[i];
    const u64 w0 = (u64)blockIdx.x * WORD_SPAN, first = w0 * 32 / b;
    const u32 sym_off = stage_text(text, n, first, WORD_SPAN * 32 / b + 8u, s_text, t, WORD_BLOCK);
    __syncthreads();
    const u16* const s16 = reinterpret_cast<const u16*>(s_text) + sym_off;
    for (u32 i = t; i < WORD_SPAN; i += WORD_BLOCK) {
        const u64 bit = (w0 + i) * 32, y = bit / b;
        u32 word = 0, s = (u32)(y - first);
        int up = 32 + (int)(bit - y * b) - (int)b; // bits of the word behind the symbol (the first one may start before the word)
        for (; up > -(int)b; up -= (int)b, ++s) {
            const u32 c = symbol_code(s_codes, s16[s]);
            word |= up >= 0 ? c << up : c >> -up;
        }
        if (w0 + i < words)
            stream[w0 + i] = word;
    }
}

// The digits of a word start inside one of its symbols, `bits` places apart at most: all of them are read off one count of the windows of a symbol and the
// seven bits behind the next one's first, which every suffix adds to once (eight digits counted one by one took 0.30 ms of 10^8 symbols, bound by LDS
// atomics; this takes 0.12).
constexpr int WINDOW_BLOCK = 1024;
constexpr u32 WINDOW_HIST_BLOCKS = 256;

template <u32 BITS> constexpr u32 WINDOW_BITS = BITS + 7; // of a symbol, a digit of eight bits from any of its places on

// windows[v] += suffixes whose first WINDOW_BITS bits in the stream are v.
template <u32 BITS>
__global__ __launch_bounds__(WINDOW_BLOCK) void window_hist_kernel(const u32* __restrict__ stream, u32 n, u32* __restrict__ windows)
{
    constexpr u32 BINS = 1u << WINDOW_BITS<BITS>;
    __shared__ u32 s_hist[BINS];
    const u32 t = threadIdx.x;
    for (u32 i = t; i < BINS; i += WINDOW_BLOCK)
        s_hist[i] = 0;
    __syncthreads();
    const u64 stride = (u64)gridDim.x * WINDOW_BLOCK;
    for (u64 x = (u64)blockIdx.x * WINDOW_BLOCK + t; x < n; x += stride)
        atomicAdd(&s_hist[(u32)packed_window(stream, x * BITS, WINDOW_BITS<BITS>)], 1u);
    __syncthreads();
    for (u32 i = t; i < BINS; i += WINDOW_BLOCK)
        if (s_hist[i])
            atomicAdd(&windows[i], s_hist[i]);
}

// ghist[p][d] = suffixes whose word has digit d at bits 8 p .. of the word (the last digit may be shorter), digit_base[p][d] = those with a smaller one: a workgroup a
// digit. Digit p is that of the windows k symbols on, so the first k windows are taken out, and k of zeros, past the text, put in. (What it takes is the latency of its loads: with four
// windows of a thread in flight and the scan in a launch of its own 16 us for symbols of seven bits, 10 now; 2^18 independent letters of 100 247 -> 240 us.)
template <u32 BITS>
__global__ __launch_bounds__(WINDOW_BLOCK) void word_digits_kernel(const u32* __restrict__ stream, const u32* __restrict__ windows, u32 n, u32 word_bits, u32* __restrict__ ghist, u32* __restrict__ digit_base)
{
    __shared__ u32 s_count[RADIX_BINS];
    __shared__ u32 s_wave[RADIX_BINS / WAVE];
    const u32 t = threadIdx.x, p = blockIdx.x, size = word_bits - 8 * p < 8 ? word_bits - 8 * p : 8u;
    const u32 from = word_bits - 8 * p - size, k = from / BITS, r = from - k * BITS; // the digit starts r bits into symbol k
    const u32 below = BITS + 7 - r - size;                                           // bits of a window behind it
    if (t < RADIX_BINS)
        s_count[t] = 0;
    __syncthreads();
    // as many threads a digit as there are: each adds up 2^(BITS - 3) windows
    const u32 d = t & ((1u << size) - 1u), first = t >> size, threads = WINDOW_BLOCK >> size;
    const bool taken_out = t < k && t < n;
    const u32 out = taken_out ? (u32)packed_window(stream, (u64)t * BITS + r, size) : 0u;
    u32 v = 0;
#pragma unroll
    for (u32 i = 0; i < 1u << (BITS - 3); ++i) {
        const u32 j = first + i * threads; // the window's bits before and behind the digit
        v += windows[(j >> below << (below + size)) | (d << below) | (j & ((1u << below) - 1u))];
    }
    if (v)
        atomicAdd(&s_count[d], v);
    if (taken_out) {
        atomicAdd(&s_count[out], ~0u); // (one less)
        atomicAdd(&s_count[0], 1u);
    }
    __syncthreads();
    const u32 count = t < RADIX_BINS ? s_count[t] : 0u, incl = wave_incl_sum(count);
    if (t < RADIX_BINS && (t & 63u) == 63u)
        s_wave[t / WAVE] = incl;
    __syncthreads();
    if (t < RADIX_BINS) {
        u32 before = incl - count;
        for (u32 w = 0; w < t / WAVE; ++w)
            before += s_wave[w];
        ghist[p * RADIX_BINS + t] = count;
        digit_base[p * RADIX_BINS + t] = before;
    }
}

// ---- the second words ----

// Texts that the second word does little for: padding, lines that come again and again, few words. Long runs of one first word are sorted again, to find them
// long and of one second word as well. Looked for at 1024 places of the sorted list, in runs of 256 or more; the runs of a written text grow with it, so from 2^26 symbols on in
// runs of n / 2^18, and in more places, from 26 of them in texts of 2^18 symbols to 220, a quarter of the list less what such a sample is off by: from a quarter on the
// second words are given up (sort_by_words). Such lists are ranked on the doubling's last context inside the first word. (Places, and us with the second words left out / read. Words of 400 to 32000,
// Zipf(1.1), letters alike: 6 * 10^5 symbols 107, 772 / 872, 10^6 99, 818 / 910, 2 * 10^6 129, 919 / 1020, 10^7 233, 2381 / 2584; log lines 10^6 526, 1202 / 1360. Words of which the
// frequent ones are short, with copies, of 28 values 10^6 symbols 1, 755 / 587, 10^7 13, 2025 / 1280; of 100 values 2 * 10^6 21, 709 / 682, 4 * 10^6 36, 923 / 871, 10^7 56, 1805 / 1418, 5 * 10^7 141, 6366 / 5293;
// with runs of spaces 5 * 10^7 190, 9560 / 8609, 252, 10716 / 11515; with a period 238, 9895 / 9030, 1.5 * 10^8 248, 27.8 / 30.1 ms.)
#ifndef CSA_WORD_LONG_FEW
#define CSA_WORD_LONG_FEW 24
#endif
constexpr u32 WORD_PLACES = 1024, WORD_LONG = 256, WORD_LONG_SHIFT = 18, WORD_LONG_FEW = CSA_WORD_LONG_FEW, WORD_LONG_FEW_SHIFT = 17, WORD_LONG_MOST = 220;

// One long run or period is enough for the settling to give up, after it has looked at the period's groups (11 groups of 1818 members, all tied for thousands of
// symbols: 0.4 ms): a region of more than ENDLESS_SYMBOLS symbols and ENDLESS_TIMES periods, or many short ones of one run that make a group of more than
// SETTLE_MAX_WORDS members on both words. A place of the list is in a region if the places behind it with the same first word stand equally far apart in the text, all
// the way. Looked for at 4096 places, by as many workgroups as take 1024 (one of 1024 threads took four times as long, 20 us). Where some are found nothing is settled,
// and in texts of fewer than CSA_WORD_ENDLESS_MIN symbols the second words are left out as well.
constexpr u32 ENDLESS_BLOCKS = 4, ENDLESS_SYMBOLS = 512, ENDLESS_TIMES = 32, PIECES_FEW = 1; // (of 1024 places)

// Places further on in the list that a region of this period is followed to. (Gaps are as long as the text allows: 2^27 symbols and its copy, whose gap times 32 is zero
// in 32 bits, took 194 ms without the settling, 24 with it.)
constexpr u32 endless_places(u32 gap) { return (u64)gap * ENDLESS_TIMES < ENDLESS_SYMBOLS ? (ENDLESS_SYMBOLS + gap - 1) / gap : ENDLESS_TIMES; }
static_assert(endless_places(1) == ENDLESS_SYMBOLS && endless_places(15) == 35 && endless_places(16) == ENDLESS_TIMES && endless_places(1u << 27) == ENDLESS_TIMES
                  && endless_places(31u << 27) == ENDLESS_TIMES, "512 symbols of short periods, 32 of all others");

// Launched before the list is counted, which it says how (rerank_count_kernel). *choice is zero before; the totals of levels are set to zero.
__global__ __launch_bounds__(WORD_PLACES) void choose_seconds_kernel(const u64* __restrict__ keys, const u32* __restrict__ sufs, u32 n, u32 syms, u32 if_endless, u32* choice, unsigned long long* level_totals)
{
    __shared__ u32 s_in[3];
    const u32 t = threadIdx.x, places = gridDim.x * WORD_PLACES, place = t * gridDim.x + blockIdx.x;
    if (t < 3)
        s_in[t] = 0;
    if (place < LEVEL_SLOTS * 8)
        level_totals[place] = 0;
    __syncthreads();
    const u32 is_long = n >> WORD_LONG_SHIFT > WORD_LONG ? n >> WORD_LONG_SHIFT : WORD_LONG;
    const u32 e = (u32)((u64)n * place / places), next = e + 1 < n ? e + 1 : e;
    const u64 key = keys[e];
    const bool equal = keys[next] == key;
    const u32 x = sufs[e], y = sufs[next];
    u32 found[3];
    found[0] = in_long_run(keys, n, is_long, place, places) ? 1u : 0u;
    const u32 gap = y > x ? y - x : 0u; // (members of a run come in text order, but for those that end the text)
    auto goes_on = [&](u32 times) { return (u64)e + times < n && keys[e + times] == key && sufs[e + times] - x == (u64)times * gap; };
    const bool near = equal && gap > 0;
    found[1] = near && goes_on(endless_places(gap)) ? 1u : 0u;
    // (gaps of up to a word: the second words are the same as well)
    found[2] = near && gap <= syms && goes_on(2 * syms / gap) && in_long_run(keys, n, (u32)SETTLE_MAX_WORDS, place, places) ? 1u : 0u;
#pragma unroll
    for (u32 i = 0; i < 3; ++i) {
        const u64 b = __ballot(found[i] != 0);
        if ((t & 63u) == 0 && b)
            atomicAdd(&s_in[i], (u32)__popcll(b));
    }
    __syncthreads();
    if (t == 0) {
        const u32 few = WORD_LONG_FEW + (n >> WORD_LONG_FEW_SHIFT);
        const bool many = blockIdx.x == 0 && s_in[0] > (few < WORD_LONG_MOST ? few : WORD_LONG_MOST); // (one sample, not the largest of several)
        const u32 mine = many ? SECONDS_LEFT_OUT : s_in[1] > 0 || s_in[2] > PIECES_FEW ? if_endless : SECONDS_AND_SETTLE;
        if (mine)
            atomicMax(choice, mine);
    }
}

constexpr int WORDS_MAX = RESOLVE_MAX;

// The list comes in virtual order (virtual_to_suffix) with the suffixes of the text's last two words in front, shortest first: among equal first words those that run
// off the text inside their second one stand before all others, as they do before those with the same padded second word, so a stable sort by
// second words leaves them there. (With one word in front a text whose end was in a long run could not use its second words: 4 * 10^6 letters of an alphabet of 100
// took 1.25 ms, 0.97 by the doubling.)
struct WordArgs {
    const u64* keys; // sorted: the first words
    const u32* sufs;
    u32 n; // suffixes, all of which the list holds
    const u32* stream;
    u32 bits, syms; // of a symbol; symbols of a word
    WordLevels levels;
    u32* sufs_out;
    u8* ties;      // of every entry, TIE_LONG and on how many of the levels it ties with its left neighbour
    u32* any_long; // zeroed: set if some run has more than WORDS_MAX members
    // the members of long runs, in list order
    u64* run_keys; // second words, and places in the lists below: what is sorted
    u32* run_slots;
    u64* words2;
    u32* members;
    u32* ordinals; // of their runs
    u32* places;
    u32* tile_agg;
    u32* tile_splits;
    const u32* tile_prefix;
    const u32* slab_total;
    u32 slab;
};

__device__ __forceinline__ u64 word_after(const WordArgs& a, u32 x)
{
    const u64 y = (u64)x + a.syms;
    return y < a.n ? packed_window(a.stream, y * a.bits, a.bits * a.syms) : 0ull;
}

// On how many levels two neighbours x and y tie whose first words differ in `diff`, or agree (diff = 0) and whose second words differ in diff2: whoever
// runs off the text inside a context ties with nobody on it.
__device__ __forceinline__ u32 levels_of(const WordArgs& a, u64 diff, u64 diff2, u32 x, u32 y)
{
    const u64 last = x > y ? x : y;
    u32 level = 0;
#pragma unroll
    for (u32 i = 0; i < WORD_LEVELS; ++i) {
        const bool inside = i < a.levels.in_first;
        const u64 left = inside ? diff >> a.levels.drop[i] : diff | (diff2 >> a.levels.drop[i]);
        level += i < a.levels.count && left == 0 && last + a.levels.context[i] < a.n ? 1u : 0u;
    }
    return level;
}

// The runs of equal first words of one tile and the halo its first and last run reach into (as in resolve_runs_kernel): every member of a run of up to
// WORDS_MAX suffixes counts those with a smaller second word. Bounded by the lines of the stream.
__global__ __launch_bounds__(RESOLVE_BLOCK) void resolve_words_kernel(WordArgs a)
{
    constexpr int H = WORDS_MAX, SPAN = RESOLVE_TILE + 2 * H;
    constexpr int ITEMS = RESOLVE_ITEMS + 1; // the last one is the thread's element of the halo
    __shared__ u64 s_head[SPAN / 64]; // bit j: the element at span place j starts a run (places outside the list count as starts)
    __shared__ u64 s_key[SPAN];       // second words
    __shared__ u32 s_suf[SPAN];
    const u32 t = threadIdx.x;
    const long long t0 = (long long)blockIdx.x * RESOLVE_TILE, lo = t0 - H, m = a.n;
    for (int j = t; j < SPAN; j += RESOLVE_BLOCK) {
        const long long e = lo + j;
        const bool in = e >= 0 && e < m, head = e <= 0 || e >= m || a.keys[e] != a.keys[e - 1];
        s_suf[j] = in ? a.sufs[e] : 0u;
        const u64 b = __ballot(head);
        if ((t & 63u) == 0)
            s_head[j / 64] = b;
    }
    __syncthreads();
    auto is_head = [&](int j) { return ((s_head[j / 64] >> (j & 63)) & 1ull) != 0; };
    // the run around place j: first place and first place behind it; false if it has more than H members
    auto run_of = [&](int j, int& first, int& last) -> bool {
        int wd = j / 64;
        u64 b = s_head[wd] & (~0ull >> (63 - (j & 63))); // starts at or before j
        while (b == 0 && wd > 0 && wd * 64 > j - H)
            b = s_head[--wd];
        first = b ? wd * 64 + 63 - __builtin_clzll(b) : -1;
        if (first < 0 || j - first > H)
            return false;
        wd = j / 64;
        b = (j & 63) == 63 ? 0ull : s_head[wd] & (~0ull << ((j & 63) + 1)); // starts behind j
        while (b == 0 && wd + 1 < SPAN / 64 && (wd + 1) * 64 <= j + H)
            b = s_head[++wd];
        last = b ? wd * 64 + __builtin_ctzll(b) : SPAN + H;
        return last - first <= H;
    };
    u32 x[ITEMS], longs = 0;
    int first[ITEMS], last[ITEMS]; // last - first = 1: alone, or nothing to do
    u64 w1[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const bool halo = k == RESOLVE_ITEMS;
        const int j = !halo ? H + k * RESOLVE_BLOCK + (int)t : (int)t < H ? (int)t : RESOLVE_TILE + (int)t;
        const long long e = lo + j;
        x[k] = 0;
        first[k] = j;
        last[k] = j + 1;
        w1[k] = 0;
        if (e < 0 || e >= m || (halo && (int)t >= 2 * H))
            continue;
        int f, l;
        if (!run_of(j, f, l)) {
            longs |= halo ? 0u : 1u << k;
            continue;
        }
        if (l - f == 1 || (halo && ((int)t < H ? l <= H : f >= H + RESOLVE_TILE)))
            continue;
        first[k] = f;
        last[k] = l;
        x[k] = s_suf[j];
        w1[k] = word_after(a, x[k]);
    }
    if (longs)
        *a.any_long = 1u;
#pragma unroll
    for (int k = 0; k < ITEMS; ++k)
        if (last[k] - first[k] > 1)
            s_key[k == RESOLVE_ITEMS ? ((int)t < H ? (int)t : RESOLVE_TILE + (int)t) : H + k * RESOLVE_BLOCK + (int)t] = w1[k];
    __syncthreads();
    int place[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const int f = first[k], l = last[k];
        const int j = k == RESOLVE_ITEMS ? ((int)t < H ? (int)t : RESOLVE_TILE + (int)t) : H + k * RESOLVE_BLOCK + (int)t;
        place[k] = j;
        if (l - f <= 1)
            continue;
        int before = 0;
        for (int i = f; i < l; ++i)
            before += s_key[i] < w1[k] || (s_key[i] == w1[k] && i < j) ? 1 : 0;
        place[k] = f + before;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ITEMS; ++k)
        if (last[k] - first[k] > 1) {
            s_suf[place[k]] = x[k];
            s_key[place[k]] = w1[k];
        }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RESOLVE_ITEMS; ++k) {
        const int j = H + k * RESOLVE_BLOCK + (int)t;
        const long long e = lo + j;
        if (e >= m)
            continue;
        const bool is_long = (longs >> k) & 1u;
        u32 tie = 0;
        if (e > 0) {
            const bool head = is_head(j);
            const u64 diff = head ? a.keys[e] ^ a.keys[e - 1] : 0ull;
            tie = levels_of(a, diff, head || is_long ? ~0ull : s_key[j] ^ s_key[j - 1], s_suf[j], s_suf[j - 1]);
        }
        a.sufs_out[e] = s_suf[j];
        a.ties[e] = (u8)(tie | (is_long ? TIE_LONG | (is_head(j) ? TIE_HEAD : 0u) : 0u));
    }
}

// The members of long runs in list order: APPLY = false counts them and their runs per tile, APPLY = true (after rerank_scan_kernel) lists them.
template <bool APPLY>
__global__ __launch_bounds__(COLLECT_BLOCK) void collect_words_kernel(WordArgs a)
{
    __shared__ u32 s_w[COLLECT_BLOCK / WAVE][2];
    const u32 t = threadIdx.x, lane = t & 63u, w = t >> 6, tile = blockIdx.x;
    const u64 base = (u64)tile * COLLECT_TILE + (u64)t * COLLECT_ITEMS;
    u32 mine = 0, heads = 0;
    u8 tie[COLLECT_ITEMS];
#pragma unroll
    for (int k = 0; k < COLLECT_ITEMS; ++k) {
        tie[k] = base + k < a.n ? a.ties[base + k] : (u8)0;
        mine += (tie[k] & TIE_LONG) ? 1u : 0u;
        heads += (tie[k] & TIE_HEAD) ? 1u : 0u;
    }
    const u32 incl = wave_incl_sum(mine), incl_heads = wave_incl_sum(heads);
    if (lane == 63u) {
        s_w[w][0] = incl;
        s_w[w][1] = incl_heads;
    }
    __syncthreads();
    u32 slot = incl - mine, total = 0, ordinal = incl_heads - heads, total_heads = 0;
    for (u32 ww = 0; ww < COLLECT_BLOCK / WAVE; ++ww) {
        if (ww < w) {
            slot += s_w[ww][0];
            ordinal += s_w[ww][1];
        }
        total += s_w[ww][0];
        total_heads += s_w[ww][1];
    }
    if (!APPLY) {
        if (t == 0) {
            *reinterpret_cast<uint4*>(a.tile_agg + (u64)tile * 4) = make_uint4(0u, 0u, total, total_heads);
            a.tile_splits[tile] = 0;
        }
        return;
    }
    if (total == 0)
        return;
    const SlabPrefix sp = slabs_before(a.slab_total, tile / a.slab);
    slot += a.tile_prefix[(u64)tile * 4 + 2] + sp.sum2;
    ordinal += a.tile_prefix[(u64)tile * 4 + 3] + sp.sum3; // runs begun before this thread's entries
#pragma unroll
    for (int k = 0; k < COLLECT_ITEMS; ++k)
        if (tie[k] & TIE_LONG) {
            ordinal += (tie[k] & TIE_HEAD) ? 1u : 0u;
            const u32 x = a.sufs_out[base + k];
            const u64 word = word_after(a, x);
            a.run_keys[slot] = a.words2[slot] = word;
            a.run_slots[slot] = slot;
            a.members[slot] = x;
            a.ordinals[slot] = ordinal - 1u;
            a.places[slot] = (u32)(base + k);
            ++slot;
        }
}

__global__ __launch_bounds__(256) void gather_ordinals_kernel(const u32* __restrict__ ordinals, const u32* __restrict__ slots, u32 count, u64* __restrict__ keys)
{
    const u64 i = (u64)blockIdx.x * 256 + threadIdx.x;
    if (i < count)
        keys[i] = ordinals[slots[i]];
}

// The members of long runs, sorted by run and second word (run_slots), to their places.
__global__ __launch_bounds__(256) void place_words_kernel(WordArgs a, u32 count)
{
    const u64 i = (u64)blockIdx.x * 256 + threadIdx.x;
    if (i >= count)
        return;
    const u32 slot = a.run_slots[i], place = a.places[i], x = a.members[slot];
    a.sufs_out[place] = x;
    const u32 before = i > 0 ? a.run_slots[i - 1] : slot;
    if (i > 0 && a.ordinals[before] == a.ordinals[slot]) // (the first of a run ties with its left neighbour as before)
        a.ties[place] = (u8)(TIE_LONG | levels_of(a, 0ull, a.words2[slot] ^ a.words2[before], x, a.members[before]));
}

} // namespace csa
