// Generation 0 of a text over a large alphabet: the first sort on 32-bit codes instead of 64-bit K-gram keys.
//
// The code of a suffix is the place of its four symbols among all four-symbol strings, weighted by how often the symbols
// occur: with cum[s] the share of symbols below s (as a 32-bit fraction) and w[s] = cum[s + 1] - cum[s],
//   code(s0 s1 s2 s3) = cum[s0] + w[s0] (cum[s1] + w[s1] (cum[s2] + w[s2] cum[s3])),
// an arithmetic code cut to 32 bits (every product is a 32 x 32 multiplication whose upper half is kept). A larger string never
// has a smaller code, whatever the shares are, so they may come from a sample of the text; frequent symbols take wide
// intervals, so that the codes spread evenly over the 32 bits where the raw symbols of a token text crowd into few values.
// Four passes over 8-byte (code, suffix) pairs put the suffixes into the order of their codes, where K-gram keys take
// eight passes over 12-byte pairs: 66 instead of 185 bytes moved per suffix (2^28 Zipf tokens: generation 0's passes 11.5 ->
// 4.1 ms). From 2^24 suffixes on two passes over the upper digits are enough, and the lower ones are sorted bucket by bucket in LDS
// (bucket_sort.hpp); codes of token texts then take 16 bits of what follows with them (EXT), which settles most of what shares a code
// without a line of the text (1e9 tokens 45.5 -> 35.7 ms).
//
// A string whose interval of codes holds at least two 32-bit values takes the second of them, which no other string can
// have: its suffixes carry a flag (OWN_CODE) through the sort and are known to be equal where their codes are.
//
// What the sort leaves open are the suffixes that share a code. resolve_runs_kernel reads the strings of those whose code is not their own
// and, of all of them, the four symbols after the string from the text (a random 128-byte line each, which is what bounds it), puts every
// run of up to RESOLVE_MAX suffixes in order inside its tile, and notes beside every suffix on how many words of four symbols it
// ties with its left neighbour, which is all the rank step needs to know: the list is that of generation 1, and what that generation
// cost (a gathered line for every suffix that is tied on four symbols, a sort of its large groups, an update of the ranks) is not
// paid (a list with many suffixes in long runs is resolved on one word: many_in_long_runs). Longer runs that are one string repeated are in order as they stand; those that are not are collected and radix sorted by the
// string itself. Then all members of long runs are sorted by the code of the next four symbols and resolved like the rest.
// Time of whole sorts when the first sort resolves four symbols and eight: 1e9 Zipf tokens 73.2 and 65.4 ms, 2^28 18.6 and 16.9, 4096
// 0.37 and 0.31; the kernel itself 8.1 and 13.8 ms on 1e9.
//
// The shares are those of single symbols, so the codes are only as even as neighbouring symbols are independent. Where a symbol has few
// successors (phrases, records), strings that are rare by the shares of their symbols are common, and most suffixes end up in long
// runs of one code: such texts lose more than they win (2^28 symbols of a chain with 3 successors each: generation 0 38.8 ms,
// 15.7 on K-gram keys). probe_codes_kernel looks for that in a sample of the suffixes, and the first sort of such a text takes
// K-gram keys. Short texts are not probed.
#pragma once

#include "device_utils.hpp"
#include "doubling.hpp"
#include "radix_sort.hpp"

namespace csa {

// ---- shares of the symbols, from a sample ----

constexpr int SYMBOLS = 1 << 16;
constexpr int SAMPLE_BLOCK = 1024;
constexpr u32 SAMPLE_CHUNK = 64;              // consecutive symbols, one wave's worth
constexpr u32 SAMPLE_CHUNKS_MIN = 256;        // 2^14 symbols are looked at, at least ...
constexpr u32 SAMPLE_CHUNKS_MAX = 1u << 14;   // ... and 2^20 at most
constexpr u32 SAMPLE_CHUNKS_WIDE = 1u << 13;  // (samples of this many chunks or more take workgroups of twice as many)
constexpr int SAMPLE_LOG2 = 20;

// Chunk (or place) c of a sample of `taken` out of `chunks`: one of the c-th of `taken` equal stretches of the text, at the place in it that the
// multiples of the golden ratio, cut to their fractions, give. At equal distances the chunks would see only a few columns of a text
// in rows of a fixed length (2^28 symbols in rows of 1024, the first 64 of each over values of their own: at a stride of
// 16384 symbols only those columns were sampled, most suffixes shared their code with thousands of others, and generation 0
// took 37.0 ms).
// `start` shifts the places.
__device__ __forceinline__ u32 sampled_chunk(u32 c, u32 chunks, u32 taken, u32 start)
{
    const u32 lo = (u32)((u64)c * chunks / taken), hi = (u32)((u64)(c + 1) * chunks / taken);
    return lo + (u32)(((u64)(c * 0x9E3779B1u + start) * (hi - lo)) >> 32);
}

// Chunks of a workgroup (a 16-bit counter holds all their symbols). What bounds the kernel is clearing the counters and adding them to the
// table: more workgroups work at it side by side, and add the same symbol more often. us for 64, 128 and 256 chunks: 2^20 Zipf tokens
// 11, 14, 18, 2^23 17, 17, 20, 2^25 24, 23, 32; independent ids 2^20 12, 15, 18, 2^23 36, 31, 29, 2^25 54, 44, 40.
__host__ __device__ __forceinline__ u32 sample_chunks_per_block(u32 taken) { return taken < SAMPLE_CHUNKS_WIDE ? 64u : 128u; }

// Whether a text with these byte counts is one that codes are not for: few enough symbols for packed keys, or symbols that differ in one
// byte alone (plan_packed_text has the last word).
__host__ __device__ __forceinline__ bool few_symbols(u32 nlo, u32 nhi) { return nlo * nhi <= 256u || nlo == 1u || nhi == 1u; }

// The different low and high bytes of a text (zero, the padding, counted in) for every thread of a workgroup of 512 or more.
__device__ __forceinline__ void count_different_bytes(const u32* __restrict__ bytehist, u32 (&s_different)[2], u32& nlo, u32& nhi)
{
    const u32 t = threadIdx.x;
    if (t < 2)
        s_different[t] = 0;
    __syncthreads();
    if (t < 512) {
        const u64 b = __ballot((t & 255u) == 0 || bytehist[t] != 0);
        if ((t & 63u) == 0)
            atomicAdd(&s_different[t / 256u], (u32)__popcll(b));
    }
    __syncthreads();
    nlo = s_different[0];
    nhi = s_different[1];
}

// counts[s] += occurrences of symbol s in the sample: `taken` chunks (all of them when the text is short). bytehist: non-null if the host has
// not seen the byte counts yet; a text that will not be sorted by codes is left alone then, and *skipped is set.
__global__ __launch_bounds__(SAMPLE_BLOCK) void sample_symbols_kernel(const u16* __restrict__ text, u32 n, u32 chunks, u32 taken,
                                                                      u32* __restrict__ counts, const u32* __restrict__ bytehist, u32* skipped)
{
    __shared__ u32 s_cnt[SYMBOLS / 2]; // two 16-bit counters per word
    __shared__ u32 s_different[2];
    if (bytehist) {
        u32 nlo, nhi;
        count_different_bytes(bytehist, s_different, nlo, nhi);
        if (few_symbols(nlo, nhi)) {
            if (blockIdx.x == 0 && threadIdx.x == 0)
                *skipped = 1u;
            return;
        }
    }
    const u32 t = threadIdx.x;
    for (u32 i = t; i < (u32)SYMBOLS / 2; i += SAMPLE_BLOCK)
        s_cnt[i] = 0;
    __syncthreads();
    const u32 per_block = sample_chunks_per_block(taken), first = blockIdx.x * per_block;
#pragma unroll 4
    for (u32 r = t / SAMPLE_CHUNK; r < per_block; r += SAMPLE_BLOCK / SAMPLE_CHUNK) {
        const u32 c = first + r;
        if (c < taken) {
            const u64 p = (u64)sampled_chunk(c, chunks, taken, 0) * SAMPLE_CHUNK + (t & (SAMPLE_CHUNK - 1));
            if (p < n) {
                const u32 s = text[p];
                atomicAdd(&s_cnt[s >> 1], (s & 1u) ? 0x10000u : 1u);
            }
        }
    }
    __syncthreads();
    for (u32 i = t; i < (u32)SYMBOLS / 2; i += SAMPLE_BLOCK) {
        const u32 v = s_cnt[i];
        if (v & 0xFFFFu)
            atomicAdd(&counts[2 * i], v & 0xFFFFu);
        if (v >> 16)
            atomicAdd(&counts[2 * i + 1], v >> 16);
    }
}

// cum[s], s <= SYMBOLS: the share of symbols below s as a 32-bit fraction, every symbol counted once more than the sample
// (scaled by 2^weight_log2) has it, so that one the sample missed has a place too. total >= the sum of all weights (the
// sample holds the text's last chunk or not, which may be a short one).
// Workgroup b writes the entries of SHARES_TILE symbols; it sums the counts of the symbols before them by itself (at most 16
// coalesced rounds over a table in the L2), which takes a third of the time of one workgroup that scans them all (18 us).
constexpr int SHARES_TILE = 1024;

__global__ __launch_bounds__(SHARES_TILE) void symbol_shares_kernel(const u32* __restrict__ counts, int weight_log2, u32 total, u32* __restrict__ cum,
                                                                    const u32* __restrict__ skipped)
{
    __shared__ u32 s_sum[16], s_own[16];
    if (*skipped)
        return;
    const u32 t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const u32 first = blockIdx.x * SHARES_TILE;
    u32 earlier = 0;
#pragma unroll 4
    for (u32 i = t * 4; i < first; i += SHARES_TILE * 4) {
        const uint4 v = *reinterpret_cast<const uint4*>(counts + i);
        earlier += v.x + v.y + v.z + v.w;
    }
    const u32 weight = (counts[first + t] << weight_log2) + 1u;
    const u32 sum = wave_reduce_sum(earlier), incl = wave_incl_sum(weight);
    if (lane == 0)
        s_sum[w] = sum;
    if (lane == 63u)
        s_own[w] = incl;
    __syncthreads();
    u32 counted = 0, before = incl - weight;
    for (u32 ww = 0; ww < 16; ++ww) {
        counted += s_sum[ww];
        before += ww < w ? s_own[ww] : 0u;
    }
    before += (counted << weight_log2) + first;
    const u64 scale = (1ull << 53) / total; // before < total: every symbol weighs at least 1
    cum[first + t] = (u32)((u64)before * scale >> 21);
    if (first + t == (u32)SYMBOLS - 1)
        cum[SYMBOLS] = 0xFFFFFFFFu;
}

// ---- do the codes tell this text's suffixes apart? ----

// The interval of codes [low, high) of the string of four symbols with shares lo[k], width[k]: the map from the last symbol's entries
// to both ends is monotone, so the next string starts at `high` or later, and low + 1, where it is below `high`, is above every
// code of a smaller string and below every code of a larger one: true if the string takes that code, which is its own then.
__device__ __forceinline__ bool string_code(const u32 (&lo)[4], const u32 (&width)[4], u32& code)
{
    u32 low = lo[3], high = lo[3] + width[3];
#pragma unroll
    for (int q = 2; q >= 0; --q) {
        low = lo[q] + (u32)(((u64)width[q] * low) >> 32);
        high = lo[q] + (u32)(((u64)width[q] * high) >> 32);
    }
    const bool alone = high - low >= 2u;
    code = low + (alone ? 1u : 0u);
    return alone;
}

// The same with 32 bits more, where the string does not take a code of its own: the place of the string inside its code's values, of which the upper
// 16 are kept. (`low` is the upper half of the longer product, which may lie above `high`, cut at every step, where the interval is short.)
__device__ __forceinline__ bool string_code(const u32 (&lo)[4], const u32 (&width)[4], u32& code, u32& within)
{
    u64 low = (u64)lo[3] << 32;
    u32 high = lo[3] + width[3];
#pragma unroll
    for (int q = 2; q >= 0; --q) {
        low = ((u64)lo[q] << 32) + (u64)width[q] * (u32)(low >> 32) + (((u64)width[q] * (u32)low) >> 32);
        high = lo[q] + (u32)(((u64)width[q] * high) >> 32);
    }
    const bool alone = (int)(high - (u32)(low >> 32)) >= 2;
    code = (u32)(low >> 32) + (alone ? 1u : 0u);
    within = (u32)low >> 16;
    return alone;
}

constexpr int PROBE_BLOCK = 256;
constexpr u32 PROBE_START = 0x55555555u; // (the sample of the symbols is taken elsewhere: what its own places show is too good)
constexpr u32 PROBE_MOST_LOG2 = 20;      // suffixes that are looked at

// What a sample of suffixes shows about codes that are not one string's alone: how often a suffix finds its code taken by one, two,
// three others and so on, by another string, by so many that a run of it is longer than RESOLVE_MAX in the whole text.
struct ProbeCounts {
    u32 again;  // suffixes that find their code taken ...
    u32 second, third, fourth; // ... by one, by two, by three others
    u32 other;  // of `again`: whose string is not that of the first one there
    u32 crowded; // of `other`: by `long_from` others or more
    u32 packed;  // suffixes, of one in bucket_skip + 1, that find `full_from` others or more in the bucket of their code (bucket_sort.hpp)
    u32 unused[3]; // (a multiple of 16 bytes is cleared by one launch)
    unsigned long long pairs; // pairs of suffixes with one code
};
constexpr u32 PROBE_FLAGS = 7; // counters before `unused`
constexpr u32 PROBE_WORDS = sizeof(ProbeCounts) / sizeof(u32);
static_assert(PROBE_WORDS % 4 == 0, "what follows the counters in the tables holds 64-bit words, and they are cleared with it");

struct ProbeArgs {
    const u16* text;
    u32 n;
    u32 taken; // suffixes, one out of each of as many stretches (sampled_chunk; not in runs, which would meet their copies in runs)
    const u32* cum;
    unsigned long long* table; // [1 << table_log2], zeroed, at least twice as many as suffixes are looked at
    u32 table_log2;
    u32 long_from;
    ProbeCounts* counts; // zeroed
    const u32* stream;   // non-null: the codes are the narrow keys of a packed text, sym_bits bits a symbol; `crowded` counts whoever
    u32 sym_bits;        // finds its code taken by long_from others or more, its own string as they are
    const u32* skipped;  // non-null: nothing is looked at if it is set
    u32* buckets;        // non-null, zeroed: suffixes that came, by the bits of their code from bucket_shift on
    u32 bucket_shift;
    u32 full_from;
    u32 bucket_skip; // one suffix of so many, a power of two, and one less here
};

// An entry of the table is a code (high half), eight bits of the first string's hash and the number of suffixes that came.
// At most 2^20 suffixes come, so a count never reaches the hash. Bounded by the latency of the table's atomics (a random line each).
__global__ __launch_bounds__(PROBE_BLOCK) void probe_codes_kernel(ProbeArgs a)
{
    __shared__ unsigned long long s_pairs[PROBE_BLOCK / WAVE];
    __shared__ u32 s_cnt[PROBE_FLAGS];
    __shared__ u32 s_bucket[PROBE_BLOCK], s_members[PROBE_BLOCK], s_before[PROBE_BLOCK];
    if (a.skipped && *a.skipped)
        return;
    const u32 t = threadIdx.x;
    if (t < PROBE_FLAGS)
        s_cnt[t] = 0;
    s_bucket[t] = ~0u;
    s_members[t] = 0;
    __syncthreads();
    u32 pairs = 0, flags = 0, bucket = ~0u, in_bucket = ~0u;
    const u32 i = blockIdx.x * PROBE_BLOCK + t;
    if (i < a.taken) {
        const u64 x = sampled_chunk(i, a.n, a.taken, PROBE_START);
        u32 lo[4], width[4], hash = 0, code;
        bool alone = false;
        if (a.stream) {
            code = (u32)packed_window(a.stream, x * a.sym_bits, 32u);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const u32 s = x + k < a.n ? a.text[x + k] : 0u;
                u32 pair[2];
                __builtin_memcpy(pair, a.cum + s, 8); // entries s and s + 1 (4-byte aligned)
                lo[k] = pair[0];
                width[k] = pair[1] - pair[0];
                hash = (hash + s + 1u) * 0x9E3779B1u;
            }
            alone = string_code(lo, width, code);
        }
        if (a.buckets && (i & a.bucket_skip) == 0) {
            bucket = code >> a.bucket_shift;
            const u32 seen = atomicCAS(&s_bucket[bucket % PROBE_BLOCK], ~0u, bucket);
            if (seen == ~0u || seen == bucket)
                in_bucket = atomicAdd(&s_members[bucket % PROBE_BLOCK], 1u);
        }
        if (!alone) {
            const unsigned long long entry = ((unsigned long long)code << 32) | (hash >> 24 << 24) | 1u;
            const u32 mask = (1u << a.table_log2) - 1u;
            u32 slot = (code * 0x9E3779B1u) >> (32 - a.table_log2);
            for (u32 tries = 0; tries <= mask; ++tries, slot = (slot + 1u) & mask) { // (half of the table stays empty)
                unsigned long long seen = atomicCAS(&a.table[slot], 0ull, entry);
                if (seen == 0)
                    break;
                if ((u32)(seen >> 32) != code)
                    continue;
                seen = atomicAdd(&a.table[slot], 1ull);
                const u32 before = (u32)seen & 0xFFFFFFu;
                const bool other = (((u32)seen ^ (u32)entry) >> 24) != 0;
                pairs = before;
                flags = 1u | (before == 1u ? 2u : 0u) | (before == 2u ? 4u : 0u) | (before == 3u ? 8u : 0u) | (other ? 16u : 0u) |
                        ((other || a.stream) && before >= a.long_from ? 32u : 0u);
                break;
            }
        }
    }
    // The members of a bucket are added by one of the workgroup's: additions to one address queue (a text of runs: 54 us, 10 without).
    if (a.buckets) {
        __syncthreads();
        u32 before = 0;
        if (in_bucket == 0)
            s_before[bucket % PROBE_BLOCK] = atomicAdd(&a.buckets[bucket], s_members[bucket % PROBE_BLOCK]);
        else if (in_bucket == ~0u && bucket != ~0u) // (its place is another bucket's)
            before = atomicAdd(&a.buckets[bucket], 1u);
        __syncthreads();
        if (in_bucket != ~0u)
            before = s_before[bucket % PROBE_BLOCK] + in_bucket;
        flags |= bucket != ~0u && before >= a.full_from ? 64u : 0u;
    }
#pragma unroll
    for (u32 k = 0; k < PROBE_FLAGS; ++k) {
        const u64 b = __ballot((flags >> k) & 1u);
        if ((t & 63u) == 0 && b)
            atomicAdd(&s_cnt[k], (u32)__popcll(b));
    }
    const u32 sum = wave_reduce_sum(pairs); // at most 64 * 2^20
    if ((t & 63u) == 0)
        s_pairs[t / WAVE] = sum;
    __syncthreads();
    if (t < PROBE_FLAGS && s_cnt[t])
        atomicAdd(reinterpret_cast<u32*>(a.counts) + t, s_cnt[t]);
    if (t == 0) {
        unsigned long long all = 0;
        for (int w = 0; w < PROBE_BLOCK / WAVE; ++w)
            all += s_pairs[w];
        if (all)
            atomicAdd(&a.counts->pairs, all);
    }
}

// ---- the codes of all suffixes, and the digit counts of the four passes ----

constexpr int CODE_BLOCK = 256;
constexpr int CODE_WIDE_BLOCK = 1024;
constexpr int CODE_ITEMS = 8;
constexpr int CODE_PASSES = 4;
constexpr int CODE_COPIES = 8;

// The radix passes over the codes: all four digits of eight bits, or those above the buckets (bucket_sort.hpp).
struct CodeDigits {
    u32 passes;
    u32 bits; // of a digit, 8 or 9
    u32 shift[CODE_PASSES];
    u32 buckets_log2; // upper bits of a code that number its bucket; 0: the passes take all bits
};
constexpr u32 CODE_BINS = CODE_PASSES * RADIX_BINS; // digit counts of all passes: four of 256, or two of 512 at most

// codes[v] = code of the suffix at virtual position v (virtual_to_suffix with `tail` = min(n, 4)); bit x & 7 of own[x >> 3]: the
// suffix at text position x has a code that only its string can have (string_code). Bounded by the lookups
// of cum[]: one 8-byte gather per symbol (the table is 256 KB: it lives in the L2s), shared by the four suffixes it appears in.
// BLOCK: the 32 KB of digit counters decide how many waves a CU holds, 16 in workgroups of 256 and 32 in workgroups of 1024,
// which code 1e9 tokens in 2.27 instead of 3.06 ms and 2^28 in 0.58 instead of 0.78 (512: 2.69, 0.66; 256 with half the
// counters: 2.92, 0.75). Short texts take 256, so that there are workgroups for every CU.
// PASSES: of `digits`. EXT: ext[v] = 16 bits that tell suffixes of one code apart, or come from equal symbols: of those that own it by their
// next four symbols (of three alone there are runs a thousand long among 1e9 tokens), of others by the rest of their string's place. Larger for none that goes before another
// suffix of the code.
template <int BLOCK, u32 PASSES, bool EXT>
__global__ __launch_bounds__(BLOCK) void code_suffixes_kernel(const u16* __restrict__ text, u32 n, u32 tail, const u32* __restrict__ cum,
                                                              u32* __restrict__ codes, u8* __restrict__ own, CodeDigits digits,
                                                              u32* __restrict__ ghist, u16* __restrict__ ext)
{
    constexpr u32 TILE = BLOCK * CODE_ITEMS, AHEAD = EXT ? 7 : 3;
    __shared__ u64 s_text[(TILE + AHEAD + 6) / 4 + 2];
    __shared__ u32 s_hist[CODE_BINS * CODE_COPIES];
    const u32 t = threadIdx.x;
    const u32 bits = PASSES == CODE_PASSES ? (u32)RADIX_BITS : digits.bits, bins = PASSES << bits;
    for (u32 i = t; i < bins * CODE_COPIES; i += BLOCK)
        s_hist[i] = 0;
    const u32 copy = t & (CODE_COPIES - 1);
    const u64 tiles = ((u64)n + TILE - 1) / TILE;
    for (u64 tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const u64 p0 = tile * TILE;
        __syncthreads(); // the counters are cleared; the stretch of the round before has been read
        const u32 sym_off = stage_text(text, n, p0, TILE + AHEAD, s_text, t, BLOCK);
        __syncthreads();
        const u16* s16 = reinterpret_cast<const u16*>(s_text) + sym_off + t * CODE_ITEMS;
        // A thread looks its own symbols up, and has those after them from the lane after it; the last lane of a wave looks them up as well. (A gather from the
        // table takes a cycle a lane, which bounded the kernel when every thread looked up all it needs.)
        u32 lo[CODE_ITEMS + AHEAD], width[CODE_ITEMS + AHEAD];
        auto look_up = [&](int k) {
            u32 pair[2];
            __builtin_memcpy(pair, cum + s16[k], 8); // entries s and s + 1 (4-byte aligned)
            lo[k] = pair[0];
            width[k] = pair[1] - pair[0];
        };
#pragma unroll
        for (int k = 0; k < CODE_ITEMS; ++k)
            look_up(k);
#pragma unroll
        for (int k = CODE_ITEMS; k < CODE_ITEMS + (int)AHEAD; ++k) {
            lo[k] = __shfl_down(lo[k - CODE_ITEMS], 1);
            width[k] = __shfl_down(width[k - CODE_ITEMS], 1);
        }
        if ((t & 63u) == 63u) {
#pragma unroll
            for (int k = CODE_ITEMS; k < CODE_ITEMS + (int)AHEAD; ++k)
                look_up(k);
        }
        u32 code[CODE_ITEMS], more[CODE_ITEMS], owners = 0;
#pragma unroll
        for (int k = 0; k < CODE_ITEMS; ++k) {
            const u32 lo4[4] = {lo[k], lo[k + 1], lo[k + 2], lo[k + 3]};
            const u32 width4[4] = {width[k], width[k + 1], width[k + 2], width[k + 3]};
            if constexpr (EXT) {
                const bool alone = string_code(lo4, width4, code[k], more[k]);
                u32 next = lo[k + 7];
#pragma unroll
                for (int q = 6; q >= 4; --q)
                    next = lo[k + q] + (u32)(((u64)width[k + q] * next) >> 32);
                more[k] = alone ? next >> 16 : more[k];
                owners |= (alone ? 1u : 0u) << k;
            } else {
                owners |= (string_code(lo4, width4, code[k]) ? 1u : 0u) << k;
            }
        }
        const u64 x0 = p0 + (u64)t * CODE_ITEMS;
        if (x0 < n)
            own[x0 / 8] = (u8)owners;
        if (tail == 4 && x0 + CODE_ITEMS + tail <= n) { // no suffix of the text's end among them: places x0 + 4 on, 16-byte aligned
            uint4* out = reinterpret_cast<uint4*>(codes + x0 + 4);
#pragma unroll
            for (int k = 0; k < CODE_ITEMS; k += 4)
                out[k / 4] = make_uint4(code[k], code[k + 1], code[k + 2], code[k + 3]);
            if constexpr (EXT) { // (x0 is a multiple of eight, ext 16-byte aligned)
                u64* const wide = reinterpret_cast<u64*>(ext + x0 + 4);
#pragma unroll
                for (int k = 0; k < CODE_ITEMS; k += 4)
                    wide[k / 4] = (u64)(more[k] | more[k + 1] << 16) | (u64)(more[k + 2] | more[k + 3] << 16) << 32;
            }
        } else {
#pragma unroll
            for (int k = 0; k < CODE_ITEMS; ++k) {
                const u64 x = x0 + k;
                if (x < n) {
                    const u64 v = x + tail >= n ? n - 1 - x : x + tail;
                    codes[v] = code[k];
                    if constexpr (EXT)
                        ext[v] = (u16)more[k];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < CODE_ITEMS; ++k)
            if (x0 + k < n) {
#pragma unroll
                for (u32 p = 0; p < PASSES; ++p) {
                    const u32 shift = PASSES == CODE_PASSES ? RADIX_BITS * p : digits.shift[p];
                    atomicAdd(&s_hist[((p << bits) + __builtin_amdgcn_ubfe(code[k], shift, bits)) * CODE_COPIES + copy], 1u);
                }
            }
    }
    __syncthreads();
    for (u32 i = t; i < bins; i += BLOCK) {
        u32 v = 0;
#pragma unroll
        for (int c = 0; c < CODE_COPIES; ++c)
            v += s_hist[i * CODE_COPIES + c];
        if (v)
            atomicAdd(&ghist[i], v);
    }
}

// ---- runs of equal codes ----

constexpr int RESOLVE_BLOCK = 512;
constexpr int RESOLVE_ITEMS = 4;
constexpr int RESOLVE_TILE = RESOLVE_BLOCK * RESOLVE_ITEMS;
#ifndef CSA_RESOLVE_MAX
#define CSA_RESOLVE_MAX 256
#endif
#ifndef CSA_WORDS_AHEAD
#define CSA_WORDS_AHEAD (1u << 22)
#endif
constexpr int RESOLVE_MAX = CSA_RESOLVE_MAX; // longest run that is sorted inside its tile
static_assert(CODE_ITEMS == 8, "a thread of the coding kernel writes one byte of flags");
static_assert(RESOLVE_MAX % 64 == 0 && 2 * RESOLVE_MAX <= RESOLVE_BLOCK, "the halo is read in whole waves, one element per thread");
constexpr u32 RESOLVE_MARK_BITS = 20;
constexpr u32 RESOLVE_MARK_WORDS = 1u << (RESOLVE_MARK_BITS - 5);

// The mark of a code: codes that share one only cost time (their runs are sorted again although they are in order).
__device__ __forceinline__ u32 resolve_mark(u32 code) { return (code * 0x9E3779B1u) >> (32 - RESOLVE_MARK_BITS); }

struct ResolveArgs {
    const u32* codes; // sorted by code: the codes (null where they have not been kept) ...
    const u64* keys;  // ... or, of the members of long runs, (ordinal of the run's string << 32 | code of the four symbols after it)
    const u32* sufs;  // OWN_CODE (with codes): no other string has this suffix's code
    u32 m;            // entries of the list ...
    const u32* open_count; // ... of open runs (OPEN), as the device has counted them; those start where bit 31 of their places is set
    const u16* text;
    u32 n;
    u32 words; // 1: the list is resolved on the symbols of the codes; 2: on as many after them, too; 0: as many_in_long_runs says ...
    u32* words_out; // ... which stands here already for long lists, and is written here for short ones
    u32 word_syms;     // symbols of a word: four, or 32 bits of the code stream of a packed text, where every code is its string's own:
    const u32* stream; // non-null
    u32 sym_bits;
    u32* sufs_out; // the list in order (the whole one: members of long runs go back to their places in it)
    u8* ties;      // of every entry, TIE_LONG and on how many words it ties with its left neighbour (doubling.hpp)
    u32* marks;    // [RESOLVE_MARK_WORDS], zeroed: codes of long runs that are not in order
    u32* unordered; // zeroed: set if there are any; with keys: if the order of a long run is not that of its strings
    u32* any_long;  // zeroed: set if there are long runs
    // the collected members of long runs (collect_runs_kernel, place_marked_kernel)
    const u32* text_codes; // the codes of all suffixes, by virtual position with `tail` suffixes at the front
    u32 tail;
    u64* run_keys;
    u32* members;
    u32* places;
    u32* tile_agg;
    u32* tile_splits;
    const u32* tile_prefix;
    const u32* slab_total;
    u32 slab;
};

// The second word of suffix x, of which the text or the stream has the end at least.
template <bool PACKED>
__device__ __forceinline__ u64 second_word(const ResolveArgs& a, u32 x)
{
    if constexpr (!PACKED)
        return load_kgram(a.text, a.n, x, 1);
    const u64 y = (u64)x + a.word_syms;
    return y < a.n ? packed_window(a.stream, y * a.sym_bits, 32u) : 0ull;
}

// A list many of whose suffixes lie in runs of RESOLVE_MAX / 2 or more is resolved on one word.
// Short lists, 12 of 64 places: members of runs that are too long for a tile would have to be sorted by the second word, those of others long for a
// tile compared by it one by one, and the generation after, with the ranks of all, costs no more. (Sorts, ms, by two words, by one,
// and before there were two: 33000 symbols of ten phrases 0.83, 0.60, 0.65; 130000 of a hundred 1.01, 0.85, 0.92; 400000 of 300 1.33, 1.12, 1.09,
// which a limit of 20 leaves at 1.35; 400000 symbols Zipf(2) 0.80, 0.69, 0.73.)
// Long lists, 543 of 1024 places, which is about where half of the list is in runs of more than RESOLVE_MAX and sort_long_runs gives it up; up to there the
// second word pays, since generation 1 would read as many lines. (ms by two words and by one, and the share of the places: 2^28 symbols
// Zipf(1.4) 0.51 25.4, 30.3; 2^29 of runs and Zipf(1.3) 0.45 52.0, 59.8; 2^26 Zipf(1.5) 0.58 9.2, 8.6; 2^28 0.66 37.9, 34.4; 2^26 Zipf(2) 0.93 14.2, 13.9;
// 5 * 10^6 of written text in 16-bit symbols 0.65 1.80, 1.63. Token texts have 0.04.)
// Lists whose lower digits were sorted in buckets (open runs) always take two words: a text so heavy that one would do has buckets that do not fit and goes
// through all passes. (3 * 10^7 symbols Zipf(1.4), open runs and two words 2.71 ms, all passes 3.05.)
constexpr u32 HALF_LONG = RESOLVE_MAX / 2, SHORT_LIST_FEW = 12, LONG_LIST_PLACES = 1024, LONG_LIST_FEW = 543;

// Lists of WORDS_AHEAD suffixes or more are looked at by a workgroup of its own: a launch costs 4 us, and the look of every tile 2 % of the sort of 2^28
// tokens (11.35 -> 11.6 ms).
constexpr u32 WORDS_AHEAD = CSA_WORDS_AHEAD;

__global__ __launch_bounds__(LONG_LIST_PLACES) void choose_words_kernel(const u32* __restrict__ codes, u32 m, u32* words_out)
{
    __shared__ u32 s_in;
    if (threadIdx.x == 0)
        s_in = 0;
    __syncthreads();
    const u64 b = __ballot(in_long_run(codes, m, HALF_LONG, threadIdx.x, LONG_LIST_PLACES));
    if ((threadIdx.x & 63u) == 0 && b)
        atomicAdd(&s_in, (u32)__popcll(b));
    __syncthreads();
    if (threadIdx.x == 0)
        *words_out = s_in > LONG_LIST_FEW ? 1u : 2u;
}

// The runs of equal codes (KEYS = false: the list of all suffixes) or of equal keys (KEYS = true: the members of the long runs, sorted
// once more by the code of the next word) of one tile and the halo its first and last run reach into, refined word by word:
// every member of a run of at most H counts those with a smaller word, which gives its place and
// the sub-run it belongs to, and the next word is compared among the members of a sub-run only. A string and its follower lie in
// one line of the text as a rule, so the second word costs one more line for one suffix in nine and saves a generation: its gather
// of a line each, its list, its rank update (1e9 Zipf tokens: 13.8 ms instead of 8.1 here, 5.5 for the long runs, and 20.0 less in
// generation 1).
// The halo's members are refined too (by both tiles their run lies in, with the same result), so that a tile knows
// all of its own places and writes them in order.
// PACKED: the words are cut from the code stream of the text, 16 bytes of which hold what 128 bytes of the text do; it fits the last-level
// cache up to 10^9 symbols of two bits.
// SHORT: lists of fewer than WORDS_AHEAD suffixes, where the slowest tile counts; what that takes costs others 1.5 % of the kernel.
// OPEN: the list is that of runs that buckets have left open (finish_buckets_kernel), wherever they stand; a workgroup takes one tile after the other.
template <int H, bool KEYS, bool PACKED, bool SHORT, bool OPEN = false> // H: the longest run that is sorted inside its tile
__global__ __launch_bounds__(RESOLVE_BLOCK, OPEN ? 8 : 1) void resolve_runs_kernel(ResolveArgs a)
{
    static_assert(!OPEN || (!KEYS && !PACKED && !SHORT), "open runs are those of codes, in long lists");
    constexpr bool PLACED = KEYS || OPEN; // the entries go to places of their own, where the ties of what starts a run are known
    constexpr u8 TIE_KNOWN = 0x20;
    const u32 entries = OPEN ? *a.open_count : a.m;
    if (OPEN && blockIdx.x == 0 && threadIdx.x == 0)
        *a.words_out = TIE_MOST_WORDS;
    for (u32 tile = blockIdx.x; !OPEN || (u64)tile * RESOLVE_TILE < entries; tile += gridDim.x) {
        constexpr int SPAN = RESOLVE_TILE + 2 * H;
        constexpr int ITEMS = RESOLVE_ITEMS + 1; // the last one is the thread's element of the halo
        constexpr int FEW = 16; // (sub-)runs of up to this many members are sorted without a look whether they are in order
        __shared__ u64 s_head[SPAN / 64]; // bit j: the element at span place j starts a run (places outside the list count as starts)
        __shared__ u64 s_down[SPAN / 64]; // bit j: its word is smaller than that of the element before it ...
        __shared__ u64 s_diff[SPAN / 64]; // ... or another one
        __shared__ u32 s_many[2];         // some run of the tile has more members, by word
        __shared__ u32 s_ends;            // some member of a run runs off the text inside its words
        __shared__ u32 s_words;
        __shared__ u32 s_off[SHORT ? 2 : 1][SHORT ? SPAN / 32 : 1]; // bit j, by word: one of the run that starts at place j does
        __shared__ __align__(16) u64 s_key[SPAN];
        __shared__ __align__(16) u32 s_suf[SPAN];
        __shared__ __align__(16) u8 s_tie[SPAN];
        u32 t = threadIdx.x;
        if (OPEN)
            opaque(t); // (what follows from it is not kept from tile to tile: 152 registers, a workgroup a SIMD)
        if (t < 2)
            s_many[t] = 0;
        if (t == 2)
            s_ends = 0;
        const u32 told = PLACED ? TIE_MOST_WORDS : SHORT || a.words ? a.words : *a.words_out;
        if (!PLACED && t < 64u) {
            const u32 w = SHORT && told == 0 ? (many_in_long_runs(a.codes, a.m, HALF_LONG, SHORT_LIST_FEW) ? 1u : 2u) : told;
            if (t == 0) {
                if (SHORT)
                    s_words = w;
                if (blockIdx.x == 0)
                    *a.words_out = w;
            }
        }
        const long long t0 = (long long)tile * RESOLVE_TILE, lo = t0 - H, m = entries;
        const u64 n = a.n;
        // whole waves take consecutive places: one ballot per wave and round gives 64 bits of s_head
        for (int j = t; j < SPAN; j += RESOLVE_BLOCK) { // (the same rounds for every lane of a wave: SPAN is a multiple of 64)
            const long long e = lo + j;
            bool head = e <= 0 || e >= m;
            u8 tie = 0;
            if (!head) {
                if constexpr (OPEN) {
                    head = (a.places[e] & RUN_START) != 0;
                } else if constexpr (KEYS) {
                    const u64 mine = a.keys[e], before = a.keys[e - 1];
                    head = mine != before;
                    tie = (mine >> 32) == (before >> 32) ? 1 : TIE_KNOWN; // (members of one string that do not run off the text inside it)
                } else {
                    head = a.codes[e] != a.codes[e - 1];
                }
            }
            s_tie[j] = !head ? (u8)TIE_MOST_WORDS : OPEN || (KEYS && e <= 0) ? TIE_KNOWN : tie;
            const u64 b = __ballot(head);
            if ((t & 63u) == 0)
                s_head[j / 64] = b;
        }
        __syncthreads();
        const u32 words = SHORT && !KEYS ? s_words : told;
        if (words < TIE_MOST_WORDS)
            for (int j = t; j < SPAN; j += RESOLVE_BLOCK) // (the thread's own places)
                s_tie[j] = s_tie[j] ? (u8)words : (u8)0;
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
        // the elements: suffix, place, run, and the words where there is company
        u32 x[ITEMS], owners = 0, longs = 0; // bit k: element k has OWN_CODE; is one of a long run
        int at[ITEMS], first[ITEMS], last[ITEMS]; // last - first = 1: alone
        u64 w0[ITEMS], w1[ITEMS];
        const bool two = PLACED || words == 2; // (keys come with two words)
        const u32 word_syms = PACKED ? a.word_syms : 4u;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const bool halo = k == RESOLVE_ITEMS;
            const int j = !halo ? H + k * RESOLVE_BLOCK + (int)t : (int)t < H ? (int)t : RESOLVE_TILE + (int)t;
            const long long e = lo + j;
            x[k] = 0;
            at[k] = first[k] = j;
            last[k] = j + 1;
            w0[k] = w1[k] = 0;
            if (e < 0 || e >= m || (halo && (int)t >= 2 * H))
                continue;
            int f, l;
            const bool is_short = run_of(j, f, l);
            if (halo) { // members of runs that reach into the tile; of a long run the left neighbour of the tile's first element alone
                const bool left = (int)t < H;
                if (is_short ? (left ? l <= H : f >= H + RESOLVE_TILE) : j != H - 1)
                    continue;
            }
            x[k] = a.sufs[e]; // (asked for before the runs are known, for all elements: no faster, 14.4 and 15.0 ms on 1e9 tokens)
            if (!KEYS && (x[k] & OWN_CODE))
                owners |= 1u << k;
            x[k] &= ~OWN_CODE;
            if (is_short) {
                first[k] = f;
                last[k] = l;
                if (l - f == 1)
                    continue;
            } else {
                longs |= 1u << k;
            }
            const bool own = (owners >> k) & 1u;
            if (!KEYS && !PACKED && !own)
                w0[k] = load_kgram(a.text, a.n, x[k], 0);
            if (two && (KEYS || is_short)) // (the members of long runs of codes get their second word when they are sorted by it)
                w1[k] = second_word<PACKED>(a, x[k]);
            if ((u64)x[k] + (u64)word_syms * words >= n)
                s_ends = 1;
            if (is_short && l - f > FEW) {
                s_many[0] = 1;
                s_many[1] = 1;
            }
        }
        __syncthreads();
        const bool ends = s_ends != 0;
        if (SHORT && ends) {
            for (int j = t; j < 2 * SPAN / 32; j += RESOLVE_BLOCK)
                s_off[j / (SPAN / 32)][j % (SPAN / 32)] = 0;
            __syncthreads();
        }
        // One word of all elements that still have company: refines their runs. Whoever runs off the text inside the word ties with
        // nobody and comes before those with the same padded word, shortest first. (SHORT: only the runs with such a member are looked at that way: a tile
        // is as slow as its slowest run, and a short text as its slowest tile. 10^5 symbols of phrases: 168 us with all runs of a tile that
        // holds one of the last suffixes, 55 without.)
        auto refine = [&](int w) {
            const u64 ctx = word_syms * (u32)(w + 1);
#pragma unroll
            for (int k = 0; k < ITEMS; ++k)
                if (last[k] - first[k] > 1 || ((longs >> k) & 1u)) {
                    s_suf[at[k]] = x[k];
                    if (w == 1 || !((owners >> k) & 1u))
                        s_key[at[k]] = w == 0 ? w0[k] : w1[k];
                    if (SHORT && ends && (u64)x[k] + ctx >= n && !((longs >> k) & 1u))
                        atomicOr(&s_off[w][first[k] / 32], 1u << (first[k] & 31));
                }
            __syncthreads();
            const bool many = s_many[w] != 0 && (SHORT || !ends);
            if (many) {
                for (int j = t; j < SPAN; j += RESOLVE_BLOCK) { // (places whose words were not wanted hold anything: no run looked at below has any)
                    const u64 down = __ballot(j > 0 && s_key[j] < s_key[j - 1]), diff = __ballot(j > 0 && s_key[j] != s_key[j - 1]);
                    if ((t & 63u) == 0) {
                        s_down[j / 64] = down;
                        s_diff[j / 64] = diff;
                    }
                }
                __syncthreads();
            }
#pragma unroll
            for (int k = 0; k < ITEMS; ++k) {
                const int f = first[k], l = last[k], j = at[k];
                if ((longs >> k) & 1u || l - f <= 1)
                    continue;
                const bool own = w == 0 && ((owners >> k) & 1u), off = ends && (!SHORT || ((s_off[w][f / 32] >> (f & 31)) & 1u));
                int nf = f, nl = l, place = j;
                if (own) { // one string: those that run off the text come first as they stand
                    if (off) {
                        while (nf < l && (u64)s_suf[nf] + ctx >= n)
                            ++nf;
                        if (j < nf) {
                            nf = j;
                            nl = j + 1;
                        }
                    }
                } else {
                    bool counted = true;
                    if (many && l - f > FEW && !off) {
                        // A run that is one string repeated, or several in order, stays as it is: its members need not be compared with
                        // each other. (In a short text the kernel takes as long as the longest run of a tile: generation 0 of 2^18
                        // symbols of phrases 221 us with all comparisons, 191 without these.)
                        u64 seen = 0;
                        for (int wd = (f + 1) / 64; wd <= (l - 1) / 64; ++wd) { // places f + 1 .. l - 1
                            u64 b = s_down[wd];
                            if (wd == (f + 1) / 64)
                                b &= ~0ull << ((f + 1) & 63);
                            if (wd == (l - 1) / 64)
                                b &= ~0ull >> (63 - ((l - 1) & 63));
                            seen |= b;
                        }
                        if (seen == 0) {
                            counted = false;
                            int wd = j / 64; // the last other word at or before j, the first behind it
                            u64 b = s_diff[wd] & (~0ull >> (63 - (j & 63)));
                            while (b == 0 && wd > f / 64)
                                b = s_diff[--wd];
                            const int start = b ? wd * 64 + 63 - __builtin_clzll(b) : f;
                            nf = start > f ? start : f;
                            wd = j / 64;
                            b = (j & 63) == 63 ? 0ull : s_diff[wd] & (~0ull << ((j & 63) + 1));
                            while (b == 0 && wd < (l - 1) / 64)
                                b = s_diff[++wd];
                            const int stop = b ? wd * 64 + __builtin_ctzll(b) : l;
                            nl = stop < l ? stop : l;
                        }
                    }
                    if (counted) {
                        const u64 mine = s_key[j];
                        int less = 0, equal = 0, before = 0; // equal: itself included
                        if (!off) {
                            for (int i = f; i < l; ++i) {
                                const u64 v = s_key[i];
                                less += v < mine ? 1 : 0;
                                equal += v == mine ? 1 : 0;
                                before += v == mine && i < j ? 1 : 0;
                            }
                        } else {
                            const bool whole = (u64)x[k] + ctx < n;
                            for (int i = f; i < l; ++i) {
                                const u64 v = s_key[i];
                                if (v < mine) {
                                    ++less;
                                } else if (v == mine) {
                                    const u32 y = s_suf[i];
                                    const bool y_whole = (u64)y + ctx < n;
                                    if (whole != y_whole)
                                        less += whole ? 1 : 0;
                                    else if (!whole)
                                        less += y > x[k] ? 1 : 0;
                                    else
                                        ++equal, before += i < j ? 1 : 0;
                                }
                            }
                            equal = whole ? equal : 1;
                        }
                        nf = f + less;
                        nl = nf + equal;
                        place = nf + before;
                    }
                }
                if (place == nf && nf != f)
                    s_tie[nf] = (u8)w;
                first[k] = nf;
                last[k] = nl;
                at[k] = place;
            }
            // the members of long runs stay where they are: do they tie with their left neighbours, are they in order?
#pragma unroll
            for (int k = 0; k < RESOLVE_ITEMS; ++k)
                if ((longs >> k) & 1u && w == (KEYS ? 1 : 0)) {
                    const int j = at[k];
                    u8 tie = s_tie[j];
                    if (!((s_head[j / 64] >> (j & 63)) & 1ull)) {
                        const bool whole = (u64)x[k] + ctx < n && (u64)s_suf[j - 1] + ctx < n;
                        const bool own = w == 0 && ((owners >> k) & 1u);
                        const u64 mine = own ? 0 : s_key[j], left = own ? 0 : s_key[j - 1];
                        tie = (u8)(w + (mine == left && whole ? 1 : 0));
                        if constexpr (KEYS) {
                            if (mine < left || !whole)
                                *a.unordered = 1u;
                        } else if (mine < left) {
                            const u32 mark = resolve_mark(OPEN ? a.text_codes[suffix_to_virtual(x[k], a.n, a.tail)] : a.codes[lo + j]), bit = 1u << (mark & 31u);
                            if (!(a.marks[mark >> 5] & bit)) // (soon set for all to see: few of a run's members get to the atomic)
                                atomicOr(&a.marks[mark >> 5], bit);
                            *a.unordered = 1u;
                        }
                    } else {
                        *a.any_long = 1u;
                        tie |= OPEN ? TIE_HEAD : 0;
                    }
                    s_tie[j] = tie | TIE_LONG;
                }
            __syncthreads();
        };
        if constexpr (!KEYS)
            refine(0);
        if (two)
            refine(1);
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (k < RESOLVE_ITEMS || (int)t < 2 * H)
                s_suf[at[k]] = x[k];
        __syncthreads();
        const int j = H + (int)t * RESOLVE_ITEMS;
        const long long e = lo + j;
        if constexpr (!PLACED) {
            if (e + RESOLVE_ITEMS <= m) { // (e is a multiple of RESOLVE_ITEMS, and the arrays are 16-byte aligned)
                static_assert(RESOLVE_ITEMS == 4 && H % 4 == 0, "four suffixes leave in one 16-byte store");
                *reinterpret_cast<uint4*>(a.sufs_out + e) = *reinterpret_cast<const uint4*>(s_suf + j);
                *reinterpret_cast<u32*>(a.ties + e) = *reinterpret_cast<const u32*>(s_tie + j);
                return;
            }
        }
#pragma unroll
        for (int k = 0; k < RESOLVE_ITEMS; ++k)
            if (e + k < m) {
                if constexpr (OPEN) { // what is as the buckets have left it is not written again (a line each)
                    const u32 place = a.places[e + k], before = place & RUN_START ? (place & RUN_TIED ? 1u : 0u) : TIE_MOST_WORDS;
                    const u32 known = s_tie[j + k], tie = known & TIE_KNOWN ? (known & ~TIE_KNOWN) | before : known;
                    const u64 to = place & RUN_PLACE;
                    if (s_suf[j + k] != (a.sufs[e + k] & ~OWN_CODE))
                        a.sufs_out[to] = s_suf[j + k];
                    if (tie != before)
                        a.ties[to] = (u8)tie;
                    continue;
                }
                const u64 to = KEYS ? (u64)a.places[e + k] : (u64)(e + k);
                u8 tie = s_tie[j + k];
                if (KEYS && (tie & TIE_KNOWN))
                    tie = (u8)((tie & ~TIE_KNOWN) | (a.ties[to] & TIE_WORDS));
                a.sufs_out[to] = s_suf[j + k];
                a.ties[to] = tie;
            }
        if (!OPEN)
            return;
        __syncthreads();
    }
}

// What a list sorted by the narrow keys of a packed text would leave at contexts shorter than a key (RerankArgs::level_drop, level_ell; the
// sums at level_totals[slot * 8 + 2 i] and [.. + 1]): an entry ties with a neighbour if neither runs off the text inside the context.
// Reads 8 bytes a suffix.
__global__ __launch_bounds__(256) void count_code_levels_kernel(RerankArgs a, const u32* __restrict__ codes, u32 levels)
{
    constexpr int ITEMS = 4;
    const u32 lane = threadIdx.x & 63u;
    u32 sums[2 * MAX_LEVELS] = {};
    const u64 stride = (u64)gridDim.x * 256 * ITEMS;
    for (u64 base = ((u64)blockIdx.x * 256 + threadIdx.x) * ITEMS; base < a.m; base += stride) {
        u32 code[ITEMS + 2] = {}, suf[ITEMS + 2] = {}; // entries base - 1 .. base + ITEMS
        if (base + ITEMS <= a.m) { // (the arrays are 16-byte aligned)
            const uint4 c = *reinterpret_cast<const uint4*>(codes + base), x = *reinterpret_cast<const uint4*>(a.sufs + base);
            code[1] = c.x, code[2] = c.y, code[3] = c.z, code[4] = c.w;
            suf[1] = x.x, suf[2] = x.y, suf[3] = x.z, suf[4] = x.w;
        } else {
#pragma unroll
            for (int k = 1; k <= ITEMS; ++k)
                if (base + k - 1 < a.m) {
                    code[k] = codes[base + k - 1];
                    suf[k] = a.sufs[base + k - 1];
                }
        }
        if (base > 0) {
            code[0] = codes[base - 1];
            suf[0] = a.sufs[base - 1];
        }
        if (base + ITEMS < a.m) {
            code[ITEMS + 1] = codes[base + ITEMS];
            suf[ITEMS + 1] = a.sufs[base + ITEMS];
        }
#pragma unroll
        for (u32 i = 0; i < MAX_LEVELS; ++i) {
            if (i >= levels)
                break;
            u32 ties = 0; // bit k: entries base + k - 1 and base + k
#pragma unroll
            for (int k = 0; k <= ITEMS; ++k) {
                const bool there = base + k > 0 && base + k < a.m;
                const u32 last = suf[k] > suf[k + 1] ? suf[k] : suf[k + 1];
                ties |= (there && ((code[k] ^ code[k + 1]) >> a.level_drop[i]) == 0 && (u64)last + a.level_ell[i] < a.n ? 1u : 0u) << k;
            }
            const u32 whole = (1u << ITEMS) - 1u;
            sums[2 * i] += (u32)__popc((ties | (ties >> 1)) & whole);
            sums[2 * i + 1] += (u32)__popc(~ties & (ties >> 1) & whole);
        }
    }
#pragma unroll
    for (u32 i = 0; i < 2 * MAX_LEVELS; ++i) {
        if (i >= 2 * levels)
            break;
        const u32 v = wave_reduce_sum(sums[i]);
        if (lane == 0 && v)
            atomicAdd(a.level_totals + (u64)((blockIdx.x * 4 + threadIdx.x / WAVE) % LEVEL_SLOTS) * 8 + i, (unsigned long long)v);
    }
}

// Members of long runs, in list order: APPLY = false counts them and the strings they begin per tile, APPLY = true (after
// rerank_scan_kernel) writes what they are to be sorted by, their suffixes and their list places. MARKED: those of runs that are out of
// order alone, by their strings; a run is marked as a whole, so the list of them sorted by string, which is also the order
// of the codes, goes back to the same places. Otherwise all of them, by the ordinal of their string (they are in order by
// now) and the code of the next four symbols.
constexpr int COLLECT_BLOCK = 256;
constexpr int COLLECT_ITEMS = 4;
constexpr int COLLECT_TILE = COLLECT_BLOCK * COLLECT_ITEMS;

// Does this entry of a long run start a string (or, of a run that is a string's with 16 bits of what follows, the run)?
__device__ __forceinline__ bool starts_string(u32 tie) { return (tie & TIE_WORDS) == 0 || (tie & TIE_HEAD); }

template <bool MARKED, bool APPLY>
__global__ __launch_bounds__(COLLECT_BLOCK) void collect_runs_kernel(ResolveArgs a)
{
    __shared__ u32 s_w[COLLECT_BLOCK / WAVE][2];
    const u32 t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const u32 tile = blockIdx.x;
    const u64 base = (u64)tile * COLLECT_TILE + (u64)t * COLLECT_ITEMS;
    static_assert(COLLECT_ITEMS == 4, "the ties of a thread's entries come in one word");
    u32 ties = 0;
    if (base + COLLECT_ITEMS <= a.m) {
        ties = *reinterpret_cast<const u32*>(a.ties + base);
    } else {
#pragma unroll
        for (int k = 0; k < COLLECT_ITEMS; ++k)
            ties |= base + k < a.m ? (u32)a.ties[base + k] << (8 * k) : 0u;
    }
    u32 flags = 0, mine = 0, heads = 0, x[COLLECT_ITEMS] = {};
    if constexpr (APPLY) // (all loads of a thread before its first store: one after the other they took 2.7 ms for 57.7 M of 1e9 suffixes, 2.0 now)
#pragma unroll
        for (int k = 0; k < COLLECT_ITEMS; ++k)
            if ((ties >> (8 * k)) & TIE_LONG)
                x[k] = a.sufs_out[base + k];
#pragma unroll
    for (int k = 0; k < COLLECT_ITEMS; ++k)
        if ((ties >> (8 * k)) & TIE_LONG) {
            u32 in = 1u;
            if constexpr (MARKED) {
                const u32 code = a.codes ? a.codes[base + k] : a.text_codes[suffix_to_virtual(a.sufs_out[base + k], a.n, a.tail)];
                const u32 mark = resolve_mark(code);
                in = (a.marks[mark >> 5] >> (mark & 31u)) & 1u;
            }
            flags |= in << k;
            mine += in;
            heads += in && starts_string(ties >> (8 * k)) ? 1u : 0u;
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
            a.tile_agg[(u64)tile * 4 + 0] = 0;
            a.tile_agg[(u64)tile * 4 + 1] = 0;
            a.tile_agg[(u64)tile * 4 + 2] = total;
            a.tile_agg[(u64)tile * 4 + 3] = total_heads;
            a.tile_splits[tile] = 0;
        }
        return;
    }
    if (total == 0)
        return;
    u64 key[COLLECT_ITEMS];
#pragma unroll
    for (int k = 0; k < COLLECT_ITEMS; ++k) {
        key[k] = 0;
        if ((flags >> k) & 1u) {
            if constexpr (MARKED) {
                key[k] = load_kgram(a.text, a.n, x[k], 0);
            } else {
                const u64 y = (u64)x[k] + a.word_syms; // (a suffix that has none there is a string of its own)
                key[k] = y >= a.n ? 0u : a.stream ? (u32)packed_window(a.stream, y * a.sym_bits, 32u) : a.text_codes[y + a.tail >= a.n ? a.n - 1 - y : y + a.tail];
            }
        }
    }
    const SlabPrefix sp = slabs_before(a.slab_total, tile / a.slab);
    slot += a.tile_prefix[(u64)tile * 4 + 2] + sp.sum2;
    ordinal += a.tile_prefix[(u64)tile * 4 + 3] + sp.sum3; // strings begun before this thread's entries
#pragma unroll
    for (int k = 0; k < COLLECT_ITEMS; ++k)
        if ((flags >> k) & 1u) {
            if constexpr (!MARKED) {
                ordinal += starts_string(ties >> (8 * k)) ? 1u : 0u;
                key[k] |= (u64)(ordinal - 1u) << 32;
            }
            a.run_keys[slot] = key[k];
            a.members[slot] = x[k];
            a.places[slot] = (u32)(base + k);
            ++slot;
        }
}

// The collected members of marked runs, sorted by string, back to their places.
__global__ __launch_bounds__(256) void place_marked_kernel(ResolveArgs a, u32 count)
{
    const u64 i = (u64)blockIdx.x * 256 + threadIdx.x;
    if (i >= count)
        return;
    const u32 x = a.members[i];
    const bool tied = i > 0 && a.run_keys[i] == a.run_keys[i - 1] && (u64)x + 4 < a.n && (u64)a.members[i - 1] + 4 < a.n;
    a.sufs_out[a.places[i]] = x;
    if (!(a.ties[a.places[i]] & TIE_HEAD)) // (whose left neighbour is none of these)
        a.ties[a.places[i]] = (u8)(TIE_LONG | (tied ? 1u : 0u));
}

} // namespace csa
