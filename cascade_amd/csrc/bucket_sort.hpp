// The lower digits of a sort by codes, bucket by bucket in LDS.
//
// Codes are even (coded_keys.hpp): after two passes on their upper digits, the suffixes of one bucket, those that share their codes' upper
// bits, are a few thousand that stand side by side, few enough for the LDS of a workgroup. One launch reads every suffix once and
// writes it once, coalesced and without waiting for other workgroups, and takes the place of the radix passes that are left.
// Buckets that do not fit (one string a hundred thousand times) are collected, sorted by radix passes and put back.
#pragma once

#include "device_utils.hpp"
#include "doubling.hpp"
#include "radix_sort.hpp"

namespace csa {

#ifndef CSA_BUCKET_BLOCK
#define CSA_BUCKET_BLOCK 1024
#endif
#ifndef CSA_BUCKET_ITEMS
#define CSA_BUCKET_ITEMS 7
#endif
#ifndef CSA_CELLS_LOG2
#define CSA_CELLS_LOG2 12
#endif
#ifndef CSA_CELL_MAX
#define CSA_CELL_MAX 512
#endif
constexpr int BUCKET_BLOCK = CSA_BUCKET_BLOCK;
constexpr int BUCKET_ITEMS = CSA_BUCKET_ITEMS;
constexpr u32 BUCKET_MAX = BUCKET_BLOCK * BUCKET_ITEMS; // most suffixes of a bucket that is sorted in LDS (two workgroups a CU)
constexpr int CELLS_LOG2 = CSA_CELLS_LOG2;
constexpr u32 CELL_MAX = CSA_CELL_MAX; // most of a cell whose members are compared with each other
static_assert(BUCKET_MAX < 1u << 16, "counters of cells are 16 bits wide");

struct BucketArgs {
    u32* codes; // sorted by their upper bits ...
    u32* sufs;
    u32 n;
    u32 tail;     // (virtual_to_suffix)
    u32 low_bits; // ... all but so many; the others number the bucket
    u32 buckets;
    u32* starts;         // [buckets + 1]: where they start
    const u32* top_base; // of the last pass: where its digits start ...
    u32 top_shift;       // ... and the bit of the code that they start from
    u32* over;           // zeroed: [0] suffixes in buckets of more than BUCKET_MAX, [1] such buckets, [2] suffixes in the largest
    u32* over_list;      // [n / BUCKET_MAX]: them, in any order
    u32* crowded;        // zeroed: buckets with a cell of more than CELL_MAX ...
    u32* crowded_list;   // ... [buckets]: them, in any order
    // EXT: sixteen bits more of every suffix (code_suffixes_kernel); the list in order goes elsewhere, with its ties
    const u16* ext;
    u32 ext_bits; // that are sorted with the lower bits of the code: 32 in all at most
    u32* sufs_out;
    u8* ties;
    u32* open_count; // zeroed: suffixes in runs of one code and one ext, which are left open (resolve_runs_kernel) ...
    u32* open_sufs;  // ... them, run after run, with OWN_CODE ...
    u32* open_places; // ... and their places in the list, with RUN_START and RUN_TIED
    // the suffixes of buckets that do not fit, collected in list order
    u32* over_before; // [buckets]: of the buckets before this one whose number is the same in its upper bits (OVER_TILE buckets) ...
    u32* over_tiles;  // ... and of all that differ in those, by them
    u64* over_keys;
    u32* over_sufs;
    u32* over_open; // EXT: where they start in the list of open runs
    u32 over_slices; // workgroups a bucket
};

constexpr int STARTS_BLOCK = 256;

// Where the buckets start, by a search inside their top digit: a thread a bucket, and one more a workgroup for the end of its last. (As many
// dependent reads as the number of suffixes of the top digit has bits: 17 to 21 where the digits are alike, 30 at most. 10 to 90 us.)
__global__ __launch_bounds__(STARTS_BLOCK) void bucket_starts_kernel(BucketArgs a)
{
    __shared__ u32 s_start[STARTS_BLOCK];
    const u32 t = threadIdx.x;
    const u32 b = blockIdx.x * (STARTS_BLOCK - 1) + t;
    u32 lo = a.n;
    if (b < a.buckets) {
        const u32 least = b << a.low_bits, d = least >> a.top_shift;
        lo = a.top_base[d];
        u32 hi = least == d << a.top_shift ? lo : d + 1u == 1u << (32u - a.top_shift) ? a.n : a.top_base[d + 1];
        while (lo < hi) {
            const u32 mid = lo + (hi - lo) / 2;
            if (a.codes[mid] < least)
                lo = mid + 1;
            else
                hi = mid;
        }
    }
    s_start[t] = lo;
    if (b <= a.buckets)
        a.starts[b] = lo;
    __syncthreads();
    if (t + 1 < STARTS_BLOCK && b < a.buckets) {
        const u32 size = s_start[t + 1] - lo;
        if (size > BUCKET_MAX) {
            a.over_list[atomicAdd(&a.over[1], 1u)] = b;
            atomicAdd(&a.over[0], size);
            atomicMax(&a.over[2], size);
        }
    }
}

// EXT: what the members of a bucket are sorted by, the lower bits of the code and the upper ones of ext.
__device__ __forceinline__ u32 bucket_key(const BucketArgs& a, u32 code, u32 ext)
{
    return (code & ((1u << a.low_bits) - 1u)) << a.ext_bits | ext >> (16u - a.ext_bits);
}

// How an entry ties with its left neighbour, whose key is another one: suffixes that own one code have one string. The last `tail` suffixes, which run off
// the text inside it, come first in virtual order and tie with nobody.
__device__ __forceinline__ u32 tie_of_strings(bool same_code, u32 mine, u32 left, u32 tail)
{
    return same_code && (mine & OWN_CODE) && (mine & ~OWN_CODE) >= tail && (left & ~OWN_CODE) >= tail ? 1u : 0u;
}

// EXT: writes a bucket whose pairs (key, virtual position and OWN_CODE) pair_of(j) gives in order, and adds the runs of one key to the open ones.
constexpr u32 BUCKET_WAVES = BUCKET_ITEMS * BUCKET_BLOCK / WAVE;
static_assert(BUCKET_WAVES <= 2 * WAVE, "one wave scans them, two a lane");

template <typename Pairs>
__device__ __forceinline__ void write_bucket(const BucketArgs& a, u32 start, u32 size, u32* s_open, Pairs pair_of)
{
    constexpr int BLOCK = BUCKET_BLOCK, ITEMS = BUCKET_ITEMS;
    const u32 t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const u32 rounds = (size + BLOCK - 1) / BLOCK;
    u32* const sufs_out = a.sufs_out + start;
    u8* const ties = a.ties + start;
    u32 suf[ITEMS], member = 0, begins = 0, tied = 0; // bit k: the entry of round k is one of a run; begins one; ties with its left neighbour on one word
#pragma unroll
    for (int k = 0; k < ITEMS; ++k)
        if ((u32)k < rounds) {
            const u32 j = k * BLOCK + t, from = j < size ? j : size - 1u;
            const u64 pair = pair_of(from), left = pair_of(from > 0 ? from - 1u : 0u), right = pair_of(from + 1u < size ? from + 1u : from);
            const u32 key = (u32)(pair >> 32), before = (u32)(left >> 32);
            const bool follows = from > 0 && key == before, precedes = from + 1u < size && key == (u32)(right >> 32);
            const bool same_code = from > 0 && (key ^ before) >> a.ext_bits == 0;
            const bool in = j < size && (follows || precedes);
            const u32 x = virtual_to_suffix((u32)pair & ~OWN_CODE, a.n, a.tail);
            suf[k] = x | ((u32)pair & OWN_CODE);
            member |= (in ? 1u : 0u) << k;
            begins |= (follows ? 0u : 1u) << k;
            const u32 tie = tie_of_strings(same_code, (u32)pair, (u32)left, a.tail);
            if (j < size) { // (most of a run are copies, tied on both words, and stay as they stand: what is to be resolved is written as if they were)
                sufs_out[j] = x;
                ties[j] = (u8)(follows ? TIE_MOST_WORDS : tie);
            }
            tied |= tie << k;
            const u64 b = __ballot(in);
            if (lane == 0)
                s_open[k * (BLOCK / WAVE) + w] = (u32)__popcll(b);
        }
    __syncthreads();
    if (w == 0) {
        const u32 used = rounds * (BLOCK / WAVE);
        const u32 c0 = 2 * lane < used ? s_open[2 * lane] : 0u, c1 = 2 * lane + 1 < used ? s_open[2 * lane + 1] : 0u;
        const u32 incl = wave_incl_sum(c0 + c1), total = __shfl(incl, 63);
        u32 base = 0;
        if (lane == 0 && total)
            base = atomicAdd(a.open_count, total);
        base = __shfl(base, 0) + incl - c0 - c1;
        if (2 * lane < used)
            s_open[2 * lane] = base;
        if (2 * lane + 1 < used)
            s_open[2 * lane + 1] = base + c0;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ITEMS; ++k)
        if ((u32)k < rounds) {
            const bool in = (member >> k) & 1u;
            const u64 b = __ballot(in);
            if (in) {
                const u32 slot = s_open[k * (BLOCK / WAVE) + w] + (u32)__popcll(b & ((1ull << lane) - 1ull));
                a.open_sufs[slot] = suf[k];
                a.open_places[slot] = (start + k * BLOCK + t) | ((begins >> k) & 1u ? RUN_START | ((tied >> k) & 1u ? RUN_TIED : 0u) : 0u);
            }
        }
}

// One bucket a workgroup. Its suffixes go to 4096 cells by the next bits of their codes, in whatever order they arrive, and everyone is compared with the
// others in its cell, of which there are one or two, by the whole code and its place in the order of the text. What bounds it are vector
// instructions: all threads do the same for whole rounds, what is past the end of the bucket going to a cell of its own. Buckets with a long
// cell, one string hundreds of times, are left to finish_crowded_kernel.
template <bool EXT>
__global__ __launch_bounds__(BUCKET_BLOCK, 2 * BUCKET_BLOCK / 256) void finish_buckets_kernel(BucketArgs a)
{
    constexpr int BLOCK = BUCKET_BLOCK, ITEMS = BUCKET_ITEMS, CAP = BUCKET_MAX, CELLS = 1 << CELLS_LOG2;
    constexpr int PER = CELLS / BLOCK; // cells of a thread in the scan
    static_assert(PER >= 2 && PER % 2 == 0 && CELLS % BLOCK == 0, "the counters are scanned by words of two");
    __shared__ u64 s_pair[CAP + WAVE]; // code, virtual position; the last ones hold nothing
    __shared__ __align__(16) u32 s_cell[CELLS / 2 + 4]; // two to a word: members of a cell, then where they start
    __shared__ u32 s_sum[BLOCK / WAVE];
    __shared__ u32 s_crowded;
    __shared__ u32 s_open[EXT ? BUCKET_WAVES : 1];
    const u32 t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const u32 start = a.starts[blockIdx.x], size = a.starts[blockIdx.x + 1] - start;
    if (size < (EXT ? 1u : 2u) || size > (u32)CAP)
        return;
    const u32 rounds = (size + BLOCK - 1) / BLOCK;
    const u32 key_bits = a.low_bits + (EXT ? a.ext_bits : 0u);
    const u32 drop = key_bits > (u32)CELLS_LOG2 ? key_bits - CELLS_LOG2 : 0u;
    const u32* const codes = a.codes + start;
    const u32* const sufs = a.sufs + start;
    u32 key[ITEMS], val[ITEMS], cell[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k)
        if ((u32)k < rounds) {
            const u32 i = k * BLOCK + t, from = i < size ? i : size - 1u;
            key[k] = codes[from];
            val[k] = sufs[from];
            if constexpr (EXT)
                key[k] = bucket_key(a, key[k], a.ext[start + from]);
        }
    for (int i = t; i < CELLS / 2 + 1; i += BLOCK)
        s_cell[i] = 0;
    if (t == 0)
        s_crowded = 0;
    __syncthreads();
    u32 at[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k)
        if ((u32)k < rounds) {
            cell[k] = k * BLOCK + t < size ? (key[k] >> drop) & (u32)(CELLS - 1) : (u32)CELLS;
            at[k] = atomicAdd(&s_cell[cell[k] / 2], 1u << (cell[k] & 1u) * 16u);
        }
    __syncthreads();
    u32 mine = 0, most = 0;
#pragma unroll
    for (int q = 0; q < PER; q += 2) {
        const u32 v = s_cell[(t * PER + q) / 2], odd = v >> 16, even = v & 0xFFFFu;
        mine += even + odd;
        most = most > even ? most : even;
        most = most > odd ? most : odd;
    }
    if (most > CELL_MAX)
        s_crowded = 1;
    const u32 incl = wave_incl_sum(mine);
    if (lane == 63u)
        s_sum[w] = incl;
    __syncthreads();
    if (s_crowded) {
        if (t == 0)
            a.crowded_list[atomicAdd(a.crowded, 1u)] = blockIdx.x;
        return;
    }
    u32 run = incl - mine;
#pragma unroll
    for (u32 ww = 0; ww < (u32)BLOCK / WAVE; ++ww)
        run += ww < w ? s_sum[ww] : 0u;
#pragma unroll
    for (int q = 0; q < PER; q += 2) {
        u32* const p = &s_cell[(t * PER + q) / 2];
        const u32 v = *p, second = run + (v & 0xFFFFu);
        *p = run | (second << 16);
        run = second + (v >> 16);
    }
    if (t == 0)
        s_cell[CELLS / 2] = size;
    __syncthreads();
    const u16* const starts = reinterpret_cast<const u16*>(s_cell);
#pragma unroll
    for (int k = 0; k < ITEMS; ++k)
        if ((u32)k < rounds) {
            const u32 virt = suffix_to_virtual(val[k] & ~OWN_CODE, a.n, a.tail);
            const u32 to = starts[cell[k]] + ((at[k] >> (cell[k] & 1u) * 16u) & 0xFFFFu);
            s_pair[cell[k] == (u32)CELLS ? CAP + lane : to] = (u64)key[k] << 32 | virt | (val[k] & OWN_CODE);
        }
    __syncthreads();
    u64 pair[EXT ? ITEMS : 1];
    u32 to_place[EXT ? ITEMS : 1];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const u32 j = k * BLOCK + t;
        if (j < size) {
            const u64 mine_pair = s_pair[j];
            const u32 code = (u32)(mine_pair >> 32), c = (code >> drop) & (u32)(CELLS - 1);
            const u32 from = starts[c], to = starts[c + 1];
            u32 place = from;
            if (to - from > 1u)
                for (u32 i = from; i < to; ++i)
                    place += s_pair[i] < mine_pair ? 1u : 0u;
            if constexpr (EXT) {
                pair[k] = mine_pair;
                to_place[k] = place;
            } else {
                a.codes[start + place] = code;
                a.sufs[start + place] = virtual_to_suffix((u32)mine_pair & ~OWN_CODE, a.n, a.tail) | ((u32)mine_pair & OWN_CODE);
            }
        }
    }
    if constexpr (EXT) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (k * BLOCK + t < size)
                s_pair[to_place[k]] = pair[k];
        __syncthreads();
        write_bucket(a, start, size, s_open, [&](u32 j) { return s_pair[j]; });
    }
}

// The crowded buckets, one at a time a workgroup: stable LSD passes over digits of eight bits, ranked as in onesweep_kernel, whose tile the bucket is.
constexpr u32 CROWDED_BLOCKS = 1024;

template <bool EXT>
__global__ __launch_bounds__(BUCKET_BLOCK) void finish_crowded_kernel(BucketArgs a)
{
    constexpr int DB = RADIX_BITS, BLOCK = BUCKET_BLOCK, ITEMS = BUCKET_ITEMS, CAP = BUCKET_MAX, WAVES = BLOCK / WAVE, BINS = 1 << DB;
    constexpr int PER = 4; // bins of a thread in the scan
    constexpr int WORDS = WAVES * BINS > 2 * CAP ? WAVES * BINS : 2 * CAP;
    static_assert(BINS <= BLOCK * PER, "the bins are scanned at once");
    __shared__ __align__(16) u32 s_mem[WORDS]; // the counters of a pass, [wave][bin]; then the pairs in the order of it
    __shared__ u32 s_carry[WAVES];
    __shared__ u32 s_open[EXT ? BUCKET_WAVES : 1];
    const u32 t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const u32 crowded = *a.crowded;
    for (u32 at = blockIdx.x; at < crowded; at += gridDim.x) {
        const u32 b = a.crowded_list[at], start = a.starts[b], size = a.starts[b + 1] - start;
        const u32 rounds = (size + BLOCK - 1) / BLOCK; // pairs of a thread: consecutive ones a wave, so that their order is that of the bucket
        const u32 first = w * rounds * WAVE + lane;
        u32 key[ITEMS], val[ITEMS], pos[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if ((u32)k < rounds) {
                const u32 i = first + k * WAVE;
                key[k] = ~0u; // behind every real pair
                val[k] = 0;
                if (i < size) {
                    key[k] = a.codes[start + i];
                    val[k] = a.sufs[start + i];
                    if constexpr (EXT)
                        key[k] = bucket_key(a, key[k], a.ext[start + i]);
                }
            }
        const u32 key_bits = a.low_bits + (EXT ? a.ext_bits : 0u);
        for (u32 shift = 0; shift < key_bits; shift += DB) {
            const u32 bits = key_bits - shift < (u32)DB ? key_bits - shift : (u32)DB;
            for (int i = t; i < WAVES * BINS / 4; i += BLOCK)
                reinterpret_cast<uint4*>(s_mem)[i] = make_uint4(0u, 0u, 0u, 0u);
            __syncthreads();
            u32* const whist = s_mem + w * BINS;
#pragma unroll
            for (int k = 0; k < ITEMS; ++k)
                if ((u32)k < rounds)
                    pos[k] = rank_in_wave<DB>(__builtin_amdgcn_ubfe(key[k], shift, bits), whist);
            __syncthreads();
            // where every wave's pairs of a digit go: all smaller digits, and this one in the waves before
            const int bin = (int)t * PER;
            u32 before[WAVES][PER], total[PER] = {};
            if (bin < BINS)
#pragma unroll
                for (int ww = 0; ww < WAVES; ++ww) {
                    const uint4 v = *reinterpret_cast<const uint4*>(s_mem + ww * BINS + bin);
                    const u32 c[PER] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int q = 0; q < PER; ++q) {
                        before[ww][q] = total[q];
                        total[q] += c[q];
                    }
                }
            const u32 mine = total[0] + total[1] + total[2] + total[3], incl = wave_incl_sum(mine);
            if (lane == 63u)
                s_carry[w] = incl;
            __syncthreads();
            u32 run = incl - mine;
            for (u32 ww = 0; ww < w; ++ww)
                run += s_carry[ww];
            if (bin < BINS) {
                u32 from[PER];
#pragma unroll
                for (int q = 0; q < PER; ++q) {
                    from[q] = run;
                    run += total[q];
                }
#pragma unroll
                for (int ww = 0; ww < WAVES; ++ww)
                    *reinterpret_cast<uint4*>(s_mem + ww * BINS + bin) =
                        make_uint4(from[0] + before[ww][0], from[1] + before[ww][1], from[2] + before[ww][2], from[3] + before[ww][3]);
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < ITEMS; ++k)
                if ((u32)k < rounds)
                    pos[k] += whist[__builtin_amdgcn_ubfe(key[k], shift, bits)];
            __syncthreads();
#pragma unroll
            for (int k = 0; k < ITEMS; ++k)
                if ((u32)k < rounds) {
                    s_mem[pos[k]] = key[k];
                    s_mem[CAP + pos[k]] = val[k];
                }
            __syncthreads();
            const bool last = shift + DB >= key_bits;
            if (EXT && last) {
                write_bucket(a, start, size, s_open, [&](u32 j) {
                    const u32 v = s_mem[CAP + j];
                    return (u64)s_mem[j] << 32 | suffix_to_virtual(v & ~OWN_CODE, a.n, a.tail) | (v & OWN_CODE);
                });
                __syncthreads();
                break;
            }
#pragma unroll
            for (int k = 0; k < ITEMS; ++k)
                if ((u32)k < rounds) {
                    const u32 i = last ? k * BLOCK + t : first + k * WAVE;
                    key[k] = s_mem[i];
                    val[k] = s_mem[CAP + i];
                    if (last && i < size) {
                        a.codes[start + i] = key[k];
                        a.sufs[start + i] = val[k];
                    }
                }
            __syncthreads();
        }
    }
}

// ---- buckets that do not fit ----

#ifndef CSA_OVER_TILE
#define CSA_OVER_TILE 1024
#endif
constexpr int OVER_TILE = CSA_OVER_TILE;
// A workgroup moves OVER_SLICE suffixes of a large bucket, a sixteenth of a small one; of many buckets, one of which is much larger than the others, more, so that there are no
// more than OVER_BLOCKS workgroups or 16 a bucket. (10^8 letters with 6 % in a run of one letter and 3 % in one of another, 16 workgroups a bucket whatever its size: 675 us there and 804 back, 37 and 36 now.)
#ifndef CSA_OVER_SLICE
#define CSA_OVER_SLICE 4096
#endif
constexpr u32 OVER_SLICE = CSA_OVER_SLICE, OVER_BLOCKS = 1u << 15;

__global__ __launch_bounds__(OVER_TILE) void over_before_kernel(BucketArgs a)
{
    __shared__ u32 s_sum[OVER_TILE / WAVE];
    const u32 t = threadIdx.x, lane = t & 63u, w = t >> 6;
    const u32 b = blockIdx.x * OVER_TILE + t;
    const u32 size = b < a.buckets ? a.starts[b + 1] - a.starts[b] : 0u;
    const u32 mine = size > BUCKET_MAX ? size : 0u, incl = wave_incl_sum(mine);
    if (lane == 63u)
        s_sum[w] = incl;
    __syncthreads();
    u32 before = incl - mine, all = 0;
    for (u32 ww = 0; ww < OVER_TILE / WAVE; ++ww) {
        before += ww < w ? s_sum[ww] : 0u;
        all += s_sum[ww];
    }
    if (b < a.buckets)
        a.over_before[b] = before;
    if (t == 0)
        a.over_tiles[blockIdx.x] = all;
    if (a.over_open && blockIdx.x == 0 && t == 0)
        *a.over_open = atomicAdd(a.open_count, a.over[0]);
}

// The suffixes of the buckets in over_list to their places in over_keys and over_sufs, or back from there (BACK), over_slices workgroups a bucket.
// EXT: by the code and ext; on the way back the ties follow from those.
template <bool BACK, bool EXT>
__global__ __launch_bounds__(256) void over_move_kernel(BucketArgs a)
{
    __shared__ u32 s_sum[256 / WAVE];
    const u32 t = threadIdx.x, b = a.over_list[blockIdx.x / a.over_slices], start = a.starts[b], size = a.starts[b + 1] - start;
    const u32 per = (size + a.over_slices - 1) / a.over_slices, first = blockIdx.x % a.over_slices * per, last = size - first < per ? size : first + per;
    if (first >= size)
        return;
    u32 earlier = 0;
    for (u32 i = t; i < b / OVER_TILE; i += 256)
        earlier += a.over_tiles[i];
    const u32 sum = wave_reduce_sum(earlier);
    if ((t & 63u) == 0)
        s_sum[t / WAVE] = sum;
    __syncthreads();
    u32 to = a.over_before[b];
    for (u32 ww = 0; ww < 256 / WAVE; ++ww)
        to += s_sum[ww];
    for (u32 i = first + t; i < last; i += 256) {
        if constexpr (!BACK) {
            a.over_keys[to + i] = EXT ? (u64)a.codes[start + i] << 16 | a.ext[start + i] : (u64)a.codes[start + i];
            a.over_sufs[to + i] = a.sufs[start + i];
        } else if constexpr (!EXT) {
            a.codes[start + i] = (u32)a.over_keys[to + i];
            a.sufs[start + i] = a.over_sufs[to + i];
        } else {
            const u64 key = a.over_keys[to + i];
            const u32 v = a.over_sufs[to + i], x = v & ~OWN_CODE;
            const bool follows = i > 0 && a.over_keys[to + i - 1] == key;
            u32 tie = 0;
            if (i > 0 && a.over_keys[to + i - 1] >> 16 == key >> 16) {
                const u32 left = a.over_sufs[to + i - 1] & ~OWN_CODE;
                tie = tie_of_strings(true, suffix_to_virtual(x, a.n, a.tail) | (v & OWN_CODE), suffix_to_virtual(left, a.n, a.tail), a.tail);
            }
            a.sufs_out[start + i] = x;
            a.ties[start + i] = (u8)(follows ? TIE_MOST_WORDS : tie);
            const u32 slot = *a.over_open + to + i; // (all of them are listed, runs or not)
            a.open_sufs[slot] = v;
            a.open_places[slot] = (start + i) | (follows ? 0u : RUN_START | (tie ? RUN_TIED : 0u));
        }
    }
}

} // namespace csa
