// Host side of the library: the handle, the radix-sort driver, the generation loop and the C ABI
// declared in include/cascade_hip.h. gfx950 only.
#include "../../include/cascade_hip.h"

#include "bucket_sort.hpp"
#include "chains.hpp"
#include "coded_keys.hpp"
#include "copies.hpp"
#include "device_pool.hpp"
#include "device_utils.hpp"
#include "doubling.hpp"
#include "messages.hpp"
#include "partition_ids.hpp"
#include "pipeline_steps.hpp"
#include "radix_sort.hpp"
#include "short_text.hpp"
#include "word_keys.hpp"

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <dlfcn.h>
#include <mutex>
#include <vector>

using namespace csa;

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

#define HIP_TRY(expr)                                                                                  \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            return fail(CSA_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)

// Named ranges for a profiler's timeline, one per partition step and per generation: the counterpart of the NVTX ranges
// the reference opens under -DPROFILE (include/profile.hpp:19-80; PROFILE_SCOPE_FMT at src/GPU_SACA.cu:1114,1717,2004,2111).
// The roctx library is looked up at run time when csa_enable_profile_ranges(1) asks for it, so the library neither
// links against a profiler nor pays for ranges nobody reads.
#ifndef HIPEMU
struct ProfileRanges {
    std::mutex mu;
    bool tried = false;
    int (*push)(const char*) = nullptr;
    int (*pop)() = nullptr;
    bool enabled = false;
} g_ranges;

int enable_ranges(bool on)
{
    std::lock_guard<std::mutex> lock(g_ranges.mu);
    if (on && !g_ranges.tried) {
        g_ranges.tried = true;
        for (const char* name : {"librocprofiler-sdk-roctx.so", "librocprofiler-sdk-roctx.so.1", "libroctx64.so", "libroctx64.so.4"}) {
            if (void* lib = dlopen(name, RTLD_NOW | RTLD_GLOBAL)) {
                g_ranges.push = reinterpret_cast<int (*)(const char*)>(dlsym(lib, "roctxRangePushA"));
                g_ranges.pop = reinterpret_cast<int (*)()>(dlsym(lib, "roctxRangePop"));
                if (g_ranges.push && g_ranges.pop)
                    break;
                g_ranges.push = nullptr;
                g_ranges.pop = nullptr;
            }
        }
    }
    g_ranges.enabled = on && g_ranges.push && g_ranges.pop;
    return on && !g_ranges.enabled ? 1 : 0;
}
#else
struct ProfileRanges {
    int (*push)(const char*) = nullptr;
    int (*pop)() = nullptr;
    bool enabled = false;
} g_ranges;
int enable_ranges(bool) { return 1; }
#endif

struct RangeScope {
    bool open = false;
    explicit RangeScope(const char* fmt, ...)
    {
        if (!g_ranges.enabled)
            return;
        char name[128];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(name, sizeof(name), fmt, ap);
        va_end(ap);
        g_ranges.push(name);
        open = true;
    }
    void close()
    {
        if (open)
            g_ranges.pop();
        open = false;
    }
    ~RangeScope() { close(); }
    RangeScope(const RangeScope&) = delete;
    RangeScope& operator=(const RangeScope&) = delete;
};

// tile shape of the radix pass; overridable at build time for tuning runs
#ifndef CSA_SORT_BLOCK
#define CSA_SORT_BLOCK 512
#endif
#ifndef CSA_SORT_ITEMS
#define CSA_SORT_ITEMS 16
#endif
#ifndef CSA_SORT32_ITEMS
#define CSA_SORT32_ITEMS CSA_SORT_ITEMS
#endif
constexpr int SORT_BLOCK = CSA_SORT_BLOCK;
constexpr int SORT_ITEMS = CSA_SORT_ITEMS;
constexpr int SORT32_ITEMS = CSA_SORT32_ITEMS; // pairs per thread when the keys are 32-bit (same LDS bytes at twice the items)
constexpr int SORT_TILE = SORT_BLOCK * SORT_ITEMS;
static_assert(SORT32_ITEMS >= SORT_ITEMS, "the look-back words are sized for tiles of SORT_TILE pairs or more");
// Long passes use workgroups of twice the threads: the runs of a digit a tile writes are twice as long, so fewer of the
// lines it writes are shared with a tile whose L2 is another one. One such workgroup fills a CU's LDS. Measured per
// sort of the 1B-token workload: 125.3 -> 121.4 ms by arrival (the default order, where neighbouring tiles run on
// different XCDs), 119.3 -> 117.4 ms under the chunked order, whose chunks keep their length in pairs (half as many
// of the larger tiles: with the full count the wide workgroups gained nothing there).
#ifndef CSA_SORT_WIDE_BLOCK
#define CSA_SORT_WIDE_BLOCK 1024
#endif
#ifndef CSA_SORT_WIDE_MIN
#define CSA_SORT_WIDE_MIN (1u << 24)
#endif
constexpr int SORT_WIDE_BLOCK = CSA_SORT_WIDE_BLOCK;
constexpr u32 SORT_WIDE_MIN = CSA_SORT_WIDE_MIN; // fewest pairs of a pass that uses the wide workgroups
static_assert(SORT_WIDE_BLOCK >= SORT_BLOCK, "the look-back words are sized for tiles of SORT_TILE pairs or more");
#ifndef CSA_RANK_BLOCK
#define CSA_RANK_BLOCK 256
#endif
#ifndef CSA_RANK_ITEMS
#define CSA_RANK_ITEMS 4
#endif
constexpr int RANK_BLOCK = CSA_RANK_BLOCK;
constexpr int RANK_ITEMS = CSA_RANK_ITEMS;
constexpr int RANK_TILE = RANK_BLOCK * RANK_ITEMS;
// Groups of up to SMALL_MAXG suffixes are sorted inside one tile of the small-group kernel; the larger ones go through
// the radix sort. A list of mostly short groups (at most SMALL_AVG_LIMIT members per group on average: token corpora)
// takes the higher limit SMALL_MAXG_HI, which leaves fewer members to the radix passes (1B-token workload: 117.5 ->
// 115.4 ms per sort). A list of long groups (small alphabets, runs) keeps the lower one: the tile's halo of SMALL_MAXG
// elements on either side and the longer member loops only cost there (4-letter workload sorted from one K-gram word:
// +6 % with the higher limit). The adversarial workload's generation 1 averages 16.5 members per group, most of them in
// groups of 65 to 256: the higher limit takes 37 M members off its radix passes (31.1 -> 29.0 ms), hence 32.
#ifndef CSA_SMALL_MAXG
#define CSA_SMALL_MAXG 64
#endif
#ifndef CSA_SMALL_MAXG_HI
#define CSA_SMALL_MAXG_HI 256
#endif
#ifndef CSA_SMALL_AVG_LIMIT
#define CSA_SMALL_AVG_LIMIT 32
#endif
// tile of the small-group kernel and of the counting / applying kernels behind it (measured per sort of the 1B-token
// workload with 16-byte loads in the applying kernel: 256 x 8 109.4 ms, 256 x 4 106.5, 512 x 4 106.2, 1024 x 4 106.7,
// 512 x 2 106.3, 512 x 8 108.8, 128 x 8 110.4)
#ifndef CSA_SMALL_BLOCK
#define CSA_SMALL_BLOCK 512
#endif
#ifndef CSA_SMALL_ITEMS
#define CSA_SMALL_ITEMS 4
#endif
constexpr int SMALL_BLOCK = CSA_SMALL_BLOCK;
constexpr int SMALL_ITEMS = CSA_SMALL_ITEMS;
constexpr int SMALL_TILE = SMALL_BLOCK * SMALL_ITEMS;
constexpr int SMALL_MAXG = CSA_SMALL_MAXG;
constexpr int SMALL_MAXG_HI = CSA_SMALL_MAXG_HI;
constexpr u32 SMALL_AVG_LIMIT = CSA_SMALL_AVG_LIMIT;
static_assert(SMALL_MAXG_HI >= SMALL_MAXG, "the higher group limit is the higher one");
constexpr u32 TICKET_POOL = 4096;
constexpr u32 PROBE_FEW = 1u << 15;           // suffixes that are probed, whose table ...
constexpr u64 PROBE_TABLE = 2ull * PROBE_FEW; // ... is one of the handle's own
constexpr u64 CODE_TABLE_WORDS = SYMBOLS + RESOLVE_MARK_WORDS + PROBE_WORDS + 2 * PROBE_TABLE + SYMBOLS + 4; // symbol counts, marks, ProbeCounts, its table, shares (and entry [SYMBOLS])
// Texts of at least this many symbols are probed before they are sorted by codes (probe_codes_kernel, 12 us with its round trip). Shorter
// ones have no runs of one code that are too long for a tile, out of order and not planted: strings of four symbols that are
// rare enough to share a code with others can come up 256 times from there on. Generation 0 of records of four symbols, one of
// them of many values, in us on K-gram keys, on codes and with the choice: 2^16.9 symbols 173, 189, -; 2^18 185, 419, 211;
// 2^18.9 202, 423, 232; of independent symbols 172, 142, -; 184, 151, 165; 203, 165, 180.
#ifndef CSA_PROBE_MIN
#define CSA_PROBE_MIN (1u << 17)
#endif
constexpr u32 PROBE_MIN = CSA_PROBE_MIN;
// Shorter texts are coded while the host waits for the probe, which takes about as long, longer ones when it has advised that: 2^22
// independent symbols 353 us coded ahead, 364 else, and 2^22 symbols of phrases, which go by K-grams then, 499 and 463.
#ifndef CSA_CODE_AHEAD_MAX
#define CSA_CODE_AHEAD_MAX (1u << 22)
#endif
constexpr u32 CODE_AHEAD_MAX = CSA_CODE_AHEAD_MAX;
static_assert(PROBE_MIN >= 32, "two suffixes are the fewest that can share a code");
constexpr u32 PINNED_HIST = 32;        // host mirror: words [0, 16) mirror the device counters, [16, 32) single values, then the histograms
constexpr u32 MSG_OFF_WORDS = 32769;   // p + 1 outbox counters, p <= 32768
constexpr int EVENT_POOL = 2 * CSA_MAX_GENERATIONS * MAX_PASSES * 2;

// Lists of at least this many suffixes update rank[] through two radix passes on the text position instead of
// scattering 4-byte writes over the whole array.
#ifndef CSA_DEFER_MIN
#define CSA_DEFER_MIN (1u << 23)
#endif
// Lists of at least this many suffixes may take the dense form of a later generation (the whole partition sorted again
// by keys read in text order); below it the generation is over before the choice matters. Smaller in test builds.
#ifndef CSA_DENSE_MIN
#define CSA_DENSE_MIN (1u << 16)
#endif
constexpr u32 DENSE_MIN = CSA_DENSE_MIN;
constexpr u32 XCD_CHUNK = 16;
// Windows of rank[] that the last step of generation 0's bucketed update assembles in LDS (1 << 14 positions; twice
// that on the largest partitions, whose two passes cover 16 position bits at most). Smaller in test builds, so that
// short lists go through the passes too.
#ifndef CSA_PLACE_WINDOW_LOG2
#define CSA_PLACE_WINDOW_LOG2 14
#endif
constexpr int PLACE_WINDOW_LOG2 = CSA_PLACE_WINDOW_LOG2;
static_assert(PLACE_WINDOW_LOG2 >= 1 && PLACE_WINDOW_LOG2 <= 14, "the placement kernel holds a window of 1 << 14 or 1 << 15 ranks");
constexpr u32 DEFER_MIN = CSA_DEFER_MIN;
// Later generations: when at least half of the sorted list changes its rank, and at least WINDOW_MIN_CHANGED
// suffixes in all, the rank writes of the generation are bucketed into windows of 1 << WINDOW_LOG2 positions of
// rank[] first. Partitions that fit one window never need it.
#ifndef CSA_WINDOW_LOG2
#define CSA_WINDOW_LOG2 23
#endif
#ifndef CSA_WINDOW_MIN_CHANGED
#define CSA_WINDOW_MIN_CHANGED (1u << 22)
#endif
constexpr int WINDOW_LOG2 = CSA_WINDOW_LOG2;
constexpr u32 WINDOW_MIN_CHANGED = CSA_WINDOW_MIN_CHANGED;
// rank-order scatter of a whole partition: partitions of at least SCATTER_WINDOW_MIN suffixes are first grouped by
// windows of 2^SCATTER_WINDOW_LOG2 ranks (40 MB of output, which the last-level cache holds)
#ifndef CSA_SCATTER_WINDOW_LOG2
#define CSA_SCATTER_WINDOW_LOG2 23
#endif
#ifndef CSA_SCATTER_WINDOW_MIN
#define CSA_SCATTER_WINDOW_MIN (1u << 25)
#endif
constexpr u32 SCATTER_WINDOW_LOG2 = CSA_SCATTER_WINDOW_LOG2;
constexpr u64 SCATTER_WINDOW_MIN = CSA_SCATTER_WINDOW_MIN;
// smallest cohort for which the message join builds a directory over the suffix-ordered cohort first
#ifndef CSA_JOIN_DIR_MIN
#define CSA_JOIN_DIR_MIN 4096u
#endif


int bit_length(u64 v)
{
    int b = 0;
    while (v) {
        ++b;
        v >>= 1;
    }
    return b;
}

} // namespace

// ---- scratch of csa_radix_sort_pairs_static_dev, the one entry point that allocates nothing ----
// One array per device, part of the code object: it exists from the moment the library is loaded until the process
// ends. Host code never uses the name `scratch` as an address (on the host it is a stand-in, not device memory): the
// address on the current device comes from hipGetSymbolAddress, once per device (static_scratch below), and everything
// that needs the memory takes that pointer.
namespace {
constexpr u64 STATIC_SORT_MAX = CSA_STATIC_SORT_MAX_PAIRS;
constexpr u64 STATIC_TILES = (STATIC_SORT_MAX + SORT_TILE - 1) / SORT_TILE;
constexpr u64 STATIC_LB_TILE_WORDS = STATIC_TILES * RADIX_BINS;                                  // per pass
constexpr u64 STATIC_LB_WORDS = STATIC_LB_TILE_WORDS + (STATIC_TILES / LB_GROUP + 1) * RADIX_BINS; // per pass, groups included
constexpr u64 align256(u64 v) { return (v + 255u) & ~(u64)255u; }
// layout: the ping-pong partners of the caller's arrays, then the control words, which every call clears
constexpr u64 STATIC_OFF_KEYS = 0;
constexpr u64 STATIC_OFF_VALS = align256(STATIC_OFF_KEYS + STATIC_SORT_MAX * sizeof(u64));
constexpr u64 STATIC_OFF_CONTROL = align256(STATIC_OFF_VALS + STATIC_SORT_MAX * sizeof(u32));
constexpr u64 STATIC_OFF_LOOKBACK = STATIC_OFF_CONTROL;
constexpr u64 STATIC_OFF_GHIST = align256(STATIC_OFF_LOOKBACK + MAX_PASSES * STATIC_LB_WORDS * sizeof(u64));
constexpr u64 STATIC_OFF_TICKETS = align256(STATIC_OFF_GHIST + MAX_PASSES * RADIX_BINS * sizeof(u32));
constexpr u64 STATIC_OFF_ERR = align256(STATIC_OFF_TICKETS + MAX_PASSES * sizeof(u32));
constexpr u64 STATIC_OFF_DIGIT_BASE = align256(STATIC_OFF_ERR + sizeof(u32)); // written before it is read: not cleared
constexpr u64 STATIC_CONTROL_END = STATIC_OFF_DIGIT_BASE;
constexpr u64 STATIC_SCRATCH_BYTES = align256(STATIC_OFF_DIGIT_BASE + MAX_PASSES * RADIX_BINS * sizeof(u32));
} // namespace

static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

// What a handle was created for (csa_create: everything; csa_create_steps: everything but the resident sort).
constexpr u32 KIND_RESIDENT = 1u;

struct csa_handle {
    int device = 0;
    u64 cap = 0;
    int key_words = 1;
    u32 kinds = 0;
    int cus = 0; // compute units of the device
    // One block of device memory for everything that scales with the partition. The resident sort uses it under a fixed
    // carve-up made at creation (the arrays below); every other entry point takes and returns columns of it as it goes
    // (device_pool.hpp). A handle serves one call at a time, so the two never meet.
    unsigned char* block = nullptr;
    DevicePool pool;
    u64 last_high_water = 0; // of the last call that used the pool
    u64* key[3] = {nullptr, nullptr, nullptr};
    u32* idx[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    u32* gid = nullptr;
    u32* rank = nullptr;
    u32* gprim[2] = {nullptr, nullptr};
    u32* gstart[2] = {nullptr, nullptr};
    // The workspace: tables whose size follows the number of tiles, and small fixed ones.
    u64* lookback = nullptr;
    u64 lookback_words = 0;
    u64 lookback_tile_words = 0;
    u32* code_tables = nullptr; // resident sort: symbol counts, marks of codes, shares of the symbols (sort_by_codes)
    u32* tile_tables = nullptr; // rerank: [rank_tiles_cap][4] tile aggregates, the same of prefixes, [rank_tiles_cap] splits,
                                // [RERANK_SLABS][5] slab totals
    u64 rank_tiles_cap = 0;
    u32* ghist = nullptr;      // [MAX_PASSES][256]
    u32* digit_base = nullptr; // [MAX_PASSES][256]
    u32* tickets = nullptr;    // [TICKET_POOL]
    u32 ticket_next = 0;
    u32* counts = nullptr; // [2] error flag; [3] verifier flag; [4] members of large groups; [6..7] tied entries;
                           // [8..9] active-set size of a step; [10..11] unserved members; [12..13] pill receipts;
                           // [14] incoherent pill receipts
    u32* msg_off = nullptr; // [MSG_OFF_WORDS]: the outbox counters of the slab-shaped steps
    u32* h_pinned = nullptr; // host mirror: [0..15] counts, [16 ..) histogram
    u32 epoch = 0;
    u32 tile_order = TILES_BY_ARRIVAL;           // how the radix passes number their tiles (radix_sort.hpp), in use
    u32 tile_order_exclusive = TILES_BY_ARRIVAL; // the order after csa_set_device_exclusive
    u32 xcd_chunk = XCD_CHUNK;                   // tiles of a radix pass that one XCD takes in a row under TILES_STATIC_CHUNKS
    u32 defer_min = DEFER_MIN; // lists at least this long use the bucketed rank update (csa_set_tuning)
    u32 window_min_changed = WINDOW_MIN_CHANGED; // csa_set_tuning (0xFFFFFFFF: never)
    u32 expect_presorted = 0; // csa_set_tuning: 1 = every generation first runs as if its large groups were in order already
    u32 settle = 1;       // csa_set_tuning: lists are settled without ranks, short texts ranked by counting; 0 once a threshold of the rank updates has been set
    u32 pack_symbols = 1; // csa_set_tuning: texts over small alphabets start from keys of many symbols (packed_text.hpp)
    csa_step_result last_step = {};              // counters of the last partition step (csa_last_step_result)
    std::vector<hipEvent_t> events;
    hipEvent_t ev_gen[CSA_MAX_GENERATIONS + 2] = {};
    bool ev_gen_ready = false;
};

namespace {

struct Launch {
    csa_handle* h;
    hipStream_t stream;
    u32 flags;
    csa_stats* stats;
    std::vector<std::pair<int, u64>> timed; // (first event index, pairs) of each timed radix launch
    int events_used = 0;
};

void add_table(TableGroup& g, void* to, const void* from, u64 bytes)
{
    g.to[g.count] = static_cast<u32*>(to);
    g.from[g.count] = static_cast<const u32*>(from);
    g.words[g.count++] = (u32)(bytes / sizeof(u32));
}

// One launch for all of them: a workgroup for every 1024 words of the largest.
int move_tables(const TableGroup& g, hipStream_t s)
{
    u32 most = 1;
    for (u32 k = 0; k < g.count; ++k)
        most = g.words[k] > most ? g.words[k] : most;
    hipLaunchKernelGGL(move_tables_kernel, dim3((most + 1023u) / 1024u), dim3(256), 0, s, g);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

int move_table(void* to, const void* from, u64 bytes, hipStream_t s)
{
    TableGroup g = {};
    add_table(g, to, from, bytes);
    return move_tables(g, s);
}

int next_ticket(Launch& L, u32** out)
{
    csa_handle* h = L.h;
    if (h->ticket_next == TICKET_POOL) {
        HIP_TRY(hipMemsetAsync(h->tickets, 0, TICKET_POOL * sizeof(u32), L.stream));
        h->ticket_next = 0;
    }
    *out = h->tickets + h->ticket_next++;
    return CSA_OK;
}

u32 next_epoch(csa_handle* h)
{
    h->epoch++;
    if (h->epoch >= (1u << 30)) { // never in practice; stale words would need a clear before reuse
        (void)hipMemset(h->lookback, 0, h->lookback_words * sizeof(u64));
        h->epoch = 1;
    }
    return h->epoch;
}

u32 hist_blocks(u64 items_per_block, u64 n)
{
    u64 blocks = (n + items_per_block - 1) / items_per_block;
    if (blocks > 2048)
        blocks = 2048;
    return (u32)(blocks ? blocks : 1);
}

// How the radix passes of a call number their tiles (radix_sort.hpp).
struct TileOrder {
    u32 order;     // TILES_BY_ARRIVAL or TILES_STATIC_CHUNKS
    u32 xcd_chunk; // tiles of SORT_TILE pairs that one XCD takes in a row under TILES_STATIC_CHUNKS
};

// tile order of a pass over a.n pairs in tiles of `tile` pairs
void set_tile_order(const TileOrder& o, OnesweepArgs& a, u32 tile)
{
    a.tiles = (u32)(((u64)a.n + tile - 1) / tile);
    a.order = o.order;
    // the chunk length is meant in tiles of SORT_TILE pairs: larger tiles, proportionally fewer per chunk
    const u32 chunk = (u32)((u64)o.xcd_chunk * SORT_TILE / tile);
    a.xcd_chunk = chunk ? chunk : 1u;
}

TileOrder tile_order_of(const csa_handle* h) { return TileOrder{h->tile_order, h->xcd_chunk}; }

bool wide_workgroups(const OnesweepArgs& a)
{
    return SORT_WIDE_BLOCK > SORT_BLOCK && a.n >= SORT_WIDE_MIN;
}

template <int SRC, int BLOCK, bool VALS>
void launch_onesweep_shape(const TileOrder& o, OnesweepArgs& a, hipStream_t s)
{
    set_tile_order(o, a, BLOCK * SORT_ITEMS);
    if (a.shift >= 32)
        hipLaunchKernelGGL((onesweep_kernel<u64, BLOCK, SORT_ITEMS, SRC, 1, VALS>), dim3(a.tiles), dim3(BLOCK), 0, s, a);
    else
        hipLaunchKernelGGL((onesweep_kernel<u64, BLOCK, SORT_ITEMS, SRC, 0, VALS>), dim3(a.tiles), dim3(BLOCK), 0, s, a);
}

template <int SRC, bool VALS = true>
void launch_onesweep(const csa_handle* h, OnesweepArgs& a, hipStream_t s)
{
    if (wide_workgroups(a))
        launch_onesweep_shape<SRC, SORT_WIDE_BLOCK, VALS>(tile_order_of(h), a, s);
    else
        launch_onesweep_shape<SRC, SORT_BLOCK, VALS>(tile_order_of(h), a, s);
}

// a.bits > RADIX_BITS: wide workgroups only (the look-back words are sized for RADIX_BINS a tile of half the size)
// EXT: wide workgroups
template <int SRC, bool EXT = false>
void launch_onesweep32(const csa_handle* hh, OnesweepArgs& a, hipStream_t s)
{
    const TileOrder h = tile_order_of(hh);
    if (a.bits > RADIX_BITS) {
        set_tile_order(h, a, SORT_WIDE_BLOCK * SORT32_ITEMS);
        hipLaunchKernelGGL((onesweep_kernel<u32, SORT_WIDE_BLOCK, SORT32_ITEMS, SRC, 0, true, RADIX_BITS + 1, EXT>), dim3(a.tiles), dim3(SORT_WIDE_BLOCK), 0, s, a);
    } else if (EXT) {
        set_tile_order(h, a, SORT_WIDE_BLOCK * SORT32_ITEMS);
        hipLaunchKernelGGL((onesweep_kernel<u32, SORT_WIDE_BLOCK, SORT32_ITEMS, SRC, 0, true, RADIX_BITS, EXT>), dim3(a.tiles), dim3(SORT_WIDE_BLOCK), 0, s, a);
    } else if (wide_workgroups(a)) {
        set_tile_order(h, a, SORT_WIDE_BLOCK * SORT32_ITEMS);
        hipLaunchKernelGGL((onesweep_kernel<u32, SORT_WIDE_BLOCK, SORT32_ITEMS, SRC, 0>), dim3(a.tiles), dim3(SORT_WIDE_BLOCK), 0, s, a);
    } else {
        set_tile_order(h, a, SORT_BLOCK * SORT32_ITEMS);
        hipLaunchKernelGGL((onesweep_kernel<u32, SORT_BLOCK, SORT32_ITEMS, SRC, 0>), dim3(a.tiles), dim3(SORT_BLOCK), 0, s, a);
    }
}

// One radix pass over n pairs, between two events where the caller asked for its time.
template <typename LaunchPass>
int launch_pass(Launch& L, u32 n, LaunchPass launch)
{
    csa_handle* h = L.h;
    const bool timed = (L.flags & CSA_FLAG_KERNEL_TIMING) && L.events_used + 2 <= (int)h->events.size();
    if (timed)
        HIP_TRY(hipEventRecord(h->events[L.events_used], L.stream));
    launch();
    if (timed) {
        HIP_TRY(hipEventRecord(h->events[L.events_used + 1], L.stream));
        L.timed.push_back({L.events_used, (u64)n});
        L.events_used += 2;
    }
    return CSA_OK;
}

// Sorts n pairs by the digits of `plan`. The first pass that runs takes its input as `src` says
// (pairs kin/vin, or keys built on the way in); passes alternate between the (kin, vin) and (kout, vout) sets, the
// very first one writing to (kout, vout). *result_in_out = 1 if the sorted pairs ended in (kout, vout).
// Passes whose digit is the same for every pair are skipped (they would be the identity).
// src = SRC_RANKS: pair i is ((rank_src[i], rank_src[i + hop]), i), i < n, built by the first pass that runs; the two
// ranks are combined as rank_pair_key says for `radix`.
// src = SRC_PACKED, SRC_TEXT: the first pass cuts its keys from the code stream, or builds them from the text, that `source`
// describes; the caller has filled ghist already.
struct TextSource {
    const u16* text;   // SRC_TEXT ...
    bool byte_wide;    // ... whose symbols may differ in one of their bytes only
    const u32* stream; // SRC_PACKED
    u64 words;
    u32 sym_bits, key_bits;
    bool scanned; // digit_base is filled as well
};

int radix_sort(Launch& L, int src, u32 text_n, u32 tail, u64* kin, u32* vin, u64* kout,
               u32* vout, u32 n, const PassPlan& plan, int* result_in_out, int* passes_run, const u32* rank_src = nullptr,
               u32 hop = 0, u32 radix = 0, const TextSource* source = nullptr)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    *result_in_out = 0;
    *passes_run = 0;
    if (n == 0)
        return CSA_OK;
    if (src == SRC_PACKED || src == SRC_TEXT) {
        if (!source)
            return fail(CSA_ERR_INTERNAL, "radix_sort: keys of the text come with their source");
    } else {
        HIP_TRY(hipMemsetAsync(h->ghist, 0, MAX_PASSES * RADIX_BINS * sizeof(u32), s));
        HistArgs ha;
        ha.keys = kin;
        ha.n = n;
        ha.plan = plan;
        ha.ghist = h->ghist;
        if (src == SRC_RANKS) {
            ha.rank = rank_src;
            ha.hop = hop;
            ha.radix = radix;
        }
        // the two halves of a (rank[i], rank[i + hop]) key are the same array, one shifted by hop: when the plan takes
        // the same digits from both halves, one histogram of rank[] and one of its first hop entries give them all
        const int half = plan.num_passes / 2;
        bool mirrored = src == SRC_RANKS && radix == 0 && plan.num_passes == 2 * half && half >= 1 && half <= RANK_HIST_PASSES;
        for (int p = 0; mirrored && p < half; ++p)
            mirrored = plan.shift[p] + plan.bits[p] <= 32 && plan.shift[half + p] == 32 + plan.shift[p] && plan.bits[half + p] == plan.bits[p];
        if (mirrored) {
            RankHistArgs ra;
            ra.rank = rank_src;
            ra.num_passes = half;
            for (int p = 0; p < half; ++p) {
                ra.shift[p] = plan.shift[p];
                ra.bits[p] = plan.bits[p];
            }
            const u32 cut = hop < n ? hop : n;
            ra.begin = 0;
            ra.end = n;
            ra.out = h->ghist + half * RADIX_BINS;
            hipLaunchKernelGGL(rank_hist_kernel, dim3(hist_blocks(256 * 16, n)), dim3(256), 0, s, ra);
            if (cut > 0) {
                ra.end = cut;
                ra.out = h->ghist;
                hipLaunchKernelGGL(rank_hist_kernel, dim3(hist_blocks(256 * 16, cut)), dim3(256), 0, s, ra);
            }
            hipLaunchKernelGGL(rank_hist_combine_kernel, dim3(1), dim3(256), 0, s, h->ghist, half, cut);
        } else {
            hipLaunchKernelGGL(radix_hist_kernel, dim3(hist_blocks(256 * 16, n)), dim3(256), 0, s, ha);
        }
    }
    if (!source || !source->scanned)
        hipLaunchKernelGGL(radix_scan_hist_kernel<RADIX_BINS>, dim3(1), dim3(RADIX_BINS), 0, s, h->ghist, h->digit_base, plan.num_passes);
    HIP_TRY(hipGetLastError());
    // (the digits of K-gram keys are the two bytes of a symbol, four times: where both take several values no pass is skipped)
    const bool all_run = src == SRC_TEXT && !source->byte_wide;
    u32* h_hist = h->h_pinned + PINNED_HIST;
    if (!all_run) {
        const int rc = move_table(h_hist, h->ghist, plan.num_passes * RADIX_BINS * sizeof(u32), s);
        if (rc)
            return rc;
        HIP_TRY(hipStreamSynchronize(s));
    }
    bool run[MAX_PASSES];
    int n_run = 0;
    for (int p = 0; p < plan.num_passes; ++p) {
        bool trivial = false;
        for (int d = 0; d < RADIX_BINS && !all_run; ++d)
            if (h_hist[p * RADIX_BINS + d] == n)
                trivial = true;
        run[p] = !trivial;
        n_run += run[p] ? 1 : 0;
    }
    if (n_run == 0 && src != SRC_PAIRS && plan.num_passes > 0) { // the pairs must still be materialised once
        run[plan.num_passes - 1] = true;
        n_run = 1;
    }
    bool first = true;
    int where = 0; // 0: current data in (kin, vin) (or the text); 1: in (kout, vout)
    for (int p = 0; p < plan.num_passes; ++p) {
        if (!run[p])
            continue;
        OnesweepArgs a;
        a.keys_in = where == 0 ? kin : kout;
        a.vals_in = where == 0 ? vin : vout;
        a.keys_out = where == 0 ? kout : kin;
        a.vals_out = where == 0 ? vout : vin;
        a.n = n;
        a.text_n = text_n;
        a.tail = tail;
        a.shift = plan.shift[p];
        a.bits = plan.bits[p];
        a.digit_base = h->digit_base + p * RADIX_BINS;
        a.lookback = h->lookback;
        a.lookback_groups = h->lookback + h->lookback_tile_words;
        a.epoch = next_epoch(h);
        a.err = h->counts + 2;
        a.rank = rank_src;
        a.hop = hop;
        a.radix = radix;
        if (source) {
            a.text = source->text;
            a.stream = source->stream;
            a.stream_words = source->words;
            a.sym_bits = source->sym_bits;
            a.key_bits = source->key_bits;
        }
        int rc = next_ticket(L, &a.ticket);
        if (rc)
            return rc;
        const int use_src = first ? src : SRC_PAIRS;
        rc = launch_pass(L, n, [&] {
            if (use_src == SRC_PAIRS)
                launch_onesweep<SRC_PAIRS>(h, a, s);
            else if (use_src == SRC_RANKS)
                launch_onesweep<SRC_RANKS>(h, a, s);
            else if (use_src == SRC_TEXT)
                launch_onesweep<SRC_TEXT>(h, a, s);
            else
                launch_onesweep<SRC_PACKED>(h, a, s);
        });
        if (rc)
            return rc;
        first = false;
        where ^= 1;
        (*passes_run)++;
    }
    HIP_TRY(hipGetLastError());
    *result_in_out = where;
    return CSA_OK;
}

PassPlan make_plan(int begin_bit, int end_bit)
{
    PassPlan p;
    p.num_passes = 0;
    // digits of up to 8 bits that never straddle bit 32 (a pass reads its digit from one half of the key)
    int s = begin_bit;
    while (s < end_bit && p.num_passes < MAX_PASSES) {
        int bits = end_bit - s < RADIX_BITS ? end_bit - s : RADIX_BITS;
        if (s < 32 && s + bits > 32)
            bits = 32 - s;
        p.shift[p.num_passes] = s;
        p.bits[p.num_passes] = bits;
        p.num_passes++;
        s += bits;
    }
    return p;
}

int ensure_events(csa_handle* h, bool kernel_timing)
{
    if (!h->ev_gen_ready) {
        for (auto& e : h->ev_gen)
            HIP_TRY(hipEventCreate(&e));
        h->ev_gen_ready = true;
    }
    if (kernel_timing && h->events.empty()) {
        h->events.resize(EVENT_POOL);
        for (auto& e : h->events)
            HIP_TRY(hipEventCreate(&e));
    }
    return CSA_OK;
}

// counts: [2] device error flag, [3] verifier flag, [4] members of large groups. Waits for the stream. `beside`: what else the host
// wants to see by then.
int read_counts(Launch& L, u32* big, TableGroup beside = {})
{
    csa_handle* h = L.h;
    add_table(beside, h->h_pinned, h->counts, 8 * sizeof(u32));
    const int rc = move_tables(beside, L.stream);
    if (rc)
        return rc;
    HIP_TRY(hipStreamSynchronize(L.stream));
    if (h->h_pinned[2]) {
        static const char* const what[] = {"", "a look-back wait ran into its spin limit",
                                           "an active suffix lies outside its group's range (small-group sort)",
                                           "a large-group member was sent outside the active list (place)",
                                           "a rank or suffix index out of range in the sorted active list (rerank)",
                                           "a large group appeared in a list whose groups were all small",
                                           "the join table of a partition step has more members than slots"};
        const u32 code = h->h_pinned[2];
        return fail(CSA_ERR_INTERNAL, "device invariant %u failed: %s", code, code < 7 ? what[code] : "unknown");
    }
    if (big)
        *big = h->h_pinned[4];
    return CSA_OK;
}


struct DeferBuffers {
    u64* recs[2]; // generation 0: [n] (position << 32 | rank) records in sorted-list order, and their ping-pong partner
    u32* vals;    // later generations: [m] new ranks in sorted-list order
    u32* t1_pos;  // ping
    u32* t1_val;
    u32* t2_pos;  // pong
    u32* t2_val;
};

// After a rerank launched with rank_recs = buf.recs[0]: rank[x] = r for each of the n records (x << 32) | r.
// The positions x are a permutation of the text positions [0, n) (the sorted suffixes of generation 0), which makes
// the digit counts of the passes a closed form. The records are sorted on the position bits above the window size
// (windows of at most 1 << 14 positions, 1 << 15 for the largest partitions), then placed window by window.
int deferred_rank_update(Launch& L, const DeferBuffers& buf, u32 n)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    const int nb = bit_length(n - 1); // <= 31
    int top = nb - PLACE_WINDOW_LOG2; // position bits to sort on
    if (top < 0)
        top = 0;
    if (top > 16)
        top = 16;
    const int window_log2 = nb - top;
    int n_pass = 0, xshift[2] = {0, 0}, xbits[2] = {0, 0};
    if (top > 8) {
        xshift[0] = window_log2;
        xbits[0] = top - 8;
        xshift[1] = window_log2 + top - 8;
        xbits[1] = 8;
        n_pass = 2;
    } else if (top > 0) {
        xshift[0] = window_log2;
        xbits[0] = top;
        n_pass = 1;
    }
    const u64* in_recs = buf.recs[0];
    if (n_pass > 0) {
        u32* h_hist = h->h_pinned + PINNED_HIST;
        for (int p = 0; p < n_pass; ++p) {
            // positions x in [0, n) whose digit (x >> shift) & mask equals d: whole periods plus a clamped remainder
            const u64 unit = 1ull << xshift[p], period = unit << xbits[p];
            const u64 whole = (u64)n / period, rest = (u64)n % period;
            for (u32 d = 0; d < (u32)RADIX_BINS; ++d) {
                u64 c = 0;
                if (d < (1u << xbits[p])) {
                    c = whole * unit;
                    if (rest > d * unit)
                        c += rest - d * unit < unit ? rest - d * unit : unit;
                }
                h_hist[p * RADIX_BINS + d] = (u32)c;
            }
        }
        HIP_TRY(hipMemcpyAsync(h->ghist, h_hist, n_pass * RADIX_BINS * sizeof(u32), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(radix_scan_hist_kernel<RADIX_BINS>, dim3(1), dim3(RADIX_BINS), 0, s, h->ghist, h->digit_base, n_pass);
        for (int p = 0; p < n_pass; ++p) {
            OnesweepArgs a;
            a.keys_in = in_recs;
            a.vals_in = nullptr; // the records travel alone
            a.keys_out = buf.recs[(p + 1) & 1];
            a.vals_out = nullptr;
            a.n = n;
            a.text_n = n;
            a.tail = 0;
            a.shift = 32 + xshift[p]; // the position is the high half of a record
            a.bits = xbits[p];
            a.digit_base = h->digit_base + p * RADIX_BINS;
            a.lookback = h->lookback;
            a.lookback_groups = h->lookback + h->lookback_tile_words;
            a.epoch = next_epoch(h);
            a.err = h->counts + 2;
                int rc = next_ticket(L, &a.ticket);
            if (rc)
                return rc;
            launch_onesweep<SRC_PAIRS, false>(h, a, s);
            in_recs = buf.recs[(p + 1) & 1];
        }
    }
    const u32 windows = (u32)((((u64)n - 1) >> window_log2) + 1);
    if (window_log2 <= 14)
        hipLaunchKernelGGL((place_ranks_kernel<14>), dim3(windows), dim3(1024), 0, s, in_recs, n, window_log2, h->rank);
    else
        hipLaunchKernelGGL((place_ranks_kernel<15>), dim3(windows), dim3(1024), 0, s, in_recs, n, window_log2, h->rank);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

// Bucketed rank update of a later generation: rank[pos[c]] = vals[c] wherever vals[c] != NO_RANK, c < m.
// A list of an eighth of the partition or more goes through two radix passes on the position bits above a window that fits LDS; the windows are
// read, brought up to date and written back whole. A shorter one goes through one pass and a plain scatter that stays inside one
// window of 1 << WINDOW_LOG2 ranks at a time. Per pair the scatter costs 19 ps, the second pass and the placing 8, and reading and writing
// every rank of the partition 1.8 (10^8 bytes of text, two such updates of 88.2 and 24.0 M pairs: device time of the sort 15.45 ms with
// the scatter, 14.82 with the windows, three processes of each in turn within 0.03).
int windowed_rank_update(Launch& L, const u32* pos, const DeferBuffers& buf, u32 m, u32 n)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    const int nb = bit_length(n - 1);
    const bool whole = m >= n / 8;
    int shift[2] = {0, 0}, bits[2] = {0, 0}, passes = 0, window_log2 = 0;
    if (whole) {
        int top = nb - PLACE_WINDOW_LOG2;
        top = top < 0 ? 0 : top > 16 ? 16 : top;
        window_log2 = nb - top;
        if (top > 8) {
            shift[passes] = window_log2;
            bits[passes++] = top - 8;
        }
        if (top > 0) {
            shift[passes] = top > 8 ? nb - 8 : window_log2;
            bits[passes++] = top > 8 ? 8 : top;
        }
    } else {
        const int top = nb - WINDOW_LOG2 < 8 ? nb - WINDOW_LOG2 : 8;
        if (top > 0) {
            shift[0] = nb - top;
            bits[passes++] = top;
        }
    }
    const u32* in_pos = pos;
    const u32* in_val = buf.vals;
    if (passes > 0) {
        int rc = move_table(h->ghist, nullptr, passes * RADIX_BINS * sizeof(u32), s);
        if (rc)
            return rc;
        for (int p = 0; p < passes; ++p)
            hipLaunchKernelGGL(position_hist_kernel, dim3(hist_blocks(256 * 16, m)), dim3(256), 0, s, pos, m, shift[p], bits[p],
                               h->ghist + p * RADIX_BINS);
        hipLaunchKernelGGL(radix_scan_hist_kernel<RADIX_BINS>, dim3(1), dim3(RADIX_BINS), 0, s, h->ghist, h->digit_base, passes);
        u32* const out_pos[2] = {buf.t1_pos, buf.t2_pos};
        u32* const out_val[2] = {buf.t1_val, buf.t2_val};
        for (int p = 0; p < passes; ++p) {
            OnesweepArgs a;
            a.keys_in = in_pos;
            a.vals_in = in_val;
            a.keys_out = out_pos[p];
            a.vals_out = out_val[p];
            a.n = m;
            a.text_n = n;
            a.tail = 0;
            a.shift = shift[p];
            a.bits = bits[p];
            a.digit_base = h->digit_base + p * RADIX_BINS;
            a.lookback = h->lookback;
            a.lookback_groups = h->lookback + h->lookback_tile_words;
            a.epoch = next_epoch(h);
            a.err = h->counts + 2;
            rc = next_ticket(L, &a.ticket);
            if (rc)
                return rc;
            launch_onesweep32<SRC_PAIRS>(h, a, s);
            in_pos = out_pos[p];
            in_val = out_val[p];
        }
    }
    if (whole) {
        const u32 windows = (u32)((((u64)n - 1) >> window_log2) + 1);
        u32* const starts = h->tile_tables; // (free between the applying kernel and the next generation's counts; 16 bytes for 1024 suffixes)
        hipLaunchKernelGGL(window_starts_kernel, dim3((u32)(((u64)m + 255) / 256)), dim3(256), 0, s, in_pos, m, window_log2, windows, starts);
        if (window_log2 <= 14)
            hipLaunchKernelGGL((place_window_kernel<14>), dim3(windows), dim3(1024), 0, s, in_pos, in_val, (const u32*)starts, n, window_log2,
                               h->rank, h->counts + 2);
        else
            hipLaunchKernelGGL((place_window_kernel<15>), dim3(windows), dim3(1024), 0, s, in_pos, in_val, (const u32*)starts, n, window_log2,
                               h->rank, h->counts + 2);
    } else {
        hipLaunchKernelGGL(scatter_ranks_kernel, dim3((u32)(((u64)m + 1023) / 1024)), dim3(256), 0, s, in_pos, in_val, m, n, h->rank,
                           h->counts + 2);
    }
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

// How far apart in rank[] two writes in a row may lie to count as one (count_ranks_kernel). Half a text of one period, ms per sort
// written in place and bucketed: 2^27 symbols, period 8 68 and 76, 10 67 and 81, 15 73 and 84; 2^29 symbols, period 7 280 and 303, 8 311
// and 310, 12 370 and 340, 15 420 and 358; 2^28 symbols, period 8 153 and 151, 12 175 and 170, 15 190 and 177. Past 2^27
// symbols rank[] is larger than the last-level cache, and a line leaves it before the next residue of the period comes by.
#ifndef CSA_FAR_REACH_MAX
#define CSA_FAR_REACH_MAX (1u << 27)
#endif
u32 run_reach(u32 n) { return n <= CSA_FAR_REACH_MAX ? 15u : 8u; }

// The smallest tile of the kernels that share the rank step's tables: the tables are sized for it.
constexpr int smaller(int a, int b) { return a < b ? a : b; }
constexpr int TABLE_TILE = smaller(smaller(RANK_TILE, SMALL_TILE), smaller(COLLECT_TILE, STEP_TILE));

// Sizes of the rank step's tables for a list of m suffixes cut into tiles of TILE elements.
struct RankTables {
    u32 tiles, slab, slabs;
    u32 *tile_agg, *tile_prefix, *tile_splits, *slab_total;
};

template <int TILE>
RankTables rank_tables(csa_handle* h, u32 m)
{
    static_assert(TILE >= TABLE_TILE, "the tables hold fewer tiles than this list has");
    RankTables r;
    r.tiles = (u32)(((u64)m + TILE - 1) / TILE);
    r.slab = (r.tiles + RERANK_SLABS - 1) / RERANK_SLABS;
    r.slabs = (r.tiles + r.slab - 1) / r.slab;
    r.tile_agg = h->tile_tables;
    r.tile_prefix = h->tile_tables + (u64)h->rank_tiles_cap * 4;
    r.tile_splits = h->tile_tables + (u64)h->rank_tiles_cap * 8;
    r.slab_total = h->tile_tables + (u64)h->rank_tiles_cap * 9;
    return r;
}

// Scans the per-tile counts, reads the totals back (the one host round trip of the step: the next list's size
// decides the launches that follow) and chooses how the ranks are written: 0 scattered by the applying kernel,
// 1 two-pass bucketed (generation 0 of large partitions), 2 one-pass bucketed (most of a later list changed).
int rank_totals(Launch& L, const RankTables& r, bool gen0, u32 m, u32 n, bool expect_no_big, u32* survivors, u32* groups,
                int* rank_update, TableGroup beside = {})
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    hipLaunchKernelGGL(rerank_scan_kernel, dim3(r.slabs), dim3(1024), 0, s, r.tile_agg, r.tile_prefix, r.tiles, r.slab,
                       r.slab_total, r.tile_splits);
    HIP_TRY(hipGetLastError());
    u32* h_slabs = h->h_pinned + PINNED_HIST;
    add_table(beside, h_slabs, r.slab_total, r.slabs * 5 * sizeof(u32));
    u32 big_seen = 0;
    int rc = read_counts(L, &big_seen, beside);
    if (rc)
        return rc;
    if (expect_no_big && big_seen != 0) // groups only split; a large group after an all-small generation is a corrupt list
        return fail(CSA_ERR_INTERNAL, "%u members of large groups appeared after a generation without any", big_seen);
    u64 surv = 0, heads = 0, changed = 0;
    for (u32 sl = 0; sl < r.slabs; ++sl) {
        surv += h_slabs[sl * 5 + 2];
        heads += h_slabs[sl * 5 + 3];
        changed += h_slabs[sl * 5 + 4];
    }
    *survivors = (u32)surv;
    *groups = (u32)heads;
    // Generation 0 ranks every suffix of the partition: on large partitions the n scattered writes go through the
    // two-pass bucketed update. Later generations write only the ranks that changed; when those are many and the
    // partition is larger than one window, they go through the one-pass bucketed update.
    const bool defer0 = gen0 && m >= h->defer_min;
    const bool windowed = !gen0 && bit_length(n - 1) > WINDOW_LOG2 && changed >= h->window_min_changed && changed >= m / 2;
    *rank_update = defer0 ? 1 : windowed ? 2 : 0;
    return CSA_OK;
}

// A dense generation: most of the partition is still active and its groups are long (a small alphabet, a periodic
// text), so nearly every member would go through the radix sort anyway; the whole partition is then sorted again by
// keys read in text order. Decided from the size of the active list and the number of its groups alone, so that the
// generation before already knows it (and leaves ordinals in rank[], which such a generation sorts in fewer passes).
bool dense_generation(u32 m, u32 groups, u32 n)
{
    return (u64)m * 5 >= (u64)n * 3 && (u64)m > (u64)groups * SMALL_MAXG_HI && (u64)m >= DENSE_MIN;
}

// Whether, and how, the first sort of a partition takes keys of many packed symbols (packed_text.hpp). From the byte
// histograms of the text: a symbol's code is made of the ranks of its two bytes among the byte values that occur, zero
// (the padding) included; with nhi * nlo <= 256 codes the text qualifies. The key takes the largest context the doubling
// of the caller's key width reaches inside 64 bits: S = 4 W 2^j symbols, which covers j generations after the first.
struct PackedPlan {
    bool enabled;
    bool byte_wide; // the symbols differ in one of their bytes only: half the passes over K-gram keys have nothing to do
    bool few;       // few_symbols
    SymbolCodes codes;
    u32 skipped; // j
    u32 values;  // codes, 256 at most; 0: too many
};

PackedPlan plan_packed_text(const u32* bytehist, u32 n, int key_words, u64 room_bytes)
{
    PackedPlan pp;
    memset(&pp, 0, sizeof(pp));
    u32 nlo = 0, nhi = 0;
    for (u32 d = 0; d < 256; ++d) {
        if (d == 0 || bytehist[d] != 0)
            pp.codes.lo[d] = (u8)nlo++;
        if (d == 0 || bytehist[256 + d] != 0)
            pp.codes.hi[d] = (u8)nhi++;
    }
    const u32 codes = nlo * nhi;
    pp.byte_wide = nlo == 1 || nhi == 1;
    pp.few = few_symbols(nlo, nhi);
    if (codes > 256)
        return pp;
    pp.values = codes;
    pp.codes.nlo = nlo;
    const u32 b = codes <= 2 ? 1u : codes <= 4 ? 2u : codes <= 16 ? 4u : 8u;
    u32 S = 4u * (u32)key_words;
    if (S * b > 64)
        return pp;
    u32 j = 0;
    while (2 * S * b <= 64) {
        S *= 2;
        ++j;
    }
    const u64 words = ((u64)n * b + 31) / 32 + 4;
    if (words * 4 > room_bytes)
        return pp;
    pp.codes.bits = b;
    pp.codes.key_syms = S;
    pp.skipped = j;
    pp.enabled = true;
    return pp;
}

// Suffixes that the probe looks at: one in 16 while they are few, then one in 512, at most 2^PROBE_MOST_LOG2.
u32 probed_suffixes(u32 n)
{
    const u32 few = n / 16 < PROBE_FEW ? n / 16 : PROBE_FEW, many = n / 512 > few ? n / 512 : few;
    return many < 1u << PROBE_MOST_LOG2 ? many : 1u << PROBE_MOST_LOG2;
}

struct CodeTables {
    u32 *counts, *marks; // zeroed together, with the counters of the probe and its table of up to PROBE_FEW suffixes
    ProbeCounts* probe;
    unsigned long long* table;
    u32* cum;
};

CodeTables code_tables(const csa_handle* h)
{
    CodeTables c;
    c.counts = h->code_tables;
    c.marks = c.counts + SYMBOLS;
    c.probe = reinterpret_cast<ProbeCounts*>(c.marks + RESOLVE_MARK_WORDS);
    c.table = reinterpret_cast<unsigned long long*>(c.probe + 1);
    c.cum = reinterpret_cast<u32*>(c.table + PROBE_TABLE);
    return c;
}

// Digits of a sort by codes whose lower bits are sorted in buckets (bucket_sort.hpp): as many upper bits as leave BUCKET_AVERAGE suffixes a bucket or
// fewer, by two passes of eight bits or two of nine. Longer texts take all digits.
#ifndef CSA_BUCKETS_MIN
#define CSA_BUCKETS_MIN ((1u << 24) + 1)
#endif
#ifndef CSA_TWO_PASS_LOG2
#define CSA_TWO_PASS_LOG2 16
#endif
#ifndef CSA_BUCKET_AVERAGE
#define CSA_BUCKET_AVERAGE 5000
#endif
constexpr u32 BUCKET_AVERAGE = CSA_BUCKET_AVERAGE;
constexpr CodeDigits ALL_DIGITS = {CODE_PASSES, RADIX_BITS, {0, 8, 16, 24}, 0};

CodeDigits bucket_digits(u32 n, bool packed)
{
    u32 log2 = 1;
    while ((n >> log2) > BUCKET_AVERAGE)
        ++log2;
    // The digits of packed keys are counted by eight bits, so there are no more buckets: as long as the average one is 2.5 standard deviations of its size below
    // BUCKET_MAX (4.5 * 10^8 symbols). (Four letters, with copies / independent, ms with all passes and with buckets: 3.4 * 10^8 symbols 16.6, 14.9 / 10.4, 8.7; 4.4 * 10^8 21.2,
    // 19.4 / 13.3, 11.2; 4.55 * 10^8 22.4, 20.5 / 14.0, 11.8; 4.62 * 10^8, where a tenth of the buckets does not fit, 22.7, 22.3 / 14.1, 13.1; 4.66 * 10^8 22.8, 28.5 / 14.3, 15.8.)
    if (packed && log2 == CSA_TWO_PASS_LOG2 + 1 && (n >> CSA_TWO_PASS_LOG2) <= BUCKET_MAX / 100 * 97)
        log2 = CSA_TWO_PASS_LOG2;
    if (log2 <= CSA_TWO_PASS_LOG2)
        return CodeDigits{2, RADIX_BITS, {16, 24}, log2};
    if (log2 <= 18 && !packed && n <= RUN_PLACE)
        return CodeDigits{2, RADIX_BITS + 1, {14, 23}, log2};
    return ALL_DIGITS;
}

// Of the suffixes that are probed, one in so many (and one less here) is counted by its bucket: 16 to 31 a bucket on average where there are more (all of
// 62500 on 256 counters: 30 us instead of 14).
u32 bucket_skip(u32 n, const CodeDigits& digits)
{
    u32 skip = 1;
    while ((probed_suffixes(n) >> digits.buckets_log2) / skip >= 32)
        skip *= 2;
    return skip - 1u;
}

// The buckets of a sample of the suffixes are counted too where the lower digits may be sorted in them, in `room` (zeroed by the caller).
void probe_buckets(ProbeArgs& a, const CodeDigits& digits, u32* room)
{
    if (digits.buckets_log2 == 0)
        return;
    a.buckets = room;
    a.bucket_shift = 32u - digits.buckets_log2;
    a.bucket_skip = bucket_skip(a.n, digits);
    const u32 full = BUCKET_MAX / 16 * 18 / (a.n / a.taken * (a.bucket_skip + 1u)); // (the average bucket shows half of that)
    a.full_from = full > 2 ? full : 2;
}

// Buckets that do not fit are sorted by radix passes after all: from a tenth of the suffixes on all passes are made at once, and from a fiftieth on in four-letter texts of
// fewer than 2^25 symbols, which save the least. (Time with all passes / with buckets, by the share that the sample shows. Tokens, strings that come often: 10^8 symbols 0.06 4417 / 3575 us,
// 0.12 5007 / 3667, 0.18 5665 / 4136; past a quarter all that do not fit are given up, 3 * 10^7 0.30 1738 / 2393. Tokens, a run and a period: 1.7 * 10^7 0.08 1908 / 1880, 0.12 1932 / 1952; 10^8 0.11
// 7983 / 7280; 4 * 10^8 0.12 31.0 / 26.9 ms, 0.19 35.2 / 38.4. Letters, two runs: 1.7 * 10^7 0.04 2253 / 2289 us, 0.08 2344 / 2425; 3 * 10^7 0.04 3395 / 3397, 0.08 3580 / 3607, 0.12 3741 / 3789; 10^8 0.08
// 9402 / 9204, 0.16 10989 / 11017; 4 * 10^8 0.10 35.6 / 34.5 ms. Texts all of whose buckets fit show up to 0.01 below 3.3 * 10^8 symbols, and 0.04 at 4.2 * 10^8.)
#ifndef CSA_MANY_LETTERS
#define CSA_MANY_LETTERS (1u << 25)
#endif
bool buckets_fit(const ProbeCounts& c, u32 n, const CodeDigits& digits, bool packed)
{
    const u32 one_in = packed && n < CSA_MANY_LETTERS ? 50 : 10;
    return (u64)c.packed * one_in * (bucket_skip(n, digits) + 1u) <= probed_suffixes(n);
}

// What a sort by codes starts from: the shares of the symbols, and for texts of PROBE_MIN symbols or more what a sample of the suffixes
// (probed_suffixes) shows about shared codes, on its way to *seen; ev_gen[1] tells that it is there. A large sample's table is
// key[0], which holds nothing yet.
// bytehist: see sample_symbols_kernel. counts[5], zeroed, says that the text was left alone.
int share_symbols(Launch& L, const u16* d_text, u32 n, ProbeCounts* seen, const u32* bytehist)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    const CodeTables c = code_tables(h);
    const u32 chunks = (n + SAMPLE_CHUNK - 1) / SAMPLE_CHUNK;
    u64 zeros = (SYMBOLS + RESOLVE_MARK_WORDS) * sizeof(u32);
    ProbeArgs a;
    memset(&a, 0, sizeof(a));
    if (n >= PROBE_MIN) {
        a.text = d_text;
        a.n = n;
        a.taken = probed_suffixes(n);
        a.cum = c.cum;
        a.table_log2 = (u32)bit_length((u64)a.taken - 1) + 1;
        // (an eighth more than a tile sorts: a run of just that many would be taken for a longer one as often as not)
        const u32 long_run = RESOLVE_MAX * 9 / 8 / (n / a.taken);
        a.long_from = long_run > 2 ? long_run : 2;
        a.counts = c.probe;
        a.skipped = h->counts + 5;
        const bool few = a.taken <= PROBE_FEW;
        a.table = few ? c.table : reinterpret_cast<unsigned long long*>(h->key[0]);
        zeros += sizeof(ProbeCounts);
        u64 large_zeros = 0;
        (few ? zeros : large_zeros) += sizeof(u64) << a.table_log2;
        if (n >= CSA_BUCKETS_MIN) {
            const CodeDigits digits = bucket_digits(n, false);
            probe_buckets(a, digits, reinterpret_cast<u32*>(reinterpret_cast<unsigned char*>(h->key[0]) + large_zeros));
            large_zeros += sizeof(u32) << digits.buckets_log2;
        }
        if (large_zeros)
            HIP_TRY(hipMemsetAsync(h->key[0], 0, large_zeros, s));
    }
    HIP_TRY(hipMemsetAsync(c.counts, 0, zeros, s));
    // one chunk in 16, at least SAMPLE_CHUNKS_MIN of them (or all there are) and at most SAMPLE_CHUNKS_MAX
    u32 taken = chunks / 16 < SAMPLE_CHUNKS_MIN ? SAMPLE_CHUNKS_MIN : chunks / 16;
    taken = taken < SAMPLE_CHUNKS_MAX ? taken : SAMPLE_CHUNKS_MAX;
    taken = taken < chunks ? taken : chunks;
    const u64 sampled = (u64)taken * SAMPLE_CHUNK < n ? (u64)taken * SAMPLE_CHUNK : (u64)n;
    const u32 per_block = sample_chunks_per_block(taken);
    hipLaunchKernelGGL(sample_symbols_kernel, dim3((taken + per_block - 1) / per_block), dim3(SAMPLE_BLOCK), 0, s, d_text, n, chunks, taken,
                       c.counts, bytehist, h->counts + 5);
    const int weight_log2 = SAMPLE_LOG2 - bit_length(sampled - 1);
    hipLaunchKernelGGL(symbol_shares_kernel, dim3(SYMBOLS / SHARES_TILE), dim3(SHARES_TILE), 0, s, (const u32*)c.counts, weight_log2,
                       (u32)((sampled << weight_log2) + SYMBOLS), c.cum, (const u32*)(h->counts + 5));
    if (n >= PROBE_MIN) {
        hipLaunchKernelGGL(probe_codes_kernel, dim3((a.taken + PROBE_BLOCK - 1) / PROBE_BLOCK), dim3(PROBE_BLOCK), 0, s, a);
        const int rc = move_table(seen, a.counts, sizeof(ProbeCounts), s);
        if (rc)
            return rc;
        HIP_TRY(hipEventRecord(h->ev_gen[1], s)); // (recorded again when the generation ends)
    }
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

// Texts of two-bit symbols from this length on may start from narrow keys: 2^25 + 5 independent letters 2.0 -> 1.2 ms, 4 * 10^8, a fifth of
// them copies, 28.4 -> 21.4. The line is not where they begin to pay: they gain at every length measured (ms, wide and narrow: 20000 letters
// with copies 0.27, 0.26; 2^17 0.29, 0.27; 2^20 0.40, 0.35; 2^22 0.56, 0.48; 2^24 1.50, 1.14), and shorter texts keep wide ones
// because callers have been told of eight passes for them. Texts of symbols of one or four bits, and keys of 48, have not been tried.
#ifndef CSA_NARROW_MIN
#define CSA_NARROW_MIN ((1u << 24) + 1)
#endif

// Whether the first sort of a packed text takes narrow keys, 32 bits of the code stream, and reads the next 32 for the suffixes that tie
// on them (sort_by_codes): four passes over 8-byte pairs instead of eight over 12-byte ones save 27 ps a suffix, less 8 for the second half; a member of a
// run that is too long for a tile costs 100 (it is collected and sorted again), and a sample of the suffixes shows how many there are.
// *digits: the radix passes that they take.
int narrow_keys_pay(Launch& L, const TextSource& ps, u32 n, bool* pay, CodeDigits* digits)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    const CodeTables c = code_tables(h);
    ProbeCounts* const seen = reinterpret_cast<ProbeCounts*>(h->h_pinned + PINNED_HIST);
    ProbeArgs a;
    memset(&a, 0, sizeof(a));
    a.n = n;
    a.taken = probed_suffixes(n);
    a.table = reinterpret_cast<unsigned long long*>(h->key[0]); // (nothing there yet)
    a.table_log2 = (u32)bit_length((u64)a.taken - 1) + 1;
    const u32 long_run = RESOLVE_MAX / (n / a.taken);
    a.long_from = long_run > 2 ? long_run : 2;
    a.counts = c.probe;
    a.stream = ps.stream;
    a.sym_bits = ps.sym_bits;
    const CodeDigits in_buckets = bucket_digits(n, true);
    probe_buckets(a, in_buckets, reinterpret_cast<u32*>(a.table + (1ull << a.table_log2)));
    HIP_TRY(hipMemsetAsync(a.table, 0, (sizeof(u64) << a.table_log2) + (sizeof(u32) << in_buckets.buckets_log2), s));
    int rc = move_table(c.probe, nullptr, sizeof(ProbeCounts), s);
    if (rc)
        return rc;
    hipLaunchKernelGGL(probe_codes_kernel, dim3((a.taken + PROBE_BLOCK - 1) / PROBE_BLOCK), dim3(PROBE_BLOCK), 0, s, a);
    if ((rc = move_table(seen, c.probe, sizeof(ProbeCounts), s)) != CSA_OK)
        return rc;
    HIP_TRY(hipStreamSynchronize(s));
    *pay = (u64)seen->crowded * 6 <= a.taken;
    *digits = buckets_fit(*seen, n, in_buckets, true) ? in_buckets : ALL_DIGITS;
    return CSA_OK;
}

// Whether a text is sorted by codes or by K-gram keys. Codes save passes, and lose time to suffixes that share one with others and
// have to be told apart by the text. Both per suffix in picoseconds, from generation 0 of texts of 2^19 to 2^28 symbols on either kind of key:
// independent symbols are 15 to 23 faster on codes, short texts by 25 us for the launches and a round trip alone; a line of the
// text for every suffix costs about 20; a suffix is compared with the others of its run, at 0.2 to 0.5 each; collecting and
// sorting the members of long runs that are out of order costs 60 each and 200 us in all.
// Measured (ms; K-grams, codes, chosen, with the probe): 2^28 Zipf tokens 16.0, 11.0, 11.0; 2^28 symbols of a chain in which a symbol
// has 3 successors 15.7, 38.8, 15.8; 20 successors 16.3, 34.4, 16.5; 2^28 symbols of 100000 phrases 16.4, 25.7, 16.5; 2^22 of them
// 0.40, 0.72, 0.45; 2^20 of them 0.23, 0.44, 0.28.
bool codes_pay(const ProbeCounts& c, u32 n)
{
    const double seen = probed_suffixes(n), per_seen = n / seen;
    const double second = 2.0 * (c.second - c.third) / seen, third = 3.0 * (c.third - c.fourth) / seen; // in codes seen twice, thrice
    const double more = ((double)c.again + c.second) / seen - second;                                    // ... thrice and more often
    // The suffixes whose company the sample missed: a code of m suffixes shows x = m / per_seen of them on average, and e^x / x
    // times as many suffixes belong to such codes as belong to codes seen twice; x follows from how many are seen thrice.
    double x = second > 0 ? 2.0 * third / second : 0.0;
    x = x < 1.0 / per_seen ? 1.0 / per_seen : x > 3.0 ? 3.0 : x;
    double company = more + second * std::exp(x) / x;
    company = company < 1.0 ? company : 1.0;
    const double others = company > 0 ? 2.0 * (double)c.pairs / seen * per_seen / company : 0.0; // with the code of one with company
    const double mixed = c.again ? (double)c.other / c.again : 0.0;
    // read from the text, and compared with its run: at most RESOLVE_MAX others
    double cost = company * (20.0 + 0.5 * mixed * (others < RESOLVE_MAX ? others : RESOLVE_MAX));
    // Collected and sorted once more. Where a long run would show two or three suffixes only, short ones do so by chance: then a
    // few of them count only if runs are long on average. (Three of them are a run of RESOLVE_MAX that shows 12 of its members at one in 32,
    // the last three of which differ from the first to arrive or do not: such a text would go one way or the other from call to call.)
    if (c.crowded > (per_seen <= 64 || x * per_seen >= RESOLVE_MAX / 2 ? 3.0 : seen / 1000))
        cost += 60.0 * c.crowded / seen + 2e8 / n;
    return cost < 18.0 + 2.5e7 / n;
}

// key[1] until the list is ranked: the codes by virtual position, which the first pass reads, the flags by text position behind them, and the
// ties of the sorted list behind those. Each starts at a multiple of 16 bytes, for the loads that wide; 5.125 bytes a suffix and 31 are fewer than 8 a
// suffix rounded up to 256.
u32* codes_of(const csa_handle* h) { return reinterpret_cast<u32*>(h->key[1]); }
u8* own_of(const csa_handle* h) { return reinterpret_cast<u8*>(h->key[1]) + (4 * h->cap + 15) / 16 * 16; }
u8* ties_of(const csa_handle* h) { return own_of(h) + ((h->cap + 7) / 8 + 15) / 16 * 16; }

u16* ext_of(const csa_handle* h) { return reinterpret_cast<u16*>(ties_of(h) + (h->cap + 15) / 16 * 16); } // (of texts that are sorted in buckets: 7.125 bytes a suffix)

int code_suffixes(Launch& L, const u16* d_text, u32 n, u32 tail, const CodeDigits& digits)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    const u32* const cum = code_tables(h).cum;
    auto launch = [&](auto kernel, int block) {
        hipLaunchKernelGGL(kernel, dim3(hist_blocks(block * CODE_ITEMS, n)), dim3(block), 0, s, d_text, n, tail, cum, codes_of(h), own_of(h), digits, h->ghist, ext_of(h));
    };
    if (digits.passes == 2)
        launch(code_suffixes_kernel<CODE_WIDE_BLOCK, 2, true>, CODE_WIDE_BLOCK);
    else if (n >= SORT_WIDE_MIN) // 2048 tiles of the wide workgroups: four for each of those a device holds at a time
        launch(code_suffixes_kernel<CODE_WIDE_BLOCK, CODE_PASSES, false>, CODE_WIDE_BLOCK);
    else
        launch(code_suffixes_kernel<CODE_BLOCK, CODE_PASSES, false>, CODE_BLOCK);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

constexpr u32 OPEN_BLOCKS = 2048; // workgroups that resolve open runs: twice as many as a device of 256 compute units holds at a time

// A list sorted by codes on its way to being ranked.
struct CodedList {
    ResolveArgs args;
    u32 words;        // words of four symbols that its order and its ties stand for, at most 2 ...
    bool told;        // ... as the device has decided (many_in_long_runs)
    u64 long_members; // suffixes in runs that were too long for their tile, sorted by their second word in ...
    int long_passes;  // ... so many radix passes
    bool long_left;   // there are runs that are too long for a tile on both words
    bool by_levels;   // the ties are those of sort_by_words: `words` of its levels, and nothing else to be done
};

// The list of open runs: where the passes of a sort by codes in buckets had their pairs, and in an array that is not used before its long runs are.
u32* open_sufs_of(const csa_handle* h) { return reinterpret_cast<u32*>(h->key[0]) + h->cap; }
u32* open_places_of(const csa_handle* h) { return h->idx[2]; }

// The bits of the codes below the passes of `digits`, in place, or with those of ext, if non-null, into idx[1] (bucket_sort.hpp). *finished = false: too many suffixes are in buckets that do
// not fit, and nothing that is used has changed. Works in the group tables, and in key[2], idx[3] and idx[4].
int finish_buckets(Launch& L, const CodeDigits& digits, u32 n, u32 tail, u32* codes, u32* sufs, const u16* ext, const u32* top_base, int* passes,
                   bool* finished)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    BucketArgs a;
    memset(&a, 0, sizeof(a));
    a.codes = codes;
    a.sufs = sufs;
    a.n = n;
    a.low_bits = 32u - digits.buckets_log2;
    a.buckets = 1u << digits.buckets_log2;
    a.starts = h->gprim[0];
    a.top_base = top_base;
    a.top_shift = digits.shift[digits.passes - 1];
    a.over = h->counts + 8;
    a.over_list = h->gprim[1];
    a.tail = tail;
    a.crowded = h->counts + 11;
    a.crowded_list = h->gstart[0]; // (done with before over_before)
    if (ext) {
        a.ext = ext;
        a.ext_bits = digits.buckets_log2 < 16u ? digits.buckets_log2 : 16u;
        a.sufs_out = h->idx[1];
        a.ties = ties_of(h);
        a.open_count = h->counts + 12;
        a.open_sufs = open_sufs_of(h);
        a.open_places = open_places_of(h);
        a.over_open = h->counts + 13;
    }
    a.over_before = h->gstart[0];
    a.over_tiles = h->gstart[1];
    hipLaunchKernelGGL(bucket_starts_kernel, dim3(a.buckets / (STARTS_BLOCK - 1) + 1), dim3(STARTS_BLOCK), 0, s, a);
    int rc = move_table(h->h_pinned + 8, a.over, 3 * sizeof(u32), s);
    if (rc)
        return rc;
    HIP_TRY(hipEventRecord(h->ev_gen[2], s)); // (recorded again when a generation ends)
    const dim3 crowded_grid(a.buckets < CROWDED_BLOCKS ? a.buckets : CROWDED_BLOCKS);
    if (ext) {
        hipLaunchKernelGGL(finish_buckets_kernel<true>, dim3(a.buckets), dim3(BUCKET_BLOCK), 0, s, a);
        hipLaunchKernelGGL(finish_crowded_kernel<true>, crowded_grid, dim3(BUCKET_BLOCK), 0, s, a);
    } else {
        hipLaunchKernelGGL(finish_buckets_kernel<false>, dim3(a.buckets), dim3(BUCKET_BLOCK), 0, s, a);
        hipLaunchKernelGGL(finish_crowded_kernel<false>, crowded_grid, dim3(BUCKET_BLOCK), 0, s, a);
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipEventSynchronize(h->ev_gen[2]));
    const u32 over = h->h_pinned[8], over_buckets = h->h_pinned[9], largest = h->h_pinned[10];
    *finished = over <= n / 4 && over <= h->cap / 2;
    if (over == 0 || !*finished)
        return CSA_OK;
    u64* const K[2] = {h->key[2], h->key[2] + h->cap / 2};
    u32* const V[2] = {h->idx[3], h->idx[4]};
    a.over_keys = K[0];
    a.over_sufs = V[0];
    hipLaunchKernelGGL(over_before_kernel, dim3((a.buckets + OVER_TILE - 1) / OVER_TILE), dim3(OVER_TILE), 0, s, a);
    const u32 wanted = (largest + OVER_SLICE - 1) / OVER_SLICE, most = OVER_BLOCKS / over_buckets;
    a.over_slices = wanted < most ? wanted : most;
    a.over_slices = a.over_slices < 16u ? 16u : a.over_slices;
    const dim3 over_grid(over_buckets * a.over_slices);
    if (ext)
        hipLaunchKernelGGL((over_move_kernel<false, true>), over_grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((over_move_kernel<false, false>), over_grid, dim3(256), 0, s, a);
    int in_out = 0, run = 0;
    rc = radix_sort(L, SRC_PAIRS, 0, 0, K[0], V[0], K[1], V[1], over, make_plan(0, ext ? 48 : 32), &in_out, &run);
    if (rc)
        return rc;
    *passes += run;
    a.over_keys = K[in_out];
    a.over_sufs = V[in_out];
    if (ext)
        hipLaunchKernelGGL((over_move_kernel<true, true>), over_grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((over_move_kernel<true, false>), over_grid, dim3(256), 0, s, a);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

// Generation 0 on codes (coded_keys.hpp): the suffixes of the text in the order of their first `words` words of four symbols (0: two, or one
// if many lie in long runs), with their ties beside them; code_suffixes ran before. Sorts (codes, idx[0]) <-> (codes', idx[1]) and resolves the runs of equal codes into
// idx[1]; the codes live in the halves of key[0]. What long runs leave open is finished by sort_marked_runs and sort_long_runs.
// packed: the codes are narrow keys, cut from its stream, of word_syms symbols (and so are the words).
// digits: the radix passes; `counted` says whose counts ghist holds, theirs or those of all digits.
int sort_by_codes(Launch& L, const u16* d_text, u32 n, u32 tail, u32 words, CodedList& list, const CodeDigits& counted, const CodeDigits& digits,
                  int* passes, const TextSource* packed = nullptr, u32 word_syms = 4)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    if (counted.bits == RADIX_BITS)
        hipLaunchKernelGGL(radix_scan_hist_kernel<RADIX_BINS>, dim3(1), dim3(RADIX_BINS), 0, s, h->ghist, h->digit_base, (int)counted.passes);
    else
        hipLaunchKernelGGL(radix_scan_hist_kernel<2 * RADIX_BINS>, dim3(1), dim3(2 * RADIX_BINS), 0, s, h->ghist, h->digit_base, (int)counted.passes);
    u32* const sorted[2] = {reinterpret_cast<u32*>(h->key[0]), reinterpret_cast<u32*>(h->key[0]) + h->cap};
    u16* const ext[2] = {reinterpret_cast<u16*>(h->gid), reinterpret_cast<u16*>(h->gid) + h->cap}; // (no groups yet)
    const u32* top_base = nullptr;
    for (u32 p = 0; p < digits.passes; ++p) {
        const u32 out = (digits.passes - 1 - p) & 1, in = out ^ 1; // the sorted codes end in the first half of key[0], their suffixes in idx[0]
        OnesweepArgs a;
        a.keys_in = p == 0 ? codes_of(h) : sorted[in];
        a.vals_in = h->idx[in];
        a.keys_out = sorted[out];
        a.vals_out = h->idx[out];
        a.n = n;
        a.text_n = n;
        a.tail = tail;
        a.own = own_of(h);
        if (packed) {
            a.stream = packed->stream;
            a.stream_words = packed->words;
            a.sym_bits = packed->sym_bits;
            a.key_bits = 32;
        }
        a.shift = (int)digits.shift[p];
        a.bits = (int)digits.bits;
        top_base = h->digit_base + ((counted.buckets_log2 ? p : digits.shift[p] / RADIX_BITS) << digits.bits);
        a.digit_base = top_base;
        a.lookback = h->lookback;
        a.lookback_groups = h->lookback + h->lookback_tile_words;
        a.epoch = next_epoch(h);
        a.err = h->counts + 2;
        int rc = next_ticket(L, &a.ticket);
        if (rc)
            return rc;
        rc = launch_pass(L, n, [&] {
            if (digits.buckets_log2 && !packed) {
                a.ext_in = p == 0 ? ext_of(h) : ext[in];
                a.ext_out = ext[out];
                if (p == 0)
                    launch_onesweep32<SRC_CODED, true>(h, a, s);
                else
                    launch_onesweep32<SRC_PAIRS, true>(h, a, s);
            } else if (p == 0 && packed)
                launch_onesweep32<SRC_PACKED>(h, a, s);
            else if (p == 0)
                launch_onesweep32<SRC_CODED>(h, a, s);
            else
                launch_onesweep32<SRC_PAIRS>(h, a, s);
        });
        if (rc)
            return rc;
    }
    *passes = CODE_PASSES; // (the digits that are sorted in buckets among them)
    if (digits.buckets_log2) {
        bool finished = false;
        int rc = finish_buckets(L, digits, n, tail, sorted[0], h->idx[0], packed ? nullptr : ext[0], top_base, passes, &finished);
        if (rc)
            return rc;
        if (!finished) { // (a sample had shown fewer suffixes in buckets that do not fit)
            if (counted.buckets_log2) {
                HIP_TRY(hipMemsetAsync(h->ghist, 0, CODE_BINS * sizeof(u32), s));
                if ((rc = code_suffixes(L, d_text, n, tail, ALL_DIGITS)) != CSA_OK)
                    return rc;
            }
            return sort_by_codes(L, d_text, n, tail, words, list, ALL_DIGITS, ALL_DIGITS, passes, packed, word_syms);
        }
    }
    memset(&list, 0, sizeof(list));
    list.words = words;
    ResolveArgs& r = list.args;
    r.codes = sorted[0];
    r.sufs = h->idx[0];
    r.m = n;
    r.text = d_text;
    r.n = n;
    r.words = words;
    r.word_syms = word_syms;
    if (packed) {
        r.stream = packed->stream;
        r.sym_bits = packed->sym_bits;
    }
    r.sufs_out = h->idx[1];
    r.ties = ties_of(h);
    r.marks = code_tables(h).marks;
    r.unordered = h->counts + 4;
    r.any_long = h->counts + 5;
    r.words_out = h->counts + 6;
    r.text_codes = codes_of(h);
    r.tail = tail;
    const dim3 resolve_grid((u32)(((u64)n + RESOLVE_TILE - 1) / RESOLVE_TILE));
    if (digits.buckets_log2 && !packed) { // the list stands in idx[1] already, but for its open runs
        r.codes = nullptr;
        r.open_count = h->counts + 12;
        r.sufs = open_sufs_of(h);
        r.places = open_places_of(h);
        hipLaunchKernelGGL((resolve_runs_kernel<RESOLVE_MAX, false, false, false, true>), dim3(resolve_grid.x < OPEN_BLOCKS ? resolve_grid.x : OPEN_BLOCKS),
                           dim3(RESOLVE_BLOCK), 0, s, r);
        HIP_TRY(hipGetLastError());
        return CSA_OK;
    }
    if (words == 0 && n >= WORDS_AHEAD)
        hipLaunchKernelGGL(choose_words_kernel, dim3(1), dim3(LONG_LIST_PLACES), 0, s, r.codes, n, r.words_out);
    if (packed)
        hipLaunchKernelGGL((resolve_runs_kernel<RESOLVE_MAX, false, true, false>), resolve_grid, dim3(RESOLVE_BLOCK), 0, s, r);
    else if (n < WORDS_AHEAD)
        hipLaunchKernelGGL((resolve_runs_kernel<RESOLVE_MAX, false, false, true>), resolve_grid, dim3(RESOLVE_BLOCK), 0, s, r);
    else
        hipLaunchKernelGGL((resolve_runs_kernel<RESOLVE_MAX, false, false, false>), resolve_grid, dim3(RESOLVE_BLOCK), 0, s, r);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

// Counts the members of long runs (of those that are marked: MARKED) per tile, scans the counts and reads the totals back.
template <bool MARKED>
int count_long_runs(Launch& L, ResolveArgs& a, u64* members, u64* strings)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    const RankTables r = rank_tables<COLLECT_TILE>(h, a.m);
    a.tile_agg = r.tile_agg;
    a.tile_splits = r.tile_splits;
    a.tile_prefix = r.tile_prefix;
    a.slab_total = r.slab_total;
    a.slab = r.slab;
    hipLaunchKernelGGL((collect_runs_kernel<MARKED, false>), dim3(r.tiles), dim3(COLLECT_BLOCK), 0, s, a);
    hipLaunchKernelGGL(rerank_scan_kernel, dim3(r.slabs), dim3(1024), 0, s, r.tile_agg, r.tile_prefix, r.tiles, r.slab, r.slab_total,
                       r.tile_splits);
    HIP_TRY(hipGetLastError());
    u32* h_slabs = h->h_pinned + PINNED_HIST;
    const int rc = move_table(h_slabs, r.slab_total, r.slabs * 5 * sizeof(u32), s);
    if (rc)
        return rc;
    HIP_TRY(hipStreamSynchronize(s));
    *members = *strings = 0;
    for (u32 sl = 0; sl < r.slabs; ++sl) {
        *members += h_slabs[sl * 5 + 2];
        *strings += h_slabs[sl * 5 + 3];
    }
    return CSA_OK;
}

// The runs whose codes are marked (long and out of order): their members are collected in list order, radix sorted by their four
// symbols and put back. Works in key[0], key[2] and idx[2..4]: the sorted codes are not needed any more once the members are collected.
int sort_marked_runs(Launch& L, ResolveArgs a, int* passes)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    u64 count = 0, strings = 0;
    int rc = count_long_runs<true>(L, a, &count, &strings);
    if (rc)
        return rc;
    u64* const K[2] = {h->key[2], h->key[0]};
    u32* const V[2] = {h->idx[3], h->idx[4]};
    a.run_keys = K[0];
    a.members = V[0];
    a.places = h->idx[2];
    hipLaunchKernelGGL((collect_runs_kernel<true, true>), dim3((u32)(((u64)a.m + COLLECT_TILE - 1) / COLLECT_TILE)), dim3(COLLECT_BLOCK), 0, s, a);
    HIP_TRY(hipGetLastError());
    int in_out = 0, run = 0;
    rc = radix_sort(L, SRC_PAIRS, 0, 0, K[0], V[0], K[1], V[1], (u32)count, make_plan(0, 64), &in_out, &run);
    if (rc)
        return rc;
    *passes += run;
    a.run_keys = K[in_out];
    a.members = V[in_out];
    hipLaunchKernelGGL(place_marked_kernel, dim3((u32)((count + 255) / 256)), dim3(256), 0, s, a, (u32)count);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

// The members of long runs, in the order of their first word by now, by their second one: collected in list order, radix sorted by the
// ordinal of their string and the code of the next four symbols, resolved like the whole list was and put back. Leaves the
// words that the list is resolved on: 1 if a run of that sort is too long again and out of order (or more than half
// of the list would have to be sorted a second time), 2 otherwise. Works in key[2] and idx[2..4].
int sort_long_runs(Launch& L, CodedList& list)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    ResolveArgs a = list.args;
    u64 count = 0, strings = 0;
    int rc = count_long_runs<false>(L, a, &count, &strings);
    if (rc)
        return rc;
    if (count > h->cap / 2 || count > a.m / 2) {
        list.words = 1;
        return CSA_OK;
    }
    u64* const K[2] = {h->key[2], h->key[2] + h->cap / 2};
    u32* const V[2] = {h->idx[3], h->idx[4]};
    a.run_keys = K[0];
    a.members = V[0];
    a.places = h->idx[2];
    hipLaunchKernelGGL((collect_runs_kernel<false, true>), dim3((u32)(((u64)a.m + COLLECT_TILE - 1) / COLLECT_TILE)), dim3(COLLECT_BLOCK), 0, s, a);
    HIP_TRY(hipMemsetAsync(h->counts + 4, 0, 2 * sizeof(u32), s));
    int in_out = 0;
    rc = radix_sort(L, SRC_PAIRS, 0, 0, K[0], V[0], K[1], V[1], (u32)count, make_plan(0, 32 + bit_length(strings - 1)), &in_out,
                    &list.long_passes);
    if (rc)
        return rc;
    list.long_members = count;
    a.codes = nullptr;
    a.keys = K[in_out];
    a.sufs = V[in_out];
    a.m = (u32)count;
    const dim3 resolve_grid((u32)((count + RESOLVE_TILE - 1) / RESOLVE_TILE));
    if (a.stream)
        hipLaunchKernelGGL((resolve_runs_kernel<RESOLVE_MAX, true, true, true>), resolve_grid, dim3(RESOLVE_BLOCK), 0, s, a);
    else
        hipLaunchKernelGGL((resolve_runs_kernel<RESOLVE_MAX, true, false, true>), resolve_grid, dim3(RESOLVE_BLOCK), 0, s, a);
    HIP_TRY(hipGetLastError());
    rc = move_table(h->h_pinned + 4, h->counts + 4, 2 * sizeof(u32), s);
    if (rc)
        return rc;
    HIP_TRY(hipStreamSynchronize(s));
    if (h->h_pinned[4] != 0)
        list.words = 1;
    list.long_left = h->h_pinned[5] != 0;
    return CSA_OK;
}

// Settles the ties of a list of short groups by where the copies they come from end (copies.hpp).
struct Settle {
    const u16* text;
    u32* sa32;      // the sorted list, whose groups are put in order
    u32 ctx, wide_ell; // symbols the groups are tied on; of the caller's key
    u64 next;          // 0, or the doubling's first context past ctx, where it has none of ctx
    const u32* stream; // null, or the codes of the text's symbols, as for the first sort, the bits of one, and of as many as 64 bits hold
    u32 sym_bits, word_bits;
    bool words;        // written text: groups may be long
    bool settled;   // the list is in order, and the doubling would have gone through num generations more, of these sizes
    u32 num;
    u64 active[SETTLE_CONTEXTS], groups[SETTLE_CONTEXTS];
};

// Whether it is tried. A failed attempt costs the list, the anchors' records and as many steps of a member as SETTLE_STEPS lets it take before
// its tile gives up, and no more for the tiles that start after that: 0.1 to 0.9 ms on texts of 10^4 to 3 * 10^6 symbols made for it, 4 to 6 % of a
// sort of 1.5 or 3 * 10^7 byte symbols of copies over copies. (Of a written text and its copy, tried on two words, 3 * 10^6 symbols 2.79 ms, 2.46 by the doubling alone;
// 3 * 10^7 21.2 and 20.1.)
// A list of copies has two or three members to a group; long groups are runs and periods, whose members agree with
// their neighbours and not with their group's root, or short strings that are in the text a hundred times: members that differ from the root
// in the same way are compared with each other one by one, and one such group holds up a short text. (Written text, us of
// the device a sort settled / doubled: 12000 symbols 316 / 288, 20000, 3.5 members to a group on average, 362 / 292, 33000, 3.9, 635 / 307.
// Token and four-letter texts with copies average 2.0 to 2.3.)
#ifndef CSA_SETTLE_AVG
#define CSA_SETTLE_AVG 3
#endif
constexpr u32 SETTLE_AVG_LIMIT = CSA_SETTLE_AVG;

// Works in key[2] (the anchors' records and bits: two bytes per suffix at most) and the symbol counts of the first sort.
int settle_copies(Launch& L, Settle& st, const RerankArgs& ra, u32 m, u32 groups)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    SettleArgs a;
    memset(&a, 0, sizeof(a));
    a.text = st.text;
    a.n = ra.n;
    a.ctx = st.ctx;
    a.log2_gap = (u32)bit_length(st.ctx) - 1u;
    a.anchors = (a.n >> a.log2_gap) + 1u;
    a.sufs = ra.sufs_out;
    a.gids = ra.gids_out;
    a.gstart = ra.gstart_out;
    a.gprim = ra.gprim_out;
    a.m = m;
    a.groups = groups;
    a.most = st.words ? SETTLE_MAX_WORDS : SETTLE_MAX;
    a.stream = st.stream;
    a.sym_bits = st.sym_bits;
    a.word_bits = st.word_bits;
    a.words[0] = (a.anchors + 63u) / 64u;
    a.words[1] = (a.words[0] + 63u) / 64u;
    a.words[2] = (a.words[1] + 63u) / 64u;
    unsigned char* at = reinterpret_cast<unsigned char*>(h->key[2]);
    unsigned char* const end = at + h->cap * sizeof(u64);
    auto take = [&](u64 bytes) {
        unsigned char* const p = at;
        at += align256(bytes);
        return p;
    };
    a.records = reinterpret_cast<u64*>(take(((u64)a.anchors + 1) * sizeof(u64)));
    for (int i = 0; i < 3; ++i)
        a.links[i] = reinterpret_cast<unsigned long long*>(take((u64)a.words[i] * sizeof(u64)));
    if (at > end)
        return CSA_OK; // (a handle of a few hundred suffixes)
    a.sa32 = st.sa32;
    u64 c = st.next ? st.next : st.ctx;
    do {
        a.contexts[a.num_contexts++] = (u32)(c < a.n ? c : a.n); // (nobody is tied on that many)
        c += c < st.wide_ell ? (c < st.wide_ell - c ? c : st.wide_ell - c) : c;
    } while (c < a.n && a.num_contexts < SETTLE_CONTEXTS);
    constexpr u32 TALLIES = 2 * (SETTLE_CONTEXTS + 1);
    static_assert(SETTLE_SLOTS * TALLIES <= SYMBOLS && SETTLE_SLOTS * TALLIES <= MAX_PASSES * RADIX_BINS, "the tallies take the symbol counts' place, and the histograms' on the host");
    a.tallies = code_tables(h).counts;
    a.failed = h->counts + 4;
    a.err = h->counts + 2;
    TableGroup zeros = {}, seen = {};
    add_table(zeros, a.failed, nullptr, sizeof(u32));
    add_table(zeros, a.tallies, nullptr, SETTLE_SLOTS * TALLIES * sizeof(u32));
    int rc = move_tables(zeros, s);
    if (rc)
        return rc;
    HIP_TRY(hipMemsetAsync(a.records, 0xFF, ((u64)a.anchors + 1) * sizeof(u64), s));
    hipLaunchKernelGGL(copy_roots_kernel, dim3((u32)(((u64)m + 255) / 256)), dim3(256), 0, s, a);
    auto* const links = st.stream ? copy_links_kernel<true> : copy_links_kernel<false>;
    hipLaunchKernelGGL(links, dim3(a.words[1]), dim3(1024), 0, s, a);
    hipLaunchKernelGGL(copy_links_top_kernel, dim3((a.words[1] + 255u) / 256u), dim3(256), 0, s, a);
    hipLaunchKernelGGL(copy_spread_kernel, dim3((u32)(((u64)a.anchors + 255) / 256)), dim3(256), 0, s, a);
    auto* const settle = st.words    ? settle_groups_kernel<SETTLE_WORDS_BLOCK, SETTLE_WORDS_ITEMS, SETTLE_MAX_WORDS, true>
                         : st.stream ? settle_groups_kernel<SETTLE_BLOCK, SETTLE_ITEMS, SETTLE_MAX, true>
                                     : settle_groups_kernel<SETTLE_BLOCK, SETTLE_ITEMS, SETTLE_MAX, false>;
    const u32 block = st.words ? SETTLE_WORDS_BLOCK : SETTLE_BLOCK, tile = block * (st.words ? SETTLE_WORDS_ITEMS : SETTLE_ITEMS);
    hipLaunchKernelGGL(settle, dim3((u32)(((u64)m + tile - 1) / tile)), dim3(block), 0, s, a);
    HIP_TRY(hipGetLastError());
    u32* const h_tallies = h->h_pinned + PINNED_HIST;
    add_table(seen, h_tallies, a.tallies, SETTLE_SLOTS * TALLIES * sizeof(u32));
    rc = read_counts(L, nullptr, seen);
    if (rc || h->h_pinned[4] != 0)
        return rc;
    u64 members[SETTLE_CONTEXTS + 1] = {}, starts[SETTLE_CONTEXTS + 1] = {};
    for (u32 slot = 0; slot < SETTLE_SLOTS; ++slot)
        for (u32 i = 0; i <= SETTLE_CONTEXTS; ++i) {
            members[i] += h_tallies[slot * TALLIES + i];
            starts[i] += (u64)(int64_t)(int32_t)h_tallies[slot * TALLIES + SETTLE_CONTEXTS + 1 + i];
        }
    // a list on context i holds the members tied on more than i contexts, and the groups that start at or before it and have not ended
    u64 above = 0;
    for (int i = (int)a.num_contexts - 1; i >= 0; --i)
        st.active[i] = above += members[i + 1];
    u64 open = 0;
    for (u32 i = 0; i < a.num_contexts; ++i)
        st.groups[i] = open += starts[i];
    st.num = 0;
    while (st.num < a.num_contexts && st.active[st.num] > 0)
        ++st.num;
    st.settled = true;
    return CSA_OK;
}

// Settles a list whose groups are runs and periods (chains.hpp): num generations of the doubling from the one about to begin, with the
// sizes that they would have had.
struct Chains {
    bool settled;
    u32 num;
    u32 active[SETTLE_CONTEXTS], groups[SETTLE_CONTEXTS], big[SETTLE_CONTEXTS];
    bool small_only[SETTLE_CONTEXTS];
};
constexpr u32 CHAIN_TRIES = 2; // failed attempts (two passes over the list and a round trip; a generation costs five times as much)

// Works in `scratch` ([groups]) and the symbol counts of the first sort.
int settle_chains(Launch& L, Chains& ch, const u16* d_text, u32 n, u64 ctx, u64 wide_ell, const u32* sufs, const u32* gids, const u32* gstart,
                  const u32* gprim, u32 m, u32 groups, u32* scratch, u32* sa32)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    ChainArgs a;
    memset(&a, 0, sizeof(a));
    memset(&ch, 0, sizeof(ch));
    a.text = d_text;
    a.n = n;
    a.ctx = (u32)ctx;
    a.sufs = sufs;
    a.gids = gids;
    a.gstart = gstart;
    a.gprim = gprim;
    a.m = m;
    a.groups = groups;
    a.sa32 = sa32;
    a.backwards = scratch;
    a.limit_lo = SMALL_MAXG;
    a.limit_hi = SMALL_MAXG_HI;
    u64 c = ctx;
    do {
        a.contexts[a.num_contexts++] = (u32)c;
        c += c < wide_ell ? (c < wide_ell - c ? c : wide_ell - c) : c;
    } while (c < n && a.num_contexts < SETTLE_CONTEXTS);
    a.tallies = code_tables(h).counts;
    a.failed = h->counts + 4;
    a.err = h->counts + 2;
    constexpr u32 TALLIES = SETTLE_CONTEXTS * CHAIN_TALLIES;
    static_assert(TALLIES <= SYMBOLS && TALLIES <= MAX_PASSES * RADIX_BINS, "the tallies take the symbol counts' place, and the histograms' on the host");
    TableGroup zeros = {}, seen = {};
    add_table(zeros, a.failed, nullptr, sizeof(u32));
    add_table(zeros, a.tallies, nullptr, TALLIES * sizeof(u32));
    int rc = move_tables(zeros, s);
    if (rc)
        return rc;
    hipLaunchKernelGGL(chain_groups_kernel, dim3((groups + 255) / 256), dim3(256), 0, s, a);
    hipLaunchKernelGGL(chain_place_kernel, dim3((u32)(((u64)m + 255) / 256)), dim3(256), 0, s, a);
    HIP_TRY(hipGetLastError());
    u32* const tallies = h->h_pinned + PINNED_HIST;
    add_table(seen, tallies, a.tallies, TALLIES * sizeof(u32));
    u32 failed = 0;
    rc = read_counts(L, &failed, seen);
    if (rc || failed)
        return rc;
    bool all_small = false;
    for (; ch.num < a.num_contexts && tallies[ch.num * CHAIN_TALLIES] > 0; ++ch.num) {
        const u32* const w = tallies + ch.num * CHAIN_TALLIES;
        ch.active[ch.num] = w[0];
        ch.groups[ch.num] = w[1];
        ch.small_only[ch.num] = all_small;
        ch.big[ch.num] = all_small ? 0u : (u64)w[0] <= (u64)w[1] * SMALL_AVG_LIMIT ? w[3] : w[2];
        all_small = all_small || ch.big[ch.num] == 0;
    }
    ch.settled = true;
    return CSA_OK;
}

// Generation 0: ranks the sorted list described by `ra`: counts per tile, scans the counts, reads the totals back, then
// applies them and brings rank[] up to date, directly from the kernel or through the two-pass bucketed update.
// coded: the list comes from sort_by_codes and carries its ties. settle: the ties of a list of short groups are settled at once if possible; the
// ranks are not needed then, nor are they when nothing is tied. counted: the counts are in the tables, and *survivors, *groups and *rank_update are set.
int rerank_step(Launch& L, RerankArgs& ra, const DeferBuffers& buf, u32* survivors, u32* groups, int* rank_update,
                u32* level_counts = nullptr, CodedList* coded = nullptr, int* passes = nullptr, Settle* settle = nullptr,
                bool counted = false)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    const RankTables r = rank_tables<RANK_TILE>(h, ra.m);
    ra.tile_agg = r.tile_agg;
    ra.tile_prefix = r.tile_prefix;
    ra.tile_splits = r.tile_splits;
    ra.slab_total = r.slab_total;
    ra.slab = r.slab;
    ra.err = h->counts + 2;
    ra.rank_recs = nullptr;
    // the level counts of packed keys ride along: accumulated in the (idle) digit histograms, read back with the totals
    unsigned long long* const h_levels = reinterpret_cast<unsigned long long*>(h->h_pinned + PINNED_HIST + 512);
    ra.level_totals = reinterpret_cast<unsigned long long*>(h->ghist);
    auto count_and_read = [&]() -> int {
        const bool levels = ra.levels > 0 || coded;
        if (levels)
            HIP_TRY(hipMemsetAsync(ra.level_totals, 0, LEVEL_SLOTS * 8 * sizeof(unsigned long long), s));
        TableGroup beside = {};
        if (coded) {
            ra.words = coded->words;
            ra.words_known = coded->told ? nullptr : coded->args.words_out;
            // (several tiles a wave on long lists: fewer additions to the level totals)
            const u32 per_wave = r.tiles >= (1u << 15) ? 8u : 1u, waves = (r.tiles + per_wave - 1) / per_wave;
            if (coded->by_levels)
                hipLaunchKernelGGL((count_ties_kernel<RANK_TILE, WORD_LEVELS>), dim3((waves + 3) / 4), dim3(256), 0, s, ra, r.tiles, per_wave);
            else
                hipLaunchKernelGGL((count_ties_kernel<RANK_TILE>), dim3((waves + 3) / 4), dim3(256), 0, s, ra, r.tiles, per_wave);
            if (ra.levels > 0)
                hipLaunchKernelGGL(count_code_levels_kernel, dim3(hist_blocks(256 * 16, ra.m)), dim3(256), 0, s, ra, coded->args.codes, ra.levels);
        } else {
            hipLaunchKernelGGL((rerank_count_kernel<RANK_BLOCK, RANK_ITEMS>), dim3(r.tiles), dim3(RANK_BLOCK), 0, s, ra);
        }
        if (levels)
            add_table(beside, h_levels, ra.level_totals, LEVEL_SLOTS * 8 * sizeof(unsigned long long));
        return rank_totals(L, r, true, ra.m, ra.n, false, survivors, groups, rank_update, beside);
    };
    int rc = counted ? CSA_OK : count_and_read();
    if (rc)
        return rc;
    if (coded && !coded->by_levels) {
        coded->words = ra.words = h->h_pinned[6];
        coded->told = true;
        const bool unordered = h->h_pinned[4] != 0, second = h->h_pinned[5] != 0 && coded->words == 2;
        if (unordered && (rc = sort_marked_runs(L, coded->args, passes)) != CSA_OK) // long runs of one code are out of order: they are sorted now
            return rc;
        if (second && (rc = sort_long_runs(L, *coded)) != CSA_OK)
            return rc;
        if ((unordered || second) && (rc = count_and_read()) != CSA_OK)
            return rc;
    }
    const u32 levels = ra.levels + (coded ? coded->words - 1 : 0);
    for (u32 i = 0; i < levels && level_counts; ++i) {
        u64 sv = 0, hd = 0;
        for (u32 slot = 0; slot < LEVEL_SLOTS; ++slot) {
            sv += h_levels[slot * 8 + 2 * i];
            hd += h_levels[slot * 8 + 2 * i + 1];
        }
        level_counts[2 * i] = (u32)sv;
        level_counts[2 * i + 1] = (u32)hd;
    }
    if (settle && *survivors == 0) {
        *rank_update = 0;
        return CSA_OK;
    }
    if (settle && (u64)*survivors <= (u64)*groups * SETTLE_AVG_LIMIT && !(coded && coded->long_left)) {
        RerankArgs list = ra;
        list.rank = nullptr;
        if (coded)
            hipLaunchKernelGGL((compact_ties_kernel<RANK_TILE>), dim3((r.tiles + 3) / 4), dim3(256), 0, s, list, r.tiles);
        else
            hipLaunchKernelGGL((rerank_kernel<RANK_BLOCK, RANK_ITEMS, false>), dim3(r.tiles), dim3(RANK_BLOCK), 0, s, list);
        HIP_TRY(hipGetLastError());
        if (coded)
            settle->ctx *= coded->words;
        rc = settle_copies(L, *settle, ra, *survivors, *groups);
        if (rc)
            return rc;
        if (settle->settled) {
            *rank_update = 0;
            return CSA_OK;
        }
    }
    // what the list becomes decides what rank[] is to hold: ordinals for a dense generation, ranks otherwise
    ra.ordinals = dense_generation(*survivors, *groups, ra.n) ? 1u : 0u;
    if (*rank_update != 0)
        ra.rank_recs = buf.recs[0];
    if (coded)
        hipLaunchKernelGGL((rerank_kernel<RANK_BLOCK, RANK_ITEMS, true>), dim3(r.tiles), dim3(RANK_BLOCK), 0, s, ra);
    else
        hipLaunchKernelGGL((rerank_kernel<RANK_BLOCK, RANK_ITEMS, false>), dim3(r.tiles), dim3(RANK_BLOCK), 0, s, ra);
    HIP_TRY(hipGetLastError());
    if (*rank_update == 1)
        return deferred_rank_update(L, buf, ra.n);
    return CSA_OK;
}

// Written text (word_keys.hpp): texts of at least this many symbols over 17 to 128 values (a symbol of eight bits gains nothing in the first word). Below,
// its round trips and launches cost as much as they save: 40000 letters of written text take 361 us by the doubling and 364 this way, independent ones of an
// alphabet of 20 217 and 238; 3 * 10^5 of written text 681 and 416. Texts that the second words are left out of (choose_seconds_kernel) are
// counted once, on the context that the doubling goes on from, and take what they took on keys of eight symbols: 2^18 symbols of log lines 940 us and 934, 10^6 1206 and
// 1193, 2 * 10^7 5.41 ms and 5.39, with runs of spaces 4.29 and 4.33.
// More than 64 values, which leave nine symbols to a word, from four times as many on (us on keys of eight symbols and by words: independent letters of 100 2^18 symbols 234 / 240,
// 3.5 * 10^5 240 / 246, 2^19 257 / 259, 10^6 291 / 293, 4 * 10^6 453 / 413; of written text with capitals, digits and marks 507 / 518, 565 / 552, 581 / 582, 663 / 632,
// 967 / 873; the same over 60 values 505 / 340, 569 / 358, 577 / 570, 659 / 623).
#ifndef CSA_WORD_KEYS_MIN
#define CSA_WORD_KEYS_MIN (1u << 18)
#endif
#ifndef CSA_WORD_KEYS_MIN_SEVEN_BITS
#define CSA_WORD_KEYS_MIN_SEVEN_BITS (1u << 20)
#endif
// Texts with a run or a period that the settling would give up at: the second words are read from this many symbols on, and the doubling goes on from them. (us with
// the second words left out / read: 10^6 letters of written text with a period of 11 over 1 % of them 1138 / 1175, 2 * 10^6 1212 / 1339, 4 * 10^6 1529 / 1537, 5.6 * 10^6
// 1740 / 1721, 1.2 * 10^7 2748 / 2540; with 2 % in runs of spaces 1257 / 1303, 1396 / 1443, 1746 / 1736, 1863 / 1878, 2941 / 2827.)
#ifndef CSA_WORD_ENDLESS_MIN
#define CSA_WORD_ENDLESS_MIN (1u << 22)
#endif
static_assert(CSA_WORD_KEYS_MIN * sizeof(u64) >= sizeof(u32) << WINDOW_BITS<7>, "the windows are counted in a list of keys");

// What sort_by_words leaves.
struct WordList {
    WordLevels levels;      // contexts that the list has been counted on: the doubling's, and the two words
    u32 survivors[WORD_LEVELS], groups[WORD_LEVELS]; // on each
    u32 valid;              // levels on which the order and the ties are those of the suffixes
    u32 members, runs;      // of long runs, sorted by the second word in ...
    int passes;             // ... so many radix passes
};

// The sorted first words of a text (syms symbols of ps.sym_bits bits each), resolved on the second ones: keys and sufs -> sufs_out, and the ties. `spare` holds the
// keys, which are not needed once the tiles are resolved. Works in key[2], idx[2..4] and spare.
int sort_by_words(Launch& L, u32 n, const TextSource& ps, u32 syms, u64* spare, const u32* sufs, u32* sufs_out, u8* ties, RerankArgs& ra, WordList& list)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    WordArgs a;
    memset(&a, 0, sizeof(a));
    a.keys = spare;
    a.sufs = sufs;
    a.n = n;
    a.stream = ps.stream;
    a.bits = ps.sym_bits;
    a.syms = syms;
    a.levels = list.levels;
    a.sufs_out = sufs_out;
    a.ties = ties;
    a.any_long = h->counts + 5;
    int rc = move_table(a.any_long, nullptr, sizeof(u32), s);
    if (rc)
        return rc;
    hipLaunchKernelGGL(resolve_words_kernel, dim3((u32)(((u64)n + RESOLVE_TILE - 1) / RESOLVE_TILE)), dim3(RESOLVE_BLOCK), 0, s, a);
    HIP_TRY(hipGetLastError());
    ra.ties = ties;
    ra.sufs = sufs_out;
    ra.words = list.levels.count;
    ra.words_known = nullptr;
    ra.first_level = 0;
    ra.levels = 0;
    const RankTables r = rank_tables<RANK_TILE>(h, n);
    unsigned long long* const h_levels = reinterpret_cast<unsigned long long*>(h->h_pinned + PINNED_HIST + 512);
    auto count_and_read = [&]() -> int {
        ra.tile_agg = r.tile_agg;
        ra.tile_prefix = r.tile_prefix;
        ra.tile_splits = r.tile_splits;
        ra.slab_total = r.slab_total;
        ra.slab = r.slab;
        ra.level_totals = reinterpret_cast<unsigned long long*>(h->ghist);
        HIP_TRY(hipMemsetAsync(ra.level_totals, 0, LEVEL_SLOTS * 8 * sizeof(unsigned long long), s));
        const u32 per_wave = r.tiles >= (1u << 15) ? 8u : 1u, waves = (r.tiles + per_wave - 1) / per_wave;
        hipLaunchKernelGGL((count_ties_kernel<RANK_TILE, WORD_LEVELS>), dim3((waves + 3) / 4), dim3(256), 0, s, ra, r.tiles, per_wave);
        TableGroup beside = {};
        add_table(beside, h_levels, ra.level_totals, LEVEL_SLOTS * 8 * sizeof(unsigned long long));
        u32 survivors = 0, groups = 0;
        int update = 0;
        const int read = rank_totals(L, r, true, n, n, false, &survivors, &groups, &update, beside);
        for (u32 i = 0; i < list.levels.count; ++i) {
            u64 sv = 0, hd = 0;
            for (u32 slot = 0; slot < LEVEL_SLOTS; ++slot) {
                sv += h_levels[slot * 8 + 2 * i];
                hd += h_levels[slot * 8 + 2 * i + 1];
            }
            list.survivors[i] = (u32)sv;
            list.groups[i] = (u32)hd;
        }
        return read;
    };
    if ((rc = count_and_read()) != CSA_OK)
        return rc;
    list.valid = list.levels.count;
    if (h->h_pinned[5] == 0)
        return CSA_OK;
    // The members of long runs: more than a quarter of the text in them are left to the doubling (runs, padding, few words).
    list.valid = list.levels.in_first;
    const RankTables cr = rank_tables<COLLECT_TILE>(h, n);
    a.tile_agg = cr.tile_agg;
    a.tile_splits = cr.tile_splits;
    a.tile_prefix = cr.tile_prefix;
    a.slab_total = cr.slab_total;
    a.slab = cr.slab;
    hipLaunchKernelGGL(collect_words_kernel<false>, dim3(cr.tiles), dim3(COLLECT_BLOCK), 0, s, a);
    hipLaunchKernelGGL(rerank_scan_kernel, dim3(cr.slabs), dim3(1024), 0, s, cr.tile_agg, cr.tile_prefix, cr.tiles, cr.slab, cr.slab_total, cr.tile_splits);
    HIP_TRY(hipGetLastError());
    u32* const h_slabs = h->h_pinned + PINNED_HIST;
    if ((rc = move_table(h_slabs, cr.slab_total, cr.slabs * 5 * sizeof(u32), s)) != CSA_OK)
        return rc;
    HIP_TRY(hipStreamSynchronize(s));
    u64 members = 0, runs = 0;
    for (u32 sl = 0; sl < cr.slabs; ++sl) {
        members += h_slabs[sl * 5 + 2];
        runs += h_slabs[sl * 5 + 3];
    }
    if (members > n / 4 || members > h->cap / 2)
        return count_and_read(); // (the tables of the tiles have been used)
    list.members = (u32)members;
    list.runs = (u32)runs;
    u64* const K[2] = {h->key[2], h->key[2] + h->cap / 2};
    u32* const V[2] = {h->idx[3], h->idx[4]};
    a.run_keys = K[0];
    a.run_slots = V[0];
    a.words2 = spare;
    a.members = reinterpret_cast<u32*>(spare + h->cap / 2);
    a.ordinals = a.members + h->cap / 2;
    a.places = h->idx[2];
    hipLaunchKernelGGL(collect_words_kernel<true>, dim3(cr.tiles), dim3(COLLECT_BLOCK), 0, s, a);
    HIP_TRY(hipGetLastError());
    int first = 0, second = 0, run = 0;
    rc = radix_sort(L, SRC_PAIRS, 0, 0, K[0], V[0], K[1], V[1], list.members, make_plan(0, (int)(ps.sym_bits * syms)), &first, &run);
    if (rc)
        return rc;
    list.passes = run;
    const dim3 member_grid((u32)((members + 255) / 256));
    hipLaunchKernelGGL(gather_ordinals_kernel, member_grid, dim3(256), 0, s, (const u32*)a.ordinals, (const u32*)V[first], list.members, K[first]);
    rc = radix_sort(L, SRC_PAIRS, 0, 0, K[first], V[first], K[first ^ 1], V[first ^ 1], list.members, make_plan(0, bit_length(runs - 1 ? runs - 1 : 1)), &second, &run);
    if (rc)
        return rc;
    list.passes += run;
    a.run_slots = V[first ^ second];
    hipLaunchKernelGGL(place_words_kernel, member_grid, dim3(256), 0, s, a, list.members);
    HIP_TRY(hipGetLastError());
    list.valid = list.levels.count;
    return count_and_read();
}

// The contexts of a list that is resolved on two words of syms symbols: the doubling's from the caller's key on, the last of those before it that the first
// word holds, from which the doubling may go on, and the two words themselves.
// (Evaluated for all of them by the compiler, which does not let one past the last level be written.)
constexpr WordLevels word_levels(u32 syms, u32 bits, u64 wide_ell)
{
    WordLevels l = {};
    auto next = [=](u64 c) { return c + (c < wide_ell ? (c < wide_ell - c ? c : wide_ell - c) : c); };
    auto add = [&](u64 c) {
        l.in_first += c <= syms ? 1u : 0u;
        l.context[l.count] = (u32)c;
        l.drop[l.count++] = (u32)(c <= syms ? syms - c : 2 * syms - c) * bits;
    };
    for (u64 c = 4; c <= 2 * syms; c = next(c))
        if (c >= wide_ell || (c <= syms && next(c) > syms))
            add(c);
    if (l.context[l.count - 1] != 2 * syms)
        add(2 * syms);
    return l;
}

template <u32 BITS>
constexpr bool word_levels_fit()
{
    constexpr WordLevels of[4] = {word_levels(64 / BITS, BITS, 4), word_levels(64 / BITS, BITS, 8), word_levels(64 / BITS, BITS, 12), word_levels(64 / BITS, BITS, 16)};
    for (const WordLevels& l : of)
        if (l.in_first == 0 || l.in_first > l.count)
            return false;
    return true;
}
static_assert(word_levels_fit<5>() && word_levels_fit<6>() && word_levels_fit<7>(), "some key width has no context of the doubling inside the first word");

// Texts of this length on are looked at before their bytes are counted (text_byte_hist_kernel). us of that kernel without the look and with it, independent ids / 26
// letters, which are counted all the same: 2^18 symbols 5.2, 4.1 / 5.1, 7.9; 2^20 7.3, 4.8 / 6.2, 9.4; 2^22 12.5, 5.0 / 10.5, 12.9; 2^24 23.0, 5.7 / 19.2, 23.3. From 2^20
// symbols on the look saves the one as much as it costs the other, and more and more in longer texts (2^22 2 % of the sort and 1 %).
#ifndef CSA_BYTE_LOOK_MIN
#define CSA_BYTE_LOOK_MIN (1u << 20)
#endif
constexpr u32 BYTE_LOOK_MIN = CSA_BYTE_LOOK_MIN;

// Texts of up to this many symbols are ranked by counting (short_text.hpp).
#ifndef CSA_SHORT_TEXT
#define CSA_SHORT_TEXT SHORT_MAX
#endif

// The whole sort of a short text: one round trip, and a second one where a group of suffixes that are tied on four symbols is long. Works in gid, rank and
// the symbol counts.
int sort_short_text(Launch& L, const u16* d_text, u32 n, u64 index_base, u8* d_sa40)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    csa_stats* st = L.stats;
    RangeScope range("sort_short_text n=%u", n);
    u32* const ranks[2] = {h->gid, h->rank};
    ShortArgs a;
    memset(&a, 0, sizeof(a));
    a.text = d_text;
    a.n = n;
    a.index_base = index_base;
    a.out = d_sa40;
    a.rank_out = ranks[0];
    a.counters = code_tables(h).counts;
    const u64 wide_ell = 4ull * (u64)h->key_words;
    u32 last = 0; // generation
    for (u64 ctx = 4; ctx < n && last + 1 < SHORT_GENERATIONS - 1;) {
        const u64 hop = ctx < wide_ell ? (ctx < wide_ell - ctx ? ctx : wide_ell - ctx) : ctx;
        a.hops[++last] = (u32)hop;
        ctx += hop;
    }
    const dim3 grid((n + SHORT_X - 1) / SHORT_X);
    HIP_TRY(hipEventRecord(h->ev_gen[0], s));
    int rc = move_table(a.counters, nullptr, SHORT_COUNTERS * sizeof(u32), s);
    if (rc)
        return rc;
    hipLaunchKernelGGL(short_first_kernel, grid, dim3(SHORT_BLOCK), 0, s, a);
    a.generation = 1;
    a.rank_in = ranks[0];
    hipLaunchKernelGGL(short_rest_kernel, dim3(1), dim3(SHORT_BLOCK), 0, s, a);
    u32* const seen = h->h_pinned + PINNED_HIST;
    static_assert(SHORT_COUNTERS <= MAX_PASSES * RADIX_BINS && SHORT_COUNTERS <= SYMBOLS, "the counters fit the tables they are kept in");
    if ((rc = move_table(seen, a.counters, SHORT_COUNTERS * sizeof(u32), s)) != CSA_OK)
        return rc;
    HIP_TRY(hipEventRecord(h->ev_gen[1], s));
    HIP_TRY(hipStreamSynchronize(s));
    if (seen[SHORT_LONG] != 0) {
        for (u32 g = 1; g <= last; ++g) {
            a.generation = g;
            a.rank_in = ranks[(g - 1) & 1];
            a.rank_out = ranks[g & 1];
            hipLaunchKernelGGL(short_next_kernel, grid, dim3(SHORT_BLOCK), 0, s, a);
        }
        if ((rc = move_table(seen, a.counters, SHORT_COUNTERS * sizeof(u32), s)) != CSA_OK)
            return rc;
        HIP_TRY(hipEventRecord(h->ev_gen[1], s));
        HIP_TRY(hipStreamSynchronize(s));
    }
    // the generations of the caller's key width: those before it has been reached belong to generation 0
    u32 folded = 0, generations = 1;
    for (u64 c = 4; c < wide_ell; c += (c < wide_ell - c ? c : wide_ell - c))
        ++folded;
    while (generations < SHORT_GENERATIONS && seen[2 * generations] != 0)
        ++generations;
    if (generations > last + 1)
        return fail(CSA_ERR_INTERNAL, "%u suffixes of a short text are tied after the last generation", seen[2 * (generations - 1)]);
    folded = folded < generations - 1 ? folded : generations - 1;
    st->generations = (int)(generations - folded);
    st->active[0] = n;
    for (u32 g = 1; g + folded < generations; ++g) {
        st->active[g] = seen[2 * (g + folded)];
        st->groups[g] = seen[2 * (g + folded) + 1];
    }
    st->key_symbols = 4;
    st->first_sort_generations = 1;
    HIP_TRY(hipEventElapsedTime(&st->ms[0], h->ev_gen[0], h->ev_gen[1]));
    st->ms_total = st->ms[0];
    return CSA_OK;
}

int sort_partition(Launch& L, const u16* d_text, u64 n64, u64 index_base, u8* d_sa40)
{
    csa_handle* h = L.h;
    hipStream_t s = L.stream;
    csa_stats* st = L.stats;
    const u32 n = (u32)n64;
    // (a caller who has set thresholds of the large sort, or asks for the times of its passes, gets that one)
    if (n <= CSA_SHORT_TEXT && h->pack_symbols && h->settle && !h->expect_presorted && !(L.flags & CSA_FLAG_KERNEL_TIMING))
        return sort_short_text(L, d_text, n, index_base, d_sa40);
    // Wide keys are not sorted word by word. A generation 0 that resolves 4 W symbols is what doubling on one-word keys
    // reaches after one or two more generations (4 -> 8 -> 16 symbols; 4 -> 8 -> 12 with the second step looking only 4
    // symbols ahead; the order of suffixes that run off the text is the same: the shorter first). So the sort always
    // starts from one-word keys, steps up to the context of the wide key, reports those generations as its generation 0
    // and doubles from there. Every reported generation then has the context, the ranks and the active set of the wide-key
    // generation it stands for. A 4-word key sorted word by word costs 32 radix passes over all suffixes (316 ms on the
    // 1B-token workload); this way it costs what the one-word key costs.
    const u64 wide_ell = 4ull * (u64)h->key_words;

    RangeScope range_sort("sort_partition n=%u", n);
    HIP_TRY(hipEventRecord(h->ev_gen[0], s));

    // ---- generation 0: every suffix sorted by its first symbols (four of them, by codes or K-gram keys, or as many as a packed
    // key holds), ties of tail suffixes broken by length ----
    RangeScope range_gen0("generation 0 m=%u", n);
    // The byte histograms of the text come first: they tell whether the alphabet is small enough for keys of more than four
    // symbols. (The digit counts are zeroed with them.)
    TableGroup zeros = {};
    add_table(zeros, h->counts, nullptr, 14 * sizeof(u32));
    add_table(zeros, h->ghist, nullptr, (MAX_PASSES + 2) * RADIX_BINS * sizeof(u32));
    int rc = move_tables(zeros, s);
    if (rc)
        return rc;
    u32* const bytehist = h->ghist + MAX_PASSES * RADIX_BINS;
    PackedPlan pp;
    memset(&pp, 0, sizeof(pp));
    // A workgroup for every 8 K symbols until there is one per CU (10^6 symbols: 12.5 us with 31 of them, 7.3 with 123), then for every
    // 32 K: more of them add the same counters more often (2 * 10^7 symbols: 1 % of the sort).
    u32 count_blocks = hist_blocks(256 * 2 * 16, n);
    count_blocks = count_blocks < 256u ? count_blocks : 256u;
    if (hist_blocks(256 * 8 * 16, n) > count_blocks)
        count_blocks = hist_blocks(256 * 8 * 16, n);
    auto count_bytes = [&](bool look) {
        if (look)
            hipLaunchKernelGGL(text_byte_hist_kernel<true>, dim3(count_blocks), dim3(256), 0, s, d_text, n, bytehist);
        else
            hipLaunchKernelGGL(text_byte_hist_kernel<false>, dim3(count_blocks), dim3(256), 0, s, d_text, n, bytehist);
    };
    bool bytes_counted = false;
    ProbeCounts* const seen = reinterpret_cast<ProbeCounts*>(h->h_pinned + PINNED_HIST + 2 * RADIX_BINS); // (behind the byte counts)
    if (h->pack_symbols) {
        count_bytes(n >= BYTE_LOOK_MIN);
        u32* h_bytes = h->h_pinned + PINNED_HIST;
        if ((rc = move_table(h_bytes, bytehist, 2 * RADIX_BINS * sizeof(u32), s)) != CSA_OK)
            return rc;
        // The symbols are sampled meanwhile: the device would stand still until the host has seen the counts, and then start with that.
        // (10^6 independent ids: 238 us with a wait in between, 226 without.)
        HIP_TRY(hipEventRecord(h->ev_gen[2], s)); // (recorded again when a generation ends)
        if ((rc = share_symbols(L, d_text, n, seen, bytehist)) != CSA_OK)
            return rc;
        HIP_TRY(hipEventSynchronize(h->ev_gen[2]));
        pp = plan_packed_text(h_bytes, n, h->key_words, (u64)h->cap * sizeof(u32));
        u64 counted_symbols = 0;
        for (u32 d = 0; d < RADIX_BINS; ++d)
            counted_symbols += h_bytes[d];
        bytes_counted = counted_symbols == n;
    }
    TextSource ps;
    memset(&ps, 0, sizeof(ps));
    const bool by_words = pp.values > 16 && pp.values <= 128 && n >= (pp.values > 64 ? CSA_WORD_KEYS_MIN_SEVEN_BITS : CSA_WORD_KEYS_MIN) && h->pack_symbols && h->settle && !h->expect_presorted;
    const u32 word_bits = by_words ? (u32)bit_length(pp.values - 1) : 0u, word_syms = by_words ? 64u / word_bits : 0u;
    const PackedPlan as_reported = pp; // what callers are told of the first sort of such texts
    if (by_words)
        pp.enabled = false;
    bool narrow = false; // keys of half as many packed symbols
    const bool in_buckets = n >= CSA_BUCKETS_MIN && h->pack_symbols;
    CodeDigits digits = ALL_DIGITS, counted = ALL_DIGITS;
    if (pp.enabled) {
        // the code stream lives in rank[], which nothing uses before the sorted list is ranked
        u32* const stream = h->rank;
        ps.stream = stream;
        ps.sym_bits = pp.codes.bits;
        ps.key_bits = pp.codes.key_syms * pp.codes.bits;
        ps.words = ((u64)n * ps.sym_bits + 31) / 32 + 4;
        if ((rc = move_table(bytehist, nullptr, RADIX_BINS * sizeof(u32), s)) != CSA_OK) // (read back already)
            return rc;
        const u64 enc_blocks = (ps.words + ENCODE_BLOCK - 1) / ENCODE_BLOCK;
        hipLaunchKernelGGL(encode_text_kernel, dim3((u32)(enc_blocks < 4096 ? enc_blocks : 4096)), dim3(ENCODE_BLOCK), 0, s, d_text, n,
                           pp.codes, stream, ps.words, bytehist);
        HIP_TRY(hipGetLastError());
        if (n >= CSA_NARROW_MIN && ps.sym_bits == 2 && ps.key_bits == 64 && pp.skipped > 0 && (rc = narrow_keys_pay(L, ps, n, &narrow, &digits)) != CSA_OK)
            return rc;
    }
    // symbols of a key of the first sort, or that its list will be taken to be resolved on
    u32 ell = pp.enabled ? (narrow ? pp.codes.key_syms / 2 : pp.codes.key_syms) : 4u;
    int folded = 0; // generations after the first that still belong to the reported generation 0
    for (u64 c = ell; c < wide_ell; c += (c < wide_ell - c ? c : wide_ell - c))
        ++folded;
    // suffixes that come first, shortest first: those that run off the text inside what the first sort resolves
    const u32 front = by_words ? 2 * word_syms : ell, tail = n < front ? n : front;
    bool coded = !pp.enabled && !pp.byte_wide && !by_words;
    if (coded) {
        const bool probed = n >= PROBE_MIN, ahead = !probed || n < CODE_AHEAD_MAX;
        if (!h->pack_symbols || pp.few) { // (few symbols, and no packed keys for them)
            if ((rc = move_table(h->counts + 5, nullptr, sizeof(u32), s)) != CSA_OK || (rc = share_symbols(L, d_text, n, seen, nullptr)) != CSA_OK)
                return rc;
        }
        if (ahead && (rc = code_suffixes(L, d_text, n, tail, counted)) != CSA_OK)
            return rc;
        if (probed) {
            HIP_TRY(hipEventSynchronize(h->ev_gen[1]));
            coded = codes_pay(*seen, n);
            if (coded && in_buckets && !ahead && buckets_fit(*seen, n, bucket_digits(n, false), false))
                digits = bucket_digits(n, false);
        }
        if (coded && !ahead && (rc = code_suffixes(L, d_text, n, tail, counted = digits)) != CSA_OK)
            return rc;
    }
    int passes = 0, p1 = 0, in_out = 0;
    u64* K[2] = {h->key[0], h->key[1]};
    u32* V[2] = {h->idx[0], h->idx[1]};
    int cur = 0; // the (K, V) set that holds the sorted pairs
    CodedList list;
    if (by_words) {
        SymbolCodes codes = pp.codes;
        codes.bits = word_bits;
        codes.key_syms = word_syms;
        ps.stream = h->rank;
        ps.sym_bits = word_bits;
        ps.key_bits = word_bits * word_syms;
        ps.words = ((u64)n * word_bits + 31) / 32 + 4;
        u32* const windows = reinterpret_cast<u32*>(K[1]); // (the first pass writes it, afterwards)
        hipLaunchKernelGGL(encode_words_kernel, dim3((u32)((ps.words + WORD_SPAN - 1) / WORD_SPAN)), dim3(WORD_BLOCK), 0, s, d_text, n, codes, h->rank, ps.words,
                           windows, 1u << (word_bits + 7));
        const u32 blocks = hist_blocks(WINDOW_BLOCK * 4, n);
        auto* const count = word_bits == 5 ? window_hist_kernel<5> : word_bits == 6 ? window_hist_kernel<6> : window_hist_kernel<7>;
        hipLaunchKernelGGL(count, dim3(blocks < WINDOW_HIST_BLOCKS ? blocks : WINDOW_HIST_BLOCKS), dim3(WINDOW_BLOCK), 0, s, (const u32*)h->rank, n, windows);
        auto* const expand = word_bits == 5 ? word_digits_kernel<5> : word_bits == 6 ? word_digits_kernel<6> : word_digits_kernel<7>;
        const PassPlan plan = make_plan(0, (int)ps.key_bits); // (digits of eight bits, and what is left)
        hipLaunchKernelGGL(expand, dim3(plan.num_passes), dim3(WINDOW_BLOCK), 0, s, (const u32*)h->rank, (const u32*)windows, n, ps.key_bits, h->ghist, h->digit_base);
        ps.scanned = true;
        HIP_TRY(hipGetLastError());
        rc = radix_sort(L, SRC_PACKED, n, tail, K[0], V[0], K[1], V[1], n, plan, &in_out, &p1, nullptr, 0, 0, &ps);
    } else if (pp.enabled) {
        const PassPlan plan = make_plan(0, narrow ? 32 : (int)ps.key_bits);
        hipLaunchKernelGGL(packed_hist_expand_kernel, dim3(1), dim3(256), 0, s, ps.stream, n, ps.sym_bits, ell, plan.num_passes, bytehist,
                           h->ghist);
        HIP_TRY(hipGetLastError());
        coded = narrow;
        if (narrow) {
            TableGroup cleared = {};
            add_table(cleared, code_tables(h).marks, nullptr, RESOLVE_MARK_WORDS * sizeof(u32));
            add_table(cleared, h->counts + 5, nullptr, sizeof(u32)); // (the sampling of the symbols has been called off with it)
            if ((rc = move_tables(cleared, s)) != CSA_OK)
                return rc;
            rc = sort_by_codes(L, d_text, n, tail, 2u, list, ALL_DIGITS, digits, &p1, &ps, ell);
            in_out = 1;
        } else {
            rc = radix_sort(L, SRC_PACKED, n, tail, K[0], V[0], K[1], V[1], n, plan, &in_out, &p1, nullptr, 0, 0, &ps);
        }
    } else if (coded) {
        rc = sort_by_codes(L, d_text, n, tail, h->pack_symbols ? 0u : 1u, list, counted, digits, &p1);
        in_out = 1; // idx[1] holds the list, key[0] and key[1] what the sort has left behind
    } else {
        if (!bytes_counted) {
            if (h->pack_symbols && (rc = move_table(bytehist, nullptr, 2 * RADIX_BINS * sizeof(u32), s)) != CSA_OK)
                return rc;
            count_bytes(false);
        }
        ps.text = d_text;
        ps.byte_wide = pp.byte_wide || !h->pack_symbols;
        hipLaunchKernelGGL(text_hist_expand_kernel, dim3(1), dim3(256), 0, s, d_text, n, (const u32*)bytehist, h->ghist);
        HIP_TRY(hipGetLastError());
        rc = radix_sort(L, SRC_TEXT, n, tail, K[0], V[0], K[1], V[1], n, make_plan(0, 64), &in_out, &p1, nullptr, 0, 0, &ps);
    }
    if (rc)
        return rc;
    passes += p1;
    if (in_out)
        cur = 1;
    u64* k_sorted = K[cur];
    u32* sa32 = V[cur]; // from here on the suffix array under construction
    // roles of the remaining arrays in generations t >= 1
    u32* ax = V[cur ^ 1];        // active list: suffixes ...
    u32* agid = h->gid;          // ... and their dense group ids
    u64* key_out = K[cur ^ 1];   // the active list sorted by (group, rank[x + h])
    u32* x_out = h->idx[2];
    u64* bkey[2] = {h->key[2], k_sorted}; // large groups on their way through the radix sort
    u32* bx[2] = {h->idx[3], h->idx[4]};  // (k_sorted is free once generation 0 has been ranked)

    RerankArgs ra;
    memset(&ra, 0, sizeof(ra));
    ra.keys = k_sorted;
    ra.sufs = sa32;
    ra.m = n;
    ra.n = n;
    ra.ell = ell;
    ra.rank = h->rank;
    ra.sufs_out = ax;
    ra.gids_out = agid;
    ra.gprim_out = h->gprim[0];
    ra.gstart_out = h->gstart[0];
    // scratch of the bucketed rank update: all free while (and after) a list is being ranked
    // (the records of generation 0 start in the third key array and swap with the sort's other output array; the sorted
    // keys themselves are still being read when the first records are written)
    auto defer_buffers = [&]() { // (by the roles the arrays have when it is asked for: a dense generation swaps two of them)
        return DeferBuffers{{bkey[0], key_out}, bx[0], bx[1], reinterpret_cast<u32*>(bkey[0]), reinterpret_cast<u32*>(bkey[1]),
                            reinterpret_cast<u32*>(bkey[1]) + h->cap};
    };
    u32 m = 0, groups = 0, big = 0;
    // packed keys: what the generations that the first sort covers would have left (contexts 4 W, 8 W, ... symbols)
    u32 level_counts[2 * MAX_LEVELS]; // (survivors, groups) of each
    if (pp.skipped > MAX_LEVELS)
        return fail(CSA_ERR_INTERNAL, "the first sort covers %u generations", pp.skipped);
    ra.levels = ra.first_level = pp.skipped - (narrow ? 1u : 0u); // (with narrow keys the last one is that of the first word)
    for (u32 i = 0; i < ra.levels; ++i) {
        ra.level_ell[i] = (u32)wide_ell << i;
        ra.level_drop[i] = (ell - ra.level_ell[i]) * pp.codes.bits;
    }
    ra.ties = ties_of(h);
    Settle settle;
    memset(&settle, 0, sizeof(settle));
    settle.text = d_text;
    settle.sa32 = sa32;
    settle.ctx = ell;
    settle.wide_ell = (u32)wide_ell;
    settle.stream = ps.stream;
    settle.sym_bits = ps.sym_bits;
    settle.word_bits = ps.stream ? 64u / ps.sym_bits * ps.sym_bits : 0u;
    WordList words;
    memset(&words, 0, sizeof(words));
    bool counted_firsts = false; // a list by words has been counted on the context it is ranked on
    u32 by_words_settled = 0; // generations of the reference that such a sort has left nothing of, and one
    if (by_words) {
        words.levels = word_levels(word_syms, word_bits, wide_ell);
        const WordLevels& lv = words.levels;
        const u32 all = lv.count - 1;
        auto next = [&](u64 c) { return c + (c < wide_ell ? (c < wide_ell - c ? c : wide_ell - c) : c); };
        auto settle_at = [&](u64 context, u32 tied, u32 in_groups, bool long_groups) -> int {
            settle.ctx = (u32)context;
            settle.words = long_groups;
            settle.next = 4;
            while (settle.next <= context)
                settle.next = next(settle.next);
            return settle_copies(L, settle, ra, tied, in_groups);
        };
        // A list with few ties on the first word has them counted and settled as they are, and so has one whose ties are copies, two or three to a
        // group: the second words would tell nothing of those apart. (Independent letters of 60 with a fifth of the text copied, 2.2 to a group, us with
        // the second words read / settled on the first, in tiles for short groups / in those for long ones: 2^18 symbols 333 / 312 / 327, 10^7 1137 / 900 /
        // 981, 5 * 10^7 4621 / 3585 / 3887. Written text from 2.67 to a group on, 2^18 letters: 327 / 530 / 373.)
        const RankTables r = rank_tables<RANK_TILE>(h, n);
        RerankArgs firsts = ra;
        firsts.ell = word_syms;
        firsts.levels = firsts.first_level = 0;
        for (u32 i = 0; i < lv.in_first; ++i) {
            firsts.level_ell[firsts.levels] = lv.context[i];
            firsts.level_drop[firsts.levels++] = lv.drop[i];
        }
        firsts.tile_agg = r.tile_agg;
        firsts.tile_prefix = r.tile_prefix;
        firsts.tile_splits = r.tile_splits;
        firsts.slab_total = r.slab_total;
        firsts.slab = r.slab;
        firsts.err = h->counts + 2;
        firsts.level_totals = reinterpret_cast<unsigned long long*>(h->ghist);
        unsigned long long* const h_levels = reinterpret_cast<unsigned long long*>(h->h_pinned + PINNED_HIST + 512);
        hipLaunchKernelGGL(choose_seconds_kernel, dim3(ENDLESS_BLOCKS), dim3(WORD_PLACES), 0, s, (const u64*)k_sorted, (const u32*)sa32, n, word_syms,
                           n < CSA_WORD_ENDLESS_MIN ? SECONDS_LEFT_OUT : SECONDS_ONLY, h->counts + 6, firsts.level_totals);
        firsts.choice = h->counts + 6;
        hipLaunchKernelGGL((rerank_count_kernel<RANK_BLOCK, RANK_ITEMS>), dim3(r.tiles), dim3(RANK_BLOCK), 0, s, firsts);
        TableGroup beside = {};
        add_table(beside, h_levels, firsts.level_totals, LEVEL_SLOTS * 8 * sizeof(unsigned long long));
        u32 tied = 0, in_groups = 0;
        int update = 0;
        if ((rc = rank_totals(L, r, true, n, n, false, &tied, &in_groups, &update, beside)) != CSA_OK)
            return rc;
        const u32 choice = h->h_pinned[6];
        u32 known = lv.in_first; // levels whose lists are known
        for (u32 i = 0; i < known; ++i) {
            u64 sv = 0, hd = 0;
            for (u32 slot = 0; slot < LEVEL_SLOTS; ++slot) {
                sv += h_levels[slot * 8 + 2 * i];
                hd += h_levels[slot * 8 + 2 * i + 1];
            }
            words.survivors[i] = (u32)sv;
            words.groups[i] = (u32)hd;
        }
        const bool few_ties = tied < n / 8, copies = 2 * (u64)tied <= 5 * (u64)in_groups;
        if (choice == SECONDS_AND_SETTLE && tied > 0 && (few_ties ? (u64)tied <= (u64)in_groups * SETTLE_AVG_LIMIT : copies)) {
            firsts.rank = nullptr;
            hipLaunchKernelGGL((rerank_kernel<RANK_BLOCK, RANK_ITEMS, false>), dim3(r.tiles), dim3(RANK_BLOCK), 0, s, firsts);
            HIP_TRY(hipGetLastError());
            if ((rc = settle_at(word_syms, tied, in_groups, few_ties)) != CSA_OK)
                return rc;
        }
        const bool seconds = choice == SECONDS_ONLY || (choice == SECONDS_AND_SETTLE && tied > 0 && !settle.settled);
        bool whole = false;
        if (seconds) {
            u8* const ties = reinterpret_cast<u8*>(K[cur ^ 1]);
            if ((rc = sort_by_words(L, n, ps, word_syms, k_sorted, sa32, ax, ties, ra, words)) != CSA_OK)
                return rc;
            std::swap(sa32, ax);
            std::swap(k_sorted, key_out);
            bkey[1] = k_sorted;
            settle.sa32 = sa32;
            ra.keys = k_sorted;
            ra.sufs_out = ax;
            passes += words.passes;
            whole = words.valid == lv.count;
            known = lv.count;
            tied = words.survivors[all];
            in_groups = words.groups[all];
            if (whole && choice == SECONDS_AND_SETTLE && tied > 0 && (u64)tied <= (u64)in_groups * SETTLE_AVG_LIMIT) {
                RerankArgs active = ra;
                active.rank = nullptr;
                hipLaunchKernelGGL((compact_ties_kernel<RANK_TILE>), dim3((r.tiles + 3) / 4), dim3(256), 0, s, active, r.tiles);
                HIP_TRY(hipGetLastError());
                if ((rc = settle_at(lv.context[all], tied, in_groups, true)) != CSA_OK)
                    return rc;
            }
        }
        if (choice != SECONDS_LEFT_OUT && (settle.settled || (tied == 0 && (whole || known == lv.in_first)))) {
            // the lists of all generations are known: those of the contexts inside the words, and those that were settled
            u32 gens = 1;
            auto report = [&](u64 active, u64 groups_of) {
                if (active == 0 || gens >= (u32)CSA_MAX_GENERATIONS)
                    return;
                st->active[gens] = active;
                st->groups[gens++] = groups_of;
            };
            for (u32 i = 0; i < known; ++i) {
                u64 c = 4;
                while (c < lv.context[i])
                    c = next(c);
                if (c == lv.context[i] && c >= wide_ell)
                    report(words.survivors[i], words.groups[i]);
            }
            for (u32 i = 0; settle.settled && i < settle.num; ++i)
                report(settle.active[i], settle.groups[i]);
            by_words_settled = gens;
        } else {
            // the doubling goes on from the last of its contexts that the list is resolved on, by the ties or by the first words
            u32 at = whole ? lv.count : lv.in_first;
            u64 c = 4;
            for (; at > 0; --at) {
                for (c = 4; c < lv.context[at - 1]; c = next(c)) {}
                if (c == lv.context[at - 1])
                    break;
            }
            if (at == 0)
                return fail(CSA_ERR_INTERNAL, "a list of words has no context of the doubling");
            ell = (u32)c;
            if (seconds) {
                memset(&list, 0, sizeof(list));
                list.words = at;
                list.told = list.by_levels = true;
                ra.words = at;
                coded = true;
            } else { // (counted on that context)
                ra.ell = ell;
                ra.drop = lv.drop[at - 1];
                m = tied;
                groups = in_groups;
                st->rank_update[0] = update;
                counted_firsts = true;
            }
            ra.levels = ra.first_level = 0;
            folded = 0;
            for (u64 f = ell; f < wide_ell; f = next(f))
                ++folded;
            pp.skipped = 0;
            for (u32 i = 0; i + 1 < at; ++i) // (counted with it)
                if (lv.context[i] >= wide_ell) {
                    level_counts[2 * pp.skipped] = words.survivors[i];
                    level_counts[2 * pp.skipped + 1] = words.groups[i];
                    ++pp.skipped;
                }
            settle.settled = false;
        }
    }
    if (by_words_settled == 0) // (a list of words has had its shorter contexts counted)
        rc = rerank_step(L, ra, defer_buffers(), &m, &groups, &st->rank_update[0], by_words ? nullptr : level_counts, coded ? &list : nullptr, &passes,
                         h->pack_symbols && h->settle && !by_words ? &settle : nullptr, counted_firsts);
    range_gen0.close();
    if (rc)
        return rc;
    bool ordinals_in_rank = ra.ordinals != 0; // rank[] holds run ordinals instead of ranks: the coming generation is dense
    st->passes[0] = passes;
    st->active[0] = n;
    st->groups[0] = 0;

    // ---- generations t >= 1 (reference loop: src/GPU_SACA.cu:1999-2103) ----
    int gen = 1;
    if (by_words) { // (its list says how far it goes, whatever the words)
        coded = false;
        if (by_words_settled) {
            gen = (int)by_words_settled;
            settle.settled = false;
            pp.skipped = 0;
            folded = 0;
        }
    }
    const u32 resolved = coded ? ell * list.words : ell;                            // symbols the first sort has resolved
    const u32 skipped = narrow ? pp.skipped + list.words - 2u : pp.skipped; // generations after the first that it stands for
    u64 ctx = resolved; // symbols resolved so far; the next generation looks hop symbols ahead
    // A list that was resolved on two words leaves what generation 1 would: that one is reported with the lists it would have had, what
    // the members of its large groups took, and no time of its own.
    if (coded && !narrow && list.words == 2) {
        if (level_counts[0] > 0) {
            st->active[1] = level_counts[0];
            st->groups[1] = level_counts[1];
            st->big[1] = list.long_members;
            st->passes[1] = list.long_passes;
            gen = 2;
        }
    } else if (coded) {
        st->passes[0] += list.long_passes;
    }
    // Nor do the generations of a list whose ties have been settled.
    if (settle.settled) {
        if (gen + settle.num > CSA_MAX_GENERATIONS)
            return fail(CSA_ERR_INTERNAL, "%u generations do not fit the statistics", gen + settle.num);
        for (u32 i = 0; i < settle.num; ++i, ++gen) {
            st->active[gen] = settle.active[i];
            st->groups[gen] = settle.groups[i];
        }
        m = 0;
    }
    const int untimed = gen - 1; // generations 1 .. untimed
    HIP_TRY(hipEventRecord(h->ev_gen[gen], s));
    int gp = 0; // gprim[gp] / gstart[gp] describe the current groups
    bool all_small = false; // no group of the current list exceeds the limit of the generation that found it so
    bool presorted_before = false; // every large group of the generation before was in order as it stood
    int chained = 0;               // the generation from which on the list was settled by settle_chains: the time is all that one's
    u32 chain_tries = 0;           // attempts at settle_chains that came to nothing
    bool high_limit = false; // that generation's limit was SMALL_MAXG_HI (groups only split: the limit stays from there on)
    const int sec_bits = bit_length(n > 1 ? n - 1 : 1);
    while (m > 0) {
        if (gen >= CSA_MAX_GENERATIONS)
            return fail(CSA_ERR_INTERNAL, "generation cap reached with %u suffixes still active", m);
        st->active[gen] = m;
        st->groups[gen] = groups;
        const u32 m_in = m;
        RangeScope range_g("generation %d m=%u groups=%u", gen, m, groups);
        const u64 hop = ctx < wide_ell ? (ctx < wide_ell - ctx ? ctx : wide_ell - ctx) : ctx;
        // A dense generation: most of the partition is still active and its groups are long (a small alphabet, a
        // periodic text), so nearly every member would go through the radix sort anyway. Then the whole partition is sorted
        // again, as in generation 0, by keys that are read in text order: (rank[x], rank[x + hop]) for x = 0, 1, ...,
        // two coalesced streams instead of one random gather per member; the ranks come out of the same run ranking as
        // in generation 0 and go back to rank[] through the bucketed update instead of scattered writes. Suffixes that had
        // retired are alone with their rank: they sort to the place they hold already and keep their rank.
        const bool dense = dense_generation(m_in, groups, n);
        if (dense) {
            // A generation that runs in this form itself, or generation 0, knew that this one would be dense (the same test on
            // the same numbers) and left ordinals in rank[]: the key runs of its sorted list numbered 0, 1, 2, ...; there
            // are as many as it had groups and singletons. Two ordinals make a key of 2 log2(runs) bits: 17 bits after
            // generation 0 of a four-letter text (256 groups and the last four suffixes), three passes where two 31-bit ranks
            // take eight. A generation of the other form leaves ranks, and the list it leaves can still qualify (its many
            // short groups dissolved, a few long ones are left): the key is then the two ranks side by side.
            passes = 0;
            if (ordinals_in_rank) {
                const u64 runs = (u64)groups + ((u64)n - m_in);
                const u32 radix = (u32)runs;
                const PassPlan plan = make_plan(0, runs > 1 ? bit_length(runs * runs - 1) : 1);
                rc = radix_sort(L, SRC_RANKS, n, 0, bkey[0], bx[0], bkey[1], bx[1], n, plan, &in_out, &passes, h->rank,
                                (u32)hop, radix);
            } else {
                PassPlan plan; // the digits of the two ranks of a key: bits [0, sec_bits) and [32, 32 + sec_bits)
                plan.num_passes = 0;
                for (int half = 0; half < 2; ++half)
                    for (int b = 0; b < sec_bits; b += RADIX_BITS) {
                        plan.shift[plan.num_passes] = 32 * half + b;
                        plan.bits[plan.num_passes] = sec_bits - b < RADIX_BITS ? sec_bits - b : RADIX_BITS;
                        plan.num_passes++;
                    }
                rc = radix_sort(L, SRC_RANKS, n, 0, bkey[0], bx[0], bkey[1], bx[1], n, plan, &in_out, &passes, h->rank,
                                (u32)hop, 0u);
            }
            if (rc)
                return rc;
            RerankArgs rd;
            memset(&rd, 0, sizeof(rd));
            rd.keys = bkey[in_out];
            rd.sufs = bx[in_out];
            rd.m = n;
            rd.n = n;
            rd.ell = 0; // no suffix is set apart for running off the text: the tied ones never do, the others are alone anyway
            rd.rank = h->rank;
            rd.sufs_out = ax;
            rd.gids_out = agid;
            rd.gprim_out = h->gprim[gp ^ 1];
            rd.gstart_out = h->gstart[gp ^ 1];
            DeferBuffers db = defer_buffers();
            db.recs[0] = bkey[in_out ^ 1]; // the records of the rank update: the two 8-byte arrays that do not hold the sorted keys
            db.recs[1] = key_out;
            rc = rerank_step(L, rd, db, &m, &groups, &st->rank_update[gen]);
            if (rc)
                return rc;
            ordinals_in_rank = rd.ordinals != 0;
            // the freshly sorted index array is the suffix array under construction from here on; the old one is scratch
            u32* const old_sa32 = sa32;
            sa32 = bx[in_out];
            bx[in_out] = old_sa32;
            big = m_in;
            st->big[gen] = m_in;
            st->passes[gen] = passes;
            st->dense[gen] = 1;
            all_small = false;
            presorted_before = false;
            gp ^= 1;
            HIP_TRY(hipEventRecord(h->ev_gen[gen + 1], s));
            gen++;
            ctx += hop;
            continue;
        }
        // Every member of the list before was one of a long group in order: runs and periods, as a rule.
        if (h->pack_symbols && h->settle && !ordinals_in_rank && gen > untimed + 1 && st->presorted[gen - 1] == st->active[gen - 1] &&
            chain_tries < CHAIN_TRIES) {
            Chains ch;
            rc = settle_chains(L, ch, d_text, n, ctx, wide_ell, ax, agid, h->gstart[gp], h->gprim[gp], m_in, groups, h->gprim[gp ^ 1], sa32);
            if (rc)
                return rc;
            if (ch.settled) {
                if (gen + ch.num > CSA_MAX_GENERATIONS)
                    return fail(CSA_ERR_INTERNAL, "%u generations do not fit the statistics", gen + ch.num);
                for (u32 i = 0; i < ch.num; ++i) {
                    st->active[gen + i] = ch.active[i];
                    st->groups[gen + i] = ch.groups[i];
                    st->big[gen + i] = st->presorted[gen + i] = ch.big[i];
                    st->small_only[gen + i] = ch.small_only[i];
                }
                chained = gen;
                gen += (int)ch.num;
                HIP_TRY(hipEventRecord(h->ev_gen[gen], s));
                break;
            }
            ++chain_tries;
        }
        if (ordinals_in_rank)
            return fail(CSA_ERR_INTERNAL, "generation %d reads ranks but the one before it left ordinals", gen);
        const RankTables r = rank_tables<SMALL_TILE>(h, m_in);
        u32* nr_list = reinterpret_cast<u32*>(key_out); // refined rank at every place of the sorted list
        // 1. gather rank[x + h]; small groups are sorted and ranked inside their tile, members of large groups set aside
        SmallSortArgs sa;
        memset(&sa, 0, sizeof(sa));
        sa.sufs = ax;
        sa.gids = agid;
        sa.gstart = h->gstart[gp];
        sa.gprim = h->gprim[gp];
        sa.rank = h->rank;
        sa.m = m_in;
        sa.n = n;
        sa.h = (u32)hop;
        sa.sec_bits = sec_bits;
        sa.groups = groups;
        sa.err = h->counts + 2;
        sa.sufs_out = x_out;
        sa.nr_out = nr_list;
        sa.big_keys = bkey[0];
        sa.big_sufs = bx[0];
        sa.big_first = reinterpret_cast<const u32*>(bkey[1]); // (free until the radix sort, which starts after the kernel that reads it)
        sa.tile_agg = r.tile_agg;
        sa.tile_splits = r.tile_splits;
        passes = 0;
        if (all_small) {
            // Groups only ever split: once a generation had no large group, none can appear again. The small-group
            // kernel then also counts for the apply step, and nothing else runs before it.
            TableGroup cleared = {};
            add_table(cleared, r.tile_agg, nullptr, (u64)r.tiles * 4 * sizeof(u32));
            add_table(cleared, r.tile_splits, nullptr, (u64)r.tiles * sizeof(u32));
            if ((rc = move_tables(cleared, s)) != CSA_OK)
                return rc;
            if (high_limit)
                hipLaunchKernelGGL((smallsort_kernel<SMALL_BLOCK, SMALL_ITEMS, SMALL_MAXG_HI, true>), dim3(r.tiles), dim3(SMALL_BLOCK), 0,
                                   s, sa);
            else
                hipLaunchKernelGGL((smallsort_kernel<SMALL_BLOCK, SMALL_ITEMS, SMALL_MAXG, true>), dim3(r.tiles), dim3(SMALL_BLOCK), 0, s,
                                   sa);
            HIP_TRY(hipGetLastError());
            st->small_only[gen] = 1;
        } else {
            // marks of the large groups whose gathered ranks are out of order, in the tables the next generation's groups
            // will be written to (free until the apply step)
            sa.big_sec = bx[1];
            sa.not_asc = h->gprim[gp ^ 1];
            sa.not_desc = h->gstart[gp ^ 1];
            high_limit = (u64)m_in <= (u64)groups * SMALL_AVG_LIMIT;
            const u32 maxg = high_limit ? (u32)SMALL_MAXG_HI : (u32)SMALL_MAXG;
            const u32 marks = m_in / maxg + 2u; // one mark index per large group at most
            TableGroup cleared = {};
            add_table(cleared, h->counts + 4, nullptr, 2 * sizeof(u32));
            add_table(cleared, sa.not_asc, nullptr, (u64)marks * sizeof(u32));
            add_table(cleared, sa.not_desc, nullptr, (u64)marks * sizeof(u32));
            if ((rc = move_tables(cleared, s)) != CSA_OK)
                return rc;
            {
                // where every large group's members start in the list of large-group members, and how many there are
                // (counts[4]): a prefix sum over the group table
                u32* big_first = reinterpret_cast<u32*>(bkey[1]);
                const RankTables gr = rank_tables<1024>(h, groups);
                hipLaunchKernelGGL((big_prefix_kernel<false>), dim3(gr.tiles), dim3(256), 0, s, (const u32*)h->gstart[gp], groups, maxg, big_first,
                                   gr.tile_agg, gr.tile_splits, (const u32*)gr.tile_prefix, (const u32*)gr.slab_total, gr.slab, gr.slabs,
                                   h->counts + 4);
                hipLaunchKernelGGL(rerank_scan_kernel, dim3(gr.slabs), dim3(1024), 0, s, gr.tile_agg, gr.tile_prefix, gr.tiles, gr.slab,
                                   gr.slab_total, gr.tile_splits);
                hipLaunchKernelGGL((big_prefix_kernel<true>), dim3(gr.tiles), dim3(256), 0, s, (const u32*)h->gstart[gp], groups, maxg, big_first,
                                   gr.tile_agg, gr.tile_splits, (const u32*)gr.tile_prefix, (const u32*)gr.slab_total, gr.slab, gr.slabs,
                                   h->counts + 4);
            }
            auto gather_and_sort_small = [&]() {
                if (high_limit)
                    hipLaunchKernelGGL((smallsort_kernel<SMALL_BLOCK, SMALL_ITEMS, SMALL_MAXG_HI, false>), dim3(r.tiles), dim3(SMALL_BLOCK),
                                       0, s, sa);
                else
                    hipLaunchKernelGGL((smallsort_kernel<SMALL_BLOCK, SMALL_ITEMS, SMALL_MAXG, false>), dim3(r.tiles), dim3(SMALL_BLOCK), 0,
                                       s, sa);
            };
            // A list whose large groups were all in order in the generation before (a run, a period: they stay so until
            // they dissolve) is expected to be so again: the (key, suffix) pairs for the radix sort, 12 of the 16 bytes the
            // kernel writes per member of a large group, are then left out, and the kernel runs once more with them in
            // the rare generation in which the marks say otherwise.
            sa.side_list = (presorted_before || h->expect_presorted) ? 0u : 1u;
            gather_and_sort_small();
            hipLaunchKernelGGL(group_order_kernel, dim3((marks + 255u) / 256u), dim3(256), 0, s, (const u32*)sa.not_asc, (const u32*)sa.not_desc,
                               marks, h->counts + 5);
            HIP_TRY(hipGetLastError());
            rc = read_counts(L, &big);
            if (rc)
                return rc;
            all_small = big == 0;
            const u32 unordered = h->h_pinned[5];
            if (big > 0 && unordered != 0 && !sa.side_list) {
                sa.side_list = 1u;
                gather_and_sort_small();
                HIP_TRY(hipGetLastError());
            }
            presorted_before = big > 0 && unordered == 0;
            if (big > 0 && unordered == 0) {
                // 2a. every large group is in order as it stands (runs of one token, periodic stretches: the gathered ranks
                //     rise or fall along the list): no sort, the members are ranked by their runs of equal gathered ranks
                PresortedArgs pa;
                pa.sufs = ax;
                pa.gids = agid;
                pa.big_sec = sa.big_sec;
                pa.gstart = h->gstart[gp];
                pa.gprim = h->gprim[gp];
                pa.big_first = sa.big_first;
                pa.not_asc = sa.not_asc;
                pa.m = m_in;
                pa.n = n;
                pa.groups = groups;
                pa.maxg = maxg;
                pa.sufs_out = x_out;
                pa.nr_out = nr_list;
                pa.err = h->counts + 2;
                // (512 x 4 tiles: 0.8 ms per sort of the adversarial workload ahead of 256 x 4; 8 elements per thread: 8 ms behind)
                constexpr int PRESORTED_BLOCK = 512, PRESORTED_ITEMS = 4;
                const RankTables pr = rank_tables<PRESORTED_BLOCK * PRESORTED_ITEMS>(h, m_in);
                pa.tile_agg = pr.tile_agg;
                pa.tile_splits = pr.tile_splits;
                pa.tile_prefix = pr.tile_prefix;
                pa.slab_total = pr.slab_total;
                pa.slab = pr.slab;
                hipLaunchKernelGGL((place_presorted_kernel<PRESORTED_BLOCK, PRESORTED_ITEMS, false>), dim3(pr.tiles), dim3(PRESORTED_BLOCK), 0, s, pa);
                hipLaunchKernelGGL(rerank_scan_kernel, dim3(pr.slabs), dim3(1024), 0, s, pr.tile_agg, pr.tile_prefix, pr.tiles, pr.slab,
                                   pr.slab_total, pr.tile_splits);
                hipLaunchKernelGGL((place_presorted_kernel<PRESORTED_BLOCK, PRESORTED_ITEMS, true>), dim3(pr.tiles), dim3(PRESORTED_BLOCK), 0, s, pa);
                HIP_TRY(hipGetLastError());
                st->presorted[gen] = big;
            }
            // 2. the large groups: radix sort on (group id, rank[x + h]), then back into the list as (suffix, refined rank)
            if (big > 0 && unordered != 0) {
                const int gid_bits = bit_length(groups > 1 ? groups - 1 : 0);
                const PassPlan plan = make_plan(0, sec_bits + gid_bits);
                rc = radix_sort(L, SRC_PAIRS, n, 0, bkey[0], bx[0], bkey[1], bx[1], big, plan, &in_out, &passes);
                if (rc)
                    return rc;
                PlaceArgs pa;
                pa.big_keys = bkey[in_out];
                pa.big_sufs = bx[in_out];
                pa.mb = big;
                pa.m = m_in;
                pa.n = n;
                pa.groups = groups;
                pa.sec_bits = sec_bits;
                pa.gstart = h->gstart[gp];
                pa.gprim = h->gprim[gp];
                pa.sufs_out = x_out;
                pa.nr_out = nr_list;
                pa.err = h->counts + 2;
                // (the tile tables are free between the small-group kernel and the counting pass below)
                const RankTables pr = rank_tables<RANK_TILE>(h, big);
                pa.tile_agg = pr.tile_agg;
                pa.tile_splits = pr.tile_splits;
                pa.tile_prefix = pr.tile_prefix;
                pa.slab_total = pr.slab_total;
                pa.slab = pr.slab;
                hipLaunchKernelGGL((place_big_kernel<RANK_BLOCK, RANK_ITEMS, false>), dim3(pr.tiles), dim3(RANK_BLOCK), 0, s, pa);
                hipLaunchKernelGGL(rerank_scan_kernel, dim3(pr.slabs), dim3(1024), 0, s, pr.tile_agg, pr.tile_prefix, pr.tiles, pr.slab,
                                   pr.slab_total, pr.tile_splits);
                hipLaunchKernelGGL((place_big_kernel<RANK_BLOCK, RANK_ITEMS, true>), dim3(pr.tiles), dim3(RANK_BLOCK), 0, s, pa);
                HIP_TRY(hipGetLastError());
            }
            // 3. per-tile counts of the sorted list (8 bytes read per member)
            hipLaunchKernelGGL((count_ranks_kernel<SMALL_BLOCK, SMALL_ITEMS>), dim3(r.tiles), dim3(SMALL_BLOCK), 0, s, nr_list, x_out, m_in,
                               run_reach(n), r.tile_agg, r.tile_splits);
            HIP_TRY(hipGetLastError());
        }
        st->big[gen] = big;
        // 4. scan, totals to the host, apply: retire singletons, compact survivors, write the changed ranks
        rc = rank_totals(L, r, false, m_in, n, all_small && big == 0, &m, &groups, &st->rank_update[gen]);
        if (rc)
            return rc;
        ApplySmallArgs aa;
        aa.sufs = x_out;
        aa.nr = nr_list;
        aa.m = m_in;
        aa.n = n;
        aa.rank = h->rank;
        const DeferBuffers defer_buf = defer_buffers();
        aa.rank_vals = st->rank_update[gen] == 2 ? defer_buf.vals : nullptr;
        aa.sa32 = sa32;
        aa.sufs_out = ax;
        aa.gids_out = agid;
        aa.gprim_out = h->gprim[gp ^ 1];
        aa.gstart_out = h->gstart[gp ^ 1];
        aa.tile_prefix = r.tile_prefix;
        aa.slab_total = r.slab_total;
        aa.slab = r.slab;
        aa.err = h->counts + 2;
        hipLaunchKernelGGL((apply_small_kernel<SMALL_BLOCK, SMALL_ITEMS>), dim3(r.tiles), dim3(SMALL_BLOCK), 0, s, aa);
        HIP_TRY(hipGetLastError());
        if (st->rank_update[gen] == 2) {
            rc = windowed_rank_update(L, x_out, defer_buf, m_in, n);
            if (rc)
                return rc;
        }
        gp ^= 1;
        st->passes[gen] = passes;
        HIP_TRY(hipEventRecord(h->ev_gen[gen + 1], s));
        gen++;
        ctx += hop;
    }
    st->generations = gen;

    // ---- output: 5-byte little-endian entries in rank order ----
    const int aligned4 = ((uintptr_t)d_sa40 & 3u) == 0;
    const u64 quads = ((u64)n + 3) / 4;
    hipLaunchKernelGGL(emit_sa40_kernel, dim3((u32)((quads + 255) / 256)), dim3(256), 0, s, sa32, n, index_base, d_sa40,
                       aligned4);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipEventRecord(h->ev_gen[gen + 1], s));
    rc = read_counts(L, nullptr); // waits for the stream; the last apply pass may still have raised the error word
    if (rc)
        return rc;

    for (int g = 0; g < gen; ++g) {
        if ((g >= 1 && g <= untimed) || (chained && g > chained))
            continue;
        HIP_TRY(hipEventElapsedTime(&st->ms[g], h->ev_gen[g], h->ev_gen[g == 0 ? untimed + 1 : chained && g == chained ? gen : g + 1]));
    }
    HIP_TRY(hipEventElapsedTime(&st->ms_output, h->ev_gen[gen], h->ev_gen[gen + 1]));
    HIP_TRY(hipEventElapsedTime(&st->ms_total, h->ev_gen[0], h->ev_gen[gen + 1]));
    for (auto& tl : L.timed) {
        float ms = 0;
        HIP_TRY(hipEventElapsedTime(&ms, h->events[tl.first], h->events[tl.first + 1]));
        st->radix_ms += ms;
        st->radix_pairs += tl.second;
        st->radix_launches++;
    }
    // wide keys: the first generations that ran stand for generation 0
    const int merged = folded < gen - 1 ? folded : gen - 1;
    if (merged > 0) {
        for (int g = 1; g <= merged; ++g) {
            st->ms[0] += st->ms[g];
            st->passes[0] += st->passes[g];
        }
        for (int g = 1; g + merged < gen; ++g) {
            st->active[g] = st->active[g + merged];
            st->groups[g] = st->groups[g + merged];
            st->big[g] = st->big[g + merged];
            st->presorted[g] = st->presorted[g + merged];
            st->passes[g] = st->passes[g + merged];
            st->rank_update[g] = st->rank_update[g + merged];
            st->small_only[g] = st->small_only[g + merged];
            st->dense[g] = st->dense[g + merged];
            st->ms[g] = st->ms[g + merged];
        }
        for (int g = gen - merged; g < gen; ++g) {
            st->active[g] = st->groups[g] = st->big[g] = st->presorted[g] = 0;
            st->passes[g] = st->rank_update[g] = st->small_only[g] = st->dense[g] = 0;
            st->ms[g] = 0.0f;
        }
        st->generations = gen - merged;
    }
    // packed keys: the first sort stands for generations 0 .. skipped of the reference; those after the first are reported
    // with the lists they would have had and no time or passes of their own
    st->key_symbols = by_words ? (as_reported.enabled ? as_reported.codes.key_syms : 4u) : pp.enabled ? resolved : ell;
    st->first_sort_generations = 1 + (int)(by_words ? as_reported.skipped : skipped);
    if (skipped > 0) {
        const int sk = (int)skipped;
        if (gen + sk > CSA_MAX_GENERATIONS)
            return fail(CSA_ERR_INTERNAL, "%d generations do not fit the statistics", gen + sk);
        for (int g = gen - 1; g >= 1; --g) {
            st->active[g + sk] = st->active[g];
            st->groups[g + sk] = st->groups[g];
            st->big[g + sk] = st->big[g];
            st->presorted[g + sk] = st->presorted[g];
            st->passes[g + sk] = st->passes[g];
            st->rank_update[g + sk] = st->rank_update[g];
            st->small_only[g + sk] = st->small_only[g];
            st->dense[g + sk] = st->dense[g];
            st->ms[g + sk] = st->ms[g];
        }
        for (int g = 1; g <= sk; ++g) {
            st->active[g] = level_counts[2 * (g - 1)];
            st->groups[g] = level_counts[2 * (g - 1) + 1];
            st->big[g] = st->presorted[g] = 0;
            st->passes[g] = st->rank_update[g] = st->small_only[g] = st->dense[g] = 0;
            st->ms[g] = 0.0f;
        }
        st->generations = gen + sk;
        // the reference stops at the first generation that leaves nothing active
        for (int g = 1; g <= sk; ++g)
            if (st->active[g] == 0) {
                st->generations = g;
                break;
            }
    }
    return CSA_OK;
}

} // namespace

extern "C" {

uint32_t csa_partition_id_bits(uint32_t p)
{
    const int id_bits = p <= 1 ? 0 : bit_length((u64)p - 1);
    return (u32)(id_bits < 1 ? 1 : id_bits) + 1u;
}

int csa_partition_ids_u16_dev(const uint16_t* d_text, uint64_t n, uint64_t text_len, const uint64_t* d_pivots,
                              int pivot_words, uint32_t p, uint16_t* d_pid, uint64_t* d_packed, uint64_t* d_psz,
                              void* stream)
{
    if (p < 1 || p > 65536u)
        return fail(CSA_ERR_ARG, "csa_partition_ids_u16_dev: p = %u is outside [1, 65536]", p);
    if (pivot_words < 1 || pivot_words > 4)
        return fail(CSA_ERR_ARG, "csa_partition_ids_u16_dev: pivot_words = %d is outside [1, 4]", pivot_words);
    if (n == 0)
        return CSA_OK;
    if (!d_text || (p > 1 && !d_pivots) || text_len < n)
        return fail(CSA_ERR_ARG, "csa_partition_ids_u16_dev: null text or pivots, or text_len < n");
    const u64 tiles64 = (n + PID_TILE - 1) / PID_TILE;
    if (tiles64 > 0xFFFFFFFFull)
        return fail(CSA_ERR_TOO_LARGE, "csa_partition_ids_u16_dev: %llu suffixes in one call", (unsigned long long)n);
    PartitionIdArgs a;
    a.text = d_text;
    a.n = n;
    a.text_len = text_len;
    a.pivots = d_pivots;
    a.p = p;
    a.bits = csa_partition_id_bits(p);
    a.pid = d_pid;
    a.packed = d_packed;
    a.psz = reinterpret_cast<unsigned long long*>(d_psz);
    a.tiles = (u32)tiles64;
    const u32 grid = a.tiles < 8192u ? a.tiles : 8192u;
    hipStream_t s = (hipStream_t)stream;
    // (the table in LDS is filled up to 2^bits(p - 1) - 1 entries)
    const bool piv_lds = (((u64)1 << bit_length((u64)(p - 1))) - 1) * (u64)pivot_words <= PID_LDS_PIVOT_WORDS;
    const u32 lds = partition_ids_lds_bytes(pivot_words, p, piv_lds, d_psz != nullptr, d_packed != nullptr, a.bits, &a.hist_copies_log2);
#define CSA_LAUNCH_PID(W)                                                                                  \
    do {                                                                                                   \
        if (piv_lds)                                                                                       \
            hipLaunchKernelGGL((partition_ids_kernel<W, true>), dim3(grid), dim3(PID_BLOCK), lds, s, a);  \
        else                                                                                               \
            hipLaunchKernelGGL((partition_ids_kernel<W, false>), dim3(grid), dim3(PID_BLOCK), lds, s, a); \
    } while (0)
    switch (pivot_words) {
    case 1: CSA_LAUNCH_PID(1); break;
    case 2: CSA_LAUNCH_PID(2); break;
    case 3: CSA_LAUNCH_PID(3); break;
    default: CSA_LAUNCH_PID(4); break;
    }
#undef CSA_LAUNCH_PID
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

namespace {
int fill_message_args(MessageArgs& a, const char* who, const uint64_t* d_sa, const uint64_t* d_keys, const uint32_t* d_beta,
                      uint64_t n, uint64_t ctx, int packed_keys, uint32_t p)
{
    if (p < 1 || p > 32768u)
        return fail(CSA_ERR_ARG, "%s: p = %u is outside [1, 32768]", who, p);
    if (n > CSA_MAX_PART_SZ)
        return fail(CSA_ERR_TOO_LARGE, "%s: %llu suffixes exceed a partition", who, (unsigned long long)n);
    if (n && (!d_sa || !d_keys || !d_beta))
        return fail(CSA_ERR_ARG, "%s: null buffer", who);
    a.sa = d_sa;
    a.keys = d_keys;
    a.beta = d_beta;
    a.n = n;
    a.ctx = ctx;
    a.packed = packed_keys ? 1 : 0;
    a.active_sz = nullptr;
    a.p = p;
    a.msg_target = nullptr;
    a.msg_rank = nullptr;
    a.msg_off = nullptr;
    a.tiles = (u32)((n + MSG_TILE - 1) / MSG_TILE);
    return CSA_OK;
}
} // namespace

int csa_count_messages_dev(const uint64_t* d_sa, const uint64_t* d_keys, const uint32_t* d_beta, uint64_t n, uint64_t ctx,
                           int packed_keys, uint32_t p, uint32_t* d_msg_count, void* stream)
{
    MessageArgs a;
    const int rc = fill_message_args(a, "csa_count_messages_dev", d_sa, d_keys, d_beta, n, ctx, packed_keys, p);
    if (rc || n == 0)
        return rc;
    if (!d_msg_count)
        return fail(CSA_ERR_ARG, "csa_count_messages_dev: null counters");
    a.msg_off = d_msg_count;
    hipLaunchKernelGGL(count_messages_kernel, dim3(a.tiles < 4096u ? a.tiles : 4096u), dim3(MSG_BLOCK), 0, (hipStream_t)stream, a);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

int csa_message_offsets_dev(uint32_t* d_msg_off, uint32_t count, void* stream)
{
    if (count == 0)
        return CSA_OK;
    if (!d_msg_off || count > 32769u)
        return fail(CSA_ERR_ARG, "csa_message_offsets_dev: null counters or more than 32769 of them");
    hipLaunchKernelGGL(message_offsets_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, d_msg_off, count);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

int csa_emit_messages_dev(const uint64_t* d_sa, const uint64_t* d_keys, const uint32_t* d_beta, uint64_t n, uint64_t ctx,
                          int packed_keys, const uint64_t* d_active_sz, uint32_t p, uint8_t* d_msg_target,
                          uint32_t* d_msg_rank, uint32_t* d_msg_off, void* stream)
{
    MessageArgs a;
    const int rc = fill_message_args(a, "csa_emit_messages_dev", d_sa, d_keys, d_beta, n, ctx, packed_keys, p);
    if (rc || n == 0)
        return rc;
    if (!d_active_sz || !d_msg_target || !d_msg_rank || !d_msg_off)
        return fail(CSA_ERR_ARG, "csa_emit_messages_dev: null buffer");
    a.active_sz = reinterpret_cast<const unsigned long long*>(d_active_sz);
    a.msg_target = d_msg_target;
    a.msg_rank = d_msg_rank;
    a.msg_off = d_msg_off;
    const u64 emit_tiles = (n + EMIT_TILE - 1) / EMIT_TILE;
    if (a.p <= EMIT_FEW_PARTS)
        hipLaunchKernelGGL((emit_messages_kernel<EMIT_FEW_PARTS>), dim3((u32)(emit_tiles < 2048u ? emit_tiles : 2048u)), dim3(EMIT_BLOCK), 0, (hipStream_t)stream, a);
    else
        hipLaunchKernelGGL((emit_messages_kernel<MSG_LDS_PARTS>), dim3((u32)(emit_tiles < 2048u ? emit_tiles : 2048u)), dim3(EMIT_BLOCK), 0, (hipStream_t)stream, a);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

extern "C++" {
namespace {
// Builds the join directory of the suffix-ordered cohort d_sa[0, n) in `dir` (room for `room` entries) and returns the
// log2 of its bucket count through *dir_log2; leaves *dir_log2 = 0 and builds nothing when the cohort is small.
int build_join_directory(const u64* d_sa, u64 n, u32* dir, u64 room, hipStream_t s, u32* dir_log2, bool sorted_probes)
{
    *dir_log2 = 0;
    if (n < CSA_JOIN_DIR_MIN || room < 3)
        return CSA_OK;
    // Probes in arrival order: one to two cohort entries per bucket, so that a probe costs the directory's line and one
    // line of the cohort (with at most 2^22 buckets a cohort of 44 M suffixes had 10 per bucket and the join of 268 M
    // messages took 14.5 ms instead of 9.5). Probes sorted by target walk the cohort and the directory in order and find
    // their lines in cache: a coarse directory (two to four entries per bucket, at most 2^22 buckets) is built four
    // times faster and serves them as well.
    u32 lg = (u32)bit_length(n) - (sorted_probes ? 2u : 1u);
    const u32 cap = sorted_probes ? 22u : 26u;
    if (lg > cap)
        lg = cap;
    while (lg && (1ull << lg) + 1 > room)
        --lg;
    if (lg == 0)
        return CSA_OK;
    hipLaunchKernelGGL(join_directory_kernel, dim3((u32)(((1ull << lg) + 256) / 256)), dim3(256), 0, s, d_sa, n, lg, dir);
    HIP_TRY(hipGetLastError());
    *dir_log2 = lg;
    return CSA_OK;
}
} // namespace
} // extern "C++"

int csa_join_messages_dev(const uint8_t* d_msg_target, const uint32_t* d_msg_rank, uint32_t msg_c, const uint64_t* d_sa,
                          const uint32_t* d_primary, uint64_t* d_keys, uint64_t n, void* stream)
{
    if (msg_c == 0)
        return CSA_OK;
    if (!d_msg_target || !d_msg_rank || (n && (!d_sa || !d_primary || !d_keys)))
        return fail(CSA_ERR_ARG, "csa_join_messages_dev: null buffer");
    if (n > CSA_MAX_PART_SZ)
        return fail(CSA_ERR_TOO_LARGE, "csa_join_messages_dev: %llu suffixes exceed a partition", (unsigned long long)n);
    hipLaunchKernelGGL(join_messages_kernel, dim3((msg_c + 255u) / 256u), dim3(256), 0, (hipStream_t)stream, d_msg_target,
                       (const u64*)nullptr, d_msg_rank, msg_c, d_sa, d_primary, d_keys, n, (const u32*)nullptr, 0u);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

int csa_join_messages_sorted_dev(csa_handle* h, const uint8_t* d_msg_target, const uint32_t* d_msg_rank, uint32_t msg_c,
                                 const uint64_t* d_sa, const uint32_t* d_primary, uint64_t* d_keys, uint64_t n, void* stream)
{
    if (!h)
        return fail(CSA_ERR_ARG, "csa_join_messages_sorted_dev: null handle");
    if (msg_c == 0)
        return CSA_OK;
    if (!d_msg_target || !d_msg_rank || (n && (!d_sa || !d_primary || !d_keys)))
        return fail(CSA_ERR_ARG, "csa_join_messages_sorted_dev: null buffer");
    if (n > CSA_MAX_PART_SZ)
        return fail(CSA_ERR_TOO_LARGE, "csa_join_messages_sorted_dev: %llu suffixes exceed a partition", (unsigned long long)n);
    if (msg_c > h->cap)
        return fail(CSA_ERR_ARG, "csa_join_messages_sorted_dev: %u messages exceed the handle's capacity %llu", msg_c,
                    (unsigned long long)h->cap);
    Launch L;
    L.h = h;
    L.stream = (hipStream_t)stream;
    L.flags = 0;
    L.stats = nullptr;
    hipStream_t s = L.stream;
    HIP_TRY(hipMemsetAsync(h->counts, 0, 4 * sizeof(u32), s));
    // (target word, rank) pairs in columns of the handle's block, sorted on the 40 target bits
    h->pool.reset();
    u64* K[2];
    u32* V[2];
    for (int i = 0; i < 2; ++i) {
        K[i] = static_cast<u64*>(h->pool.take((u64)msg_c * sizeof(u64)));
        V[i] = static_cast<u32*>(h->pool.take((u64)msg_c * sizeof(u32)));
    }
    if (!K[0] || !V[0] || !K[1] || !V[1])
        return fail(CSA_ERR_ARG, "csa_join_messages_sorted_dev: the handle's block of %llu bytes has no room for 24 bytes per message",
                    (unsigned long long)h->pool.bytes());
    // the directory over the cohort takes what is left, up to an entry per cohort member (a smaller one has longer buckets)
    u64 dir_room = n < 3 ? 3 : n;
    u32* dir = nullptr;
    while (dir_room >= 3 && !(dir = static_cast<u32*>(h->pool.take(dir_room * sizeof(u32)))))
        dir_room /= 2;
    if (!dir)
        dir_room = 0;
    h->last_high_water = h->pool.high_water();
    hipLaunchKernelGGL(unpack_lanes_kernel, dim3((msg_c + 255u) / 256u), dim3(256), 0, s, d_msg_target, (u64)msg_c, K[0]);
    HIP_TRY(hipMemcpyAsync(V[0], d_msg_rank, (u64)msg_c * sizeof(u32), hipMemcpyDeviceToDevice, s));
    int in_out = 0, passes = 0;
    const PassPlan plan = make_plan(0, 40);
    int rc = radix_sort(L, SRC_PAIRS, 0, 0, K[0], V[0], K[1], V[1], msg_c, plan, &in_out, &passes);
    if (rc)
        return rc;
    u32 dir_log2 = 0;
    rc = build_join_directory(d_sa, n, dir, dir_room, s, &dir_log2, true);
    if (rc)
        return rc;
    hipLaunchKernelGGL(join_messages_kernel, dim3((msg_c + 255u) / 256u), dim3(256), 0, s, (const u8*)nullptr,
                       (const u64*)K[in_out], (const u32*)V[in_out], msg_c, d_sa, d_primary, d_keys, n,
                       (const u32*)(dir_log2 ? dir : nullptr), dir_log2);
    HIP_TRY(hipGetLastError());
    return read_counts(L, nullptr);
}

int csa_stage_slab_u16_dev(const uint16_t* d_text, uint64_t n, const uint8_t* d_suf40, uint64_t count, int key_words,
                           const uint64_t* d_pid_map, uint32_t p, uint64_t ctx, int generation0, uint64_t* d_keys,
                           uint32_t* d_beta, void* stream)
{
    if (key_words < 1 || key_words > 4)
        return fail(CSA_ERR_ARG, "csa_stage_slab_u16_dev: key_words = %d is outside [1, 4]", key_words);
    if (p < 1 || p > 32768u)
        return fail(CSA_ERR_ARG, "csa_stage_slab_u16_dev: p = %u is outside [1, 32768] (bit 15 of a route is the retirement flag)", p);
    if (generation0 && ctx != 4ull * (u64)key_words)
        return fail(CSA_ERR_ARG, "csa_stage_slab_u16_dev: generation 0 runs at ctx = ell = %d", 4 * key_words);
    if (count == 0)
        return CSA_OK;
    if (!d_text || !d_suf40 || !d_pid_map || !d_beta)
        return fail(CSA_ERR_ARG, "csa_stage_slab_u16_dev: null buffer");
    if (n > CSA_MAX_INDEX)
        return fail(CSA_ERR_TOO_LARGE, "csa_stage_slab_u16_dev: text of %llu symbols", (unsigned long long)n);
    StageArgs a;
    a.text = d_text;
    a.n = n;
    a.suf40 = d_suf40;
    a.count = count;
    a.pid_map = d_pid_map;
    a.bits = csa_partition_id_bits(p);
    a.ctx = ctx;
    a.ell = 4u * (u32)key_words;
    a.gen0 = generation0 ? 1 : 0;
    a.keys = d_keys;
    a.beta = d_beta;
    const u64 blocks = (count + 255) / 256;
    if (blocks > 0x7FFFFFFFull)
        return fail(CSA_ERR_TOO_LARGE, "csa_stage_slab_u16_dev: %llu suffixes in one call", (unsigned long long)count);
    hipStream_t s = (hipStream_t)stream;
    switch (key_words) {
    case 1: hipLaunchKernelGGL(stage_slab_kernel<1>, dim3((u32)blocks), dim3(256), 0, s, a); break;
    case 2: hipLaunchKernelGGL(stage_slab_kernel<2>, dim3((u32)blocks), dim3(256), 0, s, a); break;
    case 3: hipLaunchKernelGGL(stage_slab_kernel<3>, dim3((u32)blocks), dim3(256), 0, s, a); break;
    default: hipLaunchKernelGGL(stage_slab_kernel<4>, dim3((u32)blocks), dim3(256), 0, s, a); break;
    }
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

extern "C++" {
namespace {
// The scatter behind csa_scatter_to_rank_order_dev and csa_scatter_slabs; takes its columns from the handle's block as
// that block stands (the caller has reset it, or holds columns of its own in it). Waits for the stream.
int scatter_to_rank_order(csa_handle* h, const char* who, const u8* d_suf, const u32* d_rank, u64 part_sz, u8* d_sa40, hipStream_t s)
{
    HIP_TRY(hipMemsetAsync(h->counts, 0, 4 * sizeof(u32), s));
    const u32 blocks = (u32)((part_sz + 255) / 256);
    u64* K[2] = {nullptr, nullptr};
    u32* V[2] = {nullptr, nullptr};
    bool windowed = part_sz >= SCATTER_WINDOW_MIN && part_sz <= h->cap;
    if (windowed) { // (a block without room for the 24 bytes per suffix of the window pass scatters directly)
        for (int i = 0; i < 2; ++i) {
            K[i] = static_cast<u64*>(h->pool.take(part_sz * sizeof(u64)));
            V[i] = static_cast<u32*>(h->pool.take(part_sz * sizeof(u32)));
        }
        windowed = K[0] && V[0] && K[1] && V[1];
    }
    if (windowed) {
        // large partition: group the pairs by the window of the output their rank falls into, then write window by window
        Launch L;
        L.h = h;
        L.stream = s;
        L.flags = 0;
        L.stats = nullptr;
        hipLaunchKernelGGL(scatter_window_keys_kernel, dim3(blocks), dim3(256), 0, s, d_suf, d_rank, part_sz, (int)SCATTER_WINDOW_LOG2,
                           K[0], V[0], h->counts + 3);
        const int window_bits = bit_length((part_sz - 1) >> SCATTER_WINDOW_LOG2);
        int in_out = 0, passes = 0;
        const int rc = radix_sort(L, SRC_PAIRS, 0, 0, K[0], V[0], K[1], V[1], (u32)part_sz,
                                  make_plan(40, 40 + window_bits), &in_out, &passes);
        if (rc)
            return rc;
        hipLaunchKernelGGL(scatter_window_lanes_kernel, dim3(blocks), dim3(256), 0, s, (const u64*)K[in_out], (const u32*)V[in_out],
                           part_sz, d_sa40);
    } else {
        hipLaunchKernelGGL(scatter_lanes_kernel, dim3(blocks), dim3(256), 0, s, d_suf, d_rank, part_sz, d_sa40, h->counts + 3);
    }
    HIP_TRY(hipGetLastError());
    for (int i = 0; i < 2; ++i) {
        h->pool.give(K[i]);
        h->pool.give(V[i]);
    }
    Launch R;
    R.h = h;
    R.stream = s;
    R.flags = 0;
    R.stats = nullptr;
    const int rc_counts = read_counts(R, nullptr); // waits for the stream; a failed wait of the bucket pass ends here
    if (h->h_pinned[3])
        return fail(CSA_ERR_ARG, "%s: a rank lies outside [0, %llu)", who, (unsigned long long)part_sz);
    return rc_counts;
}
} // namespace
} // extern "C++"

int csa_scatter_to_rank_order_dev(csa_handle* h, const uint8_t* d_suf, const uint32_t* d_rank, uint64_t part_sz,
                                  uint8_t* d_sa40, void* stream)
{
    if (!h)
        return fail(CSA_ERR_ARG, "csa_scatter_to_rank_order_dev: null handle");
    if (part_sz == 0)
        return CSA_OK;
    if (!d_suf || !d_rank || !d_sa40)
        return fail(CSA_ERR_ARG, "csa_scatter_to_rank_order_dev: null buffer");
    if (part_sz > CSA_MAX_PART_SZ)
        return fail(CSA_ERR_TOO_LARGE, "csa_scatter_to_rank_order_dev: %llu suffixes exceed a partition", (unsigned long long)part_sz);
    h->pool.reset();
    const int rc = scatter_to_rank_order(h, "csa_scatter_to_rank_order_dev", d_suf, d_rank, part_sz, d_sa40, (hipStream_t)stream);
    h->last_high_water = h->pool.high_water();
    return rc;
}

void csa_output_cut(uint64_t lo, uint64_t hi, uint64_t chunk_bytes, uint64_t c, uint64_t chunk_c, uint64_t out[6])
{
    constexpr u64 BLK = 4096; // the O_DIRECT granularity of the output file (include/Direct_File.hpp:27)
    auto clamp = [](u64 v, u64 a, u64 b) { return v < a ? a : (v > b ? b : v); };
    const u64 first_block = lo & ~(BLK - 1);       // chunks are laid out from the block that holds the range's start
    const u64 aligned_lo = (lo + BLK - 1) & ~(BLK - 1);
    u64 aligned_hi = hi & ~(BLK - 1);              // [aligned_lo, aligned_hi): the whole blocks of the range
    if (aligned_hi < aligned_lo)
        aligned_hi = aligned_lo;                   // the range lies inside one block
    // the chunk's piece: its window of chunk_bytes, clipped to the whole blocks
    out[0] = clamp(first_block + c * chunk_bytes, aligned_lo, aligned_hi);
    out[1] = clamp(first_block + (c + 1) * chunk_bytes, out[0], aligned_hi);
    // the first chunk also carries what precedes the whole blocks, the last one what follows them
    out[2] = out[3] = out[4] = out[5] = 0;
    if (c == 0) {
        out[2] = lo;
        out[3] = hi < aligned_lo ? hi : aligned_lo;
    }
    if (c + 1 == chunk_c) {
        out[4] = aligned_hi;
        out[5] = hi > aligned_hi ? hi : aligned_hi;
    }
}

const char* csa_last_error(void) { return g_err; }

uint64_t csa_bytes_per_suffix(int key_words)
{
    (void)key_words;
    // three key arrays (8 B), five index arrays (4 B), group ids, ranks, four half-size group tables
    return 3 * 8 + 5 * 4 + 4 + 4 + 4 * 2;
}

extern "C++" {
namespace {

constexpr u64 BLOCK_SLACK = 64u << 10; // what rounding every column up to DevicePool::ALIGN can cost a call

struct WorkspaceSizes {
    u64 lookback_tile_words, lookback_words, rank_tiles_cap;
    u64 bytes;
};

// The workspace: what a handle holds besides its block. It follows the number of tiles, not the number of suffixes.
WorkspaceSizes workspace_sizes(u64 cap)
{
    WorkspaceSizes w;
    const u64 sort_tiles = (cap + SORT_TILE - 1) / SORT_TILE;
    const u64 rank_tiles = (cap + TABLE_TILE - 1) / TABLE_TILE;
    // the group words of the radix pass follow the tile words (passes over nine bits have twice the words for a tile of twice the size: the last one
    // and its group may have no second half)
    w.lookback_tile_words = (sort_tiles + 1) * RADIX_BINS;
    w.lookback_words = w.lookback_tile_words + (sort_tiles / LB_GROUP + 2) * RADIX_BINS;
    if (rank_tiles * 4 > w.lookback_words)
        w.lookback_words = rank_tiles * 4;
    w.rank_tiles_cap = rank_tiles + 1;
    w.bytes = w.lookback_words * 8 + (w.rank_tiles_cap * 9 + RERANK_SLABS * 5) * sizeof(u32) + (MAX_PASSES + 2) * RADIX_BINS * 4 +
              MAX_PASSES * RADIX_BINS * 4 + TICKET_POOL * 4 + 16 * 4 + MSG_OFF_WORDS * 4;
    w.bytes += CODE_TABLE_WORDS * sizeof(u32);
    w.bytes += 10 * 4096; // ten allocations, each rounded up by the runtime
    return w;
}

u64 resident_block_bytes(u64 cap)
{
    const u64 A = DevicePool::ALIGN;
    auto up = [&](u64 b) { return (b + A - 1) & ~(A - 1); };
    return 3 * up(cap * 8) + 5 * up(cap * 4) + 2 * up(cap * 4) + 2 * up((cap / 2 + 1) * 4) + 2 * up((cap / 2 + 2) * 4);
}

int create_handle(const char* who, u64 max_part_sz, int key_words, u32 kinds, csa_handle** out)
{
    if (!out)
        return fail(CSA_ERR_ARG, "%s: out is null", who);
    *out = nullptr;
    if (key_words < 1 || key_words > 4)
        return fail(CSA_ERR_ARG, "%s: key_words = %d is outside [1, 4]", who, key_words);
    if (max_part_sz > CSA_MAX_PART_SZ)
        return fail(CSA_ERR_TOO_LARGE, "%s: %llu suffixes exceed the partition limit %llu", who,
                    (unsigned long long)max_part_sz, (unsigned long long)CSA_MAX_PART_SZ);
    csa_handle* h = new csa_handle();
    h->cap = max_part_sz ? max_part_sz : 1;
    h->key_words = key_words;
    h->kinds = kinds;
    const u64 cap = h->cap;
    const WorkspaceSizes ws = workspace_sizes(cap);
    h->lookback_tile_words = ws.lookback_tile_words;
    h->lookback_words = ws.lookback_words;
    hipError_t e = hipGetDevice(&h->device);
    if (e == hipSuccess)
        e = hipDeviceGetAttribute(&h->cus, hipDeviceAttributeMultiprocessorCount, h->device);
    // Tile order of the radix passes: by arrival, unless the caller declares the device its own
    // (csa_set_device_exclusive); the XCD-chunked order then needs 8 * XCD_CHUNK workgroups of a pass resident at once
    // and is offered only on a device with room for twice that many (csa_set_tuning changes the chunk length).
    h->tile_order = TILES_BY_ARRIVAL;
    h->tile_order_exclusive = h->cus >= 2 * 8 * (int)XCD_CHUNK ? TILES_STATIC_CHUNKS : TILES_BY_ARRIVAL;
    h->xcd_chunk = XCD_CHUNK;
    auto alloc = [&](void** p, u64 bytes) {
        if (e == hipSuccess)
            e = hipMalloc(p, bytes ? bytes : 4);
    };
    // the block: the resident sort's floor plan, or what the steps keep alive at their busiest moment
    u64 block_bytes = ((kinds & KIND_RESIDENT) ? resident_block_bytes(cap) : csa_step_bytes_per_suffix(key_words) * cap) + BLOCK_SLACK;
    block_bytes = (block_bytes + DevicePool::ALIGN - 1) & ~(DevicePool::ALIGN - 1);
    alloc((void**)&h->block, block_bytes);
    if (e == hipSuccess) {
        h->pool.attach(h->block, block_bytes);
        if (kinds & KIND_RESIDENT) { // the fixed carve-up of the resident sort
            for (int i = 0; i < 3; ++i)
                h->key[i] = static_cast<u64*>(h->pool.take(cap * 8));
            for (int i = 0; i < 5; ++i)
                h->idx[i] = static_cast<u32*>(h->pool.take(cap * 4));
            h->gid = static_cast<u32*>(h->pool.take(cap * 4));
            h->rank = static_cast<u32*>(h->pool.take(cap * 4));
            for (int i = 0; i < 2; ++i)
                h->gprim[i] = static_cast<u32*>(h->pool.take((cap / 2 + 1) * 4));
            for (int i = 0; i < 2; ++i)
                h->gstart[i] = static_cast<u32*>(h->pool.take((cap / 2 + 2) * 4));
            if (!h->gstart[1])
                e = hipErrorOutOfMemory; // (cannot happen: the block was sized by the same sum)
            h->pool.reset();
        }
    }
    alloc((void**)&h->lookback, h->lookback_words * 8);
    h->rank_tiles_cap = ws.rank_tiles_cap;
    alloc((void**)&h->tile_tables, (h->rank_tiles_cap * 9 + RERANK_SLABS * 5) * sizeof(u32));
    alloc((void**)&h->ghist, (MAX_PASSES + 2) * RADIX_BINS * 4);
    if (kinds & KIND_RESIDENT)
        alloc((void**)&h->code_tables, CODE_TABLE_WORDS * sizeof(u32));
    alloc((void**)&h->digit_base, MAX_PASSES * RADIX_BINS * 4);
    alloc((void**)&h->tickets, TICKET_POOL * 4);
    alloc((void**)&h->counts, 16 * 4);
    alloc((void**)&h->msg_off, MSG_OFF_WORDS * 4);
    if (e == hipSuccess)
        e = hipHostMalloc((void**)&h->h_pinned, (PINNED_HIST + MAX_PASSES * RADIX_BINS) * 4, hipHostMallocDefault);
    if (e == hipSuccess)
        e = hipMemset(h->lookback, 0, h->lookback_words * 8);
    if (e == hipSuccess)
        e = hipMemset(h->tickets, 0, TICKET_POOL * 4);
    if (e == hipSuccess)
        e = hipMemset(h->counts, 0, 16 * 4);
    if (e == hipSuccess)
        e = hipDeviceSynchronize();
    if (e != hipSuccess) {
        const int rc = fail(CSA_ERR_HIP, "%s: %s while allocating for %llu suffixes", who, hipGetErrorString(e), (unsigned long long)cap);
        csa_destroy(h);
        return rc;
    }
    *out = h;
    return CSA_OK;
}

} // namespace
} // extern "C++"

uint64_t csa_workspace_bytes(uint64_t max_part_sz) { return workspace_sizes(max_part_sz ? max_part_sz : 1).bytes + BLOCK_SLACK; }

int csa_create(uint64_t max_part_sz, int key_words, csa_handle** out)
{
    return create_handle("csa_create", max_part_sz, key_words, KIND_RESIDENT, out);
}

int csa_create_steps(uint64_t max_part_sz, int key_words, csa_handle** out)
{
    return create_handle("csa_create_steps", max_part_sz, key_words, 0u, out);
}

int csa_set_tuning(csa_handle* h, int knob, uint32_t value)
{
    if (!h)
        return fail(CSA_ERR_ARG, "csa_set_tuning: null handle");
    switch (knob) {
    case CSA_TUNE_DEFER_MIN: h->defer_min = value, h->settle = 0; break;
    case CSA_TUNE_WINDOW_MIN_CHANGED: h->window_min_changed = value, h->settle = 0; break;
    case CSA_TUNE_PACK_SYMBOLS: h->pack_symbols = value ? 1u : 0u; break;
    case CSA_TUNE_EXPECT_PRESORTED: h->expect_presorted = value ? 1u : 0u; break;
    case CSA_TUNE_SETTLE: h->settle = value ? 1u : 0u; break;
    case CSA_TUNE_XCD_CHUNK:
        // the chunked order waits for workgroups that are dispatched later: 8 * chunk workgroups of a pass must be able
        // to be resident together, and the device must have room for twice that many (the condition csa_create applies)
        if (value && 2ull * 8ull * value > (u64)(h->cus > 0 ? h->cus : 0))
            return fail(CSA_ERR_ARG, "csa_set_tuning: an XCD chunk of %u tiles needs %llu compute units, the device has %d", value,
                        2ull * 8ull * value, h->cus);
        h->tile_order_exclusive = value ? TILES_STATIC_CHUNKS : TILES_BY_ARRIVAL;
        if (value)
            h->xcd_chunk = value;
        if (h->tile_order != TILES_BY_ARRIVAL) // the handle is in the exclusive order already: follow
            h->tile_order = h->tile_order_exclusive;
        break;
    default: return fail(CSA_ERR_ARG, "csa_set_tuning: unknown knob %d", knob);
    }
    return CSA_OK;
}

int csa_set_device_exclusive(csa_handle* h, int exclusive)
{
    if (!h)
        return fail(CSA_ERR_ARG, "csa_set_device_exclusive: null handle");
    h->tile_order = exclusive ? h->tile_order_exclusive : TILES_BY_ARRIVAL;
    return CSA_OK;
}

void csa_destroy(csa_handle* h)
{
    if (!h)
        return;
    (void)hipFree(h->block);
    (void)hipFree(h->lookback);
    (void)hipFree(h->tile_tables);
    (void)hipFree(h->ghist);
    (void)hipFree(h->code_tables);
    (void)hipFree(h->digit_base);
    (void)hipFree(h->tickets);
    (void)hipFree(h->counts);
    (void)hipFree(h->msg_off);
    if (h->h_pinned)
        (void)hipHostFree(h->h_pinned);
    for (auto& e : h->events)
        (void)hipEventDestroy(e);
    if (h->ev_gen_ready)
        for (auto& e : h->ev_gen)
            (void)hipEventDestroy(e);
    delete h;
}

int csa_sort_partition_u16_dev(csa_handle* h, const uint16_t* d_text, uint64_t n, uint64_t index_base,
                               uint8_t* d_sa40, void* stream, uint32_t flags, csa_stats* stats)
{
    if (!h)
        return fail(CSA_ERR_ARG, "csa_sort_partition_u16_dev: handle is null");
    if (n > CSA_MAX_PART_SZ)
        return fail(CSA_ERR_TOO_LARGE, "csa_sort_partition_u16_dev: %llu suffixes exceed the partition limit %llu",
                    (unsigned long long)n, (unsigned long long)CSA_MAX_PART_SZ);
    if (index_base > CSA_MAX_INDEX || index_base + n > CSA_MAX_INDEX)
        return fail(CSA_ERR_TOO_LARGE, "csa_sort_partition_u16_dev: suffix indices up to %llu do not fit 40 bits",
                    (unsigned long long)(index_base + n));
    if (!(h->kinds & KIND_RESIDENT))
        return fail(CSA_ERR_ARG, "csa_sort_partition_u16_dev: the handle was created by csa_create_steps, which leaves out the "
                    "resident sort's arrays; use csa_create");
    if (n > h->cap)
        return fail(CSA_ERR_ARG, "csa_sort_partition_u16_dev: %llu suffixes exceed the handle's capacity %llu",
                    (unsigned long long)n, (unsigned long long)h->cap);
    csa_stats local;
    csa_stats* st = stats ? stats : &local;
    memset(st, 0, sizeof(*st));
    st->n = n;
    st->key_words = h->key_words;
    if (n == 0)
        return CSA_OK;
    if (!d_text || !d_sa40)
        return fail(CSA_ERR_ARG, "csa_sort_partition_u16_dev: null text or output pointer");
    int rc = ensure_events(h, flags & CSA_FLAG_KERNEL_TIMING);
    if (rc)
        return rc;
    Launch L;
    L.h = h;
    L.stream = (hipStream_t)stream;
    L.flags = flags;
    L.stats = st;
    return sort_partition(L, d_text, n, index_base, d_sa40);
}

int csa_pack_keys_u16_dev(const uint16_t* d_text, uint64_t n, int key_words, uint64_t* d_keys, void* stream)
{
    if (key_words < 1 || key_words > 4)
        return fail(CSA_ERR_ARG, "csa_pack_keys_u16_dev: key_words = %d is outside [1, 4]", key_words);
    if (n > CSA_MAX_PART_SZ)
        return fail(CSA_ERR_TOO_LARGE, "csa_pack_keys_u16_dev: %llu suffixes exceed the partition limit",
                    (unsigned long long)n);
    if (n == 0)
        return CSA_OK;
    if (!d_text || !d_keys)
        return fail(CSA_ERR_ARG, "csa_pack_keys_u16_dev: null pointer");
    hipLaunchKernelGGL(pack_keys_kernel, dim3((u32)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, d_text, (u32)n,
                       key_words, d_keys);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
    return CSA_OK;
}

int csa_radix_sort_pairs_dev(csa_handle* h, uint64_t* d_keys, uint32_t* d_vals, uint64_t n, int begin_bit,
                             int end_bit, void* stream)
{
    if (!h)
        return fail(CSA_ERR_ARG, "csa_radix_sort_pairs_dev: handle is null");
    if (begin_bit < 0 || end_bit > 64 || begin_bit > end_bit)
        return fail(CSA_ERR_ARG, "csa_radix_sort_pairs_dev: bad bit range [%d, %d)", begin_bit, end_bit);
    if (n > h->cap)
        return fail(CSA_ERR_ARG, "csa_radix_sort_pairs_dev: %llu pairs exceed the handle's capacity %llu",
                    (unsigned long long)n, (unsigned long long)h->cap);
    if (n == 0 || begin_bit == end_bit)
        return CSA_OK;
    if (!d_keys || !d_vals)
        return fail(CSA_ERR_ARG, "csa_radix_sort_pairs_dev: null pointer");
    Launch L;
    L.h = h;
    L.stream = (hipStream_t)stream;
    L.flags = 0;
    L.stats = nullptr;
    HIP_TRY(hipMemsetAsync(h->counts, 0, 4 * sizeof(u32), L.stream));
    h->pool.reset();
    u64* tmp_keys = static_cast<u64*>(h->pool.take(n * 8));
    u32* tmp_vals = static_cast<u32*>(h->pool.take(n * 4));
    h->last_high_water = h->pool.high_water();
    if (!tmp_keys || !tmp_vals)
        return fail(CSA_ERR_ARG, "csa_radix_sort_pairs_dev: the handle's block of %llu bytes has no room for 12 bytes per pair",
                    (unsigned long long)h->pool.bytes());
    int in_out = 0, passes = 0;
    const PassPlan plan = make_plan(begin_bit, end_bit);
    int rc = radix_sort(L, SRC_PAIRS, 0, 0, d_keys, d_vals, tmp_keys, tmp_vals, (u32)n, plan, &in_out, &passes);
    if (rc)
        return rc;
    if (in_out) {
        HIP_TRY(hipMemcpyAsync(d_keys, tmp_keys, n * 8, hipMemcpyDeviceToDevice, L.stream));
        HIP_TRY(hipMemcpyAsync(d_vals, tmp_vals, n * 4, hipMemcpyDeviceToDevice, L.stream));
    }
    return read_counts(L, nullptr);
}

extern "C++" {
namespace {
constexpr int STATIC_MAX_DEVICES = 64;
std::mutex g_static_mutex;
unsigned char* g_static_ptr[STATIC_MAX_DEVICES] = {}; // address of `scratch` on each device, asked for once per device

// The current device's copy of `scratch`.
int static_scratch(unsigned char** out)
{
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= STATIC_MAX_DEVICES)
        return fail(CSA_ERR_ARG, "csa_radix_sort_pairs_static_dev: device %d is beyond the %d devices this entry point keeps a scratch address for",
                    dev, STATIC_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_static_mutex);
    if (!g_static_ptr[dev]) {
        void* p = nullptr;
        HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p)
            return fail(CSA_ERR_HIP, "csa_radix_sort_pairs_static_dev: no address for the scratch array on device %d", dev);
        g_static_ptr[dev] = static_cast<unsigned char*>(p);
    }
    *out = g_static_ptr[dev];
    return CSA_OK;
}
} // namespace
} // extern "C++"

int csa_radix_sort_pairs_static_dev(uint64_t* d_keys, uint32_t* d_vals, uint64_t n, int begin_bit, int end_bit, void* stream)
{
    if (begin_bit < 0 || end_bit > 64 || begin_bit > end_bit)
        return fail(CSA_ERR_ARG, "csa_radix_sort_pairs_static_dev: bad bit range [%d, %d)", begin_bit, end_bit);
    if (n > STATIC_SORT_MAX)
        return fail(CSA_ERR_TOO_LARGE, "csa_radix_sort_pairs_static_dev: %llu pairs exceed the %llu this entry point's fixed scratch holds "
                    "(use csa_radix_sort_pairs_dev with a handle)", (unsigned long long)n, (unsigned long long)STATIC_SORT_MAX);
    unsigned char* base = nullptr; // the device address of the scratch array: never the array's name from here on
    int rc = static_scratch(&base);
    if (rc)
        return rc;
    if (n == 0 || begin_bit == end_bit)
        return CSA_OK;
    if (!d_keys || !d_vals)
        return fail(CSA_ERR_ARG, "csa_radix_sort_pairs_static_dev: null pointer");
    hipStream_t s = (hipStream_t)stream;
    u64* tmp_keys = reinterpret_cast<u64*>(base + STATIC_OFF_KEYS);
    u32* tmp_vals = reinterpret_cast<u32*>(base + STATIC_OFF_VALS);
    u64* lookback = reinterpret_cast<u64*>(base + STATIC_OFF_LOOKBACK);
    u32* ghist = reinterpret_cast<u32*>(base + STATIC_OFF_GHIST);
    u32* tickets = reinterpret_cast<u32*>(base + STATIC_OFF_TICKETS);
    u32* err = reinterpret_cast<u32*>(base + STATIC_OFF_ERR);
    u32* digit_base = reinterpret_cast<u32*>(base + STATIC_OFF_DIGIT_BASE);
    // The array keeps what the last call left: look-back words, digit counts, tile tickets and the error word start at
    // zero in every call (a fill kernel, not a memset node: the call may be recorded into a graph). With the words
    // cleared the launch epoch can stay the same in every call and replay.
    const u64 control_words = (STATIC_CONTROL_END - STATIC_OFF_CONTROL) / sizeof(u32);
    hipLaunchKernelGGL(fill_u32_kernel, dim3((u32)((control_words + 255) / 256)), dim3(256), 0, s,
                       reinterpret_cast<u32*>(base + STATIC_OFF_CONTROL), control_words, 0u);
    const PassPlan plan = make_plan(begin_bit, end_bit);
    HistArgs ha;
    ha.keys = d_keys;
    ha.n = (u32)n;
    ha.plan = plan;
    ha.ghist = ghist;
    hipLaunchKernelGGL(radix_hist_kernel, dim3(hist_blocks(256 * 16, n)), dim3(256), 0, s, ha);
    hipLaunchKernelGGL(radix_scan_hist_kernel<RADIX_BINS>, dim3(1), dim3(RADIX_BINS), 0, s, ghist, digit_base, plan.num_passes);
    // every pass runs (skipping the passes whose digit is constant would need the counts on the host: a round trip)
    const TileOrder by_arrival = {TILES_BY_ARRIVAL, XCD_CHUNK};
    int where = 0; // 0: the pairs are in the caller's arrays, 1: in the scratch
    for (int p = 0; p < plan.num_passes; ++p) {
        OnesweepArgs a;
        a.keys_in = where == 0 ? d_keys : tmp_keys;
        a.vals_in = where == 0 ? d_vals : tmp_vals;
        a.keys_out = where == 0 ? tmp_keys : d_keys;
        a.vals_out = where == 0 ? tmp_vals : d_vals;
        a.n = (u32)n;
        a.text_n = 0;
        a.tail = 0;
        a.shift = plan.shift[p];
        a.bits = plan.bits[p];
        a.digit_base = digit_base + p * RADIX_BINS;
        a.lookback = lookback + (u64)p * STATIC_LB_WORDS;
        a.lookback_groups = a.lookback + STATIC_LB_TILE_WORDS;
        a.ticket = tickets + p;
        a.epoch = 1;
        a.err = err;
        launch_onesweep_shape<SRC_PAIRS, SORT_BLOCK, true>(by_arrival, a, s);
        where ^= 1;
    }
    if (where)
        hipLaunchKernelGGL(copy_pairs_kernel, dim3((u32)((n + 255) / 256)), dim3(256), 0, s, (const u64*)tmp_keys, (const u32*)tmp_vals,
                           (u64)n, d_keys, d_vals);
    HIP_TRY(hipGetLastError());
    return CSA_OK;
}

int csa_radix_sort_pairs_static_status(void* stream)
{
    unsigned char* base = nullptr; // (the device address of the scratch array, as in the sort itself)
    int rc = static_scratch(&base);
    if (rc)
        return rc;
    hipStream_t s = (hipStream_t)stream;
    u32 err = 0; // one word into the caller's stack: no buffer is allocated for it
    HIP_TRY(hipMemcpyAsync(&err, base + STATIC_OFF_ERR, sizeof(u32), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    if (err)
        return fail(CSA_ERR_INTERNAL, "csa_radix_sort_pairs_static_dev: device invariant %u failed in the last sort on this device%s", err,
                    err == DEV_ERR_LOOKBACK_TIMEOUT ? " (a look-back wait ran into its spin limit): the pairs it left are not sorted" : "");
    return CSA_OK;
}

int csa_verify_sa40_dev(csa_handle* h, const uint16_t* d_text, uint64_t n, uint64_t index_base,
                        const uint8_t* d_sa40, void* stream, int* ok)
{
    if (!h || !ok)
        return fail(CSA_ERR_ARG, "csa_verify_sa40_dev: null handle or result pointer");
    *ok = 0;
    if (n > h->cap)
        return fail(CSA_ERR_ARG, "csa_verify_sa40_dev: %llu suffixes exceed the handle's capacity %llu",
                    (unsigned long long)n, (unsigned long long)h->cap);
    if (n == 0) {
        *ok = 1;
        return CSA_OK;
    }
    if (!d_text || !d_sa40)
        return fail(CSA_ERR_ARG, "csa_verify_sa40_dev: null pointer");
    hipStream_t s = (hipStream_t)stream;
    const u32 blocks = (u32)((n + 255) / 256);
    h->pool.reset();
    u32* inverse = static_cast<u32*>(h->pool.take(n * sizeof(u32))); // the inverse suffix array
    h->last_high_water = h->pool.high_water();
    if (!inverse)
        return fail(CSA_ERR_ARG, "csa_verify_sa40_dev: the handle's block of %llu bytes has no room for 4 bytes per suffix",
                    (unsigned long long)h->pool.bytes());
    HIP_TRY(hipMemsetAsync(h->counts + 3, 0, sizeof(u32), s));
    hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks), dim3(256), 0, s, inverse, n, 0xFFFFFFFFu);
    hipLaunchKernelGGL(verify_invert_kernel, dim3(blocks), dim3(256), 0, s, d_sa40, (u32)n, index_base, inverse,
                       h->counts + 3);
    hipLaunchKernelGGL(verify_order_kernel, dim3(blocks), dim3(256), 0, s, d_sa40, d_text, (u32)n, index_base, inverse,
                       h->counts + 3);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(h->h_pinned + 3, h->counts + 3, sizeof(u32), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    *ok = h->h_pinned[3] ? 0 : 1;
    return CSA_OK;
}

int csa_enable_profile_ranges(int enable)
{
    if (enable_ranges(enable != 0))
        return fail(CSA_ERR_ARG, "csa_enable_profile_ranges: no roctx library (librocprofiler-sdk-roctx.so, libroctx64.so) could be loaded");
    return CSA_OK;
}

} // extern "C"

#include "step_entries.hpp"
#include "slab_entries.hpp"
#include "host_pipeline.hpp"
