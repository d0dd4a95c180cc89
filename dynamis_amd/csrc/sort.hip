// Stable LSD radix sort for gfx950: 8-bit digits, one histogram read for all digits, then one
// "onesweep" pass per digit. Each pass ranks a tile of 4096 or 8192 keys with wave64 ballots (a key's rank
// among equal digits is the popcount of the lanes below it that hold the same digit, plus the
// counts of earlier items and earlier waves), publishes the tile's digit counts for a decoupled
// look-back across tiles, stages the ranked tile in LDS and writes it out digit-run by digit-run
// so that the global stores coalesce.
//
// Behaviour follows `RadixSort::sort` (crates/dynamis-sort/src/radix.rs:397-476): records
// [base, base+len) of (major, minor, payload), len read on the device, digits of the minor word
// first then the major word (radix.rs:312-317), ties kept in input order, result in the primaries.
// The reference ranks with per-unit serial prefix loops (sort_scatter.wgsl:45-104); the order
// produced is the same stable order.
#include "sort.h"

#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace dyn {

namespace {

constexpr uint32_t kFlagAggregate = 1u << 30;
constexpr uint32_t kFlagPrefix = 2u << 30;
constexpr uint32_t kFlagValue = (1u << 30) - 1;
constexpr uint32_t kSpinLimit = 1u << 22;

}  // namespace

// Look-back waits that gave up since the count was last cleared, over every sort this process ran
// on the device (never expected: a tile's predecessors always publish). A timed-out tile scatters
// with a partial prefix, so a non-zero count means some sort's order is wrong; dyn_sort_faults
// reads it.
__device__ uint32_t g_sort_faults = 0u;

namespace {

struct DigitList {
    uint32_t major[kSortMaxPasses];
    uint32_t shift[kSortMaxPasses];
    uint32_t count;
};

__global__ void __launch_bounds__(256) sort_prepare_kernel(uint32_t* hist, uint32_t* ctl,
                                                           const uint32_t* d_count,
                                                           const uint32_t* d_base,
                                                           uint32_t capacity) {
    const uint32_t t = threadIdx.x;
    for (uint32_t i = t; i < kSortMaxPasses * kSortBins; i += blockDim.x) hist[i] = 0;
    if (t >= 2 && t < kCtlWords) ctl[t] = 0;
    if (t == 0) {
        uint32_t base = d_base ? d_base[0] : 0u;
        if (base > capacity) base = capacity;
        uint32_t count = d_count ? d_count[0] : capacity;
        uint32_t room = capacity - base;
        ctl[kCtlLen] = count < room ? count : room;
        ctl[kCtlBase] = base;
    }
}

// Workgroups of the histogram: each adds its 256 counts a pass to the same words, so few large ones.
constexpr uint32_t kHistogramGroups = 256;
constexpr uint32_t kHistogramThreads = 1024;

__global__ void __launch_bounds__(kHistogramThreads) sort_histogram_kernel(const uint32_t* __restrict__ major,
                                                                           const uint32_t* __restrict__ minor,
                                                                           uint32_t* hist, const uint32_t* ctl,
                                                                           uint32_t* flags0, DigitList digits) {
    __shared__ uint32_t s_hist[kSortMaxPasses][kSortBins];
    const uint32_t t = threadIdx.x;
    for (uint32_t k = t; k < digits.count * kSortBins; k += kHistogramThreads) (&s_hist[0][0])[k] = 0;
    __syncthreads();
    const uint32_t len = ctl[kCtlLen];
    const uint32_t base = ctl[kCtlBase];
    bool uses_major = false, uses_minor = false;
    for (uint32_t p = 0; p < digits.count; ++p) {
        uses_major |= digits.major[p] != 0;
        uses_minor |= digits.major[p] == 0;
    }
    const uint32_t stride = gridDim.x * kHistogramThreads;
    for (uint32_t i = blockIdx.x * kHistogramThreads + t; i < len; i += stride) {
        const uint32_t hi = uses_major ? major[base + i] : 0u;
        const uint32_t lo = uses_minor ? minor[base + i] : 0u;
        for (uint32_t p = 0; p < digits.count; ++p) {
            const uint32_t word = digits.major[p] ? hi : lo;
            atomicAdd(&s_hist[p][(word >> digits.shift[p]) & 0xFFu], 1u);
        }
    }
    __syncthreads();
    for (uint32_t k = t; k < digits.count * kSortBins; k += kHistogramThreads) {
        const uint32_t c = (&s_hist[0][0])[k];
        if (c) atomicAdd(&hist[k], c);
    }
    const uint32_t words = ceil_div(len, kSortMinTile) * kSortBins;
    for (uint32_t i = blockIdx.x * kHistogramThreads + t; i < words; i += stride) flags0[i] = 0;
}

// A lane's rank among its wave's keys of digit d so far: the wave's earlier items (counted in
// `counts`), then the lanes below it; the counts move on. Lanes and items in order are input order.
__device__ __forceinline__ uint32_t wave_rank(uint32_t d, bool valid, uint32_t* counts) {
    const uint64_t live = __ballot(valid);
    uint32_t low = static_cast<uint32_t>(live), high = static_cast<uint32_t>(live >> 32);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        // all ones where the bit is set: peers keep the lanes whose bit is this lane's, a three-input
        // bit operation for each half of the wave
        const uint32_t mine = static_cast<uint32_t>(static_cast<int32_t>(d << (31 - b)) >> 31);
        const uint64_t m = __ballot(mine != 0u);
        low &= ~(static_cast<uint32_t>(m) ^ mine);
        high &= ~(static_cast<uint32_t>(m >> 32) ^ mine);
    }
    const uint32_t before = __builtin_amdgcn_mbcnt_hi(high, __builtin_amdgcn_mbcnt_lo(low, 0u));
    const uint32_t total = __popc(low) + __popc(high);
    uint32_t prior = 0;
    if (valid) prior = counts[d];
    if (valid && before == 0) counts[d] = prior + total;
    return prior + before;
}

// One lane of a short list's records moved to their places.
template <int ITEMS>
__device__ __forceinline__ void small_exchange(uint32_t (&v)[ITEMS], const uint32_t (&place)[ITEMS], uint32_t rounds,
                                               uint32_t wave_first, uint32_t len, uint32_t* stage) {
    const uint32_t lane = lane_id();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (i < static_cast<int>(rounds) && wave_first + i * kWave + lane < len) stage[place[i]] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t local = wave_first + i * kWave + lane;
        if (i < static_cast<int>(rounds) && local < len) v[i] = stage[local];
    }
    __syncthreads();
}

// Predecessor words a digit's look-back keeps in flight: it walks back over the aggregates of the
// tiles that run beside it, and one dependent read each (about 0.8 us across XCDs) would serialize
// the tiles.
constexpr int kLookBack = 8;

struct PassArgs {
    const uint32_t *in_sort, *in_other, *in_pay;
    uint32_t *out_sort, *out_other, *out_pay;
    const uint32_t* hist;
    uint32_t *flags, *flags_next, *ctl;
    uint32_t pass, shift;
};

// Passes of 8 keys a lane read the digits' counts beside the control words, and up to this many tiles draw
// their first ticket before the counts' scan: a pass of few tiles is a chain of latencies, which are then
// beside one another. A fixed grid of 8,043 boxes (10 passes) takes 120 us so and 123 without, a million
// records of six digits 129 and 131; with 16 keys a lane, where registers are short, 3,000,017 records
// took 209 us so and 206 without.
constexpr uint32_t kFewTiles = 128;

// One digit pass over tiles of kSortThreads * ITEMS keys. A workgroup with no tile leaves at once,
// and where every tile has a workgroup of its own, each takes one ticket only: the tickets are
// atomics on one word, 15 to 20 ns each, and 1,024 workgroups' tickets cost an empty pass 18 us.
// The three lanes go through one staging buffer in turn, and no load sits in a branch, so the other
// lanes' words arrive while the keys are ranked. 3,000,017 records of three lanes: 46.6 -> 31.6 us a
// pass (72 MB moved, 2.3 TB/s; what is left is the chain of a tile: ticket, load, ranking, look-back).
template <int ITEMS, bool MOVE_OTHER, bool PAYLOAD>
__device__ __forceinline__ void sort_pass(const PassArgs& a, uint32_t* s_stage) {
    constexpr int TILE = kSortThreads * ITEMS;
    constexpr int WAVES = kSortThreads / kWave;
    __shared__ uint32_t s_wave[WAVES][kSortBins];
    __shared__ uint32_t s_start[kSortBins];
    __shared__ uint32_t s_global[kSortBins];
    __shared__ uint32_t s_scan[WAVES];
    __shared__ uint32_t s_tile;
    const uint32_t *__restrict__ in_sort = a.in_sort, *__restrict__ in_other = a.in_other, *__restrict__ in_pay = a.in_pay;
    uint32_t *__restrict__ out_sort = a.out_sort, *__restrict__ out_other = a.out_other, *__restrict__ out_pay = a.out_pay;
    uint32_t *flags_pass = a.flags, *flags_next = a.flags_next, *ctl = a.ctl;
    const uint32_t pass = a.pass, shift = a.shift;
    const uint32_t t = threadIdx.x;
    const uint32_t lane = lane_id();
    const uint32_t wave = t / kWave;
    uint32_t digit_count = 0;
    if (ITEMS <= 8 && t < kSortBins) digit_count = a.hist[t];
    const uint32_t len = ctl[kCtlLen];
    const uint32_t base = ctl[kCtlBase];
    const uint32_t ntiles = ceil_div(len, TILE);
    if (blockIdx.x >= ntiles) return;

    bool drawn = ITEMS <= 8 && ntiles <= kFewTiles;
    uint32_t ticket = 0;
    if (drawn && t == 0) ticket = atomicAdd(&ctl[kCtlTiles + pass], 1u);
    // Global start of every digit: exclusive scan of this pass's histogram.
    if (ITEMS > 8 && t < kSortBins) digit_count = a.hist[t];
    const uint32_t digit_base = block_exclusive_sum<kSortThreads>(digit_count, s_scan, nullptr);
    for (;;) {
        if (!drawn && t == 0) ticket = atomicAdd(&ctl[kCtlTiles + pass], 1u);
        if (t == 0) s_tile = ticket;
        drawn = false;
        for (uint32_t k = t; k < WAVES * kSortBins; k += kSortThreads) (&s_wave[0][0])[k] = 0u;
        __syncthreads();
        const uint32_t tile = s_tile;
        if (tile >= ntiles) break;
        const uint32_t first = tile * TILE;
        const uint32_t tile_n = min(static_cast<uint32_t>(TILE), len - first);
        if (flags_next && t < kSortBins) flags_next[tile * kSortBins + t] = 0;

        uint32_t key[ITEMS], other[ITEMS], pay[ITEMS], place[ITEMS];
        const uint32_t wave_first = wave * (ITEMS * kWave);
        // Lanes past the tile's end read its last record again, so that no load sits in a branch: the
        // other lanes' words stay in flight while the keys are ranked.
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) key[i] = in_sort[base + first + min(wave_first + i * kWave + lane, tile_n - 1u)];
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t from = base + first + min(wave_first + i * kWave + lane, tile_n - 1u);
            if (PAYLOAD) pay[i] = in_pay[from];
            if (MOVE_OTHER) other[i] = in_other[from];
        }
        // Rank within the wave: items in order, lanes in order, which is input order.
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t local = wave_first + i * kWave + lane;
            const bool valid = local < tile_n;
            const uint32_t d = (key[i] >> shift) & 0xFFu;
            place[i] = wave_rank(d, valid, s_wave[wave]);
        }
        __syncthreads();

        // Digit t: per-wave offsets, tile count, tile-local start.
        uint32_t count = 0;
        if (t < kSortBins) {
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const uint32_t c = s_wave[w][t];
                s_wave[w][t] = count;
                count += c;
            }
            // the tile's counts as early as possible: later tiles wait for them
            atomic_store_agent(&flags_pass[tile * kSortBins + t], (tile == 0u ? kFlagPrefix : kFlagAggregate) | count);
        }
        const uint32_t start = block_exclusive_sum<kSortThreads>(count, s_scan, nullptr);
        if (t < kSortBins) s_start[t] = start;
        __syncthreads();
        // the keys to their local places, which do not need the look-back
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t local = wave_first + i * kWave + lane;
            if (local < tile_n) {
                const uint32_t d = (key[i] >> shift) & 0xFFu;
                place[i] += s_start[d] + s_wave[wave][d];
                s_stage[place[i]] = key[i];
            }
        }
        if (t < kSortBins) {
            // Decoupled look-back over earlier tiles for digit t, kLookBack of them at a time.
            uint32_t excl = 0;
            uint32_t spins = 0;
            bool open = tile != 0u;
            int64_t j = static_cast<int64_t>(tile) - 1;
            while (open) {
                uint32_t v[kLookBack];
#pragma unroll
                for (int b = 0; b < kLookBack; ++b) {
                    v[b] = j >= b ? atomic_load_agent(&flags_pass[(j - b) * kSortBins + t]) : kFlagPrefix;
                }
                bool waits = false;
#pragma unroll
                for (int b = 0; b < kLookBack; ++b) {
                    if (!open || waits) continue;
                    const uint32_t status = v[b] >> 30;
                    if (status == 0u) {
                        waits = true;
                        continue;
                    }
                    excl += v[b] & kFlagValue;
                    --j;
                    if (status == 2u) open = false;
                }
                if (waits) {
                    if (++spins > kSpinLimit) {
                        atomicOr(&ctl[kCtlError], 1u);
                        atomicAdd(&g_sort_faults, 1u);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
            }
            if (tile != 0u) {
                atomic_store_agent(&flags_pass[tile * kSortBins + t], kFlagPrefix | ((excl + count) & kFlagValue));
            }
            s_global[t] = digit_base + excl - start;
        }
        __syncthreads();
        // Where the staged record t + k * kSortThreads goes. Always below len when the look-back
        // completed; the guard keeps a timed-out look-back (ctl error word set) from writing outside
        // the stream.
        uint32_t at[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const uint32_t j = t + k * kSortThreads;
            at[k] = len;
            if (j < tile_n) {
                const uint32_t staged = s_stage[j];
                at[k] = s_global[(staged >> shift) & 0xFFu] + j;
                if (at[k] < len) out_sort[base + at[k]] = staged;
            }
        }
        if (PAYLOAD) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                if (wave_first + i * kWave + lane < tile_n) s_stage[place[i]] = pay[i];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < ITEMS; ++k) {
                if (at[k] < len) out_pay[base + at[k]] = s_stage[t + k * kSortThreads];
            }
        }
        if (MOVE_OTHER) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                if (wave_first + i * kWave + lane < tile_n) s_stage[place[i]] = other[i];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < ITEMS; ++k) {
                if (at[k] < len) out_other[base + at[k]] = s_stage[t + k * kSortThreads];
            }
        }
        if (gridDim.x >= ntiles) break;  // a workgroup per tile: this was its only one
        __syncthreads();
    }
}

// Streams of up to this many live records use 8 keys a lane also where the capacity (all that the
// host knows) asks for 16: 200,000 records in a stream of 4,194,304 took 119 us with 16 and 93 us with
// 8, 1,500,000 165 and 162 us, 3,000,017 208 and 237 us.
constexpr uint32_t kNarrowBelow = 1572864u;

template <int ITEMS, bool MOVE_OTHER, bool PAYLOAD>
__global__ void __launch_bounds__(kSortThreads, 4) sort_pass_kernel(PassArgs a) {
    __shared__ uint32_t s_stage[kSortThreads * ITEMS];
    if (ITEMS > 8 && a.ctl[kCtlLen] <= kNarrowBelow) sort_pass<8, MOVE_OTHER, PAYLOAD>(a, s_stage);
    else sort_pass<ITEMS, MOVE_OTHER, PAYLOAD>(a, s_stage);
}

// A short list sorted whole by one workgroup: every digit pass ranks the records where they are in
// registers and exchanges them through LDS, so nothing but the input and the result touches memory,
// in one launch instead of 2 + passes (+ 1 for an odd count). What bounds it is the latency of a
// pass (six barriers, the ranking's ballots and the exchange).
template <int ITEMS>
__global__ void __launch_bounds__(kSmallThreads) sort_small_kernel(uint32_t* major, uint32_t* minor, uint32_t* payload,
                                                                   const uint32_t* d_count, const uint32_t* d_base,
                                                                   uint32_t capacity, DigitList digits) {
    constexpr int WAVES = kSmallThreads / kWave;
    __shared__ uint32_t s_stage[kSmallThreads * ITEMS];
    __shared__ uint32_t s_wave[WAVES][kSortBins];
    __shared__ uint32_t s_start[kSortBins];
    __shared__ uint32_t s_scan[WAVES];
    const uint32_t t = threadIdx.x;
    const uint32_t lane = lane_id();
    const uint32_t wave = t / kWave;
    uint32_t base = d_base ? d_base[0] : 0u;
    if (base > capacity) base = capacity;
    const uint32_t count = d_count ? d_count[0] : capacity;
    const uint32_t len = min(count, capacity - base);
    // rounds of a wave: the records spread evenly over the waves, a wave's ones consecutive
    const uint32_t rounds = ceil_div(len, kSmallThreads);
    const uint32_t wave_first = wave * rounds * kWave;
    if (len == 0u) return;
    uint32_t rec_major[ITEMS], rec_minor[ITEMS], rec_pay[ITEMS], place[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        rec_major[i] = rec_minor[i] = rec_pay[i] = place[i] = 0u;
        if (i >= static_cast<int>(rounds)) continue;
        const uint32_t from = base + min(wave_first + i * kWave + lane, len - 1u);  // past the end: the last again
        rec_major[i] = major[from];
        if (minor) rec_minor[i] = minor[from];
        if (payload) rec_pay[i] = payload[from];
    }
    for (uint32_t p = 0; p < digits.count; ++p) {
        const uint32_t shift = digits.shift[p];
        const bool on_major = digits.major[p] != 0u;
        for (uint32_t k = t; k < WAVES * kSortBins; k += kSmallThreads) (&s_wave[0][0])[k] = 0u;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (i >= static_cast<int>(rounds)) continue;
            const uint32_t d = ((on_major ? rec_major[i] : rec_minor[i]) >> shift) & 0xFFu;
            place[i] = wave_rank(d, wave_first + i * kWave + lane < len, s_wave[wave]);
        }
        __syncthreads();
        uint32_t total = 0;
        if (t < kSortBins) {
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const uint32_t c = s_wave[w][t];
                s_wave[w][t] = total;
                total += c;
            }
        }
        const uint32_t start = block_exclusive_sum<kSmallThreads>(total, s_scan, nullptr);
        if (t < kSortBins) s_start[t] = start;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (i >= static_cast<int>(rounds)) continue;
            const uint32_t d = ((on_major ? rec_major[i] : rec_minor[i]) >> shift) & 0xFFu;
            place[i] += s_start[d] + s_wave[wave][d];
        }
        small_exchange<ITEMS>(rec_major, place, rounds, wave_first, len, s_stage);
        if (minor) small_exchange<ITEMS>(rec_minor, place, rounds, wave_first, len, s_stage);
        if (payload) small_exchange<ITEMS>(rec_pay, place, rounds, wave_first, len, s_stage);
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t local = wave_first + i * kWave + lane;
        if (i >= static_cast<int>(rounds) || local >= len) continue;
        major[base + local] = rec_major[i];
        if (minor) minor[base + local] = rec_minor[i];
        if (payload) payload[base + local] = rec_pay[i];
    }
}

__global__ void __launch_bounds__(256) sort_copy_kernel(const uint32_t* __restrict__ from_major,
                                                        const uint32_t* __restrict__ from_minor,
                                                        const uint32_t* __restrict__ from_pay,
                                                        uint32_t* to_major, uint32_t* to_minor,
                                                        uint32_t* to_pay, const uint32_t* ctl) {
    const uint32_t len = ctl[kCtlLen];
    const uint32_t base = ctl[kCtlBase];
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < len; i += stride) {
        to_major[base + i] = from_major[base + i];
        if (to_pay) to_pay[base + i] = from_pay[base + i];
        if (to_minor) to_minor[base + i] = from_minor[base + i];
    }
}

DigitList make_list(const SortDigit* digits, uint32_t passes) {
    DigitList list{};
    list.count = passes;
    for (uint32_t p = 0; p < passes; ++p) {
        list.major[p] = digits[p].major;
        list.shift[p] = digits[p].shift;
    }
    return list;
}

uint32_t histogram_groups(uint32_t capacity) {
    const uint32_t want = ceil_div(capacity ? capacity : 1u, 4u * kHistogramThreads);
    return want < kHistogramGroups ? want : kHistogramGroups;
}

uint32_t stream_groups(uint32_t capacity) {
    const uint32_t want = ceil_div(capacity ? capacity : 1u, 4096u);
    return want < 1024u ? want : 1024u;
}

}  // namespace

const SortNames kGenericSortNames = {"sort_prepare_kernel", "sort_histogram_kernel",
                                     "sort_pass_kernel", "sort_copy_kernel"};
const SortNames kEntrySortNames = {"entry_sort_prepare", "entry_sort_histogram",
                                   "entry_sort_pass", "entry_sort_copy"};
const SortNames kPairSortNames = {"pair_sort_prepare", "pair_sort_histogram", "pair_sort_pass",
                                  "pair_sort_copy"};

size_t sort_scratch_layout(uint32_t capacity, uint32_t passes, bool minor_lane, void* base,
                           SortScratch* out) {
    Carve carve(base);
    SortScratch s;
    const size_t words = capacity ? capacity : 1u;
    s.major = carve.take<uint32_t>(words);
    s.minor = minor_lane ? carve.take<uint32_t>(words) : nullptr;
    s.payload = carve.take<uint32_t>(words);
    s.hist = carve.take<uint32_t>(kSortMaxPasses * kSortBins);
    s.ctl = carve.take<uint32_t>(kCtlWords);
    s.max_tiles = ceil_div(words, kSortMinTile);
    s.flags = carve.take<uint32_t>(static_cast<size_t>(passes ? passes : 1u) * s.max_tiles *
                                   kSortBins);
    if (out) *out = s;
    return carve.used;
}

int sort_digits(uint32_t major_words, uint32_t minor_words, SortDigit* digits) {
    uint32_t n = 0;
    for (uint32_t w = 0; w < minor_words; ++w) digits[n++] = SortDigit{0u, 8u * w};
    for (uint32_t w = 0; w < major_words; ++w) digits[n++] = SortDigit{1u, 8u * w};
    return static_cast<int>(n);
}

int sort_prepare(hipStream_t stream, const SortScratch& s, const uint32_t* d_count,
                 const uint32_t* d_base, uint32_t capacity, const SortNames& names) {
    {
        ProfileScope scope(names.prepare, stream);
        sort_prepare_kernel<<<1, 256, 0, stream>>>(s.hist, s.ctl, d_count, d_base, capacity);
    }
    DYN_LAUNCHED("sort_prepare_kernel");
    return DYN_OK;
}

int sort_histogram(hipStream_t stream, const uint32_t* major, const uint32_t* minor,
                   const SortScratch& s, const SortDigit* digits, uint32_t passes,
                   uint32_t capacity, const SortNames& names) {
    {
        ProfileScope scope(names.histogram, stream);
        sort_histogram_kernel<<<histogram_groups(capacity), kHistogramThreads, 0, stream>>>(
            major, minor, s.hist, s.ctl, s.flags, make_list(digits, passes));
    }
    DYN_LAUNCHED("sort_histogram_kernel");
    return DYN_OK;
}

template <int ITEMS>
static int launch_passes(hipStream_t stream, uint32_t* major, uint32_t* minor, uint32_t* payload,
                         const SortScratch& s, const SortDigit* digits, uint32_t passes,
                         uint32_t capacity, const SortNames& names, uint32_t group_cap) {
    // Persistent workgroups take tiles in order (any count makes progress: a tile's look-back only
    // waits on earlier tiles, which running groups hold). The tiles of 8 keys a lane: a stream with
    // few live records takes those whatever ITEMS is.
    static_assert(ITEMS * kSortThreads >= kSortMinTile, "the look-back words are laid out for the narrowest tiling");
    const uint32_t tiles = ceil_div(capacity ? capacity : 1u, kSortMinTile);
    const uint32_t groups = tiles < group_cap ? tiles : group_cap;
    const size_t flag_stride = static_cast<size_t>(s.max_tiles) * kSortBins;
    uint32_t* src[3] = {major, minor, payload};
    uint32_t* dst[3] = {s.major, s.minor, s.payload};
    const bool carry_minor = minor != nullptr;
    for (uint32_t p = 0; p < passes; ++p) {
        const bool on_major = digits[p].major != 0;
        if (!on_major && !carry_minor) return fail(DYN_E_INVALID, "sort: minor digit without minor lane");
        uint32_t* in_sort = on_major ? src[0] : src[1];
        uint32_t* in_other = on_major ? src[1] : src[0];
        uint32_t* out_sort = on_major ? dst[0] : dst[1];
        uint32_t* out_other = on_major ? dst[1] : dst[0];
        uint32_t* flags_pass = s.flags + p * flag_stride;
        uint32_t* flags_next = (p + 1 < passes) ? s.flags + (p + 1) * flag_stride : nullptr;
        {
            ProfileScope scope(names.pass, stream);
            const PassArgs args{in_sort, carry_minor ? in_other : nullptr, src[2],
                                out_sort, carry_minor ? out_other : nullptr, dst[2],
                                s.hist + p * kSortBins, flags_pass, flags_next, s.ctl, p, digits[p].shift};
            auto launch = [&](auto kernel) { kernel<<<groups, kSortThreads, 0, stream>>>(args); };
            if (carry_minor && payload) launch(sort_pass_kernel<ITEMS, true, true>);
            else if (carry_minor) launch(sort_pass_kernel<ITEMS, true, false>);
            else launch(sort_pass_kernel<ITEMS, false, true>);
        }
        DYN_LAUNCHED("sort_pass_kernel");
        for (int l = 0; l < 3; ++l) {
            uint32_t* tmp = src[l];
            src[l] = dst[l];
            dst[l] = tmp;
        }
    }
    if (passes % 2 == 1) {
        {
            ProfileScope scope(names.copy, stream);
            sort_copy_kernel<<<stream_groups(capacity), 256, 0, stream>>>(
                s.major, s.minor, s.payload, major, minor, payload, s.ctl);
        }
        DYN_LAUNCHED("sort_copy_kernel");
    }
    return DYN_OK;
}

// ---- tiling: the autotuner's table ---------------------------------------------------------------
//
// A pass's tiling is keys per lane (8: 4096-key tiles; 16: 8192-key tiles, for streams with enough live
// records) and the cap on its persistent workgroups. The tuner times the candidates on the device for a
// capacity bucket (ceil(log2(capacity))) and keeps the fastest per (device, bucket); 16 keys a lane only
// above kNarrowBelow, where they differ from 8, and nothing up to kSortSmall, where no pass runs. Untuned
// buckets use the default: narrow tiles up to 2^21 keys (more of the chip busy on shorter streams), 1024
// groups (about four per CU).

struct SortTiling {
    uint32_t items, groups;
};

constexpr SortTiling kTilings[] = {{8u, 512u}, {8u, 1024u}, {8u, 2048u}, {16u, 512u}, {16u, 1024u}, {16u, 2048u}};
constexpr uint32_t kTilingCount = sizeof(kTilings) / sizeof(kTilings[0]);

std::mutex& tune_mutex() {
    static std::mutex m;
    return m;
}
std::map<std::pair<int, uint32_t>, SortTiling>& tune_table() {
    static std::map<std::pair<int, uint32_t>, SortTiling> t;
    return t;
}

uint32_t tune_bucket(uint32_t capacity) {
    return capacity <= 1u ? 0u : 32u - static_cast<uint32_t>(__builtin_clz(capacity - 1u));
}

SortTiling default_tiling(uint32_t capacity) {
    return SortTiling{capacity <= (1u << 21) ? 8u : 16u, 1024u};
}

SortTiling tiling_for(uint32_t capacity) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return default_tiling(capacity);
    std::lock_guard<std::mutex> lock(tune_mutex());
    const auto it = tune_table().find({device, tune_bucket(capacity)});
    return it == tune_table().end() ? default_tiling(capacity) : it->second;
}

int passes_with(hipStream_t stream, uint32_t* major, uint32_t* minor, uint32_t* payload, const SortScratch& s,
                const SortDigit* digits, uint32_t passes, uint32_t capacity, const SortNames& names,
                SortTiling t) {
    if (t.items == 8u) return launch_passes<8>(stream, major, minor, payload, s, digits, passes, capacity, names, t.groups);
    return launch_passes<16>(stream, major, minor, payload, s, digits, passes, capacity, names, t.groups);
}

int sort_small(hipStream_t stream, uint32_t* major, uint32_t* minor, uint32_t* payload, const uint32_t* d_count,
               const uint32_t* d_base, uint32_t capacity, const SortDigit* digits, uint32_t passes,
               const SortNames& names) {
    if (capacity > kSortSmall) return fail(DYN_E_INVALID, "sort: too many records for one workgroup");
    const DigitList list = make_list(digits, passes);
    {
        ProfileScope scope(names.pass, stream);
        auto launch = [&](auto kernel) {
            kernel<<<1, kSmallThreads, 0, stream>>>(major, minor, payload, d_count, d_base, capacity, list);
        };
        if (capacity <= 2u * kSmallThreads) launch(sort_small_kernel<2>);
        else if (capacity <= 4u * kSmallThreads) launch(sort_small_kernel<4>);
        else launch(sort_small_kernel<8>);
    }
    DYN_LAUNCHED("sort_small_kernel");
    return DYN_OK;
}

int sort_passes(hipStream_t stream, uint32_t* major, uint32_t* minor, uint32_t* payload,
                const SortScratch& s, const SortDigit* digits, uint32_t passes,
                uint32_t capacity, const SortNames& names) {
    return passes_with(stream, major, minor, payload, s, digits, passes, capacity, names, tiling_for(capacity));
}

namespace {

__global__ void __launch_bounds__(256) sort_tune_fill(uint32_t* major, uint32_t* minor, uint32_t* payload,
                                                      uint32_t count, uint32_t seed) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    uint32_t h = (i + seed) * 0x9E3779B1u;
    h ^= h >> 15;
    h *= 0x85EBCA77u;
    h ^= h >> 13;
    major[i] = h;
    minor[i] = h * 0xC2B2AE3Du;
    payload[i] = i;
}

}  // namespace

}  // namespace dyn

extern "C" {

uint32_t dyn_sort_units_for(uint32_t live) {
    uint64_t units = (static_cast<uint64_t>(live) + 255u) / 256u + 64u;
    if (units < 1u) units = 1u;
    if (units > 512u) units = 512u;
    return static_cast<uint32_t>(units);
}

uint32_t dyn_sort_key_words(uint32_t elements) {
    const uint32_t last = elements ? elements - 1u : 0u;
    const uint32_t bits = last ? 32u - static_cast<uint32_t>(__builtin_clz(last)) : 0u;
    uint32_t words = (bits + 7u) / 8u;
    if (words < 1u) words = 1u;
    if (words > 4u) words = 4u;
    return words;
}

size_t dyn_sort_scratch_bytes(uint32_t capacity, uint32_t digit_passes) {
    return dyn::sort_scratch_layout(capacity, digit_passes, true, nullptr, nullptr);
}

int dyn_sort_autotune(void* stream, uint32_t capacity, uint32_t digit_passes, uint32_t* items_out,
                      uint32_t* groups_out) {
    using namespace dyn;
    if (capacity == 0u || capacity > kSortMaxCapacity) return fail(DYN_E_INVALID, "dyn_sort_autotune: capacity out of range");
    if (digit_passes == 0u || digit_passes > kSortMaxPasses) {
        return fail(DYN_E_INVALID, "dyn_sort_autotune: digit_passes must be 1..8");
    }
    if (capacity <= kSortSmall) {  // sorted by one workgroup, which has no tiling
        const SortTiling t = default_tiling(capacity);
        if (items_out) *items_out = t.items;
        if (groups_out) *groups_out = t.groups;
        return DYN_OK;
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    const size_t scratch_bytes = sort_scratch_layout(capacity, digit_passes, true, nullptr, nullptr);
    std::vector<void*> owned;
    auto cleanup = [&](int rc) {
        (void)hipStreamSynchronize(st);
        for (void* p : owned) (void)hipFree(p);
        return rc;
    };
    uint32_t* lanes[3] = {nullptr, nullptr, nullptr};
    void* scratch = nullptr;
    for (auto*& lane : lanes) {
        if (hipMalloc(&lane, 4u * static_cast<size_t>(capacity)) != hipSuccess) return cleanup(fail(DYN_E_HIP, "dyn_sort_autotune: lanes"));
        owned.push_back(lane);
    }
    if (hipMalloc(&scratch, scratch_bytes) != hipSuccess) return cleanup(fail(DYN_E_HIP, "dyn_sort_autotune: scratch"));
    owned.push_back(scratch);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        return cleanup(fail(DYN_E_HIP, "dyn_sort_autotune: events"));
    }
    SortScratch s;
    sort_scratch_layout(capacity, digit_passes, true, scratch, &s);
    SortDigit digits[kSortMaxPasses];
    sort_digits(digit_passes > 4u ? 4u : digit_passes, digit_passes > 4u ? digit_passes - 4u : 0u, digits);
    const SortNames& names = kGenericSortNames;
    float best_ms = 0.0f;
    uint32_t best = kTilingCount;
    int rc = DYN_OK;
    for (uint32_t round = 0; round < 4 && rc == DYN_OK; ++round) {  // round 0 warms every variant
        for (uint32_t c = 0; c < kTilingCount && rc == DYN_OK; ++c) {
            if (kTilings[c].items > 8u && capacity <= kNarrowBelow) continue;  // it runs 8 keys a lane too
            sort_tune_fill<<<ceil_div(capacity, 256u), 256, 0, st>>>(lanes[0], lanes[1], lanes[2], capacity, round);
            rc = sort_prepare(st, s, nullptr, nullptr, capacity, names);
            if (rc == DYN_OK) rc = sort_histogram(st, lanes[0], lanes[1], s, digits, digit_passes, capacity, names);
            if (rc != DYN_OK || hipEventRecord(e0, st) != hipSuccess) break;
            rc = passes_with(st, lanes[0], lanes[1], lanes[2], s, digits, digit_passes, capacity, names, kTilings[c]);
            if (rc != DYN_OK || hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) break;
            float ms = 0.0f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            if (round > 0 && (best == kTilingCount || ms < best_ms)) {
                best_ms = ms;
                best = c;
            }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != DYN_OK) return cleanup(rc);
    if (best == kTilingCount) return cleanup(fail(DYN_E_HIP, "dyn_sort_autotune: timing failed"));
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return cleanup(fail(DYN_E_HIP, "dyn_sort_autotune: device"));
    {
        std::lock_guard<std::mutex> lock(tune_mutex());
        tune_table()[{device, tune_bucket(capacity)}] = kTilings[best];
    }
    if (items_out) *items_out = kTilings[best].items;
    if (groups_out) *groups_out = kTilings[best].groups;
    return cleanup(DYN_OK);
}

int dyn_sort_tuning_export(uint32_t* out, uint32_t capacity, uint32_t* count) {
    using namespace dyn;
    if (!count) return fail(DYN_E_INVALID, "dyn_sort_tuning_export: null count");
    std::lock_guard<std::mutex> lock(tune_mutex());
    *count = static_cast<uint32_t>(tune_table().size());
    uint32_t i = 0;
    for (const auto& kv : tune_table()) {
        if (i >= capacity || !out) break;
        out[4 * i + 0] = static_cast<uint32_t>(kv.first.first);
        out[4 * i + 1] = kv.first.second;
        out[4 * i + 2] = kv.second.items;
        out[4 * i + 3] = kv.second.groups;
        ++i;
    }
    return DYN_OK;
}

int dyn_sort_tuning_import(const uint32_t* entries, uint32_t count) {
    using namespace dyn;
    if (count && !entries) return fail(DYN_E_INVALID, "dyn_sort_tuning_import: null entries");
    for (uint32_t i = 0; i < count; ++i) {
        const SortTiling t{entries[4 * i + 2], entries[4 * i + 3]};
        bool known = false;
        for (const SortTiling& k : kTilings) known |= k.items == t.items && k.groups == t.groups;
        if (!known || entries[4 * i + 1] > 31u) return fail(DYN_E_INVALID, "dyn_sort_tuning_import: not a tiling of this build");
    }
    std::lock_guard<std::mutex> lock(tune_mutex());
    tune_table().clear();
    for (uint32_t i = 0; i < count; ++i) {
        tune_table()[{static_cast<int>(entries[4 * i]), entries[4 * i + 1]}] = SortTiling{entries[4 * i + 2], entries[4 * i + 3]};
    }
    return DYN_OK;
}

int dyn_sort_faults(uint32_t* out, int clear) {
    if (!out) return dyn::fail(DYN_E_INVALID, "dyn_sort_faults: null output");
    DYN_HIP(hipDeviceSynchronize());
    DYN_HIP(hipMemcpyFromSymbol(out, HIP_SYMBOL(dyn::g_sort_faults), sizeof(uint32_t), 0, hipMemcpyDeviceToHost));
    if (clear) {
        const uint32_t zero = 0u;
        DYN_HIP(hipMemcpyToSymbol(HIP_SYMBOL(dyn::g_sort_faults), &zero, sizeof(uint32_t), 0, hipMemcpyHostToDevice));
    }
    return DYN_OK;
}

int dyn_sort_pairs(void* stream, uint32_t* d_major, uint32_t* d_minor, uint32_t* d_payload,
                   uint32_t capacity, const uint32_t* d_count, const uint32_t* d_base,
                   uint32_t plan, uint32_t major_words, uint32_t minor_words, void* d_scratch,
                   size_t scratch_bytes) {
    using namespace dyn;
    (void)plan;
    if (major_words > 4u || minor_words > 4u) {
        return fail(DYN_E_INVALID, "dyn_sort_pairs: a key has at most 4 byte digits per word");
    }
    if (major_words + minor_words == 0u) {
        return fail(DYN_E_INVALID,
                    "dyn_sort_pairs: a sort needs at least one key digit to permute the payload");
    }
    if (!d_major || !d_minor || !d_payload || !d_scratch) {
        return fail(DYN_E_INVALID, "dyn_sort_pairs: null lane or scratch");
    }
    if (capacity > kSortMaxCapacity) {
        return fail(DYN_E_INVALID, "dyn_sort_pairs: capacity above 2^30-1 records");
    }
    const uint32_t passes = major_words + minor_words;
    SortScratch s;
    const size_t need = sort_scratch_layout(capacity, passes, true, d_scratch, &s);
    if (scratch_bytes < need) {
        return fail(DYN_E_CAPACITY, "dyn_sort_pairs: scratch smaller than dyn_sort_scratch_bytes");
    }
    SortDigit digits[kSortMaxPasses];
    sort_digits(major_words, minor_words, digits);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (capacity <= kSortSmall) {
        return sort_small(st, d_major, d_minor, d_payload, d_count, d_base, capacity, digits, passes);
    }
    DYN_TRY(sort_prepare(st, s, d_count, d_base, capacity));
    DYN_TRY(sort_histogram(st, d_major, d_minor, s, digits, passes, capacity));
    DYN_TRY(sort_passes(st, d_major, d_minor, d_payload, s, digits, passes, capacity));
    return DYN_OK;
}

}  // extern "C"

// ---- the sort with no allocation: its scratch is a file-scope device array ----------------------

namespace {

// The scratch of dyn_sort_pairs_static: one array per device (each GPU the library runs on holds
// its own copy until the process ends), large enough for 2^20 records at any digit count.
constexpr size_t kStaticScratchBytes = size_t{17} << 20;
__device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kStaticDevices = 64;
std::mutex static_mutex;
void* static_scratch[kStaticDevices] = {};

// The current device's address of `scratch`, looked up on the device's first call (the array's
// host-side name is no device address).
int static_scratch_of_device(void** out) {
    int device = 0;
    DYN_HIP(hipGetDevice(&device));
    if (device < 0 || device >= kStaticDevices) return dyn::fail(DYN_E_INVALID, "dyn_sort_pairs_static: device ordinal out of range");
    std::lock_guard<std::mutex> guard(static_mutex);
    if (!static_scratch[device]) {
        void* ptr = nullptr;
        const hipError_t rc = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (rc != hipSuccess || !ptr) return dyn::hip_fail(rc, "dyn_sort_pairs_static: address of the static scratch");
        static_scratch[device] = ptr;
    }
    *out = static_scratch[device];
    return DYN_OK;
}

}  // namespace

extern "C" {

size_t dyn_sort_static_scratch_bytes(void) { return kStaticScratchBytes; }

int dyn_sort_pairs_static(void* stream, uint32_t* d_major, uint32_t* d_minor, uint32_t* d_payload,
                          uint32_t capacity, const uint32_t* d_count, const uint32_t* d_base, uint32_t plan,
                          uint32_t major_words, uint32_t minor_words) {
    using namespace dyn;
    if (major_words > 4u || minor_words > 4u || major_words + minor_words == 0u) {
        return dyn_sort_pairs(stream, d_major, d_minor, d_payload, capacity, d_count, d_base, plan, major_words,
                              minor_words, nullptr, 0u);  // the same argument errors
    }
    // The capacities refused are those whose look-back words would not fit for tiles of 2,048 keys, as when
    // the array was sized, and not those that fit since tiles are larger: a caller's limit stays its limit.
    const uint32_t passes = major_words + minor_words;
    const size_t words = size_t{passes} * (ceil_div(capacity, 2048u) - ceil_div(capacity, kSortMinTile)) * kSortBins;
    if (capacity > kSortMaxCapacity ||
        sort_scratch_layout(capacity, passes, true, nullptr, nullptr) + 4u * words > kStaticScratchBytes) {
        return fail(DYN_E_CAPACITY, "dyn_sort_pairs_static: capacity beyond the static scratch (2^20 records)");
    }
    void* base = nullptr;
    DYN_TRY(static_scratch_of_device(&base));
    return dyn_sort_pairs(stream, d_major, d_minor, d_payload, capacity, d_count, d_base, plan, major_words,
                          minor_words, base, kStaticScratchBytes);
}

}  // extern "C"
