// Batch pair merger on the device: the same rounds as the host routine
// cgnn_compress_csr_batch (csrc/prep.cpp), with the same arrays as result.  It stands
// where the reference's optional GPU compressor stands
// (src/offline/bindings/batch_cuda.cpp:3-9, module compressgnn_batch_cuda; its
// kernels are not part of the reference tree).
//
// A round, on the sequence of all rows laid end to end (L entries; the last entry of a row carries a flag bit):
//   1. The pairs (seq[e], seq[e+1]) within the rows that occur at least min_pair_frequency times are the
//      candidates, in ascending order.
//   2. Greedy left-to-right parse of every row with all candidates.  A position is
//      "matched" if its pair is a candidate; the greedy parse takes the 1st, 3rd, 5th ...
//      position of every maximal stretch of matched positions (the last entry of a row
//      is never matched, so stretches do not cross rows): no sequential walk of a row, however long.
//   3. Candidates taken at least twice become rules, numbered in key order.
//   4. The parse is repeated with the rules only; a taken position becomes the rule, the position behind it goes.
//
// What bounds a round is how often it goes over the sequence and at what price, so each step keeps fewer positions:
//   - Only the pairs that can be candidates are looked at: in the first round all, later those with a rule of the round
//     before in them and those that could be candidates in it.  (Another pair was there before and was no candidate, and a
//     round makes no pair of old entries more frequent.)
//   - These are counted in a table by their hash alone, an upper bound of how often they occur; the counters stop at
//     min_pair_frequency, so that a pair met a thousand times costs its counter no thousand atomics one after the other.
//   - The positions that pass (one in seven of a web graph at 16) are listed in order, and their pairs
//     counted exactly in a table of keys.  The candidates are sorted, nothing else is.
//   - Both parses run over the list.  Positions taken are bits of a map, whose prefix sums move the entries
//     and the row starts.
// Sorting all pairs in every round (eight passes over 64-bit keys, run-length encoding, selection, a binary search per
// position, scans over all positions) took 1,950 us of the device for the three rounds of 325,557 rows and 3.2 million
// entries; this takes 620 us, 210 of them while the sequence still arrives (cgnn_compress_batch_feed).
//
// Timing decides where an atomic lands, never what comes of it: counts and sums are whole numbers, lists are in
// order of position or sorted, so the arrays are the same run to run and equal the host routine's.
//
// Offline work: the entry point waits for the device twice per round (the number of candidates, the new length).
#include <hipcub/hipcub.hpp>

#include <chrono>
#include <utility>

#include "common.h"

namespace cgnn {
namespace {

constexpr int64_t kMergerLimit = (int64_t)INT32_MAX - 65536;
constexpr uint32_t kLast = 0x80000000u;   // of an entry of the sequence: the last one of its row
constexpr uint64_t kEmpty = ~0ull;
constexpr int kItems = 8;
constexpr int kTile = kItems * kBlock;    // positions per workgroup
constexpr int kTileWords = kTile / 64;
constexpr int kScanBlock = 1024;
// Up to this many candidates are ranked by comparing all with all (10,821: 5 us); the radix sort's launches
// alone take 40 us, and at 16,384 the comparisons do, too.
constexpr int32_t kRankAll = 16384;

enum Scalar { kBad, kListed, kCandidates, kAdded, kTakenTotal, kArrived, kScalars = 8 };  // kArrived: three counters (Arrival)
enum Arrival { kPassed, kCounted, kTaken };

struct Merger {
    int64_t V;
    int32_t L, min_frequency, rules;   // rules: numbered before this round
    int32_t most;                      // pairs that can be candidates
    int32_t listed, candidates;        // once the host has read them
    int key_bits;                      // of one entry
    bool first;
    uint32_t *seq, *next_seq;
    int32_t *ptr, *next_ptr;
    uint8_t *active, *next_active;     // [L] of all rounds but the first
    uint32_t *filter;                  // counters by hash; the same memory as table_key
    uint32_t *frequent;                // a bit for each: it got to min_frequency
    uint64_t *words;                   // [L / 64] positions that pass the filter
    int32_t *tile;                     // [tiles] sums in front of a tile, or its last start of a stretch
    int32_t *tile_start;
    int32_t *position, *slot, *candidate;  // [listed] slot of the table; -1: the pair is no candidate
    uint64_t *table_key;
    int32_t *table_count;              // later the rank of the slot's candidate, -1: none
    uint64_t *cand_key, *sorted_key;   // [candidates] (first entry << key_bits) | second
    int32_t *cand_slot, *sorted_slot, *cand_rank;
    int32_t *use, *rule_of;            // [candidates] in order
    uint64_t *used;                    // [listed / 64] taken when all candidates were
    uint64_t *taken;                   // [L / 64] taken by a rule
    int32_t *word_sum;                 // [L / 64] taken positions of the tile in front of a word
    int32_t *children;
    int32_t *scalar;                   // [kScalars], and the counters of arrives_last, a line each
    int32_t *host, flag;               // pinned memory for the scalars and this flag behind them, or NULL
};

unsigned merger_grid(int64_t n) {
    const int64_t b = ceil_div(n, kBlock);
    return (unsigned)(b > 262144 ? 262144 : (b < 1 ? 1 : b));
}

unsigned tiles_of(int64_t n) { return (unsigned)(n < 1 ? 1 : ceil_div(n, kTile)); }

#define CGNN_GRID_LOOP(i, n) \
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (int64_t)gridDim.x * blockDim.x)

__device__ __forceinline__ int64_t ceil_div_dev(int64_t a, int64_t b) { return (a + b - 1) / b; }

__device__ __forceinline__ uint64_t pair_hash(uint64_t k) {
    k ^= k >> 33;
    k *= 0xff51afd7ed558ccdULL;
    k ^= k >> 33;
    return k * 0x9e3779b97f4a7c15ULL;
}

// Bits of a table with more than n entries.
__device__ __forceinline__ int table_bits(int32_t n) { return n <= 0 ? 1 : 32 - __clz(n); }

__device__ __forceinline__ int load_now(const int32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Exclusive sums over the workgroup.
template <int BLOCK>
__device__ __forceinline__ int block_scan(int v, int *total) {
    __shared__ int wave_sum[BLOCK / kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    int sum = v;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
        const int up = __shfl_up(sum, s, kWave);
        if (lane >= s) sum += up;
    }
    __syncthreads();
    if (lane == kWave - 1) wave_sum[wave] = sum;
    __syncthreads();
    int before = sum - v, all = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / kWave; ++w) {
        if (w < wave) before += wave_sum[w];
        all += wave_sum[w];
    }
    *total = all;
    return before;
}

// Sums of the tiles in front of every tile; returns the total.  FRESH: written by other workgroups of this launch.
template <int BLOCK, bool FRESH>
__device__ __forceinline__ int scan_tiles(int32_t *__restrict__ tile, int32_t tiles) {
    int running = 0;
    for (int32_t k0 = 0; k0 < tiles; k0 += BLOCK * kItems) {
        const int32_t k = k0 + threadIdx.x * kItems;
        int v[kItems], sum = 0, all;
#pragma unroll
        for (int u = 0; u < kItems; ++u) v[u] = k + u < tiles ? (FRESH ? load_now(tile + k + u) : tile[k + u]) : 0;
#pragma unroll
        for (int u = 0; u < kItems; ++u) sum += v[u];
        int before = running + block_scan<BLOCK>(sum, &all);
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            if (k + u < tiles) tile[k + u] = before;
            before += v[u];
        }
        running += all;
    }
    return running;
}

__global__ __launch_bounds__(kScanBlock) void merger_tile_sums_kernel(int32_t *__restrict__ tile, int32_t tiles,
                                                                      int32_t *__restrict__ total) {
    const int all = scan_tiles<kScanBlock, false>(tile, tiles);
    if (threadIdx.x == 0) *total = all;
}

// What the last workgroup to get here may do for the others instead of a launch behind them (3 to 5 us of the device and as
// much of the host; 14,530 vertices of degree 8.9 at a frequency of 4, twenty launches a round 636 us a call, sixteen 583; 14,163
// of 13 at 16 480, 456): true in that one, for all its threads.  What the others have left is past their L2s -- stored with
// store_now or added with an atomic -- and read with load_now: a release would write back the whole L2.  Arrivals at one counter come
// one after the other, some 12 ns each (1,600: 32 us for a launch of 12), so more than kFew workgroups arrive at one of
// kArrivalGroups counters first, and the last one there at the one for all.  Beyond kMany the launches behind stay.  (With the
// launches / one counter up to kFew / so: 121,075 vertices of degree 10.2 at a frequency of 4 1,234 / 1,199 / 1,181 us a call.
// 325,557 of 9.8 at 16, three quarters of whose 1,350 us are the link and the counts, take the same within 3 %, as their runs differ.)
constexpr unsigned kFew = 256, kArrivalGroups = 16, kMany = kFew * kArrivalGroups;
constexpr int kLine = 32;  // integers of a cache line
__device__ __forceinline__ void store_now(int32_t *p, int32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

__device__ __forceinline__ bool arrives_last(const Merger &m, Arrival at) {
    __shared__ bool last;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);  // of every wave: its stores have arrived
    __syncthreads();
    if (threadIdx.x == 0) {
        auto completes = [](int32_t *count, unsigned of) {
            return __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int32_t)of - 1;
        };
        const unsigned g = blockIdx.x % kArrivalGroups;
        last = (gridDim.x <= kFew || completes(m.scalar + kScalars + (at * kArrivalGroups + g) * kLine,
                                               (gridDim.x - g + kArrivalGroups - 1) / kArrivalGroups)) &&
               completes(m.scalar + kArrived + at, gridDim.x <= kFew ? gridDim.x : kArrivalGroups);
    }
    __syncthreads();
    return last;
}

// The scalars for the host (one thread), the flag last, when the others have arrived.
__device__ __forceinline__ void publish(const int32_t *scalar, int32_t *host, int32_t flag) {
    int32_t v[kScalars];
#pragma unroll
    for (int i = 0; i < kScalars; ++i) v[i] = load_now(scalar + i);
#pragma unroll
    for (int i = 0; i < kScalars; ++i) __hip_atomic_store(host + i, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __hip_atomic_store(host + kScalars, flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Tables of up to this many slots (12 MB) are cleared for as many pairs as there can be, in a launch that there is anyway; larger
// ones for as many as are listed, one in seven of a first round.
constexpr int64_t kClearedAhead = (int64_t)1 << 20;

__device__ __forceinline__ void clear_table(const Merger &m, int64_t slots) {
    CGNN_GRID_LOOP(i, slots / 2) {
        reinterpret_cast<ulonglong2 *>(m.table_key)[i] = make_ulonglong2(kEmpty, kEmpty);
        reinterpret_cast<int2 *>(m.table_count)[i] = make_int2(0, 0);
    }
}

// Row starts, where rows end (bits of `taken`, which the first round has no other use for yet) and the counters.
template <typename In>
__global__ void merger_rows_kernel(Merger m, const In *__restrict__ vlist, int64_t E) {
    CGNN_GRID_LOOP(i, m.V + 1) {
        const int64_t p = vlist[i], before = i > 0 ? (int64_t)vlist[i - 1] : 0;
        if (p < before || p > E || (i == 0 && p != 0) || (i == m.V && p != E)) m.scalar[kBad] = 1;
        m.ptr[i] = (int32_t)(p < 0 || p > E ? 0 : p);
        if (p > before && p <= E && before >= 0)
            atomicOr(reinterpret_cast<unsigned long long *>(m.taken + (p - 1) / 64), 1ull << ((p - 1) % 64));
    }
}

// Where the round begins: the counters, and scalars of this round.
__global__ void merger_begin_kernel(Merger m) {
    const int64_t counters = (int64_t)2 << table_bits(m.most), words = ((int64_t)m.L + kTile - 1) / kTile * kTileWords;
    CGNN_GRID_LOOP(i, counters / 4) reinterpret_cast<int4 *>(m.filter)[i] = make_int4(0, 0, 0, 0);
    CGNN_GRID_LOOP(i, ceil_div_dev(counters, 32)) m.frequent[i] = 0;
    if (m.first) CGNN_GRID_LOOP(i, words) m.taken[i] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        m.scalar[kCandidates] = 0;
        for (int i = 0; i < 3; ++i) m.scalar[kArrived + i] = 0;
        if (m.first) m.scalar[kBad] = 0;
    }
    if (blockIdx.x == 0 && threadIdx.x < 3 * kArrivalGroups) m.scalar[kScalars + threadIdx.x * kLine] = 0;
}

// A counter goes up unless it got to min_frequency, as far as the caller has seen.
__device__ __forceinline__ void count_pair(const Merger &m, uint64_t counter, uint32_t seen) {
    if (seen < (uint32_t)m.min_frequency && atomicAdd(m.filter + counter, 1u) == (uint32_t)m.min_frequency - 1)
        atomicOr(m.frequent + counter / 32, 1u << (counter % 32));
}

// Entries [from, from + n) of the first round's sequence, and the pairs that end there.
template <typename In>
__global__ __launch_bounds__(kBlock) void merger_feed_kernel(Merger m, const In *__restrict__ elist, int64_t from, int64_t n) {
    const int shift = 63 - table_bits(m.most);
    const int64_t i0 = from + (int64_t)blockIdx.x * kTile + threadIdx.x, end = from + n;
    uint64_t counter[kItems];
    uint32_t seen[kItems];
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const int64_t i = i0 + u * kBlock;
        counter[u] = kEmpty;
        if (i >= end) continue;
        int64_t c = elist[i], before = i > 0 ? (int64_t)elist[i - 1] : 0;
        if (c < 0 || c >= m.V) {
            m.scalar[kBad] = 1;
            c = 0;
        }
        if (before < 0 || before >= m.V) before = 0;
        const bool last = m.taken[i / 64] >> (i % 64) & 1;
        m.seq[i] = (uint32_t)c | (last ? kLast : 0);
        if (i > 0 && !(m.taken[(i - 1) / 64] >> ((i - 1) % 64) & 1))
            counter[u] = pair_hash((uint64_t)before << 32 | (uint64_t)c) >> shift;
    }
#pragma unroll
    for (int u = 0; u < kItems; ++u)
        if (counter[u] != kEmpty) seen[u] = __hip_atomic_load(m.filter + counter[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int u = 0; u < kItems; ++u)
        if (counter[u] != kEmpty) count_pair(m, counter[u], seen[u]);
}

// The pair at e, or kEmpty: none, or none that can be a candidate.
__device__ __forceinline__ uint64_t pair_at(const Merger &m, int64_t e) {
    if (e + 1 >= m.L || (!m.first && m.active[e] == 0)) return kEmpty;
    const uint32_t x = m.seq[e], y = m.seq[e + 1];
    return (x & kLast) ? kEmpty : (uint64_t)x << 32 | (y & ~kLast);
}

__global__ __launch_bounds__(kBlock) void merger_count_kernel(Merger m) {
    const int shift = 63 - table_bits(m.most);
    const int64_t e0 = (int64_t)blockIdx.x * kTile + threadIdx.x;
    uint64_t key[kItems];
    uint64_t counter[kItems];
    uint32_t seen[kItems];
#pragma unroll
    for (int u = 0; u < kItems; ++u) key[u] = pair_at(m, e0 + u * kBlock);
#pragma unroll
    for (int u = 0; u < kItems; ++u)
        if (key[u] != kEmpty) {
            counter[u] = pair_hash(key[u]) >> shift;
            seen[u] = __hip_atomic_load(m.filter + counter[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
    for (int u = 0; u < kItems; ++u)
        if (key[u] != kEmpty) count_pair(m, counter[u], seen[u]);
}

// The positions that pass, their number in front of every tile, and (`clear`) an empty table: the counters by hash, in whose
// memory it lies, have been read.
__global__ __launch_bounds__(kBlock) void merger_pass_kernel(Merger m, bool clear) {
    __shared__ int passed[kBlock / kWave];
    const int shift = 63 - table_bits(m.most);
    const int64_t e0 = (int64_t)blockIdx.x * kTile + threadIdx.x;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    uint64_t key[kItems];
    uint32_t seen[kItems];
#pragma unroll
    for (int u = 0; u < kItems; ++u) key[u] = pair_at(m, e0 + u * kBlock);
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const uint64_t counter = key[u] == kEmpty ? 0 : pair_hash(key[u]) >> shift;
        seen[u] = m.frequent[counter / 32] >> (counter % 32) & 1;
    }
    int count = 0;
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const uint64_t word = __ballot(key[u] != kEmpty && seen[u] != 0);
        if (lane == 0) m.words[(int64_t)blockIdx.x * kTileWords + u * (kBlock / kWave) + wave] = word;
        count += __popcll(word);
    }
    if (lane == 0) passed[wave] = count;
    __syncthreads();
    if (threadIdx.x == 0) {
        int all = 0;
        for (int w = 0; w < kBlock / kWave; ++w) all += passed[w];
        store_now(m.tile + blockIdx.x, all);
    }
    if (clear) clear_table(m, (int64_t)1 << table_bits(m.most));
    if (gridDim.x > kMany || !arrives_last(m, kPassed)) return;
    const int all = scan_tiles<kBlock, true>(m.tile, (int32_t)gridDim.x);
    if (threadIdx.x == 0) m.scalar[kListed] = all;
}

__global__ void merger_clear_table_kernel(Merger m) { clear_table(m, (int64_t)1 << table_bits(m.scalar[kListed])); }

// The list of positions, and how often their pairs occur.  Tables have more slots than pairs, so every probe ends.
__global__ __launch_bounds__(kBlock) void merger_collect_kernel(Merger m) {
    __shared__ int before[kTileWords];
    const uint64_t *words = m.words + (int64_t)blockIdx.x * kTileWords;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    if (wave == 0) {
        const int mine = lane < kTileWords ? __popcll(words[lane]) : 0;
        int sum = mine;
#pragma unroll
        for (int s = 1; s < kTileWords; s <<= 1) {
            const int up = __shfl_up(sum, s, kWave);
            if (lane >= s) sum += up;
        }
        if (lane < kTileWords) before[lane] = m.tile[blockIdx.x] + sum - mine;
    }
    __syncthreads();
    const int bits = table_bits(m.scalar[kListed]);
    const uint64_t mask = ((uint64_t)1 << bits) - 1;
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const int w = u * (kBlock / kWave) + wave;
        const uint64_t word = words[w];
        if (!(word >> lane & 1)) continue;
        const int64_t e = (int64_t)blockIdx.x * kTile + u * kBlock + threadIdx.x;
        const uint64_t key = (uint64_t)m.seq[e] << 32 | (m.seq[e + 1] & ~kLast);
        const int32_t k = before[w] + __popcll(word & (((uint64_t)1 << lane) - 1));
        uint64_t h = pair_hash(key) >> (64 - bits);
        for (;;) {
            uint64_t there = __hip_atomic_load(m.table_key + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (there == kEmpty) there = atomicCAS(reinterpret_cast<unsigned long long *>(m.table_key + h), kEmpty, key);
            if (there == kEmpty || there == key) break;
            h = (h + 1) & mask;
        }
        if (load_now(m.table_count + h) < m.min_frequency) atomicAdd(m.table_count + h, 1);
        m.position[k] = (int32_t)e;
        m.slot[k] = (int32_t)h;
    }
}

__global__ __launch_bounds__(kBlock) void merger_candidates_kernel(Merger m) {
    __shared__ int base;
    const int64_t slots = (int64_t)1 << table_bits(m.scalar[kListed]);
    for (int64_t t0 = (int64_t)blockIdx.x * kTile; t0 < slots; t0 += (int64_t)gridDim.x * kTile) {
        unsigned is = 0;
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int64_t i = t0 + u * kBlock + threadIdx.x;
            if (i < slots && m.table_count[i] >= m.min_frequency) is |= 1u << u;
        }
        int all;
        int j = block_scan<kBlock>(__popc(is), &all);
        if (threadIdx.x == 0) base = all > 0 ? atomicAdd(m.scalar + kCandidates, all) : 0;
        __syncthreads();
        j += base;
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int64_t i = t0 + u * kBlock + threadIdx.x;
            if (is >> u & 1) {
                const uint64_t key = m.table_key[i];
                m.cand_key[j] = (key >> 32) << m.key_bits | (uint32_t)key;
                m.cand_slot[j] = (int32_t)i;
                m.cand_rank[j++] = 0;
            } else if (i < slots) {
                m.table_count[i] = -1;
            }
        }
        __syncthreads();
    }
    if (m.host != nullptr && gridDim.x <= kMany && arrives_last(m, kCounted) && threadIdx.x == 0) publish(m.scalar, m.host, m.flag);
}

// Ranks of a few candidates: a workgroup compares kBlock of them with kBlock others.
__global__ __launch_bounds__(kBlock) void merger_rank_kernel(Merger m) {
    __shared__ uint64_t other[kBlock];
    const int32_t i = blockIdx.x * kBlock + threadIdx.x, j = blockIdx.y * kBlock + threadIdx.x;
    other[threadIdx.x] = j < m.candidates ? m.cand_key[j] : kEmpty;
    __syncthreads();
    if (i >= m.candidates) return;
    const uint64_t key = m.cand_key[i];
    int smaller = 0;
#pragma unroll 8
    for (int t = 0; t < kBlock; ++t) smaller += other[t] < key;
    if (smaller > 0) atomicAdd(m.cand_rank + i, smaller);
}

// The candidates take their places; none is used twice yet, and nothing is taken.
__global__ void merger_place_kernel(Merger m) {
    const bool ranked = m.candidates <= kRankAll;
    const int64_t words = ((int64_t)m.L + kTile - 1) / kTile * kTileWords, n = m.candidates > words ? m.candidates : words;
    CGNN_GRID_LOOP(i, n) {
        if (i < words) m.taken[i] = 0;
        if (i < m.candidates) {
            const int32_t r = ranked ? m.cand_rank[i] : (int32_t)i;
            if (ranked) m.sorted_key[r] = m.cand_key[i];
            m.table_count[ranked ? m.cand_slot[i] : m.sorted_slot[i]] = r;
            m.rule_of[i] = 0;
        }
    }
}

// A parse takes the list a tile per workgroup and 64 positions per wave and step.
__device__ __forceinline__ int32_t wave_begin() {
    return blockIdx.x * kTile + threadIdx.x / kWave * (kItems * kWave);
}

struct Matches {
    int32_t by[kItems], at[kItems];  // candidate or rule (-1: none), position
    uint64_t starts[kItems];         // of a stretch
    int32_t last;                    // the last one of the wave, -1: none
};

// Which positions are matched (RULES: by the rules only; FIND: the candidates are still in the table).
template <bool RULES, bool FIND>
__device__ __forceinline__ Matches matches(const Merger &m, int32_t k0, int lane) {
    auto matched_by = [&](int32_t k) {
        const int32_t c = FIND ? m.table_count[m.slot[k]] : m.candidate[k];
        return RULES && c >= 0 ? m.rule_of[c] : c;
    };
    Matches a;
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const int32_t k = k0 + u * kWave + lane;
        a.by[u] = k < m.listed ? matched_by(k) : -1;
        a.at[u] = k < m.listed ? m.position[k] : -1;
    }
    // a stretch goes on where the position in front is matched, too
    int32_t before = k0 > 0 && k0 < m.listed && matched_by(k0 - 1) >= 0 ? m.position[k0 - 1] : -2;
    a.last = -1;
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const int32_t mine = a.by[u] >= 0 ? a.at[u] : -2;
        const int32_t up = __shfl_up(mine, 1, kWave);
        a.starts[u] = __ballot(a.by[u] >= 0 && (lane == 0 ? before : up) != mine - 1);
        before = __shfl(mine, kWave - 1, kWave);
        if (a.starts[u] != 0) a.last = k0 + u * kWave + 63 - __clzll(a.starts[u]);
    }
    return a;
}

// First half of a parse: the last start of a stretch in every tile.
template <bool RULES>
__global__ __launch_bounds__(kBlock) void merger_match_kernel(Merger m) {
    __shared__ int32_t wave_start[kBlock / kWave];
    const int lane = threadIdx.x % kWave;
    const int32_t k0 = wave_begin();
    const Matches a = matches<RULES, !RULES>(m, k0, lane);
    if (!RULES)
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int32_t k = k0 + u * kWave + lane;
            if (k < m.listed) m.candidate[k] = a.by[u];
        }
    if (lane == 0) wave_start[threadIdx.x / kWave] = a.last;
    __syncthreads();
    if (threadIdx.x == 0) {
        int32_t last = -1;
        for (int w = 0; w < kBlock / kWave; ++w) last = max(last, wave_start[w]);
        m.tile_start[blockIdx.x] = last;
    }
}

// Second half: every other position of a stretch is taken.  Without RULES it leaves its name as a use of the candidate
// (any of them may stay; merger_again_kernel finds out whether there are two); with RULES the rule takes its
// place in the sequence.
template <bool RULES>
__global__ __launch_bounds__(kBlock) void merger_take_kernel(Merger m) {
    __shared__ int32_t wave_start[kBlock / kWave], carried;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int32_t k0 = wave_begin();
    const Matches a = matches<RULES, false>(m, k0, lane);
    if (lane == 0) wave_start[wave] = a.last;
    if (wave == 0) {  // the last start in front of the tile
        int32_t found = -1;
        for (int32_t b = (int32_t)blockIdx.x; b > 0 && found < 0; b -= kWave) {
            const int32_t s = b - 1 - lane >= 0 ? m.tile_start[b - 1 - lane] : -1;
            const uint64_t any = __ballot(s >= 0);
            if (any != 0) found = __shfl(s, __ffsll((unsigned long long)any) - 1, kWave);
        }
        if (lane == 0) carried = found;
    }
    __syncthreads();
    int32_t last = carried;
    for (int w = 0; w < wave; ++w) last = max(last, wave_start[w]);
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const int32_t base = k0 + u * kWave;
        const uint64_t here = a.starts[u] & (~0ull >> (63 - lane));
        const int32_t start = here != 0 ? base + 63 - __clzll(here) : last;
        if (a.starts[u] != 0) last = base + 63 - __clzll(a.starts[u]);
        const bool taken = a.by[u] >= 0 && ((base + lane - start) & 1) == 0;
        if (!RULES) {
            const uint64_t word = __ballot(taken);
            if (lane == 0 && base < m.listed) m.used[base / 64] = word;
            if (taken) m.use[a.by[u]] = base + lane;
        } else if (taken) {
            atomicOr(reinterpret_cast<unsigned long long *>(m.taken + a.at[u] / 64), 1ull << (a.at[u] % 64));
            m.seq[a.at[u]] = (uint32_t)a.by[u] | (m.seq[a.at[u] + 1] & kLast);  // the entry behind it is not taken
        }
    }
}

// A position whose candidate has the name of another use: the candidate becomes a rule.  Counting the uses with
// atomics took 42 us for the 305,000 of a web graph, because a few candidates have most of them; the names and this take 12.
__global__ __launch_bounds__(kBlock) void merger_again_kernel(Merger m) {
    const int32_t k0 = wave_begin() + threadIdx.x % kWave;
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const int32_t k = k0 + u * kWave;
        if (k >= m.listed || !(m.used[k / 64] >> (k % 64) & 1)) continue;
        const int32_t c = m.candidate[k];
        if (m.use[c] != k) m.rule_of[c] = 1;
    }
}

__global__ __launch_bounds__(kBlock) void merger_kept_kernel(Merger m) {
    const int32_t c0 = (blockIdx.x * kBlock + threadIdx.x) * kItems;
    int kept = 0, all;
#pragma unroll
    for (int u = 0; u < kItems; ++u) kept += c0 + u < m.candidates ? m.rule_of[c0 + u] : 0;
    block_scan<kBlock>(kept, &all);
    if (threadIdx.x == 0) m.tile[blockIdx.x] = all;
}

// Numbers of the new rules, and their children: kItems candidates a thread.  ALONE: one workgroup has them all; otherwise
// `tile` holds the sums of the workgroups in front.
template <int BLOCK, bool ALONE>
__global__ __launch_bounds__(BLOCK) void merger_rules_kernel(Merger m) {
    const int32_t c0 = (blockIdx.x * BLOCK + threadIdx.x) * kItems;
    int kept[kItems], sum = 0, all;
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        kept[u] = c0 + u < m.candidates ? m.rule_of[c0 + u] : 0;
        sum += kept[u];
    }
    int64_t r = m.rules + (ALONE ? 0 : m.tile[blockIdx.x]) + block_scan<BLOCK>(sum, &all);
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        if (c0 + u >= m.candidates) break;
        m.rule_of[c0 + u] = kept[u] ? (int32_t)(m.V + r) : -1;
        if (!kept[u]) continue;
        const uint64_t key = m.sorted_key[c0 + u];
        m.children[2 * r] = (int32_t)(key >> m.key_bits);
        m.children[2 * r + 1] = (int32_t)(key & (((uint64_t)1 << m.key_bits) - 1));
        ++r;
    }
    if (ALONE && threadIdx.x == 0) m.scalar[kAdded] = all;
}

// Taken positions of the tile in front of every word of the map, those in front of every tile, and all of them: with it the
// host knows the new length, while the entries still move.
__global__ __launch_bounds__(kBlock) void merger_taken_sums_kernel(Merger m, int64_t words) {
    const int64_t w = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int count = w < words ? __popcll(m.taken[w]) : 0, lane = threadIdx.x % kTileWords;
    int sum = count;
#pragma unroll
    for (int s = 1; s < kTileWords; s <<= 1) {
        const int up = __shfl_up(sum, s, kTileWords);
        if (lane >= s) sum += up;
    }
    if (w < words) {
        m.word_sum[w] = sum - count;
        if (lane == kTileWords - 1) store_now(m.tile + w / kTileWords, sum);
    }
    if (gridDim.x > kMany || !arrives_last(m, kTaken)) return;
    const int all = scan_tiles<kBlock, true>(m.tile, (int32_t)(words / kTileWords));
    if (threadIdx.x == 0) {
        store_now(m.scalar + kTakenTotal, all);
        __builtin_amdgcn_s_waitcnt(0);
        if (m.host != nullptr) publish(m.scalar, m.host, m.flag);
    }
}

// Where position e goes: to the left by the taken ones in front of it.
__device__ __forceinline__ int32_t moved(const Merger &m, int32_t e) {
    const uint64_t below = m.taken[e / 64] & (((uint64_t)1 << (e % 64)) - 1);
    return e - m.tile[e / kTile] - m.word_sum[e / 64] - __popcll(below);
}

// A wave per kItems words of the map: a word is the same for all lanes.
__global__ __launch_bounds__(kBlock) void merger_move_kernel(Merger m) {
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int64_t t0 = (int64_t)blockIdx.x * kTile;
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const int64_t v = t0 + u * kBlock + threadIdx.x;
        if (v <= m.V) {
            const int32_t p = m.ptr[v];
            m.next_ptr[v] = p < m.L ? moved(m, p) : m.L - m.scalar[kTakenTotal];
        }
    }
    if (t0 < m.L) {
        const int64_t w0 = blockIdx.x * kTileWords + wave * kItems;
        const int32_t left = m.tile[blockIdx.x];
        uint32_t entry[kItems];
        uint64_t word[kItems], passed[kItems];
        int32_t sum[kItems];
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int64_t e = (w0 + u) * 64 + lane;
            entry[u] = e < m.L ? m.seq[e] : 0;
            word[u] = m.taken[w0 + u];
            passed[u] = m.words[w0 + u];
            sum[u] = m.word_sum[w0 + u];
        }
        bool behind = w0 > 0 && m.taken[w0 - 1] >> 63;                       // the position in front is taken
        const bool next = (w0 + kItems) * 64 < m.L && (m.taken[w0 + kItems] & 1);  // the first behind these words
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int64_t e = (w0 + u) * 64 + lane;
            const uint64_t gone = word[u] << 1 | (behind ? 1 : 0);
            behind = word[u] >> 63;
            if (e >= m.L || (gone >> lane & 1)) continue;
            const uint64_t follows = word[u] >> 1 | (uint64_t)(u + 1 < kItems ? word[u + 1 < kItems ? u + 1 : u] & 1 : next) << 63;
            const int32_t to = (int32_t)e - left - sum[u] - __popcll(word[u] & (((uint64_t)1 << lane) - 1));
            // what can be a candidate next: a pair with a rule of this round in it, or one that passed the filter
            m.next_seq[to] = entry[u];
            m.next_active[to] = !(entry[u] & kLast) && ((word[u] | follows | passed[u]) >> lane & 1);
        }
    }
}

__global__ void merger_publish_kernel(const int32_t *scalar, int32_t *host, int32_t flag) { publish(scalar, host, flag); }

// out_ptr = [row starts | starts of the rule rows], out_col = [rows | children of the rules].
__global__ void merger_finish_kernel(const int32_t *__restrict__ ptr, const uint32_t *__restrict__ seq,
                                     const int32_t *__restrict__ children, int64_t V, int64_t R, int64_t L,
                                     int32_t *__restrict__ out_ptr, int32_t *__restrict__ out_col) {
    const int64_t n = L + 2 * R > V + R + 1 ? L + 2 * R : V + R + 1;
    CGNN_GRID_LOOP(i, n) {
        if (i <= V) out_ptr[i] = ptr[i];
        else if (i <= V + R) out_ptr[i] = (int32_t)(L + 2 * (i - V));
        if (i < L) out_col[i] = (int32_t)(seq[i] & ~kLast);
        else if (i < L + 2 * R) out_col[i] = children[i - L];
    }
}

struct MergerWorkspace {
    size_t seq[2], ptr[2], active[2], table_key, table_count, frequent, words, used, taken, word_sum, tile, tile_start, position,
        slot, candidate, cand_key, sorted_key, cand_slot, sorted_slot, cand_rank, use, rule_of, children, scalars, temp,
        temp_bytes, total;
};

int bits_of(int64_t n) {  // of the numbers up to n
    int bits = 1;
    while ((n >> bits) > 0) ++bits;
    return bits;
}

MergerWorkspace merger_workspace(int64_t V, int64_t E) {
    MergerWorkspace w{};
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += align_up(bytes > 0 ? bytes : 1, 256);
        return here;
    };
    const size_t n = (size_t)(E > 0 ? E : 1), tiles = tiles_of(E > V ? E : V + 1), words = tiles * kTileWords, c = n / 3 + 1;
    const size_t slots = (size_t)1 << bits_of((int64_t)n);
    for (auto &s : w.seq) s = take(n * 4);
    for (auto &p : w.ptr) p = take((size_t)(V + 1) * 4);
    for (auto &s : w.active) s = take(n);
    w.table_key = take(slots * 8);  // also the counters by hash, twice as many
    w.table_count = take(slots * 4);
    w.frequent = take(slots / 4 + 8);
    w.words = take(words * 8);
    w.used = take(words * 8);
    w.taken = take(words * 8);
    w.word_sum = take(words * 4);
    w.tile = take(tiles * 4);
    w.tile_start = take(tiles * 4);
    w.position = take(n * 4);
    w.slot = take(n * 4);
    w.candidate = take(n * 4);
    w.cand_key = take(c * 8);
    w.sorted_key = take(c * 8);
    for (auto *a : {&w.cand_slot, &w.sorted_slot, &w.cand_rank, &w.use, &w.rule_of}) *a = take(c * 4);
    w.children = take(n * 4);
    w.scalars = take((kScalars + 3 * kArrivalGroups * kLine) * 4);
    hipcub::DeviceRadixSort::SortPairs(nullptr, w.temp_bytes, (const uint64_t *)nullptr, (uint64_t *)nullptr,
                                       (const int32_t *)nullptr, (int32_t *)nullptr, (int)c, 0, 64, 0);
    w.temp = take(w.temp_bytes);
    w.total = at;
    return w;
}

int merger_fail(hipError_t e, const char *what) {
    set_error("cgnn_compress_csr_batch_device: %s: %s", what, hipGetErrorString(e));
    return CGNN_ELAUNCH;
}

Merger merger_of(int64_t V, int64_t E, int min_pair_frequency, const MergerWorkspace &w, void *workspace) {
    char *base = static_cast<char *>(workspace);
    auto i32 = [&](size_t off) { return reinterpret_cast<int32_t *>(base + off); };
    auto u32 = [&](size_t off) { return reinterpret_cast<uint32_t *>(base + off); };
    auto u64 = [&](size_t off) { return reinterpret_cast<uint64_t *>(base + off); };
    auto u8 = [&](size_t off) { return reinterpret_cast<uint8_t *>(base + off); };
    Merger m{};
    m.V = V;
    m.L = (int32_t)E;
    m.min_frequency = min_pair_frequency;
    m.first = true;
    m.most = (int32_t)E;
    m.seq = u32(w.seq[0]), m.next_seq = u32(w.seq[1]);
    m.ptr = i32(w.ptr[0]), m.next_ptr = i32(w.ptr[1]);
    m.active = u8(w.active[0]), m.next_active = u8(w.active[1]);
    m.table_key = u64(w.table_key), m.table_count = i32(w.table_count);
    m.filter = u32(w.table_key), m.frequent = u32(w.frequent);
    m.words = u64(w.words), m.used = u64(w.used), m.taken = u64(w.taken), m.word_sum = i32(w.word_sum);
    m.tile = i32(w.tile), m.tile_start = i32(w.tile_start);
    m.position = i32(w.position), m.slot = i32(w.slot), m.candidate = i32(w.candidate);
    m.cand_key = u64(w.cand_key), m.sorted_key = u64(w.sorted_key);
    m.cand_slot = i32(w.cand_slot), m.sorted_slot = i32(w.sorted_slot), m.cand_rank = i32(w.cand_rank);
    m.use = i32(w.use), m.rule_of = i32(w.rule_of), m.children = i32(w.children), m.scalar = i32(w.scalars);
    return m;
}

int merger_check(int64_t V, int64_t E, const void *vlist, const void *elist, int min_pair_frequency, const void *workspace,
                 size_t workspace_bytes, MergerWorkspace *w) {
    CGNN_REQUIRE(V >= 0 && E >= 0 && V < kMergerLimit && E < kMergerLimit,
                 "cgnn_compress_csr_batch_device: V and E must be in [0, 2^31 - 65536)");
    CGNN_REQUIRE(min_pair_frequency >= 3, "cgnn_compress_csr_batch_device: min_pair_frequency must be at least 3");
    CGNN_REQUIRE(vlist && (E == 0 || elist), "cgnn_compress_csr_batch_device: null array");
    *w = merger_workspace(V, E);
    if (workspace == nullptr || workspace_bytes < w->total) {
        set_error("cgnn_compress_csr_batch_device: workspace of %zu bytes needed, %zu given", w->total, workspace_bytes);
        return CGNN_EWORKSPACE;
    }
    return CGNN_OK;
}

// Launches that depend on a count the host has not read cover the most it can be.
void launch_begin(const Merger &m, hipStream_t stream) {
    hipLaunchKernelGGL(merger_begin_kernel, dim3(merger_grid(((int64_t)2 << bits_of(m.most)) / 4)), dim3(kBlock), 0, stream, m);
}

template <typename In>
int merger_rows(int64_t V, int64_t E, const In *vlist, int min_pair_frequency, void *workspace, size_t workspace_bytes,
                hipStream_t stream) {
    MergerWorkspace w;
    const int rc = merger_check(V, E, vlist, vlist, min_pair_frequency, workspace, workspace_bytes, &w);
    if (rc != CGNN_OK) return rc;
    const Merger m = merger_of(V, E, min_pair_frequency, w, workspace);
    launch_begin(m, stream);
    hipLaunchKernelGGL(merger_rows_kernel<In>, dim3(merger_grid(V + 1)), dim3(kBlock), 0, stream, m, vlist, E);
    return check_launch("compress_csr_batch_rows");
}

template <typename In>
int merger_feed(int64_t V, int64_t E, const In *elist, int64_t from, int64_t n, int min_pair_frequency, void *workspace,
                size_t workspace_bytes, hipStream_t stream) {
    MergerWorkspace w;
    const int rc = merger_check(V, E, elist, elist, min_pair_frequency, workspace, workspace_bytes, &w);
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(from >= 0 && n >= 0 && from + n <= E, "cgnn_compress_csr_batch_device: entries outside [0, E)");
    if (n == 0) return CGNN_OK;
    const Merger m = merger_of(V, E, min_pair_frequency, w, workspace);
    hipLaunchKernelGGL(merger_feed_kernel<In>, dim3(tiles_of(n)), dim3(kBlock), 0, stream, m, elist, from, n);
    return check_launch("compress_csr_batch_feed");
}

// The rounds, once all entries were fed.  `pinned`: kScalars + 1 integers of pinned host memory for what the host
// reads, or NULL.
int merger_rounds(int64_t V, int64_t E, int rounds, int min_pair_frequency, int32_t *out_ptr, int32_t *out_col,
                  int64_t *host_summary, int32_t *pinned, void *workspace, size_t workspace_bytes, hipStream_t stream) {
    CGNN_REQUIRE(rounds >= 1, "cgnn_compress_csr_batch_device: rounds must be positive");
    CGNN_REQUIRE(host_summary, "cgnn_compress_csr_batch_device: null array");
    MergerWorkspace w;
    const int rc = merger_check(V, E, out_ptr, out_col, min_pair_frequency, workspace, workspace_bytes, &w);
    if (rc != CGNN_OK) return rc;
    Merger m = merger_of(V, E, min_pair_frequency, w, workspace);
    const dim3 block(kBlock);
    int32_t reads = 0, host[kScalars + 1];
    if (pinned != nullptr) pinned[kScalars] = 0;
    m.host = pinned;
    // What the host needs is written, by the launch that has it last, to memory that it looks at for a while, which costs it a
    // few us; a copy and a wait cost it 40.  The launch is given the number of the read as its flag (m.flag).
    auto read = [&]() -> hipError_t {
        if (pinned == nullptr) {
            hipError_t e = hipMemcpyAsync(host, m.scalar, kScalars * sizeof(int32_t), hipMemcpyDeviceToHost, stream);
            return e == hipSuccess ? hipStreamSynchronize(stream) : e;
        }
        const auto patience = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
        while (__atomic_load_n(pinned + kScalars, __ATOMIC_ACQUIRE) != reads)
            if (std::chrono::steady_clock::now() > patience) {
                const hipError_t e = hipStreamSynchronize(stream);
                if (e != hipSuccess) return e;
                if (__atomic_load_n(pinned + kScalars, __ATOMIC_ACQUIRE) != reads) return hipErrorUnknown;
                break;
            }
        for (int i = 0; i < kScalars; ++i) host[i] = pinned[i];
        return hipSuccess;
    };
    auto publish_now = [&] {
        if (pinned != nullptr) hipLaunchKernelGGL(merger_publish_kernel, dim3(1), dim3(1), 0, stream, m.scalar, pinned, m.flag);
    };
    const int32_t all_tiles = (int32_t)tiles_of(E > V ? E : V + 1);
    hipError_t err = hipSuccess;
    bool checked = false;  // the input check is read with the first counts
    int64_t R = 0;
    for (int round = 0; round < rounds && m.L > 1; ++round) {
        const int32_t tiles = (int32_t)tiles_of(m.L);
        const dim3 grid((unsigned)tiles);
        m.key_bits = bits_of(V + R);
        m.rules = (int32_t)R;
        if (round > 0) {
            launch_begin(m, stream);
            hipLaunchKernelGGL(merger_count_kernel, grid, block, 0, stream, m);
        }
        const int64_t slots = (int64_t)1 << bits_of(m.most);
        const bool clear_here = slots <= kClearedAhead;
        hipLaunchKernelGGL(merger_pass_kernel, grid, block, 0, stream, m, clear_here);
        if (grid.x > kMany)
            hipLaunchKernelGGL(merger_tile_sums_kernel, dim3(1), dim3(kScanBlock), 0, stream, m.tile, tiles, m.scalar + kListed);
        if (!clear_here) hipLaunchKernelGGL(merger_clear_table_kernel, dim3(merger_grid(slots / 2)), block, 0, stream, m);
        hipLaunchKernelGGL(merger_collect_kernel, grid, block, 0, stream, m);
        m.flag = ++reads;
        const dim3 table(tiles_of(slots));
        hipLaunchKernelGGL(merger_candidates_kernel, table, block, 0, stream, m);
        if (table.x > kMany) publish_now();
        if ((err = read()) != hipSuccess) return merger_fail(err, "reading the candidate count");
        if (!checked && host[kBad])
            return fail(CGNN_EINVAL, "cgnn_compress_csr_batch_device: malformed CSR (row starts or columns out of range)");
        checked = true;
        m.listed = host[kListed], m.candidates = host[kCandidates];
        if (m.candidates == 0) break;
        if (m.candidates <= kRankAll) {
            const unsigned side = (unsigned)ceil_div(m.candidates, kBlock);
            hipLaunchKernelGGL(merger_rank_kernel, dim3(side, side), block, 0, stream, m);
        } else {
            size_t tb = w.temp_bytes;
            err = hipcub::DeviceRadixSort::SortPairs(static_cast<char *>(workspace) + w.temp, tb, m.cand_key, m.sorted_key,
                                                     m.cand_slot, m.sorted_slot, m.candidates, 0, 2 * m.key_bits, stream);
            if (err != hipSuccess) return merger_fail(err, "sort");
        }
        const int64_t words = (int64_t)tiles * kTileWords;
        const dim3 list(tiles_of(m.listed)), rules(tiles_of(m.candidates));
        const int64_t places = m.candidates > words ? m.candidates : words;
        hipLaunchKernelGGL(merger_place_kernel, dim3(merger_grid(places)), block, 0, stream, m);
        hipLaunchKernelGGL(merger_match_kernel<false>, list, block, 0, stream, m);
        hipLaunchKernelGGL(merger_take_kernel<false>, list, block, 0, stream, m);
        hipLaunchKernelGGL(merger_again_kernel, list, block, 0, stream, m);
        if (m.candidates <= kScanBlock * kItems) {  // a step of one workgroup costs less than three launches
            hipLaunchKernelGGL((merger_rules_kernel<kScanBlock, true>), dim3(1), dim3(kScanBlock), 0, stream, m);
        } else {
            hipLaunchKernelGGL(merger_kept_kernel, rules, block, 0, stream, m);
            hipLaunchKernelGGL(merger_tile_sums_kernel, dim3(1), dim3(kScanBlock), 0, stream, m.tile, (int32_t)rules.x,
                               m.scalar + kAdded);
            hipLaunchKernelGGL((merger_rules_kernel<kBlock, false>), rules, block, 0, stream, m);
        }
        hipLaunchKernelGGL(merger_match_kernel<true>, list, block, 0, stream, m);
        hipLaunchKernelGGL(merger_take_kernel<true>, list, block, 0, stream, m);
        m.flag = ++reads;
        const dim3 maps((unsigned)ceil_div(words, kBlock));
        hipLaunchKernelGGL(merger_taken_sums_kernel, maps, block, 0, stream, m, words);
        if (maps.x > kMany) {
            hipLaunchKernelGGL(merger_tile_sums_kernel, dim3(1), dim3(kScanBlock), 0, stream, m.tile, tiles, m.scalar + kTakenTotal);
            publish_now();
        }
        hipLaunchKernelGGL(merger_move_kernel, dim3((unsigned)all_tiles), block, 0, stream, m);
        if ((err = read()) != hipSuccess) return merger_fail(err, "reading the new length");
        const int32_t added = host[kAdded];
        if (added == 0) break;  // and nothing was taken
        if (V + R + added >= kMergerLimit) {
            hipStreamSynchronize(stream);  // the entries still move
            return fail(CGNN_EUNSUPPORTED, "cgnn_compress_csr_batch_device: node ids exceed int32");
        }
        std::swap(m.seq, m.next_seq);
        std::swap(m.ptr, m.next_ptr);
        std::swap(m.active, m.next_active);
        // at most the pairs around every new rule, and those listed before
        const int64_t most = 2 * (int64_t)host[kTakenTotal] + m.listed;
        m.L -= host[kTakenTotal];
        m.most = (int32_t)(most < m.L ? most : m.L);
        m.first = false;
        R += added;
    }
    if (!checked) {
        m.flag = ++reads;
        publish_now();
        if ((err = read()) != hipSuccess) return merger_fail(err, "reading the input check");
        if (host[kBad])
            return fail(CGNN_EINVAL, "cgnn_compress_csr_batch_device: malformed CSR (row starts or columns out of range)");
    }
    const int64_t L = m.L;
    hipLaunchKernelGGL(merger_finish_kernel, dim3(merger_grid(L + 2 * R > V + R + 1 ? L + 2 * R : V + R + 1)), block, 0,
                       stream, m.ptr, m.seq, m.children, V, R, L, out_ptr, out_col);
    host_summary[0] = R;
    host_summary[1] = L + 2 * R;
    return check_launch("compress_csr_batch_device");
}

}  // namespace
}  // namespace cgnn

using namespace cgnn;

extern "C" size_t cgnn_compress_batch_workspace_bytes(int64_t V, int64_t E) {
    if (V < 0 || E < 0 || V >= kMergerLimit || E >= kMergerLimit) return 0;
    return merger_workspace(V, E).total;
}

extern "C" int cgnn_compress_csr_batch_device(int64_t V, int64_t E, const int64_t *vlist, const int64_t *elist,
                                              int rounds, int min_pair_frequency, int32_t *out_ptr,
                                              int32_t *out_col, int64_t *host_summary, void *workspace,
                                              size_t workspace_bytes, cgnn_stream_t stream) {
    CGNN_REQUIRE(out_ptr && host_summary && (E == 0 || out_col), "cgnn_compress_csr_batch_device: null array");
    int rc = merger_rows(V, E, vlist, min_pair_frequency, workspace, workspace_bytes, stream);
    if (rc == CGNN_OK && E > 0) rc = merger_feed(V, E, elist, 0, E, min_pair_frequency, workspace, workspace_bytes, stream);
    if (rc == CGNN_OK)
        rc = merger_rounds(V, E, rounds, min_pair_frequency, out_ptr, out_col, host_summary, nullptr, workspace, workspace_bytes,
                           stream);
    if (rc != CGNN_OK) return rc;
    const hipError_t err = hipStreamSynchronize(stream);
    return err == hipSuccess ? CGNN_OK : merger_fail(err, "finishing");
}

extern "C" int cgnn_compress_batch_rows(int64_t V, int64_t E, const int32_t *vlist, int min_pair_frequency, void *workspace,
                                        size_t workspace_bytes, cgnn_stream_t stream) {
    return merger_rows(V, E, vlist, min_pair_frequency, workspace, workspace_bytes, stream);
}

extern "C" int cgnn_compress_batch_feed(int64_t V, int64_t E, const int32_t *elist, int64_t from, int64_t n,
                                        int min_pair_frequency, void *workspace, size_t workspace_bytes,
                                        cgnn_stream_t stream) {
    return merger_feed(V, E, elist, from, n, min_pair_frequency, workspace, workspace_bytes, stream);
}

extern "C" int cgnn_compress_batch_rounds(int64_t V, int64_t E, int rounds, int min_pair_frequency, int32_t *out_ptr,
                                          int32_t *out_col, int64_t *host_summary, int32_t *pinned, void *workspace,
                                          size_t workspace_bytes, cgnn_stream_t stream) {
    return merger_rounds(V, E, rounds, min_pair_frequency, out_ptr, out_col, host_summary, pinned, workspace, workspace_bytes,
                         stream);
}
