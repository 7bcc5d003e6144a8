// Neighbour sampling over a compressed graph on the device: the work of the reference's CPU
// module compressgnn_sample (src/sample/csrc/neighbor_sample.h:27-131 with
// src/sample/csrc/storage_api.h:6-118; the plain-CSC form :134-211 is the case without rules).
//
// One layer of sampling is four steps, each an entry point here:
//   count    a wave per frontier vertex: how many neighbours the vertex contributes (all of
//            them when the fan-out covers its degree, else the fan-out);
//   (prefix sums of the counts: cgnn_exclusive_sum_i32)
//   fill     a wave per frontier vertex writes its neighbours: the whole expanded in-list in the
//            reference's order (v2v entries, then the r2v entries of the rules reached from the
//            vertex in breadth-first order), or the neighbours at `fan-out` distinct random
//            positions of the expanded list (the reference's selection loop, with positions
//            resolved by descending through the rule levels with the expanded degrees);
//   relabel  local numbers for the neighbours: a vertex seen before keeps its number, new ones
//            are numbered in the order of their first occurrence, as the reference's hash map
//            does; here with a table over all vertices, integer atomic minima and a prefix sum,
//            so the numbering does not depend on timing.
//
// The breadth-first order of the full list is produced without a queue: a depth-first walk
// visits the rules of one depth in the same left-to-right order as the breadth-first walk
// does, so a first walk adds up the r2v sizes per depth and a second walk writes every rule's
// entries at (entries of shallower depths) + (entries of rules of its depth visited so far).
//
// Random positions come from a counter-based generator (a draw depends on the seed, the layer,
// the position of the frontier vertex among the samples and the step of the selection loop),
// so a sample does not depend on scheduling.  The reference draws from torch's sequential CPU
// generator; the streams differ by construction, everything downstream of a stream is the same.
//
// A call whose fan-outs bound every layer (cgnn_sample_layers) goes without the sizes in between: the neighbours of
// frontier vertex i stand in slots i * fan-out ..., whose order is the order of the list, so that nothing is summed up
// before they are drawn; the sizes stay on the device, every launch covers the most there can be, and the
// host reads once, when the outputs have to be allocated.  One mini-batch of 1,024 seeds with fan-outs 25 and 10
// took 47 launches and four host reads (256 us) layer by layer; it takes six and one (57 us);
// 16,384 seeds with 25 and 15 went from 384 to 93 us, most of it the chains of loads through the rules.
#include "common.h"

namespace cgnn {

size_t occupancy_scan_bytes(int64_t n);
int occupancy_scan(const int32_t *in, int64_t n, int32_t *out, void *scratch, hipStream_t stream);

namespace {

constexpr int kUnseen = INT32_MAX;
__device__ __forceinline__ int64_t ceil_div_dev(int64_t a, int64_t b) { return (a + b - 1) / b; }
constexpr int kLdsPicks = 1024;  // random positions a wave keeps in LDS

struct Graph {
    const int64_t *v2v_ptr, *v2v_idx, *v2r_ptr, *v2r_idx, *r2v_ptr, *r2v_idx;
    const int64_t *r2r_ptr[CGNN_SAMPLE_MAX_LEVELS], *r2r_idx[CGNN_SAMPLE_MAX_LEVELS];
    const int64_t *v_degree, *r_degree;
    int64_t vertex_cnt, rule_cnt;
    int levels;
};

Graph graph_of(const cgnn_sample_graph *g) {
    Graph d{};
    d.v2v_ptr = g->v2v_ptr, d.v2v_idx = g->v2v_idx, d.v2r_ptr = g->v2r_ptr, d.v2r_idx = g->v2r_idx;
    d.r2v_ptr = g->r2v_ptr, d.r2v_idx = g->r2v_idx;
    for (int k = 0; k < g->levels; ++k) d.r2r_ptr[k] = g->r2r_ptr[k], d.r2r_idx[k] = g->r2r_idx[k];
    d.v_degree = g->v_degree, d.r_degree = g->r_degree;
    d.vertex_cnt = g->vertex_cnt, d.rule_cnt = g->rule_cnt, d.levels = g->levels;
    return d;
}

// ---------------------------------------------------------------- random positions --
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z ^= z >> 30;
    z *= 0xbf58476d1ce4e5b9ULL;
    z ^= z >> 27;
    z *= 0x94d049bb133111ebULL;
    z ^= z >> 31;
    return z;
}

// an integer in [0, high)
__device__ __forceinline__ int64_t draw(uint64_t seed, int64_t layer, int64_t i, int64_t j, int64_t high) {
    const uint64_t key = mix64(seed ^ (0x9e3779b97f4a7c15ULL * (uint64_t)(layer + 1)));
    const uint64_t u = mix64(key + (uint64_t)i * 0xd1342543de82ef95ULL + (uint64_t)j);
    return (int64_t)__umul64hi(u, (uint64_t)high);
}

// Entry k of a rule: its own list, then the children that the descent takes.
__device__ int64_t below_rule(const Graph &g, int64_t rule, int64_t k) {
    for (int level = 0; level < g.levels; ++level) {
        const int64_t own = g.r2v_ptr[rule], own_count = g.r2v_ptr[rule + 1] - own;
        if (k < own_count) return g.r2v_idx[own + k];
        k -= own_count;
        for (int64_t c = g.r2r_ptr[level][rule]; c < g.r2r_ptr[level][rule + 1]; ++c) {
            const int64_t child = g.r2r_idx[level][c];
            const int64_t child_degree = g.r_degree[child];
            if (k < child_degree) {
                rule = child;
                break;
            }
            k -= child_degree;
        }
    }
    const int64_t own = g.r2v_ptr[rule], own_count = g.r2v_ptr[rule + 1] - own;
    if (k < own_count) return g.r2v_idx[own + k];
    // The descent found less than r_degree promised (degrees that do not fit the hierarchy).
    // The reference goes on to the next rule with k - degree, which is negative by now, and
    // indexes before that rule's list; here the position counts as out of range.
    return -1;
}

// -------------------------------------------------------- the expanded in-list ------
// The k-th neighbour in the order of storage_api.h:6-70: v2v entries; then, rule by rule of
// the vertex's v2r entries, the rule's expanded list (its r2v entries, then its children's
// lists, the children of the wave-th descent taken from level `wave` of r2r).  -1: k lies
// beyond what the descent finds (the reference throws out_of_range, or reads out of bounds: below).
__device__ int64_t neighbor_at(const Graph &g, int64_t node, int64_t k) {
    const int64_t v2v_start = g.v2v_ptr[node], v2v_count = g.v2v_ptr[node + 1] - v2v_start;
    if (k < v2v_count) return g.v2v_idx[v2v_start + k];
    if (g.v2r_ptr == nullptr) return -1;  // a plain graph: no rules
    k -= v2v_count;
    for (int64_t e = g.v2r_ptr[node]; e < g.v2r_ptr[node + 1]; ++e) {
        const int64_t rule = g.v2r_idx[e], degree = g.r_degree[rule];
        if (k < degree) return below_rule(g, rule, k);
        k -= degree;
    }
    return -1;
}

// Depth-first walk over the rules reached from `node` (depth d expands through level d of
// r2r; rules at depth `levels` are not expanded): visit(rule, depth) in pre-order.  The walk is
// uniform over the wave (every lane runs it on the same vertex).
template <typename Visit>
__device__ __forceinline__ void walk_rules(const Graph &g, int64_t node, Visit visit) {
    int64_t at[CGNN_SAMPLE_MAX_LEVELS + 1], end[CGNN_SAMPLE_MAX_LEVELS + 1];
    if (g.v2r_ptr == nullptr) return;  // a plain graph: no rules
    for (int64_t e = g.v2r_ptr[node]; e < g.v2r_ptr[node + 1]; ++e) {
        int64_t rule = g.v2r_idx[e];
        int depth = 0;
        visit(rule, 0);
        if (g.levels > 0) {
            at[0] = g.r2r_ptr[0][rule];
            end[0] = g.r2r_ptr[0][rule + 1];
        }
        // the stack holds, per depth, the range of children still to visit
        while (g.levels > 0 && depth >= 0) {
            if (at[depth] == end[depth]) {
                --depth;
                continue;
            }
            rule = g.r2r_idx[depth][at[depth]++];
            visit(rule, depth + 1);
            if (depth + 1 < g.levels) {
                ++depth;
                at[depth] = g.r2r_ptr[depth][rule];
                end[depth] = g.r2r_ptr[depth][rule + 1];
            }
        }
    }
}

// Length of the full list of storage_api.h:72-118 and the r2v entries per depth.
__device__ int64_t full_list_sizes(const Graph &g, int64_t node, int64_t per_depth[CGNN_SAMPLE_MAX_LEVELS + 1]) {
    for (int d = 0; d <= g.levels; ++d) per_depth[d] = 0;
    walk_rules(g, node, [&](int64_t rule, int depth) { per_depth[depth] += g.r2v_ptr[rule + 1] - g.r2v_ptr[rule]; });
    int64_t total = g.v2v_ptr[node + 1] - g.v2v_ptr[node];
    for (int d = 0; d <= g.levels; ++d) total += per_depth[d];
    return total;
}

struct LayerArgs {
    Graph g;
    const int64_t *frontier;  // [n] vertices
    int64_t n;
    int64_t fanout;
    int64_t first_position;   // position of frontier[0] among the samples
    int64_t layer;
    uint64_t seed;
    int32_t *counts;          // [n]
    const int32_t *offsets;   // [n + 1]
    int64_t *neighbors;       // [offsets[n]]
    int64_t *sources;         // [offsets[n]] position (among the samples) of the vertex a neighbour belongs to
    int64_t *picks;           // [offsets[n]] scratch: the chosen positions
    int32_t *status;          // device flags, see CGNN_SAMPLE_* in the header
};

__device__ __forceinline__ int64_t degree_of(const Graph &g, int64_t node) {
    return g.v_degree ? g.v_degree[node] : g.v2v_ptr[node + 1] - g.v2v_ptr[node];
}

// counts[i]: neighbours that frontier vertex i contributes (neighbor_sample.h:88-99,111).
__global__ __launch_bounds__(kBlock) void sample_count_kernel(LayerArgs a) {
    const int64_t i = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (i >= a.n) return;
    const int64_t node = a.frontier[i];
    int32_t count = 0;
    if (node < 0 || node >= a.g.vertex_cnt) {
        *a.status = CGNN_SAMPLE_BAD_VERTEX;  // every writer of a kind stores the same value
    } else {
        const int64_t degree = degree_of(a.g, node);
        if (degree > 0) {
            if (a.fanout >= degree) {
                int64_t per_depth[CGNN_SAMPLE_MAX_LEVELS + 1];
                const int64_t full = full_list_sizes(a.g, node, per_depth);
                if (full >= INT32_MAX) *a.status = CGNN_SAMPLE_TOO_MANY;
                else count = (int32_t)full;
            } else if (a.fanout >= INT32_MAX) {
                *a.status = CGNN_SAMPLE_TOO_MANY;  // one vertex alone would add 2^31 - 1 neighbours or more
            } else {
                count = (int32_t)a.fanout;
            }
        }
    }
    if (threadIdx.x % kWave == 0) a.counts[i] = count;
}

__global__ __launch_bounds__(kBlock) void sample_fill_kernel(LayerArgs a) {
    const int lane = threadIdx.x % kWave;
    const int64_t i = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (i >= a.n) return;
    const int64_t out0 = a.offsets[i], count = a.offsets[i + 1] - out0;
    if (count == 0) return;
    const Graph &g = a.g;
    const int64_t node = a.frontier[i];  // in range: the count of a vertex out of range is 0
    const int64_t position = a.first_position + i;
    for (int64_t t = lane; t < count; t += kWave) a.sources[out0 + t] = position;
    const int64_t degree = degree_of(g, node);
    auto put = [&](int64_t slot, int64_t neighbor) {
        if (neighbor < 0 || neighbor >= g.vertex_cnt) {
            // -1: the descent ran out (out_of_range in the reference); anything else: a corrupt graph
            *a.status = neighbor == -1 ? CGNN_SAMPLE_OUT_OF_RANGE : CGNN_SAMPLE_BAD_VERTEX;
            neighbor = 0;
        }
        a.neighbors[out0 + slot] = neighbor;
    };
    if (a.fanout >= degree) {
        // the whole list: v2v entries, then per depth the r2v entries of the rules of that depth
        const int64_t v2v_start = g.v2v_ptr[node], v2v_count = g.v2v_ptr[node + 1] - v2v_start;
        for (int64_t t = lane; t < v2v_count; t += kWave) put(t, g.v2v_idx[v2v_start + t]);
        int64_t next[CGNN_SAMPLE_MAX_LEVELS + 1];  // where the next rule of a depth writes
        full_list_sizes(g, node, next);
        int64_t running = v2v_count;
        for (int d = 0; d <= g.levels; ++d) {
            const int64_t size = next[d];
            next[d] = running;
            running += size;
        }
        walk_rules(g, node, [&](int64_t rule, int depth) {
            const int64_t own = g.r2v_ptr[rule], own_count = g.r2v_ptr[rule + 1] - own;
            for (int64_t t = lane; t < own_count; t += kWave) put(next[depth] + t, g.r2v_idx[own + t]);
            next[depth] += own_count;
        });
        return;
    }
    // `count` = fanout distinct positions out of `degree` (neighbor_sample.h:112-118): step j draws
    // from [0, j) and takes j itself when the draw was taken before.  The steps depend on each
    // other, so the wave runs them one after the other; all lanes compare a draw with the
    // positions chosen so far, 64 at a time.  The positions are kept in LDS; a fan-out beyond
    // kLdsPicks keeps them in the caller's scratch, accessed around the vector cache (one
    // lane writes, all lanes read).
    __shared__ int64_t lds_picks[kBlock / kWave][kLdsPicks];
    int64_t *mine = lds_picks[threadIdx.x / kWave];
    int64_t *far = a.picks + out0;
    const bool in_lds = count <= kLdsPicks;
    auto pick_at = [&](int64_t c) {
        return in_lds ? mine[c] : __hip_atomic_load(far + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    for (int64_t s = 0; s < count; ++s) {
        const int64_t j = degree - count + s;
        int64_t rnd = draw(a.seed, a.layer, position, j, j);
        bool taken = false;
        for (int64_t c0 = 0; c0 < s; c0 += kWave) {
            const int64_t c = c0 + lane;
            taken = taken || (__ballot(c < s && pick_at(c) == rnd) != 0);
        }
        if (taken) rnd = j;
        if (lane == 0) {
            if (in_lds) mine[s] = rnd;
            else __hip_atomic_store(far + s, rnd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // the position is read by all lanes in the next step
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    for (int64_t t = lane; t < count; t += kWave) put(t, neighbor_at(g, node, pick_at(t)));
}

// ------------------------------------------------------- layers of a bounded size ----
// A vertex has one entry in number_of: kUnseen, or kClaim + the first slot of the layer that holds it, or the number it
// was given.  Smaller is final, so that claims are atomic minima that never touch a number.
constexpr int32_t kClaim = 1 << 30;
constexpr int kChunkItems = 4;
constexpr int kChunk = kChunkItems * kBlock;  // most slots per workgroup when they are ranked
constexpr int kTail = 8;                      // chunks a thread sums up when all are counted
constexpr int kRegPicks = kWave;              // fan-outs up to this keep the chosen positions in registers, one a lane
// Layers of up to this many chunks are counted while they are filled: a claim that is taken over moves its vertex from one
// chunk to another, and the workgroups that rank the slots sum up the chunks in front of theirs.  A launch of 5 to 7 us
// less a layer (and one pass less over the slots, 15 us where there are 5 million), 1 to 2 us more in the fill: 1,024 seeds
// with 25 and 10 61 -> 57 us, 8,192 with 10 and 10 76 -> 70, 16,384 with 25 and 15 109 -> 93, with 25 and 25 (8,139 chunks)
// 123 -> 99.  Beyond, what they read of each other's counts (256 MB at this limit) grows with the square, and a launch of
// its own counts the slots and sums them up once.
constexpr int64_t kCountedChunks = 8192;

struct BoundedLayer {
    int64_t fanout, n_cap;   // most vertices of the frontier
    int32_t chunk;           // slots of a chunk: those of as many workgroups of bounded_fill_kernel as kChunk holds
    int32_t *slots;          // [n_cap * fanout] neighbours, -1 behind the last
    uint64_t *counts;        // [chunks] neighbours, and << 32 vertices they introduce; NULL: counted by bounded_count_kernel
    uint64_t *before;        // [chunks] the same in the chunks in front
};

__host__ __device__ __forceinline__ int bounded_lanes(int64_t fanout) { return fanout <= 16 ? 16 : fanout <= 32 ? 32 : kWave; }

// state of a layer: position of its frontier among the samples, vertices in it, edges of the layers before, chunks
// ranked so far
struct BoundedArgs {
    Graph g;
    int64_t n_input;
    const int64_t *input;
    int32_t *number_of, *samples;  // samples: without the input, which stands in front of them
    int32_t *state;          // [layers + 1][4]
    int32_t *status;         // [2] CGNN_SAMPLE_* of the first error; whether a full list went beyond its bounds
    int32_t *summary;        // last layer: number of samples, edges, status, 1 (pinned host memory)
    uint64_t seed;
    int32_t layer, layers;
    BoundedLayer at[CGNN_SAMPLE_MAX_BOUNDED];
    int64_t first_chunk[CGNN_SAMPLE_MAX_BOUNDED + 1];  // of a layer, when all are written at once
    int64_t *out_samples, *out_source, *out_neighbor;
};

__global__ __launch_bounds__(kBlock) void bounded_begin_kernel(BoundedArgs a) {
    const int64_t stride = (int64_t)gridDim.x * kBlock, t0 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    for (int64_t v = t0; v < a.g.vertex_cnt; v += stride) a.number_of[v] = kUnseen;
    for (int k = 0; k < a.layers; ++k)
        if (a.at[k].counts != nullptr)
            for (int64_t c = t0; c < a.first_chunk[k + 1] - a.first_chunk[k]; c += stride) a.at[k].counts[c] = 0;
    if (t0 < 4 * (a.layers + 1)) a.state[t0] = t0 == 1 ? (int32_t)a.n_input : 0;
    if (t0 < 2) a.status[t0] = CGNN_SAMPLE_OK;
}

template <int LANES>
__device__ __forceinline__ bool any_lane(bool yes) {
    return (__ballot(yes) >> (threadIdx.x % kWave / LANES * LANES) & (~uint64_t(0) >> (kWave - LANES))) != 0;
}

template <int LANES, typename V>
__device__ __forceinline__ V inclusive_sum(V v, int lane) {
#pragma unroll
    for (int s = 1; s < LANES; s <<= 1) {
        const V up = __shfl_up(v, s, LANES);
        if (lane >= s) v += up;
    }
    return v;
}

// The first lane whose value, none smaller than that of the lane before, is greater than k.
template <int LANES, typename V>
__device__ __forceinline__ int first_above(V values, V k) {
    int p = 0;
#pragma unroll
    for (int s = LANES / 2; s > 0; s >>= 1)
        if (__shfl(values, p + s - 1, LANES) <= k) p += s;
    return p;
}

// Entries k of a vertex's list (neighbor_at), one a lane: its rules are searched LANES at a time, because one by one
// each costs two loads that wait for each other, and a hub has hundreds.
template <int LANES>
__device__ __forceinline__ int64_t neighbors_at(const Graph &g, int64_t node, int64_t k, bool wanted, int lane) {
    const int64_t v2v_start = g.v2v_ptr[node], v2v_count = g.v2v_ptr[node + 1] - v2v_start;
    int64_t neighbor = -1;
    if (wanted && k < v2v_count) {
        neighbor = g.v2v_idx[v2v_start + k];
        wanted = false;  // all lanes stay for the exchange below
    }
    if (g.v2r_ptr == nullptr) return neighbor;
    k -= v2v_count;
    const int64_t end = g.v2r_ptr[node + 1];
    int64_t rule = -1;
    for (int64_t e0 = g.v2r_ptr[node]; e0 < end && any_lane<LANES>(wanted && rule < 0); e0 += LANES) {
        const int64_t mine = e0 + lane < end ? g.v2r_idx[e0 + lane] : -1;
        const int64_t degree = mine >= 0 ? g.r_degree[mine] : 0;
        const int64_t sum = inclusive_sum<LANES>(degree, lane);
        int64_t most = sum;
        if (any_lane<LANES>(degree < 0))  // then not every sum is above those in front of it
#pragma unroll
            for (int s = 1; s < LANES; s <<= 1) {
                const int64_t up = __shfl_up(most, s, LANES);
                if (lane >= s && up > most) most = up;
            }
        const int p = first_above<LANES>(most, k);
        const int64_t found = __shfl(mine, p, LANES), before = __shfl(sum - degree, p, LANES);
        const int64_t above = __shfl(most, LANES - 1, LANES), all = __shfl(sum, LANES - 1, LANES);
        if (rule >= 0) continue;
        if (k < above) {
            rule = found;
            k -= before;
        } else {
            k -= all;
        }
    }
    return wanted && rule >= 0 ? below_rule(g, rule, k) : neighbor;
}

// LANES lanes per frontier vertex (as many as the fan-out asks for: a step waits for one load after another, and
// with a wave per vertex most lanes of it wait for nothing), into the vertex's slots.  The first layer also
// numbers the input, a vertex given twice by its first position.  COUNTED: adds to the counts of the workgroup's chunk how
// many neighbours it found and how many vertices they introduce as far as is known; a claim that it takes from a slot
// further back, or that a number takes from a slot, is taken off that slot's chunk.
template <int LANES, bool COUNTED>
__global__ __launch_bounds__(kBlock) void bounded_fill_kernel(BoundedArgs a) {
    const BoundedLayer &l = a.at[a.layer];
    const int32_t first = a.state[4 * a.layer], n = a.state[4 * a.layer + 1];
    const int64_t i0 = (int64_t)blockIdx.x * (kBlock / LANES);
    if (i0 >= n) return;
    int live = 0, fresh = 0;
    auto displaced = [&](int32_t claim) {
        if (claim >= kClaim && claim != kUnseen)
            __hip_atomic_fetch_add(l.counts + (claim - kClaim) / l.chunk, ~uint64_t(0) << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto fill = [&](int64_t i, int lane) {
        const Graph &g = a.g;
        const int fanout = (int)l.fanout;
        const int64_t node = a.layer == 0 ? a.input[i] : a.samples[first + i], slot0 = i * fanout;
        auto put = [&](int t, int64_t neighbor) {
            if (neighbor < 0 || neighbor >= g.vertex_cnt) {
                atomicCAS(a.status, CGNN_SAMPLE_OK, neighbor == -1 ? CGNN_SAMPLE_OUT_OF_RANGE : CGNN_SAMPLE_BAD_VERTEX);
                neighbor = 0;
            }
            l.slots[slot0 + t] = (int32_t)neighbor;
            const int32_t claim = kClaim + (int32_t)(slot0 + t);
            if (a.number_of[neighbor] > claim) {
                const int32_t was = atomicMin(&a.number_of[neighbor], claim);
                if (COUNTED && was > claim) {
                    ++fresh;
                    displaced(was);
                }
            }
        };
        auto full_list = [&]() -> int {  // its length, or -1: longer than the fan-out (or by rules that lead nowhere)
            const int64_t v2v_start = g.v2v_ptr[node], v2v_count = g.v2v_ptr[node + 1] - v2v_start;
            if (v2v_count > fanout) return -1;
            if (lane < v2v_count) put(lane, g.v2v_idx[v2v_start + lane]);
            int count = (int)v2v_count;
            if (g.v2r_ptr == nullptr) return count;
            // Depth by depth, a rule a lane, in the order in which a walk in pre-order meets the rules of a depth.  Sizes
            // are cut off where they are too large in any case, so that two sums fit into one.
            const int64_t v2r_start = g.v2r_ptr[node], v2r_count = g.v2r_ptr[node + 1] - v2r_start;
            if (v2r_count > LANES) return -1;
            auto cut = [](int64_t size) { return (int)(size < 0 ? 0 : size > LANES ? LANES + 1 : size); };
            int rules = (int)v2r_count;
            int64_t rule = lane < rules ? g.v2r_idx[v2r_start + lane] : 0;
            for (int depth = 0; rules > 0; ++depth) {
                int64_t own_start = 0, child_start = 0;
                int own = 0, children = 0;
                if (lane < rules) {
                    own_start = g.r2v_ptr[rule];
                    own = cut(g.r2v_ptr[rule + 1] - own_start);
                    if (depth < g.levels) {
                        child_start = g.r2r_ptr[depth][rule];
                        children = cut(g.r2r_ptr[depth][rule + 1] - child_start);
                    }
                }
                const int sums = inclusive_sum<LANES>(own | children << 16, lane), all = __shfl(sums, LANES - 1, LANES);
                const int owns = sums & 0xffff, all_own = all & 0xffff, descend = sums >> 16, all_descend = all >> 16;
                if (count + all_own > fanout || all_descend > LANES) return -1;
                const int p = first_above<LANES>(owns, lane);
                const int64_t from = __shfl(own_start - (owns - own), p, LANES);
                if (lane < all_own) put(count + lane, g.r2v_idx[from + lane]);
                count += all_own;
                rules = all_descend;
                const int q = first_above<LANES>(descend, lane);
                const int64_t child = __shfl(child_start - (descend - children), q, LANES);
                if (lane < rules) rule = g.r2r_idx[depth][child + lane];
            }
            return count;
        };
        int count = 0;
        if (node < 0 || node >= g.vertex_cnt) {
            atomicCAS(a.status, CGNN_SAMPLE_OK, CGNN_SAMPLE_BAD_VERTEX);
        } else {
            if (a.layer == 0 && lane == 0) {
                const int32_t was = atomicMin(&a.number_of[node], (int32_t)i);
                if (COUNTED) displaced(was);
            }
            const int64_t degree = degree_of(g, node);
            if (degree > fanout) {
                // The selection loop of sample_fill_kernel with a step per lane: the draws do not depend on each other, only
                // whether a drawn position was taken before does.
                count = fanout;
                const int64_t j = degree - count + lane;
                int64_t pick = lane < count ? draw(a.seed, a.layer, first + i, j, j) : -1;
                for (int s = 1; s < count; ++s) {
                    const int64_t rnd = __shfl(pick, s, LANES);
                    const bool taken = any_lane<LANES>(lane < s && pick == rnd);
                    if (lane == s && taken) pick = j;
                }
                const int64_t neighbor = neighbors_at<LANES>(g, node, pick, lane < count, lane);
                if (lane < count) put(lane, neighbor);
            } else if (degree > 0) {
                count = full_list();
                if (count < 0) {  // the call is done again layer by layer
                    a.status[1] = 1;
                    count = 0;
                }
            }
        }
        for (int t = count + lane; t < fanout; t += LANES) l.slots[slot0 + t] = -1;
        if (lane == 0) live = count;
    };
    const int64_t mine = i0 + threadIdx.x / LANES;
    if (mine < n) fill(mine, threadIdx.x % LANES);
    if constexpr (COUNTED) {  // at most 256 of each a workgroup
        __shared__ int sums[kBlock / kWave];
        const int sum = inclusive_sum<kWave>(live | fresh << 16, (int)(threadIdx.x % kWave));
        if (threadIdx.x % kWave == kWave - 1) sums[threadIdx.x / kWave] = sum;
        __syncthreads();
        if (threadIdx.x == 0) {
            int all = 0;
#pragma unroll
            for (int w = 0; w < kBlock / kWave; ++w) all += sums[w];
            __hip_atomic_fetch_add(l.counts + i0 * l.fanout / l.chunk, (uint64_t)(all >> 16) << 32 | (uint64_t)(all & 0xffff),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// The slots of a thread in a chunk of a layer with `slots` of them: neighbours (or -1), and which introduce a vertex.
struct ChunkSlots {
    int32_t v[kChunkItems];
    unsigned introduces;
    int live, fresh;
};

__device__ __forceinline__ ChunkSlots chunk_slots(const BoundedArgs &a, const BoundedLayer &l, int64_t slots, int64_t chunk,
                                                  bool ranks) {
    ChunkSlots c;
    const int64_t s0 = chunk * l.chunk + threadIdx.x * kChunkItems;
    slots = min(slots, (chunk + 1) * l.chunk);
    if (s0 + kChunkItems <= slots) {
        const int4 four = *reinterpret_cast<const int4 *>(l.slots + s0);
        c.v[0] = four.x, c.v[1] = four.y, c.v[2] = four.z, c.v[3] = four.w;
    } else {
#pragma unroll
        for (int u = 0; u < kChunkItems; ++u) c.v[u] = s0 + u < slots ? l.slots[s0 + u] : -1;
    }
    c.introduces = 0;
    c.live = c.fresh = 0;
    int32_t number[kChunkItems];
#pragma unroll
    for (int u = 0; u < kChunkItems; ++u)  // all loads before the first use
        number[u] = ranks ? a.number_of[c.v[u] < 0 ? 0 : c.v[u]] : 0;
#pragma unroll
    for (int u = 0; u < kChunkItems; ++u) {
        if (c.v[u] < 0) continue;
        ++c.live;
        if (number[u] == kClaim + (int32_t)(s0 + u)) {
            c.introduces |= 1u << u;
            ++c.fresh;
        }
    }
    return c;
}

// Exclusive sums of two values over the workgroup, and the totals.
__device__ __forceinline__ int2 chunk_sums(int live, int fresh, int2 *total) {
    __shared__ int2 wave_sum[kBlock / kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    int a = live, b = fresh;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
        const int x = __shfl_up(a, s, kWave), y = __shfl_up(b, s, kWave);
        if (lane >= s) a += x, b += y;
    }
    __syncthreads();
    if (lane == kWave - 1) wave_sum[wave] = make_int2(a, b);
    __syncthreads();
    int2 before = make_int2(a - live, b - fresh), all = make_int2(0, 0);
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) {
        if (w < wave) before.x += wave_sum[w].x, before.y += wave_sum[w].y;
        all.x += wave_sum[w].x, all.y += wave_sum[w].y;
    }
    *total = all;
    return before;
}

// The sizes of a call, in pinned host memory: the last word last, past the caches with a wait between (a release would write
// back the whole L2).
__device__ __forceinline__ void bounded_summary(const BoundedArgs &a, int32_t samples, int32_t edges) {
    const int32_t words[3] = {samples, edges, a.status[1] ? -1 : a.status[0]};
#pragma unroll
    for (int k = 0; k < 3; ++k) __hip_atomic_store(a.summary + k, words[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __hip_atomic_store(a.summary + 3, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The vertices in the next layer's frontier.  None once a list did not fit its degree: its slots were cleared behind its
// claims, which no slot of this layer answers to, and the next layer would take them off counts that are not theirs.  The
// call is done again layer by layer in any case.
__device__ __forceinline__ int32_t bounded_frontier(const BoundedArgs &a, int32_t introduced) { return a.status[1] ? 0 : introduced; }

// How many neighbours a chunk holds and how many vertices they introduce; the last chunk to be counted sums the
// chunks up and sets the state of the next layer.
__global__ __launch_bounds__(kBlock) void bounded_count_kernel(BoundedArgs a) {
    const BoundedLayer &l = a.at[a.layer];
    int32_t *state = a.state + 4 * a.layer;
    const int64_t n = state[1], held = ceil_div_dev(n * l.fanout, l.chunk), chunks = held < 1 ? 1 : held;
    if (blockIdx.x >= chunks) return;
    const ChunkSlots c = chunk_slots(a, l, n * l.fanout, blockIdx.x, true);
    int2 total;
    chunk_sums(c.live, c.fresh, &total);
    __shared__ bool arrived_last;
    if (threadIdx.x == 0) {  // read by another XCD in this launch: as the pieces of workgroup runs (spmm.hip)
        __hip_atomic_store(l.before + blockIdx.x, (uint64_t)total.y << 32 | (uint32_t)total.x, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        arrived_last = __hip_atomic_fetch_add(state + 3, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == chunks - 1;
    }
    __syncthreads();
    if (!arrived_last) return;
    int2 running = make_int2(0, 0);
    for (int64_t k0 = (int64_t)threadIdx.x * kTail; k0 - threadIdx.x * kTail < chunks; k0 += kBlock * kTail) {
        uint64_t pair[kTail];
        int2 sum = make_int2(0, 0), all;
#pragma unroll
        for (int u = 0; u < kTail; ++u)  // all loads in flight
            pair[u] = k0 + u < chunks ? __hip_atomic_load(l.before + k0 + u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
#pragma unroll
        for (int u = 0; u < kTail; ++u) sum.x += (int)(uint32_t)pair[u], sum.y += (int)(pair[u] >> 32);
        int2 before = chunk_sums(sum.x, sum.y, &all);
        before.x += running.x, before.y += running.y;
#pragma unroll
        for (int u = 0; u < kTail; ++u) {
            if (k0 + u < chunks) l.before[k0 + u] = (uint64_t)before.y << 32 | (uint32_t)before.x;
            before.x += (int)(uint32_t)pair[u], before.y += (int)(pair[u] >> 32);
        }
        running.x += all.x, running.y += all.y;
    }
    if (threadIdx.x == 0) {
        const int32_t end = state[0] + (int32_t)n;
        state[4] = end;
        state[5] = bounded_frontier(a, running.y);
        state[6] = state[2] + running.x;
        if (a.layer == a.layers - 1) bounded_summary(a, end + running.y, state[2] + running.x);
    }
}

// The vertices that a layer introduces take the numbers behind its frontier, in the order of their slots.  COUNTED: every
// workgroup sums up the counts of the chunks, and the first sets the state of the next layer.
template <bool COUNTED>
__global__ __launch_bounds__(kBlock) void bounded_assign_kernel(BoundedArgs a) {
    const BoundedLayer &l = a.at[a.layer];
    int32_t *state = a.state + 4 * a.layer;
    const int64_t n = state[1], slots = n * l.fanout;
    if (blockIdx.x > 0 && (int64_t)blockIdx.x * l.chunk >= slots) return;
    const int32_t end = state[0] + (int32_t)n;
    int32_t fresh_before;
    if constexpr (COUNTED) {
        const int64_t chunks = ceil_div_dev(slots, l.chunk);
        uint64_t before = 0, behind = 0;  // only the first workgroup needs what stands behind
        for (int64_t c0 = threadIdx.x; c0 < (blockIdx.x == 0 ? chunks : blockIdx.x); c0 += kTail * kBlock) {
            uint64_t pair[kTail];
#pragma unroll
            for (int u = 0; u < kTail; ++u) pair[u] = c0 + u * kBlock < chunks ? l.counts[c0 + u * kBlock] : 0;
#pragma unroll
            for (int u = 0; u < kTail; ++u) {
                if (c0 + u * kBlock < blockIdx.x) before += pair[u];
                else behind += pair[u];
            }
        }
        int2 all_before, all_behind;
        chunk_sums((int)(uint32_t)before, (int)(before >> 32), &all_before);
        chunk_sums((int)(uint32_t)behind, (int)(behind >> 32), &all_behind);
        if (threadIdx.x == 0) {
            l.before[blockIdx.x] = (uint64_t)all_before.y << 32 | (uint32_t)all_before.x;
            if (blockIdx.x == 0) {
                state[4] = end;
                state[5] = bounded_frontier(a, all_behind.y);
                state[6] = state[2] + all_behind.x;
                if (a.layer == a.layers - 1) bounded_summary(a, end + all_behind.y, state[2] + all_behind.x);
            }
        }
        fresh_before = all_before.y;
    } else {
        fresh_before = (int32_t)(l.before[blockIdx.x] >> 32);
    }
    const ChunkSlots c = chunk_slots(a, l, slots, blockIdx.x, true);
    int2 total;
    int32_t number = end + fresh_before + chunk_sums(c.live, c.fresh, &total).y;
#pragma unroll
    for (int u = 0; u < kChunkItems; ++u)
        if (c.introduces >> u & 1u) {
            // no other slot has this claim
            a.number_of[c.v[u]] = number;
            a.samples[number++] = c.v[u];
        }
}

// The edges of all layers and the samples, in arrays of their exact sizes.
__global__ __launch_bounds__(kBlock) void bounded_write_kernel(BoundedArgs a) {
    const int64_t chunks = a.first_chunk[a.layers];
    if ((int64_t)blockIdx.x >= chunks) {
        const int64_t i = (blockIdx.x - chunks) * (int64_t)kBlock + threadIdx.x;
        if (i < a.state[4 * a.layers] + a.state[4 * a.layers + 1]) a.out_samples[i] = i < a.n_input ? a.input[i] : a.samples[i];
        return;
    }
    int layer = 0;
    while (layer + 1 < a.layers && (int64_t)blockIdx.x >= a.first_chunk[layer + 1]) ++layer;
    const BoundedLayer &l = a.at[layer];
    const int32_t *state = a.state + 4 * layer;
    const int64_t chunk = blockIdx.x - a.first_chunk[layer], n = state[1];
    if (chunk * l.chunk >= n * l.fanout) return;
    const ChunkSlots c = chunk_slots(a, l, n * l.fanout, chunk, false);
    int2 total;
    int64_t e = (int64_t)state[2] + (int32_t)l.before[chunk] + chunk_sums(c.live, 0, &total).x;
    const int64_t s0 = chunk * l.chunk + threadIdx.x * kChunkItems;
    int64_t i = s0 / l.fanout, t = s0 - i * l.fanout;
#pragma unroll
    for (int u = 0; u < kChunkItems; ++u) {
        if (c.v[u] >= 0) {
            a.out_source[e] = state[0] + i;
            a.out_neighbor[e++] = a.number_of[c.v[u]];
        }
        if (++t == l.fanout) t = 0, ++i;
    }
}

// ------------------------------------------------------------------- relabelling ----
// seen_at[v] = first position at which vertex v appears among the new neighbours (only for
// vertices without a local number yet).
__global__ void relabel_first_kernel(const int64_t *__restrict__ neighbors, int64_t total,
                                     const int32_t *__restrict__ local_of, int32_t *__restrict__ seen_at) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = neighbors[t];
        if (local_of[v] == kUnseen) atomicMin(&seen_at[v], (int32_t)t);  // integer minimum: any order, one result
    }
}

// introduces[t] = 1 where position t is the first occurrence of a vertex without a number.
__global__ void relabel_flag_kernel(const int64_t *__restrict__ neighbors, int64_t total,
                                    const int32_t *__restrict__ local_of, const int32_t *__restrict__ seen_at,
                                    int32_t *__restrict__ introduces) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = neighbors[t];
        introduces[t] = (local_of[v] == kUnseen && seen_at[v] == (int32_t)t) ? 1 : 0;
    }
}

// New vertices take the numbers base, base + 1, ... in the order of their first occurrence.
__global__ void relabel_assign_kernel(const int64_t *__restrict__ neighbors, int64_t total,
                                      const int32_t *__restrict__ introduces, const int32_t *__restrict__ rank,
                                      int64_t base, int32_t *__restrict__ local_of, int64_t *__restrict__ samples,
                                      int64_t *__restrict__ new_count) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        if (introduces[t]) {
            const int64_t v = neighbors[t];
            const int64_t number = base + rank[t] - 1;  // rank: inclusive count of introductions up to t
            local_of[v] = (int32_t)number;
            samples[number] = v;
        }
        if (t == total - 1) *new_count = rank[t];
    }
}

__global__ void relabel_lookup_kernel(const int64_t *__restrict__ neighbors, int64_t total,
                                      const int32_t *__restrict__ local_of, int32_t *__restrict__ seen_at,
                                      int64_t *__restrict__ numbers) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = neighbors[t];
        numbers[t] = local_of[v];
        seen_at[v] = kUnseen;  // the table is clean again for the next layer
    }
}

// The input vertices number themselves 0, 1, ...; of equal ones the first counts.
__global__ void relabel_seeds_kernel(const int64_t *__restrict__ input, int64_t n, int64_t vertex_cnt,
                                     int32_t *__restrict__ local_of, int32_t *__restrict__ status) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = input[i];
        if (v < 0 || v >= vertex_cnt) *status = CGNN_SAMPLE_BAD_VERTEX;
        else atomicMin(&local_of[v], (int32_t)i);
    }
}

__global__ void fill_i32_value_kernel(int32_t *p, int64_t n, int32_t value) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

// ---------------------------------------------------------------- prefix sums -------
// out[0] = 0, out[i + 1] = in[0] + ... + in[i] (n + 1 entries), three passes over tiles.
constexpr int kSumItems = 16;
constexpr int kSumTile = kBlock * kSumItems;

__device__ __forceinline__ int64_t block_sum_scan(int64_t v, int64_t *total) {
    __shared__ int64_t wave_sum[kBlock / kWave];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    int64_t inc = v;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
        const int64_t n = __shfl_up(inc, s, kWave);
        if (lane >= s) inc += n;
    }
    __syncthreads();
    if (lane == kWave - 1) wave_sum[wave] = inc;
    __syncthreads();
    int64_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) {
        if (w < wave) before += wave_sum[w];
        all += wave_sum[w];
    }
    *total = all;
    return before + inc;
}

__global__ __launch_bounds__(kBlock) void sum_tiles_kernel(const int32_t *__restrict__ in, int64_t n,
                                                          int64_t *__restrict__ tile_total) {
    const int64_t base = (int64_t)blockIdx.x * kSumTile + (int64_t)threadIdx.x * kSumItems;
    int64_t s = 0;
#pragma unroll
    for (int k = 0; k < kSumItems; ++k)
        if (base + k < n) s += in[base + k];
    int64_t total;
    block_sum_scan(s, &total);
    if (threadIdx.x == 0) tile_total[blockIdx.x] = total;
}

__global__ __launch_bounds__(kBlock) void sum_totals_kernel(int64_t *tile_total, int64_t tiles) {
    int64_t running = 0;
    for (int64_t base = 0; base < tiles; base += kBlock) {
        const int64_t i = base + threadIdx.x;
        const int64_t v = i < tiles ? tile_total[i] : 0;
        int64_t total;
        const int64_t inc = block_sum_scan(v, &total);
        if (i < tiles) tile_total[i] = running + inc - v;
        running += total;
    }
}

__global__ __launch_bounds__(kBlock) void sum_apply_kernel(const int32_t *__restrict__ in, int64_t n,
                                                          const int64_t *__restrict__ tile_total,
                                                          int32_t *__restrict__ out, int32_t *__restrict__ status) {
    const int64_t base = (int64_t)blockIdx.x * kSumTile + (int64_t)threadIdx.x * kSumItems;
    int32_t v[kSumItems];
    int64_t s = 0;
#pragma unroll
    for (int k = 0; k < kSumItems; ++k) {
        v[k] = base + k < n ? in[base + k] : 0;
        s += v[k];
    }
    int64_t total;
    int64_t run = tile_total[blockIdx.x] + block_sum_scan(s, &total) - s;
    if (blockIdx.x == 0 && threadIdx.x == 0) out[0] = 0;
#pragma unroll
    for (int k = 0; k < kSumItems; ++k) {
        run += v[k];
        if (base + k < n) {
            if (run >= INT32_MAX) {
                if (status) *status = CGNN_SAMPLE_TOO_MANY;
                out[base + k + 1] = INT32_MAX;
            } else {
                out[base + k + 1] = (int32_t)run;
            }
        }
    }
}

int check_graph(const cgnn_sample_graph *g, const char *name) {
    if (g == nullptr) return fail(CGNN_EINVAL, "sample: null graph");
    if (g->vertex_cnt < 0 || g->rule_cnt < 0 || g->vertex_cnt >= INT32_MAX) {
        set_error("%s: vertex_cnt must be in [0, 2^31 - 1) and rule_cnt non-negative", name);
        return CGNN_EINVAL;
    }
    if (g->levels < 0 || g->levels > CGNN_SAMPLE_MAX_LEVELS) {
        set_error("%s: %d rule levels, at most %d are supported", name, g->levels, CGNN_SAMPLE_MAX_LEVELS);
        return CGNN_EUNSUPPORTED;
    }
    bool ok = g->v2v_ptr != nullptr;
    if (g->rule_cnt > 0) ok = ok && g->v2r_ptr && g->r2v_ptr;  // a graph without rules may leave the rule blocks out
    if (g->rule_cnt == 0 && (g->v2r_ptr == nullptr) != (g->r2v_ptr == nullptr)) ok = false;
    for (int k = 0; k < g->levels; ++k) ok = ok && g->r2r_ptr[k];
    if (!ok) {
        set_error("%s: a row-pointer array of the graph is null", name);
        return CGNN_EINVAL;
    }
    if (g->rule_cnt > 0 && (g->v_degree == nullptr || g->r_degree == nullptr)) {
        set_error("%s: a graph with rules needs the expanded degrees", name);
        return CGNN_EINVAL;
    }
    return CGNN_OK;
}

LayerArgs layer_args(const cgnn_sample_graph *g, int64_t n, const int64_t *frontier, int64_t fanout, int32_t *status) {
    LayerArgs a{};
    a.g = graph_of(g);
    a.frontier = frontier;
    a.n = n;
    a.fanout = fanout;
    a.status = status;
    return a;
}

unsigned blocks_for(int64_t n) {
    int64_t b = ceil_div(n, kBlock);
    return (unsigned)(b > 16384 ? 16384 : (b < 1 ? 1 : b));
}

}  // namespace
}  // namespace cgnn

using namespace cgnn;

extern "C" size_t cgnn_exclusive_sum_workspace_bytes(int64_t n) {
    return align_up((size_t)ceil_div(n < 1 ? 1 : n, kSumTile) * sizeof(int64_t), 256);
}

extern "C" int cgnn_exclusive_sum_i32(int64_t n, const int32_t *in, int32_t *out, int32_t *status, void *workspace,
                                      size_t workspace_bytes, cgnn_stream_t stream) {
    CGNN_REQUIRE(n >= 0 && n < INT32_MAX, "cgnn_exclusive_sum_i32: n must be in [0, 2^31 - 1)");
    CGNN_REQUIRE(out != nullptr, "cgnn_exclusive_sum_i32: out is null");
    if (n == 0) {
        hipLaunchKernelGGL(fill_i32_value_kernel, dim3(1), dim3(1), 0, stream, out, (int64_t)1, 0);
        return check_launch("exclusive_sum");
    }
    CGNN_REQUIRE(in != nullptr, "cgnn_exclusive_sum_i32: in is null");
    if (workspace == nullptr || workspace_bytes < cgnn_exclusive_sum_workspace_bytes(n))
        return fail(CGNN_EWORKSPACE, "cgnn_exclusive_sum_i32: workspace too small");
    const int64_t tiles = ceil_div(n, kSumTile);
    int64_t *totals = static_cast<int64_t *>(workspace);
    hipLaunchKernelGGL(sum_tiles_kernel, dim3((unsigned)tiles), dim3(kBlock), 0, stream, in, n, totals);
    hipLaunchKernelGGL(sum_totals_kernel, dim3(1), dim3(kBlock), 0, stream, totals, tiles);
    hipLaunchKernelGGL(sum_apply_kernel, dim3((unsigned)tiles), dim3(kBlock), 0, stream, in, n, totals, out, status);
    return check_launch("exclusive_sum");
}

extern "C" int cgnn_sample_count(const cgnn_sample_graph *graph, int64_t n, const int64_t *frontier, int64_t fanout,
                                 int32_t *counts, int32_t *status, cgnn_stream_t stream) {
    int rc = check_graph(graph, "cgnn_sample_count");
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(n >= 0 && n < INT32_MAX, "cgnn_sample_count: n must be in [0, 2^31 - 1)");
    CGNN_REQUIRE(fanout >= 0, "cgnn_sample_count: the fan-out must not be negative");
    if (n == 0) return CGNN_OK;
    CGNN_REQUIRE(frontier && counts && status, "cgnn_sample_count: null array");
    LayerArgs a = layer_args(graph, n, frontier, fanout, status);
    a.counts = counts;
    hipLaunchKernelGGL(sample_count_kernel, dim3((unsigned)ceil_div(n, kBlock / kWave)), dim3(kBlock), 0, stream, a);
    return check_launch("sample_count");
}

extern "C" int cgnn_sample_fill(const cgnn_sample_graph *graph, int64_t n, const int64_t *frontier, int64_t fanout,
                                const int32_t *offsets, int64_t first_position, int64_t layer, uint64_t seed,
                                int64_t *neighbors, int64_t *sources, int64_t *picks, int32_t *status,
                                cgnn_stream_t stream) {
    int rc = check_graph(graph, "cgnn_sample_fill");
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(n >= 0 && n < INT32_MAX, "cgnn_sample_fill: n must be in [0, 2^31 - 1)");
    CGNN_REQUIRE(fanout >= 0, "cgnn_sample_fill: the fan-out must not be negative");
    if (n == 0) return CGNN_OK;
    CGNN_REQUIRE(frontier && offsets && neighbors && sources && picks && status, "cgnn_sample_fill: null array");
    LayerArgs a = layer_args(graph, n, frontier, fanout, status);
    a.offsets = offsets;
    a.first_position = first_position;
    a.layer = layer;
    a.seed = seed;
    a.neighbors = neighbors;
    a.sources = sources;
    a.picks = picks;
    hipLaunchKernelGGL(sample_fill_kernel, dim3((unsigned)ceil_div(n, kBlock / kWave)), dim3(kBlock), 0, stream, a);
    return check_launch("sample_fill");
}

extern "C" int cgnn_sample_relabel_begin(int64_t vertex_cnt, int64_t n_input, const int64_t *input, int32_t *local_of,
                                         int32_t *seen_at, int32_t *status, cgnn_stream_t stream) {
    CGNN_REQUIRE(vertex_cnt >= 0 && vertex_cnt < INT32_MAX && n_input >= 0 && n_input < INT32_MAX,
                 "cgnn_sample_relabel_begin: sizes must be in [0, 2^31 - 1)");
    CGNN_REQUIRE(status != nullptr, "cgnn_sample_relabel_begin: status is null");
    hipLaunchKernelGGL(fill_i32_value_kernel, dim3(1), dim3(1), 0, stream, status, (int64_t)1, 0);
    if (vertex_cnt > 0) {
        CGNN_REQUIRE(local_of && seen_at, "cgnn_sample_relabel_begin: null table");
        hipLaunchKernelGGL(fill_i32_value_kernel, dim3(blocks_for(vertex_cnt)), dim3(kBlock), 0, stream, local_of,
                           vertex_cnt, kUnseen);
        hipLaunchKernelGGL(fill_i32_value_kernel, dim3(blocks_for(vertex_cnt)), dim3(kBlock), 0, stream, seen_at,
                           vertex_cnt, kUnseen);
    }
    if (n_input > 0) {
        CGNN_REQUIRE(input != nullptr, "cgnn_sample_relabel_begin: input is null");
        hipLaunchKernelGGL(relabel_seeds_kernel, dim3(blocks_for(n_input)), dim3(kBlock), 0, stream, input, n_input,
                           vertex_cnt, local_of, status);
    }
    return check_launch("sample_relabel_begin");
}

extern "C" size_t cgnn_sample_relabel_workspace_bytes(int64_t total) {
    if (total <= 0) return 0;
    return 2 * align_up((size_t)total * sizeof(int32_t), 256) + occupancy_scan_bytes(total);
}

extern "C" int cgnn_sample_relabel(int64_t total, const int64_t *neighbors, int64_t base, int32_t *local_of,
                                   int32_t *seen_at, int64_t *samples, int64_t *numbers, int64_t *new_count,
                                   void *workspace, size_t workspace_bytes, cgnn_stream_t stream) {
    CGNN_REQUIRE(total >= 0 && total < INT32_MAX && base >= 0 && base + total < INT32_MAX,
                 "cgnn_sample_relabel: sizes must stay below 2^31 - 1");
    CGNN_REQUIRE(new_count != nullptr, "cgnn_sample_relabel: new_count is null");
    if (total == 0) {
        hipLaunchKernelGGL(fill_i32_value_kernel, dim3(1), dim3(1), 0, stream, reinterpret_cast<int32_t *>(new_count),
                           (int64_t)2, 0);
        return check_launch("sample_relabel");
    }
    CGNN_REQUIRE(neighbors && local_of && seen_at && samples && numbers, "cgnn_sample_relabel: null array");
    if (workspace == nullptr || workspace_bytes < cgnn_sample_relabel_workspace_bytes(total))
        return fail(CGNN_EWORKSPACE, "cgnn_sample_relabel: workspace too small");
    const size_t col = align_up((size_t)total * sizeof(int32_t), 256);
    char *wbase = static_cast<char *>(workspace);
    int32_t *introduces = reinterpret_cast<int32_t *>(wbase);
    int32_t *rank = reinterpret_cast<int32_t *>(wbase + col);
    void *scan_scratch = wbase + 2 * col;
    const unsigned blocks = blocks_for(total);
    hipLaunchKernelGGL(relabel_first_kernel, dim3(blocks), dim3(kBlock), 0, stream, neighbors, total, local_of, seen_at);
    hipLaunchKernelGGL(relabel_flag_kernel, dim3(blocks), dim3(kBlock), 0, stream, neighbors, total, local_of, seen_at,
                       introduces);
    int rc = occupancy_scan(introduces, total, rank, scan_scratch, stream);
    if (rc != CGNN_OK) return rc;
    hipLaunchKernelGGL(relabel_assign_kernel, dim3(blocks), dim3(kBlock), 0, stream, neighbors, total, introduces, rank,
                       base, local_of, samples, new_count);
    hipLaunchKernelGGL(relabel_lookup_kernel, dim3(blocks), dim3(kBlock), 0, stream, neighbors, total, local_of, seen_at,
                       numbers);
    return check_launch("sample_relabel");
}

// ------------------------------------------------------- layers of a bounded size ----
namespace {

struct BoundedLayout {
    size_t number_of, samples, state, status, total;
    size_t slots[CGNN_SAMPLE_MAX_BOUNDED], counts[CGNN_SAMPLE_MAX_BOUNDED], before[CGNN_SAMPLE_MAX_BOUNDED];
    int64_t n_cap[CGNN_SAMPLE_MAX_BOUNDED], chunks[CGNN_SAMPLE_MAX_BOUNDED];
    int32_t chunk[CGNN_SAMPLE_MAX_BOUNDED];
    int64_t samples_cap;
};

// The most slots a call may have in all its layers: 128 MB of them.  They are for the longest lists that the fan-outs
// allow, and are written and ranked however short the lists are.  With lists of two entries over 2 million vertices,
// the worst case, this form takes 132 us at 2^25 slots (16,384 seeds, fan-outs 64 and 32: 100,000 edges; layer by layer
// 311 us), 204 at 2^26 (303) and 348 at 2^27 (346), but holds 160, 294 and 525 MB where the layers take 23, 23 and 30.
constexpr int64_t kMostSlots = int64_t(1) << 25;

// false: the fan-outs do not bound the call well enough, or it has too many layers
bool bounded_layout(int64_t vertex_cnt, int64_t n_input, int layers, const int64_t *fanouts, BoundedLayout *L) {
    if (layers < 1 || layers > CGNN_SAMPLE_MAX_BOUNDED || n_input < 1 || vertex_cnt < 1) return false;
    size_t at = 0;
    auto take = [&](int64_t ints) {
        const size_t here = at;
        at += align_up((size_t)ints * sizeof(int32_t), 256);
        return here;
    };
    L->number_of = take(vertex_cnt);
    L->state = take(4 * (layers + 1));
    L->status = take(2);
    int64_t n = n_input, all = 0;
    L->samples_cap = n_input;
    for (int k = 0; k < layers; ++k) {
        if (fanouts[k] < 1 || fanouts[k] > kRegPicks || n > kMostSlots / fanouts[k]) return false;
        const int64_t slots = n * fanouts[k];
        all += slots;
        if (all > kMostSlots) return false;
        L->n_cap[k] = n;
        const int64_t workgroup = kBlock / bounded_lanes(fanouts[k]) * fanouts[k];  // a multiple of four slots, at most 256
        L->chunk[k] = (int32_t)(kChunk / workgroup * workgroup);
        L->chunks[k] = ceil_div(slots, L->chunk[k]);
        L->slots[k] = take(slots);
        L->counts[k] = L->chunks[k] <= kCountedChunks ? take(2 * L->chunks[k]) : 0;
        L->before[k] = take(2 * L->chunks[k]);
        n = slots < vertex_cnt ? slots : vertex_cnt;  // a layer adds every vertex once
        L->samples_cap += n;
    }
    if (L->samples_cap > n_input + vertex_cnt) L->samples_cap = n_input + vertex_cnt;
    L->samples = take(L->samples_cap);
    L->total = at;
    return true;
}

BoundedArgs bounded_args(const cgnn_sample_graph *graph, int64_t n_input, const int64_t *input, int layers, const int64_t *fanouts,
                         uint64_t seed, const BoundedLayout &L, void *workspace) {
    BoundedArgs a{};
    char *base = static_cast<char *>(workspace);
    auto ints = [&](size_t at) { return reinterpret_cast<int32_t *>(base + at); };
    a.g = graph_of(graph);
    a.n_input = n_input;
    a.input = input;
    a.number_of = ints(L.number_of), a.samples = ints(L.samples);
    a.state = ints(L.state), a.status = ints(L.status);
    a.seed = seed;
    a.layers = layers;
    for (int k = 0; k < layers; ++k) {
        a.at[k] = BoundedLayer{fanouts[k], L.n_cap[k], L.chunk[k], ints(L.slots[k]),
                               L.chunks[k] <= kCountedChunks ? reinterpret_cast<uint64_t *>(base + L.counts[k]) : nullptr,
                               reinterpret_cast<uint64_t *>(base + L.before[k])};
        a.first_chunk[k + 1] = a.first_chunk[k] + L.chunks[k];
    }
    return a;
}

}  // namespace

extern "C" size_t cgnn_sample_layers_workspace_bytes(int64_t vertex_cnt, int64_t n_input, int layers, const int64_t *fanouts) {
    BoundedLayout L;
    return fanouts != nullptr && vertex_cnt < INT32_MAX && bounded_layout(vertex_cnt, n_input, layers, fanouts, &L) ? L.total : 0;
}

extern "C" int cgnn_sample_layers(const cgnn_sample_graph *graph, int64_t n_input, const int64_t *input, int layers,
                                  const int64_t *fanouts, uint64_t seed, int32_t *summary, void *workspace,
                                  size_t workspace_bytes, cgnn_stream_t stream) {
    int rc = check_graph(graph, "cgnn_sample_layers");
    if (rc != CGNN_OK) return rc;
    BoundedLayout L;
    CGNN_REQUIRE(input && fanouts && summary, "cgnn_sample_layers: null array");
    if (!bounded_layout(graph->vertex_cnt, n_input, layers, fanouts, &L))
        return fail(CGNN_EUNSUPPORTED, "cgnn_sample_layers: these fan-outs do not bound the call (see the size query)");
    if (workspace == nullptr || workspace_bytes < L.total) return fail(CGNN_EWORKSPACE, "cgnn_sample_layers: workspace too small");
    BoundedArgs a = bounded_args(graph, n_input, input, layers, fanouts, seed, L, workspace);
    a.summary = summary;
    summary[3] = 0;
    hipLaunchKernelGGL(bounded_begin_kernel, dim3(blocks_for(graph->vertex_cnt)), dim3(kBlock), 0, stream, a);
    for (int k = 0; k < layers; ++k) {
        a.layer = k;
        const int lanes = bounded_lanes(fanouts[k]);
        const bool counted = a.at[k].counts != nullptr;
        const auto fill = lanes == 16   ? (counted ? bounded_fill_kernel<16, true> : bounded_fill_kernel<16, false>)
                          : lanes == 32 ? (counted ? bounded_fill_kernel<32, true> : bounded_fill_kernel<32, false>)
                                        : (counted ? bounded_fill_kernel<kWave, true> : bounded_fill_kernel<kWave, false>);
        const dim3 chunks((unsigned)L.chunks[k]);
        hipLaunchKernelGGL(fill, dim3((unsigned)ceil_div(L.n_cap[k], kBlock / lanes)), dim3(kBlock), 0, stream, a);
        if (!counted) hipLaunchKernelGGL(bounded_count_kernel, chunks, dim3(kBlock), 0, stream, a);
        hipLaunchKernelGGL(counted ? bounded_assign_kernel<true> : bounded_assign_kernel<false>, chunks, dim3(kBlock), 0, stream, a);
    }
    return check_launch("sample_layers");
}

extern "C" int cgnn_sample_layers_write(const cgnn_sample_graph *graph, int64_t n_input, const int64_t *input, int layers,
                                        const int64_t *fanouts, int64_t samples, int64_t edges, int64_t *out_samples,
                                        int64_t *out_source, int64_t *out_neighbor, void *workspace, size_t workspace_bytes,
                                        cgnn_stream_t stream) {
    int rc = check_graph(graph, "cgnn_sample_layers_write");
    if (rc != CGNN_OK) return rc;
    BoundedLayout L;
    CGNN_REQUIRE(input && fanouts && bounded_layout(graph->vertex_cnt, n_input, layers, fanouts, &L),
                 "cgnn_sample_layers_write: not the arguments of cgnn_sample_layers");
    CGNN_REQUIRE(samples >= n_input && samples <= L.samples_cap && edges >= 0, "cgnn_sample_layers_write: sizes are those of the summary");
    CGNN_REQUIRE(out_samples && (edges == 0 || (out_source && out_neighbor)), "cgnn_sample_layers_write: null array");
    if (workspace == nullptr || workspace_bytes < L.total) return fail(CGNN_EWORKSPACE, "cgnn_sample_layers_write: workspace too small");
    BoundedArgs a = bounded_args(graph, n_input, input, layers, fanouts, 0, L, workspace);
    a.out_samples = out_samples, a.out_source = out_source, a.out_neighbor = out_neighbor;
    hipLaunchKernelGGL(bounded_write_kernel, dim3((unsigned)(a.first_chunk[layers] + ceil_div(samples, kBlock))), dim3(kBlock), 0,
                       stream, a);
    return check_launch("sample_layers_write");
}
