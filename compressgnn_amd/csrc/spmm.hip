// CSR SpMM for gfx950 (wave64): Y (+)= A * X with dense row-major X, Y of width F.
//
// Geometry shared by all kernels here.  A "lane group" of LPR consecutive lanes
// (LPR a power of two, 4..64) owns one output row at a time; lane l of the group
// holds VEC consecutive features starting at (tile*LPR + l)*VEC for TILES tiles, so a
// group reads and writes LPR*VEC*sizeof(T) contiguous bytes per tile (512 B per wave
// instruction when VEC*sizeof(T) = 16, i.e. global_load_dwordx4 on every lane).
// Features beyond LPR*VEC*TILES are covered by blockIdx.y.
//
// The entries of a row (column, value, row) are loaded once per lane group, one entry per
// lane with a coalesced load, and handed to all lanes of the group through the LDS
// crossbar (ds_bpermute); the gathers of a round are issued together, none behind the end
// of the row.  Loading every entry in every lane made the kernels bound by vector
// instruction issue (address arithmetic), not by memory.
//
// Two schedules:
//   * row schedule  -- a lane group per row, entries summed in ascending order; the
//     result is bit-identical to the sequential CPU sum of the reference
//     (src/runtime/csrc/sparse/cpu/spmm_cpu.cpp:48-68): products and sums are rounded
//     separately (this file is built with -ffp-contract=off).
//   * nnz schedule  -- a lane group per run of about seg_nnz consecutive non-zeros (rows
//     of any length cost the same).  Rows of at most seg_nnz entries always lie inside
//     one run and are summed exactly as in the row schedule.  Longer rows are cut at
//     multiples of seg_nnz: the part that continues into the next run is a carry.  The
//     lane groups of one workgroup first add their carries of the same row in LDS, in
//     ascending order, so at most one carry row per output row and workgroup reaches
//     memory.  spmm_carry_reduce_kernel sums the carries of very long rows 64 at a
//     time, level by level (a row with a million entries is not walked by one lane
//     group), and spmm_fixup_kernel adds what is left, in ascending order.
//     Every output element receives its additions in a fixed order (where an atomic add
//     is used it is the only addition to that element), so results are reproducible run
//     to run.
//
//   * workgroup runs -- the nnz schedule without a pass behind it, for blocks that bring a table of their
//     runs (cgnn_csr.wg_runs).  The entries are dealt to workgroups (wg_len positions each, a row of at
//     most that many entries never divided) and a workgroup's share to its lane groups, so the pieces of a
//     row meet in LDS and the row is written there, once.  A row longer than wg_len leaves one piece
//     per workgroup in memory; the workgroup that finds itself the last to arrive at the row adds the pieces
//     up, in ascending order, so the sum does not depend on which one that is.
//
// Modes: VAL (stored values), ADD (the same, added to what Y holds), UNIT (all values 1: member lists, whose rows are gathered once), RELU_MASK (unit values, gathered
// rows zeroed where a second matrix is <= 0), SIGN_MASK (the same, the mask a bit per element), ROW_MASK (unit values, the finished
// rows of Y zeroed by a bit per element), DUAL (columns below `split` gather from
// X, the others from X1; the two partial sums are kept apart and combined as
// (0 + sum1) + sum0, which is what two successive accumulating products give).
//
// X may alias Y when accumulating (rule levels are updated in place, reference
// layer/CompressgnnSPMM.py:56-58), so X and Y carry no __restrict__; a row that is
// written is never gathered in the same launch (levels only read earlier levels).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"

namespace cgnn {
namespace {

constexpr int kUnroll = 4;        // gathers in flight per lane and tile, nnz schedule (with 7 waves per SIMD;
                                  // 8 in flight with 5 waves measured the same)
constexpr int kMidRound = 8, kDeepRound = 16;  // ... where a launch has few workgroups (launch_nnz)
// Of the nnz kernel on an MI355X at once, with kUnroll.  Not asked of the device: run lengths follow from it, and with them
// the workspaces of a product and where its sums are divided, which callers plan without a device as well.
constexpr int64_t kResidentWorkgroups = 256 * 7;
constexpr int kRowUnroll = 4;     // same for the row schedule (8: 9 % slower on web-graph out-lists, 2: 13 %, 16: 38 %)
constexpr int kXcds = 8;          // accelerator dies of an MI355X, each with its own L2
constexpr int kDefaultSeg = 64;   // non-zeros per lane group in the nnz schedule

// Where the runs of the nnz kernel come from: positions that are multiples of the run length, the table of
// workgroup runs, or the same rule worked out by every lane group (member lists, which are new with every call: a launch for
// their table would cost more than the few dependent loads) or by every workgroup from 64-bit arrays, the rows of its entries
// with it (cgnn_spmm_once).
enum { WGRUNS_NONE = 0, WGRUNS_TABLE = 1, WGRUNS_COMPUTED = 2, WGRUNS_ONCE = 3 };
enum { MODE_VAL = 0, MODE_UNIT = 1, MODE_RELU_MASK = 2, MODE_DUAL = 3, MODE_SIGN_MASK = 4, MODE_ADD = 5, MODE_ROW_MASK = 6 };
constexpr bool has_values(int mode) { return mode == MODE_VAL || mode == MODE_ADD; }

template <typename T, int VEC>
struct alignas(sizeof(T) * VEC) Pack {
    T v[VEC];
};

template <typename T>
struct SpmmArgs {
    const int32_t *rowptr;
    const int32_t *colidx;
    const int32_t *rowidx;
    const int32_t *rowmap;  // row schedule: stored row g is row rowmap[g] of Y (or NULL)
    const T *val;
    const T *X;   // gathered matrix (may alias Y)
    const T *X1;  // MODE_DUAL: source of the columns >= split
    const T *M;   // MODE_RELU_MASK: rows of X are zeroed where M <= 0
    const uint32_t *signs;  // MODE_SIGN_MASK: the same with one bit per element (set: keep), sign_words words per row
    const uint32_t *row_signs;  // MODE_ROW_MASK: such words for the rows of Y; also asked by the passes that add carries
    int32_t sign_words;
    T *Y;
    int32_t *carry_row;  // [nseg] row a run carries into, or -1
    T *carry;            // [nseg x F]
    int32_t *carry_row_out;  // spmm_carry_reduce_kernel: the next, 32 times shorter level
    T *carry_out;
    int64_t F;
    int32_t rows;
    int32_t nnz;
    int32_t nseg;
    int32_t seg_nnz;
    int32_t split;
    int32_t accumulate;
    // Runs whose carries the nnz kernel that wrote carry_row/carry has merged (see kMerged and
    // merged_runs), or 1 for the plain list a reduction level writes.
    int32_t merge_stride;
    int32_t stretch_log2;  // log2 of the workgroups per XCD stretch (see logical_block); set at launch
    int32_t blocks;        // workgroups with work (the grid rounds this up to a multiple of kXcds)
    const int32_t *cut_rows;    // spmm_fixup_rows_kernel: the stored rows that the runs cut, ascending
    const int32_t *empty_rows;  // and the stored rows without entries
    int32_t n_cut_rows, n_empty_rows;
    const int32_t *run_start;   // nnz schedule: first non-zero of every run, [nseg + 1], or NULL (run_boundary)
    int32_t *arrivals;          // workgroup runs: per workgroup and feature tile, the pieces stored so far of the row
                                // that goes on behind it; zero before and after every launch
    int32_t wg_len;             // workgroup runs: non-zeros per workgroup (run_start is the table of cgnn_csr.wg_runs, or NULL)
    int32_t keep;               // ... a row of at most this many entries is never divided, whatever the lengths
    int32_t find_empty;         // ... the rows without entries are found from rowptr, not from a list
    int32_t mean;               // MODE_UNIT, plain runs: every row is divided by its number of entries
    const int64_t *rowptr64, *col64;  // WGRUNS_ONCE: in place of rowptr, colidx and rowidx; nnz is the length of col64
};

// An entry of the table of workgroup runs is the first non-zero of a run, with this bit set when the row
// found there began before it.
constexpr int32_t kRowGoesOn = INT32_MIN;

// Where lane group g of workgroup w begins, as such an entry (the rule stands at cgnn_csr.wg_runs).
__device__ __forceinline__ int32_t wg_run_begin(const int32_t *rowptr, const int32_t *rowidx, int32_t nnz, int32_t wg_len,
                                                int32_t groups, int32_t keep, int64_t w, int g) {
    // e moved back to the start of its row when the row has at most `whole` entries
    auto begin_of = [&](int64_t e, int whole) -> int32_t {
        if (e >= nnz) return nnz;
        const int r = rowidx[e];
        const int s0 = rowptr[r];
        return rowptr[r + 1] - s0 <= whole ? s0 : (s0 < e ? (int32_t)e | kRowGoesOn : (int32_t)e);
    };
    const int run_len = wg_len / groups;
    const int32_t b0 = begin_of(w * wg_len, wg_len > keep ? wg_len : keep);
    if (g == 0) return b0;
    const int32_t b1 = begin_of((w + 1) * wg_len, wg_len > keep ? wg_len : keep);
    const int32_t first = b0 & ~kRowGoesOn, end = b1 & ~kRowGoesOn;
    const int32_t e = first + g * ((end - first + groups - 1) / groups);
    return e >= end ? b1 : begin_of(e, run_len > keep ? run_len : keep);
}

// carry_row values below zero: the run carries nothing, or its carry was added to that
// of an earlier run of the same workgroup (the row of Y is the one of that earlier run).
constexpr int kNoCarry = -1;
constexpr int kMerged = -2;

// Global memory is read and written in packs that need the alignment of one element only (the
// hardware takes a 16-byte access at any multiple of four bytes): rows of a width that is no
// whole number of packs begin anywhere.
template <typename T, int VEC>
struct Unaligned {
    typedef T type __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
};
template <typename T>
struct Unaligned<T, 1> {
    typedef T type;
};

template <typename T, int VEC>
__device__ __forceinline__ Pack<T, VEC> to_pack(const typename Unaligned<T, VEC>::type &v) {
    Pack<T, VEC> x;
    if constexpr (VEC == 1) x.v[0] = v;
    else
#pragma unroll
        for (int i = 0; i < VEC; ++i) x.v[i] = v[i];
    return x;
}
template <typename T, int VEC>
__device__ __forceinline__ typename Unaligned<T, VEC>::type of_pack(const Pack<T, VEC> &x) {
    typename Unaligned<T, VEC>::type v;
    if constexpr (VEC == 1) v = x.v[0];
    else
#pragma unroll
        for (int i = 0; i < VEC; ++i) v[i] = x.v[i];
    return v;
}

template <typename T, int VEC>
__device__ __forceinline__ Pack<T, VEC> load_pack(const T *p) {
    return to_pack<T, VEC>(*reinterpret_cast<const typename Unaligned<T, VEC>::type *>(p));
}
// Streaming load for rows that this launch reads once.
template <typename T, int VEC>
__device__ __forceinline__ Pack<T, VEC> load_pack_stream(const T *p) {
    return to_pack<T, VEC>(__builtin_nontemporal_load(reinterpret_cast<const typename Unaligned<T, VEC>::type *>(p)));
}
template <typename T, int VEC>
__device__ __forceinline__ void store_pack(T *p, const Pack<T, VEC> &x) {
    *reinterpret_cast<typename Unaligned<T, VEC>::type *>(p) = of_pack<T, VEC>(x);
}
// Streaming store for rows that are written once and not read again by this launch.
template <typename T, int VEC>
__device__ __forceinline__ void store_pack_stream(T *p, const Pack<T, VEC> &x) {
    __builtin_nontemporal_store(of_pack<T, VEC>(x), reinterpret_cast<typename Unaligned<T, VEC>::type *>(p));
}

// First feature of the pack that starts at multiple `f` of VEC: where F is no whole number of packs
// the last pack of a row is moved back to end with the row and overlaps the one before it.  Both
// lanes then compute the same values for the shared elements and store them with one
// instruction of one wave (pick_shape allows the overlap for rows of one tile only).
template <int VEC>
__device__ __forceinline__ int64_t pack_start(int64_t F, int64_t f) {
    return VEC > 1 && f > F - VEC ? F - VEC : f;
}

// Per-lane feature offsets of the TILES tiles; foff[t] < 0 marks a tile beyond F.
template <int VEC, int LPR, int TILES>
__device__ __forceinline__ void feature_offsets(int64_t F, int lane, int64_t foff[TILES]) {
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        int64_t f = ((int64_t)(blockIdx.y * TILES + t) * LPR + lane) * VEC;
        foff[t] = f < F ? pack_start<VEC>(F, f) : -1;
    }
}

// The value of the lane at byte address `from`, through the LDS crossbar.  Doubles cross it as two halves: loading every entry
// in every lane instead, products of double int64 blocks took, web graphs, us, so / with the crossbar (and in one launch):
// 6,000 vertices of 14 features, in-lists, 20.2 / 13.9, 50,001 of 32 61 / 36, 325,557 of 64 330 / 252.
template <typename T>
__device__ __forceinline__ T from_lane(int from, T v) {
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, __builtin_amdgcn_ds_bpermute(from, __builtin_bit_cast(int, v)));
    } else {
        struct Halves {
            int lo, hi;
        };
        const Halves h = __builtin_bit_cast(Halves, v);
        return __builtin_bit_cast(T, Halves{__builtin_amdgcn_ds_bpermute(from, h.lo), __builtin_amdgcn_ds_bpermute(from, h.hi)});
    }
}

// What a gather of one feature tile brings: the pack of X, and what decides which of its elements count.  Loads only: they
// stand in a branch of their own (no gathers behind the end of a row), and what used the loaded values there would have to
// wait for them before the next gather of the round is asked for -- four waits one after the other, which doubled the time of
// sums that are a chain of rounds (with sign words, us, so / as it stands: 30,011 rows of 256 features 43 / 27, 100,003 of 100
// 41 / 28, 1,000,003 of 188 211 / 188; without a mask 23, 23 and 177).
template <typename T, int VEC, int MODE>
struct Gathered {
    Pack<T, VEC> x;
    Pack<T, MODE == MODE_RELU_MASK ? VEC : 1> m;  // MODE_RELU_MASK: the rows that decide
    uint32_t word, next;                          // MODE_SIGN_MASK: the word the pack's bits begin in, and the one behind

    // the pack, zeroed where the mask drops an element
    __device__ __forceinline__ Pack<T, VEC> masked(int64_t foff) const {
        Pack<T, VEC> o = x;
        if constexpr (MODE == MODE_SIGN_MASK) {
            const uint32_t bits = __builtin_amdgcn_alignbit(next, word, (uint32_t)foff & 31u);
#pragma unroll
            for (int i = 0; i < VEC; ++i) o.v[i] = ((bits >> i) & 1u) ? o.v[i] : T(0);
        }
        if constexpr (MODE == MODE_RELU_MASK)
#pragma unroll
            for (int i = 0; i < VEC; ++i) o.v[i] = (m.v[i] <= T(0)) ? T(0) : o.v[i];
        return o;
    }
};

// kRowBytes: what the lanes of a row span.  Gather one feature tile of column c (source chosen by `src` in MODE_DUAL).
template <typename T, int VEC, int MODE, int kRowBytes>
__device__ __forceinline__ Gathered<T, VEC, MODE> gather(const SpmmArgs<T> &a, int c, int src, int64_t foff) {
    Gathered<T, VEC, MODE> g;
    if (foff < 0) {
#pragma unroll
        for (int i = 0; i < VEC; ++i) g.x.v[i] = T(0);
        if constexpr (MODE == MODE_SIGN_MASK) g.word = g.next = 0;
        if constexpr (MODE == MODE_RELU_MASK) g.m = g.x;
        return g;
    }
    const T *base = a.X;
    if constexpr (MODE == MODE_DUAL) {
        // both pointers are read first and chosen between as values (a choice between the two
        // fields of the argument block becomes a vector load of the chosen field, and a wait)
        const T *first = a.X, *second = a.X1;
        base = src ? second : first;
        c -= src ? a.split : 0;
    }
    const int64_t off = (int64_t)c * (int32_t)a.F + foff;  // F < 2^31: one 32 x 32 -> 64 bit multiply
    // Rows that are gathered once (member lists, which the modes without values exist for) are not kept in the
    // caches -- unless they are shorter than a cache line, whose other half is a row that is still to come (16
    // features, 10^6 rows: 44 us so, 32 us kept).  A choice at compile time: the compiler merges the two loads of a
    // branch into one that is kept.  Kept rows cost the kernel that writes next most: behind the means of 2.4 M rows
    // the spread of 256 features took 725 us for 485 and the gradient of the means 283 us for 175.
    if constexpr ((MODE == MODE_RELU_MASK || MODE == MODE_SIGN_MASK || MODE == MODE_UNIT || MODE == MODE_ROW_MASK) && kRowBytes > 128)
        g.x = load_pack_stream<T, VEC>(base + off);
    else
        g.x = load_pack<T, VEC>(base + off);
    if constexpr (MODE == MODE_SIGN_MASK) {
        const uint32_t *words = a.signs + (int64_t)c * a.sign_words;
        const int at = (int)(foff >> 5);
        g.word = words[at];
        g.next = 0;  // not a copy of the word, which would have to be waited for
        // VEC divides 32, so the bits of one pack lie in one word, unless the pack was moved back
        if (VEC > 1 && (a.F & (VEC - 1)) != 0) g.next = words[min(at + 1, a.sign_words - 1)];
    }
    if constexpr (MODE == MODE_RELU_MASK) g.m = load_pack_stream<T, VEC>(a.M + off);
    return g;
}

// MODE_ROW_MASK: the bits of a row of Y for one pack.  A row whose members are all masked alike (the gradient of a ReLU behind rows
// that are copies of one representative) is summed unmasked and masked once: the same value, element by element, and the words are
// one row per row of Y instead of one per member, which is a cache line a member however few of its bytes count (2,449,029 rows of
// 256 features into 41,000: 503 us with a mask per member, 462 us so; the rows and their words 494, 483).
template <int VEC>
struct RowMask {
    uint32_t word = ~0u, next = ~0u;

    __device__ __forceinline__ void load(const uint32_t *signs, int32_t sign_words, int64_t F, int row, int64_t f) {
        const uint32_t *words = signs + (int64_t)row * sign_words;
        const int at = (int)(f >> 5);
        word = words[at];
        next = 0;  // as in gather()
        if (VEC > 1 && (F & (VEC - 1)) != 0) next = words[min(at + 1, sign_words - 1)];
    }
    template <typename T>
    __device__ __forceinline__ void apply(Pack<T, VEC> &x, int64_t f) const {
        const uint32_t bits = __builtin_amdgcn_alignbit(next, word, (uint32_t)f & 31u);
#pragma unroll
        for (int i = 0; i < VEC; ++i) x.v[i] = ((bits >> i) & 1u) ? x.v[i] : T(0);
    }
};

// Accumulator of one output row.  MODE_DUAL keeps the sums over the two sources apart: the
// entries of a row are sorted by column, so those of the first source come first; when the
// first entry of the second source arrives the running sum is put aside and started anew.
template <typename T, int VEC, int TILES, int MODE>
struct Acc {
    Pack<T, VEC> a0[TILES];                          // running sum
    Pack<T, VEC> a1[MODE == MODE_DUAL ? TILES : 1];  // MODE_DUAL: finished sum over the first source
    bool second_source;                              // MODE_DUAL: a1 is in use

    __device__ __forceinline__ void clear() {
        second_source = false;
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                a0[t].v[i] = T(0);
                if constexpr (MODE == MODE_DUAL) a1[t].v[i] = T(0);
            }
    }
    // entry with gathered tiles g at features foff, value w, from source `src` (0 or 1)
    __device__ __forceinline__ void add(const Gathered<T, VEC, MODE> g[TILES], const int64_t foff[TILES], T w, int src) {
        if constexpr (MODE == MODE_DUAL) {
            // At most once per row, so the whole wave jumps over it nearly always.  Written
            // with value selects under a wave-uniform branch: a branch per lane would be
            // turned into selects on every entry.
            const bool change = src != 0 && !second_source;
            if (__ballot(change)) {
#pragma unroll
                for (int t = 0; t < TILES; ++t)
#pragma unroll
                    for (int i = 0; i < VEC; ++i) {
                        a1[t].v[i] = change ? a0[t].v[i] : a1[t].v[i];
                        a0[t].v[i] = change ? T(0) : a0[t].v[i];
                    }
                second_source = second_source || change;
            }
        }
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const Pack<T, VEC> x = g[t].masked(foff[t]);
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                if constexpr (has_values(MODE) || MODE == MODE_DUAL) a0[t].v[i] = a0[t].v[i] + x.v[i] * w;
                else a0[t].v[i] = a0[t].v[i] + x.v[i];
            }
        }
    }
    // the row's value on top of `base`: (base + sum1) + sum0 in MODE_DUAL, base + sum otherwise
    __device__ __forceinline__ T total(T base, int t, int i) const {
        if constexpr (MODE == MODE_DUAL) {
            const T sum0 = second_source ? a1[t].v[i] : a0[t].v[i];
            const T sum1 = second_source ? a0[t].v[i] : T(0);
            return (base + sum1) + sum0;
        } else {
            return base + a0[t].v[i];
        }
    }
};

// Y[row] = (MODE_ADD ? Y[row] : 0) + acc
template <typename T, int VEC, int TILES, int MODE>
__device__ __forceinline__ void write_row(T *Y, int64_t F, int row, const int64_t foff[TILES],
                                          const Acc<T, VEC, TILES, MODE> &acc, T divisor = T(1),
                                          const RowMask<VEC> *mask = nullptr) {
    T *yrow = Y + (int64_t)row * F;
    // Whether the row is added to is known at compile time: a load of Y in the block that closes a row inside a run of
    // the nnz schedule would have to be waited for, with everything asked for before it, on every path behind the block.
    constexpr bool accumulate = MODE == MODE_ADD;
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
        if (foff[t] < 0) continue;
        Pack<T, VEC> o;
        if (accumulate) {
            o = load_pack<T, VEC>(yrow + foff[t]);
        } else {
#pragma unroll
            for (int i = 0; i < VEC; ++i) o.v[i] = T(0);
        }
#pragma unroll
        for (int i = 0; i < VEC; ++i) o.v[i] = acc.total(o.v[i], t, i);
        if constexpr (MODE == MODE_UNIT)
#pragma unroll
            for (int i = 0; i < VEC; ++i) o.v[i] = o.v[i] / divisor;
        if constexpr (MODE == MODE_ROW_MASK) mask[t].template apply<T>(o, foff[t]);
        // Rows of the plain product that go out element by element are short or no whole lines, and the few of a small
        // graph are read next: kept (8 features over 4,000 vertices 4.1 us streaming, 3.7 kept; in packs 64
        // features over 50,001 vertices 12.3 us kept, 11.4 streaming).
        if constexpr (accumulate || (MODE == MODE_VAL && VEC == 1)) store_pack<T, VEC>(yrow + foff[t], o);
        else store_pack_stream<T, VEC>(yrow + foff[t], o);
    }
}

// Row of Y that stored row r stands for.
template <typename T>
__device__ __forceinline__ int out_row(const SpmmArgs<T> &a, int r) {
    return a.rowmap != nullptr ? a.rowmap[r] : r;
}

// Workgroups are dealt to the XCDs round robin.  XCD x takes every kXcds-th stretch of
// consecutive workgroups' worth of stored rows (or runs): rows that follow each other in the
// store (a locality order, or a natural order that has locality) meet in one L2, and every
// XCD gets the same mix of the matrix (one contiguous share each would leave the XCD with the
// least reuse to finish last).  A stretch holds kXcdStretchGroups lane groups, about what an
// XCD holds at a time at F = 128, so an XCD works on one region of the order at once (a
// quarter and twice that measured 1.5 % slower on the web graph, four times 20 %: too few
// stretches to even out).  Small launches take shorter stretches, at least
// kMinStretchesPerXcd per XCD.
constexpr int kXcdStretchGroups = 2048;
constexpr int kMinStretchesPerXcd = 6;

template <int GPB>
constexpr int xcd_stretch() {
    return kXcdStretchGroups / GPB > 0 ? kXcdStretchGroups / GPB : 1;
}

// log2 of the stretch (in workgroups) for a launch of `blocks` workgroups of GPB lane groups
template <int GPB>
int stretch_log2_for(int64_t blocks) {
    int lg = 0;
    while ((2 << lg) <= xcd_stretch<GPB>()) ++lg;
    while (lg > 0 && blocks < ((int64_t)kXcds * kMinStretchesPerXcd << lg)) --lg;
    return lg;
}

// Whole rounds of kXcds stretches are dealt first; what is left over is dealt the same way in
// stretches half as long, and so on down to single workgroups, so that no XCD is left with a
// whole stretch more than another.
template <typename T>
__device__ __forceinline__ int logical_block(const SpmmArgs<T> &a) {
    const int xcd = blockIdx.x % kXcds;
    int turn = blockIdx.x / kXcds;  // this workgroup's number on its XCD
    int base = 0, left = a.blocks;
    for (int lg = a.stretch_log2; lg > 0; --lg) {
        const int share = (left >> (lg + 3)) << lg;  // workgroups per XCD dealt in stretches of 2^lg  (kXcds = 2^3)
        if (turn < share) return base + ((((turn >> lg) * kXcds) + xcd) << lg) + (turn & ((1 << lg) - 1));
        turn -= share;
        base += share * kXcds;
        left -= share * kXcds;
    }
    return base + turn * kXcds + xcd;
}

// ---------------------------------------------------------------- row schedule --
template <typename T, int VEC, int LPR, int TILES, int MODE>
__global__ __launch_bounds__(kBlock) void spmm_row_kernel(SpmmArgs<T> a) {
    constexpr int GPB = kBlock / LPR;
    const int lane = threadIdx.x % LPR;
    int row = logical_block(a) * GPB + threadIdx.x / LPR;
    if constexpr (LPR == kWave) row = __builtin_amdgcn_readfirstlane(row);
    if (row >= a.rows) return;
    const int e0 = a.rowptr[row], e1 = a.rowptr[row + 1];
    row = out_row(a, row);  // from here on: the row of Y
    int64_t foff[TILES];
    feature_offsets<VEC, LPR, TILES>(a.F, lane, foff);
    Acc<T, VEC, TILES, MODE> acc;
    acc.clear();
    if (e0 == e1) {
        if constexpr (MODE != MODE_ADD) write_row<T, VEC, TILES, MODE>(a.Y, a.F, row, foff, acc);
        return;
    }
    constexpr int RU = LPR < kRowUnroll ? LPR : kRowUnroll;  // entries per round: no more than lanes to stage them
    // The lanes of the group load one entry each (one coalesced load per array for LPR
    // entries), and every entry is then handed to all lanes through the LDS crossbar:
    // no address arithmetic and no memory instruction per entry and lane for the indices.
    const int group_lane0 = 4 * ((threadIdx.x % kWave) - lane);  // byte address of the group's first lane
    // lanes beyond the width gather feature 0 again (never stored): no test per gather
    int64_t fld[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) fld[t] = foff[t] < 0 ? 0 : foff[t];
    for (int e = e0; e < e1; e += LPR) {
        int my_c = 0;
        T my_w = T(1);
        if (e + lane < e1) {
            my_c = a.colidx[e + lane];
            if (a.val) my_w = a.val[e + lane];
        }
        const int cnt = min(e1 - e, LPR);
        for (int u0 = 0; u0 < cnt; u0 += RU) {
            int c[RU];
            T w[RU];
#pragma unroll
            for (int u = 0; u < RU; ++u) {
                const int from = group_lane0 + 4 * (u0 + u);
                c[u] = __builtin_amdgcn_ds_bpermute(from, my_c);
                w[u] = from_lane(from, my_w);
            }
            // Entries of the second source are rare (columns that stand for rules): when the
            // wave has none in this round, the gathers need no choice of source per lane.
            bool second = false;
            if constexpr (MODE == MODE_DUAL) {
#pragma unroll
                for (int u = 0; u < RU; ++u) second = second || (u0 + u < cnt && c[u] >= a.split);
            }
            auto gather_and_add = [&](auto plain) {
                constexpr bool kPlain = decltype(plain)::value;  // every entry from the first source
                Gathered<T, VEC, MODE> x[RU][TILES];
#pragma unroll
                for (int u = 0; u < RU; ++u)
                    if (u0 + u < cnt) {  // no gathers behind the row's end: repeated ones still cost issue slots
#pragma unroll
                        for (int t = 0; t < TILES; ++t)
                            x[u][t] = gather<T, VEC, MODE, (int)(VEC * LPR * sizeof(T))>(a, c[u], kPlain ? 0 : c[u] >= a.split, fld[t]);
                    }
#pragma unroll
                for (int u = 0; u < RU; ++u)
                    if (u0 + u < cnt) acc.add(x[u], fld, w[u], kPlain ? 0 : c[u] >= a.split);
            };
            if (MODE != MODE_DUAL || __ballot(second) == 0) gather_and_add(std::true_type{});
            else gather_and_add(std::false_type{});
        }
    }
    write_row<T, VEC, TILES, MODE>(a.Y, a.F, row, foff, acc);
}

// ---------------------------------------------------------------- nnz schedule --
// Run s covers the non-zeros [run_boundary(s*K), run_boundary((s+1)*K)).  A boundary
// that falls inside a row of at most K entries is moved back to the start of that row,
// so such rows are never split (and are summed in the same order as the row schedule);
// only rows longer than K are cut, at multiples of K.  Runs hold fewer than 2K entries.
// Says that a loaded value is used here, so that the wait for it stands here and not at its first use.  In the run loop the
// first uses lie behind branches in which rows are stored; loads and stores are counted together, so a wait there
// also waits for the store to be acknowledged by memory.  With the waits in front -- one for the entries of a batch, one for
// the gathers of a round -- the store of a row that ended is under way together with the next round's gathers (forward
// + gradient with the rules multiplied out, us: 64 features over 50,001 vertices 36.9 -> 34.5, 32 over 100,003 45 -> 44).
// The two-source product of large graphs is bound by its traffic and took 364 us for 362 so, and the sums of short rows, whose
// gathers stand in no branch and are waited for one by one, 37.7 for 36 (10^6 rows of 16 features): these keep the waits
// where the compiler puts them.
__device__ __forceinline__ void arrive(int &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void arrive(uint32_t &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void arrive(float &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void arrive(double &v) { asm volatile("" : "+v"(v)); }
template <typename T, int VEC, int MODE>
__device__ __forceinline__ void arrive(Gathered<T, VEC, MODE> &g) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) arrive(g.x.v[i]);
    if constexpr (MODE == MODE_SIGN_MASK) arrive(g.word), arrive(g.next);
    if constexpr (MODE == MODE_RELU_MASK)
#pragma unroll
        for (int i = 0; i < VEC; ++i) arrive(g.m.v[i]);
}

template <typename T>
__device__ __forceinline__ int run_boundary(const SpmmArgs<T> &a, int e) {
    if (e >= a.nnz) return a.nnz;
    const int r = a.rowidx[e];
    const int s0 = a.rowptr[r];
    return (a.rowptr[r + 1] - s0 <= a.seg_nnz) ? s0 : e;
}

// The rows of a block given as 64-bit row pointers: entries count from rowptr[0], and pointers that are none do not lead out
// of the arrays.
struct WideRows {
    const int64_t *rowptr;
    int64_t first, last;  // the entries that belong to rows
    __device__ __forceinline__ int32_t at(int64_t r) const { return (int32_t)(max(first, min(last, rowptr[r])) - first); }
};

// Room for the entries of workgroup w: its wg_len, and those of a row that is moved to it as a whole.
inline __host__ __device__ int32_t once_room(int32_t wg_len, int32_t keep) { return wg_len + (wg_len > keep ? wg_len : keep); }

// Where workgroup w of WGRUNS_ONCE begins and the next one, as in the table, and row_of[e - begin]: the rows of the entries
// between.  A wave looks for the row at the first of its wg_len positions, 64 row pointers a step, until kNear rows are left;
// these and those behind them are read by all threads, which finds the rows at both ends, and mark their first entries;
// a running maximum spreads the marks.  pivot: row pointer lane * search_step(rows), asked for with the first loads there are.
//
// In place of a launch that made int32 arrays of the block, which the product then waited for: that cost 7.5 us, the launch
// boundary, and five dependent loads in front of a run (two now, of lines just read).  Web graphs, us, in-lists and out-lists,
// before / so: 6,000 vertices of 16 features 16.9 / 13.9 and 11.9 / 8.7, 50,001 of 16 23.5 / 19.3 and 21.8 / 15.9, 100,003 of 64
// 52.3 / 45.4 and 36.4 / 29.4, 325,557 of 128 264 / 253 and 197 / 181, of 8, 512 entries a workgroup, 83.5 / 82.9 and 72.2 /
// 63.2.  A search for each end of a stretch, down to the row, instead: in-lists of 325,557 vertices 266 us at
// 128 features; 16 row pointers a step 278.
constexpr int kNear = kBlock / 2;
// From this many rows between the two ends on (rows without entries, which may be any number) the rows are found from the entries,
// a search of them for each: a step of the walk over the rows waits for the one before, a search takes as many steps as the number of
// rows has bits.  us, all rows walked / so: 10^5 entries on both sides of 987,500 empty rows, 64 features 1,450 / 38; 1,000 in
// 10^6 rows at random, 1 feature 720 / 13; in-lists of 325,557 vertices of degree 1, 8 features 43 / 23.5, of degree 3 43.5 / 32.
// Lower bounds (two, four, eight steps) gain nothing there, and eight cost in-lists of 100,003 vertices of degree 9.8 1.5 % at
// 64 features.
constexpr int kWalked = 16 * kBlock;
__device__ __forceinline__ int search_step(int rows) { return (rows + kWave - 1) / kWave; }

template <typename T>
__device__ __forceinline__ void once_stretch(const SpmmArgs<T> &a, const WideRows &rows, int64_t w, int64_t pivot, int *row_of,
                                             int32_t &begin, int32_t &behind) {
    __shared__ int found[2], wave_count[2][kBlock / kWave], wave_max[kBlock / kWave];
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t dealt = rows.last - rows.first;
    const int32_t room = once_room(a.wg_len, a.keep);
    // the last row that begins at or before the place lies in [from, to), and row `from` does throughout
    int from = 0, to = a.rows;
    auto halve = [&](int step, int64_t start, int64_t place) {
        const bool at_or_before = lane == 0 || (from + (int64_t)step * lane < to && start - rows.first <= place);
        from += step * (__popcll(__ballot(at_or_before)) - 1);
        to = to - from > step ? from + step : to;
    };
    auto look = [&](int64_t place, int near) {
        while (to - from > near) {
            const int step = search_step(to - from);
            halve(step, rows.rowptr[min((int64_t)a.rows, from + (int64_t)step * lane)], place);
        }
        if (lane == 0) found[0] = from, found[1] = to;
    };
    const int64_t places[2] = {w * a.wg_len, (w + 1) * a.wg_len};
    if (wave == 0) {
        if (places[0] >= dealt) from = a.rows - 1;
        else if (to > kNear) halve(search_step(to), pivot, places[0]);
        look(places[0], kNear);
    }
    for (int k = threadIdx.x; k < room; k += kBlock) row_of[k] = -1;
    __syncthreads();
    from = found[0], to = found[1];
    int64_t r = (int64_t)from + threadIdx.x;
    int32_t s = r < a.rows ? rows.at(r) : 0, e = r < a.rows ? rows.at(r + 1) : 0;
    const unsigned long long before_first = __ballot(r < to && s <= places[0]), before_last = __ballot(r < a.rows && s <= places[1] && s < dealt);
    if (lane == 0) wave_count[0][wave] = __popcll(before_first), wave_count[1][wave] = __popcll(before_last);
    __syncthreads();
    int ahead[2] = {0, 0};
#pragma unroll
    for (int v = 0; v < kBlock / kWave; ++v) ahead[0] += wave_count[0][v], ahead[1] += wave_count[1][v];
    const int r0 = from + max(ahead[0], 1) - 1;
    int r1 = max(r0, from + ahead[1] - 1);
    if (ahead[1] == kBlock) {  // short rows, or many without entries
        if (wave == 0) {
            from = r1, to = a.rows;
            look(min(places[1], dealt - 1), 1);
        }
        __syncthreads();
        r1 = found[0];
    }
    const int32_t whole = a.wg_len > a.keep ? a.wg_len : a.keep;
    auto begin_of = [&](int64_t place, int row) -> int32_t {
        const int32_t s0 = rows.at(row), end = rows.at((int64_t)row + 1);
        if (place >= dealt) return (int32_t)dealt;
        // (pointers that are none would take it further back than there is room)
        if (end - s0 <= whole && place - s0 <= whole) return min(s0, (int32_t)place);
        return s0 < place ? (int32_t)place | kRowGoesOn : (int32_t)place;
    };
    begin = begin_of(places[0], r0), behind = begin_of(places[1], r1);
    const int32_t b0 = begin & ~kRowGoesOn, count = min((behind & ~kRowGoesOn) - b0, room);
    if (r1 - r0 >= kWalked) {
        constexpr int kAtOnce = 4;  // a thread's searches, whose loads do not wait for each other
        for (int k = threadIdx.x; k < count; k += kAtOnce * kBlock) {
            int lo[kAtOnce], hi[kAtOnce];
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) lo[u] = r0, hi[u] = r1 + 1;  // as from and to
            for (int span = r1 + 1 - r0; span > 1; span -= span / 2)
#pragma unroll
                for (int u = 0; u < kAtOnce; ++u) {
                    const int mid = lo[u] + (hi[u] - lo[u]) / 2;
                    if (rows.at(mid) <= b0 + min(k + u * kBlock, count - 1)) lo[u] = mid;
                    else hi[u] = max(mid, lo[u] + 1);
                }
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u)
                if (k + u * kBlock < count) row_of[k + u * kBlock] = lo[u];
        }
        if (count <= 0 && threadIdx.x == 0) row_of[0] = r0;  // row pointers that descend: a row of Y all the same
        __syncthreads();
        return;
    }
    while (r <= r1) {  // r1 < rows
        // rows without entries begin where another does: not marked, so one row a mark
        if (r > r0 && e > s && s > b0 && s - b0 < count) row_of[s - b0] = (int)r;
        r += kBlock;
        if (r <= r1) s = rows.at(r), e = rows.at(r + 1);
    }
    if (threadIdx.x == 0) row_of[0] = r0;
    __syncthreads();
    // thread t spreads the marks over entries t * each ...
    const int each = (count + kBlock - 1) / kBlock, k0 = threadIdx.x * each, k1 = min(k0 + each, count);
    int upto = -1;
    for (int k = k0; k < k1; ++k) upto = max(upto, row_of[k]);
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int n = __shfl_up(upto, d, kWave);
        if (lane >= d) upto = max(upto, n);
    }
    if (lane == kWave - 1) wave_max[wave] = upto;
    int before = __shfl_up(upto, 1, kWave);
    if (lane == 0) before = -1;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < kBlock / kWave; ++v)
        if (v < wave) before = max(before, wave_max[v]);
    for (int k = k0; k < k1; ++k) {
        before = max(before, row_of[k]);
        row_of[k] = before;
    }
    __syncthreads();
}

// What a workgroup's runs left of the rows that are divided among them, put together: the end of the
// kernel below for workgroup runs.  Every lane group holds the sum of the row that goes on behind its run
// (`continues`, in acc) and in `heads` the part of a row that came into its run and ended there; still
// `open`: one row covers the whole run; begin, behind: the table's entries for the first run of this workgroup
// and of the next.  The lane group a row begins in adds the parts of those behind it, in
// ascending order.  Slots of 2 * workgroups rows of a.carry hold the pieces of the rows that pass from one
// workgroup to the next: 2 * w for the row that comes into workgroup w, 2 * w + 1 for one that begins in it.
// end_row(e, which): the row of the workgroup's first entry (0) or its last (1); row_start(r): the first entry of row r.
template <typename T, int VEC, int LPR, int TILES, int MODE, int WGRUNS, typename EndRow, typename RowStart>
__device__ __forceinline__ void join_rows(const SpmmArgs<T> &a, int block, int lane, int grp, const int64_t foff[TILES],
                                          const Acc<T, VEC, TILES, MODE> &acc, bool continues, bool open, int y_row,
                                          int32_t begin, int32_t behind, int *flags, Pack<T, VEC> (*tails)[kBlock],
                                          Pack<T, VEC> (*heads)[kBlock], const EndRow &end_row, const RowStart &row_start) {
    constexpr int GPB = kBlock / LPR;
    constexpr int kContinues = 1, kWholeRun = 2;
    Pack<T, VEC> part[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int i = 0; i < VEC; ++i) part[t].v[i] = acc.total(T(0), t, i);
    const bool whole_run = continues && open;
    if (lane == 0) flags[grp] = (continues ? kContinues : 0) | (whole_run ? kWholeRun : 0);
    if (continues) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) tails[t][threadIdx.x] = part[t];
    }
    __syncthreads();
    const int64_t groups = (int64_t)a.blocks * GPB;
    if constexpr (MODE != MODE_ADD && WGRUNS != WGRUNS_ONCE) {  // rows without entries
        const int candidates = a.find_empty ? a.rows : a.n_empty_rows;
#pragma unroll 1
        for (int64_t item = (int64_t)block * GPB + grp; item < candidates; item += groups) {
            if (a.find_empty && a.rowptr[item] != a.rowptr[item + 1]) continue;
            T *y = a.Y + (int64_t)out_row(a, a.find_empty ? (int)item : a.empty_rows[item]) * a.F;
            Pack<T, VEC> zero;
#pragma unroll
            for (int i = 0; i < VEC; ++i) zero.v[i] = T(0);
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                if (foff[t] >= 0) store_pack_stream<T, VEC>(y + foff[t], zero);
        }
    }
    if (block >= a.blocks) return;  // the grid is rounded up
    auto add_to = [&](Pack<T, VEC>(&sum)[TILES], const Pack<T, VEC>(*from)[kBlock], int g) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const Pack<T, VEC> o = from[t][g * LPR + lane];
#pragma unroll
            for (int i = 0; i < VEC; ++i) sum[t].v[i] = sum[t].v[i] + o.v[i];
        }
    };
    // adds the parts of a row in the lane groups from g on; true if the row ends among them
    auto follow = [&](Pack<T, VEC>(&sum)[TILES], int g) {
#pragma unroll 1
        for (; g < GPB; ++g) {
            const bool on = (flags[g] & kWholeRun) != 0;
            add_to(sum, on ? tails : heads, g);
            if (!on) return true;
        }
        return false;
    };
    // A piece goes past this XCD's L2, element by element as relaxed atomics of the device's scope,
    // and so do the reads of the workgroup that adds the pieces up: a release fence instead would write back
    // and drop the whole L2, for every piece (the web graph's forward vertex stage took 785 us that way).
    auto store_piece = [&](int64_t slot, const Pack<T, VEC>(&sum)[TILES]) {
        T *p = a.carry + slot * a.F;
#pragma unroll
        for (int t = 0; t < TILES; ++t)
            if (foff[t] >= 0)
#pragma unroll
                for (int i = 0; i < VEC; ++i)
                    __hip_atomic_store(p + foff[t] + i, sum[t].v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto store_row = [&](int row, const Pack<T, VEC>(&sum)[TILES]) {
        T *y = a.Y + (int64_t)row * a.F;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            if (foff[t] < 0) continue;
            Pack<T, VEC> o = sum[t];
            if constexpr (MODE == MODE_ADD) {
                const Pack<T, VEC> base = load_pack<T, VEC>(y + foff[t]);
#pragma unroll
                for (int i = 0; i < VEC; ++i) o.v[i] = base.v[i] + o.v[i];
            }
            if constexpr (MODE == MODE_ROW_MASK) {
                RowMask<VEC> mask;
                mask.load(a.row_signs, a.sign_words, a.F, row, foff[t]);
                mask.template apply<T>(o, foff[t]);
            }
            store_pack<T, VEC>(y + foff[t], o);
        }
    };
    const bool comes_in = begin < 0, goes_out = behind < 0;
    if (grp == 0 && comes_in) {
        Pack<T, VEC> sum[TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const Pack<T, VEC> ended = heads[t][threadIdx.x];
#pragma unroll
            for (int i = 0; i < VEC; ++i) sum[t].v[i] = whole_run ? part[t].v[i] : ended.v[i];
        }
        if (whole_run) follow(sum, 1);
        store_piece(2 * (int64_t)block, sum);
    }
    if (continues && !whole_run) {
        if (follow(part, grp + 1)) store_row(y_row, part);
        else store_piece(2 * (int64_t)block + 1, part);
    }
    if (!comes_in && !goes_out) return;
    // Rows that this workgroup shares with others.
    __shared__ int arrived_last;
    const int first_row = end_row(begin & ~kRowGoesOn, 0), last_row = end_row((behind & ~kRowGoesOn) - 1, 1);
#pragma unroll 1
    for (int side = 0; side < 2; ++side) {
        if (side == 0 ? !comes_in : (!goes_out || (comes_in && first_row == last_row))) continue;
        const int row = side == 0 ? first_row : last_row;
        const int w0 = min(row_start(row) / a.wg_len, a.blocks - 1), w1 = (row_start(row + 1) - 1) / a.wg_len;
        // every store of the piece has reached memory before the arrival is counted
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (threadIdx.x == 0) {
            int32_t *count = a.arrivals + (int64_t)blockIdx.y * a.blocks + w0;
            const bool last = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == w1 - w0;
            if (last) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
            arrived_last = last;
        }
        __syncthreads();
        if (arrived_last) {
            // the lane groups take consecutive pieces each, and the first adds their sums up
            const int n = w1 - w0 + 1;
            const int j0 = (int)((int64_t)n * grp / GPB), j1 = (int)((int64_t)n * (grp + 1) / GPB);
            Pack<T, VEC> sum[TILES];
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int i = 0; i < VEC; ++i) sum[t].v[i] = T(0);
            constexpr int kBatch = 4;
#pragma unroll 1
            for (int j = j0; j < j1; j += kBatch) {
                Pack<T, VEC> piece[kBatch][TILES];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    const int64_t slot = j + u == 0 ? 2 * (int64_t)w0 + 1 : 2 * (int64_t)(w0 + j + u);
#pragma unroll
                    for (int t = 0; t < TILES; ++t)
                        if (j + u < j1 && foff[t] >= 0)
#pragma unroll
                            for (int i = 0; i < VEC; ++i)
                                piece[u][t].v[i] = __hip_atomic_load(a.carry + slot * a.F + foff[t] + i, __ATOMIC_RELAXED,
                                                                     __HIP_MEMORY_SCOPE_AGENT);
                }
#pragma unroll
                for (int u = 0; u < kBatch; ++u)
                    if (j + u < j1)
#pragma unroll
                        for (int t = 0; t < TILES; ++t)
                            if (foff[t] >= 0)
#pragma unroll
                                for (int i = 0; i < VEC; ++i) sum[t].v[i] = sum[t].v[i] + piece[u][t].v[i];
            }
#pragma unroll
            for (int t = 0; t < TILES; ++t) tails[t][threadIdx.x] = sum[t];
            __syncthreads();
            if (grp == 0) {
#pragma unroll 1
                for (int g = 1; g < GPB; ++g) add_to(sum, tails, g);
                store_row(out_row(a, row), sum);
            }
        }
        __syncthreads();
    }
}

template <typename T, int VEC, int LPR, int TILES, int MODE, int WGRUNS, int ROUND>
__global__ __launch_bounds__(kBlock, ROUND == kDeepRound ? 2 : ROUND == kMidRound ? 5 : (TILES == 1 && LPR >= 16) ? 7 : 1) void spmm_nnz_kernel(SpmmArgs<T> a) {
    constexpr int GPB = kBlock / LPR;
    static_assert(LPR % ROUND == 0, "a round's entries come from one batch");
    // What a lane group waits for between two batches of entries.  The entries of the next batch are asked for before the
    // gathers of this one, and the rows of Y they go to (rowmap, a look-up that needs the entry) are waited for behind the
    // gathers, which do not need them: a chain of entries -> gathers a batch, where it was entries -> rows -> gathers, one batch
    // behind the other.  A launch that fits the card at once is little but that chain (web graphs, forward, us, before / so:
    // 50,001 vertices of 47 features 23.5 / 22.2, 100,003 of 32 31.1 / 29.0, 200,003 of 16 45.7 / 42.7).  The two-source product
    // of large graphs is bound by its traffic and sits at its register limit: neither.  Sums of members masked one by one: neither, they
    // spilled two to four registers with the rows behind the gathers (1,000,003 rows of 100 features, 2,000 sums, by the rows'
    // signs 242 us, 222 without, by bits 165 and 157; 100,003 of 64 into 1,562 22.5 and 18).  Member lists have no rowmap to wait for, and
    // rows that end after a few entries were held up (300,007 rows of 32 features into half as many sums 20.5 us, 16.6 without; of
    // 64 29.0 and 26.5; a thirtieth as many 15.9 and 16.0): behind the gathers only up to 64 bytes a gather (2,449,029 rows of 16
    // features 121.4 us, 124.5 without), ahead but for rows of a whole wave (200,003 rows of 256 into a quarter 54.3 us, 49.3 without).
    constexpr bool kAhead = ROUND == kDeepRound || has_values(MODE) || MODE == MODE_ROW_MASK || (MODE == MODE_UNIT && LPR < kWave);
    constexpr bool kRowsBehindGathers =
        has_values(MODE) || MODE == MODE_ROW_MASK || (MODE == MODE_UNIT && VEC * LPR * sizeof(T) <= 64);
    __shared__ int wg_row[GPB];
    constexpr bool kOnce = WGRUNS == WGRUNS_ONCE;
    __shared__ Pack<T, VEC> wg_carry[kOnce ? 1 : TILES][kOnce ? 1 : kBlock];
    __shared__ Pack<T, VEC> wg_head[WGRUNS != WGRUNS_NONE ? TILES : 1][WGRUNS != WGRUNS_NONE ? kBlock : 1];
    const int lane = threadIdx.x % LPR, grp = threadIdx.x / LPR;
    const int block = logical_block(a);
    int seg = block * GPB + grp;
    if constexpr (LPR == kWave) seg = __builtin_amdgcn_readfirstlane(seg);
    // WGRUNS_ONCE: the rows of the workgroup's entries, and when all runs are done what wg_carry holds otherwise
    extern __shared__ __attribute__((aligned(16))) int row_of[];
    WideRows wide{};
    unsigned long long empties = 0;  // WGRUNS_ONCE: rows without entries, one a lane
    int e0 = 0, e1 = 0;
    bool continues = false;    // the last row of the run goes on in the next one
    bool open = false;         // WGRUNS: the row at hand began before the run
    int32_t wg_begin = 0, wg_behind = 0;
    // WGRUNS_ONCE: every wave, those without entries of their own among them (kZeroWorkgroups), looks at an equal share of the rows
    // for those without entries, which are neighbours (the youngest vertices of a graph's in-lists): zero_rows consecutive ones
    // at a time (64 a wave, so that some have many and most none: in-lists of 325,557 vertices 282 us at 128 features, 253 so).
    const int64_t waves = (int64_t)gridDim.x * (kBlock / kWave);
    const int zero_rows = (int)min((int64_t)kWave, (a.rows + waves - 1) / waves);
    const int64_t zero_row0 = ((int64_t)block * (kBlock / kWave) + threadIdx.x / kWave) * zero_rows;
    if constexpr (WGRUNS == WGRUNS_ONCE) {
        const int64_t held = a.nnz, looked_at = zero_row0 + threadIdx.x % kWave;
        wide.rowptr = a.rowptr64;
        const int64_t p = a.rowptr64[min((int64_t)a.rows, looked_at)], q = a.rowptr64[min((int64_t)a.rows, looked_at + 1)];
        const int64_t pivot = a.rowptr64[min((int64_t)a.rows, (int64_t)search_step(a.rows) * (threadIdx.x % kWave))];
        wide.first = max((int64_t)0, min(held, a.rowptr64[0]));
        wide.last = max(wide.first, min(held, a.rowptr64[a.rows]));
        if constexpr (MODE != MODE_ADD)
            empties = __ballot((int)(threadIdx.x % kWave) < zero_rows && looked_at < a.rows && min(p, wide.last) >= max(q, wide.first));
        if (a.val != nullptr) a.val += wide.first;
        a.col64 += wide.first;
        if (block < a.blocks) once_stretch(a, wide, block, pivot, row_of, wg_begin, wg_behind);
        wg_begin = __builtin_amdgcn_readfirstlane(wg_begin), wg_behind = __builtin_amdgcn_readfirstlane(wg_behind);  // no vector registers
        const int32_t first = wg_begin & ~kRowGoesOn, end = wg_behind & ~kRowGoesOn;
        const int run_len = a.wg_len / GPB, whole = run_len > a.keep ? run_len : a.keep;
        auto begin_of = [&](int g) -> int32_t {
            const int32_t e = first + g * ((end - first + GPB - 1) / GPB);
            if (g == 0) return wg_begin;
            if (e >= end) return wg_behind;
            const int row = row_of[e - first];
            const int32_t s0 = wide.at(row), behind = wide.at((int64_t)row + 1);
            return behind - s0 <= whole ? max(first, min(e, s0)) : (s0 < e ? e | kRowGoesOn : e);
        };
        const int32_t r0 = begin_of(grp), r1 = begin_of(grp + 1);
        e0 = r0 & ~kRowGoesOn, e1 = r1 & ~kRowGoesOn;
        open = r0 < 0, continues = r1 < 0;
    } else if (seg < a.nseg) {
        if constexpr (WGRUNS != WGRUNS_NONE) {
            int32_t r0, r1;
            if constexpr (WGRUNS == WGRUNS_TABLE) {
                r0 = a.run_start[seg], r1 = a.run_start[seg + 1];
            } else {
                auto begin_of = [&](int w, int g) { return wg_run_begin(a.rowptr, a.rowidx, a.nnz, a.wg_len, GPB, a.keep, w, g); };
                wg_begin = begin_of(block, 0), wg_behind = begin_of(block + 1, 0);
                r0 = begin_of(block, grp), r1 = grp + 1 < GPB ? begin_of(block, grp + 1) : wg_behind;
            }
            e0 = r0 & ~kRowGoesOn, e1 = r1 & ~kRowGoesOn;
            open = r0 < 0, continues = r1 < 0;
        } else if (a.run_start != nullptr) {  // one load instead of two dependent ones
            e0 = a.run_start[seg];
            e1 = a.run_start[seg + 1];
        } else {
            e0 = run_boundary(a, seg * a.seg_nnz);
            e1 = run_boundary(a, (seg + 1) * a.seg_nnz);
        }
    }
    auto row_at = [&](int e) -> int { return WGRUNS == WGRUNS_ONCE ? row_of[e - (wg_begin & ~kRowGoesOn)] : a.rowidx[e]; };
    auto col_at = [&](int e) -> int { return WGRUNS == WGRUNS_ONCE ? (int)a.col64[e] : a.colidx[e]; };
    // e0 >= e1 inside the list cannot happen for a well-formed CSR
    const bool active = e0 < e1;
    // means: a row that began before the run is divided by the pass that adds its carries up
    const bool began_before = WGRUNS == WGRUNS_NONE && MODE == MODE_UNIT && a.mean && active && e0 > 0 && a.rowidx[e0 - 1] == a.rowidx[e0];
    int64_t foff[TILES];
    feature_offsets<VEC, LPR, TILES>(a.F, lane, foff);
    Acc<T, VEC, TILES, MODE> acc;
    acc.clear();
    int cur = -1;
    int cur_out = -1;
    RowMask<VEC> mask[TILES];
    // A row ends inside the run: it is written, or (the part of it that lies in this run) put aside
    // for the lane group where the row began.
    int row_e0 = e0;  // where the row at hand begins in the run
    auto finish_row = [&](int y_row, int end) {
        if constexpr (WGRUNS != WGRUNS_NONE) {
            if (open) {
                open = false;
#pragma unroll
                for (int t = 0; t < TILES; ++t)
#pragma unroll
                    for (int i = 0; i < VEC; ++i) wg_head[t][threadIdx.x].v[i] = acc.total(T(0), t, i);
                return;
            }
        }
        write_row<T, VEC, TILES, MODE>(a.Y, a.F, y_row, foff, acc,
                                       MODE == MODE_UNIT && a.mean && !(began_before && row_e0 == e0) ? (T)(end - row_e0) : T(1), mask);
    };
    // A row's mask is asked for where the row begins and used where it ends, behind the gathers in between.
    auto begin_row = [&](int y_row) {
        if constexpr (MODE == MODE_ROW_MASK)
#pragma unroll
            for (int t = 0; t < TILES; ++t) mask[t].load(a.row_signs, a.sign_words, a.F, y_row, foff[t] < 0 ? 0 : foff[t]);
    };
    // the names of rows: see below
    constexpr bool kNamesRowsOfY = !(MODE == MODE_DUAL && VEC * LPR * sizeof(T) >= 512);
    auto named = [&](int stored_row) { return kNamesRowsOfY ? out_row(a, stored_row) : stored_row; };
    auto row_of_y = [&](int name) { return kNamesRowsOfY ? name : out_row(a, name); };
    if (active) {
        // A run names its rows by the row of Y they are written to (rowmap[stored row], which the
        // lanes look up beside their entries), so that closing a row inside the run needs no load
        // of its own: a load there, and the wait for it, would stand between the gathers of the run.
        // The two-source product over rows of 512 bytes and more keeps the other form -- the run names
        // its rows by their stored number and looks the row of Y up where a row ends.  The look-up
        // beside the entries puts one more load between a run's entries and its first gathers and
        // holds two more values per lane in a kernel that sits at its register limit (72 for seven
        // waves per SIMD): the F = 128 kernel, bound by its traffic either way, took 221 us with it
        // and takes 213 us without (F = 16: 76 -> 62 us with it; the 18.5 M-vertex graph at F = 64:
        // 13.6 -> 13.4 ms; the mask modes, which have no rowmap, lose the wait and nothing else).
        // looked at when the run is done: the stored row of the last entry (the row a carry belongs
        // to) and the row of the entry behind the run; asked for beside the entries
        int last_row, row_behind;
        if constexpr (!kNamesRowsOfY) {  // the names are the stored rows: the first is read here, the last is at hand at the end
            cur_out = a.rowidx[e0];
            if constexpr (WGRUNS == WGRUNS_NONE) row_behind = e1 < a.nnz ? a.rowidx[e1] : -1;
        }
        // As in the row schedule: the lanes of the group load one entry each, and the
        // entries reach all lanes through the LDS crossbar.
        const int group_lane0 = 4 * ((threadIdx.x % kWave) - lane);
        int64_t fld[TILES];  // lanes beyond the width gather feature 0 again (never stored)
#pragma unroll
        for (int t = 0; t < TILES; ++t) fld[t] = foff[t] < 0 ? 0 : foff[t];
        int my_row = 0, my_c = 0;
        T my_w = T(1);
        auto load_entry = [&](int e) {  // this lane's of the batch from e on
            my_row = 0, my_c = 0, my_w = T(1);
            if (e + lane >= e1) return;
            my_row = row_at(e + lane);
            my_c = col_at(e + lane);
            if constexpr (MODE == MODE_DUAL) my_w = a.val[e + lane];
            if constexpr (has_values(MODE)) my_w = a.val != nullptr ? a.val[e + lane] : T(1);
        };
        if constexpr (kAhead) load_entry(e0);
        for (int e = e0; e < e1; e += LPR) {
            if constexpr (!kAhead) load_entry(e);
            if constexpr (MODE != MODE_DUAL) arrive(my_c), arrive(my_row);
            if constexpr (has_values(MODE)) arrive(my_w);
            int my_o = e + lane < e1 ? named(my_row) : 0;
            if constexpr (kNamesRowsOfY) {
                // with every batch of entries, so that no load of the run waits for another but
                // the row numbers for their rows (the same two words each time)
                if constexpr (WGRUNS == WGRUNS_NONE) {
                    last_row = a.rowidx[e1 - 1];
                    row_behind = e1 < a.nnz ? a.rowidx[e1] : -1;
                }
                // the run begins with the row of its first entry
                if constexpr (!kRowsBehindGathers) {
                    const int batch_first = __builtin_amdgcn_ds_bpermute(group_lane0, my_o);
                    if (e == e0) cur_out = batch_first;
                }
            }
            const int cnt = min(e1 - e, LPR);
            const int this_c = my_c;
            const T this_w = my_w;
            if constexpr (kAhead) load_entry(e + LPR);
            for (int u0 = 0; u0 < cnt; u0 += ROUND) {
                int o[ROUND], c[ROUND];
                T w[ROUND];
#pragma unroll
                for (int u = 0; u < ROUND; ++u) {
                    const int from = group_lane0 + 4 * (u0 + u);
                    if constexpr (!kRowsBehindGathers) o[u] = __builtin_amdgcn_ds_bpermute(from, my_o);
                    c[u] = __builtin_amdgcn_ds_bpermute(from, this_c);
                    if constexpr (has_values(MODE) || MODE == MODE_DUAL)
                        w[u] = from_lane(from, this_w);
                    else
                        w[u] = T(1);
                }
                // Lanes without an entry hold column 0 (a row of X like any other) and value 1, and
                // positions behind the last entry of a batch read those: a round may gather for them,
                // nothing is added for them.  Only a block without first-source columns sees such a
                // position as one of the second source, and takes the slower path for that round.
                bool second = false;
                if constexpr (MODE == MODE_DUAL) {
#pragma unroll
                    for (int u = 0; u < ROUND; ++u) second = second | (c[u] >= a.split);
                }
                auto gather_and_add = [&](auto plain) {
                    constexpr bool kPlain = decltype(plain)::value;  // every entry from the first source
                    Gathered<T, VEC, MODE> x[ROUND][TILES];
                    // Up to 64 bytes per lane group and gather, a position behind the last entry gathers
                    // like the others (column 0, see above): the branches around four small loads cost
                    // more than the loads.  Wider rows skip it: there the extra row is what costs.
                    constexpr bool kGatherAll = VEC * LPR * sizeof(T) <= 64;
#pragma unroll
                    for (int u = 0; u < ROUND; ++u)
                        if (kGatherAll || u0 + u < cnt) {
#pragma unroll
                            for (int t = 0; t < TILES; ++t)
                                x[u][t] = gather<T, VEC, MODE, (int)(VEC * LPR * sizeof(T))>(a, c[u], kPlain ? 0 : c[u] >= a.split, fld[t]);
                        }
                    if constexpr (kRowsBehindGathers) {
                        // the names of the rows are waited for behind the gathers, which do not need them
                        if (u0 == 0) arrive(my_o);
#pragma unroll
                        for (int u = 0; u < ROUND; ++u) o[u] = __builtin_amdgcn_ds_bpermute(group_lane0 + 4 * (u0 + u), my_o);
                        if (u0 == 0 && e == e0) {  // the run begins with the row of its first entry
                            cur_out = o[0];
                            begin_row(cur_out);
                        }
                    }
                    if constexpr (MODE != MODE_DUAL && !(kGatherAll && !has_values(MODE)))
#pragma unroll
                        for (int u = 0; u < ROUND; ++u)
#pragma unroll
                            for (int t = 0; t < TILES; ++t) arrive(x[u][t]);
#pragma unroll
                    for (int u = 0; u < ROUND; ++u) {
                        if (u0 + u < cnt) {
                            if (o[u] != cur_out) {
                                // the row ends inside this run: finish it here
                                finish_row(row_of_y(cur_out), e + u0 + u);
                                row_e0 = e + u0 + u;
                                acc.clear();
                                cur_out = o[u];
                                begin_row(cur_out);
                            }
                            acc.add(x[u], fld, w[u], kPlain ? 0 : c[u] >= a.split);
                        }
                    }
                };
                if (MODE != MODE_DUAL || __ballot(second) == 0) gather_and_add(std::true_type{});
                else gather_and_add(std::false_type{});
            }
        }
        if constexpr (WGRUNS == WGRUNS_NONE) {
            cur = kNamesRowsOfY ? last_row : cur_out;
            continues = row_behind == cur;
        }
        if (!continues) finish_row(row_of_y(cur_out), e1);
    }
    if constexpr (WGRUNS != WGRUNS_NONE) {
        if constexpr (WGRUNS == WGRUNS_TABLE)
            if (seg < a.nseg) wg_begin = a.run_start[block * GPB], wg_behind = a.run_start[(block + 1) * GPB];
        if constexpr (WGRUNS == WGRUNS_ONCE && MODE != MODE_ADD) {  // rows without entries, a wave per stretch of neighbours
            Pack<T, VEC> zero;
#pragma unroll
            for (int i = 0; i < VEC; ++i) zero.v[i] = T(0);
            for (int64_t row0 = zero_row0;;) {
                while (empties != 0 && blockIdx.y == 0) {
                    const int at = __ffsll(empties) - 1, behind = __ffsll(~(empties >> at)) - 1, n = behind < 0 ? kWave : behind;
                    T *y = a.Y + (row0 + at) * a.F;
                    for (int64_t i = (int64_t)VEC * (threadIdx.x % kWave), all = n * a.F; i < all; i += VEC * kWave)
                        store_pack<T, VEC>(y + min(i, all - VEC), zero);
                    empties = n == kWave ? 0 : empties & ~(((1ull << n) - 1) << at);
                }
                row0 += waves * zero_rows;
                if (row0 >= a.rows) break;
                const int64_t r = row0 + threadIdx.x % kWave;
                empties = __ballot((int)(threadIdx.x % kWave) < zero_rows && r < a.rows && wide.at(min((int64_t)a.rows - 1, r)) >= wide.at(min((int64_t)a.rows, r + 1)));
            }
        }
        Pack<T, VEC>(*tails)[kBlock];
        int ends[2] = {0, 0};  // the rows of the workgroup's first entry and of its last
        if constexpr (kOnce) {
            const int32_t first = wg_begin & ~kRowGoesOn, end = wg_behind & ~kRowGoesOn;
            ends[0] = row_of[0], ends[1] = row_of[max(0, end - first - 1)];
            __syncthreads();
            tails = reinterpret_cast<Pack<T, VEC>(*)[kBlock]>(row_of);
        } else {
            tails = wg_carry;
        }
        auto end_row = [&](int32_t e, int which) -> int { return kOnce ? ends[which] : a.rowidx[e]; };
        auto row_start = [&](int64_t r) -> int32_t { return WGRUNS == WGRUNS_ONCE ? wide.at(r) : a.rowptr[r]; };
        join_rows<T, VEC, LPR, TILES, MODE, WGRUNS>(a, block, lane, grp, foff, acc, continues, open,
                                                    continues && active ? row_of_y(cur_out) : -1, wg_begin, wg_behind, wg_row,
                                                    tails, wg_head, end_row, row_start);
        return;
    }
    // The carries of one row are added per workgroup (or per merge_stride lane groups of it): the first lane
    // group that carries the row takes those of the groups behind it, in ascending order.
    Pack<T, VEC> part[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int i = 0; i < VEC; ++i) part[t].v[i] = acc.total(T(0), t, i);
    if (lane == 0) wg_row[grp] = continues ? cur : kNoCarry;
    if (continues) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) wg_carry[t][threadIdx.x] = part[t];
    }
    __syncthreads();
    if (seg >= a.nseg) return;
    int mark = kNoCarry;
    if (continues) {
        const int merged = a.merge_stride;  // at most GPB, a power of two
        const bool first = (grp & (merged - 1)) == 0 || wg_row[grp - 1] != cur;
        mark = first ? cur : kMerged;
        if (first) {
            for (int g = grp + 1; (g & (merged - 1)) != 0 && wg_row[g] == cur; ++g)
#pragma unroll
                for (int t = 0; t < TILES; ++t) {
                    const Pack<T, VEC> o = wg_carry[t][g * LPR + lane];
#pragma unroll
                    for (int i = 0; i < VEC; ++i) part[t].v[i] = part[t].v[i] + o.v[i];
                }
            T *crow = a.carry + (int64_t)seg * a.F;
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                if (foff[t] >= 0) store_pack<T, VEC>(crow + foff[t], part[t]);
        }
    }
    if (lane == 0 && blockIdx.y == 0) a.carry_row[seg] = mark;
}

// One level of the carry reduction.  Carries (row, vector) with equal rows are adjacent
// (in the list the nnz kernel writes, kMerged entries may lie between them: they are
// skipped); kNoCarry marks a run that carries nothing.  A lane group takes kCarryFan
// consecutive carries:
// a row whose carries all lie inside the chunk is finished here (Y += their sum, nobody
// else touches that row); the part of a row that reaches the chunk from before goes to
// slot 2*chunk of the next level, the part of a row that goes on behind the chunk to slot
// 2*chunk+1 (a row that covers the whole chunk fills slot 2*chunk and puts zeros in the
// other), so that equal rows are adjacent again on the next level.
constexpr int kCarryFan = 64;
constexpr int kReduceBatch = 16;  // carry rows in flight per lane group
constexpr int kFixBatch = 8;

template <typename T, int VEC, int LPR>
__global__ __launch_bounds__(kBlock) void spmm_carry_reduce_kernel(SpmmArgs<T> a) {
    constexpr int GPB = kBlock / LPR;
    const int sub = threadIdx.x % LPR;
    const int chunk = blockIdx.x * GPB + threadIdx.x / LPR;
    const int s0 = chunk * kCarryFan;
    if (s0 >= a.nseg) return;
    const int s1 = min(s0 + kCarryFan, a.nseg);
    const bool merged = a.merge_stride > 1;  // the list of the nnz kernel: s0 starts a workgroup
    const int before = (s0 > 0 && !merged) ? a.carry_row[s0 - 1] : -1;
    const int after = s1 < a.nseg ? a.carry_row[s1] : -1;
    // the rows of the chunk: every lane of the group reads all of them (same addresses,
    // one round trip), so no lane has to wait for another
    int rr[kCarryFan];
    if (s1 - s0 == kCarryFan) {
        const int4 *p = reinterpret_cast<const int4 *>(a.carry_row + s0);  // s0 is a multiple of 64
#pragma unroll
        for (int q = 0; q < kCarryFan / 4; ++q) {
            const int4 v = p[q];
            rr[4 * q] = v.x, rr[4 * q + 1] = v.y, rr[4 * q + 2] = v.z, rr[4 * q + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int u = 0; u < kCarryFan; ++u) rr[u] = s0 + u < s1 ? a.carry_row[s0 + u] : -1;
    }
    int any = -1;
#pragma unroll
    for (int u = 0; u < kCarryFan; ++u) any = max(any, rr[u]);
    if (any < 0) {  // nothing is carried through this chunk
        if (sub == 0) a.carry_row_out[2 * chunk] = a.carry_row_out[2 * chunk + 1] = -1;
        return;
    }
    int head_row = -1, tail_row = -1;
    T *slot0 = a.carry_out + (int64_t)(2 * chunk) * a.F;
    T *slot1 = slot0 + a.F;
    for (int64_t nominal = (int64_t)sub * VEC; nominal < a.F; nominal += (int64_t)LPR * VEC) {
        const int64_t f = pack_start<VEC>(a.F, nominal);
        Pack<T, VEC> acc, zero;
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc.v[i] = zero.v[i] = T(0);
        int cur = -1;
        bool from_before = false;
        auto close = [&](bool ends_here) {
            if (cur < 0) return;
            if (!from_before && ends_here) {
                // The one addition to these elements in this launch sequence (the row's
                // last run has stored its part already), so its result does not depend on
                // timing; sent as an atomic only so that the lane need not wait for Y.
                T *y = a.Y + (int64_t)out_row(a, cur) * a.F + f;
                if (a.row_signs != nullptr) {  // the row's last run has masked its part
                    RowMask<VEC> mask;
                    mask.load(a.row_signs, a.sign_words, a.F, cur, f);
                    mask.template apply<T>(acc, f);
                }
#pragma unroll
                for (int i = 0; i < VEC; ++i)
                    if (f + i >= nominal) unsafeAtomicAdd(y + i, acc.v[i]);  // the elements before are the lane's before
                return;
            }
            if (from_before) {
                head_row = cur;
                store_pack<T, VEC>(slot0 + f, acc);
                if (!ends_here) {
                    tail_row = cur;
                    store_pack<T, VEC>(slot1 + f, zero);
                }
            } else {
                tail_row = cur;
                store_pack<T, VEC>(slot1 + f, acc);
            }
        };
#pragma unroll
        for (int b = 0; b < kCarryFan; b += kReduceBatch) {
            Pack<T, VEC> c[kReduceBatch];
#pragma unroll
            for (int u = 0; u < kReduceBatch; ++u)
                c[u] = rr[b + u] >= 0 ? load_pack<T, VEC>(a.carry + (int64_t)(s0 + b + u) * a.F + f) : zero;
#pragma unroll
            for (int u = 0; u < kReduceBatch; ++u) {
                if (rr[b + u] != cur && rr[b + u] != kMerged) {  // entries behind the end of the last chunk are -1
                    close(true);
                    cur = rr[b + u];
                    acc = zero;
                    // is the row carried into the chunk?  In the list of the nnz kernel the
                    // run before s0 may be a merged one, so ask where the row starts.
                    from_before = (b + u == 0) && cur >= 0 &&
                                  (merged ? (int64_t)a.rowptr[cur] < (int64_t)s0 * a.seg_nnz : cur == before);
                }
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc.v[i] = acc.v[i] + c[u].v[i];
            }
        }
        close(!(cur >= 0 && cur == after));
    }
    if (sub == 0) {
        a.carry_row_out[2 * chunk] = head_row;
        a.carry_row_out[2 * chunk + 1] = tail_row;
    }
}

// Adds the carries of every row that straddles runs, in ascending run order, and
// (when not accumulating) clears the rows that have no entries (the two sets of rows are
// disjoint).  Carries: one lane group (LPR lanes across the features) per run; the group
// whose run holds the first carry of a row walks the row's carries, kFixBatch in flight,
// and adds their sum to the row.  Empty rows: one thread looks at one row, and the empty
// rows of a wave are then dealt out to its lane groups.

// Lane (within the wave) of the flagged item this lane's group should handle in the
// round that starts at rank `base`, or -1.  Uniform control flow: every lane calls it.
template <int LPR>
__device__ __forceinline__ int deal_item(bool flag, int my_rank, int base, int grp) {
    constexpr int G = kWave / LPR;
    int src = -1;
#pragma unroll
    for (int gi = 0; gi < G; ++gi) {
        const unsigned long long m = __ballot(flag && my_rank == base + gi);
        if (gi == grp && m) src = __ffsll(m) - 1;
    }
    return src;
}

template <typename T, int VEC, int LPR, bool MERGED>
__global__ __launch_bounds__(kBlock) void spmm_fixup_kernel(SpmmArgs<T> a) {
    constexpr int GPB = kBlock / LPR;
    // carry rows in flight per lane group; few, so that the many groups that find nothing
    // to do are all resident at once
    constexpr int BATCH = MERGED ? 4 : kFixBatch;
    const int lane = threadIdx.x % kWave;
    const int sub = lane % LPR, grp = lane / LPR;

    int s0 = blockIdx.x * GPB + threadIdx.x / LPR;
    if constexpr (LPR == kWave) s0 = __builtin_amdgcn_readfirstlane(s0);
    const int stride = MERGED ? a.merge_stride : 1;  // MERGED: the list of the nnz kernel
    // First carry of its row?  The list of the nnz kernel holds one carry per row and
    // workgroup: a row has an earlier carry exactly when it starts before this run, and
    // its later carries belong to the first run of every following workgroup whose end
    // still lies inside the row.  In a plain list the carries of a row are adjacent.
    int row = -1, row_end = 0;
    if (s0 < a.nseg) {
        const int r = a.carry_row[s0];
        if (r >= 0) {
            bool head;
            if constexpr (MERGED) {
                head = (int64_t)a.rowptr[r] >= (int64_t)s0 * a.seg_nnz;
                row_end = a.rowptr[r + 1];
            } else {
                head = s0 == 0 || a.carry_row[s0 - 1] != r;
            }
            if (head) row = r;
        }
    }
    if (row >= 0) {
        const int64_t group0 = (int64_t)(s0 / stride) * stride;
#pragma unroll 1
        for (int64_t nominal = (int64_t)sub * VEC; nominal < a.F; nominal += (int64_t)LPR * VEC) {
            const int64_t f = pack_start<VEC>(a.F, nominal);
            Pack<T, VEC> acc, zero;
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc.v[i] = zero.v[i] = T(0);
            bool more = true;
#pragma unroll 1
            for (int k = 0; more; k += BATCH) {
                bool take[BATCH];
                Pack<T, VEC> c[BATCH];
                if constexpr (MERGED) {
#pragma unroll
                    for (int u = 0; u < BATCH; ++u) {
                        const int64_t p = (k + u == 0) ? (int64_t)s0 : group0 + (int64_t)(k + u) * stride;
                        take[u] = (k + u == 0) || (p + 1) * a.seg_nnz < (int64_t)row_end;
                        c[u] = take[u] ? load_pack<T, VEC>(a.carry + p * a.F + f) : zero;
                    }
                } else {
                    int rr[BATCH];
#pragma unroll
                    for (int u = 0; u < BATCH; ++u) {
                        const int64_t p = (int64_t)s0 + k + u;
                        take[u] = p < a.nseg;
                        const int64_t idx = take[u] ? p : (int64_t)a.nseg - 1;
                        rr[u] = a.carry_row[idx];
                        c[u] = load_pack<T, VEC>(a.carry + idx * a.F + f);
                    }
#pragma unroll
                    for (int u = 0; u < BATCH; ++u) take[u] = take[u] && rr[u] == row;
                }
#pragma unroll
                for (int u = 0; u < BATCH; ++u) {
                    more = more && take[u];
                    if (more)
#pragma unroll
                        for (int i = 0; i < VEC; ++i) acc.v[i] = acc.v[i] + c[u].v[i];
                }
            }
            T *y = a.Y + (int64_t)out_row(a, row) * a.F + f;
            Pack<T, VEC> o = load_pack<T, VEC>(y);
            if (a.row_signs != nullptr) {  // the row's last run has masked its part
                RowMask<VEC> mask;
                mask.load(a.row_signs, a.sign_words, a.F, row, f);
                mask.template apply<T>(acc, f);
            }
#pragma unroll
            for (int i = 0; i < VEC; ++i) o.v[i] = o.v[i] + acc.v[i];
            if (MERGED && a.mean) {
                const T n = (T)(row_end - a.rowptr[row]);
#pragma unroll
                for (int i = 0; i < VEC; ++i) o.v[i] = o.v[i] / n;
            }
            store_pack<T, VEC>(y, o);
        }
    }

    if (a.accumulate) return;
    const int item = blockIdx.x * kBlock + threadIdx.x;
    const int wave_item0 = item - lane;
    if (wave_item0 >= a.rows) return;
    const bool empty = item < a.rows && a.rowptr[item] == a.rowptr[item + 1];
    const unsigned long long below = (1ull << lane) - 1ull;
    const unsigned long long empties = __ballot(empty);
    const int n_empty = __popcll(empties), empty_rank = __popcll(empties & below);
    constexpr int G = kWave / LPR;
    for (int base = 0; base < n_empty; base += G) {
        const int src = deal_item<LPR>(empty, empty_rank, base, grp);
        if (src < 0) continue;
        const int erow = out_row(a, wave_item0 + src);
        Pack<T, VEC> zero;
#pragma unroll
        for (int i = 0; i < VEC; ++i) zero.v[i] = T(0);
        for (int64_t f = (int64_t)sub * VEC; f < a.F; f += (int64_t)LPR * VEC)
            store_pack_stream<T, VEC>(a.Y + (int64_t)erow * a.F + pack_start<VEC>(a.F, f), zero);
    }
}

// The same pass for a block that comes with the lists of its cut rows and its empty rows
// (both follow from rowptr and the run length alone, so they are made once per block): a lane
// group per cut row, and nothing for the many runs that carry nothing.  The carries of a row
// sit where the nnz kernel's workgroups left them: at the run the row starts in, and at the first
// run of every following workgroup whose end still lies inside the row; they are added in that
// (ascending) order, the same as in spmm_fixup_kernel, so the result is the same bit for bit.
template <typename T, int VEC, int LPR>
__global__ __launch_bounds__(kBlock) void spmm_fixup_rows_kernel(SpmmArgs<T> a) {
    constexpr int GPB = kBlock / LPR;
    constexpr int BATCH = 8;
    const int sub = threadIdx.x % LPR;
    int item = blockIdx.x * GPB + threadIdx.x / LPR;
    if constexpr (LPR == kWave) item = __builtin_amdgcn_readfirstlane(item);
    if (item < a.n_cut_rows) {
        const int row = a.cut_rows[item];
        const int64_t row_end = a.rowptr[row + 1];
        const int64_t s0 = a.rowptr[row] / a.seg_nnz;           // the run the row starts in
        const int64_t group0 = s0 / a.merge_stride * a.merge_stride;  // first run of that run's workgroup
#pragma unroll 1
        for (int64_t nominal = (int64_t)sub * VEC; nominal < a.F; nominal += (int64_t)LPR * VEC) {
            const int64_t f = pack_start<VEC>(a.F, nominal);
            Pack<T, VEC> acc, zero;
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc.v[i] = zero.v[i] = T(0);
            bool more = true;
#pragma unroll 1
            for (int k = 0; more; k += BATCH) {
                bool take[BATCH];
                Pack<T, VEC> c[BATCH];
#pragma unroll
                for (int u = 0; u < BATCH; ++u) {
                    const int64_t p = (k + u == 0) ? s0 : group0 + (int64_t)(k + u) * a.merge_stride;
                    take[u] = (k + u == 0) || (p + 1) * a.seg_nnz < row_end;
                    c[u] = take[u] ? load_pack<T, VEC>(a.carry + p * a.F + f) : zero;
                }
#pragma unroll
                for (int u = 0; u < BATCH; ++u) {
                    more = more && take[u];
                    if (more)
#pragma unroll
                        for (int i = 0; i < VEC; ++i) acc.v[i] = acc.v[i] + c[u].v[i];
                }
            }
            T *y = a.Y + (int64_t)out_row(a, row) * a.F + f;
            Pack<T, VEC> o = load_pack<T, VEC>(y);
#pragma unroll
            for (int i = 0; i < VEC; ++i) o.v[i] = o.v[i] + acc.v[i];
            store_pack<T, VEC>(y, o);
        }
    }
    if (a.accumulate || item >= a.n_empty_rows) return;
    const int erow = out_row(a, a.empty_rows[item]);
    Pack<T, VEC> zero;
#pragma unroll
    for (int i = 0; i < VEC; ++i) zero.v[i] = T(0);
    for (int64_t f = (int64_t)sub * VEC; f < a.F; f += (int64_t)LPR * VEC)
        store_pack_stream<T, VEC>(a.Y + (int64_t)erow * a.F + pack_start<VEC>(a.F, f), zero);
}

// ------------------------------------------------------------------- dispatch --
struct Shape {
    int vec, lpr, tiles, grid_y;
};

// Lane layout for a feature width.  Packs need no alignment and the last one of a row may overlap the
// one before it (pack_start), so rows of up to 64 packs of four take packs whatever their
// width: 47 features are 12 lanes of four (the nnz kernel of a 50,001-vertex graph took 27.8 us
// with one feature a lane, 22.8 us so).  Longer rows are walked in several tiles, where an overlap
// would add a carry twice, and take the widest packs that divide the width.
// runs: the layout of the nnz schedule, which wants 16 lanes or more per run -- with 4 lanes a
// wave walks 16 runs at once, each with its own row changes (F = 16: 0.106 -> 0.089 ms for the forward
// vertex stage of the web graph) -- and so takes the narrowest packs that 16 lanes hold.
// The row schedule is faster with the widest packs (0.036 against 0.053 ms).
// two_tiles: rows beyond 64 packs as two tiles of one launch's lanes, which read every entry once for both; otherwise a part of
// the launch per 64 packs, with fewer registers, more waves and half as wide a working set in the L2s.  That is taken by
// default where it leaves no lane idle (forward, 512 features, two tiles / so: web graphs of 6,000 vertices 25.5 / 22.6 us, 100,003
// 301 / 292, 325,557 926 / 914; 1,024 features over 20,000 125 / 119); where lanes idle two tiles stay (264 features over 325,557
// vertices, forward + gradient 940 / 1,168, 400 1,198 / 1,310).  Rows of few entries cost more than they save in parts
// (row_shape), and so does the search of a small product of int64 arrays (once_layout).
template <typename T>
Shape pick_shape(int64_t F, bool runs, bool two_tiles = false) {
    Shape s;
    s.vec = 1;
    if (sizeof(T) == 4) {
        if (runs) s.vec = F <= 16 ? 1 : (F <= 32 ? 2 : 4);
        else s.vec = F < 2 ? 1 : (F < 4 ? 2 : 4);
        if (F > 4 * kWave) s.vec = F % 4 == 0 ? 4 : (F % 2 == 0 ? 2 : 1);
    }
    const int64_t slots = ceil_div(F, (int64_t)s.vec);
    int lpr = pow2_ceil(slots);
    if (lpr < 4) lpr = 4;
    if (lpr > 64) lpr = 64;
    if (s.vec != 4 || sizeof(T) != 4) {
        // fewer instantiations off the main path: 4, 16 or 64 lanes per row
        lpr = lpr <= 4 ? 4 : (lpr <= 16 ? 16 : 64);
    }
    s.lpr = lpr;
    s.tiles = (lpr == 64 && slots > 64 && sizeof(T) == 4 && (two_tiles || slots % 64 != 0)) ? 2 : 1;
    s.grid_y = (int)ceil_div(slots, (int64_t)s.lpr * s.tiles);
    return s;
}

// How many consecutive runs of the nnz schedule merge their carries before these reach memory: part of the
// order in which a long row is summed, and so a function of the width alone, not of the lane layout (a workgroup
// of the layout in use holds as many runs or a multiple of them).  What divides the rows of an assignment into
// clusters differently at the last bit flips ReLUs behind their means.
template <typename T>
int merged_runs(int64_t F) {
    int64_t vec = 1;
    if (sizeof(T) == 4) {
        vec = F % 4 == 0 ? 4 : (F % 2 == 0 ? 2 : 1);
        while (vec > 1 && F / vec < 16) vec /= 2;
    }
    int lpr = pow2_ceil(F / vec);
    if (vec != 4) lpr = lpr <= 4 ? 4 : (lpr <= 16 ? 16 : 64);
    return kBlock / (lpr < 4 ? 4 : (lpr > 64 ? 64 : lpr));
}

// The layout of the nnz schedule for a feature width.
Shape shape_of(int64_t F, int dtype) { return dtype == CGNN_F64 ? pick_shape<double>(F, true) : pick_shape<float>(F, true); }

enum { KIND_ROW = 0, KIND_NNZ = 1, KIND_FIXUP = 2, KIND_REDUCE = 3, KIND_FIXUP_ROWS = 4 };

// How many gathers a lane of the nnz schedule has in flight.  A row of up to kDefaultSeg entries is added by one lane group,
// and where a launch has few workgroups its time is that of the longest run: a batch of entries, then its gathers
// kUnroll at a time, each round waiting for memory.  With kDeepRound the gathers of 16 entries are one round, and the next
// batch of entries is on its way meanwhile; the registers for that leave two workgroups a compute unit.  us, with kUnroll / so:
// means of 30,011 rows of 64 columns in 7,584 groups 37.8 / 31.3, sums 16.8 / 12.9, masked sums 20.9 / 17.3; 9,000 rows of
// 100: 35.2 / 30.4, 18.3 / 14.5, 21.3 / 18.2; 2,708 of 64: 23.2 / 21.6, 11.0 / 10.1, 15.3 / 14.8.  Beyond 512 workgroups the means,
// whose runs are 64 entries long, would wait for a second round of workgroups (300,007 rows of 100 36.2, with kMidRound 34.8,
// with kUnroll 39.0); the runs of the others are as short as fills the card, and they gain up to 1,024 (sums of 100,003
// rows of 64 21.5 / 17.8, masked 25.5 / 22.0).  Unmasked sums take kMidRound where
// the card holds all workgroups at once, up to 3 * 2^18 entries (300,007 rows of 64 27.4 / 25.0, 600,000 38.5 / 36.3, means
// 40.7 / 38.5; at 1,000,003, where enough lane groups gather in any case, 49.3 / 51.0 and 49.2 / 50.2); masked ones do not gain by it
// (100,003 rows of 100 28.5 / 29.7), nor do the products of a plan with kDeepRound (5,000 rows of 64 9.4 / 10.1).  Those of a
// block that is new with the call gain where hubs make long runs (8,000 rows 19.6 / 18.7) and lose where rows are short
// (out-lists of 5,463 vertices, 208 features, the whole pass 14.3 / 16.7), which nothing tells apart before the launch.
template <int MODE>
constexpr bool kGoesDeep = MODE == MODE_UNIT || MODE == MODE_SIGN_MASK || MODE == MODE_ROW_MASK;

template <int MODE, int WGRUNS>
int round_of(int64_t workgroups, int64_t entries) {
    if (kGoesDeep<MODE> && workgroups <= (WGRUNS == WGRUNS_NONE ? 512 : 1024)) return kDeepRound;
    return (MODE == MODE_UNIT || MODE == MODE_ROW_MASK) && workgroups <= kResidentWorkgroups && entries <= 3 << 18 ? kMidRound : kUnroll;
}

template <typename T, int VEC, int LPR, int TILES>
void launch_nnz(int mode, const SpmmArgs<T> &a, dim3 grid, hipStream_t stream) {
    auto go = [&](auto m, auto runs) {
        constexpr int kMode = decltype(m)::value, kRuns = decltype(runs)::value;
        const dim3 block(kBlock);
        if constexpr (sizeof(T) == 4 && LPR >= kDeepRound && TILES == 1) {
            const int round = round_of<kMode, kRuns>((int64_t)grid.x * grid.y, a.nnz);
            if constexpr (kGoesDeep<kMode>)
                if (round == kDeepRound) {
                    hipLaunchKernelGGL((spmm_nnz_kernel<T, VEC, LPR, TILES, kMode, kRuns, kDeepRound>), grid, block, 0, stream, a);
                    return;
                }
            if constexpr (kMode == MODE_UNIT || kMode == MODE_ROW_MASK)
                if (round == kMidRound) {
                    hipLaunchKernelGGL((spmm_nnz_kernel<T, VEC, LPR, TILES, kMode, kRuns, kMidRound>), grid, block, 0, stream, a);
                    return;
                }
        }
        const size_t lds = kRuns != WGRUNS_ONCE ? 0
                                                : std::max((size_t)once_room(a.wg_len, a.keep) * sizeof(int),
                                                           sizeof(Pack<T, VEC>) * TILES * kBlock);
        hipLaunchKernelGGL((spmm_nnz_kernel<T, VEC, LPR, TILES, kMode, kRuns, kUnroll>), grid, block, lds, stream, a);
    };
    const std::integral_constant<int, MODE_VAL> val;
    const std::integral_constant<int, MODE_ADD> add;
    const std::integral_constant<int, MODE_UNIT> unit;
    const std::integral_constant<int, MODE_DUAL> dual;
    const std::integral_constant<int, MODE_SIGN_MASK> sign_mask;
    const std::integral_constant<int, MODE_RELU_MASK> relu_mask;
    const std::integral_constant<int, MODE_ROW_MASK> row_mask;
    if (a.rowptr64 != nullptr) {
        const std::integral_constant<int, WGRUNS_ONCE> once;
        if (a.accumulate) go(add, once);
        else go(val, once);
    } else if (a.arrivals != nullptr && a.run_start == nullptr) {
        const std::integral_constant<int, WGRUNS_COMPUTED> computed;
        if (mode == MODE_UNIT) go(unit, computed);
        else if (mode == MODE_SIGN_MASK) go(sign_mask, computed);
        else if (mode == MODE_ROW_MASK) go(row_mask, computed);
        else go(relu_mask, computed);
    } else if (a.arrivals != nullptr) {
        const std::integral_constant<int, WGRUNS_TABLE> table;
        if (mode == MODE_DUAL) go(dual, table);
        else if (a.accumulate) go(add, table);
        else go(val, table);
    } else {
        const std::integral_constant<int, WGRUNS_NONE> none;
        if (mode == MODE_VAL && a.accumulate) go(add, none);
        else if (mode == MODE_VAL) go(val, none);
        else if (mode == MODE_UNIT) go(unit, none);
        else if (mode == MODE_DUAL) go(dual, none);
        else if (mode == MODE_SIGN_MASK) go(sign_mask, none);
        else if (mode == MODE_ROW_MASK) go(row_mask, none);
        else go(relu_mask, none);
    }
}

// Products of int64 arrays that write rows without entries have at least a workgroup per kBlock rows, up to this many (as many as the
// card holds at once), however few the entries are (1,000 entries in 10^6 rows, us, with the workgroups of the entries alone / so: 1
// feature 12,500 / 13, 8 3,000 / 19, 64 2,660 / 43; a fill of the result takes 6 at 8 features, 32 at 64).  Plain stores:
// streaming ones took 49 for 36 at 64 features over 10^6 rows.
constexpr int kZeroWorkgroups = 2048;

template <typename T, int VEC, int LPR, int TILES>
int launch_shape(int kind, int mode, const SpmmArgs<T> &args, int64_t items, int grid_y, hipStream_t stream) {
    constexpr int GPB = kBlock / LPR;
    dim3 grid((unsigned)ceil_div(items, GPB), (unsigned)grid_y), block(kBlock);
    if (grid.x == 0) return CGNN_OK;
    SpmmArgs<T> a = args;
    a.stretch_log2 = 0;
    if (kind == KIND_ROW || kind == KIND_NNZ) {
        a.stretch_log2 = stretch_log2_for<GPB>(grid.x);
        a.blocks = (int32_t)grid.x;
        grid.x = (unsigned)(ceil_div((int64_t)grid.x, kXcds) * kXcds);
        if (a.rowptr64 != nullptr && !a.accumulate)
            grid.x = std::max(grid.x, (unsigned)std::min<int64_t>(kZeroWorkgroups, ceil_div((int64_t)a.rows, kBlock)));
    }
    switch (kind) {
        case KIND_ROW:
            if (mode == MODE_DUAL)
                hipLaunchKernelGGL((spmm_row_kernel<T, VEC, LPR, TILES, MODE_DUAL>), grid, block, 0, stream, a);
            else if (a.accumulate)
                hipLaunchKernelGGL((spmm_row_kernel<T, VEC, LPR, TILES, MODE_ADD>), grid, block, 0, stream, a);
            else
                hipLaunchKernelGGL((spmm_row_kernel<T, VEC, LPR, TILES, MODE_VAL>), grid, block, 0, stream, a);
            break;
        case KIND_NNZ:
            launch_nnz<T, VEC, LPR, TILES>(mode, a, grid, stream);
            break;
        case KIND_FIXUP: {  // a lane group per carry, and (when not accumulating) a thread per row
            const int64_t for_rows = a.accumulate ? 0 : ceil_div((int64_t)a.rows, kBlock);
            const int64_t for_carries = ceil_div((int64_t)a.nseg, GPB);
            const dim3 fix_grid((unsigned)(for_rows > for_carries ? for_rows : for_carries));
            if (fix_grid.x > 0 && a.merge_stride > 1)
                hipLaunchKernelGGL((spmm_fixup_kernel<T, VEC, LPR, true>), fix_grid, block, 0, stream, a);
            else if (fix_grid.x > 0)  // the short list a reduction level leaves
                hipLaunchKernelGGL((spmm_fixup_kernel<T, VEC, LPR, false>), fix_grid, block, 0, stream, a);
            break;
        }
        case KIND_FIXUP_ROWS:  // items = lane groups: one per cut row, one per empty row
            hipLaunchKernelGGL((spmm_fixup_rows_kernel<T, VEC, LPR>), dim3((unsigned)ceil_div(items, GPB)), block, 0, stream,
                               a);
            break;
        case KIND_REDUCE:  // items = chunks of kCarryFan carries, one lane group each
            hipLaunchKernelGGL((spmm_carry_reduce_kernel<T, VEC, LPR>), dim3((unsigned)ceil_div(items, GPB)), block, 0,
                               stream, a);
            break;
    }
    return check_launch("spmm launch");
}

#define CGNN_SHAPE_CASE(V, L, TL)                   \
    if (s.vec == V && s.lpr == L && s.tiles == TL)  \
        return launch_shape<T, V, L, TL>(kind, mode, a, items, s.grid_y, stream);

template <typename T>
int launch(int kind, int mode, const Shape &s, const SpmmArgs<T> &a, int64_t items, hipStream_t stream) {
    if constexpr (sizeof(T) == 4) {
        CGNN_SHAPE_CASE(4, 4, 1)
        CGNN_SHAPE_CASE(4, 8, 1)
        CGNN_SHAPE_CASE(4, 16, 1)
        CGNN_SHAPE_CASE(4, 32, 1)
        CGNN_SHAPE_CASE(4, 64, 1)
        CGNN_SHAPE_CASE(4, 64, 2)
        CGNN_SHAPE_CASE(2, 4, 1)
        CGNN_SHAPE_CASE(2, 16, 1)
        CGNN_SHAPE_CASE(2, 64, 1)
        CGNN_SHAPE_CASE(2, 64, 2)
        CGNN_SHAPE_CASE(1, 4, 1)
        CGNN_SHAPE_CASE(1, 16, 1)
        CGNN_SHAPE_CASE(1, 64, 1)
        CGNN_SHAPE_CASE(1, 64, 2)
    } else {
        CGNN_SHAPE_CASE(1, 4, 1)
        CGNN_SHAPE_CASE(1, 16, 1)
        CGNN_SHAPE_CASE(1, 64, 1)
    }
    return fail(CGNN_EUNSUPPORTED, "spmm: no kernel for this lane layout");
}

// AUTO: rows are "near regular" when the longest one is a small multiple of the mean;
// otherwise balance by non-zeros.
int schedule_for(int64_t rows, int64_t nnz, int32_t max_row_nnz, int kernel) {
    if (kernel == CGNN_SPMM_ROW || kernel == CGNN_SPMM_NNZ) return kernel;
    if (max_row_nnz <= 0) return CGNN_SPMM_NNZ;
    const double mean = rows > 0 ? (double)nnz / (double)rows : 0.0;
    const double limit = 8.0 * (mean < 8.0 ? 8.0 : mean);
    return (double)max_row_nnz <= limit ? CGNN_SPMM_ROW : CGNN_SPMM_NNZ;
}

int resolve_kernel(const cgnn_csr *A, int kernel) {
    if (kernel == CGNN_SPMM_ROW || kernel == CGNN_SPMM_NNZ) return kernel;
    if (A->rowidx == nullptr) return CGNN_SPMM_ROW;  // the nnz schedule needs the row of every non-zero
    return schedule_for(A->rows, A->nnz, A->max_row_nnz, kernel);
}

int seg_len(const cgnn_csr *A) {
    int s = A->seg_nnz > 0 ? A->seg_nnz : kDefaultSeg;
    return (s + kUnroll - 1) / kUnroll * kUnroll;
}

int check_csr(const cgnn_csr *A, const char *name) {
    if (A == nullptr) return fail(CGNN_EINVAL, "spmm: null csr");
    const int64_t lim = (int64_t)INT32_MAX - 65536;  // room for run ends past the last entry
    if (A->rows < 0 || A->cols < 0 || A->nnz < 0 || A->rows >= lim || A->nnz >= lim || A->cols >= lim) {
        set_error("%s: rows/cols/nnz must be in [0, 2^31 - 65536)", name);
        return CGNN_EINVAL;
    }
    if (A->rowptr == nullptr || (A->nnz > 0 && A->colidx == nullptr)) {
        set_error("%s: rowptr/colidx must not be null", name);
        return CGNN_EINVAL;
    }
    return CGNN_OK;
}

template <typename T>
SpmmArgs<T> make_args(const cgnn_csr *A, const void *X, const void *X1, int64_t split, const void *M, void *Y,
                      int64_t F, int accumulate) {
    SpmmArgs<T> a{};
    a.rowptr = A->rowptr;
    a.colidx = A->colidx;
    a.rowidx = A->rowidx;
    a.rowmap = A->rowmap;
    a.val = static_cast<const T *>(A->val);
    a.X = static_cast<const T *>(X);
    a.X1 = static_cast<const T *>(X1);
    a.M = static_cast<const T *>(M);
    a.Y = static_cast<T *>(Y);
    a.F = F;
    a.rows = (int32_t)A->rows;
    a.nnz = (int32_t)A->nnz;
    a.split = (int32_t)split;
    a.accumulate = accumulate ? 1 : 0;
    return a;
}

// Workspace of the nnz schedule: per level the rows of the carries, then the carries.
// Level 0 has one carry per run; every further level has two per kCarryFan carries of the
// one before; levels are added until at most kSerialCarries carries are left.
constexpr int64_t kSerialCarries = 256;
constexpr int kMaxCarryLevels = 8;

struct CarryLevels {
    int count = 0;
    int64_t n[kMaxCarryLevels];
    size_t row_off[kMaxCarryLevels], carry_off[kMaxCarryLevels];
    size_t total = 0;
};

// Rows whose carries the fix-up pass can walk directly (at most kLongChain of them, one per
// workgroup of the nnz kernel) need no reduction levels.  max_row_nnz == 0 means unknown.
constexpr int64_t kLongChain = 256;

bool wants_levels(const cgnn_csr *A, int seg, int runs_per_workgroup) {
    return A->max_row_nnz <= 0 || (int64_t)A->max_row_nnz > kLongChain * seg * runs_per_workgroup;
}

CarryLevels carry_levels(int64_t nseg, int64_t F, size_t elt, bool reduce) {
    CarryLevels L;
    int64_t n = nseg;
    while (n > 0) {
        const int k = L.count++;
        L.n[k] = n;
        L.row_off[k] = L.total;
        L.total += align_up((size_t)n * sizeof(int32_t), 256);
        L.carry_off[k] = L.total;
        L.total += align_up((size_t)n * (size_t)F * elt, 256);
        if (!reduce || n <= kSerialCarries || L.count == kMaxCarryLevels) break;
        n = 2 * ceil_div(n, kCarryFan);
    }
    return L;
}

// Pieces of the rows that workgroup runs divide among workgroups: two slots per workgroup.
size_t wg_piece_bytes(int64_t workgroups, int64_t F, size_t elt) { return 2 * (size_t)workgroups * (size_t)F * elt; }

// Non-zeros per lane group of the workgroup runs: as short as fills the card (lane groups resident at
// once: 7 workgroups per compute unit), since a run is a chain of dependent rounds of gathers and a small
// product is nothing but the time of its longest chain; not under 8 (two rounds: below that the ends of a
// run cost more than its entries); where they would be longer than `most`, the block's run length, of which several fill
// the card one after the other.

int wg_run_len(const cgnn_csr *A, int groups, int most) {
    const int64_t fill = ceil_div(ceil_div(A->nnz, kResidentWorkgroups * groups), kUnroll) * kUnroll;
    const int longest = seg_len(A);
    if (fill < 8) return longest < 8 ? longest : 8;
    return (int)(fill <= most ? fill : longest);
}

// Blocks of a plan: the run length, where two rounds of runs end more evenly than one of longer runs (forward vertex stage
// of web graphs, runs of 52 to 64 entries against 32: 80 -> 71 us for 100,000 vertices of 128 features, 89 -> 78 for 200,000
// of 64, 96 -> 87 for 200,000 of 47; of 36 to 44: 53 -> 51, 57 -> 56 and 61 -> 59 us for 47 features); rows of less than a
// cache line, whose runs are quicker, take runs a little longer (16 features, 40 and 44 entries: 28 and 31 us against 31
// and 33 of 32; 48: 39 against 34).
int most_per_run(const cgnn_csr *A, int64_t row_bytes) { return row_bytes < 128 ? seg_len(A) * 11 / 8 : seg_len(A); }

// Blocks that are new with every call: up to twice the run length.  Out-lists, near-regular rows in their natural order,
// gain from it (runs of 36 to 44 entries against 32: 42 against 50 us for 100,003 rows of 64 features), in-lists lose less
// (44 to 56 entries: 69 against 67 us for 120,000 rows, 89 against 83 for 160,000), and which a block is nobody has looked.
int most_per_new_run(const cgnn_csr *A) { return 2 * seg_len(A); }

// The layout of the row schedule.  Wide packs are for launches that fill the card several times over, where a row's
// share of the memory instructions counts.  A launch that all of it fits the card at once takes as long as its longest
// row, and that chain is shorter with more lanes: a lane group takes its entries as many at a time as it has lanes, each
// time behind a load of their columns, and a lane adds up as many features of every entry as its packs have.  There a
// row has the narrowest packs that a wave holds and as many lanes as the longest row has entries.  (118 rules of up to
// 64 vertices, 19 features: 27.5 us with packs of four on 8 lanes, 20 with 64 lanes, 17 with one feature a lane on 64;
// forward propagations over web graphs, 6,000 vertices: 8 features 36 -> 31 us, 19 38 -> 32, 47 38 -> 33, 128 38 -> 34, the
// backward vertex stage 10.3 -> 9.2; with twice the lanes the same stage of 14,000 vertices took 10.8 us instead of 9.0.)
constexpr int64_t kResidentLanes = 256 * 32 * kWave;

template <typename T>
Shape row_shape(int64_t F, int64_t rows, int64_t nnz, int32_t max_row_nnz) {
    // parts of 64 packs for rows of eight entries and more (gradient, two tiles / parts: 512 features, 325,557 vertices of 10.8
    // entries 567 / 551 us, 200,003 of 8 277 / 280, of 5 226 / 238; 10.8 entries, 5,000 vertices of 512, 768, 1,024 and 2,048 features
    // 9.0 / 9.1, 13.0 / 12.0, 15.7 / 14.8 and 27.0 / 26.0, 20,000 29.2 / 28.1, 44.2 / 39.9, 54.8 / 51.8 and 113 / 108, 100,003
    // 152 / 149, 264 / 235 and, of 1,024, 324 / 327)
    const Shape wide = pick_shape<T>(F, false, nnz < 8 * rows);
    if (sizeof(T) != 4 || wide.tiles != 1 || wide.grid_y != 1) return wide;
    Shape s = wide;
    s.vec = F <= kWave ? 1 : (F <= 2 * kWave ? 2 : 4);
    s.lpr = s.vec == 4 ? kWave : (F <= 4 * s.vec ? 4 : (F <= 16 * s.vec ? 16 : kWave));  // the layouts there are
    while (s.lpr < kWave && s.lpr < max_row_nnz) s.lpr *= 4;
    return rows * s.lpr <= kResidentLanes ? s : wide;
}

// mean (may be NULL; MODE_UNIT): whether the rows are wanted divided by their numbers of entries; false on return
// if that is left to the caller (rows so long that their carries go through the reduction levels).
template <typename T>
int spmm_typed(const cgnn_csr *A, const void *X, const void *X1, int64_t split, const void *M, void *Y, int64_t F,
               int accumulate, int kernel, int mode, void *ws, size_t ws_bytes, hipStream_t stream, bool *mean = nullptr) {
    if (A->rows == 0 || F == 0) return CGNN_OK;
    if (mode != MODE_DUAL) split = INT32_MAX;  // every column comes from X
    SpmmArgs<T> a = make_args<T>(A, X, X1, split, M, Y, F, accumulate);
    const bool masked = mode == MODE_RELU_MASK || mode == MODE_SIGN_MASK || mode == MODE_ROW_MASK;
    if (mode == MODE_SIGN_MASK || mode == MODE_ROW_MASK) {  // M holds bits, not rows
        (mode == MODE_SIGN_MASK ? a.signs : a.row_signs) = static_cast<const uint32_t *>(M);
        a.sign_words = (int32_t)ceil_div(F, 32);
        a.M = nullptr;
        M = nullptr;
    }
    const bool may_choose = kernel == CGNN_SPMM_AUTO;
    kernel = resolve_kernel(A, kernel);
    if (masked) kernel = CGNN_SPMM_NNZ;  // masks exist for the nnz schedule only
    if (mode == MODE_DUAL && A->nnz > 0 && A->val == nullptr)
        return fail(CGNN_EINVAL, "spmm: the two-source product needs stored values");
    if (kernel == CGNN_SPMM_ROW) {
        const Shape s = row_shape<T>(F, A->rows, A->nnz, A->max_row_nnz);
        return launch<T>(KIND_ROW, mode, s, a, A->rows, stream);
    }
    if (A->nnz > 0 && A->rowidx == nullptr) return fail(CGNN_EINVAL, "spmm: nnz schedule needs rowidx");
    // the lane layout decides how many runs a workgroup merges
    const Shape s = pick_shape<T>(F, true);
    const int lane_groups = kBlock / s.lpr, runs_per_workgroup = merged_runs<T>(F);
    if (may_choose && A->wg_runs != nullptr && A->arrivals != nullptr && A->wg_groups == lane_groups && A->nnz > 0) {
        const int64_t workgroups = ceil_div(A->nnz, A->wg_len);
        const size_t need = wg_piece_bytes(workgroups, F, sizeof(T));
        if (ws == nullptr || ws_bytes < need) {
            set_error("spmm: workspace of %zu bytes needed, %zu given", need, ws_bytes);
            return CGNN_EWORKSPACE;
        }
        a.run_start = A->wg_runs;
        a.arrivals = A->arrivals;
        a.wg_len = A->wg_len;
        a.nseg = (int32_t)(workgroups * lane_groups);
        a.carry = static_cast<T *>(ws);
        a.empty_rows = A->empty_rows;
        a.n_empty_rows = A->n_empty_rows;
        return launch<T>(KIND_NNZ, mode, s, a, a.nseg, stream);
    }
    const int seg = seg_len(A);
    const int64_t nseg = ceil_div(A->nnz, seg);
    const CarryLevels levels = carry_levels(nseg, F, sizeof(T), wants_levels(A, seg, runs_per_workgroup));
    if (mean != nullptr) *mean = *mean && levels.count == 1;
    a.mean = mean != nullptr && *mean;
    if (nseg > 0 && (ws == nullptr || ws_bytes < levels.total)) {
        set_error("spmm: workspace of %zu bytes needed, %zu given", levels.total, ws_bytes);
        return CGNN_EWORKSPACE;
    }
    char *base = static_cast<char *>(ws);
    auto level_rows = [&](int k) { return reinterpret_cast<int32_t *>(base + levels.row_off[k]); };
    auto level_carries = [&](int k) { return reinterpret_cast<T *>(base + levels.carry_off[k]); };
    a.nseg = (int32_t)nseg;
    a.seg_nnz = seg;
    a.run_start = A->run_start;
    a.carry_row = nseg > 0 ? level_rows(0) : nullptr;
    a.carry = nseg > 0 ? level_carries(0) : nullptr;
    a.merge_stride = runs_per_workgroup;
    if (nseg > 0) {
        int rc = launch<T>(KIND_NNZ, mode, s, a, nseg, stream);
        if (rc != CGNN_OK) return rc;
    }
    for (int k = 0; k + 1 < levels.count; ++k) {
        a.nseg = (int32_t)levels.n[k];
        a.carry_row = level_rows(k);
        a.carry = level_carries(k);
        a.carry_row_out = level_rows(k + 1);
        a.carry_out = level_carries(k + 1);
        a.merge_stride = k == 0 ? runs_per_workgroup : 1;
        int rc = launch<T>(KIND_REDUCE, mode, s, a, ceil_div(levels.n[k], kCarryFan), stream);
        if (rc != CGNN_OK) return rc;
    }
    if (levels.count > 0) {
        const int last = levels.count - 1;
        a.nseg = (int32_t)levels.n[last];
        a.carry_row = level_rows(last);
        a.carry = level_carries(last);
        a.merge_stride = last == 0 ? runs_per_workgroup : 1;
    }
    if (A->cut_rows != nullptr && levels.count == 1) {
        // the block knows which rows its runs cut (and which rows are empty): only those are looked at
        a.cut_rows = A->cut_rows;
        a.n_cut_rows = A->n_cut_rows;
        a.empty_rows = A->empty_rows;
        a.n_empty_rows = accumulate ? 0 : A->n_empty_rows;
        const int64_t items = a.n_cut_rows > a.n_empty_rows ? a.n_cut_rows : a.n_empty_rows;
        return launch<T>(KIND_FIXUP_ROWS, mode, s, a, items, stream);
    }
    const int64_t items = accumulate ? a.nseg : (a.nseg > A->rows ? a.nseg : A->rows);
    return launch<T>(KIND_FIXUP, mode, s, a, items, stream);
}

// ------------------------------------------------------- CSR preparation -------

__global__ void narrow_i64_kernel(const int64_t *__restrict__ src, int32_t *__restrict__ dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = (int32_t)src[i];
}

// run_start[s] = where the run of the nnz schedule that covers position s * seg begins.
__global__ void run_starts_kernel(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ rowidx, int32_t nnz,
                                  int32_t seg, int64_t n, int32_t *__restrict__ run_start) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int64_t e = s * seg;
    if (e >= nnz) {
        run_start[s] = nnz;
        return;
    }
    const int r = rowidx[e];
    const int s0 = rowptr[r];
    run_start[s] = (rowptr[r + 1] - s0 <= seg) ? s0 : (int32_t)e;
}

// The table of workgroup runs (cgnn_csr.wg_runs): entry w * groups + g is where lane group g of workgroup w
// begins, with kRowGoesOn set when the row there began earlier.
__global__ void wg_runs_kernel(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ rowidx, int32_t nnz,
                               int32_t wg_len, int32_t groups, int64_t n, int32_t *__restrict__ runs) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) runs[i] = wg_run_begin(rowptr, rowidx, nnz, wg_len, groups, 0, i / groups, (int)(i % groups));
}

// rowidx[e] = largest r with rowptr[r] <= e (rows without entries are skipped).
template <typename P>
__global__ void expand_rows_kernel(const P *__restrict__ rowptr, int64_t rows, int64_t nnz,
                                   int32_t *__restrict__ rowidx) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nnz;
         e += (int64_t)gridDim.x * blockDim.x) {
        int64_t lo = 0, hi = rows;  // invariant: rowptr[lo] <= e < rowptr[hi]
        while (hi - lo > 1) {
            int64_t mid = (lo + hi) >> 1;
            if ((int64_t)rowptr[mid] <= e) lo = mid;
            else hi = mid;
        }
        rowidx[e] = (int32_t)lo;
    }
}

unsigned grid_for(int64_t n) {
    int64_t b = ceil_div(n, kBlock);
    return (unsigned)(b > 16384 ? 16384 : b);
}

// narrow[c] = ids[c] as int32 (an id outside [0, groups) is replaced by the nearest valid one and
// reported): the table the composition below gathers from, half the size of the int64 ids.
__global__ void narrow_ids_kernel(const int64_t *__restrict__ ids, int64_t n, int64_t groups, int32_t *__restrict__ narrow,
                                  int32_t *__restrict__ bad) {
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x) {
        int64_t id = ids[c];
        if (id < 0 || id >= groups) {
            if (bad) *bad = 1;  // every writer stores the same value
            id = id < 0 ? 0 : groups - 1;
        }
        narrow[c] = (int32_t)id;
    }
}

// out[e] = narrow[col[e]] for the columns below first_cols, the other columns unchanged.  Four
// entries per thread, their table reads in flight together.
__global__ void compose_columns_kernel(const int32_t *__restrict__ col, int64_t nnz, int64_t first_cols,
                                       const int32_t *__restrict__ narrow, int32_t *__restrict__ out) {
    const int64_t quads = nnz / 4;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < quads; q += (int64_t)gridDim.x * blockDim.x) {
        const int4 c = reinterpret_cast<const int4 *>(col)[q];
        int4 r;
        r.x = c.x < first_cols ? narrow[c.x] : c.x;
        r.y = c.y < first_cols ? narrow[c.y] : c.y;
        r.z = c.z < first_cols ? narrow[c.z] : c.z;
        r.w = c.w < first_cols ? narrow[c.w] : c.w;
        reinterpret_cast<int4 *>(out)[q] = r;
    }
    const int64_t e = quads * 4 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < nnz) {
        const int32_t c = col[e];
        out[e] = c < first_cols ? narrow[c] : c;
    }
}

// A block with the columns from split on multiplied out (cgnn_csr_expand_columns), a wave per row: made once for a
// plan, so what counts is that a hub's entries are taken 64 at a time, and that long rules are copied by the whole wave:
// a lane takes places of the new row, not an entry (web graph of 100,003 vertices of degree 9.8: 254 us a stage
// with a lane per entry, 78 so).
__global__ __launch_bounds__(kBlock) void expand_count_kernel(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                                                              int32_t rows, int32_t split, const int32_t *__restrict__ rule_ptr,
                                                              int32_t *__restrict__ counts) {
    const int64_t row = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (row >= rows) return;
    const int lane = threadIdx.x % kWave;
    const int32_t e1 = rowptr[row + 1];
    int64_t n = 0;
    for (int64_t e = rowptr[row] + lane; e < e1; e += kWave) {
        const int32_t c = col[e];
        n += c < split ? 1 : rule_ptr[c - split + 1] - rule_ptr[c - split];
    }
#pragma unroll
    for (int s = kWave / 2; s > 0; s >>= 1) n += __shfl_xor(n, s, kWave);
    if (lane == 0) counts[row] = (int32_t)min(n, (int64_t)INT32_MAX);
}

// The magnitudes of a value as bits, in whose order they are.
__device__ __forceinline__ uint64_t magnitude(float v) { return __float_as_uint(v) & 0x7fffffffu; }
__device__ __forceinline__ uint64_t magnitude(double v) { return (uint64_t)__double_as_longlong(v) & 0x7fffffffffffffffull; }

// words of a summary that are sums, and smallest values; the others are largest ones
__host__ __device__ constexpr bool is_sum(int word) { return word == 0 || word == 2; }
__host__ __device__ constexpr bool is_least(int word) { return word == 4 || word == 6; }

__global__ void expand_summary_begin_kernel(uint64_t *__restrict__ out) {
    if (threadIdx.x < CGNN_EXPAND_SUMMARY) out[threadIdx.x] = is_least(threadIdx.x) ? ~uint64_t(0) : 0;
}

// cgnn_csr_expand_summary: integer sums and extremes, any order.  Once per plan and direction; a launch and its few rounds of
// loads (17 us for 50,001 rows of 545,000 entries), so a workgroup joins its words in LDS before it adds them to the summary.
template <typename T>
__global__ __launch_bounds__(kBlock) void expand_summary_kernel(const int32_t *__restrict__ counts, int64_t rows,
                                                                const int32_t *__restrict__ col, const T *__restrict__ val, int64_t nnz,
                                                                int32_t split, const T *__restrict__ rule_val, int64_t rule_nnz,
                                                                unsigned long long *__restrict__ out) {
    constexpr int kWaves = kBlock / kWave, kWords = CGNN_EXPAND_SUMMARY;
    __shared__ unsigned long long found[kWords][kWaves];
    unsigned long long v[kWords];
#pragma unroll
    for (int k = 0; k < kWords; ++k) v[k] = is_least(k) ? ~0ull : 0;
    auto look = [&](int k, T value) {
        const unsigned long long m = magnitude(value);
        v[k] = max(v[k], m);
        if (m != 0) v[k + 1] = min(v[k + 1], m);
    };
    const int64_t stride = (int64_t)gridDim.x * kBlock, t0 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
#pragma unroll 4
    for (int64_t r = t0; r < rows; r += stride) {
        const int32_t n = counts[r];
        v[0] += n;
        v[1] = max(v[1], (unsigned long long)n);
        v[2] += n == 0;
    }
#pragma unroll 4
    for (int64_t e = t0; e < nnz; e += stride)
        if (col[e] >= split) look(3, val[e]);
    if (rule_val != nullptr)
#pragma unroll 4
        for (int64_t e = t0; e < rule_nnz; e += stride) look(5, rule_val[e]);
    auto join = [](int k, unsigned long long a, unsigned long long b) {
        return is_sum(k) ? a + b : is_least(k) ? min(a, b) : max(a, b);
    };
#pragma unroll
    for (int k = 0; k < kWords; ++k) {
#pragma unroll
        for (int s = kWave / 2; s > 0; s >>= 1) v[k] = join(k, v[k], (unsigned long long)__shfl_xor(v[k], s, kWave));
        if (threadIdx.x % kWave == 0) found[k][threadIdx.x / kWave] = v[k];
    }
    __syncthreads();
    const int k = threadIdx.x;
    if (k >= kWords) return;
    unsigned long long all = found[k][0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) all = join(k, all, found[k][w]);
    if (is_sum(k)) atomicAdd(out + k, all);
    else if (is_least(k)) atomicMin(out + k, all);
    else atomicMax(out + k, all);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void expand_columns_kernel(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                                                                const T *__restrict__ val, int32_t rows, int32_t split,
                                                                const int32_t *__restrict__ rule_ptr,
                                                                const int32_t *__restrict__ rule_col, const T *__restrict__ rule_val,
                                                                const int32_t *__restrict__ out_ptr, int32_t *__restrict__ out_col,
                                                                T *__restrict__ out_val) {
    const int64_t row = (int64_t)blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (row >= rows) return;
    const int lane = threadIdx.x % kWave;
    const int32_t e0 = rowptr[row], e1 = rowptr[row + 1];
    int32_t out = out_ptr[row];
    const int32_t end = out_ptr[row + 1];  // nothing behind it is this row's, whatever its columns have become since they were counted
    for (int64_t base = e0; base < e1; base += kWave) {
        const int64_t e = base + lane;
        int32_t c = 0, from = 0, n = 0;
        T w = T(0);
        if (e < e1) {
            c = col[e];
            w = val[e];
            if (c >= split) from = rule_ptr[c - split];
            n = c < split ? 1 : rule_ptr[c - split + 1] - from;
        }
        int32_t upto = n;
#pragma unroll
        for (int s = 1; s < kWave; s <<= 1) {
            const int32_t below = __shfl_up(upto, s, kWave);
            if (lane >= s) upto += below;
        }
        const int32_t total = __shfl(upto, kWave - 1, kWave), before = upto - n;
        for (int32_t p0 = 0; p0 < total; p0 += kWave) {
            const int32_t p = p0 + lane;
            int k = 0;  // the entry that p comes from: as many lie wholly in front of it
#pragma unroll
            for (int s = kWave / 2; s > 0; s >>= 1)
                if (__shfl(upto, k + s - 1, kWave) <= p) k += s;
            const int32_t of = __shfl(c, k, kWave), at = __shfl(from, k, kWave) + p - __shfl(before, k, kWave);
            const T by = __shfl(w, k, kWave);
            if (p >= total || out + p >= end) continue;
            out_col[out + p] = of < split ? of : rule_col[at];
            out_val[out + p] = of >= split && rule_val != nullptr ? by * rule_val[at] : by;
        }
        out += total;
    }
}

}  // namespace

// Entry used by the cluster reductions (mean: as for spmm_typed; unit values; mask: 0 none, 1 the rows of M, where M <= 0 drops
// the element, 2 M holds ceil(F / 32) words of bits per row, where a clear bit drops it, 3 such words per sum).
static int member_mode(int mask) {
    return mask == 3 ? MODE_ROW_MASK : (mask == 2 ? MODE_SIGN_MASK : (mask == 1 ? MODE_RELU_MASK : MODE_UNIT));
}

int spmm_members(const cgnn_csr *A, int dtype, const void *X, const void *M, void *Y, int64_t F,
                 int mask, void *ws, size_t ws_bytes, hipStream_t stream, bool *mean) {
    const int mode = member_mode(mask);
    if (dtype == CGNN_F32)
        return spmm_typed<float>(A, X, nullptr, 0, M, Y, F, 0, CGNN_SPMM_NNZ, mode, ws, ws_bytes, stream, mean);
    if (dtype == CGNN_F64)
        return spmm_typed<double>(A, X, nullptr, 0, M, Y, F, 0, CGNN_SPMM_NNZ, mode, ws, ws_bytes, stream, mean);
    return fail(CGNN_EUNSUPPORTED, "spmm: dtype must be f32 or f64");
}

// The same sums in one launch (workgroup runs): mask as above.  A member list of at most kDefaultSeg rows is
// summed in ascending order, undivided, like there; a longer one in another order.
int spmm_member_runs(const cgnn_csr *A, int dtype, const void *X, const void *M, void *Y, int64_t F, int mask, int32_t *arrivals,
                     void *ws, size_t ws_bytes, hipStream_t stream) {
    auto run = [&](auto zero) {
        typedef decltype(zero) T;
        const Shape s = pick_shape<T>(F, true);
        const int groups = kBlock / s.lpr, wg_len = wg_run_len(A, groups, most_per_new_run(A)) * groups;
        const int64_t workgroups = ceil_div(A->nnz, wg_len);
        if (ws == nullptr || ws_bytes < wg_piece_bytes(workgroups, F, sizeof(T)))
            return fail(CGNN_EWORKSPACE, "member sums: workspace too small");
        SpmmArgs<T> a = make_args<T>(A, X, nullptr, INT32_MAX, M, Y, F, 0);
        const int mode = member_mode(mask);
        if (mode == MODE_SIGN_MASK || mode == MODE_ROW_MASK) {
            (mode == MODE_SIGN_MASK ? a.signs : a.row_signs) = static_cast<const uint32_t *>(M);
            a.sign_words = (int32_t)ceil_div(F, 32);
        }
        a.arrivals = arrivals;
        a.wg_len = wg_len;
        a.keep = kDefaultSeg;
        a.nseg = (int32_t)(workgroups * groups);
        a.carry = static_cast<T *>(ws);
        a.find_empty = 1;
        return launch<T>(KIND_NNZ, mode, s, a, a.nseg, stream);
    };
    return dtype == CGNN_F32 ? run(0.0f) : run(0.0);
}

// 0 arrivals: the plain runs and their pass are the better form.  That is where the launch fills the card
// several times over: a workgroup finds its runs by four dependent loads from memory and its lane groups wait for each
// other at the end, which cost 2.4 M rows of 256 features 35 us of 553, more than the pass (14 us); where the
// card is filled once or less the pass and its launch cost more (10^6 rows of 16 features: 37 us either way,
// 2,708 rows: 12 us for 18).
size_t spmm_member_runs_bytes(const cgnn_csr *A, int64_t F, int dtype, int64_t *arrivals) {
    const Shape s = shape_of(F, dtype);
    const int groups = kBlock / s.lpr;
    *arrivals = 0;
    if (A->nnz > kResidentWorkgroups * groups * kDefaultSeg) return 0;
    const int64_t workgroups = ceil_div(A->nnz, wg_run_len(A, groups, most_per_new_run(A)) * groups);
    *arrivals = workgroups * s.grid_y;
    return wg_piece_bytes(workgroups, F, dtype == CGNN_F64 ? 8 : 4);
}

// ------------------------------------------- scratch that nobody allocates -------
//
// cgnn_spmm_static runs the same kernels as cgnn_spmm with the carries of the nnz schedule in
// an array that is part of the library's device image, for callers that cannot allocate.
// Every GPU the library runs on holds its own copy of the array, at its own address, from the
// moment the image is loaded there until the process ends.
constexpr size_t kStaticScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex static_scratch_lock;
void *static_scratch_of_device[kMaxDevices] = {};

// The address of `scratch` on the device that is current in the calling thread.  In host code
// the name `scratch` is only a handle for the symbol: the device address comes from
// hipGetSymbolAddress, once per device, and is what kernels and copies are given.
int static_scratch(void **out) {
    int device = -1;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess || device < 0 || device >= kMaxDevices) {
        set_error("cgnn_spmm_static: no usable current device (%s)", e != hipSuccess ? hipGetErrorString(e) : "index out of range");
        return CGNN_ELAUNCH;
    }
    std::lock_guard<std::mutex> hold(static_scratch_lock);
    if (static_scratch_of_device[device] == nullptr) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr) {
            set_error("cgnn_spmm_static: hipGetSymbolAddress failed on device %d: %s", device, hipGetErrorString(e));
            return CGNN_ELAUNCH;
        }
        static_scratch_of_device[device] = ptr;
    }
    *out = static_scratch_of_device[device];
    return CGNN_OK;
}

}  // namespace

}  // namespace cgnn

using namespace cgnn;

extern "C" int cgnn_spmm_schedule(int64_t rows, int64_t nnz, int32_t max_row_nnz, int kernel) {
    if (kernel < CGNN_SPMM_AUTO || kernel > CGNN_SPMM_NNZ) return CGNN_SPMM_AUTO;
    return schedule_for(rows, nnz, max_row_nnz, kernel);
}

extern "C" int cgnn_spmm_run_length(const cgnn_csr *A) { return A == nullptr ? 0 : seg_len(A); }

namespace {

struct OnceLayout {
    Shape shape;
    int groups, wg_len;
    int64_t workgroups;
    size_t total;  // the pieces
};

OnceLayout once_layout(int64_t rows, int64_t nnz, int64_t F, int dtype) {
    cgnn_csr A{};
    A.rows = rows;
    A.nnz = nnz;
    A.seg_nnz = 32;  // as for the blocks of a plan
    OnceLayout L;
    // Two tiles / parts, us: 512 features, out-lists of 6,000 vertices 14.6 / 19.5, of 20,000 38.9 / 36.7, of 325,557 814 / 745.  Of
    // 768, 1,024 and 2,048 parts are faster in every block of 2^17 entries and more that was looked at, in-lists and out-lists of 20,000 and
    // 100,003 vertices of degree 5 to 9.8: 1.02 to 1.17 times.
    const bool two_tiles = nnz < (1 << 17);  // a small product
    L.shape = dtype == CGNN_F64 ? pick_shape<double>(F, true, two_tiles) : pick_shape<float>(F, true, two_tiles);
    L.groups = kBlock / L.shape.lpr;
    int run = wg_run_len(&A, L.groups, most_per_new_run(&A));
    // Floats beyond 256 features (a part of the launch per 64 packs or twice that): every part looks for the rows of its entries,
    // and the parts fill the card together, so runs are as long as that asks for, up to 64 entries of one feature a lane.  Of wider
    // packs only in small products, where runs would be shortest: in larger ones the search is little beside rows of 1 KB.
    // (In-lists and out-lists, us, runs that fill the card with one part / so: 5,000 vertices of 257 features 33.6 / 21.9 and
    // 26.2 / 18.2, of 602 38.6 / 29.7 and 29.9 / 22.9, of 2,048 67 / 67 and 44.8 / 36.4, of 4,096 123 / 115 and 82 / 63; 100,003 of
    // 513 439 / 409 and 375 / 314; 325,557 of 257 874 / 780 and 750 / 638.  Up to 32 entries whatever the packs: 20,000 vertices
    // of degree 3 and 2,048 features 63.9 / 68.9; 64 in larger products, too: 20,000 of degree 9.8 and 602 features 85 / 96.)
    if (dtype == CGNN_F32 && L.shape.grid_y > 1 && (L.shape.vec == 1 || two_tiles)) {
        const int64_t fill = ceil_div(ceil_div(nnz * L.shape.grid_y, kResidentWorkgroups * L.groups), kUnroll) * kUnroll;
        run = std::max(run, (int)std::min<int64_t>(fill, 64 / L.shape.vec));
    }
    L.wg_len = run * L.groups;
    L.workgroups = ceil_div(nnz, L.wg_len);
    L.total = wg_piece_bytes(L.workgroups, F, dtype == CGNN_F64 ? 8 : 4);
    return L;
}

template <typename T>
int spmm_once(const OnceLayout &L, int64_t rows, int64_t nnz, const int64_t *rowptr, const int64_t *col, const void *val,
              const void *X, void *Y, int64_t F, int accumulate, void *workspace, int32_t *arrivals, hipStream_t stream) {
    cgnn_csr A{};
    A.rows = rows;
    A.nnz = nnz;
    A.val = val;
    SpmmArgs<T> a = make_args<T>(&A, X, nullptr, INT32_MAX, nullptr, Y, F, accumulate);
    a.rowptr64 = rowptr;
    a.col64 = col;
    a.arrivals = arrivals;
    a.wg_len = L.wg_len;
    a.keep = kDefaultSeg;
    a.nseg = (int32_t)(L.workgroups * L.groups);
    a.carry = static_cast<T *>(workspace);
    return launch<T>(KIND_NNZ, MODE_VAL, L.shape, a, a.nseg, stream);
}

}  // namespace

extern "C" size_t cgnn_spmm_once_workspace_bytes(int64_t rows, int64_t nnz, int64_t F, int dtype, int64_t *arrivals) {
    if (arrivals) *arrivals = 0;
    if (rows <= 0 || nnz <= 0 || F <= 0) return 0;
    const OnceLayout L = once_layout(rows, nnz, F, dtype);
    if (arrivals) *arrivals = L.workgroups * L.shape.grid_y;
    return L.total;
}

extern "C" int cgnn_spmm_once(int64_t rows, int64_t nnz, const int64_t *rowptr, const int64_t *col, const void *val, int dtype,
                              const void *X, void *Y, int64_t F, int accumulate, void *workspace, size_t workspace_bytes,
                              int32_t *arrivals, cgnn_stream_t stream) {
    const int64_t lim = (int64_t)INT32_MAX - 65536;
    CGNN_REQUIRE(rows > 0 && nnz > 0 && F > 0 && rows < lim && nnz < lim, "cgnn_spmm_once: sizes must be in [1, 2^31 - 65536)");
    CGNN_REQUIRE(dtype == CGNN_F32 || dtype == CGNN_F64, "cgnn_spmm_once: dtype must be f32 or f64");
    CGNN_REQUIRE(rowptr && col && X && Y && arrivals, "cgnn_spmm_once: null array");
    const OnceLayout L = once_layout(rows, nnz, F, dtype);
    if (workspace == nullptr || workspace_bytes < L.total) return fail(CGNN_EWORKSPACE, "cgnn_spmm_once: workspace too small");
    if (dtype == CGNN_F32)
        return spmm_once<float>(L, rows, nnz, rowptr, col, val, X, Y, F, accumulate, workspace, arrivals, stream);
    return spmm_once<double>(L, rows, nnz, rowptr, col, val, X, Y, F, accumulate, workspace, arrivals, stream);
}

extern "C" int cgnn_spmm_wg_shape(const cgnn_csr *A, int64_t F, int dtype, int32_t *groups, int32_t *wg_len,
                                  int64_t *arrivals) {
    int rc = check_csr(A, "cgnn_spmm_wg_shape");
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(groups && wg_len && arrivals && F >= 1, "cgnn_spmm_wg_shape: bad argument");
    const Shape s = shape_of(F, dtype);
    *groups = kBlock / s.lpr;
    *wg_len = wg_run_len(A, *groups, most_per_run(A, F * (dtype == CGNN_F64 ? 8 : 4))) * *groups;
    *arrivals = ceil_div(A->nnz, *wg_len) * s.grid_y;
    return CGNN_OK;
}

extern "C" int cgnn_spmm_wg_runs(const cgnn_csr *A, int32_t groups, int32_t wg_len, int32_t *runs, cgnn_stream_t stream) {
    int rc = check_csr(A, "cgnn_spmm_wg_runs");
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(runs != nullptr && groups >= 1 && wg_len >= groups && wg_len % groups == 0, "cgnn_spmm_wg_runs: bad argument");
    CGNN_REQUIRE(A->nnz == 0 || A->rowidx != nullptr, "cgnn_spmm_wg_runs: the block needs rowidx");
    const int64_t n = ceil_div(A->nnz, wg_len) * groups + 1;
    hipLaunchKernelGGL(wg_runs_kernel, dim3((unsigned)ceil_div(n, kBlock)), dim3(kBlock), 0, stream, A->rowptr, A->rowidx,
                       (int32_t)A->nnz, wg_len, groups, n, runs);
    return check_launch("spmm_wg_runs");
}

extern "C" size_t cgnn_spmm_static_scratch_bytes(void) { return kStaticScratchBytes; }

extern "C" int cgnn_spmm_static_init(void) {
    void *ws = nullptr;
    return static_scratch(&ws);
}

extern "C" int cgnn_spmm_static(const cgnn_csr *A, int dtype, const void *X, void *Y, int64_t F, int accumulate,
                                int kernel, cgnn_stream_t stream) {
    int rc = check_csr(A, "cgnn_spmm_static");
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(F >= 0, "cgnn_spmm_static: F must be non-negative");
    CGNN_REQUIRE(kernel >= CGNN_SPMM_AUTO && kernel <= CGNN_SPMM_NNZ, "cgnn_spmm_static: unknown kernel id");
    CGNN_REQUIRE(dtype == CGNN_F32 || dtype == CGNN_F64, "cgnn_spmm_static: dtype must be f32 or f64");
    const size_t need = cgnn_spmm_workspace_bytes(A, F, dtype, kernel);
    if (need > kStaticScratchBytes) {
        set_error("cgnn_spmm_static: this product needs %zu bytes of scratch, the built-in array holds %zu; use "
                  "cgnn_spmm with a workspace of the caller's",
                  need, kStaticScratchBytes);
        return CGNN_EWORKSPACE;
    }
    void *ws = nullptr;
    if (need > 0) {
        rc = static_scratch(&ws);
        if (rc != CGNN_OK) return rc;
    }
    // The kernels write every carry slot and every carry-row entry they later read, so the
    // contents a previous call left in the array need no clearing.
    return cgnn_spmm(A, dtype, X, Y, F, accumulate, kernel, ws, need > 0 ? kStaticScratchBytes : 0, stream);
}

extern "C" size_t cgnn_spmm_workspace_bytes(const cgnn_csr *A, int64_t F, int dtype, int kernel) {
    if (A == nullptr || A->nnz <= 0 || F <= 0) return 0;
    if (resolve_kernel(A, kernel) == CGNN_SPMM_ROW) return 0;
    if (kernel == CGNN_SPMM_AUTO && A->wg_runs != nullptr && A->arrivals != nullptr &&
        A->wg_groups == kBlock / shape_of(F, dtype).lpr)
        return wg_piece_bytes(ceil_div(A->nnz, A->wg_len), F, dtype == CGNN_F64 ? 8 : 4);
    const int seg = seg_len(A);
    // an upper bound: the lane layout can only remove reduction levels
    return carry_levels(ceil_div(A->nnz, seg), F, dtype == CGNN_F64 ? 8 : 4, wants_levels(A, seg, 1)).total;
}

extern "C" int cgnn_spmm(const cgnn_csr *A, int dtype, const void *X, void *Y, int64_t F,
                         int accumulate, int kernel, void *workspace, size_t workspace_bytes,
                         cgnn_stream_t stream) {
    int rc = check_csr(A, "cgnn_spmm");
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(F >= 0, "cgnn_spmm: F must be non-negative");
    if (A->rows == 0 || F == 0) return CGNN_OK;
    CGNN_REQUIRE(Y != nullptr, "cgnn_spmm: Y is null");
    CGNN_REQUIRE(A->nnz == 0 || X != nullptr, "cgnn_spmm: X is null");
    CGNN_REQUIRE(kernel >= CGNN_SPMM_AUTO && kernel <= CGNN_SPMM_NNZ, "cgnn_spmm: unknown kernel id");
    if (dtype == CGNN_F32)
        return spmm_typed<float>(A, X, nullptr, 0, nullptr, Y, F, accumulate, kernel, MODE_VAL, workspace,
                                 workspace_bytes, stream);
    if (dtype == CGNN_F64)
        return spmm_typed<double>(A, X, nullptr, 0, nullptr, Y, F, accumulate, kernel, MODE_VAL, workspace,
                                  workspace_bytes, stream);
    return fail(CGNN_EUNSUPPORTED, "cgnn_spmm: dtype must be f32 or f64");
}

extern "C" int cgnn_spmm_dual(const cgnn_csr *A, int64_t split, int dtype, const void *X0, const void *X1,
                              void *Y, int64_t F, int kernel, void *workspace, size_t workspace_bytes,
                              cgnn_stream_t stream) {
    int rc = check_csr(A, "cgnn_spmm_dual");
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(F >= 0, "cgnn_spmm_dual: F must be non-negative");
    CGNN_REQUIRE(split >= 0 && split <= A->cols, "cgnn_spmm_dual: split must be in [0, cols]");
    if (A->rows == 0 || F == 0) return CGNN_OK;
    CGNN_REQUIRE(Y != nullptr, "cgnn_spmm_dual: Y is null");
    CGNN_REQUIRE(A->nnz == 0 || ((split == 0 || X0 != nullptr) && (split == A->cols || X1 != nullptr)),
                 "cgnn_spmm_dual: a source matrix is null");
    CGNN_REQUIRE(kernel >= CGNN_SPMM_AUTO && kernel <= CGNN_SPMM_NNZ, "cgnn_spmm_dual: unknown kernel id");
    if (dtype == CGNN_F32)
        return spmm_typed<float>(A, X0, X1, split, nullptr, Y, F, 0, kernel, MODE_DUAL, workspace, workspace_bytes,
                                 stream);
    if (dtype == CGNN_F64)
        return spmm_typed<double>(A, X0, X1, split, nullptr, Y, F, 0, kernel, MODE_DUAL, workspace, workspace_bytes,
                                  stream);
    return fail(CGNN_EUNSUPPORTED, "cgnn_spmm_dual: dtype must be f32 or f64");
}

extern "C" int cgnn_csr_prepare_i64(int64_t rows, int64_t nnz, const int64_t *rowptr64,
                                    const int64_t *col64, int32_t *rowptr32, int32_t *col32,
                                    int32_t *rowidx, cgnn_stream_t stream) {
    const int64_t lim = (int64_t)INT32_MAX - 65536;
    CGNN_REQUIRE(rows >= 0 && nnz >= 0 && rows < lim && nnz < lim, "cgnn_csr_prepare_i64: sizes must be in [0, 2^31 - 65536)");
    CGNN_REQUIRE(rowptr64 != nullptr, "cgnn_csr_prepare_i64: rowptr is null");
    if (rowptr32) {
        hipLaunchKernelGGL(narrow_i64_kernel, dim3(grid_for(rows + 1)), dim3(kBlock), 0, stream, rowptr64,
                           rowptr32, rows + 1);
    }
    if (col32 && nnz > 0) {
        CGNN_REQUIRE(col64 != nullptr, "cgnn_csr_prepare_i64: col is null");
        hipLaunchKernelGGL(narrow_i64_kernel, dim3(grid_for(nnz)), dim3(kBlock), 0, stream, col64, col32, nnz);
    }
    if (rowidx && nnz > 0) {
        hipLaunchKernelGGL(expand_rows_kernel<int64_t>, dim3(grid_for(nnz)), dim3(kBlock), 0, stream,
                           rowptr64, rows, nnz, rowidx);
    }
    return check_launch("csr_prepare");
}

extern "C" int cgnn_narrow_ids(int64_t n, const int64_t *ids, int64_t groups, int32_t *narrow, int32_t *bad_id,
                               cgnn_stream_t stream) {
    const int64_t lim = (int64_t)INT32_MAX - 65536;
    CGNN_REQUIRE(n >= 0 && n < lim && groups >= 1 && groups < lim, "cgnn_narrow_ids: sizes must be in [0, 2^31 - 65536), at least one group");
    if (n == 0) return CGNN_OK;
    CGNN_REQUIRE(ids && narrow, "cgnn_narrow_ids: null array");
    hipLaunchKernelGGL(narrow_ids_kernel, dim3(grid_for(n)), dim3(kBlock), 0, stream, ids, n, groups, narrow, bad_id);
    return check_launch("narrow_ids");
}

extern "C" int cgnn_csr_compose_columns(int64_t nnz, const int32_t *colidx, int64_t first_cols, const int32_t *narrow_ids,
                                        int32_t *out, cgnn_stream_t stream) {
    const int64_t lim = (int64_t)INT32_MAX - 65536;
    CGNN_REQUIRE(nnz >= 0 && nnz < lim && first_cols >= 0 && first_cols < lim, "cgnn_csr_compose_columns: sizes must be in [0, 2^31 - 65536)");
    if (nnz == 0) return CGNN_OK;
    CGNN_REQUIRE(colidx && narrow_ids && out, "cgnn_csr_compose_columns: null array");
    CGNN_REQUIRE((reinterpret_cast<uintptr_t>(colidx) | reinterpret_cast<uintptr_t>(out)) % 16 == 0,
                 "cgnn_csr_compose_columns: colidx and out must be 16-byte aligned");
    hipLaunchKernelGGL(compose_columns_kernel, dim3(grid_for((nnz + 3) / 4)), dim3(kBlock), 0, stream, colidx, nnz, first_cols,
                       narrow_ids, out);
    return check_launch("csr_compose_columns");
}

extern "C" int cgnn_spmm_run_starts(const cgnn_csr *A, int32_t *run_start, cgnn_stream_t stream) {
    int rc = check_csr(A, "cgnn_spmm_run_starts");
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(run_start != nullptr, "cgnn_spmm_run_starts: null array");
    CGNN_REQUIRE(A->nnz == 0 || A->rowidx != nullptr, "cgnn_spmm_run_starts: the block needs rowidx");
    const int seg = seg_len(A);
    const int64_t n = ceil_div(A->nnz, seg) + 1;
    hipLaunchKernelGGL(run_starts_kernel, dim3((unsigned)ceil_div(n, kBlock)), dim3(kBlock), 0, stream, A->rowptr,
                       A->rowidx, (int32_t)A->nnz, seg, n, run_start);
    return check_launch("spmm_run_starts");
}

namespace {

int check_expand(const cgnn_csr *A, int64_t split, const cgnn_csr *rules) {
    int rc = check_csr(A, "cgnn_csr_expand");
    if (rc == CGNN_OK) rc = check_csr(rules, "cgnn_csr_expand");
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(split >= 0 && split <= A->cols && A->cols - split <= rules->rows,
                 "cgnn_csr_expand: every column from split on has to be a row of the rules");
    return CGNN_OK;
}

}  // namespace

extern "C" int cgnn_csr_expand_count(const cgnn_csr *A, int64_t split, const cgnn_csr *rules, int32_t *counts,
                                     cgnn_stream_t stream) {
    int rc = check_expand(A, split, rules);
    if (rc != CGNN_OK) return rc;
    if (A->rows == 0) return CGNN_OK;
    CGNN_REQUIRE(counts != nullptr, "cgnn_csr_expand_count: counts is null");
    hipLaunchKernelGGL(expand_count_kernel, dim3((unsigned)ceil_div(A->rows, kBlock / kWave)), dim3(kBlock), 0, stream,
                       A->rowptr, A->colidx, (int32_t)A->rows, (int32_t)split, rules->rowptr, counts);
    return check_launch("csr_expand_count");
}

extern "C" int cgnn_csr_expand_summary(const cgnn_csr *A, int64_t split, const cgnn_csr *rules, int dtype, const int32_t *counts,
                                       uint64_t *summary, cgnn_stream_t stream) {
    int rc = check_expand(A, split, rules);
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(dtype == CGNN_F32 || dtype == CGNN_F64, "cgnn_csr_expand_summary: dtype must be f32 or f64");
    CGNN_REQUIRE(summary && (A->rows == 0 || counts) && (A->nnz == 0 || A->val), "cgnn_csr_expand_summary: null array");
    hipLaunchKernelGGL(expand_summary_begin_kernel, dim3(1), dim3(kWave), 0, stream, summary);
    const int64_t items = std::max(A->rows, std::max(A->nnz, rules->val != nullptr ? rules->nnz : 0));
    if (items == 0) return check_launch("csr_expand_summary");
    // as many workgroups as there are compute units: each adds seven words to the summary
    const dim3 grid((unsigned)std::min<int64_t>(ceil_div(items, 4 * kBlock), 256));
    auto run = [&](auto zero) {
        typedef decltype(zero) T;
        hipLaunchKernelGGL(expand_summary_kernel<T>, grid, dim3(kBlock), 0, stream, counts, A->rows, A->colidx,
                           static_cast<const T *>(A->val), A->nnz, (int32_t)split, static_cast<const T *>(rules->val), rules->nnz,
                           reinterpret_cast<unsigned long long *>(summary));
    };
    if (dtype == CGNN_F32) run(0.0f);
    else run(0.0);
    return check_launch("csr_expand_summary");
}

extern "C" int cgnn_csr_expand_columns(const cgnn_csr *A, int64_t split, const cgnn_csr *rules, int dtype, const int32_t *rowptr,
                                       int32_t *colidx, void *val, cgnn_stream_t stream) {
    int rc = check_expand(A, split, rules);
    if (rc != CGNN_OK) return rc;
    CGNN_REQUIRE(dtype == CGNN_F32 || dtype == CGNN_F64, "cgnn_csr_expand_columns: dtype must be f32 or f64");
    if (A->rows == 0 || A->nnz == 0) return CGNN_OK;
    CGNN_REQUIRE(A->val && rowptr && colidx && val, "cgnn_csr_expand_columns: null array");
    auto run = [&](auto zero) {
        typedef decltype(zero) T;
        hipLaunchKernelGGL(expand_columns_kernel<T>, dim3((unsigned)ceil_div(A->rows, kBlock / kWave)), dim3(kBlock), 0, stream,
                           A->rowptr, A->colidx, static_cast<const T *>(A->val), (int32_t)A->rows, (int32_t)split, rules->rowptr,
                           rules->colidx, static_cast<const T *>(rules->val), rowptr, colidx, static_cast<T *>(val));
    };
    if (dtype == CGNN_F32) run(0.0f);
    else run(0.0);
    return check_launch("csr_expand_columns");
}

extern "C" int cgnn_csr_expand_rows(int64_t rows, int64_t nnz, const int32_t *rowptr, int32_t *rowidx,
                                    cgnn_stream_t stream) {
    const int64_t lim = (int64_t)INT32_MAX - 65536;
    CGNN_REQUIRE(rows >= 0 && nnz >= 0 && rows < lim && nnz < lim, "cgnn_csr_expand_rows: sizes must be in [0, 2^31 - 65536)");
    if (nnz == 0) return CGNN_OK;
    CGNN_REQUIRE(rowptr && rowidx, "cgnn_csr_expand_rows: null array");
    hipLaunchKernelGGL(expand_rows_kernel<int32_t>, dim3(grid_for(nnz)), dim3(kBlock), 0, stream, rowptr,
                       rows, nnz, rowidx);
    return check_launch("csr_expand_rows");
}
