// libbptplan — launch plans and row groups built on the GPU (gfx950), C ABI of include/bptplan.h and include/bptbuild.h.
//
// The host builder (bptgraph.cpp) needs the index arrays on the host and tens of milliseconds per new graph.  Here the
// same plan comes out of sorts and prefix sums over the device arrays: every step is a data-parallel kernel or a
// rocPRIM primitive on the caller's stream, sizes that depend on the data stay on the device (kernels are launched
// for the upper bounds and read the actual counts from the info blocks), and all integer results are independent of
// the execution order (the only atomics are integer max / or / add whose results do not depend on their order).
//
// The reference has no plans: its kernels take the chunked CSR arrays of graph/base.py:71-86 as they are.
#include <cstring>

#include <hip/hip_runtime.h>

#include <rocprim/rocprim.hpp>

#include <cstdint>
#include <type_traits>

#include "../../include/bptattn.h"
#include "../../include/bptbuild.h"
#include "../../include/bptplan.h"

namespace {

constexpr int TPB = 256;
constexpr int FIXED_WORK = 24;        // cost of a group beyond its pairs, in pair equivalents (as the host builder)
constexpr uint32_t PAD32 = 0xFFFFFFFFu;
constexpr uint64_t PAD64 = ~uint64_t(0);

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + TPB - 1) / TPB); }

inline unsigned bits_for(uint64_t max_value) {      // bits needed to hold values 0 .. max_value
    unsigned b = 1;
    while (b < 64 && (max_value >> b) != 0) ++b;
    return b;
}

// Carves 256-byte aligned arrays out of the caller's workspace; with a null base it only adds up the sizes.
struct Bump {
    char *base;
    size_t off;
    template <typename T> T *take(int64_t n) {
        off = (off + 255) & ~size_t(255);
        T *p = base ? reinterpret_cast<T *>(base + off) : nullptr;
        off += (size_t)(n > 0 ? n : 1) * sizeof(T);
        return p;
    }
};

// ---- rocPRIM wrappers (temporary storage = one shared region of the workspace) ------------------------------------
template <typename K>
hipError_t sort_pairs(void *tmp, size_t &bytes, const K *kin, K *kout, const int32_t *vin, int32_t *vout, int64_t n,
                      unsigned end_bit, hipStream_t s) {
    return rocprim::radix_sort_pairs(tmp, bytes, kin, kout, vin, vout, (size_t)n, 0u, end_bit, s, false);
}

hipError_t scan_i32(void *tmp, size_t &bytes, const int32_t *in, int32_t *out, int64_t n, hipStream_t s) {
    return rocprim::exclusive_scan(tmp, bytes, in, out, (int32_t)0, (size_t)n, rocprim::plus<int32_t>(), s, false);
}

// largest temporary storage any primitive of the three entry points asks for
hipError_t temp_bytes(int64_t max_items, int64_t max_groups, int64_t n_edges, int64_t n_rows, size_t *out) {
    size_t best = 0, b = 0;
    hipError_t e;
    if ((e = sort_pairs<uint32_t>(nullptr, b, nullptr, nullptr, nullptr, nullptr, max_items + 1, 32, nullptr)) != hipSuccess) return e;
    best = b > best ? b : best;
    if ((e = sort_pairs<uint32_t>(nullptr, b, nullptr, nullptr, nullptr, nullptr, max_groups + 1, 32, nullptr)) != hipSuccess) return e;
    best = b > best ? b : best;
    if ((e = sort_pairs<uint64_t>(nullptr, b, nullptr, nullptr, nullptr, nullptr, n_edges + 1, 64, nullptr)) != hipSuccess) return e;
    best = b > best ? b : best;
    int64_t ns = n_rows + 1;
    ns = ns > n_edges + 1 ? ns : n_edges + 1;
    ns = ns > max_groups + 1 ? ns : max_groups + 1;
    if ((e = scan_i32(nullptr, b, nullptr, nullptr, ns, nullptr)) != hipSuccess) return e;
    best = b > best ? b : best;
    *out = best + 256;
    return hipSuccess;
}

// ---- small helpers ---------------------------------------------------------------------------------------------------
__global__ void k_fill_i32(int32_t *p, int64_t n, int32_t v) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_iota_i32(int32_t *p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) p[i] = (int32_t)i;
}

// ---- stable radix sort --------------------------------------------------------------------------------------------------
// A graph's sorts are small (10^4 .. 10^6 records, keys below the number of nodes), and there the library sort runs some twenty
// merge launches of 5 us each whatever the key width.  Here a sort is two or three least-significant-digit passes of at most 9
// bits (up to 18 key bits: two), each three launches: digit counts per tile of records, prefix over the tiles, stable
// scatter; both CSR sides share the launches (blockIdx.y).  What bounds a pass at these sizes is the launches' latency
// (4-10 us each), then the scatter's uncoalesced stores (576 k edges x 2 sides: 24 us with the 16-byte slots of the last pass).
// Both CSR sides of an edge list, call to call with the read-back: 33 765 nodes / 576 k edges 398 -> 159 us, 65 535 / 3.3 M
// 626 -> 420 us, 1 023 / 17 k 187 -> 113 us (host-bound).
// Records per thread of a tile: eight, or three for at most RS_FEW records, which then still give a tile to many CUs; the scatter
// then sums up the tiles' counts itself (at most 86 of them) instead of waiting for a third launch.
constexpr int RS_FEW = 1 << 16, RS_KPT_FEW = 3;
constexpr int RS_MAX_BITS = 9;
constexpr int RS_BINS = 1 << RS_MAX_BITS;
constexpr int RS_PREFIX_TPB = 1024;

struct RsPasses {
    int n, bits;                                  // passes, digit bits of each
};

inline RsPasses rs_passes(uint64_t max_key) {
    const unsigned b = bits_for(max_key);
    RsPasses p;
    p.n = (int)((b + RS_MAX_BITS - 1) / RS_MAX_BITS);
    p.bits = (int)((b + p.n - 1) / p.n);          // (one bit at least: the bins are taken in pairs)
    return p;
}

inline int rs_per_thread(int64_t n) { return n <= RS_FEW ? RS_KPT_FEW : 8; }
inline int64_t rs_tiles(int64_t n) { return (n + TPB * rs_per_thread(n) - 1) / (TPB * rs_per_thread(n)); }

// orders a wavefront's LDS accesses across its lanes: what one lane wrote is what another reads next
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// exclusive prefix sum of one value per thread over a block of NW wavefronts; sh holds NW + 1 ints
template <int NW> __device__ __forceinline__ int32_t block_excl_sum(int32_t v, int32_t *sh, int32_t &total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int32_t x = v;
    for (int d = 1; d < 64; d <<= 1) {
        const int32_t y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    __syncthreads();                              // (sh may still be in use by the caller's previous step)
    if (lane == 63) sh[wave] = x;
    __syncthreads();
    int32_t before = 0, all = 0;
    for (int w = 0; w < NW; ++w) {
        const int32_t c = sh[w];
        before += w < wave ? c : 0;
        all += c;
    }
    total = all;
    return before + x - v;
}

// counts[side][tile][bin]: how many records of the tile have the digit
struct RsSizes {
    int64_t n[2];                                 // records of each side
};

template <int RS_KPT, class Recs>
__global__ __launch_bounds__(TPB) void k_rs_count(Recs recs, RsSizes sizes, int shift, int bits, int32_t *counts) {
    __shared__ int32_t h[RS_BINS];
    const int bins = 1 << bits, side = blockIdx.y;
    const int64_t n = sizes.n[side];
    for (int b = threadIdx.x; b < bins; b += TPB) h[b] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t)blockIdx.x * (TPB * RS_KPT);
    bool bad = false;
    for (int r = 0; r < RS_KPT; ++r) {
        const int64_t i = i0 + r * TPB + threadIdx.x;
        const bool on = i < n;
        const int d = on ? (int)((recs.key(side, i, bad) >> shift) & (uint32_t)(bins - 1)) : -1;
        const int first = __builtin_amdgcn_readfirstlane(d);
        const uint64_t same = __ballot(d == first);
        if (same == ~uint64_t(0) && first >= 0) {             // (a high digit is often one value over a whole wavefront)
            if ((threadIdx.x & 63) == 0) atomicAdd(&h[first], 64);
        } else if (on) {
            atomicAdd(&h[d], 1);
        }
    }
    recs.report(side, __syncthreads_or(bad ? 1 : 0) != 0);
    int32_t *out = counts + ((int64_t)side * gridDim.x + blockIdx.x) * bins;
    for (int b = threadIdx.x; b < bins; b += TPB) out[b] = h[b];
}

// in place: counts[side][tile][bin] -> the records with that digit in the tiles before; totals[side][bin]: in all tiles.
// A block owns 16 bins, 64 threads share the tiles of each.
constexpr int RS_PREFIX_BINS = 16, RS_PREFIX_PARTS = RS_PREFIX_TPB / RS_PREFIX_BINS;
__global__ __launch_bounds__(RS_PREFIX_TPB) void k_rs_prefix(int32_t *counts, int32_t *totals, int64_t n_tiles, int bins) {
    __shared__ int32_t part[RS_PREFIX_PARTS][RS_PREFIX_BINS];
    const int lane = threadIdx.x % RS_PREFIX_BINS, mine = threadIdx.x / RS_PREFIX_BINS;
    const int bin = blockIdx.x * RS_PREFIX_BINS + lane, side = blockIdx.y;
    const int64_t per = (n_tiles + RS_PREFIX_PARTS - 1) / RS_PREFIX_PARTS, t0 = mine * per, t1 = t0 + per < n_tiles ? t0 + per : n_tiles;
    int32_t *c = counts + (int64_t)side * n_tiles * bins + bin;
    const bool on = bin < bins;
    int32_t sum = 0;
    if (on)
        for (int64_t t = t0; t < t1; ++t) sum += c[t * bins];
    part[mine][lane] = sum;
    __syncthreads();
    int32_t run = 0, all = 0;
    for (int w = 0; w < RS_PREFIX_PARTS; ++w) {
        run += w < mine ? part[w][lane] : 0;
        all += part[w][lane];
    }
    if (!on) return;
    if (mine == 0) totals[side * bins + bin] = all;
    for (int64_t t = t0; t < t1; t += 8) {            // (eight loads in flight: the stores in between would serialise them)
        int32_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = t + j < t1 ? c[(t + j) * bins] : 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (t + j < t1) c[(t + j) * bins] = run;
            run += v[j];
        }
    }
}

// Stable scatter of a tile: a wavefront ranks 64 records at a time among its lanes with the same digit (one ballot per digit bit)
// on top of its running counts in LDS.
// SUM: the tile sums up the counts itself (few tiles), else k_rs_prefix has.
template <int RS_KPT, bool SUM, class Recs, class Out>
__global__ __launch_bounds__(TPB) void k_rs_scatter(Recs recs, Out out, RsSizes sizes, int shift, int bits, const int32_t *counts,
                                                    const int32_t *totals) {
    const int64_t n = sizes.n[blockIdx.y];
    constexpr int NW = TPB / 64;
    __shared__ int32_t wh[NW][RS_BINS];
    __shared__ int32_t sh[NW + 1];
    const int bins = 1 << bits, side = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int b = threadIdx.x; b < bins; b += TPB)
        for (int w = 0; w < NW; ++w) wh[w][b] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t)blockIdx.x * (TPB * RS_KPT) + wave * (64 * RS_KPT) + lane;
    const uint64_t below = (uint64_t(1) << lane) - 1;
    uint32_t key[RS_KPT];
    int32_t rank[RS_KPT];
    bool bad = false;
#pragma unroll
    for (int r = 0; r < RS_KPT; ++r) key[r] = i0 + r * 64 < n ? recs.key(side, i0 + r * 64, bad) : 0u;
#pragma unroll
    for (int r = 0; r < RS_KPT; ++r) {
        const bool on = i0 + r * 64 < n;
        const int d = (int)((key[r] >> shift) & (uint32_t)(bins - 1));
        uint64_t peers = __ballot(on);
        for (int b = 0; b < bits; ++b) {
            const bool bit = (d >> b) & 1;
            const uint64_t m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const int32_t before = wh[wave][d];
        rank[r] = before + __popcll(peers & below);
        wave_lds_order();
        if (on && (peers & below) == 0) wh[wave][d] = before + __popcll(peers);
        wave_lds_order();
    }
    // where the tile's records of every digit start: two bins a thread
    int32_t tot[2] = {0, 0}, pre[2] = {0, 0}, all;
    const int b0 = 2 * threadIdx.x;
    if (SUM) {
        if (b0 < bins) {
            const int2 *c = reinterpret_cast<const int2 *>(counts + (int64_t)side * gridDim.x * bins + b0);
#pragma unroll 8
            for (unsigned t = 0; t < gridDim.x; ++t) {
                const int2 v = c[(int64_t)t * (bins / 2)];
                tot[0] += v.x;
                tot[1] += v.y;
                pre[0] += t < blockIdx.x ? v.x : 0;
                pre[1] += t < blockIdx.x ? v.y : 0;
            }
        }
    } else {
        for (int t = 0; t < 2; ++t)
            if (b0 + t < bins) {
                tot[t] = totals[side * bins + b0 + t];
                pre[t] = counts[((int64_t)side * gridDim.x + blockIdx.x) * bins + b0 + t];
            }
    }
    int32_t start = block_excl_sum<NW>(tot[0] + tot[1], sh, all);
    for (int t = 0; t < 2; ++t) {
        if (b0 + t < bins) {
            int32_t at = start + pre[t];
            for (int w = 0; w < NW; ++w) {
                const int32_t c = wh[w][b0 + t];
                wh[w][b0 + t] = at;
                at += c;
            }
        }
        start += tot[t];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_KPT; ++r) {
        const int64_t i = i0 + r * 64;
        if (i < n) out.put(side, (int64_t)wh[wave][(key[r] >> shift) & (uint32_t)(bins - 1)] + rank[r], key[r], recs.val(side, i));
    }
}

// records in plain arrays (the passes after the first)
struct RsArrays {
    const uint32_t *k[2];
    const int32_t *v[2];
    __device__ uint32_t key(int side, int64_t i, bool &) const { return k[side][i]; }
    __device__ int32_t val(int side, int64_t i) const { return v[side][i]; }
    __device__ void report(int, bool) const {}
};
struct RsToArrays {
    uint32_t *k[2];
    int32_t *v[2];
    __device__ void put(int side, int64_t at, uint32_t key, int32_t val) const {
        k[side][at] = key;
        v[side][at] = val;
    }
};

// Stable radix sort of n words in LDS by a workgroup of 16 wavefronts: by bits [shift, shift + bits), a digit of at most 8 a pass, each
// wavefront a run of up to KPT * 64 words, ranked as k_rs_scatter does.  hist: 16 x 256 ints.  (A bitonic sort in its place, 5 600 edges in
// 8 192 places: k_csr_small 17 -> 36 us, k_plan_small 19 -> 27.)
constexpr int SMALL_TPB = 1024, SMALL_NW = SMALL_TPB / 64, SMALL_BINS = 256;
template <int KPT> __device__ __forceinline__ void lds_radix(uint32_t *word, int n, int shift, int bits, int32_t *hist, int32_t *sh) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, passes = (bits + 7) / 8, digit = (bits + passes - 1) / passes, bins = 1 << digit;
    const int per = (n + SMALL_NW * 64 - 1) / (SMALL_NW * 64), i0 = wave * per * 64 + lane;          // (at most KPT)
    const uint64_t below = (uint64_t(1) << lane) - 1;
    for (int p = 0; p < passes; ++p, shift += digit) {
        uint32_t key[KPT];
        int32_t rank[KPT];
        for (int b = tid; b < SMALL_NW * bins; b += SMALL_TPB) hist[b] = 0;
#pragma unroll
        for (int r = 0; r < KPT; ++r) key[r] = r < per && i0 + r * 64 < n ? word[i0 + r * 64] : 0u;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < KPT; ++r) {
            const bool on = r < per && i0 + r * 64 < n;
            if (__ballot(on) == 0) continue;
            const int d = (int)((key[r] >> shift) & (uint32_t)(bins - 1));
            uint64_t peers = __ballot(on);
            for (int b = 0; b < digit; ++b) {
                const bool bit = (d >> b) & 1;
                const uint64_t m = __ballot(bit);
                peers &= bit ? m : ~m;
            }
            const int32_t before = hist[wave * bins + d];
            rank[r] = before + __popcll(peers & below);
            wave_lds_order();
            if (on && (peers & below) == 0) hist[wave * bins + d] = before + __popcll(peers);
            wave_lds_order();
        }
        __syncthreads();
        int32_t sum = 0, all;
        if (tid < bins)
            for (int w = 0; w < SMALL_NW; ++w) sum += hist[w * bins + tid];
        int32_t at = block_excl_sum<SMALL_NW>(sum, sh, all);
        if (tid < bins)
            for (int w = 0; w < SMALL_NW; ++w) {
                const int32_t c = hist[w * bins + tid];
                hist[w * bins + tid] = at;
                at += c;
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < KPT; ++r)
            if (r < per && i0 + r * 64 < n) word[hist[wave * bins + (int)((key[r] >> shift) & (uint32_t)(bins - 1))] + rank[r]] = key[r];
        __syncthreads();
    }
}

// start[0 .. n] of a workgroup of 16 wavefronts: where nothing was put (INT32_MAX), what was put next behind it; start[n] was put.  (The thread
// of an edge or unit that filled in the rows before its own went over all of them when only some late rows have edges: 4000 nodes whose edges all
// point to the last, both sides' CSRs 60 us by the launches for larger graphs, 153 filled in by one thread, 47 by the workgroup.)
__device__ __forceinline__ void fill_starts(int32_t *start, int n, int32_t *sh) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, per = (n + SMALL_TPB) / SMALL_TPB;
    const int r0 = min(tid * per, n + 1), r1 = min(r0 + per, n + 1);
    int32_t least = INT32_MAX;
    for (int r = r0; r < r1; ++r) least = min(least, start[r]);
    for (int d = 1; d < 64; d <<= 1) {
        const int32_t y = __shfl_down(least, d);
        if (lane + d < 64) least = min(least, y);
    }
    __syncthreads();                              // (sh may still be in use by the caller's previous step)
    if (lane == 0) sh[wave] = least;
    const int32_t next = __shfl_down(least, 1);
    int32_t after = lane < 63 ? next : INT32_MAX;
    __syncthreads();
    for (int w = wave + 1; w < SMALL_NW; ++w) after = min(after, sh[w]);
    for (int r = r1 - 1; r >= r0; --r) start[r] = after = min(start[r], after);
    __syncthreads();
}

// f(own, t) for t = 0 .. n - 1 of every lane: by itself where it has few, by the wavefront together where it has many (a row with most of a graph's
// edges).  All lanes of the wavefront are here.
template <int K, typename F> __device__ __forceinline__ void for_each_of_lane(int n, const int32_t (&own)[K], F &&f) {
    constexpr int FEW = 8;
    const int lane = threadIdx.x & 63;
    if (n <= FEW)
        for (int t = 0; t < n; ++t) f(own, t);
    for (uint64_t many = __ballot(n > FEW); many != 0; many &= many - 1) {
        const int owner = __ffsll((unsigned long long)many) - 1, k = __shfl(n, owner);
        int32_t of[K];
#pragma unroll
        for (int i = 0; i < K; ++i) of[i] = __shfl(own[i], owner);
        for (int t = lane; t < k; t += 64) f(of, t);
    }
}

// ---- base plan ---------------------------------------------------------------------------------------------------------
// Five launches and the sort: clear; narrow the indices, check the units, find the rows; emit the items; their smallest and
// largest neighbour; sort by the smallest.
constexpr int ITEM_ROWS = TPB - 1;    // rows of a block of the first two kernels (one thread more: the end of the last row)

struct GroupRec {                     // what a group is known by before the groups are numbered
    int32_t n_entries, n_pairs, key;            // key: smallest neighbour
};

// One side's arrays through all the kernels of its plan; up to two sides share the launches (blockIdx.y): most of these kernels
// take the 3-10 us that any launch over some 10^4 items takes.  Both sides' tile plans and their pair mapping, call to call:
// 33 765 nodes / 576 k edges 1831 us in library sorts, 481 one side after the other with five waits, 288 together with two.
struct PlanSide {
    const int64_t *row, *ipu, *eid, *indices;           // as the caller has them
    int64_t n_units, n_edges, n_rows, n_index_nodes, max_items;
    int32_t seg_len;
    int32_t *rowptr, *idx32, *eid32, *heavy, *info;     // the base plan
    int4 *items;
    int2 *bounds;
    int32_t *seen;                                      // its workspace
    int4 *totals;                                       // per block of ITEM_ROWS rows: items, heavy rows, slots, largest degree
    int4 *items_tmp;                                    // in row order
    int2 *bounds_tmp;
    // groups
    int32_t mode, by_work, max_groups;
    int place_bits, g_bits, key_bits, work_bits;
    int32_t *jorder;
    GroupRec *rec;
    int32_t *order, *entry0, *pair0, *chunks;           // final order: group as formed, first entry, first pair
    int4 *placed;                                       // groups in locality order: word of the final order, entries, pairs, group
    int4 *entries;                                      // parked: neighbour, mask, first pair inside the group
    int32_t *pairs;                                     // parked: edge ids in pair order
    int32_t *out_info;
};
struct PlanSides {
    PlanSide side[2];
};

inline int64_t item_row_blocks(int64_t n_rows) { return (n_rows + ITEM_ROWS) / ITEM_ROWS; }

void base_layout(Bump &b, PlanSide &S) {
    S.seen = b.take<int32_t>(S.n_edges);
    S.totals = b.take<int4>(item_row_blocks(S.n_rows));
    S.items_tmp = b.take<int4>(S.max_items);
    S.bounds_tmp = b.take<int2>(S.max_items);
}

struct SortWs {                       // the sorts of up to two sides of max_items items
    uint32_t *key[2];
    int32_t *val[2];
    int32_t *counts, *totals;
};
SortWs sort_layout(Bump &b, int64_t max_items, int n_sides) {
    SortWs w;
    for (int i = 0; i < 2; ++i) {
        w.key[i] = b.take<uint32_t>(n_sides * max_items);
        w.val[i] = b.take<int32_t>(n_sides * max_items);
    }
    w.counts = b.take<int32_t>(n_sides * rs_tiles(max_items) * RS_BINS);
    w.totals = b.take<int32_t>(n_sides * RS_BINS);
    return w;
}

__global__ void k_plan_clear(PlanSides b) {
    const PlanSide &S = b.side[blockIdx.y];
    const int64_t *ipu = S.ipu;
    const int64_t n_units = S.n_units, n_edges = S.n_edges;
    int32_t *info = S.info;
    if (threadIdx.x != 0) return;
    for (int t = 0; t < 16; ++t) info[t] = 0;
    int err = 0;
    bool covers = (n_edges == 0);
    if (n_units > 0) {
        const int64_t first = ipu[0], last = ipu[n_units];
        if (first < 0 || last >= INT32_MAX) err = 3;
        else if (last > n_edges) err = 1;
        covers = (first == 0 && last == n_edges);
    }
    info[BPT_PI_ERR] = err;
    info[BPT_PI_FLAGS] = covers ? 1 : 0;
}

// Three kinds of blocks: edge slots (indices to 32 bits, eid a permutation?), units (sorted?), rows (rowptr[r] = start of the
// first unit whose row is >= r, and what the block's rows give).  Malformed arrays set info[BPT_PI_ERR]; what the row blocks
// then wrote is not used.
__global__ __launch_bounds__(TPB) void k_plan_narrow(PlanSides b, unsigned edge_blocks, unsigned unit_blocks) {
    const PlanSide &S = b.side[blockIdx.y];
    const int64_t *row = S.row, *ipu = S.ipu, *eid = S.eid, *indices = S.indices;
    const int64_t n_units = S.n_units, n_edges = S.n_edges, n_rows = S.n_rows, n_index_nodes = S.n_index_nodes;
    const int32_t seg_len = S.seg_len;
    int32_t *info = S.info, *idx32 = S.idx32, *eid32 = S.eid32, *seen = S.seen, *rowptr = S.rowptr;
    int4 *totals = S.totals;
    if (blockIdx.x < edge_blocks) {
        const int64_t p = (int64_t)blockIdx.x * TPB + threadIdx.x;
        if (p >= n_edges) return;
        const int64_t e = eid[p], c = indices ? indices[p] : 0;
        if (e < 0 || e >= n_edges || c < 0 || (indices && c >= n_index_nodes)) {
            atomicMax(&info[BPT_PI_ERR], 1);
            eid32[p] = 0;
            idx32[p] = 0;
            return;
        }
        eid32[p] = (int32_t)e;
        idx32[p] = (int32_t)c;
        seen[e] = (int32_t)p;                          // (checked by k_plan_items' edge blocks: every slot finds itself there)
        return;
    }
    if (blockIdx.x < edge_blocks + unit_blocks) {
        const int64_t u = (int64_t)(blockIdx.x - edge_blocks) * TPB + threadIdx.x;
        if (u >= n_units) return;
        int err = 0;
        if (row[u] < 0 || row[u] >= n_rows) err = 1;
        if (u > 0 && row[u] < row[u - 1]) err = err > 2 ? err : 2;
        if (ipu[u + 1] < ipu[u]) err = err > 2 ? err : 2;
        if (err) atomicMax(&info[BPT_PI_ERR], err);
        return;
    }
    __shared__ int32_t start[TPB];
    __shared__ int32_t sh[TPB / 64 + 1];
    const unsigned blk = blockIdx.x - edge_blocks - unit_blocks;
    const int64_t r = (int64_t)blk * ITEM_ROWS + threadIdx.x;
    if (blk >= (unsigned)((n_rows + ITEM_ROWS) / ITEM_ROWS)) return;         // (the other side has more rows)
    int32_t at = 0;
    if (r <= n_rows && n_units > 0) {
        int64_t lo = 0, hi = n_units;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (row[mid] < r) lo = mid + 1; else hi = mid;
        }
        at = (int32_t)ipu[lo];
    }
    if (r <= n_rows) rowptr[r] = at;
    start[threadIdx.x] = at;
    __syncthreads();
    int32_t deg = 0, n_seg = 0;
    const bool mine = threadIdx.x < ITEM_ROWS && r < n_rows;
    if (mine) {
        deg = max(start[threadIdx.x + 1] - at, 0);
        n_seg = deg > seg_len ? (deg - 1) / seg_len + 1 : 0;
    }
    int32_t items, heavy, slots;
    block_excl_sum<TPB / 64>(mine ? max(n_seg, 1) : 0, sh, items);
    block_excl_sum<TPB / 64>(n_seg > 0 ? 1 : 0, sh, heavy);
    block_excl_sum<TPB / 64>(n_seg, sh, slots);
    for (int d = 32; d > 0; d >>= 1) deg = max(deg, __shfl_xor(deg, d));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = deg;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < TPB / 64; ++w) deg = max(deg, sh[w]);
        totals[blk] = make_int4(items, heavy, slots, deg);
    }
}

// items of every row in row order, the heavy rows, the counts; a row of more than ITEM_FEW segments is written by the whole
// block.  The blocks behind those of the rows finish the check that eid is a permutation: two slots of one edge left one
// number in `seen`, and the other slot does not find itself (plain stores and loads: the two kernels 20 us for 576 k edges,
// with a counter per edge and its clearing 27).
constexpr int ITEM_FEW = 8;
__global__ __launch_bounds__(TPB) void k_plan_items(PlanSides b, unsigned most_row_blocks) {
    const PlanSide &S = b.side[blockIdx.y];
    const int32_t *rowptr = S.rowptr, *eid32 = S.eid32, *seen = S.seen;
    const int64_t n_rows = S.n_rows, n_edges = S.n_edges;
    const int32_t seg_len = S.seg_len;
    const int4 *totals = S.totals;
    int32_t *info = S.info, *heavy = S.heavy;
    int4 *items = S.indices ? S.items_tmp : S.items;   // (without indices the items stay in row order, as on the host)
    const unsigned row_blocks = (unsigned)((n_rows + ITEM_ROWS) / ITEM_ROWS);
    __shared__ int32_t sh[TPB / 64 + 1];
    __shared__ int32_t many[TPB][3];                   // row, first item, first slot
    __shared__ int32_t n_many;
    if (info[BPT_PI_ERR]) return;
    if (blockIdx.x >= most_row_blocks) {
        const int64_t p = (int64_t)(blockIdx.x - most_row_blocks) * TPB + threadIdx.x;
        if (p < n_edges && seen[eid32[p]] != (int32_t)p) atomicAnd(&info[BPT_PI_FLAGS], ~1);
        return;
    }
    if (blockIdx.x >= row_blocks) return;
    if (threadIdx.x == 0) n_many = 0;
    const bool last = blockIdx.x == row_blocks - 1;
    int4 part = make_int4(0, 0, 0, 0);
    for (unsigned b = threadIdx.x; b < blockIdx.x; b += TPB) {
        const int4 t = totals[b];
        part.x += t.x; part.y += t.y; part.z += t.z;
        part.w = max(part.w, t.w);
    }
    int4 before;
    block_excl_sum<TPB / 64>(part.x, sh, before.x);
    block_excl_sum<TPB / 64>(part.y, sh, before.y);
    block_excl_sum<TPB / 64>(part.z, sh, before.z);
    if (last) atomicMax(&info[BPT_PI_MAX_DEGREE], threadIdx.x == 0 ? max(part.w, totals[blockIdx.x].w) : part.w);
    const int64_t r = (int64_t)blockIdx.x * ITEM_ROWS + threadIdx.x;
    const bool mine = threadIdx.x < ITEM_ROWS && r < n_rows;
    const int32_t begin = mine ? rowptr[r] : 0, end = mine ? rowptr[r + 1] : 0, deg = end - begin;
    const int32_t n_seg = deg > seg_len ? (deg - 1) / seg_len + 1 : 0;
    int32_t n_items, n_heavy, n_slots;
    const int32_t item = before.x + block_excl_sum<TPB / 64>(mine ? max(n_seg, 1) : 0, sh, n_items);
    const int32_t hv = before.y + block_excl_sum<TPB / 64>(n_seg > 0 ? 1 : 0, sh, n_heavy);
    const int32_t slot = before.z + block_excl_sum<TPB / 64>(n_seg, sh, n_slots);
    if (mine && n_seg == 0) items[item] = make_int4((int32_t)r, begin, end, -1);
    if (n_seg > 0) {
        heavy[3 * (int64_t)hv] = (int32_t)r;
        heavy[3 * (int64_t)hv + 1] = slot;
        heavy[3 * (int64_t)hv + 2] = n_seg;
        if (n_seg <= ITEM_FEW) {
            for (int32_t t = 0; t < n_seg; ++t)
                items[item + t] = make_int4((int32_t)r, begin + t * seg_len, min(end, begin + (t + 1) * seg_len), slot + t);
        } else {
            const int i = atomicAdd(&n_many, 1);
            many[i][0] = (int32_t)r;
            many[i][1] = item;
            many[i][2] = slot;
        }
    }
    __syncthreads();
    for (int i = 0; i < n_many; ++i) {
        const int32_t row = many[i][0], b = rowptr[row], e = rowptr[row + 1], n = (e - b - 1) / seg_len + 1;
        for (int32_t t = threadIdx.x; t < n; t += TPB)
            items[many[i][1] + t] = make_int4(row, b + t * seg_len, min(e, b + (t + 1) * seg_len), many[i][2] + t);
    }
    if (last && threadIdx.x == 0) {
        info[BPT_PI_N_ITEMS] = before.x + n_items;
        info[BPT_PI_N_HEAVY] = before.y + n_heavy;
        info[BPT_PI_N_SLOTS] = before.z + n_slots;
    }
}

// smallest and largest neighbour id of every item, sixteen lanes an item; an empty item: its own row id clipped to
// n_index_nodes, twice
__global__ __launch_bounds__(TPB) void k_item_bounds(PlanSides b) {
    const PlanSide &S = b.side[blockIdx.y];
    const int32_t *idx32 = S.idx32, *info = S.info;
    const int64_t n_index_nodes = S.n_index_nodes, n_edges = S.n_edges;
    const int4 *items = S.indices ? S.items_tmp : S.items;
    int2 *bounds = S.indices ? S.bounds_tmp : S.bounds;
    const int64_t i = (int64_t)blockIdx.x * (TPB / 16) + (threadIdx.x >> 4);
    if (i >= S.max_items || info[BPT_PI_ERR] || i >= info[BPT_PI_N_ITEMS]) return;
    const int4 it = items[i];
    int32_t lo, hi;
    if (it.z > it.y && it.y >= 0 && it.z <= n_edges) {          // (an item list from elsewhere is not trusted with addresses)
        lo = INT32_MAX;
        hi = 0;
        for (int32_t p = it.y + (threadIdx.x & 15); p < it.z; p += 16) {
            lo = min(lo, idx32[p]);
            hi = max(hi, idx32[p]);
        }
        for (int d = 8; d > 0; d >>= 1) {
            lo = min(lo, __shfl_xor(lo, d, 16));
            hi = max(hi, __shfl_xor(hi, d, 16));
        }
    } else {
        lo = hi = (it.x >= 0 && it.x < n_index_nodes) ? it.x : (int32_t)n_index_nodes;
    }
    if ((threadIdx.x & 15) == 0) bounds[i] = make_int2(lo, hi);
}

// the items as sort records, by their smallest or largest neighbour; places past the last item sort behind all of them
struct ItemRecs {
    PlanSides b;
    int largest;                      // by the largest, of the items as sorted by the smallest
    __device__ uint32_t key(int side, int64_t i, bool &) const {
        const PlanSide &S = b.side[side];
        if (S.info[BPT_PI_ERR] || i >= S.info[BPT_PI_N_ITEMS]) return (uint32_t)S.n_index_nodes + 1;
        return (uint32_t)(largest ? S.bounds[i].y : S.bounds_tmp[i].x);
    }
    __device__ int32_t val(int, int64_t i) const { return (int32_t)i; }
    __device__ void report(int, bool) const {}
};
struct ItemsSorted {
    PlanSides b;
    __device__ void put(int side, int64_t at, uint32_t, int32_t i) const {
        const PlanSide &S = b.side[side];
        if (S.info[BPT_PI_ERR] || i >= S.info[BPT_PI_N_ITEMS]) return;
        S.items[at] = S.items_tmp[i];
        if (S.bounds) S.bounds[at] = S.bounds_tmp[i];
    }
};

// The items in LDS: by their smallest neighbour (word: that and their place, BITS bits), the records moved, then, where groups follow, the
// order by the largest.  A sort key is n_index_nodes at most (an item without edges).
template <int BITS, int KPT> __device__ __forceinline__ void order_by_largest(const PlanSide &S, int n_items, uint32_t *word, int32_t *hist, int32_t *sh) {
    const int tid = threadIdx.x, key_bits = 32 - __clz((int)S.n_index_nodes | 1);
    for (int at = tid; at < n_items; at += SMALL_TPB) word[at] = ((uint32_t)S.bounds[at].y << BITS) | (uint32_t)at;
    __syncthreads();
    lds_radix<KPT>(word, n_items, BITS, key_bits, hist, sh);
    for (int at = tid; at < n_items; at += SMALL_TPB) S.jorder[at] = (int32_t)(word[at] & ((1u << BITS) - 1u));
}
template <int BITS, int KPT> __device__ __forceinline__ void order_items(const PlanSide &S, int n_items, uint32_t *word, int32_t *hist, int32_t *sh) {
    const int tid = threadIdx.x, key_bits = 32 - __clz((int)S.n_index_nodes | 1);
    lds_radix<KPT>(word, n_items, BITS, key_bits, hist, sh);
    for (int at = tid; at < n_items; at += SMALL_TPB) {
        const int i = (int)(word[at] & ((1u << BITS) - 1u));
        S.items[at] = S.items_tmp[i];
        if (S.bounds) S.bounds[at] = S.bounds_tmp[i];
    }
    if (!S.jorder || !S.bounds) return;
    __syncthreads();
    order_by_largest<BITS, KPT>(S, n_items, word, hist, sh);
}

// Both orders of up to 11 264 items (60 KB of LDS) by a workgroup a side, in place of the eight launches of the two sorts (5 to 7 us each).
// One CU is the bound, so the line lies where its LDS ends: 8 trees of 400 leaves, 10 900 items a side, 46 us of launches -> 27.5, a training
// pass on a new graph 551 -> 532 us (three processes each way); 16 of 100 leaves 575 -> 545.
constexpr int ORDER_ITEM_BITS = 14, ORDER_ITEMS = 11 * SMALL_TPB;
inline bool order_in_lds(const PlanSide &S) { return S.max_items <= ORDER_ITEMS && S.n_index_nodes < 1 << (32 - ORDER_ITEM_BITS); }
__global__ __launch_bounds__(SMALL_TPB) void k_item_order(PlanSides b) {
    const PlanSide &S = b.side[blockIdx.x];
    __shared__ uint32_t word[ORDER_ITEMS];
    __shared__ int32_t hist[SMALL_NW * SMALL_BINS], sh[SMALL_NW + 1];
    if (S.info[BPT_PI_ERR]) return;
    const int n_items = min(S.info[BPT_PI_N_ITEMS], ORDER_ITEMS);
    for (int i = threadIdx.x; i < n_items; i += SMALL_TPB) word[i] = ((uint32_t)S.bounds_tmp[i].x << ORDER_ITEM_BITS) | (uint32_t)i;
    __syncthreads();
    order_items<ORDER_ITEM_BITS, ORDER_ITEMS / SMALL_TPB>(S, n_items, word, hist, sh);
}

// The base plans of a small graph, and the order of their items by the largest neighbour where groups follow (jorder): a workgroup a
// side does in one launch what the launches above and their two sorts, thirteen or seventeen of 4 us and more whatever they have to do, do for
// larger ones, bit for bit.  Neighbours (16 bits) and sort words (key and place) stay in LDS, 57 KB, which set the limits; bound by the
// latency of the six steps: 19 us at 5 600 edges in place of some 70 of launches.  With k_csr_small, a training pass on new graphs: 5 trees
// of 51 leaves 725 -> 311 us, 59 of 16 in bfloat16 775 -> 357.
constexpr int SMALL_ITEM_BITS = 12, SMALL_ITEMS = 1 << SMALL_ITEM_BITS, SMALL_EDGES = 12288;
inline bool small_plan(const PlanSide &S) { return S.n_edges <= SMALL_EDGES && S.max_items <= SMALL_ITEMS && S.n_index_nodes <= 0xFFFF; }

__global__ __launch_bounds__(SMALL_TPB) void k_plan_small(PlanSides b, int32_t *info_out) {
    constexpr int NW = SMALL_TPB / 64;
    const PlanSide &S = b.side[blockIdx.x];
    const int64_t *row = S.row, *ipu = S.ipu, *eid = S.eid, *indices = S.indices;
    const int n_units = (int)S.n_units, n_edges = (int)S.n_edges, n_rows = (int)S.n_rows, seg_len = S.seg_len, tid = threadIdx.x;
    __shared__ uint32_t word[SMALL_ITEMS + 1];                    // the rows' starts, then the sort words
    __shared__ uint16_t nbr[SMALL_EDGES];
    __shared__ int32_t hist[SMALL_NW * SMALL_BINS], sh[NW + 1], err, perm;
    int32_t *const start = reinterpret_cast<int32_t *>(word);
    const int64_t first = n_units > 0 ? ipu[0] : 0, last = n_units > 0 ? ipu[n_units] : 0;
    const bool covers = n_units > 0 ? first == 0 && last == n_edges : n_edges == 0;
    if (tid == 0) {
        err = first < 0 || last >= INT32_MAX ? 3 : last > n_edges ? 1 : 0;
        perm = 1;
    }
    for (int r = tid; r <= n_rows; r += SMALL_TPB) start[r] = r < n_rows ? INT32_MAX : (int32_t)last;
    __syncthreads();
    // edge slots: indices to 32 bits, eid a permutation? (the check below); units: sorted? where the rows start
#pragma unroll 4
    for (int p = tid; p < n_edges; p += SMALL_TPB) {
        const int64_t e = eid[p], c = indices ? indices[p] : 0;
        const bool ok = e >= 0 && e < n_edges && c >= 0 && (!indices || c < S.n_index_nodes);
        if (!ok) atomicMax(&err, 1);
        S.eid32[p] = ok ? (int32_t)e : 0;
        S.idx32[p] = ok ? (int32_t)c : 0;
        nbr[p] = ok ? (uint16_t)c : (uint16_t)0;
        if (ok) S.seen[e] = p;
    }
    for (int u = tid; u < n_units; u += SMALL_TPB) {
        const int64_t r = row[u], before = u > 0 ? row[u - 1] : -1, at = ipu[u];
        int bad = r < 0 || r >= n_rows ? 1 : 0;
        if (r < before || ipu[u + 1] < at) bad = 2;
        if (bad) atomicMax(&err, bad);
        else if (r > before) start[r] = (int32_t)at;
    }
    __syncthreads();
    int32_t n_items = 0, n_heavy = 0, n_slots = 0, degree = 0;
    if (err == 0) {
        fill_starts(start, n_rows, sh);
        for (int r = tid; r <= n_rows; r += SMALL_TPB) S.rowptr[r] = start[r];
        // items of every row in row order, the heavy rows: a run of rows a thread
        int4 *const items = indices ? S.items_tmp : S.items;
        const int per = (n_rows + SMALL_TPB - 1) / SMALL_TPB, r0 = min(tid * per, n_rows), r1 = min(r0 + per, n_rows);
        auto segments = [&](int deg) { return deg > seg_len ? (deg - 1) / seg_len + 1 : 0; };
        int32_t mine = 0, heavy = 0, slots = 0;
        for (int r = r0; r < r1; ++r) {
            const int deg = start[r + 1] - start[r], n = segments(deg);
            mine += max(n, 1);
            heavy += n > 0 ? 1 : 0;
            slots += n;
            degree = max(degree, deg);
        }
        int32_t item = block_excl_sum<NW>(mine, sh, n_items), hv = block_excl_sum<NW>(heavy, sh, n_heavy), slot = block_excl_sum<NW>(slots, sh, n_slots);
        for (int d = 32; d > 0; d >>= 1) degree = max(degree, __shfl_xor(degree, d));
        __syncthreads();
        if ((tid & 63) == 0) sh[tid >> 6] = degree;
        __syncthreads();
        for (int w = 0; w < NW; ++w) degree = max(degree, sh[w]);
        for (int i = 0; i < per; ++i) {
            const int r = r0 + i, begin = r < r1 ? start[r] : 0, end = r < r1 ? start[r + 1] : 0, n = segments(end - begin);
            if (n == 0) {
                if (r < r1) items[item++] = make_int4(r, begin, end, -1);
            } else {
                S.heavy[3 * hv] = r;
                S.heavy[3 * hv + 1] = slot;
                S.heavy[3 * hv + 2] = n;
                ++hv;
            }
            const int32_t own[5] = {r, begin, end, item, slot};
            for_each_of_lane(n, own, [&](const int32_t (&o)[5], int t) {
                items[o[3] + t] = make_int4(o[0], o[1] + t * seg_len, min(o[2], o[1] + (t + 1) * seg_len), o[4] + t);
            });
            item += n;
            slot += n;
        }
        for (int p = tid; p < n_edges; p += SMALL_TPB)
            if (S.seen[S.eid32[p]] != p) perm = 0;
        __syncthreads();                                          // (the items are written, the rows' starts read)
        // smallest and largest neighbour of every item, four lanes an item; an empty item: its own row id clipped to n_index_nodes
        int2 *const bounds = indices ? S.bounds_tmp : S.bounds;
        if (bounds)
            for (int i = tid >> 2; i < n_items; i += SMALL_TPB / 4) {
                int32_t lo = INT32_MAX, hi = 0;
                const int4 it = items[i];
                if (it.z > it.y) {
                    for (int p = it.y + (tid & 3); p < it.z; p += 4) {
                        lo = min(lo, (int32_t)nbr[p]);
                        hi = max(hi, (int32_t)nbr[p]);
                    }
                    lo = min(lo, __shfl_xor(lo, 1, 4));
                    hi = max(hi, __shfl_xor(hi, 1, 4));
                    lo = min(lo, __shfl_xor(lo, 2, 4));
                    hi = max(hi, __shfl_xor(hi, 2, 4));
                } else {
                    lo = hi = (int32_t)min((int64_t)it.x, S.n_index_nodes);
                }
                if ((tid & 3) == 0) {
                    bounds[i] = make_int2(lo, hi);
                    word[i] = ((uint32_t)lo << SMALL_ITEM_BITS) | (uint32_t)i;
                }
            }
        if (indices) {
            __syncthreads();
            order_items<SMALL_ITEM_BITS, SMALL_ITEMS / SMALL_TPB>(S, n_items, word, hist, sh);
        } else if (S.jorder && S.bounds) {                        // (no edges, and groups are asked for: the items as they are)
            __syncthreads();
            order_by_largest<SMALL_ITEM_BITS, SMALL_ITEMS / SMALL_TPB>(S, n_items, word, hist, sh);
        }
    }
    if (tid < 16) {
        const int32_t v = tid == BPT_PI_ERR ? err : tid == BPT_PI_N_ITEMS ? n_items : tid == BPT_PI_N_HEAVY ? n_heavy : tid == BPT_PI_N_SLOTS ? n_slots
                          : tid == BPT_PI_MAX_DEGREE ? degree : tid == BPT_PI_FLAGS ? (covers && perm ? 1 : 0) : 0;
        S.info[tid] = v;
        if (info_out) info_out[16 * blockIdx.x + tid] = v;
    }
}

// info blocks to memory that the host reads
__global__ void k_info_out(PlanSides b, int32_t *info_out) { info_out[16 * blockIdx.x + threadIdx.x] = b.side[blockIdx.x].info[threadIdx.x]; }

// Sort key of every item: smallest (LARGEST = false) or largest neighbour id; an empty item takes its own row id,
// clipped to n_index_nodes.  Positions past n_items get the padding key, which sorts behind every real one.
template <bool LARGEST>
__global__ void k_item_keys(const int32_t *items, const int32_t *idx32, const int32_t *info, int64_t max_items,
                            int64_t n_index_nodes, int64_t n_edges, uint32_t *key) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= max_items) return;
    if (info[BPT_PI_ERR] || i >= info[BPT_PI_N_ITEMS]) {
        key[i] = PAD32;
        return;
    }
    const int4 it = reinterpret_cast<const int4 *>(items)[i];
    int32_t k = (it.x >= 0 && it.x < n_index_nodes) ? it.x : (int32_t)n_index_nodes;
    if (it.z > it.y && it.y >= 0 && it.z <= n_edges) {          // (an item list from elsewhere is not trusted with addresses)
        k = idx32[it.y];
        for (int32_t p = it.y + 1; p < it.z; ++p) k = LARGEST ? max(k, idx32[p]) : min(k, idx32[p]);
    }
    key[i] = (uint32_t)k;
}

// ---- row groups --------------------------------------------------------------------------------------------------------
struct GroupWs {
    uint32_t *key, *key_s;            // item keys, then group keys
    int32_t *iota, *jorder;           // items in the order of their largest neighbour
    int32_t *work0;                   // per group as formed
    int32_t *lorder, *lpos;           // locality numbering of the groups (by smallest neighbour) and its inverse
    int32_t *work, *prefix;           // per group in locality numbering, max_groups + 1
    int32_t *gorder, *inv;            // final group order (positions in locality numbering) and its inverse
    uint64_t *ekey, *ekey_s;          // one record per edge slot: (group, neighbour, member), unsorted and sorted
    uint64_t *mkey_s;                 // sorted (group, mask) keys of the entries (ekey is reused for the unsorted ones)
    int32_t *eval, *eval_s;           // the slot of a record; later the entry permutation
    int32_t *rank, *head, *run, *mult, *ebase, *ent_of;   // per record
    int32_t *ent_idx, *ent_g, *ent_mask, *newpos, *pop, *first;   // per entry
    void *tmp;
};

GroupWs group_layout(Bump &b, int64_t max_items, int64_t max_groups, int64_t n_edges, size_t tmp_bytes) {
    GroupWs w;
    const int64_t nk = max_items > max_groups ? max_items : max_groups;
    w.key = b.take<uint32_t>(nk);
    w.key_s = b.take<uint32_t>(nk);
    w.iota = b.take<int32_t>(nk > n_edges ? nk : n_edges);
    w.jorder = b.take<int32_t>(max_items);
    w.work0 = b.take<int32_t>(max_groups + 1);
    w.lorder = b.take<int32_t>(max_groups);
    w.lpos = b.take<int32_t>(max_groups);
    w.work = b.take<int32_t>(max_groups + 1);
    w.prefix = b.take<int32_t>(max_groups + 1);
    w.gorder = b.take<int32_t>(max_groups);
    w.inv = b.take<int32_t>(max_groups);
    w.ekey = b.take<uint64_t>(n_edges);
    w.ekey_s = b.take<uint64_t>(n_edges);
    w.mkey_s = b.take<uint64_t>(n_edges);
    w.eval = b.take<int32_t>(n_edges);
    w.eval_s = b.take<int32_t>(n_edges);
    w.rank = b.take<int32_t>(n_edges);
    w.head = b.take<int32_t>(n_edges + 1);
    w.run = b.take<int32_t>(n_edges + 1);
    w.mult = b.take<int32_t>(n_edges + 1);
    w.ebase = b.take<int32_t>(n_edges + 1);
    w.ent_of = b.take<int32_t>(n_edges);
    w.ent_idx = b.take<int32_t>(n_edges);
    w.ent_g = b.take<int32_t>(n_edges);
    w.ent_mask = b.take<int32_t>(n_edges);
    w.newpos = b.take<int32_t>(n_edges);
    w.pop = b.take<int32_t>(n_edges + 1);
    w.first = b.take<int32_t>(n_edges + 1);
    w.tmp = b.take<char>((int64_t)tmp_bytes);
    return w;
}

__device__ inline bool plan_usable(const int32_t *pinfo) { return pinfo[BPT_PI_ERR] == 0 && (pinfo[BPT_PI_FLAGS] & 1); }

__device__ inline int32_t n_groups_of(const int32_t *pinfo, int32_t R) {
    return plan_usable(pinfo) ? (pinfo[BPT_PI_N_ITEMS] + R - 1) / R : 0;
}

// work of every group as formed (its pairs plus a fixed cost) and its locality key: the smallest neighbour id any
// member reads
__global__ void k_group_work(const int32_t *items, const int32_t *jorder, const uint32_t *kmin, const int32_t *pinfo,
                             int64_t max_groups, int32_t R, int32_t *work0, uint32_t *lkey, int32_t *ginfo) {
    const int64_t g = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (g > max_groups) return;
    const int32_t ng = n_groups_of(pinfo, R), n_items = pinfo[BPT_PI_N_ITEMS];
    if (g == 0) {
        for (int i = 0; i < 16; ++i) ginfo[i] = 0;
        ginfo[BPT_GI_N_GROUPS] = ng;
    }
    int32_t w = 0;
    uint32_t key = PAD32;
    if (g < ng) {
        w = FIXED_WORK;
        for (int32_t m = 0; m < R; ++m) {
            const int64_t j = g * R + m;
            if (j < n_items) {
                const int32_t item = jorder[j];
                const int4 it = reinterpret_cast<const int4 *>(items)[item];
                w += it.z - it.y;
                key = min(key, kmin[item]);
            }
        }
    }
    work0[g] = w;
    if (g < max_groups) lkey[g] = key;
}

__global__ void k_gather_work(const int32_t *work0, const int32_t *lorder, const int32_t *ginfo, int64_t max_groups, int32_t *work) {
    const int64_t l = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (l > max_groups) return;
    work[l] = (l < ginfo[BPT_GI_N_GROUPS]) ? work0[lorder[l]] : 0;
}

// 8 contiguous ranges of about equal work: chunks[x] = number of groups whose midpoint lies before x/8 of the total
__global__ void k_chunks(const int32_t *work, const int32_t *prefix, const int32_t *pinfo, int32_t R, int32_t *chunks,
                         int32_t *ginfo) {
    __shared__ int32_t sh[9];
    const int x = threadIdx.x;
    const int32_t ng = n_groups_of(pinfo, R);
    if (x <= 8) {
        int32_t c = (x == 8) ? ng : 0;
        if (x >= 1 && x <= 7 && ng > 0) {
            const int64_t total = (int64_t)prefix[ng - 1] + work[ng - 1];
            const int64_t target = total * x / 8;
            int32_t lo = 0, hi = ng;                      // first group with prefix + work / 2 >= target
            while (lo < hi) {
                const int32_t mid = (lo + hi) >> 1;
                if ((int64_t)prefix[mid] + work[mid] / 2 < target) lo = mid + 1; else hi = mid;
            }
            c = lo;
        }
        sh[x] = c;
        chunks[x] = c;
    }
    __syncthreads();
    if (x == 0) {
        int32_t mx = 0;
        for (int i = 0; i < 8; ++i) mx = max(mx, sh[i + 1] - sh[i]);
        ginfo[BPT_GI_MAX_CHUNK] = mx;
    }
}

__global__ void k_group_keys(const int32_t *work, const int32_t *chunks, const int32_t *pinfo, int64_t max_groups, int32_t R,
                             int by_work, uint32_t *key) {
    const int64_t g = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (g >= max_groups) return;
    if (g >= n_groups_of(pinfo, R)) {
        key[g] = PAD32;
        return;
    }
    uint32_t c = 0;
    for (int x = 1; x <= 7; ++x) c += (chunks[x] <= g) ? 1u : 0u;
    key[g] = (c << 16) | (by_work ? 0xFFFFu - (uint32_t)work[g] : 0u);      // (the sort is stable: locality order otherwise)
}

__global__ void k_invert(const int32_t *order, const int32_t *count, int idx_of_count, int64_t max_n, int32_t *inv) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= max_n || i >= count[idx_of_count]) return;
    inv[order[i]] = (int32_t)i;
}

// members of the groups in their final order (members given), and one sort record per edge slot (ekey given).  inv == nullptr:
// the records carry the locality number of their group (the tile plans number their groups only once the entries are known).
__global__ void k_members_and_records(const int32_t *items, const int32_t *idx32, const int32_t *jorder, const int32_t *lpos,
                                      const int32_t *inv, const int32_t *pinfo, int64_t max_groups, int64_t n_edges, int32_t R,
                                      int32_t *members, uint64_t *ekey, int32_t *eval) {
    const int64_t j = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (j >= max_groups * R) return;
    const int32_t ng = n_groups_of(pinfo, R), n_items = pinfo[BPT_PI_N_ITEMS];
    const int64_t g0 = j / R;
    const int32_t m = (int32_t)(j % R);
    if (g0 >= ng) return;
    const int32_t gi = inv ? inv[lpos[g0]] : lpos[g0];
    if (j >= n_items) {
        if (members) {
            members[((int64_t)gi * R + m) * 2] = -1;
            members[((int64_t)gi * R + m) * 2 + 1] = -1;
        }
        return;
    }
    const int4 it = reinterpret_cast<const int4 *>(items)[jorder[j]];
    if (members) {
        members[((int64_t)gi * R + m) * 2] = it.x;
        members[((int64_t)gi * R + m) * 2 + 1] = it.w;
    }
    if (!ekey) return;
    const int32_t p_end = it.z < n_edges ? it.z : (int32_t)n_edges;
    for (int32_t p = it.y > 0 ? it.y : 0; p < p_end; ++p) {
        ekey[p] = ((uint64_t)(uint32_t)gi << 35) | ((uint64_t)(uint32_t)idx32[p] << 4) | (uint64_t)m;
        eval[p] = p;
    }
}

// Tile plans: what a group costs the matrix kernels is its number of blocks of R entries (a block costs the same whether a
// third or all of its pairs exist), known once the entries are: work[l] = 4 * (blocks + 1) for the group with locality
// number l, from the entries' group numbers (ascending, ent_g[u] = l).
__global__ void k_block_work(const int32_t *ent_g, const int32_t *ginfo, int64_t max_groups, int32_t R, int32_t *work) {
    const int64_t l = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (l > max_groups) return;
    const int32_t ng = ginfo[BPT_GI_N_GROUPS], ne = ginfo[BPT_GI_N_ENTRIES];
    if (l >= ng) {
        work[l] = 0;
        return;
    }
    int32_t bound[2];
    for (int t = 0; t < 2; ++t) {                         // first entry whose group is >= l + t
        int32_t lo = 0, hi = ne;
        while (lo < hi) {
            const int32_t mid = (lo + hi) >> 1;
            if (ent_g[mid] < (int32_t)l + t) lo = mid + 1; else hi = mid;
        }
        bound[t] = lo;
    }
    work[l] = 4 * ((bound[1] - bound[0] + R - 1) / R + 1);
}

// the entries' groups from locality numbers to final numbers
__global__ void k_renumber(int32_t *ent_g, const int32_t *inv, int64_t n_edges, const int32_t *ginfo) {
    const int64_t u = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (u >= n_edges || u >= ginfo[BPT_GI_N_ENTRIES]) return;
    ent_g[u] = inv[ent_g[u]];
}

__global__ void k_pad_records(uint64_t *ekey, int32_t *eval, int64_t n_edges, const int32_t *pinfo) {
    const int64_t p = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (p >= n_edges) return;
    if (!plan_usable(pinfo)) {
        ekey[p] = PAD64;
        eval[p] = (int32_t)p;
    }
}

// rank of a record among the equal ones before it (an edge that a member holds several times), and the starts of the
// runs of equal (group, neighbour)
__global__ void k_rank(const uint64_t *skey, int64_t n_edges, const int32_t *pinfo, int32_t *rank, int32_t *head) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i > n_edges) return;
    if (i == n_edges || !plan_usable(pinfo)) {
        head[i] = 0;
        if (i < n_edges) rank[i] = 0;
        return;
    }
    const uint64_t k = skey[i];
    int32_t t = 0;
    for (int64_t b = i - 1; b >= 0 && skey[b] == k; --b) ++t;
    rank[i] = t;
    head[i] = (i == 0 || (skey[i - 1] >> 4) != (k >> 4)) ? 1 : 0;
}

__global__ void k_multiplicity(const int32_t *rank, const int32_t *head, const int32_t *run_excl, int64_t n_edges,
                               const int32_t *pinfo, int32_t *run, int32_t *mult) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n_edges || !plan_usable(pinfo)) return;
    const int32_t r = run_excl[i] + head[i] - 1;
    run[i] = r;
    atomicMax(&mult[r], rank[i] + 1);
}

__global__ void k_entry_fill(const uint64_t *skey, const int32_t *rank, const int32_t *run, const int32_t *ebase,
                             int64_t n_edges, const int32_t *pinfo, int32_t *ent_of, int32_t *ent_idx, int32_t *ent_g,
                             int32_t *ent_mask, int32_t *ginfo) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n_edges || !plan_usable(pinfo)) return;
    if (i == 0) ginfo[BPT_GI_N_ENTRIES] = ebase[n_edges];
    const uint64_t k = skey[i];
    const int32_t u = ebase[run[i]] + rank[i];
    ent_of[i] = u;
    ent_idx[u] = (int32_t)((k >> 4) & 0x7FFFFFFFu);
    ent_g[u] = (int32_t)(k >> 35);
    atomicOr(&ent_mask[u], 1 << (int)(k & 15));
}

// sort keys of the entries inside their groups.  mode 1: by member mask, larger first; mode 2: by (neighbour mod 16,
// neighbour), which spreads a group's walk over the id range the same way in every group, so that groups running
// side by side ask for a shared row at about the same step
__global__ void k_entry_keys(const int32_t *ent_g, const int32_t *ent_mask, const int32_t *ent_idx, int64_t n_edges,
                             const int32_t *ginfo, int mode, uint64_t *ekey) {
    const int64_t u = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (u >= n_edges) return;
    uint64_t k = PAD64;
    if (u < ginfo[BPT_GI_N_ENTRIES]) {
        const uint64_t g = (uint64_t)(uint32_t)ent_g[u], x = (uint64_t)(uint32_t)ent_idx[u];
        k = (mode == 1) ? ((g << 16) | (uint64_t)(0xFFFF ^ ent_mask[u])) : (mode == 2) ? ((g << 35) | ((x & 15) << 31) | x) : ((g << 31) | x);
    }
    ekey[u] = k;
}

__global__ void k_popcounts(const int32_t *ent_mask, const int32_t *perm, int64_t n_edges, const int32_t *ginfo, int32_t *pop) {
    const int64_t u = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (u > n_edges) return;
    pop[u] = (u < ginfo[BPT_GI_N_ENTRIES]) ? __popc((uint32_t)ent_mask[perm[u]]) : 0;
}

__global__ void k_entries_out(const int32_t *ent_idx, const int32_t *ent_mask, const int32_t *perm, const int32_t *first,
                              int64_t n_edges, const int32_t *ginfo, int32_t *entries) {
    const int64_t u = (int64_t)blockIdx.x * TPB + threadIdx.x;
    const int32_t ne = ginfo[BPT_GI_N_ENTRIES];
    if (u > n_edges || u > ne) return;
    int4 e = make_int4(0, 0, 0, 0);                   // the row behind the last entry is zero
    if (u < ne) e = make_int4(ent_idx[perm[u]], ent_mask[perm[u]], first[u], 0);
    reinterpret_cast<int4 *>(entries)[u] = e;
}

__global__ void k_group_ptr(const int32_t *ent_g, const int32_t *perm, int64_t max_groups, const int32_t *ginfo, int32_t *grp_ptr) {
    const int64_t g = (int64_t)blockIdx.x * TPB + threadIdx.x;
    const int32_t ng = ginfo[BPT_GI_N_GROUPS], ne = ginfo[BPT_GI_N_ENTRIES];
    if (g > max_groups || g > ng) return;
    int32_t lo = 0, hi = ne;                          // first entry whose group is >= g
    while (lo < hi) {
        const int32_t mid = (lo + hi) >> 1;
        if (ent_g[perm[mid]] < g) lo = mid + 1; else hi = mid;
    }
    grp_ptr[g] = lo;
}

__global__ void k_edge_ids(const uint64_t *skey, const int32_t *slot_of, const int32_t *ent_of, const int32_t *newpos,
                           const int32_t *ent_mask, const int32_t *first, const int32_t *eid32, int64_t n_edges,
                           const int32_t *pinfo, int32_t R, int32_t *grp_eids, int32_t *pair_eid) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n_edges || !plan_usable(pinfo)) return;
    const int32_t m = (int32_t)(skey[i] & 15), old = ent_of[i], u = newpos[old];
    if (m >= R) return;                                   // (only with an item list that does not cover the edge slots)
    const int32_t e = eid32[slot_of[i]];
    grp_eids[(int64_t)u * R + m] = e;
    pair_eid[first[u] + __popc((uint32_t)ent_mask[old] & ((1u << m) - 1u))] = e;
}

// ---- row groups, short form -------------------------------------------------------------------------------------------
// The same groups as above for groups whose edges fit a workgroup's LDS (at most GRP_MAX_EDGES) and at most GRP_MAX_GROUPS of
// them, which are the plans of graphs up to some 10^5 nodes.  A group's records never meet another group's, so the device-wide
// sorts of all edges (fifty launches a side) become one workgroup per group that sorts its 200-1000 records in LDS and forms
// the entries, their order and the pair numbers there; two small launches then number the groups; after the caller has read the
// two counts and allocated exactly, every group writes its part of the arrays.  33 765 nodes / 576 k edges, base plan and tiles of
// one side, call to call: 868 -> 227 us (65 535 / 3.3 M: 1690 -> 384, 1 023 / 17 k: 504 -> 165, mostly launches and the waits).
constexpr int GRP_MAX_EDGES = 4096;
constexpr int GRP_MAX_GROUPS = 16384;

void short_layout(Bump &b, PlanSide &S) {
    S.placed = b.take<int4>(S.max_groups);
    S.jorder = b.take<int32_t>(S.max_items);
    S.rec = b.take<GroupRec>(S.max_groups);
    S.order = b.take<int32_t>(S.max_groups);
    S.entry0 = b.take<int32_t>(S.max_groups + 1);
    S.pair0 = b.take<int32_t>(S.max_groups + 1);
    S.chunks = b.take<int32_t>(9);
    S.entries = b.take<int4>(S.n_edges);
    S.pairs = b.take<int32_t>(S.n_edges);
}

struct ItemOrder {                    // last pass of the sort by largest neighbour
    PlanSides b;
    __device__ void put(int side, int64_t at, uint32_t, int32_t i) const { b.side[side].jorder[at] = i; }
};

// The members of a group as formed, and where its results are parked: in the edge slots of its items, which no other group has,
// one member's slots after the other's.
struct GroupSlots {
    int32_t begin[16], pre[17];
    // by 16 threads; returns the smallest neighbour of the group
    __device__ int32_t load(const int4 *items, const int2 *bounds, const int32_t *jorder, int32_t g, int32_t R, int32_t n_items, int64_t n_edges,
                            int32_t seg_len, int2 *member) {
        const int t = threadIdx.x;
        int32_t len = 0, at = 0, lo = INT32_MAX;
        const int64_t j = (int64_t)g * R + t;
        int2 who = make_int2(-1, -1);
        if (t < R && j < n_items) {
            const int32_t item = jorder[j];
            const int4 it = items[item];
            who = make_int2(it.x, it.w);
            if (it.y >= 0 && it.z > it.y && it.z <= n_edges) {
                at = it.y;
                len = min(it.z - it.y, seg_len);
            }
            if (bounds) lo = bounds[item].x;
        }
        int32_t incl = len;
        for (int d = 1; d < 16; d <<= 1) {
            const int32_t y = __shfl_up(incl, d, 16);
            if (t >= d) incl += y;
        }
        for (int d = 8; d > 0; d >>= 1) lo = min(lo, __shfl_xor(lo, d, 16));
        begin[t] = at;
        pre[t] = incl - len;
        if (t == 15) pre[16] = incl;
        if (member && t < R) *member = who;
        return lo;
    }
    __device__ int member_of(int x) const {
        int m = 0;
        for (int d = 8; d > 0; d >>= 1)
            if (m + d < 16 && pre[m + d] <= x) m += d;
        return m;
    }
    __device__ int32_t slot(int x) const {
        const int m = member_of(x);
        return begin[m] + (x - pre[m]);
    }
};

// value of lane (lane ^ M): DPP where a pattern of 16 lanes does it, through the LDS crossbar else
template <int M> __device__ __forceinline__ uint32_t lane_xor(uint32_t x) {
    auto dpp = [](uint32_t v, auto ctrl) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xf, 0xf, true); };
    if constexpr (M == 1) return dpp(x, std::integral_constant<int, 0xB1>());                      // quad_perm 1 0 3 2
    else if constexpr (M == 2) return dpp(x, std::integral_constant<int, 0x4E>());                 // quad_perm 2 3 0 1
    else if constexpr (M == 4) return dpp(dpp(x, std::integral_constant<int, 0x141>()), std::integral_constant<int, 0x1B>());   // ^7, ^3
    else if constexpr (M == 8) return dpp(x, std::integral_constant<int, 0x128>());                // row_ror 8
    else return (uint32_t)__shfl_xor((int)x, M);
}
template <int M> __device__ __forceinline__ uint64_t lane_xor(uint64_t x) {
    return (uint64_t)lane_xor<M>((uint32_t)x) | ((uint64_t)lane_xor<M>((uint32_t)(x >> 32)) << 32);
}

// the stages of stride M and below of a bitonic merge over 128 keys held by a wavefront, lane l the keys l and 64 + l
template <int M, typename K> __device__ __forceinline__ void merge_lanes(K &a, K &b, bool up_a, bool up_b, int lane) {
    if constexpr (M > 0) {
        const bool lower = (lane & M) == 0;
        const K ya = lane_xor<M>(a), yb = lane_xor<M>(b);
        a = ((a < ya) == (lower == up_a)) ? a : ya;
        b = ((b < yb) == (lower == up_b)) ? b : yb;
        merge_lanes<(M >> 1), K>(a, b, up_a, up_b, lane);
    }
}

template <int M, typename K> __device__ __forceinline__ void sort_lanes(K &a, K &b, int lane) {        // runs of 2 M
    if constexpr (M > 1) sort_lanes<(M >> 1), K>(a, b, lane);
    const bool up_a = M == 32 ? true : (lane & (2 * M)) == 0, up_b = M == 32 ? false : up_a;
    merge_lanes<M, K>(a, b, up_a, up_b, lane);
}

// Ascending bitonic sort of n keys (a power of two from 128) in LDS by NT threads: 128 keys at a time in a wavefront's registers,
// only the strides above that through LDS.  (All stages through LDS: k_group_form 66 us for 2200 tiles, so 45, and 24 since
// nothing of a group waits for a global counter.)
template <int NT, typename K> __device__ __forceinline__ void lds_sort(K *key, int n) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int c = wave * 128; c < n; c += NT * 2) {
        K a = key[c + lane], b = key[c + 64 + lane];
        sort_lanes<32, K>(a, b, lane);
        const bool up = (c & 128) == 0;
        if ((a > b) == up) { const K t = a; a = b; b = t; }
        merge_lanes<32, K>(a, b, up, up, lane);
        key[c + lane] = a;
        key[c + 64 + lane] = b;
    }
    __syncthreads();
    for (int k = 256; k <= n; k <<= 1) {
        for (int j = k >> 1; j >= 128; j >>= 1) {
            for (int t = threadIdx.x; t < (n >> 1); t += NT) {
                const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), l = i + j;
                const K a = key[i], b = key[l];
                if ((a > b) == ((i & k) == 0)) {
                    key[i] = b;
                    key[l] = a;
                }
            }
            __syncthreads();
        }
        for (int c = wave * 128; c < n; c += NT * 2) {
            K a = key[c + lane], b = key[c + 64 + lane];
            const bool up = (c & k) == 0;
            if ((a > b) == up) { const K t = a; a = b; b = t; }
            merge_lanes<32, K>(a, b, up, up, lane);
            key[c + lane] = a;
            key[c + 64 + lane] = b;
        }
        __syncthreads();
    }
}

inline __device__ int pow2_at_least(int n) {
    int p = 128;
    while (p < n) p <<= 1;
    return p;
}

// One group: its records (neighbour, member, place in the member's item) sorted, an entry per neighbour and repeat, the entries
// in the order asked for, the pairs numbered.  K: 32-bit keys where neighbour, member and place fit.
template <int CAP, typename K>
__global__ __launch_bounds__(TPB) void k_group_form(PlanSides b, int32_t R) {
    const PlanSide &S = b.side[blockIdx.y];
    const int4 *items = S.items;
    const int2 *bounds = S.bounds;
    const int32_t *jorder = S.jorder, *idx32 = S.idx32, *eid32 = S.eid32, *pinfo = S.info;
    const int64_t n_edges = S.n_edges;
    const int32_t seg_len = S.seg_len;
    const int place_bits = S.place_bits, mode = S.mode;
    GroupRec *rec = S.rec;
    int4 *entries = S.entries;
    int32_t *pairs = S.pairs;
    // (16 KB for 1024 edges with 32-bit keys: ten workgroups a CU)
    __shared__ K key[CAP];
    __shared__ uint32_t ekey[CAP], emask2[CAP / 2];                 // emask2: two entries' masks a word
    __shared__ uint16_t erec[CAP], rec_ent[CAP], efirst[CAP];       // erec: a record of the entry
    uint16_t *const rec_rep = reinterpret_cast<uint16_t *>(ekey), *const rec_cnt = rec_rep + CAP;      // (ekey is not in use yet then)
    auto mask_of = [&](int u) { return (emask2[u >> 1] >> (16 * (u & 1))) & 0xFFFFu; };
    __shared__ GroupSlots at;
    __shared__ int32_t sh[TPB / 64 + 1];
    const int32_t g = blockIdx.x, tid = threadIdx.x;
    if (g >= n_groups_of(pinfo, R)) return;
    int32_t smallest = 0;
    if (tid < 16) smallest = at.load(items, bounds, jorder, g, R, pinfo[BPT_PI_N_ITEMS], n_edges, seg_len, nullptr);
    __syncthreads();
    const int n = at.pre[16], P = pow2_at_least(n);
    for (int t = tid; t < P; t += TPB) {
        K k = (K)~(K)0;
        if (t < n) {
            const int m = at.member_of(t), place = t - at.pre[m];
            k = ((K)(uint32_t)idx32[at.begin[m] + place] << (place_bits + 4)) | (K)((m << place_bits) | place);
        }
        key[t] = k;
        if (2 * t < n) emask2[t] = 0;                               // (a full group: CAP / 2 words, all there are)
    }
    __syncthreads();
    lds_sort<TPB, K>(key, P);
    auto same_edge = [&](int a, int b) { return (key[a] >> place_bits) == (key[b] >> place_bits); };
    auto same_row = [&](int a, int b) { return (key[a] >> (place_bits + 4)) == (key[b] >> (place_bits + 4)); };
    int rep_here = 0;
    for (int i = tid; i < n; i += TPB)
        if (i > 0 && same_edge(i, i - 1)) rep_here = 1;
    const bool repeats = __syncthreads_or(rep_here) != 0;        // a member holds an edge more than once (multigraphs)
    if (repeats) {
        for (int i = tid; i < n; i += TPB) {
            int t = 0;
            for (int b = i - 1; b >= 0 && same_edge(b, i); --b) ++t;
            rec_rep[i] = (uint16_t)t;
        }
        __syncthreads();
    }
    // entries: one per record that is the first of its neighbour with its repeat number
    int n_ent = 0;
    for (int i0 = 0; i0 < n; i0 += TPB) {
        const int i = i0 + tid;
        int fresh = 0;
        if (i < n) {
            fresh = 1;
            if (!repeats) {
                if (i > 0 && same_row(i, i - 1)) fresh = 0;
            } else {
                for (int b = i - 1; b >= 0 && same_row(b, i); --b)
                    if (rec_rep[b] >= rec_rep[i]) { fresh = 0; break; }
            }
        }
        int32_t in_round;
        const int cnt = n_ent + block_excl_sum<TPB / 64>(fresh, sh, in_round);
        if (i < n) {
            rec_cnt[i] = (uint16_t)cnt;
            if (!repeats) rec_ent[i] = (uint16_t)(cnt + fresh - 1);
        }
        n_ent += in_round;
    }
    __syncthreads();
    for (int i = tid; i < n; i += TPB) {
        int u;
        if (repeats) {
            int h = i;
            while (h > 0 && same_row(h - 1, i)) --h;
            u = rec_cnt[h] + rec_rep[i];
            rec_ent[i] = (uint16_t)u;
        } else {
            u = rec_ent[i];
        }
        erec[u] = (uint16_t)i;
        atomicOr(&emask2[u >> 1], 1u << (16 * (u & 1) + (int)((key[i] >> place_bits) & 15)));
    }
    __syncthreads();
    // their order inside the group: as they are (ascending neighbour), by member mask, by (neighbour mod 16, neighbour)
    const int PE = pow2_at_least(n_ent);
    auto idx_of = [&](int u) { return (int32_t)(key[erec[u]] >> (place_bits + 4)); };
    for (int u = tid; u < PE; u += TPB)
        ekey[u] = u >= n_ent ? PAD32 : mode == 1 ? ((0xFFFFu ^ mask_of(u)) << 16) | (uint32_t)u : mode == 2 ? ((uint32_t)(idx_of(u) & 15) << 16) | (uint32_t)u
                                                                                                            : (uint32_t)u;
    __syncthreads();
    if (mode != 0) lds_sort<TPB, uint32_t>(ekey, PE);
    int n_pairs = 0;
    for (int p0 = 0; p0 < n_ent; p0 += TPB) {
        const int p = p0 + tid;
        const int u = p < n_ent ? (int)(ekey[p] & 0xFFFFu) : 0;
        int32_t in_round;
        const uint32_t mask = p < n_ent ? mask_of(u) : 0u;
        const int first = n_pairs + block_excl_sum<TPB / 64>(__popc(mask), sh, in_round);
        if (p < n_ent) {
            efirst[u] = (uint16_t)first;
            entries[at.slot(p)] = make_int4(idx_of(u), (int32_t)mask, first, 0);
        }
        n_pairs += in_round;
    }
    __syncthreads();
    for (int i = tid; i < n; i += TPB) {
        const int u = rec_ent[i], m = (int)((key[i] >> place_bits) & 15), place = (int)(key[i] & (K)((1 << place_bits) - 1));
        pairs[at.slot(efirst[u] + __popc(mask_of(u) & ((1u << m) - 1u)))] = eid32[at.begin[m] + place];
    }
    if (tid == 0) rec[g] = GroupRec{n_ent, n, smallest};
}

// Rows that have edges: a row counts at its first unit that is not empty.  Bound by the latency of one launch (a side's units are some
// 100 KB), so every workgroup leaves its own count for the host to add up, and nothing is cleared or added across workgroups.
struct UnitSide {
    const int64_t *row, *indptr;
    int32_t n;
};
struct UnitSides {
    UnitSide side[2];
};
__global__ __launch_bounds__(TPB) void k_count_rows(UnitSides b, int32_t *counts) {
    const UnitSide &S = b.side[blockIdx.y];
    __shared__ int32_t sh[TPB / 64 + 1];
    int32_t mine = 0, all;
    for (int64_t u = blockIdx.x * TPB + threadIdx.x; u < S.n; u += gridDim.x * TPB) {
        if (S.indptr[u + 1] <= S.indptr[u]) continue;
        const int64_t r = S.row[u];
        int64_t v = u;                                            // back over the row's empty units
        while (v > 0 && S.row[v - 1] == r && S.indptr[v] <= S.indptr[v - 1]) --v;
        mine += v == 0 || S.row[v - 1] != r;
    }
    block_excl_sum<TPB / 64>(mine, sh, all);
    if (threadIdx.x == 0) counts[blockIdx.y * BPT_COUNT_PARTS + blockIdx.x] = all;
}

// The groups' numbers: by locality (smallest neighbour, then as formed), cut into 8 ranges of equal work, by decreasing work inside
// a range (or not); with them every group's place in the arrays.  Two launches of comparisons of every group with every other one
// (the second: of its range): what a group is told apart by is a word that no other group has, its place is the number of smaller
// words, and what it starts at is the sum over those.  A workgroup places GRP_PLACE groups, GRP_EACH of them a thread; 64 threads
// share the others out.  Bound up to some 2000 groups by the latency of the launches and of reading the records, above by the
// comparisons.  Groups of both sides, us: 131 12, 1072 13, 2200 16.6, 4352 27, 8768 58, 13477 97 (one workgroup a side that sorted the
// words by radix passes in LDS: 12, 20, 28.6, 32, 67, 101).
constexpr int GRP_PLACE_TPB = 1024;
constexpr int GRP_EACH = 2;
constexpr int GRP_PLACE = 16 * GRP_EACH;      // groups of a workgroup
constexpr int GRP_PLACE_WAVES = GRP_PLACE_TPB / 64;
// A thread meets at most a 64th of the groups, each of which has at most GRP_MAX_EDGES entries and less than twice that as its
// work: number and sum of the smaller ones share a word, one addition for both.
constexpr int GRP_SUM_BITS = 22;
static_assert(GRP_MAX_GROUPS / 64 * (2 * GRP_MAX_EDGES) < 1 << GRP_SUM_BITS && GRP_MAX_GROUPS / 64 < 1 << (32 - GRP_SUM_BITS), "a thread's sums");

struct GroupSums {                    // over the groups with a smaller word; all: of the a of all groups
    int32_t place, a, b, all;
};
// The sums over a workgroup's threads; base: of what is smaller than all of its groups.  Valid in the first GRP_PLACE threads.
template <bool TWO>
__device__ GroupSums add_up(const uint32_t *sum, const uint32_t *b, GroupSums base) {
    __shared__ int32_t part[GRP_PLACE_WAVES][GRP_PLACE][TWO ? 3 : 2], part_base[GRP_PLACE_WAVES][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int m = 1; m < 64; m <<= 1) {
        base.all += __shfl_xor(base.all, m, 64);
        if constexpr (TWO) {
            base.place += __shfl_xor(base.place, m, 64);
            base.a += __shfl_xor(base.a, m, 64);
            base.b += __shfl_xor(base.b, m, 64);
        }
    }
    if (lane == 0) {
        part_base[wave][0] = base.place;
        part_base[wave][1] = base.a;
        part_base[wave][2] = base.b;
        part_base[wave][3] = base.all;
    }
#pragma unroll
    for (int e = 0; e < GRP_EACH; ++e) {
        int32_t place = (int32_t)(sum[e] >> GRP_SUM_BITS), a = (int32_t)(sum[e] & ((1u << GRP_SUM_BITS) - 1u)), b_here = TWO ? (int32_t)b[e] : 0;
        for (int m = 16; m < 64; m <<= 1) {
            place += __shfl_xor(place, m, 64);
            a += __shfl_xor(a, m, 64);
            if constexpr (TWO) b_here += __shfl_xor(b_here, m, 64);
        }
        if (lane < 16) {
            part[wave][16 * e + lane][0] = place;
            part[wave][16 * e + lane][1] = a;
            if constexpr (TWO) part[wave][16 * e + lane][2] = b_here;
        }
    }
    __syncthreads();
    GroupSums r{0, 0, 0, 0};
    if (tid < GRP_PLACE)
        for (int w = 0; w < GRP_PLACE_WAVES; ++w) {
            r.place += part[w][tid][0] + part_base[w][0];
            r.a += part[w][tid][1] + part_base[w][1];
            if constexpr (TWO) r.b += part[w][tid][2] + part_base[w][2];
            r.all += part_base[w][3];
        }
    return r;
}

// locality order: a group's record goes to its place there, with the word that says its final place: (range, decreasing work or
// nothing, place by locality)
__global__ __launch_bounds__(GRP_PLACE_TPB) void k_group_place(PlanSides b, int32_t R) {
    const PlanSide &S = b.side[blockIdx.y];
    const GroupRec *rec = S.rec;
    const int g_bits = S.g_bits, work_bits = S.work_bits, by_work = S.by_work;
    const int ng = n_groups_of(S.info, R), g0 = blockIdx.x * GRP_PLACE, tid = threadIdx.x;
    if (g0 >= ng) return;
    __shared__ uint2 word_work[2 * GRP_PLACE_TPB];                // word; 1 and the work
    auto work_of = [&](const GroupRec &r) { return R == 16 ? 4 * ((r.n_entries + R - 1) / R + 1) : FIXED_WORK + r.n_pairs; };
    auto word_of = [&](const GroupRec &r, int g) { return ((uint32_t)r.key << g_bits) | (uint32_t)g; };
    uint32_t mine[GRP_EACH], sum[GRP_EACH];
#pragma unroll
    for (int e = 0; e < GRP_EACH; ++e) {
        const int g = g0 + 16 * e + (tid & 15);
        mine[e] = g < ng ? word_of(rec[g], g) : 0u;
        sum[e] = 0;
    }
    GroupSums base{0, 0, 0, 0};
    for (int t0 = 0; t0 < ng; t0 += 2 * GRP_PLACE_TPB) {
        const int n = min(2 * GRP_PLACE_TPB, ng - t0);
        __syncthreads();
        for (int t = tid; t < n; t += GRP_PLACE_TPB) {
            const GroupRec r = rec[t0 + t];
            const int32_t work = work_of(r);
            word_work[t] = make_uint2(word_of(r, t0 + t), (1u << GRP_SUM_BITS) + (uint32_t)work);
            base.all += work;
        }
        __syncthreads();
#pragma unroll 8
        for (int t = tid >> 4; t < n; t += GRP_PLACE_TPB / 16) {
            const uint2 x = word_work[t];
#pragma unroll
            for (int e = 0; e < GRP_EACH; ++e) sum[e] += x.x < mine[e] ? x.y : 0u;
        }
    }
    const GroupSums at = add_up<false>(sum, nullptr, base);
    const int g = g0 + tid;
    if (tid >= GRP_PLACE || g >= ng) return;
    // range: how many of the points 1/8 ... 7/8 of the total lie at or before the group's midpoint
    const GroupRec r = rec[g];
    const int32_t work = work_of(r);
    const int64_t mid = (int64_t)at.a + work / 2, total = at.all;
    uint32_t range = 0;
    for (int x = 1; x <= 7; ++x) range += mid >= total * x / 8 ? 1u : 0u;
    const uint32_t down = by_work ? ((1u << work_bits) - 1u) - (uint32_t)work : 0u;
    S.placed[at.place] = make_int4((int)((((range << work_bits) | down) << g_bits) | (uint32_t)at.place), r.n_entries, r.n_pairs, g);
}

// final order, and every group's first entry and pair.  The ranges are runs of the locality order: a workgroup adds up what lies in
// the ranges before its groups' and compares inside theirs.  The last workgroup writes the ranges' bounds and the plan's and the
// groups' info blocks.
__global__ __launch_bounds__(GRP_PLACE_TPB) void k_group_order(PlanSides b, int32_t R) {
    const PlanSide &S = b.side[blockIdx.y];
    const int4 *placed = S.placed;
    const int32_t *pinfo = S.info;
    const int range_at = S.work_bits + S.g_bits;
    const int ng = n_groups_of(pinfo, R), tid = threadIdx.x;
    auto range_of = [&](int l) { return (int)((uint32_t)placed[l].x >> range_at); };
    if (blockIdx.x == gridDim.x - 1) {
        int32_t *chunks = S.chunks, *out_info = S.out_info;
        __shared__ int32_t cut[9], entries[GRP_PLACE_WAVES];
        if (tid < 9) cut[tid] = tid == 0 ? 0 : ng;
        __syncthreads();
        int32_t n_entries = 0;
        for (int l = tid; l < ng; l += GRP_PLACE_TPB) {
            const int from = l > 0 ? range_of(l - 1) : 0, to = range_of(l);
            for (int x = from + 1; x <= to; ++x) cut[x] = l;
            n_entries += placed[l].y;
        }
        for (int m = 1; m < 64; m <<= 1) n_entries += __shfl_xor(n_entries, m, 64);
        if ((tid & 63) == 0) entries[tid >> 6] = n_entries;
        __syncthreads();
        if (tid < 9) chunks[tid] = cut[tid];
        if (tid < 16) out_info[tid] = pinfo[tid];
        if (tid > 0) return;
        for (int w = 1; w < GRP_PLACE_WAVES; ++w) n_entries += entries[w];
        int32_t most = 0;
        for (int x = 0; x < 8; ++x) most = max(most, cut[x + 1] - cut[x]);
        S.entry0[ng] = n_entries;
        for (int i = 0; i < 16; ++i) out_info[16 + i] = i == BPT_GI_N_GROUPS ? ng : i == BPT_GI_N_ENTRIES ? n_entries : i == BPT_GI_MAX_CHUNK ? most : 0;
        return;
    }
    const int l0 = blockIdx.x * GRP_PLACE;
    if (l0 >= ng) return;
    const int first = range_of(l0), last = range_of(min(l0 + GRP_PLACE, ng) - 1);
    __shared__ uint2 word_entries[2 * GRP_PLACE_TPB];             // word; 1 and the entries
    __shared__ uint32_t n_pairs[2 * GRP_PLACE_TPB];
    uint32_t mine[GRP_EACH], sum[GRP_EACH], pairs[GRP_EACH];
#pragma unroll
    for (int e = 0; e < GRP_EACH; ++e) {
        const int l = l0 + 16 * e + (tid & 15);
        mine[e] = l < ng ? (uint32_t)placed[l].x : 0u;
        sum[e] = pairs[e] = 0;
    }
    GroupSums base{0, 0, 0, 0};
    for (int t0 = 0; t0 < ng; t0 += 2 * GRP_PLACE_TPB) {
        int lo = 0, hi = 0;                                       // of these: in the ranges before, in those and the groups' own
        for (int u = 0; u < 2; ++u) {
            const int t = u * GRP_PLACE_TPB + tid;
            bool before = false, own = false;
            if (t0 + t < ng) {
                const int4 x = placed[t0 + t];
                const int range = (int)((uint32_t)x.x >> range_at);
                before = range < first;
                own = range >= first && range <= last;
                if (before) {
                    base.place += 1;
                    base.a += x.y;
                    base.b += x.z;
                }
                if (own) {
                    word_entries[t] = make_uint2((uint32_t)x.x, (1u << GRP_SUM_BITS) + (uint32_t)x.y);
                    n_pairs[t] = (uint32_t)x.z;
                }
            }
            const int n_before = __syncthreads_count(before), n_own = __syncthreads_count(own);
            lo += n_before;
            hi += n_before + n_own;
        }
        for (int t = lo + (tid >> 4); t < hi; t += GRP_PLACE_TPB / 16) {
            const uint2 x = word_entries[t];
            const uint32_t p = n_pairs[t];
#pragma unroll
            for (int e = 0; e < GRP_EACH; ++e) {
                const bool less = x.x < mine[e];
                sum[e] += less ? x.y : 0u;
                pairs[e] += less ? p : 0u;
            }
        }
        __syncthreads();
        if (hi < min(2 * GRP_PLACE_TPB, ng - t0)) break;          // the rest lies in later ranges
    }
    const GroupSums at = add_up<true>(sum, pairs, base);
    if (tid >= GRP_PLACE || l0 + tid >= ng) return;
    S.order[at.place] = placed[l0 + tid].w;
    S.entry0[at.place] = at.a;
    S.pair0[at.place] = at.b;
}

// a group's part of the arrays; the block behind the last group writes what stands behind the last entry
struct GroupsOut {
    int32_t n_groups, n_entries, max_chunk;
    int32_t *members, *grp_ptr, *pair_eid, *grp_eids, *chunks, *ginfo;
    int4 *entries;
    int32_t *number;                  // per edge: its pair's number (or null)
};
struct GroupsOuts {
    GroupsOut side[2];
};

__global__ __launch_bounds__(TPB) void k_group_write(PlanSides b, GroupsOuts outs, int32_t R, int32_t pad_entries) {
    const PlanSide &S = b.side[blockIdx.y];
    const GroupsOut &O = outs.side[blockIdx.y];
    const int4 *items = S.items, *parked = S.entries;
    const int32_t *jorder = S.jorder, *pinfo = S.info, *order = S.order, *entry0 = S.entry0, *pair0 = S.pair0, *chunks = S.chunks,
                  *parked_pairs = S.pairs;
    const GroupRec *rec = S.rec;
    const int64_t n_edges = S.n_edges;
    const int32_t seg_len = S.seg_len, n_groups = O.n_groups, n_entries = O.n_entries, max_chunk = O.max_chunk;
    int32_t *members = O.members, *grp_ptr = O.grp_ptr, *pair_eid = O.pair_eid, *grp_eids = O.grp_eids, *out_chunks = O.chunks, *ginfo = O.ginfo;
    int4 *entries = O.entries;
    const int32_t f = blockIdx.x, tid = threadIdx.x;
    if (f > n_groups) return;                             // (the other side has more)
    if (f == n_groups) {
        if (tid == 0) {
            grp_ptr[n_groups] = n_entries;
            entries[n_entries] = make_int4(0, 0, 0, 0);
        }
        if (tid < 9) out_chunks[tid] = chunks[tid];
        if (tid < 16) ginfo[tid] = tid == BPT_GI_N_GROUPS ? n_groups : tid == BPT_GI_N_ENTRIES ? n_entries : tid == BPT_GI_MAX_CHUNK ? max_chunk : 0;
        for (int i = tid; i < pad_entries * R; i += TPB) grp_eids[(int64_t)n_entries * R + i] = (int32_t)n_edges;
        return;
    }
    __shared__ GroupSlots at;
    const int32_t g = order[f], e0 = entry0[f], p0 = pair0[f];
    const GroupRec r = rec[g];
    if (tid < 16) {
        int2 member;
        at.load(items, nullptr, jorder, g, R, pinfo[BPT_PI_N_ITEMS], n_edges, seg_len, &member);
        if (tid < R) reinterpret_cast<int2 *>(members)[(int64_t)f * R + tid] = member;
    }
    if (tid == 0) grp_ptr[f] = e0;
    __syncthreads();
    if (e0 + r.n_entries > n_entries || r.n_pairs > at.pre[16] || r.n_entries > r.n_pairs) return;    // (counts that are not this workspace's)
    for (int u = tid; u < r.n_entries; u += TPB) {
        int4 e = parked[at.slot(u)];
        e.z += p0;
        entries[e0 + u] = e;
    }
    for (int x = tid; x < r.n_pairs; x += TPB) {
        const int32_t e = parked_pairs[at.slot(x)];
        pair_eid[p0 + x] = e;
        if (O.number) O.number[e] = p0 + x;
    }
    for (int i = tid; i < r.n_entries * R; i += TPB) {
        const int u = i / R, m = i - u * R;
        const int4 e = parked[at.slot(u)];
        const uint32_t mask = (uint32_t)e.y;
        grp_eids[(int64_t)e0 * R + i] = (mask >> m) & 1u ? parked_pairs[at.slot(e.z + __popc(mask & ((1u << m) - 1u)))] : (int32_t)n_edges;
    }
}

// ---- pair numbers of the other side ---------------------------------------------------------------------------------------
__global__ void k_number_pairs(const int32_t *pair_eid, int64_t n_edges, int32_t *number) {
    const int64_t x = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (x >= n_edges) return;
    const int32_t e = pair_eid[x];
    if (e >= 0 && e < n_edges) number[e] = (int32_t)x;
}

__global__ void k_find_numbers(const int32_t *eids, int64_t n_slots, int64_t n_edges, const int32_t *number, int32_t *pairs) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n_slots) return;
    const int32_t e = eids[i];
    pairs[i] = e >= 0 && e < n_edges ? number[e] : 0;
}

// ---- link -----------------------------------------------------------------------------------------------------------------
__global__ void k_positions(const int32_t *eids_src, const int32_t *ginfo_src, int32_t R_src, int64_t n_edges, int32_t *pos) {
    const int64_t j = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (j >= (int64_t)ginfo_src[BPT_GI_N_ENTRIES] * R_src) return;
    const int32_t e = eids_src[j];
    if (e >= 0 && e < n_edges) pos[e] = (int32_t)j;
}

__global__ void k_pairs(const int32_t *eids_dst, const int32_t *ginfo_dst, int32_t R_dst, const int32_t *ginfo_src,
                        int32_t R_src, int64_t n_edges, int32_t pad, const int32_t *pos, int32_t *pairs) {
    const int64_t j = (int64_t)blockIdx.x * TPB + threadIdx.x;
    const int64_t n_real = (int64_t)ginfo_dst[BPT_GI_N_ENTRIES] * R_dst;
    if (j >= n_real + (int64_t)pad * R_dst) return;
    const int32_t spare = (ginfo_src[BPT_GI_N_ENTRIES] + pad) * R_src - 1;
    int32_t out = spare;
    if (j < n_real) {
        const int32_t e = eids_dst[j];
        if (e >= 0 && e < n_edges) out = pos[e];
    }
    pairs[j] = out;
}

// ---- edge lists of the reference's graph builder --------------------------------------------------------------------
// builder.pyx:41-116 (binary partition), :243-274 (fully connected), :171-199 (strided sparse) emit the edges token by
// token, so one thread walks one token: a first pass counts its edges, a prefix sum gives every token its place in
// the list, a second pass writes them there — the same list, in the same order, as the host walk (bptgraph.cpp).
constexpr int MAX_LEVELS = 48;
struct LevelTable {
    int64_t size[MAX_LEVELS], offset[MAX_LEVELS];
    int n;
};

struct EdgeCount {
    int64_t n = 0;
    __device__ void operator()(int64_t, int64_t, int64_t) { ++n; }
};
struct EdgeWrite {
    int64_t *src, *dst, *etype;
    int64_t shift, at;
    __device__ void operator()(int64_t s, int64_t d, int64_t t) {
        src[at] = s + shift;
        dst[at] = d + shift;
        etype[at] = t;
        ++at;
    }
};

// One token of builder.pyx:64-116: two cursors walk outwards, `step` nodes per side per level, then move one level
// up; a cursor that stops on a node whose sibling was taken continues with that child on the next level (the
// right-hand bound is checked against the current level even then, as the reference does).
template <class Sink>
__device__ void token_binary_partition(const LevelTable &lv, int64_t tok, bool causal, int64_t step, int64_t clip, Sink &out) {
    int64_t left = tok - 1, right = tok + 1, ancestor = tok;
    bool left_child = false, right_child = false;
    for (int j = 0; j < lv.n; ++j) {
        const int64_t type0 = (2 * step + 1) * (j < clip ? j : clip);
        for (int64_t s = 0; s < step; ++s) {
            if (!causal && right < lv.size[j]) {
                out(right_child ? lv.offset[j - 1] + 2 * right + 1 : lv.offset[j] + right, tok, type0 + 2 * (s + 1));
                right_child = false;
            }
            ++right;
            if (left >= 0) {
                out(left_child ? lv.offset[j - 1] + 2 * left : lv.offset[j] + left, tok, type0 + 2 * s + 1);
                left_child = false;
            }
            --left;
        }
        if ((left & 1) == 0) left_child = true;
        if ((right & 1) == 1) right_child = true;
        right >>= 1;
        left >>= 1;                           // arithmetic shift: stays negative once it is
        out(tok, lv.offset[j] + ancestor, type0);
        ancestor >>= 1;
    }
}

template <class Sink>
__device__ void token_edges(int kind, const LevelTable &lv, int64_t length, int64_t i, bool causal, int64_t a, int64_t b, Sink &out) {
    if (kind == 0) {
        token_binary_partition(lv, i, causal, a, b, out);
    } else if (kind == 1) {                   // builder.pyx:243-274: a = window
        const int64_t reach = length < a + 1 ? length : a + 1;
        out(i, i, 0);
        for (int64_t j = 1; j < reach; ++j) {
            if (i >= j) out(i - j, i, 2 * j - 1);
            if (!causal && i + j < length) out(i + j, i, 2 * j);
        }
        out(i, length, 0);
    } else {                                  // builder.pyx:171-199: a = stride, b = c
        for (int64_t j = (i / a) * a; j <= i; ++j) out(j, i, 0);
        for (int64_t blk = 1; blk <= i / a; ++blk)
            for (int64_t k = a * blk - b; k < a * blk; ++k) out(k, i, 0);
        out(i, length, 0);
    }
}

__global__ void k_graph_count(int kind, LevelTable lv, int64_t length, int causal, int64_t a, int64_t b, int32_t *counts) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i > length) return;
    EdgeCount c;
    if (i < length) token_edges(kind, lv, length, i, causal != 0, a, b, c);
    counts[i] = (int32_t)c.n;
}

__global__ void k_graph_fill(int kind, LevelTable lv, int64_t length, int causal, int64_t a, int64_t b, int64_t shift,
                             const int32_t *offsets, int64_t n_edges, int64_t *src, int64_t *dst, int64_t *etype) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= length || offsets[length] != n_edges) return;     // the caller's edge count must be the list's
    EdgeWrite w{src, dst, etype, shift, offsets[i]};
    token_edges(kind, lv, length, i, causal != 0, a, b, w);
}

bool level_table(int kind, int64_t length, LevelTable &lv) {
    lv.n = 0;
    if (kind != 0) return true;
    int64_t n = length, nodes = 0;
    while (n >= 2) {
        if (lv.n >= MAX_LEVELS - 1) return false;
        lv.size[lv.n] = n;
        lv.offset[lv.n++] = nodes;
        nodes += n;
        n = (n + 1) >> 1;
    }
    lv.size[lv.n] = 1;
    lv.offset[lv.n++] = nodes;
    return true;
}

bool graph_args_ok(int kind, int64_t length, int64_t a, int64_t b) {
    if (length < 1 || length >= INT32_MAX) return false;
    if (kind == 0) return a >= 1 && b >= 0;
    if (kind == 1) return a >= 0;
    if (kind == 2) return a >= 1 && b >= 0 && b <= a;
    return false;
}

// ---- batch of graphs --------------------------------------------------------------------------------------------------------
// Block-diagonal merge of up to MERGE_PARTS graphs a launch, described in the kernel's arguments: their edge lists one after
// the other, the node ids shifted.  Bound by its 48 bytes per edge (576 k edges of 32 graphs: 125 -> 33 us call to call
// against concatenations and a repeated shift; one graph of 3.3 M edges 1390 -> 29, where repeating one number that often took
// most of it).
constexpr int MERGE_PARTS = 64, MERGE_PER = 4;            // elements per thread
struct MergePart {
    const int64_t *src, *dst, *etype, *pos;
    int64_t edge0, node0;                                 // where its edges and nodes start in the batch
};
struct MergeParts {
    MergePart part[MERGE_PARTS];
    int64_t edge_end, node_end;
    int n;
};

__global__ __launch_bounds__(TPB) void k_merge(MergeParts m, unsigned edge_blocks, int64_t *src, int64_t *dst, int64_t *etype, int64_t *pos) {
    const bool edges = blockIdx.x < edge_blocks;
    const int64_t begin = edges ? m.part[0].edge0 : m.part[0].node0, end = edges ? m.edge_end : m.node_end;
    int64_t i = begin + (int64_t)(edges ? blockIdx.x : blockIdx.x - edge_blocks) * (TPB * MERGE_PER);
    int p = 0;
    for (int d = MERGE_PARTS / 2; d > 0; d >>= 1)         // the block's first element: last part that starts at or before it
        if (p + d < m.n && (edges ? m.part[p + d].edge0 : m.part[p + d].node0) <= i) p += d;
    const int64_t next = p + 1 < m.n ? (edges ? m.part[p + 1].edge0 : m.part[p + 1].node0) : end;
    const int64_t stop = min(i + TPB * MERGE_PER, end);
    if (edges && stop <= next) {                          // the whole block in one part: its addresses are the block's
        const MergePart &a = m.part[p];
        const int64_t *s0 = a.src - a.edge0, *d0 = a.dst - a.edge0, *e0 = a.etype - a.edge0;
        int64_t x[MERGE_PER], y[MERGE_PER], z[MERGE_PER];
        i += threadIdx.x;
#pragma unroll
        for (int r = 0; r < MERGE_PER; ++r)
            if (i + r * TPB < stop) { x[r] = s0[i + r * TPB]; y[r] = d0[i + r * TPB]; z[r] = e0[i + r * TPB]; }
#pragma unroll
        for (int r = 0; r < MERGE_PER; ++r)
            if (i + r * TPB < stop) { src[i + r * TPB] = x[r] + a.node0; dst[i + r * TPB] = y[r] + a.node0; etype[i + r * TPB] = z[r]; }
        return;
    }
    i += threadIdx.x;
    for (int r = 0; r < MERGE_PER; ++r, i += TPB) {
        if (i >= end) return;
        while (p + 1 < m.n && (edges ? m.part[p + 1].edge0 : m.part[p + 1].node0) <= i) ++p;
        const MergePart &a = m.part[p];
        if (edges) {
            const int64_t e = i - a.edge0;
            src[i] = a.src[e] + a.node0;
            dst[i] = a.dst[e] + a.node0;
            etype[i] = a.etype[e];
        } else {
            pos[i] = a.pos[i - a.node0];
        }
    }
}

// ---- CSR of an edge list ------------------------------------------------------------------------------------------------
// Both sides of a graph (or one of them) in the same launches, blockIdx.y = side.  Edges sorted by row with their ids as
// they come, so ascending edge id inside a row; the last pass writes the 64-bit eid and indices itself.
struct CsrSide {
    const int64_t *rows, *cols;
    int64_t *indptr, *indices, *eid, *unit_row, *unit_ptr;
    int32_t *info;
    uint32_t *key_s;                  // rows of the slots, sorted
    int32_t *lo_of, *unit_total;      // first slot of every row; units of every block of CSR_ROWS rows
    int32_t *bad;                     // per tile of edges: an id out of range
};
struct CsrSides {
    CsrSide side[2];
};

struct CsrEdges {                     // records of the first pass: the edges themselves; an edge with a bad id sorts behind all rows
    CsrSides g;
    int64_t n_nodes;
    __device__ uint32_t key(int side, int64_t e, bool &bad) const {
        const int64_t r = g.side[side].rows[e], c = g.side[side].cols[e];
        const bool ok = r >= 0 && r < n_nodes && c >= 0 && c < n_nodes;
        bad = bad || !ok;
        return ok ? (uint32_t)r : (uint32_t)n_nodes;
    }
    __device__ int32_t val(int, int64_t e) const { return (int32_t)e; }
    __device__ void report(int side, bool bad) const {
        if (threadIdx.x == 0) g.side[side].bad[blockIdx.x] = bad ? 1 : 0;
    }
};
struct CsrSlots {                     // what the last pass writes
    CsrSides g;
    __device__ void put(int side, int64_t at, uint32_t key, int32_t e) const {
        const CsrSide &c = g.side[side];
        c.key_s[at] = key;
        c.eid[at] = e;
        c.indices[at] = c.cols[e];
    }
};

constexpr int CSR_ROWS = TPB - 1;     // rows of a block of the two kernels below (one thread more: the end of the last row)

// indptr[r] = first slot whose row is >= r; how many chunked units the block's rows give
__global__ __launch_bounds__(TPB) void k_csr_rows(CsrSides g, int64_t n_edges, int64_t n_nodes, int32_t chunk) {
    __shared__ int32_t lo_sh[TPB];
    __shared__ int32_t sh[TPB / 64 + 1];
    const CsrSide &c = g.side[blockIdx.y];
    const int64_t r = (int64_t)blockIdx.x * CSR_ROWS + threadIdx.x;
    int64_t lo = 0, hi = n_edges;
    if (r <= n_nodes) {
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (c.key_s[mid] < (uint32_t)r) lo = mid + 1; else hi = mid;
        }
        c.indptr[r] = lo;
        c.lo_of[r] = (int32_t)lo;
    }
    lo_sh[threadIdx.x] = (int32_t)lo;
    __syncthreads();
    int32_t units = 0, total;
    if (threadIdx.x < CSR_ROWS && r < n_nodes) units = (lo_sh[threadIdx.x + 1] - (int32_t)lo + chunk - 1) / chunk;
    block_excl_sum<TPB / 64>(units, sh, total);
    if (threadIdx.x == 0) c.unit_total[blockIdx.x] = total;
}

// the units of builder.pyx:305-321: each row's slot range in chunks of at most `chunk` slots; empty rows give no unit.  A row
// of more than CSR_FEW units is written by the whole block.
constexpr int CSR_FEW = 8;
__global__ __launch_bounds__(TPB) void k_csr_units(CsrSides g, int64_t n_edges, int64_t n_nodes, int32_t chunk, int64_t n_tiles) {
    __shared__ int32_t sh[TPB / 64 + 1];
    __shared__ int32_t many[TPB][3];
    __shared__ int32_t n_many;
    const CsrSide &c = g.side[blockIdx.y];
    if (threadIdx.x == 0) n_many = 0;
    int32_t part = 0, before, total;
    for (int64_t b = threadIdx.x; b < (int64_t)blockIdx.x; b += TPB) part += c.unit_total[b];
    block_excl_sum<TPB / 64>(part, sh, before);
    const int64_t r = (int64_t)blockIdx.x * CSR_ROWS + threadIdx.x;
    const bool mine = threadIdx.x < CSR_ROWS && r < n_nodes;
    const int32_t lo = mine ? c.lo_of[r] : 0, hi = mine ? c.lo_of[r + 1] : 0, units = (hi - lo + chunk - 1) / chunk;
    const int32_t at = before + block_excl_sum<TPB / 64>(units, sh, total);
    if (units <= CSR_FEW) {
        for (int32_t u = 0; u < units; ++u) {
            c.unit_row[at + u] = r;
            c.unit_ptr[at + u] = lo + (int64_t)u * chunk;
        }
    } else {
        const int i = atomicAdd(&n_many, 1);
        many[i][0] = (int32_t)threadIdx.x;
        many[i][1] = at;
        many[i][2] = lo;
    }
    __syncthreads();
    for (int i = 0; i < n_many; ++i) {
        const int64_t row = (int64_t)blockIdx.x * CSR_ROWS + many[i][0];
        const int32_t first = many[i][1], slot = many[i][2], n = (c.lo_of[row + 1] - slot + chunk - 1) / chunk;
        for (int32_t u = threadIdx.x; u < n; u += TPB) {
            c.unit_row[first + u] = row;
            c.unit_ptr[first + u] = slot + (int64_t)u * chunk;
        }
    }
    if (blockIdx.x == gridDim.x - 1) {
        bool bad = false;
        for (int64_t t = threadIdx.x; t < n_tiles; t += TPB) bad = bad || c.bad[t] != 0;
        const int any = __syncthreads_or(bad ? 1 : 0);
        if (threadIdx.x == 0) {
            c.info[0] = any ? 1 : 0;
            c.info[1] = before + total;
            c.unit_ptr[before + total] = n_edges;
        }
    }
}

// Both sides' CSRs of a small graph, a workgroup a side in one launch: the edges sorted in LDS by (row, edge id), what the eight
// launches for larger graphs leave bit for bit: 15 to 17 us at 5 600 edges, in place of 40.  The limits are what LDS holds.
constexpr int CSR_SMALL_BITS = 14, CSR_SMALL_EDGES = 10240, CSR_SMALL_NODES = 4096;
inline bool csr_small(int64_t n_edges, int64_t n_nodes) { return n_edges <= CSR_SMALL_EDGES && n_nodes <= CSR_SMALL_NODES; }
__global__ __launch_bounds__(SMALL_TPB) void k_csr_small(CsrSides g, int n_edges, int n_nodes, int chunk) {
    constexpr int NW = SMALL_TPB / 64;
    const CsrSide &c = g.side[blockIdx.x];
    __shared__ uint32_t word[CSR_SMALL_EDGES];
    __shared__ int32_t start[CSR_SMALL_NODES + 1], sh[NW + 1];       // (start: before it is one, the sort's counts)
    static_assert(SMALL_NW * SMALL_BINS <= CSR_SMALL_NODES + 1, "the counts fit");
    const int tid = threadIdx.x;
    bool bad = false;
#pragma unroll 4
    for (int e = tid; e < n_edges; e += SMALL_TPB) {
        const int64_t r = c.rows[e], k = c.cols[e];
        const bool ok = r >= 0 && r < n_nodes && k >= 0 && k < n_nodes;
        bad = bad || !ok;
        word[e] = ((uint32_t)(ok ? r : n_nodes) << CSR_SMALL_BITS) | (uint32_t)e;
    }
    const int any_bad = __syncthreads_or(bad ? 1 : 0);
    lds_radix<CSR_SMALL_EDGES / SMALL_TPB>(word, n_edges, CSR_SMALL_BITS, 32 - __clz(n_nodes | 1), start, sh);
    for (int x = tid; x <= n_nodes; x += SMALL_TPB) start[x] = x < n_nodes ? INT32_MAX : n_edges;
    __syncthreads();
    // slots, and where the rows start
    for (int at = tid; at < n_edges; at += SMALL_TPB) {
        const uint32_t w = word[at];
        const int e = (int)(w & ((1 << CSR_SMALL_BITS) - 1)), r = (int)(w >> CSR_SMALL_BITS), before = at > 0 ? (int)(word[at - 1] >> CSR_SMALL_BITS) : -1;
        c.eid[at] = e;
        c.indices[at] = c.cols[e];
        if (r != before) start[r] = at;                           // (row n_nodes: the first bad edge)
    }
    __syncthreads();
    fill_starts(start, n_nodes, sh);
    for (int r = tid; r <= n_nodes; r += SMALL_TPB) c.indptr[r] = start[r];
    // the units of builder.pyx:305-321: a run of rows a thread
    const int per = (n_nodes + SMALL_TPB - 1) / SMALL_TPB, r0 = min(tid * per, n_nodes), r1 = min(r0 + per, n_nodes);
    auto units_of = [&](int r) { return (start[r + 1] - start[r] + chunk - 1) / chunk; };
    int32_t units = 0, total;
    for (int r = r0; r < r1; ++r) units += units_of(r);
    int32_t at = block_excl_sum<NW>(units, sh, total);
    for (int i = 0; i < per; ++i) {
        const int r = r0 + i, n = r < r1 ? units_of(r) : 0;
        const int32_t own[3] = {r, at, r < r1 ? start[r] : 0};
        for_each_of_lane(n, own, [&](const int32_t (&o)[3], int u) {
            c.unit_row[o[1] + u] = o[0];
            c.unit_ptr[o[1] + u] = o[2] + (int64_t)u * chunk;
        });
        at += n;
    }
    if (tid == 0) {
        c.info[0] = any_bad ? 1 : 0;
        c.info[1] = total;
        c.unit_ptr[total] = n_edges;
    }
}

struct CsrWs {
    uint32_t *key[2];
    int32_t *val[2];
    int32_t *counts, *totals;
};

CsrWs csr_layout(Bump &b, int64_t n_edges, int64_t n_nodes, int n_sides, CsrSides &g) {
    CsrWs w;
    const int64_t row_blocks = (n_nodes + CSR_ROWS) / CSR_ROWS;
    for (int i = 0; i < n_sides; ++i) {
        g.side[i].key_s = b.take<uint32_t>(n_edges);
        g.side[i].lo_of = b.take<int32_t>(n_nodes + 2);
        g.side[i].unit_total = b.take<int32_t>(row_blocks);
        g.side[i].bad = b.take<int32_t>(rs_tiles(n_edges));
    }
    w.key[0] = b.take<uint32_t>(n_sides * n_edges);
    w.key[1] = b.take<uint32_t>(n_sides * n_edges);
    w.val[0] = b.take<int32_t>(n_sides * n_edges);
    w.val[1] = b.take<int32_t>(n_sides * n_edges);
    w.counts = b.take<int32_t>(n_sides * rs_tiles(n_edges) * RS_BINS);
    w.totals = b.take<int32_t>(n_sides * RS_BINS);
    return w;
}

int sizes_ok(int64_t n_units, int64_t n_edges, int64_t n_rows, int64_t n_index_nodes, int32_t seg_len) {
    if (n_units < 0 || n_edges < 0 || n_rows < 0 || n_index_nodes < 0) return BPT_ERR_SIZE;
    if (n_rows >= INT32_MAX || n_edges >= INT32_MAX || n_index_nodes >= INT32_MAX || n_units > n_edges + n_rows) return BPT_ERR_SIZE;
    if (seg_len < 1) return BPT_ERR_SHAPE;
    return BPT_OK;
}

#define HIP_TRY(expr)                                   \
    do {                                                \
        const hipError_t e_ = (expr);                   \
        if (e_ != hipSuccess) return (int)e_;           \
    } while (0)

#define LAUNCH(kernel, n, ...)                                                         \
    do {                                                                               \
        if ((n) > 0) {                                                                 \
            hipLaunchKernelGGL(kernel, dim3(blocks_for(n)), dim3(TPB), 0, s, __VA_ARGS__); \
            HIP_TRY(hipGetLastError());                                                \
        }                                                                              \
    } while (0)

// one stable sort pass over one or both sides: counts, prefix, scatter
template <class Recs, class Out>
int rs_pass(const Recs &recs, const Out &out, const RsSizes &sizes, int n_sides, int shift, int bits, int32_t *counts, int32_t *totals, hipStream_t s) {
    const int64_t n = n_sides == 2 && sizes.n[1] > sizes.n[0] ? sizes.n[1] : sizes.n[0];
    const dim3 tiles((unsigned)rs_tiles(n), (unsigned)n_sides);
    const int bins = 1 << bits;
    const bool few = rs_per_thread(n) != 8;
    if (few) hipLaunchKernelGGL((k_rs_count<RS_KPT_FEW, Recs>), tiles, dim3(TPB), 0, s, recs, sizes, shift, bits, counts);
    else hipLaunchKernelGGL((k_rs_count<8, Recs>), tiles, dim3(TPB), 0, s, recs, sizes, shift, bits, counts);
    HIP_TRY(hipGetLastError());
    if (few) {
        hipLaunchKernelGGL((k_rs_scatter<RS_KPT_FEW, true, Recs, Out>), tiles, dim3(TPB), 0, s, recs, out, sizes, shift, bits, counts, totals);
    } else {
        hipLaunchKernelGGL(k_rs_prefix, dim3((unsigned)((bins + RS_PREFIX_BINS - 1) / RS_PREFIX_BINS), (unsigned)n_sides), dim3(RS_PREFIX_TPB), 0,
                           s, counts, totals, (int64_t)tiles.x, bins);
        HIP_TRY(hipGetLastError());
        hipLaunchKernelGGL((k_rs_scatter<8, false, Recs, Out>), tiles, dim3(TPB), 0, s, recs, out, sizes, shift, bits, counts, totals);
    }
    HIP_TRY(hipGetLastError());
    return BPT_OK;
}

// all passes of a sort: recs to begin with, out at the end; two arrays of keys and values (n_sides * largest n) in between
template <class Recs, class Out>
int rs_sort(const Recs &recs, const Out &out, const RsSizes &sizes, int n_sides, uint64_t max_key, uint32_t *const key[2], int32_t *const val[2],
            int32_t *counts, int32_t *totals, hipStream_t s) {
    const int64_t n = n_sides == 2 && sizes.n[1] > sizes.n[0] ? sizes.n[1] : sizes.n[0];
    if (n == 0) return BPT_OK;
    const RsPasses ps = rs_passes(max_key);
    RsToArrays to[2];
    RsArrays from[2];
    for (int t = 0; t < 2; ++t)
        for (int i = 0; i < 2; ++i) {
            to[t].k[i] = key[t] + (i < n_sides ? i : 0) * n;
            to[t].v[i] = val[t] + (i < n_sides ? i : 0) * n;
            from[t].k[i] = to[t].k[i];
            from[t].v[i] = to[t].v[i];
        }
    for (int p = 0; p < ps.n; ++p) {
        const bool first = p == 0, last = p == ps.n - 1;
        const int shift = p * ps.bits;
        int st;
        if (first && last) st = rs_pass(recs, out, sizes, n_sides, shift, ps.bits, counts, totals, s);
        else if (first) st = rs_pass(recs, to[0], sizes, n_sides, shift, ps.bits, counts, totals, s);
        else if (last) st = rs_pass(from[(p - 1) & 1], out, sizes, n_sides, shift, ps.bits, counts, totals, s);
        else st = rs_pass(from[(p - 1) & 1], to[p & 1], sizes, n_sides, shift, ps.bits, counts, totals, s);
        if (st != BPT_OK) return st;
    }
    return BPT_OK;
}

// what the kernels need to know of a side's groups, or BPT_ERR_UNSUPPORTED where they are not built in the short form: a group may
// hold more edges than fit a workgroup's LDS, or there may be more groups than it pays to compare with each other, or numbers that
// don't fit 32-bit words
int short_form(int64_t max_items, int64_t n_edges, int64_t n_index_nodes, int32_t seg_len, int32_t R, int32_t by_mask, PlanSide &S) {
    if (max_items < 0 || n_edges < 0 || n_index_nodes < 0 || max_items >= INT32_MAX || n_edges >= INT32_MAX || n_index_nodes >= INT32_MAX - 1)
        return BPT_ERR_SIZE;
    if (R < 1 || R > 16 || seg_len < 1 || by_mask < 0 || (by_mask & 3) > 2 || by_mask > 6) return BPT_ERR_SHAPE;
    if ((n_edges + 8) * R >= INT32_MAX) return BPT_ERR_SIZE;
    const int64_t max_groups = (max_items + R - 1) / R;
    if ((int64_t)R * seg_len > GRP_MAX_EDGES || max_groups > GRP_MAX_GROUPS) return BPT_ERR_UNSUPPORTED;
    S.max_items = max_items;
    S.n_edges = n_edges;
    S.n_index_nodes = n_index_nodes;
    S.seg_len = seg_len;
    S.mode = by_mask & 3;
    S.by_work = (by_mask & 4) ? 0 : 1;
    S.max_groups = (int32_t)max_groups;
    S.place_bits = (int)bits_for((uint64_t)seg_len - 1);
    S.g_bits = (int)bits_for((uint64_t)(max_groups > 0 ? max_groups - 1 : 0));
    S.key_bits = (int)bits_for((uint64_t)n_index_nodes);
    S.work_bits = (int)bits_for((uint64_t)(R == 16 ? 4 * (seg_len + 1) : FIXED_WORK + R * seg_len));
    return S.key_bits + S.g_bits > 32 || 3 + S.work_bits + S.g_bits > 32 ? BPT_ERR_UNSUPPORTED : BPT_OK;
}

int fill_side(const bpt_build_side &side, PlanSide &S) {
    const int st = sizes_ok(side.n_units, side.n_edges, side.n_rows, side.n_index_nodes, side.seg_len);
    if (st != BPT_OK) return st;
    if (!side.rowptr || !side.items || !side.info) return BPT_ERR_NULL;
    if (side.n_units > 0 && (!side.row || !side.indptr_units)) return BPT_ERR_NULL;
    if (side.n_edges > 0 && (!side.eid || !side.idx32 || !side.eid32)) return BPT_ERR_NULL;
    if (side.n_edges / ((int64_t)side.seg_len + 1) > 0 && !side.heavy) return BPT_ERR_NULL;
    S.max_items = side.n_rows + side.n_edges / side.seg_len;
    if (S.max_items >= INT32_MAX) return BPT_ERR_SIZE;
    S.row = side.row;
    S.ipu = side.indptr_units;
    S.eid = side.eid;
    S.indices = side.indices;
    S.n_units = side.n_units;
    S.n_edges = side.n_edges;
    S.n_rows = side.n_rows;
    S.n_index_nodes = side.n_index_nodes;
    S.seg_len = side.seg_len;
    S.rowptr = side.rowptr;
    S.idx32 = side.idx32;
    S.eid32 = side.eid32;
    S.heavy = side.heavy;
    S.info = side.info;
    S.items = reinterpret_cast<int4 *>(side.items);
    S.bounds = reinterpret_cast<int2 *>(side.item_bounds);
    return BPT_OK;
}

template <typename F> int64_t most_of(const PlanSides &b, int n_sides, F &&f) {
    const int64_t x = f(b.side[0]), y = n_sides == 2 ? f(b.side[1]) : 0;
    return x > y ? x : y;
}

inline bool small_plans(const PlanSides &b, int n_sides) { return small_plan(b.side[0]) && (n_sides < 2 || small_plan(b.side[1])); }

// base_build leaves both orders of the items
inline bool ordered_plans(const PlanSides &b, int n_sides) {
    bool fit = true;
    for (int i = 0; i < n_sides; ++i) fit = fit && b.side[i].indices && order_in_lds(b.side[i]);
    return fit || small_plans(b, n_sides);
}

int base_build(const PlanSides &b, int n_sides, const SortWs &w, hipStream_t s) {
    const unsigned ns = (unsigned)n_sides;
    if (small_plans(b, n_sides)) {
        hipLaunchKernelGGL(k_plan_small, dim3(ns), dim3(SMALL_TPB), 0, s, b, (int32_t *)nullptr);
        HIP_TRY(hipGetLastError());
        return BPT_OK;
    }
    hipLaunchKernelGGL(k_plan_clear, dim3(1, ns), dim3(64), 0, s, b);
    HIP_TRY(hipGetLastError());
    const unsigned edge_blocks = blocks_for(most_of(b, n_sides, [](const PlanSide &S) { return S.n_edges; }));
    const unsigned unit_blocks = blocks_for(most_of(b, n_sides, [](const PlanSide &S) { return S.n_units; }));
    const unsigned row_blocks = (unsigned)most_of(b, n_sides, [](const PlanSide &S) { return item_row_blocks(S.n_rows); });
    hipLaunchKernelGGL(k_plan_narrow, dim3(edge_blocks + unit_blocks + row_blocks, ns), dim3(TPB), 0, s, b, edge_blocks, unit_blocks);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_plan_items, dim3(row_blocks + edge_blocks, ns), dim3(TPB), 0, s, b, row_blocks);
    HIP_TRY(hipGetLastError());
    const int64_t max_items = most_of(b, n_sides, [](const PlanSide &S) { return S.max_items; });
    const bool sorted = b.side[0].indices != nullptr;          // (two sides: tiles, which have indices)
    if (max_items == 0 || (!sorted && !b.side[0].bounds)) return BPT_OK;
    hipLaunchKernelGGL(k_item_bounds, dim3(blocks_for(max_items * 16), ns), dim3(TPB), 0, s, b);
    HIP_TRY(hipGetLastError());
    if (!sorted) return BPT_OK;
    if (ordered_plans(b, n_sides)) {
        hipLaunchKernelGGL(k_item_order, dim3(ns), dim3(SMALL_TPB), 0, s, b);
        HIP_TRY(hipGetLastError());
        return BPT_OK;
    }
    const int64_t pad = most_of(b, n_sides, [](const PlanSide &S) { return S.n_index_nodes; }) + 1;
    return rs_sort(ItemRecs{b, 0}, ItemsSorted{b}, RsSizes{{b.side[0].max_items, b.side[1].max_items}}, n_sides, (uint64_t)pad, w.key, w.val, w.counts,
                   w.totals, s);
}

// ordered: base_build has left the items' order by the largest neighbour (jorder)
int groups_count(const PlanSides &b, int n_sides, int32_t R, const SortWs &w, hipStream_t s, bool ordered = false) {
    const unsigned ns = (unsigned)n_sides;
    const int64_t max_items = most_of(b, n_sides, [](const PlanSide &S) { return S.max_items; });
    if (max_items > 0) {
        // the items in the order of their largest neighbour; R consecutive ones are a group
        const int64_t n_index = most_of(b, n_sides, [](const PlanSide &S) { return S.n_index_nodes; });
        const int st = ordered ? BPT_OK : rs_sort(ItemRecs{b, 1}, ItemOrder{b}, RsSizes{{b.side[0].max_items, b.side[1].max_items}}, n_sides, (uint64_t)n_index + 1, w.key,
                               w.val, w.counts, w.totals, s);
        if (st != BPT_OK) return st;
        const int64_t place_bits = most_of(b, n_sides, [](const PlanSide &S) { return S.place_bits; });
        const bool narrow = (int64_t)bits_for((uint64_t)n_index) + 4 + place_bits <= 31;
        const dim3 grid((unsigned)most_of(b, n_sides, [](const PlanSide &S) { return S.max_groups; }), ns);
        auto form = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(TPB), 0, s, b, R);
            return hipGetLastError();
        };
        const int64_t cap = R * most_of(b, n_sides, [](const PlanSide &S) { return S.seg_len; });
        if (narrow) HIP_TRY(cap <= 1024 ? form(k_group_form<1024, uint32_t>) : cap <= 2048 ? form(k_group_form<2048, uint32_t>) : form(k_group_form<4096, uint32_t>));
        else HIP_TRY(cap <= 1024 ? form(k_group_form<1024, uint64_t>) : cap <= 2048 ? form(k_group_form<2048, uint64_t>) : form(k_group_form<4096, uint64_t>));
    }
    const int64_t max_groups = most_of(b, n_sides, [](const PlanSide &S) { return S.max_groups; });
    const unsigned places = (unsigned)((max_groups + GRP_PLACE - 1) / GRP_PLACE);
    if (places > 0) {
        hipLaunchKernelGGL(k_group_place, dim3(places, ns), dim3(GRP_PLACE_TPB), 0, s, b, R);
        HIP_TRY(hipGetLastError());
    }
    hipLaunchKernelGGL(k_group_order, dim3(places + 1, ns), dim3(GRP_PLACE_TPB), 0, s, b, R);
    HIP_TRY(hipGetLastError());
    return BPT_OK;
}

// counts: 16 ints per side, as the groups' info block
int groups_write(const PlanSides &b, int n_sides, int32_t R, const int32_t *counts, const bpt_build_tiles *out, int32_t pad_entries, hipStream_t s) {
    if (!counts || !out || pad_entries < 0) return BPT_ERR_NULL;
    GroupsOuts outs{};
    int32_t most = 0;
    for (int i = 0; i < n_sides; ++i) {
        const PlanSide &S = b.side[i];
        const bpt_build_tiles &o = out[i];
        const int32_t ng = counts[16 * i + BPT_GI_N_GROUPS], ne = counts[16 * i + BPT_GI_N_ENTRIES];
        if (ng < 0 || ng > S.max_groups || ne < 0 || ne > S.n_edges) return BPT_ERR_SIZE;
        if (!o.grp_ptr || !o.entries || !o.grp_eids || !o.chunks || !o.group_info || (ng > 0 && !o.members) || (S.n_edges > 0 && !o.pair_eid))
            return BPT_ERR_NULL;
        outs.side[i] = GroupsOut{ng, ne, counts[16 * i + BPT_GI_MAX_CHUNK], o.members, o.grp_ptr, o.pair_eid, o.grp_eids, o.chunks, o.group_info,
                                 reinterpret_cast<int4 *>(o.entries), o.number};
        most = ng > most ? ng : most;
    }
    hipLaunchKernelGGL(k_group_write, dim3((unsigned)most + 1, (unsigned)n_sides), dim3(TPB), 0, s, b, outs, R, pad_entries);
    HIP_TRY(hipGetLastError());
    return BPT_OK;
}

int csr_build(CsrSides g, int n_sides, int64_t n_edges, int64_t n_nodes, int32_t chunk, void *workspace, int64_t workspace_bytes,
              hipStream_t s) {
    if (n_edges < 0 || n_nodes < 0 || n_edges >= INT32_MAX || n_nodes >= INT32_MAX) return BPT_ERR_SIZE;
    if (chunk < 1) return BPT_ERR_SHAPE;
    if (!workspace) return BPT_ERR_NULL;
    for (int i = 0; i < n_sides; ++i) {
        const CsrSide &c = g.side[i];
        if (!c.indptr || !c.unit_ptr || !c.info) return BPT_ERR_NULL;
        if (n_edges > 0 && (!c.rows || !c.cols || !c.indices || !c.eid || !c.unit_row)) return BPT_ERR_NULL;
    }
    Bump bump{(char *)workspace, 0};
    CsrWs w = csr_layout(bump, n_edges, n_nodes, n_sides, g);
    if (workspace_bytes < (int64_t)bump.off) return BPT_ERR_WORKSPACE;
    if (csr_small(n_edges, n_nodes)) {
        hipLaunchKernelGGL(k_csr_small, dim3((unsigned)n_sides), dim3(SMALL_TPB), 0, s, g, (int)n_edges, (int)n_nodes, chunk);
        HIP_TRY(hipGetLastError());
        return BPT_OK;
    }
    // (n_nodes: the key of an edge with a bad id)
    const int st = rs_sort(CsrEdges{g, n_nodes}, CsrSlots{g}, RsSizes{{n_edges, n_edges}}, n_sides, (uint64_t)n_nodes, w.key, w.val, w.counts,
                           w.totals, s);
    if (st != BPT_OK) return st;
    const dim3 rows((unsigned)((n_nodes + CSR_ROWS) / CSR_ROWS), (unsigned)n_sides);
    hipLaunchKernelGGL(k_csr_rows, rows, dim3(TPB), 0, s, g, n_edges, n_nodes, chunk);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_csr_units, rows, dim3(TPB), 0, s, g, n_edges, n_nodes, chunk, n_edges > 0 ? rs_tiles(n_edges) : (int64_t)0);
    HIP_TRY(hipGetLastError());
    return BPT_OK;
}

}  // namespace

extern "C" {

int bpt_build_count_rows(const int64_t *const row[2], const int64_t *const indptr_units[2], const int64_t n_units[2], int n_sides, int32_t *counts,
                         void *stream) {
    if (n_sides < 1 || n_sides > 2) return BPT_ERR_SHAPE;
    if (!row || !indptr_units || !n_units || !counts) return BPT_ERR_NULL;
    UnitSides b{};
    for (int i = 0; i < n_sides; ++i) {
        if (n_units[i] < 0 || n_units[i] >= INT32_MAX) return BPT_ERR_SIZE;
        if (n_units[i] > 0 && (!row[i] || !indptr_units[i])) return BPT_ERR_NULL;
        b.side[i] = UnitSide{row[i], indptr_units[i], (int32_t)n_units[i]};
    }
    hipLaunchKernelGGL(k_count_rows, dim3(BPT_COUNT_PARTS, n_sides), dim3(TPB), 0, (hipStream_t)stream, b, counts);
    HIP_TRY(hipGetLastError());
    return BPT_OK;
}

int bpt_build_wait(void *stream) {
    HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
    return BPT_OK;
}

int bpt_graph_count_device(int kind, int64_t length, int triu, int64_t a, int64_t b, int32_t *offsets, void *workspace,
                           int64_t workspace_bytes, void *stream) {
    if (!graph_args_ok(kind, length, a, b)) return BPT_ERR_SIZE;
    if (!offsets || !workspace) return BPT_ERR_NULL;
    LevelTable lv;
    if (!level_table(kind, length, lv)) return BPT_ERR_SIZE;
    size_t tmp = 0, tb = 0;
    HIP_TRY(scan_i32(nullptr, tmp, nullptr, nullptr, length + 1, nullptr));
    Bump bump{(char *)workspace, 0};
    int32_t *counts = bump.take<int32_t>(length + 1);
    void *scratch = bump.take<char>((int64_t)tmp + 256);
    if (workspace_bytes < (int64_t)bump.off) return BPT_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    LAUNCH(k_graph_count, length + 1, kind, lv, length, triu, a, b, counts);
    tb = tmp + 256;
    HIP_TRY(scan_i32(scratch, tb, counts, offsets, length + 1, s));
    return BPT_OK;
}

int bpt_graph_fill_device(int kind, int64_t length, int triu, int64_t a, int64_t b, int64_t v_shift, const int32_t *offsets,
                          int64_t n_edges, int64_t *src, int64_t *dst, int64_t *etype, void *stream) {
    if (!graph_args_ok(kind, length, a, b) || n_edges < 0) return BPT_ERR_SIZE;
    if (!offsets || (n_edges > 0 && (!src || !dst || !etype))) return BPT_ERR_NULL;
    LevelTable lv;
    if (!level_table(kind, length, lv)) return BPT_ERR_SIZE;
    hipStream_t s = (hipStream_t)stream;
    LAUNCH(k_graph_fill, length, kind, lv, length, triu, a, b, v_shift, offsets, n_edges, src, dst, etype);
    return BPT_OK;
}

int bpt_csr_device_bounds(int64_t n_edges, int64_t n_nodes, int32_t chunk_size, int64_t bounds[2]) {
    if (!bounds) return BPT_ERR_NULL;
    if (n_edges < 0 || n_nodes < 0 || n_edges >= INT32_MAX || n_nodes >= INT32_MAX) return BPT_ERR_SIZE;
    if (chunk_size < 1) return BPT_ERR_SHAPE;
    Bump dry{nullptr, 0};
    CsrSides g;
    csr_layout(dry, n_edges, n_nodes, 2, g);
    const int64_t by_rows = n_nodes + n_edges / chunk_size;
    bounds[0] = by_rows < n_edges ? by_rows : n_edges;
    bounds[1] = (int64_t)dry.off + 256;
    return BPT_OK;
}

int bpt_csr_build_device(const int64_t *rows, const int64_t *cols, int64_t n_edges, int64_t n_nodes, int32_t chunk_size,
                         int64_t *indptr, int64_t *indices, int64_t *eid, int64_t *unit_row, int64_t *unit_ptr, int32_t *info,
                         void *workspace, int64_t workspace_bytes, void *stream) {
    CsrSides g{};
    g.side[0] = CsrSide{rows, cols, indptr, indices, eid, unit_row, unit_ptr, info, nullptr, nullptr, nullptr, nullptr};
    return csr_build(g, 1, n_edges, n_nodes, chunk_size, workspace, workspace_bytes, (hipStream_t)stream);
}

int bpt_build_merge_device(const int64_t *parts, int64_t n_parts, int64_t *src, int64_t *dst, int64_t *etype, int64_t *pos, void *stream) {
    if (n_parts < 0) return BPT_ERR_SIZE;
    if (n_parts > 0 && (!parts || !pos)) return BPT_ERR_NULL;
    hipStream_t s = (hipStream_t)stream;
    int64_t edge = 0, node = 0;
    for (int64_t p0 = 0; p0 < n_parts; p0 += MERGE_PARTS) {
        MergeParts m{};
        m.n = (int)(n_parts - p0 < MERGE_PARTS ? n_parts - p0 : MERGE_PARTS);
        const int64_t edge0 = edge, node0 = node;
        for (int i = 0; i < m.n; ++i) {
            const int64_t *a = parts + 6 * (p0 + i);
            m.part[i] = MergePart{(const int64_t *)a[0], (const int64_t *)a[1], (const int64_t *)a[2], (const int64_t *)a[3], edge, node};
            if (a[4] < 0 || a[5] < 0 || a[4] >= INT32_MAX || a[5] >= INT32_MAX) return BPT_ERR_SIZE;
            if ((a[4] > 0 && (!a[0] || !a[1] || !a[2] || !src || !dst || !etype)) || (a[5] > 0 && !a[3])) return BPT_ERR_NULL;
            edge += a[4];
            node += a[5];
        }
        m.edge_end = edge;
        m.node_end = node;
        auto blocks = [](int64_t n) { return (unsigned)((n + TPB * MERGE_PER - 1) / (TPB * MERGE_PER)); };
        const unsigned eb = blocks(edge - edge0), nb = blocks(node - node0);
        if (eb + nb == 0) continue;
        hipLaunchKernelGGL(k_merge, dim3(eb + nb), dim3(TPB), 0, s, m, eb, src, dst, etype, pos);
        HIP_TRY(hipGetLastError());
    }
    return BPT_OK;
}

int bpt_build_csrs_device(const int64_t *src, const int64_t *dst, int64_t n_edges, int64_t n_nodes, int32_t chunk_size,
                          int64_t *const out_side[5], int64_t *const in_side[5], int32_t *info, void *workspace,
                          int64_t workspace_bytes, void *stream) {
    if (!out_side || !in_side || !info) return BPT_ERR_NULL;
    CsrSides g{};
    for (int i = 0; i < 2; ++i) {
        int64_t *const *o = i == 0 ? out_side : in_side;
        g.side[i] = CsrSide{i == 0 ? src : dst, i == 0 ? dst : src, o[0], o[1], o[2], o[3], o[4], info + 2 * i,
                            nullptr, nullptr, nullptr, nullptr};
    }
    return csr_build(g, 2, n_edges, n_nodes, chunk_size, workspace, workspace_bytes, (hipStream_t)stream);
}

int bpt_plan_device_bounds(int64_t n_units, int64_t n_edges, int64_t n_rows, int32_t seg_len, int32_t R, int64_t bounds[4]) {
    if (!bounds) return BPT_ERR_NULL;
    const int st = sizes_ok(n_units, n_edges, n_rows, 0, seg_len);
    if (st != BPT_OK) return st;
    if (R < 0 || R > 16) return BPT_ERR_SHAPE;
    const int64_t max_items = n_rows + n_edges / seg_len;
    const int64_t max_heavy = n_edges / ((int64_t)seg_len + 1);
    const int64_t max_groups = R > 0 ? (max_items + R - 1) / R : 0;
    if (max_items >= INT32_MAX || (R > 0 && (n_edges + 8) * R >= INT32_MAX)) return BPT_ERR_SIZE;
    size_t tmp = 0;
    HIP_TRY(temp_bytes(max_items, max_groups, n_edges, n_rows, &tmp));
    Bump a{nullptr, 0}, b{nullptr, 0}, c{nullptr, 0};
    PlanSide S{};
    S.n_edges = n_edges;
    S.n_rows = n_rows;
    S.max_items = max_items;
    base_layout(a, S);
    sort_layout(a, max_items, 1);
    group_layout(b, max_items, max_groups, n_edges, tmp);
    c.take<int32_t>(n_edges);
    size_t ws = a.off > b.off ? a.off : b.off;
    ws = ws > c.off ? ws : c.off;
    bounds[0] = max_items;
    bounds[1] = max_heavy;
    bounds[2] = max_groups;
    bounds[3] = (int64_t)ws + 256;
    return BPT_OK;
}

int bpt_plan_build_device(const int64_t *row, const int64_t *indptr_units, int64_t n_units, const int64_t *eid,
                          const int64_t *indices, int64_t n_edges, int64_t n_rows, int64_t n_index_nodes, int32_t seg_len,
                          int32_t *rowptr, int32_t *idx32, int32_t *eid32, int32_t *items, int32_t *heavy, int32_t *info,
                          void *workspace, int64_t workspace_bytes, void *stream) {
    return bpt_build_plan_device(row, indptr_units, n_units, eid, indices, n_edges, n_rows, n_index_nodes, seg_len, rowptr, idx32, eid32,
                                 items, heavy, nullptr, info, workspace, workspace_bytes, stream);
}

int bpt_build_plan_device(const int64_t *row, const int64_t *indptr_units, int64_t n_units, const int64_t *eid,
                          const int64_t *indices, int64_t n_edges, int64_t n_rows, int64_t n_index_nodes, int32_t seg_len,
                          int32_t *rowptr, int32_t *idx32, int32_t *eid32, int32_t *items, int32_t *heavy, int32_t *item_bounds,
                          int32_t *info, void *workspace, int64_t workspace_bytes, void *stream) {
    bpt_build_side side{row, indptr_units, eid, indices, n_units, n_edges, n_rows, n_index_nodes, seg_len, 0, rowptr, idx32, eid32, items,
                        item_bounds, heavy, info};
    PlanSides b{};
    const int st = fill_side(side, b.side[0]);
    if (st != BPT_OK) return st;
    if (!workspace) return BPT_ERR_NULL;
    Bump bump{(char *)workspace, 0};
    base_layout(bump, b.side[0]);
    const SortWs w = sort_layout(bump, b.side[0].max_items, 1);
    if (workspace_bytes < (int64_t)bump.off) return BPT_ERR_WORKSPACE;
    return base_build(b, 1, w, (hipStream_t)stream);
}

int bpt_build_groups_bounds(int64_t max_items, int64_t n_edges, int64_t n_index_nodes, int32_t seg_len, int32_t R, int64_t bounds[1]) {
    if (!bounds) return BPT_ERR_NULL;
    PlanSide S{};
    const int st = short_form(max_items, n_edges, n_index_nodes, seg_len, R, 0, S);
    if (st != BPT_OK) return st;
    Bump dry{nullptr, 0};
    short_layout(dry, S);
    sort_layout(dry, max_items, 1);
    bounds[0] = (int64_t)dry.off + 256;
    return BPT_OK;
}

int bpt_build_groups_count(const int32_t *items, const int32_t *item_bounds, const int32_t *idx32, const int32_t *eid32,
                           const int32_t *plan_info, int64_t max_items, int64_t n_edges, int64_t n_index_nodes, int32_t seg_len, int32_t R,
                           int32_t by_mask, int32_t *out_info, void *workspace, int64_t workspace_bytes, void *stream) {
    PlanSides b{};
    PlanSide &S = b.side[0];
    const int st = short_form(max_items, n_edges, n_index_nodes, seg_len, R, by_mask, S);
    if (st != BPT_OK) return st;
    if (!plan_info || !out_info || !workspace || (max_items > 0 && (!items || !item_bounds))) return BPT_ERR_NULL;
    if (n_edges > 0 && (!idx32 || !eid32)) return BPT_ERR_NULL;
    S.items = (int4 *)items;
    S.bounds = (int2 *)item_bounds;
    S.idx32 = (int32_t *)idx32;
    S.eid32 = (int32_t *)eid32;
    S.info = (int32_t *)plan_info;
    S.out_info = out_info;
    Bump bump{(char *)workspace, 0};
    short_layout(bump, S);
    const SortWs w = sort_layout(bump, max_items, 1);
    if (workspace_bytes < (int64_t)bump.off) return BPT_ERR_WORKSPACE;
    return groups_count(b, 1, R, w, (hipStream_t)stream);
}

int bpt_build_groups_write(const int32_t *items, const int32_t *plan_info, int64_t max_items, int64_t n_edges, int64_t n_index_nodes,
                           int32_t seg_len, int32_t R, const int32_t *group_counts, int32_t pad_entries, int32_t *members,
                           int32_t *grp_ptr, int32_t *entries, int32_t *pair_eid, int32_t *grp_eids, int32_t *chunks, int32_t *group_info,
                           void *workspace, int64_t workspace_bytes, void *stream) {
    PlanSides b{};
    PlanSide &S = b.side[0];
    const int st = short_form(max_items, n_edges, n_index_nodes, seg_len, R, 0, S);
    if (st != BPT_OK) return st;
    if (!plan_info || !workspace || (max_items > 0 && !items)) return BPT_ERR_NULL;
    S.items = (int4 *)items;
    S.info = (int32_t *)plan_info;
    const bpt_build_tiles out{members, grp_ptr, entries, pair_eid, grp_eids, chunks, group_info, nullptr};
    Bump bump{(char *)workspace, 0};
    short_layout(bump, S);
    if (workspace_bytes < (int64_t)bump.off) return BPT_ERR_WORKSPACE;
    return groups_write(b, 1, R, group_counts, &out, pad_entries, (hipStream_t)stream);
}

// where the call below puts the sides' arrays in its workspace
static int base_sides(const bpt_build_side *sides, int n_sides, PlanSides &b, SortWs &w, Bump &bump) {
    int64_t most = 0;
    for (int i = 0; i < n_sides; ++i) {
        const bpt_build_side &side = sides[i];
        PlanSide &S = b.side[i];
        const int st = sizes_ok(side.n_units, side.n_edges, side.n_rows, side.n_index_nodes, side.seg_len);
        if (st != BPT_OK) return st;
        S.n_edges = side.n_edges;
        S.n_rows = side.n_rows;
        S.max_items = side.n_rows + side.n_edges / side.seg_len;
        if (S.max_items >= INT32_MAX) return BPT_ERR_SIZE;
        base_layout(bump, S);
        most = S.max_items > most ? S.max_items : most;
    }
    w = sort_layout(bump, most, n_sides);
    return BPT_OK;
}

int bpt_build_plans_bounds(const bpt_build_side *sides, int n_sides, int64_t bounds[1]) {
    if (!sides || !bounds || n_sides < 1 || n_sides > 2) return BPT_ERR_NULL;
    PlanSides b{};
    SortWs w;
    Bump dry{nullptr, 0};
    const int st = base_sides(sides, n_sides, b, w, dry);
    bounds[0] = (int64_t)dry.off + 256;
    return st;
}

int bpt_build_plans(const bpt_build_side *sides, int n_sides, int32_t *out_info, void *workspace, int64_t workspace_bytes, void *stream) {
    if (!sides || !out_info || !workspace || n_sides < 1 || n_sides > 2) return BPT_ERR_NULL;
    PlanSides b{};
    SortWs w;
    Bump bump{(char *)workspace, 0};
    int st = base_sides(sides, n_sides, b, w, bump);
    if (st != BPT_OK) return st;
    if (workspace_bytes < (int64_t)bump.off) return BPT_ERR_WORKSPACE;
    for (int i = 0; i < n_sides; ++i) {
        st = fill_side(sides[i], b.side[i]);
        if (st != BPT_OK) return st;
        if (!sides[i].indices && sides[i].n_edges > 0) return BPT_ERR_NULL;
    }
    hipStream_t s = (hipStream_t)stream;
    if (small_plans(b, n_sides)) {
        hipLaunchKernelGGL(k_plan_small, dim3((unsigned)n_sides), dim3(SMALL_TPB), 0, s, b, out_info);
    } else {
        st = base_build(b, n_sides, w, s);
        if (st != BPT_OK) return st;
        hipLaunchKernelGGL(k_info_out, dim3((unsigned)n_sides), dim3(16), 0, s, b, out_info);
    }
    HIP_TRY(hipGetLastError());
    return BPT_OK;
}

// where the two calls below put a side's arrays in its part of the workspace
static int tiles_sides(const bpt_build_side *sides, int n_sides, PlanSides &b, SortWs &w, Bump &bump) {
    int64_t most = 0;
    for (int i = 0; i < n_sides; ++i) {
        const bpt_build_side &side = sides[i];
        PlanSide &S = b.side[i];
        int st = fill_side(side, S);
        if (st != BPT_OK) return st;
        if (!side.item_bounds && S.max_items > 0) return BPT_ERR_NULL;
        st = short_form(S.max_items, S.n_edges, S.n_index_nodes, S.seg_len, 16, side.by_mask, S);
        if (st != BPT_OK) return st;
        base_layout(bump, S);
        short_layout(bump, S);
        most = S.max_items > most ? S.max_items : most;
    }
    w = sort_layout(bump, most, n_sides);
    return BPT_OK;
}

int bpt_build_tiles_bounds(const bpt_build_side *sides, int n_sides, int64_t bounds[1]) {
    if (!sides || !bounds || n_sides < 1 || n_sides > 2) return BPT_ERR_NULL;
    int64_t most = 0;
    Bump dry{nullptr, 0};
    for (int i = 0; i < n_sides; ++i) {
        const bpt_build_side &side = sides[i];
        int st = sizes_ok(side.n_units, side.n_edges, side.n_rows, side.n_index_nodes, side.seg_len);
        if (st != BPT_OK) return st;
        PlanSide S{};
        S.n_rows = side.n_rows;
        const int64_t max_items = side.n_rows + side.n_edges / side.seg_len;
        st = short_form(max_items, side.n_edges, side.n_index_nodes, side.seg_len, 16, side.by_mask, S);
        if (st != BPT_OK) return st;
        base_layout(dry, S);
        short_layout(dry, S);
        most = max_items > most ? max_items : most;
    }
    sort_layout(dry, most, n_sides);
    bounds[0] = (int64_t)dry.off + 256;
    return BPT_OK;
}

int bpt_build_tiles_count(const bpt_build_side *sides, int n_sides, int32_t *out_info, void *workspace, int64_t workspace_bytes, void *stream) {
    if (!sides || !out_info || !workspace || n_sides < 1 || n_sides > 2) return BPT_ERR_NULL;
    PlanSides b{};
    SortWs w;
    Bump bump{(char *)workspace, 0};
    int st = tiles_sides(sides, n_sides, b, w, bump);
    if (st != BPT_OK) return st;
    if (workspace_bytes < (int64_t)bump.off) return BPT_ERR_WORKSPACE;
    for (int i = 0; i < n_sides; ++i) b.side[i].out_info = out_info + 32 * i;
    st = base_build(b, n_sides, w, (hipStream_t)stream);
    return st != BPT_OK ? st : groups_count(b, n_sides, 16, w, (hipStream_t)stream, ordered_plans(b, n_sides));
}

int bpt_build_tiles_write(const bpt_build_side *sides, int n_sides, const int32_t *infos, const bpt_build_tiles *out, int32_t pad_entries,
                          int32_t *pairs, void *workspace, int64_t workspace_bytes, void *stream) {
    if (!sides || !infos || !out || !workspace || n_sides < 1 || n_sides > 2) return BPT_ERR_NULL;
    PlanSides b{};
    SortWs w;
    Bump bump{(char *)workspace, 0};
    int st = tiles_sides(sides, n_sides, b, w, bump);
    if (st != BPT_OK) return st;
    if (workspace_bytes < (int64_t)bump.off) return BPT_ERR_WORKSPACE;
    const int32_t counts[32] = {infos[16], infos[17], infos[18], 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
                                n_sides == 2 ? infos[48] : 0, n_sides == 2 ? infos[49] : 0, n_sides == 2 ? infos[50] : 0};
    st = groups_write(b, n_sides, 16, counts, out, pad_entries, (hipStream_t)stream);
    if (st != BPT_OK || !pairs) return st;
    if (n_sides != 2 || !out[0].number || sides[0].n_edges != sides[1].n_edges) return BPT_ERR_PLAN;
    hipStream_t s = (hipStream_t)stream;
    const int64_t n_slots = ((int64_t)counts[16 + BPT_GI_N_ENTRIES] + pad_entries) * 16;
    LAUNCH(k_find_numbers, n_slots, out[1].grp_eids, n_slots, sides[1].n_edges, out[0].number, pairs);
    return BPT_OK;
}

int bpt_build_pair_numbers(const int32_t *pair_eid_theirs, const int32_t *grp_eids_mine, int64_t n_slots, int64_t n_edges, int32_t *number,
                           int32_t *pairs, void *stream) {
    if (n_edges < 0 || n_slots < 0 || n_edges >= INT32_MAX || n_slots >= INT32_MAX) return BPT_ERR_SIZE;
    if ((n_edges > 0 && (!pair_eid_theirs || !number)) || (n_slots > 0 && (!grp_eids_mine || !pairs))) return BPT_ERR_NULL;
    hipStream_t s = (hipStream_t)stream;
    LAUNCH(k_number_pairs, n_edges, pair_eid_theirs, n_edges, number);
    LAUNCH(k_find_numbers, n_slots, grp_eids_mine, n_slots, n_edges, number, pairs);
    return BPT_OK;
}

int bpt_plan_group_device(const int32_t *items, const int32_t *idx32, const int32_t *eid32, const int32_t *plan_info,
                          int64_t max_items, int64_t n_edges, int64_t n_index_nodes, int32_t seg_len, int32_t R,
                          int32_t by_mask, int32_t *members, int32_t *grp_ptr, int32_t *entries, int32_t *pair_eid,
                          int32_t *grp_eids, int32_t *chunks, int32_t *group_info, void *workspace,
                          int64_t workspace_bytes, void *stream) {
    if (max_items < 0 || n_edges < 0 || n_index_nodes < 0 || max_items >= INT32_MAX || n_edges >= INT32_MAX ||
        n_index_nodes >= INT32_MAX)
        return BPT_ERR_SIZE;
    if (R < 1 || R > 16 || seg_len < 1 || by_mask < 0 || (by_mask & 3) > 2 || by_mask > 6) return BPT_ERR_SHAPE;
    const int by_work = (by_mask & 4) ? 0 : 1;                   // + 4: the groups of a range keep their locality order
    by_mask &= 3;
    if ((int64_t)R * seg_len + FIXED_WORK > 0xFFFF) return BPT_ERR_UNSUPPORTED;       // the work of a group is a 16-bit sort key
    if ((n_edges + 8) * R >= INT32_MAX) return BPT_ERR_SIZE;
    if (!plan_info || !grp_ptr || !entries || !grp_eids || !chunks || !group_info || !workspace) return BPT_ERR_NULL;
    if (max_items > 0 && (!items || !members)) return BPT_ERR_NULL;
    if (n_edges > 0 && (!idx32 || !eid32 || !pair_eid)) return BPT_ERR_NULL;
    const int64_t max_groups = (max_items + R - 1) / R;
    if (max_groups >= (int64_t)1 << 28) return BPT_ERR_UNSUPPORTED;                    // group numbers are 28-bit sort keys
    size_t tmp = 0;
    HIP_TRY(temp_bytes(max_items, max_groups, n_edges, 0, &tmp));
    Bump dry{nullptr, 0};
    group_layout(dry, max_items, max_groups, n_edges, tmp);
    if (workspace_bytes < (int64_t)dry.off) return BPT_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    Bump bump{(char *)workspace, 0};
    GroupWs w = group_layout(bump, max_items, max_groups, n_edges, tmp);
    size_t tb;

    // the items in the order of their largest neighbour; R consecutive ones are a group
    if (max_items > 0) {
        LAUNCH(k_item_keys<true>, max_items, items, idx32, plan_info, max_items, n_index_nodes, n_edges, w.key);
        LAUNCH(k_iota_i32, max_items, w.iota, max_items);
        tb = tmp;
        HIP_TRY(sort_pairs<uint32_t>(w.tmp, tb, w.key, w.key_s, w.iota, w.jorder, max_items, 32, s));
    }
    // the groups numbered by locality (smallest neighbour id), cut into 8 ranges of equal work, by decreasing work
    // inside a range
    if (max_items > 0) LAUNCH(k_item_keys<false>, max_items, items, idx32, plan_info, max_items, n_index_nodes, n_edges, w.key);
    LAUNCH(k_group_work, max_groups + 1, items, w.jorder, w.key, plan_info, max_groups, R, w.work0, w.key_s, group_info);
    if (max_groups > 0) {
        LAUNCH(k_iota_i32, max_groups, w.iota, max_groups);
        tb = tmp;
        HIP_TRY(sort_pairs<uint32_t>(w.tmp, tb, w.key_s, w.key, w.iota, w.lorder, max_groups, 32, s));
        LAUNCH(k_invert, max_groups, w.lorder, group_info, (int)BPT_GI_N_GROUPS, max_groups, w.lpos);
    }
    // Tiles (R = 16) are cut into ranges and ordered by their blocks of entries, which are known only after the record sort
    // below: their records carry the locality numbers first.  The other groups are balanced by their pairs, as formed.
    const bool by_blocks = (R == 16);
    auto number_groups = [&]() -> int {                   // w.work (locality numbering) -> chunks, w.gorder, w.inv
        size_t tb2 = tmp;
        HIP_TRY(scan_i32(w.tmp, tb2, w.work, w.prefix, max_groups + 1, s));
        hipLaunchKernelGGL(k_chunks, dim3(1), dim3(64), 0, s, w.work, w.prefix, plan_info, R, chunks, group_info);
        HIP_TRY(hipGetLastError());
        if (max_groups > 0) {
            LAUNCH(k_group_keys, max_groups, w.work, chunks, plan_info, max_groups, R, by_work, w.key_s);
            LAUNCH(k_iota_i32, max_groups, w.iota, max_groups);
            tb2 = tmp;
            HIP_TRY(sort_pairs<uint32_t>(w.tmp, tb2, w.key_s, w.key, w.iota, w.gorder, max_groups, 32, s));
            LAUNCH(k_invert, max_groups, w.gorder, group_info, (int)BPT_GI_N_GROUPS, max_groups, w.inv);
        }
        return BPT_OK;
    };
    if (!by_blocks) {
        LAUNCH(k_gather_work, max_groups + 1, w.work0, w.lorder, group_info, max_groups, w.work);
        const int st = number_groups();
        if (st != BPT_OK) return st;
    }
    if (max_groups > 0)
        LAUNCH(k_members_and_records, max_groups * R, items, idx32, w.jorder, w.lpos, by_blocks ? (const int32_t *)nullptr : w.inv, plan_info,
               max_groups, n_edges, R, by_blocks ? (int32_t *)nullptr : members, w.ekey, w.eval);
    // entries: distinct (group, neighbour, multiplicity) of the records sorted by (group, neighbour, member)
    LAUNCH(k_fill_i32, (n_edges + 8) * R, grp_eids, (n_edges + 8) * R, (int32_t)n_edges);
    if (n_edges > 0) {
        LAUNCH(k_pad_records, n_edges, w.ekey, w.eval, n_edges, plan_info);
        tb = tmp;
        HIP_TRY(sort_pairs<uint64_t>(w.tmp, tb, w.ekey, w.ekey_s, w.eval, w.eval_s, n_edges, 35 + bits_for((uint64_t)max_groups), s));
    }
    LAUNCH(k_rank, n_edges + 1, w.ekey_s, n_edges, plan_info, w.rank, w.head);
    tb = tmp;
    HIP_TRY(scan_i32(w.tmp, tb, w.head, w.run, n_edges + 1, s));       // w.run = exclusive scan for now
    LAUNCH(k_fill_i32, n_edges + 1, w.mult, n_edges + 1, 0);
    LAUNCH(k_fill_i32, n_edges, w.ent_mask, n_edges, 0);
    LAUNCH(k_multiplicity, n_edges, w.rank, w.head, w.run, n_edges, plan_info, w.run, w.mult);
    tb = tmp;
    HIP_TRY(scan_i32(w.tmp, tb, w.mult, w.ebase, n_edges + 1, s));
    LAUNCH(k_entry_fill, n_edges, w.ekey_s, w.rank, w.run, w.ebase, n_edges, plan_info, w.ent_of, w.ent_idx, w.ent_g,
           w.ent_mask, group_info);
    if (by_blocks) {
        // the tiles' cost is known now: their ranges, their final numbers, their members; the entries take the final numbers
        LAUNCH(k_block_work, max_groups + 1, w.ent_g, group_info, max_groups, R, w.work);
        const int st = number_groups();
        if (st != BPT_OK) return st;
        if (max_groups > 0)
            LAUNCH(k_members_and_records, max_groups * R, items, idx32, w.jorder, w.lpos, w.inv, plan_info, max_groups, n_edges, R, members,
                   (uint64_t *)nullptr, (int32_t *)nullptr);
        if (n_edges > 0) LAUNCH(k_renumber, n_edges, w.ent_g, w.inv, n_edges, group_info);
    }
    // entry order inside a group: neighbour order, or by member mask (larger first, neighbour order inside a mask); the
    // entries of renumbered groups are sorted in every case
    int32_t *perm = w.iota;                               // new position -> entry as numbered above
    LAUNCH(k_iota_i32, n_edges, w.iota, n_edges);
    if ((by_mask != 0 || by_blocks) && n_edges > 0) {
        LAUNCH(k_entry_keys, n_edges, w.ent_g, w.ent_mask, w.ent_idx, n_edges, group_info, (int)by_mask, w.ekey);
        tb = tmp;
        HIP_TRY(sort_pairs<uint64_t>(w.tmp, tb, w.ekey, w.mkey_s, w.iota, w.eval, n_edges,
                                     (by_mask == 1 ? 16 : by_mask == 2 ? 35 : 31) + bits_for((uint64_t)max_groups), s));
        perm = w.eval;
    }
    LAUNCH(k_invert, n_edges, perm, group_info, (int)BPT_GI_N_ENTRIES, n_edges, w.newpos);
    LAUNCH(k_popcounts, n_edges + 1, w.ent_mask, perm, n_edges, group_info, w.pop);
    tb = tmp;
    HIP_TRY(scan_i32(w.tmp, tb, w.pop, w.first, n_edges + 1, s));
    LAUNCH(k_entries_out, n_edges + 1, w.ent_idx, w.ent_mask, perm, w.first, n_edges, group_info, entries);
    LAUNCH(k_group_ptr, max_groups + 1, w.ent_g, perm, max_groups, group_info, grp_ptr);
    LAUNCH(k_edge_ids, n_edges, w.ekey_s, w.eval_s, w.ent_of, w.newpos, w.ent_mask, w.first, eid32, n_edges, plan_info, R, grp_eids,
           pair_eid);
    return BPT_OK;
}

int bpt_plan_link_device(const int32_t *grp_eids_dst, const int32_t *group_info_dst, int32_t R_dst,
                         const int32_t *grp_eids_src, const int32_t *group_info_src, int32_t R_src, int64_t n_edges,
                         int32_t pad_entries, int32_t *pairs, void *workspace, int64_t workspace_bytes, void *stream) {
    if (n_edges < 0 || n_edges >= INT32_MAX || pad_entries < 0) return BPT_ERR_SIZE;
    if (R_dst < 1 || R_dst > 16 || R_src < 1 || R_src > 16) return BPT_ERR_SHAPE;
    if (((int64_t)n_edges + pad_entries) * (R_dst > R_src ? R_dst : R_src) >= INT32_MAX) return BPT_ERR_SIZE;
    if (!grp_eids_dst || !group_info_dst || !grp_eids_src || !group_info_src || !pairs || !workspace) return BPT_ERR_NULL;
    if (workspace_bytes < (int64_t)((n_edges > 0 ? n_edges : 1) * sizeof(int32_t) + 256)) return BPT_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    Bump bump{(char *)workspace, 0};
    int32_t *pos = bump.take<int32_t>(n_edges);
    LAUNCH(k_fill_i32, n_edges, pos, n_edges, 0);
    LAUNCH(k_positions, n_edges * R_src, grp_eids_src, group_info_src, R_src, n_edges, pos);
    LAUNCH(k_pairs, (n_edges + pad_entries) * R_dst, grp_eids_dst, group_info_dst, R_dst, group_info_src, R_src, n_edges,
           pad_entries, pos, pairs);
    return BPT_OK;
}

}  // extern "C"
