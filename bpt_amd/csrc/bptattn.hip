// libbptattn: gfx950 HIP kernels of the BPT graph-attention path (C ABI in include/bptattn.h).
//
// Execution model.  One 64-lane wavefront owns one work item of the plan: a whole row of the
// CSR side it walks, or one segment of a row that is longer than the plan's segment length.
// Whole rows write their result directly; segments write a partial result into the workspace
// and a second kernel combines the partials of each split row in slot order.  No atomics
// anywhere, so every output is bit-reproducible run to run.
//
// Two kernel families:
//   * "generic": any h, d and f32 / f64 / bf16, lanes stride over the columns of a node row;
//   * "fast":    compile-time (h, d) for f32 / bf16.  A node row of C = h*d elements is spread
//                over the wavefront so that lane l holds C/64 elements of head l / (64/h) and
//                every 16-byte load instruction of the wavefront covers whole 128-byte lines.
//                A per-head dot product is then C/64 FMAs plus log2(64/h) DPP additions.
// Work items are dealt to workgroups so that each XCD (blocks are distributed round-robin over
// the 8 XCDs) walks a contiguous range of rows: neighbouring tokens share most of their
// neighbours, which keeps the gathered K/V rows in that XCD's L2.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <utility>
#include <vector>

#include "../../include/bptattn.h"
#include "../../include/bptattn_measure.h"

namespace {

constexpr int WAVE = 64;
constexpr int WAVES_PER_BLOCK = 4;
constexpr int BLOCK = WAVE * WAVES_PER_BLOCK;
constexpr float M_INIT_LOG2 = -1.4426950408889634e9f;   // -1e9 (graphop_kernel.cu:428) in base-2 units
constexpr float LOG2E = 1.4426950408889634f;

std::atomic<int> g_force_generic{0};

// optional measurement hook (bpt_profile_kernel): which main kernel to bracket with events
std::atomic<int> g_prof_which{0};
std::atomic<void *> g_prof_start{nullptr}, g_prof_stop{nullptr};

struct ProfScope {
    hipStream_t s;
    bool on;
    ProfScope(int which, hipStream_t stream) : s(stream), on(g_prof_which.load(std::memory_order_relaxed) == which) {
        if (on) (void)hipEventRecord((hipEvent_t)g_prof_start.load(), s);
    }
    ~ProfScope() {
        if (on) (void)hipEventRecord((hipEvent_t)g_prof_stop.load(), s);
    }
};

// ------------------------------------------------------------------------------------------
// element types
// ------------------------------------------------------------------------------------------
struct bf16_t { uint16_t bits; };
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);   // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);                                              // round to nearest even
    return (uint16_t)(u >> 16);
}

template <typename T> struct Elem;
template <> struct Elem<float> {
    using acc_t = float;
    static __device__ __forceinline__ float ld(const float *p) { return *p; }
    static __device__ __forceinline__ void st(float *p, float v) { *p = v; }
};
template <> struct Elem<double> {
    using acc_t = double;
    static __device__ __forceinline__ double ld(const double *p) { return *p; }
    static __device__ __forceinline__ void st(double *p, double v) { *p = v; }
};
template <> struct Elem<bf16_t> {
    using acc_t = float;
    static __device__ __forceinline__ float ld(const bf16_t *p) { return bf16_to_f32(p->bits); }
    static __device__ __forceinline__ void st(bf16_t *p, float v) { p->bits = f32_to_bf16(v); }
};

__device__ __forceinline__ float exp_acc(float x) { return expf(x); }
__device__ __forceinline__ double exp_acc(double x) { return exp(x); }

// ------------------------------------------------------------------------------------------
// work distribution
// ------------------------------------------------------------------------------------------
struct Item { int row, begin, end, slot; };

// Blocks go round-robin to the 8 XCDs; remap so XCD x gets a contiguous run of block indices (of those behind the first `skip`,
// a multiple of 8).
__device__ __forceinline__ int xcd_contiguous_block(int skip = 0) {
    const int nb = gridDim.x - skip, b = blockIdx.x - skip;
    const int q = nb >> 3, rem = nb & 7, x = b & 7, k = b >> 3;
    return x * q + (x < rem ? x : rem) + k;
}

__device__ __forceinline__ bool fetch_item(const bpt_plan &P, Item &it, int waves_per_block = WAVES_PER_BLOCK, int skip = 0) {
    const int w = xcd_contiguous_block(skip) * waves_per_block + (int)(threadIdx.x >> 6);
    if (w >= (int)P.n_items) return false;
    const int4 v = reinterpret_cast<const int4 *>(P.items)[w];
    // the item is the same for all lanes of the wavefront: keep it in scalar registers
    it.row = __builtin_amdgcn_readfirstlane(v.x);
    it.begin = __builtin_amdgcn_readfirstlane(v.y);
    it.end = __builtin_amdgcn_readfirstlane(v.z);
    it.slot = __builtin_amdgcn_readfirstlane(v.w);
    return true;
}

template <typename A> __device__ __forceinline__ A wave_sum(A x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    return x;
}
template <typename A> __device__ __forceinline__ A wave_max(A x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        A y = __shfl_xor(x, o);
        x = x > y ? x : y;
    }
    return x;
}

// Reduction over NW wavefronts of a block (NW == 1: a single wavefront, no LDS, no barrier).
template <typename A, int NW, bool IS_MAX> __device__ __forceinline__ A group_reduce(A x, A *smem) {
    x = IS_MAX ? wave_max(x) : wave_sum(x);
    if (NW == 1) return x;
    const int w = threadIdx.x >> 6;
    __syncthreads();                       // smem may still be read from the previous reduction
    if ((threadIdx.x & 63) == 0) smem[w] = x;
    __syncthreads();
    A r = smem[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) r = IS_MAX ? (r > smem[i] ? r : smem[i]) : r + smem[i];
    return r;
}

// ------------------------------------------------------------------------------------------
// generic kernels
// ------------------------------------------------------------------------------------------
// y[eid[p], h] = sum_d A[row, h, d] * B[..]   MODE 0: B (n, H, D) row idx[p];  MODE 1: B (E, D) row eid[p]
template <typename T, int MODE>
__global__ __launch_bounds__(BLOCK) void k_sddmm_generic(bpt_plan P, const T *__restrict__ A, const T *__restrict__ B,
                                                         T *__restrict__ y, int H, int D) {
    using acc_t = typename Elem<T>::acc_t;
    Item it;
    if (!fetch_item(P, it)) return;
    const int lane = threadIdx.x & 63;
    const T *a = A + (size_t)it.row * H * D;
    for (int p = it.begin; p < it.end; ++p) {
        const int e = P.eid[p];
        const T *b = (MODE == 0) ? B + (size_t)P.idx[p] * H * D : B + (size_t)e * D;
        for (int h = 0; h < H; ++h) {
            acc_t s = 0;
            for (int dd = lane; dd < D; dd += WAVE)
                s += (acc_t)Elem<T>::ld(a + h * D + dd) * (acc_t)Elem<T>::ld(b + (MODE == 0 ? h * D : 0) + dd);
            s = wave_sum(s);
            if (lane == 0) Elem<T>::st(y + (size_t)e * H + h, s);
        }
    }
}

// Y[row, j] = sum_p W[eid[p], j / D] * X[..]   MODE 0: X (n, H, D) row idx[p];  MODE 1: X (E, D) row eid[p], column j % D
template <typename T, int MODE>
__global__ __launch_bounds__(BLOCK) void k_spmm_generic(bpt_plan P, const T *__restrict__ W, const T *__restrict__ X,
                                                        T *__restrict__ Y, typename Elem<T>::acc_t *__restrict__ ws,
                                                        int H, int D) {
    using acc_t = typename Elem<T>::acc_t;
    Item it;
    if (!fetch_item(P, it)) return;
    const int lane = threadIdx.x & 63;
    const int C = H * D;
    for (int j = lane; j < C; j += WAVE) {
        const int h = j / D;
        acc_t s = 0;
        for (int p = it.begin; p < it.end; ++p) {
            const int e = P.eid[p];
            const acc_t w = Elem<T>::ld(W + (size_t)e * H + h);
            const acc_t xv = (MODE == 0) ? Elem<T>::ld(X + (size_t)P.idx[p] * C + j) : Elem<T>::ld(X + (size_t)e * D + (j - h * D));
            s += w * xv;
        }
        if (it.slot < 0) Elem<T>::st(Y + (size_t)it.row * C + j, s);
        else ws[(size_t)it.slot * C + j] = s;
    }
}

// Heads of fewer than 64 columns (6 x 50, 8 x 40), read and written as they are in memory by the NARROW forms of the tile kernels.
// The products keep their 64 columns: quad j of a head (the four columns a lane group position stands for) starts at column
// 4 j, or at d - 4 where that would run over the end of the head.  What a shifted quad repeats of its neighbour, and the quads past
// the end, are zero in both operands of the products over the columns (the members': tile_load16, tile_load_row_bf16; the
// entries': tile_rows_to_operand): a masking -inf in one of the last columns counts once, as in a zero-padded head, where
// zero in one operand alone would make it NaN.  Results are stored from the quads that start inside the head, a repeated column
// twice with one value.  No other head's memory is touched, so what stands there does not matter.
// Against copies padded to 64 columns and 4, 8 or 16 heads (three pads, the output and its gradient, three slices, and the
// padding heads computed with the rest): 33 765 nodes / 576 k edges at 6 x 50 with dropout, forward and backward,
// 508 -> 253 us, of which 38 are copies of q, k, v and o for the backward (Keep); of the 508 copies were 223, the rest two
// padding heads of eight.
struct Narrow {
    int d, heads;              // columns of a head, heads
    int h;                     // heads the layer is padded to where that shows: dropout keys, lse and workspace rows
    int slices;                // workgroups per group
};

// Copies that a NARROW forward writes beside its result, for a backward whose caller may have written to the rows in the meantime:
// q, k and v by workgroups of the forward's own launch that do nothing else, spread evenly between those of the tiles, and the
// result where it is stored.  The forward waits for its gathers and products and leaves much of the memory's rate unused.  Training
// pass at 33 765 nodes, 6 x 50 float32 with dropout: 265.1 us with four copies of their own behind the forward (62 us of them),
// 252.7 so, 215 with none; the copying workgroups first or last, or with loads past the L2, 253.8 to 256.5; stored the ordinary way,
// into the L2 that the tiles' rows want, 265.
struct Keep {
    const char *src[3];
    char *dst[3];              // on 16 bytes; null: no copy of this one (bytes = 0)
    int64_t bytes[3];
    int per_xcd;               // copying workgroups per XCD
    void *o;                   // second copy of the result, or null
};
constexpr int KEEP_CHUNK = 16384;          // bytes a workgroup copies

typedef float floatx4k __attribute__((ext_vector_type(4), aligned(4)));
typedef float floatx4n __attribute__((ext_vector_type(4)));
// What workgroup blockIdx.x of a launch with copying workgroups among it is to do: the number of its tile workgroup, or -1 after it
// has copied its chunk.
template <int THREADS> __device__ __forceinline__ int keep_or_tile(const Keep &keep) {
    if (keep.per_xcd == 0) return (int)blockIdx.x;
    const uint32_t x = blockIdx.x & 7, w = blockIdx.x >> 3, all = gridDim.x >> 3, c = (uint32_t)keep.per_xcd;
    const uint32_t before = (uint32_t)((uint64_t)w * c / all), upto = (uint32_t)((uint64_t)(w + 1) * c / all);
    if (before == upto) return (int)((w - before) * 8 + x);
    // (chosen by conditions, not by an index: indexed, the arguments would be copied to scratch memory by every wavefront)
    int64_t at = (int64_t)(before * 8 + x) * KEEP_CHUNK, left = keep.bytes[0];
    const char *src = keep.src[0];
    char *dst = keep.dst[0];
#pragma unroll
    for (int i = 1; i < 3; ++i) {
        const int64_t past = at - (left + KEEP_CHUNK - 1) / KEEP_CHUNK * KEEP_CHUNK;
        if (past >= 0) { at = past; left = keep.bytes[i]; src = keep.src[i]; dst = keep.dst[i]; }
        else break;
    }
    src += at;
    dst += at;
    left -= at;
    constexpr int U = 4;                                          // loads in flight
    const floatx4k *from = reinterpret_cast<const floatx4k *>(src) + threadIdx.x;
    floatx4n *to = reinterpret_cast<floatx4n *>(dst) + threadIdx.x;
    const int n = (int)min((int64_t)KEEP_CHUNK, max(left, (int64_t)0)) / 16;       // whole 16-byte pieces
    if (n == KEEP_CHUNK / 16) {
#pragma unroll 1
        for (int i = 0; i < KEEP_CHUNK / 16; i += U * THREADS) {
            floatx4k v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = from[i + u * THREADS];
#pragma unroll
            for (int u = 0; u < U; ++u) __builtin_nontemporal_store(floatx4n{v[u][0], v[u][1], v[u][2], v[u][3]}, to + (i + u * THREADS));
        }
        return -1;
    }
    // the last chunk of a tensor, and what is left of no whole number of 16 bytes (up to seven bfloat16)
#pragma unroll 1
    for (int i = threadIdx.x; i < n; i += THREADS) {
        const floatx4k v = reinterpret_cast<const floatx4k *>(src)[i];
        reinterpret_cast<floatx4n *>(dst)[i] = floatx4n{v[0], v[1], v[2], v[3]};
    }
    const int64_t end = 16 * (int64_t)n + 2 * (int)threadIdx.x;
    if (end + 2 <= left) *reinterpret_cast<uint16_t *>(dst + end) = *reinterpret_cast<const uint16_t *>(src + end);
    return -1;
}
constexpr int NARROW_HW = 2;   // heads per workgroup (6 x 50: three workgroups of two, none of them half empty)
__device__ __forceinline__ int narrow_col(const Narrow &nw, int quad) { return min(4 * quad, nw.d - 4); }
// whether column e of the quad as loaded is one that the quad before has (or, past the end of the head, any): 4 quad > d - 4 + e
template <bool NARROW> __device__ __forceinline__ bool narrow_again(const Narrow &nw, int quad, int e) {
    return NARROW && quad > (nw.d - 4 + e) >> 2;
}
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));           // such rows start anywhere on 4 bytes
typedef uint32_t uintx2u __attribute__((ext_vector_type(2), aligned(4)));

// Y[row, :] = sum of the row's partial slots.  Grid (n_heavy, ceil(C / 64), n_out): one block per split
// row, 64-column strip and output tensor (output z reads its partials n_slots*C further into the
// workspace).  Wave w adds slots w, w+4, ... (eight independent loads per step); the four wave sums
// are then added in wave order, so the result is a fixed function of the plan.
template <typename T>
__device__ __forceinline__ void combine_sum_block(const int32_t *__restrict__ hv, const typename Elem<T>::acc_t *__restrict__ ws,
                                                  T *__restrict__ Y, int C, bool accumulate = false) {
    using acc_t = typename Elem<T>::acc_t;
    __shared__ acc_t part[WAVES_PER_BLOCK][WAVE];
    const int row = hv[0], s0 = hv[1], ns = hv[2];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int j = blockIdx.y * WAVE + lane;
    acc_t s = 0;
    if (j < C) {
        const acc_t *col = ws + (size_t)s0 * C + j;
        int k = w;
        for (; k + 7 * WAVES_PER_BLOCK < ns; k += 8 * WAVES_PER_BLOCK) {
            acc_t t[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) t[u] = col[(size_t)(k + u * WAVES_PER_BLOCK) * C];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += t[u];
        }
        for (; k < ns; k += WAVES_PER_BLOCK) s += col[(size_t)k * C];
    }
    part[w][lane] = s;
    __syncthreads();
    if (w == 0 && j < C) {
        acc_t r = part[0][lane];
#pragma unroll
        for (int i = 1; i < WAVES_PER_BLOCK; ++i) r += part[i][lane];
        if (accumulate) r += Elem<T>::ld(Y + (size_t)row * C + j);
        Elem<T>::st(Y + (size_t)row * C + j, r);
    }
}

template <typename T>
__global__ __launch_bounds__(BLOCK) void k_combine_sum(const int32_t *__restrict__ heavy,
                                                       const typename Elem<T>::acc_t *__restrict__ ws, T *__restrict__ Y0,
                                                       T *__restrict__ Y1, int C, size_t ws_stride, int accumulate = 0) {
    combine_sum_block<T>(heavy + 3 * blockIdx.x, ws + (size_t)blockIdx.z * ws_stride, blockIdx.z == 0 ? Y0 : Y1, C, accumulate != 0);
}

// The three sums of the fused backward in one launch, four columns per lane (C a multiple of 256, float partials): grid
// (n_a + n_b, C / 256, 2); blocks x < n_a combine rows of list A into YA (z = 0 only), the others rows of list B into YB0
// (z = 0) and YB1 (z = 1).  Every column is added in the order combine_sum_block uses (wave w takes slots w, w + 4, ...;
// the four wave sums in wave order).
template <typename T> __device__ __forceinline__ void store4(T *p, float4 v);
template <> __device__ __forceinline__ void store4<float>(float *p, float4 v) { *reinterpret_cast<float4 *>(p) = v; }
template <> __device__ __forceinline__ void store4<bf16_t>(bf16_t *p, float4 v) {
    *reinterpret_cast<uint2 *>(p) = make_uint2((uint32_t)f32_to_bf16(v.x) | ((uint32_t)f32_to_bf16(v.y) << 16),
                                               (uint32_t)f32_to_bf16(v.z) | ((uint32_t)f32_to_bf16(v.w) << 16));
}
template <typename T> __device__ __forceinline__ float4 load4(const T *p);
template <> __device__ __forceinline__ float4 load4<float>(const float *p) { return *reinterpret_cast<const float4 *>(p); }
template <> __device__ __forceinline__ float4 load4<bf16_t>(const bf16_t *p) {
    const uint2 x = *reinterpret_cast<const uint2 *>(p);
    return make_float4(__uint_as_float(x.x << 16), __uint_as_float(x.x & 0xffff0000u), __uint_as_float(x.y << 16), __uint_as_float(x.y & 0xffff0000u));
}
// The last one to seven slots of a wavefront (those from k on, in steps of WAVES_PER_BLOCK), all asked for before the first is used: a
// launch that adds up the segments of split rows lasts as long as its longest chain of loads, and one after the other these
// are seven round trips of a chain of eight.  f(place, which of them), in order.  Sixteen before them, where there are as many.  L = 8192, k = 4:
// float32 sums 6.3 -> 5.3 us, bfloat16 6.0 -> 4.7; 16 heads at L = 32768, k = 8 28.7 -> 26.8 and the forward (256 segments in its longest row) 14.4 -> 12.6.
__device__ __forceinline__ int combine_left(int k, int ns) { return k < ns ? (ns - k + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK : 0; }
template <typename F> __device__ __forceinline__ void combine_tail(int left, F &&f) {
    if (left & 4) { f(0, 0); f(1, 1); f(2, 2); f(3, 3); }
    if (left & 2) { f(4, left & 4); f(5, (left & 4) + 1); }
    if (left & 1) f(6, left & 6);
}
template <typename T, bool NARROW = false>
__device__ __forceinline__ void combine_sum_block4(const int32_t *__restrict__ hv, const float *__restrict__ ws, T *__restrict__ Y, int C,
                                                   bool accumulate = false, int strip = -1, const Narrow &nw = Narrow{}) {
    __shared__ float4 part[WAVES_PER_BLOCK][WAVE];
    const int row = hv[0], s0 = hv[1], ns = hv[2];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = ((strip < 0 ? (int)blockIdx.y : strip) * WAVE + lane) * 4;     // strip of 256 columns: the grid's y unless given
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    const float *col = ws + (size_t)s0 * C + j;
    int k = w;
    for (; k + 15 * WAVES_PER_BLOCK < ns; k += 16 * WAVES_PER_BLOCK) {
        float4 t[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) t[u] = *reinterpret_cast<const float4 *>(col + (size_t)(k + u * WAVES_PER_BLOCK) * C);
#pragma unroll
        for (int u = 0; u < 16; ++u) { s.x += t[u].x; s.y += t[u].y; s.z += t[u].z; s.w += t[u].w; }
    }
    if (k + 7 * WAVES_PER_BLOCK < ns) {
        float4 t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = *reinterpret_cast<const float4 *>(col + (size_t)(k + u * WAVES_PER_BLOCK) * C);
#pragma unroll
        for (int u = 0; u < 8; ++u) { s.x += t[u].x; s.y += t[u].y; s.z += t[u].z; s.w += t[u].w; }
        k += 8 * WAVES_PER_BLOCK;
    }
    const int left = combine_left(k, ns);
    float4 t[7];
    combine_tail(left, [&](int u, int nth) { t[u] = *reinterpret_cast<const float4 *>(col + (size_t)(k + nth * WAVES_PER_BLOCK) * C); });
    combine_tail(left, [&](int u, int) { s.x += t[u].x; s.y += t[u].y; s.z += t[u].z; s.w += t[u].w; });
    part[w][lane] = s;
    __syncthreads();
    if (w == 0) {
        float4 r = part[0][lane];
#pragma unroll
        for (int i = 1; i < WAVES_PER_BLOCK; ++i) { r.x += part[i][lane].x; r.y += part[i][lane].y; r.z += part[i][lane].z; r.w += part[i][lane].w; }
        if constexpr (NARROW) {                                   // 64 columns of the partials per head, d of the result
            const int head = j >> 6, col = j & 63;
            T *const at = Y + (size_t)row * (nw.heads * nw.d) + head * nw.d + col;
            const float x[4] = {r.x, r.y, r.z, r.w};
            for (int e = 0; e < 4; ++e)
                if (head < nw.heads && col + e < nw.d) Elem<T>::st(at + e, x[e]);
            return;
        }
        if (accumulate) {
            const float4 y = load4<T>(Y + (size_t)row * C + j);
            r.x += y.x; r.y += y.y; r.z += y.z; r.w += y.w;
        }
        store4<T>(Y + (size_t)row * C + j, r);
    }
}
template <typename T, bool NARROW = false>
__global__ __launch_bounds__(BLOCK) void k_combine_sum3(const int32_t *__restrict__ heavy_a, int n_a, const float *__restrict__ ws_a,
                                                           T *__restrict__ YA, const int32_t *__restrict__ heavy_b,
                                                           const float *__restrict__ ws_b, T *__restrict__ YB0, T *__restrict__ YB1, int C,
                                                           size_t ws_stride_b, Narrow nw) {
    if ((int)blockIdx.x < n_a) {
        if (blockIdx.z == 0) combine_sum_block4<T, NARROW>(heavy_a + 3 * blockIdx.x, ws_a, YA, C, false, -1, nw);
    } else {
        combine_sum_block4<T, NARROW>(heavy_b + 3 * (blockIdx.x - n_a), ws_b + (size_t)blockIdx.z * ws_stride_b, blockIdx.z == 0 ? YB0 : YB1, C,
                                      false, -1, nw);
    }
}

// k_combine_sum for the specialised shapes (float partials, C a multiple of 256): grid (n_heavy, C / 256, n_out)
template <typename T>
__global__ __launch_bounds__(BLOCK) void k_combine_sum_v4(const int32_t *__restrict__ heavy, const float *__restrict__ ws, T *__restrict__ Y0,
                                                          T *__restrict__ Y1, int C, size_t ws_stride, int accumulate = 0) {
    combine_sum_block4<T>(heavy + 3 * blockIdx.x, ws + (size_t)blockIdx.z * ws_stride, blockIdx.z == 0 ? Y0 : Y1, C, accumulate != 0);
}

// dB[eid[p], d] = sum_h dy[eid[p], h] * A[row, h, d]      (graphop_kernel.cu:79-94)
template <typename T>
__global__ __launch_bounds__(BLOCK) void k_nme_dB_generic(bpt_plan P, const T *__restrict__ A, const T *__restrict__ dy,
                                                          T *__restrict__ dB, int H, int D) {
    using acc_t = typename Elem<T>::acc_t;
    Item it;
    if (!fetch_item(P, it)) return;
    const int lane = threadIdx.x & 63;
    const T *a = A + (size_t)it.row * H * D;
    for (int p = it.begin; p < it.end; ++p) {
        const int e = P.eid[p];
        for (int dd = lane; dd < D; dd += WAVE) {
            acc_t s = 0;
            for (int h = 0; h < H; ++h) s += (acc_t)Elem<T>::ld(dy + (size_t)e * H + h) * (acc_t)Elem<T>::ld(a + h * D + dd);
            Elem<T>::st(dB + (size_t)e * D + dd, s);
        }
    }
}

// Row softmax.  NW == 1: one wavefront per whole-row item (segments of split rows exit);
// NW == WAVES_PER_BLOCK: one block per split row (grid = n_heavy).
template <typename T, int NW>
__global__ __launch_bounds__(BLOCK) void k_softmax_fwd(bpt_plan P, const T *__restrict__ x, T *__restrict__ y, int H) {
    using acc_t = typename Elem<T>::acc_t;
    __shared__ acc_t smem[WAVES_PER_BLOCK];
    int begin, end, tid;
    if (NW == 1) {
        Item it;
        if (!fetch_item(P, it) || it.slot >= 0) return;
        begin = it.begin; end = it.end; tid = threadIdx.x & 63;
    } else {
        const int row = P.heavy[3 * blockIdx.x];
        begin = P.rowptr[row]; end = P.rowptr[row + 1]; tid = threadIdx.x;
    }
    constexpr int NT = NW * WAVE;
    for (int h = 0; h < H; ++h) {
        acc_t m = (acc_t)-1e9;
        for (int p = begin + tid; p < end; p += NT) {
            const acc_t v = Elem<T>::ld(x + (size_t)P.eid[p] * H + h);
            m = v > m ? v : m;
        }
        m = group_reduce<acc_t, NW, true>(m, smem);
        acc_t s = 0;
        for (int p = begin + tid; p < end; p += NT) s += exp_acc((acc_t)Elem<T>::ld(x + (size_t)P.eid[p] * H + h) - m);
        s = group_reduce<acc_t, NW, false>(s, smem);
        for (int p = begin + tid; p < end; p += NT) {
            const size_t o = (size_t)P.eid[p] * H + h;
            Elem<T>::st(y + o, exp_acc((acc_t)Elem<T>::ld(x + o) - m) / s);
        }
    }
}

// dx = dy*y - (sum_row dy*y) * y      (graphop_kernel.cu:208-230)
template <typename T, int NW>
__global__ __launch_bounds__(BLOCK) void k_softmax_bwd(bpt_plan P, const T *__restrict__ y, const T *__restrict__ dy,
                                                       T *__restrict__ dx, int H) {
    using acc_t = typename Elem<T>::acc_t;
    __shared__ acc_t smem[WAVES_PER_BLOCK];
    int begin, end, tid;
    if (NW == 1) {
        Item it;
        if (!fetch_item(P, it) || it.slot >= 0) return;
        begin = it.begin; end = it.end; tid = threadIdx.x & 63;
    } else {
        const int row = P.heavy[3 * blockIdx.x];
        begin = P.rowptr[row]; end = P.rowptr[row + 1]; tid = threadIdx.x;
    }
    constexpr int NT = NW * WAVE;
    for (int h = 0; h < H; ++h) {
        acc_t s = 0;
        for (int p = begin + tid; p < end; p += NT) {
            const size_t o = (size_t)P.eid[p] * H + h;
            s += (acc_t)Elem<T>::ld(dy + o) * (acc_t)Elem<T>::ld(y + o);
        }
        s = group_reduce<acc_t, NW, false>(s, smem);
        for (int p = begin + tid; p < end; p += NT) {
            const size_t o = (size_t)P.eid[p] * H + h;
            const acc_t yv = Elem<T>::ld(y + o);
            Elem<T>::st(dx + o, (acc_t)Elem<T>::ld(dy + o) * yv - s * yv);
        }
    }
}

// Row softmax with the heads side by side: lane l handles head l % H of edge slot l / H, so a wavefront reads
// 64 / H whole (E, H) rows per step, for up to 64 heads; lanes past the last whole row have none.  One wavefront per item.  Rows of up
// to SM_CACHE steps keep their values in registers and read memory once; longer rows re-read.  Loads are issued SM_CACHE at a time.
// Heads that do not divide 64 ran the kernels above, a pass over the row for every head: 6 heads float32, L = 8192, k = 4, all launches,
// forward 249 -> 30 us, backward 350 -> 39.
constexpr int SM_CACHE = 8;

// reduction over the threads of a block that share a head, l % H: first inside each wavefront, then over LDS
template <typename A, int NW, bool IS_MAX> __device__ __forceinline__ A head_reduce(A x, int H, int h, A *smem) {
    if ((H & (H - 1)) == 0) {
        for (int off = H; off < WAVE; off <<= 1) {
            const A o = __shfl_xor(x, off);
            x = IS_MAX ? (x > o ? x : o) : x + o;
        }
    } else {                                                      // the upper half of the n slots onto the lower one, until one is left
        const int lane = threadIdx.x & 63, slot = lane / H;
        for (int n = WAVE / H; n > 1; n = (n + 1) >> 1) {
            const int half = (n + 1) >> 1;
            const A o = __shfl(x, min(lane + half * H, WAVE - 1));
            if (slot + half < n) x = IS_MAX ? (x > o ? x : o) : x + o;
        }
        x = __shfl(x, h);
    }
    if (NW == 1) return x;
    const int w = threadIdx.x >> 6;
    __syncthreads();                       // smem may still be read from the previous reduction
    if ((int)(threadIdx.x & 63) < H) smem[w * WAVE + h] = x;
    __syncthreads();
    A r = smem[h];
    for (int i = 1; i < NW; ++i) r = IS_MAX ? (r > smem[i * WAVE + h] ? r : smem[i * WAVE + h]) : r + smem[i * WAVE + h];
    return r;
}

// WHOLE: split rows are taken whole by the first `whole` workgroups of the launch over the items, one each, and the items that are
// segments do nothing: no second and third launch, each a chain of loads of its own, and nothing kept per segment (softmax_whole_rows
// says where).
constexpr int SM_BLOCK = 512, SM_WAVES = SM_BLOCK / WAVE;
template <bool WHOLE> constexpr int sm_block() { return WHOLE ? SM_BLOCK : BLOCK; }
__device__ __forceinline__ bool split_row(const bpt_plan &P, int i, int &begin, int &end) {
    if (i >= (int)P.n_heavy) return false;                        // (their number is rounded up to a multiple of 8)
    const int row = P.heavy[3 * i];
    begin = P.rowptr[row];
    end = P.rowptr[row + 1];
    return true;
}

// seg_slot: NULL = whole rows only (segments of split rows are skipped); else it receives the item's slot (-1 = whole row)
__device__ __forceinline__ bool softmax_range(const bpt_plan &P, int &begin, int &end, int *seg_slot, int waves_per_block = WAVES_PER_BLOCK, int skip = 0) {
    Item it;
    if (!fetch_item(P, it, waves_per_block, skip) || (it.slot >= 0 && !seg_slot)) return false;
    begin = it.begin; end = it.end;
    if (seg_slot) *seg_slot = it.slot;
    return true;
}

// NW wavefronts share a row: SM_WAVES for a split row taken whole, else 1 an item
template <typename T, int NW>
__device__ __forceinline__ void softmax_fwd_heads(const bpt_plan &P, int begin, int end, int seg_slot, const T *__restrict__ x, T *__restrict__ y, int H,
                                                  typename Elem<T>::acc_t *__restrict__ seg, typename Elem<T>::acc_t *smem) {
    using acc_t = typename Elem<T>::acc_t;
    const int lane = threadIdx.x & 63, h = lane % H, slot = lane / H, per = WAVE / H, nslots = NW * per;
    const int first = slot < per ? begin + (NW > 1 ? (int)(threadIdx.x >> 6) * per : 0) + slot : end;         // (the lanes that are left over: no edges)
    const bool cached = end - begin <= SM_CACHE * nslots;
    acc_t vc[SM_CACHE];
    size_t oc[SM_CACHE];
#pragma unroll
    for (int u = 0; u < SM_CACHE; ++u) { vc[u] = (acc_t)-INFINITY; oc[u] = (size_t)-1; }    // threads past a short row's end
    acc_t m = (acc_t)-1e9;
    for (int p0 = first; p0 < end; p0 += SM_CACHE * nslots) {
        int e[SM_CACHE];
#pragma unroll
        for (int u = 0; u < SM_CACHE; ++u) { const int p = p0 + u * nslots; e[u] = p < end ? P.eid[p] : -1; }
#pragma unroll
        for (int u = 0; u < SM_CACHE; ++u) {
            oc[u] = (size_t)(e[u] < 0 ? 0 : e[u]) * H + h;
            vc[u] = e[u] < 0 ? (acc_t)-INFINITY : (acc_t)Elem<T>::ld(x + oc[u]);
            m = vc[u] > m ? vc[u] : m;
            if (e[u] < 0) oc[u] = (size_t)-1;
        }
    }
    m = head_reduce<acc_t, NW, true>(m, H, h, smem);
    acc_t s = 0;
    if (cached) {
#pragma unroll
        for (int u = 0; u < SM_CACHE; ++u) { vc[u] = exp_acc(vc[u] - m); s += vc[u]; }      // exp(-inf) = 0 for the empty slots
    } else {
        for (int p0 = first; p0 < end; p0 += SM_CACHE * nslots) {
            int e[SM_CACHE];
#pragma unroll
            for (int u = 0; u < SM_CACHE; ++u) { const int p = p0 + u * nslots; e[u] = p < end ? P.eid[p] : -1; }
            acc_t v[SM_CACHE];
#pragma unroll
            for (int u = 0; u < SM_CACHE; ++u) v[u] = e[u] < 0 ? (acc_t)-INFINITY : (acc_t)Elem<T>::ld(x + (size_t)e[u] * H + h);
#pragma unroll
            for (int u = 0; u < SM_CACHE; ++u) s += exp_acc(v[u] - m);
        }
    }
    s = head_reduce<acc_t, NW, false>(s, H, h, smem);
    if (NW == 1 && seg_slot >= 0) {
        // a segment of a split row: only its (m, s); k_softmax_seg_rows forms the row's of them and k_softmax_fwd_seg_finish writes y
        if (slot == 0) { seg[((size_t)seg_slot * H + h) * 2] = m; seg[((size_t)seg_slot * H + h) * 2 + 1] = s; }
        return;
    }
    if (cached) {
#pragma unroll
        for (int u = 0; u < SM_CACHE; ++u)
            if (oc[u] != (size_t)-1) Elem<T>::st(y + oc[u], vc[u] / s);
    } else {
        for (int p0 = first; p0 < end; p0 += SM_CACHE * nslots) {
            int e[SM_CACHE];
#pragma unroll
            for (int u = 0; u < SM_CACHE; ++u) { const int p = p0 + u * nslots; e[u] = p < end ? P.eid[p] : -1; }
            acc_t v[SM_CACHE];
#pragma unroll
            for (int u = 0; u < SM_CACHE; ++u) v[u] = e[u] < 0 ? (acc_t)0 : (acc_t)Elem<T>::ld(x + (size_t)e[u] * H + h);
#pragma unroll
            for (int u = 0; u < SM_CACHE; ++u)
                if (e[u] >= 0) Elem<T>::st(y + (size_t)e[u] * H + h, exp_acc(v[u] - m) / s);
        }
    }
}
template <typename T, bool WHOLE>
__global__ __launch_bounds__(sm_block<WHOLE>()) void k_softmax_fwd_heads(bpt_plan P, const T *__restrict__ x, T *__restrict__ y, int H,
                                                                typename Elem<T>::acc_t *__restrict__ seg, int whole) {
    int begin, end, slot = -1;
    if constexpr (WHOLE) {
        __shared__ typename Elem<T>::acc_t smem[SM_WAVES * WAVE];
        if ((int)blockIdx.x < whole) {
            if (split_row(P, blockIdx.x, begin, end)) softmax_fwd_heads<T, SM_WAVES>(P, begin, end, -1, x, y, H, nullptr, smem);
        } else if (softmax_range(P, begin, end, nullptr, SM_WAVES, whole)) {
            softmax_fwd_heads<T, 1>(P, begin, end, -1, x, y, H, nullptr, nullptr);
        }
    } else if (softmax_range(P, begin, end, seg ? &slot : nullptr)) {
        softmax_fwd_heads<T, 1>(P, begin, end, slot, x, y, H, seg, nullptr);
    }
}

template <typename T, int NW>
__device__ __forceinline__ void softmax_bwd_heads(const bpt_plan &P, int begin, int end, int seg_slot, const T *__restrict__ y, const T *__restrict__ dy,
                                                  T *__restrict__ dx, int H, typename Elem<T>::acc_t *__restrict__ seg, typename Elem<T>::acc_t *smem) {
    using acc_t = typename Elem<T>::acc_t;
    const int lane = threadIdx.x & 63, h = lane % H, slot = lane / H, per = WAVE / H, nslots = NW * per;
    const int first = slot < per ? begin + (NW > 1 ? (int)(threadIdx.x >> 6) * per : 0) + slot : end;         // (the lanes that are left over: no edges)
    const bool cached = end - begin <= SM_CACHE * nslots;
    acc_t yc[SM_CACHE], dc[SM_CACHE];
    size_t oc[SM_CACHE];
#pragma unroll
    for (int u = 0; u < SM_CACHE; ++u) { yc[u] = 0; dc[u] = 0; oc[u] = (size_t)-1; }
    acc_t s = 0;
    for (int p0 = first; p0 < end; p0 += SM_CACHE * nslots) {
        int e[SM_CACHE];
#pragma unroll
        for (int u = 0; u < SM_CACHE; ++u) { const int p = p0 + u * nslots; e[u] = p < end ? P.eid[p] : -1; }
#pragma unroll
        for (int u = 0; u < SM_CACHE; ++u) {
            oc[u] = (size_t)(e[u] < 0 ? 0 : e[u]) * H + h;
            yc[u] = e[u] < 0 ? (acc_t)0 : (acc_t)Elem<T>::ld(y + oc[u]);
            dc[u] = e[u] < 0 ? (acc_t)0 : (acc_t)Elem<T>::ld(dy + oc[u]);
            if (e[u] < 0) oc[u] = (size_t)-1;
        }
#pragma unroll
        for (int u = 0; u < SM_CACHE; ++u) s += dc[u] * yc[u];
    }
    s = head_reduce<acc_t, NW, false>(s, H, h, smem);
    if (NW == 1 && seg_slot >= 0) {
        // a segment of a split row: only its part of sum(dy * y); k_softmax_seg_rows adds the parts up and
        // k_softmax_bwd_seg_finish writes dx
        if (slot == 0) seg[(size_t)seg_slot * H + h] = s;
        return;
    }
    if (cached) {
#pragma unroll
        for (int u = 0; u < SM_CACHE; ++u)
            if (oc[u] != (size_t)-1) Elem<T>::st(dx + oc[u], dc[u] * yc[u] - s * yc[u]);
    } else {
        for (int p0 = first; p0 < end; p0 += SM_CACHE * nslots) {
            int e[SM_CACHE];
#pragma unroll
            for (int u = 0; u < SM_CACHE; ++u) { const int p = p0 + u * nslots; e[u] = p < end ? P.eid[p] : -1; }
            acc_t yv[SM_CACHE], dv[SM_CACHE];
#pragma unroll
            for (int u = 0; u < SM_CACHE; ++u) {
                const size_t o = (size_t)(e[u] < 0 ? 0 : e[u]) * H + h;
                yv[u] = e[u] < 0 ? (acc_t)0 : (acc_t)Elem<T>::ld(y + o);
                dv[u] = e[u] < 0 ? (acc_t)0 : (acc_t)Elem<T>::ld(dy + o);
            }
#pragma unroll
            for (int u = 0; u < SM_CACHE; ++u)
                if (e[u] >= 0) Elem<T>::st(dx + (size_t)e[u] * H + h, dv[u] * yv[u] - s * yv[u]);
        }
    }
}
template <typename T, bool WHOLE>
__global__ __launch_bounds__(sm_block<WHOLE>()) void k_softmax_bwd_heads(bpt_plan P, const T *__restrict__ y, const T *__restrict__ dy, T *__restrict__ dx,
                                                                int H, typename Elem<T>::acc_t *__restrict__ seg, int whole) {
    int begin, end, slot = -1;
    if constexpr (WHOLE) {
        __shared__ typename Elem<T>::acc_t smem[SM_WAVES * WAVE];
        if ((int)blockIdx.x < whole) {
            if (split_row(P, blockIdx.x, begin, end)) softmax_bwd_heads<T, SM_WAVES>(P, begin, end, -1, y, dy, dx, H, nullptr, smem);
        } else if (softmax_range(P, begin, end, nullptr, SM_WAVES, whole)) {
            softmax_bwd_heads<T, 1>(P, begin, end, -1, y, dy, dx, H, nullptr, nullptr);
        }
    } else if (softmax_range(P, begin, end, seg ? &slot : nullptr)) {
        softmax_bwd_heads<T, 1>(P, begin, end, slot, y, dy, dx, H, seg, nullptr);
    }
}

// Split rows of the softmax, second step: one block per split row.  Forward (PAIR): the segments' (m_i, s_i) are replaced by the
// row's, M = max(-1e9, m_i) and S = sum s_i exp(m_i - M); backward: the segments' partial sums are replaced by their total.  A
// lane handles head l % H of every n-th slot.
template <typename A, bool PAIR>
__global__ __launch_bounds__(BLOCK) void k_softmax_seg_rows(const int32_t *__restrict__ heavy, A *__restrict__ seg, int H) {
    __shared__ A smem[WAVES_PER_BLOCK * WAVE];
    const int s0 = heavy[3 * blockIdx.x + 1], ns = heavy[3 * blockIdx.x + 2];
    const int lane = threadIdx.x & 63, per = WAVE / H, h = lane % H, j0 = lane / H < per ? (int)(threadIdx.x >> 6) * per + lane / H : ns, nj = WAVES_PER_BLOCK * per;
    constexpr int ST = PAIR ? 2 : 1;
    if constexpr (PAIR) {
        A m = (A)-1e9;
        for (int j = j0; j < ns; j += nj) { const A v = seg[((size_t)(s0 + j) * H + h) * ST]; m = v > m ? v : m; }
        m = head_reduce<A, WAVES_PER_BLOCK, true>(m, H, h, smem);
        A s = 0;
        for (int j = j0; j < ns; j += nj) s += seg[((size_t)(s0 + j) * H + h) * ST + 1] * exp_acc(seg[((size_t)(s0 + j) * H + h) * ST] - m);
        s = head_reduce<A, WAVES_PER_BLOCK, false>(s, H, h, smem);
        for (int j = j0; j < ns; j += nj) {
            A *q = seg + ((size_t)(s0 + j) * H + h) * ST;
            q[0] = m;
            q[1] = s;
        }
    } else {
        A s = 0;
        for (int j = j0; j < ns; j += nj) s += seg[(size_t)(s0 + j) * H + h];
        s = head_reduce<A, WAVES_PER_BLOCK, false>(s, H, h, smem);
        for (int j = j0; j < ns; j += nj) seg[(size_t)(s0 + j) * H + h] = s;
    }
}

// Third step, one wavefront per item, segments only.  Forward: x is read again and y = exp(x - M) / S, rounded once, as for a whole row (a
// segment's exp(x - m) kept in y and scaled here would be rounded twice: bfloat16 results off by 7.5e-3 instead of 3.8e-3).
template <typename T>
__global__ __launch_bounds__(BLOCK) void k_softmax_fwd_seg_finish(bpt_plan P, const T *__restrict__ x, T *__restrict__ y, int H,
                                                                  const typename Elem<T>::acc_t *__restrict__ seg) {
    using acc_t = typename Elem<T>::acc_t;
    Item it;
    if (!fetch_item(P, it) || it.slot < 0) return;
    const int tid = threadIdx.x & 63, h = tid % H, nslots = WAVE / H;
    if (tid / H >= nslots) return;
    const acc_t m = seg[((size_t)it.slot * H + h) * 2], s = seg[((size_t)it.slot * H + h) * 2 + 1];
    for (int p = it.begin + tid / H; p < it.end; p += nslots) {
        const size_t o = (size_t)P.eid[p] * H + h;
        Elem<T>::st(y + o, exp_acc((acc_t)Elem<T>::ld(x + o) - m) / s);
    }
}

// Backward: dx = y * (dy - total) on the segments.
template <typename T>
__global__ __launch_bounds__(BLOCK) void k_softmax_bwd_seg_finish(bpt_plan P, const T *__restrict__ y, const T *__restrict__ dy, T *__restrict__ dx,
                                                                  int H, const typename Elem<T>::acc_t *__restrict__ seg) {
    using acc_t = typename Elem<T>::acc_t;
    Item it;
    if (!fetch_item(P, it) || it.slot < 0) return;
    const int tid = threadIdx.x & 63, h = tid % H, nslots = WAVE / H;
    if (tid / H >= nslots) return;
    const acc_t t = seg[(size_t)it.slot * H + h];
    for (int p = it.begin + tid / H; p < it.end; p += nslots) {
        const size_t o = (size_t)P.eid[p] * H + h;
        const acc_t yv = (acc_t)Elem<T>::ld(y + o);
        Elem<T>::st(dx + o, yv * ((acc_t)Elem<T>::ld(dy + o) - t));
    }
}

// The same for 4, 8 or 16 heads in float32 or bfloat16 with four heads a lane (16 bytes of a float32 record): 8 Q lanes an item,
// Q = H / 4, so a wavefront works on 8 / Q items at a time and an item of 64 edges is read with eight loads in flight a lane.  The
// kernels above give every item a wavefront, in 2.1 rounds of wavefronts at L = 8192, k = 4, and three memory instructions to every
// 64 / H slots of a row of 5 as of 64.  Two launches: the first finishes whole rows and leaves (m, s) of the segments of split rows, the
// second forms a split row's result from its segments and its edges, several blocks a row.  8 heads, 430 k edges, 16 383 rows:
// forward 20.2 + 4.4 + 9.2 -> 15.3 + 8.0 us, backward 19.1 + 4.9 + 11.3 -> 19.8 + 8.0: what is left are the 128-byte lines around the
// 32-byte records (208 k lines a tensor where 108 k would hold them: an in-row's edge ids are neighbours by twos).
template <typename T> struct Quad;                    // four neighbouring heads
template <> struct Quad<float> {
    static __device__ __forceinline__ void ld(const float *p, float (&v)[4]) {
        const float4 x = *reinterpret_cast<const float4 *>(p);
        v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
    }
    static __device__ __forceinline__ void st(float *p, const float (&v)[4]) { *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]); }
};
template <> struct Quad<bf16_t> {
    static __device__ __forceinline__ void ld(const bf16_t *p, float (&v)[4]) {
        const uint2 x = *reinterpret_cast<const uint2 *>(p);
        v[0] = __uint_as_float(x.x << 16); v[1] = __uint_as_float(x.x & 0xffff0000u);
        v[2] = __uint_as_float(x.y << 16); v[3] = __uint_as_float(x.y & 0xffff0000u);
    }
    static __device__ __forceinline__ void st(bf16_t *p, const float (&v)[4]) {
        *reinterpret_cast<uint2 *>(p) = make_uint2((uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16),
                                                   (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16));
    }
};

// over the slots of an item: the 8 Q lanes that share it, those of one quad of heads (or LANES)
template <int Q, bool IS_MAX, int LANES = 8 * Q> __device__ __forceinline__ void quad_reduce(float (&v)[4]) {
#pragma unroll
    for (int off = Q; off < LANES; off <<= 1)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float o = __shfl_xor(v[i], off);
            v[i] = IS_MAX ? (v[i] > o ? v[i] : o) : v[i] + o;
        }
}
// over all threads of a workgroup of SM_WAVES wavefronts; part: SM_WAVES x 4 Q floats that nothing else uses
template <int Q, bool IS_MAX> __device__ __forceinline__ void quad_reduce_block(float (&v)[4], float *part) {
    quad_reduce<Q, IS_MAX, WAVE>(v);
    const int lane = threadIdx.x & 63, q4 = 4 * (lane % Q);
    if (lane < Q)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[(threadIdx.x >> 6) * 4 * Q + q4 + i] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = part[q4 + i];
    for (int w = 1; w < SM_WAVES; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float o = part[w * 4 * Q + q4 + i];
            v[i] = IS_MAX ? (v[i] > o ? v[i] : o) : v[i] + o;
        }
}

// an item for every 8 Q lanes: eight slots a load, QUAD_U loads in flight (64 slots: an item of the usual length at once)
constexpr int QUAD_SLOTS = 8, QUAD_U = 8;
template <int Q, bool WHOLE> __device__ __forceinline__ bool fetch_quad_item(const bpt_plan &P, Item &it, int whole) {
    const int64_t w = ((int64_t)xcd_contiguous_block(WHOLE ? whole : 0) * sm_block<WHOLE>() + threadIdx.x) / (QUAD_SLOTS * Q);
    if (w >= P.n_items) return false;
    const int4 v = reinterpret_cast<const int4 *>(P.items)[w];
    it = Item{v.x, v.y, v.z, v.w};
    return !WHOLE || it.slot < 0;
}
// ids of this lane's slots p, p + step, ...: -1 past the end of the range
template <int U> __device__ __forceinline__ void quad_eids(const bpt_plan &P, int p, int step, int end, int (&e)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) e[u] = p + u * step < end ? P.eid[p + u * step] : -1;
}

// a split row, by a workgroup: what its threads' loads hold at once is read once, a longer row twice (max and sum of a thread together)
template <typename T, int Q> __device__ __forceinline__ void softmax_fwd_whole_row(const bpt_plan &P, const T *__restrict__ x, T *__restrict__ y) {
    constexpr int H = 4 * Q, SL = SM_BLOCK / Q, U = QUAD_U;
    __shared__ float part[2][SM_WAVES * H];
    int begin, end, e[U];
    if (!split_row(P, blockIdx.x, begin, end)) return;
    const int q4 = 4 * ((int)threadIdx.x % Q), p0 = begin + (int)threadIdx.x / Q;
    const bool once = end - begin <= U * SL;
    float v[U][4], m[4] = {-1e9f, -1e9f, -1e9f, -1e9f}, s[4] = {0.f, 0.f, 0.f, 0.f};
    auto load = [&](int p) {
        quad_eids<U>(P, p, SL, end, e);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            v[u][0] = v[u][1] = v[u][2] = v[u][3] = -INFINITY;
            if (e[u] >= 0) Quad<T>::ld(x + (size_t)e[u] * H + q4, v[u]);
        }
    };
    for (int p = p0; p < end || p == p0; p += U * SL) {
        load(p);
        float mn[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            mn[i] = m[i];
#pragma unroll
            for (int u = 0; u < U; ++u) mn[i] = v[u][i] > mn[i] ? v[u][i] : mn[i];
            if (!once) {
                s[i] *= expf(m[i] - mn[i]);
#pragma unroll
                for (int u = 0; u < U; ++u) s[i] += expf(v[u][i] - mn[i]);
            }
            m[i] = mn[i];
        }
    }
    float M[4] = {m[0], m[1], m[2], m[3]};
    quad_reduce_block<Q, true>(M, part[0]);
    if (once) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) { v[u][i] = expf(v[u][i] - M[i]); s[i] += v[u][i]; }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] *= expf(m[i] - M[i]);
    }
    quad_reduce_block<Q, false>(s, part[1]);
    for (int p = p0; p < end; p += U * SL) {
        if (!once) {
            load(p);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[u][i] = expf(v[u][i] - M[i]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (e[u] < 0) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[u][i] = v[u][i] / s[i];
            Quad<T>::st(y + (size_t)e[u] * H + q4, v[u]);
        }
    }
}

template <typename T, int Q, bool WHOLE>
__global__ __launch_bounds__(sm_block<WHOLE>()) void k_softmax_fwd_quads(bpt_plan P, const T *__restrict__ x, T *__restrict__ y, float *__restrict__ seg, int whole) {
    constexpr int H = 4 * Q, SL = QUAD_SLOTS, U = QUAD_U;
    if constexpr (WHOLE) {
        if ((int)blockIdx.x < whole) {
            softmax_fwd_whole_row<T, Q>(P, x, y);
            return;
        }
    }
    Item it;
    if (!fetch_quad_item<Q, WHOLE>(P, it, whole)) return;
    const int lane = threadIdx.x % (SL * Q), q4 = 4 * (lane % Q), p0 = it.begin + lane / Q;
    const bool once = it.end - it.begin <= U * SL;
    int e[U];
    float v[U][4], m[4] = {-1e9f, -1e9f, -1e9f, -1e9f}, s[4] = {0.f, 0.f, 0.f, 0.f};
    auto load = [&](int p) {
        quad_eids<U>(P, p, SL, it.end, e);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            v[u][0] = v[u][1] = v[u][2] = v[u][3] = -INFINITY;
            if (e[u] >= 0) Quad<T>::ld(x + (size_t)e[u] * H + q4, v[u]);
        }
    };
    for (int p = p0; p < it.end || p == p0; p += U * SL) {
        load(p);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) m[i] = v[u][i] > m[i] ? v[u][i] : m[i];
    }
    quad_reduce<Q, true>(m);
    for (int p = p0; p < it.end || p == p0; p += U * SL) {
        if (!once) load(p);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) { v[u][i] = expf(v[u][i] - m[i]); s[i] += v[u][i]; }       // exp(-inf) = 0 for the empty slots
    }
    quad_reduce<Q, false>(s);
    if (it.slot >= 0) {
        if (lane < Q) {
            float *o = seg + ((size_t)it.slot * H + q4) * 2;
#pragma unroll
            for (int i = 0; i < 4; ++i) { o[2 * i] = m[i]; o[2 * i + 1] = s[i]; }
        }
        return;
    }
    for (int p = p0; p < it.end; p += U * SL) {
        if (!once) {
            load(p);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[u][i] = expf(v[u][i] - m[i]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (e[u] < 0) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[u][i] = v[u][i] / s[i];
            Quad<T>::st(y + (size_t)e[u] * H + q4, v[u]);
        }
    }
}

template <typename T, int Q>
__device__ __forceinline__ void softmax_bwd_whole_row(const bpt_plan &P, const T *__restrict__ y, const T *__restrict__ dy, T *__restrict__ dx) {
    constexpr int H = 4 * Q, SL = SM_BLOCK / Q, U = QUAD_U;
    __shared__ float part[SM_WAVES * H];
    int begin, end, e[U];
    if (!split_row(P, blockIdx.x, begin, end)) return;
    const int q4 = 4 * ((int)threadIdx.x % Q), p0 = begin + (int)threadIdx.x / Q;
    const bool once = end - begin <= U * SL;
    float yv[U][4], dv[U][4], s[4] = {0.f, 0.f, 0.f, 0.f};
    auto load = [&](int p) {
        quad_eids<U>(P, p, SL, end, e);
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int i = 0; i < 4; ++i) yv[u][i] = dv[u][i] = 0.f;
            if (e[u] >= 0) {
                Quad<T>::ld(y + (size_t)e[u] * H + q4, yv[u]);
                Quad<T>::ld(dy + (size_t)e[u] * H + q4, dv[u]);
            }
        }
    };
    for (int p = p0; p < end || p == p0; p += U * SL) {
        load(p);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] += dv[u][i] * yv[u][i];
    }
    quad_reduce_block<Q, false>(s, part);
    for (int p = p0; p < end; p += U * SL) {
        if (!once) load(p);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (e[u] < 0) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) dv[u][i] = dv[u][i] * yv[u][i] - s[i] * yv[u][i];
            Quad<T>::st(dx + (size_t)e[u] * H + q4, dv[u]);
        }
    }
}

template <typename T, int Q, bool WHOLE>
__global__ __launch_bounds__(sm_block<WHOLE>()) void k_softmax_bwd_quads(bpt_plan P, const T *__restrict__ y, const T *__restrict__ dy, T *__restrict__ dx,
                                                                float *__restrict__ seg, int whole) {
    constexpr int H = 4 * Q, SL = QUAD_SLOTS, U = QUAD_U;
    if constexpr (WHOLE) {
        if ((int)blockIdx.x < whole) {
            softmax_bwd_whole_row<T, Q>(P, y, dy, dx);
            return;
        }
    }
    Item it;
    if (!fetch_quad_item<Q, WHOLE>(P, it, whole)) return;
    const int lane = threadIdx.x % (SL * Q), q4 = 4 * (lane % Q), p0 = it.begin + lane / Q;
    const bool once = it.end - it.begin <= U * SL;
    int e[U];
    float yv[U][4], dv[U][4], s[4] = {0.f, 0.f, 0.f, 0.f};
    auto load = [&](int p) {
        quad_eids<U>(P, p, SL, it.end, e);
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int i = 0; i < 4; ++i) yv[u][i] = dv[u][i] = 0.f;
            if (e[u] >= 0) {
                Quad<T>::ld(y + (size_t)e[u] * H + q4, yv[u]);
                Quad<T>::ld(dy + (size_t)e[u] * H + q4, dv[u]);
            }
        }
    };
    for (int p = p0; p < it.end || p == p0; p += U * SL) {
        load(p);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] += dv[u][i] * yv[u][i];
    }
    quad_reduce<Q, false>(s);
    if (it.slot >= 0) {
        if (lane < Q) {
#pragma unroll
            for (int i = 0; i < 4; ++i) seg[(size_t)it.slot * H + q4 + i] = s[i];
        }
        return;
    }
    for (int p = p0; p < it.end; p += U * SL) {
        if (!once) load(p);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (e[u] < 0) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) dv[u][i] = dv[u][i] * yv[u][i] - s[i] * yv[u][i];
            Quad<T>::st(dx + (size_t)e[u] * H + q4, dv[u]);
        }
    }
}

// Split rows, second launch: block (i, j) is the j-th of gridDim.y blocks of split row i.  Every block reduces the row's segments
// by itself (16 bytes a segment and head at most: they come from the L2), then writes its share of the row's edges.  (Its first edges asked for
// ahead of the sums: 7.7 -> 7.0 us forward and 7.8 -> 7.4 backward at L = 8192, k = 4, which has 127 split rows, but 66 -> 76 and 45 -> 52 at a
// window of 200, L = 4096, which has 4033.)
template <typename T, int Q, bool FWD>
__global__ __launch_bounds__(BLOCK) void k_softmax_split_quads(bpt_plan P, const T *__restrict__ x, const T *__restrict__ dy, T *__restrict__ y,
                                                               const float *__restrict__ seg) {
    constexpr int H = 4 * Q, SL = BLOCK / Q, U = 4;               // slots of a load of the block
    __shared__ float smem[WAVES_PER_BLOCK * WAVE];
    __shared__ float of_head[2][H];
    const int row = P.heavy[3 * blockIdx.x], s0 = P.heavy[3 * blockIdx.x + 1], ns = P.heavy[3 * blockIdx.x + 2];
    const int h = threadIdx.x % H, j0 = threadIdx.x / H, nj = BLOCK / H;
    const int begin = P.rowptr[row], deg = P.rowptr[row + 1] - begin;
    const int per = (deg + (int)gridDim.y - 1) / (int)gridDim.y, first = begin + (int)blockIdx.y * per, end = min(first + per, begin + deg);
    if constexpr (FWD) {
        float m = -1e9f, s = 0.f;
        for (int j = j0; j < ns; j += nj) { const float v = seg[((size_t)(s0 + j) * H + h) * 2]; m = v > m ? v : m; }
        m = head_reduce<float, WAVES_PER_BLOCK, true>(m, H, h, smem);
        for (int j = j0; j < ns; j += nj) s += seg[((size_t)(s0 + j) * H + h) * 2 + 1] * expf(seg[((size_t)(s0 + j) * H + h) * 2] - m);
        s = head_reduce<float, WAVES_PER_BLOCK, false>(s, H, h, smem);
        if (threadIdx.x < H) { of_head[0][h] = m; of_head[1][h] = s; }
    } else {
        float s = 0.f;
        for (int j = j0; j < ns; j += nj) s += seg[(size_t)(s0 + j) * H + h];
        s = head_reduce<float, WAVES_PER_BLOCK, false>(s, H, h, smem);
        if (threadIdx.x < H) of_head[0][h] = s;
    }
    __syncthreads();
    const int q4 = 4 * ((int)threadIdx.x % Q);
    float a[4], b[4], v[U][4], d[U][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { a[i] = of_head[0][q4 + i]; b[i] = FWD ? of_head[1][q4 + i] : 0.f; }
    int e[U];
    for (int p = first + (int)threadIdx.x / Q; p < end; p += U * SL) {
        quad_eids<U>(P, p, SL, end, e);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (e[u] >= 0) {
                Quad<T>::ld(x + (size_t)e[u] * H + q4, v[u]);
                if constexpr (!FWD) Quad<T>::ld(dy + (size_t)e[u] * H + q4, d[u]);
            }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (e[u] < 0) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[u][i] = FWD ? expf(v[u][i] - a[i]) / b[i] : v[u][i] * (d[u][i] - a[i]);
            Quad<T>::st(y + (size_t)e[u] * H + q4, v[u]);
        }
    }
}

// ------------------------------------------------------------------------------------------
// fast family: compile-time (H, D), f32 / bf16
// ------------------------------------------------------------------------------------------
template <typename T, int H_, int D_> struct Lay {
    static constexpr int H = H_, D = D_, C = H_ * D_;
    static constexpr int LPH = 64 / H_;                 // lanes per head
    static constexpr int EPL = C / 64;                  // elements per lane (all of one head)
    static constexpr int VE = 16 / (int)sizeof(T);      // elements per 16-byte vector
    static constexpr int NV = EPL / VE;                 // 16-byte vectors per lane
    static_assert(64 % H_ == 0 && C % 64 == 0 && EPL % VE == 0 && NV >= 1, "unsupported fast shape");
    static_assert(LPH >= 4, "the row-group kernels broadcast per-member values inside quads of one head");
    static_assert(D_ == NV * LPH * VE, "layout does not tile the head");
    // element offset inside a node row of vector i of `lane`: LPH consecutive lanes cover
    // LPH*16 contiguous bytes of their head
    static __device__ __forceinline__ int off(int lane, int i) { return (lane / LPH) * D + (i * LPH + lane % LPH) * VE; }
};

template <typename T, int H, int D>
__device__ __forceinline__ void load_row(const T *__restrict__ row, int lane, float (&out)[Lay<T, H, D>::EPL]) {
    using L = Lay<T, H, D>;
#pragma unroll
    for (int i = 0; i < L::NV; ++i) {
        if constexpr (sizeof(T) == 4) {
            const float4 v = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(row) + L::off(lane, i));
            out[4 * i] = v.x; out[4 * i + 1] = v.y; out[4 * i + 2] = v.z; out[4 * i + 3] = v.w;
        } else {
            const uint4 v = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(row) + L::off(lane, i));
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                out[8 * i + 2 * c] = __uint_as_float(w[c] << 16);
                out[8 * i + 2 * c + 1] = __uint_as_float(w[c] & 0xffff0000u);
            }
        }
    }
}

template <typename T, int H, int D>
__device__ __forceinline__ void store_row(T *__restrict__ row, int lane, const float (&in)[Lay<T, H, D>::EPL]) {
    using L = Lay<T, H, D>;
#pragma unroll
    for (int i = 0; i < L::NV; ++i) {
        if constexpr (sizeof(T) == 4) {
            *reinterpret_cast<float4 *>(reinterpret_cast<float *>(row) + L::off(lane, i)) =
                make_float4(in[4 * i], in[4 * i + 1], in[4 * i + 2], in[4 * i + 3]);
        } else {
            uint32_t w[4];
#pragma unroll
            for (int c = 0; c < 4; ++c)
                w[c] = (uint32_t)f32_to_bf16(in[8 * i + 2 * c]) | ((uint32_t)f32_to_bf16(in[8 * i + 2 * c + 1]) << 16);
            *reinterpret_cast<uint4 *>(reinterpret_cast<uint16_t *>(row) + L::off(lane, i)) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

// The D elements of an (E, D) edge-feature row that go with this lane's slice of a head (every head's lanes read
// the same D elements).
template <typename T, int H, int D>
__device__ __forceinline__ void load_head_row(const T *__restrict__ row, int lane, float (&out)[Lay<T, H, D>::EPL]) {
    using L = Lay<T, H, D>;
#pragma unroll
    for (int i = 0; i < L::NV; ++i) {
        const int off = (i * L::LPH + lane % L::LPH) * L::VE;
        if constexpr (sizeof(T) == 4) {
            const float4 v = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(row) + off);
            out[4 * i] = v.x; out[4 * i + 1] = v.y; out[4 * i + 2] = v.z; out[4 * i + 3] = v.w;
        } else {
            const uint4 v = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(row) + off);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                out[8 * i + 2 * c] = __uint_as_float(w[c] << 16);
                out[8 * i + 2 * c + 1] = __uint_as_float(w[c] & 0xffff0000u);
            }
        }
    }
}

// f32 partial rows in the workspace are stored in natural column order (the combine kernels
// index them by column), whatever the element type of the node tensors
template <typename T, int H, int D>
__device__ __forceinline__ void store_row_ws(float *__restrict__ row, int lane, const float (&in)[Lay<T, H, D>::EPL]) {
    using L = Lay<T, H, D>;
#pragma unroll
    for (int i = 0; i < L::NV; ++i)
#pragma unroll
        for (int c = 0; c < L::VE / 4; ++c)
            *reinterpret_cast<float4 *>(row + L::off(lane, i) + 4 * c) =
                make_float4(in[L::VE * i + 4 * c], in[L::VE * i + 4 * c + 1], in[L::VE * i + 4 * c + 2], in[L::VE * i + 4 * c + 3]);
}

template <int CTRL> __device__ __forceinline__ float dpp_mov(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}

template <int I> __device__ __forceinline__ float quad_lane(float x) { return dpp_mov<I * 0x55>(x); }   // value of lane I of the quad
__device__ __forceinline__ float quad_bcast(float x, int i) {      // the same for an index that is constant after unrolling
    switch (i & 3) {
    case 0: return quad_lane<0>(x);
    case 1: return quad_lane<1>(x);
    case 2: return quad_lane<2>(x);
    default: return quad_lane<3>(x);
    }
}

// Sum over the LPH lanes that hold one head; the result is in all of them.
template <int LPH> __device__ __forceinline__ float head_sum(float x) {
    if constexpr (LPH >= 2) x += dpp_mov<0xB1>(x);    // quad_perm [1,0,3,2]
    if constexpr (LPH >= 4) x += dpp_mov<0x4E>(x);    // quad_perm [2,3,0,1]
    if constexpr (LPH >= 8) x += dpp_mov<0x141>(x);   // row_half_mirror
    if constexpr (LPH >= 16) x += dpp_mov<0x140>(x);  // row_mirror
    if constexpr (LPH >= 32) x += __shfl_xor(x, 16);
    if constexpr (LPH >= 64) x += __shfl_xor(x, 32);
    return x;
}

template <int N> __device__ __forceinline__ float dot_n(const float (&a)[N], const float (&b)[N]) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) s = fmaf(a[i], b[i], s);
    return s;
}

// The gathers are latency bound: all row loads of a batch must be in flight before the first
// one is consumed.  Without this fence the instruction scheduler interleaves loads and FMAs to
// save registers and waits for every load separately.
__device__ __forceinline__ void issue_loads_first() { __builtin_amdgcn_sched_barrier(0); }

// weight loads for the fast SpMM: the unfused API passes T-typed edge data, the fused backward f32
template <typename WT> __device__ __forceinline__ float ld_w(const WT *p) { return Elem<WT>::ld(p); }

// NW wavefronts (a workgroup) share an item: each takes whole batches of its edges, as many as the others, and the sums meet in
// LDS.  False: no such item (the whole workgroup).  parts: how many wavefronts have edges (one at least).
template <int NW, int BATCH> __device__ __forceinline__ bool fetch_item_part(const bpt_plan &P, Item &it, int &part, int &parts) {
    part = 0;
    parts = 1;
    if constexpr (NW == 1) return fetch_item(P, it);
    const int w = xcd_contiguous_block();
    if (w >= (int)P.n_items) return false;
    const int4 v = reinterpret_cast<const int4 *>(P.items)[w];
    it.row = __builtin_amdgcn_readfirstlane(v.x);
    it.begin = __builtin_amdgcn_readfirstlane(v.y);
    it.end = __builtin_amdgcn_readfirstlane(v.z);
    it.slot = __builtin_amdgcn_readfirstlane(v.w);
    const int deg = it.end - it.begin, per = (deg + NW * BATCH - 1) / (NW * BATCH) * BATCH;
    part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    parts = max(1, (deg + max(per, 1) - 1) / max(per, 1));
    it.begin = min(it.begin + part * per, it.end);
    it.end = min(it.begin + per, it.end);
    return true;
}

// the wavefronts' sums of one item in the first wavefront, in their order; the others are done.  By the whole workgroup.
template <int NW, int N> __device__ __forceinline__ bool parts_meet(float (&acc)[N], int part, int parts, int lane) {
    if constexpr (NW > 1) {
        __shared__ float held[NW - 1][N][WAVE];
        if (part > 0 && part < parts) {
#pragma unroll
            for (int i = 0; i < N; ++i) held[part - 1][i][lane] = acc[i];
        }
        __syncthreads();
        if (part > 0) return false;
        for (int w = 0; w < parts - 1; ++w)
#pragma unroll
            for (int i = 0; i < N; ++i) acc[i] += held[w][i][lane];
    }
    return true;
}

// y[eid[p], head] = A[row, head, :] . B[idx[p], head, :]   (MODE 1: . B[eid[p], :], B an (E, D) edge feature;
// MODE 2: . B[idx[p], :], B a (n_index, D) table shared by the heads).  YT: element type of y.
template <typename T, int H, int D, int BATCH, int MODE = 0, typename YT = T>
__global__ __launch_bounds__(BLOCK) void k_sddmm_fast(bpt_plan P, const T *__restrict__ A, const T *__restrict__ B, YT *__restrict__ y) {
    using L = Lay<T, H, D>;
    Item it;
    if (!fetch_item(P, it)) return;
    const int lane = threadIdx.x & 63, head = lane / L::LPH;
    float a[L::EPL];
    load_row<T, H, D>(A + (size_t)it.row * L::C, lane, a);
    for (int p0 = it.begin; p0 < it.end; p0 += WAVE) {
        const int cnt = min(WAVE, it.end - p0);
        const int my_idx = (MODE != 1 && lane < cnt) ? P.idx[p0 + lane] : 0;
        const int my_eid = lane < cnt ? P.eid[p0 + lane] : 0;
        for (int b = 0; b < cnt; b += BATCH) {
            float bv[BATCH][L::EPL];
            int ee[BATCH];
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                const int j = (b + e < cnt) ? b + e : b;
                ee[e] = __builtin_amdgcn_readlane(my_eid, j);
                if constexpr (MODE == 0) load_row<T, H, D>(B + (size_t)__builtin_amdgcn_readlane(my_idx, j) * L::C, lane, bv[e]);
                else if constexpr (MODE == 1) load_head_row<T, H, D>(B + (size_t)ee[e] * D, lane, bv[e]);
                else load_head_row<T, H, D>(B + (size_t)__builtin_amdgcn_readlane(my_idx, j) * D, lane, bv[e]);
            }
            issue_loads_first();
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                const float s = head_sum<L::LPH>(dot_n<L::EPL>(a, bv[e]));
                if (b + e < cnt && lane % L::LPH == 0) Elem<YT>::st(y + (size_t)ee[e] * H + head, s);
            }
        }
    }
}

// Y0[row] = sum_p W0[eid[p], head] * X0[idx[p]]  (and the same with W1, X1 -> Y1 when NOUT == 2);
// MODE 1: * X0[eid[p], :], X0 an (E, D) edge feature shared by the heads
template <typename T, typename WT, int H, int D, int BATCH, int NOUT, int MODE = 0, int NW = 1>
__global__ __launch_bounds__(NW == 1 ? BLOCK : NW * WAVE) void k_spmm_fast(bpt_plan P, const WT *__restrict__ W0, const T *__restrict__ X0, T *__restrict__ Y0,
                                                     const WT *__restrict__ W1, const T *__restrict__ X1, T *__restrict__ Y1,
                                                     float *__restrict__ ws0, float *__restrict__ ws1) {
    using L = Lay<T, H, D>;
    Item it;
    int part, parts;
    if (!fetch_item_part<NW, BATCH>(P, it, part, parts)) return;
    const int lane = threadIdx.x & 63, head = lane / L::LPH;
    float acc0[L::EPL], acc1[L::EPL];
#pragma unroll
    for (int i = 0; i < L::EPL; ++i) { acc0[i] = 0.f; acc1[i] = 0.f; }
    for (int p0 = it.begin; p0 < it.end; p0 += WAVE) {
        const int cnt = min(WAVE, it.end - p0);
        const int my_idx = (MODE == 0 && lane < cnt) ? P.idx[p0 + lane] : 0;
        const int my_eid = lane < cnt ? P.eid[p0 + lane] : 0;
        for (int b = 0; b < cnt; b += BATCH) {
            float x0[BATCH][L::EPL], x1[NOUT == 2 ? BATCH : 1][L::EPL];
            float w0[BATCH], w1[BATCH];
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                const bool ok = b + e < cnt;
                const int j = ok ? b + e : b;
                const int src = __builtin_amdgcn_readlane(my_idx, j);
                const int ed = __builtin_amdgcn_readlane(my_eid, j);
                if constexpr (MODE == 0) load_row<T, H, D>(X0 + (size_t)src * L::C, lane, x0[e]);
                else load_head_row<T, H, D>(X0 + (size_t)ed * D, lane, x0[e]);
                w0[e] = ok ? ld_w(W0 + (size_t)ed * H + head) : 0.f;
                if constexpr (NOUT == 2) {
                    load_row<T, H, D>(X1 + (size_t)src * L::C, lane, x1[e]);
                    w1[e] = ok ? ld_w(W1 + (size_t)ed * H + head) : 0.f;
                }
            }
            issue_loads_first();
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
#pragma unroll
                for (int i = 0; i < L::EPL; ++i) {
                    acc0[i] = fmaf(w0[e], x0[e][i], acc0[i]);
                    if constexpr (NOUT == 2) acc1[i] = fmaf(w1[e], x1[e][i], acc1[i]);
                }
            }
        }
    }
    if constexpr (NW > 1) {
        float both[NOUT * L::EPL];
#pragma unroll
        for (int i = 0; i < L::EPL; ++i) {
            both[i] = acc0[i];
            if constexpr (NOUT == 2) both[L::EPL + i] = acc1[i];
        }
        if (!parts_meet<NW>(both, part, parts, lane)) return;
#pragma unroll
        for (int i = 0; i < L::EPL; ++i) {
            acc0[i] = both[i];
            if constexpr (NOUT == 2) acc1[i] = both[L::EPL + i];
        }
    }
    if (it.slot < 0) {
        store_row<T, H, D>(Y0 + (size_t)it.row * L::C, lane, acc0);
        if constexpr (NOUT == 2) store_row<T, H, D>(Y1 + (size_t)it.row * L::C, lane, acc1);
    } else {
        store_row_ws<T, H, D>(ws0 + (size_t)it.slot * L::C, lane, acc0);
        if constexpr (NOUT == 2) store_row_ws<T, H, D>(ws1 + (size_t)it.slot * L::C, lane, acc1);
    }
}

// dB[eid[p], d] = sum_h dy[eid[p], h] * A[row, h, d]   (graphop_kernel.cu:79-94), lane = column d (D <= 64):
// the row's H head vectors stay in registers, each edge costs one 4*H-byte load, H FMAs and one D-element store.
template <typename T, int H, int D, int BATCH>
__global__ __launch_bounds__(BLOCK) void k_nme_dB_fast(bpt_plan P, const T *__restrict__ A, const T *__restrict__ dy, T *__restrict__ dB) {
    static_assert(D <= WAVE && H <= WAVE, "one lane per column");
    Item it;
    if (!fetch_item(P, it)) return;
    const int lane = threadIdx.x & 63;
    const int col = lane < D ? lane : 0;
    float a[H];
#pragma unroll
    for (int h = 0; h < H; ++h) a[h] = Elem<T>::ld(A + (size_t)it.row * H * D + h * D + col);
    for (int p0 = it.begin; p0 < it.end; p0 += WAVE) {
        const int cnt = min(WAVE, it.end - p0);
        const int my_eid = lane < cnt ? P.eid[p0 + lane] : 0;
        for (int b = 0; b < cnt; b += BATCH) {
            int ee[BATCH];
            float g[BATCH];
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                ee[e] = __builtin_amdgcn_readlane(my_eid, (b + e < cnt) ? b + e : b);
                g[e] = Elem<T>::ld(dy + (size_t)ee[e] * H + (lane < H ? lane : 0));     // lane h holds dy[e, h]
            }
            issue_loads_first();
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                float s = 0.f;
#pragma unroll
                for (int h = 0; h < H; ++h) s = fmaf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(g[e]), h)), a[h], s);
                if (b + e < cnt && lane < D) Elem<T>::st(dB + (size_t)ee[e] * D + lane, s);
            }
        }
    }
}

// Fused forward: per destination row, online softmax over the in-edges in batches of BATCH.
// Scores are kept in base-2 units (q is pre-multiplied by scale*log2(e)).  NW: wavefronts a row (row_parts).
template <typename T, int H, int D, int BATCH, int NW = 1>
__global__ __launch_bounds__(NW == 1 ? BLOCK : NW * WAVE) void k_attn_fwd(bpt_plan P, const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v,
                                                    T *__restrict__ o, float *__restrict__ lse, float *__restrict__ ws_acc,
                                                    float *__restrict__ ws_ml, float scale_log2e) {
    using L = Lay<T, H, D>;
    Item it;
    int part, parts;
    if (!fetch_item_part<NW, BATCH>(P, it, part, parts)) return;
    const int lane = threadIdx.x & 63, head = lane / L::LPH;
    float qv[L::EPL], acc[L::EPL];
    load_row<T, H, D>(q + (size_t)it.row * L::C, lane, qv);
#pragma unroll
    for (int i = 0; i < L::EPL; ++i) { qv[i] *= scale_log2e; acc[i] = 0.f; }
    float m = M_INIT_LOG2, l = 0.f;
    for (int p0 = it.begin; p0 < it.end; p0 += WAVE) {
        const int cnt = min(WAVE, it.end - p0);
        const int my_idx = lane < cnt ? P.idx[p0 + lane] : 0;
        for (int b = 0; b < cnt; b += BATCH) {
            float kv[BATCH][L::EPL], vv[BATCH][L::EPL], s[BATCH];
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                const int src = __builtin_amdgcn_readlane(my_idx, (b + e < cnt) ? b + e : b);
                load_row<T, H, D>(k + (size_t)src * L::C, lane, kv[e]);
                load_row<T, H, D>(v + (size_t)src * L::C, lane, vv[e]);
            }
            issue_loads_first();
            float mx = m;
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                const float t = head_sum<L::LPH>(dot_n<L::EPL>(qv, kv[e]));
                s[e] = (b + e < cnt) ? t : -INFINITY;
                mx = fmaxf(mx, s[e]);
            }
            const float alpha = __builtin_amdgcn_exp2f(m - mx);
            l *= alpha;
#pragma unroll
            for (int i = 0; i < L::EPL; ++i) acc[i] *= alpha;
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                const float pe = __builtin_amdgcn_exp2f(s[e] - mx);
                l += pe;
#pragma unroll
                for (int i = 0; i < L::EPL; ++i) acc[i] = fmaf(pe, vv[e][i], acc[i]);
            }
            m = mx;
        }
    }
    if constexpr (NW > 1) {
        __shared__ float held[NW - 1][L::EPL + 2][WAVE];
        if (part > 0 && part < parts) {
#pragma unroll
            for (int i = 0; i < L::EPL; ++i) held[part - 1][i][lane] = acc[i];
            held[part - 1][L::EPL][lane] = m;
            held[part - 1][L::EPL + 1][lane] = l;
        }
        __syncthreads();
        if (part > 0) return;
        for (int w = 0; w < parts - 1; ++w) {
            const float mw = held[w][L::EPL][lane], mx = fmaxf(m, mw);
            const float a = __builtin_amdgcn_exp2f(m - mx), b = __builtin_amdgcn_exp2f(mw - mx);
            l = fmaf(b, held[w][L::EPL + 1][lane], a * l);
#pragma unroll
            for (int i = 0; i < L::EPL; ++i) acc[i] = fmaf(b, held[w][i][lane], a * acc[i]);
            m = mx;
        }
    }
    if (it.slot < 0) {
        const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
        for (int i = 0; i < L::EPL; ++i) acc[i] *= inv;
        store_row<T, H, D>(o + (size_t)it.row * L::C, lane, acc);
        if (lane % L::LPH == 0) lse[(size_t)it.row * H + head] = l > 0.f ? m + log2f(l) : 0.f;
    } else {
        store_row_ws<T, H, D>(ws_acc + (size_t)it.slot * L::C, lane, acc);
        if (lane % L::LPH == 0) {
            ws_ml[((size_t)it.slot * H + head) * 2] = m;
            ws_ml[((size_t)it.slot * H + head) * 2 + 1] = l;
        }
    }
}

// Combine the (m, l, acc) partials of each split row.  Grid (n_heavy, C / 64): one block per split row
// and 64-column strip; wave w folds slots w, w+4, ... with a running maximum (one pass, eight
// independent loads per step), then the four wave results are merged in wave order.
template <typename T, int HC, int D, bool NARROW = false>
__global__ __launch_bounds__(BLOCK) void k_attn_fwd_combine(const int32_t *__restrict__ heavy, const float *__restrict__ ws_acc,
                                                            const float *__restrict__ ws_ml, T *__restrict__ o, float *__restrict__ lse,
                                                            Narrow nw, T *__restrict__ o_keep = nullptr) {
    static_assert(HC * D % WAVE == 0, "strip width");
    const int H = NARROW ? nw.h : HC, C = H * D;                 // (NARROW: one strip per real head)
    __shared__ float pm[WAVES_PER_BLOCK][WAVE], pl[WAVES_PER_BLOCK][WAVE], pa[WAVES_PER_BLOCK][WAVE];
    const int row = heavy[3 * blockIdx.x], s0 = heavy[3 * blockIdx.x + 1], ns = heavy[3 * blockIdx.x + 2];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = blockIdx.y * WAVE + lane, head = j / D;
    const float *ml = ws_ml + ((size_t)s0 * H + head) * 2;      // slot stride 2*H
    const float *col = ws_acc + (size_t)s0 * C + j;              // slot stride C
    float M = M_INIT_LOG2, lsum = 0.f, a = 0.f;
    int kk = w;
    float tm[16], tl[16], ta[16];
    auto ask = [&](int u, int nth) {
        const size_t sl = (size_t)(kk + nth * WAVES_PER_BLOCK);
        tm[u] = ml[sl * 2 * H];
        tl[u] = ml[sl * 2 * H + 1];
        ta[u] = col[sl * C];
    };
    auto fold = [&](auto n) {
        float mx = M;
#pragma unroll
        for (int u = 0; u < n(); ++u) mx = fmaxf(mx, tm[u]);
        const float resc = __builtin_amdgcn_exp2f(M - mx);
        lsum *= resc;
        a *= resc;
#pragma unroll
        for (int u = 0; u < n(); ++u) {
            const float wgt = __builtin_amdgcn_exp2f(tm[u] - mx);
            lsum = fmaf(tl[u], wgt, lsum);
            a = fmaf(ta[u], wgt, a);
        }
        M = mx;
    };
    for (; kk + 15 * WAVES_PER_BLOCK < ns; kk += 16 * WAVES_PER_BLOCK) {
#pragma unroll
        for (int u = 0; u < 16; ++u) ask(u, u);
        fold(std::integral_constant<int, 16>{});
    }
    if (kk + 7 * WAVES_PER_BLOCK < ns) {
#pragma unroll
        for (int u = 0; u < 8; ++u) ask(u, u);
        fold(std::integral_constant<int, 8>{});
        kk += 8 * WAVES_PER_BLOCK;
    }
    const int left = combine_left(kk, ns);
    if (left > 0) {
#pragma unroll
        for (int u = 0; u < 7; ++u) { tm[u] = -INFINITY; tl[u] = ta[u] = 0.f; }
        combine_tail(left, ask);
        fold(std::integral_constant<int, 7>{});
    }
    pm[w][lane] = M; pl[w][lane] = lsum; pa[w][lane] = a;
    __syncthreads();
    if (w == 0) {
        float Mx = pm[0][lane];
#pragma unroll
        for (int i = 1; i < WAVES_PER_BLOCK; ++i) Mx = fmaxf(Mx, pm[i][lane]);
        float L = 0.f, A = 0.f;
#pragma unroll
        for (int i = 0; i < WAVES_PER_BLOCK; ++i) {
            const float wgt = __builtin_amdgcn_exp2f(pm[i][lane] - Mx);
            L = fmaf(pl[i][lane], wgt, L);
            A = fmaf(pa[i][lane], wgt, A);
        }
        if (!NARROW) Elem<T>::st(o + (size_t)row * C + j, L > 0.f ? A / L : 0.f);
        else if (lane < nw.d) {
            Elem<T>::st(o + (size_t)row * (nw.heads * nw.d) + head * nw.d + lane, L > 0.f ? A / L : 0.f);
            if (o_keep) Elem<T>::st(o_keep + (size_t)row * (nw.heads * nw.d) + head * nw.d + lane, L > 0.f ? A / L : 0.f);
        }
        if (j % D == 0) lse[(size_t)row * H + head] = L > 0.f ? Mx + log2f(L) : 0.f;
    }
}

// Fused backward, destination side: recompute p from lse, delta = dO.O, ds = p*(dO.v - delta)*scale,
// dQ[row] = sum ds*k; p and ds go to (E, H) f32 buffers addressed by edge id for the source-side pass.
template <typename T, int H, int D, int BATCH, int NW = 1>
__global__ __launch_bounds__(NW == 1 ? BLOCK : NW * WAVE) void k_attn_bwd_dst(bpt_plan P, const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v,
                                                        const T *__restrict__ o, const T *__restrict__ d_o, const float *__restrict__ lse,
                                                        T *__restrict__ dq, float *__restrict__ pbuf, float *__restrict__ dsbuf,
                                                        float *__restrict__ ws_dq, float scale, float scale_log2e) {
    using L = Lay<T, H, D>;
    Item it;
    int part, parts;
    if (!fetch_item_part<NW, BATCH>(P, it, part, parts)) return;
    const int lane = threadIdx.x & 63, head = lane / L::LPH;
    float qv[L::EPL], dov[L::EPL], dqa[L::EPL];
    float delta;
    {
        float ov[L::EPL];
        load_row<T, H, D>(o + (size_t)it.row * L::C, lane, ov);
        load_row<T, H, D>(d_o + (size_t)it.row * L::C, lane, dov);
        delta = head_sum<L::LPH>(dot_n<L::EPL>(dov, ov));
    }
    load_row<T, H, D>(q + (size_t)it.row * L::C, lane, qv);
#pragma unroll
    for (int i = 0; i < L::EPL; ++i) dqa[i] = 0.f;
    const float lse2 = lse[(size_t)it.row * H + head];
    for (int p0 = it.begin; p0 < it.end; p0 += WAVE) {
        const int cnt = min(WAVE, it.end - p0);
        const int my_idx = lane < cnt ? P.idx[p0 + lane] : 0;
        const int my_eid = lane < cnt ? P.eid[p0 + lane] : 0;
        for (int b = 0; b < cnt; b += BATCH) {
            float kv[BATCH][L::EPL], vv[BATCH][L::EPL];
            int ee[BATCH];
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                const int j = (b + e < cnt) ? b + e : b;
                const int src = __builtin_amdgcn_readlane(my_idx, j);
                ee[e] = __builtin_amdgcn_readlane(my_eid, j);
                load_row<T, H, D>(k + (size_t)src * L::C, lane, kv[e]);
                load_row<T, H, D>(v + (size_t)src * L::C, lane, vv[e]);
            }
            issue_loads_first();
#pragma unroll
            for (int e = 0; e < BATCH; ++e) {
                const float s = head_sum<L::LPH>(dot_n<L::EPL>(qv, kv[e]));
                const float dp = head_sum<L::LPH>(dot_n<L::EPL>(dov, vv[e]));
                const bool ok = b + e < cnt;
                const float pe = ok ? __builtin_amdgcn_exp2f(fmaf(s, scale_log2e, -lse2)) : 0.f;
                const float ds = pe * (dp - delta) * scale;
#pragma unroll
                for (int i = 0; i < L::EPL; ++i) dqa[i] = fmaf(ds, kv[e][i], dqa[i]);
                if (ok && lane % L::LPH == 0) {
                    pbuf[(size_t)ee[e] * H + head] = pe;
                    dsbuf[(size_t)ee[e] * H + head] = ds;
                }
            }
        }
    }
    if (!parts_meet<NW>(dqa, part, parts, lane)) return;
    if (it.slot < 0) store_row<T, H, D>(dq + (size_t)it.row * L::C, lane, dqa);
    else store_row_ws<T, H, D>(ws_dq + (size_t)it.slot * L::C, lane, dqa);
}

// ------------------------------------------------------------------------------------------
// row-group kernels of the fused path: one wavefront (= one workgroup) owns a group of up to
// R (4 or 8) rows (or row segments) that share neighbours; every neighbour row of the group's union
// ("entry") is loaded once and used for all members that have an edge to it (entry mask).
//
// The kernels issue about one instruction per four cycles and SIMD, whatever its kind, so they are
// written for a low instruction count per (member, entry) pair: 32-bit byte offsets from uniform
// base pointers (no 64-bit vector address arithmetic), the entry list of up to GRP_CHUNK entries
// held one per lane and read with v_readlane, per-pair scratch addressed by entry * R + member
// (no popcounts), unmasked scratch stores.
// ------------------------------------------------------------------------------------------
// entries whose rows are loaded together (one where a row takes 16 registers per lane)
template <int EPL> constexpr int grp_batch() { return EPL >= 16 ? 1 : 2; }
constexpr int GRP_CHUNK = 56;                      // entries per lane-held list: a multiple of twice the batch, and
                                                   // GRP_CHUNK + 3 * batch <= 64 keeps every look-ahead index a lane id
constexpr int GRP_PAD_ENTRIES = 8;                 // the per-entry arrays are readable this far past the end

template <int R> struct GroupHead {
    int rows[R], slots[R], begin, end;
};

// wavefronts per SIMD the row-group kernels are compiled for: the members' state has to stay in registers
template <typename T, int EPL, int R> constexpr int grp_wpe() { return R * EPL <= 32 ? 3 : 2; }

// Workgroup b (one wavefront) runs on XCD b % 8 and takes head slice (b / 8) % HS of group number (b / 8) / HS of
// that XCD's chunk: HS wavefronts share a group, each handling H / HS of the heads of every row.  (Dispatching all
// first slices before the second ones, to halve the rows an XCD's L2 has to hold at a time, measured slower.)
template <int R, int HS> __device__ __forceinline__ int group_slice() { return (int)((blockIdx.x >> 3) % HS); }
template <int R, int HS> __device__ __forceinline__ bool fetch_group(const bpt_plan &P, GroupHead<R> &gh) {
    const int x = blockIdx.x & 7, w = (blockIdx.x >> 3) / HS;
    const int g = __builtin_amdgcn_readfirstlane(P.grp_chunks[x]) + w;
    if (g >= __builtin_amdgcn_readfirstlane(P.grp_chunks[x + 1])) return false;
    const int lane = threadIdx.x;
    const int mem = P.grp_members[(size_t)g * (2 * R) + (lane & (2 * R - 1))];
    const int ptr = P.grp_ptr[g + (lane & 1)];
#pragma unroll
    for (int m = 0; m < R; ++m) {
        gh.rows[m] = __builtin_amdgcn_readlane(mem, 2 * m);
        gh.slots[m] = __builtin_amdgcn_readlane(mem, 2 * m + 1);
    }
    gh.begin = __builtin_amdgcn_readlane(ptr, 0);
    gh.end = __builtin_amdgcn_readlane(ptr, 1);
    return true;
}

// Row `row` of a node tensor (PITCH elements per row; the layout may cover a slice of the row's heads) through a
// uniform base pointer, a uniform 32-bit row offset and this lane's constant byte offset `loff` (global_load with scalar base + 32-bit vector offset + immediate).
template <typename T, int H, int D, int PITCH = Lay<T, H, D>::C>
__device__ __forceinline__ void load_row32(const T *__restrict__ base, uint32_t row, uint32_t loff, float (&out)[Lay<T, H, D>::EPL]) {
    using L = Lay<T, H, D>;
    const char *p = reinterpret_cast<const char *>(base) + (size_t)(row * (uint32_t)(PITCH * sizeof(T)));
#pragma unroll
    for (int i = 0; i < L::NV; ++i) {
        const char *pi = p + (size_t)(loff + (uint32_t)(i * L::LPH * 16));
        if constexpr (sizeof(T) == 4) {
            const float4 v = *reinterpret_cast<const float4 *>(pi);
            out[4 * i] = v.x; out[4 * i + 1] = v.y; out[4 * i + 2] = v.z; out[4 * i + 3] = v.w;
        } else {
            const uint4 v = *reinterpret_cast<const uint4 *>(pi);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                out[8 * i + 2 * c] = __uint_as_float(w[c] << 16);
                out[8 * i + 2 * c + 1] = __uint_as_float(w[c] & 0xffff0000u);
            }
        }
    }
}

// The same row as loaded, not yet converted: the software pipeline keeps rows in flight in this form, and
// converts them where they are used, after the wait (bf16 to f32 costs a shift or a mask per element).
template <typename T, int H, int D> struct RawRow { uint32_t w[Lay<T, H, D>::EPL * sizeof(T) / 4]; };

template <typename T, int H, int D, int PITCH = Lay<T, H, D>::C>
__device__ __forceinline__ void load_row32_raw(const T *__restrict__ base, uint32_t row, uint32_t loff, RawRow<T, H, D> &out) {
    using L = Lay<T, H, D>;
    const char *p = reinterpret_cast<const char *>(base) + (size_t)(row * (uint32_t)(PITCH * sizeof(T)));
#pragma unroll
    for (int i = 0; i < L::NV; ++i) {
        const uint4 v = *reinterpret_cast<const uint4 *>(p + (size_t)(loff + (uint32_t)(i * L::LPH * 16)));
        out.w[4 * i] = v.x; out.w[4 * i + 1] = v.y; out.w[4 * i + 2] = v.z; out.w[4 * i + 3] = v.w;
    }
}

template <typename T, int H, int D>
__device__ __forceinline__ void unpack_row(const RawRow<T, H, D> &in, float (&out)[Lay<T, H, D>::EPL]) {
    using L = Lay<T, H, D>;
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int i = 0; i < L::EPL; ++i) out[i] = __uint_as_float(in.w[i]);
    } else {
#pragma unroll
        for (int j = 0; j < L::EPL / 2; ++j) {
            out[2 * j] = __uint_as_float(in.w[j] << 16);
            out[2 * j + 1] = __uint_as_float(in.w[j] & 0xffff0000u);
        }
    }
}

// A wavefront-private row in LDS, lane-major (float4 c of lane l at slot c * 64 + l: conflict free).
template <int EPL> __device__ __forceinline__ void lds_put_row(float4 *slot, int lane, const float (&r)[EPL]) {
#pragma unroll
    for (int c = 0; c < EPL / 4; ++c) slot[c * WAVE + lane] = make_float4(r[4 * c], r[4 * c + 1], r[4 * c + 2], r[4 * c + 3]);
}
template <int EPL> __device__ __forceinline__ void lds_get_row(const float4 *slot, int lane, float (&r)[EPL]) {
#pragma unroll
    for (int c = 0; c < EPL / 4; ++c) {
        const float4 t = slot[c * WAVE + lane];
        r[4 * c] = t.x; r[4 * c + 1] = t.y; r[4 * c + 2] = t.z; r[4 * c + 3] = t.w;
    }
}

// Dropout on the attention probabilities (modules/attention.py:73): the keep / drop decision of (pair n, head h) is
// a hash of n * H + h and the call's seed, so that forward and backward agree without storing a mask.  n is the
// pair's number in the destination-side groups (entry's first pair + rank of the member in the entry's mask).
// Returns the multiplier 1 / (1 - p) or 0.
__device__ __forceinline__ float dropout_keep(uint32_t key, uint32_t seed, uint32_t thr, float inv_keep) {
    uint32_t x = key ^ seed;
    x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16;
    return x >= thr ? inv_keep : 0.f;
}

// two independent head sums, interleaved so that one hides the other's DPP wait states
template <int LPH> __device__ __forceinline__ void head_sum2(float &a, float &b) {
    if constexpr (LPH >= 2) { a += dpp_mov<0xB1>(a); b += dpp_mov<0xB1>(b); }
    if constexpr (LPH >= 4) { a += dpp_mov<0x4E>(a); b += dpp_mov<0x4E>(b); }
    if constexpr (LPH >= 8) { a += dpp_mov<0x141>(a); b += dpp_mov<0x141>(b); }
    if constexpr (LPH >= 16) { a += dpp_mov<0x140>(a); b += dpp_mov<0x140>(b); }
    if constexpr (LPH >= 32) { a += __shfl_xor(a, 16); b += __shfl_xor(b, 16); }
    if constexpr (LPH >= 64) { a += __shfl_xor(a, 32); b += __shfl_xor(b, 32); }
}

// max of three finite-or-minus-infinity values (no NaN canonicalisation of the operands)
__device__ __forceinline__ float max3f(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Forward: online softmax in base 2 over the group's entries, two entries per step.  The members' q rows
// (pre-scaled) live in LDS and are re-read for every use, which keeps the kernel at three wavefronts per SIMD.
template <typename T, int H, int D, int R, int HS, bool DROP, bool BIAS>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(grp_wpe<T, Lay<T, H / HS, D>::EPL, R>()))) void k_attn_fwd_grp(
    bpt_plan P, const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v, T *__restrict__ o,
    float *__restrict__ lse, float *__restrict__ ws_acc, float *__restrict__ ws_ml, float scale_log2e, uint32_t drop_thr,
    uint32_t drop_seed, float drop_inv, const float *__restrict__ bias) {
    constexpr int HL = H / HS, CF = H * D;                  // heads of this wavefront's slice; elements of a full row
    using L = Lay<T, HL, D>;
    constexpr int EPL = L::EPL, NQ = R / 4, GRP_BATCH = BIAS ? 1 : grp_batch<L::EPL>()   /* the score term's registers take the place of a second entry */;
    static_assert(H % HS == 0 && R % 4 == 0 && L::LPH >= 4, "members are handled in quads inside the lanes of one head");
    GroupHead<R> gh;
    if (!fetch_group<R, HS>(P, gh)) return;
    const int slice = group_slice<R, HS>(), coff = slice * HL * D;
    const int lane = threadIdx.x, head = slice * HL + lane / L::LPH;
    const uint32_t loff = (uint32_t)((coff + L::off(lane, 0)) * sizeof(T));
    const int4 *entries = reinterpret_cast<const int4 *>(P.grp_entries);
    struct Batch {
        RawRow<T, HL, D> kr[GRP_BATCH], vr[GRP_BATCH];
        int mk[GRP_BATCH], pz[GRP_BATCH];
        float bz[GRP_BATCH][BIAS ? R / 4 : 1];      // score term of (entry, member 4c + lane % 4), this lane's head
    };
    struct Rows {
        float kv[GRP_BATCH][EPL], vv[GRP_BATCH][EPL];
        int mk[GRP_BATCH], pz[GRP_BATCH];
    };
    const int4 *eids4 = reinterpret_cast<const int4 *>(P.grp_eids);
    __shared__ float4 q_lds[R * (EPL / 4) * WAVE];
    float acc[R][EPL], mrun[R], lrun[R];
#pragma unroll
    for (int m = 0; m < R; ++m) {
        float qr[EPL];
        load_row32<T, HL, D, CF>(q, (uint32_t)max(gh.rows[m], 0), loff, qr);
        mrun[m] = M_INIT_LOG2;
        lrun[m] = 0.f;
#pragma unroll
        for (int i = 0; i < EPL; ++i) { qr[i] *= scale_log2e; acc[m][i] = 0.f; }
        lds_put_row<EPL>(q_lds + m * (EPL / 4) * WAVE, lane, qr);
    }
    for (int p0 = gh.begin; p0 < gh.end; p0 += GRP_CHUNK) {
        const int cnt = min(GRP_CHUNK, gh.end - p0);
        // lanes past the end repeat the last entry with an empty mask
        int4 ent = entries[p0 + min(lane, cnt - 1)];
        ent.y = lane < cnt ? ent.y : 0;
        // edge ids of the lane's entry, four members per vector (the list is padded like the entries)
        int4 xe[R / 4];
        if constexpr (BIAS || DROP) {
#pragma unroll
            for (int c = 0; c < R / 4; ++c) xe[c] = eids4[(size_t)(p0 + min(lane, cnt - 1)) * (R / 4) + c];
        }
        auto load_batch = [&](Batch &B, int b) {
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                const uint32_t src = (uint32_t)__builtin_amdgcn_readlane(ent.x, b + e);
                B.mk[e] = __builtin_amdgcn_readlane(ent.y, b + e);
                B.pz[e] = DROP ? b + e : 0;                  // position of the entry in the chunk: the lane that holds its edge ids
                if constexpr (BIAS) {
#pragma unroll
                    for (int c = 0; c < R / 4; ++c) {
                        // lane l fetches the term of member 4c + l % 4; the quad's lanes hand it round when it is used
                        const uint32_t e0 = (uint32_t)__builtin_amdgcn_readlane(xe[c].x, b + e), e1 = (uint32_t)__builtin_amdgcn_readlane(xe[c].y, b + e);
                        const uint32_t e2 = (uint32_t)__builtin_amdgcn_readlane(xe[c].z, b + e), e3 = (uint32_t)__builtin_amdgcn_readlane(xe[c].w, b + e);
                        const uint32_t el = (lane & 3) == 0 ? e0 : (lane & 3) == 1 ? e1 : (lane & 3) == 2 ? e2 : e3;
                        B.bz[e][c] = bias[(size_t)(el * (uint32_t)H) + head];
                    }
                }
                load_row32_raw<T, HL, D, CF>(k, src, loff, B.kr[e]);
                load_row32_raw<T, HL, D, CF>(v, src, loff, B.vr[e]);
            }
        };
        // multiplier of the pair (member m, entry at position pz of the chunk): 1 without dropout; keyed by the edge id
        auto keep = [&](int m, int mk, int pz) -> float {
            if constexpr (!DROP) return 1.f;
            const int4 &x = xe[m / 4];
            const int held = (m & 3) == 0 ? x.x : (m & 3) == 1 ? x.y : (m & 3) == 2 ? x.z : x.w;
            const uint32_t edge = (uint32_t)__builtin_amdgcn_readlane(held, pz);
            return dropout_keep(edge * (uint32_t)H + (uint32_t)head, drop_seed, drop_thr, drop_inv);
        };
        auto one = [&](int m, const float (&kr)[EPL], const float (&vr)[EPL], int mk, int pz, float bz) {
            float qm[EPL];
            lds_get_row<EPL>(q_lds + m * (EPL / 4) * WAVE, lane, qm);
            const float s = head_sum<L::LPH>(dot_n<EPL>(qm, kr)) + bz;
            const float mx = fmaxf(mrun[m], s);
            const float al = __builtin_amdgcn_exp2f(mrun[m] - mx), pe = __builtin_amdgcn_exp2f(s - mx);
            lrun[m] = fmaf(lrun[m], al, pe);                       // the softmax denominator ignores dropout
            const float pk = pe * keep(m, mk, pz);
#pragma unroll
            for (int i = 0; i < EPL; ++i) acc[m][i] = fmaf(pk, vr[i], acc[m][i] * al);
            mrun[m] = mx;
        };
        auto compute = [&](const Batch &raw) {
            Rows B;
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                unpack_row<T, HL, D>(raw.kr[e], B.kv[e]);
                unpack_row<T, HL, D>(raw.vr[e], B.vv[e]);
                B.mk[e] = raw.mk[e];
                B.pz[e] = raw.pz[e];
            }
#pragma unroll
            for (int m = 0; m < R; ++m) {
                const bool h0 = (B.mk[0] >> m) & 1, h1 = (B.mk[GRP_BATCH - 1] >> m) & 1;
                // the score term in the units of the scaled scores
                const float z0 = BIAS ? quad_bcast(raw.bz[0][BIAS ? m / 4 : 0], m) * scale_log2e : 0.f;
                const float z1 = BIAS ? quad_bcast(raw.bz[GRP_BATCH - 1][BIAS ? m / 4 : 0], m) * scale_log2e : 0.f;
                if constexpr (GRP_BATCH == 1) {
                    if (h0) one(m, B.kv[0], B.vv[0], B.mk[0], B.pz[0], z0);
                } else if (h0 && h1) {
                    float qm[EPL];
                    lds_get_row<EPL>(q_lds + m * (EPL / 4) * WAVE, lane, qm);
                    float s0 = dot_n<EPL>(qm, B.kv[0]), s1 = dot_n<EPL>(qm, B.kv[GRP_BATCH - 1]);
                    head_sum2<L::LPH>(s0, s1);
                    s0 += z0;
                    s1 += z1;
                    const float mx = max3f(mrun[m], s0, s1);
                    const float al = __builtin_amdgcn_exp2f(mrun[m] - mx);
                    const float p0e = __builtin_amdgcn_exp2f(s0 - mx), p1e = __builtin_amdgcn_exp2f(s1 - mx);
                    lrun[m] = fmaf(lrun[m], al, p0e + p1e);
                    const float k0 = p0e * keep(m, B.mk[0], B.pz[0]), k1 = p1e * keep(m, B.mk[GRP_BATCH - 1], B.pz[GRP_BATCH - 1]);
#pragma unroll
                    for (int i = 0; i < EPL; ++i) acc[m][i] = fmaf(k1, B.vv[GRP_BATCH - 1][i], fmaf(k0, B.vv[0][i], acc[m][i] * al));
                    mrun[m] = mx;
                } else if (h0) {
                    one(m, B.kv[0], B.vv[0], B.mk[0], B.pz[0], z0);
                } else if (h1) {
                    one(m, B.kv[GRP_BATCH - 1], B.vv[GRP_BATCH - 1], B.mk[GRP_BATCH - 1], B.pz[GRP_BATCH - 1], z1);
                }
            }
        };
        // two-stage software pipeline: the rows of the next batch are in flight while one is used.  The loads
        // are unconditional (a branch around them would make the compiler drain the load queue at the join);
        // look-ahead past the end re-reads the chunk's last entry with an empty mask.
        Batch A, B;
        load_batch(A, 0);
        for (int b = 0; b < cnt; b += 2 * GRP_BATCH) {
            load_batch(B, b + GRP_BATCH);
            issue_loads_first();
            compute(A);
            issue_loads_first();
            load_batch(A, b + 2 * GRP_BATCH);
            issue_loads_first();
            compute(B);
            issue_loads_first();
        }
    }
#pragma unroll
    for (int m = 0; m < R; ++m) {
        if (gh.rows[m] < 0) continue;
        if (gh.slots[m] < 0) {
            const float inv = lrun[m] > 0.f ? 1.f / lrun[m] : 0.f;
#pragma unroll
            for (int i = 0; i < EPL; ++i) acc[m][i] *= inv;
            store_row<T, HL, D>(o + (size_t)gh.rows[m] * CF + coff, lane, acc[m]);
            if (lane % L::LPH == 0) lse[(size_t)gh.rows[m] * H + head] = lrun[m] > 0.f ? mrun[m] + log2f(lrun[m]) : 0.f;
        } else {
            store_row_ws<T, HL, D>(ws_acc + (size_t)gh.slots[m] * CF + coff, lane, acc[m]);
            if (lane % L::LPH == 0) {
                ws_ml[((size_t)gh.slots[m] * H + head) * 2] = mrun[m];
                ws_ml[((size_t)gh.slots[m] * H + head) * 2 + 1] = lrun[m];
            }
        }
    }
}

// ---- matrix-core forward for groups of 8 rows -------------------------------------------------------------------
// v_mfma_f32_4x4x1 works on 16 blocks of 4 lanes: D_b[i][j] += A_b[i] * B_b[j] with A_b[i] taken from lane 4b+i,
// B_b[j] from lane 4b+j and D_b[i][j] held in register i of lane 4b+j.  Block b owns the 4 * EPL columns that its
// four lanes hold in the row layout (all of one head).
//   scores   S^T = K Q^T: lane 4b+i supplies column c of the row of entry i (of a batch of four), lane 4b+j column c
//            of the q row of member j; after one instruction per column of the block and a sum over the blocks of a
//            head, register i of lane 4b+j holds (entry i, member j).  The rows reach this "one row per lane of a
//            block" arrangement through LDS: written as loaded, read back by (row, block).
//   output   O += P V: A = the lane's own probability (member j = lane % 4, entry e), B = register r of the V row
//            of entry e in the row layout; D is the accumulator of (member i, this lane's r-th column).
// A wavefront issues at most one instruction every eight cycles, so the time of a group is its instruction count:
// the matrix-core form needs about a third of the instructions per (entry, member) of the vector form.
// The exponent reference of a (member, head) is raised only when a score exceeds it by more than MFMA_TAU (base-2
// units), so the accumulators are rescaled rarely; probabilities stay below 2^MFMA_TAU times the usual ones, and
// o and lse come out the same up to rounding.
constexpr float MFMA_TAU = 8.f;
constexpr int MFMA_NB = 4;                          // entries per batch = rows of the A operand

// sum over the blocks (quads of lanes) that hold one head; the result is in all of them.  Every lane has to take
// part: a lane switched off by a branch would hand zero to its partners.
template <int BPH> __device__ __forceinline__ float block_sum(float x) {
    if constexpr (BPH >= 2) x += dpp_mov<0x1B>(dpp_mov<0x141>(x));     // lane ^ 4: row_half_mirror, then quad_perm [3,2,1,0]
    if constexpr (BPH >= 4) x += dpp_mov<0x141>(dpp_mov<0x140>(x));    // lane ^ 8: row_mirror, then row_half_mirror
    return x;
}

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef short bf16x4_t __attribute__((ext_vector_type(4)));
// two registers of bfloat16 pairs as the four-element operand of the bfloat16 matrix instructions
__device__ __forceinline__ bf16x4_t as_bf16x4(uint32_t a, uint32_t b) {
    const uint2 u = make_uint2(a, b);
    return __builtin_bit_cast(bf16x4_t, u);
}

// 16-byte vector as VE floats
template <typename T> __device__ __forceinline__ void unpack_vec(const uint4 &w, float *out) {
    const uint32_t x[4] = {w.x, w.y, w.z, w.w};
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int c = 0; c < 4; ++c) out[c] = __uint_as_float(x[c]);
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            out[2 * c] = __uint_as_float(x[c] << 16);
            out[2 * c + 1] = __uint_as_float(x[c] & 0xffff0000u);
        }
    }
}

// Two wavefronts per group of 8 rows: wavefront w owns members 4 w .. 4 w + 3 (one quad: the B operand of the
// score products), both share the staged rows.  Each wavefront loads and stages half of a batch.  With two staging
// buffers one workgroup barrier per batch orders the writes of batch b + 1 after the reads of batch b - 1; where V
// has a single buffer (W3 below) a second barrier separates the reads of batch b from the writes of batch b + 1.
template <typename T, int H, int D, int HS, bool DROP, bool BIAS>
__global__ __launch_bounds__(2 * WAVE) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 && !BIAS && !DROP ? 3 : 2))) void k_attn_fwd_mfma(
    bpt_plan P, const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v, T *__restrict__ o,
    float *__restrict__ lse, float *__restrict__ ws_acc, float *__restrict__ ws_ml, float scale_log2e, uint32_t drop_thr,
    uint32_t drop_seed, float drop_inv, const float *__restrict__ bias) {
    constexpr int R = 8, NB = MFMA_NB, HL = H / HS, CF = H * D, NE = NB / 2;      // NE: entries a wavefront loads per batch
    // float32: one V area instead of two (a second barrier per batch) and no read-ahead registers, which fits three
    // wavefronts per SIMD and six workgroups per CU (measured 5 % faster); bfloat16 rows are half as large
    constexpr bool W3 = sizeof(T) == 4 && !BIAS && !DROP;  // (the edge ids and score terms would not fit)
    using L = Lay<T, HL, D>;
    constexpr int EPL = L::EPL, NV = L::NV, VE = L::VE, BPH = L::LPH / 4, CB = 4 * EPL, PITCH = NV * WAVE + 1;
    static_assert(EPL % VE == 0 && EPL <= 8 && (BPH == 1 || BPH == 2 || BPH == 4), "shape not covered by the matrix-core kernels");
    const int lane = threadIdx.x & (WAVE - 1), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // the group of this workgroup (as fetch_group, for workgroups of two wavefronts)
    int rows[4], slots[4], g_begin, g_end;
    {
        const int x = blockIdx.x & 7, w = (blockIdx.x >> 3) / HS;
        const int g = __builtin_amdgcn_readfirstlane(P.grp_chunks[x]) + w;
        if (g >= __builtin_amdgcn_readfirstlane(P.grp_chunks[x + 1])) return;
        const int mem = P.grp_members[(size_t)g * (2 * R) + (lane & (2 * R - 1))];
        const int ptr = P.grp_ptr[g + (lane & 1)];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            rows[i] = __builtin_amdgcn_readlane(mem, 8 * wv + 2 * i);
            slots[i] = __builtin_amdgcn_readlane(mem, 8 * wv + 2 * i + 1);
        }
        g_begin = __builtin_amdgcn_readlane(ptr, 0);
        g_end = __builtin_amdgcn_readlane(ptr, 1);
    }
    const int slice = (int)((blockIdx.x >> 3) % HS), coff = slice * HL * D;
    const int head = slice * HL + lane / L::LPH, j = lane & 3, blk = lane >> 2;
    const uint32_t loff = (uint32_t)((coff + L::off(lane, 0)) * sizeof(T));
    const int4 *entries = reinterpret_cast<const int4 *>(P.grp_entries);
    const int eid_last = (int)P.n_grp_entries + GRP_PAD_ENTRIES - 1;      // last entry of grp_eids, padding included
    __shared__ uint4 kst[2][NB * PITCH];              // rows as loaded, one spare vector per row against bank conflicts
    __shared__ uint4 vst[W3 ? 1 : 2][NB * NV * WAVE];
    // q row of member 4 wv + j, the columns of this lane's block: float32 pre-scaled, or (bfloat16) as loaded, the
    // scale then being applied to the scores
    constexpr bool B16 = sizeof(T) == 2;
    float qb[B16 ? 1 : CB];
    uint4 qraw[B16 ? NV * 4 : 1];
    {
        // wavefront 0 stages its q rows through the K area, wavefront 1 through the V area
        uint4 *qst = wv == 0 ? &kst[0][0] : &vst[0][0];
        constexpr int QP = NV * WAVE;                  // unpadded: four rows fill either area exactly
        RawRow<T, HL, D> qr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) load_row32_raw<T, HL, D, CF>(q, (uint32_t)max(rows[i], 0), loff, qr[i]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < NV; ++c) qst[i * QP + c * WAVE + lane] = make_uint4(qr[i].w[4 * c], qr[i].w[4 * c + 1], qr[i].w[4 * c + 2], qr[i].w[4 * c + 3]);
        wave_lds_fence();
        if constexpr (B16) {
#pragma unroll
            for (int t = 0; t < NV * 4; ++t) qraw[t] = qst[j * QP + (t / 4) * WAVE + 4 * blk + (t % 4)];
        } else {
#pragma unroll
            for (int t = 0; t < NV * 4; ++t) unpack_vec<T>(qst[j * QP + (t / 4) * WAVE + 4 * blk + (t % 4)], &qb[t * VE]);
#pragma unroll
            for (int c = 0; c < CB; ++c) qb[c] *= scale_log2e;
        }
    }
    floatx4 acc[EPL];                                  // [row register r][member 4 wv + i]
    float mref = M_INIT_LOG2, lrun = 0.f;
#pragma unroll
    for (int r = 0; r < EPL; ++r) acc[r] = floatx4{0.f, 0.f, 0.f, 0.f};
    struct Raw {
        RawRow<T, HL, D> kr[NE], vr[NE];
        int xe[(BIAS || DROP) ? NB : 1];               // edge ids of this lane's member with the batch's entries
    };
    for (int p0 = g_begin; p0 < g_end; p0 += GRP_CHUNK) {
        const int cnt = min(GRP_CHUNK, g_end - p0);
        int4 ent = entries[p0 + min(lane, cnt - 1)];    // lanes past the end repeat the last entry with an empty mask
        ent.y = lane < cnt ? ent.y : 0;
        auto load_half = [&](Raw &B, int b) {          // this wavefront's entries of batch b
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                const uint32_t src = (uint32_t)__builtin_amdgcn_readlane(ent.x, b + NE * wv + e);
                load_row32_raw<T, HL, D, CF>(k, src, loff, B.kr[e]);
                load_row32_raw<T, HL, D, CF>(v, src, loff, B.vr[e]);
            }
            if constexpr (BIAS || DROP) {
                // the look-ahead reaches up to 2 * NB + NB - 1 entries past the group's last one: clamped to the last
                // entry of the list's padding (all values there are the spare edge id)
#pragma unroll
                for (int e = 0; e < NB; ++e) B.xe[e] = P.grp_eids[(size_t)min(p0 + b + e, eid_last) * R + 4 * wv + j];
            }
        };
        // the score terms of a batch are fetched one batch ahead, with the edge ids that came in the batch before
        float bz[NB];
        int xd[NB];                                    // edge ids of the batch in use (dropout is keyed by them)
        auto load_bias = [&](const Raw &B) {
            if constexpr (BIAS) {
#pragma unroll
                for (int e = 0; e < NB; ++e) bz[e] = bias[(size_t)((uint32_t)B.xe[e] * (uint32_t)H) + head];
            }
            if constexpr (DROP) {
#pragma unroll
                for (int e = 0; e < NB; ++e) xd[e] = B.xe[e];
            }
        };
        auto stage_half = [&](const Raw &B, int buf) {
#pragma unroll
            for (int e = 0; e < NE; ++e)
#pragma unroll
                for (int c = 0; c < NV; ++c) {
                    kst[buf][(NE * wv + e) * PITCH + c * WAVE + lane] = make_uint4(B.kr[e].w[4 * c], B.kr[e].w[4 * c + 1], B.kr[e].w[4 * c + 2], B.kr[e].w[4 * c + 3]);
                    vst[W3 ? 0 : buf][((NE * wv + e) * NV + c) * WAVE + lane] = make_uint4(B.vr[e].w[4 * c], B.vr[e].w[4 * c + 1], B.vr[e].w[4 * c + 2], B.vr[e].w[4 * c + 3]);
                }
        };
        Raw raw;
        load_half(raw, 0);
        __syncthreads();                               // the staging area is free (q rows, the previous chunk's last batch)
        stage_half(raw, 0);
        load_bias(raw);
        load_half(raw, NB);
        __syncthreads();
        for (int b = 0, buf = 0; b < cnt; b += NB, buf ^= 1) {
            int mk[NB];
#pragma unroll
            for (int e = 0; e < NB; ++e) mk[e] = __builtin_amdgcn_readlane(ent.y, b + e);
            // all LDS reads of the batch go out first: the K rows of this lane's entry by block, the V rows as loaded
            uint4 kv[NV * 4], vv[NB][NV];
#pragma unroll
            for (int t = 0; t < NV * 4; ++t) kv[t] = kst[buf][j * PITCH + (t / 4) * WAVE + 4 * blk + (t % 4)];
#pragma unroll
            for (int e = 0; e < NB; ++e)
#pragma unroll
                for (int c = 0; c < NV; ++c) vv[e][c] = vst[W3 ? 0 : buf][(e * NV + c) * WAVE + lane];
            if constexpr (!W3) issue_loads_first();
            // scores: register e of lane 4 blk + j = (entry e, member 4 wv + j), head of the block
            floatx4 st[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) st[c] = floatx4{0.f, 0.f, 0.f, 0.f};
            if constexpr (B16) {
                // four columns per instruction, operands as loaded (v_mfma_f32_4x4x4 on bfloat16)
#pragma unroll
                for (int t = 0; t < NV * 4; ++t) {
                    st[0] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(as_bf16x4(kv[t].x, kv[t].y), as_bf16x4(qraw[t].x, qraw[t].y), st[0], 0, 0, 0);
                    st[1] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(as_bf16x4(kv[t].z, kv[t].w), as_bf16x4(qraw[t].z, qraw[t].w), st[1], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int t = 0; t < NV * 4; ++t) {
                    float kf[VE];
                    unpack_vec<T>(kv[t], kf);
#pragma unroll
                    for (int c = 0; c < VE; ++c) st[c & 3] = __builtin_amdgcn_mfma_f32_4x4x1f32(kf[c], qb[t * VE + c], st[c & 3], 0, 0, 0);
                }
            }
            float sc[NB];
#pragma unroll
            for (int e = 0; e < NB; ++e) sc[e] = block_sum<BPH>((st[0][e] + st[1][e]) + (st[2][e] + st[3][e])) * (B16 ? scale_log2e : 1.f);
#pragma unroll
            for (int e = 0; e < NB; ++e) sc[e] = ((mk[e] >> (4 * wv + j)) & 1) ? (BIAS ? fmaf(bz[e], scale_log2e, sc[e]) : sc[e]) : -INFINITY;
            const float mb = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
            if (__builtin_amdgcn_ballot_w64(mb > mref + MFMA_TAU) != 0) {
                const float mn = fmaxf(mref, mb);
                const float al = __builtin_amdgcn_exp2f(mref - mn);
                mref = mn;
                lrun *= al;
                const float a0 = quad_lane<0>(al), a1 = quad_lane<1>(al), a2 = quad_lane<2>(al), a3 = quad_lane<3>(al);
#pragma unroll
                for (int r = 0; r < EPL; ++r) {
                    acc[r][0] *= a0; acc[r][1] *= a1; acc[r][2] *= a2; acc[r][3] *= a3;
                }
            }
            float pk[NB];
#pragma unroll
            for (int e = 0; e < NB; ++e) {
                const float pe = __builtin_amdgcn_exp2f(sc[e] - mref);
                lrun += pe;                                          // the softmax denominator ignores dropout
                if constexpr (DROP) {
                    pk[e] = pe * dropout_keep((uint32_t)xd[e] * (uint32_t)H + (uint32_t)head, drop_seed, drop_thr, drop_inv);
                } else {
                    pk[e] = pe;
                }
            }
            if constexpr (B16) {
                // A = the lane's four probabilities (one per entry of the batch) rounded to bfloat16; B = column r of
                // the four V rows, gathered from the rows' registers by byte permutes
                const uint32_t p01 = (uint32_t)f32_to_bf16(pk[0]) | ((uint32_t)f32_to_bf16(pk[1]) << 16);
                const uint32_t p23 = (uint32_t)f32_to_bf16(pk[2]) | ((uint32_t)f32_to_bf16(pk[3]) << 16);
                static_assert(NV == 1 && NB == 4, "one 16-byte vector per row and lane");
                const uint32_t v0[4] = {vv[0][0].x, vv[0][0].y, vv[0][0].z, vv[0][0].w}, v1[4] = {vv[1][0].x, vv[1][0].y, vv[1][0].z, vv[1][0].w};
                const uint32_t v2[4] = {vv[2][0].x, vv[2][0].y, vv[2][0].z, vv[2][0].w}, v3[4] = {vv[3][0].x, vv[3][0].y, vv[3][0].z, vv[3][0].w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const uint32_t lo01 = __builtin_amdgcn_perm(v1[c], v0[c], 0x05040100u), lo23 = __builtin_amdgcn_perm(v3[c], v2[c], 0x05040100u);
                    const uint32_t hi01 = __builtin_amdgcn_perm(v1[c], v0[c], 0x07060302u), hi23 = __builtin_amdgcn_perm(v3[c], v2[c], 0x07060302u);
                    acc[2 * c] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(as_bf16x4(p01, p23), as_bf16x4(lo01, lo23), acc[2 * c], 0, 0, 0);
                    acc[2 * c + 1] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(as_bf16x4(p01, p23), as_bf16x4(hi01, hi23), acc[2 * c + 1], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int e = 0; e < NB; ++e) {
                    float vf[EPL];
#pragma unroll
                    for (int c = 0; c < NV; ++c) unpack_vec<T>(vv[e][c], &vf[c * VE]);
#pragma unroll
                    for (int r = 0; r < EPL; ++r) acc[r] = __builtin_amdgcn_mfma_f32_4x4x1f32(pk[e], vf[r], acc[r], 0, 0, 0);
                }
            }
            // the other buffer was last read one batch ago, before the previous barrier
            if constexpr (W3) __syncthreads();
            stage_half(raw, buf ^ 1);
            load_bias(raw);
            load_half(raw, b + 2 * NB);                // look-ahead (past the end: the last entry again, unused)
            __syncthreads();
        }
    }
    const float ls[4] = {quad_lane<0>(lrun), quad_lane<1>(lrun), quad_lane<2>(lrun), quad_lane<3>(lrun)};
    const float ms[4] = {quad_lane<0>(mref), quad_lane<1>(mref), quad_lane<2>(mref), quad_lane<3>(mref)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (rows[i] < 0) continue;
        float out[EPL];
        if (slots[i] < 0) {
            const float inv = ls[i] > 0.f ? 1.f / ls[i] : 0.f;
#pragma unroll
            for (int r = 0; r < EPL; ++r) out[r] = acc[r][i] * inv;
            store_row<T, HL, D>(o + (size_t)rows[i] * CF + coff, lane, out);
            if (lane % L::LPH == 0) lse[(size_t)rows[i] * H + head] = ls[i] > 0.f ? ms[i] + log2f(ls[i]) : 0.f;
        } else {
#pragma unroll
            for (int r = 0; r < EPL; ++r) out[r] = acc[r][i];
            store_row_ws<T, HL, D>(ws_acc + (size_t)slots[i] * CF + coff, lane, out);
            if (lane % L::LPH == 0) {
                ws_ml[((size_t)slots[i] * H + head) * 2] = ms[i];
                ws_ml[((size_t)slots[i] * H + head) * 2 + 1] = ls[i];
            }
        }
    }
}

// ---- dense tiles: groups of 16 rows, one wavefront per head ---------------------------------------------------------
// A group of TILE_R = 16 rows (or row segments) and its entries (the union of the members' neighbours, each with a
// 16-bit member mask) is walked in blocks of 16 entries as a dense 16 x 16 problem on the matrix cores: the pairs a
// block does not have are computed and masked.  Adjacent rows of a BPT graph share most neighbours (35 % of a block's
// pairs exist at L = 8192, k = 4), and a dense block costs 4 cycles per pair and head in float32 against 25-35 issue
// slots of the gather form.  Workgroup = H wavefronts, wavefront = one head, so every lane keeps 1/64 of a
// 16 x 64 tile per operand and nothing is exchanged between wavefronts.
//
// v_mfma_f32_16x16x4f32: D[i][n] += sum_k A[i][k] B[k][n], lane (c = lane % 16, g = lane / 16) supplies A[c][g] and
// B[g][c] and holds D[4 g + r][c] in register r.  Which column of a row a (step, g) pair stands for is free as long as
// A and B agree, so operands are held as 16-byte vectors (the members' rows are loaded that way; the entries' rows
// reach the first layout below through LDS, see tile_rows_to_operand):
//   scores S^T = K Q^T : A = K[entry e(c)][16 t + 4 g + e], B = q[member c][16 t + 4 g + e] (steps t, e = 0..3), where
//                        row c of the product is entry e(c) = 4 (c % 4) + c / 4 of the block, so that
//                        register r of lane (c, g) = score of (entry 4 r + g, member c);
//   output O += P V    : A = register r of the probabilities as they stand (row = member c, k = g stands for entry
//                        4 r + g), B = V[entry 4 r + g][4 c + nb]; register r' of accumulator nb of lane (c, g) =
//                        O[member 4 g + r'][4 c + nb]: four consecutive columns per lane, 256 contiguous bytes per
//                        member and 16 lanes.  Step r of such a product covers the neighbouring entries 4 r .. 4 r + 3:
//                        past the end of a group's entry list (half of its last block on average) steps are left out.
//   (The bfloat16 kernels below keep entry 4 g + r in register r: their products over the entries are one instruction.)
// Softmax state is per lane for member c (the four lanes of a member hold partial denominators that are added at the
// end); the exponent reference is raised lazily as in the matrix-core forward above.
constexpr int TILE_R = 16;
constexpr int TILE_CHUNK = 128;                     // entries staged in LDS at a time = 8 blocks

typedef float floatx4v __attribute__((ext_vector_type(4)));
typedef uint32_t uintx2v __attribute__((ext_vector_type(2)));

typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
typedef float floatx2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    union { bf16x2v v; uint32_t u; } r;
    r.v = __builtin_convertvector(floatx2v{lo, hi}, bf16x2v);      // round to nearest even
    return r.u;
}

// What a tile costs beside its blocks - sums and maxima over lane groups, the rows it stores, masks - is kept to few vector instructions:
// float32 products (v_mfma_f32_16x16x4) and vector arithmetic do not run side by side on a SIMD, whichever wavefronts they come from (a
// wavefront of each takes the sum of their times: 288 + 351 -> 628 cycles; bfloat16 16 x 16 x 32 products 145 + 345 -> 405).  Lane groups
// are swapped instead of looked up through the LDS crossbar, masks are one bit field extract and one and, a member's row or slot is one
// word, rows go to 32-bit offsets from a uniform base, bfloat16 is rounded by the hardware and sums that are still zero are not rescaled;
// the float32 destination side reads masks and pair numbers back from LDS and no longer spills.  Same results to the bit.  Kernels before ->
// after, forward / destination / source side: bfloat16, L = 8192, k = 4 18.5 / 25.6 / 29.2 -> 17.1 / 24.6 / 26.5 us, 16 heads at L = 32768, k = 8
// 185 / 241 / 339 -> 184 / 240 / 333; float32, L = 8192 35.3 / 59.3 / 42.8 -> 34.1 / 58.1 / 40.9, 32-graph batch 68.6 / 105.1 / 89.4 -> 67.0 / 101.6 / 87.4.
// x of the lanes c, 16 + c, 32 + c and 48 + c, combined, in all four of them
__device__ __forceinline__ float groups_sum(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ __forceinline__ float groups_max(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// x where bit `bit` of the mask is set, -inf (0) where it is not
__device__ __forceinline__ float where_pair(int mask, int bit, float x) {
    const int m = __builtin_amdgcn_sbfe(mask, bit, 1);
    return __int_as_float((__float_as_int(x) & m) | (0xff800000 & ~m));
}
__device__ __forceinline__ float where_pair_or_zero(int mask, int bit, float x) {
    return __int_as_float(__float_as_int(x) & __builtin_amdgcn_sbfe(mask, bit, 1));
}
__device__ __forceinline__ float lane_bcast(float x, int src_lane) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(src_lane << 2, __float_as_int(x)));
}
__device__ __forceinline__ int lane_bcast(int x, int src_lane) { return __builtin_amdgcn_ds_bpermute(src_lane << 2, x); }

// Common start of the tile kernels.  HW heads (= wavefronts) per workgroup: workgroup b handles head slice
// (b / 8) % (H / HW) of group (b / 8) / (H / HW) of XCD b % 8's range.
struct TileCtx {
    int lane, wv, c, g, head, p_begin, p_end, part;
    int2 member;                 // (row, slot) of member c
    uint32_t offa, offv;         // byte offsets of this lane inside a node row: its 16-column slice of the head (operands of the
                                 // products that contract over columns, + 64 t bytes per step), and its columns 4 c .. 4 c + 3
};

template <typename T, int H, int D, int HW, bool NARROW = false, int SP = 1>
__device__ __forceinline__ bool tile_begin(const bpt_plan &P, TileCtx &t, const Narrow &nw, unsigned block = blockIdx.x) {
    static_assert(D == 64 && (H * SP) % HW == 0 && HW % SP == 0 && (sizeof(T) == 4 || sizeof(T) == 2), "64 columns per head: one 16-column slice per lane group");
    static_assert(!NARROW || SP == 1 || SP == HW, "heads a workgroup has past the last one leave its barrier alone");
    constexpr int HEADS = HW / SP;
    const int HS = NARROW ? nw.slices : H / HEADS;
    t.lane = threadIdx.x & (WAVE - 1);
    t.wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    t.c = t.lane & 15;
    t.g = t.lane >> 4;
    const int x = block & 7, w = (int)(block >> 3) / HS;
    const int grp = __builtin_amdgcn_readfirstlane(P.grp_chunks[x]) + w;
    if (grp >= __builtin_amdgcn_readfirstlane(P.grp_chunks[x + 1])) return false;
    t.member = reinterpret_cast<const int2 *>(P.grp_members)[(size_t)grp * TILE_R + t.c];
    t.p_begin = __builtin_amdgcn_readfirstlane(P.grp_ptr[grp]);
    t.p_end = __builtin_amdgcn_readfirstlane(P.grp_ptr[grp + 1]);
    t.part = SP > 1 ? t.wv / HEADS : 0;
    if constexpr (SP > 1) {
        const int per = ((t.p_end - t.p_begin + TILE_R * SP - 1) / (TILE_R * SP)) * TILE_R;
        t.p_begin = min(t.p_begin + t.part * per, t.p_end);
        t.p_end = min(t.p_begin + per, t.p_end);
    }
    t.head = (int)((block >> 3) % HS) * HEADS + (SP > 1 ? t.wv % HEADS : t.wv);
    if (NARROW) {
        if (t.head >= nw.heads) return false;
        t.offa = (uint32_t)(t.head * nw.d * sizeof(T));
        t.offv = (uint32_t)((t.head * nw.d + narrow_col(nw, t.c)) * sizeof(T));
        return true;
    }
    t.offa = (uint32_t)((t.head * D + 4 * t.g) * sizeof(T));
    t.offv = (uint32_t)((t.head * D + 4 * t.c) * sizeof(T));
    return true;
}

// The entry list of a group is staged, TILE_CHUNK entries at a time, in a wavefront-private piece of LDS as (neighbour,
// mask) pairs: every lane needs five of them per block (its A-operand row and the four rows / masks of its lane
// group), which would otherwise be five dependent global loads in front of every block's row loads.
struct TileEntryRegs {
    int4 x[TILE_CHUNK / WAVE];
};
// first half: the loads.  A kernel asks for its first piece before it reads its members' rows, so that the two round trips
// run side by side; in source order the compiler puts the members' arithmetic (and its wait) in front of these loads.
__device__ __forceinline__ void tile_ask_entries(const bpt_plan &P, int p0, int cnt, int lane, TileEntryRegs &r) {
    const int4 *entries = reinterpret_cast<const int4 *>(P.grp_entries);
#pragma unroll
    for (int u = 0; u < TILE_CHUNK / WAVE; ++u) r.x[u] = entries[p0 + min(u * WAVE + lane, cnt - 1)];   // past the end: the last entry again
}
// second half: into the wavefront's piece of LDS
__device__ __forceinline__ void tile_put_entries(const TileEntryRegs &r, int2 *lds, int cnt, int lane, int *first = nullptr) {
#pragma unroll
    for (int u = 0; u < TILE_CHUNK / WAVE; ++u) {
        const int e = u * WAVE + lane;
        int nbr = r.x[u].x, mask = r.x[u].y;
        asm volatile("" : "+v"(nbr), "+v"(mask));                 // (the values are used from here on: nothing of this half moves up to the loads)
        lds[e] = make_int2(nbr, e < cnt ? mask : 0);              // past the end: an empty mask
        if (first) first[e] = r.x[u].z;                          // number of the entry's first pair (members follow in ascending order)
    }
    wave_lds_fence();
}
__device__ __forceinline__ void tile_stage_entries(const bpt_plan &P, int2 *lds, int p0, int cnt, int lane, int *first = nullptr) {
    TileEntryRegs r;
    tile_ask_entries(P, p0, cnt, lane, r);
    tile_put_entries(r, lds, cnt, lane, first);
}
// number of the pair (entry, member c) among the plan's pairs: the entry's first pair + the members before c in its mask
__device__ __forceinline__ int tile_pair_number(int first, int mask, int c) { return first + __popc((uint32_t)mask & ((1u << c) - 1u)); }

// this lane's 16 columns of a node row (bytes offa + 64 t), as the A or B operand of a product over columns
template <bool NARROW>
__device__ __forceinline__ floatx4v tile_load4(const char *row, int t, int g, const Narrow &nw) {      // the four of step t
    if constexpr (NARROW) {
        const int quad = 4 * (4 * t + g), col = min(quad, nw.d - 4);
        const floatx4u x = *reinterpret_cast<const floatx4u *>(row + 4 * col);
        return floatx4v{col >= quad ? x[0] : 0.f, col + 1 >= quad ? x[1] : 0.f, col + 2 >= quad ? x[2] : 0.f, col + 3 >= quad ? x[3] : 0.f};
    } else {
        return *reinterpret_cast<const floatx4v *>(row + 64 * t);
    }
}
template <bool NARROW>
__device__ __forceinline__ void tile_load16(const char *row, float (&out)[16], int g, const Narrow &nw) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const floatx4v x = tile_load4<NARROW>(row, t, g, nw);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[4 * t + e] = x[e];
    }
}
// this lane's four columns of an entry's row
template <bool NARROW> __device__ __forceinline__ float4 tile_row4(const char *p) {
    if constexpr (NARROW) {
        const floatx4u x = *reinterpret_cast<const floatx4u *>(p);
        return make_float4(x[0], x[1], x[2], x[3]);
    } else {
        return *reinterpret_cast<const float4 *>(p);
    }
}

// register r of the result of lane (c, g) = sum over the 64 columns of a[row 4 g + r] * b[member c], a[row c] = what lane c passes
__device__ __forceinline__ floatx4v tile_dot(const float (&a)[16], const float (&b)[16]) {
    floatx4v s0 = floatx4v{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i + 1], b[i + 1], s1, 0, 0, 0);
    }
    return s0 + s1;
}

// acc[nb][r'] (member 4 g + r', column 4 c + nb) += sum over the block's entries of w[member][entry] * row[entry][column]:
// w = this lane's four weights (member c with entries 4 r + g), rows = columns 4 c .. 4 c + 3 of the rows of entries 4 r + g.
// Step r of the product stands for the four NEIGHBOURING entries 4 r .. 4 r + 3 (one per lane group), so a step whose
// entries lie past the end of the group's list (nv = the block's entries that exist) is left out.
__device__ __forceinline__ void tile_axpy_upto(const float (&w)[4], const float4 (&rows)[4], floatx4v (&acc)[4], int nv) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (4 * r < nv) {
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[r], rows[r].x, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[r], rows[r].y, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[r], rows[r].z, acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[r], rows[r].w, acc[3], 0, 0, 0);
        } else {
            // (the step's rows are marked as read: left in flight, they would make the next block's loads wait for
            // everything that is outstanding, this block's stores included)
            asm volatile("" ::"v"(rows[r].x), "v"(rows[r].y), "v"(rows[r].z), "v"(rows[r].w));
        }
    }
}

// The members' result rows: whole rows go to `out` (scaled by inv[member] where given), segments of split rows to the
// workspace in natural column order.  Whole rows are written past the L2 (non-temporal): this kernel does not read them again,
// and written the ordinary way they push out the neighbours' rows that the other tiles of the XCD are about to read.  Sum of a
// training step's kernels, new inputs every pass, before -> now: 32-graph batch float32 284 -> 274 us (forward 76 -> 70.5),
// L = 8192 float32 161 -> 157, bfloat16 91 -> 85.5 (forward 21.8 -> 19.2), L = 32768, k = 4 649 -> 632, window 128 97 -> 94.5;
// L = 512 level.  The same on the stores of (p, ds), which the source side reads soon, or on its loads of them: 47 -> 50.5 and
// 47 -> 55 us for the source side of L = 8192; on the loads of the members' rows: destination side 58 -> 61.6.
// where: per member, its row, -1 where there is none, -2 - slot for a segment of a split row (tile_where of lane c for member c)
__device__ __forceinline__ int tile_where(int2 member) { return member.x < 0 ? -1 : member.y < 0 ? member.x : -2 - member.y; }
template <int H, int D, bool SCALE, bool NARROW, typename T>
__device__ __forceinline__ void tile_store_row(const TileCtx &t, int r, float4 x, float inv_c, T *__restrict__ out, float *__restrict__ ws,
                                               const Narrow &nw, int where, T *__restrict__ also = nullptr) {      // also (NARROW): second copy of whole rows
    const int m = 4 * t.g + r;                                    // the member whose row this lane stores a piece of
    int at = lane_bcast(where, m);
    const float inv = SCALE ? lane_bcast(inv_c, m) : 1.f;
    if (NARROW && 4 * t.c >= nw.d) at = -1;
    const int col = NARROW ? narrow_col(nw, t.c) : 4 * t.c;
    if (at >= 0) {
        if (SCALE) { x.x *= inv; x.y *= inv; x.z *= inv; x.w *= inv; }
        // (node tensors end before 4 GiB)
        const uint32_t off = NARROW ? ((uint32_t)at * (uint32_t)(nw.heads * nw.d) + (uint32_t)(t.head * nw.d + col)) * (uint32_t)sizeof(T)
                                    : (uint32_t)at * (uint32_t)(H * D * sizeof(T)) + t.offv;
        char *const to = reinterpret_cast<char *>(out) + off;
        if constexpr (sizeof(T) == 4) {
            if constexpr (NARROW) {
                *reinterpret_cast<floatx4u *>(to) = floatx4u{x.x, x.y, x.z, x.w};
                if (also) *reinterpret_cast<floatx4u *>(reinterpret_cast<char *>(also) + off) = floatx4u{x.x, x.y, x.z, x.w};
            } else __builtin_nontemporal_store(floatx4v{x.x, x.y, x.z, x.w}, reinterpret_cast<floatx4v *>(to));
        } else {
            const uint2 y = make_uint2(pack_bf16(x.x, x.y), pack_bf16(x.z, x.w));
            if constexpr (NARROW) {
                *reinterpret_cast<uintx2u *>(to) = uintx2u{y.x, y.y};
                if (also) *reinterpret_cast<uintx2u *>(reinterpret_cast<char *>(also) + off) = uintx2u{y.x, y.y};
            } else __builtin_nontemporal_store(uintx2v{y.x, y.y}, reinterpret_cast<uintx2v *>(to));
        }
    } else if (at < -1) {
        float *const to = ws + (size_t)(-2 - at) * (NARROW ? nw.h * D : H * D) + t.head * D + col;
        if constexpr (NARROW) *reinterpret_cast<floatx4u *>(to) = floatx4u{x.x, x.y, x.z, x.w};
        else *reinterpret_cast<float4 *>(to) = x;
    }
}
template <int H, int D, bool SCALE, bool NARROW, typename T>
__device__ __forceinline__ void tile_store_rows(const TileCtx &t, const floatx4v (&acc)[4], float inv_c, T *__restrict__ out,
                                                float *__restrict__ ws, const Narrow &nw, T *__restrict__ also = nullptr) {
    const int where = tile_where(t.member);
#pragma unroll
    for (int r = 0; r < 4; ++r)
        tile_store_row<H, D, SCALE, NARROW>(t, r, make_float4(acc[0][r], acc[1][r], acc[2][r], acc[3][r]), inv_c, out, ws, nw, where, also);
}

// SP > 1: SP wavefronts of a workgroup share a tile and head, each walks a contiguous SP-th of the tile's blocks (tile_begin),
// and what they have summed up meets in LDS: every wavefront leaves its accumulators in its own piece, [r][lane] so that
// the 16-byte accesses of a wavefront are contiguous, and after one barrier adds up and stores the members 4 g + r of its
// 4 / SP registers r.  Parts are added in their order: the same bits on every run.
constexpr int TILE_PART_FLOATS = TILE_R * 64;                     // accumulators of a wavefront
__device__ __forceinline__ void tile_park(float *part, const floatx4v (&acc)[4], int lane) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
        *reinterpret_cast<floatx4v *>(part + (r * WAVE + lane) * 4) = floatx4v{acc[0][r], acc[1][r], acc[2][r], acc[3][r]};
}
// sum over the parts of register r, part s (`stride` floats after part s - 1) weighted with wgt[s] of the lane's member
template <int SP, bool WEIGHTED>
__device__ __forceinline__ float4 tile_meet(const float *part0, int stride, int r, const TileCtx &t, const float (&wgt)[SP]) {
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int s = 0; s < SP; ++s) {
        const floatx4v y = *reinterpret_cast<const floatx4v *>(part0 + s * stride + (r * WAVE + t.lane) * 4);
        if constexpr (WEIGHTED) {
            const float w = lane_bcast(wgt[s], 4 * t.g + r);
            x.x = fmaf(w, y[0], x.x); x.y = fmaf(w, y[1], x.y); x.z = fmaf(w, y[2], x.z); x.w = fmaf(w, y[3], x.w);
        } else {
            x.x += y[0]; x.y += y[1]; x.z += y[2]; x.w += y[3];
        }
    }
    return x;
}
// the same for a kernel without weights: parked accumulators of the SP parts -> result rows
template <int SP, int H, int D, bool NARROW, typename T>
__device__ __forceinline__ void tile_meet_and_store(const float *part0, int stride, const TileCtx &t, T *__restrict__ out, float *__restrict__ ws,
                                                    const Narrow &nw) {
    constexpr int RS = 4 / SP;
    const float none[SP] = {};
#pragma unroll
    for (int i = 0; i < RS; ++i) {
        const int r = t.part * RS + i;
        tile_store_row<H, D, false, NARROW>(t, r, tile_meet<SP, false>(part0, stride, r, t, none), 1.f, out, ws, nw, tile_where(t.member));
    }
}
// ... and for the forward: with the parts' exponent references and denominators (left behind the accumulators by member)
constexpr int TILE_PART_FWD_FLOATS = TILE_PART_FLOATS + 2 * TILE_R;
template <int SP, int H, int D, bool NARROW, typename T>
__device__ __forceinline__ void tile_meet_forward(float *mine, const float *part0, int stride, const TileCtx &t, const floatx4v (&acc)[4], float &mref,
                                                  float &lt, T *__restrict__ out, float *__restrict__ ws, const Narrow &nw,
                                                  T *__restrict__ also) {
    constexpr int RS = 4 / SP;
    tile_park(mine, acc, t.lane);
    if (t.g == 0) {
        mine[TILE_PART_FLOATS + 2 * t.c] = mref;
        mine[TILE_PART_FLOATS + 2 * t.c + 1] = lt;
    }
    __syncthreads();
    float wgt[SP], l = 0.f, M = M_INIT_LOG2;
#pragma unroll
    for (int s = 0; s < SP; ++s) {
        wgt[s] = part0[s * stride + TILE_PART_FLOATS + 2 * t.c];
        M = fmaxf(M, wgt[s]);
    }
#pragma unroll
    for (int s = 0; s < SP; ++s) {
        wgt[s] = __builtin_amdgcn_exp2f(wgt[s] - M);
        l = fmaf(wgt[s], part0[s * stride + TILE_PART_FLOATS + 2 * t.c + 1], l);
    }
    mref = M;
    lt = l;
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int i = 0; i < RS; ++i) {
        const int r = t.part * RS + i;
        tile_store_row<H, D, true, NARROW>(t, r, tile_meet<SP, true>(part0, stride, r, t, wgt), inv, out, ws, nw, tile_where(t.member), also);
    }
}

// Edge ids of this lane's four pairs of a block, (entry first_entry + step * r, member c): what the dropout hash and the score term are
// indexed by (n_edges, the spare row, where the pair does not exist; past the group's end the last entry is read again).
__device__ __forceinline__ void tile_pair_eids(const bpt_plan &P, int first_entry, int p_end, int c, int (&xe)[4], int step = 1) {
#pragma unroll
    for (int r = 0; r < 4; ++r) xe[r] = P.grp_eids[(size_t)min(first_entry + step * r, p_end - 1) * TILE_R + c];
}
// Which entry of a block lane c loads as row c of the products over the columns, in the float32 tile kernels: the
// scores of entries 4 r + g have to come out in register r of lane group g (row 4 g + r of the product), so that step r
// of the products over the entries stands for four NEIGHBOURING entries and can be left out past the end of the list.
__device__ __forceinline__ int tile_entry_of_row(int c) { return 4 * (c & 3) + (c >> 2); }
// Where the score term of the pair (entry, member c) sits and its gradient goes.  BIAS == 1, stored by edge id: row eid
// of (n_edges + 1, H), the spare last row for a pair that does not exist.  BIAS == 2, stored in the plan's own order:
// head-major at the pair's number, x[head * n_edges + number]: the lanes of an entry touch one run of memory and no
// index is read on the way; a pair that does not exist gets a neighbour's place, which is read and not used.
template <int H, int BIAS>
__device__ __forceinline__ uint32_t tile_bias_at(const bpt_plan &P, int head, int eid, int number) {
    if constexpr (BIAS == 2) return (uint32_t)head * (uint32_t)P.n_edges + (uint32_t)min(number, (int)P.n_edges - 1);
    else return (uint32_t)eid * (uint32_t)H + (uint32_t)head;
}

// The rows of a block's entries come from memory in the layout of the products over the entries (lane (c, g): columns
// 4 c .. 4 c + 3 of the rows of entries 4 r + g: the sixteen lanes of a lane group read one row's 256 contiguous bytes).
// The products over the COLUMNS want lane c to hold sixteen columns of ONE row (entry tile_entry_of_row(c)); loaded that
// way, neighbouring lanes read different rows and the texture addresser spends four cycles on every group of four lanes
// instead of one.  So the rows are loaded once, in the first layout, and turned in a wavefront-private piece of LDS:
// rows of TILE_KT_STRIDE floats (64 + 4: the sixteen rows of a read fall on different banks).
constexpr int TILE_KT_STRIDE = 68;
template <bool NARROW>
__device__ __forceinline__ void tile_rows_to_operand(float *kt, const float4 (&rows)[4], int c, int g, float (&out)[16], const Narrow &nw) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
        *reinterpret_cast<floatx4v *>(kt + (4 * r + g) * TILE_KT_STRIDE + 4 * c) =
            floatx4v{narrow_again<NARROW>(nw, c, 0) ? 0.f : rows[r].x, narrow_again<NARROW>(nw, c, 1) ? 0.f : rows[r].y,
                     narrow_again<NARROW>(nw, c, 2) ? 0.f : rows[r].z, narrow_again<NARROW>(nw, c, 3) ? 0.f : rows[r].w};
    wave_lds_fence();
    const float *src = kt + tile_entry_of_row(c) * TILE_KT_STRIDE + 4 * g;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const floatx4v x = *reinterpret_cast<const floatx4v *>(src + 16 * t);
        out[4 * t] = x[0]; out[4 * t + 1] = x[1]; out[4 * t + 2] = x[2]; out[4 * t + 3] = x[3];
    }
    wave_lds_fence();                                             // (read before the next block's rows are written)
}

// The members' rows likewise: lane (c, g) asks for columns 4 c .. 4 c + 3 of the row of member 4 g + r, and tile_rows_to_operand gives lane c
// the row of member c: 16 cycles of the texture addresser a load instead of 64.  Destination side, 32-graph batch 102.8 -> 99.7 us, 6 x 50 with
// dropout 90.9 -> 87.4 and its forward 97.9 -> 96.4, L = 8192, k = 4 level.  (The forward that asks for its K rows a block ahead has no
// registers for it: asked for with the entries and turned behind the first K rows, it spills: 32.8 -> 38.0 and 67 -> 75.)
template <bool NARROW, typename T>
__device__ __forceinline__ void tile_ask_members(const TileCtx &t, const T *base, uint32_t RB, float4 (&rows)[4]) {
    const int row = max(t.member.x, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r)
        rows[r] = tile_row4<NARROW>(reinterpret_cast<const char *>(base) + ((uint32_t)lane_bcast(row, 4 * t.g + r) * RB + t.offv));
}

// Block after block, a block's loads ahead of its products.  Forms measured at L = 8192, k = 4 (1217 tiles of 4 blocks) and
// dropped: the rows of the next block loaded while one is used (a two-stage register pipeline: 47 us against 44, a wavefront
// per SIMD fewer; on few, tall tiles it was the better form until the parts of a tile came to be walked side by side, see
// tile_parts), groups of 32 rows (two member blocks per wavefront sharing the K / V
// registers: a third fewer rows through the L1s, two or three wavefronts per SIMD, 56 us; two wavefronts per head in step
// on the same entries, one member block each, so that the L1 fetches a row once: 60 us: the time follows the number
// of 16 x 16 blocks, 4716 against 6324, not the bytes), five or six wavefronts per SIMD by spilling (53 / 85 us).
template <typename Blk, typename Issue, typename Compute>
__device__ __forceinline__ void tile_walk(int nblk, Issue &&issue, Compute &&compute) {
    for (int b = 0; b < nblk; ++b) {
        Blk A;
        issue(A, b);
        issue_loads_first();
        compute(A);
        issue_loads_first();
    }
}

// The rows a block needs FIRST (the K rows of its scores) are asked for one block ahead, the others (V) when the block
// begins: sixteen more registers instead of the thirty-two of the two-stage pipeline, so four wavefronts per SIMD stay.
// once_loads_left(): called once the first loads have left, for work that waits for loads asked for before them.
template <typename Blk, typename IssueFirst, typename IssueRest, typename Compute, typename Hook>
__device__ __forceinline__ void tile_walk_first_ahead(int nblk, IssueFirst &&first, IssueRest &&rest, Compute &&compute, Hook &&once_loads_left) {
    Blk A, B;
    first(A, 0);
    issue_loads_first();
    once_loads_left();
    int b = 0;
    for (; b + 2 < nblk; b += 2) {
        rest(A, b);
        first(B, b + 1);
        issue_loads_first();
        compute(A);
        issue_loads_first();
        rest(B, b + 1);
        first(A, b + 2);
        issue_loads_first();
        compute(B);
        issue_loads_first();
    }
    rest(A, b);
    if (b + 1 < nblk) {
        first(B, b + 1);
        issue_loads_first();
        compute(A);
        issue_loads_first();
        rest(B, b + 1);
        issue_loads_first();
        compute(B);
    } else {
        issue_loads_first();
        compute(A);
    }
    issue_loads_first();
}

template <typename T, int H, int D, int HW, bool DROP, int BIAS, bool NARROW = false, int SP = 1>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(4))) void k_attn_fwd_tile(
    bpt_plan P, const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v, T *__restrict__ o, float *__restrict__ lse,
    float *__restrict__ ws_acc, float *__restrict__ ws_ml, float scale_log2e, uint32_t drop_thr, uint32_t drop_seed, float drop_inv,
    const float *__restrict__ bias, Narrow nw, Keep keep) {
    const int Hs = NARROW ? nw.h : H;                             // heads as lse, workspace and dropout keys count them
    const uint32_t RB = NARROW ? (uint32_t)(nw.heads * nw.d) * sizeof(T) : (uint32_t)(H * D * sizeof(T));        // bytes of a node row
    int block = (int)blockIdx.x;
    if constexpr (NARROW) block = keep_or_tile<HW * WAVE>(keep);
    if (NARROW && block < 0) return;
    T *const o_keep = NARROW ? reinterpret_cast<T *>(keep.o) : nullptr;
    TileCtx t;
    if (!tile_begin<T, H, D, HW, NARROW, SP>(P, t, nw, (unsigned)block)) return;
    __shared__ int2 ent_lds[HW][TILE_CHUNK];
    __shared__ int fst_lds[HW][BIAS == 2 ? TILE_CHUNK : 1];      // the entries' first pair numbers: where a term in pair order sits
    int2 *ent = ent_lds[t.wv];
    int *fst = BIAS == 2 ? fst_lds[t.wv] : nullptr;
    __shared__ __attribute__((aligned(16))) float kt_lds[HW][TILE_R * TILE_KT_STRIDE];
    float *kt = kt_lds[t.wv];
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    issue_loads_first();
    const int c = t.c, g = t.g;
    const char *kb = reinterpret_cast<const char *>(k), *vb = reinterpret_cast<const char *>(v);
    float qb[16];
    // The members' q rows are asked for behind the first block's K rows: asked for here, ahead of the loop, they are waited
    // for before the entry list is (one more round trip in front of the K rows).  They stay as they are and the scores are
    // scaled instead, so nothing has to happen to them between their arrival and the first product.
    const char *const qrow = reinterpret_cast<const char *>(q) + (size_t)max(t.member.x, 0) * RB + t.offa;
    // (with the score term the sixteen registers are not there; with dropout they just are, and it does not pay: L = 8192 level, 6 x 50
    // with dropout 97.7 -> 100 us)
    constexpr bool AHEAD = !DROP && BIAS == 0;
    if constexpr (!AHEAD) {
        float4 qr[4];
        tile_ask_members<NARROW>(t, q, RB, qr);
        tile_rows_to_operand<NARROW>(kt, qr, c, g, qb, nw);
    }
    floatx4v acc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
    float mref = M_INIT_LOG2, lrun = 0.f;
    bool fresh = true;                                            // nothing has been summed up yet
    struct Blk {
        float4 kq[4];                                             // columns 4 c .. 4 c + 3 of the K rows of entries 4 r + g
        float4 vr[4];
        int mk[4], nv;                                            // bit c of mk[r]: the pair (entry 4 r + g, member c) exists; nv: entries of the block that exist
        int xe[DROP || BIAS == 1 ? 4 : 1];
        float bz[BIAS ? 4 : 1];
    };
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane, fst);
        auto issue_k = [&](Blk &B, int b) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                B.kq[r] = tile_row4<NARROW>(kb + ((uint32_t)ent[TILE_R * b + 4 * r + g].x * RB + t.offv));
        };
        auto issue_rest = [&](Blk &B, int b) {
            if constexpr (DROP || BIAS == 1) tile_pair_eids(P, p0 + TILE_R * b + g, t.p_end, c, B.xe, 4);
            B.nv = min(TILE_R, cnt - TILE_R * b);
            int idxv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int2 en = ent[TILE_R * b + 4 * r + g];
                idxv[r] = en.x; B.mk[r] = en.y;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                B.vr[r] = tile_row4<NARROW>(vb + ((uint32_t)idxv[r] * RB + t.offv));
            if constexpr (BIAS == 1) {
#pragma unroll
                for (int r = 0; r < 4; ++r) B.bz[r] = bias[tile_bias_at<H, 1>(P, t.head, B.xe[BIAS == 1 ? r : 0], 0)];
            }
            if constexpr (BIAS == 2) {
#pragma unroll
                for (int r = 0; r < 4; ++r) B.bz[r] = bias[tile_bias_at<H, 2>(P, t.head, 0, tile_pair_number(fst[TILE_R * b + 4 * r + g], B.mk[r], c))];
            }
        };
        auto compute = [&](const Blk &B) {
            float kr[16];
            tile_rows_to_operand<NARROW>(kt, B.kq, c, g, kr, nw);
            const floatx4v st = tile_dot(kr, qb);
            float sc[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                sc[r] = where_pair(B.mk[r], c, BIAS ? fmaf(st[r], scale_log2e, B.bz[BIAS ? r : 0] * scale_log2e) : st[r] * scale_log2e);
            const float mb = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
            if (__builtin_amdgcn_ballot_w64(mb > mref + MFMA_TAU) != 0) {
                const float mn = fmaxf(mref, groups_max(mb));    // over the four lanes of member c
                const float al = __builtin_amdgcn_exp2f(mref - mn);
                mref = mn;
                if (!fresh) {
                    lrun *= al;
                    // register r' of the accumulators belongs to member 4 g + r': its factor sits in lane 4 g + r'
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float a = lane_bcast(al, 4 * g + r);
#pragma unroll
                        for (int nb = 0; nb < 4; ++nb) acc[nb][r] *= a;
                    }
                }
            }
            fresh = false;
            float pr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pr[r] = __builtin_amdgcn_exp2f(sc[r] - mref);
                lrun += pr[r];                                   // the softmax denominator ignores dropout
                if constexpr (DROP)
                    pr[r] *= dropout_keep((uint32_t)B.xe[DROP ? r : 0] * (uint32_t)Hs + (uint32_t)t.head, drop_seed, drop_thr, drop_inv);
            }
            tile_axpy_upto(pr, B.vr, acc, B.nv);
        };
        auto issue = [&](Blk &B, int b) { issue_k(B, b); issue_rest(B, b); };
        if constexpr (!AHEAD) tile_walk<Blk>(nblk, issue, compute);
        else tile_walk_first_ahead<Blk>(nblk, issue_k, issue_rest, compute, [&]() { if (p0 == t.p_begin) tile_load16<NARROW>(qrow, qb, g, nw); });
        wave_lds_fence();                                         // the piece is read to the end before the next one is staged
    }
    float lt = groups_sum(lrun);                                 // denominator of member c, in its four lanes
    if constexpr (SP > 1) {
        static_assert(TILE_PART_FWD_FLOATS <= TILE_R * TILE_KT_STRIDE, "a part fits its wavefront's piece");
        tile_meet_forward<SP, H, D, NARROW>(kt, kt_lds[t.wv % (HW / SP)], (HW / SP) * TILE_R * TILE_KT_STRIDE, t, acc, mref, lt, o, ws_acc, nw, o_keep);
        if (t.part != 0) return;
    } else {
        tile_store_rows<H, D, true, NARROW>(t, acc, lt > 0.f ? 1.f / lt : 0.f, o, ws_acc, nw, o_keep);
    }
    if (g == 0 && t.member.x >= 0) {                              // lanes 0 .. 15: one member each
        if (t.member.y < 0) {
            lse[(size_t)t.member.x * Hs + t.head] = lt > 0.f ? mref + log2f(lt) : 0.f;
        } else {
            ws_ml[((size_t)t.member.y * Hs + t.head) * 2] = mref;
            ws_ml[((size_t)t.member.y * Hs + t.head) * 2 + 1] = lt;
        }
    }
}

// Backward on tiles, destination side: per block the scores and dO . v of all 16 x 16 pairs (two products over the
// columns, the K and V rows turned in LDS from the layout they are loaded in), p = 2^(s - lse),
// ds = p (dO . v - delta) scale, dq += ds K (third product, on the K rows as loaded).  With dropout or a score term the
// kernel is compiled for three wavefronts per SIMD: at four it keeps the members' q rows in scratch memory and reads
// them back for every block (83 against 58 us with dropout at L = 8192, k = 4).
// (p, ds) of the pairs that exist go to a scratch in THIS side's order, compact:
// pds[head * n_edges + t] for the pair number t of (entry, member) = the entry's first pair + the rank of the member in
// its mask, so the lanes of an entry write one contiguous run and the runs of consecutive entries follow each other.  The
// source side looks its pairs up there through its pair mapping (grp_pairs = this side's pair numbers).  Writing in the
// source side's layout instead (scattered 8-byte stores here, contiguous reads there) cost this kernel a third of its
// time (126 against 85 us at L = 4096, k = 32); letting the source side recompute p and ds (two more products there,
// delta (n, H) handed over) measured slower than either on every graph tried.
template <typename T, int H, int D, int HW, bool DROP, int BIAS, bool NARROW = false, int SP = 1>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(DROP || BIAS ? 3 : 4))) void k_attn_bwd_dst_tile(
    bpt_plan P, const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v, const T *__restrict__ o,
    const T *__restrict__ d_o, const float *__restrict__ lse, T *__restrict__ dq, float2 *__restrict__ pds, float *__restrict__ ws_dq,
    float scale, float scale_log2e, uint32_t drop_thr, uint32_t drop_seed, float drop_inv, const float *__restrict__ bias,
    float *__restrict__ ds_out, Narrow nw) {
    const int Hs = NARROW ? nw.h : H;
    const uint32_t RB = NARROW ? (uint32_t)(nw.heads * nw.d) * sizeof(T) : (uint32_t)(H * D * sizeof(T));
    TileCtx t;
    if (!tile_begin<T, H, D, HW, NARROW, SP>(P, t, nw)) return;
    __shared__ int2 ent_lds[HW][TILE_CHUNK];
    __shared__ int fst_lds[HW][TILE_CHUNK];
    int2 *ent = ent_lds[t.wv];
    int *fst = fst_lds[t.wv];
    __shared__ __attribute__((aligned(16))) float kt_lds[HW][TILE_R * TILE_KT_STRIDE];
    float *kt = kt_lds[t.wv];
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    issue_loads_first();
    const int c = t.c, g = t.g;
    const char *kb = reinterpret_cast<const char *>(k), *vb = reinterpret_cast<const char *>(v);
    const size_t mrow = (size_t)max(t.member.x, 0) * RB + t.offa;
    float2 *const pds_h = pds + (size_t)t.head * (size_t)P.n_edges;     // this head's part of the scratch
    // the member's dO columns live in LDS (lane-major, read back before every product with them): with them in registers
    // the kernel needs 144 and a SIMD holds three wavefronts, without them 128 and four
    __shared__ floatx4v dob_lds[HW / SP][4][WAVE];
    floatx4v(&dob_h)[4][WAVE] = dob_lds[t.wv % (HW / SP)];
    // (q stays as it is and the scores are scaled, as in the forward: the same roundings in both)
    float qb[16], delta, lse_c;
    if constexpr (SP > 1) {
        // each part reads its 4 / SP steps of the members' rows for all of them
        __shared__ floatx4v q_lds[HW / SP][4][WAVE];
        __shared__ float delta_lds[HW][TILE_R];
        floatx4v(&q_h)[4][WAVE] = q_lds[t.wv % (HW / SP)];
        constexpr int TS = 4 / SP;
        floatx4v xq[TS], xd[TS], xo[TS];
#pragma unroll
        for (int i = 0; i < TS; ++i) {
            const int at = t.part * TS + i;
            xq[i] = tile_load4<NARROW>(reinterpret_cast<const char *>(q) + mrow, at, g, nw);
            xd[i] = tile_load4<NARROW>(reinterpret_cast<const char *>(d_o) + mrow, at, g, nw);
            xo[i] = tile_load4<NARROW>(reinterpret_cast<const char *>(o) + mrow, at, g, nw);
        }
        lse_c = lse[(size_t)max(t.member.x, 0) * Hs + t.head];
        float part = 0.f;
#pragma unroll
        for (int i = 0; i < TS; ++i) {
            q_h[t.part * TS + i][t.lane] = xq[i];
            dob_h[t.part * TS + i][t.lane] = xd[i];
#pragma unroll
            for (int e = 0; e < 4; ++e) part = fmaf(xd[i][e], xo[i][e], part);
        }
        part = groups_sum(part);
        if (g == 0) delta_lds[t.wv][c] = part;
        __syncthreads();
        delta = 0.f;
#pragma unroll
        for (int i = 0; i < SP; ++i) delta += delta_lds[i * (HW / SP) + t.wv % (HW / SP)][c];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const floatx4v x = q_h[i][t.lane];
            qb[4 * i] = x[0]; qb[4 * i + 1] = x[1]; qb[4 * i + 2] = x[2]; qb[4 * i + 3] = x[3];
        }
    } else {
        float ob[16], dob[16];
        float4 qr[4], dr[4], orow[4];
        tile_ask_members<NARROW>(t, d_o, RB, dr);
        tile_ask_members<NARROW>(t, o, RB, orow);
        tile_ask_members<NARROW>(t, q, RB, qr);
        tile_rows_to_operand<NARROW>(kt, dr, c, g, dob, nw);
        tile_rows_to_operand<NARROW>(kt, orow, c, g, ob, nw);
        tile_rows_to_operand<NARROW>(kt, qr, c, g, qb, nw);
        float part = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) part = fmaf(dob[i], ob[i], part);
        delta = groups_sum(part);                                 // dO . O of member c, this head
        lse_c = lse[(size_t)max(t.member.x, 0) * Hs + t.head];
#pragma unroll
        for (int i = 0; i < 4; ++i) dob_h[i][t.lane] = floatx4v{dob[4 * i], dob[4 * i + 1], dob[4 * i + 2], dob[4 * i + 3]};
    }
    floatx4v acc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
    struct Blk {
        float4 kc[4], vc[4];                                      // columns 4 c .. 4 c + 3 of the K / V rows of entries 4 r + g
        int b, nv;                                                // which block of the piece; entries of it that exist
        int xe[DROP || BIAS == 1 ? 4 : 1];
        float bz[BIAS ? 4 : 1];
    };
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane, fst);
        auto issue = [&](Blk &B, int b) {
            if constexpr (DROP || BIAS == 1) tile_pair_eids(P, p0 + TILE_R * b + g, t.p_end, c, B.xe, 4);
            B.b = b;
            B.nv = min(TILE_R, cnt - TILE_R * b);
            int idxv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) idxv[r] = ent[TILE_R * b + 4 * r + g].x;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                B.kc[r] = tile_row4<NARROW>(kb + ((uint32_t)idxv[r] * RB + t.offv));
#pragma unroll
            for (int r = 0; r < 4; ++r)
                B.vc[r] = tile_row4<NARROW>(vb + ((uint32_t)idxv[r] * RB + t.offv));
            if constexpr (BIAS) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int at = TILE_R * b + 4 * r + g;
                    B.bz[r] = bias[tile_bias_at<H, BIAS>(P, t.head, B.xe[BIAS == 1 ? r : 0], BIAS == 2 ? tile_pair_number(fst[at], ent[at].y, c) : 0)];
                }
            }
        };
        auto compute = [&](const Blk &B) {
            int mask[4], number[4];                               // (read here, not kept from the block's issue on)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int at = TILE_R * B.b + 4 * r + g;
                mask[r] = ent[at].y;
                number[r] = tile_pair_number(fst[at], mask[r], c);
            }
            floatx4v st;
            {
                float kr[16];
                tile_rows_to_operand<NARROW>(kt, B.kc, c, g, kr, nw);
                st = tile_dot(kr, qb);
            }
            float va[16];
            tile_rows_to_operand<NARROW>(kt, B.vc, c, g, va, nw);
            float dob[16];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const floatx4v x = dob_h[i][t.lane];
                dob[4 * i] = x[0]; dob[4 * i + 1] = x[1]; dob[4 * i + 2] = x[2]; dob[4 * i + 3] = x[3];
            }
            const floatx4v dp = tile_dot(va, dob);
            float ds[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float pe = where_pair_or_zero(mask[r], c, __builtin_amdgcn_exp2f((BIAS ? fmaf(st[r], scale_log2e, B.bz[BIAS ? r : 0] * scale_log2e) : st[r] * scale_log2e) - lse_c));
                float mt = 1.f;                                   // dropout multiplier of this pair (as in the forward)
                if constexpr (DROP)
                    mt = dropout_keep((uint32_t)B.xe[DROP ? r : 0] * (uint32_t)Hs + (uint32_t)t.head, drop_seed, drop_thr, drop_inv);
                ds[r] = pe * (dp[r] * mt - delta) * scale;
                pe *= mt;                                         // what multiplies v (forward) and dO (dV)
                if ((mask[r] >> c) & 1) {
                    pds_h[(uint32_t)number[r]] = make_float2(pe, ds[r]);
                    if constexpr (BIAS) ds_out[tile_bias_at<H, BIAS>(P, t.head, B.xe[BIAS == 1 ? r : 0], number[r])] = ds[r];   // dL/d(score before scaling)
                }
            }
            tile_axpy_upto(ds, B.kc, acc, B.nv);
        };
        tile_walk<Blk>(nblk, issue, compute);
        wave_lds_fence();
    }
    if constexpr (SP > 1) {
        tile_park(kt, acc, t.lane);
        __syncthreads();
        tile_meet_and_store<SP, H, D, NARROW>(kt_lds[t.wv % (HW / SP)], (HW / SP) * TILE_R * TILE_KT_STRIDE, t, dq, ws_dq, nw);
    } else {
        tile_store_rows<H, D, false, NARROW>(t, acc, 1.f, dq, ws_dq, nw);
    }
}

// Backward on tiles, source side (groups of the out-CSR plan: members = source rows, entries = destinations):
// dk += ds^T q, dv += p^T dO with (p, ds) of every pair fetched from the scratch the destination side filled, at the
// destination side's pair number that this plan's grp_pairs gives for (entry, member).
//
// A lane asks for the pairs of ONE entry (destination) with four neighbouring members, not of one member with four entries:
// the destination side numbers the pairs of a tile by its entries, which are this side's members, so lanes c, the
// destinations of a block, mostly read one run of 8 bytes each per member instead of 16 places 8 bytes x (members per entry)
// apart, and the four positions are one load.  The block of (p, ds) is turned in LDS on the way into the products, which also
// frees its registers: the next block's (p, ds) are asked for behind this block's rows and the positions of the one after that,
// so neither is waited for, in 117 registers (two sets of (p, ds) in registers: 128 and 44 bytes spilled, 89 -> 100 us for the
// 32-graph batch).  The first positions leave with the entry list.  8 heads, before -> now: L = 32768, k = 4 218 -> 210 us;
// L = 4096, k = 32 54.1 -> 52.2; window 128 27.2 -> 25.6 (before: rows read a block ahead at three wavefronts per SIMD, which is
// not needed any more); 6 heads of 50 columns 68.5 -> 65.6; 32-graph batch and L = 8192, k = 4 level.
constexpr int TILE_WT_STRIDE = 18;                                // float2 per entry: 16 members + 2 (writes and reads spread over the banks)
typedef int intx4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void tile_pair_positions(const bpt_plan &P, int entry, int g, int (&pos)[4]) {
    const intx4u x = *reinterpret_cast<const intx4u *>(P.grp_pairs + (size_t)entry * TILE_R + 4 * g);
    pos[0] = x[0]; pos[1] = x[1]; pos[2] = x[2]; pos[3] = x[3];
}
template <typename T, int H, int D, int HW, bool NARROW = false, int SP = 1>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(4))) void k_attn_bwd_src_tile(
    bpt_plan P, const T *__restrict__ q, const T *__restrict__ d_o, const float2 *__restrict__ pds, T *__restrict__ dk, T *__restrict__ dv,
    float *__restrict__ ws_dk, float *__restrict__ ws_dv, Narrow nw) {
    const uint32_t RB = NARROW ? (uint32_t)(nw.heads * nw.d) * sizeof(T) : (uint32_t)(H * D * sizeof(T));
    TileCtx t;
    if (!tile_begin<T, H, D, HW, NARROW, SP>(P, t, nw)) return;
    // a wavefront's piece: its entry list and its block of (p, ds), afterwards (SP > 1) what it has summed up
    constexpr int ENT = TILE_CHUNK * 2, LIVE = ENT + TILE_R * TILE_WT_STRIDE * 2, PIECE = SP > 1 ? 2 * TILE_PART_FLOATS : LIVE;
    static_assert(PIECE >= LIVE, "the lists fit");
    __shared__ __attribute__((aligned(16))) float piece[HW][PIECE];
    int2 *ent = reinterpret_cast<int2 *>(piece[t.wv]);
    float2 *const wt = reinterpret_cast<float2 *>(piece[t.wv] + ENT);
    const int c = t.c, g = t.g;
    const char *qb = reinterpret_cast<const char *>(q), *db = reinterpret_cast<const char *>(d_o);
    const float2 *const pds_h = pds + (size_t)t.head * (size_t)P.n_edges;
    floatx4v ak[4], av[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) { ak[nb] = floatx4v{0.f, 0.f, 0.f, 0.f}; av[nb] = floatx4v{0.f, 0.f, 0.f, 0.f}; }
    // Both products contract over the block's entries, four per step; lane group g takes entries 4 r + g in step r, so that
    // the steps past the end of the group's list (half of a group's last block on average) can be left out.
    struct Blk {
        float4 qr[4], dr[4];
        int mk[4], nv;                                            // bit c of mk[r]: the pair (entry 4 r + g, member c) exists; nv: entries of the block that exist
    };
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    int pos[4];
    float2 w[4];                                                  // (p, ds) of the pairs (entry c, member 4 g + r) of the next block
    auto positions = [&](int first_entry) { tile_pair_positions(P, min(first_entry + c, t.p_end - 1), g, pos); };
    if (t.p_end > t.p_begin) positions(t.p_begin);
    issue_loads_first();
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane);
        if (p0 == t.p_begin) {
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] = pds_h[(uint32_t)pos[r]];
            positions(p0 + TILE_R);
        }
        auto put_pairs = [&]() {
            floatx4v *const wp = reinterpret_cast<floatx4v *>(wt + c * TILE_WT_STRIDE + 4 * g);
            wp[0] = floatx4v{w[0].x, w[0].y, w[1].x, w[1].y};
            wp[1] = floatx4v{w[2].x, w[2].y, w[3].x, w[3].y};
            wave_lds_fence();
        };
        auto issue_rows = [&](Blk &B, int b) {
            B.nv = min(TILE_R, cnt - TILE_R * b);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int2 en = ent[TILE_R * b + 4 * r + g];
                B.mk[r] = en.y;
                const uint32_t off = (uint32_t)en.x * RB + t.offv;
                B.qr[r] = tile_row4<NARROW>(qb + off);
                B.dr[r] = tile_row4<NARROW>(db + off);
            }
        };
        auto compute = [&](const Blk &B) {
            float pe[4], ds[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float2 w = wt[(4 * r + g) * TILE_WT_STRIDE + c];
                pe[r] = where_pair_or_zero(B.mk[r], c, w.x);      // the scratch of pairs that do not exist is not initialised
                ds[r] = where_pair_or_zero(B.mk[r], c, w.y);
            }
            wave_lds_fence();                                     // (read before the next block's are written)
            tile_axpy_upto(ds, B.qr, ak, B.nv);
            tile_axpy_upto(pe, B.dr, av, B.nv);
        };
        for (int b = 0; b < nblk; ++b) {
            Blk B;
            issue_rows(B, b);
            issue_loads_first();
            put_pairs();
            if (p0 + TILE_R * (b + 1) < t.p_end) {
#pragma unroll
                for (int r = 0; r < 4; ++r) w[r] = pds_h[(uint32_t)pos[r]];
                positions(p0 + TILE_R * (b + 2));
            }
            issue_loads_first();
            compute(B);
            issue_loads_first();
        }
        wave_lds_fence();
    }
    if constexpr (SP > 1) {
        constexpr int NEXT = (HW / SP) * PIECE;
        tile_park(piece[t.wv], ak, t.lane);
        tile_park(piece[t.wv] + TILE_PART_FLOATS, av, t.lane);
        __syncthreads();
        const float *const part0 = piece[t.wv % (HW / SP)];
        tile_meet_and_store<SP, H, D, NARROW>(part0, NEXT, t, dk, ws_dk, nw);
        tile_meet_and_store<SP, H, D, NARROW>(part0 + TILE_PART_FLOATS, NEXT, t, dv, ws_dv, nw);
    } else {
        tile_store_rows<H, D, false, NARROW>(t, ak, 1.f, dk, ws_dk, nw);
        tile_store_rows<H, D, false, NARROW>(t, av, 1.f, dv, ws_dv, nw);
    }
}

// ---- The separate operators on tiles, float32: Y[row] = sum of W[eid, head] X[idx] and y[eid, head] = <A[row, head, :], B[idx, head, :]>
// on the tile walk above, one of its products each.  Beside the rows, what these kernels move is the (n_edges, H) edge tensor, found by
// the edge ids of a block's pairs (grp_eids): a record of H floats per edge, of which a wavefront, one head, wants four bytes.  So
// the wavefronts of a workgroup share them (SHARED): each reads or writes a quarter of a block's pairs (half with two heads a
// workgroup) with all the workgroup's heads in one 16-byte access, and they meet in LDS, one barrier a block.  Every wavefront for
// itself: the texture addresser works through 64 places per instruction, four instructions a block and head.
// 8 heads, per launch without merges, row groups of 8 -> each for itself -> shared: L = 8192, k = 4 SpMM 33.9 -> 31 -> 26.6 (out-CSR) and 33 ->
// 27 -> 22.6 us (in-CSR), SDDMM 32.5 -> 27.7 -> 23.4 and 31.5 -> 28 -> 21.6; 32-graph batch SpMM 43 -> 40 -> 34, SDDMM 43 -> 41 -> 34;
// window 128 SpMM 38 -> 17 to 23 -> 12 to 19, SDDMM 29 -> 19 to 23 -> 15 to 18 (one wavefront a tile; product_parts says where).  What bounds them now: at L = 8192 the node rows read and
// written by themselves are 13 us at the rate of a large copy, the products 7; the rest is the tiles' first loads and the edge tensor's places.
template <int HW> struct HeadPack;
template <> struct HeadPack<4> { typedef floatx4v vec; };
template <> struct HeadPack<2> { typedef float vec __attribute__((ext_vector_type(2))); };

// The sums of a tile again, pair by pair.  A product over a block multiplies the weight 0 of a pair that does not exist with the row's
// columns: a row that is not finite reaches members that do not have it.  A wavefront whose sums are not all finite comes here, where
// only pairs that exist are added, so that such a row reaches its own neighbours and no others.
template <bool NARROW>
__device__ __forceinline__ void spmm_tile_by_pairs(const bpt_plan &P, const TileCtx &t, const float *Wh, uint32_t WH, const char *xb, uint32_t RB, floatx4v (&acc)[4]) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
    for (int p = t.p_begin; p < t.p_end; ++p) {
        const int4 en = reinterpret_cast<const int4 *>(P.grp_entries)[p];
        const float4 x = tile_row4<NARROW>(xb + ((uint32_t)en.x * RB + t.offv));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = 4 * t.g + r;                            // accumulators: register r of every lane belongs to member 4 g + r
            if (!((en.y >> m) & 1)) continue;
            const float w = Wh[(size_t)(uint32_t)P.grp_eids[(size_t)p * TILE_R + m] * WH];
            acc[0][r] = fmaf(w, x.x, acc[0][r]); acc[1][r] = fmaf(w, x.y, acc[1][r]); acc[2][r] = fmaf(w, x.z, acc[2][r]); acc[3][r] = fmaf(w, x.w, acc[3][r]);
        }
    }
}

template <int H, int D, int HW, bool SHARED, bool NARROW = false, int SP = 1>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(SP > 1 ? 5 : 6))) void k_spmm_tile(
    bpt_plan P, const float *__restrict__ W, const float *__restrict__ X, float *__restrict__ Y, float *__restrict__ ws, Narrow nw) {
    static_assert(SP == 1 || !SHARED, "the parts of a tile have blocks of their own: no barrier a block");
    using vec = typename HeadPack<SHARED ? HW : 2>::vec;
    constexpr int RW = SHARED ? 4 / HW : 4;                       // registers r (entries 4 r + g of a block) that a wavefront fetches weights of
    const uint32_t RB = NARROW ? (uint32_t)(nw.heads * nw.d) * 4 : (uint32_t)(H * D * 4), WH = NARROW ? (uint32_t)nw.heads : (uint32_t)H;
    TileCtx t;
    if (!tile_begin<float, H, D, HW, NARROW, SP>(P, t, nw)) return;
    constexpr int ENT = TILE_CHUNK * 2, PIECE = SP > 1 ? TILE_PART_FLOATS : ENT;
    static_assert(PIECE >= ENT, "the list fits");
    __shared__ __attribute__((aligned(16))) float piece[HW][PIECE];
    __shared__ float wt[SHARED ? 2 : 1][SHARED ? HW : 1][SHARED ? 4 * WAVE : 1];         // this block's weights and the next one's: [head][r][lane]
    int2 *ent = reinterpret_cast<int2 *>(piece[t.wv]);
    const int c = t.c, g = t.g, r0 = SHARED ? t.wv * RW : 0;
    const char *xb = reinterpret_cast<const char *>(X);
    const float *const Wh = W + t.head - (SHARED ? t.wv : 0);
    floatx4v acc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    // the edge ids of a block's pairs are asked for two blocks ahead, the weights one block ahead
    int xe[RW];
    float w[SHARED ? 1 : 4];
    vec wv[SHARED ? RW : 1];
    auto edges = [&](int first_entry) {
#pragma unroll
        for (int i = 0; i < RW; ++i) xe[i] = P.grp_eids[(size_t)min(first_entry + 4 * (r0 + i) + g, t.p_end - 1) * TILE_R + c];
    };
    auto weights = [&]() {                                        // (n_edges: the pair does not exist)
#pragma unroll
        for (int i = 0; i < RW; ++i) {
            const bool there = (uint32_t)xe[i] < (uint32_t)P.n_edges;
            const float *const at = Wh + (size_t)((uint32_t)xe[i] * WH);
            if constexpr (SHARED) {
#pragma unroll
                for (int k = 0; k < HW; ++k) wv[i][k] = 0.f;
                if (there) wv[i] = *reinterpret_cast<const vec *>(at);
            } else {
                w[i] = 0.f;
                if (there) w[i] = *at;
            }
        }
    };
    int stage = 0;
    auto put = [&]() {
        if constexpr (SHARED) {
#pragma unroll
            for (int i = 0; i < RW; ++i)
#pragma unroll
                for (int k = 0; k < HW; ++k) wt[stage][k][WAVE * (r0 + i) + t.lane] = wv[i][k];
        }
    };
    if (t.p_end > t.p_begin) edges(t.p_begin);
    issue_loads_first();
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane);
        if (p0 == t.p_begin) {
            weights();
            edges(p0 + TILE_R);
            put();
        }
        for (int b = 0; b < nblk; ++b) {
            if constexpr (SHARED) __syncthreads();                // (the other stage is read to the end too)
            const int nv = min(TILE_R, cnt - TILE_R * b);
            int mk[4];
            float4 xr[4];
            float wc[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int2 en = ent[TILE_R * b + 4 * r + g];
                mk[r] = en.y;
                xr[r] = tile_row4<NARROW>(xb + ((uint32_t)en.x * RB + t.offv));
                if constexpr (!SHARED) wc[r] = w[r];
            }
            issue_loads_first();
            const bool more = p0 + TILE_R * (b + 1) < t.p_end;
            if (more) {
                weights();
                edges(p0 + TILE_R * (b + 2));
            }
            issue_loads_first();
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (SHARED) wc[r] = wt[stage][t.wv][WAVE * r + t.lane];
                wc[r] = where_pair_or_zero(mk[r], c, wc[r]);
            }
            tile_axpy_upto(wc, xr, acc, nv);
            issue_loads_first();
            stage ^= SHARED ? 1 : 0;
            if (more) put();
        }
        wave_lds_fence();                                         // the piece is read to the end before the next one is staged
    }
    float zero = 0.f;                                             // 0 times a sum is 0 unless the sum is not finite
#pragma unroll
    for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) zero = fmaf(acc[nb][r], 0.f, zero);
    if (__builtin_amdgcn_ballot_w64(!(zero == 0.f)) != 0) spmm_tile_by_pairs<NARROW>(P, t, W + t.head, WH, xb, RB, acc);
    if constexpr (SP > 1) {
        tile_park(piece[t.wv], acc, t.lane);
        __syncthreads();
        tile_meet_and_store<SP, H, D, NARROW>(piece[t.wv % (HW / SP)], (HW / SP) * PIECE, t, Y, ws, nw);
    } else {
        tile_store_rows<H, D, false, NARROW>(t, acc, 1.f, Y, ws, nw);
    }
}

template <int H, int D, int HW, bool SHARED, bool NARROW = false, int SP = 1>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(5))) void k_sddmm_tile(
    bpt_plan P, const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ y, Narrow nw) {
    static_assert(SP == 1 || !SHARED, "the parts of a tile have blocks of their own: no barrier a block");
    using vec = typename HeadPack<SHARED ? HW : 2>::vec;
    constexpr int RW = SHARED ? 4 / HW : 4;
    const uint32_t RB = NARROW ? (uint32_t)(nw.heads * nw.d) * 4 : (uint32_t)(H * D * 4), WH = NARROW ? (uint32_t)nw.heads : (uint32_t)H;
    TileCtx t;
    if (!tile_begin<float, H, D, HW, NARROW, SP>(P, t, nw)) return;
    __shared__ int2 ent_lds[HW][TILE_CHUNK];
    __shared__ __attribute__((aligned(16))) float kt_lds[HW][TILE_R * TILE_KT_STRIDE];
    __shared__ float wt[SHARED ? 2 : 1][SHARED ? HW : 1][SHARED ? 4 * WAVE : 1];
    int2 *ent = ent_lds[t.wv];
    float *kt = kt_lds[t.wv];
    const int c = t.c, g = t.g, r0 = SHARED ? t.wv * RW : 0;
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    issue_loads_first();
    const char *bb = reinterpret_cast<const char *>(B);
    const char *const arow = reinterpret_cast<const char *>(A) + (size_t)max(t.member.x, 0) * RB + t.offa;
    float *const yh = y + t.head - (SHARED ? t.wv : 0);
    float ab[16];
    int stage = 0;
    struct Blk {
        float4 rows[4];
        int xe[RW];                                               // edge ids of the pairs that this lane stores (n_edges or more: none)
    };
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane);
        auto issue = [&](Blk &K, int b) {
#pragma unroll
            for (int i = 0; i < RW; ++i) {
                const int e = p0 + TILE_R * b + 4 * (r0 + i) + g;
                const int id = P.grp_eids[(size_t)min(e, t.p_end - 1) * TILE_R + c];
                K.xe[i] = e < t.p_end ? id : -1;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) K.rows[r] = tile_row4<NARROW>(bb + ((uint32_t)ent[TILE_R * b + 4 * r + g].x * RB + t.offv));
        };
        auto rest = [](Blk &, int) {};
        auto compute = [&](const Blk &K) {
            float kr[16];
            tile_rows_to_operand<NARROW>(kt, K.rows, c, g, kr, nw);
            const floatx4v st = tile_dot(kr, ab);
            if constexpr (SHARED) {
#pragma unroll
                for (int r = 0; r < 4; ++r) wt[stage][t.wv][WAVE * r + t.lane] = st[r];
                __syncthreads();                                  // (the stage before this one is read to the end too)
            }
#pragma unroll
            for (int i = 0; i < RW; ++i) {
                if ((uint32_t)K.xe[i] >= (uint32_t)P.n_edges) continue;
                float *const at = yh + (size_t)((uint32_t)K.xe[i] * WH);
                if constexpr (SHARED) {
                    vec x;
#pragma unroll
                    for (int k = 0; k < HW; ++k) x[k] = wt[stage][k][WAVE * (r0 + i) + t.lane];
                    *reinterpret_cast<vec *>(at) = x;
                } else {
                    *at = st[i];
                }
            }
            stage ^= SHARED ? 1 : 0;
        };
        tile_walk_first_ahead<Blk>(nblk, issue, rest, compute, [&]() { if (p0 == t.p_begin) tile_load16<NARROW>(arow, ab, g, nw); });
        wave_lds_fence();
    }
}

// ---- Dense tiles for bfloat16 rows.  Same walk and the same lane roles as the float32 tile kernels above, on
// v_mfma_f32_16x16x32_bf16 (products over the 64 columns: two instructions) and v_mfma_f32_16x16x16_bf16 (products over
// the 16 entries of a block: one instruction per four output columns), float32 accumulation:
//   lane (c, g) holds columns 16 g .. 16 g + 15 of the row of entry c (32 contiguous bytes; slot j of step t of the product
//   stands for column 16 g + 8 t + j in both operands).
// Heads of 64 columns: rows go through LDS for both kinds of product (k_attn_fwd_rows_bf16, k_attn_bwd_dst_rows_bf16,
// k_attn_bwd_src_tile_bf16_again; tile_ask_rows_bf16 says why), the next block's asked for while this one's are used.  Narrower heads, and
// the source side that reads (p, ds) back: a lane loads columns 4 c .. 4 c + 3 of the rows of entries 4 g + r (8 bytes; the B
// operand of output columns {4 c + nb} takes element nb of each of the four, packed by byte permutes), and the entries' rows
// are turned in LDS for the products over the columns (tile_rows_to_operand_bf16).
// Probabilities and ds are rounded to bfloat16 where they enter a product (the softmax denominator is summed unrounded);
// the scratch between the two backward kernels, where there is one, holds (p, ds) as two bfloat16 in 4 bytes, by head and destination-side pair number.
constexpr int TILE_BF16_WPE = 5, TILE_BF16_WPE_DST = 5, TILE_BF16_WPE_SRC = 5, TILE_BF16_WPE_AGAIN = 4;     // wavefronts per SIMD the bfloat16 tile kernels are compiled for
typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
typedef short shortx4v __attribute__((ext_vector_type(4)));
union Bf8 { bf16x8v v; uint4 q; };
union Bf4 { shortx4v v; uint32_t u[2]; };

__device__ __forceinline__ uint32_t pack_lo16(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }   // (a.lo, b.lo)
__device__ __forceinline__ uint32_t pack_hi16(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }   // (a.hi, b.hi)

// B operand of output columns {4 c + nb}: element nb of the 8-byte pieces of the rows of entries 4 g + r, r = 0 .. 3
template <int NB>
__device__ __forceinline__ Bf4 tile_cols_bf16(const uint2 (&rows)[4]) {
    Bf4 b;
    if constexpr (NB == 0) { b.u[0] = pack_lo16(rows[0].x, rows[1].x); b.u[1] = pack_lo16(rows[2].x, rows[3].x); }
    if constexpr (NB == 1) { b.u[0] = pack_hi16(rows[0].x, rows[1].x); b.u[1] = pack_hi16(rows[2].x, rows[3].x); }
    if constexpr (NB == 2) { b.u[0] = pack_lo16(rows[0].y, rows[1].y); b.u[1] = pack_lo16(rows[2].y, rows[3].y); }
    if constexpr (NB == 3) { b.u[0] = pack_hi16(rows[0].y, rows[1].y); b.u[1] = pack_hi16(rows[2].y, rows[3].y); }
    return b;
}
// acc[nb][r'] (member 4 g + r', column 4 c + nb) += sum over the block's entries of w[member c][entry 4 g + r] * row[entry][column]
__device__ __forceinline__ void tile_axpy_bf16(const Bf4 &w, const uint2 (&rows)[4], floatx4v (&acc)[4]) {
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w.v, tile_cols_bf16<0>(rows).v, acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w.v, tile_cols_bf16<1>(rows).v, acc[1], 0, 0, 0);
    acc[2] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w.v, tile_cols_bf16<2>(rows).v, acc[2], 0, 0, 0);
    acc[3] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w.v, tile_cols_bf16<3>(rows).v, acc[3], 0, 0, 0);
}
// register r of lane (c, g) = sum over the 64 columns of a[entry 4 g + r] * b[member c]
__device__ __forceinline__ floatx4v tile_dot_bf16(const Bf8 (&a)[2], const Bf8 (&b)[2]) {
    floatx4v s = floatx4v{0.f, 0.f, 0.f, 0.f};
    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0].v, b[0].v, s, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1].v, b[1].v, s, 0, 0, 0);
}
__device__ __forceinline__ void tile_load_row_bf16(const char *p, Bf8 (&out)[2], int g, const Narrow &nw) {
    uint32_t w[8];
#pragma unroll
    for (int t = 0; t < 4; ++t) {                                 // quad 4 g + t; d is even, so a quad is shifted by whole words
        const int quad = 4 * (4 * g + t), col = min(quad, nw.d - 4);
        const uintx2u x = *reinterpret_cast<const uintx2u *>(p + 2 * col);
        w[2 * t] = col >= quad ? x[0] : 0u;
        w[2 * t + 1] = col + 2 >= quad ? x[1] : 0u;
    }
    out[0].q = make_uint4(w[0], w[1], w[2], w[3]);
    out[1].q = make_uint4(w[4], w[5], w[6], w[7]);
}
template <bool NARROW> __device__ __forceinline__ uint2 tile_row4_bf16(const char *p) {
    if constexpr (NARROW) {
        const uintx2u x = *reinterpret_cast<const uintx2u *>(p);
        return make_uint2(x[0], x[1]);
    } else {
        return *reinterpret_cast<const uint2 *>(p);
    }
}
// As tile_rows_to_operand: the rows of a block's entries, loaded as columns 4 c .. 4 c + 3 of the rows of entries 4 g + r
// (the sixteen lanes of a lane group read one row's 128 contiguous bytes), turned in a wavefront-private piece of LDS
// into the operand of the products over the columns (lane (c, g): columns 16 g .. 16 g + 15 of the row of entry c).
// Rows of TILE_KT_BYTES_BF16 = 128 + 16 bytes: the sixteen rows of a read fall on different banks.
constexpr int TILE_KT_BYTES_BF16 = 144;
typedef uint32_t uintx4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void tile_rows_to_operand_bf16(char *kt, const uint2 (&rows)[4], int c, int g, Bf8 (&out)[2], const Narrow &nw) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
        *reinterpret_cast<uintx2v *>(kt + (4 * g + r) * TILE_KT_BYTES_BF16 + 8 * c) =           // (d is even: words are whole)
            uintx2v{narrow_again<true>(nw, c, 0) ? 0u : rows[r].x, narrow_again<true>(nw, c, 2) ? 0u : rows[r].y};
    wave_lds_fence();
    const char *src = kt + c * TILE_KT_BYTES_BF16 + 32 * g;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
        const uintx4v x = *reinterpret_cast<const uintx4v *>(src + 16 * h2);
        out[h2].q = make_uint4(x[0], x[1], x[2], x[3]);
    }
    wave_lds_fence();                                             // (read before the next block's rows are written)
}

constexpr int TILE_KT_FLOATS_BF16 = TILE_R * TILE_KT_BYTES_BF16 / 4;
// Rows of 64 columns, 16 bytes a lane: lane l asks for piece l % 8 of rows l / 8 and 8 + l / 8 of sixteen, puts them into LDS as
// above, and both kinds of product read them there: the products over the columns the row of entry c, the sums over the
// entries their columns, transposed (tile_axpy_rows_bf16), so that the registers are free for the next block's rows.
//
// What bounds the bfloat16 kernels is the texture addresser, which takes a vector memory instruction four lanes at a time: 16 cycles
// for one whose neighbouring lanes read on in a line, whatever a lane reads of it, 64 where each lane's line is another
// (by that count 614 k of the source side's 750 k cycles at 16 heads, L = 32768, k = 8; 250 k now).  Rows of eight bytes a lane took twice the instructions, members' rows
// read row by lane four times the cycles, (lse, delta) of a block's entries read by all 64 lanes as many as its rows.  So: rows, members'
// rows and results in 16 bytes a lane, along the rows; single words of a row by one lane group.  Nothing else helped the source side there:
// its rows a block ahead through LDS but 8 bytes a lane 333 -> 343 us; 16 bytes a lane 315; the members and (lse, delta) too 303;
// free of bank conflicts in LDS 281 to 290.  Kernels before -> after, forward / destination / source side: 16 heads at L = 32768, k = 8 184 / 240 / 333
// -> 162 / 208 / 285 us, 8 heads at L = 8192, k = 4 17.1 / 24.6 / 26.5 -> 16.4 / 22.8 / 23.6.  Training passes: window of 64 at L = 16384,
// 16 heads 163.5 -> 139.8, 32-graph batch 152 -> 139.8, L = 16384, k = 8 180 -> 158, with dropout at L = 32768, k = 8 818 -> 760.
__device__ __forceinline__ void tile_ask_rows_bf16(const char *base, const uint32_t (&off)[2], uintx4v (&rows)[2]) {
#pragma unroll
    for (int r = 0; r < 2; ++r) rows[r] = *reinterpret_cast<const uintx4v *>(base + off[r]);
}
// In LDS such rows lie 128 bytes apart, piece j of row e at place j ^ piece_turn(e): two rows of a write, the sixteen rows of an operand's
// read and the eight rows of a transposed read (32 lanes of 8 bytes, two pieces a row) fall on different banks.
constexpr int TILE_ROWS_FLOATS_BF16 = TILE_R * 32;
__device__ __forceinline__ int piece_turn(int e) { return (e & 6) | (e >> 3); }
__device__ __forceinline__ void tile_put_rows_bf16(char *kt, const uintx4v (&rows)[2], int lane) {
    const int at = (lane >> 3) * 128 + 16 * ((lane & 7) ^ piece_turn(lane >> 3));
    *reinterpret_cast<uintx4v *>(kt + at) = rows[0];
    *reinterpret_cast<uintx4v *>(kt + (at ^ 16) + 1024) = rows[1];
}
__device__ __forceinline__ void tile_operand_bf16(const char *kt, int c, int g, Bf8 (&out)[2]) {
    const int at = c * 128 + 16 * ((2 * g) ^ piece_turn(c));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uintx4v x = *reinterpret_cast<const uintx4v *>(kt + (at ^ (16 * i)));
        out[i].q = make_uint4(x[0], x[1], x[2], x[3]);
    }
}
// byte offsets of this lane's pieces of the members' rows / of the rows of the sixteen entries at `ent`
__device__ __forceinline__ uint32_t tile_piece_at(const TileCtx &t) { return (uint32_t)(t.head * 128 + 16 * (t.lane & 7)); }
template <uint32_t RB> __device__ __forceinline__ void tile_member_offsets(const TileCtx &t, uint32_t (&off)[2]) {
    const int row = max(t.member.x, 0);
#pragma unroll
    for (int r = 0; r < 2; ++r) off[r] = (uint32_t)lane_bcast(row, 8 * r + (t.lane >> 3)) * RB + tile_piece_at(t);
}
template <uint32_t RB> __device__ __forceinline__ void tile_entry_offsets(const TileCtx &t, const int2 *ent, uint32_t (&off)[2]) {
#pragma unroll
    for (int r = 0; r < 2; ++r) off[r] = (uint32_t)ent[8 * r + (t.lane >> 3)].x * RB + tile_piece_at(t);
}
// masks of entries 4 g .. 4 g + 3
__device__ __forceinline__ void tile_masks(const int2 *ent, int g, int (&mk)[4]) {
    const int4 e01 = *reinterpret_cast<const int4 *>(&ent[4 * g]), e23 = *reinterpret_cast<const int4 *>(&ent[4 * g + 2]);
    mk[0] = e01.y; mk[1] = e01.w; mk[2] = e23.y; mk[3] = e23.w;
}
// acc += w^T rows, by column: lane (c, g), register r of acc[nb] = column 16 nb + 4 g + r of member c
__device__ __forceinline__ void tile_axpy_rows_bf16(const Bf4 &w, const char *kt, int c, int g, floatx4v (&acc)[4]) {
    // sixteen lanes read four rows of sixteen columns and are given one column of the four each
    const int e = 4 * g + (c >> 2), at = e * 128 + 16 * (((c >> 1) & 1) ^ piece_turn(e)) + 8 * (c & 1);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
        const shortx4v cols = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) shortx4v *)(kt + (at ^ (32 * nb))));
        acc[nb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(cols, w.v, acc[nb], 0, 0, 0);
    }
}
// Such sums through LDS (TILE_R * TILE_TURN_STRIDE floats): into the tile kernels' other order (lane (c, g), register r: columns 4 c .. 4 c + 3
// of member 4 g + r), or to where the members' rows go.
constexpr int TILE_TURN_STRIDE = 68;
__device__ __forceinline__ void tile_put_sums(float *sh, const floatx4v (&acc)[4], int c, int g) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) *reinterpret_cast<floatx4v *>(sh + c * TILE_TURN_STRIDE + 16 * nb + 4 * g) = acc[nb];
    wave_lds_fence();
}
__device__ __forceinline__ void tile_sums_by_row(float *sh, floatx4v (&acc)[4], int c, int g) {
    tile_put_sums(sh, acc, c, g);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const floatx4v x = *reinterpret_cast<const floatx4v *>(sh + (4 * g + r) * TILE_TURN_STRIDE + 4 * c);
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[nb][r] = x[nb];
    }
    wave_lds_fence();
}
template <int H, int D>
__device__ __forceinline__ void tile_store_sums(const TileCtx &t, float *sh, const floatx4v (&acc)[4], bf16_t *__restrict__ out, float *__restrict__ ws) {
    tile_put_sums(sh, acc, t.c, t.g);
    const int where = tile_where(t.member);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int m = 8 * r + (t.lane >> 3), at = lane_bcast(where, m);
        const floatx4v *const from = reinterpret_cast<const floatx4v *>(sh + m * TILE_TURN_STRIDE + 8 * (t.lane & 7));
        const floatx4v x = from[0], y = from[1];
        if (at >= 0) {                                            // (node tensors end before 4 GiB)
            char *const to = reinterpret_cast<char *>(out) + ((uint32_t)at * (uint32_t)(H * D * 2) + tile_piece_at(t));
            __builtin_nontemporal_store(uintx4v{pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]), pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3])},
                                        reinterpret_cast<uintx4v *>(to));
        } else if (at < -1) {
            floatx4v *const to = reinterpret_cast<floatx4v *>(ws + (size_t)(-2 - at) * (H * D) + t.head * D + 8 * (t.lane & 7));
            to[0] = x;
            to[1] = y;
        }
    }
    wave_lds_fence();
}

template <int H, int D, int HW, int WPE, bool DROP, int BIAS, int SP>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(DROP || BIAS ? WPE - 1 : WPE))) void k_attn_fwd_rows_bf16(
    bpt_plan P, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v, bf16_t *__restrict__ o,
    float *__restrict__ lse, float *__restrict__ ws_acc, float *__restrict__ ws_ml, float scale_log2e, uint32_t drop_thr,
    uint32_t drop_seed, float drop_inv, const float *__restrict__ bias) {
    constexpr uint32_t RB = H * D * 2;
    const Narrow nw{};
    TileCtx t;
    if (!tile_begin<bf16_t, H, D, HW, false, SP>(P, t, nw)) return;
    __shared__ int2 ent_lds[HW][TILE_CHUNK];
    __shared__ int fst_lds[HW][BIAS == 2 ? TILE_CHUNK : 1];      // the entries' first pair numbers: where a term in pair order sits
    int2 *ent = ent_lds[t.wv];
    int *fst = BIAS == 2 ? fst_lds[t.wv] : nullptr;
    constexpr int PIECE = 2 * TILE_ROWS_FLOATS_BF16 + 4 * TILE_R;      // (the turned sums' rows are longer)
    static_assert(PIECE >= TILE_PART_FWD_FLOATS && PIECE >= TILE_R * TILE_TURN_STRIDE, "parts and turned sums fit the rows' piece");
    __shared__ __attribute__((aligned(16))) float piece[HW][PIECE];
    char *const k_lds = reinterpret_cast<char *>(piece[t.wv]), *const v_lds = k_lds + 4 * TILE_ROWS_FLOATS_BF16;
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    issue_loads_first();
    const int c = t.c, g = t.g;
    const char *kb = reinterpret_cast<const char *>(k), *vb = reinterpret_cast<const char *>(v);
    uintx4v qr[2];
    {
        uint32_t off[2];
        tile_member_offsets<RB>(t, off);
        tile_ask_rows_bf16(reinterpret_cast<const char *>(q), off, qr);
    }
    issue_loads_first();
    Bf8 qb[2];
    floatx4v acc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
    float mref = M_INIT_LOG2, lrun = 0.f;
    bool fresh = true;                                            // nothing has been summed up yet
    struct Blk {
        uintx4v kr[2], vr[2];
        int xe[DROP || BIAS == 1 ? 4 : 1];
        float bz[BIAS ? 4 : 1];
    };
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane, fst);
        auto issue = [&](Blk &B, int b) {
            if constexpr (DROP || BIAS == 1) tile_pair_eids(P, p0 + TILE_R * b + 4 * g, t.p_end, c, B.xe);
            uint32_t off[2];
            tile_entry_offsets<RB>(t, ent + TILE_R * b, off);
            tile_ask_rows_bf16(kb, off, B.kr);
            tile_ask_rows_bf16(vb, off, B.vr);
            if constexpr (BIAS == 1) {
#pragma unroll
                for (int r = 0; r < 4; ++r) B.bz[r] = bias[tile_bias_at<H, 1>(P, t.head, B.xe[BIAS == 1 ? r : 0], 0)];
            }
            if constexpr (BIAS == 2) {
                int mk[4];
                tile_masks(ent + TILE_R * b, g, mk);
#pragma unroll
                for (int r = 0; r < 4; ++r) B.bz[r] = bias[tile_bias_at<H, 2>(P, t.head, 0, tile_pair_number(fst[TILE_R * b + 4 * g + r], mk[r], c))];
            }
        };
        Blk B;
        issue(B, 0);
        issue_loads_first();
        if (p0 == t.p_begin) {
            tile_put_rows_bf16(k_lds, qr, t.lane);
            wave_lds_fence();
            tile_operand_bf16(k_lds, c, g, qb);
            wave_lds_fence();
        }
        for (int b = 0; b < nblk; ++b) {
            int mk[4], xe[DROP ? 4 : 1];
            float bz[BIAS ? 4 : 1];
            tile_masks(ent + TILE_R * b, g, mk);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (DROP) xe[DROP ? r : 0] = B.xe[DROP ? r : 0];
                if constexpr (BIAS) bz[BIAS ? r : 0] = B.bz[BIAS ? r : 0];
            }
            tile_put_rows_bf16(k_lds, B.kr, t.lane);
            tile_put_rows_bf16(v_lds, B.vr, t.lane);
            wave_lds_fence();
            if (b + 1 < nblk) issue(B, b + 1);
            issue_loads_first();
            Bf8 kr[2];
            tile_operand_bf16(k_lds, c, g, kr);
            const floatx4v st = tile_dot_bf16(kr, qb);
            float sc[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[r] = where_pair(mk[r], c, (BIAS ? st[r] + bz[BIAS ? r : 0] : st[r]) * scale_log2e);
            const float mb = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
            if (__builtin_amdgcn_ballot_w64(mb > mref + MFMA_TAU) != 0) {
                const float mn = fmaxf(mref, groups_max(mb));    // over the four lanes of member c
                const float al = __builtin_amdgcn_exp2f(mref - mn);
                mref = mn;
                if (!fresh) {
                    lrun *= al;
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb) acc[nb] *= al;
                }
            }
            fresh = false;
            float pr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pr[r] = __builtin_amdgcn_exp2f(sc[r] - mref);
                lrun += pr[r];                                   // the softmax denominator ignores dropout
                if constexpr (DROP)
                    pr[r] *= dropout_keep((uint32_t)xe[DROP ? r : 0] * (uint32_t)H + (uint32_t)t.head, drop_seed, drop_thr, drop_inv);
            }
            Bf4 pa;
            pa.u[0] = pack_bf16(pr[0], pr[1]);
            pa.u[1] = pack_bf16(pr[2], pr[3]);
            tile_axpy_rows_bf16(pa, v_lds, c, g, acc);
            wave_lds_fence();                                     // (read before the next block's are written)
            issue_loads_first();
        }
    }
    float lt = groups_sum(lrun);
    if constexpr (SP > 1) {
        tile_sums_by_row(piece[t.wv], acc, c, g);
        tile_meet_forward<SP, H, D, false>(piece[t.wv], piece[t.wv % (HW / SP)], (HW / SP) * PIECE, t, acc, mref, lt, o, ws_acc, nw, static_cast<bf16_t *>(nullptr));
        if (t.part != 0) return;
    } else {
        if (t.member.y < 0) {                                     // (segments of a split row are stored as summed up)
            const float inv = lt > 0.f ? 1.f / lt : 0.f;
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) acc[nb] *= inv;
        }
        tile_store_sums<H, D>(t, piece[t.wv], acc, o, ws_acc);
    }
    if (g == 0 && t.member.x >= 0) {
        if (t.member.y < 0) {
            lse[(size_t)t.member.x * H + t.head] = lt > 0.f ? mref + log2f(lt) : 0.f;
        } else {
            ws_ml[((size_t)t.member.y * H + t.head) * 2] = mref;
            ws_ml[((size_t)t.member.y * H + t.head) * 2 + 1] = lt;
        }
    }
}

// Destination side.  PDS: (p, ds) of the pairs go to the scratch for the source side that reads them back; otherwise that side
// forms them again (k_attn_bwd_src_tile_bf16_again) and all it is handed is (lse, delta) of the rows, `stat` (n, H): the
// segments of a split row write the same values.
template <int H, int D, int HW, int WPE, bool DROP, int BIAS, bool PDS, int SP>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(DROP || BIAS ? WPE - 1 : WPE))) void k_attn_bwd_dst_rows_bf16(
    bpt_plan P, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v, const bf16_t *__restrict__ o,
    const bf16_t *__restrict__ d_o, const float *__restrict__ lse, bf16_t *__restrict__ dq, uint32_t *__restrict__ pds,
    float2 *__restrict__ stat, float *__restrict__ ws_dq, float scale, float scale_log2e, uint32_t drop_thr, uint32_t drop_seed, float drop_inv,
    const float *__restrict__ bias, float *__restrict__ ds_out) {
    static_assert(PDS || BIAS == 0, "the score term's gradient is stored by the pair's position");
    constexpr uint32_t RB = H * D * 2;
    const Narrow nw{};
    TileCtx t;
    if (!tile_begin<bf16_t, H, D, HW, false, SP>(P, t, nw)) return;
    __shared__ int2 ent_lds[HW][TILE_CHUNK];
    __shared__ int fst_lds[HW][PDS ? TILE_CHUNK : 1];
    int2 *ent = ent_lds[t.wv];
    int *fst = PDS ? fst_lds[t.wv] : nullptr;
    constexpr int PIECE = 2 * TILE_ROWS_FLOATS_BF16 + 4 * TILE_R;      // (the turned sums' rows are longer)
    static_assert(PIECE >= TILE_PART_FLOATS && PIECE >= TILE_R * TILE_TURN_STRIDE, "parts and turned sums fit the rows' piece");
    __shared__ __attribute__((aligned(16))) float piece[HW][PIECE];
    char *const k_lds = reinterpret_cast<char *>(piece[t.wv]), *const v_lds = k_lds + 4 * TILE_ROWS_FLOATS_BF16;
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    issue_loads_first();
    const int c = t.c, g = t.g;
    const char *kb = reinterpret_cast<const char *>(k), *vb = reinterpret_cast<const char *>(v);
    uint32_t *const pds_h = pds + (size_t)t.head * (size_t)P.n_edges;     // this head's part of the scratch
    Bf8 qb[2], dob[2];
    float delta, lse_c;
    {
        uint32_t off[2];
        tile_member_offsets<RB>(t, off);
        uintx4v qr[2], dr[2], orow[2];
        tile_ask_rows_bf16(reinterpret_cast<const char *>(d_o), off, dr);
        tile_ask_rows_bf16(reinterpret_cast<const char *>(o), off, orow);
        tile_ask_rows_bf16(reinterpret_cast<const char *>(q), off, qr);
        const size_t at = (size_t)max(t.member.x, 0) * H + t.head;
        lse_c = g == 0 ? lse[at] : 0.f;
        float part[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            part[r] = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                part[r] = fmaf(__uint_as_float(dr[r][i] << 16), __uint_as_float(orow[r][i] << 16), part[r]);
                part[r] = fmaf(__uint_as_float(dr[r][i] & 0xffff0000u), __uint_as_float(orow[r][i] & 0xffff0000u), part[r]);
            }
            part[r] = head_sum<8>(part[r]);                       // dO . O of member 8 r + l / 8, this head
        }
        tile_put_rows_bf16(k_lds, qr, t.lane);
        tile_put_rows_bf16(v_lds, dr, t.lane);
        wave_lds_fence();
        tile_operand_bf16(k_lds, c, g, qb);
        tile_operand_bf16(v_lds, c, g, dob);
        wave_lds_fence();
        const float d0 = lane_bcast(part[0], 8 * (c & 7)), d1 = lane_bcast(part[1], 8 * (c & 7));
        delta = c < 8 ? d0 : d1;
        if constexpr (!PDS) {
            if (g == 0 && t.part == 0 && t.member.x >= 0) stat[at] = make_float2(lse_c, delta);
        }
        lse_c = lane_bcast(lse_c, c);
    }
    floatx4v acc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
    struct Blk {
        uintx4v kr[2], vr[2];
        int xe[DROP || BIAS == 1 ? 4 : 1];
        float bz[BIAS ? 4 : 1];
    };
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane, fst);
        auto numbers = [&](int b, const int (&mk)[4], uint32_t (&pos)[4]) {
            const int4 f4 = *reinterpret_cast<const int4 *>(&fst[TILE_R * b + 4 * g]);
            pos[0] = tile_pair_number(f4.x, mk[0], c); pos[1] = tile_pair_number(f4.y, mk[1], c);
            pos[2] = tile_pair_number(f4.z, mk[2], c); pos[3] = tile_pair_number(f4.w, mk[3], c);
        };
        auto issue = [&](Blk &B, int b) {
            if constexpr (DROP || BIAS == 1) tile_pair_eids(P, p0 + TILE_R * b + 4 * g, t.p_end, c, B.xe);
            uint32_t off[2];
            tile_entry_offsets<RB>(t, ent + TILE_R * b, off);
            tile_ask_rows_bf16(kb, off, B.kr);
            tile_ask_rows_bf16(vb, off, B.vr);
            if constexpr (BIAS) {
                int mk[4];
                uint32_t pos[4];
                tile_masks(ent + TILE_R * b, g, mk);
                numbers(b, mk, pos);
#pragma unroll
                for (int r = 0; r < 4; ++r) B.bz[r] = bias[tile_bias_at<H, BIAS>(P, t.head, B.xe[BIAS == 1 ? r : 0], pos[r])];
            }
        };
        Blk B;
        issue(B, 0);
        for (int b = 0; b < nblk; ++b) {
            int mk[4], xe[DROP || BIAS == 1 ? 4 : 1];
            float bz[BIAS ? 4 : 1];
            uint32_t pos[4];
            tile_masks(ent + TILE_R * b, g, mk);
            if constexpr (PDS) numbers(b, mk, pos);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (DROP || BIAS == 1) xe[DROP || BIAS == 1 ? r : 0] = B.xe[DROP || BIAS == 1 ? r : 0];
                if constexpr (BIAS) bz[BIAS ? r : 0] = B.bz[BIAS ? r : 0];
            }
            tile_put_rows_bf16(k_lds, B.kr, t.lane);
            tile_put_rows_bf16(v_lds, B.vr, t.lane);
            wave_lds_fence();
            if (b + 1 < nblk) issue(B, b + 1);
            issue_loads_first();
            Bf8 row[2];
            tile_operand_bf16(k_lds, c, g, row);
            const floatx4v st = tile_dot_bf16(row, qb);
            tile_operand_bf16(v_lds, c, g, row);
            const floatx4v dp = tile_dot_bf16(row, dob);
            float ds[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float pe = where_pair_or_zero(mk[r], c, __builtin_amdgcn_exp2f((BIAS ? st[r] + bz[BIAS ? r : 0] : st[r]) * scale_log2e - lse_c));
                float mt = 1.f;                                   // dropout multiplier of this pair (as in the forward)
                if constexpr (DROP)
                    mt = dropout_keep((uint32_t)xe[DROP ? r : 0] * (uint32_t)H + (uint32_t)t.head, drop_seed, drop_thr, drop_inv);
                ds[r] = pe * (dp[r] * mt - delta) * scale;
                pe *= mt;                                         // what multiplies v (forward) and dO (dV)
                if (PDS && ((mk[r] >> c) & 1)) {
                    pds_h[pos[r]] = pack_bf16(pe, ds[r]);
                    if constexpr (BIAS) ds_out[tile_bias_at<H, BIAS>(P, t.head, xe[BIAS == 1 ? r : 0], pos[r])] = ds[r];   // dL/d(score before scaling)
                }
            }
            Bf4 da;
            da.u[0] = pack_bf16(ds[0], ds[1]);
            da.u[1] = pack_bf16(ds[2], ds[3]);
            tile_axpy_rows_bf16(da, k_lds, c, g, acc);
            wave_lds_fence();                                     // (read before the next block's are written)
            issue_loads_first();
        }
    }
    if constexpr (SP > 1) {
        tile_sums_by_row(piece[t.wv], acc, c, g);
        tile_park(piece[t.wv], acc, t.lane);
        __syncthreads();
        tile_meet_and_store<SP, H, D, false>(piece[t.wv % (HW / SP)], (HW / SP) * PIECE, t, dq, ws_dq, nw);
    } else {
        tile_store_sums<H, D>(t, piece[t.wv], acc, dq, ws_dq);
    }
}

// Heads of fewer than 64 columns (their rows on 4 bytes): rows of 8 bytes a lane, kept in registers.
template <int H, int D, int HW, int WPE, bool DROP, int SP>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(WPE))) void k_attn_fwd_tile_bf16(
    bpt_plan P, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v, bf16_t *__restrict__ o,
    float *__restrict__ lse, float *__restrict__ ws_acc, float *__restrict__ ws_ml, float scale_log2e, uint32_t drop_thr,
    uint32_t drop_seed, float drop_inv, Narrow nw, Keep keep) {
    const int Hs = nw.h;                                          // heads as lse, workspace and dropout keys count them
    const uint32_t RB = (uint32_t)(nw.heads * nw.d) * 2;          // bytes of a node row
    const int block = keep_or_tile<HW * WAVE>(keep);
    if (block < 0) return;
    bf16_t *const o_keep = reinterpret_cast<bf16_t *>(keep.o);
    TileCtx t;
    if (!tile_begin<bf16_t, H, D, HW, true, SP>(P, t, nw, (unsigned)block)) return;
    __shared__ int2 ent_lds[HW][TILE_CHUNK];
    int2 *ent = ent_lds[t.wv];
    constexpr int PIECE = SP > 1 ? TILE_PART_FWD_FLOATS : TILE_KT_FLOATS_BF16;
    static_assert(PIECE >= TILE_KT_FLOATS_BF16, "the rows fit");
    __shared__ __attribute__((aligned(16))) float piece[HW][PIECE];
    char *kt = reinterpret_cast<char *>(piece[t.wv]);
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    issue_loads_first();
    const int c = t.c, g = t.g;
    const uint32_t offr = t.offa, offc = t.offv;
    const char *kb = reinterpret_cast<const char *>(k), *vb = reinterpret_cast<const char *>(v);
    Bf8 qb[2];
    tile_load_row_bf16(reinterpret_cast<const char *>(q) + (size_t)max(t.member.x, 0) * RB + offr, qb, g, nw);
    floatx4v acc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
    float mref = M_INIT_LOG2, lrun = 0.f;
    bool fresh = true;                                            // nothing has been summed up yet
    struct Blk {
        uint2 kq[4];                                              // columns 4 c .. 4 c + 3 of the K rows of entries 4 g + r
        uint2 vr[4];
        int mk[4];                                                // bit c of mk[r]: the pair (entry 4 g + r, member c) exists
        int xe[DROP ? 4 : 1];
    };
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane);
        auto issue_k = [&](Blk &B, int b) {
            const int4 e01 = *reinterpret_cast<const int4 *>(&ent[TILE_R * b + 4 * g]);
            const int4 e23 = *reinterpret_cast<const int4 *>(&ent[TILE_R * b + 4 * g + 2]);
            const int idxv[4] = {e01.x, e01.z, e23.x, e23.z};
#pragma unroll
            for (int r = 0; r < 4; ++r) B.kq[r] = tile_row4_bf16<true>(kb + ((uint32_t)idxv[r] * RB + offc));
        };
        auto issue_rest = [&](Blk &B, int b) {
            if constexpr (DROP) tile_pair_eids(P, p0 + TILE_R * b + 4 * g, t.p_end, c, B.xe);
            const int4 e01 = *reinterpret_cast<const int4 *>(&ent[TILE_R * b + 4 * g]);
            const int4 e23 = *reinterpret_cast<const int4 *>(&ent[TILE_R * b + 4 * g + 2]);
            const int idxv[4] = {e01.x, e01.z, e23.x, e23.z};
            B.mk[0] = e01.y; B.mk[1] = e01.w; B.mk[2] = e23.y; B.mk[3] = e23.w;
#pragma unroll
            for (int r = 0; r < 4; ++r) B.vr[r] = tile_row4_bf16<true>(vb + ((uint32_t)idxv[r] * RB + offc));
        };
        auto compute = [&](const Blk &B) {
            Bf8 kr[2];
            tile_rows_to_operand_bf16(kt, B.kq, c, g, kr, nw);
            const floatx4v st = tile_dot_bf16(kr, qb);
            float sc[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[r] = where_pair(B.mk[r], c, st[r] * scale_log2e);
            const float mb = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
            if (__builtin_amdgcn_ballot_w64(mb > mref + MFMA_TAU) != 0) {
                const float mn = fmaxf(mref, groups_max(mb));    // over the four lanes of member c
                const float al = __builtin_amdgcn_exp2f(mref - mn);
                mref = mn;
                if (!fresh) {
                    lrun *= al;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float a = lane_bcast(al, 4 * g + r);
#pragma unroll
                        for (int nb = 0; nb < 4; ++nb) acc[nb][r] *= a;
                    }
                }
            }
            fresh = false;
            float pr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pr[r] = __builtin_amdgcn_exp2f(sc[r] - mref);
                lrun += pr[r];                                   // the softmax denominator ignores dropout
                if constexpr (DROP)
                    pr[r] *= dropout_keep((uint32_t)B.xe[DROP ? r : 0] * (uint32_t)Hs + (uint32_t)t.head, drop_seed, drop_thr, drop_inv);
            }
            Bf4 pa;
            pa.u[0] = pack_bf16(pr[0], pr[1]);
            pa.u[1] = pack_bf16(pr[2], pr[3]);
            tile_axpy_bf16(pa, B.vr, acc);
        };
        auto issue = [&](Blk &B, int b) { issue_k(B, b); issue_rest(B, b); };
        if constexpr (DROP) tile_walk<Blk>(nblk, issue, compute);      // (the K rows ahead: eight registers more)
        else tile_walk_first_ahead<Blk>(nblk, issue_k, issue_rest, compute, []() {});
        wave_lds_fence();
    }
    float lt = groups_sum(lrun);
    if constexpr (SP > 1) {
        tile_meet_forward<SP, H, D, true>(piece[t.wv], piece[t.wv % (HW / SP)], (HW / SP) * PIECE, t, acc, mref, lt, o, ws_acc, nw, o_keep);
        if (t.part != 0) return;
    } else {
        tile_store_rows<H, D, true, true>(t, acc, lt > 0.f ? 1.f / lt : 0.f, o, ws_acc, nw, o_keep);
    }
    if (g == 0 && t.member.x >= 0) {
        if (t.member.y < 0) {
            lse[(size_t)t.member.x * Hs + t.head] = lt > 0.f ? mref + log2f(lt) : 0.f;
        } else {
            ws_ml[((size_t)t.member.y * Hs + t.head) * 2] = mref;
            ws_ml[((size_t)t.member.y * Hs + t.head) * 2 + 1] = lt;
        }
    }
}

// Destination side of such heads: (p, ds) of the pairs go to the scratch.
template <int H, int D, int HW, int WPE, bool DROP, int SP>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(DROP ? WPE - 1 : WPE))) void k_attn_bwd_dst_tile_bf16(
    bpt_plan P, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v, const bf16_t *__restrict__ o,
    const bf16_t *__restrict__ d_o, const float *__restrict__ lse, bf16_t *__restrict__ dq, uint32_t *__restrict__ pds,
    float *__restrict__ ws_dq, float scale, float scale_log2e, uint32_t drop_thr, uint32_t drop_seed, float drop_inv, Narrow nw) {
    const int Hs = nw.h;
    const uint32_t RB = (uint32_t)(nw.heads * nw.d) * 2;
    TileCtx t;
    if (!tile_begin<bf16_t, H, D, HW, true, SP>(P, t, nw)) return;
    __shared__ int2 ent_lds[HW][TILE_CHUNK];
    __shared__ int fst_lds[HW][TILE_CHUNK];
    int2 *ent = ent_lds[t.wv];
    int *fst = fst_lds[t.wv];
    constexpr int PIECE = SP > 1 ? TILE_PART_FLOATS : TILE_KT_FLOATS_BF16;
    static_assert(PIECE >= TILE_KT_FLOATS_BF16, "the rows fit");
    __shared__ __attribute__((aligned(16))) float piece[HW][PIECE];
    char *kt = reinterpret_cast<char *>(piece[t.wv]);
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    issue_loads_first();
    const int c = t.c, g = t.g;
    const uint32_t offr = t.offa, offc = t.offv;
    const char *kb = reinterpret_cast<const char *>(k), *vb = reinterpret_cast<const char *>(v);
    const size_t mrow = (size_t)max(t.member.x, 0) * RB + offr;
    uint32_t *const pds_h = pds + (size_t)t.head * (size_t)P.n_edges;     // this head's part of the scratch
    Bf8 qb[2], dob[2];
    float delta, lse_c;
    {
        Bf8 ob[2];
        tile_load_row_bf16(reinterpret_cast<const char *>(q) + mrow, qb, g, nw);
        tile_load_row_bf16(reinterpret_cast<const char *>(d_o) + mrow, dob, g, nw);
        tile_load_row_bf16(reinterpret_cast<const char *>(o) + mrow, ob, g, nw);
        float part = 0.f;
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2) {
            const uint32_t a[4] = {dob[h2].q.x, dob[h2].q.y, dob[h2].q.z, dob[h2].q.w}, b[4] = {ob[h2].q.x, ob[h2].q.y, ob[h2].q.z, ob[h2].q.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                part = fmaf(__uint_as_float(a[i] << 16), __uint_as_float(b[i] << 16), part);
                part = fmaf(__uint_as_float(a[i] & 0xffff0000u), __uint_as_float(b[i] & 0xffff0000u), part);
            }
        }
        delta = groups_sum(part);                                 // dO . O of member c, this head
        lse_c = lse[(size_t)max(t.member.x, 0) * Hs + t.head];
    }
    floatx4v acc[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) acc[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
    struct Blk {
        uint2 kc[4], vc[4];                                       // columns 4 c .. 4 c + 3 of the K / V rows of entries 4 g + r
        int mk[4];                                                // bit c of mk[r]: the pair (entry 4 g + r, member c) exists
        uint32_t pos[4];
        int xe[DROP ? 4 : 1];
    };
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane, fst);
        auto issue = [&](Blk &B, int b) {
            if constexpr (DROP) tile_pair_eids(P, p0 + TILE_R * b + 4 * g, t.p_end, c, B.xe);
            const int4 e01 = *reinterpret_cast<const int4 *>(&ent[TILE_R * b + 4 * g]);
            const int4 e23 = *reinterpret_cast<const int4 *>(&ent[TILE_R * b + 4 * g + 2]);
            const int idxv[4] = {e01.x, e01.z, e23.x, e23.z};
            B.mk[0] = e01.y; B.mk[1] = e01.w; B.mk[2] = e23.y; B.mk[3] = e23.w;
            const int4 f4 = *reinterpret_cast<const int4 *>(&fst[TILE_R * b + 4 * g]);
            B.pos[0] = tile_pair_number(f4.x, e01.y, c); B.pos[1] = tile_pair_number(f4.y, e01.w, c);
            B.pos[2] = tile_pair_number(f4.z, e23.y, c); B.pos[3] = tile_pair_number(f4.w, e23.w, c);
#pragma unroll
            for (int r = 0; r < 4; ++r) B.kc[r] = tile_row4_bf16<true>(kb + ((uint32_t)idxv[r] * RB + offc));
#pragma unroll
            for (int r = 0; r < 4; ++r) B.vc[r] = tile_row4_bf16<true>(vb + ((uint32_t)idxv[r] * RB + offc));
        };
        auto compute = [&](const Blk &B) {
            Bf8 kr[2];
            tile_rows_to_operand_bf16(kt, B.kc, c, g, kr, nw);
            const floatx4v st = tile_dot_bf16(kr, qb);
            tile_rows_to_operand_bf16(kt, B.vc, c, g, kr, nw);
            const floatx4v dp = tile_dot_bf16(kr, dob);
            float ds[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float pe = where_pair_or_zero(B.mk[r], c, __builtin_amdgcn_exp2f(st[r] * scale_log2e - lse_c));
                float mt = 1.f;                                   // dropout multiplier of this pair (as in the forward)
                if constexpr (DROP)
                    mt = dropout_keep((uint32_t)B.xe[DROP ? r : 0] * (uint32_t)Hs + (uint32_t)t.head, drop_seed, drop_thr, drop_inv);
                ds[r] = pe * (dp[r] * mt - delta) * scale;
                pe *= mt;                                         // what multiplies v (forward) and dO (dV)
                if ((B.mk[r] >> c) & 1) pds_h[B.pos[r]] = pack_bf16(pe, ds[r]);
            }
            Bf4 da;
            da.u[0] = pack_bf16(ds[0], ds[1]);
            da.u[1] = pack_bf16(ds[2], ds[3]);
            tile_axpy_bf16(da, B.kc, acc);
        };
        tile_walk<Blk>(nblk, issue, compute);
        wave_lds_fence();
    }
    if constexpr (SP > 1) {
        tile_park(piece[t.wv], acc, t.lane);
        __syncthreads();
        tile_meet_and_store<SP, H, D, true>(piece[t.wv % (HW / SP)], (HW / SP) * PIECE, t, dq, ws_dq, nw);
    } else {
        tile_store_rows<H, D, false, true>(t, acc, 1.f, dq, ws_dq, nw);
    }
}

constexpr int TILE_WT_STRIDE_BF16 = 20;
template <int H, int D, int HW, int WPE, bool NARROW = false, int SP = 1>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(WPE))) void k_attn_bwd_src_tile_bf16(
    bpt_plan P, const bf16_t *__restrict__ q, const bf16_t *__restrict__ d_o, const uint32_t *__restrict__ pds, bf16_t *__restrict__ dk,
    bf16_t *__restrict__ dv, float *__restrict__ ws_dk, float *__restrict__ ws_dv, Narrow nw) {
    const uint32_t RB = NARROW ? (uint32_t)(nw.heads * nw.d) * 2 : (uint32_t)(H * D * 2);
    TileCtx t;
    if (!tile_begin<bf16_t, H, D, HW, NARROW, SP>(P, t, nw)) return;
    constexpr int ENT = TILE_CHUNK * 2, LIVE = ENT + TILE_R * TILE_WT_STRIDE_BF16, PIECE = SP > 1 ? 2 * TILE_PART_FLOATS : LIVE;
    static_assert(PIECE >= LIVE, "the lists fit");
    __shared__ __attribute__((aligned(16))) float piece[HW][PIECE];
    int2 *ent = reinterpret_cast<int2 *>(piece[t.wv]);
    uint32_t *const wt = reinterpret_cast<uint32_t *>(piece[t.wv] + ENT);         // (turned as in the float32 kernel)
    const int c = t.c, g = t.g;
    const uint32_t offc = t.offv;
    const char *qb = reinterpret_cast<const char *>(q), *db = reinterpret_cast<const char *>(d_o);
    const uint32_t *const pds_h = pds + (size_t)t.head * (size_t)P.n_edges;
    floatx4v ak[4], av[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) { ak[nb] = floatx4v{0.f, 0.f, 0.f, 0.f}; av[nb] = floatx4v{0.f, 0.f, 0.f, 0.f}; }
    struct Blk {
        uint2 qr[4], dr[4];
        uint32_t w[4];                                            // (p, ds) of the pairs (entry c, member 4 g + r)
        int mk[4];                                                // bit c of mk[r]: the pair (entry 4 g + r, member c) exists
    };
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        tile_stage_entries(P, ent, p0, cnt, t.lane);
        // (the positions of a block's pairs in the scratch are fetched one block ahead, as in the float32 kernel, so that the
        // (p, ds) loads leave with the row loads; positions past the group's end are read at its last entry: their masks are
        // empty.  The four registers this takes are why the kernel is compiled for five wavefronts per SIMD, not six: with
        // six it spills and loses what the prefetch gains)
        auto positions = [&](int b, int (&pos)[4]) { tile_pair_positions(P, min(p0 + TILE_R * b + c, t.p_end - 1), g, pos); };
        int pos_ahead[4], ahead_of = -1;
        auto issue = [&](Blk &B, int b) {
            const int4 e01 = *reinterpret_cast<const int4 *>(&ent[TILE_R * b + 4 * g]);
            const int4 e23 = *reinterpret_cast<const int4 *>(&ent[TILE_R * b + 4 * g + 2]);
            const int idxv[4] = {e01.x, e01.z, e23.x, e23.z};
            B.mk[0] = e01.y; B.mk[1] = e01.w; B.mk[2] = e23.y; B.mk[3] = e23.w;
            int pos[4];
            if (b == ahead_of) {
#pragma unroll
                for (int r = 0; r < 4; ++r) pos[r] = pos_ahead[r];
            } else {
                positions(b, pos);
            }
            if (b + 1 < nblk) positions(b + 1, pos_ahead);
            ahead_of = b + 1;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t off = (uint32_t)idxv[r] * RB + offc;
                B.qr[r] = tile_row4_bf16<NARROW>(qb + off);
                B.dr[r] = tile_row4_bf16<NARROW>(db + off);
                B.w[r] = pds_h[(uint32_t)pos[r]];
            }
        };
        auto compute = [&](const Blk &B) {
            *reinterpret_cast<uintx4v *>(wt + c * TILE_WT_STRIDE_BF16 + 4 * g) = uintx4v{B.w[0], B.w[1], B.w[2], B.w[3]};
            wave_lds_fence();
            uint32_t w[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] = wt[(4 * g + r) * TILE_WT_STRIDE_BF16 + c];
            wave_lds_fence();                                     // (read before the next block's are written)
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] &= (uint32_t)__builtin_amdgcn_sbfe(B.mk[r], c, 1);       // the scratch of pairs that do not exist is not initialised
            Bf4 pa, da;
            pa.u[0] = pack_lo16(w[0], w[1]); pa.u[1] = pack_lo16(w[2], w[3]);
            da.u[0] = pack_hi16(w[0], w[1]); da.u[1] = pack_hi16(w[2], w[3]);
            tile_axpy_bf16(da, B.qr, ak);
            tile_axpy_bf16(pa, B.dr, av);
        };
        tile_walk<Blk>(nblk, issue, compute);
        wave_lds_fence();
    }
    if constexpr (SP > 1) {
        constexpr int NEXT = (HW / SP) * PIECE;
        tile_park(piece[t.wv], ak, t.lane);
        tile_park(piece[t.wv] + TILE_PART_FLOATS, av, t.lane);
        __syncthreads();
        const float *const part0 = piece[t.wv % (HW / SP)];
        tile_meet_and_store<SP, H, D, NARROW>(part0, NEXT, t, dk, ws_dk, nw);
        tile_meet_and_store<SP, H, D, NARROW>(part0 + TILE_PART_FLOATS, NEXT, t, dv, ws_dv, nw);
    } else {
        tile_store_rows<H, D, false, NARROW>(t, ak, 1.f, dk, ws_dk, nw);
        tile_store_rows<H, D, false, NARROW>(t, av, 1.f, dv, ws_dv, nw);
    }
}

// Source side without the scratch: p and ds of a block's pairs are formed again from the entries' q and dO rows, which are
// loaded for the products over the entries anyway and turned in LDS, the members' k and v rows (held as operands) and the
// entries' (lse, delta), which the destination side leaves in `stat` (n, H).
// Why: the scratch holds 4 bytes per pair and head, as much as the node tensors on a dense graph, and reading it back is a
// gather of 4-byte words over 16 to 32 cache lines per instruction.  At L = 32768, k = 8, 16 heads the stores cost the
// destination side 70 of 295 us and the gathers this side 105 of 370 (the kernels without them, timing only); four more
// bfloat16 matrix instructions and two turns in LDS per block cost 70: 295 + 370 -> 237 + 315 us, the step 890 -> 782.
// Both backward kernels together at 8 heads: L = 8192, k = 4 60.8 -> 57.0 us; L = 4096, k = 32 64.7 -> 48.7; window 128 39.7 ->
// 30.9; L = 32768, k = 2 235 -> 221; 32-graph batch 102.5 -> 99.2; L = 512 and L = 8192 with dropout level.  (6 heads of 50
// columns with dropout lost 2 %: heads of fewer than 64 columns keep the scratch.)  float32 keeps it too: there the two
// products are 1024 cycles of the matrix pipeline per block.  122 registers: compiled for four wavefronts per SIMD.
template <int H, int D, int HW, int WPE, bool DROP, int SP = 1>
__global__ __launch_bounds__(HW * WAVE) __attribute__((amdgpu_waves_per_eu(WPE))) void k_attn_bwd_src_tile_bf16_again(
    bpt_plan P, const bf16_t *__restrict__ q, const bf16_t *__restrict__ k, const bf16_t *__restrict__ v, const bf16_t *__restrict__ d_o,
    const float2 *__restrict__ stat, bf16_t *__restrict__ dk, bf16_t *__restrict__ dv, float *__restrict__ ws_dk, float *__restrict__ ws_dv,
    float scale, float scale_log2e, uint32_t drop_thr, uint32_t drop_seed, float drop_inv) {
    constexpr uint32_t RB = H * D * 2;
    const Narrow nw{};
    TileCtx t;
    if (!tile_begin<bf16_t, H, D, HW, false, SP>(P, t, nw)) return;
    // a wavefront's piece: its entry list, the rows being turned, the entries' (lse, delta); afterwards (SP > 1) what it has summed up
    constexpr int ENT = TILE_CHUNK * 2, ROWS = 2 * TILE_ROWS_FLOATS_BF16 + 4 * TILE_R, LIVE = ENT + ROWS + 2 * TILE_R, PIECE = SP > 1 ? 2 * TILE_PART_FLOATS : LIVE;
    static_assert(PIECE >= LIVE && ROWS >= TILE_R * TILE_TURN_STRIDE, "the lists and the turned sums fit");
    __shared__ __attribute__((aligned(16))) float piece[HW][PIECE];
    int2 *ent = reinterpret_cast<int2 *>(piece[t.wv]);
    char *const q_lds = reinterpret_cast<char *>(piece[t.wv] + ENT), *const d_lds = q_lds + 4 * TILE_ROWS_FLOATS_BF16;
    float2 *const st_lds = reinterpret_cast<float2 *>(piece[t.wv] + ENT + ROWS);
    TileEntryRegs er;
    if (t.p_end > t.p_begin) tile_ask_entries(P, t.p_begin, min(TILE_CHUNK, t.p_end - t.p_begin), t.lane, er);
    issue_loads_first();
    const int c = t.c, g = t.g;
    const char *qb = reinterpret_cast<const char *>(q), *db = reinterpret_cast<const char *>(d_o);
    const float2 *const stat_h = stat + t.head;
    Bf8 kb[2], vb[2];
    {
        uint32_t off[2];
        uintx4v kr[2], vr[2];
        tile_member_offsets<RB>(t, off);
        tile_ask_rows_bf16(reinterpret_cast<const char *>(k), off, kr);
        tile_ask_rows_bf16(reinterpret_cast<const char *>(v), off, vr);
        tile_put_rows_bf16(q_lds, kr, t.lane);
        tile_put_rows_bf16(d_lds, vr, t.lane);
        wave_lds_fence();
        tile_operand_bf16(q_lds, c, g, kb);
        tile_operand_bf16(d_lds, c, g, vb);
        wave_lds_fence();
    }
    floatx4v ak[4], av[4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) { ak[nb] = floatx4v{0.f, 0.f, 0.f, 0.f}; av[nb] = floatx4v{0.f, 0.f, 0.f, 0.f}; }
    struct Blk {
        uintx4v qr[2], dr[2];
        float2 ld;                                                // (lse, delta) of entry c, in the first lane group
        int xe[DROP ? 4 : 1];
    };
    for (int p0 = t.p_begin; p0 < t.p_end; p0 += TILE_CHUNK) {
        const int cnt = min(TILE_CHUNK, t.p_end - p0), nblk = (cnt + TILE_R - 1) / TILE_R;
        if (p0 != t.p_begin) tile_ask_entries(P, p0, cnt, t.lane, er);
        tile_put_entries(er, ent, cnt, t.lane);
        auto issue = [&](Blk &B, int b) {
            if constexpr (DROP) tile_pair_eids(P, p0 + TILE_R * b + 4 * g, t.p_end, c, B.xe);
            if (g == 0) B.ld = stat_h[(size_t)ent[TILE_R * b + c].x * H];
            uint32_t off[2];
            tile_entry_offsets<RB>(t, ent + TILE_R * b, off);
            tile_ask_rows_bf16(qb, off, B.qr);
            tile_ask_rows_bf16(db, off, B.dr);
        };
        Blk B;
        issue(B, 0);
        for (int b = 0; b < nblk; ++b) {
            int mk[4], xe[DROP ? 4 : 1];
            tile_masks(ent + TILE_R * b, g, mk);
#pragma unroll
            for (int r = 0; r < (DROP ? 4 : 0); ++r) xe[r] = B.xe[r];
            tile_put_rows_bf16(q_lds, B.qr, t.lane);
            tile_put_rows_bf16(d_lds, B.dr, t.lane);
            if (g == 0) st_lds[c] = B.ld;
            wave_lds_fence();
            if (b + 1 < nblk) issue(B, b + 1);
            issue_loads_first();
            Bf8 row[2];
            tile_operand_bf16(q_lds, c, g, row);
            const floatx4v st = tile_dot_bf16(row, kb);
            const floatx4v l01 = *reinterpret_cast<const floatx4v *>(&st_lds[4 * g]), l23 = *reinterpret_cast<const floatx4v *>(&st_lds[4 * g + 2]);
            const float lse_e[4] = {l01[0], l01[2], l23[0], l23[2]}, delta_e[4] = {l01[1], l01[3], l23[1], l23[3]};
            tile_operand_bf16(d_lds, c, g, row);
            const floatx4v dp = tile_dot_bf16(row, vb);
            float pe[4], ds[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = where_pair_or_zero(mk[r], c, __builtin_amdgcn_exp2f(st[r] * scale_log2e - lse_e[r]));
                float mt = 1.f;                                   // dropout multiplier of this pair (as in the forward)
                if constexpr (DROP)
                    mt = dropout_keep((uint32_t)xe[DROP ? r : 0] * (uint32_t)H + (uint32_t)t.head, drop_seed, drop_thr, drop_inv);
                ds[r] = where_pair_or_zero(mk[r], c, p * (dp[r] * mt - delta_e[r]) * scale);
                pe[r] = p * mt;
            }
            Bf4 pa, da;
            da.u[0] = pack_bf16(ds[0], ds[1]); da.u[1] = pack_bf16(ds[2], ds[3]);
            pa.u[0] = pack_bf16(pe[0], pe[1]); pa.u[1] = pack_bf16(pe[2], pe[3]);
            tile_axpy_rows_bf16(da, q_lds, c, g, ak);
            tile_axpy_rows_bf16(pa, d_lds, c, g, av);
            wave_lds_fence();                                     // (read before the next block's are written)
            issue_loads_first();
        }
    }
    float *const turn = reinterpret_cast<float *>(q_lds);
    if constexpr (SP > 1) {
        tile_sums_by_row(turn, ak, c, g);
        tile_sums_by_row(turn, av, c, g);
        constexpr int NEXT = (HW / SP) * PIECE;
        tile_park(piece[t.wv], ak, t.lane);
        tile_park(piece[t.wv] + TILE_PART_FLOATS, av, t.lane);
        __syncthreads();
        const float *const part0 = piece[t.wv % (HW / SP)];
        tile_meet_and_store<SP, H, D, false>(part0, NEXT, t, dk, ws_dk, nw);
        tile_meet_and_store<SP, H, D, false>(part0 + TILE_PART_FLOATS, NEXT, t, dv, ws_dv, nw);
    } else {
        tile_store_sums<H, D>(t, turn, ak, dk, ws_dk);
        tile_store_sums<H, D>(t, turn, av, dv, ws_dv);
    }
}

// Backward, destination side.  Writes (p, ds) of every pair to pds[(t * H + head)], t = the pair's
// position (entry * R + member) in the SOURCE-side plan, which P.grp_pairs gives for every
// (entry, member) of this plan (a spare position for members the entry does not have).  One store per
// entry and quad of members: lane l carries the pair of member 4c + l % 4; the same register of ds values is
// the A operand of the MFMA that accumulates dq.  The members' q rows live in LDS.
template <typename T, int H, int D, int R, int HS, bool DROP, bool BIAS>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(grp_wpe<T, Lay<T, H / HS, D>::EPL, R>()))) void k_attn_bwd_dst_grp(
    bpt_plan P, const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v, const T *__restrict__ o,
    const T *__restrict__ d_o, const float *__restrict__ lse, T *__restrict__ dq, float2 *__restrict__ pds,
    float *__restrict__ ws_dq, float scale, float scale_log2e, uint32_t drop_thr, uint32_t drop_seed, float drop_inv,
    const float *__restrict__ bias, float *__restrict__ ds_out) {
    constexpr int HL = H / HS, CF = H * D;                  // heads of this wavefront's slice; elements of a full row
    using L = Lay<T, HL, D>;
    constexpr int EPL = L::EPL, NQ = R / 4, GRP_BATCH = BIAS ? 1 : grp_batch<L::EPL>()   /* the score term's registers take the place of a second entry */;
    static_assert(H % HS == 0 && R % 4 == 0 && L::LPH >= 4, "members are handled in quads inside the lanes of one head");
    GroupHead<R> gh;
    if (!fetch_group<R, HS>(P, gh)) return;
    const int slice = group_slice<R, HS>(), coff = slice * HL * D;
    const int lane = threadIdx.x, head = slice * HL + lane / L::LPH;
    const uint32_t loff = (uint32_t)((coff + L::off(lane, 0)) * sizeof(T));
    const int mine = lane & 3;
    const uint32_t hoff = (uint32_t)head * 8u, poff = (uint32_t)mine * 4u;
    const int4 *entries = reinterpret_cast<const int4 *>(P.grp_entries);
    struct Batch {
        RawRow<T, HL, D> kr[GRP_BATCH], vr[GRP_BATCH];
        int mk[GRP_BATCH], pz[GRP_BATCH], xp[GRP_BATCH][NQ];
        int xl[GRP_BATCH][BIAS ? NQ : 1];           // edge id of (entry, member 4c + lane % 4): where ds_out gets this lane's ds
        float bz[GRP_BATCH][BIAS ? NQ : 1];         // score term of (entry, member 4c + lane % 4), this lane's head
    };
    const int4 *eids4 = reinterpret_cast<const int4 *>(P.grp_eids);
    __shared__ float4 q_lds[R * (EPL / 4) * WAVE];
    float dov[R][EPL], delta_s[R], lse2[R];
    floatx4 dqa[NQ][EPL];                       // [quad c][row register t][member 4c + i], as the source-side kernel's accumulators
#pragma unroll
    for (int m = 0; m < R; ++m) {
        const uint32_t row = (uint32_t)max(gh.rows[m], 0);
        float ov[EPL], qr[EPL];
        load_row32<T, HL, D, CF>(o, row, loff, ov);
        load_row32<T, HL, D, CF>(d_o, row, loff, dov[m]);
        load_row32<T, HL, D, CF>(q, row, loff, qr);
        lds_put_row<EPL>(q_lds + m * (EPL / 4) * WAVE, lane, qr);
        delta_s[m] = head_sum<L::LPH>(dot_n<EPL>(dov[m], ov)) * scale;
        lse2[m] = lse[(size_t)row * H + head];
    }
#pragma unroll
    for (int c = 0; c < NQ; ++c)
#pragma unroll
        for (int t = 0; t < EPL; ++t) dqa[c][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int p0 = gh.begin; p0 < gh.end; p0 += GRP_CHUNK) {
        const int cnt = min(GRP_CHUNK, gh.end - p0);
        // lanes past the end repeat the last entry with an empty mask
        int4 ent = entries[p0 + min(lane, cnt - 1)];
        ent.y = lane < cnt ? ent.y : 0;
        // edge ids of the lane's entry, four members per vector (the list is padded like the entries)
        int4 xe[R / 4];
        if constexpr (BIAS || DROP) {
#pragma unroll
            for (int c = 0; c < R / 4; ++c) xe[c] = eids4[(size_t)(p0 + min(lane, cnt - 1)) * (R / 4) + c];
        }
        auto load_batch = [&](Batch &B, int b) {
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                const uint32_t src = (uint32_t)__builtin_amdgcn_readlane(ent.x, b + e);
                B.mk[e] = __builtin_amdgcn_readlane(ent.y, b + e);
                B.pz[e] = DROP ? b + e : 0;                  // position of the entry in the chunk: the lane that holds its edge ids
                if constexpr (BIAS) {
#pragma unroll
                    for (int c = 0; c < R / 4; ++c) {
                        const uint32_t e0 = (uint32_t)__builtin_amdgcn_readlane(xe[c].x, b + e), e1 = (uint32_t)__builtin_amdgcn_readlane(xe[c].y, b + e);
                        const uint32_t e2 = (uint32_t)__builtin_amdgcn_readlane(xe[c].z, b + e), e3 = (uint32_t)__builtin_amdgcn_readlane(xe[c].w, b + e);
                        // lane l fetches the term of member 4c + l % 4; the quad's lanes hand it round when it is used
                        B.xl[e][c] = (int)(mine == 0 ? e0 : mine == 1 ? e1 : mine == 2 ? e2 : e3);
                        B.bz[e][c] = bias[(size_t)((uint32_t)B.xl[e][c] * (uint32_t)H) + head];
                    }
                }
                // lane l fetches the scratch positions of the pairs of members l % 4, 4 + l % 4, ... with this entry
                const char *pp = reinterpret_cast<const char *>(P.grp_pairs) + (size_t)((uint32_t)(p0 + b + e) * (uint32_t)(R * 4));
#pragma unroll
                for (int c = 0; c < NQ; ++c) B.xp[e][c] = *reinterpret_cast<const int *>(pp + (size_t)(poff + (uint32_t)(c * 16)));
                load_row32_raw<T, HL, D, CF>(k, src, loff, B.kr[e]);
                load_row32_raw<T, HL, D, CF>(v, src, loff, B.vr[e]);
            }
        };
        auto compute = [&](const Batch &B) {
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                float kv[EPL], vv[EPL];
                unpack_row<T, HL, D>(B.kr[e], kv);
                unpack_row<T, HL, D>(B.vr[e], vv);
                float wp[NQ], wd[NQ];
#pragma unroll
                for (int c = 0; c < NQ; ++c) { wp[c] = 0.f; wd[c] = 0.f; }
#pragma unroll
                for (int m = 0; m < R; ++m) {
                    if ((B.mk[e] >> m) & 1) {
                        float qm[EPL];
                        lds_get_row<EPL>(q_lds + m * (EPL / 4) * WAVE, lane, qm);
                        float s = dot_n<EPL>(qm, kv), dp = dot_n<EPL>(dov[m], vv);
                        head_sum2<L::LPH>(s, dp);
                        if constexpr (BIAS) s += quad_bcast(B.bz[e][BIAS ? m / 4 : 0], m);
                        float pe = __builtin_amdgcn_exp2f(fmaf(s, scale_log2e, -lse2[m]));
                        float mt = 1.f;                   // dropout multiplier of this pair (as in the forward kernel)
                        if constexpr (DROP) {
                            const int4 &x = xe[m / 4];
                            const int held = (m & 3) == 0 ? x.x : (m & 3) == 1 ? x.y : (m & 3) == 2 ? x.z : x.w;
                            const uint32_t edge = (uint32_t)__builtin_amdgcn_readlane(held, B.pz[e]);
                            mt = dropout_keep(edge * (uint32_t)H + (uint32_t)head, drop_seed, drop_thr, drop_inv);
                        }
                        const float ds = pe * fmaf(dp * mt, scale, -delta_s[m]);
                        pe *= mt;                         // what multiplies v (forward) and dO (dV)
                        wp[m / 4] = mine == (m & 3) ? pe : wp[m / 4];
                        wd[m / 4] = mine == (m & 3) ? ds : wd[m / 4];
                    }
                }
#pragma unroll
                for (int c = 0; c < NQ; ++c) {
                    if ((B.mk[e] >> (4 * c)) & 15) {      // (look-ahead batches past the group's end have empty masks)
                        char *w = reinterpret_cast<char *>(pds);
                        *reinterpret_cast<float2 *>(w + (size_t)((uint32_t)B.xp[e][c] * (uint32_t)(H * 8) + hoff)) = make_float2(wp[c], wd[c]);
                        // dL/d(score before scaling) in edge order (absent members write the spare row n_edges)
                        if constexpr (BIAS) ds_out[(size_t)((uint32_t)B.xl[e][c] * (uint32_t)H) + head] = wd[c];
                        // dq[member 4c + i] += ds[member] * k row: wd (0 for absent members) is the A operand
#pragma unroll
                        for (int t = 0; t < EPL; ++t) dqa[c][t] = __builtin_amdgcn_mfma_f32_4x4x1f32(wd[c], kv[t], dqa[c][t], 0, 0, 0);
                    }
                }
            }
        };
        // two-stage software pipeline: the rows of the next batch are in flight while one is used.  The loads
        // are unconditional (a branch around them would make the compiler drain the load queue at the join);
        // look-ahead past the end re-reads the chunk's last entry with an empty mask.
        Batch A, B;
        load_batch(A, 0);
        for (int b = 0; b < cnt; b += 2 * GRP_BATCH) {
            load_batch(B, b + GRP_BATCH);
            issue_loads_first();
            compute(A);
            issue_loads_first();
            load_batch(A, b + 2 * GRP_BATCH);
            issue_loads_first();
            compute(B);
            issue_loads_first();
        }
    }
#pragma unroll
    for (int m = 0; m < R; ++m) {
        if (gh.rows[m] < 0) continue;
        float rq[EPL];
#pragma unroll
        for (int t = 0; t < EPL; ++t) rq[t] = dqa[m / 4][t][m & 3];
        if (gh.slots[m] < 0) store_row<T, HL, D>(dq + (size_t)gh.rows[m] * CF + coff, lane, rq);
        else store_row_ws<T, HL, D>(ws_dq + (size_t)gh.slots[m] * CF + coff, lane, rq);
    }
}

// Backward, source side: dK[src] = sum ds * q[dst], dV[src] = sum p * dO[dst]; the (p, ds) of the pair
// (entry u, member m) of this plan sits at pds[(u * R + m) * H + head].  One load per entry and quad of
// members: lane l fetches the pair of member 4c + l % 4 for its head.  That is the A operand of
// v_mfma_f32_4x4x1 (16 blocks of 4 lanes: A_b[i] in lane 4b+i, B_b[j] in lane 4b+j, D_b[i][j] in register i
// of lane 4b+j): with a register of the entry's row as B, one instruction adds weight[member i] * row[..]
// to that register's slice of all four members' accumulators (register i of the result = member i).
template <typename T, int H, int D, int R, int HS>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(grp_wpe<T, Lay<T, H / HS, D>::EPL, R>()))) void k_attn_bwd_src_grp(
    bpt_plan P, const T *__restrict__ q, const T *__restrict__ d_o, const float2 *__restrict__ pds, T *__restrict__ dk,
    T *__restrict__ dv, float *__restrict__ ws_dk, float *__restrict__ ws_dv) {
    constexpr int HL = H / HS, CF = H * D;                  // heads of this wavefront's slice; elements of a full row
    using L = Lay<T, HL, D>;
    constexpr int EPL = L::EPL, NQ = R / 4, GRP_BATCH = grp_batch<L::EPL>();
    static_assert(H % HS == 0 && R % 4 == 0 && L::LPH >= 4, "members are handled in quads inside the lanes of one head");
    GroupHead<R> gh;
    if (!fetch_group<R, HS>(P, gh)) return;
    const int slice = group_slice<R, HS>(), coff = slice * HL * D;
    const int lane = threadIdx.x, head = slice * HL + lane / L::LPH;
    const uint32_t loff = (uint32_t)((coff + L::off(lane, 0)) * sizeof(T));
    const uint32_t woff = (uint32_t)(((lane & 3) * H + head) * 8);
    const int4 *entries = reinterpret_cast<const int4 *>(P.grp_entries);
    struct Batch {
        RawRow<T, HL, D> qr[GRP_BATCH], dr[GRP_BATCH];
        float2 w[GRP_BATCH][NQ];
        int mk[GRP_BATCH];
    };
    floatx4 ak[NQ][EPL], av[NQ][EPL];          // [quad c][row register t][member 4c + i]
#pragma unroll
    for (int c = 0; c < NQ; ++c)
#pragma unroll
        for (int t = 0; t < EPL; ++t) { ak[c][t] = floatx4{0.f, 0.f, 0.f, 0.f}; av[c][t] = floatx4{0.f, 0.f, 0.f, 0.f}; }
    for (int p0 = gh.begin; p0 < gh.end; p0 += GRP_CHUNK) {
        const int cnt = min(GRP_CHUNK, gh.end - p0);
        // lanes past the end repeat the last entry with an empty mask
        int4 ent = entries[p0 + min(lane, cnt - 1)];
        ent.y = lane < cnt ? ent.y : 0;
        auto load_batch = [&](Batch &B, int b) {
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                const uint32_t dst = (uint32_t)__builtin_amdgcn_readlane(ent.x, b + e);
                B.mk[e] = __builtin_amdgcn_readlane(ent.y, b + e);
                load_row32_raw<T, HL, D, CF>(q, dst, loff, B.qr[e]);
                load_row32_raw<T, HL, D, CF>(d_o, dst, loff, B.dr[e]);
                // the entry's R pairs, present or not (absent ones are zeroed before use)
                const char *pw = reinterpret_cast<const char *>(pds) + (size_t)((uint32_t)(p0 + b + e) * (uint32_t)(R * H * 8));
#pragma unroll
                for (int c = 0; c < NQ; ++c) B.w[e][c] = *reinterpret_cast<const float2 *>(pw + (size_t)(woff + (uint32_t)(c * 4 * H * 8)));
            }
        };
        auto compute = [&](const Batch &B) {
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                float qv[EPL], dv_[EPL];
                unpack_row<T, HL, D>(B.qr[e], qv);
                unpack_row<T, HL, D>(B.dr[e], dv_);
#pragma unroll
                for (int c = 0; c < NQ; ++c) {
                    if ((B.mk[e] >> (4 * c)) & 15) {
                        // all-ones where this lane's member has the edge: the scratch of absent pairs is not initialised
                        const int keep = __builtin_amdgcn_sbfe(B.mk[e], 4 * c + (lane & 3), 1);
                        const float pe = __int_as_float(__float_as_int(B.w[e][c].x) & keep);
                        const float ds = __int_as_float(__float_as_int(B.w[e][c].y) & keep);
#pragma unroll
                        for (int t = 0; t < EPL; ++t) {
                            ak[c][t] = __builtin_amdgcn_mfma_f32_4x4x1f32(ds, qv[t], ak[c][t], 0, 0, 0);
                            av[c][t] = __builtin_amdgcn_mfma_f32_4x4x1f32(pe, dv_[t], av[c][t], 0, 0, 0);
                        }
                    }
                }
            }
        };
        // two-stage software pipeline: the rows of the next batch are in flight while one is used.  The loads
        // are unconditional (a branch around them would make the compiler drain the load queue at the join);
        // look-ahead past the end re-reads the chunk's last entry with an empty mask.
        Batch A, B;
        load_batch(A, 0);
        for (int b = 0; b < cnt; b += 2 * GRP_BATCH) {
            load_batch(B, b + GRP_BATCH);
            issue_loads_first();
            compute(A);
            issue_loads_first();
            load_batch(A, b + 2 * GRP_BATCH);
            issue_loads_first();
            compute(B);
            issue_loads_first();
        }
    }
#pragma unroll
    for (int m = 0; m < R; ++m) {
        if (gh.rows[m] < 0) continue;
        float rk[EPL], rv[EPL];
#pragma unroll
        for (int t = 0; t < EPL; ++t) { rk[t] = ak[m / 4][t][m & 3]; rv[t] = av[m / 4][t][m & 3]; }
        if (gh.slots[m] < 0) {
            store_row<T, HL, D>(dk + (size_t)gh.rows[m] * CF + coff, lane, rk);
            store_row<T, HL, D>(dv + (size_t)gh.rows[m] * CF + coff, lane, rv);
        } else {
            store_row_ws<T, HL, D>(ws_dk + (size_t)gh.slots[m] * CF + coff, lane, rk);
            store_row_ws<T, HL, D>(ws_dv + (size_t)gh.slots[m] * CF + coff, lane, rv);
        }
    }
}

// Y[row] = sum over the row's edges of W[eid, head] * X[idx]: the row-group form of k_spmm_fast for the unfused ops.
// X[idx] is loaded once per entry for every member that has the edge; the weight of (entry, member 4c + lane % 4) is
// fetched by its edge id (grp_eids) and is the A operand of v_mfma_f32_4x4x1 exactly as in k_attn_bwd_src_grp.
template <typename T, int H, int D, int R, int HS>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(grp_wpe<T, Lay<T, H / HS, D>::EPL, R>()))) void k_spmm_grp(
    bpt_plan P, const T *__restrict__ W, const T *__restrict__ X, T *__restrict__ Y, float *__restrict__ ws, int accumulate) {
    constexpr int HL = H / HS, CF = H * D;                  // heads of this wavefront's slice; elements of a full row
    using L = Lay<T, HL, D>;
    constexpr int EPL = L::EPL, NQ = R / 4, GRP_BATCH = grp_batch<L::EPL>();
    static_assert(H % HS == 0 && R % 4 == 0 && L::LPH >= 4, "members are handled in quads inside the lanes of one head");
    GroupHead<R> gh;
    if (!fetch_group<R, HS>(P, gh)) return;
    const int slice = group_slice<R, HS>(), coff = slice * HL * D;
    const int lane = threadIdx.x, head = slice * HL + lane / L::LPH, mine = lane & 3;
    const uint32_t loff = (uint32_t)((coff + L::off(lane, 0)) * sizeof(T));
    const uint32_t last_edge = (uint32_t)max(P.n_edges, (int64_t)1) - 1u;
    const int4 *entries = reinterpret_cast<const int4 *>(P.grp_entries);
    const int4 *eids4 = reinterpret_cast<const int4 *>(P.grp_eids);
    struct Batch {
        RawRow<T, HL, D> xr[GRP_BATCH];
        float w[GRP_BATCH][NQ];
        int mk[GRP_BATCH];
    };
    floatx4 acc[NQ][EPL];                      // [quad c][row register t][member 4c + i]
#pragma unroll
    for (int c = 0; c < NQ; ++c)
#pragma unroll
        for (int t = 0; t < EPL; ++t) acc[c][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int p0 = gh.begin; p0 < gh.end; p0 += GRP_CHUNK) {
        const int cnt = min(GRP_CHUNK, gh.end - p0);
        // lanes past the end repeat the last entry with an empty mask
        int4 ent = entries[p0 + min(lane, cnt - 1)];
        ent.y = lane < cnt ? ent.y : 0;
        // edge ids of the lane's entry, four members per vector
        int4 xe[R / 4];
#pragma unroll
        for (int c = 0; c < R / 4; ++c) xe[c] = eids4[(size_t)(p0 + min(lane, cnt - 1)) * (R / 4) + c];
        auto load_batch = [&](Batch &B, int b) {
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                const uint32_t src = (uint32_t)__builtin_amdgcn_readlane(ent.x, b + e);
                B.mk[e] = __builtin_amdgcn_readlane(ent.y, b + e);
#pragma unroll
                for (int c = 0; c < NQ; ++c) {
                    const uint32_t e0 = (uint32_t)__builtin_amdgcn_readlane(xe[c].x, b + e), e1 = (uint32_t)__builtin_amdgcn_readlane(xe[c].y, b + e);
                    const uint32_t e2 = (uint32_t)__builtin_amdgcn_readlane(xe[c].z, b + e), e3 = (uint32_t)__builtin_amdgcn_readlane(xe[c].w, b + e);
                    // absent members carry the id n_edges: read the last edge instead, the mask zeroes the weight
                    const uint32_t el = min(mine == 0 ? e0 : mine == 1 ? e1 : mine == 2 ? e2 : e3, last_edge);
                    B.w[e][c] = ld_w(W + (size_t)el * H + head);
                }
                load_row32_raw<T, HL, D, CF>(X, src, loff, B.xr[e]);
            }
        };
        auto compute = [&](const Batch &B) {
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                float xv[EPL];
                unpack_row<T, HL, D>(B.xr[e], xv);
#pragma unroll
                for (int c = 0; c < NQ; ++c) {
                    if ((B.mk[e] >> (4 * c)) & 15) {
                        const int keep = __builtin_amdgcn_sbfe(B.mk[e], 4 * c + mine, 1);     // all-ones where the member has the edge
                        const float wt = __int_as_float(__float_as_int(B.w[e][c]) & keep);
#pragma unroll
                        for (int t = 0; t < EPL; ++t) acc[c][t] = __builtin_amdgcn_mfma_f32_4x4x1f32(wt, xv[t], acc[c][t], 0, 0, 0);
                    }
                }
            }
        };
        // two-stage software pipeline as in the fused kernels (unconditional loads; look-ahead past the end re-reads
        // the chunk's last entry with an empty mask)
        Batch A, B;
        load_batch(A, 0);
        for (int b = 0; b < cnt; b += 2 * GRP_BATCH) {
            load_batch(B, b + GRP_BATCH);
            issue_loads_first();
            compute(A);
            issue_loads_first();
            load_batch(A, b + 2 * GRP_BATCH);
            issue_loads_first();
            compute(B);
            issue_loads_first();
        }
    }
#pragma unroll
    for (int m = 0; m < R; ++m) {
        if (gh.rows[m] < 0) continue;
        float out[EPL];
#pragma unroll
        for (int t = 0; t < EPL; ++t) out[t] = acc[m / 4][t][m & 3];
        if (gh.slots[m] < 0) {
            if (accumulate) {                 // Y += the sum (rows in segments get theirs when the segments are combined)
                float old[EPL];
                load_row32<T, HL, D, CF>(Y, (uint32_t)gh.rows[m], loff, old);
#pragma unroll
                for (int t = 0; t < EPL; ++t) out[t] += old[t];
            }
            store_row<T, HL, D>(Y + (size_t)gh.rows[m] * CF + coff, lane, out);
        } else {
            store_row_ws<T, HL, D>(ws + (size_t)gh.slots[m] * CF + coff, lane, out);
        }
    }
}

// Sums, over the LPH neighbouring lanes of a head, of R values per lane, with the results spread over the lanes: a step over a
// pair of lanes halves the values a lane carries as long as it carries more than one (the other half goes to its partner),
// 12 + 6 + 3 instructions for 8 values over 8 lanes where 8 sums in every lane are 24.  Lanes are paired by the DPP patterns
// there are: mirrored within 16 and within 8, then exchanged in steps of 2 and 1.  Steps run from the widest pattern down;
// those that come before the last log2(R) add without halving.
template <int CTRL, int N> __device__ __forceinline__ void sum_halve(float (&x)[N], bool upper) {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        const float keep = upper ? x[N / 2 + i] : x[i], give = upper ? x[i] : x[N / 2 + i];
        x[i] = keep + dpp_mov<CTRL>(give);
    }
}
template <int LPH, int R> __device__ __forceinline__ float sum_scatter(float (&x)[R], int lane) {
    static_assert((LPH == 8 || LPH == 16) && (R == 4 || R == 8), "eight or sixteen lanes per head, four or eight values");
    if constexpr (LPH == 16) {
#pragma unroll
        for (int i = 0; i < R; ++i) x[i] += dpp_mov<0x140>(x[i]);
    }
    float y[4];
    if constexpr (R == 8) {
        sum_halve<0x141, 8>(x, (lane & 4) != 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = x[i];
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = x[i] + dpp_mov<0x141>(x[i]);
    }
    sum_halve<0x4E, 4>(y, (lane & 2) != 0);
    float z[2] = {y[0], y[1]};
    sum_halve<0xB1, 2>(z, (lane & 1) != 0);
    return z[0];
}
// which of the R values sum_scatter leaves in this lane; -1 where a lane further left has it too
template <int LPH, int R> __device__ __forceinline__ int sum_scatter_index(int lane) {
    const int l = lane % LPH;
    return l >= R ? -1 : l;
}

// y[eid, head] = <A[row, head, :], B[idx, head, :]> for every edge: the row-group form of k_sddmm_fast.  The
// members' A rows stay in registers, B[idx] is loaded once per entry and every member that has the edge takes its
// dot products with it; the edge id of (entry, member) comes from grp_eids.  TABLE: B is a (n, D) table whose rows
// all heads share (the rel_pos score term q[row] . table[idx], written as float32).
// All R products of an entry are formed (60 % of them belong to an edge at L = 8192, k = 4) and their sums over the head's lanes
// are spread over those lanes, so an entry is one store from all lanes, with the edge ids loaded a batch ahead.  One full sum,
// one edge id read across lanes and one 32-byte store per edge, with a branch around each, took 45 us at L = 8192, k = 4, 8
// heads float32 (two calls a training step 90.9 us), this form 37.5 (75.0); 16 heads L = 2048 43 for two, L = 512 29.
template <typename T, int H, int D, int R, int HS, bool TABLE = false, typename YT = T>
__global__ __launch_bounds__(WAVE) void k_sddmm_grp(bpt_plan P, const T *__restrict__ A, const T *__restrict__ B, YT *__restrict__ y) {
    constexpr int HL = H / HS, CF = H * D;                  // heads of this wavefront's slice; elements of a full row
    using L = Lay<T, HL, D>;
    constexpr int EPL = L::EPL, GRP_BATCH = 2;
    static_assert(H % HS == 0, "whole heads per slice");
    GroupHead<R> gh;
    if (!fetch_group<R, HS>(P, gh)) return;
    const int slice = group_slice<R, HS>(), coff = slice * HL * D;
    const int lane = threadIdx.x, head = slice * HL + lane / L::LPH;
    const uint32_t loff = (uint32_t)((coff + L::off(lane, 0)) * sizeof(T));
    const uint32_t toff = (uint32_t)((lane % L::LPH) * L::VE * sizeof(T));      // the lane's columns inside a table row
    const int4 *entries = reinterpret_cast<const int4 *>(P.grp_entries);
    const int member = sum_scatter_index<L::LPH, R>(lane);         // whose product this lane ends up with (-1: another lane has it too)
    float a[R][EPL];
#pragma unroll
    for (int m = 0; m < R; ++m) load_row32<T, HL, D, CF>(A, (uint32_t)max(gh.rows[m], 0), loff, a[m]);
    struct Batch {
        RawRow<T, HL, D> br[GRP_BATCH];
        int mk[GRP_BATCH], edge[GRP_BATCH];
    };
    for (int p0 = gh.begin; p0 < gh.end; p0 += GRP_CHUNK) {
        const int cnt = min(GRP_CHUNK, gh.end - p0);
        // lanes past the end repeat the last entry with an empty mask
        int4 ent = entries[p0 + min(lane, cnt - 1)];
        ent.y = lane < cnt ? ent.y : 0;
        auto load_batch = [&](Batch &Bt, int b) {
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                const uint32_t src = (uint32_t)__builtin_amdgcn_readlane(ent.x, b + e);
                Bt.mk[e] = __builtin_amdgcn_readlane(ent.y, b + e);
                Bt.edge[e] = P.grp_eids[(size_t)(p0 + min(b + e, cnt - 1)) * R + max(member, 0)];
                if constexpr (TABLE) load_row32_raw<T, HL, D, D>(B, src, toff, Bt.br[e]);
                else load_row32_raw<T, HL, D, CF>(B, src, loff, Bt.br[e]);
            }
        };
        auto compute = [&](const Batch &Bt) {
#pragma unroll
            for (int e = 0; e < GRP_BATCH; ++e) {
                float bv[EPL];
                unpack_row<T, HL, D>(Bt.br[e], bv);
                float x[R];
#pragma unroll
                for (int m = 0; m < R; ++m) x[m] = dot_n<EPL>(a[m], bv);
                const float s = sum_scatter<L::LPH, R>(x, lane);
                if (member >= 0 && ((Bt.mk[e] >> member) & 1)) Elem<YT>::st(y + (size_t)(uint32_t)Bt.edge[e] * H + head, s);
            }
        };
        // two-stage software pipeline as in the fused kernels (unconditional loads; look-ahead past the end re-reads
        // the chunk's last entry with an empty mask)
        Batch X0, X1;
        load_batch(X0, 0);
        for (int b = 0; b < cnt; b += 2 * GRP_BATCH) {
            load_batch(X1, b + GRP_BATCH);
            issue_loads_first();
            compute(X0);
            issue_loads_first();
            load_batch(X0, b + 2 * GRP_BATCH);
            issue_loads_first();
            compute(X1);
            issue_loads_first();
        }
    }
}

// ------------------------------------------------------------------------------------------
// rel_pos score term (modules/attention.py:69-71) over the plan of the destinations with the edge types as indices: the
// table's rows are shared by all heads and few (at most 1000, 64 columns), so the products go to the matrix cores.
// ------------------------------------------------------------------------------------------
// 16 consecutive elements as floats
template <typename T> __device__ __forceinline__ void rel_load16(const T *p, float (&out)[16]);
template <> __device__ __forceinline__ void rel_load16<float>(const float *p, float (&out)[16]) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const float4 x = *reinterpret_cast<const float4 *>(p + 4 * t);
        out[4 * t] = x.x; out[4 * t + 1] = x.y; out[4 * t + 2] = x.z; out[4 * t + 3] = x.w;
    }
}
template <> __device__ __forceinline__ void rel_load16<bf16_t>(const bf16_t *p, float (&out)[16]) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint4 x = *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(p) + 16 * t);
        const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            out[8 * t + 2 * i] = __uint_as_float(w[i] << 16);
            out[8 * t + 2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
    }
}

// floats of LDS that a wavefront of k_rel_bias_bwd stages the ds values (H heads, rows 4 floats longer than 64 slots: other banks) and the types
// of 64 slots in
constexpr int REL_STAGE_PITCH = WAVE + 4;
constexpr int REL_BWD_STAGE(int h) { return REL_STAGE_PITCH * h + WAVE; }

constexpr int REL_MAX_USED = 240;         // type numbers whose table rows fit the 64 KB of LDS of the score kernel

// A work item (a row or a segment of a long row) and the types and edge ids of its first 64 slots (lane l: slot b + l).  The plan has an edge:
// an item without any reads the types and ids of a slot that is there.
struct RelHead {
    int row, b, e, out_slot;
    int type, edge;
};
__device__ __forceinline__ void rel_head_load(const bpt_plan &P, const int4 item, int lane, RelHead &r) {
    // the item is the same for all lanes of the wavefront: keep it in scalar registers
    r.row = __builtin_amdgcn_readfirstlane(item.x); r.b = __builtin_amdgcn_readfirstlane(item.y);
    r.e = __builtin_amdgcn_readfirstlane(item.z); r.out_slot = __builtin_amdgcn_readfirstlane(item.w);
    const int slot = min(r.b + min(lane, max(min(WAVE, r.e - r.b), 1) - 1), (int)P.n_edges - 1);   // lanes past the end repeat the last slot
    r.type = P.idx[slot];
    r.edge = P.eid[slot];
}

// The rows of the table that a graph uses, as floats in LDS: row u (`pitch` floats apart) = table[used_types[u]].  All
// threads of the workgroup.
template <typename T>
__device__ __forceinline__ void rel_table_to_lds(const T *__restrict__ table, const int32_t *__restrict__ used_types, int n_used, float *lds,
                                                 int pitch) {
    constexpr int AHEAD = 4;                                      // (round trips of two dependent loads each: four rows a thread side by side)
    const int n = n_used * 16, step = (int)blockDim.x;
    for (int x = threadIdx.x; x < n; x += AHEAD * step) {
        int type[AHEAD];
        float4 row[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) type[i] = used_types[min(x + i * step, n - 1) >> 4];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) row[i] = load4<T>(table + (size_t)type[i] * 64 + (min(x + i * step, n - 1) & 15) * 4);
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            if (x + i * step < n) *reinterpret_cast<float4 *>(lds + ((x + i * step) >> 4) * pitch + ((x + i * step) & 15) * 4) = row[i];
    }
}

// bias[eid[p], head] = q[row(p), head, :] . table[used_types[idx[p]], :] for every slot p of the plan (idx = the number of
// the edge's type among the n_used types that occur).  The heads of an item's row are rows of the A operand of
// v_mfma_f32_16x16x4f32 (row number c of A = head c % H), 16 consecutive slots of the item the 16 columns of B; lane
// (g, c) holds columns 16 g .. 16 g + 15 of q for head c % H and of the table row of slot c, and receives the results of
// heads 4 g .. 4 g + 3 for slot c, which it stores as one vector where 4 g < H.  The table rows come from a copy in LDS
// (rows REL_LDS_PITCH floats apart, so that the 16 rows of an operand fall into different banks): fetched from memory
// block by block they would cost one round trip each, far longer than a block's products.  A wavefront takes
// REL_FWD_ITEMS work items and fetches for all of them at once first the items, then their q rows and the type numbers
// and edge ids of their first 64 slots.
constexpr int REL_FWD_ITEMS = 4, REL_LDS_PITCH = 68;
template <typename T, int H>
__global__ __launch_bounds__(BLOCK) void k_rel_bias_rows(bpt_plan P, const T *__restrict__ q, const T *__restrict__ table,
                                                         const int32_t *__restrict__ used_types, int n_used, float *__restrict__ bias) {
    constexpr int D = 64, K = REL_FWD_ITEMS;
    static_assert(H == 4 || H == 8 || H == 16, "four consecutive heads per lane");
    extern __shared__ float rel_lds[];
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const bool head_major = P.bias_by_pair != 0;                // results at bias[head * n_edges + eid] instead of bias[eid * H + head]
    if (blockIdx.x == 0 && threadIdx.x < H && !head_major) bias[(size_t)P.n_edges * H + threadIdx.x] = 0.f;     // the spare row the fused kernels read for absent pairs
    if (P.n_edges == 0) return;                                 // (rows, but no slot to read)
    // wavefront gw of GW takes the items gw, gw + GW, ...: the segments of a long row, which are neighbours and all full, go to
    // different wavefronts
    const int GW = (int)gridDim.x * WAVES_PER_BLOCK, i0 = (int)blockIdx.x * WAVES_PER_BLOCK + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int n_items = (int)P.n_items;
    const int4 *items = reinterpret_cast<const int4 *>(P.items);
    int4 desc[K];
#pragma unroll
    for (int k = 0; k < K; ++k) desc[k] = items[min(i0 + k * GW, n_items - 1)];
    rel_table_to_lds<T>(table, used_types, n_used, rel_lds, REL_LDS_PITCH);
    RelHead hd[K];
    float aq[K][16];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if (i0 + k * GW >= n_items) desc[k].z = desc[k].y;  // (past the last item: nothing to do)
        rel_head_load(P, desc[k], lane, hd[k]);
        rel_load16<T>(q + ((size_t)hd[k].row * H + (c % H)) * D + 16 * g, aq[k]);
    }
    __syncthreads();
    auto table_rows = [&](int type, int first, float (&bt)[16]) {          // of the 16 slots from `first` of a chunk (lane l: slot l)
        const float *row = rel_lds + lane_bcast(type, first + c) * REL_LDS_PITCH + 16 * g;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float4 x = *reinterpret_cast<const float4 *>(row + 4 * t);
            bt[4 * t] = x.x; bt[4 * t + 1] = x.y; bt[4 * t + 2] = x.z; bt[4 * t + 3] = x.w;
        }
    };
#pragma unroll
    for (int k = 0; k < K; ++k) {
        for (int p0 = hd[k].b; p0 < hd[k].e; p0 += WAVE) {
            const int cnt = min(WAVE, hd[k].e - p0);
            int type = hd[k].type, edge = hd[k].edge;
            if (p0 != hd[k].b) {                             // (items longer than 64 slots: the rest, fetched on the spot)
                const int slot = p0 + min(lane, cnt - 1);
                type = P.idx[slot]; edge = P.eid[slot];
            }
#pragma unroll
            for (int blk = 0; blk < 4; ++blk) {
                if (16 * blk < cnt) {
                    float bt[16];
                    table_rows(type, 16 * blk, bt);
                    const floatx4v acc = tile_dot(aq[k], bt);
                    const int e = lane_bcast(edge, 16 * blk + c);
                    if (16 * blk + c < cnt && 4 * g < H) {
                        if (head_major) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) bias[(size_t)(4 * g + r) * (size_t)P.n_edges + e] = acc[r];
                        } else {
                            *reinterpret_cast<float4 *>(bias + (size_t)e * H + 4 * g) = make_float4(acc[0], acc[1], acc[2], acc[3]);
                        }
                    }
                }
            }
        }
    }
}

// The same term over the TILE plan of the attention kernels, for a term kept in that plan's pair order (bias_by_pair:
// one value per pair and head at bias[head * n_edges + pair number]).  One wavefront per (tile, head), as in the attention
// kernels.  First the products of the tile's 16 member rows with every table row in use, QT[type number][member] (16
// type numbers per step: A = table rows, B = the members' q), which go to a wavefront-private piece of LDS; then the
// lanes walk the tile's pairs, which are consecutive numbers, and every pair picks its value by what pair_tm[number] =
// type number | member << 8 says.  The per-pair arrays are read and written in runs; the table rows in use are staged in
// LDS once per workgroup (fetched from memory step by step, each step waits for two dependent loads: 32 us against
// the products' 7).
//
// QT takes 64 bytes a type and wavefront, so with many types a compute unit holds a workgroup of eight wavefronts or less, and what counts is how
// few round trips and products a tile costs: a workgroup then keeps the table rows for all of its tiles, and a wavefront has its next tile's
// pairs, q rows and places in the plan on their way.  ONE: a workgroup for every tile, where all fit the chip at once or a compute unit holds 24
// wavefronts; other wavefronts are what hides the round trips there (float32 L = 8192, k = 4 25.6 -> 21.8 us, bfloat16 level).
// float32 leaves out the sixteens of types that no pair of the tile has, which its first loads tell for up to 256 (512) pairs (6 of 11 sixteens
// are left at L = 8192, k = 8 both ways, 3 of 4 at k = 4; a look through longer tiles' pairs cost what it gave).  bfloat16 multiplies on
// bfloat16 matrix instructions: the same products, summed in float32.
// Against a workgroup for every tile and float32 products throughout: float32 8 heads L = 8192, k = 4 (55 types) 25.7 -> 21.8 us, 32-graph batch (43)
// 36.7 -> 32.6, L = 8192, k = 8 both ways (173) 222 -> 65, 16 heads L = 4096, k = 16 (140) 56 -> 45, L = 100 5.1 -> 5.3; bfloat16 8 heads L = 32768,
// k = 2 (33) 59 -> 30, 16 heads a batch with k = 20 (105) 68 -> 24, L = 2048 12.5 -> 6.9.
template <typename T> struct RelTile;
template <> struct RelTile<float> {
    static constexpr int PITCH = REL_LDS_PITCH * 4;              // bytes between the table rows in LDS
    struct Row { float v[16]; };                                  // columns 16 t + 4 g + e of a 64-column row
    static __device__ __forceinline__ void cols(const float *row, int g, Row &out) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float4 x = *reinterpret_cast<const float4 *>(row + 16 * t + 4 * g);
            out.v[4 * t] = x.x; out.v[4 * t + 1] = x.y; out.v[4 * t + 2] = x.z; out.v[4 * t + 3] = x.w;
        }
    }
    static __device__ __forceinline__ floatx4v dot(const Row &a, const Row &b) { return tile_dot(a.v, b.v); }
};
template <> struct RelTile<bf16_t> {
    static constexpr int PITCH = TILE_KT_BYTES_BF16;
    struct Row { Bf8 v[2]; };                                     // columns 16 g .. 16 g + 15
    static __device__ __forceinline__ void cols(const bf16_t *row, int g, Row &out) {
#pragma unroll
        for (int t = 0; t < 2; ++t) out.v[t].q = *reinterpret_cast<const uint4 *>(row + 16 * g + 8 * t);
    }
    static __device__ __forceinline__ floatx4v dot(const Row &a, const Row &b) { return tile_dot_bf16(a.v, b.v); }
};
template <typename T, int H, int HW, bool ONE>
__global__ __launch_bounds__(HW * WAVE) void k_rel_bias_tiles(bpt_plan P, const T *__restrict__ q, const T *__restrict__ table,
                                                              const int32_t *__restrict__ used_types, int n_used,
                                                              const int32_t *__restrict__ pair_tm, float *__restrict__ bias) {
    typedef RelTile<T> R;
    constexpr int D = 64, C = H * D, HS = H / HW, PIECES = D * sizeof(T) / 16;
    constexpr int AHEAD = ONE ? 4 : 8;                          // pairs per lane whose loads are in flight together
    extern __shared__ float rel_lds[];                        // the table rows in use, then QT of every wavefront
    char *const rows = reinterpret_cast<char *>(rel_lds);
    const int lane = threadIdx.x & (WAVE - 1), wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), c = lane & 15, g = lane >> 4;
    const int n16 = (n_used + 15) & ~15;
    float *const qt = reinterpret_cast<float *>(rows + (size_t)n_used * R::PITCH) + (size_t)wv * n16 * TILE_R;
    // the workgroup's places w in the XCD's range (tile w / HS, heads from (w % HS) HW): w0, w0 + step, ...
    const int x = blockIdx.x & 7, step = (int)(gridDim.x >> 3), w0 = (int)(blockIdx.x >> 3);
    const int grp0 = __builtin_amdgcn_readfirstlane(P.grp_chunks[x]), n_places = (__builtin_amdgcn_readfirstlane(P.grp_chunks[x + 1]) - grp0) * HS;
    const int n_mine = w0 < n_places ? (ONE ? 1 : (n_places - w0 + step - 1) / step) : 0;
    struct Place { int head, p_begin, p_end, row; };            // row: of member c
    struct Pairs { int first, end; };                           // the tile's pair numbers
    struct Asked { int tm[AHEAD]; typename R::Row q; };
    auto ask_place = [&](int i, Place &y) {
        const int w = w0 + min(i, n_mine - 1) * step, grp = grp0 + w / HS;
        y.head = (w % HS) * HW + wv;
        y.p_begin = P.grp_ptr[grp];
        y.p_end = P.grp_ptr[grp + 1];
        y.row = reinterpret_cast<const int2 *>(P.grp_members)[(size_t)grp * TILE_R + c].x;
    };
    auto ask_pairs = [&](const Place &y, Pairs &e) {
        const int4 *entries = reinterpret_cast<const int4 *>(P.grp_entries);
        const int b = __builtin_amdgcn_readfirstlane(y.p_begin), l = __builtin_amdgcn_readfirstlane(y.p_end);
        const int4 last = entries[max(l - 1, 0)];
        e.first = b < l ? entries[b].z : 0;
        e.end = b < l ? last.z + __popc((uint32_t)last.y) : 0;
    };
    auto ask = [&](const Place &y, const Pairs &e, Asked &a) {
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) a.tm[k] = pair_tm[max(min(e.first + lane + k * WAVE, e.end - 1), 0)];
        R::cols(q + (size_t)max(y.row, 0) * C + y.head * D, g, a.q);
    };
    Place at[3];
    Pairs pairs[2];
    Asked cur;
    if (n_mine > 0) ask_place(0, at[0]);
    if (!ONE && n_mine > 1) ask_place(1, at[1]);
    // four pieces of the table rows a thread side by side, by two dependent loads
    for (int y = threadIdx.x, n = n_used * PIECES; y < n; y += 4 * HW * WAVE) {
        int type[4];
        uint4 piece[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) type[i] = used_types[min(y + i * HW * WAVE, n - 1) / PIECES];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            piece[i] = *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(table + (size_t)type[i] * D) + 16 * (min(y + i * HW * WAVE, n - 1) % PIECES));
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (y + i * HW * WAVE < n)
                *reinterpret_cast<uint4 *>(rows + (size_t)((y + i * HW * WAVE) / PIECES) * R::PITCH + 16 * ((y + i * HW * WAVE) % PIECES)) = piece[i];
    }
    if (n_mine > 0) {
        ask_pairs(at[0], pairs[0]);
        ask(at[0], pairs[0], cur);
    }
    if (!ONE && n_mine > 1) {
        ask_pairs(at[1], pairs[1]);
        ask_place(2, at[2]);
    }
    __syncthreads();
    for (int i = 0; i < n_mine; ++i) {
        Asked next;
        Pairs after = pairs[1];
        Place later = at[2];
        if constexpr (!ONE) next = cur;
        if (!ONE && i + 1 < n_mine) {
            ask(at[1], pairs[1], next);
            ask_pairs(at[2], after);
            ask_place(i + 3, later);
        }
        issue_loads_first();
        const int first = pairs[0].first, end = pairs[0].end;
        // bit x: one of the lane's pairs has a type number in 16 x .. 16 x + 15.  Only where all pairs are at hand and a product takes long
        uint32_t sixteens = sizeof(T) == 4 && end - first <= AHEAD * WAVE ? 0u : ~0u;
        if (sizeof(T) == 4) {
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) sixteens |= 1u << ((cur.tm[k] >> 4) & 15);
        }
        for (int tb = 0; tb < n16; tb += TILE_R) {
            if (__builtin_amdgcn_ballot_w64((sixteens >> (tb / TILE_R)) & 1) == 0) continue;
            typename R::Row kr;
            R::cols(reinterpret_cast<const T *>(rows + (size_t)min(tb + c, n_used - 1) * R::PITCH), g, kr);
            const floatx4v st = R::dot(kr, cur.q);                // register r: (type number tb + 4 g + r, member c)
#pragma unroll
            for (int r = 0; r < 4; ++r) qt[(tb + 4 * g + r) * TILE_R + c] = st[r];
        }
        wave_lds_fence();
        // (the next tile's loads, and each round's, are waited for before this round's stores: behind them the wait would include the stores)
#pragma unroll
        for (int k = 0; k < (ONE ? 0 : AHEAD); ++k) asm volatile("" ::"v"(next.tm[k]));
        float *out = bias + (size_t)at[0].head * (size_t)P.n_edges;
        for (int y = first + lane; y < end; y += AHEAD * WAVE) {
            int nt[AHEAD];
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) nt[k] = pair_tm[min(y + (AHEAD + k) * WAVE, end - 1)];
            float val[AHEAD];
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) val[k] = qt[(cur.tm[k] & 0xff) * TILE_R + (cur.tm[k] >> 8)];
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) asm volatile("" ::"v"(nt[k]));
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) {
                if (y + k * WAVE < end) out[y + k * WAVE] = val[k];
                cur.tm[k] = nt[k];
            }
        }
        if constexpr (ONE) return;
        wave_lds_fence();                                         // (read before the next tile's products are written)
        cur = next;
        pairs[0] = pairs[1];
        pairs[1] = after;
        at[0] = at[1];
        at[1] = at[2];
        at[2] = later;
    }
}

// Gradients of that term from ds[e, head] = dL/d(score of edge e before scaling): dq[row] += sum over the row's slots of
// ds[eid] * table row of the slot's type (all heads), and the table's gradient, for type number u, the sum over the slots
// with idx = u and the heads of ds[eid, head] * q[row, head].  The wavefronts walk the plan's work items (rows and
// segments of long rows; a segment's part of dq goes to the workspace slot of the item, which k_rel_finish adds to dq), sixteen
// slots at a time, on v_mfma_f32_16x16x4f32 (lane (c, g) = (lane % 16, lane / 16)):
//   dq rows (16 x 64 columns, heads in the order that spreads a row over all lanes, fewer heads than 16: zeros) += ds (heads x slots) * table rows (slots x columns): step s takes slots
//     4 g + s; the table rows in use lie in LDS, columns 4 c .. 4 c + 3 of a row are one read a lane;
//   U (slots x 64 columns) = ds^T (slots x heads) * q (heads x columns): register r of lane (c, g) is slot 4 g + r, columns 4 c ...
// Both read ds from LDS, where an item's values of 64 slots are staged.  U's rows are added to the wavefront's own sums per type number
// in LDS: all at once where the sixteen types differ (66 % of the sixteens at L = 8192, k = 4), as one row where they are the same
// (34 %: a span's edges), one slot after the other else.  The wavefronts of a workgroup add their sums in a fixed order and the
// workgroup writes one partial table, part[(u * gridDim.x + block) * 64 + column], which k_rel_finish adds up.  Every sum has one
// owner and a fixed order.
// The sums leave two wavefronts a SIMD, so what bounds the walk are the round trips of an item's loads: two items' bodies (ds, q, dq) are
// in flight while one is used, and their types and edge ids two items ahead of that, so that no wait (they are in order) includes a
// load that has just left.  A launch has a wavefront for every item up to 512 workgroups.  Against a walk that took one slot after the other
// on the vector pipeline, with one item's loads ahead and a workgroup for 512 edges, kernel alone: 8 heads float32 L = 8192, k = 4 45.5 -> 39.5 us
// (30.7 of them without any of the products: 132 MB take 26 at the rate of a copy), k = 8 both ways 297 -> 180, L = 100 25.7 -> 8.0; 16 heads
// L = 4096, k = 16 186 -> 107; bfloat16 8 heads L = 32768, k = 2 177 -> 116, 16 heads L = 2048 57 -> 24, 666 nodes 136 -> 14; 4 heads L = 1024 20 -> 14,
// L = 16384, k = 2 48 -> 49.5, the one shape that gained nothing.  Neighbouring items in neighbouring wavefronts, for the lines that
// their ds values share: 39.5 -> 42.
// CS = 2: two wavefronts take an item together, each half of the columns of q, dq and the sums (rel_bwd_shape says when).
// NB (4 or 2) neighbouring columns of a lane: of q or dq, which start on any element here (attention itself asks for 16 bytes), and of the rows in LDS
template <int NB>
struct RelCols {
    float v[NB];
};
template <int NB, typename T> __device__ __forceinline__ RelCols<NB> rel_load(const T *p) {
    RelCols<NB> y;
    if constexpr (sizeof(T) == 4) {
        typedef float floatxu __attribute__((ext_vector_type(NB), aligned(4)));
        const floatxu x = *reinterpret_cast<const floatxu *>(p);
#pragma unroll
        for (int i = 0; i < NB; ++i) y.v[i] = x[i];
    } else {
        typedef uint32_t uintxe __attribute__((ext_vector_type(NB / 2), aligned(2)));
        const uintxe x = *reinterpret_cast<const uintxe *>(p);
#pragma unroll
        for (int i = 0; i < NB / 2; ++i) {
            y.v[2 * i] = __uint_as_float(x[i] << 16);
            y.v[2 * i + 1] = __uint_as_float(x[i] & 0xffff0000u);
        }
    }
    return y;
}
template <int NB, typename T> __device__ __forceinline__ void rel_store(T *p, const RelCols<NB> &y) {
    if constexpr (sizeof(T) == 4) {
        typedef float floatxu __attribute__((ext_vector_type(NB), aligned(4)));
        floatxu x;
#pragma unroll
        for (int i = 0; i < NB; ++i) x[i] = y.v[i];
        *reinterpret_cast<floatxu *>(p) = x;
    } else {
        typedef uint32_t uintxe __attribute__((ext_vector_type(NB / 2), aligned(2)));
        uintxe x;
#pragma unroll
        for (int i = 0; i < NB / 2; ++i) x[i] = pack_bf16(y.v[2 * i], y.v[2 * i + 1]);
        *reinterpret_cast<uintxe *>(p) = x;
    }
}
template <int NB> __device__ __forceinline__ RelCols<NB> rel_row_load(const float *p) {        // (p: a multiple of NB floats)
    typedef float floatx __attribute__((ext_vector_type(NB)));
    const floatx x = *reinterpret_cast<const floatx *>(p);
    RelCols<NB> y;
#pragma unroll
    for (int i = 0; i < NB; ++i) y.v[i] = x[i];
    return y;
}
template <int NB> __device__ __forceinline__ void rel_row_store(float *p, const RelCols<NB> &y) {
    typedef float floatx __attribute__((ext_vector_type(NB)));
    floatx x;
#pragma unroll
    for (int i = 0; i < NB; ++i) x[i] = y.v[i];
    *reinterpret_cast<floatx *>(p) = x;
}
template <int H, int NB>
struct RelBody {
    float d[H];              // ds of the lane's slot
    RelCols<NB> q[H / 4], old[H / 4]; // the lane's columns of heads 4 s + g: q, and the dq row that a whole row adds to
};
// the H values of ds that belong to `edge`: of a row of (n_edges, H), or one of each head's n_edges values
struct RelStride {
    uint32_t edge, head;
};
template <int H> __device__ __forceinline__ void rel_ds_load(const float *__restrict__ ds, int edge, RelStride by, float (&out)[H]) {
#pragma unroll
    for (int h = 0; h < H; ++h) out[h] = ds[(size_t)h * by.head + (size_t)edge * by.edge];
}
// (No load stands behind a condition: where paths meet, the waits count for the one with the fewest loads.  An item without edges reads
// places that are there, and a segment its row's dq.)
template <typename T, int H, int NB>
__device__ __forceinline__ void rel_body_load(const RelHead &r, const float *__restrict__ ds, RelStride by, const T *__restrict__ q,
                                              const T *__restrict__ dq, int g, int col, RelBody<H, NB> &y) {
    constexpr int D = 64;
    rel_ds_load<H>(ds, r.edge, by, y.d);
#pragma unroll
    for (int s = 0; s < H / 4; ++s) y.q[s] = rel_load<NB, T>(q + ((size_t)r.row * H + 4 * s + g) * D + col);
#pragma unroll
    for (int s = 0; s < H / 4; ++s) y.old[s] = rel_load<NB, T>(dq + ((size_t)r.row * H + 4 * s + g) * D + col);
}
template <int NB> __device__ __forceinline__ void rel_add(float *at, const RelCols<NB> &x) {
    RelCols<NB> v = rel_row_load<NB>(at);
#pragma unroll
    for (int i = 0; i < NB; ++i) v.v[i] += x.v[i];
    rel_row_store<NB>(at, v);
}
template <typename T, int H, int NW, int CS>
__global__ __launch_bounds__(NW * CS * WAVE) void k_rel_bias_bwd(bpt_plan P, const float *__restrict__ ds, const T *__restrict__ q,
                                                            const T *__restrict__ table, const int32_t *__restrict__ used_types, int n_used,
                                                            T *__restrict__ dq, float *__restrict__ ws_dq, float *__restrict__ part) {
    constexpr int D = 64, C = H * D, PITCH = REL_STAGE_PITCH, NB = 4 / CS;
    extern __shared__ float rel_lds[];                    // NW tables of n_used x 64 sums, the table rows in use, per wavefront 64 x H staged ds values and 64 types
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), c = lane & 15, g = lane >> 4;
    const int w = wave / CS, col = (wave % CS) * (D / CS) + NB * c;       // whose items; the lane's first column
    const RelStride by = P.bias_by_pair != 0 ? RelStride{1u, (uint32_t)P.n_edges} : RelStride{(uint32_t)H, 1u};
    float *acc = rel_lds + (size_t)w * n_used * D;
    const float *rows = rel_lds + (size_t)NW * n_used * D;
    float *stage = rel_lds + (size_t)(NW + 1) * n_used * D + (size_t)wave * REL_BWD_STAGE(H);
    int *types = reinterpret_cast<int *>(stage + PITCH * H);
    // wavefront (CS > 1: the CS wavefronts) gw of GW takes the items gw, gw + GW, ...: the segments of a long row, which are neighbours, go to
    // different ones
    const int GW = (int)gridDim.x * NW, i0 = (int)blockIdx.x * NW + w, n_items = (int)P.n_items, n_mine = i0 < n_items ? (n_items - i0 + GW - 1) / GW : 0;
    const int4 *items = reinterpret_cast<const int4 *>(P.items);
    RelHead hd[4];
    RelBody<H, NB> bd[2];
    auto body = [&](const RelHead &r, RelBody<H, NB> &y) { rel_body_load<T, H, NB>(r, ds, by, q, dq, g, col, y); };
    // ds and types of up to 64 slots (past the end: zeros; the last slot's type as a negative number, no two alike)
    auto put = [&](int cnt, const float (&d)[H], int type) {
#pragma unroll
        for (int h = 0; h < H; ++h) stage[h * PITCH + lane] = lane < cnt ? d[h] : 0.f;
        types[lane] = lane < cnt ? type : ~(type | lane << 8);    // (lanes past the end hold the last slot's type, which is less than 256)
        wave_lds_fence();
    };
    // the table row of a slot: past the end one of the item's own, whatever is multiplied by zero there (an infinite row of a type that the item
    // does not have stays out of it)
    static_assert(REL_MAX_USED <= 256, "a type fits eight bits");
    auto row_of = [](int type) { return (type ^ (type >> 31)) & 255; };
    // sixteen slots of those, cnt of them exist
    auto sixteen = [&](int j, int cnt, const RelCols<NB> (&qr)[H / 4], floatx4v (&dqa)[NB]) {
        const int4 t4 = *reinterpret_cast<const int4 *>(types + j + 4 * g);               // of slots 4 g .. 4 g + 3
        const int ty[4] = {t4.x, t4.y, t4.z, t4.w}, mine = types[j + c];
        // row c of the product is head 4 (c % 4) + c / 4, so that register s of lane group g is head 4 s + g
        floatx4v a4 = *reinterpret_cast<const floatx4v *>(stage + (4 * min(c & 3, H / 4 - 1) + (c >> 2)) * PITCH + j + 4 * g);   // the same slots
        if (H < 16 && (c & 3) >= H / 4) a4 = floatx4v{0.f, 0.f, 0.f, 0.f};
        float d[H / 4];
#pragma unroll
        for (int s = 0; s < H / 4; ++s) d[s] = stage[(4 * s + g) * PITCH + j + c];
        RelCols<NB> tv[4], before[4];                             // table rows of those slots; the sums of their types so far
#pragma unroll
        for (int r = 0; r < 4; ++r) tv[r] = rel_row_load<NB>(rows + row_of(ty[r]) * D + col);
#pragma unroll
        for (int r = 0; r < 4; ++r) before[r] = rel_row_load<NB>(acc + row_of(ty[r]) * D + col);
        // slots of one type: lane (c, g) compares the type of slot c with those of slots 4 g + s
        bool twice = false;
        uint64_t same0 = 0;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const bool same = mine == ty[s];
            twice = twice || (same && c != 4 * g + s);
            if (s == 0) same0 = __builtin_amdgcn_ballot_w64(same);
        }
        issue_loads_first();                                      // (one round trip through LDS after the types', not one a product)
        floatx4v u[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) u[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < H / 4; ++s)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) u[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(d[s], qr[s].v[nb], u[nb], 0, 0, 0);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) dqa[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[s], tv[s].v[nb], dqa[nb], 0, 0, 0);
        auto slot = [&](int r) {                                  // what slot 4 g + r adds to its type's sums
            RelCols<NB> x;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) x.v[nb] = u[nb][r];
            return x;
        };
        if (__builtin_amdgcn_ballot_w64(twice) == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                RelCols<NB> x = slot(r);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) x.v[nb] = before[r].v[nb] + x.v[nb];
                if (ty[r] >= 0) rel_row_store<NB>(acc + ty[r] * D + col, x);
            }
        } else if ((int)__popcll(same0 & 0xffffu) == cnt) {       // every slot that exists has the first one's type (those past the end add nothing)
            RelCols<NB> x;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) x.v[nb] = groups_sum((u[nb][0] + u[nb][1]) + (u[nb][2] + u[nb][3]));
            if (g == 0) rel_add<NB>(acc + ty[0] * D + col, x);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                for (int gg = 0; gg < 4; ++gg) {
                    if (g == gg && ty[r] >= 0) rel_add<NB>(acc + ty[r] * D + col, slot(r));
                    wave_lds_fence();
                }
        }
        wave_lds_fence();                                         // (read before the next are staged, and written before they are added)
    };
    auto item = [&](const RelHead &cur, const RelBody<H, NB> &b) {
        floatx4v dqa[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) dqa[nb] = floatx4v{0.f, 0.f, 0.f, 0.f};
        if (cur.b < cur.e) put(min(WAVE, cur.e - cur.b), b.d, cur.type);
        for (int p0 = cur.b; p0 < cur.e; p0 += TILE_R) {
            const int at = p0 - cur.b;
            if (at > 0 && (at & (WAVE - 1)) == 0) {               // (items longer than 64 slots: the rest, fetched on the spot)
                const int cnt = min(WAVE, cur.e - p0), slot = p0 + min(lane, cnt - 1);
                float rest[H];
                rel_ds_load<H>(ds, P.eid[slot], by, rest);
                put(cnt, rest, P.idx[slot]);
            }
            sixteen(at & (WAVE - 1), min(TILE_R, cur.e - p0), b.q, dqa);
        }
        if (cur.out_slot >= 0 || cur.b < cur.e) {
#pragma unroll
            for (int s = 0; s < H / 4; ++s) {
                const int at = (4 * s + g) * D + col;
                RelCols<NB> x;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) x.v[nb] = cur.out_slot < 0 ? b.old[s].v[nb] + dqa[nb][s] : dqa[nb][s];
                if (cur.out_slot < 0) rel_store<NB, T>(dq + (size_t)cur.row * C + at, x);
                else rel_row_store<NB>(ws_dq + (size_t)cur.out_slot * C + at, x);
            }
        }
    };
    int4 descs;                                                   // of 64 items, one a lane
    int n_here = 0;
    auto head = [&](int n, RelHead &r) {                          // (past the last one: nothing to read, nothing to write)
        auto of = [&](int x, int none) {
            const int v = __builtin_amdgcn_readlane(x, n & (WAVE - 1));
            return n < n_here ? v : none;
        };
        rel_head_load(P, make_int4(of(descs.x, 0), of(descs.y, 0), of(descs.z, 0), of(descs.w, -1)), lane, r);
    };
    auto begin = [&](int first) {
        n_here = min(WAVE, n_mine - first);
        descs = items[min(i0 + (first + min(lane, max(n_here, 1) - 1)) * GW, n_items - 1)];
#pragma unroll
        for (int n = 0; n < 4; ++n) head(n, hd[n]);
#pragma unroll
        for (int n = 0; n < 2; ++n) body(hd[n], bd[n]);
    };
    begin(0);
    issue_loads_first();                                          // (on their way while the table rows are fetched)
    for (int u = wave % CS; u < n_used; u += CS) acc[u * D + lane] = 0.f;
    rel_table_to_lds<T>(table, used_types, n_used, rel_lds + (size_t)NW * n_used * D, D);
    __syncthreads();
    for (int first = 0; first < n_mine; first += WAVE) {
        if (first > 0) begin(first);
        for (int n0 = 0; n0 < n_here; n0 += 4) {
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                issue_loads_first();
                item(hd[n], bd[n & 1]);
                issue_loads_first();
                body(hd[(n + 2) & 3], bd[n & 1]);
                head(n0 + n + 4, hd[n]);
            }
        }
    }
    __syncthreads();
    for (int u = wave; u < n_used; u += NW * CS) {
        float sum = rel_lds[(size_t)u * D + lane];
#pragma unroll
        for (int x = 1; x < NW; ++x) sum += rel_lds[((size_t)x * n_used + u) * D + lane];
        part[((size_t)u * gridDim.x + blockIdx.x) * D + lane] = sum;
    }
}

// dtable[type] = the sum of the n_parts partial rows of the type's number u = used[type] (zero for a type that does
// not occur).  One workgroup per type; 16 lanes cover a row (four columns each), so a wavefront reads four partial rows
// per load: lane group s of wave w adds the rows 4 w + s, 4 w + s + 16, ...; the 16 sums are then added in a fixed order.
template <typename T>
__device__ __forceinline__ void rel_table_sum_block(int type, const float *__restrict__ part, const int32_t *__restrict__ used, int n_parts,
                                                    T *__restrict__ dtable) {
    constexpr int D = 64, GROUPS = BLOCK / 16;
    __shared__ float4 sums[GROUPS][16];
    const int u = used[type], grp = threadIdx.x >> 4, c4 = (threadIdx.x & 15) * 4;
    if (u < 0) {
        if (threadIdx.x < 16) store4<T>(dtable + (size_t)type * D + c4, make_float4(0.f, 0.f, 0.f, 0.f));
        return;
    }
    const float *p = part + (size_t)u * n_parts * D + c4;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    int x = grp;
    for (; x + 7 * GROUPS < n_parts; x += 8 * GROUPS) {
        float4 t[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) t[k] = *reinterpret_cast<const float4 *>(p + (size_t)(x + k * GROUPS) * D);
#pragma unroll
        for (int k = 0; k < 8; ++k) { s.x += t[k].x; s.y += t[k].y; s.z += t[k].z; s.w += t[k].w; }
    }
    for (; x < n_parts; x += GROUPS) {
        const float4 t = *reinterpret_cast<const float4 *>(p + (size_t)x * D);
        s.x += t.x; s.y += t.y; s.z += t.z; s.w += t.w;
    }
    sums[grp][threadIdx.x & 15] = s;
    __syncthreads();
    if (threadIdx.x < 16) {
        float4 tot = sums[0][threadIdx.x];
#pragma unroll
        for (int k = 1; k < GROUPS; ++k) { const float4 t = sums[k][threadIdx.x]; tot.x += t.x; tot.y += t.y; tot.z += t.z; tot.w += t.w; }
        store4<T>(dtable + (size_t)type * D + c4, tot);
    }
}

// What is left after k_rel_bias_bwd, in one launch of n_types + n_heavy * C / 256 workgroups: the first n_types sum
// the partial tables (above), the others add the partial dq rows of the split rows to dq (one workgroup per split row
// and strip of 256 columns, in the order combine_sum_block uses).
template <typename T>
__global__ __launch_bounds__(BLOCK) void k_rel_finish(const float *__restrict__ part, const int32_t *__restrict__ used, int n_parts, int n_types,
                                                      T *__restrict__ dtable, const int32_t *__restrict__ heavy, const float *__restrict__ ws_dq,
                                                      T *__restrict__ dq, int C) {
    const int b = blockIdx.x;
    if (b < n_types) {
        rel_table_sum_block<T>(b, part, used, n_parts, dtable);
    } else {
        const int strips = C / 256, x = b - n_types;
        combine_sum_block4<T>(heavy + 3 * (x / strips), ws_dq, dq, C, true, x % strips);
    }
}

// Measurement aid: what the memory system delivers to row gathers.  Every wavefront reads `iters` batches of
// IN_FLIGHT pseudo-random 1 KB rows (16 bytes per lane, the access pattern of the attention kernels' neighbour rows)
// of a region and keeps a checksum, so that nothing but the loads is timed.
template <int IN_FLIGHT>
__global__ __launch_bounds__(BLOCK) void k_gather_probe(const float4 *__restrict__ base, uint32_t n_rows, int iters, float *__restrict__ sink) {
    const int lane = threadIdx.x & 63;
    uint32_t r = (uint32_t)((blockIdx.x * WAVES_PER_BLOCK + (threadIdx.x >> 6)) * 2654435761u);
    float acc = 0.f;
    for (int i = 0; i < iters; ++i) {
        float4 x[IN_FLIGHT];
#pragma unroll
        for (int u = 0; u < IN_FLIGHT; ++u) {
            r = r * 1664525u + 1013904223u;                       // row = high word of r * n_rows: two instructions per address
            x[u] = base[(size_t)__umulhi(r, n_rows) * 64 + lane];
        }
#pragma unroll
        for (int u = 0; u < IN_FLIGHT; ++u) acc += x[u].x + x[u].w;
    }
    if (acc == 12345.678f) sink[0] = acc;                      // never true for the zero / random data of the probe
}

// ------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------
inline int grid_for(const bpt_plan *p) { return (int)((p->n_items + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK); }

inline int check_plan(const bpt_plan *p, bool need_idx) {
    if (!p) return BPT_ERR_NULL;
    if (p->n_rows < 0 || p->n_edges < 0 || p->n_items < 0 || p->n_heavy < 0 || p->n_slots < 0) return BPT_ERR_SIZE;
    if (p->n_items > 0 && (!p->items || !p->rowptr)) return BPT_ERR_NULL;
    if (p->n_edges > 0 && (!p->eid || (need_idx && !p->idx))) return BPT_ERR_NULL;
    if (p->n_heavy > 0 && !p->heavy) return BPT_ERR_NULL;
    if (p->n_items < p->n_rows) return BPT_ERR_SIZE;     // every row owns at least one item
    if (p->n_groups < 0 || p->grp_R < 0 || p->grp_R > 32 || p->n_grp_entries < 0) return BPT_ERR_SIZE;
    if (p->n_groups > 0 && (!p->grp_members || !p->grp_ptr || !p->grp_chunks || (p->n_edges > 0 && !p->grp_entries))) return BPT_ERR_NULL;
    if (p->n_groups > 0 && (p->grp_max_chunk < 1 || p->grp_max_chunk > p->n_groups)) return BPT_ERR_SIZE;
    if (p->n_index_nodes < 0) return BPT_ERR_SIZE;
    return BPT_OK;
}

inline int check_shape(int h, int d, int dtype) {
    if (dtype != BPT_F32 && dtype != BPT_F64 && dtype != BPT_BF16) return BPT_ERR_DTYPE;
    if (h < 1 || d < 1 || (int64_t)h * d > (1 << 20)) return BPT_ERR_SHAPE;
    return BPT_OK;
}

inline size_t acc_size(int dtype) { return dtype == BPT_F64 ? 8 : 4; }
inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int launch_status() {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? BPT_OK : (int)e;
}

// (H, D) pairs with a fast instantiation.  bf16 needs C >= 512 (eight elements per 16-byte vector).
#define BPT_FAST_SHAPES_F32(X) X(4, 64) X(8, 64) X(16, 64) X(8, 32)
#define BPT_FAST_SHAPES_BF16(X) X(8, 64) X(16, 64)

inline bool fast_shape(int h, int d, int dtype) {
    if (g_force_generic.load(std::memory_order_relaxed)) return false;
#define X(HH, DD) if (h == HH && d == DD) return true;
    if (dtype == BPT_F32) { BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { BPT_FAST_SHAPES_BF16(X) }
#undef X
    return false;
}

constexpr int FAST_BATCH = 4;

// ---- generic launchers (dtype dispatch) ----
template <typename T, int MODE>
int run_sddmm_generic(const bpt_plan *P, const void *A, const void *B, void *y, int h, int d, hipStream_t s) {
    if (P->n_items == 0) return BPT_OK;
    hipLaunchKernelGGL((k_sddmm_generic<T, MODE>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)A, (const T *)B, (T *)y, h, d);
    return launch_status();
}

template <typename T, int MODE>
int run_spmm_generic(const bpt_plan *P, const void *W, const void *X, void *Y, void *ws, int h, int d, hipStream_t s) {
    using acc_t = typename Elem<T>::acc_t;
    if (P->n_items == 0) return BPT_OK;
    hipLaunchKernelGGL((k_spmm_generic<T, MODE>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)W, (const T *)X, (T *)Y, (acc_t *)ws, h, d);
    int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0) return st;
    hipLaunchKernelGGL((k_combine_sum<T>), dim3((int)P->n_heavy, (h * d + WAVE - 1) / WAVE, 1), dim3(BLOCK), 0, s, P->heavy,
                       (const acc_t *)ws, (T *)Y, (T *)nullptr, h * d, (size_t)0);
    return launch_status();
}

// blocks of k_softmax_split_quads a split row: the longest are many times the average (16 of 127 segments at L = 8192)
inline unsigned softmax_split_blocks(const bpt_plan *P) {
    return (unsigned)std::min<int64_t>(64, std::max<int64_t>(16, P->n_slots / P->n_heavy));
}
inline unsigned softmax_item_blocks(const bpt_plan *P, int q, int block) { return (unsigned)((P->n_items * QUAD_SLOTS * q + block - 1) / block); }
// How many workgroups in front of the items' take a split row each: none where the plan does not say how long its longest row is, or where
// one is longer than `longest`.  A workgroup's CU keeps some 64 lines in flight and the records of a span's edges lie in a line
// each: with the 8192 edges of the longest row of L = 8192 the forward took 39 us and the backward 51, in two launches 22 and 27.  Kernels,
// two or three launches -> one, forward and backward: 8 heads, L = 500, both ways 9.7 + 8.6 -> 7.2 + 6.4 us; L = 1000 10.9 + 10.0 -> 8.4 + 7.6;
// 16 graphs of up to 1024 17.9 + 15.4 -> 14.6 + 13.2.  Passes of the separate operators, which
// the host bounds there: L = 100 146 -> 139 us, L = 500 151 -> 143, the 16 graphs 212 -> 206.
// Rows of `deg` edges each, forward and backward, times as fast as the launches over segments: 4, 8 or 16 heads 1.2-1.8 and 1.3-2.5 for 100 to 16 000
// rows of 70 to 1000 edges.
constexpr int SM_WHOLE_EDGES = 1024;
inline int softmax_whole_rows(const bpt_plan *P, int longest = SM_WHOLE_EDGES) {
    if (P->n_heavy == 0 || P->max_degree <= 0 || P->max_degree > longest) return 0;
    return (int)((P->n_heavy + 7) & ~(int64_t)7);
}
// The same for the kernels with the heads side by side, whose workgroups have fewer slots the more heads there are.  Times as fast as the launches over
// segments, forward and backward: where the longest row is held at once (SM_CACHE edges a slot) 1.7-2.0 and 1.7-2.1 (1000 or 700 tokens of 1, 3
// and 5 heads), just past it 1.0 and 1.0 (6 heads, 700 or 1000), 0.85 and 0.9 with one row of 1024 beside 1000 of 64 (5 and 6 heads), 0.6-0.75 and 0.8 at
// 1024 with 12 heads and more; rows of up to 512 1.6 and 1.3-1.6 with 10 and 12 heads, 1.2-1.3 and 1.1-1.4 with 32 and 64.  A short row leaves
// most of its workgroup idle, which shows once the chip is full of them: one head, 70 edges 2 and 2.2 at 100 rows, 1.07 and 1.3 at 3000, 0.76
// and 0.83 at 16 000; 200 edges (four segments) 1.2 and 1.45 at 4000; in float64 1.0 and 1.5 at 1500 rows of 70, 0.8 and 1.1 at 3000, 1.1 and 1.3 at
// 3000 of 300 (five segments).
template <typename T> inline int softmax_whole_rows_heads(const bpt_plan *P, int h) {
    constexpr bool F64 = sizeof(T) == 8;
    if (P->n_heavy > (F64 ? 1536 : 3072) && P->n_slots < (F64 ? 5 : 4) * P->n_heavy) return 0;
    return softmax_whole_rows(P, std::min(SM_WHOLE_EDGES, std::max(SM_WHOLE_EDGES / 2, SM_CACHE * SM_WAVES * (WAVE / h))));
}

template <typename T, int Q>
int run_softmax_fwd_quads(const bpt_plan *P, const void *x, void *y, void *ws, hipStream_t s) {
    const int whole = softmax_whole_rows(P);
    if (whole > 0)
        hipLaunchKernelGGL((k_softmax_fwd_quads<T, Q, true>), dim3(whole + softmax_item_blocks(P, Q, SM_BLOCK)), dim3(SM_BLOCK), 0, s, *P, (const T *)x, (T *)y,
                           (float *)nullptr, whole);
    else
        hipLaunchKernelGGL((k_softmax_fwd_quads<T, Q, false>), dim3(softmax_item_blocks(P, Q, BLOCK)), dim3(BLOCK), 0, s, *P, (const T *)x, (T *)y, (float *)ws, 0);
    const int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0 || whole > 0) return st;
    hipLaunchKernelGGL((k_softmax_split_quads<T, Q, true>), dim3((int)P->n_heavy, softmax_split_blocks(P)), dim3(BLOCK), 0, s, *P, (const T *)x,
                       (const T *)nullptr, (T *)y, (const float *)ws);
    return launch_status();
}
template <typename T, int Q>
int run_softmax_bwd_quads(const bpt_plan *P, const void *y, const void *dy, void *dx, void *ws, hipStream_t s) {
    const int whole = softmax_whole_rows(P);
    if (whole > 0)
        hipLaunchKernelGGL((k_softmax_bwd_quads<T, Q, true>), dim3(whole + softmax_item_blocks(P, Q, SM_BLOCK)), dim3(SM_BLOCK), 0, s, *P, (const T *)y, (const T *)dy, (T *)dx,
                           (float *)nullptr, whole);
    else
        hipLaunchKernelGGL((k_softmax_bwd_quads<T, Q, false>), dim3(softmax_item_blocks(P, Q, BLOCK)), dim3(BLOCK), 0, s, *P, (const T *)y, (const T *)dy, (T *)dx, (float *)ws, 0);
    const int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0 || whole > 0) return st;
    hipLaunchKernelGGL((k_softmax_split_quads<T, Q, false>), dim3((int)P->n_heavy, softmax_split_blocks(P)), dim3(BLOCK), 0, s, *P, (const T *)y,
                       (const T *)dy, (T *)dx, (const float *)ws);
    return launch_status();
}
// four heads are one load: 4, 8 or 16 heads of float32 or bfloat16 in tensors that start on 16 bytes (8 would do for bfloat16)
template <typename T> bool softmax_quads(int h, const void *a, const void *b, const void *c) {
    return sizeof(T) != 8 && (h == 4 || h == 8 || h == 16) && aligned16(a) && aligned16(b) && aligned16(c);
}

template <typename T>
int run_softmax_fwd(const bpt_plan *P, const void *x, void *y, void *ws, int h, hipStream_t s) {
    using acc_t = typename Elem<T>::acc_t;
    if (P->n_items == 0) return BPT_OK;
    if constexpr (sizeof(T) != 8) {
        if (softmax_quads<T>(h, x, y, nullptr))
            return h == 4 ? run_softmax_fwd_quads<T, 1>(P, x, y, ws, s) : h == 8 ? run_softmax_fwd_quads<T, 2>(P, x, y, ws, s) : run_softmax_fwd_quads<T, 4>(P, x, y, ws, s);
    }
    if (h <= WAVE) {           // heads side by side; split rows in three steps over their segments
        acc_t *seg = P->n_heavy > 0 ? (acc_t *)ws : nullptr;
        const int whole = softmax_whole_rows_heads<T>(P, h);
        if (whole > 0)
            hipLaunchKernelGGL((k_softmax_fwd_heads<T, true>), dim3(whole + (unsigned)((P->n_items + SM_WAVES - 1) / SM_WAVES)), dim3(SM_BLOCK), 0, s,
                               *P, (const T *)x, (T *)y, h, (acc_t *)nullptr, whole);
        else
            hipLaunchKernelGGL((k_softmax_fwd_heads<T, false>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)x, (T *)y, h, seg, 0);
        int st = launch_status();
        if (st != BPT_OK || P->n_heavy == 0 || whole > 0) return st;
        hipLaunchKernelGGL((k_softmax_seg_rows<acc_t, true>), dim3((int)P->n_heavy), dim3(BLOCK), 0, s, P->heavy, seg, h);
        st = launch_status();
        if (st != BPT_OK) return st;
        hipLaunchKernelGGL((k_softmax_fwd_seg_finish<T>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)x, (T *)y, h, (const acc_t *)seg);
        return launch_status();
    }
    hipLaunchKernelGGL((k_softmax_fwd<T, 1>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)x, (T *)y, h);
    int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0) return st;
    hipLaunchKernelGGL((k_softmax_fwd<T, WAVES_PER_BLOCK>), dim3((int)P->n_heavy), dim3(BLOCK), 0, s, *P, (const T *)x, (T *)y, h);
    return launch_status();
}

template <typename T>
int run_softmax_bwd(const bpt_plan *P, const void *y, const void *dy, void *dx, void *ws, int h, hipStream_t s) {
    using acc_t = typename Elem<T>::acc_t;
    if (P->n_items == 0) return BPT_OK;
    if constexpr (sizeof(T) != 8) {
        if (softmax_quads<T>(h, y, dy, dx))
            return h == 4 ? run_softmax_bwd_quads<T, 1>(P, y, dy, dx, ws, s) : h == 8 ? run_softmax_bwd_quads<T, 2>(P, y, dy, dx, ws, s) : run_softmax_bwd_quads<T, 4>(P, y, dy, dx, ws, s);
    }
    if (h <= WAVE) {           // heads side by side; split rows in three steps over their segments
        acc_t *seg = P->n_heavy > 0 ? (acc_t *)ws : nullptr;
        const int whole = softmax_whole_rows_heads<T>(P, h);
        if (whole > 0)
            hipLaunchKernelGGL((k_softmax_bwd_heads<T, true>), dim3(whole + (unsigned)((P->n_items + SM_WAVES - 1) / SM_WAVES)), dim3(SM_BLOCK), 0, s,
                               *P, (const T *)y, (const T *)dy, (T *)dx, h, (acc_t *)nullptr, whole);
        else
            hipLaunchKernelGGL((k_softmax_bwd_heads<T, false>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)y, (const T *)dy, (T *)dx, h, seg, 0);
        int st = launch_status();
        if (st != BPT_OK || P->n_heavy == 0 || whole > 0) return st;
        hipLaunchKernelGGL((k_softmax_seg_rows<acc_t, false>), dim3((int)P->n_heavy), dim3(BLOCK), 0, s, P->heavy, seg, h);
        st = launch_status();
        if (st != BPT_OK) return st;
        hipLaunchKernelGGL((k_softmax_bwd_seg_finish<T>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)y, (const T *)dy, (T *)dx, h,
                           (const acc_t *)seg);
        return launch_status();
    }
    hipLaunchKernelGGL((k_softmax_bwd<T, 1>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)y, (const T *)dy, (T *)dx, h);
    int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0) return st;
    hipLaunchKernelGGL((k_softmax_bwd<T, WAVES_PER_BLOCK>), dim3((int)P->n_heavy), dim3(BLOCK), 0, s, *P, (const T *)y, (const T *)dy, (T *)dx, h);
    return launch_status();
}

template <typename T>
int run_nme_dB(const bpt_plan *P, const void *A, const void *dy, void *dB, int h, int d, hipStream_t s) {
    if (P->n_items == 0) return BPT_OK;
    hipLaunchKernelGGL((k_nme_dB_generic<T>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)A, (const T *)dy, (T *)dB, h, d);
    return launch_status();
}

#define DISPATCH_DTYPE(dtype, CALL)                     \
    switch (dtype) {                                    \
        case BPT_F32: { using T = float; return CALL; } \
        case BPT_F64: { using T = double; return CALL; }\
        case BPT_BF16: { using T = bf16_t; return CALL; }\
        default: return BPT_ERR_DTYPE;                  \
    }

int sddmm_generic(const bpt_plan *P, const void *A, const void *B, void *y, int h, int d, int dtype, hipStream_t s) {
    DISPATCH_DTYPE(dtype, (run_sddmm_generic<T, 0>(P, A, B, y, h, d, s)))
}
int sddmm_edge_generic(const bpt_plan *P, const void *A, const void *B, void *y, int h, int d, int dtype, hipStream_t s) {
    DISPATCH_DTYPE(dtype, (run_sddmm_generic<T, 1>(P, A, B, y, h, d, s)))
}
int spmm_generic(const bpt_plan *P, const void *W, const void *X, void *Y, void *ws, int h, int d, int dtype, hipStream_t s) {
    DISPATCH_DTYPE(dtype, (run_spmm_generic<T, 0>(P, W, X, Y, ws, h, d, s)))
}
int spmm_edge_generic(const bpt_plan *P, const void *W, const void *X, void *Y, void *ws, int h, int d, int dtype, hipStream_t s) {
    DISPATCH_DTYPE(dtype, (run_spmm_generic<T, 1>(P, W, X, Y, ws, h, d, s)))
}

// ---- fast launchers ----
// Wavefronts a work item for the kernels that walk single rows.  The fused kernels walk them on graphs of fewer than 1536 items (with
// row groups switched off: on any), the separate operators' SpMM where it is handed a plan without groups.  There a launch lasts
// as long as its longest item: 16 batches of four edges one after the other, each a round trip to memory.  Forward / destination
// side / source side, one -> four -> eight wavefronts an item, 8 x 64 float32 unless said otherwise, us:
//   127 items (L = 64)                  9.4 / 13.7 / 7.2  -> 4.7 / 6.4 / 4.2   -> 4.8 / 5.6 / 4.2;   SpMM 7.5 -> 4.0 -> 3.8
//   539 (L = 256, k = 16)              11.1 / 16.6 / 14.4 -> 9.2 / 11.7 / 11.6 -> 8.2 / 9.4 / 10.8;  bfloat16 12.2 / 16.9 / 15.5 -> 6.0 / 7.3 / 7.4 -> 5.6 / 6.6 / 7.4
//   816 (L = 400)                      11.4 / 16.6 / 13.8 -> 7.9 / 10.0 / 11.0 -> 9.0 / 10.4 / 10.5; SpMM 10.8 -> 6.7 -> 6.7
//   1434 (L = 700, k = 1)              15.7 / 21.2 / 15.0 -> 10.1 / 12.0 / 12.2 -> 11.3 / 12.8 / 12.6; SpMM 11.6 -> 7.9 -> 7.1
//   2050 (L = 1000, k = 1, no groups)  16.8 / 22.2 / 17.9 -> 11.0 / 14.0 / 13.6 -> 14.1 / 17.0 / 15.4; SpMM 11.6 -> 8.4 -> 8.2
// Larger launches fill the GPU with a wavefront an item.  Rows of 1024 columns take twice the registers and the LDS: eight
// wavefronts an item of them are one round of the chip up to 256 items, beyond it four are faster.  16 x 64:
//   268 (L = 130, k = 4)               16.3 / 22.7 / 16.7 -> 7.9 / 10.4 / 9.3   -> 8.2 / 10.2 / 9.4;   bfloat16 16.4 / 21.3 / 19.6 -> 7.6 / 9.6 / 8.7 -> 8.3 / 8.7 / 11.4
//   324 (L = 160, k = 4)               15.7 / 22.1 / 18.1 -> 8.5 / 10.2 / 13.1  -> 10.2 / 12.0 / 12.6; bfloat16 16.0 / 20.7 / 19.8 -> 7.6 / 9.6 / 11.5 -> 10.5 / 10.8 / 12.2
//   585 (L = 256, k = 16, both ways)   18.7 / 26.8 / 23.4 -> 18.6 / 21.2 / 19.4 -> 22.3 / 24.3 / 21.2
// A float32 forward of 512 columns or more that already has a wavefront for each of the 1024 SIMDs and 25 edges or more an
// item waits for the rate of its loads, not for one item: one -> four, 8 x 64 and 16 x 64, 983 items of 25 790 edges 11.7 -> 12.4 and 19.1 ->
// 21.0; 957 of 32 613 12.0 -> 12.2 and 19.7 -> 20.4; (1018 of 23 540 11.3 -> 11.2 and 18.2 -> 18.7; 756 items 11.2 -> 10.4 and 18.6 -> 17.1).
inline int row_parts(const bpt_plan *P, int columns, bool forward_f32 = false) {
    if (P->n_items <= (columns > 512 ? 288 : 640)) return 8;
    if (forward_f32 && columns >= 512 && P->n_items > 800 && P->n_items <= 1024 && P->n_edges >= 25000) return 1;
    return P->n_items <= 2048 ? 4 : 1;
}
template <typename T, int H, int D>
int run_sddmm_fast(const bpt_plan *P, const void *A, const void *B, void *y, hipStream_t s) {
    if (P->n_items == 0) return BPT_OK;
    hipLaunchKernelGGL((k_sddmm_fast<T, H, D, FAST_BATCH>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)A, (const T *)B, (T *)y);
    return launch_status();
}

template <typename T, typename WT, int H, int D, int NOUT>
int run_spmm_fast(const bpt_plan *P, const void *W0, const void *X0, void *Y0, const void *W1, const void *X1, void *Y1,
                  float *ws, hipStream_t s) {
    if (P->n_items == 0) return BPT_OK;
    float *ws1 = ws ? ws + (size_t)P->n_slots * H * D : nullptr;
    {
        ProfScope prof(NOUT == 2 ? BPT_KERNEL_ATTN_BWD_SRC : -1, s);
#define LAUNCH_SPMM(NW)                                                                                                                  \
    hipLaunchKernelGGL((k_spmm_fast<T, WT, H, D, FAST_BATCH, NOUT, 0, NW>), dim3(NW == 1 ? grid_for(P) : (int)P->n_items),                    \
                       dim3(NW == 1 ? BLOCK : NW * WAVE), 0, s, *P, (const WT *)W0, (const T *)X0, (T *)Y0, (const WT *)W1, (const T *)X1, \
                       (T *)Y1, ws, ws1)
        switch (row_parts(P, H * D)) {
        case 8: LAUNCH_SPMM(8); break;
        case 4: LAUNCH_SPMM(4); break;
        default: LAUNCH_SPMM(1); break;
        }
#undef LAUNCH_SPMM
    }
    int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0) return st;
    hipLaunchKernelGGL((k_combine_sum_v4<T>), dim3((int)P->n_heavy, H * D / (4 * WAVE), NOUT), dim3(BLOCK), 0, s, P->heavy, (const float *)ws,
                       (T *)Y0, (T *)Y1, H * D, (size_t)P->n_slots * H * D);
    return launch_status();
}

// score term of the relative positions: bias[eid[p], head] = A[row, head, :] . table[idx[p], :], float32
bool spmm_grp_ok(const bpt_plan *P, int h, int d, int dtype);
template <typename T, int H, int D> constexpr int head_slices();
inline int group_grid(const bpt_plan *P);

// shapes of the matrix-core kernel of the rel_pos term and of its gradient kernel
inline bool rel_rows_shape(int h, int d, int dtype) {
    return !g_force_generic.load(std::memory_order_relaxed) && d == 64 && (h == 4 || h == 8 || h == 16) && (dtype == BPT_F32 || dtype == BPT_BF16);
}

constexpr int REL_MAX_PARTS = 512;        // partial tables of the gradient kernel: two workgroups per compute unit
constexpr int REL_TILES_WAVES = 24;       // wavefronts a compute unit needs to hide the score kernel's round trips, and where several tiles share a workgroup the most of them

// LDS of k_rel_bias_bwd with nw tables of sums of cs wavefronts each: the sums, the table rows, the wavefronts' staged ds values and types
inline size_t rel_bwd_lds(int nw, int cs, int64_t n_used, int h) { return ((size_t)(nw + 1) * n_used * 64 + (size_t)nw * cs * REL_BWD_STAGE(h)) * 4; }
// How k_rel_bias_bwd is launched for n_used types: a workgroup of nw (4, 2 or 1) tables of sums, cs wavefronts (1 or 2) sharing the columns of each.
struct RelBwdShape {
    int nw, cs;
};
// One wavefront a table where that puts eight on a compute unit (workgroups that fit its 160 KB of LDS x wavefronts each; more tables per
// workgroup on a tie: fewer partial tables), which it does up to 59 types with 4 heads, 56 with 8 and 49 with 16; else the shape with most of
// them.  Two wavefronts a table read and stage an item's ds and types twice.  Kernel alone, one against two: where LDS holds eight, 55 types (8
// heads, L = 8192, k = 4) 41.4 us against 52.0, 33 (8 heads bfloat16, L = 32768, k = 2) 116 against 126; where it holds two, 173 (8 heads, L = 8192,
// k = 8 both ways) 182 against 148, 134 (4 heads, L = 6215, k = 6 both ways) 101 against 79, 140 (16 heads, L = 4096, k = 16) 110 against 106.  Four a
// table: 77 in the fourth place and 138 in the last.
// A workgroup takes at most 144 KB (large_lds false: at most the 64 KB every kernel may take).  nw 0: no configuration fits.
inline RelBwdShape rel_bwd_shape(int64_t n_used, int h, bool large_lds = true) {
    const size_t cap = (large_lds ? 144 : 64) * 1024;
    RelBwdShape best{0, 0};
    int best_waves = 0;
    for (int cs = 1; cs <= 2; ++cs) {
        if (best_waves >= 8) break;
        for (int nw = 4; nw >= 1; nw >>= 1) {
            const size_t lds = rel_bwd_lds(nw, cs, n_used, h);
            if (lds > cap) continue;
            const int waves = nw * cs * (int)((160 * 1024) / lds);
            if (waves > best_waves) { best = RelBwdShape{nw, cs}; best_waves = waves; }
        }
    }
    return best;
}

// a kernel may take more than 64 KB of dynamic LDS only after it has been told so (once per kernel and device; kernels of
// one signature are different kernels, so what has been done is kept by kernel address)
inline int allow_large_lds_at(const void *kernel, size_t bytes) {
    static std::mutex lock;
    static std::vector<std::pair<const void *, int>> done;
    if (bytes <= 64 * 1024) return BPT_OK;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return BPT_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> hold(lock);
    for (const auto &x : done)
        if (x.first == kernel && x.second == dev) return BPT_OK;
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return BPT_ERR_UNSUPPORTED;          // (the caller then takes a configuration inside 64 KB)
    }
    done.emplace_back(kernel, dev);
    return BPT_OK;
}
template <typename K>
int allow_large_lds(K kernel, size_t bytes) { return allow_large_lds_at(reinterpret_cast<const void *>(kernel), bytes); }

template <typename T, int H, int NW, int CS>
int launch_rel_bias_bwd(const bpt_plan *P, const float *ds, const void *q, const void *table, const int32_t *used_types, int64_t n_used,
                        void *dq, float *ws_dq, float *part, int n_parts, hipStream_t s) {
    const size_t lds = rel_bwd_lds(NW, CS, n_used, H);
    const int st = allow_large_lds(k_rel_bias_bwd<T, H, NW, CS>, lds);
    if (st != BPT_OK) return st;
    hipLaunchKernelGGL((k_rel_bias_bwd<T, H, NW, CS>), dim3(n_parts), dim3(NW * CS * WAVE), lds, s, *P, ds, (const T *)q, (const T *)table, used_types,
                       (int)n_used, (T *)dq, ws_dq, part);
    return launch_status();
}

// f(NW, CS as compile-time numbers)
template <typename F> int rel_bwd_pick(RelBwdShape x, F &&f) {
    auto cs = [&](auto NW) -> int {
        return x.cs == 1 ? f(NW, std::integral_constant<int, 1>{}) : f(NW, std::integral_constant<int, 2>{});
    };
    return x.nw == 4 ? cs(std::integral_constant<int, 4>{}) : x.nw == 2 ? cs(std::integral_constant<int, 2>{}) : cs(std::integral_constant<int, 1>{});
}

template <typename T, int H>
int run_rel_bias_bwd(const bpt_plan *P, const float *ds, const void *q, const void *table, const int32_t *used, const int32_t *used_types,
                     int64_t n_types, int64_t n_used, void *dq, void *dtable, float *ws, hipStream_t s) {
    float *ws_dq = ws, *part = ws + (size_t)P->n_slots * H * 64;       // partial rows of dq of the split rows, then the partial tables
    int n_parts = 0;
    auto launch = [&](RelBwdShape x) {
        const int64_t fit = 256 * std::min<int64_t>(2, (160 * 1024) / (int64_t)rel_bwd_lds(x.nw, x.cs, n_used, H));
        n_parts = (int)std::min<int64_t>(std::min<int64_t>(REL_MAX_PARTS, fit), std::max<int64_t>(1, (P->n_items + x.nw - 1) / x.nw));      // (an item a table of sums at the least)
        return rel_bwd_pick(x, [&](auto NW, auto CS) {
            return launch_rel_bias_bwd<T, H, decltype(NW)::value, decltype(CS)::value>(P, ds, q, table, used_types, n_used, dq, ws_dq, part, n_parts, s);
        });
    };
    if (P->n_edges > 0) {
        const RelBwdShape x = rel_bwd_shape(n_used, H);
        int st = launch(x);
        if (st == BPT_ERR_UNSUPPORTED && rel_bwd_lds(x.nw, x.cs, n_used, H) > 64 * 1024) {      // more than 64 KB of LDS refused by the runtime
            const RelBwdShape small = rel_bwd_shape(n_used, H, false);
            if (small.nw == 0) return BPT_ERR_UNSUPPORTED;
            st = launch(small);
        }
        if (st != BPT_OK) return st;
    }
    // (without edges there are no partial tables and no partial rows: every row of dtable becomes zero)
    const bool edges = P->n_edges > 0;
    const int n_split = edges ? (int)P->n_heavy : 0;
    hipLaunchKernelGGL((k_rel_finish<T>), dim3((unsigned)(n_types + (int64_t)n_split * (H * 64 / 256))), dim3(BLOCK), 0, s, part, used,
                       edges ? n_parts : 0, (int)n_types, (T *)dtable, P->heavy, ws_dq, (T *)dq, H * 64);
    return launch_status();
}

// whether run_rel_bias_bwd has a configuration that this device accepts for n_used types (nothing is launched)
template <typename T, int H>
int rel_bias_bwd_config(int64_t n_used) {
    const RelBwdShape x = rel_bwd_shape(n_used, H);
    if (x.nw == 0) return BPT_ERR_UNSUPPORTED;
    const size_t lds = rel_bwd_lds(x.nw, x.cs, n_used, H);
    const int st = rel_bwd_pick(x, [&](auto NW, auto CS) { return allow_large_lds(k_rel_bias_bwd<T, H, decltype(NW)::value, decltype(CS)::value>, lds); });
    if (st == BPT_OK) return BPT_OK;
    return rel_bwd_shape(n_used, H, false).nw != 0 ? BPT_OK : BPT_ERR_UNSUPPORTED;      // inside the 64 KB every kernel may take
}

// the score term with the table rows in LDS: plan indices are type numbers
template <typename T, int H>
int run_rel_bias_rows(const bpt_plan *P, const void *q, const void *table, const int32_t *used_types, int64_t n_used, float *bias, hipStream_t s) {
    if (P->n_items == 0) return BPT_OK;
    const int64_t waves = (P->n_items + REL_FWD_ITEMS - 1) / REL_FWD_ITEMS;
    hipLaunchKernelGGL((k_rel_bias_rows<T, H>), dim3((unsigned)((waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK)), dim3(BLOCK),
                       (size_t)n_used * REL_LDS_PITCH * 4, s, *P, (const T *)q, (const T *)table, used_types, (int)n_used, bias);
    return launch_status();
}

// the score term over the attention kernels' tile plan, in that plan's pair order
template <typename T> size_t rel_tiles_lds(int hw, int64_t n_used) {      // the table rows, and QT of every wavefront
    return (size_t)n_used * RelTile<T>::PITCH + (size_t)hw * (size_t)((n_used + 15) & ~(int64_t)15) * TILE_R * 4;
}
template <typename T, int H, int HW>
int launch_rel_bias_tiles(const bpt_plan *P, const void *q, const void *table, const int32_t *used_types, int64_t n_used, const int32_t *pair_tm,
                          float *bias, hipStream_t s) {
    const size_t lds = rel_tiles_lds<T>(HW, n_used);
    const int resident = 256 * std::min(REL_TILES_WAVES / HW, (int)((160 * 1024) / lds)), tiles = group_grid(P) * (H / HW);   // (resident: what the chip holds)
    auto launch = [&](auto kernel, int grid) -> int {
        const int st = allow_large_lds(kernel, lds);
        if (st != BPT_OK) return st;
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(HW * WAVE), lds, s, *P, (const T *)q, (const T *)table, used_types, (int)n_used, pair_tm, bias);
        return launch_status();
    };
    return tiles <= resident || (int)((160 * 1024) / lds) * HW >= REL_TILES_WAVES ? launch(k_rel_bias_tiles<T, H, HW, true>, tiles) : launch(k_rel_bias_tiles<T, H, HW, false>, resident);
}
template <typename T, int H>
int run_rel_bias_tiles(const bpt_plan *P, const void *q, const void *table, const int32_t *used_types, int64_t n_used, const int32_t *pair_tm,
                       float *bias, hipStream_t s) {
    // eight heads share the table rows where that puts no fewer wavefronts on a compute unit
    if constexpr (H >= 8) {
        const size_t l8 = rel_tiles_lds<T>(8, n_used), l4 = rel_tiles_lds<T>(4, n_used);
        if (l8 <= 160 * 1024 && 2 * ((160 * 1024) / l8) >= (160 * 1024) / l4) {
            const int st = launch_rel_bias_tiles<T, H, 8>(P, q, table, used_types, n_used, pair_tm, bias, s);
            if (st != BPT_ERR_UNSUPPORTED) return st;             // (more than 64 KB of LDS refused by the runtime)
        }
    }
    return launch_rel_bias_tiles<T, H, 4>(P, q, table, used_types, n_used, pair_tm, bias, s);
}

template <typename T, int H, int D>
int run_rel_bias(const bpt_plan *P, const void *A, const void *table, float *bias, hipStream_t s) {
    if (P->n_items == 0) return BPT_OK;
    if (spmm_grp_ok(P, H, D, sizeof(T) == 2 ? BPT_BF16 : BPT_F32)) {      // row groups: one load of a table row per group entry
        constexpr int HS = head_slices<T, H, D>();
        if (P->grp_R == 8)
            hipLaunchKernelGGL((k_sddmm_grp<T, H, D, 8, HS, true, float>), dim3(group_grid(P) * HS), dim3(WAVE), 0, s, *P, (const T *)A,
                               (const T *)table, bias);
        else
            hipLaunchKernelGGL((k_sddmm_grp<T, H, D, 4, HS, true, float>), dim3(group_grid(P) * HS), dim3(WAVE), 0, s, *P, (const T *)A,
                               (const T *)table, bias);
        return launch_status();
    }
    hipLaunchKernelGGL((k_sddmm_fast<T, H, D, FAST_BATCH, 2, float>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)A, (const T *)table,
                       bias);
    return launch_status();
}

// node_mul_edge with the specialised kernels: y = A . B[e] (forward), dA = sum dy * B[e], dB[e] = sum_h dy * A
template <typename T, int H, int D>
int run_nme_fwd_fast(const bpt_plan *P, const void *A, const void *B, void *y, hipStream_t s) {
    if (P->n_items == 0) return BPT_OK;
    hipLaunchKernelGGL((k_sddmm_fast<T, H, D, FAST_BATCH, 1>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)A, (const T *)B, (T *)y);
    return launch_status();
}

template <typename T, int H, int D>
int run_nme_bwd_fast(const bpt_plan *P, const void *A, const void *B, const void *dy, void *dA, void *dB, float *ws, hipStream_t s) {
    if (P->n_items == 0) return BPT_OK;
    hipLaunchKernelGGL((k_spmm_fast<T, T, H, D, FAST_BATCH, 1, 1>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)dy, (const T *)B,
                       (T *)dA, (const T *)nullptr, (const T *)nullptr, (T *)nullptr, ws, (float *)nullptr);
    int st = launch_status();
    if (st != BPT_OK) return st;
    if (P->n_heavy > 0) {
        hipLaunchKernelGGL((k_combine_sum_v4<T>), dim3((int)P->n_heavy, H * D / (4 * WAVE), 1), dim3(BLOCK), 0, s, P->heavy, (const float *)ws,
                           (T *)dA, (T *)nullptr, H * D, (size_t)0);
        st = launch_status();
        if (st != BPT_OK) return st;
    }
    hipLaunchKernelGGL((k_nme_dB_fast<T, H, D, FAST_BATCH>), dim3(grid_for(P)), dim3(BLOCK), 0, s, *P, (const T *)A, (const T *)dy, (T *)dB);
    return launch_status();
}

int nme_fwd_fast(const bpt_plan *P, const void *A, const void *B, void *y, int h, int d, int dtype, hipStream_t s) {
#define X(HH, DD) if (h == HH && d == DD) return run_nme_fwd_fast<T, HH, DD>(P, A, B, y, s);
    if (dtype == BPT_F32) { using T = float; BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { using T = bf16_t; BPT_FAST_SHAPES_BF16(X) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int nme_bwd_fast(const bpt_plan *P, const void *A, const void *B, const void *dy, void *dA, void *dB, void *ws, int h, int d, int dtype,
                 hipStream_t s) {
#define X(HH, DD) if (h == HH && d == DD) return run_nme_bwd_fast<T, HH, DD>(P, A, B, dy, dA, dB, (float *)ws, s);
    if (dtype == BPT_F32) { using T = float; BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { using T = bf16_t; BPT_FAST_SHAPES_BF16(X) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int sddmm_fast(const bpt_plan *P, const void *A, const void *B, void *y, int h, int d, int dtype, hipStream_t s) {
#define X(HH, DD) if (h == HH && d == DD) return run_sddmm_fast<T, HH, DD>(P, A, B, y, s);
    if (dtype == BPT_F32) { using T = float; BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { using T = bf16_t; BPT_FAST_SHAPES_BF16(X) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int spmm_fast(const bpt_plan *P, const void *W, const void *Xp, void *Y, void *ws, int h, int d, int dtype, hipStream_t s) {
#define X(HH, DD) if (h == HH && d == DD) return run_spmm_fast<T, T, HH, DD, 1>(P, W, Xp, Y, nullptr, nullptr, nullptr, (float *)ws, s);
    if (dtype == BPT_F32) { using T = float; BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { using T = bf16_t; BPT_FAST_SHAPES_BF16(X) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

// SDDMM / SpMM with automatic family choice
bool spmm_grp_ok(const bpt_plan *P, int h, int d, int dtype);
int sddmm_grp(const bpt_plan *P, const void *A, const void *B, void *y, int h, int d, int dtype, hipStream_t s);
bool product_tiles_ok(const bpt_plan *P, int h, int d, int dtype);
int sddmm_tile(const bpt_plan *P, const void *A, const void *B, void *y, int h, int d, hipStream_t s);
int spmm_tile(const bpt_plan *P, const void *W, const void *X, void *Y, void *ws, int h, int d, hipStream_t s, bool merge = true);
int sddmm(const bpt_plan *P, const void *A, const void *B, void *y, int h, int d, int dtype, hipStream_t s) {
    if (product_tiles_ok(P, h, d, dtype)) return sddmm_tile(P, A, B, y, h, d, s);
    if (fast_shape(h, d, dtype) && aligned16(A) && aligned16(B)) {
        if (spmm_grp_ok(P, h, d, dtype)) return sddmm_grp(P, A, B, y, h, d, dtype, s);
        return sddmm_fast(P, A, B, y, h, d, dtype, s);
    }
    return sddmm_generic(P, A, B, y, h, d, dtype, s);
}
int spmm_grp(const bpt_plan *P, const void *W, const void *X, void *Y, void *ws, int h, int d, int dtype, hipStream_t s, int accumulate = 0);
int spmm(const bpt_plan *P, const void *W, const void *X, void *Y, void *ws, int h, int d, int dtype, hipStream_t s) {
    if (product_tiles_ok(P, h, d, dtype) && aligned16(ws)) return spmm_tile(P, W, X, Y, ws, h, d, s);
    if (fast_shape(h, d, dtype) && aligned16(X) && aligned16(Y) && aligned16(ws)) {
        // a plan that carries row groups and their edge ids: one row load per entry instead of one per edge
        if (spmm_grp_ok(P, h, d, dtype)) return spmm_grp(P, W, X, Y, ws, h, d, dtype, s);
        return spmm_fast(P, W, X, Y, ws, h, d, dtype, s);
    }
    return spmm_generic(P, W, X, Y, ws, h, d, dtype, s);
}

inline int64_t round16(int64_t b) { return (b + 15) & ~(int64_t)15; }
inline int product_tile_heads(int h) { return (h + 3) & ~3; }        // heads of a partial row of the separate operators on tiles, 64 columns each

// dropout of the fused path: threshold on the 32-bit hash (0 = off), seed, 1 / (1 - p)
struct Dropout {
    uint32_t thr, seed;
    float inv;
};
inline Dropout make_dropout(float p, uint64_t seed) {
    if (!(p > 0.f)) return Dropout{0u, 0u, 1.f};
    const double t = (double)p * 4294967296.0;
    return Dropout{(uint32_t)(t >= 4294967295.0 ? 4294967295.0 : (t < 1.0 ? 1.0 : t)), (uint32_t)(seed ^ (seed >> 32)), 1.f / (1.f - p)};
}

// The row-group kernels address node rows and the per-pair scratch with 32-bit byte offsets.
inline bool fits32(int64_t n, int64_t unit) { return n >= 0 && n <= (int64_t)0xffffffffu / unit; }

inline int group_grid(const bpt_plan *P) { return (int)(8 * P->grp_max_chunk); }

// The row-group kernels split a group's heads over wavefronts so that one wavefront handles at most 512 columns of
// every row (8 registers per lane and row: the members' state has to fit the register file).  Slices of 256
// float32 columns were also measured: faster on small graphs, slower at the benchmark sizes.
template <typename T, int H, int D> constexpr int head_slices() {
    constexpr int CS = 512, C = H * D;
    return (C > CS && C % CS == 0 && H % (C / CS) == 0) ? C / CS : 1;
}

// The matrix-core forward gives a wavefront at most 512 columns of every row.  0 slices = shape not covered.
template <typename T, int H, int D> constexpr int mfma_slices() {
    constexpr int CS = 512, C = H * D;
    if (C <= CS) return 1;
    return (C % CS == 0 && H % (C / CS) == 0) ? C / CS : 0;
}
template <typename T, int H, int D> constexpr bool mfma_ok() {
    constexpr int HS = mfma_slices<T, H, D>();
    if (HS == 0) return false;
    constexpr int HL = H / HS, CS = HL * D, VE = 16 / (int)sizeof(T);
    if (64 % HL != 0 || CS % 64 != 0) return false;
    constexpr int LPH = 64 / HL, EPL = CS / 64;
    return (LPH == 4 || LPH == 8 || LPH == 16) && EPL % VE == 0 && EPL <= 8;
}

// rows per group the row-group kernels exist for
inline bool group_rows_ok(int64_t R) { return R == 4 || R == 8; }

inline bool has_groups(const bpt_plan *P, int h, int d, size_t elem) {
    return P->n_groups > 0 && group_rows_ok(P->grp_R) && P->grp_members && P->grp_ptr && P->grp_entries && P->grp_chunks &&
           P->grp_max_chunk > 0 && 8 * P->grp_max_chunk >= P->n_groups && P->n_grp_entries >= 0 &&
           fits32(std::max(P->n_rows, P->n_index_nodes), (int64_t)h * d * (int64_t)elem) &&
           fits32((P->n_grp_entries + GRP_PAD_ENTRIES) * P->grp_R, (int64_t)h * 8);
}

// groups of 16 rows for the dense-tile kernels (one wavefront per head: h * 64 threads per workgroup)
inline bool has_tiles(const bpt_plan *P, int h, int d, size_t elem) {
    return P->n_groups > 0 && P->grp_R == TILE_R && P->grp_members && P->grp_ptr && P->grp_entries && P->grp_chunks &&
           P->grp_max_chunk > 0 && 8 * P->grp_max_chunk >= P->n_groups && P->n_grp_entries >= 0 && d == 64 && h <= 16 && (elem == 4 || elem == 2) &&
           fits32(std::max(P->n_rows, P->n_index_nodes), (int64_t)h * d * (int64_t)elem);
}

// Over how many wavefronts (1, 2 or 4) of a workgroup the blocks of a tile are spread.  A launch has 1024 SIMDs to fill, and one
// that does not lasts as long as its longest chain of blocks: each part's chain is a half or a quarter as long.  What
// the parts cost is the tile's header, read by each of them, and the meeting in LDS, so with more wavefronts than fill the chip
// a part has to keep enough blocks.  float32, 8 heads, forward / destination side / source side, one part -> two -> four:
//   584 wavefronts of 4 to 9 blocks (L = 512)           10.3 / 13.8 / 16.4 -> 8.0 / 10.8 / 10.9 -> 8.0 / 9.6 / 8.6 us
//   1032 of 9 (window of 128, L = 2048)                 20.5 / 29.8 / 17.0 -> 15.7 / 21.3 / 13.7 -> 14.5 / 19.4 / 13.8
//   1448 of 3 (L = 1400, k = 4)                         11.9 / 16.3 / 11.3 -> 11.4 / 14.3 / 10.2 -> 12.8 / 16.6 / 11.7
//   2056 of 9 (window of 128, L = 4096)                 25.2 / 38.6 / 25.1 -> 20.8 / 30.7 / 21.3 -> 22.9 / 32.5 / 22.3
//   2096 of 3 (16 heads, L = 1024, k = 4)               12.8 / 19.2 / 13.9 -> 13.4 / 19.6 / 15.0 -> 14.8 / 20.6 / 14.8
//   2072 of 4 / 2168 of 5 (L = 2048, k = 8)             16.8 / 26.1 / 19.0 -> 14.4 / 21.4 / 18.2 -> 15.8 / 22.4 / 17.5
//   4112 of 9 (window of 128, L = 8192)                 33.3 / 56.6 / 48.4 -> 32.3 / 53.1 / 35.5 -> 37.0 / 58.3 / 38.6
//   4160 of 5 / 4448 of 8 (L = 4096, k = 4, both ways)  24.0 / 37.6 / 37.0 -> 24.4 / 39.4 / 35.3 -> 27.8 / 42.4 / 37.1
//   8080 of 16 / 8072 of 9 (window of 256, L = 8192)    91.0 / 142 / 93.8  -> 93.2 / 140 / 85.0  -> 101 / 149 / 88.6
//   8256 of 5 (window of 64, L = 16384)                 46.5 / 72.1 / 51.4 -> 49.6 / 72.2 / 50.1 -> 57.4 / 84.7 / 61.6
// bfloat16, whose blocks are shorter against their headers:
//   552 of 5 (L = 512)      5.4 / 6.5 / 9.6 -> 5.1 / 5.7 / 7.3 -> 5.1 / 5.9 / 6.6;    1048 of 3    5.3 / 6.3 / 6.8 -> 5.7 / 6.4 / 7.2 -> 6.4 / 7.4 / 8.6
//   1032 of 9               9.6 / 11.8 / 9.0 -> 7.7 / 8.8 / 9.5 -> 7.6 / 8.4 / 10.2;  2056 of 9   10.6 / 14.1 / 11.5 -> 10.4 / 12.8 / 12.2 -> 12.0 / 14.2 / 14.4
//   2072 of 4               8.2 / 10.0 / 10.4 -> 7.9 / 10.2 / 11.9 -> 9.3 / 12.7 / 14.2;  4112 of 9   15.0 / 18.4 / 19.0 -> 16.6 / 20.0 / 21.9 -> 19.3 / 23.5 / 27.0
//   (two parts cost the last launches that take them up to 5 %: 1048 of 3)
// The same line holds with dropout, the score term and narrow heads (one head a workgroup in parts, two otherwise); float32:
//   L = 512, dropout                10.9 / 13.6 / 15.6 -> 7.9 / 10.2 / 10.4  -> 7.8 / 10.3 / 9.1;   term and dropout 11.8 / 16.5 / 16.2 -> 8.6 / 12.3 / 10.5 -> 8.0 / 11.9 / 8.2
//   window 128, L = 4096, dropout   27.9 / 39.4 / 24.5 -> 22.3 / 35.6 / 20.9 -> 25.0 / 37.2 / 22.6; 6 x 50 with dropout 34.8 / 37.8 / 21.7 -> 26.6 / 28.0 / 20.8 -> 26.8 / 30.9 / 19.9
//   L = 4096, k = 32, dropout       39.5 / 56.2 / 48.2 -> 34.8 / 54.5 / 43.6 -> 40.1 / 61.7 / 46.8; term and dropout 43.0 / 64.8 / 49.2 -> 37.5 / 63.9 / 45.1 -> 42.0 / 72.0 / 48.6
//                                   6 x 50 with dropout 55.9 / 59.4 / 42.7 -> 33.5 / 44.1 / 34.5 -> 38.4 / 49.3 / 37.4
//   L = 8192, k = 4 (one part)      35.8 / 55.6 / 38.3 -> 38.9 / 62.7 / 40.6;  6 x 50 with dropout 44.3 / 46.2 / 36.2 -> 47.0 / 50.1 / 38.4
// bfloat16, dropout: L = 512 6.3 / 7.0 / 12.8 -> 5.5 / 5.9 / 10.7 -> 5.5 / 6.2 / 7.8; window 128, L = 4096 13.2 / 14.1 / 16.6 -> 11.7 / 12.6 / 16.7 -> 13.8 /
// 15.4 / 18.8; 6 x 50 there 19.2 / 21.3 / 13.0 -> 14.4 / 17.3 / 12.8 -> 15.3 / 18.9 / 12.6.  Of 290 kernels of a hundred graphs drawn at random over all
// of these the rule slowed one by more than 1 % against one part (a window of 52, forward 16.9 -> 17.8).
// Two parts of launches that fill the chip about twice (6500 to 8192 wavefronts) pay on the source side (window 256, above) and with dropout
// (forward there 108.2 -> 106.8), not for a float32 forward without: L = 7000, k = 32 51.7 -> 53.9, L = 6000, k = 64 63.5 -> 66.0, window 128, L =
// 16000 61.1 -> 63.1, window 256 90.8 -> 92.4 (plain_forward; below, 5600 to 6300 wavefronts 42.7 -> 42.9, 46.2 -> 45.7, 48.4 -> 47.0).
inline int tile_parts(const bpt_plan *P, int heads, size_t elem, bool plain_forward = false) {
    const int64_t wavefronts = P->n_groups * heads, blocks = P->n_grp_entries / TILE_R;
    const int64_t most = plain_forward ? 13000 : 16384;
    auto pays = [&](int parts) {
        const int64_t w = wavefronts * parts, each = blocks / std::max<int64_t>(P->n_groups * parts, 1);      // (blocks of a part, rounded down)
        if (elem == 2) return w <= 2400 || (parts == 2 && w <= 4608 && each >= 4);
        return w <= 3072 || (w <= 6144 && each >= 2) || (parts == 2 && w <= most && each >= 4);
    };
    return pays(4) ? 4 : pays(2) ? 2 : 1;
}

// a tile in parts: one head a workgroup, so that no wavefront of it lies past the last head
inline Narrow narrow_parts(Narrow nw, int parts) {
    if (parts > 1) nw.slices = nw.heads;
    return nw;
}

// The separate operators on tiles: float32, groups of 16 rows with their edge ids.  Heads of 64 columns, 4, 8 or 16 of them, whose rows
// lie on 16 bytes, take the kernels of those shapes, all others of 4 to 64 columns the narrow ones (rows on 4 bytes).
bool product_tiles_ok(const bpt_plan *P, int h, int d, int dtype) {
    return dtype == BPT_F32 && !g_force_generic.load(std::memory_order_relaxed) && P->n_edges > 0 && P->grp_eids && d >= 4 && d <= 64 && h <= 16 &&
           P->n_groups > 0 && P->grp_R == TILE_R && P->grp_members && P->grp_ptr && P->grp_entries && P->grp_chunks && P->grp_max_chunk > 0 &&
           8 * P->grp_max_chunk >= P->n_groups && P->n_grp_entries >= 0 && fits32(std::max(P->n_rows, P->n_index_nodes), (int64_t)h * d * 4) &&
           fits32(P->n_edges, h);
}
inline Narrow product_narrow(int h, int d) { return Narrow{d, h, product_tile_heads(h), (h + NARROW_HW - 1) / NARROW_HW}; }

// How many heads of a workgroup access an edge's record together where one wavefront walks a tile (1: each its own), for node tensors and an
// edge tensor that start on 16 bytes or not (two heads: the edge tensor on 8).
inline bool product_whole_heads(int h, int d, bool nodes16) { return d == 64 && nodes16 && (h == 4 || h == 8 || h == 16); }
inline int shared_heads(int h, int d, bool nodes16, bool edges16, bool edges8 = true) {
    if (product_whole_heads(h, d, nodes16)) return edges16 ? 4 : 1;
    return h % NARROW_HW == 0 && edges8 ? NARROW_HW : 1;
}

// Over how many wavefronts a tile and head of the separate operators is spread (shared: as shared_heads says).  Parts have blocks of their
// own, so in parts every head goes to the edge tensor by itself: what tile_parts measured on the attention kernels holds for heads that do
// so anyway.  Heads that share take one part where a launch has wavefronts enough without parts.  SDDMM + SpMM of one side, one part ->
// two -> four:
//   four together, 8 x 64: 4112 wavefronts of 9 blocks (window of 128, L = 8192)  49 -> 70 -> 71 us;   3976 of 16 (window of 256, L = 4096)  66 -> 90 -> 86;
//     8080 of 16  129 -> 172 -> 166;   4160 of 5 (L = 4096, k = 4, both ways)  32 -> 41 -> 44;   4448 of 8  46 -> 53 -> 56
//     below, by how unequal a graph's tiles are: 2056 of 9 (window of 128)  31 -> 38 -> 40, 3288 of 18 (L = 3000, k = 16, both ways)  96 -> 86 -> 79,
//     1576 of 15 (L = 1500)  81 -> 63 -> 43, 2352 of 21 (L = 2048, k = 32)  94 -> 81 -> 74
//   16 x 64, whose edges' records are half a line: 2064 of 9 (window of 128, L = 2048)  37 -> 47 -> 49;   4112 of 9  47 -> 80 -> 85;   2176 of 3 (L = 1024,
//     k = 4)  18 -> 20 -> 22;   3024 of 9 (L = 1500, k = 16, both ways)  49 -> 59 -> 60;   of more blocks 3152 of 15 there  92 -> 78 -> 76, 2368 of 17  71 -> 72 -> 77
//   two together: 4112 of 9 (8 x 40, window of 128)  52 -> 69 -> 70;   3420 of 10 (6 x 50, L = 4096, k = 32)  52 -> 62 -> 58;   3336 of 8 (6 x 50, L = 4096, k = 4,
//     both ways)  45 -> 43 -> 43;   3288 of 18  108 -> 87 -> 77;   2982 of 9 (window of 256)  49 -> 47 -> 45
//   each by itself: 5050 of 13 (5 x 30, window of 256; both sides)  173 -> 156 -> 156
// Of 304 pairs of launches (windows, BPT graphs one way and both, k up to 64) none is slower by it than by tile_parts and those from the line
// on up to 1.9 times as fast.
inline int product_parts(const bpt_plan *P, int heads, int shared) {
    const int64_t wavefronts = P->n_groups * heads;
    const bool half_lines = shared == 4 && heads == 16 && P->n_grp_entries < 12 * TILE_R * P->n_groups;
    if (shared > 1 && wavefronts >= (half_lines ? 2050 : 3400)) return 1;
    return tile_parts(P, heads, 4);
}

template <int H>
int run_spmm_tile(const bpt_plan *P, const float *W, const float *X, float *Y, float *ws, hipStream_t s, bool merge) {
    const int shared = aligned16(W) ? 4 : 1, parts = product_parts(P, H, shared);
#define LAUNCH(SH, SP) \
    hipLaunchKernelGGL((k_spmm_tile<H, 64, 4, SH, false, SP>), dim3(group_grid(P) * (H * SP / 4)), dim3(4 * WAVE), 0, s, *P, W, X, Y, ws, Narrow{})
    if (parts == 4) LAUNCH(false, 4);
    else if (parts == 2) LAUNCH(false, 2);
    else if (shared == 4) LAUNCH(true, 1);
    else LAUNCH(false, 1);
#undef LAUNCH
    const int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0 || !merge) return st;
    hipLaunchKernelGGL((k_combine_sum_v4<float>), dim3((int)P->n_heavy, H * 64 / (4 * WAVE), 1), dim3(BLOCK), 0, s, P->heavy, (const float *)ws, Y,
                       (float *)nullptr, H * 64, (size_t)0);
    return launch_status();
}
// merge false: the split rows' partial sums are left in ws
int spmm_tile(const bpt_plan *P, const void *W_, const void *X_, void *Y_, void *ws_, int h, int d, hipStream_t s, bool merge) {
    const float *W = (const float *)W_, *X = (const float *)X_;
    float *Y = (float *)Y_, *ws = (float *)ws_;
    const bool nodes16 = aligned16(X) && aligned16(Y);
    if (product_whole_heads(h, d, nodes16)) {
        if (h == 4) return run_spmm_tile<4>(P, W, X, Y, ws, s, merge);
        if (h == 8) return run_spmm_tile<8>(P, W, X, Y, ws, s, merge);
        if (h == 16) return run_spmm_tile<16>(P, W, X, Y, ws, s, merge);
    }
    const int shared = shared_heads(h, d, nodes16, aligned16(W), (reinterpret_cast<uintptr_t>(W) & 7u) == 0), parts = product_parts(P, h, shared);
    const Narrow nw = narrow_parts(product_narrow(h, d), parts);
#define LAUNCH(HW, SH, SP) \
    hipLaunchKernelGGL((k_spmm_tile<16, 64, HW, SH, true, SP>), dim3(group_grid(P) * nw.slices), dim3(HW * WAVE), 0, s, *P, W, X, Y, ws, nw)
    if (parts == 4) LAUNCH(4, false, 4);
    else if (parts == 2) LAUNCH(2, false, 2);
    else if (shared == NARROW_HW) LAUNCH(NARROW_HW, true, 1);
    else LAUNCH(NARROW_HW, false, 1);
#undef LAUNCH
    const int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0 || !merge) return st;
    hipLaunchKernelGGL((k_combine_sum3<float, true>), dim3((int)P->n_heavy, nw.h * 64 / (4 * WAVE), 1), dim3(BLOCK), 0, s, P->heavy, (int)P->n_heavy,
                       (const float *)ws, Y, (const int32_t *)nullptr, (const float *)nullptr, (float *)nullptr, (float *)nullptr, nw.h * 64, (size_t)0, nw);
    return launch_status();
}

// Ya = the sums over Pa's rows of W * Xa, Yb over Pb's of W * Xb: the split rows of both are added up by one launch (masked_mm's gradients at 8 heads,
// L = 8192, k = 4: two launches of 3.9 + 4.7 us -> one of 4.2, the pass through the separate operators 227.8 -> 225.1)
int spmm_tile_pair(const bpt_plan *Pa, const void *Xa, void *Ya, void *ws_a, const bpt_plan *Pb, const void *Xb, void *Yb, void *ws_b, const void *W, int h, int d,
                   hipStream_t s) {
    int st = spmm_tile(Pa, W, Xa, Ya, ws_a, h, d, s, false);
    if (st != BPT_OK) return st;
    st = spmm_tile(Pb, W, Xb, Yb, ws_b, h, d, s, false);
    const int n_a = (int)Pa->n_heavy, n_b = (int)Pb->n_heavy;
    if (st != BPT_OK || n_a + n_b == 0) return st;
    const Narrow nw = product_narrow(h, d);
    const bool whole = product_whole_heads(h, d, aligned16(Xa) && aligned16(Ya));
    const int C = (whole ? h : nw.h) * 64;
#define LAUNCH(NARROW, NW) \
    hipLaunchKernelGGL((k_combine_sum3<float, NARROW>), dim3(n_a + n_b, C / (4 * WAVE), 1), dim3(BLOCK), 0, s, Pa->heavy, n_a, (const float *)ws_a, (float *)Ya, \
                       Pb->heavy, (const float *)ws_b, (float *)Yb, (float *)nullptr, C, (size_t)0, NW)
    if (whole) LAUNCH(false, Narrow{});
    else LAUNCH(true, nw);
#undef LAUNCH
    return launch_status();
}

template <int H>
int run_sddmm_tile(const bpt_plan *P, const float *A, const float *B, float *y, hipStream_t s) {
    const int shared = aligned16(y) ? 4 : 1, parts = product_parts(P, H, shared);
#define LAUNCH(SH, SP) \
    hipLaunchKernelGGL((k_sddmm_tile<H, 64, 4, SH, false, SP>), dim3(group_grid(P) * (H * SP / 4)), dim3(4 * WAVE), 0, s, *P, A, B, y, Narrow{})
    if (parts == 4) LAUNCH(false, 4);
    else if (parts == 2) LAUNCH(false, 2);
    else if (shared == 4) LAUNCH(true, 1);
    else LAUNCH(false, 1);
#undef LAUNCH
    return launch_status();
}
int sddmm_tile(const bpt_plan *P, const void *A_, const void *B_, void *y_, int h, int d, hipStream_t s) {
    const float *A = (const float *)A_, *B = (const float *)B_;
    float *y = (float *)y_;
    const bool nodes16 = aligned16(A) && aligned16(B);
    if (product_whole_heads(h, d, nodes16)) {
        if (h == 4) return run_sddmm_tile<4>(P, A, B, y, s);
        if (h == 8) return run_sddmm_tile<8>(P, A, B, y, s);
        if (h == 16) return run_sddmm_tile<16>(P, A, B, y, s);
    }
    const int shared = shared_heads(h, d, nodes16, aligned16(y), (reinterpret_cast<uintptr_t>(y) & 7u) == 0), parts = product_parts(P, h, shared);
    const Narrow nw = narrow_parts(product_narrow(h, d), parts);
#define LAUNCH(HW, SH, SP) \
    hipLaunchKernelGGL((k_sddmm_tile<16, 64, HW, SH, true, SP>), dim3(group_grid(P) * nw.slices), dim3(HW * WAVE), 0, s, *P, A, B, y, nw)
    if (parts == 4) LAUNCH(4, false, 4);
    else if (parts == 2) LAUNCH(2, false, 2);
    else if (shared == NARROW_HW) LAUNCH(NARROW_HW, true, 1);
    else LAUNCH(NARROW_HW, false, 1);
#undef LAUNCH
    return launch_status();
}

bool spmm_grp_ok(const bpt_plan *P, int h, int d, int dtype) {
    return has_groups(P, h, d, dtype == BPT_BF16 ? 2 : 4) && P->grp_eids && P->n_edges > 0;
}

template <typename T, int H, int D>
int run_spmm_grp(const bpt_plan *P, const void *W, const void *X, void *Y, float *ws, hipStream_t s, int accumulate = 0) {
    constexpr int HS = head_slices<T, H, D>();
#define LAUNCH_SPMM(RR)                                                                                                     \
    hipLaunchKernelGGL((k_spmm_grp<T, H, D, RR, HS>), dim3(group_grid(P) * HS), dim3(WAVE), 0, s, *P, (const T *)W, (const T *)X, \
                       (T *)Y, ws, accumulate)
    if (P->grp_R == 8) LAUNCH_SPMM(8);
    else LAUNCH_SPMM(4);
#undef LAUNCH_SPMM
    int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0) return st;
    hipLaunchKernelGGL((k_combine_sum_v4<T>), dim3((int)P->n_heavy, H * D / (4 * WAVE), 1), dim3(BLOCK), 0, s, P->heavy, (const float *)ws,
                       (T *)Y, (T *)nullptr, H * D, (size_t)0, accumulate);
    return launch_status();
}

template <typename T, int H, int D>
int run_sddmm_grp(const bpt_plan *P, const void *A, const void *B, void *y, hipStream_t s) {
    constexpr int HS = head_slices<T, H, D>();
    if (P->grp_R == 8) hipLaunchKernelGGL((k_sddmm_grp<T, H, D, 8, HS>), dim3(group_grid(P) * HS), dim3(WAVE), 0, s, *P, (const T *)A, (const T *)B, (T *)y);
    else hipLaunchKernelGGL((k_sddmm_grp<T, H, D, 4, HS>), dim3(group_grid(P) * HS), dim3(WAVE), 0, s, *P, (const T *)A, (const T *)B, (T *)y);
    return launch_status();
}

int sddmm_grp(const bpt_plan *P, const void *A, const void *B, void *y, int h, int d, int dtype, hipStream_t s) {
#define X(HH, DD) if (h == HH && d == DD) return run_sddmm_grp<T, HH, DD>(P, A, B, y, s);
    if (dtype == BPT_F32) { using T = float; BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { using T = bf16_t; BPT_FAST_SHAPES_BF16(X) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int spmm_grp(const bpt_plan *P, const void *W, const void *Xp, void *Y, void *ws, int h, int d, int dtype, hipStream_t s, int accumulate) {
#define X(HH, DD) if (h == HH && d == DD) return run_spmm_grp<T, HH, DD>(P, W, Xp, Y, (float *)ws, s, accumulate);
    if (dtype == BPT_F32) { using T = float; BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { using T = bf16_t; BPT_FAST_SHAPES_BF16(X) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

inline bool grouped_backward(const bpt_plan *Pin, const bpt_plan *Pout, int h, int d, size_t elem) {
    return has_groups(Pin, h, d, elem) && has_groups(Pout, h, d, elem) && Pin->grp_R == Pout->grp_R && Pin->grp_pairs;
}

// the tile kernels run the backward when both sides carry tiles and the source side the destination side's pair numbers
inline bool tiled_backward(const bpt_plan *Pin, const bpt_plan *Pout, int h, int d, size_t elem) {
    return has_tiles(Pin, h, d, elem) && has_tiles(Pout, h, d, elem) && Pout->grp_pairs;
}

// What the two backward kernels hand each other.  float2 (p, ds): one per (entry, member) of the source-side groups (plus the
// look-ahead padding) for the row-group kernels, one per edge for the per-row and the float32 tile kernels.  bfloat16 tiles: (p, ds)
// in four bytes per edge, or (lse, delta) of the rows where the source side forms the pairs again, which `plain` calls (64-column
// rows, no score term) always do if the plan has its edge ids: L = 32768, k = 8, 16 heads 8.4 MB, where the pairs would be 211.
inline int64_t pds_bytes(const bpt_plan *Pin, const bpt_plan *Pout, int h, int d, size_t elem, bool plain) {
    int64_t n = Pin->n_edges;
    if (Pout && elem == 2 && tiled_backward(Pin, Pout, h, d, elem)) {
        const int64_t rows = std::max(Pin->n_rows, Pout->n_index_nodes) * h * 8;
        return round16(plain && Pout->grp_eids ? rows : std::max(rows, n * h * 4));
    }
    if (Pout && grouped_backward(Pin, Pout, h, d, elem)) n = std::max(n, (Pout->n_grp_entries + GRP_PAD_ENTRIES) * Pout->grp_R);
    return 2 * round16(n * h * 4);
}

// Whether the source side of the bfloat16 tile kernels forms (p, ds) again instead of reading them back: with a score term
// it would have to look that up by the pair's position all the same, and the dropout decision needs the pair's edge id.
inline bool forms_pairs_again(const bpt_plan *Pout, const Dropout &drop, const float *bias) { return !bias && (drop.thr == 0 || Pout->grp_eids); }

// how the tile kernels find the score term: 0 none, 1 by edge id, 2 in the plan's own pair order, head-major
inline int tile_bias_mode(const bpt_plan *P, const float *bias) { return !bias ? 0 : P->bias_by_pair ? 2 : 1; }

template <typename T, int H, int D>
int run_attn_fwd(const bpt_plan *P, const void *q, const void *k, const void *v, void *o, float *lse, void *ws, float scale, Dropout drop,
                 const float *bias, hipStream_t s) {
    if (P->n_items == 0) return BPT_OK;
    float *ws_acc = (float *)ws;
    float *ws_ml = ws_acc ? ws_acc + (size_t)P->n_slots * H * D : nullptr;
    {
        ProfScope prof(BPT_KERNEL_ATTN_FWD, s);
        if constexpr (D == 64 && sizeof(T) == 4) {
            if (has_tiles(P, H, D, sizeof(T)) && ((drop.thr == 0 && !bias) || P->grp_eids)) {
                constexpr int HW = H >= 4 ? 4 : H;          // heads per workgroup
                const int parts = tile_parts(P, H, sizeof(T), drop.thr == 0 && !bias);
#define LAUNCH_FWD_TILE_PARTS(DR, BI, SP)                                                                                            \
    hipLaunchKernelGGL((k_attn_fwd_tile<T, H, D, HW, DR, BI, false, SP>), dim3(group_grid(P) * (H * SP / HW)), dim3(HW * WAVE), 0, s, *P, \
                       (const T *)q, (const T *)k, (const T *)v, (T *)o, lse, ws_acc, ws_ml, scale * LOG2E, drop.thr, drop.seed, drop.inv, bias, \
                       Narrow{}, Keep{})
#define LAUNCH_FWD_TILE(DR, BI)                                                                                                      \
    do {                                                                                                                             \
        if (parts == 4) LAUNCH_FWD_TILE_PARTS(DR, BI, 4);                                                                            \
        else if (parts == 2) LAUNCH_FWD_TILE_PARTS(DR, BI, 2);                                                                       \
        else LAUNCH_FWD_TILE_PARTS(DR, BI, 1);                                                                                       \
    } while (0)
                switch ((drop.thr != 0 ? 1 : 0) + 2 * tile_bias_mode(P, bias)) {
                case 0: LAUNCH_FWD_TILE(false, 0); break;
                case 1: LAUNCH_FWD_TILE(true, 0); break;
                case 2: LAUNCH_FWD_TILE(false, 1); break;
                case 3: LAUNCH_FWD_TILE(true, 1); break;
                case 4: LAUNCH_FWD_TILE(false, 2); break;
                default: LAUNCH_FWD_TILE(true, 2); break;
                }
#undef LAUNCH_FWD_TILE
#undef LAUNCH_FWD_TILE_PARTS
                goto launched;
            }
        }
        if constexpr (D == 64 && sizeof(T) == 2) {
            if (has_tiles(P, H, D, sizeof(T)) && ((drop.thr == 0 && !bias) || P->grp_eids)) {
                constexpr int HW = H >= 4 ? 4 : H;
                const int parts = tile_parts(P, H, sizeof(T));
#define LAUNCH_FWD_TILE_PARTS(DR, BI, SP)                                                                                                \
    hipLaunchKernelGGL((k_attn_fwd_rows_bf16<H, D, HW, TILE_BF16_WPE, DR, BI, SP>), dim3(group_grid(P) * (H * SP / HW)), \
                       dim3(HW * WAVE), 0, s, *P, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, (bf16_t *)o, lse, ws_acc, ws_ml, \
                       scale * LOG2E, drop.thr, drop.seed, drop.inv, bias)
#define LAUNCH_FWD_TILE(DR, BI)                                                                                                          \
    do {                                                                                                                                 \
        if (parts == 4) LAUNCH_FWD_TILE_PARTS(DR, BI, 4);                                                                                \
        else if (parts == 2) LAUNCH_FWD_TILE_PARTS(DR, BI, 2);                                                                           \
        else LAUNCH_FWD_TILE_PARTS(DR, BI, 1);                                                                                           \
    } while (0)
                switch ((drop.thr != 0 ? 1 : 0) + 2 * tile_bias_mode(P, bias)) {
                case 0: LAUNCH_FWD_TILE(false, 0); break;
                case 1: LAUNCH_FWD_TILE(true, 0); break;
                case 2: LAUNCH_FWD_TILE(false, 1); break;
                case 3: LAUNCH_FWD_TILE(true, 1); break;
                case 4: LAUNCH_FWD_TILE(false, 2); break;
                default: LAUNCH_FWD_TILE(true, 2); break;
                }
#undef LAUNCH_FWD_TILE
#undef LAUNCH_FWD_TILE_PARTS
                goto launched;
            }
        }
        if (has_groups(P, H, D, sizeof(T))) {
#define LAUNCH_FWD(RR, DR, BI)                                                                                                   \
    hipLaunchKernelGGL((k_attn_fwd_grp<T, H, D, RR, HS, DR, BI>), dim3(group_grid(P) * HS), dim3(WAVE), 0, s, *P, (const T *)q, \
                       (const T *)k, (const T *)v, (T *)o, lse, ws_acc, ws_ml, scale * LOG2E, drop.thr, drop.seed, drop.inv, bias)
#define LAUNCH_FWD_MFMA(DR, BI)                                                                                                      \
    hipLaunchKernelGGL((k_attn_fwd_mfma<T, H, D, HSM, DR, BI>), dim3(group_grid(P) * HSM), dim3(2 * WAVE), 0, s, *P, (const T *)q, \
                       (const T *)k, (const T *)v, (T *)o, lse, ws_acc, ws_ml, scale * LOG2E, drop.thr, drop.seed, drop.inv, bias)
            constexpr int HS = head_slices<T, H, D>();
            const int variant = (drop.thr != 0 ? 1 : 0) + (bias ? 2 : 0);
            if (P->grp_R == 8) {
                // every compile-time shape has the matrix-core form for groups of 8
                static_assert(mfma_ok<T, H, D>(), "groups of 8 rows need the matrix-core forward");
                constexpr int HSM = mfma_slices<T, H, D>();
                switch (variant) {
                case 0: LAUNCH_FWD_MFMA(false, false); break;
                case 1: LAUNCH_FWD_MFMA(true, false); break;
                case 2: LAUNCH_FWD_MFMA(false, true); break;
                default: LAUNCH_FWD_MFMA(true, true); break;
                }
            } else {
                switch (variant) {
                case 0: LAUNCH_FWD(4, false, false); break;
                case 1: LAUNCH_FWD(4, true, false); break;
                case 2: LAUNCH_FWD(4, false, true); break;
                default: LAUNCH_FWD(4, true, true); break;
                }
            }
#undef LAUNCH_FWD
#undef LAUNCH_FWD_MFMA
        } else {
#define LAUNCH_FWD_ROWS(NW)                                                                                                           \
    hipLaunchKernelGGL((k_attn_fwd<T, H, D, FAST_BATCH, NW>), dim3(NW == 1 ? grid_for(P) : (int)P->n_items), dim3(NW == 1 ? BLOCK : NW * WAVE), \
                       0, s, *P, (const T *)q, (const T *)k, (const T *)v, (T *)o, lse, ws_acc, ws_ml, scale * LOG2E)
            switch (row_parts(P, H * D, sizeof(T) == 4)) {
            case 8: LAUNCH_FWD_ROWS(8); break;
            case 4: LAUNCH_FWD_ROWS(4); break;
            default: LAUNCH_FWD_ROWS(1); break;
            }
#undef LAUNCH_FWD_ROWS
        }
    launched:;
    }
    int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0) return st;
    hipLaunchKernelGGL((k_attn_fwd_combine<T, H, D>), dim3((int)P->n_heavy, H * D / WAVE), dim3(BLOCK), 0, s, P->heavy,
                       (const float *)ws_acc, (const float *)ws_ml, (T *)o, lse, Narrow{}, (T *)nullptr);
    return launch_status();
}

template <typename T, int H, int D>
int run_attn_bwd(const bpt_plan *Pin, const bpt_plan *Pout, const void *q, const void *k, const void *v, const void *o,
                 const void *d_o, const float *lse, void *dq, void *dk, void *dv, void *ws, float scale, Dropout drop, const float *bias,
                 float *ds_out, hipStream_t s) {
    if (Pin->n_items == 0) return BPT_OK;
    const bool grouped = grouped_backward(Pin, Pout, H, D, sizeof(T));
    const int64_t pbytes = pds_bytes(Pin, Pout, H, D, sizeof(T), !bias);
    float *pbuf = (float *)ws;                                   // per-row kernels: p (E, H) then ds (E, H)
    float *dsbuf = pbuf + pbytes / 8;
    float2 *pds = (float2 *)ws;                                  // row-group kernels: interleaved (p, ds)
    float *ws_rows = (float *)ws + pbytes / 4;
    if constexpr (D == 64 && sizeof(T) == 4) {
        if (tiled_backward(Pin, Pout, H, D, sizeof(T)) && ((drop.thr == 0 && !bias) || Pin->grp_eids)) {
            constexpr int HW = H >= 4 ? 4 : H;
            float *ws_dk = ws_rows + (size_t)Pin->n_slots * H * D, *ws_dv = ws_dk + (size_t)Pout->n_slots * H * D;
            {
                ProfScope prof(BPT_KERNEL_ATTN_BWD_DST, s);
                const int parts = tile_parts(Pin, H, sizeof(T));
#define LAUNCH_DST_TILE_PARTS(DR, BI, SP)                                                                                              \
    hipLaunchKernelGGL((k_attn_bwd_dst_tile<T, H, D, HW, DR, BI, false, SP>), dim3(group_grid(Pin) * (H * SP / HW)), dim3(HW * WAVE), 0, s, \
                       *Pin, (const T *)q, (const T *)k, (const T *)v, (const T *)o, (const T *)d_o, lse, (T *)dq, pds, ws_rows, scale,    \
                       scale * LOG2E, drop.thr, drop.seed, drop.inv, bias, ds_out, Narrow{})
#define LAUNCH_DST_TILE(DR, BI)                                                                                                        \
    do {                                                                                                                               \
        if (parts == 4) LAUNCH_DST_TILE_PARTS(DR, BI, 4);                                                                              \
        else if (parts == 2) LAUNCH_DST_TILE_PARTS(DR, BI, 2);                                                                         \
        else LAUNCH_DST_TILE_PARTS(DR, BI, 1);                                                                                         \
    } while (0)
                switch ((drop.thr != 0 ? 1 : 0) + 2 * tile_bias_mode(Pin, bias)) {
                case 0: LAUNCH_DST_TILE(false, 0); break;
                case 1: LAUNCH_DST_TILE(true, 0); break;
                case 2: LAUNCH_DST_TILE(false, 1); break;
                case 3: LAUNCH_DST_TILE(true, 1); break;
                case 4: LAUNCH_DST_TILE(false, 2); break;
                default: LAUNCH_DST_TILE(true, 2); break;
                }
#undef LAUNCH_DST_TILE
#undef LAUNCH_DST_TILE_PARTS
            }
            int st = launch_status();
            if (st != BPT_OK) return st;
            {
                ProfScope prof(BPT_KERNEL_ATTN_BWD_SRC, s);
#define LAUNCH_SRC_TILE(SP)                                                                                                              \
    hipLaunchKernelGGL((k_attn_bwd_src_tile<T, H, D, HW, false, SP>), dim3(group_grid(Pout) * (H * SP / HW)), dim3(HW * WAVE), 0, s, *Pout,  \
                       (const T *)q, (const T *)d_o, (const float2 *)pds, (T *)dk, (T *)dv, ws_dk, ws_dv, Narrow{})
                const int parts = tile_parts(Pout, H, sizeof(T));
                if (parts == 4) LAUNCH_SRC_TILE(4);
                else if (parts == 2) LAUNCH_SRC_TILE(2);
                else LAUNCH_SRC_TILE(1);
#undef LAUNCH_SRC_TILE
            }
            st = launch_status();
            if (st != BPT_OK || Pin->n_heavy + Pout->n_heavy == 0) return st;
            hipLaunchKernelGGL((k_combine_sum3<T>), dim3((int)(Pin->n_heavy + Pout->n_heavy), H * D / (4 * WAVE), 2), dim3(BLOCK), 0, s, Pin->heavy,
                               (int)Pin->n_heavy, (const float *)ws_rows, (T *)dq, Pout->heavy, (const float *)ws_dk, (T *)dk, (T *)dv, H * D,
                               (size_t)Pout->n_slots * H * D, Narrow{});
            return launch_status();
        }
    }
    if constexpr (D == 64 && sizeof(T) == 2) {
        if (tiled_backward(Pin, Pout, H, D, sizeof(T)) && ((drop.thr == 0 && !bias) || Pin->grp_eids)) {
            const bool again = forms_pairs_again(Pout, drop, bias);
            constexpr int HW = H >= 4 ? 4 : H;
            float *ws_dk = ws_rows + (size_t)Pin->n_slots * H * D, *ws_dv = ws_dk + (size_t)Pout->n_slots * H * D;
            {
                ProfScope prof(BPT_KERNEL_ATTN_BWD_DST, s);
                const int parts = tile_parts(Pin, H, sizeof(T));
#define LAUNCH_DST_TILE_PARTS(DR, BI, PD, SP)                                                                                            \
    hipLaunchKernelGGL((k_attn_bwd_dst_rows_bf16<H, D, HW, TILE_BF16_WPE_DST, DR, BI, PD, SP>),                              \
                       dim3(group_grid(Pin) * (H * SP / HW)), dim3(HW * WAVE), 0, s, *Pin, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, (const bf16_t *)o,             \
                       (const bf16_t *)d_o, lse, (bf16_t *)dq, (uint32_t *)ws, (float2 *)ws, ws_rows, scale, scale * LOG2E, drop.thr,       \
                       drop.seed, drop.inv, bias, ds_out)
#define LAUNCH_DST_TILE(DR, BI, PD)                                                                                                      \
    do {                                                                                                                                 \
        if (parts == 4) LAUNCH_DST_TILE_PARTS(DR, BI, PD, 4);                                                                            \
        else if (parts == 2) LAUNCH_DST_TILE_PARTS(DR, BI, PD, 2);                                                                       \
        else LAUNCH_DST_TILE_PARTS(DR, BI, PD, 1);                                                                                       \
    } while (0)
                switch (again ? (drop.thr != 0 ? 7 : 6) : (drop.thr != 0 ? 1 : 0) + 2 * tile_bias_mode(Pin, bias)) {
                case 6: LAUNCH_DST_TILE(false, 0, false); break;
                case 7: LAUNCH_DST_TILE(true, 0, false); break;
                case 1: LAUNCH_DST_TILE(true, 0, true); break;
                case 2: LAUNCH_DST_TILE(false, 1, true); break;
                case 3: LAUNCH_DST_TILE(true, 1, true); break;
                case 4: LAUNCH_DST_TILE(false, 2, true); break;
                default: LAUNCH_DST_TILE(true, 2, true); break;
                }
#undef LAUNCH_DST_TILE
#undef LAUNCH_DST_TILE_PARTS
            }
            int st = launch_status();
            if (st != BPT_OK) return st;
            {
                ProfScope prof(BPT_KERNEL_ATTN_BWD_SRC, s);
                const int parts = tile_parts(Pout, H, sizeof(T));
#define LAUNCH_SRC_AGAIN_PARTS(DR, SP)                                                                                                   \
    hipLaunchKernelGGL((k_attn_bwd_src_tile_bf16_again<H, D, HW, TILE_BF16_WPE_AGAIN, DR, SP>), dim3(group_grid(Pout) * (H * SP / HW)),      \
                       dim3(HW * WAVE), 0, s, *Pout, (const bf16_t *)q, (const bf16_t *)k, (const bf16_t *)v, (const bf16_t *)d_o,         \
                       (const float2 *)ws, (bf16_t *)dk, (bf16_t *)dv, ws_dk, ws_dv, scale, scale * LOG2E, drop.thr, drop.seed, drop.inv)
#define LAUNCH_SRC_PDS(SP)                                                                                                               \
    hipLaunchKernelGGL((k_attn_bwd_src_tile_bf16<H, D, HW, TILE_BF16_WPE_SRC, false, SP>), dim3(group_grid(Pout) * (H * SP / HW)), \
                       dim3(HW * WAVE), 0, s, *Pout, (const bf16_t *)q, (const bf16_t *)d_o, (const uint32_t *)ws, (bf16_t *)dk, (bf16_t *)dv, \
                       ws_dk, ws_dv, Narrow{})
#define LAUNCH_SRC_TILE(SP)                                                                                                              \
    do {                                                                                                                                 \
        if (again && drop.thr != 0) LAUNCH_SRC_AGAIN_PARTS(true, SP);                                                                    \
        else if (again) LAUNCH_SRC_AGAIN_PARTS(false, SP);                                                                               \
        else LAUNCH_SRC_PDS(SP);                                                                                                         \
    } while (0)
                if (parts == 4) LAUNCH_SRC_TILE(4);
                else if (parts == 2) LAUNCH_SRC_TILE(2);
                else LAUNCH_SRC_TILE(1);
#undef LAUNCH_SRC_TILE
#undef LAUNCH_SRC_PDS
#undef LAUNCH_SRC_AGAIN_PARTS
            }
            st = launch_status();
            if (st != BPT_OK || Pin->n_heavy + Pout->n_heavy == 0) return st;
            hipLaunchKernelGGL((k_combine_sum3<T>), dim3((int)(Pin->n_heavy + Pout->n_heavy), H * D / (4 * WAVE), 2), dim3(BLOCK), 0, s, Pin->heavy,
                               (int)Pin->n_heavy, (const float *)ws_rows, (T *)dq, Pout->heavy, (const float *)ws_dk, (T *)dk, (T *)dv, H * D,
                               (size_t)Pout->n_slots * H * D, Narrow{});
            return launch_status();
        }
    }
    {
        ProfScope prof(BPT_KERNEL_ATTN_BWD_DST, s);
        if (grouped) {
#define LAUNCH_DST(RR, DR, BI)                                                                                                           \
    hipLaunchKernelGGL((k_attn_bwd_dst_grp<T, H, D, RR, HS, DR, BI>), dim3(group_grid(Pin) * HS), dim3(WAVE), 0, s, *Pin, (const T *)q, \
                       (const T *)k, (const T *)v, (const T *)o, (const T *)d_o, lse, (T *)dq, pds, ws_rows, scale, scale * LOG2E,      \
                       drop.thr, drop.seed, drop.inv, bias, ds_out)
            constexpr int HS = head_slices<T, H, D>();
            const int variant = (drop.thr != 0 ? 1 : 0) + (bias ? 2 : 0) + (Pin->grp_R == 8 ? 4 : 0);
            switch (variant) {
            case 0: LAUNCH_DST(4, false, false); break;
            case 1: LAUNCH_DST(4, true, false); break;
            case 2: LAUNCH_DST(4, false, true); break;
            case 3: LAUNCH_DST(4, true, true); break;
            case 4: LAUNCH_DST(8, false, false); break;
            case 5: LAUNCH_DST(8, true, false); break;
            case 6: LAUNCH_DST(8, false, true); break;
            default: LAUNCH_DST(8, true, true); break;
            }
#undef LAUNCH_DST
        } else {
#define LAUNCH_DST_ROWS(NW)                                                                                                              \
    hipLaunchKernelGGL((k_attn_bwd_dst<T, H, D, FAST_BATCH, NW>), dim3(NW == 1 ? grid_for(Pin) : (int)Pin->n_items),                         \
                       dim3(NW == 1 ? BLOCK : NW * WAVE), 0, s, *Pin, (const T *)q, (const T *)k, (const T *)v, (const T *)o, (const T *)d_o, lse, \
                       (T *)dq, pbuf, dsbuf, ws_rows, scale, scale * LOG2E)
            switch (row_parts(Pin, H * D)) {
            case 8: LAUNCH_DST_ROWS(8); break;
            case 4: LAUNCH_DST_ROWS(4); break;
            default: LAUNCH_DST_ROWS(1); break;
            }
#undef LAUNCH_DST_ROWS
        }
    }
    int st = launch_status();
    if (st != BPT_OK) return st;
    if (Pin->n_heavy > 0 && !grouped) {
        hipLaunchKernelGGL((k_combine_sum_v4<T>), dim3((int)Pin->n_heavy, H * D / (4 * WAVE), 1), dim3(BLOCK), 0, s, Pin->heavy,
                           (const float *)ws_rows, (T *)dq, (T *)nullptr, H * D, (size_t)0);
        st = launch_status();
        if (st != BPT_OK) return st;
    }
    // source side: dK[src] = sum ds * q[dst], dV[src] = sum p * dO[dst]
    if (!grouped) {
        ProfScope prof(BPT_KERNEL_ATTN_BWD_SRC, s);
        return run_spmm_fast<T, float, H, D, 2>(Pout, dsbuf, q, dk, pbuf, d_o, dv, ws_rows, s);
    }
    float *ws_dk = ws_rows + (size_t)Pin->n_slots * H * D, *ws_dv = ws_dk + (size_t)Pout->n_slots * H * D;
    {
        ProfScope prof(BPT_KERNEL_ATTN_BWD_SRC, s);
#define LAUNCH_SRC(RR)                                                                                                            \
    hipLaunchKernelGGL((k_attn_bwd_src_grp<T, H, D, RR, HS>), dim3(group_grid(Pout) * HS), dim3(WAVE), 0, s, *Pout, (const T *)q, \
                       (const T *)d_o, (const float2 *)pds, (T *)dk, (T *)dv, ws_dk, ws_dv)
        constexpr int HS = head_slices<T, H, D>();
        if (Pout->grp_R == 8) LAUNCH_SRC(8);
        else LAUNCH_SRC(4);
#undef LAUNCH_SRC
    }
    st = launch_status();
    if (st != BPT_OK || Pin->n_heavy + Pout->n_heavy == 0) return st;
    // partial rows of dq (destination side) and of dk, dv (source side) in one launch
    hipLaunchKernelGGL((k_combine_sum3<T>), dim3((int)(Pin->n_heavy + Pout->n_heavy), H * D / (4 * WAVE), 2), dim3(BLOCK), 0, s, Pin->heavy,
                       (int)Pin->n_heavy, (const float *)ws_rows, (T *)dq, Pout->heavy, (const float *)ws_dk, (T *)dk, (T *)dv, H * D,
                       (size_t)Pout->n_slots * H * D, Narrow{});
    return launch_status();
}

// ---- heads of fewer than 64 columns ----
template <typename T> bool narrow_ok(const bpt_plan *P, const Narrow &nw) {
    return has_tiles(P, nw.h, 64, sizeof(T)) && (P->grp_eids != nullptr);
}

template <typename T>
int run_attn_fwd_narrow(const bpt_plan *P, const void *q, const void *k, const void *v, void *o, float *lse, void *ws, float scale, Dropout drop,
                        const Narrow &nw, const Keep &keep, hipStream_t s) {
    float *ws_acc = (float *)ws, *ws_ml = ws_acc ? ws_acc + (size_t)P->n_slots * nw.h * 64 : nullptr;
    const int parts = tile_parts(P, nw.heads, sizeof(T));
    const Narrow np = narrow_parts(nw, parts);
    const dim3 grid(group_grid(P) * np.slices + 8 * keep.per_xcd), block((parts == 1 ? NARROW_HW : parts) * WAVE);
    if (grid.x == 0) return BPT_OK;
    {
        ProfScope prof(BPT_KERNEL_ATTN_FWD, s);
#define LAUNCH_FWD_PARTS(DR, HW, SP)                                                                                                     \
    do {                                                                                                                                 \
        if constexpr (sizeof(T) == 4)                                                                                                    \
            hipLaunchKernelGGL((k_attn_fwd_tile<T, 16, 64, HW, DR, 0, true, SP>), grid, block, 0, s, *P, (const T *)q, (const T *)k,         \
                               (const T *)v, (T *)o, lse, ws_acc, ws_ml, scale * LOG2E, drop.thr, drop.seed, drop.inv, (const float *)nullptr, np, keep); \
        else                                                                                                                             \
            hipLaunchKernelGGL((k_attn_fwd_tile_bf16<16, 64, HW, TILE_BF16_WPE, DR, SP>), grid, block, 0, s, *P,                             \
                               (const T *)q, (const T *)k, (const T *)v, (T *)o, lse, ws_acc, ws_ml, scale * LOG2E, drop.thr, drop.seed,       \
                               drop.inv, np, keep);                                                                                        \
    } while (0)
#define LAUNCH_FWD(DR)                                                                                                                   \
    do {                                                                                                                                 \
        if (parts == 4) LAUNCH_FWD_PARTS(DR, 4, 4);                                                                                      \
        else if (parts == 2) LAUNCH_FWD_PARTS(DR, 2, 2);                                                                                 \
        else LAUNCH_FWD_PARTS(DR, NARROW_HW, 1);                                                                                         \
    } while (0)
        if (drop.thr != 0) LAUNCH_FWD(true); else LAUNCH_FWD(false);
#undef LAUNCH_FWD_PARTS
#undef LAUNCH_FWD
    }
    const int st = launch_status();
    if (st != BPT_OK || P->n_heavy == 0) return st;
    hipLaunchKernelGGL((k_attn_fwd_combine<T, 16, 64, true>), dim3((int)P->n_heavy, nw.heads), dim3(BLOCK), 0, s, P->heavy, (const float *)ws_acc,
                       (const float *)ws_ml, (T *)o, lse, nw, (T *)keep.o);
    return launch_status();
}

template <typename T>
int run_attn_bwd_narrow(const bpt_plan *Pin, const bpt_plan *Pout, const void *q, const void *k, const void *v, const void *o, const void *d_o,
                        const float *lse, void *dq, void *dk, void *dv, void *ws, float scale, Dropout drop, const Narrow &nw, hipStream_t s) {
    if (Pin->n_items == 0) return BPT_OK;
    using pds_t = std::conditional_t<sizeof(T) == 4, float2, uint32_t>;
    pds_t *pds = (pds_t *)ws;
    float *ws_dq = (float *)ws + pds_bytes(Pin, Pout, nw.h, 64, sizeof(T), false) / 4;
    float *ws_dk = ws_dq + (size_t)Pin->n_slots * nw.h * 64, *ws_dv = ws_dk + (size_t)Pout->n_slots * nw.h * 64;
    const int parts = tile_parts(Pin, nw.heads, sizeof(T)), parts_src = tile_parts(Pout, nw.heads, sizeof(T));
    const Narrow np = narrow_parts(nw, parts), np_src = narrow_parts(nw, parts_src);
    const dim3 grid(group_grid(Pin) * np.slices), block((parts == 1 ? NARROW_HW : parts) * WAVE);
    const dim3 grid_src(group_grid(Pout) * np_src.slices), block_src((parts_src == 1 ? NARROW_HW : parts_src) * WAVE);
    {
        ProfScope prof(BPT_KERNEL_ATTN_BWD_DST, s);
#define LAUNCH_DST_PARTS(DR, HW, SP)                                                                                                     \
    do {                                                                                                                                 \
        if constexpr (sizeof(T) == 4)                                                                                                    \
            hipLaunchKernelGGL((k_attn_bwd_dst_tile<T, 16, 64, HW, DR, 0, true, SP>), grid, block, 0, s, *Pin, (const T *)q,                 \
                               (const T *)k, (const T *)v, (const T *)o, (const T *)d_o, lse, (T *)dq, pds, ws_dq, scale, scale * LOG2E,       \
                               drop.thr, drop.seed, drop.inv, (const float *)nullptr, (float *)nullptr, np);                                \
        else                                                                                                                             \
            hipLaunchKernelGGL((k_attn_bwd_dst_tile_bf16<16, 64, HW, TILE_BF16_WPE_DST, DR, SP>), grid, block, 0, s, *Pin,                   \
                               (const T *)q, (const T *)k, (const T *)v, (const T *)o, (const T *)d_o, lse, (T *)dq, pds, ws_dq, \
                               scale, scale * LOG2E, drop.thr, drop.seed, drop.inv, np);          \
    } while (0)
#define LAUNCH_DST(DR)                                                                                                                   \
    do {                                                                                                                                 \
        if (parts == 4) LAUNCH_DST_PARTS(DR, 4, 4);                                                                                      \
        else if (parts == 2) LAUNCH_DST_PARTS(DR, 2, 2);                                                                                 \
        else LAUNCH_DST_PARTS(DR, NARROW_HW, 1);                                                                                         \
    } while (0)
        if (drop.thr != 0) LAUNCH_DST(true); else LAUNCH_DST(false);
#undef LAUNCH_DST_PARTS
#undef LAUNCH_DST
    }
    int st = launch_status();
    if (st != BPT_OK) return st;
    {
        ProfScope prof(BPT_KERNEL_ATTN_BWD_SRC, s);
#define LAUNCH_SRC(HW, SP)                                                                                                               \
    do {                                                                                                                                 \
        if constexpr (sizeof(T) == 4)                                                                                                    \
            hipLaunchKernelGGL((k_attn_bwd_src_tile<T, 16, 64, HW, true, SP>), grid_src, block_src, 0, s, *Pout, (const T *)q, (const T *)d_o, \
                               pds, (T *)dk, (T *)dv, ws_dk, ws_dv, np_src);                                                               \
        else                                                                                                                             \
            hipLaunchKernelGGL((k_attn_bwd_src_tile_bf16<16, 64, HW, TILE_BF16_WPE_SRC, true, SP>), grid_src, block_src, 0, s, *Pout,        \
                               (const T *)q, (const T *)d_o, pds, (T *)dk, (T *)dv, ws_dk, ws_dv, np_src);                                  \
    } while (0)
        if (parts_src == 4) LAUNCH_SRC(4, 4);
        else if (parts_src == 2) LAUNCH_SRC(2, 2);
        else LAUNCH_SRC(NARROW_HW, 1);
#undef LAUNCH_SRC
    }
    st = launch_status();
    if (st != BPT_OK || Pin->n_heavy + Pout->n_heavy == 0) return st;
    hipLaunchKernelGGL((k_combine_sum3<T, true>), dim3((int)(Pin->n_heavy + Pout->n_heavy), nw.h * 64 / (4 * WAVE), 2), dim3(BLOCK), 0, s, Pin->heavy,
                       (int)Pin->n_heavy, (const float *)ws_dq, (T *)dq, Pout->heavy, (const float *)ws_dk, (T *)dk, (T *)dv, nw.h * 64,
                       (size_t)Pout->n_slots * nw.h * 64, nw);
    return launch_status();
}

// heads x d that the NARROW forms take: the padded head count has fused kernels, rows start on 4 bytes, a quad fits a head
int narrow_shape(int heads, int d, int h, int dtype, Narrow &nw) {
    if (heads < 1 || d < 1) return BPT_ERR_SHAPE;
    if (dtype != BPT_F32 && dtype != BPT_BF16) return BPT_ERR_UNSUPPORTED;
    if (!fast_shape(h, 64, dtype) || heads > h || d < 4 || d > 64 || (dtype == BPT_BF16 && d % 2 != 0)) return BPT_ERR_UNSUPPORTED;
    nw = Narrow{d, heads, h, (heads + NARROW_HW - 1) / NARROW_HW};
    return BPT_OK;
}

inline bool aligned4(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 3) == 0; }

}  // namespace

// Workspace of bpt_attention_forward_noalloc: one copy per GPU, held until the process ends.  In host code this
// name is only a handle for hipGetSymbolAddress; kernels get the device address that call returns.
static __device__ __align__(256) unsigned char scratch[BPT_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int MAX_SCRATCH_DEVICES = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[MAX_SCRATCH_DEVICES] = {};

// device address of `scratch` on the current device (looked up once per device)
int scratch_of_current_device(void **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= MAX_SCRATCH_DEVICES) return BPT_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!p) return BPT_ERR_NULL;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return BPT_OK;
}

}  // namespace

// ------------------------------------------------------------------------------------------
// C ABI
// ------------------------------------------------------------------------------------------
extern "C" {

const char *bpt_strerror(int status) {
    if (status > 0) return hipGetErrorString((hipError_t)status);
    switch (status) {
        case BPT_OK: return "ok";
        case BPT_ERR_NULL: return "required pointer is NULL";
        case BPT_ERR_SIZE: return "negative or inconsistent size";
        case BPT_ERR_DTYPE: return "unknown dtype";
        case BPT_ERR_SHAPE: return "h and d must be positive (h*d <= 2^20)";
        case BPT_ERR_WORKSPACE: return "workspace missing or too small";
        case BPT_ERR_PLAN: return "plans do not describe the same graph";
        case BPT_ERR_UNSUPPORTED: return "combination not implemented";
        case BPT_ERR_SCRATCH: return "the call needs more than the library's static scratch (BPT_NOALLOC_SCRATCH_BYTES)";
        default: return "unknown bptattn status";
    }
}

int64_t bpt_plan_struct_bytes(void) { return (int64_t)sizeof(bpt_plan); }

int bpt_set_force_generic(int on) { return g_force_generic.exchange(on ? 1 : 0); }

int bpt_gather_probe(const void *region, int64_t region_bytes, int waves_per_cu, int in_flight, int iters, float *sink, void *stream) {
    if (!region || !sink) return BPT_ERR_NULL;
    if (region_bytes < 1024 || region_bytes / 1024 > 0x7fffffff || waves_per_cu < WAVES_PER_BLOCK || waves_per_cu > 64 || iters < 1)
        return BPT_ERR_SIZE;
    if (!aligned16(region)) return BPT_ERR_UNSUPPORTED;
    const int grid = 256 * (waves_per_cu / WAVES_PER_BLOCK);      // 256 compute units
    const uint32_t n_rows = (uint32_t)(region_bytes / 1024);
    hipStream_t s = (hipStream_t)stream;
    switch (in_flight) {
    case 2: hipLaunchKernelGGL((k_gather_probe<2>), dim3(grid), dim3(BLOCK), 0, s, (const float4 *)region, n_rows, iters, sink); break;
    case 4: hipLaunchKernelGGL((k_gather_probe<4>), dim3(grid), dim3(BLOCK), 0, s, (const float4 *)region, n_rows, iters, sink); break;
    case 8: hipLaunchKernelGGL((k_gather_probe<8>), dim3(grid), dim3(BLOCK), 0, s, (const float4 *)region, n_rows, iters, sink); break;
    default: return BPT_ERR_SIZE;
    }
    return launch_status();
}

int bpt_wavefronts_per_item(const bpt_plan *plan, int kernel, int h, int d, int dtype) {
    if (!plan) return BPT_ERR_NULL;
    if (kernel < BPT_KERNEL_ATTN_FWD || kernel > BPT_KERNEL_ATTN_BWD_SRC || h < 1 || d < 1) return BPT_ERR_SHAPE;
    if (dtype != BPT_F32 && dtype != BPT_BF16) return BPT_ERR_DTYPE;
    const size_t elem = dtype == BPT_F32 ? 4 : 2;
    if (has_tiles(plan, h, d, elem)) return tile_parts(plan, h, elem, kernel == BPT_KERNEL_ATTN_FWD);
    return row_parts(plan, h * d, kernel == BPT_KERNEL_ATTN_FWD && dtype == BPT_F32);
}

int bpt_wavefronts_per_product(const bpt_plan *plan, int h, int d) {
    if (!plan) return BPT_ERR_NULL;
    if (h < 1 || d < 1) return BPT_ERR_SHAPE;
    if (!product_tiles_ok(plan, h, d, BPT_F32)) return 0;
    return product_parts(plan, h, shared_heads(h, d, true, true));
}

int bpt_profile_kernel(int which, void *start_event, void *stop_event) {
    if (which != 0 && (!start_event || !stop_event)) return BPT_ERR_NULL;
    g_prof_start.store(start_event);
    g_prof_stop.store(stop_event);
    g_prof_which.store(which);
    return BPT_OK;
}

// partial rows of a SpMM on this plan (on tiles: whole heads of 64 columns)
static int64_t spmm_rows_bytes(const bpt_plan *P, int h, int d, int dtype) {
    return P ? round16(P->n_slots * std::max((int64_t)h * d, product_tiles_ok(P, h, d, dtype) ? (int64_t)product_tile_heads(h) * 64 : 0) * (int64_t)acc_size(dtype)) : 0;
}

int64_t bpt_workspace_bytes(int op, const bpt_plan *plan, const bpt_plan *plan_t, int h, int d, int dtype) {
    if (!plan || h < 1 || d < 1) return -1;
    const int64_t C = (int64_t)h * d, a = (int64_t)acc_size(dtype);
    const int64_t s0 = plan->n_slots, s1 = plan_t ? plan_t->n_slots : 0;
    auto rows = [&](const bpt_plan *P) { return spmm_rows_bytes(P, h, d, dtype); };
    switch (op) {
        case BPT_OP_MASKEDMM_BWD:                     // (both sides' at once where one launch adds them up)
            return plan_t && product_tiles_ok(plan, h, d, dtype) && product_tiles_ok(plan_t, h, d, dtype) ? rows(plan) + rows(plan_t)
                                                                                                           : std::max(rows(plan), rows(plan_t));
        case BPT_OP_NODE_MUL_EDGE_BWD: return round16(s0 * C * a);
        case BPT_OP_SPMM_FWD: return rows(plan);
        case BPT_OP_SPMM_BWD: return rows(plan_t);
        case BPT_OP_ATTN_FWD: return round16(s0 * (C + 2 * h) * 4);
        case BPT_OP_SOFTMAX_FWD: return h <= WAVE ? round16(s0 * h * 2 * a) : 0;      // (m, s) of every segment and head
        case BPT_OP_SOFTMAX_BWD: return h <= WAVE ? round16(s0 * h * a) : 0;
        case BPT_OP_ATTN_BWD:
        case BPT_OP_ATTN_BWD_PLAIN: {
            // partial rows of dq, then of dk and dv (the three are merged by one launch after the source-side kernel)
            return pds_bytes(plan, plan_t, h, d, dtype == BPT_BF16 ? 2 : 4, op == BPT_OP_ATTN_BWD_PLAIN) + round16((s0 + 2 * s1) * C * 4);
        }
        default: return -1;
    }
}

#define CHECK(expr) do { const int st_ = (expr); if (st_ != BPT_OK) return st_; } while (0)

int bpt_maskedmm_csr_forward(const bpt_plan *plan, const void *A, const void *B, void *y, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan, true));
    CHECK(check_shape(h, d, dtype));
    if (plan->n_edges > 0 && (!A || !B || !y)) return BPT_ERR_NULL;
    return sddmm(plan, A, B, y, h, d, dtype, (hipStream_t)stream);
}

int bpt_maskedmm_csr_backward(const bpt_plan *plan_r, const bpt_plan *plan_c, const void *A, const void *B, const void *dy,
                              void *dA, void *dB, void *workspace, int64_t workspace_bytes, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan_r, true));
    CHECK(check_plan(plan_c, true));
    CHECK(check_shape(h, d, dtype));
    if (plan_r->n_edges != plan_c->n_edges) return BPT_ERR_PLAN;
    if (!dA || !dB || (plan_r->n_edges > 0 && (!A || !B || !dy))) return BPT_ERR_NULL;
    const int64_t rows_r = spmm_rows_bytes(plan_r, h, d, dtype), rows_c = spmm_rows_bytes(plan_c, h, d, dtype), need = std::max(rows_r, rows_c);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    const bool whole_r = product_whole_heads(h, d, aligned16(B) && aligned16(dA)), whole_c = product_whole_heads(h, d, aligned16(A) && aligned16(dB));
    if (product_tiles_ok(plan_r, h, d, dtype) && product_tiles_ok(plan_c, h, d, dtype) && aligned16(workspace) && workspace_bytes >= rows_r + rows_c &&
        whole_r == whole_c)
        return spmm_tile_pair(plan_r, B, dA, workspace, plan_c, A, dB, (char *)workspace + rows_r, dy, h, d, (hipStream_t)stream);
    CHECK(spmm(plan_r, dy, B, dA, workspace, h, d, dtype, (hipStream_t)stream));
    return spmm(plan_c, dy, A, dB, workspace, h, d, dtype, (hipStream_t)stream);
}

int bpt_rel_bias_forward(const bpt_plan *plan, const void *q, const void *table, const int32_t *used_types, int64_t n_used, float *bias, int h,
                         int d, int dtype, void *stream) {
    CHECK(check_plan(plan, true));
    CHECK(check_shape(h, d, dtype));
    if (plan->n_edges > 0 && (!q || !table || !bias)) return BPT_ERR_NULL;
    if (plan->bias_by_pair && !used_types) return BPT_ERR_UNSUPPORTED;      // only the kernel below writes the head-major form
    hipStream_t s = (hipStream_t)stream;
    if (used_types) {                       // plan indices are type numbers: the kernel with the table rows in LDS
        if (n_used < 0) return BPT_ERR_SIZE;
        if (!rel_rows_shape(h, d, dtype) || n_used > REL_MAX_USED || !aligned16(q) || !aligned16(table) || !aligned16(bias)) return BPT_ERR_UNSUPPORTED;
        if (plan->n_edges == 0 && (!bias || plan->bias_by_pair)) return BPT_OK;      // (no spare row to clear)
#define X(HH) if (h == HH) return run_rel_bias_rows<T, HH>(plan, q, table, used_types, n_used, bias, s);
        if (dtype == BPT_F32) { using T = float; X(4) X(8) X(16) }
        if (dtype == BPT_BF16) { using T = bf16_t; X(4) X(8) X(16) }
#undef X
        return BPT_ERR_UNSUPPORTED;
    }
    if (!fast_shape(h, d, dtype) || !aligned16(q) || !aligned16(table)) return BPT_ERR_UNSUPPORTED;
#define X(HH, DD) if (h == HH && d == DD) return run_rel_bias<T, HH, DD>(plan, q, table, bias, s);
    if (dtype == BPT_F32) { using T = float; BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { using T = bf16_t; BPT_FAST_SHAPES_BF16(X) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int bpt_rel_bias_forward_tiles(const bpt_plan *plan, const void *q, const void *table, const int32_t *used_types, int64_t n_used,
                               const int32_t *pair_types, float *bias, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan, true));
    CHECK(check_shape(h, d, dtype));
    if (n_used < 0) return BPT_ERR_SIZE;
    if (!rel_rows_shape(h, d, dtype) || n_used > REL_MAX_USED || !has_tiles(plan, h, d, dtype == BPT_BF16 ? 2 : 4)) return BPT_ERR_UNSUPPORTED;
    if (plan->n_edges == 0) return BPT_OK;
    if (!q || !table || !used_types || !pair_types || !bias) return BPT_ERR_NULL;
    if (n_used == 0) return BPT_ERR_SIZE;                        // (edges without a type in use)
    if (!aligned16(q) || !aligned16(table)) return BPT_ERR_UNSUPPORTED;
    hipStream_t s = (hipStream_t)stream;
#define X(HH) if (h == HH) return run_rel_bias_tiles<T, HH>(plan, q, table, used_types, n_used, pair_types, bias, s);
    if (dtype == BPT_F32) { using T = float; X(4) X(8) X(16) }
    if (dtype == BPT_BF16) { using T = bf16_t; X(4) X(8) X(16) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int64_t bpt_rel_bias_backward_workspace_bytes(const bpt_plan *plan, int64_t n_used, int h) {
    if (!plan || n_used < 0 || h < 1) return 0;
    return (plan->n_slots * h * 64 + n_used * REL_MAX_PARTS * 64) * 4;
}

int bpt_rel_bias_backward_supported(int64_t n_used, int h, int d, int dtype) {
    if (n_used < 0) return BPT_ERR_SIZE;
    if (!rel_rows_shape(h, d, dtype) || n_used > REL_MAX_USED) return BPT_ERR_UNSUPPORTED;
#define X(HH) if (h == HH) return rel_bias_bwd_config<T, HH>(n_used);
    if (dtype == BPT_F32) { using T = float; X(4) X(8) X(16) }
    if (dtype == BPT_BF16) { using T = bf16_t; X(4) X(8) X(16) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int bpt_rel_bias_backward(const bpt_plan *plan, const float *ds, const void *q, const void *table, const int32_t *used,
                          const int32_t *used_types, int64_t n_types, int64_t n_used, void *dq, void *dtable, void *workspace,
                          int64_t workspace_bytes, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan, true));
    CHECK(check_shape(h, d, dtype));
    if (n_types < 0 || n_used < 0 || n_used > n_types) return BPT_ERR_SIZE;
    if (!rel_rows_shape(h, d, dtype) || n_used > REL_MAX_USED || rel_bwd_shape(n_used, h).nw == 0) return BPT_ERR_UNSUPPORTED;
    if (n_types == 0) return BPT_OK;
    if (!used || !dtable || (n_used > 0 && !used_types) || (plan->n_edges > 0 && (!ds || !q || !table || !dq))) return BPT_ERR_NULL;
    if (!aligned16(ds) || !aligned16(table)) return BPT_ERR_UNSUPPORTED;
    if (!workspace || workspace_bytes < bpt_rel_bias_backward_workspace_bytes(plan, n_used, h) || !aligned16(workspace)) return BPT_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
#define X(HH) if (h == HH) return run_rel_bias_bwd<T, HH>(plan, ds, q, table, used, used_types, n_types, n_used, dq, dtable, (float *)workspace, s);
    if (dtype == BPT_F32) { using T = float; X(4) X(8) X(16) }
    if (dtype == BPT_BF16) { using T = bf16_t; X(4) X(8) X(16) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int bpt_node_mul_edge_forward(const bpt_plan *plan, const void *A, const void *B, void *y, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan, false));
    CHECK(check_shape(h, d, dtype));
    if (plan->n_edges > 0 && (!A || !B || !y)) return BPT_ERR_NULL;
    if (fast_shape(h, d, dtype) && aligned16(A) && aligned16(B)) return nme_fwd_fast(plan, A, B, y, h, d, dtype, (hipStream_t)stream);
    return sddmm_edge_generic(plan, A, B, y, h, d, dtype, (hipStream_t)stream);
}

int bpt_node_mul_edge_backward(const bpt_plan *plan, const void *A, const void *B, const void *dy, void *dA, void *dB,
                               void *workspace, int64_t workspace_bytes, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan, false));
    CHECK(check_shape(h, d, dtype));
    if (!dA || (plan->n_edges > 0 && (!A || !B || !dy || !dB))) return BPT_ERR_NULL;
    const int64_t need = bpt_workspace_bytes(BPT_OP_NODE_MUL_EDGE_BWD, plan, nullptr, h, d, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    if (fast_shape(h, d, dtype) && aligned16(B) && aligned16(dA) && aligned16(workspace))
        return nme_bwd_fast(plan, A, B, dy, dA, dB, workspace, h, d, dtype, (hipStream_t)stream);
    CHECK(spmm_edge_generic(plan, dy, B, dA, workspace, h, d, dtype, (hipStream_t)stream));
    DISPATCH_DTYPE(dtype, (run_nme_dB<T>(plan, A, dy, dB, h, d, (hipStream_t)stream)))
}

int bpt_sparse_softmax_forward(const bpt_plan *plan, const void *x, void *y, void *workspace, int64_t workspace_bytes, int h,
                               int dtype, void *stream) {
    CHECK(check_plan(plan, false));
    CHECK(check_shape(h, 1, dtype));
    if (plan->n_edges > 0 && (!x || !y)) return BPT_ERR_NULL;
    const int64_t need = bpt_workspace_bytes(BPT_OP_SOFTMAX_FWD, plan, nullptr, h, 1, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    DISPATCH_DTYPE(dtype, (run_softmax_fwd<T>(plan, x, y, workspace, h, (hipStream_t)stream)))
}

int bpt_sparse_softmax_backward(const bpt_plan *plan, const void *y, const void *dy, void *dx, void *workspace,
                                int64_t workspace_bytes, int h, int dtype, void *stream) {
    CHECK(check_plan(plan, false));
    CHECK(check_shape(h, 1, dtype));
    if (plan->n_edges > 0 && (!y || !dy || !dx)) return BPT_ERR_NULL;
    const int64_t need = bpt_workspace_bytes(BPT_OP_SOFTMAX_BWD, plan, nullptr, h, 1, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    DISPATCH_DTYPE(dtype, (run_softmax_bwd<T>(plan, y, dy, dx, workspace, h, (hipStream_t)stream)))
}

int bpt_vector_spmm_forward(const bpt_plan *plan, const void *edata, const void *x, void *y, void *workspace,
                            int64_t workspace_bytes, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan, true));
    CHECK(check_shape(h, d, dtype));
    if (!y || (plan->n_edges > 0 && (!edata || !x))) return BPT_ERR_NULL;
    const int64_t need = bpt_workspace_bytes(BPT_OP_SPMM_FWD, plan, nullptr, h, d, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    return spmm(plan, edata, x, y, workspace, h, d, dtype, (hipStream_t)stream);
}

int bpt_vector_spmm_accumulate(const bpt_plan *plan, const void *edata, const void *x, void *y, void *workspace,
                               int64_t workspace_bytes, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan, true));
    CHECK(check_shape(h, d, dtype));
    if (!y || (plan->n_edges > 0 && (!edata || !x))) return BPT_ERR_NULL;
    if (plan->n_edges == 0) return BPT_OK;
    const int64_t need = bpt_workspace_bytes(BPT_OP_SPMM_FWD, plan, nullptr, h, d, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    // exists in the row-group kernels only
    if (!(fast_shape(h, d, dtype) && aligned16(x) && aligned16(y) && aligned16(workspace) && spmm_grp_ok(plan, h, d, dtype)))
        return BPT_ERR_UNSUPPORTED;
    return spmm_grp(plan, edata, x, y, workspace, h, d, dtype, (hipStream_t)stream, 1);
}

int bpt_vector_spmm_backward(const bpt_plan *plan, const bpt_plan *plan_t, const void *edata, const void *dy, const void *x,
                             void *dedata, void *dx, void *workspace, int64_t workspace_bytes, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan, true));
    CHECK(check_plan(plan_t, true));
    CHECK(check_shape(h, d, dtype));
    if (plan->n_edges != plan_t->n_edges) return BPT_ERR_PLAN;
    if (!dx || (plan->n_edges > 0 && (!edata || !dy || !x || !dedata))) return BPT_ERR_NULL;
    const int64_t need = bpt_workspace_bytes(BPT_OP_SPMM_BWD, plan, plan_t, h, d, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    CHECK(sddmm(plan, dy, x, dedata, h, d, dtype, (hipStream_t)stream));
    return spmm(plan_t, edata, dy, dx, workspace, h, d, dtype, (hipStream_t)stream);
}

int bpt_attention_forward(const bpt_plan *plan_in, const void *q, const void *k, const void *v, const float *bias, void *o,
                          float *lse, void *workspace, int64_t workspace_bytes, float scale, float dropout_p, uint64_t dropout_seed,
                          int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan_in, true));
    CHECK(check_shape(h, d, dtype));
    if (!q || !k || !v || !o || !lse) return BPT_ERR_NULL;
    if (!(dropout_p >= 0.f && dropout_p < 1.f)) return BPT_ERR_SIZE;
    const Dropout drop = make_dropout(dropout_p, dropout_seed);
    // dropout and the score term exist in the row-group and the tile kernels only
    if ((drop.thr != 0 || bias) && !has_groups(plan_in, h, d, dtype == BPT_BF16 ? 2 : 4) && !has_tiles(plan_in, h, d, dtype == BPT_BF16 ? 2 : 4))
        return BPT_ERR_UNSUPPORTED;
    if ((bias || drop.thr != 0) && !plan_in->grp_eids) return BPT_ERR_PLAN;
    // only the tile kernels look the rows of the score term up in a numbering of the plan's own
    if (bias && plan_in->bias_by_pair && !has_tiles(plan_in, h, d, dtype == BPT_BF16 ? 2 : 4)) return BPT_ERR_PLAN;
    if (!fast_shape(h, d, dtype) || !aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o) || !aligned16(workspace))
        return BPT_ERR_UNSUPPORTED;
    const int64_t need = bpt_workspace_bytes(BPT_OP_ATTN_FWD, plan_in, nullptr, h, d, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
#define X(HH, DD) if (h == HH && d == DD) return run_attn_fwd<T, HH, DD>(plan_in, q, k, v, o, lse, workspace, scale, drop, bias, s);
    if (dtype == BPT_F32) { using T = float; BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { using T = bf16_t; BPT_FAST_SHAPES_BF16(X) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int bpt_attention_forward_noalloc(const bpt_plan *plan_in, const void *q, const void *k, const void *v, const float *bias, void *o,
                                  float *lse, float scale, float dropout_p, uint64_t dropout_seed, int h, int d, int dtype,
                                  void *stream) {
    CHECK(check_plan(plan_in, true));
    CHECK(check_shape(h, d, dtype));
    const int64_t need = bpt_workspace_bytes(BPT_OP_ATTN_FWD, plan_in, nullptr, h, d, dtype);
    if (need < 0) return BPT_ERR_SIZE;
    if (need > (int64_t)BPT_NOALLOC_SCRATCH_BYTES) return BPT_ERR_SCRATCH;
    void *ws = nullptr;
    CHECK(scratch_of_current_device(&ws));
    return bpt_attention_forward(plan_in, q, k, v, bias, o, lse, ws, (int64_t)BPT_NOALLOC_SCRATCH_BYTES, scale, dropout_p, dropout_seed,
                                 h, d, dtype, stream);
}

int bpt_attention_backward(const bpt_plan *plan_in, const bpt_plan *plan_out, const void *q, const void *k, const void *v,
                           const float *bias, const void *o, const void *d_o, const float *lse, void *dq, void *dk, void *dv,
                           float *ds_out, void *workspace, int64_t workspace_bytes, float scale, float dropout_p,
                           uint64_t dropout_seed, int h, int d, int dtype, void *stream) {
    CHECK(check_plan(plan_in, true));
    CHECK(check_plan(plan_out, true));
    CHECK(check_shape(h, d, dtype));
    if (!(dropout_p >= 0.f && dropout_p < 1.f)) return BPT_ERR_SIZE;
    const Dropout drop = make_dropout(dropout_p, dropout_seed);
    if ((drop.thr != 0 || bias) && !grouped_backward(plan_in, plan_out, h, d, dtype == BPT_BF16 ? 2 : 4) &&
        !tiled_backward(plan_in, plan_out, h, d, dtype == BPT_BF16 ? 2 : 4))
        return BPT_ERR_UNSUPPORTED;
    if ((bias != nullptr) != (ds_out != nullptr)) return BPT_ERR_NULL;       // the score term and its gradient go together
    if ((bias || drop.thr != 0) && !plan_in->grp_eids) return BPT_ERR_PLAN;
    if (bias && plan_in->bias_by_pair && !tiled_backward(plan_in, plan_out, h, d, dtype == BPT_BF16 ? 2 : 4)) return BPT_ERR_PLAN;
    // (the two sides may have different row counts: attention to a memory of another length, attention.py:144-168)
    if (plan_in->n_edges != plan_out->n_edges) return BPT_ERR_PLAN;
    if (!q || !k || !v || !o || !d_o || !lse || !dq || !dk || !dv) return BPT_ERR_NULL;
    if (!fast_shape(h, d, dtype) || !aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o) || !aligned16(d_o) ||
        !aligned16(dq) || !aligned16(dk) || !aligned16(dv) || !aligned16(workspace))
        return BPT_ERR_UNSUPPORTED;
    const int64_t need = bpt_workspace_bytes(bias ? BPT_OP_ATTN_BWD : BPT_OP_ATTN_BWD_PLAIN, plan_in, plan_out, h, d, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
#define X(HH, DD) \
    if (h == HH && d == DD) return run_attn_bwd<T, HH, DD>(plan_in, plan_out, q, k, v, o, d_o, lse, dq, dk, dv, workspace, scale, drop, bias, ds_out, s);
    if (dtype == BPT_F32) { using T = float; BPT_FAST_SHAPES_F32(X) }
    if (dtype == BPT_BF16) { using T = bf16_t; BPT_FAST_SHAPES_BF16(X) }
#undef X
    return BPT_ERR_UNSUPPORTED;
}

int bpt_attention_forward_narrow_keep(const bpt_plan *plan_in, const void *q, const void *k, const void *v, void *o, float *lse, void *const keep[4],
                                      int64_t n_q, int64_t n_k, void *workspace, int64_t workspace_bytes, float scale, float dropout_p,
                                      uint64_t dropout_seed, int heads, int d, int h, int dtype, void *stream) {
    CHECK(check_plan(plan_in, true));
    Narrow nw;
    CHECK(narrow_shape(heads, d, h, dtype, nw));
    if (!q || !k || !v || !o || !lse || !keep) return BPT_ERR_NULL;
    if (!(dropout_p >= 0.f && dropout_p < 1.f)) return BPT_ERR_SIZE;
    const Dropout drop = make_dropout(dropout_p, dropout_seed);
    if (!(dtype == BPT_F32 ? narrow_ok<float>(plan_in, nw) : narrow_ok<bf16_t>(plan_in, nw))) return BPT_ERR_UNSUPPORTED;
    if (!aligned4(q) || !aligned4(k) || !aligned4(v) || !aligned4(o) || !aligned16(workspace)) return BPT_ERR_UNSUPPORTED;
    const int64_t need = bpt_workspace_bytes(BPT_OP_ATTN_FWD, plan_in, nullptr, h, 64, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    if (n_q < 0 || n_k < 0 || (keep[3] && !aligned4(keep[3]))) return BPT_ERR_SIZE;
    Keep kp{};
    int64_t chunks = 0;
    const void *const from[3] = {q, k, v};
    for (int i = 0; i < 3; ++i) {
        if (!keep[i]) continue;
        if (!aligned16(keep[i])) return BPT_ERR_UNSUPPORTED;
        kp.src[i] = (const char *)from[i];
        kp.dst[i] = (char *)keep[i];
        kp.bytes[i] = (i == 0 ? n_q : n_k) * heads * d * (dtype == BPT_F32 ? 4 : 2);
        chunks += (kp.bytes[i] + KEEP_CHUNK - 1) / KEEP_CHUNK;
    }
    if (chunks >= (1 << 27)) return BPT_ERR_SIZE;
    kp.per_xcd = (int)((chunks + 7) / 8);
    kp.o = keep[3];
    hipStream_t s = (hipStream_t)stream;
    return dtype == BPT_F32 ? run_attn_fwd_narrow<float>(plan_in, q, k, v, o, lse, workspace, scale, drop, nw, kp, s)
                            : run_attn_fwd_narrow<bf16_t>(plan_in, q, k, v, o, lse, workspace, scale, drop, nw, kp, s);
}

int bpt_attention_forward_narrow(const bpt_plan *plan_in, const void *q, const void *k, const void *v, void *o, float *lse, void *workspace,
                                 int64_t workspace_bytes, float scale, float dropout_p, uint64_t dropout_seed, int heads, int d, int h,
                                 int dtype, void *stream) {
    void *const none[4] = {};
    return bpt_attention_forward_narrow_keep(plan_in, q, k, v, o, lse, none, 0, 0, workspace, workspace_bytes, scale, dropout_p, dropout_seed, heads, d,
                                             h, dtype, stream);
}

int bpt_attention_backward_narrow(const bpt_plan *plan_in, const bpt_plan *plan_out, const void *q, const void *k, const void *v, const void *o,
                                  const void *d_o, const float *lse, void *dq, void *dk, void *dv, void *workspace, int64_t workspace_bytes,
                                  float scale, float dropout_p, uint64_t dropout_seed, int heads, int d, int h, int dtype, void *stream) {
    CHECK(check_plan(plan_in, true));
    CHECK(check_plan(plan_out, true));
    Narrow nw;
    CHECK(narrow_shape(heads, d, h, dtype, nw));
    if (!q || !k || !v || !o || !d_o || !lse || !dq || !dk || !dv) return BPT_ERR_NULL;
    if (!(dropout_p >= 0.f && dropout_p < 1.f)) return BPT_ERR_SIZE;
    if (plan_in->n_edges != plan_out->n_edges) return BPT_ERR_PLAN;
    const Dropout drop = make_dropout(dropout_p, dropout_seed);
    if (!tiled_backward(plan_in, plan_out, h, 64, dtype == BPT_BF16 ? 2 : 4) || !plan_in->grp_eids) return BPT_ERR_UNSUPPORTED;
    if (!aligned4(q) || !aligned4(k) || !aligned4(v) || !aligned4(o) || !aligned4(d_o) || !aligned4(dq) || !aligned4(dk) || !aligned4(dv) ||
        !aligned16(workspace))
        return BPT_ERR_UNSUPPORTED;
    const int64_t need = bpt_workspace_bytes(BPT_OP_ATTN_BWD, plan_in, plan_out, h, 64, dtype);
    if (need > 0 && (!workspace || workspace_bytes < need)) return BPT_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    return dtype == BPT_F32 ? run_attn_bwd_narrow<float>(plan_in, plan_out, q, k, v, o, d_o, lse, dq, dk, dv, workspace, scale, drop, nw, s)
                            : run_attn_bwd_narrow<bf16_t>(plan_in, plan_out, q, k, v, o, d_o, lse, dq, dk, dv, workspace, scale, drop, nw, s);
}

}  // extern "C"
