// HIP kernels of the MI355X streaming DBSCAN slide step (gfx950, wave64).
//
// One slide of every stream in a batch is eight launches:
//   sort_expire (stride sort in runs + survivors per window tile) ->
//   rank (stride rank merge + survivor compaction) -> merge_final -> cells ->
//   rows -> count -> merge_cells -> border (outputs)
// (several streams and large ones: count_points -> cell_cores -> merge_cells ->
// border_regroup; small windows: update_small instead of the first four; single
// small streams and reach 1: union instead of merge_cells).
// Each kernel covers all streams of the batch in one launch: a block finds its
// stream from prefix tables of per-stream work units (tiles of positions,
// 64-position chunks) or, for the cell kernels whose sizes are only known on
// the device, walks a device-side work list in a persistent loop.
//
// Semantics follow the reference's hot path (RTDBStream level 9,
// src/dbscan/dbscan.cpp:2276-2362) and its checker (util.cpp:383-442):
// FP32 distances ((dx*dx + dy*dy) + dz*dz) without contraction, strict
// d2 < eps2, self-inclusive counts, core iff count >= min_pts, union-find
// hooking the larger root under the smaller (dbscan.cu:22-43) with slots as
// the order, so every cluster id is its minimum core slot.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include <hip/hip_ext.h>

#include "rtdbs_dev.h"
#include "rtdbs_devfn.h"

namespace rtdbs {

const char *const kPhaseNames[kNumPhases] = {"sort_expire", "rank_compact", "merge_final",
                                             "cells", "rows", "count", "union", "border"};

// ---------------------------------------------------------------------------
// small helpers


// Largest s in [0, n) with pre[s] <= g (pre[0] = 0, g < pre[n]); pre in LDS.
template <class T>
__device__ __forceinline__ int find_stream(const T *pre, int n, long long g) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if ((long long)pre[mid] <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

// The stream of cell g for a wave that walks its cells in increasing order:
// the largest s >= s0 with pre[s] <= g (pre[s0] <= g), by galloping from the
// previous cell's stream - one probe while the stream stays the same -
// instead of a full binary search per cell. Scalar loads (constant memory).
__device__ __forceinline__ int find_stream_from(const int32_t *pre, int n, int g, int s0) {
    int lo = s0, hi = s0 + 1, step = 1;
    while (hi < n && ldc(pre[hi]) <= g) {
        lo = hi;
        step <<= 1;
        hi = min(lo + step, n);
    }
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ldc(pre[mid]) <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

// The same over a per-batch prefix table in global memory, which no kernel
// writes during a launch: scalar loads (the table stays in the scalar cache),
// not a dependent vector load per step.
__device__ __forceinline__ int find_stream_c(const int32_t *pre, int n, long long g) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if ((long long)ldc(pre[mid]) <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Logical index of workgroup b of n. The dispatcher hands workgroups to the
// 8 XCDs round-robin (b runs on XCD b mod 8), and each XCD has its own L2.
// With `on`, the workgroups of XCD x take the x-th contiguous eighth of the
// logical range, so work items that are neighbours in that range (cells or
// positions whose stencils share candidates) run on one XCD and share its
// L2. A bijection on [0, n) for any n: XCD x holds n/8 workgroups, one more
// when x < n mod 8. Measured: in a 3.2 M-point batch it shortens the merge
// (385 -> 373 us) and the point-parallel output kernel (200 -> 184 us) and
// lengthens the count and rows kernels (190 -> 210 us, 127 -> 161 us); on
// single streams of 0.1-1 M points it lengthens every kernel. So the engine
// enables it per kernel (BatchArgs::xcd_groups).
__device__ __forceinline__ int xcd_block(int b, int n, bool on) {
    if (!on) return b;
    const int q = n >> 3, r = n & 7, x = b & 7;
    return x * q + min(x, r) + (b >> 3);
}

__device__ __forceinline__ uint32_t slot_mask(const StreamDev &S) {
    return (uint32_t)((1ull << S.slot_bits) - 1ull);
}

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += xor_lane(v, o);
    return v;
}

// Value of lane `l` (uniform) of a per-lane int.
__device__ __forceinline__ int lane_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// Sum over a 256-thread block.
__device__ __forceinline__ int block_sum(int v, int *lds4) {
    v = wave_sum(v);
    const int w = threadIdx.x >> 6;
    if (lane_id() == 0) lds4[w] = v;
    __syncthreads();
    int tot = lds4[0] + lds4[1] + lds4[2] + lds4[3];
    __syncthreads();
    return tot;
}

// Exclusive rank of this thread's flag within a 256-thread block, plus the
// block total (ordered stream compaction by wave ballot/popcount).
__device__ __forceinline__ int block_rank_flags(bool f, int *total, int *lds4) {
    const int lane = lane_id(), w = threadIdx.x >> 6;
    const uint64_t m = __ballot(f);
    const int below = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) lds4[w] = __popcll(m);
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        int c = lds4[i];
        base += (i < w) ? c : 0;
        tot += c;
    }
    __syncthreads();
    *total = tot;
    return base + below;
}

// Inclusive prefix (into pre[1..n], pre[0] = 0) of per-stream values over a
// block of 256 threads; n <= kMaxBatch. Values are 64-bit.
template <class F>
__device__ void block_stream_prefix(int n, long long *pre, long long *tmp4, F value) {
    const int tid = threadIdx.x;
    // each thread owns 4 consecutive streams
    long long v[4];
    long long local = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        int i = tid * 4 + q;
        v[q] = (i < n) ? value(i) : 0;
        local += v[q];
    }
    // wave inclusive scan of `local`
    const int lane = lane_id(), w = tid >> 6;
    long long x = local;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        long long y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) tmp4[w] = x;
    __syncthreads();
    long long wbase = 0;
    for (int i = 0; i < w; i++) wbase += tmp4[i];
    long long run = wbase + x - local;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        int i = tid * 4 + q;
        run += v[q];
        if (i < n) pre[i + 1] = run;
    }
    if (tid == 0) pre[0] = 0;
    __syncthreads();
}

__device__ __forceinline__ int slot_of(const StreamDev &S, int pos) {
    return (int)((uint32_t)S.skey[pos] & (uint32_t)((1ull << S.slot_bits) - 1ull));
}

// ---------------------------------------------------------------------------
// grid

// The grid of a stream read once as constant memory (uniform per block), for
// kernels that compute many keys.
struct KeyGrid {
    double lo0, lo1, lo2, inv_side;
    int64_t n0, n1, n2;
    int dim, slot_bits;
};

__device__ __forceinline__ KeyGrid key_grid(const StreamDev &S) {
    KeyGrid g;
    g.lo0 = ldc(S.lo[0]);
    g.lo1 = ldc(S.lo[1]);
    g.lo2 = ldc(S.lo[2]);
    g.inv_side = ldc(S.inv_side);
    g.n0 = ldc(S.n[0]);
    g.n1 = ldc(S.n[1]);
    g.n2 = ldc(S.n[2]);
    g.dim = ldc(S.dim);
    g.slot_bits = ldc(S.slot_bits);
    return g;
}

// Cell index per axis: floor((x - lo) / side) evaluated in double and clamped
// into the grid. Clamping keeps the search exact: |clamp(i) - clamp(j)| <=
// |i - j|, so points within reach stay within reach.
__device__ __forceinline__ int64_t bin_axis(double x, double lo, double inv, int64_t n) {
    double v = floor((x - lo) * inv);
    if (!(v >= 0.0)) v = 0.0;  // negative or NaN
    const double mx = (double)(n - 1);
    if (v > mx) v = mx;
    return (int64_t)v;
}

// Packed cell key (i0 * n1 + i1) * n2 + i2; unused axes have index 0.
__device__ __forceinline__ uint64_t cell_key_g(const KeyGrid &G, float x, float y, float z) {
    const int64_t i0 = bin_axis((double)x, G.lo0, G.inv_side, G.n0);
    const int64_t i1 = G.dim > 1 ? bin_axis((double)y, G.lo1, G.inv_side, G.n1) : 0;
    const int64_t i2 = G.dim > 2 ? bin_axis((double)z, G.lo2, G.inv_side, G.n2) : 0;
    return (uint64_t)((i0 * G.n1 + i1) * G.n2 + i2);
}

// Quotient and remainder of a cell key (< 2^52, so exact in a double) by a
// grid extent (<= 2^30), via a double-precision estimate, off by at most one,
// and an exact integer fix-up (64-bit integer division is a long software
// sequence on the GPU).
__device__ __forceinline__ void divmod_key(uint64_t x, int64_t d, int64_t *q, int64_t *r) {
    int64_t qq = (int64_t)((double)x / (double)d);
    int64_t rr = (int64_t)x - qq * d;
    while (rr < 0) {
        qq--;
        rr += d;
    }
    while (rr >= d) {
        qq++;
        rr -= d;
    }
    *q = qq;
    *r = rr;
}

// ---------------------------------------------------------------------------
// sorting: register bitonic tile sort, rank merge of the stride's tiles,
// merge-path merges of the window

__device__ __forceinline__ uint64_t readlane64(uint64_t v, int l) {
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, l);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), l);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int m) {
    const int lo = xor_lane((int)(uint32_t)v, m);
    const int hi = xor_lane((int)(uint32_t)(v >> 32), m);
    return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}

// Compare-exchange of lanes l and l ^ m (m a power of two below 64): the
// smaller key where keep_min, else the larger. For m = 16 and 32 the row-pair
// and half-wave swaps of both copies of a word leave the lower partner's
// value in one register and the upper partner's in the other, in every lane,
// so no select picks the partner out first.
__device__ __forceinline__ uint64_t lane_minmax(uint64_t v, int m, bool keep_min) {
    uint64_t x, y;
    if (m == 16 || m == 32) {
        const int lo = (int)(uint32_t)v, hi = (int)(uint32_t)(v >> 32);
        const auto rl = m == 32 ? __builtin_amdgcn_permlane32_swap(lo, lo, false, false)
                                : __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto rh = m == 32 ? __builtin_amdgcn_permlane32_swap(hi, hi, false, false)
                                : __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        x = ((uint64_t)(uint32_t)rh[0] << 32) | (uint32_t)rl[0];  // lane l & ~m
        y = ((uint64_t)(uint32_t)rh[1] << 32) | (uint32_t)rl[1];  // lane l | m
    } else {
        x = v;
        y = shfl_xor_u64(v, m);
    }
    return ((y < x) == keep_min) ? y : x;
}

// Sorts N keys ascending, E per thread: thread t (of N/E) holds positions
// Et..Et+E-1 in v. Bitonic network: exchanges between a thread's own elements
// stay in registers, exchanges within a wave use lane exchanges, and only the
// stages whose partners sit in another wave (j >= 64E) go through LDS (`lds`,
// N keys) with block barriers: none for N = 64E (one wave), three stages for
// a 512-key run over four waves (E = 2) and for N = 2048 over four waves
// (E = 8). Every thread of the block takes part in the same stages.
template <int N, int E>
__device__ __forceinline__ void bitonic_sort_regs(uint64_t (&v)[E], uint64_t *lds, int tid) {
#pragma unroll
    for (int k = 2; k <= N; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= E) {
                const int m = j / E;  // partner thread = tid ^ m, same element index
                const bool keep_min = ((tid & m) == 0) == (((tid * E) & k) == 0);
                if (j >= 64 * E) {
                    __syncthreads();
#pragma unroll
                    for (int e = 0; e < E; e++) lds[tid * E + e] = v[e];
                    __syncthreads();
#pragma unroll
                    for (int e = 0; e < E; e++) {
                        const uint64_t o = lds[(tid ^ m) * E + e];
                        v[e] = ((o < v[e]) == keep_min) ? o : v[e];
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < E; e++) v[e] = lane_minmax(v[e], m, keep_min);
                }
            } else {
#pragma unroll
                for (int e = 0; e < E; e++) {
                    if (e & j) continue;
                    const bool up = (((tid * E) + e) & k) == 0;
                    const uint64_t x = v[e], y = v[e | j];
                    const bool sw = (x > y) == up;
                    v[e] = sw ? y : x;
                    v[e | j] = sw ? x : y;
                }
            }
        }
    }
}

// Loads the packed keys (cell << slot_bits | slot) of points [tile0, tile0 +
// N) of `in` (len points, slots from slot0) into v, E per thread (tid < N/E),
// and sorts them; padding keys are ~0 and sort last. Thread tid takes points
// tid, tid + N/E, ... so each load instruction reads consecutive points (the
// network sorts any assignment; a key carries its own slot).
template <int N, int E>
__device__ __forceinline__ void sort_tile_keys(const KeyGrid &G, gptr<const float> in, int len, int tile0, int slot0,
                                               uint64_t (&v)[E], uint64_t *lds, int tid) {
    const int dim = G.dim;
    float c[E][3];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int gi = min(tile0 + e * (N / E) + tid, len - 1);
#pragma unroll
        for (int a = 0; a < 3; a++) c[e][a] = a < dim ? in[(size_t)gi * dim + a] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int gi = tile0 + e * (N / E) + tid;
        v[e] = gi < len ? (cell_key_g(G, c[e][0], c[e][1], c[e][2]) << G.slot_bits) | (uint64_t)(slot0 + gi) : ~0ull;
    }
    bitonic_sort_regs<N, E>(v, lds, tid);
}

// Bounds of a first window's points, NaNs passed over: one partial result per
// block (low per axis, then high; infinities where a block saw no number),
// written to pinned host memory, where the host joins them and lays out the
// grid. On the host the same scan is two serial chains of compares per axis:
// with it, opening a stream of 200,000 points took some 290 us longer.
__global__ __launch_bounds__(kTileThreads) void k_bounds(const float *in, int W, int dim, float *bnd) {
    __shared__ float part[kTileThreads / 64][6];
    float lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; a++) lo[a] = __builtin_inff(), hi[a] = -__builtin_inff();
    for (int p = blockIdx.x * kTileThreads + threadIdx.x; p < W; p += kBoundBlocks * kTileThreads)
#pragma unroll
        for (int a = 0; a < 3; a++) {
            if (a >= dim) break;
            const float v = gl(in)[(size_t)p * dim + a];
            lo[a] = v < lo[a] ? v : lo[a];
            hi[a] = v > hi[a] ? v : hi[a];
        }
    const int lane = lane_id(), w = threadIdx.x >> 6;
#pragma unroll
    for (int a = 0; a < 3; a++) {
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const float l = __shfl_xor(lo[a], m), h = __shfl_xor(hi[a], m);
            lo[a] = l < lo[a] ? l : lo[a];
            hi[a] = h > hi[a] ? h : hi[a];
        }
        if (lane == 0) part[w][a] = lo[a], part[w][3 + a] = hi[a];
    }
    __syncthreads();
    if (threadIdx.x >= 6) return;
    float r = part[0][threadIdx.x];
#pragma unroll
    for (int k = 1; k < kTileThreads / 64; k++) {
        const float v = part[k][threadIdx.x];
        r = (threadIdx.x < 3 ? v < r : v > r) ? v : r;
    }
    bnd[blockIdx.x * 6 + threadIdx.x] = r;
}

// The window in slot order: each position's point stored at its slot, so that
// one copy brings the whole to the host. 200,000 points in 3-D: 539 us as four
// copies put in order by the host, 176 us so.
__global__ __launch_bounds__(kTileThreads) void k_window_out(BatchArgs a, float *out, int32_t *bad) {
    const StreamDev &S = a.s[0];
    const int p = blockIdx.x * kTileThreads + threadIdx.x, W = ldc(S.W), dim = ldc(S.dim);
    if (p >= W) return;
    const uint32_t slot = (uint32_t)gl(ldc(S.skey))[p] & slot_mask(S);
    if (slot >= (uint32_t)W) {
        *bad = 1;
        return;
    }
    const gptr<float> o = gl(out) + (size_t)slot * dim;
    o[0] = gl(ldc(S.sx))[p];
    if (dim > 1) o[1] = gl(ldc(S.sy))[p];
    if (dim > 2) o[2] = gl(ldc(S.sz))[p];
}

// First window, launch 1: runs of kTile sorted keys, 16 waves per run (two keys
// per thread), into the akey (sel 0) or skey (sel 1) half of the ping-pong.
// A run is one serial chain of exchange stages, so a window of few runs takes
// as long as one of them, however the rest of the device idles: with 4 waves
// of 8 keys per thread this launch took 91 us at 200,000 points.
constexpr int kInitThreads = kTile / 2;

// Key of the first window's position p into the window arrays, with its
// coordinates taken from the input: they are the same bytes as in the runs,
// so the sort moves keys alone.
__device__ __forceinline__ void init_place(const StreamDev &S, gptr<const float> in, int p, uint64_t key, int dim) {
    const gptr<const float> c = in + (size_t)((uint32_t)key & slot_mask(S)) * dim;
    gl(ldc(S.skey))[p] = key;
    gl(ldc(S.sx))[p] = c[0];
    if (dim > 1) gl(ldc(S.sy))[p] = c[1];
    if (dim > 2) gl(ldc(S.sz))[p] = c[2];
}

template <bool LAST>
__global__ __launch_bounds__(kInitThreads) void k_init_tiles(BatchArgs a, int sel, int t, int u) {
    __shared__ uint64_t lds[kTile];
    const StreamDev &S = a.s[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) *S.mut = StreamMut{t, u, 0, {0, 0, 0, 0, 0}};
    const int tile0 = blockIdx.x * kTile, W = ldc(S.W), dim = ldc(S.dim);
    uint64_t v[2];
    sort_tile_keys<kTile, 2>(key_grid(S), gl(a.io1.in), W, tile0, 0, v, lds, threadIdx.x);
    const gptr<uint64_t> out = gl(sel ? ldc(S.skey) : ldc(S.akey));
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const int i = tile0 + threadIdx.x * 2 + e;
        if (i >= W) continue;
        if (LAST) init_place(S, gl(a.io1.in), i, v[e], dim);
        else out[i] = v[e];
    }
}


// Survivors per window tile (the reference's stable_partition,
// thrust_helper.cu:37-39, split into count + compact).
__device__ __forceinline__ void expire_count(const BatchArgs &a, int g, int *lds4) {
    const int s = find_stream_c(a.pre_wtile, a.n, g);
    const StreamDev &S = a.s[s];
    const int tile = g - ldc(a.pre_wtile[s]);
    const int W = ldc(S.W), SS = ldc(S.S);
    const gptr<const uint64_t> skey = gl((const uint64_t *)ldc(S.skey));
    const uint32_t sm = (uint32_t)((1ull << ldc(S.slot_bits)) - 1ull);
    const int p0 = tile * kWTile, p1 = min(p0 + kWTile, W);
    const int lo_slot = ldc(ldc(S.mut)->u) * SS;
    uint64_t k[kWTile / kTileThreads];
#pragma unroll
    for (int r = 0; r < kWTile / kTileThreads; r++) {
        const int p = p0 + threadIdx.x + r * kTileThreads;
        k[r] = p < p1 ? skey[p] : 0ull;
    }
    int cnt = 0;
#pragma unroll
    for (int r = 0; r < kWTile / kTileThreads; r++) {
        const int slot = (int)((uint32_t)k[r] & sm);
        cnt += (p0 + (int)threadIdx.x + r * kTileThreads < p1) && (slot < lo_slot || slot >= lo_slot + SS);
    }
    cnt = block_sum(cnt, lds4);
    if (threadIdx.x == 0) gl(ldc(S.tile_a))[tile] = cnt;
}

// Launch 1 of a slide: the first kSortParts blocks of each stride tile sort
// the stride by key (the reference's compute_cell_id + sortByCellIdAndOrder,
// aabb.cu:589-611, thrust_helper.cu:21-29) in runs of at most kRun keys into
// bkey0, four waves per run (kSortE keys per thread: a quarter of the network's
// instructions per wave of a one-wave run, for three LDS stages); the
// remaining blocks count the survivors of each window tile.
constexpr int kRun = 512;                                // most keys of a sorted run of the stride
constexpr int kSortE = 2;                                // keys per thread
constexpr int kSortParts = kTile / kRun;                 // blocks per stride tile, a run each
static_assert(kRun == kSortE * kTileThreads, "");
constexpr int kRunChunks = kRun / 64;
typedef uint64_t KeyPair __attribute__((ext_vector_type(2)));

// The runs of a stride of SS keys: as few as hold it, of equal length but for
// one key (a short last run's 64 keys would span all other runs, whose every
// chunk the rank kernel would then search).
struct Runs {
    int n, len, longer;  // runs; keys of a run, and how many of the first hold one more
    __device__ __forceinline__ Runs(int SS) : n((SS + kRun - 1) / kRun), len(SS / n), longer(SS - n * len) {}
    __device__ __forceinline__ int start(int r) const { return r * len + min(r, longer); }
};

__global__ __launch_bounds__(kTileThreads) void k_sort_expire(BatchArgs a) {
    __shared__ uint64_t lds[kTile];
    const int g = blockIdx.x;
    const int nsb = ldc(a.pre_stile[a.n]) * kSortParts;
    if (g >= nsb) {
        expire_count(a, g - nsb, (int *)lds);
        return;
    }
    const int gt = g / kSortParts;
    const int s = find_stream_c(a.pre_stile, a.n, gt);
    const StreamDev &S = a.s[s];
    const IO io = a.use_io1 ? a.io1 : a.io[s];
    const int SS = ldc(S.S);
    const Runs runs(SS);
    const int run = (gt - ldc(a.pre_stile[s])) * kSortParts + g % kSortParts;
    if (run >= runs.n) return;  // the whole block: past the stride's end
    const int start = runs.start(run), nvalid = runs.start(run + 1) - start;
    uint64_t v[kSortE];
    sort_tile_keys<kRun, kSortE>(key_grid(S), gl(io.in), start + nvalid, start, ldc(ldc(S.mut)->u) * SS, v, lds,
                                 threadIdx.x);
    // coalesced store through LDS (thread i holds positions kSortE * i ..)
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kSortE; e++) lds[threadIdx.x * kSortE + e] = v[e];
    __syncthreads();
    const gptr<uint64_t> bkey0 = gl(ldc(S.bkey0));
    for (int i = threadIdx.x; i < nvalid; i += kTileThreads) bkey0[start + i] = lds[i];
    // first and last key of every 64
    if (threadIdx.x < kRunChunks && (int)threadIdx.x * 64 < nvalid)
        gl((KeyPair *)ldc(S.bends))[run * kRunChunks + threadIdx.x] =
            KeyPair{lds[threadIdx.x * 64], lds[min((int)threadIdx.x * 64 + 63, nvalid - 1)]};
}

// Ordered compaction of the survivors into the A arrays. Each tile's offset
// is the sum of the preceding tiles' counts (no spin-waiting look-back).
__device__ __forceinline__ void expire_compact(const BatchArgs &a, int g, int *lds4) {
    const int s = find_stream_c(a.pre_wtile, a.n, g);
    const StreamDev &S = a.s[s];
    const int tile = g - ldc(a.pre_wtile[s]);
    const int p0 = tile * kWTile;
    const int W = ldc(S.W), SS = ldc(S.S), dim = ldc(S.dim);
    const uint32_t sm = (uint32_t)((1ull << ldc(S.slot_bits)) - 1ull);
    const int lo_slot = ldc(ldc(S.mut)->u) * SS;
    const gptr<const uint64_t> skey = gl((const uint64_t *)ldc(S.skey));
    const gptr<const float> sx = gl((const float *)ldc(S.sx)), sy = gl((const float *)ldc(S.sy)),
                            sz = gl((const float *)ldc(S.sz));
    const gptr<const int32_t> tile_a = gl((const int32_t *)ldc(S.tile_a));
    constexpr int per = kWTile / kTileThreads;
    // every load of the tile issued before the scan and the stores
    uint64_t key[per];
    float cx[per], cy[per], cz[per];
#pragma unroll
    for (int r = 0; r < per; r++) {
        const int p = p0 + r * kTileThreads + threadIdx.x;
        const int pp = p < W ? p : 0;
        key[r] = skey[pp];
        cx[r] = sx[pp];
        cy[r] = dim > 1 ? sy[pp] : 0.f;
        cz[r] = dim > 2 ? sz[pp] : 0.f;
    }
    int part = 0;
    for (int t = threadIdx.x; t < tile; t += kTileThreads) part += tile_a[t];
    int run = block_sum(part, lds4);
    const gptr<uint64_t> akey = gl(ldc(S.akey));
    const gptr<float> ax = gl(ldc(S.ax)), ay = gl(ldc(S.ay)), az = gl(ldc(S.az));
#pragma unroll
    for (int r = 0; r < per; r++) {
        const int p = p0 + r * kTileThreads + threadIdx.x;
        const int slot = (int)((uint32_t)key[r] & sm);
        const bool f = p < W && (slot < lo_slot || slot >= lo_slot + SS);
        int tot;
        const int rank = block_rank_flags(f, &tot, lds4);
        if (f) {
            const int d = run + rank;
            akey[d] = key[r];
            ax[d] = cx[r];
            if (dim > 1) ay[d] = cy[r];
            if (dim > 2) az[d] = cz[r];
        }
        run += tot;
    }
}

// LDS written by lanes of this wave is read by others next.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Launch 2 of a slide: blocks [0, rank_blocks) place each stride key at its rank
// in the whole stride - its index in its sorted run plus, for every other
// run, the number of that run's keys below it - and write keys and
// coordinates to the B1 arrays: the stride sorted by (cell, slot). The blocks
// after them compact the window's survivors (expire_compact), which depends on
// the same launch before.
//
// 64 consecutive keys of a run lie close together, so of another run's chunks
// of 64 keys nearly all are wholly below or wholly above them: the chunks'
// first and last keys (written by the sort) tell, one chunk per lane. Only the
// two or so chunks of each run that reach into the keys' span are loaded into
// LDS and searched, kRankChunks at a time, the next ones on their way
// meanwhile. What bounds it is the searches: seven dependent LDS reads per
// chunk and key, S / 512 runs of two chunks. Searching whole runs staged in
// LDS, as before, moved the whole stride through every block; us of the launch
// so and now: 20,501 keys 17.0 and 11.8, 50,000 keys 48 and 27.5, 10,000 keys
// 10.4 and 6.8, the 64-stream batch (321,000 keys) 57 and 42.5, of which the
// compaction takes about 20. Eight chunks a step: 12.4 and 31.6 us at 20,501
// and 50,000 keys; three probes a step 11.2 and 28.1. With SPLIT == 1 each wave ranks 64 keys by itself; with
// SPLIT == 4 the four waves of a block split the other runs between them,
// summing their partial ranks in LDS at the end, for strides too small to fill
// the device otherwise.
constexpr int kRankChunks = 4;  // chunks searched together

template <int SPLIT>
__global__ __launch_bounds__(kTileThreads) void k_rank(BatchArgs a, int rank_blocks) {
    constexpr int kWaves = kTileThreads / 64;
    constexpr int kParts = kTile / 64 / (kWaves / SPLIT);  // blocks per stride tile
    __shared__ uint64_t lds[kWaves][kRankChunks][64];
    __shared__ int part[SPLIT > 1 ? kWaves : 1][64];
    if ((int)blockIdx.x >= rank_blocks) {  // the survivor compaction shares the launch
        expire_compact(a, blockIdx.x - rank_blocks, (int *)part);
        return;
    }
    const int g = blockIdx.x;
    const int gb = g / kParts;
    const int s = find_stream_c(a.pre_stile, a.n, gb);
    const StreamDev &S = a.s[s];
    const int SS = ldc(S.S), dim = ldc(S.dim);
    const int wv = uni(threadIdx.x >> 6), lane = lane_id();
    const int sigma = wv % SPLIT;  // which of the other runs this wave searches
    const Runs runs(SS);
    // this wave's or block's 64 keys: a chunk of a run
    const int mine = ((gb - ldc(a.pre_stile[s])) * kParts + g % kParts) * (kWaves / SPLIT) + (SPLIT > 1 ? 0 : wv);
    const int myrun = mine / kRunChunks;
    const int i0 = runs.start(myrun) + mine % kRunChunks * 64;
    const int nk = min(runs.start(myrun + 1) - i0, 64);
    if (myrun >= runs.n || nk <= 0) return;  // past the stride's or the run's end (the whole block where its waves meet)
    const gptr<const uint64_t> bkey0 = gl((const uint64_t *)ldc(S.bkey0));
    const gptr<const KeyPair> bends = gl((const KeyPair *)ldc(S.bends));
    const int i = i0 + lane;
    const bool valid = lane < nk;
    const uint64_t key = valid ? bkey0[i] : ~0ull;
    // this lane's chunk among those of 8 runs, whose first is r0
    auto run_of = [&](int r0) { return r0 + (lane >> 3) * SPLIT; };
    auto ends_of = [&](int r0) { return bends[min(run_of(r0), runs.n - 1) * kRunChunks + (lane & 7)]; };
    KeyPair ends = ends_of(sigma);
    // the point's coordinates are needed only at the end: loaded now
    const IO io = a.use_io1 ? a.io1 : a.io[s];
    float px = 0.f, py = 0.f, pz = 0.f;
    if (sigma == 0) {
        const int gi = valid ? (int)((uint32_t)key & slot_mask(S)) - ldc(ldc(S.mut)->u) * SS : 0;
        const gptr<const float> p = gl(io.in) + (size_t)gi * dim;
        px = p[0];
        py = dim > 1 ? p[1] : 0.f;
        pz = dim > 2 ? p[2] : 0.f;
    }
    const uint64_t kmin = readlane64(key, 0), kmax = readlane64(key, nk - 1);
    int rank = 0, whole = 0;
    for (int r0 = sigma; r0 < runs.n; r0 += 8 * SPLIT) {
        const int r = run_of(r0);
        const int left = r < runs.n && r != myrun ? runs.start(r + 1) - runs.start(r) - (lane & 7) * 64 : 0;
        const bool below = left > 0 && ends.y < kmin;
        whole += below ? min(left, 64) : 0;
        uint64_t m = __ballot(left > 0 && !below && ends.x < kmax);
        if (r0 + 8 * SPLIT < runs.n) ends = ends_of(r0 + 8 * SPLIT);
        // the next chunks' keys; every load is issued, clamped, so that no
        // branch waits for it
        uint64_t v[kRankChunks];
        int n[kRankChunks];
        auto load = [&]() {
#pragma unroll
            for (int q = 0; q < kRankChunks; q++) {
                const int l = m ? __ffsll((unsigned long long)m) - 1 : 0;
                const int r1 = r0 + (l >> 3) * SPLIT, p0 = runs.start(r1) + (l & 7) * 64;
                n[q] = m ? runs.start(r1 + 1) - p0 : 0;
                v[q] = bkey0[min(p0 + lane, SS - 1)];
                m &= m - 1ull;
            }
        };
        load();
        while (n[0] > 0) {
#pragma unroll
            for (int q = 0; q < kRankChunks; q++) lds[wv][q][lane] = lane < n[q] ? v[q] : ~0ull;
            load();
            wave_sync();
            int pos[kRankChunks] = {};
#pragma unroll
            for (int step = 32; step > 0; step >>= 1) {
#pragma unroll
                for (int q = 0; q < kRankChunks; q++)
                    pos[q] += lds[wv][q][pos[q] + step - 1] < key ? step : 0;
            }
#pragma unroll
            for (int q = 0; q < kRankChunks; q++) rank += pos[q] + (lds[wv][q][pos[q]] < key ? 1 : 0);
            wave_sync();
        }
    }
    rank += wave_sum(whole);
    if (SPLIT > 1) {
        part[wv][lane] = rank;
        __syncthreads();
        if (sigma != 0) return;
#pragma unroll
        for (int w = 1; w < SPLIT; w++) rank += part[w][lane];
    }
    if (!valid) return;
    rank += i - runs.start(myrun);
    gl(S.bkey1)[rank] = key;
    gl(S.bx1)[rank] = px;
    if (dim > 1) gl(S.by1)[rank] = py;
    if (dim > 2) gl(S.bz1)[rank] = pz;
}

// Number of elements of A among the first d of merge(A, B); keys are unique.
// P(i) = A[i] < B[d-1-i] holds exactly for i below the answer. One wave
// samples P at 64 evenly spaced points per round, so the search costs
// ceil(log64(range)) dependent round trips instead of log2(range).
__device__ __forceinline__ int merge_path_wave(const uint64_t *A, int la, const uint64_t *B, int lb, int d) {
    const int lane = lane_id();
    int lo = max(0, d - lb), hi = min(d, la);
    while (hi > lo) {
        const int n = hi - lo;
        const int step = (n + 63) >> 6;
        const int i = lo + lane * step;
        bool p = false;
        if (i < hi) p = A[i] < B[d - 1 - i];
        const int cnt = __popcll(__ballot(p));
        if (step == 1) return lo + cnt;
        if (cnt == 0) return lo;
        const int nlo = lo + (cnt - 1) * step + 1;
        const int nhi = min(hi, lo + cnt * step);
        lo = nlo;
        hi = nhi;
    }
    return lo;
}

template <int T>
struct MergeLds {
    uint64_t in[T];
    uint64_t out[T];
    int32_t src[T];  // >= 0: index into A; < 0: ~index into B
    int32_t sp[2];
    uint64_t pred;
};

// Merges outputs [d0, d1) (d1 - d0 <= T) of merge(A, B) into m.out and, with
// SRC, their sources into m.src (block-wide).
template <int T, bool SRC = true>
__device__ __forceinline__ void merge_tile(const uint64_t *A, int la, const uint64_t *B, int lb, int d0,
                                           int d1, MergeLds<T> &m, int *a0_out, int *b0_out) {
    const int tid = threadIdx.x;
    if (tid < 128) {
        const int sp = merge_path_wave(A, la, B, lb, tid < 64 ? d0 : d1);
        if (tid == 0) m.sp[0] = sp;
        if (tid == 64) m.sp[1] = sp;
    }
    __syncthreads();
    const int a0 = m.sp[0], a1 = m.sp[1];
    const int b0 = d0 - a0, b1 = d1 - a1;
    const int na = a1 - a0, nb = b1 - b0, n = na + nb;
    constexpr int per = T / kTileThreads;
    {
        uint64_t v[per];  // every load issued before the LDS stores
#pragma unroll
        for (int r = 0; r < per; r++) {
            const int j = tid + r * kTileThreads;
            v[r] = j < na ? A[a0 + j] : (j < n ? B[b0 + j - na] : 0ull);
        }
#pragma unroll
        for (int r = 0; r < per; r++) m.in[tid + r * kTileThreads] = v[r];
    }
    __syncthreads();
    const int diag = tid * per;
    if (diag < n) {
        int lo = max(0, diag - nb), hi = min(diag, na);
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (m.in[mid] < m.in[na + diag - 1 - mid]) lo = mid + 1;
            else hi = mid;
        }
        int ai = lo, bi = diag - lo;
        for (int q = 0; q < per && diag + q < n; q++) {
            const bool takeA = (bi >= nb) || (ai < na && m.in[ai] < m.in[na + bi]);
            if (takeA) {
                m.out[diag + q] = m.in[ai];
                if (SRC) m.src[diag + q] = a0 + ai;
                ai++;
            } else {
                m.out[diag + q] = m.in[na + bi];
                if (SRC) m.src[diag + q] = ~(b0 + bi);
                bi++;
            }
        }
    }
    __syncthreads();
    *a0_out = a0;
    *b0_out = b0;
}

// One pass of the bottom-up merge sort of the first window's keys: merges runs
// of length L pairwise, from akey (sel 0) or skey (sel 1) to the other; the
// LAST pass ends in skey and places the coordinates. A pass of a window of
// some 100,000 points is a chain of dependent loads (split searches, keys,
// the merge in LDS), so the tiles are small enough to spread it over every
// CU: 512 outputs per block.
template <bool LAST>
__global__ __launch_bounds__(kTileThreads) void k_init_merge(BatchArgs a, int L, int sel) {
    __shared__ MergeLds<kWTile> m;
    const StreamDev &S = a.s[0];
    const int len = ldc(S.W), dim = ldc(S.dim);
    const int o0 = blockIdx.x * kWTile;
    const int o1 = min(o0 + kWTile, len);
    const uint64_t *sk = sel == 0 ? S.akey : S.skey;
    const gptr<uint64_t> dk = gl(sel == 0 ? ldc(S.skey) : ldc(S.akey));
    const long long L2 = 2ll * L;
    const int base = (int)((o0 / L2) * L2);
    const int la = min(L, len - base);
    const int lb = min(L, len - base - la);
    int a0, b0;
    merge_tile<kWTile, false>(sk + base, la, sk + base + la, lb, o0 - base, o1 - base, m, &a0, &b0);
#pragma unroll
    for (int r = 0; r < kWTile / kTileThreads; r++) {
        const int i = threadIdx.x + r * kTileThreads;
        if (i >= o1 - o0) break;
        if (LAST) init_place(S, gl(a.io1.in), o0 + i, m.out[i], dim);
        else dk[o0 + i] = m.out[i];
    }
}

// ---------------------------------------------------------------------------
// window update: merge the survivors with the sorted stride

// merge(survivors, sorted stride) -> window, plus cell starts per tile
// (thrust::merge at thrust_helper.cu:47-50 and the run starts of
// compute_offsets_of_cells, aabb.cu:377-395).
__global__ __launch_bounds__(kTileThreads) void k_merge_final(BatchArgs a) {
    __shared__ MergeLds<kWTile> m;
    __shared__ int lds4[4];
    const int g = blockIdx.x;
    const int s = find_stream_c(a.pre_wtile, a.n, g);
    const StreamDev &S = a.s[s];
    const int tile = g - ldc(a.pre_wtile[s]);
    const int o0 = tile * kWTile, o1 = min(o0 + kWTile, S.W);
    const int la = S.W - S.S, lb = S.S;
    const uint64_t *B = S.bkey1;
    int a0, b0;
    merge_tile(S.akey, la, B, lb, o0, o1, m, &a0, &b0);
    if (threadIdx.x == 0) {
        uint64_t pk = 0;
        if (a0 > 0) pk = S.akey[a0 - 1];
        if (b0 > 0 && B[b0 - 1] > pk) pk = B[b0 - 1];
        m.pred = pk;
    }
    __syncthreads();
    const int dim = S.dim, sb = S.slot_bits;
    constexpr int per = kWTile / kTileThreads;
    float cx[per], cy[per], cz[per];  // every gather issued before the stores
#pragma unroll
    for (int r = 0; r < per; r++) {
        const int i = threadIdx.x + r * kTileThreads;
        const int sidx = i < o1 - o0 ? m.src[i] : 0;
        const bool fromA = sidx >= 0;
        const int j = fromA ? sidx : ~sidx;
        const float *px = fromA ? S.ax : S.bx1, *py = fromA ? S.ay : S.by1, *pz = fromA ? S.az : S.bz1;
        cx[r] = px[j];
        cy[r] = dim > 1 ? py[j] : 0.f;
        cz[r] = dim > 2 ? pz[j] : 0.f;
    }
    int starts = 0;
#pragma unroll
    for (int r = 0; r < per; r++) {
        const int i = threadIdx.x + r * kTileThreads;
        if (i < o1 - o0) {
            const uint64_t key = m.out[i];
            S.skey[o0 + i] = key;
            S.sx[o0 + i] = cx[r];
            if (dim > 1) S.sy[o0 + i] = cy[r];
            if (dim > 2) S.sz[o0 + i] = cz[r];
            const uint64_t prev = i > 0 ? m.out[i - 1] : m.pred;
            starts += (o0 + i == 0) || ((key >> sb) != (prev >> sb));
        }
    }
    starts = block_sum(starts, lds4);
    if (threadIdx.x == 0) S.tile_b[tile] = starts;
}

// Cell table: ordered compaction of run starts -> cstart/ckey and position ->
// cell. Replaces compute_offsets_of_cells + thrust_sort
// (aabb.cu:377-410, thrust_helper.cu:16-19): the order comes from the scan,
// so no sort and no host round trip (dbscan.cpp:549) are needed.
__global__ __launch_bounds__(kTileThreads) void k_cells(BatchArgs a) {
    __shared__ int lds4[4];
    const int g = blockIdx.x;
    const int s = find_stream_c(a.pre_wtile, a.n, g);
    const StreamDev &S = a.s[s];
    const int tile = g - ldc(a.pre_wtile[s]);
    const int ntile = ldc(a.pre_wtile[s + 1]) - ldc(a.pre_wtile[s]);
    const int p0 = tile * kWTile;
    const int sb = S.slot_bits;
    constexpr int per = kWTile / kTileThreads;
    uint64_t kc[per], kp[per];  // keys of each position and its predecessor, loaded up front
#pragma unroll
    for (int r = 0; r < per; r++) {
        const int p = p0 + r * kTileThreads + threadIdx.x;
        kc[r] = p < S.W ? S.skey[p] : 0ull;
        kp[r] = (p < S.W && p > 0) ? S.skey[p - 1] : 0ull;
    }
    int part = 0;
    for (int t = threadIdx.x; t < tile; t += kTileThreads) part += S.tile_b[t];
    const int base = block_sum(part, lds4);
    int run = 0;
#pragma unroll
    for (int r = 0; r < per; r++) {
        const int p = p0 + r * kTileThreads + threadIdx.x;
        const bool valid = p < S.W;
        uint64_t ck = 0;
        bool f = false;
        if (valid) {
            ck = kc[r] >> sb;
            f = (p == 0) || (ck != (kp[r] >> sb));
        }
        int tot;
        const int rank = block_rank_flags(f, &tot, lds4);
        if (valid) {
            S.pcell[p] = base + run + rank + (f ? 1 : 0) - 1;
        }
        if (f) {
            const int c = base + run + rank;
            S.cstart[c] = p;
            S.ckey[c] = ck;
        }
        run += tot;
    }
    if (tile == ntile - 1 && threadIdx.x == 0) {
        const int total = base + run;
        S.mut->ncell = total;
        S.cstart[total] = S.W;
    }
}

// ---------------------------------------------------------------------------
// window update of small streams: one block per stream, the window's keys in LDS

// Inclusive prefix sum over a wave's lanes, in registers (all lanes active).
__device__ __forceinline__ int wave_scan(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast 15, 31
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
    return x;
}

// Flags of a block in position order (round r, wave, lane), counted per round
// and wave in cnt[r * 16 + wave]: before[r] = the flags before this wave's of
// round r; returns the total. Every wave scans the PER * 16 <= 128 counts, two
// per lane, for itself. Starts with the barrier that the counts need.
template <int PER>
__device__ __forceinline__ int small_scan(const int *cnt, int wv, int (&before)[PER]) {
    __syncthreads();
    const int lane = lane_id();
    const int c0 = 2 * lane < PER * 16 ? cnt[2 * lane] : 0, c1 = 2 * lane < PER * 16 ? cnt[2 * lane + 1] : 0;
    const int x = wave_scan(c0 + c1);
    const int e = (wv & 1) ? x - c1 : x - c0 - c1;
#pragma unroll
    for (int r = 0; r < PER; r++) before[r] = __builtin_amdgcn_readlane(e, r * 8 + (wv >> 1));
    return __builtin_amdgcn_readlane(x, 63);
}

// Number of the len <= 4 * q sorted keys a[0, len) in LDS below key (q a power
// of four; last: the last index of a that may be read). Three probes a step:
// a step is one LDS latency, and the latency is what it costs.
__device__ __forceinline__ int small_below(const uint64_t *a, int len, int last, int q, uint64_t key) {
    auto below = [&](int i) { return ((i < len) & (a[min(i, last)] < key)) ? 1 : 0; };
    int n = q * (below(q - 1) + below(2 * q - 1) + below(3 * q - 1) + below(4 * q - 1));
    for (q >>= 2; q > 0; q >>= 2) n += q * (below(n + q - 1) + below(n + 2 * q - 1) + below(n + 3 * q - 1));
    return n;
}

// The whole update of a stream of up to PER * 1024 points and kSmallS points a
// stride: what k_sort_expire, k_rank, k_merge_final and k_cells do together.
// At these sizes each of those is a launch and a chain of a few dependent
// round trips through memory; here the chain is the window's keys and the
// stride in, then LDS, then the new window out. A whole slide of 1,000 points
// and strides of 10 in 2-D, resident on the device: 42 us with the separate
// kernels, 32 us so; 4,000 and 400: 46.5 and 41.5 us, 64 such streams of 2,000:
// 71 and 60 us. Past 4,096 points one block's share of the work is the longer
// (8,000 and 800: 48 and 51 us with eight positions per thread). A survivor's
// place is its
// rank among the survivors plus the stride keys below it, a stride key's its
// rank in the sorted stride plus the survivors below it.
template <int PER>
__global__ __launch_bounds__(kSmallThreads) void k_update_small(BatchArgs a) {
    __shared__ uint64_t sk[PER * kSmallThreads];  // survivors' keys, then the window's
    __shared__ uint64_t bk[kSmallS + 8];          // the stride's keys, sorted, then ~0
    __shared__ float bc[3][kSmallS];              // its coordinates, as they came
    __shared__ int cnt[2][PER * 16];
    static_assert(kSmallS == kSmallThreads && kSmallThreads == 1024 && PER <= 4, "");
    const int s = blockIdx.x, tid = threadIdx.x, lane = lane_id(), wv = uni(tid >> 6);
    const StreamDev &S = a.s[s];
    const int W = ldc(S.W), SS = ldc(S.S), dim = ldc(S.dim), sb = ldc(S.slot_bits);
    const gptr<uint64_t> skey = gl(ldc(S.skey));
    const gptr<float> sx = gl(ldc(S.sx)), sy = gl(ldc(S.sy)), sz = gl(ldc(S.sz));
    const uint32_t sm = (uint32_t)((1ull << sb) - 1ull);
    const int lo_slot = ldc(ldc(S.mut)->u) * SS;
    const uint64_t lower = (1ull << lane) - 1ull;
    const IO io = a.use_io1 ? a.io1 : a.io[s];
    // the stride and the window, every load issued before the sort
    const gptr<const float> in = gl(io.in) + (size_t)min(tid, SS - 1) * dim;
    const float n0 = in[0], n1 = dim > 1 ? in[1] : 0.f, n2 = dim > 2 ? in[2] : 0.f;
    uint64_t key[PER];
    float cx[PER], cy[PER], cz[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const int p = min(r * kSmallThreads + tid, W - 1);
        key[r] = skey[p];
        cx[r] = sx[p];
        cy[r] = dim > 1 ? sy[p] : 0.f;
        cz[r] = dim > 2 ? sz[p] : 0.f;
    }
    bc[0][tid] = n0;
    bc[1][tid] = n1;
    bc[2][tid] = n2;
    uint64_t v[1] = {tid < SS ? (cell_key_g(key_grid(S), n0, n1, n2) << sb) | (uint64_t)(lo_slot + tid) : ~0ull};
    // the stride sorted: runs of 64 in each wave's lanes, then merged pairwise,
    // each key moving to its place in its run plus the partner run's keys below
    // it; the padding keys stay last
    if (wv * 64 < SS) bitonic_sort_regs<64, 1>(v, nullptr, lane);
    bk[tid] = v[0];
    if (tid < 8) bk[kSmallS + tid] = ~0ull;
    for (int L = 64, q = 16; L < SS; L <<= 1) {
        __syncthreads();
        v[0] = bk[tid];
        const int run = tid & ~(L - 1), other = run ^ L;
        int to = (run & other) + (tid - run);
        if (wv * 64 < SS) to += small_below(bk + other, min(max(SS - other, 0), L), kSmallS - 1 - other, q, v[0]);
        __syncthreads();
        if (tid < SS) bk[to] = v[0];
        if (4 * q < 2 * L) q <<= 2;
    }
    // survivors in order
    int at[PER], before[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const int slot = (int)((uint32_t)key[r] & sm);
        const bool f = r * kSmallThreads + tid < W && (slot < lo_slot || slot >= lo_slot + SS);
        const uint64_t m = __ballot(f);
        at[r] = f ? __popcll(m & lower) : -1;
        if (lane == 0) cnt[0][r * 16 + wv] = __popcll(m);
    }
    small_scan<PER>(cnt[0], wv, before);  // from its barrier on bk is whole
    v[0] = bk[tid];
    const int ns = W - SS;
#pragma unroll
    for (int r = 0; r < PER; r++)
        if (at[r] >= 0) {
            at[r] += before[r];
            sk[at[r]] = key[r];
        }
    // Survivors' places. A wave's 64 window keys rise with the lane, so the
    // stride keys between the first and the last bound every lane's count; few
    // of them as a rule, compared one by one.
    const uint64_t sample = bk[lane * 16 + 15];
    uint64_t near[PER];
    int nb[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const uint64_t k0 = readlane64(key[r], 0), k1 = readlane64(key[r], 63);
        const int b0 = 16 * __popcll(__ballot(sample < k0)), b1 = 16 * __popcll(__ballot(sample < k1));
        nb[r] = lane < 32 ? b0 : b1;
        near[r] = bk[min(nb[r] + (lane & 15), kSmallS - 1)];
    }
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const uint64_t k0 = readlane64(key[r], 0), k1 = readlane64(key[r], 63);
        const uint64_t bel = __ballot(near[r] < (lane < 32 ? k0 : k1));
        // past the array's end (every key below) the last key repeats
        const int lo = min(__builtin_amdgcn_readlane(nb[r], 0) + __popcll(bel & 0xffffull), kSmallS);
        const int hi = min(__builtin_amdgcn_readlane(nb[r], 63) + __popcll(bel & 0xffff00000000ull), kSmallS);
        int n = lo;
        if (hi - lo <= 8) {  // keys past hi are above every lane's
            uint64_t t[8];
#pragma unroll
            for (int j = 0; j < 8; j++) t[j] = bk[lo + j];
#pragma unroll
            for (int j = 0; j < 8; j++) n += t[j] < key[r] ? 1 : 0;
        } else {
            n += small_below(bk + lo, hi - lo, hi - lo, hi - lo <= 64 ? 16 : 256, key[r]);
        }
        if (at[r] >= 0) at[r] += n;
    }
    __syncthreads();  // sk holds the survivors
    int bat = -1;
    if (wv * 64 < SS) {
        bat = tid + small_below(sk, ns, PER * kSmallThreads - 1, PER == 1 ? 256 : 1024, v[0]);
        if (tid >= SS) bat = -1;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PER; r++)
        if (at[r] >= 0) {
            sk[at[r]] = key[r];
            skey[at[r]] = key[r];
            sx[at[r]] = cx[r];
            if (dim > 1) sy[at[r]] = cy[r];
            if (dim > 2) sz[at[r]] = cz[r];
        }
    if (bat >= 0) {
        const int j = (int)((uint32_t)v[0] & sm) - lo_slot;
        sk[bat] = v[0];
        skey[bat] = v[0];
        sx[bat] = bc[0][j];
        if (dim > 1) sy[bat] = bc[1][j];
        if (dim > 2) sz[bat] = bc[2][j];
    }
    __syncthreads();
    // cell table
    uint64_t prev[PER];
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const int p = r * kSmallThreads + tid;
        key[r] = sk[min(p, W - 1)];
        prev[r] = sk[max(min(p, W) - 1, 0)];
    }
    uint32_t starts = 0;  // bit r: position r * 1024 + tid starts a cell
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const int p = r * kSmallThreads + tid;
        const bool f = p < W && (p == 0 || (key[r] >> sb) != (prev[r] >> sb));
        const uint64_t m = __ballot(f);
        at[r] = __popcll(m & lower) + (f ? 1 : 0) - 1;
        starts |= (uint32_t)f << r;
        if (lane == 0) cnt[1][r * 16 + wv] = __popcll(m);
    }
    const int ncell = small_scan<PER>(cnt[1], wv, before);
    const gptr<int32_t> pcell = gl(ldc(S.pcell)), cstart = gl(ldc(S.cstart));
    const gptr<uint64_t> ckey = gl(ldc(S.ckey));
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const int p = r * kSmallThreads + tid;
        if (p >= W) continue;
        const int c = at[r] + before[r];
        pcell[p] = c;
        if ((starts >> r) & 1u) {
            cstart[c] = p;
            ckey[c] = key[r] >> sb;
        }
    }
    if (tid == 0) {
        ldc(S.mut)->ncell = ncell;
        cstart[ncell] = W;
    }
}

// ---------------------------------------------------------------------------
// stencil rows: for every cell and every row of its (2k+1)^dim stencil, the
// contiguous range of window positions holding that row's cells. A row varies
// the last used axis, whose key stride is 1 (unused axes have extent 1 and
// index 0), so its cells are the cells with keys in [lo, hi] = the target
// column's keys at zlo..zhi, consecutive in the sorted cell table. For one
// row offset, lo and hi rise with the cell's own key (the target column is
// the cell's column shifted by a constant), so one wave serves 64 consecutive
// cells: a cooperative search brackets the tile's bounds in the cell table,
// the bracket is staged in LDS and each lane binary-searches its own bounds
// there. No hashing, and a few memory round trips per 64 (cell, row) items.

constexpr int kRowTile = 64;    // cells per row-kernel item (one wave)
constexpr int kRowCap = 192;    // bracket cells staged in LDS per wave
constexpr int kRowWaves = kTileThreads / 64;

// The stencil rows of a stream's cells, (first, end) positions as one word
// each: group by group of row_w rows, which one item of the row kernel writes
// (the 2k+1 rows of one offset on the first axis in 3-D, all rows else), the
// groups' cells one after the other. An item's words are then adjacent: with
// all rows of a cell adjacent (a cell's 25 words), each of its stores was 64
// requests to L2, 18.7 M for the 24 M rows of the 64-stream batch. Row kernel
// with those and now: 64 streams 123 and 111 us, one million points 66 and 53.
// The stores put in order through LDS first: 117 and 53.
template <class T>
struct RowTable {
    gptr<T> p;
    int W, w, div;
    __device__ __forceinline__ explicit RowTable(const StreamDev &S)
        : p(gl((T *)ldc(S.rows))), W(ldc(S.W)), w(ldc(S.row_w)), div(ldc(S.row_div)) {}
    // row r of every cell c is at of(c)[row(r)]; r / w by multiplication, exact for r < kMaxRows
    __device__ __forceinline__ int row(int r) const {
        const int g = (r * div) >> 8;
        return g * (W * w - w) + r;
    }
    __device__ __forceinline__ gptr<T> of(int c) const { return p + (size_t)c * w; }
    __device__ __forceinline__ T at(int c, int r) const { return of(c)[row(r)]; }
};

// Wave-uniform view of one stream for the row kernel (scalar descriptor
// loads, global addressing).
struct RowsView {
    gptr<const uint64_t> ckey;
    gptr<const int32_t> cstart;
    RowTable<uint64_t> rows;
    gptr<uint8_t> cflag;
    int64_t n0, n1, n2;
    int k, R, dim, min_pts, dense_ok, ncell;
};

__device__ __forceinline__ RowsView rows_view(const StreamDev &S) {
    RowsView v{.rows = RowTable<uint64_t>(S)};
    v.ckey = gl(ldc(S.ckey));
    v.cstart = gl(ldc(S.cstart));
    v.cflag = gl(ldc(S.cflag));
    v.n0 = ldc(S.n[0]);
    v.n1 = ldc(S.n[1]);
    v.n2 = ldc(S.n[2]);
    v.k = ldc(S.k);
    v.R = ldc(S.R);
    v.dim = ldc(S.dim);
    v.min_pts = ldc(S.min_pts);
    v.dense_ok = ldc(S.dense_ok);
    v.ncell = ldc(ldc(S.mut)->ncell);  // written by the cell-table kernel
    return v;
}

// Ranks (number of keys below) of two wave-uniform keys in the sorted
// ckey[0, n), n >= 1: two 64-ary searches in lockstep, one probe per lane per
// key and round, then a last round over at most 64 keys.
__device__ __forceinline__ void wave_rank2(gptr<const uint64_t> ckey, int n, uint64_t k1, uint64_t k2, int *r1,
                                           int *r2) {
    const int lane = lane_id();
    int lo1 = 0, hi1 = n, lo2 = 0, hi2 = n;  // rank in [lo, hi]
    while (hi1 - lo1 > 64 || hi2 - lo2 > 64) {
        const int s1 = hi1 - lo1, s2 = hi2 - lo2;
        const int p1 = lo1 + (int)((long long)(lane + 1) * s1 / 65);  // in [lo, hi) when s > 64
        const int p2 = lo2 + (int)((long long)(lane + 1) * s2 / 65);
        const uint64_t v1 = ckey[min(p1, n - 1)];
        const uint64_t v2 = ckey[min(p2, n - 1)];
        if (s1 > 64) {
            const int c = __popcll(__ballot(v1 < k1));  // the probes below k1 are a prefix of the lanes
            const int nlo = c > 0 ? __builtin_amdgcn_readlane(p1, c - 1) + 1 : lo1;
            hi1 = c < 64 ? __builtin_amdgcn_readlane(p1, c) : hi1;
            lo1 = nlo;
        }
        if (s2 > 64) {
            const int c = __popcll(__ballot(v2 < k2));
            const int nlo = c > 0 ? __builtin_amdgcn_readlane(p2, c - 1) + 1 : lo2;
            hi2 = c < 64 ? __builtin_amdgcn_readlane(p2, c) : hi2;
            lo2 = nlo;
        }
    }
    const bool b1 = lo1 + lane < hi1 && ckey[lo1 + lane] < k1;
    const bool b2 = lo2 + lane < hi2 && ckey[lo2 + lane] < k2;
    *r1 = lo1 + __popcll(__ballot(b1));
    *r2 = lo2 + __popcll(__ballot(b2));
}

// First index in sorted a[0, n) (n >= 1) whose key is >= key.
template <class P>
__device__ __forceinline__ int lower_index(P a, int n, uint64_t key) {
    int base = 0;
    while (n > 1) {
        const int half = n >> 1;
        if (a[base + half] < key) base += half;
        n -= half;
    }
    return base + (a[base] < key ? 1 : 0);
}

// Cell classes (written once per slide by k_rows):
//   kCellSafe  - the grid is dense-safe (k*k > dim: any two points of one
//                cell are closer than eps) and the cell is interior; border
//                cells may hold points clamped in from outside the grid
//                bounds, which the side-length argument does not cover.
//   kCellDense - safe and holding >= min_pts points: all of them are core.
__device__ __forceinline__ uint8_t cell_class(const RowsView &V, int64_t i0, int64_t i1, int64_t i2, int c) {
    if (!V.dense_ok) return 0;
    if (i0 <= 0 || i0 >= V.n0 - 1) return 0;
    if (V.dim > 1 && (i1 <= 0 || i1 >= V.n1 - 1)) return 0;
    if (V.dim > 2 && (i2 <= 0 || i2 >= V.n2 - 1)) return 0;
    const int cnt = V.cstart[c + 1] - V.cstart[c];
    return cnt >= V.min_pts ? (kCellSafe | kCellDense) : kCellSafe;
}

// Storage order of a cell's stencil rows: nearest first, group by group. An
// offset d in [-k, k] ranks as 0, -1, +1, -2, +2, ... (|d| first, the
// negative side first). In 3-D row (d1, d2) - offsets on the first two axes -
// is stored at rank(d1) * (2k+1) + rank(d2): the rows of one first-axis
// offset (one rows-kernel item) stay adjacent, and the groups come nearest
// first. In 2-D row d1 is stored at rank(d1). The centre row is row 0. The
// count kernels walk rows in storage order, so a query's count meets the
// rows holding most of its neighbours first and reaches min_pts sooner; the
// other consumers need no particular order.
__device__ __forceinline__ int offset_rank(int d) { return d == 0 ? 0 : 2 * (d < 0 ? -d : d) - (d < 0 ? 1 : 0); }

// Rows per item: in 3-D one item holds the 2k+1 rows of one offset o0 on the
// first axis (o1 = -k..k on the second), whose target columns are adjacent,
// so one bracket serves all of them; in 2-D and 1-D an item is one row.
__device__ __forceinline__ int rows_groups(int dim, int k, int R) { return dim == 3 ? 2 * k + 1 : R; }

// Item g of tile t: the rows with offset o0 = g - k (3-D), or row g; the
// 64 cells of the tile one per lane. The item holding the centre row also
// records each cell's class. lk/lc: this wave's LDS. NS >= the item's row
// count (2k + 1 <= 7 in 3-D, 1 otherwise): the lower bounds of all its rows
// in the staged bracket are searched in lockstep, one LDS round per step for
// all of them.
template <int NS>
__device__ __forceinline__ void rows_tile(const RowsView &V, int t, int g, uint64_t *lk, int32_t *lc) {
    const int lane = lane_id();
    const int c = t * kRowTile + lane;
    const bool cv = c < V.ncell;
    const uint64_t ck = cv ? V.ckey[c] : 0ull;
    int64_t q, i0, i1, i2;
    divmod_key(ck, V.n2, &q, &i2);
    divmod_key((uint64_t)q, V.n1, &i0, &i1);
    const int k = V.k, w = 2 * k + 1;
    const int nsub = V.dim == 3 ? w : 1;
    // offsets of the item's rows (uniform): o0 fixed, o1 over [o1lo, o1lo + nsub)
    int o0 = 0, o1lo = 0;
    if (V.dim == 3) {
        o0 = g - k;
        o1lo = -k;
    } else if (V.dim == 2) {
        o0 = g - k;
    }
    int64_t zc, zn;
    if (V.dim == 3) {
        zc = i2;
        zn = V.n2;
    } else if (V.dim == 2) {
        zc = i1;
        zn = V.n1;
    } else {
        zc = i0;
        zn = V.n0;
    }
    // a bracket of the cell table holding every row bound of the item: the
    // bounds rise with the lane and with o1, and lo >= key + shift - k,
    // hi <= key + shift + k
    const uint64_t cvm = __ballot(cv);  // non-empty: t < ceil(ncell / 64)
    const int64_t klo = (int64_t)readlane64(ck, __ffsll((unsigned long long)cvm) - 1);
    const int64_t khi = (int64_t)readlane64(ck, 63 - __clzll((long long)cvm));
    const int64_t sh_lo = ((int64_t)o0 * V.n1 + o1lo) * V.n2, sh_hi = ((int64_t)o0 * V.n1 + o1lo + nsub - 1) * V.n2;
    const int64_t bmin = klo + sh_lo - k, bmax = khi + sh_hi + k;
    int b0 = 0, b1 = 0;
    if (bmax >= 0) wave_rank2(V.ckey, V.ncell, (uint64_t)max(bmin, (int64_t)0), (uint64_t)bmax + 1, &b0, &b1);
    const int B = b1 - b0;
    const bool staged = B > 0 && B <= kRowCap;
    if (staged) {
        for (int i = lane; i < B; i += 64) lk[i] = V.ckey[b0 + i];
        for (int i = lane; i <= B; i += 64) lc[i] = V.cstart[b0 + i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // key bounds of each row: the target column's keys at zlo..zhi
    uint64_t lo[NS], hi1[NS];
    bool ok[NS];
#pragma unroll
    for (int j = 0; j < NS; j++) {
        const int o1 = o1lo + j;
        bool okj = cv && j < nsub;
        if (V.dim == 3) okj = okj && i0 + o0 >= 0 && i0 + o0 < V.n0 && i1 + o1 >= 0 && i1 + o1 < V.n1;
        else if (V.dim == 2) okj = okj && i0 + o0 >= 0 && i0 + o0 < V.n0;
        const int64_t colbase = (int64_t)ck - zc + ((int64_t)o0 * V.n1 + (V.dim == 3 ? o1 : 0)) * V.n2;
        lo[j] = (uint64_t)(colbase + (zc - k < 0 ? 0 : zc - k));
        hi1[j] = (uint64_t)(colbase + (zc + k >= zn ? zn - 1 : zc + k)) + 1ull;
        ok[j] = okj;
    }
    int f[NS], e[NS];  // first and end positions of each row's cells in the bracket
    if (staged) {
#pragma unroll
        for (int j = 0; j < NS; j++) f[j] = e[j] = 0;
        for (int n = B; n > 1;) {
            const int half = n >> 1;
#pragma unroll
            for (int j = 0; j < NS; j++) {
                if (lk[f[j] + half] < lo[j]) f[j] += half;
                if (lk[e[j] + half] < hi1[j]) e[j] += half;
            }
            n -= half;
        }
#pragma unroll
        for (int j = 0; j < NS; j++) {
            f[j] += lk[f[j]] < lo[j] ? 1 : 0;
            e[j] += lk[e[j]] < hi1[j] ? 1 : 0;
        }
    }
#pragma unroll
    for (int j = 0; j < NS; j++) {
        if (j >= nsub) break;
        uint64_t row = 0ull;
        if (ok[j] && B > 0) {
            if (staged) {
                if (f[j] < e[j]) row = (uint64_t)(uint32_t)lc[f[j]] | ((uint64_t)(uint32_t)lc[e[j]] << 32);
            } else {
                const int fg = b0 + lower_index(V.ckey + b0, B, lo[j]);
                const int eg = b0 + lower_index(V.ckey + b0, B, hi1[j]);
                if (fg < eg) row = (uint64_t)(uint32_t)V.cstart[fg] | ((uint64_t)(uint32_t)V.cstart[eg] << 32);
            }
        }
        // stencil row number: nearest groups and rows first, the centre row 0
        const int r = V.dim == 3 ? offset_rank(o0) * w + offset_rank(o1lo + j) : (V.dim == 2 ? offset_rank(o0) : 0);
        if (cv) {
            V.rows.of(c)[V.rows.row(r)] = row;
            if (r == 0) {
                V.cflag[c] = cell_class(V, i0, i1, i2, c);
            }
        }
    }
    if (staged) __builtin_amdgcn_wave_barrier();  // reads done before the next item's stores
}

// Persistent: walks the device-side list of (stream, 64-cell tile, row group)
// items, one per wave. One block more than the walk needs publishes the
// per-stream prefixes of cells and of cell tiles for the later kernels, over
// all its threads.
__global__ __launch_bounds__(kTileThreads) void k_rows(BatchArgs a) {
    __shared__ long long pre[kMaxBatch + 1];
    __shared__ long long tmp4[4];
    __shared__ uint64_t lkey[kRowWaves][kRowCap];
    __shared__ int32_t lcs[kRowWaves][kRowCap + 1];
    const int nb = gridDim.x - 1;  // blocks of the walk
    if ((int)blockIdx.x == nb) {
        block_stream_prefix(a.n, pre, tmp4, [&](int i) { return (long long)a.s[i].mut->ncell; });
        for (int i = threadIdx.x; i <= a.n; i += kTileThreads) a.cell_pre[i] = (int32_t)pre[i];
        __syncthreads();
        block_stream_prefix(a.n, pre, tmp4, [&](int i) {
            return (long long)((a.s[i].mut->ncell + a.cell_tile - 1) / a.cell_tile);
        });
        for (int i = threadIdx.x; i <= a.n; i += kTileThreads) a.ctile_pre[i] = (int32_t)pre[i];
        return;
    }
    block_stream_prefix(a.n, pre, tmp4, [&](int i) {
        const StreamDev &S = a.s[i];
        return (long long)((S.mut->ncell + kRowTile - 1) / kRowTile) * rows_groups(S.dim, S.k, S.R);
    });
    const long long total = pre[a.n];
    const int wv = uni(threadIdx.x >> 6);
    for (long long wi = (long long)blockIdx.x * kRowWaves + wv; wi < total; wi += (long long)nb * kRowWaves) {
        const int s = uni(find_stream(pre, a.n, wi));
        const RowsView V = rows_view(a.s[s]);
        const int local = uni((int)(wi - pre[s]));
        const int G = rows_groups(V.dim, V.k, V.R);
        const int t = local / G;
        if (V.dim == 3) rows_tile<7>(V, t, local - t * G, lkey[wv], lcs[wv]);
        else rows_tile<1>(V, t, local - t * G, lkey[wv], lcs[wv]);
    }
}

// ---------------------------------------------------------------------------
// cell-parallel neighbourhood kernels: one wave per (stream, cell), walking
// the device-side cell list in a persistent loop. The candidates of a cell
// are the concatenation of its stencil rows; lanes 0..R-1 hold one row each.

struct ChunkCtx {
    int s, p0, p1;
};

__device__ __forceinline__ ChunkCtx chunk_of(const BatchArgs &a, int g) {
    ChunkCtx x;
    x.s = find_stream_c(a.pre_chunk, a.n, g);
    const int W = a.s[x.s].W;
    x.p0 = (g - ldc(a.pre_chunk[x.s])) * kChunk;
    x.p1 = min(x.p0 + kChunk, W);
    return x;
}

// Wave-uniform view of one stream for the cell-parallel kernels. The
// descriptor is read with scalar loads (no kernel writes it during a launch)
// and the arrays are addressed as global memory, so the per-lane accesses
// are global loads and stores off a scalar base.
struct CellView {
    gptr<const float> sx, sy, sz;
    gptr<const uint64_t> skey;
    gptr<const int32_t> cstart;
    RowTable<const uint64_t> rows;
    gptr<const uint8_t> cflag;
    gptr<const int32_t> pcell;
    gptr<uint8_t> flags;
    gptr<int32_t> fcore;
    gptr<uint64_t> uf;
    int W, R, dim, min_pts;
    uint32_t smask;
    float eps2;
};

__device__ __forceinline__ CellView cell_view(const StreamDev &S) {
    CellView v{.rows = RowTable<const uint64_t>(S)};
    v.sx = gl(ldc(S.sx));
    v.sy = gl(ldc(S.sy));
    v.sz = gl(ldc(S.sz));
    v.skey = gl(ldc(S.skey));
    v.cstart = gl(ldc(S.cstart));
    v.cflag = gl(ldc(S.cflag));
    v.pcell = gl(ldc(S.pcell));
    v.flags = gl(ldc(S.flags));
    v.fcore = gl(ldc(S.fcore));
    v.uf = gl(ldc(S.uf));
    v.W = ldc(S.W);
    v.R = ldc(S.R);
    v.dim = ldc(S.dim);
    v.min_pts = ldc(S.min_pts);
    v.smask = (uint32_t)((1ull << ldc(S.slot_bits)) - 1ull);
    v.eps2 = ldc(S.eps2);
    return v;
}

__device__ __forceinline__ int vslot(const CellView &V, int pos) { return (int)((uint32_t)V.skey[pos] & V.smask); }

constexpr int kRowGroup = 5;  // stencil rows fetched together

// Query ownership of a block of a point-parallel kernel with LPQ lanes per
// query: block g covers chunk g / LPQ; each query is served by LPQ adjacent
// lanes that split its stencil rows. More lanes per query shorten each
// thread's chain of dependent loads when a launch has few queries.
template <int LPQ>
struct QueryLane {
    ChunkCtx x;
    int p;    // window position of the query (may be >= x.p1: idle)
    int sub;  // 0..LPQ-1
};

template <int LPQ>
__device__ __forceinline__ QueryLane<LPQ> query_lane(const BatchArgs &a, int vb) {
    QueryLane<LPQ> q;
    const int chunk = vb / LPQ, part = vb % LPQ;
    q.x = chunk_of(a, chunk);
    q.sub = lane_id() % LPQ;
    q.p = q.x.p0 + part * (64 / LPQ) + lane_id() / LPQ;
    return q;
}

template <int LPQ>
__device__ __forceinline__ int group_sum(int v) {
#pragma unroll
    for (int o = 1; o < LPQ; o <<= 1) v += xor_lane(v, o);
    return v;
}

template <int LPQ>
__device__ __forceinline__ int group_min(int v) {
#pragma unroll
    for (int o = 1; o < LPQ; o <<= 1) v = min(v, xor_lane(v, o));
    return v;
}

// ---------------------------------------------------------------------------
// cell-parallel neighbourhood kernels: one wave per cell. The lanes hold 64
// of the cell's stencil candidates at a time - consecutive positions of its
// rows, so the loads coalesce and each candidate is read once per cell rather
// than once per query - and every query of the cell is tested against all of
// them with one ballot.

constexpr int kCellWaves = 4;  // waves (cells) per block

__device__ __forceinline__ float lane_f(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Work counters of one wave (uniform values), flushed to the per-stream
// totals with one atomic per counter when the wave moves to another stream
// or ends. The cell kernels are instantiated with WaveStats when counting is
// on (a.stats non-null) and with NoStats otherwise, so that normal launches
// carry no counting instructions.
struct WaveStats {
    int s = -1;
    unsigned long long v[kNumStats] = {};
    __device__ __forceinline__ void add(int k, unsigned long long x) { v[k] += x; }
};

struct NoStats {
    __device__ __forceinline__ void add(int, unsigned long long) {}
};

__device__ __forceinline__ void stats_flush(const BatchArgs &, NoStats &) {}
__device__ __forceinline__ void stats_stream(const BatchArgs &, NoStats &, int) {}

__device__ __forceinline__ void stats_flush(const BatchArgs &a, WaveStats &w) {
    if (a.stats && w.s >= 0 && lane_id() == 0)
        for (int k = 0; k < kNumStats; k++)
            if (w.v[k]) atomicAdd(a.stats + (size_t)w.s * kNumStats + k, w.v[k]);
    for (int k = 0; k < kNumStats; k++) w.v[k] = 0;
}

__device__ __forceinline__ void stats_stream(const BatchArgs &a, WaveStats &w, int s) {
    if (s != w.s) {
        stats_flush(a, w);
        w.s = s;
    }
}

// A cell's stencil candidates, 64 at a time. Lane r < R holds stencil row r:
// its first window position and its length. A walk in scalar registers opens
// the non-empty rows in order (a ballot mask; each row read with readlane)
// and gives every lane the position of its candidate, which belongs to the
// last row opened at or before it - no cross-lane search per chunk.
struct RowWalk {
    int rx = 0, len = 0;  // lane r: row r
    uint64_t rest = 0;    // non-empty rows not opened yet (uniform)
    int acc = 0;          // first candidate of the next row to open (uniform)
    int base = 0;         // position minus candidate index in the last row opened (uniform)
};

// Row r of cell A in lane r < R (int2 as one word), 0 in the other lanes.
__device__ __forceinline__ uint64_t row_word(const CellView &V, int A) {
    const int lane = lane_id();
    return lane < V.R ? V.rows.at(A, lane) : 0ull;
}

// The walk over rows (row_word), each cut at window position `limit`.
__device__ __forceinline__ RowWalk row_walk(uint64_t rw, int limit) {
    RowWalk w;
    w.rx = (int)(uint32_t)rw;
    w.len = max(0, min((int)(uint32_t)(rw >> 32), limit) - w.rx);
    w.rest = __ballot(w.len > 0);
    return w;
}

// Waits here for v, loaded earlier. The cell kernels issue every load that
// depends on the same thing together and then wait for all of them at once,
// so that none is moved past a branch into a round trip of its own.
template <class T>
__device__ __forceinline__ void arrived(T v) {
    asm volatile("" ::"v"(v));
}

// Opens the rows that start before jb + 64 and returns this lane's candidate
// position in chunk [jb, jb + 64); lanes past the last candidate get the last
// one. *end is the candidate count once every row is open, else INT_MAX.
// Callers stop at jb >= *end before using the position.
__device__ __forceinline__ int walk_chunk(RowWalk &w, int jb, int *end) {
    const int j = jb + lane_id();
    int base = w.base;
    while (w.rest != 0ull && w.acc < jb + 64) {
        const int r = __ffsll((unsigned long long)w.rest) - 1;
        w.rest &= w.rest - 1ull;
        const int b = __builtin_amdgcn_readlane(w.rx, r) - w.acc;
        if (j >= w.acc) base = b;
        w.base = b;
        w.acc += __builtin_amdgcn_readlane(w.len, r);
    }
    *end = w.rest != 0ull ? INT_MAX : w.acc;
    return base + min(j, *end - 1);
}

// A cell's header as each lane loaded it: run start and end, class, and
// stencil row `lane` (lanes < R). One round trip, issued ahead of its use.
struct CellHdr {
    int csv, cev, cfv;
    uint64_t rw;
};

__device__ __forceinline__ CellHdr load_hdr(const StreamDev &S, int A) {
    const gptr<const int32_t> cstart = gl((const int32_t *)ldc(S.cstart));
    const gptr<const uint8_t> cflag = gl((const uint8_t *)ldc(S.cflag));
    const RowTable<const uint64_t> rows(S);
    const int R = ldc(S.R);
    CellHdr h;
    h.csv = cstart[A];
    h.cev = cstart[A + 1];
    h.cfv = cflag[A];
    // every lane loads (no branch around the load); lanes >= R are cleared
    // where the row is used
    h.rw = rows.at(A, min(lane_id(), R - 1));
    return h;
}

// Flags of a counted point. A count that stays below min_pts is exact and
// holds the point itself, so at most one means that it has no neighbour (a
// point with a NaN or infinite coordinate has none and does not count itself):
// the output kernels write noise without reading its stencil again. 94-99% of
// the non-core points of 3-D trajectories are such, 9-63% of 2-D blobs': the
// regrouped outputs went from 163 to 139 us at 64 streams, 93 to 81 at one
// million points, 86 to 76 at 24 served streams. (A tile of 512 positions
// regrouped together instead of 64: 138, 89 and 91 us. Eight and 16 lanes a
// point instead of four: 144 and 178, 91 and 100, 101 and 128.)
__device__ __forceinline__ uint8_t count_flags(int cnt, int minpts, bool safe) {
    return cnt >= minpts ? (safe ? kFlagCore : kFlagCore | kFlagLoose) : (cnt <= 1 ? kFlagAlone : 0);
}

// A point that needs no look at its stencil to be noise. (The work counters
// cover every non-core point's stencil, so with them on all are walked.)
__device__ __forceinline__ bool known_noise(const BatchArgs &a, int flags) {
    return (flags & kFlagAlone) && !a.stats;
}

// Range count = core identification (the reference's __raygen__grid +
// __intersection__grid, dbscan.cu:155-194,250-270, and set_label,
// aabb.cu:575-587), for cell A whose header h was loaded ahead. Dense cells
// are core without counting (all pairs within eps). A cell whose whole
// stencil holds fewer than min_pts points cannot hold a core: its points are
// non-core without a distance test. Otherwise each query counts its
// neighbours, itself included, and stops once the count reaches min_pts.
// The queries and the first candidate chunk load in one round, after which
// `prefetch` issues the next cell's header, so that it arrives while this
// cell computes; each further chunk is a round of its own. `prefetch` runs
// exactly once on every path.
template <class ST, class Pre>
__device__ __forceinline__ void count_cell(const CellView &V, int A, const CellHdr &h, ST &st, Pre &&prefetch) {
    const int lane = lane_id();
    const int dim = V.dim, minpts = V.min_pts;
    const float e2 = V.eps2;
    const int cs = uni(h.csv), nA = uni(h.cev) - cs;
    const int cf = uni(h.cfv);
    if (cf & kCellDense) {
        const int rsv = vslot(V, cs);
        prefetch();
        st.add(kStatDensePoints, nA);
        const int rs = uni(rsv);
        for (int i = lane; i < nA; i += 64) V.flags[cs + i] = kFlagCore | kFlagDense;
        if (lane == 0) {
            V.fcore[A] = cs;
            V.uf[A] = ufe(rs, A);
        }
        return;
    }
    const bool safe = cf & kCellSafe;
    const RowWalk w0 = row_walk(lane < V.R ? h.rw : 0ull, INT_MAX);
    st.add(kStatQueries, nA);
    const int total = uni(wave_sum(w0.len));
    if (total < minpts) {
        // fewer candidates than min_pts: no core
        prefetch();
        for (int i = lane; i < nA; i += 64) V.flags[cs + i] = total == 1 ? kFlagAlone : 0;
        if (lane == 0) {
            V.fcore[A] = kNoCore;
            V.uf[A] = kUfNone;
        }
        return;
    }
    int fc = kNoCore, fslot = 0;
    // one block of up to 64 queries; the first block issues the prefetch
    auto block = [&](const int q0, const bool first) __attribute__((always_inline)) {
        const int nq = min(64, nA - q0);
        const int pq = cs + q0 + min(lane, nq - 1);
        const float qx = V.sx[pq];
        const float qy = dim > 1 ? V.sy[pq] : 0.f;
        const float qz = dim > 2 ? V.sz[pq] : 0.f;
        const int qslot = vslot(V, pq);
        RowWalk w = w0;
        int end;
        int pos = walk_chunk(w, 0, &end);
        const float cx = V.sx[pos];
        const float cy = dim > 1 ? V.sy[pos] : 0.f;
        const float cz = dim > 2 ? V.sz[pos] : 0.f;
        if (first) prefetch();
        arrived(qx);
        arrived(qy);
        arrived(qz);
        arrived(cx);
        arrived(cy);
        arrived(cz);
        int mine = 0;
        uint64_t open = nq == 64 ? ~0ull : ((1ull << nq) - 1ull);
        // the open queries against candidate chunk [jb, jb + 64)
        auto test = [&](const int jb, const float x, const float y, const float z) __attribute__((always_inline)) {
            const bool v = jb + lane < end;
            uint64_t m = open;
            st.add(kStatCountTests, (unsigned long long)__popcll(m) * (unsigned)min(64, end - jb));
            while (m) {
                const int qi = __ffsll((unsigned long long)m) - 1;
                m &= m - 1;
                const int c =
                    __popcll(__ballot(v & (sqd(dim, lane_f(qx, qi), lane_f(qy, qi), lane_f(qz, qi), x, y, z) < e2)));
                if (lane == qi) mine += c;
            }
            open &= ~__ballot(mine >= minpts);
        };
        // the first chunk outside the loop: its wait leaves the prefetch in flight
        test(0, cx, cy, cz);
        for (int jb = 64; open; jb += 64) {
            pos = walk_chunk(w, jb, &end);
            if (jb >= end) break;
            const float x = V.sx[pos];
            const float y = dim > 1 ? V.sy[pos] : 0.f;
            const float z = dim > 2 ? V.sz[pos] : 0.f;
            test(jb, x, y, z);
        }
        if (lane < nq) {
            V.flags[cs + q0 + lane] = count_flags(mine, minpts, safe);
            // unsafe cell: every core its own element
            if (!safe) V.uf[V.W + cs + q0 + lane] = ufe(qslot, V.W + cs + q0 + lane);
        }
        const uint64_t cm = __ballot(lane < nq && mine >= minpts);
        if (fc == kNoCore && cm != 0ull) {
            const int l = __ffsll((unsigned long long)cm) - 1;
            fc = cs + q0 + l;
            fslot = lane_i(qslot, l);
        }
    };
    block(0, true);
    for (int q0 = 64; q0 < nA; q0 += 64) block(q0, false);
    if (lane == 0) {
        V.fcore[A] = fc;  // first (minimum-slot) core: the cell's representative
        V.uf[A] = fc == kNoCore ? kUfNone : (safe ? ufe(fslot, A) : kUfUnsafe);
    }
}

// One wave per cell in a grid-stride walk over all cells of the launch; the
// next cell's header is in flight while the current cell computes.
template <class ST>
__global__ __launch_bounds__(64 * kCellWaves) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_count(BatchArgs a) {
    const int total = uni(ldc(a.cell_pre[a.n]));
    const int nw = gridDim.x * kCellWaves;
    ST st;
    int gc = uni(blockIdx.x * kCellWaves + (threadIdx.x >> 6));
    if (gc < total) {
        int s = uni(find_stream_from(a.cell_pre, a.n, gc, 0));  // cells rise, so streams do
        int c = gc - uni(ldc(a.cell_pre[s]));
        CellHdr h = load_hdr(a.s[s], c);
        while (true) {
            const int gn = gc + nw;
            int sn = s, cn = 0;
            CellHdr hn = h;
            // (past the last cell it reloads the last one: no branch around the loads)
            auto prefetch = [&]() {
                const int gq = min(gn, total - 1);
                sn = uni(find_stream_from(a.cell_pre, a.n, gq, s));
                cn = gq - uni(ldc(a.cell_pre[sn]));
                hn = load_hdr(a.s[sn], cn);
            };
            stats_stream(a, st, s);
            count_cell(cell_view(a.s[s]), c, h, st, prefetch);
            if (gn >= total) break;
            // (moved to scalar registers again: the compiler does not carry that
            // they are uniform around the loop, and would read the descriptor
            // and search the streams with vector loads)
            gc = uni(gn);
            s = uni(sn);
            c = uni(cn);
            h = hn;
        }
    }
    stats_flush(a, st);
}

// Cluster id of the core at position p of cell c, whose entry is e: the slot
// of its element's root. For kernels that run after the merge.
__device__ __forceinline__ int core_cid(const CellView &V, uint64_t e, int p) {
    if (e == kUfUnsafe) e = V.uf[V.W + p];
    return ufe_slot(ufe_root(V.uf, e));
}

// Outputs of one cell, after the merge (the reference's post_cluster_t,
// aabb.cu:173-196, and border claim, dbscan.cu:370-377): a core takes the
// root of its union-find element - the minimum core slot of its cluster; a
// non-core point takes the minimum root among the cores within eps (border,
// the deterministic form of the reference's claim) or stays noise. The roots
// are found here, so no separate flatten pass runs. The wave of each
// stream's first cell also advances the ring cursor. Loads in rounds, as in
// count_cell.
template <class ST>
__device__ void output_cell(const BatchArgs &a, int s, const CellView &V, const IO &io, int A, ST &st) {
    const int lane = lane_id();
    const int dim = V.dim;
    const float e2 = V.eps2;
    const int cfv = V.cflag[A], csv = V.cstart[A], cev = V.cstart[A + 1];
    const uint64_t ev = V.uf[A];
    const uint64_t rw = row_word(V, A);
    arrived(rw);
    // a safe cell's cores share one root, found once
    const int cidA = ufe_is(ev) ? core_cid(V, ev, 0) : 0;
    if (A == 0 && lane == 0) {
        StreamMut *m = ldc(a.s[s].mut);
        if (a.stats) a.stats[(size_t)s * kNumStats + kStatCells] += (unsigned long long)m->ncell;
        m->t = m->t + 1;
        m->u = m->u + 1 == ldc(a.s[s].units) ? 0 : m->u + 1;
    }
    const int cs = uni(csv), nA = uni(cev) - cs;
    const bool dense = uni(cfv) & kCellDense;
    gptr<int32_t> label = gl(io.label), cidv = gl(io.cid);
    const RowWalk w0 = row_walk(rw, INT_MAX);
    for (int q0 = 0; q0 < nA; q0 += 64) {
        const int nq = min(64, nA - q0);
        const int pq = cs + q0 + min(lane, nq - 1);
        const int qf = V.flags[pq];
        const uint64_t qk = V.skey[pq];
        const float qx = V.sx[pq];
        const float qy = dim > 1 ? V.sy[pq] : 0.f;
        const float qz = dim > 2 ? V.sz[pq] : 0.f;
        arrived(qk);
        arrived(qx);
        arrived(qy);
        arrived(qz);
        const int qslot = (int)((uint32_t)qk & V.smask);
        if (lane < nq && (qf & kFlagCore)) {
            label[qslot] = 0;
            cidv[qslot] = ev == kUfUnsafe ? core_cid(V, ev, pq) : cidA;
        }
        if (dense) continue;
        const bool noise = lane < nq && known_noise(a, qf);
        if (noise) {
            label[qslot] = 2;
            cidv[qslot] = qslot;
        }
        const bool isq = lane < nq && !(qf & kFlagCore) && !noise;
        const uint64_t open = __ballot(isq);
        if (open == 0ull) continue;
        int best = INT_MAX;
        RowWalk w = w0;
        for (int jb = 0;; jb += 64) {
            int end;
            const int pos = walk_chunk(w, jb, &end);
            if (jb >= end) break;
            const int f = V.flags[pos];
            const float cx = V.sx[pos];
            const float cy = dim > 1 ? V.sy[pos] : 0.f;
            const float cz = dim > 2 ? V.sz[pos] : 0.f;
            const int pc = V.pcell[pos];
            arrived(cx);
            arrived(cy);
            arrived(cz);
            arrived(pc);
            const bool core = jb + lane < end && (f & kFlagCore);
            uint64_t m = open;
            st.add(kStatBorderTests, (unsigned long long)__popcll(m) * (unsigned)min(64, end - jb));
            // roots of the chunk's cores, found once a query of the cell hits one
            int cid = INT_MAX;
            bool have = false;
            while (m) {
                const int qi = __ffsll((unsigned long long)m) - 1;
                m &= m - 1;
                const bool hit = core & (sqd(dim, lane_f(qx, qi), lane_f(qy, qi), lane_f(qz, qi), cx, cy, cz) < e2);
                if (__ballot(hit) == 0ull) continue;
                if (!have) {
                    if (core) cid = core_cid(V, V.uf[pc], pos);
                    have = true;
                }
                const int mn = wave_min(hit ? cid : INT_MAX);
                if (lane == qi) best = min(best, mn);
            }
        }
        if (isq) {
            label[qslot] = best != INT_MAX ? 1 : 2;
            cidv[qslot] = best != INT_MAX ? best : qslot;
        }
    }
}

template <class ST>
__global__ __launch_bounds__(64 * kCellWaves) void k_border(BatchArgs a) {
    const int total = uni(ldc(a.cell_pre[a.n]));
    const int nw = gridDim.x * kCellWaves;
    ST st;
    int s = 0;  // stream of the wave's current cell (cells rise, so streams do)
    for (int gc = uni(blockIdx.x * kCellWaves + (threadIdx.x >> 6)); gc < total; gc += nw) {
        s = uni(find_stream_from(a.cell_pre, a.n, gc, s));
        const int c = gc - uni(ldc(a.cell_pre[s]));
        stats_stream(a, st, s);
        output_cell(a, s, cell_view(a.s[s]), a.use_io1 ? a.io1 : a.io[s], c, st);
    }
    stats_flush(a, st);
}

// ---------------------------------------------------------------------------
// Cluster merge of streams without safe cells (reach 1): every core is an
// element.

// Touching pairs of cores of one wave, united in parallel rounds: the pairs of
// several candidate chunks and cells - of any streams of the launch - are
// collected in LDS and each lane then walks the union-find of its pair's
// stream, so the dependent loads of the walks overlap instead of adding up
// cell after cell.
constexpr int kEdgeCap = 320;

// One cell's header as the merge needs it: stream, cell within the stream,
// first core position (kNoCore: none, or no cell) and position range.
struct CellHead {
    int s, c, fc, cf, cs, ce;
};

// Streams whose cells the one-wave-per-cell merge unites.
__device__ __forceinline__ bool merged_by_wave(const BatchArgs &a, int dense_ok) { return a.wave_merge || !dense_ok; }

// Lane l's cell g = g0 + l * nw of a wave's grid-stride sequence: its stream
// by a per-lane binary search over the batch's cell prefix (a small table
// that stays in cache), then the header, all lanes' loads in one round. A cell
// past `total`, or of a stream with safe cells, reads as a cell without cores.
__device__ __forceinline__ CellHead cell_head(const BatchArgs &a, long long g, int total) {
    CellHead h{0, 0, kNoCore, 0, 0, 0};
    bool valid = g < total;
    const gptr<const int32_t> pre = gl((const int32_t *)a.cell_pre);
    int lo = 0, hi = a.n, plo = 0;  // pre[0] = 0
    while (valid && hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        const int v = pre[mid];
        if ((long long)v <= g) {
            lo = mid;
            plo = v;
        } else {
            hi = mid;
        }
    }
    h.s = lo;
    h.c = valid ? (int)(g - plo) : 0;
    const gptr<const StreamDev> sd = gl(a.s) + h.s;
    valid = valid && merged_by_wave(a, sd->dense_ok);
    if (valid) {
        h.cf = gl((const uint8_t *)sd->cflag)[h.c];
        h.fc = gl((const int32_t *)sd->fcore)[h.c];
        h.cs = gl((const int32_t *)sd->cstart)[h.c];
        h.ce = gl((const int32_t *)sd->cstart)[h.c + 1];
    }
    return h;
}

// Lane j's header, wave-uniform.
__device__ __forceinline__ CellHead lane_head(const CellHead &m, int j) {
    return CellHead{lane_i(m.s, j), lane_i(m.c, j), lane_i(m.fc, j), lane_i(m.cf, j), lane_i(m.cs, j), lane_i(m.ce, j)};
}

struct Edge {
    int x, y;  // union-find elements
    int s;     // stream
};

struct EdgeBuf {
    Edge *e;  // this wave's LDS slice
    int n;    // pairs held (uniform)
};

__device__ __forceinline__ void edge_flush(const BatchArgs &a, EdgeBuf &eb) {
    for (int i = lane_id(); i < eb.n; i += 64) {
        const Edge e = eb.e[i];
        ufe_unite<true>(gl(ldc(a.s[e.s].uf)), e.x, e.y);
    }
    eb.n = 0;
}

// Queues (target, rep) for every lane that wants it, once per run of lanes
// holding the same element (a safe cell's points are adjacent in a candidate
// chunk and share one).
template <class ST>
__device__ __forceinline__ void unite_once_per_rep(const BatchArgs &a, EdgeBuf &eb, int s, bool want, int rep,
                                                   int target, ST &st) {
    const int lane = lane_id();
    const uint64_t m = __ballot(want);
    if (m == 0ull) return;
    const uint64_t below = m & ((1ull << lane) - 1ull);
    const int prev = below ? 63 - __clzll((long long)below) : lane;
    const int prep = __shfl(rep, prev);
    const bool first = want && (below == 0ull || prep != rep);
    const uint64_t fm = __ballot(first);
    const int nf = __popcll(fm);
    st.add(kStatMergePairs, __popcll(m));
    st.add(kStatUnites, nf);
    if (eb.n + nf > kEdgeCap) edge_flush(a, eb);
    if (first) eb.e[eb.n + __popcll(fm & ((1ull << lane) - 1ull))] = Edge{target, rep, s};
    eb.n += nf;
}

// Candidate positions before which a safe cell's merge goes over candidate
// cells first (below it, scanning the positions costs fewer round trips).
constexpr int kCellLevelMin = 192;

// Cluster merge (the reference's __raygen__cluster + unite,
// dbscan.cu:279-321,354-394,9-43) by one wave per cell A with cores, for
// streams of reach 1, which have no safe cell, and for a single small stream.
// A's candidates are the stencil positions before A's own first position - the
// points of the stencil cells ordered before A, so each pair of cells is
// tested once, from its later cell - loaded 64 at a time, coalesced. A safe
// cell is one element: a candidate core within eps of any core of A joins it.
// The cores of an unsafe cell are separate elements (kFlagLoose), and the
// cell's own earlier points are candidates too.
//
// It is bound by its chain of loads, which is shorter than that of the links
// and joins (k_merge_cells), but it tests the cores of every pair. us of both:
// 3-D trajectories of 3,474 points 9.9 and 17.8, 20,588 points 10.7 and 20.8,
// 33,750 19.3 and 18.5, 40,440 15.5 and 24.2, 76,272 22.7 and 28.2; at a third of
// eps 34,240 28.6 and 21.1, 81,781 27.6 and 31.0; 2-D blobs of 831 points 8.1 and
// 13.0, 10,000 28.6 and 14.7; 100,000 1-D points 128 and 15. Six waves a SIMD,
// not eight: no spills, and few waves in such a launch (3,474 points 10.4 us with
// eight). The unites walk by cached loads (agent-scope ones: 40,440 points 16.0
// us, 81,781 30.2, 33,750 21.4).
//
// A safe cell with many candidates goes over its candidate cells first, 64 per
// round: a safe candidate cell joins A as soon as its first core is within eps
// of a core of A. Only the cells not settled that way have their points
// scanned.
template <class ST>
__device__ void union_cell(const BatchArgs &a, int s, const CellView &V, const CellHead &h, ST &st, EdgeBuf &eb,
                           uint64_t rw) {
    const int lane = lane_id();
    const int dim = V.dim;
    const float e2 = V.eps2;
    // the header comes screened (cell_head) and the stencil rows (rw, lane r:
    // row r, every lane loaded) came in with the previous cell; the first
    // queries and the first candidate chunk load in one round, then each
    // further chunk is a round of its own
    const bool safeA = h.cf & kCellSafe;
    const int cs = h.cs, nA = h.ce - h.cs;
    const RowWalk w0 = row_walk(lane < V.R ? rw : 0ull, safeA ? cs : cs + nA);
    if (w0.rest == 0ull) return;
    const bool by_cells = safeA && uni(wave_sum(w0.len)) >= kCellLevelMin;
    for (int q0 = 0; q0 < nA; q0 += 64) {
        const int nq = min(64, nA - q0);
        const int pq = cs + q0 + min(lane, nq - 1);
        const int qf = V.flags[pq];
        const float qx = V.sx[pq];
        const float qy = dim > 1 ? V.sy[pq] : 0.f;
        const float qz = dim > 2 ? V.sz[pq] : 0.f;
        // the point scan's first chunk, in the same round (not for the
        // cell-level pass, which scans other walks)
        RowWalk w1 = w0;
        int end1 = 0;
        const int pos1 = walk_chunk(w1, 0, &end1);
        const int f1 = by_cells ? 0 : V.flags[pos1];
        const float x1 = by_cells ? 0.f : V.sx[pos1];
        const float y1 = by_cells || dim < 2 ? 0.f : V.sy[pos1];
        const float z1 = by_cells || dim < 3 ? 0.f : V.sz[pos1];
        const int r1 = by_cells ? 0 : V.pcell[pos1];
        arrived(qx);
        arrived(qy);
        arrived(qz);
        arrived(x1);
        arrived(y1);
        arrived(z1);
        arrived(r1);
        const bool qcore = lane < nq && (qf & kFlagCore);
        const uint64_t qm = __ballot(qcore);
        if (qm == 0ull) continue;
        // The cores qm of this block against candidate chunk [jb, jb + 64) of
        // a walk whose candidates end at `end`.
        auto test = [&](const int jb, const int end, const int pos, const int f, const float cx, const float cy,
                        const float cz, const int rp) __attribute__((always_inline)) {
                const bool bcore = jb + lane < end && (f & kFlagCore);
                const uint64_t bm = __ballot(bcore);
                if (bm == 0ull) return;
                const int rep = bcore ? ((f & kFlagLoose) ? V.W + pos : rp) : -1;
                const unsigned chunk = (unsigned)min(64, end - jb);
                uint64_t m = qm;
                if (safeA) {
                    // lanes holding one element form a run (a safe cell's points are
                    // adjacent); one touching lane settles its whole run
                    const int prev_rep = prev_lane(rep);  // every lane takes part in the moves
                    const int prev_core = prev_lane((int)bcore);
                    const uint64_t starts = __ballot(lane == 0 || prev_rep != rep || !prev_core);
                    const uint64_t after = starts & ~((2ull << lane) - 1ull);  // run starts above this lane
                    const uint64_t upto = after ? (after & (~after + 1ull)) - 1ull : ~0ull;
                    const uint64_t below = starts & ((2ull << lane) - 1ull);
                    const uint64_t from = ~((1ull << (63 - __clzll((long long)below))) - 1ull);
                    const uint64_t run = upto & from;  // this lane's run
                    // touched candidates as one wave mask: the loop carries a scalar,
                    // not a lane predicate
                    uint64_t t = 0;
                    while (m) {
                        const int qi = __ffsll((unsigned long long)m) - 1;
                        m &= m - 1;
                        st.add(kStatMergeTests, chunk);
                        // every lane evaluates the test, no branch per query
                        t |= __ballot(sqd(dim, lane_f(qx, qi), lane_f(qy, qi), lane_f(qz, qi), cx, cy, cz) < e2) & bm;
                        if ((__ballot((t & run) != 0ull) | ~bm) == ~0ull) break;  // every candidate run settled
                    }
                    unite_once_per_rep(a, eb, s, (t >> lane) & 1ull, rep, h.c, st);
                } else {
                    while (m) {
                        const int qi = __ffsll((unsigned long long)m) - 1;
                        m &= m - 1;
                        st.add(kStatMergeTests, chunk);
                        const bool hit = bcore & (pos < cs + q0 + qi) &
                                         (sqd(dim, lane_f(qx, qi), lane_f(qy, qi), lane_f(qz, qi), cx, cy, cz) < e2);
                        unite_once_per_rep(a, eb, s, hit, rep, V.W + cs + q0 + qi, st);
                    }
                }
        };
        // the cores qm of this block against the candidate positions of walk w
        auto scan = [&](RowWalk w) __attribute__((always_inline)) {
            for (int jb = 0;; jb += 64) {
                int end;
                const int pos = walk_chunk(w, jb, &end);
                if (jb >= end) break;
                const int f = V.flags[pos];
                const float cx = V.sx[pos];
                const float cy = dim > 1 ? V.sy[pos] : 0.f;
                const float cz = dim > 2 ? V.sz[pos] : 0.f;
                const int rp = V.pcell[pos];
                arrived(cx);
                arrived(cy);
                arrived(cz);
                arrived(rp);
                test(jb, end, pos, f, cx, cy, cz, rp);
            }
        };
        if (!by_cells) {
            // the first chunk came with the queries
            if (end1 > 0) test(0, end1, pos1, f1, x1, y1, z1, r1);
            for (int jb = 64;; jb += 64) {
                int end;
                const int pos = walk_chunk(w1, jb, &end);
                if (jb >= end) break;
                const int f = V.flags[pos];
                const float cx = V.sx[pos];
                const float cy = dim > 1 ? V.sy[pos] : 0.f;
                const float cz = dim > 2 ? V.sz[pos] : 0.f;
                const int rp = V.pcell[pos];
                arrived(cx);
                arrived(cy);
                arrived(cz);
                arrived(rp);
                test(jb, end, pos, f, cx, cy, cz, rp);
            }
            continue;
        }
        // candidate cells: row r (lane r) covers positions [rx, rx + len), all
        // before cs, i.e. the cells pcell[rx] .. pcell[rx + len - 1] (< A)
        const int clo = w0.len > 0 ? V.pcell[w0.rx] : 0;
        const int chi = w0.len > 0 ? V.pcell[w0.rx + w0.len - 1] + 1 : 0;
        RowWalk cw;
        cw.rx = clo;
        cw.len = chi - clo;
        cw.rest = __ballot(cw.len > 0);
        for (int jb = 0;; jb += 64) {
            int endc;
            const int B = walk_chunk(cw, jb, &endc);
            if (jb >= endc) break;
            const bool valid = jb + lane < endc;
            const int fb = V.fcore[B];
            const int cfb = V.cflag[B];
            const int bs = V.cstart[B];
            const int be = V.cstart[B + 1];
            arrived(fb);
            arrived(be);
            const bool has = valid && fb != kNoCore;
            const int fp = has ? fb : cs;  // a valid position either way
            const float bx = V.sx[fp];
            const float by = dim > 1 ? V.sy[fp] : 0.f;
            const float bz = dim > 2 ? V.sz[fp] : 0.f;
            arrived(bx);
            arrived(by);
            arrived(bz);
            // safe candidate cells: A's cores against each cell's first core
            const uint64_t cand = __ballot(has && (cfb & kCellSafe));
            uint64_t hit = 0;
            for (uint64_t m = qm; m && hit != cand;) {
                const int qi = __ffsll((unsigned long long)m) - 1;
                m &= m - 1;
                st.add(kStatMergeTests, (unsigned)__popcll(cand & ~hit));
                hit |= __ballot(sqd(dim, lane_f(qx, qi), lane_f(qy, qi), lane_f(qz, qi), bx, by, bz) < e2) & cand;
            }
            unite_once_per_rep(a, eb, s, (hit >> lane) & 1ull, B, h.c, st);
            // the cells with cores not settled: scan their points
            RowWalk pw;
            pw.rx = bs;
            pw.len = (has && !((hit >> lane) & 1ull)) ? be - bs : 0;
            pw.rest = __ballot(pw.len > 0);
            if (pw.rest) scan(pw);
        }
    }
}

template <class ST>
__global__ __launch_bounds__(64 * kCellWaves) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_union(BatchArgs a) {
    __shared__ Edge edges[kCellWaves][kEdgeCap];
    const int total = uni(ldc(a.cell_pre[a.n]));
    const int nw = gridDim.x * kCellWaves;
    ST st;
    EdgeBuf eb{edges[threadIdx.x >> 6], 0};
    const int w = uni(xcd_block(blockIdx.x, gridDim.x, a.xcd_groups & kXcdUnion) * kCellWaves + (threadIdx.x >> 6));
    // stencil rows of a cell, lane r: row r (every lane loads, clamped to the
    // last row; lanes >= R are cleared where the rows are used)
    auto rows_of = [&](const CellHead &x) __attribute__((always_inline)) {
        const StreamDev &S = a.s[x.s];
        const int R = ldc(S.R);
        return RowTable<const uint64_t>(S).at(x.c, min(lane_id(), R - 1));
    };
    for (long long g0 = w; g0 < total; g0 += 64ll * nw) {
        const CellHead mine = cell_head(a, g0 + (long long)lane_id() * nw, total);
        uint64_t m = __ballot(mine.fc != kNoCore);
        if (m == 0ull) continue;
        CellHead h = lane_head(mine, __ffsll((unsigned long long)m) - 1);
        uint64_t rw = rows_of(h);
        while (true) {
            m &= m - 1ull;
            // the next cell's rows are in flight while this cell merges (past
            // the last cell the current one's reload: no branch around the load)
            const CellHead hn = m ? lane_head(mine, __ffsll((unsigned long long)m) - 1) : h;
            const uint64_t rwn = rows_of(hn);
            stats_stream(a, st, h.s);
            union_cell(a, h.s, cell_view(a.s[h.s]), h, st, eb, rw);
            if (m == 0ull) break;
            h = hn;
            rw = rwn;
        }
    }
    edge_flush(a, eb);
    stats_flush(a, st);
}

// ---------------------------------------------------------------------------
// Cluster merge of streams whose interior cells are safe (k*k > dim), one
// launch over tiles of consecutive cells, a tile per wave.
//
// A safe cell is one union-find element, and what the merge needs is which
// cells touch, transitively. Nearly all of that is found by very few tests:
//   links  join every cell with at most one earlier cell on each axis, a cell
//          whose first core is within eps of this cell's first core;
//   joins  go over all earlier stencil cells and compare roots. Only pairs
//          whose roots still differ are tested, in a lane where that takes few
//          tests and otherwise by several lanes together.
// Once every cell is linked (1.0-1.8 unites a cell), 0.03-4% of the cell pairs
// of the 64-stream batch, of a 1 M-point window of uneven density and of
// 100,000 trajectory points still have different roots; the one-wave-per-cell
// kernel that this replaced tested the cores of every pair. Its times and
// these, in us (events): 64 streams 360 and 138 (with the pass over the cells
// that follows the point-parallel count), 1 M points 446 and 92, 100,000 1-D
// points in dense cells 128 and 15, 100,000 trajectory points 31 and 27,
// 10,000 2-D points 28.6 and 15; 1,000 2-D points 9 and 14, 61,503 points with
// a third of eps per cell 24 and 27.
//
// What bounds it is each wave's chain of dependent loads (entry, row, the
// row's cells, their entries and first cores, the walks to the roots, the
// hook), so every step of it serves as many cells or pairs as it can: a
// tile's cells without cores take no lanes, unites and pairs are queued in
// LDS and taken 64 at a time.

// The lanes of a tile's cells for which `in` holds, in order: lane i of the
// result holds the lane of the i-th such cell (the others follow).
__device__ __forceinline__ int tile_order(bool in, uint64_t m) {
    const int lane = lane_id();
    const int below = __popcll(m & ((1ull << lane) - 1ull));
    return __builtin_amdgcn_ds_permute((in ? below : __popcll(m) + lane - below) << 2, lane);
}

__device__ __forceinline__ int from_lane(int v, int l) { return __builtin_amdgcn_ds_bpermute(l << 2, v); }

__device__ __forceinline__ uint64_t from_lane64(uint64_t v, int l) {
    const uint32_t lo = (uint32_t)from_lane((int)(uint32_t)v, l), hi = (uint32_t)from_lane((int)(uint32_t)(v >> 32), l);
    return ((uint64_t)hi << 32) | lo;
}

// First and last cell before cell A of stencil row r (Bf > Bl: none).
__device__ __forceinline__ void row_cells(const CellView &V, int A, uint64_t rw, int *Bf, int *Bl) {
    const int rx = (int)(uint32_t)rw, ry = (int)(uint32_t)(rw >> 32);
    const int f = at(V.pcell, rx), l = at(V.pcell, max(ry - 1, 0));  // an empty row is (0, 0)
    *Bf = f;
    *Bl = ry > rx ? min(l, A - 1) : f - 1;
}

// Pairs of elements of one stream, united 64 at a time, one per lane: the
// walks and hooks of a tile's unites overlap instead of adding up.
constexpr int kLinkCap = 64 * 4;  // a tile's most: 64 cells, up to 4 unites each

struct LinkBuf {
    int2 *e;  // this wave's LDS slice
    int n;    // pairs held (uniform)
};

__device__ __forceinline__ void link_push(LinkBuf &lb, bool want, int x, int y) {
    const uint64_t m = __ballot(want);
    if (want) lb.e[lb.n + __popcll(m & ((1ull << lane_id()) - 1ull))] = make_int2(x, y);
    lb.n += __popcll(m);
}

// Links of a tile's cells, lane i on the tile's i-th cell with cores. A cell
// joins the cell with cores before it in the table when their first cores are
// within eps (in a column that is its nearest neighbour; across columns the
// test fails). The resulting runs need no unites: each member hooks under the
// run's minimum slot, one atomic on its own entry. On each other axis a cell
// joins the first cell of the stencil row one step back (nearest first) whose
// first core is within eps, unless the cell before it in its run already did:
// the two rows' cells are most likely one run as well.
template <int D, class ST>
__device__ __forceinline__ void link_tile(const CellView &V, int k, int c0, int T, int ncell, LinkBuf &lb, ST &st) {
    const int lane = lane_id();
    const bool valid = lane < T && c0 + lane < ncell;
    const uint64_t w = valid ? at(V.uf, c0 + lane) : kUfNone;
    const int fc = valid ? at(V.fcore, c0 + lane) : 0;
    const uint64_t m = __ballot(ufe_is(w));
    if (m == 0ull) return;
    const int nm = __popcll(m);
    const int order = tile_order(ufe_is(w), m);
    const bool have = lane < nm;
    const int A = c0 + order;
    const uint64_t wa = from_lane64(w, order);  // (other waves may have hooked the entry already)
    const int fa = from_lane(fc, order);  // (every lane takes part in the moves)
    const int pa = have ? fa : 0;
    const float ax = at(V.sx, pa);
    const float ay = D > 1 ? at(V.sy, pa) : 0.f;
    const float az = D > 2 ? at(V.sz, pa) : 0.f;
    uint64_t rw[D];
#pragma unroll
    for (int i = 1; i < D; i++) rw[i] = have ? V.rows.at(A, i == 1 ? 1 : 2 * k + 1) : 0ull;
    // the cell before: lane - 1; for lane 0 the cell before the tile
    bool b1 = false;
    float x1 = 0.f, y1 = 0.f, z1 = 0.f;
    if (lane == 0 && c0 > 0) {
        b1 = ufe_is(at(V.uf, c0 - 1));
        const int p1 = b1 ? at(V.fcore, c0 - 1) : 0;
        x1 = at(V.sx, p1);
        y1 = D > 1 ? at(V.sy, p1) : 0.f;
        z1 = D > 2 ? at(V.sz, p1) : 0.f;
    }
    const float px = __int_as_float(prev_lane(__float_as_int(ax)));
    const float py = __int_as_float(prev_lane(__float_as_int(ay)));
    const float pz = __int_as_float(prev_lane(__float_as_int(az)));
    const bool joins = have & (lane > 0) & (sqd(D, ax, ay, az, px, py, pz) < V.eps2);
    const uint64_t lm = __ballot(joins);  // lanes that continue the run of the lane before
    const uint64_t heads = ~lm, upto = (2ull << lane) - 1ull;
    const int first = 63 - __clzll((long long)(heads & upto));  // (lane 0 is a head)
    const uint64_t later = heads & ~upto;
    const int last = later ? __ffsll((unsigned long long)later) - 2 : 63;
    uint64_t rm = wa;  // minimum entry of the run
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint64_t y = from_lane64(rm, max(lane - o, 0));
        if (lane - o >= first) rm = min(rm, y);
    }
    rm = from_lane64(rm, last);
    uint64_t old = rm;
    if (have && wa != rm) old = ufe_min(V.uf + A, rm);
    int to[D];
    int tests = have && lane > 0;
#pragma unroll
    for (int i = 1; i < D; i++) {
        int Bf, Bl;
        row_cells(V, A, rw[i], &Bf, &Bl);
        const int n = have ? Bl - Bf + 1 : 0;
        const int mid = (Bf + Bl) >> 1;
        to[i] = -1;
        for (int u0 = 0; u0 < n && to[i] < 0; u0 += 3) {
            bool wb[3];
            int cb[3];
            float bx[3], by[3], bz[3];
#pragma unroll
            for (int q = 0; q < 3; q++) {
                const int u = min(u0 + q, n - 1);
                const int B = cb[q] = mid + ((u & 1) ? (u + 1) >> 1 : -(u >> 1));
                wb[q] = ufe_is(at(V.uf, B));
                const int p = at(V.fcore, B);
                const int pp = wb[q] ? p : 0;
                bx[q] = at(V.sx, pp);
                by[q] = D > 1 ? at(V.sy, pp) : 0.f;
                bz[q] = D > 2 ? at(V.sz, pp) : 0.f;
            }
#pragma unroll
            for (int q = 0; q < 3; q++) {
                const bool t = (u0 + q < n) & (to[i] < 0) & wb[q];
                tests += t;
                if (t & (sqd(D, ax, ay, az, bx[q], by[q], bz[q]) < V.eps2)) to[i] = cb[q];
            }
        }
    }
    // (an entry that was no root any more: its ancestor joins the run)
    link_push(lb, old != rm && ufe_idx(old) != A, ufe_idx(rm), ufe_idx(old));
    const bool t1 = b1 & (sqd(D, ax, ay, az, x1, y1, z1) < V.eps2);
    link_push(lb, t1, ufe_idx(rm), c0 - 1);
    int nu = __popcll(lm) + (__ballot(t1) != 0ull);
#pragma unroll
    for (int i = 1; i < D; i++) {
        const uint64_t hit = __ballot(to[i] >= 0);
        const bool want = to[i] >= 0 && !((((hit << 1) & lm) >> lane) & 1ull);
        link_push(lb, want, ufe_idx(rm), to[i]);
        nu += __popcll(__ballot(want));
    }
    wave_sync();
    for (int i = lane; i < lb.n; i += 64) ufe_unite(V.uf, lb.e[i].x, lb.e[i].y);
    lb.n = 0;
    st.add(kStatMergeTests, wave_sum(tests));
    st.add(kStatMergePairs, nu);
    st.add(kStatUnites, nu);
}

// Cell pairs the wave tests core by core: lane of the tile's cell A in the
// upper 8 bits, cell B below.
constexpr int kPairCap = 512;  // 64 rows of at most kRowCells cells, and fewer than 64 pairs left over
constexpr int kFew = 4;  // points of a cell tested in a lane
constexpr int kRowCells = 2 * kMaxK + 1;  // most cells of a stencil row
static_assert(64 * kRowCells + 63 <= kPairCap, "");

struct PairBuf {
    uint32_t *e;  // this wave's LDS slice
    int n;        // pairs held (uniform)
};

__device__ __forceinline__ void pair_push(PairBuf &pb, bool want, int la, int B) {
    const uint64_t m = __ballot(want);
    if (want) pb.e[pb.n + __popcll(m & ((1ull << lane_id()) - 1ull))] = ((uint32_t)la << 24) | (uint32_t)B;
    pb.n += __popcll(m);
}

// (What follows is one instance for every dimension and reach, each loop with
// one call site: inlined per dimension it was 130 KB of code, twice the
// instruction cache of a pair of CUs, and no faster.)

// Minimum over groups of lp lanes: 8, 16 or 64 (uniform).
__device__ __forceinline__ float group_fmin(float v, int lp) {
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) v = fminf(v, __int_as_float(xor_lane(__float_as_int(v), o)));
    if (lp > 8) v = fminf(v, __int_as_float(xor_lane(__float_as_int(v), 8)));
    if (lp > 16) {
        v = fminf(v, __int_as_float(xor_lane(__float_as_int(v), 16)));
        v = fminf(v, __int_as_float(xor_lane(__float_as_int(v), 32)));
    }
    return v;
}

// Gap between x and the interval [lo, -nhi].
__device__ __forceinline__ float gap(float x, float lo, float nhi) {
    return x < lo ? __fsub_rn(lo, x) : (x > -nhi ? __fsub_rn(x, -nhi) : 0.f);
}

// Up to kHeld points per lane of a group of lanes, with their core flags and
// the box of the cores (upper bounds negated: one kind of reduction).
constexpr int kHeld = 4;

struct HeldCores {
    float x[kHeld], y[kHeld], z[kHeld];
    bool core[kHeld];
    float lx, ly, lz, nx, ny, nz;
};

// The points at positions [c0, c1), at most lp * kHeld of them, on lp lanes.
__device__ __forceinline__ void hold_cores(const CellView &V, int lp, bool on, int c0, int c1, HeldCores &h) {
    const int sub = lane_id() & (lp - 1);
    const float inf = __int_as_float(0x7f800000);
    h.lx = h.ly = h.lz = h.nx = h.ny = h.nz = inf;
#pragma unroll
    for (int q = 0; q < kHeld; q++) {
        const int i = c0 + q * lp + sub;
        const int p = on ? min(i, c1 - 1) : 0;
        h.x[q] = at(V.sx, p);
        h.y[q] = V.dim > 1 ? at(V.sy, p) : 0.f;
        h.z[q] = V.dim > 2 ? at(V.sz, p) : 0.f;
        h.core[q] = on && i < c1 && (at(V.flags, p) & kFlagCore);
    }
#pragma unroll
    for (int q = 0; q < kHeld; q++) {
        h.lx = fminf(h.lx, h.core[q] ? h.x[q] : inf);
        h.ly = fminf(h.ly, h.core[q] ? h.y[q] : inf);
        h.lz = fminf(h.lz, h.core[q] ? h.z[q] : inf);
        h.nx = fminf(h.nx, h.core[q] ? -h.x[q] : inf);
        h.ny = fminf(h.ny, h.core[q] ? -h.y[q] : inf);
        h.nz = fminf(h.nz, h.core[q] ? -h.z[q] : inf);
    }
}

// Do cores of A (positions [csA, ceA)) and B touch? lp lanes a pair, at most
// lp * kHeld points a side, all loaded in one round. Nearly all pairs that get
// here do not touch, so A's cores are held against the box of B's cores first
// and only those within eps of it tested against B's cores. (The rounded gap
// between a point and the box is at most its rounded difference to any point
// of the box, per axis, so nothing that touches is left out.) Called by the
// whole wave; `on` marks the groups that have a pair; A is best the smaller
// cell.
__device__ __forceinline__ bool cells_touch(const CellView &V, int lp, bool on, int csA, int ceA, int csB, int ceB,
                                            int &tests) {
    const int lane = lane_id();
    const uint64_t gm = lp == 64 ? ~0ull : ((1ull << lp) - 1ull) << (lane & ~(lp - 1));
    HeldCores a, b;
    hold_cores(V, lp, on, csA, ceA, a);
    hold_cores(V, lp, on, csB, ceB, b);
    b.lx = group_fmin(b.lx, lp);
    b.ly = group_fmin(b.ly, lp);
    b.lz = group_fmin(b.lz, lp);
    b.nx = group_fmin(b.nx, lp);
    b.ny = group_fmin(b.ny, lp);
    b.nz = group_fmin(b.nz, lp);
    const bool more = __ballot(on && ceB - csB > lp) != 0ull;  // a group holds more than a point of B per lane
    // bit q: this lane's q-th point of A is a core near the box
    uint32_t near = 0;
#pragma unroll
    for (int q = 0; q < kHeld; q++)
        near |= (a.core[q] & (sqd(3, gap(a.x[q], b.lx, b.nx), gap(a.y[q], b.ly, b.ny), gap(a.z[q], b.lz, b.nz),
                                  0.f, 0.f, 0.f) < V.eps2))
                    ? 1u << q
                    : 0u;
    bool touch = false;
    while (true) {
        const uint64_t m = __ballot(near != 0u) & gm;  // lanes of the group with such cores
        if (__ballot(m != 0ull) == 0ull) return touch;
        const int l = m ? __ffsll((unsigned long long)m) - 1 : lane;
        // this lane's next one, then the one of the group's lane l
        const int q = __ffs(near) - 1;
        float x = a.x[0], y = a.y[0], z = a.z[0];
#pragma unroll
        for (int r = 1; r < kHeld; r++) {
            x = q == r ? a.x[r] : x;
            y = q == r ? a.y[r] : y;
            z = q == r ? a.z[r] : z;
        }
        x = __int_as_float(from_lane(__float_as_int(x), l));
        y = __int_as_float(from_lane(__float_as_int(y), l));
        z = __int_as_float(from_lane(__float_as_int(z), l));
        if (lane == l) near &= near - 1u;
        bool hit = b.core[0] & (sqd(3, x, y, z, b.x[0], b.y[0], b.z[0]) < V.eps2);
        if (more) {
#pragma unroll
            for (int r = 1; r < kHeld; r++) hit |= b.core[r] & (sqd(3, x, y, z, b.x[r], b.y[r], b.z[r]) < V.eps2);
        }
        hit &= m != 0ull;
        tests += m != 0ull;
        if (__ballot(hit) & gm) {
            touch = true;
            near = 0;
        }
    }
}

// Cores of cell A against cores of cell B <= A where a cell is not safe, the
// whole wave: every touching pair of cores unites (in A = B each pair once).
__device__ __forceinline__ void join_cores(const CellView &V, int A, int B, bool safeA, bool safeB, int csA, int ceA,
                                           int csB, int ceB, int &tests, int &unites) {
    for (int pb = csB + lane_id(); pb < ceB; pb += 64) {
        const float bx = at(V.sx, pb);
        const float by = V.dim > 1 ? at(V.sy, pb) : 0.f;
        const float bz = V.dim > 2 ? at(V.sz, pb) : 0.f;
        if (!(at(V.flags, pb) & kFlagCore)) continue;
        for (int pa = csA; pa < (A != B ? ceA : pb); pa++) {
            tests++;
            if ((at(V.flags, pa) & kFlagCore) && sqd(3, at(V.sx, pa), V.dim > 1 ? at(V.sy, pa) : 0.f,
                                                 V.dim > 2 ? at(V.sz, pa) : 0.f, bx, by, bz) < V.eps2) {
                unites++;
                ufe_unite(V.uf, safeA ? A : V.W + pa, safeB ? B : V.W + pb);
            }
        }
    }
}

// The queued pairs: 64 at a time their entries, ranges and roots, one pair
// per lane; then those of safe cells with different roots, by the larger
// cell's points, on 8, 16 or 64 lanes each (most cells that get here hold a
// handful of points, and a pair's time is its chain of loads; the largest go
// 256 by 256 points); then the pairs with an unsafe cell.
template <class ST>
__device__ __forceinline__ void join_flush(const CellView &V, int c0, PairBuf &pb, ST &st) {
    const int lane = lane_id();
    int tests = 0, unites = 0;
    for (int i0 = 0; i0 < pb.n; i0 += 64) {
        const uint32_t e = pb.e[min(i0 + lane, pb.n - 1)];
        int A = c0 + (int)(e >> 24), B = (int)(e & 0xffffffu);
        const uint64_t ea = ufe_now(V.uf, A), eb = ufe_now(V.uf, B);
        int csA = at(V.cstart, A), ceA = at(V.cstart, A + 1), csB = at(V.cstart, B), ceB = at(V.cstart, B + 1);
        const bool on = i0 + lane < pb.n, safe = ufe_is(ea) && ufe_is(eb);
        bool open = on && safe;
        if (open) open = ufe_root_now(V.uf, ea) != ufe_root_now(V.uf, eb);
        if (open && ceA - csA > ceB - csB) {  // the smaller cell first
            int t = A;
            A = B;
            B = t;
            t = csA;
            csA = csB;
            csB = t;
            t = ceA;
            ceA = ceB;
            ceB = t;
        }
        // the small pairs eight a step, the larger ones four, the rest one by one
        const bool open8 = open && ceB - csB <= 8 * kHeld;
        const bool open16 = open && !open8 && ceB - csB <= 16 * kHeld;
        const uint64_t m8 = __ballot(open8), m16 = __ballot(open16);
        uint64_t bm = __ballot(open && !open8 && !open16);
        const int order8 = tile_order(open8, m8), order16 = tile_order(open16, m16);
        const int n8 = __popcll(m8), n16 = __popcll(m16);
        int a0 = 0, b0 = 0;  // the big pair's next points
        for (int k8 = 0, k16 = 0; k8 < n8 || k16 < n16 || bm != 0ull;) {
            const int lp = k8 < n8 ? 8 : (k16 < n16 ? 16 : 64);
            const int g = lane / lp + (lp == 8 ? k8 : k16), n = lp == 8 ? n8 : n16;
            const int l8 = from_lane(order8, min(g, 63)), l16 = from_lane(order16, min(g, 63));
            const int lb = bm ? __ffsll((unsigned long long)bm) - 1 : 0;
            const int l = lp == 8 ? l8 : (lp == 16 ? l16 : lb);
            const bool has = lp == 64 || g < n;
            const int x = from_lane(A, l), y = from_lane(B, l);
            int a1 = from_lane(csA, l), a2 = from_lane(ceA, l), b1 = from_lane(csB, l), b2 = from_lane(ceB, l);
            bool last = true;  // of this pair's steps
            if (lp == 64) {
                const int na = uni(a2) - uni(a1), nb = uni(b2) - uni(b1);
                a1 += a0;
                b1 += b0;
                a2 = min(a1 + 64 * kHeld, a2);
                b2 = min(b1 + 64 * kHeld, b2);
                b0 += 64 * kHeld;
                if (b0 >= nb) {
                    b0 = 0;
                    a0 += 64 * kHeld;
                }
                last = a0 >= na;
            }
            const bool touch = cells_touch(V, lp, has, a1, a2, b1, b2, tests);
            if (touch && (lane & (lp - 1)) == 0) {
                unites++;
                ufe_unite(V.uf, x, y);
            }
            if (lp == 8) {
                k8 += 8;
            } else if (lp == 16) {
                k16 += 4;
            } else if (last || uni(touch)) {
                bm &= bm - 1ull;
                a0 = b0 = 0;
            }
        }
        for (uint64_t m = __ballot(on && !safe); m; m &= m - 1ull) {
            const int l = __ffsll((unsigned long long)m) - 1;
            join_cores(V, lane_i(A, l), lane_i(B, l), lane_i(ufe_is(ea), l), lane_i(ufe_is(eb), l), lane_i(csA, l),
                       lane_i(ceA, l), lane_i(csB, l), lane_i(ceB, l), tests, unites);
        }
    }
    pb.n = 0;
    unites = wave_sum(unites);
    st.add(kStatMergeTests, wave_sum(tests));
    st.add(kStatMergePairs, unites);
    st.add(kStatUnites, unites);
}

// Joins of a tile's cells. The (cell, earlier stencil row) pairs are spread
// over the lanes and a row's cells queued as (cell, cell) pairs; the pairs'
// roots are then compared 64 at a time, one pair per lane (rows are mostly
// empty and cells few, so a lane for every cell a row could hold would idle
// 15 lanes of 16). Pairs with one root are done. The others are tested in
// their lane: cells of up to kFew points in full, larger ones by their first
// cores; larger cells that this does not join, and every pair with an unsafe
// cell, go to `far`.
template <class ST>
__device__ __forceinline__ void join_tile(const CellView &V, int k, int c0, int T, int ncell, PairBuf &pb, PairBuf &far,
                                          ST &st) {
    const int lane = lane_id(), dim = V.dim;
    const int width = 2 * k + 1;
    const int nrow = dim == 3 ? 1 + k + k * width : (dim == 2 ? 1 + k : 1);  // rows with earlier cells
    // x / nrow and x / width for the small x below, by multiplication
    const int irow = 65536 / nrow + 1, iwidth = 65536 / width + 1;
    const bool valid = lane < T && c0 + lane < ncell;
    const uint64_t w = valid ? ufe_now(V.uf, c0 + lane) : kUfNone;
    const uint64_t m = __ballot(w != kUfNone);
    if (m == 0ull) return;
    const int items = __popcll(m) * nrow;
    const int order = tile_order(w != kUfNone, m);
    // this lane's cell's root, compressed onto its entry; -1: an unsafe cell
    int ra = -1;
    if (ufe_is(w)) {
        const uint64_t r = ufe_root_now(V.uf, w);
        ra = ufe_idx(r);
        if (r != w) ufe_min(V.uf + c0 + lane, r);
    }
    const uint64_t below = (1ull << lane) - 1ull;
    for (int t0 = 0; t0 < items || pb.n > 0;) {
        if (t0 < items && pb.n < 64) {
            const int t = min(t0 + lane, items - 1);
            const int i = (t * irow) >> 16, e = t - i * nrow;
            const int la = from_lane(order, i), A = c0 + la;
            const int rA = from_lane(ra, la);
            int r = e <= k ? max(2 * e - 1, 0) : 0;  // own plane: offset -e is stored at 2e - 1
            if (dim == 3 && e > k) {
                const int f = e - 1 - k, d = (f * iwidth) >> 16;  // plane -(d + 1) is group 2d + 1
                r = (2 * d + 1) * width + f - d * width;
            }
            int Bf, Bl;
            row_cells(V, A, V.rows.at(A, r), &Bf, &Bl);
            // an unsafe cell is also paired with itself, by its own column's lane
            if (e == 0 && rA < 0) Bl = A;
            const int n = t0 + lane < items ? Bl - Bf + 1 : 0;  // at most kRowCells
            const uint64_t n1 = __ballot(n & 1), n2 = __ballot(n & 2), n4 = __ballot(n & 4);
            const int at = pb.n + __popcll(n1 & below) + 2 * __popcll(n2 & below) + 4 * __popcll(n4 & below);
            for (int u = 0; u < n; u++) pb.e[at + u] = ((uint32_t)la << 24) | (uint32_t)(Bf + u);
            pb.n += __popcll(n1) + 2 * __popcll(n2) + 4 * __popcll(n4);
            t0 += 64;
            wave_sync();
        }
        if (pb.n >= 64 || (t0 >= items && pb.n > 0)) {
            const int i = pb.n - 1 - lane;  // from the end: what stays needs no move
            const uint32_t e = pb.e[max(i, 0)];
            pb.n = max(pb.n - 64, 0);
            const int la = (int)(e >> 24), B = (int)(e & 0xffffffu);
            const int r0 = from_lane(ra, la);
            const uint64_t eb = ufe_now(V.uf, B);
            bool open = i >= 0 && eb != kUfNone && (ufe_idx(eb) != r0 || r0 < 0);
            bool hit = false, test = false;
            if (open && r0 >= 0 && ufe_is(eb)) {
                const uint64_t rb = ufe_root_now(V.uf, eb), r1 = ufe_root_now(V.uf, ufe_now(V.uf, r0));
                open = rb != r1;
                if (open) {
                    // all points of two cells of up to kFew, else the first cores
                    const int A = c0 + la;
                    const int csA = at(V.cstart, A), nA = at(V.cstart, A + 1) - csA, fA = at(V.fcore, A);
                    const int csB = at(V.cstart, B), nB = at(V.cstart, B + 1) - csB, fB = at(V.fcore, B);
                    const bool few = max(nA, nB) <= kFew;
                    float ax[kFew], ay[kFew], az[kFew];
                    bool ac[kFew];
#pragma unroll
                    for (int q = 0; q < kFew; q++) {
                        const int p = few ? csA + min(q, nA - 1) : fA;
                        ax[q] = at(V.sx, p);
                        ay[q] = dim > 1 ? at(V.sy, p) : 0.f;
                        az[q] = dim > 2 ? at(V.sz, p) : 0.f;
                        ac[q] = at(V.flags, p) & kFlagCore;
                    }
#pragma unroll
                    for (int q = 0; q < kFew; q++) {
                        const int p = few ? csB + min(q, nB - 1) : fB;
                        const float x = at(V.sx, p);
                        const float y = dim > 1 ? at(V.sy, p) : 0.f;
                        const float z = dim > 2 ? at(V.sz, p) : 0.f;
                        const bool bc = at(V.flags, p) & kFlagCore;
#pragma unroll
                        for (int o = 0; o < kFew; o++)
                            hit |= bc & ac[o] & (sqd(3, ax[o], ay[o], az[o], x, y, z) < V.eps2);
                    }
                    test = true;
                    if (hit) ufe_unite(V.uf, ufe_idx(r1), ufe_idx(rb));
                    open = !hit && !few;
                }
            }
            const int nu = __popcll(__ballot(hit));
            st.add(kStatMergeTests, __popcll(__ballot(test)));
            st.add(kStatMergePairs, nu);
            st.add(kStatUnites, nu);
            pair_push(far, open, la, B);
        }
        if (far.n > kPairCap - 64 || (t0 >= items && pb.n == 0 && far.n > 0)) {
            wave_sync();
            join_flush(V, c0, far, st);
        }
    }
}

// Walks the cell tiles of the launch's streams with safe cells, one per wave:
// tile(s, V, c0, ncell).
template <class ST, class F>
__device__ __forceinline__ void each_cell_tile(const BatchArgs &a, ST &st, F &&tile) {
    const int total = uni(ldc(a.ctile_pre[a.n]));
    const int nw = gridDim.x * kCellWaves;
    int s = 0;
    for (int g = uni(xcd_block(blockIdx.x, gridDim.x, a.xcd_groups & kXcdUnion) * kCellWaves + (threadIdx.x >> 6));
         g < total; g += nw) {
        s = uni(find_stream_from(a.ctile_pre, a.n, g, s));
        const StreamDev &S = a.s[s];
        if (merged_by_wave(a, ldc(S.dense_ok))) continue;
        stats_stream(a, st, s);
        tile(S, cell_view(S), (g - uni(ldc(a.ctile_pre[s]))) * a.cell_tile, ldc(ldc(S.mut)->ncell));
    }
    stats_flush(a, st);
}

// One launch: a tile's links, then its joins. Other waves' links may still be
// on their way when a wave compares roots; it then tests a pair that a later
// look would have found joined.
template <class ST>
__global__ __launch_bounds__(64 * kCellWaves) void k_merge_cells(BatchArgs a) {
    __shared__ int2 links[kCellWaves][kLinkCap];
    __shared__ uint32_t pairs[kCellWaves][kPairCap], rest[kCellWaves][kPairCap];
    const int wv = threadIdx.x >> 6;
    ST st;
    LinkBuf lb{links[wv], 0};
    PairBuf pb{pairs[wv], 0}, far{rest[wv], 0};
    each_cell_tile(a, st, [&](const StreamDev &S, const CellView &V, int c0, int ncell) {
        const int k = ldc(S.k), T = a.cell_tile;
        if (V.dim == 3) link_tile<3>(V, k, c0, T, ncell, lb, st);
        else if (V.dim == 2) link_tile<2>(V, k, c0, T, ncell, lb, st);
        else link_tile<1>(V, k, c0, T, ncell, lb, st);
        join_tile(V, k, c0, T, ncell, pb, far, st);
    });
}

// Range count, point-parallel form (large batches, where the device is
// saturated and per-query work matters more than coalescing): dense cells are
// core without counting (all pairs within eps); otherwise the LPQ lanes of a
// query count its neighbours (itself included) over its cell's stencil rows,
// each stopping once its own count reaches min_pts. Queries of one cell are
// adjacent and read the same candidates. D is the stream's dimension, so the
// distance test and the loads carry no per-candidate dimension selects.
//
// Walks by fours: a lane's rows, a group at a time, walked as one sequence of
// fours, each up to four candidates of one row by one 16-byte load per axis,
// kFours of them per round trip whatever the rows' lengths. Four t of a group
// lies in the last row i with pre[i] <= t (pre: the fours of the group's
// earlier rows; an empty row shares its pre with the next row, which
// overrides it) and starts at position base[i] + 4 * t; past the row's end it
// reads other candidates or up to three words past the window, which the
// coordinate arrays hold (kCandPad), and leaves them out.
//
// What bounds the walks is the work per candidate: finding its row and an
// address and a load per axis were 16 instructions of 26 when each candidate
// was found by itself, eight a round trip. A row of one or two cells fills half
// its fours, and still a four costs less than its candidates did. Count so and
// by fours: 64 streams 152 and 121 us, 24 served streams 82 and 56; outputs 137
// and 113, 71 and 72, one million points 76 and 73. One, three and four fours a
// round trip in the count: 137, 126 and 129 us at 64 streams; groups of 3, 4
// and 8 rows: 135, 128 and 125.
typedef float F4 __attribute__((ext_vector_type(4), aligned(4)));
constexpr int kFours = 2;
constexpr int kBorderRows = 8;  // rows per group of the outputs' walk (no early exit)

// The fours of a group of N rows, of `first + i * step`; past the last row none.
template <int N>
struct FourWalk {
    int base[N], pre[N], end[N];
    int n = 0;  // fours
    __device__ __forceinline__ FourWalk(const CellView &V, gptr<const uint64_t> rows, int first, int step) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int r = first + i * step;
            const uint64_t rw = r < V.R ? rows[V.rows.row(r)] : 0ull;
            const int rx = (int)(uint32_t)rw, ry = (int)(uint32_t)(rw >> 32);  // rx < ry, or both 0
            pre[i] = n;
            base[i] = rx - 4 * n;
            end[i] = ry;
            n += (ry - rx + 3) >> 2;
        }
    }
    // First position of four t, and how many candidates there are from it to
    // its row's end; past the last four (n > 0) the last one's, and none.
    __device__ __forceinline__ void at(int t, int *pos, int *left) const {
        const int tt = min(t, n - 1);
        int b = base[0], e = end[0];
#pragma unroll
        for (int i = 1; i < N; i++) {
            b = tt >= pre[i] ? base[i] : b;
            e = tt >= pre[i] ? end[i] : e;
        }
        *pos = b + 4 * tt;
        *left = t < n ? e - *pos : 0;
    }
};

template <int D>
struct Four {
    F4 x, y, z;
    __device__ __forceinline__ void load(const CellView &V, int pos) {
        x = *(gptr<const F4>)(V.sx + pos);
        if (D > 1) y = *(gptr<const F4>)(V.sy + pos);
        if (D > 2) z = *(gptr<const F4>)(V.sz + pos);
    }
    __device__ __forceinline__ float sqd_to(int v, float qx, float qy, float qz) const {
        return sqd(D, qx, qy, qz, x[v], D > 1 ? y[v] : 0.f, D > 2 ? z[v] : 0.f);
    }
};

// One lane's share of a query's stencil: rows first, first + step, ..., in
// groups of kRowGroup rows, nearest rows first. The count is checked
// against min_pts once per round trip.
template <int D>
__device__ __forceinline__ int count_walk(const CellView &V, int c, float qx, float qy, float qz, int first,
                                          int step, int &tests) {
    const int minpts = V.min_pts;
    const float e2 = V.eps2;
    int cnt = 0;
    const gptr<const uint64_t> rows = V.rows.of(c);
    for (int r0 = first; r0 < V.R; r0 += kRowGroup * step) {
        const FourWalk<kRowGroup> w(V, rows, r0, step);
        for (int t0 = 0; t0 < w.n; t0 += kFours) {
            Four<D> f[kFours];
            int left[kFours];
#pragma unroll
            for (int u = 0; u < kFours; u++) {
                int pos;
                w.at(t0 + u, &pos, &left[u]);
                f[u].load(V, pos);
            }
#pragma unroll
            for (int u = 0; u < kFours; u++) {
                tests += min(left[u], 4);
#pragma unroll
                for (int v = 0; v < 4; v++) cnt += (v < left[u]) & (f[u].sqd_to(v, qx, qy, qz) < e2);
            }
            if (cnt >= minpts) return cnt;
        }
    }
    return cnt;
}

template <int LPQ, int D>
__device__ __forceinline__ void count_vblock(const BatchArgs &a, const QueryLane<LPQ> &ql, int s,
                                             const CellView &V) {
    const int p = ql.p;
    const bool valid = p < ql.x.p1;
    const int minpts = V.min_pts;
    int cnt = 0;
    bool dense = false, safe = true;
    int c = 0;
    // the query's cell and coordinates, one round trip
    const uint32_t po = (uint32_t)(valid ? p : ql.x.p0) << 2;
    const int cv = ldo(V.pcell, po);
    const float qx = ldo(V.sx, po);
    const float qy = D > 1 ? ldo(V.sy, po) : 0.f;
    const float qz = D > 2 ? ldo(V.sz, po) : 0.f;
    arrived(qx);
    arrived(qy);
    arrived(qz);
    if (valid) {
        c = cv;
        const int cf = V.cflag[c];
        dense = cf & kCellDense;
        safe = cf & kCellSafe;
    }
    int tests = 0;
    if (valid && !dense) cnt = count_walk<D>(V, c, qx, qy, qz, ql.sub, LPQ, tests);
    if (a.stats) {
        const unsigned long long t = (unsigned long long)wave_sum(tests);
        const int nd = __popcll(__ballot(valid && dense && ql.sub == 0));
        const int nq = __popcll(__ballot(valid && !dense && ql.sub == 0));
        if (lane_id() == 0) {
            unsigned long long *st = a.stats + (size_t)s * kNumStats;
            atomicAdd(st + kStatCountTests, t);
            if (nd) atomicAdd(st + kStatDensePoints, (unsigned long long)nd);
            if (nq) atomicAdd(st + kStatQueries, (unsigned long long)nq);
        }
    }
    cnt = group_sum<LPQ>(cnt);
    if (valid && ql.sub == 0) {
        V.flags[p] = dense ? (kFlagCore | kFlagDense) : count_flags(cnt, minpts, safe);
        if (!safe) V.uf[V.W + p] = ufe(vslot(V, p), V.W + p);  // a core of an unsafe cell is an element
    }
}

template <int LPQ>
__global__ __launch_bounds__(64) void k_count_points(BatchArgs a) {
    const QueryLane<LPQ> ql = query_lane<LPQ>(a, blockIdx.x);
    const int s = uni(ql.x.s);
    const CellView V = cell_view(a.s[s]);
    if (V.dim == 3) count_vblock<LPQ, 3>(a, ql, s, V);
    else if (V.dim == 2) count_vblock<LPQ, 2>(a, ql, s, V);
    else count_vblock<LPQ, 1>(a, ql, s, V);
}

// Border / noise, point-parallel form (large batches): LPQ lanes per
// non-core point, which takes the minimum root among the cores within eps.
// The kernel also writes the cores' outputs (the root of each core's
// union-find element, found here: no separate flatten pass) and advances each
// stream's ring cursor, as the cell-parallel output kernel does. D is the
// stream's dimension.
//
// One lane's share of a non-core point's stencil in groups of
// kBorderRows rows (larger than the count's: no early exit here), without an
// early exit: the minimum root of the cores within eps. A candidate's flags
// and cell load only when it is within eps, and the cell's root only when it is
// not the cell of the last core found, whose root a safe cell's cores share
// (64 streams 139 -> 137 us, one million points 81 -> 76, 24 served 76 -> 71).
template <int D>
__device__ __forceinline__ int border_walk(const CellView &V, int c, float qx, float qy, float qz, int first,
                                           int step, int &tests) {
    const float e2 = V.eps2;
    int best = INT_MAX, seen = -1;
    const gptr<const uint64_t> rows = V.rows.of(c);
    for (int r0 = first; r0 < V.R; r0 += kBorderRows * step) {
        const FourWalk<kBorderRows> w(V, rows, r0, step);
        for (int t0 = 0; t0 < w.n; t0 += kFours) {
            Four<D> f[kFours];
            int pos[kFours], left[kFours];
#pragma unroll
            for (int u = 0; u < kFours; u++) {
                w.at(t0 + u, &pos[u], &left[u]);
                f[u].load(V, pos[u]);
            }
#pragma unroll
            for (int u = 0; u < kFours; u++) {
                tests += min(left[u], 4);
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if ((v < left[u]) & (f[u].sqd_to(v, qx, qy, qz) < e2)) {
                        const int p = pos[u] + v;
                        const int fl = ldo(V.flags, (uint32_t)p);
                        const int pc = ldo(V.pcell, (uint32_t)p << 2);
                        arrived(pc);
                        if ((fl & kFlagCore) && pc != seen) {
                            const uint64_t e = V.uf[pc];
                            if (e != kUfUnsafe) seen = pc;
                            best = min(best, core_cid(V, e, p));
                        }
                    }
            }
        }
    }
    return best;
}

template <int LPQ, int D>
__device__ __forceinline__ void border_vblock(const BatchArgs &a, const QueryLane<LPQ> &ql, int vb, int s,
                                              const CellView &V) {
    const int p = ql.p;
    // the query's flags, cell, coordinates and slot, one round trip
    const int pp = p < ql.x.p1 ? p : ql.x.p0;
    const uint32_t po = (uint32_t)pp << 2;
    const int qf = ldo(V.flags, (uint32_t)pp);
    const int c = ldo(V.pcell, po);
    const float qx = ldo(V.sx, po);
    const float qy = D > 1 ? ldo(V.sy, po) : 0.f;
    const float qz = D > 2 ? ldo(V.sz, po) : 0.f;
    const uint64_t qk = ldo(V.skey, po << 1);
    arrived(c);
    arrived(qx);
    arrived(qy);
    arrived(qz);
    arrived(qk);
    const IO io = a.use_io1 ? a.io1 : a.io[s];
    if (vb == ldc(a.pre_chunk[s]) * LPQ && lane_id() == 0) {  // the stream's first block
        StreamMut *m = ldc(a.s[s].mut);
        if (a.stats) a.stats[(size_t)s * kNumStats + kStatCells] += (unsigned long long)m->ncell;
        m->t = m->t + 1;
        m->u = m->u + 1 == ldc(a.s[s].units) ? 0 : m->u + 1;
    }
    if (p < ql.x.p1 && (qf & kFlagCore) && ql.sub == 0) {
        const int slot = (int)((uint32_t)qk & V.smask);
        gl(io.label)[slot] = 0;
        gl(io.cid)[slot] = core_cid(V, V.uf[c], pp);
    }
    const bool mine = p < ql.x.p1 && !(qf & kFlagCore);
    int best = INT_MAX;
    int tests = 0;
    if (mine && !known_noise(a, qf)) best = border_walk<D>(V, c, qx, qy, qz, ql.sub, LPQ, tests);
    if (a.stats) {
        const unsigned long long t = (unsigned long long)wave_sum(tests);
        if (lane_id() == 0 && t) atomicAdd(a.stats + (size_t)s * kNumStats + kStatBorderTests, t);
    }
    best = group_min<LPQ>(best);
    if (mine && ql.sub == 0) {
        const int slot = (int)((uint32_t)qk & V.smask);
        gl(io.label)[slot] = best != INT_MAX ? 1 : 2;
        gl(io.cid)[slot] = best != INT_MAX ? best : slot;
    }
}

template <int LPQ>
__global__ __launch_bounds__(64) void k_border_points(BatchArgs a) {
    const int vb = xcd_block(blockIdx.x, gridDim.x, a.xcd_groups & kXcdBorderPoints);
    const QueryLane<LPQ> ql = query_lane<LPQ>(a, vb);
    const int s = uni(ql.x.s);
    const CellView V = cell_view(a.s[s]);
    if (V.dim == 3) border_vblock<LPQ, 3>(a, ql, vb, s, V);
    else if (V.dim == 2) border_vblock<LPQ, 2>(a, ql, vb, s, V);
    else border_vblock<LPQ, 1>(a, ql, vb, s, V);
}

// Border / noise, point-parallel with regrouping (large batches): one wave per
// 64-position chunk, one lane per position. A core writes the root of its
// element at once; the chunk's non-core points are then regrouped 16 at a time
// onto four lanes each (a point's rank among the chunk's non-cores picks its
// group, its query passed through LDS), which split its stencil rows as in
// border_vblock. A core needs one lane and a non-core four, so a wave covers
// four times the positions of the four-lanes-per-position form with about as
// many round trips.
struct BorderQ {
    int c;
    float x, y, z;
    int slot;
};

template <int D>
__device__ __forceinline__ void border_chunk(const BatchArgs &a, const ChunkCtx &x, int g, int s, const CellView &V,
                                             BorderQ *lq) {
    const int lane = lane_id();
    const int p = x.p0 + lane;
    const bool valid = p < x.p1;
    // the query's flags, cell, coordinates and slot, one round trip
    const int pp = valid ? p : x.p0;
    const uint32_t po = (uint32_t)pp << 2;
    const int qf = ldo(V.flags, (uint32_t)pp);
    const int c = ldo(V.pcell, po);
    const float qx = ldo(V.sx, po);
    const float qy = D > 1 ? ldo(V.sy, po) : 0.f;
    const float qz = D > 2 ? ldo(V.sz, po) : 0.f;
    const uint64_t qk = ldo(V.skey, po << 1);
    arrived(c);
    arrived(qx);
    arrived(qy);
    arrived(qz);
    arrived(qk);
    const IO io = a.use_io1 ? a.io1 : a.io[s];
    if (g == ldc(a.pre_chunk[s]) && lane == 0) {  // the stream's first block
        StreamMut *m = ldc(a.s[s].mut);
        if (a.stats) a.stats[(size_t)s * kNumStats + kStatCells] += (unsigned long long)m->ncell;
        m->t = m->t + 1;
        m->u = m->u + 1 == ldc(a.s[s].units) ? 0 : m->u + 1;
    }
    const int slot = (int)((uint32_t)qk & V.smask);
    const bool core = valid && (qf & kFlagCore);
    if (core) {
        gl(io.label)[slot] = 0;
        gl(io.cid)[slot] = core_cid(V, V.uf[c], pp);
    }
    const bool noise = valid && known_noise(a, qf);
    if (noise) {
        gl(io.label)[slot] = 2;
        gl(io.cid)[slot] = slot;
    }
    const bool ask = valid && !core && !noise;
    const uint64_t nm = __ballot(ask);
    if (ask) lq[__popcll(nm & ((1ull << lane) - 1ull))] = BorderQ{c, qx, qy, qz, slot};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int nn = __popcll(nm);
    const int grp = lane >> 2, sub = lane & 3;
    int tests = 0;
    for (int b0 = 0; b0 < nn; b0 += 16) {
        const int i = b0 + grp;
        const bool have = i < nn;
        const BorderQ q = lq[have ? i : 0];
        int best = INT_MAX;
        if (have) best = border_walk<D>(V, q.c, q.x, q.y, q.z, sub, 4, tests);
        best = group_min<4>(best);
        if (have && sub == 0) {
            gl(io.label)[q.slot] = best != INT_MAX ? 1 : 2;
            gl(io.cid)[q.slot] = best != INT_MAX ? best : q.slot;
        }
    }
    if (a.stats) {
        const unsigned long long t = (unsigned long long)wave_sum(tests);
        if (lane == 0 && t) atomicAdd(a.stats + (size_t)s * kNumStats + kStatBorderTests, t);
    }
}

__global__ __launch_bounds__(64) void k_border_regroup(BatchArgs a) {
    __shared__ BorderQ lq[64];
    const int g = xcd_block(blockIdx.x, gridDim.x, a.xcd_groups & kXcdBorderPoints);
    const ChunkCtx x = chunk_of(a, g);
    const int s = uni(x.s);
    const CellView V = cell_view(a.s[s]);
    if (V.dim == 3) border_chunk<3>(a, x, g, s, V, lq);
    else if (V.dim == 2) border_chunk<2>(a, x, g, s, V, lq);
    else border_chunk<1>(a, x, g, s, V, lq);
}

// First core and union-find entry of every cell, after the point-parallel
// count: one lane per cell. Positions within a cell are in slot order, so the
// first core has the cell's minimum core slot. A dense cell's is its first
// point, and the others' flags are few (fewer than min_pts points, reach 1
// apart), read four at a time.
__global__ __launch_bounds__(64 * kCellWaves) void k_cell_cores(BatchArgs a) {
    const int total = uni(ldc(a.ctile_pre[a.n]));
    const int lane = lane_id();
    int s = 0;
    for (int g = uni(blockIdx.x * kCellWaves + (threadIdx.x >> 6)); g < total; g += gridDim.x * kCellWaves) {
        s = uni(find_stream_from(a.ctile_pre, a.n, g, s));
        const StreamDev &S = a.s[s];
        const CellView V = cell_view(S);
        const int c = (g - uni(ldc(a.ctile_pre[s]))) * a.cell_tile + lane;
        if (lane >= a.cell_tile || c >= ldc(ldc(S.mut)->ncell)) continue;
        const int cf = V.cflag[c], cs = V.cstart[c], ce = V.cstart[c + 1];
        int fc = (cf & kCellDense) ? cs : kNoCore;
        for (int i = cs; i < ce && fc == kNoCore; i += 4) {
            int f[4];
#pragma unroll
            for (int q = 0; q < 4; q++) f[q] = V.flags[min(i + q, ce - 1)];
#pragma unroll
            for (int q = 3; q >= 0; q--)
                if ((f[q] & kFlagCore) && i + q < ce) fc = i + q;
        }
        V.fcore[c] = fc;
        V.uf[c] = fc == kNoCore ? kUfNone : ((cf & kCellSafe) ? ufe(vslot(V, fc), c) : kUfUnsafe);
    }
}

// Plain device copy of 16-byte words: a kernel of known HBM traffic (reads and
// writes `n16` * 16 bytes) used to scale the profiler's byte counters.
__global__ __launch_bounds__(kTileThreads) void k_copy16(const int4 *__restrict__ src, int4 *__restrict__ dst,
                                                         size_t n16) {
    for (size_t i = (size_t)blockIdx.x * kTileThreads + threadIdx.x; i < n16; i += (size_t)gridDim.x * kTileThreads)
        dst[i] = src[i];
}

hipError_t launch_copy16(const void *src, void *dst, size_t n16, hipStream_t st) {
    if (n16 == 0) return hipSuccess;
    const size_t blocks = std::min<size_t>((n16 + kTileThreads - 1) / kTileThreads, 65536);
    hipLaunchKernelGGL(k_copy16, dim3((unsigned)blocks), dim3(kTileThreads), 0, st, (const int4 *)src, (int4 *)dst,
                       n16);
    return hipGetLastError();
}

// A list of copies in one launch: kSegWords words a block, each thread's loads
// all in flight before its stores. A copy between pinned host memory and the
// device runs as a kernel either way (the runtime's own takes 2.6-5 us for
// 20-40 KB), but submitting one costs the host 10-14 us, 16 streams' strides
// 150-170 us of a 345 us pipelined slide. The words go over the host link,
// 256 bytes per wave and load; the table is read once per block.
constexpr int kSegPer = 8;
constexpr int kSegWords = kTileThreads * kSegPer;

__global__ __launch_bounds__(kTileThreads) void k_copy_segs(const CopySeg *segs, int n, uint32_t words) {
    __shared__ CopySeg seg[kMaxBatch];
    const uint32_t w0 = blockIdx.x * kSegWords, w1 = min(w0 + kSegWords, words);
    // the block's copies: from the one holding w0 to the one holding w1 - 1
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (segs[mid].first <= w0) lo = mid;
        else hi = mid;
    }
    const int s0 = uni(lo);
    int ns = 0;  // of them, staged kMaxBatch at a time
    for (int s = s0; s < n; s += ns) {
        ns = min(n - s, kMaxBatch);
        __syncthreads();
        for (int i = threadIdx.x; i < ns; i += kTileThreads) seg[i] = segs[s + i];
        __syncthreads();
        if (seg[0].first >= w1) break;
        const uint32_t end = seg[ns - 1].first + seg[ns - 1].words;
        uint32_t v[kSegPer];
        uint32_t *to[kSegPer];
#pragma unroll
        for (int q = 0; q < kSegPer; q++) {
            const uint32_t w = w0 + q * kTileThreads + threadIdx.x;
            to[q] = nullptr;
            if (w < w1 && w >= seg[0].first && w < end) {
                int l = 0, h = ns;
                while (h - l > 1) {
                    const int mid = (l + h) >> 1;
                    if (seg[mid].first <= w) l = mid;
                    else h = mid;
                }
                v[q] = ((const uint32_t *)seg[l].src)[w - seg[l].first];
                to[q] = (uint32_t *)seg[l].dst + (w - seg[l].first);
            }
        }
#pragma unroll
        for (int q = 0; q < kSegPer; q++)
            if (to[q]) *to[q] = v[q];
    }
}

hipError_t launch_copy_segs(const CopySeg *segs, int n, uint32_t words, hipStream_t st) {
    const unsigned blocks = (unsigned)(((uint64_t)words + kSegWords - 1) / kSegWords);
    hipLaunchKernelGGL(k_copy_segs, dim3(blocks), dim3(kTileThreads), 0, st, segs, n, words);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// launchers

#define RTDBS_LAUNCH(kernel, grid, block, ...)                        \
    do {                                                              \
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, st, __VA_ARGS__); \
        hipError_t e_ = hipGetLastError();                            \
        if (e_ != hipSuccess) return e_;                              \
    } while (0)

static inline hipError_t mark(hipEvent_t *ev, uint32_t mask, int idx, hipStream_t st) {
    if (!ev || !((mask >> (idx / 2)) & 1u)) return hipSuccess;
    return hipEventRecord(ev[idx], st);
}

// Launches `kernel`; with events, they take the dispatch's own timestamps.
template <class K, class... Args>
static hipError_t launch_timed(K kernel, int grid, int block, hipStream_t st, hipEvent_t e0, hipEvent_t e1,
                               Args... args) {
    if (e0) hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, st, e0, e1, 0, args...);
    else hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, st, args...);
    return hipGetLastError();
}

hipError_t launch_slide(const BatchArgs &a, const LaunchShape &sh, hipStream_t st, hipEvent_t *ev,
                        uint32_t phase_mask) {
    hipError_t e;
#define PH_BEGIN(ph) if ((e = mark(ev, phase_mask, 2 * (ph), st)) != hipSuccess) return e
#define PH_END(ph) if ((e = mark(ev, phase_mask, 2 * (ph) + 1, st)) != hipSuccess) return e
    // per-phase times of the window update are of its separate kernels
    constexpr uint32_t kUpdatePhases =
        (1u << kPhStrideSort) | (1u << kPhMerge) | (1u << kPhMergeFinal) | (1u << kPhCells);
    if (sh.small_update && !(ev && (phase_mask & kUpdatePhases))) {
        if (sh.small_update == 1) RTDBS_LAUNCH(k_update_small<1>, a.n, kSmallThreads, a);
        else if (sh.small_update == 2) RTDBS_LAUNCH(k_update_small<2>, a.n, kSmallThreads, a);
        else RTDBS_LAUNCH(k_update_small<kSmallPer>, a.n, kSmallThreads, a);
    } else {
    PH_BEGIN(kPhStrideSort);
    RTDBS_LAUNCH(k_sort_expire, sh.stiles * kSortParts + sh.wtiles, kTileThreads, a);
    PH_END(kPhStrideSort);
    PH_BEGIN(kPhMerge);
    if (sh.rank_split) {
        const int rb = sh.stiles * (kTile / 64);
        RTDBS_LAUNCH(k_rank<4>, rb + sh.wtiles, kTileThreads, a, rb);
    } else {
        const int rb = sh.stiles * (kTile / kTileThreads);
        RTDBS_LAUNCH(k_rank<1>, rb + sh.wtiles, kTileThreads, a, rb);
    }
    PH_END(kPhMerge);
    PH_BEGIN(kPhMergeFinal);
    RTDBS_LAUNCH(k_merge_final, sh.wtiles, kTileThreads, a);
    PH_END(kPhMergeFinal);
    PH_BEGIN(kPhCells);
    RTDBS_LAUNCH(k_cells, sh.wtiles, kTileThreads, a);
    PH_END(kPhCells);
    }
    PH_BEGIN(kPhRows);
    RTDBS_LAUNCH(k_rows, sh.rows_blocks + 1, kTileThreads, a);
    PH_END(kPhRows);
    {
        // The range-count kernel is timed by its own dispatch: the events take
        // the kernel's begin and end timestamps, with no marker packets of
        // their own between it and its neighbours.
        const bool timed = ev && ((phase_mask >> kPhCount) & 1u);
        const hipEvent_t e0 = timed ? ev[2 * kPhCount] : nullptr, e1 = timed ? ev[2 * kPhCount + 1] : nullptr;
        if (sh.count_cell && a.stats)
            e = launch_timed(k_count<WaveStats>, sh.cellpar_blocks, 64 * kCellWaves, st, e0, e1, a);
        else if (sh.count_cell)
            e = launch_timed(k_count<NoStats>, sh.cellpar_blocks, 64 * kCellWaves, st, e0, e1, a);
        else if (sh.lpq >= 4) e = launch_timed(k_count_points<4>, sh.chunks * 4, 64, st, e0, e1, a);
        else if (sh.lpq == 2) e = launch_timed(k_count_points<2>, sh.chunks * 2, 64, st, e0, e1, a);
        else e = launch_timed(k_count_points<1>, sh.chunks, 64, st, e0, e1, a);
        if (e != hipSuccess) return e;
    }
    PH_BEGIN(kPhUnion);
    // the cell-parallel count wrote every cell's first core and entry; after
    // the point-parallel count a pass over the cells does
    if (!sh.count_cell) RTDBS_LAUNCH(k_cell_cores, sh.link_blocks, 64 * kCellWaves, a);
    if (sh.link && a.stats) RTDBS_LAUNCH(k_merge_cells<WaveStats>, sh.link_blocks, 64 * kCellWaves, a);
    else if (sh.link) RTDBS_LAUNCH(k_merge_cells<NoStats>, sh.link_blocks, 64 * kCellWaves, a);
    if (sh.by_wave && a.stats) RTDBS_LAUNCH(k_union<WaveStats>, sh.cellpar_blocks, 64 * kCellWaves, a);
    else if (sh.by_wave) RTDBS_LAUNCH(k_union<NoStats>, sh.cellpar_blocks, 64 * kCellWaves, a);
    PH_END(kPhUnion);
    PH_BEGIN(kPhBorder);
    if (sh.cellpar && a.stats) RTDBS_LAUNCH(k_border<WaveStats>, sh.cellpar_blocks, 64 * kCellWaves, a);
    else if (sh.cellpar) RTDBS_LAUNCH(k_border<NoStats>, sh.cellpar_blocks, 64 * kCellWaves, a);
    else if (sh.border_regroup) RTDBS_LAUNCH(k_border_regroup, sh.chunks, 64, a);
    else if (sh.lpq_border >= 4) RTDBS_LAUNCH(k_border_points<4>, sh.chunks * 4, 64, a);
    else if (sh.lpq_border == 2) RTDBS_LAUNCH(k_border_points<2>, sh.chunks * 2, 64, a);
    else RTDBS_LAUNCH(k_border_points<1>, sh.chunks, 64, a);
    PH_END(kPhBorder);
#undef PH_BEGIN
#undef PH_END
    return hipSuccess;
}

hipError_t launch_bounds_of(const float *in, int32_t W, int32_t dim, float *bnd, hipStream_t st) {
    RTDBS_LAUNCH(k_bounds, kBoundBlocks, kTileThreads, in, W, dim, bnd);
    return hipSuccess;
}

hipError_t launch_window_out(const BatchArgs &a, int32_t W, float *out, int32_t *bad, hipStream_t st) {
    RTDBS_LAUNCH(k_window_out, (W + kTileThreads - 1) / kTileThreads, kTileThreads, a, out, bad);
    return hipSuccess;
}

hipError_t launch_init(const BatchArgs &a, int32_t W, int32_t t, int32_t u, hipStream_t st) {
    const int runs = (int)(((long long)W + kTile - 1) / kTile);
    const int tiles = (int)(((long long)W + kWTile - 1) / kWTile);
    int passes = 0;
    while ((1ll << passes) < runs) passes++;
    if (passes == 0) {
        RTDBS_LAUNCH(k_init_tiles<true>, runs, kInitThreads, a, 1, t, u);
        return hipSuccess;
    }
    RTDBS_LAUNCH(k_init_tiles<false>, runs, kInitThreads, a, (passes - 1) & 1, t, u);
    for (int p = 0; p + 1 < passes; p++)
        RTDBS_LAUNCH(k_init_merge<false>, tiles, kTileThreads, a, kTile << p, (passes - 1 - p) & 1);
    RTDBS_LAUNCH(k_init_merge<true>, tiles, kTileThreads, a, kTile << (passes - 1), 0);
    return hipSuccess;
}

}  // namespace rtdbs
