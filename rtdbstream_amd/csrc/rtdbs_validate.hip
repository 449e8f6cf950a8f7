// On-device brute-force DBSCAN of one window: every pair of points is tested.
// It is the large-window validator of the slide step. It plays the role of the
// reference's own GPU check path: cluster_with_cuda and find_neighbors_t /
// find_cores_t / set_cluster_id_op_t / post_cluster_t (util.cpp:357-381,
// aabb.cu:150-261).
// It uses the same FP32 distance predicate as the slide kernels (sqd: the
// reference's un-contracted order, d2 < fl32(eps*eps)) and the same output
// rules. It shares no grid, sorting or cell logic with them: its candidates
// are all n points.
//   nn    - neighbours within eps, the point itself included (find_neighbors_t)
//   label - 0 core (nn >= min_pts), 1 border, 2 noise (find_cores_t)
//   cid   - cores: the minimum index of their cluster's cores (union-find
//           hooking the larger root under the smaller, dbscan.cu:22-43, then
//           post_cluster_t); borders: the minimum cluster id among the cores
//           within eps; noise: its own index.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <mutex>
#include <vector>

#include "rtdbs.h"
#include "rtdbs_devfn.h"
#include "rtdbs_host.h"

namespace rtdbs {

// Scratch of rtdbs_bruteforce_noalloc: union-find parents [0, kNoAllocMax)
// and, when the caller passes no nn array, neighbour counts [kNoAllocMax,
// 2 * kNoAllocMax), then one counter. One copy per GPU, held until the
// process ends (8 MiB).
constexpr int64_t kNoAllocMax = int64_t(1) << 20;
static __device__ __align__(256) int32_t scratch[2 * kNoAllocMax + 64];

namespace {

constexpr int kBfThreads = 256;
constexpr int kBfWaves = kBfThreads / 64;
constexpr int kBfGroup = 8;      // candidates read together
constexpr int kBfHitGroup = 4;   // the same where hits are queued
constexpr int kBfHits = 2048;    // hits queued per wave: a group's most (4 x 4 x 64) fits in half
constexpr int kMaxDevices = 64;

struct BfArgs {
    const float *pts;  // n points, dim floats each, point-major
    int n, dim, min_pts;
    float e2;
    int32_t *nn, *parent, *label, *cid;
    int32_t *nopen;  // number of non-core points, listed in `label` until the borders are found
    int chunk;       // candidates per wave
};

// How a pass over all pairs is laid out. A wave holds 64 * Q queries, Q per
// lane in registers, and walks `chunk` candidates. The candidates are the same
// for the whole wave, so they come through scalar loads (kBfGroup points at a
// time) and enter the distance test as scalar operands: no LDS, and no vector
// memory instruction in the loop, which is bound by vector issue (8 operations
// for a 3-D distance, one compare, one count). The four waves of a block take
// the same queries and adjacent candidate chunks; a launch has a block for
// every (query group, 4 chunks) pair: thousands for a window of tens of
// thousands of points.
struct BfUnit {
    int q0;      // first query
    int c0, c1;  // this wave's candidates
};

__device__ __forceinline__ BfUnit bf_unit(const BfArgs &a, int group, int chunk4, int per_group) {
    const int wv = uni(threadIdx.x >> 6);
    BfUnit u;
    u.q0 = group * per_group;
    u.c0 = (int)min(((long long)chunk4 * kBfWaves + wv) * a.chunk, (long long)a.n);
    u.c1 = u.c0 < a.n ? (int)min((long long)u.c0 + a.chunk, (long long)a.n) : u.c0;
    return u;
}

template <int D>
struct BfPoint {
    float x, y, z;
};

template <int D>
__device__ __forceinline__ BfPoint<D> bf_query(const BfArgs &a, int i) {
    const gptr<const float> p = gl(a.pts) + (size_t)i * D;
    BfPoint<D> q;
    q.x = p[0];
    q.y = D > 1 ? p[1] : 0.f;
    q.z = D > 2 ? p[2] : 0.f;
    return q;
}

// Calls visit(j, x, y, z) for every candidate j in [c0, c1), coordinates in
// scalar registers, and after() at least once per G candidates.
template <int D, int G, class Visit, class After>
__device__ __forceinline__ void bf_walk(const float *pts, int c0, int c1, Visit &&visit, After &&after) {
    typedef const __attribute__((address_space(4))) float *cptr;
    int j = c0;
    for (; c1 - j >= G; j += G) {
        const cptr p = (cptr)(pts + (size_t)j * D);
        float v[G * D];
#pragma unroll
        for (int k = 0; k < G * D; k++) v[k] = p[k];
#pragma unroll
        for (int k = 0; k < G; k++)
            visit(j + k, v[k * D], D > 1 ? v[k * D + (D > 1)] : 0.f, D > 2 ? v[k * D + 2 * (D > 2)] : 0.f);
        after();
    }
    for (; j < c1; j++) {
        const cptr p = (cptr)(pts + (size_t)j * D);
        visit(j, p[0], D > 1 ? p[D > 1] : 0.f, D > 2 ? p[2 * (D > 2)] : 0.f);
    }
    after();
}

__global__ __launch_bounds__(kBfThreads) void k_bf_init(BfArgs a) {
    const int i = blockIdx.x * kBfThreads + threadIdx.x;
    if (i == 0) *a.nopen = 0;
    if (i >= a.n) return;
    a.nn[i] = 0;
    a.parent[i] = i;
}

// Neighbour counts. The waves of a block add their counts in LDS, so a
// (query, 4 chunks) pair costs one atomic.
template <int Q, int D>
__global__ __launch_bounds__(kBfThreads) void k_bf_count(BfArgs a) {
    __shared__ int part[kBfWaves][Q * 64];
    const BfUnit u = bf_unit(a, blockIdx.x, blockIdx.y, Q * 64);
    const int lane = lane_id(), wv = threadIdx.x >> 6;
    BfPoint<D> q[Q];
    int cnt[Q];
#pragma unroll
    for (int r = 0; r < Q; r++) {
        q[r] = bf_query<D>(a, min(u.q0 + r * 64 + lane, a.n - 1));
        cnt[r] = 0;
    }
    const float e2 = a.e2;
    bf_walk<D, kBfGroup>(a.pts, uni(u.c0), uni(u.c1), [&](int, float x, float y, float z) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < Q; r++) cnt[r] += sqd(D, q[r].x, q[r].y, q[r].z, x, y, z) < e2;
    }, [] {});
#pragma unroll
    for (int r = 0; r < Q; r++) part[wv][r * 64 + lane] = cnt[r];
    __syncthreads();
    for (int k = threadIdx.x; k < Q * 64; k += kBfThreads) {
        int s = 0;
#pragma unroll
        for (int w = 0; w < kBfWaves; w++) s += part[w][k];
        if (s && k < a.n - u.q0) atomicAdd(a.nn + u.q0 + k, s);
    }
}

// Pairs within eps found by one wave, collected in LDS (query within the wave
// in the upper 8 bits, candidate within the chunk below; a chunk holds far
// fewer than 2^24) and handled 64 at a time, one per lane, so that the
// dependent loads of 64 hits overlap.
struct BfHits {
    uint32_t *e;
    int n;  // uniform
};

__device__ __forceinline__ void bf_push(BfHits &h, bool hit, int lq, int jo) {
    const uint64_t m = __ballot(hit);
    if (m == 0ull) return;
    if (hit) h.e[h.n + __popcll(m & ((1ull << lane_id()) - 1ull))] = ((uint32_t)lq << 24) | (uint32_t)jo;
    h.n += __popcll(m);
}

// handle(query within the wave, candidate within the chunk) for every hit
// queued, 64 at a time.
template <class Handle>
__device__ __forceinline__ void bf_flush(BfHits &h, Handle &&handle) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int k = lane_id(); k < h.n; k += 64) handle((int)(h.e[k] >> 24), (int)(h.e[k] & 0xffffffu));
    __builtin_amdgcn_wave_barrier();
    h.n = 0;
}

// Core-core unions: each core i unites with every core j < i within eps, so
// every pair is tested once.
template <int Q, int D>
__global__ __launch_bounds__(kBfThreads) void k_bf_union(BfArgs a) {
    __shared__ uint32_t hits[kBfWaves][kBfHits];
    const BfUnit u = bf_unit(a, blockIdx.x, blockIdx.y, Q * 64);
    const int lane = lane_id();
    const int qlast = (int)min((long long)u.q0 + Q * 64, (long long)a.n) - 1;
    const int c0 = uni(u.c0), c1 = uni(min(u.c1, qlast));  // candidates below the wave's last query
    if (c0 >= c1) return;
    BfPoint<D> q[Q];
    int qi[Q];  // the query's index, -1 when it is no core: no candidate is below it
    uint64_t any = 0;
#pragma unroll
    for (int r = 0; r < Q; r++) {
        const int ii = min(u.q0 + r * 64 + lane, a.n - 1);
        q[r] = bf_query<D>(a, ii);
        qi[r] = r * 64 + lane < a.n - u.q0 && a.nn[ii] >= a.min_pts ? ii : -1;
        any |= __ballot(qi[r] >= 0);
    }
    if (any == 0ull) return;
    BfHits h{hits[threadIdx.x >> 6], 0};
    auto handle = [&](int lq, int jo) {
        if (a.nn[c0 + jo] >= a.min_pts) uf_unite(a.parent, u.q0 + lq, c0 + jo);
    };
    const float e2 = a.e2;
    bf_walk<D, kBfHitGroup>(a.pts, c0, c1, [&](int j, float x, float y, float z) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < Q; r++)
            bf_push(h, (sqd(D, q[r].x, q[r].y, q[r].z, x, y, z) < e2) & (j < qi[r]), r * 64 + lane, j - c0);
    }, [&] { if (h.n > kBfHits / 2) bf_flush(h, handle); });
    bf_flush(h, handle);
}

// Cluster ids of the cores; the non-core points are listed in `label`.
__global__ __launch_bounds__(kBfThreads) void k_bf_flatten(BfArgs a) {
    const int i = blockIdx.x * kBfThreads + threadIdx.x;
    const bool v = i < a.n;
    const bool core = v && a.nn[i] >= a.min_pts;
    if (v) a.cid[i] = core ? uf_find(a.parent, i) : INT_MAX;
    const uint64_t m = __ballot(v && !core);
    if (m == 0ull) return;
    const int lead = __ffsll((unsigned long long)m) - 1;
    int base = 0;
    if (lane_id() == lead) base = atomicAdd(a.nopen, __popcll(m));
    base = __builtin_amdgcn_readlane(base, lead);
    if (v && !core) a.label[base + __popcll(m & ((1ull << lane_id()) - 1ull))] = i;
}

// Borders: the minimum cluster id among the cores within eps, for the listed
// non-core points. A persistent grid: their number is known on the device.
template <int Q, int D>
__global__ __launch_bounds__(kBfThreads) void k_bf_border(BfArgs a, int chunks4) {
    __shared__ uint32_t hits[kBfWaves][kBfHits];
    const int lane = lane_id();
    const int nopen = uni(*a.nopen);
    const long long units = (long long)((nopen + (Q * 64 - 1)) / (Q * 64)) * chunks4;
    const float e2 = a.e2;
    for (long long b = blockIdx.x; b < units; b += gridDim.x) {
        const BfUnit u = bf_unit(a, (int)(b / chunks4), (int)(b % chunks4), Q * 64);
        const int c0 = uni(u.c0), c1 = uni(u.c1);
        BfPoint<D> q[Q];
        bool mine[Q];
#pragma unroll
        for (int r = 0; r < Q; r++) {
            const int k = u.q0 + r * 64 + lane;
            q[r] = bf_query<D>(a, a.label[min(k, nopen - 1)]);
            mine[r] = k < nopen;
        }
        BfHits h{hits[threadIdx.x >> 6], 0};
        auto handle = [&](int lq, int jo) {
            if (a.nn[c0 + jo] >= a.min_pts) atomicMin(a.cid + a.label[u.q0 + lq], a.cid[c0 + jo]);
        };
        bf_walk<D, kBfHitGroup>(a.pts, c0, c1, [&](int j, float x, float y, float z) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < Q; r++)
                bf_push(h, (sqd(D, q[r].x, q[r].y, q[r].z, x, y, z) < e2) & mine[r], r * 64 + lane, j - c0);
        }, [&] { if (h.n > kBfHits / 2) bf_flush(h, handle); });
        bf_flush(h, handle);
    }
}

__global__ __launch_bounds__(kBfThreads) void k_bf_label(BfArgs a) {
    const int i = blockIdx.x * kBfThreads + threadIdx.x;
    if (i >= a.n) return;
    if (a.nn[i] >= a.min_pts) {
        a.label[i] = 0;
        return;
    }
    const int c = a.cid[i];
    a.label[i] = c != INT_MAX ? 1 : 2;
    if (c == INT_MAX) a.cid[i] = i;
}

template <int Q, int D>
hipError_t launch_bf_dim(BfArgs a, hipStream_t st) {
    const int blocks = (a.n + kBfThreads - 1) / kBfThreads;
    const int groups = (int)(((long long)a.n + Q * 64 - 1) / (Q * 64));
    // candidates per wave: waves enough for about 48 of them per SIMD (even
    // shares without a long last round), 32 to 256 candidates each (a longer
    // walk saves atomics and query loads, a shorter one latency in small
    // windows); more only where the grid's second axis would run out
    const long long waves = (long long)device_cus() * 4 * 48;
    long long chunk = std::min(std::max((long long)a.n * groups / waves, 32ll), 256ll);
    chunk = std::max(chunk, (long long)a.n / (65535ll * kBfWaves) + 1);
    a.chunk = (int)((chunk + kBfGroup - 1) / kBfGroup * kBfGroup);
    const int chunks4 = (int)(((long long)a.n + a.chunk * kBfWaves - 1) / (a.chunk * kBfWaves));
    const dim3 th(kBfThreads), pairs(groups, chunks4);
    hipLaunchKernelGGL(k_bf_init, dim3(blocks), th, 0, st, a);
    hipLaunchKernelGGL((k_bf_count<Q, D>), pairs, th, 0, st, a);
    hipLaunchKernelGGL((k_bf_union<Q, D>), pairs, th, 0, st, a);
    hipLaunchKernelGGL(k_bf_flatten, dim3(blocks), th, 0, st, a);
    const long long all = (long long)groups * chunks4;
    hipLaunchKernelGGL((k_bf_border<Q, D>), dim3((unsigned)std::min(all, (long long)device_cus() * 8)), th, 0, st, a,
                       chunks4);
    hipLaunchKernelGGL(k_bf_label, dim3(blocks), th, 0, st, a);
    return hipGetLastError();
}

// The launches of one validation, in order, on `st`. Four queries per lane
// share each candidate's loads and loop; windows of up to 8192 points take one
// instead, for four times the waves (8192 3-D points: 305 us with one, 371 us
// with four).
hipError_t launch_bf(const BfArgs &a, hipStream_t st) {
    const bool small = a.n <= 8192;
    switch (a.dim) {
    case 1: return small ? launch_bf_dim<1, 1>(a, st) : launch_bf_dim<4, 1>(a, st);
    case 2: return small ? launch_bf_dim<1, 2>(a, st) : launch_bf_dim<4, 2>(a, st);
    default: return small ? launch_bf_dim<1, 3>(a, st) : launch_bf_dim<4, 3>(a, st);
    }
}

int check_bf_args(int32_t dim, float eps, int32_t min_pts, int64_t n) {
    if (dim < 1 || dim > 3) return fail(RTDBS_EINVAL, "dim must be 1, 2 or 3 (got %d)", dim);
    if (!(eps > 0.0f) || !(eps < INFINITY)) return fail(RTDBS_EINVAL, "eps must be finite and > 0");
    if (min_pts < 1) return fail(RTDBS_EINVAL, "min_pts must be >= 1 (got %d)", min_pts);
    if (n < 1 || n > (int64_t)INT_MAX - kBfThreads) return fail(RTDBS_EINVAL, "n out of range (got %lld)", (long long)n);
    return RTDBS_OK;
}

#define BFCHK(expr)                                                                  \
    do {                                                                             \
        hipError_t e_ = (expr);                                                      \
        if (e_ != hipSuccess) {                                                      \
            rc = fail(RTDBS_EHIP, "%s failed: %s", #expr, hipGetErrorString(e_));    \
            goto done;                                                               \
        }                                                                            \
    } while (0)

// Device address of this GPU's scratch array, looked up once per device with
// the device current. Host code uses only this address, never the array's
// name (which is a host-side stand-in, not a device address).
int scratch_ptr(int32_t **out) {
    static std::mutex mu;
    static int32_t *ptr[kMaxDevices] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(RTDBS_EHIP, "hipGetDevice failed: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return fail(RTDBS_EHIP, "device %d beyond the %d supported", dev, kMaxDevices);
    std::lock_guard<std::mutex> lk(mu);
    if (!ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(RTDBS_EHIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
        ptr[dev] = (int32_t *)p;
    }
    *out = ptr[dev];
    return RTDBS_OK;
}

}  // namespace
}  // namespace rtdbs

using namespace rtdbs;

extern "C" int rtdbs_bruteforce(int32_t dim, float eps, int32_t min_pts, const float *points, int64_t n,
                                int32_t *label, int32_t *cid, int32_t *nn) {
    int rc = check_bf_args(dim, eps, min_pts, n);
    if (rc) return rc;
    if (!points || !label || !cid) return fail(RTDBS_EINVAL, "NULL argument");
    const size_t N = (size_t)n;
    char *mem = nullptr;
    BfArgs a{};
    BFCHK(hipMalloc((void **)&mem, N * (size_t)dim * 4 + (4 * N + 1) * 4));
    a.pts = (const float *)mem;
    a.nn = (int32_t *)(mem + N * (size_t)dim * 4);
    a.parent = a.nn + N;
    a.label = a.parent + N;
    a.cid = a.label + N;
    a.nopen = a.cid + N;
    a.n = (int)n;
    a.dim = dim;
    a.min_pts = min_pts;
    a.e2 = eps * eps;  // fl32(eps*eps), as the reference's radius2 (dbscan.cpp:41)
    BFCHK(hipMemcpy(mem, points, N * (size_t)dim * 4, hipMemcpyHostToDevice));
    BFCHK(launch_bf(a, 0));
    BFCHK(hipMemcpy(label, a.label, N * 4, hipMemcpyDeviceToHost));
    BFCHK(hipMemcpy(cid, a.cid, N * 4, hipMemcpyDeviceToHost));
    if (nn) BFCHK(hipMemcpy(nn, a.nn, N * 4, hipMemcpyDeviceToHost));
done:
    if (mem) (void)hipFree(mem);
    return rc;
}

extern "C" int rtdbs_bruteforce_noalloc(int32_t dim, float eps, int32_t min_pts, const float *points_dev, int64_t n,
                                        int32_t *label_dev, int32_t *cid_dev, int32_t *nn_dev) {
    int rc = check_bf_args(dim, eps, min_pts, n);
    if (rc) return rc;
    if (n > kNoAllocMax)
        return fail(RTDBS_EINVAL, "n = %lld exceeds the %lld points the allocation-free validator's scratch holds",
                    (long long)n, (long long)kNoAllocMax);
    if (!points_dev || !label_dev || !cid_dev) return fail(RTDBS_EINVAL, "NULL argument");
    int32_t *scr = nullptr;
    rc = scratch_ptr(&scr);
    if (rc) return rc;
    BfArgs a{};
    a.pts = points_dev;
    a.n = (int)n;
    a.dim = dim;
    a.min_pts = min_pts;
    a.e2 = eps * eps;  // fl32(eps*eps), as the reference's radius2 (dbscan.cpp:41)
    a.parent = scr;  // every entry < n is written by the count kernel before it is read
    a.nn = nn_dev ? nn_dev : scr + kNoAllocMax;
    a.nopen = scr + 2 * kNoAllocMax;
    a.label = label_dev;
    a.cid = cid_dev;
    hipError_t e = launch_bf(a, 0);
    if (e == hipSuccess) e = hipStreamSynchronize(0);
    if (e != hipSuccess) return fail(RTDBS_EHIP, "validator launch failed: %s", hipGetErrorString(e));
    return RTDBS_OK;
}
