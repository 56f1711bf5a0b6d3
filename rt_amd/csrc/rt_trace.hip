// rt_trace.hip -- fused per-scheme trace kernel and the C ABI of include/rt_hip.h.
//
// One launch replaces the reference's per-surface engine calls of
// Scheme::run (common-lib/scheme.cpp:983-1046): every lane owns one ray in
// registers from generation to the CCD, the packed surface table is read
// through uniform (scalar) loads and the spline pool is staged in LDS.  No
// host round trip, no Rearrange: a lost ray is masked, not compacted.
//
// Build decisions (differences from cuda_engine, each restated in the CPU
// oracle so parity is exact up to rounding):
//   D2  lost-ray counts are exact (wave ballots), not racy ++
//   D3  spline second derivatives by the serial recurrence (host)
//   D4  toric intersection by Newton on the documented F (surface.cpp:56-61)
//   D5  toric grating groove vector uses dFdZ*dFdZ (surface.cu:1438,1487)
//   D6  c == 0 aspheres go through the conic Newton; counters reset per ray
//   D7  one numerically stable quadratic root for every conic (incl. k = -1)
//   D8  the conic root is chosen by sign(c) as in surface.cu:240-244
//   D10 CCD accumulation uses atomics with a bounds check
//   D12 wavelength grids use the global ray index
//   D14 Philox4x32-10 keyed by a 64-bit seed, counter = ray index
//   D15 rectangular random beams are generated
//   D18 toric asphere derivative keeps its factor Y
//   D19 a one-sample uniform wavelength grid is range[0]
//   D20 a lost ray is frozen at the state it was lost in
#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <string>
#include <algorithm>
#include <mutex>
#include <vector>

#include "rt_device.h"
#include "rt_host.h"
#include "rt_jit.h"

using rt::Ray;

static thread_local const char* g_last_kernel = "none";

// --------------------------------------------------------------- errors
static thread_local std::string g_last_error;

int rt_set_error(int code, const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}
#define set_error rt_set_error

// ------------------------------------------------------- working buffers

int WorkBufs::ensure(Slot s, size_t bytes) {
    if (p[s] && have[s] >= bytes) return RT_OK;
    // geometric growth, so a sequence of growing calls allocates O(log) buffers
    return fresh(s, std::max(bytes, have[s] + have[s] / 2));
}

int WorkBufs::ensure_together(std::initializer_list<Part> parts) {
    size_t total = 0;
    bool none = true;
    for (const Part& q : parts) {
        total += (q.bytes + 255) / 256 * 256;
        none = none && !p[q.slot];
    }
    if (!none) {
        for (const Part& q : parts) {
            const int rc = ensure(q.slot, q.bytes);
            if (rc != RT_OK) return rc;
        }
        return RT_OK;
    }
    void* base = nullptr;
    if (hipMalloc(&base, total ? total : 8) != hipSuccess) {
        (void)hipGetLastError();
        return set_error(RT_ERR_BAD_ALLOC, "hipMalloc of %zu bytes of working memory failed", total);
    }
    owned.push_back(base);
    char* at = (char*)base;
    for (const Part& q : parts) {
        p[q.slot] = at;
        have[q.slot] = (q.bytes + 255) / 256 * 256;
        at += have[q.slot];
    }
    return RT_OK;
}

int WorkBufs::fresh(Slot s, size_t want) {
    void* q = nullptr;
    if (hipMalloc(&q, want ? want : 8) != hipSuccess) {
        (void)hipGetLastError();
        return set_error(RT_ERR_BAD_ALLOC, "hipMalloc of %zu bytes of working memory failed", want);
    }
    owned.push_back(q);
    p[s] = q;
    have[s] = want;
    return RT_OK;
}

void WorkBufs::release() {
    for (void* q : owned) (void)hipFree(q);
    owned.clear();
    params_key.clear();
    for (int s = 0; s < N_SLOTS; ++s) {
        p[s] = nullptr;
        have[s] = 0;
    }
}

// ----------------------------------------------------------------- kernel

using rt::kBlock;
using rt::kMaxPoolLds;
using rt::TraceArgs;

// BEAM < 0: rays are loaded; otherwise the beam is generated with direction type BEAM
constexpr int kLoad = -1;

// Generic kernel: the structure of every surface is read from its record.
// MODE: the recording modes (rt::kRecLoss | rt::kRecExt) or 0.
template <int BEAM, int MODE = 0>
__global__ __launch_bounds__(kBlock) void rt_trace_kernel(TraceArgs a) {
    rt::trace_body<BEAM, MODE>(a, [&](Ray& r, bool& alive, rt::TraceCtx& c, uint64_t i) {
        for (int s = 0; s < a.n_surf; ++s) {
            rt::surface_step<rt::DynSurf, MODE>(rt::DynSurf{c.table + (size_t)s * rt::DEV_STRIDE}, s, r, alive, c);
            if (a.dump) rt::dump_state(a, s, r, alive, i);
        }
    });
}

// Extents of a recording trace from its workgroups' keys (key k of workgroup w
// at keys[k * n_wg + w]; even k a minimum, odd k the minimum of the negated
// value, see rt::ext_add), as doubles, NaN where no ray was alive; workgroup
// blockIdx.x = key k.
__global__ __launch_bounds__(256) void rt_ext_reduce_kernel(const unsigned long long* keys, unsigned n_wg,
                                                            double* out) {
    __shared__ unsigned long long s[256];
    unsigned long long v = ~0ull;
    for (unsigned w = threadIdx.x; w < n_wg; w += 256) {
        const unsigned long long k = keys[(size_t)blockIdx.x * n_wg + w];
        v = k < v ? k : v;
    }
    s[threadIdx.x] = v;
    __syncthreads();
    for (int m = 128; m > 0; m >>= 1) {
        if ((int)threadIdx.x < m && s[threadIdx.x + m] < s[threadIdx.x]) s[threadIdx.x] = s[threadIdx.x + m];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double d = rt::key_value(s[0]);
        out[blockIdx.x] = s[0] == ~0ull ? __builtin_nan("") : (blockIdx.x & 1) ? -d : d;
    }
}

// Generic batched kernel (structure read from the records of each instance)
template <int BEAM>
__global__ __launch_bounds__(kBlock) void rt_trace_batch_kernel(TraceArgs a) {
    rt::trace_batch_body<BEAM>(a, [&](Ray& r, bool& alive, rt::TraceCtx& c, uint64_t) {
        for (int s = 0; s < a.n_surf; ++s)
            rt::surface_step(rt::DynSurf{c.table + (size_t)s * rt::DEV_STRIDE}, s, r, alive, c);
    });
}

// Per-instance spot from the tile moments, combined in tile order (Chan,
// Golub and LeVeque's pairwise update): n, centroid x, y, variance x, y and
// RMS radius sqrt(var x + var y).  One thread per instance.
// Spots per ray group (group of ray r = r mod G).  Moments (n, mean x,
// mean y, M2 x, M2 y) are merged with Chan et al.'s pairwise update.
struct Mom {
    double n, mx, my, qx, qy;
};

__device__ __forceinline__ Mom mom_merge(const Mom& a, const Mom& b) {
    if (b.n == 0.0) return a;
    if (a.n == 0.0) return b;
    const double nn = a.n + b.n, dx = b.mx - a.mx, dy = b.my - a.my, f = b.n / nn;
    return Mom{nn, a.mx + dx * f, a.my + dy * f, a.qx + b.qx + dx * dx * a.n * f, a.qy + b.qy + dy * dy * a.n * f};
}

// Per-instance spots of a batch from its tiles' moments (n, mean x, mean y,
// M2 x, M2 y): one workgroup per instance; lane t merges tiles t, t + 256,
// ... in ascending order, then the lanes' moments merge by a fixed tree, so
// the result depends on the tiles alone.  (One lane walking an instance's
// ~4,000 tiles serially took 2.2 ms for 1024 instances.)
constexpr int kInstSpotThreads = 256;

__global__ __launch_bounds__(kInstSpotThreads) void rt_batch_spots_kernel(const double* tm,
                                                                         const uint64_t* tile_start,
                                                                         uint64_t n_inst, double* spots) {
    __shared__ Mom s[kInstSpotThreads];
    const uint64_t i = blockIdx.x;
    Mom m{0.0, 0.0, 0.0, 0.0, 0.0};
    for (uint64_t t = tile_start[i] + threadIdx.x; t < tile_start[i + 1]; t += kInstSpotThreads) {
        const double* o = tm + t * 5;
        m = mom_merge(m, Mom{o[0], o[1], o[2], o[3], o[4]});
    }
    s[threadIdx.x] = m;
    __syncthreads();
    for (int k = kInstSpotThreads / 2; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) s[threadIdx.x] = mom_merge(s[threadIdx.x], s[threadIdx.x + k]);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const Mom r = s[0];
        double* out = spots + i * RT_SPOT_STRIDE;
        out[0] = r.n;
        out[1] = r.mx;
        out[2] = r.my;
        out[3] = r.n > 0.0 ? r.qx / r.n : 0.0;
        out[4] = r.n > 0.0 ? r.qy / r.n : 0.0;
        out[5] = r.n > 0.0 ? sqrt((r.qx + r.qy) / r.n) : 0.0;
    }
}

// Group spots of stored rays in two launches: moments of (chunk, group), then
// rt_spots_rows_kernel over each group's chunks.
//
// A workgroup of 256 lanes covers W = min(G, 256) consecutive groups and R =
// 256 / W strides of the groups side by side (lane t: stride t / W, group
// t % W), so its lanes read consecutive rays whatever G is; it walks its
// chunk of S strides kSpotRays rays a lane at a time, held in registers: sum
// and mean, then squared deviations (one division per kSpotRays rays), merged
// across the passes and, in LDS by a fixed tree, across the lanes of a group.
// One row per (chunk, group) leaves, group-major.  Bound by the row reads (17
// bytes a ray) and, for small inputs, by the two launches.  One thread per 8
// rays of a group (Welford, two divisions a ray, 40 bytes of partial per 8
// rays) and one workgroup merging all of a group's partials took 7.4 + 27.9
// us for 5e5 rays in 5 groups; this takes 6.0 + 4.4 (5e6 rays in one group:
// 19.4 + 5.1, 4.4 TB/s).
constexpr int kSpotThreads = 256;
constexpr int kSpotRays = 8;             // rays of one group per lane and pass

// strides of the groups per chunk: one pass of the workgroup, more passes
// above 2^21 rays so that a group's merge has about 1,000 rows at most (the
// rows of 1e7 rays in one group: 4,900 at one pass per chunk, 980 at five)
__host__ __device__ inline uint64_t spot_chunk_strides(uint64_t n, uint64_t G) {
    const uint64_t rows = G < (uint64_t)kSpotThreads ? kSpotThreads / G : 1;
    return rows * kSpotRays * (1 + (n >> 21));
}

// chunks of n rays in G groups (one, empty, for no rays)
__host__ __device__ inline uint64_t spot_chunk_count(uint64_t n, uint64_t G) {
    const uint64_t strides = (n + G - 1) / G, S = spot_chunk_strides(n, G);
    return strides > 0 ? (strides + S - 1) / S : 1;
}

// the moments of chunk b of n rays (X, Y, F: the first ray's) for groups g0 ..
// g0 + 255, to rows part[(g * n_rows + row) * 5 ..]
__device__ __forceinline__ void group_moments_chunk(const double* X, const double* Y, const signed char* F, uint64_t n,
                                                    uint64_t G, uint64_t b, uint64_t g0, double* part, uint64_t n_rows,
                                                    uint64_t row) {
    __shared__ Mom s[kSpotThreads];
    const unsigned W = G < (uint64_t)kSpotThreads ? (unsigned)G : (unsigned)kSpotThreads, R = kSpotThreads / W;
    const unsigned lane_row = threadIdx.x / W;
    const uint64_t g = g0 + (threadIdx.x - lane_row * W);
    const uint64_t S = spot_chunk_strides(n, G), s0 = b * S;
    const bool on = lane_row < R && g < G;
    Mom m{0.0, 0.0, 0.0, 0.0, 0.0};
    for (uint64_t p = 0; p < S; p += (uint64_t)R * kSpotRays) {
        double x[kSpotRays], y[kSpotRays];
        bool live[kSpotRays];
#pragma unroll
        for (int k = 0; k < kSpotRays; ++k) {
            const uint64_t r = (s0 + p + lane_row + (uint64_t)k * R) * G + g;
            live[k] = on && r < n && F[r] == 1;
            x[k] = live[k] ? X[r] : 0.0;
            y[k] = live[k] ? Y[r] : 0.0;
        }
        Mom q{0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < kSpotRays; ++k) {
            q.n += live[k] ? 1.0 : 0.0;
            q.mx += x[k];
            q.my += y[k];
        }
        if (q.n > 0.0) {
            q.mx /= q.n;
            q.my /= q.n;
#pragma unroll
            for (int k = 0; k < kSpotRays; ++k) {
                const double dx = live[k] ? x[k] - q.mx : 0.0, dy = live[k] ? y[k] - q.my : 0.0;
                q.qx += dx * dx;
                q.qy += dy * dy;
            }
        }
        m = mom_merge(m, q);
    }
    s[threadIdx.x] = m;
    __syncthreads();
    for (unsigned k = kSpotThreads / 2; k > 0; k >>= 1) {
        if (lane_row < k && lane_row + k < R) s[threadIdx.x] = mom_merge(s[threadIdx.x], s[threadIdx.x + k * W]);
        __syncthreads();
    }
    if (lane_row == 0 && on) {
        const Mom r = s[threadIdx.x];
        double* o = part + (g * n_rows + row) * 5;
        o[0] = r.n; o[1] = r.mx; o[2] = r.my; o[3] = r.qx; o[4] = r.qy;
    }
}

// blocks of 256 groups, a workgroup each per chunk
inline uint64_t spot_group_blocks(uint64_t G) { return (G + kSpotThreads - 1) / kSpotThreads; }

// workgroup blockIdx.x = chunk x (blocks of 256 groups)
__global__ __launch_bounds__(kSpotThreads) void rt_group_moments_kernel(const double* X, const double* Y,
                                                                        const signed char* F, uint64_t n, uint64_t G,
                                                                        uint64_t n_chunks, double* part) {
    const uint64_t gb = blockIdx.x / n_chunks, b = blockIdx.x - gb * n_chunks;
    group_moments_chunk(X, Y, F, n, G, b, gb * kSpotThreads, part, n_chunks, b);
}

// Spots from group-major partial rows (the traces' tile partials,
// TraceArgs::group_part): one workgroup per (instance, group) = blockIdx.x,
// the group's rows [row_start[i], row_start[i + 1]) of n_rows per group
// (row_start null: one instance, every row).  Thread t of NT merges rows t,
// t + NT, ... in order, loading four ahead (consecutive threads read
// consecutive rows), then a fixed tree over the threads.  NT: 1024 for one
// scheme (thousands of rows per group), 256 for a batch's instances.
template <int NT>
__global__ __launch_bounds__(NT) void rt_spots_rows_kernel(const double* part, uint64_t n_rows,
                                                           const uint64_t* row_start, uint64_t G, double* spots) {
    constexpr int kRowThreads = NT;
    __shared__ Mom s[kRowThreads];
    const uint64_t ig = blockIdx.x, i = ig / G, g = ig - i * G;
    const uint64_t r0 = row_start ? row_start[i] : 0, r1 = row_start ? row_start[i + 1] : n_rows;
    const double* base = part + g * n_rows * 5;
    Mom m{0.0, 0.0, 0.0, 0.0, 0.0};
    uint64_t b = r0 + threadIdx.x;
    for (; b + 3 * kRowThreads < r1; b += 4 * kRowThreads) {
        Mom q[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const double* o = base + (b + k * kRowThreads) * 5;
            q[k] = Mom{o[0], o[1], o[2], o[3], o[4]};
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) m = mom_merge(m, q[k]);
    }
    for (; b < r1; b += kRowThreads) {
        const double* o = base + b * 5;
        m = mom_merge(m, Mom{o[0], o[1], o[2], o[3], o[4]});
    }
    s[threadIdx.x] = m;
    __syncthreads();
    for (int k = kRowThreads / 2; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) s[threadIdx.x] = mom_merge(s[threadIdx.x], s[threadIdx.x + k]);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const Mom r = s[0];
        double* out = spots + ig * RT_SPOT_STRIDE;
        out[0] = r.n;
        out[1] = r.mx;
        out[2] = r.my;
        out[3] = r.n > 0.0 ? r.qx / r.n : 0.0;
        out[4] = r.n > 0.0 ? r.qy / r.n : 0.0;
        out[5] = r.n > 0.0 ? sqrt((r.qx + r.qy) / r.n) : 0.0;
    }
}

// Batched spots: instance i's rays are [ray_start[i], ray_start[i+1]) of the
// concatenated beam and ray r of the instance is in group r mod G.  Chunks as
// for that instance's rays alone, chunk_start the prefix over instances.
__global__ __launch_bounds__(1024) void rt_batch_chunks_kernel(const uint64_t* ray_start, uint64_t n_inst,
                                                               uint64_t G, uint64_t* chunk_start) {
    // one workgroup: chunk counts of 1024 instances at a time, an inclusive
    // scan in LDS (Hillis-Steele), the running total carried between passes
    __shared__ uint64_t sc[1024];
    uint64_t carry = 0;
    if (threadIdx.x == 0) chunk_start[0] = 0;
    for (uint64_t base = 0; base < n_inst; base += 1024) {
        const uint64_t i = base + threadIdx.x;
        sc[threadIdx.x] = i < n_inst ? spot_chunk_count(ray_start[i + 1] - ray_start[i], G) : 0;
        __syncthreads();
        for (int off = 1; off < 1024; off <<= 1) {
            const uint64_t add = (int)threadIdx.x >= off ? sc[threadIdx.x - off] : 0;
            __syncthreads();
            sc[threadIdx.x] += add;
            __syncthreads();
        }
        if (i < n_inst) chunk_start[i + 1] = carry + sc[threadIdx.x];
        carry += sc[1023];
        __syncthreads();
    }
}

// workgroup blockIdx.x = chunk of the batch x (blocks of 256 groups); the
// chunk's instance from the prefix
__global__ __launch_bounds__(kSpotThreads) void rt_batch_moments_kernel(const double* X, const double* Y,
                                                                        const signed char* F,
                                                                        const uint64_t* ray_start,
                                                                        const uint64_t* chunk_start, uint64_t n_inst,
                                                                        uint64_t G, uint64_t n_chunks, double* part) {
    const uint64_t gb = blockIdx.x / n_chunks, c = blockIdx.x - gb * n_chunks;
    uint64_t lo = 0, hi = n_inst;
    while (hi - lo > 1) {
        const uint64_t mid = (lo + hi) >> 1;
        if (chunk_start[mid] <= c) lo = mid; else hi = mid;
    }
    const uint64_t r0 = ray_start[lo];
    group_moments_chunk(X + r0, Y + r0, F + r0, ray_start[lo + 1] - r0, G, c - chunk_start[lo], gb * kSpotThreads, part,
                        n_chunks, c);
}

// One gradient-descent step on the device records of a batch: thread (i, s)
// applies p[field_k] -= lr[j_k] grad[i][j_k] for the parameters of surface s
// (map: per surface a start in a list of (j, field) pairs), then re-derives
// the record's host-derived constants (the formulas of rt_device_record) and
// the sin/cos of every updated angle.
__global__ void rt_batch_descend_kernel(double* tables, uint64_t n_inst, int n_surf, const int* map_start,
                                        const int* map, const double* grad, const double* lr, int n_par) {
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n_inst * (uint64_t)n_surf) return;
    const uint64_t i = idx / n_surf;
    const int s = (int)(idx - i * n_surf);
    const int k0 = map_start[s], k1 = map_start[s + 1];
    if (k0 == k1) return;
    double* p = tables + idx * rt::DEV_STRIDE;
    for (int k = k0; k < k1; ++k) {
        const int j = map[2 * k], f = map[2 * k + 1];
        p[f] -= lr[j] * grad[i * n_par + j];
        if (f >= RT_S_ANG && f < RT_S_ANG + 3) {
            p[RT_S_SIN + f - RT_S_ANG] = sin(p[f]);
            p[RT_S_COS + f - RT_S_ANG] = cos(p[f]);
        }
    }
    p[rt::D_INV_C] = p[RT_S_C] != 0.0 ? 1.0 / p[RT_S_C] : 0.0;
    p[rt::D_INV_D] = p[RT_S_GRCONST] != 0.0 ? 1.0 / p[RT_S_GRCONST] : 0.0;
    p[rt::D_K1C2] = (p[RT_S_K] + 1) * p[RT_S_C] * p[RT_S_C];
    for (int a = 1; a <= RT_MAX_POLY; ++a) p[rt::D_IA + a - 1] = (double)a * p[RT_S_A + a - 1];
}

// The spot loss of the adjoint and its seeds, one workgroup: per group with
// live rays, rms + w ((cx - tx)^2 + (cy - ty)^2); seeds (ax, ay, b) with
// dloss/dX_r = ax + b X_r for the group's rays: b = 1 / (n rms),
// ax = -b cx + 2 w (cx - tx) / n, likewise for y.  Thread t sums groups
// t, t + 256, ... in order, then a fixed tree: bit-reproducible.
// Loss and adjoint seeds of every group, one workgroup: each lane takes the
// groups lane, lane + kLossThreads, ... four at a time (their records loaded
// together, so a lane has four loads in flight), adds its groups' loss terms
// in that order, and the workgroup sums the lanes' terms by a fixed tree.
constexpr int kLossThreads = 1024;

__device__ __forceinline__ double spot_loss_group(const double* sp, const double* target, uint64_t g, double w,
                                                  double* seeds) {
    const double n = sp[0], cx = sp[1], cy = sp[2], rms = sp[5];
    const double tx = target ? target[2 * g] : 0.0, ty = target ? target[2 * g + 1] : 0.0;
    double ax = 0.0, ay = 0.0, b = 0.0, term = 0.0;
    if (n > 0.0) {
        term = rms + w * ((cx - tx) * (cx - tx) + (cy - ty) * (cy - ty));
        b = rms > 0.0 ? 1.0 / (n * rms) : 0.0;
        ax = -b * cx + 2.0 * w * (cx - tx) / n;
        ay = -b * cy + 2.0 * w * (cy - ty) / n;
    }
    seeds[3 * g] = ax;
    seeds[3 * g + 1] = ay;
    seeds[3 * g + 2] = b;
    return term;
}

__global__ __launch_bounds__(kLossThreads) void rt_spot_loss_kernel(const double* spots, uint64_t G,
                                                                    const double* target, double w, double* seeds,
                                                                    double* loss) {
    __shared__ double s[kLossThreads];
    constexpr uint64_t T = kLossThreads;
    double acc = 0.0;
    uint64_t g = threadIdx.x;
    for (; g + 3 * T < G; g += 4 * T) {
        double rec[4][6];
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int q = 0; q < 6; ++q) rec[k][q] = spots[(g + k * T) * RT_SPOT_STRIDE + q];
#pragma unroll
        for (int k = 0; k < 4; ++k) acc += spot_loss_group(rec[k], target, g + k * T, w, seeds);
    }
    for (; g < G; g += T) acc += spot_loss_group(spots + g * RT_SPOT_STRIDE, target, g, w, seeds);
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int k = kLossThreads / 2; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) s[threadIdx.x] += s[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss = s[0];
}

// ------------------------------------------------------------------- C ABI

// Per-wavelength table of a scheme's spline-valued functions (refractive
// indices, detector QE and spectrum), used by the generated traces of
// grid-wavelength beams: column q (layout of rt_jit_ltab_layout) at grid
// index j is the spline at pool offset off[q] evaluated at the beam's j-th
// wavelength.  Filled on the trace's stream before each such trace, so traces
// of one scheme with different wavelength grids must be stream-ordered.
struct Ltab {
    std::vector<int> base, surf, role;
    double* off_dev = nullptr;       // pool offset of each column
    double* tab_dev = nullptr;       // n_cols x kLtabMax
    bool ok = false;                 // layout set up (a column exists, offsets equal in every instance)
    void release() {
        (void)hipFree(off_dev);
        (void)hipFree(tab_dev);
        off_dev = tab_dev = nullptr;
        ok = false;
    }
};
constexpr uint64_t kLtabMax = 16384;   // wavelengths of the largest grid served by the table

// The derived per-wavelength table of a scheme's generated traces
// (rt_jit_dtab_layout): n_cols x kLtabMax doubles, filled on the launch
// stream before a trace whose wavelength grid or stream differs from those of
// the last fill (a trace on another stream is not ordered after that fill).
// Once a launch is captured into a graph, every launch fills it (a replay may
// run at any later time, with the grid it was captured with).  Traces of one
// scheme with different wavelength grids on two streams at once race on it.
struct Dtab {
    int n_cols = 0;
    double* tab_dev = nullptr;
    bool valid = false;              // tab_dev holds the grid of key
    bool always = false;             // a launch was captured: fill every time
    double key[5] = {0, 0, 0, 0, 0};
    hipStream_t stream = nullptr;    // stream of the last fill
};

constexpr int kDefaultWaves = 7, kDefaultGridMult = 16;

struct rt_hip_scheme {
    int device;
    std::string signature;           // structural key of the generated kernels
    int n_surf;
    size_t pool_len;                 // device pool (doubles)
    double* table_dev;               // n_surf records of rt::DEV_STRIDE
    mutable Dtab dt;                 // derived per-wavelength table of the generated traces
    double* pool_dev;
    std::vector<double> table;       // public packed table, as given
    std::vector<double> pool;        // public spline pool, as given
    std::vector<double> dtable;      // device records
    std::vector<double> dpool;       // device spline records
    // launch of the generated kernel (rt_hip_scheme_set_launch, rt_hip_autotune)
    // (default 256 lanes, 7 waves/SIMD, 16 workgroups per resident slot: the
    // fastest of a sweep of the batched trace over 1024 instances of uneven
    // size, 21.3 ms against 23.7-24.0 ms at a grid multiple of 2; launch_shape
    // says which traces of one scheme take another)
    int block = rt::kBlock;          // lanes per workgroup
    int waves = kDefaultWaves;       // minimum waves per SIMD asked of the compiler (0: its choice)
    int grid_mult = kDefaultGridMult;    // persistent workgroups per CU = grid_mult x resident ones
    // who set them: nobody (launch_shape's rules hold), the autotuner (taken for
    // the traces it timed) or the caller (taken for every trace)
    enum { BY_RULE, BY_TUNER, BY_CALLER } launch_by = BY_RULE;
    bool tuned_frames = false;       // the autotuner's traces formed both frames
    // surface unroll depth: 1, the whole chain unrolled (the generated
    // kernel); 0, a runtime loop over the records (the generic kernel)
    int unroll = 1;
    void* arena = nullptr;           // the allocation of table_dev, pool_dev, stat_copies and dt.tab_dev
    // kStatCopies x RT_STATS_LEN counters the trace kernels add to, folded into
    // the caller's statistics after each trace (and cleared by the fold)
    unsigned long long* stat_copies = nullptr;
    // working memory of the scheme's adjoints and spot reductions
    mutable WorkBufs work;
};

namespace {
struct DeviceInfo {
    bool valid = false;
    int device = 0;
    int cus = 0;
    hipDeviceProp_t prop;
};
thread_local DeviceInfo g_dev;

}  // namespace

int rt_ensure_device() {
    if (g_dev.valid) return RT_OK;
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev), RT_ERR_INIT_FAILED);
    HIP_TRY(hipGetDeviceProperties(&g_dev.prop, dev), RT_ERR_INIT_FAILED);
    g_dev.device = dev;
    g_dev.cus = g_dev.prop.multiProcessorCount;
    g_dev.valid = true;
    return RT_OK;
}

int rt_device_cus() { return g_dev.cus > 0 ? g_dev.cus : 256; }

namespace {
int ensure_device() { return rt_ensure_device(); }

bool fn_ref_ok(double kind, double val, size_t pool_len, const double* pool) {
    if (kind == (double)RT_FN_CONST) return true;
    if (kind != (double)RT_FN_SPLINE) return false;
    if (!(val >= 0) || val != (double)(size_t)val) return false;
    size_t o = (size_t)val;
    if (o >= pool_len) return false;
    double k = pool[o];
    if (!(k >= 2) || k > RT_MAX_SPLINE_KNOTS || k != (double)(size_t)k) return false;
    return o + 1 + 3 * (size_t)k <= pool_len;
}
}  // namespace

extern "C" int rt_hip_init(int device) {
    int count = 0;
    HIP_TRY(hipGetDeviceCount(&count), RT_ERR_INIT_FAILED);
    if (device < 0 || device >= count)
        return set_error(RT_ERR_INIT_FAILED, "device %d out of range (%d devices)", device, count);
    HIP_TRY(hipSetDevice(device), RT_ERR_INIT_FAILED);
    g_dev.valid = false;
    int rc = ensure_device();
    // the device address of the no-allocation entry point's scratch array
    return rc == RT_OK ? rt_scratch_setup(device) : rc;
}

extern "C" int rt_hip_info(char* buf, size_t len) {
    int rc = ensure_device();
    if (rc != RT_OK) return rc;
    const hipDeviceProp_t& p = g_dev.prop;
    int n = snprintf(buf, len,
                     "AMD HIP engine (gfx950 FP64)\nDevice name: %s\nArchitecture: %s\n"
                     "Global memory: %zu\nNumber of compute units: %d\nClock (kHz): %d\n",
                     p.name, p.gcnArchName, (size_t)p.totalGlobalMem, p.multiProcessorCount, p.clockRate);
    if (n < 0 || (size_t)n >= len) return set_error(RT_ERR_BAD_ALLOC, "info buffer too small");
    return RT_OK;
}

extern "C" int rt_hip_last_kernel(char* buf, size_t len) {
    if (!buf || !len) return RT_ERR_BAD_VALUE;
    snprintf(buf, len, "%s", g_last_kernel);
    return RT_OK;
}

extern "C" int rt_hip_last_error(char* buf, size_t len) {
    if (!buf || !len) return RT_ERR_BAD_VALUE;
    snprintf(buf, len, "%s", g_last_error.c_str());
    return RT_OK;
}

extern "C" int rt_hip_validate_scheme(const double* t, int n_surf, const double* pool, size_t pool_len) {
    if (!t || n_surf < 1 || n_surf > RT_MAX_SURF)
        return set_error(RT_ERR_BAD_VALUE, "n_surf %d out of range [1,%d]", n_surf, RT_MAX_SURF);
    if (pool_len && !pool) return set_error(RT_ERR_BAD_VALUE, "pool is NULL");
    for (int s = 0; s < n_surf; ++s) {
        const double* p = t + (size_t)s * RT_SURF_STRIDE;
        int cls = (int)p[RT_S_CLASS], type = (int)p[RT_S_TYPE], shape = (int)p[RT_S_SHAPE];
        if (cls < RT_PLANE || cls > RT_AUXCLASS || (double)cls != p[RT_S_CLASS])
            return set_error(RT_ERR_BAD_VALUE, "surface %d: bad class", s);
        if (type < RT_MIRROR || type > RT_AUXTYPE || (double)type != p[RT_S_TYPE])
            return set_error(RT_ERR_BAD_VALUE, "surface %d: bad type", s);
        if (shape != RT_CIRCLE && shape != RT_RECTANGLE)
            return set_error(RT_ERR_BAD_VALUE, "surface %d: bad shape", s);
        double np = p[RT_S_NPOLY];
        if (!(np >= 0 && np <= RT_MAX_POLY) || np != (double)(int)np)
            return set_error(RT_ERR_BAD_VALUE, "surface %d: bad number of aspheric terms", s);
        if (type == RT_GRATING) {
            int gt = (int)p[RT_S_GRTYPE];
            if (gt != RT_REFLECTIVE && gt != RT_TRANSPARENT)   // surface.cu:1637 BAD_VALUE
                return set_error(RT_ERR_BAD_VALUE, "surface %d: bad grating type", s);
            if (!(p[RT_S_GRCONST] != 0.0))
                return set_error(RT_ERR_BAD_VALUE, "surface %d: zero grating constant", s);
            int om = (int)p[RT_S_ORDMODE];
            if (om != RT_ORDER_FIXED && om != RT_ORDER_BLAZE)
                return set_error(RT_ERR_BAD_VALUE, "surface %d: bad order mode", s);
        }
        if (type == RT_LENS || type == RT_GRATING) {
            if (!fn_ref_ok(p[RT_S_N1KIND], p[RT_S_N1VAL], pool_len, pool) ||
                !fn_ref_ok(p[RT_S_N2KIND], p[RT_S_N2VAL], pool_len, pool))
                return set_error(RT_ERR_BAD_VALUE, "surface %d: bad refractive index reference", s);
        }
        if (type == RT_DETECTOR && p[RT_S_CCD_XDIM] > 0.0) {
            double xd = p[RT_S_CCD_XDIM], yd = p[RT_S_CCD_YDIM];
            if (!(xd >= 1 && yd >= 1 && xd * yd <= 4294967296.0) || xd != (double)(uint64_t)xd ||
                yd != (double)(uint64_t)yd)
                return set_error(RT_ERR_BAD_VALUE, "surface %d: bad CCD dimensions", s);
            if (!(p[RT_S_CCD_XPIX] > 0.0) || !(p[RT_S_CCD_YPIX] > 0.0))
                return set_error(RT_ERR_BAD_VALUE, "surface %d: bad CCD pixel size", s);
            if (!fn_ref_ok(p[RT_S_QEKIND], p[RT_S_QEVAL], pool_len, pool) ||
                !fn_ref_ok(p[RT_S_SPKIND], p[RT_S_SPVAL], pool_len, pool))
                return set_error(RT_ERR_BAD_VALUE, "surface %d: bad QE/spectrum reference", s);
        }
    }
    if (pool_len > (size_t)kMaxPoolLds - 64)
        return set_error(RT_ERR_BAD_VALUE, "spline pool of %zu doubles exceeds %d", pool_len, kMaxPoolLds - 64);
    return RT_OK;
}

void rt_device_record(const double* p, double* d) {
    for (int k = 0; k < rt::DEV_STRIDE; ++k) d[k] = k < RT_SURF_STRIDE ? p[k] : 0.0;
    d[rt::D_INV_C] = p[RT_S_C] != 0.0 ? 1.0 / p[RT_S_C] : 0.0;
    d[rt::D_INV_D] = p[RT_S_GRCONST] != 0.0 ? 1.0 / p[RT_S_GRCONST] : 0.0;
    d[rt::D_HALF_X] = p[RT_S_CCD_XSIZE] / 2.0;
    d[rt::D_HALF_Y] = p[RT_S_CCD_YSIZE] / 2.0;
    d[rt::D_INV_XPIX] = p[RT_S_CCD_XPIX] != 0.0 ? 1.0 / p[RT_S_CCD_XPIX] : 0.0;
    d[rt::D_INV_YPIX] = p[RT_S_CCD_YPIX] != 0.0 ? 1.0 / p[RT_S_CCD_YPIX] : 0.0;
    // mask bounds as the reference forms them per ray (surface.cpp:264-321, 652-699)
    const double s0 = p[RT_S_SIZE0], s1 = p[RT_S_SIZE1], c0 = p[RT_S_CEN0], c1 = p[RT_S_CEN1];
    double* m = d + rt::D_MASK;
    if ((int)p[RT_S_SHAPE] == RT_CIRCLE) {
        m[0] = s0 * s0;
    } else if ((int)p[RT_S_TYPE] == RT_SHADE) {
        m[0] = -s0 / 2.0; m[1] = s0 / 2.0; m[2] = -s1 / 2.0; m[3] = s1 / 2.0;
    } else {
        m[0] = c0 - s0 / 2.0; m[1] = c0 + s0 / 2.0; m[2] = c1 - s1 / 2.0; m[3] = c1 + s1 / 2.0;
    }
    d[rt::D_K1C2] = (p[RT_S_K] + 1) * p[RT_S_C] * p[RT_S_C];
    for (int i = 1; i <= RT_MAX_POLY; ++i) d[rt::D_IA + i - 1] = (double)i * p[RT_S_A + i - 1];
}

// Device tables: each record gets its host-derived constants (rt::DevField)
// and each referenced spline is re-laid out as [K, x0, (K-1)/(x[K-1]-x0),
// x, y, y2] with the references patched to the new offsets.
static void build_device_tables(rt_hip_scheme* s) {
    const int n = s->n_surf;
    s->dtable.assign((size_t)n * rt::DEV_STRIDE, 0.0);
    s->dpool.clear();
    std::vector<std::pair<size_t, size_t>> moved;   // (public offset, device offset)
    auto remap = [&](double& kind, double& val) {
        if (kind != (double)RT_FN_SPLINE) return;
        size_t o = (size_t)val;
        for (auto& m : moved)
            if (m.first == o) { val = (double)m.second; return; }
        const double* sp = s->pool.data() + o;
        size_t K = (size_t)sp[0];
        size_t d = s->dpool.size();
        s->dpool.push_back((double)K);
        s->dpool.push_back(sp[1]);
        s->dpool.push_back((double)(K - 1) / (sp[K] - sp[1]));
        s->dpool.insert(s->dpool.end(), sp + 1, sp + 1 + 3 * K);
        moved.push_back({o, d});
        val = (double)d;
    };
    for (int i = 0; i < n; ++i) {
        double* d = s->dtable.data() + (size_t)i * rt::DEV_STRIDE;
        const double* p = s->table.data() + (size_t)i * RT_SURF_STRIDE;
        rt_device_record(p, d);
        int type = (int)p[RT_S_TYPE];
        if (type == RT_LENS || type == RT_GRATING) {
            remap(d[RT_S_N1KIND], d[RT_S_N1VAL]);
            remap(d[RT_S_N2KIND], d[RT_S_N2VAL]);
        }
        if (type == RT_DETECTOR && p[RT_S_CCD_XDIM] > 0.0) {
            remap(d[RT_S_QEKIND], d[RT_S_QEVAL]);
            remap(d[RT_S_SPKIND], d[RT_S_SPVAL]);
        }
    }
    s->pool_len = s->dpool.size();
    s->signature = rt_jit_signature(s->dtable.data(), n);
}

__global__ __launch_bounds__(256) void rt_ltab_kernel(rt::LtabArgs a) { rt::ltab_body(a); }

__global__ __launch_bounds__(256) void rt_dtab_kernel(rt::DtabArgs a) { rt::dtab_body(a); }

__global__ __launch_bounds__(rt::kFoldThreads) void rt_stats_fold_kernel(unsigned long long* copies,
                                                                         unsigned long long* stats,
                                                                         const double* table, int n_surf, int ccd) {
    rt::stats_fold_body(copies, stats, table, n_surf, ccd != 0);
}

namespace {

// The table's layout from the signature and its column offsets from the
// device records of n_inst instances (the table is used only when every
// instance names the same spline in every column); buffers on first use.
int ltab_setup(Ltab& t, const std::string& sig, const double* dtables, int n_inst, int n_surf) {
    static const int kRoleField[4] = {RT_S_N1VAL, RT_S_N2VAL, RT_S_QEVAL, RT_S_SPVAL};
    rt_jit_ltab_layout(sig, t.base, t.surf, t.role);
    t.ok = false;
    const size_t nc = t.surf.size();
    if (nc == 0) return RT_OK;
    const size_t inst = (size_t)n_surf * rt::DEV_STRIDE;
    std::vector<double> off(nc);
    for (size_t q = 0; q < nc; ++q) {
        const size_t f = (size_t)t.surf[q] * rt::DEV_STRIDE + (size_t)kRoleField[t.role[q]];
        off[q] = dtables[f];
        for (int i = 1; i < n_inst; ++i)
            if (dtables[(size_t)i * inst + f] != off[q]) return RT_OK;
    }
    if (!t.off_dev) HIP_TRY(hipMalloc(&t.off_dev, nc * sizeof(double)), RT_ERR_BAD_ALLOC);
    if (!t.tab_dev) HIP_TRY(hipMalloc(&t.tab_dev, nc * kLtabMax * sizeof(double)), RT_ERR_BAD_ALLOC);
    HIP_TRY(hipMemcpy(t.off_dev, off.data(), nc * sizeof(double), hipMemcpyHostToDevice), RT_ERR_FAILED);
    t.ok = true;
    return RT_OK;
}

// the zeroed counter copies of a scheme or batch
int stat_copies_alloc(unsigned long long** p) {
    const size_t bytes = (size_t)rt::kStatCopies * RT_STATS_LEN * sizeof(unsigned long long);
    HIP_TRY(hipMalloc(p, bytes), RT_ERR_BAD_ALLOC);
    HIP_TRY(hipMemset(*p, 0, bytes), RT_ERR_FAILED);
    return RT_OK;
}

// where a trace of `grid` workgroups adds its counters: the caller's, or the copies
void stats_target(TraceArgs& a, unsigned long long* copies, unsigned long long* stats, unsigned grid) {
    a.direct = stats && grid <= (unsigned)rt::kStatCopies ? 1 : 0;
    a.stats = !stats ? nullptr : a.direct ? stats : copies;
}

// stats += the copies (cleared), on `st` after the trace `a`, unless it added
// to them itself
int stats_fold(const TraceArgs& a, unsigned long long* stats, hipStream_t st) {
    if (!stats || a.direct) return RT_OK;
    const int ccd = ((a.flags & RT_TRACE_HIST) && a.hist) || ((a.flags & RT_TRACE_FLUX) && a.flux);
    hipLaunchKernelGGL(rt_stats_fold_kernel, dim3(1), dim3(rt::kFoldThreads), 0, st, a.stats, stats, a.table, a.n_surf,
                       ccd);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    return RT_OK;
}

// wavelengths of the beam's grid when per-wavelength tables serve it (one
// wavelength, or a composite uniform grid of at most kLtabMax), else 0
uint64_t grid_nk(const double* beam) {
    if (!rt_jit_ltab_enabled() || !rt_jit_enabled()) return 0;
    const int distr = (int)beam[RT_B_RANGE_DISTR];
    if (distr == RT_RANGE_MONO) return 1;
    if (distr != RT_RANGE_UNIFORM || beam[RT_B_COMPOSITE] == 0.0) return 0;
    const double nl = beam[RT_B_NLAMBDA];
    if (!(nl >= 1.0) || nl > (double)kLtabMax) return 0;
    return (uint64_t)nl;
}

uint64_t ltab_nk(const Ltab& t, const double* beam) { return t.ok ? grid_nk(beam) : 0; }

// the derived table's columns for the signature
void dtab_layout(Dtab& t, const std::string& sig) {
    std::vector<int> base, surf, role;
    rt_jit_dtab_layout(sig, base, surf, role);
    t.n_cols = (int)surf.size();
}

uint64_t dtab_nk(const Dtab& t, const double* beam) { return t.n_cols > 0 ? grid_nk(beam) : 0; }

// the derived table for nk grid wavelengths of a's beam, filled on `st`
// unless it holds that grid already
int dtab_fill(Dtab& t, const TraceArgs& a, const double* table_dev, const double* pool_dev, int n_surf,
              uint64_t nk, hipStream_t st) {
    const double key[5] = {a.beam.v[RT_B_RANGE_DISTR], a.beam.v[RT_B_RANGE + 0], a.beam.v[RT_B_RANGE + 1],
                           a.beam.v[RT_B_NLAMBDA], (double)nk};
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    HIP_TRY(hipStreamIsCapturing(st, &cs), RT_ERR_FAILED);
    if (cs != hipStreamCaptureStatusNone) t.always = true;
    if (!t.always && t.valid && st == t.stream && memcmp(key, t.key, sizeof key) == 0) return RT_OK;
    t.valid = false;
    rt::DtabArgs da;
    memset(&da, 0, sizeof da);
    da.beam = a.beam;
    da.table = table_dev;
    da.pool = pool_dev;
    da.out = t.tab_dev;
    da.nk = nk;
    da.n_surf = n_surf;
    hipLaunchKernelGGL(rt_dtab_kernel, dim3((unsigned)((nk + 255) / 256), (unsigned)n_surf), dim3(256), 0, st, da);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    if (!t.always) {
        memcpy(t.key, key, sizeof key);
        t.stream = st;
        t.valid = true;
    }
    return RT_OK;
}

// fill the table for nk grid wavelengths of a's beam on `st`
int ltab_fill(const Ltab& t, const TraceArgs& a, const double* pool_dev, uint64_t nk, hipStream_t st) {
    rt::LtabArgs la;
    memset(&la, 0, sizeof la);
    la.beam = a.beam;
    la.pool = pool_dev;
    la.col_off = t.off_dev;
    la.out = t.tab_dev;
    la.nk = nk;
    la.n_cols = (int)t.surf.size();
    const uint64_t total = (uint64_t)la.n_cols * nk;
    hipLaunchKernelGGL(rt_ltab_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, la);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    return RT_OK;
}

}  // namespace

extern "C" int rt_hip_scheme_create(const double* surf_table, int n_surf, const double* spline_pool,
                                    size_t pool_len, rt_hip_scheme** out) {
    if (!out) return set_error(RT_ERR_BAD_VALUE, "out is NULL");
    *out = nullptr;
    int rc = rt_hip_validate_scheme(surf_table, n_surf, spline_pool, pool_len);
    if (rc != RT_OK) return rc;
    rc = ensure_device();
    if (rc != RT_OK) return rc;
    rt_hip_scheme* s = new (std::nothrow) rt_hip_scheme();
    if (!s) return set_error(RT_ERR_BAD_ALLOC, "out of host memory");
    s->device = g_dev.device;
    s->n_surf = n_surf;
    s->table.assign(surf_table, surf_table + (size_t)n_surf * RT_SURF_STRIDE);
    if (pool_len) s->pool.assign(spline_pool, spline_pool + pool_len);
    build_device_tables(s);
    // one allocation and one upload for all: a scheme made and destroyed, as each
    // evaluation of a loss does, 68 -> 41 us
    dtab_layout(s->dt, s->signature);
    const size_t stats = (size_t)rt::kStatCopies * RT_STATS_LEN * sizeof(unsigned long long);
    const size_t tb = (s->dtable.size() * sizeof(double) + 255) / 256 * 256;
    const size_t pb = ((s->dpool.empty() ? 1 : s->dpool.size()) * sizeof(double) + 255) / 256 * 256;
    const size_t dt = (size_t)s->dt.n_cols * kLtabMax * sizeof(double);
    char* dev = nullptr;
    if (hipMalloc(&dev, tb + pb + stats + dt) != hipSuccess) {
        delete s;
        return set_error(RT_ERR_BAD_ALLOC, "hipMalloc of scheme tables failed");
    }
    s->arena = dev;
    s->table_dev = (double*)dev;
    s->pool_dev = (double*)(dev + tb);
    s->stat_copies = (unsigned long long*)(dev + tb + pb);
    s->dt.tab_dev = dt ? (double*)(dev + tb + pb + stats) : nullptr;
    std::vector<double> up((tb + pb) / sizeof(double), 0.0);
    std::copy(s->dtable.begin(), s->dtable.end(), up.begin());
    std::copy(s->dpool.begin(), s->dpool.end(), up.begin() + tb / sizeof(double));
    if (hipMemset(s->stat_copies, 0, stats) != hipSuccess ||
        hipMemcpy(dev, up.data(), tb + pb, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(dev);
        delete s;
        return set_error(RT_ERR_FAILED, "upload of scheme tables failed");
    }
    *out = s;
    return RT_OK;
}

extern "C" int rt_jit_check_dtable(const double* dtable, int n_surf, int beam_mode, char* text, size_t len,
                                   size_t* code_size);

extern "C" int rt_hip_jit_check(const double* surf_table, int n_surf, const double* spline_pool,
                                size_t pool_len, int beam_mode, char* text, size_t len, size_t* code_size) {
    int rc = rt_hip_validate_scheme(surf_table, n_surf, spline_pool, pool_len);
    if (rc != RT_OK) return rc;
    rt_hip_scheme tmp;
    tmp.n_surf = n_surf;
    tmp.table.assign(surf_table, surf_table + (size_t)n_surf * RT_SURF_STRIDE);
    if (pool_len) tmp.pool.assign(spline_pool, spline_pool + pool_len);
    build_device_tables(&tmp);
    rc = rt_jit_check_dtable(tmp.dtable.data(), n_surf, beam_mode, text, len, code_size);
    return rc == RT_OK ? RT_OK : set_error(rc, "generated kernel did not compile");
}

extern "C" int rt_hip_scheme_destroy(rt_hip_scheme* s) {
    if (!s) return RT_OK;
    s->work.release();
    (void)hipFree(s->arena);
    delete s;
    return RT_OK;
}

static int validate_beam(const double* b) {
    if (!b) return set_error(RT_ERR_BAD_VALUE, "beam description is NULL");
    int type = (int)b[RT_B_TYPE], shape = (int)b[RT_B_SHAPE], distr = (int)b[RT_B_RANGE_DISTR];
    if (type < RT_BEAM_PARALLEL || type > RT_BEAM_GAUSS) return set_error(RT_ERR_BAD_VALUE, "bad beam type");
    if (shape != RT_CIRCLE && shape != RT_RECTANGLE) return set_error(RT_ERR_BAD_VALUE, "bad beam shape");
    if (distr < RT_RANGE_RANDOM || distr > RT_RANGE_MONO) return set_error(RT_ERR_BAD_VALUE, "bad range distribution");
    // Beam::SetParams checks (beam.cpp:78-91)
    if (!(b[RT_B_NPER] > 0)) return set_error(RT_ERR_BAD_VALUE, "number of rays must be > 0");
    if (b[RT_B_P1] < 0 || !(b[RT_B_P2] > 0)) return set_error(RT_ERR_BAD_VALUE, "beam sizes must be > 0");
    if (shape == RT_CIRCLE && b[RT_B_P1] >= b[RT_B_P2])
        return set_error(RT_ERR_BAD_VALUE, "inner radius must be below the outer one");
    if (shape == RT_RECTANGLE && !(b[RT_B_P3] > 0)) return set_error(RT_ERR_BAD_VALUE, "size ratio must be > 0");
    if (b[RT_B_COMPOSITE] != 0.0 && !(b[RT_B_NLAMBDA] >= 1))
        return set_error(RT_ERR_BAD_VALUE, "composite beam needs nlambda >= 1");
    return RT_OK;
}

// uniform values of the direction generators, on the host (beam.cu:592-598, 1034, 1099);
// params[3]*deg2rad as the macro expands (beam.cpp:383): (params[3]*RT_PI)/180.0
static void beam_uniforms(TraceArgs& a) {
    double ang = a.beam.v[RT_B_ANGUNIT] != 0.0 ? a.beam.v[RT_B_ANGPAR] : a.beam.v[RT_B_ANGPAR] * rt::kPi / 180.0;
    a.beam.u.cone_cos = cos(ang / 2.0);
    a.beam.u.cone_sin = sin(ang / 2.0);
    double stddev = a.beam.v[RT_B_ANGPAR] / 2.35482 * rt::kPi / 180 / 3600;
    a.beam.u.gauss_tg = tan(stddev);
    a.beam.u.lam_step = rt::beam_lam_step(a.beam.v);
}

namespace {
// recording traces with extents: rays from which their launch is the large one,
// and the workgroups of the default launch that the rays below it take at most
constexpr uint64_t kExtRays = 1u << 18, kExtTiles = kExtRays / kBlock;
// generated rays into both frames from which a workgroup has 512 lanes
constexpr uint64_t kFrameRays = 1u << 20;

struct LaunchShape {
    int block, waves, mult;
};

// The launch of a trace (frames: into both frames).  The caller's holds for
// every trace, the autotuner's for traces like those it timed: generated,
// recording nothing, and with both frames or without as those were.  The
// others take the defaults, but 8 waves per SIMD for rays given by the caller
// (1e6 echelle rays into both frames 123 -> 120 us, 1e7 946 -> 935; with one
// frame or none, with fewer rays and on the Czerny-Turner within 2% either
// way); where both frames take an atomic of every ray and bound the trace,
// workgroups of 512 lanes from 2^20 rays on (1e7 echelle rays of 2048
// wavelengths 1014 -> 929 us, 4e6 410 -> 400; of 64 wavelengths within 2%,
// the Czerny-Turner within 1%); and 1024 lanes and 8 waves per SIMD for
// recording traces with extents from kExtRays on, where every workgroup has
// to meet the extremes before its rays lie inside them (2^18 echelle rays 51
// -> 46 us, 2^20 161 -> 123, 2^23 857 -> 763, 2^20 of the Czerny-Turner 51 ->
// 42; 2^17 echelle rays 37 -> 45, so not there; with 4 waves, where the
// echelle's kernel does not spill its 52 bytes a lane, 2^20 130, 2^23 855).
LaunchShape launch_shape(const rt_hip_scheme* sch, bool gen, bool frames, int rec, uint64_t n) {
    if (sch->launch_by == rt_hip_scheme::BY_CALLER ||
        (sch->launch_by == rt_hip_scheme::BY_TUNER && gen && !rec && frames == sch->tuned_frames))
        return LaunchShape{sch->block, sch->waves, sch->grid_mult};
    LaunchShape l{kBlock, kDefaultWaves, kDefaultGridMult};
    if (rec & rt::kRecExt) {
        if (n >= kExtRays) {
            l.block = 1024;
            l.waves = 8;
        }
    } else if (!rec && !gen) {
        l.waves = 8;
    } else if (!rec && frames && n >= kFrameRays) {
        l.block = 512;
    }
    return l;
}

// The workgroups of a recording trace with extents: as many as are resident
// at once and no more, so that each walks many rays under bounds it has met
// (ext_add) and leaves one row of keys, in whole rounds of rays.
unsigned ext_grid(uint64_t tiles, uint64_t resident) {
    const uint64_t rounds = (tiles + resident - 1) / resident;
    return (unsigned)((tiles + rounds - 1) / rounds);
}

template <int MODE>
auto generic_kernel(int beam_mode) {
    return beam_mode == RT_BEAM_PARALLEL ? rt_trace_kernel<RT_BEAM_PARALLEL, MODE>
           : beam_mode == RT_BEAM_CONIC  ? rt_trace_kernel<RT_BEAM_CONIC, MODE>
           : beam_mode == RT_BEAM_GAUSS  ? rt_trace_kernel<RT_BEAM_GAUSS, MODE>
                                         : rt_trace_kernel<kLoad, MODE>;
}

// rt_hip_trace and rt_hip_trace_record: rec is the recording mode (rt::kRecLoss
// | rt::kRecExt or 0), loss / extents its outputs
int trace_launch(const rt_hip_scheme* sch, const double* beam_desc, uint64_t seed, size_t ray_begin, size_t n_rays,
                 double* X, double* Y, double* Z, double* cX, double* cY, double* cZ, double* lambda,
                 signed char* flag, int flags, unsigned int* ccd_hist, double* ccd_flux, unsigned long long* stats,
                 double* dump, signed char* dump_flag, int rec, unsigned char* loss, double* extents,
                 void* stream, double* group_part = nullptr, uint64_t n_groups = 0, int* block_used = nullptr) {
    if (!sch) return set_error(RT_ERR_BAD_VALUE, "scheme is NULL");
    const bool gen = (flags & RT_TRACE_GENERATE) != 0;
    if (gen) {
        int rc = validate_beam(beam_desc);
        if (rc != RT_OK) return rc;
    } else if (!X || !Y || !Z || !cX || !cY || !cZ || !lambda || !flag) {
        return set_error(RT_ERR_BAD_VALUE, "input rays missing");
    }
    if ((flags & RT_TRACE_STORE) && (!X || !Y || !Z || !cX || !cY || !cZ || !lambda || !flag))
        return set_error(RT_ERR_BAD_VALUE, "RT_TRACE_STORE needs all ray buffers");
    if (X && (!Y || !Z || !cX || !cY || !cZ || !lambda))
        return set_error(RT_ERR_BAD_VALUE, "ray buffers must be given together");
    if ((dump == nullptr) != (dump_flag == nullptr))
        return set_error(RT_ERR_BAD_VALUE, "dump and dump_flag must be given together");
    if (n_rays == 0) return RT_OK;
    int rc = ensure_device();
    if (rc != RT_OK) return rc;

    TraceArgs a;
    memset(&a, 0, sizeof a);
    if (beam_desc) memcpy(a.beam.v, beam_desc, sizeof a.beam.v);
    if (gen) beam_uniforms(a);
    a.table = sch->table_dev;
    a.pool = sch->pool_dev;
    a.n_surf = sch->n_surf;
    a.pool_len = (int)sch->pool_len;
    a.flags = flags;
    a.seed = seed;
    a.ray_begin = ray_begin;
    a.n = n_rays;
    a.X = X; a.Y = Y; a.Z = Z; a.cX = cX; a.cY = cY; a.cZ = cZ; a.L = lambda; a.F = flag;
    a.hist = ccd_hist; a.flux = ccd_flux; a.dump = dump; a.dump_flag = dump_flag;
    a.loss = loss;
    a.group_part = group_part;
    a.n_groups = n_groups;

    const int cus = rt_device_cus();
    size_t lds = sch->pool_len * sizeof(double);
    hipStream_t st = (hipStream_t)stream;
    const int beam_mode = gen ? (int)a.beam.v[RT_B_TYPE] : kLoad;

    const uint64_t nk = gen && sch->unroll ? dtab_nk(sch->dt, beam_desc) : 0;
    unsigned grid = 0;
    const bool frames = (flags & RT_TRACE_HIST) && ccd_hist && (flags & RT_TRACE_FLUX) && ccd_flux;
    const LaunchShape shape = launch_shape(sch, gen, frames, rec, n_rays);
    const int block = shape.block, waves = shape.waves;
    // The workgroups of a recording trace with extents, and their rows of keys:
    // at least the rows that any size of the default launches takes, so that a
    // later call of another size finds its memory there, also while a graph is
    // captured; a capture of a launch that could use more (smaller workgroups,
    // set since) has as many workgroups as there are rows.
    auto ext_launch = [&](uint64_t tiles, uint64_t resident) -> int {
        const size_t row = (size_t)sch->n_surf * rt::kExtPerSurf * sizeof(unsigned long long);
        const size_t bytes = row * std::max<uint64_t>(kExtTiles, std::min(tiles, resident));
        const size_t& have = sch->work.have[WorkBufs::EXT_KEYS];
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (have > 0 && have < bytes) HIP_TRY(hipStreamIsCapturing(st, &cs), RT_ERR_FAILED);
        if (cs == hipStreamCaptureStatusNone) {
            const int r = sch->work.ensure(WorkBufs::EXT_KEYS, bytes);
            if (r != RT_OK) return r;
        }
        a.ext = sch->work.get<unsigned long long>(WorkBufs::EXT_KEYS);
        grid = ext_grid(tiles, std::min<uint64_t>(resident, have / row));
        return RT_OK;
    };
    hipFunction_t fn = nullptr;
    if (rt_jit_enabled() && sch->unroll)
        fn = rt_jit_kernel(sch->signature, beam_mode | (nk ? RT_JIT_LTAB : 0),
                           (dump ? RT_JIT_VAR_DUMP : 0) | ((rec & rt::kRecLoss) ? RT_JIT_VAR_LOSS : 0) |
                               ((rec & rt::kRecExt) ? RT_JIT_VAR_EXT : 0) |
                               ((rec & rt::kRecSpots) ? RT_JIT_VAR_SPOTS : 0),
                           block, waves, sch->device);
    if (fn) {
        if (nk) {
            rc = dtab_fill(sch->dt, a, sch->table_dev, sch->pool_dev, sch->n_surf, nk, st);
            if (rc != RT_OK) return rc;
            a.ltab = sch->dt.tab_dev;
            a.lt_nk = nk;
            a.pool_len = 0;                            // every function comes from the table
            lds = 0;
        }
        // persistent grid: the workgroups that are resident at once on every CU
        // (from the compiled kernel's registers and LDS), times grid_mult
        int resident = 0;
        if (hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&resident, fn, block, lds) != hipSuccess ||
            resident < 1)
            resident = 1;
        uint64_t want = (n_rays + block - 1) / block;
        uint64_t cap = (uint64_t)cus * resident * shape.mult;
        grid = (unsigned)(want < cap ? want : cap);
        if (extents && (rc = ext_launch(want, (uint64_t)cus * resident)) != RT_OK) return rc;
        stats_target(a, sch->stat_copies, stats, grid);
        void* params[] = {&a};
        HIP_TRY(hipModuleLaunchKernel(fn, grid, 1, 1, block, 1, 1, (unsigned)lds, st, params, nullptr),
                RT_ERR_FAILED);
        g_last_kernel = "generated";
        if (block_used) *block_used = block;
        if (getenv("RT_HIP_VERBOSE"))
            fprintf(stderr, "rt_hip: trace generated kernel %p, %zu rays, block %d, waves %d, grid %u, table %llu, "
                            "record %d\n", (void*)fn, n_rays, block, waves, grid, (unsigned long long)nk,
                    rec);
    } else {
        uint64_t want = (n_rays + kBlock - 1) / kBlock;
        uint64_t cap = (uint64_t)cus * 8;      // persistent grid: 8 blocks (32 waves) per CU
        grid = (unsigned)(want < cap ? want : cap);
        if (extents && (rc = ext_launch(want, cap)) != RT_OK) return rc;
        // (a kernel that records extents writes its keys: the one without them
        // where the caller wants none)
        auto kern = rec == 0                                ? generic_kernel<0>(beam_mode)
                    : rec == rt::kRecSpots                  ? generic_kernel<rt::kRecSpots>(beam_mode)
                    : rec == (rt::kRecLoss | rt::kRecExt)   ? generic_kernel<rt::kRecLoss | rt::kRecExt>(beam_mode)
                                                            : generic_kernel<rt::kRecLoss>(beam_mode);
        stats_target(a, sch->stat_copies, stats, grid);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), lds, st, a);
        g_last_kernel = "generic";
        if (block_used) *block_used = kBlock;
        if (getenv("RT_HIP_VERBOSE"))
            fprintf(stderr, "rt_hip: trace generic kernel, %zu rays, grid %u, record %d\n", n_rays, grid, rec);
    }
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    if (extents) {
        hipLaunchKernelGGL(rt_ext_reduce_kernel, dim3((unsigned)(sch->n_surf * rt::kExtPerSurf)), dim3(256), 0, st,
                           (const unsigned long long*)a.ext, grid, extents);
        HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    }
    return stats_fold(a, stats, st);
}
}  // namespace

extern "C" int rt_hip_trace(const rt_hip_scheme* sch, const double* beam_desc, uint64_t seed,
                            size_t ray_begin, size_t n_rays, double* X, double* Y, double* Z,
                            double* cX, double* cY, double* cZ, double* lambda, signed char* flag,
                            int flags, unsigned int* ccd_hist, double* ccd_flux,
                            unsigned long long* stats, double* dump, signed char* dump_flag,
                            void* stream) {
    return trace_launch(sch, beam_desc, seed, ray_begin, n_rays, X, Y, Z, cX, cY, cZ, lambda, flag, flags, ccd_hist,
                        ccd_flux, stats, dump, dump_flag, 0, nullptr, nullptr, stream);
}

extern "C" int rt_hip_trace_spots(const rt_hip_scheme* sch, const double* beam_desc, uint64_t seed, size_t n_rays,
                                  size_t n_groups, double* spots, unsigned long long* stats, void* stream) {
    if (!sch) return set_error(RT_ERR_BAD_VALUE, "scheme is NULL");
    if (!spots || n_groups == 0) return set_error(RT_ERR_BAD_VALUE, "spots NULL or no groups");
    if (!beam_desc) return set_error(RT_ERR_BAD_VALUE, "beam_desc is NULL");
    int rc = ensure_device();
    if (rc != RT_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    const uint64_t G = n_groups;
    // one partial row per tile of the launched kernel's workgroup size (the
    // generated kernel's or the generic one's): room for the smaller
    const uint64_t b_min = (uint64_t)std::min(launch_shape(sch, true, false, rt::kRecSpots, n_rays).block, kBlock);
    const uint64_t tiles_max = (n_rays + b_min - 1) / b_min;
    if (tiles_max > (~0ull / 40) / G) return set_error(RT_ERR_BAD_VALUE, "too many rays x groups");
    rc = sch->work.ensure(WorkBufs::TRACE_PART, std::max<uint64_t>(tiles_max, 1) * G * 5 * sizeof(double));
    if (rc != RT_OK) return rc;
    double* part = sch->work.get<double>(WorkBufs::TRACE_PART);
    uint64_t rows = 0;
    if (n_rays > 0) {
        int block = 0;
        rc = trace_launch(sch, beam_desc, seed, 0, n_rays, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                          nullptr, nullptr, RT_TRACE_GENERATE, nullptr, nullptr, stats, nullptr, nullptr,
                          rt::kRecSpots, nullptr, nullptr, stream, part, G, &block);
        if (rc != RT_OK) return rc;
        rows = (n_rays + (uint64_t)block - 1) / (uint64_t)block;
    }
    hipLaunchKernelGGL(rt_spots_rows_kernel<1024>, dim3((unsigned)G), dim3(1024), 0, st, (const double*)part, rows,
                       (const uint64_t*)nullptr, G, spots);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    return RT_OK;
}

extern "C" int rt_hip_trace_record(const rt_hip_scheme* sch, const double* beam_desc, uint64_t seed, size_t n_rays,
                                   double* X, double* Y, double* Z, double* cX, double* cY, double* cZ,
                                   double* lambda, signed char* flag, int flags, unsigned long long* stats,
                                   unsigned char* loss, double* extents, void* stream) {
    if (!sch) return set_error(RT_ERR_BAD_VALUE, "scheme is NULL");
    if (n_rays > 0 && !loss) return set_error(RT_ERR_BAD_VALUE, "loss is NULL");
    if (flags & (RT_TRACE_HIST | RT_TRACE_FLUX))
        return set_error(RT_ERR_BAD_VALUE, "a recording trace accumulates no CCD frame");
    int rc = ensure_device();
    if (rc != RT_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    rc = trace_launch(sch, beam_desc, seed, 0, n_rays, X, Y, Z, cX, cY, cZ, lambda, flag, flags, nullptr, nullptr,
                      stats, nullptr, nullptr, rt::kRecLoss | (extents ? rt::kRecExt : 0), loss, extents, stream);
    if (rc != RT_OK || !extents || n_rays > 0) return rc;
    hipLaunchKernelGGL(rt_ext_reduce_kernel, dim3((unsigned)(sch->n_surf * rt::kExtPerSurf)), dim3(256), 0, st,
                       (const unsigned long long*)nullptr, 0u, extents);           // no ray: every extent empty
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    return RT_OK;
}

// ------------------------------------------------------------ launch tuning

extern "C" int rt_hip_scheme_set_launch(rt_hip_scheme* sch, int block, int waves, int grid_mult) {
    if (!sch) return set_error(RT_ERR_BAD_VALUE, "scheme is NULL");
    if (block != 64 && block != 128 && block != 256 && block != 512 && block != 1024)
        return set_error(RT_ERR_BAD_VALUE, "block must be 64, 128, 256, 512 or 1024 lanes");
    if (waves < 0 || waves > 8) return set_error(RT_ERR_BAD_VALUE, "waves must be in [0, 8]");
    if (grid_mult < 1 || grid_mult > 16) return set_error(RT_ERR_BAD_VALUE, "grid_mult must be in [1, 16]");
    sch->block = block;
    sch->waves = waves;
    sch->grid_mult = grid_mult;
    sch->launch_by = rt_hip_scheme::BY_CALLER;
    return RT_OK;
}

extern "C" int rt_hip_scheme_set_unroll(rt_hip_scheme* sch, int full) {
    if (!sch) return set_error(RT_ERR_BAD_VALUE, "scheme is NULL");
    sch->unroll = full ? 1 : 0;
    return RT_OK;
}

extern "C" int rt_hip_scheme_get_unroll(const rt_hip_scheme* sch, int* full) {
    if (!sch) return set_error(RT_ERR_BAD_VALUE, "scheme is NULL");
    if (full) *full = sch->unroll;
    return RT_OK;
}

extern "C" int rt_hip_scheme_get_launch(const rt_hip_scheme* sch, int* block, int* waves, int* grid_mult) {
    if (!sch) return set_error(RT_ERR_BAD_VALUE, "scheme is NULL");
    if (block) *block = sch->block;
    if (waves) *waves = sch->waves;
    if (grid_mult) *grid_mult = sch->grid_mult;
    return RT_OK;
}

namespace {
struct DevBuf {
    void* p = nullptr;
    ~DevBuf() { if (p) (void)hipFree(p); }
    bool alloc(size_t bytes) { return hipMalloc(&p, bytes ? bytes : 8) == hipSuccess; }
};
}  // namespace

// Time every candidate launch of the generated kernel on n_sample rays of the
// beam (generated from `seed`, traced with `flags`) and keep the fastest.
extern "C" int rt_hip_autotune(rt_hip_scheme* sch, const double* beam_desc, uint64_t seed, size_t n_sample,
                               int flags, double* best_ms, void* stream) {
    if (!sch) return set_error(RT_ERR_BAD_VALUE, "scheme is NULL");
    if (!beam_desc) return set_error(RT_ERR_BAD_VALUE, "autotuning traces a generated beam: beam_desc is NULL");
    if (n_sample == 0) return set_error(RT_ERR_BAD_VALUE, "n_sample must be > 0");
    int rc = validate_beam(beam_desc);
    if (rc != RT_OK) return rc;
    rc = ensure_device();
    if (rc != RT_OK) return rc;
    flags |= RT_TRACE_GENERATE;
    // buffers of the sample and of the detector frames
    DevBuf rays, flag, hist, flux;
    size_t npix = 0;
    for (int s = 0; s < sch->n_surf; ++s) {
        const double* p = sch->table.data() + (size_t)s * RT_SURF_STRIDE;
        if ((int)p[RT_S_TYPE] == RT_DETECTOR && p[RT_S_CCD_XDIM] > 0.0)
            npix = (size_t)p[RT_S_CCD_XDIM] * (size_t)p[RT_S_CCD_YDIM];
    }
    const bool store = (flags & RT_TRACE_STORE) != 0;
    if ((store && (!rays.alloc(7 * n_sample * sizeof(double)) || !flag.alloc(n_sample))) ||
        ((flags & RT_TRACE_HIST) && npix && !hist.alloc(npix * sizeof(unsigned))) ||
        ((flags & RT_TRACE_FLUX) && npix && !flux.alloc(npix * sizeof(double))))
        return set_error(RT_ERR_BAD_ALLOC, "autotune buffers");
    double* R = (double*)rays.p;
    // each launch traces a new beam (seed, seed + 1, ...), as a workload does:
    // repeating one beam repeats its frame accesses and runs faster
    uint64_t launch_no = 0;
    auto run = [&]() {
        return rt_hip_trace(sch, beam_desc, seed + launch_no++, 0, n_sample, store ? R : nullptr,
                            store ? R + n_sample : nullptr, store ? R + 2 * n_sample : nullptr,
                            store ? R + 3 * n_sample : nullptr, store ? R + 4 * n_sample : nullptr,
                            store ? R + 5 * n_sample : nullptr, store ? R + 6 * n_sample : nullptr,
                            store ? (signed char*)flag.p : nullptr, flags, (unsigned*)hist.p, (double*)flux.p,
                            nullptr, nullptr, nullptr, stream);
    };
    hipStream_t st = (hipStream_t)stream;
    hipEvent_t e0, e1;
    HIP_TRY(hipEventCreate(&e0), RT_ERR_FAILED);
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return set_error(RT_ERR_FAILED, "hipEventCreate");
    }
    // the launches of 128 and 256 lanes, and of as many lanes as an untuned trace
    // of these rays takes where those are more (512, for large traces into both
    // frames: the echelle's 1e7 rays 897 us, 942 with 256 lanes at best).  Of
    // those the untuned trace's waves and the compiler's choice, grid multiples
    // 8 and 16: 5 and 6 waves are within 0.5% of them, 8 waves and smaller
    // multiples 3-6% slower, and every kernel takes 0.3 s to compile.
    std::vector<int> blocks = {128, 256};
    const bool frames = (flags & RT_TRACE_HIST) && hist.p && (flags & RT_TRACE_FLUX) && flux.p;
    {
        const auto by = sch->launch_by;
        sch->launch_by = rt_hip_scheme::BY_RULE;
        const int b = launch_shape(sch, true, frames, 0, n_sample).block;
        sch->launch_by = by;
        if (b > 256) blocks.push_back(b);
    }
    const int wavess[] = {0, 5, 6, 7, 8};
    const int mults[] = {1, 2, 4, 8, 16};
    struct Cand { int b, w, m; float ms; int regs, local, u; };
    std::vector<Cand> cands;
    const int bb0 = sch->block, bw0 = sch->waves, bm0 = sch->grid_mult, bu0 = sch->unroll;
    const auto by0 = sch->launch_by;
    sch->launch_by = rt_hip_scheme::BY_CALLER;
    // mean time of `reps` back-to-back launches of candidate c
    auto timed = [&](const Cand& c, int reps, float& ms) -> int {
        sch->block = c.b; sch->waves = c.w; sch->grid_mult = c.m; sch->unroll = c.u;
        (void)hipEventRecord(e0, st);
        int r = RT_OK;
        for (int k = 0; k < reps && r == RT_OK; ++k) r = run();
        (void)hipEventRecord(e1, st);
        if (r != RT_OK) return r;
        if (hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess)
            return set_error(RT_ERR_FAILED, "autotune timing");
        ms /= (float)reps;
        return RT_OK;
    };
    // every candidate launched once (compiling its kernel); its registers and
    // private (scratch) bytes per lane as the runtime reports them
    // (surface unroll depth: the fully unrolled generated kernel under every
    // launch, and the runtime loop of the generic kernel, whose launch is fixed)
    rc = RT_OK;
    const int beam_mode = (int)beam_desc[RT_B_TYPE];
    {
        Cand c{kBlock, 0, 1, 1e30f, 0, 0, 0};
        sch->unroll = 0;
        if ((rc = run()) == RT_OK && hipStreamSynchronize(st) != hipSuccess) rc = set_error(RT_ERR_FAILED, "autotune");
        if (rc == RT_OK) cands.push_back(c);
    }
    sch->unroll = 1;
    for (int b : blocks)
        for (int w : wavess)
            for (int m : mults) {
                if (rc != RT_OK || !rt_jit_enabled()) break;
                if (b > 256 && (m < 8 || (w != 0 && w != kDefaultWaves))) continue;
                Cand c{b, w, m, 1e30f, 0, 0, 1};
                sch->block = b; sch->waves = w; sch->grid_mult = m;
                if ((rc = run()) != RT_OK) break;
                if (hipStreamSynchronize(st) != hipSuccess) { rc = set_error(RT_ERR_FAILED, "autotune"); break; }
                int local = 0;
                const int mode = beam_mode | (dtab_nk(sch->dt, beam_desc) ? RT_JIT_LTAB : 0);
                hipFunction_t fn =
                    rt_jit_enabled() ? rt_jit_kernel(sch->signature, mode, false, b, w, sch->device) : nullptr;
                if (fn && hipFuncGetAttribute(&local, HIP_FUNC_ATTRIBUTE_LOCAL_SIZE_BYTES, fn) != hipSuccess)
                    local = 0;
                if (fn && hipFuncGetAttribute(&c.regs, HIP_FUNC_ATTRIBUTE_NUM_REGS, fn) != hipSuccess) c.regs = 0;
                c.local = local;
                cands.push_back(c);
            }
    // launches that spill more than kMaxScratch bytes per lane are set aside
    // when one at or below it exists: on the fused echelle trace they timed
    // about 10% faster here than in the caller's sustained loops (7 waves/SIMD,
    // 96 B per lane: 1.20 against 1.32 ms), the lighter ones within 2%
    constexpr int kMaxScratch = 64;
    if (std::any_of(cands.begin(), cands.end(), [](const Cand& c) { return c.local <= kMaxScratch; }))
        cands.erase(std::remove_if(cands.begin(), cands.end(), [](const Cand& c) { return c.local > kMaxScratch; }),
                    cands.end());
    // Timed as the workload runs, back to back: the clock of a sustained FP64
    // load settles below that of isolated launches, and by how much depends
    // on the launch (occupancy, scratch traffic), so isolated launches rank
    // candidates differently.  The clock also drifts, so candidates are timed
    // in interleaved rounds: screening by the best of 3 rounds of 3-launch
    // bursts, then the four best ranked by the median of 5 rounds of
    // 20-launch bursts (long enough for the clock to settle under launches
    // that spill to scratch); within 0.5% the one with less scratch memory
    // wins.
    auto rounds_of = [&](std::vector<Cand>& cs, int rounds, int reps, std::vector<std::vector<float>>& t) {
        t.assign(cs.size(), {});
        for (int r = 0; r < rounds && rc == RT_OK; ++r)
            for (size_t i = 0; i < cs.size() && rc == RT_OK; ++i) {
                float ms = 0.0f;
                rc = timed(cs[i], reps, ms);
                t[i].push_back(ms);
            }
    };
    int bb = bb0, bw = bw0, bm = bm0, bu = bu0;
    double best = 1e300;
    std::vector<std::vector<float>> t;
    if (rc == RT_OK && !cands.empty()) {
        rounds_of(cands, 3, 3, t);
        for (size_t i = 0; i < cands.size() && rc == RT_OK; ++i)
            cands[i].ms = *std::min_element(t[i].begin(), t[i].end());
    }
    // RT_HIP_AUTOTUNE_LOG=1: every candidate's screening time on stderr
    const char* lg = getenv("RT_HIP_AUTOTUNE_LOG");
    const bool log = lg && lg[0] == '1';
    if (log)
        for (const Cand& c : cands)
            fprintf(stderr, "rt_hip autotune: %d,%d,%d %s, registers %d, private %d B: screening %.4f ms\n", c.b,
                    c.w, c.m, c.u ? "unrolled" : "loop", c.regs, c.local, c.ms);
    if (rc == RT_OK && !cands.empty()) {
        std::sort(cands.begin(), cands.end(), [](const Cand& x, const Cand& y) { return x.ms < y.ms; });
        if (cands.size() > 4) cands.resize(4);
        rounds_of(cands, 5, 20, t);
        int best_local = 0;
        for (size_t i = 0; i < cands.size() && rc == RT_OK; ++i) {
            std::sort(t[i].begin(), t[i].end());
            const double med = t[i][t[i].size() / 2];
            if (log) fprintf(stderr, "rt_hip autotune: %d,%d,%d %s median of 5 %.4f ms\n", cands[i].b, cands[i].w,
                             cands[i].m, cands[i].u ? "unrolled" : "loop", med);
            const bool better = best == 1e300 || med < best * (1.0 - 0.005) ||
                                (med < best * (1.0 + 0.005) && (cands[i].local < best_local ||
                                                                 (cands[i].local == best_local && med < best)));
            if (better) {
                best = med;
                best_local = cands[i].local;
                bb = cands[i].b; bw = cands[i].w; bm = cands[i].m; bu = cands[i].u;
            }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    sch->block = bb; sch->waves = bw; sch->grid_mult = bm; sch->unroll = bu;
    if (rc == RT_OK && best < 1e300) {
        sch->launch_by = rt_hip_scheme::BY_TUNER;
        sch->tuned_frames = frames;
    } else {
        sch->launch_by = by0;
    }
    if (rc != RT_OK) return rc;
    if (best_ms) *best_ms = best;
    return RT_OK;
}

// -------------------------------------------------------------- batched traces

struct rt_hip_batch {
    int device = 0, n_inst = 0, n_surf = 0;
    std::string signature;           // of the union structure (rotations/translations of any instance)
    size_t pool_len = 0;
    std::vector<double> dtables;     // n_inst x n_surf device records
    std::vector<double> dpool;
    std::vector<uint64_t> ray_start; // n_inst + 1
    double* tables_dev = nullptr;
    double* pool_dev = nullptr;
    uint64_t* ray_start_dev = nullptr;
    int block = rt::kBlock, waves = kDefaultWaves, grid_mult = kDefaultGridMult;   // as for one scheme
    int tiles_block = 0;             // workgroup size the tile arrays below are built for
    uint64_t n_tiles = 0;
    uint64_t* tile_start_dev = nullptr;
    uint32_t* tile_inst_dev = nullptr;   // instance of each tile
    double* moments_dev = nullptr;
    // descent map (rt_hip_batch_descend) in work's DESCEND slot: map_start[n_surf + 1]
    // then the (j, field) pairs, re-made (in a new buffer) when the parameter list changes
    std::vector<int> descend_key;
    // working memory of the batch's adjoints, spot reductions and descent steps
    mutable WorkBufs work;
    Ltab lt;
    unsigned long long* stat_copies = nullptr;   // as rt_hip_scheme::stat_copies
    // a beam per instance (rt_hip_batch_set_beams): n_inst x kBeamRec records,
    // used while beams_on (kept allocated until the batch is destroyed: a
    // captured graph may hold its address)
    double* beams_dev = nullptr;
    bool beams_on = false;
    int beam_type = -1;
};

struct rt_hip_graph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

namespace {

void free_batch(rt_hip_batch* b) {
    if (!b) return;
    (void)hipFree(b->tables_dev);
    (void)hipFree(b->pool_dev);
    (void)hipFree(b->ray_start_dev);
    (void)hipFree(b->tile_inst_dev);
    b->work.release();
    (void)hipFree(b->tile_start_dev);
    (void)hipFree(b->moments_dev);
    (void)hipFree(b->beams_dev);
    (void)hipFree(b->stat_copies);
    b->lt.release();
    delete b;
}

// device records of every instance (one shared pool) and the kernel signature
int build_batch_tables(rt_hip_batch* b, const double* tables, const double* pool, size_t pool_len) {
    const size_t rec = (size_t)b->n_surf * RT_SURF_STRIDE;
    const size_t drec = (size_t)b->n_surf * rt::DEV_STRIDE;
    b->dtables.assign((size_t)b->n_inst * drec, 0.0);
    std::string base;
    std::vector<double> uni;
    for (int i = 0; i < b->n_inst; ++i) {
        rt_hip_scheme tmp;
        tmp.n_surf = b->n_surf;
        tmp.table.assign(tables + i * rec, tables + (i + 1) * rec);
        if (pool_len) tmp.pool.assign(pool, pool + pool_len);
        build_device_tables(&tmp);
        std::copy(tmp.dtable.begin(), tmp.dtable.end(), b->dtables.begin() + i * drec);
        // structure without the rotations and translations must be the same for all
        std::vector<double> st = tmp.dtable;
        for (int s = 0; s < b->n_surf; ++s)
            for (int j = 0; j < 3; ++j) {
                st[s * rt::DEV_STRIDE + RT_S_ANG + j] = 0.0;
                st[s * rt::DEV_STRIDE + RT_S_DIST + j] = 0.0;
            }
        std::string sig = rt_jit_signature(st.data(), b->n_surf);
        if (i == 0) {
            base = sig;
            b->dpool = tmp.dpool;
            b->pool_len = tmp.dpool.size();
            uni = tmp.dtable;
        } else if (sig != base) {
            return set_error(RT_ERR_BAD_VALUE, "instance %d differs in structure from instance 0", i);
        }
        // union of the rotations and translations present in any instance: a zero angle or
        // offset applied as a rotation or translation leaves finite values unchanged
        for (int s = 0; s < b->n_surf; ++s)
            for (int j = 0; j < 3; ++j) {
                double* u = uni.data() + s * rt::DEV_STRIDE;
                const double* d = tmp.dtable.data() + s * rt::DEV_STRIDE;
                if (d[RT_S_ANG + j] != 0.0) u[RT_S_ANG + j] = 1.0;
                if (d[RT_S_DIST + j] != 0.0) u[RT_S_DIST + j] = 1.0;
            }
    }
    b->signature = rt_jit_signature(uni.data(), b->n_surf);
    return RT_OK;
}

// tile arrays for workgroups of b->block lanes
int prepare_tiles(rt_hip_batch* b) {
    if (b->tiles_block == b->block) return RT_OK;
    std::vector<uint64_t> ts(b->n_inst + 1, 0);
    for (int i = 0; i < b->n_inst; ++i) {
        uint64_t n = b->ray_start[i + 1] - b->ray_start[i];
        ts[i + 1] = ts[i] + (n + b->block - 1) / b->block;
    }
    // arrays of another workgroup size stay allocated until the batch is
    // destroyed: a graph captured with them may still be replayed
    for (void* q : {(void*)b->tile_start_dev, (void*)b->tile_inst_dev, (void*)b->moments_dev})
        if (q) b->work.owned.push_back(q);
    b->tile_start_dev = nullptr;
    b->tile_inst_dev = nullptr;
    b->moments_dev = nullptr;
    b->tiles_block = 0;
    b->n_tiles = ts[b->n_inst];
    std::vector<uint32_t> ti(b->n_tiles ? b->n_tiles : 1, 0);
    for (int i = 0; i < b->n_inst; ++i)
        for (uint64_t t = ts[i]; t < ts[i + 1]; ++t) ti[t] = (uint32_t)i;
    HIP_TRY(hipMalloc(&b->tile_inst_dev, ti.size() * sizeof(uint32_t)), RT_ERR_BAD_ALLOC);
    HIP_TRY(hipMemcpy(b->tile_inst_dev, ti.data(), ti.size() * sizeof(uint32_t), hipMemcpyHostToDevice),
            RT_ERR_FAILED);
    HIP_TRY(hipMalloc(&b->tile_start_dev, ts.size() * sizeof(uint64_t)), RT_ERR_BAD_ALLOC);
    HIP_TRY(hipMalloc(&b->moments_dev, (b->n_tiles ? b->n_tiles : 1) * 5 * sizeof(double)), RT_ERR_BAD_ALLOC);
    HIP_TRY(hipMemcpy(b->tile_start_dev, ts.data(), ts.size() * sizeof(uint64_t), hipMemcpyHostToDevice),
            RT_ERR_FAILED);
    b->tiles_block = b->block;
    return RT_OK;
}

}  // namespace

extern "C" int rt_hip_batch_create(const double* tables, int n_inst, int n_surf, const double* spline_pool,
                                   size_t pool_len, const uint64_t* ray_counts, rt_hip_batch** out) {
    if (!out) return set_error(RT_ERR_BAD_VALUE, "out is NULL");
    *out = nullptr;
    if (!tables || !ray_counts || n_inst < 1) return set_error(RT_ERR_BAD_VALUE, "bad batch arguments");
    const size_t rec = (size_t)n_surf * RT_SURF_STRIDE;
    for (int i = 0; i < n_inst; ++i) {
        int rc = rt_hip_validate_scheme(tables + i * rec, n_surf, spline_pool, pool_len);
        if (rc != RT_OK) return rc;
        if (ray_counts[i] > (1ull << 40)) return set_error(RT_ERR_BAD_VALUE, "instance %d: too many rays", i);
    }
    rt_hip_batch* b = new (std::nothrow) rt_hip_batch();
    if (!b) return set_error(RT_ERR_BAD_ALLOC, "out of host memory");
    b->n_inst = n_inst;
    b->n_surf = n_surf;
    b->ray_start.assign(n_inst + 1, 0);
    for (int i = 0; i < n_inst; ++i) b->ray_start[i + 1] = b->ray_start[i] + ray_counts[i];
    int rc = build_batch_tables(b, tables, spline_pool, pool_len);
    if (rc == RT_OK) rc = ensure_device();
    if (rc != RT_OK) { free_batch(b); return rc; }
    b->device = g_dev.device;
    size_t tb = b->dtables.size() * sizeof(double);
    size_t pb = (b->dpool.empty() ? 1 : b->dpool.size()) * sizeof(double);
    size_t rb = b->ray_start.size() * sizeof(uint64_t);
    if (hipMalloc(&b->tables_dev, tb) != hipSuccess || hipMalloc(&b->pool_dev, pb) != hipSuccess ||
        hipMalloc(&b->ray_start_dev, rb) != hipSuccess) {
        free_batch(b);
        return set_error(RT_ERR_BAD_ALLOC, "hipMalloc of batch tables failed");
    }
    if (hipMemcpy(b->tables_dev, b->dtables.data(), tb, hipMemcpyHostToDevice) != hipSuccess ||
        (!b->dpool.empty() &&
         hipMemcpy(b->pool_dev, b->dpool.data(), b->dpool.size() * sizeof(double), hipMemcpyHostToDevice) !=
             hipSuccess) ||
        hipMemcpy(b->ray_start_dev, b->ray_start.data(), rb, hipMemcpyHostToDevice) != hipSuccess) {
        free_batch(b);
        return set_error(RT_ERR_FAILED, "upload of batch tables failed");
    }
    rc = prepare_tiles(b);
    if (rc == RT_OK) rc = ltab_setup(b->lt, b->signature, b->dtables.data(), b->n_inst, b->n_surf);
    if (rc == RT_OK) rc = stat_copies_alloc(&b->stat_copies);
    if (rc != RT_OK) { free_batch(b); return rc; }
    *out = b;
    return RT_OK;
}

extern "C" int rt_hip_batch_update(rt_hip_batch* b, const double* tables, const double* spline_pool,
                                   size_t pool_len) {
    if (!b || !tables) return set_error(RT_ERR_BAD_VALUE, "bad batch arguments");
    const size_t rec = (size_t)b->n_surf * RT_SURF_STRIDE;
    for (int i = 0; i < b->n_inst; ++i) {
        int rc = rt_hip_validate_scheme(tables + i * rec, b->n_surf, spline_pool, pool_len);
        if (rc != RT_OK) return rc;
    }
    std::string sig = b->signature;
    size_t old_pool = b->pool_len;
    int rc = build_batch_tables(b, tables, spline_pool, pool_len);
    if (rc != RT_OK) return rc;
    if (b->signature != sig || b->pool_len != old_pool)
        return set_error(RT_ERR_BAD_VALUE, "updated tables change the batch structure; create a new batch");
    HIP_TRY(hipMemcpy(b->tables_dev, b->dtables.data(), b->dtables.size() * sizeof(double), hipMemcpyHostToDevice),
            RT_ERR_FAILED);
    if (!b->dpool.empty())
        HIP_TRY(hipMemcpy(b->pool_dev, b->dpool.data(), b->dpool.size() * sizeof(double), hipMemcpyHostToDevice),
                RT_ERR_FAILED);
    return ltab_setup(b->lt, b->signature, b->dtables.data(), b->n_inst, b->n_surf);
}

extern "C" int rt_hip_batch_set_beams(rt_hip_batch* b, const double* beam_descs) {
    if (!b) return set_error(RT_ERR_BAD_VALUE, "batch is NULL");
    if (!beam_descs) {
        b->beams_on = false;
        b->beam_type = -1;
        return RT_OK;
    }
    std::vector<double> recs((size_t)b->n_inst * rt::kBeamRec);
    const int type = (int)beam_descs[RT_B_TYPE];
    for (int i = 0; i < b->n_inst; ++i) {
        const double* d = beam_descs + (size_t)i * RT_BEAM_STRIDE;
        int rc = validate_beam(d);
        if (rc != RT_OK) return rc;
        if ((int)d[RT_B_TYPE] != type)
            return set_error(RT_ERR_BAD_VALUE, "instance %d: beam type %d differs from instance 0 (%d)", i,
                             (int)d[RT_B_TYPE], type);
        TraceArgs a;
        memset(&a, 0, sizeof a);
        memcpy(a.beam.v, d, sizeof a.beam.v);
        beam_uniforms(a);
        memcpy(recs.data() + (size_t)i * rt::kBeamRec, &a.beam, sizeof a.beam);
    }
    int rc = ensure_device();
    if (rc != RT_OK) return rc;
    if (!b->beams_dev) HIP_TRY(hipMalloc(&b->beams_dev, recs.size() * sizeof(double)), RT_ERR_BAD_ALLOC);
    HIP_TRY(hipMemcpy(b->beams_dev, recs.data(), recs.size() * sizeof(double), hipMemcpyHostToDevice),
            RT_ERR_FAILED);
    b->beam_type = type;
    b->beams_on = true;
    return RT_OK;
}

extern "C" int rt_hip_batch_destroy(rt_hip_batch* b) {
    free_batch(b);
    return RT_OK;
}

extern "C" int rt_hip_batch_info(const rt_hip_batch* b, uint64_t* total_rays, uint64_t* n_tiles) {
    if (!b) return set_error(RT_ERR_BAD_VALUE, "batch is NULL");
    if (total_rays) *total_rays = b->ray_start[b->n_inst];
    if (n_tiles) *n_tiles = b->n_tiles;
    return RT_OK;
}

extern "C" int rt_hip_batch_set_launch(rt_hip_batch* b, int block, int waves, int grid_mult) {
    if (!b) return set_error(RT_ERR_BAD_VALUE, "batch is NULL");
    if (block != 64 && block != 128 && block != 256 && block != 512 && block != 1024)
        return set_error(RT_ERR_BAD_VALUE, "block must be 64, 128, 256, 512 or 1024 lanes");
    if (waves < 0 || waves > 8) return set_error(RT_ERR_BAD_VALUE, "waves must be in [0, 8]");
    if (grid_mult < 1 || grid_mult > 16) return set_error(RT_ERR_BAD_VALUE, "grid_mult must be in [1, 16]");
    b->block = block;
    b->waves = waves;
    b->grid_mult = grid_mult;
    return prepare_tiles(b);
}

namespace {
// rt_hip_batch_trace; group_part (when set): the group spot partials of every
// tile, n_groups groups per tile (TraceArgs::group_part)
int batch_trace(const rt_hip_batch* bc, const double* beam_desc, uint64_t seed, int flags, double* X, double* Y,
                double* Z, double* cX, double* cY, double* cZ, double* lambda, signed char* flag, double* spots,
                unsigned long long* stats, void* stream, double* group_part, uint64_t n_groups) {
    rt_hip_batch* b = const_cast<rt_hip_batch*>(bc);
    if (!b) return set_error(RT_ERR_BAD_VALUE, "batch is NULL");
    int rc = validate_beam(beam_desc);
    if (rc != RT_OK) return rc;
    if ((flags & RT_TRACE_STORE) && (!X || !Y || !Z || !cX || !cY || !cZ || !lambda || !flag))
        return set_error(RT_ERR_BAD_VALUE, "RT_TRACE_STORE needs all ray buffers");
    if (flags & (RT_TRACE_HIST | RT_TRACE_FLUX))
        return set_error(RT_ERR_BAD_VALUE, "batched traces reduce spots, not CCD frames");
    rc = ensure_device();
    if (rc != RT_OK) return rc;
    rc = prepare_tiles(b);
    if (rc != RT_OK) return rc;
    if (b->n_tiles == 0) return RT_OK;

    TraceArgs a;
    memset(&a, 0, sizeof a);
    memcpy(a.beam.v, beam_desc, sizeof a.beam.v);
    beam_uniforms(a);
    a.table = b->tables_dev;
    a.pool = b->pool_dev;
    a.n_surf = b->n_surf;
    a.pool_len = (int)b->pool_len;
    a.flags = flags | RT_TRACE_GENERATE;
    a.seed = seed;
    a.n = b->ray_start[b->n_inst];
    if (flags & RT_TRACE_STORE) {
        a.X = X; a.Y = Y; a.Z = Z; a.cX = cX; a.cY = cY; a.cZ = cZ; a.L = lambda; a.F = flag;
    }
    a.tile_start = b->tile_start_dev;
    a.tile_inst = b->tile_inst_dev;
    a.ray_start = b->ray_start_dev;
    a.tile_moments = spots ? b->moments_dev : nullptr;
    a.group_part = group_part;
    a.n_groups = n_groups;
    a.n_inst = (uint64_t)b->n_inst;
    a.n_tiles = b->n_tiles;
    a.inst_stride = (uint64_t)b->n_surf * rt::DEV_STRIDE;

    const int cus = rt_device_cus();
    size_t lds = b->pool_len * sizeof(double);
    hipStream_t st = (hipStream_t)stream;
    const int beam_mode = (int)a.beam.v[RT_B_TYPE];
    if (b->beams_on) {
        if (beam_mode != b->beam_type)
            return set_error(RT_ERR_BAD_VALUE, "beam type %d differs from the instances' beams (%d)", beam_mode,
                             b->beam_type);
        a.inst_beams = b->beams_dev;
    }
    const uint64_t nk = b->beams_on ? 0 : ltab_nk(b->lt, beam_desc);
    hipFunction_t fn = nullptr;
    if (rt_jit_enabled())
        fn = rt_jit_kernel(b->signature, beam_mode | (nk ? RT_JIT_LTAB : 0), false, b->block, b->waves, b->device,
                           true);
    if (fn) {
        if (nk) {
            rc = ltab_fill(b->lt, a, b->pool_dev, nk, st);
            if (rc != RT_OK) return rc;
            a.ltab = b->lt.tab_dev;
            a.lt_nk = nk;
            a.pool_len = 0;                            // every function comes from the table
            lds = 0;
        }
        int resident = 0;
        if (hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&resident, fn, b->block, lds) != hipSuccess ||
            resident < 1)
            resident = 1;
        uint64_t cap = (uint64_t)cus * resident * b->grid_mult;
        unsigned grid = (unsigned)(b->n_tiles < cap ? b->n_tiles : cap);
        stats_target(a, b->stat_copies, stats, grid);
        void* params[] = {&a};
        HIP_TRY(hipModuleLaunchKernel(fn, grid, 1, 1, b->block, 1, 1, (unsigned)lds, st, params, nullptr),
                RT_ERR_FAILED);
        g_last_kernel = "generated";
    } else {
        if (b->block != kBlock) {
            // the generic kernel is built for kBlock lanes: retile for it
            b->block = kBlock;
            rc = prepare_tiles(b);
            if (rc != RT_OK) return rc;
            a.tile_start = b->tile_start_dev;
            a.tile_inst = b->tile_inst_dev;
            a.tile_moments = spots ? b->moments_dev : nullptr;
            a.n_tiles = b->n_tiles;
        }
        uint64_t cap = (uint64_t)cus * 8;
        unsigned grid = (unsigned)(b->n_tiles < cap ? b->n_tiles : cap);
        auto kern = beam_mode == RT_BEAM_PARALLEL ? rt_trace_batch_kernel<RT_BEAM_PARALLEL>
                  : beam_mode == RT_BEAM_CONIC    ? rt_trace_batch_kernel<RT_BEAM_CONIC>
                                                  : rt_trace_batch_kernel<RT_BEAM_GAUSS>;
        stats_target(a, b->stat_copies, stats, grid);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), lds, st, a);
        g_last_kernel = "generic";
    }
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    rc = stats_fold(a, stats, st);
    if (rc != RT_OK) return rc;
    if (spots) {
        hipLaunchKernelGGL(rt_batch_spots_kernel, dim3((unsigned)b->n_inst), dim3(kInstSpotThreads), 0, st,
                           (const double*)b->moments_dev, (const uint64_t*)b->tile_start_dev, (uint64_t)b->n_inst,
                           spots);
        HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    }
    return RT_OK;
}
}  // namespace

extern "C" int rt_hip_batch_trace(const rt_hip_batch* bc, const double* beam_desc, uint64_t seed, int flags,
                                  double* X, double* Y, double* Z, double* cX, double* cY, double* cZ,
                                  double* lambda, signed char* flag, double* spots,
                                  unsigned long long* stats, void* stream) {
    return batch_trace(bc, beam_desc, seed, flags, X, Y, Z, cX, cY, cZ, lambda, flag, spots, stats, stream, nullptr,
                       0);
}

extern "C" int rt_hip_batch_trace_group_spots(const rt_hip_batch* bc, const double* beam_desc, uint64_t seed,
                                              size_t n_groups, double* spots, unsigned long long* stats,
                                              void* stream) {
    rt_hip_batch* b = const_cast<rt_hip_batch*>(bc);
    if (!b) return set_error(RT_ERR_BAD_VALUE, "batch is NULL");
    if (!spots || n_groups == 0) return set_error(RT_ERR_BAD_VALUE, "spots NULL or no groups");
    int rc = ensure_device();
    if (rc != RT_OK) return rc;
    const uint64_t G = n_groups;
    // partial rows for the tiling of the smaller workgroup the launch may use
    // (the generic kernel retiles to its own)
    const uint64_t b_min = (uint64_t)std::min(b->block, kBlock);
    uint64_t tiles_max = 0;
    for (int i = 0; i < b->n_inst; ++i) tiles_max += (b->ray_start[i + 1] - b->ray_start[i] + b_min - 1) / b_min;
    if (tiles_max > (~0ull / 40) / G) return set_error(RT_ERR_BAD_VALUE, "too many rays x groups");
    rc = b->work.ensure(WorkBufs::TRACE_PART, std::max<uint64_t>(tiles_max, 1) * G * 5 * sizeof(double));
    if (rc != RT_OK) return rc;
    double* part = b->work.get<double>(WorkBufs::TRACE_PART);
    rc = batch_trace(b, beam_desc, seed, RT_TRACE_GENERATE, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                     nullptr, nullptr, nullptr, stats, stream, part, G);
    if (rc != RT_OK) return rc;
    // an instance with no rays has no rows: its spots stay empty
    hipLaunchKernelGGL(rt_spots_rows_kernel<256>, dim3((unsigned)(b->n_inst * G)), dim3(256), 0,
                       (hipStream_t)stream,
                       (const double*)part, (uint64_t)b->n_tiles, (const uint64_t*)b->tile_start_dev, G, spots);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    return RT_OK;
}

// A batched trace with fixed arguments recorded once as a hipGraph (trace and
// spot kernels), replayed by rt_hip_graph_launch.  Table contents may change
// between replays (rt_hip_batch_update); the stream must not be the null stream.
extern "C" int rt_hip_batch_graph_create(const rt_hip_batch* b, const double* beam_desc, uint64_t seed, int flags,
                                         double* X, double* Y, double* Z, double* cX, double* cY, double* cZ,
                                         double* lambda, signed char* flag, double* spots,
                                         unsigned long long* stats, void* stream, rt_hip_graph** out) {
    if (!out) return set_error(RT_ERR_BAD_VALUE, "out is NULL");
    *out = nullptr;
    if (!b) return set_error(RT_ERR_BAD_VALUE, "batch is NULL");
    if (!stream) return set_error(RT_ERR_BAD_VALUE, "graph capture needs a created stream");
    hipStream_t st = (hipStream_t)stream;
    // compile and load the kernel before the capture
    if (rt_jit_enabled()) {
        int rc = validate_beam(beam_desc);
        if (rc != RT_OK) return rc;
        (void)rt_jit_kernel(b->signature,
                            (int)beam_desc[RT_B_TYPE] | (rt_batch_ltab_nk(b, beam_desc) ? RT_JIT_LTAB : 0),
                            false, b->block, b->waves, b->device, true);
    }
    rt_hip_graph* g = new (std::nothrow) rt_hip_graph();
    if (!g) return set_error(RT_ERR_BAD_ALLOC, "out of host memory");
    HIP_TRY(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal), RT_ERR_FAILED);
    int rc = rt_hip_batch_trace(b, beam_desc, seed, flags, X, Y, Z, cX, cY, cZ, lambda, flag, spots, stats, stream);
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(st, &graph);
    if (rc != RT_OK || e != hipSuccess || !graph) {
        if (graph) (void)hipGraphDestroy(graph);
        delete g;
        return rc != RT_OK ? rc : set_error(RT_ERR_FAILED, "graph capture: %s", hipGetErrorString(e));
    }
    g->graph = graph;
    if (hipGraphInstantiate(&g->exec, graph, nullptr, nullptr, 0) != hipSuccess) {
        (void)hipGraphDestroy(graph);
        delete g;
        return set_error(RT_ERR_FAILED, "hipGraphInstantiate failed");
    }
    *out = g;
    return RT_OK;
}

extern "C" int rt_hip_graph_launch(rt_hip_graph* g, void* stream) {
    if (!g || !g->exec) return set_error(RT_ERR_BAD_VALUE, "graph is NULL");
    HIP_TRY(hipGraphLaunch(g->exec, (hipStream_t)stream), RT_ERR_FAILED);
    return RT_OK;
}

extern "C" int rt_hip_graph_destroy(rt_hip_graph* g) {
    if (!g) return RT_OK;
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    delete g;
    return RT_OK;
}

// device tables of a scheme, for the other translation units of the library
int rt_batch_view(const rt_hip_batch* b, BatchView* v) {
    if (!b) return set_error(RT_ERR_BAD_VALUE, "batch is NULL");
    if (b->tiles_block != b->block) return set_error(RT_ERR_FAILED, "batch tiles not prepared");
    v->device = b->device;
    v->n_inst = b->n_inst;
    v->n_surf = b->n_surf;
    v->block = b->block;
    v->signature = &b->signature;
    v->tables_dev = b->tables_dev;
    v->pool_dev = b->pool_dev;
    v->pool_len = b->pool_len;
    v->ray_start_dev = b->ray_start_dev;
    v->tile_start_dev = b->tile_start_dev;
    v->tile_inst_dev = b->tile_inst_dev;
    v->beams_dev = b->beams_on ? b->beams_dev : nullptr;
    v->beam_type = b->beam_type;
    v->n_tiles = b->n_tiles;
    v->dtables = b->dtables.data();
    v->ray_start = b->ray_start.data();
    return RT_OK;
}

const std::string& rt_scheme_signature(const rt_hip_scheme* s) { return s->signature; }

uint64_t rt_scheme_dtab_nk(const rt_hip_scheme* s, const double* beam_desc) { return dtab_nk(s->dt, beam_desc); }

int rt_scheme_dtab_fill(const rt_hip_scheme* s, const double* beam_desc, uint64_t nk, hipStream_t stream,
                        const double** tab) {
    TraceArgs a;
    memset(&a, 0, sizeof a);
    memcpy(a.beam.v, beam_desc, sizeof a.beam.v);
    *tab = s->dt.tab_dev;
    return dtab_fill(s->dt, a, s->table_dev, s->pool_dev, s->n_surf, nk, stream);
}

uint64_t rt_batch_ltab_nk(const rt_hip_batch* b, const double* beam_desc) {
    return b->beams_on ? 0 : ltab_nk(b->lt, beam_desc);
}

int rt_batch_ltab_fill(const rt_hip_batch* b, const double* beam_desc, uint64_t nk, hipStream_t stream,
                       const double** tab) {
    TraceArgs a;
    memset(&a, 0, sizeof a);
    memcpy(a.beam.v, beam_desc, sizeof a.beam.v);
    *tab = b->lt.tab_dev;
    return ltab_fill(b->lt, a, b->pool_dev, nk, stream);
}
int rt_scheme_device(const rt_hip_scheme* s) { return s->device; }
WorkBufs* rt_scheme_work(const rt_hip_scheme* s) { return &s->work; }
WorkBufs* rt_batch_work(const rt_hip_batch* b) { return &b->work; }

extern "C" int rt_hip_scheme_device_tables(const rt_hip_scheme* s, const double** table_dev, const double** pool_dev,
                                           int* n_surf, size_t* pool_len, const double** host_table) {
    if (!s) return set_error(RT_ERR_BAD_VALUE, "scheme is NULL");
    *table_dev = s->table_dev;
    *pool_dev = s->pool_dev;
    *n_surf = s->n_surf;
    *pool_len = s->pool_len;
    *host_table = s->table.data();
    return RT_OK;
}

// Spots of the alive rays per ray group; partial moments in a buffer of the
// calling thread (calls that belong to no scheme): it only grows, and a
// buffer it replaced stays allocated until the thread ends, so a graph that
// captured a call keeps valid memory.  Calls of one thread share it: they
// must run in the order of one stream.
namespace {
struct ThreadWork {
    int device = -1;
    WorkBufs w;
    ~ThreadWork() { w.release(); }
};
thread_local ThreadWork g_thread_work;

WorkBufs* thread_work(int dev) {
    if (g_thread_work.device != dev) {
        // another device: the old buffers belong to that device's context
        g_thread_work.w.release();
        g_thread_work.device = dev;
    }
    return &g_thread_work.w;
}

// moments of n rays in G groups (spot_chunk_count(n, G) rows of 5 doubles per
// group in part), then the groups' spots
int group_spots_launch(const double* X, const double* Y, const signed char* flag, uint64_t n, uint64_t G, double* part,
                       double* spots, hipStream_t st) {
    // with n == 0 the single chunk is empty and its partials are written as zeros
    const uint64_t n_chunks = spot_chunk_count(n, G);
    hipLaunchKernelGGL(rt_group_moments_kernel, dim3((unsigned)(n_chunks * spot_group_blocks(G))), dim3(kSpotThreads),
                       0, st, X, Y, flag, n, G, n_chunks, part);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    hipLaunchKernelGGL(rt_spots_rows_kernel<256>, dim3((unsigned)G), dim3(256), 0, st, (const double*)part, n_chunks,
                       (const uint64_t*)nullptr, G, spots);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    return RT_OK;
}

// partial moments of an input as the entry points' size limits count them:
// one per 8 rays of a group
uint64_t spot_partials(uint64_t n, uint64_t G) {
    const uint64_t strides = (n + G - 1) / G;
    return strides > 0 ? (strides + 7) / 8 : 1;
}
}  // namespace

extern "C" int rt_hip_group_spots(const double* X, const double* Y, const signed char* flag, size_t n,
                                  size_t n_groups, double* spots, void* stream) {
    if (!spots || n_groups == 0) return set_error(RT_ERR_BAD_VALUE, "spots NULL or no groups");
    if (n > 0 && (!X || !Y || !flag)) return set_error(RT_ERR_BAD_VALUE, "NULL ray array");
    int rc = ensure_device();
    if (rc != RT_OK) return rc;
    const uint64_t G = n_groups;
    if (spot_partials(n, G) > (1ull << 40) / G) return set_error(RT_ERR_BAD_VALUE, "too many rays or groups");
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev), RT_ERR_FAILED);
    WorkBufs* w = thread_work(dev);
    rc = w->ensure(WorkBufs::SPOT_PART, spot_chunk_count(n, G) * G * 5 * sizeof(double));
    if (rc != RT_OK) return rc;
    return group_spots_launch(X, Y, flag, n, G, w->get<double>(WorkBufs::SPOT_PART), spots, (hipStream_t)stream);
}

// ------------------------------------ group spots without allocation
//
// Partial moments of rt_hip_group_spots_noalloc live in this file-scope
// array, one copy per GPU, held until the process ends.  Host code never
// passes the array's name to a kernel (on the host it is only a stand-in):
// its device address is looked up once per device with that device current
// and kept in g_scratch_ptr.  Every call on one GPU shares the array; the
// moments kernel writes every partial it reads, so nothing has to start at
// zero, and calls that overlap on one GPU (two streams) race.
constexpr size_t kScratchDoubles = size_t(1) << 20;        // 8 MiB per GPU
__device__ __align__(256) double scratch[kScratchDoubles];

namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kScratchDevices] = {};

// the device address of `scratch` on the current device (dev)
int scratch_ptr(int dev, double** out) {
    if (dev < 0 || dev >= kScratchDevices) return set_error(RT_ERR_FAILED, "device %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            (void)hipGetLastError();
            return set_error(RT_ERR_INIT_FAILED, "hipGetSymbolAddress(scratch) on device %d: %s", dev,
                             hipGetErrorString(e));
        }
        g_scratch_ptr[dev] = (double*)p;
    }
    *out = g_scratch_ptr[dev];
    return RT_OK;
}
}  // namespace

int rt_scratch_setup(int dev) {
    double* p = nullptr;
    return scratch_ptr(dev, &p);
}

extern "C" int rt_hip_group_spots_noalloc(const double* X, const double* Y, const signed char* flag, size_t n,
                                          size_t n_groups, double* spots, void* stream) {
    if (!spots || n_groups == 0) return set_error(RT_ERR_BAD_VALUE, "spots NULL or no groups");
    if (n > 0 && (!X || !Y || !flag)) return set_error(RT_ERR_BAD_VALUE, "NULL ray array");
    const uint64_t G = n_groups;
    const uint64_t cap = kScratchDoubles / 5;                 // partial moments that fit
    const uint64_t n_part = G <= cap ? spot_partials(n, G) : 0;
    if (G > cap || n_part > cap / G)
        return set_error(RT_ERR_BAD_VALUE,
                         "%zu rays in %zu groups need %llu partial moments; the no-allocation entry point "
                         "holds %llu (use rt_hip_group_spots)",
                         n, n_groups, (unsigned long long)(G > cap ? G : n_part * G), (unsigned long long)cap);
    int rc = ensure_device();
    if (rc != RT_OK) return rc;
    int dev = 0;
    HIP_TRY(hipGetDevice(&dev), RT_ERR_FAILED);
    double* part = nullptr;
    rc = scratch_ptr(dev, &part);
    if (rc != RT_OK) return rc;
    return group_spots_launch(X, Y, flag, n, G, part, spots, (hipStream_t)stream);
}

extern "C" int rt_hip_spot_loss(const double* spots, size_t n_groups, const double* target, double weight,
                                double* seeds, double* loss, void* stream) {
    if (!spots || !seeds || !loss || n_groups == 0) return set_error(RT_ERR_BAD_VALUE, "NULL argument or no groups");
    int rc = ensure_device();
    if (rc != RT_OK) return rc;
    hipLaunchKernelGGL(rt_spot_loss_kernel, dim3(1), dim3(kLossThreads), 0, (hipStream_t)stream, spots,
                       (uint64_t)n_groups, target, weight, seeds, loss);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    return RT_OK;
}

// Spots per (instance, group) of a batch's stored rays (rt_hip_batch_trace
// with RT_TRACE_STORE): spots receives n_inst x n_groups x RT_SPOT_STRIDE.
extern "C" int rt_hip_batch_group_spots(const rt_hip_batch* b, const double* X, const double* Y,
                                        const signed char* flag, size_t n_groups, double* spots, void* stream) {
    if (!b) return set_error(RT_ERR_BAD_VALUE, "batch is NULL");
    if (!spots || n_groups == 0) return set_error(RT_ERR_BAD_VALUE, "spots NULL or no groups");
    const uint64_t total_rays = b->ray_start[b->n_inst];
    if (total_rays > 0 && (!X || !Y || !flag)) return set_error(RT_ERR_BAD_VALUE, "NULL ray array");
    int rc = ensure_device();
    if (rc != RT_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    const uint64_t G = n_groups;
    uint64_t chunks = 0;                 // the same count the device prefix forms
    for (int i = 0; i < b->n_inst; ++i) chunks += spot_chunk_count(b->ray_start[i + 1] - b->ray_start[i], G);
    // the batch's own working memory (calls on one batch are stream-ordered)
    rc = b->work.ensure(WorkBufs::SPOT_PART, chunks * G * 5 * sizeof(double));
    if (rc == RT_OK) rc = b->work.ensure(WorkBufs::SPOT_CS, ((size_t)b->n_inst + 1) * sizeof(uint64_t));
    if (rc != RT_OK) return rc;
    struct { double* part; uint64_t* cs; } buf = {b->work.get<double>(WorkBufs::SPOT_PART),
                                                  b->work.get<uint64_t>(WorkBufs::SPOT_CS)};
    hipLaunchKernelGGL(rt_batch_chunks_kernel, dim3(1), dim3(1024), 0, st, (const uint64_t*)b->ray_start_dev,
                       (uint64_t)b->n_inst, G, buf.cs);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    hipLaunchKernelGGL(rt_batch_moments_kernel, dim3((unsigned)(chunks * spot_group_blocks(G))), dim3(kSpotThreads), 0, st,
                       X, Y, flag, (const uint64_t*)b->ray_start_dev, (const uint64_t*)buf.cs, (uint64_t)b->n_inst, G,
                       chunks, buf.part);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    hipLaunchKernelGGL(rt_spots_rows_kernel<256>, dim3((unsigned)(b->n_inst * G)), dim3(256), 0, st,
                       (const double*)buf.part, chunks, (const uint64_t*)buf.cs, G, spots);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    return RT_OK;
}

// One gradient-descent step on the device tables of every instance of a batch
// for the parameters (param_surface, param_field): field -= lr[j] * grad[i][j]
// (grad: device, n_inst x n_params; lr: device, n_params).  Differentiable
// fields of the adjoint (curvature, conic constant, aspheric terms, toric cR,
// decentres, tilts, grating constant); a tilt or decentre must be non-zero on
// that surface in some instance (the generated kernels apply only the
// rotations and translations the batch had when it was created).  The host
// copy of the tables is not updated.  No allocation after the first call with
// a given parameter list, and kernels only: capturable in a hipGraph.
extern "C" int rt_hip_batch_descend(rt_hip_batch* b, const int* param_surface, const int* param_field, int n_params,
                                    const double* grad, const double* lr, void* stream) {
    if (!b) return set_error(RT_ERR_BAD_VALUE, "batch is NULL");
    if (n_params <= 0) return RT_OK;
    if (!param_surface || !param_field || !grad || !lr) return set_error(RT_ERR_BAD_VALUE, "NULL argument");
    std::vector<int> key(param_surface, param_surface + n_params);
    key.insert(key.end(), param_field, param_field + n_params);
    if (key != b->descend_key) {
        // structure flags of each surface from the signature (rotation mask, translation)
        std::vector<std::string> sig;
        size_t pos = 0;
        while (pos < b->signature.size()) {
            size_t end = b->signature.find(';', pos);
            sig.push_back(b->signature.substr(pos, end - pos));
            pos = end + 1;
        }
        std::vector<std::vector<std::pair<int, int>>> per(b->n_surf);
        for (int j = 0; j < n_params; ++j) {
            const int sf = param_surface[j], f = param_field[j];
            if (sf < 0 || sf >= b->n_surf) return set_error(RT_ERR_BAD_VALUE, "parameter %d: bad surface", j);
            const bool ok_field = f == RT_S_C || f == RT_S_K || (f >= RT_S_A && f < RT_S_A + RT_MAX_POLY) ||
                                  f == RT_S_CR || (f >= RT_S_DIST && f < RT_S_DIST + 3) ||
                                  (f >= RT_S_ANG && f < RT_S_ANG + 3) || f == RT_S_GRCONST;
            if (!ok_field) return set_error(RT_ERR_BAD_VALUE, "parameter %d: field %d cannot be stepped", j, f);
            // StatSurf<cls,type,shape,npoly,grt,ordm,ik,fnmask,rotmask,trans,ccd>
            std::vector<std::string> tp;
            std::string body = sig[sf].substr(sig[sf].find('<') + 1);
            size_t q = 0;
            while (q < body.size()) {
                size_t e = body.find_first_of(",>", q);
                tp.push_back(body.substr(q, e - q));
                q = e + 1;
                if (body[e] == '>') break;
            }
            const int rotmask = atoi(tp[8].c_str());
            const bool trans = tp[9] == "true";
            if (f >= RT_S_ANG && f < RT_S_ANG + 3 && !((rotmask >> (f - RT_S_ANG)) & 1))
                return set_error(RT_ERR_BAD_VALUE, "parameter %d: surface %d has no rotation %d in the batch", j, sf,
                                 f - RT_S_ANG);
            if (f >= RT_S_DIST && f < RT_S_DIST + 3 && !trans)
                return set_error(RT_ERR_BAD_VALUE, "parameter %d: surface %d has no translation in the batch", j, sf);
            per[sf].push_back({j, f});
        }
        std::vector<int> host(b->n_surf + 1, 0);
        for (int s = 0; s < b->n_surf; ++s) host[s + 1] = host[s] + (int)per[s].size();
        for (int s = 0; s < b->n_surf; ++s)
            for (auto& jf : per[s]) { host.push_back(jf.first); host.push_back(jf.second); }
        // a new buffer for a new list: a graph captured with the old one keeps reading it
        b->descend_key.clear();
        int rc = b->work.fresh(WorkBufs::DESCEND, host.size() * sizeof(int));
        if (rc != RT_OK) return rc;
        HIP_TRY(hipMemcpy(b->work.p[WorkBufs::DESCEND], host.data(), host.size() * sizeof(int),
                          hipMemcpyHostToDevice),
                RT_ERR_FAILED);
        b->descend_key = key;
    }
    const int* map = b->work.get<const int>(WorkBufs::DESCEND);
    const uint64_t threads = (uint64_t)b->n_inst * b->n_surf;
    hipLaunchKernelGGL(rt_batch_descend_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, b->tables_dev, (uint64_t)b->n_inst, b->n_surf,
                       map, map + b->n_surf + 1, grad, lr, n_params);
    HIP_TRY(hipGetLastError(), RT_ERR_FAILED);
    return RT_OK;
}
