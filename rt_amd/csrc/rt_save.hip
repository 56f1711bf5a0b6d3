// rt_save.hip -- the saved beam of Scheme::run on the device: the order in
// which the reference's Beam::Rearrange calls leave the rays, and the state
// of the rays lost on the way, from the loss codes of a recording trace.
//
// Scheme::run (common-lib/scheme.cpp:983-1046) keeps the good rays at the
// front of the beam arrays: after every stage that loses rays (intersection,
// surface.cpp:256-259; aperture, :316-320 and :694-697; action, :467-471 and
// :579-583) Beam::Rearrange (beam.cpp:574-598) partitions [0, N_good) with
// two pointers: the k-th lost ray from the front is swapped with the k-th
// good ray from the back while the first lies before the second.  With G the
// good count before the stage and G' after it, those pairs are exactly the
// lost rays in [0, G') in ascending order and the good rays in [G', G) in
// descending order, so one stage is a prefix count of its lost rays and one
// swap per pair, all in parallel.  The stages run in Scheme::run's order.
//
// Beam::Save (beam.cpp:636-715) writes the arrays in that order, good rays
// first.  Transform and the engine's stages touch only [0, N_good), so a lost
// ray keeps the state it was lost in, but Beam::Normalize runs over every ray
// (beam.cpp:527-571): its cosines pass through the scaled-norm formula once
// more at every later Normalize call.  rt_hip_beam_order applies them, in
// the reference's operation order with no contraction, IEEE division and
// square root, so the lost rays' cosines come out as the reference's would
// from the same state.
#include <hip/hip_runtime.h>

#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "rt_device.h"
#include "rt_host.h"

namespace {

constexpr int kTileThreads = 256;
constexpr int kPerThread = 16;
constexpr uint64_t kTile = (uint64_t)kTileThreads * kPerThread;   // positions per tile

__global__ void rt_save_zero_kernel(unsigned long long* v, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) v[i] = 0ull;
}

// Position p holds ray p before the first stage, and the counts of every loss
// code: one pass over the codes (1 byte read, 9 written a ray), V rays a lane
// (V = 4 where the codes are 4-byte aligned).  Nearly every ray has code 0, so
// those are counted in a register, the others in LDS; at most kInitBlocks
// workgroups add to the counts, which share a few lines and are served one add
// after the other.  (Two kernels, an LDS add per ray and 4,096 workgroups took
// 52 + 7 us at 2e6 rays; this takes 13.5.)
constexpr int kInitThreads = 512;
constexpr unsigned kInitBlocks = 512;

template <int V>
__global__ __launch_bounds__(kInitThreads) void rt_order_init_kernel(const unsigned char* loss, uint64_t n,
                                                                     uint64_t* perm, unsigned char* lpos,
                                                                     unsigned long long* counts) {
    __shared__ unsigned h[256];
    if (threadIdx.x < 256) h[threadIdx.x] = 0u;
    __syncthreads();
    unsigned good = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x * V;
    for (uint64_t p = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * V; p < n; p += stride) {
        if (V == 4 && p + V <= n) {
            const uint32_t c4 = *(const uint32_t*)(loss + p);
            *(uint32_t*)(lpos + p) = c4;                 // (lpos: this library's own buffer, aligned)
#pragma unroll
            for (int k = 0; k < V; ++k) {
                perm[p + k] = p + k;
                const unsigned c = (c4 >> (8 * k)) & 255u;
                if (c) atomicAdd(&h[c], 1u);
                else ++good;
            }
        } else {
            for (uint64_t q = p; q < n && q < p + V; ++q) {
                const unsigned c = loss[q];
                lpos[q] = (unsigned char)c;
                perm[q] = q;
                if (c) atomicAdd(&h[c], 1u);
                else ++good;
            }
        }
    }
    for (int m = 32; m >= 1; m >>= 1) good += __shfl_xor(good, m);
    if (__lane_id() == 0 && good) atomicAdd(&h[0], good);
    __syncthreads();
    if (threadIdx.x < 256 && h[threadIdx.x]) atomicAdd(&counts[threadIdx.x], (unsigned long long)h[threadIdx.x]);
}

// the 16 codes of a thread's positions base .. base + 15 (lpos is padded to a
// whole tile), as bit k of a mask: position base + k is below G and has `code`
__device__ __forceinline__ unsigned code_mask(const unsigned char* lpos, uint64_t base, uint64_t G,
                                              unsigned char code) {
    const uint4 v = *(const uint4*)(lpos + base);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    unsigned m = 0;
#pragma unroll
    for (int k = 0; k < kPerThread; ++k)
        m |= (base + k < G && ((w[k / 4] >> (8 * (k % 4))) & 255u) == code) ? 1u << k : 0u;
    return m;
}

// lost rays of this stage (code) per tile of [0, G)
__global__ __launch_bounds__(kTileThreads) void rt_stage_count_kernel(const unsigned char* lpos, uint64_t G,
                                                                      unsigned char code, uint64_t* tile_bad) {
    __shared__ unsigned s[kTileThreads / 64];
    const uint64_t base = (uint64_t)blockIdx.x * kTile + (uint64_t)threadIdx.x * kPerThread;
    unsigned c = __popc(code_mask(lpos, base, G, code));
    for (int m = 32; m >= 1; m >>= 1) c += __shfl_xor(c, m);
    if (__lane_id() == 0) s[threadIdx.x / 64] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned t = 0;
        for (int w = 0; w < kTileThreads / 64; ++w) t += s[w];
        tile_bad[blockIdx.x] = t;
    }
}

// exclusive prefix over the tiles (one workgroup, chunks of 1024 with a carry)
__global__ __launch_bounds__(1024) void rt_tile_scan_kernel(uint64_t* tile_bad, uint64_t n_tiles) {
    __shared__ uint64_t s[1024];
    __shared__ uint64_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (uint64_t b0 = 0; b0 < n_tiles; b0 += 1024) {
        const uint64_t b = b0 + threadIdx.x;
        const uint64_t v = b < n_tiles ? tile_bad[b] : 0;
        s[threadIdx.x] = v;
        __syncthreads();
        for (int off = 1; off < 1024; off <<= 1) {       // inclusive Hillis-Steele scan
            const uint64_t t = threadIdx.x >= (unsigned)off ? s[threadIdx.x - off] : 0;
            __syncthreads();
            s[threadIdx.x] += t;
            __syncthreads();
        }
        const uint64_t c = carry;
        if (b < n_tiles) tile_bad[b] = c + s[threadIdx.x] - v;
        __syncthreads();
        if (threadIdx.x == 1023) carry = c + s[1023];
        __syncthreads();
    }
}

// bad: this thread's mask of lost rays of the stage in tile `tile`
// (code_mask); returns the lost rays before its first position, counted from
// the start of [0, G) (tile_off: the tile's offset).  The workgroup is the
// tile; every read of the tile completes before the function returns
// (barrier).
__device__ __forceinline__ uint64_t tile_prefix(const unsigned char* lpos, uint64_t G, unsigned char code,
                                                uint64_t tile, uint64_t tile_off, unsigned& bad) {
    __shared__ unsigned s[kTileThreads / 64];
    bad = code_mask(lpos, tile * kTile + (uint64_t)threadIdx.x * kPerThread, G, code);
    const unsigned c = __popc(bad), lane = __lane_id();
    unsigned run = c;                                    // inclusive scan over the wave
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned t = __shfl_up(run, off);
        if (lane >= (unsigned)off) run += t;
    }
    if (lane == 63) s[threadIdx.x / 64] = run;
    __syncthreads();
    for (unsigned w = 0; w < threadIdx.x / 64; ++w) run += s[w];
    return tile_off + run - c;
}

// good rays of [G', G): the k-th from the back (k = 1, 2, ...) at gpos[k - 1];
// workgroup b takes tile first_tile + b
__global__ __launch_bounds__(kTileThreads) void rt_stage_tail_kernel(const unsigned char* lpos, uint64_t G,
                                                                     uint64_t Gn, uint64_t nb, unsigned char code,
                                                                     const uint64_t* tile_off, uint64_t first_tile,
                                                                     uint64_t* gpos) {
    const uint64_t tile = first_tile + blockIdx.x;
    unsigned bad;
    uint64_t pre = tile_prefix(lpos, G, code, tile, tile_off[tile], bad);
    const uint64_t base = tile * kTile + (uint64_t)threadIdx.x * kPerThread;
    for (int k = 0; k < kPerThread; ++k) {
        const uint64_t q = base + k;
        if ((bad >> k) & 1u) {
            ++pre;
            continue;
        }
        if (q < Gn || q >= G) continue;
        // lost rays after q: all of them but the `pre` before q (q is good)
        const uint64_t good_after = (G - 1 - q) - (nb - pre);
        gpos[good_after] = q;
    }
}

// lost rays of [0, G'): the k-th (k = 1, 2, ...) swaps places with gpos[k - 1]
__global__ __launch_bounds__(kTileThreads) void rt_stage_head_kernel(unsigned char* lpos, uint64_t G, uint64_t Gn,
                                                                     unsigned char code, const uint64_t* tile_off,
                                                                     const uint64_t* gpos, uint64_t* perm) {
    unsigned bad;
    uint64_t pre = tile_prefix(lpos, G, code, blockIdx.x, tile_off[blockIdx.x], bad);
    const uint64_t base = (uint64_t)blockIdx.x * kTile + (uint64_t)threadIdx.x * kPerThread;
    for (; bad; bad &= bad - 1) {
        const uint64_t p = base + (uint64_t)(__ffs((int)bad) - 1);
        if (p >= Gn) break;
        const uint64_t q = gpos[pre++];
        const uint64_t rp = perm[p], rq = perm[q];
        perm[p] = rq;
        perm[q] = rp;
        const unsigned char lq = lpos[q];
        lpos[q] = lpos[p];
        lpos[p] = lq;
    }
}

// Beam::Normalize on one ray (beam.cpp:541-569): the scaled norm, in the
// reference's operation order with no contraction
__device__ __forceinline__ void normalize_reference(double& cX, double& cY, double& cZ) {
#pragma clang fp contract(off)
    const double acX = fabs(cX), acY = fabs(cY), acZ = fabs(cZ);
    double norm;
    if (acX >= acY) {
        if (acX >= acZ) norm = acX * sqrt(1.0 + acY * acY / acX / acX + acZ * acZ / acX / acX);
        else norm = acZ * sqrt(1.0 + acX * acX / acZ / acZ + acY * acY / acZ / acZ);
    } else {
        if (acY >= acZ) norm = acY * sqrt(1.0 + acX * acX / acY / acY + acZ * acZ / acY / acY);
        else norm = acZ * sqrt(1.0 + acX * acX / acZ / acZ + acY * acY / acZ / acZ);
    }
    cX /= norm;
    cY /= norm;
    cZ /= norm;
}

struct OrderArgs {
    const double* in[7];
    double* out;
    const uint64_t* perm;
    const unsigned char* loss;
    uint64_t n;
    unsigned char renorm[256];
};

// Bound by the 7 rows read and written and the permutation (121 bytes a ray);
// the rows' loads are issued together, the renormalisation counts read from
// LDS (indexed in the argument segment they went through scratch memory, with
// the rows behind a call: 82 us at 2e6 rays, now 56).
__global__ __launch_bounds__(256) void rt_beam_order_kernel(OrderArgs a) {
    __shared__ unsigned char s_renorm[256];
    typedef const __attribute__((address_space(4))) unsigned char* cbytes;
    if (threadIdx.x < 256)
        s_renorm[threadIdx.x] = ((cbytes)__builtin_amdgcn_kernarg_segment_ptr())[__builtin_offsetof(OrderArgs, renorm) +
                                                                                 threadIdx.x];
    __syncthreads();
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < a.n; p += stride) {
        const uint64_t r = a.perm[p];
        double v[7];
#pragma unroll
        for (int k = 0; k < 7; ++k) v[k] = a.in[k][r];
        const int m = s_renorm[a.loss[r]];
        for (int j = 0; j < m; ++j) normalize_reference(v[3], v[4], v[5]);
#pragma unroll
        for (int k = 0; k < 7; ++k) a.out[(uint64_t)k * a.n + p] = v[k];
    }
}

unsigned grid_for(uint64_t n, unsigned block) {
    const uint64_t want = (n + block - 1) / block;
    const uint64_t cap = (uint64_t)rt_device_cus() * 16;
    return (unsigned)std::max<uint64_t>(1, std::min(want, cap));
}

struct SaveWork {
    int device = -1;
    WorkBufs w;
    ~SaveWork() { w.release(); }
};
thread_local SaveWork g_save_work;

}  // namespace

extern "C" int rt_hip_rearrange(const unsigned char* loss_dev, size_t n, uint64_t* perm_dev, uint64_t* counts,
                                void* stream) {
    if (n > 0 && (!loss_dev || !perm_dev)) return rt_set_error(RT_ERR_BAD_VALUE, "NULL loss or perm buffer");
    if (!counts) return rt_set_error(RT_ERR_BAD_VALUE, "counts is NULL");
    memset(counts, 0, 256 * sizeof(uint64_t));
    if (n == 0) return RT_OK;
    int rc = rt_ensure_device();
    if (rc != RT_OK) return rc;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return rt_set_error(RT_ERR_FAILED, "hipGetDevice failed");
    if (g_save_work.device != dev) {
        g_save_work.w.release();
        g_save_work.device = dev;
    }
    WorkBufs& w = g_save_work.w;
    const uint64_t n_tiles = (n + kTile - 1) / kTile;
    if ((rc = w.ensure(WorkBufs::SAVE_HIST, 256 * sizeof(unsigned long long))) != RT_OK ||
        (rc = w.ensure(WorkBufs::SAVE_LPOS, n_tiles * kTile)) != RT_OK ||
        (rc = w.ensure(WorkBufs::SAVE_TILES, n_tiles * sizeof(uint64_t))) != RT_OK ||
        (rc = w.ensure(WorkBufs::SAVE_GPOS, n * sizeof(uint64_t))) != RT_OK)
        return rc;
    hipStream_t st = (hipStream_t)stream;
    unsigned long long* hist = w.get<unsigned long long>(WorkBufs::SAVE_HIST);
    unsigned char* lpos = w.get<unsigned char>(WorkBufs::SAVE_LPOS);
    uint64_t* tiles = w.get<uint64_t>(WorkBufs::SAVE_TILES);
    uint64_t* gpos = w.get<uint64_t>(WorkBufs::SAVE_GPOS);

    hipLaunchKernelGGL(rt_save_zero_kernel, dim3(1), dim3(256), 0, st, hist, 256);
    const int V = ((uintptr_t)loss_dev & 3u) == 0 ? 4 : 1;
    const uint64_t want = (n + (uint64_t)kInitThreads * V - 1) / ((uint64_t)kInitThreads * V);
    hipLaunchKernelGGL(V == 4 ? rt_order_init_kernel<4> : rt_order_init_kernel<1>,
                       dim3((unsigned)std::min<uint64_t>(want, kInitBlocks)), dim3(kInitThreads), 0, st, loss_dev,
                       (uint64_t)n, perm_dev, lpos, hist);
    if (hipGetLastError() != hipSuccess) return rt_set_error(RT_ERR_FAILED, "rearrange launch failed");
    if (hipMemcpyAsync(counts, hist, 256 * sizeof(uint64_t), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return rt_set_error(RT_ERR_FAILED, "rearrange: reading the loss counts failed");

    // stages in Scheme::run's order: codes 1, 2, 3, ... (kLossDead rays never
    // were good and sit outside [0, G) from the start)
    uint64_t G = n - counts[rt::kLossDead];
    if (counts[rt::kLossDead]) return rt_set_error(RT_ERR_BAD_VALUE, "rays that entered dead cannot be ordered");
    for (int code = 1; code < rt::kLossDead; ++code) {
        const uint64_t nb = counts[code];
        if (nb == 0) continue;
        const uint64_t Gn = G - nb;
        const uint64_t tiles_G = (G + kTile - 1) / kTile;
        hipLaunchKernelGGL(rt_stage_count_kernel, dim3((unsigned)tiles_G), dim3(kTileThreads), 0, st,
                           (const unsigned char*)lpos, G, (unsigned char)code, tiles);
        hipLaunchKernelGGL(rt_tile_scan_kernel, dim3(1), dim3(1024), 0, st, tiles, tiles_G);
        const uint64_t t0 = Gn / kTile;
        hipLaunchKernelGGL(rt_stage_tail_kernel, dim3((unsigned)(tiles_G - t0)), dim3(kTileThreads), 0, st,
                           (const unsigned char*)lpos, G, Gn, nb, (unsigned char)code, (const uint64_t*)tiles, t0,
                           gpos);
        const uint64_t tiles_Gn = (Gn + kTile - 1) / kTile;
        if (tiles_Gn)
            hipLaunchKernelGGL(rt_stage_head_kernel, dim3((unsigned)tiles_Gn), dim3(kTileThreads), 0, st, lpos, G, Gn,
                               (unsigned char)code, (const uint64_t*)tiles, (const uint64_t*)gpos, perm_dev);
        if (hipGetLastError() != hipSuccess) return rt_set_error(RT_ERR_FAILED, "rearrange stage launch failed");
        G = Gn;
    }
    return RT_OK;
}

extern "C" int rt_hip_beam_order(size_t n, const uint64_t* perm_dev, const unsigned char* loss_dev,
                                 const unsigned char* renorm, const double* X, const double* Y, const double* Z,
                                 const double* cX, const double* cY, const double* cZ, const double* lambda,
                                 double* out_dev, void* stream) {
    if (n == 0) return RT_OK;
    if (!perm_dev || !loss_dev || !renorm || !X || !Y || !Z || !cX || !cY || !cZ || !lambda || !out_dev)
        return rt_set_error(RT_ERR_BAD_VALUE, "NULL argument");
    int rc = rt_ensure_device();
    if (rc != RT_OK) return rc;
    OrderArgs a;
    memset(&a, 0, sizeof a);
    a.in[0] = X; a.in[1] = Y; a.in[2] = Z; a.in[3] = cX; a.in[4] = cY; a.in[5] = cZ; a.in[6] = lambda;
    a.out = out_dev;
    a.perm = perm_dev;
    a.loss = loss_dev;
    a.n = n;
    memcpy(a.renorm, renorm, 256);
    hipLaunchKernelGGL(rt_beam_order_kernel, dim3(grid_for(n, 256)), dim3(256), 0, (hipStream_t)stream, a);
    if (hipGetLastError() != hipSuccess) return rt_set_error(RT_ERR_FAILED, "beam order launch failed");
    return RT_OK;
}
