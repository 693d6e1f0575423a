// traverse.hip — raw closest-hit / any-hit traversal kernels for gfx950.
// These are the kernels behind wl_trace_closest and wl_trace_any, which stand
// in for optixTrace (PathTracing.cu:72-75, :92-102).
//
// One ray per lane, 256 lanes per workgroup, an LDS stack per lane, and a
// persistent grid whose lanes refill from their wave's range of rays
// (traverse_persistent.h).  The LDS stack is sized per launch: a BVH at most
// 16 levels deep needs at most 15 entries, so its kernels reserve 16
// (16 KiB per workgroup) instead of 32.  The instrumented closest-hit kernel
// (node / triangle counts) keeps one ray per lane without refill.
#include "traverse_persistent.h"
#include "wl_internal.h"

namespace wl
{

constexpr int kTraceBlock = 256;
// The first nodes of the BVH (laid out breadth first: the root, its group of
// 8 and their groups, levels 0-2 of a full tree) are copied to LDS per
// workgroup; every ray starts there, so about half of a ray's node visits
// read LDS instead of the L1/L2 path.  9,344 bytes beside the 16-entry stack
// keep 6 workgroups (24 waves) per CU; the 32-entry-stack kernels for deep
// BVHs have no room for it.
constexpr uint32_t kTopNodes = 73;

// Chunks of this many rays (traverse_persistent.h), taken at run time from one
// counter per XCD, each counter in a cache line of its own and each chunk asked
// for one ahead.  2^23 rays, closest / any hit: 64: 696 / 534 us, 96: 688 / 522,
// 128: 691 / 521, 256: 713 / 523, 512: 730 / 524 (727 / 603 us with 256 and the
// eight counters in one line).  A launch with fewer than 128 rays per resident
// wave takes 64, which fill one wave's lanes: 100,003 rays 112 -> 65 us (16: 94,
// 32: 79, 128: 81 before the last rays' both-steps rule of trav_persistent).
constexpr uint32_t kTraceChunk = 128;

// The chunk counters' values at launch, one per XCD, and the launch's chunk.
struct TraceSched
{
    uint32_t base[8];
    uint32_t chunk;
};

template <int STACK>
constexpr uint32_t top_nodes() { return STACK == 16 ? kTopNodes : 0u; }

// Copies nodes [0, ntop) to LDS (all threads of the workgroup, then a barrier).
__device__ __forceinline__ void load_top(uint4 *top, const WlBvh8Node *__restrict__ nodes,
                                         uint32_t ntop)
{
    const uint4 *src = reinterpret_cast<const uint4 *>(nodes);
    for (uint32_t i = threadIdx.x; i < 8u * ntop; i += kTraceBlock)
        top[i] = src[i];
    __syncthreads();
}

// ntop: nodes copied to LDS, min(node count, top_nodes<STACK>()); sched /
// base: the launching stream's chunk counters and their values at launch.
// The grid is a multiple of 8.
template <int STACK, bool WIDE>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(6, 8)))
void k_trace_closest_p(
    const WlBvh8Node *__restrict__ nodes, const WlTriRecord *__restrict__ tris,
    const wl_ray *__restrict__ rays, uint32_t n, wl_hit *__restrict__ hits, uint32_t ntop,
    uint32_t *__restrict__ sched, TraceSched base)
{
    __shared__ uint32_t stack[STACK * kTraceBlock];
    __shared__ uint4 top[8 * (top_nodes<STACK>() ? top_nodes<STACK>() : 1)];
    if (top_nodes<STACK>())
        load_top(top, nodes, ntop);
    const EighthChunks range(n, blockIdx.x % 8u, base.chunk);
    trav_persistent<kClosest, kTraceBlock, WIDE, top_nodes<STACK>() != 0>(
        nodes, tris, stack,
        XcdChunks<kTraceBlock, decltype(range)>(range, sched + kSchedStride * (blockIdx.x % 8u),
                                                base.base[blockIdx.x % 8u]),
        [&](uint32_t i, TravRay &r, uint32_t &) { load_ray_nt(rays, i, r); },
        [&](uint32_t i, const TravRay &, const TravResult &h) { store_hit_nt(hits, i, h); },
        reinterpret_cast<const WlBvh8Node *>(top), top_nodes<STACK>() ? ntop : 0u);
}

template <int STACK, bool WIDE>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(7, 8)))
void k_trace_any_p(const WlBvh8Node *__restrict__ nodes, const WlTriRecord *__restrict__ tris,
                   const wl_ray *__restrict__ rays, uint32_t n, uint32_t *__restrict__ bits,
                   uint32_t ntop, uint32_t *__restrict__ sched, TraceSched base)
{
    __shared__ uint32_t stack[STACK * kTraceBlock];
    __shared__ uint4 top[8 * (top_nodes<STACK>() ? top_nodes<STACK>() : 1)];
    if (top_nodes<STACK>())
        load_top(top, nodes, ntop);
    const EighthChunks range(n, blockIdx.x % 8u, base.chunk);
    trav_persistent<kAny, kTraceBlock, WIDE, top_nodes<STACK>() != 0>(
        nodes, tris, stack,
        XcdChunks<kTraceBlock, decltype(range)>(range, sched + kSchedStride * (blockIdx.x % 8u),
                                                base.base[blockIdx.x % 8u]),
        [&](uint32_t i, TravRay &r, uint32_t &) { load_ray_nt(rays, i, r); },
        [&](uint32_t i, const TravRay &, const TravResult &h) {
            if (h.prim != WL_INVALID)
                atomicOr(&bits[i >> 5], 1u << (i & 31u));
        },
        reinterpret_cast<const WlBvh8Node *>(top), top_nodes<STACK>() ? ntop : 0u);
}

// Instrumented closest hit: one ray per lane, per-ray node/triangle counts.
template <int STACK>
__global__ __launch_bounds__(kTraceBlock) void k_trace_closest_counted(
    const WlBvh8Node *__restrict__ nodes, const WlTriRecord *__restrict__ tris,
    const wl_ray *__restrict__ rays, uint32_t n, wl_hit *__restrict__ hits,
    uint32_t *__restrict__ counts)
{
    __shared__ uint32_t stack[STACK * kTraceBlock];
    const uint32_t rid = blockIdx.x * kTraceBlock + threadIdx.x;
    const bool active = rid < n;
    TravRay r;
    if (active)
        load_ray_nt(rays, rid, r);
    else
        trav_setup(r, 0, 0, 0, 1, 0, 0, 0, 0);
    uint32_t nn = 0, nt = 0;
    TravResult h = trav_run<kClosest, true, kTraceBlock>(nodes, tris, r, active, stack,
                                                     threadIdx.x, nn, nt);
    if (active)
    {
        reinterpret_cast<float4 *>(hits)[rid] =
            make_float4(h.t, __uint_as_float(h.prim), h.b1, h.b2);
        counts[2 * (size_t)rid] = nn;
        counts[2 * (size_t)rid + 1] = nt;
    }
}

// Zeroes the any-hit occlusion words (the kernel ORs bits in).
__global__ void k_zero_words(uint32_t *words, uint32_t nwords)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t k = i; k < nwords; k += gridDim.x * blockDim.x)
        words[k] = 0;
}

// Persistent grid: the workgroups that fit the GPU at once (the launch then
// takes at most one workgroup per 256 rays).
template <class K>
static uint32_t persistent_grid(K kernel, int num_cus)
{
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kTraceBlock, 0) !=
            hipSuccess ||
        per_cu < 1)
        per_cu = 4;
    return (uint32_t)(per_cu * std::max(1, num_cus));
}

// Rays per chunk of a launch of n rays on a GPU that holds `grid_cache`
// workgroups at once.
static uint32_t trace_chunk(uint32_t n, uint32_t grid_cache)
{
    const uint32_t waves = grid_cache * (kTraceBlock / 64);
    return n / kTraceChunk < waves ? 64u : kTraceChunk;
}

// The counters' values for a launch over n rays, advanced past it.
static TraceSched take_bases(wl_context_s::SchedBlock *sb, uint32_t n, uint32_t chunk)
{
    TraceSched t;
    t.chunk = chunk;
    for (uint32_t x = 0; x < 8; ++x)
    {
        t.base[x] = sb->base[x];
        sb->base[x] += EighthChunks(n, x, t.chunk).count();
    }
    return t;
}

// The persistent grid for n rays in chunks of `chunk`, rounded up to a multiple
// of 8 so that each XCD's eighth of the rays has workgroups.
static uint32_t xcd_grid(uint32_t grid_cache, uint32_t n, uint32_t chunk)
{
    const uint32_t per_block = chunk * (kTraceBlock / 64);
    const uint32_t g = (uint32_t)std::min<uint64_t>(
        grid_cache, ((uint64_t)n + per_block - 1) / per_block);
    return (g + 7u) & ~7u;
}

template <class V>
static hipError_t closest_impl(const wl_accel_s *a, const wl_ray *rays, uint32_t n,
                               wl_hit *hits, hipStream_t s)
{
    static uint32_t grid_cache = 0; // depends only on the kernel and the device
    static int cus_cache = -1;
    if (cus_cache != a->ctx->num_cus)
    {
        grid_cache = persistent_grid(k_trace_closest_p<V::STACK, V::WIDE>, a->ctx->num_cus);
        cus_cache = a->ctx->num_cus;
    }
    const uint32_t chunk = trace_chunk(n, grid_cache);
    const uint32_t grid = xcd_grid(grid_cache, n, chunk);
    std::lock_guard<std::mutex> lock(a->ctx->sched_mu);
    wl_context_s::SchedBlock *sb = nullptr;
    const hipError_t e = sched_block(a->ctx, s, &sb);
    if (e != hipSuccess)
        return e;
    const TraceSched base = take_bases(sb, n, chunk);
    hipLaunchKernelGGL((k_trace_closest_p<V::STACK, V::WIDE>), dim3(grid), dim3(kTraceBlock), 0, s,
                       a->d_nodes, a->d_tris, rays, n, hits,
                       std::min<uint32_t>(a->num_nodes, top_nodes<V::STACK>()), sb->dev, base);
    return hipGetLastError();
}

template <class V>
static hipError_t any_impl(const wl_accel_s *a, const wl_ray *rays, uint32_t n,
                           uint32_t *bits, hipStream_t s)
{
    static uint32_t grid_cache = 0;
    static int cus_cache = -1;
    if (cus_cache != a->ctx->num_cus)
    {
        grid_cache = persistent_grid(k_trace_any_p<V::STACK, V::WIDE>, a->ctx->num_cus);
        cus_cache = a->ctx->num_cus;
    }
    const uint32_t chunk = trace_chunk(n, grid_cache);
    const uint32_t grid = xcd_grid(grid_cache, n, chunk);
    std::lock_guard<std::mutex> lock(a->ctx->sched_mu);
    wl_context_s::SchedBlock *sb = nullptr;
    const hipError_t e = sched_block(a->ctx, s, &sb);
    if (e != hipSuccess)
        return e;
    const TraceSched base = take_bases(sb, n, chunk);
    const uint32_t words = (n + 31) / 32;
    hipLaunchKernelGGL(k_zero_words, dim3(std::min<uint32_t>((words + 255) / 256, 4096)),
                       dim3(256), 0, s, bits, words);
    hipLaunchKernelGGL((k_trace_any_p<V::STACK, V::WIDE>), dim3(grid), dim3(kTraceBlock), 0, s, a->d_nodes,
                       a->d_tris, rays, n, bits,
                       std::min<uint32_t>(a->num_nodes, top_nodes<V::STACK>()), sb->dev, base);
    return hipGetLastError();
}

// f(first, rays) for every launch of a trace of n rays.
template <class F>
static hipError_t for_launches(uint32_t n, F f)
{
    hipError_t e = hipSuccess;
    for (uint32_t first = 0; e == hipSuccess && first < n;)
    {
        const uint32_t m = launch_rays(n - first);
        e = f(first, m);
        first += m;
    }
    return e;
}

hipError_t launch_trace_closest(const wl_accel_s *a, const wl_ray *rays,
                                uint32_t n, wl_hit *hits, uint32_t *counts,
                                hipStream_t s)
{
    if (n == 0)
        return hipSuccess;
    if (counts)
    {
        dim3 grid(n / kTraceBlock + (n % kTraceBlock != 0)), block(kTraceBlock);
        if (a->trav_variant == WL_TRAV_DEEP)
            hipLaunchKernelGGL(k_trace_closest_counted<WL_BVH8_STACK_DEPTH>, grid, block, 0, s,
                               a->d_nodes, a->d_tris, rays, n, hits, counts);
        else
            hipLaunchKernelGGL(k_trace_closest_counted<WL_BVH8_SHALLOW_DEPTH>, grid, block, 0, s,
                               a->d_nodes, a->d_tris, rays, n, hits, counts);
        return hipGetLastError();
    }
    return with_variant(a->trav_variant, [&](auto v) {
        return for_launches(n, [&](uint32_t first, uint32_t m) {
            return closest_impl<decltype(v)>(a, rays + first, m, hits + first, s);
        });
    });
}

hipError_t launch_trace_any(const wl_accel_s *a, const wl_ray *rays,
                            uint32_t n, uint32_t *bits, hipStream_t s)
{
    if (n == 0)
        return hipSuccess;
    return with_variant(a->trav_variant, [&](auto v) {
        return for_launches(n, [&](uint32_t first, uint32_t m) {
            return any_impl<decltype(v)>(a, rays + first, m, bits + first / 32, s);
        });
    });
}

} // namespace wl
