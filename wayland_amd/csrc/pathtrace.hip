// pathtrace.hip — wavefront path tracer for gfx950.
//
// Restates the per-pixel megakernel of the reference (raygen loop
// PathTracing.cu:40-139, __closesthit__radiance :181-289, __miss__radiance
// :163-171, NEE :81-128, RR :130-138) as queue kernels:
//
//   first trace -> [shade -> trace] x max_depth -> accumulate
//
//   trace      BVH8 traversal: closest hits of the next bounce's rays and, in
//              the same launch, any hits of this bounce's shadow rays, whose
//              precomputed NEE contribution is added where unoccluded.  The
//              first one of a single-scene batch traces path i's camera
//              ray (TEA seed (pixel, frame), pinhole ray) computed in place,
//              and the first shade pass recomputes that vertex's state and
//              starts the path's radiance: nothing is written per path
//              before the first traversal.  Multi-request batches keep a
//              raygen pass (k_raygen_multi).
//   shade      miss / emitter hit with MIS / depth cap / Disney BSDF
//              sample-pdf-eval / NEE light sample + BSDF eval / RR, in the
//              reference's RNG draw order; appends the continuing paths and
//              the shadow rays to compacted queues (wave64 ballot + mbcnt
//              prefix, one atomic per workgroup).
//   finish     batches that are small and alone: all bounces after the second
//              in one kernel, every workgroup looping over a slice of the queue
//              (k_finish).
//   accumulate compensated (Kahan) FP32 film: sum + compensation per pixel.
//
// Radiance contributions reach a path in the reference's order (one per
// bounce at most), so per-sample radiance matches a serial evaluation.
// Every kernel loops over a device-side queue count with a fixed grid, so the
// host enqueues a whole batch without synchronising.
//
// The queues are split into eight segments, one per XCD (workgroups with
// blockIdx % 8 == x run on XCD x): a workgroup appends to its XCD's segment
// and the next kernel's workgroups on that XCD read it, so the append counter
// and the entries stay in one L2.  The first queue is the identity over the
// batch's paths (entry i is path i, blocks of kPtBlock dealt to the XCDs in
// turn) and is never written.
#include "guide_device.h"
#include "shading_device.h"
#include "traverse_persistent.h"
#include "serve_plan.h"
#include "wl_pt.h"

namespace wl
{

// A pointer to device memory that was itself loaded from memory (a request's
// scene): without this the compiler reads through it with flat instructions,
// which wait on the LDS counter too.
template <class T>
__device__ __forceinline__ const T *global_ptr(const T *p)
{
    return (const T *)(const __attribute__((address_space(1))) T *)(uintptr_t)p;
}

// b if parity, else a.  Written on the address bits: as a select between two
// members of PtBuffers the compiler indexes a copy of them in scratch memory.
template <class T>
__device__ __forceinline__ T *pick(int parity, T *a, T *b)
{
    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
    return (T *)(__attribute__((address_space(1))) T *)(x ^ ((x ^ y) & (0 - (uintptr_t)parity)));
}

// ---- queues -------------------------------------------------------------------
// XCD x's queue lengths of one parity: low word the ray queue's segment, high
// word the shadow queue's.
__device__ __forceinline__ unsigned long long *queue_len(const PtBuffers &B, uint32_t xcd,
                                                         int parity)
{
    return reinterpret_cast<unsigned long long *>(B.counters +
                                                  kPtCounterStride * (4 * xcd + (uint32_t)parity));
}
// XCD x's chunk counter of the traversal (zero when a trace kernel starts).
__device__ __forceinline__ uint32_t *queue_chunks(const PtBuffers &B, uint32_t xcd)
{
    return B.counters + kPtCounterStride * (4 * xcd + 2);
}

// The entries of the ray queue that this XCD's workgroups take.
__device__ __forceinline__ QueueWalk queue_walk(const PtBuffers &B, int parity, bool first)
{
    const uint32_t x = blockIdx.x % 8u;
    if (first)
        return dealt_walk<kPtBlock>(B.counters[kPtFlatCount], x);
    const uint32_t lo = x * B.segcap;
    return QueueWalk{ lo, kPtBlock, lo + (uint32_t)*queue_len(B, x, parity) };
}

// Workgroup-level append to the XCD's segments of two queues.  Every wave of
// the workgroup calls this in the same loop pass.  Per wave a ballot and
// mbcnt prefix; per workgroup one 64-bit atomic for both queues, issued by one
// thread.  The LDS slots alternate between passes (pass parity), so two
// barriers per pass suffice.
struct BlockAppendLds
{
    uint32_t cnt[2][2][kPtBlock / 64]; // [pass parity][queue][wave]
    uint32_t base[2][2];               // [pass parity][queue]
};

__device__ __forceinline__ void block_append2(BlockAppendLds &L, uint32_t pass,
                                              unsigned long long *len, bool p0, bool p1,
                                              uint32_t &slot0, uint32_t &slot1)
{
    const uint32_t par = pass & 1u;
    const uint32_t wave = threadIdx.x / 64u, lane = __lane_id();
    const uint64_t m0 = __ballot(p0), m1 = __ballot(p1);
    if (lane == 0)
    {
        L.cnt[par][0][wave] = (uint32_t)__popcll(m0);
        L.cnt[par][1][wave] = (uint32_t)__popcll(m1);
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        uint32_t t0 = 0, t1 = 0;
        for (uint32_t w = 0; w < kPtBlock / 64; ++w)
        {
            t0 += L.cnt[par][0][w];
            t1 += L.cnt[par][1][w];
        }
        const unsigned long long add = (unsigned long long)t1 << 32 | t0;
        const unsigned long long old = add ? atomicAdd(len, add) : 0ull;
        L.base[par][0] = (uint32_t)old;
        L.base[par][1] = (uint32_t)(old >> 32);
    }
    __syncthreads();
    uint32_t o0 = L.base[par][0], o1 = L.base[par][1];
    for (uint32_t w = 0; w < wave; ++w)
    {
        o0 += L.cnt[par][0][w];
        o1 += L.cnt[par][1][w];
    }
    slot0 = o0 + lane_prefix(m0);
    slot1 = o1 + lane_prefix(m1);
}

__device__ __forceinline__ float4 f4(V3 v, float w) { return make_float4(v.x, v.y, v.z, w); }
__device__ __forceinline__ V3 v3of(float4 a) { return mk(a.x, a.y, a.z); }

// ---- camera rays ----------------------------------------------------------
// Camera ray of path p of a batch: its pixel and sample, the seed after
// PinholeGenerateRay's two draws (Camera.h:28-35: u, then v), the direction.
__device__ __forceinline__ void camera_ray(const PtParams &P, uint32_t p, V3 &o, V3 &d,
                                           uint32_t &seed)
{
    const uint32_t pixel = P.pix0 + p % P.npix;
    const uint32_t s = p / P.npix;
    const uint32_t x = pixel % P.width, y = pixel / P.width;
    seed = tea4(pixel, P.frame0 + s);
    const float u = 2.f * ((float)(int)x + rnd(seed)) / (float)(int)P.width - 1.f;
    const float v = 2.f * ((float)(int)y + rnd(seed)) / (float)(int)P.height - 1.f;
    d = normalize(ld3(P.cam.lookat) + ld3(P.cam.right) * u + ld3(P.cam.up) * v);
    o = ld3(P.cam.pos);
}

// Clears the queue lengths and chunk counters and sets the first queue's length.
__device__ __forceinline__ void start_counters(const PtBuffers &B, uint32_t npaths)
{
    for (uint32_t i = threadIdx.x; i < kPtCounters; i += blockDim.x)
        B.counters[i] = i == kPtFlatCount ? npaths : 0u;
}

// Start of a single-scene batch: the queue counters and the material bins.
// No per-path state is written: the first trace computes each
// path's camera ray with camera_ray, and the first shade pass recomputes the
// first vertex's state (origin, direction and seed, throughput 1, depth 0,
// lastTraceTerm 1, lastPdf 1) and writes the path's radiance (and, when
// training a guide, its record accumulator), so a path costs no ray, queue
// or radiance write and read before its first traversal.
__global__ void k_batch_start(PtParams P, PtBuffers B)
{
    start_counters(B, P.npix * P.nsamples);
    for (uint32_t b = threadIdx.x; b < P.sort_bins; b += blockDim.x)
        B.sort_bins[b] = 0;
}

// ---- top BVH levels in LDS ---------------------------------------------------
// The single-scene traversal kernels with the 16-entry stack copy the first
// 73 nodes (levels 0-2 of the breadth-first node layout: root, its group and
// their groups) to LDS; every ray starts there.  9,344 bytes beside the
// stack keep 6 workgroups per CU.  Multi-request launches start rays at other
// roots of the node arena and keep the plain loads.
constexpr uint32_t kPtTopNodes = 73;

template <int STACK, bool MULTI>
constexpr uint32_t pt_top_nodes() { return (STACK == 16 && !MULTI) ? kPtTopNodes : 0u; }

template <int STACK, bool MULTI>
__device__ __forceinline__ uint32_t pt_load_top(uint4 *top, const PtScene &S)
{
    if (!pt_top_nodes<STACK, MULTI>())
        return 0u;
    const uint32_t ntop = min(S.num_nodes, pt_top_nodes<STACK, MULTI>());
    const uint4 *src = reinterpret_cast<const uint4 *>(S.nodes);
    for (uint32_t i = threadIdx.x; i < 8u * ntop; i += kPtBlock)
        top[i] = src[i];
    __syncthreads();
    return ntop;
}

// ---- trace: closest hits of the ray queue, any hits of the shadow queue -----
// Rays per chunk (traverse_persistent.h): 64 fill one wave's lanes, more share
// the counter's latency once every wave has plenty.
__device__ __forceinline__ uint32_t queue_chunk(uint32_t n_xcd)
{
    const uint32_t wavesx = (gridDim.x / 8u) * (kPtBlock / 64);
    return n_xcd / 128u < wavesx ? 64u : 128u;
}

__device__ __forceinline__ DealtChunks<kPtBlock> first_chunks(uint32_t n)
{
    return DealtChunks<kPtBlock>(n, blockIdx.x % 8u, queue_chunk(n / 8u));
}

// The first bounce of a single-scene batch: queue entry i is path i, and its
// camera ray is computed here (the same camera_ray as the shade pass uses),
// not read from a ray queue: nothing is written before the first traversal.
template <int STACK, bool WIDE>
__global__ __launch_bounds__(kPtBlock) __attribute__((amdgpu_waves_per_eu(5)))
void k_trace_first(PtParams P, PtScene S, PtBuffers B)
{
    __shared__ uint32_t stack[STACK * kPtBlock];
    __shared__ uint4 top[8 * (pt_top_nodes<STACK, false>() ? pt_top_nodes<STACK, false>() : 1)];
    const uint32_t ntop = pt_load_top<STACK, false>(top, S);
    const uint32_t count = P.npix * P.nsamples;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        B.stats[0] += count;
    const auto range = first_chunks(count);
    trav_persistent<kClosest, kPtBlock, WIDE, pt_top_nodes<STACK, false>() != 0>(
        S.nodes, S.tris, stack,
        XcdChunks<kPtBlock, decltype(range)>(range, queue_chunks(B, blockIdx.x % 8u), 0u),
        [&](uint32_t i, TravRay &r, uint32_t &) {
            V3 o, d;
            uint32_t seed;
            camera_ray(P, i, o, d, seed);
            trav_setup(r, o.x, o.y, o.z, d.x, d.y, d.z, P.epsilon, 1e30f);
        },
        [&](uint32_t i, const TravRay &, const TravResult &h) { store_hit_nt(B.hits, i, h); },
        reinterpret_cast<const WlBvh8Node *>(top), ntop);
}

// Ray i of a queue: the shadow queue or the ray queue of the given parity.
template <bool MULTI>
__device__ __forceinline__ void queue_fetch(const PtBuffers &B, int parity,
                                            const PtReq *__restrict__ reqs, float eps, bool shadow,
                                            uint32_t i, TravRay &r, uint32_t &root)
{
    // the ray queues carry the path's lastPdf and seed in the rays' w words
    // (the shade pass reads its state back from the ray): every extension ray
    // is traced on [epsilon, 1e30], epsilon the batch's or the ray's request's
    const wl_ray *rays = pick(parity, B.rays0, B.rays1);
    const f4v *rp = reinterpret_cast<const f4v *>((shadow ? B.srays : rays) + i);
    const f4v a = __builtin_nontemporal_load(rp), b = __builtin_nontemporal_load(rp + 1);
    float tmin = a.w, tmax = b.w;
    if (!shadow)
    {
        tmin = eps;
        tmax = 1e30f;
    }
    if constexpr (MULTI) // the node and triangle arrays are the arena of the requests' BVHs
    {
        if (shadow)
            root = B.sreq[i];
        else
        {
            const PtReq &rq = reqs[pick(parity, B.qreq0, B.qreq1)[i]];
            root = rq.root;
            tmin = rq.P.epsilon;
        }
    }
    trav_setup(r, a.x, a.y, a.z, b.x, b.y, b.z, tmin, tmax);
    r.code |= shadow ? kAnyRay : 0u;
}

// Its result: the hit of a path's ray, or the NEE contribution of an unoccluded
// shadow ray (one per path) added to its path's radiance.
__device__ __forceinline__ void queue_emit(const PtBuffers &B, uint32_t i, const TravRay &r,
                                           const TravResult &h)
{
    if (!(r.code & kAnyRay))
    {
        store_hit_nt(B.hits, i, h);
        return;
    }
    if (h.prim != WL_INVALID)
        return;
    const uint32_t path = B.spath[i];
    const float4 c = B.scontrib[i];
    float4 rr = B.rad[path];
    rr.x = rr.x + c.x;
    rr.y = rr.y + c.y;
    rr.z = rr.z + c.z;
    B.rad[path] = rr;
    if (c.w != 0.0f) // the path records guide training radiance
    {
        float4 ga = B.gacc[path];
        ga.x += c.x;
        ga.y += c.y;
        ga.z += c.z;
        B.gacc[path] = ga;
    }
}

// The two queues of a bounce are independent (a shadow ray adds to its path's
// radiance, which the closest hits do not touch), so one launch traces both:
// each XCD's chunks are those of its ray segment, then those of its shadow
// segment.  The shadow rays fill the waves that the last closest hits leave
// idle, and a bounce costs one launch less.  The chunks handed out at run time
// replace equal ranges per wave, which waited for the most expensive one (the
// caustic's shadow kernel took 87 us on average for what its closest hits did
// in 64).  With the per-XCD queues: 1024^2 caustic pass 3.01 -> 2.05 ms, two
// 1024^2 Cornell frames of 25 bounces 3.33 -> 2.53 ms, 517 x 389 x 3 textured
// 1.35 -> 0.87 ms, 1080p x 64 spp 40.2 -> 36.0 ms, 64 serving requests 393 (at
// equal ranges before any of this) -> 309 ms.
// first: the multi-request raygen's queue (all rays, no shadow rays).
template <int STACK, bool WIDE, bool MULTI>
__global__ __launch_bounds__(kPtBlock) __attribute__((amdgpu_waves_per_eu(STACK == 16 ? 6 : 5)))
void k_trace(PtScene S, PtBuffers B, int parity, const PtReq *__restrict__ reqs, float eps,
             int first)
{
    __shared__ uint32_t stack[STACK * kPtBlock];
    __shared__ uint4 top[8 * (pt_top_nodes<STACK, MULTI>() ? pt_top_nodes<STACK, MULTI>() : 1)];
    const uint32_t ntop = pt_load_top<STACK, MULTI>(top, S);
    const uint32_t x = blockIdx.x % 8u;
    const unsigned long long len = *queue_len(B, x, parity);
    const uint32_t flat = first ? B.counters[kPtFlatCount] : 0u;
    const uint32_t nrays = (uint32_t)len, nshadow = (uint32_t)(len >> 32);
    if (blockIdx.x < 8u && threadIdx.x == 0)
    {
        *queue_len(B, x, parity ^ 1) = 0ull; // the next shade pass appends there
        const unsigned long long n0 = first ? (x == 0 ? flat : 0u) : nrays;
        if (n0)
            atomicAdd(&B.stats[0], n0); // extension rays
        if (nshadow)
            atomicAdd(&B.stats[1], (unsigned long long)nshadow);
    }
    const auto flat_range = first_chunks(flat);
    const SegmentChunks seg_range(x * B.segcap, nrays, nshadow, queue_chunk(nrays + nshadow));
    bool shadow = false; // the kind of the wave's current chunk
    auto range = [&](uint32_t c, uint32_t &next, uint32_t &end) {
        if (first)
            flat_range(c, next, end);
        else
            seg_range(c, next, end, shadow);
    };
    trav_persistent<kMixed, kPtBlock, WIDE, pt_top_nodes<STACK, MULTI>() != 0>(
        S.nodes, S.tris, stack, XcdChunks<kPtBlock, decltype(range)>(range, queue_chunks(B, x), 0u),
        [&](uint32_t i, TravRay &r, uint32_t &root) {
            queue_fetch<MULTI>(B, parity, reqs, eps, shadow, i, r, root);
        },
        [&](uint32_t i, const TravRay &r, const TravResult &h) { queue_emit(B, i, r, h); },
        reinterpret_cast<const WlBvh8Node *>(top), ntop);
}

// ---- material sort of the shade queue ------------------------------------------
// Counting sort of the queue entries by the mesh (= material slot) they hit;
// misses take the last bin.  Per block: an LDS histogram, one global atomic per
// bin; the scatter reserves each block's range per bin the same way, so the
// global atomics per bounce are (blocks x bins), not one per entry.
constexpr uint32_t kSortMaxBins = 1024;

__device__ __forceinline__ uint32_t sort_key(const PtScene &S, uint32_t prim, uint32_t nbins)
{
    if (prim == WL_INVALID)
        return nbins - 1;
    const float4 *sr = reinterpret_cast<const float4 *>(S.prims) + 3 * (size_t)prim;
    return min(__float_as_uint(sr[2].y), nbins - 2);
}

__global__ __launch_bounds__(kPtBlock) void k_sort_count(PtParams P, PtScene S, PtBuffers B,
                                                         int parity, int first)
{
    __shared__ uint32_t hist[kSortMaxBins];
    const uint32_t nb = P.sort_bins;
    for (uint32_t b = threadIdx.x; b < nb; b += kPtBlock)
        hist[b] = 0;
    __syncthreads();
    const QueueWalk q = queue_walk(B, parity, first != 0);
    for (uint32_t k = blockIdx.x / 8u; q.at(k) < q.limit; k += gridDim.x / 8u)
    {
        const uint32_t i = q.at(k) + threadIdx.x;
        if (i >= q.limit)
            break;
        const uint32_t key =
            sort_key(S, __float_as_uint(reinterpret_cast<const float4 *>(B.hits)[i].y), nb);
        B.sort_keys[i] = key;
        atomicAdd(&hist[key], 1u);
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < nb; b += kPtBlock)
        if (hist[b])
            atomicAdd(&B.sort_bins[b], hist[b]);
}

// One block: bin counts -> running bin offsets and their total; clears the counts.
__global__ void k_sort_scan(PtParams P, PtBuffers B)
{
    __shared__ uint32_t part[kPtBlock];
    const uint32_t nb = P.sort_bins;
    const uint32_t per = (nb + kPtBlock - 1) / kPtBlock;
    const uint32_t b0 = threadIdx.x * per, b1 = min(nb, b0 + per);
    uint32_t s = 0;
    for (uint32_t b = b0; b < b1; ++b)
        s += B.sort_bins[b];
    part[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        uint32_t run = 0;
        for (int t = 0; t < kPtBlock; ++t)
        {
            const uint32_t v = part[t];
            part[t] = run;
            run += v;
        }
        B.counters[kPtSortTotal] = run;
    }
    __syncthreads();
    uint32_t run = part[threadIdx.x];
    for (uint32_t b = b0; b < b1; ++b)
    {
        const uint32_t c = B.sort_bins[b];
        B.sort_bins[kSortMaxBins + b] = run;
        B.sort_bins[b] = 0;
        run += c;
    }
}

__global__ __launch_bounds__(kPtBlock) void k_sort_scatter(PtParams P, PtBuffers B, int parity,
                                                           int first)
{
    __shared__ uint32_t hist[kSortMaxBins];
    __shared__ uint32_t base[kSortMaxBins];
    const uint32_t nb = P.sort_bins;
    const QueueWalk q = queue_walk(B, parity, first != 0);
    for (uint32_t k = blockIdx.x / 8u; q.at(k) < q.limit; k += gridDim.x / 8u)
    {
        for (uint32_t b = threadIdx.x; b < nb; b += kPtBlock)
            hist[b] = 0;
        __syncthreads();
        const uint32_t i = q.at(k) + threadIdx.x;
        uint32_t key = 0, local = 0;
        if (i < q.limit)
        {
            key = B.sort_keys[i];
            local = atomicAdd(&hist[key], 1u);
        }
        __syncthreads();
        for (uint32_t b = threadIdx.x; b < nb; b += kPtBlock)
            if (hist[b])
                base[b] = atomicAdd(&B.sort_bins[kSortMaxBins + b], hist[b]);
        __syncthreads();
        if (i < q.limit)
            B.sort_perm[base[key] + local] = i;
        __syncthreads();
    }
}

// ---- guide inference for the active queue ------------------------------------
// Query of a hit: position normalised to the scene box, geometric normal
// facing the incoming ray, outgoing direction.  The shade kernel builds the
// same query from the same values for its training records.
__device__ __forceinline__ void guide_query(const PtParams &P, V3 hitPos, V3 Ng, V3 rayDir,
                                            float q[9])
{
    q[0] = (hitPos.x - P.gbox_lo[0]) * P.gbox_inv[0];
    q[1] = (hitPos.y - P.gbox_lo[1]) * P.gbox_inv[1];
    q[2] = (hitPos.z - P.gbox_lo[2]) * P.gbox_inv[2];
    q[3] = Ng.x;
    q[4] = Ng.y;
    q[5] = Ng.z;
    q[6] = -rayDir.x;
    q[7] = -rayDir.y;
    q[8] = -rayDir.z;
}

// Path state word thr.w: bits 0-15 the path's depth, bits 16-30 the number of
// guided vertices it has passed, bit 31 set once its guide training record
// is taken.
constexpr uint32_t kDepthMask = 0xFFFFu;
constexpr uint32_t kGvisMask = 0x7FFFu;
constexpr uint32_t kGrecBit = 1u << 31;

// Whether the shade pass samples the guide at the vertex of queue item i: a
// hit on a mesh that emits nothing, below the depth cap, whose material has
// trans = 0 and clearcoat = 0, on a path that has passed fewer than gverts
// guided vertices (gverts = 0: no limit).  The shade kernel decides from the
// same values (its emitter, depth-cap and material branches, then gverts).
// SEL 0: every hit (no path state: diagnostics), 1: a path's first vertex
// (depth 0, none guided), 2: any later vertex (state read from thr).
template <int SEL>
__device__ __forceinline__ bool guide_wanted(const PtParams &P, const PtScene &S,
                                             const PtBuffers &B, const uint32_t *qin,
                                             uint32_t prim, uint32_t i)
{
    if (prim == WL_INVALID)
        return false;
    if (SEL == 0)
        return true;
    uint32_t depth = 0, gvis = 0;
    if (SEL == 2)
    {
        const uint32_t raw = __float_as_uint(B.thr[qin[i]].w);
        depth = raw & kDepthMask;
        gvis = (raw >> 16) & kGvisMask;
    }
    if (depth + 1 >= P.max_depth || (P.gverts != 0 && gvis >= P.gverts))
        return false;
    const uint32_t mesh = __float_as_uint(S.prims[12 * (size_t)prim + 9]);
    const PtMesh M = S.meshes[mesh];
    if (M.light != WL_INVALID)
        return false;
    const wl_disney_material &m = S.materials[M.material];
    return m.trans == 0.0f && m.clearcoat == 0.0f;
}

// Guide inference for the active queue.  Each wave walks its 64-item chunks
// of the queue, appends the items whose vertex the shade pass will guide to a
// ring of item indices in LDS, and runs the network on full 16-query tiles
// from the ring (the remainder at the end), so the MFMA work follows the
// guided vertices, not the queue length.  Results go to gout at the item's
// queue index; other items' slots are not written.
template <int SEL>
__global__ __launch_bounds__(kPtBlock)
void k_guide_infer_pt(PtParams P, PtScene S, PtBuffers B, int parity)
{
    constexpr int kRing = 128; // holds < 16 left over + 64 appended
    __shared__ bf16x8 sA[kGuideFwdVecs];
    __shared__ float sb[kGuideBiases];
    __shared__ float sq[9 * kPtBlock];
    __shared__ uint32_t sring[(kPtBlock / 64) * kRing];
    float *q = sq + 9 * threadIdx.x;
    uint32_t *ring = sring + (threadIdx.x / 64) * kRing;
    const bf16x8 *fwd = reinterpret_cast<const bf16x8 *>(P.gfwd);
    guide_stage<kPtBlock, kGuideFwdVecs>(sA, fwd);
    guide_stage_biases<kPtBlock>(sb, P.gparams);
    __syncthreads();
    const QueueWalk qw = queue_walk(B, parity, SEL != 2);
    const uint32_t *qin = parity ? B.qpath1 : B.qpath0;
    const wl_ray *rays = parity ? B.rays1 : B.rays0;
    const int lane = threadIdx.x & 63, g = lane >> 4;
    // one tile: ring entries [head, head + n), n <= 16 (wave-uniform)
    auto run_tile = [&](uint32_t head, uint32_t n) {
        const uint32_t k = (uint32_t)(lane & 15);
        const bool valid = k < n;
        const uint32_t i = valid ? ring[(head + k) % kRing] : 0u;
#pragma unroll
        for (int t = 0; t < 9; ++t)
            q[t] = 0.f;
        if (valid)
        {
            const float4 hit = reinterpret_cast<const float4 *>(B.hits)[i];
            float4 r0, r1;
            if (SEL == 1)
            {
                // the first queue: path i's camera ray (no ray queue is written)
                V3 co, cd;
                uint32_t sd;
                camera_ray(P, i, co, cd, sd);
                r0 = f4(co, P.epsilon);
                r1 = f4(cd, 1e30f);
            }
            else
            {
                const float4 *rp = reinterpret_cast<const float4 *>(rays + i);
                r0 = rp[0];
                r1 = rp[1];
            }
            const uint32_t prim = __float_as_uint(hit.y);
            const float4 *sr = reinterpret_cast<const float4 *>(S.prims) + 3 * (size_t)prim;
            const float4 w0 = sr[0], w1 = sr[1], w2 = sr[2];
            const V3 o = mk(r0.x, r0.y, r0.z), d = mk(r1.x, r1.y, r1.z);
            const V3 va = mk(w0.x, w0.y, w0.z), vb = mk(w0.w, w1.x, w1.y),
                     vc = mk(w1.z, w1.w, w2.x);
            V3 Ng = normalize(cross(vb - va, vc - va));
            if (dot(Ng, d) > 0)
                Ng = -Ng;
            guide_query(P, o + d * hit.x, Ng, d, q);
        }
        bf16x8 x[2];
        guide_encode(q, g, x);
        floatx4 o[2];
        guide_forward<false>(sA, sb, lane, x, o, nullptr);
        guide_decode_lanes(o, g, B.gout + kGuideDecoded * (size_t)i, valid);
    };
    uint32_t head = 0, tail = 0; // ring positions, wave-uniform
    // wave w of a workgroup takes the 64 entries 64 w of each of its blocks
    for (uint32_t b = blockIdx.x / 8u; qw.at(b) < qw.limit; b += gridDim.x / 8u)
    {
        const uint32_t i = qw.at(b) + threadIdx.x;
        bool want = false;
        if (i < qw.limit)
        {
            const uint32_t prim = reinterpret_cast<const uint32_t *>(B.hits)[4 * (size_t)i + 1];
            want = guide_wanted<SEL>(P, S, B, qin, prim, i);
        }
        const uint64_t m = __ballot(want);
        if (want)
            ring[(tail + lane_prefix(m)) % kRing] = i;
        tail += (uint32_t)__popcll(m);
        // the ring is read by other lanes of this wave: order the LDS
        // accesses at wave scope
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        while (tail - head >= 16u)
        {
            run_tile(head, 16u);
            head += 16u;
        }
    }
    if (tail != head)
        run_tile(head, tail - head);
}

// ---- shade ------------------------------------------------------------------
// GSAMPLE: one-sample MIS of the learned guide and the BSDF at vertices whose
// material has trans = 0 and clearcoat = 0.  There the reference's pdf equals
// the density its sampler draws from wherever the BSDF is non-zero, so
// mixing in the guide keeps the estimator's expectation unchanged.  The mixed
// density replaces the BSDF pdf everywhere the reference uses it (the path
// weight, lastPdf for emitter-hit MIS, the NEE MIS weight).
// MULTI: paths of many requests; each lane shades with its request's scene
// and parameters.
// GTRAIN: paths carry guide training records (radiance after the recorded
// vertex is summed; GSAMPLE vertices record themselves).
// TRACE: also writes the per-vertex record of PtBuffers::trace.
// The pass is bound by VALU issue (81 % busy on the 2M-triangle scene), so what
// counts is the instructions of the BSDF: with the terms that vanish for plain
// materials behind a branch and one sine and cosine for all lobes, two 1024^2
// Cornell frames 2.53 -> 2.32 ms, 256 small serving requests 9.2 -> 8.8 ms.  Four
// waves per SIMD: five (96 VGPRs, no spills) is 2-6 % slower.

// What a shaded vertex does next.
struct Vertex
{
    bool cont = false, shadow = false, shadow_gacc = false;
    uint32_t path = 0, req = 0, root = 0;
    wl_ray next_ray{}, shadow_ray{};
    V3 contrib{};
};

// Shades entry i of the ray queue: what its path does next, in `out`.
template <bool GSAMPLE, bool GTRAIN, bool MULTI, bool TRACE>
__device__ __forceinline__ void shade_vertex(const PtParams &P0, const PtScene &S0,
                                             const PtBuffers &B, int parity,
                                             const PtReq *__restrict__ reqs, int first, uint32_t i,
                                             Vertex &out)
{
    const uint32_t *qin = pick(parity, B.qpath0, B.qpath1);
    const uint32_t *req_in = pick(parity, B.qreq0, B.qreq1);
    // the first queue is the identity: entry i is path i
    const bool ident = first != 0;
    out.path = ident ? i : qin[i];
    if (MULTI)
        out.req = req_in[i];
    const PtReq *rq = MULTI ? reqs + out.req : nullptr;
    if (MULTI)
        out.root = rq->root;
    const PtParams &P = MULTI ? rq->P : P0;
    const PtScene &S = MULTI ? rq->S : S0;
    const float4 hit = reinterpret_cast<const float4 *>(B.hits)[i];
    float4 s_pos, s_dir, s_thr, s_ltt;
    if (first)
    {
        // the first vertex: single-scene batches recompute the camera
        // ray; multi-request ones read it (with lastPdf 1 and the
        // seed in its w words) from the queue the raygen pass wrote,
        // whose item lookup the shade pass would otherwise repeat
        if (MULTI)
        {
            const float4 *rp = reinterpret_cast<const float4 *>(B.rays0 + i);
            s_pos = rp[0];
            s_dir = rp[1];
        }
        else
        {
            V3 o, d;
            uint32_t sd;
            camera_ray(P, out.path, o, d, sd);
            s_pos = f4(o, 1.0f);                // w: lastPdf
            s_dir = f4(d, __uint_as_float(sd)); // w: seed
        }
        s_thr = f4(mk(1, 1, 1), __uint_as_float(0u)); // w: depth
        s_ltt = f4(mk(1, 1, 1), 1.0f); // w: miss weight
    }
    else
    {
        // the ray this pass shades: origin and lastPdf, then the
        // direction and the seed (written so by the last pass)
        const float4 *rp =
            reinterpret_cast<const float4 *>(pick(parity, B.rays0, B.rays1) + i);
        s_pos = rp[0];
        s_dir = rp[1];
        s_thr = B.thr[out.path];
        s_ltt = B.ltt[out.path];
    }
    V3 rayPos = v3of(s_pos);
    float lastPdf = s_pos.w;
    V3 rayDir = v3of(s_dir);
    uint32_t seed = __float_as_uint(s_dir.w);
    V3 throughput = v3of(s_thr);
    const uint32_t sw = __float_as_uint(s_thr.w);
    uint32_t depth = sw & kDepthMask;
    uint32_t gvis = (sw >> 16) & kGvisMask; // guided vertices passed
    V3 lastTraceTerm = v3of(s_ltt);
    float missw = 1.0f; // miss weight of the ray this vertex samples
    // radiance changes only at a miss or an emitter hit: read and
    // written back only then
    const bool gtrain = GTRAIN && (P.gmode & 2u);
    V3 radiance = mk(0, 0, 0), rad_in = mk(0, 0, 0);
    bool rad_dirty = false;
    const uint32_t prim = __float_as_uint(hit.y);
    bool done = false;
    // guiding: the path's training record is taken (its first guided
    // vertex); the radiance added after it goes to gacc
    const bool grec_done = gtrain && (sw & kGrecBit) != 0;
    bool grec_now = false;
    if (prim == WL_INVALID)
    {
        // __miss__radiance: radiance += throughput * bg.  The
        // reference leaves the last vertex's weight f |cos| / pdf
        // out of this term, so its expectation is throughput * bg
        // times the probability that the last vertex's sampler
        // sends the ray to the background.  s_ltt.w keeps that
        // expectation when a guided vertex sampled the ray: the
        // reference sampler's density over the mixed density
        // there, and exactly 1 after every other vertex.
        radiance = ident ? mk(0, 0, 0) : v3of(B.rad[out.path]);
        rad_in = radiance;
        radiance = radiance + throughput * ld3(P.bg) * s_ltt.w;
        rad_dirty = true;
        done = true;
    }
    else
    {
        depth += 1;
        const float t = hit.x, b1 = hit.z, b2 = hit.w;
        const float4 *sr = reinterpret_cast<const float4 *>(global_ptr(S.prims)) + 3 * (size_t)prim;
        const float4 w0 = sr[0], w1 = sr[1], w2 = sr[2];
        const V3 va = mk(w0.x, w0.y, w0.z), vb = mk(w0.w, w1.x, w1.y),
                 vc = mk(w1.z, w1.w, w2.x);
        const uint32_t mesh = __float_as_uint(w2.y);
        const PtMesh M = global_ptr(S.meshes)[mesh];
        V3 Ng = normalize(cross(vb - va, vc - va));
        V3 Ns;
        if (M.has_normal)
        {
            const float4 *nr = reinterpret_cast<const float4 *>(global_ptr(S.normals)) + 3 * (size_t)prim;
            const float4 n0 = nr[0], n1 = nr[1], n2 = nr[2];
            const V3 na = mk(n0.x, n0.y, n0.z), nb = mk(n0.w, n1.x, n1.y),
                     nc = mk(n1.z, n1.w, n2.x);
            Ns = normalize(na * (1 - b1 - b2) + nb * b1 + nc * b2);
        }
        else
            Ns = Ng;
        const V3 hitPos = rayPos + rayDir * t;
        if (M.light != WL_INVALID)
        {
            const PtLight lt = global_ptr(S.lights)[M.light];
            if (depth == 1 || (P.strategy != WL_STRATEGY_NEE &&
                               (lt.two_sided || dot(Ns, rayDir) < 0)))
            {
                float neePdf = 0.f;
                if (P.strategy != WL_STRATEGY_UPT && depth > 1)
                {
                    // PdfAreaLightPos (Pdf.h:20-31)
                    float pdf = 1.0f / (float)P.num_lights;
                    pdf /= (float)lt.tri_count;
                    pdf /= tri_area(va, vb, vc);
                    const float dist = t;
                    neePdf = pdf * dist * dist / fabsf(dot(Ns, rayDir));
                }
                const float uptPdf = lastPdf;
                radiance = ident ? mk(0, 0, 0) : v3of(B.rad[out.path]);
                rad_in = radiance;
                rad_dirty = true;
                radiance = radiance + throughput * ld3(lt.L) * lastTraceTerm *
                                          (uptPdf / (uptPdf + neePdf));
            }
            done = true;
        }
        else if (depth >= P.max_depth)
        {
            throughput = mk(0, 0, 0);
            done = true;
        }
        else
        {
            const Mat mat = load_mat(global_ptr(S.materials) + M.material);
            // texture colour (PathTracing.cu:261-268)
            V3 tex = mk(1, 1, 1);
            if (M.texture != WL_INVALID)
            {
                const float4 *ur = reinterpret_cast<const float4 *>(global_ptr(S.uvs)) + 2 * (size_t)prim;
                const float4 u01 = ur[0], u2 = ur[1];
                const float w0 = 1 - b1 - b2;
                const float tu = (u01.x * w0 + u01.z * b1) + u2.x * b2;
                const float tv = (u01.y * w0 + u01.w * b1) + u2.y * b2;
                const PtTexture T = global_ptr(S.textures)[M.texture];
                tex = tex_bilinear(global_ptr(S.texels) + T.offset, T.width, T.height, tu, tv);
            }
            if (mat.trans < 0.1f)
            {
                if (dot(Ng, rayDir) > 0)
                    Ng = -Ng;
                if (dot(Ns, rayDir) > 0)
                    Ns = -Ns;
            }
            const bool guided = GSAMPLE && mat.trans == 0.0f &&
                                mat.clearcoat == 0.0f && (P.gmode & 1u) &&
                                (P.gverts == 0 || gvis < P.gverts);
            if (GSAMPLE && guided)
                gvis += 1;
            GuideMix gm;
            bool took_guide = false;
            V3 nd;
            if (GSAMPLE && guided)
            {
                const float *gsrc = B.gout + kGuideDecoded * (size_t)i;
                guide_load(gsrc, gm);
                if (rnd(seed) < P.galpha)
                {
                    const float u0 = rnd(seed);
                    const float u1 = rnd(seed);
                    const float u2 = rnd(seed);
                    nd = guide_sample(gm, gsrc + 40, u0, u1, u2);
                    took_guide = true;
                }
            }
            if (!took_guide)
            {
                nd = sample_disney(mat, Ns, -rayDir, seed);
                nd = normalize(nd);
            }
            float pdf = pdf_disney(mat, Ns, -rayDir, nd);
            if (GSAMPLE && guided && !(pdf < 0.0f || __builtin_isnan(pdf)))
            {
                // the reference sampler's own density: its pdf less
                // the diffuse term below the surface, where the
                // sampler draws nothing (trans = 0, clearcoat = 0)
                const float cl = dot(nd, Ns);
                const float pb = pdf;
                float sdens = pdf;
                if (cl < 0.0f)
                    sdens -= 0.5f * (1.0f - mat.metallic) * (-cl * (1.0f / kPi));
                pdf = P.galpha * guide_pdf(gm, nd) + (1.0f - P.galpha) * pdf;
                if (!(pdf > 0.0f))
                    pdf = -1.0f; // a zero mixed density ends the path
                else if (__builtin_isinf(pb))
                    // the reference pdf is infinite where its GGX
                    // reflection folds back onto -V (1 / |L.H|, and
                    // its sampler does land there): the limit of
                    // s / p_mix as p_bsdf grows, not inf / inf
                    missw = 1.0f / (1.0f - P.galpha);
                else
                    missw = fmaxf(sdens, 0.0f) / pdf; // 0 if only q is infinite
            }
            if (pdf < 0.0f || __builtin_isnan(pdf))
            {
                done = true;
            }
            else
            {
                throughput = throughput * lastTraceTerm;
                const float cosWeight = dot(nd, Ns);
                V3 bsdf = eval_disney(mat, Ns, Ng, -rayDir, nd, tex);
                bsdf = clamp3(bsdf, 0.f, 1e30f);
                lastTraceTerm = bsdf * fabsf(cosWeight) / pdf;
                if (TRACE && depth - 1 < B.trace_max)
                {
                    float4 *tr = reinterpret_cast<float4 *>(
                        B.trace + 8 * ((size_t)out.path * B.trace_max + depth - 1));
                    tr[0] = make_float4((float)depth, (float)mesh, pdf,
                                        (lastTraceTerm.x + lastTraceTerm.y +
                                         lastTraceTerm.z) / 3.0f);
                    tr[1] = make_float4((throughput.x + throughput.y + throughput.z) /
                                            3.0f,
                                        0.0f, 0.0f, mat.trans);
                }
                const V3 lastRayDir = rayDir;
                if (GSAMPLE && guided && gtrain && !grec_done)
                {
                    // training record: query, sampled direction and
                    // the throughput reaching this vertex
                    float q[9];
                    guide_query(P, hitPos, Ng, rayDir, q);
                    float4 *r = reinterpret_cast<float4 *>(B.grec + 16 * (size_t)out.path);
                    r[0] = make_float4(q[0], q[1], q[2], q[3]);
                    r[1] = make_float4(q[4], q[5], q[6], q[7]);
                    r[2] = make_float4(q[8], nd.x, nd.y, nd.z);
                    r[3] = make_float4(0.0f, (throughput.x + throughput.y + throughput.z) *
                                                 (1.0f / 3.0f),
                                       0.0f, 0.0f);
                    grec_now = true;
                }
                rayPos = hitPos;
                rayDir = nd;
                lastPdf = pdf;
                // ---- NEE at this vertex (PathTracing.cu:81-128)
                if (P.strategy != WL_STRATEGY_UPT && P.num_lights > 0)
                {
                    uint32_t lid = (uint32_t)((float)P.num_lights * rnd(seed));
                    lid = lid < P.num_lights ? lid : P.num_lights - 1;
                    const PtLight lt = global_ptr(S.lights)[lid];
                    float lpdf = 1.0f / (float)P.num_lights;
                    uint32_t triIdx = (uint32_t)(rnd(seed) * (float)lt.tri_count);
                    triIdx = triIdx < lt.tri_count ? triIdx : lt.tri_count - 1;
                    lpdf = lpdf / (float)lt.tri_count;
                    const uint32_t lprim = lt.tri_offset + triIdx;
                    const float4 *lr = reinterpret_cast<const float4 *>(global_ptr(S.prims)) + 3 * (size_t)lprim;
                    const float4 l0 = lr[0], l1 = lr[1], l2 = lr[2];
                    const V3 p0 = mk(l0.x, l0.y, l0.z), p1 = mk(l0.w, l1.x, l1.y),
                             p2 = mk(l1.z, l1.w, l2.x);
                    float u = rnd(seed), v = rnd(seed);
                    if (u + v > 1)
                    {
                        u = 1 - u;
                        v = 1 - v;
                    }
                    const float cx = 1 - u - v, cy = u;
                    const V3 lpos = p0 + u * (p1 - p0) + v * (p2 - p0);
                    lpdf = lpdf / tri_area(p0, p1, p2);
                    V3 lN;
                    if (lt.has_normal)
                    {
                        const float4 *nr = reinterpret_cast<const float4 *>(global_ptr(S.normals)) + 3 * (size_t)lprim;
                        const float4 n0 = nr[0], n1 = nr[1], n2 = nr[2];
                        const V3 na = mk(n0.x, n0.y, n0.z), nb = mk(n0.w, n1.x, n1.y),
                                 nc = mk(n1.z, n1.w, n2.x);
                        // weights (1 - cx - cy, cx, cy), as Sample.h:121 applies them
                        lN = normalize(na * (1 - cx - cy) + nb * cx + nc * cy);
                    }
                    else
                        lN = normalize(cross(p1 - p0, p2 - p0));
                    V3 visRay = lpos - rayPos;
                    const float dist = length(visRay);
                    visRay = visRay / dist;
                    const float cosTheta1 = dot(lN, visRay);
                    if (lt.two_sided || cosTheta1 < 0)
                    {
                        const float cosTheta2 = dot(Ns, visRay);
                        const float neePdf = lpdf * dist * dist / fabsf(cosTheta1);
                        float uptPdf = 0.f;
                        if (P.strategy != WL_STRATEGY_NEE)
                        {
                            uptPdf = pdf_disney(mat, Ns, -lastRayDir, visRay);
                            if (uptPdf < 0 || __builtin_isnan(uptPdf))
                                uptPdf = 0.f;
                            if (GSAMPLE && guided)
                                uptPdf = P.galpha * guide_pdf(gm, visRay) +
                                         (1.0f - P.galpha) * uptPdf;
                        }
                        V3 bv = eval_disney(mat, Ns, Ng, -lastRayDir, visRay, tex);
                        bv = clamp3(bv, 0.f, 1e30f);
                        out.contrib = throughput * bv * fabsf(cosTheta2) * ld3(lt.L) / neePdf *
                                  (1 - uptPdf / (uptPdf + neePdf));
                        out.shadow = true;
                        out.shadow_ray = wl_ray{ rayPos.x, rayPos.y, rayPos.z, P.epsilon,
                                             visRay.x, visRay.y, visRay.z,
                                             dist * (1 - P.epsilon) };
                    }
                }
                // ---- Russian roulette (PathTracing.cu:130-138)
                if (depth > P.rr_depth)
                {
                    if (rnd(seed) > P.rr_prob)
                    {
                        throughput = mk(0, 0, 0);
                        done = true;
                    }
                    else
                        throughput = throughput / P.rr_prob;
                }
            }
        }
    }
    if (rad_dirty || ident) // the first pass starts every path's radiance
        B.rad[out.path] = f4(radiance, 0.0f);
    if (gtrain)
    {
        // radiance reaching the path after its first guided vertex
        if (grec_done && rad_dirty)
        {
            float4 gacc = B.gacc[out.path];
            gacc.x += radiance.x - rad_in.x;
            gacc.y += radiance.y - rad_in.y;
            gacc.z += radiance.z - rad_in.z;
            B.gacc[out.path] = gacc;
        }
        if (grec_now) // nothing gathered yet; w marks the record
            B.gacc[out.path] = make_float4(0.f, 0.f, 0.f, 1.0f);
        else if (ident) // no record yet
            B.gacc[out.path] = make_float4(0.f, 0.f, 0.f, 0.f);
        out.shadow_gacc = grec_done;
    }
    if (!done)
    {
        out.cont = true;
        B.thr[out.path] = f4(throughput,
                         __uint_as_float(depth | (gvis << 16) |
                                         (grec_done || grec_now ? kGrecBit : 0u)));
        B.ltt[out.path] = f4(lastTraceTerm, missw);
        // the path's lastPdf and seed ride in the ray's w words
        out.next_ray = wl_ray{ rayPos.x, rayPos.y, rayPos.z, lastPdf,
                           rayDir.x, rayDir.y, rayDir.z, __uint_as_float(seed) };
    }
}

// Writes a shaded vertex's ray to the other ray queue and its shadow ray.
template <bool MULTI>
__device__ __forceinline__ void store_vertex(const PtBuffers &B, int parity, const Vertex &v,
                                             uint32_t slot, uint32_t sslot)
{
    if (v.cont)
    {
        pick(parity, B.qpath1, B.qpath0)[slot] = v.path;
        pick(parity, B.rays1, B.rays0)[slot] = v.next_ray;
        if (MULTI)
            pick(parity, B.qreq1, B.qreq0)[slot] = v.req;
    }
    if (v.shadow)
    {
        B.spath[sslot] = v.path;
        if (MULTI)
            B.sreq[sslot] = v.root;
        B.srays[sslot] = v.shadow_ray;
        B.scontrib[sslot] = f4(v.contrib, v.shadow_gacc ? 1.0f : 0.0f);
    }
}

template <bool GSAMPLE, bool GTRAIN, bool MULTI, bool TRACE = false>
__global__ __launch_bounds__(kPtBlock)
__attribute__((amdgpu_waves_per_eu(GSAMPLE || GTRAIN ? 3 : 4)))
void k_shade(PtParams P0, PtScene S0, PtBuffers B, int parity, const PtReq *__restrict__ reqs,
             int first)
{
    QueueWalk q = queue_walk(B, parity, first != 0);
    if (!MULTI && P0.sort_bins)
    {
        // the sorted order of the whole queue, dealt in blocks as the first's
        // (one word: the eight segments' lengths cost every workgroup 2 us more)
        q = dealt_walk<kPtBlock>(B.counters[kPtSortTotal], blockIdx.x % 8u);
    }
    if (blockIdx.x < 8u && threadIdx.x == 0)
        *queue_chunks(B, blockIdx.x) = 0u; // the next trace counts from zero
    const uint32_t seg = (blockIdx.x % 8u) * B.segcap;
    __shared__ BlockAppendLds app;
    uint32_t pass = 0;
    // every thread of the workgroup runs the same passes (k is per
    // workgroup), as the workgroup barriers of the append require
    for (uint32_t k = blockIdx.x / 8u; q.at(k) < q.limit; k += gridDim.x / 8u)
    {
        const uint32_t j = q.at(k) + threadIdx.x;
        const bool in_range = j < q.limit;
        // material-sorted order: the j-th entry of the sorted queue
        const uint32_t i = (!MULTI && P0.sort_bins && in_range) ? B.sort_perm[j] : j;
        Vertex v;
        if (in_range)
            shade_vertex<GSAMPLE, GTRAIN, MULTI, TRACE>(P0, S0, B, parity, reqs, first, i, v);
        // ---- compaction (whole wave participates)
        uint32_t slot, sslot;
        block_append2(app, pass++, queue_len(B, blockIdx.x % 8u, parity ^ 1), v.cont, v.shadow,
                      slot, sslot);
        store_vertex<MULTI>(B, parity, v, seg + slot, seg + sslot);
    }
}

// ---- finish: the remaining bounces of every path --------------------------------
// In a batch of up to a few million paths a launch soon takes as long as its
// slowest ray (70-90 us from the caustic's third bounce on, for a few thousand
// rays) and an empty one 4.5 us.  So after kLaunchedBounces bounces each
// workgroup takes a slice of its XCD's ray
// segment and runs that slice's bounces to the end by itself: shade (appending
// to its own slice of the other queue), barrier, trace the slice's rays and
// shadow rays, barrier.  A slow ray then holds up its own workgroup's slice
// only, and the remaining bounces need no launches of their own.  The slices
// reuse the queues' memory: an entry appends at most one to each queue, so the
// slice [e0, e0 + n) of one queue always fits [e0, e0 + n) of the others.
// Measured with bounces launched / finished here (after 2): 65,536 Cornell paths
// of 25 bounces 557 / 368 us, 1M 1179 / 956, 3M 2455 / 2256; 1M paths on the
// 2M-triangle scene 2827 / 2092, 3M 4161 / 3652; 1M caustic paths 1874 / 1320.
// Finishing after 1, 3 or 5 bounces: within 2 % of 2 on Cornell, 1406 / 1388 /
// 1498 on the caustic.  Larger batches keep the launched bounces (as two lanes
// of 3M Cornell paths each 4098 / 4679): their queues stay long, and this kernel
// holds four waves per SIMD, the shade pass's registers, where k_trace holds six.
// A material-sorted batch sorts its launched bounces only.  Long paths that lie
// together in the image do not undo the gain by keeping few workgroups busy: with
// a deep cavity behind 1/2 to 1/32 of a flat scene's pixels, 66K to 4M paths of 25
// to 100 bounces take 0.31 to 0.63 of what they took before k_trace and this kernel.
constexpr uint32_t kLaunchedBounces = 2;
constexpr uint32_t kMaxSlice = 4096;

template <int STACK, bool WIDE, bool GTRAIN, bool MULTI>
__global__ __launch_bounds__(kPtBlock) __attribute__((amdgpu_waves_per_eu(4)))
void k_finish(PtParams P0, PtScene S0, PtBuffers B, int parity, const PtReq *__restrict__ reqs)
{
    __shared__ uint32_t stack[STACK * kPtBlock];
    __shared__ uint4 top[8 * (pt_top_nodes<STACK, MULTI>() ? pt_top_nodes<STACK, MULTI>() : 1)];
    __shared__ BlockAppendLds app;
    __shared__ unsigned long long s_len; // the slice's queue lengths: rays, shadow rays
    __shared__ uint32_t s_chunk;         // its chunk counter
    const uint32_t x = blockIdx.x % 8u, nblk = gridDim.x / 8u;
    const uint32_t total = (uint32_t)*queue_len(B, x, parity);
    // equal slices of whole waves, one per workgroup while they are short
    const uint32_t share = ((total + nblk - 1u) / nblk + 63u) & ~63u;
    const uint32_t slice = min(share, kMaxSlice);
    if ((blockIdx.x / 8u) * slice >= total)
        return;
    const uint32_t ntop = pt_load_top<STACK, MULTI>(top, S0);
    unsigned long long rays = 0, shadows = 0; // traced by this workgroup
    uint32_t pass = 0;
    for (uint32_t at = (blockIdx.x / 8u) * slice; at < total; at += nblk * slice)
    {
        const uint32_t e0 = x * B.segcap + at;
        int par = parity;
        uint32_t n = min(slice, total - at);
        while (n != 0)
        {
            if (threadIdx.x == 0)
            {
                s_len = 0ull;
                s_chunk = 0u;
            }
            __syncthreads();
            for (uint32_t k = 0; k < n; k += kPtBlock)
            {
                Vertex v;
                if (k + threadIdx.x < n)
                    shade_vertex<false, GTRAIN, MULTI, false>(P0, S0, B, par, reqs, 0,
                                                              e0 + k + threadIdx.x, v);
                uint32_t slot, sslot;
                block_append2(app, pass++, &s_len, v.cont, v.shadow, slot, sslot);
                store_vertex<MULTI>(B, par, v, e0 + slot, e0 + sslot);
            }
            par ^= 1;
            __syncthreads(); // the appended entries and lengths
            const unsigned long long len = s_len;
            const uint32_t nrays = __builtin_amdgcn_readfirstlane((uint32_t)len);
            const uint32_t nshadow = __builtin_amdgcn_readfirstlane((uint32_t)(len >> 32));
            rays += nrays;
            shadows += nshadow;
            const SegmentChunks range(e0, nrays, nshadow, 64u);
            bool shadow = false; // the kind of the wave's current chunk
            trav_persistent<kMixed, kPtBlock, WIDE, pt_top_nodes<STACK, MULTI>() != 0>(
                S0.nodes, S0.tris, stack,
                [&](bool, uint32_t &next, uint32_t &end) {
                    uint32_t c = 0;
                    if (__lane_id() == 0)
                        c = atomicAdd(&s_chunk, 1u);
                    range(__builtin_amdgcn_readfirstlane(c), next, end, shadow);
                },
                [&](uint32_t i, TravRay &r, uint32_t &root) {
                    queue_fetch<MULTI>(B, par, reqs, P0.epsilon, shadow, i, r, root);
                },
                [&](uint32_t i, const TravRay &r, const TravResult &h) {
                    queue_emit(B, i, r, h);
                },
                reinterpret_cast<const WlBvh8Node *>(top), ntop);
            __syncthreads(); // every hit and NEE contribution of this bounce
            n = nrays;
        }
    }
    if (threadIdx.x == 0)
    {
        atomicAdd(&B.stats[0], rays);
        atomicAdd(&B.stats[1], shadows);
    }
}

// ---- batched serving: raygen and film update of a multi-request megabatch ----
__global__ void k_batch_begin(PtMultiLaunch L, PtBuffers B)
{
    const PtBatchHeader h = L.batches[*L.batch_index];
    if (threadIdx.x == 0)
        *L.header = h;
    start_counters(B, h.paths);
}

__global__ void k_batch_end(PtMultiLaunch L)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
    {
        const uint32_t b = *L.batch_index;
        L.times[b] = (unsigned long long)wall_clock64(); // the batch's film update is done
        *L.batch_index = b + 1;
    }
}

__global__ void k_clock_stamp(unsigned long long *dst)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *dst = (unsigned long long)wall_clock64();
}

__global__ __launch_bounds__(kPtBlock) void k_raygen_multi(PtMultiLaunch L, PtBuffers B)
{
    const PtBatchHeader h = *L.header;
    const uint32_t npaths = h.paths, nitems = h.items;
    const PtItem *items = L.items + h.item_offset;
    for (uint32_t p = blockIdx.x * kPtBlock + threadIdx.x; p < npaths;
         p += gridDim.x * kPtBlock)
    {
        const PtItem it = items[find_item(items, nitems, p, false)];
        const PtParams &P = L.reqs[it.req].P;
        const uint32_t local = p - it.path0;
        const uint32_t pixel = local % it.npix;
        const uint32_t s = local / it.npix;
        const uint32_t x = pixel % P.width, y = pixel / P.width;
        uint32_t seed = tea4(pixel, it.frame0 + s);
        // PinholeGenerateRay (Camera.h:28-35): two draws, u then v
        const float u = 2.f * ((float)(int)x + rnd(seed)) / (float)(int)P.width - 1.f;
        const float v = 2.f * ((float)(int)y + rnd(seed)) / (float)(int)P.height - 1.f;
        const V3 d = normalize(ld3(P.cam.lookat) + ld3(P.cam.right) * u + ld3(P.cam.up) * v);
        const V3 o = ld3(P.cam.pos);
        // the ray carries lastPdf 1 and the seed in its w words, as the
        // shade pass writes its rays; the first shade pass takes path = p
        // and starts the path's radiance and state
        B.rays0[p] = wl_ray{ o.x, o.y, o.z, 1.0f, d.x, d.y, d.z, __uint_as_float(seed) };
        B.qreq0[p] = it.req;
    }
}

// Kahan update of each item's film, samples in ascending order (the order
// a single-request render adds them in).
__global__ __launch_bounds__(kPtBlock) void k_accumulate_multi(PtMultiLaunch L, PtBuffers B)
{
    const PtBatchHeader h = *L.header;
    const uint32_t nitems = h.items, npix = h.pixels;
    const PtItem *items = L.items + h.item_offset;
    for (uint32_t x = blockIdx.x * kPtBlock + threadIdx.x; x < npix; x += gridDim.x * kPtBlock)
    {
        const PtItem it = items[find_item(items, nitems, x, true)];
        const uint32_t px = x - it.px0;
        float *f = L.reqs[it.req].film + 6 * (size_t)px;
        float sum[3] = { f[0], f[1], f[2] }, c[3] = { f[3], f[4], f[5] };
        for (uint32_t s = 0; s < it.nsamples; ++s)
        {
            const float4 r = B.rad[it.path0 + (size_t)s * it.npix + px];
            const float v[3] = { r.x, r.y, r.z };
#pragma unroll
            for (int k = 0; k < 3; ++k)
            {
                const float y = v[k] - c[k];
                const float t = sum[k] + y;
                c[k] = (t - sum[k]) - y;
                sum[k] = t;
            }
        }
        for (int k = 0; k < 3; ++k)
        {
            f[k] = sum[k];
            f[3 + k] = c[k];
        }
    }
}

// ---- guide training samples -----------------------------------------------------
// A recorded vertex's weight is F/p of its sampled direction: the radiance
// the path gathered through that direction divided by the throughput that
// reached the vertex (channel means).  Zero-weight records carry no gradient
// and are dropped.
// Each thread takes kCollectPer paths per pass (coalesced: path base + k
// kPtBlock + thread) and the workgroup claims the training slots of the whole
// pass with one atomic: one per 2048 paths, where one per wave serialised
// the kernel on the counter.
constexpr uint32_t kCollectPer = 8;

__global__ __launch_bounds__(kPtBlock) void k_guide_collect(PtParams P, PtBuffers B)
{
    __shared__ uint32_t s_cnt[kPtBlock / 64];
    __shared__ uint32_t s_base;
    const uint32_t npaths = P.npix * P.nsamples;
    const uint32_t wave = threadIdx.x / 64u, lane = __lane_id();
    constexpr uint32_t span = kPtBlock * kCollectPer;
    // block-uniform loop: every thread runs the same passes (barriers)
    for (uint32_t base = blockIdx.x * span; base < npaths; base += gridDim.x * span)
    {
        float w[kCollectPer];
        uint64_t m[kCollectPer];
        uint32_t wtotal = 0;
#pragma unroll
        for (uint32_t k = 0; k < kCollectPer; ++k)
        {
            const uint32_t p = base + k * kPtBlock + threadIdx.x;
            bool keep = false;
            w[k] = 0.f;
            if (p < npaths)
            {
                const float4 ga = B.gacc[p];
                if (ga.w != 0.0f)
                {
                    const float thr = B.grec[16 * (size_t)p + 13];
                    const float wk = (ga.x + ga.y + ga.z) * (1.0f / 3.0f) / fmaxf(thr, 1e-30f);
                    keep = wk > 0.0f; // false for NaN
                    w[k] = fminf(wk, B.gwmax);
                }
            }
            m[k] = __ballot(keep);
            wtotal += (uint32_t)__popcll(m[k]);
        }
        if (lane == 0)
            s_cnt[wave] = wtotal;
        __syncthreads();
        if (threadIdx.x == 0)
        {
            uint32_t t = 0;
            for (uint32_t v = 0; v < kPtBlock / 64; ++v)
                t += s_cnt[v];
            s_base = t ? atomicAdd(B.gcount, t) : 0u;
        }
        __syncthreads();
        uint32_t o = s_base;
        for (uint32_t v = 0; v < wave; ++v)
            o += s_cnt[v];
#pragma unroll
        for (uint32_t k = 0; k < kCollectPer; ++k)
        {
            if ((m[k] >> lane) & 1u)
            {
                const uint32_t slot = o + lane_prefix(m[k]);
                const uint32_t p = base + k * kPtBlock + threadIdx.x;
                if (slot < B.gtrain_cap)
                {
                    const float4 *src = reinterpret_cast<const float4 *>(B.grec + 16 * (size_t)p);
                    float4 *dst = reinterpret_cast<float4 *>(B.gtrain + 16 * (size_t)slot);
                    dst[0] = src[0];
                    dst[1] = src[1];
                    dst[2] = src[2];
                    dst[3] = make_float4(w[k], 0.0f, 0.0f, 0.0f);
                }
            }
            o += (uint32_t)__popcll(m[k]);
        }
        __syncthreads(); // s_cnt and s_base are rewritten by the next pass
    }
}

// ---- film -----------------------------------------------------------------
// Kahan-compensated sum over the batch's samples of each pixel, in sample
// order: film = [sum RGB, compensation RGB] per pixel.
__global__ __launch_bounds__(kPtBlock) void k_accumulate(PtParams P, PtBuffers B, float *film)
{
    for (uint32_t px = blockIdx.x * kPtBlock + threadIdx.x; px < P.npix;
         px += gridDim.x * kPtBlock)
    {
        float *f = film + 6 * ((size_t)P.pix0 + px);
        float sum[3] = { f[0], f[1], f[2] }, c[3] = { f[3], f[4], f[5] };
        for (uint32_t s = 0; s < P.nsamples; ++s)
        {
            const float4 r = B.rad[(size_t)s * P.npix + px];
            const float v[3] = { r.x, r.y, r.z };
#pragma unroll
            for (int k = 0; k < 3; ++k)
            {
                const float y = v[k] - c[k];
                const float t = sum[k] + y;
                c[k] = (t - sum[k]) - y;
                sum[k] = t;
            }
        }
        for (int k = 0; k < 3; ++k)
        {
            f[k] = sum[k];
            f[3 + k] = c[k];
        }
    }
}

__global__ void k_store_samples(PtParams P, PtBuffers B, float *rgb)
{
    for (uint32_t px = blockIdx.x * blockDim.x + threadIdx.x; px < P.npix;
         px += gridDim.x * blockDim.x)
    {
        const float4 r = B.rad[px];
        const size_t o = 3 * ((size_t)P.pix0 + px);
        rgb[o] = r.x;
        rgb[o + 1] = r.y;
        rgb[o + 2] = r.z;
    }
}

// Reference progressive film (PathTracing.cu:140-158): running mean with
// float factors and double temporaries in an RGBA float buffer, clamp,
// ACES, x255, truncate to u8.
__global__ void k_frame_update(PtParams P, PtBuffers B, uint32_t frame, float *acc,
                               uint8_t *color)
{
    for (uint32_t px = blockIdx.x * blockDim.x + threadIdx.x; px < P.npix;
         px += gridDim.x * blockDim.x)
    {
        const float4 r = B.rad[px];
        const double tf[4] = { 0.0 + (double)(r.x / 1), 0.0 + (double)(r.y / 1),
                               0.0 + (double)(r.z / 1), 1.0 };
        float *a = acc + 4 * ((size_t)P.pix0 + px);
        if (frame == 0)
        {
            for (int k = 0; k < 4; ++k)
                a[k] = (float)tf[k];
        }
        else
        {
            const double f0 = (double)((float)frame / ((float)frame + 1.0f));
            const double f1 = (double)(1.0f / ((float)frame + 1.0f));
            for (int k = 0; k < 4; ++k)
                a[k] = (float)((double)a[k] * f0 + tf[k] * f1);
        }
        uint8_t *c = color + 4 * ((size_t)P.pix0 + px);
        for (int k = 0; k < 3; ++k)
            c[k] = (uint8_t)(aces1(clampf(a[k], 0.f, 1e30f)) * 255.0f);
        c[3] = (uint8_t)(1.0f * 255.0f);
    }
}

__global__ void k_resolve(const float *film, uint32_t npix, uint32_t nsamples, float *rgb)
{
    for (uint32_t px = blockIdx.x * blockDim.x + threadIdx.x; px < npix;
         px += gridDim.x * blockDim.x)
    {
        for (int k = 0; k < 3; ++k)
            rgb[3 * (size_t)px + k] =
                (film[6 * (size_t)px + k] - film[6 * (size_t)px + 3 + k]) / (float)nsamples;
    }
}

// ---- host side: one batch ---------------------------------------------------
// Workgroups of `kernel` that fit a CU at once.
template <class K>
static int blocks_per_cu(K kernel)
{
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kPtBlock, 0) != hipSuccess ||
        n < 1)
        n = 4;
    return n;
}

// A grid of at most `blocks` workgroups and per_cu per CU, a multiple of 8.
static uint32_t grid8(uint32_t blocks, int num_cus, int per_cu)
{
    const uint32_t fit = (uint32_t)std::max(1, num_cus) * (uint32_t)per_cu;
    return (std::min<uint32_t>(blocks, fit) + 7u) & ~7u;
}

hipError_t pt_run_batch(const PtParams &P, const PtScene &S, const PtBuffers &B0,
                        bool alone, int num_cus, hipStream_t st)
{
    const uint32_t npaths = P.npix * P.nsamples;
    const uint32_t blocks_all = (npaths + kPtBlock - 1) / kPtBlock;
    // persistent traversal grids: the workgroups that fit the GPU at once.  All
    // grids are multiples of 8 (each XCD its share).
    static int occ[3] = {}, occ_first[3] = {}; // per traversal variant
    const uint32_t trav = S.trav_variant;
    if (!occ[trav])
        with_variant(trav, [&](auto v) {
            using V = decltype(v);
            occ_first[trav] = blocks_per_cu(k_trace_first<V::STACK, V::WIDE>);
            occ[trav] = blocks_per_cu(k_trace<V::STACK, V::WIDE, false>);
        });
    const uint32_t g_trav = grid8(4 * blocks_all, num_cus, occ[trav]);
    const uint32_t g_first = grid8(4 * blocks_all, num_cus, occ_first[trav]);
    const uint32_t g_shade = grid8(blocks_all, num_cus, 8);
    const uint32_t g_sort = grid8(blocks_all, num_cus, 4);
    // guide inference: up to 4 workgroups per CU
    const uint32_t g_guide = grid8(blocks_all, num_cus, 4);
    PtBuffers B = B0;
    B.segcap = pt_segment(npaths);
    auto trace = [&](int parity) {
        with_variant(trav, [&](auto v) {
            using V = decltype(v);
            hipLaunchKernelGGL((k_trace<V::STACK, V::WIDE, false>), dim3(g_trav), dim3(kPtBlock),
                               0, st, S, B, parity, nullptr, P.epsilon, 0);
        });
    };
    hipLaunchKernelGGL(k_batch_start, dim3(1), dim3(kPtBlock), 0, st, P, B);
    with_variant(trav, [&](auto v) {
        using V = decltype(v);
        hipLaunchKernelGGL((k_trace_first<V::STACK, V::WIDE>), dim3(g_first), dim3(kPtBlock), 0,
                           st, P, S, B);
    });
    // the guide's inference and the per-vertex trace belong to the launched bounces
    const bool finish = alone && npaths < kFinishMaxPaths &&
                        P.max_depth > kLaunchedBounces + 1 && !B.trace &&
                        (!(P.gmode & 1u) || (P.gbounces != 0 && P.gbounces <= kLaunchedBounces));
    const uint32_t bounces = finish ? kLaunchedBounces : P.max_depth;
    for (uint32_t b = 0; b < bounces; ++b)
    {
        const int parity = (int)(b & 1u), first = b == 0 ? 1 : 0;
        if (P.sort_bins)
        {
            hipLaunchKernelGGL(k_sort_count, dim3(g_sort), dim3(kPtBlock), 0, st, P, S, B, parity,
                               first);
            hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(kPtBlock), 0, st, P, B);
            hipLaunchKernelGGL(k_sort_scatter, dim3(g_sort), dim3(kPtBlock), 0, st, P, B, parity,
                               first);
        }
        // guided sampling on the first gbounces bounces (0 = all)
        const bool gsample = (P.gmode & 1u) && (P.gbounces == 0 || b < P.gbounces);
        const bool gtrain = (P.gmode & 2u) != 0;
        if (gsample)
        {
            if (b == 0)
                hipLaunchKernelGGL(k_guide_infer_pt<1>, dim3(g_guide), dim3(kPtBlock), 0, st, P,
                                   S, B, parity);
            else
                hipLaunchKernelGGL(k_guide_infer_pt<2>, dim3(g_guide), dim3(kPtBlock), 0, st, P,
                                   S, B, parity);
            if (gtrain)
                hipLaunchKernelGGL((k_shade<true, true, false>), dim3(g_shade), dim3(kPtBlock), 0,
                                   st, P, S, B, parity, nullptr, first);
            else
                hipLaunchKernelGGL((k_shade<true, false, false>), dim3(g_shade), dim3(kPtBlock),
                                   0, st, P, S, B, parity, nullptr, first);
        }
        else if (gtrain)
            hipLaunchKernelGGL((k_shade<false, true, false>), dim3(g_shade), dim3(kPtBlock), 0, st,
                               P, S, B, parity, nullptr, first);
        else if (B.trace)
            hipLaunchKernelGGL((k_shade<false, false, false, true>), dim3(g_shade),
                               dim3(kPtBlock), 0, st, P, S, B, parity, nullptr, first);
        else
            hipLaunchKernelGGL((k_shade<false, false, false>), dim3(g_shade), dim3(kPtBlock), 0,
                               st, P, S, B, parity, nullptr, first);
        trace(parity ^ 1); // the next bounce's rays, this bounce's shadow rays
    }
    if (finish)
    {
        const bool gtrain = (P.gmode & 2u) != 0;
        with_variant(trav, [&](auto v) {
            using V = decltype(v);
            hipLaunchKernelGGL((gtrain ? k_finish<V::STACK, V::WIDE, true, false>
                                       : k_finish<V::STACK, V::WIDE, false, false>),
                               dim3(grid8(4 * blocks_all, num_cus, 4)), dim3(kPtBlock), 0, st, P,
                               S, B, (int)(kLaunchedBounces & 1u), nullptr);
        });
    }
    return hipGetLastError();
}

static int g_multi_occ[3] = {}; // per traversal variant

void pt_multi_init()
{
    for (uint32_t trav = 3; trav-- > 0;)
        if (!g_multi_occ[trav])
            with_variant(trav, [&](auto v) {
                using V = decltype(v);
                g_multi_occ[trav] = blocks_per_cu(k_trace<V::STACK, V::WIDE, true>);
            });
}

hipError_t pt_clock_stamp(unsigned long long *dst, hipStream_t st)
{
    hipLaunchKernelGGL(k_clock_stamp, dim3(1), dim3(64), 0, st, dst);
    return hipGetLastError();
}

hipError_t pt_run_multi(const PtMultiLaunch &L, const PtBuffers &B0, int num_cus, hipStream_t st)
{
    pt_multi_init();
    const uint32_t blocks_all = (L.capacity + kPtBlock - 1) / kPtBlock;
    const uint32_t g_gen = grid8(blocks_all, num_cus, 8);
    const uint32_t g_trav = grid8(4 * blocks_all, num_cus, g_multi_occ[L.trav_variant]);
    const uint32_t g_shade =
        grid8(blocks_all, num_cus, (int)std::max<uint32_t>(1, L.shade_blocks_per_cu));
    const PtParams P0{};
    const PtScene S0{};
    PtScene SA{}; // traversal: the node/triangle arena of the requests' BVHs
    SA.nodes = L.nodes;
    SA.tris = L.tris;
    PtBuffers B = B0;
    B.segcap = pt_segment(L.capacity);
    auto trace = [&](int parity, int first) {
        with_variant(L.trav_variant, [&](auto v) {
            using V = decltype(v);
            hipLaunchKernelGGL((k_trace<V::STACK, V::WIDE, true>), dim3(g_trav), dim3(kPtBlock), 0,
                               st, SA, B, parity, L.reqs, 0.0f, first);
        });
    };
    hipLaunchKernelGGL(k_batch_begin, dim3(1), dim3(kPtBlock), 0, st, L, B);
    hipLaunchKernelGGL(k_raygen_multi, dim3(g_gen), dim3(kPtBlock), 0, st, L, B);
    trace(0, 1);
    const bool finish = L.finish && L.max_depth > kLaunchedBounces + 1;
    const uint32_t bounces = finish ? kLaunchedBounces : L.max_depth;
    for (uint32_t b = 0; b < bounces; ++b)
    {
        const int parity = (int)(b & 1u);
        hipLaunchKernelGGL((k_shade<false, false, true>), dim3(g_shade), dim3(kPtBlock), 0, st,
                           P0, S0, B, parity, L.reqs, b == 0 ? 1 : 0);
        trace(parity ^ 1, 0);
    }
    if (finish)
        with_variant(L.trav_variant, [&](auto v) {
            using V = decltype(v);
            hipLaunchKernelGGL((k_finish<V::STACK, V::WIDE, false, true>),
                               dim3(grid8(4 * blocks_all, num_cus, 4)), dim3(kPtBlock), 0, st, P0,
                               SA, B, (int)(kLaunchedBounces & 1u), L.reqs);
        });
    hipLaunchKernelGGL(k_accumulate_multi, dim3(g_gen), dim3(kPtBlock), 0, st, L, B);
    hipLaunchKernelGGL(k_batch_end, dim3(1), dim3(64), 0, st, L);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_arena_copy_nodes(WlBvh8Node *__restrict__ dst,
                                                          const WlBvh8Node *__restrict__ src,
                                                          uint32_t n, uint32_t node0,
                                                          uint32_t tri0)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    WlBvh8Node v = src[i];
    v.child_base += node0;
    v.tri_base += tri0;
    dst[node0 + i] = v;
}

hipError_t pt_arena_copy_nodes(WlBvh8Node *dst, const WlBvh8Node *src, uint32_t n,
                               uint32_t node0, uint32_t tri0, hipStream_t st)
{
    if (n == 0)
        return hipSuccess;
    hipLaunchKernelGGL(k_arena_copy_nodes, dim3((n + 255) / 256), dim3(256), 0, st, dst, src, n,
                       node0, tri0);
    return hipGetLastError();
}

hipError_t pt_guide_infer_queue(const PtParams &P, const PtScene &S, const PtBuffers &B,
                                uint32_t n, int num_cus, hipStream_t st)
{
    const uint32_t g = grid8((n + kPtBlock - 1) / kPtBlock, num_cus, 4);
    hipLaunchKernelGGL(k_guide_infer_pt<0>, dim3(g), dim3(kPtBlock), 0, st, P, S, B, 0);
    return hipGetLastError();
}

hipError_t pt_guide_collect(const PtParams &P, const PtBuffers &B, int num_cus, hipStream_t st)
{
    const uint32_t npaths = P.npix * P.nsamples;
    const uint32_t span = kPtBlock * kCollectPer;
    const uint32_t g =
        std::max<uint32_t>(1, std::min<uint32_t>((npaths + span - 1) / span, (uint32_t)num_cus * 8));
    hipLaunchKernelGGL(k_guide_collect, dim3(g), dim3(kPtBlock), 0, st, P, B);
    return hipGetLastError();
}

hipError_t pt_accumulate(const PtParams &P, const PtBuffers &B, float *film, int num_cus,
                         hipStream_t st)
{
    const uint32_t g = std::min<uint32_t>((P.npix + kPtBlock - 1) / kPtBlock, (uint32_t)num_cus * 8);
    hipLaunchKernelGGL(k_accumulate, dim3(g), dim3(kPtBlock), 0, st, P, B, film);
    return hipGetLastError();
}

hipError_t pt_store_samples(const PtParams &P, const PtBuffers &B, float *rgb, hipStream_t st)
{
    const uint32_t g = std::min<uint32_t>((P.npix + 255) / 256, 4096);
    hipLaunchKernelGGL(k_store_samples, dim3(g), dim3(256), 0, st, P, B, rgb);
    return hipGetLastError();
}

hipError_t pt_frame_update(const PtParams &P, const PtBuffers &B, uint32_t frame, float *acc,
                           uint8_t *color, hipStream_t st)
{
    const uint32_t g = std::min<uint32_t>((P.npix + 255) / 256, 4096);
    hipLaunchKernelGGL(k_frame_update, dim3(g), dim3(256), 0, st, P, B, frame, acc, color);
    return hipGetLastError();
}

hipError_t pt_resolve(const float *film, uint32_t npix, uint32_t nsamples, float *rgb,
                      hipStream_t st)
{
    const uint32_t g = std::min<uint32_t>((npix + 255) / 256, 4096);
    hipLaunchKernelGGL(k_resolve, dim3(g), dim3(256), 0, st, film, npix, nsamples, rgb);
    return hipGetLastError();
}

} // namespace wl
