// traverse_persistent.h — persistent traversal with lane refill (gfx950).
//
// Incoherent rays finish after very different numbers of steps, so a wave
// that runs one ray per lane to completion idles most of its lanes near the
// end.  Here a fixed grid of waves loops; once at least kRefillLanes lanes of
// a wave are idle, they hand out their finished results and start the next rays of
// the wave's own ray indices (after Aila & Laine, "Understanding the
// Efficiency of Ray Traversal on GPUs", HPG 2009).
//
// Each pass of the loop runs the triangle step, the node step or both, for the
// lanes that can take it.  The kernels are bound by VALU issue (a node step is
// about 165 instructions, a triangle step about 120, whatever the number of
// lanes in it), so a step waits until enough lanes need it: the triangle step
// until kTriLanes hold a pending triangle, the node step until kNodeLanes can
// take a node, unless nothing else can run.  Once the wave's rays are used up
// every pass runs both: the last rays' latency counts then, not the issue
// slots.  Running both on every pass left
// 9 lanes of 64 in the triangle step on the 2M-triangle soup, and 21 in the
// node step on a 36-triangle box.  With the steps apart, 32-bit node offsets
// and results handed out at the refill: 2^23 incoherent rays 842 -> 727 us
// (closest hit) and 679 -> 603 us (any hit), the 1080p wavefront render
// 46.2 -> 40.9 ms, the 256 small serving requests 13.2 -> 11.5 ms.
//
// The rays come in chunks that a wave takes one after the other (XcdChunks for
// a launch over the whole GPU).  It leaves the loop when it got an empty chunk
// and none of its lanes holds a ray.
#pragma once
#include "../../include/wayland_hip.h"
#include "traverse_device.h"

namespace wl
{

// Ray and hit streams are read once and written once: non-temporal accesses
// keep them from displacing BVH nodes in the caches.
typedef float f4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void load_ray_nt(const wl_ray *__restrict__ rays, uint32_t i,
                                            TravRay &r)
{
    const f4v *rp = reinterpret_cast<const f4v *>(rays + i);
    const f4v a = __builtin_nontemporal_load(rp), b = __builtin_nontemporal_load(rp + 1);
    trav_setup(r, a.x, a.y, a.z, b.x, b.y, b.z, a.w, b.w);
}

__device__ __forceinline__ void store_hit_nt(wl_hit *__restrict__ hits, uint32_t i,
                                             const TravResult &h)
{
    const f4v v = { h.t, __uint_as_float(h.prim), h.b1, h.b2 };
    __builtin_nontemporal_store(v, reinterpret_cast<f4v *>(hits) + i);
}

// A wave refills once at least this many of its lanes are idle.
constexpr int kRefillLanes = 16;

// Lanes that must wait for a step before a wave runs it while the other step
// has work (see above).
constexpr int kTriLanes = 16;
constexpr int kNodeLanes = 40;

// Number of lanes in m, kept in a scalar register (a compare of the 64-bit
// count would go to the vector unit).
__device__ __forceinline__ int lane_count(uint64_t m)
{
    int c = __popcll(m);
    asm("" : "+s"(c));
    return c;
}

__device__ __forceinline__ uint32_t lane_prefix(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Chunks of a launch over the whole GPU, a list of them per XCD: the hardware
// deals workgroups round-robin to the 8 XCDs, each with its own L2, so XCD x's
// workgroups are those with blockIdx % 8 == x (the grid is a multiple of 8).
// An XCD's W waves start on its chunks 0 .. W-1 and then each takes chunk W + k,
// k counted by `dyn`, the XCD's counter (dyn_base: its value at launch).
// range(c, next, end): the ray indices [next, end) of the XCD's chunk c, empty
// past its last.  Every wave that had a chunk makes exactly one fetch past the
// XCD's last, so a launch advances the counter by the XCD's number of chunks.
// A wave that got a chunk asks for its next at once (lane 0 holds the answer,
// `ahead`), so the atomic's latency passes behind the chunk's own rays.
template <int BLOCK, class Range>
struct XcdChunks
{
    Range &range;
    uint32_t *dyn;
    uint32_t next_chunk, wavesx, dyn_base, ahead;
    __device__ __forceinline__ XcdChunks(Range &r, uint32_t *d, uint32_t base)
        : range(r), dyn(d),
          next_chunk((blockIdx.x / 8u) * (BLOCK / 64) +
                     __builtin_amdgcn_readfirstlane(threadIdx.x / 64)),
          wavesx((gridDim.x / 8u) * (BLOCK / 64)), dyn_base(base), ahead(0)
    {
    }
    __device__ __forceinline__ void operator()(bool first, uint32_t &next, uint32_t &end)
    {
        range(first ? next_chunk : wavesx + __builtin_amdgcn_readfirstlane(ahead) - dyn_base, next,
              end);
        if (next < end && __lane_id() == 0)
            ahead = atomicAdd(dyn, 1u);
    }
};

// chunks(first, next, end): the wave's next chunk [next, end) of ray indices,
// wave-uniform, empty when there is none left.  fetch(i, TravRay&, root) sets
// up ray i of the current chunk (root: the index of its first node, 0 unless
// several BVHs share the node array); emit(i, const TravRay&, const
// TravResult&) consumes its result.  RAYS: kClosest, kAny, or kMixed, where
// fetch marks any-hit rays with kAnyRay in TravRay::code.  BLOCK must be a
// multiple of 64.
// top / ntop (with TOP): nodes [0, ntop) copied to LDS by the caller (see
// node_visit).
template <int RAYS, int BLOCK, bool WIDE, bool TOP, class Chunks, class Fetch, class Emit>
__device__ __forceinline__ void trav_persistent(const WlBvh8Node *__restrict__ nodes,
                                                const WlTriRecord *__restrict__ tris,
                                                uint32_t *stack, Chunks chunks, Fetch fetch,
                                                Emit emit, const WlBvh8Node *top, uint32_t ntop)
{
    static_assert(BLOCK % 64 == 0, "whole waves only");
    constexpr uint32_t kNone = 0xFFFFFFFFu;
    uint32_t next, end;
    chunks(true, next, end);
    TravRay r;
    trav_setup(r, 0, 0, 0, 1, 0, 0, 0, 0);
    TravState st;
    trav_init(st, r, false, threadIdx.x);
    uint32_t rid = kNone; // the ray whose state or unwritten result this lane holds
    for (;;)
    {
        const uint64_t busy = __ballot(!trav_done(st));
        const uint32_t nidle = (uint32_t)lane_count(~busy);
        if ((next < end && nidle >= (uint32_t)kRefillLanes) || busy == 0)
        {
            const bool idle = trav_done(st);
            if (idle && rid != kNone)
            {
                trav_finish(st.res);
                emit(rid, r, st.res);
                rid = kNone;
            }
            if (next >= end)
                break; // busy == 0: the wave's rays are used up
            if (idle)
            {
                const uint32_t k = next + lane_prefix(~busy);
                if (k < end)
                {
                    rid = k;
                    uint32_t root = 0;
                    fetch(rid, r, root);
                    trav_init(st, r, true, threadIdx.x, root);
                }
            }
            next = next + nidle < end ? next + nidle : end;
            if (next >= end)
                chunks(false, next, end);
        }
        // a lane with a pending triangle takes the triangle step next, any
        // other unfinished lane the node step
        const int nt = lane_count(__ballot(st.trimask != 0));
        const int nn = lane_count(__ballot(st.trimask == 0 && st.grp_mask != 0));
        const bool last = next >= end;
        const bool tri = nt >= kTriLanes || (nt > 0 && (last || nn < kNodeLanes));
        if (tri && st.trimask != 0)
            trav_tri<RAYS, false, WIDE>(tris, r, st);
        const bool can = st.trimask == 0 && st.grp_mask != 0;
        const int nn2 = lane_count(__ballot(can));
        if ((!tri || last || nn2 >= kNodeLanes) && can)
            trav_node<BLOCK, TOP, WIDE>(nodes, r, st, stack, top, ntop);
    }
}

} // namespace wl
