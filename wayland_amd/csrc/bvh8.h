// bvh8.h — in-memory layout of the 8-wide compressed BVH shared by the host
// builder (bvh_builder.cpp) and the gfx950 traversal kernels (traverse.hip).
//
// It replaces the opaque acceleration structure that optixAccelBuild produces
// (src/Backend/Optix/Core/AccelStructure.cpp:133-162).
//
// Node: 128 bytes, one L2 cache line on gfx950, fetched by one lane as eight
// 16-byte loads:
//   bytes   0..11  p[3]        box origin (float)
//   bytes  12..14  e[3]        per-axis scale exponent, scale = 2^(e-127)
//   byte   15      imask       bit s set: slot s is an inner node
//   bytes  16..19  child_base  inner child of slot s lives at child_base + s
//   bytes  20..23  tri_base    first triangle record of this node's leaves
//   bytes  24..27  trivalid    nibble s: the triangles of leaf slot s, bits
//                              0 .. count - 1 (0: inner or empty slot); the
//                              leaves' records follow each other in slot
//                              order from tri_base
//   bytes  28..31  unused
//   bytes  32..127 q[6][8]     quantised child boxes: lo_x, hi_x, lo_y, hi_y,
//                              lo_z, hi_z; plane = p + scale * q, q an
//                              integer 0..2047 held as binary16 (exact), so
//                              gfx950's v_fma_mix_f32 reads it directly.
// Child boxes are rounded outward and padded by one quantum, so the decoded
// box always contains the exact child box.  Empty slots have lo = 65504 (the
// largest finite binary16) and hi = 0, which a near/far-plane slab test never
// hits.
//
// Inner children are addressed as child_base + slot: every node that has an
// inner child owns a group of eight node slots.  That costs node memory for
// unused slots (never fetched) and buys a 4-byte traversal stack entry,
// (child_base / 8) << 8 | remaining-hit-mask, with no node reload on pop.
//
// Slots are assigned per node so that, for a ray whose direction sign bits
// are o (bit k set: d_k < 0), visiting slots in increasing (slot ^ o ^ 7)
// order is approximately front to back (child centroids matched to octant
// directions, Ylitie, Karras, Laine, HPG 2017).
//
// Triangle record: 48 bytes, world-space vertices gathered once at build time
// plus the global primitive id (mesh triangle offset + local index), the
// build input it came from and its index within that input.
#pragma once
#include <stdint.h>

#define WL_BVH8_STACK_DEPTH 32
#define WL_BVH8_SHALLOW_DEPTH 16 // trees up to here: half the stack, more wavefronts
#define WL_BVH8_MAX_LEAF_TRIS 4

struct alignas(16) WlBvh8Node
{
    float p[3];
    uint8_t e[3];
    uint8_t imask;
    uint32_t child_base;
    uint32_t tri_base;
    uint32_t trivalid;
    uint32_t pad_;
    uint16_t q[6][8];
};

struct alignas(16) WlTriRecord
{
    float v0[3];
    float v1[3];
    float v2[3];
    uint32_t prim;
    uint32_t input;
    uint32_t local;
};

static_assert(sizeof(WlBvh8Node) == 128, "BVH8 node must be 128 bytes");
static_assert(sizeof(WlTriRecord) == 48, "triangle record must be 48 bytes");

// The traversal kernels' variants: the short stack (with it the wavefronts and,
// in single-BVH launches, the top levels in LDS) wherever the tree is shallow,
// and byte offsets of 32 bits from a uniform base where they reach every node
// and triangle record; a BVH whose arrays pass 4 GB (89M triangles or 33M node
// slots) takes 64-bit addresses.  Deep trees, which are rare, share one variant.
// All three on the same 2M-triangle scene, in this order: 2^23 closest hits 666 /
// 690 / 831 us, any hits 504 / 525 / 649 us, 1024^2 x 16 spp 10.8 / 11.7 / 12.0 ms.
enum
{
    WL_TRAV_SHORT = 0,      // WL_BVH8_SHALLOW_DEPTH entries, 32-bit offsets
    WL_TRAV_SHORT_WIDE = 1, // WL_BVH8_SHALLOW_DEPTH entries, 64-bit addresses
    WL_TRAV_DEEP = 2        // WL_BVH8_STACK_DEPTH entries, 64-bit addresses
};
static inline uint32_t wl_bvh8_variant(uint32_t depth, uint64_t nodes, uint64_t tris)
{
    const bool narrow = nodes * sizeof(WlBvh8Node) <= (1ull << 32) &&
                        tris * sizeof(WlTriRecord) < (1ull << 32);
    return depth > WL_BVH8_SHALLOW_DEPTH ? WL_TRAV_DEEP
                                         : (narrow ? WL_TRAV_SHORT : WL_TRAV_SHORT_WIDE);
}
