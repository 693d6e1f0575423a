// traverse_device.h — gfx950 BVH8 traversal, one ray per lane.
//
// Watertight FP32 ray/triangle test (Woop, Benthin, Wald, JCGT 2013) with the
// same operation order as the host oracle: this translation unit is compiled
// with -ffp-contract=off, so every + - * / below rounds separately and the
// division and square root are IEEE correctly rounded.  Box tests use
// explicit fmaf (only the triangle test must match the host bit for bit: the
// box test decides what is visited, never what is hit, because boxes are
// conservative).
//
// Traversal state per lane: a current node group (child_base, hit mask in
// key space), the pending triangles of the node visited last, and an LDS
// stack of 4-byte group entries, WL_BVH8_STACK_DEPTH deep, laid out
// [depth][lane] so the 64 lanes of a wave touch 64 consecutive words.
//
// A ray alternates two steps: trav_node (the next node of the group: eight
// child boxes) while no triangle is pending, and trav_tri (one pending
// triangle).  It is finished once its group and its pending triangles are
// both empty.  trav_run takes one ray to completion (the instrumented kernel,
// the example program, the CPU emulation); the persistent kernels
// (traverse_persistent.h) choose per wave which of the two steps to run.  A
// ray's own steps come in the same order either way, so the results are the
// same.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bvh8.h"

#define WL_INVALID 0xFFFFFFFFu

// Compiled for the device by hipcc and, for the CPU emulation used by the
// tests (hostemu.cpp), for the host.  WL_TRAV_CHECK is empty on the device;
// the host emulation defines it to record out-of-range accesses.
#define WL_HD __host__ __device__ __forceinline__
#ifndef WL_TRAV_CHECK
#define WL_TRAV_CHECK(cond, what) ((void)0)
#endif

namespace wl
{

WL_HD float wl_u2f(uint32_t u) { return __builtin_bit_cast(float, u); }
WL_HD uint32_t wl_f2u(float f) { return __builtin_bit_cast(uint32_t, f); }

// Keeps the compiler from seeing through x: a multiplication written as shifts
// and adds stays that (the 32-bit integer multiply is a quarter-rate
// instruction).
WL_HD uint32_t opaque(uint32_t x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+v"(x));
#endif
    return x;
}

struct TravRay
{
    float o[3];
    float tmin, tmax;
    float inv[3];
    float Sx, Sy, Sz;
    // bits 0-2: visit key, bit k clear for d_k < 0 (slots in increasing
    // slot ^ key order are near first); bits 4-6: bit 4 + k set for d_k < 0
    // (16 x bit = the byte offset of the near plane in its lo / hi pair);
    // bits 8, 9: the largest component is x, y (else z); bit 31: it is < 0;
    // bit 10: kAnyRay
    uint32_t code;
};

WL_HD void trav_setup(TravRay &r, float ox, float oy,
                                           float oz, float dx, float dy,
                                           float dz, float tmin, float tmax)
{
    r.o[0] = ox;
    r.o[1] = oy;
    r.o[2] = oz;
    r.tmin = tmin;
    r.tmax = tmax;
    float d[3] = { dx, dy, dz };
    // axes (kx, ky, kz), kz the largest component of d: y z x, z x y or x y z
    // (the winding swap of kx and ky for d[kz] < 0 is tri_test's sign)
    const bool cy = fabsf(dy) > fabsf(dx);
    const float dm = cy ? dy : dx;
    const bool cz = fabsf(dz) > fabsf(dm);
    const float dkz = cz ? dz : dm;
    const float dkx = cz ? dx : (cy ? dz : dy);
    const float dky = cz ? dy : (cy ? dx : dz);
    r.Sx = dkx / dkz;
    r.Sy = dky / dkz;
    r.Sz = 1.0f / dkz;
    const uint32_t axis = (cz ? 0u : (cy ? 2u << 8 : 1u << 8)) | (dkz < 0.0f ? 1u << 31 : 0u);
    uint32_t neg = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
    {
        float di = d[i];
        if (fabsf(di) < 1e-30f)
            di = copysignf(1e-30f, di);
        // the reciprocals only place box planes, which are padded; the
        // triangle test uses the correctly rounded Sx, Sy, Sz
#if defined(__HIP_DEVICE_COMPILE__)
        r.inv[i] = __builtin_amdgcn_rcpf(di);
#else
        r.inv[i] = 1.0f / di;
#endif
        if (r.inv[i] < 0.0f)
            neg |= 1u << i;
    }
    r.code = (neg ^ 7u) | neg << 4 | axis;
}

// Watertight test; returns true and (t, b1, b2) for tmin <= t <= tmax.
WL_HD bool tri_test(const TravRay &r, const float4 w0,
                                         const float4 w1, const float4 w2,
                                         float tmax, float &t_out, float &b1_out,
                                         float &b2_out)
{
    // A = v0 - o, B = v1 - o, C = v2 - o, subtracted in world axes, then the
    // components permuted to (kx, ky, kz)
    const bool zx = (r.code & 1u << 8) != 0, zy = (r.code & 2u << 8) != 0;
    const float A0 = w0.x - r.o[0], A1 = w0.y - r.o[1], A2 = w0.z - r.o[2];
    const float B0 = w0.w - r.o[0], B1 = w1.x - r.o[1], B2 = w1.y - r.o[2];
    const float C0 = w1.z - r.o[0], C1 = w1.w - r.o[1], C2 = w2.x - r.o[2];
    const float Akx = zx ? A1 : (zy ? A2 : A0), Aky = zx ? A2 : (zy ? A0 : A1),
                Akz = zx ? A0 : (zy ? A1 : A2);
    const float Bkx = zx ? B1 : (zy ? B2 : B0), Bky = zx ? B2 : (zy ? B0 : B1),
                Bkz = zx ? B0 : (zy ? B1 : B2);
    const float Ckx = zx ? C1 : (zy ? C2 : C0), Cky = zx ? C2 : (zy ? C0 : C1),
                Ckz = zx ? C0 : (zy ? C1 : C2);
    // The published test swaps kx and ky where d[kz] < 0, which turns each
    // product pair below round: U = Cx By - Cy Bx becomes Cy Bx - Cx By.
    // Flipping the sign of the three x components gives exactly that,
    // signed zeros included, for three instructions instead of six more
    // selection conditions.
    auto flip = [&](float x) { return wl_u2f(wl_f2u(x) ^ (r.code & 0x80000000u)); };
    const float Ax = flip(Akx - r.Sx * Akz);
    const float Ay = Aky - r.Sy * Akz;
    const float Bx = flip(Bkx - r.Sx * Bkz);
    const float By = Bky - r.Sy * Bkz;
    const float Cx = flip(Ckx - r.Sx * Ckz);
    const float Cy = Cky - r.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f)
    {
        double CxBy = (double)Cx * (double)By, CyBx = (double)Cy * (double)Bx;
        U = (float)(CxBy - CyBx);
        double AxCy = (double)Ax * (double)Cy, AyCx = (double)Ay * (double)Cx;
        V = (float)(AxCy - AyCx);
        double BxAy = (double)Bx * (double)Ay, ByAx = (double)By * (double)Ax;
        W = (float)(BxAy - ByAx);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f))
        return false;
    const float det = U + V + W;
    if (det == 0.0f)
        return false;
    const float Az = r.Sz * Akz;
    const float Bz = r.Sz * Bkz;
    const float Cz = r.Sz * Ckz;
    const float T = U * Az + V * Bz + W * Cz;
    const float rcp = 1.0f / det;
    const float t = T * rcp;
    if (!(t >= r.tmin && t <= tmax))
        return false;
    t_out = t;
    b1_out = V * rcp;
    b2_out = W * rcp;
    return true;
}

// Quantised planes are binary16 halves of a word; the fma that consumes the
// widened value compiles to one v_fma_mix_f32 (conversion folded in).
WL_HD float q_lo16(uint32_t w)
{
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu));
}
WL_HD float q_hi16(uint32_t w)
{
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
}

struct TravResult
{
    float t;
    uint32_t prim;
    float b1, b2;
    uint32_t input, local; // build input and input-local index (AUX only)
};

// Resumable traversal state of one ray: the current node group, the stack
// position, the pending triangles and the best hit so far.  The stack itself
// lives in LDS: sp indexes it as lane + BLOCK x depth.
struct TravState
{
    TravResult res;
    uint32_t grp_base, grp_mask;
    uint32_t sp;
    uint32_t trimask, trivalid, tri_base; // pending triangles (see NodeHits)
};

// Starts (active) at node `root`, the only member of the first group.
WL_HD void trav_init(TravState &st, const TravRay &r, bool active, uint32_t lane,
                     uint32_t root = 0)
{
    st.res.t = r.tmax;
    st.res.prim = WL_INVALID;
    st.res.b1 = 0.0f;
    st.res.b2 = 0.0f;
    st.res.input = WL_INVALID;
    st.res.local = WL_INVALID;
    st.sp = lane;
    st.grp_base = root;
    st.grp_mask = active ? 1u << (r.code & 7u) : 0u; // slot 0's key
    st.trimask = 0;
    st.trivalid = 0;
    st.tri_base = 0;
}

// The eight child boxes of `node` against [tmin, min(t_best, ...)]: inner
// hits in key space (bit s ^ key), and the triangles of the hit leaves: bit
// 4 s + i for triangle i of leaf slot s, whose record is tri_base + the number
// of trivalid bits below it.
struct NodeHits
{
    uint32_t child_base, tri_base, inner, trimask, trivalid;
};

// TOP: nodes [0, ntop) are also held in LDS at `top`, read there instead of
// from memory (the builder lays the top levels out first) with byte offsets of
// 32 bits.  WIDE: 64-bit addresses per lane for the rest; otherwise the same
// offsets from the uniform base (wl_bvh8_variant).
template <bool TOP, bool WIDE>
WL_HD NodeHits node_visit(const WlBvh8Node *__restrict__ nodes, uint32_t node,
                          const TravRay &r, float t_best, const WlBvh8Node *top = nullptr,
                          uint32_t ntop = 0)
{
    // near/far quantised planes chosen by the ray's direction signs: the lo and
    // hi planes of an axis are a 16-byte aligned pair, so a per-lane bit of the
    // address picks one and its complement the other
    const bool in_top = TOP && node < ntop;
    const uint32_t at = WIDE && !in_top ? 0u : node << 7;
    const uint32_t nx = at | (r.code & 16u), ny = at | ((r.code >> 1) & 16u),
                   nz = at | ((r.code >> 2) & 16u);
    uint4 h0, h1, nqx, fqx, nqy, fqy, nqz, fqz;
    auto fetch = [&](auto base, auto as) {
        auto ld = [&](uint32_t off, uint32_t imm) { return *as(base + off + imm); };
        h0 = ld(at, 0);
        h1 = ld(at, 16);
        nqx = ld(nx, 32);
        fqx = ld(nx ^ 16u, 32);
        nqy = ld(ny, 64);
        fqy = ld(ny ^ 16u, 64);
        nqz = ld(nz, 96);
        fqz = ld(nz ^ 16u, 96);
    };
#if defined(__HIP_DEVICE_COMPILE__)
    // distinct address spaces keep the two paths apart: LDS reads for the
    // cached nodes, global loads for the rest (not one generic-pointer load)
    typedef __attribute__((address_space(3))) const uint4 lds_u4;
    typedef __attribute__((address_space(1))) const uint4 glb_u4;
    typedef __attribute__((address_space(3))) const char lds_c;
    typedef __attribute__((address_space(1))) const char glb_c;
    auto as_lds = [](lds_c *p) { return (lds_u4 *)p; };
    auto as_glb = [](glb_c *p) { return (glb_u4 *)p; };
    if (in_top)
        fetch((lds_c *)reinterpret_cast<const char *>(top), as_lds);
    else
        fetch((glb_c *)reinterpret_cast<const char *>(WIDE ? nodes + node : nodes), as_glb);
#else
    auto as_any = [](const char *p) { return reinterpret_cast<const uint4 *>(p); };
    fetch(reinterpret_cast<const char *>(in_top ? top : WIDE ? nodes + node : nodes), as_any);
#endif
    const float px = wl_u2f(h0.x), py = wl_u2f(h0.y), pz = wl_u2f(h0.z);
    const uint32_t ew = h0.w;
    const float sx = wl_u2f((ew & 0xFFu) << 23);
    const float sy = wl_u2f(((ew >> 8) & 0xFFu) << 23);
    const float sz = wl_u2f(((ew >> 16) & 0xFFu) << 23);
    const uint32_t imask = ew >> 24;
    // per-axis plane parameters: t = q * sinv + adj
    const float ax = (px - r.o[0]) * r.inv[0];
    const float ay = (py - r.o[1]) * r.inv[1];
    const float az = (pz - r.o[2]) * r.inv[2];
    const float six = sx * r.inv[0], siy = sy * r.inv[1], siz = sz * r.inv[2];
    const float cull = t_best * 1.00001f;
    const float tmin = r.tmin;
    const uint32_t nxw[4] = { nqx.x, nqx.y, nqx.z, nqx.w };
    const uint32_t fxw[4] = { fqx.x, fqx.y, fqx.z, fqx.w };
    const uint32_t nyw[4] = { nqy.x, nqy.y, nqy.z, nqy.w };
    const uint32_t fyw[4] = { fqy.x, fqy.y, fqy.z, fqy.w };
    const uint32_t nzw[4] = { nqz.x, nqz.y, nqz.z, nqz.w };
    const uint32_t fzw[4] = { fqz.x, fqz.y, fqz.z, fqz.w };
    // all eight tests first, without branches: the hit mask
    uint32_t hitmask = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s)
    {
        const int wi = s >> 1;
        float qnx, qfx, qny, qfy, qnz, qfz;
        if (s & 1)
        {
            qnx = q_hi16(nxw[wi]); qfx = q_hi16(fxw[wi]);
            qny = q_hi16(nyw[wi]); qfy = q_hi16(fyw[wi]);
            qnz = q_hi16(nzw[wi]); qfz = q_hi16(fzw[wi]);
        }
        else
        {
            qnx = q_lo16(nxw[wi]); qfx = q_lo16(fxw[wi]);
            qny = q_lo16(nyw[wi]); qfy = q_lo16(fyw[wi]);
            qnz = q_lo16(nzw[wi]); qfz = q_lo16(fzw[wi]);
        }
        const float tnx = __builtin_fmaf(qnx, six, ax);
        const float tfx = __builtin_fmaf(qfx, six, ax);
        const float tny = __builtin_fmaf(qny, siy, ay);
        const float tfy = __builtin_fmaf(qfy, siy, ay);
        const float tnz = __builtin_fmaf(qnz, siz, az);
        const float tfz = __builtin_fmaf(qfz, siz, az);
        const float tn = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, tmin));
        float tf = fminf(fminf(tfx, tfy), tfz);
        tf = __builtin_fmaf(fabsf(tf), 4e-6f, tf);
        hitmask |= (tn <= fminf(tf, cull)) ? (1u << s) : 0u;
    }
    NodeHits h;
    h.child_base = h1.x;
    h.tri_base = h1.y;
    h.trivalid = h1.z;
    // hit leaves: every slot's bit to a nibble, the nibbles' valid triangles
    uint32_t x = hitmask;
    x = (x | x << 12) & 0x000F000Fu;
    x = (x | x << 6) & 0x03030303u;
    x = (x | x << 3) & 0x11111111u;
    h.trimask = (opaque(x << 4) - x) & h.trivalid;
    // inner hits to key space: bit s -> bit s ^ k (xor of a 3-bit index =
    // swaps of single bits, pairs and nibbles)
    uint32_t m = hitmask & imask;
    const uint32_t k = r.code;
    m = (k & 1u) ? (((m & 0x55u) << 1) | ((m >> 1) & 0x55u)) : m;
    m = (k & 2u) ? (((m & 0x33u) << 2) | ((m >> 2) & 0x33u)) : m;
    m = (k & 4u) ? (((m & 0x0Fu) << 4) | ((m >> 4) & 0x0Fu)) : m;
    h.inner = m;
    return h;
}

// Which rays a traversal takes: closest hit, any hit, or both kinds, the
// any-hit rays marked with kAnyRay in TravRay::code.
enum
{
    kClosest = 0,
    kAny = 1,
    kMixed = 2
};
constexpr uint32_t kAnyRay = 1u << 10;

// Test triangle record i; keeps the closest hit (ties to the smaller
// primitive id).  Returns true for an accepted hit.
template <int RAYS, bool AUX, bool WIDE>
WL_HD bool tri_visit(const WlTriRecord *__restrict__ tris, uint32_t i, const TravRay &r,
                     TravState &st)
{
    const float4 *tp;
    if (WIDE)
        tp = reinterpret_cast<const float4 *>(tris + i);
    else
    {
        const uint32_t i3 = opaque((i << 1) + i);
        tp = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(tris) + (i3 << 4));
    }
    const float4 w0 = tp[0], w1 = tp[1], w2 = tp[2];
    float t, b1, b2;
    // the best hit so far bounds t: closest hit keeps only t <= res.t (ties to
    // the smaller primitive id below); any-hit holds res.t = tmax until its hit
    if (tri_test(r, w0, w1, w2, st.res.t, t, b1, b2))
    {
        const uint32_t prim = wl_f2u(w2.y);
        if (RAYS == kAny || t < st.res.t || (t == st.res.t && prim < st.res.prim))
        {
            st.res.t = t;
            st.res.prim = prim;
            st.res.b1 = b1;
            st.res.b2 = b2;
            if (AUX)
            {
                st.res.input = wl_f2u(w2.z);
                st.res.local = wl_f2u(w2.w);
            }
            return true;
        }
    }
    return false;
}

// A traversal variant (WL_TRAV_*) as template arguments, and f called with that
// of v.
template <int STACK_, bool WIDE_>
struct TravVariant
{
    static constexpr int STACK = STACK_;
    static constexpr bool WIDE = WIDE_;
};
template <class F>
auto with_variant(uint32_t v, F f)
{
    return v == WL_TRAV_SHORT        ? f(TravVariant<WL_BVH8_SHALLOW_DEPTH, false>{})
           : v == WL_TRAV_SHORT_WIDE ? f(TravVariant<WL_BVH8_SHALLOW_DEPTH, true>{})
                                     : f(TravVariant<WL_BVH8_STACK_DEPTH, true>{});
}

// ---- chunks of ray indices (traverse_persistent.h hands them out) ------------
// chunk c of an XCD is [next, end), empty past its last; no chunk after an empty
// one holds a ray.

// Rays of the next launch of a raw trace with `left` to go: the kernels' ray
// indices are 32 bits and run up to 64 past the last one, so a trace of more than
// 2^31 rays takes two launches.
WL_HD uint32_t launch_rays(uint32_t left) { return left < 1u << 31 ? left : 1u << 31; }

// The raw traces: XCD xcd's eighth of n rays is [xcd * ceil(n / 8),
// (xcd + 1) * ceil(n / 8)) clipped to n, so its rays and hits go through one L2.
struct EighthChunks
{
    uint32_t lo, hi, chunk;
    WL_HD EighthChunks(uint32_t n, uint32_t xcd, uint32_t chunk_) : chunk(chunk_)
    {
        const uint32_t n8 = (n + 7u) / 8u;
        lo = xcd * n8 < n ? xcd * n8 : n;
        hi = lo + n8 < n ? lo + n8 : n;
    }
    // what a launch advances the XCD's counter by
    WL_HD uint32_t count() const { return (hi - lo + chunk - 1u) / chunk; }
    WL_HD void operator()(uint32_t c, uint32_t &next, uint32_t &end) const
    {
        const uint64_t s0 = lo + (uint64_t)c * chunk;
        next = (uint32_t)(s0 < hi ? s0 : hi);
        end = (uint32_t)(s0 + chunk < hi ? s0 + chunk : hi);
    }
};

// The entries of a path tracer's queue that an XCD's workgroups take, in blocks
// of BLOCK: block k of the walk is [at(k), at(k) + BLOCK) clipped to limit.
struct QueueWalk
{
    uint32_t base, step, limit;
    WL_HD uint32_t at(uint32_t k) const { return base + k * step; }
};
// A queue without segments (a batch's first, or a sorted one): the blocks are
// dealt to the XCDs in turn.
template <uint32_t BLOCK>
WL_HD QueueWalk dealt_walk(uint32_t n, uint32_t xcd)
{
    return QueueWalk{ xcd * BLOCK, 8u * BLOCK, n };
}

// That queue's traversal: the XCD's blocks in pieces.
template <uint32_t BLOCK>
struct DealtChunks
{
    uint32_t n, xcd, chunk, per;
    WL_HD DealtChunks(uint32_t n_, uint32_t xcd_, uint32_t chunk_)
        : n(n_), xcd(xcd_), chunk(chunk_), per(BLOCK / chunk_)
    {
    }
    WL_HD void operator()(uint32_t c, uint32_t &next, uint32_t &end) const
    {
        const uint64_t s0 = ((uint64_t)(c / per) * 8u + xcd) * BLOCK + (c % per) * chunk;
        next = (uint32_t)(s0 < n ? s0 : n);
        end = (uint32_t)(s0 + chunk < n ? s0 + chunk : n);
    }
};

// A segment's traversal: the chunks of its rays, then those of its shadow rays,
// both from entry lo on in queues of their own.
struct SegmentChunks
{
    uint32_t lo, nrays, nshadow, chunk, ray_chunks;
    WL_HD SegmentChunks(uint32_t lo_, uint32_t nrays_, uint32_t nshadow_, uint32_t chunk_)
        : lo(lo_), nrays(nrays_), nshadow(nshadow_), chunk(chunk_),
          ray_chunks((nrays_ + chunk_ - 1u) / chunk_)
    {
    }
    WL_HD void operator()(uint32_t c, uint32_t &next, uint32_t &end, bool &shadow) const
    {
        shadow = c >= ray_chunks;
        const uint32_t n = shadow ? nshadow : nrays;
        const uint64_t s0 = (uint64_t)(shadow ? c - ray_chunks : c) * chunk;
        next = lo + (uint32_t)(s0 < n ? s0 : n);
        end = lo + (uint32_t)(s0 + chunk < n ? s0 + chunk : n);
    }
};

// Whether the ray has nothing left to do.
WL_HD bool trav_done(const TravState &st) { return (st.grp_mask | st.trimask) == 0; }

// One node: the next of the current group (which must not be empty; no
// triangle may be pending).  Its hit children become the group, with what was
// left of the old one pushed; without any, the group goes on, and once it is
// used up the stack's top is popped.  So the group is empty only when the
// stack is, and a node without inner hits touches the stack at most once.
template <int BLOCK, bool TOP = false, bool WIDE = true>
WL_HD bool trav_node(const WlBvh8Node *__restrict__ nodes, const TravRay &r, TravState &st,
                     uint32_t *lds_stack, const WlBvh8Node *top = nullptr, uint32_t ntop = 0)
{
    const uint32_t pos = __builtin_ctz(st.grp_mask);
    const uint32_t rest = st.grp_mask & (st.grp_mask - 1u);
    const uint32_t node = st.grp_base + (pos ^ (r.code & 7u));
    WL_TRAV_CHECK(node < wl_trav_nodes_bound, "node index");
    const NodeHits h = node_visit<TOP, WIDE>(nodes, node, r, st.res.t, top, ntop);
    st.trimask = h.trimask;
    st.trivalid = h.trivalid;
    st.tri_base = h.tri_base;
    if (h.inner)
    {
        if (rest)
        {
            WL_TRAV_CHECK(st.sp < wl_trav_stack_bound * BLOCK, "stack depth");
            lds_stack[st.sp] = st.grp_base << 5 | rest; // base / 8 in the upper 24 bits
            st.sp += BLOCK;
        }
        st.grp_base = h.child_base;
        st.grp_mask = h.inner;
    }
    else
    {
        st.grp_mask = rest;
        if (rest == 0 && st.sp >= BLOCK)
        {
            st.sp -= BLOCK;
            const uint32_t e = lds_stack[st.sp];
            st.grp_base = e >> 5 & ~7u;
            st.grp_mask = e & 0xFFu;
        }
    }
    return false;
}

// One pending triangle (there must be one).  A hit of an any-hit ray ends it.
template <int RAYS, bool AUX = false, bool WIDE = true>
WL_HD bool trav_tri(const WlTriRecord *__restrict__ tris, const TravRay &r, TravState &st)
{
    const uint32_t b = __builtin_ctz(st.trimask);
    st.trimask &= st.trimask - 1u;
    const uint32_t i = st.tri_base + (uint32_t)__builtin_popcount(st.trivalid & ((1u << b) - 1u));
    WL_TRAV_CHECK(i < wl_trav_tris_bound, "triangle index");
    if (tri_visit<RAYS, AUX, WIDE>(tris, i, r, st) &&
        (RAYS == kAny || (RAYS == kMixed && (r.code & kAnyRay))))
    {
        st.trimask = 0;
        st.grp_mask = 0;
    }
    return false;
}

WL_HD void trav_finish(TravResult &res)
{
    if (res.prim == WL_INVALID)
        res.t = wl_u2f(0x7F800000u); // +inf
}

// Traverse one ray to completion.  lane: the ray's first entry of the stack.
template <int RAYS, bool COUNT, int BLOCK, bool AUX = false, bool TOP = false, bool WIDE = true>
WL_HD TravResult trav_run(const WlBvh8Node *__restrict__ nodes,
                          const WlTriRecord *__restrict__ tris, const TravRay &r, bool active,
                          uint32_t *lds_stack, uint32_t lane, uint32_t &n_nodes,
                          uint32_t &n_tris, const WlBvh8Node *top = nullptr, uint32_t ntop = 0)
{
    TravState st;
    trav_init(st, r, active, lane);
    while (st.grp_mask)
    {
        if (trav_node<BLOCK, TOP, WIDE>(nodes, r, st, lds_stack, top, ntop))
            break; // CPU emulation only: an index out of range
        if (COUNT)
            ++n_nodes;
        while (st.trimask)
        {
            if (COUNT)
                ++n_tris;
            if (trav_tri<RAYS, AUX, WIDE>(tris, r, st))
                break;
        }
    }
    trav_finish(st.res);
    return st.res;
}

} // namespace wl
