// bvh_builder.cpp — host SAH builder: binned-SAH BVH2, collapse to BVH8 by
// dynamic programming over its subtrees, octant slot ordering and 16-bit
// outward-rounded box quantisation.
// Replaces the closed GPU builder behind optixAccelBuild
// (src/Backend/Optix/Core/AccelStructure.cpp:133-162).
#include "bvh_builder.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <deque>
#include <future>
#include <limits>

namespace wl
{
namespace
{

constexpr int kBins = 32;
// SAH cost of a traversal step relative to one triangle test.  Measured on
// the 2M-triangle soup (closest hit steps one node or one triangle): 0.7
// keeps incoherent closest hit level with 1.0 and makes the path tracer's
// extension and shadow rays 2 % faster (fewer triangle tests per ray).
constexpr double kSahTraversal = 0.7;
constexpr uint32_t kParallelMin = 1u << 16;

struct Aabb
{
    float lo[3] = { INFINITY, INFINITY, INFINITY };
    float hi[3] = { -INFINITY, -INFINITY, -INFINITY };
    void grow(const Aabb &o)
    {
        for (int k = 0; k < 3; ++k)
        {
            lo[k] = std::min(lo[k], o.lo[k]);
            hi[k] = std::max(hi[k], o.hi[k]);
        }
    }
    void grow_point(const float *p)
    {
        for (int k = 0; k < 3; ++k)
        {
            lo[k] = std::min(lo[k], p[k]);
            hi[k] = std::max(hi[k], p[k]);
        }
    }
    double area() const
    {
        double d[3];
        for (int k = 0; k < 3; ++k)
        {
            d[k] = (double)hi[k] - (double)lo[k];
            if (!(d[k] >= 0))
                return 0.0;
        }
        return 2.0 * (d[0] * d[1] + d[1] * d[2] + d[2] * d[0]);
    }
};

struct Node2
{
    Aabb box;
    uint32_t left = 0, right = 0; // inner; both after their parent
    uint32_t first = 0, total = 0; // the subtree's range of prims
    uint32_t count = 0;            // total in a leaf, 0 in an inner node
};

// The cheapest way to hang a BVH2 subtree into an 8-wide node (after Ylitie,
// Karras, Laine, HPG 2017, who follow Aila and others): CollapseCost::k[k - 1] is
// the SAH cost of it as at most k children, k = 1..7.  A single child is a leaf of
// the subtree's triangles or a node of its own; k children are i from the left
// subtree and k - i from the right: nibble k - 2 of `split` holds the i of
// k = 2..7, 0 where k - 1 children cost no more.  The subtree's own node has
// own_k children, own_i of them from the left.
// Against opening the largest child until eight are found: the 2M-triangle soup
// takes 294,000 nodes instead of 497,000 and 5.75 visits a ray instead of 5.89;
// 1080p x 64 spp 35.5 -> 34.7 ms, 1M caustic paths 1.43 -> 1.38 ms, 100,003 rays
// 65 -> 62 us, 2^23 closest hits 680 -> 674 us.  The build takes about 6 % longer
// (2M triangles on 8 CPUs, four builds each twice: 3.7-5.0 -> 4.0-5.3 s).
struct Collapse
{
    uint32_t split : 24, own_k : 4, own_i : 4;
};
struct CollapseCost // while choosing only: the larger part of the two
{
    float k[7];
};
// Cost of a triangle test relative to a node visit: 1.5 and 2.5 are equally
// fast, 1.0 (more triangles per leaf) is 2-3 % slower, 0.6 7 %.
constexpr float kTriCost = 2.0f;

struct Bvh2Builder
{
    const float *tris;
    uint32_t n;
    std::vector<Aabb> pbox;
    std::vector<float> cen;
    std::vector<uint32_t> prims;
    std::vector<Node2> nodes;
    std::atomic<uint32_t> next_node{ 0 };
    std::atomic<int> threads_left{ 0 };

    uint32_t alloc_nodes(uint32_t k) { return next_node.fetch_add(k); }

    void build_range(uint32_t node, uint32_t begin, uint32_t end)
    {
        // iterative on the right child, recursive (maybe async) on the left
        for (;;)
        {
            Node2 &nd = nodes[node];
            Aabb box, cbox;
            for (uint32_t i = begin; i < end; ++i)
            {
                uint32_t p = prims[i];
                box.grow(pbox[p]);
                cbox.grow_point(&cen[3 * (size_t)p]);
            }
            nd.box = box;
            uint32_t cnt = end - begin;
            nd.first = begin;
            nd.total = cnt;
            int best_axis = -1, best_bin = 0;
            double best_cost = std::numeric_limits<double>::infinity();
            double leaf_cost = (double)cnt;
            double parea = box.area();
            if (cnt > 1)
            {
                for (int axis = 0; axis < 3; ++axis)
                {
                    float lo = cbox.lo[axis], hi = cbox.hi[axis];
                    if (!(hi > lo))
                        continue;
                    Aabb bins[kBins];
                    uint32_t counts[kBins] = {};
                    double scale = kBins / ((double)hi - lo);
                    for (uint32_t i = begin; i < end; ++i)
                    {
                        uint32_t p = prims[i];
                        int b = (int)(((double)cen[3 * (size_t)p + axis] - lo) * scale);
                        b = std::min(std::max(b, 0), kBins - 1);
                        counts[b]++;
                        bins[b].grow(pbox[p]);
                    }
                    double rarea[kBins];
                    uint32_t rcnt[kBins];
                    Aabb acc;
                    uint32_t c = 0;
                    for (int b = kBins - 1; b > 0; --b)
                    {
                        acc.grow(bins[b]);
                        c += counts[b];
                        rarea[b] = acc.area();
                        rcnt[b] = c;
                    }
                    acc = Aabb();
                    c = 0;
                    for (int b = 0; b < kBins - 1; ++b)
                    {
                        acc.grow(bins[b]);
                        c += counts[b];
                        if (c == 0 || rcnt[b + 1] == 0)
                            continue;
                        double cost =
                            kSahTraversal + (acc.area() * c + rarea[b + 1] * rcnt[b + 1]) /
                                      (parea > 0 ? parea : 1.0);
                        if (cost < best_cost)
                        {
                            best_cost = cost;
                            best_axis = axis;
                            best_bin = b;
                        }
                    }
                }
            }
            bool make_leaf = cnt <= WL_BVH8_MAX_LEAF_TRIS &&
                             (best_axis < 0 || leaf_cost <= best_cost);
            if (cnt == 0 || make_leaf)
            {
                nd.count = cnt;
                return;
            }
            uint32_t mid;
            if (best_axis >= 0)
            {
                float lo = cbox.lo[best_axis], hi = cbox.hi[best_axis];
                double scale = kBins / ((double)hi - lo);
                auto it = std::partition(
                    prims.begin() + begin, prims.begin() + end, [&](uint32_t p) {
                        int b = (int)(((double)cen[3 * (size_t)p + best_axis] - lo) *
                                      scale);
                        b = std::min(std::max(b, 0), kBins - 1);
                        return b <= best_bin;
                    });
                mid = (uint32_t)(it - prims.begin());
            }
            else
            {
                // all centroids coincide: split the range in half
                mid = begin + cnt / 2;
            }
            if (mid == begin || mid == end)
                mid = begin + cnt / 2;
            uint32_t l = alloc_nodes(2);
            nd.left = l;
            nd.right = l + 1;
            nd.count = 0;
            if (cnt >= kParallelMin && threads_left.fetch_sub(1) > 0)
            {
                auto fut = std::async(std::launch::async,
                                      [this, l, begin, mid] { build_range(l, begin, mid); });
                build_range(l + 1, mid, end);
                fut.get();
                return;
            }
            build_range(l, begin, mid);
            node = l + 1;
            begin = mid;
        }
    }
};

// A box without area, triangles collapsed into a point or a line, counts as this
// in the choice: the cheapest one is then that of the fewest nodes (4096 triangles
// in one point: 1023 nodes at 0, 147 so).
constexpr float kNoArea = 1e-30f;

// The collapse choice of every subtree (children come after their parents);
// subtrees that are cheaper as one leaf become leaves.  Areas are scaled by a
// power of two that puts the root's near 2^64, so that a float holds them, and
// their sums over 2^31 triangles, in any unit (unscaled, all costs were equal at
// coordinates of 1e20 or 1e-23, and a ray took 46 to 60 visits where it takes 24).
std::vector<Collapse> choose_collapse(std::vector<Node2> &nodes, uint32_t n)
{
    std::vector<Collapse> out(n);
    std::vector<CollapseCost> costs(n);
    const double root_area = nodes[0].box.area();
    const double unit = root_area > 0 && std::isfinite(root_area)
                            ? std::ldexp(1.0, 64 - std::ilogb(root_area))
                            : 1.0;
    for (uint32_t i = n; i-- > 0;)
    {
        Node2 &nd = nodes[i];
        Collapse &c = out[i];
        float *cost = costs[i].k;
        const double box_area = nd.box.area() * unit;
        const float area = box_area > 0 ? (float)box_area : kNoArea;
        c.split = 0;
        c.own_k = 0;
        c.own_i = 0;
        if (nd.count > 0 || nd.total == 0)
        {
            std::fill(cost, cost + 7, area * kTriCost * (float)nd.total);
            continue;
        }
        const float *l = costs[nd.left].k, *r = costs[nd.right].k;
        float as[9]; // cost as k children, k = 2..8, and the left subtree's share
        uint32_t share[9];
        for (uint32_t k = 2; k <= 8; ++k)
        {
            float best = INFINITY;
            uint32_t at = 1;
            for (uint32_t j = 1; j < k; ++j)
                if (l[j - 1] + r[k - j - 1] < best)
                {
                    best = l[j - 1] + r[k - j - 1];
                    at = j;
                }
            as[k] = best;
            share[k] = at;
        }
        uint32_t own = 8;
        for (uint32_t k = 7; k >= 2; --k)
            if (as[k] <= as[own])
                own = k;
        c.own_k = own;
        c.own_i = share[own];
        cost[0] = area + as[own];
        const float leaf = area * kTriCost * (float)nd.total;
        if (nd.total <= WL_BVH8_MAX_LEAF_TRIS && leaf <= cost[0])
        {
            cost[0] = leaf;
            nd.count = nd.total;
        }
        for (uint32_t k = 2; k <= 7; ++k)
        {
            const bool fewer = cost[k - 2] <= as[k];
            cost[k - 1] = fewer ? cost[k - 2] : as[k];
            if (!fewer)
                c.split |= share[k] << (4 * (k - 2));
        }
    }
    return out;
}

// The children of node n's 8-wide node under that choice.
void chosen_children(const std::vector<Node2> &nodes, const std::vector<Collapse> &choice,
                     uint32_t n, std::vector<uint32_t> &kids)
{
    struct Part
    {
        uint32_t node, k; // subtree, children it may take
    };
    Part stack[16]; // at most eight parts are open at once
    int sp = 0;
    stack[sp++] = { nodes[n].left, choice[n].own_i };
    stack[sp++] = { nodes[n].right, (uint32_t)(choice[n].own_k - choice[n].own_i) };
    while (sp > 0)
    {
        Part p = stack[--sp];
        const Node2 &nd = nodes[p.node];
        uint32_t at = 0;
        if (nd.count == 0)
            while (p.k > 1 && (at = choice[p.node].split >> (4 * (p.k - 2)) & 0xFu) == 0)
                --p.k;
        if (at == 0) // a child by itself
        {
            kids.push_back(p.node);
            continue;
        }
        stack[sp++] = { nd.left, at };
        stack[sp++] = { nd.right, p.k - at };
    }
}

inline float exp2i(int e) { return std::ldexp(1.0f, e); }

// Quantised planes are integers 0..kQMax, stored as binary16 (exact for
// integers up to 2048): the traversal's fma then takes them as a
// mixed-precision operand with no separate conversion.
constexpr int kQMax = 2047;

// Per-axis exponent so that (hi - p) / 2^e <= kQMax - 2 (the outward
// rounding and one quantum of padding on either side then stay in range).
int choose_exponent(float lo, float hi)
{
    const double room = kQMax - 2;
    double ext = (double)hi - (double)lo;
    if (!(ext > 0))
        return -120;
    int x;
    std::frexp(ext / room, &x); // ext/room = m * 2^x, m in [0.5, 1)
    int e = x;
    if (std::ldexp(1.0, e - 1) >= ext / room)
        e -= 1;
    while (std::ldexp(1.0, e) * room < ext)
        ++e;
    return std::min(std::max(e, -120), 127);
}

// binary16 bits of an integer 0 <= n <= 2047 (exact: 11 significant bits).
uint16_t half_of_int(int n)
{
    if (n <= 0)
        return 0;
    int e = 0;
    while ((n >> (e + 1)) != 0)
        ++e; // 2^e <= n < 2^(e+1), e <= 10
    const uint32_t mant = ((uint32_t)n << (10 - e)) & 0x3FFu;
    return (uint16_t)(((uint32_t)(e + 15) << 10) | mant);
}
constexpr uint16_t kHalfMaxFinite = 0x7BFF; // 65504: the empty slot's lo plane

constexpr size_t kMaxNodes = (size_t)0xFFFFFF * 8; // 24-bit node-group index

// BVH2 -> BVH8 (breadth-first, so the top levels sit together): by `choice`, or
// without one by opening the largest child until there are eight.  Returns the
// SAH cost (node 1, triangle 1).
double collapse_bvh8(const float *tris, uint32_t ntris, const std::vector<Node2> &nodes,
                     const std::vector<uint32_t> &prims, const std::vector<Collapse> *choice,
                     Bvh8Host *out)
{
    out->nodes.clear();
    out->tris.clear();
    // the root owns a group of 8 slots like every other node, so that every
    // child group starts at a multiple of 8 (the stack stores base / 8)
    out->nodes.resize(8);
    out->tris.reserve(ntris);
    out->depth = 1;
    out->inner_nodes = 0;
    out->leaves = 0;
    double root_area = nodes[0].box.area();
    double sah = 0.0;
    struct Work
    {
        uint32_t n2, n8, depth;
    };
    std::deque<Work> queue;
    queue.push_back({ 0, 0, 1 });
    while (!queue.empty())
    {
        Work w = queue.front();
        queue.pop_front();
        out->depth = std::max(out->depth, w.depth);
        out->inner_nodes++;
        const Node2 &src = nodes[w.n2];
        std::vector<uint32_t> kids;
        if (src.count > 0 || ntris == 0)
        {
            if (ntris > 0)
                kids.push_back(w.n2);
        }
        else if (choice)
            chosen_children(nodes, *choice, w.n2, kids);
        else
        {
            kids.push_back(src.left);
            kids.push_back(src.right);
            while (kids.size() < 8)
            {
                int best = -1;
                double best_area = -1.0;
                for (size_t i = 0; i < kids.size(); ++i)
                {
                    const Node2 &k = nodes[kids[i]];
                    if (k.count == 0 && k.box.area() > best_area)
                    {
                        best_area = k.box.area();
                        best = (int)i;
                    }
                }
                if (best < 0)
                    break;
                uint32_t id = kids[best];
                kids[best] = nodes[id].left;
                kids.push_back(nodes[id].right);
            }
        }
        if (root_area > 0)
            sah += src.box.area() / root_area;

        // octant slot assignment (greedy max matching of centroid offsets)
        int slot_of[8];
        for (int i = 0; i < 8; ++i)
            slot_of[i] = -1;
        {
            float pc[3];
            for (int k = 0; k < 3; ++k)
                pc[k] = 0.5f * (src.box.lo[k] + src.box.hi[k]);
            double cost[8][8];
            for (size_t i = 0; i < kids.size(); ++i)
            {
                const Aabb &cb = nodes[kids[i]].box;
                double off[3];
                for (int k = 0; k < 3; ++k)
                    off[k] = 0.5 * ((double)cb.lo[k] + cb.hi[k]) - pc[k];
                for (int s = 0; s < 8; ++s)
                    cost[i][s] = ((s & 1) ? -off[0] : off[0]) +
                                 ((s & 2) ? -off[1] : off[1]) +
                                 ((s & 4) ? -off[2] : off[2]);
            }
            bool slot_used[8] = {};
            for (size_t round = 0; round < kids.size(); ++round)
            {
                double bestc = -INFINITY;
                int bi = -1, bs = -1;
                for (size_t i = 0; i < kids.size(); ++i)
                {
                    if (slot_of[i] >= 0)
                        continue;
                    for (int s = 0; s < 8; ++s)
                        if (!slot_used[s] && cost[i][s] > bestc)
                        {
                            bestc = cost[i][s];
                            bi = (int)i;
                            bs = s;
                        }
                }
                slot_of[bi] = bs;
                slot_used[bs] = true;
            }
        }

        WlBvh8Node node;
        std::memset(&node, 0, sizeof node);
        for (int s = 0; s < 8; ++s)
        {
            for (int k = 0; k < 3; ++k)
            {
                node.q[2 * k][s] = kHalfMaxFinite;
                node.q[2 * k + 1][s] = 0;
            }
        }
        // quantisation frame = this node's box
        const Aabb &nb = src.box;
        float scale[3];
        for (int k = 0; k < 3; ++k)
        {
            float lo = ntris ? nb.lo[k] : 0.0f;
            float hi = ntris ? nb.hi[k] : 0.0f;
            node.p[k] = lo;
            int e = choose_exponent(lo, hi);
            node.e[k] = (uint8_t)(e + 127);
            scale[k] = exp2i(e);
            (void)hi;
        }
        bool any_inner = false;
        for (size_t i = 0; i < kids.size(); ++i)
            if (nodes[kids[i]].count == 0)
                any_inner = true;
        if (any_inner)
        {
            node.child_base = (uint32_t)out->nodes.size();
            out->nodes.resize(out->nodes.size() + 8);
        }
        node.tri_base = (uint32_t)out->tris.size();
        // leaves in slot order
        for (int s = 0; s < 8; ++s)
        {
            int i = -1;
            for (size_t j = 0; j < kids.size(); ++j)
                if (slot_of[j] == s)
                    i = (int)j;
            if (i < 0)
                continue;
            const Node2 &k = nodes[kids[i]];
            for (int a = 0; a < 3; ++a)
            {
                double qlo = std::floor(((double)k.box.lo[a] - node.p[a]) / scale[a]) - 1.0;
                double qhi = std::ceil(((double)k.box.hi[a] - node.p[a]) / scale[a]) + 1.0;
                qlo = std::max(qlo, 0.0);
                qhi = std::min(qhi, (double)kQMax);
                node.q[2 * a][s] = half_of_int((int)qlo);
                node.q[2 * a + 1][s] = half_of_int((int)qhi);
            }
            if (k.count == 0)
            {
                node.imask |= (uint8_t)(1u << s);
                queue.push_back({ kids[i], node.child_base + (uint32_t)s, w.depth + 1 });
            }
            else
            {
                node.trivalid |= ((1u << k.count) - 1u) << (4 * s);
                for (uint32_t t = 0; t < k.count; ++t)
                {
                    uint32_t p = prims[k.first + t];
                    WlTriRecord r;
                    std::memcpy(r.v0, tris + 9 * (size_t)p, 36);
                    r.prim = p;
                    r.input = 0;
                    r.local = p;
                    out->tris.push_back(r);
                }
                out->leaves++;
                if (root_area > 0)
                    sah += k.box.area() / root_area * k.count;
            }
        }
        out->nodes[w.n8] = node;
    }
    return sah;
}

} // namespace

bool build_bvh8(const float *tris, uint32_t ntris, int nthreads, Bvh8Host *out,
                std::string *err)
{
    auto t0 = std::chrono::steady_clock::now();
    Bvh2Builder b;
    b.tris = tris;
    b.n = ntris;
    b.pbox.resize(ntris);
    b.cen.resize(3 * (size_t)ntris);
    b.prims.resize(ntris);
    for (uint32_t i = 0; i < ntris; ++i)
    {
        Aabb a;
        for (int v = 0; v < 3; ++v)
            a.grow_point(tris + 9 * (size_t)i + 3 * v);
        b.pbox[i] = a;
        for (int k = 0; k < 3; ++k)
            b.cen[3 * (size_t)i + k] = 0.5f * (a.lo[k] + a.hi[k]);
        b.prims[i] = i;
    }
    b.nodes.resize(std::max<size_t>(1, 2 * (size_t)ntris));
    b.next_node = 1;
    b.threads_left = std::max(0, nthreads - 1);
    b.build_range(0, 0, ntris);
    // not needed any more, and about as large as the costs of the choice
    std::vector<Aabb>().swap(b.pbox);
    std::vector<float>().swap(b.cen);

    const uint32_t n2 = b.next_node;
    double sah;
    {
        // A tree that the choice makes deeper than the kernels' short stack is
        // also collapsed greedily, and the shallower one is taken: chains of
        // ever smaller triangles, of which the greedy collapse opens the large
        // near ones first, come out either way (300 triangles that shrink by
        // 0.65 each: 34 levels, 24 greedily; 600 that shrink by 0.9: 27, 34
        // greedily, more than the traversal stack holds).
        const std::vector<Collapse> choice = choose_collapse(b.nodes, n2);
        sah = collapse_bvh8(tris, ntris, b.nodes, b.prims, &choice, out);
        const bool fits = out->nodes.size() <= kMaxNodes;
        if (out->depth > WL_BVH8_SHALLOW_DEPTH || !fits)
        {
            for (uint32_t i = 0; i < n2; ++i) // leaves that the choice made
                if (b.nodes[i].left != 0)
                    b.nodes[i].count = 0;
            Bvh8Host greedy;
            const double greedy_sah = collapse_bvh8(tris, ntris, b.nodes, b.prims, nullptr,
                                                    &greedy);
            const bool greedy_fits = greedy.nodes.size() <= kMaxNodes;
            if (greedy_fits != fits ? greedy_fits : greedy.depth < out->depth)
            {
                *out = std::move(greedy);
                sah = greedy_sah;
            }
        }
    }
    out->sah_cost = sah;
    auto t1 = std::chrono::steady_clock::now();
    out->build_seconds = std::chrono::duration<double>(t1 - t0).count();
    if (out->depth > WL_BVH8_STACK_DEPTH)
    {
        if (err)
            *err = "BVH8 depth " + std::to_string(out->depth) +
                   " exceeds the traversal stack depth " +
                   std::to_string(WL_BVH8_STACK_DEPTH);
        return false;
    }
    if (out->nodes.size() > kMaxNodes)
    {
        if (err)
            *err = "BVH8 node count exceeds the 24-bit node-group index";
        return false;
    }
    return true;
}

} // namespace wl
