// trace.hip -- wavefront path tracer kernels for gfx950.
//
// One camera-sample batch of a Path render runs as
//   traverse(primary) -> shade_primary -> { traverse -> shade }* -> finish -> accumulate
// (primary rays are generated from their index where they are used)
// over ping-pong SoA ray queues (float4 origin|tnear, float4 dir|job,
// float4 attenuation, uint4 job|pixel|sample|depth).  shade appends the rays
// that continue with one atomic per wavefront (ballot + popcount) and writes a
// termination record per light-sample path; accumulate replays the records of
// each pixel in (sample, light sample) order, which is the order the
// reference adds them (fresnel/cpu/TracerPath.cc:141-239), so the image does
// not depend on how paths were scheduled.
#include "rt/isect.h"
#include "rt/shade.h"
#include "kernels/tiles.hip"

namespace fh
{
// >= 3 pushes per level of a 4-wide tree of depth 32 (half the depth of a
// Karras tree over 64-bit keys; the binary packet search pushes one per level)
constexpr uint32_t STACK_MAX = 96;

struct HitT
    {
    float t;
    uint32_t geom;
    uint32_t prim;
    };

__device__ __forceinline__ void slab(v3 o, v3 inv, float lx, float ly, float lz, float hx, float hy, float hz,
                                     float& tmin, float& tmax)
    {
    const float tx0 = (lx - o.x) * inv.x, tx1 = (hx - o.x) * inv.x;
    const float ty0 = (ly - o.y) * inv.y, ty1 = (hy - o.y) * inv.y;
    const float tz0 = (lz - o.z) * inv.z, tz1 = (hz - o.z) * inv.z;
    tmin = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fminf(tz0, tz1));
    tmax = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fmaxf(tz0, tz1));
    }

// Lower bound on the computed distance of any primitive inside a box whose
// slab interval is [tmin, tmax] (see CULL_K).  A box is culled when this
// bound exceeds the closest hit, so every primitive that could still win is
// tested and the result does not depend on the hierarchy or the visiting
// order (but for polyhedra's hits below their bound, CULL_K).  margin = CULL_K
// * 3 * the scene's largest primitive half-extent.
__device__ __forceinline__ float cull_bound(float tmin, float tmax, float margin)
    {
    return tmin - (CULL_K * fmaxf(tmax, 0.0f) + margin);
    }

__device__ __forceinline__ bool better(float t, uint32_t g, uint32_t p, const HitT& b)
    {
    // every comparison evaluated (no short circuit): lane masks, no branches
    const bool lt = t < b.t, eq = t == b.t, g_lt = g < b.geom, g_eq = g == b.geom, p_lt = p < b.prim;
    return lt | (eq & (g_lt | (g_eq & p_lt)));
    }

// Element i of an array in global memory (a direct global load, not a flat one).
typedef float F4v __attribute__((ext_vector_type(4)));
typedef uint32_t U4v __attribute__((ext_vector_type(4)));
typedef uint32_t U2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float4 ldg(const float4* p, size_t i)
    {
    const F4v v = ((const F4v __attribute__((address_space(1)))*)p)[i];
    return make_float4(v.x, v.y, v.z, v.w);
    }
__device__ __forceinline__ uint4 ldg(const uint4* p, size_t i)
    {
    const U4v v = ((const U4v __attribute__((address_space(1)))*)p)[i];
    return make_uint4(v.x, v.y, v.z, v.w);
    }
__device__ __forceinline__ uint2 ldg(const uint2* p, size_t i)
    {
    const U2v v = ((const U2v __attribute__((address_space(1)))*)p)[i];
    return make_uint2(v.x, v.y);
    }
__device__ __forceinline__ void stg(uint2* p, size_t i, uint2 e)
    {
    U2v v = {e.x, e.y};
    ((U2v __attribute__((address_space(1)))*)p)[i] = v;
    }

// Stack with the top SS entries in LDS (interleaved by thread) and the rest
// in a per-thread global region.
template<int SS> struct LdsStack
    {
    uint2* lds;
    uint2* glob;
    uint32_t lstride, gstride;
    uint32_t sp;
    __device__ __forceinline__ void push(uint32_t n, float t, uint32_t& err)
        {
        const uint2 e = make_uint2(n, __float_as_uint(t));
        if (sp < SS)
            lds[sp * lstride] = e;
        else if (sp < STACK_MAX)
            stg(glob, (size_t)(sp - SS) * gstride, e);
        else
            {
            err = 1;
            return;
            }
        sp++;
        }
    // Push the entries whose key is finite, the first argument pair first
    // (sorted by descending key, so the finite ones are the last).  With room
    // in LDS for all three there is no branch: each is written where the next
    // entry goes, and stays when its key is finite.
    __device__ __forceinline__ void push3(uint32_t n3, float k3, uint32_t n2, float k2, uint32_t n1, float k1,
                                          uint32_t& err)
        {
        const float inf = __builtin_huge_valf();
        if (sp + 3 <= SS)
            {
            lds[sp * lstride] = make_uint2(n3, __float_as_uint(k3));
            sp += (k3 < inf) ? 1u : 0u;
            lds[sp * lstride] = make_uint2(n2, __float_as_uint(k2));
            sp += (k2 < inf) ? 1u : 0u;
            lds[sp * lstride] = make_uint2(n1, __float_as_uint(k1));
            sp += (k1 < inf) ? 1u : 0u;
            return;
            }
        if (k3 < inf)
            push(n3, k3, err);
        if (k2 < inf)
            push(n2, k2, err);
        if (k1 < inf)
            push(n1, k1, err);
        }
    __device__ __forceinline__ void pop(uint32_t& n, float& t)
        {
        sp--;
        uint2 e;
        if (sp < SS)
            e = lds[sp * lstride];
        else
            e = ldg(glob, (size_t)(sp - SS) * gstride);
        n = e.x;
        t = __uint_as_float(e.y);
        }
    };

// Stack in private memory (for the diagnostic kernels).
struct LocalStack
    {
    uint2 s[STACK_MAX];
    uint32_t sp;
    __device__ __forceinline__ void push(uint32_t n, float t, uint32_t& err)
        {
        if (sp < STACK_MAX)
            s[sp++] = make_uint2(n, __float_as_uint(t));
        else
            err = 1;
        }
    __device__ __forceinline__ void push3(uint32_t n3, float k3, uint32_t n2, float k2, uint32_t n1, float k1,
                                          uint32_t& err)
        {
        const float inf = __builtin_huge_valf();
        if (k3 < inf)
            push(n3, k3, err);
        if (k2 < inf)
            push(n2, k2, err);
        if (k1 < inf)
            push(n1, k1, err);
        }
    __device__ __forceinline__ void pop(uint32_t& n, float& t)
        {
        sp--;
        n = s[sp].x;
        t = __uint_as_float(s[sp].y);
        }
    };


// Candidate distance of one primitive; TYPES lists the geometry types the
// scene can hold, so a spheres-only traversal compiles without the other
// intersectors (fewer registers, more wavefronts in flight).
template<uint32_t TYPES>
__device__ __forceinline__ bool leaf_test(const GeomDev& g, uint32_t prim, v3 o, v3 d, float tnear, float& t)
    {
    if constexpr (TYPES == T_SPHERES)
        {
        const float4 s = g.a[prim];
        float de;
        bool first;
        return sphere_t(o, d, mk3(s.x, s.y, s.z), s.w, t, de, first) && (tnear < t);
        }
    else
        return intersect_prim<false>(g, prim, o, d, tnear, t, nullptr);
    }

typedef const Node __attribute__((address_space(1))) GlobalNode;

// State of a ray's search of the binary hierarchy (below a tile-list subtree).
struct TraceState
    {
    v3 o, d, inv;
    float tnear;
    float margin;
    HitT best;
    uint32_t node;
    };

// One node visit of the closest-hit search over the binary hierarchy (the
// subtrees of tile lists): the primitives of leaf children are tested, the
// nearer hit inner child is visited next and the farther one pushed.  Returns
// false when the search is complete.  The closest hit is
// the smallest (t, geometry, primitive) over the primitives whose bounds pass
// the slab test with tmax >= tnear; a subtree is culled when the lower bound
// of its primitives' distances (cull_bound) exceeds the closest hit.
template<class Stack, bool COUNT, uint32_t TYPES>
__device__ __forceinline__ bool trace_visit2(const Node* __restrict__ nodes, const GeomDev* __restrict__ geoms,
                                            TraceState& r, Stack& st, uint32_t& n_nodes, uint32_t& n_prims,
                                            uint32_t& err)
    {
    if (r.node == EMPTY)
        return false;
    // global address space: direct global loads instead of flat ones
    const GlobalNode* np = (const GlobalNode*)(nodes + r.node);
    const float4 A = make_float4(np->a_lo.x, np->a_lo.y, np->a_lo.z, np->a_lo.w);
    const float4 B = make_float4(np->a_hi.x, np->a_hi.y, np->a_hi.z, np->a_hi.w);
    const float4 C = make_float4(np->b_box.x, np->b_box.y, np->b_box.z, np->b_box.w);
    const uint4 lk = make_uint4(np->link.x, np->link.y, np->link.z, np->link.w);
    if (COUNT)
        n_nodes++;
    float t0min, t0max, t1min, t1max;
    slab(r.o, r.inv, A.x, A.y, A.z, A.w, B.x, B.y, t0min, t0max);
    slab(r.o, r.inv, B.z, B.w, C.x, C.y, C.z, C.w, t1min, t1max);
    const float c0 = cull_bound(t0min, t0max, r.margin);
    const float c1 = cull_bound(t1min, t1max, r.margin);
    bool h0 = (t0min <= t0max) && (t0max >= r.tnear) && !(c0 > r.best.t);
    bool h1 = (t1min <= t1max) && (t1max >= r.tnear) && !(c1 > r.best.t);
    if (h0 && (lk.x & LEAF))
        {
        const uint32_t prim = lk.x & ~LEAF;
        float t;
        if (COUNT)
            n_prims++;
        if (leaf_test<TYPES>(geoms[lk.z], prim, r.o, r.d, r.tnear, t) && better(t, lk.z, prim, r.best))
            {
            r.best.t = t;
            r.best.geom = lk.z;
            r.best.prim = prim;
            }
        h0 = false;
        }
    if (h1 && (lk.y & LEAF))
        {
        const uint32_t prim = lk.y & ~LEAF;
        float t;
        if (COUNT)
            n_prims++;
        if (leaf_test<TYPES>(geoms[lk.w], prim, r.o, r.d, r.tnear, t) && better(t, lk.w, prim, r.best))
            {
            r.best.t = t;
            r.best.geom = lk.w;
            r.best.prim = prim;
            }
        h1 = false;
        }
    h0 = h0 && !(c0 > r.best.t);
    h1 = h1 && !(c1 > r.best.t);
    if (h0 && h1)
        {
        const bool swap = t1min < t0min;
        st.push(swap ? lk.x : lk.y, swap ? c0 : c1, err);
        r.node = swap ? lk.y : lk.x;
        return true;
        }
    if (h0)
        {
        r.node = lk.x;
        return true;
        }
    if (h1)
        {
        r.node = lk.y;
        return true;
        }
    while (st.sp > 0)
        {
        uint32_t n;
        float tm;
        st.pop(n, tm);
        if (!(tm > r.best.t))
            {
            r.node = n;
            return true;
            }
        }
    r.node = EMPTY;
    return false;
    }

// Intersector of one primitive of type G, if the state's types hold it.
template<uint32_t G, uint32_t TYPES, bool COUNT>
__device__ __forceinline__ void test_binary(const GeomDev* __restrict__ geoms, TraceState& r, uint32_t ty,
                                            uint32_t slot, uint32_t prim, uint32_t& n_prims)
    {
    if constexpr ((TYPES & (1u << G)) != 0)
        if (ty == G)
            {
            float t;
            if (COUNT)
                n_prims++;
            if (intersect_prim<false, 1u << G>(geoms[slot], prim, r.o, r.d, r.tnear, t, nullptr)
                && better(t, slot, prim, r.best))
                {
                r.best.t = t;
                r.best.geom = slot;
                r.best.prim = prim;
                }
            }
    }

// Closest hit of each lane's ray by the binary search from the root: for each
// lane the visits, tests and comparisons of trace_visit2 in the same order,
// but a lane that reaches leaves stops in the middle of its visit until the
// waiting lanes are twice those that can go on, and the primitive tests run
// for all of them, one type at a time (20,000 polyhedra, 1280 x 720, 64
// samples: 18.6 ms with the tests on the spot, 16.8 so).
template<class Stack, bool COUNT, uint32_t TYPES>
__device__ inline void trace_binary(const SceneDev& sc, v3 o, v3 d, float tnear, HitT& best, Stack& st,
                                    uint32_t& n_nodes, uint32_t& n_prims, uint32_t& err)
    {
    const Node* __restrict__ nodes = sc.nodes;
    const GeomDev* __restrict__ geoms = sc.geoms;
    TraceState r;
    r.o = o;
    r.d = d;
    r.inv = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    r.tnear = tnear;
    r.margin = sc.cull_margin;
    r.best.t = __builtin_huge_valf();
    r.best.geom = EMPTY;
    r.best.prim = EMPTY;
    r.node = sc.root;
    st.sp = 0;
    bool wait = false, h0 = false, h1 = false, swap = false;
    float c0 = 0.0f, c1 = 0.0f;
    uint4 lk = make_uint4(0, 0, 0, 0);
    // the rest of a visit once its leaves are tested
    auto advance = [&]()
    {
        const bool a = h0 && !(lk.x & LEAF) && !(c0 > r.best.t);
        const bool b = h1 && !(lk.y & LEAF) && !(c1 > r.best.t);
        if (a && b)
            st.push(swap ? lk.x : lk.y, swap ? c0 : c1, err);
        if (a || b)
            {
            r.node = (b && (!a || swap)) ? lk.y : lk.x;
            return;
            }
        r.node = EMPTY;
        while (st.sp > 0)
            {
            uint32_t n;
            float tm;
            st.pop(n, tm);
            if (!(tm > r.best.t))
                {
                r.node = n;
                return;
                }
            }
    };
    for (;;)
        {
        for (;;)
            {
            const bool go = r.node != EMPTY && !wait;
            const uint32_t n_go = (uint32_t)__popcll(__ballot(go));
            const uint32_t n_wait = (uint32_t)__popcll(__ballot(wait));
            if (n_go == 0 || n_wait >= 2 * n_go)
                break;
            if (go)
                {
                const float4* np = (const float4*)(nodes + r.node);
                const float4 A = ldg(np, 0), B = ldg(np, 1), C = ldg(np, 2);
                lk = ldg((const uint4*)np, 3);
                if (COUNT)
                    n_nodes++;
                float t0min, t0max, t1min, t1max;
                slab(r.o, r.inv, A.x, A.y, A.z, A.w, B.x, B.y, t0min, t0max);
                slab(r.o, r.inv, B.z, B.w, C.x, C.y, C.z, C.w, t1min, t1max);
                c0 = cull_bound(t0min, t0max, r.margin);
                c1 = cull_bound(t1min, t1max, r.margin);
                h0 = (t0min <= t0max) && (t0max >= r.tnear) && !(c0 > r.best.t);
                h1 = (t1min <= t1max) && (t1max >= r.tnear) && !(c1 > r.best.t);
                swap = t1min < t0min;
                wait = (h0 && (lk.x & LEAF)) || (h1 && (lk.y & LEAF));
                if (!wait)
                    advance();
                }
            }
        if (__ballot(wait) == 0)
            break;
        for (uint32_t k = 0; k < 2; k++)
            {
            const uint32_t ref = k ? lk.y : lk.x, slot = k ? lk.w : lk.z;
            const uint32_t ty = (wait && (k ? h1 : h0) && (ref & LEAF)) ? geoms[slot].type : 0xffu;
            const uint32_t prim = ref & ~LEAF;
            test_binary<G_SPHERE, TYPES, COUNT>(geoms, r, ty, slot, prim, n_prims);
            test_binary<G_CYLINDER, TYPES, COUNT>(geoms, r, ty, slot, prim, n_prims);
            test_binary<G_POLYHEDRON, TYPES, COUNT>(geoms, r, ty, slot, prim, n_prims);
            test_binary<G_MESH, TYPES, COUNT>(geoms, r, ty, slot, prim, n_prims);
            test_binary<G_POLYGON, TYPES, COUNT>(geoms, r, ty, slot, prim, n_prims);
            }
        if (wait)
            {
            advance();
            wait = false;
            }
        }
    best = r.best;
    }

// ---------------------------------------------------------------- 4-wide search
// Closest-hit search over the 4-wide hierarchy.  A ray walks the nodes with a
// cheap test that only has to be conservative, and the primitives it reaches
// are tested later, many lanes together:
//   * a child box is 8-bit steps of the node's interval (k_bvh4_fill); the
//     ray's direction signs pick the near and far ends, so an axis of a
//     child's slab interval is two byte conversions and two fmas.  The node's
//     origin less the ray's is one rounding of exact operands, so an end at
//     distance t is off by at most 3 x 2^-24 t, 3 x 2^-24 of the node's width
//     times the reciprocal, and the 2 x 2^-24 t of a primitive's float slab
//     interval (lo - o) * inv; the node's pad (2^-22 of its width and more)
//     and the factor 1 + 2^-19 in the comparison cover them, so every child
//     whose primitives' own test could pass is open;
//   * the exact slab gate of a primitive's own bounds and its intersector run
//     at the leaf step.  Leaf children are sorted and pushed like inner ones;
//     a lane that takes one waits until enough lanes hold one.
// A child is culled when its key, max(tmin, 0 or tnear) - CULL_K tmax, exceeds
// the closest hit plus the scene's margin (cull_bound with the margin moved to
// the other side; CULL_K's factor of two covers the roundings of key and sum;
// a hit lies past tnear, so the larger of the two bounds holds).
// So every primitive whose bounds pass the slab test and whose hit does not lie
// below its own culling bound is tested if it could still win, and the result
// is the smallest (t, geometry, primitive) of those whatever the hierarchy and
// the order.  Only polyhedra have hits below that bound (CULL_K): where one is
// the smallest, this search and the binary one may differ, as either may from
// the checker's.
//
// Bound by VALU issue (99 % on the lattice) with under half the lanes active.
// Exact boxes and leaf tests on the spot took about 450 instructions per
// visit, with a few lanes in the sphere solves; this form takes about 160 per
// visit and 100 per leaf step.  With 128-byte nodes of float centres and half
// extents (seven 16-byte loads per visit instead of four) the loads bound it:
// 11.6 ms on the lattice against 9.2.
//
// What the search reads of a scene.  UNI (one scene for the whole wavefront):
// the pointers are read once, through scalar loads, and stay in scalar
// registers; otherwise each lane reads its own scene's record when it needs
// it, which costs every node visit a load that its node's loads wait for.
template<bool UNI> struct SearchScene;
template<> struct SearchScene<true>
    {
    const Node4* n4;
    const float4* lf;
    const uint2* lr;
    const GeomDev* g;
    __device__ __forceinline__ SearchScene(const SceneDev& s) : n4(s.nodes4), lf(s.leaf), lr(s.leaf_ref), g(s.geoms) { }
    __device__ __forceinline__ const Node4* nodes4() const { return n4; }
    __device__ __forceinline__ const float4* leaf() const { return lf; }
    __device__ __forceinline__ const uint2* leaf_ref() const { return lr; }
    __device__ __forceinline__ const GeomDev* geoms() const { return g; }
    };
template<> struct SearchScene<false>
    {
    const SceneDev& s;
    __device__ __forceinline__ SearchScene(const SceneDev& sc) : s(sc) { }
    __device__ __forceinline__ const Node4* nodes4() const { return s.nodes4; }
    __device__ __forceinline__ const float4* leaf() const { return s.leaf; }
    __device__ __forceinline__ const uint2* leaf_ref() const { return s.leaf_ref; }
    __device__ __forceinline__ const GeomDev* geoms() const { return s.geoms; }
    };

struct Search
    {
    v3 o, d, ic;      // the ray; reciprocals of d, bounded (node_rcp)
    float tnear;
    float margin;
    float cull;       // best.t + margin
    HitT best;        // spheres-only: prim is the leaf position until search_end
    uint32_t cur;     // inner node, LEAF | leaf position, or EMPTY: done
    };

// Reciprocal of a direction component for the node tests.  Below 2^-60 it is
// taken as 2^60: a box the origin lies beside by more than the node's pad is
// missed, and inside one the interval reaches 2^60 times that pad, at least
// 2^36 times the node's largest coordinate, past every hit.
constexpr float RCP_MAX = 0x1p60f;
__device__ __forceinline__ float node_rcp(float d)
    {
    const float inv = 1.0f / d;
    return (fabsf(d) < 1.0f / RCP_MAX) ? copysignf(RCP_MAX, d) : inv;
    }
// The exact reciprocals, for the gate of a primitive's own bounds.
__device__ __forceinline__ v3 exact_rcp(const Search& r)
    {
    v3 i = r.ic;
    if (fabsf(i.x) == RCP_MAX)
        i.x = 1.0f / r.d.x;
    if (fabsf(i.y) == RCP_MAX)
        i.y = 1.0f / r.d.y;
    if (fabsf(i.z) == RCP_MAX)
        i.z = 1.0f / r.d.z;
    return i;
    }

template<class Stack>
__device__ __forceinline__ void search_begin(const SceneDev& sc, v3 o, v3 d, float tnear, Search& r, Stack& st)
    {
    r.o = o;
    r.d = d;
    r.ic = mk3(node_rcp(d.x), node_rcp(d.y), node_rcp(d.z));
    r.tnear = tnear;
    r.margin = sc.cull_margin;
    r.cull = __builtin_huge_valf();
    r.best.t = __builtin_huge_valf();
    r.best.geom = EMPTY;
    r.best.prim = EMPTY;
    r.cur = sc.root;
    st.sp = 0;
    }

// Next entry of the stack that is not culled (EMPTY: the search is complete).
template<class Stack> __device__ __forceinline__ void search_pop(Search& r, Stack& st)
    {
    r.cur = EMPTY;
    while (st.sp > 0)
        {
        uint32_t n;
        float key;
        st.pop(n, key);
        if (!(key > r.cull))
            {
            r.cur = n;
            return;
            }
        }
    }

__device__ __forceinline__ void order2(float& ka, uint32_t& na, float& kb, uint32_t& nb)
    {
    const bool sw = kb < ka;
    const float k = sw ? kb : ka;
    const uint32_t n = sw ? nb : na;
    kb = sw ? ka : kb;
    nb = sw ? na : nb;
    ka = k;
    na = n;
    }

// One node visit: the nearest open child is taken next, the others are pushed,
// farthest first.  The near distance is held at tnear, which a primitive's own
// gate asks its far end to reach, so a ray that leaves a surface does not open
// the boxes it only starts in: in flat systems those are most of them (20,000
// overlapping polygons, 800 x 600, 16 samples: at 0 in place of tnear 89 visits
// a secondary ray and 14.7 ms a call, so 1.0 and 8.6; 10,000 hexagons 2.70 and
// 2.59 ms).  Spheres-only kernels keep 0: their rays' origins lie in few boxes,
// and 4,096 spheres took 2 % more with tnear.
template<class Stack, bool COUNT, uint32_t TYPES>
__device__ __forceinline__ void search_visit(const Node4* __restrict__ nodes, Search& r, Stack& st, uint32_t& n_nodes,
                                             uint32_t& err)
    {
    if (COUNT)
        n_nodes++;
    const uint4* np = (const uint4*)(nodes + r.cur);
    const uint4 A = ldg(np, 0), B = ldg(np, 1), C = ldg(np, 2), ref = ldg(np, 3);
    // A: origin, step x | B: step y z, low x y | C: low z, high x y z
    const float ox = __uint_as_float(A.x), oy = __uint_as_float(A.y), oz = __uint_as_float(A.z);
    const float sx = __uint_as_float(A.w) * r.ic.x, sy = __uint_as_float(B.x) * r.ic.y,
                sz = __uint_as_float(B.y) * r.ic.z;
    const float bx = (ox - r.o.x) * r.ic.x, by = (oy - r.o.y) * r.ic.y, bz = (oz - r.o.z) * r.ic.z;
    const bool px = r.ic.x >= 0.0f, py = r.ic.y >= 0.0f, pz = r.ic.z >= 0.0f;
    const uint32_t qnx = px ? B.z : C.y, qfx = px ? C.y : B.z;
    const uint32_t qny = py ? B.w : C.z, qfy = py ? C.z : B.w;
    const uint32_t qnz = pz ? C.x : C.w, qfz = pz ? C.w : C.x;
    uint32_t nd[4] = {ref.x, ref.y, ref.z, ref.w};
    float key[4];
#pragma unroll
    for (int k = 0; k < 4; k++)
        {
        auto byte = [k](uint32_t q) { return (float)((q >> (8 * k)) & 0xffu); };
        const float tx = __builtin_fmaf(byte(qnx), sx, bx), ux = __builtin_fmaf(byte(qfx), sx, bx);
        const float ty = __builtin_fmaf(byte(qny), sy, by), uy = __builtin_fmaf(byte(qfy), sy, by);
        const float tz = __builtin_fmaf(byte(qnz), sz, bz), uz = __builtin_fmaf(byte(qfz), sz, bz);
        const float lo = fmaxf(fmaxf(fmaxf(tx, ty), tz), TYPES == T_SPHERES ? 0.0f : r.tnear);
        const float hi = fminf(fminf(ux, uy), uz) * (1.0f + 0x1p-19f);
        const float q = __builtin_fmaf(-CULL_K, hi, lo);
        const bool open = (lo <= hi) & !(q > r.cull) & (k < 2 || nd[k] != EMPTY);
        key[k] = open ? q : __builtin_huge_valf();
        }
    order2(key[0], nd[0], key[1], nd[1]);
    order2(key[2], nd[2], key[3], nd[3]);
    order2(key[0], nd[0], key[2], nd[2]);
    order2(key[1], nd[1], key[3], nd[3]);
    order2(key[1], nd[1], key[2], nd[2]);
    if (key[0] < __builtin_huge_valf())
        {
        st.push3(nd[3], key[3], nd[2], key[2], nd[1], key[1], err);
        r.cur = nd[0];
        }
    else
        search_pop(r, st);
    }

// Leaf step of the lanes whose cur is a leaf (in a spheres-only scene): the
// exact slab gate of the sphere's bounds as the builder computes them
// (GeometrySphere.cc:60-73), then the sphere test.
template<bool COUNT, bool UNI>
__device__ __forceinline__ void search_sphere(const SearchScene<UNI>& sc, Search& r, uint32_t& n_prims)
    {
    const uint32_t p = r.cur & ~LEAF;
    const float4 s = ldg(sc.leaf(), p);
    float tmin, tmax;
    slab(r.o, exact_rcp(r), s.x - s.w, s.y - s.w, s.z - s.w, s.x + s.w, s.y + s.w, s.z + s.w, tmin, tmax);
    if (!((tmin <= tmax) && (tmax >= r.tnear)))
        return;
    if (COUNT)
        n_prims++;
    float t, de;
    bool first;
    if (!sphere_t(r.o, r.d, mk3(s.x, s.y, s.z), s.w, t, de, first) || !(r.tnear < t))
        return;
    bool win = t < r.best.t;
    if (t == r.best.t)
        {
        win = true;
        if (r.best.prim != EMPTY)
            {
            const uint2 a = ldg(sc.leaf_ref(), p), b = ldg(sc.leaf_ref(), r.best.prim);
            win = a.x < b.x || (a.x == b.x && a.y < b.y);
            }
        }
    if (win)
        {
        r.best.t = t;
        r.best.prim = p;
        r.cull = t + r.margin;
        }
    }

// Primitive tests of type G: the lanes that hold a primitive of that type run
// its intersector together.
template<uint32_t G, uint32_t TYPES, bool COUNT>
__device__ __forceinline__ void test_type(const GeomDev* __restrict__ geoms, Search& r, uint32_t ty, uint32_t slot,
                                          uint32_t prim, uint32_t& n_prims)
    {
    if constexpr ((TYPES & (1u << G)) != 0)
        if (ty == G)
            {
            float t;
            if (COUNT)
                n_prims++;
            if (intersect_prim<false, 1u << G>(geoms[slot], prim, r.o, r.d, r.tnear, t, nullptr)
                && better(t, slot, prim, r.best))
                {
                r.best.t = t;
                r.best.geom = slot;
                r.best.prim = prim;
                r.cull = t + r.margin;
                }
            }
    }

// Leaf step in other scenes (the leaf array's form depends on the scene:
// kernels of other types are never given a spheres-only scene): the gate with
// the stored bounds, then one geometry type at a time.
template<uint32_t TYPES, bool COUNT, bool UNI>
__device__ __forceinline__ void search_mixed(const SearchScene<UNI>& sc, Search& r, uint32_t& n_prims)
    {
    const uint32_t p = r.cur & ~LEAF;
    const float4 a = ldg(sc.leaf(), 2 * (size_t)p), b = ldg(sc.leaf(), 2 * (size_t)p + 1);
    float tmin, tmax;
    slab(r.o, exact_rcp(r), a.x, a.y, a.z, b.x, b.y, b.z, tmin, tmax);
    if (!((tmin <= tmax) && (tmax >= r.tnear)))
        return;
    const uint32_t slot = __float_as_uint(a.w), prim = __float_as_uint(b.w);
    const uint32_t ty = sc.geoms()[slot].type;
    test_type<G_SPHERE, TYPES, COUNT>(sc.geoms(), r, ty, slot, prim, n_prims);
    test_type<G_CYLINDER, TYPES, COUNT>(sc.geoms(), r, ty, slot, prim, n_prims);
    test_type<G_POLYHEDRON, TYPES, COUNT>(sc.geoms(), r, ty, slot, prim, n_prims);
    test_type<G_MESH, TYPES, COUNT>(sc.geoms(), r, ty, slot, prim, n_prims);
    test_type<G_POLYGON, TYPES, COUNT>(sc.geoms(), r, ty, slot, prim, n_prims);
    }

template<uint32_t TYPES, bool COUNT, bool UNI>
__device__ __forceinline__ void search_leaf(const SearchScene<UNI>& sc, Search& r, uint32_t& n_prims)
    {
    if constexpr (TYPES == T_SPHERES)
        search_sphere<COUNT, UNI>(sc, r, n_prims);
    else
        search_mixed<TYPES, COUNT, UNI>(sc, r, n_prims);
    }

template<uint32_t TYPES, bool UNI>
__device__ __forceinline__ HitT search_end(const SearchScene<UNI>& sc, const Search& r)
    {
    HitT h = r.best;
    if (TYPES == T_SPHERES && h.prim != EMPTY)
        {
        const uint2 id = ldg(sc.leaf_ref(), h.prim);
        h.geom = id.x;
        h.prim = id.y;
        }
    return h;
    }

// Closest hit of one ray per lane.  The wavefront visits nodes until the lanes
// waiting at leaves are at least LEAF_WAIT times those still at inner nodes:
// 1 for spheres (1/4, 1/2, 1, 2: 9.3, 9.1, 9.2, 9.3 ms of traversal on the
// lattice of 1M spheres, 84M rays), 2 for the longer tests of other types
// (1/2, 1, 2, 4: 12.5, 11.4, 10.9, 10.9 ms on the mixed scene of 1.8M
// primitives, 14M rays).
template<class Stack, bool COUNT, uint32_t TYPES, bool UNI>
__device__ inline void trace_closest(const SceneDev& scene, v3 o, v3 d, float tnear, HitT& best, Stack& st,
                                     uint32_t& n_nodes, uint32_t& n_prims, uint32_t& err)
    {
    constexpr uint32_t LEAF_WAIT = TYPES == T_SPHERES ? 1 : 2;
    const SearchScene<UNI> sc(scene);
    Search r;
    search_begin(scene, o, d, tnear, r, st);
    for (;;)
        {
        for (;;)
            {
            const bool inner = !(r.cur & LEAF);
            const uint32_t n_in = (uint32_t)__popcll(__ballot(inner));
            const uint32_t n_leaf = (uint32_t)__popcll(__ballot((r.cur & LEAF) && r.cur != EMPTY));
            if (n_in == 0 || n_leaf >= LEAF_WAIT * n_in)
                break;
            if (inner)
                search_visit<Stack, COUNT, TYPES>(sc.nodes4(), r, st, n_nodes, err);
            }
        const bool leaf = (r.cur & LEAF) && r.cur != EMPTY;
        if (__ballot(leaf) == 0)
            break;
        if (leaf)
            {
            search_leaf<TYPES, COUNT, UNI>(sc, r, n_prims);
            search_pop(r, st);
            }
        }
    best = search_end<TYPES, UNI>(sc, r);
    }

// A ray queue is cut into QSEG segments with one append counter each, the
// counters QSEG_STRIDE words (256 bytes) apart: a producer unit (a claimed
// chunk of a persistent kernel, or a workgroup) appends to segment
// unit % QSEG, so the append atomics spread over QSEG addresses instead of
// queueing on one (one counter's atomic rate bounded the shading kernels).
// Segment s keeps its entries at [s seg_cap, s seg_cap + count_s); the host
// sizes seg_cap from the producers' per-unit output bounds, so no segment can
// overflow (a full segment raises a flag instead of writing past it).
// Consumers see the entries as one dense index range: entry i of the queue
// lives at slot i + adj[s] for the last segment s with pre[s] <= i.
constexpr uint32_t QSEG = 16, QSEG_STRIDE = 64;
constexpr uint32_t QSEG_FLAG = QSEG * QSEG_STRIDE; // overflow flag word after the counters

struct Queue
    {
    float4* o;   // origin, tnear
    float4* d;   // direction, job (bits)
    float4* att; // attenuation
    uint4* meta; // job, pixel, sample-in-batch | light sample << 16, depth
    uint32_t* count;      // producer: append counters (count[s * QSEG_STRIDE]) and flag
    uint32_t seg_cap;     // slots per segment
    uint32_t pre[QSEG];   // consumer: first dense index of each segment
    uint32_t adj[QSEG];   // consumer: slot - index within segment s (s seg_cap - pre[s])
    };

// Consumer view of a queue, written on the device by k_queue_view from its
// producer's segment counters: the entry count, the segment prefix (as
// Queue::pre/adj) and which of the next kernels act on it.  A bounce step's
// kernels all read it, so no count goes back to the host between bounces.
constexpr uint32_t VIEW_IDLE = 0, VIEW_BOUNCE = 1, VIEW_FINISH = 2;
struct QueueView
    {
    uint32_t n;
    uint32_t mode;
    uint32_t pad[2];
    uint32_t pre[QSEG];
    uint32_t adj[QSEG];
    };

// A kernel of `mode` reading a queue: false when it has nothing to do;
// otherwise n and q's segment prefix come from the view (no view: the values
// passed by the host stand).  The view is the same for every thread.
__device__ __forceinline__ bool take_view(const QueueView* __restrict__ view, uint32_t mode, Queue& q, uint32_t& n)
    {
    if (!view)
        return true;
    if (view->mode != mode)
        return false;
    n = view->n;
#pragma unroll
    for (uint32_t s = 0; s < QSEG; s++)
        {
        q.pre[s] = view->pre[s];
        q.adj[s] = view->adj[s];
        }
    return true;
    }

// One wavefront: the consumer view of the queue whose segment counters are
// `count` (filled by the previous producer), then those counters and the
// traversal's work counters cleared for the next producer and consumer.  The
// view's mode is FINISH when at most `tail` entries are left or `force` is
// set, BOUNCE for more, IDLE when the queue is empty or a segment overflowed
// (then CTR_QUEUE_OVERFLOW is raised; the host reports it).  steps[2 step],
// steps[2 step + 1] record the count and mode (pinned host memory).
__global__ __launch_bounds__(64) void k_queue_view(uint32_t* count, uint32_t seg_cap, uint32_t tail, uint32_t force,
                                                   QueueView* view, uint32_t* work, uint32_t* steps, uint32_t step,
                                                   unsigned long long* counters)
    {
    const uint32_t lane = threadIdx.x;
    const uint32_t c = lane < QSEG ? count[lane * QSEG_STRIDE] : 0u;
    const uint32_t flag = count[QSEG_FLAG];
    uint32_t incl = c;
    for (uint32_t off = 1; off < QSEG; off <<= 1)
        {
        const uint32_t t = __shfl_up(incl, off, 64);
        if (lane >= off)
            incl += t;
        }
    const uint32_t total = __shfl(incl, QSEG - 1, 64);
    const bool bad = flag != 0 || __ballot(lane < QSEG && c > seg_cap) != 0;
    const uint32_t mode = (bad || total == 0) ? VIEW_IDLE : ((total <= tail || force) ? VIEW_FINISH : VIEW_BOUNCE);
    if (lane < QSEG)
        {
        const uint32_t pre = incl - c;
        view->pre[lane] = pre;
        view->adj[lane] = lane * seg_cap - pre;
        count[lane * QSEG_STRIDE] = 0u;
        }
    if (lane < 8)
        work[lane * QSEG_STRIDE] = 0u;
    if (lane == 0)
        {
        view->n = total;
        view->mode = mode;
        steps[2 * step] = total;
        steps[2 * step + 1] = mode;
        count[QSEG_FLAG] = 0u;
        if (bad)
            atomicOr((unsigned int*)(counters + CTR_QUEUE_OVERFLOW), 1u);
        }
    }

// slot - index for dense index i (pre is non-decreasing, pre[0] = 0)
__device__ __forceinline__ uint32_t seg_adj(const Queue& q, uint32_t i)
    {
    uint32_t a = 0;
#pragma unroll
    for (uint32_t s = 1; s < QSEG; s++)
        a = (i >= q.pre[s]) ? q.adj[s] : a;
    return a;
    }

// Slot of dense index i, for lanes whose indices lie in [lo, hi] (both
// wavefront-uniform): one scalar offset when the range is in one segment.
__device__ __forceinline__ uint32_t q_slot(const Queue& q, uint32_t i, uint32_t lo, uint32_t hi)
    {
    lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
    hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)hi);
    const uint32_t a = seg_adj(q, lo);
    if (a == seg_adj(q, hi))
        return i + a;
    return i + seg_adj(q, i);
    }

// First slot of a reservation of `total` entries in segment seg, or EMPTY
// (and the flag set) when the segment is full.
__device__ __forceinline__ uint32_t seg_reserve(const Queue& q, uint32_t seg, uint32_t total)
    {
    const uint32_t p = atomicAdd(q.count + seg * QSEG_STRIDE, total);
    if ((uint64_t)p + total <= q.seg_cap)
        return seg * q.seg_cap + p;
    atomicOr(q.count + QSEG_FLAG, 1u);
    return EMPTY;
    }

__device__ __forceinline__ uint32_t lane_id()
    {
    return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    }

// Append slot for lanes with pred set: one atomic per wavefront.  Every lane
// of the wavefront must call it.
__device__ __forceinline__ uint32_t wave_append(bool pred, const Queue& q, uint32_t seg)
    {
    const uint64_t m = __ballot(pred);
    const uint32_t lane = lane_id();
    uint32_t base = EMPTY;
    if (lane == 0 && m)
        base = seg_reserve(q, seg, (uint32_t)__popcll(m));
    base = __shfl(base, 0, 64);
    return (base == EMPTY) ? EMPTY : base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    }

// Append slot in segment seg of q for lanes with pred set (EMPTY if the
// segment is full): one atomic per workgroup of BS threads (wavefront counts
// combined in LDS).  Every thread of the workgroup must call it; sh holds
// BS / 64 + 1 words.
template<int BS>
__device__ __forceinline__ uint32_t block_append(bool pred, const Queue& q, uint32_t seg, uint32_t* sh)
    {
    const uint64_t m = __ballot(pred);
    const uint32_t lane = lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    if (lane == 0)
        sh[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0)
        {
        uint32_t total = 0;
        for (int w = 0; w < BS / 64; w++)
            {
            const uint32_t c = sh[w];
            sh[w] = total;
            total += c;
            }
        sh[BS / 64] = total ? seg_reserve(q, seg, total) : EMPTY;
        }
    __syncthreads();
    const uint32_t b = sh[BS / 64];
    const uint32_t slot = (b == EMPTY) ? EMPTY : b + sh[wave] + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    __syncthreads(); // sh is reused by the next call
    return slot;
    }

// Rank of this thread among the workgroup's threads with `pred` (in thread
// order) and, in `total`, their number.  Every thread must call it.
template<int BS>
__device__ __forceinline__ uint32_t block_rank(bool pred, uint32_t* sh, uint32_t& total)
    {
    const uint64_t m = __ballot(pred);
    const uint32_t lane = lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    if (lane == 0)
        sh[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (uint32_t w = 0; w < BS / 64; w++)
        {
        const uint32_t c = sh[w];
        before += (w < wave) ? c : 0u;
        all += c;
        }
    __syncthreads(); // sh is reused by the next call
    total = all;
    return before + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    }

template<int BS>
__device__ __forceinline__ uint32_t block_max(uint32_t v, uint32_t* sh)
    {
    for (int off = 32; off > 0; off >>= 1)
        v = max(v, (uint32_t)__shfl_xor(v, off, 64));
    if (lane_id() == 0)
        sh[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t r = 0;
    for (int w = 0; w < BS / 64; w++)
        r = max(r, sh[w]);
    __syncthreads();
    return r;
    }

__device__ __forceinline__ uint32_t wave_max(uint32_t v)
    {
    for (int off = 32; off > 0; off >>= 1)
        v = max(v, (uint32_t)__shfl_xor(v, off, 64));
    return v;
    }

__device__ __forceinline__ uint32_t find_job(const JobDev* jobs, uint32_t n_jobs, uint32_t i)
    {
    // last job with ray_base <= i
    uint32_t lo = 0, hi = n_jobs;
    while (hi - lo > 1)
        {
        const uint32_t mid = (lo + hi) >> 1;
        if (jobs[mid].ray_base <= i)
            lo = mid;
        else
            hi = mid;
        }
    return lo;
    }

__device__ __forceinline__ uint4 make_rec(v3 c, uint32_t code)
    {
    return make_uint4(__float_as_uint(c.x), __float_as_uint(c.y), __float_as_uint(c.z), code);
    }

// Termination record of light sample ls of camera sample k at pixel ordinal
// j (the primary order below): chunk-major, [j / 64][k][j % 64][ls], so the
// 64 paths of a wavefront's tile are stored and read back contiguously.
__device__ __forceinline__ uint64_t rec_index(const JobDev& J, uint32_t k, uint32_t j, uint32_t ls)
    {
    return J.rec_base + (((uint64_t)(j >> 6) * J.K + k) * 64u + (j & 63u)) * J.L + ls;
    }


// ---------------------------------------------------------------- traverse
// Persistent threads: each wavefront takes 64 rays at a time from a counter
// until the queue is exhausted.
// Primary ray i of a batch: job, camera sample and pixel from the index
// (fresnel/cpu/TracerPath.cc:100-136, tnear 1e-3).
// Order of a job's primary rays: the image is cut into chunks of 64 pixels
// (8x8 tiles over the largest multiple-of-8 region, then the right and bottom
// strips row by row), and the K samples of a chunk are consecutive.  A
// wavefront therefore traces one sample of one compact tile, and the rays in
// flight at any time cover a K times smaller part of the image than in
// sample-major order.  local in [0, npix K) -> (sample k, pixel px, py).
// Pixel of ordinal j of the primary order (below).
__device__ __forceinline__ void ordinal_pixel(const JobDev& J, uint32_t j, uint32_t& px, uint32_t& py)
    {
    const uint32_t W8 = J.W & ~7u, H8 = J.H & ~7u;
    if (j < W8 * H8)
        {
        const uint32_t tile = j >> 6, within = j & 63u, tiles_x = W8 >> 3;
        const uint32_t ty = fdiv(tile, J.div_tiles); // tile / tiles_x
        px = (tile - ty * tiles_x) * 8u + (within & 7u);
        py = ty * 8u + (within >> 3);
        return;
        }
    uint32_t r = j - W8 * H8;
    const uint32_t rw = J.W - W8;
    if (r < rw * H8)
        {
        py = r / rw;
        px = W8 + (r - py * rw);
        return;
        }
    r -= rw * H8;
    const uint32_t by = r / J.W;
    py = H8 + by;
    px = r - by * J.W;
    }

// Ordinal of pixel (px, py): the inverse of ordinal_pixel.
__device__ __forceinline__ uint32_t pixel_ordinal(const JobDev& J, uint32_t px, uint32_t py)
    {
    const uint32_t W8 = J.W & ~7u, H8 = J.H & ~7u;
    if (px < W8 && py < H8)
        return (((py >> 3) * (W8 >> 3) + (px >> 3)) << 6) | ((py & 7u) << 3) | (px & 7u);
    const uint32_t rw = J.W - W8;
    if (py < H8)
        return W8 * H8 + py * rw + (px - W8);
    return W8 * H8 + rw * H8 + (py - H8) * J.W + px;
    }

// Ordinal of the pixel with raster index `pixel`.
__device__ __forceinline__ uint32_t raster_ordinal(const JobDev& J, uint32_t pixel)
    {
    const uint32_t py = fdiv(pixel, J.div_w);
    return pixel_ordinal(J, pixel - py * J.W, py);
    }

typedef const float __attribute__((address_space(4))) ConstF;
typedef const uint32_t __attribute__((address_space(4))) ConstU;

// Whether chunk c (64 pixels of the primary order, the same for the whole
// wavefront) is a full tile whose candidate list is empty: every ray of its
// pixels misses.  Nothing is traced, shaded or recorded for such a chunk;
// k_accumulate and k_preview take its samples as background.
__device__ __forceinline__ bool empty_chunk(const JobDev& J, uint32_t c)
    {
    if (!J.use_tiles || c >= J.tiles_x * J.tiles_y)
        return false;
    c = (uint32_t)__builtin_amdgcn_readfirstlane((int)c);
    return ((const ConstU*)J.tile_start)[c] == ((const ConstU*)J.tile_end)[c];
    }

__device__ __forceinline__ void primary_order(const JobDev& J, uint32_t local, uint32_t& k, uint32_t& px,
                                              uint32_t& py, uint32_t& j)
    {
    const uint32_t chunk = fdiv(local, J.div_chunk); // local / (64 K)
    const uint32_t rem = local - chunk * 64u * J.K;
    const uint32_t size = min(64u, J.npix - chunk * 64u);
    k = (size == 64u) ? (rem >> 6) : rem / size;
    j = chunk * 64u + (rem - k * size);
    ordinal_pixel(J, j, px, py);
    }

// Primary ray i of job J (the job whose ray range holds i).
__device__ __forceinline__ void primary_ray_of(const JobDev& J, uint32_t i, uint32_t& k, uint32_t& px, uint32_t& py,
                                               uint32_t& jord, v3& o, v3& d)
    {
    primary_order(J, i - J.ray_base, k, px, py, jord);
    camera_ray(J.cam, J.W, J.H, J.xs_off, J.inv_h, J.seed, px, py, J.n_base + k + 1, true, o, d);
    }

__device__ __forceinline__ void primary_ray(const JobDev* __restrict__ jobs, uint32_t n_jobs, uint32_t i, uint32_t& job,
                                            uint32_t& k, uint32_t& px, uint32_t& py, uint32_t& jord, v3& o, v3& d)
    {
    job = find_job(jobs, n_jobs, i);
    primary_ray_of(jobs[job], i, k, px, py, jord, o, d);
    }

__device__ __forceinline__ void primary_ray(const JobDev* __restrict__ jobs, uint32_t n_jobs, uint32_t i, uint32_t& job,
                                            uint32_t& k, uint32_t& pixel, uint32_t& jord, v3& o, v3& d)
    {
    uint32_t px, py;
    primary_ray(jobs, n_jobs, i, job, k, px, py, jord, o, d);
    pixel = py * jobs[job].W + px;
    }

// Persistent traversal: each wavefront claims `chunk` rays (a multiple of 64)
// per atomic on the work counter and claims its next chunk before tracing the
// current one, so the atomic's round trip overlaps the traversal.
// Work claims of the persistent traversal.  Without bands the wavefronts
// claim `chunk` rays at a time from [0, n).  With bands the queue's 16
// segments hold the rays of 16 image bands (k_primary) and the dense range is
// cut into 8 ranges of two segments, one per XCD: a workgroup starts on the
// range of the XCD it runs on (workgroups are dispatched to the 8 XCDs in
// turn) and moves to the next range once its own is exhausted, so each XCD's
// L2 mostly serves the hierarchy around two bands.  Each range's counter only
// grows, so every wavefront stops after at most 8 exhausted ranges.
struct Claims
    {
    uint32_t* work; // one counter per range, QSEG_STRIDE words apart
    uint32_t chunk, n, r, ranges, tried;
    // q.pre[2 k] (constant indices only, so the prefix stays in registers)
    __device__ __forceinline__ static uint32_t even_pre(const Queue& q, uint32_t k)
        {
        uint32_t v = 0;
#pragma unroll
        for (uint32_t j = 1; j < QSEG / 2; j++)
            v = (k == j) ? q.pre[2 * j] : v;
        return v;
        }
    __device__ __forceinline__ uint32_t lo(const Queue& q, uint32_t k) const
        {
        return ranges == 1 ? 0u : even_pre(q, k);
        }
    __device__ __forceinline__ uint32_t hi(const Queue& q, uint32_t k) const
        {
        return (ranges == 1 || k == ranges - 1) ? n : even_pre(q, k + 1);
        }
    // next claimed [base, end) of the calling wavefront, or base = EMPTY
    __device__ __forceinline__ void next(const Queue& q, uint32_t lane, uint32_t& base, uint32_t& end)
        {
        while (tried < ranges)
            {
            uint32_t c = 0;
            if (lane == 0)
                c = atomicAdd(work + r * QSEG_STRIDE, chunk);
            c = __shfl(c, 0, 64);
            const uint32_t a = lo(q, r), b = hi(q, r);
            if (c < b - a)
                {
                base = a + c;
                end = min(b, base + chunk);
                return;
                }
            r = (r + 1 == ranges) ? 0u : r + 1;
            tried++;
            }
        base = EMPTY;
        end = EMPTY;
        }
    };

// Each wavefront searches 64 rays at a time and takes new ones as soon as
// `refill` lanes are idle, so lanes do not wait for the longest ray of 64.  A
// wavefront's rays belong to one job at a time (nearly all chunks do: the
// queues are filled chunk by chunk), whose scene pointers are scalar.  Bound
// by VALU issue and the latency of node and leaf loads.  Traversal per call
// with 64 rays at a time to their ends, and so: lattice of 1M spheres 9.0 and
// 8.3 ms, small scene 0.55 and 0.36, meshes 9.1 and 6.0, mixed 9.5 and 5.9,
// spherocylinders 2.2 and 1.0 (refill at 16, 24, 32, 40 idle lanes: lattice
// 8.8, 8.7, 8.4, 8.1, meshes 6.1, 6.0, 6.2, 6.3, mixed 5.95, 5.98, 6.01, 6.19:
// 32 serves both kernels, spheres alone would take 40).
// Held to 7 wavefronts per SIMD in spheres-only scenes (6: lattice 8.8; 8
// spills), 6 otherwise (5: mixed 6.4, 7: meshes 7.5 against 6.9 then).
template<int BLOCK, int SS, bool COUNT, bool PRIMARY, uint32_t TYPES>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(TYPES == T_SPHERES ? 7 : 6))) void k_traverse(
    const JobDev* __restrict__ jobs, uint32_t n_jobs, Queue q, uint32_t n, const QueueView* __restrict__ view,
    uint4* hits, uint32_t* work, uint32_t chunk, uint32_t bands, uint32_t refill, uint2* gstack, uint32_t gstride,
    unsigned long long* counters)
    {
    if (!take_view(view, VIEW_BOUNCE, q, n))
        return;
    constexpr uint32_t LEAF_WAIT = TYPES == T_SPHERES ? 1 : 2;
    __shared__ uint2 lds[SS * BLOCK];
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    LdsStack<SS> st;
    st.lds = lds + threadIdx.x;
    st.lstride = BLOCK;
    st.glob = gstack + gtid;
    st.gstride = gstride;
    st.sp = 0;
    const uint32_t lane = lane_id();
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t n_nodes = 0, n_prims = 0, err = 0, n_rays = 0;
    Claims cl;
    cl.work = work;
    // at least eight claims a wavefront, down to 64 rays each: a launch of a few
    // million rays in claims of 256 leaves half the wavefronts without work
    // (claims of 256: small scene 0.48 ms, meshes 7.0, mixed 6.5; two, four,
    // eight, sixteen claims a wavefront: mixed 6.05, 6.01, 5.86, 5.75, lattice
    // 8.35, 8.40, 8.35, 8.42)
    const uint32_t share = n / (gridDim.x * (BLOCK / 64) * 8);
    cl.chunk = max(64u, min(chunk, share & ~63u));
    cl.n = n;
    cl.ranges = (bands && !PRIMARY) ? 8u : 1u;
    cl.r = (cl.ranges == 8u) ? (blockIdx.x & 7u) : 0u;
    cl.tried = 0;
    uint32_t pool, pool_end; // untaken rays of the wavefront's chunk; the next chunk is claimed ahead
    uint32_t next, next_end;
    cl.next(q, lane, pool, pool_end);
    cl.next(q, lane, next, next_end);
    uint32_t job = 0; // of every ray the wavefront holds
    Search r;
    r.cur = EMPTY;
    uint32_t i = EMPTY; // the lane's ray (EMPTY: none)
    for (;;)
        {
        // store finished rays, take new ones
        const uint32_t n_idle = (uint32_t)__popcll(__ballot(r.cur == EMPTY));
        const bool stop = n_idle >= refill || n_idle == 64;
        const SearchScene<true> done(jobs[job].scene);
        if (stop && r.cur == EMPTY && i != EMPTY)
            {
            const HitT h = search_end<TYPES, true>(done, r);
            hits[i] = make_uint4(__float_as_uint(h.t), h.geom, h.prim, 0);
            i = EMPTY;
            if (COUNT)
                n_rays++;
            }
        bool blocked = false; // the next unclaimed ray belongs to another job
        while (stop && pool != EMPTY && !blocked)
            {
            const uint64_t need = __ballot(i == EMPTY);
            if (need == 0)
                break;
            const uint32_t avail = pool_end - pool;
            const uint32_t rank = (uint32_t)__popcll(need & below);
            const bool take = i == EMPTY && rank < avail;
            uint32_t took = min((uint32_t)__popcll(need), avail);
            v3 o = mk3(0, 0, 0), d = mk3(0, 0, 1);
            float tnear = 1e-3f;
            uint32_t j = 0;
            if (take)
                {
                if (PRIMARY)
                    {
                    uint32_t k, pixel, jord;
                    primary_ray(jobs, n_jobs, pool + rank, j, k, pixel, jord, o, d);
                    }
                else
                    {
                    const uint32_t sl = q_slot(q, pool + rank, pool, pool_end - 1u);
                    const float4 a = q.o[sl];
                    const float4 b = q.d[sl];
                    o = mk3(a.x, a.y, a.z);
                    d = mk3(b.x, b.y, b.z);
                    tnear = a.w;
                    j = __float_as_uint(b.w);
                    }
                }
            bool mine = take;
            if (n_jobs > 1)
                {
                // rays of one job at a time: an idle wavefront takes its first
                // ray's job, the rays before the first of another job are taken
                const uint32_t first = (uint32_t)(__ffsll((unsigned long long)need) - 1);
                if (need == ~0ull)
                    job = (uint32_t)__builtin_amdgcn_readlane((int)j, first);
                const uint64_t other = __ballot(take && j != job);
                if (other != 0)
                    {
                    blocked = true;
                    took = (uint32_t)__popcll(need & ((other & (~other + 1ull)) - 1ull));
                    mine = take && rank < took;
                    }
                }
            if (mine)
                {
                i = pool + rank;
                search_begin(jobs[job].scene, o, d, tnear, r, st);
                }
            pool += took;
            if (pool == pool_end)
                {
                pool = next;
                pool_end = next_end;
                if (next != EMPTY)
                    cl.next(q, lane, next, next_end);
                }
            }
        if (__ballot(r.cur != EMPTY) == 0)
            {
            if (__ballot(i != EMPTY) == 0)
                break;
            continue; // rays of an empty scene: stored above
            }
        const SearchScene<true> sc(jobs[job].scene);
        const bool more = pool != EMPTY && !blocked;
        uint32_t n_in, n_leaf;
        for (;;)
            {
            const bool inner = !(r.cur & LEAF);
            n_in = (uint32_t)__popcll(__ballot(inner));
            n_leaf = (uint32_t)__popcll(__ballot((r.cur & LEAF) && r.cur != EMPTY));
            if (n_in == 0 || n_leaf >= LEAF_WAIT * n_in || (more && n_in + n_leaf + refill <= 64))
                break;
            if (inner)
                search_visit<LdsStack<SS>, COUNT, TYPES>(sc.nodes4(), r, st, n_nodes, err);
            }
        if (n_leaf != 0 && n_leaf >= LEAF_WAIT * n_in)
            if ((r.cur & LEAF) && r.cur != EMPTY)
                {
                search_leaf<TYPES, COUNT, true>(sc, r, n_prims);
                search_pop(r, st);
                }
        }
    if (COUNT)
        {
        const int c = PRIMARY ? CTR_PRIMARY : CTR_SECONDARY;
        atomicAdd(counters + c + 0, (unsigned long long)n_rays);
        atomicAdd(counters + c + 1, (unsigned long long)n_nodes);
        atomicAdd(counters + c + 2, (unsigned long long)n_prims);
        }
    if (err)
        atomicOr((unsigned int*)(counters + CTR_OVERFLOW), 1u);
    }

// ---------------------------------------------------------------- shading
// Shading attributes of the closest hit: re-evaluate the winning primitive.
template<uint32_t TYPES = T_ALL>
__device__ __forceinline__ void hit_attributes(const SceneDev& sc, const HitT& h, v3 o, v3 d, float tnear, Attr& at,
                                               const GeomDev*& g)
    {
    g = sc.geoms + h.geom;
    if (TYPES == T_SPHERES || g->type == G_SPHERE)
        {
        // the search's t is the sphere solve's: no second solve
        // (GeometrySphere.cc:81-117 attributes, unflipped Ng)
        const float4 s = g->a[h.prim];
        const v3 p = xyz(s);
        const v3 w = cross(p - o, d);
        at.Ng = mk3(o.x + h.t * d.x - p.x, o.y + h.t * d.y - p.y, o.z + h.t * d.z - p.z);
        at.d = s.w - sqrtf(dot(w, w));
        at.color = ld3(g->color, h.prim);
        return;
        }
    float t2;
    intersect_prim<true, TYPES>(*g, h.prim, o, d, tnear, t2, &at);
    }

// Depth-0 shading: one primary hit spawns the L light-sample paths
// (fresnel/cpu/TracerPath.cc:141-155 reuse the cached primary hit).
// Depth-0 shading of a workgroup's primary hits: each hit spawns the job's L
// light-sample paths (fresnel/cpu/TracerPath.cc:141-155 reuse the cached
// primary hit); continuing paths are appended to `out` with one atomic per
// workgroup and light sample, terminated ones write their record.  Every
// thread of the workgroup must call it.
template<int BS, uint32_t TYPES>
__device__ __forceinline__ void shade_primary_block(const JobDev* __restrict__ jobs, bool valid, uint32_t job,
                                                    uint32_t k, uint32_t pixel, uint32_t jord, v3 o, v3 d,
                                                    const HitT& h,
                                                    const Queue& out, uint32_t seg, uint4* records, uint32_t* sh)
    {
    const float tnear = 1e-3f;
    uint32_t L = 0;
    const JobDev& J = jobs[job];
    if (valid)
        {
        L = J.L;
        if (h.geom == EMPTY)
            {
            // primary miss: background for the whole camera sample (TracerPathMethods.h:44-49)
            records[rec_index(J, k, jord, 0)] = make_rec(mk3(0, 0, 0), REC_BG);
            L = 0;
            }
        }
    Attr at;
    const GeomDev* g = nullptr;
    const Mat* m = nullptr;
    if (L)
        {
        hit_attributes<TYPES>(J.scene, h, o, d, tnear, at, g);
        m = (at.d >= g->outline_width) ? &g->mat : &g->outline;
        }
    const uint32_t Lmax = block_max<BS>(L, sh);
    const uint32_t n_sample = valid ? J.n_base + k + 1 : 0;
    for (uint32_t ls = 0; ls < Lmax; ls++)
        {
        bool cont = false;
        v3 att = mk3(1.0f, 1.0f, 1.0f), no, nd, add;
        if (ls < L)
            {
            bool addv;
            cont = path_hit(*m, at, o, d, h.t, pixel, J.seed, 0, (n_sample - 1) * J.L + ls, att, no, nd, add, addv);
            if (!cont)
                records[rec_index(J, k, jord, ls)] = make_rec(addv ? add : mk3(0, 0, 0), addv ? REC_ADD : REC_NONE);
            }
        const uint32_t slot = block_append<BS>(cont, out, seg, sh);
        if (cont && slot != EMPTY)
            {
            out.o[slot] = make_float4(no.x, no.y, no.z, 1e-3f);
            out.d[slot] = make_float4(nd.x, nd.y, nd.z, __uint_as_float(job));
            out.att[slot] = make_float4(att.x, att.y, att.z, 0.0f);
            out.meta[slot] = make_uint4(job, pixel, k | (ls << 16), 1);
            }
        }
    }

template<int BS, uint32_t TYPES>
__global__ __launch_bounds__(BS) void k_shade_primary(const JobDev* __restrict__ jobs, uint32_t n_jobs,
                                                      const uint4* __restrict__ hits, uint32_t n, Queue out,
                                                      uint4* records)
    {
    __shared__ uint32_t sh[BS / 64 + 1];
    const uint32_t i = blockIdx.x * BS + threadIdx.x;
    const bool valid = i < n;
    uint32_t job = 0, pixel = 0, k = 0, jord = 0;
    HitT h;
    h.geom = EMPTY;
    v3 o = mk3(0, 0, 0), d = mk3(0, 0, 1);
    if (valid)
        {
        // the primary ray is regenerated rather than stored (bit-identical)
        primary_ray(jobs, n_jobs, i, job, k, pixel, jord, o, d);
        const uint4 hh = hits[i];
        h.t = __uint_as_float(hh.x);
        h.geom = hh.y;
        h.prim = hh.z;
        }
    shade_primary_block<BS, TYPES>(jobs, valid, job, k, pixel, jord, o, d, h, out, blockIdx.x % QSEG, records, sh);
    }

// Shade one hit or miss of a path at depth >= 1.  Returns true when the path
// continues with (no, nd, att); otherwise rec holds its termination record.
template<uint32_t TYPES>
__device__ inline bool shade_bounce(const JobDev& J, const HitT& h, v3 o, v3 d, float tnear, uint32_t pixel,
                                    uint32_t k, uint32_t ls, uint32_t depth, v3& att, v3& no, v3& nd, uint4& rec)
    {
    if (h.geom == EMPTY)
        {
        // miss: lights whose cone contains the direction (TracerPathMethods.h:50-73)
        rec = make_rec(att, REC_LIGHTS | (light_mask(J.lights, d) << 2));
        return false;
        }
    Attr at;
    const GeomDev* g;
    hit_attributes<TYPES>(J.scene, h, o, d, tnear, at, g);
    const Mat& m = (at.d >= g->outline_width) ? g->mat : g->outline;
    const uint32_t n_sample = J.n_base + k + 1;
    v3 add;
    bool addv;
    const bool cont = path_hit(m, at, o, d, h.t, pixel, J.seed, depth, (n_sample - 1) * J.L + ls, att, no, nd, add,
                               addv);
    if (!cont)
        rec = make_rec(addv ? add : mk3(0, 0, 0), addv ? REC_ADD : REC_NONE);
    return cont;
    }

// Shade the queued hit h of job J (ray o, d from tnear, entry meta mt, path
// attenuation att): returns whether its path continues with (no, nd, att); a
// terminated path's record is written.
template<uint32_t TYPES>
__device__ __forceinline__ bool shade_queued(const JobDev& J, const HitT& h, v3 o, v3 d, float tnear, const uint4& mt,
                                             uint4* records, uint32_t max_depth, unsigned long long* counters,
                                             v3& att, v3& no, v3& nd)
    {
    const uint32_t k = mt.z & 0xffffu, ls = mt.z >> 16;
    uint4 rec;
    bool cont = shade_bounce<TYPES>(J, h, o, d, tnear, mt.y, k, ls, mt.w, att, no, nd, rec);
    if (cont && mt.w + 1 >= max_depth)
        {
        // depth cap (the reference has none): stop without contribution
        cont = false;
        rec = make_rec(mk3(0, 0, 0), REC_NONE);
        atomicAdd(counters + CTR_CAPPED, 1ull);
        }
    if (!cont)
        records[rec_index(J, k, raster_ordinal(J, mt.y), ls)] = rec;
    return cont;
    }

// Hit list of one shading unit: queue index, slot, geometry, primitive and
// distance of each ray that hit, in queue order.
template<int BS>
struct ShadeLds
    {
    uint4 ent[BS];
    float t[BS];
    uint32_t sh[BS / 64 + 1];
    };

// Shade the BS queued rays of `unit`.  A ray that missed ends on its own
// thread with its lights record; the rays that hit are listed in LDS in queue
// order and shaded by the workgroup's first threads, so a wavefront's lanes
// all run the surface interaction (on a lattice of spheres most bounce rays
// escape, and a wavefront of mixed rays would run it with few lanes).  The
// continuing paths are appended to segment unit % QSEG in queue order.  Each
// path's arithmetic depends only on its own entry, so the result is the same
// as shading every ray on its own thread.  A wavefront whose entries all
// belong to one job (every one of a single-job batch, most of a multi-job
// one, whose queues are filled chunk by chunk) reads the job record through
// scalar loads; otherwise each ray reads its own job's record.  Every thread
// of the workgroup must call it.
template<int BS, uint32_t TYPES>
__device__ __forceinline__ void shade_unit(const JobDev* __restrict__ jobs, uint32_t n_jobs, const Queue& in,
                                           uint32_t n, uint32_t unit, const uint4* __restrict__ hits,
                                           const Queue& out, uint4* records, uint32_t max_depth,
                                           unsigned long long* counters, ShadeLds<BS>& L)
    {
    const uint32_t first = unit * BS;
    const uint32_t i = first + threadIdx.x;
    const uint32_t sl = q_slot(in, i, first, min(n, first + BS) - 1u);
    bool hit = false;
    uint4 hh = make_uint4(0, 0, 0, 0);
    if (i < n)
        {
        hh = hits[i];
        hit = hh.y != EMPTY;
        if (!hit)
            {
            // miss: lights whose cone contains the direction (TracerPathMethods.h:50-73)
            const uint4 mt = in.meta[sl];
            const float4 b = in.d[sl];
            const float4 a4 = in.att[sl];
            const uint32_t j0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)mt.x);
            const JobDev& J = (n_jobs == 1 || __ballot(mt.x != j0) == 0) ? jobs[j0] : jobs[mt.x];
            const uint32_t k = mt.z & 0xffffu, ls = mt.z >> 16;
            records[rec_index(J, k, raster_ordinal(J, mt.y), ls)] =
                make_rec(mk3(a4.x, a4.y, a4.z), REC_LIGHTS | (light_mask(J.lights, mk3(b.x, b.y, b.z)) << 2));
            }
        }
    uint32_t n_hit;
    const uint32_t pos = block_rank<BS>(hit, L.sh, n_hit);
    if (hit)
        {
        L.ent[pos] = make_uint4(i, sl, hh.y, hh.z);
        L.t[pos] = __uint_as_float(hh.x);
        }
    __syncthreads();
    bool cont = false;
    v3 att, no, nd;
    uint4 mt = make_uint4(0, 0, 0, 0);
    if (threadIdx.x < n_hit)
        {
        const uint4 e = L.ent[threadIdx.x];
        HitT h;
        h.t = L.t[threadIdx.x];
        h.geom = e.z;
        h.prim = e.w;
        const uint32_t hs = e.y;
        mt = in.meta[hs];
        const float4 a = in.o[hs];
        const float4 b = in.d[hs];
        const float4 at4 = in.att[hs];
        att = mk3(at4.x, at4.y, at4.z);
        const v3 o = mk3(a.x, a.y, a.z), d = mk3(b.x, b.y, b.z);
        const uint32_t j0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)mt.x);
        if (n_jobs == 1 || __ballot(mt.x != j0) == 0)
            cont = shade_queued<TYPES>(jobs[j0], h, o, d, a.w, mt, records, max_depth, counters, att, no, nd);
        else
            cont = shade_queued<TYPES>(jobs[mt.x], h, o, d, a.w, mt, records, max_depth, counters, att, no, nd);
        }
    const uint32_t slot = block_append<BS>(cont, out, unit % QSEG, L.sh);
    if (cont && slot != EMPTY)
        {
        out.o[slot] = make_float4(no.x, no.y, no.z, 1e-3f);
        out.d[slot] = make_float4(nd.x, nd.y, nd.z, __uint_as_float(mt.x));
        out.att[slot] = make_float4(att.x, att.y, att.z, 0.0f);
        out.meta[slot] = make_uint4(mt.x, mt.y, mt.z, mt.w + 1);
        }
    }

// Units of BS rays from unit0 + blockIdx.x; LOOP: grid-stride over every
// further unit, else one unit per workgroup (the host sizes the grid from the
// live-path fraction recent renders had at this bounce and launches the LOOP
// form from the first unit beyond it, so no ray is left out).  Unit u appends
// to segment u % QSEG.  The LOOP form is held to 7 wavefronts per SIMD: its
// loop would otherwise keep the loop's constants (Philox, the sine/cosine
// polynomial) in registers across iterations instead of rematerializing them.
template<int BS, uint32_t TYPES, bool LOOP>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(LOOP ? 7 : 1))) void k_shade(
    const JobDev* __restrict__ jobs, uint32_t n_jobs, Queue in, uint32_t n, const QueueView* __restrict__ view,
    uint32_t unit0, const uint4* __restrict__ hits, Queue out, uint4* records, uint32_t max_depth,
    unsigned long long* counters)
    {
    if (!take_view(view, VIEW_BOUNCE, in, n))
        return;
    __shared__ ShadeLds<BS> lds;
    const uint32_t units = (n + BS - 1) / BS;
    for (uint32_t unit = unit0 + blockIdx.x; unit < units; unit += gridDim.x)
        {
        shade_unit<BS, TYPES>(jobs, n_jobs, in, n, unit, hits, out, records, max_depth, counters, lds);
        if (!LOOP)
            break;
        __syncthreads(); // the next unit rewrites the hit list
        }
    }

// Primary rays as wavefront packets.  The 64 rays of a wavefront come from
// one 8x8 pixel tile of one camera sample, so they need nearly the same
// nodes: the wavefront walks one node sequence (uniform node index, one
// fetch per visit) and every lane tests the visited node's children against
// its own ray, with its own closest hit, cull and leaf tests.  A lane acts
// only on nodes it wants (its own slab and cull tests passed at the parent),
// so each ray's result is the one the per-ray search returns; the wavefront
// descends into a child when any lane wants it, nearer child first by lane
// majority, and pushes the other with each lane's own cull bound.  A group of
// 64 rays that straddles jobs is searched once for each.
constexpr uint32_t UNWANTED = 0x80000000u; // stack flag: this lane does not need the node
typedef const GeomDev __attribute__((address_space(4))) ConstGeom;

// Leaf test of a primitive every lane of the wavefront shares: the geometry
// record and the primitive's data arrive through scalar loads.
template<uint32_t TYPES>
__device__ __forceinline__ bool leaf_test_uniform(const GeomDev* geoms, uint32_t slot, uint32_t prim, v3 o, v3 d,
                                                  float tnear, float& t)
    {
    if constexpr (TYPES == T_SPHERES)
        {
        const ConstGeom* g = (const ConstGeom*)geoms + slot;
        const ConstF* sp = (const ConstF*)g->a + 4 * (size_t)prim;
        float de;
        bool first;
        return sphere_t(o, d, mk3(sp[0], sp[1], sp[2]), sp[3], t, de, first) && (tnear < t);
        }
    else
        {
        const GeomDev g = uniform_geom(geoms, slot);
        return intersect_prim<false, TYPES, true>(g, prim, o, d, tnear, t, nullptr);
        }
    }

// Tile-list entries examined (counting kernels only): all, and those of
// spherocylinders, convex polyhedra and mesh triangles.
struct EntryCount
    {
    uint32_t all = 0, cyl = 0, poly = 0, mesh = 0;
    };

// Closest hits of one wavefront's 64 primary rays (lane ray o, d of job `job`
// at pixel px, py; `valid` lanes only): tile lists when all 64 rays form one
// full tile of a job that has them, else a wavefront-packet BVH search for
// each job.  ONE_JOB: every lane's job is the same (a scalar).
template<int SS, bool COUNT, uint32_t TYPES, bool ONE_JOB>
__device__ __forceinline__ void primary_group_hit(const JobDev* __restrict__ jobs, bool valid, uint32_t job,
                                                  uint32_t px, uint32_t py, v3 o, v3 d, float tnear,
                                                  LdsStack<SS>& st, HitT& best, uint32_t& n_nodes,
                                                  uint32_t& n_prims, EntryCount& n_entries, uint32_t& err)
    {
    // one job at a time (nearly always all 64 rays belong to one)
    uint64_t left = __ballot(valid);
    if (left == 0)
        return;
    do
    {
    const uint32_t first = ONE_JOB ? 0u : (uint32_t)(__ffsll((unsigned long long)left) - 1);
    const uint32_t job0 = (uint32_t)__builtin_amdgcn_readlane((int)job, first);
    const bool mine = ONE_JOB ? valid : (valid && job == job0);
    const uint64_t m_mine = __ballot(mine);
    left &= ~m_mine;
    // the tile of this group, if all 64 rays belong to one full 8x8 tile
    uint32_t tile = EMPTY;
    if (m_mine == ~0ull && jobs[job0].use_tiles)
        {
        const JobDev& J = jobs[job0];
        if (px < J.tiles_x * TILE && py < J.tiles_y * TILE)
            tile = (py / TILE) * J.tiles_x + px / TILE;
        const uint32_t t0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)tile);
        if (__ballot(tile != t0) != 0)
            tile = EMPTY;
        tile = (uint32_t)__builtin_amdgcn_readfirstlane((int)tile);
        }
    if (tile != EMPTY)
        {
        // candidate list of the tile (kernels/tiles.hip), nearest bound
        // first; the next entry is loaded while the current one is tested
        const JobDev& J = jobs[job0];
        const GeomDev* __restrict__ geoms = J.scene.geoms;
        const v3 inv = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
        best.t = __builtin_huge_valf();
        best.geom = EMPTY;
        best.prim = EMPTY;
        const uint32_t e0 = ((const ConstU*)J.tile_start)[tile];
        const uint32_t e1 = ((const ConstU*)J.tile_end)[tile];
        const ConstU* ent = (const ConstU*)J.tile_entries;
        uint32_t cur[8], nxt[8];
        if (e0 < e1)
            for (int k = 0; k < 8; k++)
                cur[k] = ent[8 * (size_t)e0 + k];
        for (uint32_t e = e0; e < e1; e++)
            {
            const size_t en = (e + 1 < e1) ? (size_t)e + 1 : (size_t)e;
            for (int k = 0; k < 8; k++)
                nxt[k] = ent[8 * en + k];
            const float q = __uint_as_float(cur[0]);
            const bool want = !(q > best.t);
            if (__ballot(want) == 0)
                break;
            if (COUNT)
                {
                n_entries.all++;
                if constexpr (TYPES != T_SPHERES)
                    if (!(cur[7] & NODE_REF))
                        {
                        const uint32_t type = J.scene.geoms[__float_as_uint(J.prim_lo[cur[7]].w)].type;
                        n_entries.cyl += type == G_CYLINDER;
                        n_entries.poly += type == G_POLYHEDRON;
                        n_entries.mesh += type == G_MESH;
                        }
                }
            if (want)
                {
                float lx, ly, lz, hx, hy, hz;
                float4 sph;
                uint32_t slot, prim;
                if constexpr (TYPES == T_SPHERES)
                    {
                    sph = make_float4(__uint_as_float(cur[1]), __uint_as_float(cur[2]),
                                      __uint_as_float(cur[3]), __uint_as_float(cur[4]));
                    // the sphere's bounds, as the builder computes them (GeometrySphere.cc:60-73)
                    lx = sph.x - sph.w;
                    ly = sph.y - sph.w;
                    lz = sph.z - sph.w;
                    hx = sph.x + sph.w;
                    hy = sph.y + sph.w;
                    hz = sph.z + sph.w;
                    slot = cur[5];
                    prim = cur[6];
                    }
                else
                    {
                    lx = __uint_as_float(cur[1]);
                    ly = __uint_as_float(cur[2]);
                    lz = __uint_as_float(cur[3]);
                    hx = __uint_as_float(cur[4]);
                    hy = __uint_as_float(cur[5]);
                    hz = __uint_as_float(cur[6]);
                    slot = 0;
                    prim = 0;
                    }
                float tmin, tmax;
                slab(o, inv, lx, ly, lz, hx, hy, hz, tmin, tmax);
                if ((tmin <= tmax) && (tmax >= tnear))
                    {
                    float t;
                    bool hit;
                    if constexpr (TYPES == T_SPHERES)
                        {
                        float de;
                        bool first;
                        if (COUNT)
                            n_prims++;
                        hit = sphere_t(o, d, mk3(sph.x, sph.y, sph.z), sph.w, t, de, first) && (tnear < t);
                        }
                    else
                        {
                        const uint32_t r = cur[7];
                        hit = false;
                        if (r & NODE_REF)
                            {
                            // a subtree: the BVH search below its root, from this
                            // lane's closest hit so far (same slab and cull tests)
                            if (!(cull_bound(tmin, tmax, J.scene.cull_margin) > best.t))
                                {
                                TraceState ts;
                                ts.o = o;
                                ts.d = d;
                                ts.inv = inv;
                                ts.tnear = tnear;
                                ts.margin = J.scene.cull_margin;
                                ts.best = best;
                                ts.node = r & ~NODE_REF;
                                st.sp = 0;
                                while (trace_visit2<LdsStack<SS>, COUNT, TYPES>(J.scene.nodes, geoms, ts, st, n_nodes,
                                                                                n_prims, err))
                                    {
                                    }
                                best = ts.best;
                                }
                            }
                        else
                            {
                            if (COUNT)
                                n_prims++;
                            // the entry's primitive is the same in every lane: its
                            // record and data arrive through scalar loads
                            slot = __float_as_uint(((ConstF*)J.prim_lo)[4 * (size_t)r + 3]);
                            prim = __float_as_uint(((ConstF*)J.prim_hi)[4 * (size_t)r + 3]);
                            const GeomDev g = uniform_geom(geoms, slot);
                            hit = intersect_prim<false, TYPES, true>(g, prim, o, d, tnear, t, nullptr);
                            }
                        }
                    if (hit && better(t, slot, prim, best))
                        {
                        best.t = t;
                        best.geom = slot;
                        best.prim = prim;
                        }
                    }
                }
            for (int k = 0; k < 8; k++)
                cur[k] = nxt[k];
            }
        }
    else
        {
        const SceneDev& sc = jobs[job0].scene;
        const Node* __restrict__ nodes = sc.nodes;
        const GeomDev* __restrict__ geoms = sc.geoms;
        const v3 inv = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
        const float margin = sc.cull_margin;
        if (mine)
            {
            best.t = __builtin_huge_valf();
            best.geom = EMPTY;
            best.prim = EMPTY;
            }
        st.sp = 0;
        uint32_t node = sc.root;
        bool want = mine;
        while (node != EMPTY)
            {
            // the node index is uniform: fetch through the constant address
            // space so the node arrives in scalar registers
            node = (uint32_t)__builtin_amdgcn_readfirstlane((int)node);
            const ConstF* nf = (const ConstF*)(nodes + node);
            const ConstU* nu = (const ConstU*)(nodes + node);
            const float4 A = make_float4(nf[0], nf[1], nf[2], nf[3]);
            const float4 B = make_float4(nf[4], nf[5], nf[6], nf[7]);
            const float4 C = make_float4(nf[8], nf[9], nf[10], nf[11]);
            const uint4 lk = make_uint4(nu[12], nu[13], nu[14], nu[15]);
            if (COUNT && want)
                n_nodes++;
            float t0min, t0max, t1min, t1max;
            slab(o, inv, A.x, A.y, A.z, A.w, B.x, B.y, t0min, t0max);
            slab(o, inv, B.z, B.w, C.x, C.y, C.z, C.w, t1min, t1max);
            const float c0 = cull_bound(t0min, t0max, margin);
            const float c1 = cull_bound(t1min, t1max, margin);
            bool w0 = want && (t0min <= t0max) && (t0max >= tnear) && !(c0 > best.t);
            bool w1 = want && (t1min <= t1max) && (t1max >= tnear) && !(c1 > best.t);
            if (lk.x & LEAF)
                {
                if (w0)
                    {
                    const uint32_t prim = lk.x & ~LEAF;
                    float t;
                    if (COUNT)
                        n_prims++;
                    if (leaf_test_uniform<TYPES>(geoms, lk.z, prim, o, d, tnear, t) && better(t, lk.z, prim, best))
                        {
                        best.t = t;
                        best.geom = lk.z;
                        best.prim = prim;
                        }
                    }
                w0 = false;
                }
            if (lk.y & LEAF)
                {
                if (w1)
                    {
                    const uint32_t prim = lk.y & ~LEAF;
                    float t;
                    if (COUNT)
                        n_prims++;
                    if (leaf_test_uniform<TYPES>(geoms, lk.w, prim, o, d, tnear, t) && better(t, lk.w, prim, best))
                        {
                        best.t = t;
                        best.geom = lk.w;
                        best.prim = prim;
                        }
                    }
                w1 = false;
                }
            w0 = w0 && !(c0 > best.t);
            w1 = w1 && !(c1 > best.t);
            const uint64_t b0 = __ballot(w0), b1 = __ballot(w1);
            if (b0 && b1)
                {
                const uint64_t both = b0 & b1;
                const uint64_t pref1 = __ballot(w0 && w1 && t1min < t0min);
                const bool near1 = 2 * __popcll(pref1) > __popcll(both);
                const uint32_t far_node = near1 ? lk.x : lk.y;
                const bool far_want = near1 ? w0 : w1;
                st.push(far_want ? far_node : (far_node | UNWANTED), near1 ? c0 : c1, err);
                node = near1 ? lk.y : lk.x;
                want = near1 ? w1 : w0;
                continue;
                }
            if (b0)
                {
                node = lk.x;
                want = w0;
                continue;
                }
            if (b1)
                {
                node = lk.y;
                want = w1;
                continue;
                }
            node = EMPTY;
            while (st.sp > 0)
                {
                uint32_t e;
                float cv;
                st.pop(e, cv);
                const bool w = !(e & UNWANTED) && !(cv > best.t);
                if (__ballot(w) != 0)
                    {
                    node = (uint32_t)__builtin_amdgcn_readfirstlane((int)e) & ~UNWANTED;
                    want = w;
                    break;
                    }
                }
            }
        }
    } while (!ONE_JOB && left != 0);
    }

template<int BLOCK, int SS, bool COUNT, uint32_t TYPES>
__global__ __launch_bounds__(BLOCK) void k_traverse_packet(const JobDev* __restrict__ jobs, uint32_t n_jobs,
                                                           uint32_t n, uint4* hits, uint32_t* work, uint32_t chunk,
                                                           uint2* gstack, uint32_t gstride,
                                                           unsigned long long* counters)
    {
    __shared__ uint2 lds[SS * BLOCK];
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    LdsStack<SS> st;
    st.lds = lds + threadIdx.x;
    st.lstride = BLOCK;
    st.glob = gstack + gtid;
    st.gstride = gstride;
    st.sp = 0;
    const uint32_t lane = lane_id();
    uint32_t n_nodes = 0, n_prims = 0, err = 0, n_rays = 0;
    EntryCount n_entries;
    uint32_t claim = 0;
    if (lane == 0)
        claim = atomicAdd(work, chunk);
    uint32_t base = __shfl(claim, 0, 64);
    while (base < n)
        {
        uint32_t next = 0;
        if (lane == 0)
            next = atomicAdd(work, chunk);
        const uint32_t end = min(n, base + chunk);
        for (uint32_t sub = base; sub < end; sub += 64)
            {
            const uint32_t i = sub + lane;
            const bool valid = i < end;
            v3 o = mk3(0.0f, 0.0f, 0.0f), d = mk3(0.0f, 0.0f, 1.0f);
            uint32_t job = 0, px = 0, py = 0;
            if (valid)
                {
                uint32_t k, jord;
                primary_ray(jobs, n_jobs, i, job, k, px, py, jord, o, d);
                }
            HitT best;
            primary_group_hit<SS, COUNT, TYPES, false>(jobs, valid, job, px, py, o, d, 1e-3f, st, best, n_nodes,
                                                       n_prims, n_entries, err);
            if (valid)
                {
                hits[i] = make_uint4(__float_as_uint(best.t), best.geom, best.prim, 0);
                if (COUNT)
                    n_rays++;
                }
            }
        base = __shfl(next, 0, 64);
        }
    if (COUNT)
        {
        atomicAdd(counters + CTR_PRIMARY + 0, (unsigned long long)n_rays);
        atomicAdd(counters + CTR_PRIMARY + 1, (unsigned long long)n_nodes);
        atomicAdd(counters + CTR_PRIMARY + 2, (unsigned long long)n_prims);
        atomicAdd(counters + CTR_TILE_ENTRIES, (unsigned long long)n_entries.all);
        atomicAdd(counters + CTR_TILE_ENTRIES + 1, (unsigned long long)n_entries.cyl);
        atomicAdd(counters + CTR_TILE_ENTRIES + 2, (unsigned long long)n_entries.poly);
        atomicAdd(counters + CTR_TILE_ENTRIES + 3, (unsigned long long)n_entries.mesh);
        }
    if (err)
        atomicOr((unsigned int*)(counters + CTR_OVERFLOW), 1u);
    }

// Primary rays traced and shaded in one persistent kernel: the workgroup
// claims `groups` x its size rays per atomic, each wavefront traces `groups`
// groups of 64 rays (primary_group_hit) and the workgroup shades them
// together (shade_primary_block), so no hit is stored and no primary ray is
// generated twice.  Same arithmetic as k_traverse_packet + k_shade_primary.
// The spheres-only variant is held to 128 registers (4 wavefronts per SIMD; a
// few values spill): with the double-precision sine and cosine of the depth-0
// lobe sample it would take 147 (3 wavefronts) and run 1.7x longer, and at 5
// wavefronts it spills more and runs 17 % longer.  The variant for other
// scenes, whose list search waits on primitive loads, runs best at 6 (C3's
// primary kernel: 31.2 ms per frame at 4, 29.8 at 5, 27.7 at 6, 28.2 at 8).
template<int BLOCK, int SS, bool COUNT, uint32_t TYPES>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(TYPES == T_SPHERES ? 4 : 6))) void k_primary(
    const JobDev* __restrict__ jobs, uint32_t n_jobs, uint32_t n, uint32_t* work, uint32_t groups, uint32_t bands,
    uint2* gstack, uint32_t gstride, Queue out, uint4* records, unsigned long long* counters)
    {
    __shared__ uint2 lds[SS * BLOCK];
    __shared__ uint32_t sh[BLOCK / 64 + 1];
    __shared__ uint32_t s_claim;
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    LdsStack<SS> st;
    st.lds = lds + threadIdx.x;
    st.lstride = BLOCK;
    st.glob = gstack + gtid;
    st.gstride = gstride;
    st.sp = 0;
    const uint32_t lane = lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t chunk = BLOCK * groups;
    uint32_t n_nodes = 0, n_prims = 0, err = 0, n_rays = 0;
    EntryCount n_entries;
    // Chunk u of n_units goes to queue segment u % QSEG, or with bands to
    // segment u / G (16 contiguous bands of G chunks, i.e. of the image); the
    // claims then visit the bands in turn, claim c -> chunk (c % QSEG) G + c /
    // QSEG, so the chunks in flight still append to all 16 segments.
    const uint32_t n_units = (n + chunk - 1) / chunk;
    const uint32_t G = (n_units + QSEG - 1) / QSEG;
    const uint32_t n_claims = bands ? QSEG * G : n_units;
    if (threadIdx.x == 0)
        s_claim = atomicAdd(work, 1u);
    __syncthreads();
    uint32_t c = s_claim;
    __syncthreads();
    while (c < n_claims)
        {
        if (threadIdx.x == 0)
            s_claim = atomicAdd(work, 1u); // the next chunk, claimed ahead
        const uint32_t u = bands ? (c % QSEG) * G + c / QSEG : c;
        const uint32_t seg = bands ? u / G : u % QSEG; // the chunk's output segment
        const uint32_t base = u * chunk;
        // the chunk's jobs one after the other (one, unless it straddles two):
        // the job's index is workgroup-uniform, so its record arrives by scalar
        // loads and the loop is taken by the whole workgroup, barriers included
        const uint32_t last = min(n, base + chunk) - 1u;
        const uint32_t job_first = (uint32_t)__builtin_amdgcn_readfirstlane((int)find_job(jobs, n_jobs, base));
        const uint32_t job_last = (uint32_t)__builtin_amdgcn_readfirstlane((int)find_job(jobs, n_jobs, last));
        for (uint32_t job = job_first; job <= job_last && u < n_units; job++)
            {
            const JobDev& J = jobs[job];
            const uint32_t end = (job == job_last) ? n : jobs[job + 1].ray_base;
            // chunks of 64 pixels of this job's first and last ray here
            const uint32_t c0 = fdiv(max(base, J.ray_base) - J.ray_base, J.div_chunk);
            const uint32_t c1 = fdiv(min(last + 1u, end) - 1u - J.ray_base, J.div_chunk);
            if (c0 == c1 && empty_chunk(J, c0))
                {
                if (COUNT)
                    for (uint32_t g = 0; g < groups; g++)
                        {
                        const uint32_t i = base + (wave * groups + g) * 64 + lane;
                        n_rays += (i >= J.ray_base && i < end) ? 1u : 0u;
                        }
                continue;
                }
            for (uint32_t g = 0; g < groups; g++)
                {
                const uint32_t i0 = base + ((uint32_t)__builtin_amdgcn_readfirstlane((int)wave) * groups + g) * 64;
                const uint32_t i = i0 + lane;
                bool valid = i >= J.ray_base && i < end;
                if (COUNT && valid)
                    n_rays++;
                if (c0 != c1 && i0 >= J.ray_base && i0 < end)
                    {
                    // the group's chunk, if its rays belong to one
                    const uint32_t a = fdiv(i0 - J.ray_base, J.div_chunk);
                    if (a == fdiv(min(i0 + 64u, end) - 1u - J.ray_base, J.div_chunk) && empty_chunk(J, a))
                        valid = false;
                    }
                v3 o = mk3(0.0f, 0.0f, 0.0f), d = mk3(0.0f, 0.0f, 1.0f);
                uint32_t k = 0, px = 0, py = 0, jord = 0;
                if (valid)
                    primary_ray_of(J, i, k, px, py, jord, o, d);
                HitT best;
                best.t = __builtin_huge_valf();
                best.geom = EMPTY;
                best.prim = EMPTY;
                primary_group_hit<SS, COUNT, TYPES, true>(jobs, valid, job, px, py, o, d, 1e-3f, st, best, n_nodes,
                                                          n_prims, n_entries, err);
                shade_primary_block<BLOCK, TYPES>(jobs, valid, job, k, py * J.W + px, jord, o, d, best, out, seg,
                                                  records, sh);
                }
            }
        __syncthreads();
        c = s_claim;
        __syncthreads();
        }
    if (COUNT)
        {
        atomicAdd(counters + CTR_PRIMARY + 0, (unsigned long long)n_rays);
        atomicAdd(counters + CTR_PRIMARY + 1, (unsigned long long)n_nodes);
        atomicAdd(counters + CTR_PRIMARY + 2, (unsigned long long)n_prims);
        atomicAdd(counters + CTR_TILE_ENTRIES, (unsigned long long)n_entries.all);
        atomicAdd(counters + CTR_TILE_ENTRIES + 1, (unsigned long long)n_entries.cyl);
        atomicAdd(counters + CTR_TILE_ENTRIES + 2, (unsigned long long)n_entries.poly);
        atomicAdd(counters + CTR_TILE_ENTRIES + 3, (unsigned long long)n_entries.mesh);
        }
    if (err)
        atomicOr((unsigned int*)(counters + CTR_OVERFLOW), 1u);
    }

// One bounce of the secondary rays in one persistent kernel: each wavefront
// claims `chunk` rays of the queue per atomic (the next chunk ahead), traces
// each ray and shades its hit or miss (shade_bounce); continuing paths are
// appended to `out` with one atomic per 64 rays, terminated ones write their
// record.  Same arithmetic as k_traverse + k_shade.
template<int BLOCK, int SS, bool COUNT, uint32_t TYPES>
__global__ __launch_bounds__(BLOCK) void k_bounce(const JobDev* __restrict__ jobs, Queue in, uint32_t n,
                                                  const QueueView* __restrict__ view, uint32_t* work, uint32_t chunk,
                                                  uint2* gstack, uint32_t gstride, Queue out, uint4* records,
                                                  uint32_t max_depth, unsigned long long* counters)
    {
    if (!take_view(view, VIEW_BOUNCE, in, n))
        return;
    __shared__ uint2 lds[SS * BLOCK];
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    LdsStack<SS> st;
    st.lds = lds + threadIdx.x;
    st.lstride = BLOCK;
    st.glob = gstack + gtid;
    st.gstride = gstride;
    st.sp = 0;
    const uint32_t lane = lane_id();
    uint32_t n_nodes = 0, n_prims = 0, err = 0, n_rays = 0;
    uint32_t claim = 0;
    if (lane == 0)
        claim = atomicAdd(work, chunk);
    uint32_t base = __shfl(claim, 0, 64);
    while (base < n)
        {
        uint32_t next = 0;
        if (lane == 0)
            next = atomicAdd(work, chunk);
        const uint32_t end = min(n, base + chunk);
        const uint32_t seg = (base / chunk) % QSEG; // the chunk's output segment
        for (uint32_t sub = base; sub < end; sub += 64)
            {
            const uint32_t i = sub + lane;
            const uint32_t sl = q_slot(in, i, sub, min(end, sub + 64u) - 1u);
            bool cont = false;
            v3 att, no, nd;
            uint4 mt = make_uint4(0, 0, 0, 0);
            if (i < end)
                {
                mt = in.meta[sl];
                const JobDev& J = jobs[mt.x];
                const float4 a = in.o[sl];
                const float4 b = in.d[sl];
                const float4 at4 = in.att[sl];
                const v3 o = mk3(a.x, a.y, a.z), d = mk3(b.x, b.y, b.z);
                HitT h;
                trace_closest<LdsStack<SS>, COUNT, TYPES, false>(J.scene, o, d, a.w, h, st, n_nodes, n_prims, err);
                if (COUNT)
                    n_rays++;
                att = mk3(at4.x, at4.y, at4.z);
                const uint32_t k = mt.z & 0xffffu, ls = mt.z >> 16;
                uint4 rec;
                cont = shade_bounce<TYPES>(J, h, o, d, a.w, mt.y, k, ls, mt.w, att, no, nd, rec);
                if (cont && mt.w + 1 >= max_depth)
                    {
                    // depth cap (the reference has none): stop without contribution
                    cont = false;
                    rec = make_rec(mk3(0, 0, 0), REC_NONE);
                    atomicAdd(counters + CTR_CAPPED, 1ull);
                    }
                if (!cont)
                    records[rec_index(J, k, raster_ordinal(J, mt.y), ls)] = rec;
                }
            const uint32_t slot = wave_append(cont, out, seg);
            if (cont && slot != EMPTY)
                {
                out.o[slot] = make_float4(no.x, no.y, no.z, 1e-3f);
                out.d[slot] = make_float4(nd.x, nd.y, nd.z, __uint_as_float(mt.x));
                out.att[slot] = make_float4(att.x, att.y, att.z, 0.0f);
                out.meta[slot] = make_uint4(mt.x, mt.y, mt.z, mt.w + 1);
                }
            }
        base = __shfl(next, 0, 64);
        }
    if (COUNT)
        {
        atomicAdd(counters + CTR_SECONDARY + 0, (unsigned long long)n_rays);
        atomicAdd(counters + CTR_SECONDARY + 1, (unsigned long long)n_nodes);
        atomicAdd(counters + CTR_SECONDARY + 2, (unsigned long long)n_prims);
        }
    if (err)
        atomicOr((unsigned int*)(counters + CTR_OVERFLOW), 1u);
    }

// One bounce of a path in the tail: trace and shade.  Returns whether the path
// goes on (o, d, att, mt.w moved to its next segment); otherwise its record is
// written.
template<int SS, bool COUNT, uint32_t TYPES, bool UNI>
__device__ __forceinline__ bool finish_bounce(const JobDev& J, uint4& mt, v3& o, v3& d, v3& att, LdsStack<SS>& st,
                                              uint4* records, uint32_t max_depth, unsigned long long* counters,
                                              uint32_t& n_nodes, uint32_t& n_prims, uint32_t& err)
    {
    const uint32_t k = mt.z & 0xffffu, ls = mt.z >> 16;
    uint4 rec;
    HitT h;
    trace_closest<LdsStack<SS>, COUNT, TYPES, UNI>(J.scene, o, d, 1e-3f, h, st, n_nodes, n_prims, err);
    v3 no, nd;
    bool cont = shade_bounce<TYPES>(J, h, o, d, 1e-3f, mt.y, k, ls, mt.w, att, no, nd, rec);
    if (cont && mt.w + 1 >= max_depth)
        {
        cont = false;
        rec = make_rec(mk3(0, 0, 0), REC_NONE);
        atomicAdd(counters + CTR_CAPPED, 1ull);
        }
    if (!cont)
        {
        records[rec_index(J, k, raster_ordinal(J, mt.y), ls)] = rec;
        return false;
        }
    o = no;
    d = nd;
    mt.w++;
    return true;
    }

// Tail: the paths still queued are traced and shaded to their ends by the
// resident wavefronts.  Up to 64 a wavefront they are dealt out evenly, so a
// few thousand paths run a few lanes each on every SIMD and a wavefront waits
// for the longest of few rays; beyond that, a lane whose path has ended takes
// the next one from the pool (one atomic per wavefront and bounce), so lanes
// stay busy until the pool is empty.  A wavefront whose paths all belong to
// one job reads the job record through scalar loads, as in k_shade.  gstride
// is the grid's thread count.  Bound by the latency of the longest paths' node
// loads.  One thread per path to its end (7 of 64 lanes active) took 4.6 ms on
// the mesh scene's 1.9M tail rays, 1.26 on the lens scene's 0.6M, 0.49 on the
// small scene's; this takes 3.06, 0.94 and 0.36 (held to 5 or 6 wavefronts per
// SIMD instead of 4: 3.8 and 2.9 on the meshes, 0.45 and 0.39 on the small one).
template<int BLOCK, int SS, bool COUNT, uint32_t TYPES>
__global__ __launch_bounds__(BLOCK) void k_finish(const JobDev* __restrict__ jobs, uint32_t n_jobs, Queue in,
                                                  uint32_t n, const QueueView* __restrict__ view, uint32_t* work,
                                                  uint4* records, uint32_t max_depth, uint2* gstack,
                                                  uint32_t gstride, unsigned long long* counters)
    {
    if (!take_view(view, VIEW_FINISH, in, n))
        return;
    __shared__ uint2 lds[SS * BLOCK];
    LdsStack<SS> st;
    st.lds = lds + threadIdx.x;
    st.lstride = BLOCK;
    st.glob = gstack + blockIdx.x * BLOCK + threadIdx.x;
    st.gstride = gstride;
    st.sp = 0;
    uint32_t n_nodes = 0, n_prims = 0, n_rays = 0, err = 0;
    const uint32_t lane = lane_id();
    const uint32_t waves = gridDim.x * (BLOCK / 64);
    const uint32_t wave = blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
    const uint32_t per = min(64u, (n + waves - 1) / waves);
    const uint32_t dealt = waves * per; // paths from here on form the pool
    bool pool = dealt < n;
    bool active = false;
    uint32_t i = wave * per + lane;
    bool take = lane < per && i < n;
    uint4 mt = make_uint4(0, 0, 0, 0);
    v3 o = mk3(0, 0, 0), d = mk3(0, 0, 1), att = mk3(0, 0, 0);
    for (;;)
        {
        if (take)
            {
            const uint32_t sl = i + seg_adj(in, i);
            mt = in.meta[sl];
            const float4 a = in.o[sl];
            const float4 b = in.d[sl];
            const float4 at4 = in.att[sl];
            o = mk3(a.x, a.y, a.z);
            d = mk3(b.x, b.y, b.z);
            att = mk3(at4.x, at4.y, at4.z);
            active = true;
            }
        if (__ballot(active) == 0)
            break;
        if (active)
            {
            if (COUNT)
                n_rays++;
            const uint32_t j0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)mt.x);
            if (n_jobs == 1 || __ballot(mt.x != j0) == 0)
                active = finish_bounce<SS, COUNT, TYPES, true>(jobs[j0], mt, o, d, att, st, records, max_depth,
                                                               counters, n_nodes, n_prims, err);
            else
                active = finish_bounce<SS, COUNT, TYPES, false>(jobs[mt.x], mt, o, d, att, st, records, max_depth,
                                                                counters, n_nodes, n_prims, err);
            }
        take = false;
        const uint64_t idle = __ballot(!active);
        if (pool && idle != 0)
            {
            uint32_t c = 0;
            if (lane == 0)
                c = atomicAdd(work, (uint32_t)__popcll(idle));
            // (the counter stays below n + 64 x the wavefronts: one claim past the end each)
            i = dealt + __shfl(c, 0, 64) + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
            take = !active && i < n;
            pool = __ballot(!active && i >= n) == 0;
            }
        }
    if (COUNT)
        {
        atomicAdd(counters + CTR_TAIL + 0, (unsigned long long)n_rays);
        atomicAdd(counters + CTR_TAIL + 1, (unsigned long long)n_nodes);
        atomicAdd(counters + CTR_TAIL + 2, (unsigned long long)n_prims);
        }
    if (err)
        atomicOr((unsigned int*)(counters + CTR_OVERFLOW), 1u);
    }

// ---------------------------------------------------------------- accumulate
// Replay each camera sample's records in light-sample order, then the Welford
// mean and sRGB of fresnel/cpu/TracerPath.cc:229-249.
__global__ void k_accumulate(const JobDev* __restrict__ jobs, uint32_t n_jobs, uint32_t total,
                             const uint4* __restrict__ records)
    {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total)
        return;
    uint32_t lo = 0, hi = n_jobs;
    while (hi - lo > 1)
        {
        const uint32_t mid = (lo + hi) >> 1;
        if (jobs[mid].pix_base <= i)
            lo = mid;
        else
            hi = mid;
        }
    const JobDev& J = jobs[lo];
    // thread i handles pixel ordinal j (records are chunk-major, so a
    // wavefront reads 64 contiguous records per sample)
    const uint32_t jord = i - J.pix_base;
    uint32_t px, py;
    ordinal_pixel(J, jord, px, py);
    const uint32_t pixel = py * J.W + px;
    float4 mean = J.linear[pixel];
    const uint32_t K = J.K;
    // a chunk nothing was traced for has no records (empty_chunk; a wavefront
    // of a later job may straddle two chunks)
    const uint32_t chunk = jord >> 6;
    const bool empty = J.use_tiles && chunk < J.tiles_x * J.tiles_y && J.tile_start[chunk] == J.tile_end[chunk];
    // the first records of four camera samples are loaded together, then
    // folded into the mean in sample order
    constexpr uint32_t U = 4;
    for (uint32_t k0 = 0; k0 < K; k0 += U)
    {
    uint4 rk[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++)
        rk[u] = (k0 + u < K && !empty) ? records[rec_index(J, k0 + u, jord, 0)] : make_uint4(0, 0, 0, REC_BG);
#pragma unroll
    for (uint32_t u = 0; u < U; u++)
        {
        const uint32_t k = k0 + u;
        if (k < K)
        {
        v3 result = mk3(0, 0, 0);
        float a = 1.0f;
        const uint4 r0 = rk[u];
        if ((r0.w & 3u) == REC_BG)
            {
            result = J.bg * float(J.L);
            a = J.bg_alpha;
            }
        else
            {
            auto fold = [&](const uint4 r)
            {
                const v3 val = mk3(__uint_as_float(r.x), __uint_as_float(r.y), __uint_as_float(r.z));
                const uint32_t kind = r.w & 3u;
                if (kind == REC_ADD)
                    result = result + val;
                else if (kind == REC_LIGHTS)
                    {
                    const uint32_t mask = r.w >> 2;
                    for (uint32_t li = 0; li < J.lights.N; li++)
                        if (mask & (1u << li))
                            result = result + (val * J.lights.color[li]) * J.lights.inv_sin[li];
                    }
            };
            fold(r0);
            for (uint32_t ls = 1; ls < J.L; ls++)
                fold(records[rec_index(J, k, jord, ls)]);
            }
        const v3 s = div_rcp(result, float(J.L));
        const float q = 1.0f / float(J.n_base + k + 1);
        mean.x = mean.x + (s.x - mean.x) * q;
        mean.y = mean.y + (s.y - mean.y) * q;
        mean.z = mean.z + (s.z - mean.z) * q;
        mean.w = mean.w + (a - mean.w) * q;
        }
        }
    }
    J.linear[pixel] = mean;
    if (!J.highlight || (mean.x <= 1.0f && mean.y <= 1.0f && mean.z <= 1.0f))
        J.srgb[pixel] = to_srgb(mean);
    else
        J.srgb[pixel] = to_srgb(make_float4(J.hw_color.x, J.hw_color.y, J.hw_color.z, mean.w));
    }

// ---------------------------------------------------------------- preview
// fresnel/cpu/TracerDirect.cc:77-218: aa_n^2 primary rays with tnear 0 and
// representative-point direct lighting, plain mean.

// Color and opacity of one preview ray's closest hit h (background on a miss).
template<uint32_t TYPES>
__device__ __forceinline__ float4 preview_shade(const JobDev& J, const HitT& h, v3 o, v3 d)
    {
    if (h.geom == EMPTY)
        return make_float4(J.bg.x, J.bg.y, J.bg.z, J.bg_alpha);
    Attr at;
    const GeomDev* g;
    hit_attributes<TYPES>(J.scene, h, o, d, 0.0f, at, g);
    const v3 n = div_true(at.Ng, sqrtf(dot(at.Ng, at.Ng)));
    const v3 v = div_rcp(-d, sqrtf(dot(d, d)));
    const Mat& m = (at.d >= g->outline_width) ? g->mat : g->outline;
    v3 c;
    if (m.solid > 0.5f)
        c = get_color(m, at.color);
    else
        {
        c = mk3(0, 0, 0);
        for (uint32_t li = 0; li < J.lights.N; li++)
            {
            const v3 l = J.lights.dir[li];
            v3 r = -v + (2.0f * n * dot(n, v));
            const float half = J.lights.theta[li];
            const float ldotr = dot(l, r);
            if (ldotr < J.lights.cos_theta[li])
                {
                v3 ax = cross(l, r);
                ax = div_rcp(ax, sqrtf(dot(ax, ax)));
                const float ang = -acosf(ldotr) + half;
                quat qr;
                qr.s = cosf(ang / 2.0f);
                qr.v = sinf(ang / 2.0f) * ax;
                r = rotate(qr, r);
                }
            const float ndotl = dot(n, l);
            const v3 f_d = (ndotl >= 0.0f) ? brdf_diffuse(m, l, v, n, at.color) * ndotl : mk3(0, 0, 0);
            const v3 f_s = (dot(n, r) >= 0.0f)
                               ? brdf_specular(m, r, v, n, at.color, half, J.lights.tan_clamped[li]) * dot(n, r)
                               : mk3(0, 0, 0);
            c = c + (f_d + f_s) * PI_F * J.lights.color[li];
            }
        }
    return make_float4(c.x, c.y, c.z, 1.0f);
    }

// One workgroup per unit of the primary-ray order, grid-stride.  A wavefront
// traces one sample of the 64 pixels of a chunk (an 8x8 tile), so its rays
// take the tile's candidate list or one packet search (primary_group_hit)
// instead of 64 searches of their own.  SPLIT: a unit is one chunk, and its
// samples go round the workgroup's wavefronts; each round's colors meet in
// LDS, where one thread per pixel and channel adds them in sample order (the
// order of the reference's loop, so the sum does not depend on the split).
// Otherwise (fewer samples than wavefronts) each wavefront has a chunk to
// itself.  own_search: each lane searches the binary hierarchy for its own ray
// (scenes with convex polyhedra, whose hits may lie units below their box's
// entry, see CULL_K: which one is found first decides then, and the order stays
// that of the search per ray).
// The kernel is bound by VALU issue (camera rays with Philox, the
// lights' acos, sin and cos).  One pixel per thread with its own search and
// 64 serial samples, in raster order with the stack in scratch, took 5.99 ms
// for 500 spheres at 600 x 370 and 34.3 ms for 20,000 polyhedra at 1280 x
// 720, 64 samples each, image read included; this form takes 0.67 and 16.8 ms.
// Held to 80 registers (6 wavefronts per SIMD, what the LDS allows; some values
// spill): 1280 x 720, 64 samples of 500 spheres 0.69 -> 0.62 ms of kernel,
// 20,000 spherocylinders 2.8 -> 2.5, 500 meshes 6.4 -> 5.6, mixed 17.8 -> 16.2
// against the 4 that 113 to 127 registers allow.
template<int BLOCK, int SS, uint32_t TYPES, bool SPLIT>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(6))) void k_preview(
    const JobDev* __restrict__ jobp, uint32_t aa_n, uint32_t own_search, uint2* gstack, uint32_t gstride,
    unsigned long long* counters)
    {
    constexpr uint32_t WAVES = BLOCK / 64;
    static_assert(BLOCK == 256, "one thread per pixel and channel of a chunk");
    __shared__ uint2 lds[SS * BLOCK];
    __shared__ float4 col[SPLIT ? 2 : 1][SPLIT ? WAVES * 64 : 1];
    const JobDev& J = *jobp;
    LdsStack<SS> st;
    st.lds = lds + threadIdx.x;
    st.lstride = BLOCK;
    st.glob = gstack + blockIdx.x * BLOCK + threadIdx.x;
    st.gstride = gstride;
    st.sp = 0;
    const uint32_t lane = lane_id();
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t samples = aa_n * aa_n;
    const uint32_t n_chunks = (J.npix + 63) / 64;
    const uint32_t n_units = SPLIT ? n_chunks : (n_chunks + WAVES - 1) / WAVES;
    const float q = 1.0f / float(samples);
    uint32_t n_nodes = 0, n_prims = 0, err = 0;
    EntryCount n_entries;
    for (uint32_t u = blockIdx.x; u < n_units; u += gridDim.x)
        {
        const uint32_t chunk = SPLIT ? u : u * WAVES + wave;
        const uint32_t j = chunk * 64 + lane;
        const bool valid = j < J.npix;
        uint32_t px = 0, py = 0;
        if (valid)
            ordinal_pixel(J, j, px, py);
        float4 sum = make_float4(0, 0, 0, 0); // SPLIT: .x is this thread's channel
        uint32_t rounds = SPLIT ? (samples + WAVES - 1) / WAVES : samples;
        if (empty_chunk(J, SPLIT ? chunk : (uint32_t)__builtin_amdgcn_readfirstlane((int)chunk)))
            {
            // every sample is background, added as often
            const uint32_t ch = threadIdx.x & 3u;
            const float4 b = make_float4(J.bg.x, J.bg.y, J.bg.z, J.bg_alpha);
            const float x = (ch == 0u) ? b.x : (ch == 1u) ? b.y : (ch == 2u) ? b.z : b.w;
            for (uint32_t k = 0; k < samples; k++)
                {
                sum.x += SPLIT ? x : b.x;
                sum.y += b.y;
                sum.z += b.z;
                sum.w += b.w;
                }
            rounds = 0;
            }
        for (uint32_t r = 0; r < rounds; r++)
            {
            const uint32_t sample = SPLIT ? r * WAVES + wave : r;
            float4 c = make_float4(0, 0, 0, 0);
            if (sample < samples)
                {
                v3 o = mk3(0.0f, 0.0f, 0.0f), d = mk3(0.0f, 0.0f, 1.0f);
                if (valid)
                    camera_ray(J.cam, J.W, J.H, J.xs_off, J.inv_h, J.seed, px, py, sample, aa_n != 1, o, d);
                HitT h;
                h.t = __builtin_huge_valf();
                h.geom = EMPTY;
                h.prim = EMPTY;
                if (TYPES != T_SPHERES && own_search)
                    {
                    if (valid)
                        trace_binary<LdsStack<SS>, false, TYPES>(J.scene, o, d, 0.0f, h, st, n_nodes, n_prims, err);
                    }
                else
                    primary_group_hit<SS, false, TYPES, true>(jobp, valid, 0, px, py, o, d, 0.0f, st, h, n_nodes,
                                                              n_prims, n_entries, err);
                if (valid)
                    c = preview_shade<TYPES>(J, h, o, d);
                }
            if constexpr (SPLIT)
                {
                float4* buf = col[r & 1u];
                buf[wave * 64 + lane] = c;
                __syncthreads(); // the other half of col is rewritten only after the next round's barrier
                const float* f = (const float*)buf;
                const uint32_t n = min(WAVES, samples - r * WAVES);
                for (uint32_t w = 0; w < n; w++)
                    sum.x += f[w * 256 + threadIdx.x];
                }
            else
                {
                sum.x += c.x;
                sum.y += c.y;
                sum.z += c.z;
                sum.w += c.w;
                }
            }
        if constexpr (SPLIT)
            {
            // thread 4 k + channel holds its channel of pixel k
            const uint32_t ch = threadIdx.x & 3u;
            const uint32_t jp = chunk * 64 + (threadIdx.x >> 2);
            float v = sum.x * q;
            const uint64_t low = __ballot(ch == 3u || v <= 1.0f);
            const bool plain = !J.highlight || ((low >> (lane & ~3u)) & 15u) == 15u;
            if (jp < J.npix)
                {
                ordinal_pixel(J, jp, px, py);
                const size_t at = 4 * ((size_t)py * J.W + px) + ch;
                ((float*)J.linear)[at] = v;
                if (!plain && ch < 3u)
                    v = (ch == 0u) ? J.hw_color.x : (ch == 1u) ? J.hw_color.y : J.hw_color.z;
                ((unsigned char*)J.srgb)[at] = (ch == 3u) ? (unsigned char)(v * 255.0f + 0.5f) : srgb_channel(v);
                }
            __syncthreads(); // the next unit writes col[0] again
            }
        else if (valid)
            {
            const uint32_t pixel = py * J.W + px;
            const float4 outp = make_float4(sum.x * q, sum.y * q, sum.z * q, sum.w * q);
            J.linear[pixel] = outp;
            if (!J.highlight || (outp.x <= 1.0f && outp.y <= 1.0f && outp.z <= 1.0f))
                J.srgb[pixel] = to_srgb(outp);
            else
                J.srgb[pixel] = to_srgb(make_float4(J.hw_color.x, J.hw_color.y, J.hw_color.z, outp.w));
            }
        }
    if (err)
        atomicOr((unsigned int*)(counters + CTR_OVERFLOW), 1u);
    }

// ---------------------------------------------------------------- diagnostics
// Plain streaming copy, the reference point that scales the HBM byte counters.
__global__ void k_debug_copy(const float4* __restrict__ src, float4* __restrict__ dst, uint64_t n)
    {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
    }

__global__ void k_debug_philox(const uint32_t* in, uint32_t n, uint32_t* out)
    {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const uint32_t* c = in + 6 * i;
    const u4 r = philox(c[0], c[1], c[2], c[3], c[4], c[5]);
    for (int q = 0; q < 4; q++)
        out[4 * i + q] = r.v[q];
    }

// The shading code's sinf/cosf (cr_sincosf) of n arguments.
__global__ void k_debug_sincos(const float* x, uint32_t n, float* s, float* c)
    {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    float a, b;
    cr_sincosf(x[i], a, b);
    s[i] = a;
    c[i] = b;
    }

// Primary ray and closest hit per pixel for camera sample `sample`.
template<uint32_t TYPES>
__global__ void k_debug_primary(const JobDev* __restrict__ jobp, uint32_t sample, float* rays, uint4* hits)
    {
    const JobDev& J = *jobp;
    const uint32_t pixel = blockIdx.x * blockDim.x + threadIdx.x;
    if (pixel >= J.npix)
        return;
    const uint32_t py = pixel / J.W, px = pixel - py * J.W;
    v3 o, d;
    camera_ray(J.cam, J.W, J.H, J.xs_off, J.inv_h, J.seed, px, py, sample, true, o, d);
    LocalStack st;
    uint32_t dummy = 0, err = 0;
    HitT h;
    trace_closest<LocalStack, false, TYPES, true>(J.scene, o, d, 1e-3f, h, st, dummy, dummy, err);
    float* r = rays + 6 * (size_t)pixel;
    r[0] = o.x;
    r[1] = o.y;
    r[2] = o.z;
    r[3] = d.x;
    r[4] = d.y;
    r[5] = d.z;
    hits[pixel] = make_uint4(__float_as_uint(h.t), h.geom, h.prim, err);
    }

template<uint32_t TYPES>
__global__ void k_debug_trace(const SceneDev sc, const float* rays, uint32_t n, float tnear, uint4* hits)
    {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const float* r = rays + 6 * (size_t)i;
    LocalStack st;
    uint32_t dummy = 0, err = 0;
    HitT h;
    const v3 o = mk3(r[0], r[1], r[2]), d = mk3(r[3], r[4], r[5]);
    // the 4-wide search takes boxes behind the origin as closed
    if (tnear < 0.0f)
        trace_binary<LocalStack, false, TYPES>(sc, o, d, tnear, h, st, dummy, dummy, err);
    else
        trace_closest<LocalStack, false, TYPES, true>(sc, o, d, tnear, h, st, dummy, dummy, err);
    hits[i] = make_uint4(__float_as_uint(h.t), h.geom, h.prim, err);
    }
    } // namespace fh
