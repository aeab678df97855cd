// bvh.hip -- linear BVH construction and refit on gfx950.
//
//   prim_bounds  per-primitive boxes (the reference bounds callbacks)
//   centroid bounds reduction
//   morton       30-bit Morton code of each box centroid
//   radix sort   stable LSD sort of (code, index), 4 passes of 8 bits; ranks
//                inside a block come from wavefront ballots and LDS counters
//   karras       hierarchy emission over the sorted codes with the position
//                as tie break (Karras, HPG 2012): every key is distinct, so the
//                tree depth is at most 64
//   refit        bottom-up box union with one atomic arrival counter per node
#include "rt/isect.h"

namespace fh
{
constexpr int SORT_BLOCK = 256;

// ---------------------------------------------------------------- bounds
__global__ void k_prim_bounds(const GeomDev* __restrict__ geoms, const uint32_t* __restrict__ prefix,
                              const uint32_t* __restrict__ slots, uint32_t n_active, uint32_t N, float4* lo_out,
                              float4* hi_out)
    {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N)
        return;
    uint32_t lo = 0, hi = n_active;
    while (hi - lo > 1)
        {
        const uint32_t mid = (lo + hi) >> 1;
        if (prefix[mid] <= i)
            lo = mid;
        else
            hi = mid;
        }
    const uint32_t slot = slots[lo];
    const uint32_t local = i - prefix[lo];
    v3 bl, bh;
    prim_bounds(geoms[slot], local, bl, bh);
    lo_out[i] = make_float4(bl.x, bl.y, bl.z, __uint_as_float(slot));
    hi_out[i] = make_float4(bh.x, bh.y, bh.z, __uint_as_float(local));
    }

// Centroid bounds: per-block partials, then one block reduces the partials.
__device__ __forceinline__ void block_minmax(float v[6], float* sh)
    {
    // v[0..2] minimum, v[3..5] maximum; sh holds 6 * blockDim floats
    for (int k = 0; k < 6; k++)
        sh[k * blockDim.x + threadIdx.x] = v[k];
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1)
        {
        if (threadIdx.x < s)
            for (int k = 0; k < 6; k++)
                {
                const float a = sh[k * blockDim.x + threadIdx.x], b = sh[k * blockDim.x + threadIdx.x + s];
                sh[k * blockDim.x + threadIdx.x] = (k < 3) ? fminf(a, b) : fmaxf(a, b);
                }
        __syncthreads();
        }
    for (int k = 0; k < 6; k++)
        v[k] = sh[k * blockDim.x];
    }

__global__ void k_centroid_partial(const float4* __restrict__ lo, const float4* __restrict__ hi, uint32_t N,
                                   float* partial)
    {
    __shared__ float sh[6 * 256];
    float v[6] = {__builtin_huge_valf(), __builtin_huge_valf(), __builtin_huge_valf(),
                  -__builtin_huge_valf(), -__builtin_huge_valf(), -__builtin_huge_valf()};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        {
        const float4 a = lo[i], b = hi[i];
        const float c[3] = {(a.x + b.x) * 0.5f, (a.y + b.y) * 0.5f, (a.z + b.z) * 0.5f};
        for (int k = 0; k < 3; k++)
            {
            v[k] = fminf(v[k], c[k]);
            v[3 + k] = fmaxf(v[3 + k], c[k]);
            }
        }
    block_minmax(v, sh);
    if (threadIdx.x == 0)
        for (int k = 0; k < 6; k++)
            partial[6 * blockIdx.x + k] = v[k];
    }

__global__ void k_centroid_final(const float* partial, uint32_t n_part, float* out)
    {
    __shared__ float sh[6 * 256];
    float v[6] = {__builtin_huge_valf(), __builtin_huge_valf(), __builtin_huge_valf(),
                  -__builtin_huge_valf(), -__builtin_huge_valf(), -__builtin_huge_valf()};
    for (uint32_t i = threadIdx.x; i < n_part; i += blockDim.x)
        for (int k = 0; k < 6; k++)
            v[k] = (k < 3) ? fminf(v[k], partial[6 * i + k]) : fmaxf(v[k], partial[6 * i + k]);
    block_minmax(v, sh);
    if (threadIdx.x == 0)
        for (int k = 0; k < 6; k++)
            out[k] = v[k];
    }

// ---------------------------------------------------------------- morton
__device__ __forceinline__ uint32_t expand10(uint32_t x)
    {
    x &= 0x3ffu;
    x = (x | (x << 16)) & 0x030000ffu;
    x = (x | (x << 8)) & 0x0300f00fu;
    x = (x | (x << 4)) & 0x030c30c3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
    }
__device__ __forceinline__ uint32_t quant10(float c, float lo, float hi)
    {
    const float e = hi - lo;
    const float f = (e > 0.0f) ? (c - lo) / e : 0.5f;
    const float s = fminf(fmaxf(f * 1024.0f, 0.0f), 1023.0f);
    return (uint32_t)s;
    }
__global__ void k_morton(const float4* __restrict__ lo, const float4* __restrict__ hi, uint32_t N,
                         const float* __restrict__ cb, uint32_t* keys, uint32_t* vals)
    {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N)
        return;
    const float4 a = lo[i], b = hi[i];
    const uint32_t x = quant10((a.x + b.x) * 0.5f, cb[0], cb[3]);
    const uint32_t y = quant10((a.y + b.y) * 0.5f, cb[1], cb[4]);
    const uint32_t z = quant10((a.z + b.z) * 0.5f, cb[2], cb[5]);
    keys[i] = (expand10(x) << 2) | (expand10(y) << 1) | expand10(z);
    vals[i] = i;
    }

// ---------------------------------------------------------------- radix sort
// ITEMS keys per thread: a workgroup sorts SORT_BLOCK * ITEMS keys of a pass
// (its ranks take ITEMS dependent rounds).
template<int ITEMS>
__global__ __launch_bounds__(SORT_BLOCK) void k_radix_hist(const uint32_t* __restrict__ keys, uint32_t N,
                                                           uint32_t shift, uint32_t n_blocks, uint32_t* hist)
    {
    __shared__ uint32_t cnt[256];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t base = blockIdx.x * (SORT_BLOCK * ITEMS);
    for (int r = 0; r < ITEMS; r++)
        {
        const uint32_t i = base + r * SORT_BLOCK + threadIdx.x;
        if (i < N)
            atomicAdd(&cnt[(keys[i] >> shift) & 0xffu], 1u);
        }
    __syncthreads();
    hist[threadIdx.x * n_blocks + blockIdx.x] = cnt[threadIdx.x];
    }

// Exclusive scan of n uint32 in place: blocks of 2048 (256 x 8), then the
// block sums (at most 2048) in one block, then the add-back.
__device__ __forceinline__ uint32_t block_excl_scan256(uint32_t v, uint32_t* sh, uint32_t& total)
    {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (uint32_t off = 1; off < 256; off <<= 1)
        {
        const uint32_t t = (threadIdx.x >= off) ? sh[threadIdx.x - off] : 0u;
        __syncthreads();
        sh[threadIdx.x] += t;
        __syncthreads();
        }
    total = sh[255];
    const uint32_t incl = sh[threadIdx.x];
    __syncthreads();
    return incl - v;
    }
__global__ __launch_bounds__(256) void k_scan_blocks(uint32_t* data, uint32_t n, uint32_t* sums)
    {
    __shared__ uint32_t sh[256];
    const uint32_t base = blockIdx.x * 2048 + threadIdx.x * 8;
    uint32_t v[8], s = 0;
    for (int k = 0; k < 8; k++)
        {
        v[k] = (base + k < n) ? data[base + k] : 0u;
        s += v[k];
        }
    uint32_t total;
    uint32_t run = block_excl_scan256(s, sh, total);
    for (int k = 0; k < 8; k++)
        {
        if (base + k < n)
            data[base + k] = run;
        run += v[k];
        }
    if (threadIdx.x == 0)
        sums[blockIdx.x] = total;
    }
__global__ __launch_bounds__(256) void k_scan_top(uint32_t* sums, uint32_t n)
    {
    __shared__ uint32_t sh[256];
    const uint32_t base = threadIdx.x * 8;
    uint32_t v[8], s = 0;
    for (int k = 0; k < 8; k++)
        {
        v[k] = (base + k < n) ? sums[base + k] : 0u;
        s += v[k];
        }
    uint32_t total;
    uint32_t run = block_excl_scan256(s, sh, total);
    for (int k = 0; k < 8; k++)
        {
        if (base + k < n)
            sums[base + k] = run;
        run += v[k];
        }
    }
// Exclusive scan of n <= SCAN_SINGLE_MAX uint32 in place in one workgroup
// (1024 threads x 16 consecutive items): the scans of small builds take one
// launch instead of three.
constexpr uint32_t SCAN_SINGLE_MAX = 16384;
__global__ __launch_bounds__(1024) void k_scan_single(uint32_t* data, uint32_t n)
    {
    __shared__ uint32_t sh[1024];
    const uint32_t base = threadIdx.x * 16;
    uint32_t v[16], s = 0;
    for (int k = 0; k < 16; k++)
        {
        v[k] = (base + k < n) ? data[base + k] : 0u;
        s += v[k];
        }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t off = 1; off < 1024; off <<= 1)
        {
        const uint32_t t = (threadIdx.x >= off) ? sh[threadIdx.x - off] : 0u;
        __syncthreads();
        sh[threadIdx.x] += t;
        __syncthreads();
        }
    uint32_t run = sh[threadIdx.x] - s;
    for (int k = 0; k < 16; k++)
        {
        if (base + k < n)
            data[base + k] = run;
        run += v[k];
        }
    }
__global__ void k_scan_add(uint32_t* data, uint32_t n, const uint32_t* sums)
    {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        data[i] += sums[i / 2048];
    }

template<int ITEMS>
__global__ __launch_bounds__(SORT_BLOCK) void k_radix_scatter(const uint32_t* __restrict__ kin,
                                                              const uint32_t* __restrict__ vin, uint32_t* kout,
                                                              uint32_t* vout, uint32_t N, uint32_t shift,
                                                              uint32_t n_blocks, const uint32_t* __restrict__ offs)
    {
    constexpr int WAVES = SORT_BLOCK / 64;
    __shared__ uint32_t running[256];
    __shared__ uint32_t wcnt[WAVES * 256];
    running[threadIdx.x] = offs[threadIdx.x * n_blocks + blockIdx.x];
    for (int w = 0; w < WAVES; w++)
        wcnt[w * 256 + threadIdx.x] = 0;
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint64_t lt_mask = (1ull << lane) - 1ull;
    const uint32_t base = blockIdx.x * (SORT_BLOCK * ITEMS);
    for (int r = 0; r < ITEMS; r++)
        {
        const uint32_t i = base + r * SORT_BLOCK + threadIdx.x;
        const bool valid = i < N;
        const uint32_t key = valid ? kin[i] : 0u;
        const uint32_t val = valid ? vin[i] : 0u;
        const uint32_t digit = (key >> shift) & 0xffu;
        // lanes holding the same digit
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++)
            {
            const bool bit = (digit >> b) & 1u;
            const uint64_t m = __ballot(valid && bit);
            peers &= bit ? m : ~m;
            }
        const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
        if (valid && rank == 0)
            wcnt[wave * 256 + digit] = (uint32_t)__popcll(peers);
        __syncthreads();
        if (valid)
            {
            uint32_t pos = running[digit] + rank;
            for (uint32_t w = 0; w < wave; w++)
                pos += wcnt[w * 256 + digit];
            kout[pos] = key;
            vout[pos] = val;
            }
        __syncthreads();
        uint32_t add = 0;
        for (int w = 0; w < WAVES; w++)
            {
            add += wcnt[w * 256 + threadIdx.x];
            wcnt[w * 256 + threadIdx.x] = 0;
            }
        running[threadIdx.x] += add;
        __syncthreads();
        }
    }

// ---------------------------------------------------------------- karras
__device__ __forceinline__ int kdelta(const uint32_t* keys, int N, int i, int j)
    {
    if (j < 0 || j >= N)
        return -1;
    const uint64_t a = ((uint64_t)keys[i] << 32) | (uint32_t)i;
    const uint64_t b = ((uint64_t)keys[j] << 32) | (uint32_t)j;
    return __clzll(a ^ b);
    }

__device__ __forceinline__ void leaf_link(const uint32_t* vals, const float4* lo, const float4* hi, int p, uint32_t& c,
                                          uint32_t& g)
    {
    const uint32_t orig = vals[p];
    g = __float_as_uint(lo[orig].w);
    c = LEAF | __float_as_uint(hi[orig].w);
    }

// Internal node i of N-1; parent[] holds (parent << 1 | side) for inner nodes
// [0, N-1) and leaves [N-1, 2N-1).
__global__ void k_karras(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                         const float4* __restrict__ lo, const float4* __restrict__ hi, int N, Node* nodes,
                         uint32_t* parent)
    {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N - 1)
        return;
    const int d = (kdelta(keys, N, i, i + 1) - kdelta(keys, N, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = kdelta(keys, N, i, i - d);
    int lmax = 2;
    while (kdelta(keys, N, i, i + lmax * d) > dmin)
        lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (kdelta(keys, N, i, i + (l + t) * d) > dmin)
            l += t;
    const int j = i + l * d;
    const int dnode = kdelta(keys, N, i, j);
    int s = 0;
    for (int div = 2;; div <<= 1)
        {
        const int t = (l + div - 1) / div;
        if (kdelta(keys, N, i, i + (s + t) * d) > dnode)
            s += t;
        if (t <= 1)
            break;
        }
    const int gamma = i + s * d + (d < 0 ? d : 0);
    uint32_t c0, c1, g0 = 0, g1 = 0;
    const int first = i < j ? i : j, last = i < j ? j : i;
    if (first == gamma)
        {
        leaf_link(vals, lo, hi, gamma, c0, g0);
        parent[(N - 1) + gamma] = (uint32_t)(i << 1);
        }
    else
        {
        c0 = (uint32_t)gamma;
        parent[gamma] = (uint32_t)(i << 1);
        }
    if (last == gamma + 1)
        {
        leaf_link(vals, lo, hi, gamma + 1, c1, g1);
        parent[(N - 1) + gamma + 1] = (uint32_t)(i << 1) | 1u;
        }
    else
        {
        c1 = (uint32_t)(gamma + 1);
        parent[gamma + 1] = (uint32_t)(i << 1) | 1u;
        }
    nodes[i].link = make_uint4(c0, c1, g0, g1);
    }

// Data of the leaf at position p (primitive bounds a, b) for the 4-wide
// search (SceneDev::leaf): neighbours in space lie next to each other.
__device__ __forceinline__ void store_leaf(uint32_t p, float4 a, float4 b, const GeomDev* __restrict__ sphere_geoms,
                                           float4* __restrict__ leaf, uint2* __restrict__ leaf_ref)
    {
    if (sphere_geoms)
        {
        const uint32_t slot = __float_as_uint(a.w), prim = __float_as_uint(b.w);
        leaf[p] = sphere_geoms[slot].a[prim];
        leaf_ref[p] = make_uint2(slot, prim);
        }
    else
        {
        leaf[2 * (size_t)p] = a;
        leaf[2 * (size_t)p + 1] = b;
        }
    }

// One-primitive scene: root with the leaf and an EMPTY child whose NaN box
// fails every slab test.
__global__ void k_single_leaf(const float4* __restrict__ lo, const float4* __restrict__ hi, Node* nodes,
                              const GeomDev* __restrict__ sphere_geoms, float4* __restrict__ leaf,
                              uint2* __restrict__ leaf_ref)
    {
    const float4 a = lo[0], b = hi[0];
    const float nan = __builtin_nanf("");
    nodes[0].a_lo = make_float4(a.x, a.y, a.z, b.x);
    nodes[0].a_hi = make_float4(b.y, b.z, nan, nan);
    nodes[0].b_box = make_float4(nan, nan, nan, nan);
    nodes[0].link = make_uint4(LEAF | __float_as_uint(b.w), EMPTY, __float_as_uint(a.w), 0u);
    store_leaf(0, a, b, sphere_geoms, leaf, leaf_ref);
    }

// ---------------------------------------------------------------- refit
__device__ __forceinline__ void store_box(Node* n, uint32_t side, const float b[6])
    {
    float* f = reinterpret_cast<float*>(n);
    const int o = side ? 6 : 0;
    for (int k = 0; k < 6; k++)
        __hip_atomic_store(f + o + k, b[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
__device__ __forceinline__ void load_box(Node* n, uint32_t side, float b[6])
    {
    float* f = reinterpret_cast<float*>(n);
    const int o = side ? 6 : 0;
    for (int k = 0; k < 6; k++)
        b[k] = __hip_atomic_load(f + o + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

__global__ void k_refit(const uint32_t* __restrict__ vals, const float4* __restrict__ lo,
                        const float4* __restrict__ hi, int N, Node* nodes, const uint32_t* __restrict__ parent,
                        uint32_t* flags, float* root_box, const GeomDev* __restrict__ sphere_geoms,
                        float4* __restrict__ leaf, uint2* __restrict__ leaf_ref)
    {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N)
        return;
    const uint32_t orig = vals[p];
    const float4 a = lo[orig], b = hi[orig];
    store_leaf((uint32_t)p, a, b, sphere_geoms, leaf, leaf_ref);
    float box[6] = {a.x, a.y, a.z, b.x, b.y, b.z};
    uint32_t par = parent[(N - 1) + p];
    for (;;)
        {
        const uint32_t node = par >> 1;
        // Boxes and flags are device-scope atomics, which are coherent across
        // the XCDs' L2 caches without flushing them.  s_waitcnt 0 (every
        // counter of this wave drained) makes the box stores complete at the
        // device coherence point before the flag increment is issued; the
        // sibling's box loads are issued only after its increment returned 1.
        // A device-scope fence here would write back and invalidate the whole
        // L2 once per thread and level.
        // The compiler sees only relaxed atomics to different addresses and an
        // intrinsic it models as touching no memory, so the signal fences
        // (compiler barriers, no instruction) keep the box stores before the
        // wait and the increment, and the sibling's box loads after its
        // increment, in program order; the wait then orders them in hardware.
        store_box(nodes + node, par & 1u, box);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        const uint32_t prev = __hip_atomic_fetch_add(flags + node, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        if (prev == 0)
            return; // the sibling finishes this node
        float b0[6], b1[6];
        load_box(nodes + node, 0, b0);
        load_box(nodes + node, 1, b1);
        for (int k = 0; k < 3; k++)
            {
            box[k] = fminf(b0[k], b1[k]);
            box[3 + k] = fmaxf(b0[3 + k], b1[3 + k]);
            }
        if (node == 0)
            {
            for (int k = 0; k < 6; k++)
                root_box[k] = box[k];
            return;
            }
        par = parent[node];
        }
    }
// ---------------------------------------------------------------- 4-wide hierarchy
// The binary hierarchy's inner nodes at even depth become the nodes of a
// 4-wide hierarchy whose children are their grandchildren (a child that is a
// leaf stays a child), so a search makes half as many dependent node fetches.
// The binary tree is the one built and refit; the 4-wide nodes hold its boxes
// rounded outwards
// (k_bvh4_fill after every build and refit, the topology from k_depth_even and
// a scan of its flags).

// even[i] = 1 for inner nodes at even depth (the root has depth 0); even[n] = 0.
__global__ void k_depth_even(const uint32_t* __restrict__ parent, uint32_t n, uint32_t* even)
    {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n)
        return;
    if (i == n)
        {
        even[n] = 0;
        return;
        }
    uint32_t d = 0;
    for (uint32_t k = i; k != 0; k = parent[k] >> 1)
        d++;
    even[i] = (d & 1u) ? 0u : 1u;
    }

__device__ __forceinline__ void child_box(const Node& n, uint32_t side, float b[6])
    {
    if (side == 0)
        {
        b[0] = n.a_lo.x; b[1] = n.a_lo.y; b[2] = n.a_lo.z;
        b[3] = n.a_lo.w; b[4] = n.a_hi.x; b[5] = n.a_hi.y;
        }
    else
        {
        b[0] = n.a_hi.z; b[1] = n.a_hi.w; b[2] = n.b_box.x;
        b[3] = n.b_box.y; b[4] = n.b_box.z; b[5] = n.b_box.w;
        }
    }

// 4-wide node idx4[i] from inner node i of n, for the nodes at even depth:
// idx4 is the exclusive scan of k_depth_even's flags (n + 1 entries).  A leaf
// child is referred to by its position in leaf order (k_karras's key order).
// On each axis the children's boxes are rounded outwards to 8-bit steps of
// the node's own interval, after a pad of 2^-22 of that interval's width, what
// the search's slab test loses to rounding (search_visit), and of 2^-24 of the
// node's largest coordinate, for the roundings here and for rays along a box's
// face (node_rcp).  (A pad of 2^-20 of the coordinate opened what lies beside a
// ray far from the origin: 100,000 spheres of radius 0.5 moved by 10^6, 16
// samples, 800 x 600, 5.1 ms and 38 node visits a ray, so 2.0 and 14.6.)
// An end that is infinite, NaN or beyond 2^66 becomes -2^66 (a low end) or 2^66
// (a high one), the largest interval whose slab test cannot overflow (2^67
// times RCP_MAX, 2^60), above the 2^64 at which squared distances overflow in
// the primitives' own tests; only that axis takes their pad.  A primitive's own
// bounds are tested exactly at its leaf, so one out there is still found by
// every ray that starts within.
__global__ void k_bvh4_fill(const Node* __restrict__ nodes, uint32_t n, const uint32_t* __restrict__ idx4,
                            const uint32_t* __restrict__ parent, Node4* __restrict__ out)
    {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || idx4[i + 1] == idx4[i])
        return;
    float box[4][6];
    uint32_t ref[4];
    uint32_t m = 0;
    // leaf position of child `side` of binary node j (split position g: the
    // children's key ranges end at g and begin at g + 1, and an inner child's
    // index is that end); a node of two leaves is one of their positions
    auto leaf_position = [&](uint32_t j, const uint4& l, uint32_t side)
    {
        uint32_t g;
        if (l.y == EMPTY)
            g = 0; // one-primitive scene
        else if (!(l.x & LEAF))
            g = l.x;
        else if (!(l.y & LEAF))
            g = l.y - 1;
        else
            g = (parent[n + j] == (j << 1)) ? j : j - 1;
        return g + side;
    };
    const Node a = nodes[i];
    const uint32_t la[2] = {a.link.x, a.link.y};
    for (uint32_t s = 0; s < 2; s++)
        {
        if (la[s] & LEAF) // a leaf or EMPTY (not a child)
            {
            child_box(a, s, box[m]);
            ref[m] = LEAF | leaf_position(i, a.link, s);
            if (la[s] != EMPTY)
                m++;
            continue;
            }
        const Node b = nodes[la[s]];
        const uint32_t lb[2] = {b.link.x, b.link.y};
        for (uint32_t t = 0; t < 2; t++)
            {
            child_box(b, t, box[m]);
            ref[m] = (lb[t] & LEAF) ? (LEAF | leaf_position(la[s], b.link, t)) : idx4[lb[t]];
            m++;
            }
        }
    if (m == 1)
        {
        // one-primitive scene: its leaf twice
        for (int x = 0; x < 6; x++)
            box[1][x] = box[0][x];
        ref[1] = ref[0];
        m = 2;
        }
    // a box of NaN alone (primitives of NaN positions, and nodes of nothing
    // else) lets no ray pass its slab test: that child is closed, high below low
    constexpr float FAR = 0x1p66f;
    bool closed[4];
    bool far[3] = {false, false, false};
    float big = 0.0f;
    for (uint32_t k = 0; k < m; k++)
        {
        closed[k] = true;
        for (int x = 0; x < 6; x++)
            closed[k] = closed[k] && box[k][x] != box[k][x];
        for (int x = 0; x < 6 && !closed[k]; x++)
            {
            if (fabsf(box[k][x]) <= FAR)
                big = fmaxf(big, fabsf(box[k][x]));
            else
                {
                box[k][x] = (x < 3) ? -FAR : FAR;
                far[x % 3] = true;
                }
            }
        }
    Node4 r;
    for (int x = 0; x < 3; x++)
        {
        // swapped ends (a negative radius) count as the interval between them
        double lo = 1e300, hi = -1e300;
        for (uint32_t k = 0; k < m; k++)
            if (!closed[k])
                {
                lo = fmin(lo, (double)fminf(box[k][x], box[k][3 + x]));
                hi = fmax(hi, (double)fmaxf(box[k][x], box[k][3 + x]));
                }
        if (!(lo <= hi))
            {
            // every child closed: ends as far apart as can be
            lo = -(double)FAR;
            hi = (double)FAR;
            far[x] = true;
            }
        const double pad = NODE_PAD * (hi - lo) + NODE_PAD_FLOOR * (far[x] ? FAR : big);
        // origin rounded down, 255 steps from it reach the high end
        float org = (float)(lo - pad);
        if ((double)org > lo - pad)
            org = nextafterf(org, -__builtin_huge_valf());
        float step = fmaxf((float)((hi + pad - (double)org) * (1.0 / 255.0)), 0x1p-126f);
        if ((double)step * 255.0 < hi + pad - (double)org)
            step = nextafterf(step, __builtin_huge_valf());
        const double per_step = 1.0 / (double)step;
        uint32_t ql = 0, qh = 0;
        for (uint32_t k = 0; k < m; k++)
            {
            const double a = (double)fminf(box[k][x], box[k][3 + x]) - pad - (double)org;
            const double b = (double)fmaxf(box[k][x], box[k][3 + x]) + pad - (double)org;
            const double fa = closed[k] ? 255.0 : floor(a * per_step);
            const double fb = closed[k] ? 0.0 : ceil(b * per_step);
            ql |= (uint32_t)fmin(fmax(fa, 0.0), 255.0) << (8 * k);
            qh |= (uint32_t)fmin(fmax(fb, 0.0), 255.0) << (8 * k);
            }
        r.o[x] = org;
        r.s[x] = step;
        r.qlo[x] = ql;
        r.qhi[x] = qh;
        }
    for (uint32_t k = 0; k < 4; k++)
        r.ref[k] = (k < m) ? ref[k] : EMPTY;
    out[idx4[i]] = r;
    }

// ---------------------------------------------------------------- quality
// Surface-area cost of a hierarchy: the sum over internal nodes of their two
// child boxes' half surface areas.  A random ray visits a node with
// probability proportional to its box's area, so the sum tracks traversal
// cost; the refit policy compares it with the value right after a build.
__device__ __forceinline__ float half_area(float x0, float y0, float z0, float x1, float y1, float z1)
    {
    const float dx = x1 - x0, dy = y1 - y0, dz = z1 - z0;
    return dx * dy + dy * dz + dz * dx;
    }

__device__ __forceinline__ float block_sum(float v, float* sh)
    {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1)
        {
        if (threadIdx.x < s)
            sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
        }
    return sh[0];
    }

// Largest primitive half-extent of the scene (sets the traversal's cull margin).
__device__ __forceinline__ float block_maxf(float v, float* sh)
    {
    sh[threadIdx.x] = v;
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1)
        {
        if (threadIdx.x < s)
            sh[threadIdx.x] = fmaxf(sh[threadIdx.x], sh[threadIdx.x + s]);
        __syncthreads();
        }
    return sh[0];
    }

__global__ void k_extent_partial(const float4* __restrict__ lo, const float4* __restrict__ hi, uint32_t N,
                                 float* partial)
    {
    __shared__ float sh[256];
    float v = 0.0f;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        {
        const float4 a = lo[i], b = hi[i];
        v = fmaxf(v, fmaxf(fmaxf(b.x - a.x, b.y - a.y), b.z - a.z) * 0.5f);
        }
    v = block_maxf(v, sh);
    if (threadIdx.x == 0)
        partial[blockIdx.x] = v;
    }

__global__ void k_extent_final(const float* __restrict__ partial, uint32_t n_part, float* out)
    {
    __shared__ float sh[256];
    float v = 0.0f;
    for (uint32_t i = threadIdx.x; i < n_part; i += blockDim.x)
        v = fmaxf(v, partial[i]);
    v = block_maxf(v, sh);
    if (threadIdx.x == 0)
        out[0] = v;
    }

__global__ void k_sah_partial(const Node* __restrict__ nodes, uint32_t n_nodes, float* partial)
    {
    __shared__ float sh[256];
    float v = 0.0f;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n_nodes; i += gridDim.x * blockDim.x)
        {
        const Node n = nodes[i];
        v += half_area(n.a_lo.x, n.a_lo.y, n.a_lo.z, n.a_lo.w, n.a_hi.x, n.a_hi.y);
        if (n.link.y != EMPTY)
            v += half_area(n.a_hi.z, n.a_hi.w, n.b_box.x, n.b_box.y, n.b_box.z, n.b_box.w);
        }
    v = block_sum(v, sh);
    if (threadIdx.x == 0)
        partial[blockIdx.x] = v;
    }

__global__ void k_sah_final(const float* __restrict__ partial, uint32_t n_part, float* out)
    {
    __shared__ float sh[256];
    float v = 0.0f;
    for (uint32_t i = threadIdx.x; i < n_part; i += blockDim.x)
        v += partial[i];
    v = block_sum(v, sh);
    if (threadIdx.x == 0)
        out[0] = v;
    }
    } // namespace fh
