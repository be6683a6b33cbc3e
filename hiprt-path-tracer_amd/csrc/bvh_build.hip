// bvh_build.hip -- GPU LBVH builder (replaces hiprtBuildGeometry,
// src/HIPRT-Orochi/HIPRTScene.h:87-150, whose implementation lives in the
// absent HIPRT library).
//
// Pipeline (all on the device, one stream):
//   1. per-triangle boxes + scene/centroid bounds (block partials, folded
//      without atomics)
//   2. 63-bit Morton code of each box centre (21 bits per axis)
//   3. radix sort (Morton, primitive) pairs
//   4. Karras 2012 hierarchy: node i of n-1 interior nodes from the key prefixes
//   5. bottom-up refit with arrival counters; each node also gets its SAH cost
//      and a collapse flag (subtree of <= MAX_LEAF_SIZE triangles becomes one
//      leaf when that is cheaper)
//   6. emit 64-byte BvhNodes and 48-byte TriRecords in Morton order.
// Boxes are padded (bvh_common.h). finalize_bvh validates the tree, computes its
// statistics and lays it out depth first for both builders, on the device: as
// host passes over a copy of the tree that took 85 of the 107 ms of a build of
// 1,040,384 triangles.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include <rocprim/rocprim.hpp>

#include "bvh_common.h"

namespace mipt {
namespace {

using bvhc::f2o;
using bvhc::f4max;
using bvhc::f4min;
using bvhc::half_area;
using bvhc::o2f;
using bvhc::SAH_C_NODE;
using bvhc::SAH_C_TRI;

__device__ __forceinline__ uint64_t expand21(uint64_t v)
{
    v &= 0x1fffffull;
    v = (v | (v << 32)) & 0x1f00000000ffffull;
    v = (v | (v << 16)) & 0x1f0000ff0000ffull;
    v = (v | (v << 8)) & 0x100f00f00f00f00full;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}

// Codes, and what the later kernels find set: no visits, no parents, nothing
// collapsed (four memsets, seven kernels, otherwise).
__global__ void k_morton(const float4* __restrict__ lo, const float4* __restrict__ hi, int32_t n,
                         const uint32_t* __restrict__ bounds, uint64_t* __restrict__ keys,
                         uint32_t* __restrict__ vals, int32_t ninner, uint32_t* __restrict__ visits,
                         int32_t* __restrict__ node_parent, int32_t* __restrict__ leaf_parent,
                         uint8_t* __restrict__ collapse)
{
    int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    leaf_parent[i] = -1;
    if (i < ninner)
    {
        visits[i] = 0u;
        node_parent[i] = -1;
        collapse[i] = 0;
    }
    float clo[3], cext[3];
    for (int k = 0; k < 3; k++)
    {
        clo[k] = o2f(bounds[6 + k]);
        float e = o2f(bounds[9 + k]) - clo[k];
        cext[k] = e > 0.0f ? e : 1.0f;
    }
    float4 a = lo[i], b = hi[i];
    float c[3] = {0.5f * (a.x + b.x), 0.5f * (a.y + b.y), 0.5f * (a.z + b.z)};
    uint64_t code = 0;
    for (int k = 0; k < 3; k++)
    {
        float f = (c[k] - clo[k]) / cext[k];
        f = fminf(fmaxf(f, 0.0f), 1.0f);
        uint64_t q = (uint64_t)fminf(f * 2097152.0f, 2097151.0f);
        code |= expand21(q) << (2 - k);
    }
    keys[i] = code;
    vals[i] = (uint32_t)i;
}

__device__ __forceinline__ int delta(const uint64_t* __restrict__ keys, int32_t n, int32_t i, int32_t j)
{
    if (j < 0 || j >= n)
        return -1;
    uint64_t x = keys[i] ^ keys[j];
    if (x == 0)
        return 64 + __clz((uint32_t)(i ^ j));
    return __clzll(x);
}

// Karras 2012, "Maximizing Parallelism in the Construction of BVHs, Octrees,
// and k-d Trees", Figure 4. Child refs: >= 0 interior node, < 0 ~leaf index.
__global__ void k_karras(const uint64_t* __restrict__ keys, int32_t n, int32_t* __restrict__ child,
                         int32_t* __restrict__ node_parent, int32_t* __restrict__ leaf_parent,
                         int32_t* __restrict__ range_lo, int32_t* __restrict__ range_hi)
{
    int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1)
        return;
    int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = delta(keys, n, i, i - d);
    int32_t lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin)
        lmax *= 2;
    int32_t l = 0;
    for (int32_t t = lmax / 2; t >= 1; t /= 2)
        if (delta(keys, n, i, i + (l + t) * d) > dmin)
            l += t;
    int32_t j = i + l * d;
    int dnode = delta(keys, n, i, j);
    int32_t s = 0;
    int32_t t = l;
    do
    {
        t = (t + 1) / 2;
        if (delta(keys, n, i, i + (s + t) * d) > dnode)
            s += t;
    } while (t > 1);
    int32_t gamma = i + s * d + (d < 0 ? -1 : 0);
    int32_t first = i < j ? i : j;
    int32_t last = i < j ? j : i;
    int32_t left = (first == gamma) ? ~gamma : gamma;
    int32_t right = (last == gamma + 1) ? ~(gamma + 1) : gamma + 1;
    child[2 * i] = left;
    child[2 * i + 1] = right;
    if (left < 0) leaf_parent[~left] = i; else node_parent[left] = i;
    if (right < 0) leaf_parent[~right] = i; else node_parent[right] = i;
    range_lo[i] = first;
    range_hi[i] = last;
    if (i == 0)
        node_parent[0] = -1;
}

// Padded box of sorted leaf k.
__device__ __forceinline__ void leaf_box(const float4* __restrict__ plo, const float4* __restrict__ phi,
                                         const uint32_t* __restrict__ vals, int32_t k, float abs_pad,
                                         float4& lo, float4& hi)
{
    const uint32_t p = vals[k];
    bvhc::pad_box(plo[p], phi[p], abs_pad, lo, hi);
}

__global__ void k_refit(int32_t n, const float4* __restrict__ plo, const float4* __restrict__ phi,
                        const uint32_t* __restrict__ vals, const int32_t* __restrict__ child,
                        const int32_t* __restrict__ node_parent, const int32_t* __restrict__ leaf_parent,
                        const int32_t* __restrict__ range_lo, const int32_t* __restrict__ range_hi,
                        uint32_t* __restrict__ visits, float4* __restrict__ nlo, float4* __restrict__ nhi,
                        float* __restrict__ cost, uint8_t* __restrict__ collapse, const float* __restrict__ pad)
{
    int32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n)
        return;
    const float abs_pad = pad[0];
    int32_t p = leaf_parent[k];
    // A binary radix tree over distinct 96-bit (key, index) prefixes is at
    // most 96 levels deep; the bound only guards against a malformed tree.
    for (int level = 0; p >= 0 && p < n - 1 && level < 128; level++)
    {
        __threadfence();
        if (atomicAdd(&visits[p], 1u) == 0)
            return; // the other child is not done yet; its thread continues
        __threadfence();
        float4 lo[2], hi[2];
        float c[2];
        for (int s = 0; s < 2; s++)
        {
            int32_t ch = child[2 * p + s];
            if (ch < 0)
            {
                leaf_box(plo, phi, vals, ~ch, abs_pad, lo[s], hi[s]);
                c[s] = half_area(lo[s], hi[s]) * SAH_C_TRI;
            }
            else
            {
                lo[s] = nlo[ch];
                hi[s] = nhi[ch];
                c[s] = cost[ch];
            }
        }
        float4 blo = f4min(lo[0], lo[1]), bhi = f4max(hi[0], hi[1]);
        float a = half_area(blo, bhi);
        int32_t count = range_hi[p] - range_lo[p] + 1;
        float c_split = a * SAH_C_NODE + c[0] + c[1];
        float c_leaf = a * (float)count * SAH_C_TRI;
        bool as_leaf = count <= MAX_LEAF_SIZE && c_leaf <= c_split;
        nlo[p] = blo;
        nhi[p] = bhi;
        cost[p] = as_leaf ? c_leaf : c_split;
        collapse[p] = as_leaf ? 1 : 0;
        p = node_parent[p];
    }
}

__global__ void k_emit_nodes(int32_t n, const float4* __restrict__ plo, const float4* __restrict__ phi,
                             const uint32_t* __restrict__ vals, const int32_t* __restrict__ child,
                             const int32_t* __restrict__ range_lo, const int32_t* __restrict__ range_hi,
                             const float4* __restrict__ nlo, const float4* __restrict__ nhi,
                             const uint8_t* __restrict__ collapse, const float* __restrict__ pad,
                             const int32_t* __restrict__ node_parent, BvhNode* __restrict__ nodes)
{
    int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1)
        return;
    // depth, and whether a collapsed node (a leaf of the tree) lies on the
    // way to the root; at most 96 levels (see k_refit)
    int32_t depth = 0;
    bool unused = false;
    for (int32_t p = i; p > 0 && depth < 128; p = node_parent[p], depth++)
        unused |= collapse[p] != 0;
    if (unused)
    {
        nodes[i].d = make_int4(0, 0, 0, NODE_UNUSED);
        return;
    }
    float4 lo[2], hi[2];
    int32_t ref[2];
    for (int s = 0; s < 2; s++)
    {
        int32_t ch = child[2 * i + s];
        if (ch < 0)
        {
            leaf_box(plo, phi, vals, ~ch, pad[0], lo[s], hi[s]);
            ref[s] = make_leaf(~ch, 1);
        }
        else
        {
            lo[s] = nlo[ch];
            hi[s] = nhi[ch];
            ref[s] = collapse[ch] ? make_leaf(range_lo[ch], range_hi[ch] - range_lo[ch] + 1) : ch;
        }
    }
    BvhNode nd;
    nd.a = make_float4(lo[0].x, lo[0].y, lo[0].z, hi[0].x);
    nd.b = make_float4(hi[0].y, hi[0].z, lo[1].x, lo[1].y);
    nd.c = make_float4(lo[1].z, hi[1].x, hi[1].y, hi[1].z);
    nd.d = make_int4(ref[0], ref[1], range_lo[i], depth);
    nodes[i] = nd;
}

using bvhc::blocks;

} // namespace

void write_single_triangle_root(BvhNode* d_node, const float4* d_lo, const float4* d_hi)
{
    float4 lo, hi;
    HIP_CHECK(hipMemcpy(&lo, d_lo, sizeof(float4), hipMemcpyDeviceToHost));
    HIP_CHECK(hipMemcpy(&hi, d_hi, sizeof(float4), hipMemcpyDeviceToHost));
    const float ext = std::max({hi.x - lo.x, hi.y - lo.y, hi.z - lo.z});
    float4 plo, phi;
    bvhc::pad_box(lo, hi, ext * bvhc::PAD_ABS, plo, phi);
    BvhNode nd;
    nd.a = make_float4(plo.x, plo.y, plo.z, phi.x);
    // Empty second child: every slab of an all-(+inf) box is at +inf or -inf,
    // so the box test always fails.
    nd.b = make_float4(phi.y, phi.z, INFINITY, INFINITY);
    nd.c = make_float4(INFINITY, INFINITY, INFINITY, INFINITY);
    nd.d = make_int4(make_leaf(0, 1), make_leaf(0, 1), 0, 0);
    HIP_CHECK(hipMemcpy(d_node, &nd, sizeof(nd), hipMemcpyHostToDevice));
}

namespace {

constexpr int CHECK_BLOCK = 256;
constexpr int TREE_BLOCK = 1024;
// Triangles up to which one block checks and lays out the tree, in LDS.
constexpr int32_t TREE_SMALL = 4096;

__device__ __forceinline__ double box_area(float lx, float ly, float lz, float hx, float hy, float hz)
{
    const double dx = (double)hx - lx, dy = (double)hy - ly, dz = (double)hz - lz;
    if (dx < 0 || dy < 0 || dz < 0)
        return 0.0;
    return dx * dy + dy * dz + dz * dx;
}

__device__ __forceinline__ double root_box_area(const BvhNode& nd, int32_t n)
{
    return n == 1 ? box_area(nd.a.x, nd.a.y, nd.a.z, nd.a.w, nd.b.x, nd.b.y)
                  : box_area(fminf(nd.a.x, nd.b.z), fminf(nd.a.y, nd.b.w), fminf(nd.a.z, nd.c.x),
                             fmaxf(nd.a.w, nd.c.y), fmaxf(nd.b.x, nd.c.z), fmaxf(nd.b.y, nd.c.w));
}

// Checks node j and its children and adds them up. start(begin, depth)
// records a node whose range starts at triangle `begin`; see_node(r) and see_tri(q)
// mark a node as referenced and a triangle as held, and say whether they were.
template <class Start, class SeeNode, class SeeTri>
__device__ __forceinline__ void check_node(const BvhNode* __restrict__ nodes, int32_t j, int32_t count, int32_t n,
                                           TreeStats& t, const Start& start, const SeeNode& see_node,
                                           const SeeTri& see_tri)
{
    const BvhNode nd = nodes[j];
    const int32_t begin = nd.d.z, depth = nd.d.w;
    if (depth == NODE_UNUSED)
        return;
    t.inner++;
    if (begin < 0 || begin >= n || depth < 0 || (depth == 0) != (j == 0))
    {
        t.errors++;
        return;
    }
    start(begin, depth);
    const double area[2] = {box_area(nd.a.x, nd.a.y, nd.a.z, nd.a.w, nd.b.x, nd.b.y),
                            box_area(nd.b.z, nd.b.w, nd.c.x, nd.c.y, nd.c.z, nd.c.w)};
    const int32_t refs[2] = {nd.d.x, nd.d.y};
    for (int s = 0; s < (n == 1 ? 1 : 2); s++)
    {
        const int32_t r = refs[s];
        if (r >= 0)
        {
            t.sah += SAH_C_NODE * area[s];
            if (r >= count || nodes[r].d.w != depth + 1 || (s == 0 && nodes[r].d.z != begin) || see_node(r))
                t.errors++;
            continue;
        }
        const int32_t first = leaf_first(r), cnt = leaf_count(r);
        t.leaves++;
        t.max_leaf = max(t.max_leaf, (uint32_t)cnt);
        t.max_depth = max(t.max_depth, (uint32_t)depth + 1u);
        t.sah += SAH_C_TRI * cnt * area[s];
        if (first < 0 || first + cnt > n || (s == 0 && first != begin))
        {
            t.errors++;
            continue;
        }
        for (int32_t q = first; q < first + cnt; q++)
            t.errors += see_tri(q) ? 1u : 0u;
    }
}

// Sums over the block, in thread 0; `part` holds a record per wave.
template <int BLOCK> __device__ __forceinline__ TreeStats block_sum(TreeStats t, TreeStats* part)
{
    for (int off = 32; off > 0; off >>= 1)
    {
        t.sah += __shfl_xor(t.sah, off, 64);
        t.inner += __shfl_xor(t.inner, off, 64);
        t.leaves += __shfl_xor(t.leaves, off, 64);
        t.errors += __shfl_xor(t.errors, off, 64);
        t.max_depth = max(t.max_depth, (uint32_t)__shfl_xor(t.max_depth, off, 64));
        t.max_leaf = max(t.max_leaf, (uint32_t)__shfl_xor(t.max_leaf, off, 64));
    }
    if ((threadIdx.x & 63) == 0)
        part[threadIdx.x / 64] = t;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < BLOCK / 64; w++)
        {
            t.sah += part[w].sah;
            t.inner += part[w].inner;
            t.leaves += part[w].leaves;
            t.errors += part[w].errors;
            t.max_depth = max(t.max_depth, part[w].max_depth);
            t.max_leaf = max(t.max_leaf, part[w].max_leaf);
        }
    return t;
}

// Nodes whose range starts at the same triangle are a chain of first children,
// so a node's place in the depth-first order is the number of nodes that start
// before it, plus its depth below the chain's top.
__device__ __forceinline__ void lay_out(const BvhNode* __restrict__ nodes, int32_t j, int32_t n,
                                        const uint32_t* before, const int32_t* top_depth, BvhNode* __restrict__ out)
{
    BvhNode nd = nodes[j];
    if (nd.d.w == NODE_UNUSED)
        return;
    auto place = [&](const int4 d) { return (int32_t)before[d.z] + d.w - top_depth[d.z]; };
    const int32_t at = place(nd.d);
    if (nd.d.x >= 0)
        nd.d.x = place(nodes[nd.d.x].d);
    if (nd.d.y >= 0 && n > 1)
        nd.d.y = place(nodes[nd.d.y].d);
    nd.d.z = nd.d.w = 0;
    out[at] = nd;
}

__global__ void k_check_init(uint32_t* __restrict__ tri_seen, uint32_t* __restrict__ starts,
                             int32_t* __restrict__ top_depth, int32_t n, uint32_t* __restrict__ node_seen, int32_t count)
{
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
    {
        tri_seen[i] = 0u;
        starts[i] = 0u;
        top_depth[i] = 0x7fffffff;
    }
    if (i < count)
        node_seen[i] = 0u;
}

// Checks every node, adds up the statistics per block, and counts the nodes whose
// range starts at each triangle, with the depth of the topmost. A last record holds
// the root's area in sah.
__global__ __launch_bounds__(CHECK_BLOCK) void k_tree_check(const BvhNode* __restrict__ nodes, int32_t count, int32_t n,
                                                            uint32_t* __restrict__ tri_seen,
                                                            uint32_t* __restrict__ node_seen,
                                                            uint32_t* __restrict__ starts,
                                                            int32_t* __restrict__ top_depth,
                                                            TreeStats* __restrict__ stats)
{
    __shared__ TreeStats part[CHECK_BLOCK / 64];
    const int32_t j = blockIdx.x * CHECK_BLOCK + threadIdx.x;
    TreeStats t{};
    if (j == 0)
        stats[gridDim.x].sah = root_box_area(nodes[0], n);
    if (j < count)
        check_node(
            nodes, j, count, n, t,
            [&](int32_t begin, int32_t depth) {
                atomicAdd(&starts[begin], 1u);
                atomicMin(&top_depth[begin], depth);
            },
            [&](int32_t r) { return atomicAdd(&node_seen[r], 1u) != 0u; },
            [&](int32_t q) { return atomicAdd(&tri_seen[q], 1u) != 0u; });
    t = block_sum<CHECK_BLOCK>(t, part);
    if (threadIdx.x == 0)
        stats[blockIdx.x] = t;
}

// Every used node but the root is referenced (once: k_tree_check), every
// triangle seen; the rest adds to the errors of block 0's record.
__global__ void k_tree_complete(const BvhNode* __restrict__ nodes, int32_t count, int32_t n,
                                const uint32_t* __restrict__ tri_seen, const uint32_t* __restrict__ node_seen,
                                TreeStats* __restrict__ stats)
{
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool bad = i < n && tri_seen[i] == 0u;
    if (i < count && i > 0 && nodes[i].d.w != NODE_UNUSED)
        bad |= node_seen[i] == 0u;
    if (bad)
        atomicAdd(&stats[0].errors, 1u);
}

__global__ void k_tree_layout(const BvhNode* __restrict__ nodes, int32_t count, int32_t n,
                              const uint32_t* __restrict__ before, const int32_t* __restrict__ top_depth,
                              BvhNode* __restrict__ out)
{
    const int32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < count)
        lay_out(nodes, j, n, before, top_depth, out);
}

// The same for a tree of at most TREE_SMALL triangles in one block, without the
// host between check and layout: a tree with errors is not laid out.
__global__ __launch_bounds__(TREE_BLOCK) void k_tree_small(const BvhNode* __restrict__ nodes, int32_t count, int32_t n,
                                                           BvhNode* __restrict__ out, TreeReport* __restrict__ report)
{
    __shared__ uint32_t starts[TREE_SMALL]; // nodes that start at a triangle, then before it
    __shared__ int32_t top_depth[TREE_SMALL];
    __shared__ uint32_t tri_seen[TREE_SMALL / 32], node_seen[TREE_SMALL / 32];
    __shared__ TreeStats part[TREE_BLOCK / 64];
    __shared__ uint32_t wave_total[TREE_BLOCK / 64];
    __shared__ uint32_t missing, errors;
    const int32_t tid = (int32_t)threadIdx.x;
    for (int32_t i = tid; i < TREE_SMALL; i += TREE_BLOCK)
    {
        starts[i] = 0u;
        top_depth[i] = 0x7fffffff;
    }
    if (tid < TREE_SMALL / 32)
        tri_seen[tid] = node_seen[tid] = 0u;
    if (tid == 0)
        missing = 0u;
    __syncthreads();
    TreeStats t{};
    auto see = [](uint32_t* bits, int32_t i) {
        const uint32_t bit = 1u << (i & 31);
        return (atomicOr(&bits[i >> 5], bit) & bit) != 0u;
    };
    for (int32_t j = tid; j < count; j += TREE_BLOCK)
        check_node(
            nodes, j, count, n, t,
            [&](int32_t begin, int32_t depth) {
                atomicAdd(&starts[begin], 1u);
                atomicMin(&top_depth[begin], depth);
            },
            [&](int32_t r) { return see(node_seen, r); }, [&](int32_t q) { return see(tri_seen, q); });
    __syncthreads();
    for (int32_t i = tid; i < n; i += TREE_BLOCK)
    {
        bool bad = ((tri_seen[i >> 5] >> (i & 31)) & 1u) == 0u;
        if (i < count && i > 0 && nodes[i].d.w != NODE_UNUSED)
            bad |= ((node_seen[i >> 5] >> (i & 31)) & 1u) == 0u;
        if (bad)
            atomicAdd(&missing, 1u);
    }
    // exclusive scan of starts: four a thread
    static_assert(TREE_SMALL == 4 * TREE_BLOCK, "four a thread");
    uint32_t own[4], sum = 0u;
    for (int k = 0; k < 4; k++)
    {
        own[k] = starts[4 * tid + k];
        sum += own[k];
    }
    uint32_t incl = sum;
    for (int off = 1; off < 64; off <<= 1)
    {
        const uint32_t v = __shfl_up(incl, off, 64);
        if ((tid & 63) >= off)
            incl += v;
    }
    if ((tid & 63) == 63)
        wave_total[tid / 64] = incl;
    __syncthreads();
    uint32_t at = incl - sum;
    for (int w = 0; w < tid / 64; w++)
        at += wave_total[w];
    for (int k = 0; k < 4; k++)
    {
        starts[4 * tid + k] = at;
        at += own[k];
    }
    t = block_sum<TREE_BLOCK>(t, part);
    if (tid == 0)
    {
        t.errors += missing;
        errors = t.errors;
        report->sums = t;
        report->root_area = root_box_area(nodes[0], n);
    }
    __syncthreads();
    if (errors != 0u)
        return;
    for (int32_t j = tid; j < count; j += TREE_BLOCK)
        lay_out(nodes, j, n, starts, top_depth, out);
}

} // namespace

TreeScratch tree_scratch(BuildScratch& sc, int32_t n, int32_t count)
{
    TreeScratch t{};
    const size_t N = (size_t)n, C = (size_t)count;
    if (n > TREE_SMALL)
    {
        t.o_tri = sc.add(4 * N);
        t.o_starts = sc.add(4 * N);
        t.o_before = sc.add(4 * N);
        t.o_top = sc.add(4 * N);
        t.o_node = sc.add(4 * C);
        t.o_stats = sc.add(sizeof(TreeStats) * (blocks(count, CHECK_BLOCK) + 1));
        HIP_CHECK(rocprim::exclusive_scan(nullptr, t.scan_bytes, (const uint32_t*)nullptr, (uint32_t*)nullptr, 0u, N,
                                          rocprim::plus<uint32_t>(), (hipStream_t) nullptr));
        t.o_scan = sc.add(t.scan_bytes > 0 ? t.scan_bytes : 1);
    }
    t.o_item_ref = sc.add(sizeof(int32_t) * C);
    t.o_item_stack = sc.add(sizeof(uint32_t) * C);
    t.o_tri_src = sc.add(sizeof(uint32_t) * N);
    t.o_report = sc.add(sizeof(TreeReport));
    return t;
}

void set_statistics(Ctx& ctx, const TreeStats& t, double root_area)
{
    Bvh& bvh = ctx.bvh;
    if (t.errors != 0u)
        fail(MIPT_ERR_HIP, "BVH validation failed: " + std::to_string(t.errors) +
                               " nodes or triangles missing, out of range or in two places");
    bvh.node_count = (int32_t)t.inner;
    bvh.leaf_count = (int32_t)t.leaves;
    bvh.max_depth = (int32_t)t.max_depth;
    bvh.max_leaf_size = (int32_t)t.max_leaf;
    bvh.sah_cost = root_area > 0 ? (t.sah + SAH_C_NODE * root_area) / root_area : 0.0;
}

void finalize_bvh(Ctx& ctx, const BuildScratch& sc, TreeScratch& t, const BvhNode* d_nodes, int32_t count)
{
    Bvh& bvh = ctx.bvh;
    const int32_t n = bvh.triangle_count;
    const hipStream_t s = nullptr;
    t.item_ref = sc.get<int32_t>(t.o_item_ref);
    t.item_stack = sc.get<uint32_t>(t.o_item_stack);
    t.tri_src = sc.get<uint32_t>(t.o_tri_src);
    t.report = sc.get<TreeReport>(t.o_report);
    if (n <= TREE_SMALL)
    {
        bvh.nodes.reserve(sizeof(BvhNode) * (size_t)count);
        hipLaunchKernelGGL(k_tree_small, dim3(1), dim3(TREE_BLOCK), 0, s, d_nodes, count, n, bvh.nodes.as<BvhNode>(),
                           t.report);
        build_wide(ctx, count, false, t);
        bvh.valid = true;
        return;
    }
    const unsigned check_blocks = blocks(count, CHECK_BLOCK);
    uint32_t *tri_seen = sc.get<uint32_t>(t.o_tri), *starts = sc.get<uint32_t>(t.o_starts),
             *before = sc.get<uint32_t>(t.o_before), *node_seen = sc.get<uint32_t>(t.o_node);
    int32_t* top_depth = sc.get<int32_t>(t.o_top);
    TreeStats* stats = sc.get<TreeStats>(t.o_stats);
    const unsigned wide_grid = blocks(std::max(n, count), 256);
    hipLaunchKernelGGL(k_check_init, dim3(wide_grid), dim3(256), 0, s, tri_seen, starts, top_depth, n, node_seen, count);
    hipLaunchKernelGGL(k_tree_check, dim3(check_blocks), dim3(CHECK_BLOCK), 0, s, d_nodes, count, n, tri_seen,
                       node_seen, starts, top_depth, stats);
    hipLaunchKernelGGL(k_tree_complete, dim3(wide_grid), dim3(256), 0, s, d_nodes, count, n, tri_seen, node_seen,
                       stats);
    size_t scan_bytes = t.scan_bytes;
    HIP_CHECK(rocprim::exclusive_scan(sc.get<void>(t.o_scan), scan_bytes, (const uint32_t*)starts, before, 0u,
                                      (size_t)n, rocprim::plus<uint32_t>(), s));
    HIP_CHECK(hipGetLastError());
    std::vector<TreeStats> hs(check_blocks + 1);
    HIP_CHECK(hipMemcpy(hs.data(), stats, sizeof(TreeStats) * hs.size(), hipMemcpyDeviceToHost));
    const double root_area = hs.back().sah;
    hs.pop_back();
    TreeStats sum{};
    for (const TreeStats& b : hs)
    {
        sum.sah += b.sah;
        sum.inner += b.inner;
        sum.leaves += b.leaves;
        sum.errors += b.errors;
        sum.max_depth = std::max(sum.max_depth, b.max_depth);
        sum.max_leaf = std::max(sum.max_leaf, b.max_leaf);
    }
    set_statistics(ctx, sum, root_area);
    bvh.nodes.reserve(sizeof(BvhNode) * (size_t)bvh.node_count);
    hipLaunchKernelGGL(k_tree_layout, dim3(blocks(count, 256)), dim3(256), 0, s, d_nodes, count, n, before, top_depth,
                       bvh.nodes.as<BvhNode>());
    HIP_CHECK(hipGetLastError());
    build_wide(ctx, bvh.node_count, true, t);
    bvh.valid = true;
}

void build_lbvh(Ctx& ctx)
{
    const int32_t n = ctx.triangle_count;
    Bvh& bvh = ctx.bvh;
    bvh.valid = false;
    bvh.builder = MIPT_BVH_LBVH;
    bvh.triangle_count = n;
    if (n <= 0)
    {
        bvh.node_count = bvh.leaf_count = bvh.max_depth = bvh.max_leaf_size = bvh.wide_stack = 0;
        bvh.valid = true;
        return;
    }
    const float* verts = ctx.vertices.as<float>();
    const int32_t* idx = ctx.indices.as<int32_t>();

    hipEvent_t ev0, ev1;
    HIP_CHECK(hipEventCreate(&ev0));
    HIP_CHECK(hipEventCreate(&ev1));

    const unsigned bgrid = bvhc::bounds_grid(n);
    const int32_t ninner = n > 1 ? n - 1 : 1;
    const hipStream_t s = nullptr;
    size_t tmp_bytes = 0;
    HIP_CHECK(rocprim::radix_sort_pairs(nullptr, tmp_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr, (uint32_t*)nullptr,
                                        (uint32_t*)nullptr, (size_t)n, 0u, 63u, s));
    BuildScratch sc;
    const size_t N = (size_t)n, I = (size_t)ninner;
    const size_t o_plo = sc.add(sizeof(float4) * N), o_phi = sc.add(sizeof(float4) * N), o_bounds = sc.add(4 * 12),
                 o_pad = sc.add(4), o_partial = sc.add(4 * 12 * (size_t)bgrid), o_keys = sc.add(8 * N),
                 o_keys_sorted = sc.add(8 * N), o_vals = sc.add(4 * N), o_vals_sorted = sc.add(4 * N),
                 o_sort = sc.add(tmp_bytes > 0 ? tmp_bytes : 1), o_child = sc.add(8 * I), o_parent = sc.add(4 * I),
                 o_leaf_parent = sc.add(4 * N), o_range_lo = sc.add(4 * I), o_range_hi = sc.add(4 * I),
                 o_visits = sc.add(4 * I), o_nlo = sc.add(sizeof(float4) * I), o_nhi = sc.add(sizeof(float4) * I),
                 o_cost = sc.add(4 * I), o_collapse = sc.add(I), o_nodes = sc.add(sizeof(BvhNode) * I);
    TreeScratch tree = tree_scratch(sc, n, ninner);
    sc.allocate();
    float4 *plo = sc.get<float4>(o_plo), *phi = sc.get<float4>(o_phi), *nlo = sc.get<float4>(o_nlo),
           *nhi = sc.get<float4>(o_nhi);
    uint32_t *bounds = sc.get<uint32_t>(o_bounds), *vals = sc.get<uint32_t>(o_vals),
             *vals_sorted = sc.get<uint32_t>(o_vals_sorted), *visits = sc.get<uint32_t>(o_visits);
    float *pad = sc.get<float>(o_pad), *partial = sc.get<float>(o_partial), *cost = sc.get<float>(o_cost);
    uint64_t *keys = sc.get<uint64_t>(o_keys), *keys_sorted = sc.get<uint64_t>(o_keys_sorted);
    int32_t *child = sc.get<int32_t>(o_child), *node_parent = sc.get<int32_t>(o_parent),
            *leaf_parent = sc.get<int32_t>(o_leaf_parent), *range_lo = sc.get<int32_t>(o_range_lo),
            *range_hi = sc.get<int32_t>(o_range_hi);
    uint8_t* collapse = sc.get<uint8_t>(o_collapse);
    BvhNode* nodes = sc.get<BvhNode>(o_nodes);
    bvh.tris.reserve(sizeof(TriRecord) * n);

    HIP_CHECK(hipEventRecord(ev0, s));
    const int B = 256;
    hipLaunchKernelGGL(bvhc::k_tri_boxes, dim3(bgrid), dim3(bvhc::BOUNDS_BLOCK), 0, s, verts, idx, n, plo, phi,
                       partial);
    hipLaunchKernelGGL(bvhc::k_bounds_final, dim3(1), dim3(bvhc::BOUNDS_FINAL_BLOCK), 0, s, partial, (int32_t)bgrid, bounds, pad);
    hipLaunchKernelGGL(k_morton, dim3(blocks(n, B)), dim3(B), 0, s, plo, phi, n, bounds, keys, vals,
                       ninner, visits, node_parent, leaf_parent, collapse);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(rocprim::radix_sort_pairs(sc.get<void>(o_sort), tmp_bytes, keys, keys_sorted, vals, vals_sorted, (size_t)n,
                                        0u, 63u, s));

    if (n == 1)
        write_single_triangle_root(nodes, plo, phi);
    else
    {
        hipLaunchKernelGGL(k_karras, dim3(blocks(n - 1, B)), dim3(B), 0, s, keys_sorted, n, child, node_parent,
                           leaf_parent, range_lo, range_hi);
        hipLaunchKernelGGL(k_refit, dim3(blocks(n, B)), dim3(B), 0, s, n, plo, phi, vals_sorted, child, node_parent,
                           leaf_parent, range_lo, range_hi, visits, nlo, nhi, cost, collapse, pad);
        hipLaunchKernelGGL(k_emit_nodes, dim3(blocks(n - 1, B)), dim3(B), 0, s, n, plo, phi, vals_sorted, child,
                           range_lo, range_hi, nlo, nhi, collapse, pad, node_parent, nodes);
    }
    hipLaunchKernelGGL(bvhc::k_emit_tris, dim3(blocks(n, B)), dim3(B), 0, s, verts, idx, n, vals_sorted,
                       bvh.tris.as<TriRecord>());
    HIP_CHECK(hipGetLastError());
    tree.done = ev1;
    finalize_bvh(ctx, sc, tree, nodes, ninner);
    HIP_CHECK(hipEventSynchronize(ev1));
    float ms = 0.0f;
    HIP_CHECK(hipEventElapsedTime(&ms, ev0, ev1));
    bvh.build_ms = ms;
    HIP_CHECK(hipEventDestroy(ev0));
    HIP_CHECK(hipEventDestroy(ev1));
}

} // namespace mipt
