// bvh_wide.hip -- collapses the built binary tree into the 6-wide quantised
// tree the traversal walks (layout.h: WideNode). Wide trees whose child boxes are
// quantised on their node's own grid: Ylitie, Karras and Laine 2017,
// "Efficient Incoherent Ray Traversal on GPUs Through Compressed Wide BVHs"; six
// children, the 64-byte record and its references are this file's own.
//
// Eight lanes to a wide node, level by level: they open the binary node's children,
// largest box first, until six are held, write the quantised record and
// list its interior children for the next level. One block does the first levels,
// or a small tree; each larger level is a launch. The
// children of a node, and the triangles of its leaf children, are contiguous;
// the triangles are copied into the order this gives by a last kernel.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bvh_common.h"
#include "internal.h"
#include "lane_groups.h"

namespace mipt {
namespace {

constexpr int WIDE_BLOCK = 512;
constexpr int SMALL_BLOCK = 1024;
constexpr uint32_t SMALL_LEVEL = SMALL_BLOCK / 8; // what the block does at once
constexpr int LEVELS_AT_A_TIME = 4;
constexpr unsigned LEVEL_BLOCKS = 2048; // they fill the GPU; larger levels go around
constexpr uint32_t LAST_OF_LEAF = 0x80000000u; // with a triangle's place in the binary tree's order

// Exclusive prefix sum over the wave; total gets the wave's sum.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, uint32_t& total)
{
    const uint32_t lane = __lane_id();
    uint32_t incl = v;
    for (int off = 1; off < 64; off <<= 1)
    {
        const uint32_t t = __shfl_up(incl, off, 64);
        if (lane >= (uint32_t)off)
            incl += t;
    }
    total = __shfl(incl, 63, 64);
    return incl - v;
}

// A leaf child's first triangle is 4 bits from the node's first: with the
// largest leaf last, the others may hold 15 triangles at most.
__device__ __forceinline__ bool offsets_fit(int32_t sum, int32_t largest) { return sum - largest <= 15; }

// Box coordinates as finite numbers (a triangle may reach infinity or hold a
// NaN; its box then covers everything on that axis).
__device__ __forceinline__ float finite_lo(float x) { return fminf(fmaxf(x, -WIDE_MAX_COORD), WIDE_MAX_COORD); }
__device__ __forceinline__ float finite_hi(float x) { return fmaxf(fminf(x, WIDE_MAX_COORD), -WIDE_MAX_COORD); }

__device__ __forceinline__ int32_t tris_of(int32_t ref) { return ref < 0 ? leaf_count(ref) : 0; }

// The child that a lane holds.
struct Child {
    float lo[3], hi[3];
    int32_t ref;   // binary reference: node index, or leaf (< 0)
    int32_t tris;  // triangles of a leaf, 0 for an interior child
    uint32_t key;  // larger for a larger box; 0: not to be opened
};

__device__ __forceinline__ Child child_of(const BvhNode& nd, bool second)
{
    Child c;
    c.lo[0] = second ? nd.b.z : nd.a.x;
    c.lo[1] = second ? nd.b.w : nd.a.y;
    c.lo[2] = second ? nd.c.x : nd.a.z;
    c.hi[0] = second ? nd.c.y : nd.a.w;
    c.hi[1] = second ? nd.c.z : nd.b.x;
    c.hi[2] = second ? nd.c.w : nd.b.y;
    c.ref = second ? nd.d.y : nd.d.x;
    c.tris = tris_of(c.ref);
    const float dx = c.hi[0] - c.lo[0], dy = c.hi[1] - c.lo[1], dz = c.hi[2] - c.lo[2];
    const float area = dx * dy + dy * dz + dz * dx;
    // areas order as their bits, a NaN is the largest
    c.key = c.ref < 0 ? 0u : (area < 0.0f ? 1u : (__float_as_uint(area) & 0x7fffffffu) + 1u);
    return c;
}

// One axis of the children's boxes, quantised: lower and upper planes of
// children 0 to 3 a byte each, and the tail word of children 4 and 5.
struct Planes {
    uint32_t lo, hi, tail;
    float origin;
    uint32_t exponent; // biased
};

// Quantises to 8 bits of the node's extent: q * 2^e + origin, lower bounds rounded
// down and upper bounds up (in double: the differences of two floats and the
// scaling by a power of two are exact enough that no bound moves inwards).
__device__ __forceinline__ Planes quantise_axis(float lo, float hi, bool held, uint32_t c)
{
    lo = finite_lo(lo);
    hi = finite_hi(hi);
    const float mn = group_min_f(held ? lo : INFINITY), mx = group_max_f(held ? hi : -INFINITY);
    const double extent = fmax((double)mx - (double)mn, 0.0);
    // the smallest e with 255 * 2^e >= extent
    int e = -100;
    if (extent > 0.0)
        e = max(e, __builtin_amdgcn_frexp_exp(extent) - 8);
    if (ldexp(255.0, e) < extent)
        e++;
    const double inv = ldexp(1.0, -e);
    const double a = floor(((double)lo - (double)mn) * inv), b = ceil(((double)hi - (double)mn) * inv);
    // a child that is not there is empty
    const uint32_t ql = held ? (uint32_t)fmin(fmax(a, 0.0), 255.0) : 255u;
    const uint32_t qh = held ? (uint32_t)fmin(fmax(b, 0.0), 255.0) : 0u;
    Planes p;
    const uint32_t shift = 8u * (c & 3u);
    p.lo = group_or(c < 4u ? ql << shift : 0u);
    p.hi = group_or(c < 4u ? qh << shift : 0u);
    p.tail = group_or(c == 4u || c == 5u ? (ql << shift) | (qh << (shift + 16u)) : 0u);
    p.origin = mn;
    p.exponent = (uint32_t)(e + 127);
    return p;
}

// Makes wide nodes, one for each group of eight lanes, lane c holding child c
// (every lane of the wave must call it, with the group's node j). Child nodes are
// numbered from first_node + *node_count on. BLOCK: the counters are in global memory,
// where one address serves an atomic after another (751 us for 217,557 nodes with
// three for each wave, 345 us with two for each block), and every thread of the block
// must call it; 0: they are in LDS. A level of the
// tree is a chain of up to five node fetches with work between them: with a
// thread to a node that work was 4500 instructions, and a level took 8 us however
// few its nodes (20 us with the children in scratch memory and the triangles copied
// here; now 4 us). The tree of 1000 triangles takes 31 us, for 50 and 116.
template <int BLOCK>
__device__ __forceinline__ void collapse(const BvhNode* __restrict__ nodes, int32_t single, uint32_t j, bool active,
                                         int32_t* item_ref, uint32_t* item_stack, WideNode* __restrict__ out,
                                         uint32_t* __restrict__ tri_src, uint32_t first_node, uint32_t* node_count,
                                         uint32_t* tri_count, uint32_t* max_stack)
{
    const uint32_t lane = __lane_id(), c = lane & 7u, shift = lane & 56u;
    Child ch{};
    int32_t more = 0; // first triangle of a second leaf merged into this one
    uint32_t count = 0;
    if (active)
    {
        const BvhNode root = nodes[item_ref[j]];
        ch = child_of(root, c == 1u);
        count = 1u;
        if (!single)
        {
            count = 2u;
            const int32_t t0 = tris_of(root.d.x), t1 = tris_of(root.d.y);
            if (t0 > 15 && t1 > 15)
            {
                // two full leaves: one leaf of both
                const Child second = child_of(root, true);
                for (int a = 0; a < 3; a++)
                {
                    ch.lo[a] = fminf(ch.lo[a], second.lo[a]);
                    ch.hi[a] = fmaxf(ch.hi[a], second.hi[a]);
                }
                more = leaf_first(root.d.y);
                ch.tris = t0 + t1;
                count = 1u;
            }
        }
        while (count < (uint32_t)WIDE_CHILDREN)
        {
            const uint32_t key = c < count ? ch.key : 0u, best_key = group_max(key);
            if (best_key == 0u)
                break;
            const uint32_t best = (uint32_t)__ffs((int)group_ballot(key == best_key, shift)) - 1u;
            const BvhNode nd = nodes[__shfl(ch.ref, (int)(shift + best))];
            // the child to be opened has no triangles itself
            const uint32_t own = c < count ? (uint32_t)ch.tris : 0u;
            const int32_t ta = tris_of(nd.d.x), tb = tris_of(nd.d.y);
            uint32_t sum = own + group_xor<1>(own);
            sum += group_xor<2>(sum);
            sum += group_xor<7>(sum);
            const int32_t largest = max(max(ta, tb), (int32_t)group_max(own));
            if (!offsets_fit((int32_t)sum + ta + tb, largest))
            {
                if (c == best)
                    ch.key = 0u;
                continue;
            }
            if (c == best || c == count)
                ch = child_of(nd, c == count);
            count++;
        }
        // the largest leaf last: two lanes change places
        const uint32_t own = c < count ? (uint32_t)ch.tris : 0u;
        const uint32_t most = group_max(own); // by all eight lanes
        const uint32_t fullest = group_ballot(c < count && own == most, shift);
        const uint32_t big = 31u - (uint32_t)__clz((int)fullest);
        const int src = (int)(shift + (c == big ? count - 1u : (c == count - 1u ? big : c)));
        for (int a = 0; a < 3; a++)
        {
            ch.lo[a] = __shfl(ch.lo[a], src);
            ch.hi[a] = __shfl(ch.hi[a], src);
        }
        ch.ref = __shfl(ch.ref, src);
        ch.tris = __shfl(ch.tris, src);
    }
    const bool held = c < count, interior = held && ch.tris == 0;
    const uint32_t inner = group_ballot(interior, shift);
    const uint32_t rank = (uint32_t)__popc(inner & ((1u << c) - 1u));
    // contiguous blocks of child nodes and triangles: a scan over the wave's
    // children (at most 48 nodes and 1536 triangles)
    uint32_t total;
    const uint32_t before = wave_scan((interior ? 0x10000u : 0u) + (held ? (uint32_t)ch.tris : 0u), total);
    uint32_t node_base = 0, tri_base = 0;
    if (BLOCK > 0)
    {
        constexpr int WAVES = BLOCK > 0 ? BLOCK / 64 : 1;
        __shared__ uint32_t wave_nodes[WAVES], wave_tris[WAVES], base[2];
        if (lane == 0)
        {
            wave_nodes[threadIdx.x / 64u] = total >> 16;
            wave_tris[threadIdx.x / 64u] = total & 0xffffu;
        }
        __syncthreads();
        if (threadIdx.x < 2u)
        {
            uint32_t sum = 0u;
            for (int w = 0; w < WAVES; w++)
                sum += threadIdx.x == 0u ? wave_nodes[w] : wave_tris[w];
            if (sum > 0u)
                base[threadIdx.x] = atomicAdd(threadIdx.x == 0u ? node_count : tri_count, sum);
        }
        __syncthreads();
        node_base = base[0];
        tri_base = base[1];
        for (uint32_t w = 0; w < threadIdx.x / 64u; w++)
        {
            node_base += wave_nodes[w];
            tri_base += wave_tris[w];
        }
    }
    else
    {
        if (lane == 0)
        {
            node_base = atomicAdd(node_count, total >> 16);
            tri_base = atomicAdd(tri_count, total & 0xffffu);
        }
        node_base = __shfl(node_base, 0);
        tri_base = __shfl(tri_base, 0);
    }
    const uint32_t group_before = __shfl(before, (int)shift);
    node_base += first_node + (group_before >> 16);
    tri_base += group_before & 0xffffu;
    uint32_t need = 0;
    if (active)
    {
        need = item_stack[j] + count - 1u;
        const uint32_t off = (before & 0xffffu) - (group_before & 0xffffu);
        if (interior)
        {
            item_ref[node_base + rank] = ch.ref;
            item_stack[node_base + rank] = need;
        }
        else if (held)
        {
            const uint32_t first = (uint32_t)leaf_first(ch.ref), cnt = (uint32_t)leaf_count(ch.ref);
            for (uint32_t q = 0; q < (uint32_t)ch.tris; q++)
                tri_src[tri_base + off + q] = (q < cnt ? first + q : (uint32_t)more + q - cnt) |
                                              (q + 1u == (uint32_t)ch.tris ? LAST_OF_LEAF : 0u);
        }
        const uint32_t meta = group_or(held ? (interior ? 16u + rank : off) << (5u * c + 1u) : 0u);
        const Planes x = quantise_axis(ch.lo[0], ch.hi[0], held, c), y = quantise_axis(ch.lo[1], ch.hi[1], held, c),
                     z = quantise_axis(ch.lo[2], ch.hi[2], held, c);
        const uint32_t exps = (count << 17) | x.exponent | (y.exponent << 9) | (z.exponent << 23);
        if (c == 0u)
        {
            WideNode w;
            w.origin = make_float4(x.origin, y.origin, z.origin, __int_as_float((int32_t)exps));
            w.refs = make_uint4(node_base - 16u, tri_base | WIDE_LEAF, meta, x.tail);
            w.qxy = make_uint4(x.lo, x.hi, y.lo, y.hi);
            w.qz = make_uint4(z.lo, z.hi, y.tail, z.tail);
            out[j] = w;
        }
    }
    for (int o = 32; o > 0; o >>= 1)
        need = max(need, (uint32_t)__shfl_xor(need, o));
    // the bound is read first: most waves are below it
    if (lane == 0 && need > *(volatile uint32_t*)max_stack)
        atomicMax(max_stack, need);
    if (BLOCK > 0)
        __syncthreads(); // before the next round writes the sums
}

// The root and the levels after it, up to one of more than `small_level` nodes
// (none: level[0] is then empty). Nothing is done where `errors` (null:
// none) says that the binary tree is not valid.
__global__ __launch_bounds__(SMALL_BLOCK) void k_wide_small(const BvhNode* __restrict__ nodes, int32_t single,
                                                            uint32_t small_level, const uint32_t* errors,
                                                            int32_t* item_ref, uint32_t* item_stack,
                                                            WideNode* __restrict__ out,
                                                            uint32_t* __restrict__ tri_src, WideCounters* counters)
{
    __shared__ uint32_t node_count, tri_count, max_stack;
    if (threadIdx.x == 0)
    {
        item_ref[0] = 0;
        item_stack[0] = 0u;
        node_count = errors && *errors != 0u ? 0u : 1u;
        tri_count = max_stack = 0u;
    }
    __syncthreads();
    uint32_t begin = 0;
    for (;;)
    {
        const uint32_t end = node_count;
        if (begin == end || end - begin > small_level)
            break;
        __syncthreads();
        for (uint32_t base = begin; base < end; base += SMALL_BLOCK / GROUP)
        {
            const uint32_t j = base + threadIdx.x / GROUP;
            collapse<0>(nodes, single, j, j < end, item_ref, item_stack, out, tri_src, 0u, &node_count, &tri_count,
                     &max_stack);
        }
        __syncthreads();
        begin = end;
    }
    for (uint32_t k = threadIdx.x; k < (uint32_t)WIDE_LEVELS + 1u; k += SMALL_BLOCK)
    {
        counters->level[k].begin = k == 0u ? begin : 0u;
        counters->level[k].count = k == 0u ? node_count - begin : 0u;
    }
    if (threadIdx.x == 0)
    {
        counters->tris = tri_count;
        counters->max_stack = max_stack;
    }
}

// Level k of those left. The host knows a bound of its size alone.
__global__ __launch_bounds__(WIDE_BLOCK) void k_wide_level(const BvhNode* __restrict__ nodes, int32_t single, int k,
                                                           int32_t* item_ref, uint32_t* item_stack,
                                                           WideNode* __restrict__ out,
                                                           uint32_t* __restrict__ tri_src, WideCounters* counters)
{
    const uint32_t begin = counters->level[k].begin, end = begin + counters->level[k].count;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        counters->level[k + 1].begin = end;
    for (uint32_t base = begin + blockIdx.x * (WIDE_BLOCK / GROUP); base < end; base += gridDim.x * (WIDE_BLOCK / GROUP))
    {
        const uint32_t j = base + threadIdx.x / GROUP;
        collapse<WIDE_BLOCK>(nodes, single, j, j < end, item_ref, item_stack, out, tri_src, end,
                             &counters->level[k + 1].count, &counters->tris, &counters->max_stack);
    }
}

// The triangle records in the wide leaves' order, 16 bytes a thread.
__global__ __launch_bounds__(256) void k_wide_tris(const float4* __restrict__ tris, const uint32_t* __restrict__ tri_src,
                                                   uint32_t n, float4* __restrict__ out)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const uint32_t rec = i / 3u, part = i - 3u * rec;
    if (rec >= n)
        return;
    const uint32_t src = tri_src[rec];
    if ((src & ~LAST_OF_LEAF) >= n)
        return; // not listed: the counts are checked on the host
    float4 v = tris[3u * (size_t)(src & ~LAST_OF_LEAF) + part];
    if (part == 1u)
        v.w = __int_as_float((src & LAST_OF_LEAF) ? 1 : 0);
    out[i] = v;
}

} // namespace

void build_wide(Ctx& ctx, int32_t capacity, bool checked, const TreeScratch& t)
{
    Bvh& bvh = ctx.bvh;
    const int32_t n = bvh.triangle_count;
    const hipStream_t s = nullptr;
    // a wide node is rooted at a binary node of its own
    bvh.wide.reserve(sizeof(WideNode) * (size_t)capacity);
    bvh.wide_tris.reserve(sizeof(TriRecord) * (size_t)n);
    const BvhNode* nodes = bvh.nodes.as<BvhNode>();
    WideNode* out = bvh.wide.as<WideNode>();
    WideCounters* counters = &t.report->wide;
    const int32_t single = n == 1;
    // A tree that is not checked yet is a small one: one block makes all its
    // levels (4000 triangles: 69 us; the host then waits once for everything).
    const uint32_t small_level = checked ? SMALL_LEVEL : ~0u;
    hipLaunchKernelGGL(k_wide_small, dim3(1), dim3(SMALL_BLOCK), 0, s, nodes, single, small_level,
                       checked ? nullptr : &t.report->sums.errors, t.item_ref, t.item_stack, out, t.tri_src, counters);
    auto copy_tris = [&] {
        hipLaunchKernelGGL(k_wide_tris, dim3(bvhc::blocks(3 * (int64_t)n, 256)), dim3(256), 0, s, bvh.tris.as<float4>(),
                           t.tri_src, (uint32_t)n, bvh.wide_tris.as<float4>());
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipEventRecord(t.done, s));
    };
    // Levels are launched LEVELS_AT_A_TIME without asking how large they are; a
    // level has at most six times the nodes of the one before. (5000 triangles: 15 us
    // for the first levels and 28 for four launches, where one block took 87.)
    TreeReport r{};
    uint64_t bound = (uint64_t)WIDE_CHILDREN * small_level;
    for (int k = 0;;)
    {
        for (int i = 0; checked && i < LEVELS_AT_A_TIME; i++, k++)
        {
            if (k >= WIDE_LEVELS)
                fail(MIPT_ERR_HIP, "wide BVH: too many levels");
            bound = std::min<uint64_t>(bound, (uint64_t)capacity);
            const unsigned blocks = std::min(bvhc::blocks(GROUP * (int64_t)bound, WIDE_BLOCK), LEVEL_BLOCKS);
            hipLaunchKernelGGL(k_wide_level, dim3(blocks), dim3(WIDE_BLOCK), 0, s, nodes, single, k, t.item_ref,
                               t.item_stack, out, t.tri_src, counters);
            bound *= WIDE_CHILDREN;
        }
        if (!checked)
            copy_tris();
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipMemcpy(&r, t.report, sizeof(r), hipMemcpyDeviceToHost));
        if (!checked)
            set_statistics(ctx, r.sums, r.root_area);
        const uint64_t made = (uint64_t)r.wide.level[k].begin + r.wide.level[k].count;
        if (made > (uint64_t)capacity || r.wide.tris > (uint32_t)n)
            fail(MIPT_ERR_HIP, "wide BVH: more nodes or triangles than the binary tree holds");
        if (r.wide.level[k].count == 0u || !checked)
            break;
        bound = r.wide.level[k].count;
    }
    if (r.wide.tris != (uint32_t)n)
        fail(MIPT_ERR_HIP, "wide BVH: triangles lost in the collapse");
    if (checked)
        copy_tris();
    bvh.wide_stack = (int32_t)r.wide.max_stack + 1; // a node pushes every child it enters, then takes one
}

} // namespace mipt
