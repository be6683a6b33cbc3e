// bvh_wide.hip -- collapses the built binary tree into the 6-wide quantised
// tree the traversal walks (layout.h: WideNode).
//
// A thread per wide node, level by level: it opens the binary node's children,
// largest box first, until six are held, writes the quantised record and
// lists its interior children for the next level. One block does the levels
// of up to SMALL_LEVEL nodes without the host; each larger level is a launch. The
// children of a node, and the triangles of its leaf children, are contiguous;
// the triangles are copied into the order this gives.
#include <hip/hip_runtime.h>

#include "bvh_common.h"
#include "internal.h"

namespace mipt {
namespace {

constexpr int WIDE_BLOCK = 64;
constexpr int SMALL_BLOCK = 256;
constexpr uint32_t SMALL_LEVEL = 1024;

struct Counters {
    uint32_t nodes;
    uint32_t tris;
    uint32_t max_stack;
    uint32_t begin; // first node of the level that k_wide_small left to do
};

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

struct Child {
    float4 lo, hi;
    int32_t ref;       // binary reference: node index, or leaf (< 0)
    int32_t extra_ref; // a second leaf merged into this one, or 0
    int32_t tris;      // triangles of a leaf, 0 for an interior child
    bool closed;       // opening it would break the offset limit
};

__device__ __forceinline__ Child make_child(float4 lo, float4 hi, int32_t ref)
{
    return Child{lo, hi, ref, 0, ref < 0 ? leaf_count(ref) : 0, ref < 0};
}

__device__ __forceinline__ Child child0(const BvhNode& nd)
{
    return make_child(make_float4(nd.a.x, nd.a.y, nd.a.z, 0.0f), make_float4(nd.a.w, nd.b.x, nd.b.y, 0.0f), nd.d.x);
}

__device__ __forceinline__ Child child1(const BvhNode& nd)
{
    return make_child(make_float4(nd.b.z, nd.b.w, nd.c.x, 0.0f), make_float4(nd.c.y, nd.c.z, nd.c.w, 0.0f), nd.d.y);
}

// A leaf child's first triangle is 4 bits from the node's first: with the
// largest leaf last, the others may hold 15 triangles at most.
__device__ __forceinline__ bool offsets_fit(int32_t sum, int32_t largest) { return sum - largest <= 15; }

// Box coordinates as finite numbers (a triangle may reach infinity or hold a
// NaN; its box then covers everything on that axis).
__device__ __forceinline__ float finite_lo(float x) { return fminf(fmaxf(x, -WIDE_MAX_COORD), WIDE_MAX_COORD); }
__device__ __forceinline__ float finite_hi(float x) { return fmaxf(fminf(x, WIDE_MAX_COORD), -WIDE_MAX_COORD); }

// Quantises one axis of the children's boxes to 8 bits of the node's extent:
// q * 2^e + origin, lower bounds rounded down and upper bounds up (in double:
// the differences of two floats and the scaling by a power of two are exact
// enough that no bound moves inwards). Returns the biased exponent.
__device__ uint32_t quantise_axis(const float* lo, const float* hi, int count, float& origin, uint8_t* qlo,
                                  uint8_t* qhi)
{
    float mn = finite_lo(lo[0]), mx = finite_hi(hi[0]);
    for (int k = 1; k < count; k++)
    {
        mn = fminf(mn, finite_lo(lo[k]));
        mx = fmaxf(mx, finite_hi(hi[k]));
    }
    origin = mn;
    const double extent = fmax((double)mx - (double)mn, 0.0);
    int e = -100;
    if (extent > 0.0)
        e = max(e, (int)ceil(log2(extent / 255.0)));
    while (e < 120 && ldexp(255.0, e) < extent)
        e++;
    const double inv = ldexp(1.0, -e);
    for (int k = 0; k < WIDE_CHILDREN; k++)
    {
        if (k >= count)
        {
            qlo[k] = 255;
            qhi[k] = 0;
            continue;
        }
        const double a = floor(((double)finite_lo(lo[k]) - (double)mn) * inv);
        const double b = ceil(((double)finite_hi(hi[k]) - (double)mn) * inv);
        qlo[k] = (uint8_t)fmin(fmax(a, 0.0), 255.0);
        qhi[k] = (uint8_t)fmin(fmax(b, 0.0), 255.0);
    }
    return (uint32_t)(e + 127);
}

__device__ __forceinline__ uint32_t pack4(const uint8_t* q)
{
    return (uint32_t)q[0] | ((uint32_t)q[1] << 8) | ((uint32_t)q[2] << 16) | ((uint32_t)q[3] << 24);
}

__device__ __forceinline__ uint32_t pack_tail(const uint8_t* qlo, const uint8_t* qhi)
{
    return (uint32_t)qlo[4] | ((uint32_t)qlo[5] << 8) | ((uint32_t)qhi[4] << 16) | ((uint32_t)qhi[5] << 24);
}

// Makes wide node j (every lane of the wave must call it).
__device__ __forceinline__ void collapse(const BvhNode* __restrict__ nodes, const TriRecord* __restrict__ tris,
                                         int32_t single, uint32_t j, bool active, int32_t* item_ref,
                                         uint32_t* item_stack, WideNode* __restrict__ out,
                                         TriRecord* __restrict__ tri_out, Counters* counters)
{
    Child c[WIDE_CHILDREN];
    int count = 0;
    if (active)
    {
        const BvhNode root = nodes[item_ref[j]];
        c[0] = child0(root);
        count = 1;
        if (!single)
        {
            c[1] = child1(root);
            count = 2;
            // two full leaves: one leaf of both
            if (c[0].tris > 15 && c[1].tris > 15)
            {
                c[0].lo = bvhc::f4min(c[0].lo, c[1].lo);
                c[0].hi = bvhc::f4max(c[0].hi, c[1].hi);
                c[0].extra_ref = c[1].ref;
                c[0].tris += c[1].tris;
                count = 1;
            }
        }
        while (count < WIDE_CHILDREN)
        {
            int best = -1;
            float best_area = -1.0f;
            for (int k = 0; k < count; k++)
            {
                const float area = bvhc::half_area(c[k].lo, c[k].hi);
                if (!c[k].closed && !(area <= best_area))
                {
                    best = k;
                    best_area = area;
                }
            }
            if (best < 0)
                break;
            const BvhNode nd = nodes[c[best].ref];
            const Child a = child0(nd), b = child1(nd);
            int32_t sum = a.tris + b.tris, largest = max(a.tris, b.tris);
            for (int k = 0; k < count; k++)
                if (k != best)
                {
                    sum += c[k].tris;
                    largest = max(largest, c[k].tris);
                }
            if (!offsets_fit(sum, largest))
            {
                c[best].closed = true;
                continue;
            }
            c[best] = a;
            c[count++] = b;
        }
        // the largest leaf last
        int big = 0;
        for (int k = 1; k < count; k++)
            if (c[k].tris >= c[big].tris)
                big = k;
        const Child last = c[big];
        c[big] = c[count - 1];
        c[count - 1] = last;
    }
    uint32_t inner = 0, ntri = 0;
    for (int k = 0; k < count; k++)
    {
        inner += c[k].tris == 0;
        ntri += (uint32_t)c[k].tris;
    }
    // contiguous blocks of child nodes and triangles: one atomic per wave
    uint32_t wave_inner, wave_tris;
    const uint32_t inner_off = wave_scan(inner, wave_inner), tri_off = wave_scan(ntri, wave_tris);
    uint32_t node_base = 0, tri_base = 0;
    if (__lane_id() == 0)
    {
        node_base = atomicAdd(&counters->nodes, wave_inner);
        tri_base = atomicAdd(&counters->tris, wave_tris);
    }
    node_base = __shfl(node_base, 0, 64) + inner_off;
    tri_base = __shfl(tri_base, 0, 64) + tri_off;
    uint32_t need = 0;
    if (active)
    {
        need = item_stack[j] + (uint32_t)(count - 1);
        WideNode w;
        uint32_t meta = 0, rank = 0, off = 0;
        for (int k = 0; k < count; k++)
        {
            if (c[k].tris == 0)
            {
                meta |= (16u + rank) << (5 * k + 1);
                item_ref[node_base + rank] = c[k].ref;
                item_stack[node_base + rank] = need;
                rank++;
                continue;
            }
            meta |= off << (5 * k + 1);
            const int32_t refs[2] = {c[k].ref, c[k].extra_ref};
            uint32_t t = off;
            for (int h = 0; h < 2 && refs[h] < 0; h++)
            {
                const int32_t first = leaf_first(refs[h]), cnt = leaf_count(refs[h]);
                for (int32_t q = 0; q < cnt; q++)
                {
                    TriRecord r = tris[first + q];
                    t++;
                    r.e1.w = __int_as_float(t == off + (uint32_t)c[k].tris ? 1 : 0);
                    tri_out[tri_base + t - 1] = r;
                }
            }
            off += (uint32_t)c[k].tris;
        }
        uint8_t qlo[3][WIDE_CHILDREN], qhi[3][WIDE_CHILDREN];
        float origin[3], lo[WIDE_CHILDREN], hi[WIDE_CHILDREN];
        uint32_t exps = (uint32_t)count << 17;
        for (int a = 0; a < 3; a++)
        {
            for (int k = 0; k < count; k++)
            {
                lo[k] = a == 0 ? c[k].lo.x : (a == 1 ? c[k].lo.y : c[k].lo.z);
                hi[k] = a == 0 ? c[k].hi.x : (a == 1 ? c[k].hi.y : c[k].hi.z);
            }
            const int at[3] = {0, 9, 23};
            exps |= quantise_axis(lo, hi, count, origin[a], qlo[a], qhi[a]) << at[a];
        }
        w.origin = make_float4(origin[0], origin[1], origin[2], __int_as_float((int32_t)exps));
        w.refs = make_uint4(node_base - 16u, tri_base | WIDE_LEAF, meta, pack_tail(qlo[0], qhi[0]));
        w.qxy = make_uint4(pack4(qlo[0]), pack4(qhi[0]), pack4(qlo[1]), pack4(qhi[1]));
        w.qz = make_uint4(pack4(qlo[2]), pack4(qhi[2]), pack_tail(qlo[1], qhi[1]), pack_tail(qlo[2], qhi[2]));
        out[j] = w;
    }
    for (int off = 32; off > 0; off >>= 1)
        need = max(need, (uint32_t)__shfl_xor(need, off, 64));
    if (__lane_id() == 0 && need > 0)
        atomicMax(&counters->max_stack, need);
}

// The root and the levels after it, up to one of more than SMALL_LEVEL nodes;
// counters->begin is then that level's first node (all nodes: the tree is done).
__global__ __launch_bounds__(SMALL_BLOCK) void k_wide_small(const BvhNode* __restrict__ nodes,
                                                            const TriRecord* __restrict__ tris, int32_t single,
                                                            int32_t* item_ref, uint32_t* item_stack,
                                                            WideNode* __restrict__ out, TriRecord* __restrict__ tri_out,
                                                            Counters* counters)
{
    __shared__ uint32_t level_end;
    if (threadIdx.x == 0)
    {
        item_ref[0] = 0;
        item_stack[0] = 0u;
        *counters = Counters{1u, 0u, 0u, 0u};
        level_end = 1u;
    }
    __threadfence_block();
    __syncthreads();
    uint32_t begin = 0;
    for (;;)
    {
        const uint32_t end = level_end;
        if (begin == end || end - begin > SMALL_LEVEL)
            break;
        for (uint32_t base = begin; base < end; base += SMALL_BLOCK)
        {
            const uint32_t j = base + threadIdx.x;
            collapse(nodes, tris, single, j, j < end, item_ref, item_stack, out, tri_out, counters);
        }
        __threadfence();
        __syncthreads();
        if (threadIdx.x == 0)
            level_end = atomicAdd(&counters->nodes, 0u);
        __syncthreads();
        begin = end;
    }
    if (threadIdx.x == 0)
        counters->begin = begin;
}

__global__ __launch_bounds__(WIDE_BLOCK) void k_wide_level(const BvhNode* __restrict__ nodes,
                                                           const TriRecord* __restrict__ tris, int32_t single,
                                                           uint32_t begin, uint32_t end, int32_t* item_ref,
                                                           uint32_t* item_stack, WideNode* __restrict__ out,
                                                           TriRecord* __restrict__ tri_out, Counters* counters)
{
    const uint32_t j = begin + blockIdx.x * WIDE_BLOCK + threadIdx.x;
    collapse(nodes, tris, single, j, j < end, item_ref, item_stack, out, tri_out, counters);
}

} // namespace

void build_wide(Ctx& ctx)
{
    Bvh& bvh = ctx.bvh;
    const int32_t n = bvh.triangle_count;
    const hipStream_t s = nullptr;
    // a wide node is rooted at a binary node of its own
    const size_t capacity = (size_t)bvh.node_count;
    bvh.wide.reserve(sizeof(WideNode) * capacity);
    bvh.wide_tris.reserve(sizeof(TriRecord) * (size_t)n);
    BuildScratch sc;
    const size_t o_ref = sc.add(sizeof(int32_t) * capacity), o_stack = sc.add(sizeof(uint32_t) * capacity),
                 o_counters = sc.add(sizeof(Counters));
    sc.allocate();
    int32_t* item_ref = sc.get<int32_t>(o_ref);
    uint32_t* item_stack = sc.get<uint32_t>(o_stack);
    Counters* counters = sc.get<Counters>(o_counters);
    const BvhNode* nodes = bvh.nodes.as<BvhNode>();
    const TriRecord* tris = bvh.tris.as<TriRecord>();
    WideNode* out = bvh.wide.as<WideNode>();
    TriRecord* tri_out = bvh.wide_tris.as<TriRecord>();
    Counters h{};
    auto read_counters = [&] {
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipMemcpy(&h, counters, sizeof(h), hipMemcpyDeviceToHost));
        if (h.nodes > capacity || h.tris > (uint32_t)n)
            fail(MIPT_ERR_HIP, "wide BVH: more nodes or triangles than the binary tree holds");
    };
    hipLaunchKernelGGL(k_wide_small, dim3(1), dim3(SMALL_BLOCK), 0, s, nodes, tris, (int32_t)(n == 1), item_ref,
                       item_stack, out, tri_out, counters);
    read_counters();
    for (uint32_t begin = h.begin; begin < h.nodes;)
    {
        const uint32_t end = h.nodes;
        hipLaunchKernelGGL(k_wide_level, dim3(bvhc::blocks(end - begin, WIDE_BLOCK)), dim3(WIDE_BLOCK), 0, s, nodes,
                           tris, (int32_t)(n == 1), begin, end, item_ref, item_stack, out, tri_out, counters);
        read_counters();
        begin = end;
    }
    if (h.tris != (uint32_t)n)
        fail(MIPT_ERR_HIP, "wide BVH: triangles lost in the collapse");
    bvh.wide_count = (int32_t)h.nodes;
    bvh.wide_stack = (int32_t)h.max_stack + 1; // a node pushes every child it enters, then takes one
}

} // namespace mipt
