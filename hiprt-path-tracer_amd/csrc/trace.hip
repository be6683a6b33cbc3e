// trace.hip -- closest-hit and any-hit BVH traversal for gfx950.
//
// Replaces hiprtGeomTraversalClosest / hiprtGeomTraversalAnyHit as used by
// trace_main_path_ray, evaluate_shadow_ray_occluded and
// evaluate_bsdf_light_sample_ray (src/Device/includes/Intersect.h:200-324,
// :544-643). CDNA4 has no ray-tracing units, so this is a plain stackful
// traversal of a 6-wide tree (layout.h: WideNode), one ray per lane:
//   * one 64-byte node fetch tests the quantised boxes of up to six children;
//     those hit are sorted by entry distance, the nearest is taken and the
//     others are pushed with their distances, so that an entry behind the
//     closest hit found since is dropped without a fetch;
//   * a leaf is a reference to its first triangle (Moller-Trumbore, exact
//     reference arithmetic), taken from the stack like a node. Lanes at leaves
//     wait until LEAF_LANES of them are there (or no lane is at a node): the
//     wave then pays for the triangle test once for many;
//   * the per-lane stack lives in LDS, laid out [depth][lane]; entries
//     deeper than the LDS stack spill to a per-thread global array, without
//     their distances: few do, and the arrays, sized for the deepest stack a
//     tree allows, are half as large (two million bounce rays: 509 us a launch,
//     511 us with the distances);
//   * a persistent grid sized from occupancy; each wave takes batches of rays
//     from a global counter and hands them to lanes whose ray is done, once
//     REFILL_LANES of them are. When none are left, its last GROUPS rays get
//     eight lanes each;
//   * optionally the rays to trace come from segmented queues of slot
//     indices (seglist.h) whose lengths are read on the device (the path
//     passes enqueue only live rays); results go to the rays' own slots.
//
// Results are exact: the box test is conservative (boxes padded at build time,
// quantised outwards, and the slab interval relatively widened by 2^-16), so
// it never rejects a node holding the closest Moller-Trumbore hit, and ties in
// t go to the smaller primitive index. Hit IDs and t are therefore
// bit-identical to a brute-force loop over all triangles with the same
// arithmetic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <utility>

#include "internal.h"
#include "lane_groups.h"
#include "pt_math.h"
#include "seglist.h"

namespace mipt {
namespace {

enum Mode { CLOSEST = 0, ANY = 1, CLOSEST_COUNTED = 2, QUEUED = 3 };

constexpr float WIDEN_LO = 1.0f - 1.52587890625e-05f; // 1 - 2^-16
constexpr float WIDEN_HI = 1.0f + 1.52587890625e-05f;

__device__ __forceinline__ float safe_inv(float d)
{
    const float tiny = 1.0e-20f;
    return 1.0f / (fabsf(d) > tiny ? d : copysignf(tiny, d));
}

__global__ void k_reset_counter(uint32_t* c) { c[0] = 0u; }

// Lanes at a leaf that make the wave test triangles, one after another while that
// many are left (1 to 24 measured within 2 % of each other, 32 lost 20 %: lanes that
// wait test no boxes; one test at a time cost the same in closest_bounce's scene,
// 1.96 ms for 1.57 with 100,000 rays among 20,000 large overlapping triangles,
// and with coincident triangles it was slower than a loop over a leaf: 300 of
// them, a million rays, 755 us for 584, now 527), and lanes without a ray that
// make it take more (8 to 24: the same).
constexpr int LEAF_LANES = 8;
constexpr int REFILL_LANES = 16;
// Fewer rays than the grid has lanes are dealt to 3 waves per SIMD, at least
// MIN_BATCH to a wave, one for each of its groups of eight lanes (120,000
// bounce rays of the 1M-triangle scene: 120 us at 2 waves, 116 us at 3, 119 to
// 126 us at 4 to 6; 1 to 8 rays a wave measure the same).
constexpr uint32_t MIN_BATCH = 8;
constexpr uint32_t FEW_WAVES_PER_CU = 12;

constexpr int MAX_LDS_STACK = 32;

constexpr int32_t IDLE = 0x7fffffff; // no node or leaf to visit (node indices stay below)

// A ray set: `rays` indexed by slot; with `occluded` it is traced any-hit
// (shadow rays: tmax is the light distance), else closest-hit into `hits`.
// Slots come from a segmented queue, or are 0 .. n-1 without one.
struct QueueJob {
    const float4* rays;
    int4* hits;
    uint8_t* occluded;
    const uint32_t* slots;
    const uint32_t* counts;
    uint32_t seg_cap;
};

struct TraceArgs {
    const WideNode* nodes;
    const TriRecord* tris;
    QueueJob job[3];
    uint2* counts;      // nodes and triangles per ray (instrumented variant)
    uint32_t n;         // rays without a queue
    uint32_t* spill;    // references of stack entries past the LDS ones, a column per thread
    uint32_t spill_stride;
    uint32_t* work_counter;
    uint32_t tile;
    uint32_t few_waves; // waves that fewer rays than the grid's lanes are dealt to
    uint32_t last_tri;  // index of the last triangle record
};

__device__ __forceinline__ uint32_t med3(uint32_t a, uint32_t b, uint32_t c) { return max(min(a, b), min(max(a, b), c)); }

// Sorts six keys: two triples by three-operand minimum, median and maximum
// (one instruction each), then a merge: 18 instructions against 24 of a
// network of two-operand comparators.
__device__ __forceinline__ void sort6(uint32_t k[6])
{
    const uint32_t a0 = min(min(k[0], k[1]), k[2]), a1 = med3(k[0], k[1], k[2]), a2 = max(max(k[0], k[1]), k[2]);
    const uint32_t b0 = min(min(k[3], k[4]), k[5]), b1 = med3(k[3], k[4], k[5]), b2 = max(max(k[3], k[4]), k[5]);
    const uint32_t x = max(a0, b0), y = min(a2, b2), p = min(a1, b1), q = max(a1, b1);
    const uint32_t m = max(x, p), n = min(q, y);
    k[0] = min(a0, b0);
    k[1] = min(x, p);
    k[2] = min(m, n);
    k[3] = max(m, n);
    k[4] = max(q, y);
    k[5] = max(a2, b2);
}

// Rays that a wave takes at a time.
__host__ __device__ __forceinline__ uint32_t wave_batch(uint32_t total, uint32_t waves, uint32_t tile, uint32_t few_waves)
{
    if (total >= waves * 64u)
        return 64u * tile;
    const uint32_t share = (total + few_waves - 1u) / few_waves;
    return share <= MIN_BATCH ? MIN_BATCH : (share < 64u ? share : 64u);
}

// The last GROUPS rays of a wave are traced by eight lanes each, lane c of a
// group taking child c of a node and triangle c of a leaf. What ends a launch is
// its longest ray: a round of one lane to a ray issues about 300 instructions
// (four cycles each) after waiting for its node, a round of eight lanes about
// 200 for a node and a leaf whose loads are under way together. 61 camera rays:
// 21.6 us with one lane to a ray, 15.3 us so; 12,513 bounce rays 59.6 us and
// 41 us, 120,000 (which end one lane to a ray until eight are left in a wave)
// 142 us and 116 us; 2,073,600 516 us and 506 us. Eight rays is what the lanes
// hold; a wave with more has enough to issue.
constexpr int GROUPS = 64 / GROUP;

template <int I> __device__ __forceinline__ float byte_of(uint32_t w) { return (float)((w >> (8 * I)) & 0xffu); }

// One ray set, or (QUEUED) the rays of up to three segmented queues: dense
// index w runs over queue 0, then 1, then 2. One launch instead of three keeps
// the grid busy when the queues are short (a launch costs about the traversal
// latency of its longest ray, whatever its length).
//
// Bound by instruction issue: the vector units are busy 85 % of the time over
// 2,073,600 incoherent rays on 1,040,384 triangles (17 nodes and 4.6 triangles
// a ray, 45 of 64 lanes at a node in a mean node step, about 210 instructions;
// the 64-byte record costs 4 loads, the L2 serves 2.4 GB). A binary tree of
// 64-byte nodes with float boxes took 43.8 nodes a ray, and the same 4
// loads for each: 910 us, now 506 us; 700,001 shadow rays 564 us, now 296 us.
// Reading the nodes by groups of four lanes through LDS (a quarter of the cache
// accesses) cost more in instructions and LDS than it saved (680 us), a second
// put-aside leaf per lane let culling lag (552 us).
template <int BLOCK, int STACK, int MODE>
__global__ __launch_bounds__(BLOCK) void k_trace(TraceArgs a)
{
    constexpr bool QUEUES = MODE == QUEUED;
    __shared__ uint2 stack[STACK * BLOCK];
    // Segment starts of the three queues (the same for every wave): read
    // from LDS by a per-lane binary search, so no registers hold them while
    // the rays are traversed.
    __shared__ uint32_t seg_start[QUEUES ? 3 : 1][SEG_COUNT];
    __shared__ uint32_t queue_end[3];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    uint32_t total = a.n, end0 = 0u, end1 = 0u;
    if (QUEUES)
    {
        if (threadIdx.x < 64u)
        {
            uint32_t sum = 0;
#pragma unroll
            for (int k = 0; k < 3; k++)
            {
                SegMap m{};
                m.excl = 0u;
                m.total = 0u;
                if (a.job[k].slots)
                    m.init(a.job[k].counts, a.job[k].seg_cap);
                seg_start[QUEUES ? k : 0][lane] = m.excl;
                sum += m.total;
                if (lane == 0)
                    queue_end[k] = sum;
            }
        }
        __syncthreads();
        end0 = __builtin_amdgcn_readfirstlane(queue_end[0]);
        end1 = __builtin_amdgcn_readfirstlane(queue_end[1]);
        total = __builtin_amdgcn_readfirstlane(queue_end[2]);
    }

    // The wave's rays: its first batch by index, later ones from the work
    // counter, past the statically assigned ones (a same-address atomic from
    // every wave costs tens of microseconds per launch). With fewer rays than
    // lanes the batches shrink, down to MIN_BATCH rays: more waves, each with
    // fewer different paths through the tree, end sooner.
    const uint32_t waves = gridDim.x * (BLOCK / 64u);
    const uint32_t batch = wave_batch(total, waves, a.tile, a.few_waves);
    uint32_t next = __builtin_amdgcn_readfirstlane(blockIdx.x * (BLOCK / 64u) + threadIdx.x / 64u) * batch;
    uint32_t batch_end = min(next + batch, total);
    bool more = next < total;

    // the lane's ray
    pt::f3 o{}, d{};
    float inv_nx = 0.0f, inv_ny = 0.0f, inv_nz = 0.0f, inv_fx = 0.0f, inv_fy = 0.0f, inv_fz = 0.0f;
    float best_t = 0.0f, best_u = 0.0f, best_v = 0.0f;
    int32_t best_prim = -1, last_prim = -1;
    uint32_t slot = 0u, job = 0u;
    uint32_t n_nodes = 0, n_tris = 0;
    bool any = MODE == ANY, has_ray = false;
    int32_t cur = IDLE;  // node or leaf to visit next
    int32_t leaf = 0;    // leaf whose triangles wait to be tested, 0 for none
    int sp = 0;

    auto write_result = [&]() {
        if (any)
        {
            uint8_t* occ = a.job[0].occluded;
            if (QUEUES)
                occ = job == 0u ? a.job[0].occluded : (job == 1u ? a.job[1].occluded : a.job[2].occluded);
            occ[slot] = best_prim >= 0 ? 1 : 0;
        }
        else
        {
            int4* hits = a.job[0].hits;
            if (QUEUES)
                hits = job == 0u ? a.job[0].hits : (job == 1u ? a.job[1].hits : a.job[2].hits);
            hits[slot] = best_prim >= 0 ? make_int4(best_prim, __float_as_int(best_t), __float_as_int(best_u),
                                                    __float_as_int(best_v))
                                        : make_int4(-1, __float_as_int(-1.0f), 0, 0);
            if (MODE == CLOSEST_COUNTED)
                a.counts[slot] = make_uint2(n_nodes, n_tris);
        }
    };

    // The instrumented variant counts a ray's visits one lane to a ray.
    constexpr int LAST_RAYS = MODE == CLOSEST_COUNTED ? 0 : GROUPS;
    for (;;)
    {
        const uint64_t idle = __ballot(cur == IDLE && leaf == 0 && sp == 0);
        const int live = 64 - __popcll(idle);
        if (more ? live <= 64 - REFILL_LANES : live <= LAST_RAYS)
        {
            const bool free = cur == IDLE && leaf == 0 && sp == 0;
            if (free && has_ray)
            {
                has_ray = false;
                write_result();
            }
            if (more && next >= batch_end)
            {
                // with every ray assigned by index there is nothing to ask for
                if (waves * batch >= total)
                    more = false;
                else
                {
                    uint32_t base = 0u;
                    if (lane == 0u)
                        base = atomicAdd(a.work_counter, batch);
                    next = __builtin_amdgcn_readfirstlane(base) + waves * batch;
                    batch_end = min(next + batch, total);
                    more = next < total;
                }
            }
            if (more)
            {
                const uint32_t left = batch_end - next;
                const uint32_t rank = (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
                if (free && rank < left)
                {
                    const uint32_t w = next + rank;
                    const float4* rays = a.job[0].rays;
                    slot = w;
                    if (QUEUES)
                    {
                        // fields picked by selects: indexing the argument
                        // struct by a run-time value would copy it to scratch
                        job = w < end0 ? 0u : (w < end1 ? 1u : 2u);
                        const uint32_t local = w - (job == 0u ? 0u : (job == 1u ? end0 : end1));
                        rays = job == 0u ? a.job[0].rays : (job == 1u ? a.job[1].rays : a.job[2].rays);
                        const uint32_t* slots =
                            job == 0u ? a.job[0].slots : (job == 1u ? a.job[1].slots : a.job[2].slots);
                        const uint32_t seg_cap =
                            job == 0u ? a.job[0].seg_cap : (job == 1u ? a.job[1].seg_cap : a.job[2].seg_cap);
                        any = job == 0u ? a.job[0].occluded != nullptr
                                        : (job == 1u ? a.job[1].occluded != nullptr : a.job[2].occluded != nullptr);
                        // last segment whose start is <= local
                        int lo = 0, hi = (int)SEG_COUNT - 1;
                        for (int step = 0; step < 6; step++)
                        {
                            const int mid = (lo + hi + 1) >> 1;
                            if (seg_start[QUEUES ? job : 0][mid] <= local)
                                lo = mid;
                            else
                                hi = mid - 1;
                        }
                        slot = slots[(size_t)lo * seg_cap + (local - seg_start[QUEUES ? job : 0][lo])];
                    }
                    const float4 ra = rays[2 * (size_t)slot], rb = rays[2 * (size_t)slot + 1];
                    o = pt::mk(ra.x, ra.y, ra.z);
                    d = pt::mk(rb.x, rb.y, rb.z);
                    last_prim = __float_as_int(ra.w);
                    best_t = rb.w;
                    best_prim = -1;
                    best_u = best_v = 0.0f;
                    const float ix = safe_inv(d.x), iy = safe_inv(d.y), iz = safe_inv(d.z);
                    inv_nx = ix * WIDEN_LO;
                    inv_ny = iy * WIDEN_LO;
                    inv_nz = iz * WIDEN_LO;
                    inv_fx = ix * WIDEN_HI;
                    inv_fy = iy * WIDEN_HI;
                    inv_fz = iz * WIDEN_HI;
                    if (MODE == CLOSEST_COUNTED)
                        n_nodes = n_tris = 0u;
                    has_ray = true;
                    sp = 0;
                    // Nothing is hit at or past tmax, nor by a ray with an
                    // infinite or NaN component (every triangle test then
                    // compares a NaN, an infinity or 0).
                    const bool finite = __builtin_isfinite(o.x) && __builtin_isfinite(o.y) && __builtin_isfinite(o.z) &&
                                        __builtin_isfinite(d.x) && __builtin_isfinite(d.y) && __builtin_isfinite(d.z);
                    cur = best_t > 0.0f && finite ? 0 : IDLE;
                }
                next += min((uint32_t)__popcll(idle), left);
            }
            else if (live <= LAST_RAYS)
                break;
        }

        const bool at_node = (uint32_t)cur < (uint32_t)IDLE;
        if (at_node)
        {
            const WideNode* np = a.nodes + cur;
            const float4 org = np->origin;
            const uint4 refs = np->refs, qxy = np->qxy, qz = np->qz;
            if (MODE == CLOSEST_COUNTED)
                n_nodes++;
            const uint32_t ex = (uint32_t)__float_as_int(org.w);
            const float sx = __uint_as_float(ex << 23), sy = __uint_as_float((ex << 14) & 0x7f800000u),
                        sz = __uint_as_float(ex & 0x7f800000u);
            const uint32_t count = (ex >> 17) & 7u;
            const float px = org.x - o.x, py = org.y - o.y, pz = org.z - o.z;
            const float nbx = px * inv_nx, nby = py * inv_ny, nbz = pz * inv_nz;
            const float fbx = px * inv_fx, fby = py * inv_fy, fbz = pz * inv_fz;
            const float nsx = sx * inv_nx, nsy = sy * inv_ny, nsz = sz * inv_nz;
            const float fsx = sx * inv_fx, fsy = sy * inv_fy, fsz = sz * inv_fz;
            // entry and exit planes by the sign of the direction
            const bool bx = inv_nx < 0.0f, by = inv_ny < 0.0f, bz = inv_nz < 0.0f;
            const uint32_t tx = bx ? __builtin_rotateright32(refs.w, 16) : refs.w;
            const uint32_t ty = by ? __builtin_rotateright32(qz.z, 16) : qz.z;
            const uint32_t tz = bz ? __builtin_rotateright32(qz.w, 16) : qz.w;
            const uint32_t nx = bx ? qxy.y : qxy.x, fx = bx ? qxy.x : qxy.y;
            const uint32_t ny = by ? qxy.w : qxy.z, fy = by ? qxy.z : qxy.w;
            const uint32_t nz = bz ? qz.y : qz.x, fz = bz ? qz.x : qz.y;
            const float far_limit = best_t * WIDEN_HI;
            uint32_t key[WIDE_CHILDREN], hits = 0u;
#define MIPT_CHILD(K, NX, FX, NY, FY, NZ, FZ)                                                                          \
    {                                                                                                                  \
        const float tn = fmaxf(fmaxf(fmaxf(__builtin_fmaf(NX, nsx, nbx), __builtin_fmaf(NY, nsy, nby)),                \
                                     __builtin_fmaf(NZ, nsz, nbz)),                                                    \
                               0.0f);                                                                                  \
        const float tf = fminf(fminf(fminf(__builtin_fmaf(FX, fsx, fbx), __builtin_fmaf(FY, fsy, fby)),                \
                                     __builtin_fmaf(FZ, fsz, fbz)),                                                    \
                               far_limit);                                                                             \
        const bool hit = tn <= tf && K < count;                                                                        \
        key[K] = hit ? ((__float_as_uint(tn) & ~31u) | (5u * K + 1u)) : ~0u;                                           \
        hits += hit ? 1u : 0u;                                                                                         \
    }
            MIPT_CHILD(0, byte_of<0>(nx), byte_of<0>(fx), byte_of<0>(ny), byte_of<0>(fy), byte_of<0>(nz), byte_of<0>(fz))
            MIPT_CHILD(1, byte_of<1>(nx), byte_of<1>(fx), byte_of<1>(ny), byte_of<1>(fy), byte_of<1>(nz), byte_of<1>(fz))
            MIPT_CHILD(2, byte_of<2>(nx), byte_of<2>(fx), byte_of<2>(ny), byte_of<2>(fy), byte_of<2>(nz), byte_of<2>(fz))
            MIPT_CHILD(3, byte_of<3>(nx), byte_of<3>(fx), byte_of<3>(ny), byte_of<3>(fy), byte_of<3>(nz), byte_of<3>(fz))
            MIPT_CHILD(4, byte_of<0>(tx), byte_of<2>(tx), byte_of<0>(ty), byte_of<2>(ty), byte_of<0>(tz), byte_of<2>(tz))
            MIPT_CHILD(5, byte_of<1>(tx), byte_of<3>(tx), byte_of<1>(ty), byte_of<3>(ty), byte_of<1>(tz), byte_of<3>(tz))
#undef MIPT_CHILD
            sort6(key); // nearest first, misses last
            auto ref_of = [&](uint32_t k) {
                const uint32_t m = __builtin_amdgcn_ubfe(refs.z, k, 5u);
                return (m < 16u ? refs.y : refs.x) + m;
            };
            // the nearest is next, the others go on the stack, farthest first:
            // the k-th nearest to entry sp + hits - 1 - k
            const int top = sp + (int)hits - 1;
            if (!__any(top > STACK))
            {
#pragma unroll
                for (int k = 1; k < WIDE_CHILDREN; k++)
                    if (key[k] != ~0u)
                        stack[(top - k) * BLOCK + threadIdx.x] = make_uint2(key[k], ref_of(key[k]));
            }
            else
            {
#pragma unroll
                for (int k = 1; k < WIDE_CHILDREN; k++)
                    if (key[k] != ~0u)
                    {
                        const uint2 e = make_uint2(key[k], ref_of(key[k]));
                        if (top - k < STACK)
                            stack[(top - k) * BLOCK + threadIdx.x] = e;
                        else
                            a.spill[(size_t)(top - k - STACK) * a.spill_stride + gtid] = e.y;
                    }
            }
            cur = IDLE;
            if (hits > 0u)
            {
                sp = top;
                cur = (int32_t)ref_of(key[0]);
            }
        }
        // A leaf is put aside and the lane goes on; with one put aside already
        // it waits for its turn. A lane without a node takes one entry: one
        // behind the closest hit costs it this round, which is cheaper than a
        // loop that runs as long as any lane drops entries.
        auto put_aside = [&]() {
            if (cur < 0 && leaf == 0)
            {
                leaf = cur;
                cur = IDLE;
            }
        };
        put_aside();
        if (cur == IDLE && sp > 0)
        {
            sp--;
            uint2 e = make_uint2(0u, 0u); // a spilled entry: distance 0, always in reach
            if (sp < STACK)
                e = stack[sp * BLOCK + threadIdx.x];
            else
                e.y = a.spill[(size_t)(sp - STACK) * a.spill_stride + gtid];
            // the entry's distance is already widened downwards
            if (__uint_as_float(e.x) <= best_t * WIDEN_HI)
                cur = (int32_t)e.y;
            put_aside();
        }

        uint64_t leaves = __ballot(leaf != 0);
        if (leaves && (!more || __popcll(leaves) >= LEAF_LANES || !__ballot((uint32_t)cur < (uint32_t)IDLE)))
        {
            do
            {
                if (leaf != 0)
                {
                    const TriRecord* tr = a.tris + ((uint32_t)leaf & ~WIDE_LEAF);
                    const float4 v0 = tr->v0, e1 = tr->e1, e2 = tr->e2;
                    const int32_t prim = __float_as_int(v0.w);
                    if (MODE == CLOSEST_COUNTED)
                        n_tris++;
                    float t, u, v;
                    leaf = __float_as_int(e1.w) != 0 ? 0 : leaf + 1;
                    if (pt::mt_intersect(pt::mk(v0.x, v0.y, v0.z), pt::mk(e1.x, e1.y, e1.z), pt::mk(e2.x, e2.y, e2.z), o, d,
                                         t, u, v) &&
                        prim != last_prim && (t < best_t || (t == best_t && prim < best_prim)))
                    {
                        best_t = t;
                        best_prim = prim;
                        best_u = u;
                        best_v = v;
                        if (any)
                        {
                            cur = IDLE;
                            leaf = 0;
                            sp = 0;
                        }
                    }
                }
                leaves = __ballot(leaf != 0);
            } while (__popcll(leaves) >= LEAF_LANES);
        }
    }

    // The wave's last rays, eight lanes to each.
    const uint64_t live_lanes = __ballot(has_ray);
    if (MODE == CLOSEST_COUNTED || live_lanes == 0ull)
        return;
    const uint32_t c = lane & 7u, group = lane >> 3, group_shift = lane & 56u;
    uint64_t mine = live_lanes;
#pragma unroll
    for (uint32_t i = 0; i + 1 < GROUPS; i++)
        mine = i < group ? mine & (mine - 1ull) : mine;
    const int owner = mine ? __ffsll((unsigned long long)mine) - 1 : (int)lane;
    auto from_owner_f = [&](float v) { return __shfl(v, owner); };
    auto from_owner_i = [&](int32_t v) { return __shfl(v, owner); };
    o = pt::mk(from_owner_f(o.x), from_owner_f(o.y), from_owner_f(o.z));
    d = pt::mk(from_owner_f(d.x), from_owner_f(d.y), from_owner_f(d.z));
    inv_nx = from_owner_f(inv_nx);
    inv_ny = from_owner_f(inv_ny);
    inv_nz = from_owner_f(inv_nz);
    inv_fx = from_owner_f(inv_fx);
    inv_fy = from_owner_f(inv_fy);
    inv_fz = from_owner_f(inv_fz);
    best_t = from_owner_f(best_t);
    best_u = from_owner_f(best_u);
    best_v = from_owner_f(best_v);
    best_prim = from_owner_i(best_prim);
    last_prim = from_owner_i(last_prim);
    slot = (uint32_t)from_owner_i((int32_t)slot);
    job = (uint32_t)from_owner_i((int32_t)job);
    any = from_owner_i(any ? 1 : 0) != 0;
    cur = mine ? from_owner_i(cur) : IDLE;
    leaf = mine ? from_owner_i(leaf) : 0;
    sp = mine ? from_owner_i(sp) : 0;
    if (!mine)
    {
        cur = IDLE;
        leaf = 0;
        sp = 0;
    }
    // the ray's stack stays in its owner's columns
    uint2* const column = stack + ((threadIdx.x & ~63u) + (uint32_t)owner);
    uint32_t* const deep = a.spill + (gtid - lane + (uint32_t)owner);
    const bool bx = inv_nx < 0.0f, by = inv_ny < 0.0f, bz = inv_nz < 0.0f;
    // children 4 and 5 have their planes in the tail words: entry planes in
    // bytes 0 and 1, exit planes in bytes 2 and 3, swapped by the direction
    const bool tail = c >= 4u;
    const uint32_t lo_shift = tail ? 8u * (c & 1u) : 8u * c, hi_shift = tail ? lo_shift + 16u : lo_shift;
    const uint32_t nx_shift = bx ? hi_shift : lo_shift, fx_shift = bx ? lo_shift : hi_shift;
    const uint32_t ny_shift = by ? hi_shift : lo_shift, fy_shift = by ? lo_shift : hi_shift;
    const uint32_t nz_shift = bz ? hi_shift : lo_shift, fz_shift = bz ? lo_shift : hi_shift;

    auto put_leaf_aside = [&]() {
        if (cur < 0 && leaf == 0)
        {
            leaf = cur;
            cur = IDLE;
        }
    };
    // Stack entries written by one lane of a group are read by the others: the
    // lanes of a wave run in step and its memory operations stay in order, so
    // only the compiler has to keep that order.
    auto stack_fence = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
    stack_fence();
    for (;;)
    {
        // The eight topmost entries at once: the first in reach of the closest
        // hit is next, those above it are dropped.
        auto pop = [&]() {
            if (cur == IDLE && sp > 0)
            {
                const int at = sp - 1 - (int)c;
                uint2 e = make_uint2(0x7f800001u, 0u); // NaN: out of reach
                if (at >= STACK)
                    e = make_uint2(0u, deep[(size_t)(at - STACK) * a.spill_stride]);
                else if (at >= 0)
                    e = column[at * BLOCK];
                const uint32_t in_reach = group_ballot(__uint_as_float(e.x) <= best_t * WIDEN_HI, group_shift);
                const int first = in_reach ? __ffs((int)in_reach) - 1 : 0;
                const int32_t ref = __shfl((int32_t)e.y, (int)group_shift + first);
                if (in_reach)
                {
                    cur = ref;
                    sp -= first + 1;
                }
                else
                    sp = max(sp - GROUP, 0);
            }
        };
        put_leaf_aside();
        pop();
        put_leaf_aside();
        if (!__any(cur != IDLE || leaf != 0 || sp > 0))
            break;
        // both loads go out together; a group without a node or leaf reads the
        // first one
        const bool at_node = (uint32_t)cur < (uint32_t)IDLE;
        const WideNode* np = a.nodes + (at_node ? cur : 0);
        const float4 org = np->origin;
        const uint4 refs = np->refs, qxy = np->qxy, qz = np->qz;
        const TriRecord* tr = a.tris + (leaf != 0 ? min(((uint32_t)leaf & ~WIDE_LEAF) + c, a.last_tri) : 0u);
        const float4 v0 = tr->v0, e1 = tr->e1, e2 = tr->e2;

        if (leaf != 0)
        {
            // lanes past the leaf's last triangle have nothing
            const uint32_t lasts = group_ballot(__float_as_int(e1.w) != 0, group_shift);
            const bool in_leaf = (((lasts ^ (lasts - 1u)) >> c) & 1u) != 0u;
            leaf = lasts ? 0 : leaf + GROUP;
            const int32_t prim = __float_as_int(v0.w);
            float t, u, v;
            const bool hit = in_leaf &&
                             pt::mt_intersect(pt::mk(v0.x, v0.y, v0.z), pt::mk(e1.x, e1.y, e1.z),
                                              pt::mk(e2.x, e2.y, e2.z), o, d, t, u, v) &&
                             prim != last_prim && (t < best_t || (t == best_t && prim < best_prim));
            // positive floats order as their bits
            const uint32_t tb = hit ? __float_as_uint(t) : ~0u;
            const uint32_t t_min = group_min(tb);
            const bool nearest = hit && tb == t_min;
            const uint32_t p_min = group_min(nearest ? (uint32_t)prim : ~0u);
            const uint32_t winner = group_ballot(nearest && (uint32_t)prim == p_min, group_shift);
            if (winner)
            {
                const int src = (int)group_shift + __ffs((int)winner) - 1;
                best_u = __shfl(u, src);
                best_v = __shfl(v, src);
                best_t = __uint_as_float(t_min);
                best_prim = (int32_t)p_min;
                if (any)
                {
                    cur = IDLE;
                    leaf = 0;
                    sp = 0;
                }
            }
        }
        if ((uint32_t)cur < (uint32_t)IDLE)
        {
            const uint32_t ex = (uint32_t)__float_as_int(org.w);
            const float sx = __uint_as_float(ex << 23), sy = __uint_as_float((ex << 14) & 0x7f800000u),
                        sz = __uint_as_float(ex & 0x7f800000u);
            const float px = org.x - o.x, py = org.y - o.y, pz = org.z - o.z;
            const uint32_t wnx = tail ? refs.w : (bx ? qxy.y : qxy.x), wfx = tail ? refs.w : (bx ? qxy.x : qxy.y);
            const uint32_t wny = tail ? qz.z : (by ? qxy.w : qxy.z), wfy = tail ? qz.z : (by ? qxy.z : qxy.w);
            const uint32_t wnz = tail ? qz.w : (bz ? qz.y : qz.x), wfz = tail ? qz.w : (bz ? qz.x : qz.y);
            auto plane = [](uint32_t w, uint32_t shift) { return (float)__builtin_amdgcn_ubfe(w, shift, 8u); };
            const float tn = fmaxf(fmaxf(fmaxf(__builtin_fmaf(plane(wnx, nx_shift), sx * inv_nx, px * inv_nx),
                                               __builtin_fmaf(plane(wny, ny_shift), sy * inv_ny, py * inv_ny)),
                                         __builtin_fmaf(plane(wnz, nz_shift), sz * inv_nz, pz * inv_nz)),
                                   0.0f);
            const float tf = fminf(fminf(fminf(__builtin_fmaf(plane(wfx, fx_shift), sx * inv_fx, px * inv_fx),
                                               __builtin_fmaf(plane(wfy, fy_shift), sy * inv_fy, py * inv_fy)),
                                         __builtin_fmaf(plane(wfz, fz_shift), sz * inv_fz, pz * inv_fz)),
                                   best_t * WIDEN_HI);
            const bool hit = tn <= tf && c < ((ex >> 17) & 7u);
            const uint32_t key = hit ? ((__float_as_uint(tn) & ~31u) | (5u * c + 1u)) : ~0u;
            // children nearer than this lane's: keys differ by their child
            uint32_t rank = 0u;
            rank += group_xor<1>(key) < key ? 1u : 0u;
            rank += group_xor<2>(key) < key ? 1u : 0u;
            rank += group_xor<3>(key) < key ? 1u : 0u;
            rank += group_xor<4>(key) < key ? 1u : 0u;
            rank += group_xor<5>(key) < key ? 1u : 0u;
            rank += group_xor<6>(key) < key ? 1u : 0u;
            rank += group_xor<7>(key) < key ? 1u : 0u;
            const uint32_t nearest = group_min(key);
            const int hits = __popc(group_ballot(hit, group_shift));
            auto ref_of = [&](uint32_t k) {
                const uint32_t m = __builtin_amdgcn_ubfe(refs.z, k, 5u);
                return (m < 16u ? refs.y : refs.x) + m;
            };
            const int top = sp + hits - 1;
            if (hit && rank > 0u)
            {
                const int at = top - (int)rank;
                const uint2 e = make_uint2(key, ref_of(key));
                if (at < STACK)
                    column[at * BLOCK] = e;
                else
                    deep[(size_t)(at - STACK) * a.spill_stride] = e.y;
            }
            stack_fence();
            cur = IDLE;
            if (hits > 0)
            {
                sp = top;
                cur = (int32_t)ref_of(nearest);
            }
        }
    }
    if (mine && c == 0u)
        write_result();
}

__global__ void k_all_miss(int4* __restrict__ hits, uint8_t* __restrict__ occluded, uint32_t n)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    if (hits)
        hits[i] = make_int4(-1, __float_as_int(-1.0f), 0, 0);
    if (occluded)
        occluded[i] = 0;
}

using TraceFn = void (*)(TraceArgs);

template <int BLOCK, int STACK>
TraceFn pick_mode(int mode)
{
    switch (mode)
    {
    case CLOSEST: return k_trace<BLOCK, STACK, CLOSEST>;
    case ANY: return k_trace<BLOCK, STACK, ANY>;
    case QUEUED: return k_trace<BLOCK, STACK, QUEUED>;
    default: return k_trace<BLOCK, STACK, CLOSEST_COUNTED>;
    }
}

template <int BLOCK>
TraceFn pick_stack(int stack, int mode)
{
    switch (stack)
    {
    case 8: return pick_mode<BLOCK, 8>(mode);
    case 16: return pick_mode<BLOCK, 16>(mode);
    case 24: return pick_mode<BLOCK, 24>(mode);
    default: return pick_mode<BLOCK, 32>(mode);
    }
}

TraceFn pick(int block, int stack, int mode)
{
    switch (block)
    {
    case 64: return pick_stack<64>(stack, mode);
    case 128: return pick_stack<128>(stack, mode);
    default: return pick_stack<256>(stack, mode);
    }
}

struct Launch {
    TraceFn fn;
    unsigned grid;
};

// Persistent grid: the blocks that fit on the device at once, at most enough
// for n rays.
unsigned persistent_grid(Ctx& ctx, const void* fn, uint32_t n)
{
    const int block = ctx.trace_cfg.block_size;
    // Blocks per CU of each kernel on each device, computed once; contexts on
    // several host threads share the table.
    static std::map<std::pair<const void*, int>, int> occupancy;
    static std::mutex occupancy_lock;
    const auto key = std::make_pair(fn, ctx.device);
    int per_cu = 0;
    {
        std::lock_guard<std::mutex> guard(occupancy_lock);
        auto it = occupancy.find(key);
        if (it != occupancy.end())
            per_cu = it->second;
    }
    if (per_cu == 0)
    {
        HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, block, 0));
        if (per_cu < 1)
            per_cu = 1;
        std::lock_guard<std::mutex> guard(occupancy_lock);
        occupancy[key] = per_cu;
    }
    const uint64_t max_grid = (uint64_t)per_cu * (uint64_t)ctx.cu_count;
    // a wave may take as few as MIN_BATCH rays
    const uint64_t need = ((uint64_t)n + (uint64_t)(MIN_BATCH * (block / 64)) - 1) / (uint64_t)(MIN_BATCH * (block / 64));
    const uint64_t g = need < max_grid ? need : max_grid;
    return (unsigned)(g ? g : 1);
}

Launch plan(Ctx& ctx, int mode, uint32_t n, int lds_stack)
{
    Launch l;
    l.fn = pick(ctx.trace_cfg.block_size, lds_stack, mode);
    l.grid = persistent_grid(ctx, reinterpret_cast<const void*>(l.fn), n);
    return l;
}

// Work counter and spill columns of a persistent grid of `threads` threads.
struct Scratch {
    uint32_t* counter;
    uint32_t* spill;
};

Scratch trace_scratch(Ctx& ctx, uint32_t threads)
{
    // The columns are sized for every thread the device can hold (32 waves
    // per CU), not for this launch's grid, so that launches of different grids
    // on one stream never reallocate the buffer under queued kernels.
    const int spill_depth = ctx.bvh.wide_stack - ctx.trace_cfg.lds_stack;
    const size_t spill_off = 256; // work counters live at the front
    const size_t columns = std::max<size_t>(threads, (size_t)ctx.cu_count * 32u * 64u);
    size_t spill_bytes = spill_off;
    if (spill_depth > 0)
        spill_bytes = spill_off + sizeof(uint32_t) * (size_t)spill_depth * columns;
    ctx.spill.reserve(spill_bytes);
    return Scratch{ctx.spill.as<uint32_t>(),
                   reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(ctx.spill.ptr) + spill_off)};
}

TraceArgs trace_args(Ctx& ctx, uint32_t threads, const Scratch& sc)
{
    TraceArgs a{};
    a.nodes = ctx.bvh.wide.as<WideNode>();
    a.tris = ctx.bvh.wide_tris.as<TriRecord>();
    a.spill = sc.spill;
    a.spill_stride = threads;
    a.work_counter = sc.counter;
    a.tile = (uint32_t)ctx.trace_cfg.queue_tile;
    a.few_waves = (uint32_t)ctx.cu_count * FEW_WAVES_PER_CU;
    a.last_tri = (uint32_t)ctx.bvh.triangle_count - 1u;
    return a;
}

// Whether a launch of n rays gives any wave more than the batch that it takes
// by its index. Without, the work counter is not read and needs no reset: its
// kernel is 4.5 us of a launch of 61 rays' 15.
bool takes_from_counter(const TraceArgs& a, unsigned grid, uint32_t n, int block)
{
    const uint32_t waves = grid * (uint32_t)(block / 64);
    return (uint64_t)waves * wave_batch(n, waves, a.tile, a.few_waves) < n;
}

bool trace_ready(Ctx& ctx)
{
    if (!ctx.bvh.valid)
        fail(MIPT_ERR_NO_BVH, "no BVH: call mipt_build_bvh first");
    return ctx.bvh.triangle_count != 0;
}

void launch(Ctx& ctx, int mode, const mipt_ray* rays, mipt_hit* hits, uint8_t* occluded, uint32_t* counts, uint32_t n,
            hipStream_t stream)
{
    if (n == 0)
        return;
    if (!trace_ready(ctx))
    {
        hipLaunchKernelGGL(k_all_miss, dim3((n + 255) / 256), dim3(256), 0, stream, reinterpret_cast<int4*>(hits),
                           occluded, n);
        HIP_CHECK(hipGetLastError());
        return;
    }
    const Launch l = plan(ctx, mode, n, ctx.trace_cfg.lds_stack);
    const int block = ctx.trace_cfg.block_size;
    const uint32_t threads = l.grid * (uint32_t)block;
    const Scratch sc = trace_scratch(ctx, threads);
    TraceArgs a = trace_args(ctx, threads, sc);
    a.job[0].rays = reinterpret_cast<const float4*>(rays);
    a.job[0].hits = reinterpret_cast<int4*>(hits);
    a.job[0].occluded = occluded;
    a.counts = reinterpret_cast<uint2*>(counts);
    a.n = n;
    if (takes_from_counter(a, l.grid, n, block))
        hipLaunchKernelGGL(k_reset_counter, dim3(1), dim3(1), 0, stream, sc.counter);
    hipLaunchKernelGGL(l.fn, dim3(l.grid), dim3(block), 0, stream, a);
    HIP_CHECK(hipGetLastError());
}

// ---- closest hit without allocation ---------------------------------
// Work counter and spill columns of mipt_trace_closest_noalloc, in a
// file-scope device array: each device holds its own copy from module load
// until the process ends. Host code reaches it only through the per-device
// address from hipGetSymbolAddress (the name itself is a host stand-in).
constexpr size_t NOALLOC_COUNTER_BYTES = 256;
static_assert(MIPT_TRACE_NOALLOC_SCRATCH_BYTES > NOALLOC_COUNTER_BYTES, "scratch too small");
static __device__ __align__(256) uint8_t scratch[MIPT_TRACE_NOALLOC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex noalloc_lock;
void* noalloc_ptr[MAX_DEVICES] = {};
hipError_t noalloc_err[MAX_DEVICES] = {};
bool noalloc_done[MAX_DEVICES] = {};

} // namespace

void noalloc_scratch_init(int device)
{
    if (device < 0 || device >= MAX_DEVICES)
        return;
    std::lock_guard<std::mutex> guard(noalloc_lock);
    if (noalloc_done[device])
        return;
    // the device is current (mipt_create set it)
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    noalloc_err[device] = e;
    noalloc_ptr[device] = e == hipSuccess ? p : nullptr;
    noalloc_done[device] = true;
}

void trace_closest_noalloc(Ctx& ctx, const mipt_ray* rays, mipt_hit* hits, uint32_t n, hipStream_t stream)
{
    if (n == 0)
        return;
    void* base = nullptr;
    {
        std::lock_guard<std::mutex> guard(noalloc_lock);
        if (ctx.device < 0 || ctx.device >= MAX_DEVICES || !noalloc_done[ctx.device])
            fail(MIPT_ERR_HIP, "mipt_trace_closest_noalloc: no scratch address for this device");
        if (noalloc_err[ctx.device] != hipSuccess)
            fail(MIPT_ERR_HIP, std::string("mipt_trace_closest_noalloc: hipGetSymbolAddress(scratch): ") +
                                   hipGetErrorString(noalloc_err[ctx.device]));
        base = noalloc_ptr[ctx.device];
    }
    if (!trace_ready(ctx))
    {
        hipLaunchKernelGGL(k_all_miss, dim3((n + 255) / 256), dim3(256), 0, stream, reinterpret_cast<int4*>(hits),
                           nullptr, n);
        HIP_CHECK(hipGetLastError());
        return;
    }
    const int block = ctx.trace_cfg.block_size;
    // Spill columns of the persistent grid: where the whole grid's columns do
    // not fit, it shrinks to the blocks whose columns do (every wave takes
    // rays from the work counter, so fewer blocks trace the same rays), or
    // more of the stack stays in LDS: of the LDS depths from the context's on,
    // the one that leaves the most blocks. 1,040,384 triangles, 2,073,600
    // bounce rays, stacks of 57 (SAH) and 59 entries: 581 and 690 us with 16 and
    // 24 LDS entries (plain call: 509 and 561), where spilled entries of 8 bytes
    // behind 8 LDS ones left 668 and 642 of 3072 blocks: 1098 and 1366 us.
    const size_t room = MIPT_TRACE_NOALLOC_SCRATCH_BYTES - NOALLOC_COUNTER_BYTES;
    Launch l{nullptr, 0u};
    for (int lds = ctx.trace_cfg.lds_stack; lds <= MAX_LDS_STACK; lds += 8)
    {
        Launch c = plan(ctx, CLOSEST, n, lds);
        const unsigned whole = c.grid;
        const size_t per_block =
            sizeof(uint32_t) * (size_t)std::max(0, ctx.bvh.wide_stack - lds) * (size_t)block;
        if (per_block > 0)
            c.grid = (unsigned)std::min<size_t>(whole, room / per_block);
        if (c.grid > l.grid)
            l = c;
        if (c.grid == whole)
            break;
    }
    if (l.grid == 0)
        fail(MIPT_ERR_INVALID_ARGUMENT,
             "mipt_trace_closest_noalloc: a BVH of " + std::to_string(ctx.bvh.wide_stack) +
                 " stack entries needs more than the " + std::to_string(MIPT_TRACE_NOALLOC_SCRATCH_BYTES) +
                 "-byte scratch for one block's spill stack");
    const unsigned grid = l.grid;
    const uint32_t threads = grid * (uint32_t)block;
    const Scratch sc{reinterpret_cast<uint32_t*>(base),
                     reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(base) + NOALLOC_COUNTER_BYTES)};
    TraceArgs a = trace_args(ctx, threads, sc);
    a.job[0].rays = reinterpret_cast<const float4*>(rays);
    a.job[0].hits = reinterpret_cast<int4*>(hits);
    a.n = n;
    if (takes_from_counter(a, grid, n, block))
        hipLaunchKernelGGL(k_reset_counter, dim3(1), dim3(1), 0, stream, sc.counter);
    hipLaunchKernelGGL(l.fn, dim3(grid), dim3(block), 0, stream, a);
    HIP_CHECK(hipGetLastError());
}

uint32_t* trace_counters(Ctx& ctx)
{
    static_assert(TRACE_COUNTERS <= 64, "they lie in front of the spill columns");
    return trace_scratch(ctx, 0u).counter;
}

// A scene without triangles has work counters too (the passes reset them).
void trace_reserve(Ctx& ctx)
{
    if (ctx.bvh.valid)
        (void)trace_scratch(ctx, 0u);
}

void autotune_trace(Ctx& ctx, const mipt_ray* rays, uint32_t n, int32_t repeats, hipStream_t stream,
                    mipt_trace_tuning* out, double* table)
{
    static const int blocks[3] = {64, 128, 256};
    static const int stacks[4] = {8, 16, 24, 32};
    static const int tiles[3] = {1, 2, 4};
    if (!trace_ready(ctx))
        fail(MIPT_ERR_INVALID_ARGUMENT, "mipt_autotune_trace: the scene has no triangles");
    const TraceConfig keep = ctx.trace_cfg;
    ctx.autotune_hits.reserve(sizeof(mipt_hit) * (size_t)n);
    mipt_hit* hits = ctx.autotune_hits.as<mipt_hit>();
    hipEvent_t e0, e1;
    HIP_CHECK(hipEventCreate(&e0));
    HIP_CHECK(hipEventCreate(&e1));
    double best = 0.0, at_default = 0.0;
    TraceConfig best_cfg = keep;
    int tried = 0;
    try
    {
        for (int bi = 0; bi < 3; bi++)
            for (int si = 0; si < 4; si++)
                for (int ti = 0; ti < 3; ti++)
                {
                    ctx.trace_cfg.block_size = blocks[bi];
                    ctx.trace_cfg.lds_stack = stacks[si];
                    ctx.trace_cfg.queue_tile = tiles[ti];
                    // one untimed launch: occupancy query, spill columns
                    launch(ctx, CLOSEST, rays, hits, nullptr, nullptr, n, stream);
                    HIP_CHECK(hipEventRecord(e0, stream));
                    for (int r = 0; r < repeats; r++)
                        launch(ctx, CLOSEST, rays, hits, nullptr, nullptr, n, stream);
                    HIP_CHECK(hipEventRecord(e1, stream));
                    HIP_CHECK(hipEventSynchronize(e1));
                    float ms = 0.0f;
                    HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
                    const double mean = (double)ms / repeats;
                    if (table)
                        table[(bi * 4 + si) * 3 + ti] = mean;
                    if (blocks[bi] == TraceConfig{}.block_size && stacks[si] == TraceConfig{}.lds_stack &&
                        tiles[ti] == TraceConfig{}.queue_tile)
                        at_default = mean;
                    if (tried == 0 || mean < best)
                    {
                        best = mean;
                        best_cfg = ctx.trace_cfg;
                    }
                    tried++;
                }
    }
    catch (...)
    {
        ctx.trace_cfg = keep;
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        throw;
    }
    HIP_CHECK(hipEventDestroy(e0));
    HIP_CHECK(hipEventDestroy(e1));
    ctx.trace_cfg = best_cfg;
    if (out)
    {
        out->block_size = best_cfg.block_size;
        out->lds_stack = best_cfg.lds_stack;
        out->queue_tile = best_cfg.queue_tile;
        out->configurations = tried;
        out->best_ms = best;
        out->default_ms = at_default;
    }
}

void trace_closest(Ctx& ctx, const mipt_ray* rays, mipt_hit* hits, uint32_t* counts, uint32_t n, hipStream_t stream)
{
    launch(ctx, counts ? CLOSEST_COUNTED : CLOSEST, rays, hits, nullptr, counts, n, stream);
}

void trace_any(Ctx& ctx, const mipt_ray* rays, uint8_t* occluded, uint32_t n, hipStream_t stream)
{
    launch(ctx, ANY, rays, nullptr, occluded, nullptr, n, stream);
}

void trace_queues(Ctx& ctx, const TraceQueue* q, int count, uint32_t* counter, hipStream_t stream)
{
    uint64_t capacity = 0;
    for (int k = 0; k < count; k++)
        capacity += q[k].capacity;
    if (capacity == 0)
        return;
    if (count > 3)
        fail(MIPT_ERR_INVALID_ARGUMENT, "trace_queues: at most 3 queues");
    if (!trace_ready(ctx))
    {
        for (int k = 0; k < count; k++)
            hipLaunchKernelGGL(k_all_miss, dim3((q[k].capacity + 255) / 256), dim3(256), 0, stream,
                               reinterpret_cast<int4*>(q[k].hits), q[k].occluded, q[k].capacity);
        HIP_CHECK(hipGetLastError());
        return;
    }
    const Launch l = plan(ctx, QUEUED, (uint32_t)std::min<uint64_t>(capacity, 0xffffffffull), ctx.trace_cfg.lds_stack);
    const int block = ctx.trace_cfg.block_size;
    const uint32_t threads = l.grid * (uint32_t)block;
    const Scratch sc = trace_scratch(ctx, threads);
    TraceArgs a = trace_args(ctx, threads, sc);
    for (int k = 0; k < count; k++)
    {
        QueueJob& j = a.job[k];
        j.rays = reinterpret_cast<const float4*>(q[k].rays);
        j.hits = reinterpret_cast<int4*>(q[k].hits);
        j.occluded = q[k].occluded;
        j.slots = q[k].queue->slots;
        j.counts = q[k].queue->counts;
        j.seg_cap = q[k].queue->seg_cap;
    }
    a.work_counter = counter;
    hipLaunchKernelGGL(l.fn, dim3(l.grid), dim3(block), 0, stream, a);
    HIP_CHECK(hipGetLastError());
}

} // namespace mipt
