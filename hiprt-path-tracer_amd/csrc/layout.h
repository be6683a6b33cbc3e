// layout.h -- HBM layout of the acceleration structure.
//
// BvhNode: one 64-byte record per interior node of a binary BVH = one cache
// line. It carries the boxes of BOTH children, so a traversal step is one
// 64-byte fetch that decides which children to visit:
//   a = (c0.lo.x, c0.lo.y, c0.lo.z, c0.hi.x)
//   b = (c0.hi.y, c0.hi.z, c1.lo.x, c1.lo.y)
//   c = (c1.lo.z, c1.hi.x, c1.hi.y, c1.hi.z)
//   d = (child0, child1, 0, 0)
// A child >= 0 is an interior node index; a child < 0 is a leaf
// ~((first << LEAF_COUNT_BITS) | (count - 1)) over TriRecords [first, first+count).
//
// TriRecord: 48 bytes per triangle in leaf order: (a, prim), (b - a, 0),
// (c - a, 0). The edges are the exact binary32 differences the reference
// computes per test (src/Renderer/Triangle.h:26-27).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mipt {

constexpr int LEAF_COUNT_BITS = 4;
constexpr int MAX_LEAF_SIZE = 1 << LEAF_COUNT_BITS; // 16

struct alignas(64) BvhNode {
    float4 a, b, c;
    int4 d;
};
static_assert(sizeof(BvhNode) == 64, "BvhNode must be one 64-byte line");

struct alignas(16) TriRecord {
    float4 v0; // w = primitive index (int bits)
    float4 e1;
    float4 e2;
};
static_assert(sizeof(TriRecord) == 48, "TriRecord must be 48 bytes");

// WideNode: one 64-byte record per node of the 6-wide tree the traversal
// walks (bvh_wide.hip), half a 128-byte L2 line. The children's boxes are 8-bit steps
// of the node's own grid, lower bounds rounded down and upper ones up:
//   plane = origin + q * 2^(e - 127)
//   origin = (x, y, z, exponents e of x, y and z at bits 0, 9 and 23 and the
//             number of children at bit 17)
//   refs   = (first child node - 16, first triangle | WIDE_LEAF, meta, x tail)
//   qxy    = (x lo 0..3, x hi 0..3, y lo 0..3, y hi 0..3), a byte per child
//   qz     = (z lo 0..3, z hi 0..3, y tail, z tail)
//   tail   = (lo 4, lo 5, hi 4, hi 5)
// meta holds 5 bits per child, child k's at bit 5k + 1: below 16 a leaf, whose triangles start that far
// from the first triangle and run to the record with e1.w != 0; 16 + k the
// node's k-th interior child. So a reference is (meta < 16 ? refs.y : refs.x) + meta, its sign
// bit telling a leaf.
constexpr int WIDE_CHILDREN = 6;
constexpr uint32_t WIDE_LEAF = 0x80000000u;
constexpr float WIDE_MAX_COORD = 1.0e30f;

struct alignas(64) WideNode {
    float4 origin;
    uint4 refs;
    uint4 qxy;
    uint4 qz;
};
static_assert(sizeof(WideNode) == 64, "WideNode must be 64 bytes");

__host__ __device__ inline int32_t make_leaf(int32_t first, int32_t count)
{
    return ~((first << LEAF_COUNT_BITS) | (count - 1));
}
__host__ __device__ inline int32_t leaf_first(int32_t child) { return (~child) >> LEAF_COUNT_BITS; }
__host__ __device__ inline int32_t leaf_count(int32_t child) { return ((~child) & (MAX_LEAF_SIZE - 1)) + 1; }

} // namespace mipt
