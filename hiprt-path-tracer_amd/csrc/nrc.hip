// nrc.hip -- learned radiance cache: a multiresolution hash-grid encoding of
// the position plus one-blob encodings of direction, normal, roughness and
// albedo (64 inputs), a 6-matrix ReLU MLP of width 64 with BF16 weights on the
// MFMA units (FP32 accumulation), a relative-L2 loss and Adam, all trained on
// the GPU from the tracer's own paths.
//
// MFMA: v_mfma_f32_16x16x32_bf16. Operand layout of lane l (0..63):
// A[m = l%16][k = 8*(l/16) + j], B[k = 8*(l/16) + j][n = l%16] for j < 8;
// D[m = 4*(l/16) + i][n = l%16] for i < 4. Inference has a wave for 64 rows, whose
// activations stay in registers (k_nrc_forward); training one for a 16-row tile,
// whose activations move between layers through a padded LDS tile
// (D layout -> row-major -> A layout).
#include <hip/hip_runtime.h>

#include <cstring>

#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "nrc.h"

namespace mipt {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4))); // in a caller's array of floats

// Rows from which the grid gradient is binned instead of added by global
// atomics: the bins' five launches cost the same with few levels as with many,
// the atomics by the level. A whole training step, atomics against bins, tables
// of 2^14 (2^19) entries a level: 16 levels 3000 rows 121 / 116 us (237 / 236),
// 4096 rows 138 / 117 (255 / 238); 7 levels 4096 rows 106 / 112 (143 / 152),
// 6000 rows 125 / 118 (163 / 154); 3 levels 6000 rows 109 / 114 (124 / 132), 8192 rows
// 123 / 117 (137 / 134); 1 level 10,000 rows 123 / 132 (126 / 141), 16,384 rows
// 132 / 125 (136 / 134). 65,536 rows of 16 levels: 1188 / 314 (1384 / 492).
constexpr uint32_t grad_bin_min_rows(uint32_t levels) { return std::max(4096u, 3072u + 12288u / levels); }
constexpr uint32_t GRAD_MAX_RANGES = 1u << (24 - 13); // per level (log2_table is at most 24)
constexpr uint32_t GRAD_BIN_ROWS = 1u << 16;          // rows binned at a time: 100 MB of updates at most
constexpr int TILE_LD = NRC_WIDTH + 8; // LDS row stride (bf16) of an activation tile

// binary32 -> bfloat16, round to nearest even (finite inputs).
__device__ __forceinline__ uint16_t to_bf16(float x)
{
    uint32_t u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float from_bf16(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

__device__ __forceinline__ v8bf load_v8(const uint16_t* p)
{
    const uint4 q = *reinterpret_cast<const uint4*>(p);
    return __builtin_bit_cast(v8bf, q);
}

__device__ __forceinline__ v4f mfma(v8bf a, v8bf b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// Encoding
// ---------------------------------------------------------------------------
__device__ __forceinline__ void oct_uv(float x, float y, float z, float& u, float& v)
{
    const float s = fabsf(x) + fabsf(y) + fabsf(z);
    float px = x / s, py = y / s;
    if (z < 0.0f)
    {
        const float ox = (1.0f - fabsf(py)) * (px >= 0.0f ? 1.0f : -1.0f);
        const float oy = (1.0f - fabsf(px)) * (py >= 0.0f ? 1.0f : -1.0f);
        px = ox;
        py = oy;
    }
    u = px * 0.5f + 0.5f;
    v = py * 0.5f + 0.5f;
}

// One-blob with NRC_BLOB bins: bin i holds max(0, 1 - |x * NRC_BLOB - (i + 0.5)|).
__device__ __forceinline__ void one_blob(float x, uint16_t* out)
{
    const float t = x * (float)NRC_BLOB;
    for (int i = 0; i < NRC_BLOB; i++)
        out[i] = to_bf16(fmaxf(0.0f, 1.0f - fabsf(t - ((float)i + 0.5f))));
}

__device__ __forceinline__ uint32_t grid_index(const NrcGridLevel& L, uint32_t x, uint32_t y, uint32_t z, uint32_t tmask)
{
    if (L.dense) // res^3 fits the table; the mask keeps any index inside it
        return (x + y * L.res + z * L.res * L.res) & tmask;
    return ((x * 1u) ^ (y * 2654435761u) ^ (z * 805459861u)) & tmask;
}

// Corner c of the cell containing the scaled position, its weight and index.
__device__ __forceinline__ void corner(const NrcGridLevel& L, const float pos[3], int c, uint32_t tmask, uint32_t& idx,
                                       float& w)
{
    uint32_t g[3];
    float wk[3];
    for (int a = 0; a < 3; a++)
    {
        const float s = pos[a] * L.scale + 0.5f;
        const float f = floorf(s);
        const float fr = s - f;
        const uint32_t gi = (uint32_t)f + (((c >> a) & 1) ? 1u : 0u);
        g[a] = gi;
        wk[a] = ((c >> a) & 1) ? fr : 1.0f - fr;
    }
    w = (wk[0] * wk[1]) * wk[2];
    idx = grid_index(L, g[0], g[1], g[2], tmask);
}

__device__ __forceinline__ void normalized_position(const NrcDev& P, const float* q, float pos[3])
{
    for (int a = 0; a < 3; a++)
        pos[a] = fminf(1.0f, fmaxf(0.0f, (q[a] - P.bmin[a]) * P.inv_extent));
}

// The inputs of a query record (16 floats: position, direction, normal,
// roughness, albedo) that are not the grid's, in pairs, and its position in the
// grid's cube.
__device__ __forceinline__ void record_inputs(const NrcDev& P, const float4* __restrict__ queries, size_t rec,
                                              uint32_t pairs[NRC_MISC / 2], float pos[3])
{
    const float4 a = queries[4 * rec], b = queries[4 * rec + 1], c = queries[4 * rec + 2], d = queries[4 * rec + 3];
    const float q[16] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w};
    normalized_position(P, q, pos);
    uint16_t m[NRC_MISC];
    float u, v;
    oct_uv(q[3], q[4], q[5], u, v);
    one_blob(u, m);
    one_blob(v, m + NRC_BLOB);
    oct_uv(q[6], q[7], q[8], u, v);
    one_blob(u, m + 2 * NRC_BLOB);
    one_blob(v, m + 3 * NRC_BLOB);
    one_blob(q[9], m + 4 * NRC_BLOB);
    m[5 * NRC_BLOB] = to_bf16(q[10]);
    m[5 * NRC_BLOB + 1] = to_bf16(q[11]);
    m[5 * NRC_BLOB + 2] = to_bf16(q[12]);
    m[5 * NRC_BLOB + 3] = to_bf16(1.0f);
    for (int k = 5 * NRC_BLOB + 4; k < NRC_MISC; k++)
        m[k] = 0;
    for (int k = 0; k < NRC_MISC / 2; k++)
        pairs[k] = (uint32_t)m[2 * k] | ((uint32_t)m[2 * k + 1] << 16);
}

// A row's inputs that are not the grid's; zeros for a row of padding.
__device__ __forceinline__ void write_inputs(const NrcDev& P, const float4* __restrict__ queries, const RowSel& sel,
                                             uint32_t row, uint32_t rows, const EncDev& E)
{
    uint4* out = reinterpret_cast<uint4*>(E.misc + (size_t)row * NRC_MISC);
    uint32_t m[NRC_MISC / 2] = {};
    if (row < rows)
    {
        float pos[3];
        record_inputs(P, queries, sel.record(row), m, pos);
        for (int i = 0; i < 3; i++)
            E.pos[(size_t)i * E.stride + row] = pos[i];
    }
    for (int k = 0; k < NRC_MISC / 8; k++)
        out[k] = make_uint4(m[4 * k], m[4 * k + 1], m[4 * k + 2], m[4 * k + 3]);
}

// Encodes the selected rows into E rows [0, rows) and zero-fills the rows up
// to the next multiple of pad (at most n rows in all), in two kernels.
//
// k_nrc_inputs reads each record once: the inputs that are not grid features,
// and the position in the grid's cube.
__global__ __launch_bounds__(256) void k_nrc_inputs(NrcDev P, const float4* __restrict__ queries, RowSel sel,
                                                    uint32_t n, uint32_t pad, EncDev E)
{
    const uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t rows = sel.rows();
    const uint32_t padded = (rows + pad - 1) / pad * pad;
    if (row >= n || row >= padded)
        return;
    write_inputs(P, queries, sel, row, rows, E);
}

// k_nrc_grid interpolates one level for one row per thread. Workgroups go to
// the 8 XCDs round-robin, so block b runs on XCD b % 8: it takes level
// b % 8 for every row first and level b % 8 + 8 after that, so that an XCD's L2
// (4 MB) holds one level's table (2 MB of FP16 pairs at 2^19 entries) and the
// position planes stream past it. The two corners along x are next to
// each other in the table when the lower one's x is even (hashed: the
// index is x XOR terms of y and z) or the level is dense and its index
// even: one 8-byte load then brings both.
//
// Bound by the gathers (a lane's 4 or 8 bytes are a cache access of their own).
// Reading the 64-byte records on every XCD and writing 4 bytes of each
// 128-byte input row from each of them cost more than the gathers:
// 1,000,003 rows x 16 levels took 800 us that way.
constexpr uint32_t NRC_XCDS = 8;

// A row's two features of level l at its normalised position.
__device__ __forceinline__ uint32_t grid_features(const NrcDev& P, int l, const float pos[3])
{
    const uint32_t tmask = (1u << P.log2_table) - 1u;
    const NrcGridLevel& L = P.level[l];
    const uint32_t* table = reinterpret_cast<const uint32_t*>(P.grid_f16) + ((size_t)l << P.log2_table);
    uint32_t pair[8];
    float w[8];
    for (int cc = 0; cc < 8; cc += 2)
    {
        uint32_t i0, i1;
        corner(L, pos, cc, tmask, i0, w[cc]);
        corner(L, pos, cc + 1, tmask, i1, w[cc + 1]);
        const uint2 both = *reinterpret_cast<const uint2*>(table + (i0 & ~1u));
        pair[cc] = (i0 & 1u) ? both.y : both.x;
        pair[cc + 1] = (i0 & 1u) ? both.x : both.y;
        if (i1 != (i0 ^ 1u))
            pair[cc + 1] = table[i1];
    }
    float f0 = 0.0f, f1 = 0.0f;
    for (int cc = 0; cc < 8; cc++)
    {
        f0 += w[cc] * (float)__builtin_bit_cast(_Float16, (uint16_t)(pair[cc] & 0xffffu));
        f1 += w[cc] * (float)__builtin_bit_cast(_Float16, (uint16_t)(pair[cc] >> 16));
    }
    return (uint32_t)to_bf16(f0) | ((uint32_t)to_bf16(f1) << 16);
}

__global__ __launch_bounds__(256) void k_nrc_grid(NrcDev P, RowSel sel, uint32_t n, uint32_t pad, uint32_t chunks,
                                                  EncDev E)
{
    const uint32_t turn = blockIdx.x / NRC_XCDS;
    const int l = (int)(blockIdx.x % NRC_XCDS + NRC_XCDS * (turn / chunks));
    const uint32_t row = (turn % chunks) * blockDim.x + threadIdx.x;
    const uint32_t rows = sel.rows();
    const uint32_t padded = (rows + pad - 1) / pad * pad;
    if (l >= P.levels || row >= n || row >= padded)
        return;
    uint32_t* out = E.feat + (size_t)l * E.stride + row;
    if (row >= rows)
    {
        *out = 0u;
        return;
    }
    float pos[3];
    for (int i = 0; i < 3; i++)
        pos[i] = E.pos[(size_t)i * E.stride + row];
    *out = grid_features(P, l, pos);
}

// Both in one launch for few rows: block row l of the levels, then one for the
// other inputs. A level's block reads the whole record for its position, which
// costs bandwidth that few rows leave free.
__global__ __launch_bounds__(256) void k_nrc_encode_few(NrcDev P, const float4* __restrict__ queries, RowSel sel,
                                                        uint32_t n, uint32_t pad, EncDev E)
{
    const uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    const int l = (int)blockIdx.y;
    const uint32_t rows = sel.rows();
    const uint32_t padded = (rows + pad - 1) / pad * pad;
    if (row >= n || row >= padded)
        return;
    if (l == P.levels)
    {
        write_inputs(P, queries, sel, row, rows, E);
        return;
    }
    uint32_t f = 0u;
    if (row < rows)
    {
        const float4 a = queries[4 * sel.record(row)];
        const float q[3] = {a.x, a.y, a.z};
        float pos[3];
        normalized_position(P, q, pos);
        f = grid_features(P, l, pos);
    }
    E.feat[(size_t)l * E.stride + row] = f;
}

// Rows of NRC_WIDTH inputs as the network counts them: the grid features,
// the other inputs, zeros. In one launch for few rows: `chunks` blocks for the
// other inputs, then the levels' in k_nrc_grid's order.
__global__ __launch_bounds__(256) void k_nrc_encode_rows(NrcDev P, const float4* __restrict__ queries, uint32_t n,
                                                         uint32_t chunks, uint32_t* __restrict__ out)
{
    const uint32_t turn = blockIdx.x / NRC_XCDS;
    int l = (int)(blockIdx.x % NRC_XCDS + NRC_XCDS * (turn / chunks));
    uint32_t chunk = turn % chunks;
    const uint32_t grid_blocks = (uint32_t)(P.levels + NRC_XCDS - 1) / NRC_XCDS * NRC_XCDS * chunks;
    if (blockIdx.x >= grid_blocks)
    {
        l = P.levels;
        chunk = blockIdx.x - grid_blocks;
    }
    else if (l >= P.levels)
        return;
    const uint32_t row = chunk * blockDim.x + threadIdx.x;
    if (row >= n)
        return;
    uint32_t* o = out + (size_t)row * (NRC_WIDTH / 2);
    if (l == P.levels)
    {
        uint32_t m[NRC_MISC / 2];
        float pos[3];
        record_inputs(P, queries, row, m, pos);
        for (int k = 0; k < NRC_MISC / 2; k++)
            o[l + k] = m[k];
        for (int k = l + NRC_MISC / 2; k < NRC_WIDTH / 2; k++)
            o[k] = 0u;
        return;
    }
    const float4 a = queries[4 * (size_t)row];
    const float q[3] = {a.x, a.y, a.z};
    float pos[3];
    normalized_position(P, q, pos);
    o[l] = grid_features(P, l, pos);
}

// The same from encoded planes (a thread per pair of inputs).
__global__ void k_nrc_rows(EncDev E, int levels, uint32_t n, uint32_t* __restrict__ out)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t row = (uint32_t)(i / (NRC_WIDTH / 2));
    const int k = (int)(i % (NRC_WIDTH / 2));
    if (row >= n)
        return;
    uint32_t v = 0u;
    if (k < levels)
        v = E.feat[(size_t)k * E.stride + row];
    else if (k - levels < NRC_MISC / 2)
        v = reinterpret_cast<const uint32_t*>(E.misc + (size_t)row * NRC_MISC)[k - levels];
    out[i] = v;
}

// The cache's encode workspace for n rows.
EncDev enc_buffer(Nrc& C, uint32_t n)
{
    EncDev E{};
    E.stride = (n + 63u) & ~63u;
    const size_t S = E.stride;
    const int levels = C.settings.grid_levels;
    C.enc.reserve(S * (4 * (size_t)levels + 2 * NRC_MISC + 4 * 3));
    E.feat = C.enc.as<uint32_t>();
    E.misc = reinterpret_cast<uint16_t*>(E.feat + S * levels);
    E.pos = reinterpret_cast<float*>(E.misc + S * NRC_MISC);
    return E;
}

// Up to here one launch encodes faster (16 levels of 2^19, 7 of 2^14): 300 rows
// 13.9 us an inference for 17.7 in two launches, 5000 rows 18.6 for 19.7; past it
// the order of levels over the XCDs counts: 20,000 rows 32.9 us (16.4) for 26.6
// (19.2), 60,000 61.5 us for 43.8, a million 478 us for 463. (The weights' loads
// going out together then took 1 to 2 us off every one of these.)
constexpr uint32_t FEW_ROWS = 16384;
// The same line for rows as the caller gets them (one launch against the planes'
// launches and k_nrc_rows; 16 levels of 2^19, 7 of 2^14): 1 to 5000 rows 6.2 us
// for 9.5 and 9.9, 20,000 rows 15.8 us (8.8) for 19.0 (14.2), 40,000 28.7 us (13.9) for
// 29.9 (17.3), 65,536 42.5 us (21.9) for 42.0 (22.4); there each row's 128 bytes
// are written 4 at a time from eight XCDs.
constexpr uint32_t FEW_OUTPUT_ROWS = 49152;

void encode_launch(const NrcDev& P, const float* d_queries, const RowSel& sel, uint32_t n, uint32_t pad,
                   const EncDev& E, hipStream_t s)
{
    const unsigned chunks = (n + 255u) / 256u;
    if (n <= FEW_ROWS)
    {
        hipLaunchKernelGGL(k_nrc_encode_few, dim3(chunks, (unsigned)P.levels + 1u), dim3(256), 0, s, P,
                           reinterpret_cast<const float4*>(d_queries), sel, n, pad, E);
        return;
    }
    const unsigned turns = ((unsigned)P.levels + NRC_XCDS - 1) / NRC_XCDS;
    hipLaunchKernelGGL(k_nrc_inputs, dim3(chunks), dim3(256), 0, s, P, reinterpret_cast<const float4*>(d_queries), sel,
                       n, pad, E);
    hipLaunchKernelGGL(k_nrc_grid, dim3(NRC_XCDS * turns * chunks), dim3(256), 0, s, P, sel, n, pad, chunks, E);
}

// ---------------------------------------------------------------------------
// Fused MLP
// ---------------------------------------------------------------------------
__device__ __forceinline__ void load_weights_lds(const uint16_t* __restrict__ src, uint16_t* dst, int count)
{
    for (int i = threadIdx.x * 8; i < count; i += blockDim.x * 8)
        *reinterpret_cast<uint4*>(dst + i) = *reinterpret_cast<const uint4*>(src + i);
}

// One layer on a 16-row tile: A fragments (two k-steps) times W^T (n-major
// [N][64] in LDS) -> D for the n-block nb.
__device__ __forceinline__ v4f layer_block(const v8bf a[2], const uint16_t* wt, int nb, int lane)
{
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const int n = 16 * nb + (lane & 15);
    for (int s = 0; s < 2; s++)
        acc = mfma(a[s], load_v8(wt + n * NRC_WIDTH + 32 * s + 8 * (lane >> 4)), acc);
    return acc;
}

typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

// Two binary32 -> bfloat16 (round to nearest even), in one instruction.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{a, b}), v2bf));
}

constexpr int FWD_FRAGS = (NRC_LAYERS - 1) * 8 + 2; // 64-lane weight fragments: 4 feature blocks x 2 k-steps a layer

// Inference: out[row] = MLP(encoded row) (RGB + 0), rows < count.
//
// Each layer is the transposed product W^T X^T: the rows are the columns of
// the MFMA's result, and a lane that holds features 16 mb + 4 g + i (g = lane / 16,
// i < 4) of a row feeds them to the next layer as they are, with the next
// weights' k order permuted to match (fragment (mb, s), slot 8 g + j of k-step s:
// feature 16 (2 s + j / 4) + 4 g + j % 4). The activations never leave the
// registers, and a weight fragment read from LDS serves the 64 rows (4
// columns blocks) of a wave: through LDS tiles of 16 rows, with the fragments
// read for each, 1,000,003 rows took 132 us.
__global__ __launch_bounds__(256, 3) void k_nrc_forward(const uint16_t* __restrict__ wt_global, EncDev E, int levels,
                                                     const uint32_t* count, uint32_t n, v4f_any* __restrict__ out)
{
    __shared__ uint4 frag[FWD_FRAGS * 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t rows = count && *count < n ? *count : n;
    if (blockIdx.x * 4u * 64u >= rows)
        return;
    // Every weight is on its way before the first is stored: with few rows the
    // launch is mostly this wait.
    uint4 v[(FWD_FRAGS + 3) / 4];
#pragma unroll
    for (int i = 0; i < (FWD_FRAGS + 3) / 4; i++)
    {
        const int f = wave + 4 * i < FWD_FRAGS ? wave + 4 * i : FWD_FRAGS - 1;
        const int layer = f < 40 ? f / 8 : 5, mb = f < 40 ? (f % 8) / 2 : 0, k_step = f % 2;
        const int g = lane >> 4;
        const uint16_t* w = wt_global + NRC_WOFF(layer) + (size_t)(16 * mb + (lane & 15)) * NRC_WIDTH;
        if (i >= 2) // layers past the first: two runs of four weights
        {
            const uint2 lo = *reinterpret_cast<const uint2*>(w + 32 * k_step + 4 * g);
            const uint2 hi = *reinterpret_cast<const uint2*>(w + 32 * k_step + 16 + 4 * g);
            v[i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
        }
        else
        {
            // layer 0 takes the grid features in k-step 0 and the other inputs
            // in step 1: pairs of weights, none past either's end
            const int first = k_step == 0 ? 8 * g : 2 * levels + 8 * g, end = k_step == 0 ? 2 * levels : NRC_WIDTH;
            uint32_t pair[4];
            for (int p = 0; p < 4; p++)
                pair[p] = first + 2 * p < end ? *reinterpret_cast<const uint32_t*>(w + first + 2 * p) : 0u;
            v[i] = make_uint4(pair[0], pair[1], pair[2], pair[3]);
        }
    }
#pragma unroll
    for (int i = 0; i < (FWD_FRAGS + 3) / 4; i++)
        if (wave + 4 * i < FWD_FRAGS)
            frag[(wave + 4 * i) * 64 + lane] = v[i];
    __syncthreads();
    const uint32_t tiles = (rows + 63) / 64;
    const int col = lane & 15, g = lane >> 4;
    for (uint32_t t = blockIdx.x * 4 + wave; t < tiles; t += gridDim.x * 4)
    {
        // rows 4 col + q of the 64 (q < 4: the column block)
        const uint32_t r = t * 64 + 4 * col;
        uint32_t x[4][2][4]; // [column block][k-step][8 bf16]
        for (int p = 0; p < 4; p++)
        {
            const int l = 4 * g + p;
            uint4 f = make_uint4(0u, 0u, 0u, 0u);
            if (l < levels)
                f = *reinterpret_cast<const uint4*>(E.feat + (size_t)l * E.stride + r);
            x[0][0][p] = f.x;
            x[1][0][p] = f.y;
            x[2][0][p] = f.z;
            x[3][0][p] = f.w;
        }
        for (int q = 0; q < 4; q++)
        {
            const uint4 m = *reinterpret_cast<const uint4*>(E.misc + (size_t)(r + q) * NRC_MISC + 8 * g);
            x[q][1][0] = m.x;
            x[q][1][1] = m.y;
            x[q][1][2] = m.z;
            x[q][1][3] = m.w;
        }
        auto operand = [](const uint32_t* v) { return __builtin_bit_cast(v8bf, make_uint4(v[0], v[1], v[2], v[3])); };
#pragma unroll 1
        for (int layer = 0; layer < NRC_LAYERS - 1; layer++)
        {
            uint32_t y[4][2][4];
#pragma unroll
            for (int mb = 0; mb < 4; mb++)
            {
                const v8bf a0 = __builtin_bit_cast(v8bf, frag[(layer * 8 + 2 * mb) * 64 + lane]);
                const v8bf a1 = __builtin_bit_cast(v8bf, frag[(layer * 8 + 2 * mb + 1) * 64 + lane]);
#pragma unroll
                for (int q = 0; q < 4; q++)
                {
                    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
                    acc = mfma(a0, operand(x[q][0]), acc);
                    acc = mfma(a1, operand(x[q][1]), acc);
                    y[q][mb >> 1][2 * (mb & 1)] = pack_bf16(fmaxf(acc[0], 0.0f), fmaxf(acc[1], 0.0f));
                    y[q][mb >> 1][2 * (mb & 1) + 1] = pack_bf16(fmaxf(acc[2], 0.0f), fmaxf(acc[3], 0.0f));
                }
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                for (int s = 0; s < 2; s++)
                    for (int i = 0; i < 4; i++)
                        x[q][s][i] = y[q][s][i];
        }
        const v8bf a0 = __builtin_bit_cast(v8bf, frag[40 * 64 + lane]);
        const v8bf a1 = __builtin_bit_cast(v8bf, frag[41 * 64 + lane]);
#pragma unroll
        for (int q = 0; q < 4; q++)
        {
            v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = mfma(a0, operand(x[q][0]), acc);
            acc = mfma(a1, operand(x[q][1]), acc);
            if (g == 0 && r + q < rows)
                out[r + q] = v4f_any{acc[0], acc[1], acc[2], 0.0f};
        }
    }
}

// Training: forward, loss gradient and backward of one 16-row tile per wave.
// Writes the layer inputs X_l and output gradients dY_l column-major
// ([64][batch_stride], bf16) for the weight-gradient GEMMs, dX0 (float,
// column-major) for the grid, and adds the loss to *loss_sum. Tiles
// cover the rows rounded up to 32 (the k-step of the dW GEMM); the encoded
// rows past the count are zero, so their activations and gradients are zero.
__global__ __launch_bounds__(256) void k_nrc_train_fwd_bwd(NrcTrainDev T)
{
    __shared__ uint16_t wt[NRC_WEIGHTS];   // W^T, [N][K]
    __shared__ uint16_t wk[NRC_WEIGHTS];   // W, [K][N]
    __shared__ uint16_t acts[4][NRC_LAYERS][16 * TILE_LD];
    load_weights_lds(T.wt, wt, NRC_WEIGHTS);
    load_weights_lds(T.wk, wk, NRC_WEIGHTS);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t rows = T.sel.rows();
    const uint32_t tiles_total = ((rows + 31) & ~31u) / 16;
    const uint32_t S = T.batch_stride;
    for (uint32_t t = blockIdx.x * 4 + wave; t < tiles_total; t += gridDim.x * 4)
    {
        const uint32_t r0 = t * 16;
        // layer-0 input tile (row-major in LDS) from the encoded rows: 4 rows
        // of a level's plane, and a quarter of a row's other inputs, per lane
        uint16_t* x_in = acts[wave][0];
        {
            const int l = lane >> 2, r = 4 * (lane & 3);
            if (l < T.levels)
            {
                const uint4 f = *reinterpret_cast<const uint4*>(T.enc.feat + (size_t)l * T.enc.stride + r0 + r);
                const uint32_t v[4] = {f.x, f.y, f.z, f.w};
                for (int i = 0; i < 4; i++)
                    *reinterpret_cast<uint32_t*>(x_in + (r + i) * TILE_LD + 2 * l) = v[i];
            }
            const int row = lane >> 2, k0 = 8 * (lane & 3);
            const uint4 m = *reinterpret_cast<const uint4*>(T.enc.misc + (size_t)(r0 + row) * NRC_MISC + k0);
            const uint32_t v[4] = {m.x, m.y, m.z, m.w};
            uint16_t* dst = x_in + row * TILE_LD + 2 * T.levels + k0;
            for (int i = 0; i < 4; i++)
                *reinterpret_cast<uint32_t*>(dst + 2 * i) = v[i];
            // zeros after them (with fewer than 16 levels)
            for (int k = 2 * T.levels + NRC_MISC + 2 * (lane & 3); k < NRC_WIDTH; k += 8)
                *reinterpret_cast<uint32_t*>(x_in + row * TILE_LD + k) = 0u;
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_wave_barrier();
        v4f pred = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int layer = 0; layer < NRC_LAYERS; layer++)
        {
            const uint16_t* xin = acts[wave][layer];
            // column-major copy of this layer's input for dW: lane = column
            {
                uint16_t* dst = T.xcm + (size_t)layer * NRC_WIDTH * S + (size_t)lane * S + r0;
                for (int r = 0; r < 16; r++)
                    dst[r] = xin[r * TILE_LD + lane];
            }
            v8bf a[2];
            for (int s = 0; s < 2; s++)
                a[s] = load_v8(xin + (lane & 15) * TILE_LD + 32 * s + 8 * (lane >> 4));
            const uint16_t* w = wt + NRC_WOFF(layer);
            if (layer < NRC_LAYERS - 1)
            {
                uint16_t* xo = acts[wave][layer + 1];
                for (int nb = 0; nb < 4; nb++)
                {
                    const v4f acc = layer_block(a, w, nb, lane);
                    for (int i = 0; i < 4; i++)
                        xo[(4 * (lane >> 4) + i) * TILE_LD + 16 * nb + (lane & 15)] = to_bf16(fmaxf(acc[i], 0.0f));
                }
                __builtin_amdgcn_s_waitcnt(0xc07f);
                __builtin_amdgcn_wave_barrier();
            }
            else
                pred = layer_block(a, w, 0, lane);
        }
        // relative L2: sum over rows and RGB of (p - y)^2 / (p^2 + 0.01); the
        // denominator is held constant in the gradient.
        uint16_t* dy = acts[wave][0]; // reuse: dY of the current layer, row-major
        float lsum = 0.0f;
        {
            const int col = lane & 15;
            for (int i = 0; i < 4; i++)
            {
                const uint32_t row = r0 + 4 * (lane >> 4) + i;
                float g = 0.0f;
                if (col < 3 && row < rows)
                {
                    const float p = pred[i];
                    const float y = T.targets[4 * T.sel.record(row) + col];
                    const float den = p * p + 0.01f;
                    const float d = p - y;
                    lsum += d * d / den;
                    g = 2.0f * d / den;
                }
                dy[(4 * (lane >> 4) + i) * TILE_LD + col] = to_bf16(g);
                dy[(4 * (lane >> 4) + i) * TILE_LD + 16 + col] = 0;
            }
        }
        for (int off = 32; off > 0; off >>= 1)
            lsum += __shfl_down(lsum, off, 64);
        if (lane == 0)
            atomicAdd(T.loss_sum, lsum);
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_wave_barrier();
        for (int layer = NRC_LAYERS - 1; layer >= 0; layer--)
        {
            const int N = layer == NRC_LAYERS - 1 ? NRC_OUT : NRC_WIDTH;
            // column-major copy of dY_layer for dW (lanes < N are columns)
            if (lane < N)
            {
                uint16_t* dst = T.dycm + (size_t)layer * NRC_WIDTH * S + (size_t)lane * S + r0;
                for (int r = 0; r < 16; r++)
                    dst[r] = dy[r * TILE_LD + lane];
            }
            // dX = dY W^T: A = dY (k' = n), B[k' = n][col = k] = W[k][n] from the [K][N] layout
            v8bf a[2];
            for (int s = 0; s < 2; s++)
            {
                const int n0 = 32 * s + 8 * (lane >> 4);
                if (n0 < N)
                    a[s] = load_v8(dy + (lane & 15) * TILE_LD + n0);
                else
                    a[s] = __builtin_bit_cast(v8bf, make_uint4(0u, 0u, 0u, 0u));
            }
            const uint16_t* w = wk + NRC_WOFF(layer);
            __builtin_amdgcn_s_waitcnt(0xc07f);
            __builtin_amdgcn_wave_barrier();
            for (int kb = 0; kb < 4; kb++)
            {
                v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
                const int k = 16 * kb + (lane & 15);
                for (int s = 0; s < 2; s++)
                {
                    const int n0 = 32 * s + 8 * (lane >> 4);
                    const v8bf b = n0 < N ? load_v8(w + k * N + n0) : __builtin_bit_cast(v8bf, make_uint4(0u, 0u, 0u, 0u));
                    acc = mfma(a[s], b, acc);
                }
                if (layer > 0)
                {
                    // ReLU mask of the layer input (the previous layer's output)
                    const uint16_t* xin = acts[wave][layer];
                    for (int i = 0; i < 4; i++)
                    {
                        const int r = 4 * (lane >> 4) + i;
                        const float m = from_bf16(xin[r * TILE_LD + k]) > 0.0f ? acc[i] : 0.0f;
                        dy[r * TILE_LD + k] = to_bf16(m);
                    }
                }
                else
                {
                    // gradient of the grid features (columns < 2 * levels)
                    const uint32_t row = r0 + 4 * (lane >> 4);
                    if (k < 2 * T.levels)
                        *reinterpret_cast<float4*>(T.dx0 + (size_t)k * S + row) =
                            make_float4(row < rows ? acc[0] : 0.0f, row + 1 < rows ? acc[1] : 0.0f,
                                        row + 2 < rows ? acc[2] : 0.0f, row + 3 < rows ? acc[3] : 0.0f);
                }
            }
            __builtin_amdgcn_s_waitcnt(0xc07f);
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// dW_l[k][n] += scale * sum_r X_l[r][k] dY_l[r][n] over one chunk of rows.
// Block = 4 waves = the 4 k-blocks of 16; each wave keeps the n-blocks of its
// k-block in registers and adds them to the FP32 gradient once.
__global__ __launch_bounds__(256) void k_nrc_weight_grad(NrcTrainDev T, uint32_t chunk)
{
    const int layer = blockIdx.y;
    const int lane = threadIdx.x & 63, kb = threadIdx.x >> 6;
    const uint32_t rows = T.sel.rows();
    const uint32_t rows_pad = (rows + 31) & ~31u;
    const uint32_t begin = blockIdx.x * chunk;
    if (begin >= rows_pad)
        return;
    const uint32_t end = begin + chunk < rows_pad ? begin + chunk : rows_pad;
    const int N = layer == NRC_LAYERS - 1 ? NRC_OUT : NRC_WIDTH;
    const int nbs = N / 16;
    const uint32_t S = T.batch_stride;
    const uint16_t* X = T.xcm + (size_t)layer * NRC_WIDTH * S;
    const uint16_t* D = T.dycm + (size_t)layer * NRC_WIDTH * S;
    v4f acc[4];
    for (int nb = 0; nb < 4; nb++)
        acc[nb] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const int k = 16 * kb + (lane & 15);
    for (uint32_t r = begin; r < end; r += 32)
    {
        const uint32_t rr = r + 8 * (lane >> 4);
        const v8bf a = load_v8(X + (size_t)k * S + rr);
        for (int nb = 0; nb < nbs; nb++)
        {
            const v8bf b = load_v8(D + (size_t)(16 * nb + (lane & 15)) * S + rr);
            acc[nb] = mfma(a, b, acc[nb]);
        }
    }
    const float scale = 1.0f / (3.0f * (float)rows);
    float* g = T.wgrad + NRC_WOFF(layer);
    for (int nb = 0; nb < nbs; nb++)
        for (int i = 0; i < 4; i++)
        {
            const int kk = 16 * kb + 4 * (lane >> 4) + i;
            const int nn = 16 * nb + (lane & 15);
            atomicAdd(g + kk * N + nn, acc[nb][i] * scale);
        }
}

// Grid gradient by global atomics: a thread per (row, level) adds the feature
// gradients to the level's 8 corners.
__global__ __launch_bounds__(128) void k_nrc_grid_grad(NrcDev P, NrcTrainDev T)
{
    const int l = (int)blockIdx.y;
    const uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t rows = T.sel.rows();
    if (row >= rows)
        return;
    float pos[3];
    for (int i = 0; i < 3; i++)
        pos[i] = T.enc.pos[(size_t)i * T.enc.stride + row];
    const uint32_t tmask = (1u << P.log2_table) - 1u;
    const float scale = 1.0f / (3.0f * (float)rows);
    const NrcGridLevel& L = P.level[l];
    const float g0 = T.dx0[(size_t)(2 * l) * T.batch_stride + row] * scale;
    const float g1 = T.dx0[(size_t)(2 * l + 1) * T.batch_stride + row] * scale;
    for (int cc = 0; cc < 8; cc++)
    {
        uint32_t idx;
        float w;
        corner(L, pos, cc, tmask, idx, w);
        const size_t e = ((size_t)l << P.log2_table) + idx;
        atomicAdd(T.ggrad + 2 * e, w * g0);
        atomicAdd(T.ggrad + 2 * e + 1, w * g1);
    }
}

// The same without global atomics on the gradient, which the memory side serves at
// 18 G/s however they are ordered, and slower where they meet in few entries
// (a step of 65,536 rows, 16 levels: 12.9 ms at 2^4 entries a level, 1.25 ms at
// 2^9; binned 0.32 ms both): the corner updates are binned by ranges of 2^log2_e
// table entries of a level (count, prefix sums, scatter), then a block adds the
// updates of one range in LDS and writes the range once.
struct GradBins {
    uint32_t* counts;  // [levels][ranges]
    uint32_t* cursors; // [levels][ranges]: first free place of each bin
    uint32_t* entry;   // [levels][rows * 8]: entry within its range
    float2* value;     // the same places: the two features' addends
    uint2* items;      // (bin, first update of it) a block adds; item_count of them
    uint32_t* item_count;
    uint32_t places;   // rows * 8: places of a level
    uint32_t first_row, rows; // this pass's rows
    int log2_e;
    uint32_t ranges;   // per level
};

// The 8 corners of a row at a level.
__device__ __forceinline__ void row_corners(const NrcDev& P, const EncDev& E, int l, uint32_t row, uint32_t idx[8],
                                            float w[8])
{
    float pos[3];
    for (int i = 0; i < 3; i++)
        pos[i] = E.pos[(size_t)i * E.stride + row];
    const uint32_t tmask = (1u << P.log2_table) - 1u;
#pragma unroll
    for (int cc = 0; cc < 8; cc++)
        corner(P.level[l], pos, cc, tmask, idx[cc], w[cc]);
}

constexpr int GRAD_BIN_BLOCK = 512;
constexpr int GRAD_ADD_BLOCK = 512;
constexpr uint32_t GRAD_SHARE = 8192; // updates a block adds (4096 and 16384: within 10 %)

__global__ void k_nrc_bins_reset(GradBins B, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        B.counts[i] = 0u;
    if (i == 0u)
        *B.item_count = 0u;
}

template <bool SCATTER>
__global__ __launch_bounds__(GRAD_BIN_BLOCK) void k_nrc_bin(NrcDev P, NrcTrainDev T, GradBins B)
{
    __shared__ uint32_t hist[GRAD_MAX_RANGES], base[GRAD_MAX_RANGES];
    const int l = (int)blockIdx.y;
    const uint32_t ranges = B.ranges;
    const uint32_t rows = T.sel.rows();
    const uint32_t end = min(B.first_row + B.rows, rows);
    const uint32_t row = B.first_row + blockIdx.x * GRAD_BIN_BLOCK + threadIdx.x;
    if (row - threadIdx.x >= end)
        return;
    for (uint32_t i = threadIdx.x; i < ranges; i += GRAD_BIN_BLOCK)
        hist[i] = 0u;
    __syncthreads();
    uint32_t idx[8], rank[8];
    float w[8];
    if (row < end)
    {
        row_corners(P, T.enc, l, row, idx, w);
#pragma unroll
        for (int cc = 0; cc < 8; cc++)
            rank[cc] = atomicAdd(&hist[idx[cc] >> B.log2_e], 1u);
    }
    __syncthreads();
    uint32_t* global = (SCATTER ? B.cursors : B.counts) + (size_t)l * ranges;
    for (uint32_t i = threadIdx.x; i < ranges; i += GRAD_BIN_BLOCK)
        if (hist[i] > 0u)
            base[i] = atomicAdd(&global[i], hist[i]);
    if (!SCATTER)
        return;
    __syncthreads();
    if (row >= end)
        return;
    const float scale = 1.0f / (3.0f * (float)rows);
    const float g0 = T.dx0[(size_t)(2 * l) * T.batch_stride + row] * scale;
    const float g1 = T.dx0[(size_t)(2 * l + 1) * T.batch_stride + row] * scale;
#pragma unroll
    for (int cc = 0; cc < 8; cc++)
    {
        const size_t at = (size_t)l * B.places + base[idx[cc] >> B.log2_e] + rank[cc];
        B.entry[at] = idx[cc] & ((1u << B.log2_e) - 1u);
        B.value[at] = make_float2(w[cc] * g0, w[cc] * g1);
    }
}

// Start of each bin within its level (one block per level), and the list of the
// blocks' shares: GRAD_SHARE updates of a bin at most.
__global__ __launch_bounds__(256) void k_nrc_bin_starts(GradBins B, uint32_t ranges)
{
    __shared__ uint32_t part[256];
    const uint32_t* counts = B.counts + (size_t)blockIdx.x * ranges;
    uint32_t* cursors = B.cursors + (size_t)blockIdx.x * ranges;
    const uint32_t per = (ranges + 255u) / 256u, first = threadIdx.x * per;
    uint32_t sum = 0u;
    for (uint32_t i = first; i < min(first + per, ranges); i++)
        sum += counts[i];
    part[threadIdx.x] = sum;
    __syncthreads();
    for (uint32_t off = 1; off < 256u; off <<= 1)
    {
        const uint32_t v = threadIdx.x >= off ? part[threadIdx.x - off] : 0u;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    uint32_t start = part[threadIdx.x] - sum;
    for (uint32_t i = first; i < min(first + per, ranges); i++)
    {
        cursors[i] = start;
        start += counts[i];
        const uint32_t shares = (counts[i] + GRAD_SHARE - 1u) / GRAD_SHARE;
        if (shares > 0u)
        {
            const uint32_t at = atomicAdd(B.item_count, shares);
            for (uint32_t k = 0; k < shares; k++)
                B.items[at + k] = make_uint2(blockIdx.x * ranges + i, k * GRAD_SHARE);
        }
    }
}

// A share of a bin: a whole bin's sums are added to the gradient by plain stores,
// those of a bin in several shares by atomics. The LDS serves float atomics at
// 3.6 cycles a lane: one block for the 300,000 updates that a coarse
// level's only bin gets from a frame took 730 us.
template <int LOG2_E>
__global__ __launch_bounds__(GRAD_ADD_BLOCK) void k_nrc_bin_add(NrcDev P, NrcTrainDev T, GradBins B)
{
    constexpr uint32_t ENTRIES = 1u << LOG2_E;
    __shared__ float4 sums4[ENTRIES / 2];
    float* sums = reinterpret_cast<float*>(sums4);
    if (blockIdx.x >= *B.item_count)
        return;
    const uint2 item = B.items[blockIdx.x];
    const uint32_t bin = item.x; // level * ranges + range
    const uint32_t ranges = B.ranges;
    const int l = (int)(bin / ranges);
    const uint32_t count = B.counts[bin], end = min(item.y + GRAD_SHARE, count);
    for (uint32_t i = threadIdx.x; i < ENTRIES / 2; i += GRAD_ADD_BLOCK)
        sums4[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    __syncthreads();
    // after the scatter the cursor is the bin's end
    const size_t first = (size_t)l * B.places + B.cursors[bin] - count;
#pragma unroll 4
    for (uint32_t i = item.y + threadIdx.x; i < end; i += GRAD_ADD_BLOCK)
    {
        const uint32_t e = B.entry[first + i];
        const float2 v = B.value[first + i];
        atomicAdd(&sums[2 * e], v.x);
        atomicAdd(&sums[2 * e + 1], v.y);
    }
    __syncthreads();
    float* out = T.ggrad + 2 * (((size_t)l << P.log2_table) + (size_t)(bin % ranges) * ENTRIES);
    if (count > GRAD_SHARE)
    {
        for (uint32_t i = threadIdx.x; i < 2 * ENTRIES; i += GRAD_ADD_BLOCK)
            if (sums[i] != 0.0f)
                atomicAdd(out + i, sums[i]);
        return;
    }
    float4* out4 = reinterpret_cast<float4*>(out);
    for (uint32_t i = threadIdx.x; i < ENTRIES / 2; i += GRAD_ADD_BLOCK)
    {
        const float4 v = sums4[i];
        if (v.x != 0.0f || v.y != 0.0f || v.z != 0.0f || v.w != 0.0f)
        {
            const float4 o = out4[i];
            out4[i] = make_float4(o.x + v.x, o.y + v.y, o.z + v.z, o.w + v.w);
        }
    }
}

void grid_grad_launch(Nrc& C, const NrcDev& P, const NrcTrainDev& T, uint32_t batch, hipStream_t s)
{
    const int lt = P.log2_table;
    const unsigned levels = (unsigned)P.levels;
    if (batch < grad_bin_min_rows(levels))
    {
        hipLaunchKernelGGL(k_nrc_grid_grad, dim3((batch + 127u) / 128u, levels), dim3(128), 0, s, P, T);
        return;
    }
    GradBins B{};
    // Both range sizes are within 6 % of each other from 2^15 to 2^19 entries
    // (16 levels of 37,000 rows, 2^10 against 2^13: 264 / 273 us and 381 / 376).
    // Below, the larger one leaves a level few blocks and sums in LDS that no
    // update reaches (2^14: 238 / 273); above, the smaller one splits the updates over
    // more ranges than there are blocks at a time (2^21: 792 / 745), and a level of
    // 2^24 has as many ranges of 2^13 as the histograms hold. A table smaller than a
    // range is one range, whose other sums stay 0.
    B.log2_e = lt <= 14 ? 10 : 13;
    const uint32_t ranges = lt > B.log2_e ? 1u << (lt - B.log2_e) : 1u;
    const uint32_t pass = std::min<uint32_t>(batch, GRAD_BIN_ROWS);
    B.ranges = ranges;
    const size_t bins = (size_t)levels * ranges, places = (size_t)8 * pass;
    const size_t max_items = bins + places * levels / GRAD_SHARE;
    C.grad_bins.reserve(8 * bins + 12 * places * levels + 8 * max_items + 8);
    B.value = C.grad_bins.as<float2>();
    B.items = reinterpret_cast<uint2*>(B.value + places * levels);
    B.entry = reinterpret_cast<uint32_t*>(B.items + max_items);
    B.counts = B.entry + places * levels;
    B.cursors = B.counts + bins;
    B.item_count = B.cursors + bins;
    B.places = (uint32_t)places;
    for (uint32_t r = 0; r < batch; r += pass)
    {
        B.first_row = r;
        B.rows = std::min(pass, batch - r);
        const dim3 grid((B.rows + GRAD_BIN_BLOCK - 1) / GRAD_BIN_BLOCK, levels);
        hipLaunchKernelGGL(k_nrc_bins_reset, dim3((unsigned)((bins + 255) / 256)), dim3(256), 0, s, B, (uint32_t)bins);
        hipLaunchKernelGGL(k_nrc_bin<false>, grid, dim3(GRAD_BIN_BLOCK), 0, s, P, T, B);
        hipLaunchKernelGGL(k_nrc_bin_starts, dim3(levels), dim3(256), 0, s, B, ranges);
        hipLaunchKernelGGL(k_nrc_bin<true>, grid, dim3(GRAD_BIN_BLOCK), 0, s, P, T, B);
        if (B.log2_e == 10)
            hipLaunchKernelGGL(k_nrc_bin_add<10>, dim3((unsigned)max_items), dim3(GRAD_ADD_BLOCK), 0, s, P, T, B);
        else
            hipLaunchKernelGGL(k_nrc_bin_add<13>, dim3((unsigned)max_items), dim3(GRAD_ADD_BLOCK), 0, s, P, T, B);
    }
}

// Adam (Kingma & Ba 2015) with bias correction; also writes the low-precision
// copies the kernels read and clears the gradient.
__global__ void k_nrc_adam_mlp(NrcTrainDev T, float lr1, float lr_scale_b1, float lr_scale_b2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= NRC_WEIGHTS || T.sel.rows() == 0)
        return;
    const float g = T.wgrad[i];
    T.wgrad[i] = 0.0f;
    float m = T.wm[i] = T.beta1 * T.wm[i] + (1.0f - T.beta1) * g;
    float v = T.wv[i] = T.beta2 * T.wv[i] + (1.0f - T.beta2) * g * g;
    const float mh = m / lr_scale_b1, vh = v / lr_scale_b2;
    const float p = T.wmaster[i] - lr1 * mh / (sqrtf(vh) + T.eps);
    T.wmaster[i] = p;
    // i indexes the [K][N] layout of its layer; mirror into [N][K]
    int layer = i < NRC_WOFF(NRC_LAYERS - 1) ? i / (NRC_WIDTH * NRC_WIDTH) : NRC_LAYERS - 1;
    const int N = layer == NRC_LAYERS - 1 ? NRC_OUT : NRC_WIDTH;
    const int local = i - NRC_WOFF(layer);
    const int k = local / N, n = local % N;
    const uint16_t b = to_bf16(p);
    T.wk_rw[i] = b;
    T.wt_rw[NRC_WOFF(layer) + n * NRC_WIDTH + k] = b;
}

__global__ void k_nrc_adam_grid(NrcTrainDev T, size_t count, float lr1, float lr_scale_b1, float lr_scale_b2)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count || T.sel.rows() == 0)
        return;
    const float g = T.ggrad[i];
    T.ggrad[i] = 0.0f;
    float m = T.gm[i] = T.beta1 * T.gm[i] + (1.0f - T.beta1) * g;
    float v = T.gv[i] = T.beta2 * T.gv[i] + (1.0f - T.beta2) * g * g;
    const float mh = m / lr_scale_b1, vh = v / lr_scale_b2;
    const float p = T.gmaster[i] - lr1 * mh / (sqrtf(vh) + T.eps);
    T.gmaster[i] = p;
    T.grid_rw[i] = (_Float16)p;
}

__global__ void k_set_u32(uint32_t* p, uint32_t v) { *p = v; }

__global__ void k_nrc_zero(float* p, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = 0.0f;
}

inline unsigned blocks_for(size_t n, int b) { return (unsigned)((n + b - 1) / b); }

uint32_t xorshift(uint32_t& s)
{
    s ^= s << 13;
    s ^= s >> 17;
    s ^= s << 5;
    return s;
}

uint16_t host_to_bf16(float x)
{
    uint32_t u;
    std::memcpy(&u, &x, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

} // namespace

void nrc_set_params(Ctx& ctx, const float* mlp_master, const float* grid_master)
{
    Nrc& C = ctx.nrc;
    if (mlp_master)
    {
        std::vector<uint16_t> wk(NRC_WEIGHTS), wt(NRC_WEIGHTS);
        for (int layer = 0; layer < NRC_LAYERS; layer++)
        {
            const int N = layer == NRC_LAYERS - 1 ? NRC_OUT : NRC_WIDTH;
            for (int k = 0; k < NRC_WIDTH; k++)
                for (int n = 0; n < N; n++)
                {
                    const int i = NRC_WOFF(layer) + k * N + n;
                    wk[i] = host_to_bf16(mlp_master[i]);
                    wt[NRC_WOFF(layer) + n * NRC_WIDTH + k] = wk[i];
                }
        }
        HIP_CHECK(hipMemcpy(C.w_master.ptr, mlp_master, 4 * NRC_WEIGHTS, hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(C.wk.ptr, wk.data(), 2 * NRC_WEIGHTS, hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(C.wt.ptr, wt.data(), 2 * NRC_WEIGHTS, hipMemcpyHostToDevice));
    }
    if (grid_master)
    {
        std::vector<_Float16> gh(C.grid_count);
        for (size_t i = 0; i < C.grid_count; i++)
            gh[i] = (_Float16)grid_master[i];
        HIP_CHECK(hipMemcpy(C.grid_master.ptr, grid_master, 4 * C.grid_count, hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(C.grid_f16.ptr, gh.data(), 2 * C.grid_count, hipMemcpyHostToDevice));
    }
}

void nrc_configure(Ctx& ctx, const mipt_radiance_cache_settings& s)
{
    Nrc& C = ctx.nrc;
    C.settings = s;
    const int L = s.grid_levels;
    const size_t T = (size_t)1 << s.grid_log2_table;
    C.grid_count = (size_t)L * T * 2;
    C.grid_f16.reserve(2 * C.grid_count);
    C.grid_master.reserve(4 * C.grid_count);
    C.grid_m.reserve(4 * C.grid_count);
    C.grid_v.reserve(4 * C.grid_count);
    C.grid_grad.reserve(4 * C.grid_count);
    C.w_master.reserve(4 * NRC_WEIGHTS);
    C.w_m.reserve(4 * NRC_WEIGHTS);
    C.w_v.reserve(4 * NRC_WEIGHTS);
    C.w_grad.reserve(4 * NRC_WEIGHTS);
    C.wt.reserve(2 * NRC_WEIGHTS);
    C.wk.reserve(2 * NRC_WEIGHTS);
    C.loss.reserve(64);
    // Host initialisation: Glorot-uniform weights, grid features U(-1e-4, 1e-4),
    // from a xorshift32 stream seeded with `seed`.
    uint32_t st = s.seed ? s.seed : 1u;
    std::vector<float> w(NRC_WEIGHTS);
    std::vector<uint16_t> wk(NRC_WEIGHTS), wt(NRC_WEIGHTS);
    for (int layer = 0; layer < NRC_LAYERS; layer++)
    {
        const int N = layer == NRC_LAYERS - 1 ? NRC_OUT : NRC_WIDTH;
        const int fan_out = layer == NRC_LAYERS - 1 ? 3 : NRC_WIDTH;
        const float lim = std::sqrt(6.0f / (float)(NRC_WIDTH + fan_out));
        for (int k = 0; k < NRC_WIDTH; k++)
            for (int n = 0; n < N; n++)
            {
                float u = (float)xorshift(st) * (1.0f / 4294967296.0f);
                float x = (2.0f * u - 1.0f) * lim;
                if (layer == NRC_LAYERS - 1 && n >= 3)
                    x = 0.0f;
                const int i = NRC_WOFF(layer) + k * N + n;
                w[i] = x;
                wk[i] = host_to_bf16(x);
                wt[NRC_WOFF(layer) + n * NRC_WIDTH + k] = wk[i];
            }
    }
    std::vector<float> gm(C.grid_count);
    std::vector<_Float16> gh(C.grid_count);
    for (size_t i = 0; i < C.grid_count; i++)
    {
        float u = (float)xorshift(st) * (1.0f / 4294967296.0f);
        gm[i] = (2.0f * u - 1.0f) * 1.0e-4f;
        gh[i] = (_Float16)gm[i];
    }
    HIP_CHECK(hipMemcpy(C.w_master.ptr, w.data(), 4 * NRC_WEIGHTS, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(C.wk.ptr, wk.data(), 2 * NRC_WEIGHTS, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(C.wt.ptr, wt.data(), 2 * NRC_WEIGHTS, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(C.grid_master.ptr, gm.data(), 4 * C.grid_count, hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(C.grid_f16.ptr, gh.data(), 2 * C.grid_count, hipMemcpyHostToDevice));
    for (DeviceBuffer* b : {&C.w_m, &C.w_v, &C.w_grad})
        HIP_CHECK(hipMemset(b->ptr, 0, 4 * NRC_WEIGHTS));
    for (DeviceBuffer* b : {&C.grid_m, &C.grid_v, &C.grid_grad})
        HIP_CHECK(hipMemset(b->ptr, 0, 4 * C.grid_count));
    C.step = 0;
    C.configured = true;
}

NrcDev nrc_dev(const Ctx& ctx)
{
    const Nrc& C = ctx.nrc;
    const mipt_radiance_cache_settings& s = C.settings;
    NrcDev P{};
    for (int a = 0; a < 3; a++)
        P.bmin[a] = ctx.scene_bmin[a];
    float ext = 0.0f;
    for (int a = 0; a < 3; a++)
        ext = std::fmax(ext, ctx.scene_bmax[a] - ctx.scene_bmin[a]);
    P.inv_extent = ext > 0.0f ? 1.0f / ext : 1.0f;
    P.levels = s.grid_levels;
    P.log2_table = s.grid_log2_table;
    const double T = std::ldexp(1.0, s.grid_log2_table);
    for (int l = 0; l < s.grid_levels; l++)
    {
        // Instant-NGP resolution schedule: scale_l = base * b^l - 1. Corners
        // reach floor(scale + 0.5) + 1 along an axis, so a dense level holds
        // floor(scale + 0.5) + 2 points per axis.
        const double scale = (double)s.grid_base_resolution * std::pow((double)s.grid_per_level_scale, l) - 1.0;
        const uint32_t res = (uint32_t)std::floor((double)(float)scale + 0.5) + 2u;
        P.level[l].scale = (float)scale;
        P.level[l].res = res;
        P.level[l].dense = (double)res * res * res <= T ? 1u : 0u;
    }
    P.grid_f16 = C.grid_f16.as<_Float16>();
    return P;
}

// Spreads the 10 low bits of v to every third bit.
__device__ __forceinline__ uint32_t spread3(uint32_t v)
{
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Morton key of each valid row's position (10 bits per axis of the grid's
// cube); rows past the count get the largest key and sort last.
__global__ void k_nrc_order_keys(NrcDev P, const float4* __restrict__ queries, const uint32_t* count, uint32_t n,
                                 uint32_t* __restrict__ keys, uint32_t* __restrict__ vals)
{
    const uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= n)
        return;
    vals[row] = row;
    if (row >= *count)
    {
        keys[row] = 0xffffffffu;
        return;
    }
    const float4 a = queries[4 * (size_t)row];
    const float q[3] = {a.x, a.y, a.z};
    float pos[3];
    normalized_position(P, q, pos);
    uint32_t c[3];
    for (int k = 0; k < 3; k++)
        c[k] = (uint32_t)fminf(pos[k] * 1024.0f, 1023.0f);
    keys[row] = spread3(c[0]) | (spread3(c[1]) << 1) | (spread3(c[2]) << 2);
}

__global__ void k_nrc_order_gather(const float4* __restrict__ queries, const uint32_t* __restrict__ pix,
                                   const uint32_t* __restrict__ perm, const uint32_t* count, float4* __restrict__ q_out,
                                   uint32_t* __restrict__ pix_out)
{
    const uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= *count)
        return;
    const uint32_t src = perm[row];
    for (int k = 0; k < 4; k++)
        q_out[4 * (size_t)row + k] = queries[4 * (size_t)src + k];
    pix_out[row] = pix[src];
}

void nrc_spatial_order(Ctx& ctx, const float4* d_queries, const uint32_t* d_pix, const uint32_t* d_count, uint32_t n,
                       float4* q_out, uint32_t* pix_out, hipStream_t s)
{
    Nrc& C = ctx.nrc;
    if (n == 0)
        return;
    C.sort_keys.reserve(4 * (size_t)n);
    C.sort_keys_out.reserve(4 * (size_t)n);
    C.sort_vals.reserve(4 * (size_t)n);
    C.sort_vals_out.reserve(4 * (size_t)n);
    const NrcDev P = nrc_dev(ctx);
    hipLaunchKernelGGL(k_nrc_order_keys, dim3(blocks_for(n, 256)), dim3(256), 0, s, P, d_queries, d_count, n,
                       C.sort_keys.as<uint32_t>(), C.sort_vals.as<uint32_t>());
    size_t tmp_bytes = 0;
    HIP_CHECK(rocprim::radix_sort_pairs(nullptr, tmp_bytes, C.sort_keys.as<uint32_t>(), C.sort_keys_out.as<uint32_t>(),
                                        C.sort_vals.as<uint32_t>(), C.sort_vals_out.as<uint32_t>(), (size_t)n, 0u, 32u,
                                        s));
    C.sort_tmp.reserve(tmp_bytes > 0 ? tmp_bytes : 1);
    HIP_CHECK(rocprim::radix_sort_pairs(C.sort_tmp.ptr, tmp_bytes, C.sort_keys.as<uint32_t>(),
                                        C.sort_keys_out.as<uint32_t>(), C.sort_vals.as<uint32_t>(),
                                        C.sort_vals_out.as<uint32_t>(), (size_t)n, 0u, 32u, s));
    hipLaunchKernelGGL(k_nrc_order_gather, dim3(blocks_for(n, 256)), dim3(256), 0, s, d_queries, d_pix,
                       C.sort_vals_out.as<uint32_t>(), d_count, q_out, pix_out);
    HIP_CHECK(hipGetLastError());
}

void nrc_infer(Ctx& ctx, const float* d_queries, const uint32_t* d_count, uint32_t n, float* d_out, hipStream_t s)
{
    Nrc& C = ctx.nrc;
    if (!C.configured)
        fail(MIPT_ERR_INVALID_ARGUMENT, "radiance cache not configured: call mipt_set_radiance_cache first");
    if (n == 0)
        return;
    const EncDev E = enc_buffer(C, n);
    const NrcDev P = nrc_dev(ctx);
    encode_launch(P, d_queries, RowSel{d_count, 1u, 0u, n}, n, 1u, E, s);
    const unsigned grid = (unsigned)std::min<size_t>(blocks_for((n + 63) / 64, 4), (size_t)ctx.cu_count * 3);
    hipLaunchKernelGGL(k_nrc_forward, dim3(grid), dim3(256), 0, s, C.wt.as<uint16_t>(), E, P.levels, d_count, n,
                       reinterpret_cast<v4f_any*>(d_out));
    HIP_CHECK(hipGetLastError());
}

void nrc_encode(Ctx& ctx, const float* d_queries, uint32_t n, uint16_t* d_out, hipStream_t s)
{
    Nrc& C = ctx.nrc;
    if (!C.configured)
        fail(MIPT_ERR_INVALID_ARGUMENT, "radiance cache not configured: call mipt_set_radiance_cache first");
    if (n == 0)
        return;
    const NrcDev P = nrc_dev(ctx);
    if (n <= FEW_OUTPUT_ROWS)
    {
        const unsigned chunks = (n + 255u) / 256u, turns = ((unsigned)P.levels + NRC_XCDS - 1) / NRC_XCDS;
        hipLaunchKernelGGL(k_nrc_encode_rows, dim3((NRC_XCDS * turns + 1u) * chunks), dim3(256), 0, s, P,
                           reinterpret_cast<const float4*>(d_queries), n, chunks, reinterpret_cast<uint32_t*>(d_out));
        HIP_CHECK(hipGetLastError());
        return;
    }
    const EncDev E = enc_buffer(C, n);
    encode_launch(P, d_queries, RowSel{nullptr, 1u, 0u, n}, n, 1u, E, s);
    hipLaunchKernelGGL(k_nrc_rows, dim3(blocks_for((size_t)n * (NRC_WIDTH / 2), 256)), dim3(256), 0, s, E,
                       (int)C.settings.grid_levels, n, reinterpret_cast<uint32_t*>(d_out));
    HIP_CHECK(hipGetLastError());
}

void nrc_gradients(Ctx& ctx, const float* d_queries, const float* d_targets, const uint32_t* d_count, uint32_t n,
                   uint32_t rec_stride, uint32_t rec_offset, bool clear_loss, hipStream_t s)
{
    Nrc& C = ctx.nrc;
    if (!C.configured)
        fail(MIPT_ERR_INVALID_ARGUMENT, "radiance cache not configured: call mipt_set_radiance_cache first");
    // rows of this batch at most (records below n)
    const uint32_t avail = n > rec_offset ? (n - rec_offset + rec_stride - 1) / rec_stride : 0u;
    const uint32_t batch = std::min<uint32_t>(avail, (uint32_t)C.settings.batch_size);
    C.last_sel_count = nullptr;
    if (batch == 0)
        return;
    const uint32_t stride = (batch + 31) & ~31u;
    const EncDev E = enc_buffer(C, stride);
    C.xcm.reserve(2 * (size_t)NRC_LAYERS * NRC_WIDTH * stride);
    C.dycm.reserve(2 * (size_t)NRC_LAYERS * NRC_WIDTH * stride);
    C.dx0.reserve(4 * (size_t)stride * NRC_GRID_MAX);
    C.count.reserve(4);
    const uint32_t* cnt = d_count;
    if (!cnt)
    {
        hipLaunchKernelGGL(k_set_u32, dim3(1), dim3(1), 0, s, C.count.as<uint32_t>(), n);
        cnt = C.count.as<uint32_t>();
    }
    const RowSel sel{cnt, rec_stride, rec_offset, batch};
    C.last_sel_count = cnt;
    C.last_sel_stride = rec_stride;
    C.last_sel_offset = rec_offset;
    C.last_sel_limit = batch;
    const NrcDev P = nrc_dev(ctx);
    // encode the batch; rows past its count up to a multiple of 32 are zero
    encode_launch(P, d_queries, sel, stride, 32u, E, s);
    if (clear_loss)
        hipLaunchKernelGGL(k_nrc_zero, dim3(1), dim3(64), 0, s, C.loss.as<float>(), (size_t)1);
    NrcTrainDev T{};
    T.wt = C.wt.as<uint16_t>();
    T.wk = C.wk.as<uint16_t>();
    T.enc = E;
    T.targets = d_targets;
    T.sel = sel;
    T.batch_stride = stride;
    T.levels = C.settings.grid_levels;
    T.xcm = C.xcm.as<uint16_t>();
    T.dycm = C.dycm.as<uint16_t>();
    T.dx0 = C.dx0.as<float>();
    T.loss_sum = C.loss.as<float>();
    T.wgrad = C.w_grad.as<float>();
    T.ggrad = C.grid_grad.as<float>();
    const unsigned grid = (unsigned)std::min<size_t>(blocks_for(stride / 16, 4), (size_t)ctx.cu_count);
    hipLaunchKernelGGL(k_nrc_train_fwd_bwd, dim3(grid), dim3(256), 0, s, T);
    const uint32_t chunk = 1024;
    hipLaunchKernelGGL(k_nrc_weight_grad, dim3(blocks_for(stride, chunk), NRC_LAYERS), dim3(256), 0, s, T, chunk);
    grid_grad_launch(C, P, T, batch, s);
    HIP_CHECK(hipGetLastError());
}

void nrc_train_pass(Ctx& ctx, hipStream_t s)
{
    Nrc& C = ctx.nrc;
    if (!C.configured || C.train_capacity == 0)
        fail(MIPT_ERR_INVALID_ARGUMENT,
             "RADIANCE_CACHE_TRAIN: no training records; run a path-trace pass with radiance_cache on first");
    const uint32_t cap = C.train_capacity;
    const uint32_t batch = (uint32_t)C.settings.batch_size;
    const uint32_t steps = (cap + batch - 1) / batch;
    const uint32_t* count = C.counters.as<uint32_t>() + 1;
    for (uint32_t i = 0; i < steps; i++)
    {
        nrc_gradients(ctx, C.train_queries.as<float>(), C.train_targets.as<float>(), count, cap, steps, i, i == 0,
                      s);
        nrc_apply_adam(ctx, s);
    }
}

void nrc_apply_adam(Ctx& ctx, hipStream_t s)
{
    Nrc& C = ctx.nrc;
    if (!C.last_sel_count)
        return; // no batch
    C.step++;
    const mipt_radiance_cache_settings& st = C.settings;
    const float b1t = 1.0f - (float)std::pow((double)st.adam_beta1, (double)C.step);
    const float b2t = 1.0f - (float)std::pow((double)st.adam_beta2, (double)C.step);
    NrcTrainDev T{};
    T.beta1 = st.adam_beta1;
    T.beta2 = st.adam_beta2;
    T.eps = st.adam_eps;
    T.wgrad = C.w_grad.as<float>();
    T.wm = C.w_m.as<float>();
    T.wv = C.w_v.as<float>();
    T.wmaster = C.w_master.as<float>();
    T.wk_rw = C.wk.as<uint16_t>();
    T.wt_rw = C.wt.as<uint16_t>();
    T.ggrad = C.grid_grad.as<float>();
    T.gm = C.grid_m.as<float>();
    T.gv = C.grid_v.as<float>();
    T.gmaster = C.grid_master.as<float>();
    T.grid_rw = C.grid_f16.as<_Float16>();
    T.sel = RowSel{C.last_sel_count, C.last_sel_stride, C.last_sel_offset, C.last_sel_limit};
    hipLaunchKernelGGL(k_nrc_adam_mlp, dim3(blocks_for(NRC_WEIGHTS, 256)), dim3(256), 0, s, T, st.learning_rate, b1t,
                       b2t);
    hipLaunchKernelGGL(k_nrc_adam_grid, dim3(blocks_for(C.grid_count, 256)), dim3(256), 0, s, T, C.grid_count,
                       st.learning_rate, b1t, b2t);
    HIP_CHECK(hipGetLastError());
}

} // namespace mipt
