// Device code shared by the MFMA translation units (moe_mfma.hip,
// moe_half.hip, moe_half_full.hip): vector types, the unit dealing over the
// XCDs, fp16 operand helpers and the grid bounds.
#pragma once

#include "moe_device.hpp"

#include <algorithm>

#pragma clang fp contract(off)

namespace moe {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int kSub = 32;                   // tokens per MFMA tile (N)
constexpr int kSubs = kMfmaTile / kSub;    // tiles per item
struct Unit {
    int item, slice;
    bool ok;
};

// blockIdx -> (item, slice).  Workgroup i runs on XCD i % 8; XCD x takes
// chunks of kUnitChunk consecutive units round-robin (chunk c goes to XCD
// c % 8), so the units of one item slice share an XCD while the work of the
// popular experts is spread over all XCDs.
constexpr int kUnitChunk = 4;

// The dealing permutes each round of 8 * kUnitChunk consecutive ids.  Within
// an XCD the dispatcher hands consecutive workgroups to its four shader
// engines in turn (measured: a workgroup's engine follows its position
// modulo 4 in the XCD's sequence for three quarters of them), so the unit
// at position p of chunk k is unit (p + k) % 4 of that chunk: the gate/up
// kernel's token tile `sub` (empty for the tail tiles of small items) then
// visits every engine instead of pinning the working tiles to one.
__device__ __forceinline__ int dealt_unit(int id) {
    const int n = id >> 3, x = id & 7, k = n / kUnitChunk;
    return (k * 8 + x) * kUnitChunk + (n + k) % kUnitChunk;
}

// Chunks of kGuChunkRows row slices per XCD (the gate/up kernel): the
// item-major sequence of (item, row slice) pairs is cut into chunks of
// kGuChunkRows, chunk c runs on XCD c % 8, and the activations of an item's
// token tiles, read by every row slice, are fetched into fewer L2s.  Within a
// chunk, row slice r's token tiles are rotated by r + c over the four
// positions so each engine sees every tile index.  Chunk rows, layer ms
// (2048/512, two runs each): 1 (one row slice): 4K 1.47-1.49, 16K 4.61,
// stack 26.65; 4: 1.47-1.48, 4.53-4.55, 26.56; 8: 1.46-1.47, 4.51-4.56,
// 26.90; 16 (whole items): 1.48-1.50, 4.52, 27.7 (items dealt whole leave
// the XCDs unevenly loaded on the stack's 1,032-token layers).
constexpr int kGuChunkRows = 4;
template<int Rows = kGuChunkRows>
__device__ __forceinline__ Unit row_chunk_unit(int count, int slices) {
    constexpr int kGuChunk = Rows * kSubs;   // units of one chunk
    const int id = static_cast<int>(blockIdx.x);
    const int n = id >> 3, x = id & 7, k = n / kGuChunk, p = n - k * kGuChunk;
    const int rl = p / kSubs;
    const int u = (k * 8 + x) * kGuChunk + rl * kSubs + (p + rl + k) % kSubs;
    Unit r;
    r.ok = u < count * slices;
    r.item = r.ok ? u / slices : 0;
    r.slice = r.ok ? u % slices : 0;
    return r;
}

__device__ __forceinline__ Unit mfma_unit(int count, int slices) {
    const int units = count * slices;
    const int u = dealt_unit(static_cast<int>(blockIdx.x));
    Unit r;
    r.ok = u < units;
    r.item = r.ok ? u / slices : 0;
    r.slice = r.ok ? u % slices : 0;
    return r;
}

__device__ __forceinline__ float half_lo(uint32_t w) { return h2f(w); }
__device__ __forceinline__ float half_hi(uint32_t w) { return h2f(w >> 16); }

// 8 fp16 values as an MFMA operand.
__device__ __forceinline__ v8h pack8(const uint32_t (&w)[4]) {
    v4i v = {static_cast<int>(w[0]), static_cast<int>(w[1]), static_cast<int>(w[2]), static_cast<int>(w[3])};
    return __builtin_bit_cast(v8h, v);
}

// fp16 -> fp32 conversions the compiler cannot fold into v_fma_mix_f32.  On
// gfx950 v_fma_mix_f32 issues at about the rate of a conversion (measured:
// 0.5 wave-instructions per SIMD per ns against 0.9 for v_fma_f32, v_mul_f32
// and v_add_f32), so a scale used by several products is converted once and
// the products are plain fp32 fmas.  (Same values: fp16 -> fp32 is exact.)
__device__ __forceinline__ float cvt_half_lo(uint32_t w) {
    float r;
    asm("v_cvt_f32_f16 %0, %1" : "=v"(r) : "v"(w));
    return r;
}
__device__ __forceinline__ float cvt_half_hi(uint32_t w) {
    float r;
    asm("v_cvt_f32_f16_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_1" : "=v"(r) : "v"(w));
    return r;
}

// acc[v] = fma(d4[v], fma(float(I[v]), d8, c4), acc[v]); d4 read as fp16 by
// v_fma_mix_f32 (lo / hi half of each word).
__device__ __forceinline__ float fma_mix_lo(uint32_t h2, float t, float acc) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h2), "v"(t), "v"(acc));
    return r;
}
__device__ __forceinline__ float fma_mix_hi(uint32_t h2, float t, float acc) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h2), "v"(t), "v"(acc));
    return r;
}

// SiLU(gate) * up and the middle Q8 of one 32-row tile, its gate and up waves
// sharing the work (the IEEE divisions, expf and rounding of 32 tokens took the
// gate wave alone about 750 instructions while the up wave idled; shared, the
// 2560/640 layer of 3,001 tokens 2053 -> 2002 us): wave `mat` finishes
// tokens 16 mat .. + 15, lane l rows 8 (l / 16) .. + 7 of token 16 mat + l % 16.
// gate / up: [register v][lane] of the tile's sums (row 16h + v, token m); token
// i of the tile is pair first + j0 + i, valid below ncols.
template<bool Dbg>
__device__ __forceinline__ void finish_gate_up(const FfnArgs &a, const float (*gate)[64], const float (*up)[64], int mat,
                                               int first, int j0, int ncols, int R0) {
    const int lane = threadIdx.x & 63, nbi = a.shape.I / 32;
    const int part = lane >> 4, m = 16 * mat + (lane & 15), j = j0 + m;
    int flags = 0;
    float mid[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int v = 8 * (part & 1) + e, l = 32 * (part >> 1) + m;
        mid[e] = silu_mul(gate[v][l], up[v][l], flags);
    }
    float keep[8];
    if constexpr (Dbg) {
#pragma unroll
        for (int e = 0; e < 8; ++e) keep[e] = mid[e];
    }
    const Q8Part<4> q8 = quantize_part<4>(mid);
    if (j < ncols) {
        const size_t pair = static_cast<size_t>(first + j), mb = pair * nbi + R0 / 32;
        *reinterpret_cast<uint2 *>(a.mq.codes + mb * 32 + 8 * part) = make_uint2(q8.codes[0], q8.codes[1]);
        if (part == 0) a.mq.heads[mb] = q8.head;
        if constexpr (Dbg) {
            if (a.middle_f32)
#pragma unroll
                for (int e = 0; e < 8; ++e) a.middle_f32[pair * a.shape.I + R0 + 8 * part + e] = keep[e];
        }
        const int f = flags | (part == 0 ? q8.flags : 0);
        if (f) atomicOr(a.error, f);
    }
}

constexpr uint32_t kNibbles = 0x0f0f0f0fu;
constexpr int kGuMaxBlocks = 64, kGu96MaxBlocks = 96;

// Upper bound on MFMA items: a group of n >= mfma_min pairs gives
// ceil(n / 128) items, and at most min(Ep, pairs / mfma_min) groups qualify.
inline size_t mfma_item_bound(const FfnArgs &a) {
    const size_t P = static_cast<size_t>(a.pairs_bound);
    const size_t G = std::min(P, static_cast<size_t>(a.shape.Ep));
    const size_t big = a.mfma_min >= 1 ? std::min(G, P / static_cast<size_t>(a.mfma_min)) : G;
    return std::max<size_t>(P / kMfmaTile + big, 1);
}

// row_chunk_unit's grid: the units rounded up to whole rounds of 8 chunks.
inline unsigned chunk_grid(const FfnArgs &a, int slices, int rows = kGuChunkRows) {
    const size_t units = mfma_item_bound(a) * static_cast<size_t>(slices);
    const size_t round = 8 * static_cast<size_t>(rows) * kSubs;
    return static_cast<unsigned>((units + round - 1) / round * round);
}

}  // namespace
}  // namespace moe
