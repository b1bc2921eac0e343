#pragma once

#include "moe_mfma_device.hpp"

#pragma clang fp contract(off)

namespace moe {
namespace {

// ---- fp16 fragment dots over operands staged in LDS (rows of <= 64 blocks).
// The matrix core takes both sides without a conversion (moe_internal.hpp,
// half_slot): nibbles as fp16 subnormals n * 2^-24 / n * 2^-20 and the codes
// from the fp16 operand plane; the result is float(I_f) * 2^-24 exactly, so
// the int32 -> fp32 conversions of an int8 MFMA (a fifth of the epilogue) are
// gone and the power of two moves into d8: fma(I 2^-24, d8 2^24, -4 s8) rounds
// the same real number.
//
// What bounds it: VALU issue (counters: VALU active 95 % of the time at about
// 4 cycles an instruction), so what counts is instructions per leaf: 322 with
// int8 dots, 257 here, 192 of them the reference's own fma / multiply / adds.
// The operands are 64 bytes a block, and reading them per lane from L2
// touches 32 lines an instruction (measured: 4K layer 1.39 -> 1.63 ms), so
// a workgroup of 4 waves (4 row tiles of 32 against the same 32 tokens) copies
// each node's blocks into LDS with whole 128-byte lines, double buffered,
// one barrier per node, and the heads are converted once per workgroup.
// Three waves per SIMD matter more than overlap inside a wave: tree levels 3-4
// are parked in LDS to stay under 168 VGPRs (4K / 16K layers, us: all levels
// in registers, two waves 1470 / 4660; the same with every MFMA and LDS read
// issued a step ahead 1336 / 4280; this form 1250 / 4003).
constexpr float kHalfScale = 16777216.0f;   // 2^24
constexpr int kHtWaves = 4;                 // waves (row tiles) per workgroup
constexpr int kHtThreads = 64 * kHtWaves;

// The 8 nibbles of dword 2F + h of a chunk in half_slot order.
__device__ __forceinline__ v8h nibble_operand(uint32_t d) {
    const uint32_t e = d >> 8;
    return pack8({d & 0x000f000fu, e & 0x000f000fu, d & 0x00f000f0u, e & 0x00f000f0u});
}
__device__ __forceinline__ v16f frag_dot(uint32_t nibbles, uint4 x) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(nibble_operand(nibbles), pack8({x.x, x.y, x.z, x.w}), v16f{}, 0, 0, 0);
}
// fma(d4, fma(float(I), d8, -4 s8), +0) with F = float(I) 2^-24, s = {d8 2^24, -4 s8}.
__device__ __forceinline__ float half_value(float F, float2 s, const uint32_t (&d4)[8], int v) {
    const float t = fmaf(F, s.x, s.y);
    return (v & 1) ? mul_half_hi(d4[v >> 1], t) : mul_half_lo(d4[v >> 1], t);
}

// tree_merge with the merged node left in w (after node 15: the tree's sum).
__device__ __forceinline__ void merge_node(float (*park)[16][64], int lane, int p, float (&w)[16], float (&l1)[16],
                                           float (&l2)[16]) {
    if ((p & 1) == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) l1[i] = w[i];
        return;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = l1[i] + w[i];
    if ((p & 2) == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) l2[i] = w[i];
        return;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = l2[i] + w[i];
    if ((p & 4) == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) park[0][i][lane] = w[i];
        return;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = park[0][i][lane] + w[i];
    if ((p & 8) == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) park[1][i][lane] = w[i];
        return;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = park[1][i][lane] + w[i];
}

struct HalfLds {
    uint4 x[2][2][32][8];                        // [buffer][blocks 2p, +1 / 2p + 32, +33][token][piece, swizzled]
    float2 hd[2][4][32];                         // [buffer][block][token]: d8 * 2^24, -4 s8
    uint4 d4[2][kHtWaves][4][4];                 // [buffer][wave][block][32 halfs]
    float park[kHtWaves][2][16][64];             // [wave]: pending tree levels 3, 4
};

// One wave's 32 rows and the workgroup's token columns.
struct HalfTile {
    __amdgpu_buffer_rsrc_t wr, sr, xr, hr;   // weight codes and scales of the 32 rows; token operands and heads
    uint32_t x_base, h_base;                 // staged token's row (tid / 8) in xr, head token's row (tid % 32) in hr
    int nb;
};

// Canon: xr / hr are canonical 36-byte blocks, converted to operands while
// they are staged (once per workgroup).
template<bool Canon> constexpr uint32_t HtXStride = Canon ? 36u : 64u;
template<bool Canon> constexpr uint32_t HtHStride = Canon ? 36u : 4u;

// Four codes as fp16 in half_slot order, high: divided by 16.  code ^ 0x80
// under 0x64 is the fp16 1024 + (code + 128).
__device__ __forceinline__ uint2 codes_to_half(uint32_t c, bool high) {
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    const uint32_t u = c ^ 0x80808080u;
    const v2h a = __builtin_bit_cast(v2h, (u & 0x00ff00ffu) | 0x64006400u);
    const v2h b = __builtin_bit_cast(v2h, ((u >> 8) & 0x00ff00ffu) | 0x64006400u);
    const v2h o = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
    const v2h q = {static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
    const v2h p = {static_cast<_Float16>(-72.0f), static_cast<_Float16>(-72.0f)};
    return make_uint2(__builtin_bit_cast(uint32_t, high ? __builtin_elementwise_fma(a, q, p) : a + o),
                      __builtin_bit_cast(uint32_t, high ? __builtin_elementwise_fma(b, q, p) : b + o));
}

// The tree of the wave's 32 rows over the workgroup's 32 tokens, left in nd
// (register v of lane half h, lane m: row 16h + v, token m).  Every wave of the
// workgroup runs it (barriers); Full: 64 blocks, no block of a node is missing.
// A missing block is staged as zeros (operand, head and scale), so its value
// is the +0 of the reference's unused lane; nodes and halves of nodes without
// a block are left out (no lane value is -0, so adding +0 changes nothing).  dots(p, i, q, F0, F1) receives the
// fragments of block 2p + i + 32q in the debug build.
template<bool Full, bool Canon, bool Dbg, class Dots>
__device__ __forceinline__ void half_tree(HalfLds &st, const HalfTile &t, int wave, float (&nd)[16], Dots &&dots) {
    constexpr int Q = 2;   // block pairs of node p: 2p, 2p + 32
    constexpr uint32_t xst = HtXStride<Canon>, hst = HtHStride<Canon>;
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, h = lane >> 5;
    const int nb = t.nb;
    const int prow = 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
    const uint32_t row_bytes = static_cast<uint32_t>(nb) * 16u;
    const uint32_t w_off = static_cast<uint32_t>(prow) * row_bytes + 32u * 16u * h;      // block 2p + i (+ 32 h)
    // Staging: thread t moves piece t % 8 (block of the pair, lane half,
    // fragment) of token t / 8 for both pairs; thread t < 128 the head of
    // token t % 32, block t / 32; lane l < 16 of a wave scale group l / 4 of
    // block l % 4.
    const int tok = tid >> 3, piece = tid & 7, slot = piece ^ ((tok >> 1) & 7);
    const int pi = piece >> 2, ph = (piece >> 1) & 1, pf = piece & 1;
    const uint32_t x_off = t.x_base + static_cast<uint32_t>(pi) * xst + (Canon ? 4u + 8u * pf + 4u * ph : 16u * (piece & 3));
    const int hb = tid >> 5;                                        // block slot: pair hb / 2, block hb % 2
    const int hblk = (hb & 1) + 32 * (hb >> 1);
    const uint32_t h_off = t.h_base + static_cast<uint32_t>(hblk) * hst;
    const int sblk = lane & 3, sgrp = lane >> 2;
    const int sb = (sblk & 1) + 32 * (sblk >> 1);
    const uint32_t s_off = static_cast<uint32_t>((sgrp & 3) * nb + sb) * 16u;

    uint4 xs[Q];
    uint4 wn[2], dn;
    uint32_t hs = 0;
    auto fetch = [&](int p) {
        const uint32_t b0 = static_cast<uint32_t>(2 * p);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const bool ok = Full || static_cast<int>(b0) + pi + 32 * q < nb;
            const uint32_t o = (b0 + 32u * q) * xst;
            if constexpr (Canon) {
                xs[q].x = ok ? buffer_load4(t.xr, x_off, o) : 0u;
                xs[q].y = ok ? buffer_load4(t.xr, x_off, o + 16u) : 0u;
            } else {
                xs[q] = make_uint4(0, 0, 0, 0);
                if (ok) xs[q] = buffer_load16(t.xr, x_off, o);
            }
        }
        if (wave < 2) {
            hs = 0;
            if (Full || static_cast<int>(b0) + hblk < nb) hs = buffer_load4(t.hr, h_off, b0 * hst);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) wn[i] = buffer_load16(t.wr, w_off, (b0 + i) * 16u);
        dn = make_uint4(0, 0, 0, 0);
        if (Full || static_cast<int>(b0) + sb < nb) dn = buffer_load16(t.sr, s_off, b0 * 16u);
    };
    auto commit = [&](int buf) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            if constexpr (Canon) {
                const uint2 lo = codes_to_half(xs[q].x, false), hi = codes_to_half(xs[q].y, true);
                st.x[buf][q][tok][slot] = make_uint4(lo.x, lo.y, hi.x, hi.y);
            } else {
                st.x[buf][q][tok][slot] = xs[q];
            }
        }
        if (wave < 2) st.hd[buf][hb][tid & 31] = make_float2(cvt_half_lo(hs) * kHalfScale, -4.0f * cvt_half_hi(hs));
        if (lane < 16) st.d4[buf][wave][sblk][sgrp] = dn;
    };
    fetch(0);
    commit(0);
    __syncthreads();

    const int xrow = 8 * m + ((2 * h) ^ ((m >> 1) & 7));   // piece 4 i + 2 h + f of token m: xrow ^ (4 i + f)
    float l1[16], l2[16];
#pragma unroll 1
    for (int p = 0; p < 16; ++p) {
        if (!Full && 2 * p >= nb) {   // uniform: no block left in this node or any later one
#pragma unroll
            for (int v = 0; v < 16; ++v) nd[v] = 0.0f;
            merge_node(st.park[wave], lane, p, nd, l1, l2);
            continue;
        }
        const int buf = p & 1;
        const bool both = Full || 2 * p + 32 < nb;   // uniform: the node has blocks 2p + 32, + 33
        const uint4 w[2] = {wn[0], wn[1]};
        fetch(p < 15 ? p + 1 : p);
        __builtin_amdgcn_sched_barrier(0);
        // An opaque zero keeps the operand addresses (one register and XORs)
        // from being hoisted out of the loop into registers.
        int zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        const int row = xrow + zero;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t wv[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
            const auto scales = [&](int blk, uint32_t (&d)[8]) {
                const uint4 q0 = st.d4[buf][wave][blk][2 * h], q1 = st.d4[buf][wave][blk][2 * h + 1];
                d[0] = q0.x; d[1] = q0.y; d[2] = q0.z; d[3] = q0.w;
                d[4] = q1.x; d[5] = q1.y; d[6] = q1.z; d[7] = q1.w;
            };
            uint32_t da[8], db[8];
            scales(i, da);
            scales(2 + i, db);
            const float2 sa = st.hd[buf][i][m], sb2 = st.hd[buf][2 + i][m];
            float u[2][16];
            v16f ka[2], kb[2];
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                const auto r = __builtin_amdgcn_permlane32_swap(wv[2 * f], wv[2 * f + 1], false, false);
                const int sl = row ^ (4 * i + f);
                const v16f Fa = frag_dot(r[0], (&st.x[buf][0][0][0])[sl]);
                if (both) {
                    const v16f Fb = frag_dot(r[1], (&st.x[buf][1][0][0])[sl]);
#pragma unroll
                    for (int v = 0; v < 16; ++v) u[f][v] = half_value(Fa[v], sa, da, v) + half_value(Fb[v], sb2, db, v);
                    if constexpr (Dbg) kb[f] = Fb;
                } else {
#pragma unroll
                    for (int v = 0; v < 16; ++v) u[f][v] = half_value(Fa[v], sa, da, v);
                }
                if constexpr (Dbg) ka[f] = Fa;
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float leaf = u[0][v] + u[1][v];
                nd[v] = i == 0 ? leaf : nd[v] + leaf;
            }
            if constexpr (Dbg) {
                dots(p, i, 0, ka[0], ka[1]);
                if (both) dots(p, i, 1, kb[0], kb[1]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        merge_node(st.park[wave], lane, p, nd, l1, l2);
        commit(buf ^ 1);
        __syncthreads();
    }
}

// Gate / up: waves 2r and 2r + 1 take the gate and up rows of row tile r (two
// tiles of 32 rows a workgroup) against token tile `sub` of an MFMA item, then
// share the tile's SiLU and quantisation (finish_gate_up).
constexpr int kGuTiles = kHtWaves / 2;

template<bool Full, bool Dbg>
__global__ __launch_bounds__(kHtThreads, Dbg ? 2 : 3) void k_gate_up_half(FfnArgs a) {
    __shared__ HalfLds st;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int mat = wave & 1, rs = wave >> 1;
    const int H = a.shape.H, I = a.shape.I, nb = H / 32, nbi = I / 32;
    const int slices = (nbi + kGuTiles - 1) / kGuTiles * kSubs;
    const Unit un = row_chunk_unit<kGuChunkRows / kGuTiles>(a.routes.item_counts[1], slices);
    if (!un.ok) return;   // uniform per workgroup
    const Item *itp = a.routes.mfma_items + un.item;
    const int expert = itp->expert, first = itp->first, ncols = itp->ncols;
    const int sub = un.slice % kSubs;
    if (kSub * sub >= ncols) return;   // uniform per workgroup: no tokens in this tile
    const int rt = un.slice / kSubs * kGuTiles + rs;    // 32-row tile
    const bool active = rt < nbi;                       // wave-uniform; an idle wave repeats the last tile
    const int R0 = std::min(rt, nbi - 1) * 32;
    const int tid = threadIdx.x, lane = tid & 63;

    const size_t rbase = static_cast<size_t>(expert) * I + R0;
    const uint32_t row_bytes = static_cast<uint32_t>(nb) * 16u;
    const auto token_row = [&](int i) {   // activation row of the tile's token i (past ncols: the last one)
        return static_cast<uint32_t>(a.routes.pair_token[first + std::min(kSub * sub + i, ncols - 1)]) * static_cast<uint32_t>(nb);
    };
    HalfTile t;
    t.wr = buffer_rsrc((mat ? a.bank.up_codes : a.bank.gate_codes) + rbase * row_bytes, 32u * row_bytes);
    t.sr = buffer_rsrc((mat ? a.bank.up_scales : a.bank.gate_scales) + rbase * nb, 32u * static_cast<uint32_t>(nb) * 2u);
    t.xr = buffer_rsrc(a.xhalf, static_cast<uint32_t>(a.tokens) * static_cast<uint32_t>(nb) * 64u);
    t.hr = buffer_rsrc(a.xq.heads, static_cast<uint32_t>(a.tokens) * static_cast<uint32_t>(nb) * 4u);
    t.x_base = token_row(tid >> 3) * 64u;
    t.h_base = token_row(tid & 31) * 4u;
    t.nb = nb;
    float res[16];
    half_tree<Full, false, Dbg>(st, t, wave, res, [&](int p, int i, int q, v16f F0, v16f F1) {
        if constexpr (Dbg) {
            int32_t *dots = mat ? a.up_dots : a.gate_dots;
            const int m = lane & 31, j = kSub * sub + m, b = 2 * p + i + 32 * q;
            if (dots && active && j < ncols && b < nb)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    dots[(static_cast<size_t>(first + j) * I + R0 + 16 * (lane >> 5) + v) * nb + b] =
                        static_cast<int>((F0[v] + F1[v]) * kHalfScale);
        }
    });
    // Both waves' sums, each in its own wave's park area: no barrier follows the
    // merges of nodes without blocks, so the other wave may still be merging.
    const float (*xch[2])[64] = {st.park[2 * rs][0], st.park[2 * rs + 1][0]};   // [mat][v][lane]
#pragma unroll
    for (int v = 0; v < 16; ++v) st.park[wave][0][v][lane] = res[v];
    __syncthreads();
    if (!active) return;
    finish_gate_up<Dbg>(a, xch[0], xch[1], mat, first, kSub * sub, ncols, R0);
}

// Q4_0 linear on wide grids: 4 row tiles of 32 a workgroup against the same 32
// columns.  Ids are XCD-aware: the column tiles of one row group run on one
// XCD.  (The tree of one tile is one wave's work here; k_linear_mfma splits it
// over a workgroup for grids that leave SIMDs idle.)
template<bool Full, bool Canon>
__global__ __launch_bounds__(kHtThreads, 3) void k_linear_half(LinearMfmaArgs a) {
    __shared__ HalfLds st;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int id = static_cast<int>(blockIdx.x), local = id >> 3;
    const int rg = (id & 7) + 8 * (local / a.col_tiles), c0 = local % a.col_tiles * kSub;
    if (rg * kHtWaves >= a.row_tiles) return;   // uniform per workgroup (grid padded to 8 row groups)
    const int rt = rg * kHtWaves + wave;
    const bool active = rt < a.row_tiles;       // wave-uniform; an idle wave repeats the last tile
    const int R0 = std::min(rt, a.row_tiles - 1) * 32, nb = a.nb;
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t row_bytes = static_cast<uint32_t>(nb) * 16u;
    const auto column_row = [&](int i) {   // column c0 + i's first block (past N: the last column)
        return static_cast<uint32_t>(std::min(c0 + i, a.N - 1)) * static_cast<uint32_t>(nb);
    };
    HalfTile t;
    t.wr = buffer_rsrc(a.codes + static_cast<size_t>(R0) * row_bytes, 32u * row_bytes);
    t.sr = buffer_rsrc(a.scales + static_cast<size_t>(R0) * nb, 32u * static_cast<uint32_t>(nb) * 2u);
    const uint32_t blocks = static_cast<uint32_t>(a.N) * static_cast<uint32_t>(nb);
    t.xr = Canon ? buffer_rsrc(a.q8, blocks * 36u) : buffer_rsrc(a.xq.codes, blocks * 64u);
    t.hr = Canon ? t.xr : buffer_rsrc(a.xq.heads, blocks * 4u);
    t.x_base = column_row(tid >> 3) * HtXStride<Canon>;
    t.h_base = column_row(tid & 31) * HtHStride<Canon>;
    t.nb = nb;
    float out[16];
    half_tree<Full, Canon, false>(st, t, wave, out, [](int, int, int, v16f, v16f) {});
    const int c = c0 + (lane & 31), row = R0 + 16 * (lane >> 5);
    if (!active || c >= a.N) return;
    float *yr = a.y + static_cast<size_t>(c) * a.M + row;
    if (row + 16 <= a.M && (a.M & 3) == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            reinterpret_cast<float4 *>(yr)[q] = make_float4(out[4 * q], out[4 * q + 1], out[4 * q + 2], out[4 * q + 3]);
        return;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v)
        if (row + v < a.M) yr[v] = out[v];
}

}  // namespace
}  // namespace moe
