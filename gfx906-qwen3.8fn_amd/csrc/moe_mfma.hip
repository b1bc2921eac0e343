// Int8-MFMA grouped expert projections for prefill-width groups (gfx950): the
// down projection, and gate / up of rows of more than 64 blocks (shorter rows:
// moe_half.hpp).
//
// Replaces the reference's MMQ path (src/hip/mmq.hip:139-381, mmq<Q4_0,J>) and
// the Session's MMVQ expert projections for wide groups
// (src/hip/linear.hip:156-490), with the same arithmetic contract:
//   per-block int32 dot  I = sum (qs&15)*c[i] + (qs>>4)*c[i+16]  src/quant.cpp:48-55
//   block value          d4 * (I*d8 - 8*s8)                       src/quant.cpp:88-93
//   SiLU(g)*u + Q8_1     src/hip/linear.hip:99-150, :509-525
//
// One v_mfma_i32_32x32x32_i8 is one Q4_0 block (K = 32) of a 32-row x
// 32-token tile, so its int32 results are exactly the reference's per-block
// dots.  The per-block scaling cannot be chained through the MFMA, so every
// result needs a vector epilogue; it is kept to two VALU instructions:
//   * the MFMA accumulates onto the constant 0x4B400000 (1.5 * 2^23), so the
//     result bits read as the float F = 12582912 + I exactly (|I| <= 61440);
//   * t = fma(F, d8, -12582912*d8) = round(I*d8)  (12582912*d8 is exact: d8 is
//     an fp16 value, 3*2^22 times it needs at most 13 significand bits);
//   * acc = fma(d4, t, acc) with d4 taken straight from its fp16 plane
//     (v_fma_mix_f32).
// The -8*d4*s8 terms form a [rows x blocks] x [blocks x tokens] product of
// fp16 values; one v_mfma_f32_32x32x16_f16 covers 16 blocks of it (fp16
// products are exact in fp32), and it seeds the accumulators.
//
// Work unit = (MFMA item of <= 128 grouped pairs of one expert, row slice),
// ordered item-major and dealt to the XCDs in chunks (see mfma_unit).
#include "moe_leaf.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace moe {
namespace {

constexpr int kMagic = 0x4B400000;         // bits of 12582912.0f
constexpr float kMagicF = 12582912.0f;


// The fp16 hi halves (s of a Q8_1 head) of 8 heads, zero for blocks >= nb.
__device__ __forceinline__ v8h head_sums(uint4 h0, uint4 h1, int kb0, int nb) {
    const uint32_t hv[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t lo = kb0 + 2 * e < nb ? hv[2 * e] >> 16 : 0u;
        const uint32_t hi = kb0 + 2 * e + 1 < nb ? hv[2 * e + 1] & 0xffff0000u : 0u;
        w[e] = lo | hi;
    }
    return pack8(w);
}

// As scale_block below, with the 16 row scales already in fp32.
__device__ __forceinline__ void scale_block_f32(float (&acc)[16], v16i r, uint32_t head, const float (&d4)[16]) {
    const v16f f = __builtin_bit_cast(v16f, r);
    const float d8 = cvt_half_lo(head);
    const float nk = -kMagicF * d8;
    // Eight independent products, then their eight accumulations: at two
    // waves per SIMD back-to-back dependent fmas issue at about 60 % of the
    // rate of independent ones (measured).
#pragma unroll
    for (int g = 0; g < 16; g += 8) {
        float t[8];
#pragma unroll
        for (int v = 0; v < 8; ++v) t[v] = fmaf(f[g + v], d8, nk);
#pragma unroll
        for (int v = 0; v < 8; ++v) acc[g + v] = fmaf(d4[g + v], t[v], acc[g + v]);
    }
}

// acc[v] += d4[v] * round(I[v] * d8) for one MFMA result (see the file comment).
__device__ __forceinline__ void scale_block(float (&acc)[16], v16i r, uint32_t head, const uint32_t (&d4)[8]) {
    const v16f f = __builtin_bit_cast(v16f, r);
    const float d8 = half_lo(head);
    const float nk = -kMagicF * d8;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const float t = fmaf(f[v], d8, nk);
        const float s = (v & 1) ? half_hi(d4[v >> 1]) : half_lo(d4[v >> 1]);
        acc[v] = fmaf(s, t, acc[v]);
    }
}

// a + the lo / hi fp16 half of h2.
__device__ __forceinline__ float add_half_lo(uint32_t h2, float a) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h2), "v"(a));
    return r;
}
__device__ __forceinline__ float add_half_hi(uint32_t h2, float a) {
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h2), "v"(a));
    return r;
}

// Q4_1 blocks {d4, m4, codes}: the reference's per-fragment value is
// fma(float(I_f), half(d4*d8), half(m4*s8) / 2) (src/cpu_expert.cpp:167-194),
// i.e. per block half(d4*d8) * I + half(m4*s8) with both products rounded to
// fp16.  Here, per block: acc = fma(I, dd, acc) + ms with the same two fp16
// roundings, two rows a packed multiply; only the fp32 summation order is
// this kernel's own.  Four VALU operations an element (subtract, half a
// multiply each for dd and ms, two mixed fmas) where separate products and
// conversions took nine: 2560/640 layer of 3,001 tokens
// 2113 -> 2056 us.
__device__ __forceinline__ void scale_block_q41(float (&acc)[16], v16i r, uint32_t head, const uint32_t (&d4)[8],
                                                const uint32_t (&m4)[8]) {
    const v16f f = __builtin_bit_cast(v16f, r);
    const uint32_t dp = __builtin_amdgcn_perm(head, head, 0x01000100u), sp = __builtin_amdgcn_perm(head, head, 0x03020302u);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t dd = pk_mul_half(d4[i], dp), ms = pk_mul_half(m4[i], sp);
        const float I0 = f[2 * i] - kMagicF, I1 = f[2 * i + 1] - kMagicF;   // exact: F = 12582912 + I
        acc[2 * i] = add_half_lo(ms, fma_mix_lo(dd, I0, acc[2 * i]));
        acc[2 * i + 1] = add_half_hi(ms, fma_mix_hi(dd, I1, acc[2 * i + 1]));
    }
}

// What one wave needs to project its 32 weight rows against up to kSubs
// token tiles.  Offsets are per lane; per-block steps are uniform.
struct TileArgs {
    __amdgpu_buffer_rsrc_t wr, sr, xr, hr;   // weight codes, weight scales, activation codes, activation heads
    __amdgpu_buffer_rsrc_t mr;               // Q4_1: weight mins (the scales' layout); unused for Q4_0
    uint32_t w_off;                          // lane's A row (block b at + 16 b)
    uint32_t s_off0, s_off1, s_step;         // lane's two 16-byte scale groups (block b at + b s_step)
    uint32_t x_off[kSubs], h_off[kSubs];     // lane's token rows (block b at + 32 b / + 4 b)
    const uint16_t *cscale;                  // lane's A-row scale of block kb at cscale[kb * cstride]
    int cstride;
    int nb;                                  // blocks per row (K / 32)
    int shift;                               // 0: low nibbles (lane half 0), 4: high nibbles
    int32_t *dots;                           // debug: per-block dots [pair][rows][nb] or null
    size_t dot_rows;                         // rows per pair in `dots`
    int dot_row0, dot_pair0, ncols, m, h;
};

// Debug-dot row of accumulator register v in lane half h.
template<bool Down>
__device__ __forceinline__ int acc_row(int v, int h) {
    return Down ? 4 * (v & 7) + 2 * h + (v >> 3) : 16 * h + v;
}

struct Loads {
    uint4 w, d0, d1, m0, m1;
    uint4 x[kSubs];
    uint32_t hd[kSubs];
};

template<int NS, bool Q41 = false>
__device__ __forceinline__ Loads tile_loads(const TileArgs &t, int b) {
    Loads l;
    const uint32_t ub = static_cast<uint32_t>(b);
    l.w = buffer_load16(t.wr, t.w_off, ub * 16u);
    l.d0 = buffer_load16(t.sr, t.s_off0, ub * t.s_step);
    l.d1 = buffer_load16(t.sr, t.s_off1, ub * t.s_step);
    if constexpr (Q41) {
        l.m0 = buffer_load16(t.mr, t.s_off0, ub * t.s_step);
        l.m1 = buffer_load16(t.mr, t.s_off1, ub * t.s_step);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        l.x[s] = buffer_load16(t.xr, t.x_off[s], ub * 32u);
        l.hd[s] = buffer_load4(t.hr, t.h_off[s], ub * 4u);
    }
    return l;
}

// acc[s] = -8 * sum_b d4 s8 + sum_b d4 round(I d8) for the NS token tiles
// (Q41: sum_b of scale_block_q41's terms from +0).
// The loads of block b + 1 are issued before block b is computed.
template<int NS, bool Dbg, bool Down, bool Q41 = false>
__device__ __forceinline__ void tile_project(const TileArgs &t, float (&acc)[kSubs][16]) {
    v16f corr[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) corr[s] = v16f{};
    for (int c = 0; c < (Q41 ? 0 : t.nb); c += 16) {
        const int kb0 = c + 8 * t.h;
        uint32_t dw[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k0 = kb0 + 2 * e, k1 = k0 + 1;
            const uint32_t lo = t.cscale[std::min(k0, t.nb - 1) * t.cstride];
            const uint32_t hi = t.cscale[std::min(k1, t.nb - 1) * t.cstride];
            dw[e] = (k0 < t.nb ? lo : 0u) | (k1 < t.nb ? hi << 16 : 0u);
        }
        const v8h da = pack8(dw);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const uint4 h0 = buffer_load16(t.hr, t.h_off[s] + 4u * kb0, 0);
            const uint4 h1 = buffer_load16(t.hr, t.h_off[s] + 4u * kb0, 16);
            corr[s] = __builtin_amdgcn_mfma_f32_32x32x16_f16(da, head_sums(h0, h1, kb0, t.nb), corr[s], 0, 0, 0);
        }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[s][v] = Q41 ? 0.0f : -8.0f * corr[s][v];

    v16i magic;
#pragma unroll
    for (int v = 0; v < 16; ++v) magic[v] = kMagic;
    Loads cur = tile_loads<NS, Q41>(t, 0);
#pragma unroll 1
    for (int b = 0; b < t.nb; ++b) {
        const Loads nxt = tile_loads<NS, Q41>(t, std::min(b + 1, t.nb - 1));
        const uint32_t d4[8] = {cur.d0.x, cur.d0.y, cur.d0.z, cur.d0.w, cur.d1.x, cur.d1.y, cur.d1.z, cur.d1.w};
        const uint32_t m4[8] = {cur.m0.x, cur.m0.y, cur.m0.z, cur.m0.w, cur.m1.x, cur.m1.y, cur.m1.z, cur.m1.w};
        const v4i A = {static_cast<int>((cur.w.x >> t.shift) & kNibbles), static_cast<int>((cur.w.y >> t.shift) & kNibbles),
                       static_cast<int>((cur.w.z >> t.shift) & kNibbles), static_cast<int>((cur.w.w >> t.shift) & kNibbles)};
        v16i r[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const v4i B = {static_cast<int>(cur.x[s].x), static_cast<int>(cur.x[s].y), static_cast<int>(cur.x[s].z),
                           static_cast<int>(cur.x[s].w)};
            r[s] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B, magic, 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if constexpr (Q41) scale_block_q41(acc[s], r[s], cur.hd[s], d4, m4);
            else scale_block(acc[s], r[s], cur.hd[s], d4);
            if constexpr (Dbg) {
                const int j = kSub * s + t.m;
                if (t.dots && j < t.ncols)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        t.dots[(static_cast<size_t>(t.dot_pair0 + j) * t.dot_rows + t.dot_row0 + acc_row<Down>(v, t.h)) *
                                   t.nb + b] = r[s][v] - kMagic;
            }
        }
        cur = nxt;
    }
}

template<bool Dbg, bool Down, bool Q41 = false>
__device__ __forceinline__ void tile_dispatch(const TileArgs &t, int nsub, float (&acc)[kSubs][16]) {
    switch (nsub) {
    case 1: tile_project<1, Dbg, Down, Q41>(t, acc); break;
    case 2: tile_project<2, Dbg, Down, Q41>(t, acc); break;
    case 3: tile_project<3, Dbg, Down, Q41>(t, acc); break;
    default: tile_project<4, Dbg, Down, Q41>(t, acc); break;
    }
}

// Workgroup = 2 waves: wave 0 gate rows R0..R0+31, wave 1 the same up rows,
// both for token tile `sub` (32 pairs) of an MFMA item.  A-row m of the MFMA
// is physical row 16*((m>>2)&1) + 4*(m>>3) + (m&3), so accumulator register v
// of lane half h is row 16h + v: the lane's 16 scales per block are two
// 16-byte groups of the [rows/8][blocks][8] plane, and its 16 middle values
// are elements 16h..16h+15 of one Q8_1 block.  Units are ordered
// (item, slice, sub) so the 4 tiles of an item that read the same weight rows
// are adjacent on one XCD.
// Rows of at most 64 blocks take k_gate_up_half (moe_half.hpp) instead; here
// Fold is kFoldGrouped96 (2048 < H <= 3072: the grouped leaves plus block
// kp + 64 in chain A; 2560/640 4K Zipf layer 3.40 -> 2.83 ms with Q4_0 downs,
// 3.54 -> 2.98 ms with Q4_1, against kFoldMulti; the fp16-operand form with a
// third block pair, two waves per SIMD at 63 KB of LDS, measured 3 % slower)
// or kFoldMulti (H > 3072); one instantiation per shape keeps only that
// path's registers.  The linear kernel (moe_leaf.hpp) also takes kFoldStaged
// (< 64 blocks) and kFoldGrouped (64).
template<int Fold, bool Dbg>
__global__ __launch_bounds__(128, 2) void k_gate_up_mfma(FfnArgs a) {
    // Pending tree levels 3-4 per wave; after the tree, the waves' results.
    __shared__ float park[2][2][16][64];
    __shared__ uint4 d4_lds[2][Fold == kFoldGrouped96 ? kGu96MaxBlocks : 1][4];   // [mat][block][32 halfs]
    const int mat = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int H = a.shape.H, I = a.shape.I, nb = H / 32, nbi = I / 32;
    const int slices = nbi * kSubs;
    const Unit un = row_chunk_unit(a.routes.item_counts[1], slices);
    if (!un.ok) return;   // uniform per workgroup
    const Item *itp = a.routes.mfma_items + un.item;
    const int expert = itp->expert, first = itp->first, ncols = itp->ncols;
    const int sub = un.slice % kSubs;
    const int R0 = (un.slice / kSubs) * 32;
    if (kSub * sub >= ncols) return;   // uniform per workgroup: no tokens in this tile
    const int lane = threadIdx.x & 63;
    const int m = lane & 31, h = lane >> 5;
    const int prow = 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
    const int j = kSub * sub + m;
    const int pair = first + std::min(j, ncols - 1);

    const size_t rbase = static_cast<size_t>(expert) * I + R0;
    const uint32_t row_bytes = static_cast<uint32_t>(nb) * 16u;
    GuTile t;
    t.wr = buffer_rsrc((mat ? a.bank.up_codes : a.bank.gate_codes) + rbase * row_bytes, 32u * row_bytes);
    t.sr = buffer_rsrc((mat ? a.bank.up_scales : a.bank.gate_scales) + rbase * nb, 32u * static_cast<uint32_t>(nb) * 2u);
    t.xr = buffer_rsrc(a.xq.codes, static_cast<uint32_t>(a.tokens) * static_cast<uint32_t>(nb) * 32u);
    t.hr = buffer_rsrc(a.xq.heads, static_cast<uint32_t>(a.tokens) * static_cast<uint32_t>(nb) * 4u);
    t.w_off = static_cast<uint32_t>(prow) * row_bytes;
    t.s_off0 = static_cast<uint32_t>(2 * h * nb) * 16u;
    t.s_off1 = t.s_off0 + static_cast<uint32_t>(nb) * 16u;
    const uint32_t tok = static_cast<uint32_t>(a.routes.pair_token[pair]);
    t.x_off = tok * static_cast<uint32_t>(nb) * 32u + 16u * h;
    t.h_off = tok * static_cast<uint32_t>(nb) * 4u;
    t.nb = nb;
    t.shift = 4 * h;
    t.dots = Dbg ? (mat ? a.up_dots : a.gate_dots) : nullptr;
    t.dot_base = (static_cast<size_t>(pair) * I + R0 + 16 * h) * nb;
    t.dot_ok = Dbg && t.dots && j < ncols;

    float res[16];
    // Node 0's weight half is issued before the scale staging, so the two
    // round trips overlap.
    const uint32_t w_off = static_cast<uint32_t>(prow) * row_bytes + 32u * 16u * h;
    uint4 wn[2] = {};
    if constexpr (Fold == kFoldGrouped96) {
        half_load_w(t, w_off, 0, wn);
        // Stage the tile's scales (both matrices).
        // Scale group g (rows 8g..8g+7) of block b is one 16-byte chunk of the
        // [rows/8][blocks][8] plane and lands at halfs 8g..8g+7 of [mat][b].
        for (int c = threadIdx.x; c < 8 * nb; c += blockDim.x) {
            const int mm = c / (4 * nb), rem = c % (4 * nb), gi = rem / nb, b = rem % nb;
            const uint16_t *plane = mm ? a.bank.up_scales : a.bank.gate_scales;
            d4_lds[mm][b][gi] = *reinterpret_cast<const uint4 *>(plane + (rbase + 8 * gi) * nb + b * 8);
        }
        __syncthreads();
        const GuStage g{reinterpret_cast<const uint32_t *>(&d4_lds[mat][0][0]), nullptr};
        fold_tree_grouped96<Dbg>(t, g, w_off, park[mat], lane, wn, res);
    } else {
        fold_tree_multi<Dbg>(t, park[mat], lane, res);
    }
    // Both waves' sums meet in LDS (each wave's own park area) and each wave
    // finishes 16 tokens (finish_gate_up).
#pragma unroll
    for (int v = 0; v < 16; ++v) park[mat][0][v][lane] = res[v];
    __syncthreads();
    finish_gate_up<Dbg>(a, park[0][0], park[1][0], mat, first, kSub * sub, ncols, R0);
}

// ------------------------------------------------------------------ down ---
// Workgroup = 4 waves x 32 output rows = 128 rows of H.  A-row m maps to
// physical row rho = 4*(v&7) + 2*hh + (v>>3) with v = 4*(m>>3) + (m&3) and
// hh = (m>>2)&1, so accumulator register v of lane half h is row
// 4*(v&7) + 2h + (v>>3), whose scale sits at slot 16h + v of the
// [rows/32][blocks][32] plane (slot (r%4)*8 + (r%32)/4): one 32-byte read per
// lane and block.  Before the stores, lanes l and l^32 trade 8 values so each
// lane holds 16 consecutive rows (4 float4 stores per tile).
//
// I <= 512 (16 blocks): the four waves read the same middle rows, so the
// item's middle codes and heads are staged once in LDS, and each wave stages
// its 32-row scale tile there.  Weight blocks stream through a window of
// kDnWin registers: block b's register is reloaded with block b + kDnWin as
// soon as block b's A operand is formed.  With Q4_0 rows and 8 or 16 blocks
// a workgroup runs kDnSlicesPerGroup slices of 128 rows against the
// one staging: the window runs on into the next slice's blocks, and the next
// slice's scale tile goes to the other half of a double buffer.
constexpr int kDnMaxBlocks = 16;
constexpr int kDnWin = 8;
constexpr int kDnSlicesPerGroup = 4;

template<int NB, int W = 4>
struct DownStageT {
    static constexpr bool kMins = false;
    uint4 x[kDnMaxBlocks][kMfmaTile][2];     // middle codes [block][pair][32 bytes]
    uint32_t hd[kDnMaxBlocks][kMfmaTile];    // middle heads [block][pair]
    uint4 d4[NB][W][kDnMaxBlocks][4];        // [buffer][wave]: scales [block][32 slots]
};
using DownStage = DownStageT<2>;             // Q4_0 rows: 80 KiB, two workgroups per CU
// Q4_1 rows also stage their mins (80 KiB: two workgroups per CU) and take
// one slice per workgroup (a second scale buffer would not fit twice).
template<int W = 4>
struct DownStageQ41T : DownStageT<1, W> {
    static constexpr bool kMins = true;
    uint4 m4[W][kDnMaxBlocks][4];            // per wave: mins [block][32 slots]
};
using DownStageQ41 = DownStageQ41T<4>;
// Rows of 17..32 Q4_0 blocks: a workgroup of 8 waves takes two 128-row
// slices against one staging of each round (80 KiB).
using DownStage2 = DownStageT<1, 8>;

// Slices of 128 rows per work unit of the down kernel.  Running on into the
// next slice keeps block j of every slice in window register j % kDnWin only
// when the block count is a multiple of kDnWin.
__host__ __device__ constexpr int down_span(int nbi, bool q41) {
    return nbi % kDnWin == 0 && nbi <= kDnMaxBlocks && !q41 ? kDnSlicesPerGroup : 1;
}
// Work units per item.
__host__ __device__ constexpr int down_groups(int H, int nbi, bool q41) {
    const int slices = (H + 127) / 128, span = down_span(nbi, q41);
    return (slices + span - 1) / span;
}

// d4s: the wave's staged scale tile ([block][4] chunks); m4s: its staged
// Q4_1 mins (same layout), or nullptr for Q4_0 rows.  wa: the weight window
// (block b in register b % kDnWin); block b + kDnWin is read through wr
// (this slice's 32 rows, and the next slice's 32 rows at next_off when there
// is a next slice: past its end the descriptor reads zeros), at lane offset
// w_off.
template<int NS, bool Dbg, bool Q41, class Stage>
__device__ __forceinline__ void down_staged(const FfnArgs &a, const Stage &st, const uint4 (*d4s)[4], const uint4 (*m4s)[4],
                                            uint4 (&wa)[kDnWin], __amdgpu_buffer_rsrc_t wr, uint32_t next_off,
                                            uint32_t w_off, int nbi, int first, int ncols, int R0, int pslot, int lane,
                                            float (&acc)[kSubs][16]) {
    const int m = lane & 31, h = lane >> 5, shift = 4 * h;
    const uint16_t *d4h = reinterpret_cast<const uint16_t *>(&d4s[0][0]);
    if constexpr (Q41) {
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[s][v] = 0.0f;
    } else {
    // Seed: -8 * sum_b d4 s8, 16 blocks in one f16 MFMA.
    uint32_t dw[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int k0 = 8 * h + 2 * e, k1 = k0 + 1;
        const uint32_t lo = k0 < nbi ? d4h[k0 * 32 + pslot] : 0u;
        const uint32_t hi = k1 < nbi ? d4h[k1 * 32 + pslot] : 0u;
        dw[e] = lo | (hi << 16);
    }
    const v8h da = pack8(dw);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        uint32_t sw[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k0 = 8 * h + 2 * e, k1 = k0 + 1;
            const uint32_t lo = k0 < nbi ? st.hd[k0][kSub * s + m] >> 16 : 0u;
            const uint32_t hi = k1 < nbi ? st.hd[k1][kSub * s + m] & 0xffff0000u : 0u;
            sw[e] = lo | hi;
        }
        const v16f corr = __builtin_amdgcn_mfma_f32_32x32x16_f16(da, pack8(sw), v16f{}, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[s][v] = -8.0f * corr[v];
    }
    }
    v16i magic;
#pragma unroll
    for (int v = 0; v < 16; ++v) magic[v] = kMagic;
    // Each step's B operand and head are read from LDS one step ahead (block
    // b + 1's first at block b's last step; past nbi they are never used).
    uint4 xb = st.x[0][m][h];
    uint32_t hx = st.hd[0][m];
#pragma unroll
    for (int b = 0; b < kDnMaxBlocks; ++b) {
        if (b < nbi) {   // uniform; a guard rather than a break keeps the loop unrolled
        const uint4 w = wa[b % kDnWin];
        const uint4 d0 = d4s[b][2 * h], d1 = d4s[b][2 * h + 1];
        const uint32_t d4[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
        uint32_t m4[8] = {};
        float d4f[16];
        if constexpr (Q41) {
            const uint4 n0 = m4s[b][2 * h], n1 = m4s[b][2 * h + 1];
            m4[0] = n0.x; m4[1] = n0.y; m4[2] = n0.z; m4[3] = n0.w;
            m4[4] = n1.x; m4[5] = n1.y; m4[6] = n1.z; m4[7] = n1.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                d4f[2 * e] = cvt_half_lo(d4[e]);
                d4f[2 * e + 1] = cvt_half_hi(d4[e]);
            }
        }
        const v4i A = {static_cast<int>((w.x >> shift) & kNibbles), static_cast<int>((w.y >> shift) & kNibbles),
                       static_cast<int>((w.z >> shift) & kNibbles), static_cast<int>((w.w >> shift) & kNibbles)};
        {
            // The offset goes into the per-lane operand, which the range check covers.
            const int nb = b + kDnWin;
            const uint32_t o = nb < nbi ? static_cast<uint32_t>(nb) * 16u : next_off + static_cast<uint32_t>(nb - nbi) * 16u;
            wa[b % kDnWin] = buffer_load16(wr, w_off + o, 0);
        }
        // Each tile's MFMA is issued before the previous tile is scaled, so
        // the matrix unit works under the scaling and two results are live.
        v16i rp;
        uint32_t hp = 0;
        auto scale_prev = [&](int sp) {
            if constexpr (Q41) scale_block_q41(acc[sp], rp, hp, d4, m4);
            else scale_block_f32(acc[sp], rp, hp, d4f);
            if constexpr (Dbg) {
                const int j = kSub * sp + m;
                if (a.down_dots && j < ncols)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        a.down_dots[(static_cast<size_t>(first + j) * a.shape.H + R0 + 4 * (v & 7) + 2 * h + (v >> 3)) * nbi + b] =
                            rp[v] - kMagic;
            }
        };
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const v4i B = {static_cast<int>(xb.x), static_cast<int>(xb.y), static_cast<int>(xb.z), static_cast<int>(xb.w)};
            const v16i r = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B, magic, 0, 0, 0);
            const uint32_t hs = hx;
            if (s + 1 < NS) {
                xb = st.x[b][kSub * (s + 1) + m][h];
                hx = st.hd[b][kSub * (s + 1) + m];
            } else if (b + 1 < kDnMaxBlocks) {
                xb = st.x[b + 1][m][h];
                hx = st.hd[b + 1][m];
            }
            if (s > 0) scale_prev(s - 1);
            __builtin_amdgcn_sched_barrier(0);
            rp = r;
            hp = hs;
        }
        scale_prev(NS - 1);
        }
    }
}

// down_staged for one of two staging rounds (down_two_rounds): blocks B0 ..
// B0 + 15 of the row sit at local indices 0..15.
template<int NS, bool Dbg, bool Q41, class Stage, int B0>
__device__ __forceinline__ void down_staged_round(const FfnArgs &a, const Stage &st, const uint4 (*d4s)[4], const uint4 (*m4s)[4],
                                            uint4 (&wa)[kDnWin], __amdgpu_buffer_rsrc_t wr, uint32_t next_off,
                                            uint32_t w_off, int nbi, int first, int ncols, int R0, int pslot, int lane,
                                            float (&acc)[kSubs][16]) {
    const int m = lane & 31, h = lane >> 5, shift = 4 * h;
    // Blocks B0 .. B0 + nloc - 1 are staged at local indices 0 .. nloc - 1
    // (the scales, mins, codes and heads); the weight window and the dots
    // use the block's own index.
    static_assert(B0 % kDnWin == 0, "block B0 + b sits in window register b % kDnWin");
    // (B0 == 0: every local index below kDnMaxBlocks is also below nbi, so
    // nbi itself bounds the first round.)
    const int nloc = B0 == 0 ? nbi : min(nbi - B0, kDnMaxBlocks);
    const uint16_t *d4h = reinterpret_cast<const uint16_t *>(&d4s[0][0]);
    if constexpr (Q41) {
        if constexpr (B0 == 0) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[s][v] = 0.0f;
        }
    } else {
    // Seed: -8 * sum_b d4 s8, 16 blocks in one f16 MFMA.
    uint32_t dw[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int k0 = 8 * h + 2 * e, k1 = k0 + 1;
        const uint32_t lo = k0 < nloc ? d4h[k0 * 32 + pslot] : 0u;
        const uint32_t hi = k1 < nloc ? d4h[k1 * 32 + pslot] : 0u;
        dw[e] = lo | (hi << 16);
    }
    const v8h da = pack8(dw);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        uint32_t sw[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int k0 = 8 * h + 2 * e, k1 = k0 + 1;
            const uint32_t lo = k0 < nloc ? st.hd[k0][kSub * s + m] >> 16 : 0u;
            const uint32_t hi = k1 < nloc ? st.hd[k1][kSub * s + m] & 0xffff0000u : 0u;
            sw[e] = lo | hi;
        }
        const v16f corr = __builtin_amdgcn_mfma_f32_32x32x16_f16(da, pack8(sw), v16f{}, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            if constexpr (B0 == 0) acc[s][v] = -8.0f * corr[v];
            else acc[s][v] = acc[s][v] + -8.0f * corr[v];
        }
    }
    }
    v16i magic;
#pragma unroll
    for (int v = 0; v < 16; ++v) magic[v] = kMagic;
    // Each step's B operand and head are read from LDS one step ahead (block
    // b + 1's first at block b's last step; past nbi they are never used).
    uint4 xb = st.x[0][m][h];
    uint32_t hx = st.hd[0][m];
#pragma unroll
    for (int b = 0; b < kDnMaxBlocks; ++b) {
        if (b < nloc) {   // uniform; a guard rather than a break keeps the loop unrolled
        const uint4 w = wa[b % kDnWin];
        const uint4 d0 = d4s[b][2 * h], d1 = d4s[b][2 * h + 1];
        const uint32_t d4[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
        uint32_t m4[8] = {};
        float d4f[16];
        if constexpr (Q41) {
            const uint4 n0 = m4s[b][2 * h], n1 = m4s[b][2 * h + 1];
            m4[0] = n0.x; m4[1] = n0.y; m4[2] = n0.z; m4[3] = n0.w;
            m4[4] = n1.x; m4[5] = n1.y; m4[6] = n1.z; m4[7] = n1.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                d4f[2 * e] = cvt_half_lo(d4[e]);
                d4f[2 * e + 1] = cvt_half_hi(d4[e]);
            }
        }
        const v4i A = {static_cast<int>((w.x >> shift) & kNibbles), static_cast<int>((w.y >> shift) & kNibbles),
                       static_cast<int>((w.z >> shift) & kNibbles), static_cast<int>((w.w >> shift) & kNibbles)};
        {
            // The offset goes into the per-lane operand, which the range check covers.
            const int nb = B0 + b + kDnWin;
            const uint32_t o = nb < nbi ? static_cast<uint32_t>(nb) * 16u : next_off + static_cast<uint32_t>(nb - nbi) * 16u;
            wa[b % kDnWin] = buffer_load16(wr, w_off + o, 0);
        }
        // Each tile's MFMA is issued before the previous tile is scaled, so
        // the matrix unit works under the scaling and two results are live.
        v16i rp;
        uint32_t hp = 0;
        auto scale_prev = [&](int sp) {
            if constexpr (Q41) scale_block_q41(acc[sp], rp, hp, d4, m4);
            else scale_block_f32(acc[sp], rp, hp, d4f);
            if constexpr (Dbg) {
                const int j = kSub * sp + m;
                if (a.down_dots && j < ncols)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        a.down_dots[(static_cast<size_t>(first + j) * a.shape.H + R0 + 4 * (v & 7) + 2 * h + (v >> 3)) * nbi + B0 + b] =
                            rp[v] - kMagic;
            }
        };
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const v4i B = {static_cast<int>(xb.x), static_cast<int>(xb.y), static_cast<int>(xb.z), static_cast<int>(xb.w)};
            const v16i r = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B, magic, 0, 0, 0);
            const uint32_t hs = hx;
            if (s + 1 < NS) {
                xb = st.x[b][kSub * (s + 1) + m][h];
                hx = st.hd[b][kSub * (s + 1) + m];
            } else if (b + 1 < kDnMaxBlocks) {
                xb = st.x[b + 1][m][h];
                hx = st.hd[b + 1][m];
            }
            if (s > 0) scale_prev(s - 1);
            __builtin_amdgcn_sched_barrier(0);
            rp = r;
            hp = hs;
        }
        scale_prev(NS - 1);
        }
    }
}

// Writes a wave's 32-row x (32 x nsub)-pair result tile to the pairs'
// contribution rows.  Lane half h holds rows 4q + 2h (v = q) and
// 4q + 2h + 1 (v = 8 + q), q = 0..7; after the trade lane half h holds rows
// 16h .. 16h + 15 (4 float4 stores per tile).
__device__ __forceinline__ void store_down_tile(const FfnArgs &a, const float (&acc)[kSubs][16], int nsub, int first,
                                                int ncols, int R0) {
    const int lane = threadIdx.x & 63, m = lane & 31, h = lane >> 5;
#pragma unroll
    for (int s = 0; s < kSubs; ++s) {
        if (s >= nsub) break;
        const int j = kSub * s + m;
        const bool valid = j < ncols;
        const int p = first + std::min(j, ncols - 1);
        const size_t orow = static_cast<size_t>(a.routes.pair_token[p]) * a.out_stride_k + a.routes.pair_rank[p];
        float *dst = a.out + orow * a.shape.H + R0 + 16 * h;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // v_permlane32_swap(a, b): lanes < 32 get (own a, a of lane + 32),
            // lanes >= 32 (b of lane - 32, own b) -- for both halves the
            // float4's x and z; the same for y and w.
            const auto xz = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[s][q]),
                                                             __float_as_uint(acc[s][4 + q]), false, false);
            const auto yw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[s][8 + q]),
                                                             __float_as_uint(acc[s][12 + q]), false, false);
            const float4 o = make_float4(__uint_as_float(xz[0]), __uint_as_float(yw[0]), __uint_as_float(xz[1]),
                                         __uint_as_float(yw[1]));
            if (valid) *reinterpret_cast<float4 *>(dst + 4 * q) = o;
        }
    }
}

// The staged path's slices s0 .. s1-1 for one wave, after the staging
// barrier.  wa holds slice s0's first kDnWin weight blocks; buffer 0 of
// st.d4 its scales.
template<int NS, bool Dbg, bool Q41, class Stage>
__device__ __forceinline__ void down_slices(const FfnArgs &a, Stage &st, int wave, uint4 (&wa)[kDnWin], int nbi,
                                            int expert, int first, int ncols, int s0, int s1, uint32_t w_off, int pslot) {
    const int lane = threadIdx.x & 63, H = a.shape.H;
    const uint32_t row_bytes = static_cast<uint32_t>(nbi) * 16u;
    for (int sl = s0; sl < s1; ++sl) {
        const int R0 = sl * 128 + wave * 32;
        if (R0 >= H) break;                     // wave-uniform; later slices lie further down
        // Opaque zeros added to the lane index, the weight offset and the
        // block count keep the per-lane LDS and weight addresses (about 80
        // VGPRs) and the window's block offsets (16 SGPRs) from being
        // hoisted out of the loop into registers.
        int zero, szero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        asm volatile("s_mov_b32 %0, 0" : "=s"(szero));
        const int buf = Q41 ? 0 : (sl - s0) & 1;
        const int Rn = R0 + 128;
        const bool pf = sl + 1 < s1 && Rn < H;
        // Loads are unconditional: past the last slice the descriptors are
        // empty and read zeros.
        const size_t rc = static_cast<size_t>(expert) * H + R0, rn = static_cast<size_t>(expert) * H + (pf ? Rn : R0);
        // Rows R0 .. R0 + 31, and R0 + 128 .. R0 + 159 when there is a next slice.
        const auto wr = buffer_rsrc(a.bank.down_codes + rc * row_bytes, (pf ? 160u : 32u) * row_bytes);
        // The next slice's scale tile: nbi * 4 chunks of 16 bytes, one per lane.
        uint4 dn = make_uint4(0, 0, 0, 0);
        if constexpr (!Q41)
            dn = buffer_load16(buffer_rsrc(a.bank.down_scales + rn * nbi, pf ? static_cast<uint32_t>(nbi) * 64u : 0u),
                               16u * static_cast<uint32_t>(lane), 0);
        float acc[kSubs][16];
        const uint4 (*m4s)[4] = nullptr;
        if constexpr (Q41) m4s = st.m4[wave];
        down_staged<NS, Dbg, Q41>(a, st, st.d4[buf][wave], m4s, wa, wr, 128u * row_bytes, w_off + static_cast<uint32_t>(zero), nbi + szero,
                                  first, ncols, R0, pslot, lane + zero, acc);
        if constexpr (!Q41) {
            // The other buffer was last read by slice sl - 1 of this wave.
            if (lane < nbi * 4) st.d4[buf ^ 1][wave][lane >> 2][lane & 3] = dn;
            __builtin_amdgcn_wave_barrier();
        }
        store_down_tile(a, acc, NS, first, ncols, R0);
    }
}

// Stages blocks B0 .. B0 + 15 (those below nbi) of an item's middle codes
// and heads, and of each active wave's 32-row scale (and min) tile, at local
// block indices 0..15.  Thread t keeps one (block, half) of the code rows,
// local block (t % 32) / 2 and half t % 2, for pairs t / 32 + 8 i, and one
// block of the heads, t % 16, for pairs t / 16 + 16 i.  The descriptors end
// at the item's last pair: pairs past ncols read zero.  All loads are issued
// before the first LDS write.
template<int T>
struct DownStager {
    __amdgpu_buffer_rsrc_t xr, hr;
    const uint4 *scales, *mins;   // the wave's [nbi][4] chunks
    uint32_t pair_bytes;
    int cols, nbi, xb, xh, xj, hb, hj;

    __device__ static DownStager make(const FfnArgs &a, int first, int ncols, int nsub, int nbi, size_t rbase) {
        static_assert(kMfmaTile == 128 && kDnMaxBlocks == 16 && (T == 256 || T == 512),
                      "staging map: 256 or 512 threads, 128 pairs, 16 blocks");
        DownStager g;
        g.pair_bytes = static_cast<uint32_t>(nbi) * 32u;
        g.xr = buffer_rsrc(a.mq.codes + static_cast<size_t>(first) * g.pair_bytes, static_cast<uint32_t>(ncols) * g.pair_bytes);
        g.hr = buffer_rsrc(a.mq.heads + static_cast<size_t>(first) * nbi, static_cast<uint32_t>(ncols * nbi) * 4u);
        g.scales = reinterpret_cast<const uint4 *>(a.bank.down_scales + rbase * nbi);
        g.mins = a.bank.down_mins ? reinterpret_cast<const uint4 *>(a.bank.down_mins + rbase * nbi) : nullptr;
        g.cols = nsub * kSub;
        g.nbi = nbi;
        const int tid = static_cast<int>(threadIdx.x);
        g.xb = (tid & 31) >> 1;
        g.xh = tid & 1;
        g.xj = tid >> 5;
        g.hb = tid & 15;
        g.hj = tid >> 4;
        return g;
    }

    template<class Stage>
    __device__ void run(Stage &st, int B0, int wave, int lane, bool active) const {
        const int bx = B0 + xb, bh = B0 + hb;
        const uint32_t x_off = static_cast<uint32_t>(xj) * pair_bytes + static_cast<uint32_t>(32 * bx + 16 * xh);
        const uint32_t h_off = static_cast<uint32_t>(hj * nbi + bh) * 4u;
        // Thread t keeps (block, half) ((t % 32) / 2, t % 2) of pairs t / 32 + PX i
        // and the head of block t % 16 of pairs t / 16 + PH i.
        constexpr int PX = T / 32, PH = T / 16;
        uint4 xv[kMfmaTile / PX];
        uint32_t hv[kMfmaTile / PH];
#pragma unroll
        for (int i = 0; i < kMfmaTile / PX; ++i)
            if (PX * i < cols && bx < nbi) xv[i] = buffer_load16(xr, x_off, static_cast<uint32_t>(PX * i) * pair_bytes);
#pragma unroll
        for (int i = 0; i < kMfmaTile / PH; ++i)
            if (PH * i < cols && bh < nbi) hv[i] = buffer_load4(hr, h_off, static_cast<uint32_t>(PH * i * nbi) * 4u);
#pragma unroll
        for (int i = 0; i < kMfmaTile / PX; ++i)
            if (PX * i < cols && bx < nbi) st.x[xb][xj + PX * i][xh] = xv[i];
#pragma unroll
        for (int i = 0; i < kMfmaTile / PH; ++i)
            if (PH * i < cols && bh < nbi) st.hd[hb][hj + PH * i] = hv[i];
        const int nl = min(nbi - B0, kDnMaxBlocks);
        if (active)
            for (int c = lane; c < nl * 4; c += 64) st.d4[0][wave][c >> 2][c & 3] = scales[B0 * 4 + c];
        if constexpr (Stage::kMins) {
            if (active)
                for (int c = lane; c < nl * 4; c += 64) st.m4[wave][c >> 2][c & 3] = mins[B0 * 4 + c];
        }
    }
};

// Rows of 17..32 down blocks (I = 544..1024; the reference model's 640: 20):
// one 128-row slice per workgroup, its blocks staged in two rounds into the
// same LDS (0..15, then 16..nbi - 1) with the accumulators carried across.
// The weight window already holds blocks 16..23 when the second round
// starts.  Every wave reaches both barriers.
template<int NS, bool Dbg, bool Q41, class Stage, class Stager>
__device__ __forceinline__ void down_two_rounds(const FfnArgs &a, Stage &st, const Stager &sg, int wave, bool active,
                                                uint4 (&wa)[kDnWin], int nbi, int first, int ncols, int R0, size_t rbase,
                                                uint32_t w_off, int pslot) {
    const int lane = threadIdx.x & 63;
    const uint32_t row_bytes = static_cast<uint32_t>(nbi) * 16u;
    // This slice's 32 rows; past them (no next slice) the descriptor reads zeros.
    const auto wr = buffer_rsrc(a.bank.down_codes + rbase * row_bytes, 32u * row_bytes);
    const uint4 (*m4s)[4] = nullptr;
    if constexpr (Q41) m4s = st.m4[wave];
    float acc[kSubs][16];
    if (active)
        down_staged_round<NS, Dbg, Q41, Stage, 0>(a, st, st.d4[0][wave], m4s, wa, wr, 32u * row_bytes, w_off, nbi, first, ncols,
                                            R0, pslot, lane, acc);
    __syncthreads();   // every wave is done with blocks 0..15
    sg.run(st, kDnMaxBlocks, wave, lane, active);
    __syncthreads();
    if (!active) return;
    down_staged_round<NS, Dbg, Q41, Stage, kDnMaxBlocks>(a, st, st.d4[0][wave], m4s, wa, wr, 32u * row_bytes, w_off, nbi, first,
                                                   ncols, R0, pslot, lane, acc);
    store_down_tile(a, acc, NS, first, ncols, R0);
}

// R2: rows of 17..32 blocks, staged in two rounds (down_two_rounds); a
// separate instantiation, so the other shapes' kernel keeps its registers.
template<bool Dbg, bool Q41, bool R2 = false>
__global__ __launch_bounds__(256, 2) void k_down_mfma(FfnArgs a) {
    __shared__ std::conditional_t<Q41, DownStageQ41, DownStage> st;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int H = a.shape.H, nbi = a.shape.I / 32;
    const int slices = (H + 127) / 128;
    const bool staged = R2 || nbi <= kDnMaxBlocks;
    const int span = down_span(nbi, Q41);
    const Unit un = mfma_unit(a.routes.item_counts[1], down_groups(H, nbi, Q41));
    if (!un.ok) return;
    const Item *itp = a.routes.mfma_items + un.item;
    const int expert = itp->expert, first = itp->first, ncols = itp->ncols;
    const int s0 = un.slice * span, s1 = std::min(slices, s0 + span);
    const int R0 = s0 * 128 + wave * 32;
    const bool active = R0 < H;      // wave-uniform
    const int nsub = (ncols + kSub - 1) / kSub;
    const int m = lane & 31, h = lane >> 5;
    const int mv = 4 * (m >> 3) + (m & 3);
    const int prow = 4 * (mv & 7) + 2 * ((m >> 2) & 1) + (mv >> 3);
    const int pslot = (prow & 3) * 8 + (prow >> 2);

    const size_t rbase = static_cast<size_t>(expert) * H + (active ? R0 : 0);
    const uint32_t row_bytes = static_cast<uint32_t>(nbi) * 16u;
    const uint16_t *scales = a.bank.down_scales + rbase * nbi;        // [nbi][32] halfs of this 32-row group
    if (staged) {
        // The first weight blocks first (their HBM latency overlaps the staging).
        const auto wr = buffer_rsrc(a.bank.down_codes + rbase * row_bytes, 32u * row_bytes);
        const uint32_t w_off = static_cast<uint32_t>(prow) * row_bytes;
        uint4 wa[kDnWin];
#pragma unroll
        for (int b = 0; b < kDnWin; ++b) wa[b] = buffer_load16(wr, w_off, static_cast<uint32_t>(b < nbi ? b : 0) * 16u);
        if constexpr (R2) {
            // Middle codes and heads of the item's pairs, every load issued
            // before the first LDS write (DownStager).
            const DownStager<256> sg = DownStager<256>::make(a, first, ncols, nsub, nbi, rbase);
            sg.run(st, 0, wave, lane, active);
            __syncthreads();
            switch (nsub) {   // two staging rounds; every wave takes part in their barriers
            case 1: down_two_rounds<1, Dbg, Q41>(a, st, sg, wave, active, wa, nbi, first, ncols, R0, rbase, w_off, pslot); break;
            case 2: down_two_rounds<2, Dbg, Q41>(a, st, sg, wave, active, wa, nbi, first, ncols, R0, rbase, w_off, pslot); break;
            case 3: down_two_rounds<3, Dbg, Q41>(a, st, sg, wave, active, wa, nbi, first, ncols, R0, rbase, w_off, pslot); break;
            default: down_two_rounds<4, Dbg, Q41>(a, st, sg, wave, active, wa, nbi, first, ncols, R0, rbase, w_off, pslot); break;
            }
            return;
        }
        // Middle codes and heads of the item's pairs, every load issued
        // before the first LDS write.  Thread t keeps one (block, half) of the
        // code rows, block (t % 32) / 2 and half t % 2, for pairs t / 32 + 8 i,
        // and one block of the heads, t % 16, for pairs t / 16 + 16 i.  The
        // descriptors end at the item's last pair: pairs past ncols read zero.
        static_assert(kMfmaTile == 128 && kDnMaxBlocks == 16, "staging map: 256 threads, 128 pairs, 16 blocks");
        const int cols = nsub * kSub;
        const uint32_t pair_bytes = static_cast<uint32_t>(nbi) * 32u;
        const auto xr = buffer_rsrc(a.mq.codes + static_cast<size_t>(first) * pair_bytes,
                                    static_cast<uint32_t>(ncols) * pair_bytes);
        const auto hr = buffer_rsrc(a.mq.heads + static_cast<size_t>(first) * nbi,
                                    static_cast<uint32_t>(ncols * nbi) * 4u);
        const int tid = static_cast<int>(threadIdx.x);
        const int xb = (tid & 31) >> 1, xh = tid & 1, xj = tid >> 5, hb = tid & 15, hj = tid >> 4;
        const uint32_t x_off = static_cast<uint32_t>(xj) * pair_bytes + static_cast<uint32_t>(32 * xb + 16 * xh);
        const uint32_t h_off = static_cast<uint32_t>(hj * nbi + hb) * 4u;
        uint4 xv[kMfmaTile / 8];
        uint32_t hv[kMfmaTile / 16];
#pragma unroll
        for (int i = 0; i < kMfmaTile / 8; ++i)
            if (8 * i < cols && xb < nbi) xv[i] = buffer_load16(xr, x_off, 8u * i * pair_bytes);
#pragma unroll
        for (int i = 0; i < kMfmaTile / 16; ++i)
            if (16 * i < cols && hb < nbi) hv[i] = buffer_load4(hr, h_off, 64u * i * static_cast<uint32_t>(nbi));
#pragma unroll
        for (int i = 0; i < kMfmaTile / 8; ++i)
            if (8 * i < cols && xb < nbi) st.x[xb][xj + 8 * i][xh] = xv[i];
#pragma unroll
        for (int i = 0; i < kMfmaTile / 16; ++i)
            if (16 * i < cols && hb < nbi) st.hd[hb][hj + 16 * i] = hv[i];
        if (active)
            for (int c = lane; c < nbi * 4; c += 64)
                st.d4[0][wave][c >> 2][c & 3] = reinterpret_cast<const uint4 *>(scales)[c];
        if constexpr (Q41) {
            const uint16_t *mins = a.bank.down_mins + rbase * nbi;   // same layout as the scales
            if (active)
                for (int c = lane; c < nbi * 4; c += 64)
                    st.m4[wave][c >> 2][c & 3] = reinterpret_cast<const uint4 *>(mins)[c];
        }
        __syncthreads();
        if (!active) return;
        switch (nsub) {
        case 1: down_slices<1, Dbg, Q41>(a, st, wave, wa, nbi, expert, first, ncols, s0, s1, w_off, pslot); break;
        case 2: down_slices<2, Dbg, Q41>(a, st, wave, wa, nbi, expert, first, ncols, s0, s1, w_off, pslot); break;
        case 3: down_slices<3, Dbg, Q41>(a, st, wave, wa, nbi, expert, first, ncols, s0, s1, w_off, pslot); break;
        default: down_slices<4, Dbg, Q41>(a, st, wave, wa, nbi, expert, first, ncols, s0, s1, w_off, pslot); break;
        }
        return;
    }
    if (!active) return;   // no barrier on this path
    float acc[kSubs][16];
    const uint32_t pairs = static_cast<uint32_t>(a.pairs_bound);
    TileArgs t;
    t.wr = buffer_rsrc(a.bank.down_codes + rbase * row_bytes, 32u * row_bytes);
    t.sr = buffer_rsrc(scales, static_cast<uint32_t>(nbi) * 64u);
    t.mr = buffer_rsrc(Q41 ? a.bank.down_mins + rbase * nbi : scales, static_cast<uint32_t>(nbi) * 64u);
    t.xr = buffer_rsrc(a.mq.codes, pairs * static_cast<uint32_t>(nbi) * 32u);
    t.hr = buffer_rsrc(a.mq.heads, pairs * static_cast<uint32_t>(nbi) * 4u);
    t.w_off = static_cast<uint32_t>(prow) * row_bytes;
    t.s_off0 = 32u * h;
    t.s_off1 = 32u * h + 16u;
    t.s_step = 64u;
#pragma unroll
    for (int s = 0; s < kSubs; ++s) {
        const uint32_t p = static_cast<uint32_t>(first + std::min(kSub * s + m, ncols - 1));
        t.x_off[s] = p * static_cast<uint32_t>(nbi) * 32u + 16u * h;
        t.h_off[s] = p * static_cast<uint32_t>(nbi) * 4u;
    }
    t.cscale = scales + pslot;
    t.cstride = 32;
    t.nb = nbi;
    t.shift = 4 * h;
    t.dots = Dbg ? a.down_dots : nullptr;
    t.dot_rows = static_cast<size_t>(H);
    t.dot_row0 = R0;
    t.dot_pair0 = first;
    t.ncols = ncols;
    t.m = m;
    t.h = h;
    tile_dispatch<Dbg, true, Q41>(t, nsub, acc);
    store_down_tile(a, acc, nsub, first, ncols, R0);
}

// Q4_0 rows of 17..32 down blocks without debug outputs: a workgroup of 8
// waves takes slices 2u (waves 0-3) and 2u + 1 (waves 4-7) of an item, so
// each staging round (down_two_rounds) serves 256 rows instead of 128.  The
// CU holds one such workgroup (8 waves at 236 VGPRs: two per SIMD, as two
// 4-wave workgroups would).
__global__ __launch_bounds__(512, 1) void k_down_mfma_pair(FfnArgs a) {
    constexpr bool Q41 = false;
    __shared__ DownStage2 st;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int H = a.shape.H, nbi = a.shape.I / 32;
    const int slices = (H + 127) / 128;
    const Unit un = mfma_unit(a.routes.item_counts[1], (slices + 1) / 2);
    if (!un.ok) return;   // uniform per workgroup
    const Item *itp = a.routes.mfma_items + un.item;
    const int expert = itp->expert, first = itp->first, ncols = itp->ncols;
    const int R0 = (2 * un.slice + (wave >> 2)) * 128 + (wave & 3) * 32;
    const bool active = R0 < H;      // wave-uniform
    const int nsub = (ncols + kSub - 1) / kSub;
    const int m = lane & 31;
    const int mv = 4 * (m >> 3) + (m & 3);
    const int prow = 4 * (mv & 7) + 2 * ((m >> 2) & 1) + (mv >> 3);
    const int pslot = (prow & 3) * 8 + (prow >> 2);
    const size_t rbase = static_cast<size_t>(expert) * H + (active ? R0 : 0);
    const uint32_t row_bytes = static_cast<uint32_t>(nbi) * 16u;
    // The first weight blocks first (their HBM latency overlaps the staging).
    const auto wr = buffer_rsrc(a.bank.down_codes + rbase * row_bytes, 32u * row_bytes);
    const uint32_t w_off = static_cast<uint32_t>(prow) * row_bytes;
    uint4 wa[kDnWin];
#pragma unroll
    for (int b = 0; b < kDnWin; ++b) wa[b] = buffer_load16(wr, w_off, static_cast<uint32_t>(b) * 16u);
    const DownStager<512> sg = DownStager<512>::make(a, first, ncols, nsub, nbi, rbase);
    sg.run(st, 0, wave, lane, active);
    __syncthreads();
    switch (nsub) {   // two staging rounds; every wave takes part in their barriers
    case 1: down_two_rounds<1, false, Q41>(a, st, sg, wave, active, wa, nbi, first, ncols, R0, rbase, w_off, pslot); break;
    case 2: down_two_rounds<2, false, Q41>(a, st, sg, wave, active, wa, nbi, first, ncols, R0, rbase, w_off, pslot); break;
    case 3: down_two_rounds<3, false, Q41>(a, st, sg, wave, active, wa, nbi, first, ncols, R0, rbase, w_off, pslot); break;
    default: down_two_rounds<4, false, Q41>(a, st, sg, wave, active, wa, nbi, first, ncols, R0, rbase, w_off, pslot); break;
    }
}

unsigned mfma_grid(const FfnArgs &a, int slices) {
    const size_t units = mfma_item_bound(a) * static_cast<size_t>(slices);
    const size_t round = 8 * static_cast<size_t>(kUnitChunk);
    return static_cast<unsigned>((units + round - 1) / round * round);
}

}  // namespace

hipError_t launch_linear_mfma(const LinearMfmaArgs &a, hipStream_t s) {
    const bool w8 = a.waves == 8;
    if (a.q8) {
        if (w8) launch_linear_mfma_t<true, 8, false>(a, s);
        else launch_linear_mfma_t<true, 4, false>(a, s);
    } else {
        if (w8) launch_linear_mfma_t<false, 8, false>(a, s);
        else launch_linear_mfma_t<false, 4, false>(a, s);
    }
    return hipGetLastError();
}

hipError_t launch_gate_up_mfma(const FfnArgs &a, hipStream_t s) {
    const bool dbg = a.middle_f32 || a.gate_dots || a.up_dots;
    const int nb = a.shape.H / 32;
    if (nb <= kHalfMaxBlocks) return launch_gate_up_half(a, s);
    const unsigned grid = chunk_grid(a, a.shape.I / 32 * kSubs);
    if (nb <= kGu96MaxBlocks) {
        if (dbg) k_gate_up_mfma<kFoldGrouped96, true><<<grid, 128, 0, s>>>(a);
        else k_gate_up_mfma<kFoldGrouped96, false><<<grid, 128, 0, s>>>(a);
    } else if (dbg) k_gate_up_mfma<kFoldMulti, true><<<grid, 128, 0, s>>>(a);
    else k_gate_up_mfma<kFoldMulti, false><<<grid, 128, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_down_mfma(const FfnArgs &a, hipStream_t s) {
    const bool q41 = a.bank.down_mins != nullptr;
    const unsigned grid = mfma_grid(a, down_groups(a.shape.H, a.shape.I / 32, q41));
    // Rows of 17..32 blocks take two staging rounds; the debug build (per-block
    // dots) keeps them on the tile path, whose register use it can afford.
    const int nbi = a.shape.I / 32;
    const bool r2 = nbi > kDnMaxBlocks && nbi <= 2 * kDnMaxBlocks;
    if (a.down_dots) {
        if (q41) k_down_mfma<true, true><<<grid, 256, 0, s>>>(a);
        else k_down_mfma<true, false><<<grid, 256, 0, s>>>(a);
    } else if (r2 && !q41) {
        // Two slices per 8-wave workgroup (2560/640 4K Zipf(1.1) layer with
        // Q4_0 downs 2.70-2.71 -> 2.46 ms); with Q4_1 rows (254 VGPRs, 88 KB
        // of LDS) it ran 2.71 -> 2.75 ms, so those keep one slice per workgroup.
        const unsigned pgrid = mfma_grid(a, ((a.shape.H + 127) / 128 + 1) / 2);   // k_down_mfma_pair's units per item
        k_down_mfma_pair<<<pgrid, 512, 0, s>>>(a);
    } else if (r2) {
        k_down_mfma<false, true, true><<<grid, 256, 0, s>>>(a);
    } else if (q41) k_down_mfma<false, true><<<grid, 256, 0, s>>>(a);
    else k_down_mfma<false, false><<<grid, 256, 0, s>>>(a);
    return hipGetLastError();
}

}  // namespace moe
