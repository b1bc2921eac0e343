// Exact-order leaves of the reference's pairwise tree on int8 MFMA, and the
// linear kernel built from them.  moe_mfma.hip uses them for gate / up rows of
// more than 64 blocks and for Q4_0 linears, moe_linear_q41.hip for Q4_1 ones.
#pragma once

#include "moe_mfma_device.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace moe {
namespace {

// ------------------------------------------------------------- gate / up ---
// The gate and up projections feed SiLU and the middle Q8, and one middle
// code that rounds differently moves its token's output by ~1e-2 rms, so they
// reproduce the reference's fp32 arithmetic exactly (cpu_expert's
// matrix_gpu_order, src/cpu_expert.cpp:156-213, the order of the gfx906
// MMVQ kernel src/hip/linear.hip:156-281):
//   fragment f of block k: bytes 8f..8f+7 of the code chunk, i.e. elements
//     8f..8f+7 (low nibbles) and 16+8f..16+8f+7 (high nibbles);
//   lane L = 2*(k%64) + f:  acc[L] = fma(d4, fma(float(I_f), d8, -4*s8), acc[L])
//     over k = L/2, L/2 + 64, ... in increasing k;
//   u_f(k') = acc[2k'+f] + acc[2(k'+32)+f],  v(k') = u_0(k') + u_1(k')  (k' < 32);
//   result = pairwise tree of v(0..31) in index order (XOR butterfly 1..32).
// Every add and fma is the same IEEE fp32 operation, so the gate and up
// values are bit-identical to the reference's, and with moe_expf so is the
// middle.  Fragment dots come from two MFMAs per block whose A operands keep
// only that fragment's bytes (the other half zero); both MFMAs start from 0.

// A block's scales against one token, for the 16 rows of a lane half.
//   Q4_0: the lane value is fma(d4, fma(float(I_f), d8, -4 s8), acc).
//   Q4_1: acc + fma(float(I_f), half(d4 d8), half(m4 s8) / 2): both products
//     rounded to fp16 by packed multiplies, once per block for its two
//     fragments.  The nibbles are taken doubled (nibbles<true>), so the MFMA
//     gives 2 I and fma(2 I, dd, ms) is twice the reference's value, exactly;
//     the tree's sum is halved at the end.
template<bool Q41> struct BlkScale {
    float d8, c4;
    uint32_t d4[8];
};
template<> struct BlkScale<true> {
    uint32_t dd[8], ms[8];   // fp16 pairs: rows 2i, 2i + 1
};

__device__ __forceinline__ uint32_t pk_mul_half(uint32_t a, uint32_t b) {
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, a) * __builtin_bit_cast(v2h, b));
}

template<bool Q41>
__device__ __forceinline__ BlkScale<Q41> blk_scale(uint32_t head, uint4 d0, uint4 d1, uint4 m0, uint4 m1) {
    BlkScale<Q41> s;
    const uint32_t d[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
    if constexpr (Q41) {
        const uint32_t m[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
        const uint32_t dp = __builtin_amdgcn_perm(head, head, 0x01000100u), sp = __builtin_amdgcn_perm(head, head, 0x03020302u);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            s.dd[i] = pk_mul_half(d[i], dp);
            s.ms[i] = pk_mul_half(m[i], sp);
        }
    } else {
        s.d8 = cvt_half_lo(head);
        s.c4 = -4.0f * cvt_half_hi(head);
#pragma unroll
        for (int i = 0; i < 8; ++i) s.d4[i] = d[i];
    }
    return s;
}

// fma(a, dd, ms) with the fp16 pair's lo / hi half of dd and ms.
__device__ __forceinline__ float fma_mix_dm_lo(float a, uint32_t dd, uint32_t ms) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[0,1,1]" : "=v"(r) : "v"(a), "v"(dd), "v"(ms));
    return r;
}
__device__ __forceinline__ float fma_mix_dm_hi(float a, uint32_t dd, uint32_t ms) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[0,1,1] op_sel_hi:[0,1,1]" : "=v"(r) : "v"(a), "v"(dd), "v"(ms));
    return r;
}

// The reference's lane value of one block and fragment for register v.
template<bool Q41>
__device__ __forceinline__ float frag_value(int I, const BlkScale<Q41> &s, int v) {
    if constexpr (Q41) {
        const float f = static_cast<float>(I);
        return (v & 1) ? fma_mix_dm_hi(f, s.dd[v >> 1], s.ms[v >> 1]) : fma_mix_dm_lo(f, s.dd[v >> 1], s.ms[v >> 1]);
    } else {
        const float t = fmaf(static_cast<float>(I), s.d8, s.c4);
        return (v & 1) ? mul_half_hi(s.d4[v >> 1], t) : mul_half_lo(s.d4[v >> 1], t);
    }
}

// The lane's accumulator over one more block and fragment.
template<bool Q41>
__device__ __forceinline__ void fragment_scale(float (&acc)[16], v16i I, const BlkScale<Q41> &s) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        if constexpr (Q41) {
            acc[v] = acc[v] + frag_value<true>(I[v], s, v);
        } else {
            const float t = fmaf(static_cast<float>(I[v]), s.d8, s.c4);
            acc[v] = (v & 1) ? fma_mix_hi(s.d4[v >> 1], t, acc[v]) : fma_mix_lo(s.d4[v >> 1], t, acc[v]);
        }
    }
}

// The nibbles of a dword at `shift` (0 low, 4 high) as bytes; Q4_1: doubled.
template<bool Q41>
__device__ __forceinline__ uint32_t nibbles(uint32_t w, int shift) {
    if constexpr (Q41) return (shift ? w >> 3 : w << 1) & (kNibbles << 1);
    else return (w >> shift) & kNibbles;
}

struct GuTile {
    __amdgpu_buffer_rsrc_t wr, sr, xr, hr;
    __amdgpu_buffer_rsrc_t mr;   // Q4_1: weight mins (the scales' layout); unused for Q4_0
    uint32_t w_off, s_off0, s_off1, x_off, h_off;   // token block b at x_off + b XStride / h_off + b HStride
    int nb, shift;
    int32_t *dots;     // debug: [pair][I][nb] or null
    size_t dot_base;   // dots index of (pair of this lane, row R0 + 16h, block 0)
    bool dot_ok;
};

// Per-block steps of a token's codes and head: split planes (32 / 4 bytes),
// or canonical 36-byte Q8_1 blocks read in place (Canon).
template<bool Canon> constexpr uint32_t XStride = Canon ? 36u : 32u;
template<bool Canon> constexpr uint32_t HStride = Canon ? 36u : 4u;

struct BlockLoads {
    uint4 w, d0, d1, m0, m1, x;
    uint32_t hd;
};

template<bool Canon, bool Q41>
__device__ __forceinline__ BlockLoads block_loads(const GuTile &t, int b) {
    const uint32_t ub = static_cast<uint32_t>(b);
    BlockLoads l;
    l.w = buffer_load16(t.wr, t.w_off, ub * 16u);
    l.d0 = buffer_load16(t.sr, t.s_off0, ub * 16u);
    l.d1 = buffer_load16(t.sr, t.s_off1, ub * 16u);
    if constexpr (Q41) {
        l.m0 = buffer_load16(t.mr, t.s_off0, ub * 16u);
        l.m1 = buffer_load16(t.mr, t.s_off1, ub * 16u);
    }
    l.x = buffer_load16(t.xr, t.x_off, ub * XStride<Canon>);
    l.hd = buffer_load4(t.hr, t.h_off, ub * HStride<Canon>);
    return l;
}

// Fragment f's dots of one block for the wave's 32 rows x 32 tokens.
template<int F, bool Q41>
__device__ __forceinline__ v16i fragment_dots(const GuTile &t, const BlockLoads &l) {
    const v16i zero = {};
    const v4i B = {static_cast<int>(l.x.x), static_cast<int>(l.x.y), static_cast<int>(l.x.z), static_cast<int>(l.x.w)};
    const v4i A = F == 0 ? v4i{static_cast<int>(nibbles<Q41>(l.w.x, t.shift)), static_cast<int>(nibbles<Q41>(l.w.y, t.shift)), 0, 0}
                         : v4i{0, 0, static_cast<int>(nibbles<Q41>(l.w.z, t.shift)), static_cast<int>(nibbles<Q41>(l.w.w, t.shift))};
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B, zero, 0, 0, 0);
}

template<bool Dbg>
__device__ __forceinline__ void store_dots(const GuTile &t, int b, v16i I0, v16i I1) {
    if constexpr (Dbg) {
        if (t.dot_ok)
#pragma unroll
            for (int v = 0; v < 16; ++v) t.dots[t.dot_base + static_cast<size_t>(v) * t.nb + b] = I0[v] + I1[v];
    }
}

// ---- H <= 2048 (one block per reference lane): staged scales and heads,
// weights and activations prefetched one leaf pair ahead.

struct GuStage {
    const uint32_t *d4;   // LDS [nb][32 halfs] of this wave's rows (row 16h + v at half 16h + v)
    const uint32_t *m4;   // Q4_1: LDS mins, the scales' layout
};

struct Blk {
    uint4 w, x;           // code chunk of the lane's A row, Q8 codes of its token (16 bytes each)
};

template<bool Canon = false>
__device__ __forceinline__ Blk blk_load(const GuTile &t, int b) {
    const uint32_t ub = static_cast<uint32_t>(b);
    return Blk{buffer_load16(t.wr, t.w_off, ub * 16u), buffer_load16(t.xr, t.x_off, ub * XStride<Canon>)};
}

// Fragment F's dots of one block with v_mfma_i32_32x32x16_i8 (K = 16 = one
// fragment): lane half h supplies the fragment's 8 nibbles of elements
// 16h + 8F .. +7 and the same 8 Q8 codes.
template<int F, bool Q41>
__device__ __forceinline__ v16i frag_mfma(const Blk &k, int shift) {
    const uint32_t w0 = F ? k.w.z : k.w.x, w1 = F ? k.w.w : k.w.y;
    const uint32_t x0 = F ? k.x.z : k.x.x, x1 = F ? k.x.w : k.x.y;
    const long A = static_cast<long>((static_cast<uint64_t>(nibbles<Q41>(w1, shift)) << 32) | nibbles<Q41>(w0, shift));
    const long B = static_cast<long>((static_cast<uint64_t>(x1) << 32) | x0);
    return __builtin_amdgcn_mfma_i32_32x32x16_i8(A, B, v16i{}, 0, 0, 0);
}

// Block `blk`'s staged scales (and mins) against a token's head.
template<bool Q41>
__device__ __forceinline__ BlkScale<Q41> staged_scale(const GuStage &g, int blk, int h, uint32_t head) {
    const uint4 *d = reinterpret_cast<const uint4 *>(g.d4 + blk * 16 + 8 * h);
    if constexpr (Q41) {
        const uint4 *m = reinterpret_cast<const uint4 *>(g.m4 + blk * 16 + 8 * h);
        return blk_scale<true>(head, d[0], d[1], m[0], m[1]);
    } else {
        return blk_scale<false>(head, d[0], d[1], uint4{}, uint4{});
    }
}

// v(k') = (acc[2k'] + acc[2(k'+32)]) + (acc[2k'+1] + acc[2(k'+32)+1]) with
// acc[2j+f] the fragment-f value of block j (+0 past nb).  Full: nb == 64.
// Blocks k' and k'+32 are loaded here; the fragment-0 pair is finished before
// the fragment-1 MFMAs so only two MFMA results are live.
// A block past the row's end is an unused lane of the reference, +0: its dots
// are not computed at all (rows of 20 blocks: 20 blocks' work instead of 64;
// Q4_1 640 x 2560 at 128 / 1032 columns 17.1 / 62.7 -> 11.5 / 35.1 us, Q4_0
// 1024 x 4096 at 128 / 512 16.9 / 53.8 -> 10.7 / 33.9).
template<bool Canon, bool Q41>
__device__ __forceinline__ void leaf_staged(const GuTile &t, const GuStage &g, int kp, int h, float (&v)[16]) {
    const int jb = kp + 32;
    if (kp >= t.nb) {   // uniform
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = 0.0f;
        return;
    }
    const Blk ka = blk_load<Canon>(t, kp);
    const uint32_t ha = buffer_load4(t.hr, t.h_off, static_cast<uint32_t>(kp) * HStride<Canon>);
    if (jb >= t.nb) {   // uniform
        const BlkScale<Q41> sa = staged_scale<Q41>(g, kp, h, ha);
        const v16i I0 = frag_mfma<0, Q41>(ka, t.shift), I1 = frag_mfma<1, Q41>(ka, t.shift);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = frag_value<Q41>(I0[i], sa, i) + frag_value<Q41>(I1[i], sa, i);
    } else {
        const Blk kb = blk_load<Canon>(t, jb);
        const uint32_t hb = buffer_load4(t.hr, t.h_off, static_cast<uint32_t>(jb) * HStride<Canon>);
        const BlkScale<Q41> sa = staged_scale<Q41>(g, kp, h, ha), sb = staged_scale<Q41>(g, jb, h, hb);
        float u0[16];
        {
            const v16i Ia = frag_mfma<0, Q41>(ka, t.shift), Ib = frag_mfma<0, Q41>(kb, t.shift);
#pragma unroll
            for (int i = 0; i < 16; ++i) u0[i] = frag_value<Q41>(Ia[i], sa, i) + frag_value<Q41>(Ib[i], sb, i);
        }
        {
            const v16i Ia = frag_mfma<1, Q41>(ka, t.shift), Ib = frag_mfma<1, Q41>(kb, t.shift);
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = u0[i] + (frag_value<Q41>(Ia[i], sa, i) + frag_value<Q41>(Ib[i], sb, i));
        }
    }
    // One leaf at a time: hoisting the next leaf's loads and MFMAs above this
    // point multiplies the live registers.
    __builtin_amdgcn_sched_barrier(0);
}

// ---- H == 2048 (64 blocks): loads in groups of four leaves that use whole
// cache lines.  Group g covers blocks 4g..4g+3 and 4g+32..4g+35, loaded half
// (two leaves) at a time.  Lane half h of row m reads contiguous bytes of its
// row (blocks 4g+32h+i); a v_permlane32_swap of the low- and high-nibble
// words then gives, per leaf, the MFMA operand of block 4g+i (low nibbles in
// lanes < 32, high in lanes >= 32) and of block 4g+32+i.  Lane half h of
// token n reads bytes 16h..16h+15 of consecutive 32-byte Q8 blocks, so the
// two halves of a token use the same lines.
struct HalfGroup {
    uint4 w[2];           // A row: blocks 4g+2q+i (h = 0) / 4g+32+2q+i (h = 1)
    uint4 xa[2], xb[2];   // token codes, half h: blocks 4g+2q+i / 4g+32+2q+i
    uint2 ha, hb;         // token heads of blocks 4g+2q, +1 / 4g+32+2q, +1
};

// The operands of level-1 node p = 2g + q (leaves 4g + 2q and 4g + 2q + 1).
// Loading half a line group at a time keeps the kernel at three waves per
// SIMD (a whole group in registers needed 211 VGPRs: two waves).  The weight
// half (8 VGPRs) of node p + 1 is loaded while node p computes (157 VGPRs;
// 16K layer 5.42 -> 5.35 ms); the activation half as well would need 177
// VGPRs, two waves per SIMD.
__device__ __forceinline__ void half_load_w(const GuTile &t, uint32_t w_off, int p, uint4 (&w)[2]) {
    const uint32_t b0 = static_cast<uint32_t>(4 * (p >> 1) + 2 * (p & 1));
#pragma unroll
    for (int i = 0; i < 2; ++i) w[i] = buffer_load16(t.wr, w_off, (b0 + i) * 16u);
}
template<bool Canon = false>
__device__ __forceinline__ void half_load_x(const GuTile &t, int p, HalfGroup &G) {
    constexpr uint32_t xs = XStride<Canon>, hs = HStride<Canon>;
    const uint32_t b0 = static_cast<uint32_t>(4 * (p >> 1) + 2 * (p & 1));
#pragma unroll
    for (int i = 0; i < 2; ++i) G.xa[i] = buffer_load16(t.xr, t.x_off, (b0 + i) * xs);
#pragma unroll
    for (int i = 0; i < 2; ++i) G.xb[i] = buffer_load16(t.xr, t.x_off, (b0 + 32 + i) * xs);
    if constexpr (Canon) {
        G.ha = make_uint2(buffer_load4(t.hr, t.h_off, b0 * hs), buffer_load4(t.hr, t.h_off, (b0 + 1) * hs));
        G.hb = make_uint2(buffer_load4(t.hr, t.h_off, (b0 + 32) * hs), buffer_load4(t.hr, t.h_off, (b0 + 33) * hs));
    } else {   // head plane: the two heads are adjacent
        const auto a = __builtin_amdgcn_raw_buffer_load_b64(t.hr, t.h_off, b0 * hs, 0);
        const auto b = __builtin_amdgcn_raw_buffer_load_b64(t.hr, t.h_off, (b0 + 32) * hs, 0);
        G.ha = make_uint2(a[0], a[1]);
        G.hb = make_uint2(b[0], b[1]);
    }
}

__device__ __forceinline__ v16i frag_mfma2(uint32_t a0, uint32_t a1, uint32_t x0, uint32_t x1) {
    const long A = static_cast<long>((static_cast<uint64_t>(a1) << 32) | a0);
    const long B = static_cast<long>((static_cast<uint64_t>(x1) << 32) | x0);
    return __builtin_amdgcn_mfma_i32_32x32x16_i8(A, B, v16i{}, 0, 0, 0);
}

// Rows of 65..96 blocks in the grouped form (the reference model's 2560:
// 80 blocks).  Reference lane j also holds block j + 64 when j + 64 < nb, and
// its accumulator continues with fma(d4, t, acc) over that block; lane j + 32
// holds no second block (j + 96 >= nb).  So leaf kp's chain A gets one more
// block, kp + 64, for kp < nb - 64.  Its operands per node (leaves 2p, 2p+1):
// the lane's row chunk of the block, the token's half block and its head.
struct ExtraBlk {
    uint4 w[2], x[2];
    uint32_t hd[2];
};

template<bool Canon = false>
__device__ __forceinline__ void extra_load(const GuTile &t, int p, ExtraBlk &E) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t e = static_cast<uint32_t>(std::min(64 + 2 * p + i, t.nb - 1));   // past nb: unused
        E.w[i] = buffer_load16(t.wr, t.w_off, e * 16u);
        E.x[i] = buffer_load16(t.xr, t.x_off, e * XStride<Canon>);
        E.hd[i] = buffer_load4(t.hr, t.h_off, e * HStride<Canon>);
    }
}

// Block kp + 64's fragment F, after block kp's value (the chain of reference
// lane kp).
template<int F, bool Q41>
__device__ __forceinline__ v16i extra_dots(const ExtraBlk &E, int i, int shift) {
    return frag_mfma<F, Q41>(Blk{E.w[i], E.x[i]}, shift);
}

// The MFMA operands and scales of leaf kp's blocks kp (a) and kp + 32 (b).
template<bool Q41> struct LeafOps {
    uint32_t a[4], b[4];
    BlkScale<Q41> sa, sb;
    __device__ __forceinline__ LeafOps(const GuStage &g, const HalfGroup &G, int i, int kp, int h) {
        const uint4 wi = G.w[i];
        const uint32_t wv[4] = {wi.x, wi.y, wi.z, wi.w};
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const auto r = __builtin_amdgcn_permlane32_swap(nibbles<Q41>(wv[d], 0), nibbles<Q41>(wv[d], 4), false, false);
            a[d] = r[0];   // block kp: low nibbles (lanes < 32), high nibbles (lanes >= 32)
            b[d] = r[1];   // block kp + 32
        }
        sa = staged_scale<Q41>(g, kp, h, i ? G.ha.y : G.ha.x);
        sb = staged_scale<Q41>(g, kp + 32, h, i ? G.hb.y : G.hb.x);
    }
};

// Leaf kp with block kp + 64 in chain A: v = (A0 + B0) + (A1 + B1), with
// A_f = fma(d4', t', fma(d4, t, +0)) over blocks kp, kp + 64 and B_f block
// kp + 32's value, as leaf_grouped without the extra block.
template<bool Dbg, bool Q41>
__device__ __forceinline__ void leaf_grouped_extra(const GuTile &t, const GuStage &g, const HalfGroup &G,
                                                   const ExtraBlk &E, int i, int kp, int h, const LeafOps<Q41> &o,
                                                   float (&v)[16]) {
    const uint4 xa = G.xa[i], xb = G.xb[i];
    float u0[16];
    v16i keep_a0, keep_b0, keep_e0;
    {
        float za[16];
        const v16i Ia = frag_mfma2(o.a[0], o.a[1], xa.x, xa.y);
#pragma unroll
        for (int j = 0; j < 16; ++j) za[j] = frag_value<Q41>(Ia[j], o.sa, j);
        const v16i Ie = extra_dots<0, Q41>(E, i, t.shift);
        fragment_scale<Q41>(za, Ie, staged_scale<Q41>(g, kp + 64, h, E.hd[i]));
        const v16i Ib = frag_mfma2(o.b[0], o.b[1], xb.x, xb.y);
#pragma unroll
        for (int j = 0; j < 16; ++j) u0[j] = za[j] + frag_value<Q41>(Ib[j], o.sb, j);
        if constexpr (Dbg) { keep_a0 = Ia; keep_b0 = Ib; keep_e0 = Ie; }
    }
    {
        float za[16];
        const v16i Ia = frag_mfma2(o.a[2], o.a[3], xa.z, xa.w);
#pragma unroll
        for (int j = 0; j < 16; ++j) za[j] = frag_value<Q41>(Ia[j], o.sa, j);
        const v16i Ie = extra_dots<1, Q41>(E, i, t.shift);
        fragment_scale<Q41>(za, Ie, staged_scale<Q41>(g, kp + 64, h, E.hd[i]));
        const v16i Ib = frag_mfma2(o.b[2], o.b[3], xb.z, xb.w);
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = u0[j] + (za[j] + frag_value<Q41>(Ib[j], o.sb, j));
        if constexpr (Dbg) {
            store_dots<Dbg>(t, kp, keep_a0, Ia);
            store_dots<Dbg>(t, kp + 32, keep_b0, Ib);
            store_dots<Dbg>(t, kp + 64, keep_e0, Ie);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
}

// Shared: with an extra block, the operands are formed once, before the uniform
// branch; else on each side of it (the compiler then schedules the two sides
// each on its own).  us, shared / not, rows of 80 blocks x 2560: planes at 200 /
// 1,032 columns 28.2 / 86.2 against 28.7 / 87.0, Q4_1 91.1 against 91.8 at
// 1,032; but canonical Q4_0 blocks 24.2 / 79.1 against 23.9 / 78.2, and the
// gate / up kernel's layers lose 0.5 %.
template<bool Dbg, bool Extra, bool Q41, bool Shared>
__device__ __forceinline__ void leaf_grouped(const GuTile &t, const GuStage &g, const HalfGroup &G, int i, int kp, int h,
                                             float (&v)[16], const ExtraBlk &E) {
    if constexpr (Extra && !Shared) {
        if (kp < t.nb - 64) {   // uniform
            leaf_grouped_extra<Dbg, Q41>(t, g, G, E, i, kp, h, LeafOps<Q41>(g, G, i, kp, h), v);
            return;
        }
    }
    const LeafOps<Q41> o(g, G, i, kp, h);
    if constexpr (Extra && Shared) {
        if (kp < t.nb - 64) {   // uniform
            leaf_grouped_extra<Dbg, Q41>(t, g, G, E, i, kp, h, o, v);
            return;
        }
    }
    const uint4 xa = G.xa[i], xb = G.xb[i];
    float u0[16];
    v16i keep_a0, keep_b0;
    {
        const v16i Ia = frag_mfma2(o.a[0], o.a[1], xa.x, xa.y), Ib = frag_mfma2(o.b[0], o.b[1], xb.x, xb.y);
#pragma unroll
        for (int j = 0; j < 16; ++j) u0[j] = frag_value<Q41>(Ia[j], o.sa, j) + frag_value<Q41>(Ib[j], o.sb, j);
        if constexpr (Dbg) { keep_a0 = Ia; keep_b0 = Ib; }
    }
    {
        const v16i Ia = frag_mfma2(o.a[2], o.a[3], xa.z, xa.w), Ib = frag_mfma2(o.b[2], o.b[3], xb.z, xb.w);
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = u0[j] + (frag_value<Q41>(Ia[j], o.sa, j) + frag_value<Q41>(Ib[j], o.sb, j));
        if constexpr (Dbg) {
            store_dots<Dbg>(t, kp, keep_a0, Ia);
            store_dots<Dbg>(t, kp + 32, keep_b0, Ib);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
}

// Merge of the level-1 node p (= w, leaves 2p and 2p + 1) into the pairwise
// tree over v(0..31), upward like a binary counter, so each level holds at
// most one pending left operand.  Levels 1-2 stay in registers; levels 3-4
// (touched every 8, 16 leaves) wait in LDS (`park`, 2 x 16 floats per lane of
// this wave).
__device__ __forceinline__ void tree_merge(float (*park)[16][64], int lane, int p, float (&w)[16], float (&l1)[16],
                                           float (&l2)[16], float (&res)[16]) {
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
    int lvl = 0;
    for (; lvl < 2; ++lvl) {
        if (((p >> (lvl + 2)) & 1) == 0) break;
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i] = park[lvl][i][lane] + w[i];
    }
    if (lvl < 2) {
#pragma unroll
        for (int i = 0; i < 16; ++i) park[lvl][i][lane] = w[i];
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) res[i] = w[i];
    }
}

// The tree of a row of 65..96 blocks.
template<bool Dbg>
__device__ __forceinline__ void fold_tree_grouped96(const GuTile &t, const GuStage &g, uint32_t w_off, float (*park)[16][64],
                                                    int lane, uint4 (&wn)[2], float (&res)[16]) {
    // wn: node 0's weight half, already in flight.
    const int h = lane >> 5;
    float l1[16], l2[16];
#pragma unroll 1
    for (int p = 0; p < 16; ++p) {
        HalfGroup G;
        G.w[0] = wn[0];
        G.w[1] = wn[1];
        half_load_x(t, p, G);
        ExtraBlk E;
        if (2 * p < t.nb - 64) extra_load(t, p, E);   // uniform
        half_load_w(t, w_off, p < 15 ? p + 1 : p, wn);   // node p + 1's weights in flight during node p
        float w[16], x[16];
        leaf_grouped<Dbg, true, false, false>(t, g, G, 0, 2 * p, h, w, E);
        leaf_grouped<Dbg, true, false, false>(t, g, G, 1, 2 * p + 1, h, x, E);
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i] = w[i] + x[i];
        tree_merge(park, lane, p, w, l1, l2, res);
    }
}

// ---- H > 2048 (reference lanes holding several blocks): per-block loads.
// One block of a reference lane's chain: both fragment dots scaled into the
// lane's accumulators, acc = fma(d4, fma(float(I_f), d8, c4), acc).
template<bool Dbg, bool Q41>
__device__ __forceinline__ void chain_block(const GuTile &t, const BlockLoads &l, int b, float (&c0)[16],
                                            float (&c1)[16]) {
    const v16i I0 = fragment_dots<0, Q41>(t, l), I1 = fragment_dots<1, Q41>(t, l);
    const BlkScale<Q41> s = blk_scale<Q41>(l.hd, l.d0, l.d1, l.m0, l.m1);
    fragment_scale<Q41>(c0, I0, s);
    fragment_scale<Q41>(c1, I1, s);
    store_dots<Dbg>(t, b, I0, I1);
}

// Leaf kp for rows of more than 64 blocks: reference lanes kp and kp + 32,
// each the chain over its blocks j, j + 64, ... in increasing order (the
// reference lane array's acc[2j + f]), walked as one sequence -- kp's chain,
// then kp + 32's -- with
// each block's loads issued before the previous block is scaled.
template<bool Dbg, bool Canon, bool Q41>
__device__ __forceinline__ void fold_leaf_multi(const GuTile &t, int kp, float (&v)[16]) {
    float a0[16], a1[16], b0[16], b1[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) { a0[i] = 0.0f; a1[i] = 0.0f; b0[i] = 0.0f; b1[i] = 0.0f; }
    // nb > 64 here, so kp + 32 < nb and both chains hold a block.
    const int na = (t.nb - kp + 63) / 64, nc = (t.nb - kp - 32 + 63) / 64;
    BlockLoads cur = block_loads<Canon, Q41>(t, kp);
#pragma unroll 1
    for (int s = 0; s < na; ++s) {   // uniform
        const BlockLoads nxt = block_loads<Canon, Q41>(t, s + 1 < na ? kp + 64 * (s + 1) : kp + 32);
        chain_block<Dbg, Q41>(t, cur, kp + 64 * s, a0, a1);
        cur = nxt;
    }
#pragma unroll 1
    for (int s = 0; s < nc; ++s) {   // uniform
        BlockLoads nxt = cur;
        if (s + 1 < nc) nxt = block_loads<Canon, Q41>(t, kp + 32 + 64 * (s + 1));
        chain_block<Dbg, Q41>(t, cur, kp + 32 + 64 * s, b0, b1);
        cur = nxt;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = (a0[i] + b0[i]) + (a1[i] + b1[i]);
    __builtin_amdgcn_sched_barrier(0);
}

template<bool Dbg>
__device__ __forceinline__ void fold_tree_multi(const GuTile &t, float (*park)[16][64], int lane, float (&res)[16]) {
    float l1[16], l2[16];
#pragma unroll 1
    for (int p = 0; p < 16; ++p) {
        float w[16], x[16];
        fold_leaf_multi<Dbg, false, false>(t, 2 * p, w);
        fold_leaf_multi<Dbg, false, false>(t, 2 * p + 1, x);
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i] = w[i] + x[i];
        tree_merge(park, lane, p, w, l1, l2, res);
    }
}

enum { kFoldStaged = 0, kFoldGrouped = 1, kFoldMulti = 2, kFoldGrouped96 = 3 };


// ---------------------------------------------------------------- linear ---
// One matrix against wide column batches (moe_linear), in the gate/up kernel's
// exact order (Q4_1: its own block value) without the SiLU epilogue.  The reference's pairwise
// tree over the 16 level-1 nodes (leaves 2p, 2p+1; leaf k' = blocks k' and
// k' + 32 and, past 64 blocks, their lane's later blocks) splits into four
// 4-node subtrees whose roots combine as (R0 + R1) + (R2 + R3): workgroup =
// one 32-row x 32-column tile, wave w builds subtree w, so a tile's
// sequential work is a quarter of the gate/up kernel's.  The waves share the
// rows' scales staged in LDS.  Ids are XCD-aware: the column tiles of one row
// tile run on one XCD, so its rows are fetched from HBM once.
__device__ __forceinline__ void subtree4_merge(int q, float (&w)[16], float (&l1)[16], float (&l2)[16],
                                               float (&res)[16]) {
    if ((q & 1) == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) l1[i] = w[i];
        return;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = l1[i] + w[i];
    if ((q & 2) == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) l2[i] = w[i];
        return;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) res[i] = l2[i] + w[i];
}

// The two-node form for 8-wave workgroups: res = node 0 + node 1.
__device__ __forceinline__ void subtree2_merge(int q, float (&w)[16], float (&l1)[16], float (&res)[16]) {
    if ((q & 1) == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) l1[i] = w[i];
        return;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) res[i] = l1[i] + w[i];
}

// NPW level-1 nodes per wave (4: a 4-wave workgroup, 2: an 8-wave one).  wn: the
// wave's first node's weight half, already in flight (grouped folds).
template<int Fold, bool Canon, int NPW, bool Q41>
__device__ __forceinline__ void subtree(const GuTile &t, const GuStage &g, uint32_t w_off, int wave, int lane,
                                        uint4 (&wn)[2], float (&res)[16]) {
    static_assert(NPW == 4 || NPW == 2, "subtree: 2 or 4 nodes per wave");
    const int h = lane >> 5;
    float l1[16], l2[16];
    if constexpr (Fold == kFoldGrouped || Fold == kFoldGrouped96) {
        constexpr bool X = Fold == kFoldGrouped96;
        // Node q + 1's weight half is in flight while node q computes.
#pragma unroll 1
        for (int q = 0; q < NPW; ++q) {
            const int p = NPW * wave + q;
            HalfGroup G;
            G.w[0] = wn[0];
            G.w[1] = wn[1];
            half_load_x<Canon>(t, p, G);
            ExtraBlk E;
            if constexpr (X) {
                if (2 * p < t.nb - 64) extra_load<Canon>(t, p, E);   // uniform
            }
            half_load_w(t, w_off, q < NPW - 1 ? p + 1 : p, wn);
            float w[16], x[16];
            leaf_grouped<false, X, Q41, Q41 || !Canon>(t, g, G, 0, 2 * p, h, w, E);
            leaf_grouped<false, X, Q41, Q41 || !Canon>(t, g, G, 1, 2 * p + 1, h, x, E);
#pragma unroll
            for (int i = 0; i < 16; ++i) w[i] = w[i] + x[i];
            if constexpr (NPW == 4) subtree4_merge(q, w, l1, l2, res);
            else subtree2_merge(q, w, l1, res);
        }
    } else {
#pragma unroll 1
        for (int q = 0; q < NPW; ++q) {
            const int p = NPW * wave + q;
            float w[16], x[16];
            if constexpr (Fold == kFoldStaged) {
                leaf_staged<Canon, Q41>(t, g, 2 * p, h, w);
                leaf_staged<Canon, Q41>(t, g, 2 * p + 1, h, x);
            } else {
                fold_leaf_multi<false, Canon, Q41>(t, 2 * p, w);
                fold_leaf_multi<false, Canon, Q41>(t, 2 * p + 1, x);
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) w[i] = w[i] + x[i];
            if constexpr (NPW == 4) subtree4_merge(q, w, l1, l2, res);
            else subtree2_merge(q, w, l1, res);
        }
    }
}

template<bool Q41> using LinearArgsOf = std::conditional_t<Q41, LinearMfmaQ41Args, LinearMfmaArgs>;

// Canon: the columns are canonical Q8_1 blocks, read in place (codes at
// byte 4 of each 36-byte block, the head at byte 0); else the split planes.
// W = 8: eight waves of two level-1 nodes each, the roots combined
// ((R0 + R1) + (R2 + R3)) + ((R4 + R5) + (R6 + R7)) -- the same tree levels
// as the 4-wave form's (R0 + R1) + (R2 + R3) over 4-node subtrees -- for
// launches whose 4-wave grid leaves SIMDs with one wave.
template<int Fold, bool Canon, int W, bool Q41>
__global__ __launch_bounds__(64 * W, W == 8 ? 1 : 2) void k_linear_mfma(LinearArgsOf<Q41> a) {
    constexpr int NPW = 16 / W, VPW = 16 / W;   // level-1 nodes and finished values per wave
    __shared__ float roots[W][16][64];          // subtree roots [wave][value][lane]
    constexpr int SB = Fold == kFoldGrouped96 ? kGu96MaxBlocks : Fold == kFoldMulti ? 1 : kGuMaxBlocks;
    __shared__ uint4 d4_lds[SB][4];             // [block][32 halfs]
    __shared__ uint4 m4_lds[Q41 ? SB : 1][4];   // Q4_1 mins
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int id = static_cast<int>(blockIdx.x), local = id >> 3;
    const int rt = (id & 7) + 8 * (local / a.col_tiles), ct = local % a.col_tiles;
    if (rt >= a.row_tiles) return;   // uniform per workgroup (grid padded to 8 row tiles)
    const int nb = a.nb, R0 = rt * 32, c0 = ct * kSub;
    const int lane = threadIdx.x & 63;
    const int m = lane & 31, h = lane >> 5;
    const int prow = 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
    const uint32_t col = static_cast<uint32_t>(std::min(c0 + m, a.N - 1));
    const uint32_t row_bytes = static_cast<uint32_t>(nb) * 16u;
    GuTile t;
    t.wr = buffer_rsrc(a.codes + static_cast<size_t>(R0) * row_bytes, 32u * row_bytes);
    t.sr = buffer_rsrc(a.scales + static_cast<size_t>(R0) * nb, 32u * static_cast<uint32_t>(nb) * 2u);
    if constexpr (Q41) t.mr = buffer_rsrc(a.mins + static_cast<size_t>(R0) * nb, 32u * static_cast<uint32_t>(nb) * 2u);
    if constexpr (Canon) {
        t.xr = buffer_rsrc(a.q8, static_cast<uint32_t>(a.N) * static_cast<uint32_t>(nb) * 36u);
        t.hr = t.xr;
        t.x_off = col * static_cast<uint32_t>(nb) * 36u + 4u + 16u * h;
        t.h_off = col * static_cast<uint32_t>(nb) * 36u;
    } else {
        t.xr = buffer_rsrc(a.xq.codes, static_cast<uint32_t>(a.N) * static_cast<uint32_t>(nb) * 32u);
        t.hr = buffer_rsrc(a.xq.heads, static_cast<uint32_t>(a.N) * static_cast<uint32_t>(nb) * 4u);
        t.x_off = col * static_cast<uint32_t>(nb) * 32u + 16u * h;
        t.h_off = col * static_cast<uint32_t>(nb) * 4u;
    }
    t.w_off = static_cast<uint32_t>(prow) * row_bytes;
    t.s_off0 = static_cast<uint32_t>(2 * h * nb) * 16u;
    t.s_off1 = t.s_off0 + static_cast<uint32_t>(nb) * 16u;
    t.nb = nb;
    t.shift = 4 * h;
    t.dots = nullptr;
    t.dot_base = 0;
    t.dot_ok = false;
    // The first node's weight half is issued before the scale staging, so the
    // two round trips overlap.
    const uint32_t w_off = static_cast<uint32_t>(prow) * row_bytes + 32u * 16u * h;
    uint4 wn[2] = {};
    if constexpr (Fold == kFoldGrouped || Fold == kFoldGrouped96) half_load_w(t, w_off, NPW * wave, wn);
    if constexpr (Fold != kFoldMulti) {
        // Scale group g (rows 8g..8g+7) of block b lands at halfs 8g..8g+7 of d4_lds[b].
        for (int c = threadIdx.x; c < 4 * nb; c += blockDim.x) {
            const int gi = c / nb, b = c % nb;
            const size_t at = static_cast<size_t>(R0 + 8 * gi) * nb + b * 8;
            d4_lds[b][gi] = *reinterpret_cast<const uint4 *>(a.scales + at);
            if constexpr (Q41) m4_lds[b][gi] = *reinterpret_cast<const uint4 *>(a.mins + at);
        }
        __syncthreads();
    }
    const GuStage g{reinterpret_cast<const uint32_t *>(&d4_lds[0][0]), reinterpret_cast<const uint32_t *>(&m4_lds[0][0])};
    float res[16];
    subtree<Fold, Canon, NPW, Q41>(t, g, w_off, wave, lane, wn, res);
#pragma unroll
    for (int v = 0; v < 16; ++v) roots[wave][v][lane] = res[v];
    __syncthreads();
    // Wave w finishes values VPW w .. VPW w + VPW - 1: rows R0 + 16h + VPW w + i
    // of column c0 + m.
    const int c = c0 + m;
    const int row = R0 + 16 * h + VPW * wave;
    if (c >= a.N || row >= a.M) return;
    float out[VPW];
#pragma unroll
    for (int i = 0; i < VPW; ++i) {
        const int v = VPW * wave + i;
        const float q0 = (roots[0][v][lane] + roots[1][v][lane]) + (roots[2][v][lane] + roots[3][v][lane]);
        if constexpr (W == 4) out[i] = q0;
        else out[i] = q0 + ((roots[4][v][lane] + roots[5][v][lane]) + (roots[6][v][lane] + roots[7][v][lane]));
        // Q4_1: half of the doubled sum; + 0: the reference's lanes start from
        // +0, so none of its sums is -0 (Q4_0's lane values do so as well).
        if constexpr (Q41) out[i] = 0.5f * out[i] + 0.0f;
    }
    float *yr = a.y + static_cast<size_t>(c) * a.M + row;
    if constexpr (W == 4) {
        if (row + 4 <= a.M && (a.M & 3) == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0) {
            *reinterpret_cast<float4 *>(yr) = make_float4(out[0], out[1], out[2], out[3]);
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < VPW; ++i)
        if (row + i < a.M) yr[i] = out[i];
}

template<bool Canon, int W, bool Q41>
void launch_linear_mfma_t(const LinearArgsOf<Q41> &a, hipStream_t s) {
    constexpr unsigned T = 64 * W;
    const unsigned grid = static_cast<unsigned>((a.row_tiles + 7) / 8 * 8) * static_cast<unsigned>(a.col_tiles);
    // Only 64-block rows take the 8-wave form: for the other folds the
    // compiler's register allocator fails on it (with the iterative-ILP
    // scheduler that moe_mfma.hip is built with).
    if (a.nb == kGuMaxBlocks) k_linear_mfma<kFoldGrouped, Canon, W, Q41><<<grid, T, 0, s>>>(a);
    else if (a.nb > kGuMaxBlocks && a.nb <= kGu96MaxBlocks) k_linear_mfma<kFoldGrouped96, Canon, 4, Q41><<<grid, 256, 0, s>>>(a);
    else if (a.nb < kGuMaxBlocks) k_linear_mfma<kFoldStaged, Canon, 4, Q41><<<grid, 256, 0, s>>>(a);
    else k_linear_mfma<kFoldMulti, Canon, 4, Q41><<<grid, 256, 0, s>>>(a);
}
}  // namespace
}  // namespace moe
