// jk_gemm_few.hip -- repacked GEMM where the output has few tiles (3 tokens up to a few hundred).
//
// The products of jk_gemm.hip (execute_gemm_repacked_rows, repack.rs:2718-3042) where the tiled
// kernels cannot fill the GPU. Those give a wave 32 weight rows and all of K, with one 128-element
// chunk of weights in flight, so a small launch of any size waits out the same chain of loads:
// Q4_K with 4096 columns took 33 us for 1024 rows and 38 us for 14336 at any count up to 32
// tokens, Q6_K 4096 x 14336 201 us up to 256 tokens.
//
// A workgroup owns 16 RW weight rows x 16 TW tokens as 16 x 16 tiles, one per wave, and K advances in
// chunks of KU units of 256 elements, moved from global memory straight into one of two LDS stages
// while the other is evaluated. With few tiles, K is split over KW = KU waves per tile, unit u of a
// chunk on wave u: a wave computes every scale group's addend of its unit,
//     term = f32(dot) * (xs * ws)  [- xsum * wm],
// into registers -- the exact integer dot from v_mfma_i32_16x16x32_i8, the scale products of four
// groups from one v_mfma_f32_16x16x1_4b_f32 (each a single rounded f32 product) -- and then waits
// for its turn: the tile's running sums travel through LDS from the wave of the unit before, which
// has added its terms, to this one, which adds its own in group order. Each output is therefore the
// reference's sum in the reference's order, bit for bit, while loads, unpacking, products and
// scale products run on all the waves; only the additions are a chain. In tolerance mode the order
// is free: each wave keeps sums of its own (one fused multiply-add per group), added at the end.
//
// What bounds it: the chain's hand-over at few tiles (Q6_K 4096 x 14336 at 4 tokens: VALU busy 50% of the
// cycles, a wave waiting 44% of its time; 24 us), and from about eight tiles per CU the VALU (512 tokens: 99%;
// Q4_0 11008 x 4096 at 150 tokens in tolerance mode 74%, and 29% f32 and integer MFMAs, of which the f32 ones
// stall it). Of its instructions a unit and tile some 130 in 215 are the four operations per output and group
// that the recipe takes (Q4_K); unpacking, swapping and scaling the operands for a single 16 x 16 tile are
// the rest. Next to these, loads straight from global memory in the operands' layout (64 lines a load) had
// kept the address unit busy 80% of the time.
//
// Operands: lane l holds weight row (or token) l % 16 and part kq = l / 16 of K. For a pair of
// 32-element groups lane kq reads 16 bytes -- piece kq % 2 of group kq / 2 of the pair -- and
// v_permlane32_swap_b32 of dwords 0 and 2, and 1 and 3, leaves each group's 8 operand bytes in every
// lane: lane kq holds piece kq % 2, bytes 8 (kq / 2) .. of the group. Weights and activations use
// the same order of K within a group, so the dot is the group's.
#include "jk_device.hpp"

namespace jk {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
// (named address space: through a generic pointer a volatile access is a flat instruction, which
// waits for the global loads in flight too)
typedef __attribute__((address_space(3))) v4f lds_v4f_t;
typedef __attribute__((address_space(3))) int lds_int_t;

template <int Q> struct FewFmt {
    static constexpr bool B32 = fmt_of(Q).be == 32;
    static constexpr bool G16 = Q == JK_Q6_K;                   // 16-element scale groups
    static constexpr bool MINS = Q == JK_Q4_K || Q == JK_Q5_K;
    static constexpr int NG = G16 ? 16 : 8;                     // scale groups per unit
    static constexpr int NP = NG / 4;                           // scale-product MFMAs per unit
    static constexpr int NL = Q == JK_Q8_0 || Q == JK_Q4_0 ? 4 : Q == JK_Q6_K || Q == JK_Q5_K ? 3 : 2;  // 16-byte loads
    // quants are stored biased by this: -BIAS times the group's activation sum, from an MFMA
    // against a constant operand, starts the group's accumulator (one MFMA for all the row tiles
    // instead of three VALU instructions per weight dword)
    static constexpr int BIAS = Q == JK_Q4_0 ? 8 : Q == JK_Q6_K ? 32 : 0;
};

// One lane's share of a unit of 16 weight rows.
template <int Q> struct FewW {
    u32x4 q[FewFmt<Q>::NL];  // Q5_K: q[2] is qh; Q6_K: q[2] is qh
    u32x4 hd;                // Q4_K / Q5_K: d, dmin, packed scales and mins of the row
    uint32_t d[2];           // 32-element formats: f16 scales of groups 2 kq, 2 kq + 1; Q6_K: d, 4 scales
};
// One lane's share of a unit of 16 tokens.
struct FewX {
    u32x4 q[4];
    float2 s, m;  // scales (and sums) of 32-blocks 2 kq, 2 kq + 1 of the unit
};

// A chunk of KU units in LDS, 16-byte pieces and dwords placed so that the 16 rows (or tokens) an
// operand read covers fall on distinct banks: the slot of a piece is XORed with its row or token.
template <int Q, int RW, int TW, int KU> struct alignas(16) FewStage {
    static constexpr int C = fmt_of(Q).chunks;
    static constexpr int SB = FewFmt<Q>::B32 ? 8 * KU : KU;  // blocks of a row
    static constexpr int SW = SB < 16 ? SB : 16;
    static constexpr bool D = fmt_of(Q).d_off >= 0;
    // scale dwords of a row (256-element blocks: room for KU scales from an odd element on)
    static constexpr int DW = !D ? 0 : FewFmt<Q>::B32 ? 4 * KU : KU > 4 ? 8 : 4;
    static_assert(!D || FewFmt<Q>::B32 || 2 * DW > KU, "KU scales from an odd element on");
    uint8_t w[C * 16 * RW * SB * 16];  // [plane][row][block]
    uint8_t x[16 * TW * KU * 256];     // [token][16-byte piece]
    float xs[16 * TW * KU * 8];        // [token][32-block]
    float xm[FewFmt<Q>::MINS ? 16 * TW * KU * 8 : 4];
    uint32_t d[D ? 16 * RW * DW : 4];  // [row][dword]: the row's f16 scales from an even element on
    static __device__ __forceinline__ int wslot(int row, int blk) { return blk ^ ((row / (16 / SW)) & (SW - 1)); }
    static __device__ __forceinline__ int sslot(int tok, int blk) { return blk ^ ((2 * tok) & (8 * KU - 1)); }
};

// This wave's share of the global-to-LDS loads of chunk c (addresses past the row or token range
// are clamped: read and never used).
template <int Q, int RW, int TW, int KU, int KW>
__device__ __forceinline__ void few_issue(FewStage<Q, RW, TW, KU> &S, const WeightDev &w, const jk_act_q8 &a, int n0,
                                          int r1, int m0, int c, int wave, int lane) {
    using St = FewStage<Q, RW, TW, KU>;
    constexpr int NW = RW * TW * KW;
    const int nb = w.nb, M = (int)a.m;
    static_assert(St::C * RW * St::SB % 4 == 0 && RW * St::DW % 4 == 0, "whole loads");
    constexpr int NWI = St::C * RW * St::SB / 4, NXI = 4 * TW * KU, NSI = 2 * TW * KU, NDI = RW * St::DW / 4;
#pragma unroll
    for (int i = 0; i < (NWI + NW - 1) / NW; ++i) {
        const int n = min(wave + NW * i, NWI - 1), p = 64 * n + lane;
        const int slot = p % St::SB, row = p / St::SB % (16 * RW), plane = p / (St::SB * 16 * RW);
        const int b = min(St::SB * c + St::wslot(row, slot), nb - 1);
        const size_t at = ((size_t)plane * (size_t)w.rows + (size_t)min(n0 + row, r1 - 1)) * (size_t)nb + (size_t)b;
        lds_dma16(w.planes + at * 16, (lds_u8_t *)S.w + 1024 * n);
    }
#pragma unroll
    for (int i = 0; i < (NXI + NW - 1) / NW; ++i) {
        const int n = min(wave + NW * i, NXI - 1), p = 64 * n + lane;
        const int slot = p % (16 * KU), tok = p / (16 * KU);
        const int k = min(256 * KU * c + 16 * (slot ^ (tok & 15)), (int)a.k_padded - 16);
        lds_dma16(a.qs + (size_t)min(m0 + tok, M - 1) * a.k_padded + k, (lds_u8_t *)S.x + 1024 * n);
    }
#pragma unroll
    for (int i = 0; i < (NSI + NW - 1) / NW; ++i) {
        const int n = min(wave + NW * i, NSI - 1), e = 64 * n + lane;
        const int slot = e % (8 * KU), tok = e / (8 * KU);
        const size_t at = (size_t)min(m0 + tok, M - 1) * a.k_blocks32 +
                          (size_t)min(8 * KU * c + St::sslot(tok, slot), (int)a.k_blocks32 - 1);
        lds_dma4(a.scales + at, (lds_u8_t *)S.xs + 256 * n);
        if constexpr (FewFmt<Q>::MINS) lds_dma4(a.sums + at, (lds_u8_t *)S.xm + 256 * n);
    }
    if constexpr (St::D)
#pragma unroll
        for (int i = 0; i < (NDI + NW - 1) / NW; ++i) {
            const int n = min(wave + NW * i, NDI - 1), e = 64 * n + lane;
            const int dw = e % St::DW, row = e / St::DW;
            const size_t first = (size_t)min(n0 + row, r1 - 1) * (size_t)nb + (size_t)(St::SB * c);
            // (the scale plane is padded to whole dwords)
            const size_t at = min(first / 2 + (size_t)dw, ((size_t)w.rows * (size_t)nb - 1) / 2);
            lds_dma4(reinterpret_cast<const uint32_t *>(w.dplane) + at, (lds_u8_t *)S.d + 256 * n);
        }
}

// Reads of unit v of the staged chunk: weight row 16 rw + jl, token 16 tw + jl.
template <int Q, int RW, int TW, int KU>
__device__ __forceinline__ void few_wread(FewW<Q> &o, const FewStage<Q, RW, TW, KU> &S, int row, int v, int kq,
                                          int dodd) {
    using St = FewStage<Q, RW, TW, KU>;
    auto piece = [&](int plane, int blk) {
        return S.w + ((plane * 16 * RW + row) * St::SB + St::wslot(row, blk)) * 16;
    };
    auto ld16 = [](const uint8_t *p) { return *reinterpret_cast<const u32x4 *>(p); };
    if constexpr (FewFmt<Q>::B32) {
        // pair j: group kq / 2 of it, piece kq % 2 (Q4_0: one piece)
#pragma unroll
        for (int j = 0; j < 4; ++j) o.q[j] = ld16(piece(Q == JK_Q8_0 ? kq & 1 : 0, 8 * v + 2 * j + (kq >> 1)));
        const uint32_t dd = S.d[row * St::DW + 4 * v + kq];
        o.d[0] = dd & 0xFFFFu;
        o.d[1] = dd >> 16;
    } else if constexpr (Q == JK_Q6_K) {
        o.q[0] = ld16(piece(kq, v));      // ql of half 0
        o.q[1] = ld16(piece(4 + kq, v));  // ql of half 1
        o.q[2] = ld16(piece(8 + kq, v));  // qh: half kq / 2, piece kq % 2
        o.d[0] = reinterpret_cast<const uint16_t *>(S.d + row * St::DW)[dodd + v];
        o.d[1] = *reinterpret_cast<const uint32_t *>(piece(12, v) + 4 * kq);
    } else {
        constexpr int Q0 = Q == JK_Q5_K ? 3 : 1;
        o.q[0] = ld16(piece(Q0 + kq, v));      // quarters 0, 1
        o.q[1] = ld16(piece(Q0 + 4 + kq, v));  // quarters 2, 3
        o.hd = ld16(piece(0, v));
        if constexpr (Q == JK_Q5_K) o.q[2] = ld16(piece(1 + (kq & 1), v));
    }
}
template <int Q, int RW, int TW, int KU>
__device__ __forceinline__ void few_xread(FewX &o, const FewStage<Q, RW, TW, KU> &S, int tok, int v, int kq) {
    using St = FewStage<Q, RW, TW, KU>;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        o.q[j] = *reinterpret_cast<const u32x4 *>(S.x + (tok * 16 * KU + ((16 * v + 4 * j + kq) ^ (tok & 15))) * 16);
    const int e = tok * 8 * KU + St::sslot(tok, 8 * v + 2 * kq);
    o.s = *reinterpret_cast<const float2 *>(S.xs + e);
    if constexpr (FewFmt<Q>::MINS) o.m = *reinterpret_cast<const float2 *>(S.xm + e);
}

// Leaves the 8 operand bytes of the pair's two groups in dwords 0, 1 and 2, 3 of the lane's piece.
__device__ __forceinline__ void pair_swap(u32x4 &v) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const auto s = __builtin_amdgcn_permlane32_swap(v[k], v[2 + k], false, false);
        v[k] = s[0];
        v[2 + k] = s[1];
    }
}
template <int Q> __device__ __forceinline__ void few_swap(FewW<Q> &w) {
#pragma unroll
    for (int i = 0; i < FewFmt<Q>::NL; ++i)
        if (!(Q == JK_Q5_K && i == 2)) pair_swap(w.q[i]);
}

__device__ __forceinline__ long op64(uint32_t lo, uint32_t hi) { return (long)(((unsigned long)hi << 32) | lo); }

// Weight operand of 32-element group 2 j + e of the unit (i8 values, plus BIAS).
template <int Q>
__device__ __forceinline__ long few_wop(const FewW<Q> &w, int j, int e, int kq) {
    uint32_t g[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if constexpr (Q == JK_Q8_0) {
            g[k] = w.q[j][2 * e + k];
        } else if constexpr (Q == JK_Q4_0) {
            // piece 0 of a group is the low nibbles of its 16 bytes, piece 1 the high ones
            g[k] = (w.q[j][2 * e + k] >> (4 * (kq & 1))) & 0x0F0F0F0Fu;
        } else if constexpr (Q == JK_Q4_K || Q == JK_Q5_K) {
            // quarter j, in the pair of q[j / 2]: its low nibbles are group 2 j, its high ones 2 j + 1
            g[k] = (w.q[j >> 1][2 * (j & 1) + k] >> (4 * e)) & 0x0F0F0F0Fu;
            if constexpr (Q == JK_Q5_K) {  // bit n of qh[l] for element l of group n
                const uint32_t h = (kq >> 1) ? w.q[2][2 + k] : w.q[2][k];
                const int n = 2 * j + e;
                g[k] |= (n <= 4 ? h << (4 - n) : h >> (n - 4)) & 0x10101010u;
            }
        } else {
            // Q6_K: quarter qq of half j / 2: ql pieces of quarter qq % 2 (the pair of q[j / 2]), low
            // nibbles for qq < 2, and bits 2 qq, 2 qq + 1 of qh (the pair of q[2] is the two halves)
            const int qq = 2 * (j & 1) + e;
            const uint32_t l = w.q[j >> 1][2 * e + k], h = w.q[2][2 * (j >> 1) + k];
            g[k] = ((l >> (4 * (j & 1))) & 0x0F0F0F0Fu) | ((qq < 2 ? h << (4 - 2 * qq) : h >> (2 * qq - 4)) & 0x30303030u);
        }
    }
    return op64(g[0], g[1]);
}

// The lane's weight scales (and mins) for the scale-product MFMAs: MFMA s covers groups NP blk + s
// in its blocks blk = 0..3, and lane kq supplies block kq.
template <int Q>
__device__ __forceinline__ void few_scales(const FewW<Q> &w, int kq, float (&ws)[FewFmt<Q>::NP], float (&wm)[2]) {
    if constexpr (FewFmt<Q>::B32) {
        ws[0] = f16_finite(w.d[0]);
        ws[1] = f16_finite(w.d[1]);
    } else if constexpr (Q == JK_Q6_K) {
        const float d = f16_finite(w.d[0]);
#pragma unroll
        for (int s = 0; s < 4; ++s) ws[s] = d * (float)(int8_t)(w.d[1] >> (8 * s));
    } else {
        // unpack_k4_scales_mins (repack.rs:1158-1170), groups 2 kq and 2 kq + 1
        const uint32_t x = w.hd[0], y = w.hd[1], z = w.hd[2], v = w.hd[3];
        const float d = f16_finite(x & 0xFFFFu), dmin = f16_finite(x >> 16);
        const uint32_t lo = (uint32_t)((kq >> 1) - 1);  // all ones for kq < 2 (a mask: no branch)
        const uint32_t sc = (lo & y & 0x3F3F3F3Fu) | (~lo & ((v & 0x0F0F0F0Fu) | ((y >> 2) & 0x30303030u)));
        const uint32_t mv = (lo & z & 0x3F3F3F3Fu) | (~lo & (((v >> 4) & 0x0F0F0F0Fu) | ((z >> 2) & 0x30303030u)));
        const int sh = 16 * (kq & 1);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            ws[s] = d * (float)((sc >> (sh + 8 * s)) & 255u);
            wm[s] = dmin * (float)((mv >> (sh + 8 * s)) & 255u);
        }
    }
}

// The terms of one unit for one 16 x 16 tile: t[s][4 j + i] of group NP j + s.
template <int Q>
__device__ __forceinline__ void few_terms(FewW<Q> &W, FewX &X, int kq, v16f (&t)[FewFmt<Q>::NP]) {
    using F = FewFmt<Q>;
    constexpr int NP = F::NP;
    float ws[NP];
    [[maybe_unused]] float wm[2];
    few_scales<Q>(W, kq, ws, wm);
    few_swap<Q>(W);
#pragma unroll
    for (int j = 0; j < 4; ++j) pair_swap(X.q[j]);
#pragma unroll
    for (int s = 0; s < NP; ++s) {
        // groups NP j + s: 32-element group 2 j + e, for 16-element groups its piece `part`
        const int e = F::G16 ? s >> 1 : s, part = s & 1;
        v16f pm;
        t[s] = __builtin_amdgcn_mfma_f32_16x16x1f32(ws[s], e ? X.s.y : X.s.x, v16f{0}, 0, 0, 0);
        if constexpr (F::MINS) pm = __builtin_amdgcn_mfma_f32_16x16x1f32(wm[s], s ? X.m.y : X.m.x, v16f{0}, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            long xv = op64(X.q[j][2 * e], X.q[j][2 * e + 1]);
            // 16-element groups: the K = 32 MFMA with the other piece's lanes zeroed
            if constexpr (F::G16) xv = (kq & 1) == part ? xv : 0l;
            v4i c = v4i{0, 0, 0, 0};
            if constexpr (F::BIAS != 0) {
                constexpr uint32_t bb = (uint32_t)((256 - F::BIAS) & 255) * 0x01010101u;
                c = __builtin_amdgcn_mfma_i32_16x16x32_i8(op64(bb, bb), xv, c, 0, 0, 0);
            }
            c = __builtin_amdgcn_mfma_i32_16x16x32_i8(few_wop<Q>(W, j, e, kq), xv, c, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float p = (float)c[i] * t[s][4 * j + i];
                if constexpr (F::MINS) p = p - pm[4 * j + i];
                t[s][4 * j + i] = p;
            }
        }
        // the terms are in registers before the wait for the unit's turn (left to itself the
        // compiler sinks their arithmetic past it, into the chain)
        asm volatile("" : "+v"(t[s]));
    }
}

// Tolerance mode: one unit of one tile into 16 accumulators, acc[4 j + i] taking the groups NP j + s:
// acc = fma(f32(dot), xs * ws, acc), and the mins' -(xsum * wm) through the outer-product MFMA
// accumulating into the same registers.
template <int Q>
__device__ __forceinline__ void few_accumulate(FewW<Q> &W, FewX &X, int kq, v16f &acc, int ng) {
    using F = FewFmt<Q>;
    constexpr int NP = F::NP;
    float ws[NP];
    [[maybe_unused]] float wm[2];
    few_scales<Q>(W, kq, ws, wm);
    few_swap<Q>(W);
#pragma unroll
    for (int j = 0; j < 4; ++j) pair_swap(X.q[j]);
#pragma unroll
    for (int s = 0; s < NP; ++s) {
        const int e = F::G16 ? s >> 1 : s, part = s & 1;
        // (a group past the row's end, in the partial last unit, has no weight: its scale is dropped)
        if (F::B32) ws[s] = NP * kq + s < ng ? ws[s] : 0.0f;
        const v16f p = __builtin_amdgcn_mfma_f32_16x16x1f32(ws[s], e ? X.s.y : X.s.x, v16f{0}, 0, 0, 0);
        if constexpr (F::MINS) acc = __builtin_amdgcn_mfma_f32_16x16x1f32(-wm[s], s ? X.m.y : X.m.x, acc, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            long xv = op64(X.q[j][2 * e], X.q[j][2 * e + 1]);
            if constexpr (F::G16) xv = (kq & 1) == part ? xv : 0l;
            v4i c = v4i{0, 0, 0, 0};
            if constexpr (F::BIAS != 0) {
                constexpr uint32_t bb = (uint32_t)((256 - F::BIAS) & 255) * 0x01010101u;
                c = __builtin_amdgcn_mfma_i32_16x16x32_i8(op64(bb, bb), xv, c, 0, 0, 0);
            }
            c = __builtin_amdgcn_mfma_i32_16x16x32_i8(few_wop<Q>(W, j, e, kq), xv, c, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[4 * j + i] = __builtin_fmaf((float)c[i], p[4 * j + i], acc[4 * j + i]);
        }
    }
}

// KW: waves along K (1, or KU: one unit of a chunk each)
template <int Q, int RW, int TW, int KU, int KW, bool TOL>
__global__ __launch_bounds__(64 * RW * TW * KW) void gemm_few_kernel(WeightDev w, jk_act_q8 a, float *__restrict__ y,
                                                                     int r0, int r1) {
    using F = FewFmt<Q>;
    using St = FewStage<Q, RW, TW, KU>;
    static_assert(KW == 1 || KW == KU, "waves along K");
    constexpr int NG = F::NG, NP = F::NP;
    __shared__ St st[2];
    __shared__ __align__(16) v4f s_acc[KW > 1 ? RW * TW : 1][64];  // running sums of each 16 x 16 tile
    __shared__ int s_turn[RW * TW];                   // units whose terms have been added to them
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int jl = lane & 15, kq = lane >> 4;
    const int kw = wave / (RW * TW), tile = wave % (RW * TW), rw = tile % RW, tw = tile / RW;
    // an eighth of the tiles per XCD (workgroup i runs on XCD i % 8), a row tile's token tiles together
    // (whole row tiles per XCD left XCDs idle or a round behind: Q5_K 1603 x 14336, 1564 tokens 480 us, now
    // 349; Q8_0 731 x 1024, 1111 tokens 16.6 us, now 9.4)
    const int ntn = (r1 - r0 + 16 * RW - 1) / (16 * RW), ntm = ((int)a.m + 16 * TW - 1) / (16 * TW);
    const int wg = (int)blockIdx.x, t = (wg & 7) * ((int)gridDim.x >> 3) + (wg >> 3);
    if (t >= ntn * ntm) return;  // workgroup-uniform
    const int tn = t / ntm, tm = t % ntm;
    const int n0 = r0 + 16 * RW * tn, m0 = 16 * TW * tm, M = (int)a.m;
    const int steps = w.cols / 32, units = (steps + 7) / 8, nchunks = (units + KU - 1) / KU;
    const int row = 16 * rw + jl, tok = 16 * tw + jl;
    v4f acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    [[maybe_unused]] v16f tacc = v16f{0};

    auto add = [&](const v16f(&t)[NP], int u) {
        const int ng = min(8, steps - 8 * u) * (NG / 8);  // groups of this unit (a partial last unit: fewer)
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            if (F::B32 && g >= ng) break;  // (256-element blocks: whole units only)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += t[g % NP][4 * (g / NP) + i];
        }
    };
    auto unit = [&](const St &S, int u, int v) {
        FewW<Q> W;
        FewX X;
        [[maybe_unused]] const int dodd = (int)(((size_t)min(n0 + row, r1 - 1) * (size_t)w.nb + (size_t)(u - v)) & 1);
        few_wread(W, S, row, v, kq, dodd);
        few_xread(X, S, tok, v, kq);
        if constexpr (TOL) {
            few_accumulate<Q>(W, X, kq, tacc, steps - 8 * u);
            return;
        }
        v16f t[NP];
        few_terms<Q>(W, X, kq, t);
        if constexpr (KW == 1) {
            add(t, u);
            return;
        }
        // this unit's turn: the sums of units 0 .. u - 1, then its terms in group order. The LDS
        // executes a wave's accesses in order, so sums read after the turn's value are the ones
        // that were written before it.
        if (u > 0) {
            int turn;
            do {
                turn = *(volatile lds_int_t *)&s_turn[tile];
                acc = *(volatile lds_v4f_t *)&s_acc[tile][lane];
            } while (__builtin_amdgcn_readfirstlane(turn) != u);
        }
        add(t, u);
        if (u + 1 < units) {
            *(volatile lds_v4f_t *)&s_acc[tile][lane] = acc;
            *(volatile lds_int_t *)&s_turn[tile] = u + 1;  // (every lane the same word)
        }
    };

    few_issue<Q, RW, TW, KU, KW>(st[0], w, a, n0, r1, m0, 0, wave, lane);
    if (threadIdx.x < RW * TW) s_turn[threadIdx.x] = 0;
    for (int c = 0; c < nchunks; ++c) {
        // chunk c is in LDS (each wave has waited for its own loads), and every wave is done with the
        // other stage, which is refilled while this one is evaluated (three stages measured the same,
        // and cost a resident workgroup)
        JK_WAIT_VMCNT(0);
        stage_barrier();
        if (c + 1 < nchunks) few_issue<Q, RW, TW, KU, KW>(st[(c + 1) & 1], w, a, n0, r1, m0, c + 1, wave, lane);
        const St &S = st[c & 1];
        if constexpr (KW == 1) {
            for (int v = 0; v < KU; ++v)
                if (KU * c + v < units) unit(S, KU * c + v, v);
        } else {
            if (KU * c + kw < units) unit(S, KU * c + kw, kw);
        }
    }
    if constexpr (TOL) {
        acc = v4f{tacc[0], tacc[1], tacc[2], tacc[3]};
#pragma unroll
        for (int j = 1; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += tacc[4 * j + i];
        if constexpr (KW > 1) {  // the waves' partial tiles, through the first stage's LDS, in wave order
            v4f *part = reinterpret_cast<v4f *>(&st[0]);
            static_assert(sizeof(St) >= KW * RW * TW * 1024, "room for the partial tiles");
            __syncthreads();
            if (kw > 0) part[(kw * RW * TW + tile) * 64 + lane] = acc;
            __syncthreads();
            if (kw > 0) return;
#pragma unroll
            for (int k = 1; k < KW; ++k) {
                const v4f o = part[(k * RW * TW + tile) * 64 + lane];
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] += o[i];
            }
        }
    } else {
        if (KW > 1 && (units - 1) % KU != kw) return;
    }
    // the last unit's wave: lane holds token jl, weight rows 4 kq + i of its tile
    const int m = m0 + tok, n = n0 + 16 * rw + 4 * kq;
    if (m < M) {
        float *dst = y + (size_t)m * (size_t)(r1 - r0) + (size_t)(n - r0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n + i < r1) dst[i] = acc[i];
    }
}

template <int Q, int RW, int TW, int KU, int KW>
static jk_status launch_few_t(hipStream_t s, const WeightDev &w, const jk_act_q8 &a, float *y, int r0, int r1, bool tol) {
    const size_t ntn = (size_t)(r1 - r0 + 16 * RW - 1) / (16 * RW), ntm = (a.m + 16 * TW - 1) / (16 * TW);
    const dim3 grid((unsigned)((ntn * ntm + 7) / 8 * 8)), block(64 * RW * TW * KW);
    if (tol)
        JK_LAUNCH("gemm_few_kernel<tolerance>", (gemm_few_kernel<Q, RW, TW, KU, KW, true>), grid, block, 0, s, w, a, y, r0, r1);
    else
        JK_LAUNCH("gemm_few_kernel", (gemm_few_kernel<Q, RW, TW, KU, KW, false>), grid, block, 0, s, w, a, y, r0, r1);
    return check_launch("gemm_few_kernel");
}

// RW x TW (x K waves) by the number T of 16 x 16 output tiles (us, bit-exact, Q4_K x 4096 columns
// unless said): one tile and eight K waves a workgroup while every CU has at most one (1024 rows, 16
// tokens 7.1 against 8.7 on 2x1x4; 4096 rows 8.2 against 10.0); two row tiles and four K waves up to
// four tiles per CU (14336 rows, 16 tokens 15.7 against 20.9 on 1x1x4, 23.9 on 2x2x4), with two token
// tiles where there are two and two tiles per CU already (4096 rows, 64 tokens 12.8 against 14.0);
// two K waves up to ten (1024 rows, 512 tokens 20.1 against 22.3 on 2x2x4, 21.6 unsplit); beyond,
// tiles enough for unsplit K (4096 rows, 512 tokens 64.3 against 70.7 on 2x2x2), except for
// Q6_K, whose 16 groups a unit make the longer serial stretch (4096 x 14336, 512 tokens 334 on 2x2x2
// against 409). Unsplit, a workgroup takes all of 33 to 64 tokens (14336 rows, 33 tokens 29.6 against
// 36.6 on two token tiles); Q8_0's larger weight stages are shared by four token tiles (14336
// rows, 128 tokens 53.6 against 72.4), and at few tiles it takes two K waves (16 tokens 15.7
// against 20.9).
enum FewShape { kFew1x1x8, kFew2x1x4, kFew2x2x4, kFew2x2x2, kFew4x2, kFew4x3, kFew4x4 };
static FewShape few_shape(int quant, long rows, long m, long ncu) {
    const long tm = (m + 15) / 16, T = (rows + 15) / 16 * tm;
    if (T <= ncu) return kFew1x1x8;
    if (T <= 4 * ncu) return tm == 1 || T <= 2 * ncu ? kFew2x1x4 : kFew2x2x4;
    if (T <= 10 * ncu || quant == JK_Q6_K) return kFew2x2x2;
    if (tm == 3) return kFew4x3;
    return tm == 4 || quant == JK_Q8_0 ? kFew4x4 : kFew4x2;
}

long gemm_few_workgroups(int quant, long rows, long m, long ncu) {
    static constexpr int kRows[] = {16, 32, 32, 32, 64, 64, 64}, kTokens[] = {16, 16, 32, 32, 32, 48, 64};
    const FewShape f = few_shape(quant, rows, m, ncu);
    return (rows + kRows[f] - 1) / kRows[f] * ((m + kTokens[f] - 1) / kTokens[f]);
}

template <int Q>
static jk_status launch_few_q(hipStream_t s, const WeightDev &w, const jk_act_q8 &a, float *y, int r0, int r1, long ncu,
                              bool tol) {
    switch (few_shape(w.quant, r1 - r0, (long)a.m, ncu)) {
    case kFew1x1x8: return launch_few_t<Q, 1, 1, 8, 8>(s, w, a, y, r0, r1, tol);
    case kFew2x1x4:
        if constexpr (Q == JK_Q8_0) return launch_few_t<Q, 2, 1, 2, 2>(s, w, a, y, r0, r1, tol);
        else return launch_few_t<Q, 2, 1, 4, 4>(s, w, a, y, r0, r1, tol);
    case kFew2x2x4: return launch_few_t<Q, 2, 2, 4, 4>(s, w, a, y, r0, r1, tol);
    case kFew2x2x2: return launch_few_t<Q, 2, 2, 2, 2>(s, w, a, y, r0, r1, tol);
    case kFew4x2:
        if constexpr (Q != JK_Q6_K && Q != JK_Q8_0) return launch_few_t<Q, 4, 2, 2, 1>(s, w, a, y, r0, r1, tol);
        break;
    case kFew4x3:
        if constexpr (Q != JK_Q6_K) return launch_few_t<Q, 4, 3, 2, 1>(s, w, a, y, r0, r1, tol);
        break;
    default:
        if constexpr (Q != JK_Q6_K) return launch_few_t<Q, 4, 4, 2, 1>(s, w, a, y, r0, r1, tol);
        break;
    }
    return fail(JK_DEVICE_ERROR, "gemm: no few-tile launch of quant %d", w.quant);  // (few_shape gives none of these)
}

bool gemm_few_ok(const WeightDev &w, const jk_act_q8 &a) {
    switch (w.quant) {
    case JK_Q8_0:
    case JK_Q4_0:
        if (w.nb % 2) return false;  // the scale plane is read by dwords
        break;
    case JK_Q4_K:
    case JK_Q5_K:
    case JK_Q6_K: break;
    default: return false;
    }
    return a.m >= 3 && (uintptr_t)a.qs % 16 == 0 && a.k_padded == (size_t)w.cols && a.k_blocks32 == (size_t)w.cols / 32;
}

jk_status launch_gemm_few(hipStream_t s, const WeightDev &w, const jk_act_q8 &a, float *y, int r0, int r1, long ncu,
                          bool tol) {
    switch (w.quant) {
    case JK_Q8_0: return launch_few_q<JK_Q8_0>(s, w, a, y, r0, r1, ncu, tol);
    case JK_Q4_0: return launch_few_q<JK_Q4_0>(s, w, a, y, r0, r1, ncu, tol);
    case JK_Q4_K: return launch_few_q<JK_Q4_K>(s, w, a, y, r0, r1, ncu, tol);
    case JK_Q5_K: return launch_few_q<JK_Q5_K>(s, w, a, y, r0, r1, ncu, tol);
    case JK_Q6_K: return launch_few_q<JK_Q6_K>(s, w, a, y, r0, r1, ncu, tol);
    default: return fail(JK_CAPABILITY_MISMATCH, "gemm: unsupported quant %d", w.quant);
    }
}

}  // namespace jk
