// jk_gemm_split.hip -- tolerance-mode repacked GEMM of Q4_K and Q5_K for launches that fill the GPU.
//
// The other tolerance kernels multiply whole numbers and scale each 32-element group's sum by xs * ws,
// a product per output and group that costs an f32 MFMA (which no VALU work of its wave overlaps) beside
// the VALU's multiply-add, and another MFMA for the mins. Here the weight's 6-bit group scale goes into
// its operand: q * sc is at most 15 * 63 (Q4_K) or 31 * 63 (Q5_K), exact in f16, as the i8 activations
// are, and a group's sum of 32 products stays below 2^24, exact in the MFMA's f32. A lane of the result
// holds one token, so what is left per output and group is
//     part = fma(sum, xs, part)
// and per 256-element block acc = fma(d, part, acc) and the mins, acc = fma(-dmin, sum(xsum * mn), acc),
// whose sums over the 8 groups are two bf16 MFMAs: xsum as three bf16 numbers (24 bits), mn exact.
//
// Formed before d and dmin come in, a block's sums can pass f32's range where the outputs do not: they
// reach 2^12 times its xs (with the operands' 2^-14) and 2^9 times its xsum. Both are taken times 2^-13,
// which d and dmin give back, so that no finite xs or xsum overflows; the quantizer's xs are zero or
// at least 1e-30 / 127, far enough from f32's smallest.
//
// A workgroup owns 256 weight rows x 128 tokens, a wave 32 x 128. Weights go from global memory straight
// into one of two LDS stages a 256-element block ahead, activations through registers a 64-element
// quarter ahead, converted to f16 once per workgroup; a wave unpacks the weights that it multiplies.
//
// What bounds it: each wave's own chain, LDS read -> MFMA -> multiply-adds, one tile deep, at two waves a
// SIMD and a workgroup barrier every 64 elements. Counted at 14336 x 4096, 2048 tokens: the VALU is busy 53%
// of the cycles (2.2 instructions per output and group, of which the multiply-add is one; unpacking,
// converting and the blocks' ends are the rest), the matrix cores 27%, the LDS 39% (a third of it bank
// conflicts), and a wave waits a third of its time. 14336 x 4096, Q4_K: 2048 tokens 443 us (543 TOPS) against
// 533 us on the 128 x 128 tiles (launched back to back; 485 us and more under a profiler), 512 tokens 130
// against 167 us, and the error against 64 bits 1.7e-7 against 3.1e-7. Timed with work left out: loading no
// weights 408 us. (The weights' loads are asm that the compiler does not count, so its wait for the
// activations' loads, two tiles into a quarter, waits for the quarter's weights too: more than needed, never
// less. The explicit wait at a block's end is for all of them.)
// Also tried, both with the activation scales in the operands (x * xs as two f16 numbers, no multiply-add
// per group): 552 us, the conversion and twice the MFMAs taking more than they save, and 565 us with its
// MFMAs and VALU work interleaved by hand. What made it fast: each tile's sum pinned where it is added (the
// compiler otherwise sinks the adds, keeps the products and spills 130 registers), and a quarter's last
// tile added after the barrier, while the next quarter's operands are read (466 us without).
#include "jk_device.hpp"

namespace jk {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

constexpr int kSplitN = 256, kSplitM = 128, kSplitThreads = 512;
constexpr float kSplitDown = 0x1p-13f, kSplitUp = 0x1p13f;

template <int Q> struct alignas(16) SplitLds {
    static constexpr int P = fmt_of(Q).chunks;
    uint8_t x[2][kSplitM][128];         // [stage][token]: 8 16-byte pieces of f16, XORed with the token
    float xs[2][kSplitM][8];            // [block & 1][token][group], times 2^-13
    uint16_t xm[2][4][kSplitM][8];      // the groups' sums times 2^-13 in three bf16 parts, and zeros
    float d[kSplitN], dm[kSplitN];      // the rows' 2^27 d and 2^13 dmin
    uint8_t w[2][P][kSplitN][16];       // [stage][plane][row] (last: the others within an instruction's offset)
};

__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ h8 op8(h2 a, h2 b, h2 c, h2 d) { return h8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]}; }

template <int Q>
__global__ __launch_bounds__(kSplitThreads) __attribute__((amdgpu_waves_per_eu(2))) void
gemm_split_kernel(WeightDev w, jk_act_q8 a, float *__restrict__ y, int r0, int r1, int vec) {
    using S = SplitLds<Q>;
    constexpr int Q0 = Q == JK_Q5_K ? 3 : 1;
    constexpr int NWI = S::P * kSplitN / 64, NWL = (NWI + 7) / 8;  // weight loads of a block, and a wave's
    __shared__ S L;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ntn = (r1 - r0 + kSplitN - 1) / kSplitN, ntm = ((int)a.m + kSplitM - 1) / kSplitM;
    // an eighth of the tiles per XCD (workgroup i runs on XCD i % 8), a row tile's token tiles together
    // (whole row tiles per XCD leave some XCDs a round more: 11008 rows, 1300 tokens 319 us)
    const int wg = (int)blockIdx.x, tile = (wg & 7) * ((int)gridDim.x >> 3) + (wg >> 3);
    if (tile >= ntn * ntm) return;  // workgroup-uniform
    const int tn = tile / ntm, tm = tile % ntm;
    const int n0 = r0 + kSplitN * tn, m0 = kSplitM * tm, M = (int)a.m, nb = w.nb, nsteps = 4 * nb;
    const int row0 = 32 * wave;
    // LDS addresses are rebuilt in every quarter from a thread index that the compiler cannot see
    // through: kept across the loop they would not fit the registers
    int tv = tid;
    auto jl = [&] { return tv & 31; };        // weight row of an operand, token of a result
    auto hf = [&] { return (tv >> 5) & 1; };  // half of a 32-element group

    // activations: the thread's token and 16 of a quarter's 64 bytes (rows past the end are clamped)
    const int xtok = tid >> 2, part = tid & 3;
    const uint32_t xrow = (uint32_t)min(xtok, M - 1 - m0);
    const uint32_t xqo = xrow * (uint32_t)a.k_padded + 16u * (uint32_t)part;
    const uint32_t xso = (xrow * (uint32_t)a.k_blocks32 + 2u * (uint32_t)part) * 4u;
    const int8_t *xqb = a.qs + (size_t)m0 * a.k_padded;
    const float *xsb = a.scales + (size_t)m0 * a.k_blocks32, *xmb = a.sums + (size_t)m0 * a.k_blocks32;
    auto xload = [&](int s) { return *reinterpret_cast<const u32x4 *>(xqb + 64 * min(s, nsteps - 1) + xqo); };
    auto sload = [&](const float *base, int b) {
        return *reinterpret_cast<const float2 *>(reinterpret_cast<const char *>(base + 8 * b) + xso);
    };
    // constants that v_and_or_b32 and v_bitop3_b32 take from registers (opaque, or the compiler splits
    // each use into two instructions with a literal)
    uint32_t k6400 = 0x64006400u, k6480 = 0x64806480u;
    asm("" : "+v"(k6400), "+v"(k6480));
    // dwords 2 i, 2 i + 1 of the thread's bytes to f16 (elements 0 2 1 3 of a dword), piece 2 part + i
    auto xconv = [&](const u32x4 &raw, int stage, int i) {
        h2 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)  // (byte ^ 0x80 with f16's exponent: 1024 + 128 + x)
            v[k] = as_h2(((raw[2 * i + (k >> 1)] >> (8 * (k & 1))) & 0x00FF00FFu) ^ k6480) -
                   h2{(_Float16)1152, (_Float16)1152};
        *reinterpret_cast<h8 *>(&L.x[stage][(tv >> 2)][16 * ((2 * (tv & 3) + i) ^ (((tv >> 2) >> 1) & 7))]) = op8(v[0], v[1], v[2], v[3]);
    };
    // the token's scales and sums of groups 2 part, 2 part + 1 of block b
    auto sstore = [&](float2 fs, float2 fm, int b) {
        *reinterpret_cast<float2 *>(&L.xs[b & 1][(tv >> 2)][2 * (tv & 3)]) = float2{fs.x * kSplitDown, fs.y * kSplitDown};
        float v0 = fm.x * kSplitDown, v1 = fm.y * kSplitDown;
#pragma unroll
        for (int k = 0; k < 3; ++k) {  // (truncated to 8 bits each: the differences are exact)
            const uint32_t c0 = __float_as_uint(v0) & 0xFFFF0000u, c1 = __float_as_uint(v1) & 0xFFFF0000u;
            *reinterpret_cast<uint32_t *>(&L.xm[b & 1][k][(tv >> 2)][2 * (tv & 3)]) = (c0 >> 16) | c1;
            // (nothing is left of an infinite sum, whose difference from itself is NaN)
            v0 = __builtin_isinf(v0) ? 0.0f : v0 - __uint_as_float(c0);
            v1 = __builtin_isinf(v1) ? 0.0f : v1 - __uint_as_float(c1);
        }
    };
    // this wave's share of the weight loads: plane wave / 4 + 2 i, 64 rows
    const uint32_t wvo = (uint32_t)min(64 * (wave & 3) + lane, r1 - 1 - n0) * (uint32_t)nb * 16u;
    auto wload = [&](int b, int i) {
        if (wave + 8 * i >= NWI) return;  // wave-uniform
        const uint8_t *src = w.planes + (((size_t)((wave >> 2) + 2 * i) * (size_t)w.rows + (size_t)n0) * (size_t)nb +
                                         (size_t)b) * 16;
        asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(wvo), "s"(src),
                     "{m0}"((unsigned)(size_t)((lds_u8_t *)&L.w[b & 1][(wave >> 2) + 2 * i][64 * (wave & 3)][0]))
                     : "memory");
    };

    h2 ws[4];  // the row's group scales in pairs (0, 2), (1, 3), (4, 6), (5, 7), times 2^10, odd groups' 2^6
    b8 mn;     // and its mins
    // unpack_k4_scales_mins (repack.rs:1158-1170)
    auto header = [&](int b) {
        const u32x4 hd = *reinterpret_cast<const u32x4 *>(L.w[b & 1][0][row0 + jl()]);
        const uint32_t s0 = hd[1] & 0x3F3F3F3Fu, s1 = (hd[3] & 0x0F0F0F0Fu) | ((hd[1] >> 2) & 0x30303030u);
        const uint32_t m0w = hd[2] & 0x3F3F3F3Fu, m1w = ((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] >> 2) & 0x30303030u);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const _Float16 f = (_Float16)(k & 1 ? 64 : 1024);
            ws[k] = (as_h2((((k >> 1 ? s1 : s0) >> (8 * (k & 1))) & 0x00FF00FFu) | k6400) -
                     h2{(_Float16)1024, (_Float16)1024}) * h2{f, f};
        }
        uint32_t mv[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t m2 = (k >> 1 ? m1w : m0w) >> (16 * (k & 1));
            mv[k] = (__float_as_uint((float)(m2 & 255u)) >> 16) | (__float_as_uint((float)((m2 >> 8) & 255u)) & 0xFFFF0000u);
        }
        mn = __builtin_bit_cast(b8, u32x4{mv[0], mv[1], mv[2], mv[3]});
    };
    // weight operand of 8 elements: group 2 j + e, elements 16 hf + 8 i .. of it (times 2^-14)
    auto unpack = [&](const u32x4 &q, const u32x4 &qh, int j, int e, int i) {
        const h2 wp = ws[2 * (j >> 1) + e];
        const h2 sv = j & 1 ? h2{wp[1], wp[1]} : h2{wp[0], wp[0]};
        h2 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t u = (q[2 * i + (k >> 1)] >> (8 * (k & 1))) & (e ? 0x00F000F0u : 0x000F000Fu);
            if constexpr (Q == JK_Q5_K) {  // bit n of qh's byte to bit 4 (or 8) of the quant's
                const int n = 2 * j + e, at = n + 8 * (k & 1) - (e ? 8 : 4);
                const uint32_t hv = qh[2 * i + (k >> 1)];
                u |= (at >= 0 ? hv >> (at & 31) : hv << (-at & 31)) & (e ? 0x01000100u : 0x00100010u);
            }
            v[k] = as_h2(u) * sv;  // (as an f16 number the quant is q * 2^-24, or 2^-20: denormal, exact)
        }
        return op8(v[0], v[1], v[2], v[3]);
    };
    // activation operand: token 32 t + jl, group e of the quarter, elements 16 hf + 8 i ..
    uint32_t xbase;
    auto bread = [&](int stage, int t, int e, int i) {
        return *reinterpret_cast<const h8 *>(&L.x[stage][32 * t][0] + (xbase ^ (uint32_t)(16 * (4 * e + i))));
    };

    float acc[4][16], sum[4][16];
#pragma unroll
    for (int i = 0; i < 64; ++i) acc[i >> 4][i & 15] = 0.0f;
    h8 A[2], B[3][2];
    v16f P[2];
    float2 xs[4], xn[4];  // the lane's tokens' scales of a quarter's two groups, and the next quarter's
    float xlast = 0.0f;
    u32x4 q, qh;
    auto qread = [&](int b, int j) {
        q = *reinterpret_cast<const u32x4 *>(L.w[b & 1][Q0 + 2 * j + hf()][row0 + jl()]);
        if constexpr (Q == JK_Q5_K) qh = *reinterpret_cast<const u32x4 *>(L.w[b & 1][1 + hf()][row0 + jl()]);
        else qh = q;
    };
    auto xsread = [&](int b, int j) {
#pragma unroll
        for (int t = 0; t < 4; ++t) xn[t] = *reinterpret_cast<const float2 *>(&L.xs[b & 1][32 * t + jl()][2 * j]);
    };
    auto add = [&](int p, int t, float x, bool first) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            sum[t][i] = first ? P[p][i] * x : __builtin_fmaf(P[p][i], x, sum[t][i]);
            asm volatile("" : "+v"(sum[t][i]));  // (added here: not sunk into a later block)
        }
    };

    u32x4 raw = xload(0);
    float2 fs = sload(xsb, 0), fm = sload(xmb, 0);
    sstore(fs, fm, 0);
    xconv(raw, 0, 0);
    xconv(raw, 0, 1);
    *reinterpret_cast<uint32_t *>(&L.xm[0][3][(tv >> 2)][2 * (tv & 3)]) = 0;
    *reinterpret_cast<uint32_t *>(&L.xm[1][3][(tv >> 2)][2 * (tv & 3)]) = 0;
    raw = xload(1);
#pragma unroll
    for (int i = 0; i < NWL; ++i) wload(0, i);
    JK_WAIT_VMCNT(0);
    stage_barrier();

    for (int b = 0; b < nb; ++b) {
        header(b);
        const int bn = min(b + 1, nb - 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int s = 4 * b + j;
            auto bread2 = [&](int u) {
                B[u % 3][0] = bread(s & 1, u & 3, u >> 2, 0);
                B[u % 3][1] = bread(s & 1, u & 3, u >> 2, 1);
            };
            asm volatile("" : "+v"(tv));
            xbase = (uint32_t)(128 * jl() + 16 * ((2 * hf()) ^ ((jl() >> 1) & 7)));
            if (j < 3 && b + 1 < nb)
#pragma unroll
                for (int i = j * NWL / 3; i < (j + 1) * NWL / 3; ++i) wload(b + 1, i);
            if (j == 0) {
                fs = sload(xsb, bn);
                fm = sload(xmb, bn);
            }
            if (j == 1 && wave < kSplitN / 64) {  // (the last block's have been read)
                const uint32_t dd = *reinterpret_cast<const uint32_t *>(L.w[b & 1][0][tv]);
                L.d[tv] = 16384.0f * kSplitUp * f16_finite(dd & 0xFFFFu);
                L.dm[tv] = kSplitUp * f16_finite(dd >> 16);
            }
            if (j == 2) sstore(fs, fm, b + 1);
            if (j == 0) {
                qread(b, 0);
                xsread(b, 0);
            }
            bread2(0);
            bread2(1);
            A[0] = unpack(q, qh, j, 0, 0);
            A[1] = unpack(q, qh, j, 0, 1);
            if (j > 0) add(1, 3, xlast, false);  // (the quarter before's last tile: its MFMAs ran into the barrier)
#pragma unroll
            for (int t = 0; t < 4; ++t) xs[t] = xn[t];
            // tile u % 4 of group u / 4: its MFMAs run while the tile before is added up
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (u == 4) {
                    A[0] = unpack(q, qh, j, 1, 0);
                    A[1] = unpack(q, qh, j, 1, 1);
                }
                P[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[0], B[u % 3][0], v16f{0}, 0, 0, 0);
                P[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[1], B[u % 3][1], P[u & 1], 0, 0, 0);
                if (u < 6) bread2(u + 2);
                if (u == 2) xconv(raw, (s + 1) & 1, 0);  // (past the last quarter: written, never used)
                if (u == 3) {
                    xconv(raw, (s + 1) & 1, 1);
                    raw = xload(s + 2);
                }
                if (u == 5 && j < 3) {
                    qread(b, j + 1);
                    xsread(b, j + 1);
                }
                if (u > 0) add((u - 1) & 1, (u - 1) & 3, (u - 1) >> 2 ? xs[(u - 1) & 3].y : xs[(u - 1) & 3].x, j == 0 && u <= 4);
                __builtin_amdgcn_sched_barrier(0);  // (or the compiler runs MFMAs ahead and spills)
            }
            xlast = xs[3].y;
            if (j == 3) add(1, 3, xlast, false);
            if (j == 3) {
                v16f mm[2];
                auto minsum = [&](int t) {
                    const int tok = 32 * t + jl();
                    const v16f c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        mn, *reinterpret_cast<const b8 *>(L.xm[b & 1][hf()][tok]), v16f{0}, 0, 0, 0);
                    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        mn, *reinterpret_cast<const b8 *>(L.xm[b & 1][2 + hf()][tok]), c, 0, 0, 0);
                };
                mm[0] = minsum(0);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    if (t < 3) mm[(t + 1) & 1] = minsum(t + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int rr = row0 + 8 * k + 4 * hf();
                        const float4 d4 = *reinterpret_cast<const float4 *>(&L.d[rr]);
                        const float4 m4 = *reinterpret_cast<const float4 *>(&L.dm[rr]);
                        const float dv[4] = {d4.x, d4.y, d4.z, d4.w}, mv[4] = {m4.x, m4.y, m4.z, m4.w};
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float c = acc[t][4 * k + i];
                            c = __builtin_fmaf(dv[i], sum[t][4 * k + i], c);
                            acc[t][4 * k + i] = __builtin_fmaf(-mv[i], mm[t & 1][4 * k + i], c);
                        }
                    }
                }
                JK_WAIT_VMCNT(0);  // the next block's weights
            }
            stage_barrier();
        }
    }

    const size_t R = (size_t)(r1 - r0);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int m = m0 + 32 * t + jl();
        if (m >= M) continue;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int n = n0 + row0 + 8 * k + 4 * hf();
            float *dst = y + (size_t)m * R + (size_t)(n - r0);
            const float(&c)[16] = acc[t];
            if (vec && n + 3 < r1) {
                *reinterpret_cast<float4 *>(dst) = float4{c[4 * k], c[4 * k + 1], c[4 * k + 2], c[4 * k + 3]};
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < r1) dst[i] = c[4 * k + i];
            }
        }
    }
}

bool gemm_split_ok(const WeightDev &w, const jk_act_q8 &a) {
    return (w.quant == JK_Q4_K || w.quant == JK_Q5_K) && (uintptr_t)a.qs % 16 == 0 && (uintptr_t)a.scales % 8 == 0 &&
           (uintptr_t)a.sums % 8 == 0 && a.k_padded == (size_t)w.cols && a.k_blocks32 == (size_t)w.cols / 32;
}

jk_status launch_gemm_split(hipStream_t s, const WeightDev &w, const jk_act_q8 &a, float *y, int r0, int r1) {
    const size_t ntn = (size_t)(r1 - r0 + kSplitN - 1) / kSplitN, ntm = (a.m + kSplitM - 1) / kSplitM;
    const dim3 grid((unsigned)((ntn * ntm + 7) / 8 * 8)), block(kSplitThreads);
    const int vec = (r1 - r0) % 4 == 0 && (uintptr_t)y % 16 == 0;
    if (w.quant == JK_Q4_K) JK_LAUNCH("gemm_split_kernel", gemm_split_kernel<JK_Q4_K>, grid, block, 0, s, w, a, y, r0, r1, vec);
    else JK_LAUNCH("gemm_split_kernel", gemm_split_kernel<JK_Q5_K>, grid, block, 0, s, w, a, y, r0, r1, vec);
    return check_launch("gemm_split_kernel");
}

}  // namespace jk
