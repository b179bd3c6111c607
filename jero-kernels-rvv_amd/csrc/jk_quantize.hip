// jk_quantize.hip -- activation quantizers, bit-exact with the reference recipes.
//
// Maxima are order-independent, so they are reduced across lanes; sums that the
// reference accumulates in f32 are accumulated sequentially in one lane in the
// reference's order; integer sums are reduced across lanes.
#include <type_traits>

#include "jk_device.hpp"

namespace jk {

// quantize_block_q8_0_scalar (quant_q8.rs:203-219): 32 lanes per block, one element each.
__global__ __launch_bounds__(256) void quantize_q8_0_kernel(const float *__restrict__ x, size_t nblocks,
                                                            jk_block_q8_0 *__restrict__ out) {
    const size_t blk = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) >> 5;
    const int l = threadIdx.x & 31;
    const bool live = blk < nblocks;
    const float v = live ? x[blk * 32 + l] : 0.0f;
    const float amax = wave_max<32>(__builtin_isfinite(v) ? fabsf(v) : 0.0f);
    if (!live) return;
    if (amax == 0.0f || !__builtin_isfinite(amax)) {
        out[blk].qs[l] = 0;
        if (l == 0) out[blk].d = 0.0f;
        return;
    }
    const float inv = 127.0f / amax;
    out[blk].qs[l] = (int8_t)round_scaled_to_i8(v, inv);
    if (l == 0) out[blk].d = amax / 127.0f;
}

jk_status launch_quantize_q8_0(hipStream_t s, const float *x, size_t nblocks, jk_block_q8_0 *out) {
    const size_t threads = nblocks * 32;
    hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, x, nblocks, out);
    return check_launch("quantize_q8_0_kernel");
}

// quantize_block_q8_k_scalar (quant_q8.rs:447-475): one wave per block, 4 elements per lane,
// bsums[j] = sum of the 16 quants of lanes 4j..4j+3. With ACT != 0 the input element is the
// gated activation gated<ACT>(x[i], up[i]) (SwiGLU or ReLU^2), computed in the load. V4: the inputs
// are 16-byte aligned and a lane reads its four elements with one load each. The block maximum and
// the bsums are DPP reductions (a maximum and an integer sum: exact in any order), with no LDS
// round trip on the launch's critical path.
template <int ACT, bool V4>
__global__ __launch_bounds__(256) void quantize_q8_k_kernel(const float *__restrict__ x, const float *__restrict__ up,
                                                            size_t nblocks, jk_block_q8k *__restrict__ out) {
    const size_t blk = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int l = threadIdx.x & 63;
    const bool live = blk < nblocks;
    const size_t e0 = min(blk, nblocks - 1) * 256 + 4 * l;  // (clamped: in bounds for every lane)
    float g[4], u[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (V4) {
        const float4 gv = *reinterpret_cast<const float4 *>(x + e0);
        g[0] = gv.x, g[1] = gv.y, g[2] = gv.z, g[3] = gv.w;
        if constexpr (ACT != 0) {
            const float4 uv = *reinterpret_cast<const float4 *>(up + e0);
            u[0] = uv.x, u[1] = uv.y, u[2] = uv.z, u[3] = uv.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            g[i] = x[e0 + i];
            if constexpr (ACT != 0) u[i] = up[e0 + i];
        }
    }
    float v[4];
    float a = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[i] = live ? gated<ACT>(g[i], u[i]) : 0.0f;
        a = fmaxf(a, __builtin_isfinite(v[i]) ? fabsf(v[i]) : 0.0f);
    }
    const float amax = wave_max64_dpp(a);
    int q[4] = {0, 0, 0, 0};
    const bool zero = amax == 0.0f || !__builtin_isfinite(amax);
    if (!zero) {
        const float inv = 127.0f / amax;
        for (int i = 0; i < 4; ++i) q[i] = round_scaled_to_i8(v[i], inv);
    }
    const int part = sum4_dpp(q[0] + q[1] + q[2] + q[3]);
    if (!live) return;
    uint32_t packed = (uint32_t)(q[0] & 255) | ((uint32_t)(q[1] & 255) << 8) | ((uint32_t)(q[2] & 255) << 16) |
                      ((uint32_t)(q[3] & 255) << 24);
    *reinterpret_cast<uint32_t *>(&out[blk].qs[4 * l]) = packed;
    if ((l & 3) == 0) out[blk].bsums[l >> 2] = (int16_t)part;
    if (l == 0) out[blk].d = zero ? 0.0f : amax / 127.0f;
}

jk_status launch_quantize_q8_k(hipStream_t s, const float *x, size_t nblocks, jk_block_q8k *out) {
    return launch_quantize_q8_k_gated(s, kActNone, x, nullptr, nblocks, out);
}

jk_status launch_quantize_q8_k_gated(hipStream_t s, int act, const float *x, const float *up, size_t nblocks,
                                     jk_block_q8k *out) {
    const dim3 grid((unsigned)((nblocks * 64 + 255) / 256)), block(256);
    const bool v4 = (uintptr_t)x % 16 == 0 && (act == kActNone || (uintptr_t)up % 16 == 0);
    if (act == kActSwiglu) {
        if (v4) hipLaunchKernelGGL((quantize_q8_k_kernel<kActSwiglu, true>), grid, block, 0, s, x, up, nblocks, out);
        else hipLaunchKernelGGL((quantize_q8_k_kernel<kActSwiglu, false>), grid, block, 0, s, x, up, nblocks, out);
    } else if (act == kActRelu2) {
        if (v4) hipLaunchKernelGGL((quantize_q8_k_kernel<kActRelu2, true>), grid, block, 0, s, x, up, nblocks, out);
        else hipLaunchKernelGGL((quantize_q8_k_kernel<kActRelu2, false>), grid, block, 0, s, x, up, nblocks, out);
    } else {
        if (v4) hipLaunchKernelGGL((quantize_q8_k_kernel<kActNone, true>), grid, block, 0, s, x, up, nblocks, out);
        else hipLaunchKernelGGL((quantize_q8_k_kernel<kActNone, false>), grid, block, 0, s, x, up, nblocks, out);
    }
    return check_launch("quantize_q8_k_kernel");
}

// Ordered f32 fold of N consecutive lanes (N = 4 or 8) that hold four values each, in
// element order: lane j of the group computes (((prev + v0) + v1) + v2) + v3 where prev is
// lane j-1's result (init for j == 0). After N steps lane N-1 holds the group's fold.
template <int N>
__device__ __forceinline__ float lane_chain(const float (&v)[4], float init) {
    const int j = (int)(threadIdx.x & (N - 1));
    float run = init;
#pragma unroll
    for (int step = 0; step < N; ++step) {
        const float prev = __shfl_up(run, 1, N);  // lane j - 1 of the group (lane 0 keeps its own)
        const float base = j == 0 ? init : prev;
        const float r = (((base + v[0]) + v[1]) + v[2]) + v[3];
        run = j == step ? r : run;
    }
    return run;
}

// QuantizedActQ8::quantize_into (repack.rs:542-650): one wave per (row, 256-element
// superblock), lane l holding elements 4l..4l+3 (coalesced loads), 8 lanes per 32-block.
// Per block, quantize_block32_scalar (repack.rs:175-204): non-finite -> 0, absmax over the
// block (zero block below 1e-30), scale = absmax / 127, q = round(x * 127 / absmax) clamped
// to +-127, and the sequential sum from +0.0; the two x_sums_16 entries are Rust `.sum()`
// folds from -0.0; super_scales_256 (repack.rs:612-621) is the max of the superblock's
// block scales from 0.0. Elements past k (the zero-padded tail) take part as +0.0. With ACT != 0
// the element is the gated activation gated<ACT>(x, up) of the two input rows.
template <bool V4, int ACT>
__global__ __launch_bounds__(256) void quantize_act_q8_kernel(const float *__restrict__ x, const float *__restrict__ up,
                                                              jk_act_q8 a) {
    const size_t wv = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (wv >= a.m * a.sb256) return;  // wave-uniform
    const int l = (int)(threadIdx.x & 63);
    const size_t row = wv / a.sb256, sb = wv % a.sb256;
    const size_t e0 = sb * 256 + 4 * (size_t)l;
    const float *src = x + row * a.k;
    const float *usrc = ACT ? up + row * a.k : nullptr;
    float v[4];
    if constexpr (V4) {
        if (e0 + 3 < a.k) {
            const float4 f = *reinterpret_cast<const float4 *>(src + e0);
            v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
            if constexpr (ACT != kActNone) {
                const float4 u = *reinterpret_cast<const float4 *>(usrc + e0);
                v[0] = gated<ACT>(v[0], u.x); v[1] = gated<ACT>(v[1], u.y);
                v[2] = gated<ACT>(v[2], u.z); v[3] = gated<ACT>(v[3], u.w);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = e0 + i < a.k ? gated<ACT>(src[e0 + i], ACT ? usrc[e0 + i] : 0.0f) : 0.0f;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = e0 + i < a.k ? gated<ACT>(src[e0 + i], ACT ? usrc[e0 + i] : 0.0f) : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __builtin_isfinite(v[i]) ? v[i] : 0.0f;
    const float absmax = max8_dpp(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
    const bool zero = absmax < 1e-30f;
    const float inv = zero ? 0.0f : 127.0f / absmax;
    const float scale = zero ? 0.0f : absmax / 127.0f;
    uint32_t packed = 0;
    if (!zero) {
#pragma unroll
        for (int i = 0; i < 4; ++i) packed |= (uint32_t)(rust_round_clamp_i8(v[i] * inv, -127.0f, 127.0f) & 255) << (8 * i);
    }
    const float sum = lane_chain<8>(v, 0.0f);
    const float s16 = lane_chain<4>(v, -0.0f);
    // superblock max of the block scales (lanes 8b hold block b's scale), from 0.0
    float mx = fmaxf(0.0f, scale);
    mx = fmaxf(mx, __shfl_xor(mx, 8));
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));

    const size_t b = sb * 8 + (size_t)(l >> 3);
    if (b < a.k_blocks32) {
        *reinterpret_cast<uint32_t *>(a.qs + row * a.k_padded + e0) = packed;
        const int j = l & 7;
        if (j == 0) a.scales[row * a.k_blocks32 + b] = scale;
        if (j == 7) a.sums[row * a.k_blocks32 + b] = sum;
        if ((l & 3) == 3) a.sums16[row * a.k_chunks + 2 * b + (j >> 2)] = s16;
    }
    if (l == 0) a.super256[row * a.sb256 + sb] = mx;
}

template <int ACT>
static void launch_act_q8(hipStream_t s, const float *x, const float *up, const jk_act_q8 &a) {
    const size_t waves = a.m * a.sb256;
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
    const bool v4 = (a.k & 3) == 0 && ((uintptr_t)x & 15) == 0 && (!ACT || ((uintptr_t)up & 15) == 0);
    if (v4) hipLaunchKernelGGL((quantize_act_q8_kernel<true, ACT>), grid, block, 0, s, x, up, a);
    else hipLaunchKernelGGL((quantize_act_q8_kernel<false, ACT>), grid, block, 0, s, x, up, a);
}

jk_status launch_quantize_act_q8(hipStream_t s, const float *x, const jk_act_q8 &a) {
    return launch_quantize_act_q8_gated(s, kActNone, x, nullptr, a);
}

jk_status launch_quantize_act_q8_gated(hipStream_t s, int act, const float *x, const float *up, const jk_act_q8 &a) {
    if (act == kActSwiglu) launch_act_q8<kActSwiglu>(s, x, up, a);
    else if (act == kActRelu2) launch_act_q8<kActRelu2>(s, x, up, a);
    else launch_act_q8<kActNone>(s, x, up, a);
    return check_launch("quantize_act_q8_kernel");
}

// quantize_absmax_i8 of a row, with NORM of x * inv * nw: the maximum over the workgroup, then the codes.
// V4: k % 4 == 0 and 16-byte aligned rows and norm weights (the codes are then stored 4 at a time).
// NT: threads of the workgroup.
template <bool V4, bool NORM, int NT>
__device__ __forceinline__ void absmax_codes(const float *src, const float *nw, float inv, size_t k, int8_t *dst,
                                             float *scale_out) {
    constexpr int VE = V4 ? 4 : 1;
    __shared__ float s_max[NT / 64];
    const int t = threadIdx.x;
    auto xnorm = [&](size_t i, float (&o)[VE]) {  // of elements i .. i + VE - 1
        if constexpr (V4) {
            const float4 v = *reinterpret_cast<const float4 *>(src + i);
            o[0] = v.x, o[1] = v.y, o[2] = v.z, o[3] = v.w;
            if constexpr (NORM) {
                const float4 g = *reinterpret_cast<const float4 *>(nw + i);
                o[0] = o[0] * inv * g.x, o[1] = o[1] * inv * g.y, o[2] = o[2] * inv * g.z, o[3] = o[3] * inv * g.w;
            }
        } else {
            o[0] = NORM ? src[i] * inv * nw[i] : src[i];
        }
    };
    float mx = 0.0f;
    for (size_t i = (size_t)VE * t; i < k; i += (size_t)VE * NT) {
        float xn[VE];
        xnorm(i, xn);
#pragma unroll
        for (int e = 0; e < VE; ++e) {
            const float av = fabsf(xn[e]);
            if (av > mx) mx = av;
        }
    }
    mx = wave_max<64>(mx);
    if ((t & 63) == 0) s_max[t >> 6] = mx;
    __syncthreads();
    mx = s_max[0];
#pragma unroll
    for (int i = 1; i < NT / 64; ++i) mx = fmaxf(mx, s_max[i]);
    const bool zero = __builtin_isnan(mx) || mx < 1e-12f;
    const float scale = zero ? 1.0f / 127.0f : mx / 127.0f;
    for (size_t i = (size_t)VE * t; i < k; i += (size_t)VE * NT) {
        float xn[VE];
        int c[VE];
        xnorm(i, xn);
#pragma unroll
        for (int e = 0; e < VE; ++e) c[e] = zero ? 0 : rust_round_clamp_i8(xn[e] / scale, -128.0f, 127.0f);
        if constexpr (V4)
            *reinterpret_cast<uint32_t *>(dst + i) = (uint32_t)(c[0] & 255) | ((uint32_t)(c[1] & 255) << 8) |
                                                     ((uint32_t)(c[2] & 255) << 16) | ((uint32_t)(c[3] & 255) << 24);
        else dst[i] = (int8_t)c[0];
    }
    if (t == 0) *scale_out = scale;
}

// quantize_absmax_i8 (lib.rs:1072-1098) per row, one workgroup each: a wave for short rows, of which thousands come
// at once, up to sixteen where a row is long enough to keep them reading. Two passes over the row bound
// it. (us, 64 / 256 / 1024 threads, launched back to back: 8192 x 256 6.6 / 7.1 / 25, 8192 x 2560 29 / 23 /
// 38, 1 x 14336 32 / 9.9 / 7.0, 2048 x 14336 59 / 41 / 34)
template <bool V4, int NT>
__global__ __launch_bounds__(NT) void absmax_i8_kernel(const float *__restrict__ x, size_t k, int8_t *__restrict__ q,
                                                       float *__restrict__ scales) {
    const size_t row = blockIdx.x;
    absmax_codes<V4, false, NT>(x + row * k, nullptr, 1.0f, k, q + row * k, scales + row);
}

// subln_quantize_absmax_i8 (lib.rs:1042-1101) per row, one workgroup each.
//
// The sum of squares is the reference's sequential f32 sum (dot_product_f32_scalar, lib.rs:770-778):
// k additions that each wait for the one before, about 7 cycles each from LDS (20 us for 6912; 190 us by
// one thread from global memory). For few rows it is put together in parallel instead, bit for bit: while
// the running sum stays inside one binade it is an integer A times its ulp u, and adding x >= 0 gives
// RNE(A + x / u) u: A grows by round(x / u), where a tie goes to the even neighbour and so depends on
// whether A is even. What a run of elements adds is therefore a pair of integers, for A even and for A
// odd, and pairs are put together by a scan. (Ties are common: squares of bf16 values have few low
// bits.) An approximate prefix sum tells each element's binade. The elements where the rule does not
// hold (within 2e-5 of a power of two, about one per doubling of the sum; the first element; NaN and
// Inf; sums near the ends of the exponent range) are added one by one by the first wave, between them
// the runs, each as one integer addition to the float's bits. That addition is checked to start and to
// end in the expected binade, and all its elements to have been given that binade (a thread's
// approximate prefix can lie a few ulps below the end of the thread before it, put together in another
// order, and fall back into the binade below); where a check fails, or with too many elements outside
// the rule, the first wave adds the whole row in order. Normal rows of 2560 and 6912 have 12 and 14 such
// elements, of f32 and of bf16 values alike: 7.6 and 9.3 us a launch (with every tie added one by one
// 8.0 and 10 us, and for bf16 values, 325 and 726 ties, 59 and 151 us). What bounds it now: the scans'
// cross-lane steps, the elements added one by one (a scalar round trip each) and three passes over the row.
constexpr int kAbsThreads = 1024;
constexpr int kSqSerial = 256;    // pieces up to this length are added one by one
constexpr int kSqEvents = 256;    // elements outside the rule, at most

// What adding a run of elements adds to the running sum's integer A, for A even and for A odd.
struct SumRun {
    int even, odd;
};
__device__ __forceinline__ SumRun run_then(SumRun f, SumRun g) {
    return {f.even + ((f.even & 1) ? g.odd : g.even), f.odd + ((f.odd & 1) ? g.even : g.odd)};
}

// Inclusive scans over the lanes of a 16-lane row (WAVE: of the wave) by DPP moves, whose lanes without a
// source get zeros, the identity of all three.
template <int CTRL, int ROWS = 0xF> __device__ __forceinline__ int dpp_or0(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}
template <bool WAVE> __device__ __forceinline__ float scan_add(float v) {
    auto f = [](int x) { return __int_as_float(x); };
    v += f(dpp_or0<0x111>(__float_as_int(v)));  // row_shr:1, 2, 4, 8
    v += f(dpp_or0<0x112>(__float_as_int(v)));
    v += f(dpp_or0<0x114>(__float_as_int(v)));
    v += f(dpp_or0<0x118>(__float_as_int(v)));
    if constexpr (WAVE) {
        v += f(dpp_or0<0x142, 0xA>(__float_as_int(v)));  // row_bcast:15 into rows 1 and 3
        v += f(dpp_or0<0x143, 0xC>(__float_as_int(v)));  // row_bcast:31 into rows 2 and 3
    }
    return v;
}
// run: since the last of cnt events
template <int CTRL, int ROWS = 0xF> __device__ __forceinline__ void scan_run_step(SumRun &run, int &cnt) {
    const SumRun r = run_then({dpp_or0<CTRL, ROWS>(run.even), dpp_or0<CTRL, ROWS>(run.odd)}, run);
    const int c = dpp_or0<CTRL, ROWS>(cnt);
    run = cnt ? run : r;
    cnt += c;
}
template <bool WAVE> __device__ __forceinline__ void scan_runs(SumRun &run, int &cnt) {
    scan_run_step<0x111>(run, cnt);
    scan_run_step<0x112>(run, cnt);
    scan_run_step<0x114>(run, cnt);
    scan_run_step<0x118>(run, cnt);
    if constexpr (WAVE) {
        scan_run_step<0x142, 0xA>(run, cnt);
        scan_run_step<0x143, 0xC>(run, cnt);
    }
}

struct SumLds {
    static constexpr int NW = kAbsThreads / 64;
    float part[NW];                  // per wave: sum of its squares
    SumRun run[NW];                  // and its run after its last event, and its events
    int cnt[NW];
    uint32_t first[NW], last[NW];    // binades of the wave's first and last elements
    int split[NW];                   // whether a run changes its binade between two threads of the wave
    int4 ev[kSqEvents];              // position and binade, the run before it, the square's bits
    int tail_eb;                     // binade after the last element
};

// acc + s[0] + s[1] + ... + s[n - 1], in order (s: 16-byte aligned LDS, the same for every lane; up to
// the next multiple of 32 it holds -0.0, the identity of f32 addition), from 16-byte broadcast reads
// requested 32 values ahead, so that an addition waits only for the one before it.
__device__ __forceinline__ float ordered_sum(float acc, const float *s, int n) {
    const float4 *s4 = reinterpret_cast<const float4 *>(s);
    const int n32 = (n + 31) / 32;
    float4 cur[8], nxt[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) cur[i] = s4[i];
    for (int c = 0; c < n32; ++c) {
        const int cn = min(c + 1, n32 - 1);
#pragma unroll
        for (int i = 0; i < 8; ++i) nxt[i] = s4[8 * cn + i];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc = (((acc + cur[i].x) + cur[i].y) + cur[i].z) + cur[i].w;
#pragma unroll
        for (int i = 0; i < 8; ++i) cur[i] = nxt[i];
    }
    return acc;
}

// The same sum of n values >= 0 (or NaN) by the whole workgroup, as described above; the result is
// the first wave's. PER: values per thread, odd (the threads' reads then fall on distinct banks).
template <int PER>
__device__ __forceinline__ float parallel_ordered_sum(float acc0, const float *sq, int n, SumLds &L) {
    constexpr int NW = kAbsThreads / 64;
    static_assert(NW <= 16, "the waves' values in one row");
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lo = t * PER;
    float v[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) v[i] = sq[min(lo + i, n - 1)];
    float part = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        v[i] = lo + i < n ? v[i] : 0.0f;
        part += v[i];
    }
    const float incl = scan_add<true>(part);
    if (lane == 63) L.part[wave] = incl;
    __syncthreads();
    const float waves = scan_add<false>(lane < NW ? L.part[lane] : 0.0f);
    const float before_wave = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(waves), max(wave - 1, 0)));
    const float pre = acc0 + (wave > 0 ? before_wave : 0.0f) + (incl - part);  // approximate sum before the thread
    // adds element i, after an approximate sum p, to a run: its binade, and whether it goes by the rule
    auto element = [&](int i, float p, SumRun &run, uint32_t &eb) {
        eb = __float_as_uint(p * 0.99998f) >> 23;
        const uint32_t ee = __float_as_uint((p + v[i]) * 1.00002f) >> 23;
        const float to_ulp = __uint_as_float((277u - min(max(eb, 30u), 220u)) << 23);  // 1 / u, a power of two
        const float w = v[i] * to_ulp, fl = floorf(w), fr = w - fl;
        const int r = (int)fl + (fr > 0.5f), tie = fr == 0.5f;
        const int a = run.even + r, b = run.odd + r;  // (a tie: one more if that makes the sum even)
        run = {a + (a & tie), b + (~b & tie)};
        return eb == ee && eb >= 30 && eb <= 220 && w < 16777216.0f;
    };
    uint32_t events = 0;
    SumRun run = {0, 0};  // since the last event
    float p = pre;
    uint32_t first = 0, last = 0;  // binades of the first and the last element (kNoRun: no run goes on past it)
    constexpr uint32_t kNoRun = 1u << 16;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        uint32_t eb;
        const bool ok = element(i, p, run, eb), live = lo + i < n;  // (past the end: zeros, which add nothing)
        p += v[i];
        if (live && !ok) run = {0, 0};
        events |= (uint32_t)(live && !ok) << i;
        if (lo + i == n - 1) L.tail_eb = (int)eb;
        if (i == 0) first = live ? eb : kNoRun;
        if (i == PER - 1) last = live && ok ? eb : kNoRun;
    }
    // the elements of a run share a binade: within a thread by construction (an element by the rule ends in
    // the binade that the next one starts from), from one thread to the next by this test
    const uint32_t before = (uint32_t)dpp_or0<0x138>((int)last);  // wave_shr:1
    const bool split = lane > 0 && ((before | first) & kNoRun) == 0 && before != first;
    const uint64_t any_split = __ballot(split);
    if (lane == 0) L.first[wave] = first, L.split[wave] = any_split != 0;
    if (lane == 63) L.last[wave] = last;
    const int cnt = __popc(events);
    int pc = cnt;
    scan_runs<true>(run, pc);
    if (lane == 63) L.run[wave] = run, L.cnt[wave] = pc;
    const SumRun ex = {dpp_or0<0x138>(run.even), dpp_or0<0x138>(run.odd)};  // before the thread, in its wave
    __syncthreads();
    SumRun wr = lane < NW ? L.run[lane] : SumRun{0, 0};
    int wc = lane < NW ? L.cnt[lane] : 0;
    scan_runs<false>(wr, wc);
    const int prev = max(wave - 1, 0);
    const SumRun wp = {__builtin_amdgcn_readlane(wr.even, prev), __builtin_amdgcn_readlane(wr.odd, prev)};
    const int before_c = __builtin_amdgcn_readlane(wc, prev), total_c = __builtin_amdgcn_readlane(wc, NW - 1);
    if (events) {
        int ci = (wave > 0 ? before_c : 0) + pc - cnt;
        run = pc > cnt || wave == 0 ? ex : run_then(wp, ex);
        p = pre;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const SumRun before = run;
            uint32_t eb;
            element(i, p, run, eb);
            p += v[i];
            const bool event = (events >> i) & 1u;
            if (event && ci < kSqEvents)
                L.ev[ci] = make_int4((lo + i) << 9 | (int)eb, before.even, before.odd, __float_as_int(v[i]));
            ci += event;
            if (event) run = {0, 0};
        }
    }
    __syncthreads();
    if (t >= 64) return 0.0f;
    uint32_t bits = (uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(acc0));
    const int w1 = min(lane, NW - 1), w0 = max(w1 - 1, 0);
    const uint32_t l0 = L.last[w0], f1 = L.first[w1];
    const bool gap = L.split[w1] || (w1 > 0 && ((l0 | f1) & kNoRun) == 0 && l0 != f1);
    bool fits = total_c <= kSqEvents && __ballot(gap) == 0;
    const SumRun tail = {__builtin_amdgcn_readlane(wr.even, NW - 1), __builtin_amdgcn_readlane(wr.odd, NW - 1)};
    int pos = -1;  // the last element added (scalars)
    // the run up to (not including) element p, all in binade e
    auto advance = [&](int p, int even, int odd, uint32_t e) {
        const uint32_t to = bits + (uint32_t)((bits & 1u) ? odd : even);
        if (p > pos + 1 && ((bits >> 23) != e || (to >> 23) != e)) fits = false;
        bits = to;
    };
    for (int g = 0; fits && g < total_c; g += 64) {
        const int4 ev = L.ev[min(g + lane, total_c - 1)];  // lane l: event g + l
        for (int j = 0; j < min(64, total_c - g); ++j) {
            const uint32_t at = (uint32_t)__builtin_amdgcn_readlane(ev.x, j);
            const int p = (int)(at >> 9);
            advance(p, __builtin_amdgcn_readlane(ev.y, j), __builtin_amdgcn_readlane(ev.z, j), at & 511u);
            const float acc = __uint_as_float(bits) + __int_as_float(__builtin_amdgcn_readlane(ev.w, j));
            bits = (uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(acc));
            pos = p;
        }
    }
    advance(n, tail.even, tail.odd, (uint32_t)__builtin_amdgcn_readfirstlane(L.tail_eb));
    return fits ? __uint_as_float(bits) : ordered_sum(acc0, sq, n);
}

// SQ: values of a row summed at once, in LDS (a multiple of 32; a longer row in such pieces). PER: values per thread
// of the parallel sum (odd, see above; of 15, 14 are used: a workgroup's squares stay below 64 KB), or 0
// for the sum in order by the first wave.
template <bool V4, int NT, int PER, int SQ>
__global__ __launch_bounds__(NT) void absmax_i8_norm_kernel(const float *__restrict__ x, const float *__restrict__ nw,
                                                            size_t k, float eps, int8_t *__restrict__ q,
                                                            float *__restrict__ scales) {
    static_assert(PER == 0 || (NT == kAbsThreads && SQ <= PER * NT), "the parallel sum's threads");
    constexpr int VE = V4 ? 4 : 1;
    __shared__ __align__(16) float s_sq[SQ];
    __shared__ float s_inv;
    const size_t row = blockIdx.x;
    const float *src = x + row * k;
    const int t = threadIdx.x;
    float sum_sq = 0.0f;  // (the first wave's)
    for (size_t c0 = 0; c0 < k; c0 += SQ) {
        const int len = (int)min((size_t)SQ, k - c0);
        if (c0 > 0) {
            if (t == 0) s_inv = sum_sq;
            __syncthreads();  // the piece before is summed; its running sum is every thread's
            sum_sq = s_inv;
        }
        for (int i = VE * t; i < len; i += VE * NT) {
            if constexpr (V4) {
                const float4 v = *reinterpret_cast<const float4 *>(src + c0 + i);
                *reinterpret_cast<float4 *>(s_sq + i) = make_float4(v.x * v.x, v.y * v.y, v.z * v.z, v.w * v.w);
            } else {
                const float v = src[c0 + i];
                s_sq[i] = v * v;
            }
        }
        if (t < (-len & 31)) s_sq[len + t] = -0.0f;
        __syncthreads();
        if (PER == 0 || len <= kSqSerial) {
            sum_sq = t < 64 ? ordered_sum(sum_sq, s_sq, len) : 0.0f;
        } else if constexpr (PER > 0) {
            __shared__ __align__(16) SumLds s_sum;
            sum_sq = parallel_ordered_sum<PER>(sum_sq, s_sq, len, s_sum);
        }
    }
    if (t == 0) {
        const float mean_sq = sum_sq / (float)k;
        s_inv = 1.0f / sqrtf(mean_sq + eps);
    }
    __syncthreads();
    absmax_codes<V4, true, NT>(src, nw, s_inv, k, q + row * k, scales + row);
}

template <bool V4>
static void launch_absmax_plain(hipStream_t s, const float *x, size_t m, size_t k, int8_t *q, float *scales) {
    const dim3 grid((unsigned)m);
    if (k <= 1024) hipLaunchKernelGGL((absmax_i8_kernel<V4, 64>), grid, dim3(64), 0, s, x, k, q, scales);
    else if (k <= 4096) hipLaunchKernelGGL((absmax_i8_kernel<V4, 256>), grid, dim3(256), 0, s, x, k, q, scales);
    else hipLaunchKernelGGL((absmax_i8_kernel<V4, 1024>), grid, dim3(1024), 0, s, x, k, q, scales);
}

// The parallel sum takes a workgroup per CU and its time is its latency, so it is for as many rows as there are
// CUs, or few rounds of long ones; more rows go in order, in small workgroups of which a CU holds many
// (us, launched back to back: 64 threads 8192 x 256 8.8, 8192 x 1000 26, 600 x 1000 9.1; 256 threads 600 x 2560
// 14.8, 2048 x 2560 18, 2048 x 6912 49; the parallel sum 8192 x 256 219, 8192 x 1000 114, 600 x 1000 13.9, 600 x 2560
// 15.9, 2048 x 2560 35, 2048 x 6912 82; and 600 x 6912 31 against 34 in order). Rows of up to 256 values
// are as soon added by one wave as shared out.
template <bool V4>
static void launch_absmax_norm(hipStream_t s, const float *x, const float *nw, size_t m, size_t k, float eps, int8_t *q,
                               float *scales) {
    const dim3 grid((unsigned)m);
    const size_t ncu = (size_t)cu_count();
    auto launch = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, grid, dim3((unsigned)threads), 0, s, x, nw, k, eps, q, scales);
    };
    constexpr int T = kAbsThreads;
    if (k <= kSqSerial || (m > ncu && k <= 1024)) launch(absmax_i8_norm_kernel<V4, 64, 0, 1024>, 64);
    else if (m > ncu && (k <= 4096 || m > 4 * ncu)) launch(absmax_i8_norm_kernel<V4, 256, 0, 2048>, 256);
    else if (k <= 3 * T) launch(absmax_i8_norm_kernel<V4, T, 3, 3 * T>, T);
    else if (k <= 7 * T) launch(absmax_i8_norm_kernel<V4, T, 7, 7 * T>, T);
    else launch(absmax_i8_norm_kernel<V4, T, 15, 14 * T>, T);
}

jk_status launch_absmax_i8(hipStream_t s, const float *x, const float *norm_w, size_t m, size_t k, float eps,
                           int8_t *q, float *scales) {
    const bool v4 = k % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)norm_w % 16 == 0 && (uintptr_t)q % 4 == 0;
    if (norm_w) (v4 ? launch_absmax_norm<true> : launch_absmax_norm<false>)(s, x, norm_w, m, k, eps, q, scales);
    else (v4 ? launch_absmax_plain<true> : launch_absmax_plain<false>)(s, x, m, k, q, scales);
    return check_launch("absmax_i8_kernel");
}

}  // namespace jk
