// Device helpers of the decoder's kernels: constants, f16 and vector access, LDS DMA, serial chains in segments with
// candidate starts, rmsnorm and quantization of a row. Used by qh_decoder.hip and qh_attn_few.hip.
#pragma once

#include <type_traits>

#include "qh_device.h"
#include "qh_gemv.h"
#include "qh_internal.h"
#include "qh_math.h"

namespace qh {

namespace {

constexpr int kChunk = 32;            // prefill chunk (reference Model::kBatch, model.h:52)
constexpr int kMaxStack = 1024;       // prefill stack limit (tokens whose matmuls share a launch)
constexpr int kMaxCtx = 8192;         // positions the attention kernel's score array holds
constexpr int kVStageBytes = 96 * 1024;  // LDS for staged V rows (768 rows at head_dim 64)
constexpr int kFuseLds = 65536;       // dynamic LDS limit of the fused GEMV kernels

// Positions the V cache holds per layer: the context rounded up to its 8-position blocks.
inline int v_ctx(int ctx) { return (ctx + 7) & ~7; }

// Floats per attention workgroup's exp row: the context rounded up to 16 (64-byte aligned rows) plus 64 of slack for
// whole-batch scalar reads past the last position.
inline int escr_stride(int ctx) { return ((ctx + 15) & ~15) + 64; }

enum { kStatusCtx = 1, kStatusToken = 2 };


__device__ __forceinline__ float h2f(uint16_t h) { return f16_to_f32(h); }

// A 16-byte register value as a native vector (register arrays of HIP's uint4 struct are not always split into
// registers by the compiler; native vectors are).
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4u ld4(const void* p) { return *reinterpret_cast<const v4u*>(p); }

// LDS DMA (global_load_lds_dwordx4): lane l's 16 bytes at g go to lds_wave + 16 l, where lds_wave is the same LDS
// address in every lane of the wave. Counted by vmcnt; the LDS data is valid after s_waitcnt vmcnt(0). Issued in
// inline assembly, behind the compiler's back: the compiler counts a DMA it knows of as a transfer that may complete
// out of order, so after one it waits for every outstanding load (vmcnt(0)) before using any earlier load's result
// and before any LDS access. This way the earlier loads keep their waits, LDS accesses wait for nothing, the caller
// waits for the transfer itself (s_waitcnt vmcnt(0)) before reading its LDS, and the compiler's waits for loads
// issued before it become conservative (they also cover the transfers), never short. M0, which the transfer takes
// its LDS address from, is an input operand of the asm ("{m0}" constraint): the compiler writes it and knows what M0
// holds afterwards. The s_nop covers the wait state between an M0 write and the transfer that reads it. The body
// exists only in the device pass (the host pass cannot form an LDS address).
__device__ __forceinline__ void lds_dma16_async(const void* g, void* lds_wave) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds_wave);
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(m0) : "memory");
#endif
}
// f32 -> f16 (round to nearest even) of an already rounded f32 value, as the reference stores its f32 K / V results
// into the f16 cache. The empty asm makes the value opaque, so the compiler cannot fuse the FMA that produced it and
// this conversion into one v_fma_mixlo_f16, which rounds only once (straight to f16) and differs on double-rounding
// cases.
__device__ __forceinline__ uint16_t f2h(float f) {
    asm volatile("" : "+v"(f));
    return __builtin_bit_cast(uint16_t, (_Float16)f);
}

// quantize_q8 of one 32-block held one value per lane of a half-wave (ops_ref.cpp:69-83): the block's absolute
// maximum / 127, codes rounded half away from zero. Every lane of the half-wave must be active.
// Maximum over the whole wave (every lane active) with the select o > a ? o : a at each step: DPP within rows of
// 16, then the gfx950 row swaps (16 and 32 lanes apart).
__device__ __forceinline__ float wave_max_sel(float a) {
    auto step = [](float x, float o) { return o > x ? o : x; };
    a = step(a, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0xB1, 0xF, 0xF, false)));
    a = step(a, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0x4E, 0xF, 0xF, false)));
    a = step(a, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0x141, 0xF, 0xF, false)));
    a = step(a, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0x140, 0xF, 0xF, false)));
    uint32_t u = __builtin_bit_cast(uint32_t, a);
    const auto s16 = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    a = step(__builtin_bit_cast(float, (uint32_t)s16[0]), __builtin_bit_cast(float, (uint32_t)s16[1]));
    u = __builtin_bit_cast(uint32_t, a);
    const auto s32 = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return step(__builtin_bit_cast(float, (uint32_t)s32[0]), __builtin_bit_cast(float, (uint32_t)s32[1]));
}

// quantize_q8 of the row xs[0, D) (16-byte aligned, D % 32 == 0) into q / d: 8 lanes per block, 32 blocks per pass
// of 256 threads.
__device__ __forceinline__ void quant_row_x8(const float* xs, int D, int8_t* __restrict__ q, float* __restrict__ d) {
    const int nb = D / QK;
    for (int t = (int)threadIdx.x; t < nb * 8; t += 256) {  // whole 8-lane groups
        const int b = t >> 3;
        quant_block_x8(reinterpret_cast<const float4*>(xs)[t], q + b * QK, d + b);
    }
}

// acc = op(acc, p[i]) for i = 0 .. n-1 in order, by one thread, over floats in LDS (16-byte aligned, n >= 1). A wave
// issues about one instruction per 4 cycles whatever its kind, so the loop is shaped for the fewest instructions
// per element: batches of 32 values read as 8 b128 at immediate offsets from one base, two register sets that
// alternate without copies (the next batch in flight while the current one is consumed), no clamping. It reads up
// to kChainPad floats past n: callers size the array n + kChainPad.
constexpr int kChainPad = 64;

// An LDS address the compiler treats as per-lane: uniform LDS addresses otherwise get rematerialized into a VGPR for
// every read, costing an instruction each (mbcnt_lo(0, 0) is 0 in every lane).
template <typename T>
__device__ __forceinline__ const T* lane_ptr(const T* p) {
    return p + __builtin_amdgcn_mbcnt_lo(0u, 0u);
}

template <typename Op>
__device__ __forceinline__ float lds_chain(const float* p, int n, Op op, float acc0 = 0.0f) {
    float4 a[8], b[8];
    auto ld = [](float4(&r)[8], const float* q) {
        const float4* q4 = reinterpret_cast<const float4*>(q);
#pragma unroll
        for (int k = 0; k < 8; ++k) r[k] = q4[k];
    };
    float acc = acc0;
    auto use = [&](const float4(&r)[8], int cnt) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (4 * k + 0 < cnt) acc = op(acc, r[k].x);
            if (4 * k + 1 < cnt) acc = op(acc, r[k].y);
            if (4 * k + 2 < cnt) acc = op(acc, r[k].z);
            if (4 * k + 3 < cnt) acc = op(acc, r[k].w);
        }
    };
    int j = 0;
    p = lane_ptr(p);
    ld(a, p);
    // sched_barrier keeps each prefetch ahead of the values it overlaps (the scheduler would sink it)
    for (; j + 64 <= n; j += 64) {
        ld(b, p + j + 32);
        __builtin_amdgcn_sched_barrier(0);
        use(a, 32);
        ld(a, p + j + 64);
        __builtin_amdgcn_sched_barrier(0);
        use(b, 32);
    }
    if (j + 32 <= n) {
        ld(b, p + j + 32);
        __builtin_amdgcn_sched_barrier(0);
        use(a, 32);
        use(b, n - j - 32);  // cnt is uniform
    } else {
        use(a, n - j);
    }
    return acc;
}

// R float4 per thread of a row of n4 <= 256 R float4 with every load issued before the first use: slot k holds
// element tid + 256 k (clamped onto the last element, so the loads are unconditional). Kernels take R = row_slots(n4):
// one load per thread up to D = 1024, eight (D <= 8192) above.
template <int R>
struct RowF4 {
    float4 v[R];
    __device__ __forceinline__ void load(const float* __restrict__ src, int n4) {
        const float4* s4 = reinterpret_cast<const float4*>(src);
#pragma unroll
        for (int k = 0; k < R; ++k) v[k] = s4[min((int)threadIdx.x + 256 * k, n4 - 1)];
    }
};
constexpr int row_slots(int n4) { return n4 <= 256 ? 1 : 8; }

// ------------------------------------------------------------------------------ segmented sum of squares
// rmsnorm's sum of squares is one serial chain, ss = fma(x_i, x_i, ss) for i = 0 .. D-1 in order (ops_ref.cpp:195-197):
// D dependent FMAs, the longest dependency of a decode layer. seg_sum_squares runs it as four segments at once, one
// per wave, and still returns the chain's value bit for bit:
//  - wave 0 runs segment 0 from 0;
//  - the wave of segment k >= 1 runs it from 64 start values at once, one per lane: the f32 rounding of the exact
//    (double) sum of squares before the segment, and its neighbours 32 below to 31 above in bit order. The chain's
//    value at the segment start differs from that guess only by the chain's own accumulated rounding (at most 26 ulps
//    over 2*10^5 random rows of 896, including rows with outliers), so some lane almost always started at exactly
//    the chain's value, and that lane's result is then the chain's value at the segment end;
//  - every thread then follows the chain from segment 0 through the lanes whose start matches bit for bit; a value
//    outside a window (rare) is continued by running that segment serially from it.
// The chains read x through scalar loads (x is in global memory and no workgroup writes it during the kernel): one
// 64-byte load feeds 16 FMAs of all 64 lanes with scalar operands, and the LDS stays free for the other waves.
// Scalar loads can return out of order, so the loop waits for everything outstanding after each 32-value batch,
// with the next batch already issued; each wave first touches every 64-byte line of its segment (SegWarm) so these
// loads hit the scalar cache.
typedef float v16f __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(4))) v16f* const_v16f_ptr;
typedef const __attribute__((address_space(4))) uint32_t* const_u32_ptr;

// lgkmcnt(0) with the vector-memory and export counters left alone (gfx9 s_waitcnt encoding).
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xc07f); }

// acc = fma(g[i], g[i], acc) for i = 0 .. n-1 in order, g uniform across the wave and 64-byte aligned, n % 32 == 0.
__device__ __forceinline__ float ss_chain_scalar(const float* g, int n, float acc) {
    const_v16f_ptr p = (const_v16f_ptr)g;
    const int nv = n / 16;  // even
    v16f a0 = p[0], a1 = p[1];
    wait_lgkm0();
    __builtin_amdgcn_sched_barrier(0);
    int i = 0;
#pragma unroll 1
    for (; i + 4 <= nv; i += 4) {
        const v16f b0 = p[i + 2], b1 = p[i + 3];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = __builtin_fmaf(a0[k], a0[k], acc);
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = __builtin_fmaf(a1[k], a1[k], acc);
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkm0();
        __builtin_amdgcn_sched_barrier(0);
        a0 = p[min(i + 4, nv - 2)];
        a1 = p[min(i + 5, nv - 1)];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = __builtin_fmaf(b0[k], b0[k], acc);
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = __builtin_fmaf(b1[k], b1[k], acc);
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkm0();
        __builtin_amdgcn_sched_barrier(0);
    }
    if (i + 2 <= nv) {  // nv % 4 == 2: the last batch, loaded by the loop (or before it)
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = __builtin_fmaf(a0[k], a0[k], acc);
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = __builtin_fmaf(a1[k], a1[k], acc);
    }
    return acc;
}

// One scalar load per 64-byte line of the first 256 values of g[0, n): brings them into the scalar cache; the values
// are held until consume() so the loads cannot be dropped.
struct SegWarm {
    uint32_t v[16];
    __device__ __forceinline__ void issue(const float* g, int n) {
        const_u32_ptr q = (const_u32_ptr)g;
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = q[min(i * 16, n - 1)];
    }
    __device__ __forceinline__ void consume() const {
        asm volatile("" ::"s"(v[0]), "s"(v[1]), "s"(v[2]), "s"(v[3]), "s"(v[4]), "s"(v[5]), "s"(v[6]), "s"(v[7]));
        asm volatile("" ::"s"(v[8]), "s"(v[9]), "s"(v[10]), "s"(v[11]), "s"(v[12]), "s"(v[13]), "s"(v[14]), "s"(v[15]));
    }
};

// Sum over the wave of a double, in lane 63 (DPP: pairs, quads, half rows, rows, then rows 0+1 and 2+3 across).
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double wave_sum_lane63(double v) {
    v += dpp_f64<0xb1>(v);         // quad_perm [1,0,3,2]
    v += dpp_f64<0x4e>(v);         // quad_perm [2,3,0,1]
    v += dpp_f64<0x141>(v);        // row_half_mirror
    v += dpp_f64<0x140>(v);        // row_mirror
    v += dpp_f64<0x142, 0xa>(v);   // row_bcast:15 into rows 1, 3
    v += dpp_f64<0x143, 0xc>(v);   // row_bcast:31 into rows 2, 3
    return v;
}

// acc = op(acc, g[i]) for i = 0 .. n-1 in order (n >= 1), g uniform across the wave and 4-byte aligned. Whole
// batches of 32 values are read, so up to 32 values past n must be readable.
template <typename Op>
__device__ __forceinline__ float chain_scalar(const float* g, int n, float acc, Op op) {
    const_v16f_ptr p = (const_v16f_ptr)g;
    const int nb = n >> 5, rem = n & 31;
    auto use = [&](const v16f& x0, const v16f& x1, int cnt) {  // cnt is uniform
#pragma unroll
        for (int k = 0; k < 16; ++k)
            if (k < cnt) acc = op(acc, x0[k]);
#pragma unroll
        for (int k = 0; k < 16; ++k)
            if (16 + k < cnt) acc = op(acc, x1[k]);
    };
    v16f a0 = p[0], a1 = p[1];
    wait_lgkm0();
    __builtin_amdgcn_sched_barrier(0);
    int b = 0;
#pragma unroll 1
    for (; b + 2 <= nb; b += 2) {
        const v16f c0 = p[2 * b + 2], c1 = p[2 * b + 3];
        __builtin_amdgcn_sched_barrier(0);
        use(a0, a1, 32);
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkm0();
        __builtin_amdgcn_sched_barrier(0);
        a0 = p[2 * b + 4];
        a1 = p[2 * b + 5];
        __builtin_amdgcn_sched_barrier(0);
        use(c0, c1, 32);
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkm0();
        __builtin_amdgcn_sched_barrier(0);
    }
    if (b < nb) {  // a full batch in a, the partial one after it
        const v16f c0 = p[2 * b + 2], c1 = p[2 * b + 3];
        __builtin_amdgcn_sched_barrier(0);
        use(a0, a1, 32);
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkm0();
        __builtin_amdgcn_sched_barrier(0);
        use(c0, c1, rem);
    } else {
        use(a0, a1, rem);
    }
    return acc;
}

// Four segments of a chain over n values, wave w running segment w: [0, b1), [b1, b1 + L), [b1 + L, b1 + 2 L),
// [b1 + 2 L, n).
struct Segs4 {
    int b1, L, n;
    __device__ __forceinline__ int start(int k) const { return k == 0 ? 0 : b1 + (k - 1) * L; }
    __device__ __forceinline__ int len(int k) const { return k == 0 ? b1 : k == 3 ? n - b1 - 2 * L : L; }
};

// Workgroup state of one segmented chain.
struct SegShared {
    double part[4][4];  // [wave][k]: the wave's share of the exact sum of the chain's terms below segment k's start
    float res[256];     // every lane's segment result
    uint32_t gbits[4];  // segment k's guess
};

// Sums three per-lane partials over the wave into part[wave][1..3]; a barrier must follow before seg_chain_run.
__device__ __forceinline__ void seg_partials(SegShared& sh, double p1, double p2, double p3) {
    p1 = wave_sum_lane63(p1);
    p2 = wave_sum_lane63(p2);
    p3 = wave_sum_lane63(p3);
    if ((threadIdx.x & 63) == 63) {
        const int w = (int)threadIdx.x >> 6;
        sh.part[w][1] = p1;
        sh.part[w][2] = p2;
        sh.part[w][3] = p3;
    }
}

// Runs the segments (wave 0 from 0, the wave of segment k from the 64 candidates around its guess), a barrier, then
// follows the chain through the candidates; returns the chain's end value in every thread. chain(k, start) runs
// segment k from start in the calling wave (k and start uniform across the wave) and returns its end value. All 256
// threads call it after the barrier that published part.
template <typename Chain>
__device__ __forceinline__ float seg_chain_run(SegShared& sh, Chain chain) {
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float start = 0.0f;
    if (wave > 0) {
        const double g = sh.part[0][wave] + sh.part[1][wave] + sh.part[2][wave] + sh.part[3][wave];
        const uint32_t gb = __float_as_uint((float)g);
        start = __uint_as_float(gb + (uint32_t)lane - 32u);
        if (lane == 0) sh.gbits[wave] = gb;
    }
    sh.res[tid] = chain(wave, start);
    __syncthreads();
    float s = sh.res[0];
    const uint32_t g1 = sh.gbits[1], g2 = sh.gbits[2], g3 = sh.gbits[3];
#pragma unroll
    for (int k = 1; k < 4; ++k) {
        const uint32_t j = __float_as_uint(s) - (k == 1 ? g1 : k == 2 ? g2 : g3) + 32u;
        if (j < 64u)
            s = sh.res[64 * k + j];
        else
            s = chain(k, s);
    }
    return s;
}

// The chain's value ss of x[0, D) in every thread: segments [0, S0) and three of L = (D / 4) rounded down to a
// multiple of 32 (S0 = D - 3 L >= L). x: global, 64-byte aligned, not written during the kernel; xr: this thread's
// RowF4 of x; warm: seg_warm(x, D), issued by the same thread. All 256 threads of the workgroup call it (two barriers
// inside). D % 64 == 0, 128 <= D <= 8192.
__device__ __forceinline__ Segs4 seg_split(int D) {
    const int L = (D / 4) & ~31;
    return Segs4{D - 3 * L, L, D};
}
// The scalar loads that bring this wave's segment of x into the scalar cache (issued early, consumed by
// seg_sum_squares).
__device__ __forceinline__ SegWarm seg_warm(const float* __restrict__ x, int D) {
    const Segs4 sg = seg_split(D);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    SegWarm warm;
    warm.issue(x + sg.start(wave), sg.len(wave));
    return warm;
}
template <int R>
__device__ float seg_sum_squares(const float* __restrict__ x, int D, const RowF4<R>& xr, const SegWarm& warm,
                                 int tlk = -1) {
    (void)tlk;
    __shared__ SegShared sh;
    const int tid = (int)threadIdx.x, n4 = D / 4;
    const Segs4 sg = seg_split(D);
    double p1 = 0.0, p2 = 0.0, p3 = 0.0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i4 = tid + 256 * k;
        if (i4 < n4) {
            const float4 v = xr.v[k];
            const double s = (double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z + (double)v.w * v.w;
            const int e = 4 * i4;
            p1 += e < sg.start(1) ? s : 0.0;
            p2 += e < sg.start(2) ? s : 0.0;
            p3 += e < sg.start(3) ? s : 0.0;
        }
    }
    seg_partials(sh, p1, p2, p3);
    __syncthreads();
    QH_WSTAMP(tlk, 4);
    warm.consume();
    const float r = seg_chain_run(sh, [&](int k, float s0) { return ss_chain_scalar(x + sg.start(k), sg.len(k), s0); });
    QH_WSTAMP(tlk, 5);
    return r;
}

// seg_sum_squares for a row held in LDS (xs, complete, 16-byte aligned, kChainPad floats of slack; written in this
// kernel, so not readable through scalar loads): the same segments and candidate starts, each segment's chain reading
// its operands from LDS (the four waves' broadcast reads slow each other, ~12 cycles per element, against ~6 for
// scalar operands, still a quarter of the serial chain). xr: this thread's RowF4 of the row's values. All 256 threads
// call it (two barriers inside).
template <int R>
__device__ float seg_sum_squares_lds(const float* xs, int D, const RowF4<R>& xr) {
    __shared__ SegShared sh;
    const int tid = (int)threadIdx.x, n4 = D / 4;
    const Segs4 sg = seg_split(D);
    double p1 = 0.0, p2 = 0.0, p3 = 0.0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i4 = tid + 256 * k;
        if (i4 < n4) {
            const float4 v = xr.v[k];
            const double s = (double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z + (double)v.w * v.w;
            const int e = 4 * i4;
            p1 += e < sg.start(1) ? s : 0.0;
            p2 += e < sg.start(2) ? s : 0.0;
            p3 += e < sg.start(3) ? s : 0.0;
        }
    }
    seg_partials(sh, p1, p2, p3);
    __syncthreads();
    return seg_chain_run(sh, [&](int k, float s0) {
        return lds_chain(xs + sg.start(k), sg.len(k), [](float acc, float v) { return __builtin_fmaf(v, v, acc); }, s0);
    });
}

// rmsnorm scale 1 / sqrt(ss / D + eps) (ops_ref.cpp:197-198).
__device__ __forceinline__ float rms_scale(float ss, int D, float eps) {
    return 1.0f / __builtin_sqrtf(ss / (float)D + eps);
}

// The sum of squares of xs[0, D) (LDS, complete, kChainPad floats of slack) by thread 0, in every thread.
__device__ __forceinline__ float lds_sum_squares(const float* xs, int D) {
    __shared__ float ss_sh;
    if (threadIdx.x == 0) ss_sh = lds_chain(xs, D, [](float acc, float v) { return __builtin_fmaf(v, v, acc); });
    __syncthreads();
    return ss_sh;
}

// y = x * scale * w of the row xs[0..D) (LDS; each thread reads and rewrites its own float4s, slot k = tid + 256 k),
// also to `normed` when given, then quantize_q8 of y. All 256 threads call it; xs is free after its return only
// after a barrier.
template <int R>
__device__ void normalize_quant_lds(float* xs, int D, float scale, const RowF4<R>& wr, int8_t* __restrict__ oq,
                                    float* __restrict__ od, float* __restrict__ normed) {
    const int tid = (int)threadIdx.x, n4 = D / 4;
    float4* x4 = reinterpret_cast<float4*>(xs);
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i4 = tid + 256 * k;
        if (i4 < n4) {
            float4 xv = x4[i4];
            xv.x = xv.x * scale * wr.v[k].x;
            xv.y = xv.y * scale * wr.v[k].y;
            xv.z = xv.z * scale * wr.v[k].z;
            xv.w = xv.w * scale * wr.v[k].w;
            x4[i4] = xv;
            if (normed) reinterpret_cast<float4*>(normed)[i4] = xv;
        }
    }
    __syncthreads();
    quant_row_x8(xs, D, oq, od);
}

// rmsnorm of the row xs[0..D) (LDS, 16-byte aligned, complete) with weight w (loaded into wr by the caller before
// the row was complete, so its latency is hidden), then quantize_q8 of the normed row; also written to `normed`
// when given (ops_ref.cpp:195-199: ss += x*x as one FMA per element in order, scale = 1/sqrt(ss/n + eps),
// y = x * scale * w). Called by all 256 threads of a workgroup; D % 64 == 0, D <= 8192.
template <int R>
__device__ void norm_quant_lds(float* xs, int D, const RowF4<R>& wr, float eps, int8_t* __restrict__ oq,
                               float* __restrict__ od, float* __restrict__ normed) {
    normalize_quant_lds(xs, D, rms_scale(lds_sum_squares(xs, D), D, eps), wr, oq, od, normed);
}

}  // namespace

}  // namespace qh
