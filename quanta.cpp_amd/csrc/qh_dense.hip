// Unquantized weights (F32 / F16): matvec_ref (reference ops_ref.cpp:8-27) for n tokens, out[t * ldo + r] = acc with
// acc = fma(w_ri, x_ti, acc) from +0 in column order (the reference build contracts acc += w * x; an F16 weight converts
// exactly). Up to three matrices of one type and width over the same activations share a launch (q / k / v, gate / up).
//
// One token: a row is one serial chain, so the time is the chain's, cols dependent multiply-adds, as long as the weights
// keep up. A workgroup owns 16 rows, one lane each: wave 0 runs the chains, its weights from LDS (four columns to a
// 16-byte read, rows 4 banks apart) and the activation as scalar operands, while waves 1-3 load the tile after next and
// stage the next, 256 columns at a time, coalesced and widened; wave 1 also brings the next tile's activation lines
// into the scalar cache. Against 64 rows to a workgroup with the activation from LDS: F16 896x4864 53 -> 23 us,
// 200x14336 154 -> 62 us, F32 9000x8192 113 -> 79 us, F16 4864x896 11 -> 7 us (the call). With many rows the
// memory bounds it, not the chain, and a workgroup takes 64 rows by 64 columns, with or without loading waves
// (gemv_form). The arguments of a launch of one matrix are plain values, which are in registers when a wave starts; out
// of the three matrices' struct they cost every wave a read of the kernel's arguments before its first load (0.1 us a
// round of workgroups: F16 60000x256 8.0 -> 7.5 us, F32 16384x128 4.3 -> 3.8).
// Several tokens: the chains of 16 rows x 16 tokens are an f32 matrix product summed in order (v_mfma_f32_16x16x4_f32:
// each k step one fused multiply-add, see qh_attn.hip), 32 rows x 32 tokens to a workgroup of four waves, weights and
// activations staged in LDS in operand order, 64 columns at a time.
#include "qh_device.h"
#include "qh_internal.h"

namespace qh {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(4))) v16f* const_v16f_ptr;
typedef const __attribute__((address_space(4))) uint32_t* const_u32_ptr;

struct DenseSegs {
    const uint8_t* w[3];
    float* out[3];
    int ldo[3], r0[3], r1[3];
    int tiles[3];  // row tiles per matrix
};
struct DenseSeg {
    const uint8_t* w;
    float* out;
    int ldo, r0, r1;
    __device__ __forceinline__ DenseSeg(const uint8_t* w_, float* out_, int r0_, int r1_)
        : w(w_), out(out_), ldo(0), r0(r0_), r1(r1_) {}
    __device__ __forceinline__ DenseSeg(const DenseSegs& g, int& t) {  // t: the launch's row tile, then the matrix's
        int s = 0;
        if (t >= g.tiles[0]) {
            t -= g.tiles[0];
            s = 1;
            if (t >= g.tiles[1]) {
                t -= g.tiles[1];
                s = 2;
            }
        }
        w = s == 0 ? g.w[0] : s == 1 ? g.w[1] : g.w[2];
        out = s == 0 ? g.out[0] : s == 1 ? g.out[1] : g.out[2];
        ldo = s == 0 ? g.ldo[0] : s == 1 ? g.ldo[1] : g.ldo[2];
        r0 = s == 0 ? g.r0[0] : s == 1 ? g.r0[1] : g.r0[2];
        r1 = s == 0 ? g.r1[0] : s == 1 ? g.r1[1] : g.r1[2];
    }
};

// The 4 (F32) or 8 (F16) weights of a 16-byte unit in f32.
template <int DT>
__device__ __forceinline__ void widen(const uint4& u, float (&f)[DT == kF32 ? 4 : 8]) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (DT == kF32) {
            f[i] = __uint_as_float(w[i]);
        } else {
            f[2 * i] = f16_to_f32((uint16_t)(w[i] & 0xffffu));
            f[2 * i + 1] = f16_to_f32((uint16_t)(w[i] >> 16));
        }
    }
}

constexpr int kGvLoaders = 192;

}  // namespace

// ONE: the matrix is w0 / out0, rows [r0, r1); else segs has them. res: out[r] = res[r] + acc (a residual stream, read
// and written by the same lane), or null.
template <int DT, int kGvRows, bool ONE>
__global__ __launch_bounds__(256) void gemv_dense_kernel(const uint8_t* __restrict__ w0, float* out0, const float* __restrict__ x,
                                                         const float* res, int cols, int r0, int r1, DenseSegs segs) {
    constexpr int kGvCols = 4096 / kGvRows, kGvStride = kGvCols + 4;
    constexpr int kSize = DT == kF32 ? 4 : 2, kPer = 16 / kSize;                    // bytes per weight, weights per unit
    constexpr int kUnits = (kGvRows * kGvCols / kPer + kGvLoaders - 1) / kGvLoaders;  // units per loading thread
    constexpr int kUpr = kGvCols / kPer;                                              // units per row and tile
    __shared__ __align__(16) float ws[2][kGvRows * kGvStride];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int rt = (int)blockIdx.x;
    const DenseSeg sg = ONE ? DenseSeg(w0, out0, r0, r1) : DenseSeg(segs, rt);
    const int rbase = sg.r0 + rt * kGvRows, ntiles = (cols + kGvCols - 1) / kGvCols;
    if (wave == 0) {
        float acc = 0.0f;
        const int row = rbase + (lane & (kGvRows - 1));
        const float rv = res && row < sg.r1 ? res[row] : 0.0f;
        auto xload = [&](int c, v16f& a, v16f& b) {  // 32 activations from column c (clamped: the last of the row)
            const const_v16f_ptr p = (const_v16f_ptr)(x + min(c, cols - 32));
            a = p[0];
            b = p[1];
        };
        auto wait = [] { __builtin_amdgcn_s_waitcnt(0xc07f); };  // lgkmcnt(0)
        v16f xa0, xa1, xb0, xb1;
        xload(0, xa0, xa1);
        for (int t = 0; t < ntiles; ++t) {
            __syncthreads();  // tile t is staged
            const float4* wr = reinterpret_cast<const float4*>(&ws[t & 1][(lane & (kGvRows - 1)) * kGvStride]);
            const int nc = min(kGvCols, cols - t * kGvCols) / 32;  // batches of 32 columns
            float4 wa[8], wb[8];
            auto wload = [&](int b, float4(&w)[8]) {
#pragma unroll
                for (int i = 0; i < 8; ++i) w[i] = wr[8 * b + i];
            };
            auto use = [&](const float4(&w)[8], const v16f& a, const v16f& b) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float f[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc = __builtin_fmaf(f[e], i < 4 ? a[(4 * i + e) & 15] : b[(4 * i + e) & 15], acc);
                }
            };
            wload(0, wa);
            for (int b = 0; b < nc; b += 2) {  // a batch's reads are issued under the one before
                wait();
                __builtin_amdgcn_sched_barrier(0);
                xload(t * kGvCols + 32 * (b + 1), xb0, xb1);
                wload(min(b + 1, kGvCols / 32 - 1), wb);
                __builtin_amdgcn_sched_barrier(0);
                use(wa, xa0, xa1);
                __builtin_amdgcn_sched_barrier(0);
                wait();
                __builtin_amdgcn_sched_barrier(0);
                if (b + 1 < nc) {  // uniform
                    xload(t * kGvCols + 32 * (b + 2), xa0, xa1);
                    wload(min(b + 2, kGvCols / 32 - 1), wa);
                    __builtin_amdgcn_sched_barrier(0);
                    use(wb, xb0, xb1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if (lane < kGvRows && row < sg.r1) sg.out[row] = res ? rv + acc : acc;
        return;
    }
    // waves 1-3: unit e = 192 j + (tid - 64) of the tile is row e / kUpr, columns kPer (e % kUpr) ..; rows past
    // r1 and columns past cols are clamped (loaded, never used)
    const int lt = tid - 64;
    uint4 u[2][kUnits];
    auto load = [&](uint4(&r)[kUnits], int t) {
        const int c0 = min(t, ntiles - 1) * kGvCols;
#pragma unroll
        for (int j = 0; j < kUnits; ++j) {
            const int e = min(kGvLoaders * j + lt, kGvRows * kUpr - 1);
            const int row = min(rbase + e / kUpr, sg.r1 - 1), c = min(c0 + kPer * (e % kUpr), cols - kPer);
            r[j] = *reinterpret_cast<const uint4*>(sg.w + ((size_t)row * cols + c) * kSize);
        }
    };
    auto stage = [&](const uint4(&r)[kUnits], int buf) {
#pragma unroll
        for (int j = 0; j < kUnits; ++j) {
            const int e = min(kGvLoaders * j + lt, kGvRows * kUpr - 1);  // past the tile: the last unit again
            float f[kPer];
            widen<DT>(r[j], f);
            float4* d = reinterpret_cast<float4*>(&ws[buf][(e / kUpr) * kGvStride + kPer * (e % kUpr)]);
#pragma unroll
            for (int i = 0; i < kPer / 4; ++i) d[i] = make_float4(f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]);
        }
    };
    auto warm = [&](int t) {  // one scalar load per 64-byte line of tile t's activations
        if (wave != 1) return;
        uint32_t v[16];
        const_u32_ptr p = (const_u32_ptr)x;
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = p[min(t * kGvCols + 16 * i, cols - 1)];
#pragma unroll
        for (int i = 0; i < 16; i += 8)
            asm volatile("" ::"s"(v[i]), "s"(v[i + 1]), "s"(v[i + 2]), "s"(v[i + 3]), "s"(v[i + 4]), "s"(v[i + 5]), "s"(v[i + 6]),
                         "s"(v[i + 7]));
    };
    load(u[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    load(u[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    warm(0);
    for (int t = 0; t < ntiles; t += 2) {  // barrier t: tile t is staged, and tile t - 1 is chained
        stage(u[0], 0);
        load(u[0], t + 2);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        warm(t + 1);
        if (t + 1 < ntiles) {  // uniform
            stage(u[1], 1);
            load(u[1], t + 3);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            warm(t + 2);
        }
    }
}

// The same for short rows, or where many rows bound it: every wave loads and stages 64 rows by 64 columns (the LDS rows
// one bank apart), the next tile's loads in flight under this one's chains, which wave 0 runs with the activation as LDS
// broadcasts. No hand-over between waves, and a third more of them loading.
template <int DT, bool ONE>
__global__ __launch_bounds__(256) void gemv_dense_plain_kernel(const uint8_t* __restrict__ w0, float* out0, const float* __restrict__ x,
                                                         const float* res, int cols, int r0, int r1, DenseSegs segs) {
    constexpr int kRows = 64, kCols = 64, kStride = kCols + 1;
    constexpr int kSize = DT == kF32 ? 4 : 2, kPer = 16 / kSize, kUpr = kCols / kPer;  // weights, units per row
    constexpr int kUnits = kRows * kUpr / 256;
    __shared__ float ws[2][kRows * kStride];
    __shared__ __align__(16) float xs[2][kCols];
    const int tid = (int)threadIdx.x;
    int rt = (int)blockIdx.x;
    const DenseSeg sg = ONE ? DenseSeg(w0, out0, r0, r1) : DenseSeg(segs, rt);
    const int rbase = sg.r0 + rt * kRows, row = rbase + tid, ntiles = (cols + kCols - 1) / kCols;
    uint4 w[kUnits];
    float4 xr = make_float4(0.f, 0.f, 0.f, 0.f);
    auto load = [&](int c0) {  // rows past r1 and columns past cols are clamped (loaded, never used)
#pragma unroll
        for (int j = 0; j < kUnits; ++j) {
            const int u = 256 * j + tid, r = min(rbase + u / kUpr, sg.r1 - 1), c = min(c0 + kPer * (u % kUpr), cols - kPer);
            w[j] = *reinterpret_cast<const uint4*>(sg.w + ((size_t)r * cols + c) * kSize);
        }
        if (tid < kCols / 4) xr = *reinterpret_cast<const float4*>(x + min(c0 + 4 * tid, cols - 4));
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int j = 0; j < kUnits; ++j) {
            const int u = 256 * j + tid;
            float f[kPer];
            widen<DT>(w[j], f);
            float* d = &ws[buf][(u / kUpr) * kStride + kPer * (u % kUpr)];
#pragma unroll
            for (int e = 0; e < kPer; ++e) d[e] = f[e];
        }
        if (tid < kCols / 4) reinterpret_cast<float4*>(xs[buf])[tid] = xr;
    };
    const bool run = tid < kRows && row < sg.r1;
    const float rv = res && run ? res[row] : 0.0f;
    float acc = 0.0f;
    load(0);
    stage(0);
    __syncthreads();
    for (int t = 0; t < ntiles; ++t) {
        const int buf = t & 1;
        if (t + 1 < ntiles) load((t + 1) * kCols);
        if (run) {
            const float* wrow = &ws[buf][tid * kStride];
            const float* xt = xs[buf];
            if (cols - t * kCols >= kCols) {
#pragma unroll
                for (int c = 0; c < kCols; ++c) acc = __builtin_fmaf(wrow[c], xt[c], acc);
            } else {  // cols % 32 == 0
#pragma unroll
                for (int c = 0; c < kCols / 2; ++c) acc = __builtin_fmaf(wrow[c], xt[c], acc);
            }
        }
        if (t + 1 < ntiles) stage(buf ^ 1);
        __syncthreads();
    }
    if (run) sg.out[row] = res ? rv + acc : acc;
}

namespace {
constexpr int kMmTile = 32, kMmCols = 64;
}

template <int DT>
__global__ __launch_bounds__(256) void matmul_dense_kernel(DenseSegs segs, int cols, const float* __restrict__ x, int ldx,
                                                           int n, int n_tg) {
    constexpr int kSize = DT == kF32 ? 4 : 2, kPer = 16 / kSize, kUpr = kMmCols / kPer;
    constexpr int kWu = kMmTile * kUpr / 256, kXu = kMmTile * kMmCols / 4 / 256;  // units per thread: 2 / 1 and 2
    // [buffer][16 columns][row or token tile][k step row * 16 + row or token] -> 4 k steps
    __shared__ float4 wt[2][kMmCols / 16][2][64], xt[2][kMmCols / 16][2][64];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroups of one row tile run on one XCD, whose L2 the weights they share stay in
    const int Gd = (int)gridDim.x, pid = (int)blockIdx.x, per = Gd / 8, rem = Gd % 8;
    const int logical = (pid % 8) * per + min(pid % 8, rem) + pid / 8;
    int rt = logical / n_tg;
    const int tbase = logical % n_tg * kMmTile;
    const DenseSeg sg(segs, rt);
    const int rbase = sg.r0 + rt * kMmTile;
    uint4 w[2][kWu];
    float4 xv[2][kXu];
    auto load = [&](uint4(&a)[kWu], float4(&b)[kXu], int c0) {  // rows, tokens and columns past the end are clamped
#pragma unroll
        for (int j = 0; j < kWu; ++j) {
            const int e = 256 * j + tid, row = min(rbase + e / kUpr, sg.r1 - 1);
            a[j] = *reinterpret_cast<const uint4*>(sg.w + ((size_t)row * cols + min(c0 + kPer * (e % kUpr), cols - kPer)) * kSize);
        }
#pragma unroll
        for (int j = 0; j < kXu; ++j) {
            const int e = 256 * j + tid, tok = min(tbase + e / 16, n - 1);
            b[j] = *reinterpret_cast<const float4*>(x + (size_t)tok * ldx + min(c0 + 4 * (e % 16), cols - 4));
        }
    };
    auto stage = [&](const uint4(&a)[kWu], const float4(&b)[kXu], int buf) {
#pragma unroll
        for (int j = 0; j < kWu; ++j) {
            const int e = 256 * j + tid, row = e / kUpr, c = kPer * (e % kUpr);
            float f[kPer];
            widen<DT>(a[j], f);
            float* d = reinterpret_cast<float*>(&wt[buf][c / 16][row / 16][row % 16]) + c / 4 % 4;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if constexpr (DT == kF32)
                    d[64 * k] = f[k];
                else
                    *reinterpret_cast<float2*>(d + 64 * k) = make_float2(f[k], f[4 + k]);
            }
        }
#pragma unroll
        for (int j = 0; j < kXu; ++j) {
            const int e = 256 * j + tid, tok = e / 16, c = 4 * (e % 16);
            float* d = reinterpret_cast<float*>(&xt[buf][c / 16][tok / 16][tok % 16]) + c / 4 % 4;
            d[0] = b[j].x;
            d[64] = b[j].y;
            d[128] = b[j].z;
            d[192] = b[j].w;
        }
    };
    const int wr = wave >> 1, wc = wave & 1, nchunk = (cols + kMmCols - 1) / kMmCols;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    load(w[0], xv[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    load(w[1], xv[1], kMmCols);
    __builtin_amdgcn_sched_barrier(0);
    stage(w[0], xv[0], 0);
    load(w[0], xv[0], 2 * kMmCols);
    __syncthreads();
    auto chunk = [&](auto uc, int c) {
        constexpr int U = decltype(uc)::value;
        float4 a[kMmCols / 16], b[kMmCols / 16];
#pragma unroll
        for (int i = 0; i < kMmCols / 16; ++i) {
            a[i] = wt[U][i][wr][lane];
            b[i] = xt[U][i][wc][lane];
        }
        __builtin_amdgcn_sched_barrier(0);
        if (c + 1 < nchunk) {  // uniform
            stage(w[U ^ 1], xv[U ^ 1], U ^ 1);
            load(w[U ^ 1], xv[U ^ 1], (c + 3) * kMmCols);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kMmCols / 16; ++i) {
            if (c * kMmCols + 16 * i < cols) {  // uniform; cols % 32 == 0
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].x, b[i].x, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].y, b[i].y, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].z, b[i].z, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].w, b[i].w, acc, 0, 0, 0);
            }
        }
        __syncthreads();
    };
    for (int c = 0; c < nchunk; c += 2) {
        chunk(std::integral_constant<int, 0>{}, c);
        if (c + 1 < nchunk) chunk(std::integral_constant<int, 1>{}, c + 1);
    }
    const int tok = tbase + 16 * wc + (lane & 15);
    if (tok < n) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = rbase + 16 * wr + 4 * (lane >> 4) + i;
            if (row < sg.r1) sg.out[(size_t)tok * sg.ldo + row] = acc[i];
        }
    }
}

// The one-token launch. 64 rows per workgroup where a launch has so many workgroups of 16 that their starts and loads,
// not their chains, bound it (F16 30000x1024 18.5 us with 16, 14.9 with 64; F32 16384x448 8.3 and 6.7; F16 151936x896 68
// and 53), 16 below and for long rows (F16 16384x14336 100 us with 16, 192 with 64; F32 4096x896 7.0 and 8.1, 32768x8192
// 241 and 256). The plain kernel
//   for a tile of columns or half (F32 20000x32 2.5 us, 2.8 with loading waves; 128x64 2.1 and 2.25; F16 8192x32 2.40 and
//     2.44, 8192x64 2.54 and 2.47),
//   for short F32 rows by the tens of thousands (100000x128 10.9 and 12.7; 12000x128 3.6 and 3.5, 100000x256 21.5 and
//     20.4),
//   where two to four workgroups share a CU in one round (F32 45000x448 16.0 and 16.8, 16384x448 7.4 and 6.7, 80000x1024
//     70 and 60; F16 60000x192 6.1 and 6.6, 60000x448 11.7 and 11.9, 32768x256 5.6 and 5.2, 80000x192 8.3 and 8.1), and
//   for long F32 rows that workgroups of 16 would take in a round and a half, four to a CU (24000x8192 172 and 182 us,
//     28000x8192 224 and 216).
struct GemvForm {
    int rows;  // per workgroup
    bool plain;
};
static GemvForm gemv_form(int dtype, int rows, int cols) {
    const long cus = device_cus();
    const bool f32 = dtype == kF32;
    const bool one_round = rows > 128 * cus && rows <= 256 * cus && cols <= (f32 ? 1024 : 256);
    const bool uneven = f32 && cols >= 8192 && rows > 64 * cus && rows <= 96 * cus;
    if (cols <= (f32 ? 64 : 32) || one_round || uneven || (f32 && rows > 64 * cus && cols <= 192)) return {64, true};
    return {cols < 8192 && (rows >= 128 * cus || (rows >= 32 * cus && cols < 4096)) ? 64 : 16, false};
}

hipError_t launch_dense_segs(const MmOut* m, int n_mats, const float* x, int ldx, int n, const float* res, hipStream_t s) {
    if (n_mats < 1 || n_mats > 3 || (res && (n != 1 || n_mats != 1))) return hipErrorInvalidValue;
    const qh_tensor& W = *m[0].W;
    DenseSegs sg{};
    int tiles = 0, rows = 0;
    for (int i = 0; i < n_mats; ++i) rows += m[i].r1 - m[i].r0;
    const GemvForm form = gemv_form(W.dtype, rows, W.cols);
    const int tile = n > 1 ? kMmTile : form.rows;
    for (int i = 0; i < n_mats; ++i) {
        if (m[i].W->dtype != W.dtype || m[i].W->cols != W.cols) return hipErrorInvalidValue;
        sg.w[i] = static_cast<const uint8_t*>(m[i].W->data);
        sg.out[i] = m[i].out;
        sg.ldo[i] = m[i].ldo;
        sg.r0[i] = m[i].r0;
        sg.r1[i] = m[i].r1;
        sg.tiles[i] = (m[i].r1 - m[i].r0 + tile - 1) / tile;
        tiles += sg.tiles[i];
    }
    if (W.dtype != kF32 && W.dtype != kF16) return hipErrorInvalidValue;
    if (n == 1) {
        const dim3 grid((unsigned)tiles);
        auto launch = [&](auto dt, auto one) {
            constexpr int DT = decltype(dt)::value;
            constexpr bool ONE = decltype(one)::value;
            if (form.plain)
                qh_launch((gemv_dense_plain_kernel<DT, ONE>), grid, dim3(256), 0, s, sg.w[0], sg.out[0], x, res, W.cols,
                          sg.r0[0], sg.r1[0], sg);
            else if (tile == 16)
                qh_launch((gemv_dense_kernel<DT, 16, ONE>), grid, dim3(256), 0, s, sg.w[0], sg.out[0], x, res, W.cols,
                          sg.r0[0], sg.r1[0], sg);
            else
                qh_launch((gemv_dense_kernel<DT, 64, ONE>), grid, dim3(256), 0, s, sg.w[0], sg.out[0], x, res, W.cols,
                          sg.r0[0], sg.r1[0], sg);
        };
        auto typed = [&](auto one) {
            if (W.dtype == kF32)
                launch(std::integral_constant<int, kF32>{}, one);
            else
                launch(std::integral_constant<int, kF16>{}, one);
        };
        if (n_mats == 1)
            typed(std::true_type{});
        else
            typed(std::false_type{});
        return hipGetLastError();
    }
    const int n_tg = (n + kMmTile - 1) / kMmTile;
    if (W.dtype == kF32)
        qh_launch(matmul_dense_kernel<kF32>, dim3((unsigned)(tiles * n_tg)), dim3(256), 0, s, sg, W.cols, x, ldx, n, n_tg);
    else
        qh_launch(matmul_dense_kernel<kF16>, dim3((unsigned)(tiles * n_tg)), dim3(256), 0, s, sg, W.cols, x, ldx, n, n_tg);
    return hipGetLastError();
}

hipError_t launch_gemv_dense(float* out, int ldo, const qh_tensor& W, const float* x, int ldx, int n, int r0, int r1,
                             hipStream_t s) {
    const MmOut m{&W, out, ldo, r0, r1};
    return launch_dense_segs(&m, 1, x, ldx, n, nullptr, s);
}

}  // namespace qh
