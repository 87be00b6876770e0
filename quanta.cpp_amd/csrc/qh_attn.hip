// Attention of a prefill stack over the f16 KV cache (reference model.cpp:115-137, ops_ref.cpp:201-226): the same
// arithmetic in the same order as the decoder's other attention kernels, for n tokens whose cache rows are all stored
// already (kv_store_kernel).
//
// Both chains of the definition, a score's s = fma(q_i, k_i, s) over the dimensions and an output's
// o = fma(a_j, v_j, o) over the positions, are matrix products summed in order, and the f32 matrix instructions sum in
// order: each of their k steps is one fused multiply-add, rounded once, subnormals kept, so a 16x16x4 product equals
// four v_fma_f32 per element bit for bit (tests/test_gpu_dense.py: f32 and f16 weights over their whole range, infinite
// and NaN ones among them, against multiply-add chains on the CPU; tests/test_gpu_stack_attention.py: all shapes on this
// file's operands, with infinite keys and values). They run 32 multiply-adds per cycle and SIMD with one
// dependent accumulator; v_fma_f32 with a scalar, DPP or f16 operand runs 15, and with its operands broadcast from
// LDS the LDS bounds it at about 5.
//
// The rows of both products are (token, query head) pairs of one KV head, numbered token * G + head-in-group (G query
// heads share a KV head). Up to kShortRows rows one launch does everything (attn_short_kernel); beyond, the scores go
// through a device workspace, pairs in groups of 64:
//   attn_scores_kernel   s_j * scale, and each wave's maximum per pair
//   attn_softmax_kernel  e_j = expf(s_j - max) in place, the sum in position order, 1 / sum
//   attn_values_kernel   out_i = chain of fma(e_j * inv, v_ji, out_i), quantized per 32 dimensions
// Scores in the workspace: [n_kv * groups][row / 16][pair / 16][row % 4][pair % 16][row / 4 % 4], so that a lane's 16
// bytes are its operand of four 16x16x4 products.
//
// Measured per layer (14 heads, 2 KV heads, head_dim 64) against one token to a wave, lane per position for the scores
// and per dimension for the outputs, weights as LDS broadcasts: 512 tokens 35 -> 24 us (26 before the exponentials lost
// their branches, which is what the comparisons below were measured against), 1,024 tokens 108 -> 55 us; 1,024 tokens at
// position 1,024 576 -> 127 us, 952 at 2,048 811 -> 170 us (scores 60, softmax 50, values 60). Stacks of few workgroups
// go elsewhere (few_workgroups, qh_decoder.hip).
#include "qh_device.h"
#include "qh_internal.h"

namespace qh {

namespace {

typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
__device__ __forceinline__ v4u ld4(const void* p) { return *reinterpret_cast<const v4u*>(p); }
__device__ __forceinline__ float half_of(uint32_t w, int hi) {
    return f16_to_f32((uint16_t)(hi ? w >> 16 : w & 0xffffu));
}

constexpr int kSoftWaves = 16;   // waves of a softmax workgroup
constexpr int kSoftTile = 256;   // positions per softmax pass (16 per wave)
constexpr int kRowPad = 32;      // the workspace's rows per pair group are a multiple of this

// Pair p of KV head kvh (past the last: the last again, computed and never stored): its token, head and cache rows.
struct Pair {
    int token, head, rows;
    __device__ __forceinline__ Pair(const AttnStack& a, int kvh, int p) {
        const int G = a.n_heads / a.n_kv;
        p = min(p, a.n * G - 1);
        token = p / G;
        head = kvh * G + (p - token * G);
        rows = a.pos0 + token + 1;
    }
};
// Cache rows of pair p alone (uniform p: the first or last of a group).
__device__ __forceinline__ int pair_rows(const AttnStack& a, int p) {
    const int G = a.n_heads / a.n_kv;
    return a.pos0 + min(p, a.n * G - 1) / G + 1;
}

// Scores of one pair group: each of the workgroup's 4 waves takes pt positions, 32 at a time, as the product
// [32 positions][HD] . [HD][64 pairs] (two v_mfma_f32_32x32x2_f32 per two dimensions). The rotated queries stay in
// registers, the next 32 positions' keys load while this product runs. Lane l holds pair l % 32 of each half group,
// register i position 8 (i / 4) + 4 (l / 32) + i % 4.
template <int HD>
__global__ __launch_bounds__(256) void attn_scores_kernel(AttnStack a, int ng, int pt, int n_pt) {
    constexpr int HALF = HD / 2, CPR = HD / 8, QS = HD + 1;
    __shared__ float qs[64 * QS];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kvh = (int)blockIdx.y / ng, g = ng - 1 - (int)blockIdx.y % ng;  // the longest groups first
    const int hi = pair_rows(a, g * 64 + 63);
    if (4 * (int)blockIdx.x * pt >= hi) return;
    const int tile = 4 * (int)blockIdx.x + wave, j0 = tile * pt, j1 = min(j0 + pt, (hi + 31) & ~31);
    const int li = lane & 31, lh = lane >> 5;
    // K chunk c of position j, 16 bytes: [n_kv][HD / 8][ctx]; positions past the context repeat its last
    const char* kb = reinterpret_cast<const char*>(a.kc) + (size_t)kvh * CPR * a.ctx * 16;
    const size_t cstep = (size_t)a.ctx * 16;
    v4u k[CPR];
    auto load = [&](int c, int j) { k[c] = ld4(kb + c * cstep + (size_t)min(j + li, a.ctx - 1) * 16); };
#pragma unroll
    for (int c = 0; c < CPR; ++c) load(c, j0);
    {  // q with bias, rotated (model.cpp:183-195, ops_ref.cpp:201-214): 4 threads per pair
        const Pair pr(a, kvh, g * 64 + (tid & 63));
        const float* row = a.q + ((size_t)pr.token * a.n_heads + pr.head) * HD;
        const float* crow = a.cs + (size_t)(pr.rows - 1) * HD;
        const float* b = a.bq ? a.bq + pr.head * HD : nullptr;
        float* dst = qs + (tid & 63) * QS;
#pragma unroll
        for (int n = 0; n < HALF / 16; ++n) {
            const int i = 4 * (4 * n + wave);
            const float4 u4 = *reinterpret_cast<const float4*>(row + i), v4 = *reinterpret_cast<const float4*>(row + HALF + i);
            const float4 c0 = *reinterpret_cast<const float4*>(crow + 2 * i), c1 = *reinterpret_cast<const float4*>(crow + 2 * i + 4);
            float u[4] = {u4.x, u4.y, u4.z, u4.w}, v[4] = {v4.x, v4.y, v4.z, v4.w};
            const float c[4] = {c0.x, c0.z, c1.x, c1.z}, s[4] = {c0.y, c0.w, c1.y, c1.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (b) {
                    u[e] = u[e] + b[i + e];
                    v[e] = v[e] + b[i + e + HALF];
                }
                dst[i + e] = __builtin_fmaf(u[e], c[e], -(v[e] * s[e]));
                dst[HALF + i + e] = __builtin_fmaf(v[e], c[e], u[e] * s[e]);
            }
        }
    }
    __syncthreads();
    if (j0 >= hi) return;  // uniform per wave; nothing below synchronises across waves
    float q[2][HALF];  // dimensions 2 t + lh of pairs li and 32 + li
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < HALF; ++t) q[h][t] = qs[(32 * h + li) * QS + 2 * t + lh];
    const int rows[2] = {Pair(a, kvh, g * 64 + li).rows, Pair(a, kvh, g * 64 + 32 + li).rows};
    const int lo = pair_rows(a, g * 64), shift = 16 * lh;
    const float scale = 1.0f / __builtin_sqrtf((float)HD);
    const size_t gi = (size_t)(kvh * ng + g);
    float4* out = reinterpret_cast<float4*>(a.s) + gi * (a.rs / 4) * 64 + (li >> 4) * 64 + lh * 32 + (li & 15);
    float mx[2] = {-__builtin_inff(), -__builtin_inff()};
    for (int j = j0; j < j1; j += 32) {
        v16f acc[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.0f;
#pragma unroll
        for (int c = 0; c < CPR; ++c) {
            float kf[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) kf[d] = f16_to_f32((uint16_t)((k[c][d] >> shift) & 0xffffu));
            load(c, min(j + 32, j1 - 32));
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[d], q[0][4 * c + d], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[d], q[1][4 * c + d], acc[1], 0, 0, 0);
            }
        }
        auto finish = [&](auto masked) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float s = acc[h][i] * scale, m = __builtin_fmaxf(s, mx[h]);  // NaN scores never win
                    mx[h] = !decltype(masked)::value || j + 8 * (i / 4) + 4 * lh + (i & 3) < rows[h] ? m : mx[h];
                    acc[h][i] = s;
                }
                // lanes 0-31 hold steps 0 and 2 of each 16 positions, lanes 32-63 steps 1 and 3, at all four rows:
                // exchanged, lanes 0-31 hold the four steps at rows 0 and 1, lanes 32-63 at rows 2 and 3
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        float v[4];
#pragma unroll
                        for (int n = 0; n < 2; ++n) {
                            const float lo2 = acc[h][8 * b + 4 * n + k], hi2 = acc[h][8 * b + 4 * n + k + 2];
                            const auto w = __builtin_amdgcn_permlane32_swap(
                                __builtin_bit_cast(uint32_t, lo2), __builtin_bit_cast(uint32_t, hi2), false, false);
                            v[2 * n] = __builtin_bit_cast(float, (uint32_t)w[0]);
                            v[2 * n + 1] = __builtin_bit_cast(float, (uint32_t)w[1]);
                        }
                        out[(size_t)(j / 16 + b) * 256 + 128 * h + 16 * k] = make_float4(v[0], v[1], v[2], v[3]);
                    }
            }
        };
        if (j + 32 <= lo)  // uniform: rows of every pair
            finish(std::false_type{});
        else
            finish(std::true_type{});
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t u = __builtin_bit_cast(uint32_t, mx[h]);
        const auto w = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        const float x = __builtin_bit_cast(float, (uint32_t)w[0]), y = __builtin_bit_cast(float, (uint32_t)w[1]);
        if (lh == 0) a.pm[(gi * n_pt + tile) * 64 + 32 * h + li] = y > x ? y : x;
    }
}

// Softmax of half a pair group (ops_ref.cpp:216-226): the maximum over the score waves' maxima (independent of the
// order of comparison), the exponentials 256 positions a pass (a wave takes 16 positions of 16 pairs at a time), written
// back and to LDS, where one wave (another each pass) adds them to the pairs' sums in position order while the others
// go on with the next pass. The exponentials bound it (about 40 instructions each).
__global__ __launch_bounds__(64 * kSoftWaves) void attn_softmax_kernel(AttnStack a, int ng, int pt, int n_pt) {
    constexpr int kBlocks = kSoftTile / 16, kUnits = kBlocks * 2 / kSoftWaves;  // 16-position blocks, units per wave
    __shared__ float4 es[2][kBlocks][2][64];
    __shared__ float red[kSoftWaves][64];
    __shared__ float run[32];
    __shared__ uint64_t exptab[32];
    ExpTab et;
    et.load();
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int gg = 2 * ng - 1 - (int)blockIdx.x % (2 * ng), kvh = (int)blockIdx.x / (2 * ng), g = gg >> 1, half = gg & 1;
    const int li = lane & 31, lh = lane >> 5, p0 = gg * 32;
    if (p0 >= a.n * (a.n_heads / a.n_kv)) return;
    const int hi = pair_rows(a, p0 + 31), nb = (hi + 15) / 16;
    const size_t gi = (size_t)(kvh * ng + g);
    // this wave's units: pairs 16 sub .. of the half group, blocks b0 + 8 k of each pass
    const int sub = wave & 1, b0 = wave >> 1, rows = pair_rows(a, p0 + 16 * sub + (lane & 15));
    float4* s = reinterpret_cast<float4*>(a.s) + gi * (a.rs / 4) * 64 + (2 * half + sub) * 64 + lane;  // + 256 per block
    float4 cur[kUnits];
    auto load = [&](float4(&v)[kUnits], int t) {
#pragma unroll
        for (int k = 0; k < kUnits; ++k) v[k] = s[(size_t)min(t * kBlocks + b0 + kSoftWaves / 2 * k, nb - 1) * 256];
    };
    load(cur, 0);
    float mx = -__builtin_inff(), part = mx;  // of this lane's pair in the units; of pair li
    const int tiles = (hi + pt - 1) / pt;
    for (int t = 2 * wave + lh; t < tiles; t += 2 * kSoftWaves) {
        const float m = a.pm[(gi * n_pt + t) * 64 + half * 32 + li];
        part = m > part ? m : part;
    }
    red[wave][lane] = part;
    et.store(exptab);
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 2 * kSoftWaves; ++w) {
        const float m = red[w >> 1][(w & 1) * 32 + 16 * sub + (lane & 15)];
        mx = m > mx ? m : mx;
    }
    const int passes = (hi + kSoftTile - 1) / kSoftTile;
    for (int t = 0; t < passes; ++t) {
        float4 nxt[kUnits];
        load(nxt, t + 1 < passes ? t + 1 : t);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < kUnits; ++k) {
            const int b = b0 + kSoftWaves / 2 * k, bg = t * kBlocks + b;
            if (bg < nb) {  // uniform
                const float x[4] = {cur[k].x, cur[k].y, cur[k].z, cur[k].w};
                float e[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    e[i] = dev_expf_nonpos(x[i] - mx, exptab);
                    e[i] = 16 * bg + 4 * i + (lane >> 4) < rows ? e[i] : 0.0f;  // +0 leaves a pair's sum as it is
                }
                const float4 v = make_float4(e[0], e[1], e[2], e[3]);
                s[(size_t)bg * 256] = v;
                es[t & 1][b][sub][lane] = v;
            }
        }
        __syncthreads();
        if (wave == t % kSoftWaves) {  // lane li (and its copy 32 + li): pair li
            float sum = t ? run[li] : 0.0f;
            const int cb = min(kBlocks, nb - t * kBlocks);
#pragma unroll 2
            for (int b = 0; b < cb; ++b) {
                float4 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = es[t & 1][b][li >> 4][16 * k + (li & 15)];
#pragma unroll
                for (int k = 0; k < 4; ++k) sum = sum + v[k].x;
#pragma unroll
                for (int k = 0; k < 4; ++k) sum = sum + v[k].y;
#pragma unroll
                for (int k = 0; k < 4; ++k) sum = sum + v[k].z;
#pragma unroll
                for (int k = 0; k < 4; ++k) sum = sum + v[k].w;
            }
            run[li] = sum;
            if (t + 1 == passes && lh == 0) a.inv[gi * 64 + half * 32 + li] = 1.0f / sum;
        }
#pragma unroll
        for (int k = 0; k < kUnits; ++k) cur[k] = nxt[k];
    }
}

// Outputs of one pair group for 32 dimensions (one quantization block): wave w takes pairs 16 w .. of the group as the
// product [16 pairs][positions] . [positions][32 dimensions], two v_mfma_f32_16x16x4_f32 per 4 positions. The values
// go through LDS, 64 positions at a time, widened and in operand order (a lane's 4 k steps in one 16-byte read), staged
// once for the four waves; the weights are 16 bytes of a lane's own per 16 positions. Both load two tiles ahead (memory takes
// about two tiles' products to answer). Lane l holds dimension l % 16 of each half block, register i pair
// 4 (l / 16) + i.
constexpr int kValTile = 64;
template <int HD>
__global__ __launch_bounds__(256) void attn_values_kernel(AttnStack a, int ng) {
    constexpr int kSteps = kValTile / 4;
    __shared__ float4 vs[2][kValTile / 16][2][64];  // [16 positions][half block][k step row * 16 + dimension] -> 4 steps
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kvh = (int)blockIdx.x / ng, g = ng - 1 - (int)blockIdx.x % ng, d0 = 32 * (int)blockIdx.y;
    const int G = a.n_heads / a.n_kv, np = a.n * G, p0 = g * 64 + 16 * wave;
    const int li = lane & 15, lq = lane >> 4;
    const int lo = pair_rows(a, p0), hi = pair_rows(a, p0 + 15);
    const size_t gi = (size_t)(kvh * ng + g);
    const float4* sw = reinterpret_cast<const float4*>(a.s) + gi * (a.rs / 4) * 64 + 64 * wave;  // + 256 per 16 positions
    const float inv = a.inv[gi * 64 + 16 * wave + li];
    // value block b of 8 positions, 16 bytes per dimension: [ctx / 8][n_kv * HD]; thread: dimension tid % 32, block
    // tid / 32 of the tile
    const char* vb = reinterpret_cast<const char*>(a.vc) + ((size_t)kvh * HD + d0) * 16;
    const size_t vstep = (size_t)a.n_kv * HD * 16;
    const int last = (pair_rows(a, g * 64 + 63) - 1) / 8;
    auto vload = [&](int t) { return ld4(vb + (size_t)min(t * (kValTile / 8) + tid / 32, last) * vstep + (tid & 31) * 16); };
    auto stage = [&](const v4u& v, int buf) {
        const int b = tid / 32, dl = tid & 15;
        float* dst = reinterpret_cast<float*>(&vs[buf][b >> 1][(tid >> 4) & 1][dl]) + 2 * (b & 1);
#pragma unroll
        for (int k = 0; k < 4; ++k)  // positions k and 4 + k of the block: row k of two steps
            *reinterpret_cast<float2*>(dst + 64 * k) = make_float2(half_of(v[k / 2], k & 1), half_of(v[2 + k / 2], k & 1));
    };
    struct Weights {
        float4 p[kSteps / 4];
    };
    auto wload = [&](Weights& w, int t) {  // up to three tiles past the group's rows: kWsPad
        const float4* p = sw + (size_t)t * (kValTile * 16) + lane;
#pragma unroll
        for (int k = 0; k < kSteps / 4; ++k) w.p[k] = p[256 * k];
    };
    v4f acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    Weights w[2];
    v4u v[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {  // in the order of the loop, so that its waits count
        v[u] = vload(u);
        wload(w[u], u);
        __builtin_amdgcn_sched_barrier(0);
    }
    stage(v[0], 0);
    v[0] = vload(2);
    __syncthreads();
    // Tile t (ring slot U = t % 2): stages tile t + 1, loads t + 2 and t + 3. FULL: all its positions are rows of every
    // pair of the group; else the wave's steps that are rows of its pairs.
    auto tile = [&](auto uc, auto full, int t) {
        constexpr int U = decltype(uc)::value;
        float4 x[2][2] = {{vs[U][0][0][lane], vs[U][0][1][lane]}, {}};
        __builtin_amdgcn_sched_barrier(0);
        stage(v[U ^ 1], U ^ 1);
        v[U ^ 1] = vload(t + 3);
        __builtin_amdgcn_sched_barrier(0);
        const int steps = decltype(full)::value ? kSteps : lo / 4 - t * kSteps;
        float p[kSteps];
#pragma unroll
        for (int k = 0; k < kSteps / 4; ++k) {
            p[4 * k] = w[U].p[k].x * inv;
            p[4 * k + 1] = w[U].p[k].y * inv;
            p[4 * k + 2] = w[U].p[k].z * inv;
            p[4 * k + 3] = w[U].p[k].w * inv;
        }
        wload(w[U], t + 2);
#pragma unroll
        for (int b = 0; b < kSteps / 4; ++b) {  // the next 4 steps' values are read under this product
            if (b + 1 < kSteps / 4) {
                x[(b + 1) & 1][0] = vs[U][b + 1][0][lane];
                x[(b + 1) & 1][1] = vs[U][b + 1][1][lane];
            }
            __builtin_amdgcn_sched_barrier(0);
            if (decltype(full)::value || 4 * b < steps) {  // uniform per wave
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if (decltype(full)::value || 4 * b + k < steps) {
#pragma unroll
                        for (int d = 0; d < 2; ++d) {
                            const float4 y = x[b & 1][d];
                            acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                p[4 * b + k], k == 0 ? y.x : k == 1 ? y.y : k == 2 ? y.z : y.w, acc[d], 0, 0, 0);
                        }
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };
    using std::integral_constant;
    const int full = pair_rows(a, g * 64) / kValTile;                                // uniform
    const int tiles = (pair_rows(a, g * 64 + 48) / 4 * 4 + kValTile - 1) / kValTile;  // of the last wave
    int t = 0;
    for (; t + 2 <= full; t += 2) {
        tile(integral_constant<int, 0>{}, std::true_type{}, t);
        tile(integral_constant<int, 1>{}, std::true_type{}, t + 1);
    }
    for (; t < tiles; t += 2) {
        tile(integral_constant<int, 0>{}, std::false_type{}, t);
        if (t + 1 < tiles) tile(integral_constant<int, 1>{}, std::false_type{}, t + 1);
    }
    if (p0 >= np) return;  // uniform per wave; nothing below synchronises across waves
    // The rows past the first pair's whole steps, for the pairs that have them (a later token's row is not an earlier
    // one's, and 0 times an infinite value is not 0): lane l's pairs 4 lq + i, 4 positions at a time.
    int rows[4];
    float pinv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        rows[i] = pair_rows(a, p0 + 4 * lq + i);
        pinv[i] = a.inv[gi * 64 + 16 * wave + 4 * lq + i];
    }
    const float* sp = reinterpret_cast<const float*>(sw + 4 * lq);
    for (int j = lo & ~3; j < hi; j += 4) {
        float e4[4][4];  // [pair][position]
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) e4[i][k] = sp[(size_t)(j / 16) * 1024 + 4 * (16 * k + i) + ((j >> 2) & 3)];
        uint2 x2[2];
#pragma unroll
        for (int d = 0; d < 2; ++d) x2[d] = *reinterpret_cast<const uint2*>(vb + (size_t)(j / 8) * vstep + 256 * d + 16 * li + (j & 4) * 2);
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const float x = half_of(k < 2 ? x2[d].x : x2[d].y, k & 1);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float r = __builtin_fmaf(e4[i][k] * pinv[i], x, acc[d][i]);
                    acc[d][i] = j + k < rows[i] ? r : acc[d][i];
                }
            }
    }
    // quantize_q8 (ops_ref.cpp:69-83) of each pair's 32 dimensions: 16 lanes, two values each
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int p = p0 + 4 * lq + i;
        const float x0 = acc[0][i], x1 = acc[1][i];
        const float m = dpp_max<0x140>(max8_lanes(__builtin_fmaxf(__builtin_fabsf(x0), __builtin_fabsf(x1))));
        const float sc = m / 127.0f;
        const float r = sc > 0.0f ? 1.0f / sc : 0.0f;
        if (p < np) {
            const int token = p / G, col = (kvh * G + (p - token * G)) * HD + d0;
            const size_t at = (size_t)token * a.n_heads * HD + col;
            a.oq[at + li] = (int8_t)(int)round_half_away(x0 * r);
            a.oq[at + 16 + li] = (int8_t)(int)round_half_away(x1 * r);
            if (li == 0) a.od[at / QK] = sc;
            if (a.of) {
                a.of[at + li] = x0;
                a.of[at + 16 + li] = x1;
            }
        }
    }
}

// All of it in one launch for up to kShortRows rows: a workgroup takes 16 pairs and keeps their scores in LDS (64 bytes
// per row, in the order of a 16x16x4 product's operand; 1,024 rows leave two workgroups to a CU). Its 4 waves score 16
// positions at a time each (the product [16 positions][HD] . [HD][16 pairs]), exponentiate, one sums, and each takes
// HD / 4 of the output dimensions. Keys and values come straight from the cache as whole 16-byte units, the next unit's
// load in flight, four lanes to a unit, each selecting its two halves (as 4-byte loads, which the address unit serves
// no faster, 512 tokens took 39 us against 26). Serial latency bounds it: 8 or 16 waves a workgroup measured no faster.
// Up to 1,024 rows it is ahead of the three launches (512 tokens 26 against 32 us and two launches, 1,024 tokens 55
// against 70, 64 tokens at position 900 equal).
constexpr int kShortRows = 1024;
template <int HD>
__global__ __launch_bounds__(256) void attn_short_kernel(AttnStack a, int ng16) {
    constexpr int HALF = HD / 2, CPR = HD / 8, QS = HD + 1, DT = HD / 64;  // DT: 16-dimension tiles per wave
    extern __shared__ float4 es[];  // [row / 16][row % 4][pair] -> rows 4 t + row % 4, t = 0 .. 3
    __shared__ float qs[16 * QS];   // the queries, then the outputs
    __shared__ float red[4][16];
    __shared__ float sums[16];
    __shared__ uint64_t exptab[32];
    ExpTab et;
    et.load();
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kvh = (int)blockIdx.x / ng16, p0 = 16 * (ng16 - 1 - (int)blockIdx.x % ng16);  // the longest first
    const int G = a.n_heads / a.n_kv, np = a.n * G;
    const int li = lane & 15, lq = lane >> 4;
    const int lo = pair_rows(a, p0), hi = pair_rows(a, p0 + 15), nb = (hi + 15) / 16;
    // K chunk c of position j, 16 bytes: [n_kv][HD / 8][ctx] (positions past the rows repeat the last); this lane's
    // dimensions 8 c + lq and 8 c + 4 + lq are halves lq & 1 of dwords lq / 2 and 2 + lq / 2
    const char* kb = reinterpret_cast<const char*>(a.kc) + (size_t)kvh * CPR * a.ctx * 16;
    const size_t cstep = (size_t)a.ctx * 16;
    const int shift = 16 * (lq & 1);
    auto half = [&](uint32_t w) { return f16_to_f32((uint16_t)((w >> shift) & 0xffffu)); };
    const bool second = lq >= 2;
    v4u k[CPR];
    auto kload = [&](int b) {
        const char* p = kb + (size_t)min(16 * b + li, hi - 1) * 16;
#pragma unroll
        for (int c = 0; c < CPR; ++c) k[c] = ld4(p + c * cstep);
    };
    kload(min(wave, nb - 1));
    {  // q with bias, rotated (model.cpp:183-195, ops_ref.cpp:201-214): 16 threads per pair
        const Pair pr(a, kvh, p0 + tid / 16);
        const float* row = a.q + ((size_t)pr.token * a.n_heads + pr.head) * HD;
        const float* crow = a.cs + (size_t)(pr.rows - 1) * HD;
        const float* b = a.bq ? a.bq + pr.head * HD : nullptr;
        float* dst = qs + (tid / 16) * QS;
#pragma unroll
        for (int n = 0; n < HALF / 16; ++n) {
            const int i = 16 * n + (tid & 15);
            float u = row[i], v = row[HALF + i];
            const float2 c = *reinterpret_cast<const float2*>(crow + 2 * i);
            if (b) {
                u = u + b[i];
                v = v + b[i + HALF];
            }
            dst[i] = __builtin_fmaf(u, c.x, -(v * c.y));
            dst[HALF + i] = __builtin_fmaf(v, c.x, u * c.y);
        }
    }
    et.store(exptab);
    __syncthreads();
    float q[HD / 4];  // dimensions 4 t + lq of pair li
#pragma unroll
    for (int t = 0; t < HD / 4; ++t) q[t] = qs[li * QS + 4 * t + lq];
    const float scale = 1.0f / __builtin_sqrtf((float)HD);
    const int rows = pair_rows(a, p0 + li);
    float mx = -__builtin_inff();
    for (int b = wave; b < nb; b += 4) {  // register i: position 16 b + 4 lq + i of pair li
        v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
        float kf[HD / 4];
#pragma unroll
        for (int c = 0; c < CPR; ++c) {
            uint32_t w[4] = {k[c][0], k[c][1], k[c][2], k[c][3]};
            asm("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
            kf[2 * c] = half(second ? w[1] : w[0]);
            kf[2 * c + 1] = half(second ? w[3] : w[2]);
        }
        kload(min(b + 4, nb - 1));
#pragma unroll
        for (int t = 0; t < HD / 4; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t], q[t], acc, 0, 0, 0);
        float* dst = reinterpret_cast<float*>(es + 64 * b + li) + lq;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float s = acc[i] * scale;
            mx = 16 * b + 4 * lq + i < rows ? __builtin_fmaxf(s, mx) : mx;  // NaN scores never win
            dst[64 * i] = s;
        }
    }
    mx = __builtin_fmaxf(mx, __shfl_xor(mx, 16));
    mx = __builtin_fmaxf(mx, __shfl_xor(mx, 32));
    if (lane < 16) red[wave][lane] = mx;
    // the first value blocks go out under the softmax: dimension 16 (DT wave + d) + li, positions as the keys' dimensions
    const char* vb = reinterpret_cast<const char*>(a.vc) + ((size_t)kvh * HD + 16 * DT * wave + li) * 16;
    const size_t vstep = (size_t)a.n_kv * HD * 16;
    const int last = (hi - 1) / 8;
    constexpr int kAhead = 4;
    struct Vals {
        v4u w[DT][2];
    };
    auto vload = [&](int b) {
        Vals v;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const char* p = vb + (size_t)min(2 * b + h, last) * vstep;
#pragma unroll
            for (int d = 0; d < DT; ++d) v.w[d][h] = ld4(p + 256 * d);
        }
        return v;
    };
    Vals v[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {  // in the order of the loop, so that its waits count
        v[u] = vload(u);
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    mx = red[0][li];
#pragma unroll
    for (int w = 1; w < 4; ++w) mx = __builtin_fmaxf(mx, red[w][li]);
    for (int b = wave; b < nb; b += 4) {  // rows 16 b + 4 t + lq of pair li
        float4 x = es[64 * b + lane];
        float e[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            e[t] = dev_expf_nonpos(e[t] - mx, exptab);
            e[t] = 16 * b + 4 * t + lq < rows ? e[t] : 0.0f;  // +0 leaves a pair's sum as it is
        }
        es[64 * b + lane] = make_float4(e[0], e[1], e[2], e[3]);
    }
    __syncthreads();
    if (wave == 0) {  // the sum in position order (ops_ref.cpp:220-224), each pair in 4 lanes alike
        float sum = 0.0f;
        float4 x[2][4];
#pragma unroll
        for (int r = 0; r < 4; ++r) x[0][r] = es[16 * r + li];
        auto add = [&](const float4(&y)[4]) {
#pragma unroll
            for (int r = 0; r < 4; ++r) sum = sum + y[r].x;
#pragma unroll
            for (int r = 0; r < 4; ++r) sum = sum + y[r].y;
#pragma unroll
            for (int r = 0; r < 4; ++r) sum = sum + y[r].z;
#pragma unroll
            for (int r = 0; r < 4; ++r) sum = sum + y[r].w;
        };
        for (int b = 0; b < nb; b += 2) {  // a block past the last repeats it, and is not added
#pragma unroll
            for (int r = 0; r < 4; ++r) x[1][r] = es[64 * min(b + 1, nb - 1) + 16 * r + li];
            __builtin_amdgcn_sched_barrier(0);
            add(x[0]);
#pragma unroll
            for (int r = 0; r < 4; ++r) x[0][r] = es[64 * min(b + 2, nb - 1) + 16 * r + li];
            __builtin_amdgcn_sched_barrier(0);
            if (b + 1 < nb) add(x[1]);
        }
        if (lane < 16) sums[lane] = 1.0f / sum;
    }
    __syncthreads();
    const float inv = sums[li];
    v4f acc[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d) acc[d] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    const int steps = lo / 4;  // of 4 positions that are rows of every pair
    float4 x = es[lane];
    auto block = [&](auto full, int u, int b) {
        const float p[4] = {x.x * inv, x.y * inv, x.z * inv, x.w * inv};
        float vf[DT][4];
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t w[4] = {v[u].w[d][h][0], v[u].w[d][h][1], v[u].w[d][h][2], v[u].w[d][h][3]};
                asm("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
                vf[d][2 * h] = half(second ? w[1] : w[0]);
                vf[d][2 * h + 1] = half(second ? w[3] : w[2]);
            }
        v[u] = vload(b + kAhead);
        x = es[64 * min(b + 1, nb - 1) + lane];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (decltype(full)::value || 4 * b + t < steps)  // uniform
#pragma unroll
                for (int d = 0; d < DT; ++d) acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[t], vf[d][t], acc[d], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    int vbk = 0;
    for (; 4 * (vbk + kAhead) <= steps; vbk += kAhead)
#pragma unroll
        for (int u = 0; u < kAhead; ++u) block(std::true_type{}, u, vbk + u);
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
        if (4 * (vbk + u) < steps) block(std::false_type{}, u, vbk + u);  // uniform
    // The rows past the first pair's whole steps, for the pairs that have them (a later token's row is not an earlier
    // one's, and 0 times an infinite value is not 0): lane l's pairs 4 lq + i.
    for (int j = 4 * steps; j < hi; ++j) {
        const float* ep = reinterpret_cast<const float*>(es + (j / 16) * 64 + (j & 3) * 16 + 4 * lq) + (j / 4) % 4;
        float xv[DT];
#pragma unroll
        for (int d = 0; d < DT; ++d)
            xv[d] = f16_to_f32(a.vc[((size_t)(j / 8) * a.n_kv * HD + (size_t)kvh * HD + 16 * (DT * wave + d) + li) * 8 + (j & 7)]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float p = ep[4 * i] * sums[4 * lq + i];
            const bool in = j < pair_rows(a, p0 + 4 * lq + i);
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const float r = __builtin_fmaf(p, xv[d], acc[d][i]);
                acc[d][i] = in ? r : acc[d][i];
            }
        }
    }
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i) qs[(4 * lq + i) * QS + 16 * (DT * wave + d) + li] = acc[d][i];
    __syncthreads();
    for (int e = tid / 32; e < 16 * (HD / QK); e += 8) {  // quantize_q8 by 32 lanes
        const int r = e / (HD / QK), p = p0 + r, d0 = e % (HD / QK) * QK;
        if (p < np) {  // uniform per 32 lanes
            const int token = p / G;
            const size_t at = (size_t)token * a.n_heads * HD + (kvh * G + (p - token * G)) * HD + d0;
            const float y = qs[r * QS + d0 + (tid & 31)];
            if (a.of) a.of[at + (tid & 31)] = y;
            quant_block32(y, a.oq + at, a.od + at / QK);
        }
    }
}

// Workspace floats per (pair group, KV head) whose last token has `rows` rows: the scores, the score waves' maxima (at
// least 32 positions each) and the inverse sums.
constexpr size_t kWsPad = 4 * kValTile * 256;  // bytes: four tiles of rows that attn_values_kernel may load past a group's
size_t group_floats(int rs) { return 64 * ((size_t)rs + rs / 32 + 1); }
int row_stride(int rows) { return (rows + kRowPad - 1) / kRowPad * kRowPad; }

}  // namespace

// Bytes for `tokens` at the end of the context, at most kAttnWsBytes unless one token's pairs need more, which is the
// least that works (*least); 0 for a context whose every stack one launch takes.
size_t attn_stack_ws_bytes(int n_heads, int n_kv, int ctx, int tokens, size_t* least_bytes) {
    *least_bytes = 0;
    if (ctx <= kShortRows) return 0;
    const size_t G = (size_t)(n_heads / n_kv), groups = (tokens * G + 63) / 64, least = (G + 63) / 64;
    const size_t per = (size_t)n_kv * group_floats(row_stride(ctx)) * 4, fit = kAttnWsBytes / per;
    *least_bytes = per * least + kWsPad;
    return per * (groups < fit ? groups : fit > least ? fit : least) + kWsPad;
}

hipError_t launch_attention_stack(AttnStack a, int head_dim, float* ws, size_t ws_bytes, hipStream_t s) {
    const int G = a.n_heads / a.n_kv, n = a.n, pos0 = a.pos0, qd = a.n_heads * head_dim;
    const AttnStack all = a;
    if (pos0 + n <= kShortRows) {
        const int ng16 = (n * G + 15) / 16;
        const size_t lds = (size_t)((pos0 + n + 15) / 16) * 1024;
        if (head_dim == 64)
            qh_launch(attn_short_kernel<64>, dim3((unsigned)(a.n_kv * ng16)), dim3(256), lds, s, a, ng16);
        else
            qh_launch(attn_short_kernel<128>, dim3((unsigned)(a.n_kv * ng16)), dim3(256), lds, s, a, ng16);
        return hipGetLastError();
    }
    for (int t0 = 0; t0 < n; t0 += a.n) {  // as many tokens at a time as the workspace holds
        a = all;
        a.rs = row_stride(pos0 + n);
        const long fit = (long)((ws_bytes - kWsPad) / 4 / ((size_t)a.n_kv * group_floats(a.rs)));  // pair groups per KV head
        a.n = (int)(fit * 64 / G < n - t0 ? fit * 64 / G : n - t0);
        if (a.n < 1) return hipErrorInvalidValue;
        a.pos0 = pos0 + t0;
        a.q += (size_t)t0 * qd;
        a.oq += (size_t)t0 * qd;
        a.od += (size_t)t0 * (qd / QK);
        if (a.of) a.of += (size_t)t0 * qd;
        const int ng = (a.n * G + 63) / 64, rows = a.pos0 + a.n;
        // positions per score wave: a wave loads and rotates its queries once, so as many as still fill the GPU
        const long units = (long)a.n_kv * ng * (a.pos0 + a.n / 2) / 32;  // products of 32 positions, about
        const int pt = units >= 16L * device_cus() * 4 ? 128 : units >= 8L * device_cus() ? 64 : 32;
        const int n_pt = (rows + pt - 1) / pt;
        a.s = ws;
        a.pm = a.s + (size_t)a.n_kv * ng * a.rs * 64;
        a.inv = a.pm + (size_t)a.n_kv * ng * n_pt * 64;
        const dim3 gs((unsigned)((n_pt + 3) / 4), (unsigned)(a.n_kv * ng)), gx((unsigned)(a.n_kv * ng * 2));
        const dim3 gv((unsigned)(a.n_kv * ng), (unsigned)(head_dim / 32));
        if (head_dim == 64)
            qh_launch(attn_scores_kernel<64>, gs, dim3(256), 0, s, a, ng, pt, n_pt);
        else
            qh_launch(attn_scores_kernel<128>, gs, dim3(256), 0, s, a, ng, pt, n_pt);
        qh_launch(attn_softmax_kernel, gx, dim3(64 * kSoftWaves), 0, s, a, ng, pt, n_pt);
        if (head_dim == 64)
            qh_launch(attn_values_kernel<64>, gv, dim3(256), 0, s, a, ng);
        else
            qh_launch(attn_values_kernel<128>, gv, dim3(256), 0, s, a, ng);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace qh
