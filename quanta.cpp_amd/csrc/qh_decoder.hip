// GPU-resident decoder for the q4mix Qwen2-shaped model: the reference's Model::forward and forward_batch
// (engine/src/model.cpp:165-228, 349-433) with the operation order of its CPU build, so every hidden state, logit and
// greedy token is bit-identical to the reference.
//
// Decode (one token) runs five kernels per layer, each with its elementwise work fused in:
//   qkv        one launch for the q, k and v GEMVs (three row segments, same activation); every workgroup first runs
//              the layer's rmsnorm (serial FMA sum of squares, one rounded 1/sqrt) and quantizes the normed row into
//              its LDS (layer 0: the token's embedding row)                (model.cpp:179-182, ops_ref.cpp:195-199)
//   attention  one 16-wave workgroup per query head: biases, RoPE (host table of glibc powf/cosf/sinf of the
//              reference's formula), this token's f16 K/V row into the cache, scores (serial FMA dot over head_dim),
//              max, glibc-identical expf, serial sum in position order, normalise, serial weighted V sum in position
//              order, and the int8 quantization of the head's two 32-blocks of output
//                                                                         (model.cpp:115-137, 183-208, ops_ref.cpp:201-226)
//   o          GEMV and residual add                                     (model.cpp:207-209)
//   gate/up    the MLP's rmsnorm in every workgroup's prologue as above, one GEMV over the same rows of both matrices,
//              g / (1 + expf(-g)) * u, quantization                     (model.cpp:212-218, ops_ref.cpp:243-248)
//   down       GEMV and residual add                                     (model.cpp:219-221)
// then the final norm and the head (Exact Shortlist Head for top-k queries, full 8-bit head + argmax otherwise). The
// position and the token live on the device, so a decode step is a fixed launch sequence that can be captured in a HIP
// graph and replayed: the step reads the token the previous step chose, and its last kernel writes the new token,
// appends it to the output list and advances the position. A step at a position beyond the context writes nothing
// into the cache and raises bit 0 of the status word; a prompt token outside the vocabulary raises bit 1.
//
// Prefill (chunks of up to 32 tokens) uses the int8-MFMA matmul for every projection (q / k / v in one launch, gate /
// up in one launch) and an attention kernel over a (head, token) grid: a token's keys and values for the chunk's
// positions come from the chunk's own projections, so no kernel reads a cache row another workgroup of the same launch
// writes.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <type_traits>
#include <vector>

#include "qh_attn_chunk.h"
#include "qh_decoder_device.h"
#include "qh_device.h"
#include "qh_gemv.h"
#include "qh_internal.h"
#include "qh_math.h"

namespace qh {

namespace {

// Activation fill for a GEMV tile whose input is rmsnorm(x) * w quantized (the decode step's q/k/v and gate/up
// inputs): every workgroup normalises the residual row itself, while its first pass of weight loads is in flight,
// and quantizes it straight into the tile's LDS codes / scales, so no kernel of its own and no cross-workgroup
// synchronisation is needed. With eq set, the row is instead the embedding of token *tok (the first layer), and
// workgroup 0 also stores it as the residual stream x_out. tmp: LDS scratch of D + kChainPad floats (16-byte
// aligned).
struct NormAct {
    static constexpr bool kGlobalScales = false;  // the scales are computed into LDS
    const float* x;
    const int8_t* eq;
    const uint16_t* es;
    const int32_t* tok;
    int V;
    float* x_out;
    int* status;
    const float* w;
    float eps;
    int D;
    float* tmp;
    int tlk;  // timeline id of the kernel (stamps compiled in only with QH_TIMELINE)

    // The loads the norm starts from (issued before the tile's weight loads, whose issue would otherwise hold them
    // up): the residual row and its scalar-cache warm-up, and the norm weight.
    template <int R>
    struct Pre {
        RowF4<R> wr, xr;
        SegWarm warm;
    };
    // EMB: the row is the embedding of *tok (eq set); the same loads whatever the branch below, so the compiler counts
    // the outstanding loads exactly where the row is first used.
    template <int R, bool EMB>
    __device__ __forceinline__ Pre<R> begin() const {
        Pre<R> p;
        load_row<R, EMB>(p.xr, (int)threadIdx.x, D / 4);
        if (!EMB && D >= 128) p.warm = seg_warm(x, D);  // uniform
        p.wr.load(w, D / 4);
        return p;
    }

    template <bool XL, int R, bool EMB>
    __device__ __forceinline__ void fill(const Pre<R>& p, int8_t* xs, float* xds) const {
        static_assert(XL, "the normed activation is produced in LDS");
        const int tid = (int)threadIdx.x, n4 = D / 4;
        const RowF4<R>& wr = p.wr;
        const RowF4<R>& xr = p.xr;
        float4* t4 = reinterpret_cast<float4*>(tmp);
        float ss;
        if (!EMB && D >= 128) {  // uniform
            ss = seg_sum_squares(x, D, xr, p.warm, tlk);
        } else {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int i4 = tid + 256 * k;
                if (i4 < n4) {
                    t4[i4] = xr.v[k];
                    if (x_out && blockIdx.x == 0) reinterpret_cast<float4*>(x_out)[i4] = xr.v[k];
                }
            }
            __syncthreads();
            ss = lds_sum_squares(tmp, D);
        }
        const float scale = rms_scale(ss, D, eps);
        if constexpr (R == 1) {
            // thread t holds float4 t, so the 8-lane groups of quant_block_x8 are the row's 32-blocks: each thread
            // quantizes its own values, with no LDS round trip and no barrier (n4 % 8 == 0: whole groups)
            if (tid < n4) {
                float4 y = xr.v[0];
                y.x = y.x * scale * wr.v[0].x;
                y.y = y.y * scale * wr.v[0].y;
                y.z = y.z * scale * wr.v[0].z;
                y.w = y.w * scale * wr.v[0].w;
                quant_block_x8(y, xs + (tid >> 3) * QK, xds + (tid >> 3));
            }
        } else {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int i4 = tid + 256 * k;
                if (i4 < n4) {
                    float4 y = xr.v[k];
                    y.x = y.x * scale * wr.v[k].x;
                    y.y = y.y * scale * wr.v[k].y;
                    y.z = y.z * scale * wr.v[k].z;
                    y.w = y.w * scale * wr.v[k].w;
                    t4[i4] = y;
                }
            }
            __syncthreads();
            quant_row_x8(tmp, D, xs, xds);
        }
    }

    // The row to normalise into xr: the embedding of *tok (EMB) or x.
    template <int R, bool EMB>
    __device__ __forceinline__ void load_row(RowF4<R>& xr, int tid, int n4) const {
        const int nb = D / QK;
        if constexpr (EMB) {
            int t = *tok;
            const bool bad = t < 0 || t >= V;
            if (bad && tid == 0 && blockIdx.x == 0) atomicOr(status, kStatusToken);
            t = bad ? 0 : t;
            const int8_t* er = eq + (size_t)t * D;
            const uint16_t* sr = es + (size_t)t * nb;
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int i4 = min(tid + 256 * k, n4 - 1);
                const uint32_t c4 = *reinterpret_cast<const uint32_t*>(er + 4 * i4);
                const float sc = h2f(sr[i4 / (QK / 4)]);
                xr.v[k].x = bad ? 0.0f : (float)(int8_t)(c4 & 0xff) * sc;
                xr.v[k].y = bad ? 0.0f : (float)(int8_t)((c4 >> 8) & 0xff) * sc;
                xr.v[k].z = bad ? 0.0f : (float)(int8_t)((c4 >> 16) & 0xff) * sc;
                xr.v[k].w = bad ? 0.0f : (float)(int8_t)(c4 >> 24) * sc;
            }
        } else {
            xr.load(x, n4);
        }
    }
};

// A NormAct with its row slots (R = row_slots(D / 4)) and row source (EMB: the embedding, eq set) fixed, in the
// interface gemv_tile takes.
template <int R, bool EMB>
struct NormActR {
    static constexpr bool kGlobalScales = false;
    NormAct a;
    template <bool XL>
    __device__ __forceinline__ NormAct::Pre<R> begin() const { return a.template begin<R, EMB>(); }
    template <bool XL>
    __device__ __forceinline__ void fill(const NormAct::Pre<R>& p, int8_t* xs, float* xds) const {
        a.template fill<XL, R, EMB>(p, xs, xds);
    }
};

// ------------------------------------------------------------------------------------------------------ kernels

// x[t] = embedding row of tokens[t] (get_row, ops_ref.cpp:162-192: F32 as stored, F16 converted, Q8_0 / Q4_0 code *
// f16 scale, all exact in f32), then the first layer's rmsnorm and quantization; the normed row also to normed[t]
// when given (the f32 input of unquantized matrices). One workgroup per token.
template <int R>
__global__ __launch_bounds__(256) void embed_norm_quant_kernel(const int32_t* __restrict__ tokens,
                                                               const uint8_t* __restrict__ emb, int dtype, int D,
                                                               int V, float* __restrict__ x,
                                                               const float* __restrict__ w, float eps,
                                                               int8_t* __restrict__ oq, float* __restrict__ od,
                                                               float* __restrict__ normed, int* __restrict__ status) {
    __shared__ __align__(16) float xs[8192 + kChainPad];
    const int t = blockIdx.x, tid = threadIdx.x;
    RowF4<R> wr;
    wr.load(w, D / 4);
    int tok = tokens[t];
    const bool bad = tok < 0 || tok >= V;
    if (bad) {
        if (tid == 0) atomicOr(status, kStatusToken);
        tok = 0;
    }
    const size_t nq = dtype == kQ4 ? (size_t)V * D / 2 : (size_t)V * D;  // quant bytes (both planes) before the scales
    const uint16_t* sr = reinterpret_cast<const uint16_t*>(emb + nq) + (size_t)tok * (D / QK);
    for (int i4 = tid; i4 < D / 4; i4 += 256) {  // elements 4 i4 .. 4 i4 + 3 (one block, one half of a Q4_0 block)
        float4 v;
        if (dtype == kF32) {
            v = reinterpret_cast<const float4*>(emb + (size_t)tok * D * 4)[i4];
        } else if (dtype == kF16) {
            const uint2 h = reinterpret_cast<const uint2*>(emb + (size_t)tok * D * 2)[i4];
            v = make_float4(h2f((uint16_t)(h.x & 0xffffu)), h2f((uint16_t)(h.x >> 16)), h2f((uint16_t)(h.y & 0xffffu)),
                            h2f((uint16_t)(h.y >> 16)));
        } else {
            const float sc = h2f(sr[i4 / (QK / 4)]);
            uint32_t c4;
            if (dtype == kQ8) {
                c4 = *reinterpret_cast<const uint32_t*>(emb + (size_t)tok * D + 4 * i4);
            } else if (dtype == kQ8P) {  // q = 16 (h + 8) + l - 128: the byte (h + 8) << 4 | l, top bit flipped
                const int e = 4 * i4, j = e % QK;
                const size_t off = (size_t)tok * D / 2 + (e / QK) * 16 + j % 16;
                const uint32_t hb = *reinterpret_cast<const uint32_t*>(emb + off);
                const uint32_t lb = *reinterpret_cast<const uint32_t*>(emb + (size_t)V * D / 2 + off);
                const uint32_t hn = j < 16 ? hb & 0x0F0F0F0Fu : (hb >> 4) & 0x0F0F0F0Fu;
                const uint32_t ln = j < 16 ? lb & 0x0F0F0F0Fu : (lb >> 4) & 0x0F0F0F0Fu;
                c4 = ((hn << 4) | ln) ^ 0x80808080u;
            } else {  // element j of a block: low nibble of byte j (j < 16), high nibble of byte j - 16
                const int e = 4 * i4, j = e % QK;
                const uint32_t b4 = *reinterpret_cast<const uint32_t*>(emb + (size_t)tok * D / 2 + (e / QK) * 16 + j % 16);
                c4 = nibbles_to_i8(j < 16 ? b4 & 0x0F0F0F0Fu : (b4 >> 4) & 0x0F0F0F0Fu);
            }
            v = make_float4((float)(int8_t)(c4 & 0xff) * sc, (float)(int8_t)((c4 >> 8) & 0xff) * sc,
                            (float)(int8_t)((c4 >> 16) & 0xff) * sc, (float)(int8_t)(c4 >> 24) * sc);
        }
        if (bad) v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        reinterpret_cast<float4*>(x + (size_t)t * D)[i4] = v;
        reinterpret_cast<float4*>(xs)[i4] = v;
    }
    __syncthreads();
    norm_quant_lds(xs, D, wr, eps, oq + (size_t)t * D, od + (size_t)t * (D / QK), normed ? normed + (size_t)t * D : nullptr);
}

// One workgroup per token: residual add x += o, then rmsnorm with weight w and int8 quantization of the normed row;
// the normed row is also written to normed[t] when given. D <= 8192.
template <int R>
__global__ __launch_bounds__(256) void add_rmsnorm_quant_kernel(float* __restrict__ x, const float* __restrict__ o,
                                                                const float* __restrict__ w, int D, float eps,
                                                                int8_t* __restrict__ xq, float* __restrict__ xd,
                                                                float* __restrict__ normed) {
    __shared__ __align__(16) float xs[8192 + kChainPad];
    const int t = blockIdx.x, tid = threadIdx.x, n4 = D / 4;
    RowF4<R> wr, xr, orow;
    wr.load(w, n4);
    xr.load(x + (size_t)t * D, n4);
    orow.load(o + (size_t)t * D, n4);
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i4 = tid + 256 * k;
        if (i4 < n4) {
            float4 v = xr.v[k];
            v.x = v.x + orow.v[k].x;
            v.y = v.y + orow.v[k].y;
            v.z = v.z + orow.v[k].z;
            v.w = v.w + orow.v[k].w;
            xr.v[k] = v;
            reinterpret_cast<float4*>(x + (size_t)t * D)[i4] = v;
            reinterpret_cast<float4*>(xs)[i4] = v;
        }
    }
    __syncthreads();
    const float ss = D >= 128 ? seg_sum_squares_lds(xs, D, xr) : lds_sum_squares(xs, D);  // uniform
    normalize_quant_lds(xs, D, rms_scale(ss, D, eps), wr, xq + (size_t)t * D, xd + (size_t)t * (D / QK),
                        normed ? normed + (size_t)t * D : nullptr);
}

// The f16 cache rows of n tokens at positions *pos_dev .. + n - 1 (a prefill stack) from their projections k / v
// ([n][n_kv * HD]): bias, RoPE as a*c - b*s and b*c + a*s with the reference build's contraction
// (fma(a, c, -(b*s)), fma(b, c, a*s)), rounded to f16, exactly what attention_kernel rebuilds and stores
// (model.cpp:183-206, ops_ref.cpp:201-214), in the K chunk and V block layouts. One workgroup per token; positions
// past the context store nothing (attention_kernel raises the status).
template <int HD>
__global__ __launch_bounds__(256) void kv_store_kernel(const float* __restrict__ k, const float* __restrict__ v,
                                                       const float* __restrict__ bk, const float* __restrict__ bv,
                                                       const float* __restrict__ cs, const int* __restrict__ pos_dev,
                                                       int ctx, int n_kv, uint16_t* __restrict__ kc,
                                                       uint16_t* __restrict__ vc) {
    constexpr int HALF = HD / 2, CPR = HD / 8;
    const int t = blockIdx.x, tid = threadIdx.x, pos = *pos_dev + t;
    if (pos >= ctx || pos < 0) return;
    const int kvd = n_kv * HD;
    const float* krow = k + (size_t)t * kvd;
    const float* crow = cs + (size_t)pos * HD;
    for (int e = tid; e < n_kv * HALF; e += 256) {
        const int kvh = e / HALF, i = e % HALF;
        float a = krow[kvh * HD + i], b = krow[kvh * HD + i + HALF];
        if (bk) {
            a = a + bk[kvh * HD + i];
            b = b + bk[kvh * HD + i + HALF];
        }
        const float c = crow[2 * i], sn = crow[2 * i + 1];
        const float lo = __builtin_fmaf(a, c, -(b * sn)), hi = __builtin_fmaf(b, c, a * sn);
        const size_t base = (size_t)kvh * CPR * ctx;
        kc[((base + (size_t)(i >> 3) * ctx + pos) << 3) + (i & 7)] = f2h(lo);
        kc[((base + (size_t)((i + HALF) >> 3) * ctx + pos) << 3) + ((i + HALF) & 7)] = f2h(hi);
    }
    for (int e = tid; e < kvd; e += 256) {
        const float x = v[(size_t)t * kvd + e];
        vc[((size_t)(pos / 8) * kvd + e) * 8 + (pos & 7)] = f2h(bv ? x + bv[e] : x);
    }
}

// Attention over an f32 KV cache (the reference's --kv-f32, model.cpp:96-104, 197-204: the cache keeps k / v as
// computed, no f16 rounding), laid out as the reference keeps it, [ctx][n_kv * head_dim] per layer. One 256-thread
// workgroup per (query head, token of the chunk), prefill and decode alike: the chunk's K / V rows 0..t are rebuilt
// from the projections (bias, RoPE) in LDS, so no workgroup reads a cache row another one writes; scores
// s = fma(q_i, k_i, s) in dimension order, * 1 / sqrt(head_dim); max; glibc expf; the sum in position order (four
// segments with candidate starts, as attention_kernel); normalise; out_i = fma(a_j, v_ji, out_i) in position order
// over V rows staged in LDS; the output quantized per 32-block (model.cpp:115-137, ops_ref.cpp:201-226).
template <int HD>
__global__ __launch_bounds__(256) void attention_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ bq, const float* __restrict__ bk, const float* __restrict__ bv,
    const float* __restrict__ cs, const int* __restrict__ pos_dev, int ctx, int n_heads, int n_kv,
    float* __restrict__ kc, float* __restrict__ vc, int8_t* __restrict__ oq, float* __restrict__ od,
    int* __restrict__ status, float* __restrict__ of) {
    constexpr int HALF = HD / 2, C4 = HD / 4;
    constexpr int kVR = 16384 / HD;  // V rows per LDS stage (64 KB)
    __shared__ __align__(16) float att[kMaxCtx + kChainPad];
    __shared__ __align__(16) float vst[kVR * HD];
    __shared__ __align__(16) float kloc[kChunk * HD];
    __shared__ __align__(16) float vloc[kChunk * HD];
    __shared__ __align__(16) float qs[HD];
    __shared__ float red[4];
    __shared__ float sum_sh;
    __shared__ uint64_t exptab[32];
    __shared__ SegShared ssh;
    ExpTab et;
    et.load();
    const int h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int pos0 = *pos_dev, pos = pos0 + t, nrows = pos + 1;
    if (pos >= ctx || pos0 < 0) {  // uniform: a step past the context touches no cache row
        if (tid == 0 && h == 0) atomicOr(status, kStatusCtx);
        return;
    }
    const int qd = n_heads * HD, kvd = n_kv * HD, group = n_heads / n_kv, kvh = h / group;
    // add_bias, then rope: a * c - b * s and b * c + a * s with the reference build's contraction
    for (int e = tid; e < (t + 1) * HALF; e += 256) {
        const int r = e / HALF, i = e % HALF;
        const float* row = k + (size_t)r * kvd + kvh * HD;
        float a = row[i], b = row[i + HALF];
        if (bk) {
            a = a + bk[kvh * HD + i];
            b = b + bk[kvh * HD + i + HALF];
        }
        const float* crow = cs + (size_t)(pos0 + r) * HD;
        kloc[r * HD + i] = __builtin_fmaf(a, crow[2 * i], -(b * crow[2 * i + 1]));
        kloc[r * HD + i + HALF] = __builtin_fmaf(b, crow[2 * i], a * crow[2 * i + 1]);
    }
    for (int e = tid; e < (t + 1) * HD; e += 256) {
        const int r = e / HD, i = e % HD;
        const float x = v[(size_t)r * kvd + kvh * HD + i];
        vloc[e] = bv ? x + bv[kvh * HD + i] : x;
    }
    if (tid < HALF) {
        const float* row = q + (size_t)t * qd + h * HD;
        float a = row[tid], b = row[tid + HALF];
        if (bq) {
            a = a + bq[h * HD + tid];
            b = b + bq[h * HD + tid + HALF];
        }
        const float* crow = cs + (size_t)pos * HD;
        qs[tid] = __builtin_fmaf(a, crow[2 * tid], -(b * crow[2 * tid + 1]));
        qs[tid + HALF] = __builtin_fmaf(b, crow[2 * tid], a * crow[2 * tid + 1]);
    }
    et.store(exptab);
    __syncthreads();
    if (h % group == 0)
        for (int i = tid; i < HD; i += 256) {
            kc[(size_t)pos * kvd + kvh * HD + i] = kloc[t * HD + i];
            vc[(size_t)pos * kvd + kvh * HD + i] = vloc[t * HD + i];
        }
    // scores (model.cpp:122-125): cached rows below pos0 from the cache, the chunk's rows from LDS
    const float scale = 1.0f / __builtin_sqrtf((float)HD);
    const float4* q4 = reinterpret_cast<const float4*>(qs);
    float mx = -__builtin_inff();
    for (int j = tid; j < nrows; j += 256) {
        const float* kr = j < pos0 ? kc + (size_t)j * kvd + kvh * HD : kloc + (j - pos0) * HD;
        float sc = 0.0f;
#pragma unroll 4
        for (int c = 0; c < C4; ++c) {
            const float4 kk = reinterpret_cast<const float4*>(kr)[c], qq = q4[c];
            sc = __builtin_fmaf(qq.x, kk.x, sc);
            sc = __builtin_fmaf(qq.y, kk.y, sc);
            sc = __builtin_fmaf(qq.z, kk.z, sc);
            sc = __builtin_fmaf(qq.w, kk.w, sc);
        }
        const float a = sc * scale;
        att[j] = a;
        mx = a > mx ? a : mx;
    }
    mx = wave_max_sel(mx);  // the maximum does not depend on the order of comparison
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = red[0];
    for (int w = 1; w < 4; ++w) mx = red[w] > mx ? red[w] : mx;
    // exp, with each lane's exact partial sums below the segment starts; the sum in position order (ops_ref.cpp:216-226)
    const bool seg = nrows >= 128;  // uniform; shorter rows keep the single chain
    const int Ls = (nrows / 4) & ~15;
    const Segs4 sg{(nrows - 3 * Ls) & ~15, Ls, nrows};
    double p1 = 0.0, p2 = 0.0, p3 = 0.0;
    for (int j = tid; j < nrows; j += 256) {
        const float e = dev_expf(att[j] - mx, exptab);
        att[j] = e;
        p1 += j < sg.start(1) ? (double)e : 0.0;
        p2 += j < sg.start(2) ? (double)e : 0.0;
        p3 += j < sg.start(3) ? (double)e : 0.0;
    }
    if (seg) seg_partials(ssh, p1, p2, p3);
    __syncthreads();
    auto add = [](float acc, float a) { return acc + a; };
    float sum;
    if (seg) {
        sum = seg_chain_run(ssh, [&](int kk, float s0) { return lds_chain(att + sg.start(kk), sg.len(kk), add, s0); });
    } else {
        if (tid == 0) sum_sh = lds_chain(att, nrows, add);
        __syncthreads();
        sum = sum_sh;
    }
    const float inv = 1.0f / sum;
    for (int j = tid; j < nrows; j += 256) att[j] = att[j] * inv;
    // out_i = sum_j a_j * v_ji (model.cpp:131-135): thread i per dimension, V rows staged in LDS
    float acc = 0.0f;
    for (int s0 = 0; s0 < nrows; s0 += kVR) {
        const int sn = min(nrows, s0 + kVR);
        __syncthreads();  // the weights are final, the previous stage is consumed
        for (int e = tid; e < (sn - s0) * C4; e += 256) {
            const int r = s0 + e / C4, c = e % C4;
            const float* src = r < pos0 ? vc + (size_t)r * kvd + kvh * HD : vloc + (r - pos0) * HD;
            reinterpret_cast<float4*>(vst + (r - s0) * HD)[c] = reinterpret_cast<const float4*>(src)[c];
        }
        __syncthreads();
        if (tid < HD)
            for (int j = s0; j < sn; ++j) acc = __builtin_fmaf(att[j], vst[(j - s0) * HD + tid], acc);
    }
    if (tid < HD) {  // quantize_q8 of the attention output
        const int col = h * HD + (tid & ~31);
        if (of) of[(size_t)t * qd + h * HD + tid] = acc;  // the f32 input of an unquantized o projection
        quant_block32(acc, oq + (size_t)t * qd + col, od + (size_t)t * (qd / QK) + col / QK);
    }
}

// h = g / (1 + expf(-g)) * u (ops_ref.cpp:243-248) over a 256-value block, then the block's Walsh-Hadamard transform
// (FLAG_HADAMARD_DOWN, model.cpp:219, 424: fwht_blocks, ops_ref.cpp:228-241: butterflies v[j] = a + c, v[j + h] = a - c
// for h = 1, 2, .., 128, then * 1 / sqrt(256)) and the quantization of its 8 32-blocks for the down projection. Each
// butterfly adds or subtracts the same two values as the reference's loop, so the result does not depend on the
// order the butterflies of a stage run in. Grid (ffn_dim / 256, tokens).
__global__ __launch_bounds__(256) void swiglu_fwht_quant_kernel(const float* __restrict__ g, const float* __restrict__ u,
                                                                int F, int8_t* __restrict__ oq, float* __restrict__ od,
                                                                float* __restrict__ of) {
    __shared__ float vb[256];
    const int tid = threadIdx.x;
    const size_t b0 = (size_t)blockIdx.y * F + (size_t)blockIdx.x * 256;
    const float gv = g[b0 + tid];
    vb[tid] = gv / (1.0f + dev_expf(-gv)) * u[b0 + tid];
    __syncthreads();
    for (int hh = 1; hh < 256; hh *= 2) {
        const int j = (tid / hh) * 2 * hh + tid % hh;  // butterfly tid (< 128): v[j], v[j + hh]
        float a = 0.0f, c = 0.0f;
        if (tid < 128) {
            a = vb[j];
            c = vb[j + hh];
        }
        __syncthreads();
        if (tid < 128) {
            vb[j] = a + c;
            vb[j + hh] = a - c;
        }
        __syncthreads();
    }
    const float norm = 1.0f / __builtin_sqrtf(256.0f);
    const size_t blk = b0 + (tid & ~31);
    const float hv = vb[tid] * norm;
    if (of) of[b0 + tid] = hv;
    quant_block32(hv, oq + blk, od + blk / QK);
}

// ------------------------------------------------------------------------------ decode attention, 16 waves per head
// Timeline stamps for phase measurements: compiled in only with -DQH_TIMELINE (thread 0 of workgroup 0 records the
// shader clock at each stamp; qh_timeline_read copies them out).
#if defined(QH_TIMELINE)
__device__ uint64_t qh_tl[64];
#define QH_STAMP(i)                                                                    \
    do {                                                                               \
        if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) qh_tl[i] = __builtin_readcyclecounter(); \
    } while (0)
#else
#define QH_STAMP(i) \
    do {            \
    } while (0)
#endif

// Brings every 64-byte line of g[0, n) (g uniform across the wave, 4-byte aligned) into the scalar cache: one scalar
// load per line, all in flight at once, then one wait. The loads land in one scratch register, since only their
// cache fill matters.
__device__ __forceinline__ void warm_lines(const float* g, int n) {
#if defined(__HIP_DEVICE_COMPILE__)
    uint32_t sink;
    for (int i = 0; i < n; i += 16)
        asm volatile("s_load_dword %0, %1, 0x0" : "=s"(sink) : "s"(g + i) : "memory");
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#endif
}

// Workgroup state of a four-segment chain run by waves 0-3 of a 16-wave workgroup (seg16_*).
struct SegShared16 {
    double part[16][4];  // [wave][k]: the wave's share of the exact sum of the chain's terms below segment k's start
    float res[256];      // every lane's segment result (waves 0-3)
    uint32_t gbits[4];   // segment k's guess
};

// Sums three per-lane partials over the wave into part[wave][1..3]; a barrier must follow before seg16_run.
__device__ __forceinline__ void seg16_partials(SegShared16& sh, double p1, double p2, double p3) {
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

// seg_chain_run for a 16-wave workgroup: waves 0-3 run the four segments (wave 0 from 0, wave k from the 64 candidates
// around its guess, the f32 rounding of the exact sum below the segment), the others wait at the barrier; then every
// thread follows the chain through the candidates and returns its end value. chain(k, start) runs segment k from
// start in the calling wave (k and start uniform across the wave). All 1024 threads call it after the barrier that
// published part.
template <typename Chain>
__device__ __forceinline__ float seg16_run(SegShared16& sh, Chain chain) {
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (wave < 4) {
        float start = 0.0f;
        if (wave > 0) {
            double g = 0.0;
#pragma unroll
            for (int w = 0; w < 16; ++w) g += sh.part[w][wave];
            const uint32_t gb = __float_as_uint((float)g);
            start = __uint_as_float(gb + (uint32_t)lane - 32u);
            if (lane == 0) sh.gbits[wave] = gb;
        }
        sh.res[tid] = chain(wave, start);
    }
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

// Decode attention of one token (position *pos_dev) for query head h = blockIdx.x over positions [0, pos], head_dim 64:
// the same arithmetic, order and cache layouts as attention_kernel with one token, spread over 16 waves. Every thread
// scores one cached row held in registers (rows beyond 1024 in a loop), the 16 waves share the V DMA of the first LDS
// stage (a few transfers each, issued after their scores, so the scores keep exact load waits), and the exp and
// normalisation run one position per thread. The serial softmax sum runs as four segments on waves 0-3 (seg16_run), the
// weighted V chain on wave 0 with the weights as scalar operands while the other waves bring the weight row into the
// scalar cache. Workgroups of the first query head of each KV group store the token's K / V row.
// Grid (group, n_kv) with group = n_heads / n_kv: query head h = blockIdx.y * group + blockIdx.x of KV head blockIdx.y,
// so no division is needed. The arguments the first loads need come first: the first 16 dwords arrive in registers at
// dispatch, the rest (and the grid's size) take a load.
template <int HD>
__global__ __launch_bounds__(1024) void attention_decode_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    uint16_t* __restrict__ kc, const int* __restrict__ pos_dev, int ctx, int group, const float* __restrict__ bq,
    const float* __restrict__ bk, int n_kv, const float* __restrict__ bv, const float* __restrict__ cs,
    uint16_t* __restrict__ vc, int8_t* __restrict__ oq, float* __restrict__ od, float* __restrict__ escr,
    int escr_stride, int* __restrict__ status, float* __restrict__ of) {
    static_assert(HD == 64, "one chain wave and one K row of 8 chunks per thread");
    constexpr int NT = 1024, NW = NT / 64;
    constexpr int HALF = HD / 2, CPR = HD / 8;
    constexpr int kVRows = kVStageBytes / (HD * 2);  // V rows one LDS stage holds (a multiple of 8)
    constexpr int kVBlk = kVRows / 8;                // 8-row blocks per stage
    __shared__ __align__(16) float att[kMaxCtx + kChainPad];
    __shared__ __align__(16) uint4 vst[(kVBlk + 4) * HD];  // [block][dim] -> 8 rows; 4 blocks of read padding
    __shared__ __align__(16) uint16_t kloc[HD];
    __shared__ __align__(16) uint16_t vloc[HD];
    __shared__ __align__(16) float qs[HD];
    __shared__ float red[NW];
    __shared__ float sum_sh;
    __shared__ uint64_t exptab[32];
    __shared__ SegShared16 ssh;
    QH_STAMP(0);
    QH_WSTAMP(1, 0);
    const int n_heads = group * n_kv;
    const int kvh = (int)blockIdx.y, h = kvh * group + (int)blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kvd = n_kv * HD;
    // The token's raw q (wave 0), k (wave 1) and v (wave 2) values and biases do not depend on the position: their
    // loads go out before it arrives.
    float pa = 0.0f, pb = 0.0f, ba = 0.0f, bb = 0.0f, pc = 0.0f, ps = 0.0f;
    if (wave < 2 && lane < HALF) {
        const float* src = wave == 0 ? q + h * HD : k + kvh * HD;
        const float* bias = wave == 0 ? (bq ? bq + h * HD : nullptr) : (bk ? bk + kvh * HD : nullptr);
        pa = src[lane];
        pb = src[lane + HALF];
        ba = bias ? bias[lane] : 0.0f;
        bb = bias ? bias[lane + HALF] : 0.0f;
    } else if (wave == 2) {
        pa = v[kvh * HD + lane];
        ba = bv ? bv[kvh * HD + lane] : 0.0f;
    }
    ExpTab et;
    et.load();
    const uint4* vc4 = reinterpret_cast<const uint4*>(vc);
    auto vchunk = [&](int blk, int d) { return (size_t)blk * kvd + kvh * HD + d; };  // uint4 index of (block, dim)
    auto kchunk = [&](int c, int p) { return ((size_t)kvh * CPR + c) * ctx + p; };    // 16-byte K chunk c of row p
    // The position (a scalar load, back before the vector loads above), then this thread's K row: cached rows only
    // (tid < pos; row pos is the token's own, written by this launch). The K rows are the largest of the kernel's first
    // transfers and one CU issues them at ~40 bytes per cycle, so rows past the position are not read.
    const int pos = *pos_dev, nrows = pos + 1;
    if (pos >= ctx || pos < 0) {  // uniform: a step past the context touches no cache row
        if (tid == 0 && h == 0) atomicOr(status, kStatusCtx);
        return;
    }
    v4u kk[CPR];
    if (tid < pos) {
        const uint16_t* kg = kc + (kchunk(0, tid) << 3);
#pragma unroll
        for (int i = 0; i < CPR; ++i) kk[i] = ld4(kg + (size_t)i * ctx * 8);
    }
    QH_STAMP(8);
    // Then the RoPE angles of the position (ops_ref.cpp:201-214, with the reference build's contraction).
    if (wave < 2 && lane < HALF) {
        const float* crow = cs + (size_t)pos * HD;
        pc = crow[2 * lane];
        ps = crow[2 * lane + 1];
    }
    const bool has_bias = wave == 0 ? bq != nullptr : wave == 1 ? bk != nullptr : bv != nullptr;
    if (wave < 2 && lane < HALF) {
        float a = pa, b = pb;
        if (has_bias) {
            a = a + ba;
            b = b + bb;
        }
        const float lo = __builtin_fmaf(a, pc, -(b * ps)), hi = __builtin_fmaf(b, pc, a * ps);
        QH_STAMP(9);
        if (wave == 0) {
            qs[lane] = lo;
            qs[lane + HALF] = hi;
        } else {
            kloc[lane] = f2h(lo);
            kloc[lane + HALF] = f2h(hi);
        }
    } else if (wave == 2) {
        vloc[lane] = f2h(has_bias ? pa + ba : pa);
    }
    et.store(exptab);
    __syncthreads();
    QH_STAMP(1);
    if (h % group == 0 && tid < HD) {
        kc[(kchunk(tid >> 3, pos) << 3) + (tid & 7)] = kloc[tid];
        vc[vchunk(pos / 8, tid) * 8 + (pos & 7)] = vloc[tid];
    }

    // scores s_j = (sum_i q_i * k_ji as one FMA per element in dimension order) * (1 / sqrt(HD)) (model.cpp:122-125);
    // q comes from LDS by broadcast reads (every lane the same address), which keeps the kernel within the 128
    // registers a 16-wave workgroup allows
    const float scale = 1.0f / __builtin_sqrtf((float)HD);
    const float4* q4 = reinterpret_cast<const float4*>(lane_ptr(qs));
    auto dot_row = [&](const v4u(&r)[CPR], const float4* q4) {
        float sc = 0.0f;
#pragma unroll
        for (int i = 0; i < CPR; ++i) {
            const float4 qa = q4[2 * i], qb = q4[2 * i + 1];
            const float qq[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sc = __builtin_fmaf(qq[2 * e], h2f((uint16_t)(r[i][e] & 0xffffu)), sc);
                sc = __builtin_fmaf(qq[2 * e + 1], h2f((uint16_t)(r[i][e] >> 16)), sc);
            }
        }
        return sc;
    };
    float mx = -__builtin_inff();
    if (tid < nrows) {  // row tid: the cached row in registers, or the token's own row (tid == pos)
        if (tid == pos) {
#pragma unroll
            for (int i = 0; i < CPR; ++i) kk[i] = ld4(kloc + i * 8);
        }
        const float a = dot_row(kk, q4) * scale;
        att[tid] = a;
        mx = a;
    }
    if (pos >= NT) {  // contexts beyond NT positions: the other cached rows one at a time, then the token's own row
        for (int j = tid + NT; j < pos; j += NT) {
            const uint16_t* kg = kc + (kchunk(0, j) << 3);
#pragma unroll
            for (int i = 0; i < CPR; ++i) kk[i] = ld4(kg + (size_t)i * ctx * 8);
            const float4* qo = q4;
            asm volatile("" : "+v"(qo));  // keeps the q reads inside the loop (hoisted, they would not fit)
            const float a = dot_row(kk, qo) * scale;
            att[j] = a;
            mx = a > mx ? a : mx;
        }
        if (tid == pos % NT) {
#pragma unroll
            for (int i = 0; i < CPR; ++i) kk[i] = ld4(kloc + i * 8);
            const float a = dot_row(kk, q4) * scale;
            att[pos] = a;
            mx = a > mx ? a : mx;
        }
    }
    QH_STAMP(2);
    mx = wave_max_sel(mx);  // the maximum does not depend on the order of comparison
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = red[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = red[w] > mx ? red[w] : mx;
    QH_STAMP(3);
    // exp (the exp row also goes to global memory for the segmented sum's scalar loads), with each lane's exact partial
    // sums below the segment starts
    float* erow = escr + (size_t)h * escr_stride;
    float* arow = escr + (size_t)(n_heads + h) * escr_stride;
    const bool seg = nrows >= 128;  // uniform; shorter rows keep the single chain
    const int Ls = (nrows / 4) & ~15;
    const Segs4 sg{(nrows - 3 * Ls) & ~15, Ls, nrows};
    double p1 = 0.0, p2 = 0.0, p3 = 0.0;
    for (int j = tid; j < nrows; j += NT) {
        const float e = dev_expf(att[j] - mx, exptab);
        att[j] = e;
        erow[j] = e;
        p1 += j < sg.start(1) ? (double)e : 0.0;
        p2 += j < sg.start(2) ? (double)e : 0.0;
        p3 += j < sg.start(3) ? (double)e : 0.0;
    }
    QH_STAMP(10);
    if (seg) seg16_partials(ssh, p1, p2, p3);
    QH_STAMP(11);
    __builtin_amdgcn_s_waitcnt(0);  // the exp row's stores (read through scalar loads after the barrier)
    QH_STAMP(12);
    __syncthreads();
    QH_STAMP(4);
    // The first stage's V blocks straight into LDS by DMA while waves 0-3 run the softmax sum: waves 4-15 take 1 KB
    // chunks wave - 4, wave + 8, ... (clamped onto the last chunk, whose repeats write the same data). A wave's DMA
    // issue waits while the memory pipeline drains, so the chain waves issue none. Cache blocks stop below pos: the
    // block holding pos, if any, carries a stale row pos that the stage build replaces. The normalisation's
    // s_waitcnt(0) completes the transfers before the barrier that precedes the V chain.
    const int ncb = min((pos + 7) / 8, kVBlk);
    if (wave >= 4) {
        constexpr int kDmaWaves = NW - 4, kPerWave = (kVBlk + kDmaWaves - 1) / kDmaWaves;
        const int last = max(ncb - 1, 0);
#pragma unroll
        for (int e = 0; e < kPerWave; ++e) {
            const int c = min(wave - 4 + kDmaWaves * e, last);
            lds_dma16_async(vc4 + vchunk(c, lane), vst + c * 64);
        }
    }
    // softmax sum in position order (ops_ref.cpp:220-224)
    auto add = [](float acc, float a) { return acc + a; };
    float sum;
    if (seg) {
        sum = seg16_run(ssh, [&](int kk_, float s0) {
            warm_lines(erow + sg.start(kk_), sg.len(kk_));  // the exp row was just written: not in the scalar cache
            return chain_scalar(erow + sg.start(kk_), sg.len(kk_), s0, add);
        });
    } else {
        if (tid == 0) sum_sh = lds_chain(att, nrows, add);
        __syncthreads();
        sum = sum_sh;
    }
    QH_STAMP(5);
    const float inv = 1.0f / sum;
    for (int j = tid; j < nrows; j += NT) {
        const float a = att[j] * inv;
        att[j] = a;
        arow[j] = a;
    }
    QH_STAMP(13);
    // the weight row's stores and the V DMA complete before the barrier; then the token's own row, if it falls inside
    // the first stage, is written over the DMA's block
    __builtin_amdgcn_s_waitcnt(0);
    QH_STAMP(14);
    __syncthreads();
    uint16_t* vst16 = reinterpret_cast<uint16_t*>(vst);
    if (pos < kVRows && tid < HD) vst16[((pos >> 3) * HD + tid) * 8 + (pos & 7)] = vloc[tid];
    __syncthreads();
    QH_STAMP(6);

    // out_i = sum_j a_j * v_ji, one FMA per position in order (model.cpp:131-135): lane i of wave 0 per dimension,
    // the weights as scalar operands (as in attention_kernel); the other waves warm the weight row's lines and load the
    // next stage's cache blocks into registers while the chain runs, so that only LDS stores stand between two stages
    // (position 3,500: 37.3 -> 31.7 us a layer).
    constexpr int kLoaders = NT - HD, kPre = (kVBlk * HD + kLoaders - 1) / kLoaders;
    v4u nxt[kPre];
    float acc = 0.0f;
    for (int s0 = 0;;) {
        const int se = min(nrows, s0 + kVRows);
        if (tid >= HD && se < nrows) {  // uniform per wave; pos >= 1 here (a second stage)
            const int nb8 = (min(nrows, se + kVRows) - se + 7) / 8, lastc = (pos - 1) / 8;
#pragma unroll
            for (int u = 0; u < kPre; ++u) {  // units past the stage repeat its last (never stored)
                const int c = min(tid - HD + kLoaders * u, nb8 * HD - 1);
                nxt[u] = ld4(vc4 + vchunk(min(se / 8 + c / HD, lastc), c % HD));
            }
        }
        if (tid < HD) {
            const_v16f_ptr wp = (const_v16f_ptr)(arow + s0);  // s0 is a multiple of 32: 64-byte aligned
            auto ldv = [&](uint4(&vv)[4], int jr) {  // rows s0 + jr .. + 31 (jr % 32 == 0)
                const uint4* vp = vst + (jr >> 3) * HD + tid;
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) vv[q4] = vp[q4 * HD];
            };
            auto use = [&](const uint4(&vv)[4], const v16f& w0, const v16f& w1, int cnt) {
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    const uint32_t w[4] = {vv[q4].x, vv[q4].y, vv[q4].z, vv[q4].w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int kx = 8 * q4 + e;
                        if (kx < cnt)
                            acc = __builtin_fmaf(kx < 16 ? w0[kx & 15] : w1[kx & 15],
                                                 h2f((uint16_t)(e & 1 ? w[e >> 1] >> 16 : w[e >> 1] & 0xffffu)), acc);
                    }
                }
            };
            const int n = se - s0;
            uint4 vA[4], vB[4];
            v16f wA0 = wp[0], wA1 = wp[1], wB0, wB1;
            ldv(vA, 0);
            int jr = 0;
#pragma unroll 1
            for (; jr + 64 <= n; jr += 64) {
                wait_lgkm0();
                __builtin_amdgcn_sched_barrier(0);
                wB0 = wp[(jr + 32) / 16];
                wB1 = wp[(jr + 32) / 16 + 1];
                ldv(vB, jr + 32);
                __builtin_amdgcn_sched_barrier(0);
                use(vA, wA0, wA1, 32);
                wait_lgkm0();
                __builtin_amdgcn_sched_barrier(0);
                wA0 = wp[(jr + 64) / 16];
                wA1 = wp[(jr + 64) / 16 + 1];
                ldv(vA, jr + 64);
                __builtin_amdgcn_sched_barrier(0);
                use(vB, wB0, wB1, 32);
            }
            wait_lgkm0();
            __builtin_amdgcn_sched_barrier(0);
            if (jr + 32 <= n) {
                wB0 = wp[(jr + 32) / 16];
                wB1 = wp[(jr + 32) / 16 + 1];
                ldv(vB, jr + 32);
                __builtin_amdgcn_sched_barrier(0);
                use(vA, wA0, wA1, 32);
                wait_lgkm0();
                __builtin_amdgcn_sched_barrier(0);
                use(vB, wB0, wB1, n - jr - 32);
            } else {
                use(vA, wA0, wA1, n - jr);
            }
        } else if (s0 == 0) {  // the other waves: 16 lines of the weight row per scalar-load batch
            const int wi = __builtin_amdgcn_readfirstlane(wave - 1);
            for (int b = wi * 256; b < nrows; b += (NW - 1) * 256) {
                SegWarm warm;
                warm.issue(arow + b, nrows - b);
                warm.consume();
            }
        }
        s0 = se;
        if (s0 >= nrows) break;
        __syncthreads();  // the stage is consumed; load rows [s0, min(nrows, s0 + kVRows)) (s0 % 8 == 0)
        const int sn = min(nrows, s0 + kVRows);
        const int nb8 = (sn - s0 + 7) / 8;
        if (tid >= HD) {
#pragma unroll
            for (int u = 0; u < kPre; ++u) {  // whole cache blocks; the token's row is written after
                const int c = tid - HD + kLoaders * u;
                if (c < nb8 * HD) *reinterpret_cast<v4u*>(&vst[c]) = nxt[u];
            }
        }
        __syncthreads();
        if (pos >= s0 && pos < sn && tid < HD) vst16[(((pos - s0) >> 3) * HD + tid) * 8 + (pos & 7)] = vloc[tid];
        __syncthreads();
    }
    QH_STAMP(7);
    QH_WSTAMP(1, 3);
    if (tid < HD) {  // quantize_q8 of the attention output, two 32-blocks per 64 dimensions
        const int col = h * HD + (tid & ~31);
        if (of) of[h * HD + tid] = acc;  // the f32 input of an unquantized o projection
        quant_block32(acc, oq + col, od + col / QK);
    }
}

// h = g / (1 + expf(-g)) * u (ops_ref.cpp:243-248) over n_blocks 32-blocks, quantized per block.
__global__ __launch_bounds__(256) void swiglu_quant_kernel(const float* __restrict__ g, const float* __restrict__ u,
                                                           long n_blocks, int8_t* __restrict__ oq,
                                                           float* __restrict__ od, float* __restrict__ of) {
    const long blk = ((long)blockIdx.x * 256 + threadIdx.x) >> 5;
    if (blk >= n_blocks) return;  // whole half-waves leave together
    const long i = blk * QK + (threadIdx.x & 31);
    const float gv = g[i];
    const float hv = gv / (1.0f + dev_expf(-gv)) * u[i];
    if (of) of[i] = hv;  // the f32 input of an unquantized down projection
    quant_block32(hv, oq + blk * QK, od + blk);
}

// Prefill gate / up, SwiGLU and quantization of the down projection's input in one launch (model.cpp:212-218 for a
// chunk of n tokens; ops_ref.cpp:122-160, 243-248, 69-83). Workgroup (b, g): rows [32 b, 32 b + 32) of gate and of up
// for tokens [16 g, 16 g + 16). The chunk's 64 weight rows, 16 activation rows and their scales are staged in LDS
// by coalesced 16-byte loads, 16 blocks at a time (the next chunk's loads in flight); wave w multiplies row tile w
// (gate rows 0-15, 16-31, up rows 0-15, 16-31 of the block) by the token tile with one int8 MFMA per block and runs
// the chains of its own results in registers: lane l holds rows 4 (l / 16) + i, token l % 16, acc = fma(float(s) *
// dw, dx, acc) in block order, as the other matmul kernels. Then h = g / (1 + expf(-g)) * u and the quantization of
// each token's 32 values (one block of the down projection's input) by 32 lanes. SHORT: at most two chunks
// (cols <= 1024), straight-line.
constexpr int kSwKC = 16;  // blocks per chunk
template <int DT>
struct SwRegs {
    static constexpr int kBw = DT == kQ8 ? QK : QK / 2;           // weight bytes per block
    static constexpr int kAu = 64 * kSwKC * kBw / 16 / 256;        // 16-byte weight units per thread (8 / 4)
    static constexpr int kXu = 16 * kSwKC * QK / 16 / 256;         // 16-byte activation units per thread (2)
    static constexpr int kWu = 64 * kSwKC / 256;                   // row scales per thread (4)
    uint4 a[kAu];
    uint4 x[kXu];
    uint16_t dw[kWu];
    float dx;
};

template <int DT, bool SHORT>
__global__ __launch_bounds__(256) void matmul_swiglu_kernel(const uint8_t* __restrict__ wg,
                                                            const uint16_t* __restrict__ sgt,
                                                            const uint8_t* __restrict__ wu,
                                                            const uint16_t* __restrict__ sut,
                                                            const int8_t* __restrict__ xq, const float* __restrict__ xd,
                                                            int cols, int rows, int n, int n_tg,
                                                            int8_t* __restrict__ oq, float* __restrict__ od) {
    using R = SwRegs<DT>;
    constexpr int KC = kSwKC, kBw = R::kBw;
    constexpr int kArow = KC * kBw + 16;  // LDS row strides in bytes (= 4 dwords mod 64 banks: the 16 rows of an
    constexpr int kXrow = KC * QK + 16;   // operand read hit distinct banks)
    constexpr int kAupr = KC * kBw / 16, kXupr = KC * QK / 16;
    constexpr int kDxRow = KC + 4;        // token scale row stride (floats): 16-byte reads of 16 tokens, no conflict
    __shared__ __align__(16) uint8_t as[2][64 * kArow];
    __shared__ __align__(16) int8_t xs[2][16 * kXrow];
    __shared__ __align__(16) float dws[2][64 * KC];
    __shared__ __align__(16) float dxs[2][16 * kDxRow];
    __shared__ float hg[32][17], hu[32][17];
    __shared__ uint64_t exptab[32];
    ExpTab et;
    et.load();
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, lq = lane >> 4;
    // workgroups of one row block (its token groups) are numbered onto one XCD, as in the matmul kernels
    const int G = (int)gridDim.x, p = (int)blockIdx.x;
    const int xcd = p % 8, per = G / 8, rem = G % 8;
    const int logical = xcd * per + min(xcd, rem) + p / 8;
    const int rb = logical / n_tg, tg = logical % n_tg;
    const int r0 = rb * 32, tbase = tg * 16;
    const int nb = cols / QK;
    const size_t wrow = (size_t)nb * kBw;

    // staged row s (0..63): gate row r0 + s for s < 32, else up row r0 + s - 32; tokens past n are clamped
    const uint8_t* asrc[R::kAu];
    int aoff[R::kAu];
#pragma unroll
    for (int j = 0; j < R::kAu; ++j) {
        const int e = j * 256 + tid, r = e / kAupr;
        asrc[j] = r < 32 ? wg + (size_t)(r0 + r) * wrow : wu + (size_t)(r0 + r - 32) * wrow;
        aoff[j] = (e % kAupr) * 16;
    }
    const int8_t* xsrc[R::kXu];
    int xoff[R::kXu];
#pragma unroll
    for (int j = 0; j < R::kXu; ++j) {
        const int e = j * 256 + tid;
        xsrc[j] = xq + (size_t)min(tbase + e / kXupr, n - 1) * cols;
        xoff[j] = (e % kXupr) * 16;
    }
    const uint16_t* wsrc[R::kWu];
#pragma unroll
    for (int j = 0; j < R::kWu; ++j) {
        const int r = (j * 256 + tid) / KC;
        wsrc[j] = r < 32 ? sgt + (size_t)(r0 + r) * nb : sut + (size_t)(r0 + r - 32) * nb;
    }
    const float* dxsrc = xd + (size_t)min(tbase + tid / KC, n - 1) * nb;
    const int sk = tid % KC;  // the block of this thread's staged scales (256 is a multiple of KC)

    auto load = [&](R& S, int c0) {
#pragma unroll
        for (int j = 0; j < R::kAu; ++j)
            S.a[j] = load16(asrc[j] + min((size_t)c0 * kBw + aoff[j], wrow - 16));
#pragma unroll
        for (int j = 0; j < R::kXu; ++j) S.x[j] = load16(xsrc[j] + min(c0 * QK + xoff[j], cols - 16));
        const int b = min(c0 + sk, nb - 1);
#pragma unroll
        for (int j = 0; j < R::kWu; ++j) S.dw[j] = wsrc[j][b];
        S.dx = dxsrc[b];
    };
    auto stage = [&](const R& S, int buf) {
#pragma unroll
        for (int j = 0; j < R::kAu; ++j) {
            const int e = j * 256 + tid;
            *reinterpret_cast<uint4*>(&as[buf][(e / kAupr) * kArow + (e % kAupr) * 16]) = S.a[j];
        }
#pragma unroll
        for (int j = 0; j < R::kXu; ++j) {
            const int e = j * 256 + tid;
            *reinterpret_cast<uint4*>(&xs[buf][(e / kXupr) * kXrow + (e % kXupr) * 16]) = S.x[j];
        }
#pragma unroll
        for (int j = 0; j < R::kWu; ++j) {
            uint32_t h = S.dw[j];
            asm volatile("" : "+v"(h));  // keeps the conversion here (hoisted, it would wait for later loads)
            dws[buf][j * 256 + tid] = f16_to_f32((uint16_t)h);
        }
        dxs[buf][(tid / KC) * kDxRow + sk] = S.dx;
    };
    // wave w: staged rows 16 w + li (operand) / 16 w + 4 lq + i (results); chains acc[i] of (row 16 w + 4 lq + i,
    // token li)
    const int shift = DT == kQ8 ? 0 : (lq >> 1) * 4;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto compute = [&](int buf, int c0) {
        const int nblk = min(KC, nb - c0);
        const float4* dw4 = reinterpret_cast<const float4*>(dws[buf]) + (16 * wave + 4 * lq) * (KC / 4);
        const float4* dx4 = reinterpret_cast<const float4*>(dxs[buf] + li * kDxRow);
#pragma unroll
        for (int g4 = 0; g4 < KC / 4; ++g4) {
            long a[4], x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int b = 4 * g4 + i;
                a[i] = *reinterpret_cast<const long*>(
                    &as[buf][(16 * wave + li) * kArow + b * kBw + (DT == kQ8 ? lq * 8 : (lq & 1) * 8)]);
                x[i] = *reinterpret_cast<const long*>(&xs[buf][li * kXrow + b * QK + lq * 8]);
            }
            float4 dwv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) dwv[r] = dw4[r * (KC / 4) + g4];
            const float4 dxv = dx4[g4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                long ai = a[i];
                if (DT == kQ4) {
                    const uint64_t v = (uint64_t)ai;
                    const uint32_t lo = nibbles_to_i8(((uint32_t)v >> shift) & 0x0F0F0F0Fu);
                    const uint32_t hi = nibbles_to_i8(((uint32_t)(v >> 32) >> shift) & 0x0F0F0F0Fu);
                    ai = (long)(((uint64_t)hi << 32) | lo);
                }
                const v4i c = __builtin_amdgcn_mfma_i32_16x16x32_i8(ai, x[i], (v4i){0, 0, 0, 0}, 0, 0, 0);
                const float dx = i == 0 ? dxv.x : i == 1 ? dxv.y : i == 2 ? dxv.z : dxv.w;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float dw = i == 0 ? dwv[r].x : i == 1 ? dwv[r].y : i == 2 ? dwv[r].z : dwv[r].w;
                    const float nx = __builtin_fmaf((float)c[r] * dw, dx, acc[r]);
                    acc[r] = 4 * g4 + i < nblk ? nx : acc[r];
                }
            }
        }
    };

    const int n_chunks = (nb + KC - 1) / KC;
    if constexpr (SHORT) {
        R A, B;
        load(A, 0);
        load(B, KC);
        __builtin_amdgcn_sched_barrier(0);
        stage(A, 0);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        compute(0, 0);
        stage(B, 1);  // buffer 1 is not read by chunk 0
        __syncthreads();
        compute(1, KC);  // a chunk past nb adds nothing
    } else {
        // chunk c in buffer c % 2 and register set c % 2, refilled with chunk c + 2 once staged (clamped re-reads
        // past the last chunk)
        R S[2];
        load(S[0], 0);
        load(S[1], KC);
        __builtin_amdgcn_sched_barrier(0);
        stage(S[0], 0);
        load(S[0], 2 * KC);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        for (int c = 0;; c += 2) {
            compute(0, c * KC);
            if (c + 1 >= n_chunks) break;
            stage(S[1], 1);
            load(S[1], (c + 3) * KC);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            compute(1, (c + 1) * KC);
            if (c + 2 >= n_chunks) break;
            stage(S[0], 0);
            load(S[0], (c + 4) * KC);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
        }
    }
    (void)n_chunks;

    // h = g / (1 + expf(-g)) * u (ops_ref.cpp:243-248) and its quantization per token: 32 lanes per block
    {
        float(*dst)[17] = wave < 2 ? hg : hu;
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[16 * (wave & 1) + 4 * lq + r][li] = acc[r];
    }
    et.store(exptab);
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        const int tk = pass * 8 + tid / 32, rr = tid % 32, tok = tbase + tk;
        if (tok < n) {  // uniform per 32-lane group
            const float gv = hg[rr][tk], uv = hu[rr][tk];
            quant_block32(gv / (1.0f + dev_expf(-gv, exptab)) * uv, oq + (size_t)tok * rows + r0,
                          od + (size_t)tok * (rows / QK) + rb);
        }
    }
}

// q, k and v GEMVs of one token in one launch: three row segments of one dtype and width over one activation,
// the layer's normed input, which every workgroup builds itself (NormAct).
struct QkvSegs {
    const uint8_t *w0, *w1, *w2;
    const uint16_t *s0, *s1, *s2;
    float *o0, *o1, *o2;
    int rows0, rows1, rows2;
    int tiles0, tiles1;
};

template <int DT, int U, int R, bool EMB>
__global__ __launch_bounds__(256) void gemv_qkv_norm_kernel(QkvSegs a, NormAct act, int nb, int tile_rows,
                                                            uint32_t nb_magic) {
    extern __shared__ __align__(16) float smem[];
    QH_WSTAMP(0, 0);
    int blk = (int)blockIdx.x;
    const uint8_t* w = a.w0;
    const uint16_t* sc = a.s0;
    float* out = a.o0;
    int rows = a.rows0;
    if (blk >= a.tiles0) {
        blk -= a.tiles0;
        if (blk >= a.tiles1) {
            blk -= a.tiles1;
            w = a.w2, sc = a.s2, out = a.o2, rows = a.rows2;
        } else {
            w = a.w1, sc = a.s1, out = a.o1, rows = a.rows1;
        }
    }
    const int ra = blk * tile_rows;
    const int nrows = min(tile_rows, rows - ra);
    act.tmp = smem + gemv_tile_lds_bytes(nb * QK, tile_rows, true) / 4;
    constexpr int kBlockBytes = DT == kQ8 ? QK : QK / 2;
    const GemvSegs<1> segs{{w + (size_t)ra * nb * kBlockBytes}, {sc + (size_t)ra * nb}};
    const float val =
        gemv_tile<DT, U, true, 1>(segs, nullptr, nullptr, nb, nrows, tile_rows, nb_magic, smem,
                                  NormActR<R, EMB>{act}, 0);
    QH_WSTAMP(0, 3);
    if ((int)threadIdx.x < nrows) out[ra + threadIdx.x] = val;
}

// One token's projection added into the residual stream: x[r] += (W . xq)[r] (model.cpp:208-210, 224-226).
template <int DT, int U, bool XL>
__global__ __launch_bounds__(256) void gemv_residual_kernel(const uint8_t* __restrict__ wq,
                                                            const uint16_t* __restrict__ wscale,
                                                            const int8_t* __restrict__ xq,
                                                            const float* __restrict__ xd, int nb, int rows,
                                                            int tile_rows, uint32_t nb_magic, float* __restrict__ x) {
    extern __shared__ __align__(16) float smem[];
    const int tlk = nb > 64 ? 4 : 2;  // timeline id: the down projection (K = 4864) or o (K = 896)
    (void)tlk;
    QH_WSTAMP(tlk, 0);
    const int tid = (int)threadIdx.x;
    const int ra = (int)blockIdx.x * tile_rows;
    const int nrows = min(tile_rows, rows - ra);
    const float x0 = x[ra + min(tid, nrows - 1)];  // the residual row, in flight with the weights
    const float val = gemv_tile<DT, U, XL>(wq, wscale, xq, xd, nb, ra, nrows, tile_rows, nb_magic, smem, tlk);
    QH_WSTAMP(tlk, 3);
    if (tid < nrows) x[ra + tid] = x0 + val;
}

// One token's gate and up GEMVs over the same 32 rows of both matrices, from the normed MLP input each workgroup
// builds itself (NormAct), then h = g / (1 + expf(-g)) * u and the quantization of those 32 values (one block) for
// the down projection.
template <int DT, int U, int R>
__global__ __launch_bounds__(256) void gemv_swiglu_norm_kernel(const uint8_t* __restrict__ wg,
                                                               const uint16_t* __restrict__ sg,
                                                               const uint8_t* __restrict__ wu,
                                                               const uint16_t* __restrict__ su, NormAct act, int nb,
                                                               uint32_t nb_magic, int8_t* __restrict__ oq,
                                                               float* __restrict__ od) {
    extern __shared__ __align__(16) float smem[];
    __shared__ uint64_t exptab[32];
    QH_WSTAMP(3, 0);
    ExpTab et;
    et.load();
    const int tid = (int)threadIdx.x, ra = (int)blockIdx.x * QK;
    act.tmp = smem + gemv_tile_lds_bytes(nb * QK, 2 * QK, true) / 4;
    constexpr int kBlockBytes = DT == kQ8 ? QK : QK / 2;
    const GemvSegs<2> segs{{wg + (size_t)ra * nb * kBlockBytes, wu + (size_t)ra * nb * kBlockBytes},
                           {sg + (size_t)ra * nb, su + (size_t)ra * nb}};
    const float val =
        gemv_tile<DT, U, true, 2>(segs, nullptr, nullptr, nb, QK, 2 * QK, nb_magic, smem, NormActR<R, false>{act}, 3);
    QH_WSTAMP(3, 3);
    // wave 0 holds the block's 32 gate rows in lanes 0-31 and its 32 up rows in lanes 32-63: one half swap hands
    // lane l its up value (the exp table is stored by lanes 0-31 of the same wave, so no barrier is needed)
    if (tid < 2 * QK) {  // wave 0
        et.store(exptab);
        const uint32_t vb = __builtin_bit_cast(uint32_t, val);
        const auto sw = __builtin_amdgcn_permlane32_swap(vb, vb, false, false);
        const float u = __builtin_bit_cast(float, (uint32_t)sw[1]);
        if (tid < QK) quant_block32(val / (1.0f + dev_expf(-val, exptab)) * u, oq + ra, od + blockIdx.x);
    }
}

__global__ __launch_bounds__(256) void residual_add_kernel(float* __restrict__ x, const float* __restrict__ o, int n) {
    const int i = (int)(blockIdx.x * 256 + threadIdx.x);
    if (i < n) x[i] = x[i] + o[i];
}

// rmsnorm + quantization of one row (the final norm before the head), normed row also to `normed`.
template <int R>
__global__ __launch_bounds__(256) void norm_quant_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                         int D, float eps, int8_t* __restrict__ oq,
                                                         float* __restrict__ od, float* __restrict__ normed) {
    __shared__ __align__(16) float xs[8192 + kChainPad];
    const int tid = threadIdx.x, n4 = D / 4;
    RowF4<R> wr, xr;
    xr.load(x, n4);
    const SegWarm warm = D >= 128 ? seg_warm(x, D) : SegWarm{};
    wr.load(w, n4);
#pragma unroll
    for (int k = 0; k < R; ++k)
        if (tid + 256 * k < n4) reinterpret_cast<float4*>(xs)[tid + 256 * k] = xr.v[k];
    if (D >= 128) {  // uniform
        normalize_quant_lds(xs, D, rms_scale(seg_sum_squares(x, D, xr, warm), D, eps), wr, oq, od, normed);
    } else {
        __syncthreads();
        norm_quant_lds(xs, D, wr, eps, oq, od, normed);
    }
}

// Prefill / decode bookkeeping on the device.
__global__ void set_int_kernel(int* p, int value) { *p = value; }

// The first positions of a prefill stack's 32-token attention sub-chunks: p[i] = base + 32 i, i < n.
__global__ void set_subpos_kernel(int* p, int base, int n) {
    const int i = (int)threadIdx.x;
    if (i < n) p[i] = base + kChunk * i;
}

// The token a step chose: the sampler's pick when there is one, else the head's greedy top-1.
struct Pick {
    const int32_t* sampled;
    const qh_head_stats* stats;
    const int32_t* top1_full;
    __device__ __forceinline__ int id() const { return sampled ? *sampled : stats ? stats->top1 : *top1_full; }
};

// The chosen token becomes the next input, is appended to out[] and to the token history (session.cpp:45-46), and,
// after a decode step (advance), the position moves on.
__global__ void advance_kernel(Pick pick, TokenFeedback fb, int advance) { fb.apply(pick.id(), advance != 0); }

// Appends a prompt chunk to the token history (Session::feed, session.cpp:13-30), first emptying it when the chunk
// starts a sequence (reset). One workgroup.
__global__ __launch_bounds__(256) void history_append_kernel(const int32_t* __restrict__ tokens, int n, int reset,
                                                             int32_t* __restrict__ hist, int* __restrict__ hist_len,
                                                             int hist_cap) {
    __shared__ int base;
    if (threadIdx.x == 0) base = reset ? 0 : *hist_len;
    __syncthreads();
    const int b = base;
    for (int i = (int)threadIdx.x; i < n; i += 256)
        if (b + i < hist_cap) hist[b + i] = tokens[i];
    if (threadIdx.x == 0) *hist_len = b + n < hist_cap ? b + n : hist_cap;
}

}  // namespace

// ------------------------------------------------------------------------------------------------- host side

struct Decoder {
    qh_model_desc hp;
    std::vector<qh_tensor> t;  // the caller's device tensors, in the qh_decoder_create order
    const qh_tensor* lmh = nullptr;  // the LM head: the embedding, or lm_head.weight when untied (model.cpp:16)
    bool hadamard = false;           // FLAG_HADAMARD_DOWN (model_file.h:21)
    bool kv32 = false;               // an f32 KV cache (Model::load kv_f16 false)
    bool dense = false;              // some matrix is F32 / F16 (matvec_ref): f32 copies of the activations are kept
    float *fa = nullptr, *fb = nullptr;  // f32 normed layer input [kChunk][dim]; attention / SwiGLU output
                                         // [kChunk][max(dim, ffn_dim)] (the unquantized matrices' inputs)
    // device state
    uint16_t *kc = nullptr, *vc = nullptr;  // f16 cache (the default)
    float *kcf = nullptr, *vcf = nullptr;   // f32 cache, [n_layers][ctx][kv_dim] each
    float* cs = nullptr;
    float *x = nullptr, *o = nullptr, *q = nullptr, *k = nullptr, *v = nullptr, *g = nullptr, *u = nullptr,
          *hidden = nullptr;
    // int8 activations: qa holds a layer's normed input (and the head's), qb the attention / MLP inner activation
    int8_t *qa = nullptr, *qb = nullptr;
    float *da = nullptr, *db = nullptr;
    float* escr = nullptr;      // decode attention: a row of exp values, then one of weights, per head
    int escr_stride = 0;
    float* aws = nullptr;       // prefill stack attention: the scores
    size_t aws_bytes = 0;
    int32_t* tokens = nullptr;  // [kChunk] prefill input / [0] decode input
    // Prefill stack: the tokens whose norms and matmuls share one launch (kChunk, the reference's Model::kBatch, by
    // default; larger stacks run the matmul tile kernels at M up to kMaxStack). Over an f32 cache, or without the fused
    // kernels, attention runs each stack as 32-token sub-chunks in order, the sub-chunk i starting at subpos[i].
    int stack = kChunk;
    int* subpos = nullptr;
    int stack_end = 0;  // the current prefill stack's end position (host-side, for the attention plan)
    // token history (prompt ids since position 0, then each chosen id) and the optional query / sampler settings
    int32_t* hist = nullptr;  // [ctx_len + 1]
    int* hist_len = nullptr;
    bool has_query = false, has_sampler = false;
    qh_sampler_params qp{}, sp{};
    uint64_t* rng = nullptr;
    int32_t* sampled = nullptr;
    int* pos = nullptr;         // current position
    int* n_out = nullptr;
    int* status = nullptr;
    int32_t* out = nullptr;
    int out_cap = 0;
    // head
    float *logits = nullptr, *coarse = nullptr, *upper = nullptr;
    int32_t* rows = nullptr;
    qh_head_stats* stats = nullptr;
    void* head_ws = nullptr;
    size_t head_ws_bytes = 0;
    void* am_ws = nullptr;
    size_t am_ws_bytes = 0;
    void* sample_ws = nullptr;  // the sampler's sorted path (more than QH_SAMPLE_MAX_TOPK survivors)
    int32_t* top1_full = nullptr;
    bool fuse = true;  // fused decode kernels (QH_DECODER_FUSE=0 at creation selects one launch per operation)
    std::vector<void*> allocs;
    // The stage the kernels launched since the previous mark belong to (qh_decoder_step_timed).
    void mark(int id) const {
        if (KernelTimer* t = kernel_timer()) t->mark(id);
    }
};

namespace {

enum { T_EMBED, T_NORM, T_LAYER0 };
enum { L_ATTN_NORM, L_WQ, L_WK, L_WV, L_WO, L_BQ, L_BK, L_BV, L_FFN_NORM, L_WG, L_WU, L_WD, L_COUNT };

const qh_tensor& lt(const Decoder* d, int l, int which) { return d->t[T_LAYER0 + l * L_COUNT + which]; }
const float* lf(const Decoder* d, int l, int which) { return static_cast<const float*>(lt(d, l, which).data); }
const float* bias(const Decoder* d, int l, int which) { return d->hp.qkv_bias ? lf(d, l, which) : nullptr; }
const qh_tensor& head4(const Decoder* d) { return d->t[T_LAYER0 + d->hp.n_layers * L_COUNT]; }
const qh_tensor& head_err(const Decoder* d) { return d->t[T_LAYER0 + d->hp.n_layers * L_COUNT + 1]; }
const float* final_norm(const Decoder* d) { return static_cast<const float*>(d->t[T_NORM].data); }
bool dense_w(const qh_tensor& W) { return W.dtype == kF32 || W.dtype == kF16; }

const uint8_t* quants(const qh_tensor& W) { return static_cast<const uint8_t*>(W.data); }
const uint16_t* scales(const qh_tensor& W) {
    return reinterpret_cast<const uint16_t*>(quants(W) + qh_quant_bytes(W.dtype, W.rows, W.cols));
}
uint32_t nb_magic(int nb) { return nb == 1 ? 0u : (uint32_t)((0x100000000ull + (uint64_t)nb - 1) / (uint64_t)nb); }

hipError_t dalloc(Decoder* d, void** p, size_t bytes) {
    if (fault_alloc_fires()) return hipErrorOutOfMemory;  // qh_fault_alloc's forced failure
    hipError_t e = hipMalloc(p, bytes < 256 ? 256 : bytes);
    if (e == hipSuccess) d->allocs.push_back(*p);
    return e;
}

void dfree(Decoder* d, void* p) {
    if (!p) return;
    for (size_t i = 0; i < d->allocs.size(); ++i)
        if (d->allocs[i] == p) {
            d->allocs.erase(d->allocs.begin() + (long)i);
            break;
        }
    (void)hipFree(p);
}

// Whether a prefill stack's tokens go through attention together (attention_stack), not as 32-token sub-chunks.
bool stack_attention(const Decoder* d) { return d->fuse && !d->kv32; }

// The work buffers of a prefill stack of c tokens: the residual stream, projections, MLP rows, int8 activations and
// their scales, the f32 copies for unquantized matrices and the attention sub-chunks' positions. On failure the ones
// allocated stay listed (the caller frees them).
hipError_t alloc_stack(Decoder* d, int c) {
    const qh_model_desc& hp = d->hp;
    const size_t D = hp.dim, F = hp.ffn_dim, wide = D > F ? D : F, kvd = (size_t)hp.n_kv_heads * hp.head_dim;
    hipError_t e = hipSuccess;
    auto A = [&](void** p, size_t b) {
        if (e == hipSuccess) e = dalloc(d, p, b);
    };
    A((void**)&d->x, sizeof(float) * c * D);
    A((void**)&d->o, sizeof(float) * c * D);
    A((void**)&d->q, sizeof(float) * c * D);
    A((void**)&d->k, sizeof(float) * c * kvd);
    A((void**)&d->v, sizeof(float) * c * kvd);
    A((void**)&d->g, sizeof(float) * c * F);
    A((void**)&d->u, sizeof(float) * c * F);
    A((void**)&d->qa, c * wide);
    A((void**)&d->qb, c * wide);
    A((void**)&d->da, sizeof(float) * c * (wide / QK));
    A((void**)&d->db, sizeof(float) * c * (wide / QK));
    if (d->dense) {
        A((void**)&d->fa, sizeof(float) * c * D);
        A((void**)&d->fb, sizeof(float) * c * wide);
    }
    A((void**)&d->subpos, sizeof(int) * (kMaxStack / kChunk));
    // the stack attention's scores, where it runs: any size from the least works, so less is taken where the rest of
    // the memory is in use
    size_t least = 0, b = c > kChunk && stack_attention(d)
                              ? attn_stack_ws_bytes(hp.n_heads, hp.n_kv_heads, hp.ctx_len, c, &least) : 0;
    for (; b && e == hipSuccess; b = b / 2 < least ? least : b / 2) {
        e = dalloc(d, (void**)&d->aws, b);
        if (e == hipSuccess) {
            d->aws_bytes = b;
            break;
        }
        (void)hipGetLastError();
        if (e == hipErrorOutOfMemory && b > least) e = hipSuccess;
    }
    return e;
}

#define QH_TRY(expr)                                 \
    do {                                             \
        const hipError_t e_ = (expr);                \
        if (e_ != hipSuccess) return e_;             \
    } while (0)

// Calls f(dt, u, xl) with std::integral_constant arguments for the plan's dtype, unroll and activation staging, so a
// caller can launch KERNEL<dt, u, xl> for any plan gemv_plan makes.
// Calls f with the row-slot count (std::integral_constant) of rows of D floats.
template <typename F>
void by_row_slots(int D, F&& f) {
    if (row_slots(D / 4) == 1)
        f(std::integral_constant<int, 1>{});
    else
        f(std::integral_constant<int, 8>{});
}

template <typename F>
hipError_t plan_dispatch(int dtype, const GemvPlan& p, F&& f) {
    using std::integral_constant;
    auto go = [&](auto dt, auto u) {
        if (p.act_lds)
            f(dt, u, std::true_type{});
        else
            f(dt, u, std::false_type{});
        return hipGetLastError();
    };
    auto by_unroll = [&](auto dt) {
        switch (p.unroll) {
            case 1: return go(dt, integral_constant<int, 1>{});
            case 2: return go(dt, integral_constant<int, 2>{});
            case 4: return go(dt, integral_constant<int, 4>{});
            case 8: return go(dt, integral_constant<int, 8>{});
            default: return hipErrorInvalidValue;
        }
    };
    if (dtype == kQ8) return by_unroll(integral_constant<int, kQ8>{});
    if (dtype == kQ4) return by_unroll(integral_constant<int, kQ4>{});
    return hipErrorInvalidValue;
}

hipError_t embed(Decoder* d, const int32_t* tokens, int n, hipStream_t s) {
    const qh_tensor& emb = d->t[T_EMBED];
    by_row_slots(d->hp.dim, [&](auto r) {
        qh_launch((embed_norm_quant_kernel<decltype(r)::value>), dim3(n), dim3(256), 0, s, tokens, quants(emb),
                  emb.dtype, d->hp.dim, d->hp.vocab_size, d->x, lf(d, 0, L_ATTN_NORM), d->hp.norm_eps, d->qa, d->da,
                  d->fa, d->status);
    });
    return hipGetLastError();
}

// Model::linear / linear_batch (model.cpp:150-157, 336-347) of n tokens into out [n][ldo] (n == 1: out[r]): the
// integer-dot GEMV / matmul on the quantized activation for a Q8_0 / Q4_0 W, matvec_ref on its f32 copy for an
// F32 / F16 W. inner: the attention / SwiGLU output (qb / db / fb), else the normed layer input (qa / da / fa).
hipError_t linear(Decoder* d, float* out, int ldo, const qh_tensor& W, bool inner, int n, hipStream_t s) {
    if (dense_w(W)) return launch_gemv_dense(out, ldo, W, inner ? d->fb : d->fa, W.cols, n, 0, W.rows, s);
    const int8_t* xq = inner ? d->qb : d->qa;
    const float* xd = inner ? d->db : d->da;
    if (n == 1) return launch_gemv(out, W, xq, xd, 0, W.rows, gemv_plan(W.dtype, W.cols, W.rows), s);
    return launch_matmul(out, ldo, W, xq, xd, n, 0, W.rows, s);
}

// linear() of up to three matrices over one activation, the unquantized ones of one dtype that follow one another in one
// launch.
hipError_t linear_group(Decoder* d, const MmOut* m, int k, bool inner, int n, hipStream_t s) {
    for (int i = 0; i < k;) {
        int j = i + 1;
        if (dense_w(*m[i].W)) {
            while (j < k && m[j].W->dtype == m[i].W->dtype && m[j].W->cols == m[i].W->cols) ++j;
            QH_TRY(launch_dense_segs(m + i, j - i, inner ? d->fb : d->fa, m[i].W->cols, n, nullptr, s));
        } else {
            QH_TRY(linear(d, m[i].out, m[i].ldo, *m[i].W, inner, n, s));
        }
        i = j;
    }
    return hipSuccess;
}

// The normed-input fill of a decode kernel: layer input from the residual stream x, or (first layer) from the
// embedding of the current token, which workgroup 0 also stores as x.
NormAct make_norm(Decoder* d, bool embedding, const float* w) {
    NormAct a{};
    if (embedding) {
        const qh_tensor& emb = d->t[T_EMBED];
        a.eq = reinterpret_cast<const int8_t*>(quants(emb));
        a.es = reinterpret_cast<const uint16_t*>(quants(emb) + (size_t)emb.rows * emb.cols);
        a.tok = d->tokens;
        a.V = d->hp.vocab_size;
        a.x_out = d->x;
    } else {
        a.x = d->x;
    }
    a.status = d->status;
    a.w = w;
    a.eps = d->hp.norm_eps;
    a.D = d->hp.dim;
    a.tlk = -1;
    return a;
}

// LDS of a normed-input GEMV tile: the tile (codes staged in LDS) plus the D-float scratch of the norm.
size_t norm_tile_lds(int cols, int tile_rows, int D) {
    return gemv_tile_lds_bytes(cols, tile_rows, true) + 4 * ((size_t)D + kChainPad);
}

// Plan of the fused q/k/v launch, or false (one launch per operation) where the three projections differ in dtype
// or the plain GEMV would stream or the tile does not fit.
bool qkv_plan(const Decoder* d, int l, GemvPlan* p, size_t* lds) {
    const qh_tensor &wq = lt(d, l, L_WQ), &wk = lt(d, l, L_WK), &wv = lt(d, l, L_WV);
    if (!d->fuse || dense_w(wq) || wq.dtype != wk.dtype || wq.dtype != wv.dtype) return false;
    *p = gemv_plan(wq.dtype, wq.cols, wq.rows);
    *lds = norm_tile_lds(wq.cols, p->tile_rows, d->hp.dim);
    return !p->stream && *lds <= kFuseLds;
}

hipError_t launch_qkv_norm(Decoder* d, int l, const GemvPlan& p, size_t lds, const NormAct& act, hipStream_t s) {
    const qh_tensor &wq = lt(d, l, L_WQ), &wk = lt(d, l, L_WK), &wv = lt(d, l, L_WV);
    const int T = p.tile_rows;
    QkvSegs a{quants(wq), quants(wk), quants(wv), scales(wq), scales(wk), scales(wv), d->q, d->k, d->v,
              wq.rows, wk.rows, wv.rows, (wq.rows + T - 1) / T, (wk.rows + T - 1) / T};
    const unsigned grid = (unsigned)(a.tiles0 + a.tiles1 + (wv.rows + T - 1) / T);
    const int nb = wq.cols / QK;
    return plan_dispatch(wq.dtype, p, [&](auto dt, auto u, auto) {
        by_row_slots(act.D, [&](auto r) {
            if (act.eq)
                qh_launch((gemv_qkv_norm_kernel<decltype(dt)::value, decltype(u)::value, decltype(r)::value,
                                                         true>),
                                   dim3(grid), dim3(256), lds, s, a, act, nb, T, nb_magic(nb));
            else
                qh_launch((gemv_qkv_norm_kernel<decltype(dt)::value, decltype(u)::value, decltype(r)::value,
                                                         false>),
                                   dim3(grid), dim3(256), lds, s, a, act, nb, T, nb_magic(nb));
        });
    });
}

// x += W . (xq, xd) for one token: the GEMV tile kernel with the add in its epilogue, or (a streaming-size W, or
// one launch per operation) GEMV into d->o and a separate add.
hipError_t residual(Decoder* d, const qh_tensor& W, hipStream_t s) {
    const int8_t* xq = d->qb;
    const float* xd = d->db;
    if (dense_w(W)) {
        const MmOut m{&W, d->x, 0, 0, W.rows};
        return launch_dense_segs(&m, 1, d->fb, W.cols, 1, d->x, s);
    }
    const GemvPlan p = gemv_plan(W.dtype, W.cols, W.rows);
    if (d->fuse && !p.stream) {
        const int T = p.tile_rows, nb = W.cols / QK;
        const unsigned grid = (unsigned)((W.rows + T - 1) / T);
        const size_t lds = gemv_lds_bytes(W.cols, T, p.act_lds);
        return plan_dispatch(W.dtype, p, [&](auto dt, auto u, auto xl) {
            qh_launch((gemv_residual_kernel<decltype(dt)::value, decltype(u)::value, decltype(xl)::value>),
                               dim3(grid), dim3(256), lds, s, quants(W), scales(W), xq, xd, nb, W.rows, T,
                               nb_magic(nb), d->x);
        });
    }
    QH_TRY(launch_gemv(d->o, W, xq, xd, 0, W.rows, p, s));
    qh_launch(residual_add_kernel, dim3((unsigned)((W.rows + 255) / 256)), dim3(256), 0, s, d->x, d->o,
                       W.rows);
    return hipGetLastError();
}

// The down projection's input from gate / up rows g, u of n tokens (ffn values each): SwiGLU and quantization, with
// the block-256 Walsh-Hadamard transform between them when the model has FLAG_HADAMARD_DOWN (model.cpp:216-220).
hipError_t swiglu_down_input(Decoder* d, int F, int n, hipStream_t s) {
    if (d->hadamard) {
        qh_launch(swiglu_fwht_quant_kernel, dim3((unsigned)(F / 256), (unsigned)n), dim3(256), 0, s, d->g, d->u, F,
                  d->qb, d->db, d->fb);
    } else {
        const long nblk = (long)n * F / QK;
        qh_launch(swiglu_quant_kernel, dim3((unsigned)((nblk * QK + 255) / 256)), dim3(256), 0, s, d->g, d->u, nblk,
                  d->qb, d->db, d->fb);
    }
    return hipGetLastError();
}

hipError_t norm_quant(Decoder* d, const float* w, float* normed, hipStream_t s) {
    by_row_slots(d->hp.dim, [&](auto r) {
        qh_launch((norm_quant_kernel<decltype(r)::value>), dim3(1), dim3(256), 0, s, d->x, w, d->hp.dim,
                           d->hp.norm_eps, d->qa, d->da, normed);
    });
    return hipGetLastError();
}

// rmsnorm (ffn_norm) of one token, gate / up, SwiGLU and quantization into qb / db.
hipError_t gate_up(Decoder* d, int l, hipStream_t s) {
    const qh_tensor &wg = lt(d, l, L_WG), &wu = lt(d, l, L_WU);
    const int nb = wg.cols / QK;
    const size_t lds = norm_tile_lds(wg.cols, 2 * QK, d->hp.dim);
    if (d->fuse && !d->hadamard && !d->dense && wg.dtype == wu.dtype && lds <= kFuseLds) {
        const unsigned grid = (unsigned)(wg.rows / QK);
        NormAct act = make_norm(d, false, lf(d, l, L_FFN_NORM));
        act.tlk = 3;
        by_row_slots(d->hp.dim, [&](auto r) {
            constexpr int R = decltype(r)::value;
            if (wg.dtype == kQ8)
                qh_launch((gemv_swiglu_norm_kernel<kQ8, 8, R>), dim3(grid), dim3(256), lds, s, quants(wg),
                                   scales(wg), quants(wu), scales(wu), act, nb, nb_magic(nb), d->qb, d->db);
            else
                qh_launch((gemv_swiglu_norm_kernel<kQ4, 8, R>), dim3(grid), dim3(256), lds, s, quants(wg),
                                   scales(wg), quants(wu), scales(wu), act, nb, nb_magic(nb), d->qb, d->db);
        });
        return hipGetLastError();
    }
    QH_TRY(norm_quant(d, lf(d, l, L_FFN_NORM), d->fa, s));
    const MmOut m[2] = {{&wg, d->g, 0, 0, wg.rows}, {&wu, d->u, 0, 0, wu.rows}};
    QH_TRY(linear_group(d, m, 2, false, 1, s));
    return swiglu_down_input(d, wg.rows, 1, s);
}

// Attention of a chunk of n <= kChunk tokens at positions *pos_dev .. + n - 1 whose projections start at row r0 of
// q / k / v; outputs to rows r0 .. of qb / db (and fb).
hipError_t attention_chunk(Decoder* d, int l, int n, int r0, const int* pos_dev, hipStream_t s) {
    const qh_model_desc& hp = d->hp;
    const size_t layer_k = (size_t)hp.ctx_len * hp.n_kv_heads * hp.head_dim;
    const size_t layer_v = (size_t)v_ctx(hp.ctx_len) * hp.n_kv_heads * hp.head_dim;
    const size_t qd = (size_t)hp.n_heads * hp.head_dim, kvd = (size_t)hp.n_kv_heads * hp.head_dim;
    const float *q = d->q + r0 * qd, *k = d->k + r0 * kvd, *v = d->v + r0 * kvd;
    int8_t* oq = d->qb + r0 * qd;
    float* od = d->db + r0 * (qd / QK);
    float* of = d->fb ? d->fb + r0 * qd : nullptr;
    const dim3 grid(hp.n_heads, n);
    if (d->kv32) {  // the f32 cache: prefill and decode alike
        const size_t layer_kv = (size_t)hp.ctx_len * hp.n_kv_heads * hp.head_dim;
        if (hp.head_dim == 64)
            qh_launch((attention_f32_kernel<64>), grid, dim3(256), 0, s, q, k, v, bias(d, l, L_BQ),
                      bias(d, l, L_BK), bias(d, l, L_BV), d->cs, pos_dev, hp.ctx_len, hp.n_heads, hp.n_kv_heads,
                      d->kcf + l * layer_kv, d->vcf + l * layer_kv, oq, od, d->status, of);
        else
            qh_launch((attention_f32_kernel<128>), grid, dim3(256), 0, s, q, k, v, bias(d, l, L_BQ),
                      bias(d, l, L_BK), bias(d, l, L_BV), d->cs, pos_dev, hp.ctx_len, hp.n_heads, hp.n_kv_heads,
                      d->kcf + l * layer_kv, d->vcf + l * layer_kv, oq, od, d->status, of);
    } else if (hp.head_dim == 64) {
        qh_launch((attention_kernel<64, 2>), grid, dim3(256), 0, s, q, k, v, bias(d, l, L_BQ), bias(d, l, L_BK),
                  bias(d, l, L_BV), d->cs, pos_dev, hp.ctx_len, hp.n_heads, hp.n_kv_heads, d->kc + l * layer_k,
                  d->vc + l * layer_v, oq, od, d->status, of);
    } else {
        qh_launch((attention_kernel<128>), grid, dim3(256), 0, s, q, k, v, bias(d, l, L_BQ), bias(d, l, L_BK),
                  bias(d, l, L_BV), d->cs, pos_dev, hp.ctx_len, hp.n_heads, hp.n_kv_heads, d->kc + l * layer_k,
                  d->vc + l * layer_v, oq, od, d->status, of);
    }
    return hipGetLastError();
}

// Whether a prefill stack of n tokens at pos0 has so few workgroups that a workgroup per query head and token
// (attention_kernel), or per query head and four tokens (attention_stack_kernel, up to kStackCtx rows), is faster than
// the pair groups of launch_attention_stack, which take a quarter to a sixteenth of the workgroups and are serial for
// longer. Measured in us a layer (whole layer, these kernels and the pair groups):
//   head_dim 64, up to 1,024 rows, two workgroups of four tokens to a CU: 14 heads, 33 tokens at 896 58 and 71, 128 at 256
//     56 and 58, 146 at 200 61.8 and 60.4; where the tokens' row counts differ the short ones fill in: 4 heads, 740 at 0
//     67 and 71, 900 at 0 79.9 and 80.6, 620 at 400 84.5 and 82.1.
//   head_dim 64, beyond: two workgroups to a CU, 4 heads 128 tokens at 4,000 94 and 138, 14 heads 33 at 7,000 133 and 196;
//     a second round of them pays until the rows outweigh it: 14 heads, 64 at 2,500 110 and 116, 73 at 5,500 183 and 176.
//   head_dim 128, one workgroup to a CU: 2 heads, 128 at 700 55 and 75, 1,000 64 and 79, 4,000 151 and 138; a second
//     round only up to 1,024 rows and past about 200: 2 heads, 140 at 700 72 and 78, at 0 52.0 and 50.0, at 1,000 89 and 82.
bool few_workgroups(const qh_model_desc& hp, int n, int pos0) {
    const long cus = device_cus(), w = (long)hp.n_heads * n, w4 = (long)hp.n_heads * ((n + kStackTok - 1) / kStackTok);
    const long rows = pos0 + n, twice_mean = 2l * pos0 + n;  // the last token's rows, and twice their mean
    if (hp.head_dim == 64) {
        if (rows <= kStackCtx) return w4 <= 2 * cus || 5 * w4 * twice_mean <= 16 * cus * rows;
        return w <= 2 * cus || (w <= 4 * cus && w * rows <= 4 * cus * 4096);
    }
    if (rows <= kStackCtx) return w <= cus || (w <= 2 * cus && twice_mean >= 400);
    return w <= cus && rows <= 2700;
}

// Attention of a prefill stack of n > kChunk tokens at positions *d->pos ..: the f16 cache rows of every token of the
// stack first (kv_store_kernel), then the stack's (token, head) pairs together (launch_attention_stack), or, where those
// are few, one workgroup per head and token (each its own chunk, every earlier row read from the cache) or four tokens.
hipError_t attention_stack(Decoder* d, int l, int n, hipStream_t s) {
    const qh_model_desc& hp = d->hp;
    const size_t layer_k = (size_t)hp.ctx_len * hp.n_kv_heads * hp.head_dim;
    const size_t layer_v = (size_t)v_ctx(hp.ctx_len) * hp.n_kv_heads * hp.head_dim;
    uint16_t *kc = d->kc + l * layer_k, *vc = d->vc + l * layer_v;
    if (hp.head_dim == 64)
        qh_launch((kv_store_kernel<64>), dim3(n), dim3(256), 0, s, d->k, d->v, bias(d, l, L_BK), bias(d, l, L_BV),
                  d->cs, d->pos, hp.ctx_len, hp.n_kv_heads, kc, vc);
    else
        qh_launch((kv_store_kernel<128>), dim3(n), dim3(256), 0, s, d->k, d->v, bias(d, l, L_BK), bias(d, l, L_BV),
                  d->cs, d->pos, hp.ctx_len, hp.n_kv_heads, kc, vc);
    QH_TRY(hipGetLastError());
    const int pos0 = d->stack_end - n;
    if (few_workgroups(hp, n, pos0))
        return launch_attention_few({d->q, d->k, d->v, bias(d, l, L_BQ), bias(d, l, L_BK), bias(d, l, L_BV), d->cs, d->pos,
                                     n, hp.ctx_len, hp.n_heads, hp.n_kv_heads, kc, vc, d->qb, d->db, d->status, d->fb},
                                    hp.head_dim, d->stack_end, s);
    AttnStack a{};
    a.q = d->q;
    a.bq = bias(d, l, L_BQ);
    a.cs = d->cs;
    a.kc = kc;
    a.vc = vc;
    a.ctx = hp.ctx_len;
    a.n_heads = hp.n_heads;
    a.n_kv = hp.n_kv_heads;
    a.n = n;
    a.pos0 = pos0;
    a.oq = d->qb;
    a.od = d->db;
    a.of = d->fb;
    return launch_attention_stack(a, hp.head_dim, d->aws, d->aws_bytes, s);
}

hipError_t attention(Decoder* d, int l, int n, hipStream_t s) {
    const qh_model_desc& hp = d->hp;
    if (n > kChunk && stack_attention(d)) return attention_stack(d, l, n, s);
    if (n > kChunk) {  // a prefill stack without it: its 32-token sub-chunks in order (each reads the rows the ones before wrote)
        for (int i = 0; i * kChunk < n; ++i)
            QH_TRY(attention_chunk(d, l, min(kChunk, n - i * kChunk), i * kChunk, d->subpos + i, s));
        return hipSuccess;
    }
    if (n == 1 && hp.head_dim == 64 && d->fuse && !d->kv32) {  // decode: one 16-wave workgroup per head
        const size_t layer_k = (size_t)hp.ctx_len * hp.n_kv_heads * hp.head_dim;
        const size_t layer_v = (size_t)v_ctx(hp.ctx_len) * hp.n_kv_heads * hp.head_dim;
        qh_launch((attention_decode_kernel<64>), dim3(hp.n_heads / hp.n_kv_heads, hp.n_kv_heads), dim3(1024), 0, s,
                  d->q, d->k, d->v, d->kc + l * layer_k, d->pos, hp.ctx_len, hp.n_heads / hp.n_kv_heads,
                  bias(d, l, L_BQ), bias(d, l, L_BK), hp.n_kv_heads, bias(d, l, L_BV), d->cs, d->vc + l * layer_v,
                  d->qb, d->db, d->escr, d->escr_stride, d->status, d->fb);
        return hipGetLastError();
    }
    return attention_chunk(d, l, n, 0, d->pos, s);  // a chunk of the prefill (either cache), or the f32 cache
}

// One decode step's layers for the token in d->tokens[0], from its embedding. Leaves the final normed hidden state
// in d->hidden and its quantization in qa / da for the head.
hipError_t decode_layers(Decoder* d, hipStream_t s) {
    const qh_model_desc& hp = d->hp;
    for (int l = 0; l < hp.n_layers; ++l) {
        GemvPlan p;
        size_t lds = 0;
        if (qkv_plan(d, l, &p, &lds) && (l > 0 || d->t[T_EMBED].dtype == kQ8)) {
            NormAct act = make_norm(d, l == 0, lf(d, l, L_ATTN_NORM));
            act.tlk = 0;
            QH_TRY(launch_qkv_norm(d, l, p, lds, act, s));
        } else {
            if (l == 0)
                QH_TRY(embed(d, d->tokens, 1, s));
            else
                QH_TRY(norm_quant(d, lf(d, l, L_ATTN_NORM), d->fa, s));
            const qh_tensor &wq = lt(d, l, L_WQ), &wk = lt(d, l, L_WK), &wv = lt(d, l, L_WV);
            const MmOut m[3] = {{&wq, d->q, 0, 0, wq.rows}, {&wk, d->k, 0, 0, wk.rows}, {&wv, d->v, 0, 0, wv.rows}};
            QH_TRY(linear_group(d, m, 3, false, 1, s));
        }
        d->mark(l * QH_STAGES_PER_LAYER + QH_STAGE_QKV);
        QH_TRY(attention(d, l, 1, s));
        d->mark(l * QH_STAGES_PER_LAYER + QH_STAGE_ATTENTION);
        QH_TRY(residual(d, lt(d, l, L_WO), s));
        d->mark(l * QH_STAGES_PER_LAYER + QH_STAGE_O);
        QH_TRY(gate_up(d, l, s));
        d->mark(l * QH_STAGES_PER_LAYER + QH_STAGE_GATE_UP);
        QH_TRY(residual(d, lt(d, l, L_WD), s));
        d->mark(l * QH_STAGES_PER_LAYER + QH_STAGE_DOWN);
    }
    QH_TRY(norm_quant(d, final_norm(d), d->hidden, s));
    d->mark(QH_STAGE_FINAL_NORM);
    return hipSuccess;
}

// Matrices over one activation, in as few launches as their formats allow: runs of one dtype and width share one.
// Gate / up / SwiGLU / quantization of a prefill chunk as one launch (matmul_swiglu_kernel) into qb / db, or false
// (the matmul launch and swiglu_quant_kernel instead: one launch per operation, different formats or widths, rows
// not a multiple of 32, unaligned operands).
bool swiglu_fused(Decoder* d, const qh_tensor& wg, const qh_tensor& wu, int n, hipStream_t s) {
    if (n > kChunk || !d->fuse || d->hadamard || d->dense || wg.dtype != wu.dtype || wg.rows != wu.rows || wg.cols != wu.cols || wg.rows % QK != 0 ||
        (wg.dtype != kQ8 && wg.dtype != kQ4) || wg.cols % QK != 0 || wg.cols < 2 * QK)
        return false;
    const uint8_t *qg = quants(wg), *qu = quants(wu);
    if (((reinterpret_cast<uintptr_t>(qg) | reinterpret_cast<uintptr_t>(qu) | reinterpret_cast<uintptr_t>(d->qa)) &
         15u) != 0)
        return false;
    const int n_tg = (n + 15) / 16;
    const dim3 grid((unsigned)(wg.rows / QK * n_tg));
    const bool short_rows = wg.cols / QK <= 2 * kSwKC;
#define QH_SW(DT, SH)                                                                                            \
    qh_launch((matmul_swiglu_kernel<DT, SH>), grid, dim3(256), 0, s, qg, scales(wg), qu, scales(wu), d->qa, d->da, \
              wg.cols, wg.rows, n, n_tg, d->qb, d->db)
    if (wg.dtype == kQ4) {
        if (short_rows)
            QH_SW(kQ4, true);
        else
            QH_SW(kQ4, false);
    } else {
        if (short_rows)
            QH_SW(kQ8, true);
        else
            QH_SW(kQ8, false);
    }
#undef QH_SW
    return true;
}

hipError_t matmul_group(const MmOut* m, int k, const int8_t* xq, const float* xd, int n, hipStream_t s) {
    for (int i = 0; i < k;) {
        int j = i + 1;
        while (j < k && m[j].W->dtype == m[i].W->dtype && m[j].W->cols == m[i].W->cols) ++j;
        QH_TRY(launch_matmul_segs(m + i, j - i, xq, xd, n, s));
        i = j;
    }
    return hipSuccess;
}

// All layers for a chunk of n tokens whose embeddings are in d->x[0..n) and normed inputs in qa / da, positions
// from *d->pos. Leaves the last layer's down projection in d->o (not yet added to the residual stream).
hipError_t prefill_layers(Decoder* d, int n, hipStream_t s) {
    const qh_model_desc& hp = d->hp;
    const int D = hp.dim, F = hp.ffn_dim;
    for (int l = 0; l < hp.n_layers; ++l) {
        if (l > 0) {
            by_row_slots(D, [&](auto r) {
                qh_launch((add_rmsnorm_quant_kernel<decltype(r)::value>), dim3(n), dim3(256), 0, s, d->x,
                                   d->o, lf(d, l, L_ATTN_NORM), D, hp.norm_eps, d->qa, d->da, d->fa);
            });
            QH_TRY(hipGetLastError());
        }
        const qh_tensor &wq = lt(d, l, L_WQ), &wk = lt(d, l, L_WK), &wv = lt(d, l, L_WV);
        const MmOut qkv[3] = {{&wq, d->q, wq.rows, 0, wq.rows}, {&wk, d->k, wk.rows, 0, wk.rows},
                              {&wv, d->v, wv.rows, 0, wv.rows}};
        if (dense_w(wq) || dense_w(wk) || dense_w(wv)) {
            QH_TRY(linear_group(d, qkv, 3, false, n, s));
        } else {
            QH_TRY(matmul_group(qkv, 3, d->qa, d->da, n, s));
        }
        QH_TRY(attention(d, l, n, s));
        const qh_tensor& wo = lt(d, l, L_WO);
        QH_TRY(linear(d, d->o, wo.rows, wo, true, n, s));
        by_row_slots(D, [&](auto r) {
            qh_launch((add_rmsnorm_quant_kernel<decltype(r)::value>), dim3(n), dim3(256), 0, s, d->x, d->o,
                               lf(d, l, L_FFN_NORM), D, hp.norm_eps, d->qa, d->da, d->fa);
        });
        QH_TRY(hipGetLastError());
        const qh_tensor &wg = lt(d, l, L_WG), &wu = lt(d, l, L_WU), &wd = lt(d, l, L_WD);
        // a prefill stack: gate / up with the SwiGLU epilogue in one tile launch where the plan allows it
        const hipError_t sw = n > kChunk && d->fuse && !d->hadamard && !d->dense
                                  ? launch_matmul_swiglu(wg, wu, d->qa, d->da, n, d->qb, d->db, s)
                                  : hipErrorNotSupported;
        if (sw != hipErrorNotSupported) {
            QH_TRY(sw);
        } else if (!swiglu_fused(d, wg, wu, n, s)) {
            const MmOut gu[2] = {{&wg, d->g, wg.rows, 0, wg.rows}, {&wu, d->u, wu.rows, 0, wu.rows}};
            if (dense_w(wg) || dense_w(wu)) {
                QH_TRY(linear_group(d, gu, 2, false, n, s));
            } else {
                QH_TRY(matmul_group(gu, 2, d->qa, d->da, n, s));
            }
            QH_TRY(swiglu_down_input(d, F, n, s));
        }
        QH_TRY(hipGetLastError());
        QH_TRY(linear(d, d->o, wd.rows, wd, true, n, s));
    }
    return hipSuccess;
}

// The head on the quantized final hidden state in qa / da; top_k > 0 uses the shortlist.
// The head query of a forward (Session::head_query, session.cpp:63-79): with a query set, top_k follows its
// temperature and top_k, and its repetition penalty makes the history window the must ids; else the caller's top_k.
int query_top_k(const Decoder* d, int top_k) {
    if (!d->has_query) return top_k;
    return d->qp.temperature <= 0.f ? 1 : d->qp.top_k;
}

// The token history as a device-resident id list: its last `window` ids (all when window <= 0).
HeadMust history_window(const Decoder* d, int window) {
    HeadMust m;
    m.ids = d->hist;
    m.len_dev = d->hist_len;
    m.window = window;
    return m;
}

// The shortlist head runs for top_k > 0 queries on a model with head_q4 / head_err or with a nibble-plane LM head.
bool has_shortlist(const Decoder* d) { return head4(d).data != nullptr || d->lmh->dtype == kQ8P; }
bool shortlist_on(const Decoder* d, int top_k) { return query_top_k(d, top_k) > 0 && has_shortlist(d); }

// The feedback of a chosen token into the decoder's state.
TokenFeedback token_feedback(Decoder* d) {
    TokenFeedback fb;
    fb.token = d->tokens;
    fb.pos = d->pos;
    fb.n_out = d->n_out;
    fb.out = d->out;
    fb.out_cap = d->out_cap;
    fb.hist = d->hist;
    fb.hist_len = d->hist_len;
    fb.hist_cap = d->hp.ctx_len + 1;
    return fb;
}

// advance: a greedy decode step through the shortlist head, whose last kernel then also feeds the token back.
hipError_t run_head(Decoder* d, int top_k, hipStream_t s, bool advance = false) {
    const qh_tensor& h8 = *d->lmh;
    if (shortlist_on(d, top_k)) {
        qh_head_query q{query_top_k(d, top_k), d->hp.vocab_size, nullptr, 0};
        qh_head_out out{d->logits, d->coarse, d->upper, d->rows, d->stats};
        const HeadMust must = d->has_query && d->qp.repeat_penalty != 1.f ? history_window(d, d->qp.repeat_window)
                                                                           : HeadMust{};
        const TokenFeedback fb = token_feedback(d);
        return launch_shortlist_head(h8, head4(d), head_err(d), d->qa, d->da, q, must, out, d->head_ws, s,
                                     advance ? &fb : nullptr);
    }
    if (dense_w(h8))  // Model::linear on the final normed state itself (matvec_ref)
        QH_TRY(launch_gemv_dense(d->logits, 0, h8, d->hidden, h8.cols, 1, 0, h8.rows, s));
    else if (h8.dtype == kQ8P)
        QH_TRY(launch_gemv_planes(d->logits, h8, d->qa, d->da, 0, h8.rows, s));
    else
        QH_TRY(launch_gemv(d->logits, h8, d->qa, d->da, 0, h8.rows, gemv_plan(h8.dtype, h8.cols, h8.rows), s));
    return launch_argmax(d->logits, d->hp.vocab_size, d->top1_full, d->am_ws, s);
}


}  // namespace

// ------------------------------------------------------------------------------------------------- C-ABI glue

int decoder_create(const qh_model_desc* hp, const qh_tensor* tensors, int n_tensors, Decoder** out) {
    auto* d = new Decoder();
    d->hp = *hp;
    const char* fuse = getenv("QH_DECODER_FUSE");
    d->fuse = !(fuse && strcmp(fuse, "0") == 0);
    d->t.assign(tensors, tensors + n_tensors);
    const size_t n_lm = T_LAYER0 + (size_t)hp->n_layers * L_COUNT + 2;  // lm_head.weight's slot, when given
    d->lmh = d->t.size() > n_lm && d->t[n_lm].data ? &d->t[n_lm] : &d->t[T_EMBED];
    d->hadamard = (hp->flags & QH_FLAG_HADAMARD_DOWN) != 0;
    d->kv32 = hp->kv_f32 != 0;
    d->dense = dense_w(*d->lmh);
    for (int l = 0; l < hp->n_layers; ++l)
        for (int m : {L_WQ, L_WK, L_WV, L_WO, L_WG, L_WU, L_WD}) d->dense = d->dense || dense_w(lt(d, l, m));
    const int D = hp->dim, V = hp->vocab_size, hd = hp->head_dim;
    const size_t kvd = (size_t)hp->n_kv_heads * hd;
    const size_t kv_bytes = (size_t)hp->n_layers * hp->ctx_len * kvd * 2;
    const size_t v_bytes = (size_t)hp->n_layers * v_ctx(hp->ctx_len) * kvd * 2;
    const size_t kv32_bytes = (size_t)hp->n_layers * hp->ctx_len * kvd * 4;
    hipError_t e = hipSuccess;
    auto A = [&](void** p, size_t b) {
        if (e == hipSuccess) e = dalloc(d, p, b);
    };
    if (d->kv32) {
        A((void**)&d->kcf, kv32_bytes);
        A((void**)&d->vcf, kv32_bytes);
    } else {
        A((void**)&d->kc, kv_bytes);
        A((void**)&d->vc, v_bytes);
    }
    A((void**)&d->cs, sizeof(float) * (size_t)hp->ctx_len * hd);
    if (e == hipSuccess) e = alloc_stack(d, kChunk);
    A((void**)&d->hidden, sizeof(float) * D);
    d->escr_stride = escr_stride(hp->ctx_len);
    A((void**)&d->escr, sizeof(float) * 2 * (size_t)hp->n_heads * d->escr_stride);  // exp rows, weight rows
    A((void**)&d->tokens, sizeof(int32_t) * kChunk);
    A((void**)&d->hist, sizeof(int32_t) * ((size_t)hp->ctx_len + 1));
    A((void**)&d->hist_len, 256);
    A((void**)&d->rng, 256);
    A((void**)&d->sampled, 256);
    A((void**)&d->pos, 256);
    A((void**)&d->n_out, 256);
    A((void**)&d->status, 256);
    A((void**)&d->logits, sizeof(float) * V);
    A((void**)&d->coarse, sizeof(float) * V);
    A((void**)&d->upper, sizeof(float) * V);
    A((void**)&d->rows, sizeof(int32_t) * (size_t)(V + 64));
    A((void**)&d->stats, sizeof(qh_head_stats));
    A((void**)&d->top1_full, 256);
    if (has_shortlist(d)) {
        d->head_ws_bytes = head_workspace_bytes(V, D, 1);  // the same for every top_k the selection holds
        A(&d->head_ws, d->head_ws_bytes);
    }
    d->am_ws_bytes = argmax_workspace_bytes(V);
    A(&d->am_ws, d->am_ws_bytes);
    if (V <= QH_SAMPLE_MAX_VOCAB) A(&d->sample_ws, sample_workspace_bytes(V));
    if (e != hipSuccess) {
        decoder_destroy(d);
        return check_hip(e, "qh_decoder_create allocation");
    }
    // RoPE angle table with the reference's formula and the host's libm (ops_ref.cpp:201-214).
    std::vector<float> cs((size_t)hp->ctx_len * hd);
    const int half = hd / 2;
    for (int p = 0; p < hp->ctx_len; ++p)
        for (int i = 0; i < half; ++i) {
            const float freq = powf(hp->rope_theta, -2.0f * (float)i / (float)hd);
            const float angle = (float)p * freq;
            cs[((size_t)p * half + i) * 2] = cosf(angle);
            cs[((size_t)p * half + i) * 2 + 1] = sinf(angle);
        }
    e = hipMemcpy(d->cs, cs.data(), sizeof(float) * cs.size(), hipMemcpyHostToDevice);
    for (int* p : {d->n_out, d->pos, d->status, d->hist_len})
        if (e == hipSuccess) e = hipMemset(p, 0, 256);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e != hipSuccess) {
        decoder_destroy(d);
        return check_hip(e, "qh_decoder_create upload");
    }
    *out = d;
    return QH_OK;
}

void decoder_destroy(Decoder* d) {
    if (!d) return;
    for (void* p : d->allocs) (void)hipFree(p);
    delete d;
}

hipError_t decoder_set_prefill_stack(Decoder* d, int c) {
    if (c == d->stack) return hipSuccess;
    QH_TRY(hipDeviceSynchronize());  // nothing in flight uses the buffers that are replaced
    void** slots[] = {(void**)&d->x,  (void**)&d->o,  (void**)&d->q,  (void**)&d->k,  (void**)&d->v,
                      (void**)&d->g,  (void**)&d->u,  (void**)&d->qa, (void**)&d->qb, (void**)&d->da,
                      (void**)&d->db, (void**)&d->fa, (void**)&d->fb, (void**)&d->subpos, (void**)&d->aws};
    constexpr int kSlots = (int)(sizeof(slots) / sizeof(slots[0]));
    void* old[kSlots];
    for (int i = 0; i < kSlots; ++i) {
        old[i] = *slots[i];
        *slots[i] = nullptr;
    }
    const hipError_t e = alloc_stack(d, c);
    for (int i = 0; i < kSlots; ++i) {
        void* drop = e == hipSuccess ? old[i] : *slots[i];
        if (e != hipSuccess) *slots[i] = old[i];  // keep the previous stack on failure
        dfree(d, drop);
    }
    if (e == hipSuccess) d->stack = c;
    return e;
}

hipError_t decoder_prefill(Decoder* d, const int32_t* tokens, int n, int pos0, int top_k, hipStream_t s) {
    const qh_model_desc& hp = d->hp;
    const int D = hp.dim;
    qh_launch(set_int_kernel, dim3(1), dim3(1), 0, s, d->status, 0);
    QH_TRY(hipGetLastError());
    qh_launch(history_append_kernel, dim3(1), dim3(256), 0, s, tokens, n, pos0 == 0 ? 1 : 0, d->hist,
                       d->hist_len, hp.ctx_len + 1);
    QH_TRY(hipGetLastError());
    int last = 0;
    for (int c0 = 0; c0 < n; c0 += d->stack) {
        const int m = n - c0 < d->stack ? n - c0 : d->stack;
        if (m > kChunk && !stack_attention(d)) {
            qh_launch(set_subpos_kernel, dim3(1), dim3(kMaxStack / kChunk), 0, s, d->subpos, pos0 + c0,
                      (m + kChunk - 1) / kChunk);
            QH_TRY(hipGetLastError());
        }
        qh_launch(set_int_kernel, dim3(1), dim3(1), 0, s, d->pos, pos0 + c0);
        QH_TRY(hipGetLastError());
        d->stack_end = pos0 + c0 + m;
        QH_TRY(embed(d, tokens + c0, m, s));
        QH_TRY(prefill_layers(d, m, s));
        last = m - 1;
    }
    // final residual add, norm and quantization of the last token only, then the head
    by_row_slots(D, [&](auto r) {
        qh_launch((add_rmsnorm_quant_kernel<decltype(r)::value>), dim3(1), dim3(256), 0, s,
                           d->x + (size_t)last * D, d->o + (size_t)last * D, final_norm(d), D, hp.norm_eps, d->qa,
                           d->da, d->hidden);
    });
    QH_TRY(hipGetLastError());
    QH_TRY(run_head(d, top_k, s));
    qh_launch(set_int_kernel, dim3(1), dim3(1), 0, s, d->pos, pos0 + n);
    return hipGetLastError();
}

// Picks the token from the last head call (the sampler when one is set) and feeds it back (advance: a decode step).
hipError_t pick_and_advance(Decoder* d, int top_k, bool advance, hipStream_t s) {
    const bool sl = shortlist_on(d, top_k);
    Pick pick{nullptr, sl ? d->stats : nullptr, d->top1_full};
    if (d->has_sampler) {
        const HeadMust hist = d->sp.repeat_penalty != 1.f ? history_window(d, d->sp.repeat_window) : HeadMust{};
        QH_TRY(launch_sample(d->logits, d->hp.vocab_size, sl ? d->rows : nullptr, sl ? d->stats : nullptr, hist,
                             d->sp, d->rng, d->sampled, d->sample_ws, s));
        pick.sampled = d->sampled;
    }
    qh_launch(advance_kernel, dim3(1), dim3(1), 0, s, pick, token_feedback(d), advance ? 1 : 0);
    return hipGetLastError();
}

hipError_t decoder_step(Decoder* d, int top_k, hipStream_t s) {
    QH_TRY(decode_layers(d, s));
    if (!d->has_sampler && shortlist_on(d, top_k)) {  // greedy: fed back in the head
        QH_TRY(run_head(d, top_k, s, true));
        d->mark(QH_STAGE_HEAD);
        return hipSuccess;
    }
    QH_TRY(run_head(d, top_k, s));
    d->mark(QH_STAGE_HEAD);
    QH_TRY(pick_and_advance(d, top_k, true, s));
    d->mark(QH_STAGE_PICK);
    return hipSuccess;
}

int decoder_step_timed(Decoder* d, int top_k, hipStream_t s, float* us, int32_t* stage, int cap, int32_t* n) {
    KernelTimer t;
    t.ev.assign(2 * (size_t)cap, nullptr);
    int rc = QH_OK;
    for (hipEvent_t& e : t.ev)
        if (!rc) rc = check_hip(hipEventCreate(&e), "hipEventCreate");
    if (!rc) {
        kernel_timer() = &t;
        const hipError_t e = decoder_step(d, top_k, s);
        kernel_timer() = nullptr;
        rc = check_hip(e, "qh_decoder_step_timed");
    }
    if (!rc) rc = check_hip(hipStreamSynchronize(s), "hipStreamSynchronize");
    if (!rc && t.launched > cap)
        rc = fail(QH_ERR_NOMEM, "qh_decoder_step_timed: the step launched %d kernels, more than the %d timing slots (the "
                  "step has run)", t.launched, cap);
    for (int i = 0; !rc && i < t.n; ++i) {
        rc = check_hip(hipEventElapsedTime(&us[i], t.ev[2 * i], t.ev[2 * i + 1]), "hipEventElapsedTime");
        us[i] *= 1e3f;
        stage[i] = t.stage[i];
    }
    for (hipEvent_t e : t.ev)
        if (e) (void)hipEventDestroy(e);
    if (!rc || t.launched > cap) *n = t.launched;
    return rc;
}

hipError_t decoder_begin(Decoder* d, int top_k, int32_t* out, int out_cap, hipStream_t s) {
    d->out = out;
    d->out_cap = out_cap;
    qh_launch(set_int_kernel, dim3(1), dim3(1), 0, s, d->n_out, 0);
    QH_TRY(hipGetLastError());
    return pick_and_advance(d, top_k, false, s);
}

int decoder_ctx(const Decoder* d) { return d->hp.ctx_len; }

#if defined(QH_TIMELINE)
extern "C" int qh_timeline_pa_read(uint64_t* host, int n) {
    return hipMemcpyFromSymbol(host, HIP_SYMBOL(qh_tl_pa), sizeof(uint64_t) * (n < 16 ? n : 16)) == hipSuccess ? 0 : 1;
}

extern "C" int qh_timeline_read(uint64_t* host, int n) {
    return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(qh_tl), sizeof(uint64_t) * (size_t)n);
}
extern "C" int qh_timeline_wg_read(uint64_t* host) {
    return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(qh_tl_wg), sizeof(qh_tl_wg));
}
#endif

void decoder_views(Decoder* d, qh_decoder_state* v) {
    v->logits = d->logits;
    v->hidden = d->hidden;
    v->xq = d->qa;
    v->xd = d->da;
    v->stats = d->stats;
    v->top1_full = d->top1_full;
    v->pos = d->pos;
    v->n_out = d->n_out;
    v->token = d->tokens;
    v->kcache = d->kc;
    v->vcache = d->vc;
    v->kcache_f32 = d->kcf;
    v->vcache_f32 = d->vcf;
    v->status = d->status;
    v->history = d->hist;
    v->history_len = d->hist_len;
    v->rng_state = d->rng;
}

int decoder_vocab(const Decoder* d) { return d->hp.vocab_size; }

bool decoder_has_shortlist(const Decoder* d) { return has_shortlist(d); }

int decoder_set_query(Decoder* d, const qh_sampler_params* p) {
    d->has_query = p != nullptr;
    if (p) d->qp = *p;
    return 0;
}

hipError_t decoder_set_sampler(Decoder* d, const qh_sampler_params* p, uint64_t seed) {
    d->has_sampler = p != nullptr;
    if (!p) return hipSuccess;
    d->sp = *p;
    const uint64_t st = seed | 1u;  // Sampler's constructor (sampler.cpp:10-13)
    return hipMemcpy(d->rng, &st, sizeof st, hipMemcpyHostToDevice);
}

}  // namespace qh
