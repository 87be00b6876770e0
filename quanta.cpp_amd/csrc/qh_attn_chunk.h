// Attention of a prefill chunk, one workgroup per (query head, token): qh_decoder.hip's 32-token chunks, and (SINGLE) the
// small stacks of qh_attn_few.hip.
#pragma once

#include "qh_decoder_device.h"

namespace qh {

namespace {

// Attention of token t (position pos0 + t) and query head h over positions [0, pos0 + t], for a chunk of n <= 32
// tokens whose raw projections are q [n][n_heads*HD], k / v [n][n_kv*HD]. One workgroup per (head, token).
// Cache layouts (f16 bits, per layer): K in 16-byte chunks of 8 dimensions, [n_kv][HD/8][ctx][8], so the lanes of a
// wave that read chunk c of 64 consecutive positions read 1 KB of contiguous memory (one row per lane, each lane's
// row complete after HD/8 reads); V in blocks of 8 positions, [pos/8][n_kv*HD][8], so one 16-byte read gives a lane 8
// consecutive positions of its dimension. Rows below pos0 come from the cache; the
// chunk's own rows are rebuilt from k / v (bias, RoPE, f16 rounding, exactly as stored), and workgroups of the first
// query head of each KV group store their token's row. The output (HD values) is quantized straight into oq / od
// ([n][n_heads*HD] codes, one scale per 32 values).
// WPE = 1: a 96 KB V stage, one workgroup per CU (one wave per SIMD, which lets the compiler keep three cached K rows
// per thread in registers). WPE = 2 (prefill chunks at head_dim 64): a 32 KB stage (256 rows) and two cached K rows
// per thread, so two workgroups share a CU (LDS under 80 KB, registers under 256 each) and the 448 workgroups of a
// 14-head chunk run in one round instead of two; their serial chains leave each SIMD mostly idle.
// Timeline stamps of the chunk's last token, query head 0 (compiled in only with -DQH_TIMELINE; the last launch's
// stamps stay in qh_tl_pa, qh_timeline_pa_read copies them out).
#if defined(QH_TIMELINE)
__device__ uint64_t qh_tl_pa[16];
#define QH_PASTAMP(i)                                                                                        \
    do {                                                                                                     \
        if (blockIdx.x == 0 && blockIdx.y == gridDim.y - 1 && threadIdx.x == 0) qh_tl_pa[i] = __builtin_readcyclecounter(); \
    } while (0)
#else
#define QH_PASTAMP(i) \
    do {              \
    } while (0)
#endif
template <int HD, int WPE = 1, bool SINGLE = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void attention_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ bq, const float* __restrict__ bk, const float* __restrict__ bv,
    const float* __restrict__ cs, const int* __restrict__ pos_dev, int ctx, int n_heads, int n_kv,
    uint16_t* __restrict__ kc, uint16_t* __restrict__ vc, int8_t* __restrict__ oq, float* __restrict__ od,
    int* __restrict__ status, float* __restrict__ of) {
    constexpr int HALF = HD / 2, CPR = HD / 8;           // 16-byte chunks per f16 K row
    constexpr int kVRows = (WPE == 1 ? kVStageBytes : 32 * 1024) / (HD * 2);  // V rows one LDS stage holds (mult. of 8)
    constexpr int kVBlk = kVRows / 8;                    // 8-row blocks per stage
    __shared__ __align__(16) float att[kMaxCtx + kChainPad];
    __shared__ __align__(16) uint4 vst[(kVBlk + 4) * HD];  // [block][dim] -> 8 rows; 4 blocks of read padding
    __shared__ __align__(16) uint16_t kloc[kChunk * HD];
    __shared__ __align__(16) uint16_t vloc[kChunk * HD];
    __shared__ __align__(16) float qs[HD];
    __shared__ float red[4];
    __shared__ float sum_sh;
    __shared__ uint64_t exptab[32];
    ExpTab et;
    et.load();
    // SINGLE: every token of a prefill stack is its own chunk (token y = blockIdx.y at position *pos_dev + y), its
    // earlier rows all in the cache already (kv_store_kernel), so the workgroup rebuilds only its own row and stores
    // none.
    const int h = blockIdx.x, y = blockIdx.y, t = SINGLE ? 0 : y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int pos0 = *pos_dev + (SINGLE ? y : 0), pos = pos0 + t, nrows = pos + 1;
    if (pos >= ctx || pos0 < 0) {  // uniform: a step past the context touches no cache row
        if (tid == 0 && h == 0) atomicOr(status, kStatusCtx);
        return;
    }
    const int qd = n_heads * HD, kvd = n_kv * HD, group = n_heads / n_kv, kvh = h / group;
    if (SINGLE) {  // this token's rows of the projections and of the output
        q += (size_t)y * qd;
        k += (size_t)y * kvd;
        v += (size_t)y * kvd;
        oq += (size_t)y * qd;
        od += (size_t)y * (qd / QK);
        if (of) of += (size_t)y * qd;
    }
    QH_PASTAMP(0);
    // V block b of this head: HD uint4 at vbase + b * kvd (in uint4 units, kvd / 8 per position... see vblock())
    const uint4* vc4 = reinterpret_cast<const uint4*>(vc);
    auto vchunk = [&](int blk, int d) { return (size_t)blk * kvd + kvh * HD + d; };  // uint4 index of (block, dim)
    // K chunk (8 dimensions, 16 bytes) c of position p of this KV head, in 16-byte units: [kv head][HD/8][ctx]
    auto kchunk = [&](int c, int p) { return ((size_t)kvh * CPR + c) * ctx + p; };

    // this token's q (this head), k and v (its KV head) rows among the chunk's projections
    const float* qsrc = q + (size_t)t * qd + h * HD;  // row r of k / v: ksrc + r * kvd
    const float* ksrc = k + kvh * HD;
    const float* vsrc = v + kvh * HD;
    const int nk = (t + 1) * HALF, nv = (t + 1) * HD;
    // q of this head with bias, rotated; keys and values of the chunk's tokens 0..t (model.cpp:183-195, rope
    // ops_ref.cpp:201-214: a*c - b*s and b*c + a*s with the reference build's contraction fma(a, c, -(b*s)) and
    // fma(b, c, a*s)). A pair's inputs: the raw values a = row[i], b = row[i + HALF], their biases, cos / sin.
    struct Pair {
        float a, b, ba, bb, c, s;
    };
    auto load_pair = [&](const float* row, const float* bias, int i, const float* crow) {
        Pair pr;
        pr.a = row[i];
        pr.b = row[i + HALF];
        pr.ba = bias ? bias[i] : 0.0f;
        pr.bb = bias ? bias[i + HALF] : 0.0f;
        pr.c = crow[2 * i];
        pr.s = crow[2 * i + 1];
        return pr;
    };
    auto rope = [](const Pair& pr, bool has_bias, float& lo, float& hi) {
        float a = pr.a, b = pr.b;
        if (has_bias) {
            a = a + pr.ba;
            b = b + pr.bb;
        }
        lo = __builtin_fmaf(a, pr.c, -(b * pr.s));
        hi = __builtin_fmaf(b, pr.c, a * pr.s);
    };
    const float* bqh = bq ? bq + h * HD : nullptr;
    const float* bkh = bk ? bk + kvh * HD : nullptr;
    // Every element this thread rebuilds is loaded before any is used (indices clamped, so every load is
    // unconditional and the loads are one round trip): K pair elements tid + 256 i and V elements tid + 256 i of the
    // chunk's rows 0..t. 256 is a multiple of HD, so a thread's elements share their dimension, and its biases.
    static_assert(256 % HD == 0, "a thread's rebuilt elements share one dimension");
    constexpr int KPT = kChunk * HALF / 256, VPT = kChunk * HD / 256;  // elements per thread at n = kChunk
    const int tq = min(tid, HALF - 1);
    const Pair qp = load_pair(qsrc, bqh, tq, cs + (size_t)pos * HD);
    const int ik = tid % HALF, iv = tid % HD;
    const float kba = bkh ? bkh[ik] : 0.0f, kbb = bkh ? bkh[ik + HALF] : 0.0f;
    const float vb = bv ? bv[kvh * HD + iv] : 0.0f;
    float ka[KPT], kb[KPT], vv[VPT];
    float2 kcs[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        const int rk = min(tid + 256 * i, nk - 1) / HALF;
        const float* row = ksrc + (size_t)rk * kvd;
        ka[i] = row[ik];
        kb[i] = row[ik + HALF];
        kcs[i] = *reinterpret_cast<const float2*>(cs + (size_t)(pos0 + rk) * HD + 2 * ik);
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) vv[i] = vsrc[(size_t)(min(tid + 256 * i, nv - 1) / HD) * kvd + iv];
    __builtin_amdgcn_sched_barrier(0);

    // This thread's cached K rows for the first score rows (registers) go out behind those (a load waits for every
    // load issued before it), and their issue, which stalls while the memory pipeline drains, covers the q / k / v
    // latency. No row read here is written by this launch: K rows stop below pos0.
    constexpr int kKPre = WPE == 1 ? 3 : 2;  // score rows per thread loaded up front (768 / 512 positions)
    const int grow = pos0 > 0 ? pos0 - 1 : 0;
    v4u kpre[kKPre][CPR];
#pragma unroll
    for (int r = 0; r < kKPre; ++r) {
        const uint16_t* kg = kc + (kchunk(0, min(tid + 256 * r, grow)) << 3);
#pragma unroll
        for (int i = 0; i < CPR; ++i) kpre[r][i] = ld4(kg + (size_t)i * ctx * 8);
    }
    if (tid < HALF) rope(qp, bq != nullptr, qs[tid], qs[tid + HALF]);
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        const int e = tid + 256 * i;
        if (e < nk) {
            const int r = e / HALF;
            float lo, hi;
            rope(Pair{ka[i], kb[i], kba, kbb, kcs[i].x, kcs[i].y}, bk != nullptr, lo, hi);
            kloc[r * HD + ik] = f2h(lo);
            kloc[r * HD + ik + HALF] = f2h(hi);
        }
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int e = tid + 256 * i;
        if (e < nv) vloc[(e / HD) * HD + iv] = f2h(bv ? vv[i] + vb : vv[i]);
    }
    et.store(exptab);
    __syncthreads();
    QH_PASTAMP(1);
    if (!SINGLE && h % group == 0)
        for (int i = tid; i < HD; i += 256) {
            kc[(kchunk(i >> 3, pos) << 3) + (i & 7)] = kloc[t * HD + i];
            vc[vchunk(pos / 8, i) * 8 + (pos & 7)] = vloc[t * HD + i];
        }

    // scores: s = sum_i q_i * k_i as one FMA per element in order, then * scale (model.cpp:122-125)
    float qv[HD];
#pragma unroll
    for (int i = 0; i < HD; ++i) qv[i] = qs[i];
    const float scale = 1.0f / __builtin_sqrtf((float)HD);
    float mx = -__builtin_inff();
    // one dot product: s = fma(q_i, k_i, s) in dimension order
    auto dot_row = [&](const v4u(&kk)[CPR]) {
        float sc = 0.0f;
#pragma unroll
        for (int i = 0; i < CPR; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sc = __builtin_fmaf(qv[i * 8 + 2 * e], h2f((uint16_t)(kk[i][e] & 0xffffu)), sc);
                sc = __builtin_fmaf(qv[i * 8 + 2 * e + 1], h2f((uint16_t)(kk[i][e] >> 16)), sc);
            }
        }
        return sc;
    };
    // the chunk's own rows j >= pos0 (keys in LDS)
    for (int j = pos0 + tid; j < nrows; j += 256) {
        v4u kk[CPR];
        const uint16_t* kl = kloc + (j - pos0) * HD;
#pragma unroll
        for (int i = 0; i < CPR; ++i) kk[i] = ld4(kl + i * 8);
        const float a = dot_row(kk) * scale;
        att[j] = a;
        mx = a > mx ? a : mx;
    }
    // The first stage's V blocks go straight into LDS (DMA, no registers), in two halves of the whole stage per wave
    // (clamped onto the last block, whose repeats write the same data): the first once the scores are done and the
    // second after the exp row (the issue of a half stalls its wave while the memory pipeline drains, so neither
    // holds up the scores, and the second is issued after the wait that completes the first). Everything is waited
    // for before the stage is built. Cache blocks stop below pos0: none is written by
    // this launch (the block holding pos0 carries stale rows from pos0 on, replaced when the stage is built).
    const int ncb = min((pos0 + 7) / 8, kVBlk);  // cache blocks of the first stage (the last may be partial)
    constexpr int kDmaPerBlk = HD / 64;          // 1 KB (one wave instruction) per DMA chunk
    constexpr int kVEarly = kVBlk * kDmaPerBlk / 4;  // DMA chunks per wave
    auto dma_v = [&](int e0, int e1) {           // chunks wave + 4 e, e in [e0, e1)
        const int last = max(ncb * kDmaPerBlk - 1, 0);
#pragma unroll
        for (int e = e0; e < e1; ++e) {
            const int c = min(wave + 4 * e, last);
            lds_dma16_async(vc4 + vchunk(c / kDmaPerBlk, (c % kDmaPerBlk) * 64 + lane), vst + c * 64);
        }
    };

    // the cached rows tid + 256 r (registers only), their chains interleaved; stored after the barrier below
    float sc[kKPre];
    {
#pragma unroll
        for (int r = 0; r < kKPre; ++r)  // uniform: no thread has a cached row tid + 256 r at or past pos0
            sc[r] = 256 * r < pos0 ? dot_row(kpre[r]) * scale : 0.0f;
#pragma unroll
        for (int r = 0; r < kKPre; ++r) {
            const int j = tid + 256 * r;
            if (j < pos0) mx = sc[r] > mx ? sc[r] : mx;
        }
    }
    for (int j = tid + 256 * kKPre; j < pos0; j += 256) {  // longer contexts: one row at a time
        v4u kk[CPR];
        const uint16_t* kg = kc + (kchunk(0, j) << 3);
#pragma unroll
        for (int i = 0; i < CPR; ++i) kk[i] = ld4(kg + (size_t)i * ctx * 8);
        const float a = dot_row(kk) * scale;
        att[j] = a;
        mx = a > mx ? a : mx;
    }
    // the maximum does not depend on the order of comparison
    QH_PASTAMP(2);
    mx = wave_max_sel(mx);
    if (lane == 0) red[wave] = mx;
    dma_v(0, kVEarly / 2);
#pragma unroll
    for (int r = 0; r < kKPre; ++r) {
        const int j = tid + 256 * r;
        if (j < pos0) att[j] = sc[r];
    }
    __syncthreads();
    mx = red[0];
    for (int w = 1; w < 4; ++w) mx = red[w] > mx ? red[w] : mx;
    QH_PASTAMP(3);
    // exp, kept in LDS, with each lane's exact partial sums below the segment starts
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
    QH_PASTAMP(4);
    __shared__ SegShared ssh;
    if (seg) seg_partials(ssh, p1, p2, p3);
    __builtin_amdgcn_s_waitcnt(0);  // the first half of the V DMA
    dma_v(kVEarly / 2, kVEarly);
    __syncthreads();
    // softmax sum in position order (ops_ref.cpp:220-224)
    auto add = [](float acc, float a) { return acc + a; };
    float sum;
    if (seg) {
        // segments read as LDS broadcasts (through scalar loads of a global copy written just before, the sum of
        // 512 positions took 2.3 us against 1.4 us)
        sum = seg_chain_run(ssh, [&](int k, float s0) { return lds_chain(att + sg.start(k), sg.len(k), add, s0); });
    } else {
        __syncthreads();
        if (tid == 0) sum_sh = lds_chain(att, nrows, add);
        __syncthreads();
        sum = sum_sh;
    }
    QH_PASTAMP(5);
    const float inv = 1.0f / sum;
    for (int j = tid; j < nrows; j += 256) {
        att[j] = att[j] * inv;
    }
    // the V DMA is complete before the barrier; then the chunk's rows that fall inside
    // the first stage are written over the DMA's blocks
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    uint16_t* vst16 = reinterpret_cast<uint16_t*>(vst);
    {
        const int s1 = min(nrows, kVRows);
        for (int e = tid; e < (s1 - pos0) * HD; e += 256) {  // empty when pos0 >= kVRows
            const int r = pos0 + e / HD, d = e % HD;
            vst16[((r >> 3) * HD + d) * 8 + (r & 7)] = vloc[(r - pos0) * HD + d];
        }
        __syncthreads();
    }
    QH_PASTAMP(6);

    // out_i = sum_j a_j * v_ji, one FMA per position in order (model.cpp:131-135): thread i per dimension, over
    // the rows of each LDS stage. The weights are broadcast LDS reads of att (every lane the same address), so a
    // batch of 32 positions is 4 V reads, 8 weight reads and 32 FMAs, the next batch's reads in flight while one is
    // consumed. (With scalar operands from a global copy of the weights, written just before, the first stage's
    // chain ran 1.4x slower at two workgroups per CU.) V reads past the stage stay inside its padding, weight reads
    // inside att's padding.
    // Past the first stage, the threads without a dimension load the next stage's cache blocks into registers while
    // the chain runs (kPreload: at most 12 16-byte units each), so only LDS stores stand between two stages.
    constexpr int kLoaders = 256 - HD, kPre = (kVBlk * HD + kLoaders - 1) / kLoaders;
    constexpr bool kPreload = kPre <= 12;
    uint4 nxt[kPreload ? kPre : 1];
    float acc = 0.0f;
    for (int s0 = 0;;) {
        const int se = min(nrows, s0 + kVRows);
        if (kPreload && tid >= HD && se < nrows) {  // uniform per wave; pos0 >= 1 here (a second stage)
            const int nb8 = (min(nrows, se + kVRows) - se + 7) / 8, lastc = (pos0 - 1) / 8;
#pragma unroll
            for (int u = 0; u < kPre; ++u) {
                const int c = tid - HD + kLoaders * u, blk = se / 8 + c / HD, d = c % HD;
                const uint4 x = vc4[vchunk(min(blk, lastc), d)];
                nxt[u] = c < nb8 * HD && blk * 8 < pos0 ? x : make_uint4(0u, 0u, 0u, 0u);
            }
        }
        if (tid < HD) {
            // The weights are LDS broadcast reads of att (one 16-byte read gives every lane 4 weights), a batch
            // ahead of the chain.
            const float4* ap = reinterpret_cast<const float4*>(att + s0);  // s0 is a multiple of 32
            auto ldv = [&](uint4(&vv)[4], float4(&w)[8], int jr) {  // rows s0 + jr .. + 31 (jr % 32 == 0)
                const uint4* vp = vst + (jr >> 3) * HD + tid;
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) vv[q4] = vp[q4 * HD];
#pragma unroll
                for (int q = 0; q < 8; ++q) w[q] = ap[jr / 4 + q];
            };
            auto use = [&](const uint4(&vv)[4], const float4(&w)[8], int cnt) {
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    const uint32_t v[4] = {vv[q4].x, vv[q4].y, vv[q4].z, vv[q4].w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int k = 8 * q4 + e;
                        const float4 wq = w[k >> 2];
                        const float wk = (k & 3) == 0 ? wq.x : (k & 3) == 1 ? wq.y : (k & 3) == 2 ? wq.z : wq.w;
                        if (k < cnt)
                            acc = __builtin_fmaf(wk, h2f((uint16_t)(e & 1 ? v[e >> 1] >> 16 : v[e >> 1] & 0xffffu)),
                                                 acc);
                    }
                }
            };
            const int n = se - s0;
            uint4 vA[4], vB[4];
            float4 wA[8], wB[8];
            // sched_barrier keeps each batch's reads ahead of the chain steps they overlap (the scheduler would sink
            // them next to their first use)
            ldv(vA, wA, 0);
            int jr = 0;
#pragma unroll 1
            for (; jr + 64 <= n; jr += 64) {
                ldv(vB, wB, jr + 32);
                __builtin_amdgcn_sched_barrier(0);
                use(vA, wA, 32);
                ldv(vA, wA, jr + 64);
                __builtin_amdgcn_sched_barrier(0);
                use(vB, wB, 32);
            }
            if (jr + 32 <= n) {
                ldv(vB, wB, jr + 32);
                __builtin_amdgcn_sched_barrier(0);
                use(vA, wA, 32);
                use(vB, wB, n - jr - 32);
            } else {
                use(vA, wA, n - jr);
            }
        }
        s0 = se;
        if (s0 >= nrows) break;
        __syncthreads();  // the stage is consumed; load rows [s0, min(nrows, s0 + kVRows)) (s0 % 8 == 0)
        const int sn = min(nrows, s0 + kVRows);
        const int nb8 = (sn - s0 + 7) / 8;
        if constexpr (kPreload) {
            if (tid >= HD) {
#pragma unroll
                for (int u = 0; u < kPre; ++u) {
                    const int c = tid - HD + kLoaders * u;
                    if (c < nb8 * HD) vst[c] = nxt[u];
                }
            }
        } else {
            for (int c = tid; c < nb8 * HD; c += 256) {  // whole cache blocks; the chunk's rows are written after
                const int blk = s0 / 8 + c / HD, d = c % HD;
                vst[c] = blk * 8 < pos0 ? vc4[vchunk(blk, d)] : make_uint4(0u, 0u, 0u, 0u);
            }
        }
        __syncthreads();
        for (int e = tid; e < (sn - max(s0, pos0)) * HD; e += 256) {
            const int r = max(s0, pos0) + e / HD, d = e % HD;
            vst16[(((r - s0) >> 3) * HD + d) * 8 + (r & 7)] = vloc[(r - pos0) * HD + d];
        }
        __syncthreads();
    }
    QH_PASTAMP(7);
    if (tid < HD) {  // quantize_q8 of the attention output, two 32-blocks per 64 dimensions
        const int col = h * HD + (tid & ~31);
        if (of) of[(size_t)t * qd + h * HD + tid] = acc;  // the f32 input of an unquantized o projection
        quant_block32(acc, oq + (size_t)t * qd + col, od + (size_t)t * (qd / QK) + col / QK);
    }
}

}  // namespace

}  // namespace qh
