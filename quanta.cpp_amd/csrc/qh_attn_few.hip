// Attention of a prefill stack of few workgroups, its cache rows stored (kv_store_kernel): one workgroup per query head and
// four tokens up to kStackCtx rows at head_dim 64, else one per query head and token. In a code object of its own: three
// kernels more in the decoder's made a decode step slower though its kernels' code was the same (24 layers at position
// 512 by 0.5%; two layers at 3,500, with the first of them in front of the step's kernels, 1,891 -> 1,915 us for 16).
#include "qh_attn_chunk.h"
#include "qh_decoder_device.h"
#include "qh_device.h"
#include "qh_internal.h"

namespace qh {

namespace {

// Attention of a prefill stack at head_dim 64 with kStackTok consecutive tokens of one query head per workgroup, once
// kv_store_kernel has stored every row of the stack, so the workgroup rebuilds nothing and its tokens share the K and
// V rows it reads: positions *pos_dev + y0 .. + kStackTok - 1 (y0 = kStackTok * blockIdx.y, tokens below n), all
// below kStackCtx. The same arithmetic and order as attention_kernel for each token (model.cpp:115-137,
// ops_ref.cpp:216-226): q with bias and RoPE in f32; wave i takes token i: its q as 64 scalar operands, lane l
// scores cached rows l, l + 64, ... up to the token's row count (s = fma(q_i, k_i, s) in dimension order, the f16 key
// as a mixed-precision operand, then * 1/sqrt(64)), the next row's key loaded while a row is scored; the maximum over
// the wave; glibc expf; the softmax sum in position order, its normalisation, and the weighted V chain over V rows
// staged in LDS (lane d for dimension d, the weights as LDS broadcast reads), the four tokens' chains on four SIMDs
// at once. The V stages' loads are issued a stage ahead (the first at the start), so their latency hides under the
// scores and the previous stage's chains. The output is quantized per 32-block. Its LDS holds two workgroups per CU,
// so the register budget is that of two waves per SIMD.
template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void attention_stack_kernel(
    const float* __restrict__ q, const float* __restrict__ bq, const float* __restrict__ cs,
    const int* __restrict__ pos_dev, int n, int ctx, int n_heads, int n_kv, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, int8_t* __restrict__ oq, float* __restrict__ od, int* __restrict__ status,
    float* __restrict__ of) {
    static_assert(HD == 64, "a lane per dimension");
    constexpr int HALF = HD / 2, CPR = HD / 8, NTK = kStackTok;
    constexpr int kVRows = 256, kVBlk = kVRows / 8;  // V rows per LDS stage (32 KB)
    constexpr int kVPer = kVBlk * HD / 256;          // 16-byte V units per thread and stage
    __shared__ __align__(16) float att[NTK][kStackCtx + kChainPad];
    __shared__ __align__(16) uint4 vst[(kVBlk + 4) * HD];  // [block][dim] -> 8 rows; 4 blocks of read padding
    __shared__ __align__(16) float qs[NTK][HD];
    __shared__ uint64_t exptab[32];
    ExpTab et;
    et.load();
    // groups in reverse order: the longest (the stack's last tokens) are dispatched first, the short ones fill in
    const int h = blockIdx.x, y0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * NTK, tid = threadIdx.x, lane = tid & 63,
              wave = tid >> 6;
    const int nt = min(NTK, n - y0);  // tokens of this workgroup (uniform)
    const int base = *pos_dev + y0;   // position of token 0
    const int nmax = base + nt;       // rows of the last token
    if (base < 0 || nmax > ctx || nmax > kStackCtx) {  // uniform; the host launches this only within both limits
        if (tid == 0) atomicOr(status, kStatusCtx);
        return;
    }
    const int qd = n_heads * HD, kvd = n_kv * HD, group = n_heads / n_kv, kvh = h / group;
    auto kchunk = [&](int c, int p) { return ((size_t)kvh * CPR + c) * ctx + p; };
    auto vchunk = [&](int blk, int d) { return (size_t)blk * kvd + kvh * HD + d; };
    const uint4* vc4 = reinterpret_cast<const uint4*>(vc);
    // V units of the stage at s0 (whole cache blocks of 8 positions below nmax) into registers, then into vst
    v4u vreg[kVPer];
    auto vload = [&](int s0) {  // units past the stage's blocks: re-reads, never stored
        const int nb8 = (min(nmax, s0 + kVRows) - s0 + 7) / 8;
#pragma unroll
        for (int k = 0; k < kVPer; ++k) {
            const int c = min(tid + 256 * k, nb8 * HD - 1);
            vreg[k] = ld4(vc4 + vchunk(s0 / 8 + c / HD, c % HD));
        }
    };
    auto vput = [&]() {  // the whole stage area (rows past the stage: never read)
#pragma unroll
        for (int k = 0; k < kVPer; ++k) *reinterpret_cast<v4u*>(&vst[tid + 256 * k]) = vreg[k];
    };
    vload(0);
    // q of token `wave` (lanes 0-31: one rotated pair each), with bias (model.cpp:183-195, ops_ref.cpp:201-214)
    if (wave < nt && lane < HALF) {
        const float* src = q + (size_t)(y0 + wave) * qd + h * HD;
        const float* crow = cs + (size_t)(base + wave) * HD;
        float a = src[lane], b = src[lane + HALF];
        if (bq) {
            a = a + bq[h * HD + lane];
            b = b + bq[h * HD + lane + HALF];
        }
        const float c = crow[2 * lane], sn = crow[2 * lane + 1];
        qs[wave][lane] = __builtin_fmaf(a, c, -(b * sn));
        qs[wave][lane + HALF] = __builtin_fmaf(b, c, a * sn);
    }
    et.store(exptab);
    __syncthreads();

    // wave tk: token tk's scores, maximum, exponentials, softmax sum in position order (ops_ref.cpp:220-224) and
    // normalisation, all within the wave (its rows of att are its own)
    const int tk = wave, nrows = base + tk + 1;
    if (tk < nt) {
        const float scale = 1.0f / __builtin_sqrtf((float)HD);
        const float qv = qs[tk][lane];
        float qsg[HD];  // q_i, wave-uniform
#pragma unroll
        for (int d = 0; d < HD; ++d) qsg[d] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, qv), d));
        float mx = -__builtin_inff();
        v4u kA[CPR], kB[CPR];
        auto kload = [&](v4u(&kk)[CPR], int j) {  // row j's key, clamped to the token's last row
            const uint16_t* kg = kc + (kchunk(0, min(j, nrows - 1)) << 3);
#pragma unroll
            for (int c = 0; c < CPR; ++c) kk[c] = ld4(kg + (size_t)c * ctx * 8);
        };
        auto score = [&](const v4u(&kk)[CPR], int j) {
            float sc = 0.0f;
#pragma unroll
            for (int c = 0; c < CPR; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sc = __builtin_fmaf(qsg[8 * c + 2 * e], h2f((uint16_t)(kk[c][e] & 0xffffu)), sc);
                    sc = __builtin_fmaf(qsg[8 * c + 2 * e + 1], h2f((uint16_t)(kk[c][e] >> 16)), sc);
                }
            if (j < nrows) {
                const float a = sc * scale;
                att[tk][j] = a;
                mx = a > mx ? a : mx;
            }
        };
        kload(kA, lane);
        int j0 = 0;
        for (; j0 + 64 < nrows; j0 += 128) {
            kload(kB, j0 + 64 + lane);
            score(kA, j0 + lane);
            kload(kA, j0 + 128 + lane);
            score(kB, j0 + 64 + lane);
        }
        if (j0 < nrows) score(kA, j0 + lane);
        mx = wave_max_sel(mx);  // the maximum does not depend on the order of comparison
        __builtin_amdgcn_wave_barrier();
        for (int j = lane; j < nrows; j += 64) att[tk][j] = dev_expf(att[tk][j] - mx, exptab);
        __builtin_amdgcn_wave_barrier();
        const float sum = lds_chain(att[tk], nrows, [](float acc, float a) { return acc + a; });
        const float inv = 1.0f / sum;
        for (int j = lane; j < nrows; j += 64) att[tk][j] = att[tk][j] * inv;
    }
    // out_i = sum_j a_j * v_ji, one FMA per position in order (model.cpp:131-135): wave i, lane d, over the rows of
    // each V stage (whole cache blocks of 8 positions; rows past a token's count are never used)
    float acc = 0.0f;
    for (int s0 = 0; s0 < nmax; s0 += kVRows) {
        const int sn = min(nmax, s0 + kVRows);
        __syncthreads();  // the previous stage is consumed (and, for the first, the normalised rows are written)
        vput();
        if (s0 + kVRows < nmax) vload(s0 + kVRows);  // the next stage's loads run under this stage's chains
        __syncthreads();
        if (tk < nt && s0 < nrows) {
            const int n_ = min(nrows, sn) - s0;
            const float4* ap = reinterpret_cast<const float4*>(lane_ptr(att[tk] + s0));  // s0 % 32 == 0
            auto ldv = [&](uint4(&vv)[4], float4(&w)[8], int jr) {  // rows s0 + jr .. + 31 (jr % 32 == 0)
                const uint4* vp = vst + (jr >> 3) * HD + lane;
#pragma unroll
                for (int q4i = 0; q4i < 4; ++q4i) vv[q4i] = vp[q4i * HD];
#pragma unroll
                for (int qi = 0; qi < 8; ++qi) w[qi] = ap[jr / 4 + qi];
            };
            auto use = [&](const uint4(&vv)[4], const float4(&w)[8], int cnt) {
#pragma unroll
                for (int q4i = 0; q4i < 4; ++q4i) {
                    const uint32_t vw[4] = {vv[q4i].x, vv[q4i].y, vv[q4i].z, vv[q4i].w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int kx = 8 * q4i + e;
                        const float4 wq = w[kx >> 2];
                        const float wk = (kx & 3) == 0 ? wq.x : (kx & 3) == 1 ? wq.y : (kx & 3) == 2 ? wq.z : wq.w;
                        if (kx < cnt)
                            acc = __builtin_fmaf(wk, h2f((uint16_t)(e & 1 ? vw[e >> 1] >> 16 : vw[e >> 1] & 0xffffu)),
                                                 acc);
                    }
                }
            };
            uint4 vA[4], vB[4];
            float4 wA[8], wB[8];
            ldv(vA, wA, 0);
            int jr = 0;
#pragma unroll 1
            for (; jr + 64 <= n_; jr += 64) {
                ldv(vB, wB, jr + 32);
                __builtin_amdgcn_sched_barrier(0);
                use(vA, wA, 32);
                ldv(vA, wA, jr + 64);
                __builtin_amdgcn_sched_barrier(0);
                use(vB, wB, 32);
            }
            if (jr + 32 <= n_) {
                ldv(vB, wB, jr + 32);
                __builtin_amdgcn_sched_barrier(0);
                use(vA, wA, 32);
                use(vB, wB, n_ - jr - 32);
            } else {
                use(vA, wA, n_ - jr);
            }
        }
    }
    if (tk < nt) {  // quantize_q8 of the output, two 32-blocks per 64 dimensions
        const size_t row = (size_t)(y0 + tk) * qd;
        const int col = h * HD + (lane & ~31);
        if (of) of[row + h * HD + lane] = acc;
        quant_block32(acc, oq + row + col, od + row / QK + col / QK);
    }
}

}  // namespace

hipError_t launch_attention_few(const AttnFew& a, int head_dim, int rows, hipStream_t s) {
    const dim3 grid(a.n_heads, a.n);
    if (head_dim == 64 && rows <= kStackCtx)
        qh_launch((attention_stack_kernel<64>), dim3(a.n_heads, (a.n + kStackTok - 1) / kStackTok), dim3(256), 0, s, a.q,
                  a.bq, a.cs, a.pos, a.n, a.ctx, a.n_heads, a.n_kv, a.kc, a.vc, a.oq, a.od, a.status, a.of);
    else if (head_dim == 64)
        qh_launch((attention_kernel<64, 2, true>), grid, dim3(256), 0, s, a.q, a.k, a.v, a.bq, a.bk, a.bv, a.cs, a.pos,
                  a.ctx, a.n_heads, a.n_kv, a.kc, a.vc, a.oq, a.od, a.status, a.of);
    else
        qh_launch((attention_kernel<128, 1, true>), grid, dim3(256), 0, s, a.q, a.k, a.v, a.bq, a.bk, a.bv, a.cs, a.pos,
                  a.ctx, a.n_heads, a.n_kv, a.kc, a.vc, a.oq, a.od, a.status, a.of);
    return hipGetLastError();
}

}  // namespace qh
