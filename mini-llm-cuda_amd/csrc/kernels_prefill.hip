// Prefill: many tokens of one or more sequences through the stack at once.
//
// Rows of the activation matrices are tokens (all segments concatenated); the projections are MFMA
// GEMMs (kernels_gemm.hip, kernels_tile.hip) against copies of the weights as halves or planes, or, in short calls, the row
// kernels of the decode step (kernels_rows.hip); per layer
//
//   rmsnorm rows -> GEMM Wa -> attention: per-head QK-norm + RoPE + KV-page write, tiled causal attention
//                              GDN:       chunked recurrence, one head of one sequence per workgroup
//                -> (PLE rows) -> GEMM Wo (+ residual) (+ GEMM pleUp accumulate)
//                -> rmsnorm rows -> GEMM W13 with SiLU(gate)*up epilogue -> GEMM W2 (+ residual)
//
// and at the end the LM head runs for the last row of every segment only (the reference computes
// logits for all L columns, inference.cu:723-743, and uses the last one).  With bf16 weights the GEMM
// inputs (normed activations, mixing output, FFN activations) are rounded to half; with fp32 weights they are
// stored as two halves, the weights as three (h2.h), or, where a model's weights spread further than halves reach
// (operand_spread), both as three bf16 planes that add up to the fp32 value (p3.h).  Accumulation, the
// residual stream, K/V and GDN states stay fp32.  This is what runInference(L) (inference.cu:376-751)
// does for L columns, minus the columns that are already in the cache.
#include <math.h>
#include <string.h>

#include <algorithm>

#include "h2.h"
#include "mlh_internal.h"
#include "p3.h"
#include "persist_common.h"
#include "sample.h"

#define PWG 256
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct PfArgs {
    StepArgs a;        // model dimensions and shared pointers (rope, page table, E, gains ...)
    int n;             // rows (tokens) in this call
    int nseg;
    const int* ids;    // [n]
    const int* rowSeq; // [n] sequence of the row
    const int* rowPos; // [n] position of the row's token in its sequence
    const int* segStart;
    const int* segLen;
    const int* segSeq;
    const int* segPos0;
    const int* blkSeg; // attention query blocks: segment and first query of the block
    const int* blkQ0;
    float* X;          // [n, dim] residual stream
    void* Xn;          // [n, dim] GEMM input (fp32 models: pairs of halves, h2.h, or planes, p3.h; else halves); planes: that of the output projection too, [n, aLd]
    int* exps;         // exponents of pairs' rows
    float* QKV;        // [n, qkvLd]
    int qkvLd;
    void* Amix;        // [n, aLd] GEMM input of the output projection: mixing output, then (at column L.ad) the PLE row (fp32 models: floats, then pairs in place)
    int aLd;
    float* H1;         // [n, dim]
    void* U;           // [n, ffn]
    uint16_t* Kh;      // [n, dim] IEEE-half copies of this call's K and V rows (after norm and RoPE), or null: what the MFMA
    uint16_t* Vh;      //          attention reads when every segment starts at position 0 (all of its keys are rows of the call)
    unsigned char* rows; // short calls: the mixing output goes into the planes of the row products (rows.h) instead of Amix
    RowsLayout lay;
    int half;            // bf16 weights
};

__device__ __forceinline__ float pf_wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float pf_wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int pf_wave_max(int v) { return (int)pwave_max((float)v); } // (exponents: exact)
__device__ __forceinline__ float pf_sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); } // inference.cu:248
__device__ __forceinline__ float pf_silu(float v) { return v / (1.0f + expf(-v)); }       // inference.cu:270

// store a float as the GEMM input type (IEEE half for bf16 models, whose MFMA path runs in fp16)
template <typename AT> __device__ __forceinline__ void put(AT* p, float v);
template <> __device__ __forceinline__ void put<f16_t>(f16_t* p, float v) {
    const _Float16 h = (_Float16)half_range(v);
    p->bits = __builtin_bit_cast(uint16_t, h);
}
template <> __device__ __forceinline__ void put<float>(float* p, float v) { *p = v; }
// element `col` of row `row` of a GEMM input matrix (leading dimension ld in elements)
template <typename AT> __device__ __forceinline__ void put_at(void* base, size_t row, int ld, int col, float v) { put<AT>((AT*)base + row * ld + col, v); }
// element `col` of a token's mixing output (behind it: its PLE columns)
template <typename AT> __device__ __forceinline__ void put_mix(const PfArgs& P, size_t row, int col, float v) {
    if (P.rows) rows_put(P.rows, col, (int)row, P.lay, P.half != 0, v);
    else put_at<AT>(P.Amix, row, P.aLd, col, v);
}
template <typename WT> __device__ __forceinline__ float getw(const WT* p);
template <> __device__ __forceinline__ float getw<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float getw<bf16_t>(const bf16_t* p) { return __uint_as_float(((uint32_t)*p) << 16); }

// inference.cu:9-22
template <typename WT>
__global__ void k_pf_embed(PfArgs P) {
    const int row = blockIdx.y, i = blockIdx.x * PWG + threadIdx.x;
    if (i >= P.a.dim) return;
    P.X[(size_t)row * P.a.dim + i] = getw<WT>((const WT*)P.a.E + (size_t)P.ids[row] * P.a.dim + i);
}

// inference.cu:24-50 + 83-95, one wave per row (d is a multiple of 8 on this path: 16-byte loads).  Rows of up to
// 4096 elements stay in registers between the sum of squares and the scaling (one pass over memory), and a lane's
// four results leave as one store.
template <typename AT> __device__ __forceinline__ void put4(AT* o, float a, float b, float c, float d);
template <> __device__ __forceinline__ void put4<f16_t>(f16_t* o, float a, float b, float c, float d) {
    *reinterpret_cast<uint2*>(o) = make_uint2(pack_half_range(a, b), pack_half_range(c, d));
}

template <> __device__ __forceinline__ void put4<float>(float* o, float a, float b, float c, float d) { *reinterpret_cast<f32x4*>(o) = f32x4{a, b, c, d}; }

template <typename AT> __device__ __forceinline__ void put4_at(void* base, size_t row, int ld, int col, float a, float b, float c, float d) { put4<AT>((AT*)base + row * ld + col, a, b, c, d); }
template <> __device__ __forceinline__ void put4_at<p3_t>(void* base, size_t row, int ld, int col, float a, float b, float c, float d) { p3_put4((unsigned char*)base + row * ld * 6, col, a, b, c, d); }
// Four columns of the mixing output.
template <typename AT> __device__ __forceinline__ void put_mix4(const PfArgs& P, size_t row, int col, const f32x4& v) {
    if (P.rows) rows_put4(P.rows, col, (int)row, P.lay, P.half != 0, v.x, v.y, v.z, v.w);
    else put4_at<AT>(P.Amix, row, P.aLd, col, v.x, v.y, v.z, v.w);
}

// PLE columns of `rows` rows from row0 on, e[row][j] = silu(ple gate output) * P[tok][j], behind the mixing output (fp32 models' calls of more rows than the row
// kernels take: k_pf_operand_rows).  Workgroups of their own in the launches that mix: a launch for them took 4.4 us a layer, whatever it did.  24 bf16 layers of width
// 2048, us: 17 rows 1945 -> 1884, 70 2094 -> 2019, 300 3081 -> 3006, 777 4512 -> 4442; 16 384 rows the same.
// AT_ONCE: elements of a thread on their way together; one after the other a chunk of 64 rows x 128 columns was a chain of 32 latencies, and what a
// launch of few chunks ended with (8 bf16 layers of width 1024, us: 64 rows 588 -> 538, 600 820 -> 749, 1500 1340 -> 1262, 8 prompts of 1160 rows 1126 -> 1047).
template <int AT_ONCE, typename WT, typename AT> __device__ __forceinline__ void ple_columns(const PfArgs& P, const LayerDev& L, int row0, int rows, int tid, int threads) {
    const int ple = P.a.ple, total = rows * ple;
    for (int i0 = tid; i0 < total; i0 += AT_ONCE * threads) {
        float gate[AT_ONCE], emb[AT_ONCE];
#pragma unroll
        for (int k = 0; k < AT_ONCE; k++) {
            const int i = min(i0 + k * threads, total - 1), r = i / ple, j = i - r * ple;
            const size_t row = (size_t)row0 + r;
            gate[k] = P.QKV[row * P.qkvLd + L.offPle + j];
            emb[k] = getw<WT>((const WT*)L.pleTable + (size_t)P.ids[row] * ple + j);
        }
#pragma unroll
        for (int k = 0; k < AT_ONCE; k++) {
            const int i = i0 + k * threads, r = i / ple, j = i - r * ple;
            if (i < total) put_mix<AT>(P, (size_t)row0 + r, L.ad + j, pf_silu(gate[k]) * emb[k]);
        }
    }
}
template <int AT_ONCE> __device__ __forceinline__ void ple_columns(const PfArgs& P, const LayerDev& L, int row0, int rows, int tid, int threads) {
    if (P.half) ple_columns<AT_ONCE, bf16_t, f16_t>(P, L, row0, rows, tid, threads);
    else ple_columns<AT_ONCE, float, float>(P, L, row0, rows, tid, threads);
}

// KEEP: 16-byte pieces a lane keeps, rows of up to 256 KEEP elements.  All loads of a row and of the gains go out at once: a load under a comparison, or the
// gains asked for behind the sum, each add a memory latency.  Measured: 777 rows of 2048 5.4 us (6.3), 517 rows of 768 5.0 us (4.9); 16384 rows of
// 2048 32 us (37), 6.2 TB/s: part of it comes out of the caches.
template <typename AT, int KEEP>
__global__ void __launch_bounds__(PWG) k_pf_rmsnorm(const float* __restrict__ X, const float* __restrict__ gamma, void* out, int* exps, int n, int d) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= n) return;
    const float* x = X + (size_t)row * d;
    f32x4 keep[KEEP], gain[KEEP];
#pragma unroll
    for (int k = 0; k < KEEP; k++) keep[k] = *reinterpret_cast<const f32x4*>(x + min(lane * 4 + k * 256, d - 4));
#pragma unroll
    for (int k = 0; k < KEEP; k++) gain[k] = *reinterpret_cast<const f32x4*>(gamma + min(lane * 4 + k * 256, d - 4));
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < KEEP; k++) {
        const f32x4 v = lane * 4 + k * 256 < d ? keep[k] : (f32x4)(0.f);
        s = fmaf(v.x, v.x, s); s = fmaf(v.y, v.y, s); s = fmaf(v.z, v.z, s); s = fmaf(v.w, v.w, s);
    }
    for (int i = lane * 4 + KEEP * 256; i < d; i += 256) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(x + i);
        s = fmaf(v.x, v.x, s); s = fmaf(v.y, v.y, s); s = fmaf(v.z, v.z, s); s = fmaf(v.w, v.w, s);
    }
    s = pf_wave_sum(s);
    const float r = sqrtf(s / (float)d + 1e-8f);
    auto normed = [&](const f32x4& v, const f32x4& g) { return f32x4{g.x * (v.x / r), g.y * (v.y / r), g.z * (v.z / r), g.w * (v.w / r)}; };
    auto later = [&](int i) { return normed(*reinterpret_cast<const f32x4*>(x + i), *reinterpret_cast<const f32x4*>(gamma + i)); }; // past the kept ones
#pragma unroll
    for (int k = 0; k < KEEP; k++) keep[k] = normed(keep[k], gain[k]);
    int e = 0;
    if constexpr (__is_same(AT, h2_t)) { // the row's scale
        int most = -100000;
#pragma unroll
        for (int k = 0; k < KEEP; k++) most = max(most, h2_size4(keep[k].x, keep[k].y, keep[k].z, keep[k].w)); // (past the end: the last columns once more)
        for (int i = lane * 4 + KEEP * 256; i < d; i += 256) {
            const f32x4 v = later(i);
            most = max(most, h2_size4(v.x, v.y, v.z, v.w));
        }
        e = h2_exponent(pf_wave_max(most));
        if (lane == 0) exps[row] = e;
    }
    auto store = [&](int i, const f32x4& v) {
        if constexpr (__is_same(AT, h2_t)) h2_put4<false>((unsigned char*)out + (size_t)row * d * 4, i, ldexpf(v.x, -e), ldexpf(v.y, -e), ldexpf(v.z, -e), ldexpf(v.w, -e));
        else put4_at<AT>(out, (size_t)row, d, i, v.x, v.y, v.z, v.w);
    };
#pragma unroll
    for (int k = 0; k < KEEP; k++)
        if (lane * 4 + k * 256 < d) store(lane * 4 + k * 256, keep[k]);
    for (int i = lane * 4 + KEEP * 256; i < d; i += 256) store(i, later(i));
}
template <typename AT> static void launch_rmsnorm(hipStream_t st, const float* X, const float* gamma, void* out, int* exps, int n, int d) {
    const dim3 grid((n + 3) / 4);
    if (d <= 1024) hipLaunchKernelGGL((k_pf_rmsnorm<AT, 4>), grid, dim3(PWG), 0, st, X, gamma, out, exps, n, d);
    else if (d <= 2048) hipLaunchKernelGGL((k_pf_rmsnorm<AT, 8>), grid, dim3(PWG), 0, st, X, gamma, out, exps, n, d);
    else hipLaunchKernelGGL((k_pf_rmsnorm<AT, 16>), grid, dim3(PWG), 0, st, X, gamma, out, exps, n, d);
}

// Per (head, row): per-head RMSNorm of q and k (inference.cu:52-81, 97-111), RoPE on adjacent pairs at the
// row's position (inference.cu:113-134), q written back in place, k and v written to the KV pages.

template <int HD>
__global__ void __launch_bounds__(64) k_pf_qk_rope_kv(PfArgs P, LayerDev L) {
    constexpr int EPL = HD / 64;
    const StepArgs& a = P.a;
    const int h = blockIdx.x, row = blockIdx.y, lane = threadIdx.x;
    if (h == a.heads) { ple_columns<1>(P, L, row, 1, lane, 64); return; }
    const int seq = P.rowSeq[row], pos = P.rowPos[row];
    float* qkv = P.QKV + (size_t)row * P.qkvLd;
    float qv[EPL], kv[EPL], vv[EPL];
#pragma unroll
    for (int e = 0; e < EPL; e++) {
        const int i = lane * EPL + e;
        qv[e] = qkv[h * HD + i]; kv[e] = qkv[L.offK + h * HD + i]; vv[e] = qkv[L.offV + h * HD + i];
    }
    if (a.qkNorm) {
        float sq = 0.f, sk = 0.f;
#pragma unroll
        for (int e = 0; e < EPL; e++) { sq = fmaf(qv[e], qv[e], sq); sk = fmaf(kv[e], kv[e], sk); }
        sq = pf_wave_sum(sq); sk = pf_wave_sum(sk);
        const float rq = sqrtf(sq / (float)HD + 1e-8f), rk = sqrtf(sk / (float)HD + 1e-8f);
#pragma unroll
        for (int e = 0; e < EPL; e++) {
            const int i = lane * EPL + e;
            qv[e] = L.gq[h * HD + i] * (qv[e] / rq);
            kv[e] = L.gk[h * HD + i] * (kv[e] / rk);
        }
    }
    if (EPL == 1) {
        const float c = a.rope[(size_t)pos * HD + (lane & ~1)], s = a.rope[(size_t)pos * HD + (lane | 1)];
        const float qo = __shfl_xor(qv[0], 1, 64), ko = __shfl_xor(kv[0], 1, 64);
        if (lane & 1) { qv[0] = s * qo + c * qv[0]; kv[0] = s * ko + c * kv[0]; }
        else { qv[0] = c * qv[0] - s * qo; kv[0] = c * kv[0] - s * ko; }
    } else {
        const float c = a.rope[(size_t)pos * HD + 2 * lane], s = a.rope[(size_t)pos * HD + 2 * lane + 1];
        const float q0 = qv[0], q1 = qv[EPL - 1], k0 = kv[0], k1 = kv[EPL - 1];
        qv[0] = c * q0 - s * q1; qv[EPL - 1] = s * q0 + c * q1;
        kv[0] = c * k0 - s * k1; kv[EPL - 1] = s * k0 + c * k1;
    }
    const int page = a.pageTable[seq * a.pagesPerSeq + (pos >> 6)];
    const size_t o = ((size_t)page * MLH_KV_PAGE + (pos & 63)) * a.dim + h * HD;
#pragma unroll
    for (int e = 0; e < EPL; e++) {
        const int i = lane * EPL + e;
        qkv[h * HD + i] = qv[e];
        L.K[o + i] = kv[e];
        L.V[o + i] = vv[e];
    }
    if (P.Kh) { // the half copies, rounded exactly as the attention kernel rounds the fp32 rows on its way into LDS
        const size_t ho = (size_t)row * a.dim + h * HD + lane * EPL;
        if (EPL == 2) {
            *reinterpret_cast<uint32_t*>(P.Kh + ho) = pack_f16(kv[0], kv[1]);
            *reinterpret_cast<uint32_t*>(P.Vh + ho) = pack_f16(vv[0], vv[1]);
        } else {
#pragma unroll
            for (int e = 0; e < EPL; e++) {
                P.Kh[ho + e] = __builtin_bit_cast(uint16_t, (_Float16)kv[e]);
                P.Vh[ho + e] = __builtin_bit_cast(uint16_t, (_Float16)vv[e]);
            }
        }
    }
}

// Causal attention for 16 queries of one head at fp32 precision (inference.cu:136-239, 511-573 for these columns), optional sigmoid gate
// (:241-250), on the fp32 matrix cores (v_mfma_f32_16x16x4_f32: every product and sum fp32).
//
// The four or eight waves of a workgroup take key tiles of 16 in turn, each with an online softmax of its own, and meet once at the end; nothing goes through
// LDS on the way.  S^T[key, query] = K . Q^T: lane 16 g + n holds a key's (a query's) columns [g HD/4, (g + 1) HD/4), the order of the contraction being
// free.  The accumulator leaves the lane the scores of keys 4 g .. 4 g + 3 of query n, which is the operand P of O^T += V^T . P^T as it stands; row m of the
// V operand of block b is dimension m HD/16 + b, so V comes in 16-byte pieces as well.  Loads of the wave's next tile go out before this one's products.
// Bound by the matrix cores' fp32 rate and, for few rows, by the longest chain of tiles: eight waves where that leaves a unit one workgroup (84 rows, 6 heads
// of 128: 9.0 us, 11.4 by four; 517: 21.6, 31.4).  Measured: 517 rows 107 us on the vector ALU through LDS tiles of 64 keys; 17 376 rows of 64 sequences,
// 12 heads of 64: 170 us (899; 178 while the compiler put a tile's loads behind the products they were to run under).
#define PF_QB 16
template <int HD, int NW, typename AT>
__global__ void __launch_bounds__(NW * 64) k_pf_attn(PfArgs P, LayerDev L) {
    constexpr int KC = HD / 4, VB = HD / 16, LDO = HD + 4;
    __shared__ float part[NW][PF_QB][LDO], stat[NW][2][PF_QB];
    const StepArgs& a = P.a;
    const int h = blockIdx.x, blk = blockIdx.y, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int seg = P.blkSeg[blk], q0 = P.blkQ0[blk];
    const int seq = P.segSeq[seg], pos0 = P.segPos0[seg], len = P.segLen[seg], row0 = P.segStart[seg] + q0;
    const int nq = min(PF_QB, len - q0), maxPos = pos0 + q0 + nq - 1, qpos = pos0 + q0 + n;
    f32x4 q[KC / 4];
    {
        const float* qr = P.QKV + (size_t)(row0 + min(n, nq - 1)) * P.qkvLd + h * HD + g * KC;
#pragma unroll
        for (int c = 0; c < KC / 4; c++) q[c] = *reinterpret_cast<const f32x4*>(qr + 4 * c);
    }
    const float scale = 1.0f / sqrtf((float)HD);
    f32x4 k[2][KC / 4], v[2][4][VB / 4], acc[VB];
#pragma unroll
    for (int b = 0; b < VB; b++) acc[b] = (f32x4)(0.f);
    float m = -1.0e30f, l = 0.f; // of query n; l: over this lane's keys
    const int ntiles = (maxPos >> 4) + 1;
    auto fetch = [&](int t, int set) __attribute__((always_inline)) { // (rows behind the last position that a query here sees: that row again, with weight zero)
        const int j0 = t * 16, last = maxPos - j0;
        const size_t base = ((size_t)a.pageTable[seq * a.pagesPerSeq + (j0 >> 6)] * MLH_KV_PAGE + (j0 & 63)) * a.dim + h * HD;
        const float* kr = L.K + base + (size_t)min(n, last) * a.dim + g * KC;
#pragma unroll
        for (int c = 0; c < KC / 4; c++) k[set][c] = *reinterpret_cast<const f32x4*>(kr + 4 * c);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float* vr = L.V + base + (size_t)min(4 * g + i, last) * a.dim + n * VB;
#pragma unroll
            for (int c = 0; c < VB / 4; c++) v[set][i][c] = *reinterpret_cast<const f32x4*>(vr + 4 * c);
        }
    };
    auto tile = [&](int t, int set) __attribute__((always_inline)) {
        f32x4 s0 = (f32x4)(0.f), s1 = (f32x4)(0.f); // two chains
#pragma unroll
        for (int c = 0; c < KC / 4; c++) {
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[set][c].x, q[c].x, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[set][c].y, q[c].y, s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[set][c].z, q[c].z, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[set][c].w, q[c].w, s1, 0, 0, 0);
        }
        const int key = t * 16 + 4 * g;
        float s[4], mt = m;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s[i] = key + i <= qpos ? (s0[i] + s1[i]) * scale : -1.0e30f;
            mt = fmaxf(mt, s[i]);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
        mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
        const float corr = expf(m - mt);
        l *= corr;
        m = mt;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s[i] = key + i <= qpos ? expf(s[i] - mt) : 0.f;
            l += s[i];
        }
#pragma unroll
        for (int b = 0; b < VB; b++) acc[b] *= corr;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int b = 0; b < VB; b++) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[set][i][b / 4][b % 4], s[i], acc[b], 0, 0, 0);
    };
    int t = wave;
    if (t < ntiles) fetch(t, 0);
    while (t < ntiles) { // (no further tile: the same loads again, dropped)
        fetch(min(t + NW, ntiles - 1), 1);
        __builtin_amdgcn_sched_barrier(0); // (the compiler would put the loads behind the products)
        tile(t, 0);
        t += NW;
        if (t >= ntiles) break;
        fetch(min(t + NW, ntiles - 1), 0);
        __builtin_amdgcn_sched_barrier(0);
        tile(t, 1);
        t += NW;
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (g == 0) { stat[wave][0][n] = m; stat[wave][1][n] = l; }
    __syncthreads();
    { // this wave's share, at the common maximum
        float M = stat[0][0][n];
#pragma unroll
        for (int w = 1; w < NW; w++) M = fmaxf(M, stat[w][0][n]);
        const float f = expf(m - M);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int b = 0; b < VB; b += 4)
                *reinterpret_cast<f32x4*>(&part[wave][n][(4 * g + i) * VB + b]) = f32x4{acc[b][i], acc[b + 1][i], acc[b + 2][i], acc[b + 3][i]} * f;
    }
    __syncthreads();
    for (int i = tid; i < nq * (HD / 4); i += NW * 64) {
        const int qi = i / (HD / 4), c4 = (i % (HD / 4)) * 4;
        float M = stat[0][0][qi], den = 0.f;
#pragma unroll
        for (int w = 1; w < NW; w++) M = fmaxf(M, stat[w][0][qi]);
        f32x4 o = (f32x4)(0.f);
#pragma unroll
        for (int w = 0; w < NW; w++) {
            den = fmaf(stat[w][1][qi], expf(stat[w][0][qi] - M), den);
            o += *reinterpret_cast<const f32x4*>(&part[w][qi][c4]);
        }
        const size_t row = (size_t)(row0 + qi);
        o.x /= den; o.y /= den; o.z /= den; o.w /= den;
        if (a.gating) {
            const f32x4 z = *reinterpret_cast<const f32x4*>(P.QKV + row * P.qkvLd + L.offG + h * HD + c4);
            o.x *= pf_sigmoid(z.x); o.y *= pf_sigmoid(z.y); o.z *= pf_sigmoid(z.z); o.w *= pf_sigmoid(z.w);
        }
        put_mix4<AT>(P, row, h * HD + c4, o);
    }
}

// ----------------------------------------------------------------------------
// fp16 MFMA causal attention (bf16-weight models; their MFMA path computes in IEEE half, see the host section).  A workgroup owns one head and 128 consecutive
// queries of one segment, a wave 32 of them.  Per 64-key page:
//   S^T[key, query] = K . Q^T      (A = K tile from LDS, B = Q^T held in registers)
//   online softmax down the key axis -- with the transposed product every lane owns ONE query column
//   (accumulator element i of lane l is row 8(i/4) + 4(l/32) + i%4, column l%32), so the running max,
//   the running sum and the rescale of the output are in-lane, plus one exchange between lane halves
//   O^T[hd, query] += V^T . P^T    (B = the lane's own P values, A = V transposed in LDS)
// The contraction index of the second product may be permuted freely as long as A and B agree: slot
// (half, e) of 16-key step t is the key the accumulator layout puts there, and the V tile is written
// to LDS transposed in exactly that order, so P never leaves its registers.
// K and V come from the fp32 pages and are rounded to fp16 on the way into LDS; scores, softmax
// statistics and the output accumulate in fp32.
// ----------------------------------------------------------------------------
#define PF_MQB 128
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));


// position of key k (0..63) of a page along the permuted contraction axis of O^T += V^T . P^T
__device__ __forceinline__ int pv_slot(int k) {
    const int b = k >> 5, k32 = k & 31;
    const int i = 4 * (k32 >> 3) + (k32 & 3), hh = (k32 >> 2) & 1;
    return 16 * (2 * b + (i >> 3)) + 8 * hh + (i & 7);
}

template <int HD, bool H16>
__global__ void __launch_bounds__(PWG, H16 ? 2 : 1) k_pf_attn_mfma(PfArgs P, LayerDev L) {
    constexpr int KP = HD + 8;   // K tile row pitch (16-bit elements): 16-byte reads, rows 4 banks apart
    constexpr int VP = 64 + 8;   // V^T row pitch
    constexpr int KS = HD / 16;  // 16-wide contraction steps of K . Q^T
    constexpr int MB = HD / 32;  // 32-row blocks of O^T
    __shared__ __attribute__((aligned(16))) uint16_t Kt[64 * KP];
    __shared__ __attribute__((aligned(16))) uint16_t Vt[HD * VP];
    const StepArgs& a = P.a;
    const int h = blockIdx.x, blk = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int seg = P.blkSeg[blk], q0 = P.blkQ0[blk];
    const int seq = P.segSeq[seg], pos0 = P.segPos0[seg], len = P.segLen[seg];
    const int n32 = lane & 31, half = lane >> 5;
    const int qi = q0 + wave * 32 + n32;              // this lane's query within the segment
    const int qrow = P.segStart[seg] + min(qi, len - 1);
    const int qpos = pos0 + qi;
    const int waveMaxPos = pos0 + min(q0 + wave * 32 + 31, len - 1);
    const int maxPos = pos0 + min(q0 + PF_MQB, len) - 1;
    const bool waveActive = q0 + wave * 32 < len;

    // Q^T operand (fp16): for step s the lane holds q[16 s + 8 half .. +7] of its query, times log2(e) / sqrt(HD): the
    // scores come out of the MFMA ready for exp2
    u32x4 qop[KS];
    {
        const float* q = P.QKV + (size_t)qrow * P.qkvLd + h * HD + 8 * half;
        const float qs = 1.44269504088896341f / sqrtf((float)HD);
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const f32x4 lo = *reinterpret_cast<const f32x4*>(q + 16 * s), hi = *reinterpret_cast<const f32x4*>(q + 16 * s + 4);
            // one at a time: product and conversion are then one instruction (v_fma_mixlo_f16) and the product is rounded once
            auto pair = [&](float a, float b) { return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(a * qs)) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(b * qs)) << 16); };
            qop[s].x = pair(lo.x, lo.y); qop[s].y = pair(lo.z, lo.w);
            qop[s].z = pair(hi.x, hi.y); qop[s].w = pair(hi.z, hi.w);
        }
    }
    f32x16 oacc[MB];
#pragma unroll
    for (int b = 0; b < MB; b++)
#pragma unroll
        for (int i = 0; i < 16; i++) oacc[b][i] = 0.f;
    float m_run = -1.0e30f, l_run = 0.f;
    const int waveMinPos = pos0 + q0 + wave * 32; // the lowest query position of the wave
    const int ntiles = (maxPos >> 6) + 1;

    // A tile's K and V rows travel global -> registers -> LDS; the loads of tile t + 1 are issued before tile t is
    // multiplied, so their latency runs under the MFMAs.  Rows beyond the last position any query of the workgroup
    // may see are read from a clamped row and zeroed (every load unconditional: all of them in flight at once).
    // H16: every segment of the call starts at position 0, so key j of the segment is row segStart + j of the call and
    // its K and V rows exist as halves (written by the QK-norm / RoPE kernel): half the bytes, no conversion, and few
    // enough registers for two workgroups per compute unit -- one multiplies while the other does its softmax.
    constexpr int NK = 64 * (HD / 4) / PWG, NV = 32 * (HD / 4) / PWG;
    constexpr int NK16 = 64 * (HD / 8) / PWG, NV16 = 32 * (HD / 8) / PWG;
    f32x4 kreg[H16 ? 1 : NK], vreg[H16 ? 1 : NV][2];
    u32x4 kreg16[H16 ? NK16 : 1], vreg16[H16 ? NV16 : 1][2];
    auto fetch = [&](int t) {
        const int j0 = t << 6;
        const int rmax = maxPos - j0; // >= 0
        if (H16) {
            const size_t base = ((size_t)P.segStart[seg] + j0) * a.dim + h * HD; // pos0 == 0: key position == row within the segment
#pragma unroll
            for (int n = 0; n < NK16; n++) {
                const int i = tid + n * PWG, r = i / (HD / 8), c8 = (i % (HD / 8)) * 8;
                kreg16[n] = *reinterpret_cast<const u32x4*>(P.Kh + base + (size_t)min(r, rmax) * a.dim + c8);
            }
#pragma unroll
            for (int n = 0; n < NV16; n++) {
                const int i = tid + n * PWG, kp = i & 7, g = (i >> 3) % (HD / 8), ko = (i >> 3) / (HD / 8);
                const int k = 16 * ko + 2 * kp, c8 = 8 * g;
                vreg16[n][0] = *reinterpret_cast<const u32x4*>(P.Vh + base + (size_t)min(k, rmax) * a.dim + c8);
                vreg16[n][1] = *reinterpret_cast<const u32x4*>(P.Vh + base + (size_t)min(k + 1, rmax) * a.dim + c8);
            }
            return;
        }
        const int page = a.pageTable[seq * a.pagesPerSeq + t];
        const size_t base = ((size_t)page * MLH_KV_PAGE) * a.dim + h * HD;
#pragma unroll
        for (int n = 0; n < NK; n++) {
            const int i = tid + n * PWG, r = i / (HD / 4), c4 = (i % (HD / 4)) * 4;
            kreg[n] = *reinterpret_cast<const f32x4*>(L.K + base + (size_t)min(r, rmax) * a.dim + c4);
        }
#pragma unroll
        for (int n = 0; n < NV; n++) {
            const int i = tid + n * PWG, kp = i & 7, g = (i >> 3) % (HD / 4), ko = (i >> 3) / (HD / 4);
            const int k = 16 * ko + 2 * kp, c4 = 4 * g;
            vreg[n][0] = *reinterpret_cast<const f32x4*>(L.V + base + (size_t)min(k, rmax) * a.dim + c4);
            vreg[n][1] = *reinterpret_cast<const f32x4*>(L.V + base + (size_t)min(k + 1, rmax) * a.dim + c4);
        }
    };
    fetch(0);
    for (int t = 0; t < ntiles; t++) {
        const int j0 = t << 6;
        const int rmax = maxPos - j0;
        __syncthreads(); // the previous tile has been consumed
        if (H16) {
            // ---- K tile: natural layout, sixteen bytes per store ----
#pragma unroll
            for (int n = 0; n < NK16; n++) {
                const int i = tid + n * PWG, r = i / (HD / 8), c8 = (i % (HD / 8)) * 8;
                *reinterpret_cast<u32x4*>(Kt + r * KP + c8) = r <= rmax ? kreg16[n] : (u32x4)(0u);
            }
            // ---- V tile: transposed, keys in contraction-slot order; a lane carries two keys that are neighbours there:
            // for every column the halves of both keys go into one 32-bit word (v_perm picks the two 16-bit pieces) ----
#pragma unroll
            for (int n = 0; n < NV16; n++) {
                const int i = tid + n * PWG, kp = i & 7, g = (i >> 3) % (HD / 8), ko = (i >> 3) / (HD / 8);
                const int k = 16 * ko + 2 * kp, c8 = 8 * g;
                const u32x4 v0 = k <= rmax ? vreg16[n][0] : (u32x4)(0u), v1 = k + 1 <= rmax ? vreg16[n][1] : (u32x4)(0u);
                const int slot = pv_slot(k); // even, and pv_slot(k + 1) == slot + 1
#pragma unroll
                for (int w = 0; w < 4; w++) { // word w holds columns c8 + 2 w (low half) and c8 + 2 w + 1 (high half)
                    *reinterpret_cast<uint32_t*>(Vt + (c8 + 2 * w + 0) * VP + slot) = __builtin_amdgcn_perm(v1[w], v0[w], 0x05040100u);
                    *reinterpret_cast<uint32_t*>(Vt + (c8 + 2 * w + 1) * VP + slot) = __builtin_amdgcn_perm(v1[w], v0[w], 0x07060302u);
                }
            }
        } else {
        // ---- K tile: natural layout ----
#pragma unroll
            for (int n = 0; n < NK; n++) {
                const int i = tid + n * PWG, r = i / (HD / 4), c4 = (i % (HD / 4)) * 4;
                const f32x4 kk = r <= rmax ? kreg[n] : (f32x4)(0.f);
                u32x2 w; w.x = pack_f16(kk.x, kk.y); w.y = pack_f16(kk.z, kk.w);
                *reinterpret_cast<u32x2*>(Kt + r * KP + c4) = w;
            }
            // ---- V tile: transposed, keys in contraction-slot order; a lane carries two keys that are neighbours there ----
#pragma unroll
            for (int n = 0; n < NV; n++) {
                const int i = tid + n * PWG, kp = i & 7, g = (i >> 3) % (HD / 4), ko = (i >> 3) / (HD / 4); // key pair, column chunk, group of 8 pairs
                const int k = 16 * ko + 2 * kp, c4 = 4 * g;
                const f32x4 v0 = k <= rmax ? vreg[n][0] : (f32x4)(0.f), v1 = k + 1 <= rmax ? vreg[n][1] : (f32x4)(0.f);
                const int slot = pv_slot(k); // even, and pv_slot(k + 1) == slot + 1
                *reinterpret_cast<uint32_t*>(Vt + (c4 + 0) * VP + slot) = pack_f16(v0.x, v1.x);
                *reinterpret_cast<uint32_t*>(Vt + (c4 + 1) * VP + slot) = pack_f16(v0.y, v1.y);
                *reinterpret_cast<uint32_t*>(Vt + (c4 + 2) * VP + slot) = pack_f16(v0.z, v1.z);
                *reinterpret_cast<uint32_t*>(Vt + (c4 + 3) * VP + slot) = pack_f16(v0.w, v1.w);
            }
        }
        __syncthreads();
        if (t + 1 < ntiles) fetch(t + 1);
        if (!waveActive || j0 > waveMaxPos) continue; // wave-uniform; the barriers above are still reached by every wave
        // ---- S^T = K . Q^T for the two 32-key blocks ----
        f32x16 sacc[2];
#pragma unroll
        for (int b = 0; b < 2; b++) {
#pragma unroll
            for (int i = 0; i < 16; i++) sacc[b][i] = 0.f;
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const u32x4 kop = *reinterpret_cast<const u32x4*>(Kt + (32 * b + n32) * KP + 16 * s + 8 * half);
                sacc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, kop), __builtin_bit_cast(f16x8, qop[s]), sacc[b], 0, 0, 0);
            }
        }
        // ---- causal mask, online softmax down the key axis (base 2: the scores carry log2(e) / sqrt(HD)) ----
        // A tile that lies entirely at or below the wave's lowest query position needs no mask (all but the last one or
        // two tiles of a wave), and the output is only rescaled when some query's running maximum moved.
        float mx = -1.0e30f;
        const bool fullTile = j0 + 63 <= waveMinPos; // wave-uniform
        if (fullTile) {
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 16; i += 2) mx = fmaxf(mx, fmaxf(sacc[b][i], sacc[b][i + 1]));
        } else {
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int key = j0 + 32 * b + 8 * (i >> 2) + 4 * half + (i & 3);
                    const float sv = key <= qpos ? sacc[b][i] : -1.0e30f;
                    sacc[b][i] = sv;
                    mx = fmaxf(mx, sv);
                }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mn = fmaxf(m_run, mx);
        float ls = 0.f;
        if (fullTile) {
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float pv = __builtin_amdgcn_exp2f(sacc[b][i] - mn);
                    sacc[b][i] = pv;
                    ls += pv;
                }
        } else {
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float pv = sacc[b][i] > -1.0e29f ? __builtin_amdgcn_exp2f(sacc[b][i] - mn) : 0.f;
                    sacc[b][i] = pv;
                    ls += pv;
                }
        }
        ls += __shfl_xor(ls, 32, 64);
        if (__any(mn > m_run)) { // wave-uniform
            const float corr = __builtin_amdgcn_exp2f(m_run - mn);
            l_run *= corr;
#pragma unroll
            for (int b = 0; b < MB; b++)
#pragma unroll
                for (int i = 0; i < 16; i++) oacc[b][i] *= corr;
        }
        l_run += ls;
        m_run = mn;
        // ---- O^T += V^T . P^T ----
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const int b = st >> 1, e0 = 8 * (st & 1);
            u32x4 pop;
            pop.x = pack_f16(sacc[b][e0 + 0], sacc[b][e0 + 1]); pop.y = pack_f16(sacc[b][e0 + 2], sacc[b][e0 + 3]);
            pop.z = pack_f16(sacc[b][e0 + 4], sacc[b][e0 + 5]); pop.w = pack_f16(sacc[b][e0 + 6], sacc[b][e0 + 7]);
#pragma unroll
            for (int mb = 0; mb < MB; mb++) {
                const u32x4 vop = *reinterpret_cast<const u32x4*>(Vt + (32 * mb + n32) * VP + 16 * st + 8 * half);
                oacc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, vop), __builtin_bit_cast(f16x8, pop), oacc[mb], 0, 0, 0);
            }
        }
    }
    if (qi >= len) return;
    const float inv_l = 1.0f / l_run;
    const size_t row = (size_t)qrow;
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int i4 = 0; i4 < 4; i4++) {
            const int dcol = h * HD + 32 * mb + 8 * i4 + 4 * half;
            f32x4 o;
            o.x = oacc[mb][4 * i4] * inv_l; o.y = oacc[mb][4 * i4 + 1] * inv_l; o.z = oacc[mb][4 * i4 + 2] * inv_l; o.w = oacc[mb][4 * i4 + 3] * inv_l;
            if (a.gating) {
                const f32x4 gt = *reinterpret_cast<const f32x4*>(P.QKV + row * P.qkvLd + L.offG + dcol);
                o.x *= pf_sigmoid(gt.x); o.y *= pf_sigmoid(gt.y); o.z *= pf_sigmoid(gt.z); o.w *= pf_sigmoid(gt.w);
            }
            if (P.rows) { rows_put4(P.rows, dcol, (int)row, P.lay, true, o.x, o.y, o.z, o.w); continue; }
            u32x2 w; w.x = pack_f16(o.x, o.y); w.y = pack_f16(o.z, o.w);
            *reinterpret_cast<u32x2*>((bf16_t*)P.Amix + row * P.aLd + dcol) = w;
        }
}

// Gated-delta-net prefill.  The rows of a head's state evolve independently of each other
//   S[r,:] <- alpha S[r,:] + beta (v_r - alpha u_r) k^T,  u_r = S[r,:].k,   o_r = S_new[r,:].q
// (the decode kernel's update, regrouped; k, q L2-normalised), so one workgroup carries GR rows of
// one head of one segment in registers across the whole segment: eight lanes per two rows (GR = 64) or one (32), each with DK/8
// columns of them.  Sixteen tokens of q, k, v and gate inputs are staged in LDS at a time, the next sixteen
// being loaded into registers meanwhile.  The decay is kept out of the element loop: within the sixteen the registers hold S / a,
// a the product of their alphas so far, so a token costs three FMAs per element -- S.k, S.q and the rank-1 update --
// instead of four.  With p = S_old[r,:].q the read-out needs no second pass:
// o_r = (alpha p + w (k.q)) / |q|,  w = beta (v_r - alpha u_r) / |k|.
// A token's constants are ready before the sixteen begin, nothing in them branches, and the outputs leave together behind them: what is left
// from token to token is u's sum, two FMAs and the update.  Bound by that chain with one workgroup on a unit, by issue and by the LDS reads of
// k and q (why a lane has two rows) with three.  Measured (12 heads of 64): 19 segments of up to 333 tokens 101 us with 64 rows, 82 with 32 (148 with a
// branch and the output's conversion inside the token), 64 of up to 512 215 and 222 (263).
#define PF_GC 16
// Workgroup barrier that orders LDS traffic only: __syncthreads() also waits for every outstanding global
// load (loads and stores share one counter), which would put the next chunk's prefetch on the critical path.
__device__ __forceinline__ void pf_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
template <int CTRL> __device__ __forceinline__ float dpp_of(float v, float other = 0.f) { // lanes whose source lies outside the row of sixteen: `other`
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(other), __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float sum8(float v) { // over eight lanes, in all of them: in the vector ALU (a shuffle through LDS costs some 100 cycles)
    v += dpp_of<0xB1>(v);         // lanes 0<->1, 2<->3
    v += dpp_of<0x4E>(v);         // lanes 0<->2, 1<->3
    return v + dpp_of<0x141>(v);  // lane i <-> 7 - i
}
template <int DK, int GR, typename AT>
__global__ void __launch_bounds__(PWG) k_pf_gdn(PfArgs P, LayerDev L, int skipFrom) {
    constexpr int DV = DK, TPR = 8, RPT = GR * TPR / PWG, CPT = DK / TPR;
    static_assert(RPT == 1 || RPT == 2, "rows per eight lanes");
    constexpr int NQK = PF_GC * DK / 4 / PWG; // f32x4 loads per thread for each of q and k
    __shared__ __attribute__((aligned(16))) float qs[PF_GC][DK];
    __shared__ __attribute__((aligned(16))) float ks[PF_GC][DK];
    __shared__ __attribute__((aligned(16))) float vs[PF_GC][GR];
    __shared__ __attribute__((aligned(16))) float os[PF_GC][GR];
    __shared__ float zs[PF_GC][2];
    __shared__ float gate[PF_GC][5]; // alpha, beta, 1/|q|, 1/|k|, k.q
    __shared__ __attribute__((aligned(16))) f32x4 cst[PWG / 64][PF_GC]; // by wave: the factors of u, w, p in the read-out and w in the read-out
    const StepArgs& a = P.a;
    const int h = blockIdx.x, seg = blockIdx.y, r0 = blockIdx.z * GR, tid = threadIdx.x, wave = tid >> 6;
    const int seq = P.segSeq[seg], len = P.segLen[seg], row0 = P.segStart[seg];
    if (len >= skipFrom) return; // taken by the chunk-parallel kernels
    if (h == a.gdnHeads) { // the segment's PLE columns, a share of its rows each
        const int share = (len + gridDim.z - 1) / gridDim.z, from = min((int)blockIdx.z * share, len);
        ple_columns<8>(P, L, row0 + from, min(share, len - from), tid, PWG);
        return;
    }
    const int r = tid / TPR * RPT, cg = tid % TPR, c0 = cg * CPT;
    float* Srow = L.S + (((size_t)seq * a.gdnHeads + h) * DV + r0 + r) * DK + c0;
    float S[RPT][CPT];
#pragma unroll
    for (int j = 0; j < RPT; j++)
#pragma unroll
        for (int c = 0; c < CPT; c += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(Srow + j * DK + c);
            S[j][c] = v.x; S[j][c + 1] = v.y; S[j][c + 2] = v.z; S[j][c + 3] = v.w;
        }
    const float ba = L.gdnBa[h], bb = L.gdnBb[h]; // (loaded inside the loop they would wait for the next sixteen tokens, issued before them)
    f32x4 qreg[NQK], kreg[NQK];
    float vreg[PF_GC * GR / PWG], zreg = 0.f;
    auto fetch = [&](int t0) {
        const int last = len - 1 - t0; // >= 0
#pragma unroll
        for (int it = 0; it < NQK; it++) {
            const int i = it * PWG + tid, c = i / (DK / 4), e4 = (i % (DK / 4)) * 4;
            const float* qkv = P.QKV + (size_t)(row0 + t0 + min(c, last)) * P.qkvLd;
            qreg[it] = *reinterpret_cast<const f32x4*>(qkv + h * DK + e4);
            kreg[it] = *reinterpret_cast<const f32x4*>(qkv + L.offK + h * DK + e4);
        }
#pragma unroll
        for (int it = 0; it < PF_GC * GR / PWG; it++) {
            const int i = it * PWG + tid, c = i / GR, e = i % GR;
            vreg[it] = P.QKV[(size_t)(row0 + t0 + min(c, last)) * P.qkvLd + L.offV + h * DV + r0 + e];
        }
        if (tid < 2 * PF_GC) {
            const int c = tid >> 1;
            zreg = P.QKV[(size_t)(row0 + t0 + min(c, last)) * P.qkvLd + ((tid & 1) ? L.offGb : L.offGa) + h];
        }
    };
    auto put_outputs = [&](int t0, int nt) { // of the chunk from t0 on
        const int c = tid / (GR / 4), e4 = tid % (GR / 4) * 4;
        if (c < nt) put_mix4<AT>(P, (size_t)(row0 + t0 + c), h * DV + r0 + e4, *reinterpret_cast<const f32x4*>(&os[c][e4]));
    };
    fetch(0);
    for (int t0 = 0; t0 < len; t0 += PF_GC) {
        const int nt = min(PF_GC, len - t0);
        pf_lds_barrier(); // the previous chunk has been consumed
#pragma unroll
        for (int it = 0; it < NQK; it++) {
            const int i = it * PWG + tid, c = i / (DK / 4), e4 = (i % (DK / 4)) * 4;
            *reinterpret_cast<f32x4*>(&qs[c][e4]) = qreg[it];
            *reinterpret_cast<f32x4*>(&ks[c][e4]) = kreg[it];
        }
#pragma unroll
        for (int it = 0; it < PF_GC * GR / PWG; it++) {
            const int i = it * PWG + tid;
            vs[i / GR][i % GR] = vreg[it];
        }
        if (tid < 2 * PF_GC) zs[tid >> 1][tid & 1] = zreg;
        pf_lds_barrier();
        if (t0 + PF_GC < len) fetch(t0 + PF_GC); // in flight during this chunk's arithmetic
        if (t0 > 0) put_outputs(t0 - PF_GC, PF_GC);
        { // per token: |q|, |k|, k.q and the gates -- 16 threads per token
            const int c = tid >> 4, sub = tid & 15;
            float sq = 0.f, sk = 0.f, kq = 0.f;
#pragma unroll
            for (int e = sub * 4; e < DK; e += 64) {
                const f32x4 qv = *reinterpret_cast<const f32x4*>(&qs[c][e]), kv = *reinterpret_cast<const f32x4*>(&ks[c][e]);
#pragma unroll
                for (int i = 0; i < 4; i++) { sq = fmaf(qv[i], qv[i], sq); sk = fmaf(kv[i], kv[i], sk); kq = fmaf(kv[i], qv[i], kq); }
            }
            sq = sum8(sq); sk = sum8(sk); kq = sum8(kq);
            sq += dpp_of<0x140>(sq); sk += dpp_of<0x140>(sk); kq += dpp_of<0x140>(kq); // lane i <-> 15 - i
            const float za = zs[c][0] + ba, zb = zs[c][1] + bb;
            const float rq = 1.0f / sqrtf(sq + 1e-6f), rk = 1.0f / sqrtf(sk + 1e-6f);
            const float sp = fmaxf(za, 0.f) + log1pf(expf(-fabsf(za)));
            const bool past = c >= nt; // a token past the segment's end leaves the state as it is
            if (sub == 0) {
                gate[c][0] = past ? 1.f : expf(-sp);
                gate[c][1] = past ? 0.f : pf_sigmoid(zb);
                gate[c][2] = rq; gate[c][3] = rk; gate[c][4] = kq * rq * rk; // k.q of the normalised vectors
            }
        }
        pf_lds_barrier();
        float aprod; // the product of the chunk's alphas
        bool fold;   // ... is too small to carry: every token folds its alpha into the registers instead
        { // a token's constants, by lane (each wave for itself; lanes that agree mod 16 alike)
            const int c = tid & 15;
            const float alpha = gate[c][0], beta = gate[c][1], rq = gate[c][2], rk = gate[c][3], kqn = gate[c][4];
            float pr = alpha; // of the alphas up to this token
            pr *= dpp_of<0x111>(pr, 1.f); pr *= dpp_of<0x112>(pr, 1.f); pr *= dpp_of<0x114>(pr, 1.f); pr *= dpp_of<0x118>(pr, 1.f);
            aprod = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pr), 15));
            fold = !(aprod >= 1.0e-12f);
            const float before = fold ? 1.f : dpp_of<0x111>(pr, 1.f), after = fold ? 1.f : pr;
            f32x4 k4;
            k4.x = alpha * rk * before; k4.y = beta * rk / after; k4.z = alpha * rq * before; k4.w = beta * kqn;
            if ((tid & 63) < 16) cst[wave][c] = k4;
        }
        float kept[2][RPT] = {}; // outputs of tokens cg and cg + 8: row r (and r + 1)
        struct Token { f32x4 k[CPT / 4], q[CPT / 4], f; float v[RPT]; };
        auto load = [&](int c) __attribute__((always_inline)) {
            Token t;
#pragma unroll
            for (int e = 0; e < CPT / 4; e++) {
                t.k[e] = *reinterpret_cast<const f32x4*>(&ks[c][c0 + 4 * e]);
                t.q[e] = *reinterpret_cast<const f32x4*>(&qs[c][c0 + 4 * e]);
            }
            t.f = cst[wave][c];
#pragma unroll
            for (int j = 0; j < RPT; j++) t.v[j] = vs[c][r + j];
            return t;
        };
        auto token = [&](int c, const Token& t, bool folding) __attribute__((always_inline)) {
            float ua[RPT][2] = {}, pa[RPT][2] = {}; // two chains each
#pragma unroll
            for (int e = 0; e < CPT; e++)
#pragma unroll
                for (int j = 0; j < RPT; j++) {
                    ua[j][e & 1] = fmaf(S[j][e], t.k[e / 4][e % 4], ua[j][e & 1]);
                    pa[j][e & 1] = fmaf(S[j][e], t.q[e / 4][e % 4], pa[j][e & 1]);
                }
            const float alpha = folding ? gate[c][0] : 1.f;
#pragma unroll
            for (int j = 0; j < RPT; j++) {
                const float w = fmaf(-t.f.x, sum8(ua[j][0] + ua[j][1]), t.v[j]), s = t.f.y * w; // s: the coefficient of k
#pragma unroll
                for (int e = 0; e < CPT; e++) S[j][e] = fmaf(s, t.k[e / 4][e % 4], folding ? alpha * S[j][e] : S[j][e]);
                const float o = fmaf(t.f.z, sum8(pa[j][0] + pa[j][1]), t.f.w * w);
                kept[c >> 3][j] = cg == (c & 7) ? o : kept[c >> 3][j];
            }
        };
        if (!fold) {
            Token t[2];
            t[0] = load(0);
#pragma unroll
            for (int c = 0; c < PF_GC; c++) { // the next token's values are on their way out of LDS during this one
                if (c + 1 < PF_GC) t[(c + 1) & 1] = load(c + 1);
                __builtin_amdgcn_sched_barrier(0);
                token(c, t[c & 1], false);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < RPT; j++)
#pragma unroll
                for (int e = 0; e < CPT; e++) S[j][e] *= aprod;
        } else {
            for (int c = 0; c < PF_GC; c++) token(c, load(c), true);
        }
#pragma unroll
        for (int j = 0; j < RPT; j++) { os[cg][r + j] = kept[0][j]; os[cg + 8][r + j] = kept[1][j]; }
    }
    pf_lds_barrier();
    const int tail = (len - 1) / PF_GC * PF_GC;
    put_outputs(tail, len - tail);
#pragma unroll
    for (int j = 0; j < RPT; j++)
#pragma unroll
        for (int c = 0; c < CPT; c += 4) {
            f32x4 v; v.x = S[j][c]; v.y = S[j][c + 1]; v.z = S[j][c + 2]; v.w = S[j][c + 3];
            *reinterpret_cast<f32x4*>(Srow + j * DK + c) = v;
        }
}

// ----------------------------------------------------------------------------
// Chunk-parallel gated-delta-net prefill on the MFMA units (bf16 models, segments of 64 tokens or more).
//
// Over a chunk of C = 64 tokens starting from state S0, with g_t = sum_{j<=t} log(alpha_j):
//   S_t = e^{g_t} S0 + sum_{i<=t} e^{g_t - g_i} w_i k_i^T,      w_t = beta_t (v_t - alpha_t S_{t-1} k_t)
// (k, q L2-normalised).  Substituting S_{t-1} gives a unit-lower-triangular system for the w_t:
//   (I + A) W^T = beta (.) V - diag(beta e^{g}) K S0^T,   A[t,i] = beta_t e^{g_t - g_i} (k_i . k_t), i < t
// so W^T = Vt - Kt S0^T with Vt = (I+A)^{-1} (beta (.) V) and Kt = (I+A)^{-1} diag(beta e^{g}) K, both free
// of S0.  The outputs and the next state are then plain products:
//   O   = diag(e^{g}) Q S0^T + M W^T,      M[t,i] = e^{g_t - g_i} (k_i . q_t), i <= t
//   S_C = e^{g_C} S0 + W Kh,               Kh[i,:] = e^{g_C - g_i} k_i
// k_gdn_prep builds Vt, Kt, diag(e^g) Q, M, Kh for every chunk of every head in parallel (forward
// substitution, 64 steps, one column per thread); k_gdn_scan walks the chunks of one head of one
// segment in order with the state -- transposed, S^T[dk, dv] -- in MFMA accumulators, 56 MFMAs per
// chunk and wave.  Operands are IEEE half, accumulation and the state fp32.  Every contraction index
// (dk in Kt S0^T and Q S0^T, the chunk's token index in M W^T and Kh^T W^T) is stored in the order
// the accumulator layout holds it (slot_of below), so S0^T and W^T are used as MFMA B operands straight
// from the accumulator registers, without a transpose through LDS.
// ----------------------------------------------------------------------------
#define GD_C 64
// accumulator element i of lane (n, half) of a 32x32 tile is row 8(i/4) + 4 half + i%4; a 16-wide MFMA step
// st takes elements 8 st .. 8 st + 7 of both halves.  slot_of(x) = position of row x of a (multi-tile)
// contraction axis in that order: tile x/32, then step, half, element.
__host__ __device__ __forceinline__ int slot_of(int x) {
    const int x32 = x & 31;
    const int i = 4 * (x32 >> 3) + (x32 & 3), hh = (x32 >> 2) & 1;
    return (x & ~31) + 16 * (i >> 3) + 8 * hh + (i & 7);
}
// One chunk's operands as fragments of 1 KB: what a wave's lanes take of a 32-row, 16-step operand, 16 bytes each.
template <int DK> struct GdLayout {
    static constexpr int JT = DK / 32;
    static constexpr int fKt = 0, fQh = fKt + 4 * JT, fM = fQh + 4 * JT, fKhT = fM + 6, fVt = fKhT + 4 * JT; // [token tile][dk step]; M's three tiles; [dk tile][token step]; [dv tile][token step]
    static constexpr int frags = fVt + 4 * JT, total = frags * 1024;
};
__device__ __forceinline__ uint16_t f16_bits(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }

template <int DK>
__global__ void __launch_bounds__(2 * DK, 2) k_gdn_prep(PfArgs P, LayerDev L, const int* __restrict__ chunkSeg, const int* __restrict__ chunkT0,
                                                      unsigned char* __restrict__ ws, float* __restrict__ gCexp) {
    constexpr int DV = DK, NT = 2 * DK, JT = DK / 32;
    typedef GdLayout<DK> Lay;
    extern __shared__ __attribute__((aligned(16))) unsigned char pls[];
    float* Am = reinterpret_cast<float*>(pls);            // [64][64]
    float* gs = Am + GD_C * GD_C;                         // g[64], beta[64], sp[64], 1/|k|[64], 1/|q|[64], partial sums [4][64]
    uint16_t* k16 = reinterpret_cast<uint16_t*>(gs + 12 * GD_C); // [64][DK + 8] normalised k, half
    uint16_t* q16 = k16 + GD_C * (DK + 8);
    const StepArgs& a = P.a;
    const int chunk = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int seg = chunkSeg[chunk], t0 = chunkT0[chunk];
    const int nv = min(GD_C, P.segLen[seg] - t0), row0 = P.segStart[seg] + t0;
    if (h == a.gdnHeads) { ple_columns<8>(P, L, row0, nv, tid, NT); return; }
    unsigned char* img = ws + ((size_t)chunk * a.gdnHeads + h) * Lay::total;
    float* g = gs; float* beta = gs + GD_C; float* sp = gs + 2 * GD_C; float* rk = gs + 3 * GD_C; float* rq = gs + 4 * GD_C;
    float* part = gs + 5 * GD_C;
    float* eg = gs + 9 * GD_C;   // e^{g_t}
    float* egc = gs + 10 * GD_C; // e^{g_C - g_t}

    // Thread (sel, cidx) keeps column cidx of q (sel 0: threads [0, DK)) or k (sel 1: threads [DK, 2 DK)) for the 64
    // tokens of the chunk in registers (tokens past the segment end: zero).
    const int sel = tid / DK, cidx = tid % DK;
    float colv[GD_C];
    {
        const float* src = P.QKV + (size_t)row0 * P.qkvLd + (sel ? L.offK : 0) + h * DK + cidx;
#pragma unroll
        for (int t = 0; t < GD_C; t++) { // unconditional loads of clamped rows: 64 loads in flight, no branch per row
            const float v = src[(size_t)min(t, nv - 1) * P.qkvLd];
            colv[t] = t < nv ? v : 0.f;
        }
    }
    if (tid < GD_C) { // gates
        const int t = tid;
        float s_ = 0.f, b_ = 0.f;
        if (t < nv) {
            const float* qkv = P.QKV + (size_t)(row0 + t) * P.qkvLd;
            const float za = qkv[L.offGa + h] + L.gdnBa[h], zb = qkv[L.offGb + h] + L.gdnBb[h];
            s_ = fmaxf(za, 0.f) + log1pf(expf(-fabsf(za))); // -log(alpha)
            b_ = pf_sigmoid(zb);
        }
        sp[t] = s_; beta[t] = b_;
        float v = -s_; // inclusive prefix sum over the 64 tokens (one wave)
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const float u = __shfl_up(v, o, 64); if (tid >= o) v += u; }
        g[t] = v;
    }
    { // squared norms per token: reduce-scatter over the 64 lanes of a wave (lane t ends up with token t), then over waves
        float r[GD_C];
#pragma unroll
        for (int t = 0; t < GD_C; t++) r[t] = colv[t] * colv[t];
#pragma unroll
        for (int o = 32, n = 32; o > 0; o >>= 1, n >>= 1) {
            const bool up = (lane & o) != 0;
#pragma unroll
            for (int i = 0; i < n; i++) {
                const float keep = up ? r[i + n] : r[i], send = up ? r[i] : r[i + n];
                r[i] = keep + __shfl_xor(send, o, 64);
            }
        }
        part[wave * GD_C + lane] = r[0];
    }
    __syncthreads();
    if (tid < 2 * GD_C) { // 1 / norm of q (threads 0..63) and k (64..127)
        const int t = tid & 63, m = tid >> 6; // m 0: q, 1: k
        constexpr int WPM = DK / 64;          // waves per matrix
        float ss = 0.f;
#pragma unroll
        for (int w = 0; w < WPM; w++) ss += part[(m * WPM + w) * GD_C + t];
        (m ? rk : rq)[t] = 1.0f / sqrtf(ss + 1e-6f);
        if (m == 0) { eg[t] = expf(g[t]); egc[t] = expf(g[GD_C - 1] - g[t]); }
    }
    __syncthreads();
    { // normalise the register column, publish the half copy for the MFMAs
        const float* rr = sel ? rk : rq;
        uint16_t* d16 = sel ? k16 : q16;
#pragma unroll
        for (int t = 0; t < GD_C; t++) {
            colv[t] *= rr[t];
            d16[t * (DK + 8) + cidx] = f16_bits(colv[t]);
        }
    }
    __syncthreads();
    { // K K^T and Q K^T on the MFMA units: 2 x 2 tiles each
        const int n32 = lane & 31, half = lane >> 5;
        for (int tix = wave; tix < 8; tix += NT / 64) {
            const int which = tix >> 2, tt = (tix >> 1) & 1, ti = tix & 1;
            const uint16_t* Aop = (which ? q16 : k16) + (32 * tt + n32) * (DK + 8) + 8 * half;
            const uint16_t* Bop = k16 + (32 * ti + n32) * (DK + 8) + 8 * half;
            const int i_ = 32 * ti + n32;
            f32x4 gt[4], bt[4]; // of the lane's sixteen tokens, read ahead: behind the stores below every one would wait for its way out of LDS
#pragma unroll
            for (int q = 0; q < 4; q++) {
                gt[q] = *reinterpret_cast<const f32x4*>(g + 32 * tt + 8 * q + 4 * half);
                bt[q] = *reinterpret_cast<const f32x4*>(beta + 32 * tt + 8 * q + 4 * half);
            }
            const float gi = g[i_];
            f32x16 acc;
#pragma unroll
            for (int i = 0; i < 16; i++) acc[i] = 0.f;
#pragma unroll
            for (int s_ = 0; s_ < DK / 16; s_++)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4*>(Aop + 16 * s_)),
                                                             __builtin_bit_cast(f16x8, *reinterpret_cast<const u32x4*>(Bop + 16 * s_)), acc, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int t = 32 * tt + 8 * (e >> 2) + 4 * half + (e & 3);
                const float dec = expf(gt[e >> 2][e & 3] - gi); // <= 1 where it is used (i <= t)
                if (which == 0) Am[t * GD_C + i_] = i_ < t ? bt[e >> 2][e & 3] * dec * acc[e] : 0.f;
                else if (ti <= tt) // (the tile above the diagonal is zero and not stored)
                    *reinterpret_cast<uint16_t*>(img + (Lay::fM + (tt + ti) * 2 + ((slot_of(i_) >> 4) & 1)) * 1024 + (((slot_of(i_) >> 3) & 1) * 32 + (t & 31)) * 16 + 2 * (slot_of(i_) & 7)) =
                        f16_bits(i_ <= t ? dec * acc[e] : 0.f);
            }
        }
    }
    __syncthreads();
    // forward substitution, one column per thread: threads [0, DV) solve beta (.) V, threads [DV, 2 DV) -- the ones
    // that hold the k columns -- solve diag(beta e^g) K
    float X[GD_C];
    const int col = cidx;
    if (tid < DV) {
        const float* vsrc = P.QKV + (size_t)row0 * P.qkvLd + L.offV + h * DV + col;
#pragma unroll
        for (int t = 0; t < GD_C; t++) X[t] = vsrc[(size_t)min(t, nv - 1) * P.qkvLd]; // all 64 loads in flight at once
#pragma unroll
        for (int t = 0; t < GD_C; t++) X[t] *= beta[t]; // beta is zero for tokens past the segment end
    } else {
#pragma unroll
        for (int t = 0; t < GD_C; t++) X[t] = beta[t] * eg[t] * colv[t];
    }
    // Blocked forward substitution.  The 64 rows go in four blocks of 16: inside a block a thread solves its column in
    // fp32 as before (the block's own triangle, 120 multiply-adds); what the solved block contributes to all later rows,
    // A[later rows, block] X[block], is a matrix product and runs on the MFMA units with half operands -- a wave takes
    // its own 64 columns (two column tiles), so nothing here needs a workgroup barrier: LDS instructions of a wave
    // execute in order.  Per wave 8 MFMAs replace three quarters of the 2016 multiply-adds a thread had on its chain.
    {
        constexpr int AHP = GD_C + 8;                       // pitch of the half copy of A (elements): 16-byte reads, rows 4 banks apart
        uint16_t* Ah = k16;                                 // [64][AHP]; k16 / q16 are free: their MFMAs are done (barrier above)
        unsigned char* wsc = reinterpret_cast<unsigned char*>(Ah + GD_C * AHP) + wave * (64 * 80); // this wave's exchange area
        // X of the solved block as halves, [column][16] with pitch 48 bytes (B operand); the update of the next block's
        // rows, [column][16] floats with pitch 80 bytes -- both conflict-free for 16-byte accesses, and they may share
        // the area: the MFMAs have read the one before the other is written (same wave, in order)
        for (int i = tid; i < GD_C * GD_C / 2; i += NT) { // half copy of A, two elements per thread and trip
            const int t = i / (GD_C / 2), i2 = (i % (GD_C / 2)) * 2;
            *reinterpret_cast<uint32_t*>(Ah + t * AHP + i2) = pack_f16(Am[t * GD_C + i2], Am[t * GD_C + i2 + 1]);
        }
        __syncthreads();
        const int n32 = lane & 31, half = lane >> 5;
        f32x16 upd[2]; // [column tile of the wave]: what the solved blocks contribute to rows 32 .. 63
#pragma unroll
        for (int ct = 0; ct < 2; ct++)
#pragma unroll
            for (int e = 0; e < 16; e++) upd[ct][e] = 0.f;
        auto hand_over = [&](const f32x16& u, int ct, int e0) { // elements e0 .. e0 + 7 = 16 rows of a tile, to the owners of the columns
#pragma unroll
            for (int j = 0; j < 2; j++) {
                f32x4 v;
                v.x = u[e0 + 4 * j]; v.y = u[e0 + 4 * j + 1]; v.z = u[e0 + 4 * j + 2]; v.w = u[e0 + 4 * j + 3];
                *reinterpret_cast<f32x4*>(wsc + (32 * ct + n32) * 80 + (8 * j + 4 * half) * 4) = v; // rows 8 j + 4 half + 0..3 of the block
            }
        };
#pragma unroll
        for (int b = 0; b < 4; b++) {
            if (b > 1) { // rows 16 b .. 16 b + 15: elements 8 (b & 1) .. + 7 of the tile of rows 32 .. 63 (block 1's were handed over by block 0)
                hand_over(upd[0], 0, 8 * (b & 1));
                hand_over(upd[1], 1, 8 * (b & 1));
            }
            if (b > 0) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const f32x4 u = *reinterpret_cast<const f32x4*>(wsc + lane * 80 + q * 16);
                    X[16 * b + 4 * q] -= u.x; X[16 * b + 4 * q + 1] -= u.y; X[16 * b + 4 * q + 2] -= u.z; X[16 * b + 4 * q + 3] -= u.w;
                }
            }
#pragma unroll
            for (int tt = 1; tt < 16; tt++) { // the block's own triangle
                const int t = 16 * b + tt;
                float acc0 = X[t], acc1 = 0.f, acc2 = 0.f, acc3 = 0.f; // four chains: the row's dot product is on the serial path
#pragma unroll
                for (int i4 = 0; i4 < tt; i4 += 4) {
                    const f32x4 a4 = *reinterpret_cast<const f32x4*>(Am + t * GD_C + 16 * b + i4); // zero at and beyond the diagonal
                    acc0 = fmaf(-a4.x, X[16 * b + i4], acc0);
                    if (i4 + 1 < tt) acc1 = fmaf(-a4.y, X[16 * b + i4 + 1], acc1);
                    if (i4 + 2 < tt) acc2 = fmaf(-a4.z, X[16 * b + i4 + 2], acc2);
                    if (i4 + 3 < tt) acc3 = fmaf(-a4.w, X[16 * b + i4 + 3], acc3);
                }
                X[t] = (acc0 + acc1) + (acc2 + acc3);
            }
            if (b < 3) { // publish the block as halves and add its contribution to the later rows
                u32x4 w0, w1;
                w0.x = pack_f16(X[16 * b + 0], X[16 * b + 1]); w0.y = pack_f16(X[16 * b + 2], X[16 * b + 3]);
                w0.z = pack_f16(X[16 * b + 4], X[16 * b + 5]); w0.w = pack_f16(X[16 * b + 6], X[16 * b + 7]);
                w1.x = pack_f16(X[16 * b + 8], X[16 * b + 9]); w1.y = pack_f16(X[16 * b + 10], X[16 * b + 11]);
                w1.z = pack_f16(X[16 * b + 12], X[16 * b + 13]); w1.w = pack_f16(X[16 * b + 14], X[16 * b + 15]);
                *reinterpret_cast<u32x4*>(wsc + lane * 48) = w0;
                *reinterpret_cast<u32x4*>(wsc + lane * 48 + 16) = w1;
                u32x4 xop[2];
#pragma unroll
                for (int ct = 0; ct < 2; ct++) xop[ct] = *reinterpret_cast<const u32x4*>(wsc + (32 * ct + n32) * 48 + 16 * half);
                const u32x4 aop1 = *reinterpret_cast<const u32x4*>(Ah + (32 + n32) * AHP + 16 * b + 8 * half);
#pragma unroll
                for (int ct = 0; ct < 2; ct++)
                    upd[ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, aop1), __builtin_bit_cast(f16x8, xop[ct]), upd[ct], 0, 0, 0);
                if (b == 0) { // rows 16 .. 31 are fed by block 0 alone: their tile lives only until it is handed over
                    const u32x4 aop0 = *reinterpret_cast<const u32x4*>(Ah + n32 * AHP + 8 * half);
#pragma unroll
                    for (int ct = 0; ct < 2; ct++) {
                        f32x16 u0;
#pragma unroll
                        for (int e = 0; e < 16; e++) u0[e] = 0.f;
                        u0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, aop0), __builtin_bit_cast(f16x8, xop[ct]), u0, 0, 0, 0);
                        hand_over(u0, ct, 8); // (the exchange area is free: both column tiles' operands are in registers)
                    }
                }
            }
        }
    }
    const float gC = g[GD_C - 1];
    const int sl = slot_of(col);
    // Kt, diag(e^g) Q and Kh^T are assembled in LDS in the image layout (the half copies of k and q are no longer
    // needed: the MFMAs are done), Vt in slot order as well, and leave in fragment order, 16 bytes a lane; element-wise
    // 2-byte stores to global would touch a different cache line per lane.
    uint16_t* khs = q16 + GD_C * (DK + 8); // [DK][64 + 8]
    __syncthreads();                       // every column is solved: the triangular matrix has been read for the last time
    uint16_t* vts = reinterpret_cast<uint16_t*>(Am); // V^T [DV][64] takes its place (the same 64 * DV * 2 bytes)
    if (tid < DV) { // holds the q column
#pragma unroll
        for (int q = 0; q < 8; q++) { // piece q: step q / 2, half q % 2; at a place of the row that spreads the rows over the banks
            const int t = 16 * (q >> 1) + 4 * (q & 1);
            u32x4 w;
            w.x = pack_f16(X[t], X[t + 1]); w.y = pack_f16(X[t + 2], X[t + 3]); w.z = pack_f16(X[t + 8], X[t + 9]); w.w = pack_f16(X[t + 10], X[t + 11]);
            *reinterpret_cast<u32x4*>(vts + col * GD_C + (q ^ (col & 7)) * 8) = w;
        }
#pragma unroll
        for (int t = 0; t < GD_C; t++) q16[t * (DK + 8) + sl] = f16_bits(eg[t] * colv[t]);
    } else { // holds the k column
#pragma unroll
        for (int t = 0; t < GD_C; t++) {
            k16[t * (DK + 8) + sl] = f16_bits(X[t]);
            khs[col * (GD_C + 8) + slot_of(t)] = f16_bits(egc[t] * colv[t]); // e^{g_C - g_t} k_t, token axis in slot order
        }
    }
    __syncthreads();
    {
        u32x4* d1 = reinterpret_cast<u32x4*>(img);
        for (int i = tid; i < 2 * 4 * JT * 64; i += NT) { // Kt and Qh: the rows of k16 and q16 follow one another
            const int f = i >> 6, l32 = i & 31, hh = (i >> 5) & 1, f1 = f % (4 * JT);
            d1[i] = *reinterpret_cast<const u32x4*>((f < 4 * JT ? k16 : q16) + (32 * (f1 / (2 * JT)) + l32) * (DK + 8) + 16 * (f1 % (2 * JT)) + 8 * hh);
        }
        for (int i = tid; i < 4 * JT * 64; i += NT) { // Kh^T and Vt^T
            const int f = i >> 6, l32 = i & 31, hh = (i >> 5) & 1, row = 32 * (f >> 2) + l32;
            d1[Lay::fKhT * 64 + i] = *reinterpret_cast<const u32x4*>(khs + row * (GD_C + 8) + 16 * (f & 3) + 8 * hh);
            d1[Lay::fVt * 64 + i] = *reinterpret_cast<const u32x4*>(vts + row * GD_C + ((2 * (f & 3) + hh) ^ (row & 7)) * 8);
        }
    }
    if (tid == 0) gCexp[(size_t)chunk * a.gdnHeads + h] = expf(gC);
}

// One wave per 32 state columns dv of a head: nothing of a chunk's products crosses columns, so the waves of a head are workgroups of their own, on
// different compute units.  An operand is used once by a wave: it comes from memory straight into registers, and the load of the next chunk's same
// operand goes out behind its use, a whole chunk ahead.  Bound by the MFMA chain of a chunk (56 a wave) where few heads times segments run, by the
// operands' way through the caches where many do.  Measured (head size 128): 13 chunks, 16 heads: 26 us (51 with the four waves of a head in one
// workgroup and the operands through LDS); 32 chunks, 8 x 16 heads: 95 us (122).
template <int DK>
__global__ void __launch_bounds__(64, 1) k_gdn_scan(PfArgs P, LayerDev L, const int* __restrict__ chunkBase, const unsigned char* __restrict__ ws,
                                                      const float* __restrict__ gCexp) {
    constexpr int DV = DK, JT = DK / 32; // dk tiles
    typedef GdLayout<DK> Lay;
    const StepArgs& a = P.a;
    const int h = blockIdx.x, seg = blockIdx.y, dt = blockIdx.z, lane = threadIdx.x;
    const int len = P.segLen[seg];
    if (len < GD_C) return; // short segments take the recurrent kernel
    const int seq = P.segSeq[seg], row0 = P.segStart[seg], nch = (len + GD_C - 1) / GD_C, cb = chunkBase[seg];
    const int n32 = lane & 31, half = lane >> 5, dv = 32 * dt + n32;
    float* Sg = L.S + ((size_t)seq * a.gdnHeads + h) * DV * DK;
    f32x16 St[JT]; // S^T tile j: rows dk = 32 j + 8(i/4) + 4 half + i%4, column dv
#pragma unroll
    for (int j = 0; j < JT; j++)
#pragma unroll
        for (int i = 0; i < 16; i++) St[j][i] = Sg[(size_t)dv * DK + 32 * j + 8 * (i >> 2) + 4 * half + (i & 3)];
    u32x4 kt[4 * JT], qh[4 * JT], mm[6], kh[4 * JT], vt[4]; // this chunk's fragments, each the next chunk's once it has been used
    auto frag = [&](int c, int f) __attribute__((always_inline)) {
        return reinterpret_cast<const u32x4*>(ws + ((size_t)(cb + c) * a.gdnHeads + h) * Lay::total + f * 1024)[lane];
    };
#pragma unroll
    for (int f = 0; f < 4 * JT; f++) { kt[f] = frag(0, Lay::fKt + f); qh[f] = frag(0, Lay::fQh + f); }
#pragma unroll
    for (int f = 0; f < 4; f++) vt[f] = frag(0, Lay::fVt + 4 * dt + f);
#pragma unroll
    for (int f = 0; f < 6; f++) mm[f] = frag(0, Lay::fM + f);
#pragma unroll
    for (int f = 0; f < 4 * JT; f++) kh[f] = frag(0, Lay::fKhT + f);
    auto mfma = [](const u32x4& x, const u32x4& y, const f32x16& z) __attribute__((always_inline)) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, x), __builtin_bit_cast(f16x8, y), z, 0, 0, 0);
    };
    float gC = gCexp[(size_t)cb * a.gdnHeads + h];
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0), as a builtin: the compiler then knows that no load from before the loop is open in it, and does not
    asm volatile("" ::: "memory");      // wait for the state at the head of every trip
    for (int c = 0; c < nch; c++) {
        const int cn = min(c + 1, nch - 1); // (behind the last chunk: that one again, dropped)
        const float gN = gCexp[(size_t)(cb + cn) * a.gdnHeads + h];
        // S0^T as B operands: step (j, st) = elements 8 st .. 8 st + 7 of tile j, rounded to half
        u32x4 sop[JT][2];
#pragma unroll
        for (int j = 0; j < JT; j++)
#pragma unroll
            for (int st = 0; st < 2; st++) {
                sop[j][st].x = pack_f16(St[j][8 * st + 0], St[j][8 * st + 1]); sop[j][st].y = pack_f16(St[j][8 * st + 2], St[j][8 * st + 3]);
                sop[j][st].z = pack_f16(St[j][8 * st + 4], St[j][8 * st + 5]); sop[j][st].w = pack_f16(St[j][8 * st + 6], St[j][8 * st + 7]);
            }
        // X = Kt S0^T : [64 tokens, 32 dv] (lane = dv), Y^T = S0 (diag(e^g) Q)^T : [32 dv, 64 tokens] (lane = token: the
        // operands swapped), so that an output row leaves as four neighbouring columns per store.
        f32x16 X[2], Y[2];
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
#pragma unroll
            for (int i = 0; i < 16; i++) { X[tt][i] = 0.f; Y[tt][i] = 0.f; }
#pragma unroll
            for (int j = 0; j < JT; j++)
#pragma unroll
                for (int st = 0; st < 2; st++) {
                    const int f = 2 * JT * tt + 2 * j + st;
                    X[tt] = mfma(kt[f], sop[j][st], X[tt]);
                    Y[tt] = mfma(sop[j][st], qh[f], Y[tt]);
                    kt[f] = frag(cn, Lay::fKt + f);
                    qh[f] = frag(cn, Lay::fQh + f);
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
        // W^T = Vt - X, as B operands (token axis in slot order by construction)
        u32x4 wop[2][2];
#pragma unroll
        for (int tt = 0; tt < 2; tt++)
#pragma unroll
            for (int st = 0; st < 2; st++) {
                const f16x8 v = __builtin_bit_cast(f16x8, vt[2 * tt + st]);
                float w[8];
#pragma unroll
                for (int e = 0; e < 8; e++) w[e] = (float)v[e] - X[tt][8 * st + e];
                wop[tt][st].x = pack_f16(w[0], w[1]); wop[tt][st].y = pack_f16(w[2], w[3]);
                wop[tt][st].z = pack_f16(w[4], w[5]); wop[tt][st].w = pack_f16(w[6], w[7]);
                vt[2 * tt + st] = frag(cn, Lay::fVt + 4 * dt + 2 * tt + st);
            }
        // O = Y + M W^T (M is lower triangular: tokens of tile 0 see only tile 0)
#pragma unroll
        for (int tt = 0; tt < 2; tt++)
#pragma unroll
            for (int t2 = 0; t2 <= tt; t2++)
#pragma unroll
                for (int st = 0; st < 2; st++) {
                    Y[tt] = mfma(wop[t2][st], mm[2 * (tt + t2) + st], Y[tt]);
                    mm[2 * (tt + t2) + st] = frag(cn, Lay::fM + 2 * (tt + t2) + st);
                }
        __builtin_amdgcn_sched_barrier(0);
        // S^T <- e^{g_C} S^T + Kh^T W^T
#pragma unroll
        for (int j = 0; j < JT; j++)
#pragma unroll
            for (int i = 0; i < 16; i++) St[j][i] *= gC;
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int j = 0; j < JT; j++) {
                St[j] = mfma(kh[4 * j + s], wop[s >> 1][s & 1], St[j]);
                kh[4 * j + s] = frag(cn, Lay::fKhT + 4 * j + s);
            }
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
            // lane = token n32 of this tile; element i = column 32 dt + 8 (i / 4) + 4 half + i % 4.  The two lanes of a
            // token (half 0 and 1) swap two of their four 8-byte pieces so that each holds two whole 16-byte pieces:
            // half as many store instructions, and the address unit works through a store per lane and instruction.
            u32x2 w[4];
#pragma unroll
            for (int g = 0; g < 4; g++) {
                w[g].x = pack_half_range(Y[tt][4 * g], Y[tt][4 * g + 1]); w[g].y = pack_half_range(Y[tt][4 * g + 2], Y[tt][4 * g + 3]);
            }
            // half 0 keeps pieces g = 0, 2 (and gets the partner's upper halves of them), half 1 keeps g = 1, 3
            u32x2 give[2], got[2];
            give[0] = half ? w[0] : w[1]; give[1] = half ? w[2] : w[3];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                got[k].x = (uint32_t)__shfl_xor((int)give[k].x, 32, 64);
                got[k].y = (uint32_t)__shfl_xor((int)give[k].y, 32, 64);
            }
            if (n32 < len - (c * GD_C + 32 * tt)) {
                f16_t* orow = (f16_t*)P.Amix + (size_t)(row0 + c * GD_C + 32 * tt + n32) * P.aLd + h * DV + 32 * dt + 8 * half;
#pragma unroll
                for (int k = 0; k < 2; k++) { // columns 16 k + 8 half .. + 7: lower four from the half-0 lane, upper four from the half-1 lane
                    const u32x2 mine = half ? w[2 * k + 1] : w[2 * k];
                    u32x4 v;
                    v.x = half ? got[k].x : mine.x; v.y = half ? got[k].y : mine.y;
                    v.z = half ? mine.x : got[k].x; v.w = half ? mine.y : got[k].y;
                    *reinterpret_cast<u32x4*>(orow + 16 * k) = v;
                }
            }
        }
        gC = gN;
    }
#pragma unroll
    for (int j = 0; j < JT; j++)
#pragma unroll
        for (int i = 0; i < 16; i++) Sg[(size_t)dv * DK + 32 * j + 8 * (i >> 2) + 4 * half + (i & 3)] = St[j][i];
}

// The same with one wave per 16 columns, on 16 x 16 x 32 products, where few heads times segments run: half the products, packing and outputs of a chunk
// on a wave's chain, for twice the operands' way through the caches.  The operand image is the one above.  Its pieces hold the contraction's elements
// {4 hh .. 4 hh + 3, 8 + 4 hh .. + 3} of step st; lane (n, q) takes those of st = q / 2, hh = q % 2, which makes row 4 q + i of a 16-row tile number
// 16 (q / 2) + 4 (q % 2) + i of its 32 (tile 0 of a pair) or 8 more (tile 1): the state's dk and X's tokens are kept in that order, so that they are
// operands as they stand here too.  Measured (head size 128, 13 chunks): 16 heads 16.8 us (26.2 with 32 columns a wave), 4 x 16 heads 24.4 (27.5).
template <int DK>
__global__ void __launch_bounds__(64, 1) k_gdn_scan16(PfArgs P, LayerDev L, const int* __restrict__ chunkBase, const unsigned char* __restrict__ ws,
                                                        const float* __restrict__ gCexp) {
    constexpr int DV = DK, JT = DK / 32;
    typedef GdLayout<DK> Lay;
    const StepArgs& a = P.a;
    const int h = blockIdx.x, seg = blockIdx.y, dt = blockIdx.z, lane = threadIdx.x, n = lane & 15, q = lane >> 4;
    const int len = P.segLen[seg];
    if (len < GD_C) return; // short segments take the recurrent kernel
    const int seq = P.segSeq[seg], row0 = P.segStart[seg], nch = (len + GD_C - 1) / GD_C, cb = chunkBase[seg];
    auto place = [](int x) { return 16 * (x >> 3) + 4 * ((x >> 2) & 1) + (x & 3); }; // row x of a pair's first tile among its 32
    unsigned offR[2], offN[2]; // this lane's piece: rows in that order (tile of the pair), columns in their own (half of the 32)
#pragma unroll
    for (int t = 0; t < 2; t++) {
        offR[t] = (q >> 1) * 1024 + ((q & 1) * 32 + place(n) + 8 * t) * 16;
        offN[t] = (q >> 1) * 1024 + ((q & 1) * 32 + n + 16 * t) * 16;
    }
    float* Srow = L.S + (((size_t)seq * a.gdnHeads + h) * DV + 16 * dt + n) * DK + place(4 * q);
    f32x4 St[JT][2]; // S^T: rows dk = 32 j + place(4 q) + 8 t + i, column dv = 16 dt + n
#pragma unroll
    for (int j = 0; j < JT; j++)
#pragma unroll
        for (int t = 0; t < 2; t++) St[j][t] = *reinterpret_cast<const f32x4*>(Srow + 32 * j + 8 * t);
    u32x4 kt[2][2][JT], qh[4][JT], mm[3][2], kh[JT][2][2], vt[2]; // this chunk's pieces, each the next chunk's once it has been used
    auto frag = [&](int c, int f, unsigned off) __attribute__((always_inline)) {
        return *reinterpret_cast<const u32x4*>(ws + ((size_t)(cb + c) * a.gdnHeads + h) * Lay::total + f * 1024 + off);
    };
    auto get_kt = [&](int c, int u, int t, int j) __attribute__((always_inline)) { return frag(c, Lay::fKt + u * 2 * JT + 2 * j, offR[t]); };
    auto get_qh = [&](int c, int v, int j) __attribute__((always_inline)) { return frag(c, Lay::fQh + (v >> 1) * 2 * JT + 2 * j, offN[v & 1]); };
    auto get_mm = [&](int c, int p, int o) __attribute__((always_inline)) { return frag(c, Lay::fM + 2 * p, offN[o]); };
    auto get_kh = [&](int c, int j, int t, int u) __attribute__((always_inline)) { return frag(c, Lay::fKhT + 4 * j + 2 * u, offR[t]); };
    const unsigned offV = (dt >> 1) * 4096 + ((dt & 1) ? offN[1] : offN[0]);
    auto get_vt = [&](int c, int u) __attribute__((always_inline)) { return frag(c, Lay::fVt + 2 * u, offV); };
    auto mfma = [](const u32x4& x, const u32x4& y, const f32x4& z) __attribute__((always_inline)) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x), __builtin_bit_cast(f16x8, y), z, 0, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < JT; j++)
#pragma unroll
        for (int v = 0; v < 4; v++) { kt[v >> 1][v & 1][j] = get_kt(0, v >> 1, v & 1, j); qh[v][j] = get_qh(0, v, j); kh[j][v & 1][v >> 1] = get_kh(0, j, v & 1, v >> 1); }
#pragma unroll
    for (int u = 0; u < 2; u++) vt[u] = get_vt(0, u);
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
        for (int o = 0; o < 2; o++) mm[p][o] = get_mm(0, p, o);
    float gC = gCexp[(size_t)cb * a.gdnHeads + h];
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0), as a builtin: as above
    asm volatile("" ::: "memory");
    for (int c = 0; c < nch; c++) {
        const int cn = min(c + 1, nch - 1); // (behind the last chunk: that one again, dropped)
        const float gN = gCexp[(size_t)(cb + cn) * a.gdnHeads + h];
        u32x4 sop[JT];
#pragma unroll
        for (int j = 0; j < JT; j++) {
            sop[j].x = pack_f16(St[j][0].x, St[j][0].y); sop[j].y = pack_f16(St[j][0].z, St[j][0].w);
            sop[j].z = pack_f16(St[j][1].x, St[j][1].y); sop[j].w = pack_f16(St[j][1].z, St[j][1].w);
        }
        f32x4 X[2][2], Y[4]; // X = Kt S0^T: [tokens 32 u + .., dv];  Y^T = S0 (diag(e^g) Q)^T: [dv, tokens 16 v + ..]
#pragma unroll
        for (int v = 0; v < 4; v++) { X[v >> 1][v & 1] = (f32x4)(0.f); Y[v] = (f32x4)(0.f); }
#pragma unroll
        for (int j = 0; j < JT; j++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                X[v >> 1][v & 1] = mfma(kt[v >> 1][v & 1][j], sop[j], X[v >> 1][v & 1]);
                kt[v >> 1][v & 1][j] = get_kt(cn, v >> 1, v & 1, j);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        u32x4 wop[2]; // W^T = Vt - X
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const f16x8 v = __builtin_bit_cast(f16x8, vt[u]);
            wop[u].x = pack_f16((float)v[0] - X[u][0].x, (float)v[1] - X[u][0].y); wop[u].y = pack_f16((float)v[2] - X[u][0].z, (float)v[3] - X[u][0].w);
            wop[u].z = pack_f16((float)v[4] - X[u][1].x, (float)v[5] - X[u][1].y); wop[u].w = pack_f16((float)v[6] - X[u][1].z, (float)v[7] - X[u][1].w);
            vt[u] = get_vt(cn, u);
        }
        // S^T <- e^{g_C} S^T + Kh^T W^T: what the next chunk waits for
#pragma unroll
        for (int j = 0; j < JT; j++)
#pragma unroll
            for (int t = 0; t < 2; t++) St[j][t] *= gC;
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int j = 0; j < JT; j++)
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    St[j][t] = mfma(kh[j][t][u], wop[u], St[j][t]);
                    kh[j][t][u] = get_kh(cn, j, t, u);
                }
        __builtin_amdgcn_sched_barrier(0);
        // O = Y + M W^T (M is lower triangular: tokens of the first 32 see only those)
#pragma unroll
        for (int j = 0; j < JT; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                Y[v] = mfma(sop[j], qh[v][j], Y[v]);
                qh[v][j] = get_qh(cn, v, j);
            }
#pragma unroll
        for (int p = 0; p < 3; p++) // (0, 0), (1, 0), (1, 1)
#pragma unroll
            for (int o = 0; o < 2; o++) {
                const int v = (p ? 2 : 0) + o;
                Y[v] = mfma(wop[p >> 1], mm[p][o], Y[v]);
                mm[p][o] = get_mm(cn, p, o);
            }
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (n < len - (c * GD_C + 16 * v))
                put4<f16_t>((f16_t*)P.Amix + (size_t)(row0 + c * GD_C + 16 * v + n) * P.aLd + h * DV + 16 * dt + 4 * q, Y[v].x, Y[v].y, Y[v].z, Y[v].w);
        gC = gN;
    }
#pragma unroll
    for (int j = 0; j < JT; j++)
#pragma unroll
        for (int t = 0; t < 2; t++) *reinterpret_cast<f32x4*>(Srow + 32 * j + 8 * t) = St[j][t];
}

// fp32 models: the row of mixing output (floats, from several workgroups) and its PLE columns as pairs (h2.h) and the row's exponent, in place: 32
// columns take 128 bytes either way, and a block's eight lanes read it in an instruction before the one that writes it; or as planes (p3.h), to Xn.  A wave a
// row; up to 256 KEEP columns stay in registers between the maximum and the split.
template <typename T, int KEEP>
__global__ void __launch_bounds__(PWG) k_pf_operand_rows(PfArgs P, LayerDev L) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, cols = L.ad + P.a.ple;
    if (row >= P.n) return;
    float* x = (float*)P.Amix + (size_t)row * P.aLd;
    const float* gate = P.QKV + (size_t)row * P.qkvLd + L.offPle;
    const float* table = (const float*)L.pleTable + (size_t)P.ids[row] * P.a.ple;
    auto value = [&](int i) {
        if (i < L.ad) return *reinterpret_cast<const f32x4*>(x + i);
        const int j = i - L.ad;
        return f32x4{pf_silu(gate[j]) * table[j], pf_silu(gate[j + 1]) * table[j + 1], pf_silu(gate[j + 2]) * table[j + 2], pf_silu(gate[j + 3]) * table[j + 3]};
    };
    if constexpr (__is_same(T, p3_t)) {
        for (int i = lane * 4; i < cols; i += 256) {
            const f32x4 v = value(i);
            put4_at<p3_t>(P.Xn, (size_t)row, P.aLd, i, v.x, v.y, v.z, v.w);
        }
        return;
    }
    f32x4 keep[KEEP];
    int most = -100000;
#pragma unroll
    for (int k = 0; k < KEEP; k++) keep[k] = value(min(lane * 4 + k * 256, cols - 4));
#pragma unroll
    for (int k = 0; k < KEEP; k++) most = max(most, h2_size4(keep[k].x, keep[k].y, keep[k].z, keep[k].w));
    for (int i = lane * 4 + KEEP * 256; i < cols; i += 256) {
        const f32x4 v = value(i);
        most = max(most, h2_size4(v.x, v.y, v.z, v.w));
    }
    const int e = h2_exponent(pf_wave_max(most));
    if (lane == 0) P.exps[row] = e;
    auto store = [&](int i, const f32x4& v) { h2_put4<false>(x, i, ldexpf(v.x, -e), ldexpf(v.y, -e), ldexpf(v.z, -e), ldexpf(v.w, -e)); };
#pragma unroll
    for (int k = 0; k < KEEP; k++)
        if (lane * 4 + k * 256 < cols) store(lane * 4 + k * 256, keep[k]);
    for (int i = lane * 4 + KEEP * 256; i < cols; i += 256) store(i, value(i));
}

// Exponents of the FFN units' columns, a wave each: |x / rms| <= sqrt(d), so by Cauchy and Schwarz a gate or up value is at most sqrt(d) |row (.) gain| and the
// unit, |silu(g)| <= |g|, the product of the two.  It is brought under 2^15; the largest half is twice that.
__global__ void __launch_bounds__(PWG) k_unit_exps(const float* __restrict__ W13, const float* __restrict__ gain, int* exps, int units, int d) {
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (j >= units) return;
    const float *g = W13 + (size_t)2 * j * d, *u = g + d;
    double sg = 0.0, su = 0.0;
    for (int i = lane; i < d; i += 64) {
        const double a = (double)g[i] * gain[i], b = (double)u[i] * gain[i];
        sg += a * a; su += b * b;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { sg += __shfl_xor(sg, o, 64); su += __shfl_xor(su, o, 64); }
    const double bound = (double)d * sqrt(sg) * sqrt(su);
    if (lane == 0) exps[j] = bound > 0.0 ? __builtin_amdgcn_frexp_exp(bound) - 15 : 0;
}

// One workgroup per segment: argmax over the LM head's partial maxima of its last row (lowest index on ties); the
// sequence's length advances by the segment's.  picks: pinned host memory, by sequence.
__global__ void __launch_bounds__(PWG) k_pf_finish(PfArgs P, int nparts, int* picks) {
    __shared__ float sv[PWG];
    __shared__ int si[PWG];
    __shared__ double sd[PWG + 1];
    const StepArgs& a = P.a;
    const int tid = threadIdx.x, seg = blockIdx.x;
    if (P.n < MLH_PREFILL_GEMM_MIN_ROWS && a.temperature > 0.f) { // short calls draw, as the decode step they take the place of does
        const int seq = P.segSeq[seg], end = P.segPos0[seg] + P.segLen[seg];
        const int nxt = mlh_sample_row<PWG>(a.logits + (size_t)seq * a.vocab, a.vocab, a.temperature, mlh_sample_uniform(a.sampleSeed, seq, end), sd, si);
        if (tid == 0) { a.nextTok[seq] = nxt; picks[seq] = nxt; a.pos[seq] = end; }
        return;
    }
    float v = -3.0e38f;
    int idx = 0x7fffffff;
    for (int i = tid; i < nparts; i += PWG) {
        const float v2 = a.amaxVal[(size_t)seg * a.amaxParts + i];
        const int i2 = a.amaxIdx[(size_t)seg * a.amaxParts + i];
        if (v2 > v || (v2 == v && i2 < idx)) { v = v2; idx = i2; }
    }
    sv[tid] = v; si[tid] = idx;
    __syncthreads();
    for (int s = PWG / 2; s > 0; s >>= 1) {
        if (tid < s && (sv[tid + s] > sv[tid] || (sv[tid + s] == sv[tid] && si[tid + s] < si[tid]))) { sv[tid] = sv[tid + s]; si[tid] = si[tid + s]; }
        __syncthreads();
    }
    if (tid == 0) {
        int nxt = si[0];
        if (nxt < 0 || nxt >= a.vocab) nxt = 0; // only reachable with non-finite logits
        const int seq = P.segSeq[seg];
        a.nextTok[seq] = nxt;
        picks[seq] = nxt;
        a.pos[seq] += P.segLen[seg];
    }
}

// Row-wise softmax over the vocabulary (inference.cu:293-362) and the cross-entropy of the next token:
// probs[row] = softmax(logits[row]); nll[row] = -log max(probs[row][target[row]], 1e-4), the clamp of
// training_orchestrator.cu:343-347 (target < 0: none).
// A workgroup takes a row and keeps it in registers, NR elements a thread, all asked for at once: what bounds it is the way to memory and back, and one pass
// less makes half of it.  Measured (rows of 20 224): 84 of them 9.8 us, 517 26.2;
// three passes of 256 threads, an element at a time, took 51.5 and 82.9.
// Longer rows than 32 x 1024 are read again in every pass.
#define SMT 1024
__device__ __forceinline__ float sm_block_sum(float v, float* red, int lane, int wave) {
    v = pf_wave_sum(v);
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < SMT / 64; w++) s += red[w];
    return s;
}
template <int NR> // 0: any length
__global__ void __launch_bounds__(SMT) k_pf_softmax_rows(const float* __restrict__ logits, float* __restrict__ probs, const int* __restrict__ target, float* __restrict__ nll, int V) {
    __shared__ float red[2][SMT / 64];
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float* lg = logits + (size_t)row * V;
    const float at = nll && tid == 0 && target[row] >= 0 ? lg[target[row]] : 0.f;
    float x[NR ? NR : 1] = {}, m = -3.0e38f;
    if (NR) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(lg), 0, V * 4, 0x00027000);
#pragma unroll
        for (int j = 0; j < NR; j++) x[j] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (unsigned)(tid + j * SMT) * 4u, 0, 0));
#pragma unroll
        for (int j = 0; j < NR; j++)
            if (tid + j * SMT < V) m = fmaxf(m, x[j]);
    } else {
#pragma unroll 4
        for (int i = tid; i < V; i += SMT) m = fmaxf(m, lg[i]);
    }
    m = pf_wave_max(m);
    if (lane == 0) red[0][wave] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < SMT / 64; w++) m = fmaxf(m, red[0][w]);
    float sum = 0.f;
    if (NR) {
#pragma unroll
        for (int j = 0; j < NR; j++) {
            x[j] = tid + j * SMT < V ? expf(x[j] - m) : 0.f;
            sum += x[j];
        }
    } else {
#pragma unroll 4
        for (int i = tid; i < V; i += SMT) sum += expf(lg[i] - m);
    }
    sum = sm_block_sum(sum, red[1], lane, wave);
    if (probs) {
        float* pr = probs + (size_t)row * V;
        if (NR) {
#pragma unroll
            for (int j = 0; j < NR; j++)
                if (tid + j * SMT < V) pr[tid + j * SMT] = x[j] / sum;
        } else {
#pragma unroll 4
            for (int i = tid; i < V; i += SMT) pr[i] = expf(lg[i] - m) / sum;
        }
    }
    if (nll && tid == 0) nll[row] = target[row] >= 0 ? -logf(fmaxf(expf(at - m) / sum, 0.0001f)) : 0.f;
}

int mlh_launch_softmax_rows(mlh_ctx* c, const float* logits, float* probs, const int* target, float* nll, int rows) {
    const int V = c->hp.vocabSize;
#define SOFTMAX_ROWS(NR_) hipLaunchKernelGGL((k_pf_softmax_rows<NR_>), dim3(rows), dim3(SMT), 0, c->stream, logits, probs, target, nll, V)
    if (V <= 8 * SMT) SOFTMAX_ROWS(8);
    else if (V <= 20 * SMT) SOFTMAX_ROWS(20);
    else if (V <= 32 * SMT) SOFTMAX_ROWS(32);
    else SOFTMAX_ROWS(0);
#undef SOFTMAX_ROWS
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { c->err = std::string("softmax launch: ") + hipGetErrorString(e); return -2; }
    return 0;
}

// ----------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------
static int cdiv(int a, int b) { return (a + b - 1) / b; }

bool mlh_prefill_gemm_supported(const mlh_ctx* c) { return c->operands; }

// widths that the MFMA kernels take: whole chunks of 128 bytes
static bool operand_widths(const mlh_ctx* c) {
    const mlh_hparams& hp = c->hp;
    const int esz = c->wbytes, kmul = 128 / esz;
    if (hp.dim % kmul || hp.ffnDim % kmul || (hp.pleDim && hp.pleDim % kmul)) return false;
    for (const LayerDev& L : c->layers)
        if (L.ad % kmul) return false;
    return true;
}

// ---- fp16 operands of the MFMA path for bf16 models ----
// A bf16 value has 8 significand bits, an IEEE half 11: scaled by a power of two that brings the
// matrix's largest magnitude just under the half range, every weight down to 2^-29 of that maximum
// converts exactly, so the MFMA path multiplies the very bf16-rounded weights the GEMV path reads --
// but against activations that keep 11 significand bits instead of 8.  (Accumulation is fp32 either way.)
__global__ void k_absmax_bf16(const bf16_t* __restrict__ w, size_t n, unsigned* out) {
    unsigned m = 0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) m = max(m, (unsigned)(w[i] & 0x7fffu));
    for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
    if ((threadIdx.x & 63) == 0 && m) atomicMax(out, m);
}
__global__ void k_bf16_to_f16(const bf16_t* __restrict__ w, f16_t* __restrict__ out, size_t n, float scale, unsigned* inexact) {
    unsigned bad = 0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float v = __uint_as_float(((uint32_t)w[i]) << 16) * scale;
        const _Float16 h = (_Float16)v;
        out[i].bits = __builtin_bit_cast(uint16_t, h);
        bad += ((float)h != v);
    }
    if (bad) atomicAdd(inexact, bad);
}

int mlh_operand_alloc(mlh_ctx* c, void** p, size_t bytes) {
    const hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) { (void)hipGetLastError(); return MLH_NO_ROOM; }
    MLH_CHECK(c, e);
    c->mirrorAllocs.push_back(*p);
    c->operandBytes += bytes;
    return 0;
}

static int build_mirror(mlh_ctx* c, const void* src, size_t n, const void** dst, float* alpha, unsigned* d_scratch) {
    void* buf = nullptr;
    if (const int rc = mlh_operand_alloc(c, &buf, n * 2)) return rc;
    MLH_CHECK(c, hipMemsetAsync(d_scratch, 0, 8, c->stream));
    hipLaunchKernelGGL(k_absmax_bf16, dim3(1024), dim3(256), 0, c->stream, (const bf16_t*)src, n, d_scratch);
    unsigned h[2] = {0, 0};
    MLH_CHECK(c, hipMemcpyAsync(h, d_scratch, 4, hipMemcpyDeviceToHost, c->stream));
    MLH_CHECK(c, hipStreamSynchronize(c->stream));
    // largest magnitude = bf16 bits h[0]; its exponent e (unbiased): scale 2^(14 - e) puts it in [2^14, 2^15)
    const int e = (int)((h[0] >> 7) & 0xff) - 127;
    const int k = h[0] ? 14 - e : 0;
    const float scale = ldexpf(1.0f, k);
    hipLaunchKernelGGL(k_bf16_to_f16, dim3(1024), dim3(256), 0, c->stream, (const bf16_t*)src, (f16_t*)buf, n, scale, d_scratch + 1);
    MLH_CHECK(c, hipMemcpyAsync(h, d_scratch, 8, hipMemcpyDeviceToHost, c->stream));
    MLH_CHECK(c, hipStreamSynchronize(c->stream));
    c->f16Inexact += h[1];
    *dst = buf;
    *alpha = ldexpf(1.0f, -k);
    return 0;
}

// Sets *found when the magnitude of one of n elements (as bits: infinities and NaN are the largest) reaches `limit`.
template <typename WT>
__global__ void __launch_bounds__(256) k_find_beyond(const uint4* __restrict__ w, size_t n, uint32_t limit, unsigned* found) {
    const size_t n16 = n / (16 / sizeof(WT));
    bool any = false;
    if (sizeof(WT) == 4 && blockIdx.x == 0 && threadIdx.x < n - n16 * 4) any = (reinterpret_cast<const uint32_t*>(w)[n16 * 4 + threadIdx.x] & 0x7fffffffu) >= limit; // (a gate bias per head)
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += (size_t)gridDim.x * 256) {
        const uint4 v = w[i];
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (sizeof(WT) == 4) any = any || (x[e] & 0x7fffffffu) >= limit;
            else any = any || (x[e] & 0x7fffu) >= limit || (x[e] >> 16 & 0x7fffu) >= limit;
        }
    }
    if (any) *found = 1;
}

// Whether the MFMA kernels may multiply this model's matrices.  Their products are sums over planes (of the activations, and of fp32
// weights) or of scaled halves, which an infinite operand turns into NaN where inf * x is infinite; the GEMV and
// single-launch kernels multiply in fp32 and keep it.  So no weight may lie beyond the planes, and no gain above 2^60: rows
// are multiplied by it before they are normalised, and their squares overflow from 2^64 on.  Nor may a per-layer embedding lie beyond the planes
// (what it scales is multiplied by PLE up), or a gate bias above 2^60: the chunked delta rule adds up logarithms of decays and takes
// differences of the sums.  One pass over the weights per finalize.
static int operand_values(mlh_ctx* c, bool* within) {
    const mlh_hparams& hp = c->hp;
    const size_t d = hp.dim, F = hp.ffnDim, pl = hp.pleDim;
    unsigned* found = nullptr;
    unsigned h = 0;
    MLH_CHECK(c, hipMalloc((void**)&found, 4));
    hipError_t e = hipMemsetAsync(found, 0, 4, c->stream);
    auto matrix = [&](const void* w, size_t n) { // (rows are multiples of 128 bytes)
        if (c->wbytes == 4) hipLaunchKernelGGL((k_find_beyond<float>), dim3(2048), dim3(256), 0, c->stream, (const uint4*)w, n, P3_BEYOND, found);
        else hipLaunchKernelGGL((k_find_beyond<bf16_t>), dim3(2048), dim3(256), 0, c->stream, (const uint4*)w, n, 0x7f80u, found);
    };
    auto vector = [&](const float* g, size_t n) { hipLaunchKernelGGL((k_find_beyond<float>), dim3(4), dim3(256), 0, c->stream, (const uint4*)g, n, 0x5d800000u, found); };
    matrix(c->E, (size_t)hp.vocabSize * d);
    vector(c->gF, d);
    for (const LayerDev& L : c->layers) {
        matrix(L.Wa, L.rowsA * d); matrix(L.Wo, d * L.ad); matrix(L.W13, 2 * F * d); matrix(L.W2, d * F);
        if (pl) { matrix(L.pleUp, d * pl); matrix(L.pleTable, (size_t)hp.vocabSize * pl); }
        vector(L.g1, d); vector(L.g2, d);
        if (L.gq) { vector(L.gq, d); vector(L.gk, d); }
        if (L.gdnBa) { vector(L.gdnBa, hp.gdnHeads); vector(L.gdnBb, hp.gdnHeads); }
    }
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(&h, found, 4, hipMemcpyDeviceToHost, c->stream);
    const hipError_t e2 = hipStreamSynchronize(c->stream);
    (void)hipFree(found);
    MLH_CHECK(c, e);
    MLH_CHECK(c, e2);
    *within = h == 0;
    return 0;
}

// Whether scaled halves reach over an fp32 model's operands.  A row of halves ends 2^-39 below its largest element (h2.h), where floats and planes end
// at 2^-126: elements far below the largest are kept in fewer bits, and where the large ones meet zeros the sum is made of those.  So
//   - a row of weights has its typical element (mean of the exponents, zeros apart) within 2^12 of its largest: with its columns' scales in W2, whose
//     columns the units' exponents go into;
//   - the rows that are multiplied have theirs within 2^8, as far as that follows from the model: residual columns (E's columns, rows of [Wo | pleUp] and W2, each
//     about its own mean) with the gain in front of a product; value rows and PLE columns (gate row and table) beside each other;
//   - an FFN unit, whose scale comes from its bound, is dim below that on rows without a direction; on rows as uneven as the residual columns at most 2^4 more.
// What is lost at 2^-39 of the largest is then 2^-27 of a typical weight, 2^-31 of a typical element of a row, 2^-24 of a typical unit (dim 2048).
// Models beyond multiply planes.  Normally distributed weights have 4 or 5, 1 and 1 octaves.  Exponents and integer sums: the answer is the same at every finalize.
#define SPREAD_WEIGHTS 12
#define SPREAD_ROWS 8
#define SPREAD_UNITS 4
#define SPREAD_NONE (-100000)
__device__ __forceinline__ void spread_worst(int* worst, int v) { // (a row that does not add to it leaves the word alone: one address for all)
    if (v > __hip_atomic_load(worst, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(worst, v);
}
// the exponents of rows of [W | U] with those of the columns: the largest of each row to rowMost, and the largest distance of one from its row's mean to worst
__global__ void __launch_bounds__(PWG) k_spread_rows(const float* __restrict__ W, int cols, const float* __restrict__ U, int cols2, const int* __restrict__ colExps, int* rowMost, int* worst, int rows) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    int most = SPREAD_NONE, sum = 0, count = 0;
    for (int i = lane; i < cols + cols2; i += 64) {
        const float x = i < cols ? W[(size_t)row * cols + i] : U[(size_t)row * cols2 + i - cols];
        if (x == 0.f) continue;
        const int e = h2_size(x) + (colExps ? colExps[i] : 0);
        most = max(most, e); sum += e; count++;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { most = max(most, __shfl_xor(most, o, 64)); sum += __shfl_xor(sum, o, 64); count += __shfl_xor(count, o, 64); }
    if (lane) return;
    if (rowMost) rowMost[row] = most;
    if (count) spread_worst(worst, most - (int)floorf((float)sum / (float)count));
}
// ... the largest of each column to colMost (x: columns, y: strips of rows)
__global__ void __launch_bounds__(PWG) k_spread_cols(const float* __restrict__ W, int rows, int cols, int* colMost) {
    const int col = blockIdx.x * PWG + threadIdx.x, strip = (rows + gridDim.y - 1) / gridDim.y, end = min(rows, (int)(blockIdx.y + 1) * strip);
    if (col >= cols) return;
    int most = SPREAD_NONE;
    for (int r = blockIdx.y * strip; r < end; r++) most = max(most, h2_size(W[(size_t)r * cols + col]));
    atomicMax(colMost + col, most);
}
// ... and how far a unit's bound lies above dim times its size on rows of elements `like`, of mean square 1 (a power of two, the largest to worst)
__global__ void __launch_bounds__(PWG) k_spread_units(const float* __restrict__ W13, const float* __restrict__ gain, const float* __restrict__ like, int* worst, int units, int d) {
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (j >= units) return;
    const float *g = W13 + (size_t)2 * j * d, *u = g + d;
    double s[4] = {};
    for (int i = lane; i < d; i += 64) {
        const double a = (double)g[i] * gain[i], b = (double)u[i] * gain[i], x = like[i];
        s[0] += a * a; s[1] += b * b; s[2] += a * a * x * x; s[3] += b * b * x * x;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int k = 0; k < 4; k++) s[k] += __shfl_xor(s[k], o, 64);
    if (lane || s[0] == 0.0 || s[1] == 0.0) return; // (a unit that is always 0)
    const double size = sqrt(s[2]) * sqrt(s[3]);
    spread_worst(worst, size > 0.0 ? __builtin_amdgcn_frexp_exp(sqrt(s[0]) * sqrt(s[1]) / size) : -SPREAD_NONE);
}
static int spread_mean(const int* v, int n) { // rounded down; of the elements there are
    long sum = 0, count = 0;
    for (int i = 0; i < n; i++)
        if (v[i] > SPREAD_NONE / 2) { sum += v[i]; count++; }
    return count ? (int)floor((double)sum / (double)count) : SPREAD_NONE;
}
static bool spread_even(const std::vector<int>& v) {
    const int mean = spread_mean(v.data(), (int)v.size());
    return mean == SPREAD_NONE || *std::max_element(v.begin(), v.end()) - mean <= SPREAD_ROWS;
}
static int operand_spread(mlh_ctx* c, bool* within) {
    const mlh_hparams& hp = c->hp;
    const int d = hp.dim, F = hp.ffnDim, p = hp.pleDim, V = hp.vocabSize, n = (int)c->layers.size(), per = c->maxRowsA + p + 2 * d;
    // ints: the worst row, E's columns, units; a layer's rows of Wa, table columns, rows of [Wo | pleUp] and W2
    const size_t ints = 1 + 2 * (size_t)d + F + (size_t)n * per; // (at the end floats: a row like the residual's)
    int* dev = nullptr;
    std::vector<int> h(ints);
    std::vector<float> gains((size_t)(2 * n + 1) * d);
    MLH_CHECK(c, hipMalloc((void**)&dev, ints * 4));
    hipError_t e = hipMemsetAsync(dev, 0x80, ints * 4, c->stream); // (far below SPREAD_NONE)
    int *const worst = dev, *const colE = dev + 1, *const units = colE + d, *const first = units + F;
    float* const like = (float*)(first + (size_t)n * per);
    auto rows = [&](const void* W, int cols, const void* U, int cols2, const int* colExps, int* most, int count) {
        hipLaunchKernelGGL(k_spread_rows, dim3(cdiv(count, 4)), dim3(PWG), 0, c->stream, (const float*)W, cols, (const float*)U, cols2, colExps, most, worst, count);
    };
    auto cols = [&](const void* W, int count, int width, int* most) { hipLaunchKernelGGL(k_spread_cols, dim3(cdiv(width, PWG), 64), dim3(PWG), 0, c->stream, (const float*)W, count, width, most); };
    rows(c->E, d, nullptr, 0, nullptr, nullptr, V);
    cols(c->E, V, d, colE);
    for (int t = 0; t < n; t++) {
        const LayerDev& L = c->layers[t];
        int *a = first + (size_t)t * per, *table = a + c->maxRowsA, *o = table + p, *w2 = o + d;
        rows(L.Wa, d, nullptr, 0, nullptr, a, L.rowsA);
        rows(L.Wo, L.ad, L.pleUp, p, nullptr, o, d);
        rows(L.W13, d, nullptr, 0, nullptr, nullptr, 2 * F);
        hipLaunchKernelGGL(k_unit_exps, dim3(cdiv(F, 4)), dim3(PWG), 0, c->stream, (const float*)L.W13, L.g2, units, F, d);
        rows(L.W2, F, nullptr, 0, units, w2, d);
        if (p) { rows(L.pleTable, p, nullptr, 0, nullptr, nullptr, V); cols(L.pleTable, V, p, table); }
        if (e == hipSuccess) e = hipMemcpyAsync(gains.data() + (size_t)2 * t * d, L.g1, (size_t)d * 4, hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipMemcpyAsync(gains.data() + (size_t)(2 * t + 1) * d, L.g2, (size_t)d * 4, hipMemcpyDeviceToHost, c->stream);
    }
    if (e == hipSuccess) e = hipMemcpyAsync(gains.data() + (size_t)2 * n * d, c->gF, (size_t)d * 4, hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(h.data(), dev, ints * 4, hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    bool ok = h[0] <= SPREAD_WEIGHTS;
    std::vector<int> resid(d, SPREAD_NONE); // how far a residual column may lie above the others
    auto contributes = [&](const int* v) {
        const int mean = spread_mean(v, d);
        for (int j = 0; j < d; j++)
            if (v[j] > SPREAD_NONE / 2) resid[j] = std::max(resid[j], v[j] - mean);
    };
    contributes(h.data() + 1);
    for (int t = 0; t < n; t++) {
        const LayerDev& L = c->layers[t];
        const int *a = h.data() + (first - dev) + (size_t)t * per, *table = a + c->maxRowsA, *o = table + p, *w2 = o + d;
        contributes(o);
        contributes(w2);
        std::vector<int> mix(a + L.offV, a + L.offV + L.ad);
        for (int j = 0; j < p; j++) mix.push_back(a[L.offPle + j] > SPREAD_NONE / 2 && table[j] > SPREAD_NONE / 2 ? a[L.offPle + j] + table[j] : SPREAD_NONE);
        ok = ok && spread_even(mix);
    }
    for (int g = 0; g < 2 * n + 1; g++) {
        std::vector<int> x(d, SPREAD_NONE);
        for (int j = 0; j < d; j++) {
            const float v = gains[(size_t)g * d + j];
            int ex = 0;
            (void)frexpf(v, &ex);
            if (v != 0.f && resid[j] > SPREAD_NONE / 2) x[j] = ex + resid[j];
        }
        ok = ok && spread_even(x);
    }
    if (e == hipSuccess && ok) {
        const int most = *std::max_element(resid.begin(), resid.end());
        std::vector<float> row(d);
        double ss = 0.0;
        for (int j = 0; j < d; j++) { const double x = resid[j] > SPREAD_NONE / 2 ? ldexp(1.0, resid[j] - most) : 0.0; row[j] = (float)x; ss += x * x; }
        for (float& x : row) x = ss > 0.0 ? (float)(x / sqrt(ss / d)) : 1.f;
        e = hipMemcpyAsync(like, row.data(), (size_t)d * 4, hipMemcpyHostToDevice, c->stream);
        if (e == hipSuccess) e = hipMemsetAsync(worst, 0, 4, c->stream);
        for (const LayerDev& L : c->layers) hipLaunchKernelGGL(k_spread_units, dim3(cdiv(F, 4)), dim3(PWG), 0, c->stream, (const float*)L.W13, L.g2, (const float*)like, worst, F, d);
        if (e == hipSuccess) e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(h.data(), worst, 4, hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        ok = h[0] <= SPREAD_UNITS;
    }
    (void)hipStreamSynchronize(c->stream);
    (void)hipFree(dev);
    MLH_CHECK(c, e);
    *within = ok;
    return 0;
}

// An fp32 matrix as three bf16 planes or as triples of halves, what the tiled products of the prefill multiply.
static int build_planes(mlh_ctx* c, const void* src, int rows, int cols, const void** dst) {
    void* buf = nullptr;
    if (const int rc = mlh_operand_alloc(c, &buf, (size_t)rows * cols * 6)) return rc;
    MLH_CHECK(c, mlh_split_p3(c->stream, (const float*)src, cols, buf, cols, rows, cols));
    *dst = buf;
    return 0;
}
static int build_triples(mlh_ctx* c, const void* src, int rows, int cols, const int* colExps, const void** dst, const int** exps) {
    void *buf = nullptr, *e = nullptr;
    int rc;
    if ((rc = mlh_operand_alloc(c, &buf, (size_t)rows * cols * 6)) || (rc = mlh_operand_alloc(c, &e, (size_t)rows * 4))) return rc;
    MLH_CHECK(c, mlh_split_h2(c->stream, true, (const float*)src, cols, buf, cols, colExps, (int*)e, rows, cols));
    *dst = buf;
    *exps = (const int*)e;
    return 0;
}

// A chunk's operands of all heads (bf16 models with gated-delta-net layers; else 0).
static size_t gdn_chunk_bytes(const mlh_ctx* c) {
    const mlh_hparams& hp = c->hp;
    if (hp.weightDtype != MLH_DTYPE_BF16) return 0;
    for (const LayerDev& L : c->layers)
        if (L.kind == MLH_KIND_GDN) return (size_t)hp.gdnHeads * ((hp.gdnDk == 64 ? GdLayout<64>::total : GdLayout<128>::total) + 4);
    return 0;
}
// Elements of the products' inputs: halves, pairs of them or planes; of the mixing output, which becomes planes in Xn; columns of Xn.
static size_t input_bytes(const mlh_ctx* c) { return c->hp.weightDtype == MLH_DTYPE_BF16 ? 2 : c->pfDtype == MLH_GEMM_P3 ? 6 : 4; }
static size_t mix_bytes(const mlh_ctx* c) { return std::min<size_t>(input_bytes(c), 4); }
static size_t xn_cols(const mlh_ctx* c) { return c->pfDtype == MLH_GEMM_P3 ? std::max(c->hp.dim, c->maxAd + c->hp.pleDim) : c->hp.dim; }
// Work buffers of a prefill call: per row, and of the chunks that segments of 64 rows or more are cut into (ensure_prefill_buffers).
static size_t prefill_row_bytes(const mlh_ctx* c) {
    const mlh_hparams& hp = c->hp;
    const size_t wb = input_bytes(c), d = hp.dim;
    return d * (8 + (wb == 2 ? 4 : 0)) + xn_cols(c) * wb + (size_t)c->maxRowsA * 4 + ((size_t)c->maxAd + hp.pleDim) * mix_bytes(c) + hp.ffnDim * wb + 68;
}
// ... of one over every position of the context, with the products' split-K workspace.
size_t mlh_prefill_work_bytes(const mlh_ctx* c) {
    const size_t rows = (size_t)c->hp.maxSeqs * c->hp.maxL, chunks = (size_t)c->hp.maxSeqs * cdiv(c->hp.maxL, GD_C);
    return rows * prefill_row_bytes(c) + chunks * gdn_chunk_bytes(c) + mlh_gemm_workspace_bytes();
}

// Whether the copies fit: into the caller's limit, and onto the device with room left for a prefill call over every position of the
// context or, if that is less, a sixteenth of the device's memory.  Without them a model of which only the matrices
// fit still runs (they take 2.5 times the matrices' bytes in fp32, twice in bf16, [Wo | pleUp] once more).
static int operand_room(mlh_ctx* c, bool* fits) {
    const mlh_hparams& hp = c->hp;
    const size_t d = hp.dim, F = hp.ffnDim, pl = hp.pleDim, wb = c->wbytes, per = wb == 4 ? 10 : 4;
    auto rows16 = [](size_t n) { return (n + 15) / 16 * 16; };
    const size_t exps = c->pfDtype == MLH_GEMM_H2 ? 4 : 0; // of every row, and of the FFN units
    size_t need = rows16(hp.vocabSize) * d * per + hp.vocabSize * exps;
    for (const LayerDev& L : c->layers)
        need += (rows16(L.rowsA) * d + rows16(d) * (L.ad + pl) + rows16(2 * F) * d + rows16(d) * F) * per + (pl ? d * (L.ad + pl) * wb : 0) + (L.rowsA + 2 * d + 3 * F) * exps;
    size_t free = 0, total = 0;
    MLH_CHECK(c, hipMemGetInfo(&free, &total));
    const size_t have = c->pfRows * prefill_row_bytes(c) + c->pfGdnChunks * gdn_chunk_bytes(c) + (c->gemmWs ? mlh_gemm_workspace_bytes() : 0); // (of earlier calls)
    const size_t work = std::min(mlh_prefill_work_bytes(c), total / 16);
    *fits = need <= c->operandLimit && need + (work > have ? work - have : 0) <= free;
    return 0;
}

void mlh_drop_operands(mlh_ctx* c) {
    c->operands = false;
    for (void* p : c->mirrorAllocs) (void)hipFree(p);
    c->mirrorAllocs.clear();
    c->operandBytes = 0;
    for (LayerDev& L : c->layers) L.eWa = L.eWo = L.eW13 = L.eW2 = L.eU = nullptr, L.WaP = L.WoP = L.W13P = L.W2P = L.WaR = L.WoR = L.W13R = L.W2R = nullptr;
    c->EP = c->ER = nullptr;
    c->eE = nullptr;
}

// The halves or planes; on MLH_NO_ROOM what has been allocated so far is still there.
static int build_operands(mlh_ctx* c, unsigned* d_scratch) {
    const mlh_hparams& hp = c->hp;
    const bool mirror = hp.weightDtype == MLH_DTYPE_BF16;
    const size_t d = hp.dim, F = hp.ffnDim, pl = hp.pleDim, wb = c->wbytes;
    int rc = 0;
    for (LayerDev& L : c->layers) {
        L.sWa = L.sWo = L.sW13 = L.sW2 = 1.0f;
        const void* wo = L.Wo;
        if (pl > 0) { // [Wo | pleUp] along K, in the storage type
            void* cat = nullptr;
            if ((rc = mlh_operand_alloc(c, &cat, d * (L.ad + pl) * wb))) return rc;
            MLH_CHECK(c, hipMemcpy2D(cat, (L.ad + pl) * wb, L.Wo, L.ad * wb, L.ad * wb, d, hipMemcpyDeviceToDevice));
            MLH_CHECK(c, hipMemcpy2D((char*)cat + L.ad * wb, (L.ad + pl) * wb, L.pleUp, pl * wb, pl * wb, d, hipMemcpyDeviceToDevice));
            wo = cat;
        }
        L.WoR = wo;
        if (mirror) {
            if ((rc = build_mirror(c, L.Wa, (size_t)L.rowsA * d, &L.WaP, &L.sWa, d_scratch)) ||
                (rc = build_mirror(c, wo, d * (L.ad + pl), &L.WoP, &L.sWo, d_scratch)) ||
                (rc = build_mirror(c, L.W13, 2 * F * d, &L.W13P, &L.sW13, d_scratch)) ||
                (rc = build_mirror(c, L.W2, d * F, &L.W2P, &L.sW2, d_scratch)))
                return rc;
        } else if (c->pfDtype == MLH_GEMM_P3) {
            if ((rc = build_planes(c, L.Wa, L.rowsA, (int)d, &L.WaP)) || (rc = build_planes(c, wo, (int)d, L.ad + (int)pl, &L.WoP)) ||
                (rc = build_planes(c, L.W13, 2 * (int)F, (int)d, &L.W13P)) || (rc = build_planes(c, L.W2, (int)d, (int)F, &L.W2P)))
                return rc;
        } else {
            void* units = nullptr;
            if ((rc = mlh_operand_alloc(c, &units, F * 4))) return rc;
            hipLaunchKernelGGL(k_unit_exps, dim3(cdiv((int)F, 4)), dim3(PWG), 0, c->stream, (const float*)L.W13, L.g2, (int*)units, (int)F, (int)d);
            MLH_CHECK(c, hipGetLastError());
            L.eU = (const int*)units;
            if ((rc = build_triples(c, L.Wa, L.rowsA, (int)d, nullptr, &L.WaP, &L.eWa)) || (rc = build_triples(c, wo, (int)d, L.ad + (int)pl, nullptr, &L.WoP, &L.eWo)) ||
                (rc = build_triples(c, L.W13, 2 * (int)F, (int)d, nullptr, &L.W13P, &L.eW13)) || (rc = build_triples(c, L.W2, (int)d, (int)F, L.eU, &L.W2P, &L.eW2)))
                return rc;
        }
    }
    c->sE = 1.0f;
    return mirror ? build_mirror(c, c->E, (size_t)hp.vocabSize * hp.dim, &c->EP, &c->sE, d_scratch) :
           c->pfDtype == MLH_GEMM_P3 ? build_planes(c, c->E, hp.vocabSize, hp.dim, &c->EP) : build_triples(c, c->E, hp.vocabSize, hp.dim, nullptr, &c->EP, &c->eE);
}

static void drop_prefill_buffers(mlh_ctx* c) { // (hipFree waits for the device)
    for (void* p : c->pfAllocs) (void)hipFree(p);
    c->pfAllocs.clear();
    c->pfRows = 0;
}

int mlh_build_gemm_operands(mlh_ctx* c) {
    mlh_drop_operands(c); // a repeated finalize rebuilds them
    c->f16Inexact = 0;
    if (!operand_widths(c)) return 0;
    int rc = 0;
    bool ok = false, halves = true;
    if ((rc = operand_values(c, &ok)) || !ok) return rc;
    if (c->wbytes == 4 && (rc = operand_spread(c, &halves))) return rc;
    const int form = c->wbytes == 2 ? MLH_GEMM_F16 : halves ? MLH_GEMM_H2 : MLH_GEMM_P3;
    if (form != c->pfDtype) drop_prefill_buffers(c); // (their rows' size follows from it)
    c->pfDtype = form;
    if ((rc = operand_room(c, &ok)) || !ok) return rc;
    unsigned* d_scratch = nullptr;
    MLH_CHECK(c, hipMalloc((void**)&d_scratch, 8));
    rc = build_operands(c, d_scratch);
    (void)hipFree(d_scratch);
    if (rc == 0) rc = mlh_rows_prepare(c);
    if (rc) mlh_drop_operands(c);
    c->operands = rc == 0;
    return rc == MLH_NO_ROOM ? 0 : rc; // (another context or process took the room in between)
}

// The headDim-128 attention tiles exceed the 64 KB a launch may use without opting in.
static size_t gdn_prep_lds(int dk) { return ((size_t)GD_C * GD_C + 12 * GD_C) * 4 + (size_t)2 * GD_C * (dk + 8) * 2 + (size_t)dk * (GD_C + 8) * 2; }

int mlh_init_prefill_kernels(mlh_ctx* c) {
    MLH_CHECK(c, hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gdn_prep<64>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)gdn_prep_lds(64)));
    MLH_CHECK(c, hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gdn_prep<128>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)gdn_prep_lds(128)));
    return 0;
}

static int ensure_prefill_buffers(mlh_ctx* c, int rows) {
    if (rows <= c->pfRows) return 0;
    const mlh_hparams& hp = c->hp;
    (void)hipStreamSynchronize(c->stream);
    drop_prefill_buffers(c);
    const size_t n = (size_t)rows, wb = input_bytes(c);
    auto alloc = [&](void** p, size_t bytes) -> int {
        MLH_CHECK(c, hipMalloc(p, std::max<size_t>(bytes, 16)));
        c->pfAllocs.push_back(*p);
        return 0;
    };
    int rc;
    const size_t nblk = cdiv(rows, PF_QB) + hp.maxSeqs, nchunk = cdiv(rows, GD_C) + hp.maxSeqs;
    const size_t meta = 3 * n + 5 * (size_t)hp.maxSeqs + 2 * nblk + 2 * nchunk; // ids, sequence and position of every row; segments; attention blocks; GDN chunks
    if ((rc = alloc((void**)&c->pfX, n * hp.dim * 4)) || (rc = alloc(&c->pfXn, n * xn_cols(c) * wb)) ||
        (rc = alloc((void**)&c->pfQKV, n * c->maxRowsA * 4)) || (rc = alloc(&c->pfA, n * (c->maxAd + hp.pleDim) * mix_bytes(c))) ||
        (rc = alloc((void**)&c->pfH1, n * hp.dim * 4)) || (rc = alloc((void**)&c->pfExp, n * 4)) ||
        (rc = alloc(&c->pfU, n * hp.ffnDim * wb)) ||
        (hp.weightDtype == MLH_DTYPE_BF16 && ((rc = alloc((void**)&c->pfKh, n * hp.dim * 2)) || (rc = alloc((void**)&c->pfVh, n * hp.dim * 2)))) ||
        (rc = alloc((void**)&c->pfMeta, meta * 4)))
        return rc;
    if ((rc = mlh_pin(c, c->pinMeta, meta * 4)) || (rc = mlh_pin(c, c->pinNext, (size_t)hp.maxSeqs * 4))) return rc;
    c->pfRows = rows;
    return 0;
}

// Split-K workspace of the GEMMs; its launches are ordered on the context's stream.
static int ensure_gemm_workspace(mlh_ctx* c) {
    if (c->gemmWs) return 0;
    void* ws = nullptr;
    MLH_CHECK(c, hipMalloc(&ws, mlh_gemm_workspace_bytes()));
    c->allocs.push_back(ws);
    MLH_CHECK(c, hipMemset(ws, 0, mlh_gemm_workspace_bytes()));
    c->gemmWs = ws;
    return 0;
}

#define PF_DISPATCH_WT(c, expr_f32, expr_bf16) do { if ((c)->hp.weightDtype == MLH_DTYPE_BF16) { expr_bf16; } else { expr_f32; } } while (0)

// Calls of up to this many tokens run through the row kernels: fewer launches (norms and embedding ride along) and, for bf16
// models, fp32 precision of the activations.  Measured against the tiled products (us per call): 12 fp32 layers of dim 768, 5 / 16 / 64
// tokens 461 / 510 / 771 -- 672 / 724 / 1012, and beyond 64 rows the weights would be fetched once more; 24 bf16 layers of dim 2048,
// 16 / 32 / 48 tokens 1511 / 2155 / 3767 -- 1953 / 2255 / 2723: three plane products against one of halves.
#define MLH_ROWS_PREFILL_F32 64
#define MLH_ROWS_PREFILL_BF16 32
bool mlh_prefill_by_rows(const mlh_ctx* c, int tokens) { return tokens <= (c->hp.weightDtype == MLH_DTYPE_F32 ? MLH_ROWS_PREFILL_F32 : MLH_ROWS_PREFILL_BF16); }

// Appends lens[s] tokens to sequence seqs[s] for every segment s (token ids concatenated in `ids`).
// allLogits: null, or a device buffer [rows, vocab] that receives the logits of every position.
int mlh_run_prefill_gemm(mlh_ctx* c, int nseg, const int32_t* seqs, const int32_t* ids, const int32_t* lens, float* allLogits) {
    const mlh_hparams& hp = c->hp;
    int n = 0;
    for (int s = 0; s < nseg; s++) n += lens[s];
    int rc = ensure_prefill_buffers(c, n);
    if (rc == 0) rc = ensure_gemm_workspace(c);
    if (rc) return rc;
    const bool rowsPath = mlh_prefill_by_rows(c, n);
    // ---- metadata: laid out in pinned memory as on the device, one copy ----
    // bf16 models: fp16 MFMA attention, 128 queries per workgroup; below 16 tokens as precise as the token-by-token path
    const bool mfmaAttn = hp.weightDtype == MLH_DTYPE_BF16 && n >= MLH_PREFILL_GEMM_MIN_ROWS;
    const int qb = mfmaAttn ? PF_MQB : PF_QB;
    bool anyGdn = false, fresh = true; // fresh: every segment starts its sequence, all keys of the call are rows of the call
    for (const LayerDev& L : c->layers) anyGdn = anyGdn || L.kind == MLH_KIND_GDN;
    const bool gdnChunked = anyGdn && c->pfDtype == MLH_GEMM_F16 && !rowsPath; // segments of 64 tokens or more: chunk-parallel MFMA path
    int nblk = 0, nchunk = 0, chunked = 0; // chunked: segments on that path
    for (int s = 0; s < nseg; s++) {
        nblk += cdiv(lens[s], qb);
        if (gdnChunked && lens[s] >= GD_C) { nchunk += cdiv(lens[s], GD_C); chunked++; }
    }
    int* const h = c->pinMeta.p;
    int *h_ids = h, *h_rowSeq = h + n, *h_rowPos = h + 2 * n, *h_seg = h + 3 * n, *h_blk = h_seg + 5 * nseg, *h_chunk = h_blk + 2 * nblk;
    const size_t metaInts = (size_t)(h_chunk - h) + 2 * (size_t)nchunk;
    memcpy(h_ids, ids, (size_t)n * 4);
    for (int s = 0, r = 0, b = 0, k = 0; s < nseg; s++) { // segStart, segLen, segSeq, segPos0, chunkBase; blkSeg, blkQ0; chunkSeg, chunkT0
        const int pos0 = c->h_len[seqs[s]];
        h_seg[s] = r; h_seg[nseg + s] = lens[s]; h_seg[2 * nseg + s] = seqs[s]; h_seg[3 * nseg + s] = pos0; h_seg[4 * nseg + s] = k;
        fresh = fresh && pos0 == 0;
        for (int q0 = 0; q0 < lens[s]; q0 += qb, b++) { h_blk[b] = s; h_blk[nblk + b] = q0; }
        if (gdnChunked && lens[s] >= GD_C)
            for (int t0 = 0; t0 < lens[s]; t0 += GD_C, k++) { h_chunk[k] = s; h_chunk[nchunk + k] = t0; }
        for (int i = 0; i < lens[s]; i++, r++) { h_rowSeq[r] = seqs[s]; h_rowPos[r] = pos0 + i; }
    }
    if (nchunk > 0) {
        const size_t per = (size_t)hp.gdnHeads * (hp.gdnDk == 64 ? GdLayout<64>::total : GdLayout<128>::total);
        if ((size_t)nchunk > c->pfGdnChunks) {
            MLH_CHECK(c, hipStreamSynchronize(c->stream));
            if (c->pfGdnWs) { (void)hipFree(c->pfGdnWs); (void)hipFree(c->pfGdnG); c->pfGdnWs = nullptr; c->pfGdnG = nullptr; c->pfGdnChunks = 0; }
            MLH_CHECK(c, hipMalloc(&c->pfGdnWs, (size_t)nchunk * per));
            MLH_CHECK(c, hipMalloc((void**)&c->pfGdnG, (size_t)nchunk * hp.gdnHeads * 4));
            c->pfGdnChunks = nchunk;
        }
    }
    int* d = c->pfMeta;
    int *d_seg = d + 3 * n, *d_blk = d_seg + 5 * nseg, *d_chunk = d_blk + 2 * nblk;
    hipStream_t st = c->stream;
    MLH_CHECK(c, hipMemcpyAsync(d, h, metaInts * 4, hipMemcpyHostToDevice, st)); // (the call ends with a synchronisation: the pinned copy is free again)

    PfArgs P;
    mlh_fill_args(c, P.a, nseg, c->d_tok);
    P.n = n; P.nseg = nseg; P.ids = d; P.rowSeq = d + n; P.rowPos = d + 2 * n;
    P.segStart = d_seg; P.segLen = d_seg + nseg; P.segSeq = d_seg + 2 * nseg; P.segPos0 = d_seg + 3 * nseg;
    P.blkSeg = d_blk; P.blkQ0 = d_blk + nblk;
    P.X = c->pfX; P.Xn = c->pfXn; P.QKV = c->pfQKV; P.qkvLd = c->maxRowsA; P.Amix = c->pfA; P.aLd = c->maxAd + hp.pleDim;
    P.H1 = c->pfH1; P.U = c->pfU; P.exps = c->pfExp;
    P.Kh = mfmaAttn && fresh ? c->pfKh : nullptr;
    P.Vh = mfmaAttn && fresh ? c->pfVh : nullptr;
    P.lay = rows_layout(std::min(n, 64)); P.rows = rowsPath ? c->rowsMix : nullptr; P.half = hp.weightDtype == MLH_DTYPE_BF16;
    RowsArgs base = {};
    base.M = n; base.lay = P.lay; base.normDim = hp.dim;
    const int d_ = hp.dim, F = hp.ffnDim, dt = c->pfDtype;
    // Up to 64 rows of halves are one row of 64 x 64 tiles: their two groups of waves keep four stages in flight, where a wave of the weight-streaming kernel (what
    // mlh_gemm_tn_epi takes) has one chunk.  Whole prefills, 24 layers of width 2048, us: 33 rows 2237 -> 1756, 48 2406 -> 1819, 64 2707 -> 2002 (65: 2084).
    // (FFN units go through the hardware's exp2 and reciprocal in tiles, through expf and a division in that kernel: both 2.085e-4 of their norm from float64, K 2048.)
    auto* const product = dt == MLH_GEMM_F16 && n <= 64 ? mlh_gemm_tile : mlh_gemm_tn_epi;
#define GEMM(A, lda, eA, B, alpha, eB, ldb, C, ldc, R, ldr, M, N, K)                                                           \
    do {                                                                                                                     \
        hipError_t e_ = product(st, dt, 0, A, lda, B, ldb, C, ldc, R, ldr, M, N, K, c->gemmWs, alpha, eA, eB, nullptr); \
        if (e_ != hipSuccess) { c->err = std::string("prefill GEMM: ") + hipGetErrorString(e_); return -2; } \
    } while (0)

#define NORM(X_, gain_)                                                                                                        \
    do {                                                                                                                     \
        if (dt == MLH_GEMM_F16) launch_rmsnorm<f16_t>(st, X_, gain_, P.Xn, nullptr, n, d_);                                   \
        else if (dt == MLH_GEMM_P3) launch_rmsnorm<p3_t>(st, X_, gain_, P.Xn, nullptr, n, d_);                                \
        else launch_rmsnorm<h2_t>(st, X_, gain_, P.Xn, P.exps, n, d_);                                                        \
    } while (0)
    const int pleWgs = hp.pleDim > 0 && (P.half || rowsPath) ? 1 : 0; // a row's (segment's, chunk's) workgroup for the PLE columns

    if (rowsPath) mlh_rows_embed(c, P.ids, n, P.X, P.lay);
    else PF_DISPATCH_WT(c, hipLaunchKernelGGL((k_pf_embed<float>), dim3(cdiv(d_, PWG), n), dim3(PWG), 0, st, P),
                   hipLaunchKernelGGL((k_pf_embed<bf16_t>), dim3(cdiv(d_, PWG), n), dim3(PWG), 0, st, P));
    for (int t = hp.transformers - 1; t >= 0; t--) { // file block 0 is the top (inference.cu:384-385)
        const LayerDev& L = c->layers[t];
        if (rowsPath) {
            RowsArgs R = base;
            R.K = d_; R.A = c->rowsX; R.ssqIn = c->rowsSsqX; R.nparts = t == hp.transformers - 1 ? 1 : d_ / RW_TILE; R.C = P.QKV; R.ldc = P.qkvLd;
            mlh_rows_gemm(c, RW_PLAIN, L.WaR, L.rowsA, R);
        } else {
            NORM(P.X, L.g1);
            GEMM(P.Xn, d_, P.exps, L.WaP, L.sWa, L.eWa, d_, P.QKV, P.qkvLd, nullptr, 0, n, L.rowsA, d_);
        }
        if (L.kind == MLH_KIND_ATTENTION) {
#define ATTN_ROWS(HD_, AT_)                                                                                                    \
    do {                                                                                                                     \
        if (hp.attnHeads * nblk <= c->numCUs) hipLaunchKernelGGL((k_pf_attn<HD_, 8, AT_>), dim3(hp.attnHeads, nblk), dim3(512), 0, st, P, L); \
        else hipLaunchKernelGGL((k_pf_attn<HD_, 4, AT_>), dim3(hp.attnHeads, nblk), dim3(256), 0, st, P, L);                 \
    } while (0)
            if (hp.headDim == 64) {
                hipLaunchKernelGGL((k_pf_qk_rope_kv<64>), dim3(hp.attnHeads + pleWgs, n), dim3(64), 0, st, P, L);
                if (mfmaAttn && P.Kh) hipLaunchKernelGGL((k_pf_attn_mfma<64, true>), dim3(hp.attnHeads, nblk), dim3(PWG), 0, st, P, L);
                else if (mfmaAttn) hipLaunchKernelGGL((k_pf_attn_mfma<64, false>), dim3(hp.attnHeads, nblk), dim3(PWG), 0, st, P, L);
                else if (P.half) ATTN_ROWS(64, f16_t);
                else ATTN_ROWS(64, float);
            } else {
                hipLaunchKernelGGL((k_pf_qk_rope_kv<128>), dim3(hp.attnHeads + pleWgs, n), dim3(64), 0, st, P, L);
                if (mfmaAttn && P.Kh) hipLaunchKernelGGL((k_pf_attn_mfma<128, true>), dim3(hp.attnHeads, nblk), dim3(PWG), 0, st, P, L);
                else if (mfmaAttn) hipLaunchKernelGGL((k_pf_attn_mfma<128, false>), dim3(hp.attnHeads, nblk), dim3(PWG), 0, st, P, L);
                else if (P.half) ATTN_ROWS(128, f16_t);
                else ATTN_ROWS(128, float);
            }
        } else {
            const int skipFrom = gdnChunked ? GD_C : 0x7fffffff;
            // 32 state rows a workgroup up to two heads a compute unit: half the products of a token on a wave's chain.  Measured (heads of 64; us, 64 and 32
            // rows): 12 heads x 1 segment 44, 34; x 5 66, 47; x 19 101, 82; x 32 177, 141; x 64 215, 222.
            if (chunked < nseg) { // (a launch whose workgroups all return takes 4.7 us a layer)
                const bool half = hp.weightDtype == MLH_DTYPE_BF16, few = hp.gdnHeads * nseg <= 2 * c->numCUs;
#define RECUR(DK_, GR_, AT_) hipLaunchKernelGGL((k_pf_gdn<DK_, GR_, AT_>), dim3(hp.gdnHeads + pleWgs, nseg, DK_ / GR_), dim3(PWG), 0, st, P, L, skipFrom)
#define RECUR_ROWS(DK_, AT_) do { if (few) RECUR(DK_, 32, AT_); else RECUR(DK_, 64, AT_); } while (0)
                if (hp.gdnDk == 64) { if (half) RECUR_ROWS(64, f16_t); else RECUR_ROWS(64, float); }
                else { if (half) RECUR_ROWS(128, f16_t); else RECUR_ROWS(128, float); }
#undef RECUR_ROWS
#undef RECUR
            }
            if (nchunk > 0) {
                const int *dcs = d_chunk, *dct = d_chunk + nchunk, *dcb = d_seg + 4 * nseg;
                // 16 columns a wave up to two waves a compute unit (4 segments of 16 heads of 128: 24.4 us, 27.5 with 32 columns); beyond, the operands'
                // second way through the caches costs more than the shorter chain gives (8 segments: 51, 41).
                const bool narrow = hp.gdnHeads * chunked * (hp.gdnDv / 16) <= 2 * c->numCUs;
#define SCAN(K_, DK_, W_) hipLaunchKernelGGL((K_<DK_>), dim3(hp.gdnHeads, nseg, DK_ / W_), dim3(64), 0, st, P, L, dcb, (const unsigned char*)c->pfGdnWs, c->pfGdnG)
                if (hp.gdnDk == 64) {
                    hipLaunchKernelGGL((k_gdn_prep<64>), dim3(nchunk, hp.gdnHeads + pleWgs), dim3(128), gdn_prep_lds(64), st, P, L, dcs, dct, (unsigned char*)c->pfGdnWs, c->pfGdnG);
                    if (narrow) SCAN(k_gdn_scan16, 64, 16);
                    else SCAN(k_gdn_scan, 64, 32);
                } else {
                    hipLaunchKernelGGL((k_gdn_prep<128>), dim3(nchunk, hp.gdnHeads + pleWgs), dim3(256), gdn_prep_lds(128), st, P, L, dcs, dct, (unsigned char*)c->pfGdnWs, c->pfGdnG);
                    if (narrow) SCAN(k_gdn_scan16, 128, 16);
                    else SCAN(k_gdn_scan, 128, 32);
#undef SCAN
                }
            }
        }
        if (!P.half && !rowsPath) {
            const int cols = L.ad + hp.pleDim;
            if (dt == MLH_GEMM_P3) hipLaunchKernelGGL((k_pf_operand_rows<p3_t, 1>), dim3(cdiv(n, 4)), dim3(PWG), 0, st, P, L);
            else if (cols <= 1024) hipLaunchKernelGGL((k_pf_operand_rows<h2_t, 4>), dim3(cdiv(n, 4)), dim3(PWG), 0, st, P, L);
            else hipLaunchKernelGGL((k_pf_operand_rows<h2_t, 8>), dim3(cdiv(n, 4)), dim3(PWG), 0, st, P, L);
        }
        if (rowsPath) {
            mlh_rows_rest_of_layer(c, t, base, P.X, P.H1);
            continue;
        }
        GEMM(dt == MLH_GEMM_P3 ? P.Xn : P.Amix, P.aLd, P.exps, L.WoP, L.sWo, L.eWo, L.ad + hp.pleDim, P.H1, d_, P.X, d_, n, d_, L.ad + hp.pleDim); // Wo . a + pleUp . e + x
        NORM(P.H1, L.g2);
        { // gate/up projection with SiLU(gate) * up in the epilogue (inference.cu:262-281): U comes out in the GEMM input type
            hipError_t e_ = product(st, dt, 1, P.Xn, d_, L.W13P, d_, P.U, F, nullptr, 0, n, 2 * F, d_, c->gemmWs, L.sW13, P.exps, L.eW13, L.eU);
            if (e_ != hipSuccess) { c->err = std::string("prefill GEMM: ") + hipGetErrorString(e_); return -2; }
        }
        GEMM(P.U, F, nullptr, L.W2P, L.sW2, L.eW2, F, P.X, d_, P.H1, d_, n, d_, F);
    }
#undef GEMM
    if (allLogits && rowsPath) { // tied LM head of every normalised row (inference.cu:705-743 computes all L columns)
        RowsArgs R = base;
        R.K = d_; R.A = c->rowsX; R.ssqIn = c->rowsSsqX; R.nparts = d_ / RW_TILE; R.C = allLogits; R.ldc = hp.vocabSize;
        mlh_rows_gemm(c, RW_PLAIN, c->ER, hp.vocabSize, R);
    } else if (allLogits) {
        NORM(P.X, c->gF);
        hipError_t e_ = product(st, dt, 0, P.Xn, d_, c->EP, d_, allLogits, hp.vocabSize, nullptr, 0, n, hp.vocabSize, d_, c->gemmWs, c->sE, P.exps, c->eE, nullptr);
        if (e_ != hipSuccess) { c->err = std::string("prefill GEMM: ") + hipGetErrorString(e_); return -2; }
    }
    for (int s0 = 0; s0 < nseg; s0 += 64)
        mlh_rows_lm_head(c, std::min(64, nseg - s0), P.X, P.segStart + s0, P.segLen + s0, P.segSeq + s0, c->amaxVal + (size_t)s0 * c->amaxParts, c->amaxIdx + (size_t)s0 * c->amaxParts);
    hipLaunchKernelGGL(k_pf_finish, dim3(nseg), dim3(PWG), 0, st, P, cdiv(hp.vocabSize, RW_TILE), c->pinNext.p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { c->err = std::string("prefill launch: ") + hipGetErrorString(e); return -2; }
    MLH_CHECK(c, hipStreamSynchronize(st));
    for (int s = 0; s < nseg; s++) {
        c->h_len[seqs[s]] += lens[s];
        c->h_next[seqs[s]] = c->pinNext.p[seqs[s]];
        c->h_nextKnown[seqs[s]] = 1;
    }
    return 0;
}
