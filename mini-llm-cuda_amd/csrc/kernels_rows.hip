// The products of a decode step and of short prefills: C[M, N] = A[M, K] . W[N, K]^T for at most 64 rows of A, fp32 or bf16
// weights packed once into the order the waves fetch them in (rows.h), at fp32 precision.
//
// Every weight is read once and the activations once per workgroup, so a product is a launch, a memory latency and the bytes
// behind it; the arithmetic must not add to that.  A workgroup of eight waves owns 16 weight rows at a time and MB blocks of
// tokens; the waves split K in chunks of 128 bytes per weight row and multiply straight from registers on
// v_mfma_f32_16x16x32_bf16: the activations come as three bf16 planes in operand order (rows.h, written by whichever kernel
// produced them), fp32 weights are split into planes in registers (six plane products, as in p3.h), bf16 weights are one plane
// (three products); the eight partial sums meet in LDS.  Two forms: k_rows keeps its activations in registers while it walks several
// tiles of weight rows, the next tile's weights on their way (K of up to CNT chunks per wave); k_rows_long streams both (long K,
// which is the down projection with its few rows).  Measured (launch included, us): d 768, 5 fp32 sequences: first phase 5.5, output
// projection 5.4, gate / up 6.5, down 7.7 -- 12.7, 11.5, 12.9, 14.4 as GEMVs over groups of four sequences; 64 sequences 7.7, 5.2,
// 10.1, 7.6 -- 10.6, 10, 10.6, 14 through the fp32 matrix cores with rows of 16 lines per fetch; d 2048, 8 bf16 sequences 9.2, 6.3,
// 12.3 (46 MB: 3.7 TB/s), 13.2 -- 10.4, 8.5, 15.5, 16 with activations rounded to half.
//
// RMSNorm rides along: the kernel that writes a residual row also writes the planes of gain (.) row for the product that follows and, per
// workgroup, the row's partial sum of squares; the product adds those up (in order) and scales its result by 1 / rms.
#include <algorithm>

#include "mlh_internal.h"
#include "rows.h"
#include "rows_mul.h"
#include "sample.h"

#define RW_WAVES 8
#define RW_THREADS (RW_WAVES * 64)
// the activations of a chunk: [32-wide step][plane][token block]
template <typename WT, int MB> struct RowsA {
    u32x4 v[RowsW<WT>::SUB][3][MB];
    __device__ __forceinline__ void load(const unsigned char* chunk, int stride, int block) {
#pragma unroll
        for (int s = 0; s < RowsW<WT>::SUB; s++)
#pragma unroll
            for (int pl = 0; pl < 3; pl++)
#pragma unroll
                for (int mb = 0; mb < MB; mb++) v[s][pl][mb] = *reinterpret_cast<const u32x4*>(chunk + (s * 3 + pl) * stride + mb * block);
    }
};
__device__ __forceinline__ const unsigned char* rows_a_base(const RowsArgs& P, int tb0, int lane) { // this lane's place in the first column block
    return P.A + (size_t)(tb0 * 4 + (lane >> 4)) * P.lay.t * 16 + (lane & 15 & (P.lay.t - 1)) * 16;
}

template <int MB> struct RowsShared {
    f32x4 red[2][RW_WAVES][MB][64]; // tiles alternate
    float rms[MB * 16], part[RW_THREADS];
};

// Sums of squares of the workgroup's token rows -> 1 / rms: 512 / (16 MB) threads per row, each a fixed share of the partial sums.
template <int MB> __device__ __forceinline__ void rows_ssq(const RowsArgs& P, RowsShared<MB>& sh, int tb0) {
    constexpr int TPR = RW_THREADS / (16 * MB);
    if (!P.ssqIn) return;
    const int r = threadIdx.x / TPR, j = threadIdx.x % TPR;
    float s = 0.f;
    for (int i = j; i < P.nparts; i += TPR) s += P.ssqIn[(size_t)i * 64 + tb0 * 16 + r];
    sh.part[threadIdx.x] = s;
}
template <int MB> __device__ __forceinline__ void rows_rms(const RowsArgs& P, RowsShared<MB>& sh) { // after a barrier behind rows_ssq
    constexpr int TPR = RW_THREADS / (16 * MB);
    if (!P.ssqIn) return;
    if (threadIdx.x < 16 * MB) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < TPR; j++) s += sh.part[threadIdx.x * TPR + j];
        sh.rms[threadIdx.x] = 1.0f / sqrtf(s / (float)P.normDim + 1e-8f);
    }
    __syncthreads();
}

// The workgroup's partial sums of a tile are in sh.red[buf]: wave mb finishes token block mb; lane 16 q + t has the tile's columns
// 4 q .. 4 q + 3 of token 16 (tb0 + mb) + t.
template <typename WT, int MB, int EPI>
__device__ __forceinline__ void rows_epilogue(const RowsArgs& P, const RowsShared<MB>& sh, int buf, int tile, int tb0) {
    constexpr bool HALFK = sizeof(WT) == 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, t16 = lane & 15, q = lane >> 4, n = tile * RW_TILE + 4 * q;
    if (wave >= MB) return;
    f32x4 v = (f32x4)(0.f);
#pragma unroll
    for (int k = 0; k < RW_WAVES; k += 2) v += sh.red[buf][k][wave][lane] + sh.red[buf][k + 1][wave][lane];
    if (P.ssqIn) v *= sh.rms[wave * 16 + t16];
    const int m = (tb0 + wave) * 16 + t16;
    const bool live = m < P.M;
    if (EPI == RW_SWIGLU) {
        if (live && n < P.N) { // columns 2 j, 2 j + 1: gate and up of unit j
            uint32_t s[3];
            p3_split2((v.x / (1.0f + expf(-v.x))) * v.y, (v.z / (1.0f + expf(-v.z))) * v.w, s);
            const int j = n >> 1; // even: the two units are half of a group of four
            unsigned char* o = P.out + rows_offset(j & ~3, m, P.lay, HALFK) + (j & 2) * 2;
#pragma unroll
            for (int pl = 0; pl < 3; pl++) *reinterpret_cast<uint32_t*>(o + pl * P.lay.stride()) = s[pl];
        }
    } else if (EPI == RW_RESID) { // N and ldc are multiples of 16
        if (live) v += *reinterpret_cast<const f32x4*>(P.R + (size_t)m * P.ldc + n);
        else v = (f32x4)(0.f);
        float s = v.x * v.x;
        s = fmaf(v.y, v.y, s); s = fmaf(v.z, v.z, s); s = fmaf(v.w, v.w, s);
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        if (q == 0) P.ssqOut[(size_t)tile * 64 + m] = s;
        if (live) {
            *reinterpret_cast<f32x4*>(P.C + (size_t)m * P.ldc + n) = v;
            const f32x4 g = *reinterpret_cast<const f32x4*>(P.outGain + n);
            rows_put4(P.out, n, m, P.lay, HALFK, g.x * v.x, g.y * v.y, g.z * v.z, g.w * v.w);
        }
    } else {
        if (live) {
            float* c = P.C + (size_t)(EPI == RW_LOGITS ? P.sidx[m] : m) * P.ldc + n;
            if ((P.ldc & 3) == 0 && n + 3 < P.N) *reinterpret_cast<f32x4*>(c) = v;
            else
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < P.N) c[e] = v[e];
        }
        if (EPI == RW_LOGITS) { // largest of the 16 rows, lowest index on ties
            if (P.stepCounter && tile == 0 && tb0 == 0 && threadIdx.x == 0) *P.stepCounter += 1; // steps begun: the finish logs into row (counter - 1)
            float best = -3.0e38f;
            int bi = 0x7fffffff;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < P.N && v[e] > best) { best = v[e]; bi = n + e; }
#pragma unroll
            for (int o = 16; o < 64; o <<= 1) {
                const float ov = __shfl_xor(best, o, 64);
                const int oi = __shfl_xor(bi, o, 64);
                if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
            }
            if (live && q == 0) {
                P.amaxVal[(size_t)m * P.amaxParts + tile] = best;
                P.amaxIdx[(size_t)m * P.amaxParts + tile] = bi;
            }
        }
    }
}

// K of at most CNT chunks per wave: the activations stay in registers, workgroup x walks the tiles x, x + gridDim.x, ...
template <typename WT, int MB, int CNT, int EPI>
__global__ void __launch_bounds__(RW_THREADS, 2) k_rows(RowsArgs P) {
    __shared__ RowsShared<MB> sh;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tb0 = blockIdx.y * MB;
    const int nchunks = P.K / RowsW<WT>::KE, cnt = (nchunks - wave + RW_WAVES - 1) / RW_WAVES; // chunks wave, wave + 8, ...
    RowsW<WT> w[2][CNT];
    RowsA<WT, MB> a[CNT];
    const unsigned char* W = P.W + lane * 16;
    auto loadW = [&](int tile, int buf) { // (a wave with fewer chunks fetches its matrix row's last one again)
#pragma unroll
        for (int i = 0; i < CNT; i++) w[buf][i].load(W + ((size_t)tile * nchunks + min(wave + i * RW_WAVES, nchunks - 1)) * 2048);
    };
    int tile = blockIdx.x;
    loadW(tile, 0);
    {
        const unsigned char* A = rows_a_base(P, tb0, lane);
        const int stride = P.lay.stride(), block = 64 * P.lay.t;
#pragma unroll
        for (int i = 0; i < CNT; i++) a[i].load(A + (size_t)min(wave + i * RW_WAVES, nchunks - 1) * (RowsW<WT>::SUB * 3) * stride, stride, block);
    }
    rows_ssq<MB>(P, sh, tb0);
    auto multiply = [&](int buf) {
        f32x4 acc[MB];
#pragma unroll
        for (int mb = 0; mb < MB; mb++) acc[mb] = (f32x4)(0.f);
#pragma unroll
        for (int i = 0; i < CNT; i++)
            if (i < cnt) w[buf][i].template mul<MB>(a[i].v, acc);
#pragma unroll
        for (int mb = 0; mb < MB; mb++) sh.red[buf][wave][mb][lane] = acc[mb];
    };
    bool first = true;
    auto pass = [&](int buf) -> bool { // a tile whose weights are in buffer buf; returns whether there is another one
        const int next = tile + gridDim.x;
        const bool more = next < P.tiles;
        if (more) { // (two copies of the product: the waits in front of it differ)
            loadW(next, buf ^ 1);
            multiply(buf);
        } else {
            multiply(buf);
        }
        __syncthreads();
        if (first) rows_rms<MB>(P, sh);
        first = false;
        rows_epilogue<WT, MB, EPI>(P, sh, buf, tile, tb0);
        tile = next;
        return more;
    };
    while (pass(0) && pass(1)) {}
}

// One tile per workgroup, weights D chunks and activations AD chunks ahead.
template <typename WT, int MB, int D, int AD, int EPI>
__global__ void __launch_bounds__(RW_THREADS, 2) k_rows_long(RowsArgs P) {
    static_assert(D % AD == 0, "the activation ring must line up with the weight ring");
    __shared__ RowsShared<MB> sh;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tile = blockIdx.x, tb0 = blockIdx.y * MB;
    const int nchunks = P.K / RowsW<WT>::KE, cnt = (nchunks - wave + RW_WAVES - 1) / RW_WAVES;
    RowsW<WT> w[D];
    RowsA<WT, MB> a[AD];
    const unsigned char *W = P.W + (size_t)tile * nchunks * 2048 + lane * 16, *A = rows_a_base(P, tb0, lane);
    const int stride = P.lay.stride(), block = 64 * P.lay.t;
    auto loadW = [&](int i, int slot) { w[slot].load(W + (size_t)min(wave + i * RW_WAVES, nchunks - 1) * 2048); };
    auto loadA = [&](int i, int slot) { a[slot].load(A + (size_t)min(wave + i * RW_WAVES, nchunks - 1) * (RowsW<WT>::SUB * 3) * stride, stride, block); };
#pragma unroll
    for (int j = 0; j < D; j++) loadW(j, j);
#pragma unroll
    for (int j = 0; j < AD; j++) loadA(j, j);
    rows_ssq<MB>(P, sh, tb0);
    f32x4 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++) acc[mb] = (f32x4)(0.f);
    int i = 0;
    for (; i + D < cnt; i += D) {
#pragma unroll
        for (int j = 0; j < D; j++) {
            w[j].template mul<MB>(a[j % AD].v, acc);
            loadW(i + j + D, j);
            loadA(i + j + AD, j % AD);
        }
    }
#pragma unroll
    for (int j = 0; j < D; j++) {
        if (i + j < cnt) w[j].template mul<MB>(a[j % AD].v, acc);
        if (j + AD < D) loadA(i + j + AD, j % AD);
    }
#pragma unroll
    for (int mb = 0; mb < MB; mb++) sh.red[0][wave][mb][lane] = acc[mb];
    __syncthreads();
    rows_rms<MB>(P, sh);
    rows_epilogue<WT, MB, EPI>(P, sh, 0, tile, tb0);
}

template <typename WT, int EPI>
static void launch_rows(hipStream_t st, const RowsArgs& P, int cus) {
    const int cnt = (P.K / RowsW<WT>::KE + RW_WAVES - 1) / RW_WAVES; // chunks per wave
    // Token blocks per workgroup: all of them, so that a weight row is fetched by one workgroup -- unless so few workgroups
    // would be left that splitting the tokens (the weights then come from the cache) keeps more compute units busy.
    int mb = P.lay.blocks;
    while (mb > 1 && P.tiles * (P.lay.blocks / mb) <= 160) mb /= 2;
    const int gy = P.lay.blocks / mb, rounds = (P.tiles * gy + cus - 1) / cus;
    // one workgroup per compute unit, the tiles dealt evenly
    const dim3 walk((P.tiles + rounds - 1) / rounds, gy), each(P.tiles, gy);
#define ROWS(MB_, CNT_) do { hipLaunchKernelGGL((k_rows<WT, MB_, CNT_, EPI>), walk, dim3(RW_THREADS), 0, st, P); return; } while (0)
#define ROWS_LONG(MB_, D_, AD_) do { hipLaunchKernelGGL((k_rows_long<WT, MB_, D_, AD_, EPI>), each, dim3(RW_THREADS), 0, st, P); return; } while (0)
    // CNT, the chunks per wave whose activations stay in registers (12 MB registers per fp32 chunk, 24 MB per bf16 chunk, beside two
    // tiles' weights): the steps are those that widths of 256, 768, 1024 and 2048 need, alone and beside 64 PLE columns (fp32 K up to
    // 256, 768, 1024; bf16 up to 1024, 2048, 2560), where the form was timed, and not every depth there could be.  K in between takes the next deeper form: a wave that is a chunk
    // short fetches its row's last chunk once more, from the cache, and does not multiply it.  The deepest are bounded by the 256
    // registers of two waves per SIMD (250 with one block of bf16, 248 with four blocks of fp32); beyond them, and where four blocks
    // of bf16 would not fit at all, both operands are streamed.
    if constexpr (sizeof(WT) == 4) {
        if (mb == 1) { if (cnt <= 1) ROWS(1, 1); if (cnt <= 3) ROWS(1, 3); if (cnt <= 4) ROWS(1, 4); ROWS_LONG(1, 8, 4); }
        if (mb == 2) { if (cnt <= 1) ROWS(2, 1); if (cnt <= 3) ROWS(2, 3); ROWS_LONG(2, 4, 2); }
        if (cnt <= 1) ROWS(4, 1);
        if (cnt <= 3) ROWS(4, 3);
        ROWS_LONG(4, 4, 2);
    } else {
        if (mb == 1) { if (cnt <= 2) ROWS(1, 2); if (cnt <= 4) ROWS(1, 4); if (cnt <= 5) ROWS(1, 5); ROWS_LONG(1, 8, 2); }
        if (mb == 2) { if (cnt <= 2) ROWS(2, 2); ROWS_LONG(2, 4, 2); }
        ROWS_LONG(4, 4, 1);
    }
#undef ROWS
#undef ROWS_LONG
}

// row-major [rows, K] -> fetch order (rows.h); rows past the end: zero
__global__ void __launch_bounds__(256) k_rows_pack(const unsigned char* __restrict__ src, unsigned char* __restrict__ dst, int rows, int rowBytes, size_t pieces) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < pieces; i += (size_t)gridDim.x * 256) {
        const int lane = (int)(i & 63), p = (int)(i >> 6) & 1, nch = rowBytes / 128;
        const size_t tc = i >> 7, row = tc / nch * RW_TILE + (lane & 15);
        u32x4 v = (u32x4)(0u);
        if (row < (size_t)rows) v = *reinterpret_cast<const u32x4*>(src + row * rowBytes + tc % nch * 128 + p * 64 + (lane >> 4) * 16);
        *reinterpret_cast<u32x4*>(dst + i * 16) = v;
    }
}

// ---- the step's other kernels ----
template <typename WT> __device__ __forceinline__ float rw_get(const WT* p);
template <> __device__ __forceinline__ float rw_get<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float rw_get<bf16_t>(const bf16_t* p) { return __uint_as_float(((uint32_t)*p) << 16); }

struct RowsEmbed { // what the embedding of a row writes
    float* x;           // residual rows
    unsigned char* out; // planes of gain (.) row
    const float* gain;  // of the first applied layer
    float* ssq;         // partial sums of squares [.][64]: the row's whole sum in the first
    RowsLayout lay;
};

// Residual row `slot` from the fp32 or weight-typed row src: its copy, its planes and its sum of squares.  Every thread of a
// 256-thread workgroup calls it; half: bf16 weights.
template <typename ST>
__device__ __forceinline__ void rows_begin(const RowsEmbed& e, int dim, bool half, int slot, const ST* src, float* sh) {
    const int tid = threadIdx.x;
    float s = 0.f;
    for (int i = tid * 4; i < dim; i += 1024) {
        f32x4 v;
        v.x = rw_get<ST>(src + i); v.y = rw_get<ST>(src + i + 1); v.z = rw_get<ST>(src + i + 2); v.w = rw_get<ST>(src + i + 3);
        if (e.x) *reinterpret_cast<f32x4*>(e.x + (size_t)slot * dim + i) = v;
        const f32x4 g = *reinterpret_cast<const f32x4*>(e.gain + i);
        rows_put4(e.out, i, slot, e.lay, half, g.x * v.x, g.y * v.y, g.z * v.z, g.w * v.w);
        s = fmaf(v.x, v.x, s); s = fmaf(v.y, v.y, s); s = fmaf(v.z, v.z, s); s = fmaf(v.w, v.w, s);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((tid & 63) == 0) sh[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) e.ssq[slot] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// the embedding of a token (inference.cu:9-22)
template <typename WT>
__global__ void __launch_bounds__(256) k_rows_embed(StepArgs a, RowsEmbed e) {
    __shared__ float sh[4];
    rows_begin<WT>(e, a.dim, sizeof(WT) == 2, blockIdx.x, (const WT*)a.E + (size_t)a.tok[blockIdx.x] * a.dim, sh);
}

// the last row of every segment of a prefill, for the LM head: segment seg0 + x becomes row x
__global__ void __launch_bounds__(256) k_rows_last(RowsEmbed e, const float* X, int dim, bool half, const int* segStart, const int* segLen) {
    __shared__ float sh[4];
    rows_begin<float>(e, dim, half, blockIdx.x, X + (size_t)(segStart[blockIdx.x] + segLen[blockIdx.x] - 1) * dim, sh);
}

// Attention over several workgroups per (head, sequence): their partial results combined, gated (inference.cu:241-250) and,
// with the PLE columns e = silu(gate) * P[tok], written as planes.  Grid: slots x pieces of the row.
__global__ void __launch_bounds__(256) k_rows_mix(StepArgs a, LayerDev L) {
    const int slot = blockIdx.x, tid = threadIdx.x, hd = a.hd;
    const float* qkv = a.qkv + (size_t)slot * a.qkvStride;
    const bool half = a.wbytes == 2;
    const int i = blockIdx.y * 256 + tid;
    if (i < L.ad) {
        const int h = i / hd, e = i - h * hd;
        const float* pp = a.part + (((size_t)slot * a.nsplit) * a.heads + h) * (hd + 2);
        const size_t sstride = (size_t)a.heads * (hd + 2);
        float M = -1.0e30f;
        for (int s = 0; s < a.nsplit; s++) M = fmaxf(M, pp[s * sstride + hd]);
        float num = 0.f, den = 0.f;
        for (int s = 0; s < a.nsplit; s++) {
            const float w = expf(pp[s * sstride + hd] - M);
            num = fmaf(w, pp[s * sstride + e], num);
            den = fmaf(w, pp[s * sstride + hd + 1], den);
        }
        float v = num / den;
        if (a.gating) v = v / (1.0f + expf(-qkv[L.offG + i]));
        rows_put(a.mixRows, i, slot, a.mixLay, half, v);
    } else if (i - L.ad < a.ple) {
        const int j = i - L.ad;
        const size_t t = (size_t)a.tok[slot] * a.ple + j;
        const float g = qkv[L.offPle + j], p = half ? rw_get<bf16_t>((const bf16_t*)L.pleTable + t) : ((const float*)L.pleTable)[t];
        rows_put(a.mixRows, i, slot, a.mixLay, half, g / (1.0f + expf(-g)) * p);
    }
}

// One workgroup per slot: the pick from the LM head's partial maxima (lowest index on ties) or a draw from the logits,
// the bookkeeping (next token, id log, position) and, when another step follows, that step's embedding.
template <typename WT>
__global__ void __launch_bounds__(256) k_rows_finish(StepArgs a, RowsEmbed e, int nparts, int* tokOut, int embedNext) {
    __shared__ float sv[256];
    __shared__ int si[256];
    __shared__ double sd[257];
    const int slot = blockIdx.x, tid = threadIdx.x, seq = a.sidx[slot];
    int nxt;
    if (a.temperature > 0.f) {
        nxt = mlh_sample_row<256>(a.logits + (size_t)seq * a.vocab, a.vocab, a.temperature, mlh_sample_uniform(a.sampleSeed, seq, a.pos[seq] + 1), sd, si);
        __syncthreads();
    } else {
        float v = -3.0e38f;
        int idx = 0x7fffffff;
        for (int i = tid; i < nparts; i += 256) {
            const float v2 = a.amaxVal[(size_t)slot * a.amaxParts + i];
            const int i2 = a.amaxIdx[(size_t)slot * a.amaxParts + i];
            if (v2 > v || (v2 == v && i2 < idx)) { v = v2; idx = i2; }
        }
        sv[tid] = v; si[tid] = idx;
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if (tid < s && (sv[tid + s] > sv[tid] || (sv[tid + s] == sv[tid] && si[tid + s] < si[tid]))) { sv[tid] = sv[tid + s]; si[tid] = si[tid + s]; }
            __syncthreads();
        }
        nxt = si[0];
        if (nxt < 0 || nxt >= a.vocab) nxt = 0; // only reachable with non-finite logits
        __syncthreads();
    }
    if (tid == 0) {
        const int step = *a.stepCounter - 1; // counted up by the LM head
        tokOut[slot] = nxt;
        a.nextTok[seq] = nxt;
        if (step >= 0 && step < a.outCapacity) a.outIds[(size_t)step * a.nseq + slot] = nxt;
        a.pos[seq] += 1;
    }
    if (embedNext) rows_begin<WT>(e, a.dim, sizeof(WT) == 2, slot, (const WT*)a.E + (size_t)nxt * a.dim, sv);
}

__global__ void k_rows_advance(StepArgs a) { // a token that needs no logits
    const int slot = threadIdx.x;
    if (slot < a.nseq) a.pos[a.sidx[slot]] += 1;
}

// ----------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------
bool mlh_rows_applicable(const mlh_ctx* c, int nseq) { return c->prefillMode == 0 && nseq <= 64 && mlh_prefill_gemm_supported(c); }

// The row step's weights (owned by the context's operand list, rebuilt by a repeated finalize) and work buffers.
static int pack(mlh_ctx* c, const void* src, int rows, int cols, const void** dst) {
    const int rowBytes = cols * c->wbytes;
    const size_t pieces = (size_t)((rows + RW_TILE - 1) / RW_TILE) * RW_TILE * rowBytes / 16;
    void* buf = nullptr;
    if (const int rc = mlh_operand_alloc(c, &buf, pieces * 16)) return rc;
    hipLaunchKernelGGL(k_rows_pack, dim3(4096), dim3(256), 0, c->stream, (const unsigned char*)src, (unsigned char*)buf, rows, rowBytes, pieces);
    MLH_CHECK(c, hipGetLastError());
    *dst = buf;
    return 0;
}

int mlh_rows_prepare(mlh_ctx* c) {
    const mlh_hparams& hp = c->hp;
    int rc = 0;
    for (LayerDev& L : c->layers) // (WoR holds [Wo | pleUp] as one row-major matrix so far)
        if ((rc = pack(c, L.Wa, L.rowsA, hp.dim, &L.WaR)) || (rc = pack(c, L.WoR, hp.dim, L.ad + hp.pleDim, &L.WoR)) ||
            (rc = pack(c, L.W13, 2 * hp.ffnDim, hp.dim, &L.W13R)) || (rc = pack(c, L.W2, hp.dim, hp.ffnDim, &L.W2R)))
            return rc;
    if ((rc = pack(c, c->E, hp.vocabSize, hp.dim, &c->ER))) return rc;
    if (c->rowsBuf) return 0;
    const size_t d = (size_t)hp.dim * 384, mix = (size_t)(c->maxAd + hp.pleDim) * 384, u = (size_t)hp.ffnDim * 384, ssq = (size_t)(hp.dim / RW_TILE) * 64 * 4;
    void* p = nullptr;
    if ((rc = mlh_dev_alloc_bytes(c, &p, 2 * d + mix + u + 2 * ssq))) return rc;
    unsigned char* b = (unsigned char*)p;
    c->rowsX = b; c->rowsH = b + d; c->rowsMix = b + 2 * d; c->rowsU = b + 2 * d + mix;
    c->rowsSsqX = (float*)(b + 2 * d + mix + u);
    c->rowsSsqH = c->rowsSsqX + ssq / 4;
    c->rowsBuf = p;
    return 0;
}

void mlh_rows_gemm(mlh_ctx* c, int epi, const void* w, int n, RowsArgs P) {
    P.W = (const unsigned char*)w; P.N = n; P.tiles = (n + RW_TILE - 1) / RW_TILE;
    const bool half = c->hp.weightDtype == MLH_DTYPE_BF16;
#define ROWS_EPI(E_) do { if (half) launch_rows<bf16_t, E_>(c->stream, P, c->numCUs); else launch_rows<float, E_>(c->stream, P, c->numCUs); } while (0)
    if (epi == RW_PLAIN) ROWS_EPI(RW_PLAIN);
    else if (epi == RW_RESID) ROWS_EPI(RW_RESID);
    else if (epi == RW_SWIGLU) ROWS_EPI(RW_SWIGLU);
    else ROWS_EPI(RW_LOGITS);
#undef ROWS_EPI
}

// Output projection, gate / up and down projection of file block t over the rows of `base`: residual rows x -> h1 -> x.
void mlh_rows_rest_of_layer(mlh_ctx* c, int t, const RowsArgs& base, float* x, float* h1) {
    const mlh_hparams& hp = c->hp;
    const LayerDev& L = c->layers[t];
    const int d = hp.dim, F = hp.ffnDim;
    RowsArgs P = base; // h1 = [Wo | pleUp] . [mix | e] + x (inference.cu:582-610)
    P.K = L.ad + hp.pleDim; P.A = c->rowsMix; P.C = h1; P.ldc = d; P.R = x; P.out = c->rowsH; P.outGain = L.g2; P.ssqOut = c->rowsSsqH;
    mlh_rows_gemm(c, RW_RESID, L.WoR, d, P);
    mlh_mark(c, MLH_K_OPROJ);
    P = base; // silu(gate) * up of the normalised rows (inference.cu:612-672)
    P.K = d; P.A = c->rowsH; P.ssqIn = c->rowsSsqH; P.nparts = d / RW_TILE; P.out = c->rowsU;
    mlh_rows_gemm(c, RW_SWIGLU, L.W13R, 2 * F, P);
    mlh_mark(c, MLH_K_FFN_GATEUP);
    P = base; // x = W2 . u + h1 (inference.cu:675-699), and the planes for the next layer's first product or the LM head
    P.K = F; P.A = c->rowsU; P.C = x; P.ldc = d; P.R = h1; P.out = c->rowsX; P.outGain = t > 0 ? c->layers[t - 1].g1 : c->gF; P.ssqOut = c->rowsSsqX;
    mlh_rows_gemm(c, RW_RESID, L.W2R, d, P);
    mlh_mark(c, MLH_K_FFN_DOWN);
}

void mlh_rows_embed(mlh_ctx* c, const int* tok, int n, float* x, RowsLayout lay) {
    StepArgs a;
    mlh_fill_args(c, a, n, tok);
    const RowsEmbed emb = {x, c->rowsX, c->layers[c->hp.transformers - 1].g1, c->rowsSsqX, lay};
    if (c->hp.weightDtype == MLH_DTYPE_BF16) hipLaunchKernelGGL((k_rows_embed<bf16_t>), dim3(n), dim3(256), 0, c->stream, a, emb);
    else hipLaunchKernelGGL((k_rows_embed<float>), dim3(n), dim3(256), 0, c->stream, a, emb);
}

// Final norm and LM head of the last row of each of n <= 64 segments: logits of sequence segSeq[i], partial maxima of slot i.
void mlh_rows_lm_head(mlh_ctx* c, int n, const float* X, const int* segStart, const int* segLen, const int* segSeq, float* amaxVal, int* amaxIdx) {
    const mlh_hparams& hp = c->hp;
    const RowsLayout lay = rows_layout(n);
    const RowsEmbed emb = {nullptr, c->rowsX, c->gF, c->rowsSsqX, lay};
    hipLaunchKernelGGL(k_rows_last, dim3(n), dim3(256), 0, c->stream, emb, X, hp.dim, hp.weightDtype == MLH_DTYPE_BF16, segStart, segLen);
    RowsArgs P = {};
    P.M = n; P.K = hp.dim; P.lay = lay; P.normDim = hp.dim; P.A = c->rowsX; P.ssqIn = c->rowsSsqX; P.nparts = 1; P.C = c->logits; P.ldc = hp.vocabSize;
    P.sidx = segSeq; P.amaxVal = amaxVal; P.amaxIdx = amaxIdx; P.amaxParts = c->amaxParts;
    mlh_rows_gemm(c, RW_LOGITS, c->ER, hp.vocabSize, P);
}

// One step of nseq sequences on the context's stream (no allocation, no synchronisation: can be captured).  embedded: the step
// before it has already written the residual rows; embedNext: this one does that for the next.
int mlh_rows_step(mlh_ctx* c, int nseq, const int* tokPtr, bool lmHead, bool embedded, bool embedNext) {
    if (!c->rowsBuf) { c->err = "row step buffers not prepared"; return -1; }
    const mlh_hparams& hp = c->hp;
    hipStream_t st = c->stream;
    const RowsLayout lay = rows_layout(nseq);
    const int first = hp.transformers - 1, d = hp.dim;
    c->mixRows = c->rowsMix;
    c->mixLay = lay;
    StepArgs a;
    mlh_fill_args(c, a, nseq, tokPtr);
    if (!embedded) mlh_rows_embed(c, tokPtr, nseq, c->x, lay);
    if (!embedded) mlh_mark(c, MLH_K_EMBED);
    RowsArgs base = {};
    base.M = nseq; base.lay = lay; base.normDim = d; base.sidx = c->d_sidx;
    int nparts = 1; // partial sums behind rowsX: one from the embedding, one per workgroup from a down projection
    int rc = 0;
    for (int t = first; t >= 0 && rc == 0; t--) { // file block 0 is the top (inference.cu:384-385)
        const LayerDev& L = c->layers[t];
        RowsArgs P = base; // q | k | v | ... of the normalised rows (inference.cu:388-465, 487-507)
        P.K = d; P.A = c->rowsX; P.ssqIn = c->rowsSsqX; P.nparts = nparts; P.C = c->qkv; P.ldc = c->maxRowsA;
        mlh_rows_gemm(c, RW_PLAIN, L.WaR, L.rowsA, P);
        mlh_mark(c, MLH_K_QKV);
        rc = mlh_launch_mix(c, a, L);
        if (L.kind == MLH_KIND_ATTENTION && c->nsplit > 1) hipLaunchKernelGGL(k_rows_mix, dim3(nseq, (L.ad + hp.pleDim + 255) / 256), dim3(256), 0, st, a, L);
        mlh_mark(c, L.kind == MLH_KIND_ATTENTION ? MLH_K_ATTN : MLH_K_GDN); // (the combination of the partial results with it)
        mlh_rows_rest_of_layer(c, t, base, c->x, c->h1);
        nparts = d / RW_TILE;
    }
    c->mixRows = nullptr;
    if (rc) return rc;
    if (lmHead) { // tied LM head of the normalised rows (inference.cu:705-743)
        RowsArgs P = base;
        P.K = d; P.A = c->rowsX; P.ssqIn = c->rowsSsqX; P.nparts = nparts; P.C = c->logits; P.ldc = hp.vocabSize;
        P.amaxVal = c->amaxVal; P.amaxIdx = c->amaxIdx; P.amaxParts = c->amaxParts; P.stepCounter = c->d_stepCounter;
        mlh_rows_gemm(c, RW_LOGITS, c->ER, hp.vocabSize, P);
        mlh_mark(c, MLH_K_LMHEAD);
        const RowsEmbed emb = {c->x, c->rowsX, c->layers[first].g1, c->rowsSsqX, lay};
        const int np = (hp.vocabSize + RW_TILE - 1) / RW_TILE, next = embedNext ? 1 : 0;
        if (hp.weightDtype == MLH_DTYPE_BF16) hipLaunchKernelGGL((k_rows_finish<bf16_t>), dim3(nseq), dim3(256), 0, st, a, emb, np, c->d_tok, next);
        else hipLaunchKernelGGL((k_rows_finish<float>), dim3(nseq), dim3(256), 0, st, a, emb, np, c->d_tok, next);
        mlh_mark(c, MLH_K_FINISH);
    } else {
        hipLaunchKernelGGL(k_rows_advance, dim3(1), dim3(64), 0, st, a);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) { c->err = std::string("row step launch: ") + hipGetErrorString(e); return -2; }
    return 0;
}
