// Decode of up to 16 sequences in one launch, every XCD of the MI355X a tensor-parallel rank (gfx950, wave64).
//
// As kernels of their own the products of a step are five dependent launches a layer, and a launch costs 4 to 8 us whatever it
// multiplies.  Here one launch runs all steps of a call: the layers are cut up over the XCDs as in the one-sequence kernel
// (kernels_xcd.hip: heads X, X + 8 and FFN units [X F/8, (X + 1) F/8) on XCD X), so that a layer has two exchanges across the XCDs
// (the partial sums of the output and the down projection) and five inside one.  Exchanged values are (value, tag) words whose tag is
// the number of the layer pass: the arrival of the data is the synchronisation.  Every buffer is rewritten one pass later, by
// workgroups that have meanwhile gathered a slice from every workgroup of their XCD, so nobody is still reading it.
//
// A workgroup (one per compute unit, 32 per XCD) is eight workers and four communicators.
//   Workers multiply: 16 weight rows a tile in the row kernels' fetch order (rows.h), on v_mfma_f32_16x16x32_bf16 at fp32 precision
//   (fp32 weights as three planes, activations as three planes).  They touch global memory for weights only, issued a phase or two
//   ahead into registers, and never wait for an exchange.
//   Communicators do the rest: add the partial sums of the workgroup's slice of the columns (the residual stays with them), gather
//   what the next product needs, split it into planes in LDS, and run the token mixing (attention over the pages, the delta rule on
//   state rows).  They poll; loads return in issue order on this ISA, so a wave that polled behind its own weight loads would see
//   the answer late.
// The sides meet at workgroup barriers.
//
// What bounds it: the chain of exchanges and what a communicator executes between them; for the widest models HBM as well.  Time stamps: d 768,
// 5 sequences, a gated-delta-net layer 17.7 us, its bytes 6 at the copy kernel's rate: partial sums from all XCDs 2.3, residual rows gathered and
// split 3.0, the products with their words' way out and in 7.2, delta rule 1.0, mixing output 1.0, barriers and 1 / rms 2.6.  d 2048 bf16: 28 us for
// one sequence, 42 for eight (bytes 22 and 25), of which the residual rows are 2.7 and 10.6.  Hence the care below for what is formed when: a value made
// of the thread's place that the compiler keeps, spills or moves behind a barrier costs more than forming it again.
// Measured, us per step, here and as the row kernels' sequence: hybrid, fp32, d 768, 12 layers: 2 sequences 219 and 367, 5 sequences 232
// and 373, 16 sequences 315 and 394; hybrid, bf16, d 2048, 24 layers: 1 sequence 705 and 1161, 8 sequences 1050 and 1265.  More than
// 16, and from 6 to 9 on where it covers the model and is faster: kernels_wide.hip.
//
// The launch starts with a meeting of all 256 workgroups: if one is missing after a bounded wait nothing has been written and the
// call runs as the sequence of row kernels instead.  Behind it every workgroup is resident, and every wait is bounded as well: when
// one expires the launch ends early and the row kernels redo the steps.  What a redo cannot write anew, the gated-delta-net states, is
// therefore read from one place in the first step and written to another, which counts when the launch has ended well (the host keeps
// which one that is, mlh_ranks_done; other kernels know the first only, mlh_ranks_settle).  The same bytes as in place; a copy of the
// rows made on the way cost 10 to 33 us a launch (d 2048 bf16, 1 and 8 sequences).
#include <string.h>

#include <algorithm>

#include "mlh_internal.h"
#include "xcd_exchange.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

#define RK_WORK 8                             // worker waves
#define RK_COMM 4                             // communicator waves
#define RK_CT (RK_COMM * 64)                  // their threads
#define RK_THREADS ((RK_WORK + RK_COMM) * 64)
#define RK_SPLITS 16                          // key splits of a (head, sequence) at most

struct RanksArgs {
    StepArgs a;
    const LayerDev* layers;
    const unsigned char* ER;
    unsigned char* xw; // exchange words
    unsigned xwBytes, tagBase;
    int NL, steps, fs;
    int rowsQ;         // words per token of the first phase's region
    int planeBytes;    // of the operand planes in LDS
    unsigned *abortFlag, *xcdCount;
    int abortAtStep;   // test hook: workgroup 0 gives up when it reaches this step (> 0)
    int otherAt;       // floats from a sequence's gated-delta-net states to their second place
    unsigned sides;    // bit s: the states of sequence s are in the second place before the launch
    unsigned area, oPart, oMl, oMix, oX, oH, oU, oXP, oHP, oAmax, oTok; // bytes of exchange words per XCD and what lies where in them; oAmax, oTok: behind all of them
};

// ---- weights ----
template <typename WT> struct RkW { u32x4 raw[2]; }; // this lane's share of a chunk: 16 rows x 128 bytes
template <typename WT> struct RkOp;                  // ... ready to multiply
template <> struct RkOp<float> {
    static constexpr int KE = 32, SUB = 1; // K per chunk, 32-wide steps per chunk
    u32x4 w[3];
    __device__ __forceinline__ void from(const RkW<float>& r) {
        uint32_t s[4][3];
#pragma unroll
        for (int p = 0; p < 2; p++) {
            p3_split2(__uint_as_float(r.raw[p].x), __uint_as_float(r.raw[p].y), s[2 * p]);
            p3_split2(__uint_as_float(r.raw[p].z), __uint_as_float(r.raw[p].w), s[2 * p + 1]);
        }
#pragma unroll
        for (int pl = 0; pl < 3; pl++) { w[pl].x = s[0][pl]; w[pl].y = s[1][pl]; w[pl].z = s[2][pl]; w[pl].w = s[3][pl]; }
    }
    __device__ __forceinline__ void pin() { asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2])); }
};
template <> struct RkOp<bf16_t> { // as it comes
    static constexpr int KE = 64, SUB = 2;
    __device__ __forceinline__ void from(const RkW<bf16_t>&) {}
    __device__ __forceinline__ void pin() {}
};
// 32-wide step s of a chunk: six plane products (p3.h) on two chains of accumulators / three on the step's chain
__device__ __forceinline__ void rk_mul(const RkW<float>&, const RkOp<float>& o, int, const u32x4 (&a)[3], f32x4& c0, f32x4& c1) {
#define RK_MM(C_, W_, A_) C_ = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, o.w[W_]), __builtin_bit_cast(bf16x8, a[A_]), C_, 0, 0, 0)
    RK_MM(c0, 0, 2); RK_MM(c1, 1, 1); RK_MM(c0, 2, 0); RK_MM(c1, 0, 1); RK_MM(c0, 1, 0); RK_MM(c1, 0, 0);
#undef RK_MM
}
__device__ __forceinline__ void rk_mul(const RkW<bf16_t>& w, const RkOp<bf16_t>&, int s, const u32x4 (&a)[3], f32x4& c0, f32x4& c1) {
    f32x4& c = s ? c1 : c0;
#pragma unroll
    for (int pl = 2; pl >= 0; pl--)
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w.raw[s]), __builtin_bit_cast(bf16x8, a[pl]), c, 0, 0, 0);
}

// Register sets of a worker.  w1: two tiles over the whole width, K dealt in chunks to the eight workers (first phase, gate / up, LM head);
// w1b: a third tile of gate / up, then the rest of the down projection; w2: output projection, then the down projection, TW tiles of which
// NS workers share one.
template <typename WT, int HD> struct RkCfg;
template <> struct RkCfg<float, 64> { static constexpr int CA = 3, NTB = 0, TW = 2, CO = 2, CW = 2; }; // (8 heads of 128 are wider than fp32 weights fit)
template <int HD> struct RkCfg<bf16_t, HD> { static constexpr int CA = 4, NTB = 1, TW = 4, CO = HD == 64 ? 2 : 3, CW = 6; };

struct RkShared {
    unsigned char* planes; // operand planes of the product at hand
    f32x4* red;            // [2][slots][parts][64] partial sums of the tiles
    float2* resid;         // [RK_CT] residual elements of the communicators' threads
    float *sq, *rms;       // [RK_CT], [16]
    f32x4* ple;            // [64] the XCD's PLE values, four columns of a token each
    float* gain;           // of the next norm
    int *tok, *pos, *seq;  // [16] per slot
    int* ctl;              // [0] leave, [2] XCD, [3] rank
};

// What the workers make of the thread's place is formed again from here on, and not kept, spilled or moved across the phases.
#define RK_FORGET()                              \
    do {                                         \
        X = X0; r = r0; lane = threadIdx.x & 63; \
        asm volatile("" : "+s"(X), "+s"(r), "+v"(lane)); \
    } while (0)
#define RK_BAR() lds_barrier()
// Once per layer, and not at every barrier (0.1 us each): whether a wait was given up.  Until then the waves go on with what they have and
// no further wait waits; what they publish carries valid tags, so K/V rows from the first step's position on, the states' other
// place, logits, picks and positions may all be written from it.  The redo writes them again (positions: mlh_ranks_failed).
#define RK_CHECK()                  \
    do {                            \
        if (runi(S.ctl[0])) return; \
    } while (0)

// The planes of four neighbouring columns k .. k + 3 of token t of mb (rows.h, with as many tokens per block as there are).
__device__ __forceinline__ void rk_put4(unsigned char* planes, int k, int t, int mb, bool half, const float (&v)[4]) {
    uint32_t x[3], y[3];
    p3_split2(v[0], v[1], x);
    p3_split2(v[2], v[3], y);
    const int stride = 64 * mb, q = half ? (k & 31) >> 3 : (k & 15) >> 2, e = half ? k & 4 : (k & 16) >> 2;
    unsigned char* p = planes + (k >> 5) * 3 * stride + (q * mb + t) * 16 + e * 2;
#pragma unroll
    for (int pl = 0; pl < 3; pl++) *reinterpret_cast<uint2*>(p + pl * stride) = make_uint2(x[pl], y[pl]);
}

// Four neighbouring values of a matrix row, fetched now and converted when they are used.
template <typename WT> struct RkRow4;
template <> struct RkRow4<float> {
    f32x4 v;
    __device__ __forceinline__ void load(const void* p, size_t i) { v = *reinterpret_cast<const f32x4*>((const float*)p + i); }
    __device__ __forceinline__ void get(float (&o)[4]) const { o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w; }
};
template <> struct RkRow4<bf16_t> {
    u32x2 v;
    __device__ __forceinline__ void load(const void* p, size_t i) { v = *reinterpret_cast<const u32x2*>((const bf16_t*)p + i); }
    __device__ __forceinline__ void get(float (&o)[4]) const {
        o[0] = __uint_as_float(v.x << 16); o[1] = __uint_as_float(v.x & 0xffff0000u);
        o[2] = __uint_as_float(v.y << 16); o[3] = __uint_as_float(v.y & 0xffff0000u);
    }
};

// tiles of the first phase of a layer on an XCD: its heads' q, k, v (and gate) rows, the tile with its PLE gate rows, the tiles of all gate scalars
template <int HD>
__device__ __forceinline__ int rk_tilesA(LayerPtr L, int heads, int ple, int np, int nh, int& idxPle, int& idxG) {
    const bool gdn = L->kind != MLH_KIND_ATTENTION;
    int n = nh * (gdn ? 3 : np) * (HD / 16);
    idxPle = n;
    if (ple > 0) n++;
    idxG = n;
    if (gdn) n += ((L->offGb + heads - 1) >> 4) - (L->offGa >> 4) + 1;
    return n;
}

// ------------------------------------------------------------------------------------------------ communicators
template <typename WT, int HD>
__device__ __forceinline__ void rk_communicator(const RanksArgs& P, const RkShared& S, int X0, int r0) {
    constexpr bool HALF = sizeof(WT) == 2;
    constexpr int KE = RkOp<WT>::KE, LPR = HD / 4, RPI = 64 / LPR, BR = 4 * RPI, ITS = 64 / (4 * RPI); // (state rows: at most 64 per workgroup)
    const StepArgs& a = P.a;
    const int d = a.dim, cw = runi((int)(threadIdx.x >> 6)) - RK_WORK;
    int id = threadIdx.x - RK_WORK * 64;
    int X = X0, r = r0, lane = threadIdx.x & 63;
    const int nh = (a.heads - X0 + RK_XCDS - 1) / RK_XCDS, pleX = a.ple / RK_XCDS, part = nh * HD, NL = P.NL, mb = a.nseq;
    const int npAttn = 3 + (a.gating ? 1 : 0);
    const unsigned area = P.area;
    const rsrc_t W = __builtin_amdgcn_make_buffer_rsrc(P.xw, 0, P.xwBytes, 0x00027000);
    const int stepRow = *a.stepCounter; // (advanced when everybody has read it)
    const int batches = ((a.vocab + 15) / 16 + 2 * RK_XCDS * RK_PER - 1) / (2 * RK_XCDS * RK_PER); // of the LM head's tiles, two per workgroup
    bool ok = true;
    auto give_up = [&](unsigned spins) { // bounded waits
        if (!ok || spins > RK_SPIN || ((spins & 127) == 127 && aldu(P.abortFlag))) { ok = false; return true; }
        return false;
    };
    auto tell = [&]() { if (!ok) { S.ctl[0] = 1; astu(P.abortFlag, 3u); } };
    // A thread has token tk and every G-th group of four columns from g0 on, this workgroup state rows of one pair of a head and a
    // sequence, this wave a share of the keys of one.
    const int G = runi(RK_CT / mb), pairs = mb * nh;
    const bool act = id < G * mb;
    const int g00 = act ? id / mb : 0, tk0 = act ? id - g00 * mb : 0;
    int g0 = g00, tk = tk0;
    int rows = 4 * RPI; // of a pair per workgroup: the XCD's 32 workgroups share its pairs
    while (rows < 64 && pairs * HD > rows * RK_PER) rows *= 2;
    const int gPair = runi(r0 / (HD / rows)), gIts = gPair < pairs ? rows / (4 * RPI) : 0; // RPI rows a wave, gIts times; 0: none
    const int gHead = runi(gPair / mb), gTok = gPair - gHead * mb, gMove = runi((int)(P.sides >> S.seq[gTok])) & 1 ? -P.otherAt : P.otherAt, gRow = (r0 - gPair * (HD / rows)) * rows + cw * (rows / 4);
    const int aSplit = runi((cw * RK_PER + r0) / pairs), aPair = cw * RK_PER + r0 - aSplit * pairs, aHead = runi(aPair / mb), aTok = aPair - aHead * mb;
    int lanesLog = 6; // of the lanes that sum up a row's squares
    while ((mb << lanesLog) > 64) lanesLog--;
    int lrow = 0, c4 = 0;  // of a wave on rows of HD: row among RPI, column
    unsigned own = 0;      // the XCD's exchange words
    auto forget = [&]() __attribute__((always_inline)) { // what is made of the thread's place is formed again from here on, and not kept or hoisted
        X = X0; r = r0; lane = threadIdx.x & 63; g0 = g00; tk = tk0;
        asm volatile("" : "+s"(X), "+s"(r), "+v"(lane), "+v"(g0), "+v"(tk));
        id = cw * 64 + lane; lrow = lane / LPR; c4 = (lane % LPR) * 4; own = (unsigned)X * area;
    };
    // Four columns of a token, four or eight times per thread: a region of ng groups, read until every tag is there, to use(group, values).
    auto fetch = [&](auto rbTag, unsigned base, int ng, int g, unsigned tag, auto&& use) __attribute__((always_inline)) {
        constexpr int RB = decltype(rbTag)::value;
        const unsigned half = (unsigned)(ng * mb) * 16u;
        u32x4 w[RB][2];
        unsigned off[RB];
#pragma unroll
        for (int k = 0; k < RB; k++) off[k] = (unsigned)(min(g + k * G, ng - 1) * mb + tk) * 16u;
        for (unsigned spins = 0;; spins++) {
            asm volatile("" ::: "memory");
            bool all = true;
#pragma unroll
            for (int k = 0; k < RB; k++) {
                w[k][0] = xget<LD_XCD>(W, off[k], base);
                w[k][1] = xget<LD_XCD>(W, off[k], base + half);
            }
#pragma unroll
            for (int k = 0; k < RB; k++) all = all && xfresh(w[k][0], tag) && xfresh(w[k][1], tag);
            if (__all(all) || give_up(spins)) break;
        }
#pragma unroll
        for (int k = 0; k < RB; k++)
            if (act && g + k * G < ng) {
                float v[4] = {__uint_as_float(w[k][0].x), __uint_as_float(w[k][0].z), __uint_as_float(w[k][1].x), __uint_as_float(w[k][1].z)};
                use(g + k * G, v);
            }
    };
    auto gather = [&](unsigned base, int ng, unsigned tag, auto&& use) __attribute__((always_inline)) {
#pragma unroll 1
        for (int g = 0; g < ng;) {
            if (ng - g > 4 * G) { fetch(std::integral_constant<int, 8>(), base, ng, g + g0, tag, use); g += 8 * G; }
            else { fetch(std::integral_constant<int, 4>(), base, ng, g + g0, tag, use); g += 4 * G; }
        }
    };
    // Residual rows into planes: the workgroup's slice of the columns is the sum of the XCDs' partial sums and the residual,
    // published inside the XCD and gathered from its 32 workgroups; the gain on the way into LDS, the sums of squares beside it.
    auto residual = [&](unsigned partials, unsigned pub, unsigned tag) __attribute__((always_inline)) {
        const int mine = (d / 64) * mb; // pairs of columns x tokens of the slice
        if (cw * 64 < mine) {
            const int p = id < mine ? g0 : 0, t = id < mine ? tk : 0;
            const unsigned off = (unsigned)(((p & 1) * (d / 4) + r * (d / 128) + (p >> 1)) * mb + t) * 16u;
            float2 res = S.resid[id];
            u32x4 w[RK_XCDS];
            for (unsigned spins = 0;; spins++) {
                asm volatile("" ::: "memory");
                bool all = true;
#pragma unroll
                for (int x = 0; x < RK_XCDS; x++) w[x] = xget<LD_CROSS>(W, off, partials + (unsigned)x * area);
#pragma unroll
                for (int x = 0; x < RK_XCDS; x++) all = all && xfresh(w[x], tag);
                if (__all(all) || give_up(spins)) break;
            }
            float s0 = 0.f, s1 = 0.f; // fixed order
#pragma unroll
            for (int x = 0; x < RK_XCDS; x++) { s0 += __uint_as_float(w[x].x); s1 += __uint_as_float(w[x].z); }
            if (id < mine) {
                res.x += s0; res.y += s1;
                xput<ST_XCD>(W, off, own + pub, res.x, res.y, tag);
                S.resid[id] = res;
            }
        }
        float sq = 0.f;
        gather(own + pub, d / 4, tag, [&](int g, float (&v)[4]) {
            const f32x4 gn = *reinterpret_cast<const f32x4*>(S.gain + 4 * g);
            sq = fmaf(v[0], v[0], sq); sq = fmaf(v[1], v[1], sq); sq = fmaf(v[2], v[2], sq); sq = fmaf(v[3], v[3], sq);
            v[0] *= gn.x; v[1] *= gn.y; v[2] *= gn.z; v[3] *= gn.w;
            rk_put4(S.planes, 4 * g, tk, mb, HALF, v);
        });
        S.sq[id] = sq;
        tell();
    };
    // the first layer's: the embedding rows (inference.cu:9-22), read by every workgroup
    auto embed = [&]() __attribute__((always_inline)) {
        const size_t row = (size_t)S.tok[tk] * d;
        if (id < (d / 64) * mb) {
            float v[4];
            RkRow4<WT> e;
            e.load(a.E, row + 4 * (r * (d / 128) + (g0 >> 1)));
            e.get(v);
            S.resid[id] = (g0 & 1) ? make_float2(v[2], v[3]) : make_float2(v[0], v[1]);
        }
        float sq = 0.f;
#pragma unroll 1
        for (int gr = g0; runi(gr) < d / 4; gr += 4 * G) {
            RkRow4<WT> e[4];
#pragma unroll
            for (int k = 0; k < 4; k++) e[k].load(a.E, row + 4 * min(gr + k * G, d / 4 - 1));
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int g = gr + k * G;
                float v[4];
                e[k].get(v);
                if (act && g < d / 4) {
                    const f32x4 gn = *reinterpret_cast<const f32x4*>(S.gain + 4 * g);
                    sq = fmaf(v[0], v[0], sq); sq = fmaf(v[1], v[1], sq); sq = fmaf(v[2], v[2], sq); sq = fmaf(v[3], v[3], sq);
                    v[0] *= gn.x; v[1] *= gn.y; v[2] *= gn.z; v[3] *= gn.w;
                    rk_put4(S.planes, 4 * g, tk, mb, HALF, v);
                }
            }
        }
        S.sq[id] = sq;
    };
    // 1 / rms of the rows, behind the barrier that makes the sums visible (one wave)
    auto rms = [&]() {
        if (cw) return;
        const int lt = 1 << lanesLog, t = lane >> lanesLog, j = lane & (lt - 1); // lanes per token
        float z[8], s = 0.f; // (at most seven sums a lane)
#pragma unroll
        for (int k = 0; k < 8; k++) z[k] = S.sq[min(min(j + k * lt, G - 1) * mb + t, RK_CT - 1)];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 8; k++) s += j + k * lt < G ? z[k] : 0.f;
        for (int o = 1; o < lt; o <<= 1) s += __shfl_xor(s, o, 64);
        if (j == 0 && t < mb) S.rms[t] = 1.0f / sqrtf(s / (float)d + 1e-8f);
    };

    const int pageSeq = runi(S.seq[aTok]), pages = a.pageTable[pageSeq * a.pagesPerSeq + min(lane, a.pagesPerSeq - 1)]; // lane i: page i of the sequence whose keys this wave reads
    LayerPtr layers = (LayerPtr)P.layers;
    auto gain4 = [&](const float* g, int k) { return *reinterpret_cast<const f32x4*>(g + min(id * 4 + k * RK_CT * 4, d - 4)); };
    auto keep4 = [&](int k, const f32x4& v) { if (id * 4 + k * RK_CT * 4 < d) *reinterpret_cast<f32x4*>(S.gain + id * 4 + k * RK_CT * 4) = v; };

    for (int step = 0; step < P.steps; step++) {
#pragma unroll
        for (int k = 0; k < 2; k++) keep4(k, gain4(layers[NL - 1].g1, k)); // the first norm's gain
        RK_BAR(); // tokens, positions and the first gain in LDS
        RK_CHECK();
        if (P.abortAtStep > 0 && step == P.abortAtStep && X0 == 0 && r0 == 0) ok = false;
        // A half layer is one product over the residual rows and what follows it: even ones the first phase, the token mixing and the
        // output projection, odd ones gate / up and the down projection; behind them the LM head.
#pragma unroll 1
        for (int u = 0; u <= 2 * NL; u++) {
            const int l = u >> 1;
            const bool head = u == 2 * NL, odd = u & 1;
            const unsigned lt = P.tagBase + (unsigned)(step * (NL + 1) + l + 1);
            forget();
            const LayerPtr L = layers + (head ? 0 : NL - 1 - l); // file block 0 is the top (inference.cu:384-385)
            const bool gdn = L->kind != MLH_KIND_ATTENTION;
            // the next norm's gain, fetched now, in LDS behind the first barrier
            f32x4 gn[2];
            {
                const float* g = odd ? l + 1 < NL ? layers[NL - 2 - l].g1 : a.gF : L->g2;
#pragma unroll
                for (int k = 0; k < 2; k++) gn[k] = gain4(g, k);
            }
            auto splits = [&]() { // pieces of a pair's keys, one per wave of the XCD's communicators
                const int longest = (int)pwave_max((float)S.pos[min(lane, mb - 1)]);
                return max(1, min(min(RK_COMM * RK_PER / pairs, RK_SPLITS), (longest + BR - 1) / BR));
            };
            // this wave's first state row (elements, below 2^31: ranks_model), as it is read in this step
            unsigned stateAt = (unsigned)(runi(((S.seq[gTok] * a.gdnHeads + X + RK_XCDS * gHead) * HD + gRow) * HD) + ((gMove > 0) == (step > 0) ? P.otherAt : 0));
            auto key_base = [&](int h, int j) { // row 0 of key block j
                const int q = j * BR / MLH_KV_PAGE;
                const int page = q < 64 ? __builtin_amdgcn_readlane(pages, q) : runi(a.pageTable[pageSeq * a.pagesPerSeq + q]);
                return ((size_t)page * MLH_KV_PAGE + (j * BR) % MLH_KV_PAGE) * d + h * HD;
            };
            auto key_rows = [&](int p, int h, int j, f32x4 (&kv)[8]) __attribute__((always_inline)) { // (rows at and beyond p are not read: they may be written any time)
                const size_t base = key_base(h, j);
                const float *K = L->K + base, *V = L->V + base;
#pragma unroll
                for (int it = 0; it < 4; it++) {
                    unsigned o = (unsigned)(min(it * RPI + lrow, p - 1 - j * BR) * d + c4);
                    asm volatile("" : "+v"(o));
                    kv[it] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(K + o));
                    kv[it + 4] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(V + o));
                }
            };
            // What the token mixing reads of earlier tokens (state rows, or a wave's first block of keys) is brought into the L2 before this wave polls
            // for anything of this layer: one load touches 64 lines.  The gate biases or the position's rotations, and the PLE table's rows, are fetched.
            float touched = 0.f;
            f32x4 side = {};
            RkRow4<WT> pt = {};
            const int gPle = (((int)L->ad + X * pleX) % KE) / 4; // the XCD's PLE columns in the chunk of the output projection they lie in
            auto prefetch = [&]() __attribute__((always_inline)) {
                if (gdn) {
                    if (gIts) {
                        touched = *(L->S + stateAt + min(lane * 32, gIts * RPI * HD - 1));
                        side.x = L->gdnBa[X + RK_XCDS * gHead];
                        side.y = L->gdnBb[X + RK_XCDS * gHead];
                    }
                } else {
                    const int p = runi(S.pos[aTok]);
                    if (aSplit < splits()) {
                        if (aSplit * BR < p) {
                            const int row = min((lane & 31) / (HD / 32), p - 1 - aSplit * BR);
                            touched = *((lane < 32 ? L->K : L->V) + key_base(X + RK_XCDS * aHead, aSplit) + (unsigned)(row * d + (lane % (HD / 32)) * 32));
                        }
                        side = *reinterpret_cast<const f32x4*>(a.rope + (size_t)p * HD + c4);
                    }
                }
                if (a.ple > 0 && act && g0 >= gPle && g0 < gPle + pleX / 4) pt.load(L->pleTable, (size_t)S.tok[tk] * a.ple + X * pleX + 4 * (g0 - gPle));
            };
            // where the token mixing finds things: formed here, where there is time
            int idxPle, idxG;
            rk_tilesA<HD>(L, a.heads, a.ple, npAttn, nh, idxPle, idxG);
            const int gePle = g0 - gPle;
            const bool ple = a.ple > 0 && act && gePle >= 0 && gePle < pleX / 4;
            unsigned po = (unsigned)((ple ? tk * P.rowsQ + 4 * gePle : 0) + idxPle * 16 + ((L->offPle + X * pleX) & 15)) * 8u;
            unsigned mixAt = gdn ? (unsigned)(gTok * P.rowsQ + gHead * 3 * HD) * 8u : (unsigned)(aTok * P.rowsQ + aHead * npAttn * HD) * 8u; // its q rows
            unsigned gateAt = (unsigned)(gTok * P.rowsQ + idxG * 16 + (L->offGa & 15) + X + RK_XCDS * gHead) * 8u, gateStep = (unsigned)(L->offGb - L->offGa) * 8u;
            unsigned qLane = (unsigned)c4 * 8u, vLane = (unsigned)(2 * HD + gRow + lrow) * 8u;
            mixAt = (unsigned)runi((int)mixAt); gateAt = (unsigned)runi((int)gateAt); gateStep = (unsigned)runi((int)gateStep);
            asm volatile("" : "+v"(po), "+s"(mixAt), "+s"(gateAt), "+s"(gateStep), "+v"(qLane), "+v"(vLane), "+s"(stateAt));
            if (!odd && !head) prefetch();
            // ---------------------------------------------------------------- the product's input rows
            if (u == 0) embed();
            else residual(odd ? P.oHP : P.oXP, odd ? P.oH : P.oX, odd ? lt : lt - 1);
            RK_BAR();
            rms();
            RK_BAR();
            if (head)
                for (int k = 1; k < batches; k++) RK_BAR();
#pragma unroll
            for (int k = 0; k < 2; k++) keep4(k, gn[k]); // (nobody reads the gain between here and the next half layer)
            forget();
            if (head) break;
            if (odd) {
                // ------------------------------------------------------------ the XCD's FFN activations
                gather(own + P.oU, P.fs / 4, lt, [&](int g, float (&v)[4]) { rk_put4(S.planes, 4 * g, tk, mb, HALF, v); });
                tell();
                RK_BAR();
                RK_BAR();
                RK_CHECK();
                continue;
            }
            // ---------------------------------------------------------------- token mixing
            const unsigned ngm = (unsigned)(part / 4); // groups of four columns of the XCD's mixing output
            u32x4 e0 = {}, e1 = {};
            asm volatile("" : : "v"(touched));
            // PLE: e = silu(gate) * P[tok], read with the first words of the block and kept by the thread that puts it into planes
            auto ple_words = [&]() {
                if (a.ple == 0) return true;
                e0 = xget<LD_XCD>(W, po, own); e1 = xget<LD_XCD>(W, po + 16u, own);
                return xfresh(e0, lt) && xfresh(e1, lt);
            };
            if (gdn && gIts) {
                // state rows: u = S k; S <- alpha (S - beta u k^T) + beta v k^T; o = S q
                float* St = L->S + stateAt;
                unsigned sLane = (unsigned)(lrow * HD + c4);
                asm volatile("" : "+v"(sLane));
                f32x4 st[ITS];
#pragma unroll
                for (int i = 0; i < ITS; i++) st[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(St + min(i, gIts - 1) * RPI * HD + (size_t)sLane));
                const unsigned tb = own + mixAt, gb = own + gateAt;
                u32x4 w[4];
                u32x2 vv[ITS], ga, gz;
                for (unsigned spins = 0;; spins++) {
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int k = 0; k < 4; k++) w[k] = xget<LD_XCD>(W, qLane + (unsigned)((k >> 1) * HD * 8 + (k & 1) * 16), tb);
                    ga = __builtin_amdgcn_raw_buffer_load_b64(W, 0u, gb, LD_XCD);
                    gz = __builtin_amdgcn_raw_buffer_load_b64(W, gateStep, gb, LD_XCD);
#pragma unroll
                    for (int i = 0; i < ITS; i++) vv[i] = __builtin_amdgcn_raw_buffer_load_b64(W, vLane + (unsigned)(min(i, gIts - 1) * RPI) * 8u, tb, LD_XCD);
                    bool all = ple_words();
#pragma unroll
                    for (int k = 0; k < 4; k++) all = all && xfresh(w[k], lt);
                    all = all && ga.y == lt && gz.y == lt;
#pragma unroll
                    for (int i = 0; i < ITS; i++) all = all && vv[i].y == lt;
                    if (__all(all) || give_up(spins)) break;
                }
                float qf[4] = {__uint_as_float(w[0].x), __uint_as_float(w[0].z), __uint_as_float(w[1].x), __uint_as_float(w[1].z)};
                float kf[4] = {__uint_as_float(w[2].x), __uint_as_float(w[2].z), __uint_as_float(w[3].x), __uint_as_float(w[3].z)};
                float sq = 0.f, sk = 0.f;
#pragma unroll
                for (int e = 0; e < 4; e++) { sq = fmaf(qf[e], qf[e], sq); sk = fmaf(kf[e], kf[e], sk); }
                const float rq = rsqrtf(rk_row_sum<LPR>(sq) + 1e-6f), rk = rsqrtf(rk_row_sum<LPR>(sk) + 1e-6f);
#pragma unroll
                for (int e = 0; e < 4; e++) { qf[e] *= rq; kf[e] *= rk; }
                const float za = __uint_as_float(ga.x) + side.x, zb = __uint_as_float(gz.x) + side.y;
                const float alpha = psigmoid(-za), beta = psigmoid(zb); // (exp(-softplus(z)) = sigmoid(-z))
#pragma unroll
                for (int i = 0; i < ITS; i++)
                    if (i < gIts) {
                        f32x4& s = st[i];
                        float u = s.x * kf[0];
                        u = fmaf(s.y, kf[1], u); u = fmaf(s.z, kf[2], u); u = fmaf(s.w, kf[3], u);
                        u = rk_row_sum<LPR>(u);
                        const float bu = beta * u, bv = beta * __uint_as_float(vv[i].x);
                        s.x = fmaf(alpha, s.x - bu * kf[0], bv * kf[0]); s.y = fmaf(alpha, s.y - bu * kf[1], bv * kf[1]);
                        s.z = fmaf(alpha, s.z - bu * kf[2], bv * kf[2]); s.w = fmaf(alpha, s.w - bu * kf[3], bv * kf[3]);
                        float o = s.x * qf[0];
                        o = fmaf(s.y, qf[1], o); o = fmaf(s.z, qf[2], o); o = fmaf(s.w, qf[3], o);
                        o = rk_row_sum<LPR>(o);
                        if (c4 == 0) {
                            const int c = gHead * HD + gRow + lrow + i * RPI;
                            const u32x2 z = {__float_as_uint(o), lt};
                            __builtin_amdgcn_raw_buffer_store_b64(z, W, ((((c >> 1) & 1) * ngm + (c >> 2)) * mb + gTok) * 16u + (c & 1) * 8u, own + P.oMix, ST_XCD);
                        }
                    }
                if (step == 0) St += gMove;
                if (ok)
#pragma unroll
                    for (int i = 0; i < ITS; i++)
                        if (i < gIts) *reinterpret_cast<f32x4*>(St + i * RPI * HD + (size_t)sLane) = st[i];
            } else if (!gdn && aSplit < splits()) {
                // key blocks s, s + nsplit, ... of a pair; split 0 adds this step's own row
                const int nsplit = splits(), s = aSplit, h = X + RK_XCDS * aHead, p = runi(S.pos[aTok]), nblk = (p + BR - 1) / BR;
                f32x4 pre[8] = {}, next[8]; // a block of keys: K, then V
                if (s < nblk) key_rows(p, h, s, pre);
                f32x4 gq = (f32x4)(1.f), gk = (f32x4)(1.f);
                if (a.qkNorm) {
                    gq = *reinterpret_cast<const f32x4*>(L->gq + h * HD + c4);
                    gk = *reinterpret_cast<const f32x4*>(L->gk + h * HD + c4);
                }
                const unsigned tb = own + mixAt;
                u32x4 w[6];
                for (unsigned spins = 0;; spins++) {
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int k = 0; k < 6; k++) w[k] = xget<LD_XCD>(W, qLane + (unsigned)((k >> 1) * HD * 8 + (k & 1) * 16), tb);
                    bool all = ple_words();
#pragma unroll
                    for (int k = 0; k < 6; k++) all = all && xfresh(w[k], lt);
                    if (__all(all) || give_up(spins)) break;
                }
                auto vec = [&](int k) { return f32x4{__uint_as_float(w[k].x), __uint_as_float(w[k].z), __uint_as_float(w[k + 1].x), __uint_as_float(w[k + 1].z)}; };
                auto norm_rope = [&](f32x4 v, const f32x4& g) { // inference.cu:52-134
                    if (a.qkNorm) {
                        float ss = v.x * v.x;
                        ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss);
                        const float ri = rsqrtf(rk_row_sum<LPR>(ss) * (1.0f / HD) + 1e-8f);
                        v.x = g.x * (v.x * ri); v.y = g.y * (v.y * ri); v.z = g.z * (v.z * ri); v.w = g.w * (v.w * ri);
                    }
                    return f32x4{side.x * v.x - side.y * v.y, side.y * v.x + side.x * v.y, side.z * v.z - side.w * v.w, side.w * v.z + side.z * v.w};
                };
                const f32x4 q = norm_rope(vec(0), gq), kn = norm_rope(vec(2), gk), vn = vec(4);
                const float scale = 1.0f / sqrtf((float)HD);
                auto dot = [&](const f32x4& k) {
                    float z = k.x * q.x;
                    z = fmaf(k.y, q.y, z); z = fmaf(k.z, q.z, z); z = fmaf(k.w, q.w, z);
                    return rk_row_sum<LPR>(z) * scale;
                };
                float m = -1.0e30f, lsum = 0.f; // of this lane's row group
                f32x4 acc = (f32x4)(0.f);
                const float sn = dot(kn);
                if (s == 0 && lrow == 0) {
                    m = sn; lsum = 1.f; acc = vn;
                    if (ok) {
                        const size_t o = key_base(h, p / BR) + (size_t)(p % BR) * d + c4;
                        *reinterpret_cast<f32x4*>(L->K + o) = kn;
                        *reinterpret_cast<f32x4*>(L->V + o) = vn;
                    }
                }
                auto keys = [&](int j, auto& kv) __attribute__((always_inline)) {
                    float sc[4];
#pragma unroll
                    for (int it = 0; it < 4; it++) {
                        sc[it] = dot(kv[it]);
                        sc[it] = j * BR + it * RPI + lrow < p ? sc[it] : -1.0e30f;
                    }
                    const float mn = fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), m), corr = expf(m - mn);
                    lsum *= corr;
                    acc *= corr;
#pragma unroll
                    for (int it = 0; it < 4; it++) {
                        const float e = j * BR + it * RPI + lrow < p ? expf(sc[it] - mn) : 0.f;
                        lsum += e;
                        acc.x = fmaf(e, kv[it + 4].x, acc.x); acc.y = fmaf(e, kv[it + 4].y, acc.y);
                        acc.z = fmaf(e, kv[it + 4].z, acc.z); acc.w = fmaf(e, kv[it + 4].w, acc.w);
                    }
                    m = mn;
                };
                int j = s;
                while (j < nblk) { // the next block's loads before this one's arithmetic (no next one: the same again, from the cache)
                    const int j1 = j + nsplit;
                    key_rows(p, h, j1 < nblk ? j1 : j, next);
                    __builtin_amdgcn_sched_barrier(0);
                    keys(j, pre);
                    __builtin_amdgcn_sched_barrier(0);
                    j = j1;
#pragma unroll
                    for (int k = 0; k < 8; k++) pre[k] = next[k];
                }
#pragma unroll
                for (int o = LPR; o < 64; o <<= 1) { // the row groups of the wave
                    const float mo = __shfl_xor(m, o, 64), lo = __shfl_xor(lsum, o, 64);
                    f32x4 ao;
                    ao.x = __shfl_xor(acc.x, o, 64); ao.y = __shfl_xor(acc.y, o, 64); ao.z = __shfl_xor(acc.z, o, 64); ao.w = __shfl_xor(acc.w, o, 64);
                    const float mm = fmaxf(m, mo), ca = expf(m - mm), cb = expf(mo - mm);
                    lsum = lsum * ca + lo * cb;
                    acc = acc * ca + ao * cb;
                    m = mm;
                }
                if (lane < LPR) {
                    const unsigned o = (((unsigned)(s * 2) * ngm + aHead * LPR + lane) * mb + aTok) * 16u;
                    xput<ST_XCD>(W, o, own + P.oPart, acc.x, acc.y, lt);
                    xput<ST_XCD>(W, o + ngm * mb * 16u, own + P.oPart, acc.z, acc.w, lt);
                    if (lane == 0) xput<ST_XCD>(W, (unsigned)((s * nh + aHead) * mb + aTok) * 16u, own + P.oMl, m, lsum, lt);
                }
            } else if (a.ple > 0) {
                for (unsigned spins = 0;; spins++) {
                    asm volatile("" ::: "memory");
                    if (__all(ple_words()) || give_up(spins)) break;
                }
            }
            if (ple) {
                float pv[4];
                pt.get(pv);
                S.ple[gePle * mb + tk] = f32x4{psilu(__uint_as_float(e0.x)) * pv[0], psilu(__uint_as_float(e0.z)) * pv[1],
                                                      psilu(__uint_as_float(e1.x)) * pv[2], psilu(__uint_as_float(e1.z)) * pv[3]};
            }
            // ---------------------------------------------------------------- the XCD's mixing output and PLE columns into planes
            forget();
            if (a.ple > 0 && act && g0 < KE / 4) { // (the other XCDs' columns of the chunk count as zero here)
                const int ge = g0 - gPle;
                const bool in = ge >= 0 && ge < pleX / 4;
                const f32x4 e = in ? S.ple[ge * mb + tk] : (f32x4)(0.f);
                const float v[4] = {e.x, e.y, e.z, e.w};
                rk_put4(S.planes, part + 4 * g0, tk, mb, HALF, v);
            }
            if (gdn) {
                gather(own + P.oMix, (int)ngm, lt, [&](int g, float (&v)[4]) { rk_put4(S.planes, 4 * g, tk, mb, HALF, v); });
            } else {
                const int nsplit = splits();
#pragma unroll 1
                for (int gr = g0; runi(gr) < (int)ngm; gr += G) {
                    const int g = min(gr, (int)ngm - 1), hl = g / LPR;
                    float m = -1.0e30f, den = 0.f, num[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                    for (int s0 = 0; s0 < nsplit; s0 += 4) { // four splits at a time
                        u32x4 w0[4], w1[4], ml[4];
                        for (unsigned spins = 0;; spins++) {
                            asm volatile("" ::: "memory");
                            bool all = true;
#pragma unroll
                            for (int k = 0; k < 4; k++) {
                                const int s = min(s0 + k, nsplit - 1);
                                const unsigned o = (unsigned)(g * mb + tk) * 16u, so = own + P.oPart + (unsigned)(s * 2 * mb) * ngm * 16u;
                                w0[k] = xget<LD_XCD>(W, o, so);
                                w1[k] = xget<LD_XCD>(W, o, so + ngm * mb * 16u);
                                ml[k] = xget<LD_XCD>(W, (unsigned)(hl * mb + tk) * 16u, own + P.oMl + (unsigned)(s * nh * mb) * 16u);
                            }
#pragma unroll
                            for (int k = 0; k < 4; k++) all = all && xfresh(w0[k], lt) && xfresh(w1[k], lt) && xfresh(ml[k], lt);
                            if (__all(all) || give_up(spins)) break;
                        }
                        float mn = m;
#pragma unroll
                        for (int k = 0; k < 4; k++) mn = s0 + k < nsplit ? fmaxf(mn, __uint_as_float(ml[k].x)) : mn;
                        const float corr = expf(m - mn);
                        den *= corr;
#pragma unroll
                        for (int e = 0; e < 4; e++) num[e] *= corr;
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            const float c = s0 + k < nsplit ? expf(__uint_as_float(ml[k].x) - mn) : 0.f;
                            den = fmaf(c, __uint_as_float(ml[k].z), den);
                            num[0] = fmaf(c, __uint_as_float(w0[k].x), num[0]); num[1] = fmaf(c, __uint_as_float(w0[k].z), num[1]);
                            num[2] = fmaf(c, __uint_as_float(w1[k].x), num[2]); num[3] = fmaf(c, __uint_as_float(w1[k].z), num[3]);
                        }
                        m = mn;
                    }
                    const float inv = 1.0f / den;
#pragma unroll
                    for (int e = 0; e < 4; e++) num[e] *= inv;
                    if (a.gating) { // inference.cu:241-250 (these words are older than the partial results)
                        const unsigned o = (unsigned)(tk * P.rowsQ + hl * npAttn * HD + 3 * HD + (g * 4) % HD) * 8u;
                        u32x4 z0, z1;
                        for (unsigned spins = 0;; spins++) {
                            asm volatile("" ::: "memory");
                            z0 = xget<LD_XCD>(W, o, own); z1 = xget<LD_XCD>(W, o + 16u, own);
                            if (__all(xfresh(z0, lt) && xfresh(z1, lt)) || give_up(spins)) break;
                        }
                        num[0] *= psigmoid(__uint_as_float(z0.x)); num[1] *= psigmoid(__uint_as_float(z0.z));
                        num[2] *= psigmoid(__uint_as_float(z1.x)); num[3] *= psigmoid(__uint_as_float(z1.z));
                    }
                    if (act && gr < (int)ngm) rk_put4(S.planes, 4 * g, tk, mb, HALF, num);
                }
            }
            tell();
            RK_BAR();
            RK_BAR();
        }
        const unsigned lt = P.tagBase + (unsigned)(step * (NL + 1) + NL + 1);
        // the pick: token slot s is decided by workgroup s out of two candidates per workgroup, lowest index on ties
        const int gw = r * RK_XCDS + X;
        if (cw == 0) {
            if (gw < a.nseq) {
                constexpr int N = 2 * RK_XCDS * RK_PER / 64;
                const unsigned base = P.oAmax + (unsigned)(gw * 2 * RK_XCDS * RK_PER) * 16u;
                u32x4 c[N];
                for (unsigned spins = 0;; spins++) {
                    asm volatile("" ::: "memory");
                    bool all = true;
#pragma unroll
                    for (int k = 0; k < N; k++) c[k] = xget<LD_CROSS>(W, (unsigned)(k * 64 + lane) * 16u, base);
#pragma unroll
                    for (int k = 0; k < N; k++) all = all && xfresh(c[k], lt);
                    if (__all(all) || give_up(spins)) break;
                }
                float v = -3.0e38f;
                int i = 0x7fffffff;
#pragma unroll
                for (int k = 0; k < N; k++) {
                    const float v2 = __uint_as_float(c[k].x);
                    const int i2 = (int)c[k].z;
                    if (v2 > v || (v2 == v && i2 < i)) { v = v2; i = i2; }
                }
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    const float v2 = __shfl_xor(v, o, 64);
                    const int i2 = __shfl_xor(i, o, 64);
                    if (v2 > v || (v2 == v && i2 < i)) { v = v2; i = i2; }
                }
                if (i < 0 || i >= a.vocab) i = 0; // only reachable with non-finite logits
                if (lane == 0 && ok) {
                    xput<ST_CROSS>(W, (unsigned)gw * 16u, P.oTok, __int_as_float(i), 0.f, lt);
                    const int row = stepRow + step, seq = S.seq[gw];
                    if (row >= 0 && row < a.outCapacity) a.outIds[(size_t)row * a.nseq + gw] = i;
                    if (step + 1 == P.steps) {
                        a.nextTok[seq] = i;
                        ((int*)a.tok)[gw] = i;
                        a.pos[seq] = S.pos[gw] + 1;
                        if (gw == 0) *a.stepCounter = stepRow + P.steps;
                    }
                }
            }
            if (step + 1 < P.steps) {
                u32x4 c;
                for (unsigned spins = 0;; spins++) {
                    asm volatile("" ::: "memory");
                    c = xget<LD_CROSS>(W, (unsigned)min(lane, a.nseq - 1) * 16u, P.oTok);
                    if (__all(xfresh(c, lt)) || give_up(spins)) break;
                }
                if (lane < mb && ok) { S.tok[lane] = (int)c.x; S.pos[lane] += 1; }
            }
            tell();
        }
    }
}

// ------------------------------------------------------------------------------------------------ workers
template <typename WT, int HD>
__device__ __forceinline__ void rk_worker(const RanksArgs& P, const RkShared& S, int X0, int r0) {
    typedef RkCfg<WT, HD> C;
    typedef RkOp<WT> Op;
    constexpr int KE = Op::KE, SUB = Op::SUB, CA = C::CA, TW = C::TW, NS = RK_WORK / TW, CO = C::CO, CW = C::CW, NTB = C::NTB;
    constexpr int C2 = NTB ? (CO > CW / 2 ? CO : CW / 2) : (CO > CW ? CO : CW), SLOTS = NTB ? 3 : 2;
    const StepArgs& a = P.a;
    const int d = a.dim, wave = runi(threadIdx.x >> 6), NL = P.NL, mb = a.nseq, fs = P.fs, rowsQ = P.rowsQ;
    int X = X0, r = r0, lane = threadIdx.x & 63;
    const int nh = (a.heads - X0 + RK_XCDS - 1) / RK_XCDS, pleX = a.ple / RK_XCDS, npAttn = 3 + (a.gating ? 1 : 0);
    const int nch = d / KE, ko = nh * (HD / KE) + (a.ple > 0 ? 1 : 0);
    const int slot2 = wave / NS, part2 = wave % NS; // output and down projection: tile r + 32 slot2, chunks part2, part2 + NS, ...
    const unsigned area = P.area, oXP = P.oXP, oHP = P.oHP, oU = P.oU;
    const rsrc_t W = __builtin_amdgcn_make_buffer_rsrc(P.xw, 0, P.xwBytes, 0x00027000);
    LayerPtr layers = (LayerPtr)P.layers;
    auto own = [&]() { return (unsigned)X * area; };

    RkW<WT> w1[2][CA], w1b[CA], w2[C2];
    auto chunk = [&](RkW<WT>& w, const unsigned char* m, size_t index) __attribute__((always_inline)) { // chunk `index` of a packed matrix
        unsigned lb = lane * 16u;
        asm volatile("" : "+v"(lb));
        const unsigned char* p = m + index * 2048;
        const u32x4 *q0 = reinterpret_cast<const u32x4*>(p + (size_t)lb), *q1 = reinterpret_cast<const u32x4*>(p + (size_t)lb + 1024);
        if constexpr (sizeof(WT) == 2) { w.raw[0] = __builtin_nontemporal_load(q0); w.raw[1] = __builtin_nontemporal_load(q1); }
        else { w.raw[0] = *q0; w.raw[1] = *q1; }
    };
    auto tile1 = [&](RkW<WT> (&w)[CA], const unsigned char* m, int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < CA; i++) chunk(w[i], m, (size_t)tile * nch + min(wave + RK_WORK * i, nch - 1));
    };
    // tile number idx of the first phase of layer L on this XCD (rk_tilesA)
    auto tileA = [&](LayerPtr L, int idx) {
        constexpr int HT = HD / 16;
        const int np = L->kind != MLH_KIND_ATTENTION ? 3 : npAttn;
        int idxPle, idxG;
        const int n = rk_tilesA<HD>(L, a.heads, a.ple, npAttn, nh, idxPle, idxG);
        idx = min(idx, n - 1);
        if (idx < idxPle) {
            const int hl = idx >= np * HT ? 1 : 0, rem = idx - hl * (np * HT), p = rem / HT, i = rem - p * HT; // (two heads at most)
            const int off = p == 0 ? 0 : p == 1 ? L->offK : p == 2 ? L->offV : L->offG;
            return ((off + (X + RK_XCDS * hl) * HD) >> 4) + i;
        }
        if (idx < idxG) return (L->offPle + X * pleX) >> 4;
        return (L->offGa >> 4) + idx - idxG;
    };
    auto issueA = [&](LayerPtr L, bool lm) __attribute__((always_inline)) { // (lm: the LM head's first tiles instead; one set of loads with selected addresses)
        const int last = (a.vocab + 15) / 16 - 1, gw = r * RK_XCDS + X;
        const unsigned char* m = lm ? P.ER : (const unsigned char*)L->WaR;
#pragma unroll
        for (int k = 0; k < 2; k++) tile1(w1[k], m, lm ? min(gw + k * RK_XCDS * RK_PER, last) : tileA(L, r + RK_PER * k));
    };
    auto issueO = [&](LayerPtr L) __attribute__((always_inline)) {
        constexpr int cph = HD / KE;
        const int total = (L->ad + a.ple) / KE, tile = min(r + RK_PER * slot2, d / 16 - 1);
#pragma unroll
        for (int i = 0; i < CO; i++) {
            const int c = min(part2 + NS * i, ko - 1), hl = c / cph;
            const int gc = c < nh * cph ? (X + RK_XCDS * hl) * cph + c - hl * cph : (L->ad + X * pleX) / KE;
            chunk(w2[i], (const unsigned char*)L->WoR, (size_t)tile * total + gc);
        }
    };
    auto issue13 = [&](LayerPtr L) __attribute__((always_inline)) {
        const int n = fs / 8;
        const unsigned char* m = (const unsigned char*)L->W13R;
#pragma unroll
        for (int k = 0; k < 2; k++) tile1(w1[k], m, X * n + min(r + RK_PER * k, n - 1));
        if constexpr (NTB > 0) tile1(w1b, m, X * n + min(r + RK_PER * 2, n - 1));
    };
    auto issueW2 = [&](LayerPtr L, RkW<WT>* dst, int i0, int cnt) __attribute__((always_inline)) {
        const int n = fs / KE, tile = min(r + RK_PER * slot2, d / 16 - 1);
#pragma unroll
        for (int i = 0; i < CW; i++)
            if (i >= i0 && i < i0 + cnt) chunk(dst[i - i0], (const unsigned char*)L->W2R, (size_t)tile * (RK_XCDS * n) + X * n + min(part2 + NS * i, n - 1));
    };
    // operand planes of 32-wide step kb
    auto operand = [&](u32x4 (&v)[3], int kb) __attribute__((always_inline)) {
        const int stride = 64 * mb;
        const unsigned char* p = S.planes + kb * 3 * stride + ((lane >> 4) * mb + min(lane & 15, mb - 1)) * 16;
#pragma unroll
        for (int pl = 0; pl < 3; pl++) v[pl] = *reinterpret_cast<const u32x4*>(p + pl * stride);
    };
    auto red = [&](int buf, int slot, int part) -> f32x4& { return S.red[((buf * SLOTS + slot) * RK_WORK + part) * 64 + lane]; };
    auto red2 = [&](int buf, int slot, int part) -> f32x4& { return S.red[(buf * SLOTS * RK_WORK + slot * NS + part) * 64 + lane]; };
    auto sum = [&](int buf, int slot) { // (all reads out before the first addition)
        f32x4 t[RK_WORK];
#pragma unroll
        for (int k = 0; k < RK_WORK; k++) t[k] = red(buf, slot, k);
        __builtin_amdgcn_sched_barrier(0);
        return ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
    };
    auto sum2 = [&](int buf, int slot) {
        f32x4 t[NS];
#pragma unroll
        for (int k = 0; k < NS; k++) t[k] = red2(buf, slot, k);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 v = t[0];
#pragma unroll
        for (int k = 1; k < NS; k++) v += t[k];
        return v;
    };

    // fp32 weights are split into planes before the barrier they wait at (of two tiles, the first; pinned: left alone the compiler moves the split
    // behind the barrier)
    Op op1[CA], op2[C2];
    unsigned ahead = 0; // (a load that only touches)
    auto ready = [&](Op& o, RkW<WT>& w, bool real) __attribute__((always_inline)) { // (not real: past the last chunk, counts as zero)
        if constexpr (sizeof(WT) == 2) return;
        if (!real) w.raw[0] = w.raw[1] = (u32x4)(0u);
        o.from(w);
        o.pin();
    };
    auto ready1 = [&](int n1) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < CA; i++) ready(op1[i], w1[0][i], wave + RK_WORK * i < nch);
        if (sizeof(WT) == 4 && wave + RK_WORK * (CA - 1) >= nch)
#pragma unroll
            for (int i = 0; i < CA; i++)
                if (wave + RK_WORK * i >= nch) {
                    w1[1][i].raw[0] = w1[1][i].raw[1] = (u32x4)(0u);
                    if constexpr (NTB > 0) w1b[i].raw[0] = w1b[i].raw[1] = (u32x4)(0u);
                }
    };
    // n1 tiles over the whole width -> red
    auto multiplyT = [&](auto tilesTag, int buf) __attribute__((always_inline)) { // fp32 weights: one or two tiles
        constexpr int T = decltype(tilesTag)::value, CH = T == 1 ? 2 : 1; // accumulator chains per tile
        f32x4 acc[T][CH];
#pragma unroll
        for (int k = 0; k < T; k++)
#pragma unroll
            for (int c = 0; c < CH; c++) acc[k][c] = (f32x4)(0.f);
        u32x4 v[2][3]; // operand planes of a step and of the next one
        operand(v[0], min(wave, nch - 1));
#pragma unroll
        for (int i = 0; i < CA; i++) {
            if (i + 1 < CA) operand(v[(i + 1) & 1], min(wave + RK_WORK * (i + 1), nch - 1));
            __builtin_amdgcn_sched_barrier(0);
            rk_mul(w1[0][i], op1[i], 0, v[i & 1], acc[0][0], acc[0][CH - 1]);
            if constexpr (T > 1) {
                Op o;
                RkW<WT> w = w1[1][i];
                asm volatile("" : "+v"(w.raw[0]), "+v"(w.raw[1]));
                o.from(w);
                rk_mul(w, o, 0, v[i & 1], acc[T > 1 ? 1 : 0][0], acc[T > 1 ? 1 : 0][CH - 1]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int k = 0; k < T; k++) red(buf, k, wave) = CH == 2 ? acc[k][0] + acc[k][CH - 1] : acc[k][0];
    };
    auto multiplyHalf = [&](int buf, int n1) __attribute__((always_inline)) { // two-byte weights: up to three tiles, as they come
        f32x4 acc[SLOTS];
#pragma unroll
        for (int k = 0; k < SLOTS; k++) acc[k] = (f32x4)(0.f);
#pragma unroll
        for (int i = 0; i < CA; i++)
            if (wave + RK_WORK * i < nch)
#pragma unroll
                for (int p = 0; p < SUB; p++) {
                    u32x4 v[3];
                    operand(v, (wave + RK_WORK * i) * SUB + p);
                    rk_mul(w1[0][i], op1[i], p, v, acc[0], acc[0]);
                    if (n1 > 1) rk_mul(w1[1][i], op1[i], p, v, acc[1], acc[1]);
                    if (SLOTS > 2 && n1 > 2) rk_mul(w1b[i], op1[i], p, v, acc[SLOTS - 1], acc[SLOTS - 1]);
                }
#pragma unroll
        for (int k = 0; k < SLOTS; k++)
            if (k < n1) red(buf, k, wave) = acc[k];
    };
    auto multiply1 = [&](int buf, int n1) __attribute__((always_inline)) {
        if constexpr (sizeof(WT) == 2) multiplyHalf(buf, n1);
        else if (n1 <= 1) multiplyT(std::integral_constant<int, 1>(), buf);
        else multiplyT(std::integral_constant<int, 2>(), buf);
    };

    issueA(layers + NL - 1, false);
    issueO(layers + NL - 1);
    for (int step = 0; step < P.steps; step++) {
        RK_BAR(); // tokens, positions, first gain
        RK_CHECK();
#pragma unroll 1
        for (int l = 0; l < NL; l++) {
            RK_FORGET();
            const LayerPtr L = layers + (NL - 1 - l), Ln = layers + (l + 1 < NL ? NL - 2 - l : NL - 1);
            const unsigned lt = P.tagBase + (unsigned)(step * (NL + 1) + l + 1);
            const bool last = l + 1 == NL;
            // tiles over several workers: chunks part2 + NS i < n of w2 (op2), then of w1b; partial tiles across the XCDs
            auto multiply2 = [&](auto countTag, int n) __attribute__((always_inline)) {
                constexpr int CNT = decltype(countTag)::value;
                f32x4 acc[2] = {(f32x4)(0.f), (f32x4)(0.f)};
                if constexpr (sizeof(WT) == 2) {
#pragma unroll
                    for (int i = 0; i < CNT; i++)
                        if (part2 + NS * i < n)
#pragma unroll
                            for (int p = 0; p < SUB; p++) {
                                u32x4 v[3];
                                operand(v, (part2 + NS * i) * SUB + p);
                                if (i < C2) rk_mul(w2[i < C2 ? i : 0], op2[0], p, v, acc[0], acc[1]);
                                else rk_mul(w1b[i < C2 || NTB == 0 ? 0 : i - C2], op2[0], p, v, acc[0], acc[1]);
                            }
                } else {
                    u32x4 v[2][3];
                    operand(v[0], min(part2, n - 1));
#pragma unroll
                    for (int i = 0; i < CNT; i++) {
                        if (i + 1 < CNT) operand(v[(i + 1) & 1], min(part2 + NS * (i + 1), n - 1));
                        __builtin_amdgcn_sched_barrier(0);
                        rk_mul(w2[i < C2 ? i : 0], op2[i < C2 ? i : 0], 0, v[i & 1], acc[0], acc[1]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                red2(0, slot2, part2) = acc[0] + acc[1];
            };
            auto publish2 = [&](unsigned to) __attribute__((always_inline)) {
                const int tile = r + RK_PER * wave, t16 = lane & 15, q = lane >> 4;
                if (wave < TW && tile < d / 16 && t16 < mb) {
                    const f32x4 v = sum2(0, wave);
                    const unsigned base = own() + to, o = (unsigned)((tile * 4 + q) * mb + t16) * 16u;
                    xput<ST_CROSS>(W, o, base, v.x, v.y, lt);
                    xput<ST_CROSS>(W, o, base + (unsigned)(d / 4 * mb) * 16u, v.z, v.w, lt);
                }
            };
            const int t16 = lane & 15, q = lane >> 4;
            // ---------------------------------------------------------------- first phase (inference.cu:388-465)
            {
                int ip, ig;
                const int n = rk_tilesA<HD>(L, a.heads, a.ple, npAttn, nh, ip, ig), n1 = r >= n ? 0 : r + RK_PER < n ? 2 : 1;
                ready1(n1);
                RK_BAR();
                multiply1(0, n1);
                RK_BAR();
                if (wave < n1 && t16 < mb) {
                    const f32x4 v = sum(0, wave) * S.rms[t16];
                    const unsigned o = (unsigned)(t16 * rowsQ + (r + RK_PER * wave) * 16 + 4 * q) * 8u;
                    xput<ST_XCD>(W, o, own(), v.x, v.y, lt);
                    xput<ST_XCD>(W, o, own() + 16u, v.z, v.w, lt);
                }
                issue13(L);
            }
            RK_FORGET();
            // ---------------------------------------------------------------- output projection over the XCD's columns (inference.cu:582-610)
            {
#pragma unroll
                for (int i = 0; i < CO; i++) ready(op2[i], w2[i], part2 + NS * i < ko);
                RK_BAR();
                multiply2(std::integral_constant<int, CO>(), ko);
                RK_BAR();
                publish2(oHP);
                issueW2(L, w2, 0, C2);
                if constexpr (CW > C2) { // the rest has no registers before gate / up is done: into the L2 meanwhile, 64 lines a load
                    const int n = fs / KE, tile = min(r + RK_PER * slot2, d / 16 - 1), line = min(lane, (CW - C2) * 16 - 1);
                    const int c = min(part2 + NS * (C2 + line / 16), n - 1);
                    ahead = *reinterpret_cast<const unsigned*>((const unsigned char*)L->W2R + ((size_t)tile * (RK_XCDS * n) + X * n + c) * 2048 + (line % 16) * 128);
                }
            }
            RK_FORGET();
            // ---------------------------------------------------------------- gate / up of the XCD's FFN units (inference.cu:612-672)
            {
                const int n = fs / 8, n1 = r >= n ? 0 : r + 2 * RK_PER < n ? 3 : r + RK_PER < n ? 2 : 1;
                ready1(n1);
                RK_BAR();
                multiply1(0, n1);
                if constexpr (CW > C2) {
                    asm volatile("" : : "v"(ahead));
                    issueW2(L, w1b, C2, CW - C2);
                }
                RK_BAR();
                if (wave < n1 && t16 < mb) {
                    const f32x4 v = sum(0, wave) * S.rms[t16];
                    const int k = r + RK_PER * wave;
                    xput<ST_XCD>(W, (unsigned)(((q & 1) * (fs / 4) + 2 * k + (q >> 1)) * mb + t16) * 16u, own() + oU, psilu(v.x) * v.y, psilu(v.z) * v.w, lt);
                }
                issueA(Ln, last);
            }
            RK_FORGET();
            // ---------------------------------------------------------------- down projection over the XCD's columns (inference.cu:675-699)
            {
#pragma unroll
                for (int i = 0; i < C2; i++) ready(op2[i], w2[i], part2 + NS * i < fs / KE);
                RK_BAR();
                multiply2(std::integral_constant<int, CW>(), fs / KE);
                RK_BAR();
                publish2(oXP);
                RK_CHECK();
                issueO(Ln);
            }
        }
        RK_FORGET();
        // -------------------------------------------------------------------- LM head (inference.cu:705-743)
        {
            const unsigned lt = P.tagBase + (unsigned)(step * (NL + 1) + NL + 1);
            constexpr int GRID = RK_XCDS * RK_PER;
            const int tiles = (a.vocab + 15) / 16, batches = (tiles + 2 * GRID - 1) / (2 * GRID), gw = r * RK_XCDS + X, t16 = lane & 15, q = lane >> 4;
            float best = -3.0e38f;
            int bi = 0x7fffffff;
            RK_BAR();
#pragma unroll 1
            for (int k = 0; k <= batches; k++) { // two tiles at a time; the sums of a batch while the next is multiplied
                if (k > 0 && wave < 2) {
                    const int tile = gw + (2 * k - 2 + wave) * GRID;
                    if (tile < tiles && t16 < mb) {
                        const f32x4 v = sum((k - 1) & 1, wave) * S.rms[t16];
                        const int n = tile * 16 + 4 * q;
                        float* c = a.logits + (size_t)S.seq[t16] * a.vocab + n;
                        if ((a.vocab & 3) == 0 && n + 3 < a.vocab) *reinterpret_cast<f32x4*>(c) = v;
                        else
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                if (n + e < a.vocab) c[e] = v[e];
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (n + e < a.vocab && v[e] > best) { best = v[e]; bi = n + e; }
                    }
                    if (k == batches) {
#pragma unroll
                        for (int o = 16; o < 64; o <<= 1) {
                            const float ov = __shfl_xor(best, o, 64);
                            const int oi = __shfl_xor(bi, o, 64);
                            if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
                        }
                        if (q == 0 && t16 < mb) xput<ST_CROSS>(W, (unsigned)(t16 * 2 * GRID + gw * 2 + wave) * 16u, P.oAmax, best, __int_as_float(bi), lt);
                    }
                }
                if (k < batches) {
                    const int n1 = gw + 2 * k * GRID >= tiles ? 0 : gw + (2 * k + 1) * GRID < tiles ? 2 : 1;
                    ready1(n1);
                    if constexpr (sizeof(WT) == 2) multiplyHalf(k & 1, n1);
                    else multiplyT(std::integral_constant<int, 2>(), k & 1); // (a tile past the last one: the last one again, dropped)
                    // the next two tiles, or the next step's first phase
                    const LayerPtr L0 = layers + NL - 1;
                    const bool done = k + 1 == batches;
                    const unsigned char* m = done ? (const unsigned char*)L0->WaR : P.ER;
#pragma unroll
                    for (int j = 0; j < 2; j++) tile1(w1[j], m, done ? tileA(L0, r + RK_PER * j) : min(gw + (2 * k + 2 + j) * GRID, tiles - 1));
                    RK_BAR();
                }
            }
        }
    }
}

template <typename WT, int HD>
__global__ void __launch_bounds__(RK_THREADS) k_decode_ranks(RanksArgs P) {
    extern __shared__ __align__(16) unsigned char lds[];
    constexpr int SLOTS = RkCfg<WT, HD>::NTB ? 3 : 2;
    RkShared S;
    S.planes = lds;
    S.red = reinterpret_cast<f32x4*>(lds + P.planeBytes);
    S.resid = reinterpret_cast<float2*>(S.red + 2 * SLOTS * RK_WORK * 64);
    S.sq = reinterpret_cast<float*>(S.resid + RK_CT);
    S.rms = S.sq + RK_CT;
    S.ple = reinterpret_cast<f32x4*>(S.rms + 16);
    S.gain = reinterpret_cast<float*>(S.ple + 64);
    S.tok = reinterpret_cast<int*>(S.gain + P.a.dim);
    S.pos = S.tok + 16;
    S.seq = S.pos + 16;
    S.ctl = S.seq + 16;
    if (threadIdx.x < P.a.nseq) {
        const int s = P.a.sidx[threadIdx.x];
        S.tok[threadIdx.x] = P.a.tok[threadIdx.x];
        S.seq[threadIdx.x] = s;
        S.pos[threadIdx.x] = P.a.pos[s];
    }
    if (threadIdx.x < 64) {
        unsigned xcc, rank;
        const unsigned code = rk_meeting(P.xcdCount, xcc, rank);
        if (threadIdx.x == 0) {
            if (code) astu(P.abortFlag, code);
            S.ctl[0] = code ? 1 : 0;
            S.ctl[2] = (int)xcc;
            S.ctl[3] = (int)rank;
        }
    }
    lds_barrier();
    if (runi(S.ctl[0])) return;
    const int X = runi(S.ctl[2]), r = runi(S.ctl[3]);
    if (threadIdx.x >= RK_WORK * 64) {
        __builtin_amdgcn_s_setprio(3);
        rk_communicator<WT, HD>(P, S, X, r);
    } else {
        rk_worker<WT, HD>(P, S, X, r);
    }
}

// the meeting's words and the abort flag, before every launch
__global__ void k_ranks_prep(unsigned* abortFlag, unsigned* xcdCount, unsigned startCount) {
    if (threadIdx.x == 0) *abortFlag = 0u;
    if (threadIdx.x <= RK_XCDS) xcdCount[threadIdx.x] = threadIdx.x < RK_XCDS ? startCount : 0u;
}
// states of sequences that are in their second place, to the first (x: pieces, y: layer, z: sequence)
__global__ void __launch_bounds__(256) k_ranks_settle(const LayerDev* layers, size_t otherAt4, unsigned long long which, size_t per4) {
    f32x4* S = reinterpret_cast<f32x4*>(layers[blockIdx.y].S);
    if (!S || !(which >> blockIdx.z & 1)) return;
    S += blockIdx.z * per4;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < per4; i += (size_t)gridDim.x * 256) S[i] = S[otherAt4 + i];
}
__global__ void k_ranks_positions(const int* lens, int* pos, int nseq) {
    if (threadIdx.x < nseq) pos[threadIdx.x] = lens[threadIdx.x];
}
__global__ void k_ranks_zero(u32x4* p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = (u32x4)(0u);
}

// ----------------------------------------------------------------------------
// host side
// ----------------------------------------------------------------------------
struct RanksPlan { // how a launch of n sequences is laid out
    int planeBytes, rowsQ;
    size_t lds, words;
    unsigned area, oPart, oMl, oMix, oX, oH, oU, oXP, oHP, oAmax, oTok;
};

static bool ranks_plan(const mlh_ctx* c, int n, RanksPlan& p) {
    const mlh_hparams& hp = c->hp;
    const bool half = hp.weightDtype == MLH_DTYPE_BF16;
    const int d = hp.dim, fs = hp.ffnDim / RK_XCDS, ke = half ? 64 : 32, slots = half ? 3 : 2, nh = (hp.attnHeads + RK_XCDS - 1) / RK_XCDS;
    const int cols = std::max(std::max(d, fs), nh * hp.headDim + ke);
    p.planeBytes = cols * 6 * n;
    p.lds = (size_t)p.planeBytes + 2 * slots * RK_WORK * 1024 + RK_CT * 8 + (RK_CT + 16 + 64 * 4 + d + 3 * 16 + 16) * 4;
    // n tokens are the columns of one MFMA; a residual element per communicator thread, state rows of a pair of a head and a sequence per workgroup,
    // a group of the PLE chunk's columns per thread
    if (n > MLH_RANKS_MAX_SEQS || n > RK_CT / (d / 64) || n * nh * hp.headDim > RK_PER * 64 || n > RK_CT / (ke / 4) || p.lds > RK_LDS) return false;
    p.lds = std::max(p.lds, (size_t)RK_LDS / 2 + 1024); // one workgroup per compute unit
    int tiles = 0;
    for (const LayerDev& L : c->layers) {
        const bool gdn = L.kind != MLH_KIND_ATTENTION;
        int t = nh * (gdn || !hp.queryGating ? 3 : 4) * (hp.headDim / 16) + (hp.pleDim > 0 ? 1 : 0);
        if (gdn) t += (L.offGb + hp.gdnHeads - 1) / 16 - L.offGa / 16 + 1;
        tiles = std::max(tiles, t);
    }
    if (tiles > 2 * RK_PER) return false;
    p.rowsQ = tiles * 16;
    size_t at = 0;
    auto place = [&](size_t bytes) { const size_t o = at; at += (bytes + 255) / 256 * 256; return (unsigned)o; };
    place((size_t)p.rowsQ * n * 8);
    p.oPart = place((size_t)RK_COMM * RK_PER * hp.headDim * 8);
    p.oMl = place((size_t)RK_COMM * RK_PER * 16);
    p.oMix = place((size_t)nh * hp.headDim * n * 8);
    p.oX = place((size_t)d * n * 8);
    p.oH = place((size_t)d * n * 8);
    p.oXP = place((size_t)d * n * 8);
    p.oHP = place((size_t)d * n * 8);
    p.oU = place((size_t)fs * n * 8);
    p.area = (unsigned)at;
    at *= RK_XCDS;
    p.oAmax = place((size_t)n * 2 * RK_XCDS * RK_PER * 16);
    p.oTok = place((size_t)n * 16);
    p.words = at;
    return at < ((size_t)1 << 31);
}

// Floats of one sequence's states of a layer (0: no layer has states).
static size_t state_floats(const mlh_ctx* c) {
    for (const LayerDev& L : c->layers)
        if (L.kind == MLH_KIND_GDN) return (size_t)c->hp.gdnHeads * c->hp.gdnDk * c->hp.gdnDv;
    return 0;
}

// Sequences whose states have a second place, in a model that the kernel covers: those of a launch of this kernel or of kernels_wide.hip.
// (Both places of all states lie within 32-bit offsets; where 64 more do not, 16 may.)
static bool places_fit(const mlh_ctx* c, int others) { return (c->hp.maxSeqs + others) * state_floats(c) < (size_t)1 << 31; }
static int other_seqs(const mlh_ctx* c) {
    const int wide = std::min(c->hp.maxSeqs, MLH_WIDE_MAX_SEQS);
    return mlh_wide_model(c) && places_fit(c, wide) ? wide : std::min(c->hp.maxSeqs, MLH_RANKS_MAX_SEQS);
}

// Whether the kernel covers a model of these hyper-parameters on this device.
static bool ranks_model(const mlh_ctx* c) {
    const mlh_hparams& hp = c->hp;
    const bool half = hp.weightDtype == MLH_DTYPE_BF16;
    const int ke = half ? 64 : 32, ca = half ? 4 : 3, tw = half ? 4 : 2, ns = RK_WORK / tw, cw = half ? 6 : 2, t13 = half ? 3 : 2;
    if (c->numCUs != RK_XCDS * RK_PER) return false;
    if (hp.headDim != 64 && (!half || hp.headDim != 128)) return false;
    if (hp.attnHeads < RK_XCDS || hp.attnHeads > 2 * RK_XCDS || hp.dim != hp.attnHeads * hp.headDim) return false;
    for (const LayerDev& L : c->layers)
        if (L.kind != MLH_KIND_ATTENTION && (hp.gdnHeads != hp.attnHeads || hp.gdnDk != hp.headDim || hp.gdnDv != hp.headDim)) return false;
    if (hp.dim % 128 || hp.dim % ke || hp.dim / ke > ca * RK_WORK || hp.dim / 16 > RK_PER * tw) return false;
    const int fs = hp.ffnDim / RK_XCDS, pleX = hp.pleDim / RK_XCDS;
    if (hp.ffnDim % (RK_XCDS * ke) || fs / ke > cw * ns || fs / 8 > RK_PER * t13) return false;
    if (hp.pleDim > 0) {
        if (hp.pleDim % (RK_XCDS * 4) || 16 % pleX || hp.pleDim % ke) return false;
        for (const LayerDev& L : c->layers)
            if (L.offPle % 16) return false;
    }
    return places_fit(c, other_seqs(c));
}

// Sequences whose states have a second place behind those of all maxSeqs (mlh_create allocates both).
int mlh_ranks_other_seqs(const mlh_ctx* c) { return ranks_model(c) ? other_seqs(c) : 0; }

// Whether the kernel covers this context's model as it has been finalized (memory for its exchange words apart).
static bool ranks_shape(const mlh_ctx* c) { return ranks_model(c) && mlh_rows_applicable(c, 1); }

// Whether kernels_wide.hip takes a call.  Here a pair of a head and a sequence has four workgroups of its XCD up to 64 pairs, fewer beyond; there it has one or a share
// of one whatever their number, and attention layers cost a little more, the others less.  Measured, us per step, here and there (12 layers, fp32, 100 keys; in
// brackets 350 keys):
//   hybrid (3 in 4 gated delta net)  8 heads   6: 212, 209 (216, 216)   8: 216, 211 (221, 219)   9: 243, 211
//                                   10 heads   6: 232, 242 (238, 249)   7: 257, 242 (264, 250)   9: 272, 244
//                                   12 heads   5: 241, 253              6: 267, 255 (272, 263)   12: 321, 260   16: 328, 263
//   attention only                   8 heads   6: 224, 239 (249, 267)   8: 237, 240 (264, 269)   9: 266, 240   8, gated and normed (272, 272)
//                                   10 heads   6: 247, 261 (266, 285)   7: 275, 262 (299, 287)
//              gated and normed     12 heads   6: 302, 303 (322, 331)   7: 310, 304 (338, 333)   8: 307, 306 (333, 337)   9: 339, 306 (374, 340)
static bool wide_is_faster(const mlh_ctx* c, int nseq) {
    int gdn = 0;
    for (const LayerDev& L : c->layers) gdn += L.kind != MLH_KIND_ATTENTION;
    const bool hybrid = 2 * gdn >= (int)c->layers.size();
    return nseq >= (hybrid ? 6 : 7) && (nseq * c->hp.attnHeads > 64 || (hybrid && c->hp.attnHeads == RK_XCDS));
}
bool mlh_ranks_wide(const mlh_ctx* c, int nseq) { return c->wideMax >= nseq && (wide_is_faster(c, nseq) || nseq > std::max(c->ranksMax, 5)); }

bool mlh_ranks_applicable(const mlh_ctx* c, int nseq) { return (mlh_ranks_wide(c, nseq) || c->ranksMax >= nseq) && mlh_rows_applicable(c, nseq); }

template <typename WT, int HD>
static int ranks_launch(mlh_ctx* c, const RanksArgs* P, size_t lds) {
    const void* f = reinterpret_cast<const void*>(&k_decode_ranks<WT, HD>);
    if (!P) { // preparation
        MLH_CHECK(c, hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, RK_LDS));
        int perCu = 0;
        MLH_CHECK(c, hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, k_decode_ranks<WT, HD>, RK_THREADS, RK_LDS));
        return perCu < 1 ? 1 : 0;
    }
    hipLaunchKernelGGL((k_decode_ranks<WT, HD>), dim3(RK_XCDS * RK_PER), dim3(RK_THREADS), lds, c->stream, *P);
    MLH_CHECK(c, hipGetLastError());
    return 0;
}
static int ranks_launch(mlh_ctx* c, const RanksArgs* P, size_t lds) {
    const bool half = c->hp.weightDtype == MLH_DTYPE_BF16, wide = c->hp.headDim == 128;
    if (half) return wide ? ranks_launch<bf16_t, 128>(c, P, lds) : ranks_launch<bf16_t, 64>(c, P, lds);
    return ranks_launch<float, 64>(c, P, lds);
}

int mlh_ranks_reset(mlh_ctx* c) {
    c->ranksTag = 0;
    void* const bufs[] = {c->ranksBuf, c->wideBuf};
    const size_t bytes[] = {c->ranksBytes, c->wideBytes};
    for (int i = 0; i < 2; i++) {
        if (!bufs[i]) continue;
        hipLaunchKernelGGL(k_ranks_zero, dim3(1024), dim3(256), 0, c->stream, (u32x4*)bufs[i], bytes[i] / 16);
        MLH_CHECK(c, hipGetLastError());
    }
    return 0;
}

// At finalize: how many sequences the kernel takes (none where the model or the device does not suit it), and its exchange words.
int mlh_ranks_prepare(mlh_ctx* c) {
    c->ranksMax = c->wideMax = 0;
    if (!ranks_shape(c)) return 0;
    int rc = ranks_launch(c, nullptr, 0);
    if (rc) return rc < 0 ? rc : 0;
    int most = 0;
    size_t bytes = 0;
    RanksPlan p;
    for (int n = 1; n <= std::min(c->hp.maxSeqs, MLH_RANKS_MAX_SEQS) && ranks_plan(c, n, p); n++) { most = n; bytes = std::max(bytes, p.words); }
    if (bytes > c->ranksBytes) {
        void* q = nullptr;
        if (hipMalloc(&q, bytes) != hipSuccess) { // no room: the row kernels
            (void)hipGetLastError();
            return 0;
        }
        c->allocs.push_back(q);
        c->ranksBuf = q;
        c->ranksBytes = bytes;
    }
    c->ranksMax = most;
    if ((rc = mlh_wide_prepare(c))) return rc;
    return mlh_ranks_reset(c);
}

// `steps` decode steps of sequences 0 .. nseq - 1 in one launch.
int mlh_launch_ranks(mlh_ctx* c, int nseq, int steps) {
    const mlh_hparams& hp = c->hp;
    const bool wide = mlh_ranks_wide(c, nseq);
    RanksPlan p;
    if (!wide && (!ranks_plan(c, nseq, p) || p.words > c->ranksBytes)) { c->err = "decode of several sequences: no plan"; return -1; }
    // tags are a running count of layer passes; before it could wrap and meet a stale word, everything goes back to zero
    const unsigned long long need = (unsigned long long)steps * (hp.transformers + 1) + 1;
    if (c->ranksTag + need >= 0xFFFFFFFFull)
        if (const int rc = mlh_ranks_reset(c)) return rc;
    const unsigned tagBase = (unsigned)c->ranksTag;
    c->ranksTag += need;
    const int otherAt = (int)(hp.maxSeqs * state_floats(c));
    const unsigned startCount = c->injectAbort > 0 ? (unsigned)RK_PER : 0u; // test hook: no workgroup finds a place
    if (c->injectAbort > 0) c->injectAbort--;
    hipLaunchKernelGGL(k_ranks_prep, dim3(1), dim3(64), 0, c->stream, c->d_sync + 64 * 20, c->d_sync + 64 * 23, startCount);
    MLH_CHECK(c, hipGetLastError());
    if (wide) return mlh_launch_wide(c, nseq, steps, tagBase, otherAt);
    RanksArgs P;
    mlh_fill_args(c, P.a, nseq, c->d_tok);
    P.layers = c->d_layers;
    P.ER = (const unsigned char*)c->ER;
    P.xw = (unsigned char*)c->ranksBuf;
    P.xwBytes = (unsigned)c->ranksBytes;
    P.NL = hp.transformers;
    P.steps = steps;
    P.fs = hp.ffnDim / RK_XCDS; P.rowsQ = p.rowsQ; P.planeBytes = p.planeBytes;
    P.abortFlag = c->d_sync + 64 * 20;
    P.xcdCount = c->d_sync + 64 * 23;
    P.area = p.area; P.oPart = p.oPart; P.oMl = p.oMl; P.oMix = p.oMix; P.oX = p.oX; P.oH = p.oH; P.oU = p.oU; P.oXP = p.oXP; P.oHP = p.oHP;
    P.oAmax = p.oAmax; P.oTok = p.oTok;
    P.tagBase = tagBase;
    P.otherAt = otherAt;
    P.sides = (unsigned)c->ranksSides;
    P.abortAtStep = c->injectAbortStep;
    c->injectAbortStep = 0;
    return ranks_launch(c, &P, p.lds);
}

// A launch of nseq sequences has ended well: their states are in the place they were not in.
void mlh_ranks_done(mlh_ctx* c, int nseq) {
    if (state_floats(c)) c->ranksSides ^= ~0ull >> (64 - nseq); // (64 at most)
}

// It has given up (and its stream has drained): positions are what they were, and no word of it is met again.
int mlh_ranks_failed(mlh_ctx* c, int nseq) {
    memcpy(c->pinIo.p, c->h_len.data(), (size_t)nseq * 4);
    hipLaunchKernelGGL(k_ranks_positions, dim3(1), dim3(64), 0, c->stream, (const int*)c->pinIo.p, c->d_pos, nseq);
    MLH_CHECK(c, hipGetLastError());
    return mlh_ranks_reset(c);
}

// Before any other kernel works on n sequences (seqs: which; null: the first n): their states are in the first place.
int mlh_ranks_settle(mlh_ctx* c, const int* seqs, int n) {
    if (!c->ranksSides) return 0;
    unsigned long long which = 0;
    for (int i = 0; i < n; i++)
        if (const int s = seqs ? seqs[i] : i; s < MLH_WIDE_MAX_SEQS) which |= c->ranksSides & 1ull << s;
    if (!which) return 0;
    const size_t per4 = state_floats(c) / 4;
    hipLaunchKernelGGL(k_ranks_settle, dim3((unsigned)std::min<size_t>(16, (per4 + 255) / 256), c->hp.transformers, MLH_WIDE_MAX_SEQS), dim3(256), 0, c->stream,
                       (const LayerDev*)c->d_layers, c->hp.maxSeqs * per4, which, per4);
    MLH_CHECK(c, hipGetLastError());
    c->ranksSides &= ~which;
    return 0;
}
