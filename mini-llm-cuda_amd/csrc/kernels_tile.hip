// Tiled MFMA GEMM for the prefill's products: those of fp32 models (prompts of more than 64 tokens in a call; fewer run through
// kernels_rows.hip), and those of bf16 models that are too small for the 256 x 256 tiles of kernels_gemm.hip:
//
//     C[M, N] = A[M, K] . B[N, K]^T  (+ R[M, N])        A, B: IEEE half, fp32 as scaled halves (h2.h), fp32 as bf16 planes (p3.h), or bf16
//
// (bf16 operands: the GEMM self-test only; models with bf16 weights multiply halves, those with fp32 weights pairs of them by triples, or planes where
// their weights spread further than halves reach.)
//
// KG groups of 2 x NW waves own one TM x TN tile, 128 x 128 or 64 x 64, every wave WM x WN blocks of 16 x 16.  K goes by in slices of RA and RB bytes per row of A
// and B: 64 two-byte elements (128 bytes), 32 elements of three planes or halves (192 bytes) or 32 of two (128).  Slices go global -> LDS directly into a ring
// of S stages, one barrier per stage: stage s + S - 1 is asked for when stage s is about to be multiplied.  A slice's loads
// take the wave about as long to issue as its MFMAs take, and nothing inside the wave hides that (loads spread between
// the MFMAs measured no better): what hides it is another wave on the SIMD, hence eight waves or several workgroups per unit.
// Two groups (KG 2) take turns at the slices, a slice each per stage, and add their sums through LDS: for launches that put one workgroup on a unit,
// where a tile's chain of slices is what takes the time.  The chain is half as long, and each half of the eight waves multiplies what it has read once;
// eight waves of 32 x 16 on one slice read half as much again.  Pairs by triples, 64 x 64 tiles, weights cold: four waves with six stages 0.37 us per slice,
// two groups of them with three 0.24 and about 6 per launch (90 x 2560 x 768, K split in three: 11.1 and 9.6 us).
// A launch with 64 x 64 tiles spends half its time outside the slices, so nothing there waits for anything else: all arguments are fetched at once, a workgroup's
// tile and slices come from one division, scales and missing partial tiles need no branch (64 x 64 x 768: 9.4 us before that, 8.8 with it).
// The planes of a slice are read into registers once and used for all their products, so the fp32 forms need
// half the LDS reads per MFMA of a plain two-byte product with the same tile.
#include <algorithm>
#include <atomic>

#include "h2.h"
#include "mlh_internal.h"
#include "p3.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct TileTraits;
template <> struct TileTraits<f16_t> {
    static constexpr int RA = 128, RB = 128, KE = 64, NFA = 2, NFB = 2, ESA = 2, ESB = 2; // of A and B: bytes per row and slice, elements, fragments per slice, bytes per element
    static constexpr int NP = 2, PA[2] = {0, 1}, PB[2] = {0, 1}; // products per slice: of which fragments
    static __device__ __forceinline__ int phys(int p, int r) { return p ^ ((r >> 1) & 7); }
    // fragment f of a slice: elements 32 f .. 32 f + 31, lane quarter kq takes eight of them
    static __device__ __forceinline__ int frag(int f, int kq, int r) { return ((4 * f + kq) ^ ((r >> 1) & 7)) * 16; }
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4& b, f32x4& c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
};
template <> struct TileTraits<bf16_t> {
    static constexpr int RA = 128, RB = 128, KE = 64, NFA = 2, NFB = 2, ESA = 2, ESB = 2;
    static constexpr int NP = 2, PA[2] = {0, 1}, PB[2] = {0, 1};
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4& b, f32x4& c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
};
template <> struct TileTraits<p3_t> {
    static constexpr int RA = P3_BYTES, RB = P3_BYTES, KE = P3_BLOCK, NFA = 3, NFB = 3, ESA = 6, ESB = 6; // fragments: the planes
    static constexpr int NP = 6, PA[6] = {0, 0, 1, 0, 1, 2}, PB[6] = {0, 1, 0, 2, 1, 0};
    // Rows are 192 bytes apart: four neighbouring rows cover the four quarters of the 256 bytes the LDS serves at a time, and
    // rows that share a quarter (row / 4 = g differs) must use different 16-byte slots of it.  A 16-byte read is served
    // sixteen lanes at a time, lanes 0-3, 12-15, 20-27 together, then 4-11, 16-19, 28-31, and so on: g = 0, 3 with kq and
    // g = 1, 2 with kq + 1 meet.  Slot kq ^ (-g & 3) keeps both sets apart (kq ^ g does not: counted, every read took twice as long).
    static __device__ __forceinline__ int phys(int p, int r) { return (p & ~3) | ((p & 3) ^ (-(r >> 2) & 3)); }
    static __device__ __forceinline__ int frag(int f, int kq, int r) { return f * P3_PLANE + ((kq ^ (-(r >> 2) & 3)) * 16); }
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4& b, f32x4& c) { TileTraits<bf16_t>::mma(a, b, c); }
};

template <> struct TileTraits<h2_t> { // rows of A lie as those of 64 halves (fragments hi, lo), rows of B as those of planes (hi, lo, tiny)
    static constexpr int RA = 128, RB = 192, KE = 32, NFA = 2, NFB = 3, ESA = 4, ESB = 6;
    static constexpr int NP = 4, PA[4] = {0, 1, 0, 0}, PB[4] = {2, 0, 1, 0};
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4& b, f32x4& c) { TileTraits<f16_t>::mma(a, b, c); }
};
// where a lane's 16 bytes of a row lie in a slice of R bytes, and what a lane of an operand reads: the rules of 128 and 192 bytes
template <int R> __device__ __forceinline__ int tile_phys(int p, int r) { return R == 128 ? TileTraits<f16_t>::phys(p, r) : TileTraits<p3_t>::phys(p, r); }
template <int R> __device__ __forceinline__ int tile_frag(int f, int kq, int r) { return R == 128 ? TileTraits<f16_t>::frag(f, kq, r) : TileTraits<p3_t>::frag(f, kq, r); }

// XCD-aware order, as in kernels_gemm.hip: ids congruent mod 8 share an L2 and take a contiguous eighth of the tiles, which
// walk panels of four N tiles
__device__ __forceinline__ bool tile_of(unsigned id, unsigned tilesM, unsigned tilesN, int& tm, int& tn) {
    const unsigned total = tilesM * tilesN, per = (total + 7) / 8;
    const unsigned t = (id & 7) * per + (id >> 3);
    if ((id >> 3) >= per || t >= total) return false;
    const unsigned panel = t / (4 * tilesM), pw = min(4u, tilesN - 4 * panel), r = t - panel * 4 * tilesM;
    tm = (int)(pw == 4 ? r >> 2 : pw == 3 ? r / 3 : r >> (pw - 1)); // r / pw without a division's chain in front of the first load
    tn = (int)(4 * panel + r - tm * pw);
    return true;
}

#define TL_AGENT 16 // cache policy of partial tiles: sc1, agent scope

// workgroups whose stages fit the LDS of a compute unit (the register allocation must leave room for as many)
template <typename T> constexpr int tile_wgs(int rowsA, int rowsB, int stages) { return std::min(3, 160 * 1024 / ((rowsA * TileTraits<T>::RA + rowsB * TileTraits<T>::RB) * stages)); }

// WM x WN blocks of 16 x 16 per wave.  lda / ldb in elements; EPI as in kernels_gemm.hip.  gridDim.y > 1: that many
// workgroups split K of a tile; each writes its partial tile to `partials`, the last to arrive adds them in slice order.
template <typename T, int WM, int WN, int NW, int S, int KG, int EPI>
__global__ void __launch_bounds__(128 * NW * KG, NW * KG / 2 * tile_wgs<T>(32 * WM, 16 * NW * WN, S * KG)) k_gemm_tile(const void* __restrict__ A, int lda, const void* __restrict__ B, int ldb, void* Cv, int ldc,
                                                         const float* R, int ldr, int M, int N, int K, int tilesM, int tilesN, float alpha, const int* __restrict__ eA, const int* __restrict__ eB, const int* __restrict__ eC,
                                                         int ks, int kn, int kr, unsigned* counters, unsigned long long* partials) {
    typedef TileTraits<T> TT;
    constexpr int RA = TT::RA, RB = TT::RB, TM = 32 * WM, TN = 16 * NW * WN, THREADS = 128 * NW * KG;
    constexpr int SLICE = TM * RA + TN * RB, STAGE = KG * SLICE;
    constexpr int NWV = 2 * NW, CA = TM * RA / 1024, NL = SLICE / (1024 * NWV); // waves of a group; 1 KB pieces of A; load instructions per wave and slice
    static_assert(WM % KG == 0 && SLICE % (1024 * NWV) == 0, "a slice is a whole number of rounds of loads");
    extern __shared__ __attribute__((aligned(16))) unsigned char tls[];
    // (every argument in front of the first load in one go: fetched where each is first used they are waits one behind the other)
    asm volatile("" ::"s"(A), "s"(B), "s"(lda), "s"(ldb), "s"(M), "s"(N), "s"(K), "s"(tilesM), "s"(tilesN), "s"(eA), "s"(eB), "s"(kn), "s"(kr));
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = wave / NWV, wg = wave % NWV; // group, wave of it
    const int wm = wg / NW, wn = wg % NW, r16 = lane & 15, kq = lane >> 4;
    int tm, tn;
    if (!tile_of(blockIdx.x, tilesM, tilesN, tm, tn)) return;
    const int m0 = tm * TM, n0 = tn * TN;
    const int by = blockIdx.y, sbeg = by * kn + min(by, kr), send = sbeg + kn + (by < kr); // slices: kn for each of ks workgroups, the first kr one more
    const size_t ldaB = (size_t)lda * TT::ESA, ldbB = (size_t)ldb * TT::ESB;

    // load side: 1 KB per instruction, piece q * NWV + wg of the group's slice (the rows of A, then those of B); the lane fetches what
    // belongs into its slot (rows past the end: the last one)
    unsigned off[NL];
    bool fromB[NL];
#pragma unroll
    for (int q = 0; q < NL; q++) {
        const int c = q * NWV + wg;
        fromB[q] = c >= CA;
        const int o = (c - (fromB[q] ? CA : 0)) * 1024 + lane * 16, r = fromB[q] ? o / RB : o / RA, p = (fromB[q] ? o % RB : o % RA) >> 4;
        off[q] = (unsigned)((size_t)(fromB[q] ? min(r, N - 1 - n0) : min(r, M - 1 - m0)) * (fromB[q] ? ldbB : ldaB)) + (unsigned)(fromB[q] ? tile_phys<RB>(p, r) : tile_phys<RA>(p, r)) * 16;
    }
    auto uniform64 = [](unsigned long long v) {
        const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
        return ((unsigned long long)hi << 32) | lo;
    };
    unsigned long long baseA = uniform64((unsigned long long)A + (size_t)m0 * ldaB + (size_t)(sbeg + g) * RA);
    unsigned long long baseB = uniform64((unsigned long long)B + (size_t)n0 * ldbB + (size_t)(sbeg + g) * RB);
    const unsigned lds0 = (unsigned)(unsigned long long)tls;
    auto dma16 = [](unsigned long long sbase, unsigned laneOff, unsigned ldsAddr) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(ldsAddr), "v"(laneOff), "s"(sbase) : "memory", "m0");
    };
    const unsigned ldsW = __builtin_amdgcn_readfirstlane(lds0 + g * SLICE + wg * 1024);
    auto issue = [&](unsigned stageOff) { // the group's next slice into a stage
#pragma unroll
        for (int q = 0; q < NL; q++) dma16(fromB[q] ? baseB : baseA, off[q], ldsW + stageOff + q * NWV * 1024);
        baseA += KG * RA; baseB += KG * RB;
    };

    typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
    unsigned rdA[TT::NFA], rdB[TT::NFB];
#pragma unroll
    for (int f = 0; f < TT::NFA; f++) rdA[f] = lds0 + g * SLICE + (wm * 16 * WM + r16) * RA + tile_frag<RA>(f, kq, r16);
#pragma unroll
    for (int f = 0; f < TT::NFB; f++) rdB[f] = lds0 + g * SLICE + TM * RA + (wn * 16 * WN + r16) * RB + tile_frag<RB>(f, kq, r16);
    f32x4 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int j = 0; j < WN; j++) acc[i][j] = (f32x4)(0.f);

    // which blocks of its tile a wave has at the end: every group WO of the WM rows
    constexpr int WO = WM / KG;
    const int wr = (wm * WM + g * WO) * 16; // ... of rows m0 + wr ..
    constexpr bool PAIRS = __is_same(T, h2_t);
    int ea[PAIRS ? WO : 1] = {}, eb[PAIRS ? WN : 1][4] = {}; // the rows' scales, asked for in front of the slices
    if constexpr (PAIRS) { // (past the end, and rows without scales: zero)
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(eA), 0, eA ? M * 4 : 0, 0x00027000), rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(eB), 0, N * 4, 0x00027000);
#pragma unroll
        for (int bm = 0; bm < WO; bm++) ea[bm] = __builtin_amdgcn_raw_buffer_load_b32(ra, (unsigned)(m0 + wr + r16) * 4u + bm * 64, 0, 0);
#pragma unroll
        for (int bn = 0; bn < WN; bn++)
#pragma unroll
            for (int e = 0; e < 4; e++) eb[bn][e] = __builtin_amdgcn_raw_buffer_load_b32(rb, (unsigned)(n0 + wn * WN * 16 + 4 * kq) * 4u + bn * 64 + e * 4, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
    const int steps = (send - sbeg + KG - 1) / KG, mine = (send - sbeg - g + KG - 1) / KG; // slices of a group: sbeg + g + KG i
    unsigned cur = 0, nxt = (S - 1) * STAGE; // stage of step s, stage of step s + S - 1
#pragma unroll
    for (int q = 0; q < S - 1; q++)
        if (q < mine) issue(q * STAGE);
    for (int s = 0; s < steps; s++) {
        if (S > 2 && s + S - 2 < mine) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * NL) : "memory"); // slice s has landed, the ones after it may be on their way
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier(); // ... for every wave, and every wave has read slice s - 1
        __builtin_amdgcn_sched_barrier(0);
        if (KG > 1 && s >= mine) break; // (an odd one: the last step only)
        if (s + S - 1 < mine) issue(nxt);
        u32x4 fa[TT::NFA][WM], fb[TT::NFB][WN];
#pragma unroll
        for (int f = 0; f < TT::NFB; f++) {
#pragma unroll
            for (int b = 0; b < WN; b++) fb[f][b] = *(const lds_u32x4*)(rdB[f] + cur + b * 16 * RB);
            if (f < TT::NFA)
#pragma unroll
                for (int b = 0; b < WM; b++) fa[f][b] = *(const lds_u32x4*)(rdA[f] + cur + b * 16 * RA);
        }
        // (transposed product, weights as the first operand: a lane ends up with four neighbouring columns of one row)
#pragma unroll
        for (int pr = 0; pr < TT::NP; pr++)
#pragma unroll
            for (int bn = 0; bn < WN; bn++)
#pragma unroll
                for (int bm = 0; bm < WM; bm++) TT::mma(fb[TT::PB[pr]][bn], fa[TT::PA[pr]][bm], acc[bm][bn]);
        __builtin_amdgcn_sched_barrier(0);
        cur = cur == (S - 1) * STAGE ? 0 : cur + STAGE;
        nxt = nxt == (S - 1) * STAGE ? 0 : nxt + STAGE;
    }

    if constexpr (KG > 1) { // the groups' sums meet in LDS; each group goes on with its share of the rows, acc[0 .. WO - 1]
        static_assert(KG == 2, "two groups");
        __syncthreads(); // everyone is done with the stages
        u32x4* swap = reinterpret_cast<u32x4*>(tls) + wg * 64 + lane;
#pragma unroll
        for (int i = 0; i < WO; i++)
#pragma unroll
            for (int j = 0; j < WN; j++) swap[(g * WO * WN + i * WN + j) * (128 * NW)] = __builtin_bit_cast(u32x4, g == 0 ? acc[WO + i][j] : acc[i][j]);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < WO; i++)
#pragma unroll
            for (int j = 0; j < WN; j++) {
                const f32x4 other = __builtin_bit_cast(f32x4, swap[((1 - g) * WO * WN + i * WN + j) * (128 * NW)]);
                acc[i][j] = g == 0 ? acc[i][j] + other : other + acc[WO + i][j];
            }
    }

    if (ks > 1) {
        // Partial tiles go past the L2s (agent scope), 16 bytes at a time.  (Offsets in the lanes' register alone: with a scalar one beside it
        // the compiler lets the next instruction overwrite a store's data, and lanes 12 to 15 of sixteen have then stored what that wrote.)
        constexpr unsigned TB = TM * TN * 4;
        const __amdgpu_buffer_rsrc_t ws = __builtin_amdgcn_make_buffer_rsrc(partials, 0, MLH_GEMM_WS_PARTIALS * 4, 0x00027000);
        const unsigned at = (unsigned)(blockIdx.x * ks + blockIdx.y) * TB;
#pragma unroll
        for (int i = 0; i < WO; i++)
#pragma unroll
            for (int j = 0; j < WN; j++)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), ws, at + (unsigned)(tid + (i * WN + j) * THREADS) * 16u, 0, TL_AGENT);
        stores_landed();  // the partial tile is where the last to arrive will read it ...
        __syncthreads();  // ... for every wave of the workgroup
        if (tid == 0) {
            const unsigned prev = __hip_atomic_fetch_add(counters + blockIdx.x, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool last = prev == (unsigned)(ks - 1);
            *reinterpret_cast<int*>(tls) = last; // (the stages are done with; an int of its own would cost triples their second workgroup a unit)
            if (last) __hip_atomic_store(counters + blockIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!*reinterpret_cast<const int*>(tls)) return;
        // those behind the last of them lie outside the buffer and come as zeros: no branch around a load
        constexpr int CH = WO * WN > 4 ? 2 : 8; // partial tiles whose loads are in flight together; added in slice order
        const __amdgpu_buffer_rsrc_t parts = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)partials + (size_t)(blockIdx.x * ks) * TB, 0, ks * TB, 0x00027000);
#pragma unroll
        for (int i = 0; i < WO * WN; i++) acc[i / WN][i % WN] = (f32x4)(0.f);
#pragma unroll 1
        for (int q0 = 0; q0 < ks; q0 += CH) {
            u32x4 u[CH][WO * WN];
#pragma unroll
            for (int q = 0; q < CH; q++)
#pragma unroll
                for (int w = 0; w < WO * WN; w++) u[q][w] = __builtin_amdgcn_raw_buffer_load_b128(parts, (unsigned)(q0 + q) * TB + (unsigned)(tid + w * THREADS) * 16u, 0, TL_AGENT);
#pragma unroll
            for (int q = 0; q < CH; q++)
#pragma unroll
                for (int w = 0; w < WO * WN; w++) acc[w / WN][w % WN] += __builtin_bit_cast(f32x4, u[q][w]);
        }
    }

    // lane (r16, kq) holds, per 16 x 16 block, row r16 of C and the columns 4 kq .. 4 kq + 3
    if constexpr (PAIRS) { // back from the rows' scales
#pragma unroll
        for (int bn = 0; bn < WN; bn++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int bm = 0; bm < WO; bm++) acc[bm][bn][e] = ldexpf(acc[bm][bn][e], ea[bm] + eb[bn][e]);
    }
    if (EPI == 0) {
        const bool vec = ((ldc & 3) == 0) && (!R || (ldr & 3) == 0) && (((unsigned long long)Cv & 15) == 0) && (((unsigned long long)R & 15) == 0);
#pragma unroll
        for (int bm = 0; bm < WO; bm++) {
            const int row = m0 + wr + bm * 16 + r16;
            if (row >= M) continue;
#pragma unroll
            for (int bn = 0; bn < WN; bn++) {
                const int col = n0 + (wn * WN + bn) * 16 + 4 * kq;
                f32x4 v = acc[bm][bn] * alpha;
                float* cp = (float*)Cv + (size_t)row * ldc + col;
                const float* rp = R ? R + (size_t)row * ldr + col : nullptr;
                if (vec && col + 3 < N) {
                    if (R) v += *reinterpret_cast<const f32x4*>(rp);
                    *reinterpret_cast<f32x4*>(cp) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (col + e < N) cp[e] = v[e] + (rp ? rp[e] : 0.f);
                }
            }
        }
    } else { // SwiGLU: columns 2 j, 2 j + 1 are gate and up of unit j; the units leave in the operand type, through LDS so that stores are whole pieces
        constexpr int UB = sizeof(T) == 6 ? (TN / 64) * P3_BYTES : PAIRS ? (TN / 64) * 128 : TN; // bytes of a row of units (TN / 2 of them)
        constexpr int UP = UB + 16;                                    // its pitch in LDS
        __syncthreads();                                               // everyone is done with the stages
#pragma unroll
        for (int bm = 0; bm < WO; bm++)
#pragma unroll
            for (int bn = 0; bn < WN; bn++) {
                const f32x4 v = acc[bm][bn] * alpha;
                unsigned char* row = tls + (wr + bm * 16 + r16) * UP;
                const int j = (wn * WN + bn) * 8 + 2 * kq;
                if (sizeof(T) == 6) {
                    uint32_t w[3];
                    p3_split2((v.x / (1.0f + expf(-v.x))) * v.y, (v.z / (1.0f + expf(-v.z))) * v.w, w);
#pragma unroll
                    for (int p = 0; p < 3; p++) *reinterpret_cast<uint32_t*>(row + p3_offset(j) + p * P3_PLANE) = w[p];
                } else if (PAIRS) {
                    const int u = (n0 >> 1) + j, last = (N >> 1) - 1; // units u, u + 1 at their columns' scale
                    const float x = ldexpf((v.x / (1.0f + expf(-v.x))) * v.y, -eC[min(u, last)]), y = ldexpf((v.z / (1.0f + expf(-v.z))) * v.w, -eC[min(u + 1, last)]);
                    const h2_f16x2 hi = {(_Float16)x, (_Float16)y}, lo = {(_Float16)(x - (float)hi[0]), (_Float16)(y - (float)hi[1])};
                    unsigned char* to = row + (j >> 5) * 128 + (j & 31) * 2;
                    *reinterpret_cast<uint32_t*>(to) = __builtin_bit_cast(uint32_t, hi);
                    *reinterpret_cast<uint32_t*>(to + 64) = __builtin_bit_cast(uint32_t, lo);
                } else { // exp2 and reciprocal of the hardware (1 ulp each): far inside the rounding of a two-byte result
                    float o[2] = {v.x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * v.x)) * v.y, // (the factor that can be 0 before the one that could overflow)
                                  v.z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * v.z)) * v.w};
                    uint32_t w;
                    if (__is_same(T, f16_t)) w = pack_half_range(o[0], o[1]);
                    else w = __builtin_bit_cast(uint16_t, (__bf16)o[0]) | (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)o[1]) << 16;
                    *reinterpret_cast<uint32_t*>(row + j * 2) = w;
                }
            }
        __syncthreads();
        const int NU = N >> 1, j0 = n0 >> 1;
        const size_t ldcB = (size_t)ldc * TT::ESA;
        const bool vec = sizeof(T) != 2 || ((ldcB & 15) == 0 && ((unsigned long long)Cv & 15) == 0);
        for (int i = tid; i < TM * (UB / 16); i += THREADS) {
            const int r = i / (UB / 16), p = i % (UB / 16), row = m0 + r;
            if (row >= M) continue;
            const unsigned char* src = tls + r * UP + p * 16;
            if (sizeof(T) == 6) { // (rows of units are padded to whole blocks)
                if (j0 + (p / 12) * P3_BLOCK < NU) *reinterpret_cast<u32x4*>((unsigned char*)Cv + row * ldcB + (size_t)(j0 / P3_BLOCK) * P3_BYTES + p * 16) = *reinterpret_cast<const u32x4*>(src);
            } else if (PAIRS) {
                if (j0 + (p / 8) * 32 < NU) *reinterpret_cast<u32x4*>((unsigned char*)Cv + row * ldcB + (size_t)(j0 / 32) * 128 + p * 16) = *reinterpret_cast<const u32x4*>(src);
            } else {
                const int j = j0 + p * 8;
                uint16_t* up = (uint16_t*)Cv + (size_t)row * ldc + j;
                if (vec && j + 7 < NU) *reinterpret_cast<u32x4*>(up) = *reinterpret_cast<const u32x4*>(src);
                else
                    for (int e = 0; e < 8; e++)
                        if (j + e < NU) up[e] = reinterpret_cast<const uint16_t*>(src)[e];
            }
        }
    }
}

template <typename T, int WM, int WN, int NW, int S, int KG = 1>
static hipError_t launch_tile(hipStream_t stream, int epi, const void* A, int lda, const void* B, int ldb, void* C, int ldc,
                              const float* R, int ldr, int M, int N, int K, void* ws, float alpha, const int* eA, const int* eB, const int* eC, int ks) {
    constexpr int TM = 32 * WM, TN = 16 * NW * WN;
    const int tilesM = (M + TM - 1) / TM, tilesN = (N + TN - 1) / TN;
    const size_t lds = std::max((size_t)S * KG * (TM * TileTraits<T>::RA + TN * TileTraits<T>::RB), (size_t)TM * (3 * TN + 16));
    static std::atomic<bool> attr{false}; // set-up is idempotent: two threads that race here both do it
    if (!attr) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_tile<T, WM, WN, NW, S, KG, 0>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_tile<T, WM, WN, NW, S, KG, 1>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        attr = true;
    }
    const int slices = K / TileTraits<T>::KE;
    const dim3 grid((tilesM * tilesN + 7) / 8 * 8, ks);
    unsigned* counters = (unsigned*)ws;
    unsigned long long* partials = ws ? (unsigned long long*)((unsigned char*)ws + MLH_GEMM_WS_COUNTERS * 4) : nullptr;
    if (epi) hipLaunchKernelGGL((k_gemm_tile<T, WM, WN, NW, S, KG, 1>), grid, dim3(128 * NW * KG), lds, stream, A, lda, B, ldb, C, ldc, R, ldr, M, N, K, tilesM, tilesN, alpha, eA, eB, eC, ks, slices / ks, slices % ks, counters, partials);
    else hipLaunchKernelGGL((k_gemm_tile<T, WM, WN, NW, S, KG, 0>), grid, dim3(128 * NW * KG), lds, stream, A, lda, B, ldb, C, ldc, R, ldr, M, N, K, tilesM, tilesN, alpha, eA, eB, eC, ks, slices / ks, slices % ks, counters, partials);
    return hipGetLastError();
}

// What a launch takes, in microseconds: `slots` workgroups share a compute unit at a time; a round of the chip with k of
// them on a unit takes slices * us[k - 1] + 3; the way of partial tiles through memory and their sum, K split ks times, split + part * ks.  us: measured per K slice with one, two and three workgroups on every
// unit (the loads, barriers and LDS reads of a workgroup hide behind the others' MFMAs).
struct TileCost { int tm, tn, slots; double us[3], split, part; };
// Variants of the two-byte types: 64 x 64; 128 x 128 with two stages, two workgroups a unit; halves only (what the models multiply): 128 x 128
// with four stages, for launches that put one on a unit: nothing but its own stages then covers the way of a slice from memory.  777 x 2048 x 5888, K split in two, weights cold
// (a prefill reads each once): 36.8 us against 48.3 with two stages; on 512 workgroups (3270 rows) 114 against 110; and 64 x 64 by two groups of four
// waves with four stages of two slices, for launches that put one on a unit.  Prefills of 24 layers, weights cold (us): 100 x 6336 x 2048 12.6 (four waves, three stages:
// 14.9), 300 x 2048 x 2048 12.2 (15.2); whole prefills of 70, 150, 300, 500 tokens 2124 (2318), 2546 (2718), 3122 (3218), 3483 (3647).
static const TileCost kCostHalf[4] = {{64, 64, 3, {0.26, 0.38, 0.58}, 4.0, 0.5}, {128, 128, 2, {0.64, 1.04, 0.0}, 4.0, 0.5}, {128, 128, 1, {0.58, 0.0, 0.0}, 4.0, 0.5}, {64, 64, 1, {0.22, 0.0, 0.0}, 1.6, 0.1}};
// Pairs by triples: 64 x 64 by four waves, three stages (60 KB: two workgroups a unit); 128 x 128 by eight, two
// stages (80 KB, two a unit to the byte; three stages, one a unit: 0.98); 64 x 64 by two groups of four, three stages of two slices, for launches that put one on a
// unit.  What bounds a slice of 128 x 128: its 40 KB on the way into LDS and the reads behind them
// take 0.55, its matrix instructions 0.43 at the full clock, and they overlap in part.  Against planes (us): 19470 x 4096 x 768 490 and 757,
// 17400 x 768 x 2048 219 and 366, 1200 x 2560 x 768 30 and 34; in prefills of 12 layers, weights cold, 90 rows: 2560 x 768 9.9 and 10.3,
// SwiGLU 4096 x 768 12.5 and 14.5, 768 x 2048 10.9 and 11.8; 130 x 3072 x 768 11.0 and 12.8 (K split in three on 64 x 64 tiles of four waves, two a unit, 12.5:
// their partial tiles are what the third figures' split stands for).  Dealing the waves into two halves that take turns at reading and
// multiplying was no faster (tried on planes: 754 to 826 for 776), nor slices contiguous in memory (483 for 495).
static const TileCost kCostH2[3] = {{64, 64, 2, {0.395, 0.55, 0.0}, 3.0, 0.4}, {128, 128, 2, {0.93, 1.84, 0.0}, 1.6, 0.4}, {64, 64, 1, {0.30, 0.0, 0.0}, 1.6, 0.1}};
static const TileCost kCostP3[2] = {{64, 64, 2, {0.39, 0.75, 0.0}, 4.0, 0.5}, {128, 128, 1, {1.28, 0.0, 0.0}, 4.0, 0.5}};

static double tile_us(const TileCost& c, int M, int N, int slices, int cus, int ks) {
    const long tiles = (long)((M + c.tm - 1) / c.tm) * ((N + c.tn - 1) / c.tn) * ks;
    const long full = tiles / ((long)cus * c.slots), rest = tiles - full * cus * c.slots;
    const double n = (double)((slices + ks - 1) / ks);
    double us = full * (n * c.us[c.slots - 1] + 3.0);
    if (rest) us += n * c.us[(rest + cus - 1) / cus - 1] + 3.0;
    return us + (ks > 1 ? c.split + c.part * ks : 0.0); // (the partial tiles' way through memory and their sum)
}

// The split of K that is fastest: the workspace holds 4 M partial sums and 1024 tile counters, and a workgroup keeps eight slices or more.
static double best_split(const TileCost& c, int M, int N, int slices, int cus, bool ws, int& ks) {
    const long tiles = (long)((M + c.tm - 1) / c.tm) * ((N + c.tn - 1) / c.tn);
    double best = tile_us(c, M, N, slices, cus, 1);
    ks = 1;
    for (int k = 2; ws && k <= 8 && slices / k >= 8 && tiles <= MLH_GEMM_WS_COUNTERS - 8 && (tiles + 7) * k * c.tm * c.tn <= MLH_GEMM_WS_PARTIALS; k++) {
        const double us = tile_us(c, M, N, slices, cus, k);
        if (us < best) { best = us; ks = k; }
    }
    return best;
}

// The fastest variant of a type, and what it is expected to take.
struct TileChoice { int variant, ks; };
static double tile_choice(int dtype, int M, int N, int K, int cus, bool ws, TileChoice& c) {
    const TileCost* cost = dtype == MLH_GEMM_P3 ? kCostP3 : dtype == MLH_GEMM_H2 ? kCostH2 : kCostHalf;
    const int slices = K / (dtype == MLH_GEMM_P3 || dtype == MLH_GEMM_H2 ? 32 : 64);
    double best = 0.0;
    for (int v = 0; v < (dtype == MLH_GEMM_F16 ? 4 : dtype == MLH_GEMM_H2 ? 3 : 2); v++) {
        int ks;
        const double us = best_split(cost[v], M, N, slices, cus, ws, ks);
        if (v == 0 || us < best) { best = us; c.variant = v; c.ks = ks; }
    }
    return best;
}
double mlh_gemm_tile_us(int dtype, int M, int N, int K, int cus, bool ws) {
    TileChoice c;
    return tile_choice(dtype, M, N, K, cus, ws, c);
}

hipError_t mlh_gemm_tile(hipStream_t stream, int dtype, int epi, const void* A, int lda, const void* B, int ldb, void* C, int ldc,
                         const float* R, int ldr, int M, int N, int K, void* ws, float alpha, const int* eA, const int* eB, const int* eC) {
    const int cus = mlh_gemm_num_cus();
    if (!cus) return hipErrorInvalidDevice;
    TileChoice c;
    tile_choice(dtype, M, N, K, cus, ws != nullptr, c);
#define TILE(T_, WM_, WN_, NW_, ...) launch_tile<T_, WM_, WN_, NW_, __VA_ARGS__>(stream, epi, A, lda, B, ldb, C, ldc, R, ldr, M, N, K, ws, alpha, eA, eB, eC, c.ks)
    // Measured (517 x 768 x 3072, 517 x 6144 x 768, 17000 x 768 x 2048; us): planes 27, 35, 335 -- fp32 MFMA tiles of 256 x 256 took
    // 701, 187, 512 --, halves 13, 13, 69.  Planes: 64 x 64 by eight waves of 32 x 16, three stages (two workgroups a unit), or
    // 128 x 128 by eight waves of 64 x 32, two stages.  Two-byte operands: 64 x 64 by four waves of 32 x 32, three stages, or
    // 128 x 128 by eight waves, two stages (two workgroups a unit) or, halves, four (one).
    if (dtype == MLH_GEMM_P3) return c.variant == 0 ? TILE(p3_t, 2, 1, 4, 3) : TILE(p3_t, 4, 2, 4, 2);
    if (dtype == MLH_GEMM_H2) return c.variant == 0 ? TILE(h2_t, 2, 2, 2, 3) : c.variant == 1 ? TILE(h2_t, 4, 2, 4, 2) : TILE(h2_t, 2, 2, 2, 3, 2);
    if (dtype == MLH_GEMM_F16) return c.variant == 0 ? TILE(f16_t, 2, 2, 2, 3) : c.variant == 1 ? TILE(f16_t, 4, 2, 4, 2) : c.variant == 2 ? TILE(f16_t, 4, 2, 4, 4) : TILE(f16_t, 2, 2, 2, 4, 2);
    return c.variant == 0 ? TILE(bf16_t, 2, 2, 2, 3) : TILE(bf16_t, 4, 2, 4, 2);
#undef TILE
}

// fp32 rows -> plane rows (weights at finalize; the self-test's operands, which alone may lie beyond P3_BEYOND).  ldd >= cols, columns past `cols` become zero.
__global__ void __launch_bounds__(256) k_split_p3(const float* __restrict__ src, int lds_, void* dst, int ldd, int rows, int cols) {
    const size_t n4 = (size_t)rows * (ldd / 4);
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
        const int r = (int)(i / (ldd / 4)), c = (int)(i % (ldd / 4)) * 4;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = c + e < cols ? src[(size_t)r * lds_ + c + e] : 0.f;
        unsigned char* row = (unsigned char*)dst + (size_t)r * ldd * 6;
        p3_put4(row, c, v[0], v[1], v[2], v[3]);
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (p3_beyond(v[e])) {
                uint32_t h[3];
                p3_split_beyond(v[e], h);
#pragma unroll
                for (int k = 0; k < 3; k++) *reinterpret_cast<uint16_t*>(row + p3_offset(c + e) + k * P3_PLANE) = (uint16_t)h[k];
            }
    }
}
hipError_t mlh_split_p3(hipStream_t stream, const float* src, int lds_, void* dst, int ldd, int rows, int cols) {
    hipLaunchKernelGGL(k_split_p3, dim3(2048), dim3(256), 0, stream, src, lds_, dst, ldd, rows, cols);
    return hipGetLastError();
}

// fp32 rows -> rows of triples (weights at finalize; colExps: exponents that the columns take over from the other operand's, or null) or pairs (the self-test's
// other operand), and their exponents.  A wave a row; cols, lds and ldd: multiples of 32.
template <bool TRIPLES>
__global__ void __launch_bounds__(256) k_split_h2(const float* __restrict__ src, int lds_, void* dst, int ldd, const int* __restrict__ colExps, int* exps, int rows, int cols) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float* x = src + (size_t)row * lds_;
    unsigned char* out = (unsigned char*)dst + (size_t)row * ldd * (TRIPLES ? 6 : 4);
    auto col = [&](int i) { return colExps ? colExps[i] : 0; };
    int most = -100000;
    for (int i = lane; i < cols; i += 64)
        if (x[i] != 0.f) most = max(most, h2_size(x[i]) + col(i));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, 64));
    const int e = h2_exponent(most);
    if (lane == 0) exps[row] = e;
    for (int i = lane * 4; i < cols; i += 256) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(x + i);
        h2_put4<TRIPLES>(out, i, ldexpf(v.x, col(i) - e), ldexpf(v.y, col(i + 1) - e), ldexpf(v.z, col(i + 2) - e), ldexpf(v.w, col(i + 3) - e));
    }
}
hipError_t mlh_split_h2(hipStream_t stream, bool triples, const float* src, int lds_, void* dst, int ldd, const int* colExps, int* exps, int rows, int cols) {
    const dim3 grid((rows + 3) / 4);
    if (triples) hipLaunchKernelGGL((k_split_h2<true>), grid, dim3(256), 0, stream, src, lds_, dst, ldd, colExps, exps, rows, cols);
    else hipLaunchKernelGGL((k_split_h2<false>), grid, dim3(256), 0, stream, src, lds_, dst, ldd, colExps, exps, rows, cols);
    return hipGetLastError();
}
