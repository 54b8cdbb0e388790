// Tiled MFMA GEMM for the prefill's products: those of fp32 models (prompts of more than 64 tokens in a call; fewer run through
// kernels_rows.hip), and those of bf16 models that are too small for the 256 x 256 tiles of kernels_gemm.hip:
//
//     C[M, N] = A[M, K] . B[N, K]^T  (+ R[M, N])        A, B: IEEE half, fp32 as three bf16 planes (p3.h), or bf16
//
// (bf16 operands: the GEMM self-test only; models with bf16 weights multiply halves.)
//
// A workgroup of 2 x NW waves owns one TM x TN tile, 128 x 128 or 64 x 64, every wave WM x WN blocks of 16 x 16.  K goes by in slices of RB bytes per row: 64
// two-byte elements (128 bytes) or 32 elements of three planes (192 bytes).  Slices go global -> LDS directly into a ring
// of S stages, one barrier per slice: slice s + S - 1 is asked for when slice s is about to be multiplied.  A slice's loads
// take the wave about as long to issue as its MFMAs take, and nothing inside the wave hides that (loads spread between
// the MFMAs measured no better): what hides it is another wave on the SIMD, hence eight waves or several workgroups per unit.
// The three planes of a slice are read into registers once and used for all six plane products, so the fp32 form needs
// half the LDS reads per MFMA of a plain two-byte product with the same tile.
#include <algorithm>
#include <atomic>

#include "mlh_internal.h"
#include "p3.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct TileTraits;
template <> struct TileTraits<f16_t> {
    static constexpr int RB = 128, KE = 64, NF = 2, ES = 2; // bytes and elements per row and slice, fragments per slice, bytes per element
    static __device__ __forceinline__ int phys(int p, int r) { return p ^ ((r >> 1) & 7); }
    // fragment f of a slice: elements 32 f .. 32 f + 31, lane quarter kq takes eight of them
    static __device__ __forceinline__ int frag(int f, int kq, int r) { return ((4 * f + kq) ^ ((r >> 1) & 7)) * 16; }
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4& b, f32x4& c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
};
template <> struct TileTraits<bf16_t> {
    static constexpr int RB = 128, KE = 64, NF = 2, ES = 2;
    static __device__ __forceinline__ int phys(int p, int r) { return p ^ ((r >> 1) & 7); }
    static __device__ __forceinline__ int frag(int f, int kq, int r) { return ((4 * f + kq) ^ ((r >> 1) & 7)) * 16; }
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4& b, f32x4& c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
};
template <> struct TileTraits<p3_t> {
    static constexpr int RB = P3_BYTES, KE = P3_BLOCK, NF = 3, ES = 6; // fragments: the planes
    // Rows are 192 bytes apart: four neighbouring rows cover the four quarters of the 256 bytes the LDS serves at a time, and
    // rows that share a quarter (row / 4 = g differs) must use different 16-byte slots of it.  A 16-byte read is served
    // sixteen lanes at a time, lanes 0-3, 12-15, 20-27 together, then 4-11, 16-19, 28-31, and so on: g = 0, 3 with kq and
    // g = 1, 2 with kq + 1 meet.  Slot kq ^ (-g & 3) keeps both sets apart (kq ^ g does not: counted, every read took twice as long).
    static __device__ __forceinline__ int phys(int p, int r) { return (p & ~3) | ((p & 3) ^ (-(r >> 2) & 3)); }
    static __device__ __forceinline__ int frag(int f, int kq, int r) { return f * P3_PLANE + ((kq ^ (-(r >> 2) & 3)) * 16); }
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4& b, f32x4& c) { TileTraits<bf16_t>::mma(a, b, c); }
};

// XCD-aware order, as in kernels_gemm.hip: ids congruent mod 8 share an L2 and take a contiguous eighth of the tiles, which
// walk panels of four N tiles
__device__ __forceinline__ bool tile_of(int id, int tilesM, int tilesN, int& tm, int& tn) {
    const int total = tilesM * tilesN, per = (total + 7) / 8;
    const int t = (id & 7) * per + (id >> 3);
    if ((id >> 3) >= per || t >= total) return false;
    const int panel = t / (4 * tilesM), pw = min(4, tilesN - 4 * panel), r = t - panel * 4 * tilesM;
    tm = r / pw;
    tn = 4 * panel + r % pw;
    return true;
}

__device__ __forceinline__ unsigned long long tl_ald(const unsigned long long* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void tl_ast(unsigned long long* p, unsigned long long v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// workgroups whose stages fit the LDS of a compute unit (the register allocation must leave room for as many)
template <typename T> constexpr int tile_wgs(int rows, int stages) { return std::min(3, 160 * 1024 / (rows * TileTraits<T>::RB * stages + 16)); }

// WM x WN blocks of 16 x 16 per wave.  lda / ldb in elements; EPI as in kernels_gemm.hip.  gridDim.y > 1: that many
// workgroups split K of a tile; each writes its partial tile to `partials`, the last to arrive adds them in slice order.
template <typename T, int WM, int WN, int NW, int S, int EPI>
__global__ void __launch_bounds__(128 * NW, NW / 2 * tile_wgs<T>(32 * WM + 16 * NW * WN, S)) k_gemm_tile(const void* __restrict__ A, int lda, const void* __restrict__ B, int ldb, void* Cv, int ldc,
                                                         const float* R, int ldr, int M, int N, int K, int tilesM, int tilesN, float alpha,
                                                         unsigned* counters, unsigned long long* partials) {
    typedef TileTraits<T> TT;
    constexpr int RB = TT::RB, NF = TT::NF, TM = 32 * WM, TN = 16 * NW * WN, THREADS = 128 * NW;
    constexpr int STAGE = (TM + TN) * RB;
    constexpr int NWV = 2 * NW, CA = TM * RB / 1024, NL = (TM + TN) * RB / (1024 * NWV); // waves; 1 KB pieces of A; load instructions per wave and slice
    static_assert((TM + TN) * RB % (1024 * NWV) == 0, "a slice is a whole number of rounds of loads");
    extern __shared__ __attribute__((aligned(16))) unsigned char tls[];
    __shared__ int lastFlag;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / NW, wn = wave % NW, r16 = lane & 15, kq = lane >> 4;
    int tm, tn;
    if (!tile_of(blockIdx.x, tilesM, tilesN, tm, tn)) return;
    const int m0 = tm * TM, n0 = tn * TN;
    const int nslices = K / TT::KE, ks = gridDim.y;
    const int sbeg = ks == 1 ? 0 : (int)((unsigned)nslices * blockIdx.y / (unsigned)ks);
    const int send = ks == 1 ? nslices : (int)((unsigned)nslices * (blockIdx.y + 1) / (unsigned)ks);
    const size_t ldaB = (size_t)lda * TT::ES, ldbB = (size_t)ldb * TT::ES;

    // load side: 1 KB per instruction, piece q * NWV + wave of the slice (the rows of A, then those of B); the lane fetches what
    // belongs into its slot (rows past the end: the last one)
    unsigned off[NL];
    bool fromB[NL];
#pragma unroll
    for (int q = 0; q < NL; q++) {
        const int c = q * NWV + wave;
        fromB[q] = c >= CA;
        const int o = (c - (fromB[q] ? CA : 0)) * 1024 + lane * 16, r = o / RB, p = (o % RB) >> 4;
        off[q] = (unsigned)((size_t)(fromB[q] ? min(r, N - 1 - n0) : min(r, M - 1 - m0)) * (fromB[q] ? ldbB : ldaB)) + (unsigned)TT::phys(p, r) * 16;
    }
    auto uniform64 = [](unsigned long long v) {
        const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
        return ((unsigned long long)hi << 32) | lo;
    };
    unsigned long long baseA = uniform64((unsigned long long)A + (size_t)m0 * ldaB + (size_t)sbeg * RB);
    unsigned long long baseB = uniform64((unsigned long long)B + (size_t)n0 * ldbB + (size_t)sbeg * RB);
    const unsigned lds0 = (unsigned)(unsigned long long)tls;
    auto dma16 = [](unsigned long long sbase, unsigned laneOff, unsigned ldsAddr) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(ldsAddr), "v"(laneOff), "s"(sbase) : "memory", "m0");
    };
    const unsigned ldsW = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024);
    auto issue = [&](unsigned stageOff) { // the next slice into a stage
#pragma unroll
        for (int q = 0; q < NL; q++) dma16(fromB[q] ? baseB : baseA, off[q], ldsW + stageOff + q * NWV * 1024);
        baseA += RB; baseB += RB;
    };

    typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
    unsigned rdA[NF], rdB[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        rdA[f] = lds0 + (wm * 16 * WM + r16) * RB + TT::frag(f, kq, r16);
        rdB[f] = lds0 + TM * RB + (wn * 16 * WN + r16) * RB + TT::frag(f, kq, r16);
    }
    f32x4 acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int j = 0; j < WN; j++) acc[i][j] = (f32x4)(0.f);

    unsigned cur = 0, nxt = (S - 1) * STAGE; // stage of slice s, stage of slice s + S - 1
#pragma unroll
    for (int q = 0; q < S - 1; q++)
        if (sbeg + q < send) issue(q * STAGE);
    for (int s = sbeg; s < send; s++) {
        if (S > 2 && s + S - 2 < send) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * NL) : "memory"); // slice s has landed, the ones after it may be on their way
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier(); // ... for every wave, and every wave has read slice s - 1
        __builtin_amdgcn_sched_barrier(0);
        if (s + S - 1 < send) issue(nxt);
        u32x4 fa[NF][WM], fb[NF][WN];
#pragma unroll
        for (int f = 0; f < NF; f++) {
#pragma unroll
            for (int b = 0; b < WN; b++) fb[f][b] = *(const lds_u32x4*)(rdB[f] + cur + b * 16 * RB);
#pragma unroll
            for (int b = 0; b < WM; b++) fa[f][b] = *(const lds_u32x4*)(rdA[f] + cur + b * 16 * RB);
        }
        // (transposed product, weights as the first operand: a lane ends up with four neighbouring columns of one row)
        constexpr int NP = NF == 3 ? 6 : NF;
        constexpr int PA[6] = {0, NF == 3 ? 0 : 1, 1, 0, 1, 2}, PB[6] = {0, 1, 0, 2, 1, 0}; // plane pairs, or the two halves of the slice
#pragma unroll
        for (int pr = 0; pr < NP; pr++)
#pragma unroll
            for (int bn = 0; bn < WN; bn++)
#pragma unroll
                for (int bm = 0; bm < WM; bm++) TT::mma(fb[PB[pr]][bn], fa[PA[pr]][bm], acc[bm][bn]);
        __builtin_amdgcn_sched_barrier(0);
        cur = cur == (S - 1) * STAGE ? 0 : cur + STAGE;
        nxt = nxt == (S - 1) * STAGE ? 0 : nxt + STAGE;
    }

    if (ks > 1) {
        constexpr int TW = TM * TN / 2; // 8-byte words of a partial tile
        unsigned long long* mine = partials + ((size_t)blockIdx.x * ks + blockIdx.y) * TW + tid;
#pragma unroll
        for (int i = 0; i < WM; i++)
#pragma unroll
            for (int j = 0; j < WN; j++) {
                tl_ast(mine + (size_t)(2 * (i * WN + j)) * THREADS, (unsigned long long)__float_as_uint(acc[i][j].x) | ((unsigned long long)__float_as_uint(acc[i][j].y) << 32));
                tl_ast(mine + (size_t)(2 * (i * WN + j) + 1) * THREADS, (unsigned long long)__float_as_uint(acc[i][j].z) | ((unsigned long long)__float_as_uint(acc[i][j].w) << 32));
            }
        stores_landed();  // the partial tile is where the last to arrive will read it ...
        __syncthreads();  // ... for every wave of the workgroup
        if (tid == 0) {
            const unsigned prev = __hip_atomic_fetch_add(counters + blockIdx.x, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            lastFlag = prev == (unsigned)(ks - 1);
            if (lastFlag) __hip_atomic_store(counters + blockIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!lastFlag) return;
        const unsigned long long* all = partials + (size_t)blockIdx.x * ks * TW + tid;
        constexpr int CH = 8 / (WM * WN) > 0 ? 8 / (WM * WN) : 1;
        for (int q0 = 0; q0 < ks; q0 += CH) { // CH partial tiles at a time, all their loads in flight; added in slice order
            unsigned long long u[CH][2 * WM * WN];
#pragma unroll
            for (int q = 0; q < CH; q++)
#pragma unroll
                for (int w = 0; w < 2 * WM * WN; w++) u[q][w] = tl_ald(all + (size_t)min(q0 + q, ks - 1) * TW + (size_t)w * THREADS);
#pragma unroll
            for (int q = 0; q < CH; q++) {
                if (q0 + q >= ks) break;
#pragma unroll
                for (int i = 0; i < WM; i++)
#pragma unroll
                    for (int j = 0; j < WN; j++) {
                        const unsigned long long lo = u[q][2 * (i * WN + j)], hi = u[q][2 * (i * WN + j) + 1];
                        f32x4 v;
                        v.x = __uint_as_float((unsigned)lo); v.y = __uint_as_float((unsigned)(lo >> 32));
                        v.z = __uint_as_float((unsigned)hi); v.w = __uint_as_float((unsigned)(hi >> 32));
                        acc[i][j] = q0 + q == 0 ? v : acc[i][j] + v;
                    }
            }
        }
    }

    // lane (r16, kq) holds, per 16 x 16 block, row r16 of C and the columns 4 kq .. 4 kq + 3
    if (EPI == 0) {
        const bool vec = ((ldc & 3) == 0) && (!R || (ldr & 3) == 0) && (((unsigned long long)Cv & 15) == 0) && (((unsigned long long)R & 15) == 0);
#pragma unroll
        for (int bm = 0; bm < WM; bm++) {
            const int row = m0 + (wm * WM + bm) * 16 + r16;
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
        constexpr int UB = sizeof(T) == 6 ? (TN / 64) * P3_BYTES : TN; // bytes of a row of units (TN / 2 of them)
        constexpr int UP = UB + 16;                                    // its pitch in LDS
        __syncthreads();                                               // everyone is done with the stages
#pragma unroll
        for (int bm = 0; bm < WM; bm++)
#pragma unroll
            for (int bn = 0; bn < WN; bn++) {
                const f32x4 v = acc[bm][bn] * alpha;
                unsigned char* row = tls + ((wm * WM + bm) * 16 + r16) * UP;
                const int j = (wn * WN + bn) * 8 + 2 * kq;
                if (sizeof(T) == 6) {
                    uint32_t w[3];
                    p3_split2((v.x / (1.0f + expf(-v.x))) * v.y, (v.z / (1.0f + expf(-v.z))) * v.w, w);
#pragma unroll
                    for (int p = 0; p < 3; p++) *reinterpret_cast<uint32_t*>(row + p3_offset(j) + p * P3_PLANE) = w[p];
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
        const size_t ldcB = (size_t)ldc * TT::ES;
        const bool vec = sizeof(T) == 6 || ((ldcB & 15) == 0 && ((unsigned long long)Cv & 15) == 0);
        for (int i = tid; i < TM * (UB / 16); i += THREADS) {
            const int r = i / (UB / 16), p = i % (UB / 16), row = m0 + r;
            if (row >= M) continue;
            const unsigned char* src = tls + r * UP + p * 16;
            if (sizeof(T) == 6) { // (rows of units are padded to whole blocks)
                if (j0 + (p / 12) * P3_BLOCK < NU) *reinterpret_cast<u32x4*>((unsigned char*)Cv + row * ldcB + (size_t)(j0 / P3_BLOCK) * P3_BYTES + p * 16) = *reinterpret_cast<const u32x4*>(src);
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

template <typename T, int WM, int WN, int NW, int S>
static hipError_t launch_tile(hipStream_t stream, int epi, const void* A, int lda, const void* B, int ldb, void* C, int ldc,
                              const float* R, int ldr, int M, int N, int K, void* ws, float alpha, int ks) {
    constexpr int TM = 32 * WM, TN = 16 * NW * WN;
    const int tilesM = (M + TM - 1) / TM, tilesN = (N + TN - 1) / TN;
    const size_t lds = std::max((size_t)S * (TM + TN) * TileTraits<T>::RB, (size_t)TM * (3 * TN + 16));
    static std::atomic<bool> attr{false}; // set-up is idempotent: two threads that race here both do it
    if (!attr) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_tile<T, WM, WN, NW, S, 0>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_gemm_tile<T, WM, WN, NW, S, 1>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        attr = true;
    }
    const dim3 grid((tilesM * tilesN + 7) / 8 * 8, ks);
    unsigned* counters = (unsigned*)ws;
    unsigned long long* partials = ws ? (unsigned long long*)((unsigned char*)ws + MLH_GEMM_WS_COUNTERS * 4) : nullptr;
    if (epi) hipLaunchKernelGGL((k_gemm_tile<T, WM, WN, NW, S, 1>), grid, dim3(128 * NW), lds, stream, A, lda, B, ldb, C, ldc, R, ldr, M, N, K, tilesM, tilesN, alpha, counters, partials);
    else hipLaunchKernelGGL((k_gemm_tile<T, WM, WN, NW, S, 0>), grid, dim3(128 * NW), lds, stream, A, lda, B, ldb, C, ldc, R, ldr, M, N, K, tilesM, tilesN, alpha, counters, partials);
    return hipGetLastError();
}

// What a launch takes, in microseconds: `slots` workgroups share a compute unit at a time; a round of the chip with k of
// them on a unit takes slices * us[k - 1] + 3.  us: measured per K slice with one, two and three workgroups on every
// unit (the loads, barriers and LDS reads of a workgroup hide behind the others' MFMAs).
struct TileCost { int tm, tn, slots; double us[3]; };
// Variants of the two-byte types: 64 x 64; 128 x 128 with two stages, two workgroups a unit; halves only (what the models multiply): 128 x 128
// with four stages, for launches that put one on a unit: nothing but its own stages then covers the way of a slice from memory.  777 x 2048 x 5888, K split in two, weights cold
// (a prefill reads each once): 36.8 us against 48.3 with two stages; on 512 workgroups (3270 rows) 114 against 110.
static const TileCost kCostHalf[3] = {{64, 64, 3, {0.26, 0.38, 0.58}}, {128, 128, 2, {0.64, 1.04, 0.0}}, {128, 128, 1, {0.58, 0.0, 0.0}}};
static const TileCost kCostP3[2] = {{64, 64, 2, {0.39, 0.75, 0.0}}, {128, 128, 1, {1.28, 0.0, 0.0}}};
#define TL_SPLIT_US(ks) ((ks) > 1 ? 4.0 + 0.5 * (ks) : 0.0) // the partial tiles' way through memory and their sum

static double tile_us(const TileCost& c, int M, int N, int slices, int cus, int ks) {
    const long tiles = (long)((M + c.tm - 1) / c.tm) * ((N + c.tn - 1) / c.tn) * ks;
    const long full = tiles / ((long)cus * c.slots), rest = tiles - full * cus * c.slots;
    const double n = (double)((slices + ks - 1) / ks);
    double us = full * (n * c.us[c.slots - 1] + 3.0);
    if (rest) us += n * c.us[(rest + cus - 1) / cus - 1] + 3.0;
    return us + TL_SPLIT_US(ks);
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
    const bool p3 = dtype == MLH_GEMM_P3;
    const int slices = K / (p3 ? P3_BLOCK : 64);
    double best = 0.0;
    for (int v = 0; v < (dtype == MLH_GEMM_F16 ? 3 : 2); v++) {
        int ks;
        const double us = best_split(p3 ? kCostP3[v] : kCostHalf[v], M, N, slices, cus, ws, ks);
        if (v == 0 || us < best) { best = us; c.variant = v; c.ks = ks; }
    }
    return best;
}
double mlh_gemm_tile_us(int dtype, int M, int N, int K, int cus, bool ws) {
    TileChoice c;
    return tile_choice(dtype, M, N, K, cus, ws, c);
}

hipError_t mlh_gemm_tile(hipStream_t stream, int dtype, int epi, const void* A, int lda, const void* B, int ldb, void* C, int ldc,
                         const float* R, int ldr, int M, int N, int K, void* ws, float alpha) {
    const int cus = mlh_gemm_num_cus();
    if (!cus) return hipErrorInvalidDevice;
    TileChoice c;
    tile_choice(dtype, M, N, K, cus, ws != nullptr, c);
#define TILE(T_, WM_, WN_, NW_, S_) launch_tile<T_, WM_, WN_, NW_, S_>(stream, epi, A, lda, B, ldb, C, ldc, R, ldr, M, N, K, ws, alpha, c.ks)
    // Measured (517 x 768 x 3072, 517 x 6144 x 768, 17000 x 768 x 2048; us): planes 27, 35, 335 -- fp32 MFMA tiles of 256 x 256 took
    // 701, 187, 512 --, halves 13, 13, 69.  fp32: 64 x 64 by eight waves of 32 x 16, three stages (two workgroups a unit), or
    // 128 x 128 by eight waves of 64 x 32, two stages.  Two-byte operands: 64 x 64 by four waves of 32 x 32, three stages, or
    // 128 x 128 by eight waves, two stages (two workgroups a unit) or, halves, four (one).
    if (dtype == MLH_GEMM_P3) return c.variant == 0 ? TILE(p3_t, 2, 1, 4, 3) : TILE(p3_t, 4, 2, 4, 2);
    if (dtype == MLH_GEMM_F16) return c.variant == 0 ? TILE(f16_t, 2, 2, 2, 3) : c.variant == 1 ? TILE(f16_t, 4, 2, 4, 2) : TILE(f16_t, 4, 2, 4, 4);
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
