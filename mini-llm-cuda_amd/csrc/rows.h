// Operands of the products of a decode step of up to 64 sequences (kernels_rows.hip).
//
// Activations: three bf16 planes (p3.h) in the order of the MFMA operand.  Token rows go in blocks of T = 1, 2, 4, 8 or 16 (the
// smallest that holds the batch; up to four blocks of 16), columns in blocks of 32.  Block (kb, plane, tb) is 64 T bytes: position
// q T + t has the 16 bytes of token t of the block, eight of the 32 columns: columns 8 q .. 8 q + 7 beside bf16 weights, columns
// 4 q .. 4 q + 3 and 16 + 4 q .. 19 + 4 q beside fp32 weights.
//
// Weights: the matrix once more in the order the waves fetch it.  A tile is 16 rows, a chunk 128 bytes of each; (tile, chunk) is 2 KB:
// load p (0, 1) of lane 16 q + r is the 16 bytes at p 64 + q 16 of row r's 128.  A fetch of 1 KB contiguous bytes runs three
// times as fast through a compute unit's L1 as one of 16 rows of 64 bytes.
#pragma once
#include "p3.h"

struct RowsLayout {
    int t, blocks; // tokens per block, blocks
    __host__ __device__ __forceinline__ int stride() const { return 64 * t * blocks; } // bytes from one plane of a column block to the next
};
inline RowsLayout rows_layout(int n) {
    RowsLayout l = {1, n <= 16 ? 1 : n <= 32 ? 2 : 4};
    while (l.t < 16 && l.t < n) l.t *= 2;
    return l;
}

// byte offset, in plane 0, of the four neighbouring columns k .. k + 3 (k a multiple of 4) of token m; `half`: bf16 weights
__device__ __forceinline__ size_t rows_offset(int k, int m, RowsLayout l, bool half) {
    const int q = half ? (k & 31) >> 3 : (k & 15) >> 2, e = half ? k & 4 : (k & 16) >> 2, tb = m >> 4; // (more than one block: t is 16)
    return (size_t)(k >> 5) * 3 * l.stride() + (size_t)((tb * 4 + q) * l.t + (m & 15)) * 16 + e * 2;
}
__device__ __forceinline__ void rows_put4(void* planes, int k, int m, RowsLayout l, bool half, float a, float b, float c, float d) {
    uint32_t x[3], y[3];
    p3_split2(a, b, x);
    p3_split2(c, d, y);
    unsigned char* p = (unsigned char*)planes + rows_offset(k, m, l, half);
#pragma unroll
    for (int pl = 0; pl < 3; pl++) *reinterpret_cast<uint2*>(p + pl * l.stride()) = make_uint2(x[pl], y[pl]);
}
__device__ __forceinline__ void rows_put(void* planes, int k, int m, RowsLayout l, bool half, float v) {
    uint32_t w[3];
    p3_split2(v, 0.f, w);
    unsigned char* p = (unsigned char*)planes + rows_offset(k & ~3, m, l, half) + (k & 3) * 2;
#pragma unroll
    for (int pl = 0; pl < 3; pl++) *reinterpret_cast<uint16_t*>(p + pl * l.stride()) = (uint16_t)w[pl];
}

#define RW_TILE 16 // weight rows of a tile
enum { RW_PLAIN, RW_RESID, RW_SWIGLU, RW_LOGITS };

struct RowsArgs {
    const unsigned char* W;         // in fetch order (rows.h)
    int M, N, K, tiles;
    RowsLayout lay;                 // of the plane buffers
    const unsigned char* A;         // planes of the input rows
    const float* ssqIn;             // [nparts][64] partial sums of squares of the rows behind A, or null: no normalisation
    int nparts, normDim;
    float* C;                       // RW_PLAIN, RW_RESID: [M, ldc] fp32; RW_LOGITS: row sidx[m] of [*, ldc]
    int ldc;
    const float* R;                 // RW_RESID: added to the product, [M, ldc]
    unsigned char* out;             // RW_RESID: planes of outGain (.) C; RW_SWIGLU: planes of silu(gate) * up
    const float* outGain;
    float* ssqOut;                  // RW_RESID: [workgroup][64]
    const int* sidx;
    float* amaxVal;                 // RW_LOGITS: [M, amaxParts] largest logit of each workgroup's rows and its index
    int* amaxIdx;
    int amaxParts;
    int* stepCounter;               // RW_LOGITS: counted up once
};
