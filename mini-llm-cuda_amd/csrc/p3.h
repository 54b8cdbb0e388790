// fp32 matrices as three bf16 planes, for products on the bf16 matrix cores at fp32 precision.
//
// x = hi + mid + lo with hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid), each rounded to nearest even: three
// times eight significand bits hold the 24 of x, so the sum is exact (down to the bf16 denormals).  A product a.b is formed from
// the six plane products hi.hi, hi.mid, mid.hi, mid.mid, hi.lo, lo.hi, every one exact in the fp32 accumulator; what
// is left out (mid.lo, lo.mid, lo.lo) is below 2^-25 of |a||b|, less than one fp32 rounding of it.
//
// Storage: 32 elements of a row take 192 bytes, their hi, mid and lo halves in turn (64 bytes each); a row of K elements
// (K a multiple of 32) is K * 6 bytes.  Leading dimensions are counted in elements.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define P3_BLOCK 32   // elements per block
#define P3_BYTES 192  // bytes per block
#define P3_PLANE 64   // bytes from one plane of a block to the next

struct p3_t { uint16_t bits[3]; }; // only its size (6 bytes per element) is used; rows are addressed in bytes

typedef float p3_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 p3_bf16x2 __attribute__((ext_vector_type(2)));

// the planes of two neighbouring elements, packed two to a word
__device__ __forceinline__ void p3_split2(float a, float b, uint32_t (&w)[3]) {
#pragma unroll
    for (int p = 0; p < 3; p++) {
        const p3_f32x2 v = {a, b};
        w[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, p3_bf16x2));
        a -= __uint_as_float(w[p] << 16);
        b -= __uint_as_float(w[p] & 0xffff0000u);
    }
}
__device__ __forceinline__ size_t p3_offset(int col) { return (size_t)(col >> 5) * P3_BYTES + (size_t)(col & 31) * 2; }
// one element / four neighbouring elements (col a multiple of 4) of the row that starts at `row`
__device__ __forceinline__ void p3_put(void* row, int col, float v) {
    uint32_t w[3];
    p3_split2(v, 0.f, w);
    unsigned char* p = (unsigned char*)row + p3_offset(col);
#pragma unroll
    for (int k = 0; k < 3; k++) *reinterpret_cast<uint16_t*>(p + k * P3_PLANE) = (uint16_t)w[k];
}
__device__ __forceinline__ void p3_put4(void* row, int col, float a, float b, float c, float d) {
    uint32_t x[3], y[3];
    p3_split2(a, b, x);
    p3_split2(c, d, y);
    unsigned char* p = (unsigned char*)row + p3_offset(col);
#pragma unroll
    for (int k = 0; k < 3; k++) *reinterpret_cast<uint2*>(p + k * P3_PLANE) = make_uint2(x[k], y[k]);
}
