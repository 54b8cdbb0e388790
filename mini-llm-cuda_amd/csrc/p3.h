// fp32 matrices as three bf16 planes, for products on the bf16 matrix cores at fp32 precision.
//
// x = hi + mid + lo with hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid), each rounded to nearest even: three
// times eight significand bits hold the 24 of x, so the sum is exact (down to the bf16 denormals).  A product a.b is formed from
// the six plane products hi.hi, hi.mid, mid.hi, mid.mid, hi.lo, lo.hi, every one exact in the fp32 accumulator; what
// is left out (mid.lo, lo.mid, lo.lo) is below 2^-24 of |a||b|: over all significands |mid| <= 2^-8.006 |a| and |lo| <= 2^-17.003 |a|,
// at worst 0.995 2^-24 together, which is what rounding the product to fp32 may cost.  In sums it is far less: of 768 normal terms it
// moves the result by 5.7e-9 (rms, of |a||b| / sqrt(768)), a sequential fp32 sum by 5.1e-7; of 3072, 5.6e-9 against 1.0e-6.
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

// Magnitudes from here on (as bits: infinities and NaN too) have no finite bf16 nearest to them.
#define P3_BEYOND 0x7f7f8000u
__device__ __forceinline__ bool p3_beyond(float v) { return (__float_as_uint(v) & 0x7fffffffu) >= P3_BEYOND; }

// The planes of two neighbouring elements, packed two to a word.  Beyond P3_BEYOND they make NaN of every product: weights and gains
// that reach it keep a model off this path (mlh_build_gemm_operands).  An activation that does has overflowed: its row's sum of
// squares is infinite or NaN at the next norm, whatever this product gives.
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
// The planes of an element beyond.  An infinity goes into the plane that meets the other operand's hi plane alone, with
// +-1 in front of it: its plane products with a finite b are +-b, 0 and the infinity times hi(b), so their sum is what inf * b
// is (NaN for b = 0), and with another infinity it is that infinity.  The largest finite values are cut instead of rounded (no
// plane exceeds the value; exact as well).
__device__ __forceinline__ void p3_split_beyond(float a, uint32_t (&h)[3]) {
    const uint32_t u = __float_as_uint(a);
    if ((u & 0x7fffffffu) >= 0x7f800000u) {
        const bool nan = (u & 0x7fffffu) != 0;
        h[0] = nan ? 0x7fc0u : 0x3f80u | (u >> 31 << 15);
        h[1] = 0;
        h[2] = nan ? 0u : u >> 16;
        return;
    }
    h[0] = u >> 16;
    a -= __uint_as_float(u & 0xffff0000u);
    h[1] = __float_as_uint(a) >> 16;
    a -= __uint_as_float(h[1] << 16);
    h[2] = __float_as_uint(a) >> 16;
}
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
