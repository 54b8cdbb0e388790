// fp32 matrices as IEEE halves, for the prefill's products on the half-precision matrix cores at fp32 precision.
//
// A row is scaled by a power of two that brings its largest element into [2^14, 2^15).  An element x of it is hi + lo + tiny with hi = half(x),
// lo = half(x - hi), tiny = half(x - hi - lo), each rounded to nearest even.  Weights keep the three: elements down to 2^-15 of the row's largest
// exactly, smaller ones to 2^-39 of it.  Activations keep hi and lo: elements down to 2^-16 of the row's largest to 2^-23 of themselves, three in four of them
// exactly, smaller ones to 2^-39 of the largest.  (Models whose rows spread far enough for that to matter multiply planes: operand_spread in
// kernels_prefill.hip.)  A product a.b is
// formed from hi.tiny, lo.hi, hi.lo and hi.hi, every one exact in the fp32 accumulator; lo.lo and lo.tiny, below 2^-22 of |a||b|, are left out.  That
// moves a sum of normal terms by 6.2e-8 (rms, of |a||b| / sqrt(K)), whatever K is; what the accumulator rounds on the way is more, and grows with the
// number of matrix instructions: four here for 32 columns where three bf16 planes (p3.h) take six.  Measured against float64 (rms, of the product's
// norm), K = 768, 832, 2048: planes 4.3e-7, 4.5e-7, 7.1e-7; here 3.1e-7, 3.2e-7, 5.0e-7; an fp32 library product 5.0e-7, 5.2e-7, 8.1e-7.  Logits of six layers of
// width 768, 90 to 200 tokens, weights of 0.02 to 0.1: 2.2 to 3.8e-6 with planes, 1.6 to 2.7e-6 here.
// (Pairs for the weights too: 422 us, not 496, at 19470 x 4096 x 768, and no further off; but then weights are not what was uploaded.)
//
// Storage: 32 activations of a row take 128 bytes, their hi and then their lo halves, which is what 32 floats take: rows are converted in
// place.  32 weights take 192.  Beside a matrix an exponent per row, of the power of two that takes the scaled row back; the epilogue adds the row's of both.
//
// FFN units are written by many workgroups a row, and no pass finds their rows' scale: they have a scale per column instead, from a bound on what the
// unit can be (k_unit_exps in kernels_prefill.hip), and W2's columns take it back before its rows are scaled.  Units are typically 2^-11 of
// the bound; those of 2^-16 of it and more are kept to 2^-23, the rest to 2^-39 of the bound.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

struct h2_t { uint16_t bits[2]; }; // names the form; rows are addressed in bytes

typedef _Float16 h2_f16x2 __attribute__((ext_vector_type(2)));

// The exponent of a row: of the largest of h2_size over its elements.  (Infinite or NaN elements: the row's products are NaN whatever it is.)
__device__ __forceinline__ int h2_size(float x) { return x != 0.f ? __builtin_amdgcn_frexp_expf(x) : -100000; }
__device__ __forceinline__ int h2_size4(float a, float b, float c, float d) { return max(max(h2_size(a), h2_size(b)), max(h2_size(c), h2_size(d))); }
__device__ __forceinline__ int h2_exponent(int most) { return most > -100000 ? most - 15 : 0; }
// four neighbouring elements, scaled (col a multiple of 4), of the row that starts at `row`
template <bool TRIPLES> __device__ __forceinline__ void h2_put4(void* row, int col, float a, float b, float c, float d) {
    float v[4] = {a, b, c, d};
    unsigned char* p = (unsigned char*)row + (size_t)(col >> 5) * (TRIPLES ? 192 : 128) + (size_t)(col & 31) * 2;
#pragma unroll
    for (int k = 0; k < (TRIPLES ? 3 : 2); k++) {
        const h2_f16x2 x = {(_Float16)v[0], (_Float16)v[1]}, y = {(_Float16)v[2], (_Float16)v[3]};
        *reinterpret_cast<uint2*>(p + k * 64) = make_uint2(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y));
        v[0] -= (float)x[0]; v[1] -= (float)x[1]; v[2] -= (float)y[0]; v[3] -= (float)y[1];
    }
}
