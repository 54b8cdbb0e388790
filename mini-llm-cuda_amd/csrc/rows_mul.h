// One chunk of a product of the row kernels' operands (rows.h): 16 weight rows x 128 bytes, straight from registers.
#pragma once
#include "p3.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <typename WT> struct RowsW;
template <> struct RowsW<float> {
    static constexpr int KE = 32, SUB = 1; // K per chunk, 32-wide steps per chunk
    u32x4 raw[2];
    __device__ __forceinline__ void load(const unsigned char* chunk) { // this lane's place in a chunk
#pragma unroll
        for (int p = 0; p < 2; p++) raw[p] = *reinterpret_cast<const u32x4*>(chunk + p * 1024);
    }
    template <int MB> __device__ __forceinline__ void mul(const u32x4 (&a)[1][3][MB], f32x4 (&acc)[MB]) const {
        u32x4 w[3];
        uint32_t s[4][3];
#pragma unroll
        for (int p = 0; p < 2; p++) {
            p3_split2(__uint_as_float(raw[p].x), __uint_as_float(raw[p].y), s[2 * p]);
            p3_split2(__uint_as_float(raw[p].z), __uint_as_float(raw[p].w), s[2 * p + 1]);
        }
#pragma unroll
        for (int pl = 0; pl < 3; pl++) { w[pl].x = s[0][pl]; w[pl].y = s[1][pl]; w[pl].z = s[2][pl]; w[pl].w = s[3][pl]; }
#pragma unroll
        for (int sum = 2; sum >= 0; sum--)
#pragma unroll
            for (int pw = 0; pw <= sum; pw++)
#pragma unroll
                for (int mb = 0; mb < MB; mb++)
                    acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[pw]), __builtin_bit_cast(bf16x8, a[0][sum - pw][mb]), acc[mb], 0, 0, 0);
    }
};
template <> struct RowsW<bf16_t> {
    static constexpr int KE = 64, SUB = 2;
    u32x4 raw[2];
    __device__ __forceinline__ void load(const unsigned char* chunk) {
#pragma unroll
        for (int p = 0; p < 2; p++) raw[p] = *reinterpret_cast<const u32x4*>(chunk + p * 1024);
    }
    template <int MB> __device__ __forceinline__ void mul(const u32x4 (&a)[2][3][MB], f32x4 (&acc)[MB]) const {
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
            for (int pl = 2; pl >= 0; pl--)
#pragma unroll
                for (int mb = 0; mb < MB; mb++)
                    acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, raw[p]), __builtin_bit_cast(bf16x8, a[p][pl][mb]), acc[mb], 0, 0, 0);
    }
};
