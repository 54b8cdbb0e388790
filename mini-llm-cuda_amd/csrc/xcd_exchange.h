// What the single-launch decodes of several sequences share: an XCD as a tensor-parallel rank of 32 workgroups, words exchanged through its
// L2 or past it, and the meeting at the start of a launch.
#pragma once
#include "persist_common.h"

typedef __amdgpu_buffer_rsrc_t rsrc_t;

#define RK_XCDS 8
#define RK_PER 32                             // workgroups per XCD
#define RK_SPIN (1u << 20)
#define RK_MEET_SPIN (1u << 14)               // of the meeting at the start (about 20 ms)
#define RK_LEFT 0x10000u                      // in the word that counts them: somebody has gone
#define RK_LDS (160 * 1024)

enum { LD_XCD = 2, LD_CROSS = 16, ST_XCD = 0, ST_CROSS = 16 }; // cache policy of exchange loads and stores: nt leaves no line in the L1 (measured, not promised: words with tags, that are loaded until they are new), sc1 goes past the L2

__device__ __forceinline__ int runi(int v) { return __builtin_amdgcn_readfirstlane(v); }
// The layer table is read by scalar loads where it is used.
typedef const __attribute__((address_space(4))) LayerDev* LayerPtr;

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
template <int POL> __device__ __forceinline__ u32x4 xget(rsrc_t r, unsigned lane, unsigned base) { return __builtin_amdgcn_raw_buffer_load_b128(r, lane, base, POL); }
template <int POL> __device__ __forceinline__ void xput(rsrc_t r, unsigned lane, unsigned base, float a, float b, unsigned tag) { // two words
    const u32x4 v = {__float_as_uint(a), tag, __float_as_uint(b), tag};
    __builtin_amdgcn_raw_buffer_store_b128(v, r, lane, base, POL);
}
__device__ __forceinline__ bool xfresh(const u32x4& v, unsigned tag) { return v.y == tag && v.w == tag; }
template <int W> __device__ __forceinline__ float rk_row_sum(float v) { // over aligned groups of 16 or 32 lanes
    v = pgroup_sum<16>(v);
    if (W == 32) { // the rows of 16 in pairs
        const u32x2 t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(t.x) + __uint_as_float(t.y);
    }
    return v;
}

// Lanes of one wave call it: the workgroup's XCD from the hardware register, its rank inside it from the order of arrival, then a meeting of
// all.  0, or why the launch does not take place (in lane 0).  Nothing has been written by then.
__device__ __forceinline__ unsigned rk_meeting(unsigned* xcdCount, unsigned& xcc, unsigned& rank) {
    // the XCD from the hardware register, the rank inside it from the order of arrival; then a meeting of all
    rank = RK_PER;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    xcc &= 15u;
    if (xcc < RK_XCDS && threadIdx.x == 0) rank = __hip_atomic_fetch_add(xcdCount + xcc, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    rank = (unsigned)runi((int)rank);
    // One word decides: the 256th arrival makes it 256 for good, a workgroup that waits no longer (or has no place) adds
    // RK_LEFT before that, and then nobody goes on.
    unsigned* meet = xcdCount + RK_XCDS;
    unsigned code = rank >= RK_PER ? 2u : 0u;
    if (threadIdx.x == 0) {
        if (code) __hip_atomic_fetch_or(meet, RK_LEFT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else __hip_atomic_fetch_add(meet, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (unsigned spins = 0; !code; spins++) {
            unsigned n = aldu(meet);
            if (n == RK_XCDS * RK_PER) break;
            if (n & RK_LEFT) code = 1u;
            else if (spins > RK_MEET_SPIN) {
                if (__hip_atomic_compare_exchange_strong(meet, &n, n | RK_LEFT, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) code = 1u;
                else spins = RK_MEET_SPIN; // somebody arrived just now: look again
            }
            __builtin_amdgcn_s_sleep(2);
        }
    }
    return code;
}
