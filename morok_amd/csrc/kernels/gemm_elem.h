// What the 16-bit product kernels share: element vectors, roundings, the sum with an addend, and the order in which
// workgroups take the output tiles.
#pragma once
#include <hip/hip_runtime.h>

namespace mrk::dev {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
// the same in memory where a row of 16-bit (of 32-bit) elements may start on any element
typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef f32x4 f32x4_any __attribute__((aligned(4)));

#define LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

// Maps the linear workgroup id to an output tile so that the workgroups that land on one
// XCD (ids congruent mod 8 share an L2) cover a compact block of tiles: first regroup
// ids by XCD, then walk tiles in column groups of 4 tile-rows.
__device__ __forceinline__ void tile_of_block(int bid, int tiles_m, int tiles_n, int* tm, int* tn) {
    const int total = tiles_m * tiles_n;
    const int per = total >> 3, rem = total & 7;
    const int xcd = bid & 7, idx = bid >> 3;
    int id = xcd * per + (xcd < rem ? xcd : rem) + idx;
    if (total < 8) id = bid;
    constexpr int kGroup = 4;
    const int group_sz = kGroup * tiles_n;
    const int g = id / group_sz;
    const int first_m = g * kGroup;
    const int gm = (tiles_m - first_m) < kGroup ? (tiles_m - first_m) : kGroup;
    const int in = id - g * group_sz;
    *tm = first_m + in % gm;
    *tn = in / gm;
}

// Sixteen zero bytes in device memory: where the copies of a partial last K step point the
// lanes whose k lies beyond K.
static __device__ __attribute__((aligned(16))) const unsigned g_zero16[4] = {0u, 0u, 0u, 0u};

template <bool kF16>
__device__ __forceinline__ bf16x4 round_to_elem(const f32x4& v) {
    if constexpr (kF16) return __builtin_bit_cast(bf16x4, __builtin_convertvector(v, f16x4));
    else return __builtin_convertvector(v, bf16x4);
}
// the sum of two chunks of eight 16-bit elements, taken in f32 and rounded once
template <bool kF16>
__device__ __forceinline__ u32x4 add_elems(const u32x4& a, const u32x4& b) {
    if constexpr (kF16) {
        const f32x8 s = __builtin_convertvector(__builtin_bit_cast(f16x8, a), f32x8) + __builtin_convertvector(__builtin_bit_cast(f16x8, b), f32x8);
        return __builtin_bit_cast(u32x4, __builtin_convertvector(s, f16x8));
    } else {
        const f32x8 s = __builtin_convertvector(__builtin_bit_cast(bf16x8, a), f32x8) + __builtin_convertvector(__builtin_bit_cast(bf16x8, b), f32x8);
        return __builtin_bit_cast(u32x4, __builtin_convertvector(s, bf16x8));
    }
}

}  // namespace mrk::dev
