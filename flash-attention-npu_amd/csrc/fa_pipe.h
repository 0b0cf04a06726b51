// fa_pipe.h -- what the kernels with one wave per SIMD share: 32x32x16
// products, LDS tiles of 256-byte rows that are read by rows and transposed,
// loads straight into LDS.
#pragma once
#include "fa_common.h"

namespace fa {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// 32x32x16 MFMA on 16-byte packed operands. Lane l holds A[l%32][8*(l/32)+e]
// and B[8*(l/32)+e][l%32]; the result lane l holds D[8*(i/4)+4*(l/32)+i%4][l%32].
template <int DT>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (DT == DT_FP16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <int DT>
__device__ __forceinline__ uint32_t pack2(float x, float y) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    if constexpr (DT == DT_FP16) {
        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x, y}), f16x2));
    } else {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x, y}), bf16x2));
    }
}

// Slot of 16-byte chunk c in row r of a tile. Conflict free for ds_read_b128 of
// one chunk of 32 rows and for the transpose reads of 4 rows x 4 chunks.
__device__ __forceinline__ int swz(int r, int c) { return c ^ (((r & 3) << 2) | ((r >> 2) & 3)); }

__device__ __forceinline__ u32x4 tr_read(unsigned lo, unsigned hi) {
    const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(size_t)lo));
    const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(size_t)hi));
    return u32x4{a[0], a[1], b[0], b[1]};
}
// 8 rows of one byte column: of 16 lanes, lane i gives the address of 8 bytes
// (half i & 1 of 16 columns) of row i >> 1 and gets column i
__device__ __forceinline__ u32x2 tr8_read(unsigned a) {
    typedef int i32x2 __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) i32x2 lds_i32x2;
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*)(size_t)a));
}
__device__ __forceinline__ u32x4 row_read(unsigned a) {
    return *(const __attribute__((address_space(3))) u32x4*)(size_t)a;
}
__device__ __forceinline__ float float_read(unsigned a) {
    return *(const __attribute__((address_space(3))) float*)(size_t)a;
}
// A pointer that is the same in all lanes, for an operand that has to be scalar
__device__ __forceinline__ const char* uniform(const char* p) {
    const uint64_t x = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x), hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
    return (const char*)(((uint64_t)hi << 32) | lo);
}
// Loads straight into LDS: 16 bytes per lane from base + off[u] to the LDS
// address lds + 1024 u + 16 lane (u < 4; 4 bytes to lds + 4 lane). The
// instruction's offset moves both addresses, so off[u] holds (3 - u) KB more
// and `base` is 3 KB less. In assembly, because the compiler would wait for
// every such load before any LDS read; wait_loads<N> waits until all but the
// wave's last N are there. Nor does it put wait states inside the block: five
// instructions' worth lie between the readfirstlanes of the address and the first
// load (gfx9's distance from a vector write of a scalar register to a memory
// instruction that reads it), the write of m0 among them.
__device__ __forceinline__ void dma16x4(unsigned lds, const char* base, const unsigned (&off)[4]) {
    base = uniform(base);
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile(
        "s_mov_b32 m0, %0\n\ts_nop 3\n\t"
        "global_load_lds_dwordx4 %2, %1\n\t"
        "global_load_lds_dwordx4 %3, %1 offset:1024\n\t"
        "global_load_lds_dwordx4 %4, %1 offset:2048\n\t"
        "global_load_lds_dwordx4 %5, %1 offset:3072" ::"s"(lds), "s"(base), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3])
        : "memory", "m0");
}
// The same by the lanes of mask[u] in load u; the LDS bytes of the others stay
__device__ __forceinline__ void dma16x4(unsigned lds, const char* base, const unsigned (&off)[4], const uint64_t (&mask)[4]) {
    base = uniform(base);
    lds = __builtin_amdgcn_readfirstlane(lds);
    uint64_t all;
    asm volatile(
        "s_mov_b32 m0, %1\n\ts_mov_b64 %0, exec\n\ts_nop 1\n\t"
        "s_mov_b64 exec, %7\n\tglobal_load_lds_dwordx4 %3, %2\n\t"
        "s_mov_b64 exec, %8\n\tglobal_load_lds_dwordx4 %4, %2 offset:1024\n\t"
        "s_mov_b64 exec, %9\n\tglobal_load_lds_dwordx4 %5, %2 offset:2048\n\t"
        "s_mov_b64 exec, %10\n\tglobal_load_lds_dwordx4 %6, %2 offset:3072\n\t"
        "s_mov_b64 exec, %0"
        : "=&s"(all)
        : "s"(lds), "s"(base), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(mask[0]), "s"(mask[1]), "s"(mask[2]), "s"(mask[3])
        : "memory", "m0");
}
__device__ __forceinline__ void dma4(unsigned lds, const char* base, unsigned off) {
    base = uniform(base);
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dword %2, %1" ::"s"(lds), "s"(base), "v"(off) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}
__device__ __forceinline__ void row_write(unsigned a, u32x4 v) {
    *(__attribute__((address_space(3))) u32x4*)(size_t)a = v;
}
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }


}  // namespace fa
