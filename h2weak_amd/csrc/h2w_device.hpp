// h2w_device.hpp -- device helpers that the real and the complex kernels share: exchanges between the
// lanes of a wave, streaming and buffer loads, scalar reads of the work lists.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "h2w_internal.hpp"

namespace h2w {
// the FP64 buffer atomic's intrinsic (no clang builtin; a compiler that did not know it would fail at the link)
__device__ double buf_fadd64(double v, __amdgpu_buffer_rsrc_t r, int voff, int soff, int aux) __asm(
    "llvm.amdgcn.raw.ptr.buffer.atomic.fadd.f64");
namespace {

// Value of lane (lane ^ O) for a power of two O < 64: quad permutes (DPP) for 1 and 2,
// ds_swizzle in its bit-mask mode for 4 .. 16, ds_bpermute for 32.  Every lane of the
// aligned group of 2 O lanes must be active.
template <int O>
__device__ __forceinline__ int xor_lane(int v) {
    if constexpr (O == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);
    else if constexpr (O == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);
    else if constexpr (O < 32) return __builtin_amdgcn_ds_swizzle(v, 0x1F | (O << 10));
    else return __builtin_amdgcn_ds_bpermute((int)(((threadIdx.x & 63) ^ O) << 2), v);
}
template <int O>
__device__ __forceinline__ float xor_lane(float v) {
    return __int_as_float(xor_lane<O>(__float_as_int(v)));
}
template <int O>
__device__ __forceinline__ double xor_lane(double v) {
    const int64_t b = __double_as_longlong(v);
    const int lo = xor_lane<O>((int)(uint32_t)b), hi = xor_lane<O>((int)(b >> 32));
    return __longlong_as_double((int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}
// Value of a lane that differs in bit O (1, 2: lane ^ O; 4, 8: rotation by O within a row of 16 lanes,
// which flips bit O and keeps the bits below): enough for sums over whole rows, without the LDS crossbar.
template <int O>
__device__ __forceinline__ double fold_lane(double v) {
    constexpr int ctrl = O == 1 ? 0xB1 : O == 2 ? 0x4E : 0x120 + O;
    const int64_t b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)b, ctrl, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), ctrl, 0xF, 0xF, false);
    return __longlong_as_double((int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}
// sum of a value's four copies at lanes equal modulo 16
__device__ __forceinline__ double sum_halves(double v) {
    auto fold = [](double x, auto swap) {
        const int64_t b = __double_as_longlong(x);
        const auto lo = swap((uint32_t)b), hi = swap((uint32_t)(b >> 32));
        return __longlong_as_double((int64_t)(((uint64_t)hi[0] << 32) | lo[0])) +
               __longlong_as_double((int64_t)(((uint64_t)hi[1] << 32) | lo[1]));
    };
    v = fold(v, [](uint32_t w) { return __builtin_amdgcn_permlane16_swap(w, w, false, false); });
    return fold(v, [](uint32_t w) { return __builtin_amdgcn_permlane32_swap(w, w, false, false); });
}
// the same with O known only after unrolling
template <typename T>
__device__ __forceinline__ T xor_lane_n(T v, int o) {
    switch (o) {
    case 1: return xor_lane<1>(v);
    case 2: return xor_lane<2>(v);
    case 4: return xor_lane<4>(v);
    case 8: return xor_lane<8>(v);
    case 16: return xor_lane<16>(v);
    default: return xor_lane<32>(v);
    }
}

// Streaming load through a global-address-space pointer: operator pointers taken from a
// table in memory are generic to the compiler, whose flat loads would also count against
// the LDS wait counter.
template <typename V>
__device__ __forceinline__ V ld_nt(const V *p) {
    return __builtin_nontemporal_load((const __attribute__((address_space(1))) V *)p);
}

// Raw buffer access (gfx9 resource word 3): a lane whose offset lies at or past the
// resource's size reads zeros and writes nothing, without a branch.
constexpr int kBufWord3 = 0x00020000;
constexpr uint32_t kOutOfRange = 0xFFFFFFF0u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, kBufWord3);
}
// An offset the compiler cannot see through: keeps a load whose offset is selected per
// lane a single unconditional load (instead of one load per alternative under branches).
// The asm is empty and loads nothing.
__device__ __forceinline__ uint32_t opaque_off(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}
template <typename T>
__device__ __forceinline__ T buf_ld(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
template <typename V>
__device__ __forceinline__ V buf_ld16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
template <typename V>
__device__ __forceinline__ V buf_ld16_nt(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2));
}
// Atomic addition without a result; lanes out of range add nothing.
__device__ __forceinline__ void buf_atomic_add(__amdgpu_buffer_rsrc_t r, uint32_t off, double v) {
    (void)buf_fadd64(v, r, (int)off, 0, 0);
}
__device__ __forceinline__ void buf_atomic_add(__amdgpu_buffer_rsrc_t r, uint32_t off, float v) {
    (void)__builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(v, r, (int)off, 0, 0);
}
// one 4-, 8- or 16-byte vector, streamed (not kept in the caches)
template <typename V>
__device__ __forceinline__ V buf_ldv_nt(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    if constexpr (sizeof(V) == 16) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2));
    else if constexpr (sizeof(V) == 8) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 2));
    else return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 2));
}
// N consecutive elements (N sizeof(T) = 8, 16, 32 or 64 bytes) in 8- or 16-byte loads
template <typename T, int N>
__device__ __forceinline__ void buf_ld_n(T (&out)[N], __amdgpu_buffer_rsrc_t r, uint32_t off) {
    constexpr int B = N * (int)sizeof(T);
    if constexpr (B == 8) {
        typedef unsigned int U2 __attribute__((ext_vector_type(2)));
        typedef T W __attribute__((ext_vector_type(N)));
        const W w = __builtin_bit_cast(W, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
#pragma unroll
        for (int k = 0; k < N; ++k) out[k] = w[k];
    } else {
        constexpr int E = 16 / sizeof(T);
        typedef T W __attribute__((ext_vector_type(E)));
#pragma unroll
        for (int p = 0; p < B / 16; ++p) {
            const W w = __builtin_bit_cast(W, __builtin_amdgcn_raw_buffer_load_b128(r, off + 16 * p, 0, 0));
#pragma unroll
            for (int k = 0; k < E; ++k) out[E * p + k] = w[k];
        }
    }
}

// Work lists are never written by a kernel: read through the constant address space, their
// wave-uniform loads stay scalar after the kernel's own stores (a vector load there would
// wait for every load in flight).
typedef const __attribute__((address_space(4))) GTerm CGTerm;
__device__ __forceinline__ GTerm term_at(const CGTerm *p, int k) {
    GTerm t;
    t.a = p[k].a;
    t.x = p[k].x;
    t.t = p[k].t;
    t.cols = p[k].cols;
    t.ld = p[k].ld;
    return t;
}

}  // namespace
}  // namespace h2w
