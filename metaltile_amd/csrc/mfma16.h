// Helpers of the GEMV kernels on the 16x16x32 matrix instruction (qmv_runs_impl.h).
#pragma once
#include "mtq_device.h"

#include <type_traits>

namespace mtq {

typedef uint32_t kr_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t kr_u32x2 __attribute__((ext_vector_type(2)));
typedef float kr_f32x4 __attribute__((ext_vector_type(4)));

template <int DT> __device__ __forceinline__ kr_f32x4 kr_mfma(kr_u32x4 a, kr_u32x4 b, kr_f32x4 c) {
    if constexpr (DT == DT_BF16) {
        typedef __attribute__((ext_vector_type(8))) __bf16 v8;
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    } else {
        typedef __attribute__((ext_vector_type(8))) _Float16 v8;
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
    }
}

template <int B, int E, class F> __device__ __forceinline__ void kr_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        kr_for<B + 1, E>(f);
    }
}

// Between a wave's writes to its own LDS and its reads of what other lanes wrote (LDS operations of a wave complete in order: no wait).
__device__ __forceinline__ void kr_turned() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

constexpr uint32_t KR_OOB = 0x80000000u;   // every buffer is shorter than 2 GiB (host): base + KR_OOB is out of range for any base below 2 GiB
constexpr int KR_NT = 2;                   // cache policy of the weights: read once

__device__ __forceinline__ __amdgpu_buffer_rsrc_t kr_rsrc(uint64_t a, uint32_t bytes) {
    // (the base is the same in every lane: the descriptor is kept in scalar registers)
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), 0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

template <int DT> __device__ __forceinline__ float kr_elem(uint32_t dw, int odd) {
    if constexpr (DT == DT_BF16) return __uint_as_float(odd ? (dw & 0xFFFF0000u) : (dw << 16));
    else return f16_bits_to_f32(odd ? (dw >> 16) : (dw & 0xFFFFu));
}

}  // namespace mtq
