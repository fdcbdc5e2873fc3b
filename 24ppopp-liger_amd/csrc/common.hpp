// common.hpp -- shared device helpers for the gfx950 (CDNA4, wave64) kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/liger_hip.h"

namespace lg {

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef unsigned uint2_t __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;

// thread-local error text, set by the host-side launchers
void set_error(const char* fmt, ...);
int check_launch(const char* what);

// What is known about a stream (runtime.hip): the compute units its kernels may run on (fewer than the device for a CU-masked
// stream) and its split-K workspace (nullptr for a stream the library neither created nor was told about with lg_stream_attach).
constexpr size_t LG_SPLITK_WORKSPACE_BYTES = (size_t)64 << 20;
constexpr int LG_ARRIVAL_COUNTERS = 4096;
struct StreamInfo {
    int cus;
    float* ws;
    size_t ws_bytes;
    unsigned* arrivals;  // LG_ARRIVAL_COUNTERS counters behind the workspace, zero between launches
};
StreamInfo stream_info(hipStream_t stream);
int device_cu_count();

// A butterfly step v = op(v of this lane, v of lane ^ O) as vector instructions (data-parallel primitives and lane swaps, a few cycles each)
// instead of a trip through the LDS crossbar (over a hundred), with the same bits: LayerNorm of 32 rows of 12288 halves 4.7 -> 4.1 us, of 4096 35.2 -> 33.4,
// 4096 fp32 rows of 1024 8.4 -> 6.2.  Steps of 8 and 4 rotate rows of 16 lanes:
// rotating by 4 reaches lane ^ 4 only where lanes 8 apart hold the same value (AFTER8), as they do after the step of 8; else it takes two moves.
template <int O, bool AFTER8, class Op>
__device__ __forceinline__ float lane_step(float v, Op op) {
    const int u = __builtin_bit_cast(int, v);
    auto moved = [](int x, auto control) { return __builtin_amdgcn_update_dpp(0, x, decltype(control)::value, 0xf, 0xf, false); };
    typedef std::integral_constant<int, 0xb1> Swap1;            // lanes 1 0 3 2 of every four
    typedef std::integral_constant<int, 0x4e> Swap2;            // 2 3 0 1
    typedef std::integral_constant<int, 0x1b> Reverse4;         // 3 2 1 0
    typedef std::integral_constant<int, 0x141> Reverse8;        // 7 .. 0 of every eight
    typedef std::integral_constant<int, 0x124> Rotate4;
    typedef std::integral_constant<int, 0x128> Rotate8;
    if constexpr (O >= 16) {  // of both results one is this lane's own value and the other its partner's
        uint2_t r;
        if constexpr (O == 16) r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        else r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        const unsigned first = r[0], second = r[1];
        return op(__builtin_bit_cast(float, first), __builtin_bit_cast(float, second));
    } else {
        int w;
        if constexpr (O == 8) w = moved(u, Rotate8{});
        else if constexpr (O == 4 && AFTER8) w = moved(u, Rotate4{});
        else if constexpr (O == 4) w = moved(moved(u, Reverse8{}), Reverse4{});
        else if constexpr (O == 2) w = moved(u, Swap2{});
        else w = moved(u, Swap1{});
        return op(v, __builtin_bit_cast(float, w));
    }
}
// all steps from G / 2 down to 1: every lane of G adjacent ones gets the result over them
template <int G, class Op>
__device__ __forceinline__ float lanes_reduce(float v, Op op) {
    static_assert(G == 4 || G == 8 || G == 16 || G == 32 || G == 64, "groups in use");
    if constexpr (G == 64) v = lane_step<32, false>(v, op);
    if constexpr (G >= 32) v = lane_step<16, false>(v, op);
    if constexpr (G >= 16) v = lane_step<8, false>(v, op);
    if constexpr (G >= 8) v = lane_step<4, (G >= 16)>(v, op);
    v = lane_step<2, false>(v, op);
    return lane_step<1, false>(v, op);
}
template <int G>
__device__ __forceinline__ float lanes_sum(float v) {
    return lanes_reduce<G>(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_sum(float v) { return lanes_sum<kWave>(v); }
template <int G>
__device__ __forceinline__ float lanes_max(float v) {
    return lanes_reduce<G>(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_max(float v) { return lanes_max<kWave>(v); }

// Block-wide sum for up to 1024 threads (16 waves); every thread gets the result.
// `scratch` must hold 16 floats; two back-to-back calls may reuse it (barrier at entry).
__device__ __forceinline__ float block_sum(float v, float* scratch) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    v = wave_sum(v);
    if (nw == 1) return v;
    __syncthreads();
    if (lane == 0) scratch[wid] = v;
    __syncthreads();
    float r = (lane < nw) ? scratch[lane] : 0.f;
    return wave_sum(r);
}
__device__ __forceinline__ float block_max(float v, float* scratch) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    v = wave_max(v);
    if (nw == 1) return v;
    __syncthreads();
    if (lane == 0) scratch[wid] = v;
    __syncthreads();
    float r = (lane < nw) ? scratch[lane] : -3.0e38f;
    return wave_max(r);
}

// scalar load/store helpers that work for both element types
template <typename T> __device__ __forceinline__ float ldf(const T* p) { return (float)(*p); }
template <typename T> __device__ __forceinline__ void stf(T* p, float v) { *p = (T)v; }

// 16-byte vector of T
// at any alignment: global memory takes loads and stores of these as whole ones
typedef half_t half4u_t __attribute__((ext_vector_type(4), aligned(2)));
typedef half_t half8u_t __attribute__((ext_vector_type(8), aligned(2)));

template <typename T> struct Vec16;
template <> struct Vec16<float> {
    static constexpr int N = 4;
    float4_t v;
    __device__ __forceinline__ float get(int i) const { return v[i]; }
    __device__ __forceinline__ void set(int i, float x) { v[i] = x; }
};
template <> struct Vec16<half_t> {
    static constexpr int N = 8;
    half8_t v;
    __device__ __forceinline__ float get(int i) const { return (float)v[i]; }
    __device__ __forceinline__ void set(int i, float x) { v[i] = (half_t)x; }
};

__device__ __forceinline__ float gelu_tanh(float x) {
    // 0.5 x (1 + tanh(0.79788456 (x + 0.044715 x^3)))   (reference cuda_kernels.cu:9-15)
    // evaluated as x / (1 + exp(-2u)), the same function with one hardware exp2 and one reciprocal
    const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    const float e = __builtin_amdgcn_exp2f(-2.0f * 1.4426950408889634f * u);  // inf for very negative x: result -0
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
__device__ __forceinline__ bool aligned_dev16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace lg
