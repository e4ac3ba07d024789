// Device helpers of the on-chip solvers (chip.hip, chip_complex.hip): sums over a wavefront and a
// workgroup on the VALU, and register arrays indexed by constants.
#pragma once

#include <utility>

#include "chip.h"
#include "krylov_dev.h"

namespace mpf {

// cross-lane moves on the VALU: quad permutes for l ^ 1 and l ^ 2, rotations within 16 lanes,
// and for the 16- and 32-lane halves gfx950's swaps, which leave both halves' values side by side
constexpr int kXor1 = 0xB1, kXor2 = 0x4E;   // quad_perm [1, 0, 3, 2], [2, 3, 0, 1]
constexpr int kRor4 = 0x124, kRor8 = 0x128;
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const uint64_t b = __double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xF, 0xF, true);
    const uint32_t hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((uint64_t)hi << 32) | lo);
}
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
template <int HALF>
__device__ __forceinline__ v2u swap_halves(uint32_t v) {
    if constexpr (HALF == 16) return __builtin_amdgcn_permlane16_swap(v, v, false, false);
    else return __builtin_amdgcn_permlane32_swap(v, v, false, false);
}
// v of both 16-lane (32-lane) halves of each 32 (64) lanes added, in every lane
template <int HALF>
__device__ __forceinline__ float add_halves(float v) {
    const v2u s = swap_halves<HALF>(__float_as_uint(v));
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
template <int HALF>
__device__ __forceinline__ double add_halves(double v) {
    const uint64_t b = __double_as_longlong(v);
    const v2u lo = swap_halves<HALF>((uint32_t)b), hi = swap_halves<HALF>((uint32_t)(b >> 32));
    return __longlong_as_double(((uint64_t)hi[0] << 32) | lo[0]) + __longlong_as_double(((uint64_t)hi[1] << 32) | lo[1]);
}
// both of them, apart: the lower half's value first
template <int HALF>
__device__ __forceinline__ void both_halves(double v, double (&o)[2]) {
    const uint64_t b = __double_as_longlong(v);
    const v2u lo = swap_halves<HALF>((uint32_t)b), hi = swap_halves<HALF>((uint32_t)(b >> 32));
    o[0] = __longlong_as_double(((uint64_t)hi[0] << 32) | lo[0]);
    o[1] = __longlong_as_double(((uint64_t)hi[1] << 32) | lo[1]);
}
// LDS accesses of one wavefront made visible to its own lanes
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// sum over the lanes that agree in l mod 4
template <class T>
__device__ __forceinline__ T add_quads(T v) {
    v += dpp<kRor4>(v);
    v += dpp<kRor8>(v);
    v = add_halves<16>(v);
    return add_halves<32>(v);
}

// column of the group that lane l holds after wave_sum, and the lowest lane holding column c
template <int G>
__device__ __forceinline__ int col_of(int l) {
    return G == 4 ? ((l & 1) << 1) | ((l >> 1) & 1) : (G == 2 ? (l & 1) : 0);
}
template <int G>
constexpr int lane_of(int c) { return G == 4 ? ((c >> 1) & 1) | ((c & 1) << 1) : c; }

// per-lane values of G columns summed over quads: lane l returns column col_of(l).  The steps halve
// the columns (each lane keeps one half and sends the other).
template <int G, class T>
__device__ __forceinline__ T quad_sum(const T (&v)[G], int l) {
    T a;
    if constexpr (G == 4) {
        const bool hi = l & 1;
        const T k0 = hi ? v[2] : v[0], k1 = hi ? v[3] : v[1];
        const T s0 = hi ? v[0] : v[2], s1 = hi ? v[1] : v[3];
        const T a0 = k0 + dpp<kXor1>(s0), a1 = k1 + dpp<kXor1>(s1);
        const bool od = l & 2;
        const T k = od ? a1 : a0, s = od ? a0 : a1;
        a = k + dpp<kXor2>(s);
    } else if constexpr (G == 2) {
        const bool hi = l & 1;
        const T k = hi ? v[1] : v[0], s = hi ? v[0] : v[1];
        a = k + dpp<kXor1>(s);
        a += dpp<kXor2>(a);
    } else {
        a = v[0];
        a += dpp<kXor1>(a);
        a += dpp<kXor2>(a);
    }
    return a;
}
// the same over the wavefront
template <int G, class T>
__device__ __forceinline__ T wave_sum(const T (&v)[G], int l) {
    return add_quads(quad_sum<G>(v, l));
}
// FP32 values: 16 lanes in FP32, their sums in FP64
template <int G>
__device__ __forceinline__ double wave_sum_wide(const float (&v)[G], int l) {
    float a = quad_sum<G>(v, l);
    a += dpp<kRor4>(a);
    a += dpp<kRor8>(a);
    return add_halves<32>(add_halves<16>((double)a));
}

// the wavefronts' wave_sum results (red[wave][column]) summed in a fixed tree: every lane
// returns its column's total
template <int G>
__device__ __forceinline__ double across_waves(const double* red, int stride, int nw, int l) {
    const int w = l / G;                 // at most 16 wavefronts: lanes past them add 0
    double a = w < nw ? red[w * stride + col_of<G>(l)] : 0.0;
    if constexpr (G == 1) a += dpp<kXor1>(a);
    if constexpr (G <= 2) a += dpp<kXor2>(a);
    return add_quads(a);
}

__device__ __forceinline__ float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

template <int G> struct ChipVec;
template <> struct ChipVec<1> { typedef float type; };
template <> struct ChipVec<2> { typedef float2 type; };
template <> struct ChipVec<4> { typedef float4 type; };
template <int G>
__device__ __forceinline__ void unpack(const typename ChipVec<G>::type& v, float (&o)[G]) {
    if constexpr (G == 1) o[0] = v;
    else if constexpr (G == 2) { o[0] = v.x; o[1] = v.y; }
    else { o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w; }
}
template <int G>
__device__ __forceinline__ typename ChipVec<G>::type pack(const float (&v)[G]) {
    if constexpr (G == 1) return v[0];
    else if constexpr (G == 2) return make_float2(v[0], v[1]);
    else return make_float4(v[0], v[1], v[2], v[3]);
}

// Reference rule: the first column's group decides for its pair, and the others keep pace with it
// instead of running after it.  After step k the leader publishes 2 k, or 2 k + 1 where it stops;
// a follower ends step k only when it has seen that decision, so it never passes the leader's
// last step.  The wait is bounded (kLeadPolls: about 0.1 ms): a follower that gives up keeps its
// state and goes on in the next phase.  In place of leader first, followers after: forward solves of
// 817 nodes 1.02 -> 0.58 ms, of two complex frames of 1261 nodes 1.57 -> 0.88 ms.
__device__ __forceinline__ int lead_seen(const int* progress) {
    return __hip_atomic_load(progress, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void lead_tell(int* progress, int v) {
    __hip_atomic_store(progress, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// the leader's word on `step` (`seen`: an earlier look); -1: none in time
__device__ __forceinline__ int lead_word(const int* progress, int step, int seen, int polls) {
    for (int i = 0; (seen >> 1) < step; ++i) {
        if (i >= polls) return -1;
        __builtin_amdgcn_s_sleep(1);
        seen = lead_seen(progress);
    }
    return seen;
}

// f(0), ..., f(K - 1) with constant arguments: the per-row arrays are only ever indexed by
// constants, so that they are registers from the start (unrolled late they become vectors
// that every branch copies)
template <int K, class F, int... I>
__device__ __forceinline__ void each_row_of(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>()), ...);
}
template <int K, class F>
__device__ __forceinline__ void each_row(F&& f) {
    each_row_of<K>(f, std::make_integer_sequence<int, K>());
}

}  // namespace mpf
