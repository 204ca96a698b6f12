// Wave-level pieces shared by the diagonal-block kernels: lane broadcasts, compile-time loops and
// the 16 x 16 x 4 matrix instruction.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>

namespace elx {
namespace wv {

// v of lane `src` (uniform) for every lane
__device__ __forceinline__ float bcast_lane(float v, int src) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}
__device__ __forceinline__ double bcast_lane(double v, int src) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), src);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Entry J of the 16-lane row that a lane belongs to, in every lane of that row (all lanes on).
template <int J>
__device__ __forceinline__ double row_bcast(double v) {
    return __longlong_as_double(
        __builtin_amdgcn_update_dpp(0LL, (long long)__double_as_longlong(v), 0x150 + J, 0xF, 0xF, true));
}
template <int J>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + J, 0xF, 0xF, true));
}
// Orders LDS accesses between the lanes of one wave (their hardware order is program order; the
// compiler, which sees one lane at a time, must not move them past each other).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}
__device__ __forceinline__ bool finite(double v) { return fabs(v) <= 1.7976931348623157e308; }
__device__ __forceinline__ bool finite(float v) { return fabsf(v) <= 3.4028234663852886e38f; }

// The 16 x 16 x 4 matrix instruction: D(i, j) = fma over k = 0..3 ascending of a(i, k) b(k, j)
// onto C(i, j), one rounding each -- bit for bit the FMA chain. Lane l feeds a(l % 16, l / 16)
// and b(l / 16, l % 16); its register r holds D(row(l / 16, r), l % 16).
template <typename T>
struct Mfma4;
template <>
struct Mfma4<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    __device__ static acc run(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static int row(int kq, int r) { return kq + 4 * r; }
};
template <>
struct Mfma4<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    __device__ static acc run(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static int row(int kq, int r) { return 4 * kq + r; }
};

}  // namespace wv
}  // namespace elx
