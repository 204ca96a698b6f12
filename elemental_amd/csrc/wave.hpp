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

// x / d by the reciprocal r = 1 / d: x r and one correction with the exact remainder, then rounded
// as the division rounds it (compared with it on the quotients that lie closest to a rounding
// boundary, for every FP32 divisor). That holds where nothing leaves the exponent range on the way:
// divisor_ok(d) and dividend_ok(x). A zero x keeps the quotient's sign.
__device__ __forceinline__ double quot(double x, double d, double r) {
    const double q = x * r;
    return __builtin_copysign(__builtin_fma(__builtin_fma(-q, d, x), r, q), q);
}
__device__ __forceinline__ float quot(float x, float d, float r) {
    const float q = x * r;
    return __builtin_copysignf(__builtin_fmaf(__builtin_fmaf(-q, d, x), r, q), q);
}
__device__ __forceinline__ bool divisor_ok(double d) { return fabs(d) <= 0x1p400 && fabs(d) >= 0x1p-400; }
__device__ __forceinline__ bool divisor_ok(float d) { return fabsf(d) <= 0x1p60f && fabsf(d) >= 0x1p-60f; }
__device__ __forceinline__ bool dividend_ok(double x) {
    return x == 0.0 || (fabs(x) <= 0x1p600 && fabs(x) >= 0x1p-600);
}
__device__ __forceinline__ bool dividend_ok(float x) {
    return x == 0.0f || (fabsf(x) <= 0x1p64f && fabsf(x) >= 0x1p-64f);
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
