// Sentinels of the sweeps' exchange buffers: signalling NaNs, which arithmetic
// never produces (results that are NaN come out quiet).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace m4g {

template <typename T> struct Sentinel;
template <> struct Sentinel<double> {
    static constexpr uint64_t bits = 0x7FF0DEADBEEF0001ull;
    __device__ static double value() { return __longlong_as_double((long long)bits); }
    __device__ static bool is(double v) { return (uint64_t)__double_as_longlong(v) == bits; }
    __device__ static double canon(double v) { return is(v) ? __longlong_as_double(0x7FF8000000000000ll) : v; }
};
template <> struct Sentinel<float> {
    static constexpr uint32_t bits = 0x7F80BEEFu;
    __device__ static float value() { return __int_as_float((int)bits); }
    __device__ static bool is(float v) { return (uint32_t)__float_as_int(v) == bits; }
    __device__ static float canon(float v) { return is(v) ? __int_as_float(0x7FC00000) : v; }
};

}  // namespace m4g
