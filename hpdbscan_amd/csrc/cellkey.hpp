// The cell key of a row: the reference's linearised cell id
// (spatial_index.h:144-165) offset by the job's key base, followed by the
// row's sub-box digit, and the grid it lies in.  Shared by the kernel that keys
// the rows for the sort and the one that labels rows in input order, which must
// find the very key the sort used, and by the kernels of small inputs.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <limits>
#include <type_traits>

#include "internal.hpp"

namespace hpd {

// floor((x - min) / eps) as the reference build computes it
// (spatial_index.h:156): (x - min) * rcp with rcp = 1/eps rounded once, in
// float for float and integer data, in double for double data.
template <typename T>
__device__ __forceinline__ uint64_t cell_index(T x, T mn, float rcp_f, double rcp_d);

template <>
__device__ __forceinline__ uint64_t cell_index<float>(float x, float mn, float rcp_f, double) {
    const float v = (x - mn) * rcp_f;
    return static_cast<uint64_t>(floorf(v));
}
template <>
__device__ __forceinline__ uint64_t cell_index<double>(double x, double mn, float, double rcp_d) {
    const double v = (x - mn) * rcp_d;
    return static_cast<uint64_t>(floor(v));
}

// (x - min) is evaluated in T's promoted type and converted to float
template <typename T>
__device__ __forceinline__ float int_diff_f32(T x, T mn) {
    using P = decltype(x - mn);
    if constexpr (sizeof(T) < sizeof(int)) {
        return static_cast<float>(static_cast<int>(x) - static_cast<int>(mn));
    } else {
        using U = std::make_unsigned_t<P>;
        return static_cast<float>(static_cast<P>(static_cast<U>(x) - static_cast<U>(mn)));
    }
}

#define HPD_INT_CELL_INDEX(T)                                                             \
    template <>                                                                           \
    __device__ __forceinline__ uint64_t cell_index<T>(T x, T mn, float rcp_f, double) {   \
        const float v = int_diff_f32<T>(x, mn) * rcp_f;                                   \
        return static_cast<uint64_t>(floorf(v));                                          \
    }
HPD_INT_CELL_INDEX(int8_t)
HPD_INT_CELL_INDEX(int16_t)
HPD_INT_CELL_INDEX(int32_t)
HPD_INT_CELL_INDEX(int64_t)
HPD_INT_CELL_INDEX(uint8_t)
HPD_INT_CELL_INDEX(uint16_t)
HPD_INT_CELL_INDEX(uint32_t)
HPD_INT_CELL_INDEX(uint64_t)
#undef HPD_INT_CELL_INDEX

// (x - min) * (1/eps) as the cell index computes it (float product for
// float data, double for double), returned exactly as a double
template <typename T>
__device__ __forceinline__ double scaled_value(T x, T mn, float rcp_f, double rcp_d);
template <>
__device__ __forceinline__ double scaled_value<float>(float x, float mn, float rcp_f, double) {
    return static_cast<double>((x - mn) * rcp_f);
}
template <>
__device__ __forceinline__ double scaled_value<double>(double x, double mn, float, double rcp_d) {
    return (x - mn) * rcp_d;
}
template <typename T>
__device__ __forceinline__ double scaled_value(T, T, float, double) {
    return 0.0;  // integer data has no sub-boxes
}

// key = (key_base + cell id) << sub_bits | sub-box digit, where the digit is
// the box of the cell's sub_k^D split along the same scaled coordinate
// v = (x - min) * (1/eps) that the cell index floors (v held exactly in
// double): sub_j = clamp(floor(v_j sub_k) - sub_k floor(v_j), 0, sub_k - 1)
template <typename T, int D>
__device__ __forceinline__ uint64_t row_key(const T* __restrict__ p, const JobParams<T>& jp,
                                            int sub_k, int sub_bits) {
    T row[D];
#pragma unroll
    for (int j = 0; j < D; ++j) row[j] = p[j];
    uint64_t cell = 0;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        const int j = jp.cp.swapped[k];
        T xj = row[0];
        T mj = jp.minv[0];
#pragma unroll
        for (int t = 1; t < D; ++t)
            if (t == j) {
                xj = row[t];
                mj = jp.minv[t];
            }
        cell += cell_index<T>(xj, mj, jp.rcp_f, jp.rcp_d) * jp.cp.stride[k];
    }
    uint64_t sub = 0, mul = 1;
    if (sub_bits > 0) {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            const double v = scaled_value<T>(row[j], jp.minv[j], jp.rcp_f, jp.rcp_d);
            const double c = floor(v);
            long long sd = static_cast<long long>(floor(v * sub_k)) - static_cast<long long>(c) * sub_k;
            sd = sd < 0 ? 0 : (sd >= sub_k ? sub_k - 1 : sd);
            sub += static_cast<uint64_t>(sd) * mul;
            mul *= static_cast<uint64_t>(sub_k);
        }
    }
    return ((jp.key_base + cell) << sub_bits) | sub;
}

// The reference starts max at numeric_limits<T>::min(): FLT_MIN / DBL_MIN for
// floating types (the smallest positive normal), the lowest value for
// integers.
template <typename T>
__device__ __forceinline__ T max_init() {
    return std::numeric_limits<T>::min();
}
template <typename T>
__device__ __forceinline__ T min_init() {
    return std::numeric_limits<T>::max();
}

// std::min(m, c) == (c < m) ? c : m ; std::max(m, c) == (m < c) ? c : m
template <typename T>
__device__ __forceinline__ T ref_min(T m, T c) {
    return (c < m) ? c : m;
}
template <typename T>
__device__ __forceinline__ T ref_max(T m, T c) {
    return (m < c) ? c : m;
}

// float / double -> integer as x86-64 cvttss2si / cvttsd2si produce it
// (out of range or NaN: the "integer indefinite" value)
__device__ __forceinline__ int64_t d2i64_x86(double v) {
    if (!(v >= -9223372036854775808.0 && v < 9223372036854775808.0)) return INT64_MIN;
    return static_cast<int64_t>(v);
}
__device__ __forceinline__ uint64_t d2u64_x86(double v) {
    if (v < 9223372036854775808.0) return static_cast<uint64_t>(d2i64_x86(v));
    return static_cast<uint64_t>(d2i64_x86(v - 9223372036854775808.0)) ^ 0x8000000000000000ull;
}

// cells of one dimension, ceil((max - min) / eps) + 1 (spatial_index.h:124-131)
// with the reciprocal form and the flushing of the reference's build (device
// code flushes denormal inputs and results itself)
template <typename T>
__device__ __forceinline__ uint64_t cells_of_dev(T mx, T mn, float rcp_f, double rcp_d) {
    if constexpr (std::is_same<T, float>::value) {
        const float v = (mx - mn) * rcp_f;
        return d2u64_x86(static_cast<double>(ceilf(v))) + 1;
    } else if constexpr (std::is_same<T, double>::value) {
        const double v = (mx - mn) * rcp_d;
        return d2u64_x86(ceil(v)) + 1;
    } else {
        const float v = int_diff_f32<T>(mx, mn) * rcp_f;
        return d2u64_x86(static_cast<double>(ceilf(v))) + 1;
    }
}

// The grid of one job from its min / max (mm: D minima, D maxima), into jp
// (whose reciprocals the host wrote): cells per dimension, dimension order (an
// insertion sort ascending by cells, which is what std::sort does for so few
// keys: ties keep their order), strides, minima.  Returns the number of
// cells; overflow becomes true when they exceed 2^64.
template <typename T, int D>
__device__ __forceinline__ uint64_t make_grid(const T* mm, JobParams<T>& jp, bool& overflow) {
    uint64_t c[D];
    uint64_t tot = 1;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        c[k] = cells_of_dev<T>(mm[D + k], mm[k], jp.rcp_f, jp.rcp_d);
        uint64_t t;
        if (__builtin_mul_overflow(tot, c[k], &t)) overflow = true;
        tot = t;
    }
    int sw[D];
#pragma unroll
    for (int k = 0; k < D; ++k) sw[k] = k;
    for (int k = 1; k < D; ++k) {
        const int v = sw[k];
        int i = k - 1;
        while (i >= 0 && c[v] < c[sw[i]]) {
            sw[i + 1] = sw[i];
            --i;
        }
        sw[i + 1] = v;
    }
    uint64_t acc = 1;
    jp.cp.d = D;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        jp.minv[k] = mm[k];
        jp.cp.swapped[k] = sw[k];
        jp.cp.stride[k] = acc;
        jp.cp.ncell[k] = c[sw[k]];
        acc *= c[sw[k]];
    }
    return tot;
}

}  // namespace hpd
