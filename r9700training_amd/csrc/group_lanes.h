// group_lanes.h -- groups of an activation held across a wave's lanes, for the quantisers: a lane holds 8
// consecutive columns (one 16-byte load of bf16), a group of 2^lg columns (8 .. 512) spans 2^(lg-3)
// neighbouring lanes, and a wave covers 512 consecutive columns. The unnormalised Walsh-Hadamard
// transform's stages then run h = 1, 2, 4 inside a lane's registers and h = 8, 16, .. between
// lanes 1, 2, .. apart: data-parallel moves (DPP) inside a row of 16 lanes and the row swaps past it,
// no LDS traffic (an f64 __shfl_xor is two LDS permutes). The butterflies are the host rows'
// (src/adjoint/host/quant.cpp:181-191: sum in the lower, difference in the upper value, h
// ascending), so the transform is theirs bit for bit.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/r97q.h"
#include "iqr_device.h"

namespace r97q {
namespace lanes {

constexpr int kV = 8;                        // columns a lane
constexpr int kMinLog = 3, kMaxLog = 9;      // groups of 8 .. 512 columns
constexpr int kThreads = 256;

// the value of lane ^ H (H 1, 2, 4 or 8: inside a row of 16 lanes; every lane of the row active)
template <int H>
__device__ __forceinline__ uint32_t other(uint32_t x) {
    if constexpr (H == 1) return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, true);  // quad [1,0,3,2]
    if constexpr (H == 2) return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, true);  // quad [2,3,0,1]
    if constexpr (H == 4) {  // ^7 (half-row mirror), then ^3 (the quad reversed)
        const int m = __builtin_amdgcn_mov_dpp((int)x, 0x141, 0xF, 0xF, true);
        return (uint32_t)__builtin_amdgcn_mov_dpp(m, 0x1B, 0xF, 0xF, true);
    }
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x128, 0xF, 0xF, true);  // the row rotated by 8
}

// (lower, upper) of the pair of lanes H apart (16 or 32), in both of them
template <int H>
__device__ __forceinline__ void pair(double v, double& lo, double& hi) {
    static_assert(H == 16 || H == 32, "the row swaps");
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t x = (uint32_t)b, y = (uint32_t)(b >> 32);
    // the swap exchanges the odd 16-lane rows (H 16) or the upper half (H 32) of its first operand
    // with the even rows (the lower half) of its second: given x twice, the lower and the upper
    const auto sx = H == 16 ? __builtin_amdgcn_permlane16_swap(x, x, false, false)
                            : __builtin_amdgcn_permlane32_swap(x, x, false, false);
    const auto sy = H == 16 ? __builtin_amdgcn_permlane16_swap(y, y, false, false)
                            : __builtin_amdgcn_permlane32_swap(y, y, false, false);
    lo = __builtin_bit_cast(double, (uint64_t)sy[0] << 32 | sx[0]);
    hi = __builtin_bit_cast(double, (uint64_t)sy[1] << 32 | sx[1]);
}

// one stage between lanes H apart: lo + hi in the lower lane, lo - hi in the upper. For H < 16 the
// partner's value plus or minus the lane's own: o + v (the sum commutes) or o - v.
template <int H>
__device__ __forceinline__ void stage(double (&v)[kV], int lane) {
    const uint32_t flip = (lane & H) ? 0x80000000u : 0u;  // negates the subtrahend in the upper lane
    auto negated = [&](double d) {
        return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, d) ^ ((uint64_t)flip << 32));
    };
#pragma unroll
    for (int k = 0; k < kV; ++k) {
        if constexpr (H < 16) {
            const uint64_t b = __builtin_bit_cast(uint64_t, v[k]);
            const uint64_t o = (uint64_t)other<H>((uint32_t)(b >> 32)) << 32 | other<H>((uint32_t)b);
            v[k] = __builtin_bit_cast(double, o) + negated(v[k]);
        } else {
            double lo, hi;
            pair<H>(v[k], lo, hi);
            v[k] = lo + negated(hi);
        }
    }
}

// the transform of each group of 2^lg columns (lg uniform; every lane of the wave calls it)
__device__ __forceinline__ void fwht(double (&v)[kV], int lg, int lane) {
#pragma unroll
    for (int h = 1; h < kV; h <<= 1)
#pragma unroll
        for (int k = 0; k < kV; ++k)
            if (!(k & h)) {
                const double a = v[k], b = v[k + h];
                v[k] = a + b;
                v[k + h] = a - b;
            }
    if (lg > 3) stage<1>(v, lane);
    if (lg > 4) stage<2>(v, lane);
    if (lg > 5) stage<4>(v, lane);
    if (lg > 6) stage<8>(v, lane);
    if (lg > 7) stage<16>(v, lane);
    if (lg > 8) stage<32>(v, lane);
}

template <int H>
__device__ __forceinline__ double max_with(double m) {
    double lo, hi;
    if constexpr (H < 16) {
        const uint64_t b = __builtin_bit_cast(uint64_t, m);
        lo = m;
        hi = __builtin_bit_cast(double, (uint64_t)other<H>((uint32_t)(b >> 32)) << 32 | other<H>((uint32_t)b));
    } else {
        pair<H>(m, lo, hi);
    }
    return fmax(lo, hi);
}

// the largest |v| of each group (a NaN passed over, as the host's comparisons pass it over)
__device__ __forceinline__ double group_amax(const double (&v)[kV], int lg) {
    double m = 0.0;
#pragma unroll
    for (int k = 0; k < kV; ++k) m = fmax(m, fabs(v[k]));
    if (lg > 3) m = max_with<1>(m);
    if (lg > 4) m = max_with<2>(m);
    if (lg > 5) m = max_with<4>(m);
    if (lg > 6) m = max_with<8>(m);
    if (lg > 7) m = max_with<16>(m);
    if (lg > 8) m = max_with<32>(m);
    return m;
}

// a / s rounded to nearest, given inv = 1 / s rounded to nearest: one Newton correction of a * inv
// gives the correctly rounded quotient (Markstein's theorem; f32 operands widened to f64 stay far
// from f64's exponent limits), and the fixup puts the IEEE result where a or s is 0, inf or NaN
__device__ __forceinline__ double quotient(double a, double s, double inv) {
    const double q = a * inv;
    const double r = __builtin_fma(-q, s, a);
    return __builtin_amdgcn_div_fixup(__builtin_fma(r, inv, q), s, a);
}

// eight codes rint(v * inv) clamped to +-127 (ties to even; the conversion saturates, NaN gives 0),
// packed for one 8-byte store
__device__ __forceinline__ uint2 codes_of(const double (&v)[kV], double inv) {
    uint32_t i[kV];
#pragma unroll
    for (int k = 0; k < kV; ++k) {
        int32_t c;
        asm("v_cvt_i32_f64 %0, %1" : "=v"(c) : "v"(__builtin_rint(v[k] * inv)));
        i[k] = (uint32_t)(c > 127 ? 127 : c < -127 ? -127 : c);
    }
    // the low bytes of two, then of four: byte selectors 0..3 the second operand's, 4..7 the first's
    uint32_t w[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
        w[h] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(i[4 * h + 3], i[4 * h + 2], 0x0C0C0400u),
                                     __builtin_amdgcn_perm(i[4 * h + 1], i[4 * h], 0x0C0C0400u), 0x05040100u);
    return uint2{w[0], w[1]};
}

// eight values as bf16 (the hardware's round to nearest even), packed for one 16-byte store
__device__ __forceinline__ uint4 bf16_of(const double (&v)[kV]) {
    typedef __bf16 bf16x2 __attribute__((__vector_size__(4)));
    uint32_t w[kV / 2];
#pragma unroll
    for (int k = 0; k < kV / 2; ++k) {
        const bf16x2 b = {(__bf16)(float)v[2 * k], (__bf16)(float)v[2 * k + 1]};
        w[k] = __builtin_bit_cast(uint32_t, b);
    }
    return uint4{w[0], w[1], w[2], w[3]};
}

// eight consecutive bf16 or f32 values from 16-byte-aligned p
template <class T>
__device__ __forceinline__ void load8(const T* p, float (&x)[kV]) {
    if constexpr (sizeof(T) == 2) {
        const uint4 v = *reinterpret_cast<const uint4*>(p);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            x[2 * q] = __builtin_bit_cast(float, w[q] << 16);
            x[2 * q + 1] = __builtin_bit_cast(float, w[q] & 0xFFFF0000u);
        }
    } else {
        const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
        x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
        x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
    }
}
__device__ __forceinline__ void store8(float* p, const float (&x)[kV]) {
    *reinterpret_cast<float4*>(p) = float4{x[0], x[1], x[2], x[3]};
    *reinterpret_cast<float4*>(p + 4) = float4{x[4], x[5], x[6], x[7]};
}

// log2 of a group these kernels take, or -1
inline int group_log(int64_t group) {
    for (int lg = kMinLog; lg <= kMaxLog; ++lg)
        if (group == int64_t(1) << lg) return lg;
    return -1;
}
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace lanes
}  // namespace r97q
