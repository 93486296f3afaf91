// fused_quant.hip -- the fused quantiser producers on the card: rmsnorm_had_quant_i8g,
// gated_had_quant_i8g and gate_had_quant_i8g (the reference's host rows
// src/adjoint/host/quant.cpp:896-1405 and device rows src/adjoint/device/quant.hip:959-961).
//
// Each applies an elementwise part to its inputs -- the RMS norm x * rs * (w + wadd) * mult, the
// gated activation silu(gate) * up over gate_up's two halves, or the gate sigmoid(a) * b
// (src/adjoint/host/elementwise.cpp:278-347, 459-641) -- then had_quant_act_i8g over the part's
// output: per group of `group` columns, the unnormalised Walsh-Hadamard transform, scale = amax / 127,
// codes = clamp(rint(v / scale), +-127). The adjoint is the parts' adjoints composed in the order
// the host row composes them: the codes' cotangent divided by the forward's scale, dropped where
// |v / scale| > 127, rotated back; the output write's cotangent added; then the part's adjoint.
//
// Two families. Groups of 8 .. 512 columns over aligned bf16 or f32 buffers are held across lanes, eight
// columns a lane (the second half of this file); every other call takes the general kernels:
//
// One workgroup a row, four waves; each wave takes whole groups. A lane holds max(1, group / 64)
// values of a group (element lane + 64 k), so a group of 64 or more is one wave and a smaller
// group shares a wave with its neighbours. The butterfly stages run in the host's order (h = 1, 2,
// 4, ...): the stages below 64 exchange with lane ^ h, the rest stay in a lane's registers. The
// part's output is formed in f64 from the inputs the way the host twin forms it, so the rotated
// values, the clamp decision and the codes are the host row's; the row's sums (the norm's sum of
// squares and its adjoint's shared term) run in a different order than the host's sequential loops,
// which moves them by an f64 ulp at most. This file is built with -ffp-contract=off so no FMA
// changes a rounding the host loop makes.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "../../include/r97q.h"
#include "group_lanes.h"
#include "iqr_device.h"
#include "status.h"

namespace r97q {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxLogGroup = 10;  // the reference's rows serve groups up to 1024 (quant.hip:129-137)

struct Args {
    const void* x0;
    const void* x1;
    int32_t dtype;
    int64_t n;
    double eps, wadd, mult;
    int8_t* codes;      // forward
    float* scale;       // forward: written; adjoint: the forward's
    uint16_t* y_out;    // forward, may be null
    const float* gc;    // adjoint: the codes' cotangent
    const float* gout;  // adjoint: the output write's cotangent, may be null
    float* dx0;
    float* dx1;
};

__device__ __forceinline__ double ld(const void* p, int32_t dt, int64_t i) {
    if (dt == R97Q_BF16) return (double)bf16_to_f32(static_cast<const uint16_t*>(p)[i]);
    if (dt == R97Q_F32) return (double)static_cast<const float*>(p)[i];
    return static_cast<const double*>(p)[i];
}

// src/adjoint/host/elementwise.cpp:121
__device__ __forceinline__ double sigm(double x) { return 1.0 / (1.0 + exp(-x)); }

template <int G>
struct Geo {
    static constexpr int V = G >= 64 ? G / 64 : 1;  // values a lane holds
    static constexpr int L = G >= 64 ? 64 : G;       // lanes a group spans
    static constexpr int E = 64 * V;                  // columns one wave step covers
};

// the unnormalised Walsh-Hadamard transform of each group (src/adjoint/host/quant.cpp:181-191)
template <int G>
__device__ __forceinline__ void fwht(double (&v)[Geo<G>::V], int lane) {
    constexpr int V = Geo<G>::V;
#pragma unroll
    for (int h = 1; h < G; h <<= 1) {
        if (h < 64) {
#pragma unroll
            for (int k = 0; k < V; ++k) {
                const double o = __shfl_xor(v[k], h);
                v[k] = (lane & h) ? o - v[k] : v[k] + o;
            }
        } else {
            const int hb = h / 64;
#pragma unroll
            for (int k = 0; k < V; ++k)
                if (!(k & hb)) {
                    const double a = v[k], b = v[k + hb];
                    v[k] = a + b;
                    v[k + hb] = a - b;
                }
        }
    }
}

// the four waves' partial sums, added in wave order; every thread gets the total
__device__ double block_sum(double s, double* red) {
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    double t = red[0];
    for (int w = 1; w < kWaves; ++w) t += red[w];
    __syncthreads();
    return t;
}

// the norm's 1 / sqrt(mean(x^2) + eps) of row r (src/adjoint/host/elementwise.cpp:526-529)
__device__ double row_rs(const Args& a, int64_t r, double* red) {
    double ss = 0.0;
    for (int64_t j = threadIdx.x; j < a.n; j += kThreads) {
        const double x = ld(a.x0, a.dtype, r * a.n + j);
        ss += x * x;
    }
    return 1.0 / sqrt(block_sum(ss, red) / (double)a.n + a.eps);
}

// the part's output at column j of row r (elementwise.cpp:284-289, 322-324, 530-537)
template <int PART>
__device__ __forceinline__ double part_y(const Args& a, int64_t r, int64_t j, double rs) {
    if constexpr (PART == R97Q_PART_RMSNORM) {
        return ld(a.x0, a.dtype, r * a.n + j) * rs * (ld(a.x1, a.dtype, j) + a.wadd) * a.mult;
    } else if constexpr (PART == R97Q_PART_SILU_MUL) {
        const int64_t b = r * 2 * a.n + j;
        const double g = ld(a.x0, a.dtype, b);
        return g * sigm(g) * ld(a.x0, a.dtype, b + a.n);
    } else {
        const int64_t b = r * a.n + j;
        return sigm(ld(a.x0, a.dtype, b)) * ld(a.x1, a.dtype, b);
    }
}

// grid (rows): codes, scale and (when asked) the part's output rounded to f32 then bf16
template <int PART, int G>
__global__ __launch_bounds__(kThreads) void fused_fwd_kernel(Args a) {
    using Gm = Geo<G>;
    __shared__ double red[kWaves];
    const int64_t r = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const double rs = PART == R97Q_PART_RMSNORM ? row_rs(a, r, red) : 0.0;
    const int64_t n = a.n, ngrp = n / G, steps = (n + Gm::E - 1) / Gm::E;
    for (int64_t st = wave; st < steps; st += kWaves) {
        const int64_t e0 = st * Gm::E + lane;
        const bool valid = e0 < n;  // groups are whole: a lane's values are all in or all out
        double v[Gm::V];
#pragma unroll
        for (int k = 0; k < Gm::V; ++k) {
            v[k] = valid ? part_y<PART>(a, r, e0 + 64 * k, rs) : 0.0;
            if (valid && a.y_out) a.y_out[r * n + e0 + 64 * k] = f32_to_bf16((float)v[k]);
        }
        fwht<G>(v, lane);
        double m = 0.0;
#pragma unroll
        for (int k = 0; k < Gm::V; ++k) m = fabs(v[k]) > m ? fabs(v[k]) : m;
#pragma unroll
        for (int o = 1; o < Gm::L; o <<= 1) {
            const double other = __shfl_xor(m, o);
            m = other > m ? other : m;
        }
        const double s = m > 0.0 ? m * (1.0 / 127.0) : 1.0;  // quant.cpp:222-224
        const double inv = 1.0 / s;
        if (valid) {
#pragma unroll
            for (int k = 0; k < Gm::V; ++k) {
                const double c = rint(v[k] * inv);
                a.codes[r * n + e0 + 64 * k] = (int8_t)(c > 127.0 ? 127.0 : c < -127.0 ? -127.0 : c);
            }
            if (lane % Gm::L == 0) a.scale[r * ngrp + e0 / G] = (float)s;
        }
    }
}

// grid (rows): dx0 (and dx1 for the gate) += the composed adjoint. The norm takes two passes over
// its row: the first forms the shared term t = sum r_j x_j c_j, the second writes dx with it.
template <int PART, int G>
__global__ __launch_bounds__(kThreads) void fused_bwd_kernel(Args a) {
    using Gm = Geo<G>;
    __shared__ double red[kWaves];
    const int64_t r = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t n = a.n, ngrp = n / G, steps = (n + Gm::E - 1) / Gm::E;
    const double rs = PART == R97Q_PART_RMSNORM ? row_rs(a, r, red) : 0.0;
    double t = 0.0;
    constexpr int passes = PART == R97Q_PART_RMSNORM ? 2 : 1;
    for (int pass = 0; pass < passes; ++pass) {
        double tp = 0.0;
        for (int64_t st = wave; st < steps; st += kWaves) {
            const int64_t e0 = st * Gm::E + lane;
            const bool valid = e0 < n;
            double v[Gm::V], d[Gm::V];
#pragma unroll
            for (int k = 0; k < Gm::V; ++k) v[k] = valid ? part_y<PART>(a, r, e0 + 64 * k, rs) : 0.0;
            fwht<G>(v, lane);
            // the straight-through rule at the forward's scale (quant.cpp:349-368)
#pragma unroll
            for (int k = 0; k < Gm::V; ++k) {
                const int64_t e = e0 + 64 * k;
                d[k] = 0.0;
                if (valid) {
                    const double s = (double)a.scale[r * ngrp + e / G];
                    d[k] = fabs(v[k] * (1.0 / s)) > 127.0 ? 0.0 : (double)a.gc[r * n + e] / s;
                }
            }
            fwht<G>(d, lane);
            if (!valid) continue;
#pragma unroll
            for (int k = 0; k < Gm::V; ++k) {
                const int64_t j = e0 + 64 * k;
                const double rr = a.gout ? d[k] + (double)a.gout[r * n + j] : d[k];
                if constexpr (PART == R97Q_PART_RMSNORM) {
                    // elementwise.cpp:628-640
                    const double x = ld(a.x0, a.dtype, r * n + j), c = ld(a.x1, a.dtype, j) + a.wadd;
                    if (pass == 0) {
                        tp += rr * x * c;
                    } else {
                        const double shared = rs * rs * rs * x * t / (double)n;
                        float* o = a.dx0 + r * n + j;
                        *o = (float)((double)*o + a.mult * (rs * c * rr - shared));
                    }
                } else if constexpr (PART == R97Q_PART_SILU_MUL) {
                    // elementwise.cpp:305-311
                    const int64_t b = r * 2 * n + j;
                    const double g = ld(a.x0, a.dtype, b), u = ld(a.x0, a.dtype, b + n), sg = sigm(g);
                    a.dx0[b] = (float)((double)a.dx0[b] + rr * u * (sg * (1.0 + g * (1.0 - sg))));
                    a.dx0[b + n] = (float)((double)a.dx0[b + n] + rr * (g * sigm(g)));
                } else {
                    // elementwise.cpp:342-345
                    const int64_t b = r * n + j;
                    const double x = ld(a.x0, a.dtype, b), bv = ld(a.x1, a.dtype, b), sx = sigm(x);
                    a.dx0[b] = (float)((double)a.dx0[b] + rr * (sx * (1.0 - sx)) * bv);
                    a.dx1[b] = (float)((double)a.dx1[b] + rr * sigm(x));
                }
            }
        }
        if (PART == R97Q_PART_RMSNORM && pass == 0) t = block_sum(tp, red);
    }
}

template <int PART, int LG>
void launch_part(bool bwd, int64_t rows, const Args& a, hipStream_t s) {
    if constexpr (LG > kMaxLogGroup) {
        return;
    } else {
        if (bwd)
            hipLaunchKernelGGL((fused_bwd_kernel<PART, 1 << LG>), dim3((unsigned)rows), dim3(kThreads), 0, s, a);
        else
            hipLaunchKernelGGL((fused_fwd_kernel<PART, 1 << LG>), dim3((unsigned)rows), dim3(kThreads), 0, s, a);
    }
}

template <int PART, int LG = 0>
void dispatch_group(int lg, bool bwd, int64_t rows, const Args& a, hipStream_t s) {
    if constexpr (LG <= kMaxLogGroup) {
        if (lg == LG) return launch_part<PART, LG>(bwd, rows, a, s);
        dispatch_group<PART, LG + 1>(lg, bwd, rows, a, s);
    }
}

// ---------------------------------------------------------------- groups of 8 .. 512 columns, bf16 and f32
// The same producers with the groups held across lanes (group_lanes.h): eight columns a lane, every
// buffer read and written in 16-byte accesses, each input read once. The f64 arithmetic is the host
// twins' as above (the sigmoid formed once a value; divisions by the scale through lanes::quotient,
// correctly rounded as the division is), so the gates' outputs are the kernels' above bit for bit.
struct LaneArgs {
    Args a;
    int lg;         // log2 of the group
    int64_t upr;    // 8-column units a row
    int64_t units;  // in all
};

template <class T>
__device__ __forceinline__ const T* in(const void* p) {
    return static_cast<const T*>(p);
}

// the unit's row and first column (32-bit when the units fit: the 64-bit division is ~5x the code)
__device__ __forceinline__ void unit_at(const LaneArgs& q, int64_t u, int64_t& r, int64_t& c) {
    if (q.units <= UINT32_MAX) {
        const uint32_t w = (uint32_t)u, d = (uint32_t)q.upr;
        r = w / d;
        c = (int64_t)(w - (uint32_t)r * d) * lanes::kV;
    } else {
        r = u / q.upr;
        c = (u - r * q.upr) * lanes::kV;
    }
}

// codes, scale and (when asked) the part's output of a unit at row r, column c, from the output v
__device__ __forceinline__ void put_codes(const LaneArgs& q, int64_t r, int64_t c, bool valid, double (&v)[lanes::kV],
                                          int lane) {
    const int64_t e = r * q.a.n + c;
    if (valid && q.a.y_out) *reinterpret_cast<uint4*>(q.a.y_out + e) = lanes::bf16_of(v);
    lanes::fwht(v, q.lg, lane);
    const double m = lanes::group_amax(v, q.lg);
    const double s = m > 0.0 ? m * (1.0 / 127.0) : 1.0;
    const uint2 codes = lanes::codes_of(v, 1.0 / s);
    if (!valid) return;
    *reinterpret_cast<uint2*>(q.a.codes + e) = codes;
    if ((c & ((int64_t(1) << q.lg) - 1)) == 0) q.a.scale[e >> q.lg] = (float)s;
}

// the part output's cotangent of a unit: the straight-through rule on the rotated output v at the
// forward's scale, rotated back, plus the output write's cotangent
__device__ __forceinline__ void out_cot(const LaneArgs& q, int64_t e, bool valid, double (&v)[lanes::kV], int lane,
                                        double (&rr)[lanes::kV]) {
    float g[lanes::kV] = {}, go[lanes::kV] = {}, sf = 1.0f;
    if (valid) {
        sf = q.a.scale[e >> q.lg];
        lanes::load8(q.a.gc + e, g);
        if (q.a.gout) lanes::load8(q.a.gout + e, go);
    }
    lanes::fwht(v, q.lg, lane);
    const double s = (double)sf, inv = 1.0 / s;
#pragma unroll
    for (int k = 0; k < lanes::kV; ++k) {
        const double d = lanes::quotient((double)g[k], s, inv);
        rr[k] = fabs(v[k] * inv) > 127.0 ? 0.0 : d;
    }
    lanes::fwht(rr, q.lg, lane);
    if (q.a.gout) {
#pragma unroll
        for (int k = 0; k < lanes::kV; ++k) rr[k] = rr[k] + (double)go[k];
    }
}

// the sigmoid: the reciprocal of d = 1 + exp(-x) >= 1, which needs none of a division's scaling. Two Newton
// steps and a last correction from the remainder round it to nearest, as the division does; the fixup
// puts 0 for an infinite d and passes a NaN. (With the compiler's
// division, bf16 rounding in integer code and the clamp in f64 the gates' forward took 294 us, not 253.)
__device__ __forceinline__ double sigm_lane(double x) {
    const double d = 1.0 + exp(-x);
    double r = __builtin_amdgcn_rcp(d);
#pragma unroll
    for (int i = 0; i < 3; ++i) r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    return __builtin_amdgcn_div_fixup(r, d, 1.0);
}

// The gates, flat over the units. Bound by memory in the adjoint and by the f64 instructions (the
// exponential, the division, the butterflies) in the forward. Measured at 4096 x 17408 bf16, silu_mul,
// group 128, with y and its cotangent: forward 222 us (2.3 TB/s) and adjoint 368 us (5.4 TB/s), against
// 338 and 1074 us for one column a lane and LDS permutes.
template <int PART, class T>
__global__ __launch_bounds__(lanes::kThreads) void lane_fwd_kernel(const LaneArgs q) {
    const int64_t u = (int64_t)blockIdx.x * lanes::kThreads + threadIdx.x;
    const bool valid = u < q.units;
    int64_t r, c;
    unit_at(q, valid ? u : 0, r, c);
    const int64_t n = q.a.n, e = r * n + c;
    float x[lanes::kV] = {}, y[lanes::kV] = {};
    if (valid) {
        lanes::load8(in<T>(q.a.x0) + (PART == R97Q_PART_SILU_MUL ? e + r * n : e), x);
        lanes::load8(PART == R97Q_PART_SILU_MUL ? in<T>(q.a.x0) + e + r * n + n : in<T>(q.a.x1) + e, y);
    }
    double v[lanes::kV];
#pragma unroll
    for (int k = 0; k < lanes::kV; ++k) {
        const double g = (double)x[k], o = (double)y[k];
        v[k] = PART == R97Q_PART_SILU_MUL ? g * sigm_lane(g) * o : sigm_lane(g) * o;
    }
    put_codes(q, r, c, valid, v, threadIdx.x & 63);
}

template <int PART, class T>
__global__ __launch_bounds__(lanes::kThreads) void lane_bwd_kernel(const LaneArgs q) {
    const int64_t u = (int64_t)blockIdx.x * lanes::kThreads + threadIdx.x;
    const bool valid = u < q.units;
    int64_t r, c;
    unit_at(q, valid ? u : 0, r, c);
    const int64_t n = q.a.n, e = r * n + c;
    constexpr bool kSilu = PART == R97Q_PART_SILU_MUL;
    const int64_t b = kSilu ? e + r * n : e;
    float x[lanes::kV] = {}, y[lanes::kV] = {};
    if (valid) {
        lanes::load8(in<T>(q.a.x0) + b, x);
        lanes::load8(kSilu ? in<T>(q.a.x0) + b + n : in<T>(q.a.x1) + e, y);
    }
    double sg[lanes::kV], v[lanes::kV], rr[lanes::kV];
#pragma unroll
    for (int k = 0; k < lanes::kV; ++k) {
        const double g = (double)x[k];
        sg[k] = sigm_lane(g);
        v[k] = kSilu ? g * sg[k] * (double)y[k] : sg[k] * (double)y[k];
    }
    out_cot(q, e, valid, v, threadIdx.x & 63, rr);
    if (!valid) return;
    float* d0 = q.a.dx0 + b;
    float* d1 = kSilu ? q.a.dx0 + b + n : q.a.dx1 + e;
    float o0[lanes::kV], o1[lanes::kV];
    lanes::load8(d0, o0);
    lanes::load8(d1, o1);
#pragma unroll
    for (int k = 0; k < lanes::kV; ++k) {
        const double g = (double)x[k], w = (double)y[k], s = sg[k];
        if constexpr (kSilu) {  // elementwise.cpp:305-311
            o0[k] = (float)((double)o0[k] + rr[k] * w * (s * (1.0 + g * (1.0 - s))));
            o1[k] = (float)((double)o1[k] + rr[k] * (g * s));
        } else {  // elementwise.cpp:342-345
            o0[k] = (float)((double)o0[k] + rr[k] * (s * (1.0 - s)) * w);
            o1[k] = (float)((double)o1[k] + rr[k] * s);
        }
    }
    lanes::store8(d0, o0);
    lanes::store8(d1, o1);
}

// The norm: a workgroup a row, as many threads as the row has units up to 1024, IT units a thread,
// the row held from its one read to the last use -- in registers, but for the adjoint past 8192 columns,
// which spills (17 registers a lane at IT 2, 78 at IT 3). Measured with group 128 (y and its cotangent
// written and read), against four waves walking the row three times: 64 x 5120 f32 forward 6.0 us and
// adjoint 7.8, against 21 and 58; 64 x 12288 8.2 and 15, against 48 and 133; 64 x 17408 10 and 31, against 67
// and 186; 2048 x 17408 bf16 83 and 378, against 177 and 961.
constexpr int kNormMaxIt = 3;

__device__ double row_sum(double s, double* red) {
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    double t = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) t += red[w];
    __syncthreads();
    return t;
}

template <class T, int IT, bool BWD>
__global__ __launch_bounds__(1024) void lane_norm_kernel(const LaneArgs q) {
    __shared__ double red[16];
    const int lane = threadIdx.x & 63;
    const int64_t r = blockIdx.x, n = q.a.n;
    float x[IT][lanes::kV], w[IT][lanes::kV];
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int64_t u = (int64_t)i * blockDim.x + threadIdx.x;
#pragma unroll
        for (int k = 0; k < lanes::kV; ++k) x[i][k] = w[i][k] = 0.0f;
        if (u < q.upr) {
            lanes::load8(in<T>(q.a.x0) + r * n + u * lanes::kV, x[i]);
            lanes::load8(in<T>(q.a.x1) + u * lanes::kV, w[i]);
        }
#pragma unroll
        for (int k = 0; k < lanes::kV; ++k) ss += (double)x[i][k] * (double)x[i][k];
    }
    const double rs = 1.0 / sqrt(row_sum(ss, red) / (double)n + q.a.eps);
    double rr[IT][lanes::kV], tp = 0.0;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int64_t u = (int64_t)i * blockDim.x + threadIdx.x;
        const bool valid = u < q.upr;
        double v[lanes::kV];
#pragma unroll
        for (int k = 0; k < lanes::kV; ++k)
            v[k] = valid ? (double)x[i][k] * rs * ((double)w[i][k] + q.a.wadd) * q.a.mult : 0.0;
        if constexpr (!BWD) {
            put_codes(q, r, u * lanes::kV, valid, v, lane);
        } else {
            out_cot(q, r * n + u * lanes::kV, valid, v, lane, rr[i]);
            if (valid) {
#pragma unroll
                for (int k = 0; k < lanes::kV; ++k) tp += rr[i][k] * (double)x[i][k] * ((double)w[i][k] + q.a.wadd);
            }
        }
    }
    if constexpr (BWD) {
        // elementwise.cpp:628-640
        const double t = row_sum(tp, red), nd = (double)n, ninv = 1.0 / nd;
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int64_t u = (int64_t)i * blockDim.x + threadIdx.x;
            if (u >= q.upr) continue;
            float* d = q.a.dx0 + r * n + u * lanes::kV;
            float o[lanes::kV];
            lanes::load8(d, o);
#pragma unroll
            for (int k = 0; k < lanes::kV; ++k) {
                const double c = (double)w[i][k] + q.a.wadd;
                const double shared = lanes::quotient(rs * rs * rs * (double)x[i][k] * t, nd, ninv);
                o[k] = (float)((double)o[k] + q.a.mult * (rs * c * rr[i][k] - shared));
            }
            lanes::store8(d, o);
        }
    }
}

template <class T, bool BWD>
void launch_norm(const LaneArgs& q, int64_t rows, hipStream_t s) {
    const int it = (int)((q.upr + 1023) / 1024);
    const int threads = (int)(((q.upr + it - 1) / it + 63) / 64 * 64);
    const dim3 grid((unsigned)rows), block((unsigned)threads);
    if (it == 1) hipLaunchKernelGGL((lane_norm_kernel<T, 1, BWD>), grid, block, 0, s, q);
    else if (it == 2) hipLaunchKernelGGL((lane_norm_kernel<T, 2, BWD>), grid, block, 0, s, q);
    else hipLaunchKernelGGL((lane_norm_kernel<T, 3, BWD>), grid, block, 0, s, q);
}

template <class T>
void launch_lanes(int32_t part, bool bwd, int64_t rows, const LaneArgs& q, hipStream_t s) {
    if (part == R97Q_PART_RMSNORM) return bwd ? launch_norm<T, true>(q, rows, s) : launch_norm<T, false>(q, rows, s);
    const dim3 grid((unsigned)((q.units + lanes::kThreads - 1) / lanes::kThreads)), block(lanes::kThreads);
    if (part == R97Q_PART_SILU_MUL) {
        if (bwd) hipLaunchKernelGGL((lane_bwd_kernel<R97Q_PART_SILU_MUL, T>), grid, block, 0, s, q);
        else hipLaunchKernelGGL((lane_fwd_kernel<R97Q_PART_SILU_MUL, T>), grid, block, 0, s, q);
    } else {
        if (bwd) hipLaunchKernelGGL((lane_bwd_kernel<R97Q_PART_SIGMOID_MUL, T>), grid, block, 0, s, q);
        else hipLaunchKernelGGL((lane_fwd_kernel<R97Q_PART_SIGMOID_MUL, T>), grid, block, 0, s, q);
    }
}

// Whether a call goes across lanes: groups of 8 .. 512 columns over bf16 or f32 inputs, every buffer on
// 16 bytes (the codes on 8), a norm's row of at most kNormMaxIt x 1024 units. The other groups, f64
// inputs (the rows' host operands), wider norms, overlapping gradients and unaligned views take the
// kernels above.
bool takes_lanes(int32_t part, const Args& a, int lg, int64_t rows) {
    if (lg < lanes::kMinLog || lg > lanes::kMaxLog || a.dtype == R97Q_F64) return false;
    if (part == R97Q_PART_RMSNORM && a.n > (int64_t)kNormMaxIt * 1024 * lanes::kV) return false;
    if (part != R97Q_PART_RMSNORM && rows * (a.n / lanes::kV) / lanes::kThreads >= INT32_MAX) return false;
    // the gate's two gradients added into overlapping buffers: one at a time, as the kernel above does
    const uintptr_t d0 = (uintptr_t)a.dx0, d1 = (uintptr_t)a.dx1, bytes = (uintptr_t)(rows * a.n) * 4;
    if (part == R97Q_PART_SIGMOID_MUL && a.dx0 && d0 < d1 + bytes && d1 < d0 + bytes) return false;
    const void* p[] = {a.x0, a.x1, a.y_out, a.gc, a.gout, a.dx0, a.dx1};
    for (const void* b : p)
        if (!lanes::aligned16(b)) return false;
    return (reinterpret_cast<uintptr_t>(a.codes) & 7) == 0;
}

const char* part_name(int32_t part) {
    return part == R97Q_PART_RMSNORM ? "rmsnorm_had_quant_i8g"
           : part == R97Q_PART_SILU_MUL ? "gated_had_quant_i8g"
                                        : "gate_had_quant_i8g";
}

// the record rules the reference's rows apply (quant.hip:129-159, the group; elementwise.cpp, the
// parts' operands): 0 and log2(group) in *lg, or an error code with the message set
int check_args(int32_t part, const void* x0, const void* x1, int32_t dtype, int64_t rows, int64_t n, int64_t group,
               const char* who, int* lg) {
    if (part < R97Q_PART_RMSNORM || part > R97Q_PART_SIGMOID_MUL) {
        set_error("fused quantiser: part %d is not rmsnorm (0), silu_mul (1) or sigmoid_mul (2)", (int)part);
        return R97Q_EINVAL;
    }
    if (!x0 || (part != R97Q_PART_SILU_MUL && !x1)) {
        set_error("%s: null %s", who, !x0 ? "first input" : part == R97Q_PART_RMSNORM ? "gain" : "second input");
        return R97Q_EINVAL;
    }
    if (dtype != R97Q_BF16 && dtype != R97Q_F32 && dtype != R97Q_F64) {
        set_error("%s: the inputs are bf16, f32 or f64", who);
        return R97Q_EINVAL;
    }
    if (rows <= 0 || n <= 0) {
        set_error("%s: rows and n must be positive", who);
        return R97Q_EINVAL;
    }
    if (group <= 0 || (group & (group - 1)) != 0 || n % group != 0) {
        set_error("%s: 'group' must be a power of two that divides 'n' (n=%lld group=%lld)", who, (long long)n,
                  (long long)group);
        return R97Q_EINVAL;
    }
    if (group > (1 << kMaxLogGroup)) {
        set_error("%s: a group of %lld is wider than the rows serve (%d)", who, (long long)group, 1 << kMaxLogGroup);
        return R97Q_EUNSUPPORTED;
    }
    if (rows > 0x7fffffffLL) {
        set_error("%s: %lld rows; at most 2^31 - 1 a call", who, (long long)rows);
        return R97Q_EUNSUPPORTED;
    }
    *lg = 0;
    while ((1LL << *lg) < group) ++*lg;
    return R97Q_OK;
}

void launch(int32_t part, int lg, bool bwd, int64_t rows, const Args& a, hipStream_t s) {
    if (takes_lanes(part, a, lg, rows)) {
        const int64_t upr = a.n / lanes::kV;
        const LaneArgs q{a, lg, upr, rows * upr};
        return a.dtype == R97Q_BF16 ? launch_lanes<uint16_t>(part, bwd, rows, q, s) : launch_lanes<float>(part, bwd, rows, q, s);
    }
    if (part == R97Q_PART_RMSNORM) dispatch_group<R97Q_PART_RMSNORM>(lg, bwd, rows, a, s);
    else if (part == R97Q_PART_SILU_MUL) dispatch_group<R97Q_PART_SILU_MUL>(lg, bwd, rows, a, s);
    else dispatch_group<R97Q_PART_SIGMOID_MUL>(lg, bwd, rows, a, s);
}

}  // namespace
}  // namespace r97q

using namespace r97q;

extern "C" {

int r97q_fused_had_quant_i8g(int32_t part, const void* x0, const void* x1, int32_t x_dtype, int64_t rows, int64_t n,
                             int64_t group, double eps, double wadd, double mult, int8_t* codes, float* scale,
                             uint16_t* y_out, R97IqrStream stream) {
    clear_error();
    int lg = 0;
    const char* who = part_name(part);
    if (int e = check_args(part, x0, x1, x_dtype, rows, n, group, who, &lg)) return e;
    if (!codes || !scale) {
        set_error("%s: null codes or scale", who);
        return R97Q_EINVAL;
    }
    Args a{x0, x1, x_dtype, n, eps, wadd, mult, codes, scale, y_out, nullptr, nullptr, nullptr, nullptr};
    launch(part, lg, false, rows, a, (hipStream_t)stream);
    return launch_status("fused_fwd_kernel");
}

int r97q_fused_had_quant_i8g_bwd(int32_t part, const void* x0, const void* x1, int32_t x_dtype, int64_t rows,
                                 int64_t n, int64_t group, double eps, double wadd, double mult, const float* scale,
                                 const float* g_codes, const float* g_out, float* dx0, float* dx1,
                                 R97IqrStream stream) {
    clear_error();
    int lg = 0;
    const char* who = part_name(part);
    if (int e = check_args(part, x0, x1, x_dtype, rows, n, group, who, &lg)) return e;
    if (!scale || !g_codes || !dx0 || (part == R97Q_PART_SIGMOID_MUL && !dx1)) {
        set_error("%s adjoint: null scale, codes' cotangent or %s", who, !dx0 ? "dx0" : "dx1");
        return R97Q_EINVAL;
    }
    Args a{x0, x1, x_dtype, n, eps, wadd, mult, nullptr, const_cast<float*>(scale), nullptr, g_codes, g_out, dx0,
           dx1};
    launch(part, lg, true, rows, a, (hipStream_t)stream);
    return launch_status("fused_bwd_kernel");
}

}  // extern "C"
