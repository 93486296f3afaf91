// sm_finish.hip -- the second launch of the few-token path (qlinear_sm.h): the products' partials added
// in range order with the adapter's up-projection, the down product's sum t, and the factor gradients,
// each a kind of workgroup of one launch.
//
//   Y[m][n]  = sum_z part[z][m][n] + sum_j u[m][j] B[n][j]      u = s . sum_z tpart[z]   (forward)
//   dX[m][k] (+)= sum_z part[z][m][k] + sum_j u[m][j] A[j][k]   u = dt                   (backward)
//   dA[j][k] += sum_m u[m][j] X[m][k]      dB[n][j] += sum_m s t[m][j] dY[m][n]
//
// The adapter's sums run over the exact f32 u and t (the larger calls' bf16 MFMAs take them as two
// halves): the up-projection in f32 FMAs, a few microseconds of the chip's vector rate at the token counts
// of this path, less than staging it for MFMAs would need; the factor gradients on the f32 MFMAs
// (grad_item). All sums run in an order that the shape alone fixes.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "iqr_device.h"
#include "qlinear_sm.h"
#include "status.h"

namespace r97q {
namespace sm {
namespace {

constexpr int kThreads = 512;
constexpr int kRows = 32;       // token rows of an output workgroup
constexpr int kCols = 128;      // its columns: four a thread, two rows
constexpr int kGradCols = 32;   // columns of a gradient workgroup
constexpr int kCopy = 32 * kThreads;  // values of a copy workgroup

__device__ __forceinline__ float4 add4(float4 a, float4 b) { return {a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w}; }

// sum over z < SU of U[z][i], the ranges in order, four loads in flight
__device__ __forceinline__ float sum_ranges(const float* U, int SU, int64_t n, int64_t i) {
    if (SU == 1) return U[i];
    float v = 0.0f;
    int z = 0;
    for (; z + 4 <= SU; z += 4) {
        float x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = U[(int64_t)(z + q) * n + i];
#pragma unroll
        for (int q = 0; q < 4; ++q) v += x[q];
    }
    for (; z < SU; ++z) v += U[(int64_t)z * n + i];
    return v;
}

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xFFFF0000u); }

// rows m0 .. m0+31, columns c0 .. c0+127 of the output
__device__ __forceinline__ void output_item(const Finish& f, float* u, int64_t m0, int64_t c0) {
    const int tid = threadIdx.x, r = f.rank;
    for (int i = tid; i < kRows * r; i += kThreads) {
        const int64_t m = m0 + i / r;
        u[i] = m < f.T ? f.scale * sum_ranges(f.U, f.SU, f.T * r, m0 * r + i) : 0.0f;
    }
    __syncthreads();
    const int64_t c = c0 + 4 * (tid & 31);
    const int rl = 2 * (tid >> 5);
    float4 v[2] = {};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int64_t m = m0 + rl + h;
        if (m >= f.T) continue;
        const float* src = f.part + m * f.outs + c;
        const int64_t ld = f.T * f.outs;
        int z = 0;
        for (; z + 4 <= f.S; z += 4) {
            float4 x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = *reinterpret_cast<const float4*>(src + (z + q) * ld);
#pragma unroll
            for (int q = 0; q < 4; ++q) v[h] = add4(v[h], x[q]);
        }
        for (; z < f.S; ++z) v[h] = add4(v[h], *reinterpret_cast<const float4*>(src + z * ld));
    }
    if (m0 + rl >= f.T) return;
    const float* ul = u + rl * r;
    if (r > 0 && f.fwd) {
        for (int j = 0; j < r; j += 8) {
            uint4 b[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) b[q] = *reinterpret_cast<const uint4*>(f.F + (c + q) * r + j);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float4 ua = *reinterpret_cast<const float4*>(ul + h * r + j);
                const float4 ub = *reinterpret_cast<const float4*>(ul + h * r + j + 4);
                float* y = &v[h].x;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float a = y[q];
                    a = __builtin_fmaf(ua.x, bf16_lo(b[q].x), a);
                    a = __builtin_fmaf(ua.y, bf16_hi(b[q].x), a);
                    a = __builtin_fmaf(ua.z, bf16_lo(b[q].y), a);
                    a = __builtin_fmaf(ua.w, bf16_hi(b[q].y), a);
                    a = __builtin_fmaf(ub.x, bf16_lo(b[q].z), a);
                    a = __builtin_fmaf(ub.y, bf16_hi(b[q].z), a);
                    a = __builtin_fmaf(ub.z, bf16_lo(b[q].w), a);
                    y[q] = __builtin_fmaf(ub.w, bf16_hi(b[q].w), a);
                }
            }
        }
    } else if (r > 0) {
        for (int j = 0; j < r; j += 8) {
            uint2 a[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const uint16_t* p = f.F + (int64_t)(j + q) * f.outs + c;
                a[q] = f.fvec ? *reinterpret_cast<const uint2*>(p)
                              : uint2{(uint32_t)p[0] | (uint32_t)p[1] << 16, (uint32_t)p[2] | (uint32_t)p[3] << 16};
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const float w = ul[h * r + j + q];
                    v[h].x = __builtin_fmaf(w, bf16_lo(a[q].x), v[h].x);
                    v[h].y = __builtin_fmaf(w, bf16_hi(a[q].x), v[h].y);
                    v[h].z = __builtin_fmaf(w, bf16_lo(a[q].y), v[h].z);
                    v[h].w = __builtin_fmaf(w, bf16_hi(a[q].y), v[h].w);
                }
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int64_t m = m0 + rl + h;
        if (m >= f.T) continue;
        const int64_t at = m * f.outs + c;
        float* y = &v[h].x;
        if (f.out_f32) {
            float* o = static_cast<float*>(f.out) + at;
            if (f.vec) {
                if (f.accumulate) v[h] = add4(v[h], *reinterpret_cast<const float4*>(o));
                *reinterpret_cast<float4*>(o) = v[h];
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) o[q] = f.accumulate ? y[q] + o[q] : y[q];
            }
        } else {
            uint16_t* o = static_cast<uint16_t*>(f.out) + at;
            if (f.vec) {
                if (f.accumulate) {
                    const uint2 d = *reinterpret_cast<const uint2*>(o);
                    v[h] = add4(v[h], float4{bf16_lo(d.x), bf16_hi(d.x), bf16_lo(d.y), bf16_hi(d.y)});
                }
                *reinterpret_cast<uint2*>(o) =
                    uint2{(uint32_t)f32_to_bf16(y[0]) | (uint32_t)f32_to_bf16(y[1]) << 16,
                          (uint32_t)f32_to_bf16(y[2]) | (uint32_t)f32_to_bf16(y[3]) << 16};
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) o[q] = f32_to_bf16(f.accumulate ? y[q] + bf16_to_f32(o[q]) : y[q]);
            }
        }
    }
}

// out[j][c] or out[c][j] += sum over m of g[m][j] V[m][c] for the 32 columns from c0, g = mul * sum over
// z < SU of U[z]. Wave w takes an eighth of the token rows; the eight sums of a column meet in LDS,
// added in order. The products run on the f32 MFMAs (32 x 32 x 2; 16 x 16 x 4 up to rank 16, rank 8 with
// zero rows): exact f32 operands and f32 sums as FMAs give, and a lane's operand is the value it loaded.
// FMAs with g broadcast from LDS were bound by the LDS reads (16 bytes for four FMAs of a wave): the
// 777-token, 2560 + 1408-column launch at rank 32 took 41 us, now 26.
template <int R>
__device__ __forceinline__ void grad_item(const float* U, int SU, float mul, int64_t T, const uint16_t* V, int64_t C, int64_t c0,
                          float* out, bool transposed, float* lds) {
    using Acc = float __attribute__((ext_vector_type(R >= 32 ? 16 : 4)));
    constexpr int kW = kThreads / 64;
    constexpr int kM = R >= 32 ? 32 : 16;     // an MFMA's factor rows and columns
    constexpr int kRowsMf = 64 / kM;          // its token rows: lane / kM
    constexpr int kJ = R > kM ? R / kM : 1;   // factor-row tiles
    constexpr int kC = kGradCols / kM;        // column tiles
    constexpr int kBatch = 16;  // token rows loaded at a time, the next while these multiply (32: no faster, and slower to 256 tokens)
    constexpr int kN = kBatch / kRowsMf;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, hi = lane / kM, lo = lane % kM;
    const int64_t per = ((T + kW - 1) / kW + kRowsMf - 1) / kRowsMf * kRowsMf;
    const int64_t b = wave * per, e = b + per < T ? b + per : T;
    Acc acc[kJ][kC] = {};
    float x[kN][kC], h[kN][kJ];
    const int c32 = (int)C, lu = lo < R ? lo : 0;
    // rows past e (and factor rows past R) load a valid element and count as zero
    auto load = [&](int64_t m) {
        const int rows = (int)(e - m);
        const uint16_t* vp = V + m * C + c0 + lo;
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            const int row = kRowsMf * i + hi;
#pragma unroll
            for (int c = 0; c < kC; ++c) {
                const uint16_t v = vp[(row < rows ? row * c32 : 0) + c * kM];
                x[i][c] = row < rows ? bf16_to_f32(v) : 0.0f;
            }
        }
        const float* u = U + m * R + lu;
#pragma unroll
        for (int i = 0; i < kN; ++i)
#pragma unroll
            for (int j = 0; j < kJ; ++j) h[i][j] = u[(kRowsMf * i + hi < rows ? kRowsMf * i + hi : 0) * R + j * kM];
        for (int z = 1; z < SU; ++z) {
            u += T * R;
#pragma unroll
            for (int i = 0; i < kN; ++i)
#pragma unroll
                for (int j = 0; j < kJ; ++j) h[i][j] += u[(kRowsMf * i + hi < rows ? kRowsMf * i + hi : 0) * R + j * kM];
        }
#pragma unroll
        for (int i = 0; i < kN; ++i)
#pragma unroll
            for (int j = 0; j < kJ; ++j) h[i][j] = kRowsMf * i + hi < rows && lo < R ? mul * h[i][j] : 0.0f;
    };
    if (b < e) load(b);
    for (int64_t m = b; m < e; m += kBatch) {
        float xc[kN][kC], hc[kN][kJ];
#pragma unroll
        for (int i = 0; i < kN; ++i) {
#pragma unroll
            for (int c = 0; c < kC; ++c) xc[i][c] = x[i][c];
#pragma unroll
            for (int j = 0; j < kJ; ++j) hc[i][j] = h[i][j];
        }
        if (m + kBatch < e) load(m + kBatch);  // on their way while these rows multiply
#pragma unroll
        for (int i = 0; i < kN; ++i)
#pragma unroll
            for (int j = 0; j < kJ; ++j)
#pragma unroll
                for (int c = 0; c < kC; ++c) {
                    if constexpr (kM == 32)
                        acc[j][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(hc[i][j], xc[i][c], acc[j][c], 0, 0, 0);
                    else
                        acc[j][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(hc[i][j], xc[i][c], acc[j][c], 0, 0, 0);
                }
    }
    // [wave][R][32 columns]; a lane holds factor rows 4 * (lane / kM) + .. of the column lane % kM
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
        for (int c = 0; c < kC; ++c)
#pragma unroll
            for (int q = 0; q < (kM == 32 ? 16 : 4); ++q) {
                const int row = j * kM + q / 4 * 8 + 4 * hi + q % 4;
                if (row < R) lds[(wave * R + row) * kGradCols + c * kM + lo] = acc[j][c][q];
            }
    __syncthreads();
    for (int i = threadIdx.x; i < R * kGradCols; i += kThreads) {
        // neighbouring threads neighbouring elements of the output
        const int j = transposed ? i % R : i / kGradCols, c = transposed ? i / R : i % kGradCols;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < kW; ++w) v += lds[(w * R + j) * kGradCols + c];
        out[transposed ? (c0 + c) * R + j : (int64_t)j * C + c0 + c] += v;
    }
}

struct Counts {
    int dA, dB, outputs, rows, copies[2];  // workgroups of each kind, in this order (the longest first)
    int ctiles;
};

template <int R>
__global__ __launch_bounds__(kThreads, R <= 32 ? 4 : 2) void sm_finish_kernel(const Finish f, const Counts n) {
    // the gradients' sums [8][R][32]; the output's u [32][R]
    __shared__ __attribute__((aligned(16))) float lds[8 * kGradCols * (R < 8 ? 8 : R)];
    int b = blockIdx.x;
    if constexpr (R > 0) {
        if (b < n.dA + n.dB) {  // one call, so that it inlines
            const bool a = b < n.dA;
            return grad_item<R>(a ? f.U : f.t, a ? f.SU : 1, a ? f.scale : f.tscale, f.T, a ? f.X : f.dY, a ? f.K : f.N,
                                (int64_t)(a ? b : b - n.dA) * kGradCols, a ? f.dA : f.dB, !a, lds);
        }
        b -= n.dA + n.dB;
    }
    if (b < n.outputs) return output_item(f, lds, (int64_t)(b / n.ctiles) * kRows, (int64_t)(b % n.ctiles) * kCols);
    b -= n.outputs;
    if constexpr (R > 0) {
        if (b < n.rows) {
            const int64_t i = (int64_t)b * kThreads + threadIdx.x, tr = f.T * R;
            if (i >= tr) return;
            if (f.t_out || f.u_out) {
                const float v = sum_ranges(f.U, f.SU, tr, i);
                if (f.t_out) f.t_out[i] = v;
                if (f.u_out) f.u_out[i] = f.u_add ? f.u_out[i] + f.scale * v : f.scale * v;
            }
            if (f.ts) f.ts[i] = f.tscale * f.t[i];
            return;
        }
        b -= n.rows;
    }
    const Finish::Copy& c = f.copy[b < n.copies[0] ? 0 : 1];
    if (b >= n.copies[0]) b -= n.copies[0];
    // (A as the caller holds it may lie off 16 bytes: a value at a time)
    const bool vec = (reinterpret_cast<uintptr_t>(c.from) & 15) == 0;
    for (int64_t i = (int64_t)b * kCopy + 8 * threadIdx.x; i < c.n && i < (int64_t)(b + 1) * kCopy; i += 8 * kThreads) {
        uint4 v;
        if (vec) {
            v = *reinterpret_cast<const uint4*>(c.from + i);
        } else {
            const uint16_t* p = c.from + i;
            v = uint4{(uint32_t)p[0] | (uint32_t)p[1] << 16, (uint32_t)p[2] | (uint32_t)p[3] << 16,
                      (uint32_t)p[4] | (uint32_t)p[5] << 16, (uint32_t)p[6] | (uint32_t)p[7] << 16};
        }
        *reinterpret_cast<uint4*>(c.to + i) = v;
    }
}

}  // namespace

int launch_finish(const Finish& f, hipStream_t s) {
    Counts n{};
    if (f.out) {
        n.ctiles = (int)(f.outs / kCols);
        n.outputs = (int)((f.T + kRows - 1) / kRows) * n.ctiles;
    }
    if (f.rank > 0) {
        if (f.dA) n.dA = (int)(f.K / kGradCols);
        if (f.dB) n.dB = (int)(f.N / kGradCols);
        if (f.t_out || f.u_out || f.ts) n.rows = (int)((f.T * f.rank + kThreads - 1) / kThreads);
    }
    for (int i = 0; i < 2; ++i)
        if (f.copy[i].to) n.copies[i] = (int)((f.copy[i].n + kCopy - 1) / kCopy);
    const int grid = n.outputs + n.dA + n.dB + n.rows + n.copies[0] + n.copies[1];
    if (grid == 0) return R97Q_OK;
    const dim3 g((unsigned)grid), t(kThreads);
    switch (f.rank) {
        case 0: hipLaunchKernelGGL(sm_finish_kernel<0>, g, t, 0, s, f, n); break;
        case 8: hipLaunchKernelGGL(sm_finish_kernel<8>, g, t, 0, s, f, n); break;
        case 16: hipLaunchKernelGGL(sm_finish_kernel<16>, g, t, 0, s, f, n); break;
        case 32: hipLaunchKernelGGL(sm_finish_kernel<32>, g, t, 0, s, f, n); break;
        default: hipLaunchKernelGGL(sm_finish_kernel<64>, g, t, 0, s, f, n); break;
    }
    return launch_status("sm_finish_kernel");
}

}  // namespace sm
}  // namespace r97q
