// adamw.hip -- the LoRA factors' AdamW on the card: the reference's Optimiser::step
// (src/optim.cpp:223-307, include/r97/optim.h) over device f32 master weights, moments and
// accumulation buffers.
//
// Bit for bit with the reference's host optimiser: every element operation is the reference's f32
// operation in its order (correctly rounded, never contracted into an FMA; the square root
// through f64, measured: the f32 one differs from the correctly rounded value in ~15% of inputs); the global
// norm is the reference's -- one double partial a fixed 4096-element chunk of the parameters'
// concatenation, each summed in element order (a chunk that spans two parameters continues across
// them), the partials added in chunk order; the schedule and the bias corrections are the
// reference's host expressions.
//
// Launches: an update is one elementwise pass over every parameter (a table of up to kTable
// rows a launch), reading this call's gradients and/or the accumulation buffers, and writing
// the weights, both moments, the cleared buffers and (optionally) the weights' bf16 copies. The
// reference's in-place passes over the buffers (the sum, the mean, the clip's scaling) are folded
// into that pass as the same f32 operations on the value. With clipping, two launches come first:
// the chunk partials, then one workgroup that adds them and leaves the clip factor on the card -- no
// host read-back, nothing to synchronise.
//
// Staged gradients (R97Q_ADAMW_GRADS_STAGED): the gradients are the device rows' f32 staging
// buffers; the call takes each value as the reference's grad_stage flush leaves it in a zero-filled
// leaf (one bf16 rounding, src/adjoint/device/grad_stage.cpp:69-73) and clears the buffers in the
// same pass -- the flush, the leaf fill and the optimiser's step in one.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "../../include/r97q.h"
#include "status.h"

// hipcc contracts a * b + c into one FMA by default (one rounding instead of the reference's two):
// contraction is off for this file's arithmetic (written with plain operators: the __f*_rn helpers
// are header functions, compiled outside this pragma, whose products still contract).
#pragma clang fp contract(off)

namespace {

constexpr int64_t kNormChunk = 4096;
constexpr int64_t kScaleBytes = 16;  // the workspace's head: the clip factor (f32), then the partials

// where this call's gradient total comes from
constexpr int kFromAcc = 1;  // the accumulation buffers (earlier calls' sums)
constexpr int kFromG = 2;    // this call's gradients
constexpr int kStaged = 4;   // ... staged: rounded once to bf16, and the staging buffers cleared

// The parameters of one elementwise launch (the table travels in the kernel arguments, which hold
// 4 KiB: 70 rows of 56 bytes and the scalars). A parameter longer than kRowMax goes in as several
// rows. Measured over the 192 factors of the 24-layer stack (12.6 M values, 377 MB): 16 rows a
// launch and a value a thread, 12 launches of 9.7 us; see update_kernel for this form.
constexpr int kTable = 70;
constexpr int64_t kRowMax = int64_t(1) << 29;
constexpr int kPerThread = 4, kPerBlock = 256 * kPerThread;

struct Row {
    float* w;
    float* m;
    float* v;
    float* acc;
    float* g;
    uint16_t* wb;
    uint32_t block0;  // first block of this row in the launch
    uint32_t n_flags; // the row's values << 2 | kVec | kDecay
};
constexpr uint32_t kVec = 1;    // every buffer of the row takes 4-value accesses (16-byte aligned; wb 8)
constexpr uint32_t kDecay = 2;  // the weight decay applies
static_assert(sizeof(Row) == 56 && kTable * sizeof(Row) + 128 <= 4096, "the table fits the kernel arguments");

struct Table {
    Row r[kTable];
    int count;
};

// the row that holds block `block`: a binary search, uniform over the workgroup
__device__ __forceinline__ int row_of_block(const Table& t, uint32_t block) {
    int lo = 0, hi = t.count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (block >= t.r[mid].block0) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ uint16_t bf16_rne(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x7FFFFFFFu) > 0x7F800000u ? (uint16_t)((u >> 16) | 0x0040u)
                                           : (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// a gradient value (staged: as the flush leaves it in the leaf)
__device__ __forceinline__ float grad_of(float g, int mode) {
    return (mode & kStaged) ? __uint_as_float((uint32_t)bf16_rne(g) << 16) : g;
}

// the accumulated gradient as the reference's buffer holds it when the update reads it:
// (acc + g) (the last call's accumulation), x 1/k (the mean, when k > 1). With the gradients alone
// the buffer held zero: 0 + g is g (a -0 that would turn +0 changes no result).
__device__ __forceinline__ float grad_total(float acc, float g, int mode, float inv_k) {
    const float x = (mode & kFromAcc) ? acc + grad_of(g, mode) : grad_of(g, mode);
    return inv_k != 1.0f ? x * inv_k : x;
}

// values j .. j+3 of a buffer, j + 4 <= n when `vec` (one 16-byte access), else those below n
__device__ __forceinline__ void load4(const float* p, uint32_t j, uint32_t n, bool vec, float (&x)[4]) {
    if (vec) {
        const float4 v = *reinterpret_cast<const float4*>(p + j);
        x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = j + u < n ? p[j + u] : 0.0f;
    }
}
__device__ __forceinline__ void store4(float* p, uint32_t j, uint32_t n, bool vec, const float (&x)[4]) {
    if (vec) {
        *reinterpret_cast<float4*>(p + j) = float4{x[0], x[1], x[2], x[3]};
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (j + u < n) p[j + u] = x[u];
    }
}

__global__ __launch_bounds__(256) void accumulate_kernel(const Table t, int mode) {
    const Row& r = t.r[row_of_block(t, blockIdx.x)];
    const uint32_t n = r.n_flags >> 2, j = (blockIdx.x - r.block0) * kPerBlock + threadIdx.x * kPerThread;
    if (j >= n) return;
    const bool vec = (r.n_flags & kVec) && j + 4 <= n;
    float a[4], g[4];
    load4(r.acc, j, n, vec, a);
    load4(r.g, j, n, vec, g);
#pragma unroll
    for (int u = 0; u < 4; ++u) a[u] = a[u] + grad_of(g[u], mode);
    store4(r.acc, j, n, vec, a);
    if (mode & kStaged) store4(r.g, j, n, vec, {0.0f, 0.0f, 0.0f, 0.0f});
}

// ---------------------------------------------------------------- the global norm
// The parameters of one norm launch: the gradients' (and, with ACC, the accumulation buffers')
// pointers and their first elements in the concatenation (off[count] its end).
template <bool ACC>
struct NormTable {
    static constexpr int kRows = ACC ? 160 : 240;
    const float* g[kRows];
    const float* acc[ACC ? kRows : 1];
    int64_t off[kRows + 1];
    int count;
};
static_assert(sizeof(NormTable<true>) <= 4032 && sizeof(NormTable<false>) <= 4032, "the table fits the kernel arguments");

// The chunks' partials. A chunk's 4096 squares are one serial chain of f64 adds (the reference's
// order), so a launch takes at least that chain's latency, and everything else has to stay out of
// its way: a workgroup takes kNormLanes chunks, a loader wave each and one adding wave. A loader
// brings in a segment of its chunk (coalesced, the next segment's loads in flight meanwhile) and
// squares it into one of two LDS slots in f64 (the square of an f32 is exact there, so the product's
// rounding is no question); the adding wave runs the chains, one a lane, two squares an LDS
// access. More chunks a workgroup would leave CUs idle, fewer would put several adding waves on a
// SIMD. Measured over the 24-layer stack's 12.6 M values: 38.7 us against 12 x 1000 us for a lane a chunk,
// each lane loading its own chunk's values (64 lines an instruction), and 92 us for one wave that
// both loads and adds.
constexpr int kNormLanes = 4;
constexpr int kNormSeg = 256;  // values of a chunk a step
constexpr int kNormHold = kNormSeg / 64;
constexpr int kNormThreads = 64 * (kNormLanes + 1);

template <bool ACC>
__global__ __launch_bounds__(kNormThreads) void norm_partials_kernel(const NormTable<ACC> t, int mode, float inv_k,
                                                                     int64_t c0, int64_t c1,
                                                                     double* __restrict__ partials) {
    __shared__ __attribute__((aligned(16))) double sq[2][kNormLanes][kNormSeg + 2];  // rows 4 banks apart
    constexpr int kSteps = (int)kNormChunk / kNormSeg;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t first = t.off[0], end = t.off[t.count];
    const int64_t cb = c0 + (int64_t)blockIdx.x * kNormLanes;
    // the LDS reads and writes of a step are done; a loader's global loads stay in flight
    auto step_end = []() {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        asm volatile("s_barrier" ::: "memory");
    };
    if (wave < kNormLanes) {
        const int64_t c = cb + wave;
        int row = 0;
        float g[kNormHold], acc[kNormHold];
        // the values of a step as they are held, zero outside this launch's parameters (adding the
        // zero's square leaves a partial as it is)
        auto load = [&](int step) {
            const int64_t s0 = c * kNormChunk + step * kNormSeg;
#pragma unroll
            for (int h = 0; h < kNormHold; ++h) g[h] = acc[h] = 0.0f;
            if (c >= c1) return;
            while (row + 1 < t.count && s0 >= t.off[row + 1]) ++row;
            if (s0 >= t.off[row] && s0 + kNormSeg <= t.off[row + 1]) {  // the segment lies in one parameter
                const int64_t j = s0 - t.off[row] + lane;
#pragma unroll
                for (int h = 0; h < kNormHold; ++h) {
                    g[h] = t.g[row][j + 64 * h];
                    if constexpr (ACC) acc[h] = t.acc[row][j + 64 * h];
                }
            } else {
#pragma unroll
                for (int h = 0; h < kNormHold; ++h) {
                    const int64_t e = s0 + 64 * h + lane;
                    if (e >= first && e < end) {
                        int i = row;
                        while (e >= t.off[i + 1]) ++i;
                        g[h] = t.g[i][e - t.off[i]];
                        if constexpr (ACC) acc[h] = t.acc[i][e - t.off[i]];
                    }
                }
            }
        };
        load(0);
        for (int step = 0; step < kSteps; ++step) {
#pragma unroll
            for (int h = 0; h < kNormHold; ++h) {
                const double v = (double)grad_total(acc[h], g[h], mode, inv_k);
                sq[step & 1][wave][64 * h + lane] = v * v;
            }
            if (step + 1 < kSteps) load(step + 1);
            step_end();  // step's squares are in; the adder reads them while the other slot is filled
        }
        return;
    }
    const int mine = lane & (kNormLanes - 1);  // the chunk this lane adds (lanes past kNormLanes repeat)
    const int64_t c = cb + mine;
    // a chunk that starts before the launch's first element continues the partial an earlier launch left
    double part = c < c1 && c * kNormChunk < first ? partials[c] : 0.0;
    step_end();
    for (int step = 0; step < kSteps; ++step) {
        const double2* s = reinterpret_cast<const double2*>(sq[step & 1][mine]);
        double2 a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] = s[u];
        for (int q = 0; q < kNormSeg / 2; q += 16) {
#pragma unroll
            for (int u = 0; u < 8; ++u) b[u] = s[q + 8 + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                part += a[u].x;
                part += a[u].y;
            }
            const int qn = q + 16 < kNormSeg / 2 ? q + 16 : 0;
#pragma unroll
            for (int u = 0; u < 8; ++u) a[u] = s[qn + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                part += b[u].x;
                part += b[u].y;
            }
        }
        if (step + 1 < kSteps) step_end();
    }
    if (lane < kNormLanes && c < c1) partials[c] = part;
}

// src/optim.cpp:131-184: the norm from the chunk partials (added in chunk order), and the factor
// the clip multiplies by (1 when it does not bite: x * 1 is x). One workgroup: the partials into LDS
// a piece at a time, added serially from there (3072 partials: 20.6 us, 5 ns an add; one thread
// loading each as it adds, 172 us).
constexpr int kFactorPiece = 4096;
__global__ __launch_bounds__(256) void clip_factor_kernel(const double* __restrict__ partials, int64_t chunks, float clip,
                                                          float* __restrict__ factor) {
    __shared__ __attribute__((aligned(16))) double s[kFactorPiece];
    double sq = 0.0;
    for (int64_t c0 = 0; c0 < chunks; c0 += kFactorPiece) {
        const int n = (int)(chunks - c0 < kFactorPiece ? chunks - c0 : kFactorPiece);
        const int up = (n + 15) & ~15;  // zeros up to a whole step: they leave the sum as it is
#pragma unroll 4
        for (int i = threadIdx.x; i < up; i += 256) s[i] = i < n ? partials[c0 + i] : 0.0;
        __syncthreads();
        if (threadIdx.x < 64) {
            const double2* d = reinterpret_cast<const double2*>(s);
            double2 a[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) a[u] = d[u];
            for (int q = 0; q < up / 2; q += 8) {
                double2 b[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) b[u] = d[q + 8 < up / 2 ? q + 8 + u : u];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    sq += a[u].x;
                    sq += a[u].y;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) a[u] = b[u];
            }
        }
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    const float norm = (float)sqrt(sq);
    *factor = norm > clip && norm > 0.0f ? clip / norm : 1.0f;
}

// the AdamW element update (src/optim.cpp:278-289); the accumulation buffer cleared when it was read.
// Bound by memory (30 bytes a value): four values a thread in 16-byte accesses. Measured over the
// 24-layer stack (377 MB): 66 us (5.7 TB/s) for three launches of up to 70 factors, against 116 us
// for twelve of 16 with a value a thread.
__global__ __launch_bounds__(256) void update_kernel(const Table t, int mode, float inv_k,
                                                     const float* __restrict__ clip, float lr, float b1, float b2,
                                                     float omb1, float omb2, float eps, float bc1, float bc2,
                                                     float weight_decay) {
    const Row& r = t.r[row_of_block(t, blockIdx.x)];
    const uint32_t n = r.n_flags >> 2, j = (blockIdx.x - r.block0) * kPerBlock + threadIdx.x * kPerThread;
    if (j >= n) return;
    const bool vec = (r.n_flags & kVec) && j + 4 <= n;
    const float wd = (r.n_flags & kDecay) ? weight_decay : 0.0f;
    float a[4] = {}, g[4], w[4], m[4], v[4];
    if (mode & kFromAcc) load4(r.acc, j, n, vec, a);
    load4(r.g, j, n, vec, g);
    load4(r.w, j, n, vec, w);
    load4(r.m, j, n, vec, m);
    load4(r.v, j, n, vec, v);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        float x = grad_total(a[u], g[u], mode, inv_k);
        if (clip) x = x * *clip;
        m[u] = b1 * m[u] + omb1 * x;
        v[u] = b2 * v[u] + omb2 * x * x;
        const float mh = m[u] / bc1;
        const float vh = v[u] / bc2;
        // sqrt through f64: the f32 square root here is not always the correctly rounded one, the f64
        // one rounded to f32 is (53 >= 2 * 24 + 2 significant bits: the double rounding is innocuous)
        const float sq = (float)sqrt((double)vh);
        w[u] = w[u] - lr * (mh / (sq + eps) + wd * w[u]);
    }
    store4(r.m, j, n, vec, m);
    store4(r.v, j, n, vec, v);
    store4(r.w, j, n, vec, w);
    if (mode & kFromAcc) store4(r.acc, j, n, vec, {0.0f, 0.0f, 0.0f, 0.0f});
    if (mode & kStaged) store4(r.g, j, n, vec, {0.0f, 0.0f, 0.0f, 0.0f});
    if (!r.wb) return;
    uint16_t o[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) o[u] = bf16_rne(w[u]);
    if (vec) {
        *reinterpret_cast<uint2*>(r.wb + j) =
            uint2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (j + u < n) r.wb[j + u] = o[u];
    }
}

__global__ __launch_bounds__(256) void to_bf16_kernel(const float* __restrict__ x, uint16_t* __restrict__ y, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = bf16_rne(x[i]);
}

unsigned blocks(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

int64_t total_of(const R97qAdamWParam* p, int32_t count) {
    int64_t t = 0;
    for (int32_t i = 0; i < count; ++i) t += p[i].n;
    return t;
}

// every buffer of parameter q takes 4-value accesses (and so do its rows: kRowMax is a multiple of 4)
bool aligned(const R97qAdamWParam& q, const float* g) {
    const uintptr_t f = (uintptr_t)q.w | (uintptr_t)q.m | (uintptr_t)q.v | (uintptr_t)q.acc | (uintptr_t)g;
    return f % 16 == 0 && (uintptr_t)q.w_bf16 % 8 == 0;
}

// the elementwise launches: tables of up to kTable rows
template <class F>
int for_each_table(const R97qAdamWParam* p, float* const* grads, int32_t count, F&& f) {
    Table t{};
    uint32_t nblocks = 0;
    auto flush = [&]() {
        if (t.count == 0) return R97Q_OK;
        const int e = f(t, nblocks);
        t = Table{};
        nblocks = 0;
        return e;
    };
    for (int32_t i = 0; i < count; ++i) {
        const R97qAdamWParam& q = p[i];
        const uint32_t flags = (aligned(q, grads[i]) ? kVec : 0) | (q.decay ? kDecay : 0);
        for (int64_t at = 0; at < q.n; at += kRowMax) {
            const int64_t n = q.n - at < kRowMax ? q.n - at : kRowMax;
            if (t.count == kTable || (int64_t)nblocks + blocks(n, kPerBlock) > INT32_MAX)
                if (int e = flush()) return e;
            t.r[t.count++] = Row{q.w + at, q.m + at, q.v + at, q.acc + at, grads[i] + at,
                                 q.w_bf16 ? q.w_bf16 + at : nullptr, nblocks, (uint32_t)n << 2 | flags};
            nblocks += blocks(n, kPerBlock);
        }
    }
    return flush();
}

// the chunk partials of the global norm: tables of up to NormTable<ACC>::kRows parameters
template <bool ACC>
int launch_norm(const R97qAdamWParam* p, float* const* grads, int32_t count, int mode, float inv_k, double* partials,
                hipStream_t s) {
    int64_t off = 0;
    for (int32_t first = 0; first < count; first += NormTable<ACC>::kRows) {
        NormTable<ACC> t{};
        t.count = count - first < NormTable<ACC>::kRows ? count - first : NormTable<ACC>::kRows;
        for (int i = 0; i < t.count; ++i) {
            t.g[i] = grads[first + i];
            if constexpr (ACC) t.acc[i] = p[first + i].acc;
            t.off[i] = off;
            off += p[first + i].n;
        }
        t.off[t.count] = off;
        const int64_t c0 = t.off[0] / kNormChunk, c1 = (off + kNormChunk - 1) / kNormChunk;
        hipLaunchKernelGGL(norm_partials_kernel<ACC>, dim3(blocks(c1 - c0, kNormLanes)), dim3(kNormThreads), 0, s, t, mode, inv_k,
                           c0, c1, partials);
        if (int e = r97q::launch_status("adamw norm partials")) return e;
    }
    return R97Q_OK;
}

}  // namespace

extern "C" {

// src/optim.cpp:113-126
float r97q_scheduled_lr(const R97qAdamWConfig* cfg, int32_t step) {
    if (step <= 0) return 0.0f;
    const double base = cfg->lr > 0.0f ? double(cfg->lr) : 0.0;
    if (cfg->warmup_steps > 0 && step <= cfg->warmup_steps) {
        const double r = double(step) / double(cfg->warmup_steps);
        return float(base * r);
    }
    if (cfg->total_steps <= 0 || cfg->total_steps <= cfg->warmup_steps) return cfg->lr;
    const double floor_v = base * (cfg->lr_floor_frac >= 0.0f ? double(cfg->lr_floor_frac) : 0.0);
    const double horizon = double(cfg->total_steps - cfg->warmup_steps);
    const double tt = double(step - cfg->warmup_steps);
    const double t = tt < horizon ? tt : horizon;
    const double angle = 3.14159265358979323846 * t / horizon;
    return float(floor_v + (base - floor_v) * 0.5 * (1.0 + std::cos(angle)));
}

int64_t r97q_adamw_workspace_bytes(const R97qAdamWParam* params, int32_t count) {
    if (!params || count <= 0) return -1;
    return kScaleBytes + (total_of(params, count) + kNormChunk - 1) / kNormChunk * (int64_t)sizeof(double);
}

int r97q_adamw_step(const R97qAdamWConfig* cfg, const R97qAdamWParam* params, float* const* grads,
                    int32_t count, int32_t flags, int32_t* updates, int32_t* pending, int32_t* applied,
                    void* workspace, int64_t workspace_bytes, R97IqrStream stream) {
    r97q::clear_error();
    const char* who = "r97q_adamw_step";
    if (!cfg || !params || !grads || count <= 0 || !updates || !pending || cfg->accum_steps <= 0 ||
        (flags & ~R97Q_ADAMW_GRADS_STAGED)) {
        r97q::set_error("%s: null argument, no parameters, accum_steps < 1 or unknown flags", who);
        return R97Q_EINVAL;
    }
    for (int32_t i = 0; i < count; ++i)
        if (!params[i].w || !params[i].m || !params[i].v || !params[i].acc || !grads[i] || params[i].n <= 0) {
            r97q::set_error("%s: parameter %d: null buffer or n <= 0", who, (int)i);
            return R97Q_EINVAL;
        }
    const bool clipping = cfg->clip_norm > 0.0f;
    const int64_t need = r97q_adamw_workspace_bytes(params, count);
    if (clipping && (workspace_bytes < need || !workspace)) {
        r97q::set_error("%s: workspace %lld bytes, needs %lld", who, (long long)workspace_bytes, (long long)need);
        return R97Q_EWORKSPACE;
    }
    const hipStream_t s = (hipStream_t)stream;
    if (applied) *applied = 0;
    const int staged = (flags & R97Q_ADAMW_GRADS_STAGED) ? kStaged : 0;
    const int32_t before = *pending;
    if (++*pending < cfg->accum_steps) {
        // not the update's call: add the gradients into the buffers
        return for_each_table(params, grads, count, [&](const Table& t, uint32_t nb) {
            hipLaunchKernelGGL(accumulate_kernel, dim3(nb), dim3(256), 0, s, t, kFromG | staged);
            return r97q::launch_status("adamw accumulate");
        });
    }
    const int mode = (before > 0 ? kFromAcc : 0) | kFromG | staged;
    const float inv_k = 1.0f / float(*pending);  // the mean (x 1/k; k = 1 leaves the sum as it is)
    float* factor = nullptr;
    if (clipping) {
        factor = static_cast<float*>(workspace);
        double* partials = reinterpret_cast<double*>(static_cast<uint8_t*>(workspace) + kScaleBytes);
        if (int e = before > 0 ? launch_norm<true>(params, grads, count, mode, inv_k, partials, s)
                               : launch_norm<false>(params, grads, count, mode, inv_k, partials, s))
            return e;
        const int64_t chunks = (total_of(params, count) + kNormChunk - 1) / kNormChunk;
        hipLaunchKernelGGL(clip_factor_kernel, dim3(1), dim3(256), 0, s, partials, chunks, cfg->clip_norm, factor);
        if (int e2 = r97q::launch_status("adamw clip factor")) return e2;
    }
    const int32_t t = *updates + 1;
    const float lr = r97q_scheduled_lr(cfg, t);
    const float b1 = cfg->beta1, b2 = cfg->beta2;
    const float bc1 = 1.0f - std::pow(b1, float(t));
    const float bc2 = 1.0f - std::pow(b2, float(t));
    int e = for_each_table(params, grads, count, [&](const Table& tb, uint32_t nb) {
        hipLaunchKernelGGL(update_kernel, dim3(nb), dim3(256), 0, s, tb, mode, inv_k, (const float*)factor, lr, b1, b2,
                           1.0f - b1, 1.0f - b2, cfg->eps, bc1, bc2, cfg->weight_decay);
        return r97q::launch_status("adamw update");
    });
    if (e) return e;
    ++*updates;
    *pending = 0;
    if (applied) *applied = 1;
    return R97Q_OK;
}

int r97q_f32_to_bf16(const float* x, uint16_t* y, int64_t n, R97IqrStream stream) {
    r97q::clear_error();
    if (!x || !y || n < 0) {
        r97q::set_error("r97q_f32_to_bf16: null buffer or n < 0");
        return R97Q_EINVAL;
    }
    if (n == 0) return R97Q_OK;
    hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks(n, 256)), dim3(256), 0, (hipStream_t)stream, x, y, n);
    return r97q::launch_status("r97q_f32_to_bf16");
}

}  // extern "C"
