// qlinear_sm.h -- parameters and launchers of the few-token path of the linear + LoRA layer: the split
// products (qlinear_sm.hip, compiled once per code width) and the launch that finishes them
// (sm_finish.hip).
//
// Two launches a direction. The first deals each output tile's reduction over S ranges, a workgroup
// each, and beside them the adapter's down product (t = X.A^T or dY.B) over SD ranges: every
// workgroup writes an f32 partial. The second adds the partials in range order, folds the adapter's
// up-projection in, and writes Y or dX; in the backward other workgroups of it add the factor
// gradients. No launch reads what another workgroup of the same launch writes.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qlinear_rt.h"

namespace r97q {
namespace sm {

// tokens a workgroup's tile holds
inline int tile_tokens(int64_t T) { return T <= 32 ? 32 : T <= 64 ? 64 : 128; }

struct Params {
    rt::Params w;         // the weight: stream, scale_t, a24, b, run_rows, N, K; and T
    const uint16_t* act;  // X [T, K] (forward) or dY [T, N] (dX), row-major
    const uint16_t* F;    // the down product's factor: A [r, K] (forward) or B [N, r] (dX)
    int fvec;             // F takes 16-byte loads (A as the caller holds it may not: a value at a time)
    int rank;
    int S;                // ranges the products' reduction is dealt over
    int SD;               // and the down product's
    int mtiles, otiles;
    int mblocks;          // 32-token blocks, the down product's
    int ndown;            // down workgroups: mblocks * SD, or 0
    int nprod;            // product workgroups: mtiles * otiles * S, or 0
    float* part;          // [S][T][outputs]
    float* tpart;         // [SD][T][r]
    const float* a_scale; // launch_coded_dx: f32 [T, otiles]
};
template <int BITS>
void launch_products(const Params& p, bool fwd, hipStream_t s);

// gemm_nt_q's adjoint (w.out (+)= a_scale[m, k/128] * (act . W)[m, k]; S 1, nprod tiles) with tiles of
// `tile` tokens, and the tile it takes: the smallest of 32 (up to 32 tokens), 64 (up to 64), 128 and 256
// with at most a tile a CU, or 0 where 256 are still more (the 512-token tiles then fill the chip)
template <int BITS>
void launch_coded_dx(const Params& p, int tile, hipStream_t s);
inline int coded_tile(int64_t T, int64_t K) {
    if (T <= 32) return 32;
    if (T <= 64) return 64;
    for (int bm : {128, 256})
        if ((T + bm - 1) / bm * (K / 128) <= 256) return bm;
    return 0;
}

// One finishing launch: the parts whose counts are non-zero. `u` below is scale * sum over z < SU of
// U[z] (f32 [T, r] each): s.t in the forward, dt in the backward.
struct Finish {
    int64_t T;
    int rank;
    const float* U;
    int SU;
    float scale;
    // Y or dX [T, outs] (+)= sum over z < S of part[z] + u . F^T (forward: F = B [outs, r]) or
    // u . F (dX: F = A [r, outs]); S may be 0; null out: none
    const float* part;
    int S;
    int64_t outs;
    const uint16_t* F;
    int fvec;  // F takes 16-byte (forward) or 8-byte (dX) loads
    int fwd;
    void* out;
    int out_f32, accumulate, vec;  // vec: out takes 4-value accesses
    // t_out [T, r] = sum over z of U[z]; u_out [T, r] = u (+= with u_add; either may be null)
    float* t_out;
    float* u_out;
    int u_add;
    // dA [r, K] += u^T . X, dB [N, r] += tscale * dY^T . t (either may be null)
    const uint16_t* X;
    int64_t K;
    float* dA;
    const uint16_t* dY;
    const float* t;
    float tscale;
    int64_t N;
    float* dB;
    // what a later stage reads: ts [T, r] = tscale * t, and copies of bf16 operands (n a multiple of 8, `to`
    // on 16 bytes, `from` anywhere; null `to`: none)
    float* ts;
    struct Copy {
        const uint16_t* from;
        uint16_t* to;
        int64_t n;
    } copy[2];
};
int launch_finish(const Finish& f, hipStream_t s);

}  // namespace sm
}  // namespace r97q
