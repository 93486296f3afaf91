// qlinear_sm.hip -- the products of a call with few tokens, for CDNA4 (gfx950). Compiled once per code
// width (-DR97Q_BITS=3..6, or 8 for the int8-code form).
//
//   part[z][m][o] = sum over range z of the reduction of act[m] . W     (W decoded as in qlinear_rt.hip)
//   tpart[z][m][j] = sum over range z of act[m] . factor                (the adapter's down product)
//
// The 512-token tile of qlinear_rt.hip leaves most of the chip idle below about a thousand tokens: a
// 4096 x 4096 layer has 32 of its tiles at one token, each multiplying 511 rows of padding. Here a
// tile holds 32, 64 or 128 tokens x 128 outputs and its reduction is dealt over S ranges, one or two
// workgroups a CU in all. Per 64-deep step a workgroup decodes the 128 x 64 weight tile and brings in its
// tokens' 64 values, both into LDS (two slots each, one barrier a step), and multiplies them; below 128
// tokens the decode's vector instructions, not the MFMAs, are the work, and a range of a few steps
// is latency: a step's loads are issued two steps ahead, and two workgroups share a CU (128
// registers a lane; rings of four sets in one workgroup a CU measured 8-14% slower). The token
// operand comes row-major as the caller holds it, so no launch writes a tiled copy.
// Measured at 4096 x 4096, b5 trellis, a launch: 1 token 12 us, 64 tokens 16 us, 128 tokens 19 us, against 27
// (and a reduction of 4.6) for the 512-token tile.
//
// The decode is qlinear_rt.hip's, value for value, with the wave's row slice a run-time shift instead of
// a compile-time one (the window's dwords are shifted down to the slice's first bit, an operation or
// two for each column's 4 or 8 rows): eight waves then run one copy of the loop, which the
// instruction cache holds.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "qlinear_sm.h"
#include "rt_core.h"

#ifndef R97Q_BITS
#error "compile with -DR97Q_BITS=<code width>"
#endif

namespace r97q {
namespace sm {
namespace {

using rt::as_bf16x8;
using rt::bf16x8;
using rt::f32x16;
using rt::kBN;
using rt::kStep;
using rt::kTileBytes;
using rt::mfma32;
using rt::pack_bf16;
using rt::tile_barrier;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // a native 16-byte vector (registers)
typedef short s16x4 __attribute__((__vector_size__(4 * sizeof(short))));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr int kWaves = 8;
constexpr int kRing = 2;  // register sets: a step's loads are issued kRing steps before its products
constexpr int BITS = R97Q_BITS;
constexpr bool C8 = BITS == R97Q_CODES8;

// the steps of range z of S
__device__ __forceinline__ void range_of(int z, int S, int nsteps, int& s0, int& s1) {
    s0 = (int)((int64_t)z * nsteps / S);
    s1 = (int)((int64_t)(z + 1) * nsteps / S);
}

// ---------------------------------------------------------------- the weight's decode
__device__ __forceinline__ void scale_of(uint32_t w, bool upper, float& sc, float& off) {
    sc = __builtin_bit_cast(float, upper ? (w & 0xFFFF0000u) : (w << 16));
    off = (C8 ? -128.0f : -1150.0f) * sc;
}
// the trellis state's value times the scale, less the offset (qlinear_rt.hip's header): one rounding
// is left for the bf16 conversion
[[maybe_unused]] __device__ __forceinline__ float state_value(uint32_t st, uint32_t a24, uint32_t b, float sc, float off) {
    const uint32_t h = (st * a24 + b) & 0x3F3F3F3Fu;
    const uint32_t d = __builtin_amdgcn_sad_u8(h, 0u, 0x6400u);  // f16(1024 + sum)
    return __builtin_fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)d), sc, off);
}
// the 16-bit window at bit o of hi:lo
[[maybe_unused]] __device__ __forceinline__ uint32_t window(uint32_t hi, uint32_t lo, int o) {
    if (o + 16 <= 32) return (lo >> o) & 0xFFFFu;
    if (o >= 32) return (hi >> (o - 32)) & 0xFFFFu;
    return __builtin_amdgcn_alignbit(hi, lo, o) & 0xFFFFu;
}
// code byte `byte` of w times the scale, less the offset
[[maybe_unused]] __device__ __forceinline__ float code_value(uint32_t w, int byte, float sc, float off) {
    return __builtin_fmaf((float)(((w ^ 0x80808080u) >> (8 * byte)) & 0xFFu), sc, off);
}

// One lane's share of a tile. Forward: tile [128 n][64 k]; wave w decodes rows 4w .. 4w+3 of each of the
// four 32-row segments, lane = (segment lane>>4, columns 4*(lane&15) .. +3). dX: tile [128 k][64 n];
// wave w decodes rows 8*(w&3) .. +7 of segment w>>2, lane = columns 2*lane, 2*lane+1.
template <bool FWD>
struct Lane {
    static constexpr int ROWS = FWD ? 4 : 8;
    static constexpr int NW = FWD ? 2 : 3;  // dwords a column's window spans, from any start bit
    struct Words {
        uint32_t w[8];         // forward: [dword][4 columns]; dX: [dword][2 columns] (6); codes: 4
        uint32_t s[ROWS / 2];  // the rows' bf16 scales
    };
    const uint32_t* base[NW];  // forward: the lane's dwords at step 0
    const uint16_t* scale;     // the lane's rows' scales at step 0 (forward) or its block's (dX)
    const uint8_t* units;      // codes: the lane's bytes at step 0
    int64_t stride;            // codes: bytes between steps (dX)
    uint32_t a24, b;
    int off;                   // the window's first bit within the first dword
    int d0;                    // dX: the window's first dword
    int seg, rs, ns;           // dX: the wave's segment of a step; segments a run; in all
    int64_t K;
    int N;
    int lds[FWD ? 4 : 2];      // the lane's LDS offsets: forward a row each, dX a column each

    __device__ __forceinline__ void setup(const rt::Params& p, int64_t o0, int wave, int lane) {
        K = p.K;
        N = (int)p.N;
        a24 = p.a24;
        b = p.b;
        const int slice = FWD ? wave : wave & 3;
        seg = FWD ? 0 : wave >> 2;
        const int lo = BITS * (32 - ROWS * (slice + 1));
        d0 = lo >> 5;
        off = lo & 31;
        if constexpr (FWD) {
            const int sg = lane >> 4, cg = lane & 15;
            const int64_t g = (o0 >> 5) + sg, srow = 32 * g + 4 * wave;
            scale = p.scale_t + srow;
            if constexpr (C8) {
                const int h = (int)(srow & 7) >> 2;
                units = reinterpret_cast<const uint8_t*>(p.stream) + ((srow >> 3) * (K >> 2) + cg) * 32 + 8 * h;
            } else {
                const int64_t r = p.run_rows >> 5, n = p.N >> 5;
                const int64_t top = (g / r + 1) * r;
                const int64_t gh = g % r != 0 ? g - 1 : (top < n ? top : n) - 1;
#pragma unroll
                for (int t = 0; t < NW; ++t)
                    base[t] = p.stream + (d0 + t < BITS ? (g * BITS + d0 + t) : gh * BITS) * K + 4 * cg;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 32 * sg + 4 * wave + i;
                lds[i] = row * 128 + (((cg >> 1) ^ rt::swz(row)) << 4) + ((cg & 1) << 3);
            }
        } else {
            scale = p.scale_t + (o0 >> 7) * p.N + 32 * seg + 8 * slice;
            if constexpr (C8) {
                units = reinterpret_cast<const uint8_t*>(p.stream) +
                        ((int64_t)(4 * seg + slice) * (K >> 2) + (o0 >> 2) + (lane >> 1)) * 32 + 16 * (lane & 1);
                stride = 8 * (K >> 2) * 32;
            } else {
                rs = (int)(p.run_rows >> 5);
                ns = (int)(p.N >> 5);
                base[0] = p.stream + o0 + 2 * lane;
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int row = 2 * lane + c;
                lds[c] = row * 128 + (((4 * seg + slice) ^ rt::swz(row)) << 4);
            }
        }
    }

    __device__ __forceinline__ void load(int s, Words& x) const {
        if constexpr (FWD) {
            if constexpr (C8) {
                const uint8_t* u = units + (int64_t)s * (kStep / 4 * 32);
                const uint2 a = *reinterpret_cast<const uint2*>(u), c = *reinterpret_cast<const uint2*>(u + 16);
                x.w[0] = a.x; x.w[1] = a.y; x.w[2] = c.x; x.w[3] = c.y;
            } else {
#pragma unroll
                for (int t = 0; t < NW; ++t) {
                    const uint4 v = *reinterpret_cast<const uint4*>(base[t] + (int64_t)s * kStep);
                    x.w[4 * t] = v.x; x.w[4 * t + 1] = v.y; x.w[4 * t + 2] = v.z; x.w[4 * t + 3] = v.w;
                }
            }
            const uint2 v = *reinterpret_cast<const uint2*>(scale + (int64_t)(s >> 1) * N);
            x.s[0] = v.x; x.s[1] = v.y;
        } else {
            if constexpr (C8) {
                const uint4 v = *reinterpret_cast<const uint4*>(units + (int64_t)s * stride);
                x.w[0] = v.x; x.w[1] = v.y; x.w[2] = v.z; x.w[3] = v.w;
            } else {
                // the wave's segment and the one its windows run on into (the segment below, or the
                // run's top one at the seam): uniform
                const int g = 2 * s + seg, q = g / rs, top = (q + 1) * rs;
                const int gh = g != q * rs ? g - 1 : (top < ns ? top : ns) - 1;
#pragma unroll
                for (int t = 0; t < NW; ++t) {
                    const int d = d0 + t < BITS ? d0 + t : BITS;  // a dword past the halo's first is never used
                    const int64_t row = d < BITS ? (int64_t)g * BITS + d : (int64_t)gh * BITS;
                    const uint2 v = *reinterpret_cast<const uint2*>(base[0] + row * K);
                    x.w[2 * t] = v.x; x.w[2 * t + 1] = v.y;
                }
            }
            const uint4 v = *reinterpret_cast<const uint4*>(scale + (int64_t)s * kStep);
            x.s[0] = v.x; x.s[1] = v.y; x.s[2] = v.z; x.s[3] = v.w;
        }
    }

    __device__ __forceinline__ void decode(const Words& x, uint8_t* tile) const {
        if constexpr (FWD) {
            uint32_t wl[4], wh[4];
            if constexpr (!C8) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    wl[c] = __builtin_amdgcn_alignbit(x.w[4 + c], x.w[c], off);
                    wh[c] = 3 * BITS + 16 > 32 ? x.w[4 + c] >> off : 0u;
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float sc, of, v[4];
                scale_of(x.s[i >> 1], i & 1, sc, of);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if constexpr (C8) {
                        const int byte = 8 * (c >> 1) + 2 * i + (c & 1);
                        v[c] = code_value(x.w[byte >> 2], byte & 3, sc, of);
                    } else {
                        v[c] = state_value(window(wh[c], wl[c], BITS * (3 - i)), a24, b, sc, of);
                    }
                }
                *reinterpret_cast<uint2*>(tile + lds[i]) = uint2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
            }
        } else {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                uint32_t wl = 0u, wh = 0u;
                if constexpr (!C8) {
                    wl = __builtin_amdgcn_alignbit(x.w[2 + c], x.w[c], off);
                    wh = __builtin_amdgcn_alignbit(x.w[4 + c], x.w[2 + c], off);
                }
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    float sc, of;
                    scale_of(x.s[i >> 1], i & 1, sc, of);
                    if constexpr (C8) {
                        const int byte = 2 * i + c;
                        v[i] = code_value(x.w[byte >> 2], byte & 3, sc, of);
                    } else {
                        v[i] = state_value(window(wh, wl, BITS * (7 - i)), a24, b, sc, of);
                    }
                }
                *reinterpret_cast<uint4*>(tile + lds[c]) = uint4{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]),
                                                                 pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
            }
        }
    }
};

// the lane's token fragments of step s from its row: reduction values 64s + 32 half + 8j .. +8
template <int NJ>
__device__ __forceinline__ void load_tokens(const uint16_t* row, int s, uint4 (&t)[NJ]) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) t[j] = *reinterpret_cast<const uint4*>(row + (int64_t)s * kStep + 8 * j);
}

// A product workgroup: MT token blocks of 32. With eight, a wave takes one block and all four 32-output
// blocks; with four, one block and two output blocks; with two, one block and one output block; with one, one output block and half of
// each step's reduction (two of its four 16-deep slices), the halves added at the end. A step's
// tokens are read whole-row (eight lanes a 128-byte line) and go through LDS in the weight tile's
// layout: as fragments straight from the rows, 32 lines an instruction and every block loaded by as many
// waves as share it, the loads cost more than the decode.
// DIRECT: the whole reduction (S 1), the product in the code basis of an activation written (or added)
// into the output: times a_scale[m, output tile]; else the range's partial.
template <bool FWD, int MT, bool DIRECT = false>
__device__ __forceinline__ void product_item(const Params& p, uint8_t* tiles, uint8_t* toks, int mt, int ot, int z) {
    constexpr int NN = MT == 8 ? 4 : MT == 4 ? 2 : 1;
    constexpr int NJ = MT == 1 ? 2 : 4;
    constexpr int NT = MT >= 4 ? MT / 2 : 1;  // 16-byte token pieces a thread loads a step
    constexpr int kTokBytes = MT * 32 * 2 * kStep;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int half = lane >> 5, l32 = lane & 31;
    const int blk = MT == 8 ? wave : MT == 4 ? wave >> 1 : MT == 2 ? wave >> 2 : 0;
    const int ni0 = MT == 8 ? 0 : MT == 4 ? 2 * (wave & 1) : wave & 3;
    const int j0 = MT == 1 ? 2 * (wave >> 2) : 0;
    const int64_t red = FWD ? p.w.K : p.w.N, outs = FWD ? p.w.N : p.w.K;
    int s0, s1;
    range_of(z, p.S, (int)(red / kStep), s0, s1);
    const int64_t o0 = (int64_t)ot * kBN;
    // the thread's token pieces: row tid/8 (+ 64) of the tile, 16-byte chunk tid%8 (with one block the
    // second 256 threads repeat the first's, the same bytes to the same place). Rows past T read row
    // T-1: their products are never stored.
    const uint16_t* src[NT];
    int dst[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        const int r = (MT == 1 ? (threadIdx.x & 255) : threadIdx.x + 512 * q) >> 3, c = threadIdx.x & 7;
        int64_t m = (int64_t)mt * 32 * MT + r;
        if (m > p.w.T - 1) m = p.w.T - 1;
        src[q] = p.act + m * red + 8 * c;
        dst[q] = r * 128 + ((c ^ rt::swz(r)) << 4);
    }
    Lane<FWD> w;
    w.setup(p.w, o0, wave, lane);
    // the wave's fragments in LDS: slice j is chunk 4 half + j of a row, at the row's byte 0 plus
    // (chunk ^ swz) * 16, which is this base with j's two bits flipped in
    const int fx = (((4 * half) ^ rt::swz(l32)) << 4) + 128 * l32;
    const int fr = 4096 * ni0 + fx, ft = 4096 * blk + fx;
    f32x16 acc[NN];
#pragma unroll
    for (int ni = 0; ni < NN; ++ni) acc[ni] = (f32x16){};
    typename Lane<FWD>::Words wd[kRing];
    u32x4 tk[kRing][NT];
    const int last = s1 - 1;
    auto at = [&](int s) { return s < last ? s : last; };
    auto fetch = [&](int s, typename Lane<FWD>::Words& x, u32x4 (&t)[NT]) {
        w.load(at(s), x);
#pragma unroll
        for (int q = 0; q < NT; ++q) t[q] = *reinterpret_cast<const u32x4*>(src[q] + (int64_t)at(s) * kStep);
    };
    auto fill = [&](const typename Lane<FWD>::Words& x, const u32x4 (&t)[NT], uint8_t* tok, uint8_t* tile) {
#pragma unroll
        for (int q = 0; q < NT; ++q) *reinterpret_cast<u32x4*>(tok + dst[q]) = t[q];
        w.decode(x, tile);
        tile_barrier();
    };
#pragma unroll
    for (int i = 0; i < kRing; ++i) fetch(s0 + i, wd[i], tk[i]);
    fill(wd[0], tk[0], toks, tiles);
    // step s + I: the loads of step s + I + kRing on their way, the step's products from one LDS slot beside
    // the next step's decode into the other
    auto multiply = [&](const uint8_t* tok, const uint8_t* cur) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const bf16x8 a = as_bf16x8(*reinterpret_cast<const uint4*>(tok + (ft ^ ((j0 + j) << 4))));
#pragma unroll
            for (int ni = 0; ni < NN; ++ni)
                acc[ni] = mfma32(a, as_bf16x8(*reinterpret_cast<const uint4*>(cur + (fr ^ ((j0 + j) << 4)) + 4096 * ni)), acc[ni]);
        }
    };
    for (int s = s0; s < s1; s += kRing) {  // the steps leave by their break (without this bound the compiler does not end)
#define R97Q_SM_STEP(I)                                 \
    fetch(s + I + kRing, wd[I], tk[I]);                 \
    multiply(toks + (I & 1) * kTokBytes, tiles + (I & 1) * kTileBytes);   \
    if (s + I >= last) break;                           \
    fill(wd[(I + 1) % kRing], tk[(I + 1) % kRing], toks + ((I + 1) & 1) * kTokBytes, tiles + ((I + 1) & 1) * kTileBytes);
        R97Q_SM_STEP(0)
        R97Q_SM_STEP(1)
#undef R97Q_SM_STEP
    }
    const int64_t m0 = (int64_t)mt * 32 * MT + 32 * blk;
    if constexpr (MT == 1) {  // the reduction's second half, from waves 4-7 through the LDS tiles
        float* h = reinterpret_cast<float*>(tiles) + (wave & 3) * 1024;
        tile_barrier();
        if (wave >= 4) {
#pragma unroll
            for (int e = 0; e < 16; ++e) h[64 * e + lane] = acc[0][e];
        }
        tile_barrier();
        if (wave >= 4) return;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[0][e] += h[64 * e + lane];
    }
    // accumulator element e: row 8*(e/4) + 4*half + e%4 of the block, column 32 ni + l32
    if constexpr (DIRECT) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int64_t m = m0 + 8 * (e >> 2) + 4 * half + (e & 3);
            if (m >= p.w.T) continue;
            const float f = p.a_scale[m * p.otiles + ot];
            const int64_t at = m * outs + o0 + 32 * ni0 + l32;
#pragma unroll
            for (int ni = 0; ni < NN; ++ni) {
                float v = acc[ni][e] * f;
                if (p.w.out_f32) {
                    float* d = static_cast<float*>(p.w.out) + at + 32 * ni;
                    *d = p.w.accumulate ? *d + v : v;
                } else {
                    uint16_t* d = static_cast<uint16_t*>(p.w.out) + at + 32 * ni;
                    if (p.w.accumulate) v += bf16_to_f32(*d);
                    *d = f32_to_bf16(v);
                }
            }
        }
        return;
    }
    float* out = p.part + (int64_t)z * p.w.T * outs + o0 + 32 * ni0 + l32;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int64_t m = m0 + 8 * (e >> 2) + 4 * half + (e & 3);
        if (m >= p.w.T) continue;
#pragma unroll
        for (int ni = 0; ni < NN; ++ni) out[m * outs + 32 * ni] = acc[ni][e];
    }
}

// A down workgroup: 32 tokens against the factor's r columns over range z of SD, 32 columns a pass. The
// waves take the range's steps in turn; their sums meet in LDS, added in wave order. A [r, K] is the
// MFMA's operand as it lies; of B [N, r] a step's 64 rows go through the wave's 4 KiB of LDS (64 bytes a
// row, columns past r zero) and come back transposed.
template <bool FWD>
__device__ __forceinline__ void down_item(const Params& p, uint8_t* lds, int mb, int z) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int half = lane >> 5, l32 = lane & 31;
    const int64_t n = FWD ? p.w.K : p.w.N;
    const int r = p.rank;
    int s0, s1;
    range_of(z, p.SD, (int)(n / kStep), s0, s1);
    const int64_t m0 = (int64_t)mb * 32;
    int64_t row = m0 + l32;
    if (row > p.w.T - 1) row = p.w.T - 1;
    const uint16_t* tok = p.act + row * n + 32 * half;
    uint8_t* own = lds + 4096 * wave;
    float* red = reinterpret_cast<float*>(lds);  // the waves' sums, 4 KiB each: the same places
    const int pieces = r < 32 ? r >> 3 : 4;      // 16-byte pieces of a B row a pass takes
    for (int c0 = 0; c0 < r; c0 += 32) {
        const int j = c0 + l32;
        f32x16 acc = (f32x16){};
        if constexpr (!FWD) {
#pragma unroll
            for (int q = 0; q < 4; ++q) *reinterpret_cast<u32x4*>(own + 1024 * q + 16 * lane) = u32x4{0u, 0u, 0u, 0u};
        }
        for (int s = s0 + wave; s < s1; s += kWaves) {
            uint4 t[4];
            bf16x8 f[4];
            load_tokens<4>(tok, s, t);
            if constexpr (FWD) {
                const uint16_t* fp = p.F + (int64_t)(j < r ? j : 0) * n + (int64_t)s * kStep + 32 * half;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    u32x4 v;
                    if (p.fvec) {
                        v = *reinterpret_cast<const u32x4*>(fp + 8 * q);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] = (uint32_t)fp[8 * q + 2 * i] | (uint32_t)fp[8 * q + 2 * i + 1] << 16;
                    }
                    if (j >= r) v = u32x4{0u, 0u, 0u, 0u};
                    f[q] = __builtin_bit_cast(bf16x8, v);
                }
            } else {
                const uint8_t* src = reinterpret_cast<const uint8_t*>(p.F + (int64_t)s * kStep * r + c0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (q >= pieces) break;
                    const int i = lane + 64 * q, br = i / pieces, bc = i % pieces;
                    *reinterpret_cast<u32x4*>(own + 64 * br + 16 * bc) =
                        *reinterpret_cast<const u32x4*>(src + (int64_t)br * 2 * r + 16 * bc);
                }
                // one wave's LDS operations run in order. A transposing read gives 16 lanes 4 rows of
                // one column each: lane i's address is row i/4, columns 4 (i%4)
                const int i16 = lane & 15, cb = (lane >> 4) & 1;
                const uint8_t* at = own + (32 * half + (i16 >> 2)) * 64 + 32 * cb + 8 * (i16 & 3);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 512 * q));
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 512 * q + 256));
                    const u32x4 v = {(uint32_t)(uint16_t)lo[0] | (uint32_t)(uint16_t)lo[1] << 16,
                                     (uint32_t)(uint16_t)lo[2] | (uint32_t)(uint16_t)lo[3] << 16,
                                     (uint32_t)(uint16_t)hi[0] | (uint32_t)(uint16_t)hi[1] << 16,
                                     (uint32_t)(uint16_t)hi[2] | (uint32_t)(uint16_t)hi[3] << 16};
                    f[q] = __builtin_bit_cast(bf16x8, v);
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) acc = mfma32(as_bf16x8(t[q]), f[q], acc);
        }
        if (wave > 0) {
#pragma unroll
            for (int e = 0; e < 16; ++e) red[(wave * 16 + e) * 64 + lane] = acc[e];
        }
        __syncthreads();
        if (wave == 0 && j < r) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                float v = acc[e];
#pragma unroll
                for (int q = 1; q < kWaves; ++q) v += red[(q * 16 + e) * 64 + lane];
                const int64_t m = m0 + 8 * (e >> 2) + 4 * half + (e & 3);
                if (m < p.w.T) p.tpart[((int64_t)z * p.w.T + m) * r + j] = v;
            }
        }
        __syncthreads();
    }
}

// The down workgroups come first (short of work but long of latency), then the products, each XCD a
// contiguous run of (range, output tile) pairs with the token tiles inner: a weight tile's readers
// share an L2.
template <bool FWD, int MT>
__global__ __launch_bounds__(64 * kWaves, 4) void sm_products_kernel(const Params p) {
    __shared__ __attribute__((aligned(16))) uint8_t tiles[2 * kTileBytes];
    __shared__ __attribute__((aligned(16))) uint8_t toks[2 * MT * 32 * 2 * kStep];
    const int b = blockIdx.x;
    if (b < p.ndown) return down_item<FWD>(p, tiles, b % p.mblocks, b / p.mblocks);
    const int i = rt::xcd_tile(b - p.ndown, p.nprod);
    const int mt = i % p.mtiles, q = i / p.mtiles;
    product_item<FWD, MT>(p, tiles, toks, mt, q % p.otiles, q / p.otiles);
}

// gemm_nt_q's adjoint where the 512-token tiles of qlinear_fused.hip would leave CUs idle: the whole
// reduction a workgroup, as many token blocks a tile as keep the tiles within one a CU (sm::coded_tile).
// Measured at 4096 x 4096, int8-code weight, with the call's gap: 1 token 30 us, 128 tokens 46, 1024
// tokens 57, 2048 tokens 90, against 98, 105, 120 and 127.
template <int MT>
__global__ __launch_bounds__(64 * kWaves, MT == 8 ? 2 : 4) void sm_coded_dx_kernel(const Params p) {
    __shared__ __attribute__((aligned(16))) uint8_t tiles[2 * kTileBytes];
    __shared__ __attribute__((aligned(16))) uint8_t toks[2 * MT * 32 * 2 * kStep];
    const int i = rt::xcd_tile(blockIdx.x, p.nprod);
    product_item<false, MT, true>(p, tiles, toks, i % p.mtiles, i / p.mtiles, 0);
}

}  // namespace

template <>
void launch_coded_dx<R97Q_BITS>(const Params& p, int tile, hipStream_t s) {
    const dim3 grid((unsigned)p.nprod), block(64 * kWaves);
    switch (tile) {
        case 32: hipLaunchKernelGGL(sm_coded_dx_kernel<1>, grid, block, 0, s, p); break;
        case 64: hipLaunchKernelGGL(sm_coded_dx_kernel<2>, grid, block, 0, s, p); break;
        case 128: hipLaunchKernelGGL(sm_coded_dx_kernel<4>, grid, block, 0, s, p); break;
        default: hipLaunchKernelGGL(sm_coded_dx_kernel<8>, grid, block, 0, s, p); break;
    }
}

template <>
void launch_products<R97Q_BITS>(const Params& p, bool fwd, hipStream_t s) {
    const dim3 grid((unsigned)(p.ndown + p.nprod)), block(64 * kWaves);
    const int mt = tile_tokens(p.w.T) / 32;
#define R97Q_SM_LAUNCH(F, M) hipLaunchKernelGGL((sm_products_kernel<F, M>), grid, block, 0, s, p)
    if (fwd) {
        if (mt == 1) R97Q_SM_LAUNCH(true, 1);
        else if (mt == 2) R97Q_SM_LAUNCH(true, 2);
        else R97Q_SM_LAUNCH(true, 4);
    } else {
        if (mt == 1) R97Q_SM_LAUNCH(false, 1);
        else if (mt == 2) R97Q_SM_LAUNCH(false, 2);
        else R97Q_SM_LAUNCH(false, 4);
    }
#undef R97Q_SM_LAUNCH
}

}  // namespace sm
}  // namespace r97q
