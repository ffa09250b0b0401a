// gemv_any_multi.hip -- decode GEMV for several activation rows (up to 16 per pass) over tensors of other formats than plain OIL4
// (Qwen35Engine::gemm with small B, src/adapters/tools/qwen35_engine.cpp:47-85, over dequantize_block_all,
// src/block_codec.cpp:576-720): uniform SPARK_Q0, OIL2, OIL8 and grouped lattices, and the mixes of the planner (OIL1, SPARK_Q0) and
// of the registry (OIL1_GRP, OIL2_GRP, OIL4_GRP, OIL8_GRP).
//
// The products run on v_mfma_f32_16x16x32_f16 and are exact: an activation is scaled by a power of two per (token, block) and cut
// into three FP16 pieces (33 bits), which are three rows of the matrix instruction's A operand; a weight is an exact FP16 number
// times a factor that its block, or its group of 64, shares.  (A piece counts from the largest magnitude of its block: an outlier over a run whose scale is 0 costs
// the other runs bits.  SPARK_Q0 and OIL1, five rows, an outlier over a run of scale 0 in every block, error against 64 bits: of 1e5 1.1e-7, 1e6 5.6e-7, 1e8 7e-5;
// one to four rows, where gemv_signs serves them, 0.8e-7 throughout.)
//   SPARK_Q0, OIL1, OIL1_GRP   the weight itself (+- an FP16 scale, an FP16 mean)
//   OIL2, OIL2_GRP             10^4 times the level (15104, 4528)
//   OIL4_GRP                   10^4 / 256 times the level as a sum of two (signed bytes a and b / 256 of 256 a + b)
//   OIL8, OIL8_GRP             2 q - 255, q
// Sums are FP32; the factor and the power of two meet a block's or group's sum.  The zero points of grouped formats are
// one more matrix instruction (group sums of the activations, in three pieces, times the FP16 zero points).
// A wavefront takes every n-th block of the row for a run of 16-row groups, keeps the activations of its block in registers, and
// the wavefronts' sums meet in LDS once per run; every sum has a fixed order.  All but OIL8 are stored as
// window streams or sign tiles; a block is found through its descriptor, two steps ahead.  The pieces lie in a workspace of the caller's or in scratch of the
// stream; a call that is being captured without a workspace is left to the kernels that pack nothing.
//
// What bounds it: latency at two wavefronts per SIMD and the two launches where rows are short or few (planner's mix, 11008 x 4096, five rows: vector
// issue 27 %, matrix cores 7 %, memory 1.3 TB/s); the decode's vector instructions in the grouped formats (registry's mix 42 %); towards
// 16 rows and wide rows the activations' way into each compute unit (8 KB per block and five rows, once per workgroup).  Tried: shares of K for several workgroups of a range
// of rows, added by the last one, 10 to 20 % faster on the widest rows only and two to three times slower on others.
// Before (window-stream kernel in passes of up to four rows, OIL8 kernel likewise) -> now, pre-pass included:
//   16795 x 12032 SPARK_Q0, 15 rows 498 -> 53 us;  11008 x 4096 planner mix, 5 / 16 rows 26.7 / 70 -> 11.8 / 16.3 us;  OIL2, 8 rows 46.6 -> 15.8 us
//   6613 x 8192, registry mix, 9 rows 99.6 -> 40.6 us;  4096 x 4096 OIL8, 32 rows 87 -> 27.4 us;  649 x 768 planner mix, 5 rows 11.3 -> 5.5 us
// Other mixes of formats stay with the window-stream kernel, four rows at a time (11008 x 4096, 75 % OIL2 and 25 % OIL4, 8 rows 58 us).
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "level_digits.h"
#include "oil4_lds.h"
#include "pack_activations.h"

namespace oilhip {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x3 __attribute__((ext_vector_type(3)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxWaves = 8;
// tiles of 16 operand rows for M tokens of three pieces each
constexpr int tiles_for(int M) { return (3 * M + 15) / 16; }
constexpr int kPassTokens = 16;

// What the weights are: kOrderA formats have one factor per block at most, kOrderC formats one per group of 64 columns.
// Operand columns: step s of a block, lane group kq, element e is column 64 kq + 8 s + e (A), or 64 (s / 2) + 16 kq + 8 (s % 2) + e (C).
enum Source { kSpark = 0, kPlanner, kOil2, kOil8, kOil2Grp, kOil4Grp, kOil8Grp, kSparkMix };
constexpr bool grouped(int S) { return S >= kOil2Grp; }
constexpr bool by_descriptor(int S) { return S != kOil8; }                 // stored as window streams or sign tiles (common.h)
constexpr int steps_of(int S) { return grouped(S) ? 9 : 8; }               // the ninth: group sums
__host__ __device__ constexpr uint32_t tile_bytes(bool grp) { return (grp ? 9u : 8u) * 1024u; }

// ---- pre-pass --------------------------------------------------------------------------------------------------------
struct PackArgs {
    Activations in;
    uint8_t* xp;            // powers of two [block][16 NT] floats, one block of zeros, then the operands [block][tile][step][lane][8 halves]
    uint32_t bpr, tiles, grp;
    int M;
};

__global__ void __launch_bounds__(256)
pack_pieces_kernel(const PackArgs a) {
    // (all arguments at once: read where they are needed, each adds a scalar load's latency)
    asm volatile("" :: "s"(a.in.x), "s"(a.in.x2), "s"(a.in.norm_w), "s"(a.in.ldx), "s"(a.in.aligned), "s"(a.xp), "s"(a.bpr), "s"(a.tiles), "s"(a.grp), "s"(a.M));
    const uint32_t lane = threadIdx.x & 63u, blk = blockIdx.x, t = blockIdx.y * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t rows = 16u * a.tiles;
    if (3u * t >= rows) return;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if ((int)t < a.M) load_activations(a.in, t, blk, a.bpr, lane, v);
    // the largest magnitude as a bit pattern: infinities and NaN are the largest of all
    uint32_t top = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) top = max(top, __float_as_uint(v[e]) & 0x7FFFFFFFu);
    auto dpp = [&](auto ctrl) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, decltype(ctrl)::value, 0xF, 0xF, true); };
    using std::integral_constant;
    top = max(top, dpp(integral_constant<int, 0xB1>{}));                   // quad_perm [1,0,3,2]
    top = max(top, dpp(integral_constant<int, 0x4E>{}));                   // [2,3,0,1]
    top = max(top, dpp(integral_constant<int, 0x141>{}));                  // row_half_mirror
    top = max(top, dpp(integral_constant<int, 0x140>{}));                  // row_mirror
    top = max(max((uint32_t)__builtin_amdgcn_readlane((int)top, 0), (uint32_t)__builtin_amdgcn_readlane((int)top, 16)),
              max((uint32_t)__builtin_amdgcn_readlane((int)top, 32), (uint32_t)__builtin_amdgcn_readlane((int)top, 48)));
    const bool bad = top >= 0x7F800000u;
    int ex = top == 0u || bad ? 0 : 14 - ((int)(top >> 23) - 127);         // to [2^14, 2^15)
    ex = ex > 140 ? 140 : ex;
    _Float16 h[3][4];
    float sum = 0.0f;
    auto cut = [](float f, _Float16& h0, _Float16& h1, _Float16& h2) {
        h0 = (_Float16)f;
        const float r = f - (float)h0;
        h1 = (_Float16)r;
        h2 = (_Float16)(r - (float)h1);
    };
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float f = bad ? 0.0f : ldexpf(v[e], ex);
        sum += f;
        cut(f, h[0][e], h[1][e], h[2][e]);
    }
    float undo[3];
    undo[0] = undo[1] = undo[2] = bad ? __uint_as_float(0x7FC00000u) : ldexpf(1.0f, -ex);
    uint32_t step, kq;
    if (a.grp) { step = 2u * (lane >> 4) + ((lane & 3u) >> 1); kq = (lane & 15u) >> 2; }
    else { step = (lane & 15u) >> 1; kq = lane >> 4; }
    uint8_t* base = a.xp + (a.bpr + 1u) * rows * 4u + (size_t)blk * a.tiles * tile_bytes(a.grp);
    sum += oil4::dpp_quad_xor1(sum);
    sum += oil4::dpp_quad_xor2(sum);
    sum += oil4::dpp_half_mirror(sum);
    sum += oil4::dpp_row_mirror(sum);                                       // of the lane's group of 64 columns: below 2^21
    _Float16 g[3];
    cut(sum * 0x1p-6f, g[0], g[1], g[2]);
    if (top == 0x7F800000u) {                                              // infinities, no NaN (uniform)
        // Up to three of them: each is +-1 in a piece of its own, the rest of the block 0, and the piece's power of two is
        // infinity, so that an output gets the infinity with its weight's sign (NaN of a zero weight), as in FP32.  More: NaN.
        uint32_t before = 0;
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) {
            const bool here = (__float_as_uint(v[e]) & 0x7FFFFFFFu) == 0x7F800000u;
            const uint64_t m = __ballot(here);
            const uint32_t rank = before + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
#pragma unroll
            for (uint32_t d = 0; d < 3u; ++d) h[d][e] = here && rank == d ? (_Float16)(v[e] > 0.0f ? 1.0f : -1.0f) : (_Float16)0.0f;
            before += (uint32_t)__popcll(m);
        }
#pragma unroll
        for (uint32_t d = 0; d < 3u; ++d) {
            if (before <= 3u) undo[d] = d < before ? __builtin_inff() : 1.0f;
            float s = ((float)h[d][0] + (float)h[d][1]) + ((float)h[d][2] + (float)h[d][3]);
            s += oil4::dpp_quad_xor1(s);
            s += oil4::dpp_quad_xor2(s);
            s += oil4::dpp_half_mirror(s);
            s += oil4::dpp_row_mirror(s);
            g[d] = (_Float16)(s * 0x1p-6f);
        }
    }
#pragma unroll
    for (uint32_t d = 0; d < 3u; ++d) {
        const uint32_t r = 3u * t + d;
        if (r >= rows) break;
        uint8_t* tile = base + (r >> 4) * tile_bytes(a.grp);
        const f16x2 lo = f16x2{h[d][0], h[d][1]}, hi = f16x2{h[d][2], h[d][3]};
        *reinterpret_cast<uint2*>(tile + (step * 64u + kq * 16u + (r & 15u)) * 16u + (lane & 1u) * 8u) =
            make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
        if (a.grp && (lane & 15u) == 0u) {                                  // group lane / 16 at lane group lane / 16, element 0
            const f16x2 s = f16x2{g[d], (_Float16)0.0f};
            *reinterpret_cast<uint4*>(tile + (8u * 64u + (lane >> 4) * 16u + (r & 15u)) * 16u) = make_uint4(__builtin_bit_cast(uint32_t, s), 0u, 0u, 0u);
        }
        if (lane == 0) {
            reinterpret_cast<float*>(a.xp)[blk * rows + r] = undo[d];
            if (blk == 0) reinterpret_cast<float*>(a.xp)[a.bpr * rows + r] = 0.0f;
        }
    }
}

// ---- weights ---------------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t pair16(uint32_t h) { return __builtin_amdgcn_perm(h, h, 0x01000100u); }   // the low half twice
__device__ __forceinline__ uint32_t pk_add(uint32_t a, _Float16 b) {
    const f16x2 r = __builtin_bit_cast(f16x2, a) + f16x2{b, b};
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint32_t pk_fma(uint32_t a, _Float16 b, _Float16 c) {
    const f16x2 r = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, a), f16x2{b, b}, f16x2{c, c});
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ f16x8 eight(uint32_t a, uint32_t b, uint32_t c, uint32_t d) { return __builtin_bit_cast(f16x8, u32x4{a, b, c, d}); }

// bits 0..7 of b: set -> +scale, clear -> -scale; minus = the scale's halves with their signs flipped
__device__ __forceinline__ f16x8 signs(uint32_t b, uint32_t minus) {
    uint32_t t = b | (b << 15);                                             // bit 2 d at 2 d, bit 2 d + 1 at 2 d + 16
    asm("" : "+v"(t));                                                     // shifts below, not 32-bit multiplications of b
    return eight(((t << 15) & 0x80008000u) ^ minus, ((t << 13) & 0x80008000u) ^ minus, ((t << 11) & 0x80008000u) ^ minus,
                 ((t << 9) & 0x80008000u) ^ minus);
}
// eight 2-bit codes -> 10^4 times their levels (-15104, -4528, 4528, 15104)
__device__ __forceinline__ f16x8 levels2(uint32_t c) {
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        uint32_t t = (c >> (8 * i)) & 0xFFu;
        t |= t << 6;
        t = (t | (t << 12)) & 0x03030303u;
        const uint32_t hi = __builtin_amdgcn_perm(0u, 0x736CECF3u, t), lo = __builtin_amdgcn_perm(0u, 0x606C6C60u, t);
        d[2 * i] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
        d[2 * i + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
    }
    return eight(d[0], d[1], d[2], d[3]);
}
// four bytes -> 1024 + byte as FP16, two per dword
__device__ __forceinline__ void widen(uint32_t b, uint32_t& d0, uint32_t& d1) {
    d0 = __builtin_amdgcn_perm(0x64646464u, b, 0x04010400u);
    d1 = __builtin_amdgcn_perm(0x64646464u, b, 0x04030402u);
}
// eight bytes q -> 2 q - 255 (centred) or q
template <bool CENTRED>
__device__ __forceinline__ f16x8 bytes8(uint32_t b0, uint32_t b1) {
    uint32_t d[4];
    widen(b0, d[0], d[1]);
    widen(b1, d[2], d[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (CENTRED) d[i] = pk_fma(pk_add(d[i], (_Float16)-1151.0f), (_Float16)2.0f, (_Float16)-1.0f);
        else d[i] = pk_add(d[i], (_Float16)-1024.0f);
    }
    return eight(d[0], d[1], d[2], d[3]);
}

// eight 4-bit codes of c -> the two summands
__device__ __forceinline__ void levels4(uint32_t c, f16x8& va, f16x8& vb) {
    uint32_t ae, be, ao, bo, d[8];
    level_digits(c, ae, be);                                                    // codes 0, 2, 4, 6
    level_digits(c >> 4, ao, bo);                                              // codes 1, 3, 5, 7
    // bytes to code order, then to FP16: 1024 + (digit + 128)
    const uint32_t a0 = __builtin_amdgcn_perm(ao, ae, 0x05010400u) ^ 0x80808080u, a1 = __builtin_amdgcn_perm(ao, ae, 0x07030602u) ^ 0x80808080u;
    const uint32_t b0 = __builtin_amdgcn_perm(bo, be, 0x05010400u) ^ 0x80808080u, b1 = __builtin_amdgcn_perm(bo, be, 0x07030602u) ^ 0x80808080u;
    widen(a0, d[0], d[1]);
    widen(a1, d[2], d[3]);
    widen(b0, d[4], d[5]);
    widen(b1, d[6], d[7]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        d[i] = pk_add(d[i], (_Float16)-1152.0f);
        d[4 + i] = pk_fma(d[4 + i], (_Float16)0x1p-8f, (_Float16)-4.5f);
    }
    va = eight(d[0], d[1], d[2], d[3]);
    vb = eight(d[4], d[5], d[6], d[7]);
}

// dwords of a block that a lane holds
constexpr int raw_dwords(int S) {
    return S == kSpark || S == kPlanner ? 3 : S == kOil2 ? 6 : S == kOil8 ? 18 : S == kOil2Grp ? 5 : S == kOil4Grp ? 9 : 17;
}
__host__ __device__ constexpr uint32_t block_bytes(int S) { return S == kSpark ? 48u : S == kOil2 ? 64u : S == kOil8 ? 256u : S == kOil2Grp ? 80u : S == kOil4Grp ? 144u : 272u; }
// row groups of a run, at most: as many as registers and LDS take
constexpr int run_groups(int S, int NT) { return NT == 3 && grouped(S) ? 1 : NT > 1 || raw_dwords(S) > 6 ? 2 : 4; }
// blocks of activations that a wavefront holds
constexpr int x_slots(int S, int NT) { return NT == 1 ? (grouped(S) || raw_dwords(S) > 9 ? 2 : 3) : 1; }

struct BodyArgs {
    const uint8_t* W;
    const DevBlock* blocks;        // by_descriptor
    const uint8_t* xp;
    float* y;
    uint32_t wbytes;               // size of the payload (by_descriptor)
    uint32_t rows, bpr, ldy, parts, part_blocks, chunk, g_base, g_rem;
    int M;
};

template <int S, int NT, int G>
__global__ void __launch_bounds__(64 * kMaxWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemv_any_multi_kernel(const BodyArgs a) {
    constexpr int XD = x_slots(S, NT), ST = steps_of(S), N = raw_dwords(S), ROWS = 16 * NT;
    extern __shared__ __align__(16) float red[];
    const uint32_t wgid = blockIdx.x, g_begin = wgid * a.g_base + (wgid < a.g_rem ? wgid : a.g_rem), g_end = g_begin + a.g_base + (wgid < a.g_rem ? 1u : 0u);
    const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), waves = blockDim.x >> 6;
    const uint32_t li = lane & 15u, kq = lane >> 4, bpr = a.bpr;
    const uint32_t iters = (a.part_blocks + waves - 1u) / waves;
    const uint32_t stride = block_bytes(S), row_bytes = bpr * stride;
    const uint32_t last = a.rows - 1u - 16u * g_begin, ngroups = g_end - g_begin;      // rows past the end repeat the last one
    const auto wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(by_descriptor(S) ? a.W : a.W + (size_t)g_begin * 16u * row_bytes), (short)0,
                                                       (int)(by_descriptor(S) ? a.wbytes : 0xFFFFFFFFu), 0x00020000);
    const auto drs = __builtin_amdgcn_make_buffer_rsrc(const_cast<DevBlock*>(by_descriptor(S) ? a.blocks + (size_t)g_begin * 16u * bpr : nullptr), (short)0,
                                                       (int)0xFFFFFFFFu, 0x00020000);
    const float* undo = reinterpret_cast<const float*>(a.xp);
    const uint8_t* xblocks = a.xp + (bpr + 1u) * ROWS * 4u;
    auto place = [&](uint32_t part, uint32_t i) { const uint32_t b = wave + i * waves; return b < a.part_blocks ? part * a.part_blocks + b : 0xFFFFFFFFu; };
    auto block_at = [&](uint32_t part, uint32_t i) { const uint32_t b = place(part, i); return b < bpr ? b : bpr - 1u; };

    uint32_t w[G][N];
    uint32_t fmt[G], dnext[G], fnext[G];                                   // by_descriptor: format of w; place and format of the step after
    auto load_desc = [&](int g, uint32_t part, uint32_t run, uint32_t i) {
        if constexpr (by_descriptor(S)) {
            uint32_t r = (run + (uint32_t)g) * 16u + li;
            r = r < last ? r : last;
            const u32x4 d = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(drs, r * bpr * 16u, block_at(part, i) * 16u, 0));
            dnext[g] = d.x * 16u;
            fnext[g] = (d.w >> 16) & 0xFFu;
        }
    };
    auto b32 = [&](uint32_t off, uint32_t so) { return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(wrs, off, so, 0); };
    auto load_w = [&](int g, uint32_t part, uint32_t run, uint32_t i) {
        uint32_t (&o)[N] = w[g];
        uint32_t r = (run + (uint32_t)g) * 16u + li;
        r = r < last ? r : last;
        const uint32_t off = by_descriptor(S) ? dnext[g] : r * row_bytes, so = by_descriptor(S) ? 0u : block_at(part, i) * stride;
        if constexpr (by_descriptor(S)) fmt[g] = fnext[g];
        auto group_loads = [&](auto bits) {
            constexpr uint32_t B = decltype(bits)::value, GB = 4u + 8u * B, Q = B / 2u;
            o[0] = b32(off + kq * GB, so);                                 // zero point and scale of group kq
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) {
                const uint32_t at = off + j * GB + 4u + 2u * B * kq;
                if constexpr (B == 2u) o[1 + Q * j] = b32(at, so);
                if constexpr (B == 4u) { const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(wrs, at, so, 0)); o[1 + Q * j] = v.x; o[2 + Q * j] = v.y; }
                if constexpr (B == 8u) { const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs, at, so, 0)); o[1 + Q * j] = v.x; o[2 + Q * j] = v.y; o[3 + Q * j] = v.z; o[4 + Q * j] = v.w; }
            }
        };
        if constexpr (S == kSpark || S == kPlanner) {                      // runs 2 kq and 2 kq + 1: 12 bytes, or (OIL1) 4
            const uint32_t at = S == kPlanner && fmt[g] != 1u ? 4u : 12u;
            const u32x3 v = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(wrs, off + at * kq, so, 0));
            o[0] = v.x; o[1] = v.y; o[2] = v.z;
        } else if constexpr (S == kOil2) {                                 // 124 bits from bit 16 + 124 kq; the scale
            const uint32_t at = off + ((16u + 124u * kq) >> 5) * 4u;
            const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs, at, so, 0));
            o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
            o[4] = kq < 3u ? b32(at + 16u, so) : 0u;
            o[5] = b32(off, so);
        } else if constexpr (S == kOil8) {                                 // bytes 64 kq .. 64 kq + 67; the scale
#pragma unroll
            for (uint32_t j = 0; j < 4u; ++j) {
                const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs, off + 64u * kq + 16u * j, so, 0));
                o[4 * j] = v.x; o[4 * j + 1] = v.y; o[4 * j + 2] = v.z; o[4 * j + 3] = v.w;
            }
            o[16] = kq < 3u ? b32(off + 64u * kq + 64u, so) : 0u;
            o[17] = b32(off, so);
        } else if constexpr (S == kOil2Grp) {
            group_loads(std::integral_constant<uint32_t, 2u>{});
        } else if constexpr (S == kOil4Grp) {
            group_loads(std::integral_constant<uint32_t, 4u>{});
        } else if constexpr (S == kOil8Grp) {
            group_loads(std::integral_constant<uint32_t, 8u>{});
        } else {
            // four 16-byte places of which a format fills what it has
            auto b64 = [&](uint32_t at) { const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(wrs, at, so, 0)); return u32x4{v.x, v.y, 0u, 0u}; };
            auto b128 = [&](uint32_t at) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs, at, so, 0)); };
            u32x4 q0 = {0u, 0u, 0u, 0u}, q1 = q0, q2 = q0, q3 = q0;
            const uint32_t f = fmt[g];
            const uint32_t header = f == 7u ? 0u : (f == 9u ? 20u : f == 10u ? 36u : 68u) * kq;
            const uint32_t hdr = b32(off + header, so);
            if (f == 9u) {
                const uint32_t at = off + 4u + 4u * kq;
                q0.x = b32(at, so); q1.x = b32(at + 20u, so); q2.x = b32(at + 40u, so); q3.x = b32(at + 60u, so);
            } else if (f == 7u) {                                          // all 32 bytes
                q0 = b128(off); q1 = b128(off + 16u);
            } else if (f == 10u) {
                const uint32_t at = off + 4u + 8u * kq;
                q0 = b64(at); q1 = b64(at + 36u); q2 = b64(at + 72u); q3 = b64(at + 108u);
            } else {
                const uint32_t at = off + 4u + 16u * kq;
                q0 = b128(at); q1 = b128(at + 68u); q2 = b128(at + 136u); q3 = b128(at + 204u);
            }
            o[0] = hdr;
#pragma unroll
            for (int k = 0; k < 4; ++k) { o[1 + k] = q0[k]; o[5 + k] = q1[k]; o[9 + k] = q2[k]; o[13 + k] = q3[k]; }
        }
    };
    f16x8 x[XD][NT][ST];
    f32x4 un[XD][NT];
    auto load_part = [&](uint32_t part) {
#pragma unroll
        for (int s = 0; s < XD; ++s)
            if (s == 0 || (uint32_t)s < iters) {
                // a wavefront that has a block less than the others takes the last one again, times 0
                const uint32_t blk = block_at(part, (uint32_t)s), scale_of = place(part, (uint32_t)s) < bpr ? blk : bpr;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const f16x8* p = reinterpret_cast<const f16x8*>(xblocks + ((size_t)blk * NT + (uint32_t)t) * tile_bytes(grouped(S))) + lane;
#pragma unroll
                    for (int k = 0; k < ST; ++k) x[s][t][k] = p[64 * k];
                    un[s][t] = *reinterpret_cast<const f32x4*>(undo + scale_of * ROWS + 16u * (uint32_t)t + 4u * kq);
                }
            }
    };
    float acc[G][NT][4];
    // The sums of a chain of matrix instructions, before anything reads them.  A result must not be read for 8 wait states, which the
    // hardware does not enforce and the compiler leaves; but where a branch follows the last instruction of a chain, the
    // compiler counts the wait states of the code that falls through, and a read at the branch's target came one wait state behind
    // the instruction: the sums lacked its products.  So a chain ends with its wait states, in front of any branch.
    auto settle = [](f32x4& v) { asm volatile("s_nop 7" : "+v"(v)); };
    // One block of 16 rows into acc[g].  The weights' factor meets the sum before the power of two does, so that no partial sum is
    // larger than it would be in FP32.
    auto multiply = [&](int xs, int g) {
        const uint32_t (&o)[N] = w[g];
        f32x4 sum[NT];
        if constexpr (!grouped(S)) {
            const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
            float factor = 1.0f;
            // Several chains, whose sums meet afterwards: an instruction rounds its sums four times, one after the other (eight products of a
            // lane group at a time), so one chain of eight rounds 32 times.  SPARK_Q0, 4096 columns, 16 rows, error against 64 bits with 1 / 2 / 4
            // chains: 12.2e-8 / 10.1e-8 / 9.3e-8 (one row at a time in FP32: 10.7e-8).
            constexpr int CH = NT == 3 && S == kOil8 ? 2 : 4;              // (as many as the registers take)
            f32x4 chain[NT][CH];
            uint32_t minus[2], bits[2], c[16];
            if constexpr (S == kSpark || S == kPlanner) {
                const bool spark = S == kSpark || fmt[g] == 1u;
                minus[0] = pair16(o[0]) ^ 0x80008000u;
                minus[1] = pair16((spark ? o[1] : o[0]) >> 16) ^ 0x80008000u;
                bits[0] = spark ? __builtin_amdgcn_alignbit(o[1], o[0], 16) : 0xFFFFFFFFu;
                bits[1] = spark ? o[2] : 0xFFFFFFFFu;
            } else if constexpr (S == kOil2) {
                factor = __half2float(__ushort_as_half((unsigned short)o[5])) * 1e-4f;
                const uint32_t sh = 16u - 4u * kq;
#pragma unroll
                for (int j = 0; j < 4; ++j) c[j] = __builtin_amdgcn_alignbit(o[j + 1], o[j], sh);
            } else {
                factor = __half2float(__ushort_as_half((unsigned short)o[17])) * (8.0f / 255.0f);
                const uint32_t sh = kq < 2u ? 2u : 1u;
#pragma unroll
                for (int j = 0; j < 16; ++j) c[j] = __builtin_amdgcn_alignbyte(o[j + 1], o[j], sh);
            }
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                f16x8 v;
                if constexpr (S == kSpark || S == kPlanner) {
                    v = signs((bits[s >> 2] >> (8 * (s & 3))) & 0xFFu, minus[s >> 2]);
                } else if constexpr (S == kOil2) {                         // columns 31 and 63 of the lane are slots: 31 codes a run
                    const int at = 62 * (s >> 2) + 16 * (s & 3);
                    uint32_t q = at % 32 == 0 ? c[at / 32] : __builtin_amdgcn_alignbit(at / 32 + 1 < 4 ? c[at / 32 + 1] : 0u, c[at / 32], at % 32);
                    v = levels2(q & 0xFFFFu);
                    if ((s & 3) == 3) v[7] = (_Float16)0.0f;
                } else {
                    v = bytes8<true>(c[2 * s], c[2 * s + 1]);
                    if (s == 7) v[7] = (kq & 1u) ? (_Float16)0.0f : v[7];  // columns 127 and 255 are slots
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) chain[t][s * CH / 8] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[xs][t][s], v, s % (8 / CH) ? chain[t][s * CH / 8] : zero, 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
#pragma unroll
                for (int c = 0; c < CH; ++c) settle(chain[t][c]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sum[t][e] = chain[t][0][e] + chain[t][1][e];
                    if constexpr (CH == 4) sum[t][e] += chain[t][2][e] + chain[t][3][e];
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[g][t][e] = fmaf(sum[t][e] * factor, un[xs][t][e], acc[g][t][e]);
        } else {
            // zero point and scale of group kq, this lane's row (the group sums are packed divided by 64)
            const bool own = S != kSparkMix || fmt[g] != 7u;
            float sc = __half2float(__ushort_as_half((unsigned short)(o[0] >> 16)));
            const float unit = S == kOil2Grp ? 1e-4f : S == kOil4Grp ? 256e-4f : S == kOil8Grp ? 1.0f / 255.0f
                             : fmt[g] == 9u ? 1e-4f : fmt[g] == 10u ? 256e-4f : 1.0f / 255.0f;
            sc = own ? sc * unit : 1.0f;
            const uint32_t zbits = own ? o[0] & 0xFFFFu : 0u;
            const f16x8 zv = eight(zbits, 0u, 0u, 0u);
            float factor[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) factor[j] = __int_as_float(__builtin_amdgcn_ds_bpermute((int)((li + 16u * (uint32_t)j) * 4u), __float_as_int(sc)));
            const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[xs][t][8], zv, zero, 0, 0, 0);
                settle(sum[t]);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[t][e] *= 64.0f;
            }
            const uint32_t minus = S == kSparkMix ? pair16(o[1]) ^ 0x80008000u : 0u;      // OIL1_GRP: the scale
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f32x4 part[NT];
                f16x8 vs[2], vs2[2];                                       // both halves first: their decoding may branch
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    f16x8 v, v2 = eight(0u, 0u, 0u, 0u);
                    if constexpr (S == kOil2Grp) {
                        v = levels2((o[1 + j] >> (16 * h)) & 0xFFFFu);
                    } else if constexpr (S == kOil4Grp) {
                        levels4(o[1 + 2 * j + h], v, v2);
                    } else if constexpr (S == kOil8Grp) {
                        v = bytes8<false>(o[1 + 4 * j + 2 * h], o[2 + 4 * j + 2 * h]);
                    } else {
                        v = levels2((o[1 + 4 * j] >> (16 * h)) & 0xFFFFu);
                        if (fmt[g] == 7u) {                                // 15 bits from 16 + 15 (4 j + kq)
                            const int d = (16 + 60 * j) / 32, r = (16 + 60 * j) % 32;
                            const uint64_t lo = o[1 + d] | (uint64_t)o[2 + d] << 32;
                            const uint64_t win = (lo >> r) | (r ? (uint64_t)(d + 2 < 8 ? o[3 + d] : 0u) << (64 - r) : 0ull);
                            const uint32_t b = (uint32_t)(win >> (15u * kq)) & 0x7FFFu;
                            v = signs((b >> (8 * h)) & 0xFFu, minus);
                            if (h == 1) v[7] = (_Float16)0.0f;
                        } else if (fmt[g] == 10u) {
                            levels4(o[1 + 4 * j + h], v, v2);
                        } else if (fmt[g] == 11u) {
                            v = bytes8<false>(o[1 + 4 * j + 2 * h], o[2 + 4 * j + 2 * h]);
                        }
                    }
                    vs[h] = v;
                    vs2[h] = v2;
                }
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        part[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[xs][t][2 * j + h], vs[h], h ? part[t] : zero, 0, 0, 0);
                        if constexpr (S == kOil4Grp || S == kSparkMix) part[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[xs][t][2 * j + h], vs2[h], part[t], 0, 0, 0);
                    }
#pragma unroll
                for (int t = 0; t < NT; ++t) settle(part[t]);
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[t][e] = fmaf(part[t][e], factor[j], sum[t][e]);
                __builtin_amdgcn_sched_barrier(0);                         // one group's weights in registers at a time
            }
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[g][t][e] = fmaf(sum[t][e], un[xs][t][e], acc[g][t][e]);
        }
    };
    auto lds_barrier = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    constexpr uint32_t OUT = (uint32_t)(G * NT * 4) * 64u, AREA = (uint32_t)kMaxWaves * OUT;
    float* keep = red + 2u * AREA;
    if (waves < (uint32_t)kMaxWaves)
        for (uint32_t o = waves * OUT + threadIdx.x; o < AREA; o += blockDim.x) { red[o] = 0.0f; red[AREA + o] = 0.0f; }
    // outputs of a run: the eight wavefronts' sums of a token's three pieces (in 64 bits for the formats that gemv_signs serves one row of: its sums are of whole
    // numbers, and several rows are to be no less accurate than one)
    using Sum = std::conditional_t<S == kSpark || S == kPlanner, double, float>;
    auto finish = [&](uint32_t part, uint32_t run, const float* area) {
        for (uint32_t o = threadIdx.x; o < (uint32_t)(G * 16) * (uint32_t)a.M; o += blockDim.x) {
            const uint32_t l = o & 15u, g = (o >> 4) % G, token = (o >> 4) / G;
            Sum sum = 0;
#pragma unroll
            for (uint32_t d = 0; d < 3u; ++d) {
                const uint32_t q = 3u * token + d;
                const float* p = area + ((g * NT + (q >> 4)) * 4u + (q & 3u)) * 64u + ((q >> 2) & 3u) * 16u + l;
                sum += (((Sum)p[0] + (Sum)p[OUT]) + ((Sum)p[2u * OUT] + (Sum)p[3u * OUT])) + (((Sum)p[4u * OUT] + (Sum)p[5u * OUT]) + ((Sum)p[6u * OUT] + (Sum)p[7u * OUT]));
            }
            float s = (float)sum;
            float* k = keep + ((run % a.chunk) / G) * (uint32_t)(G * 16 * kPassTokens) + o;
            if (part) s += *k;
            if (part + 1u < a.parts) { *k = s; continue; }
            const uint32_t r = (g_begin + run + g) * 16u + l;
            if (run + g < ngroups && r < a.rows) a.y[(size_t)token * a.ldy + r] = s;
        }
    };
    // the step after (part, run, i)
    uint32_t chunk_begin = 0, chunk_end = a.chunk < ngroups ? a.chunk : ngroups;
    struct At { uint32_t part, run, i, cb, ce; };
    auto after = [&](At p) {                                               // selects: the walk is on the way of every step
        const bool turn = p.i + 1u >= iters, done = turn & (p.run + G >= p.ce), over = done & (p.part + 1u >= a.parts);
        const uint32_t cb = over ? (p.ce < ngroups ? p.ce : 0u) : p.cb, far = cb + a.chunk < ngroups ? cb + a.chunk : ngroups;
        return At{over ? 0u : done ? p.part + 1u : p.part, done ? cb : turn ? p.run + G : p.run, turn ? 0u : p.i + 1u, cb, over ? far : p.ce};
    };
    load_part(0u);
    At here{0u, 0u, 0u, chunk_begin, chunk_end}, next = after(here), then = after(next);
#pragma unroll
    for (int g = 0; g < G; ++g) load_desc(g, 0u, 0u, 0u);
#pragma unroll
    for (int g = 0; g < G; ++g) { load_w(g, 0u, 0u, 0u); load_desc(g, next.part, next.run, next.i); }
    uint32_t odd = 0, done_part = 0, done_run = 0xFFFFFFFFu;
    for (; chunk_begin < ngroups; chunk_begin = chunk_end, chunk_end = chunk_end + a.chunk < ngroups ? chunk_end + a.chunk : ngroups)
    for (uint32_t part = 0; part < a.parts; ++part) {
        if (a.parts > 1u && (part || chunk_begin)) load_part(part);
        for (uint32_t run = chunk_begin; run < chunk_end; run += G) {
            if (done_run != 0xFFFFFFFFu) finish(done_part, done_run, red + (odd ^ 1u) * AREA);
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[g][t][e] = 0.0f;
#pragma unroll
            for (int i = 0; i < XD; ++i)
                if (i == 0 || (uint32_t)i < iters) {
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        multiply(i, g);
                        load_w(g, next.part, next.run, next.i);
                        load_desc(g, then.part, then.run, then.i);
                    }
                    next = then;
                    then = after(then);
                }
            float* area = red + odd * AREA + wave * OUT;
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) area[(uint32_t)((g * NT + t) * 4 + e) * 64u + lane] = acc[g][t][e];
            lds_barrier();
            odd ^= 1u;
            done_part = part; done_run = run;
        }
    }
    finish(done_part, done_run, red + (odd ^ 1u) * AREA);
}

constexpr uint32_t kKeepGroups = 48;                                       // groups whose sums wait in LDS between parts: a multiple of every run length

template <int S, int NT, int G>
int launch_run(const BodyArgs& a, uint32_t wgs, uint32_t waves, hipStream_t s) {
    const size_t lds = (size_t)2u * kMaxWaves * G * NT * 1024u + (a.parts > 1u ? (size_t)kKeepGroups * 16u * kPassTokens * 4u : 0u);
    static std::atomic<uint64_t> raised{0};
    auto kern = gemv_any_multi_kernel<S, NT, G>;
    if (int rc = ensure_max_lds(raised, (const void*)kern, 160 * 1024)) return rc;
    hipLaunchKernelGGL(kern, dim3(wgs), dim3(64u * waves), lds, s, a);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

template <int S, int NT>
int launch_one(BodyArgs a, hipStream_t s) {
    constexpr int G = run_groups(S, NT), XD = x_slots(S, NT);
    const uint32_t most = (uint32_t)(kMaxWaves * XD);
    a.parts = (a.bpr + most - 1u) / most;
    a.part_blocks = (a.bpr + a.parts - 1u) / a.parts;
    a.parts = (a.bpr + a.part_blocks - 1u) / a.part_blocks;
    const uint32_t each = (a.part_blocks + kMaxWaves - 1u) / kMaxWaves, waves = (a.part_blocks + each - 1u) / each;
    a.chunk = a.parts > 1u ? kKeepGroups : 0x7FFFFFFFu;
    const uint32_t groups = (a.rows + 15u) / 16u, slots = (uint32_t)device_cu_count() * std::max(1u, (uint32_t)kMaxWaves / waves);
    const uint32_t wgs = std::min(groups, slots);
    a.g_base = groups / wgs;
    a.g_rem = groups % wgs;
    // The longest run that divides the fullest workgroup's groups: a run that is not full costs as much as a full one (5120 x 4096,
    // 4 rows, runs of 1 / 2 / 4 for 2 groups: SPARK_Q0 9.9 / 9.7 / 12.7 us, OIL2_GRP 12.4 / 12.7 / 18.7; 11008 x 4096, 3 groups: OIL2 14.9 / 16.8 /
    // 18.5, the registry's mix 28.2 / 34.0; 16384 x 4096, 4 groups: SPARK_Q0 14.5 / 13.2 / 13.4).
    const uint32_t most_groups = a.g_base + (a.g_rem ? 1u : 0u);
    if constexpr (G > 2)
        if (most_groups % (uint32_t)G == 0u) return launch_run<S, NT, G>(a, wgs, waves, s);
    if constexpr (G > 1)
        if (most_groups % 2u == 0u) return launch_run<S, NT, 2>(a, wgs, waves, s);
    return launch_run<S, NT, 1>(a, wgs, waves, s);
}

template <int S>
int launch_tiles(int tiles, const BodyArgs& a, hipStream_t s) {
    return tiles == 1 ? launch_one<S, 1>(a, s) : tiles == 2 ? launch_one<S, 2>(a, s) : launch_one<S, 3>(a, s);
}

int source_of(const oilhip_weights& w) {
    if (w.seg.by_descriptor()) {
        uint32_t formats = 0;
        for (uint32_t i = 0; i < w.seg.nf; ++i) {
            if (w.seg.cb_bytes[i] != full_block_cb_bytes((int)w.seg.fmt[i]) || w.seg.cb_bytes[i] + w.seg.idx_bytes[i] != full_block_bytes((int)w.seg.fmt[i])) return -1;
            formats |= 1u << w.seg.fmt[i];
        }
        if (w.alloc_bytes >= 0xFFFFFFF0ull) return -1;                     // 32-bit offsets
        switch (formats) {
            case 1u << OILHIP_SPARK_Q0: return kSpark;
            case 1u << OILHIP_OIL2: return kOil2;
            case 1u << OILHIP_OIL2_GRP: return kOil2Grp;
            case 1u << OILHIP_OIL4_GRP: return kOil4Grp;
            case 1u << OILHIP_OIL8_GRP: return kOil8Grp;
        }
        if ((formats & ~(1u << OILHIP_OIL1 | 1u << OILHIP_SPARK_Q0)) == 0) return kPlanner;
        if ((formats & ~(1u << OILHIP_OIL1_GRP | 1u << OILHIP_OIL2_GRP | 1u << OILHIP_OIL4_GRP | 1u << OILHIP_OIL8_GRP)) == 0) return kSparkMix;
        return -1;
    }
    return w.uniform_fmt == OILHIP_OIL8 && w.uniform_stride == 256u && w.uniform_cb == 0 && w.uniform_idx == 256u && (w.uniform_base & 3u) == 0 ? kOil8 : -1;
}

// Whether two to four rows (OIL8: to eight) are faster here than through the kernels of up to four rows per pass (window streams: two where
// four rows of activations do not fit their LDS).  From 36 shapes of 0.26 to 123 M weights per format, all timed both ways; "M weights" are
// millions.
bool faster_than_row_kernels(int src, const oilhip_weights& w, int M) {
    const uint64_t weights = w.rows * w.cols;
    const bool light = src == kSpark || src == kPlanner;
    if (src == kOil8) return M <= 4 ? weights >= 12000000u : M > 2 && weights >= 2000000u;
    // Two rows: tall tensors, which are packed for one row at a time, and of these the formats whose error is no larger here (as window streams; stored as
    // sign tiles they come here only with outputs that lie over the activations: 11008 x 4096
    // SPARK_Q0 16.5 against 12.3 us, planner's mix 12.0 against 12.4; 22016 x 4096 24 against 13, 19 against 15).
    if (M == 2) return light && w.seg.waves == 16;
    // Three and four: SPARK_Q0 and the planner's mix always (1000 x 2048, 3 rows 7.2 against 6.1 us, 4096 x 11008, 4 rows 43 against 14).
    if (light || w.seg.waves == 16) return true;
    // Heavier decoding needs a full chip.  Workgroups of which few have a second group: 5120 x 4096, 3 rows OIL4_GRP 15.8 against 16.7 us,
    // registry's mix 18.9 against 20.8; 6144 x 2048 OIL2_GRP 10.1 against 11.2; 7000 x 3072 14.0 against 11.4.
    const uint64_t groups = (w.rows + 15u) / 16u, cus = (uint64_t)device_cu_count();
    if (grouped(src) && w.cols <= 5120u && groups > cus && groups * 5u < cus * 8u) return false;
    // Rows of more than 16 blocks are two parts or more of at most 16, with little work each where rows are few: 2048 x 6144, 3 rows
    // OIL4_GRP 13.3 against 15.2, registry's mix 16.8 against 20.7; 4096 x 5120 mix 18.3 against 20.6; 1024 x 8192 OIL4_GRP 17.2 against
    // 16.0, mix 17.8 against 21.5; 4096 x 8192 mix 25.5 against 22.3.
    if ((src == kOil4Grp || src == kSparkMix) && w.cols > 4096u && weights < 30000000u) return src == kOil4Grp ? w.cols >= 8192u : M == 4 && w.cols > 8192u;
    // 12 M weights: 2048 x 2048, 3 rows OIL4_GRP 7.8 against 8.1; 1500 x 4096 OIL2_GRP 8.9 against 9.6; 4096 x 4096 OIL2 11.5 against 9.2.
    // Wider than 5120 columns four rows take two passes there: 1000 x 11008 OIL2 22.3 against 14.6.
    return weights >= 12000000u || w.cols > 5120u;
}

// what the tensor's weights are, or -1 where these kernels do not cover the tensor and the batch, or another one is faster
int source_for(const oilhip_weights& w, int M) {
    const int src = source_of(w);
    if (src < 0 || M < 2 || !w.all_full || (w.cols & 255u) || w.cols == 0 || w.cols > kGemvPackMaxCols || w.rows == 0 || w.rows > 0x7FFFFFFFull) return -1;
    if (M <= (src == kOil8 ? 8 : 4) && !faster_than_row_kernels(src, w, M)) return -1;
    const uint32_t bpr = (uint32_t)(w.cols >> 8);
    // 32-bit byte offsets inside a workgroup's rows (blocks, or descriptors)
    const uint64_t per_row = std::max<uint64_t>(16u, by_descriptor(src) ? 16u : block_bytes(src)) * bpr;
    if ((w.rows / (16u * (uint64_t)device_cu_count()) + 8u) * 16u * per_row >= 0x80000000ull) return -1;
    return src;
}

}  // namespace

size_t gemv_any_multi_bytes(const oilhip_weights& w, int M) {
    const int src = source_for(w, M);
    if (src < 0) return 0;
    const size_t tiles = (size_t)tiles_for(std::min(M, kPassTokens));
    return tiles * (64u + (size_t)(w.cols >> 8) * (64u + tile_bytes(grouped(src))));
}

// Returns 1 where these kernels do not serve the call.  Without d_pack, a call that is being captured is left to the kernels that
// use no scratch: two graphs captured on one stream would share the stream's, and they may be replayed side by side.
int launch_gemv_any_multi(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s, uint8_t* d_pack, const MultiInput& in, uint32_t ldx) {
    const int src = source_for(w, M);
    if (src < 0 || (!d_pack && stream_capturing(s))) return 1;
    const uint32_t bpr = (uint32_t)(w.cols >> 8);
    const StreamLock lock(s);
    uint8_t* xp = d_pack;
    if (!xp)
        if (int rc = stream_scratch(lock, kScratchGemvPack, kGemvPackBytes, reinterpret_cast<void**>(&xp))) return rc;
    for (int m0 = 0; m0 < M; m0 += kPassTokens) {
        const int m = std::min(M - m0, kPassTokens), tiles = tiles_for(m);
        if (!ldx) ldx = (uint32_t)w.cols;
        const size_t skip = (size_t)m0 * ldx;
        const uint32_t aligned = ((reinterpret_cast<uintptr_t>(d_x) | reinterpret_cast<uintptr_t>(in.x2)) & 15u) == 0 && (ldx & 3u) == 0;
        const PackArgs p{{d_x + skip, in.x2 ? in.x2 + skip : nullptr, in.norm_w, in.xn ? in.xn + skip : nullptr, ldx, aligned, in.inv_form ? 1u : 0u},
                         xp, bpr, (uint32_t)tiles, grouped(src) ? 1u : 0u, m};
        const uint32_t tokens = (16u * (uint32_t)tiles + 2u) / 3u;
        hipLaunchKernelGGL(pack_pieces_kernel, dim3(bpr, (tokens + 3u) / 4u), dim3(256), 0, s, p);
        OILHIP_HIP(hipGetLastError());
        const BodyArgs a{w.d_payload + (by_descriptor(src) ? 0u : w.uniform_base), w.d_blocks, xp, d_y + (size_t)m0 * w.rows, (uint32_t)w.alloc_bytes,
                         (uint32_t)w.rows, bpr, (uint32_t)w.rows, 0u, 0u, 0u, 0u, 0u, m};
        int rc = 1;
        switch (src) {
            case kSpark: rc = launch_tiles<kSpark>(tiles, a, s); break;
            case kPlanner: rc = launch_tiles<kPlanner>(tiles, a, s); break;
            case kOil2: rc = launch_tiles<kOil2>(tiles, a, s); break;
            case kOil8: rc = launch_tiles<kOil8>(tiles, a, s); break;
            case kOil2Grp: rc = launch_tiles<kOil2Grp>(tiles, a, s); break;
            case kOil4Grp: rc = launch_tiles<kOil4Grp>(tiles, a, s); break;
            case kOil8Grp: rc = launch_tiles<kOil8Grp>(tiles, a, s); break;
            case kSparkMix: rc = launch_tiles<kSparkMix>(tiles, a, s); break;
        }
        if (rc) return rc;
    }
    return OILHIP_OK;
}

}  // namespace oilhip
