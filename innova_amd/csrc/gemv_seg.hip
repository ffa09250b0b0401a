// gemv_seg.hip -- decode GEMV for tensors whose rows mix wire formats (the SPARK mixes of
// FormatRegistry::allocate_mix_blocks, src/format_registry.cpp:477-599, and the stacks of FormatPlanner::allocate, src/format_planner.cpp:133-315,
// that hold more than SPARK_Q0 and OIL1, whose mix gemv_signs.hip serves): Qwen35Engine::gemm
// (src/adapters/tools/qwen35_engine.cpp:47-85) fused with dequantize_block_all (src/block_codec.cpp:576-720).
//
// Such a tensor is a few MB of small blocks (16 bytes for OIL1, 48 for SPARK_Q0), so the launch is bound by
// dependent memory round trips, not by bandwidth.  The upload therefore stores it as one stream of windows (at most
// 4 KB each) per wavefront, the first at an address that follows from the wavefront's number alone: it is fetched
// blind together with the activations, and a window describes itself and says where the next one is (entries: format, block count, where the blocks and their tags
// sit in the window, which rows they belong to).  A stream covers rows chosen so that all streams weigh about the same, in tiles of up to four;
// inside a tile the blocks are ordered by format, inside a format by row and column, so a step of 8 blocks has one
// format for all 64 lanes.  The wavefront copies a window to LDS with plain 16-byte loads, fetches the next one while it works,
// and decodes from LDS: a lane owns one run of 32 weights and adds its dot product to its accumulator of the run's
// row; when an entry closes its tile each row is summed across the wavefront in a fixed order.
//
// SPARK_Q0 runs (FP16 scale + 32 sign bits) are multiplied as FP16 pairs (+-scale is exact in FP16) through the
// mixed-precision FMA; OIL1 runs are mean * (sum of the run's activations), the sums formed once per launch while x
// is staged.
#include "common.h"
#include "oil4_lds.h"
#include "run_decode.h"

namespace oilhip {
namespace {

constexpr int kRunPad = 36;                // floats per run of 32 activations in LDS: 16-byte reads of neighbouring lanes
                                           // fall into different banks
// Wavefronts per workgroup, one workgroup per CU: 16 (four per SIMD, windows of at most 2 KB) for one activation row
// of a tensor that was packed for them, else 8 (two per SIMD, windows of at most 4 KB).  The decoding is bound by instruction
// issue with waits on LDS in between (a step of 8 SPARK_Q0 blocks is 91 vector and 10 LDS instructions), so more wavefronts
// side by side fill the waits: 11008 x 4096 at the registry's SPARK mix went from 15.7 to 13.5 us, at the planner's mix from 9.2 to
// 8.8.  More rows need more registers than four wavefronts per SIMD leave (128): there a workgroup has 8,
// and each takes two streams, one after the other (two rows with 16 wavefronts spill 31 registers to memory: 11008 x 4096 at the
// planner's mix 15.1 us, OIL8_GRP 35 us; with 8 wavefronts 12.0 and 21.6; packed for 8 wavefronts they took 11.7 and 17.9).
constexpr uint32_t window_of(int waves) { return waves == 16 ? kSegWindow / 2 : kSegWindow; }
constexpr int TR = kSegTileRows;           // accumulators per lane and activation row: a tile has at most this many rows
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// (Figures of the planner's mix and of SPARK_Q0 alone in this file are from before gemv_signs.hip served them.)
// Sign table of one activation row: for every four columns all sixteen sums +-x0 +-x1 +-x2 +-x3, entry n the one in which bit j of n makes x[j]
// positive.  A SPARK_Q0 run is then eight reads instead of 32 products of unpacked signs: 30 vector instructions fewer per step, and
// about 10 clocks of LDS for each read (16 for 16 bytes per lane of plain activations).  Where another format of the tensor works on few instructions per weight
// beside it that pays: planner's mix, 12288 x 4096 7.53 -> 7.38 us, 22016 x 4096 12.3 -> 11.4, 30000 x 2048 10.4 -> 9.5.  SPARK_Q0 alone is bound by LDS
// then (11008 x 4096 10.2 -> 10.4), and with eight wavefronts building the table costs more than it saves (4096 x 4096 5.03 -> 5.22): both stay.  Error
// against 64 bits (2-norm, planner's mix) 1.0e-7 -> 0.94e-7.  The sums are of x / 32, so that those of a run's 32 activations stay below the largest float
// where the activations do, and the block's scale is taken 32 times: both exact, but for activations below 2^-121, whose lowest bits go
// (2^-150 at most: with weights below 1/32 that is less than the rounding of a subnormal product).  That costs 0.05 to 0.1 us at these sizes, which the figures
// include.
constexpr uint32_t kSignRunBytes = 8u * 64u + 64u;        // a run's eight tables; the gap spreads runs over the LDS banks
constexpr uint32_t kSignTab = kLevelTabBytes + 64;        // where the table starts in LDS
typedef __attribute__((address_space(3))) f32x4_t lds_f4;

// the entries of columns 4 * c4 .. 4 * c4 + 3
__device__ __forceinline__ void put_signs(uint32_t c4, float4 t) {
    t.x *= 0.03125f; t.y *= 0.03125f; t.z *= 0.03125f; t.w *= 0.03125f;
    // neighbouring lanes write their four 16-byte pieces in different orders, so that eight of them hit all banks: piece j ^ sw holds the
    // sums with the signs of j and those that sw flips
    const uint32_t g = c4 & 7u, sw = g >> 1, at = kSignTab + (c4 >> 3) * kSignRunBytes + g * 64u + sw * 16u;
    const float p = t.x + t.y, q = t.x - t.y;
    const float x2 = __uint_as_float(__float_as_uint(t.z) ^ (sw << 31)), x3 = __uint_as_float(__float_as_uint(t.w) ^ ((sw >> 1) << 31));
#pragma unroll
    for (uint32_t j = 0; j < 4u; ++j) {
        const float b = (j & 1u ? x2 : -x2) + (j & 2u ? x3 : -x3);
        *(lds_f4*)(uintptr_t)(at ^ (j * 16u)) = f32x4_t{b - p, b + q, b - q, b + p};
    }
}

// a 32nd of the sum of +-x over the run whose table is at `base`: bit k of u set -> +x[k], else -x[k]
__device__ __forceinline__ float signed_sum(uint32_t u, uint32_t base) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = *(lds_cf*)(uintptr_t)((((i == 0 ? u << 2 : u >> (4 * i - 2)) & 0x3Cu) | base) + 64u * i);
    return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
}

struct SegArgs {
    uint32_t nstreams, blind16, tag_bytes, keep_x;
    uint64_t stream_bytes;
};

static_assert(TR == 4, "a closed tile's rows are summed in the four lanes of a quad");
__device__ __forceinline__ float dpp_row_ror4(float v) {                  // lane i: lane i - 4 of its sixteen
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0x124, 0xF, 0xF, true));
}
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// One entry of a window: nblk blocks of format FMT (of the size the quantizer writes: no other is packed into windows) from `data`, their tags from `tags`
// (both in LDS).
// adds a run's dot products to the accumulators of its row of the tile
template <int MB>
__device__ __forceinline__ void add_to_row(float (&acc)[MB][TR], uint32_t rowl, const float (&part)[MB]) {
#pragma unroll
    for (int j = 0; j < TR; ++j) {
        const bool mine = rowl == (uint32_t)j;
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[m][j] += mine ? part[m] : 0.f;
    }
}

template <int FMT, int MB, bool SIGNS>
__device__ __forceinline__ void run_entry(const uint8_t* data, const uint8_t* tags, uint32_t tagw, uint32_t nblk,
                                          const DecodeTables* __restrict__ T, const LdsTables& L, const float* xs, const float* rs,
                                          float (&acc)[MB][TR], uint32_t xpad, uint32_t nruns, uint32_t lane) {
    constexpr int N = run_raw_dwords(FMT);
    constexpr uint32_t stride = (full_block_bytes(FMT) + 15u) & ~15u;
    uint32_t cb_bytes = full_block_cb_bytes(FMT), idx_bytes = full_block_bytes(FMT) - cb_bytes;
    // (four activation rows leave no registers for what the compiler makes of known sizes in the sparse formats: 244 bytes of spills, 1000 x 1280 of
    // the registry's mix 9.9 -> 13.6 us)
    if constexpr (MB >= 4) asm volatile("" : "+s"(cb_bytes), "+s"(idx_bytes));
    const uint32_t steps = (nblk + 7u) >> 3, r = lane & 7u, g = lane >> 3;
    // a block's tag: row of the tile and column block, one byte (row << 6 | column) or two (row << 12 | column)
    const uint32_t tshift = tagw == 1u ? 6u : 12u, tmask = tagw == 1u ? 0x3Fu : 0xFFFu;
    auto tag_of = [&](uint32_t b) -> uint32_t {
        return tagw == 1u ? (uint32_t)tags[b] : (uint32_t)reinterpret_cast<const uint16_t*>(tags)[b];
    };
    if constexpr (FMT == 0) {
        // a block is 8 FP16 run means: a lane takes a whole block, 16 bytes of means against 8 run sums
        for (uint32_t b0 = 0; b0 < nblk; b0 += 64u) {
            const uint32_t blk = b0 + lane;
            const bool live = blk < nblk;
            const uint32_t bc = live ? blk : nblk - 1u;
            const uint32_t tag = tag_of(bc);
            const u32x4 mv = *reinterpret_cast<const u32x4*>(data + bc * stride);
            const float mean[8] = {f16_bits(mv.x), f16_bits(mv.x >> 16), f16_bits(mv.y), f16_bits(mv.y >> 16),
                                   f16_bits(mv.z), f16_bits(mv.z >> 16), f16_bits(mv.w), f16_bits(mv.w >> 16)};
            float part[MB];
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const float4* sp = reinterpret_cast<const float4*>(rs + (size_t)m * nruns + (tag & tmask) * 8u);
                const float4 s0 = sp[0], s1 = sp[1];
                float a0 = mean[0] * s0.x, a1 = mean[1] * s0.y;
                a0 = __fmaf_rn(mean[2], s0.z, a0);
                a1 = __fmaf_rn(mean[3], s0.w, a1);
                a0 = __fmaf_rn(mean[4], s1.x, a0);
                a1 = __fmaf_rn(mean[5], s1.y, a1);
                a0 = __fmaf_rn(mean[6], s1.z, a0);
                a1 = __fmaf_rn(mean[7], s1.w, a1);
                part[m] = live ? a0 + a1 : 0.f;
            }
            add_to_row<MB>(acc, tag >> tshift, part);
        }
    } else {
    for (uint32_t st = 0; st < steps; ++st) {
        const uint32_t blk = st * 8u + g;
        const bool live = blk < nblk;
        const uint32_t bc = live ? blk : nblk - 1u;                     // past the end: the last block again, result unused
        const uint32_t tag = tag_of(bc);
        const uint8_t* cb = data + bc * stride;
        uint32_t raw[N];
        fetch_run<FMT>(cb, cb_bytes, r, raw);
        const uint32_t rowl = tag >> tshift, run = (tag & tmask) * 8u + r;
        float part[MB];
        if constexpr (FMT == 1 && SIGNS) {
            part[0] = (32.0f * f16_bits(raw[0])) * signed_sum(raw[1], kSignTab + run * kSignRunBytes);
        } else if constexpr (FMT == 1) {
            // weight k = bit k ? +scale : -scale; as FP16: |scale| with the sign bit from the (inverted) sign word.
            // Pair k holds weights k (low half) and k + 16 (high half).
            const uint32_t s16 = raw[0] & 0xFFFFu;
            const uint32_t mag = s16 & 0x7FFFu;
            uint32_t mag2 = mag | (mag << 16);
            asm volatile("" : "+v"(mag2));                             // one v_and_or_b32 per pair below, not a multiply-add
            const uint32_t negm = ~raw[1] ^ (0u - (s16 >> 15));
            uint32_t w2[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) w2[k] = ((negm << (15 - k)) & 0x80008000u) | mag2;
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const float* xr = xs + (size_t)m * xpad + run * kRunPad;
                float4 xv[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) xv[c] = *reinterpret_cast<const float4*>(xr + 4 * c);
                float a0 = 0.f, a1 = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const h2v p0 = __builtin_bit_cast(h2v, w2[4 * c]), p1 = __builtin_bit_cast(h2v, w2[4 * c + 1]);
                    const h2v p2 = __builtin_bit_cast(h2v, w2[4 * c + 2]), p3 = __builtin_bit_cast(h2v, w2[4 * c + 3]);
                    a0 = __fmaf_rn((float)p0[0], xv[c].x, a0);
                    a1 = __fmaf_rn((float)p0[1], xv[c + 4].x, a1);
                    a0 = __fmaf_rn((float)p1[0], xv[c].y, a0);
                    a1 = __fmaf_rn((float)p1[1], xv[c + 4].y, a1);
                    a0 = __fmaf_rn((float)p2[0], xv[c].z, a0);
                    a1 = __fmaf_rn((float)p2[1], xv[c + 4].z, a1);
                    a0 = __fmaf_rn((float)p3[0], xv[c].w, a0);
                    a1 = __fmaf_rn((float)p3[1], xv[c + 4].w, a1);
                }
                part[m] = a0 + a1;
            }
        } else if constexpr (has_dot_run(FMT)) {
            constexpr int MH = MB > 2 ? 2 : MB;          // activation rows per pass: 32 registers of x each
#pragma unroll
            for (int h = 0; h < MB; h += MH) {
                f32x4_t xv[MH][8];
                float xsum[MH], sub[MH];
#pragma unroll
                for (int m = 0; m < MH; ++m) {
                    const float* xr = xs + (size_t)(h + m) * xpad + run * kRunPad;
#pragma unroll
                    for (int c = 0; c < 8; ++c) xv[m][c] = *reinterpret_cast<const f32x4_t*>(xr + 4 * c);
                    xsum[m] = rs[(size_t)(h + m) * nruns + run];
                }
                dot_run<FMT, MH>(raw, r, xv, xsum, sub);
#pragma unroll
                for (int m = 0; m < MH; ++m) part[h + m] = sub[m];
            }
        } else {
            float w[32];
            expand_run<FMT>(raw, cb, cb_bytes, idx_bytes, r, T, L, w);
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const float* xr = xs + (size_t)m * xpad + run * kRunPad;
                float a0 = 0.f, a1 = 0.f;
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    const float4 xv = *reinterpret_cast<const float4*>(xr + 4 * c);
                    a0 = __fmaf_rn(w[4 * c], xv.x, a0);
                    a1 = __fmaf_rn(w[4 * c + 1], xv.y, a1);
                    a0 = __fmaf_rn(w[4 * c + 2], xv.z, a0);
                    a1 = __fmaf_rn(w[4 * c + 3], xv.w, a1);
                }
                part[m] = a0 + a1;
            }
        }
        if (!live) {
#pragma unroll
            for (int m = 0; m < MB; ++m) part[m] = 0.f;
        }
        add_to_row<MB>(acc, rowl, part);
    }
    }
}

#define OILHIP_SEG_FORMATS(X) X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14)

// MB activation rows per launch.  Dynamic LDS: level tables, MB * (padded x + run sums), two windows per wavefront.
// XF (one activation row only) transforms x while it is staged: 1 = the row holds 2 * cols floats h and the kernel
// multiplies with siluf(h[k]) * h[cols + k] (the SwiGLU product of Qwen35Engine::mlp_step,
// src/adapters/tools/qwen35_engine.cpp:611-621); 2 = x * (1 + xw[k]) is staged and every output is scaled by
// 1 / sqrt(mean(x^2) + 1e-6), which each workgroup forms from the row it loads anyway (Qwen35Engine::rmsnorm, :39-44).
template <int MB, int XF, int kWaves, bool SIGNS>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kWaves / 4, kWaves / 4)))
gemv_seg_kernel(const uint8_t* __restrict__ streams, const DecodeTables* __restrict__ T, const float* __restrict__ x,
                const float* __restrict__ xw, float* __restrict__ y, uint32_t rows, uint32_t cols, int m0, int M,
                const SegArgs A) {
    static_assert((XF == 0 && !SIGNS) || MB == 1, "the fused input transforms and the sign table serve one activation row");
    constexpr uint32_t WIN = window_of(kWaves);
    constexpr int NW = WIN / 1024;                     // 16-byte pieces of a window per lane
    extern __shared__ __align__(16) float smem[];
    const uint32_t nruns = cols >> 5, xpad = nruns * kRunPad;
    float* ssq_part = smem + kLevelTabBytes / 4;       // XF = 2: sum(x^2) per wavefront
    float* xs = ssq_part + 16;                         // [MB][nruns][36], behind the level tables of dot_run (and the sign table)
    if constexpr (SIGNS) xs += nruns * (kSignRunBytes / 4u);
    float* rs = xs + (!SIGNS || A.keep_x ? (size_t)MB * xpad : 0);                // [MB][nruns] run sums
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = uniform(tid >> 6);
    constexpr uint32_t NBUF = SIGNS ? 1u : 2u;         // windows in LDS (the next one waits in registers: it may overwrite the one that is worked off)
    uint8_t* win = reinterpret_cast<uint8_t*>(rs + (size_t)MB * nruns) + (size_t)wave * NBUF * WIN;
    const LdsTables L{nullptr, nullptr, nullptr, nullptr};      // the formats that expand weight by weight here use no level table

    uint32_t sid = blockIdx.x * kWaves + wave;
    const bool active = sid < A.nstreams;
    const uint8_t* sp = streams + (active ? (size_t)sid * A.stream_bytes : 0);
    u32x4 wreg[NW];                                    // a window in flight
    // the first window is fetched before anything is known about it: as many 16-byte pieces as the fullest first
    // window of the tensor has
    // (pieces past that size repeat the last one: every lane loads, unconditionally, so that nothing waits here)
#pragma unroll
    for (int j = 0; j < NW; ++j) {
        const uint32_t piece = j * 64u + lane < A.blind16 ? j * 64u + lane : A.blind16 - 1u;
        wreg[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(sp + (size_t)piece * 16u));
    }

    build_level_tables(smem, tid);
    // x -> LDS, 36 floats per run; 8 consecutive threads hold one run and add it up on the way
    const uint32_t nq = cols >> 2;
    float ssq = 0.f;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const bool on = m0 + m < M;
        const float4* xrow = reinterpret_cast<const float4*>(x + (size_t)(on ? m0 + m : 0) * cols * (XF == 1 ? 2u : 1u));
        for (uint32_t c0 = tid; c0 < nq; c0 += 256u * kWaves) {
            float4 v[4], b[XF ? 4 : 1];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t c4 = c0 + 64u * kWaves * j;
                v[j] = xrow[c4 < nq ? c4 : c0];
                if constexpr (XF == 1) b[j] = xrow[nq + (c4 < nq ? c4 : c0)];
                if constexpr (XF == 2) b[j] = reinterpret_cast<const float4*>(xw)[c4 < nq ? c4 : c0];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t c4 = c0 + 64u * kWaves * j;
                if (c4 < nq) {
                    float4 t = on ? v[j] : make_float4(0.f, 0.f, 0.f, 0.f);
                    if constexpr (XF == 1) {
                        t.x = (t.x * __builtin_amdgcn_rcpf(1.0f + __expf(-t.x))) * b[j].x;
                        t.y = (t.y * __builtin_amdgcn_rcpf(1.0f + __expf(-t.y))) * b[j].y;
                        t.z = (t.z * __builtin_amdgcn_rcpf(1.0f + __expf(-t.z))) * b[j].z;
                        t.w = (t.w * __builtin_amdgcn_rcpf(1.0f + __expf(-t.w))) * b[j].w;
                    }
                    if constexpr (XF == 2) {
                        ssq = __fmaf_rn(t.x, t.x, __fmaf_rn(t.y, t.y, __fmaf_rn(t.z, t.z, __fmaf_rn(t.w, t.w, ssq))));
                        t.x *= 1.0f + b[j].x; t.y *= 1.0f + b[j].y; t.z *= 1.0f + b[j].z; t.w *= 1.0f + b[j].w;
                    }
                    if constexpr (SIGNS) put_signs(c4, t);
                    if (!SIGNS || A.keep_x) *reinterpret_cast<float4*>(xs + (size_t)m * xpad + (c4 >> 3) * kRunPad + (c4 & 7u) * 4) = t;
                    float s = (t.x + t.y) + (t.z + t.w);
                    s += oil4::dpp_quad_xor1(s);
                    s += oil4::dpp_quad_xor2(s);
                    s += oil4::dpp_half_mirror(s);
                    if ((c4 & 7u) == 0u) rs[(size_t)m * nruns + (c4 >> 3)] = s;
                }
            }
        }
    }
    if constexpr (XF == 2) {
        float v = ssq;
        v += oil4::dpp_quad_xor1(v);
        v += oil4::dpp_quad_xor2(v);
        v += oil4::dpp_half_mirror(v);
        v += oil4::dpp_row_mirror(v);
        v += oil4::dpp_row_bcast15(v);
        v += oil4::dpp_row_bcast31(v);
        if (lane == 63) ssq_part[wave] = v;
    }
#pragma unroll
    for (int j = 0; j < NW; ++j) *reinterpret_cast<u32x4*>(win + ((size_t)j * 64u + lane) * 16u) = wreg[j];
    __syncthreads();
    if (!active) return;
    float yscale = 1.0f;
    if constexpr (XF == 2) {
        float tot = 0.f;
#pragma unroll
        for (int j = 0; j < kWaves; j += 4) tot += (ssq_part[j] + ssq_part[j + 1]) + (ssq_part[j + 2] + ssq_part[j + 3]);
        yscale = 1.0f / sqrtf(tot / (float)cols + 1e-6f);
    }

    float acc[MB][TR];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int j = 0; j < TR; ++j) acc[m][j] = 0.f;
    for (uint32_t wi = 0;; ++wi) {
        const uint8_t* cur = win + (NBUF == 2u ? (wi & 1u) * WIN : 0u);
        // the header and the records, 8 bytes each: a lane holds one of 64 in a row, and an entry costs no LDS round trip of its own
        const uint2* units = reinterpret_cast<const uint2*>(cur);
        uint2 held = units[lane];
        uint32_t held0 = 0;
        auto unit = [&](uint32_t u) -> uint2 {
            if (u - held0 >= 64u) { held0 = u; held = units[u + lane < WIN / 8u ? u + lane : u]; }
            return make_uint2((uint32_t)__builtin_amdgcn_readlane((int)held.x, (int)(u - held0)), (uint32_t)__builtin_amdgcn_readlane((int)held.y, (int)(u - held0)));
        };
        const uint2 hdr = unit(0u);
        const uint32_t h0 = hdr.x;                     // 8-byte units of records | another window follows << 12 | its 16-byte pieces << 16
        bool more = (h0 >> 12) & 1u;
        uint32_t used16 = h0 >> 16;                    // the next window: its size and place are in this one's header, ...
        const uint8_t* np = streams + (size_t)hdr.y * 16u;
        if (MB > 1 && !more && (sid += gridDim.x * kWaves) < A.nstreams) {         // ... or it is the first one of this wavefront's next stream
            more = true;
            used16 = A.blind16;
            np = streams + (size_t)sid * A.stream_bytes;
        }
        if (more) {
#pragma unroll
            for (int j = 0; j < NW; ++j) {
                const uint32_t piece = j * 64u + lane < used16 ? j * 64u + lane : used16 - 1u;
                wreg[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(np + (size_t)piece * 16u));
            }
        }
        const uint32_t ne = h0 & 0xFFFu;               // an entry is one unit, the row numbers behind a closing entry two
        for (uint32_t i = 1; i <= ne; ++i) {
            const uint2 rec = unit(i);
            const uint32_t r0 = rec.x, r1 = rec.y, nblk = r0 >> 16, nrows = (r0 >> 9) & 7u;
            const uint8_t* data = cur + (r1 & 0xFFFFu);
            const uint8_t* tags = cur + (r1 >> 16);
#define OILHIP_SEG_CASE(F)                                                                                              \
    case F:                                                                                                             \
        run_entry<F, MB, SIGNS>(data, tags, A.tag_bytes, nblk, T, L, xs, rs, acc, xpad, nruns, lane);                                                                                  \
        break;
            switch ((r0 >> 4) & 15u) { OILHIP_SEG_FORMATS(OILHIP_SEG_CASE) default: break; }
#undef OILHIP_SEG_CASE
            if ((r0 >> 8) & 1u) {                      // the tile is complete: sum its rows across the wavefront, row q in every lane with lane % 4 = q
                // (two units with the row numbers follow a closing entry)
                const uint32_t trow = reinterpret_cast<const uint32_t*>(cur + 8u * (i + 1u))[lane & 3u];
                const bool b0 = lane & 1u, b1 = lane & 2u;
                i += 2;
#pragma unroll
                for (int m = 0; m < MB; ++m) {
                    const float r01 = (b0 ? acc[m][1] : acc[m][0]) + oil4::dpp_quad_xor1(b0 ? acc[m][0] : acc[m][1]);
                    const float r23 = (b0 ? acc[m][3] : acc[m][2]) + oil4::dpp_quad_xor1(b0 ? acc[m][2] : acc[m][3]);
                    float v = (b1 ? r23 : r01) + oil4::dpp_quad_xor2(b1 ? r01 : r23);
                    v += dpp_row_ror4(v);                                  // lanes 4 to 7 and 12 to 15: with the quad before
                    v += oil4::dpp_row_ror8(v);                            // ... and the other two
                    const auto rows2 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
                    v = __uint_as_float(rows2[0]) + __uint_as_float(rows2[1]);
                    const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
                    v = __uint_as_float(halves[0]) + __uint_as_float(halves[1]);
                    if ((lane & ~3u) == 4u && (lane & 3u) < nrows && m0 + m < M) y[(size_t)(m0 + m) * rows + trow] = v * yscale;
#pragma unroll
                    for (int j = 0; j < TR; ++j) acc[m][j] = 0.f;
                }
            }
        }
        if (more) {
            uint8_t* nxt = win + (NBUF == 2u ? ((wi + 1u) & 1u) * WIN : 0u);
#pragma unroll
            for (int j = 0; j < NW; ++j) *reinterpret_cast<u32x4*>(nxt + ((size_t)j * 64u + lane) * 16u) = wreg[j];
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");       // other lanes read what this lane wrote
        } else {
            break;
        }
    }
}

template <int MB>
size_t seg_lds_bytes(const oilhip_weights& w) {        // the windows take 64 KB with 8 wavefronts and with 16
    return kLevelTabBytes + 64 + (size_t)MB * ((w.cols >> 5) * (kRunPad + 1)) * 4 + 16 * (size_t)kSegWindow;
}

// whether a format of the tensor reads the activations themselves (OIL1 takes their sums, SPARK_Q0 the sign table)
bool keeps_x(const SegLayout& g) {
    for (uint32_t i = 0; i < g.nf; ++i)
        if (g.fmt[i] > 1u) return true;
    return false;
}

size_t signs_lds_bytes(const oilhip_weights& w) {
    const size_t nruns = w.cols >> 5;
    return kSignTab + nruns * (kSignRunBytes + (keeps_x(w.seg) ? kRunPad * 4 : 0) + 4) + 8 * (size_t)kSegWindow;
}

// The sign table: SPARK_Q0 beside other formats, sixteen wavefronts, and a row short enough for it (7168 columns of the planner's mix).
bool takes_signs(const oilhip_weights& w) {
    bool spark = false;
    for (uint32_t i = 0; i < w.seg.nf; ++i) spark |= w.seg.fmt[i] == OILHIP_SPARK_Q0;
    return spark && w.seg.nf > 1 && w.seg.waves == 16 && signs_lds_bytes(w) <= 160 * 1024;
}

template <int MB, int XF, int kWaves, bool SIGNS>
int launch_waves(const oilhip_weights& w, const DecodeTables* T, const float* d_x, float* d_y, int m0, int M, hipStream_t s,
                 const float* d_xw) {
    static std::atomic<uint64_t> attr_done{0};
    auto kern = gemv_seg_kernel<MB, XF, kWaves, SIGNS>;
    const SegLayout& g = w.seg;
    const size_t lds = SIGNS ? signs_lds_bytes(w) : seg_lds_bytes<MB>(w);
    if (lds > 160 * 1024) return 1;
    if (int rc = ensure_max_lds(attr_done, reinterpret_cast<const void*>(kern), 160 * 1024)) return rc;
    SegArgs A{};
    A.nstreams = g.nstreams; A.blind16 = g.blind16; A.tag_bytes = g.tag_bytes; A.keep_x = keeps_x(g); A.stream_bytes = g.stream_bytes;
    const uint32_t per = (g.waves + kWaves - 1) / kWaves;              // streams per wavefront
    hipLaunchKernelGGL(kern, dim3((g.nstreams + kWaves * per - 1) / (kWaves * per)), dim3(64 * kWaves), lds, s, w.d_payload, T, d_x, d_xw,
                       d_y, (uint32_t)w.rows, (uint32_t)w.cols, m0, M, A);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

template <int MB, int XF = 0>
int launch_seg(const oilhip_weights& w, const DecodeTables* T, const float* d_x, float* d_y, int m0, int M, hipStream_t s,
               const float* d_xw = nullptr) {
    if constexpr (MB == 1) {
        if (takes_signs(w)) return launch_waves<MB, XF, 16, true>(w, T, d_x, d_y, m0, M, s, d_xw);
        if (w.seg.waves == 16) return launch_waves<MB, XF, 16, false>(w, T, d_x, d_y, m0, M, s, d_xw);
    }
    return launch_waves<MB, XF, 8, false>(w, T, d_x, d_y, m0, M, s, d_xw);
}

}  // namespace

// Returns 1 when the tensor has no window streams or the shape is outside what this kernel covers.
int launch_gemv_seg(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s) {
    if (!w.seg.nstreams || !w.all_full || (w.cols & 255u) || w.rows == 0) return 1;
    const DecodeTables* T = nullptr;
    if (int rc = get_tables(&T)) return rc;
    if (seg_lds_bytes<1>(w) > 160 * 1024) return 1;
    int m0 = 0;
    while (m0 < M) {
        const int left = M - m0;
        int rc;
        if (left >= 3 && seg_lds_bytes<4>(w) <= 160 * 1024) { rc = launch_seg<4>(w, T, d_x, d_y, m0, M, s); m0 += 4; }
        else if (left >= 2 && seg_lds_bytes<2>(w) <= 160 * 1024) { rc = launch_seg<2>(w, T, d_x, d_y, m0, M, s); m0 += 2; }
        else { rc = launch_seg<1>(w, T, d_x, d_y, m0, M, s); m0 += 1; }
        if (rc) return rc;
    }
    return OILHIP_OK;
}

// y = W . (siluf(h[0..K)) * h[K..2K)) for one activation row h of 2K floats.  Returns 1 when the tensor is not covered.
int launch_gemv_seg_swiglu(const oilhip_weights& w, const float* d_h, float* d_y, hipStream_t s) {
    if (!w.seg.nstreams || !w.all_full || (w.cols & 255u) || w.rows == 0 || seg_lds_bytes<1>(w) > 160 * 1024) return 1;
    const DecodeTables* T = nullptr;
    if (int rc = get_tables(&T)) return rc;
    return launch_seg<1, 1>(w, T, d_h, d_y, 0, 1, s);
}

// y = W . rmsnorm(x; xw) for one activation row.  Returns 1 when the tensor is not covered.
int launch_gemv_seg_rmsnorm(const oilhip_weights& w, const float* d_x, const float* d_xw, float* d_y, hipStream_t s) {
    if (!w.seg.nstreams || !w.all_full || (w.cols & 255u) || w.rows == 0 || seg_lds_bytes<1>(w) > 160 * 1024) return 1;
    const DecodeTables* T = nullptr;
    if (int rc = get_tables(&T)) return rc;
    return launch_seg<1, 2>(w, T, d_x, d_y, 0, 1, s, d_xw);
}

}  // namespace oilhip
