// generic_kernels.hip -- the all-format kernels: bit-exact tensor dequantize and a
// GEMV/GEMM that decodes every weight through decode_weight().  They cover every
// wire format, mixed-format rows and ragged tail blocks; the specialised kernels
// (gemv_oil4.hip, ...) take over for the shapes that matter for throughput.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "gemm_tiles.h"

namespace oilhip {
namespace {

// One workgroup per block, one thread per weight (strided for blocks > 256).
// Mirrors OILReader::read_tensor's loop over dequantize_block_all
// (src/oil_format.cpp:464-477).
__global__ void __launch_bounds__(256)
dequant_kernel(const uint8_t* __restrict__ payload, const DevBlock* __restrict__ blocks,
               const uint64_t* __restrict__ out_off, const DecodeTables* __restrict__ T,
               float* __restrict__ out, uint32_t nblocks, uint32_t uniform_nw) {
    for (uint32_t b = blockIdx.x; b < nblocks; b += gridDim.x) {
        const DevBlock d = blocks[b];
        const uint8_t* cb = payload + (size_t)d.off16 * 16;
        const uint8_t* idx = cb + d.cb_bytes;
        float* o = out + (out_off ? out_off[b] : (uint64_t)b * uniform_nw);
        for (uint32_t i = threadIdx.x; i < d.nw; i += 256)
            o[i] = decode_weight(d.fmt, cb, d.cb_bytes, idx, d.idx_bytes, d.nw, i, T);
    }
}

// ---- full 256-weight blocks of nominal size: a wavefront per block, lane l decodes weights 4l .. 4l+3 and stores one
// float4, so a block is one coalesced 1 KB store.  Every value is formed exactly as decode_weight forms it (level
// from the literal / host-built tables times the FP16 scale widened by the integer rule, one fused multiply-add for
// the grouped formats, scale == 0 -> zero point, slots 0).  Blocks sit back to back at a regular stride (`blocks`
// null) or wherever their descriptors say (tensors stored as window streams or sign tiles).
struct FullTables { const float* lv8; const float* t255; const float* q127; const float* lv4; const float* lv2; };   // LDS copies


// BITS_OF_NAN: FP16 widened by the integer rule of the reference, NaN payloads included; else by the hardware's conversion (the same
// value for everything but NaN payloads)
template <int FMT, bool BITS_OF_NAN = true>
__device__ __forceinline__ float4 decode_full4(const uint8_t* __restrict__ p, uint32_t lane, const FullTables& L) {
    auto widen = [](uint32_t h) { return BITS_OF_NAN ? half_bits_to_float(h) : __half2float(__ushort_as_half((unsigned short)h)); };
    const uint32_t* q = reinterpret_cast<const uint32_t*>(p);
    const uint32_t i0 = 4u * lane;
    if constexpr (FMT == 2 || FMT == 3 || FMT == 4) {                      // OIL2 / OIL4 / OIL8 (src/block_codec.cpp:173-182)
        constexpr uint32_t BITS = FMT == 2 ? 2u : (FMT == 3 ? 4u : 8u);
        const float* lv = FMT == 2 ? L.lv2 : (FMT == 3 ? L.lv4 : L.lv8);
        const float scale = widen(q[0] & 0xFFFFu);
        // first code bit of weight 4l: 16 + BITS * (4l - slots before it); one slot per 16*BITS weights
        const uint32_t bit = 16u + BITS * (i0 - i0 / (16u * BITS));
        const uint32_t lo = q[bit >> 5], hi = q[(bit >> 5) + 1u];            // hi may be the first dword after the block: unused bits
        const uint32_t v = __builtin_amdgcn_alignbit(hi, lo, bit & 31u);
        const bool last_is_slot = ((i0 + 4u) % (16u * BITS)) == 0u;
        constexpr uint32_t mask = (1u << BITS) - 1u;
        return make_float4(lv[v & mask] * scale, lv[(v >> BITS) & mask] * scale, lv[(v >> (2u * BITS)) & mask] * scale,
                           last_is_slot ? 0.0f : lv[(v >> (3u * BITS)) & mask] * scale);
    } else if constexpr (FMT == 0) {                                       // OIL1: eight FP16 run means (:615-626)
        const float m = widen(reinterpret_cast<const uint16_t*>(p)[lane >> 3]);
        return make_float4(m, m, m, m);
    } else if constexpr (FMT == 1) {                                       // SPARK_Q0: per run FP16 scale + 32 sign bits (:643-654)
        const uint16_t* h = reinterpret_cast<const uint16_t*>(p);
        const uint32_t run = lane >> 3, j0 = 4u * (lane & 7u);
        const float sc = widen(h[3u * run]);
        const uint32_t bits = ((uint32_t)h[3u * run + 1u] | ((uint32_t)h[3u * run + 2u] << 16)) >> j0;
        return make_float4((bits & 1u) ? sc : -sc, (bits & 2u) ? sc : -sc, (bits & 4u) ? sc : -sc, (bits & 8u) ? sc : -sc);
    } else if constexpr (FMT == 5 || FMT == 12) {                          // OIL16 / OIL16_GRP: 512 bytes of FP16 (:588-596)
        const uint32_t a = q[2u * lane], c = q[2u * lane + 1u];
        return make_float4(widen(a & 0xFFFFu), widen(a >> 16), widen(c & 0xFFFFu),
                           widen(c >> 16));
    } else if constexpr (FMT == 6) {                                       // OIL32: raw FP32 (:585-587)
        const uint4 v = reinterpret_cast<const uint4*>(p)[lane];
        return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
    } else if constexpr (FMT == 7) {                                       // OIL1_GRP: scale, 240 sign bits, every 16th weight a slot (:627-642)
        const float scale = widen(q[0] & 0xFFFFu);
        const uint32_t bit = 16u + i0 - i0 / 16u;
        const uint32_t v = __builtin_amdgcn_alignbit(q[(bit >> 5) + 1u], q[bit >> 5], bit & 31u);
        const bool last_is_slot = ((i0 + 4u) & 15u) == 0u;
        return make_float4((v & 1u) ? scale : -scale, (v & 2u) ? scale : -scale, (v & 4u) ? scale : -scale,
                           last_is_slot ? 0.0f : ((v & 8u) ? scale : -scale));
    } else if constexpr (FMT == 8) {                                       // SPARK_Q0_GRP: scale, 256 signs, 112 refinement bits (:655-676)
        const float scale = widen(q[0] & 0xFFFFu);
        const uint32_t sbit = 16u + i0;                                    // four signs inside one dword
        const uint32_t sg = q[sbit >> 5] >> (sbit & 31u);
        float r[4];
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) {
            const uint32_t i = i0 + e;
            float mag = scale;
            if (((i + 1u) * 112u) / 256u != (i * 112u) / 256u) {           // a refined position (is_slot with 112 of 256)
                const uint32_t rpos = 16u + 256u + (i * 112u) / 256u;
                mag = __fmul_rn(scale, ((q[rpos >> 5] >> (rpos & 31u)) & 1u) ? 1.893f : 0.567f);
            }
            r[e] = ((sg >> e) & 1u) ? mag : -mag;
        }
        return make_float4(r[0], r[1], r[2], r[3]);
    } else if constexpr (FMT == 9 || FMT == 10 || FMT == 11) {             // grouped lattice: 4 x {FP16 zp, FP16 scale, 64 codes} (:308-331)
        constexpr uint32_t bits = FMT == 9 ? 2u : (FMT == 10 ? 4u : 8u), gbytes = 4u + 8u * bits;
        const float* lv = FMT == 9 ? L.lv2 : (FMT == 10 ? L.lv4 : L.t255);
        const uint32_t g = lane >> 4, j0 = 4u * (lane & 15u);              // group, first weight of the lane inside it
        const uint32_t hdr = *reinterpret_cast<const uint32_t*>(p + g * gbytes);
        const float zp = widen(hdr & 0xFFFFu), sc = widen(hdr >> 16);
        const uint32_t cbit = j0 * bits;                                   // 4 codes: 8, 16 or 32 bits inside one dword
        const uint32_t v = *reinterpret_cast<const uint32_t*>(p + g * gbytes + 4u + (cbit >> 5) * 4u) >> (cbit & 31u);
        float r[4];
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e)
            r[e] = sc == 0.0f ? zp : __fmaf_rn(lv[(v >> (e * bits)) & ((1u << bits) - 1u)], sc, zp);
        return make_float4(r[0], r[1], r[2], r[3]);
    } else {                                                               // SPARK_SPARSE / _GRP: header + 20 records, later ones win (:677-716)
        const uint4* p4 = reinterpret_cast<const uint4*>(p);
        const uint4 v0 = p4[0], v1 = p4[1], v2 = p4[2], v3 = p4[3];
        const uint32_t d[16] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w, v2.x, v2.y, v2.z, v2.w, v3.x, v3.y, v3.z, v3.w};
        float s0, s1;
        bool dead;
        if (FMT == 13) { s0 = s1 = __uint_as_float(d[0]); dead = s0 == 0.0f; }
        else { s0 = widen(d[0] & 0xFFFFu); s1 = widen(d[0] >> 16); dead = s0 == 0.0f && s1 == 0.0f; }
        float r[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < 20; ++k) {
            const int o = 4 + 3 * k;                                       // byte offset of record k
            const uint32_t lo = d[o >> 2], hi = d[(o >> 2) + ((o & 3) ? 1 : 0)];
            const uint32_t rec = __builtin_amdgcn_alignbyte(hi, lo, o & 3) & 0xFFFFFFu;
            const uint32_t rel = rec & 0xFFFFu, e = rel - i0;
            const float val = L.q127[rec >> 16] * (rel < 128u ? s0 : s1);
#pragma unroll
            for (uint32_t t = 0; t < 4u; ++t) r[t] = e == t ? val : r[t];
        }
        return dead ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : make_float4(r[0], r[1], r[2], r[3]);
    }
}

#define OILHIP_ALL_FORMATS(X) X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14)

// FMT >= 0: every block has that format; FMT < 0: each block's format from its descriptor (tensors that mix formats)
template <int FMT>
__global__ void __launch_bounds__(256)
dequant_full_kernel(const uint8_t* __restrict__ base, uint32_t stride, const DevBlock* __restrict__ blocks,
                    const DecodeTables* __restrict__ T, float* __restrict__ out, uint32_t nblocks) {
    __shared__ float tb[256 * 3 + 20];
    {
        const uint32_t t = threadIdx.x;
        tb[t] = T->lv8[t]; tb[256 + t] = T->t255[t]; tb[512 + t] = T->q127[t];
        if (t < 16) tb[768 + t] = kLv4[t];
        if (t < 4) tb[784 + t] = kLv2[t];
    }
    __syncthreads();
    const FullTables L{tb, tb + 256, tb + 512, tb + 768, tb + 784};
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for (uint32_t b = blockIdx.x * 4u + wave; b < nblocks; b += gridDim.x * 4u) {
        const uint8_t* p = base + (blocks ? (size_t)blocks[b].off16 * 16u : (size_t)b * stride);
        float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if constexpr (FMT >= 0) {
            o = decode_full4<FMT>(p, lane, L);
        } else {
            const int f = __builtin_amdgcn_readfirstlane((int)blocks[b].fmt);
#define OILHIP_CASE(F) case F: o = decode_full4<F>(p, lane, L); break;
            switch (f) { OILHIP_ALL_FORMATS(OILHIP_CASE) default: break; }
#undef OILHIP_CASE
        }
        reinterpret_cast<float4*>(out + (size_t)b * 256u)[lane] = o;
    }
}

// ---- the operands of the prefill GEMM in fragment order: [32-row block][16-column group][lane][8 bf16], lane = 32 * (column
// half) + row % 32 ---------------------------------------------------------------------------------------------------------
// A workgroup takes one 256-column block of 32 rows, of the weights or (past nw workgroups) of the activations.  Weights: a wavefront
// fetches its rows' blocks whole, 16 bytes per lane, all in flight, and parks them in LDS; then a lane decodes eight weights of
// one row at a time from there (each value rounded once to bf16, to nearest even), which are its 16 bytes of a fragment.
// Activations are parked as bf16 and read back the same way.
// What bounds it: writing the operands.
struct PrepareArgs {
    const uint8_t* base;
    const DevBlock* blocks;         // null: blocks `stride` apart, all of format fmt
    const DecodeTables* T;
    uint16_t *wf, *xf;
    const void* x;
    uint32_t* arrived;              // counters to clear
    uint32_t stride, need_tables, row0, rows, bpr, nw, M, x_is_f32, raw_pitch, ncount;
};
constexpr uint32_t kParkPitch = 256u + 8u;     // bf16 per parked row: 16-byte reads of 16 rows hit every bank once

__host__ __device__ constexpr uint32_t largest_block(uint32_t formats) {
    uint32_t n = 0;
    for (int f = 0; f < 15; ++f) n = (formats >> f & 1u) && full_block_bytes(f) > n ? full_block_bytes(f) : n;
    return n;
}

// FORMATS: the formats that may occur, as bits; several: each block's format from its descriptor
// NW: wavefronts of a workgroup
template <uint32_t FORMATS, uint32_t NW>
__global__ void __launch_bounds__(64 * NW, 4)
dense_prepare_kernel(const PrepareArgs a) {
    constexpr uint32_t R = 32u / NW, PIECES = 16u / NW;                      // rows per wavefront, fragments (and 8-column pieces of x) per thread
    constexpr int ONLY = (FORMATS & (FORMATS - 1u)) == 0 ? __builtin_ctz(FORMATS) : -1;
    extern __shared__ __align__(16) uint8_t lds[];
    uint16_t* park = reinterpret_cast<uint16_t*>(lds);
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef u32x4 u32x4_4 __attribute__((aligned(4)));
    typedef u32x4 u32x4_2 __attribute__((aligned(2)));
    typedef f32x4 f32x4_4 __attribute__((aligned(4)));
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    // Neighbouring blocks to one XCD: with every eighth block an XCD reads addresses that are a power of two apart and so lie in few of its L2's channels.
    // The launch alone, 5000 x 2816 of the planner's mix 13.1 -> 9.3 us; whole calls: 11008 x 4096 SPARK_Q0, 512 tokens 78.4 -> 72.5, 900 x 1024
    // planner's mix, 50 tokens 10.6 -> 9.3, 4096 x 4096 registry's mix, 64 tokens 28.7 -> 27.3, 11008 x 4096 OIL8, 256 tokens 58.7 -> 57.9.
    const bool of_x = blockIdx.x >= a.nw;
    const uint32_t id = of_x ? blockIdx.x - a.nw : xcd_chunk(blockIdx.x, a.nw), rb = id / a.bpr, blk = id % a.bpr;
    if (blockIdx.x == 0)
        for (uint32_t i = tid; i < a.ncount; i += 64u * NW) a.arrived[i] = 0u;
    if (of_x) {
        constexpr uint32_t T = 2u * NW;                                      // threads per row: 8-column pieces q, q + T, ...
        const uint32_t r = tid / T, q = tid % T, m = rb * 32u + r;
        const size_t at = (size_t)min(m, a.M - 1u) * a.bpr * 256u + blk * 256u + q * 8u;
        uint4 o[PIECES];
        auto rounded = [](f32x4 f0, f32x4 f1) {
            const bf2 d0 = bf2{(__bf16)f0.x, (__bf16)f0.y}, d1 = bf2{(__bf16)f0.z, (__bf16)f0.w};
            const bf2 d2 = bf2{(__bf16)f1.x, (__bf16)f1.y}, d3 = bf2{(__bf16)f1.z, (__bf16)f1.w};
            return make_uint4(__builtin_bit_cast(uint32_t, d0), __builtin_bit_cast(uint32_t, d1), __builtin_bit_cast(uint32_t, d2), __builtin_bit_cast(uint32_t, d3));
        };
        // 16-byte loads wherever the rows start
        if (a.x_is_f32) {
            const f32x4_4* x = reinterpret_cast<const f32x4_4*>(static_cast<const float*>(a.x) + at);
            f32x4 f[2 * PIECES];
#pragma unroll
            for (uint32_t j = 0; j < 2u * PIECES; ++j) f[j] = x[2u * T * (j >> 1) + (j & 1u)];
#pragma unroll
            for (uint32_t j = 0; j < PIECES; ++j) o[j] = rounded(f[2 * j], f[2 * j + 1]);
        } else {
            const u32x4_2* x = reinterpret_cast<const u32x4_2*>(static_cast<const uint16_t*>(a.x) + at);
#pragma unroll
            for (uint32_t j = 0; j < PIECES; ++j) { const u32x4 v = x[T * j]; o[j] = make_uint4(v.x, v.y, v.z, v.w); }
        }
#pragma unroll
        for (uint32_t j = 0; j < PIECES; ++j) *reinterpret_cast<uint4*>(park + r * kParkPitch + (q + T * j) * 8u) = m < a.M ? o[j] : make_uint4(0u, 0u, 0u, 0u);
    } else {
        float* tb = reinterpret_cast<float*>(lds);                          // decode tables, then the formats of the rows, then the raw blocks
        uint32_t* fmts = reinterpret_cast<uint32_t*>(tb + 256 * 3 + 20);
        uint8_t* raw = reinterpret_cast<uint8_t*>(fmts + 32);
        // R rows of this wavefront (rows past the end repeat the last one); blocks of up to 64 bytes: four lanes per row and one load for all rows, else
        // one load per row.
        constexpr uint32_t LANES = largest_block(FORMATS) <= 64u ? 4u : 1u;
        const uint32_t mine_of = lane / LANES % R, row = min(rb * 32u + wave * R + mine_of, a.rows - 1u) + a.row0;
        uint64_t off;
        uint32_t fmt = ONLY >= 0 ? (uint32_t)ONLY : 0u;
        if (a.blocks) {
            const DevBlock d = a.blocks[(size_t)row * a.bpr + blk];
            off = (uint64_t)d.off16 * 16u;
            if constexpr (ONLY < 0) fmt = d.fmt;
        } else {
            off = ((uint64_t)row * a.bpr + blk) * a.stride;
        }
        // 16-byte pieces of the row's block: one byte per format (full_block_bytes / 16), no table in memory
        constexpr auto sizes = [](int first) { uint64_t t = 0; for (int i = 0; i < 8; ++i) t |= (uint64_t)(full_block_bytes(first + i) / 16u) << (8 * i); return t; };
        const uint32_t pieces = (uint32_t)((fmt < 8u ? sizes(0) : sizes(8)) >> (8u * (fmt & 7u))) & 0xFFu;
        constexpr uint32_t LOADS = LANES == 1u ? R : 1u;
        u32x4 v[LOADS];
        uint32_t f[LOADS];
        const bool own_piece = lane < LANES * R && lane % LANES < pieces;
        if constexpr (LANES > 1u) {
            v[0] = u32x4{0, 0, 0, 0};
            if (own_piece) v[0] = *reinterpret_cast<const u32x4_4*>(a.base + off + lane % LANES * 16u);
        } else {
#pragma unroll
            for (int i = 0; i < (int)R; ++i) {
                const uint64_t o = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)off, i) |
                                   (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(off >> 32), i) << 32;
                f[i] = (uint32_t)__builtin_amdgcn_readlane((int)pieces, i);
                v[i] = u32x4{0, 0, 0, 0};
                if (lane < f[i]) v[i] = *reinterpret_cast<const u32x4_4*>(a.base + o + lane * 16u);
            }
        }
        if (a.need_tables) {
            for (uint32_t i = tid; i < 256u; i += 64u * NW) { tb[i] = a.T->lv8[i]; tb[256 + i] = a.T->t255[i]; tb[512 + i] = a.T->q127[i]; }
        }
        if (tid < 16) tb[768 + tid] = kLv4[tid];
        if (tid < 4) tb[784 + tid] = kLv2[tid];
        if (ONLY < 0 && lane < LANES * R && lane % LANES == 0u) fmts[wave * R + mine_of] = fmt;
        if constexpr (LANES > 1u) {
            if (own_piece) *reinterpret_cast<u32x4*>(raw + (wave * R + mine_of) * a.raw_pitch + lane % LANES * 16u) = v[0];
        } else {
#pragma unroll
            for (int i = 0; i < (int)R; ++i)
                if (lane < f[i]) *reinterpret_cast<u32x4*>(raw + (wave * R + (uint32_t)i) * a.raw_pitch + lane * 16u) = v[i];
        }
        __syncthreads();
        const FullTables L{tb, tb + 256, tb + 512, tb + 768, tb + 784};
        const uint8_t* p = raw + (lane & 31u) * a.raw_pitch;
        const uint32_t mine = ONLY < 0 ? fmts[lane & 31u] : 0u;
        uint4* out = reinterpret_cast<uint4*>(a.wf) + ((size_t)rb * a.bpr * 16u + blk * 16u) * 64u + lane;
        auto decode = [&](auto fc, uint32_t g) {                             // columns 16 g + 8 (lane / 32) .. + 7
            constexpr int F = decltype(fc)::value;
            const float4 lo = decode_full4<F, false>(p, 4u * g + 2u * (lane >> 5), L), hi = decode_full4<F, false>(p, 4u * g + 2u * (lane >> 5) + 1u, L);
            const bf2 d0 = bf2{(__bf16)lo.x, (__bf16)lo.y}, d1 = bf2{(__bf16)lo.z, (__bf16)lo.w};
            const bf2 d2 = bf2{(__bf16)hi.x, (__bf16)hi.y}, d3 = bf2{(__bf16)hi.z, (__bf16)hi.w};
            return make_uint4(__builtin_bit_cast(uint32_t, d0), __builtin_bit_cast(uint32_t, d1), __builtin_bit_cast(uint32_t, d2), __builtin_bit_cast(uint32_t, d3));
        };
        // the formats one after the other, each for the lanes whose row has it; the column groups together, for their LDS reads to overlap
        uint4 o[PIECES];
#define OILHIP_CASE(F)                                                                                                        \
    if constexpr ((FORMATS >> F) & 1u) {                                                                                      \
        if (ONLY >= 0 || mine == (uint32_t)F)                                                                                 \
            _Pragma("unroll") for (uint32_t g = 0; g < PIECES; ++g) o[g] = decode(std::integral_constant<int, F>{}, wave + NW * g); \
    }
        OILHIP_ALL_FORMATS(OILHIP_CASE)
#undef OILHIP_CASE
#pragma unroll
        for (uint32_t g = 0; g < PIECES; ++g) out[(wave + NW * g) * 64u] = o[g];
        return;
    }
    __syncthreads();
    for (uint32_t g = wave; g < 16u; g += NW)
        *reinterpret_cast<uint4*>(a.xf + (((size_t)rb * a.bpr * 16u + blk * 16u + g) * 64u + lane) * 8u) =
            *reinterpret_cast<const uint4*>(park + (lane & 31u) * kParkPitch + g * 16u + (lane >> 5) * 8u);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Y[m][row] = sum_k W[row][k] * X[m][k] for MB batch rows at a time; one
// workgroup per output row, thread t owns weight t of every block in the row
// (Qwen35Engine::gemm, src/adapters/tools/qwen35_engine.cpp:66-81).
template <int MB>
__global__ void __launch_bounds__(256)
gemv_generic_kernel(const uint8_t* __restrict__ payload, const DevBlock* __restrict__ blocks,
                    const DecodeTables* __restrict__ T, const float* __restrict__ x,
                    float* __restrict__ y, uint32_t rows, uint32_t cols, int M, int m0) {
    __shared__ float part[MB][4];
    const uint32_t row = blockIdx.x, t = threadIdx.x, bpr = cols >> 8;
    float acc[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[b] = 0.0f;
    for (uint32_t k = 0; k < bpr; ++k) {
        const DevBlock d = blocks[(size_t)row * bpr + k];
        const uint8_t* cb = payload + (size_t)d.off16 * 16;
        const float v = decode_weight(d.fmt, cb, d.cb_bytes, cb + d.cb_bytes, d.idx_bytes, 256, t, T);
#pragma unroll
        for (int b = 0; b < MB; ++b)
            if (m0 + b < M) acc[b] = __fmaf_rn(v, x[(size_t)(m0 + b) * cols + (size_t)k * 256 + t], acc[b]);
    }
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const float s = wave_sum(acc[b]);
        if ((t & 63) == 0) part[b][t >> 6] = s;
    }
    __syncthreads();
    if (t < MB && m0 + (int)t < M)
        y[(size_t)(m0 + t) * rows + row] = (part[t][0] + part[t][1]) + (part[t][2] + part[t][3]);
}

// Mean squared error of one decoded block against the original weights it encodes:
// FormatRegistry::measure_mse (src/format_registry.cpp:281-289) over dequantize_block_all,
// one thread per block, double accumulation in index order with the fused multiply-add the
// reference build uses, rounded to float at the end.
__global__ void __launch_bounds__(64)
block_mse_kernel(const uint8_t* __restrict__ payload, const DevBlock* __restrict__ blocks,
                 const DecodeTables* __restrict__ T, const float* __restrict__ orig,
                 const uint64_t* __restrict__ start, float* __restrict__ out, uint32_t nblocks) {
    const uint32_t b = blockIdx.x * 64 + threadIdx.x;
    if (b >= nblocks) return;
    const DevBlock d = blocks[b];
    const uint8_t* cb = payload + (size_t)d.off16 * 16;
    const float* o = orig + start[b];
    double s = 0.0;
    for (uint32_t i = 0; i < d.nw; ++i) {
        const double diff = (double)o[i] - (double)decode_weight(d.fmt, cb, d.cb_bytes, cb + d.cb_bytes, d.idx_bytes, d.nw, i, T);
        s = fma(diff, diff, s);
    }
    out[b] = (float)(s / (double)d.nw);
}

}  // namespace

int launch_block_mse(const oilhip_weights& w, const float* d_orig, const uint64_t* d_start, float* d_out, hipStream_t s) {
    const DecodeTables* T = nullptr;
    if (int rc = get_tables(&T)) return rc;
    if (w.nblocks == 0) return OILHIP_OK;
    hipLaunchKernelGGL(block_mse_kernel, dim3((w.nblocks + 63) / 64), dim3(64), 0, s, w.d_payload, w.d_blocks, T,
                       d_orig, d_start, d_out, w.nblocks);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

// full blocks of nominal size: one format at a regular stride (1), or (window streams and sign tiles) the place
// and format of every block from its descriptor (2); 0: neither
static int full_block_layout(const oilhip_weights& w) {
    if (!w.all_full || w.d_out_off) return 0;
    const bool by_stride = w.uniform_fmt >= 0 && w.uniform_stride > 0 && (w.uniform_base & 3u) == 0 &&
                           w.uniform_stride == full_block_bytes(w.uniform_fmt) &&
                           w.uniform_cb == full_block_cb_bytes(w.uniform_fmt) &&
                           w.uniform_cb + w.uniform_idx == w.uniform_stride;
    if (by_stride) return 1;
    bool by_desc = w.seg.by_descriptor();
    for (uint32_t i = 0; by_desc && i < w.seg.nf; ++i)
        by_desc = w.seg.cb_bytes[i] == full_block_cb_bytes((int)w.seg.fmt[i]) &&
                  w.seg.cb_bytes[i] + w.seg.idx_bytes[i] == full_block_bytes((int)w.seg.fmt[i]);
    return by_desc ? 2 : 0;
}

bool dense_prepare_covers(const oilhip_weights& w) { return full_block_layout(w) != 0; }

// Weight rows [row0, row0 + rows) to wf and, with x, M activation rows to xf, in fragment order; clears ncount counters at `arrived`.
// Rows past the end of the last 32-row block hold copies (weights) or zeros.  Returns 1 when the tensor's blocks are not full blocks
// of nominal size.
int launch_dense_prepare(const oilhip_weights& w, uint32_t row0, uint32_t rows, uint16_t* wf, const void* x, bool x_is_f32, uint32_t M,
                         uint16_t* xf, uint32_t* arrived, uint32_t ncount, hipStream_t s) {
    const int layout = full_block_layout(w);
    if (!layout) return 1;
    PrepareArgs a{};
    if (int rc = get_tables(&a.T)) return rc;
    const bool by_stride = layout == 1;
    a.base = w.d_payload + (by_stride ? w.uniform_base : 0u);
    a.blocks = by_stride ? nullptr : w.d_blocks;
    a.stride = w.uniform_stride;
    uint32_t formats = by_stride ? 1u << w.uniform_fmt : 0u, largest = 0;
    for (uint32_t i = 0; !by_stride && i < w.seg.nf; ++i) formats |= 1u << w.seg.fmt[i];
    for (int f = 0; f < 15; ++f)
        if (formats >> f & 1u) largest = std::max(largest, full_block_bytes(f));
    a.need_tables = (formats & (1u << 4 | 1u << 11 | 1u << 13 | 1u << 14)) != 0;
    // a decoder may read a dword past the end; an odd number of 16-byte pieces spreads the rows over the banks
    a.raw_pitch = (largest + 16u) / 16u % 2u ? largest + 16u : largest + 32u;
    a.wf = wf; a.xf = xf; a.x = x;
    a.row0 = row0; a.rows = rows; a.bpr = (uint32_t)(w.cols >> 8);
    a.nw = (rows + 31u) / 32u * a.bpr;
    a.arrived = arrived; a.ncount = arrived ? ncount : 0u;
    a.M = M; a.x_is_f32 = x_is_f32;
    const uint32_t nx = x ? (M + 31u) / 32u * a.bpr : 0u;
    const size_t lds = std::max<size_t>(32u * kParkPitch * 2u, (256u * 3u + 20u + 32u) * 4u + 32u * a.raw_pitch);
    // The two mixes that the planner and the registry produce have kernels of their own: with every decoder in it the kernel takes
    // 17 us for a tensor of any size, most of them to fetch its instructions.
    constexpr uint32_t kPlanner = 1u << OILHIP_OIL1 | 1u << OILHIP_SPARK_Q0;
    constexpr uint32_t kSparkMix = 1u << OILHIP_OIL1_GRP | 1u << OILHIP_OIL2_GRP | 1u << OILHIP_OIL4_GRP | 1u << OILHIP_OIL8_GRP;
    const bool one = (formats & (formats - 1u)) == 0;
    // Twice the wavefronts per workgroup, with half of the work each, while the chip has room for all of them (719 x 3840 of four
    // formats 10 instead of 16 us); half as many beyond (11008 x 4096 OIL8 27 instead of 32 us).
    const bool wide = a.nw + nx <= 4u * (uint32_t)device_cu_count();
#define OILHIP_KERNEL(FORMATS) (wide ? dense_prepare_kernel<FORMATS, 8u> : dense_prepare_kernel<FORMATS, 4u>)
    auto kern = OILHIP_KERNEL(0x7FFFu);
#define OILHIP_CASE(F) if (formats == 1u << F) kern = OILHIP_KERNEL(1u << F);
    OILHIP_ALL_FORMATS(OILHIP_CASE)
#undef OILHIP_CASE
    if (!one && (formats & ~kPlanner) == 0) kern = OILHIP_KERNEL(kPlanner);
    else if (!one && (formats & ~kSparkMix) == 0) kern = OILHIP_KERNEL(kSparkMix);
#undef OILHIP_KERNEL
    hipLaunchKernelGGL(kern, dim3(a.nw + nx), dim3(wide ? 512 : 256), lds, s, a);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

int launch_dequant(const oilhip_weights& w, float* d_out, hipStream_t s) {
    const DecodeTables* T = nullptr;
    if (int rc = get_tables(&T)) return rc;
    if (w.nblocks == 0) return OILHIP_OK;
    {
        const uint32_t g = std::min<uint32_t>((w.nblocks + 3u) / 4u, (uint32_t)device_cu_count() * 16u);
        const int layout = full_block_layout(w);
        const bool by_stride = layout == 1;
        if (layout) {
            const uint8_t* base = w.d_payload + (by_stride ? w.uniform_base : 0u);
            const DevBlock* bl = by_stride ? nullptr : w.d_blocks;
            const int f = by_stride || w.seg.nf == 1 ? w.uniform_fmt : -1;
#define OILHIP_CASE(F) case F: hipLaunchKernelGGL((dequant_full_kernel<F>), dim3(g), dim3(256), 0, s, base, w.uniform_stride, bl, T, d_out, w.nblocks); break;
            switch (f) {
                OILHIP_ALL_FORMATS(OILHIP_CASE)
                default: hipLaunchKernelGGL((dequant_full_kernel<-1>), dim3(g), dim3(256), 0, s, base, 0u, bl, T, d_out, w.nblocks); break;
            }
#undef OILHIP_CASE
            OILHIP_HIP(hipGetLastError());
            return OILHIP_OK;
        }
    }
    const uint32_t grid = w.nblocks < (1u << 20) ? w.nblocks : (1u << 20);
    hipLaunchKernelGGL(dequant_kernel, dim3(grid), dim3(256), 0, s, w.d_payload, w.d_blocks,
                       w.d_out_off, T, d_out, w.nblocks, 256u);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

int launch_gemv_generic(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s) {
    const DecodeTables* T = nullptr;
    if (int rc = get_tables(&T)) return rc;
    constexpr int MB = 4;
    for (int m0 = 0; m0 < M; m0 += MB) {
        hipLaunchKernelGGL(gemv_generic_kernel<MB>, dim3((uint32_t)w.rows), dim3(256), 0, s,
                           w.d_payload, w.d_blocks, T, d_x, d_y, (uint32_t)w.rows, (uint32_t)w.cols, M, m0);
        OILHIP_HIP(hipGetLastError());
    }
    return OILHIP_OK;
}

}  // namespace oilhip
