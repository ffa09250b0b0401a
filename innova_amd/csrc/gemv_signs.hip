// gemv_signs.hip -- decode GEMV for tensors whose blocks are SPARK_Q0 and OIL1 in any mix (the 1.50-bpw stacks FormatPlanner::allocate
// produces, src/format_planner.cpp:133-315, and either format alone): Qwen35Engine::gemm (src/adapters/tools/qwen35_engine.cpp:47-85)
// fused with dequantize_block_all (src/block_codec.cpp:576-720), one to four activation rows per launch.
//
// Both formats say the same thing: a run of 32 weights is an FP16 number times 32 signs, and an OIL1 run has the sign + everywhere.  So a
// tile of 16 rows by one block is four INT8 matrix instructions (16x16x64) whatever its blocks are.  One operand are the signs as bytes of
// +-64, two vector instructions per four weights (a shift, and one that masks and sets the magnitude).  The other are the activations as
// four signed byte digits relative to the largest magnitude of their run (31 bits).  (Not of their block: where an outlier meets a scale of 0 or a small one,
// the other runs would be left with few bits.  16 blocks, x N(0, 1), an outlier of 1e6 in each over a run of scale 0: 1.4e-4 with one power of two per
// block, 0.8e-7 with one per run.)  The digits of the run pair 2 q, 2 q + 1 are rows
// 4 q .. 4 q + 3 and are zero in the lane groups of other runs, so a lane gets the four digit sums of the two runs whose signs and scales it
// holds: they become one float, exact but for its rounding, meet the two scales in FP32 (a scale times its run's power of two is exact), and no lane ever holds another row's sum.
//
// A wavefront keeps the digits of its one to four column blocks in registers and walks down the workgroup's tiles; every workgroup packs
// the activations itself (each wavefront its own blocks, without a barrier), so there is no second launch and no scratch.  The wavefronts'
// sums meet in LDS once per 16 tiles, in a fixed order.
//
// What bounds it: vector issue (about 60 instructions per tile of one block, 30 of them making sign bytes; as many to pack a block of activations) and, below
// ten tiles a workgroup, latency: the launch, the tiles' places, the blocks, each behind the other.  Before (window streams, gemv_seg.hip; several rows
// gemv_any_multi.hip) -> now, us, planner's mix, launches of a graph over a ring of tensors in memory:
//   one row   649 x 768 4.0 -> 2.5   4096 x 4096 5.3 -> 3.9   12288 x 4096 8.1 -> 5.3   22016 x 4096 12.3 -> 7.1   60000 x 4096 23.6 -> 13.6
//             4096 x 11008 8.1 -> 6.2   SPARK_Q0 alone 11008 x 4096 10.8 -> 5.3   with the norm 12288 x 4096 8.7 -> 5.9
//   two       4096 x 4096 6.7 -> 4.7   22016 x 4096 14.8 -> 8.7   4096 x 11008 15.3 -> 9.8   with the norm 12288 x 4096 13.2 -> 7.5
//   three     1000 x 1280 5.6 -> 3.7   11008 x 4096 11.8 -> 8.2;   four   11008 x 4096 11.8 -> 9.1   with the norm 12288 x 4096 13.6 -> 10.7
// (One power of two per run instead of per block is an instruction more per tile of one block and row, and 82 vector instructions instead of 93 to pack a block; the
// sums of runs held as floats stand behind the loop.  Launches of many tiles up to 2 % slower for it, the others 1 to 5 % faster.)
// Error against 64 bits (2-norm, 4096 columns, one row) 1.1e-7 -> 0.8e-7.
// Level or slower: an operand of 0 and 1 with the activations' sums as the matrix instruction's addend (24 registers per block instead of 16); sums over
// the lane groups in front of LDS instead of behind it (22016 x 4096 8.5 us against 6.9, with the loop's waits then counting no loads).
//
// Runs whose activations are not finite, or too small for the power of two that undoes the digits, add up their signed activations in FP32.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "oil4_lds.h"

namespace oilhip {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x3 __attribute__((ext_vector_type(3)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// wavefronts of a CU: four per SIMD with 128 registers each, or two where the digits take more
constexpr uint32_t waves_for(int M) { return M <= 2 ? 16u : 8u; }
enum Form { kPlain = 0, kSwiglu = 1, kNorm = 2 };
// tiles between two meetings of the wavefronts' sums: as many as LDS takes beside the digits
constexpr uint32_t chunk_for(int M) { return M == 1 ? 16u : 8u; }
// column blocks of a wavefront, at most (sixteen registers of digits per block and activation row), and its loads in flight per column block
// (what is read ahead of a further chunk or part takes registers too)
constexpr int most_blocks(int M, int XF, bool loop) { return M == 1 ? (loop ? 2 : XF == kNorm ? 3 : 4) : M == 2 ? 1 : M == 3 || !loop ? 2 : 1; }
constexpr int loads_ahead(int M, int CB) { return CB == 1 ? 4 : CB == 2 && M < 4 ? 2 : 1; }

struct SignArgs {
    const uint8_t* W;                      // SignTiles' buffer (common.h)
    const float *x, *x2, *norm_w;
    float *y, *xn;
    uint32_t wbytes, rows, bpr, ntiles, ldx, parts, per, t_base, t_rem, waves;
};

__device__ __forceinline__ uint32_t scalar(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ float half_lo(uint32_t v) { return (float)__builtin_bit_cast(_Float16, (unsigned short)v); }

// four signs as bytes: bit set -> -64, clear -> +64; bits K, K + 8, K + 16, K + 24 of s.  (Inverted: the power of two that undoes the
// digits is negative.)
template <int K>
__device__ __forceinline__ int sign_bytes(uint32_t s, uint32_t tops, uint32_t size) { return (int)(((s << (7 - K)) & tops) | size); }

// LOOP: more than one chunk of tiles or part of K
template <int M, int CB, int XF, bool LOOP>
__global__ void __launch_bounds__(64 * waves_for(M))
gemv_signs_kernel(const SignArgs a) {
    constexpr int P = loads_ahead(M, CB);
    constexpr uint32_t CHUNK = chunk_for(M);
    // (all arguments at once: read where they are needed, each adds a scalar load's latency)
    asm volatile("" :: "s"(a.W), "s"(a.x), "s"(a.y), "s"(a.wbytes), "s"(a.rows), "s"(a.bpr), "s"(a.ntiles), "s"(a.ldx), "s"(a.t_base), "s"(a.t_rem), "s"(a.waves));
    extern __shared__ __align__(16) uint32_t smem[];
    const uint32_t lane = threadIdx.x & 63u, wave = scalar(threadIdx.x >> 6), waves = a.waves;
    const uint32_t li = lane & 15u, q = lane >> 4;
    const uint32_t wg = blockIdx.x, t_begin = wg * a.t_base + (wg < a.t_rem ? wg : a.t_rem), t_end = t_begin + a.t_base + (wg < a.t_rem ? 1u : 0u);
    uint32_t* mine = smem + wave * ((uint32_t)(CB * M) * 256u + 16u);      // digits (or floats) of this wavefront's blocks, 1 KB each, and 64 bytes of zeros
    mine[(uint32_t)(CB * M) * 256u + li] = 0u;
    float* sums = reinterpret_cast<float*>(smem) + waves * ((uint32_t)(CB * M) * 256u + 16u);      // [tile of the chunk][wavefront][row of y][lane]
    float* ssq_part = sums + (LOOP ? CHUNK : t_end - t_begin) * waves * (uint32_t)(64 * M);   // kNorm: [wavefront][row of y], negative where x or its weight is not finite
    const auto wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.W), (short)0, (int)a.wbytes, 0x00020000);
    const uint32_t* heads = reinterpret_cast<const uint32_t*>(a.W);        // [block of the row][tile]: {place / 16, mask of SPARK_Q0 rows}
    const uint32_t row_bit = 1u << li, rows_before = row_bit - 1u, at_mean = 16u * li + 4u * q, at_sign = 16u * li + 12u * q;
    const uint32_t col = 32u * (lane >> 3) + (lane & 7u);                  // a lane packs columns col + 8 j of a block
    uint32_t tops = 0x80808080u, size = 0x40404040u;                       // in registers: one instruction masks and sets the magnitude
    asm volatile("" : "+s"(tops), "+v"(size));

    // what a wavefront reads of the activations and the tiles' places for a chunk of tiles and a part of K (place of tile i in lane i, its mask in lane 16 + i)
    struct Input { uint32_t head[CB]; float v[CB][M][4], u[CB][XF == kSwiglu ? M : 1][4]; };
    auto tiles_of = [&](uint32_t chunk) { return !LOOP || t_end - chunk < CHUNK ? t_end - chunk : CHUNK; };
    auto block_of = [&](uint32_t part, int s, bool& live) {
        const uint32_t first = LOOP ? part * a.per : 0u, last = LOOP && first + a.per < a.bpr ? first + a.per : a.bpr, b = first + (uint32_t)s * waves + wave;
        live = b < last;
        return live ? b : a.bpr - 1u;
    };
    auto fetch = [&](Input& in, uint32_t chunk, uint32_t part) {
        const uint32_t n = tiles_of(chunk);
        bool live;
#pragma unroll
        for (int s = 0; s < CB; ++s) in.head[s] = heads[2u * (block_of(part, s, live) * a.ntiles + chunk + (li < n ? li : n - 1u)) + (q & 1u)];
#pragma unroll
        for (int s = 0; s < CB; ++s) {
            const uint32_t b = 256u * block_of(part, s, live);
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    in.v[s][m][j] = (a.x + (size_t)m * a.ldx + b)[col + 8 * j];
                    if constexpr (XF == kSwiglu) in.u[s][m][j] = (a.x2 + (size_t)m * a.ldx + b)[col + 8 * j];
                    if constexpr (XF == kNorm) if (m == 0) in.u[s][0][j] = (a.norm_w + b)[col + 8 * j];
                }
        }
    };

    i32x4 dig[CB][M][4];
    float undo[CB][M], ssq[M], endless[M];                                             // undo: of the run that this lane packs, lane / 8; positive where it is held as floats; endless: kNorm: 0, or NaN where x or a
                                                                           // weight of the norm is not finite
    uint32_t slow = 0;                                                     // bit s * M + m: runs of that block add up in FP32
#pragma unroll
    for (int m = 0; m < M; ++m) ssq[m] = endless[m] = 0.0f;
    // one block of one row to digits
    auto pack = [&](int s, int m, float (&f)[4], const float (&u)[4], bool on, bool counts) {
#pragma unroll
        for (int j = 0; j < 4; ++j) f[j] = on ? f[j] : 0.0f;               // a wavefront without a block of its own here: zeros
        if constexpr (XF == kSwiglu) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (M == 1) f[j] = (f[j] * __builtin_amdgcn_rcpf(1.0f + __expf(-f[j]))) * u[j];
                else f[j] = (f[j] * (1.0f / (1.0f + expf(-f[j])))) * u[j];
            }
        }
        if constexpr (XF == kNorm) {
#pragma unroll
            for (int j = 0; j < 4; ++j) endless[m] = fmaf(f[j], 0.0f, fmaf(u[j], 0.0f, endless[m]));
            ssq[m] += counts ? (f[0] * f[0] + f[1] * f[1]) + (f[2] * f[2] + f[3] * f[3]) : 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) f[j] *= 1.0f + u[j];
        }
        uint32_t top = 0;                                                  // the largest magnitude of this lane's run as a bit pattern
#pragma unroll
        for (int j = 0; j < 4; ++j) top = max(top, __float_as_uint(f[j]) & 0x7FFFFFFFu);
        top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
        top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x4E, 0xF, 0xF, true));    // [2,3,0,1]
        top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x141, 0xF, 0xF, true));   // row_half_mirror
        // to [2^30, 2^31), one less where the top digit would pass 127
        int ex = 30 - ((int)(top >> 23) - 127) - ((top & 0x7FFFFFu) > 0x7EFEFEu ? 1 : 0);
        ex = top == 0u ? 0 : ex;
        const bool odd = top >= 0x7F800000u || ex > 119;                   // (a half is a multiple of 2^-24: times 2^-119 / 64 it is still exact)
        undo[s][m] = top >= 0x7F800000u ? 64.0f : odd ? 1.0f : -ldexpf(1.0f, -ex - 6);
        slow = (slow & ~(1u << (s * M + m))) | (__ballot(odd) ? 1u << (s * M + m) : 0u);
        uint32_t b[4];                                                     // signed digits: the bytes of X + 128 (1 + 2^8 + 2^16 + 2^24), less 128 each
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = odd ? __float_as_uint(f[j]) : ((uint32_t)(int)rintf(ldexpf(f[j], ex)) + 0x80808080u) ^ 0x80808080u;
        // digit d (of a run of floats: byte d) of the four columns in one dword: piece (q, d) of 64 bytes, run of the pair, dword lane % 8
        const uint32_t l01 = __builtin_amdgcn_perm(b[1], b[0], 0x05010400u), h01 = __builtin_amdgcn_perm(b[1], b[0], 0x07030602u);
        const uint32_t l23 = __builtin_amdgcn_perm(b[3], b[2], 0x05010400u), h23 = __builtin_amdgcn_perm(b[3], b[2], 0x07030602u);
        uint32_t* area = mine + (uint32_t)(s * M + m) * 256u;
        uint32_t* o = area + 64u * q + li;
        o[0] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
        o[16] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
        o[32] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
        o[48] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
        // operand row 4 q + d: digit d of lane group q's runs, zero in the other lane groups
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const i32x4* p = reinterpret_cast<const i32x4*>((li >> 2) == q ? area + 64u * q + 16u * (li & 3u) : mine + (uint32_t)(CB * M) * 256u);
#pragma unroll
        for (int k = 0; k < 4; ++k) dig[s][m][k] = p[k];
        if constexpr (LOOP || M > 2 || CB > 3) __builtin_amdgcn_sched_barrier(0);    // one block's floats become digits at a time: registers
    };
    // of run 2 q + r: lane 8 r of the row of sixteen, which a multiplication takes as it reads its operand (row_newbcast)
    auto undo_of = [&](int s, int m, auto r) {
        return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(undo[s][m]), 0x150 + 8 * decltype(r)::value, 0xF, 0xF, true));
    };
    auto barrier = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    // (m is the same for a wavefront; a lane per wavefront's sum, then over the sixteen lanes: one read of LDS instead of one behind the other)
    auto norm_of = [&](uint32_t m, bool& finite) {
        const float p = li < waves ? ssq_part[li * (uint32_t)M + m] : 0.0f;
        float t = fabsf(p);
        auto add = [&](auto how) { t += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(t), decltype(how)::value, 0xF, 0xF, true)); };
        add(std::integral_constant<int, 0xB1>{});                          // quad_perm [1,0,3,2]
        add(std::integral_constant<int, 0x4E>{});                          // [2,3,0,1]
        add(std::integral_constant<int, 0x141>{});                         // row_half_mirror
        add(std::integral_constant<int, 0x140>{});                         // row_mirror
        finite = __ballot((int)__float_as_uint(p) < 0) == 0u;
        return 1.0f / sqrtf(t / (float)(256u * a.bpr) + 1e-6f);
    };

    Input in;
    fetch(in, t_begin, 0u);
    for (uint32_t chunk = t_begin, part = 0;;) {
        const uint32_t n = tiles_of(chunk);
        const bool ends = !LOOP || part + 1u == a.parts, over = ends && (!LOOP || t_end - chunk <= CHUNK);
        uint32_t head[CB];
        bool live[CB];
#pragma unroll
        for (int s = 0; s < CB; ++s) { head[s] = in.head[s]; block_of(part, s, live[s]); }
        Input next;
        if constexpr (LOOP) fetch(next, ends && !over ? chunk + CHUNK : chunk, over ? part : ends ? 0u : part + 1u);
        u32x3 w[P][CB];
        auto load = [&](int p, int s, uint32_t i) {
            const uint32_t at = i < n ? i : n - 1u, off = i < n && live[s] ? 0u : 0x80000000u;     // past the end: out of range, zeros and no fetch
            const uint32_t place = (uint32_t)__builtin_amdgcn_readlane((int)head[s], (int)at), mask = (uint32_t)__builtin_amdgcn_readlane((int)head[s], (int)(16u + at));
            const uint32_t before = 32u * (uint32_t)__builtin_popcount(mask & rows_before) + ((mask & row_bit) ? at_sign : at_mean);
            w[p][s] = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(wrs, before + off, place * 16u, 0));
        };
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int s = 0; s < CB; ++s) load(p, s, (uint32_t)p);
        __builtin_amdgcn_sched_barrier(0);
        if (!LOOP || a.parts > 1u || chunk == t_begin) {
#pragma unroll
            for (int s = 0; s < CB; ++s)
#pragma unroll
                for (int m = 0; m < M; ++m) pack(s, m, in.v[s][m], in.u[s][XF == kSwiglu ? m : 0], live[s], chunk == t_begin);
        }
        auto share_norm = [&] {
            if (!ends || chunk != t_begin) return;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const float t = oil4::wave_sum(ssq[m]);
                const bool any = __ballot(endless[m] != 0.0f) != 0u;
                if (lane == 0) ssq_part[wave * (uint32_t)M + (uint32_t)m] = __uint_as_float((__float_as_uint(t) & 0x7FFFFFFFu) | (any ? 0x80000000u : 0u));
            }
        };
        if constexpr (XF == kNorm && M > 1) share_norm();                  // (one row: below, where the loads have arrived; several: registers)
        float acc[M];
        auto multiply = [&](int p, int s, uint32_t i) {
            const uint32_t mask = (uint32_t)__builtin_amdgcn_readlane((int)head[s], (int)(16u + i));
            const bool spark = (mask & row_bit) != 0u;
            const u32x3 o = w[p][s];
            const uint32_t s0 = spark ? __builtin_amdgcn_alignbit(o.y, o.x, 16) : 0xFFFFFFFFu, s1 = spark ? o.z : 0xFFFFFFFFu;
            const float c0 = half_lo(o.x), c1 = half_lo((spark ? o.y : o.x) >> 16);
            const i32x4 b0 = {sign_bytes<0>(s0, tops, size), sign_bytes<1>(s0, tops, size), sign_bytes<2>(s0, tops, size), sign_bytes<3>(s0, tops, size)};
            const i32x4 b1 = {sign_bytes<4>(s0, tops, size), sign_bytes<5>(s0, tops, size), sign_bytes<6>(s0, tops, size), sign_bytes<7>(s0, tops, size)};
            const i32x4 b2 = {sign_bytes<0>(s1, tops, size), sign_bytes<1>(s1, tops, size), sign_bytes<2>(s1, tops, size), sign_bytes<3>(s1, tops, size)};
            const i32x4 b3 = {sign_bytes<4>(s1, tops, size), sign_bytes<5>(s1, tops, size), sign_bytes<6>(s1, tops, size), sign_bytes<7>(s1, tops, size)};
            const i32x4 zero = {0, 0, 0, 0};
            i32x4 d0[M], d1[M];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                d0[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(dig[s][m][0], b0, zero, 0, 0, 0);
                d1[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(dig[s][m][2], b2, zero, 0, 0, 0);
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                d0[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(dig[s][m][1], b1, d0[m], 0, 0, 0);
                d1[m] = __builtin_amdgcn_mfma_i32_16x16x64_i8(dig[s][m][3], b3, d1[m], 0, 0, 0);
            }
            // (the wait states that a reader of the last result needs, in front of the branch below: the compiler counts one way only)
#pragma unroll
            for (int m = 0; m < M; ++m) asm volatile("s_nop 7" : "+v"(d0[m]), "+v"(d1[m]));
#pragma unroll
            for (int m = 0; m < M; ++m) {
                auto one = [](const i32x4& d) { return fmaf((float)(d[3] * 256 + d[2]), 65536.0f, (float)(d[1] * 256 + d[0])); };
                float f0 = one(d0[m]), f1 = one(d1[m]);
                if (__builtin_expect((slow & (1u << (s * M + m))) != 0u, 0)) {   // uniform; behind the loop: a branch that is not taken
                    const uint8_t* x = reinterpret_cast<const uint8_t*>(mine + (uint32_t)(s * M + m) * 256u + 64u * q);
                    auto floats = [&](float f, auto r, uint32_t signs, const uint8_t* run) {
                        // (a 64th of each beside an infinity: finite ones must not add up to the other one)
                        const bool infinite = undo_of(s, m, r) == 64.0f;
                        float e = 0.0f;
#pragma unroll 1
                        for (uint32_t k = 0; k < 32u; ++k) {
                            const uint8_t* p = run + 4u * (k & 7u) + (k >> 3);                  // bytes 64 apart
                            const uint32_t b = p[0] | p[64] << 8 | p[128] << 16 | (uint32_t)p[192] << 24;
                            const float v = __uint_as_float(b ^ (~(signs << (31u - k)) & 0x80000000u));
                            e += infinite ? v * 0.015625f : v;
                        }
                        return undo_of(s, m, r) > 0.0f ? e : f;
                    };
                    f0 = floats(f0, std::integral_constant<int, 0>{}, s0, x);
                    f1 = floats(f1, std::integral_constant<int, 1>{}, s1, x + 32);
                }
                acc[m] = fmaf(undo_of(s, m, std::integral_constant<int, 0>{}) * c0, f0, acc[m]);
                acc[m] = fmaf(undo_of(s, m, std::integral_constant<int, 1>{}) * c1, f1, acc[m]);
            }
        };
        // the loop is left, never skipped within: so every wait for a load counts the loads behind it
        bool more = true;
        for (uint32_t i = 0; more;) {
#pragma unroll
            for (int p = 0; p < P; ++p) {
#pragma unroll
                for (int m = 0; m < M; ++m) acc[m] = 0.0f;
#pragma unroll
                for (int s = 0; s < CB; ++s) {
                    multiply(p, s, i);
                    if (CB > 1) load(p, s, i + (uint32_t)P);
                }
                float* o = sums + (i * waves + wave) * (uint32_t)(64 * M) + lane;
#pragma unroll
                for (int m = 0; m < M; ++m) o[64 * m] = LOOP && part ? o[64 * m] + acc[m] : acc[m];
                if (++i == n) { more = false; break; }
                if (CB == 1) load(p, 0, i + (uint32_t)(P - 1));
            }
        }
        if constexpr (XF == kNorm && M == 1) share_norm();
        if (ends) {
            barrier();
            // a wavefront per tile and row of y: first over the wavefronts, four sums side by side, then over the lane groups
            for (uint32_t i = wave; i < n * (uint32_t)M; i += waves) {
                const uint32_t t = i / (uint32_t)M, m = i % (uint32_t)M;
                const float* p = sums + (t * waves * (uint32_t)M + m) * 64u + lane;
                float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                for (uint32_t j = 0; j < waves; j += 4u)
#pragma unroll
                    for (uint32_t e = 0; e < 4u; ++e) s[e] += j + e < waves ? p[(j + e) * (uint32_t)(64 * M)] : 0.0f;
                float y = (s[0] + s[1]) + (s[2] + s[3]);
                const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
                y = __uint_as_float(h[0]) + __uint_as_float(h[1]);
                const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
                y = __uint_as_float(r[0]) + __uint_as_float(r[1]);
                if constexpr (XF == kNorm) {
                    // a sum of squares past the largest float makes every finite x zero, before it meets a weight
                    bool finite;
                    const float r = norm_of(m, finite);
                    y = r == 0.0f && finite ? 0.0f : y * r;
                }
                const uint32_t row = (chunk + t) * 16u + lane;
                if (lane < 16u && row < a.rows) a.y[(size_t)m * a.rows + row] = y;
            }
            if constexpr (XF == kNorm && M > 1) {
                // the normalised rows: a workgroup writes every gridDim.x-th block of them
                if (a.xn && chunk == t_begin)
                    for (uint32_t b = wg; b < a.bpr; b += gridDim.x)
                        for (uint32_t o = threadIdx.x; o < 256u * M; o += blockDim.x) {
                            const uint32_t m = o >> 8, c = 256u * b + (o & 255u);
                            bool finite;
                            a.xn[(size_t)m * a.ldx + c] = a.x[(size_t)m * a.ldx + c] * norm_of(m, finite) * (1.0f + a.norm_w[c]);
                        }
            }
            if (over) break;
            barrier();
        }
        chunk = ends ? chunk + CHUNK : chunk;
        part = ends ? 0u : part + 1u;
        if constexpr (LOOP) in = next;
    }
}

template <int M, int CB, int XF, bool LOOP>
int launch_form(const SignArgs& a, uint32_t wgs, hipStream_t s) {
    static std::atomic<uint64_t> raised{0};
    auto kern = gemv_signs_kernel<M, CB, XF, LOOP>;
    if (int rc = ensure_max_lds(raised, reinterpret_cast<const void*>(kern), 160 * 1024)) return rc;
    const size_t lds = (size_t)a.waves * (CB * M * 1024u + 64u + (LOOP ? chunk_for(M) : a.t_base + (a.t_rem ? 1u : 0u)) * 256u * M + 4u * M);
    hipLaunchKernelGGL(kern, dim3(wgs), dim3(64u * a.waves), lds, s, a);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

// K in parts that a workgroup's wavefronts cover at once, evenly, and the tiles in as many workgroups as the chip holds.  Returns 1 where LOOP is
// false and the call needs more than one part or chunk.
template <int M, int XF, bool LOOP>
int launch_rows(SignArgs a, hipStream_t s) {
    constexpr uint32_t W = waves_for(M), most = W * (uint32_t)most_blocks(M, XF, LOOP);
    a.parts = (a.bpr + most - 1u) / most;
    a.per = (a.bpr + a.parts - 1u) / a.parts;
    a.parts = (a.bpr + a.per - 1u) / a.per;
    const uint32_t cb = (a.per + W - 1u) / W;
    a.waves = (a.per + cb - 1u) / cb;
    const uint32_t wgs = std::min(a.ntiles, (uint32_t)device_cu_count() * (W / a.waves));
    a.t_base = a.ntiles / wgs;
    a.t_rem = a.ntiles % wgs;
    if (!LOOP && (a.parts > 1u || a.t_base + (a.t_rem ? 1u : 0u) > chunk_for(M))) return 1;
    if constexpr (most_blocks(M, XF, LOOP) > 1) if (cb == 2u) return launch_form<M, 2, XF, LOOP>(a, wgs, s);
    if constexpr (most_blocks(M, XF, LOOP) > 2) {
        if (cb == 3u) return launch_form<M, 3, XF, LOOP>(a, wgs, s);
        if constexpr (most_blocks(M, XF, LOOP) > 3) if (cb == 4u) return launch_form<M, 4, XF, LOOP>(a, wgs, s);
    }
    return launch_form<M, 1, XF, LOOP>(a, wgs, s);
}

template <int M, int XF>
int launch_any(const SignArgs& a, hipStream_t s) {
    const int rc = launch_rows<M, XF, false>(a, s);
    return rc == 1 ? launch_rows<M, XF, true>(a, s) : rc;
}

template <int XF>
int launch_pass(const SignArgs& a, int M, hipStream_t s) {
    return M == 1 ? launch_any<1, XF>(a, s) : M == 2 ? launch_any<2, XF>(a, s) : M == 3 ? launch_any<3, XF>(a, s) : launch_any<4, XF>(a, s);
}

}  // namespace

// One and two rows always, also of tensors that are tall and wide, where every chunk of tiles packs part after part (two rows, planner's mix, us before -> here: 12288 x 8192
// 18.4 -> 10.8, 28672 x 8192 38.8 -> 18.6, 30000 x 16640 68.0 -> 44.3, 12000 x 20480 48.3 -> 22.4, 2048 x 8192 7.3 -> 7.3).  Three and four while eight wavefronts hold the digits of the whole row (two blocks each): beyond, every workgroup packs part after
// part, which costs more than the other kernel's pre-pass, us there -> here: 11008 x 4096 11.8 -> 8.2 (3 rows), 11.8 -> 9.1 (4); 60000 x 4096 40.1 -> 25.2, 40.2 -> 34.9;
// 8192 x 5120 10.5 -> 11.9, 10.5 -> 12.0; 4096 x 11008 13.5 -> 17.1 (4).  Five rows and more are two passes: 11008 x 4096, 8 rows 13.9 -> 18.
bool signs_fastest(const oilhip_weights& w, int M) {
    return w.seg.sign_tiles && (M <= 2 || (M <= kSignRows && (w.cols >> 8) <= waves_for(M) * (uint32_t)most_blocks(M, kPlain, false)));
}

// Returns 1 when the tensor is not stored as sign tiles.
int launch_gemv_signs(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s, const MultiInput& in, uint32_t ldx) {
    if (!w.seg.sign_tiles) return 1;
    if (!ldx) ldx = (uint32_t)w.cols;
    for (int m0 = 0; m0 < M; m0 += kSignRows) {
        const size_t skip = (size_t)m0 * ldx;
        const SignArgs a{w.d_payload, d_x + skip, in.x2 ? in.x2 + skip : nullptr, in.norm_w, d_y + (size_t)m0 * w.rows, in.xn ? in.xn + skip : nullptr,
                         (uint32_t)w.alloc_bytes, (uint32_t)w.rows, (uint32_t)(w.cols >> 8), w.seg.sign_tiles, ldx, 0u, 0u, 0u, 0u, 0u};
        const int m = std::min(M - m0, kSignRows);
        if (int rc = in.x2 ? launch_pass<kSwiglu>(a, m, s) : in.norm_w ? launch_pass<kNorm>(a, m, s) : launch_pass<kPlain>(a, m, s)) return rc;
    }
    return OILHIP_OK;
}

}  // namespace oilhip
