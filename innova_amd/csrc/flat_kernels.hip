// flat_kernels.hip -- the reference's flat-codebook matmul entry points on the
// device: one caller-supplied codebook, plain row-major index matrices.
//   oil::kernel::oil8_gemm / oil4_gemm          src/kernel_oil8.cpp, src/kernel_oil4.cpp
//   oil::adapters::prod::gemv_{spark,oil4,oil8} src/kernel_production.cpp:79-128,345-364
//   oil::engines::OIL{8,4,2}Engine::quant_gemm  src/oil_engines_oil{8,4,2}.cpp
#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"
#include "oil4_lds.h"

namespace oilhip {
namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

// sum over the wavefront, in lane 63
__device__ __forceinline__ float wave_sum(float v) {
    v += oil4::dpp_quad_xor1(v);
    v += oil4::dpp_quad_xor2(v);
    v += oil4::dpp_half_mirror(v);
    v += oil4::dpp_row_mirror(v);
    v += oil4::dpp_row_bcast15(v);
    v += oil4::dpp_row_bcast31(v);
    return v;
}

// FP16 codebook entry exactly as fp16_to_float (src/kernel_oil4.cpp:15-29).
__device__ __forceinline__ float flat_half(uint16_t h) {
    const uint32_t e = (h >> 10) & 31u, m = h & 0x3FFu;
    if (e == 31u && m != 0u) return __uint_as_float(0x7FC00000u);
    return half_bits_to_float(h);
}

// One row (or R rows) of codes against activations: kernel::oil4_gemm, the production GEMVs and the index-byte forms that
// gemv_oil8.hip does not take.  BITS = 8: a byte per weight, codebook of 256 floats; 4: a nibble, FP16 codebook of 16; 2:
// SPARK ternary (0 -> -1, 1 -> 0, 2 and 3 -> +1).
// What bounds it: bytes from memory at the large sizes, the launch at the small ones; the form this replaces (a workgroup
// per row, a byte load, a shift and a table read in LDS per weight and thread) was bound by its instructions.  A lane takes
// UNIT consecutive weights of every row with one load, at any alignment, and the activations of those weights once for
// the R rows; nibbles and ternary codes become FP16 pairs by byte permutes of a codebook held in registers (16 entries are
// two 8-byte tables for each half of an FP16 value; the code's top bit selects between them) and enter the FP32 sum
// through v_fma_mix.  The four wavefronts of a workgroup take every fourth 64 * UNIT weights of the same rows, so that a
// short row still occupies them all.  4096 x 4096, M = 1, before -> after: SPARK 10.9 -> 6.7 us (the host's launch rate); M = 4:
// SPARK 19.9 -> 7.6, production OIL4 22.1 -> 9.0, M = 8: OIL8 63 -> 16; oil4_gemm M = 6, 3000 x 2044: 42.6 -> 20.8.
struct FlatRows {
    const uint8_t* w;            // row r starts at byte r * row_bytes; PAIR: row (m, n) at byte ((m * rows + n) * K) / 2
    const void* cb;
    const float* x;              // activation row b at x + b * K; PAIR: row n
    float* y;                    // y[b * rows + r]; PAIR: y[m * rows + n]
    float scale;
    uint32_t rows, K, batch;     // PAIR: batch = M
    uint64_t row_bytes;
    const uint8_t* last = nullptr;   // the codes' last dword, when a lane's codes can start off a dword; else nullptr
};

// The dword at an address that was computed as a number.  The address space is said because a pointer made from an integer is generic to
// the compiler: a flat load counts as an LDS access too and returns out of order, so the next wait on LDS waits for memory.
__device__ __forceinline__ uint32_t load_dword(uintptr_t at) { return *(const __attribute__((address_space(1))) uint32_t*)at; }
typedef uint32_t u32x4_at4 __attribute__((ext_vector_type(4), aligned(4)));
// N neighbouring dwords, dword-aligned, four to a load
template <int N>
__device__ __forceinline__ void load_dwords(uint32_t (&d)[N], uintptr_t at) {
#pragma unroll
    for (int i = 0; i + 4 <= N; i += 4) {
        const u32x4_at4 v = *(const __attribute__((address_space(1))) u32x4_at4*)(at + 4 * i);
        d[i] = v.x; d[i + 1] = v.y; d[i + 2] = v.z; d[i + 3] = v.w;
    }
#pragma unroll
    for (int i = N / 4 * 4; i < N; ++i) d[i] = load_dword(at + 4 * i);
}
// 32 bits that start at bit `bit` behind p, from the one or two dwords they lie in; `last` keeps the second inside the array.
__device__ __forceinline__ uint32_t load_bits32(const uint8_t* p, uint32_t bit, const uint8_t* last) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(p) + (bit >> 3), q = at & ~(uintptr_t)3, l = reinterpret_cast<uintptr_t>(last);
    const uint32_t a = load_dword(q), b = load_dword(q < l ? q + 4 : l);
    return __builtin_amdgcn_alignbit(b, a, (uint32_t)(at & 3) * 8u + (bit & 7u));
}
__device__ __forceinline__ float4 load_f4(const float* p) { float4 v; __builtin_memcpy(&v, p, 16); return v; }

template <int BITS>
struct FlatBook;

template <>
struct FlatBook<4> {                                       // low bytes of entries 0-3, 4-7, 8-11, 12-15, then high bytes
    uint32_t lo[4], hi[4];
    __device__ __forceinline__ void init(const void* cb, const float*) {
        const uint16_t* c = reinterpret_cast<const uint16_t*>(cb);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            lo[g] = hi[g] = 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) { const uint32_t h = c[4 * g + j]; lo[g] |= (h & 255u) << (8 * j); hi[g] |= (h >> 8) << (8 * j); }
        }
    }
    // eight nibbles of d -> f(i, value), i = 0 .. 7
    template <class F>
    __device__ __forceinline__ void each(uint32_t d, F&& f) const {
#pragma unroll
        for (int odd = 0; odd < 2; ++odd) {
            const uint32_t n = odd ? d >> 4 : d, at = n & 0x07070707u;
            const uint32_t top = __builtin_amdgcn_perm(0u, 0u, (n & 0x08080808u) | 0x05050505u);   // 0xFF in bytes whose code is 8 or more (selector 13), else 0
            const uint32_t l = (__builtin_amdgcn_perm(lo[1], lo[0], at) & ~top) | (__builtin_amdgcn_perm(lo[3], lo[2], at) & top);
            const uint32_t h = (__builtin_amdgcn_perm(hi[1], hi[0], at) & ~top) | (__builtin_amdgcn_perm(hi[3], hi[2], at) & top);
            const auto p0 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(h, l, 0x05010400u));
            const auto p1 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(h, l, 0x07030602u));
            f(odd, (float)p0[0]); f(odd + 2, (float)p0[1]); f(odd + 4, (float)p1[0]); f(odd + 6, (float)p1[1]);
        }
    }
    __device__ __forceinline__ float one(uint32_t code) const {
        const uint32_t g = code >> 2, sh = 8u * (code & 3u);
        const uint32_t l = g == 0u ? lo[0] : g == 1u ? lo[1] : g == 2u ? lo[2] : lo[3], h = g == 0u ? hi[0] : g == 1u ? hi[1] : g == 2u ? hi[2] : hi[3];
        return flat_half((uint16_t)(((l >> sh) & 255u) | (((h >> sh) & 255u) << 8)));
    }
};

template <>
struct FlatBook<2> {
    __device__ __forceinline__ void init(const void*, const float*) {}
    // sixteen codes of d; codes i and i + 8 become one FP16 pair (only the high bytes differ: 0xBC, 0x00, 0x3C, 0x3C)
    template <class F>
    __device__ __forceinline__ void each(uint32_t d, F&& f) const {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t at = ((i < 4 ? d << (8 - 2 * i) : d >> (2 * i - 8)) & 0x03000300u) | 0x000C000Cu;
            const auto p = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0u, 0x3C3C00BCu, at));
            f(i, (float)p[0]); f(i + 8, (float)p[1]);
        }
    }
    __device__ __forceinline__ float one(uint32_t code) const { return code == 0u ? -1.0f : code == 1u ? 0.0f : 1.0f; }
};

template <>
struct FlatBook<8> {
    const float* tab;                                      // LDS: entry v of copy c at v * 16 + c
    uint32_t copy;
    __device__ __forceinline__ void init(const void*, const float* lds) { tab = lds; copy = threadIdx.x & 15u; }
    template <class F>
    __device__ __forceinline__ void each(uint32_t d, F&& f) const {
#pragma unroll
        for (int i = 0; i < 4; ++i) f(i, tab[((d >> (8 * i)) & 255u) * 16u + copy]);
    }
    __device__ __forceinline__ float one(uint32_t code) const { return tab[code * 16u + copy]; }
};

// R rows (PAIR: the rows of R values of m for one n) against B activation rows (PAIR: one).
template <int BITS, int R, int B, bool PAIR>
__global__ void __launch_bounds__(256)
flat_rows_kernel(const FlatRows a) {
    constexpr uint32_t PER = 32 / BITS, WORDS = BITS == 2 ? 1 : 8 / PER, UNIT = PER * WORDS;   // weights of a lane per step: 16 or 8
    __shared__ float tab[BITS == 8 ? 256 * 16 : 1];
    __shared__ float part[4][R * B];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (BITS == 8) {
        for (uint32_t i = tid; i < 256u * 16u; i += 256u) tab[i] = reinterpret_cast<const float*>(a.cb)[i >> 4];
        __syncthreads();
    }
    FlatBook<BITS> book;
    book.init(a.cb, tab);
    const uint32_t groups = PAIR ? a.rows : (a.rows + R - 1) / R, bg = blockIdx.x / groups, rg = blockIdx.x - bg * groups;
    const uint32_t r0 = PAIR ? rg : rg * R, b0 = bg * (PAIR ? R : B);
    const uint8_t* w[R];
    const float* x[B];
#pragma unroll
    for (int r = 0; r < R; ++r) {                          // rows past the end repeat the last one
        if (PAIR) {
            const uint64_t pair = (uint64_t)min(b0 + r, a.batch - 1u) * a.rows + r0;
            w[r] = a.w + pair * a.K / 2;
        } else {
            w[r] = a.w + (uint64_t)min(r0 + r, a.rows - 1u) * a.row_bytes;
        }
    }
#pragma unroll
    for (int b = 0; b < B; ++b) x[b] = a.x + (uint64_t)(PAIR ? r0 : min(b0 + b, a.batch - 1u)) * a.K;
    float acc[R][B] = {};
    if (a.K >= UNIT) {
        for (uint32_t k0 = (wave * 64u + lane) * UNIT; k0 < a.K; k0 += 256u * UNIT) {
            // the lane that would run past the row's end takes the row's last UNIT weights and leaves out what its
            // neighbour has: a remainder walked weight by weight is a chain of loads (K = 4092: 12.3 us with it, 7.1 without)
            const uint32_t k = k0 + UNIT <= a.K ? k0 : a.K - UNIT, skip = k0 - k;
            uint32_t d[R][WORDS];
            if (a.last) {
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (uint32_t q = 0; q < WORDS; ++q) d[r][q] = load_bits32(w[r], (k + q * PER) * BITS, a.last);
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (uint32_t q = 0; q < WORDS; ++q) d[r][q] = reinterpret_cast<const uint32_t*>(w[r] + k * BITS / 8)[q];
            }
            float xv[B][UNIT];
#pragma unroll
            for (int b = 0; b < B; ++b)
#pragma unroll
                for (uint32_t q = 0; q < UNIT / 4; ++q) {
                    const float4 v = load_f4(x[b] + k + 4 * q);
                    xv[b][4 * q] = v.x; xv[b][4 * q + 1] = v.y; xv[b][4 * q + 2] = v.z; xv[b][4 * q + 3] = v.w;
                }
            auto products = [&](auto masked) {
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (uint32_t q = 0; q < WORDS; ++q)
                        book.each(d[r][q], [&](int i, float v) {
                            if (masked.value) v = q * PER + i >= skip ? v : 0.0f;       // both factors: the other may be infinite
#pragma unroll
                            for (int b = 0; b < B; ++b) acc[r][b] = __builtin_fmaf(v, xv[b][q * PER + i], acc[r][b]);
                        });
            };
            if (__ballot(skip != 0u) == 0ull) {
                products(std::false_type{});
            } else {
#pragma unroll
                for (int b = 0; b < B; ++b)
#pragma unroll
                    for (uint32_t i = 0; i < UNIT; ++i) xv[b][i] = i >= skip ? xv[b][i] : 0.0f;
                products(std::true_type{});
            }
        }
    } else if (tid < a.K) {                                // rows shorter than a lane's share
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float v = book.one((w[r][tid * BITS / 8] >> (tid * BITS % 8)) & ((1u << BITS) - 1u));
#pragma unroll
            for (int b = 0; b < B; ++b) acc[r][b] = v * x[b][tid];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const float v = wave_sum(acc[r][b]);
            if (lane == 63u) part[wave][r * B + b] = v;
        }
    __syncthreads();
    if (tid < R * B) {
        const uint32_t r = tid / B, b = tid % B;
        const float v = ((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid])) * a.scale;
        if (PAIR) { if (b0 + r < a.batch) a.y[(uint64_t)(b0 + r) * a.rows + r0] = v; }
        else if (r0 + r < a.rows && b0 + b < a.batch) a.y[(uint64_t)(b0 + b) * a.rows + r0 + r] = v;
    }
}

template <int BITS, int R, int B, bool PAIR>
int launch_flat_rows(FlatRows a, hipStream_t s) {
    const uint64_t bytes = PAIR ? ((uint64_t)a.batch * a.rows * a.K + 1) / 2 : a.rows * a.row_bytes;
    if (bytes && ((reinterpret_cast<uintptr_t>(a.w) & 3u) || (a.K & (32u / BITS - 1u)) || (!PAIR && (a.row_bytes & 3u))))
        a.last = reinterpret_cast<const uint8_t*>((reinterpret_cast<uintptr_t>(a.w) + bytes - 1) & ~(uintptr_t)3);
    const uint64_t gx = PAIR ? a.rows : (a.rows + R - 1) / R, gy = (a.batch + (PAIR ? R : B) - 1) / (PAIR ? R : B);
    if (gx * gy > 0x7FFFFFFFull) return fail(OILHIP_E_ARG, "outputs exceed the grid limit");
    hipLaunchKernelGGL((flat_rows_kernel<BITS, R, B, PAIR>), dim3((uint32_t)(gx * gy)), dim3(256), 0, s, a);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

// Rows per workgroup: four share the activations' loads; few rows go one per workgroup so that every CU has some.
template <int BITS>
int launch_flat_rows(const FlatRows& a, hipStream_t s) {
    if (a.rows < 2048u) return a.batch == 1 ? launch_flat_rows<BITS, 1, 1, false>(a, s) : a.batch == 2 ? launch_flat_rows<BITS, 1, 2, false>(a, s) : launch_flat_rows<BITS, 1, 4, false>(a, s);
    return a.batch == 1 ? launch_flat_rows<BITS, 4, 1, false>(a, s) : a.batch == 2 ? launch_flat_rows<BITS, 4, 2, false>(a, s) : launch_flat_rows<BITS, 4, 4, false>(a, s);
}

// OIL{8,4,2}Engine::quant_gemm: codes packed along the flat [K][N] index, every output one k-ordered chain of fused
// multiply-adds, terms with A == 0 skipped, bit for bit as in the reference loop.
// The chain bounds it: K dependent FMAs of one wavefront, at least 4 cycles each.  Instructions on the wavefront that carries it cost the
// most, so a workgroup splits the work by role: producer wavefronts fetch, unpack and look up the levels of COLS columns and a tile of
// steps into LDS while one wavefront per row of A walks an earlier tile with 1.25 instructions per step (an FMA, a quarter of a 16-byte LDS
// read; A sits in a register of 16 lanes and the broadcast is part of the FMA).  16 columns per workgroup, three quarters of the chain's
// lanes idle: the chain costs the same for any number of lanes, and 256 workgroups at N = 4096 share the unpacking and
// the fetches.  A producer lane takes one k step: its columns' codes are neighbouring dwords at any bit
// offset, its levels go to as many rows of the tile (lanes side by side, no bank conflicts), and four tiles of codes are in
// flight.  For that the loops over whole tiles have no branch between a fetch and its use, or the compiler waits for all loads, and
// the loads say that they are global (load_dword): with either missing, every tile waited out a trip to memory, 13 cycles per step.
// Three buffers let the chain pass the next tile's barrier and start its reads before it ends a tile.  ONE (one row of A, COLS < 64): the
// chain has a SIMD to itself; with 64 columns the producers need all four (N = 11008, 4-bit: 28.5 us on three, 26.5).
// K = 4096, M = 1, 4-bit, N = 300 / 4096 / 8192 / 11008: 20.5 / 22.6 / 27.0 / 36.5 -> 17.0 / 18.7 / 21.6 / 26.5 us; 8-bit 21.5 / 23.8 / 35.6 / 49.5 ->
// 18.2 / 19.8 / 24.6 / 31; M = 8, N = 4096, 4-bit 48 -> 41.  Now 8 cycles per step: 4.6 for the FMA with its broadcast, 1.2 for the LDS
// reads' issue (both measured alone), the rest around a tile's barrier, its test for zeros and its loads of A.
constexpr int kEngMaxRows = 4, kEngTile = 192, kEngPitch = kEngTile + 4, kEngBuffers = 3;
constexpr int eng_parts(int cols) { return cols > 16 ? 2 : 1; }             // producers that share a tile's step
constexpr int eng_producers(int cols) { return kEngTile / 64 * eng_parts(cols); }
constexpr int eng_copies(int bits, int cols) { return bits != 8 ? 64 : cols == 64 ? 8 : 16; }   // lane-private copies of the codebook
constexpr size_t eng_lds(int bits, int cols) { return 4u * ((size_t)eng_copies(bits, cols) << bits) + 4u * (size_t)(kEngBuffers * cols * kEngPitch); }

// Sixteen steps of a chain: acc += a * level, step 4 i + e with A from a[e] of lane J + i of every 16.  The broadcast rides on the FMA
// (the compiler keeps it as a move of its own, which doubles the chain's instructions).  A register that a VALU instruction has just
// written must not be read this way: a[] is written by memory loads only.
template <int J>
__device__ __forceinline__ void eng_steps(float& acc, const float4& a, const float4* q) {
#define ENG_FOUR(I, L0, L1, L2, L3)                                                                                                          \
    "v_fmac_f32_dpp %0, %1, %" #L0 " row_newbcast:%" #I " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %0, %2, %" #L1 " row_newbcast:%" #I   \
    " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %0, %3, %" #L2 " row_newbcast:%" #I " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %0, %4, %" #L3 \
    " row_newbcast:%" #I " row_mask:0xf bank_mask:0xf\n\t"
    asm(ENG_FOUR(21, 5, 6, 7, 8) ENG_FOUR(22, 9, 10, 11, 12) ENG_FOUR(23, 13, 14, 15, 16) ENG_FOUR(24, 17, 18, 19, 20)
        : "+v"(acc) : "v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(q[0].x), "v"(q[0].y), "v"(q[0].z), "v"(q[0].w), "v"(q[1].x), "v"(q[1].y),
          "v"(q[1].z), "v"(q[1].w), "v"(q[2].x), "v"(q[2].y), "v"(q[2].z), "v"(q[2].w), "v"(q[3].x), "v"(q[3].y), "v"(q[3].z), "v"(q[3].w),
          "n"(J), "n"(J + 1), "n"(J + 2), "n"(J + 3));
#undef ENG_FOUR
}

template <int BITS, int COLS, bool ONE>
__global__ void __launch_bounds__(ONE ? 256 * eng_parts(COLS) : 64 * (eng_producers(COLS) + kEngMaxRows))
engine_kernel(const float* __restrict__ A, const uint8_t* __restrict__ bq, const float* __restrict__ cb, float* __restrict__ C,
              long long M, long long N, long long K) {
    constexpr int TILE = kEngTile, PITCH = kEngPitch, PRODUCERS = eng_producers(COLS);
    constexpr int OWN = COLS / eng_parts(COLS);       // a producer's lanes take a step each, OWN columns of it
    constexpr int W = OWN * BITS / 32;                     // dwords of one step's codes
    constexpr uint32_t COPIES = eng_copies(BITS, COLS), SHIFT = COPIES == 64 ? 8 : COPIES == 16 ? 6 : 5;   // an entry's copies take 1 << SHIFT bytes
    constexpr int AHEAD = 4;                               // tiles of codes in flight
    extern __shared__ __align__(16) float eng_mem[];
    float* tab = eng_mem;
    float* lev0 = eng_mem + (COPIES << BITS);              // three tiles: [column][step]
    const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    for (uint32_t i = threadIdx.x; i < (1u << BITS) * COPIES; i += blockDim.x) tab[i] = cb[i / COPIES];
    // workgroups are dealt to the eight XCDs in turn: each takes a run of neighbouring columns, whose codes share lines
    const uint32_t q8 = gridDim.x >> 3, r8 = gridDim.x & 7u, xcd = blockIdx.x & 7u;
    const long long n0 = (long long)(xcd * q8 + (xcd < r8 ? xcd : r8) + (blockIdx.x >> 3)) * COLS;
    const long long full = K / TILE, tiles = (K + TILE - 1) / TILE;
    __syncthreads();
    // ONE: wavefront 0 is the chain, and wavefront 4, which would share its SIMD, ends here
    if (ONE && wave == 4u) return;
    if (ONE ? wave != 0u : wave < (uint32_t)PRODUCERS) {
        const uint32_t step0 = (ONE ? (wave & 3u) - 1u : wave % 3u) * 64u + lane, col0 = (ONE ? wave >> 2 : wave / 3u) * OWN;
        uint32_t raw[AHEAD][W + 1], sh[AHEAD];
        const uintptr_t base = reinterpret_cast<uintptr_t>(bq);
        const uintptr_t last = (base + ((unsigned long long)K * (unsigned long long)N * BITS + 7) / 8 - 1) & ~(uintptr_t)3;
        // This lane's step of the next tile, as wide loads where no lane's dwords can reach past the codes' end (the first `safe`
        // tiles), else dword by dword; past the end: the last step again.
        const unsigned long long first = (unsigned long long)n0 + col0, end_bit = ((unsigned long long)(K - 1) * N + first) * BITS;
        unsigned long long next_bit = ((unsigned long long)step0 * N + first) * BITS;
        const long long safe = (K - (COLS * BITS + 95) / (N * BITS) - 1) / TILE;
        auto fetch = [&](int slot, auto wide) {
            const unsigned long long bit = next_bit < end_bit ? next_bit : end_bit;
            next_bit += (unsigned long long)TILE * N * BITS;
            const uintptr_t at = base + (bit >> 3), word = at & ~(uintptr_t)3;
            sh[slot] = (uint32_t)(at & 3) * 8u + (uint32_t)(bit & 7);
            if (wide.value) {
                load_dwords<W + 1>(raw[slot], word);
                return;
            }
#pragma unroll
            for (int i = 0; i <= W; ++i) raw[slot][i] = load_dword(word + 4 * i < last ? word + 4 * i : last);
        };
        uint32_t buffer = 0;
        auto decode = [&](int slot, auto partial, bool live) {   // a tile that K ends in: zeros past K
            float lv[OWN];
#pragma unroll
            for (int c = 0; c < OWN; ++c) {
                const uint32_t d = __builtin_amdgcn_alignbit(raw[slot][c * BITS / 32 + 1], raw[slot][c * BITS / 32], sh[slot]);
                constexpr uint32_t MASK = ((1u << BITS) - 1u) << SHIFT;
                const int right = c * BITS % 32 - (int)SHIFT;
                const uint32_t at = ((right > 0 ? d >> right : d << -right) & MASK) | ((lane & (COPIES - 1)) * 4u);   // byte offset of the entry's copy
                lv[c] = *reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(tab) + at);
            }
            float* dst = lev0 + buffer * (COLS * PITCH) + col0 * PITCH + step0;
#pragma unroll
            for (int c = 0; c < OWN; ++c) dst[c * PITCH] = partial.value && !live ? 0.0f : lv[c];
            buffer = buffer == kEngBuffers - 1 ? 0u : buffer + 1u;
        };
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) fetch(u, std::false_type{});
        long long t = 0;
        for (; t + 2 * AHEAD <= safe; t += AHEAD)          // no branch inside, so that a wait counts exactly the loads before it
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                decode(u, std::false_type{}, true);        // tile t + u: the chain has left tile t + u - 3
                fetch(u, std::true_type{});
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);         // the next tile's waits stay behind this tile
            }
        for (; t < tiles; t += AHEAD)
#pragma unroll
            for (int u = 0; u < AHEAD; ++u)
                if (t + u < tiles) {                       // uniform over the workgroup, as in the other role
                    decode(u, std::true_type{}, (t + u) * TILE + step0 < K);
                    fetch(u, std::false_type{});
                    __syncthreads();
                }
        return;
    }
    __builtin_amdgcn_s_setprio(3);                         // the chain goes first where it shares a SIMD with producers
    const uint32_t row = ONE ? 0u : wave - PRODUCERS, rows = ONE ? 1u : (blockDim.x >> 6) - PRODUCERS;
    const long long m = (long long)blockIdx.y * rows + row;
    const bool live = m < M;
    const float* a_row = A + (live ? m : M - 1) * K;
    const float* mine = lev0 + (lane & (COLS - 1)) * PITCH;
    constexpr int GA = TILE / 64;                          // A of a tile: lane j of every 16 holds steps 64 g + 4 j to 64 g + 4 j + 3
    auto fetch_a = [&](float4 (&dst)[GA], long long t) {
        const float* p = a_row + t * TILE + 4u * (lane & 15u);
#pragma unroll
        for (int g = 0; g < GA; ++g) dst[g] = load_f4(p + 64 * g);
    };
    auto fetch_last = [&](float4 (&dst)[GA]) {             // the tile that K ends in
#pragma unroll
        for (int g = 0; g < GA; ++g) {
            const long long k = full * TILE + 64 * g + 4u * (lane & 15u);
            // past K: -0 meets a zero level, and adding their product, -0, changes no sum, not even a zero's sign
            dst[g].x = k < K ? a_row[k] : -0.0f; dst[g].y = k + 1 < K ? a_row[k + 1] : -0.0f;
            dst[g].z = k + 2 < K ? a_row[k + 2] : -0.0f; dst[g].w = k + 3 < K ? a_row[k + 3] : -0.0f;
        }
    };
    float acc = 0.0f;
    constexpr int BATCHES = TILE / 32, RING = ONE ? 3 : 2; // batches of 32 steps; the levels of one, and of those that are read ahead
    static_assert(BATCHES % RING == 0);
    float4 lv[RING][8];
    const float* src = mine;
    auto read = [&](float4 (&dst)[8], const float* tile, int b) {
#pragma unroll
        for (int j = 0; j < 8; ++j) dst[j] = *reinterpret_cast<const float4*>(tile + 32 * b + 4 * j);
    };
    auto after = [&](const float* tile) { return tile == mine + (kEngBuffers - 1) * (COLS * PITCH) ? mine : tile + COLS * PITCH; };
    // A tile's steps.  The next tile's barrier and first reads come before this one's end.
    // for LDS alone, whose writers wait for their writes: reads stay in flight across it
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto walk = [&](const float4 (&a)[GA], auto partial, int steps, bool more) {
        float low = INFINITY;                              // smallest magnitude of the tile's A: is there a zero?
        if (!partial.value) {
#pragma unroll
            for (int g = 0; g < GA; ++g) {
                asm("v_min3_f32 %0, %0, |%1|, |%2|" : "+v"(low) : "v"(a[g].x), "v"(a[g].y));
                asm("v_min3_f32 %0, %0, |%1|, |%2|" : "+v"(low) : "v"(a[g].z), "v"(a[g].w));
            }
        } else {
#pragma unroll
            for (int g = 0; g < GA; ++g) {
                const int k = 64 * g + 4 * (int)(lane & 15u);
                if (k < steps) low = fminf(low, fabsf(a[g].x));
                if (k + 1 < steps) low = fminf(low, fabsf(a[g].y));
                if (k + 2 < steps) low = fminf(low, fabsf(a[g].z));
                if (k + 3 < steps) low = fminf(low, fabsf(a[g].w));
            }
        }
        const float* next = after(src);
        if (__builtin_expect(__ballot(low == 0.0f) == 0ull, 1)) {
            auto batch = [&](auto number) {
                constexpr int b = decltype(number)::value, FAR = RING - 1;
                if constexpr (b + FAR < BATCHES) {
                    read(lv[(b + FAR) % RING], src, b + FAR);
                } else if (more) {
                    if (b + FAR == BATCHES) barrier();
                    read(lv[(b + FAR) % RING], next, b + FAR - BATCHES);
                }
                __builtin_amdgcn_sched_barrier(0);
                const float4* l = lv[b % RING];
                eng_steps<8 * (b & 1)>(acc, a[b / 2], l);  // one statement per 16 steps: the compiler puts a wait state between two
                eng_steps<8 * (b & 1) + 4>(acc, a[b / 2], l + 4);
                __builtin_amdgcn_sched_barrier(0);
            };
            [&]<int... B>(std::integer_sequence<int, B...>) { (batch(std::integral_constant<int, B>{}), ...); }(std::make_integer_sequence<int, BATCHES>{});
        } else {                                           // a zero: the reference skips the term, 0 * inf must not reach the sum
#pragma unroll
            for (int g = 0; g < GA; ++g)
_Pragma("unroll 1")
                for (int j = 0; j < 16; ++j) {
                    const float v[4] = {a[g].x, a[g].y, a[g].z, a[g].w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {          // steps past K: -0, whose terms change nothing
                        const float x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[e]), j));
                        const float r = __fmaf_rn(x, src[64 * g + 4 * j + e], acc);
                        acc = x != 0.0f ? r : acc;
                    }
                }
            if (more) {
                barrier();
#pragma unroll
                for (int b = 0; b < RING - 1; ++b) read(lv[b], next, b);
            }
        }
        src = next;
    };
    float4 a0[GA], a1[GA];
    auto fetch_any = [&](float4 (&dst)[GA], long long t) { if (t < full) fetch_a(dst, t); else if (t < tiles) fetch_last(dst); };
    auto walk_any = [&](const float4 (&a)[GA], long long t) { walk(a, std::true_type{}, t < full ? TILE : (int)(K - full * TILE), t + 1 < tiles); };
    fetch_any(a0, 0);
    __syncthreads();
#pragma unroll
    for (int b = 0; b < RING - 1; ++b) read(lv[b], src, b);
    long long t = 0;
    for (; t + 2 < full; t += 2) {                         // no branch but walk's own: A of the next tile stays in flight
        fetch_a(a1, t + 1);
        walk(a0, std::false_type{}, TILE, true);
        fetch_a(a0, t + 2);
        walk(a1, std::false_type{}, TILE, true);
    }
    for (; t < tiles; t += 2) {                            // at most three tiles
        fetch_any(a1, t + 1);
        walk_any(a0, t);
        if (t + 1 == tiles) break;
        fetch_any(a0, t + 2);
        walk_any(a1, t + 1);
    }
    if (live && lane < (uint32_t)COLS && n0 + lane < N) C[m * N + n0 + lane] = acc;
}

__global__ void __launch_bounds__(256) engine_empty_kernel(float* __restrict__ C, long long n) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) C[i] = 0.0f;
}

// The engines whose B operand is not a codebook index: kind 1 = Oil1Engine (one float per 32 flat positions,
// src/oil_engines_oil1.cpp:61-82), 3 = SparkEngine (2-bit codes: 2 -> +s, 0 -> -s, else 0, with s = a * scale of
// the flat position's block, src/oil_engines_spark.cpp:154-186), 16 = OIL16Engine (FP16 widened as
// math::vec_fp16_to_fp32 does, src/math.cpp:509-526; src/oil_engines_fp.cpp:433-451), 32 = OIL32Engine (:531-547).
// Terms with a == 0 are skipped and k runs in ascending order, as in the reference loops.
template <int KIND>
__global__ void __launch_bounds__(64)
engine_dense_kernel(const float* __restrict__ A, const void* __restrict__ B, const float* __restrict__ scales,
                    long long block, float* __restrict__ C, long long M, long long N, long long K) {
    // Same frame as engine_kernel: a wavefront per 64 outputs, the operand of 32 steps fetched together and one
    // batch ahead, the k-ordered chain of every output untouched.
    const long long n = (long long)blockIdx.x * 64 + threadIdx.x;
    const long long m = blockIdx.y;
    const bool live = n < N;
    const unsigned long long nn = (unsigned long long)(live ? n : N - 1);
    constexpr int UN = KIND == 3 ? 16 : 32;              // kind 3 fetches two operands per step
    const float* a_row = A + m * K;
    struct Term { float b; float s; };                   // kind 3: b = +1 / -1 / 0 by code, s = scale of the flat position's block
    // kind 3: block index and offset of the next flat position to be fetched (fetches go through k in order)
    const unsigned long long ublock = block > 0 ? (unsigned long long)block : 1ull;
    unsigned long long fq = nn / ublock, fr = nn % ublock;
    const unsigned long long dq = (unsigned long long)N / ublock, dr = (unsigned long long)N % ublock;
    auto fetch_one = [&](long long kk) {
        const unsigned long long flat = (unsigned long long)kk * (unsigned long long)N + nn;
        Term t{0.0f, 1.0f};
        if (KIND == 1) t.b = reinterpret_cast<const float*>(B)[flat / 32];
        else if (KIND == 32) t.b = reinterpret_cast<const float*>(B)[flat];
        else if (KIND == 16) t.b = __uint_as_float((uint32_t)reinterpret_cast<const uint16_t*>(B)[flat]);   // raw half, widened later
        else {
            t.s = scales[fq];
            t.b = __uint_as_float((uint32_t)((reinterpret_cast<const uint8_t*>(B)[flat / 4] >> ((flat % 4) * 2)) & 3u));
            fq += dq; fr += dr;
            if (fr >= ublock) { fr -= ublock; ++fq; }
        }
        return t;
    };
    auto widen = [](float raw) {                          // math::vec_fp16_to_fp32: -0 widens to +0; selects only
        const uint32_t h = __float_as_uint(raw);
        const uint32_t sg = (h & 0x8000u) << 16, e = (h >> 10) & 31u, mt = h & 0x3FFu;
        const uint32_t normal = sg | ((e + 112u) << 23) | (mt << 13);
        const uint32_t infnan = sg | 0x7F800000u | (mt << 13);
        const uint32_t sub = sg | __float_as_uint(__uint2float_rn(mt) * 0x1p-24f);      // exact
        const uint32_t r = e == 31u ? infnan : (e != 0u ? normal : sub);
        return (h & 0x7FFFu) == 0u ? 0.0f : __uint_as_float(r);
    };
    auto fold = [&](float acc, float a, const Term& t) {
        if (KIND == 1 || KIND == 32) {
            const float r = __fmaf_rn(a, t.b, acc);
            return a != 0.0f ? r : acc;
        } else if (KIND == 16) {
            const float r = __fmaf_rn(a, t.b, acc);                                  // widened before the chain starts
            return a != 0.0f ? r : acc;
        } else {
            const float s = __fmul_rn(a, t.s);                                       // a product, then a sum: no fused form here
            const uint32_t code = __float_as_uint(t.b);
            const float r = code == 2u ? __fadd_rn(acc, s) : (code == 0u ? __fsub_rn(acc, s) : acc);
            return a != 0.0f ? r : acc;
        }
    };
    float acc = 0.0f;
    long long k = 0;
    Term cur[UN], nxt[UN];
    if (K >= UN) {
#pragma unroll
        for (int j = 0; j < UN; ++j) cur[j] = fetch_one(j);
    }
    for (; k + UN <= K; k += UN) {
        const bool more = k + 2 * UN <= K;
        if (more) {
#pragma unroll
            for (int j = 0; j < UN; ++j) nxt[j] = fetch_one(k + UN + j);
        }
        if (KIND == 16) {
#pragma unroll
            for (int j = 0; j < UN; ++j) cur[j].b = widen(cur[j].b);
        }
#pragma unroll
        for (int j = 0; j < UN; ++j) acc = fold(acc, a_row[k + j], cur[j]);
        if (more) {
#pragma unroll
            for (int j = 0; j < UN; ++j) cur[j] = nxt[j];
        }
    }
    for (; k < K; ++k) {
        Term t = fetch_one(k);
        if (KIND == 16) t.b = widen(t.b);
        acc = fold(acc, a_row[k], t);
    }
    if (live) C[m * N + n] = acc;
}

// OIL{8,4,2}Engine::dequant_tensor (src/oil_engines_oil8.cpp:171-183, oil4.cpp:205-220, oil2.cpp:184-193): packed
// codes -> codebook values; with scales, OIL8Engine / OIL4Engine::dequantize_per_block (oil8.cpp:121-134:
// cb[i] * scale; oil4.cpp:136-150: cb[i] * half_range + center, one multiply-add in the reference build) over
// one index byte per weight.
__global__ void __launch_bounds__(256)
engine_dequant_kernel(int bits, const uint8_t* __restrict__ idx, const float* __restrict__ cb, long long n,
                      const float* __restrict__ scales, long long block, float* __restrict__ out) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        if (!scales) {
            const int per = 8 / bits;
            const uint32_t code = (idx[i / per] >> ((i % per) * bits)) & ((1u << bits) - 1u);
            out[i] = cb[code];
        } else if (bits == 8) {
            out[i] = cb[idx[i]] * scales[i / block];
        } else {
            const long long b = i / block;
            out[i] = __fmaf_rn(cb[idx[i] & 15u], scales[2 * b + 1], scales[2 * b]);
        }
    }
}

template <int BITS, int COLS, bool ONE>
int launch_engine(const float* a, const uint8_t* b, const float* cb, float* c, int64_t M, int64_t N, int64_t K, hipStream_t s) {
    static std::atomic<uint64_t> raised{0};
    constexpr size_t lds = eng_lds(BITS, COLS);
    if (int rc = ensure_max_lds(raised, (const void*)engine_kernel<BITS, COLS, ONE>, (int)lds)) return rc;
    const int64_t rows = std::min<int64_t>(M, kEngMaxRows), groups = (N + COLS - 1) / COLS;   // rows of A of one workgroup share the levels
    if (groups > 0x7FFFFFFFll) return fail(OILHIP_E_ARG, "N exceeds the grid limit");
    hipLaunchKernelGGL((engine_kernel<BITS, COLS, ONE>), dim3((uint32_t)groups, (uint32_t)((M + rows - 1) / rows)),
                       dim3((uint32_t)(ONE ? 256 * eng_parts(COLS) : 64 * (eng_producers(COLS) + rows))), lds, s, a, b, cb, c, (long long)M, (long long)N, (long long)K);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

template <int BITS>
int launch_engine_bits(int cols, const float* a, const uint8_t* b, const float* cb, float* c, int64_t M, int64_t N, int64_t K, hipStream_t s) {
    if (M == 1 && cols < 64) return cols == 16 ? launch_engine<BITS, 16, true>(a, b, cb, c, M, N, K, s) : launch_engine<BITS, 32, true>(a, b, cb, c, M, N, K, s);
    return cols == 16 ? launch_engine<BITS, 16, false>(a, b, cb, c, M, N, K, s)
         : cols == 32 ? launch_engine<BITS, 32, false>(a, b, cb, c, M, N, K, s) : launch_engine<BITS, 64, false>(a, b, cb, c, M, N, K, s);
}

// Negative sizes are errors; an empty output (M or N zero) needs no pointers at all.
int check(const void* a, const void* b, const void* c, const void* d, long long M, long long N, long long K) {
    if (M < 0 || N < 0 || K < 0) return fail(OILHIP_E_ARG, "negative dimension");
    if (M == 0 || N == 0) return OILHIP_OK;
    if (!a || !b || !c || !d) return fail(OILHIP_E_ARG, "null argument");
    return OILHIP_OK;
}

}  // namespace
}  // namespace oilhip

using namespace oilhip;

extern "C" {

int oilhip_flat_oil8_gemm(const uint8_t* d_idx, const float* d_cb, const float* d_act, float* d_out,
                          int M, int N, int K, void* stream) {
    if (int rc = check(d_idx, d_cb, d_act, d_out, M, N, K)) return rc;
    if (M == 0 || N == 0) return OILHIP_OK;
    if (M <= 4) {                                     // decode shapes: the register-resident kernel
        const int rc = launch_gemv_flat8(d_idx, d_cb, d_act, d_out, M, N, K, 1.0f, (hipStream_t)stream);
        if (rc <= 0) return rc;
    }
    return launch_flat_rows<8>(FlatRows{d_idx, d_cb, d_act, d_out, 1.0f, (uint32_t)N, (uint32_t)K, (uint32_t)M, (uint64_t)K}, (hipStream_t)stream);
}

int oilhip_flat_oil4_gemm(const uint8_t* d_packed, const uint16_t* d_cb16, const float* d_act, float* d_out,
                          int M, int N, int K, void* stream) {
    if (int rc = check(d_packed, d_cb16, d_act, d_out, M, N, K)) return rc;
    if (M == 0 || N == 0) return OILHIP_OK;
    if ((long long)M * N > 0x7FFFFFFFll) return fail(OILHIP_E_ARG, "M*N exceeds the grid limit");
    const FlatRows a{d_packed, d_cb16, d_act, d_out, 1.0f, (uint32_t)N, (uint32_t)K, (uint32_t)M, 0};
    return M == 1 ? launch_flat_rows<4, 1, 1, true>(a, (hipStream_t)stream) : M == 2 ? launch_flat_rows<4, 2, 1, true>(a, (hipStream_t)stream)
                  : launch_flat_rows<4, 4, 1, true>(a, (hipStream_t)stream);
}

int oilhip_prod_gemv_spark(const uint8_t* d_w, float scale, const float* d_x, float* d_y,
                           int M, int K, int batch, void* stream) {
    if (int rc = check(d_w, d_x, d_y, d_y, M, batch, K)) return rc;
    if (M == 0 || batch == 0) return OILHIP_OK;
    return launch_flat_rows<2>(FlatRows{d_w, nullptr, d_x, d_y, scale, (uint32_t)M, (uint32_t)K, (uint32_t)batch, ((uint64_t)K + 3) / 4}, (hipStream_t)stream);
}

int oilhip_prod_gemv_oil4(const uint8_t* d_w, const uint16_t* d_cb16, float scale, const float* d_x,
                          float* d_y, int M, int K, int batch, void* stream) {
    if (int rc = check(d_w, d_cb16, d_x, d_y, M, batch, K)) return rc;
    if (M == 0 || batch == 0) return OILHIP_OK;
    if (batch == 1) {                                 // decode: the register-resident kernel (11008 x 4096: 7.6 us against 11.4)
        const int rc = launch_gemv_flat4(d_w, d_cb16, scale, d_x, d_y, M, K, (hipStream_t)stream);
        if (rc <= 0) return rc;
    }
    return launch_flat_rows<4>(FlatRows{d_w, d_cb16, d_x, d_y, scale, (uint32_t)M, (uint32_t)K, (uint32_t)batch, ((uint64_t)K + 1) / 2}, (hipStream_t)stream);
}

// Y[b*M + m]: the flat OIL8 kernel with (rows = M weight rows, batch = activation rows).
int oilhip_prod_gemv_oil8(const uint8_t* d_w, const float* d_cb, float scale, const float* d_x, float* d_y,
                          int M, int K, int batch, void* stream) {
    if (int rc = check(d_w, d_cb, d_x, d_y, M, batch, K)) return rc;
    if (M == 0 || batch == 0) return OILHIP_OK;
    if (batch <= 4) {
        const int rc = launch_gemv_flat8(d_w, d_cb, d_x, d_y, batch, M, K, scale, (hipStream_t)stream);
        if (rc <= 0) return rc;
    }
    return launch_flat_rows<8>(FlatRows{d_w, d_cb, d_x, d_y, scale, (uint32_t)M, (uint32_t)K, (uint32_t)batch, (uint64_t)K}, (hipStream_t)stream);
}

// profile_gemv_{spark,oil4,oil8} (src/kernel_production.cpp:433-485): `repeats` launches of the tiled GEMV between two
// events on `stream`; waits for them.  Not capturable.
int oilhip_profile_gemv(int kind, const uint8_t* d_w, const void* d_cb, float scale, const float* d_x, float* d_y,
                        int M, int K, int repeats, oilhip_kernel_perf_t* out, void* stream) {
    if (!out) return fail(OILHIP_E_ARG, "profile_gemv: null result");
    if (kind != 0 && kind != 4 && kind != 8) return fail(OILHIP_E_ARG, "profile_gemv: kind must be 0 (SPARK), 4 (OIL4) or 8 (OIL8)");
    if (repeats < 1) repeats = 1;
    auto run = [&]() {
        return kind == 0 ? oilhip_prod_gemv_spark(d_w, scale, d_x, d_y, M, K, 1, stream)
             : kind == 4 ? oilhip_prod_gemv_oil4(d_w, static_cast<const uint16_t*>(d_cb), scale, d_x, d_y, M, K, 1, stream)
                         : oilhip_prod_gemv_oil8(d_w, static_cast<const float*>(d_cb), scale, d_x, d_y, M, K, 1, stream);
    };
    if (int rc = run()) return rc;                    // first-use set-up stays outside the timed launches
    auto s = static_cast<hipStream_t>(stream);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    OILHIP_HIP(hipEventCreate(&e0));
    if (hipError_t e = hipEventCreate(&e1); e != hipSuccess) {
        (void)hipEventDestroy(e0);
        return fail(OILHIP_E_DEVICE, std::string("hipEventCreate: ") + hipGetErrorString(e));
    }
    int rc = OILHIP_OK;
    float ms = 0.f;
    hipError_t he = hipEventRecord(e0, s);
    for (int r = 0; r < repeats && rc == OILHIP_OK && he == hipSuccess; ++r) rc = run();
    if (he == hipSuccess) he = hipEventRecord(e1, s);
    if (he == hipSuccess) he = hipEventSynchronize(e1);
    if (he == hipSuccess) he = hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != OILHIP_OK) return rc;
    if (he != hipSuccess) return fail(OILHIP_E_DEVICE, std::string("profile_gemv: ") + hipGetErrorString(he));
    int dev = 0, khz = 0;
    OILHIP_HIP(hipGetDevice(&dev));
    OILHIP_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeClockRate, dev));
    const double sec = (double)ms * 1e-3 / repeats;
    const uint64_t m = (uint64_t)(M > 0 ? M : 0), k = (uint64_t)(K > 0 ? K : 0);
    out->cycles = (uint64_t)(sec * (double)khz * 1e3);            // shader clocks at the device's peak frequency
    out->bytes_read = kind == 0 ? m * k * 2 : kind == 4 ? m * k / 2 + m * k * 4 : m * k + m * 1024;   // the reference's formulas
    out->bytes_written = m * 4;
    out->gflops = sec > 0.0 ? 2.0 * (double)m * (double)k / (sec * 1.0e9) : 0.0;
    return OILHIP_OK;
}

int oilhip_engine_quant_gemm(int bits, const float* d_a, const uint8_t* d_b, const float* d_cb, float* d_c,
                             int64_t M, int64_t N, int64_t K, void* stream) {
    if (int rc = check(d_a, d_b, d_cb, d_c, M, N, K)) return rc;
    if (bits != 2 && bits != 4 && bits != 8) return fail(OILHIP_E_ARG, "bits must be 2, 4 or 8");
    if (M == 0 || N == 0) return OILHIP_OK;
    if (M > 65535) return fail(OILHIP_E_ARG, "M exceeds the grid limit");
    if (K == 0) {                                          // empty sums
        hipLaunchKernelGGL(engine_empty_kernel, dim3((uint32_t)std::min<int64_t>((M * N + 255) / 256, 65535)), dim3(256), 0, (hipStream_t)stream, d_c, (long long)(M * N));
        OILHIP_HIP(hipGetLastError());
        return OILHIP_OK;
    }
    // as few columns per workgroup as keeps the launch at one workgroup per CU: two chains on one SIMD take turns
    const int cus = device_cu_count(), cols = N <= 16ll * cus ? 16 : N <= 32ll * cus ? 32 : 64;
    hipStream_t s = (hipStream_t)stream;
    return bits == 8 ? launch_engine_bits<8>(cols, d_a, d_b, d_cb, d_c, M, N, K, s)
         : bits == 4 ? launch_engine_bits<4>(cols, d_a, d_b, d_cb, d_c, M, N, K, s)
                     : launch_engine_bits<2>(cols, d_a, d_b, d_cb, d_c, M, N, K, s);
}

int oilhip_engine_dequant(int bits, const uint8_t* d_idx, const float* d_cb, int64_t n, const float* d_scales,
                          int64_t block, float* d_out, void* stream) {
    if (n < 0) return fail(OILHIP_E_ARG, "negative length");
    if (n == 0) return OILHIP_OK;
    if (!d_idx || !d_cb || !d_out) return fail(OILHIP_E_ARG, "null argument");
    if (bits != 2 && bits != 4 && bits != 8) return fail(OILHIP_E_ARG, "bits must be 2, 4 or 8");
    if (d_scales && (bits == 2 || block <= 0)) return fail(OILHIP_E_ARG, "per-block dequantize exists for 4 and 8 bits with a positive block size");
    const uint32_t grid = (uint32_t)std::min<int64_t>((n + 255) / 256, 65535);
    hipLaunchKernelGGL(engine_dequant_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream, bits, d_idx, d_cb, (long long)n,
                       d_scales, (long long)block, d_out);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

int oilhip_engine_dense_gemm(int kind, const float* d_a, const void* d_b, const float* d_scales, int64_t block,
                             float* d_c, int64_t M, int64_t N, int64_t K, void* stream) {
    if (int rc = check(d_a, d_b, d_c, d_c, M, N, K)) return rc;
    if (kind != 1 && kind != 3 && kind != 16 && kind != 32) return fail(OILHIP_E_ARG, "kind must be 1, 3, 16 or 32");
    if (M == 0 || N == 0) return OILHIP_OK;
    if (kind == 3 && (!d_scales || block <= 0)) return fail(OILHIP_E_ARG, "the SPARK engine needs scales and a block size");
    if (M > 65535) return fail(OILHIP_E_ARG, "M exceeds the grid limit");
    const dim3 grid((uint32_t)((N + 63) / 64), (uint32_t)M);
    hipStream_t s = (hipStream_t)stream;
    if (kind == 1) hipLaunchKernelGGL(engine_dense_kernel<1>, grid, dim3(64), 0, s, d_a, d_b, d_scales, (long long)block, d_c, M, N, K);
    else if (kind == 3) hipLaunchKernelGGL(engine_dense_kernel<3>, grid, dim3(64), 0, s, d_a, d_b, d_scales, (long long)block, d_c, M, N, K);
    else if (kind == 16) hipLaunchKernelGGL(engine_dense_kernel<16>, grid, dim3(64), 0, s, d_a, d_b, d_scales, (long long)block, d_c, M, N, K);
    else hipLaunchKernelGGL(engine_dense_kernel<32>, grid, dim3(64), 0, s, d_a, d_b, d_scales, (long long)block, d_c, M, N, K);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

}  // extern "C"
