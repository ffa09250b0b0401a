// gemm_signs.hip -- prefill GEMM for tensors that are stored as sign tiles (SPARK_Q0 and OIL1 blocks, common.h): Y[M][N] = X[M][K] . W^T
// with bf16 operands on v_mfma_f32_32x32x16_bf16, FP32 accumulation and output (the contraction of Qwen35Engine::gemm with B up to 512,
// src/adapters/tools/qwen35_engine.cpp:47-85,630-753).
//
// A workgroup is four wavefronts side by side: 64 tokens times 32 FN weight rows each.  A wavefront makes the weights' fragments in registers: a lane
// holds two runs of its row per stage of 64 columns, rounds their scales to bf16 once, and makes a pair of weights with a shift and one
// instruction that masks two signs and flips them.  A pair is columns k and k + 16 of the run, so the activations are packed in that
// order.  Nothing of the weights is shared, so they cost neither LDS nor much of the way into the compute unit that bounds the product over decoded
// operands (gemm_dense.hip), and no launch decodes them.  The activations' fragments and the runs' bits (12 bytes per pair of runs, 4 for OIL1) go
// from memory straight to LDS, three and four stages ahead; one barrier per stage.
//
// What bounds it: with one workgroup per compute unit the issue of its instructions (about 130 beside 16 matrix instructions, one wavefront per SIMD); with
// several, what comes into the compute unit: 12 KB per stage of 64 x 128 outputs.  Loads taken out: 28.4 -> 24.0 us below.
// Weights decoded to bf16 by a launch of their own -> here, whole call, us: planner's mix 5000 x 2816, 437 tokens 33.8 -> 26.3; 4096 x 11008, 64 tokens
// 37.2 -> 22.1; 11008 x 4096, 1024 / 2048 tokens 114 / 200 -> 99 / 178; SPARK_Q0 11008 x 4096, 512 tokens 72.8 -> 52.2;
// 900 x 1024, 50 tokens 9.3 -> 10.6 and 2000 x 4096, 200 tokens 19.9 -> 17.6 stay there.
// Tried and slower: weights through LDS, each made once per workgroup of 128 x 128 (40 us for the first of these: LDS and issue), tiles in groups of four
// token blocks (28.1), a stage more of activations in LDS (a workgroup less per compute unit: 512 tokens 55 -> 62), parts of K with 64 x 256 tiles (60).
#include <algorithm>
#include <string>

#include "common.h"
#include "gemm_tiles.h"

namespace oilhip {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_4 __attribute__((aligned(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_2 __attribute__((aligned(2)));

constexpr int FM = 2, GS = 4;              // 32-token blocks of a workgroup, 16-column groups per stage
constexpr uint32_t A_STAGE = (uint32_t)FM * GS * 1024u;
constexpr uint32_t NA = 4u;                // stages of activations, and of bits, in LDS: stage s in place s % 4
constexpr uint32_t bits_stage(int FN) { return 4u * (uint32_t)FN * 1024u; }

struct SignGemmArgs {
    const uint8_t* W;               // sign tiles
    const uint16_t* Xf;             // [32-token block][16-column group][lane][8 bf16]
    float* Y;
    float* partial;                 // [tile][part][sums] when parts > 1
    uint32_t* arrived;              // per tile, zero before the launch
    uint32_t wbytes, M, N, bpr, ntiles, MT, NT, parts;
};

__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ u32x4 resource(const void* p, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    return u32x4{uni((uint32_t)a), uni((uint32_t)(a >> 32) & 0xFFFFu), uni(bytes), 0x00020000u};
}
__device__ __forceinline__ uint32_t bf16_bits(float f) { return (uint32_t)__builtin_bit_cast(unsigned short, (__bf16)f); }

// ---- activations: a thread takes a run of 32 columns of one token; position 2 k of a run is column k, 2 k + 1 column k + 16
struct SignPackArgs {
    const void* x;
    uint16_t* xf;
    uint32_t* arrived;              // counters to clear
    uint32_t M, bpr, x_is_f32, ncount;
};
__global__ void __launch_bounds__(256)
sign_pack_kernel(const SignPackArgs a) {
    const uint32_t t = threadIdx.x & 31u, run = threadIdx.x >> 5, blk = blockIdx.x, rb = blockIdx.y, m = rb * 32u + t;
    if (blockIdx.x + blockIdx.y == 0)
        for (uint32_t i = threadIdx.x; i < a.ncount; i += 256u) a.arrived[i] = 0u;
    const size_t at = ((size_t)min(m, a.M - 1u) * a.bpr + blk) * 256u + run * 32u;
    uint32_t d[16];
    if (a.x_is_f32) {
        const f32x4_4* x = reinterpret_cast<const f32x4_4*>(static_cast<const float*>(a.x) + at);
        f32x4 f[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = x[j];
#pragma unroll
        for (int j = 0; j < 16; ++j) d[j] = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)f[j >> 2][j & 3], (__bf16)f[4 + (j >> 2)][j & 3]});
    } else {
        const u32x4_2* x = reinterpret_cast<const u32x4_2*>(static_cast<const uint16_t*>(a.x) + at);
        u32x4 f[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) f[j] = x[j];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t lo = f[j >> 2][j & 3], hi = f[2 + (j >> 2)][j & 3];
            d[2 * j] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
            d[2 * j + 1] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
        }
    }
    const bool in = m < a.M;
    u32x4* o = reinterpret_cast<u32x4*>(a.xf) + (((size_t)rb * a.bpr + blk) * 16u + 2u * run) * 64u + t;
#pragma unroll
    for (int p = 0; p < 4; ++p) o[32 * p] = in ? u32x4{d[4 * p], d[4 * p + 1], d[4 * p + 2], d[4 * p + 3]} : u32x4{0u, 0u, 0u, 0u};
}

// ---- product
template <int FN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
gemm_signs_kernel(const SignGemmArgs a) {
    constexpr uint32_t B_STAGE = bits_stage(FN), BITS0 = NA * A_STAGE, HEAD0 = BITS0 + 4u * B_STAGE;
    constexpr int LOADS = FM + FN;                         // per stage and thread: activations, bits
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = uni(tid >> 6), half = lane >> 5;
    const uint32_t tiles = a.MT * a.NT, item = xcd_chunk(blockIdx.x, tiles * a.parts), tile = item / a.parts, part = item % a.parts;
    // all rows of a token block one after the other: an XCD keeps few token blocks in its L2, and the weights' bits are a tenth of their bytes
    const uint32_t mt = tile / a.NT, nt = tile % a.NT;
    const uint32_t bpr = a.bpr, G = 16u * bpr, bbeg = bpr * part / a.parts, bend = bpr * (part + 1u) / a.parts, nblk = bend - bbeg, nst = 4u * nblk;

    // places of the blocks of this workgroup's tiles of 16 rows (past the last tile: the last one again, whose rows are not stored)
    uint2* heads = reinterpret_cast<uint2*>(lds + HEAD0);
    for (uint32_t i = tid; i < 8u * FN * nblk; i += 256u) {
        const uint32_t t = nt * (8u * FN) + i % (8u * FN);
        heads[i] = reinterpret_cast<const uint2*>(a.W)[(size_t)(bbeg + i / (8u * FN)) * a.ntiles + (t < a.ntiles ? t : a.ntiles - 1u)];
    }
    __syncthreads();

    // (to the end of the part's columns of the last row block: a stage past them reads zeros)
    const u32x4 xrs = resource(a.Xf + (size_t)mt * FM * G * 512u + (size_t)bbeg * 8192u, ((uint32_t)(FM - 1) * G + 16u * nblk) * 1024u), wrs = resource(a.W, a.wbytes);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    uint32_t voff[FM];
#pragma unroll
    for (int c = 0; c < FM; ++c) voff[c] = ((uint32_t)c * G + wave) * 1024u + lane * 16u;      // group `wave` of the stage, row block c
    auto load_x = [&](uint32_t st, uint32_t slot) {
        const uint32_t dst = uni(lds0 + slot * A_STAGE + wave * 1024u), so = uni((st < nst ? st : nst - 1u) * (GS * 1024u));
#pragma unroll
        for (int c = 0; c < FM; ++c)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(dst + (uint32_t)c * (GS * 1024u)), "v"(voff[c]), "s"(xrs), "s"(so) : "memory");
    };
    // this lane's row of row block j: 32 j + lane % 32 of the wavefront's; where its block of the row starts, how far apart its run pairs are
    const uint32_t row_bit = 1u << (lane & 15u), rows_before = row_bit - 1u;
    struct Block { uint32_t at, step; };
    auto head_of = [&](uint32_t b, int j) { return heads[(b < nblk ? b : nblk - 1u) * (8u * FN) + 2u * (FN * wave + (uint32_t)j) + ((lane >> 4) & 1u)]; };
    auto block_of = [&](uint2 h) {
        return Block{h.x * 16u + 16u * (lane & 15u) + 32u * (uint32_t)__builtin_popcount(h.y & rows_before), (h.y & row_bit) ? 12u : 4u};
    };
    auto load_bits = [&](uint32_t slot, int j, const Block& k) {           // 16 bytes from run pair `slot` of the block on
        const uint32_t dst = uni(lds0 + BITS0 + slot * B_STAGE + (FN * wave + (uint32_t)j) * 1024u);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" :: "s"(dst), "v"(k.at + slot * k.step), "s"(wrs) : "memory");
    };
    auto bits_of = [&](uint32_t slot, int j) { return *reinterpret_cast<const u32x4*>(lds + BITS0 + slot * B_STAGE + (FN * wave + (uint32_t)j) * 1024u + lane * 16u); };
    struct Run { uint32_t bits, pair; };
    auto runs_of = [&](Run (&r)[2], const u32x4& o, uint32_t step) {
        const bool spark = step == 12u;
        auto pair = [](uint32_t h) { const __bf16 b = (__bf16)-(float)__builtin_bit_cast(_Float16, (unsigned short)h); return __builtin_bit_cast(uint32_t, bf16x2{b, b}); };
        r[0].pair = pair(o.x);                             // of clear bits: minus
        r[1].pair = pair((spark ? o.y : o.x) >> 16);
        r[0].bits = (spark ? __builtin_amdgcn_alignbit(o.y, o.x, 16) : 0xFFFFFFFFu) >> (4u * half);
        r[1].bits = (spark ? o.z : 0xFFFFFFFFu) >> (4u * half);
    };
    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    bf16x8 fa[2][FM];
    u32x4 fb[2][FN];
    Run run[2][FN][2];                                     // of even and odd stages
    auto read_a = [&](int set, uint32_t slot, uint32_t g, int i) { fa[set][i] = *reinterpret_cast<const bf16x8*>(lds + slot * A_STAGE + (uint32_t)i * (GS * 1024u) + g * 1024u + lane * 16u); };
    // element e of group g's fragment: pair 8 (g % 2) + 4 half + e of run g / 2
    auto make_b = [&](int set, const Run (&r)[2], int g, int j, int e) { fb[set][j][e] = ((r[g >> 1].bits << (15 - 8 * (g & 1) - e)) & 0x80008000u) ^ r[g >> 1].pair; };

    Block cur[FN], next[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) { cur[j] = block_of(head_of(0u, j)); next[j] = block_of(head_of(1u, j)); }
#pragma unroll
    for (uint32_t q = 0; q < 2u; ++q)
#pragma unroll
        for (int j = 0; j < FN; ++j) load_bits(q, j, cur[j]);
#pragma unroll
    for (uint32_t i = 0; i < NA - 2u; ++i) load_x(i, i);
#pragma unroll
    for (int j = 0; j < FN; ++j) load_bits(2u, j, cur[j]);
    load_x(NA - 2u, NA - 2u);
#pragma unroll
    for (int j = 0; j < FN; ++j) load_bits(3u, j, cur[j]);
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(LOADS) : "memory");     // the activations of stages 0 and 1, the bits of stages 0 and 1
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        runs_of(run[0][j], bits_of(0u, j), cur[j].step);
#pragma unroll
        for (int e = 0; e < 4; ++e) make_b(0, run[0][j], 0, j, e);
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) read_a(0, 0u, 0u, i);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // slot 0 of the bits is read before it is loaded again
    for (uint32_t b = 0; b < nblk; ++b) {
        uint2 head[FN];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t st = 4u * b + (uint32_t)q;
            // in place: the activations of this stage and the next, the bits of the next
            u32x4 raw[FN];
#pragma unroll
            for (int g = 0; g < GS; ++g) {
                const int set = g & 1, gn = (g + 1) % GS;
#pragma unroll
                for (int e = 0; e < FM * FN; ++e) {
                    const int i = e / FN, j = e % FN;
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[set][i], __builtin_bit_cast(bf16x8, fb[set][j]), acc[i][j], 0, 0, 0);
                    // beside it, for the next group: its fragments; for the next stage: its runs; and the loads
                    if (e < FM) read_a(set ^ 1, (uint32_t)(g + 1 < GS ? q : (q + 1) & 3), (uint32_t)gn, e);
                    constexpr int EACH = 4 / FM;                           // elements of a fragment beside one of FM matrix instructions
#pragma unroll
                    for (int v = 0; v < EACH; ++v) make_b(set ^ 1, run[(q + (g + 1 < GS ? 0 : 1)) & 1][j], gn, j, i * EACH + v);
                    if (i == 0 && g == 0) raw[j] = bits_of((uint32_t)(q + 1) & 3u, j);
                    if (i == FM - 1 && g == 2) runs_of(run[(q + 1) & 1][j], raw[j], q < 3 ? cur[j].step : next[j].step);
                    if (i == 0 && g == 1 && q == 2) head[j] = head_of(b + 2u, j);
                    if (e == 0 && g == 1) load_x(st + 3u, (uint32_t)(q + 3) & 3u);
                    if (i == 0 && g == 2) load_bits((uint32_t)q, j, next[j]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (q == 3) {
#pragma unroll
                for (int j = 0; j < FN; ++j) { cur[j] = next[j]; next[j] = block_of(head[j]); }
            }
            // in place from here on: what all but this iteration loaded
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(%1)" :: "n"(LOADS), "n"(FM) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may write LDS after the end
    // 12 wait states between the last matrix instruction and a read of its sums, which the compiler does not count along a branch
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) asm volatile("s_nop 11" : "+v"(acc[i][j]));

    // lane l holds column l % 32; register v holds row 8 * (v / 4) + 4 * (l / 32) + v % 4
    if (a.parts > 1u) {
        // the parts meet in memory; the last workgroup of a tile adds them up in order (stores and loads that are coherent by themselves)
        float* mine = a.partial + ((size_t)tile * a.parts + part) * (4096u * FM * FN) + tid;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) __hip_atomic_store(mine + ((i * FN + j) * 16 + v) * 256, acc[i][j][v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __shared__ uint32_t order;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this thread's part is in place before the barrier, the others' before theirs
        __syncthreads();
        if (tid == 0) order = __hip_atomic_fetch_add(a.arrived + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (order + 1u != a.parts) return;
        const float* all_parts = a.partial + (size_t)tile * a.parts * (4096u * FM * FN) + tid;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
        for (uint32_t p = 0; p < a.parts; ++p)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) {
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        acc[i][j][v] += __hip_atomic_load(all_parts + (size_t)p * (4096u * FM * FN) + ((i * FN + j) * 16 + v) * 256, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    asm volatile("" ::: "memory");         // not all loads at once
                }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const uint32_t col = nt * (128u * FN) + (wave * FN + (uint32_t)j) * 32u + (lane & 31u);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const uint32_t r = mt * (32u * FM) + (uint32_t)i * 32u + 8u * (v >> 2) + 4u * (lane >> 5) + (v & 3u);
                if (r < a.M && col < a.N) a.Y[(size_t)r * a.N + col] = acc[i][j][v];
            }
        }
}

template <int FN>
int launch_tiles(const SignGemmArgs& a, hipStream_t s) {
    static std::atomic<uint64_t> raised{0};
    auto kern = gemm_signs_kernel<FN>;
    if (int rc = ensure_max_lds(raised, reinterpret_cast<const void*>(kern), 160 * 1024 - 64)) return rc;
    const size_t lds = NA * A_STAGE + 4u * bits_stage(FN) + 64u * FN * (size_t)((a.bpr + a.parts - 1u) / a.parts);
    hipLaunchKernelGGL(kern, dim3(a.MT * a.NT * a.parts), dim3(256), lds, s, a);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

// Row blocks of a wavefront and parts along K for M tokens and N weight rows, by an estimate of the microseconds: 5.6 (FN = 1) or 7.6 for the launches, the
// first loads and the last stores; 1.53 per million activations that are packed; 0.278 or 0.45 per stage of a workgroup that has a compute unit to itself,
// more where several share one; and the parts' meeting.  Fitted to 21 pairs of shape and batch (500 to 11008 rows, 1024 to 11008 columns, 40 to 2048
// tokens) with all plans timed: what it chooses is 1.4 % slower than the best on average, 9 % at most.
struct SignPlan { uint32_t fn, parts; double us; };
SignPlan sign_plan(uint32_t M, uint32_t N, uint32_t bpr) {
    const double cus = (double)device_cu_count(), pack = 1.53e-6 * 256.0 * M * bpr;
    SignPlan best{1u, 1u, 1e30};
    for (uint32_t fn = 1; fn <= 2u; ++fn)
        for (uint32_t parts = 1; parts <= (fn == 1u ? 8u : 1u) && parts <= bpr; parts *= 2u) {
            const double wgs = (double)((M + 32u * FM - 1u) / (32u * FM)) * (double)((N + 128u * fn - 1u) / (128u * fn)) * parts, each = wgs / cus;
            const double load = each <= 1.0 ? 1.0 : fn == 1u ? std::max(0.65 * each + 0.8, 0.88 * each) : 0.95 * each + 0.35;
            const double us = (fn == 1u ? 5.6 : 7.6) + pack + 4.0 * (double)((bpr + parts - 1u) / parts) * (fn == 1u ? 0.278 : 0.45) * load + (parts > 1u ? 0.6 + 0.9 * parts + 0.01 * wgs : 0.0);
            if (us < best.us) best = {fn, parts, us};
        }
    return best;
}

}  // namespace

// The kernel takes its loops' lengths from its part of K, and a part without blocks has none: the plan's parts are checked where they become a launch.
int check_sign_parts(uint32_t bpr, uint32_t parts) {
    return parts >= 1u && parts <= bpr ? OILHIP_OK : fail(OILHIP_E_ARG, "prefill plan of " + std::to_string(parts) + " parts for " + std::to_string(bpr) + " blocks");
}

// Returns 1 when the tensor is not stored as sign tiles, or decoding it first may be as fast (small products).  Both times are estimates, this one 11 % short at most and
// the other 14 % long at most, so a fifth less is asked for.
int launch_gemm_signs(const oilhip_weights& w, const void* d_x, bool x_is_f32, float* d_y, int M_, hipStream_t s) {
    if (!w.seg.sign_tiles) return 1;
    const uint32_t N = (uint32_t)w.rows, bpr = (uint32_t)(w.cols >> 8), M = (uint32_t)M_;
    if ((uint64_t)M * w.cols * 2u >= 0x80000000ull) return fail(OILHIP_E_ARG, "activation matrix too large for the prefill kernel");
    const SignPlan pl = sign_plan(M, N, bpr);
    if (64ull * pl.fn * ((bpr + pl.parts - 1u) / pl.parts) > 49152u || (uint64_t)w.cols * 512u >= 0x80000000ull) return 1;
    if (pl.us > 0.8 * dense_estimate_us(M, N, (uint32_t)w.cols)) return 1;
    if (int rc = check_sign_parts(bpr, pl.parts)) return rc;
    const StreamLock lock(s);
    uint16_t* xf = nullptr;
    const uint32_t mpad = (M + 255u) & ~255u;
    if (int rc = stream_scratch(lock, kScratchGemmX, (size_t)mpad * w.cols * 2, reinterpret_cast<void**>(&xf))) return rc;
    const uint32_t tm = 32u * FM, tn = 128u * pl.fn;
    SignGemmArgs a{w.d_payload, xf, d_y, nullptr, nullptr, (uint32_t)w.alloc_bytes, M, N, bpr, w.seg.sign_tiles, (M + tm - 1u) / tm, (N + tn - 1u) / tn, pl.parts};
    if (a.parts > 1u) {
        void* p = nullptr;
        const size_t counters = ((size_t)a.MT * a.NT * 4u + 255u) & ~(size_t)255u;
        if (int rc = stream_scratch(lock, kScratchGemmP, counters + (size_t)a.MT * a.NT * a.parts * tm * tn * 4u, &p)) return rc;
        a.arrived = static_cast<uint32_t*>(p);
        a.partial = reinterpret_cast<float*>(static_cast<uint8_t*>(p) + counters);
    }
    const SignPackArgs pk{d_x, xf, a.arrived, M, bpr, x_is_f32 ? 1u : 0u, a.parts > 1u ? a.MT * a.NT : 0u};
    hipLaunchKernelGGL(sign_pack_kernel, dim3(bpr, a.MT * tm / 32u), dim3(256), 0, s, pk);
    OILHIP_HIP(hipGetLastError());
    return pl.fn == 2u ? launch_tiles<2>(a, s) : launch_tiles<1>(a, s);
}

}  // namespace oilhip
