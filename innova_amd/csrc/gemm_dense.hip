// gemm_dense.hip -- prefill GEMM for tensors of any format but plain OIL4: Y[M][N] = X[M][K] . W^T over two bf16 operands that a
// pre-pass (dense_prepare_kernel, generic_kernels.hip) has written in fragment order, v_mfma_f32_32x32x16_bf16, FP32 accumulation
// and output (the contraction of Qwen35Engine::gemm with B up to 512, src/adapters/tools/qwen35_engine.cpp:47-85,630-753).
//
// Fragment order: [32-row block][16-column group][lane][8 bf16]; one fragment is 1 KB, lane = 32 * (column half) + row % 32.
// A workgroup is 2 x 2 wavefronts of FM x FN blocks of 32 x 32 outputs.  Its operands go from memory to LDS without passing
// through registers (buffer_load ... lds: 64 lanes x 16 bytes land in order, which is a fragment), GS column groups per stage,
// ST stages around; a wavefront reads fragments back with conflict-free 16-byte reads.  One workgroup barrier per stage; the
// first fragments of a stage are read during the last matrix instructions of the stage before.  The waits on memory are counted
// by hand (the loads are invisible to the compiler).
//
// What bounds it: the operands' way into the compute unit.  A lone workgroup and a full chip both move about 30 bytes per clock
// and compute unit, through LDS or straight into registers, whatever is in flight; the matrix cores would take 64 for tiles of
// 128 x 128.  Tried and slower (11008 x 4096, 1024 tokens; this: 95 us): loads through registers into LDS 105 us, no LDS and K cut
// among the wavefronts 105 us, tiles of 256 x 256 105 to 110 us, 256 x 128 105 us (whole call at 2048 / 4096 tokens: 128 x 128 203 / 363 us,
// 256 x 128 with three stages 202 / 376, 256 x 256 236 / 365).
// Before (pipelined tiles of 256 x 128 and 128 x 128, operands in row order, activations rounded and weights decoded by launches of
// their own) -> now, whole call: 5000 x 2816 planner mix, 437 tokens 55.2 -> 36.7 us; 719 x 3840, four formats, 81 tokens 47.9 ->
// 20.3 us; 4096 x 11008 planner mix, 64 tokens 252 -> 42.5 us; 7532 x 4864 OIL8, 602 tokens 151 -> 113 us; 11008 x 4096 OIL8, 1024
// tokens 154 -> 145 us; 11008 x 4096 SPARK_Q0, 512 / 1024 / 2048 / 4096 tokens 111 / 144 / 237 / 441 -> 79 / 120 / 204 / 363 us.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "gemm_tiles.h"

namespace oilhip {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct DenseArgs {
    const uint16_t *Xf, *Wf;        // fragments
    float* Y;
    float* partial;                 // [tile][part][TM * TN] when parts > 1
    uint32_t* arrived;              // per tile, zero before the launch
    uint32_t M, N, K, ldy, MT, NT, parts;
};

__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ u32x4 resource(const void* p) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    return u32x4{uni((uint32_t)a), uni((uint32_t)(a >> 32) & 0xFFFFu), 0xFFFFFFFFu, 0x00020000u};
}

// GS: column groups per stage (an even divisor of 16), ST: stages around (at least 3)
template <int FM, int FN, int GS, int ST>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
gemm_dense_kernel(const DenseArgs a) {
    constexpr int CH = (FM + FN) * GS / 2;                 // 1 KB pieces a wavefront brings per stage
    constexpr uint32_t STAGE = 4u * CH * 1024u;            // A: 2 FM row blocks x GS groups, then B
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = uni(tid >> 6), wm = wave >> 1, wn = wave & 1u;
    const uint32_t tiles = a.MT * a.NT, item = xcd_chunk(blockIdx.x, tiles * a.parts), tile = item / a.parts, part = item % a.parts;
    uint32_t mt, nt;
    frag_tile_of(tile, a.MT, a.NT, mt, nt);
    const uint32_t G = a.K >> 4, all = G / GS;             // stages of a row: K is a multiple of 256
    const uint32_t sbeg = (uint32_t)((uint64_t)all * part / a.parts), send = (uint32_t)((uint64_t)all * (part + 1u) / a.parts), last = send - 1u;

    const u32x4 xrs = resource(a.Xf + (size_t)mt * (2u * FM) * G * 512u), wrs = resource(a.Wf + (size_t)nt * (2u * FN) * G * 512u);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    uint32_t voff[CH];
    bool is_x[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const uint32_t piece = wave * CH + (uint32_t)c;    // < 2 FM GS: A piece (row block piece / GS, group piece % GS)
        is_x[c] = piece < 2u * FM * GS;
        const uint32_t q = is_x[c] ? piece : piece - 2u * FM * GS;
        voff[c] = (q / GS * G + q % GS) * 1024u + lane * 16u;
    }
    auto load_stage = [&](uint32_t st) {
        const uint32_t so = uni((st < last ? st : last) * (GS * 1024u));                  // past the end: the last one again, never read
        const uint32_t dst = uni(lds0 + (st % (uint32_t)ST) * STAGE + wave * (CH * 1024u));
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const u32x4 rs = is_x[c] ? xrs : wrs;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         :: "s"(dst + (uint32_t)c * 1024u), "v"(voff[c]), "s"(rs), "s"(so) : "memory");
        }
    };
    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    bf16x8 fa[2][FM], fb[2][FN];
    auto read_frags = [&](int set, uint32_t st, uint32_t g) {
        const uint8_t* p = lds + (st % (uint32_t)ST) * STAGE + g * 1024u + lane * 16u;
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[set][i] = *reinterpret_cast<const bf16x8*>(p + (wm * FM + (uint32_t)i) * (GS * 1024u));
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[set][j] = *reinterpret_cast<const bf16x8*>(p + 2u * FM * GS * 1024u + (wn * FN + (uint32_t)j) * (GS * 1024u));
    };
    auto multiply = [&](int set) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[set][i], fb[set][j], acc[i][j], 0, 0, 0);
    };
    for (uint32_t s = 0; s < (uint32_t)ST - 1u; ++s) load_stage(sbeg + s);
    // all but the youngest ST - 2 (here), ST - 3 (in the loop) stages have arrived
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"((ST - 2) * CH) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_frags(0, sbeg, 0);
    for (uint32_t st = sbeg; st < send; ++st) {
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"((ST - 3) * CH) : "memory");
        __builtin_amdgcn_s_barrier();                      // stage st + 1 is in place, stage st - 1 is read
        asm volatile("" ::: "memory");
#pragma unroll
        for (int g = 0; g < GS; ++g) {                     // reads stay a group of matrix instructions ahead
            if (g + 1 < GS) read_frags((g + 1) & 1, st, (uint32_t)g + 1u);
            else read_frags(0, st + 1u, 0);                // after the last stage: what lies there, unused
            __builtin_amdgcn_sched_barrier(0);
            if (g == 0) load_stage(st + (uint32_t)ST - 1u);
            multiply(g & 1);
            __builtin_amdgcn_sched_barrier(0);
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
        // the parts meet in memory; the last workgroup of a tile adds them up in order
        // (stores and loads that are coherent across the device by themselves: a release fence would write a whole L2 back)
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
            const uint32_t col = nt * (64u * FN) + (wn * FN + (uint32_t)j) * 32u + (lane & 31u);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const uint32_t row = mt * (64u * FM) + (wm * FM + (uint32_t)i) * 32u + 8u * (v >> 2) + 4u * (lane >> 5) + (v & 3u);
                if (row < a.M && col < a.N) a.Y[(size_t)row * a.ldy + col] = acc[i][j][v];
            }
        }
}

template <int FM, int FN, int GS, int ST>
int launch_tiles(const DenseArgs& a, hipStream_t s) {
    static std::atomic<uint64_t> raised{0};
    auto kern = gemm_dense_kernel<FM, FN, GS, ST>;
    if (int rc = ensure_max_lds(raised, reinterpret_cast<const void*>(kern), 160 * 1024 - 64)) return rc;
    hipLaunchKernelGGL(kern, dim3(a.MT * a.NT * a.parts), dim3(256), (size_t)ST * 2u * GS * (FM + FN) * 1024u, s, a);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

}  // namespace

// Workgroup tile (64 f x 64 f) and parts along K for M tokens and N weight rows, by an estimate of the clocks.  A workgroup's stage
// (16 KB) takes 480 (f = 1) or 540; the stages of the workgroups of a compute unit add up, and the last of them leave others without
// work.  A workgroup that has a part of K stores its whole tile, 2500 f^2 clocks that add up in the same way, and one of a tile's
// workgroups reads all of its parts.  (Counted once instead of for every workgroup, the stores let large products be cut in two:
// 11008 x 4096, 2048 tokens 276 us instead of 201, 512 tokens 97 instead of 78.)
// Over 30 measured pairs of shape and batch (500 to 11008 rows, 1024 to 11008 columns, 33 to 2048 tokens) the choice is 0.4 % slower
// than the best of f = 1, 2 and 1, 2, 4, 8 parts on average, 3.5 % at most; over 20 others that the numbers were not taken from (35 to
// 3000 tokens) 1.4 %, 12 % at most.  719 x 3840, 81 tokens: f = 1 in 1 / 4 parts 23.5 / 17.1 us,
// f = 2 in 1 / 4 39.1 / 24.6; 4096 x 11008, 700 tokens: f = 2 in 1 / 2 / 4 parts 114 / 111 / 134 us.
struct DensePlan { uint32_t f, parts; double clocks; };
static DensePlan dense_plan(uint32_t M, uint32_t N, uint32_t K) {
    const double cus = (double)device_cu_count();
    DensePlan best{2u, 1u, 1e30};
    for (uint32_t f = 1; f <= 2u; ++f)
        for (uint32_t parts = 1; parts <= 8u && parts * 4u <= K / 64u; parts *= 2u) {
            const uint32_t t = 64u * f;
            const double wgs = (double)((M + t - 1u) / t) * (double)((N + t - 1u) / t) * parts, each = std::max(wgs / cus, 1.0);
            const double stages = (double)K * f / 64.0 / parts * (f == 1u ? 480.0 : 540.0);
            const double clocks = (wgs <= cus ? 1.0 : each + 0.2) * stages + (parts > 1u ? (2500.0 * each + 1000.0 * parts) * f * f : 0.0);
            if (clocks < best.clocks) best = {f, parts, clocks};
        }
    return best;
}

// The whole call, for the choice between this product and the one that decodes its weights itself: the launch that writes the operands at 5.3 TB/s behind
// 5 us, the product at 1.9 GHz.  Planner's mix, estimate and time: 5000 x 2816, 437 tokens 36 / 33.8 us; 900 x 1024, 50 tokens 9.8 / 9.3; 2000 x 4096, 200 tokens
// 18.8 / 19.9; 4096 x 11008, 64 tokens 36 / 37; 11008 x 4096, 512 / 2048 tokens 78 / 73, 224 / 200.
double dense_estimate_us(uint32_t M, uint32_t N, uint32_t K) {
    return dense_plan(M, N, K).clocks / 1900.0 + 5.0 + 2.0 * K * ((double)N + M) / 5.3e6;
}

// Prefill over a tensor of any format (full 256-weight blocks): slabs of weight rows are decoded to bf16 in a scratch
// buffer of the stream (dequantize_block_all's values, each rounded once to bf16) in the launch that also brings the activations
// into fragment order.  Returns 1 when the tensor's layout is not covered.
int launch_gemm_any(const oilhip_weights& w, const void* d_x, bool x_is_f32, float* d_y, int M_, hipStream_t s) {
    if (w.rows > 0x7FFFFFFFull || w.cols > 0x7FFFFFFFull) return fail(OILHIP_E_ARG, "matrix too large for the prefill kernel");
    const uint32_t N = (uint32_t)w.rows, K = (uint32_t)w.cols, M = (uint32_t)M_;
    if ((uint64_t)M * K * 2u >= 0x80000000ull) return fail(OILHIP_E_ARG, "activation matrix too large for the prefill kernel");
    if (!dense_prepare_covers(w)) return 1;            // before any scratch is allocated for it
    // slab: at most 128 MB of bf16, a multiple of 256 rows
    const uint32_t slab = (uint32_t)std::min<uint64_t>((N + 255u) & ~255u, std::max<uint64_t>(256, ((128ull << 20) / ((uint64_t)K * 2u)) & ~255ull));
    if ((uint64_t)K * 512u >= 0x80000000ull) return fail(OILHIP_E_ARG, "rows too wide for the prefill kernel");
    const StreamLock lock(s);
    uint16_t *wf = nullptr, *xf = nullptr;
    if (int rc = stream_scratch(lock, kScratchGemmW, (size_t)slab * K * 2, reinterpret_cast<void**>(&wf))) return rc;
    const uint32_t mpad = (M + 255u) & ~255u;
    if (int rc = stream_scratch(lock, kScratchGemmX, (size_t)mpad * K * 2, reinterpret_cast<void**>(&xf))) return rc;
    for (uint32_t n0 = 0; n0 < N; n0 += slab) {
        const uint32_t nc = std::min(slab, N - n0);
        const DensePlan pl = dense_plan(M, nc, K);
        const uint32_t t = 64u * pl.f;
        DenseArgs a{xf, wf, d_y + n0, nullptr, nullptr, M, nc, K, N, (M + t - 1u) / t, (nc + t - 1u) / t, pl.parts};
        if (a.parts > 1u) {
            void* p = nullptr;
            const size_t counters = ((size_t)a.MT * a.NT * 4u + 255u) & ~(size_t)255u;
            if (int rc = stream_scratch(lock, kScratchGemmP, counters + (size_t)a.MT * a.NT * a.parts * t * t * 4u, &p)) return rc;
            a.arrived = static_cast<uint32_t*>(p);
            a.partial = reinterpret_cast<float*>(static_cast<uint8_t*>(p) + counters);
        }
        if (int rc = launch_dense_prepare(w, n0, nc, wf, n0 == 0 ? d_x : nullptr, x_is_f32, M, xf, a.arrived, a.MT * a.NT, s)) return rc;
        const int rc = pl.f == 1u ? launch_tiles<1, 1, 4, 4>(a, s) : launch_tiles<2, 2, 2, 4>(a, s);
        if (rc) return rc;
    }
    return OILHIP_OK;
}

}  // namespace oilhip
