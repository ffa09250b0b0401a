// gemv_oil4_multi.hip -- decode GEMV over uniform OIL4 tensors for a handful of activation rows (up to 4, 8, 16 or 32 tokens
// per pass): Qwen35Engine::gemm with small B (src/adapters/tools/qwen35_engine.cpp:47-85) and the per-expert batches of
// moe_dispatch_batched (src/moe_variants.cpp:767-827).
//
// The products run on the matrix cores in INT8, exactly.  The sixteen levels (src/block_codec.cpp:18-23) have four decimals:
// 10000 times a level is an integer n of at most 15 bits, n = 256 a + b with a and b signed bytes, neither of them 0 or
// -128, and level q < 8 is minus level 15 - q.  So a code becomes its two digits without a table in memory: three bits
// of four codes at a time select bytes of an 8-byte table held in two registers (v_perm_b32), and the sign is applied to
// the four bytes at once (x ^ m) + (m & 1) (v_xad_u32; no carry crosses bytes because no digit is 0): 17 vector instructions
// per dword of eight codes.  An activation is scaled by a power of two per (token, block of 256) and rounded to four
// signed bytes (|X| < 127.5 * 2^24: the rounding is 2^-31 to 2^-32 of the block's largest magnitude, and values from a 128th of it on are
// exact); sums over a block are exact in INT32, then scaled in FP32 by the block's FP16 scale and the power of two.
// Three bytes would leave 23 bits of the largest value to all of them: with one activation of 1000 among ordinary ones in every block,
// an error of 6e-7 instead of 1e-7 with FP16 pairs or four bytes.  v_mfma_i32_16x16x64_i8 takes the
// activations as its rows and 16 weight rows as its columns, so a lane's outputs belong to one weight row and meet one scale.
//
// A wavefront takes every n-th block of the row for a run of 16-row groups; the activations of its block sit in registers
// and serve every group of the run, and the wavefronts' sums meet in LDS once per run.  Where a workgroup would have few row groups,
// several share them and cut K (best_cut): their sums meet in memory and the last to arrive adds them up in order, so the order of every sum is fixed.
// Long launches read a byte's digits from a 64 KB table in LDS (whole_cut) instead of forming them: 8 vector instructions and 4 LDS reads
// for eight codes.
// What bounds it: the intake of activations, then the work on them, one after the other.  A compute unit takes in about 30 bytes per clock;
// activations are 4 to 32 KB per block and workgroup, weights 2 KB per block and row group.  Clocks inside a workgroup (4096 x 11008, 16 tokens,
// K whole, one row group): loads issued at 3200, the first wavefront's data at 5000 and its sums at 7900, the last one's sums at
// 14200; the next third of K the same, the end at 33600.  On tall tensors vector issue (about 170 instructions per block of 16 rows, of which
// 4.6 to 5 clocks each; 100 with the table) beside 8 to 56 matrix instructions (16 clocks each, 6.5 of which hold the issue back), and memory:
// 131072 x 4096, 4 tokens 5.2 TB/s.
// Before (FP16 halves of levels from a 64 KB LDS table, K cut between workgroups) -> now, pre-pass included, weights from memory:
//   11008 x 4096, 4 / 8 / 16 / 32 tokens: 12.9 / 12.9 / 15.0 / 19.9 us -> 11.7 / 13.2 / 15.3 / 21.0 us
//   4096 x 11008: 17.4 / 18.0 / 20.5 / 25.8 us -> 13.9 / 16.1 / 18.0 / 24.5 us
//   131072 x 4096, 4 / 16 / 32 tokens: 81 / 86 / 127 us -> 62 / 90 / 141 us;  30000 x 14336: 77 / 81 / 120 us -> 61 / 85 / 131 us
//   2838 x 512, 5 / 16 / 32 tokens: 7.5 / 8.7 / 9.3 -> 5.4 / 5.7 / 7.1 us
// (slower with more than 16 tokens of tall tensors, where four digits cost more than the table did)
// Error against 64 bits (2-norm): 1.8e-7 -> 0.9e-7, whatever the distribution of the activations.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "level_digits.h"
#include "oil4_lds.h"
#include "pack_activations.h"

namespace oilhip {
namespace {

using namespace oil4;

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Passes by token count.  The activation operand of one matrix instruction has 16 rows.  Few: up to four tokens, their
// four digits side by side (row 4 t + d is digit d of token t), so two instructions (digits a and b of the weights) give all eight
// products.  Digits: 16 tokens per tile and a tile of rows per digit, seven instructions.  The product of the two lowest
// digits is left out (2^-31 of the result's scale).  NT tiles of tokens share the decoded weights.
// 9 to 12 tokens: three tiles of few (24 matrix instructions for a block of 16 rows instead of 28, and 3 sums of a lane instead of 28).  17 to 24: a
// tile by digits and one or two of few (36 or 44 instead of 56).  With tiles by digits alone -> now, 12 / 20 / 24 tokens: 11008 x 4096 14.3 / 18.9 / 18.7 ->
// 13.8 / 15.2 / 16.4 us, 2816 x 7424 14.3 / 20.4 / 20.4 -> 13.1 / 15.0 / 15.2, 20000 x 8192 33.0 / 47.0 / 47.0 -> 30.7 / 38.3 / 42.9.
enum PassKind { kFew4 = 0, kFew8 = 1, kFew12 = 2, kDigits16 = 3, kMixed20 = 4, kMixed24 = 5, kDigits32 = 6, kPassKinds = 7 };
__host__ __device__ constexpr bool kind_few(int k) { return k < kDigits16; }
__host__ __device__ constexpr bool tile_few(int k, int t) { return kind_few(k) || ((k == kMixed20 || k == kMixed24) && t > 0); }
__host__ __device__ constexpr int kind_tiles(int k) { return k == kFew4 || k == kDigits16 ? 1 : k == kFew12 || k == kMixed24 ? 3 : 2; }
__host__ __device__ constexpr int tile_outputs(int k, int t) { return tile_few(k, t) ? 1 : 4; }             // of a lane
__host__ __device__ constexpr int outputs_before(int k, int t) { return t == 0 ? 0 : outputs_before(k, t - 1) + tile_outputs(k, t - 1); }
__host__ __device__ constexpr int lane_outputs(int k) { return outputs_before(k, kind_tiles(k)); }
__host__ __device__ constexpr uint32_t tokens_before(int k, int t) { return t == 0 ? 0u : tokens_before(k, t - 1) + (tile_few(k, t - 1) ? 4u : 16u); }
__host__ __device__ constexpr uint32_t kind_tokens(int k) { return tokens_before(k, kind_tiles(k)); }
// packed bytes of one block: 1 KB pieces (64 lanes x 16 bytes), four per operand (half of the block x half of its nibbles) for a
// tile of few, sixteen for one by digits: 1 KB per token
__host__ __device__ constexpr uint32_t kind_block_bytes(int k) { return kind_tokens(k) * 1024u; }
inline int kind_of(int tokens) { return tokens <= 4 ? kFew4 : tokens <= 8 ? kFew8 : tokens <= 12 ? kFew12 : tokens <= 16 ? kDigits16 : tokens <= 20 ? kMixed20 : tokens <= 24 ? kMixed24 : kDigits32; }

// blocks of activations that a wavefront holds: as many as the registers take
// (8 wavefronts per CU, 256 registers each, or 16 with 128)
constexpr int x_slots(int kind, int waves) { return kind == kFew4 ? 4 : kind == kFew8 ? 3 : (kind == kFew12 || kind == kDigits16) && waves == 8 ? 2 : 1; }
constexpr int kMaxTokens = 32;
constexpr uint32_t kMaxSplit = 8;
// row groups of a run
constexpr int longest_run(int kind, int waves) { return kind >= kMixed24 ? 3 : waves == 16 ? 2 : 4; }
constexpr uint32_t kMaxKeep = 24u * 1024u, kMaxKeepNoTable = 48u * 1024u;  // bytes of LDS for sums that are carried from part to part

// ---- pre-pass: activations to digits in operand order -----------------------------------------------------------------
// A wavefront takes one (token, block): 256 columns as one 16-byte load per lane, optionally silu(x) * x2 or the RMSNorm's
// x / rms * (1 + w), the largest magnitude, the digits by nibble position in LDS, and 64 16-byte pieces out.  Column i of a block sits at nibble p = 4 + i - i / 64 (columns 63,
// 127, 191, 255 meet empty slots and nibbles 0..3 the block's scale: both see activation 0).
// Several batches in one launch (the experts of a mixture-of-experts step): batch j packs M[j] rows of x into
// xp + xp_off[j]; its rows are list[row0[j] + m] when use_list is set, else row0[j] + m.  The list travels by value with
// the launch, so the host needs no copy and no synchronisation.
// (more than 16 tokens: the table leaves room for runs of two groups only, 3.6 -> 3.7 us per group of 16 blocks)
__host__ __device__ constexpr bool jobs_table(int kind) { return kind <= kDigits16; }
// row groups of a run beside the other bodies, without spilling registers
constexpr int jobs_run(int kind) { return kind == kDigits32 ? 2 : kind == kMixed24 ? 3 : 4; }
constexpr int kMaxJobs = 32, kMaxListed = 448;
struct PackJobs {
    uint32_t n;                 // 0: one batch, described by PackArgs alone
    uint32_t begin[kMaxJobs + 1];   // workgroups of batch j
    uint16_t M[kMaxJobs], row0[kMaxJobs];
    uint32_t xp_off[kMaxJobs];
    uint8_t kind[kMaxJobs];
    int use_list;
    bool table;                 // pack in the order of multi_body's TABLE, where jobs_table allows it
    int16_t list[kMaxListed];
};
// where a batch's powers of two start (floats [block][kMaxTokens]) and its packed blocks after them
__host__ __device__ constexpr uint32_t undo_bytes(uint32_t bpr) { return bpr * (uint32_t)kMaxTokens * 4u; }

struct PackArgs {
    Activations in;
    const int* tok;
    uint8_t* xp;                // undo floats at the start, then the blocks
    uint32_t bpr, xrows;
    int M, kind;
    uint32_t* arrived;          // counters that the main launch wants zero
    uint32_t ncount;
};

// A block's 256 columns (four per lane) to digits: put(e, p, bytes) receives for column e of the lane its nibble p and the digits
// as bytes 0 (low) to 3.  Returns what undoes the scaling.  Uniform over the wavefront.
template <class Put>
__device__ __forceinline__ float block_to_digits(float (&v)[4], uint32_t lane, Put&& put) {
    if ((lane & 15u) == 15u) v[3] = 0.0f;                                  // column 64 n + 63: no weight there
    // the largest magnitude as a bit pattern: infinities and NaN are the largest of all
    uint32_t top = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) top = max(top, __float_as_uint(v[e]) & 0x7FFFFFFFu);
    top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
    top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x4E, 0xF, 0xF, true));    // [2,3,0,1]
    top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x141, 0xF, 0xF, true));   // row_half_mirror
    top = max(top, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x140, 0xF, 0xF, true));   // row_mirror
    top = max(max((uint32_t)__builtin_amdgcn_readlane((int)top, 0), (uint32_t)__builtin_amdgcn_readlane((int)top, 16)),
              max((uint32_t)__builtin_amdgcn_readlane((int)top, 32), (uint32_t)__builtin_amdgcn_readlane((int)top, 48)));
    const bool bad = top >= 0x7F800000u;
    // the power of two that brings the largest magnitude to [2^30, 2^31), one less where its top digit would pass 127 (above
    // 0x7F7F7F7F, a mantissa above 0x7EFEFE); magnitudes below 2^-119 go lower, so that the power that undoes it stays a float
    int ex = 30 - ((int)(top >> 23) - 127) - ((top & 0x7FFFFFu) > 0x7EFEFEu ? 1 : 0);
    ex = top == 0u || bad ? 0 : ex > 149 ? 149 : ex;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t i = 4u * lane + (uint32_t)e, p = 4u + i - (i >> 6);
        const int X = bad ? 0 : (int)rintf(ldexpf(v[e], ex));
        if ((i & 63u) != 63u) put(e, p, ((uint32_t)X + 0x80808080u) ^ 0x80808080u);   // signed digits: the bytes of X + 128 (1 + 2^8 + 2^16 + 2^24), less 128 each
    }
    return bad ? __uint_as_float(0x7FC00000u) : ldexpf(1.0f, -ex);
}

// BY_TABLE: in the order of multi_body's TABLE.  (One batch, without the jobs: 1.4 KB of arguments cost the host 1.2 us of a launch.)
template <bool BY_TABLE>
__device__ __forceinline__ void pack_body(const PackArgs& a, uint32_t blk, uint32_t four, uint32_t jobs, bool use_list, uint32_t row0, const int16_t* list);

template <bool BY_TABLE>
__global__ void __launch_bounds__(256)
pack_digits_kernel(const PackArgs a) {
    // all arguments at once: read where they are needed, each adds a scalar load's latency (3.04 -> 2.85 us for a few blocks)
    asm volatile("" :: "s"(a.in.x), "s"(a.in.x2), "s"(a.in.norm_w), "s"(a.in.ldx), "s"(a.in.aligned), "s"(a.tok), "s"(a.xp), "s"(a.xrows), "s"(a.M), "s"(a.kind));
    pack_body<BY_TABLE>(a, blockIdx.x, blockIdx.y, 0u, false, 0u, nullptr);
    if (a.ncount && blockIdx.x + blockIdx.y == 0) for (uint32_t i = threadIdx.x; i < a.ncount; i += 256u) a.arrived[i] = 0u;
}
__global__ void __launch_bounds__(256)
pack_digits_jobs_kernel(PackArgs a, const PackJobs jobs) {
    uint32_t j = 0, bid = blockIdx.x;
    while (j + 1u < jobs.n && bid >= jobs.begin[j + 1u]) ++j;              // uniform
    a.M = jobs.M[j]; a.kind = jobs.kind[j]; a.xp += jobs.xp_off[j];
    bid -= jobs.begin[j];
    const uint32_t four = bid / a.bpr, blk = bid - four * a.bpr;
    if (jobs.table && jobs_table(a.kind)) pack_body<true>(a, blk, four, jobs.n, jobs.use_list, jobs.row0[j], jobs.list);
    else pack_body<false>(a, blk, four, jobs.n, jobs.use_list, jobs.row0[j], jobs.list);
}

template <bool BY_TABLE>
__device__ __forceinline__ void pack_body(const PackArgs& a, uint32_t blk, uint32_t four, uint32_t jobs, bool use_list, uint32_t row0, const int16_t* list) {
    __shared__ __align__(16) uint8_t lds[4][1024];
    const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // workgroup = four tokens (number `four`) of one block
    const uint32_t t = four * 4u + wave;
    uint32_t src = 0xFFFFFFFFu;
    if ((int)t < a.M) src = jobs ? (use_list ? (uint32_t)list[row0 + t] : row0 + t) : a.tok ? (uint32_t)a.tok[t] : t;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (src < a.xrows) load_activations(a.in, src, blk, a.bpr, lane, v);
    // digit d of nibble p at byte d * 256 + ((2 (p / 128) + s) * 4 + (p / 32) % 4) * 16 + i: 16-byte pieces by (operand, lane group); the
    // operands of a half are its even and odd nibbles, s = p % 2 and i = (p % 32) / 2, or by table the halves of a lane's 32
    auto place = [&](uint32_t p) {
        const uint32_t sub = BY_TABLE ? (p >> 4) & 1u : p & 1u, i = BY_TABLE ? p & 15u : (p & 31u) >> 1;
        return (((p >> 7) * 2u + sub) * 4u + ((p >> 5) & 3u)) * 16u + i;
    };
    uint8_t* mine = lds[wave];
    if (lane < 4u) {
        const uint32_t at = place(lane);
        mine[at] = 0; mine[256u + at] = 0; mine[512u + at] = 0; mine[768u + at] = 0;
    }
    const float undo = block_to_digits(v, lane, [&](int, uint32_t p, uint32_t bytes) {
        const uint32_t at = place(p);
        mine[at] = (uint8_t)bytes; mine[256u + at] = (uint8_t)(bytes >> 8); mine[512u + at] = (uint8_t)(bytes >> 16); mine[768u + at] = (uint8_t)(bytes >> 24);
    });
    // the token's tile: by digits (the first sixteen, or all), or of few
    const bool few = kind_few(a.kind) || (t >= 16u && a.kind != kDigits32);
    const uint32_t tokens = few ? 4u : 16u, tt = t & (tokens - 1u);
    if (lane == 0) reinterpret_cast<float*>(a.xp)[blk * (uint32_t)kMaxTokens + t] = undo;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // lane = (digit, operand, lane group): one 16-byte piece
    const uint32_t d = lane >> 4, op = (lane >> 2) & 3u, kq = lane & 3u;
    const uint4 piece = *reinterpret_cast<const uint4*>(mine + 16u * lane);
    uint8_t* o = a.xp + undo_bytes(a.bpr) + (size_t)blk * kind_block_bytes(a.kind);
    o += (t - tt) * 1024u;                                                 // the tiles before: 1 KB per token
    if (few) *reinterpret_cast<uint4*>(o + op * 1024u + (kq * 16u + tt * 4u + d) * 16u) = piece;
    else *reinterpret_cast<uint4*>(o + (d * 4u + op) * 1024u + (kq * 16u + tt) * 16u) = piece;
}

// ---- main kernel --------------------------------------------------------------------------------------------------
// Several tensors of one shape in one launch (the experts of a mixture-of-experts step).  A tensor brings its packed activations,
// batch size and output; with K cut, the products of part p > 0 go to rows row0 + m of sums[p - 1].  A job is one tensor's row groups for one part of K; the jobs
// lie one behind the other (tensor by tensor, part by part) and the launch's workgroups take pieces of that line: of job j workgroup wg[j]
// takes the first `first` groups, the ones behind it `each` each, and one that has room left goes on with the job after it.
constexpr uint32_t kMaxLines = 64;
struct MultiJobs {
    uint32_t n, split;
    uint32_t first[kMaxLines], each[kMaxLines];
    uint16_t wg[kMaxLines];
    const uint8_t* W[kMaxJobs];
    float* y[kMaxJobs];
    float* sums[kMaxBatchParts - 1];
    uint32_t ld[kMaxBatchParts];
    uint32_t xp_off[kMaxJobs];
    uint16_t row0[kMaxJobs];
    uint8_t M[kMaxJobs], kind[kMaxJobs];
};

// how a pass size walks a job's blocks: steps begin[k][p] to end[k][p] - 1 of blocks[k][p] blocks each
struct PartsOf { uint16_t begin[kPassKinds][kMaxBatchParts], end[kPassKinds][kMaxBatchParts], blocks[kPassKinds][kMaxBatchParts]; uint32_t chunk[kPassKinds]; };

template <int KIND>
struct Sums {                                                              // one block's integer sums of one token tile
    static constexpr int N = kind_few(KIND) ? 2 : 4;
    i32x4 s[N];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < N; ++i) s[i] = i32x4{0, 0, 0, 0};
    }
};

// Digits of a packed byte, 64 KB at LDS offset 0: entry of byte value v at byte 256 v + 4 lane (a copy per lane: no bank conflicts),
// {a, b} of its low nibble, {a, b} of its high one.
constexpr uint32_t kDigitTab = 65536u;
__device__ __forceinline__ void build_digit_table(uint8_t* lds) {
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t q = threadIdx.x >> 6; q < 64u; q += blockDim.x >> 6) {   // four entries at a time: byte values 4 q + lane / 16
        uint32_t a, b;
        level_digits(((q & 3u) * 4u + (lane >> 4)) | (q >> 2) << 8, a, b);
        const uint32_t e = __builtin_amdgcn_perm(b, a, 0x05010400u);
        reinterpret_cast<uint4*>(lds)[q * 64u + lane] = make_uint4(e, e, e, e);
    }
}
// the entries of a dword's four bytes; `lane4`: 4 * lane
__device__ __forceinline__ void digit_entries(uint32_t w, uint32_t lane4, uint32_t* e) {
    e[0] = *(lds_cuint*)(uintptr_t)__builtin_amdgcn_perm(w, lane4, 0x0C0C0400u);
    e[1] = *(lds_cuint*)(uintptr_t)__builtin_amdgcn_perm(w, lane4, 0x0C0C0500u);
    e[2] = *(lds_cuint*)(uintptr_t)__builtin_amdgcn_perm(w, lane4, 0x0C0C0600u);
    e[3] = *(lds_cuint*)(uintptr_t)__builtin_amdgcn_perm(w, lane4, 0x0C0C0700u);
}

struct BodyArgs {
    const uint8_t* W;
    const uint8_t* xp;             // packed activations
    float* y;
    uint32_t rows, bpr, ldy;
    uint32_t parts, part_blocks;   // the row's blocks, cut so that the wavefronts hold the activations of a part
    uint32_t chunk;                // groups that go through all parts together: their sums wait in LDS
    int M;
    uint32_t part0 = 0;            // this workgroup walks parts part0 to parts - 1
};

// K cut between workgroups: `n` workgroups (1: no cut) share the rows and take each parts / n parts (rounded up).  Their sums meet
// in memory, [workgroup][token][row], and the last of them to arrive adds them up in order.
struct Split {
    uint32_t n = 1, each = 0, ld = 0;
    float* partial = nullptr;
    uint32_t* arrived = nullptr;
};

// G: row groups of a run.  Workgroups of a runtime number of at most kMaxWaves wavefronts, so that a part's blocks divide
// evenly among them; one that has a block less than the others takes the last one again, scaled by 0.  A workgroup walks the
// runs of a chunk of its groups for one part of the rows after the other: activations that are fetched once per part cost nothing, fetched
// once per run they cost as much as the products (37449 x 14336, 16 tokens: 98 us against 73).  The sums wait in LDS.
// FROM: a workgroup may begin with a later part than the first.  SPLIT: its sums go to `partial`.
template <int KIND, int G, int kMaxWaves, bool TABLE, bool SPLIT, bool FROM = SPLIT>
__device__ __forceinline__ void
multi_body(const BodyArgs& a, uint32_t g_begin, uint32_t g_end, float* lds, float* partial = nullptr, uint32_t ldp = 0) {
    constexpr int NT = kind_tiles(KIND), PER = kind_few(KIND) ? 1 : 4, DIG = PER;   // at most: outputs of a lane per tile, operand pieces per half and parity
    constexpr int XD = x_slots(KIND, kMaxWaves);
    constexpr int WD = G < 3 ? XD : 1;                                     // weights in flight: the run's, for short runs of all blocks of the part
    const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), waves = blockDim.x >> 6;
    const uint32_t li = lane & 15u, kq = lane >> 4;
    const uint32_t row_bytes = a.bpr * 128u, bpr = a.bpr, part0 = FROM ? a.part0 : 0u;
    const uint32_t iters = (a.part_blocks + waves - 1u) / waves;           // blocks per wavefront and part, at most XD
    // this workgroup's rows: 32-bit offsets from its first group
    const uint8_t* base = a.W + (size_t)g_begin * 16u * row_bytes;
    const uint32_t last = a.rows - 1u - 16u * g_begin, ngroups = g_end - g_begin;   // rows past the end repeat the last one
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), (short)0, (int)0xFFFFFFFFu, 0x00020000);
    const float* undo = reinterpret_cast<const float*>(a.xp);
    const uint8_t* xblocks = a.xp + undo_bytes(bpr);
    // five to twelve tokens: rows of absent ones in the last tile repeat a present one, and nothing more is fetched (5 tokens, 4096 x 4096
    // 8.95 -> 8.40 us; for the other sizes level)
    uint32_t xlane[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) xlane[t] = kind_few(KIND) && t > 0 && t == NT - 1 ? kq * 16u + min(li >> 2, (uint32_t)a.M - 4u * t - 1u) * 4u + (li & 3u) : lane;
    const uint32_t scale_lane = li * 4u;                                   // ds_bpermute address of lane li: it holds the block's scale
    auto place = [&](uint32_t part, uint32_t i) { const uint32_t b = wave + i * waves; return b < a.part_blocks ? part * a.part_blocks + b : 0xFFFFFFFFu; };
    auto block_at = [&](uint32_t part, uint32_t i) { const uint32_t b = place(part, i); return b < bpr ? b : bpr - 1u; };

    // the levels' integer form (10^-4), and the 2^8 of the lowest digit product kept: a power of two with the scale, exactly, the rest at the end
    constexpr float kScaleUnit = 0x1p-6f, kAccUnit = 1.6384f;
    u32x4 w[WD][G][2];
    auto load_w = [&](int slot, int g, uint32_t part, uint32_t run, uint32_t i) {
        uint32_t r = (run + (uint32_t)g) * 16u + li;
        r = r < last ? r : last;
        const uint32_t off = r * row_bytes + kq * 16u, so = block_at(part, i) * 128u;
        w[slot][g][0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, so, 2));
        w[slot][g][1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + 64u, so, 2));
    };
    i32x4 x[XD][NT][DIG][4];
    float un[XD][NT][PER];
    auto load_x_operand = [&](int slot, int o, uint32_t blk) {
        const i32x4* p = reinterpret_cast<const i32x4*>(xblocks + (size_t)blk * kind_block_bytes(KIND));
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int d = 0; d < tile_outputs(KIND, t); ++d) x[slot][t][d][o] = p[(int)tokens_before(KIND, t) * 64 + (d * 4 + o) * 64 + (int)xlane[t]];
    };
    auto load_undo = [&](int slot, uint32_t blk) {
        const float* u = undo + blk * (uint32_t)kMaxTokens;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (tile_few(KIND, t)) {
                un[slot][t][0] = u[tokens_before(KIND, t) + kq];
            } else {
                const float4 f = *reinterpret_cast<const float4*>(u + tokens_before(KIND, t) + 4 * kq);
                const float all[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
                for (int v = 0; v < PER; ++v) un[slot][t][v] = all[v];
            }
        }
    };
    auto load_part = [&](uint32_t part) {
#pragma unroll
        for (int s = 0; s < XD; ++s)
            if (s == 0 || (uint32_t)s < iters) {
                const uint32_t blk = block_at(part, (uint32_t)s);
#pragma unroll
                for (int o = 0; o < 4; ++o) load_x_operand(s, o, blk);
                load_undo(s, blk);
            }
    };
    load_part(part0);                                                      // activations first: loads return in order
#pragma unroll
    for (int s = 0; s < WD; ++s)
        if (s == 0 || (uint32_t)s < iters)
#pragma unroll
            for (int g = 0; g < G; ++g) load_w(s, g, part0, 0u, (uint32_t)s);
    // a barrier for LDS alone: __syncthreads() would also wait for the weights that are in flight
    auto lds_barrier = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    if constexpr (TABLE) {
        build_digit_table(reinterpret_cast<uint8_t*>(lds));
        lds_barrier();
    }
    const uint32_t lane4 = 4u * lane;
    float* red = lds + (TABLE ? kDigitTab / 4u : 0u);
    constexpr uint32_t LANE = (uint32_t)lane_outputs(KIND), OUT = (uint32_t)G * LANE * 64u;
    const uint32_t held = kMaxWaves == 8 ? 8u : (waves + 3u) & ~3u, AREA = held * OUT;   // wavefronts that sums are held for
    float* keep = red + 2u * AREA;                                         // sums of the parts before, by run
    if (waves < held) {                                                  // the sums of absent wavefronts read as zero
        for (uint32_t o = waves * OUT + threadIdx.x; o < AREA; o += blockDim.x) { red[o] = 0.0f; red[AREA + o] = 0.0f; }
    }

    float acc[G][NT][PER];
    uint32_t chunk_begin = 0, chunk_end = a.chunk < ngroups ? a.chunk : ngroups;
    auto step = [&](auto slot, uint32_t part, uint32_t run) {
        constexpr int XS = decltype(slot)::value, WS = WD > 1 ? XS : 0;
        constexpr uint32_t i = (uint32_t)XS;
        const bool spare = place(part, i) >= bpr;                          // uniform
        // the step that takes this one's registers: the next one, or this block's in the next run; after the last one: any
        uint32_t ni = WD > 1 ? i : i + 1u, nrun = run, npart = part;
        if (WD > 1 || ni >= iters) { ni = WD > 1 ? i : 0u; nrun += G; }
        if (nrun >= chunk_end) {
            if (npart + 1u < a.parts) { ++npart; nrun = chunk_begin; }
            else { npart = part0; nrun = chunk_end < ngroups ? chunk_end : 0u; }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            Sums<KIND> sum[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) sum[t].clear();
            // the block's FP16 scale: the low half of the first dword of lane li.  It meets the integer sum before the power of two does: a
            // partial sum is below the output's own size then and overflows where the output would (kAccUnit).  A spare block adds 0, or the NaN that its output has anyway.
            float scale = __half2float(__ushort_as_half((unsigned short)__builtin_amdgcn_ds_bpermute((int)scale_lane, (int)w[WS][g][0].x)));
            scale = spare ? 0.0f : scale * kScaleUnit;
#pragma unroll
            for (int o = 0; o < 4; ++o) {                                  // operand: half o / 2 of the block, half of its nibbles
                i32x4 da, db;
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    if constexpr (!TABLE) {
                        uint32_t ad, bd;
                        level_digits((o & 1) ? w[WS][g][o >> 1][d] >> 4 : w[WS][g][o >> 1][d], ad, bd);
                        da[d] = (int)ad; db[d] = (int)bd;
                    } else if (d == 0) {
                        uint32_t e[8];
                        digit_entries(w[WS][g][o >> 1][(o & 1) * 2], lane4, e);
                        digit_entries(w[WS][g][o >> 1][(o & 1) * 2 + 1], lane4, e + 4);
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            da[i] = (int)__builtin_amdgcn_perm(e[2 * i + 1], e[2 * i], 0x06040200u);
                            db[i] = (int)__builtin_amdgcn_perm(e[2 * i + 1], e[2 * i], 0x07050301u);
                        }
                    }
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    if (tile_few(KIND, t)) {
                        sum[t].s[0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[XS][t][0][o], da, sum[t].s[0], 0, 0, 0);
                        sum[t].s[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[XS][t][0][o], db, sum[t].s[1], 0, 0, 0);
                    } else if constexpr (!kind_few(KIND)) {                // digits of the activations: [0] low to [3] high
                        // (an order in which no instruction waits for the one before the last)
                        sum[t].s[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[XS][t][3][o], db, sum[t].s[1], 0, 0, 0);     // 2^24
                        sum[t].s[2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[XS][t][2][o], db, sum[t].s[2], 0, 0, 0);     // 2^16
                        sum[t].s[3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[XS][t][1][o], db, sum[t].s[3], 0, 0, 0);     // 2^8
                        sum[t].s[0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[XS][t][3][o], da, sum[t].s[0], 0, 0, 0);     // 2^32
                        sum[t].s[1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[XS][t][2][o], da, sum[t].s[1], 0, 0, 0);
                        sum[t].s[2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[XS][t][1][o], da, sum[t].s[2], 0, 0, 0);
                        sum[t].s[3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[XS][t][0][o], da, sum[t].s[3], 0, 0, 0);
                    }
                }
            }
            load_w(WS, g, npart, nrun, ni);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (tile_few(KIND, t)) {                                   // element d is digit d of this lane's token
                    // below 252 (128 * 27178 + 128 * 106) < 2^30; the product of the two lowest digits is left out here as well
                    const float f = fmaf((float)(sum[t].s[0][3] * 256 + sum[t].s[1][3]), 65536.0f,
                                         fmaf((float)(sum[t].s[0][2] * 256 + sum[t].s[1][2]), 256.0f, (float)(sum[t].s[0][1] * 256 + (sum[t].s[1][1] + sum[t].s[0][0]))));
                    acc[g][t][0] = fmaf(f * scale, un[XS][t][0], acc[g][t][0]);
                } else if constexpr (!kind_few(KIND)) {
#pragma unroll
                    for (int v = 0; v < PER; ++v) {
                        // below 252 (128 * 128 + 128 * 106) (256 + 1) < 2^31
                        const float f = fmaf((float)(sum[t].s[0][v] * 256 + sum[t].s[1][v]), 65536.0f, (float)(sum[t].s[2][v] * 256 + sum[t].s[3][v]));
                        acc[g][t][v] = fmaf(f * scale, un[XS][t][v], acc[g][t][v]);
                    }
                }
            }
        }
    };
    // the sums of a run, out of the area that all wavefronts have written
    auto finish = [&](uint32_t part, uint32_t run, const float* area) {
        for (uint32_t o = threadIdx.x; o < OUT; o += blockDim.x) {
            float p[kMaxWaves];
#pragma unroll
            for (uint32_t wv = 0; wv < (uint32_t)kMaxWaves; ++wv) p[wv] = area[(kMaxWaves == 8 || wv < 4u || (wv & ~3u) < held ? wv : 0u) * OUT + o];   // all in flight
            float s = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            if constexpr (kMaxWaves == 16) {
                s = held > 4u ? s : (p[0] + p[1]) + (p[2] + p[3]);
                s = held > 8u ? s + ((p[8] + p[9]) + (p[10] + p[11])) : s;
                s = held > 12u ? s + ((p[12] + p[13]) + (p[14] + p[15])) : s;
            }
            float* k = keep + ((run % a.chunk) / G) * OUT + o;             // this thread's own from part to part
            if (part > part0) s += *k;
            if (part + 1u < a.parts) { *k = s; continue; }
            const uint32_t l = o & 63u, e = o >> 6, g = e / LANE, q = e % LANE;   // output q of the lane for group g
            const bool few = kind_few(KIND) || (KIND != kDigits32 && q >= 4u);
            const uint32_t token = few ? 4u * q + (l >> 4) : 16u * (q >> 2) + 4u * (l >> 4) + (q & 3u);
            const uint32_t r = (g_begin + run + g) * 16u + (l & 15u);
            if (run + g < ngroups && r < a.rows && (int)token < a.M) {
                // (stores that are coherent across the device by themselves: a release fence would write a whole L2 back)
                if (SPLIT) __hip_atomic_store(partial + (size_t)token * ldp + r, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else a.y[(size_t)token * a.ldy + r] = s * kAccUnit;
            }
        }
    };
    uint32_t odd = 0, done_part = 0, done_run = 0xFFFFFFFFu;
    for (; chunk_begin < ngroups; chunk_begin = chunk_end, chunk_end = chunk_end + a.chunk < ngroups ? chunk_end + a.chunk : ngroups)
    for (uint32_t part = part0; part < a.parts; ++part) {
        if (a.parts > part0 + 1u && (part > part0 || chunk_begin)) load_part(part);
        for (uint32_t run = chunk_begin; run < chunk_end; run += G) {
            // the run before: its sums are complete since the barrier; the area is written again after the next barrier
            if (done_run != 0xFFFFFFFFu) finish(done_part, done_run, red + (odd ^ 1u) * AREA);
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int v = 0; v < tile_outputs(KIND, t); ++v) acc[g][t][v] = 0.0f;
            step(std::integral_constant<int, 0>{}, part, run);
            if constexpr (XD > 1) if (iters > 1u) step(std::integral_constant<int, 1>{}, part, run);
            if constexpr (XD > 2) if (iters > 2u) step(std::integral_constant<int, 2>{}, part, run);
            if constexpr (XD > 3) if (iters > 3u) step(std::integral_constant<int, 3>{}, part, run);
            float* area = red + odd * AREA + wave * OUT;
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int v = 0; v < tile_outputs(KIND, t); ++v) area[((uint32_t)g * LANE + (uint32_t)(outputs_before(KIND, t) + v)) * 64u + lane] = acc[g][t][v];
            lds_barrier();
            odd ^= 1u;
            done_part = part; done_run = run;
        }
    }
    finish(done_part, done_run, red + (odd ^ 1u) * AREA);
}

template <int KIND, int G, int W, bool TABLE>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(W / 4, W / 4)))
gemv_oil4_multi_kernel(const BodyArgs a, uint32_t g_base, uint32_t g_rem) {
    extern __shared__ __align__(16) float lds[];
    const uint32_t b = blockIdx.x, g0 = b * g_base + (b < g_rem ? b : g_rem);
    multi_body<KIND, G, W, TABLE, false>(a, g0, g0 + g_base + (b < g_rem ? 1u : 0u), lds);
}

// K cut between workgroups.  Workgroups are dealt to the eight XCDs in turn, so neighbours in blockIdx take different parts: with two,
// four or eight parts an XCD's L2 holds one part of the activations.
template <int KIND, int G, int W, bool TABLE>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(W / 4, W / 4)))
gemv_oil4_multi_split_kernel(BodyArgs a, uint32_t g_base, uint32_t g_rem, const Split sp) {
    extern __shared__ __align__(16) float lds[];
    const uint32_t b = blockIdx.x / sp.n, mine = blockIdx.x - b * sp.n, g0 = b * g_base + (b < g_rem ? b : g_rem), g1 = g0 + g_base + (b < g_rem ? 1u : 0u);
    const uint32_t all = a.parts;
    a.part0 = mine * sp.each;
    a.parts = a.part0 + sp.each < all ? a.part0 + sp.each : all;
    multi_body<KIND, G, W, TABLE, true>(a, g0, g1, lds, sp.partial + (size_t)mine * a.M * sp.ld, sp.ld);
    uint32_t* order = reinterpret_cast<uint32_t*>(lds);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this thread's sums are in place before the barrier, the others' before theirs
    __syncthreads();
    if (threadIdx.x == 0) *order = __hip_atomic_fetch_add(sp.arrived + b, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*order + 1u != sp.n) return;
    // four rows of a token at a time, all parts' loads in flight together (rows are padded to sixteen)
    const uint32_t r0 = 16u * g0, quads = 4u * (g1 - g0);
    const auto sums = __builtin_amdgcn_make_buffer_rsrc(sp.partial, (short)0, 0x7FFFFFFF, 0x00020000);
    for (uint32_t o = threadIdx.x; o < quads * (uint32_t)a.M; o += blockDim.x) {
        const uint32_t token = o / quads, r = r0 + 4u * (o - token * quads);
        f32x4 p[kMaxSplit];
        const uint32_t at = (token * sp.ld + r) * 4u, step = (uint32_t)a.M * sp.ld * 4u;
#pragma unroll
        for (uint32_t i = 0; i < kMaxSplit; ++i)           // 16: sc1, past the XCD's own cache; beyond the parts: out of range, zeros
            p[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(sums, i < sp.n ? at + i * step : 0x80000000u, 0, 16));
        f32x4 s = p[0];
#pragma unroll
        for (uint32_t i = 1; i < kMaxSplit; ++i) s += p[i];
        float* y = a.y + (size_t)token * a.ldy + r;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (r + e < a.rows) y[e] = s[e] * 1.6384f;
    }
    if (threadIdx.x == 0) __hip_atomic_store(sp.arrived + b, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch on these activations
}

// Batches of different pass sizes side by side: the job's pass size selects the body.
// What bounds it: 4 and 8 tokens memory (a CU's pace of 23 KB per us is 6 TB/s), more tokens vector and matrix issue, one after the other.  A launch
// lasts as long as its longest workgroup, so the line is cut by an estimate that was fitted to the workgroups themselves, and the down projections cut K
// (with all of K their workgroups had 7 to 13 row groups each and four to seven intakes of activations).  Eight experts 4096 <-> 14336,
// 64 tokens, top-2, whole workgroups per job and K whole -> now: gate / up ends at 157 to 196 us -> 143 to 150, down 105 to 135 -> 76 to 83.
template <bool TABLE>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemv_oil4_multi_jobs_kernel(const uint8_t* __restrict__ xp, uint32_t rows, uint32_t bpr, const PartsOf parts, const MultiJobs jobs) {
    extern __shared__ __align__(16) float lds[];
    const uint32_t lane = threadIdx.x & 63u, lines = jobs.n * jobs.split, groups = (rows + 15u) / 16u;
    // Workgroups are dealt to the eight XCDs in turn: an XCD takes neighbouring pieces of the line, so that its L2 holds one or two jobs' activations.
    const uint32_t wg = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    // the last job that begins before this workgroup (it may reach into it), or the first one
    const uint64_t before = __ballot(lane < lines && (uint32_t)jobs.wg[lane] < wg);
    for (uint32_t line = before ? 63u - (uint32_t)__builtin_clzll(before) : 0u; line < lines && jobs.wg[line] <= wg; ++line) {
        const uint32_t at = wg - jobs.wg[line], f = jobs.first[line], e = jobs.each[line];
        const uint32_t g0 = at ? f + (at - 1u) * e : 0u, to = at ? g0 + e : f, g1 = to < groups ? to : groups;
        if (g0 >= groups) continue;
        const uint32_t j = line / jobs.split, part = line - j * jobs.split, kind = jobs.kind[j];
        float* y = part ? jobs.sums[part - 1u] + (size_t)jobs.row0[j] * jobs.ld[part] : jobs.y[j];
        const BodyArgs a{jobs.W[j], xp + jobs.xp_off[j], y, rows, bpr, jobs.ld[part], parts.end[kind][part], parts.blocks[kind][part], parts.chunk[kind], jobs.M[j], parts.begin[kind][part]};
        switch (kind) {
            case kFew4: multi_body<kFew4, jobs_run(kFew4), 8, TABLE, false, true>(a, g0, g1, lds); break;
            case kFew8: multi_body<kFew8, jobs_run(kFew8), 8, TABLE, false, true>(a, g0, g1, lds); break;
            case kFew12: multi_body<kFew12, jobs_run(kFew12), 8, TABLE, false, true>(a, g0, g1, lds); break;
            case kDigits16: multi_body<kDigits16, jobs_run(kDigits16), 8, TABLE, false, true>(a, g0, g1, lds); break;
            case kMixed20: multi_body<kMixed20, jobs_run(kMixed20), 8, false, false, true>(a, g0, g1, lds); break;
            case kMixed24: multi_body<kMixed24, jobs_run(kMixed24), 8, false, false, true>(a, g0, g1, lds); break;
            default: multi_body<kDigits32, jobs_run(kDigits32), 8, false, false, true>(a, g0, g1, lds); break;
        }
        __syncthreads();                                                   // the next job's sums go to the same places in LDS
    }
}

// How a row's blocks are cut into parts of at most x_slots blocks per wavefront, and the wavefronts of a workgroup: as many as
// divide a part with the least left over.
void cut_row(int kind, int max_waves, uint32_t bpr, uint32_t& parts, uint32_t& part_blocks) {
    const uint32_t most = (uint32_t)(max_waves * x_slots(kind, max_waves));
    parts = (bpr + most - 1u) / most;
    part_blocks = (bpr + parts - 1u) / parts;
    parts = (bpr + part_blocks - 1u) / part_blocks;
}
uint32_t waves_of(int max_waves, uint32_t blocks) { const uint32_t each = (blocks + (uint32_t)max_waves - 1u) / (uint32_t)max_waves; return (blocks + each - 1u) / each; }
// groups whose sums may wait in LDS between parts (a multiple of every run length), and the LDS of a workgroup with `most` groups
constexpr uint32_t chunk_of(int kind, bool table) { return (table ? kMaxKeep : kMaxKeepNoTable) / ((uint32_t)lane_outputs(kind) * 256u) / 12u * 12u; }
size_t lds_of(int kind, int max_waves, uint32_t waves, bool table, int g, uint32_t parts, uint32_t most) {
    const size_t unit = (size_t)lane_outputs(kind) * 256u, waiting = std::min((most + g - 1u) / g * g, chunk_of(kind, table));
    return (table ? kDigitTab : 0u) + unit * (2u * (max_waves == 8 ? 8u : (waves + 3u) & ~3u) * g + (parts > 1u ? waiting : 0u));
}

// How a launch cuts the tensor.
struct Cut {
    uint32_t parts, part_blocks, wgs, most;                                // parts of a row, workgroups along the rows, row groups of the fullest
    uint32_t split, each;                                                  // workgroups along K, parts of each
    int waves, run;                                                        // most wavefronts of a workgroup, row groups of a run
    bool table;                                                            // digits from the table in LDS
};
Cut cut_for(int kind, int waves, bool table, uint32_t rows, uint32_t bpr, uint32_t split) {
    Cut c{};
    c.waves = waves; c.table = table;
    cut_row(kind, waves, (bpr + split - 1u) / split, c.each, c.part_blocks);
    c.parts = (bpr + c.part_blocks - 1u) / c.part_blocks;
    c.split = (c.parts + c.each - 1u) / c.each;
    // eight or sixteen wavefronts per CU, as far as LDS goes
    const uint32_t groups = (rows + 15u) / 16u, w = waves_of(waves, c.part_blocks), cus = (uint32_t)device_cu_count();
    const uint32_t fit = (uint32_t)(kMaxLds / lds_of(kind, waves, w, table, longest_run(kind, waves), c.each, 1u << 20));
    c.wgs = std::max(1u, std::min(groups, cus * std::max(1u, std::min((uint32_t)waves / w, fit)) / c.split));
    c.most = (groups + c.wgs - 1u) / c.wgs;
    // The longest run that divides the fullest workgroup's groups: a run that is not full costs as much as a full one.  Over 136
    // measured shapes (256 to 3000 groups, 2048 to 11008 columns, 4 to 32 tokens) 2.2 % behind the best run length on average, 16 % at most;
    // 16384 x 11008, 32 tokens: runs of 2 / 3 for 4 groups 55 / 78 us; 20480 x 4096, 8 tokens: 1 / 3 / 4 for 5 groups 17.0 / 18.6 / 23.6 us.
    c.run = longest_run(kind, waves);
    while (c.most % (uint32_t)c.run) --c.run;
    return c;
}
// Without a cut along K.  Sixteen wavefronts and the table for 9 to 16 tokens where eight would not fill the SIMDs evenly, or walk many runs
// of one group (8448 x 2816, 16 tokens 13.1 -> 12.3 us, 20000 x 8192 34.1 -> 32.0; 12288 x 4096 stays, 14.7 against 15.2); up to 8 tokens the
// table alone where a wavefront has enough to do to earn its 0.5 us (131072 x 4096, 4 / 8 tokens 60.6 / 66.5 -> 57.1 / 63.1).
Cut whole_cut(int kind, uint32_t rows, uint32_t bpr) {
    Cut c = cut_for(kind, 8, false, rows, bpr, 1u);
    const uint32_t w = waves_of(8, c.part_blocks);
    if (kind == kDigits16 && (w < 8u ? bpr > 8u : c.most >= 16u || (c.run == 1 && c.most >= 5u))) return cut_for(kind, 16, true, rows, bpr, 1u);
    if (kind_few(kind) && c.most * c.each * ((c.part_blocks + w - 1u) / w) >= 16u) return cut_for(kind, 8, true, rows, bpr, 1u);
    return c;
}
// Where a workgroup has few row groups, what it takes in is mostly activations: K is cut between workgroups then.  The line is an estimate in
// us that counts a workgroup's bytes of activations, its work and what the meeting of the sums costs (with more than 16 tokens also their way through memory,
// 0.35 us per 1000 rows and four parts); it was fitted to 1 to 8 parts on 25 shapes (300 to 131072 rows, 1024 to 14336 columns), `least` to 16 more
// (600 to 20000 rows, 2048 to 14336 columns, 4 to 32 tokens): there its choice is 0.4 % slower than the better of cut and whole on average, 7 % at most, and never
// slower than no cut by more than 3 %.  5 tokens, 1 / best: 600 x 14336 15.7 / 10.5 us, 5120 x 13824 23.1 / 18.5; 16 tokens 4096 x 11008 19.4 / 16.5;
// 32 tokens 30.0 / 23.9; 24 tokens 25.2 / 21.2, 14336 x 5120 25.4 / 31.7: stays whole.
Cut best_cut(int kind, uint32_t rows, uint32_t bpr) {
    static const struct { double x, weights, unit, run, meet, meet_part, sums, rows, least; } kCost[kPassKinds] = {
        {1.59e-5, 0.0, 0.517, 0.131, 1.95, 0.19, 0.43, 0.0, 0.97}, {0.92e-5, 0.0, 0.574, 0.103, 2.01, 0.19, 0.0, 0.0, 0.97},
        {0.92e-5, 0.0, 0.630, 0.103, 2.01, 0.19, 0.0, 0.0, 0.95}, {0.99e-5, 7.0e-5, 0.0, 0.0, 2.65, 0.27, 0.0, 0.0, 0.90},
        {0.96e-5, 8.3e-5, 0.0, 0.039, 1.91, 0.37, 0.0, 0.0875e-3, 0.97}, {0.96e-5, 9.3e-5, 0.0, 0.039, 1.91, 0.37, 0.0, 0.0875e-3, 0.97},
        {0.96e-5, 11.3e-5, 0.0, 0.039, 1.91, 0.37, 0.0, 0.0875e-3, 0.97}};
    const auto& k = kCost[kind];
    Cut best = whole_cut(kind, rows, bpr);
    const double x_block = (double)kind_block_bytes(kind);
    if (x_block * bpr < 96e3) return best;
    auto cost = [&](const Cut& c) {
        const uint32_t w = waves_of(c.waves, c.part_blocks), blocks = c.part_blocks * c.each, cus = (uint32_t)device_cu_count();
        const double turns = (double)((c.wgs * c.split + cus - 1u) / cus), side = std::max(1.0, w * turns / 4.0);
        const double units = (double)(c.most * c.each * ((c.part_blocks + w - 1u) / w)) * side;
        double t = turns * blocks * (k.x * x_block + k.weights * 2048.0 * c.most) + k.unit * units + k.run * (double)(c.each * (c.most / (uint32_t)c.run));
        if (c.split > 1u) t += k.meet + (k.meet_part + k.rows * rows) * c.split + k.sums * c.split * c.most * kind_tokens(kind) / 256.0;
        return t;
    };
    // the estimate of the whole row is for the forms that it was fitted on; 4.6 us are in all of them
    double least = (4.6 + cost(cut_for(kind, 8, false, rows, bpr, 1u))) * k.least - 4.6;
    for (uint32_t n : {2u, 3u, 4u, 5u, 6u, 8u}) {
        const Cut c = kind == kDigits16 ? cut_for(kind, 16, true, rows, bpr, n) : cut_for(kind, 8, false, rows, bpr, n);
        if (c.split != n) continue;
        const double t = cost(c);
        if (t < least) { least = t; best = c; }
    }
    return best;
}
// bytes of a split launch's counters and sums
size_t split_bytes(const Cut& c, uint32_t rows, int M) {
    return c.split < 2u ? 0u : (((size_t)c.wgs * 4u + 255u) & ~(size_t)255u) + (size_t)c.split * (size_t)M * ((rows + 15u) & ~15u) * 4u;
}

template <int KIND, int G, int W, bool TABLE, bool SPLIT>
int launch_one(const BodyArgs& a, const Cut& c, const Split& sp, hipStream_t s) {
    static std::atomic<uint64_t> raised{0};
    const uint32_t groups = (a.rows + 15u) / 16u, waves = waves_of(W, a.part_blocks);
    const size_t lds = lds_of(KIND, W, waves, TABLE, G, c.each, c.most);
    if constexpr (SPLIT) {
        if (int rc = ensure_max_lds(raised, (const void*)gemv_oil4_multi_split_kernel<KIND, G, W, TABLE>, kMaxLds)) return rc;
        hipLaunchKernelGGL((gemv_oil4_multi_split_kernel<KIND, G, W, TABLE>), dim3(c.wgs * c.split), dim3(64u * waves), lds, s, a, groups / c.wgs, groups % c.wgs, sp);
    } else {
        if (int rc = ensure_max_lds(raised, (const void*)gemv_oil4_multi_kernel<KIND, G, W, TABLE>, kMaxLds)) return rc;
        hipLaunchKernelGGL((gemv_oil4_multi_kernel<KIND, G, W, TABLE>), dim3(c.wgs), dim3(64u * waves), lds, s, a, groups / c.wgs, groups % c.wgs);
    }
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}
template <int KIND, int W, bool TABLE, bool SPLIT>
int launch_run(const BodyArgs& a, const Cut& c, const Split& sp, hipStream_t s) {
    constexpr int LONGEST = longest_run(KIND, W);
    if constexpr (LONGEST >= 4) if (c.run == 4) return launch_one<KIND, 4, W, TABLE, SPLIT>(a, c, sp, s);
    if constexpr (LONGEST >= 3) if (c.run == 3) return launch_one<KIND, 3, W, TABLE, SPLIT>(a, c, sp, s);
    if (c.run == 2) return launch_one<KIND, 2, W, TABLE, SPLIT>(a, c, sp, s);
    return launch_one<KIND, 1, W, TABLE, SPLIT>(a, c, sp, s);
}
template <int KIND>
int launch_kind(BodyArgs a, const Cut& c, const Split& sp, hipStream_t s) {
    a.parts = c.parts;
    a.part_blocks = c.part_blocks;
    a.chunk = c.each > 1u ? chunk_of(KIND, c.table) : 0x7FFFFFFFu;
    if constexpr (KIND == kDigits16) {
        if (c.split > 1u) return launch_run<KIND, 16, true, true>(a, c, sp, s);
        return c.table ? launch_run<KIND, 16, true, false>(a, c, sp, s) : launch_run<KIND, 8, false, false>(a, c, sp, s);
    } else {
        if (c.split > 1u) return launch_run<KIND, 8, false, true>(a, c, sp, s);
        if constexpr (KIND < kDigits16)
            if (c.table) return launch_run<KIND, 8, true, false>(a, c, sp, s);
        return launch_run<KIND, 8, false, false>(a, c, sp, s);
    }
}

int launch_main(int kind, const BodyArgs& a, const Cut& c, const Split& sp, hipStream_t s) {
    switch (kind) {
        case kFew4: return launch_kind<kFew4>(a, c, sp, s);
        case kFew8: return launch_kind<kFew8>(a, c, sp, s);
        case kFew12: return launch_kind<kFew12>(a, c, sp, s);
        case kDigits16: return launch_kind<kDigits16>(a, c, sp, s);
        case kMixed20: return launch_kind<kMixed20>(a, c, sp, s);
        case kMixed24: return launch_kind<kMixed24>(a, c, sp, s);
        default: return launch_kind<kDigits32>(a, c, sp, s);
    }
}

// 32-bit byte offsets inside a workgroup's rows, 32-bit row numbers
bool shape_covered(const oilhip_weights& w, uint64_t xrows, uint32_t ldx) {
    return w.rows > 0 && w.rows <= 0x7FFFFFFFull && w.cols <= kGemvPackMaxCols && (w.cols & 255u) == 0 && w.cols > 0 &&
           xrows * ldx <= 0x1FFFFFFFFull && (w.rows / (16u * (uint64_t)device_cu_count()) + 6u) * 16u * (w.cols / 2u) < 0x80000000ull;
}

// The scratch of the entry point that allocates nothing: a fixed array in the code object (8 MB, held by every GPU the library
// runs on until the process ends).  In host code the array's name is only a stand-in: the device address comes from
// hipGetSymbolAddress, once per device with that device current, and only that pointer is ever handed to a kernel.
constexpr size_t kStaticScratchBytes = 8u << 20;
static_assert(kStaticScratchBytes >= kGemvPackBytes, "the static scratch holds the packed activations");
static __device__ __align__(256) uint8_t scratch[kStaticScratchBytes];
std::mutex g_static_mu;
uint8_t* g_static_ptr[64] = {};

int static_pack_buffer(uint8_t** out) {
    int dev = 0;
    OILHIP_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return fail(OILHIP_E_ARG, "device index out of range");
    std::lock_guard<std::mutex> lk(g_static_mu);
    if (!g_static_ptr[dev]) {
        void* p = nullptr;
        OILHIP_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(OILHIP_E_DEVICE, "hipGetSymbolAddress returned a null address for the static scratch");
        g_static_ptr[dev] = static_cast<uint8_t*>(p);
    }
    *out = g_static_ptr[dev];
    return OILHIP_OK;
}

}  // namespace

static size_t pack_bytes(uint32_t bpr, int kind) { return undo_bytes(bpr) + (size_t)bpr * kind_block_bytes(kind); }
// What a pass may take of a stream's scratch: it comes in two sizes, one pass, and from rows of more than 4096 weights on the static scratch's.
static size_t pass_room(uint32_t bpr) { return bpr > 16u ? kStaticScratchBytes : kGemvPackBytes; }
// How a pass of m tokens is cut: K only as far as the sums fit behind the activations in a stream's scratch, whatever the scratch of the call is, so that
// captured calls (a workspace) and those that allocate nothing add in the order of the eager one.
static Cut pass_cut(int kind, uint32_t rows, uint32_t bpr, int m) {
    const Cut c = best_cut(kind, rows, bpr);
    return pack_bytes(bpr, kind) + split_bytes(c, rows, m) > pass_room(bpr) ? whole_cut(kind, rows, bpr) : c;
}

size_t gemv_oil4_multi_bytes(const oilhip_weights& w, int M) {
    if (!plain_oil4(w) || !shape_covered(w, 1, (uint32_t)w.cols)) return 0;
    const uint32_t bpr = (uint32_t)(w.cols >> 8);
    auto pass = [&](int m) { return m < 1 ? 0u : pack_bytes(bpr, kind_of(m)) + split_bytes(pass_cut(kind_of(m), (uint32_t)w.rows, bpr, m), (uint32_t)w.rows, m); };
    return M < kMaxTokens ? pass(M) : std::max(pass(kMaxTokens), pass(M % kMaxTokens));
}

// Y[m][r] for m < M: x row tok[m] (or m when tok is null) of an [xrows][ldx] activation matrix; with w2 the same activations
// also go through a second tensor of the same width into d_y2 (the gate and up projections of an expert): they are packed
// once per pass for both.  `in` says what the activations are (common.h).  Returns 1 when the shape is outside what this
// kernel covers.
int launch_gemv_oil4_multi(const oilhip_weights& w, const float* d_x, const int* d_tok, float* d_y, int M, uint32_t ldx, uint32_t ldy,
                           uint32_t xrows, hipStream_t s, const MultiInput& in, const oilhip_weights* w2, float* d_y2, uint32_t ldy2,
                           uint8_t* d_pack, size_t pack_room) {
    if (!shape_covered(w, xrows, ldx)) return 1;
    if (w2 && (w2->cols != w.cols || !shape_covered(*w2, xrows, ldx) || !plain_oil4(*w2) || !d_y2)) return 1;
    const uint32_t bpr = (uint32_t)(w.cols >> 8);
    const StreamLock lock(s);
    uint8_t* xp = d_pack;
    size_t room = pass_room(bpr);
    if (!xp) {
        if (int rc = stream_scratch(lock, kScratchGemvPack, room, reinterpret_cast<void**>(&xp))) return rc;
    } else {
        room = pack_room ? pack_room : gemv_oil4_multi_bytes(w, M);
    }
    // (a second tensor's sums may need more room than a workspace that was made for the first has)
    auto cut = [&](const oilhip_weights& t, int kind, int m, uint8_t* behind, Split& sp) {
        const uint32_t rows = (uint32_t)t.rows;
        Cut c = pass_cut(kind, rows, bpr, m);
        if (c.split > 1u && pack_bytes(bpr, kind) + split_bytes(c, rows, m) > room) c = whole_cut(kind, rows, bpr);
        if (c.split > 1u) sp = {c.split, c.each, (rows + 15u) & ~15u, reinterpret_cast<float*>(behind + (((size_t)c.wgs * 4u + 255u) & ~(size_t)255u)), reinterpret_cast<uint32_t*>(behind)};
        return c;
    };
    const uintptr_t at = reinterpret_cast<uintptr_t>(d_x) | reinterpret_cast<uintptr_t>(in.x2);
    const uint32_t aligned = (at & 15u) == 0 && (ldx & 3u) == 0;
    for (int m0 = 0; m0 < M; m0 += kMaxTokens) {
        const int m = std::min(M - m0, kMaxTokens), kind = kind_of(m);
        const size_t skip = d_tok ? 0 : (size_t)m0 * ldx;
        const Activations act{d_x + skip, in.x2 ? in.x2 + skip : nullptr, in.norm_w, in.xn ? in.xn + skip : nullptr, ldx, aligned, in.inv_form ? 1u : 0u};
        uint8_t* behind = xp + pack_bytes(bpr, kind);
        Split sp{}, sp2{};
        Cut c = cut(w, kind, m, behind, sp), c2 = w2 ? cut(*w2, kind, m, behind, sp2) : Cut{};
        if (w2 && c.table != c2.table) {                                   // the activations are packed in one order
            c = cut_for(kind, 8, false, (uint32_t)w.rows, bpr, 1u);
            c2 = cut_for(kind, 8, false, (uint32_t)w2->rows, bpr, 1u);
            sp = sp2 = Split{};
        }
        const uint32_t counters = std::max(sp.n > 1u ? c.wgs : 0u, sp2.n > 1u ? c2.wgs : 0u);
        hipLaunchKernelGGL(c.table ? pack_digits_kernel<true> : pack_digits_kernel<false>, dim3(bpr, kind_tokens(kind) / 4u), dim3(256), 0, s,
                           PackArgs{act, d_tok ? d_tok + m0 : nullptr, xp, bpr, d_tok ? xrows : xrows - (uint32_t)m0, m, kind, reinterpret_cast<uint32_t*>(behind), counters});
        OILHIP_HIP(hipGetLastError());
        if (int rc = launch_main(kind, BodyArgs{w.d_payload, xp, d_y + (size_t)m0 * ldy, (uint32_t)w.rows, bpr, ldy, 0u, 0u, 0u, m}, c, sp, s)) return rc;
        if (w2)
            if (int rc = launch_main(kind, BodyArgs{w2->d_payload, xp, d_y2 + (size_t)m0 * ldy2, (uint32_t)w2->rows, bpr, ldy2, 0u, 0u, 0u, m}, c2, sp2, s)) return rc;
    }
    return OILHIP_OK;
}

// ---- several batches in one launch (the experts of a mixture-of-experts step) ---------------------------------------
// Batch b multiplies M[b] <= 32 activation rows with tensor wa[b] (and, with wb, with a second tensor of the same shape:
// an expert's gate and up projections share their activations).  All tensors have one shape; the batches may differ in pass
// size.  The activation rows of batch b are rows list[row0[b] + m] of x when `list` is given (the list is passed by value
// with the launch), else rows row0[b] + m; with x2 they are silu(x) * x2.  Outputs: ya[b][m * ldy + r].
// With `sums` K may be cut into up to kMaxBatchParts parts: part p > 0 goes to rows row0[b] + m of sums->to[p - 1], sums->n says how many there
// are, and the caller adds them up.
size_t gemv_oil4_multi_batches_bytes(int nb, uint64_t cols) {
    const uint32_t bpr = (uint32_t)(cols >> 8);
    return (size_t)nb * (undo_bytes(bpr) + (size_t)bpr * kind_block_bytes(kDigits32));
}

namespace {
// Estimated us of a workgroup's piece of a job: a start per step (its activations, the table), then its runs of row groups at the pace of a
// wavefront's blocks.  Fitted to the workgroups of seven steps of four to eight experts (1024 <-> 3584 to 4096 <-> 14336, 1 to 32 tokens
// each) without and with the table, 2 us off on average in pieces of 5 to 170 us.
struct PieceCost { double start, run; };                                   // run: of jobs_run groups
PieceCost piece_cost(int kind, bool table, uint32_t steps, uint32_t blocks, uint32_t waves) {
    static const double kStart[2][kPassKinds] = {{3.6, 3.2, 3.5, 3.9, 2.0, 2.4, 1.9}, {4.5, 4.3, 4.4, 4.5, 2.0, 2.4, 1.9}},
                        kRun[2][kPassKinds] = {{0.083, 0.296, 0.4, 0.533, 0.01, 0.01, 0.01}, {0.1, 0.36, 0.567, 0.79, 0.01, 0.01, 0.01}},
                        kGroupBlock[2][kPassKinds] = {{0.0936, 0.1081, 0.119, 0.1267, 0.169, 0.190, 0.229}, {0.0880, 0.0955, 0.1091, 0.1130, 0.169, 0.190, 0.229}};
    return {kStart[table][kind] * steps, steps * (kRun[table][kind] + 8.0 * ((blocks + waves - 1u) / waves) * kGroupBlock[table][kind] * jobs_run(kind))};
}
}  // namespace

int launch_gemv_oil4_multi_batches(int nb, const oilhip_weights* const* wa, float* const* ya, const oilhip_weights* const* wb, float* const* yb,
                                   const int* M, const int* row0, const int* list, int nlist, const float* d_x, const float* d_x2,
                                   uint32_t ldx, uint32_t xrows, uint32_t ldy, void* d_ws, size_t ws_bytes, hipStream_t s, BatchSums* sums) {
    const int per = wb ? 2 : 1, njobs = per * nb;
    if (nb < 1 || njobs > kMaxJobs || nlist > kMaxListed) return 1;
    const oilhip_weights& w0 = *wa[0];
    if (!shape_covered(w0, xrows, ldx) || xrows > 32767u) return 1;
    if (ws_bytes < gemv_oil4_multi_batches_bytes(nb, w0.cols)) return 1;
    const uint32_t bpr = (uint32_t)(w0.cols >> 8), groups = ((uint32_t)w0.rows + 15u) / 16u;
    PackJobs pj{};
    pj.n = (uint32_t)nb;
    pj.use_list = list ? 1 : 0;
    for (int i = 0; i < nlist; ++i) pj.list[i] = (int16_t)list[i];
    MultiJobs mj{};
    int of_kind[kPassKinds] = {};
    uint32_t xp_at = 0;
    for (int b = 0; b < nb; ++b) {
        if (M[b] < 1 || M[b] > kMaxTokens) return fail(OILHIP_E_ARG, "multi-row batches: a batch exceeds the pass size");
        const int kind = kind_of(M[b]);
        pj.M[b] = (uint16_t)M[b]; pj.row0[b] = (uint16_t)row0[b]; pj.kind[b] = (uint8_t)kind; pj.xp_off[b] = xp_at;
        pj.begin[b + 1] = pj.begin[b] + bpr * kind_tokens(kind) / 4u;
        xp_at += undo_bytes(bpr) + bpr * kind_block_bytes(kind);
        of_kind[kind] += per;
        for (int t = 0; t < per; ++t) {
            const int j = b * per + t;
            const oilhip_weights* w = t ? wb[b] : wa[b];
            if (!plain_oil4(*w) || w->rows != w0.rows || w->cols != w0.cols) return 1;
            mj.W[j] = w->d_payload; mj.y[j] = t ? yb[b] : ya[b]; mj.row0[j] = (uint16_t)row0[b];
            mj.M[j] = (uint8_t)M[b]; mj.kind[j] = (uint8_t)kind; mj.xp_off[j] = pj.xp_off[b];
        }
    }
    // How K is cut: parts of whole steps of eight blocks (the last one takes what is left), walked in the longest steps that the
    // wavefronts hold the activations of; without a cut, steps of one size.
    struct Plan { PartsOf parts; uint32_t split, waves, wgs; bool table; double us; PieceCost cost[kPassKinds][kMaxBatchParts]; };
    auto plan_for = [&](uint32_t split, bool table, Plan& p) {
        p = Plan{};
        p.table = table; p.split = split; p.waves = split > 1u ? 8u : 1u;
        const uint32_t eights = (bpr + 7u) / 8u, q = (eights + split - 1u) / split;
        if (split > 1u && (eights + q - 1u) / q != split) return false;
        for (int k = 0; k < kPassKinds; ++k) {
            if (!of_kind[k]) continue;
            bool steps = false;
            if (split == 1u) {
                uint32_t n, blocks;
                cut_row(k, 8, bpr, n, blocks);
                p.parts.end[k][0] = (uint16_t)n; p.parts.blocks[k][0] = (uint16_t)blocks;
                p.waves = std::max(p.waves, waves_of(8, blocks));
                steps = n > 1u;
            }
            for (uint32_t i = 0; split > 1u && i < split; ++i) {
                const uint32_t at = i * q, mine = std::min(q, eights - at);
                uint32_t step = (uint32_t)x_slots(k, 8);
                while (mine % step || at % step) --step;
                p.parts.begin[k][i] = (uint16_t)(at / step); p.parts.end[k][i] = (uint16_t)((at + mine) / step); p.parts.blocks[k][i] = (uint16_t)(8u * step);
                steps |= mine > step;
            }
            p.parts.chunk[k] = steps ? chunk_of(k, table && jobs_table(k)) : 0x7FFFFFFFu;
        }
        double work = 0.0, start = 0.0, grain = 0.0;
        for (int k = 0; k < kPassKinds; ++k)
            for (uint32_t i = 0; of_kind[k] && i < split; ++i) {
                const uint32_t run = (uint32_t)jobs_run(k);
                const PieceCost c = p.cost[k][i] = piece_cost(k, table, p.parts.end[k][i] - p.parts.begin[k][i], p.parts.blocks[k][i], p.waves);
                const double w = (double)of_kind[k] * ((groups + run - 1u) / run) * c.run;
                work += w; start += w * c.start; grain += w * c.run;
            }
        const uint32_t side = std::max(1u, 8u / p.waves);
        if (table && side > 1u) return false;                              // no room for two tables
        p.wgs = (uint32_t)device_cu_count() * side;
        p.us = work / p.wgs + (start + 0.5 * grain) / work + 0.7 * (split - 1u);
        return true;
    };
    Plan plan, other;
    if (!plan_for(1u, false, plan)) return 1;
    // No plan is below a piece of one run of one step, so small experts, whose steps are bound by the host, leave it at the first plan: working
    // out the others took 1 to 2 us of a step (1 token, 1536 <-> 2048, top-2: 32.8 us -> 31.4; 8 tokens, 1280 <-> 1280: 33.3 -> 30.9).
    double least[2] = {plan.us, plan.us};
    for (int table = 0; table < 2; ++table)
        for (int k = 0; k < kPassKinds; ++k) {
            const PieceCost c = piece_cost(k, table, 1u, 8u, 8u);
            if (of_kind[k]) least[table] = std::min(least[table], c.start + 0.5 * c.run);
        }
    for (uint32_t n = 1; n <= (sums ? (uint32_t)sums->most : 1u) && (uint32_t)njobs * n <= kMaxLines; ++n)
        for (bool table : {false, true})
            if ((n > 1u || table) && least[table] + 0.7 * (n - 1u) < plan.us && plan_for(n, table, other) && other.us < plan.us) plan = other;
    pj.table = plan.table;
    // The line of jobs, cut into pieces of at most `most` us each: the least `most`, to 1 %, that the workgroups suffice for.
    mj.n = (uint32_t)njobs; mj.split = plan.split;
    uint32_t wgs = 0, fullest = 0;
    auto cut_line = [&](double most, MultiJobs& o) {
        uint32_t wg = 0, longest = 0;
        double used = 0.0;
        for (uint32_t line = 0; line < mj.n * mj.split; ++line) {
            const int kind = mj.kind[line / mj.split];
            const uint32_t run = (uint32_t)jobs_run(kind);
            const PieceCost& c = plan.cost[kind][line % mj.split];
            auto fits = [&](double room) { return room > c.run + c.start ? (uint32_t)((room - c.start) / c.run) * run : 0u; };
            const uint32_t e = std::max(fits(most), run);
            uint32_t f = used > 0.0 ? fits(most - used) : e;
            if (f == 0u) { ++wg; used = 0.0; f = e; }
            f = std::min(f, groups);
            const uint32_t more = (groups - f + e - 1u) / e, last = more ? groups - f - (more - 1u) * e : f;
            o.wg[line] = (uint16_t)std::min(wg, 65535u); o.first[line] = f; o.each[line] = e;
            wg += more;
            used = (more ? 0.0 : used) + c.start + (last + run - 1u) / run * c.run;
            longest = std::max({longest, f, more ? e : 0u});
        }
        if (wg >= plan.wgs) return false;
        wgs = wg + 1u; fullest = longest;
        return true;
    };
    double most = plan.us;
    while (!cut_line(most, mj)) most *= 1.02;
    for (double less : {0.92, 0.96, 0.98, 0.99}) {                         // (pieces of one run each get no shorter)
        if (fullest <= 4u) break;
        MultiJobs shorter = mj;
        if (cut_line(most * less, shorter)) { mj = shorter; most *= less; }
    }
    if ((fullest + 6ull) * 16u * (w0.cols / 2u) >= 0x80000000ull) return 1;
    size_t lds = 0;
    for (int k = 0; k < kPassKinds; ++k)
        if (of_kind[k]) lds = std::max(lds, lds_of(k, 8, plan.waves, plan.table && jobs_table(k), jobs_run(k), plan.parts.chunk[k] != 0x7FFFFFFFu ? 2u : 1u, fullest));
    mj.ld[0] = ldy;
    if (sums) {
        sums->n = (int)plan.split;
        for (uint32_t p = 1; p < plan.split; ++p) { mj.sums[p - 1] = sums->to[p - 1]; mj.ld[p] = sums->ld[p - 1]; }
    }
    const uint32_t aligned = ((reinterpret_cast<uintptr_t>(d_x) | reinterpret_cast<uintptr_t>(d_x2)) & 15u) == 0 && (ldx & 3u) == 0;
    const PackArgs a{{d_x, d_x2, nullptr, nullptr, ldx, aligned, 0u}, nullptr, static_cast<uint8_t*>(d_ws), bpr, xrows, 0, 0, nullptr, 0u};
    hipLaunchKernelGGL(pack_digits_jobs_kernel, dim3(pj.begin[nb]), dim3(256), 0, s, a, pj);
    OILHIP_HIP(hipGetLastError());
    static std::atomic<uint64_t> raised[2]{};
    auto kern = plan.table ? gemv_oil4_multi_jobs_kernel<true> : gemv_oil4_multi_jobs_kernel<false>;
    if (int rc = ensure_max_lds(raised[plan.table], (const void*)kern, kMaxLds)) return rc;
    hipLaunchKernelGGL(kern, dim3((wgs + 7u) & ~7u), dim3(64u * plan.waves), lds, s, static_cast<const uint8_t*>(d_ws),
                       (uint32_t)w0.rows, bpr, plan.parts, mj);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

}  // namespace oilhip

extern "C" int oilhip_gemv_oil4_f32_noalloc(const oilhip_weights* w, const float* d_x, float* d_y, int M, void* stream) {
    using namespace oilhip;
    if (int rc = check_matmul_shape(w, d_x, d_y, M)) return rc;
    if (!plain_oil4(*w)) return fail(OILHIP_E_ARG, "gemv_oil4_f32_noalloc: the tensor must be uniform OIL4 in the plain 128-byte block layout");
    if (w->cols > kGemvPackMaxCols)
        return fail(OILHIP_E_ARG, "gemv_oil4_f32_noalloc: rows of " + std::to_string(w->cols) + " weights exceed the static scratch (at most " +
                                      std::to_string(kGemvPackMaxCols) + " columns)");
    hipStream_t s = (hipStream_t)stream;
    int rc = 1;                                                             // 1: shape not covered by that kernel
    if (M <= 2) rc = launch_gemv_oil4(*w, d_x, d_y, M, s);                  // the register-resident kernel uses no scratch
    if (rc == 1 && M >= 2) {
        // the documented limit of this entry point on partial sums, which its callers may rely on being refused at
        const uint64_t parts = M > 16 ? (w->cols + 2047u) / 2048u : (w->cols + 4095u) / 4096u;
        if (parts > 2u && parts * (uint64_t)std::min(M, M > 16 ? 32 : 16) * w->rows > 1043456u)
            return fail(OILHIP_E_ARG, "gemv_oil4_f32_noalloc: this shape needs a kernel that allocates; use oilhip_gemv_f32");
        uint8_t* pack = nullptr;
        if (int e = static_pack_buffer(&pack)) return e;
        rc = launch_gemv_oil4_multi(*w, d_x, nullptr, d_y, M, (uint32_t)w->cols, (uint32_t)w->rows, (uint32_t)M, s, {}, nullptr, nullptr, 0, pack, kStaticScratchBytes);
    }
    if (rc == 1 && M > 2 && M <= 4) rc = launch_gemv_oil4(*w, d_x, d_y, M, s);
    if (rc == 1) return fail(OILHIP_E_ARG, "gemv_oil4_f32_noalloc: this shape needs a kernel that allocates; use oilhip_gemv_f32");
    return rc;
}

// The sums of the decode kernels have a fixed order whatever this says, also where workgroups take parts of K.
extern "C" int oilhip_set_ordered_sums(int ordered) {
    (void)ordered;
    return OILHIP_OK;
}
