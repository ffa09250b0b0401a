// common.h -- shared host-side declarations of liboilhip (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>
#include <string>

#include "../../include/oilhip.h"
#include "block_decode.h"

namespace oilhip {

// bytes of a full 256-weight block of each format (codebook channel + index channel) and of its codebook channel,
// as quantize_block_all writes them (src/block_codec.cpp:368-574)
__host__ __device__ constexpr uint32_t full_block_bytes(int f) {
    constexpr uint32_t n[15] = {16, 48, 64, 128, 256, 512, 1024, 32, 48, 80, 144, 272, 512, 64, 64};
    return f >= 0 && f < 15 ? n[f] : 0u;
}
__host__ __device__ constexpr uint32_t full_block_cb_bytes(int f) { return f == 0 ? 16u : 0u; }

// Thread-local text behind oilhip_last_error().
void set_error(const std::string& msg);
int fail(int code, const std::string& msg);

#define OILHIP_HIP(call)                                                                  \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess)                                                             \
            return ::oilhip::fail(OILHIP_E_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Per-device decode tables (device pointer), created on first use.
int get_tables(const DecodeTables** out);
int device_cu_count();
// shape rules shared by every matmul entry point: non-null pointers, M >= 1, full blocks, cols a multiple of 256
int check_matmul_shape(const oilhip_weights* w, const void* x, const void* y, int M);

// Raises a kernel's dynamic LDS limit once per device.  `done` is the call site's own flag word (one bit per device);
// concurrent first calls may both set the attribute, which is harmless.
int ensure_max_lds(std::atomic<uint64_t>& done, const void* kernel, int bytes);

// Device scratch of at least `bytes` that belongs to (current device, stream, slot): kernels queued on one stream run
// in order, so calls on different streams never share a buffer.  A buffer is never freed or moved while the process
// lives (a captured graph or a queued kernel may still point at it): a request that outgrows it gets a new, larger
// one and the old one stays allocated.  No allocation can happen while the stream is being captured, so the first
// call of a given size on a stream has to be made outside capture; otherwise the call fails with OILHIP_E_ARG.
// New buffers are zero-filled.
// One call's launches write and read the scratch one after the other; a second thread's launches on the same stream must
// not come between them.  So the scratch is asked for under the stream's lock, which the caller holds until the last launch
// that uses it is queued.
enum ScratchSlot { kScratchGemvPack = 0, kScratchGemmX = 1, kScratchTl = 2, kScratchGemmW = 3, kScratchGemmP = 4 };
std::mutex& stream_mutex(hipStream_t s);
class StreamLock {
public:
    explicit StreamLock(hipStream_t s) : stream(s), held_(stream_mutex(s)) {}
    const hipStream_t stream;
private:
    std::lock_guard<std::mutex> held_;
};
int stream_scratch(const StreamLock& lock, int slot, size_t bytes, void** out);
bool stream_capturing(hipStream_t s);

// Tensors whose rows mix formats are stored as `nstreams` streams of windows of at most 4 KB, made for one wavefront each,
// `waves` (8, or 16 with windows of at most 2 KB) wavefronts per CU (gemv_seg.hip).  The first window of stream s sits at byte s * stream_bytes of the payload buffer, the later ones
// behind all first windows, each found through its predecessor.  A stream covers a set of rows (chosen so that all
// streams weigh about the same) in tiles of at most kSegTileRows; inside a tile the blocks are ordered by format (in the
// order of `fmt`), inside a format by row and column.  Window: 2 dwords {8-byte units of records | 1 << 12 if another
// window follows | 16-byte pieces that window fills << 16, its byte offset / 16 in the buffer}; the records: per entry
// 2 dwords {slot | format << 4 | closes its tile << 8 | rows of the tile << 9 | blocks << 16, byte offset of the blocks |
// byte offset of their tags << 16}, and behind an entry that closes its tile 4 dwords with the tile's row numbers; the
// tags (per block: row of the tile and column block, in one byte (row << 6 | column) while a row has at most 64 blocks,
// else two (row << 12 | column)); the blocks, 16-byte aligned, whole.  `blind16` = 16-byte pieces the fullest first
// window fills.
// Most tensors of SPARK_Q0 and OIL1 blocks alone (api.hip says which) are stored as `sign_tiles` tiles of 16 rows instead (gemv_signs.hip): at the start 8 bytes per (block of the row, tile), all tiles of the row's first block first: {byte offset / 16 in the buffer, a
// bit per row that is SPARK_Q0 there}; then tile by tile, block of the row by block of the row, the up to 16 rows' blocks in the order of the rows, whole.
// `nstreams` is 0 then.
constexpr int kSegMaxFormats = 15;
constexpr uint32_t kSegWindow = 4096;
constexpr int kSegTileRows = 4;
struct SegLayout {
    uint32_t nf = 0, sign_tiles = 0, nstreams = 0, waves = 8, blind16 = 0, tag_bytes = 2;
    uint64_t stream_bytes = 0;
    bool by_descriptor() const { return nstreams || sign_tiles; }      // blocks are found through their descriptors
    uint32_t fmt[kSegMaxFormats] = {}, cb_bytes[kSegMaxFormats] = {}, idx_bytes[kSegMaxFormats] = {}, stride[kSegMaxFormats] = {};
};

}  // namespace oilhip

// The handle behind oilhip_weights*.
struct oilhip_weights {
    int device = 0;
    uint8_t* d_payload = nullptr;           // block payloads, each 16-byte aligned
    oilhip::DevBlock* d_blocks = nullptr;   // one descriptor per block
    oilhip::SegLayout seg;                  // mixed-format tensors of full blocks: tile- and format-ordered storage
    uint64_t* d_out_off = nullptr;          // first output index per block (only when nw varies)
    uint64_t alloc_bytes = 0;               // size of d_payload
    uint64_t payload_bytes = 0;             // sum of cb_bytes + idx_bytes
    uint64_t rows = 0, cols = 0;
    uint32_t nblocks = 0;
    int uniform_fmt = -1;                   // single format id, or -1
    uint32_t uniform_stride = 0;            // bytes between consecutive blocks when regular, else 0
    uint32_t uniform_cb = 0, uniform_idx = 0;   // channel sizes of every block when regular
    uint32_t uniform_base = 0;              // byte offset of block 0 when regular
    bool all_full = false;                  // every block holds exactly 256 weights
    bool nominal = false;                   // ... and has the channel sizes the quantizer writes for its format
};

namespace oilhip {
// Uniform OIL4 / OIL8 tensors in the plain layout the specialised kernels read: every block's bytes in the index
// channel, blocks back to back from byte 0.  Anything else (a non-empty codebook channel, padding between blocks)
// goes through the kernels that follow the descriptors.
inline bool plain_oil4(const oilhip_weights& w) {
    return w.uniform_fmt == OILHIP_OIL4 && w.uniform_stride == 128 && w.uniform_cb == 0 && w.uniform_idx == 128 && w.uniform_base == 0;
}
inline bool plain_oil8(const oilhip_weights& w) {
    return w.uniform_fmt == OILHIP_OIL8 && w.uniform_stride == 256 && w.uniform_cb == 0 && w.uniform_idx == 256 && w.uniform_base == 0;
}

// kernels (each returns an OILHIP_* code and sets the error text)
int launch_dequant(const oilhip_weights& w, float* d_out, hipStream_t s);
// operands of the prefill GEMM in fragment order (generic_kernels.hip)
int launch_dense_prepare(const oilhip_weights& w, uint32_t row0, uint32_t rows, uint16_t* wf, const void* x, bool x_is_f32, uint32_t M,
                         uint16_t* xf, uint32_t* arrived, uint32_t ncount, hipStream_t s);
bool dense_prepare_covers(const oilhip_weights& w);   // whether launch_dense_prepare takes this tensor's layout
int launch_gemv_generic(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s);
// fast paths return 1 when they do not cover the case (caller falls through to the general kernel)
int launch_gemv_oil4(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s);
// production gemv_oil4 form for one activation row: rows of K/2 code bytes, FP16 codebook of 16, one scale
int launch_gemv_flat4(const uint8_t* d_w, const uint16_t* d_cb16, float scale, const float* d_x, float* d_y, int rows, int K,
                      hipStream_t s);
int launch_gemv_oil8(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s);
// kernel::oil8_gemm form: rows of K index bytes, any 256-entry codebook; out[m*N + n] = scale * dot
int launch_gemv_flat8(const uint8_t* d_idx, const float* d_cb, const float* d_act, float* d_out, int M, int N, int K, float scale,
                      hipStream_t s);
// several activation rows at once (INT8 MFMA, gemv_oil4_multi.hip); x row tok[m] (or m) of an [xrows][ldx] matrix, y row
// stride ldy.  What a row is multiplied as: itself, silu(x) * x2, or x * (1 + norm_w) / rms(x)
struct MultiInput {
    const float* x2 = nullptr;      // same layout as x
    const float* norm_w = nullptr;  // cols floats
    bool inv_form = false;          // silu as x * (1 / (1 + exp(-x))) instead of x / (1 + exp(-x))
    float* xn = nullptr;            // with norm_w: receives the normalised rows, same layout as x, no overlap with it
};
int launch_gemv_oil4_multi(const oilhip_weights& w, const float* d_x, const int* d_tok, float* d_y, int M, uint32_t ldx, uint32_t ldy,
                           uint32_t xrows, hipStream_t s, const MultiInput& in = {}, const oilhip_weights* w2 = nullptr, float* d_y2 = nullptr,
                           uint32_t ldy2 = 0, uint8_t* d_pack = nullptr, size_t pack_room = 0);
// several batches of one tensor shape in one launch, at most 32 rows each; BatchSums: where parts of K may leave their sums
constexpr int kMaxBatchParts = 4;
struct BatchSums {
    int most, n;                                    // parts that may be used, and that were
    float* to[kMaxBatchParts - 1];                  // part p > 0: row i of all activation rows at to[p - 1] + i * ld[p - 1]
    uint32_t ld[kMaxBatchParts - 1];
};
size_t gemv_oil4_multi_batches_bytes(int nb, uint64_t cols);
int launch_gemv_oil4_multi_batches(int nb, const oilhip_weights* const* wa, float* const* ya, const oilhip_weights* const* wb, float* const* yb,
                                   const int* M, const int* row0, const int* list, int nlist, const float* d_x, const float* d_x2,
                                   uint32_t ldx, uint32_t xrows, uint32_t ldy, void* d_ws, size_t ws_bytes, hipStream_t s, BatchSums* sums = nullptr);
// other formats, up to 16 rows per pass (FP16 MFMA, gemv_any_multi.hip)
int launch_gemv_any_multi(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s, uint8_t* d_pack = nullptr,
                          const MultiInput& in = {}, uint32_t ldx = 0);
// bytes of d_pack that these two kernels need (0: they do not serve the tensor)
size_t gemv_oil4_multi_bytes(const oilhip_weights& w, int M);
size_t gemv_any_multi_bytes(const oilhip_weights& w, int M);
// oilhip_gemv_f32 after its checks; d_pack as in oilhip_gemv_f32_ws
int gemv_f32(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s, uint8_t* d_pack);
int check_workspace(const oilhip_weights& w, int M, const void* d_ws, size_t ws_bytes);
// widest row that these kernels take and the bytes of packed activations that any pass needs (d_pack, or stream scratch): per
// block 32 floats (powers of two) and four digits of 256 activations for 32 tokens, or 48 floats and 27 KB of FP16 pieces
constexpr uint32_t kGemvPackMaxCols = 32768;
constexpr size_t kGemvPackBytes = (size_t)(kGemvPackMaxCols >> 8) * (192u + 32768u);
// rows that mix formats, stored tile by tile and format by format
int launch_gemv_seg(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s);
// SPARK_Q0 and OIL1 blocks stored as sign tiles, kSignRows activation rows per launch
constexpr int kSignRows = 4;
bool signs_fastest(const oilhip_weights& w, int M);       // whether this kernel is faster than gemv_any_multi's
// Whether arrays of na and nb floats share memory.  Several rows whose outputs lie over something that workgroups read, or store besides, go through a kernel
// whose activations are packed by a launch of their own, before any output is stored, where there is one.
inline bool overlap(const float* a, uint64_t na, const float* b, uint64_t nb) {
    const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
    return a0 < b0 + 4u * nb && b0 < a0 + 4u * na;
}
int launch_gemv_signs(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s, const MultiInput& in = {}, uint32_t ldx = 0);
// every format, a lane per run of 32 weights
int launch_gemv_runs(const oilhip_weights& w, const float* d_x, float* d_y, int M, hipStream_t s);
// prefill: x is bf16 bit patterns, or FP32 (rounded once to bf16) when x_is_f32; any tensor of full blocks (gemm_dense.hip) ...
double dense_estimate_us(uint32_t M, uint32_t N, uint32_t K);
int launch_gemm_any(const oilhip_weights& w, const void* d_x, bool x_is_f32, float* d_y, int M, hipStream_t s);
// ... sign tiles, decoded inside the kernel (gemm_signs.hip) ...
int check_sign_parts(uint32_t bpr, uint32_t parts);       // a plan's parts of K, checked before its launch
int launch_gemm_signs(const oilhip_weights& w, const void* d_x, bool x_is_f32, float* d_y, int M, hipStream_t s);
// ... and plain uniform OIL4, decoded inside the kernel (gemm_oil4_frag.hip)
int launch_gemm_oil4_frag(const oilhip_weights& w, const void* d_x, bool x_is_f32, float* d_y, int M, hipStream_t s);
}  // namespace oilhip
