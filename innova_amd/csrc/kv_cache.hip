// kv_cache.hip -- the OIL4 KV cache of the reference (oil::OIL4KVCache, include/oil/kv_cache_oil4.h:26-83,
// src/kv_cache_oil4.cpp) held in HBM: 4-bit codes, two per byte (low nibble first), and 16 FP16 centroids per block of
// 32 / 64 / 128 consecutive values of a layer's [token][heads * dim] stream.
//
//   append    : every chunk (a token's values cut at block boundaries, :207-291) is quantized by 16 lanes, one per
//               cluster, with the reference's 16-level Lloyd-Max (:75-153) step for step -- same initial centroids, same 20
//               iterations over the sorted values, same sequential sums -- so codes and centroids are identical.
//   get_range : codes -> centroids -> FP32 [len][heads * dim] through the cache's own half decode
//               (CodebookOIL4::half_to_float, src/codebook.cpp:36-64, which is not IEEE for subnormals).
//
// A chunk's codes are packed from its own first byte, block * (block / 2) + offset / 2 (:246).  With an even number
// of values per token that makes element e of a layer nibble e & 1 of byte e / 2.  With an odd number a chunk that
// starts at an even offset and holds an odd count shares its last byte with the chunk behind it, and the later write
// wins (the earlier chunk's last code is lost, as in the reference); the kernels reproduce that by leaving the shared
// byte to the later chunk.
#include <algorithm>
#include <new>
#include <type_traits>
#include <vector>

#include "common.h"

struct oilhip_kv {
    int device = 0;
    int layers = 0;
    int64_t max_seq = 0, heads = 0, dim = 0, block = 64, per_token = 0;
    int64_t idx_bytes = 0;          // per layer and side, (max_seq * per_token + 1) / 2
    int64_t nblocks = 0;            // per layer and side
    int64_t idx_stride = 0;         // idx_bytes rounded up to 256
    uint8_t* d_idx = nullptr;       // [layers][2 (K, V)][idx_stride]
    uint16_t* d_cb = nullptr;       // [layers][2][nblocks * 16]
    std::vector<int64_t> pos;       // tokens appended per layer (the reference's current_pos: counts dropped tokens too)
};

namespace oilhip {
namespace {

// CodebookOIL4::float_to_half (src/codebook.cpp:16-34): the mantissa is truncated, magnitudes below 2^-25 become zero.
__device__ __forceinline__ uint32_t kv_float_to_half(float f) {
    const uint32_t u = __float_as_uint(f);
    const uint32_t sign = (u >> 16) & 0x8000u;
    const int e = (int)((u >> 23) & 0xFFu) - 112;
    uint32_t mant = u & 0x007FFFFFu;
    if (e <= 0) {
        if (e < -10) return sign;
        mant = (mant | 0x00800000u) >> (1 - e);
        return sign | (mant >> 13);
    }
    if (e >= 31) return sign | 0x7C00u | (mant ? 0x0200u : 0u);
    return sign | ((uint32_t)e << 10) | (mant >> 13);
}

// CodebookOIL4::half_to_float (src/codebook.cpp:36-64).  A subnormal half whose highest set mantissa bit is p gets the
// exponent field 113 - p, and of its normalised mantissa << 13 only the low 16 bits (the reference holds it in a
// uint16_t, :52).
__device__ __forceinline__ float kv_half_to_float(uint32_t h) {
    const uint32_t sign = (h & 0x8000u) << 16;
    const uint32_t e = (h >> 10) & 0x1Fu;
    const uint32_t mant = h & 0x03FFu;
    uint32_t f;
    if (e == 0) {
        if (mant == 0) {
            f = sign;
        } else {
            const uint32_t p = 31u - (uint32_t)__clz((int)mant);
            f = sign | ((113u - p) << 23) | ((((mant << (10u - p)) & 0x03FFu) << 13) & 0xFFFFu);
        }
    } else if (e == 31) {
        f = sign | 0x7F800000u | (mant << 13);
    } else {
        f = sign | ((e + 112u) << 23) | (mant << 13);
    }
    return __uint_as_float(f);
}

// the first of the nearest centroids (a loop over LDS: this path is for rare chunks and should cost the common one no registers)
__device__ __forceinline__ uint32_t kv_nearest(const float* cen, float x) {
    float best = fabsf(__fsub_rn(x, cen[0]));
    uint32_t bi = 0;
#pragma unroll 1
    for (uint32_t c = 1; c < 16; ++c) {
        const float d = fabsf(__fsub_rn(x, cen[c]));
        if (d < best) { best = d; bi = c; }
    }
    return bi;
}

struct KvLds {
    float srt[128];
    float cen[16];
    uint8_t code[128];
};

// Minimum (the first of equal values: the sign of a zero minimum reaches a constant chunk's centroids) and maximum of
// the chunk, in every lane.
__device__ __forceinline__ void kv_min_max(float x0, float x1, uint32_t n, uint32_t lane, float& lo, float& hi) {
    lo = lane < n ? x0 : __builtin_inff();
    uint32_t lo_i = lane;
    if (lane + 64 < n && x1 < lo) { lo = x1; lo_i = lane + 64; }
    hi = lane < n ? x0 : -__builtin_inff();
    if (lane + 64 < n && x1 > hi) hi = x1;
    for (int o = 32; o > 0; o >>= 1) {
        const float ol = __shfl_xor(lo, o, 64);
        const uint32_t oi = (uint32_t)__shfl_xor((int)lo_i, o, 64);
        if (ol < lo || (ol == lo && oi < lo_i)) { lo = ol; lo_i = oi; }
        const float oh = __shfl_xor(hi, o, 64);
        if (oh > hi) hi = oh;
    }
}

// lloyd_max_16 (src/kv_cache_oil4.cpp:75-153) for n <= 128 values by one wavefront, for any values.  Leaves the n codes in L.code and
// the 16 centroids (FP32) in L.cen.
__device__ __forceinline__ void kv_quantize_chunk(const float* __restrict__ src, uint32_t n, uint32_t lane, KvLds& L) {
    const float x0 = lane < n ? src[lane] : 0.f;
    const float x1 = lane + 64 < n ? src[lane + 64] : 0.f;
    float lo, hi;
    kv_min_max(x0, x1, n, lane, lo, hi);
    const float range = __fsub_rn(hi, lo);
    if (range < 1e-10f) {
        if (lane < n) L.code[lane] = 8;
        if (lane + 64 < n) L.code[lane + 64] = 8;
        if (lane < 16) L.cen[lane] = lo;
        __syncthreads();
        return;
    }
    if (lane < 16) L.cen[lane] = __fadd_rn(lo, __fdiv_rn(__fmul_rn(range, (float)lane + 0.5f), 16.0f));
    // ascending bitonic sort over 128 slots, +inf behind the values
    L.srt[lane] = lane < n ? x0 : __builtin_inff();
    L.srt[lane + 64] = lane + 64 < n ? x1 : __builtin_inff();
    __syncthreads();
    for (uint32_t k = 2; k <= 128; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            const uint32_t i = ((lane & ~(j - 1)) << 1) | (lane & (j - 1));
            const uint32_t p = i | j;
            const bool up = (i & k) == 0;
            const float a = L.srt[i], b = L.srt[p];
            if ((a > b) == up) { L.srt[i] = b; L.srt[p] = a; }
            __syncthreads();
        }
    }
    for (int it = 0; it < 20; ++it) {
        // lane c < 16 collects the members of cluster c as bit masks over the sorted order and adds them up in that
        // order, as the reference's loop over the sorted values does
        const uint32_t b0 = lane < n ? kv_nearest(L.cen, L.srt[lane]) : 16u;
        const uint32_t b1 = lane + 64 < n ? kv_nearest(L.cen, L.srt[lane + 64]) : 16u;
        uint64_t m0 = 0, m1 = 0;
#pragma unroll 1
        for (uint32_t c = 0; c < 16; ++c) {
            const uint64_t w0 = __ballot(b0 == c), w1 = __ballot(b1 == c);
            if (lane == c) { m0 = w0; m1 = w1; }
        }
        float sum = 0.f;
        const int cnt = __popcll(m0) + __popcll(m1);
        for (; m0; m0 &= m0 - 1) sum = __fadd_rn(sum, L.srt[__builtin_ctzll(m0)]);
        for (; m1; m1 &= m1 - 1) sum = __fadd_rn(sum, L.srt[64 + __builtin_ctzll(m1)]);
        bool moved = false;
        if (lane < 16 && cnt > 0) {                                                  // an empty cluster keeps its centroid
            const float nv = __fdiv_rn(sum, (float)cnt);
            moved = __float_as_uint(nv) != __float_as_uint(L.cen[lane]);
            L.cen[lane] = nv;
        }
        __syncthreads();
        if (__ballot(moved) == 0) break;     // a fixed point: the remaining iterations would reproduce these centroids bit for bit
    }
    if (lane < n) L.code[lane] = (uint8_t)kv_nearest(L.cen, x0);
    if (lane + 64 < n) L.code[lane + 64] = (uint8_t)kv_nearest(L.cen, x1);
    __syncthreads();
}

// ---- the same quantizer, 16 lanes per chunk ----------------------------------------------------------------------------
// A wavefront takes up to four chunks of at most 16 V values, one per row of 16 lanes; lane c of a row holds values c V ..
// c V + V - 1 and is cluster c.  The values are sorted across the row in registers and kept in LDS.  Sorted values
// that belong to one cluster are neighbours, so an iteration is: every cluster moves its first member's position (from where it
// was) until |x - cen[c]| < |x - cen[c - 1]| holds at it and not before it, and adds its members up in sorted order, as the
// reference's loop does.  A cluster whose range stays has the same sum as before, and when all ranges stay the centroids are a fixed
// point.
// That the comparison of neighbours is monotone over the sorted values and equals the reference's scan over all 16 needs
// centroids that are finite and rise by more than the rounding of the distances (at most range * 2^-22); this is checked in every
// iteration, and chunks that fail it (large values: a cluster's sum overflows although its members are finite), hold infinities or
// NaN, or are constant, go through kv_quantize_chunk.
// What bounds it: vector issue of the iterations (about 60 instructions for four chunks each, of which a long append takes about a
// dozen); the chain of dependent instructions and LDS round trips when a decode step appends one token, where each wavefront
// takes one chunk.  One wavefront per chunk before (every value compared with all 16 centroids in each iteration, sums passed
// from lane to lane) -> now, 4096 values per token, K and V: 2048 tokens 490 -> 93 us with blocks of 64, 1024 tokens of 2048
// values with blocks of 32 300 -> 37 us and of 128 268 -> 40 us (clearing included), one token 13 -> 6 us.
// Sorting floats instead of keys, tokens of whole blocks without index arithmetic, and sums by lane masks (BUSY) -> kernel alone, 2048 tokens of 4096
// values 85 -> 72 us, 1024 tokens of 2048 values with blocks of 32 29.5 -> 23.6 us and of 128 33.4 -> 32.4 us, one token of 4096 7.0 -> 6.6 us.
// Windows of four positions per move and sums of eight values per round need fewer steps, and were slower by 12 %.
constexpr int kSrtPad = 8;                 // floats before a row's values

template <int CTRL>
__device__ __forceinline__ int row_dpp(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true); }

template <int CTRL>
__device__ __forceinline__ float row_dpp(float v) { return __int_as_float(row_dpp<CTRL>(__float_as_int(v))); }

// Finite values and +inf (a chunk with a NaN or an infinity in it takes the other path, whatever becomes of it here).  A zero may
// change its sign where zeros of both signs meet: no sum, distance or comparison notices.
__device__ __forceinline__ float lesser(float a, float b) { float r; asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b)); return r; }
__device__ __forceinline__ float greater(float a, float b) { float r; asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b)); return r; }

template <int V>
__device__ __forceinline__ void in_lane_merge(float (&k)[V]) {
#pragma unroll
    for (int j = V / 2; j > 0; j >>= 1)
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (!(e & j)) { const float a = k[e], b = k[e | j]; k[e] = lesser(a, b); k[e | j] = greater(a, b); }
}

// Ascending bitonic sort of 16 V values, element c V + e in lane c.  A merge begins with the mirrored partner, so that all
// comparisons point the same way; `bound[i]` is -inf in lanes whose bit i is clear (they keep the smaller value), else +inf.
template <int V>
__device__ __forceinline__ void row_sort(float (&k)[V], uint32_t c) {
    auto med3 = [](float a, float b, float m) { return __builtin_amdgcn_fmed3f(a, b, m); };
    float bound[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) bound[i] = (c >> i) & 1u ? __builtin_inff() : -__builtin_inff();
    // inside a lane
#pragma unroll
    for (int m = 2; m <= V; m <<= 1) {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const int o = e ^ (m - 1);
            if (e < o) { const float a = k[e], b = k[o]; k[e] = lesser(a, b); k[o] = greater(a, b); }
        }
#pragma unroll
        for (int j = m / 4; j > 0; j >>= 1)
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (!(e & j)) { const float a = k[e], b = k[e | j]; k[e] = lesser(a, b); k[e | j] = greater(a, b); }
    }
    auto flip = [&](auto ctrl, int bit) {
        float o[V];
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = row_dpp<decltype(ctrl)::value>(k[V - 1 - e]);
#pragma unroll
        for (int e = 0; e < V; ++e) k[e] = med3(k[e], o[e], bound[bit]);
    };
    auto step = [&](auto ctrl, int bit) {
#pragma unroll
        for (int e = 0; e < V; ++e) k[e] = med3(k[e], row_dpp<decltype(ctrl)::value>(k[e]), bound[bit]);
    };
    using std::integral_constant;
    flip(integral_constant<int, 0xB1>{}, 0);                               // lane ^ 1
    in_lane_merge<V>(k);
    flip(integral_constant<int, 0x1B>{}, 1);                               // ^ 3
    step(integral_constant<int, 0xB1>{}, 0);
    in_lane_merge<V>(k);
    flip(integral_constant<int, 0x141>{}, 2);                              // ^ 7
    step(integral_constant<int, 0x4E>{}, 1);                               // ^ 2
    step(integral_constant<int, 0xB1>{}, 0);
    in_lane_merge<V>(k);
    flip(integral_constant<int, 0x140>{}, 3);                              // ^ 15
#pragma unroll
    for (int e = 0; e < V; ++e) k[e] = med3(k[e], row_dpp<0x141>(row_dpp<0x1B>(k[e])), bound[2]);   // ^ 4
    step(integral_constant<int, 0x4E>{}, 1);
    step(integral_constant<int, 0xB1>{}, 0);
    in_lane_merge<V>(k);
}

// sum / count, correctly rounded, for a count of at most 128: sum * (1 / count) in two floats has an error of about 2^-46 of it, and a
// quotient with so small a divisor is never closer than 2^-32 to the middle between two floats.
__device__ __forceinline__ float kv_mean(float sum, float count) {
#pragma clang fp contract(off)
    const float r = __builtin_amdgcn_rcpf(count), r2 = __builtin_fmaf(-count, r, 1.0f) * r;
    const float q = sum * r;
    float d = q + __builtin_fmaf(sum, r2, __builtin_fmaf(sum, r, -q));
    const bool tiny = fabsf(sum) < 0x1p-90f;                               // the remainders may not be floats
    if (__ballot(tiny)) {
        asm volatile("" : "+v"(sum));                                      // keeps the division inside the branch
        d = tiny ? __fdiv_rn(sum, count) : d;
    }
    return d;
}

// `n` values (x[e] = value c V + e of the row's chunk; anything past n).  Returns false where the chunk has to take the other path;
// n = 0: nothing to do.  Uniform over a row of lanes; all 64 lanes take part.  srt: room for kSrtPad + 32 V floats, from
// -kSrtPad on.
// BUSY: with wavefronts enough to wait for each other a member costs one vector instruction and a comparison for all lanes, instead of a comparison,
// a selection and an addition of zero; a wavefront by itself waits longer for that.
template <int V, bool BUSY>
__device__ __forceinline__ bool kv_lloyd_rows(const float (&x)[V], uint32_t n, uint32_t lane, float* srt, uint32_t (&code)[V], float& cen_out) {
    const uint32_t c = lane & 15u;
    const int nan = 0x7FC00000;
    float k[V];
    bool finite = true;
#pragma unroll
    for (int e = 0; e < V; ++e) {
        const bool in = c * V + (uint32_t)e < n;
        finite &= !in || fabsf(x[e]) < __builtin_inff();
        k[e] = in ? x[e] : __builtin_inff();                               // +infinity behind the values
    }
    row_sort<V>(k, c);
#pragma unroll
    for (int e = 0; e < V; ++e) srt[c * V + (uint32_t)e] = k[e];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const float lo = srt[0], hi = srt[n ? n - 1u : 0u];
    const float range = __fsub_rn(hi, lo);
    bool ok = range >= 1e-10f && range < __builtin_inff();
    ok &= ((__ballot(!finite) >> (lane & 48u)) & 0xFFFFull) == 0;
    float cen = __fadd_rn(lo, __fdiv_rn(__fmul_rn(range, (float)c + 0.5f), 16.0f));
    ok &= ((__ballot(!(fabsf(cen) < __builtin_inff())) >> (lane & 48u)) & 0xFFFFull) == 0;
    const float least_gap = range * 0x1p-20f;
    // NaN before the first value and behind the last one: no comparison holds there.  Likewise the centroid before the first one, and
    // all centroids of a row that takes the other path: its boundaries stay where they are.
    if (c < 2u) srt[c ? (int)n : -1] = __int_as_float(nan);
    cen = ok ? cen : __int_as_float(nan);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    auto lane_below = [&](float v) { return __int_as_float(__builtin_amdgcn_update_dpp(nan, __float_as_int(v), 0x111, 0xF, 0xF, false)); };
    float below = lane_below(cen);
    // p: the first sorted value of this cluster, the end of the one before
    uint32_t p = 0;
#pragma unroll
    for (uint32_t h = 8u * V; h > 0; h >>= 1) {
        const float v = srt[p + h - 1u];
        p += ((p + h <= n) & (fabsf(__fsub_rn(v, below)) <= fabsf(__fsub_rn(v, cen)))) ? h : 0u;
    }
    uint32_t p_was = 0xFFFFFFFFu, end = 0, end_was = 0;
    for (int it = 0;; ++it) {
        for (int moves = 0; moves <= 16 * V; ++moves) {                    // towards the boundary; a direction never turns
            const float left = srt[(int)p - 1], right = srt[p];
            const bool up = fabsf(__fsub_rn(right, below)) <= fabsf(__fsub_rn(right, cen));
            const bool down = fabsf(__fsub_rn(left, cen)) < fabsf(__fsub_rn(left, below));
            p += up ? 1u : down ? 0xFFFFFFFFu : 0u;
            if ((__ballot(up) | __ballot(down)) == 0) break;
        }
        end = (uint32_t)__builtin_amdgcn_update_dpp((int)n, (int)p, 0x101, 0xF, 0xF, false);   // p of cluster c + 1
        const bool changed = (p != p_was) | (end != end_was);
        if (it == 20 || __ballot(changed) == 0) break;
        const int cnt = changed ? (int)(end - p) : 0;                      // an empty cluster keeps its centroid
        float sum = 0.f;
        const float* at = srt + p;                                         // up to 16 V + 16 V floats on, in lanes that are done
        int left = cnt;
        do {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = at[u];
            if constexpr (BUSY) {                                          // lanes drop out as their members end
                const uint64_t first = __ballot(left > 0), second = __ballot(left > 1), third = __ballot(left > 2), fourth = __ballot(left > 3);
                uint64_t all;
                asm volatile("s_mov_b64 %1, exec\n\ts_mov_b64 exec, %6\n\tv_add_f32_e32 %0, %0, %2\n\ts_mov_b64 exec, %7\n\tv_add_f32_e32 %0, %0, %3\n\t"
                             "s_mov_b64 exec, %8\n\tv_add_f32_e32 %0, %0, %4\n\ts_mov_b64 exec, %9\n\tv_add_f32_e32 %0, %0, %5\n\ts_mov_b64 exec, %1"
                             : "+v"(sum), "=&s"(all) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "s"(first), "s"(second), "s"(third), "s"(fourth));
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) sum = __fadd_rn(sum, left > u ? v[u] : 0.f);   // sum is never -0: + 0 changes nothing
            }
            at += 4;
            left -= 4;
        } while (__ballot(left > 0));
        const float mean = kv_mean(cnt > 0 ? sum : 1.0f, (float)(cnt > 0 ? cnt : 1));
        cen = cnt > 0 ? mean : cen;
        below = lane_below(cen);
        const bool tight = __fsub_rn(cen, below) <= least_gap;             // false for the first one
        ok &= !tight & (fabsf(cen) < __builtin_inff());                    // of an infinite sum kv_mean makes NaN
        p_was = p;
        end_was = end;
    }
    ok = ((__ballot(!ok) >> (lane & 48u)) & 0xFFFFull) == 0;
    // a value's cluster is the last one whose first member is not larger
    const float first = p < n ? srt[p] : __builtin_inff();
#pragma unroll
    for (int e = 0; e < V; ++e) {
        uint32_t q = 0;
#pragma unroll
        for (uint32_t h = 8; h > 0; h >>= 1) {
            const float t = __int_as_float(__builtin_amdgcn_ds_bpermute((int)(4u * ((lane & 48u) + q + h)), __float_as_int(first)));
            q = x[e] >= t ? q + h : q;
        }
        code[e] = q;
    }
    cen_out = cen;
    return ok || n == 0;
}

// Up to four chunks of a wavefront: chunk(g, src, n) says where row g's chunk is (n = 0: none).  Leaves the codes of values c V + e in
// code[e] and centroid c in cen.
template <int V>
struct KvRows {
    float srt[4 * (16 * V + kSrtPad) + 16 * V];
    KvLds slow;
};
// WHOLE: all chunks have 16 V values and begin at a multiple of their loads' size.
template <int V, bool BUSY, bool WHOLE>
__device__ __forceinline__ void kv_quantize_rows(const float* src, uint32_t n, uint32_t lane, KvRows<V>& L, uint32_t (&code)[V], float& cen) {
    const uint32_t c = lane & 15u;
    float x[V];
    if (WHOLE) n = 16u * V;
    if (WHOLE || (n == 16u * V && (reinterpret_cast<uintptr_t>(src) & (V == 2 ? 7u : 15u)) == 0)) {
        if constexpr (V == 2) {
            const float2 f = reinterpret_cast<const float2*>(src)[c];
            x[0] = f.x; x[1] = f.y;
        } else {
#pragma unroll
            for (int h = 0; h < V / 4; ++h) {
                const float4 f = reinterpret_cast<const float4*>(src)[c * (V / 4) + (uint32_t)h];
                x[4 * h] = f.x; x[4 * h + 1] = f.y; x[4 * h + 2] = f.z; x[4 * h + 3] = f.w;
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < V; ++e) x[e] = c * V + (uint32_t)e < n ? src[c * V + (uint32_t)e] : 0.f;
    }
    const bool ok = kv_lloyd_rows<V, BUSY>(x, n, lane, L.srt + (lane >> 4) * (16 * V + kSrtPad) + kSrtPad, code, cen);
    uint64_t left = __ballot(!ok);
    while (left) {                                                         // chunk by chunk, by all 64 lanes
        const uint32_t at = (uint32_t)__builtin_ctzll(left);
        left &= ~(0xFFFFull << (at & 48u));
        const uint64_t p = reinterpret_cast<uint64_t>(src);
        const uint64_t q = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)p, (int)at) |
                           (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(p >> 32), (int)at) << 32;
        kv_quantize_chunk(reinterpret_cast<const float*>(q), (uint32_t)__builtin_amdgcn_readlane((int)n, (int)at), lane, L.slow);
        if ((lane & 48u) == (at & 48u)) {
#pragma unroll
            for (int e = 0; e < V; ++e) code[e] = L.slow.code[(c * V + (uint32_t)e) & 127u];
            cen = L.slow.cen[c];
        }
        __syncthreads();
    }
}

// One row of 16 lanes per (token, chunk of the token, K or V), `per_wave` rows of a wavefront in use.  pos = tokens the layer
// held before this call, ntok = tokens of this call that fit.  K centroids are stored by the chunk that opens a block, or -- while the layer is empty, and
// for V always -- by the last chunk of the call that touches the block (:256-261, :277-279: later writes win).
template <int V, bool BUSY>
__global__ void __launch_bounds__(64)
kv_append_kernel(uint8_t* __restrict__ k_idx, uint8_t* __restrict__ v_idx, uint16_t* __restrict__ k_cb,
                 uint16_t* __restrict__ v_cb, const float* __restrict__ k, const float* __restrict__ v, int64_t pos,
                 int64_t ntok, int64_t per_token, uint32_t chunks_per_token, uint32_t items, uint32_t per_wave, int64_t idx_bytes) {
    __shared__ KvRows<V> L;
    constexpr int64_t block = 16 * V;
    const uint32_t lane = threadIdx.x, row = lane >> 4, c = lane & 15u;
    const bool is_v = blockIdx.y != 0;
    const uint32_t item = blockIdx.x * per_wave + row;
    const bool in = row < per_wave && item < items;
    const int64_t s = in ? item / chunks_per_token : 0;
    const uint32_t ch = in ? item % chunks_per_token : 0u;
    const int64_t tok_lo = (pos + s) * per_token, tok_hi = tok_lo + per_token;
    const int64_t blk = tok_lo / block + ch;
    const int64_t a = ch == 0 ? tok_lo : blk * block;
    const int64_t b = (blk + 1) * block < tok_hi ? (blk + 1) * block : tok_hi;
    const uint32_t n = in && a < tok_hi ? (uint32_t)(b - a) : 0u;
    const float* src = (is_v ? v : k) + (n ? a - pos * per_token : 0);
    uint32_t code[V];
    float cen;
    kv_quantize_rows<V, BUSY, false>(src, n, lane, L, code, cen);
    if (n == 0) return;
    const bool last_on_block = (b & (block - 1)) == 0 || b == (pos + ntok) * per_token;
    const uint32_t off = (uint32_t)(a & (block - 1));
    const int64_t at = blk * (block >> 1) + (off >> 1);
    uint32_t nbytes = (n + 1) >> 1;
    if (!(off & 1u) && (n & 1u) && !last_on_block) --nbytes;        // that byte belongs to the next chunk of this call
    if (at + nbytes > idx_bytes) nbytes = at < idx_bytes ? (uint32_t)(idx_bytes - at) : 0u;   // :248-249
    uint8_t* idx = (is_v ? v_idx : k_idx) + at;
    uint32_t bytes = 0;
#pragma unroll
    for (int e = 0; e < V; ++e) bytes |= (c * V + (uint32_t)e < n ? code[e] : 0u) << (4 * e);
    if (nbytes == (uint32_t)block / 2u) {                            // whole block: aligned
        if constexpr (V == 2) idx[c] = (uint8_t)bytes;
        if constexpr (V == 4) reinterpret_cast<uint16_t*>(idx)[c] = (uint16_t)bytes;
        if constexpr (V == 8) reinterpret_cast<uint32_t*>(idx)[c] = bytes;
    } else {
#pragma unroll
        for (int i = 0; i < V / 2; ++i)
            if (c * (V / 2) + (uint32_t)i < nbytes) idx[c * (V / 2) + (uint32_t)i] = (uint8_t)(bytes >> (8 * i));
    }
    const bool store_cb = (is_v || pos == 0) ? last_on_block : off == 0;
    if (store_cb) (is_v ? v_cb : k_cb)[blk * 16 + c] = (uint16_t)kv_float_to_half(cen);
}

// The same where a token is whole blocks and the inputs are aligned: the call's chunks lie one behind the other, in memory and in the cache, and
// every one writes its block's codes and centroids.  Rows without a chunk repeat the last one.
template <int V, bool BUSY>
__global__ void __launch_bounds__(64)
kv_append_whole_kernel(uint8_t* __restrict__ k_idx, uint8_t* __restrict__ v_idx, uint16_t* __restrict__ k_cb, uint16_t* __restrict__ v_cb,
                       const float* __restrict__ k, const float* __restrict__ v, int64_t first_block, uint32_t items, uint32_t per_wave) {
    __shared__ KvRows<V> L;
    const uint32_t lane = threadIdx.x, row = lane >> 4, c = lane & 15u;
    const bool is_v = blockIdx.y != 0;
    const uint32_t item = min(blockIdx.x * per_wave + row, items - 1u);
    uint32_t code[V];
    float cen;
    kv_quantize_rows<V, BUSY, true>((is_v ? v : k) + (size_t)item * (16u * V), 16u * V, lane, L, code, cen);
    if (row >= per_wave || blockIdx.x * per_wave + row >= items) return;
    const size_t blk = (size_t)first_block + item;
    uint8_t* idx = (is_v ? v_idx : k_idx) + blk * (8u * V);
    uint32_t bytes = code[0];
#pragma unroll
    for (int e = 1; e < V; ++e) bytes |= code[e] << (4 * e);
    if constexpr (V == 2) idx[c] = (uint8_t)bytes;
    if constexpr (V == 4) reinterpret_cast<uint16_t*>(idx)[c] = (uint16_t)bytes;
    if constexpr (V == 8) reinterpret_cast<uint32_t*>(idx)[c] = bytes;
    (is_v ? v_cb : k_cb)[blk * 16 + c] = (uint16_t)kv_float_to_half(cen);
}

// OIL4KVCache::quantize_block_oil4 over nblocks independent runs of n <= 16 V values: one code per byte, 16 centroids.
template <int V>
__global__ void __launch_bounds__(64)
kv_quantize_blocks_kernel(const float* __restrict__ src, uint32_t n, uint32_t nblocks, uint32_t per_wave, uint8_t* __restrict__ codes,
                          uint16_t* __restrict__ cb) {
    __shared__ KvRows<V> L;
    const uint32_t lane = threadIdx.x, row = lane >> 4, c = lane & 15u;
    const uint32_t item = blockIdx.x * per_wave + row;
    const bool in = row < per_wave && item < nblocks;
    const size_t at = in ? (size_t)item * n : 0;
    uint32_t code[V];
    float cen;
    kv_quantize_rows<V, false, false>(src + at, in ? n : 0u, lane, L, code, cen);
    if (!in) return;
#pragma unroll
    for (int e = 0; e < V; ++e)
        if (c * V + (uint32_t)e < n) codes[at + c * V + (uint32_t)e] = (uint8_t)code[e];
    cb[(size_t)item * 16 + c] = (uint16_t)kv_float_to_half(cen);
}

// Chunks per wavefront: four fill its lanes; with fewer chunks than keep two wavefronts on every SIMD, one each, so that a chunk waits
// for its own iterations only.
uint32_t kv_per_wave(uint64_t chunks) { return chunks >= 8ull * (uint64_t)device_cu_count() ? 4u : 1u; }

// Eight wavefronts for every SIMD (that many: 16 x 128 values, blocks of 128, 1024 tokens 32.9 -> 32.4 us with masks; two for every SIMD, 400 values,
// blocks of 64, 500 tokens 9.8 -> 10.3; one token of 4096 6.6 -> 7.0).
bool kv_busy(uint64_t wavefronts) { return wavefronts >= 32ull * (uint64_t)device_cu_count(); }

// dequantize_block_oil4 (:155-161): dst[b][i] = half_to_float(cb[b][codes[b][i] & 15])
__global__ void __launch_bounds__(256)
kv_dequantize_blocks_kernel(const uint8_t* __restrict__ codes, const uint16_t* __restrict__ cb, float* __restrict__ dst,
                            uint32_t n, uint64_t total) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    dst[i] = kv_half_to_float(cb[(i / n) * 16 + (codes[i] & 15u)]);
}

// get_range for tokens whose value count is a multiple of 4 (value e is then nibble e & 1 of byte e / 2).  A workgroup decodes kTile consecutive elements of K
// (blockIdx.y = 0) or V (1): the centroids of the blocks under the tile go to LDS as FP32 once, then each thread
// turns 2 bytes of codes into one 16-byte store, four times.  Bound by the stores, which bypass the caches: 2056 tokens of
// 4096 (67 MB out) take 13.9 us, with ordinary stores 16.9.
constexpr uint32_t kTile = 4096;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(256)
kv_get_range_kernel(const uint8_t* __restrict__ k_idx, const uint8_t* __restrict__ v_idx, const uint16_t* __restrict__ k_cb,
                    const uint16_t* __restrict__ v_cb, float* __restrict__ k_out, float* __restrict__ v_out, uint64_t first,
                    uint64_t count, uint32_t block_shift, uint64_t ncb) {
    __shared__ float cen[(kTile / 32 + 1) * 16];
    const uint8_t* idx = blockIdx.y ? v_idx : k_idx;
    const uint16_t* cb = blockIdx.y ? v_cb : k_cb;
    float* out = blockIdx.y ? v_out : k_out;
    const uint64_t j0 = (uint64_t)blockIdx.x * kTile;
    const uint64_t jn = count - j0 < kTile ? count - j0 : kTile;
    const uint64_t blk0 = (first + j0) >> block_shift;
    const uint32_t nent = (uint32_t)((((first + j0 + jn - 1) >> block_shift) - blk0 + 1) * 16);
    for (uint32_t i = threadIdx.x; i < nent; i += 256) {
        const uint64_t at = blk0 * 16 + i;
        cen[i] = at < ncb ? kv_half_to_float(cb[at]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t it = 0; it < kTile / 1024; ++it) {
        const uint64_t j = (uint64_t)it * 1024 + threadIdx.x * 4;
        if (j < jn) {
            const uint64_t e = first + j0 + j;
            const uint32_t codes = *reinterpret_cast<const uint16_t*>(idx + (e >> 1));
            const float* t = cen + (uint32_t)((e >> block_shift) - blk0) * 16;
            f32x4 o;
            o.x = t[codes & 15u]; o.y = t[(codes >> 4) & 15u]; o.z = t[(codes >> 8) & 15u]; o.w = t[(codes >> 12) & 15u];
            __builtin_nontemporal_store(o, reinterpret_cast<f32x4*>(out + j0 + j));
        }
    }
}

// get_range, one value per thread, with the reference's chunk arithmetic (:318-334): the chunk of a value starts at
// the later of its token's first value and its block's first value, and its codes count from the chunk's own byte.
__global__ void __launch_bounds__(256)
kv_get_range_scalar_kernel(const uint8_t* __restrict__ k_idx, const uint8_t* __restrict__ v_idx,
                           const uint16_t* __restrict__ k_cb, const uint16_t* __restrict__ v_cb, float* __restrict__ k_out,
                           float* __restrict__ v_out, uint64_t first, uint64_t count, uint32_t block_shift, uint64_t per_token,
                           uint64_t idx_bytes) {
    const uint64_t j = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= count) return;
    const uint64_t e = first + j;
    const uint64_t blk = e >> block_shift;
    const uint64_t tok_lo = e / per_token * per_token, blk_lo = blk << block_shift;
    const uint64_t a = tok_lo > blk_lo ? tok_lo : blk_lo;
    const uint64_t at = (blk << (block_shift - 1)) + ((a - blk_lo) >> 1) + ((e - a) >> 1);
    const uint8_t* idx = blockIdx.y ? v_idx : k_idx;
    const uint16_t* cb = blockIdx.y ? v_cb : k_cb;
    const uint32_t byte = at < idx_bytes ? idx[at] : 0u;                              // :322-325
    const uint32_t code = (byte >> (4 * (uint32_t)((e - a) & 1))) & 15u;
    (blockIdx.y ? v_out : k_out)[j] = kv_half_to_float(cb[blk * 16 + code]);
}

// codes and centroids in one launch
__global__ void __launch_bounds__(256) kv_zero_kernel(uint4* p, uint64_t np, uint4* q, uint64_t nq) {
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < np + nq; i += (uint64_t)gridDim.x * 256)
        __builtin_nontemporal_store(u32x4{0, 0, 0, 0}, reinterpret_cast<u32x4*>((i < np ? p : q - np) + i));
}

int kv_alloc(oilhip_kv* c) {
    const int64_t total = c->max_seq * c->per_token;
    c->idx_bytes = (total + 1) / 2;
    c->nblocks = (total + c->block - 1) / c->block;
    c->idx_stride = (c->idx_bytes + 255) / 256 * 256;
    const size_t ib = (size_t)c->layers * 2 * (size_t)c->idx_stride;
    const size_t cbb = (size_t)c->layers * 2 * (size_t)c->nblocks * 32;
    c->d_idx = nullptr;
    c->d_cb = nullptr;
    if (ib == 0) return OILHIP_OK;
    if (hipMalloc((void**)&c->d_idx, ib) != hipSuccess) return fail(OILHIP_E_NOMEM, "kv cache: hipMalloc of the code arrays failed");
    if (hipMalloc((void**)&c->d_cb, cbb) != hipSuccess) {
        (void)hipFree(c->d_idx);
        c->d_idx = nullptr;
        return fail(OILHIP_E_NOMEM, "kv cache: hipMalloc of the centroid arrays failed");
    }
    OILHIP_HIP(hipMemset(c->d_idx, 0, ib));
    OILHIP_HIP(hipMemset(c->d_cb, 0, cbb));
    return OILHIP_OK;
}

inline uint8_t* kv_idx(const oilhip_kv* c, int layer, int side) { return c->d_idx + ((size_t)layer * 2 + side) * (size_t)c->idx_stride; }
inline uint16_t* kv_cb(const oilhip_kv* c, int layer, int side) { return c->d_cb + ((size_t)layer * 2 + side) * (size_t)c->nblocks * 16; }

}  // namespace
}  // namespace oilhip

using namespace oilhip;

extern "C" {

int oilhip_kv_create(int num_layers, int64_t max_seq_len, int64_t num_heads, int64_t head_dim, int64_t block_size,
                     oilhip_kv** out) {
    if (!out) return fail(OILHIP_E_ARG, "kv_create: out is null");
    *out = nullptr;
    if (num_layers < 0 || max_seq_len < 0 || num_heads < 0 || head_dim < 0) return fail(OILHIP_E_ARG, "kv_create: negative size");
    const int64_t per_token = num_heads * head_dim;
    if (per_token > 0 && max_seq_len > ((int64_t)1 << 40) / per_token) return fail(OILHIP_E_ARG, "kv_create: cache too large");
    oilhip_kv* c = new (std::nothrow) oilhip_kv;
    if (!c) return fail(OILHIP_E_NOMEM, "kv_create: out of host memory");
    if (hipGetDevice(&c->device) != hipSuccess) { delete c; return fail(OILHIP_E_NOGPU, "kv_create: no HIP device"); }
    c->layers = num_layers;
    c->max_seq = max_seq_len;
    c->heads = num_heads;
    c->dim = head_dim;
    c->per_token = per_token;
    c->block = (block_size == 32 || block_size == 64 || block_size == 128) ? block_size : 64;   // kv_cache_oil4.cpp:25-26
    c->pos.assign((size_t)num_layers, 0);
    const int rc = kv_alloc(c);
    if (rc != OILHIP_OK) { delete c; return rc; }
    *out = c;
    return OILHIP_OK;
}

int oilhip_kv_destroy(oilhip_kv* c) {
    if (!c) return OILHIP_OK;
    if (c->d_idx) (void)hipFree(c->d_idx);
    if (c->d_cb) (void)hipFree(c->d_cb);
    delete c;
    return OILHIP_OK;
}

int oilhip_kv_append(oilhip_kv* c, int layer, const float* d_k, const float* d_v, int64_t seq_len, void* stream) {
    if (!c) return fail(OILHIP_E_ARG, "kv_append: cache is null");
    if (layer < 0 || seq_len < 0) return fail(OILHIP_E_ARG, "kv_append: negative layer or length");
    if (layer >= c->layers) return OILHIP_OK;                                       // :209
    const int64_t pos = c->pos[(size_t)layer];
    int64_t ntok = c->max_seq - pos;                                               // tokens past max_seq_len are dropped (:224)
    if (ntok > seq_len) ntok = seq_len;
    if (ntok > 0 && c->per_token > 0) {
        if (!d_k || !d_v) return fail(OILHIP_E_ARG, "kv_append: null input");
        // chunks of a token: one more where its ends may lie inside blocks
        const int64_t cpt = (c->per_token + c->block - 1) / c->block + (c->per_token % c->block ? 1 : 0);
        if (ntok * cpt > 0x7FFFFFFF) return fail(OILHIP_E_ARG, "kv_append: too many tokens for one call");
        const uint32_t items = (uint32_t)(ntok * cpt), per_wave = kv_per_wave(2ull * items);
        const dim3 grid((items + per_wave - 1u) / per_wave, 2);
        const bool busy = kv_busy(2ull * grid.x);
        if (c->per_token % c->block == 0 && (((uintptr_t)d_k | (uintptr_t)d_v) & 15) == 0) {
            auto kern = busy ? (c->block == 32 ? kv_append_whole_kernel<2, true> : c->block == 64 ? kv_append_whole_kernel<4, true> : kv_append_whole_kernel<8, true>)
                             : (c->block == 32 ? kv_append_whole_kernel<2, false> : c->block == 64 ? kv_append_whole_kernel<4, false> : kv_append_whole_kernel<8, false>);
            hipLaunchKernelGGL(kern, grid, dim3(64), 0, (hipStream_t)stream, kv_idx(c, layer, 0), kv_idx(c, layer, 1), kv_cb(c, layer, 0),
                               kv_cb(c, layer, 1), d_k, d_v, pos * cpt, items, per_wave);
        } else {
            auto kern = busy ? (c->block == 32 ? kv_append_kernel<2, true> : c->block == 64 ? kv_append_kernel<4, true> : kv_append_kernel<8, true>)
                             : (c->block == 32 ? kv_append_kernel<2, false> : c->block == 64 ? kv_append_kernel<4, false> : kv_append_kernel<8, false>);
            hipLaunchKernelGGL(kern, grid, dim3(64), 0, (hipStream_t)stream, kv_idx(c, layer, 0), kv_idx(c, layer, 1), kv_cb(c, layer, 0),
                               kv_cb(c, layer, 1), d_k, d_v, pos, ntok, c->per_token, (uint32_t)cpt, items, per_wave, c->idx_bytes);
        }
        OILHIP_HIP(hipGetLastError());
    }
    c->pos[(size_t)layer] = pos + seq_len;                                          // :290, dropped tokens counted as well
    return OILHIP_OK;
}

int oilhip_kv_held(const oilhip_kv* c, int layer, int64_t* tokens) {
    if (!c || !tokens) return fail(OILHIP_E_ARG, "kv_held: null argument");
    // the reference would read past its arrays where tokens were dropped; those are not returned
    *tokens = layer < 0 || layer >= c->layers || c->per_token == 0 ? 0 : std::min(c->pos[(size_t)layer], c->max_seq);
    return OILHIP_OK;
}

int oilhip_kv_get_range(const oilhip_kv* c, int layer, int64_t start, int64_t end, float* d_k, float* d_v, int64_t* len_out,
                        void* stream) {
    if (len_out) *len_out = 0;
    if (!c) return fail(OILHIP_E_ARG, "kv_get_range: cache is null");
    if (layer < 0 || start < 0) return fail(OILHIP_E_ARG, "kv_get_range: negative layer or start");
    if (layer >= c->layers) return OILHIP_OK;                                       // :295
    int64_t held = 0;
    if (int rc = oilhip_kv_held(c, layer, &held)) return rc;
    int64_t len = end - start;
    if (len <= 0) return OILHIP_OK;
    if (start + len > held) len = held - start;
    if (len <= 0) return OILHIP_OK;
    if (!d_k || !d_v) return fail(OILHIP_E_ARG, "kv_get_range: null output");
    const uint64_t first = (uint64_t)start * (uint64_t)c->per_token, count = (uint64_t)len * (uint64_t)c->per_token;
    const uint32_t shift = c->block == 32 ? 5u : c->block == 64 ? 6u : 7u;
    if ((c->per_token & 3) == 0 && (((uintptr_t)d_k | (uintptr_t)d_v) & 15) == 0) {
        const uint64_t tiles = (count + kTile - 1) / kTile;
        if (tiles > 0x7FFFFFFFull) return fail(OILHIP_E_ARG, "kv_get_range: range too long for one call");
        hipLaunchKernelGGL(kv_get_range_kernel, dim3((uint32_t)tiles, 2), dim3(256), 0, (hipStream_t)stream, kv_idx(c, layer, 0),
                           kv_idx(c, layer, 1), kv_cb(c, layer, 0), kv_cb(c, layer, 1), d_k, d_v, first, count, shift,
                           (uint64_t)c->nblocks * 16);
    } else {
        const uint64_t groups = (count + 255) / 256;
        if (groups > 0x7FFFFFFFull) return fail(OILHIP_E_ARG, "kv_get_range: range too long for one call");
        hipLaunchKernelGGL(kv_get_range_scalar_kernel, dim3((uint32_t)groups, 2), dim3(256), 0, (hipStream_t)stream,
                           kv_idx(c, layer, 0), kv_idx(c, layer, 1), kv_cb(c, layer, 0), kv_cb(c, layer, 1), d_k, d_v, first, count,
                           shift, (uint64_t)c->per_token, (uint64_t)c->idx_bytes);
    }
    OILHIP_HIP(hipGetLastError());
    if (len_out) *len_out = len;
    return OILHIP_OK;
}

int oilhip_kv_info(const oilhip_kv* c, int* context_len, int64_t* block_size, uint64_t* size_bytes, uint64_t* fp32_bytes) {
    if (!c) return fail(OILHIP_E_ARG, "kv_info: cache is null");
    const int64_t tokens = c->pos.empty() ? 0 : c->pos[0];                          // context_len(): layer 0 (:368-370)
    if (context_len) *context_len = (int)tokens;
    if (block_size) *block_size = c->block;
    if (size_bytes) *size_bytes = (uint64_t)c->layers * (2ull * (uint64_t)c->idx_bytes + 2ull * (uint64_t)c->nblocks * 32ull);   // :372-380
    if (fp32_bytes) *fp32_bytes = (uint64_t)(tokens * c->per_token * 2 * 4);        // :382-386
    return OILHIP_OK;
}

int oilhip_kv_clear(oilhip_kv* c, void* stream) {
    if (!c) return fail(OILHIP_E_ARG, "kv_clear: cache is null");
    const uint64_t n_idx = (uint64_t)c->layers * 2 * (uint64_t)c->idx_stride / 16, n_cb = (uint64_t)c->layers * 2 * (uint64_t)c->nblocks * 32 / 16;
    if (n_idx + n_cb)
        hipLaunchKernelGGL(kv_zero_kernel, dim3((uint32_t)std::min<uint64_t>((n_idx + n_cb + 255) / 256, 4096)), dim3(256), 0, (hipStream_t)stream,
                           reinterpret_cast<uint4*>(c->d_idx), n_idx, reinterpret_cast<uint4*>(c->d_cb), n_cb);
    OILHIP_HIP(hipGetLastError());
    for (auto& p : c->pos) p = 0;
    return OILHIP_OK;
}

int oilhip_kv_resize(oilhip_kv* c, int64_t new_max_seq_len) {
    if (!c) return fail(OILHIP_E_ARG, "kv_resize: cache is null");
    if (new_max_seq_len < 0) return fail(OILHIP_E_ARG, "kv_resize: negative length");
    OILHIP_HIP(hipDeviceSynchronize());
    if (c->d_idx) (void)hipFree(c->d_idx);
    if (c->d_cb) (void)hipFree(c->d_cb);
    c->max_seq = new_max_seq_len;
    for (auto& p : c->pos) p = 0;                                                   // :408 -- every layer starts empty again
    return kv_alloc(c);
}

int oilhip_kv_state(const oilhip_kv* c, int layer, uint8_t* k_idx, uint8_t* v_idx, uint16_t* k_cb, uint16_t* v_cb) {
    if (!c || layer < 0 || layer >= c->layers) return fail(OILHIP_E_ARG, "kv_state: bad cache or layer");
    OILHIP_HIP(hipDeviceSynchronize());
    if (c->idx_bytes) {
        if (k_idx) OILHIP_HIP(hipMemcpy(k_idx, kv_idx(c, layer, 0), (size_t)c->idx_bytes, hipMemcpyDeviceToHost));
        if (v_idx) OILHIP_HIP(hipMemcpy(v_idx, kv_idx(c, layer, 1), (size_t)c->idx_bytes, hipMemcpyDeviceToHost));
        if (k_cb) OILHIP_HIP(hipMemcpy(k_cb, kv_cb(c, layer, 0), (size_t)c->nblocks * 32, hipMemcpyDeviceToHost));
        if (v_cb) OILHIP_HIP(hipMemcpy(v_cb, kv_cb(c, layer, 1), (size_t)c->nblocks * 32, hipMemcpyDeviceToHost));
    }
    return OILHIP_OK;
}

int oilhip_kv_quantize_blocks(const float* d_src, int64_t n, int64_t nblocks, uint8_t* d_codes, uint16_t* d_cb16, void* stream) {
    if (n < 0 || nblocks < 0) return fail(OILHIP_E_ARG, "kv_quantize_blocks: negative size");
    if (n > 128) return fail(OILHIP_E_ARG, "kv_quantize_blocks: at most 128 values per block on the device (the cache's largest block)");
    if (n == 0 || nblocks == 0) return OILHIP_OK;                                   // :78
    if (!d_src || !d_codes || !d_cb16) return fail(OILHIP_E_ARG, "kv_quantize_blocks: null pointer");
    if (nblocks > 0x7FFFFFFF) return fail(OILHIP_E_ARG, "kv_quantize_blocks: too many blocks for one call");
    const uint32_t per_wave = kv_per_wave((uint64_t)nblocks);
    auto kern = n <= 32 ? kv_quantize_blocks_kernel<2> : n <= 64 ? kv_quantize_blocks_kernel<4> : kv_quantize_blocks_kernel<8>;
    hipLaunchKernelGGL(kern, dim3(((uint32_t)nblocks + per_wave - 1u) / per_wave), dim3(64), 0, (hipStream_t)stream, d_src, (uint32_t)n,
                       (uint32_t)nblocks, per_wave, d_codes, d_cb16);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

int oilhip_kv_dequantize_blocks(const uint8_t* d_codes, const uint16_t* d_cb16, float* d_dst, int64_t n, int64_t nblocks, void* stream) {
    if (n < 0 || nblocks < 0) return fail(OILHIP_E_ARG, "kv_dequantize_blocks: negative size");
    if (n == 0 || nblocks == 0) return OILHIP_OK;
    if (!d_codes || !d_cb16 || !d_dst) return fail(OILHIP_E_ARG, "kv_dequantize_blocks: null pointer");
    const uint64_t total = (uint64_t)n * (uint64_t)nblocks;
    if ((total + 255) / 256 > 0x7FFFFFFFull || n > 0x7FFFFFFF) return fail(OILHIP_E_ARG, "kv_dequantize_blocks: too large for one call");
    hipLaunchKernelGGL(kv_dequantize_blocks_kernel, dim3((uint32_t)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, d_codes, d_cb16, d_dst, (uint32_t)n, total);
    OILHIP_HIP(hipGetLastError());
    return OILHIP_OK;
}

}  // extern "C"
