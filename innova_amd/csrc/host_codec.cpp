// host_codec.cpp -- host-side OIL block quantizer (the producer of block
// payloads).  In the reference the quantizer is CPU code as well
// (quantize_block_all, src/block_codec.cpp:368-574); it is not part of the
// accelerated decode path.  The reference build fuses a*b+c (its -mfma flag
// with the compiler's default contraction), so sums of products below use
// std::fma explicitly and this file is compiled with -ffp-contract=off.
#include <immintrin.h>
#include <sched.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <limits>
#include <span>
#include <thread>
#include <utility>
#include <vector>

#include "../../include/oilhip.h"

namespace oilhip {
int fail(int code, const std::string& msg);
}

namespace {

// quantize_tensor: at least this many weights per thread (0.2 ms of work; starting one costs 0.02 to 0.05 ms: 300,000 weights take 0.35 ms on one thread and 0.4 to 0.5
// on four), at most this many threads (67 MB of weights took 3.0 ms on 16 and on 32 of them)
constexpr uint64_t kWeightsPerThread = 262144;
constexpr int kMaxThreads = 32;

constexpr std::array<float, 4> kL2 = {-1.5104f, -0.4528f, 0.4528f, 1.5104f};
constexpr std::array<float, 16> kL4 = {-2.7178f, -2.0522f, -1.5995f, -1.2392f, -0.9275f, -0.6508f,
                                       -0.3976f, -0.1260f, 0.1260f,  0.3976f,  0.6508f,  0.9275f,
                                       1.2392f,  1.5995f,  2.0522f,  2.7178f};

// block_codec.cpp:26-59 -- round to nearest even, overflow and NaN to infinity,
// magnitudes under 2^-24 to signed zero.
uint16_t to_half(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    const uint32_t sgn = (u >> 16) & 0x8000u;
    int ex = int((u >> 23) & 0xFF) - 127;
    if (ex > 15) return uint16_t(sgn | 0x7C00u);
    if (ex < -24) return uint16_t(sgn);
    const uint32_t sig = (u & 0x7FFFFFu) | 0x800000u;
    const int cut = ex >= -14 ? 13 : -ex - 1;
    uint32_t keep = sig >> cut;
    const uint32_t lost = sig & ((1u << cut) - 1u), mid = 1u << (cut - 1);
    keep += (lost > mid) || (lost == mid && (keep & 1u));
    if (ex < -14) return uint16_t(sgn | keep);
    if (keep >= 0x800u) {
        keep >>= 1;
        if (++ex > 15) return uint16_t(sgn | 0x7C00u);
    }
    return uint16_t(sgn | uint32_t(ex + 15) << 10 | (keep & 0x3FFu));
}

// LSB-first bit sink over a fixed-size byte span (block_codec.cpp:87-100).
class BitSink {
public:
    explicit BitSink(std::span<uint8_t> out) : out_(out) { std::fill(out.begin(), out.end(), uint8_t{0}); }
    void put(uint32_t v, int n) {
        for (int i = 0; i < n; ++i, ++at_)
            if ((at_ >> 3) < out_.size() && ((v >> i) & 1u)) out_[at_ >> 3] |= uint8_t(1u << (at_ & 7));
    }
    void skip(size_t n) { at_ += n; }
private:
    std::span<uint8_t> out_;
    size_t at_ = 0;
};

bool is_slot(long long i, long long n, int count) {   // block_codec.cpp:122-126
    return count > 0 && n > 0 && ((i + 1) * count) / n != (i * count) / n;
}

template <size_t N>
uint32_t nearest(float v, const std::array<float, N>& lv) {   // :139-146, ties keep the lower index
    uint32_t best = 0;
    float bd = std::fabs(v - lv[0]);
    for (uint32_t i = 1; i < N; ++i) {
        const float d = std::fabs(v - lv[i]);
        if (d < bd) { bd = d; best = i; }
    }
    return best;
}

uint32_t nearest_level(float v, int bits) {
    if (bits == 2) return nearest(v, kL2);
    if (bits == 4) return nearest(v, kL4);
    const float c = std::max(-8.0f, std::min(8.0f, v));
    return uint32_t(std::lround((c + 8.0f) * 255.0f / 16.0f));
}

float rms(std::span<const float> w) {   // :149-154
    if (w.empty()) return 0.0f;
    double s = 0.0;
    for (float x : w) s = std::fma(double(x), double(x), s);
    return float(std::sqrt(s / double(w.size())));
}

uint32_t cap255(long v) { return uint32_t(v) > 255u ? 255u : uint32_t(v); }

size_t grp_header_bits(int n) { return n < 64 ? (n < 8 ? 0u : 16u) : size_t(n / 64) * 32u; }

size_t payload_bound(int fmt, int n) {
    if (n <= 0) return 0;
    const size_t N = size_t(n);
    switch (fmt) {
        case OILHIP_OIL32: return N * 4;
        case OILHIP_OIL16: case OILHIP_OIL16_GRP: return N * 2;
        case OILHIP_OIL8: return N;
        case OILHIP_OIL4: return (N * 4 + 7) / 8;
        case OILHIP_OIL2: return (N * 2 + 7) / 8;
        case OILHIP_OIL8_GRP: return (grp_header_bits(n) + N * 8 + 7) / 8;
        case OILHIP_OIL4_GRP: return (grp_header_bits(n) + N * 4 + 7) / 8;
        case OILHIP_OIL2_GRP: return (grp_header_bits(n) + N * 2 + 7) / 8;
        case OILHIP_OIL1: return ((N + 31) / 32) * 2;
        case OILHIP_OIL1_GRP: return (N + 7) / 8;
        case OILHIP_SPARK_Q0: return (N * 3 + 15) / 16;
        case OILHIP_SPARK_Q0_GRP: return n < 32 ? (N + 7) / 8 : (N * 3 + 15) / 16;
        case OILHIP_SPARK_SPARSE: return N / 4 < 4 ? 0 : 4 + std::min<size_t>(20, (N / 4 - 4) / 3) * 3;
        case OILHIP_SPARK_SPARSE_GRP: return N / 4 < 8 ? 0 : 4 + ((N / 4 - 4) / 3) * 3;
        default: return 0;
    }
}

size_t encode_lattice(std::span<const float> w, int bits, uint8_t* out) {   // :157-171
    const int n = int(w.size());
    const size_t bytes = (size_t(bits) * n + 7) / 8;
    BitSink sink({out, bytes});
    const float scale = rms(w);
    sink.put(to_half(scale), 16);
    const float s = scale <= 1e-12f ? 0.0f : scale;
    for (int i = 0; i < n; ++i) {
        if (is_slot(i, n, 16 / bits)) continue;
        sink.put(nearest_level(s == 0.0f ? 0.0f : w[i] / s, bits), bits);
    }
    return bytes;
}

size_t encode_grouped(std::span<const float> w, int bits, uint8_t* out) {   // :191-306
    const int n = int(w.size()), full = n / 64;
    const bool wide = bits == 8;
    const size_t bytes = (grp_header_bits(n) + size_t(n) * bits + 7) / 8;
    BitSink sink({out, bytes});
    auto code = [&](float v, float zp, float sc) -> uint32_t {
        if (wide) return cap255(std::lround((v - zp) / sc * 255.0f));
        return nearest_level(float((double(v) - zp) / double(sc)), bits);
    };
    float pzp = 0.0f, psc = 1.0f;
    for (int g = 0; g < full; ++g) {
        const auto grp = w.subspan(size_t(g) * 64, 64);
        float zp, sc;
        if (wide) {
            const auto [lo, hi] = std::minmax_element(grp.begin(), grp.end());
            zp = *lo;
            sc = *hi - *lo;
        } else {
            double mu = 0.0, ss = 0.0;
            for (float x : grp) mu += x;
            mu /= 64.0;
            for (float x : grp) { const double d = double(x) - mu; ss = std::fma(d, d, ss); }
            zp = float(mu);
            sc = ss > 0.0 ? float(std::sqrt(ss / 64.0)) : 0.0f;
        }
        sink.put(to_half(zp), 16);
        sink.put(to_half(sc), 16);
        pzp = zp;
        psc = sc;
        if (sc == 0.0f) { sink.skip(size_t(64) * bits); continue; }
        for (float x : grp) sink.put(code(x, zp, sc), bits);
    }
    const auto tail = w.subspan(size_t(full) * 64);
    if (tail.empty()) return bytes;
    if (full > 0) {                               // partial tail reuses the last group's zp/scale
        for (float x : tail) sink.put(psc == 0.0f ? 0u : code(x, pzp, psc), bits);
        return bytes;
    }
    if (n < 8) {                                  // headerless: implicit scale 1, zero-point 0
        for (float x : tail)
            sink.put(wide ? cap255(std::lround((x + 1.0f) * 127.5f)) : nearest_level(x, bits), bits);
        return bytes;
    }
    float sc;
    if (wide) {
        sc = std::fabs(tail[0]);
        for (float x : tail.subspan(1)) sc = std::max(sc, std::fabs(x));
    } else {
        double ss = 0.0;
        for (float x : tail) ss = std::fma(double(x), double(x), ss);
        sc = ss > 0.0 ? float(std::sqrt(ss / double(n))) : 0.0f;
    }
    sink.put(to_half(sc), 16);
    if (sc == 0.0f) return bytes;
    for (float x : tail)
        sink.put(wide ? cap255(std::lround((x / sc + 1.0f) * 127.5f)) : nearest_level(x / sc, bits), bits);
    return bytes;
}

size_t encode_sparse(std::span<const float> w, bool grouped, uint8_t* out) {   // :484-570
    const int n = int(w.size());
    const size_t budget = size_t(n) / 4;
    if (budget < (grouped ? 8u : 4u)) return 0;
    int keep = int((budget - 4) / 3);
    if (!grouped) keep = std::min(keep, 20);
    if (grouped && keep <= 0) return 0;
    const int half = n / 2;
    std::vector<std::pair<float, int>> mag(static_cast<size_t>(n));
    float s0 = 0.0f, s1 = 0.0f;
    for (int i = 0; i < n; ++i) {
        const float a = std::fabs(w[i]);
        mag[size_t(i)] = {a, i};
        float& top = (!grouped || i < half) ? s0 : s1;
        top = std::max(top, a);
    }
    if (!grouped) {
        if (s0 <= 1e-12f) { std::memset(out, 0, 4); return 4; }
        std::memcpy(out, &s0, 4);
    } else {
        if (s0 <= 1e-12f) s0 = 1.0f;
        if (s1 <= 1e-12f) s1 = 1.0f;
        const uint16_t h0 = to_half(s0), h1 = to_half(s1);
        out[0] = uint8_t(h0); out[1] = uint8_t(h0 >> 8); out[2] = uint8_t(h1); out[3] = uint8_t(h1 >> 8);
    }
    if (keep > 0)   // same call as the reference: equal magnitudes land where libstdc++'s heap puts them
        std::partial_sort(mag.begin(), mag.begin() + keep, mag.end(),
                          [](const auto& a, const auto& b) { return a.first > b.first; });
    for (int r = 0; r < keep; ++r) {
        const int at = mag[size_t(r)].second;
        const float s = (!grouped || at < half) ? s0 : s1;
        const int q = std::clamp(int(std::lround(w[at] / s * 127.0f)), -127, 127);
        uint8_t* rec = out + 4 + 3 * size_t(r);
        rec[0] = uint8_t(at); rec[1] = uint8_t(at >> 8); rec[2] = uint8_t(int8_t(q));
    }
    return 4 + 3 * size_t(keep);
}

// Encodes one block; returns false for an unknown format.  cb receives the OIL1
// run means, idx everything else.
bool encode_block(int fmt, std::span<const float> w, uint8_t* idx, size_t& il, uint8_t* cb, size_t& cl) {
    const int n = int(w.size());
    il = cl = 0;
    auto sign_bit = [](float v) { return v >= 0.0f ? 1u : 0u; };
    switch (fmt) {
        case OILHIP_OIL32: std::memcpy(idx, w.data(), size_t(n) * 4); il = size_t(n) * 4; return true;
        case OILHIP_OIL16: case OILHIP_OIL16_GRP:
            for (int i = 0; i < n; ++i) { const uint16_t h = to_half(w[i]); idx[2 * i] = uint8_t(h); idx[2 * i + 1] = uint8_t(h >> 8); }
            il = size_t(n) * 2; return true;
        case OILHIP_OIL8: il = encode_lattice(w, 8, idx); return true;
        case OILHIP_OIL4: il = encode_lattice(w, 4, idx); return true;
        case OILHIP_OIL2: il = encode_lattice(w, 2, idx); return true;
        case OILHIP_OIL8_GRP: il = encode_grouped(w, 8, idx); return true;
        case OILHIP_OIL4_GRP: il = encode_grouped(w, 4, idx); return true;
        case OILHIP_OIL2_GRP: il = encode_grouped(w, 2, idx); return true;
        case OILHIP_OIL1:                                       // :406-420
            for (int a = 0, r = 0; a < n; a += 32, ++r) {
                const auto run = w.subspan(size_t(a), size_t(std::min(32, n - a)));
                double s = 0.0;
                for (float x : run) s += x;
                const uint16_t h = to_half(float(s / double(run.size())));
                cb[2 * r] = uint8_t(h); cb[2 * r + 1] = uint8_t(h >> 8);
                cl += 2;
            }
            return true;
        case OILHIP_OIL1_GRP: {                                 // :421-443
            il = (size_t(n) + 7) / 8;
            BitSink sink({idx, il});
            if (n >= 32) sink.put(to_half(rms(w)), 16);
            for (int i = 0; i < n; ++i)
                if (n < 32 || !is_slot(i, n, 16)) sink.put(sign_bit(w[i]), 1);
            return true;
        }
        case OILHIP_SPARK_Q0: {                                 // :444-458
            il = (size_t(n) * 3 + 15) / 16;
            BitSink sink({idx, il});
            for (int a = 0; a < n; a += 32) {
                const auto run = w.subspan(size_t(a), size_t(std::min(32, n - a)));
                if (run.size() == 32) sink.put(to_half(rms(run)), 16);
                for (float x : run) sink.put(sign_bit(x), 1);
            }
            return true;
        }
        case OILHIP_SPARK_Q0_GRP: {                             // :459-483
            if (n < 32) {
                il = (size_t(n) + 7) / 8;
                BitSink sink({idx, il});
                for (float x : w) sink.put(sign_bit(x), 1);
                return true;
            }
            il = (size_t(n) * 3 + 15) / 16;
            BitSink sink({idx, il});
            const float scale = rms(w);
            sink.put(to_half(scale), 16);
            for (float x : w) sink.put(sign_bit(x), 1);
            const float thr = scale * 1.23f;
            for (int i = 0; i < n; ++i)
                if (is_slot(i, n, n / 2 - 16)) sink.put(std::fabs(w[i]) > thr ? 1u : 0u, 1);
            return true;
        }
        case OILHIP_SPARK_SPARSE: il = encode_sparse(w, false, idx); return true;
        case OILHIP_SPARK_SPARSE_GRP: il = encode_sparse(w, true, idx); return true;
        default: return false;
    }
}

// ---- full 256-weight blocks ------------------------------------------------------------------------------------
// What a model's tensors consist of, so the encoders below are written for the vector units: the same rounded
// operations as above in the same order per result, laid out so that independent results run side by side.
//   * sums of squares and means are sequential chains in double: one chain per block, group or run as above, but
//     several of them interleaved (a single chain waits four cycles per weight).  A float's square is exact in
//     double, so adding it rounds as the fused form does.
//   * nearest() over a sorted table is a step function of v: the code is the number of thresholds that v reaches.
//     The thresholds are found once with nearest() itself (threshold_table), ties and rounding included.  Only values
//     of bounded magnitude come here (|v| <= 16: a weight over the RMS of its 256), where distances to distant levels
//     never round to the same float.
//   * codes are laid out one per byte and packed a dword at a time instead of bit by bit.
// Blocks with a non-finite or enormous weight go through encode_block.  The plain forms are compiled for AVX2 and the baseline; for AVX-512 the parts
// that are bound by their instructions are written out: sums of runs whose floats are transposed eight by eight so that a lane is a chain, codes by a
// search of four steps over thresholds that are in the weights' scale (no division per weight), halves and signs a register at a time, and
// the next sixteen blocks fetched while these are encoded.  One thread, ns per weight without the output pages' first touch (Xeon 2.7 GHz), bit by bit -> plain
// forms -> AVX-512, weights in cache: OIL4 54 -> 1.6 to 2.3 -> 0.6 to 0.9, OIL8 53 -> 0.8 to 1.2 -> 0.6 to 0.9, SPARK_Q0 11.9 -> 1.7 to 2.5 -> 0.3 to 0.5; whole calls of 4 M weights, ms:
// OIL4_GRP 18.1 -> 7.9, OIL8_GRP 12.9 -> 6.4, SPARK_Q0 and OIL1 mixed 10.7 -> 3.0, OIL2 7.6 -> 4.0.  16 M weights of OIL4 on eight threads 8.5 -> 5.0 ms, of
// which the first touch of the output pages is a third.
#define OIL_INLINE inline __attribute__((always_inline))

template <size_t N>
std::array<float, N - 1> threshold_table(const std::array<float, N>& lv) {
    std::array<float, N - 1> t;
    for (uint32_t i = 1; i < N; ++i) {
        // the smallest float between two levels at which nearest() answers i; bit patterns of floats of one sign are
        // ordered, so the search runs over integers that order floats of both signs
        auto key = [](float f) { int32_t b; std::memcpy(&b, &f, 4); return b < 0 ? int32_t(0x80000000u - uint32_t(b)) : b; };
        auto val = [](int32_t k) { const int32_t b = k < 0 ? int32_t(0x80000000u - uint32_t(k)) : k; float f; std::memcpy(&f, &b, 4); return f; };
        int64_t lo = key(lv[i - 1]), hi = key(lv[i]);                  // nearest(lo) = i - 1, nearest(hi) = i
        while (hi - lo > 1) {
            const int64_t mid = lo + (hi - lo) / 2;
            (nearest(val(int32_t(mid)), lv) >= i ? hi : lo) = mid;
        }
        t[i - 1] = val(int32_t(hi));
    }
    return t;
}
const std::array<float, 3> kT2 = threshold_table(kL2);
const std::array<float, 15> kT4 = threshold_table(kL4);

OIL_INLINE void put16(uint8_t* p, uint16_t v) { std::memcpy(p, &v, 2); }

// sum of squares of `runs` consecutive runs of `len` floats each, every run a chain of its own
template <int RUNS, int LEN>
OIL_INLINE void square_sums(const float* w, double* s) {
    for (int r = 0; r < RUNS; ++r) s[r] = 0.0;
    for (int i = 0; i < LEN; ++i)
        for (int r = 0; r < RUNS; ++r) { const double x = w[r * LEN + i]; s[r] += x * x; }
}

// ---- the parts that are bound by their instructions, for AVX-512; plain functions of a block or more: a call costs nothing beside them ----
#define OIL_AVX512 __attribute__((target("avx512f,avx512bw,avx512dq,avx512vl,avx2,fma")))
#pragma clang attribute push(OIL_AVX512, apply_to = function)                // lambdas included

// Eight floats each of eight runs -> element k of all runs in column k.
template <class Run>
OIL_INLINE void transpose8(Run&& run, __m256 (&t)[8]) {
    __m256 r[8], u[8];
    for (int j = 0; j < 8; ++j) r[j] = _mm256_loadu_ps(run(j));
    for (int j = 0; j < 8; j += 2) { u[j] = _mm256_unpacklo_ps(r[j], r[j + 1]); u[j + 1] = _mm256_unpackhi_ps(r[j], r[j + 1]); }
    for (int j = 0; j < 8; j += 4)
        for (int k = 0; k < 2; ++k) {
            r[j + 2 * k] = _mm256_shuffle_ps(u[j + k], u[j + k + 2], 0x44);
            r[j + 2 * k + 1] = _mm256_shuffle_ps(u[j + k], u[j + k + 2], 0xEE);
        }
    for (int k = 0; k < 4; ++k) {
        t[k] = _mm256_permute2f128_ps(r[k], r[k + 4], 0x20);
        t[k + 4] = _mm256_permute2f128_ps(r[k], r[k + 4], 0x31);
    }
}

// Sums of squares (or of the floats themselves) of 8 * SETS runs of LEN floats: a lane of a register is a run's chain.  (Loads that are whole runs
// apart, one float each, took 0.8 ns per weight.)
template <int SETS, int LEN, bool SQUARES = true>
void run_sums_avx512(const float* w, double* s) {
    __m512d acc[SETS];
    for (int r = 0; r < SETS; ++r) acc[r] = _mm512_setzero_pd();
    for (int i = 0; i < LEN; i += 8)
        for (int r = 0; r < SETS; ++r) {
            __m256 t[8];
            transpose8([&](int j) { return w + size_t(8 * r + j) * LEN + i; }, t);
            for (int k = 0; k < 8; ++k) {
                const __m512d x = _mm512_cvtps_pd(t[k]);
                acc[r] = SQUARES ? _mm512_fmadd_pd(x, x, acc[r]) : _mm512_add_pd(acc[r], x);
            }
        }
    for (int r = 0; r < SETS; ++r) _mm512_storeu_pd(s + 8 * r, acc[r]);
}

// to_half of eight floats.  The instruction rounds as to_half does but for magnitudes below 2^-24, which to_half makes zero.
OIL_INLINE void halves8(__m256 v, uint16_t* out) {
    const __m256 mag = _mm256_andnot_ps(_mm256_set1_ps(-0.0f), v);
    const __mmask8 small = _mm256_cmp_ps_mask(mag, _mm256_set1_ps(0x1p-24f), _CMP_LT_OQ);
    _mm_storeu_si128(reinterpret_cast<__m128i*>(out), _mm256_cvtps_ph(_mm256_mask_and_ps(v, small, v, _mm256_set1_ps(-0.0f)), _MM_FROUND_TO_NEAREST_INT));
}

inline void spark_avx512(const float* w, uint8_t* out) {
    alignas(64) double s[8];
    alignas(16) uint16_t h[8];
    run_sums_avx512<1, 32>(w, s);
    halves8(_mm512_cvtpd_ps(_mm512_sqrt_pd(_mm512_div_pd(_mm512_load_pd(s), _mm512_set1_pd(32.0)))), h);
    for (int r = 0; r < 8; ++r) {
        const __mmask16 lo = _mm512_cmp_ps_mask(_mm512_loadu_ps(w + 32 * r), _mm512_setzero_ps(), _CMP_GE_OQ);
        const __mmask16 hi = _mm512_cmp_ps_mask(_mm512_loadu_ps(w + 32 * r + 16), _mm512_setzero_ps(), _CMP_GE_OQ);
        const uint64_t six = uint64_t(h[r]) | uint64_t(uint32_t(lo) | uint32_t(hi) << 16) << 16;
        std::memcpy(out + 6 * r, &six, 6);
    }
}

inline void means_avx512(const float* w, uint8_t* out) {
    alignas(64) double s[8];
    run_sums_avx512<1, 32, false>(w, s);
    halves8(_mm512_cvtpd_ps(_mm512_div_pd(_mm512_load_pd(s), _mm512_set1_pd(32.0))), reinterpret_cast<uint16_t*>(out));
}

// A weight's code is the number of thresholds (sorted, padded with infinity) that v reaches: four steps for fifteen, two for three.
template <int N>
OIL_INLINE __m128i search_avx512(__m512 v, __m512 from, __m512 middle) {
    __m512i q = _mm512_maskz_set1_epi32(_mm512_cmp_ps_mask(v, middle, _CMP_GE_OQ), (N + 1) / 2);
    for (int half = (N + 1) / 4; half >= 1; half /= 2) {                 // thresholds q .. q + 2 half - 2 are left: the one in their middle
        const __m512 m = _mm512_permutexvar_ps(_mm512_add_epi32(q, _mm512_set1_epi32(half - 1)), from);
        q = _mm512_mask_add_epi32(q, _mm512_cmp_ps_mask(v, m, _CMP_GE_OQ), q, _mm512_set1_epi32(half));
    }
    return _mm512_cvtepi32_epi8(q);
}

// The codes of 256 weights over their scale.  The quotient rises with the weight, so that it reaches a threshold t from one weight on, which is a
// float or two from t * scale: found by dividing there, once for all thresholds, and no weight is divided.  False where a neighbour on either side does
// not settle a threshold (t * scale just above a power of two).
template <size_t N>
bool codes_avx512(const float* w, float scale, const std::array<float, N>& thresholds, uint8_t* code) {
    alignas(64) float t[16];
    for (size_t j = 0; j < 16; ++j) t[j] = thresholds[j < N ? j : N - 1];
    const __m512 tv = _mm512_load_ps(t), sv = _mm512_set1_ps(scale), c = _mm512_mul_ps(tv, sv);
    const __m512i up = _mm512_mask_blend_epi32(_mm512_movepi32_mask(_mm512_castps_si512(c)), _mm512_set1_epi32(1), _mm512_set1_epi32(-1));     // to the next float
    auto reaches = [&](__m512 v) { return _mm512_cmp_ps_mask(_mm512_div_ps(v, sv), tv, _CMP_GE_OQ); };
    const __m512 above = _mm512_castsi512_ps(_mm512_add_epi32(_mm512_castps_si512(c), up));
    const __m512 below = _mm512_castsi512_ps(_mm512_sub_epi32(_mm512_castps_si512(c), up));
    const __m512 lower = _mm512_castsi512_ps(_mm512_sub_epi32(_mm512_castps_si512(below), up));
    if (reaches(above) != 0xFFFF || reaches(lower) != 0) return false;
    __m512 from = _mm512_mask_blend_ps(reaches(c), above, c);
    from = _mm512_mask_blend_ps(reaches(below), from, below);
    if constexpr (N == 15) from = _mm512_mask_blend_ps(0x8000, from, _mm512_set1_ps(std::numeric_limits<float>::infinity()));
    const __m512 middle = _mm512_permutexvar_ps(_mm512_set1_epi32(int(N) / 2), from);
    for (int i = 0; i < 256; i += 16) _mm_store_si128(reinterpret_cast<__m128i*>(code + i), search_avx512<int(N)>(_mm512_loadu_ps(w + i), from, middle));
    return true;
}

// level_code<8> of 256 weights over their scale, straight into the block: 254 bytes, the last of every 128 left out
inline void codes8_avx512(const float* w, float scale, uint8_t* out) {
    const __m512 sv = _mm512_set1_ps(scale);
    for (int i = 0; i < 256; i += 16) {
        const __m512 c = _mm512_max_ps(_mm512_min_ps(_mm512_div_ps(_mm512_loadu_ps(w + i), sv), _mm512_set1_ps(8.0f)), _mm512_set1_ps(-8.0f));
        const __m512 r = _mm512_mul_ps(_mm512_mul_ps(_mm512_add_ps(c, _mm512_set1_ps(8.0f)), _mm512_set1_ps(255.0f)), _mm512_set1_ps(0.0625f));
        const __m512i k = _mm512_cvttps_epi32(r);
        const __mmask16 half = _mm512_cmp_ps_mask(_mm512_sub_ps(r, _mm512_cvtepi32_ps(k)), _mm512_set1_ps(0.5f), _CMP_GE_OQ);
        const __m128i b = _mm512_cvtepi32_epi8(_mm512_mask_add_epi32(k, half, k, _mm512_set1_epi32(1)));
        if (i < 240) _mm_storeu_si128(reinterpret_cast<__m128i*>(out + i - i / 128), b);       // (code 127 lies under the next run's first)
        else _mm_mask_storeu_epi8(out + 239, 0x7FFF, b);
    }
}

// 64 codes, one per byte -> 8 BITS bytes, first code in the low bits
template <int BITS>
OIL_INLINE auto pack64_avx512(__m512i c) {
    if constexpr (BITS == 4) {
        return _mm512_cvtepi16_epi8(_mm512_maddubs_epi16(c, _mm512_set1_epi16(0x1001)));                       // a byte's code + 16 times the next
    } else {
        const __m512i pairs = _mm512_maddubs_epi16(c, _mm512_set1_epi16(0x0401));
        return _mm512_cvtepi32_epi8(_mm512_madd_epi16(pairs, _mm512_set1_epi32(0x00100001)));
    }
}

// The codes of 256 weights, one per byte, without the last of every 16 * BITS: 32 BITS - 2 bytes
template <int BITS>
void pack_lattice_avx512(const uint8_t* code, uint8_t* out) {
    constexpr int RUN = 16 * BITS;
    alignas(64) uint8_t dense[256 + 64];
    for (int r = 0; r < 256 / RUN; ++r) {
        if constexpr (BITS == 4) _mm512_storeu_si512(dense + r * (RUN - 1), _mm512_load_si512(code + r * RUN));
        else _mm256_storeu_si256(reinterpret_cast<__m256i*>(dense + r * (RUN - 1)), _mm256_load_si256(reinterpret_cast<const __m256i*>(code + r * RUN)));
    }
    for (int i = 0; i < 4; ++i) {
        const auto b = pack64_avx512<BITS>(_mm512_load_si512(dense + 64 * i));
        if constexpr (BITS == 4) {
            if (i < 3) _mm256_storeu_si256(reinterpret_cast<__m256i*>(out + 32 * i), b);
            else _mm256_mask_storeu_epi8(out + 96, 0x3FFFFFFFu, b);
        } else {
            if (i < 3) _mm_storeu_si128(reinterpret_cast<__m128i*>(out + 16 * i), b);
            else _mm_mask_storeu_epi8(out + 48, 0x3FFFu, b);
        }
    }
}

// Mean and deviation of the four groups of 64 of each of four blocks, every sum in order in a lane of its own: one block's four sums would wait four
// cycles per weight for each other.
inline void moments_avx512(const float* const (&block)[4], float (&zp)[4][4], float (&sc)[4][4]) {
    __m512d mu[2] = {_mm512_setzero_pd(), _mm512_setzero_pd()}, ss[2] = {_mm512_setzero_pd(), _mm512_setzero_pd()};
    for (int i = 0; i < 64; i += 8)
        for (int h = 0; h < 2; ++h) {
            __m256 t[8];
            transpose8([&](int j) { return block[2 * h + j / 4] + 64 * (j % 4) + i; }, t);
            for (int k = 0; k < 8; ++k) mu[h] = _mm512_add_pd(mu[h], _mm512_cvtps_pd(t[k]));
        }
    for (int h = 0; h < 2; ++h) mu[h] = _mm512_div_pd(mu[h], _mm512_set1_pd(64.0));
    for (int i = 0; i < 64; i += 8)
        for (int h = 0; h < 2; ++h) {
            __m256 t[8];
            transpose8([&](int j) { return block[2 * h + j / 4] + 64 * (j % 4) + i; }, t);
            for (int k = 0; k < 8; ++k) { const __m512d d = _mm512_sub_pd(_mm512_cvtps_pd(t[k]), mu[h]); ss[h] = _mm512_fmadd_pd(d, d, ss[h]); }
        }
    for (int h = 0; h < 2; ++h) {
        _mm256_storeu_ps(zp[2 * h], _mm512_cvtpd_ps(mu[h]));
        _mm256_storeu_ps(sc[2 * h], _mm512_cvtpd_ps(_mm512_sqrt_pd(_mm512_div_pd(ss[h], _mm512_set1_pd(64.0)))));
    }
}

// full_grouped<BITS> with the groups' zero points and scales
template <int BITS>
void grouped_avx512(const float* w, const float* zp, const float* sc, uint8_t* out) {
    constexpr int N = BITS == 4 ? 15 : 3;
    alignas(64) float t[16];
    for (int j = 0; j < 16; ++j) t[j] = j >= N ? std::numeric_limits<float>::infinity() : BITS == 4 ? kT4[size_t(j % 15)] : kT2[size_t(j % 3)];
    const __m512 from = _mm512_load_ps(t), middle = _mm512_set1_ps(t[N / 2]);
    for (int g = 0; g < 4; ++g) {
        uint8_t* o = out + g * (4 + 8 * BITS);
        put16(o, to_half(zp[g]));
        put16(o + 2, to_half(sc[g]));
        if (sc[g] == 0.0f) { std::memset(o + 4, 0, 8 * BITS); continue; }
        const __m512d z = _mm512_set1_pd(double(zp[g])), c = _mm512_set1_pd(double(sc[g]));
        alignas(64) uint8_t code[64];
        for (int i = 0; i < 64; i += 16) {
            auto half = [&](int at) { return _mm512_cvtpd_ps(_mm512_div_pd(_mm512_sub_pd(_mm512_cvtps_pd(_mm256_loadu_ps(w + 64 * g + at)), z), c)); };
            const __m512 v = _mm512_insertf32x8(_mm512_castps256_ps512(half(i)), half(i + 8), 1);
            _mm_store_si128(reinterpret_cast<__m128i*>(code + i), search_avx512<N>(v, from, middle));
        }
        const auto b = pack64_avx512<BITS>(_mm512_load_si512(code));
        if constexpr (BITS == 4) _mm256_storeu_si256(reinterpret_cast<__m256i*>(o + 4), b);
        else _mm_storeu_si128(reinterpret_cast<__m128i*>(o + 4), b);
    }
}
inline bool grouped8_avx512(const float* w, uint8_t* out) {
    for (int g = 0; g < 4; ++g) {
        __m512 v[4], lo, hi;
        for (int i = 0; i < 4; ++i) v[i] = _mm512_loadu_ps(w + 64 * g + 16 * i);
        lo = _mm512_min_ps(_mm512_min_ps(v[0], v[1]), _mm512_min_ps(v[2], v[3]));
        hi = _mm512_max_ps(_mm512_max_ps(v[0], v[1]), _mm512_max_ps(v[2], v[3]));
        const float zp = _mm512_reduce_min_ps(lo), sc = _mm512_reduce_max_ps(hi) - zp;
        if (zp == 0.0f) return false;                                  // which of several zeros is the first: encode_block finds it
        uint8_t* o = out + g * 68;
        put16(o, to_half(zp));
        put16(o + 2, to_half(sc));
        for (int i = 0; i < 4; ++i) {
            const __m512 r = _mm512_mul_ps(_mm512_div_ps(_mm512_sub_ps(v[i], _mm512_set1_ps(zp)), _mm512_set1_ps(sc)), _mm512_set1_ps(255.0f));
            const __m512i k = _mm512_cvttps_epi32(r);
            const __mmask16 half = _mm512_cmp_ps_mask(_mm512_sub_ps(r, _mm512_cvtepi32_ps(k)), _mm512_set1_ps(0.5f), _CMP_GE_OQ);
            const __m128i b = _mm512_cvtusepi32_epi8(_mm512_mask_add_epi32(k, half, k, _mm512_set1_epi32(1)));
            _mm_storeu_si128(reinterpret_cast<__m128i*>(o + 4 + 16 * i), sc == 0.0f ? _mm_setzero_si128() : b);
        }
    }
    return true;
}
#pragma clang attribute pop

template <int BITS>
OIL_INLINE uint32_t level_code(float v) {
    if constexpr (BITS == 8) {
        const float lo = v < 8.0f ? v : 8.0f, c = -8.0f < lo ? lo : -8.0f;
        const float r = (c + 8.0f) * 255.0f / 16.0f;                   // lround: halves away from zero, r >= 0
        const int k = int(r);
        return uint32_t(k + (r - float(k) >= 0.5f ? 1 : 0));
    } else {
        uint32_t q = 0;
        if constexpr (BITS == 4) for (float t : kT4) q += v >= t ? 1u : 0u;
        else for (float t : kT2) q += v >= t ? 1u : 0u;
        return q;
    }
}

// codes (one per byte, `n` of them, n * BITS a multiple of 8) -> bytes, first code in the low bits
template <int BITS>
OIL_INLINE void pack_codes(const uint8_t* c, int n, uint8_t* out) {
    if constexpr (BITS == 8) std::memcpy(out, c, size_t(n));
    else if constexpr (BITS == 4) for (int i = 0; i < n / 2; ++i) out[i] = uint8_t(c[2 * i] | c[2 * i + 1] << 4);
    else for (int i = 0; i < n / 4; ++i) out[i] = uint8_t(c[4 * i] | c[4 * i + 1] << 2 | c[4 * i + 2] << 4 | c[4 * i + 3] << 6);
}

// WIDE: the processor has AVX-512
template <int BITS, bool WIDE>
OIL_INLINE void full_lattice(const float* w, double sum_sq, uint8_t* out) {
    const float scale = float(std::sqrt(sum_sq / 256.0));
    put16(out, to_half(scale));
    alignas(64) uint8_t code[256], dense[256];
    if constexpr (WIDE && BITS == 8) {
        if (scale > 1e-12f) { codes8_avx512(w, scale, out + 2); return; }
    }
    if (scale <= 1e-12f) {
        const uint32_t q = level_code<BITS>(0.0f);
        for (int i = 0; i < 256; ++i) code[i] = uint8_t(q);
    } else {
        bool done = false;
        if constexpr (WIDE && BITS == 4) done = codes_avx512(w, scale, kT4, code);
        if constexpr (WIDE && BITS == 2) done = codes_avx512(w, scale, kT2, code);
        if (!done) for (int i = 0; i < 256; ++i) code[i] = uint8_t(level_code<BITS>(w[i] / scale));
    }
    if constexpr (WIDE && BITS != 8) {
        pack_lattice_avx512<BITS>(code, out + 2);
        return;
    }
    // 16 / BITS weights, the last of every 16 * BITS, have no code: their bits hold the scale
    constexpr int RUN = 16 * BITS;
    for (int r = 0; r < 256 / RUN; ++r) std::memcpy(dense + r * (RUN - 1), code + r * RUN, RUN - 1);
    pack_codes<BITS>(dense, 256 - 256 / RUN, out + 2);
}

template <int BITS>
OIL_INLINE bool full_grouped(const float* w, uint8_t* out) {
    float zp[4], sc[4];
    if constexpr (BITS == 8) {
        for (int g = 0; g < 4; ++g) {
            float lo = w[g * 64], hi = lo;
            for (int i = 1; i < 64; ++i) { const float x = w[g * 64 + i]; lo = x < lo ? x : lo; hi = x > hi ? x : hi; }
            if (lo == 0.0f) return false;                              // which of several zeros is the first: encode_block finds it
            zp[g] = lo;
            sc[g] = hi - lo;
        }
    } else {
        double mu[4] = {0, 0, 0, 0}, ss[4] = {0, 0, 0, 0};
        for (int i = 0; i < 64; ++i)
            for (int g = 0; g < 4; ++g) mu[g] += w[g * 64 + i];
        for (int g = 0; g < 4; ++g) mu[g] /= 64.0;
        for (int i = 0; i < 64; ++i)
            for (int g = 0; g < 4; ++g) { const double d = double(w[g * 64 + i]) - mu[g]; ss[g] = std::fma(d, d, ss[g]); }
        for (int g = 0; g < 4; ++g) { zp[g] = float(mu[g]); sc[g] = ss[g] > 0.0 ? float(std::sqrt(ss[g] / 64.0)) : 0.0f; }
    }
    constexpr int GROUP = 4 + 8 * BITS;
    for (int g = 0; g < 4; ++g) {
        uint8_t* o = out + g * GROUP;
        put16(o, to_half(zp[g]));
        put16(o + 2, to_half(sc[g]));
        alignas(64) uint8_t code[64];
        if (sc[g] == 0.0f) {
            std::memset(code, 0, sizeof code);
        } else if constexpr (BITS == 8) {
            for (int i = 0; i < 64; ++i) {
                const float r = (w[g * 64 + i] - zp[g]) / sc[g] * 255.0f;
                const int k = int(r), q = k + (r - float(k) >= 0.5f ? 1 : 0);
                code[i] = uint8_t(q > 255 ? 255 : q);
            }
        } else {
            for (int i = 0; i < 64; ++i) code[i] = uint8_t(level_code<BITS>(float((double(w[g * 64 + i]) - zp[g]) / double(sc[g]))));
        }
        pack_codes<BITS>(code, 64, o + 4);
    }
    return true;
}

OIL_INLINE uint32_t sign_bits(const float* w, int n) {                 // n <= 32
    uint32_t m = 0;
    for (int i = 0; i < n; ++i) m |= (w[i] >= 0.0f ? 1u : 0u) << i;
    return m;
}

// the largest magnitude of 256 weights as a bit pattern; the vector code takes it up to 1.6e29
constexpr uint32_t kLargestBits = 0x70000000u;
OIL_INLINE uint32_t largest_bits(const float* w) {
    uint32_t top = 0;
    for (int i = 0; i < 256; ++i) { uint32_t b; std::memcpy(&b, w + i, 4); b &= 0x7FFFFFFFu; top = b > top ? b : top; }
    return top;
}

// One full block; `sum_sq` is its sum of squares where the format is scaled by the block's RMS.  False: not covered
// here, encode_block takes it.
template <bool WIDE>
OIL_INLINE bool encode_full(int fmt, const float* w, double sum_sq, uint8_t* out) {
    if (largest_bits(w) > kLargestBits) return false;
    switch (fmt) {
        case OILHIP_OIL2: full_lattice<2, WIDE>(w, sum_sq, out); return true;
        case OILHIP_OIL4: full_lattice<4, WIDE>(w, sum_sq, out); return true;
        case OILHIP_OIL8: full_lattice<8, WIDE>(w, sum_sq, out); return true;
        case OILHIP_OIL2_GRP: if constexpr (!WIDE) return full_grouped<2>(w, out); else return false;      // (WIDE: encode_range takes four blocks' groups side by side)
        case OILHIP_OIL4_GRP: if constexpr (!WIDE) return full_grouped<4>(w, out); else return false;
        case OILHIP_OIL8_GRP: if constexpr (!WIDE) return full_grouped<8>(w, out); else return grouped8_avx512(w, out);
        case OILHIP_OIL1: {
            if constexpr (WIDE) { means_avx512(w, out); return true; }
            double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            for (int i = 0; i < 32; ++i)
                for (int r = 0; r < 8; ++r) s[r] += w[r * 32 + i];
            for (int r = 0; r < 8; ++r) put16(out + 2 * r, to_half(float(s[r] / 32.0)));
            return true;
        }
        case OILHIP_SPARK_Q0: {
            if constexpr (WIDE) { spark_avx512(w, out); return true; }
            double s[8];
            square_sums<8, 32>(w, s);
            for (int r = 0; r < 8; ++r) {
                const uint32_t m = sign_bits(w + 32 * r, 32);
                put16(out + 6 * r, to_half(float(std::sqrt(s[r] / 32.0))));
                std::memcpy(out + 6 * r + 2, &m, 4);
            }
            return true;
        }
        case OILHIP_OIL1_GRP: {                                        // a scale, then 15 signs of every 16 weights
            uint64_t word = to_half(float(std::sqrt(sum_sq / 256.0)));
            int held = 16;
            for (int r = 0; r < 16; ++r) {
                word |= uint64_t(sign_bits(w + 16 * r, 15)) << held;
                held += 15;
                if (held >= 32) { const uint32_t lo = uint32_t(word); std::memcpy(out, &lo, 4); out += 4; word >>= 32; held -= 32; }
            }
            return true;
        }
        default: return false;
    }
}

// Blocks [b0, b1) into payload + blocks[b].cb_off; only the last block of a tensor can be shorter than 256.
template <bool WIDE>
OIL_INLINE void encode_range(const uint8_t* fmts, const float* w, uint64_t numel, const oilhip_block_t* blocks, uint8_t* payload,
                             uint32_t b0, uint32_t b1) {
    constexpr uint32_t SIDE = WIDE ? 16 : 8;                           // blocks whose sums run side by side
    auto encode_plain = [&](uint32_t b) {                              // one channel is empty in every format: both may point at the block's place
        uint8_t* out = payload + blocks[b].cb_off;
        size_t il = 0, cl = 0;
        encode_block(fmts[b], {w + uint64_t(b) * 256, size_t(std::min<uint64_t>(256, numel - uint64_t(b) * 256))}, out, il, out, cl);
    };
    const uint32_t whole = uint32_t(std::min<uint64_t>(b1, numel / 256));
    if (whole < b1) encode_plain(whole);                               // the tensor's last block, shorter than the others
    for (uint32_t b = b0; b < whole; b += SIDE) {
        const uint32_t nb = std::min(SIDE, whole - b);
        auto scaled_by_rms = [](uint8_t f) { return f == OILHIP_OIL2 || f == OILHIP_OIL4 || f == OILHIP_OIL8 || f == OILHIP_OIL1_GRP; };
        double s[SIDE] = {};
        bool scaled = false;
        for (uint32_t j = 0; j < nb; ++j) scaled |= scaled_by_rms(fmts[b + j]);
        if (scaled) {
            if (nb < SIDE) for (uint32_t j = 0; j < nb; ++j) square_sums<1, 256>(w + uint64_t(b + j) * 256, s + j);
            else if constexpr (WIDE) run_sums_avx512<SIDE / 8, 256>(w + uint64_t(b) * 256, s);
            else square_sums<SIDE, 256>(w + uint64_t(b) * 256, s);
        }
        float zp[WIDE ? SIDE : 1][4], sc[WIDE ? SIDE : 1][4];          // of the 2- and 4-bit groups, block by block of those formats
        uint32_t grouped = 0;
        if constexpr (WIDE) {
            const float* block[SIDE + 3];
            uint32_t n = 0;
            for (uint32_t j = 0; j < nb; ++j)
                if (fmts[b + j] == OILHIP_OIL2_GRP || fmts[b + j] == OILHIP_OIL4_GRP) block[n++] = w + uint64_t(b + j) * 256;
            for (uint32_t j = n; n && j < (n + 3) / 4 * 4; ++j) block[j] = block[n - 1];
            for (uint32_t j = 0; j < n; j += 4) {
                float z[4][4], c[4][4];
                moments_avx512({block[j], block[j + 1], block[j + 2], block[j + 3]}, z, c);
                std::memcpy(zp[j], z, sizeof z);
                std::memcpy(sc[j], c, sizeof c);
            }
        }
        for (uint32_t j = 0; j < nb; ++j) {
            const uint64_t at = uint64_t(b + j) * 256;
            uint8_t* out = payload + blocks[b + j].cb_off;
            // the block as far behind it, while this one is worked on
            if (WIDE && at + (SIDE + 1) * 256 <= numel) for (int i = 0; i < 16; ++i) __builtin_prefetch(w + at + SIDE * 256 + 16 * i);
            const int fmt = fmts[b + j];
            if constexpr (WIDE) {
                if (fmt == OILHIP_OIL2_GRP || fmt == OILHIP_OIL4_GRP) {
                    const uint32_t g = grouped++;
                    if (largest_bits(w + at) > kLargestBits) encode_plain(b + j);
                    else if (fmt == OILHIP_OIL2_GRP) grouped_avx512<2>(w + at, zp[g], sc[g], out);
                    else grouped_avx512<4>(w + at, zp[g], sc[g], out);
                    continue;
                }
            }
            if (!encode_full<WIDE>(fmt, w + at, s[j], out)) encode_plain(b + j);
        }
    }
}

using RangeFn = void (*)(const uint8_t*, const float*, uint64_t, const oilhip_block_t*, uint8_t*, uint32_t, uint32_t);
OIL_AVX512
void encode_range_avx512(const uint8_t* f, const float* w, uint64_t n, const oilhip_block_t* b, uint8_t* p, uint32_t b0, uint32_t b1) { encode_range<true>(f, w, n, b, p, b0, b1); }
__attribute__((target("avx2,fma")))
void encode_range_avx2(const uint8_t* f, const float* w, uint64_t n, const oilhip_block_t* b, uint8_t* p, uint32_t b0, uint32_t b1) { encode_range<false>(f, w, n, b, p, b0, b1); }
void encode_range_base(const uint8_t* f, const float* w, uint64_t n, const oilhip_block_t* b, uint8_t* p, uint32_t b0, uint32_t b1) { encode_range<false>(f, w, n, b, p, b0, b1); }

RangeFn range_fn() {
    if (__builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") && __builtin_cpu_supports("avx512dq") && __builtin_cpu_supports("avx512vl"))
        return encode_range_avx512;
    return __builtin_cpu_supports("avx2") && __builtin_cpu_supports("fma") ? encode_range_avx2 : encode_range_base;
}

// Threads for a tensor when the caller names no number: those this process may run on, each with enough work to pay for
// being started.
int auto_threads(uint64_t numel) {
    cpu_set_t set;
    const int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : int(std::max(1u, std::thread::hardware_concurrency()));
    return int(std::clamp<uint64_t>(numel / kWeightsPerThread, 1, uint64_t(std::min(cpus, kMaxThreads))));
}

}  // namespace

extern "C" {

size_t oilhip_payload_bound(int fmt, int n) { return payload_bound(fmt, n); }

int oilhip_quantize_block(int fmt, const float* w, int n, uint8_t* idx, size_t idx_cap, size_t* idx_len,
                          uint8_t* cb, size_t cb_cap, size_t* cb_len) {
    if (!w || n <= 0 || !idx_len || !cb_len) return oilhip::fail(OILHIP_E_ARG, "quantize_block: bad arguments");
    if (fmt < 0 || fmt >= OILHIP_NUM_FORMATS) return oilhip::fail(OILHIP_E_ARG, "quantize_block: unknown format");
    const size_t need = payload_bound(fmt, n);
    if (fmt == OILHIP_OIL1 ? (cb_cap < need || !cb) : (need > 0 && (idx_cap < need || !idx)))
        return oilhip::fail(OILHIP_E_ARG, "quantize_block: output buffer too small");
    encode_block(fmt, {w, size_t(n)}, idx, *idx_len, cb, *cb_len);
    return OILHIP_OK;
}

int oilhip_quantize_tensor(const uint8_t* fmts, uint32_t nblocks, const float* w, uint64_t numel,
                           uint8_t* payload, uint64_t cap, oilhip_block_t* blocks, uint64_t* total, int threads) {
    if (!fmts || !w || !total || nblocks == 0) return oilhip::fail(OILHIP_E_ARG, "quantize_tensor: bad arguments");
    if (uint64_t(nblocks) * 256 < numel || uint64_t(nblocks - 1) * 256 >= numel)
        return oilhip::fail(OILHIP_E_ARG, "quantize_tensor: nblocks does not match numel");
    if (threads <= 0) threads = auto_threads(numel);
    threads = int(std::min<uint32_t>(uint32_t(std::min(threads, 64)), nblocks));
    const uint32_t chunk = (nblocks + uint32_t(threads) - 1) / uint32_t(threads);
    // how many blocks of each format there are, up to the end of each thread's share
    uint64_t count[256] = {};
    std::vector<std::array<uint32_t, OILHIP_NUM_FORMATS>> upto;
    for (uint64_t b = 0; b < nblocks;) {
        uint32_t part[4][256] = {};                                    // four tables: neighbours of one format would wait for each other
        const uint64_t end = std::min<uint64_t>(nblocks, b + chunk);
        for (; b + 4 <= end; b += 4) { ++part[0][fmts[b]]; ++part[1][fmts[b + 1]]; ++part[2][fmts[b + 2]]; ++part[3][fmts[b + 3]]; }
        for (; b < end; ++b) ++part[0][fmts[b]];
        for (int f = 0; f < 256; ++f) count[f] += uint64_t(part[0][f]) + part[1][f] + part[2][f] + part[3][f];
        upto.emplace_back();
        for (int f = 0; f < OILHIP_NUM_FORMATS; ++f) upto.back()[size_t(f)] = uint32_t(count[f]);
    }
    for (int f = OILHIP_NUM_FORMATS; f < 256; ++f)
        if (count[f]) return oilhip::fail(OILHIP_E_ARG, "quantize_tensor: unknown format");
    const bool sparse = count[OILHIP_SPARK_SPARSE] || count[OILHIP_SPARK_SPARSE_GRP];     // an all-zero block is shorter there
    size_t widest = 0, full[OILHIP_NUM_FORMATS];
    uint64_t bound = 0;
    for (int f = 0; f < OILHIP_NUM_FORMATS; ++f) {
        full[f] = payload_bound(f, 256);
        if (count[f]) widest = std::max(widest, full[f]);
        bound += count[f] * ((full[f] + 15) & ~size_t(15));
    }
    if (!payload) { *total = bound; return OILHIP_OK; }
    if (!blocks) return oilhip::fail(OILHIP_E_ARG, "quantize_tensor: blocks is null");
    // a thread starts half of the others of its share first: sixteen are running after four starts one behind the other instead of fifteen
    auto in_chunks = [&](auto&& work) {
        auto share = [&](auto&& self, int t0, int t1) -> void {        // threads t0 .. t1 - 1
            std::vector<std::thread> others;
            for (; t1 - t0 > 1; t1 = t0 + (t1 - t0 + 1) / 2) {
                const int mid = t0 + (t1 - t0 + 1) / 2;
                if (uint64_t(mid) * chunk < nblocks) others.emplace_back([&self, mid, t1] { self(self, mid, t1); });
            }
            const uint64_t b0 = uint64_t(t0) * chunk;
            if (b0 < nblocks) work(uint32_t(b0), uint32_t(std::min<uint64_t>(nblocks, b0 + chunk)));
            for (auto& th : others) th.join();
        };
        share(share, 0, threads);
    };
    auto weights_of = [&](uint32_t b) { return uint32_t(std::min<uint64_t>(256, numel - uint64_t(b) * 256)); };
    uint64_t off = 0;
    if (!sparse) {
        // every block's size follows from its format and length, so the blocks are encoded where they belong; a full block's is a multiple of 16
        std::vector<uint64_t> start(upto.size() + 1, 0);
        for (size_t c = 0; c < upto.size(); ++c)
            for (size_t f = 0; f < OILHIP_NUM_FORMATS; ++f) start[c + 1] += uint64_t(upto[c][f]) * full[f];
        const uint32_t n_last = weights_of(nblocks - 1);
        off = start.back();
        if (n_last < 256) off += payload_bound(fmts[nblocks - 1], int(n_last)) - full[fmts[nblocks - 1]];
        if (off > cap) return oilhip::fail(OILHIP_E_ARG, "quantize_tensor: payload buffer too small");
        const RangeFn encode = range_fn();
        in_chunks([&](uint32_t b0, uint32_t b1) {
            uint64_t at = start[b0 / chunk];
            for (uint32_t b = b0; b < b1; ++b) {
                const uint32_t n = weights_of(b), bytes = uint32_t(n == 256 ? full[fmts[b]] : payload_bound(fmts[b], int(n)));
                const uint32_t cl = fmts[b] == OILHIP_OIL1 ? bytes : 0u;
                blocks[b] = oilhip_block_t{at, at + cl, cl, bytes - cl, n, fmts[b], {0, 0, 0}};
                at += bytes;
            }
            encode(fmts, w, numel, blocks, payload, b0, b1);
        });
        *total = off;
        return OILHIP_OK;
    }
    struct Enc { uint32_t il, cl; };
    const size_t stride = widest + 32;             // [32 bytes codebook channel][index channel]
    std::vector<uint8_t> tmp(size_t(nblocks) * stride);
    std::vector<Enc> len(nblocks);
    in_chunks([&](uint32_t b0, uint32_t b1) {
        for (uint32_t b = b0; b < b1; ++b) {
            size_t il = 0, cl = 0;
            uint8_t* slot = tmp.data() + size_t(b) * stride;
            encode_block(fmts[b], {w + uint64_t(b) * 256, weights_of(b)}, slot + 32, il, slot, cl);
            len[b] = {uint32_t(il), uint32_t(cl)};
        }
    });
    for (uint32_t b = 0; b < nblocks; ++b) {
        off = (off + 15) & ~uint64_t(15);
        if (off + len[b].cl + len[b].il > cap) return oilhip::fail(OILHIP_E_ARG, "quantize_tensor: payload buffer too small");
        const uint8_t* slot = tmp.data() + size_t(b) * stride;
        std::memcpy(payload + off, slot, len[b].cl);
        std::memcpy(payload + off + len[b].cl, slot + 32, len[b].il);
        blocks[b] = oilhip_block_t{off, off + len[b].cl, len[b].cl, len[b].il, weights_of(b), fmts[b], {0, 0, 0}};
        off += len[b].cl + len[b].il;
    }
    *total = off;
    return OILHIP_OK;
}

}  // extern "C"
