// pack_activations.h -- what the pre-passes of the several-row kernels read: the activation rows, optionally as the caller's SwiGLU product
// or RMSNorm forms them (Qwen35Engine::rmsnorm and mlp_step, src/adapters/tools/qwen35_engine.cpp:39-44,611-621), so that neither is a launch of its own
// (a layer of OIL2 2560 <-> 6400, 14 rows 68.6 -> 64.4 us, registry's mix 1024 <-> 3328, 9 rows 53.9 -> 48.2).  Bound by latency: one load, for the norm
// a walk over the row by every wavefront, and the exchange of a maximum.
#pragma once
#include "oil4_lds.h"

namespace oilhip {

// What the rows are multiplied as: x, silu(x) * x2, or x * (1 + norm_w) / rms(x).
struct Activations {
    const float *x, *x2, *norm_w;
    float* xn;                  // with norm_w: the normalised rows go here as well (optional, laid out like x)
    uint32_t ldx, aligned, inv_form;
};

// this lane's four columns of block `blk` of row `src`
__device__ __forceinline__ void load_activations(const Activations& a, uint32_t src, uint32_t blk, uint32_t bpr, uint32_t lane, float (&v)[4]) {
    const float* row = a.x + (size_t)src * a.ldx;
    const float* p = row + 256u * blk + 4u * lane;
    auto load = [&](const float* q, float (&o)[4]) {
        if (a.aligned) { const float4 f = *reinterpret_cast<const float4*>(q); o[0] = f.x; o[1] = f.y; o[2] = f.z; o[3] = f.w; }
        else { for (int e = 0; e < 4; ++e) o[e] = q[e]; }
    };
    load(p, v);
    if (a.x2) {
        float u[4];
        load(a.x2 + (p - a.x), u);
        // silu(g) * u as ExpertFFN::forward (src/moe_variants.cpp:77-91) or mlp_step (qwen35_engine.cpp:31,37,617) forms it
        for (int e = 0; e < 4; ++e) v[e] = (a.inv_form ? v[e] * (1.0f / (1.0f + expf(-v[e]))) : v[e] / (1.0f + expf(-v[e]))) * u[e];
    } else if (a.norm_w) {
        float s = 0.0f;
        for (uint32_t b = 0; b < bpr; b += 8u) {                           // eight loads in flight; past the end: the last block, counted as 0
            float f[8][4];
#pragma unroll
            for (uint32_t i = 0; i < 8u; ++i) load(row + 256u * (b + i < bpr ? b + i : bpr - 1u) + 4u * lane, f[i]);
#pragma unroll
            for (uint32_t i = 0; i < 8u; ++i)
                s += b + i < bpr ? (f[i][0] * f[i][0] + f[i][1] * f[i][1]) + (f[i][2] * f[i][2] + f[i][3] * f[i][3]) : 0.0f;
        }
        s = oil4::wave_sum(s);
        const float r = 1.0f / sqrtf(s / (float)(256u * bpr) + 1e-6f);
        for (int e = 0; e < 4; ++e) v[e] = v[e] * r * (1.0f + a.norm_w[256u * blk + 4u * lane + e]);
        if (a.xn) {
            float* o = a.xn + (size_t)src * a.ldx + 256u * blk + 4u * lane;
            for (int e = 0; e < 4; ++e) o[e] = v[e];
        }
    }
}

}  // namespace oilhip
