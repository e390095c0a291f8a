// loss_device.h — the training loss of one ray and the count of valid rays, for the loss's
// own kernels and for the integrator that takes the loss in its stride.
#pragma once
#include "ngp_common.h"

namespace ngp {

// The valid rays among n flags, by one workgroup of kThreads (the batch's flags are a few
// hundred KB; 16 bytes per load, `wsum` one word per wavefront).  Valid in thread 0.
template <int kThreads>
__device__ __forceinline__ uint32_t count_flags(uint32_t n, const bool *__restrict__ flags, uint32_t *wsum) {
    const uint8_t *f = reinterpret_cast<const uint8_t *>(flags);
    uint32_t c = 0;
    const uint32_t n16 = (reinterpret_cast<uintptr_t>(f) & 15u) == 0 ? n / 16 : 0;
    // eight 16-byte loads in flight per thread (one round for 2^17 flags; sixteen do not
    // fit the registers of a workgroup of 1024 and took 45 us instead of 10)
    constexpr uint32_t kU = 8;
    for (uint32_t q0 = 0; q0 < n16; q0 += kU * kThreads) {
        uint4 v[kU];
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
            const uint32_t q = q0 + u * kThreads + threadIdx.x;
            v[u] = q < n16 ? reinterpret_cast<const uint4 *>(f)[q] : make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
            // bools are 0 or 1: a word's set bits are its true bytes
            c += (uint32_t)(__popc(v[u].x) + __popc(v[u].y) + __popc(v[u].z) + __popc(v[u].w));
        }
    }
    for (uint32_t i = 16 * n16 + threadIdx.x; i < n; i += kThreads) c += f[i] ? 1u : 0u;
    c = wave_sum(c);
    if (lane_id() == 0) wsum[threadIdx.x / kWave] = c;
    __syncthreads();
    uint32_t t = 0;
    if (threadIdx.x == 0)
        for (int w = 0; w < kThreads / kWave; ++w) t += wsum[w];
    return t;
}

// optax.huber_loss(pred, target, delta): 0.5 e^2 if |e| <= delta else delta (|e| - delta/2),
// averaged over the three channels and nv rays; `grad` is its gradient times ls.
__device__ __forceinline__ float huber_ray(float r, float g, float b, const float *__restrict__ gt, float delta, float nv,
                                           float ls, float4 &grad) {
    const float e[3] = {r - gt[0], g - gt[1], b - gt[2]};
    float h = 0.0f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float ae = fabsf(e[c]);
        h += ae <= delta ? 0.5f * e[c] * e[c] : delta * (ae - 0.5f * delta);
    }
    const float s = 1.0f / (3.0f * nv);
    grad = make_float4((fminf(fmaxf(e[0], -delta), delta) * s) * ls, (fminf(fmaxf(e[1], -delta), delta) * s) * ls,
                       (fminf(fmaxf(e[2], -delta), delta) * s) * ls, 0.0f);
    return (h / 3.0f) / nv;
}

}  // namespace ngp
