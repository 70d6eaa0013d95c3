// A mixture's choice of experts for one row, by one workgroup: a launch of its own (moe.hip), or one workgroup more in the launch of a parallel layer's mixer, which reads the same
// row and takes as long (delta.hip, latent.hip).
#pragma once
#include "common.h"
#include "kernels.h"

namespace lmx {

constexpr int MOE_MAX_E = 256, MOE_MAX_TOP = 32;

// the `top` largest of z[0, E) (lowest index first among equals) and their softmax, by one wave: an expert's place is the number of experts ahead of it.
// z is padded with -inf to a multiple of 4
__device__ __forceinline__ void pick_top(const float* z, int E, int top, int lane, int* place, int* ids, float* wt) {
    float v[MOE_MAX_E / 64]; int rank[MOE_MAX_E / 64];
    if (lane < top) place[lane] = lane;                      // only non-finite logits leave a place empty
#pragma unroll
    for (int i = 0; i < MOE_MAX_E / 64; ++i) { v[i] = lane + 64 * i < E ? z[lane + 64 * i] : -INFINITY; rank[i] = 0; }
    for (int j = 0; j < E; j += 4) {
        const float4 q = *reinterpret_cast<const float4*>(z + j);
        const float o[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int i = 0; i < MOE_MAX_E / 64; ++i) rank[i] += o[n] > v[i] || (o[n] == v[i] && j + n < lane + 64 * i);
    }
#pragma unroll
    for (int i = 0; i < MOE_MAX_E / 64; ++i) if (lane + 64 * i < E && rank[i] < top) place[rank[i]] = lane + 64 * i;
    __builtin_amdgcn_wave_barrier();
    const int id = lane < top ? place[lane] : 0;
    const float e = lane < top ? expf(z[id] - z[place[0]]) : 0.f;
    const float sum = wave_sum(e);
    if (lane < top) { ids[lane] = id; wt[lane] = e / sum; }
}

inline void check_router(const MoeRouterArgs& a) {
    if (!a.x) return;
    LMX_REQUIRE(a.E >= 1 && a.E <= MOE_MAX_E && a.top >= 1 && a.top <= a.E && a.top <= MOE_MAX_TOP, "moe_router: 1..256 experts, at most 32 of them per row");
    LMX_REQUIRE(a.K % 8 == 0 && a.ldx % 8 == 0 && a.w && a.ids && a.wt, "moe_router: bad arguments");
}

// 64 NW threads: a wave takes two experts at a time, their rows and the input row on their way together
template <typename T, int NW>
__device__ __forceinline__ void moe_router_row(const MoeRouterArgs& a, int row) {
    __shared__ __attribute__((aligned(16))) float z[MOE_MAX_E];
    __shared__ int place[MOE_MAX_TOP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const T* x = reinterpret_cast<const T*>(a.x) + (size_t)row * a.ldx;
    for (int i = tid; i < MOE_MAX_E; i += 64 * NW) if (i >= a.E) z[i] = -INFINITY;
    for (int e = wave; e < a.E; e += 2 * NW) {
        const bool two = e + NW < a.E;
        const T* w = reinterpret_cast<const T*>(a.w) + (size_t)e * a.K;
        const T* w2 = two ? w + (size_t)NW * a.K : w;
        const float b = a.bias ? to_f32(reinterpret_cast<const T*>(a.bias)[e]) : 0.f, b2 = a.bias && two ? to_f32(reinterpret_cast<const T*>(a.bias)[e + NW]) : 0.f;
        float s = 0.f, s2 = 0.f;
#pragma unroll 4
        for (int c = lane * 8; c < a.K; c += 512) {
            float f[8], g[8], v[8]; load8<T>(w + c, f); load8<T>(w2 + c, g); load8<T>(x + c, v);
#pragma unroll
            for (int i = 0; i < 8; ++i) { s = fmaf(f[i], v[i], s); s2 = fmaf(g[i], v[i], s2); }
        }
        s = wave_sum(s); s2 = wave_sum(s2);
        if (lane == 0) { z[e] = s + b; if (two) z[e + NW] = s2 + b2; }
    }
    __syncthreads();
    if (wave == 0) pick_top(z, a.E, a.top, lane, place, a.ids + (size_t)row * a.top, a.wt + (size_t)row * a.top);
}

}  // namespace lmx
