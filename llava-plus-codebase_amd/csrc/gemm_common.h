// Pieces shared by the prefill GEMM kernels (gemm.hip, gemm8p.hip, gemm4w.h): MFMA wrappers, the LDS tile image / swizzle, and the
// register epilogue (bias / activation / SiLU·mul / residual, 8-byte packed stores).
#pragma once
#include "common.h"
#include "kernels.h"

namespace lmx {

// ---------------------------------------------------------------------------------------------
// MFMA wrappers
// ---------------------------------------------------------------------------------------------
template <typename T> struct Mfma32x32x16;
template <> struct Mfma32x32x16<bf16_t> {
    static __device__ __forceinline__ f32x16 run(const uint4& a, const uint4& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_v, a), __builtin_bit_cast(bf16x8_v, b), c, 0, 0, 0);
    }
};
template <> struct Mfma32x32x16<f16_t> {
    static __device__ __forceinline__ f32x16 run(const uint4& a, const uint4& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_v, a), __builtin_bit_cast(f16x8_v, b), c, 0, 0, 0);
    }
};

// ---------------------------------------------------------------------------------------------
// shared epilogue math
// ---------------------------------------------------------------------------------------------
template <typename T = bf16_t> __device__ __forceinline__ float apply_act(float v, int act) {
    if (act == kActQuickGelu) return act_quick_gelu<T>(v);
    if (act == kActGeluErf) return act_gelu_erf(v);
    return v;
}

// the same on N values of one output row, with the choice made ONCE: inlined per element, the erf and exp code of the branches not taken lies between any two elements and
// every element jumps over it into an instruction-cache line of its own
template <int N> __device__ __forceinline__ void apply_act_n(float (&v)[N], int act) {
    if (act == kActNone) return;
    if (act == kActQuickGelu) {
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = act_quick_gelu(v[e]);
    } else if (act == kActGeluErf) {
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = act_gelu_erf(v[e]);
    }
}

template <typename T> __device__ __forceinline__ void store4(T* p, const float (&v)[4]);
template <> __device__ __forceinline__ void store4<bf16_t>(bf16_t* p, const float (&v)[4]) {
    uint2 u; u.x = pack2<bf16_t>(v[0], v[1]); u.y = pack2<bf16_t>(v[2], v[3]);
    *reinterpret_cast<uint2*>(p) = u;
}
template <> __device__ __forceinline__ void store4<f16_t>(f16_t* p, const float (&v)[4]) {
    uint2 u; u.x = pack2<f16_t>(v[0], v[1]); u.y = pack2<f16_t>(v[2], v[3]);
    *reinterpret_cast<uint2*>(p) = u;
}
template <> __device__ __forceinline__ void store4<float>(float* p, const float (&v)[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
template <typename T> __device__ __forceinline__ void load4(const T* p, float (&v)[4]);
template <> __device__ __forceinline__ void load4<bf16_t>(const bf16_t* p, float (&v)[4]) {
    uint2 u = *reinterpret_cast<const uint2*>(p);
    v[0] = unpack_lo<bf16_t>(u.x); v[1] = unpack_hi<bf16_t>(u.x); v[2] = unpack_lo<bf16_t>(u.y); v[3] = unpack_hi<bf16_t>(u.y);
}
template <> __device__ __forceinline__ void load4<f16_t>(const f16_t* p, float (&v)[4]) {
    uint2 u = *reinterpret_cast<const uint2*>(p);
    v[0] = unpack_lo<f16_t>(u.x); v[1] = unpack_hi<f16_t>(u.x); v[2] = unpack_lo<f16_t>(u.y); v[3] = unpack_hi<f16_t>(u.y);
}
template <> __device__ __forceinline__ void load4<float>(const float* p, float (&v)[4]) {
    float4 u = *reinterpret_cast<const float4*>(p);
    v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
}

// ---------------------------------------------------------------------------------------------
// 16-bit MFMA GEMM
// ---------------------------------------------------------------------------------------------
constexpr int GEMM_BK = 64;               // K elements per stage = 128 bytes per row
constexpr int GEMM_ROWB = GEMM_BK * 2;    // row pitch in LDS (bytes)

// LDS byte offset of 16-byte chunk `chunk` (0..7) of tile row `row`: rows 2r,2r+1 share a 256-B bank row, and
// the 8 chunk slots are XORed with (row>>1)&7 so 16 consecutive rows reading the same logical chunk hit 16
// distinct 16-B slots (ds_read_b128 lane groups are 16 lanes wide).
__device__ __forceinline__ int lds_chunk_off(int row, int chunk) {
    return row * GEMM_ROWB + (((chunk ^ (row >> 1)) & 7) << 4);
}

// ---------------------------------------------------------------------------------------------
// shared epilogue: acc[i][j][4q+e] = C[m = m_base + j*32 + l31][n = n_base + i*32 + 8q + 4hi + e]
// (weight fragment = MFMA A operand, so a lane owns 4 consecutive n of one row m per accumulator quad)
//
// Written for SHORT CODE.  A workgroup of a big tile runs this once, with instructions it has not fetched before, and waits for every cache line of them: unrolled over all
// accumulators, with the activation's branches around every element, it took 54,500 cycles behind the last MFMA of a 256 x 256 tile whatever K (24 - 26 us of the 55 us of
// 4096 x 4096 x 1024, of the 141 us of 4096 x 4096 x 4096), stores in row order or not; now 9,500 cycles, 5 us (gated 15,700; with a residual 19,800).  So a wave turns its tile into row order through LDS of its own, 32 rows at a
// time (pitch 32 NTL + 4 floats: 16-byte writes and reads without bank conflicts, no barrier), and one rolled body does bias, gating, activation, residual, rounding and
// the 8-byte stores on row pieces (4 rows x 128 bytes a store instruction at NTL = 2).
// Values and rounding: bias -> activation -> residual -> one rounding, fp32 until then.
// ---------------------------------------------------------------------------------------------
template <int NTL> constexpr int epilogue_pitch() { return 32 * NTL + 4; }
template <int NTL> constexpr int epilogue_wave_bytes() { return 32 * epilogue_pitch<NTL>() * 4; }       // LDS a wave needs: the caller's operand buffers, dead by then

// F32: the instantiation whose output is fp32 with an optional soft cap (GemmArgs::c_f32); its own template so that the hot kernels do not carry the branch
template <typename T, int MT, int NTL, bool F32 = false>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& a, f32x16 (&acc)[NTL][MT], int m_base, int n_base, int lane, char* wave_lds) {
    constexpr int PITCH = epilogue_pitch<NTL>();
    T* __restrict__ C = reinterpret_cast<T*>(a.C);
    const T* __restrict__ bias = reinterpret_cast<const T*>(a.bias);
    const T* R = reinterpret_cast<const T*>(a.R);
    const int act = a.act;
    const int hi = lane >> 5, l31 = lane & 31;
    float* img = reinterpret_cast<float*>(wave_lds);
    const bool gated = NTL % 2 == 0 && act_gated(act);
    const int pk_q = a.pk_kc ? a.pk_heads * a.pk_D : 0x7fffffff;         // first column that leaves through the K / V^T pack (CLIP q|k|v)

    // plain: LPR lanes a row of 32 NTL columns; gated: fused columns are interleaved [32 gate | 32 up] per 64, half as many lanes a row of 16 NTL outputs
    constexpr int LPR = 8 * NTL, RPP = 64 / LPR, NP = 32 / RPP;          // lanes of a row, rows of a pass, passes
    const int c = (lane % LPR) * 4, n = n_base + c;
    const bool n_in = n < a.N;
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias && n_in && !gated) load4<T>(bias + n, b);
    uint2 rq[NP], rn[NP];                                                // residual rows, requested one 32-row block ahead (C may alias R: a block's stores touch none of the next's rows)
    auto want = [&](uint2 (&d)[NP], int j) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int m = m_base + j * 32 + p * RPP + lane / LPR;
            d[p] = m < a.M && n_in && n < pk_q ? *reinterpret_cast<const uint2*>(R + (size_t)m * a.ldr + n) : uint2{0u, 0u};
        }
    };
    if (R) want(rn, 0);
#pragma unroll 1
    for (int j = 0; j < MT; ++j) {
        const int m0 = m_base + j * 32;
        if (m0 >= a.M) break;
        if (R) {
#pragma unroll
            for (int p = 0; p < NP; ++p) rq[p] = rn[p];
            if (j + 1 < MT) want(rn, j + 1);
        }
#pragma unroll
        for (int jj = 0; jj < MT; ++jj)
            if (jj == j) {
#pragma unroll
                for (int i = 0; i < NTL; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<float4*>(img + l31 * PITCH + i * 32 + 8 * q + 4 * hi) =
                            make_float4(acc[i][jj][4 * q], acc[i][jj][4 * q + 1], acc[i][jj][4 * q + 2], acc[i][jj][4 * q + 3]);
            }
        __builtin_amdgcn_wave_barrier();
        if (gated) {
            constexpr int GPR = 4 * NTL;                                 // lanes of a row of 16 NTL outputs
            const int o = (lane % GPR) * 4, f = (o >> 5) * 64 + (o & 31);
            float bg[4] = {0.f, 0.f, 0.f, 0.f}, bu[4] = {0.f, 0.f, 0.f, 0.f};
            if (bias && n_base + f < a.N) { load4<T>(bias + n_base + f, bg); load4<T>(bias + n_base + f + 32, bu); }
#pragma unroll
            for (int p = 0; p < GPR / 2; ++p) {
                const int r = p * (64 / GPR) + lane / GPR;
                const float4 g = *reinterpret_cast<const float4*>(img + r * PITCH + f), u = *reinterpret_cast<const float4*>(img + r * PITCH + f + 32);
                float v[4] = {g.x + bg[0], g.y + bg[1], g.z + bg[2], g.w + bg[3]};
                const float w[4] = {u.x + bu[0], u.y + bu[1], u.z + bu[2], u.w + bu[3]};
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = gate_mul(act, v[e], w[e]);
                if (m0 + r < a.M && n_base + f < a.N) store4<T>(C + (size_t)(m0 + r) * a.ldc + n_base / 2 + o, v);
            }
        } else {
            float4 t[NP];
#pragma unroll
            for (int p = 0; p < NP; ++p) t[p] = *reinterpret_cast<const float4*>(img + (p * RPP + lane / LPR) * PITCH + c);
#pragma unroll
            for (int p = 0; p < NP; ++p) t[p] = make_float4(t[p].x + b[0], t[p].y + b[1], t[p].z + b[2], t[p].w + b[3]);
            if (act != kActNone) {
#pragma unroll 1
                for (int p = 0; p < NP; ++p)
#pragma unroll
                    for (int pp = 0; pp < NP; ++pp)
                        if (pp == p) {
                            float v[4] = {t[pp].x, t[pp].y, t[pp].z, t[pp].w};
                            apply_act_n<4>(v, act);
                            t[pp] = make_float4(v[0], v[1], v[2], v[3]);
                        }
            }
            if (R) {
#pragma unroll
                for (int p = 0; p < NP; ++p)
                    t[p] = make_float4(t[p].x + unpack_lo<T>(rq[p].x), t[p].y + unpack_hi<T>(rq[p].x), t[p].z + unpack_lo<T>(rq[p].y), t[p].w + unpack_hi<T>(rq[p].y));
            }
            if constexpr (F32) {
#pragma unroll
                for (int p = 0; p < NP; ++p) t[p] = make_float4(soft_cap(t[p].x, a.cap), soft_cap(t[p].y, a.cap), soft_cap(t[p].z, a.cap), soft_cap(t[p].w, a.cap));
            }
            if (n < pk_q) {
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    const int m = m0 + p * RPP + lane / LPR;
                    const float v[4] = {t[p].x, t[p].y, t[p].z, t[p].w};
                    if (m < a.M && n_in) {
                        if constexpr (F32) store4<float>(reinterpret_cast<float*>(a.C) + (size_t)m * a.ldc + n, v);
                        else store4<T>(C + (size_t)m * a.ldc + n, v);
                    }
                }
            } else if (n_in && n - pk_q < pk_q) {
                const int kcol = n - pk_q, head = kcol / a.pk_D, d = kcol - head * a.pk_D;      // K rows [head][pos][D]
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    const int m = m0 + p * RPP + lane / LPR, pimg = m / a.pk_rows, pos = m - pimg * a.pk_rows;
                    const float v[4] = {t[p].x, t[p].y, t[p].z, t[p].w};
                    if (m < a.M) store4<T>(reinterpret_cast<T*>(a.pk_kc) + pimg * a.pk_img_stride + ((size_t)head * a.pk_spad + pos) * a.pk_D + d, v);
                }
            }
        }
        if (a.pk_kc && m0 + l31 < a.M) {
            // v columns -> V^T [head][d][pos]: a lane owns one row here, so a store instruction makes two 64-byte runs
            const int m = m0 + l31, pimg = m / a.pk_rows, pos = m - pimg * a.pk_rows;
            const int first = 2 * pk_q - n_base, c0 = first > 0 ? first : 0, c1 = a.N - n_base < 32 * NTL ? a.N - n_base : 32 * NTL;
#pragma unroll 1
            for (int cc = c0 + hi; cc < c1; cc += 2) {
                float v[1] = {img[l31 * PITCH + cc] + (bias ? to_f32(bias[n_base + cc]) : 0.f)};
                apply_act_n<1>(v, act);
                const int vcol = n_base + cc - 2 * pk_q;                 // = head * D + d
                reinterpret_cast<T*>(a.pk_vt)[pimg * a.pk_img_stride + (size_t)vcol * a.pk_spad + pos] = from_f32<T>(v[0]);
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}


}  // namespace lmx
