// Four-wave prefill GEMM for gfx950: C[M,N] = act(X[M,K] · W[N,K]ᵀ + bias) (+ residual), 16-bit operands, fp32 accumulate.
//
// Replaces the same torch.nn.Linear calls as gemm.hip (HF5:models/llama/modeling_llama.py:163-176,243-281) for every prompt-sized linear: the decoder's q|k|v, gate|up, o and
// down, the CLIP tower's, the training step's forward and data gradients.
//
// Bound: power in a full round.  With random operands the chip's matrix cores run at the clock their power allows: 4096 x 4096 x 8192, one round of 256 tiles, takes 187 us at 1.85 GHz
// with the matrix cores 76 % busy, the same on zeros 146 us at 2.30 GHz and 78 % (eight waves of 32x32x16: 208 us at 1.63 GHz, 145 at 2.26; by counters).  So a form is as fast as it is
// frugal, and a launch as fast as its tiles divide over the CUs: q|k|v, gate|up and down of a 7B prompt of 1087 rows hold 2.03 .. 2.13 GHz at 59 .. 61 % busy; o, 224 tiles with 0.24 us
// of fixed cost in a K-step of 0.56, is not bound by power: 2.4 GHz at 34 %.  From memory, every XCD's L2 reads X once and the weights once between them: 199 MB at q|k|v are 8 x 8.9 of
// X, 101 of W and 27 of output; 123 at o, 335 at down with its partial tiles; 371 at gate|up, whose second round reads X once more.
// Both decide the shape (4096 x 4096 x 8192, us on random operands / on zeros):
//   * one wave a SIMD with a 128 x 128 piece of the tile: a K-step of 256 x 256 x 64 reads 128 KB of fragments from LDS (eight waves of 128 x 64: 192 KB; LDS is busy
//     in 19 % of the cycles against 30).  204 / 137 with eight waves of v_mfma_f32_32x32x16, 174 / 136 here;
//   * v_mfma_f32_16x16x32, not 32x32x16: 177 / 126 against 192 / 121 without the epilogue.  The larger instruction is the better one on zeros and takes more power on numbers;
//   * both K halves of an accumulator back to back: 178 / 138 -> 174 / 136;
//   * tiles of 32 MB x 32 NB for many MB, NB, because the power limit makes the time of a K-step follow the tile's area (0.12 + 0.018 us x MB NB): whichever divides
//     the problem into the fullest rounds wins (gemm4w_form).
//
// Structure: 4 waves = 2 (M) x 2 (N), wave wm takes the 16-row blocks 2 j + wm (so a ragged last tile leaves both waves the same work), wave wn the columns 16 NB wn .. + 16 NB - 1.
//   * A K-step (64 k) is four phases, one quadrant (half of the wave's row blocks x half of its column blocks) each.  Even K-steps take  X0 Wa, X0 Wb, X1 Wb, X1 Wa  with
//     Wa = W half 0, odd ones with Wa = W half 1: so every phase needs exactly one half-tile that its predecessor did not, and reads it into registers that are free one
//     phase ahead.  The reads sit between the phase's first MFMAs, one for every two, then the DMA instructions.
//   * Operands are staged as half-tiles (X half: the tile's first / second MB0 / MB1 x 32 rows, W half: the first / second NB0 / NB1 x 16 columns of both wave columns) of 64 k in
//     a ring of NR K-steps, as many as 160 KB hold up to four, filled by LDS-DMA (buffer_load_dwordx4 ... lds).  With half-tiles numbered in the order of their first use, h is
//     read in phase h - 2, and phase h stages the half-tile NR K-steps on that takes its slot.  A barrier closes every second phase:
//       RAW  h is read behind the barrier at the end of the last odd phase before h - 2; in front of it every wave has waited until only half-tiles behind h + 1 (h even) or h (odd)
//            are in flight, a compile-time count;
//       WAR  the reads of h were retired (lgkmcnt(0)) in front of the barrier behind phase h - 2 or h - 1; its slot is filled again from phase h on.
//     (Rings of two throughout -> of up to four, inside a prompt: 2308 x 3072 x 1024 24.1 -> 23.2 us, 2308 x 4096 x 1024 37.5 -> 36.8, 2048 x 2048 x 5632 and x 2048 38.8 -> 38.2.)
//   * Behind the last K-step the descriptors are emptied: loads past it read no memory, write zeros to slots that are not read (an odd last K-step is followed by one of zeros)
//     and keep every count.
//   * LDS image of a half-tile: rows of 128 bytes, 16-byte chunk c of row r at chunk c ^ ((r >> 1) & 7); LDS-DMA is lane-linear, so the permutation is on the source address.
//   * Rows beyond M / N are clamped to the last valid row at load time (their accumulators are never stored).
//   * The weight fragment is the MFMA A operand, so a lane owns four consecutive n of one row; v_permlane16_swap makes eight of two blocks, and the rows leave in 16-byte
//     stores straight from the registers: 6 us behind the last MFMA of a full round (its 32 MB of output), 10 through an LDS image in row order or with 8-byte stores.
//   * Gated weights ([32 gate | 32 up] rows): a 16-column block of the tile is 8 gate and 8 up rows of the same outputs, whatever the tile's width.
//   * K slices (S > 1): fp32 partial tiles in accumulator order, plain stores; gemm4w_reduce_kernel, the next launch, adds them in slice order and runs the epilogue.
#pragma once
#include <mutex>
#include <set>

#include "common.h"
#include "kernels.h"
#include "gemm_common.h"

namespace lmx {

namespace {

typedef int v4i_t __attribute__((ext_vector_type(4)));
typedef unsigned frag_t __attribute__((ext_vector_type(4)));

template <int N> struct IC { static constexpr int value = N; };

__device__ __forceinline__ v4i_t make_rsrc(const void* p, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    v4i_t r;
    r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    r.y = __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32));
    r.z = __builtin_amdgcn_readfirstlane((int)bytes);
    r.w = 0x00020000;
    return r;
}

// d += a b on the accumulator registers.  Written out so that the accumulators stay in AGPRs: left to itself the register allocator moves them (and the fragments) back and
// forth between the two files inside the loop.  The wait states in front of the first use and behind the last one are the caller's (mfma_settle).
template <typename T> __device__ __forceinline__ void mfma16(f32x4& d, frag_t a, frag_t b);
template <> __device__ __forceinline__ void mfma16<bf16_t>(f32x4& d, frag_t a, frag_t b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(d) : "v"(a), "v"(b));
}
template <> __device__ __forceinline__ void mfma16<f16_t>(f32x4& d, frag_t a, frag_t b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(d) : "v"(a), "v"(b));
}
// read where it stands: left to itself the compiler copies all accumulators out of their registers ahead of the epilogue's branches, and spills
__device__ __forceinline__ f32x4 from_acc(const f32x4& d) {
    float x, y, z, w;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(d[0])); asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(y) : "a"(d[1]));
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(z) : "a"(d[2])); asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(w) : "a"(d[3]));
    return f32x4{x, y, z, w};
}
__device__ __forceinline__ void mfma_settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// fused column f of a gated tile -> weight row: the tile's 16-column blocks hold 8 gate and 8 up columns of the same outputs, the weight 32 and 32
__device__ __forceinline__ int gated_row(int f) {
    const int j = (f >> 4) * 8 + (f & 7);
    return (j >> 5) * 64 + (j & 31) + ((f & 8) << 2);
}

template <int MB, int NB> struct Shape4w {
    static constexpr int BM = 32 * MB, BN = 32 * NB;
    static constexpr int MB0 = (MB + 1) / 2, MB1 = MB / 2, NB0 = (NB + 1) / 2, NB1 = NB / 2;
    static constexpr int STEP = (MB + NB) * 4096;            // bytes of one K-step (64 k) of both operands
    static constexpr int OX0 = 0, OW0 = MB0 * 4096, OW1 = OW0 + NB0 * 4096, OX1 = OW1 + NB1 * 4096;
    static constexpr int NR = 160 * 1024 / STEP < 4 ? 160 * 1024 / STEP : 4;      // K-steps of the ring
    static constexpr int LDS = NR * STEP;
    static_assert(LDS + BM * 4 <= 160 * 1024, "the grouped form keeps its rows' slots beside the ring");
};
constexpr int QF4_PITCH = 264;                               // elements per LDS row of the q|k|v epilogue

}  // namespace

// a, b: the same register of two 16-column blocks -> lanes of even groups of 16 hold the first block's columns (a: their own four, b: the next group's four), odd groups the second's
__device__ __forceinline__ void swap16(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0]; b = r[1];
}
// a's upper 32 lanes <-> b's lower 32
__device__ __forceinline__ void swap32(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]); b = __uint_as_float(r[1]);
}
// 8 values of one row (4 where the row ends); `wide`: 16-byte rows
template <typename T> __device__ __forceinline__ void put8(T* p, uint4 u, bool wide, bool whole = true) {
    if (wide && whole) *reinterpret_cast<uint4*>(p) = u;
    else {
        *reinterpret_cast<uint2*>(p) = uint2{u.x, u.y};
        if (whole) *reinterpret_cast<uint2*>(p + 4) = uint2{u.z, u.w};
    }
}

// two rotation pairs at once: T( T(x1 c) + T(-x2 s) ), T( T(x2 c) + T(x1 s) ), the arithmetic of rope_term with two roundings an instruction
template <typename T> __device__ __forceinline__ void rope_pairs(uint32_t x1, uint32_t x2, uint32_t c, uint32_t s, uint32_t& o1, uint32_t& o2) {
#pragma clang fp contract(off)
    const float al = unpack_lo<T>(x1), ah = unpack_hi<T>(x1), bl = unpack_lo<T>(x2), bh = unpack_hi<T>(x2);
    const float cl = unpack_lo<T>(c), ch = unpack_hi<T>(c), sl = unpack_lo<T>(s), sh = unpack_hi<T>(s);
    const uint32_t p1 = pack2<T>(al * cl, ah * ch), q1 = pack2<T>(-bl * sl, -bh * sh), p2 = pack2<T>(bl * cl, bh * ch), q2 = pack2<T>(al * sl, ah * sh);
    o1 = pack2<T>(unpack_lo<T>(p1) + unpack_lo<T>(q1), unpack_hi<T>(p1) + unpack_hi<T>(q1));
    o2 = pack2<T>(unpack_lo<T>(p2) + unpack_lo<T>(q2), unpack_hi<T>(p2) + unpack_hi<T>(q2));
}

// q|k|v epilogue with RoPE + KV-cache append (GemmArgs::qf_*).  A 256-column tile covers whole heads of ONE of the three regions (the launcher checks the alignment), a wave's 128
// columns one head of 128 or two of 64: both members of a rotation pair (d, d + D / 2) are the same register of two of its blocks.
//   q / k tile: rounded to T (the rounding point of GEMM + rope_kv_kernel), out = T( T(x cos) + T(rot(x) sin) ) with cos / sin of the row's position from the fp32 table, requested
//               four row blocks at a time; 16-byte stores into the q columns of C / the K-cache row of the position.
//   v tile:     LDS image TRANSPOSED [col][row], so that a work item (d, 8 consecutive positions) is one 16-byte LDS read and one 16-byte store into V^T[kv head][d][pos ..] (pos0
//               and the row group are multiples of 8).
template <typename T, int MB>
__device__ __forceinline__ void qkv_rope_epilogue4(const GemmArgs& a, f32x4 (&acc)[8][MB], char* smem, int m0, int n0, int wm, int wn, int lane, int tid) {
    constexpr int BM = 32 * MB;
    const int D = a.qf_D, HALF = D >> 1;
    const int q_cols = a.qf_nh * D, k_cols = a.qf_nkv * D;
    const int region = n0 < q_cols ? 0 : (n0 < q_cols + k_cols ? 1 : 2);
    const int l15 = lane & 15, g4 = lane >> 4;
    if (region < 2) {
        // four row blocks at a time: their table values are requested in front of the batch's first store (a load behind a store waits for it: vmcnt counts both in order)
        constexpr int JB = 4;
        auto heads = [&](auto d_c) {
            constexpr int DD = decltype(d_c)::value, HB = DD / 32;       // blocks of half a head: block i turns with i + HB
            const int head = (n0 - (region ? q_cols : 0) + wn * 128) / DD;      // first of the wave's heads in its region
#pragma unroll 1
            for (int j0 = 0; j0 < MB; j0 += JB) {
                if (m0 + j0 * 32 + wm * 16 >= a.M) break;
                f32x4 cs[JB][HB][2];
#pragma unroll
                for (int jj = 0; jj < JB; ++jj) {
                    int m = m0 + (j0 + jj) * 32 + wm * 16 + l15; m = m < a.M ? m : a.M - 1;
                    const float* row = a.qf_rope + (size_t)(a.qf_pos0 + m) * DD + 4 * g4;
#pragma unroll
                    for (int p = 0; p < HB; ++p) {
                        cs[jj][p][0] = *reinterpret_cast<const f32x4*>(row + 16 * p);
                        cs[jj][p][1] = *reinterpret_cast<const f32x4*>(row + DD / 2 + 16 * p);
                    }
                }
#pragma unroll
                for (int jj = 0; jj < JB; ++jj) {
                    const int m = m0 + (j0 + jj) * 32 + wm * 16 + l15;
                    f32x4 t[8];
#pragma unroll
                    for (int b0 = 0; b0 < MB; b0 += JB)
                        if (b0 == j0 && b0 + jj < MB) {
#pragma unroll
                            for (int i = 0; i < 8; ++i) t[i] = from_acc(acc[i][b0 + jj < MB ? b0 + jj : 0]);
                        }
                    uint32_t o[8][2];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int p = q % HB, i = q / HB * 2 * HB + p, k = i + HB;
#pragma unroll
                        for (int e = 0; e < 4; e += 2)
                            rope_pairs<T>(pack2<T>(t[i][e], t[i][e + 1]), pack2<T>(t[k][e], t[k][e + 1]), pack2<T>(cs[jj][p][0][e], cs[jj][p][0][e + 1]),
                                          pack2<T>(cs[jj][p][1][e], cs[jj][p][1][e + 1]), o[i][e >> 1], o[k][e >> 1]);
                    }
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        swap16(o[2 * p][0], o[2 * p + 1][0]); swap16(o[2 * p][1], o[2 * p + 1][1]);
                        const int c = 32 * p + (g4 & 1) * 16 + (g4 >> 1) * 8;
                        T* dst = region == 0 ? reinterpret_cast<T*>(a.C) + (size_t)m * a.ldc + n0 + wn * 128 + c
                                             : reinterpret_cast<T*>(a.qf_kc) + ((size_t)(head + c / DD) * a.qf_smax + a.qf_pos0 + m) * DD + c % DD;
                        if (m < a.M && j0 + jj < MB) *reinterpret_cast<uint4*>(dst) = uint4{o[2 * p][0], o[2 * p][1], o[2 * p + 1][0], o[2 * p + 1][1]};
                    }
                }
            }
        };
        if (D == 128) heads(IC<128>{});
        else heads(IC<64>{});
    } else {
        uint16_t* tt = reinterpret_cast<uint16_t*>(smem);     // [col][row]
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < MB; ++j) {
                const f32x4 t = from_acc(acc[i][j]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = j * 32 + wm * 16 + l15, col = wn * 128 + i * 16 + 4 * g4 + r;
                    tt[col * QF4_PITCH + row] = (uint16_t)(pack2<T>(t[r], 0.f) & 0xffffu);
                }
            }
        __syncthreads();
        T* vt = reinterpret_cast<T*>(a.qf_vt);
        const int row0 = n0 - q_cols - k_cols;                  // first V^T row [kv head][d] of the tile
        const int rg = tid & 31, m = m0 + rg * 8;               // 8 positions, every eighth column
        if (rg < BM / 8 && m < a.M) {
            T* dst = vt + (size_t)(row0 + (tid >> 5)) * a.qf_smax + a.qf_pos0 + m;
#pragma unroll 1
            for (int c0 = tid >> 5; c0 < 256; c0 += 64) {
                uint4 v[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) v[k] = *reinterpret_cast<const uint4*>(tt + (c0 + 8 * k) * QF4_PITCH + rg * 8);
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    T* p = dst + (size_t)(c0 - (tid >> 5) + 8 * k) * a.qf_smax;
                    if (m + 8 <= a.M) *reinterpret_cast<uint4*>(p) = v[k];
                    else                                        // the last, partial row group of the prompt
                        for (int e = 0; m + e < a.M; ++e) reinterpret_cast<uint16_t*>(p)[e] = tt[(c0 + 8 * k) * QF4_PITCH + rg * 8 + e];
                }
            }
        }
        if (m0 + BM >= a.M) {                                   // V^T behind the last row: cleared to the end of its 64 keys, as rope_kv_kernel does
            const int end = a.qf_pos0 + a.M, whole = (end + 63) & ~63, pos = end + (tid & 63);
            if (pos < (whole < a.qf_smax ? whole : a.qf_smax))
                for (int c = tid >> 6; c < 256; c += 4)
                    reinterpret_cast<uint16_t*>(vt)[(size_t)(row0 + c) * a.qf_smax + pos] = 0;
        }
    }
}

// out_row(m): row of C that row m of the tile's problem is written to
template <typename T, int MB, int NB, typename F>
__device__ __forceinline__ void epilogue4(const GemmArgs& a, f32x4 (&acc)[NB][MB], int m0, int n0, int wm, int wn, int lane, F&& out_row) {
    constexpr int P = (NB + 1) / 2;                                     // pairs of blocks
    T* C = reinterpret_cast<T*>(a.C);
    const T* bias = reinterpret_cast<const T*>(a.bias);
    const T* R = reinterpret_cast<const T*>(a.R);
    const int act = a.act;
    const int l15 = lane & 15, g4 = lane >> 4;
    const bool gated = act_gated(act);
    const bool wide = a.ldc % 8 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0, wide_r = a.ldr % 8 == 0 && reinterpret_cast<uintptr_t>(R) % 16 == 0;
    const int pk_q = a.pk_kc ? a.pk_heads * a.pk_D : 0x3fffffff;
    const int nb = n0 + wn * NB * 16;
    const int cb = (g4 & 1) * 16 + (g4 >> 1) * 8;                       // columns of pair p: nb + 32 p + cb .. + 7
    auto want = [&](uint4 (&d)[P], int j) {
        const int m = m0 + j * 32 + wm * 16 + l15;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int c = 32 * p + cb, n = nb + c;
            d[p] = uint4{0u, 0u, 0u, 0u};
            if (m < a.M && c < 16 * NB && n < a.N && n < pk_q) {
                const T* r = R + (size_t)m * a.ldr + n;
                const bool whole = n + 8 <= a.N;
                if (wide_r && whole) d[p] = *reinterpret_cast<const uint4*>(r);
                else {
                    const uint2 x = *reinterpret_cast<const uint2*>(r), y = whole ? *reinterpret_cast<const uint2*>(r + 4) : uint2{0u, 0u};
                    d[p] = uint4{x.x, x.y, y.x, y.y};
                }
            }
        }
    };
    auto take = [&](f32x4 (&t)[2 * P], int j) {
        t[2 * P - 1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NB; ++i) t[i] = from_acc(acc[i][j]);
    };
    if (gated) {
#pragma unroll 1
        for (int j = 0; j < MB; ++j) {
            const int mb = m0 + j * 32 + wm * 16, m = mb + l15;
            if (mb >= a.M) break;
            f32x4 t[2 * P];
#pragma unroll
            for (int jj = 0; jj < MB; ++jj)
                if (jj == j) take(t, jj);
            T* row = C + (size_t)out_row(m) * a.ldc + (nb >> 1);
            uint32_t o2[2 * ((P + 1) / 2)][2];                           // four outputs a lane of pair p
#pragma unroll
            for (int p = 0; p < P; ++p) {
                float g[4] = {t[2 * p][0], t[2 * p][1], t[2 * p][2], t[2 * p][3]}, u[4] = {t[2 * p + 1][0], t[2 * p + 1][1], t[2 * p + 1][2], t[2 * p + 1][3]};
#pragma unroll
                for (int e = 0; e < 4; ++e) swap32(g[e], u[e]);
                if (bias) {
                    const int oc = (nb >> 1) + 16 * p + 8 * (g4 >> 1) + 4 * (g4 & 1), ng = (oc >> 5) * 64 + (oc & 31);
                    if (ng < a.N) {
                        float b[4], c[4]; load4<T>(bias + ng, b); load4<T>(bias + ng + 32, c);
#pragma unroll
                        for (int e = 0; e < 4; ++e) { g[e] += b[e]; u[e] += c[e]; }
                    }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) g[e] = gate_mul(act, g[e], u[e]);
                o2[p][0] = pack2<T>(g[0], g[1]); o2[p][1] = pack2<T>(g[2], g[3]);
            }
            if constexpr (P % 2 == 1) o2[P][0] = o2[P][1] = 0u;
#pragma unroll
            for (int p = 0; p < P; p += 2) {
                swap16(o2[p][0], o2[p + 1][0]); swap16(o2[p][1], o2[p + 1][1]);
                const int b = 2 * p + 2 * (g4 & 1) + (g4 >> 1);            // the lane's block
                if (m < a.M && b < NB && nb + 16 * b < a.N) put8(row + 8 * b, uint4{o2[p][0], o2[p][1], o2[p + 1][0], o2[p + 1][1]}, wide);
            }
        }
        return;
    }
    auto columns = [&](const f32x4 (&t)[2 * P], float (&v)[P][8]) {
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) { v[p][e] = t[2 * p][e]; v[p][4 + e] = t[2 * p + 1][e]; swap16(v[p][e], v[p][4 + e]); }
    };
    auto residual = [&](float (&v)[P][8], const uint4 (&rq)[P]) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            v[p][0] += unpack_lo<T>(rq[p].x); v[p][1] += unpack_hi<T>(rq[p].x); v[p][2] += unpack_lo<T>(rq[p].y); v[p][3] += unpack_hi<T>(rq[p].y);
            v[p][4] += unpack_lo<T>(rq[p].z); v[p][5] += unpack_hi<T>(rq[p].z); v[p][6] += unpack_lo<T>(rq[p].w); v[p][7] += unpack_hi<T>(rq[p].w);
        }
    };
    auto packed = [&](const float (&v)[8]) { return uint4{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]), pack2<T>(v[4], v[5]), pack2<T>(v[6], v[7])}; };
    auto add_bias = [&](float (&v)[P][8]) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int c = 32 * p + cb, n = nb + c;
            if (c < 16 * NB && n < a.N) {
                float b[4], c4[4] = {0.f, 0.f, 0.f, 0.f};
                load4<T>(bias + n, b);
                if (n + 8 <= a.N) load4<T>(bias + n + 4, c4);
#pragma unroll
                for (int e = 0; e < 4; ++e) { v[p][e] += b[e]; v[p][4 + e] += c4[e]; }
            }
        }
    };
    if (act == kActNone && !a.pk_kc) {
        // the residual of the whole tile is requested at once, into the registers of the fragments: a row block ahead, every block waited for its rows and, vmcnt being in order, for
        // the stores in front of them
        uint4 rows[MB][P];
        if (R) {
#pragma unroll
            for (int j = 0; j < MB; ++j) want(rows[j], j);
        }
#pragma unroll
        for (int j = 0; j < MB; ++j) {
            const int mb = m0 + j * 32 + wm * 16, m = mb + l15;
            if (mb >= a.M) break;
            f32x4 t[2 * P];
            take(t, j);
            float v[P][8];
            columns(t, v);
            if (bias) add_bias(v);
            if (R) residual(v, rows[j]);
            T* row = C + (size_t)out_row(m) * a.ldc;
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int c = 32 * p + cb, n = nb + c;
                if (m < a.M && c < 16 * NB && n < a.N) put8(row + n, packed(v[p]), wide, n + 8 <= a.N);
            }
        }
        return;
    }
    uint4 rq[P], rn[P];
    if (R) want(rn, 0);
#pragma unroll 1
    for (int j = 0; j < MB; ++j) {
        const int mb = m0 + j * 32 + wm * 16, m = mb + l15;
        if (mb >= a.M) break;
        if (R) {
#pragma unroll
            for (int p = 0; p < P; ++p) rq[p] = rn[p];
            if (j + 1 < MB) want(rn, j + 1);
        }
        f32x4 t[2 * P];
#pragma unroll
        for (int jj = 0; jj < MB; ++jj)
            if (jj == j) take(t, jj);
        float v[P][8];
        columns(t, v);
        if (bias) add_bias(v);
        if (act != kActNone) {
#pragma unroll 1
            for (int p = 0; p < P; ++p) {
                float w[8];
#pragma unroll
                for (int pp = 0; pp < P; ++pp)
                    if (pp == p)
#pragma unroll
                        for (int e = 0; e < 8; ++e) w[e] = v[pp][e];
                apply_act_n<8>(w, act);
#pragma unroll
                for (int pp = 0; pp < P; ++pp)
                    if (pp == p)
#pragma unroll
                        for (int e = 0; e < 8; ++e) v[pp][e] = w[e];
            }
        }
        if (R) residual(v, rq);
        T* row = C + (size_t)out_row(m) * a.ldc;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int c = 32 * p + cb, n = nb + c;
            const uint4 u = packed(v[p]);
            if (m >= a.M || c >= 16 * NB || n >= a.N) continue;
            if (n < pk_q) put8(row + n, u, wide, n + 8 <= a.N);
            else {
                const int pimg = m / a.pk_rows, pos = m - pimg * a.pk_rows;
                if (n < 2 * pk_q) {                                      // K rows [head][pos][D]
                    const int kcol = n - pk_q, head = kcol / a.pk_D, d = kcol - head * a.pk_D;
                    put8(reinterpret_cast<T*>(a.pk_kc) + pimg * a.pk_img_stride + ((size_t)head * a.pk_spad + pos) * a.pk_D + d, u, false);
                } else {                                                 // V^T [head][d][pos]: a store instruction makes runs of 16 positions
                    uint16_t* vt = reinterpret_cast<uint16_t*>(a.pk_vt) + pimg * a.pk_img_stride + (size_t)(n - 2 * pk_q) * a.pk_spad + pos;
                    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) vt[(size_t)e * a.pk_spad] = (uint16_t)(e & 1 ? w[e >> 1] >> 16 : w[e >> 1] & 0xffffu);
                }
            }
        }
    }
}

// weight row behind buffer row rb + 32 i of a tile's W halves
template <int NB> __device__ __forceinline__ int weight_row(int i, int rb, int n0, int N, bool gated) {
    constexpr int NB0 = (NB + 1) / 2, NB1 = NB / 2;
    const int half = i >= NB0, blocks = half ? NB1 : NB0, r = (half ? i - NB0 : i) * 32 + rb;      // buffer row of the half
    const int w = r >= 16 * blocks, c = r - w * 16 * blocks;
    int n = n0 + w * NB * 16 + half * NB0 * 16 + c;
    if (gated) n = gated_row(n);
    return n < N ? n : N - 1;
}

// the K-steps [kt_begin, kt_begin + nk) of one tile.  vx, vw: byte offsets of the thread's DMA pieces in the operands; x1_live: the tile has rows in X half 1 (without, its phases are skipped)
template <typename T, int MB, int NB>
__device__ __forceinline__ void product4(f32x4 (&acc)[NB][MB], char* smem, v4i_t rsX, v4i_t rsW, const uint32_t (&vx)[MB], const uint32_t (&vw)[NB], int kt_begin, int nk, bool x1_live,
                                         int tid) {
    using SH = Shape4w<MB, NB>;
    constexpr int MB0 = SH::MB0, MB1 = SH::MB1, NB0 = SH::NB0, NB1 = SH::NB1;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1, l15 = lane & 15, g4 = lane >> 4;
    const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    const unsigned lds_wave = __builtin_amdgcn_readfirstlane(lds_base + wave * 1024);

    // An LDS-DMA instruction lands lane-linear at M0; M0 is set at least one instruction ahead.  Written as asm so that the compiler neither sees an LDS write (it would drain
    // the queue in front of the next ds_read) nor counts the loads.  Nothing else in this kernel uses M0.
    auto aim = [&](unsigned dst) { asm volatile("s_mov_b32 m0, %0" : : "s"(dst)); };
    auto fire = [&](uint32_t v, const v4i_t& rs, unsigned so) { asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" : : "v"(v), "s"(rs), "s"(so) : "memory"); };

    // ---- fragment read addresses --------------------------------------------------------------------------------------------------
    int ox[2], ow0[2], ow1[2];                               // [ks]
    {
        const int sw = (l15 >> 1) & 7;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int c = ((4 * ks + g4) ^ sw) << 4;
            ox[ks] = (wm * 16 + l15) * 128 + c;
            ow0[ks] = SH::OW0 + (wn * 16 * NB0 + l15) * 128 + c;
            ow1[ks] = SH::OW1 + (wn * 16 * NB1 + l15) * 128 + c;
        }
    }

#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    frag_t x0[2][MB0], x1[2][MB1], w0[2][NB0], w1[2][NB1];
    auto at = [&](int off) { return *reinterpret_cast<const frag_t*>(smem + off); };
    auto rd_x0 = [&](int ring, int t) { const int ks = t / MB0, i = t % MB0; x0[ks][i] = at(ox[ks] + ring + i * 4096); };
    auto rd_x1 = [&](int ring, int t) { const int ks = t / MB1, i = t % MB1; x1[ks][i] = at(ox[ks] + ring + SH::OX1 + i * 4096); };
    auto rd_w0 = [&](int ring, int t) { const int ks = t / NB0, i = t % NB0; w0[ks][i] = at(ow0[ks] + ring + i * 2048); };
    auto rd_w1 = [&](int ring, int t) { const int ks = t / NB1, i = t % NB1; w1[ks][i] = at(ow1[ks] + ring + i * 2048); };

    auto main_loop = [&](auto live_c) {
        constexpr bool X1 = decltype(live_c)::value;
        constexpr int C1 = X1 ? MB1 : 0;                     // DMA instructions of X half 1
        unsigned so = 0;                                     // byte offset along K of the K-step that is staged next
        // half j (0: X0, 1: W0, 2: W1, 3: X1), piece t, ring slot at `ring`
        auto st_aim = [&](int j, int ring, int t) { aim(lds_wave + ring + (j == 0 ? SH::OX0 : j == 1 ? SH::OW0 : j == 2 ? SH::OW1 : SH::OX1) + t * 4096); };
        auto st_fire = [&](int j, int t) {
            if (j == 0) fire(vx[t], rsX, so);
            else if (j == 1) fire(vw[t], rsW, so);
            else if (j == 2) fire(vw[NB0 + t], rsW, so);
            else fire(vx[MB0 + t], rsX, so);
        };
        auto st = [&](int j, int ring, int t) { st_aim(j, ring, t); asm volatile("s_nop 0"); st_fire(j, t); };
        auto mma = [&](int nh, int mh, int t) {              // MFMA t of the quadrant (W half nh, X half mh)
            const int nw = nh ? NB1 : NB0, nx = mh ? MB1 : MB0;
            const int ks = t & 1, r = t >> 1, i = r / nx, j = (i & 1) ? nx - 1 - r % nx : r % nx;
            f32x4& d = acc[nh ? NB0 + i : i][mh ? MB0 + j : j];
            mfma16<T>(d, nh ? w1[ks][i] : w0[ks][i], mh ? x1[ks][j] : x0[ks][j]);
        };
        constexpr int NR = SH::NR, STEPC = MB0 + NB + C1;    // K-steps of the ring, DMA instructions of one
        // ---- prologue: the whole ring on its way, the first K-step landed and its first halves in registers ---------------------------
        so = (unsigned)kt_begin * 128u;
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            if (k >= nk) { rsX.z = 0; rsW.z = 0; }           // nothing behind the last K-step: empty descriptors read no memory and keep every count
            const int first = (k ^ NR) & 1;                  // the W half that the loop stages first for this K-step
#pragma unroll
            for (int t = 0; t < MB0; ++t) st(0, k * SH::STEP, t);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < ((h ^ first) ? NB1 : NB0); ++t) st((h ^ first) ? 2 : 1, k * SH::STEP, t);
#pragma unroll
            for (int t = 0; t < C1; ++t) st(3, k * SH::STEP, t);
            so += 128u;
        }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NR - 1) * STEPC) : "memory");
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int t = 0; t < 2 * MB0; ++t) rd_x0(0, t);
#pragma unroll
        for (int t = 0; t < 2 * NB0; ++t) rd_w0(0, t);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();

        // one phase: the quadrant's MFMAs, between them the next half's fragment reads, then one half's DMA (M0 of a piece set two MFMAs ahead of it)
        auto phase = [&](auto nh_c, auto mh_c, auto reads_c, auto j_c, auto pieces_c, int ring, auto&& rd) {
            constexpr int NH = decltype(nh_c)::value, MH = decltype(mh_c)::value, READS = decltype(reads_c)::value, J = decltype(j_c)::value, PIECES = decltype(pieces_c)::value;
            constexpr int NM = (MH && !X1) ? 0 : 2 * (NH ? NB1 : NB0) * (MH ? MB1 : MB0);
            constexpr int G = READS + PIECES > 0 ? READS + PIECES : 1;
            constexpr int EVERY = NM / G > 0 ? NM / G : 1;
            auto aux = [&](int k) {
                if (k < READS) rd(k);
                else st_fire(J, k - READS);
                if (k + 1 >= READS && k + 1 < READS + PIECES) st_aim(J, ring, k + 1 - READS);
            };
            int done = 0;
            if constexpr (READS == 0 && PIECES > 0) { st_aim(J, ring, 0); asm volatile("s_nop 0"); }
#pragma unroll
            for (int t = 0; t < NM; ++t) {
                mma(NH, MH, t);
                if (t % EVERY == EVERY - 1 && done < READS + PIECES) {
                    aux(done++);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int t = 0; t < READS + PIECES; ++t)
                if (t >= done) { if (t >= READS) asm volatile("s_nop 0"); aux(t); }
            __builtin_amdgcn_sched_barrier(0);
        };
        int cur = 0, nxt = SH::STEP;                         // ring slots of this K-step and the next
        auto kstep = [&](auto par_c, int left) {             // left: K-steps behind this one
            constexpr int A = decltype(par_c)::value, B = 1 - A;      // W half that comes first in this K-step, second
            constexpr int NA = A ? NB1 : NB0, NBB = B ? NB1 : NB0;
            if (left < NR) { rsX.z = 0; rsW.z = 0; }
            phase(IC<A>{}, IC<0>{}, IC<2 * NBB>{}, IC<0>{}, IC<MB0>{}, cur, [&](int t) { if constexpr (B) rd_w1(cur, t); else rd_w0(cur, t); });
            phase(IC<B>{}, IC<0>{}, IC<X1 ? 2 * MB1 : 0>{}, IC<A ? 2 : 1>{}, IC<NA>{}, cur, [&](int t) { rd_x1(cur, t); });
            // in flight: behind the first two halves of the next K-step (an odd ring stages the W halves of a K-step in the other order)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NR % 2 ? 0 : NA) + C1 + (NR - 2) * STEPC + MB0 + NA) : "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            phase(IC<B>{}, IC<1>{}, IC<2 * MB0>{}, IC<B ? 2 : 1>{}, IC<NBB>{}, cur, [&](int t) { rd_x0(nxt, t); });
            phase(IC<A>{}, IC<1>{}, IC<2 * NBB>{}, IC<3>{}, IC<C1>{}, cur, [&](int t) { if constexpr (B) rd_w1(nxt, t); else rd_w0(nxt, t); });
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NR - 1) * STEPC) : "memory");       // behind the next K-step
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            so += 128u;
            cur = nxt;
            nxt = nxt + SH::STEP == SH::LDS ? 0 : nxt + SH::STEP;
        };
        // an odd last K-step is followed by one of zeros: one exit, so that the accumulators stay where they are
#pragma unroll 1
        for (int left = nk; left > 0; left -= 2) {
            kstep(IC<0>{}, left - 1);
            kstep(IC<1>{}, left - 2);
        }
    };
    if (x1_live) main_loop(IC<1>{});
    else main_loop(IC<0>{});
    mfma_settle();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // no LDS write is on its way when the workgroup, or its ring, ends
}

template <typename T, int MB, int NB, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm4w_kernel(GemmArgs a) {
    using SH = Shape4w<MB, NB>;
    constexpr int MB0 = SH::MB0;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int l15 = lane & 15, g4 = lane >> 4;

    const int S = SPLIT ? a.split_k : 1;
    const int mtiles = (a.M + SH::BM - 1) / SH::BM, ntiles = (a.N + SH::BN - 1) / SH::BN;
    const int lid = xcd_remap(blockIdx.x, mtiles * ntiles * S);
    const int tile = SPLIT ? lid / S : lid, slice = SPLIT ? lid - tile * S : 0;
    int tile_m, tile_n;
    if constexpr (!SPLIT) gemm_tile_of(tile, mtiles, ntiles, tile_m, tile_n);
    else { tile_n = tile / mtiles; tile_m = tile - tile_n * mtiles; }
    const int m0 = tile_m * SH::BM, n0 = tile_n * SH::BN;
    const int nk_all = a.K >> 6;
    const int pairs = (nk_all + 1) >> 1;                     // slices of whole pairs: only the last one can end on an odd K-step
    const int kt_begin = SPLIT ? 2 * (int)((long)pairs * slice / S) : 0;
    const int kt_end = SPLIT && slice + 1 < S ? 2 * (int)((long)pairs * (slice + 1) / S) : nk_all;
    const int nk = kt_end - kt_begin;

    // ---- LDS-DMA sources: piece i of a half covers buffer rows 8 (wave + 4 i) .. + 7 -----------------------------------------------
    v4i_t rsX = make_rsrc(a.X, (uint32_t)((size_t)a.M * a.ldx * sizeof(T)));
    v4i_t rsW = make_rsrc(a.W, (uint32_t)((size_t)a.N * a.ldw * sizeof(T)));
    uint32_t vx[MB], vw[NB];
    {
        const int rb = 8 * wave + (lane >> 3);
        const int chunk = ((lane & 7) ^ (rb >> 1)) & 7;
        const bool gated = act_gated(a.act);
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            int m = m0 + i * 32 + rb;                        // tile rows in order: half 1 follows half 0
            m = m < a.M ? m : a.M - 1;
            vx[i] = (uint32_t)(((size_t)m * a.ldx + chunk * 8) * sizeof(T));
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int n = weight_row<NB>(i, rb, n0, a.N, gated);
            vw[i] = (uint32_t)(((size_t)n * a.ldw + chunk * 8) * sizeof(T));
        }
    }
    f32x4 acc[NB][MB];
    product4<T, MB, NB>(acc, smem, rsX, rsW, vx, vw, kt_begin, nk, a.M - m0 > 32 * MB0, tid);

    if constexpr (!SPLIT) {
        if constexpr (NB == 8) {
            if (a.qf_kc) {
                __syncthreads();                             // the operand ring is dead
                qkv_rope_epilogue4<T, MB>(a, acc, smem, m0, n0, wm, wn, lane, tid);
                return;
            }
        }
        epilogue4<T, MB, NB>(a, acc, m0, n0, wm, wn, lane, [](int m) { return m; });
    } else {
        // fp32 partial tile in accumulator order: float4 number j NB + i of thread tid at ((j NB + i) 256 + tid) 16 of the slab
        f32x4* slab = reinterpret_cast<f32x4*>(a.skw) + ((size_t)tile * S + slice) * (SH::BM * SH::BN / 4) + tid;
#pragma unroll
        for (int j = 0; j < MB; ++j) {
            if (m0 + j * 32 + wm * 16 >= a.M) continue;
#pragma unroll
            for (int i = 0; i < NB; ++i) slab[(j * NB + i) * 256] = acc[i][j];
        }
    }
}

// The rows of a group times its weight (GroupGemmArgs with a plan; bound and figures: as the linears above, group_gemm_bm): tile rows are slots, their X rows gathered through the DMA offsets, their C rows scattered by the
// epilogue.  Tiles run group by group, a group's row tiles next to each other for one panel of its weight.  The grid is an upper bound: workgroups past the plan's tiles leave.
template <typename T, int MB, int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void group_gemm4w_kernel(GroupGemmArgs a) {
    using SH = Shape4w<MB, NB>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
    const int ntiles = (a.N + SH::BN - 1) / SH::BN, total = *a.plan.n_tiles * ntiles;
    if ((int)blockIdx.x >= total) return;
    const int lid = xcd_remap(blockIdx.x, total);
    const GroupTile t = a.plan.tiles[lid / ntiles];
    const int rel = lid - t.first * ntiles;
    const GroupTile u = a.plan.tiles[t.first + rel % t.n_tiles];
    const int grp = __builtin_amdgcn_readfirstlane(u.group), row0 = __builtin_amdgcn_readfirstlane(u.row0), rows = __builtin_amdgcn_readfirstlane(u.rows);
    const int n0 = __builtin_amdgcn_readfirstlane(rel / t.n_tiles) * SH::BN;
    const int* order = a.plan.order + row0;
    __shared__ int slots[SH::BM];                            // (the product's first barriers stand between this and the epilogue)
    if (tid < SH::BM) slots[tid] = order[tid < rows ? tid : rows - 1];
    const v4i_t rsX = make_rsrc(a.X, (uint32_t)((size_t)(a.rows / a.per_row) * a.ldx * sizeof(T)));
    const v4i_t rsW = make_rsrc(reinterpret_cast<const T*>(a.W) + (size_t)grp * a.w_group, (uint32_t)((size_t)a.N * a.ldw * sizeof(T)));
    uint32_t vx[MB], vw[NB];
    const int rb = 8 * wave + (lane >> 3), chunk = ((lane & 7) ^ (rb >> 1)) & 7;
    const bool gated = act_gated(a.act);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int r = i * 32 + rb;
        vx[i] = (uint32_t)(((size_t)(order[r < rows ? r : rows - 1] / a.per_row) * a.ldx + chunk * 8) * sizeof(T));
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) vw[i] = (uint32_t)(((size_t)weight_row<NB>(i, rb, n0, a.N, gated) * a.ldw + chunk * 8) * sizeof(T));
    f32x4 acc[NB][MB];
    product4<T, MB, NB>(acc, smem, rsX, rsW, vx, vw, 0, a.K >> 6, rows > 32 * SH::MB0, tid);
    GemmArgs e{};
    e.C = a.C; e.ldc = a.ldc; e.M = rows; e.N = a.N; e.act = a.act;
    epilogue4<T, MB, NB>(e, acc, 0, n0, wm, wn, lane, [&](int m) { return slots[m]; });
}

template <typename T, int MB, int NB>
void group_gemm4w_launch(const GroupGemmArgs& a, int m_tiles, hipStream_t st) {
    using SH = Shape4w<MB, NB>;
    auto kern = group_gemm4w_kernel<T, MB, NB>;
    static std::once_flag once;
    std::call_once(once, [&] { LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SH::LDS)); });
    LMX_LAUNCH(kern, dim3(m_tiles * cdiv(a.N, SH::BN)), dim3(256), SH::LDS, st, a);
    LMX_CHECK_HIP(hipGetLastError());
}

// sum of the slices in slice order + epilogue, in row order through LDS: workgroup (tile, j) makes rows 32 j .. + 31 of the tile
template <typename T, int MB, int NB, int S>
__global__ __launch_bounds__(256) void gemm4w_reduce_kernel(GemmArgs a) {
    using SH = Shape4w<MB, NB>;
    constexpr int PITCH = SH::BN + 4;
    __shared__ __attribute__((aligned(16))) float sums[32 * PITCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave & 1, wn = wave >> 1, l15 = lane & 15, g4 = lane >> 4;
    const int mtiles = (a.M + SH::BM - 1) / SH::BM;
    const int tile = blockIdx.x / MB, j = blockIdx.x - tile * MB;
    const int tile_n = tile / mtiles, tile_m = tile - tile_n * mtiles;
    const int m_base = tile_m * SH::BM + j * 32, n0 = tile_n * SH::BN;
    if (m_base >= a.M) return;
    const bool gated = act_gated(a.act);
    const int r_out = tid >> 3, seg = tid & 7, m_out = m_base + r_out;
    const T* R = reinterpret_cast<const T*>(a.R);
    const T* bias = reinterpret_cast<const T*>(a.bias);
    uint2 rr[NB];
    if (R && m_out < a.M) {
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            const int n = n0 + (seg + 8 * k) * 4;
            rr[k] = n < a.N ? *reinterpret_cast<const uint2*>(R + (size_t)m_out * a.ldr + n) : uint2{0u, 0u};
        }
    }
    if (m_base + wm * 16 < a.M) {
        const f32x4* slab = reinterpret_cast<const f32x4*>(a.skw) + (size_t)tile * S * (SH::BM * SH::BN / 4) + tid;
        f32x4 w[S][NB];
#pragma unroll
        for (int sl = 0; sl < S; ++sl)
#pragma unroll
            for (int i = 0; i < NB; ++i) w[sl][i] = slab[(size_t)sl * (SH::BM * SH::BN / 4) + (j * NB + i) * 256];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            f32x4 t = w[0][i];
#pragma unroll
            for (int sl = 1; sl < S; ++sl) t += w[sl][i];
            *reinterpret_cast<f32x4*>(sums + (wm * 16 + l15) * PITCH + wn * NB * 16 + i * 16 + 4 * g4) = t;
        }
    }
    __syncthreads();
    if (m_out >= a.M) return;
    T* __restrict__ C = reinterpret_cast<T*>(a.C);
    const float* row = sums + r_out * PITCH;
    if (gated) {
        for (int o = seg * 4; o < SH::BN / 2; o += 32) {
            const int f = (o >> 3) * 16 + (o & 7), oc = n0 / 2 + o, ng = (oc >> 5) * 64 + (oc & 31);
            if (oc * 2 >= a.N) continue;
            const float4 g = *reinterpret_cast<const float4*>(row + f), u = *reinterpret_cast<const float4*>(row + f + 8);
            float v[4] = {g.x, g.y, g.z, g.w}, w[4] = {u.x, u.y, u.z, u.w};
            if (bias) {
                float bg[4], bu[4]; load4<T>(bias + ng, bg); load4<T>(bias + ng + 32, bu);
#pragma unroll
                for (int e = 0; e < 4; ++e) { v[e] += bg[e]; w[e] += bu[e]; }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gate_mul(a.act, v[e], w[e]);
            store4<T>(C + (size_t)m_out * a.ldc + oc, v);
        }
        return;
    }
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        const int c = (seg + 8 * k) * 4, n = n0 + c;
        if (n >= a.N) continue;
        const f32x4 t = *reinterpret_cast<const f32x4*>(row + c);
        float v[4] = {t.x, t.y, t.z, t.w};
        if (bias) {
            float b[4]; load4<T>(bias + n, b);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += b[e];
        }
        apply_act_n<4>(v, a.act);
        if (R) {
            v[0] += unpack_lo<T>(rr[k].x); v[1] += unpack_hi<T>(rr[k].x); v[2] += unpack_lo<T>(rr[k].y); v[3] += unpack_hi<T>(rr[k].y);
        }
        store4<T>(C + (size_t)m_out * a.ldc + n, v);
    }
}

// launcher of one tile form: the caller has checked the shapes (launch_gemm4w)
template <typename T, int MB, int NB>
void gemm4w_launch(GemmArgs a, int S, hipStream_t st) {
    using SH = Shape4w<MB, NB>;
    const int tiles = cdiv(a.M, SH::BM) * cdiv(a.N, SH::BN);
    a.split_k = S;
    constexpr int QF = 256 * QF4_PITCH * 2;
    const int lds = a.qf_kc && QF > SH::LDS ? QF : SH::LDS;
    // a K-sliced product is two launches; an armed kernel timer (in-situ profile) spans both, the boundary between them included
    KernelTimer* kt = g_kernel_timer;
    const bool timed = S > 1 && kt && !kt->used;
    auto launch = [&](auto kern) {
        // one opt-in per kernel instantiation (every instantiation decays to the same pointer TYPE, so the flag is keyed on the pointer value)
        static std::mutex mu; static std::set<const void*> done;
        {
            std::lock_guard<std::mutex> lk(mu);
            if (!done.count(reinterpret_cast<const void*>(kern))) {
                LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, QF > SH::LDS ? QF : SH::LDS));
                done.insert(reinterpret_cast<const void*>(kern));
            }
        }
        if (timed) { kt->used = true; hipExtLaunchKernelGGL(kern, dim3(tiles * S), dim3(256), lds, st, kt->e0, nullptr, 0, a); }
        else LMX_LAUNCH(kern, dim3(tiles * S), dim3(256), lds, st, a);
        LMX_CHECK_HIP(hipGetLastError());
    };
    if (S == 1) { launch(gemm4w_kernel<T, MB, NB, false>); return; }
    launch(gemm4w_kernel<T, MB, NB, true>);
    auto reduce = [&](auto kern) {
        if (timed) hipExtLaunchKernelGGL(kern, dim3(tiles * MB), dim3(256), 0, st, nullptr, kt->e1, 0, a);
        else hipLaunchKernelGGL(kern, dim3(tiles * MB), dim3(256), 0, st, a);
        LMX_CHECK_HIP(hipGetLastError());
    };
    if (S == 2) reduce(gemm4w_reduce_kernel<T, MB, NB, 2>);
    else reduce(gemm4w_reduce_kernel<T, MB, NB, 3>);
}

// the tile forms, in the order of gemm4w.hip's table; each dtype's in two source files
#define LMX_GEMM4W_LARGE(X, T) X(T, 8, 8) X(T, 7, 8) X(T, 7, 7) X(T, 8, 6)
#define LMX_GEMM4W_SMALL(X, T) X(T, 5, 8) X(T, 6, 6) X(T, 5, 6) X(T, 5, 4) X(T, 4, 5) X(T, 4, 4)
#define LMX_GEMM4W_EXTERN(T, MB, NB) extern template void gemm4w_launch<T, MB, NB>(GemmArgs, int, hipStream_t); \
                                     extern template void group_gemm4w_launch<T, MB, NB>(const GroupGemmArgs&, int, hipStream_t);
#define LMX_GEMM4W_INST(T, MB, NB) template void gemm4w_launch<T, MB, NB>(GemmArgs, int, hipStream_t); \
                                   template void group_gemm4w_launch<T, MB, NB>(const GroupGemmArgs&, int, hipStream_t);

}  // namespace lmx
