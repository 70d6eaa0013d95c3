// Linears of a few dozen to a few hundred rows (a later turn's prompt, short prompts, the rows behind a cached prefix):  C = epilogue(X[M, K] · W[N, K]^T).
//
// Such a launch has to read every weight once and is short of everything else: 256 x 256 tiles leave half their rows empty and give 43 - 86 workgroups, 128 x 128 and
// 64 x 64 tiles read the weights several times over and keep one K-slab of DMA in flight.  Here a workgroup owns ALL rows of an M tile (32 MT <= 256, so up to 256 rows
// there is one M tile and a weight is read by one workgroup), 64 or 128 weight rows, and one of S slices of K:
//   * LDS ring of 64-deep slabs, as many as fit 160 KB (3 .. 6): at 139 rows 110 KB of DMA stay in flight per CU, which is what 5 TB/s x the loaded latency asks for
//     (a 2-slot ring of 128 x 128 tiles: 32 KB);
//   * 8 waves = (BN / 32) column groups x KW groups of the slab's four 16-deep steps: a wave multiplies one 32-row weight fragment with MT row fragments, the KW partial
//     tiles are added through LDS in group order (deterministic);
//   * the finished tile sits in LDS in row order, so that bias, activation, gating, residual and rounding run on 16-byte row pieces; with S > 1 the fp32 tile goes to the
//     slab [slice][M][N] instead and rows_reduce_kernel, the next launch, adds the slices in order and runs the same epilogue.
//   * every workgroup starts its walk over K somewhere else.
// Bound: DMA into LDS.  At 139 rows the q|k|v product without its reads and MFMAs takes 32 us of 36 (64 weight rows, one slice), the weights alone 19: 100 MB of weights from
// HBM and 250 MB of rows from L2 share the way into LDS.  Figures by shape: gemm_rows_form.
#include <algorithm>

#include "common.h"
#include "kernels.h"
#include "gemm_common.h"

namespace lmx {

namespace {

// bias -> activation -> residual -> round, 8 columns of one row at once (the order of gemm_epilogue)
template <typename T> __device__ __forceinline__ void rows_store(const GemmArgs& a, int m, int n, float (&v)[8]) {
    if (a.bias) {
        float b[8]; load8<T>(static_cast<const T*>(a.bias) + n, b);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += b[e];
    }
    apply_act_n<8>(v, a.act);
    if (a.R) {
        float r[8]; load8<T>(static_cast<const T*>(a.R) + (size_t)m * a.ldr + n, r);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += r[e];
    }
    if (a.c_f32) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = soft_cap(v[e], a.cap);
        store8<float>(static_cast<float*>(a.C) + (size_t)m * a.ldc + n, v);
    } else store8<T>(static_cast<T*>(a.C) + (size_t)m * a.ldc + n, v);
}
// gated: 8 outputs from 8 gate and 8 up columns; ng = fused column of the first gate
template <typename T> __device__ __forceinline__ void rows_store_gated(const GemmArgs& a, int m, int ng, float (&g)[8], float (&u)[8]) {
    if (a.bias) {
        float b[8]; load8<T>(static_cast<const T*>(a.bias) + ng, b);
        float c[8]; load8<T>(static_cast<const T*>(a.bias) + ng + 32, c);
#pragma unroll
        for (int e = 0; e < 8; ++e) { g[e] += b[e]; u[e] += c[e]; }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = gate_mul(a.act, g[e], u[e]);
    store8<T>(static_cast<T*>(a.C) + (size_t)m * a.ldc + (ng >> 6) * 32 + (ng & 31), g);
}

typedef int rows_v4i __attribute__((ext_vector_type(4)));
__device__ __forceinline__ rows_v4i rows_rsrc(const void* p) {           // raw buffer view: 32-bit byte offsets (the launcher checks the operands' sizes)
    const uint64_t u = reinterpret_cast<uint64_t>(p);
    return rows_v4i{__builtin_amdgcn_readfirstlane((int)(uint32_t)u), __builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32)), -1, 0x00020000};
}

template <int MT, int BN> constexpr int rows_stages() {
    constexpr int n = 160 * 1024 / ((32 * MT + BN) * GEMM_ROWB);
    return n > 6 ? 6 : n;
}
template <int MT, int BN> constexpr int rows_smem() {
    constexpr int ring = rows_stages<MT, BN>() * (32 * MT + BN) * GEMM_ROWB, tile = 32 * MT * (BN + 4) * 4;
    return ring > tile ? ring : tile;
}
// at most min(younger, N) groups of P loads of this wave stay in flight
template <int N, int P> __device__ __forceinline__ void rows_wait(int younger) {
    static_assert(N * P <= 63, "vmcnt is a 6-bit field");
    if constexpr (N == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (younger >= N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N * P) : "memory");
    else rows_wait<N - 1, P>(younger);
}

}  // namespace

template <typename T, int MT, int BN>
__global__ __launch_bounds__(512) void gemm_rows_kernel(GemmArgs a, int mtiles, int S) {
    constexpr int NW = 8, BM = 32 * MT;
    constexpr int WN = BN / 32, KW = NW / WN, KPW = 4 / KW;     // column groups, groups of a slab's 16-deep steps, steps per group
    constexpr int NSTAGE = rows_stages<MT, BN>(), ROWS = BM + BN, BUF = ROWS * GEMM_ROWB;
    constexpr int PIECES = ROWS / 8, PPW = (PIECES + NW - 1) / NW;
    static_assert(KW * KPW == 4 && KPW <= 2 && NSTAGE >= 3, "shape");
    constexpr int PITCH = BN + 4;                               // floats of a tile row in LDS: 16 rows x 16 bytes hit 16 distinct bank groups

    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN, grp = wave / WN;
    const int hi = lane >> 5, l31 = lane & 31;

    const int ntiles = (a.N + BN - 1) / BN;
    const int lid = xcd_remap(blockIdx.x, mtiles * ntiles * S);
    const int tile_m = lid % mtiles, ns = lid / mtiles, tile_n = ns / S, slice = ns % S;
    const int m0 = tile_m * BM, n0 = tile_n * BN;

    const int nk_all = a.K / GEMM_BK;
    const int k_first = (int)((long)nk_all * slice / S), nk = (int)((long)nk_all * (slice + 1) / S) - k_first;

    // 1-KiB pieces of a slab (8 rows x 128 bytes; X rows first), swizzled on the source side as in gemm_mfma_kernel.  Where the pieces do not divide over the waves the
    // last one is fetched by several: the same bytes to the same place, and every wave counts the same number of loads.
    rows_v4i rs[PPW];
    uint32_t voff[PPW];
    unsigned pdst[PPW];
#pragma unroll
    for (int i = 0; i < PPW; ++i) {
        int p = wave + NW * i; p = p < PIECES ? p : PIECES - 1;
        pdst[i] = (unsigned)p * 1024u;
        const int row = p * 8 + (lane >> 3), chunk = ((lane & 7) ^ (row >> 1)) & 7;
        const bool isx = p * 8 < BM;
        int r = isx ? m0 + row : n0 + row - BM;
        const int last = (isx ? a.M : a.N) - 1;
        r = r < last ? r : last;
        rs[i] = rows_rsrc(isx ? a.X : a.W);
        voff[i] = (uint32_t)(((size_t)r * (isx ? a.ldx : a.ldw) + (size_t)k_first * GEMM_BK + chunk * 8) * sizeof(T));
    }
    const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    // workgroups walk K from different places: in step, all of them ask for the same 128 bytes of every row at a time (weights alone: 5.2 -> 5.7 TB/s)
    const int rot = tile_n * 5 % nk;
    auto stage = [&](int kt, int slot) {         // LDS-DMA from inline asm: the compiler must not drain the queue before every slab's first ds_read (gemm_pipe_kernel)
        int k = kt + rot; k = k < nk ? k : k - nk;
        const unsigned so = (unsigned)k * (unsigned)(GEMM_BK * sizeof(T));
#pragma unroll
        for (int i = 0; i < PPW; ++i) {
            const unsigned dst = __builtin_amdgcn_readfirstlane(lds_base + (unsigned)slot * BUF + pdst[i]);
            unsigned keep;
            asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
                         : "=&s"(keep) : "s"(dst), "v"(voff[i]), "s"(rs[i]), "s"(so) : "memory");
        }
    };

    f32x16 acc[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;

    // Fragments are read one 16-deep step ahead of their MFMAs: behind the barrier that publishes slab kt + 1 a wave requests that slab's first fragments and then multiplies
    // the last ones of slab kt, so the LDS round trip runs beside the matrix pipe.  The slot of slab kt is free for a new slab there: every wave has waited for its last
    // fragments of it (lgkmcnt(0)) in front of that barrier.
    struct Frag { uint4 w, x[MT]; };
    Frag f[2];
    const int wrow = BM + wn * 32 + l31;
    auto read = [&](Frag& d, int slot, int i) {
        const char* buf = smem + slot * BUF;
        const int chunk = (grp * KPW + i) * 2 + hi;
        d.w = *reinterpret_cast<const uint4*>(buf + lds_chunk_off(wrow, chunk));
#pragma unroll
        for (int j = 0; j < MT; ++j) d.x[j] = *reinterpret_cast<const uint4*>(buf + lds_chunk_off(j * 32 + l31, chunk));
    };
    auto mma = [&](const Frag& d) {
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[j] = Mfma32x32x16<T>::run(d.w, d.x[j], acc[j]);
    };
    int slot = 0;
    auto slab = [&](int kt, Frag& cur, Frag& nxt) {      // the last step's fragments are in `cur` (KPW = 1) / `nxt` (KPW = 2); leaves the next slab's first ones in the other
        if constexpr (KPW == 2) {
            read(nxt, slot, 1);
            mma(cur);
        }
        Frag& last = KPW == 2 ? nxt : cur;
        Frag& first = KPW == 2 ? cur : nxt;
        if (kt + 1 < nk) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            rows_wait<NSTAGE - 2, PPW>(nk - 2 - kt);     // slab kt + 1 has landed; the slabs behind it stay in flight
            __builtin_amdgcn_s_barrier();
            const int freed = slot;
            slot = slot + 1 == NSTAGE ? 0 : slot + 1;
            read(first, slot, 0);
            if (kt + NSTAGE < nk) stage(kt + NSTAGE, freed);
        }
        mma(last);
    };
#pragma unroll
    for (int i = 0; i < NSTAGE; ++i)
        if (i < nk) stage(i, i);
    rows_wait<NSTAGE - 1, PPW>(nk - 1);
    __builtin_amdgcn_s_barrier();
    read(f[0], 0, 0);
    if constexpr (KPW == 2) {
        for (int kt = 0; kt < nk; ++kt) slab(kt, f[0], f[1]);
    } else {
        int kt = 0;
        for (; kt + 1 < nk; kt += 2) { slab(kt, f[0], f[1]); slab(kt + 1, f[1], f[0]); }
        if (kt < nk) slab(kt, f[0], f[1]);
    }

    // ---- the KW partial tiles into one fp32 tile in row order (acc[j][4 q + e] = row j * 32 + l31, column wn * 32 + 8 q + 4 hi + e) ----
    float* tile = reinterpret_cast<float*>(smem);
    __syncthreads();
#pragma unroll
    for (int g = 0; g < KW; ++g) {
        if (grp == g) {
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float4* p = reinterpret_cast<float4*>(tile + (j * 32 + l31) * PITCH + wn * 32 + 8 * q + 4 * hi);
                    float4 v = make_float4(acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]);
                    if (g) { const float4 o = *p; v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w; }
                    *p = v;
                }
        }
        __syncthreads();
    }
    const int rows = a.M - m0 < BM ? a.M - m0 : BM;
    if (S > 1) {
        float* slab = static_cast<float*>(a.skw) + (size_t)slice * a.M * a.N;
        for (int i = tid; i < rows * (BN / 4); i += NW * 64) {
            const int m = i / (BN / 4), c = (i % (BN / 4)) * 4;
            if (n0 + c < a.N) *reinterpret_cast<float4*>(slab + (size_t)(m0 + m) * a.N + n0 + c) = *reinterpret_cast<const float4*>(tile + m * PITCH + c);
        }
        return;
    }
    if (act_gated(a.act)) {
        for (int i = tid; i < rows * (BN / 16); i += NW * 64) {
            const int m = i / (BN / 16), o = (i % (BN / 16)) * 8, c = (o >> 5) * 64 + (o & 31);
            if (n0 + c >= a.N) continue;
            float g[8], u[8];
            load8<float>(tile + m * PITCH + c, g); load8<float>(tile + m * PITCH + c + 32, u);
            rows_store_gated<T>(a, m0 + m, n0 + c, g, u);
        }
        return;
    }
    const int pk_q = a.pk_kc ? a.pk_heads * a.pk_D : 0x3fffffff;        // CLIP q|k|v: the k columns leave as K rows, the v columns as V^T (GemmArgs::pk_kc)
    for (int i = tid; i < rows * (BN / 8); i += NW * 64) {
        const int m = i / (BN / 8), c = (i % (BN / 8)) * 8;
        if (n0 + c >= a.N || n0 + c >= 2 * pk_q) continue;
        float v[8]; load8<float>(tile + m * PITCH + c, v);
        if (n0 + c < pk_q) { rows_store<T>(a, m0 + m, n0 + c, v); continue; }
        if (a.bias) {
            float b[8]; load8<T>(static_cast<const T*>(a.bias) + n0 + c, b);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += b[e];
        }
        apply_act_n<8>(v, a.act);
        const int im = (m0 + m) / a.pk_rows, pos = m0 + m - im * a.pk_rows, kc = n0 + c - pk_q, head = kc / a.pk_D, d = kc - head * a.pk_D;
        store8<T>(static_cast<T*>(a.pk_kc) + im * a.pk_img_stride + ((size_t)head * a.pk_spad + pos) * a.pk_D + d, v);
    }
    const int v0 = 2 * pk_q > n0 ? 2 * pk_q - n0 : 0, v1 = a.N - n0 < BN ? a.N - n0 : BN;
    if (v0 >= v1) return;
    for (int i = tid; i < rows * (v1 - v0); i += NW * 64) {               // lanes along the rows: consecutive positions of one V^T row
        const int c = v0 + i / rows, m = i % rows;
        float v[1] = {tile[m * PITCH + c] + (a.bias ? to_f32(static_cast<const T*>(a.bias)[n0 + c]) : 0.f)};
        apply_act_n<1>(v, a.act);
        const int im = (m0 + m) / a.pk_rows, pos = m0 + m - im * a.pk_rows;
        static_cast<T*>(a.pk_vt)[im * a.pk_img_stride + (size_t)(n0 + c - 2 * pk_q) * a.pk_spad + pos] = from_f32<T>(v[0]);
    }
}

// sum of the S slabs in slice order + epilogue; a thread makes 8 outputs
template <typename T>
__global__ __launch_bounds__(256) void rows_reduce_kernel(GemmArgs a, int S) {
    const bool gated = act_gated(a.act);
    const int per_row = (gated ? a.N / 2 : a.N) / 8;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long)a.M * per_row) return;
    const int m = (int)(i / per_row), o = (int)(i % per_row) * 8;
    const float* slab = static_cast<const float*>(a.skw) + (size_t)m * a.N;
    const size_t step = (size_t)a.M * a.N;
    auto sum = [&](int n, float (&v)[8]) {
        load8<float>(slab + n, v);
        for (int s = 1; s < S; ++s) {
            float t[8]; load8<float>(slab + s * step + n, t);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += t[e];
        }
    };
    if (gated) {
        const int c = (o >> 5) * 64 + (o & 31);
        float g[8], u[8];
        sum(c, g); sum(c + 32, u);
        rows_store_gated<T>(a, m, c, g, u);
    } else {
        float v[8];
        sum(o, v);
        rows_store<T>(a, m, o, v);
    }
}

// The same sum with residual rows, and the RMSNorm of the finished row in the same launch: a workgroup owns a row (rmsnorm_reg_kernel's order of its sum, so its bits).  Its time is the
// launch, one slice's round trip behind the other and the row's sum: 139 rows of 4096 in six slices (13.7 MB from L2) 4.8 + 4.8 us in two launches -> 5.8.  A layer of prompts of 33 .. 384
// rows, hidden 4096, 2 .. 4 us less of 125 .. 255 for down, and as much for o where that is sliced.
template <typename T, int NP>
__global__ __launch_bounds__(256) void rows_reduce_norm_kernel(GemmArgs a, int S, const T* __restrict__ w, T* __restrict__ xn, float eps) {
    __shared__ float red[4];
    const int m = blockIdx.x, tid = threadIdx.x, HC = a.N >> 3;
    const float* slab = static_cast<const float*>(a.skw) + (size_t)m * a.N;
    const size_t step = (size_t)a.M * a.N;
    const T* R = static_cast<const T*>(a.R);
    float v[NP][8], r[NP][8];
    Chunk8<T> g[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int c = tid + i * 256;
        if (c >= HC) continue;
        load8<float>(slab + c * 8, v[i]);
        if (R) load8<T>(R + (size_t)m * a.ldr + c * 8, r[i]);
        g[i].load(w + c * 8);
    }
    for (int s = 1; s < S; ++s) {
        float t[NP][8];
#pragma unroll
        for (int i = 0; i < NP; ++i) { const int c = tid + i * 256; if (c < HC) load8<float>(slab + s * step + c * 8, t[i]); }
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] += t[i][e];
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int c = tid + i * 256;
        if (c >= HC) continue;
#pragma unroll
        for (int e = 0; e < 8; ++e) { v[i][e] = round_to<T>(R ? v[i][e] + r[i][e] : v[i][e]); ss += v[i][e] * v[i][e]; }
        store8<T>(static_cast<T*>(a.C) + (size_t)m * a.ldc + c * 8, v[i]);
    }
    ss = block_sum<4>(ss, red);
    const float inv = rsqrtf(ss / (float)a.N + eps);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int c = tid + i * 256;
        if (c >= HC) continue;
        float o[8]; g[i].get(o);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = round_to<T>(v[i][e] * inv) * o[e];
        store8<T>(xn + (size_t)m * a.N + c * 8, o);
    }
}
void launch_rows_reduce_norm(int dtype, const GemmArgs& a, int S, const void* norm_w, void* xn, float eps, hipStream_t st) {
    LMX_REQUIRE(dtype != kF32 && a.N <= 8192 && !a.bias && a.act == kActNone && !a.c_f32 && !a.pk_kc, "rows_reduce_norm: a plain 16-bit linear of up to 8192 outputs");
    const int np = cdiv(a.N / 8, 256);
#define R(TT, NPV) hipLaunchKernelGGL((rows_reduce_norm_kernel<TT, NPV>), dim3(a.M), dim3(256), 0, st, a, S, (const TT*)norm_w, (TT*)xn, eps)
#define RT(TT) do { if (np == 1) R(TT, 1); else if (np == 2) R(TT, 2); else if (np == 3) R(TT, 3); else R(TT, 4); } while (0)
    if (dtype == kBF16) RT(bf16_t); else RT(f16_t);
#undef RT
#undef R
    LMX_CHECK_HIP(hipGetLastError());
}

template <typename T, int MT, int BN>
static void launch_rows_cfg(const GemmArgs& a, int mtiles, int S, hipStream_t st, bool keep) {
    constexpr int smem = rows_smem<MT, BN>();
    static_assert(smem <= 160 * 1024, "LDS");
    auto kern = gemm_rows_kernel<T, MT, BN>;
    static bool attr_set = false;
    if (!attr_set) {
        LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
        attr_set = true;
    }
    const dim3 grid(mtiles * cdiv(a.N, BN) * S);
    KernelTimer* kt = g_kernel_timer;
    if (S > 1 && !keep && kt && !kt->used) {              // an armed kernel timer spans both launches, the boundary between them included
        const dim3 rg((unsigned)cdiv64((int64_t)a.M * (act_gated(a.act) ? a.N / 2 : a.N) / 8, 256));
        kt->used = true;
        hipExtLaunchKernelGGL(kern, grid, dim3(512), smem, st, kt->e0, nullptr, 0, a, mtiles, S);
        hipExtLaunchKernelGGL(rows_reduce_kernel<T>, rg, dim3(256), 0, st, nullptr, kt->e1, 0, a, S);
    } else {
        LMX_LAUNCH(kern, grid, dim3(512), smem, st, a, mtiles, S);
        if (S > 1 && !keep) {
            const dim3 rg((unsigned)cdiv64((int64_t)a.M * (act_gated(a.act) ? a.N / 2 : a.N) / 8, 256));
            hipLaunchKernelGGL(rows_reduce_kernel<T>, rg, dim3(256), 0, st, a, S);
        }
    }
    LMX_CHECK_HIP(hipGetLastError());
}

template <typename T, int BN>
static void launch_rows_n(const GemmArgs& a, int mtiles, int S, hipStream_t st, bool keep) {
    switch (cdiv(cdiv(a.M, mtiles), 32)) {
        case 1: launch_rows_cfg<T, 1, BN>(a, mtiles, S, st, keep); break;
        case 2: launch_rows_cfg<T, 2, BN>(a, mtiles, S, st, keep); break;
        case 3: launch_rows_cfg<T, 3, BN>(a, mtiles, S, st, keep); break;
        case 4: launch_rows_cfg<T, 4, BN>(a, mtiles, S, st, keep); break;
        case 5: launch_rows_cfg<T, 5, BN>(a, mtiles, S, st, keep); break;
        case 6: launch_rows_cfg<T, 6, BN>(a, mtiles, S, st, keep); break;
        case 7: launch_rows_cfg<T, 7, BN>(a, mtiles, S, st, keep); break;
        default: launch_rows_cfg<T, 8, BN>(a, mtiles, S, st, keep); break;
    }
}

bool gemm_rows_applies(int dtype, const GemmArgs& a) {
    auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return (dtype == kBF16 || dtype == kF16) && a.K % GEMM_BK == 0 && a.N % 8 == 0 && a.ldc % 8 == 0 && al(a.C) && (!a.bias || al(a.bias)) && (!a.R || (al(a.R) && a.ldr % 8 == 0)) &&
           (!act_gated(a.act) || a.N % 64 == 0) && !a.qf_kc && (!a.pk_kc || (a.pk_D % 8 == 0 && al(a.pk_kc) && a.pk_img_stride % 8 == 0 && !a.c_f32)) && (size_t)a.M * a.ldx * 2 < ((size_t)1 << 32) && (size_t)a.N * a.ldw * 2 < ((size_t)1 << 32);
}

size_t gemm_rows_slab_bytes(int M, int N, int S) { return S > 1 ? (size_t)S * M * N * sizeof(float) : 0; }

// The form launch_gemm takes for this product: {row tiles, weight rows of a workgroup, K slices}, or row tiles 0 = not here.  LLaVA-1.5-7B's four linears (q|k|v 12288 x 4096,
// o 4096 x 4096, gate|up 22016 x 4096, down 4096 x 11008), us a launch with the reduction, weights cold: the other kernels -> here
//   rows      q|k|v        o            gate|up      down
//     20   24.4 -> 22.3  17.2 -> 12.3  67.8 -> 33.2  43.1 -> 21.9      64 weight rows (gate|up 128), slices to 256 workgroups
//    100   34.6 -> 30.7  18.6 -> 16.2  71.0 -> 43.3  48.4 -> 29.5
//    139   58.0 -> 33.7  17.4 (19.3)   70.8 -> 50.4  41.7 -> 34.9      128 weight rows, up to 6 slices; o stays where it was
//    250   58.7 -> 43.1  20.8 (25.6)   78.5 -> 62.6  53.3 -> 50.9
//    290   61.9 -> 45.4  31.7 -> 26.0  80.5 (90.4)   85.5 -> 46.5      two row tiles; gate|up (344 workgroups) stays
//    512   74.1 -> 64.3  33.6 -> 31.1  94.3 (128.7)  90.0 -> 76.0
// so: 64 weight rows up to 128 rows, where the weights are the time; 128 above, where the rows' re-reads are; no more than one workgroup per CU; slices of at least 10 slabs,
// and above 128 rows no slicing of a short K (the slabs of o cost what its weights cost).  Short products (K < 1024, under 4 M weights) are launch time on any form.
//
// Of products past the lines of the four-wave tiles (gemm4w_form) come here those with fp32 output, those that these tiles make in less time (linear_form) and all with LMX_GEMM8P=0.
//
// More rows (or what the slices above do not take): tiles of 32 .. 256 rows x 128 weight rows, as many as make ONE round of workgroups, where 256 x 256 tiles would be too few and
// small tiles several rounds (us, best other form -> here; 16-bit, weights cold):
//   2048 x 2048 x 2048  33.6 -> 23.9   1400 x 2048 x 2048  30.9 -> 20.0   2679 x 1280 x 2048  30.9 -> 22.9   600 x 4096 x 4096  40.5 -> 32.8   1087 x 4096 x 4096  51.9 -> 47.1
//   2048 x 2048 x 5632  58.8 -> 56.6   2308 x 1024 x 4096  61.2 -> 37.0   4616 x 1024 x 4096  59.1 -> 56.9   577 x 4096 x 1024   17.3 -> 13.8   2308 x 1024 x 1024   17.9 -> 14.9
// Not: long K under tiles of 160 rows and more (1087 x 4096 x 11008: 100.7 (116.4): three slices of 256 x 256 tiles read less), 160 and more tiles of 256 x 256, and the few small
// tiles of 577 x 1024 and its like (7.4, 16.9 us on 64 x 64), whose time is their chain of K steps.
//
// Where the others are the faster ones (30 weights x 24 row counts, launches back to back, weights cold; other (here)):
//   a short K in slices: the second launch costs what is saved.  257 x 3072 x 2048 10.7 (19.9), 128 x 4096 x 2048 11.9 (15.9), 256 x 8192 x 1536 16.5 (25.1); rows at 33 .. 64
//     over up to 64 tiles of 64 x 64 stay here, and up to 256 rows over more than 640: 64 x 3072 x 2048 12.2 -> 10.9, 251 x 11456 x 2304 37.3 -> 31.9;
//   one round of 64 x 64 tiles: 96 x 6656 x 4096 19.2 (21.3), 257 x 3072 x 3072 14.2 (19.7), 257 x 2560 x 5120 21.4 (24.6); two rounds: 257 x 4096 x 4096 30.4 -> 24.4;
//   256 x 256 tiles in slices where one slice leaves CUs idle: 258 x 9792 x 7296 59.4 (75.8), 183 x 18176 x 7744 84.5 (96.4).  (Where it does not they win back to back, 512 x 12288 x
//     4096 60.6 (63.5), 256 x 15360 x 5120 61.6 (65.3), 256 x 27648 x 5120 87.8 (96.7), and lose inside a prompt: 500 rows 12 us a layer of 4096, 250 rows 4 us a layer of 5120);
//   tall tiles over a short K: 2048 x 4096 x 2048 42.6 (47.8), 2308 x 3072 x 1024 21.3 (26.1); 2048 x 3072 x 2048 39.9 -> 36.0.
// Over all 720 products 1.135 times as fast as the others alone (1.115 without these lines).
RowsForm gemm_rows_form(int dtype, const GemmArgs& a) {
    const RowsForm none{0, 0, 1};
    if (a.K < 1024 || (size_t)a.N * a.K < ((size_t)1 << 20) || !gemm_rows_applies(dtype, a)) return none;
    const int nk = a.K / GEMM_BK;
    const int64_t t64 = (int64_t)cdiv(a.M, 64) * cdiv(a.N, 64);
    const int t256 = cdiv(a.M, 256) * cdiv(a.N, 256), big = t256 * gemm_slices(a);       // workgroups of the ping-pong kernel
    const bool plain = !act_gated(a.act) && !a.c_f32;                                   // (the others have one tile form for fp32 output and no small ones for gated)
    if (a.M <= 512 && (size_t)a.N * a.K >= ((size_t)4 << 20)) {
        const int mt = cdiv(a.M, 256);
        const bool few = a.M <= 128 && cdiv(a.N, 64) <= 256;
        const int bn = few ? 64 : 128, tiles = mt * cdiv(a.N, bn);
        if (tiles <= 256) {
            int s = std::min(256 / tiles, few ? 4 : mt == 2 ? 4 : 6);
            while (s > 1 && (nk / s < 10 || !a.skw || a.pk_kc || gemm_rows_slab_bytes(a.M, a.N, s) > a.skw_bytes())) --s;
            bool take = tiles * s >= 128 && (few || s <= 2 || nk >= 128 || (mt == 2 && a.M <= 384));
            if (take && plain) {
                if (a.K < 2560 && (s == 1 ? few && a.M <= 64 : (a.M <= 32 || a.M > 64 || t64 > 64) && (mt == 2 || t64 <= 640))) take = false;
                else if (few && a.M > 64 && s == 2 && t64 <= 256 && a.K < 8192) take = false;
                else if (mt == 2 && s > 1 && t64 <= (a.K <= 3072 ? 320 : 256)) take = false;
            }
            if (take && !a.c_f32 && s == 1 && a.M > 96 && tiles < (mt == 2 ? 176 : 160) && big >= 192) return none;
            if (take) return RowsForm{mt, bn, s};
        }
    }
    if (a.M <= (a.K < 2560 ? 256 : 384) || t256 >= 160 || t64 <= (a.K >= 2048 ? 320 : 512)) return none;
    const int nt = cdiv(a.N, 128), fit = 256 / nt;
    if (fit < 1 || cdiv(a.M, fit) > 256) return none;
    const int mt = cdiv(a.M, cdiv(cdiv(a.M, fit), 32) * 32), rows32 = cdiv(cdiv(a.M, mt), 32);
    if (mt * nt < 144 || (rows32 > 4 && nk > 64) || (rows32 > 3 && nk > 128)) return none;
    if (rows32 >= 7 && (a.K <= 1024 || (a.K <= 2048 && (int64_t)cdiv(a.M, 128) * cdiv(a.N, 128) > 400))) return none;
    return RowsForm{mt, 128, 1};
}

void launch_gemm_rows(int dtype, const GemmArgs& a, int mtiles, int BN, int S, hipStream_t st, bool keep) {
    LMX_REQUIRE(gemm_rows_applies(dtype, a) && mtiles >= 1 && cdiv(a.M, mtiles) <= 256 && (BN == 64 || BN == 128), "gemm_rows: shape or alignment");
    LMX_REQUIRE(S >= 1 && S <= a.K / GEMM_BK && (S == 1 || (a.skw && gemm_rows_slab_bytes(a.M, a.N, S) <= a.skw_bytes() && !a.pk_kc)), "gemm_rows: K slices");
    // every M tile covers cdiv(rows per tile, 32) * 32 rows: the tiles that start past M are left out
    mtiles = cdiv(a.M, cdiv(cdiv(a.M, mtiles), 32) * 32);
    if (dtype == kBF16) { if (BN == 64) launch_rows_n<bf16_t, 64>(a, mtiles, S, st, keep); else launch_rows_n<bf16_t, 128>(a, mtiles, S, st, keep); }
    else { if (BN == 64) launch_rows_n<f16_t, 64>(a, mtiles, S, st, keep); else launch_rows_n<f16_t, 128>(a, mtiles, S, st, keep); }
}

}  // namespace lmx
