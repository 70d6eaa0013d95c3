// Gated delta rule with a decay per key channel (kernels.h: DeltaShape).  Everything that enters the recurrence is fp32: unit norms, decays, step sizes, the state.
//
//   delta_prep_kernel    prompt rows: short convolutions and silu, unit q and k, decays, step sizes, and per chunk of 16 tokens what the recurrence needs of them
//   delta_scan_kernel    prompt rows: the recurrence, chunk by chunk, on fp32 MFMA tiles; a workgroup owns 16 columns of S (value channels), its 4 waves the key channels
//   delta_gate_kernel    prompt rows: o / rms(o) * weight * sigmoid(gate)
//   delta_decode_kernel  one new token per sequence: all of it in one launch, one workgroup per head
//
// A chunk.  With D_t the product of the chunk's decays up to token t (elementwise over key channels) and S the state before the chunk, the recurrence unrolls to
//   u_t = beta_t (v_t - (D_t k_t)^T S - sum_{s<t} A_ts u_s)      A_ts = k_t . (D_t / D_s) k_s
//   o_t = (D_t q_t)^T S + sum_{s<=t} P_ts u_s                    P_ts = q_t . (D_t / D_s) k_s
//   S'  = D_15 S + sum_s ((D_15 / D_s) k_s) u_s^T
// The quotients are products of the decays in between, never divisions, so a decay of any strength is exact to rounding.  A, P and T = (1 + diag(beta) A)^-1 diag(beta)
// (unit lower triangular: forward substitution) do not depend on S: delta_prep_kernel forms them for all chunks at once, the scan is left with U = T (V - (D k) S) and
// the products above.
//
// Decode: the read-out o = S^T q after the write equals (g S)^T q + (k . q) u, so both products of a token run over the decayed state at once and the state update is
// off the critical path.  What bounds one sequence is not bytes (2 MB on 16 heads) but memory latencies in a row: with every load requested ahead of the first wait
// 12.9 -> 10.0 us at 16 heads of 128 x 128, 54 -> 39 us at 32 sequences of 32 heads (3.4 TB/s of state).
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "moe_pick.h"
#include "gemv2.h"

namespace lmx {

// sum over the LPC lanes of a column (8, 16 or 32 consecutive lanes); every lane gets it
template <int LPC> __device__ __forceinline__ float lanes_sum(float v) {
    v = sum8(v);
    if constexpr (LPC >= 16) v += dpp_get<0x140>(v);       // mirror in 16
    if constexpr (LPC >= 32) v = fold16(v, OpSum{});
    return v;
}
__device__ __forceinline__ float softplus_f32(float z) { return z > 20.f ? z : log1pf(expf(z)); }
__device__ __forceinline__ float sigmoid_acc(float z) { return 1.f / (1.f + expf(-z)); }
__device__ __forceinline__ float decay_f32(float rate, float z) { return expf(-rate * softplus_f32(z)); }      // rate = exp(A_log)
__device__ __forceinline__ float silu_acc(float z) { return z / (1.f + expf(-z)); }

// ---------------------------------------------------------------------------------------------------------------
// prompt rows
// ---------------------------------------------------------------------------------------------------------------
constexpr int DELTA_C = 16;              // tokens of a chunk

// segment of a chunk (its index, or -1)
__device__ __forceinline__ int delta_segment(const DeltaPrefillArgs& a, int chunk) {
    int s = a.n_seg - 1;
    while (s > 0 && a.seg[s].chunk0 > chunk) --s;
    return (chunk - a.seg[s].chunk0) * DELTA_C < a.seg[s].n ? s : -1;
}

// 8 channels of token t: sum over the taps, then silu.  Inputs before the portion come from the ring, before the sequence they are zero
template <typename T>
__device__ __forceinline__ void conv_silu8(const DeltaPrefillArgs& a, const DeltaSeg& sg, int t, int c, float (&out)[8]) {
    const int taps = a.s.taps, C = a.s.channels();
    const T* w = reinterpret_cast<const T*>(a.w.conv) + c;
    const T* proj = reinterpret_cast<const T*>(a.proj) + (size_t)sg.row0 * a.ld + c;
    const T* ring = reinterpret_cast<const T*>(sg.ring) + c;
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = 0.f;
#pragma unroll 4
    for (int j = 0; j < taps; ++j) {
        const int r = t - (taps - 1) + j, p = sg.pos0 + r;
        if (p < 0) continue;
        float x[8], f[8];
        const T* src = proj + (ptrdiff_t)r * a.ld;
        if (r < 0) src = ring + (size_t)(p % taps) * C;
        load8<T>(src, x);
        load8<T>(w + (size_t)j * C, f);
#pragma unroll
        for (int e = 0; e < 8; ++e) out[e] = fmaf(x[e], f[e], out[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = silu_acc(out[e]);
}

// grid (chunks, heads), 256 threads
template <typename T, int LPC>
__global__ __launch_bounds__(256) void delta_prep_kernel(DeltaPrefillArgs a) {
    constexpr int DK = LPC * 8, C = DELTA_C, CW = DK / 16;
    extern __shared__ __attribute__((aligned(16))) float dsm[];
    float *g = dsm, *k = g + C * DK, *q = k + C * DK;        // [C][DK]; the value tile comes first in the same place, the written-out keys last
    __shared__ float A[C][C], P[C][C], beta[C];
    const int tid = threadIdx.x, H = a.s.H, G = a.s.G, DV = a.s.DV;
    const int si = __builtin_amdgcn_readfirstlane(delta_segment(a, blockIdx.x));
    if (si < 0) return;
    const DeltaSeg sg = a.seg[si];
    const int t0 = ((int)blockIdx.x - sg.chunk0) * DELTA_C;
    const int nt = sg.n - t0 < C ? sg.n - t0 : C;
    const int h = blockIdx.y, kh = h / (H / G);
    const size_t ch = (size_t)(sg.chunk0 + t0 / C) * H + h;
    // ---- values, transposed: [DV][C]
    T* vt = reinterpret_cast<T*>(dsm);
    for (int i = tid; i < C * (DV / 8); i += 256) {
        const int t = i / (DV / 8), c = (i % (DV / 8)) * 8;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 0.f;
        if (t < nt) conv_silu8<T>(a, sg, t0 + t, 2 * G * DK + h * DV + c, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) vt[(c + e) * C + t] = from_f32<T>(v[e]);
    }
    __syncthreads();
    {
        const uint4* src = reinterpret_cast<const uint4*>(dsm);
        uint4* dst = reinterpret_cast<uint4*>(reinterpret_cast<T*>(a.v) + ch * DV * C);
        for (int i = tid; i < DV * C * (int)sizeof(T) / 16; i += 256) dst[i] = src[i];
    }
    __syncthreads();
    // ---- unit q and k (rows 0..15: q, 16..31: k); tokens past the portion are zero rows with decay 1
    for (int r = tid / LPC; r < 2 * C; r += 256 / LPC) {
        const int t = r % C, c = (tid % LPC) * 8;
        const bool is_k = r >= C;
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = 0.f;
        if (t < nt) conv_silu8<T>(a, sg, t0 + t, (is_k ? G + kh : kh) * DK + c, x);
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
        ss = lanes_sum<LPC>(ss);
        const float inv = is_k ? 1.f / sqrtf(ss + 1e-6f) : 1.f / (sqrtf(ss + 1e-6f) * sqrtf((float)a.s.dk));
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] *= inv;
        store8<float>((is_k ? k : q) + t * DK + c, x);
    }
    const float rate = expf(to_f32(reinterpret_cast<const T*>(a.w.A_log)[h]));
    for (int i = tid; i < C * LPC; i += 256) {
        const int t = i / LPC, c = (i % LPC) * 8;
        float z[8], d[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) z[e] = 1.f;
        if (t < nt) {
            load8<T>(reinterpret_cast<const T*>(a.ag) + ((size_t)sg.row0 + t0 + t) * a.ag_ld + h * DK + c, z);
            load8<T>(reinterpret_cast<const T*>(a.w.dt_bias) + h * DK + c, d);
#pragma unroll
            for (int e = 0; e < 8; ++e) z[e] = decay_f32(rate, z[e] + d[e]);
        }
        store8<float>(g + t * DK + c, z);
    }
    if (tid < C) beta[tid] = tid < nt ? sigmoid_acc(to_f32(reinterpret_cast<const T*>(a.proj)[((size_t)sg.row0 + t0 + tid) * a.ld + a.s.channels() + h])) : 0.f;
    A[tid / C][tid % C] = 0.f; P[tid / C][tid % C] = 0.f;
    __syncthreads();
    // ---- A and P: 16 lanes own one key s and carry it through the decays behind it
    const int s = tid / 16, sub = tid % 16;
    float r[CW];
#pragma unroll
    for (int j = 0; j < CW / 4; ++j) {
        const float4 x = *reinterpret_cast<const float4*>(k + s * DK + j * 64 + sub * 4);
        r[j * 4] = x.x; r[j * 4 + 1] = x.y; r[j * 4 + 2] = x.z; r[j * 4 + 3] = x.w;
    }
    for (int t = (tid >> 6) * 4; t < C; ++t) {
        float ak = 0.f, aq = 0.f;
#pragma unroll
        for (int j = 0; j < CW / 4; ++j) {
            const int c = t * DK + j * 64 + sub * 4;
            const float4 gg = *reinterpret_cast<const float4*>(g + c), kk = *reinterpret_cast<const float4*>(k + c), qq = *reinterpret_cast<const float4*>(q + c);
            if (t > s) { r[j * 4] *= gg.x; r[j * 4 + 1] *= gg.y; r[j * 4 + 2] *= gg.z; r[j * 4 + 3] *= gg.w; }
            ak = fmaf(kk.x, r[j * 4], ak); ak = fmaf(kk.y, r[j * 4 + 1], ak); ak = fmaf(kk.z, r[j * 4 + 2], ak); ak = fmaf(kk.w, r[j * 4 + 3], ak);
            aq = fmaf(qq.x, r[j * 4], aq); aq = fmaf(qq.y, r[j * 4 + 1], aq); aq = fmaf(qq.z, r[j * 4 + 2], aq); aq = fmaf(qq.w, r[j * 4 + 3], aq);
        }
        ak = lanes_sum<16>(ak); aq = lanes_sum<16>(aq);
        if (sub == 0 && t >= s) { P[t][s] = aq; if (t > s) A[t][s] = ak; }
    }
    // ---- D_t k_t, D_t q_t, D_15
    {
        constexpr int PARTS = 256 / DK;
        const int c = tid % DK, part = tid / DK;
        float D = 1.f;
#pragma unroll
        for (int t = 0; t < C; ++t) {
            D *= g[t * DK + c];
            if (t % PARTS != part) continue;
            a.kd[(ch * C + t) * DK + c] = D * k[t * DK + c];
            a.qd[(ch * C + t) * DK + c] = D * q[t * DK + c];
        }
        if (part == 0) a.dc[ch * DK + c] = D;
    }
    __syncthreads();
    a.pm[ch * C * C + tid] = P[tid / C][tid % C];
    if (tid < C) {                                           // column tid of T
        float x[C];
#pragma unroll
        for (int t = 0; t < C; ++t) {
            float v = t == tid ? 1.f : 0.f;
#pragma unroll
            for (int i = 0; i < t; ++i) v = fmaf(-A[t][i], x[i], v);
            x[t] = beta[t] * v;
            a.tm[(ch * C + t) * C + tid] = x[t];
        }
    }
#pragma unroll
    for (int j = 0; j < CW; ++j) dsm[((j / 4) * 64 + sub * 4 + j % 4) * (C + 1) + s] = r[j];
    __syncthreads();
    for (int i = tid; i < DK * C; i += 256) a.kt[ch * DK * C + i] = dsm[(i / C) * (C + 1) + i % C];
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 ldg4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// grid (heads x DV / 16, segments), 256 threads: wave w owns key channels [w DK / 4, (w + 1) DK / 4) of 16 columns.  Everything is laid out so that no operand changes
// lanes: register i of lane l of an accumulator is row 4 (l / 16) + i, column l % 16, which as a B operand is k index l / 16 of the i-th of four products whose A operands
// hold columns 4 (l / 16) + i.  The waves' parts of (D k) S and of o meet in LDS.
template <typename T, int LPC>
__global__ __launch_bounds__(256, LPC <= 16 && sizeof(T) == 2 ? 2 : 1) void delta_scan_kernel(DeltaPrefillArgs a) {
    constexpr int DK = LPC * 8, NT = DK / 64, C = DELTA_C;
    __shared__ __attribute__((aligned(16))) f32x4 wb[2][4][64], ob[2][4][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int H = a.s.H, DV = a.s.DV;
    const int lid = xcd_remap(blockIdx.x, gridDim.x), nblk = DV / 16, h = lid / nblk, c0 = (lid % nblk) * 16;
    const DeltaSeg sg = a.seg[blockIdx.y];
    const int r16 = lane & 15, q4 = (lane >> 4) * 4, cb = wave * (DK / 4);
    float* st = sg.state + ((size_t)h * DV + c0 + r16) * DK + cb + q4;
    f32x4 S[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) S[j] = sg.pos0 > 0 ? ldg4(st + j * 16) : f32x4{0.f, 0.f, 0.f, 0.f};
    using Raw = std::conditional_t<sizeof(T) == 2, uint2, f32x4>;
    struct Chunk { f32x4 kd[NT], qd[NT], kt[NT], dc[NT], tm; float pm; Raw v; };
    // a chunk's base is uniform, a lane's place in it does not change: one 32-bit offset a lane for each array
    const unsigned o_kd = r16 * DK + cb + q4, o_kt = (cb + r16) * C + q4, o_dc = cb + q4, o_tm = r16 * C + q4, o_v = (c0 + r16) * C + q4;
    auto fetch = [&](int n, Chunk& x) {
        const size_t ch = (size_t)(sg.chunk0 + n) * H + h;
        const float *kd = a.kd + ch * C * DK, *qd = a.qd + ch * C * DK, *kt = a.kt + ch * DK * C, *dc = a.dc + ch * DK, *tm = a.tm + ch * C * C, *pm = a.pm + ch * C * C;
        const T* v = reinterpret_cast<const T*>(a.v) + ch * DV * C;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            x.kd[j] = ldg4(kd + o_kd + j * 16);
            x.qd[j] = ldg4(qd + o_kd + j * 16);
            x.kt[j] = ldg4(kt + o_kt + j * 16 * C);
            x.dc[j] = ldg4(dc + o_dc + j * 16);
        }
        x.tm = ldg4(tm + o_tm);
        x.pm = pm[o_tm + wave];
        x.v = *reinterpret_cast<const Raw*>(v + o_v);
    };
    // a read-out of the chunk before, one element a thread; its parts are in LDS since the barrier of this step
    const int ot = (tid >> 6) * 4 + (tid & 3), ocol = (tid >> 2) & 15;
    float* const obase = a.o + (size_t)sg.row0 * H * DV + (size_t)h * DV + c0;
    const unsigned o_o = (unsigned)ot * H * DV + ocol;
    auto put_o = [&](int n, float v) { if (n * C + ot < sg.n) (obase + (size_t)n * C * H * DV)[o_o] = v; };
    auto sum_o = [&](int n) {
        const float* p = reinterpret_cast<const float*>(&ob[n & 1][0][0]) + tid;
        return (p[0] + p[256]) + (p[512] + p[768]);
    };
    const int nc = (sg.n + C - 1) / C;
    // The chain of a chunk is W (8 products of 32 cycles), its way through LDS, U (4) and the new S (8); what does not hang on it fills the waits: O's products cover the
    // write, the barrier and the reads.  The fences keep it in this order.
    auto step = [&](int n, const Chunk& cur, auto fetch_next) {
        f32x4 W = {0.f, 0.f, 0.f, 0.f}, O = W, U = W, X;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) W = mfma4(cur.kd[j][i], S[j][i], W);
        fetch_next();
        __builtin_amdgcn_sched_barrier(0);
        constexpr int NO = NT * 4;
        auto part_o = [&](int k) { O = mfma4(cur.qd[k / 4][k % 4], S[k / 4][k % 4], O); };
        part_o(0);
        __builtin_amdgcn_sched_barrier(0);
        wb[n & 1][wave][lane] = W;
#pragma unroll
        for (int k = 1; k < NO / 2; ++k) part_o(k);
        __builtin_amdgcn_sched_barrier(0);
        // LDS only: a full barrier would also wait for the chunks that are on their way
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const f32x4 w0 = wb[n & 1][0][lane], w1 = wb[n & 1][1][lane], w2 = wb[n & 1][2][lane], w3 = wb[n & 1][3][lane];
        float o_prev = 0.f;
        if (n > 0) o_prev = sum_o(n - 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = NO / 2; k < NO; ++k) part_o(k);
        f32x4 v;
        if constexpr (sizeof(T) == 2) v = f32x4{unpack_lo<T>(cur.v.x), unpack_hi<T>(cur.v.x), unpack_lo<T>(cur.v.y), unpack_hi<T>(cur.v.y)}; else v = cur.v;
#pragma unroll
        for (int i = 0; i < 4; ++i) X[i] = v[i] - ((w0[i] + w1[i]) + (w2[i] + w3[i]));
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) S[j][i] *= cur.dc[j][i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) U = mfma4(cur.tm[i], X[i], U);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) S[j] = mfma4(cur.kt[j][i], U[i], S[j]);
        const float u = wave < 2 ? (wave == 0 ? U[0] : U[1]) : (wave == 2 ? U[2] : U[3]);
        O = mfma4(cur.pm, u, O);                             // a quarter of P U per wave
        ob[n & 1][wave][lane] = O;
        if (n > 0) put_o(n - 1, o_prev);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Two chunks in registers, one of them on its way; past the last chunk the last one is read again.  More of them gave nothing (the chain above bounds a step) and took the
    // registers of a second workgroup on the CU, which short and many sequences need.  us at 16 heads x 1100 rows / 16 heads x (1100, 890, 680) / 32 heads x 16 sequences of
    // about 50: four chunks and one workgroup 73.5 / 106 / 108, this 62 / 94 / 64
    constexpr int NB = 2;
    Chunk buf[NB];
    auto at = [&](int n) { return n < nc ? n : nc - 1; };
#pragma unroll
    for (int u = 0; u < NB - 1; ++u) fetch(at(u), buf[u]);
    int n = 0;
    for (; n + NB <= nc; n += NB)
#pragma unroll
        for (int u = 0; u < NB; ++u) step(n + u, buf[u], [&] { fetch(at(n + u + NB - 1), buf[(u + NB - 1) % NB]); });
#pragma unroll
    for (int u = 0; u < NB - 1; ++u) if (n + u < nc) step(n + u, buf[u], [] {});
    __syncthreads();
    put_o(nc - 1, sum_o(nc - 1));
#pragma unroll
    for (int j = 0; j < NT; ++j) *reinterpret_cast<f32x4*>(st + j * 16) = S[j];
    // the newest inputs of the convolutions: every channel once, spread over the segment's workgroups
    const int CH = a.s.channels(), taps = a.s.taps, keep = sg.n < taps ? sg.n : taps;
    for (int c = blockIdx.x * 256 + tid; c < CH; c += gridDim.x * 256)
        for (int j = 0; j < keep; ++j) {
            const int t = sg.n - keep + j;
            reinterpret_cast<T*>(sg.ring)[(size_t)((sg.pos0 + t) % taps) * CH + c] = reinterpret_cast<const T*>(a.proj)[((size_t)sg.row0 + t) * a.ld + c];
        }
}

// `lpv` lanes (a power of two, 8 lpv >= DV) per (row, head)
template <typename T>
__global__ __launch_bounds__(256) void delta_gate_kernel(DeltaPrefillArgs a, int pairs, int row_base, int lpv) {
    const int p = blockIdx.x * (256 / lpv) + threadIdx.x / lpv, c = (threadIdx.x % lpv) * 8, pp = p < pairs ? p : pairs - 1;      // every lane stays for the sums
    const int H = a.s.H, DV = a.s.DV, h = pp % H, cc = c < DV ? c : 0;
    const size_t row = (size_t)row_base + pp / H;
    float o[8], gate[8], w[8], ss = 0.f;
    load8<float>(a.o + (row * H + h) * DV + cc, o);
    load8<T>(reinterpret_cast<const T*>(a.ag) + row * a.ag_ld + H * a.s.DK + h * DV + cc, gate);
    load8<T>(reinterpret_cast<const T*>(a.w.norm) + cc, w);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(o[e], o[e], ss);
    ss = c < DV ? ss : 0.f;
    for (int d = lpv >> 1; d > 0; d >>= 1) ss += __shfl_xor(ss, d, 64);
    const float inv = 1.f / sqrtf(ss / (float)a.s.dv + a.eps);
    if (p >= pairs || c >= DV) return;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= inv * w[e] * sigmoid_acc(gate[e]);
    store8<T>(reinterpret_cast<T*>(a.out) + row * a.out_ld + h * DV + c, o);
}

// scratch of `rows` rows in segments that start anywhere: a launch holds up to rows / 16 + DELTA_MAX_SEG chunks
static size_t delta_regions(const DeltaShape& s, int rows, int es, size_t (&b)[8]) {
    const size_t n = ((size_t)rows / DELTA_C + DELTA_MAX_SEG) * s.H, C = DELTA_C;
    const size_t raw[8] = {n * C * s.DK * 4, n * C * s.DK * 4, n * C * s.DK * 4, n * s.DK * 4, n * C * C * 4, n * C * C * 4, n * C * s.DV * es, (size_t)rows * s.H * s.DV * 4};
    size_t sum = 0;
    for (int i = 0; i < 8; ++i) { b[i] = (raw[i] + 255) / 256 * 256; sum += b[i]; }
    return sum;
}
size_t delta_scratch_bytes(const DeltaShape& s, int rows, int es) { size_t b[8]; return delta_regions(s, rows, es, b); }
void delta_carve(DeltaPrefillArgs& a, void* scratch, int rows, int es) {
    size_t b[8];
    delta_regions(a.s, rows, es, b);
    char* p = static_cast<char*>(scratch);
    void* at[8];
    for (int i = 0; i < 8; ++i) { at[i] = p; p += b[i]; }
    a.kd = static_cast<float*>(at[0]); a.qd = static_cast<float*>(at[1]); a.kt = static_cast<float*>(at[2]); a.dc = static_cast<float*>(at[3]);
    a.tm = static_cast<float*>(at[4]); a.pm = static_cast<float*>(at[5]); a.v = at[6]; a.o = static_cast<float*>(at[7]);
}

static void delta_check(const DeltaShape& s) {
    LMX_REQUIRE(s.H >= 1 && s.G >= 1 && s.H % s.G == 0, "delta: heads must be a multiple of key heads");
    LMX_REQUIRE((s.DK == 64 || s.DK == 128 || s.DK == 256) && s.DV >= 64 && s.DV % 64 == 0 && s.dk >= 1 && s.dk <= s.DK && s.dv >= 1 && s.dv <= s.DV, "delta: bad head widths");
    LMX_REQUIRE(s.taps >= 1, "delta: at least one tap");
}
static void delta_check(const DeltaPrefillArgs& a) {
    delta_check(a.s);
    LMX_REQUIRE(a.ld % 8 == 0 && a.ld >= a.s.channels() + a.s.H && a.ag_ld % 8 == 0 && a.ag_ld >= a.s.H * (a.s.DK + a.s.DV), "delta: bad row pitch");
    LMX_REQUIRE(a.n_seg >= 1 && a.n_seg <= DELTA_MAX_SEG, "delta: 1..16 segments a launch");
    for (int i = 0, at = 0; i < a.n_seg; ++i) { LMX_REQUIRE(a.seg[i].chunk0 == at, "delta: chunks follow each other"); at += cdiv(a.seg[i].n, DELTA_C); }
    for (int i = 0; i < a.n_seg; ++i) LMX_REQUIRE(a.seg[i].n >= 1 && a.seg[i].pos0 >= 0 && a.seg[i].row0 >= 0 && a.seg[i].state && a.seg[i].ring, "delta: bad segment");
}
#define DELTA_KB(KERN, GRID, NTH, SMEM, ...) do { if (a.s.DK == 64) LMX_LAUNCH((KERN<TT, 8>), GRID, dim3(NTH), SMEM, st, __VA_ARGS__); \
                                            else if (a.s.DK == 128) LMX_LAUNCH((KERN<TT, 16>), GRID, dim3(NTH), SMEM, st, __VA_ARGS__); \
                                            else LMX_LAUNCH((KERN<TT, 32>), GRID, dim3(NTH), SMEM, st, __VA_ARGS__); } while (0)
#define DELTA_K(KERN, GRID, SMEM, ...) DELTA_KB(KERN, GRID, 256, SMEM, __VA_ARGS__)

void launch_delta_prep(int dtype, const DeltaPrefillArgs& a, hipStream_t st) {
    delta_check(a);
    int tiles = 0;
    for (int i = 0; i < a.n_seg; ++i) tiles += cdiv(a.seg[i].n, DELTA_C);
    const dim3 grid(tiles, a.s.H);
    const size_t smem = std::max((size_t)3 * DELTA_C * a.s.DK * 4, (size_t)DELTA_C * a.s.DV * dtype_size(dtype));
    LMX_REQUIRE(smem <= 60 * 1024, "delta_prep: head widths too large");
    if (dtype == kBF16) { using TT = bf16_t; DELTA_K(delta_prep_kernel, grid, smem, a); }
    else if (dtype == kF16) { using TT = f16_t; DELTA_K(delta_prep_kernel, grid, smem, a); }
    else { using TT = float; DELTA_K(delta_prep_kernel, grid, smem, a); }
    LMX_CHECK_HIP(hipGetLastError());
}
void launch_delta_scan(int dtype, const DeltaPrefillArgs& a, hipStream_t st) {
    delta_check(a);
    const dim3 grid(a.s.H * (a.s.DV / 16), a.n_seg);
    if (dtype == kBF16) { using TT = bf16_t; DELTA_K(delta_scan_kernel, grid, 0, a); }
    else if (dtype == kF16) { using TT = f16_t; DELTA_K(delta_scan_kernel, grid, 0, a); }
    else { using TT = float; DELTA_K(delta_scan_kernel, grid, 0, a); }
    LMX_CHECK_HIP(hipGetLastError());
}
void launch_delta_gate(int dtype, const DeltaPrefillArgs& a, hipStream_t st) {
    delta_check(a);
    int lpv = 8;
    while (lpv * 8 < a.s.DV) lpv <<= 1;
    LMX_REQUIRE(lpv <= 64, "delta_gate: value heads up to 512");
    for (int i = 0; i < a.n_seg;) {                          // neighbouring segments are one run of rows
        int k = i + 1, rows = a.seg[i].n;
        while (k < a.n_seg && a.seg[k].row0 == a.seg[k - 1].row0 + a.seg[k - 1].n) rows += a.seg[k++].n;
        const int pairs = rows * a.s.H;
#define L(TT) LMX_LAUNCH(delta_gate_kernel<TT>, dim3(cdiv(pairs, 256 / lpv)), dim3(256), 0, st, a, pairs, a.seg[i].row0, lpv)
        if (dtype == kBF16) L(bf16_t); else if (dtype == kF16) L(f16_t); else L(float);
#undef L
        i = k;
    }
    LMX_CHECK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------------------------
// one new token per sequence: grid (heads, sequences), NTH threads
// ---------------------------------------------------------------------------------------------------------------
template <typename T, int LPC, int NTH>
__device__ __forceinline__ void delta_decode_head(const DeltaDecodeArgs& a, int h, int z, float* sm, float* red) {
    constexpr int DK = LPC * 8, CPP = NTH / LPC, PF = 2048 / NTH, RP = 2048 / NTH;      // columns of one pass over the state, passes in flight, low-rank rows at a time
    const int tid = threadIdx.x;
    const int H = a.s.H, G = a.s.G, DV = a.s.DV, taps = a.s.taps, C = a.s.channels();
    const int rep = H / G, kh = h / rep;
    float *q = sm, *k = q + DK, *g = k + DK, *v = g + DK, *gate = v + DV, *o = gate + DV;
    const DecodeFusedSeq e = a.tab ? a.tab[z] : a.one;
    const T* row = reinterpret_cast<const T*>(a.proj) + (size_t)z * a.ld;
    float* st = reinterpret_cast<float*>(e.K) + (size_t)h * DV * DK;
    T* ring = reinterpret_cast<T*>(e.VT);
    const T* conv = reinterpret_cast<const T*>(a.w.conv);
    const int sub = tid % LPC, col = tid / LPC;
    // Everything that is read from memory is requested before anything waits: state, the first pass over the low-rank rows, inputs and weights of the convolutions (every
    // slot of the ring, so that no address waits for the position), biases, norm weights.  Addresses past an end are clamped and their values dropped.
    float S[PF][8];
#pragma unroll
    for (int p = 0; p < PF; ++p) {
        const int c = p * CPP + col;
        load8<float>(st + (size_t)(c < DV ? c : DV - 1) * DK + sub * 8, S[p]);
    }
    const int pos = *e.pos_ptr;
    const T* wdt = reinterpret_cast<const T*>(a.w.dt_bias) + h * DK;
    // decays and output gates: 8 lanes per row of the second low-rank matrices, RP rows at a time.  Rows of a wave are on one side of DK and of DK + DV (multiples of 64)
    auto low_rank = [&](int i, const T*& w, const T*& x, int& n) {
        i = i < DK + DV ? i : DK + DV - 1;
        const bool is_g = __builtin_amdgcn_readfirstlane(i) < DK;
        w = reinterpret_cast<const T*>(a.wag) + (size_t)(is_g ? h * DK + i : H * DK + h * DV + i - DK) * a.wag_ld + (is_g ? 0 : a.ra);
        x = row + a.a_off + (is_g ? 0 : a.ra);
        n = is_g ? a.ra : a.rg;
    };
    const int c8 = (tid & 7) * 8;
    Chunk8<T> wf[RP][2], xf[RP][2];
    float bias[RP];
#pragma unroll
    for (int m = 0; m < RP; ++m) {
        const T *w, *x;
        int n;
        low_rank((tid >> 3) + m * (NTH / 8), w, x, n);
        const int c1 = n > 64 ? c8 + 64 : c8;
        wf[m][0].load(w + c8); wf[m][1].load(w + c1); xf[m][0].load(x + c8); xf[m][1].load(x + c1);
        const int i = (tid >> 3) + m * (NTH / 8);
        bias[m] = to_f32(wdt[i < DK ? i : DK - 1]);
    }
    const int n_conv = 2 * DK + DV;
    auto channel = [&](int i) { return i >= 2 * DK ? 2 * G * DK + h * DV + i - 2 * DK : (i < DK ? kh * DK + i : (G + kh) * DK + i - DK); };
    constexpr int RT = 4;                                    // a ring of up to so many taps is read whole
    const int ci = channel(tid < n_conv ? tid : n_conv - 1);
    const T x_new = row[ci];
    T rv[RT], cv[RT];
#pragma unroll
    for (int j = 0; j < RT; ++j) {
        const int t = j < taps ? j : taps - 1;
        rv[j] = ring[(size_t)t * C + ci];
        cv[j] = conv[(size_t)t * C + ci];
    }
    const T beta_in = row[C + h], rate_in = reinterpret_cast<const T*>(a.w.A_log)[h], norm_w = reinterpret_cast<const T*>(a.w.norm)[tid < DV ? tid : DV - 1];
    const bool frozen = e.done && *e.done != 0;
    const float beta = sigmoid_acc(to_f32(beta_in));
    const float rate = expf(to_f32(rate_in));
    for (int i0 = tid >> 3; i0 < DK + DV; i0 += 256) {
        const bool first = i0 == tid >> 3;
        const T *w[RP], *x[RP];
        int n[RP];
        float s[RP] = {};
#pragma unroll
        for (int m = 0; m < RP; ++m) low_rank(i0 + m * (NTH / 8), w[m], x[m], n[m]);
        if (first) {
#pragma unroll
            for (int m = 0; m < RP; ++m)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    if (u == 1 && n[m] <= 64) continue;
                    float f[8], y[8]; wf[m][u].get(f); xf[m][u].get(y);
#pragma unroll
                    for (int e2 = 0; e2 < 8; ++e2) s[m] = fmaf(f[e2], y[e2], s[m]);
                }
        }
        const int most = a.ra > a.rg ? a.ra : a.rg;
#pragma unroll 2
        for (int c = c8 + (first ? 128 : 0); c < most; c += 64)
#pragma unroll
            for (int m = 0; m < RP; ++m) {
                if (c >= n[m]) continue;
                float f[8], y[8]; load8<T>(w[m] + c, f); load8<T>(x[m] + c, y);
#pragma unroll
                for (int e2 = 0; e2 < 8; ++e2) s[m] = fmaf(f[e2], y[e2], s[m]);
            }
#pragma unroll
        for (int m = 0; m < RP; ++m) {
            const int i = i0 + m * (NTH / 8);
            s[m] = round_to<T>(lanes_sum<8>(s[m]));          // the prompt path stores this product in the model dtype
            if ((tid & 7) != 0 || i >= DK + DV) continue;
            if (i < DK) g[i] = decay_f32(rate, s[m] + (first ? bias[m] : to_f32(wdt[i])));
            else gate[i - DK] = sigmoid_acc(s[m]);
        }
    }
    // ---- short convolutions: thread per channel; the ring slot of this position is not one that any tap reads
    const int slot = pos % taps;
    for (int i = tid; i < n_conv; i += NTH) {
        const bool is_v = i >= 2 * DK;
        const int c = channel(i);
        T xin;
        float s;
        if (i == tid && taps <= RT) {
            xin = x_new;
            const int last = taps - 1;
            const float r0 = to_f32(rv[0]), r1 = to_f32(rv[1]), r2 = to_f32(rv[2]), r3 = to_f32(rv[3]), w0 = to_f32(cv[0]), w1 = to_f32(cv[1]), w2 = to_f32(cv[2]), w3 = to_f32(cv[3]);
            s = to_f32(xin) * (last == 0 ? w0 : last == 1 ? w1 : last == 2 ? w2 : w3);
#pragma unroll
            for (int j = 1; j < RT; ++j) {
                if (j >= taps || pos - j < 0) continue;
                const int sl = slot >= j ? slot - j : slot - j + taps, t = last - j;
                s = fmaf(sl == 0 ? r0 : sl == 1 ? r1 : sl == 2 ? r2 : r3, t == 0 ? w0 : t == 1 ? w1 : w2, s);
            }
        } else {
            xin = row[c];
            s = to_f32(xin) * to_f32(conv[(size_t)(taps - 1) * C + c]);
            for (int j = 1, sl = slot; j < taps; ++j) {
                sl = sl == 0 ? taps - 1 : sl - 1;
                if (pos - j >= 0) s = fmaf(to_f32(ring[(size_t)sl * C + c]), to_f32(conv[(size_t)(taps - 1 - j) * C + c]), s);
            }
        }
        if (is_v || h % rep == 0) ring[(size_t)slot * C + c] = xin;
        s = silu_acc(s);
        if (is_v) v[i - 2 * DK] = round_to<T>(s); else sm[i] = s;      // (values: the prompt path stores them in the model dtype)
    }
    __syncthreads();
    // every lane group has whole q and k: unit vectors and their product without another round
    float kr[8], qr[8], gr[8], qq = 0.f, kk = 0.f, kq = 0.f;
    load8<float>(k + sub * 8, kr); load8<float>(q + sub * 8, qr); load8<float>(g + sub * 8, gr);
#pragma unroll
    for (int n = 0; n < 8; ++n) { qq = fmaf(qr[n], qr[n], qq); kk = fmaf(kr[n], kr[n], kk); }
    qq = lanes_sum<LPC>(qq); kk = lanes_sum<LPC>(kk);
    const float qi = 1.f / (sqrtf(qq + 1e-6f) * sqrtf((float)a.s.dk)), ki = 1.f / sqrtf(kk + 1e-6f);
#pragma unroll
    for (int n = 0; n < 8; ++n) { qr[n] *= qi; kr[n] *= ki; kq = fmaf(qr[n], kr[n], kq); }
    kq = lanes_sum<LPC>(kq);
    float ss = 0.f;
    auto column = [&](float (&s)[8], int c) {
        float r0 = 0.f, r1 = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int n = 0; n < 8; n += 2) {
            s[n] *= gr[n]; s[n + 1] *= gr[n + 1];
            r0 = fmaf(s[n], kr[n], r0); r1 = fmaf(s[n + 1], kr[n + 1], r1);
            o0 = fmaf(s[n], qr[n], o0); o1 = fmaf(s[n + 1], qr[n + 1], o1);
        }
        const float r = lanes_sum<LPC>(r0 + r1), oo = lanes_sum<LPC>(o0 + o1);
        const float u = beta * (v[c] - r);
#pragma unroll
        for (int n = 0; n < 8; ++n) s[n] = fmaf(kr[n], u, s[n]);
        const float out = fmaf(kq, u, oo);
        if (sub == 0) { o[c] = out; ss += out * out; }
        if (!frozen) store8<float>(st + (size_t)c * DK + sub * 8, s);
    };
    for (int c0 = 0; c0 < DV; c0 += PF * CPP) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            const int c = c0 + p * CPP + col;
            if (c < DV) column(S[p], c);                     // uniform in a lane group
        }
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            const int c = c0 + (PF + p) * CPP + col;
            if (c < DV) load8<float>(st + (size_t)c * DK + sub * 8, S[p]);
        }
    }
    ss = block_sum<NTH / 64>(ss, red);                       // (its barriers also publish o)
    const float inv = 1.f / sqrtf(ss / (float)a.s.dv + a.eps);
    T* out = reinterpret_cast<T*>(a.out) + (size_t)z * a.out_ld + h * DV;
    for (int c = tid; c < DV; c += NTH) out[c] = from_f32<T>(o[c] * inv * to_f32(c == tid ? norm_w : reinterpret_cast<const T*>(a.w.norm)[c]) * gate[c]);
}

template <typename T, int LPC, int NTH>
__global__ __launch_bounds__(NTH, NTH == 512 && sizeof(T) == 2 ? 4 : 1) void delta_decode_kernel(DeltaDecodeArgs a) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    __shared__ float red[NTH / 64];
    if ((int)blockIdx.x == a.s.H) { moe_router_row<T, NTH / 64>(a.router, blockIdx.y); return; }
    delta_decode_head<T, LPC, NTH>(a, blockIdx.x, blockIdx.y, sm, red);
}

// One sequence's step beside a linear that reads the layer's normalised row too (a parallel layer's gate | up): the heads' workgroups are the first of the launch, the linear's, sixteen
// waves of R rows, follow.  The step is a chain of latencies on 16 .. 32 CUs, the linear a stream that wants the others; in launches of their own each waits for the other's end.
template <typename T, int LPC, int R>
__global__ __launch_bounds__(1024) void delta_decode_linear_kernel(DeltaDecodeArgs a, GemvArgs g) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    __shared__ float red[16];
    if ((int)blockIdx.x < a.s.H) delta_decode_head<T, LPC, 1024>(a, blockIdx.x, 0, sm, red);
    else gemv2_body<T, R, 4, 1, false, false, 16>(g, (int)blockIdx.x - a.s.H, reinterpret_cast<char*>(sm), nullptr, 0u);
}

static bool joined_one_round(int heads, int rows) { return cdiv(rows, 64) + heads <= 256; }      // four rows a wave of the linear beside the step
static bool one_round(const DeltaShape& s, int n_seq) { return s.H * n_seq <= 256; }
// past one round the routers are a tail of their own: 32 x 32 heads x sequences 39.1 us without, 50.4 with them, 9.8 alone; in one round (16 x 1) 9.9 either way, 8.1 alone.  On the line,
// where the routers' own workgroups are the ones past the round, they still cost less than their launches: a decode step with two of them, 16 x 16 728 us in the step's launch, 734 in
// their own; 32 x 8 1458, 1461
bool delta_decode_routes(const DeltaShape& s, int n_seq) { return one_round(s, n_seq); }
static size_t delta_decode_smem(const DeltaShape& s) { return (size_t)(3 * s.DK + 3 * s.DV) * 4; }
static void delta_decode_check(const DeltaDecodeArgs& a) {
    delta_check(a.s);
    LMX_REQUIRE(a.ra % 64 == 0 && a.rg % 64 == 0 && a.ra >= 64 && a.rg >= 64 && a.wag_ld >= a.ra + a.rg && a.wag_ld % 8 == 0, "delta_decode: low-rank widths in whole 64-column groups");
    LMX_REQUIRE(a.a_off >= a.s.channels() + a.s.H && a.ld >= a.a_off + a.ra + a.rg, "delta_decode: bad row pitch");
    LMX_REQUIRE(a.n_seq >= 1 && (a.tab || (a.n_seq == 1 && a.one.K && a.one.VT && a.one.pos_ptr)), "delta_decode: bad sequence");
    LMX_REQUIRE(delta_decode_smem(a.s) <= 60 * 1024 && a.a_off % 8 == 0, "delta_decode: head widths too large");
}
void launch_delta_decode(int dtype, const DeltaDecodeArgs& a, hipStream_t st) {
    delta_decode_check(a);
    check_router(a.router);
    const dim3 grid(a.s.H + (a.router.x ? 1 : 0), a.n_seq);
    const size_t smem = delta_decode_smem(a.s);
#define L(TT, NTH) do { if (a.s.DK == 64) LMX_LAUNCH((delta_decode_kernel<TT, 8, NTH>), grid, dim3(NTH), smem, st, a); \
                        else if (a.s.DK == 128) LMX_LAUNCH((delta_decode_kernel<TT, 16, NTH>), grid, dim3(NTH), smem, st, a); \
                        else LMX_LAUNCH((delta_decode_kernel<TT, 32, NTH>), grid, dim3(NTH), smem, st, a); } while (0)
#define LN(TT) do { if (wide) L(TT, 1024); else L(TT, 512); } while (0)
    // 1024 threads a head while every workgroup has a CU of its own; past that two workgroups of 512 on a CU, whose reads and arithmetic overlap.  us at 16 x 16 / 16 x 24 /
    // 32 x 32 heads x sequences: 1024 threads 13.8 / 22.5 / 45.4, 512 threads 15.9 / 20.0 / 40.5 (bf16 at 128 registers: 20 bytes a lane in scratch at DK 256, none at 128; f16 none)
    const bool wide = one_round(a.s, a.n_seq);
    LMX_REQUIRE(wide || !a.router.x, "delta_decode: no router here");
    if (dtype == kBF16) LN(bf16_t); else if (dtype == kF16) LN(f16_t); else LN(float);
#undef LN
#undef L
    LMX_CHECK_HIP(hipGetLastError());
}

// Where the shared launch takes less than the two (us a layer of one token, two launches -> one; heads of 128):
//   one round of workgroups (four rows a wave)   N x K  8192 x 2048 31.3 -> 26.8   11264 x 4096 64.0 -> 58.6   11264 x 8192 154.3 -> 150.7,
//     but few workgroups with long rows are the longer of the two:   1024 x 4096 44.4 : 45.8   5632 x 5120 67.8 : 68.1   1024 x 8192 118.2 : 126.1   (5632 x 4096 53.3 : 51.3, 1024 x 3072 32.7 : 32.4)
//   several rounds (two rows a wave)   16384 x 2048 39.0 -> 36.0   22016 x 3072 63.2 -> 58.3   18432 x 4608 91.0 -> 87.4   22016 x 6144 134.9 -> 132.0   18432 x 7168 148.6 -> 148.1,
//     but the launch of its own streams faster, by more than the step the more there is:   32768 x 6144 165.4 : 166.0   22016 x 7168 161.8 : 164.6, and with rows a multiple of 8 KiB apart at
//     once:   16384 x 4096 73.7 : 74.8   32768 x 4096 108.3 : 112.4   22016 x 8192 197.9 : 204.3
//   heads of 256, whose step is twice as long   11264 x 2048 43.5 -> 35.5   22016 x 4096 95.1 -> 87.7   1024 x 4096 55.8 -> 51.6;   32768 x 8192 250 : 254
// More than 64 heads: 96 of 64 beside 22016 x 4096 93.4 either way.
bool delta_decode_joins(int dtype, const DeltaShape& s, const GemvArgs& g) {
    if (s.H > 64 || g.K > 8192 || !gemv2_applies(dtype, g)) return false;
    const bool bounded = (size_t)g.N * g.K <= ((size_t)1 << 27);
    if (s.DK == 256 && g.K <= 4096) return bounded;
    if (joined_one_round(s.H, g.N)) return g.K <= 3072 || g.N >= 6144;
    return bounded && g.K % 4096 != 0;
}
void launch_delta_decode_linear(int dtype, const DeltaDecodeArgs& a, const GemvArgs& g, hipStream_t st) {
    delta_decode_check(a);
    LMX_REQUIRE(a.n_seq == 1 && !a.tab && !a.router.x && delta_decode_joins(dtype, a.s, g) && !g.norm_w, "delta_decode_linear: one sequence, a plain linear of the weight stream");
    LMX_REQUIRE(!act_gated(g.act) || g.N % 64 == 0, "delta_decode_linear: gated rows come in groups of 64");
    // four rows a wave where that leaves every workgroup a CU of its own (all of a row of 2048 is on the wire at once), two where the workgroups come in rounds: a layer of one token at four
    // rows / two  11264 x 2048 29.5 / 29.9 us   16384 x 3072 51.4 / 51.9   22016 x 4096 82.7 / 83.1, but  32768 x 6144 165.4 / 163.3
    const bool four = joined_one_round(a.s.H, g.N);
    const size_t smem = std::max(delta_decode_smem(a.s), gemv2_smem_bytes(g.K, 2, 16));
    const dim3 grid(a.s.H + cdiv(g.N, four ? 64 : 32));
#define L(TT, LPC) do { if (four) LMX_LAUNCH((delta_decode_linear_kernel<TT, LPC, 4>), grid, dim3(1024), smem, st, a, g); \
                        else LMX_LAUNCH((delta_decode_linear_kernel<TT, LPC, 2>), grid, dim3(1024), smem, st, a, g); } while (0)
#define LD(TT) do { if (a.s.DK == 64) L(TT, 8); else if (a.s.DK == 128) L(TT, 16); else L(TT, 32); } while (0)
    if (dtype == kBF16) LD(bf16_t); else LD(f16_t);
#undef LD
#undef L
    LMX_CHECK_HIP(hipGetLastError());
}

}  // namespace lmx
