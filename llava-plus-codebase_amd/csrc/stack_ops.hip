// Kernels of the layer-stack decoders (stack.cpp): models described layer by layer, with an fp32 residual stream, norms on both sides of a sublayer, per-head
// query / key norms, partial rotary positions, sliding windows, a softmax sink and output gates.  Every size and constant is an argument.
//
//   residual_norm_kernel       x <- x + m rms_norm(y) w_post (+ injected row), xn <- rms_norm(x) w_pre : one launch between any two linears of a prefill / batch
//   qkv_norm_rope_kv_kernel    query / key norm, rotation, KV append of a prompt portion (q stays in its row, k rows and V^T columns go to the caches)
//   rows_attn_kernel           any dtype, VALU: one workgroup per (row, head); the fp32 engine's prefill and head widths past the MFMA kernel's
//   decode_win_kernel          one new token per sequence: query / key norm, rotation, append, attention over the window, sink, gate, split merge in one launch
// (16-bit prefill attention with head widths up to 128 is flash_prefill2_kernel's windowed form, attention.hip.)
//
// Head vectors are stored padded to D in {64, 128, 256} lanes: the padding weights are zero, so padded lanes of q, k and v are zero and add nothing; the query / key
// norm divides by the true width.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "attention_batch.h"
#include "attention_decode.h"

namespace lmx {

// ---------------------------------------------------------------------------------------------------------------
// residual + norms
// ---------------------------------------------------------------------------------------------------------------
// AHEAD: both norms' weights and the injected row are on their way with the rows, four experts' rows at a time (each behind the sum in front of it was a trip to memory of its own)
template <typename T, int NP, bool AHEAD>
__global__ __launch_bounds__(256) void residual_norm_kernel(ResidualNormArgs a) {
    __shared__ float red[4];
    const int row = blockIdx.x, tid = threadIdx.x, HC = a.H >> 3;
    const float rH = 1.f / (float)a.H_real;
    const float* xin = a.x_in ? a.x_in + (size_t)row * a.H : nullptr;
    const T* y = a.y ? reinterpret_cast<const T*>(a.y) + (size_t)row * a.H : nullptr;
    const T* inj = a.inject ? reinterpret_cast<const T*>(a.inject) + (size_t)row * a.H : nullptr;
    const T* post = y || a.top > 0 ? reinterpret_cast<const T*>(a.post_w) : nullptr;
    const T* pre = reinterpret_cast<const T*>(a.pre_w);
    float x[NP][8], yv[NP][8];
    Chunk8<T> gp[NP], gn[NP], gi[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int c = tid + i * 256;
        if (!AHEAD || c >= HC) continue;
        if (post) gp[i].load(post + c * 8);
        if (pre) gn[i].load(pre + c * 8);
        if (inj) gi[i].load(inj + c * 8);
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int c = tid + i * 256;
        if (c >= HC) continue;
        if (xin) load8<float>(xin + c * 8, x[i]);
        else {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[i][e] = 0.f;
        }
        if (y) load8<T>(y + c * 8, yv[i]);
        else {
#pragma unroll
            for (int e = 0; e < 8; ++e) yv[i][e] = 0.f;
        }
        constexpr int KE = AHEAD ? 4 : 1;
        for (int k0 = 0; k0 < a.top; k0 += KE) {
            Chunk8<T> m[KE];
            float wk[KE];
#pragma unroll
            for (int k = 0; k < KE; ++k) {
                const size_t slot = (size_t)row * a.top + (k0 + k < a.top ? k0 + k : k0);
                wk[k] = a.moe_w[slot];
                m[k].load(reinterpret_cast<const T*>(a.moe_y) + slot * a.H + c * 8);
            }
#pragma unroll
            for (int k = 0; k < KE; ++k) {
                if (k0 + k >= a.top) continue;
                float v[8]; m[k].get(v);
#pragma unroll
                for (int e = 0; e < 8; ++e) yv[i][e] = fmaf(wk[k], v[e], yv[i][e]);
            }
        }
        if (post) {
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += yv[i][e] * yv[i][e];
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[i][e] += a.mult * yv[i][e];
        }
    }
    if (post) {
        ss = block_sum<4>(ss, red);
        const float inv = a.mult / sqrtf(ss * rH + a.eps);
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int c = tid + i * 256;
            if (c >= HC) continue;
            if (!AHEAD) gp[i].load(post + c * 8);
            float g[8]; gp[i].get(g);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[i][e] += yv[i][e] * inv * g[e];
        }
    }
    float s2 = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int c = tid + i * 256;
        if (c >= HC) continue;
        if (inj) {
            if (!AHEAD) gi[i].load(inj + c * 8);
            float g[8]; gi[i].get(g);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[i][e] += g[e];
        }
        if (a.x_out) store8<float>(a.x_out + (size_t)row * a.H + c * 8, x[i]);
#pragma unroll
        for (int e = 0; e < 8; ++e) s2 += x[i][e] * x[i][e];
    }
    T* xn = reinterpret_cast<T*>(a.xn) + (size_t)row * (a.xn_ld ? a.xn_ld : a.H);
    if (a.cast) {
#pragma unroll
        for (int i = 0; i < NP; ++i) { const int c = tid + i * 256; if (c < HC) store8<T>(xn + c * 8, x[i]); }
        return;
    }
    if (!pre) return;
    s2 = block_sum<4>(s2, red);
    const float inv2 = 1.f / sqrtf(s2 * rH + a.eps);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const int c = tid + i * 256;
        if (c >= HC) continue;
        if (!AHEAD) gn[i].load(pre + c * 8);
        float g[8], o[8]; gn[i].get(g);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = x[i][e] * inv2 * g[e];
        store8<T>(xn + c * 8, o);
    }
}

// ---------------------------------------------------------------------------------------------------------------
// input rows of a model whose embedding depends on the token before: x = embed[t] + bigram[(prev mul_prev + t mul_cur) mod buckets] (row `buckets` without a previous
// token), summed in fp32.  One workgroup per row.
// ---------------------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void embed_rows_kernel(EmbedRowsArgs a) {
    const int row = blockIdx.x, tid = threadIdx.x;
    int64_t t, prev = -1;
    if (a.tab) { t = *a.tab[row].tok; prev = *a.tab[row].prev; }
    else if (a.ids) {
        t = a.ids[row];
        if (row > 0) prev = a.ids[row - 1];
        else if (a.prev_id) prev = *a.prev_id;
        else if (a.prev_tok) prev = *a.prev_tok;
    } else { t = *a.tok; prev = *a.prev_tok; }
    t = t < 0 ? 0 : (t >= a.vocab ? a.vocab - 1 : t);
    int64_t b = a.buckets;
    if (prev >= 0) {
        b = (prev * a.mul_prev + t * a.mul_cur) % a.buckets;
        if (b < 0) b += a.buckets;
    }
    const T* e = reinterpret_cast<const T*>(a.embed) + (size_t)t * a.H;
    const T* g = reinterpret_cast<const T*>(a.bigram) + (size_t)b * a.H;
    for (int c = tid; c < (a.H >> 3); c += 256) {
        float v[8], u[8];
        load8<T>(e + c * 8, v); load8<T>(g + c * 8, u);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] += u[i];
        store8<float>(a.x + (size_t)row * a.H + c * 8, v);
        if (a.x0) store8<T>(reinterpret_cast<T*>(a.x0) + (size_t)row * a.x0_ld + c * 8, v);
    }
}

void launch_embed_rows(int dtype, const EmbedRowsArgs& a, int rows, hipStream_t st) {
    LMX_REQUIRE(a.embed && a.bigram && a.x && a.buckets >= 1 && a.H % 8 == 0 && a.vocab >= 1, "embed_rows: bad arguments");
    LMX_REQUIRE(a.tab || a.ids || (rows == 1 && a.tok && a.prev_tok), "embed_rows: no tokens");
    LMX_REQUIRE(!a.x0 || a.x0_ld % 8 == 0, "embed_rows: bad pitch");
    if (rows <= 0) return;
#define L(TT) LMX_LAUNCH(embed_rows_kernel<TT>, dim3(rows), dim3(256), 0, st, a)
    if (dtype == kBF16) L(bf16_t); else if (dtype == kF16) L(f16_t); else L(float);
#undef L
    LMX_CHECK_HIP(hipGetLastError());
}

// Loads ahead: fewer trips to memory a row, but registers for fewer rows on a CU.  16-bit rows of up to 2048 either way eight, of up to 4096 six for eight, of up to 8192 three for six: not
// where the rows are one round without and two with it, past 4096 nor where they are few rounds (with an injected row, one trip more, a round fewer; from 3073 to 4096 always).  us without /
// with, rows from L2 and, in brackets, from memory:  128 x 4096 4.2 / 3.5, 512 x 4096 6.4 / 5.8 (8.0 / 7.3), 1700 x 3072 11.9 / 12.1 (13.8 / 14.7), 1664 x 2560 10.6 / 11.1 and injected
// 10.4 / 11.1, 2560 x 4096 21.7 / 20.6 (25.1 / 23.7), 1664 x 4096 injected 15.5 / 14.3;  512 x 8192 11.4 / 10.6, 1024 x 8192 18.6 / 19.0, 1536 x 8192 24.4 / 26.7 (888 x 8192 18.7 / 19.9),
// 2560 x 8192 40.7 / 42.2 and injected 44.1 / 43.0, 4096 x 8192 84.3 / 80.5.  fp32 rows keep twice as much on the way: ahead only in one round.
bool residual_norm_ahead(int dtype, const ResidualNormArgs& a, int rows) {
    const int np = (a.H / 8 + 255) / 256;
    if (dtype == kF32) return rows <= (np == 1 ? 1792 : np == 2 ? 1024 : 512);
    if (np == 1) return true;
    if (np == 2) return rows <= 1536 || rows > 2048 || (a.inject && a.H > 3072);
    return rows <= 768 || rows > (a.inject ? 1536 : 2560);
}
void launch_residual_norm(int dtype, const ResidualNormArgs& a, int rows, hipStream_t st) {
    LMX_REQUIRE(a.H % 8 == 0 && a.H > 0 && a.H <= 8192 && a.H_real >= 1 && a.H_real <= a.H, "residual_norm: width must be a multiple of 8, at most 8192");
    LMX_REQUIRE(a.top >= 0 && (a.top == 0 || (a.moe_y && a.moe_w)), "residual_norm: expert outputs need their weights");
    LMX_REQUIRE((!a.pre_w && !a.cast) || a.xn, "residual_norm: the normalised rows need a buffer");
    LMX_REQUIRE(!(a.pre_w && a.cast) && a.xn_ld % 8 == 0, "residual_norm: norm or cast, in 16-byte rows");
    if (rows <= 0) return;
    const int np = (a.H / 8 + 255) / 256;
#define R(TT, NPV) do { if (residual_norm_ahead(dtype, a, rows)) LMX_LAUNCH((residual_norm_kernel<TT, NPV, true>), dim3(rows), dim3(256), 0, st, a); \
                        else LMX_LAUNCH((residual_norm_kernel<TT, NPV, false>), dim3(rows), dim3(256), 0, st, a); } while (0)
#define RT(TT) do { if (np == 1) R(TT, 1); else if (np == 2) R(TT, 2); else R(TT, 4); } while (0)
    if (dtype == kBF16) RT(bf16_t); else if (dtype == kF16) RT(f16_t); else RT(float);
#undef RT
#undef R
    LMX_CHECK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------------------------
// query / key norm + rotation + KV append of prompt rows.  grid (ceil(T / 64), H + 2 G), 256 threads.
//   PAIRED (rot_dims % 16 == 0): D / 16 lanes own one head vector, two 8-element chunks each — a chunk of the rotated part with its partner half a rotation away, or two
//   neighbouring chunks of the rest — so a lane rotates what it loaded: no LDS, no barrier.
//   otherwise: D / 8 lanes, 8 consecutive elements each, the partner i +- rot_dims / 2 through LDS (any even number of rotated dimensions).
// V^T behind the last row is cleared to the end of its 64 keys (or to zero_to).
// ---------------------------------------------------------------------------------------------------------------
template <typename T, int D, bool PAIRED>
__device__ __forceinline__ void qkv_norm_rope_body(const QkvNormRopeArgs& a, const int block, char* smem) {
    const int tid = threadIdx.x;
    const int tok0 = block * 64, slot = blockIdx.y;
    const int ntok = (a.T - tok0) < 64 ? (a.T - tok0) : 64;                // <= 0: a block of nothing but rows to clear
    const int nzero = (a.zero_to - tok0) < 64 ? (a.zero_to - tok0) : 64;
    T* qkv = reinterpret_cast<T*>(a.qkv);
    constexpr int LPV = D / 8, VPP = 256 / LPV;          // lanes per vector, vectors per pass
    if (PAIRED && slot < a.n_heads + a.n_kv_heads) {
        constexpr int LP = D / 16, ITER = 64 * LP / 256;
        const bool is_k = slot >= a.n_heads;
        const int half8 = a.rot_dims >> 4, k = tid % LP;                   // rotated chunks per half
        const bool rot = k < half8;
        const int c0 = rot ? k : 2 * half8 + 2 * (k - half8), c1 = rot ? k + half8 : c0 + 1;
        const T* nw = reinterpret_cast<const T*>(is_k ? a.k_norm : a.q_norm);
        T* kc = reinterpret_cast<T*>(a.K) + (size_t)(is_k ? slot - a.n_heads : 0) * a.s_max * D;
        float x[ITER][2][8], g0[8], g1[8];
#pragma unroll
        for (int it = 0; it < ITER; ++it) {
            const int t = it * (256 / LP) + tid / LP;
            const T* xp = qkv + (size_t)(t < ntok ? tok0 + t : a.T - 1) * a.qkv_stride + slot * D;
            load8<T>(xp + c0 * 8, x[it][0]); load8<T>(xp + c1 * 8, x[it][1]);
        }
        if (nw) { load8<T>(nw + c0 * 8, g0); load8<T>(nw + c1 * 8, g1); }
#pragma unroll
        for (int it = 0; it < ITER; ++it) {
            const int t = it * (256 / LP) + tid / LP;
            const bool live = t < ntok;
            float (&u)[8] = x[it][0];
            float (&v)[8] = x[it][1];
            if (nw) {
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += u[e] * u[e] + v[e] * v[e];
#pragma unroll
                for (int o = LP / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
                const float inv = 1.f / sqrtf(ss / (float)a.qk_dim + a.eps);
#pragma unroll
                for (int e = 0; e < 8; ++e) { u[e] *= inv * g0[e]; v[e] *= inv * g1[e]; }
            }
            const int pos = a.pos0 + tok0 + t;
            if (!live && is_k && t < nzero) {
#pragma unroll
                for (int e = 0; e < 8; ++e) { u[e] = 0.f; v[e] = 0.f; }
                store8<T>(kc + (size_t)pos * D + c0 * 8, u); store8<T>(kc + (size_t)pos * D + c1 * 8, v);
            }
            if (!live) continue;
            if (rot) {
                const float* cs = a.cos_sin + (size_t)pos * a.rot_dims + k * 8;
                float c[8], s[8];
                load8<float>(cs, c); load8<float>(cs + half8 * 8, s);
#pragma unroll
                for (int e = 0; e < 8; ++e) { const float p = u[e], q = v[e]; u[e] = p * c[e] - q * s[e]; v[e] = q * c[e] + p * s[e]; }
            }
            T* o = is_k ? kc + (size_t)pos * D : qkv + (size_t)(tok0 + t) * a.qkv_stride + slot * D;
            store8<T>(o + c0 * 8, u); store8<T>(o + c1 * 8, v);
        }
        return;
    }
    if (slot < a.n_heads + a.n_kv_heads) {
        float* vec = reinterpret_cast<float*>(smem);     // [VPP][D] normalised vectors of this pass
        const bool is_k = slot >= a.n_heads;
        const int sub = tid % LPV, v = tid / LPV, i0 = sub * 8;
        const T* nw = reinterpret_cast<const T*>(is_k ? a.k_norm : a.q_norm);
        T* kc = reinterpret_cast<T*>(a.K) + (size_t)(is_k ? slot - a.n_heads : 0) * a.s_max * D;
        const int half = a.rot_dims >> 1;
        for (int t0 = 0; t0 < 64; t0 += VPP) {
            const int t = t0 + v;
            const bool live = t < ntok;
            T* xp = qkv + (size_t)(tok0 + (live ? t : 0)) * a.qkv_stride + slot * D + i0;
            float x[8]; load8<T>(xp, x);
            if (nw) {
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
#pragma unroll
                for (int o = LPV / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
                const float inv = 1.f / sqrtf(ss / (float)a.qk_dim + a.eps);
                float g[8]; load8<T>(nw + i0, g);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = x[e] * inv * g[e];
            }
            __syncthreads();                             // the previous pass has been read
            store8<float>(vec + v * D + i0, x);
            __syncthreads();
            const int pos = a.pos0 + tok0 + (live ? t : 0);
            const float* cs = a.cos_sin + (size_t)pos * a.rot_dims;
            if (i0 < a.rot_dims) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int i = i0 + e;
                    if (i >= a.rot_dims) continue;
                    const bool lo = i < half;
                    const int j = lo ? i : i - half;
                    const float p = vec[v * D + (lo ? i + half : i - half)];
                    x[e] = x[e] * cs[j] + (lo ? -p : p) * cs[half + j];
                }
            }
            if (!live) continue;
            store8<T>(is_k ? kc + (size_t)pos * D + i0 : xp, x);
        }
        return;
    }
    // ---- v: [tok][D] -> V^T[d][pos] through LDS (64-key runs) ----
    const int kvh = slot - a.n_heads - a.n_kv_heads;
    constexpr int PITCH = D + 2;
    T* tile = reinterpret_cast<T*>(smem);
    for (int g = tid; g < 64 * (D / 8); g += 256) {
        const int t = g / (D / 8), c = (g % (D / 8)) * 8;
        if (t >= ntok) continue;
        float v[8]; load8<T>(qkv + (size_t)(tok0 + t) * a.qkv_stride + slot * D + c, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) tile[t * PITCH + c + e] = from_f32<T>(v[e]);
    }
    __syncthreads();
    T* vt = reinterpret_cast<T*>(a.VT) + (size_t)kvh * D * a.s_max;
    const int t = tid & 63;
    if (t < ntok || t < nzero) {
        const int pos = a.pos0 + tok0 + t;
        for (int d = tid >> 6; d < D; d += 4) vt[(size_t)d * a.s_max + pos] = t < ntok ? tile[t * PITCH + d] : from_f32<T>(0.f);
    }
    if (ntok > 0 && tok0 + 64 >= a.T && a.zero_to == 0) {     // as in rope_kv_kernel: to the end of the last row's 64 keys
        const int end = a.pos0 + a.T, whole = (end + 63) & ~63, pos = end + t;
        if (pos < (whole < a.s_max ? whole : a.s_max))
            for (int d = tid >> 6; d < D; d += 4) vt[(size_t)d * a.s_max + pos] = from_f32<T>(0.f);
    }
}

template <typename T, int D, bool PAIRED>
__global__ __launch_bounds__(256) void qkv_norm_rope_kv_kernel(QkvNormRopeArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    qkv_norm_rope_body<T, D, PAIRED>(a, blockIdx.x, smem);
}

template <typename T, int D>
__global__ __launch_bounds__(256) void qkv_norm_rope_segs_kernel(QkvNormRopeArgs a, RowSegs g) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int block = blockIdx.x;
    const RowSeg& s = g.s[row_segs_at(g, block)];
    a.qkv = reinterpret_cast<T*>(a.qkv) + (size_t)s.row0 * a.qkv_stride;
    a.K = s.K; a.VT = s.VT; a.T = s.n; a.pos0 = s.pos0; a.s_max = s.s_max; a.zero_to = s.zero_to;
    qkv_norm_rope_body<T, D, true>(a, block, smem);
}

void launch_qkv_norm_rope_segs(int dtype, int D, const QkvNormRopeArgs& a, const RowSegs& segs, hipStream_t st) {
    RowSegs g = segs;
    LMX_REQUIRE((dtype == kBF16 || dtype == kF16) && (D == 64 || D == 128), "qkv_norm_rope_kv: rows of several sequences are of 16 bits and padded to heads of 64 or 128");
    LMX_REQUIRE(a.qkv && a.qkv_stride % 8 == 0 && a.qkv_stride >= (a.n_heads + 2 * a.n_kv_heads) * D, "qkv_norm_rope_kv: bad row pitch");
    LMX_REQUIRE(a.rot_dims % 16 == 0 && a.rot_dims <= a.qk_dim && a.qk_dim <= D && (a.rot_dims == 0 || a.cos_sin), "qkv_norm_rope_kv: bad rotation");
    LMX_REQUIRE(g.n >= 0 && g.n <= ROW_SEGS, "qkv_norm_rope_kv: too many segments");
    for (int i = 0; i < g.n; ++i) {
        const RowSeg& s = g.s[i];
        LMX_REQUIRE(s.K && s.VT && s.n >= 1 && s.row0 >= 0 && s.pos0 >= 0 && s.pos0 + s.n <= s.s_max && s.pos0 + s.zero_to <= s.s_max, "qkv_norm_rope_kv: rows past the cache");
        LMX_REQUIRE(s.zero_to == 0 || a.n_heads == 0, "qkv_norm_rope_kv: clearing is for key / value rows");
    }
    if (g.n == 0) return;
    const dim3 grid(row_segs_blocks(g, [](const RowSeg& s) { return cdiv(std::max(s.n, s.zero_to), 64); }), a.n_heads + 2 * a.n_kv_heads);
    const size_t smem = (size_t)64 * (D + 2) * dtype_size(dtype);
#define L(TT, DD) do {                                                                                                                   \
        auto kern = qkv_norm_rope_segs_kernel<TT, DD>;                                                                                   \
        static bool attr_set = false;                                                                                                    \
        if (!attr_set) { LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024)); attr_set = true; } \
        hipLaunchKernelGGL(kern, grid, dim3(256), smem, st, a, g);                                                                       \
    } while (0)
#define LD(TT) do { if (D == 128) L(TT, 128); else L(TT, 64); } while (0)
    if (dtype == kBF16) LD(bf16_t); else LD(f16_t);
#undef LD
#undef L
    LMX_CHECK_HIP(hipGetLastError());
}

void launch_qkv_norm_rope_kv(int dtype, int D, const QkvNormRopeArgs& a, hipStream_t st) {
    LMX_REQUIRE(D == 64 || D == 128 || D == 256, "qkv_norm_rope_kv: padded head width must be 64, 128 or 256");
    LMX_REQUIRE(a.qkv_stride % 8 == 0 && a.qkv_stride >= (a.n_heads + 2 * a.n_kv_heads) * D, "qkv_norm_rope_kv: bad row pitch");
    LMX_REQUIRE(a.rot_dims % 2 == 0 && a.rot_dims <= a.qk_dim && a.qk_dim <= D && (a.rot_dims == 0 || a.cos_sin), "qkv_norm_rope_kv: bad rotation");
    LMX_REQUIRE(a.pos0 >= 0 && a.pos0 + a.T <= a.s_max && a.pos0 + a.zero_to <= a.s_max, "qkv_norm_rope_kv: rows past the cache");
    if (a.T <= 0) return;
    const dim3 grid(cdiv(a.zero_to > a.T ? a.zero_to : a.T, 64), a.n_heads + 2 * a.n_kv_heads);
    const bool paired = a.rot_dims % 16 == 0;
    LMX_REQUIRE(a.zero_to == 0 || (paired && a.n_heads == 0), "qkv_norm_rope_kv: clearing is for key / value rows of whole rotation groups");
    size_t smem = (size_t)64 * (D + 2) * dtype_size(dtype);
    if (!paired && smem < 256 * 8 * sizeof(float)) smem = 256 * 8 * sizeof(float);
#define L(TT, DD) do {                                                                                                                   \
        auto kern = paired ? qkv_norm_rope_kv_kernel<TT, DD, true> : qkv_norm_rope_kv_kernel<TT, DD, false>;                                                                                     \
        static bool attr_set[2] = {false, false};                                                                                        \
        if (!attr_set[paired]) { LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024)); attr_set[paired] = true; } \
        hipLaunchKernelGGL(kern, grid, dim3(256), smem, st, a);                                                                          \
    } while (0)
#define LD(TT) do { if (D == 256) L(TT, 256); else if (D == 128) L(TT, 128); else L(TT, 64); } while (0)
    if (dtype == kBF16) LD(bf16_t); else if (dtype == kF16) LD(f16_t); else LD(float);
#undef LD
#undef L
    LMX_CHECK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------------------------
// attention of prompt rows on the vector ALUs: grid (n_heads, rows).  Scores of the row's visible keys wait in LDS.
// ---------------------------------------------------------------------------------------------------------------
template <typename T, int D>
__global__ __launch_bounds__(256) void rows_attn_kernel(FlashArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float* p_lds = reinterpret_cast<float*>(smem) + 8;       // probabilities of keys [k0, kv_len), k0 = first visible key rounded down to 64
    float* red = reinterpret_cast<float*>(smem);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int head = blockIdx.x, row = blockIdx.y;
    const int kvh = head / (a.n_heads / a.n_kv_heads);
    const int pos = a.q_pos0 + row;
    const int lo = a.window > 0 && pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
    const int k0 = lo & ~63, nk = ((pos + 1 - k0) + 63) & ~63;
    const T* Q = reinterpret_cast<const T*>(a.Q) + (size_t)row * a.q_stride + head * D;
    const T* Kc = reinterpret_cast<const T*>(a.K) + (size_t)kvh * a.s_max * D;
    const T* Vt = reinterpret_cast<const T*>(a.VT) + (size_t)kvh * D * a.s_max;
    constexpr int LPK = D / 8, KPW = 64 / LPK;
    const float scl = a.scale * 1.4426950408889634f;
    {
        const int sub = lane % LPK, kslot = lane / LPK;
        float qv[8]; load8<T>(Q + sub * 8, qv);
        for (int b = wave * KPW; b < nk; b += 4 * KPW) {
            const int key = k0 + b + kslot;
            float kv[8]; load8<T>(Kc + (size_t)(key <= pos ? key : pos) * D + sub * 8, kv);
            float s = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) s = fmaf(qv[e], kv[e], s);
            s = group_sum<LPK>(s);
            if (sub == 0) p_lds[b + kslot] = key >= lo && key <= pos ? s * scl : -INFINITY;
        }
    }
    __syncthreads();
    float mx = -INFINITY;
    for (int k = tid; k < nk; k += 256) mx = fmaxf(mx, p_lds[k]);
    mx = block_max<4>(mx, red);
    float sum = 0.f;
    for (int k = tid; k < nk; k += 256) { const float e = __builtin_amdgcn_exp2f(p_lds[k] - mx); p_lds[k] = e; sum += e; }
    sum = block_sum<4>(sum, red);
    __syncthreads();
    float out = softmax_scale(sum, mx, a.sink != 0);
    if (a.gate) out *= sigmoid_f32(to_f32(reinterpret_cast<const T*>(a.gate)[(size_t)row * a.q_stride + head]));
    T* O = reinterpret_cast<T*>(a.O) + (size_t)row * a.o_stride + head * D;
    const int sub = tid & 7, drow = tid >> 3;
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
        const int d = db * 32 + drow;
        float acc = 0.f;
        for (int b = 0; b < nk; b += 64) {
            float vv[8]; load8<T>(Vt + (size_t)d * a.s_max + k0 + b + sub * 8, vv);
            float pv[8]; load8<float>(p_lds + b + sub * 8, pv);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc = fmaf(pv[e], pv[e] != 0.f ? vv[e] : 0.f, acc);
        }
        acc = sum8(acc);
        if (sub == 0) O[d] = from_f32<T>(acc * out);
    }
}

void launch_rows_attn(int dtype, int D, const FlashArgs& a, hipStream_t st) {
    LMX_REQUIRE(D == 64 || D == 128 || D == 256, "rows_attn: padded head width must be 64, 128 or 256");
    LMX_REQUIRE(a.s_max % 64 == 0 && a.q_len > 0 && a.q_pos0 >= 0 && a.q_pos0 + a.q_len <= a.s_max, "rows_attn: bad lengths");
    const int last = a.q_pos0 + a.q_len;
    const int span = a.window > 0 && a.window < last ? a.window : last;
    const size_t smem = ((size_t)span + 136) * sizeof(float);
    LMX_REQUIRE(smem <= 160 * 1024, "rows_attn: score row does not fit LDS");
#define L(TT, DD) do {                                                                                                                   \
        auto kern = rows_attn_kernel<TT, DD>;                                                                                            \
        static bool attr_set = false;                                                                                                    \
        if (!attr_set) { LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024)); attr_set = true; } \
        hipLaunchKernelGGL(kern, dim3(a.n_heads, a.q_len), dim3(256), smem, st, a);                                                      \
    } while (0)
#define LD(TT) do { if (D == 256) L(TT, 256); else if (D == 128) L(TT, 128); else L(TT, 64); } while (0)
    if (dtype == kBF16) LD(bf16_t); else if (dtype == kF16) LD(f16_t); else LD(float);
#undef LD
#undef L
    LMX_CHECK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------------------------
// one new token per sequence.  grid (n_heads, n_split, sequences), 256 threads.  Split s of n_split walks the 128-key chunks c0 + s, c0 + s + n_split, ... of the
// window [pos - window + 1, pos] with an online softmax; every K / V^T load of a chunk is requested before anything waits, the first chunk's ahead of the query's own
// norm and rotation.  The workgroup that walks the chunk of position `pos` takes the new key from the qkv row (and, for the first query head of a kv group, appends
// it); it is never read back from the cache inside the launch.  Splits are merged by the last workgroup of a head to arrive (write-through partials, one ticket).
// ---------------------------------------------------------------------------------------------------------------
// one head vector by one wave: norm over the true width, rotation, into out[D] (fp32 LDS); tmp[D] is scratch of this wave
template <typename T, int D>
__device__ __forceinline__ void norm_rope_vec(const T* __restrict__ x, const T* __restrict__ nw, float eps, int qk_dim, const float* __restrict__ cs, int rot_dims,
                                              float* tmp, float* out, int lane) {
    constexpr int E = D / 64;
    float v[E];
#pragma unroll
    for (int j = 0; j < E; ++j) v[j] = to_f32(x[lane + 64 * j]);
    if (nw) {
        float ss = 0.f;
#pragma unroll
        for (int j = 0; j < E; ++j) ss += v[j] * v[j];
        const float inv = 1.f / sqrtf(wave_sum(ss) / (float)qk_dim + eps);
#pragma unroll
        for (int j = 0; j < E; ++j) v[j] = v[j] * inv * to_f32(nw[lane + 64 * j]);
    }
#pragma unroll
    for (int j = 0; j < E; ++j) tmp[lane + 64 * j] = v[j];
    __builtin_amdgcn_wave_barrier();
    const int half = rot_dims >> 1;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int i = lane + 64 * j;
        if (i < rot_dims) {
            const bool lo = i < half;
            const int k = lo ? i : i - half;
            const float p = tmp[lo ? i + half : i - half];
            v[j] = v[j] * cs[k] + (lo ? -p : p) * cs[half + k];
        }
        // the same rounding as the prompt's rows: q enters the scores and k the cache in the model dtype
        out[i] = round_to<T>(v[j]);
    }
}

template <typename T, int D, bool LEAVE = false>
__global__ __launch_bounds__(256) void decode_win_kernel(WinDecodeArgs a) {
    __shared__ __attribute__((aligned(16))) float sc[DF_CHUNK];
    __shared__ __attribute__((aligned(16))) float qs[D], ks[D];
    __shared__ float tmp[2][D];
    __shared__ float red[8];
    __shared__ float mg_m[DF_MAX_SPLIT], mg_w[DF_MAX_SPLIT];
    __shared__ float mg_o[256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int head = blockIdx.x, split = blockIdx.y, z = blockIdx.z;
    const DecodeFusedSeq e = a.tab ? a.tab[z] : a.one;
    int pos = a.pos >= 0 ? a.pos : *e.pos_ptr;
    pos = pos < a.s_max ? pos : a.s_max - 1;               // the host keeps len + steps <= s_max; never index past the cache whatever the device word holds
    const int group = a.n_heads / a.n_kv_heads, kvh = head / group;
    const int lo = a.window > 0 && pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
    const int c0 = lo / DF_CHUNK, c1 = pos / DF_CHUNK;
    const T* row = reinterpret_cast<const T*>(a.qkv) + (size_t)z * a.qkv_stride;
    T* Kc = reinterpret_cast<T*>(e.K) + (size_t)kvh * a.s_max * D;
    T* Vt = reinterpret_cast<T*>(e.VT) + (size_t)kvh * D * a.s_max;
    const T* vnew = row + (a.n_heads + a.n_kv_heads + kvh) * D;
    const float* cs = a.cos_sin + (size_t)pos * a.rot_dims;
    const bool owner = (c1 - c0) % a.n_split == split;      // this workgroup walks the new key's chunk
    constexpr int WS = D + 4;
    float* ws = e.ws + ((size_t)head * a.n_split + split) * WS;

    constexpr int LPK = D / 8, KPW = 64 / LPK, KU = DF_CHUNK / (4 * KPW), DB = D / 32;
    const float scl = a.scale * 1.4426950408889634f;
    const int sub = lane % LPK, kslot = lane / LPK;
    const int s8 = tid & 7, drow = tid >> 3;
    Chunk8<T> kr[KU], vr[2][DB];
    auto load_chunk = [&](int c) {
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            int key = c * DF_CHUNK + (u * 4 + wave) * KPW + kslot;
            key = key < pos ? key : (pos > 0 ? pos - 1 : 0);             // rows past the cached keys re-read the last one; their scores are dropped
            kr[u].load(Kc + (size_t)key * D + sub * 8);
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int db = 0; db < DB; ++db) vr[kb][db].load(Vt + (size_t)(db * 32 + drow) * a.s_max + c * DF_CHUNK + kb * 64 + s8 * 8);
    };
    if (c0 + split <= c1) load_chunk(c0 + split);
    if (wave == 0) norm_rope_vec<T, D>(row + head * D, reinterpret_cast<const T*>(a.q_norm), a.eps, a.qk_dim, cs, a.rot_dims, tmp[0], qs, lane);
    else if (wave == 1 && owner) norm_rope_vec<T, D>(row + (a.n_heads + kvh) * D, reinterpret_cast<const T*>(a.k_norm), a.eps, a.qk_dim, cs, a.rot_dims, tmp[1], ks, lane);
    __syncthreads();
    if (owner && wave == 0) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < D / 64; ++j) s = fmaf(qs[lane + 64 * j], ks[lane + 64 * j], s);
        s = wave_sum(s);
        if (lane == 0) red[6] = s * scl;
    }
    __syncthreads();
    if (owner && head % group == 0) {
        for (int d = tid; d < D; d += 256) {
            Kc[(size_t)pos * D + d] = from_f32<T>(ks[d]);
            Vt[(size_t)d * a.s_max + pos] = vnew[d];
        }
    }
    float qv[8]; load8<float>(qs + sub * 8, qv);
    float m = -INFINITY, l = 0.f, acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db] = 0.f;
    for (int c = c0 + split; c <= c1; c += a.n_split) {
        const int kb0 = c * DF_CHUNK;
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const int kl = (u * 4 + wave) * KPW + kslot, key = kb0 + kl;
            float kv[8]; kr[u].get(kv);
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) s = fmaf(qv[i], kv[i], s);
            s = group_sum<LPK>(s);
            if (sub == 0) sc[kl] = key == pos ? red[6] : (key >= lo && key < pos ? s * scl : -INFINITY);
        }
        __syncthreads();
        const float s = tid < DF_CHUNK ? sc[tid] : -INFINITY;
        const float m_new = fmaxf(m, block_max<4>(s, red));              // finite: a walked chunk holds at least one visible key
        const float alpha = __builtin_amdgcn_exp2f(m - m_new);           // first chunk: exp2(-inf) = 0 on zero accumulators
        const float ex = __builtin_amdgcn_exp2f(s - m_new);
        l = l * alpha + block_sum<4>(ex, red);
        m = m_new;
        float p_new = 0.f;
        if (c == c1) {                                                   // the newest key's value comes from the row, not from the cache
            if (tid == pos - kb0) red[7] = ex;
            if (tid < DF_CHUNK) sc[tid] = tid == pos - kb0 ? 0.f : ex;
        } else if (tid < DF_CHUNK) sc[tid] = ex;
        __syncthreads();
        if (c == c1) p_new = red[7];
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] *= alpha;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            float p[8]; load8<float>(sc + kb * 64 + s8 * 8, p);
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                float v[8]; vr[kb][db].get(v);
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[db] = fmaf(p[i], p[i] != 0.f ? v[i] : 0.f, acc[db]);      // columns outside the window or past the cache never enter, whatever they hold
            }
        }
        if (c == c1 && s8 == 0) {
#pragma unroll
            for (int db = 0; db < DB; ++db) acc[db] = fmaf(p_new, to_f32(vnew[db * 32 + drow]), acc[db]);
        }
        if (c + a.n_split <= c1) load_chunk(c + a.n_split);
        __syncthreads();                                                 // sc is rewritten by the next chunk
    }
    float gate = 1.f;
    if (a.gate_off >= 0) gate = sigmoid_f32(to_f32(row[a.gate_off + head]));
    T* out = reinterpret_cast<T*>(a.out) + (size_t)z * a.out_stride + head * D;
    const float fin = a.n_split == 1 ? softmax_scale(l, m, a.sink != 0) * gate : 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        float t = acc[db];
        t = sum8(t);
        if (s8 == 0) {
            const int d = db * 32 + drow;
            if (a.n_split == 1) out[d] = from_f32<T>(t * fin);
            else if constexpr (LEAVE) ws[d] = t;
            else __hip_atomic_store(ws + d, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (a.n_split == 1) return;
    if constexpr (LEAVE) {                                   // the next launch adds the splits (gemv2.h)
        if (tid == 0) { ws[D] = m; ws[D + 1] = l; }
        return;
    }
    if (tid == 0) {
        __hip_atomic_store(ws + D, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(ws + D + 1, l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // ---- merge by the last workgroup to arrive for this head (decode_fused_body's protocol: write-through payload, every wave drains, one relaxed ticket) ----
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) red[5] = __hip_atomic_fetch_add(e.counters + head, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.n_split - 1 ? 1.f : 0.f;
    __syncthreads();
    if (red[5] == 0.f) return;
    const float* wsh = e.ws + (size_t)head * a.n_split * WS;
    if (tid < a.n_split) {
        mg_m[tid] = __hip_atomic_load(wsh + tid * WS + D, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        mg_w[tid] = __hip_atomic_load(wsh + tid * WS + D + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    constexpr int NG = 256 / D, SPG = DF_MAX_SPLIT / NG;
    const int g = tid / D, d = tid % D;
    float ov[SPG];
#pragma unroll
    for (int i = 0; i < SPG; ++i) {
        const int sp = g + i * NG;
        ov[i] = sp < a.n_split ? __hip_atomic_load(wsh + sp * WS + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.f;
    }
    __syncthreads();
    float M = -INFINITY, lt = 0.f, o = 0.f;
    for (int sp = 0; sp < a.n_split; ++sp) M = fmaxf(M, mg_m[sp]);
    for (int sp = 0; sp < a.n_split; ++sp) lt += __builtin_amdgcn_exp2f(mg_m[sp] - M) * mg_w[sp];          // a split without a chunk left (-inf, 0): weight 0
#pragma unroll
    for (int i = 0; i < SPG; ++i) {
        const int sp = g + i * NG;
        if (sp < a.n_split) o += __builtin_amdgcn_exp2f(mg_m[sp] - M) * ov[i];
    }
    mg_o[tid] = o;
    __syncthreads();
    if (g == 0) {
#pragma unroll
        for (int i = 1; i < NG; ++i) o += mg_o[i * D + d];
        out[d] = from_f32<T>(o * softmax_scale(lt, M, a.sink != 0) * gate);
    }
    if (tid == 0) __hip_atomic_store(e.counters + head, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);    // re-arm for the next launch
}

// The same launch for 16-bit models with head widths up to 128: one workgroup per (kv head, split, sequence) serves ALL query heads of the kv head on MFMA tiles, so a cached
// key and value leaves memory once instead of once per query head.  A wave walks 64-key pieces (no barrier inside the walk): keys and V^T rows come in whole lines (16 loads of
// 1 KiB each, marked streaming) and reach the operands' order through 16 KiB of wave-private LDS, chunks XOR-swizzled; the next piece is requested as soon as this one is in LDS.
// Scores = K tile (16 keys) x query heads (16 columns), the softmax over the lane's 16 keys and 4 lanes, then V^T rows x probabilities.  The C layout of the scores (lane = head,
// 4 rows a tile) is the B layout of the probabilities when row 4 q + r of tile t is key 8 q + 4 t + r of 32, so no probability changes lanes.  Probabilities keep fp32's 24
// bits: three 16-bit terms, three MFMAs; f16 terms of a probability times 2^15, because f16 ends at 2^-24: without the factor a probability of 2^-12 kept 12 bits and one below 2^-25
// none, with it the sums are off by 2^-40 a key.  Bound: the cache stream (32 sequences x 1024 keys, 8 kv heads of 128: 134 MB a launch): straight operand loads 36.9 us, whole lines through LDS with the next piece on the
// wire 32.0 (4.2 TB/s), with one split (straight: 2 splits 36.4, 4 43.3: the merge and a shorter walk cost more than a fuller chip gives); which launches: decode_win_form.
template <typename T> struct WinMfma;
template <> struct WinMfma<bf16_t> {
    static __device__ __forceinline__ f32x4 run(const uint4& a, const uint4& b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_v, a), __builtin_bit_cast(bf16x8_v, b), c, 0, 0, 0);
    }
};
template <> struct WinMfma<f16_t> {
    static __device__ __forceinline__ f32x4 run(const uint4& a, const uint4& b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_v, a), __builtin_bit_cast(f16x8_v, b), c, 0, 0, 0);
    }
};
constexpr int WIN_GROUP_MAX = 16;                              // query heads of a kv head: the columns of a tile
// q heads, new key, one row of scratch per wave | the waves' partial rows [wave][head][D], statistics | the waves' tiles (the partial rows take their place after the walk)
static int win_group_smem(int group, int D, int nw) { return ((group + 1 + nw) * D + 2 * nw * 16 + 8 + std::max(nw * 64 * D / 2, nw * group * D)) * (int)sizeof(float); }

template <typename T, int D, int NW>
__global__ __launch_bounds__(NW * 64) void decode_win_group_kernel(WinDecodeArgs a) {
    extern __shared__ __attribute__((aligned(16))) float wsm[];
    const int group = a.n_heads / a.n_kv_heads;
    float *qs = wsm, *ks = qs + group * D, *tmp = ks + D, *wm = tmp + NW * D, *wl = wm + NW * 16, *flag = wl + NW * 16, *wo = flag + 8;      // wo: [wave][head][D] after the walk, [wave] tiles of 64 keys before
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15, q4 = lane >> 4;
    const int kvh = blockIdx.x, split = blockIdx.y, z = blockIdx.z;
    const DecodeFusedSeq e = a.tab ? a.tab[z] : a.one;
    int pos = a.pos >= 0 ? a.pos : *e.pos_ptr;
    pos = __builtin_amdgcn_readfirstlane(pos < a.s_max ? pos : a.s_max - 1);
    const int lo = a.window > 0 && pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
    const int p0 = lo / 64, np = (pos + 63) / 64 - p0;         // 64-key pieces with a cached key that is seen (np <= 0: none); split's wave w takes NW split + w, + NW n_split, ...
    const T* row = reinterpret_cast<const T*>(a.qkv) + (size_t)z * a.qkv_stride;
    T* Kc = reinterpret_cast<T*>(e.K) + (size_t)kvh * a.s_max * D;
    T* Vt = reinterpret_cast<T*>(e.VT) + (size_t)kvh * D * a.s_max;
    const T* vnew = row + (a.n_heads + a.n_kv_heads + kvh) * D;
    const float* cs = a.cos_sin + (size_t)pos * a.rot_dims;
    const bool owner = split == a.n_split - 1;                 // this workgroup takes the new key
    constexpr int NT = D / 32, ND = D / 16;                    // 32-deep steps of a score, 16-row tiles of V^T
    constexpr float UP = std::is_same_v<T, f16_t> ? 32768.f : 1.f;      // the accumulators hold UP times the sums (probabilities are <= 1); the normaliser l does not
    const float scl = a.scale * 1.4426950408889634f;

    // piece loads: instruction u brings 1 KiB = whole key rows (K) or 8 V^T rows of 64 keys; lane l's 16 bytes land at l 16 of the tile's KiB u, so the chunk it fetches is the swizzled one
    constexpr int NL = D / 8, CPR = D / 8;                     // loads a tile; 16-byte chunks of a key row
    char* tile = reinterpret_cast<char*>(wo) + wave * 64 * D * 2;
    const int krow = lane / CPR, kch = lane % CPR, vrow = lane >> 3, vch = lane & 7;
    auto kswz = [](int row) { return ((row & 3) | (row >> 1 & 12)) & (CPR - 1); };      // the 16 rows a fragment read takes are 8 a + 4 t + b: distinct
    uint32_t k_lane[NL];                                       // u-dependent only through the swizzle; the row offsets are whole KiB
#pragma unroll
    for (int u = 0; u < NL; ++u) { const int row = u * (64 / CPR) + krow; k_lane[u] = (uint32_t)((krow * CPR + (kch ^ kswz(row))) * 16); }
    const uint32_t v_lane = ((uint32_t)vrow * (uint32_t)a.s_max) * 2u + (uint32_t)((vch ^ (vrow >> 1)) * 16);      // rows 8 u + vrow: (row >> 1) & 7 = 4 (u & 1) + (vrow >> 1)
    uint4 kr[NL], vr[NL];
    auto view = [](const T* p, bool on) {                      // the table's words come by vector loads: as they are, every buffer load would loop over the lanes' views
        const uint64_t v = reinterpret_cast<uint64_t>(p);
        return ba_rsrc(reinterpret_cast<const void*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)v) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32), on);
    };
    auto load_k = [&](int p, bool on) {                        // a piece that is not there: an empty view, no traffic and no branch around the loads
        const __amdgpu_buffer_rsrc_t rs = view(Kc, on);
#pragma unroll
        for (int u = 0; u < NL; ++u) kr[u] = __builtin_bit_cast(uint4, ba_ld16<true>(rs, k_lane[u], (uint32_t)((p * 64) * D * 2 + u * 1024)));
    };
    auto load_v = [&](int p, bool on) {
        const __amdgpu_buffer_rsrc_t rs = view(Vt, on);
#pragma unroll
        for (int u = 0; u < NL; ++u) vr[u] = __builtin_bit_cast(uint4, ba_ld16<true>(rs, v_lane ^ (u & 1 ? 64u : 0u), (uint32_t)(8 * u) * (uint32_t)a.s_max * 2u + (uint32_t)p * 128u));
    };
    auto to_lds = [&](const uint4 (&r)[NL]) {
#pragma unroll
        for (int u = 0; u < NL; ++u) *reinterpret_cast<uint4*>(tile + u * 1024 + lane * 16) = r[u];
        asm volatile("" ::: "memory");                         // the wave's LDS operations retire in order; the compiler must not turn them round either
    };
    const int first = NW * split + wave, step = NW * a.n_split;
    load_k(p0 + first, first < np);
    asm volatile("" ::: "memory");                             // keys before values: the order of the walk
    load_v(p0 + first, first < np);
    asm volatile("" ::: "memory");
    for (int h = wave; h < group + (owner ? 1 : 0); h += NW) {  // the query heads, then the new key
        const bool isk = h == group;
        norm_rope_vec<T, D>(row + (isk ? a.n_heads + kvh : kvh * group + h) * D, reinterpret_cast<const T*>(isk ? a.k_norm : a.q_norm), a.eps, a.qk_dim, cs, a.rot_dims, tmp + wave * D,
                            qs + h * D, lane);
    }
    __syncthreads();
    auto frag = [&](const float* v) -> uint4 {                 // 8 consecutive fp32 values that are 16-bit ones already
        float x[8]; load8<float>(v, x);
        return uint4{pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3]), pack2<T>(x[4], x[5]), pack2<T>(x[6], x[7])};
    };
    uint4 qf[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) qf[t] = i16 < group ? frag(qs + i16 * D + q4 * (D / 4) + 8 * t) : uint4{0u, 0u, 0u, 0u};

    float m = -INFINITY, l = 0.f;                              // of head i16; l: this lane's keys
    f32x4 acc[ND];                                             // [16 d + 4 q4 + r][head i16]
#pragma unroll
    for (int d = 0; d < ND; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = first; i < np; i += step) {
        const int base = (p0 + i) * 64;
        to_lds(kr);
        load_k(p0 + i + step, i + step < np);
        f32x4 s[4];                                            // [2 h + t]: keys 32 h + 8 q4 + 4 t + r
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            s[g] = f32x4{0.f, 0.f, 0.f, 0.f};
            const int row = 32 * (g >> 1) + 8 * (i16 >> 2) + 4 * (g & 1) + (i16 & 3);
#pragma unroll
            for (int t = 0; t < NT; ++t)
                s[g] = WinMfma<T>::run(*reinterpret_cast<const uint4*>(tile + row * D * 2 + (((q4 * NT + t) ^ kswz(row)) * 16)), qf[t], s[g]);
        }
        const bool edge = base < lo || base + 64 > pos;        // some of the piece's keys are outside: their scores are dropped and their values, whatever they hold, cleared
        float mx = -INFINITY;
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = base + 32 * (g >> 1) + 8 * q4 + 4 * (g & 1) + r;
                s[g][r] = !edge || (key >= lo && key < pos) ? s[g][r] * scl : -INFINITY;
                mx = fmaxf(mx, s[g][r]);
            }
        mx = fold16(mx, OpMax{}); mx = fold32(mx, OpMax{});
        const float m_new = fmaxf(m, mx), ms = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - ms);
        m = m_new;
        float ps = 0.f;
        uint4 pf[2][3];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float p[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) p[k] = __builtin_amdgcn_exp2f(s[2 * h + (k >> 2)][k & 3] - ms);
            ps += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
#pragma unroll
            for (int k = 0; k < 8; ++k) p[k] *= UP;
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                pf[h][n] = uint4{pack2<T>(p[0], p[1]), pack2<T>(p[2], p[3]), pack2<T>(p[4], p[5]), pack2<T>(p[6], p[7])};
                p[0] -= unpack_lo<T>(pf[h][n].x); p[1] -= unpack_hi<T>(pf[h][n].x); p[2] -= unpack_lo<T>(pf[h][n].y); p[3] -= unpack_hi<T>(pf[h][n].y);
                p[4] -= unpack_lo<T>(pf[h][n].z); p[5] -= unpack_hi<T>(pf[h][n].z); p[6] -= unpack_lo<T>(pf[h][n].w); p[7] -= unpack_hi<T>(pf[h][n].w);
            }
        }
        l = l * alpha + ps;
        asm volatile("" ::: "memory");                         // the keys have been read out of the tile
        to_lds(vr);
        load_v(p0 + i + step, i + step < np);
#pragma unroll
        for (int d = 0; d < ND; ++d) acc[d] *= alpha;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t keep[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int key = base + 32 * h + 8 * q4 + 2 * c;
                keep[c] = !edge ? 0xffffffffu : (key >= lo && key < pos ? 0x0000ffffu : 0u) | (key + 1 >= lo && key + 1 < pos ? 0xffff0000u : 0u);
            }
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                uint4 vf = *reinterpret_cast<const uint4*>(tile + (d * 16 + i16) * 128 + (((4 * h + q4) ^ (i16 >> 1)) * 16));
                vf.x &= keep[0]; vf.y &= keep[1]; vf.z &= keep[2]; vf.w &= keep[3];
#pragma unroll
                for (int n = 2; n >= 0; --n) acc[d] = WinMfma<T>::run(vf, pf[h][n], acc[d]);
            }
        }
        asm volatile("" ::: "memory");                         // the next piece's keys go into the tile after every read of this one's values
    }
    // into the caches after the walk: a store in flight (to a pointer out of the table) makes every wait of the walk one for everything
    if (owner) {
        for (int d = tid; d < D; d += NW * 64) {
            Kc[(size_t)pos * D + d] = from_f32<T>(ks[d]);
            Vt[(size_t)d * a.s_max + pos] = vnew[d];
        }
    }
    if (owner && wave == 0) {                                  // the new key: its score from the MFMA (every row of the tile is the key), its value from the row
        f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < NT; ++t) s = WinMfma<T>::run(frag(ks + q4 * (D / 4) + 8 * t), qf[t], s);
        const float sn = s[0] * scl, m_new = fmaxf(m, sn);
        const float alpha = __builtin_amdgcn_exp2f(m - m_new), pn = __builtin_amdgcn_exp2f(sn - m_new);
        m = m_new;
        l = l * alpha + (q4 == 0 ? pn : 0.f);
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            const uint2 v = *reinterpret_cast<const uint2*>(vnew + d * 16 + 4 * q4);
            const f32x4 vv = {unpack_lo<T>(v.x), unpack_hi<T>(v.x), unpack_lo<T>(v.y), unpack_hi<T>(v.y)};
            acc[d] = acc[d] * alpha + vv * (pn * UP);
        }
    }
    // ---- the waves, then the splits ----
    l = fold16(l, OpSum{}); l = fold32(l, OpSum{});
    if (q4 == 0) { wm[wave * 16 + i16] = m; wl[wave * 16 + i16] = l; }
    __syncthreads();                                           // every wave is done with its tile: the partial rows take their place
    if (i16 < group) {
#pragma unroll
        for (int d = 0; d < ND; ++d) *reinterpret_cast<f32x4*>(wo + (wave * group + i16) * D + d * 16 + 4 * q4) = acc[d] * (1.f / UP);
    }
    __syncthreads();
    constexpr int WS = D + 4;
    T* out = reinterpret_cast<T*>(a.out) + (size_t)z * a.out_stride + kvh * group * D;
    auto gate = [&](int h) { return a.gate_off >= 0 ? sigmoid_f32(to_f32(row[a.gate_off + kvh * group + h])) : 1.f; };
    for (int i = tid; i < group * D; i += NW * 64) {
        const int h = i / D, d = i % D;
        float M = -INFINITY, lt = 0.f, o = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) M = fmaxf(M, wm[w * 16 + h]);
        const float Ms = M == -INFINITY ? 0.f : M;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float f = __builtin_amdgcn_exp2f(wm[w * 16 + h] - Ms);
            lt += f * wl[w * 16 + h]; o += f * wo[(w * group + h) * D + d];
        }
        if (a.n_split == 1) out[i] = from_f32<T>(o * softmax_scale(lt, M, a.sink != 0) * gate(h));
        else {
            float* ws = e.ws + ((size_t)(kvh * group + h) * a.n_split + split) * WS;
            __hip_atomic_store(ws + d, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (d == 0) {
                __hip_atomic_store(ws + D, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(ws + D + 1, lt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    if (a.n_split == 1) return;
    // merge by the last workgroup to arrive for this kv head (decode_win_kernel's protocol; the ticket is the group's first head's)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* ticket = e.counters + kvh * group;
    if (tid == 0) flag[0] = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.n_split - 1 ? 1.f : 0.f;
    __syncthreads();
    if (flag[0] == 0.f) return;
    for (int i = tid; i < group * D; i += NW * 64) {
        const int h = i / D, d = i % D;
        const float* wsh = e.ws + (size_t)(kvh * group + h) * a.n_split * WS;
        float M = -INFINITY, lt = 0.f, o = 0.f;
        for (int s0 = 0; s0 < a.n_split; s0 += 8) {            // eight splits' words are on their way together
            float mi[8], li[8], oi[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float* w = wsh + (s0 + k) * WS;
                const bool in = s0 + k < a.n_split;
                mi[k] = in ? __hip_atomic_load(w + D, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : -INFINITY;
                li[k] = in ? __hip_atomic_load(w + D + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.f;
                oi[k] = in ? __hip_atomic_load(w + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.f;
            }
            float Mn = M;
#pragma unroll
            for (int k = 0; k < 8; ++k) Mn = fmaxf(Mn, mi[k]);
            const float Ms = Mn == -INFINITY ? 0.f : Mn, f = __builtin_amdgcn_exp2f(M - Ms);      // a split without a key of its own: (-inf, 0, 0)
            lt *= f; o *= f;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float fk = __builtin_amdgcn_exp2f(mi[k] - Ms);
                lt += li[k] * fk; o += oi[k] * fk;
            }
            M = Mn;
        }
        out[i] = from_f32<T>(o * softmax_scale(lt, M, a.sink != 0) * gate(h));
    }
    if (tid == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);          // re-arm for the next launch
}

bool decode_win_groups(int dtype, int D, int n_heads, int n_kv_heads, int n_seq) {
    return dtype != kF32 && D <= 128 && n_heads / n_kv_heads <= WIN_GROUP_MAX && n_seq > 1;
}
// Which kernel and how many splits.  The grouped one reads a cached key once instead of once per query head, in whole lines, but has a group-th of the workgroups, a longer start
// and, over splits, one workgroup that merges all heads of the group.  us, one head a workgroup -> grouped, 16-bit, caches cold (in a step the weights pass between two layers):
//   32 heads on  8 of 128   32 sequences of 1200 keys 116 -> 33   8 of 130  15 -> 12     2 of 600  14 -> 13     4 of 20  9 -> 11      16 of 60  13 -> 11
//   24 heads on 12          32 of 1200 108 -> 53                  2 of 130  12 -> 11     32 of 60  17 -> 19
//   32 heads on 32           8 of 1200  74 -> 32                  2 of 300  14 -> 12     16 of 130 33 -> 23     16 of 60  18 -> 20
//    8 heads on  1          32 of 600   34 -> 15                  8 of 600  14 -> 15     2 of 600  12 -> 15      8 of 60  9 -> 12     (16 on 1: 16 of 600 25 -> 20, 4 of 600 13 -> 20)
// so: up to groups of four from one chunk of keys on, larger groups by the bytes that one head a workgroup asks for (the merge grows with the group); shorter contexts only where
// a group is three or four.  One sequence of 601 keys, 16 heads on 4: 11.1 us either way (9.7 since sums over lanes pass LDS by), all of it latency, so the form with more workgroups stays.
// Eight waves instead of four: where a workgroup has a CU to itself, some of eight waves get a second piece, and the busiest workgroup takes no more pieces than with four (24 pieces in two
// splits are 16 + 8 for 12 + 12).  A step of 10 layers of small linears, 5 .. 32 sequences, 4 or 8 kv heads, contexts of 260 .. 4000, four waves -> eight, us a layer:  one split, 8 pieces
// 52.5 -> 51.9, 12 60.7 -> 59.6, 16 68.0 -> 65.8, 32 85.6 -> 83.4, 63 110.1 -> 109.5;  two, 17 48.6 -> 47.5, 34 59.0 -> 57.4, 52 67.9 -> 67.0, but 24 49.2 : 50.8 and 53.2 : 54.8, 41 56.1 : 57.1;
// three, 48 58.9 -> 57.8, but 34 52.2 : 54.1;  four, 34 49.1 -> 47.9, but 42 50.2 : 52.1;  five, 42 44.8 -> 44.0, but 52 46.1 : 48.8.  Level where the busiest takes as many either way and more
// workgroups are as busy (52 pieces in four splits 51.0 : 51.4).  Groups of two in one split 2 % more to 4 % less, in two 46.1 : 45.9, 59.7 : 60.4; a head a group 50.8 : 51.1, 58.7 : 57.8,
// 63.7 : 64.9.  Five to eight pieces stay with four waves: 1 .. 4 % less with groups of three and more, 1 .. 2 % more with two.  32 sequences of 600 .. 1024 keys, 8 kv heads: 31.4 -> 29.3 us
// a launch (4.6 TB/s of keys and values).
// Splits: as many as make ONE round of workgroups of the grouped kernel (its waves fill a CU: 96 x 3 and 160 x 2 workgroups took a second round, 15 -> 19 and 21 -> 25 us).
// pieces of 64 keys that the busiest of `splits` workgroups of nw waves takes of np
static int win_most_pieces(int np, int splits, int nw) { return np / (nw * splits) * nw + std::min(nw, np % (nw * splits)); }
WinForm decode_win_form(int dtype, int D, int n_heads, int n_kv_heads, int n_seq, int max_len, int window) {
    // chunks the longest member's window can touch; enough workgroups to fill the chip, no more
    const int span = window > 0 && window + 127 < max_len + 1 ? window + 127 : max_len + 1;
    const int group = n_heads / n_kv_heads, chunks = std::max(1, std::min((span + 127) / 128, DF_MAX_SPLIT));
    const double mb = (double)n_heads * n_seq * span * D * 4e-6;
    bool grouped = decode_win_groups(dtype, D, n_heads, n_kv_heads, n_seq);
    if (group <= 4) grouped = grouped && (span >= 128 || (group >= 3 && mb >= 10));
    else grouped = grouped && mb >= 0.6 * group * group;
    const int wgs = (grouped ? n_kv_heads : n_heads) * n_seq, n_split = std::max(1, std::min(chunks, grouped ? 256 / wgs : (1024 + wgs - 1) / wgs));
    // cached keys in sight, wherever in a piece the window begins
    const int np = window > 0 && window <= max_len ? std::min((max_len + 63) / 64, (window + 61) / 64 + 1) : (max_len + 63) / 64;
    const bool wide = grouped && wgs * n_split <= 256 && np > 8 * n_split && win_most_pieces(np, n_split, 8) <= win_most_pieces(np, n_split, 4) && group >= (n_split > 1 ? 3 : 2);
    return WinForm{grouped, n_split, wide};
}

void launch_decode_win(int dtype, int D, const WinDecodeArgs& a, bool grouped, bool wide, hipStream_t st) {
    LMX_REQUIRE(D == 64 || D == 128 || D == 256, "decode_win: padded head width must be 64, 128 or 256");
    LMX_REQUIRE(a.s_max % DF_CHUNK == 0 && a.n_split >= 1 && a.n_split <= DF_MAX_SPLIT && a.n_seq >= 1, "decode_win: cache in whole 128-key chunks, 1..32 splits");
    LMX_REQUIRE(a.n_heads >= 1 && a.n_kv_heads >= 1 && a.n_heads % a.n_kv_heads == 0 && a.qkv && a.out, "decode_win: bad arguments");
    LMX_REQUIRE(a.rot_dims % 2 == 0 && a.rot_dims <= a.qk_dim && a.qk_dim <= D && (a.rot_dims == 0 || a.cos_sin), "decode_win: bad rotation");
    LMX_REQUIRE(a.tab || (a.n_seq == 1 && a.one.K && a.one.VT && a.one.ws && a.one.counters && (a.pos >= 0 || a.one.pos_ptr)), "decode_win: bad sequence");
    LMX_REQUIRE(!a.leave || (a.n_seq == 1 && !grouped && dtype != kF32), "decode_win: splits are left to the next launch by one sequence of a 16-bit model");
    if (grouped && decode_win_groups(dtype, D, a.n_heads, a.n_kv_heads, a.n_seq) && a.qkv_stride % 4 == 0 && reinterpret_cast<uintptr_t>(a.qkv) % 8 == 0) {
        const dim3 grid(a.n_kv_heads, a.n_split, a.n_seq);
        const int group = a.n_heads / a.n_kv_heads;
#define L(TT, DD, NWV)                                                                                                                                     \
    do {                                                                                                                                                   \
        static bool attr_set = false;                                                                                                                      \
        if (!attr_set) {                                                                                                                                   \
            LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&decode_win_group_kernel<TT, DD, NWV>), hipFuncAttributeMaxDynamicSharedMemorySize, win_group_smem(WIN_GROUP_MAX, DD, NWV))); \
            attr_set = true;                                                                                                                               \
        }                                                                                                                                                  \
        LMX_LAUNCH((decode_win_group_kernel<TT, DD, NWV>), grid, dim3(NWV * 64), win_group_smem(group, DD, NWV), st, a);                                   \
    } while (0)
#define LD(TT) do { if (wide) { if (D == 128) L(TT, 128, 8); else L(TT, 64, 8); } else if (D == 128) L(TT, 128, 4); else L(TT, 64, 4); } while (0)
        if (dtype == kBF16) LD(bf16_t); else LD(f16_t);
#undef LD
#undef L
        LMX_CHECK_HIP(hipGetLastError());
        return;
    }
    const dim3 grid(a.n_heads, a.n_split, a.n_seq);
#define L(TT, DD, LV) LMX_LAUNCH((decode_win_kernel<TT, DD, LV>), grid, dim3(256), 0, st, a)
#define LD(TT, LV) do { if (D == 256) L(TT, 256, LV); else if (D == 128) L(TT, 128, LV); else L(TT, 64, LV); } while (0)
    if (dtype == kF32) LD(float, false);
    else if (a.leave) { if (dtype == kBF16) LD(bf16_t, true); else LD(f16_t, true); }
    else if (dtype == kBF16) LD(bf16_t, false); else LD(f16_t, false);
#undef LD
#undef L
    LMX_CHECK_HIP(hipGetLastError());
}

}  // namespace lmx
