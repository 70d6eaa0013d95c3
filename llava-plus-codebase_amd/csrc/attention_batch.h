// Decode attention of the decode BATCH (continuous batching), 16-bit models with head_dim 128: one workgroup per (sequence, head) whose waves STREAM the head's
// keys (attention.hip includes this; launch_decode_fused takes it for the batch form).  As the SINGLE request's launch the same body loses, 16.8 -> 20.4 us a layer: 32
// workgroups cannot pull 19 MB fast enough.
//
// Why: the batch launch of decode_fused_kernel — one workgroup per (sequence, head, 128-key chunk), the whole chunk in registers, partials through memory, ticket, merge by
// the last arriver — moves a batch-8 layer's 142 MB of K / V^T at 3.2 TB/s (4.0 at 32 sequences): its resident workgroups start together, request everything at once, then
// compute and merge together with the HBM idle.  Contract reproduced: the single-token branch of
// llava/model/llava_arch.py:103-112 -> HF5:models/llama/modeling_llama.py:191-214, 243-281 (RoPE on q and the new key, KV append, softmax in fp32, probabilities x V),
// same inputs and outputs as decode_fused_kernel's batch form (DecodeFusedArgs with `tab`); NOT the same summation order (online softmax over 64-key pieces instead
// of 128-key partials merged in chunk order), so parity is by tolerance against the reference arithmetic, not bit-identity with the chunked launch.
//
// Shape: four waves per workgroup; wave w walks the 64-key pieces w, w + 4, ... of the cached keys [0, pos): 16 K
// loads (4 keys x 256 B = 1 KiB contiguous per instruction) + 16 V^T loads (8 d-rows x 128 B per instruction).  Scores are two-element dot products (a 16-bit pair times a
// 16-bit pair, fp32 sum) whose 16 lanes' partial sums are reduced AND dealt out in 15 lane exchanges, so that each lane ends with the score of its own key; an online softmax;
// the piece's 64 probabilities go from the score layout (key 4 sub + kslot) into the V^T layout (8 consecutive keys per lane) through 256 bytes of wave-private LDS; P x V in
// fp32 on the lane's 16 d-rows.  No workgroup barrier inside the loop, nothing goes through global memory.  The next piece's keys are requested as soon as this one's are in
// the scores and its values when this one's are in the sums, into the same registers: a wave always has half a piece on the wire.  Loads are raw buffer loads (base + 32-bit
// lane offset + scalar offset): as 64-bit pointers the 32 addresses of a piece cost 64 registers.  After the loop: one barrier, the four wave states + the NEW key (rotated
// from the qkv row, value from the qkv row) are merged by threads d < D, and one workgroup per kv head appends the new key / value to the caches.
// Bound: the cache stream.  16 sequences of 516 - 1090 keys, 32 heads: 48.3 us a launch with a piece's loads requested together and plain, rows of V^T 4 KiB apart; 47.6 with
// the prefetch and the dealt-out sums; 43.2 (4.9 TB/s) with loads marked streaming and rows 4.25 KiB apart (Model::kv_pitch); 40.9 with the sequences in
// batch_attn_order.  The same loads with no arithmetic, sequences as they come: 38.7.
#pragma once
#include "common.h"
#include "kernels.h"
#include "attention_decode.h"

namespace lmx {

constexpr int BA_PIECE = 64;      // keys per piece
typedef uint32_t ba_u32x4 __attribute__((ext_vector_type(4)));
// raw (stride 0) buffer view: a load is base + 32-bit lane offset + wave-uniform scalar offset.  (As 64-bit pointers hipcc kept the 32 per-load addresses of a
// piece alive across the loop: 64 registers, spilled in the two-phase form.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ba_rsrc(const void* p, bool on = true) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, on ? 0x7fffffff : 0, 0x00020000); }
template <bool NT> __device__ __forceinline__ ba_u32x4 ba_ld16(__amdgpu_buffer_rsrc_t rs, uint32_t lane_off, uint32_t wave_off) { return __builtin_amdgcn_raw_buffer_load_b128(rs, lane_off, wave_off, NT ? 2 : 0); }

template <int CTRL> __device__ __forceinline__ float ba_dpp(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true)); }
// c + a.x b.x + a.y b.y of one 32-bit word of a 16-bit type
template <typename T> __device__ __forceinline__ float ba_dot2(uint32_t a, uint32_t b, float c);
template <> __device__ __forceinline__ float ba_dot2<bf16_t>(uint32_t a, uint32_t b, float c) {
    typedef __bf16 v2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c, false);
}
template <> __device__ __forceinline__ float ba_dot2<f16_t>(uint32_t a, uint32_t b, float c) {
    typedef _Float16 v2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c, false);
}

constexpr int BA_NW = 4;          // waves per workgroup

// decode batch: grid (heads, sequences); K / V^T / position of sequence z from the per-layer table, q|k|v and output rows by stride
// NT: the loads are marked streaming, where no other workgroup reads the same keys
template <typename T, bool NT>
__global__ __launch_bounds__(BA_NW * 64) void decode_attn_wave_kernel(DecodeFusedArgs a, BatchOrder order) {
    constexpr int D = 128, NW = BA_NW;
    __shared__ __attribute__((aligned(16))) float p_lds[NW][BA_PIECE];      // wave-private: probabilities of the current piece, by key
    __shared__ float part[NW + 1][D + 2];                                    // wave states (o[D], m, l) + the new key's
    const int zseq = order.z[blockIdx.y], head = blockIdx.x;
    const DecodeFusedSeq e = a.tab[zseq];
    int pos = *e.pos_ptr;                                                   // keys [0, pos) are cached; this token's key goes to row pos
    pos = pos < a.s_max ? pos : a.s_max - 1;                                // the host keeps len + steps <= s_max; never index past the cache whatever the device word holds
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int s_max = a.s_max, group = a.n_heads / a.n_kv_heads, kvh = head / group;
    const T* qkv = reinterpret_cast<const T*>(a.QKV) + (size_t)zseq * a.qkv_stride;
    const T* knew = qkv + (a.n_heads + kvh) * D;
    const T* vnew = qkv + (a.n_heads + a.n_kv_heads + kvh) * D;
    T* Kc = reinterpret_cast<T*>(e.K) + (size_t)kvh * s_max * D;
    T* Vt = reinterpret_cast<T*>(e.VT) + (size_t)kvh * D * s_max;
    const float* cs = a.cos_sin + (size_t)pos * D;

    const int sub = lane & 15, kslot = lane >> 4;                           // K layout: 16 lanes per key (8 dims each), 4 keys per instruction
    const int s8 = lane & 7, drow8 = lane >> 3;                             // V^T layout: 8 lanes per d-row (8 keys each), 8 d-rows per instruction
    const float scl = a.scale * 1.4426950408889634f;                        // log2 domain

    ba_u32x4 kraw[16], vraw[16];
    const uint32_t k_lane = (uint32_t)(kslot * D + sub * 8) * (uint32_t)sizeof(T);
    const uint32_t v_lane = ((uint32_t)drow8 * (uint32_t)s_max + (uint32_t)s8 * 8u) * (uint32_t)sizeof(T);
    // a load of a piece that is not there goes through an empty view: no traffic, and no branch around the loads (the wait counts behind a branch would cover the prefetch too)
    auto load_k = [&](int k0, bool on) {                                    // rows past the cached keys lie inside the cache (s_max is whole pieces); their scores are dropped
        const __amdgpu_buffer_rsrc_t rs = ba_rsrc(Kc, on);
#pragma unroll
        for (int u = 0; u < 16; ++u) kraw[u] = ba_ld16<NT>(rs, k_lane, (uint32_t)(k0 + 4 * u) * (uint32_t)(D * sizeof(T)));
    };
    auto load_v = [&](int k0, bool on) {
        const __amdgpu_buffer_rsrc_t rs = ba_rsrc(Vt, on);
#pragma unroll
        for (int i = 0; i < 16; ++i) vraw[i] = ba_ld16<NT>(rs, v_lane, ((uint32_t)(8 * i) * (uint32_t)s_max + (uint32_t)k0) * (uint32_t)sizeof(T));
    };
    const int n_piece = (pos + BA_PIECE - 1) / BA_PIECE;

    float qv[8];
    rope8<T, D>(qkv + head * D, cs, sub * 8, qv);
    const uint32_t qp[4] = {pack2<T>(qv[0], qv[1]), pack2<T>(qv[2], qv[3]), pack2<T>(qv[4], qv[5]), pack2<T>(qv[6], qv[7])};      // exact: rotated q is rounded to T

    float m_run = -INFINITY, l_run = 0.f;                                   // m: of the wave; l: of this lane's keys
    float acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    if (wave < n_piece) {                                                   // (a wave without a piece asks for nothing: 32 loads of an empty view are 32 trips through the address unit)
    load_k(wave * BA_PIECE, true);
    asm volatile("" ::: "memory");                                          // keys before values: the order the loop's wait counts rely on
    load_v(wave * BA_PIECE, true);
    asm volatile("" ::: "memory");
    for (int pc = wave; pc < n_piece; pc += NW) {
        const int nk = pos - pc * BA_PIECE;                                            // >= 1 live keys
        // ---- scores: 16 partial sums per lane, reduced over the key's 16 lanes and dealt out: lane (kslot, sub) ends with key 4 sub + kslot ------------------------
        float dot[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            dot[u] = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c) dot[u] = ba_dot2<T>(kraw[u][c], qp[c], dot[u]);
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) asm volatile("" : "+v"(dot[u]) :: "memory");        // the next keys are not requested above the products that read the registers: 64 more
        load_k((pc + NW) * BA_PIECE, pc + NW < n_piece);
        const bool b3 = sub & 8, b2 = sub & 4, b1 = sub & 2, b0 = sub & 1;
#pragma unroll
        for (int j = 0; j < 8; ++j) dot[j] = (b3 ? dot[j + 8] : dot[j]) + ba_dpp<0x140>(b3 ? dot[j] : dot[j + 8]);       // mirror in 16
#pragma unroll
        for (int j = 0; j < 4; ++j) dot[j] = (b2 ? dot[j + 4] : dot[j]) + ba_dpp<0x141>(b2 ? dot[j] : dot[j + 4]);       // mirror in 8
#pragma unroll
        for (int j = 0; j < 2; ++j) dot[j] = (b1 ? dot[j + 2] : dot[j]) + ba_dpp<0x1B>(b1 ? dot[j] : dot[j + 2]);        // mirror in 4
        const float mine = (b0 ? dot[1] : dot[0]) + ba_dpp<0xB1>(b0 ? dot[0] : dot[1]);
        const int my_key = 4 * sub + kslot;                                 // this lane's key inside the piece
        const bool live = my_key < nk;
        const float s = live ? mine * scl : -INFINITY;
        // ---- online softmax over the piece --------------------------------------------------------------------------------------------------------------
        float mx = fmaxf(s, ba_dpp<0x140>(s));
        mx = fmaxf(mx, ba_dpp<0x141>(mx)); mx = fmaxf(mx, ba_dpp<0x1B>(mx)); mx = fmaxf(mx, ba_dpp<0xB1>(mx));
        mx = fold16(mx, OpMax{}); mx = fold32(mx, OpMax{});
        const float m_new = fmaxf(m_run, mx);                               // finite: the piece has at least one live key
        const float p = live ? __builtin_amdgcn_exp2f(s - m_new) : 0.f;
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);          // first piece: exp2(-inf) = 0 on zero accumulators
        l_run = l_run * alpha + p;
        m_run = m_new;
        p_lds[wave][my_key] = p;                                            // the wave's LDS operations retire in order: the reads below see these writes;
        __builtin_amdgcn_wave_barrier();                                    // the compiler must not move them above the writes of the OTHER lanes either
        const float4 p0 = *reinterpret_cast<const float4*>(&p_lds[wave][s8 * 8]);
        const float4 p1 = *reinterpret_cast<const float4*>(&p_lds[wave][s8 * 8 + 4]);
        if (nk < BA_PIECE) {
            // the partial piece: the V^T lines run past the cached keys (stale or never-written columns).  Their probabilities are 0, but 0 x Inf / NaN is
            // NaN, so the values themselves are cleared (wave-uniform branch, once per head: keys 8 s8 + 2 c, + 1 of word c)
            uint32_t msk[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) msk[c] = (8 * s8 + 2 * c < nk ? 0x0000ffffu : 0u) | (8 * s8 + 2 * c + 1 < nk ? 0xffff0000u : 0u);
#pragma unroll
            for (int i = 0; i < 16; ++i)
#pragma unroll
                for (int c = 0; c < 4; ++c) vraw[i][c] &= msk[c];
        }
        // ---- o = o alpha + P V on this lane's d-rows (8 i + drow8) and keys (8 s8 .. + 8) --------------------------------------------------------------
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t w4[4] = {vraw[i][0], vraw[i][1], vraw[i][2], vraw[i][3]};
            float t = acc[i] * alpha;
            t = fmaf(p0.x, unpack_lo<T>(w4[0]), t); t = fmaf(p0.y, unpack_hi<T>(w4[0]), t);
            t = fmaf(p0.z, unpack_lo<T>(w4[1]), t); t = fmaf(p0.w, unpack_hi<T>(w4[1]), t);
            t = fmaf(p1.x, unpack_lo<T>(w4[2]), t); t = fmaf(p1.y, unpack_hi<T>(w4[2]), t);
            t = fmaf(p1.z, unpack_lo<T>(w4[3]), t); t = fmaf(p1.w, unpack_hi<T>(w4[3]), t);
            acc[i] = t;
        }
        __builtin_amdgcn_wave_barrier();                                    // next piece's probabilities are written only after every lane has read this one's
#pragma unroll
        for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(acc[i]) :: "memory");
        load_v((pc + NW) * BA_PIECE, pc + NW < n_piece);
    }
    }
    // ---- the wave's state: o[d] = sum over the 8 lanes of a d-row, then (o, m, l) into LDS ------------------------------------------------------------------
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        float t = acc[i];
        t += ba_dpp<0xB1>(t); t += ba_dpp<0x4E>(t); t += ba_dpp<0x141>(t);
        if (s8 == 0) part[wave][8 * i + drow8] = t;
    }
    l_run = wave_sum(l_run);
    if (lane == 0) { part[wave][D] = m_run; part[wave][D + 1] = l_run; }
    // ---- the new key: rotated from the qkv row by wave 0 (same arithmetic as decode_fused_body), its value straight from the qkv row ---------------------------
    if (wave == 0) {
        float kr[8];
        rope8<T, D>(knew, cs, sub * 8, kr);
        float dot = 0.f;
#pragma unroll
        for (int c = 0; c < 8; ++c) dot = fmaf(qv[c], kr[c], dot);
        dot = group_sum<16>(dot);
        if (lane == 0) { part[NW][D] = dot * scl; part[NW][D + 1] = 1.f; }
        if (head % group == 0 && kslot == 0) store8<T>(Kc + (size_t)pos * D + sub * 8, kr);          // one workgroup per kv head appends
    }
    if (tid >= 64 && tid < 64 + D) {
        const T v = vnew[tid - 64];
        part[NW][tid - 64] = to_f32(v);
        if (head % group == 0) Vt[(size_t)(tid - 64) * s_max + pos] = v;
    }
    __syncthreads();
    // thread d < D merges the wave states and the new key (fixed order: deterministic)
    if (tid >= D) return;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w <= NW; ++w) M = fmaxf(M, part[w][D]);
    float l = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w <= NW; ++w) {
        const float m = part[w][D];
        if (m != -INFINITY) {
            const float f = __builtin_amdgcn_exp2f(m - M);
            l += f * part[w][D + 1];
            o += f * part[w][tid];
        }
    }
    (reinterpret_cast<T*>(a.O) + (size_t)zseq * a.o_stride)[head * D + tid] = from_f32<T>(l > 0.f ? o / l : 0.f);
}

// The batch form of launch_decode_fused through the kernel above.  Workgroup forms measured at equal contexts, with a piece's loads requested together (ms per batched step at
// 8 / 16 / 24 / 32 sequences): 8 waves x 1 head 3.75 / 5.19 / 6.51 / 7.76, 8 x 2 3.95 / 5.16 / 6.71 / 7.76, 4 x 2 4.01 / 5.10 / 6.59 / 7.62, **4 x 1 3.77 / 5.10 / 6.38 /
// 7.62**, 4 or 8 waves x 4 heads 25 - 30 % slower: two independent 4-wave workgroups per CU, one head each, drift apart, so one's merge tail and start-up run under the
// other's stream; walking several heads per workgroup only lengthens the tail.
template <typename T>
inline void launch_decode_attn_wave_t(const DecodeFusedArgs& all, hipStream_t st) {
    constexpr int MOST = (int)sizeof(BatchOrder::z);
    for (int z0 = 0; z0 < all.n_seq; z0 += MOST) {                          // (an engine's batch is one launch)
        DecodeFusedArgs a = all;
        a.n_seq = all.n_seq - z0 < MOST ? all.n_seq - z0 : MOST;
        a.tab = all.tab + z0;
        a.QKV = static_cast<const T*>(all.QKV) + (size_t)z0 * all.qkv_stride;
        a.O = static_cast<T*>(all.O) + (size_t)z0 * all.o_stride;
        BatchOrder o;
        for (int z = 0; z < a.n_seq; ++z) o.z[z] = all.order && all.n_seq <= MOST ? all.order[z] : (uint8_t)z;
        if (a.n_heads == a.n_kv_heads) hipLaunchKernelGGL((decode_attn_wave_kernel<T, true>), dim3(a.n_heads, a.n_seq), dim3(BA_NW * 64), 0, st, a, o);
        else hipLaunchKernelGGL((decode_attn_wave_kernel<T, false>), dim3(a.n_heads, a.n_seq), dim3(BA_NW * 64), 0, st, a, o);
    }
}

}  // namespace lmx
