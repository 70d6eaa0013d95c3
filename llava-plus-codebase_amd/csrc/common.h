// Common device/host helpers for the MI355X (gfx950 / CDNA4) LLaVA forward path.
// Everything here is written for wave64 + MFMA; there is no portability layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string>

namespace lmx {

// ---------------------------------------------------------------------------------------------
// dtypes (mirrors include/llava_mi355x.h: LMX_DTYPE_*)
// ---------------------------------------------------------------------------------------------
enum DType : int { kF32 = 0, kBF16 = 1, kF16 = 2 };

static inline size_t dtype_size(int dt) { return dt == kF32 ? 4 : 2; }

struct bf16_t { uint16_t x; };   // storage-only tags; arithmetic is always fp32
struct f16_t  { uint16_t x; };

typedef __attribute__((ext_vector_type(8))) __bf16   bf16x8_v;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_v;
typedef __attribute__((ext_vector_type(16))) float   f32x16;
typedef __attribute__((ext_vector_type(4)))  float   f32x4;

template <typename T> struct TypeInfo;
template <> struct TypeInfo<float>  { static constexpr int id = kF32;  static constexpr int vec16 = 4; };
template <> struct TypeInfo<bf16_t> { static constexpr int id = kBF16; static constexpr int vec16 = 8; };
template <> struct TypeInfo<f16_t>  { static constexpr int id = kF16;  static constexpr int vec16 = 8; };

// ---- scalar conversions -------------------------------------------------------------------
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __uint_as_float(b << 16); }
// round-to-nearest-even, NaN stays NaN (same rounding torch uses for .to(bfloat16)).  The native __bf16 cast lowers to the
// gfx950 hardware converter (v_cvt_pk_bf16_f32): branch-free, one instruction per pair.
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f);
}
__device__ __forceinline__ float f16_bits_to_f32(uint32_t b) {
    _Float16 h = __builtin_bit_cast(_Float16, (uint16_t)b);
    return (float)h;
}
__device__ __forceinline__ uint32_t f32_to_f16_bits(float f) {
    _Float16 h = (_Float16)f;   // RNE
    return (uint32_t)__builtin_bit_cast(uint16_t, h);
}

template <typename T> __device__ __forceinline__ float to_f32(T v);
template <> __device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f32<bf16_t>(bf16_t v) { return bf16_bits_to_f32(v.x); }
template <> __device__ __forceinline__ float to_f32<f16_t>(f16_t v) { return f16_bits_to_f32(v.x); }

template <typename T> __device__ __forceinline__ T from_f32(float f);
template <> __device__ __forceinline__ float from_f32<float>(float f) { return f; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float f) { bf16_t r; r.x = (uint16_t)f32_to_bf16_bits(f); return r; }
template <> __device__ __forceinline__ f16_t from_f32<f16_t>(float f) { f16_t r; r.x = (uint16_t)f32_to_f16_bits(f); return r; }

// round an fp32 value through T (used where the reference rounds an intermediate to model dtype)
template <typename T> __device__ __forceinline__ float round_to(float f) { return to_f32<T>(from_f32<T>(f)); }

// One RoPE output with HF's rounding chain, T( T(x c) + T(r s) ) (HF5:models/llama/modeling_llama.py:130-160 on tensors of the model dtype: every
// elementwise op rounds).  Contraction is switched OFF here: for fp16 hipcc narrows T(x c) with half operands to a half multiply (exact) and would then be
// free to fuse it with the add into ONE half fma — skipping the rounding of the product — in one kernel and not in another (seen: rope_kv_kernel and the
// q|k|v epilogue of the prompt GEMM disagreed in 25 % of the fp16 elements by one ulp).  With the pragma every kernel computes the same, HF's, bits.
template <typename T> __device__ __forceinline__ float rope_term(float x, float c, float r, float s) {
#pragma clang fp contract(off)
    const float p = round_to<T>(x * c);
    const float q = round_to<T>(r * s);
    return round_to<T>(p + q);
}

// ---- 16-bit pair pack / unpack ------------------------------------------------------------
template <typename T> __device__ __forceinline__ uint32_t pack2(float lo, float hi);
typedef __bf16 bf16x2_v __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_v __attribute__((ext_vector_type(2)));
template <> __device__ __forceinline__ uint32_t pack2<bf16_t>(float lo, float hi) {
    const bf16x2_v v = {(__bf16)lo, (__bf16)hi};          // one v_cvt_pk_bf16_f32
    return __builtin_bit_cast(uint32_t, v);
}
template <> __device__ __forceinline__ uint32_t pack2<f16_t>(float lo, float hi) {
    const f16x2_v v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
}
template <typename T> __device__ __forceinline__ float unpack_lo(uint32_t w);
template <typename T> __device__ __forceinline__ float unpack_hi(uint32_t w);
template <> __device__ __forceinline__ float unpack_lo<bf16_t>(uint32_t w) { return __uint_as_float(w << 16); }
template <> __device__ __forceinline__ float unpack_hi<bf16_t>(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
template <> __device__ __forceinline__ float unpack_lo<f16_t>(uint32_t w) { return f16_bits_to_f32(w & 0xffffu); }
template <> __device__ __forceinline__ float unpack_hi<f16_t>(uint32_t w) { return f16_bits_to_f32(w >> 16); }

// Load / store 8 consecutive elements of T as fp32 (16-byte access for 16-bit types, 2x16 B for f32).
template <typename T> __device__ __forceinline__ void load8(const T* p, float (&v)[8]);
template <> __device__ __forceinline__ void load8<float>(const float* p, float (&v)[8]) {
    float4 a = *reinterpret_cast<const float4*>(p);
    float4 b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
template <> __device__ __forceinline__ void load8<bf16_t>(const bf16_t* p, float (&v)[8]) {
    uint4 u = *reinterpret_cast<const uint4*>(p);
    v[0] = unpack_lo<bf16_t>(u.x); v[1] = unpack_hi<bf16_t>(u.x);
    v[2] = unpack_lo<bf16_t>(u.y); v[3] = unpack_hi<bf16_t>(u.y);
    v[4] = unpack_lo<bf16_t>(u.z); v[5] = unpack_hi<bf16_t>(u.z);
    v[6] = unpack_lo<bf16_t>(u.w); v[7] = unpack_hi<bf16_t>(u.w);
}
template <> __device__ __forceinline__ void load8<f16_t>(const f16_t* p, float (&v)[8]) {
    uint4 u = *reinterpret_cast<const uint4*>(p);
    v[0] = unpack_lo<f16_t>(u.x); v[1] = unpack_hi<f16_t>(u.x);
    v[2] = unpack_lo<f16_t>(u.y); v[3] = unpack_hi<f16_t>(u.y);
    v[4] = unpack_lo<f16_t>(u.z); v[5] = unpack_hi<f16_t>(u.z);
    v[6] = unpack_lo<f16_t>(u.w); v[7] = unpack_hi<f16_t>(u.w);
}
template <typename T> __device__ __forceinline__ void store8(T* p, const float (&v)[8]);
template <> __device__ __forceinline__ void store8<float>(float* p, const float (&v)[8]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
template <> __device__ __forceinline__ void store8<bf16_t>(bf16_t* p, const float (&v)[8]) {
    uint4 u;
    u.x = pack2<bf16_t>(v[0], v[1]); u.y = pack2<bf16_t>(v[2], v[3]);
    u.z = pack2<bf16_t>(v[4], v[5]); u.w = pack2<bf16_t>(v[6], v[7]);
    *reinterpret_cast<uint4*>(p) = u;
}
template <> __device__ __forceinline__ void store8<f16_t>(f16_t* p, const float (&v)[8]) {
    uint4 u;
    u.x = pack2<f16_t>(v[0], v[1]); u.y = pack2<f16_t>(v[2], v[3]);
    u.z = pack2<f16_t>(v[4], v[5]); u.w = pack2<f16_t>(v[6], v[7]);
    *reinterpret_cast<uint4*>(p) = u;
}

// 8 elements of T as they lie in memory: requested now, converted when they are needed
template <typename T> struct Chunk8;
template <> struct Chunk8<bf16_t> {
    uint4 r;
    __device__ __forceinline__ void load(const bf16_t* p) { r = *reinterpret_cast<const uint4*>(p); }
    __device__ __forceinline__ void get(float (&v)[8]) const {
        v[0] = unpack_lo<bf16_t>(r.x); v[1] = unpack_hi<bf16_t>(r.x); v[2] = unpack_lo<bf16_t>(r.y); v[3] = unpack_hi<bf16_t>(r.y);
        v[4] = unpack_lo<bf16_t>(r.z); v[5] = unpack_hi<bf16_t>(r.z); v[6] = unpack_lo<bf16_t>(r.w); v[7] = unpack_hi<bf16_t>(r.w);
    }
};
template <> struct Chunk8<f16_t> {
    uint4 r;
    __device__ __forceinline__ void load(const f16_t* p) { r = *reinterpret_cast<const uint4*>(p); }
    __device__ __forceinline__ void get(float (&v)[8]) const {
        v[0] = unpack_lo<f16_t>(r.x); v[1] = unpack_hi<f16_t>(r.x); v[2] = unpack_lo<f16_t>(r.y); v[3] = unpack_hi<f16_t>(r.y);
        v[4] = unpack_lo<f16_t>(r.z); v[5] = unpack_hi<f16_t>(r.z); v[6] = unpack_lo<f16_t>(r.w); v[7] = unpack_hi<f16_t>(r.w);
    }
};
template <> struct Chunk8<float> {
    float r[8];
    __device__ __forceinline__ void load(const float* p) { load8<float>(p, r); }
    __device__ __forceinline__ void get(float (&v)[8]) const {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = r[e];
    }
};

// ---- wave64 / block reductions --------------------------------------------------------------
// Lanes meet in DPP moves and, past a row of 16, permlane swaps (a few cycles each; through LDS, as a shuffle goes, every step is a round trip of some 70).  The pairs are those of
// xor shuffles with N/2 .. 1: behind the step of 8 a row is periodic, so rotations are as good as the xor.  Whole waves only.  (decode_win_kernel, 16 heads x 600 keys: 11.95 -> 9.7 us; a gated linear of 11264 x 2048 with its norms 12.9 -> 11.9)
template <int CTRL> __device__ __forceinline__ float dpp_get(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true)); }
template <typename OP> __device__ __forceinline__ float fold32(float v, OP op) {      // lanes l and l ^ 32
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <typename OP> __device__ __forceinline__ float fold16(float v, OP op) {      // lanes l and l ^ 16
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
struct OpSum { __device__ __forceinline__ float operator()(float x, float y) const { return x + y; } };
struct OpMax { __device__ __forceinline__ float operator()(float x, float y) const { return fmaxf(x, y); } };
template <int N, typename OP> __device__ __forceinline__ float group_fold(float v, OP op) {
    static_assert(N == 8 || N == 16 || N == 32 || N == 64, "lanes of a group");
    if constexpr (N >= 64) v = fold32(v, op);
    if constexpr (N >= 32) v = fold16(v, op);
    if constexpr (N >= 16) { v = op(v, dpp_get<0x128>(v)); v = op(v, dpp_get<0x124>(v)); }
    else v = op(v, __shfl_xor(v, 4, 64));
    v = op(v, dpp_get<0x4E>(v));
    return op(v, dpp_get<0xB1>(v));
}
template <int N> __device__ __forceinline__ float group_sum(float v) { return group_fold<N>(v, OpSum{}); }
__device__ __forceinline__ float wave_sum(float v) { return group_sum<64>(v); }
__device__ __forceinline__ float wave_max(float v) { return group_fold<64>(v, OpMax{}); }
// sum over 8 consecutive lanes, neighbours first
__device__ __forceinline__ float sum8(float v) {
    v += dpp_get<0xB1>(v);                                  // lane ^ 1
    v += dpp_get<0x4E>(v);                                  // lane ^ 2
    return v + dpp_get<0x141>(v);                           // mirror in 8
}
// Block-wide sum for blocks of NW waves; `red` is NW floats of LDS. All threads get the result.
template <int NW> __device__ __forceinline__ float block_sum(float v, float* red) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();            // protect `red` from a previous use
    if (lane == 0) red[w] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += red[i];
    return t;
}
template <int NW> __device__ __forceinline__ float block_max(float v, float* red) {
    v = wave_max(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    float t = red[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) t = fmaxf(t, red[i]);
    return t;
}

// ---- activations (epilogue codes; mirrors include/llava_mi355x.h LMX_ACT_*) -------------------
enum Act : int { kActNone = 0, kActQuickGelu = 1, kActGeluErf = 2, kActSiluMul = 3, kActReluMul = 4 };
// gated forms: the weight's rows come in [32 gate | 32 up] groups and the output is f(gate) * up
__host__ __device__ __forceinline__ bool act_gated(int act) { return act == kActSiluMul || act == kActReluMul; }

// SiLU and quick GELU, x / (1 + e^-kx) with k = 1 and 1.702, in 32 bits.  The exponent kx log2 e is kept in two parts: rounded to one, its error is the largest of the result's, |kx| / 2 units
// of its last place.  The argument is held where the exponential is 0 or infinite either way, so that the parts are finite.  Over [-12, 12], against 64 bits and with the division, one part /
// two: SiLU 1.07 / 0.45 units of 2^-24 in the mean, 14.5 / 3.1 at most, 0.0142 / 0.0068 % of f16 and 0.0019 / 0.0009 % of bf16 results rounded the other way; quick GELU 2.11 / 0.43, 31.6 / 3.7.
constexpr float kLog2e[2] = {0x1.715476p+0f, 0x1.4ae0c0p-26f}, kQuickLog2e[2] = {0x1.3a4cbep+1f, 0x1.7c622ep-28f};      // log2 e and 1.702f log2 e to 48 bits
__device__ __forceinline__ float exp_minus(float x, const float (&k)[2]) {
    const float end = 150.f / k[0], y = -__builtin_amdgcn_fmed3f(x, -end, end), t = y * k[0];
    return __builtin_amdgcn_exp2f(t) * fmaf(fmaf(y, k[1], fmaf(y, k[0], -t)), 0x1.62e430p-1f, 1.f);
}
// x / (1 + e).  For 16-bit outputs by the reciprocal, corrected by the quotient's remainder: the division's result but for the last bit of a hundredth, in seven instructions for ten, which pays
// for the exponent (four images 3320 -> 3325 us, a 1087-position prompt 15.45 -> 15.44 ms; by the reciprocal alone 3252 and 15.31, with 0.59 units in the mean for 0.54 over [-4, 4]).  A quarter
// of both keeps the reciprocal a normal number up to the largest exponential; the fixup gives the division's answer for an infinite one.
template <typename T> __device__ __forceinline__ float over_one_plus(float x, float e) {
    if constexpr (sizeof(T) == 4) return x / (1.f + e);
    const float n = 0.25f * x, d = fmaf(0.25f, e, 0.25f), r = __builtin_amdgcn_rcpf(d), q = n * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, n), r, q), d, n);
}
template <typename T = bf16_t> __device__ __forceinline__ float act_quick_gelu(float x) { return over_one_plus<T>(x, exp_minus(x, kQuickLog2e)); }
__device__ __forceinline__ float act_gelu_erf(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }
template <typename T = bf16_t> __device__ __forceinline__ float act_silu(float x) { return over_one_plus<T>(x, exp_minus(x, kLog2e)); }
template <typename T = bf16_t> __device__ __forceinline__ float gate_mul(int act, float g, float u) { return (act == kActReluMul ? fmaxf(g, 0.f) : act_silu<T>(g)) * u; }

// logits <- cap tanh(logits / cap); cap <= 0: unchanged
__device__ __forceinline__ float soft_cap(float v, float cap) { return cap > 0.f ? cap * tanhf(v / cap) : v; }

// ---- XCD-aware block remap (8 XCDs, block b is dispatched to XCD b % 8). Bijective for any nwg.
__device__ __forceinline__ int xcd_remap(int bid, int nwg) {
    const int xcd = bid & 7, idx = bid >> 3;
    const int q = nwg >> 3, r = nwg & 7;
    const int base = (xcd < r) ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q;
    return base + idx;
}

// Logical tile id -> (tile_m, tile_n) of a 256 x 256-tile GEMM.  An XCD runs ~32 CONSECUTIVE logical ids at a time (xcd_remap), each XCD behind its own L2.
// Column-major ids (tile_m fastest) make that window 32 M-tiles of ONE N-panel: the W panel is shared by all of them, but every X panel has a single reader, so X
// is re-read from HBM once per N-panel — harmless at M ~ 1k (five M-tiles: X lives in the L2s), 9 - 12 x the algorithmic traffic at M = 32768 (3.1 GB per
// wgrad launch, 5 TB/s of HBM reads under a "compute-bound" kernel).  From 16 M-tiles on the ids walk groups of GM M-tiles, M fastest inside a group, then N:
// the window is GM x 32 / GM tiles, each X panel read by 32 / GM tiles and each W panel by GM, and a group's X panels stay hot across its whole sweep over N
// (the W panels — the weights, 100 MB at most — come back from the memory-side cache).  Same tiles, same arithmetic: only the order in which they run.
__device__ __forceinline__ void gemm_tile_of(int lid, int mtiles, int ntiles, int& tile_m, int& tile_n) {
    constexpr int GM = 4;               // measured on the 16 x 2048 training step: GM = 16 / 8 / 4 / 2 / 1 -> 1446 / 1359 / 1320 - 1333 / 1323 / 1336 ms
    if (mtiles < 16) { tile_n = lid / mtiles; tile_m = lid - tile_n * mtiles; return; }
    const int gsz = GM * ntiles;
    const int grp = lid / gsz, first = grp * GM;
    const int gm = mtiles - first < GM ? mtiles - first : GM;
    const int in = lid - grp * gsz;
    tile_n = in / gm; tile_m = first + (in - tile_n * gm);
}

// ---------------------------------------------------------------------------------------------
// host-side error plumbing: every C-ABI entry returns int; message is thread-local.
// ---------------------------------------------------------------------------------------------
void set_last_error(const std::string& s);
const char* get_last_error();

struct Error { std::string msg; };

#define LMX_CHECK_HIP(expr)                                                                        \
    do {                                                                                           \
        hipError_t _e = (expr);                                                                    \
        if (_e != hipSuccess) {                                                                    \
            throw ::lmx::Error{std::string(#expr) + " failed: " + hipGetErrorString(_e) + " (" +  \
                               __FILE__ + ":" + std::to_string(__LINE__) + ")"};                  \
        }                                                                                          \
    } while (0)

#define LMX_REQUIRE(cond, what)                                                                    \
    do {                                                                                           \
        if (!(cond)) {                                                                             \
            throw ::lmx::Error{std::string("requirement failed: ") + #cond + " — " + (what) +     \
                               " (" + __FILE__ + ":" + std::to_string(__LINE__) + ")"};          \
        }                                                                                          \
    } while (0)

static inline int cdiv(int a, int b) { return (a + b - 1) / b; }
static inline int64_t cdiv64(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace lmx
