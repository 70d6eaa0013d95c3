// Host side of the four-wave GEMM (kernels: gemm4w.h): which tile and how many K slices, and the launch.
#include <algorithm>
#include <iterator>
#include <mutex>

#include "gemm4w.h"

namespace lmx {

LMX_GEMM4W_LARGE(LMX_GEMM4W_EXTERN, bf16_t)
LMX_GEMM4W_SMALL(LMX_GEMM4W_EXTERN, bf16_t)
LMX_GEMM4W_LARGE(LMX_GEMM4W_EXTERN, f16_t)
LMX_GEMM4W_SMALL(LMX_GEMM4W_EXTERN, f16_t)

namespace {

struct Tile { int8_t mb, nb; };
#define LMX_GEMM4W_TILE(T, MB, NB) {MB, NB},
constexpr Tile kTiles[] = {LMX_GEMM4W_LARGE(LMX_GEMM4W_TILE, ) LMX_GEMM4W_SMALL(LMX_GEMM4W_TILE, )};

// Time of a launch (us).  K-steps fitted to 112 linears back to back; epilogues, slices and the rest to 900 products of 257 .. 8000 rows x 512 .. 28000 weights x 64 .. 14000, every
// activation, with and without residual and bias, every tile of the table, 1 .. 3 slices, each form for 3.5 ms ahead of its timing (the chip at its power limit) on weights from memory
// (1.6 GB of them in turn).  7 % rms at the form it picks, which is 0.9 % behind the best one of the table in the mean, 30 % at most.  256 workgroups are a round, one a CU.
//   a K-step:  0.24 us + 0.0129 a block of the tile + 0.0066 a block of its sides
//   a round that leaves CUs idle has their power: its K-steps take 0.76 + 0.24 x (the share of CUs at work) of that
//   an epilogue:  2 us + 0.093 a block, more with an activation (vector ALUs at one wave a SIMD), a residual or a bias; of a slice 5 us, then the reduction's launch and its reads
float cost(const GemmArgs& a, int mb, int nb, int S) {
    const int area = mb * nb, tiles = cdiv(a.M, 32 * mb) * cdiv(a.N, 32 * nb) * S;
    const bool gated = act_gated(a.act);
    const float steps = cdiv(a.K / 64, S) * (0.24f + 0.0129f * area + 0.0066f * (mb + nb));
    float block = gated ? 0.187f : a.act == kActQuickGelu ? 0.429f : a.act != kActNone ? 0.642f : 0.093f;
    if (a.R) block += 0.152f;
    if (a.bias && (gated || a.act == kActNone)) block += 0.077f;      // (the other activations were timed with theirs)
    const float epi = S > 1 ? 5.1f : block * area + 2.06f;
    float t = (tiles / 256) * (steps + epi);
    if (const int rem = tiles % 256) t += steps * (0.76f + 0.24f * (rem / 256.f)) + epi;
    if (S > 1) t += 4.5f + 1.27e-6f * S * a.M * a.N;
    return 1.6f + 1.03f * t;
}

// fallback K-slice scratch for callers that bring none and ask for slices (lmx_op_gemm: unit tests, microbenchmarks; ONE stream at a time).
// The engine passes per-sequence scratch instead (Model::prefill), so concurrent request threads never share it.
struct FallbackWs {
    std::mutex mu;
    void* ws = nullptr; size_t ws_bytes = 0;
};
FallbackWs g_fb;

template <typename T> void launch_t(const GemmArgs& a, const TileForm& f, hipStream_t st) {
#define LMX_GEMM4W_CASE(T_, MB, NB) case MB * 16 + NB: gemm4w_launch<T_, MB, NB>(a, f.slices, st); return;
    switch (f.mb * 16 + f.nb) {
        LMX_GEMM4W_LARGE(LMX_GEMM4W_CASE, T)
        LMX_GEMM4W_SMALL(LMX_GEMM4W_CASE, T)
        default: throw Error{"gemm4w: no such tile"};
    }
}

// A grouped product on tiles of mb x nb blocks, by rounds fitted to back-to-back launches of 112 linears of 139 .. 6528 rows (6 % rms).  The host does not know the groups' rows: the mean
// over loads around the average.  Over 75 .. 670 rows a group of two mixtures (16 groups, 2816 x 2048 and 2048 x 1408, 5504 x 4096 and 4096 x 2752, rows spread at random) the tile this
// picks is 2.5 % behind the best one in the mean; over ten grouped products of 70 .. 900 rows a group 3.1 %
float group_rounds(int tiles, int n, int act, int mb, int nb) {
    const int area = mb * nb;
    const float steps = n * (0.24f + 0.0129f * area + 0.0066f * (mb + nb)), epi = (act_gated(act) ? 0.34f : act != kActNone ? 0.64f : 0.215f) * area - 2.2f;
    float t = (tiles / 256) * (steps + epi);
    if (const int rem = tiles % 256) {
        const float share = rem / 256.f;
        t += steps * (0.76f + 0.24f * share) + epi * std::max(0.5f, share);
    }
    return t;
}
float group_cost(const GroupGemmArgs& a, int mb, int nb) {
    const float avg = (float)a.rows / a.groups;
    float t = 0.f;
    for (const float load : {0.85f, 0.92f, 1.f, 1.08f, 1.15f}) {
        const int m_tiles = a.groups * std::max(1, cdiv((int)(avg * load), 32 * mb));
        t += 0.2f * group_rounds(m_tiles * cdiv(a.N, 32 * nb), a.K / 64, a.act, mb, nb);
    }
    return t;
}
int group_nb(const GroupGemmArgs& a, int mb, float* least) {
    int best = 0;
    for (const Tile& t : kTiles) {
        if (t.mb != mb) continue;
        const float c = group_cost(a, mb, t.nb);
        if (!best || c < *least) { best = t.nb; *least = c; }
    }
    return best;
}
template <typename T> void launch_group_t(const GroupGemmArgs& a, int mb, int nb, int m_tiles, hipStream_t st) {
#define LMX_GROUP4W_CASE(T_, MB, NB) case MB * 16 + NB: group_gemm4w_launch<T_, MB, NB>(a, m_tiles, st); return;
    switch (mb * 16 + nb) {
        LMX_GEMM4W_LARGE(LMX_GROUP4W_CASE, T)
        LMX_GEMM4W_SMALL(LMX_GROUP4W_CASE, T)
        default: throw Error{"group_gemm: no such tile"};
    }
}

}  // namespace

bool group_gemm4w_applies(const GroupGemmArgs& a) {
    return a.plan.n_tiles && a.rows % a.per_row == 0 && (size_t)(a.rows / a.per_row) * a.ldx * 2 < ((size_t)1 << 32) && (size_t)a.N * a.ldw * 2 < ((size_t)1 << 32);
}
int group_gemm4w_bm(const GroupGemmArgs* a, int n) {
    int best = 0;
    float least = 0.f;
    for (int mb = 4; mb <= 8; ++mb) {
        float sum = 0.f, c = 0.f;
        for (int i = 0; i < n; ++i) { group_nb(a[i], mb, &c); sum += c; }
        if (!best || sum < least) { best = mb; least = sum; }
    }
    return 32 * best;
}
void launch_group_gemm4w(int dtype, const GroupGemmArgs& a, int bm, int nb, int m_tiles, hipStream_t st) {
    LMX_REQUIRE(bm % 32 == 0 && bm >= 128 && bm <= 256 && group_gemm4w_applies(a), "group_gemm: bad tiles");
    float c = 0.f;
    if (nb == 0) nb = group_nb(a, bm / 32, &c);
    if (dtype == kBF16) launch_group_t<bf16_t>(a, bm / 32, nb, m_tiles, st);
    else launch_group_t<f16_t>(a, bm / 32, nb, m_tiles, st);
}

// what the slices of a product may need at most: the scratch of any tile form (and of 256 x 256 tiles, which callers size theirs by)
size_t gemm4w_slab_bytes(int M, int N, const TileForm& f) {
    if (f.slices <= 1) return 0;
    const size_t tile = (size_t)cdiv(M, 32 * f.mb) * cdiv(N, 32 * f.nb) * f.mb * f.nb * 1024, whole = (size_t)cdiv(M, 256) * cdiv(N, 256) * 65536;
    return f.slices * std::max(tile, whole) * sizeof(float);
}

// Which products: more than 256 rows (below, the row tiles of gemm_rows.hip read every weight once) and more than 640 tiles of 64 x 64; past 384 rows, with a K from 8192 on, more than 160
// and, with a K from 5120 on and 1024 weights or more, more than 256; of these those that no other form makes in less time (linear_form).  Long K under the line of 640: 144 products of
// 385 .. 3000 rows x 768 .. 5504 weights, time of the form before / here 1.24 in the mean, 0.975 .. 1.6 (957 x 1280 x 11008 69.8 / 46.1 us, 800 x 1536 x 5632 32.2 / 25.2), 90 with SiLU, GELU
// or quick GELU 1.33, 0.98 .. 2.2; up to 384 rows, where the row tiles come in slices, 1.07 (351 x 2816 x 11008 42.4 / 43.8).  Under 1024 weights and a K of 8192 the times err most, both
// ways: 2878 x 832 x 5120 with a residual 38.6 / 44.1, 2622 x 768 x 5120 31.3 / 35.0, 3068 x 512 x 5824 30.1 / 33.5, but 2638 x 960 x 6144 49.6 / 40.2, 1641 x 768 x 7680 55.4 / 35.4.
// K of 4096 0.83 .. 1.13, of 1024 .. 2560 0.64 .. 1.13.  Below the line otherwise, us theirs / here, by shape:  800 x 1024 x 2048 10.3 / 14.1   2000 x 512 x 2048 12.9 / 14.8
//   257 x 6208 x 2048 15.1 / 17.1   330 x 4544 x 2304 15.9 / 17.3   577 x 4096 x 1024 13.3 / 13.9,  but  700 x 3072 x 1024 11.4 / 9.8   2308 x 1024 x 4096 30.5 / 27.2
//   500 x 4096 x 11008 74.3 / 63.3.
TileForm gemm4w_form(int dtype, const GemmArgs& a, float* us) {
    const TileForm none{0, 0, 1};
    if ((dtype != kBF16 && dtype != kF16) || a.c_f32 || a.K % 64 != 0 || a.N % 8 != 0 || (act_gated(a.act) && a.N % 64 != 0) || (a.pk_kc && a.pk_D % 8 != 0)) return none;
    if (a.R && a.ldr % 4 != 0) return none;                  // residual rows of any pitch: another kernel's
    if ((size_t)a.M * a.ldx * 2 >= ((size_t)1 << 32) || (size_t)a.N * a.ldw * 2 >= ((size_t)1 << 32)) return none;
    const int line = a.M <= 384 ? 640 : a.K >= 8192 ? 160 : a.K >= 5120 && a.N >= 1024 ? 256 : 640;
    if (!a.qf_kc && (a.M <= 256 || (int64_t)cdiv(a.M, 64) * cdiv(a.N, 64) <= line)) return none;      // (the q|k|v epilogue is here alone: gemm_fuses_qkv's lines)
    TileForm best = none;
    float least = 0.f;
    for (const Tile& t : kTiles) {
        if (a.qf_kc && t.nb != 8) continue;
        const int64_t tiles = (int64_t)cdiv(a.M, 32 * t.mb) * cdiv(a.N, 32 * t.nb);
        for (int S = 1; S <= 3; ++S) {
            const TileForm f{t.mb, t.nb, S};
            if (S > 1 && (!a.skw || a.pk_kc || a.qf_kc || tiles * S > 272 || a.K / 64 / S < 10 || gemm4w_slab_bytes(a.M, a.N, f) > a.skw_bytes())) break;
            const float c = cost(a, t.mb, t.nb, S);
            if (!best.mb || c < least) { best = f; least = c; }
        }
    }
    if (us) *us = least;
    return best;
}

void launch_gemm4w(int dtype, GemmArgs a, TileForm f, hipStream_t st) {
    // (forms by number come here without launch_gemm's and gemm4w_form's checks)
    LMX_REQUIRE(dtype == kBF16 || dtype == kF16, "gemm4w: 16-bit dtypes only");
    LMX_REQUIRE(std::any_of(std::begin(kTiles), std::end(kTiles), [&](const Tile& t) { return t.mb == f.mb && t.nb == f.nb; }), "gemm4w: no such tile");
    LMX_REQUIRE(a.K % 64 == 0, "gemm4w: K must be a multiple of 64");
    LMX_REQUIRE(a.ldx % 8 == 0 && a.ldw % 8 == 0, "gemm4w: leading dims must keep 16-byte row alignment");
    LMX_REQUIRE((size_t)a.M * a.ldx * 2 < ((size_t)1 << 32) && (size_t)a.N * a.ldw * 2 < ((size_t)1 << 32), "gemm4w: operands must be addressable with 32-bit byte offsets");
    LMX_REQUIRE(!act_gated(a.act) || a.N % 64 == 0, "gemm4w: SiLU·mul needs N % 64 == 0");
    LMX_REQUIRE(a.N % 4 == 0 && a.ldc % 4 == 0 && (!a.R || a.ldr % 4 == 0) && !a.c_f32, "gemm4w: rows of 8 bytes, 16-bit output");
    f.slices = std::max(1, std::min({f.slices, 3, cdiv(a.K / 64, 2)}));       // slices of whole pairs of K-steps
    if (f.slices > 1 && !a.skw) {
        std::lock_guard<std::mutex> lk(g_fb.mu);
        const size_t need = (gemm4w_slab_bytes(a.M, a.N, f) + 1023) / 1024 * 1024;
        if (need > g_fb.ws_bytes) {
            LMX_CHECK_HIP(hipStreamSynchronize(st));
            if (g_fb.ws) (void)hipFree(g_fb.ws);
            g_fb.ws = nullptr; g_fb.ws_bytes = 0;
            LMX_CHECK_HIP(hipMalloc(&g_fb.ws, need)); g_fb.ws_bytes = need;
        }
        a.scratch(g_fb.ws, g_fb.ws_bytes);
    }
    LMX_REQUIRE(f.slices == 1 || gemm4w_slab_bytes(a.M, a.N, f) <= a.skw_bytes(), "gemm4w: the partial tiles do not fit the scratch");
    if (a.qf_kc) LMX_REQUIRE(f.slices == 1 && f.nb == 8 && a.qf_rope && a.qf_vt && (a.qf_D == 64 || a.qf_D == 128) && (a.qf_nh * a.qf_D) % 256 == 0 && (a.qf_nkv * a.qf_D) % 256 == 0 &&
                             a.N == (a.qf_nh + 2 * a.qf_nkv) * a.qf_D && a.qf_pos0 % 8 == 0 && a.qf_smax % 8 == 0 && !a.bias && !a.R && a.act == kActNone && a.ldc % 8 == 0,
                             "gemm4w: the fused q|k|v epilogue needs an un-split launch over head-aligned tiles (gemm_fuses_qkv)");
    // the CLIP K / V^T pack lives in the un-split epilogue only: a K-sliced launch's reduction would write the k | v columns to C and leave the pack untouched
    if (a.pk_kc) LMX_REQUIRE(f.slices == 1 && !act_gated(a.act) && a.pk_D % 8 == 0 && a.N % 8 == 0, "gemm4w: the K / V^T pack epilogue needs an un-split launch of a plain linear");
    if (dtype == kBF16) launch_t<bf16_t>(a, f, st);
    else launch_t<f16_t>(a, f, st);
}

}  // namespace lmx
