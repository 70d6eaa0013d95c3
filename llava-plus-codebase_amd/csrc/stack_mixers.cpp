// Mixers and mixtures of the layer-stack decoders besides softmax attention (stack.cpp): launch sequences of latent attention, the gated delta rule and the mixture of
// experts, for the rows of a prompt piece and for one new token per sequence.
#include "engine.h"

namespace lmx {

struct StackProf { const char *delta, *norm, *uq, *qlat, *attn, *olat, *router, *plan, *gate_up, *down; };
#define NAMES(P, UQ) {P ".delta", P ".latent_norm", UQ, P ".latent_q", P ".attn", P ".latent_o", P ".moe.router", P ".moe.plan", P ".moe.gate_up", P ".moe.down"}
const StackProf stack_prof_prefill = NAMES("prefill", "prefill.gemm.uq"), stack_prof_decode = NAMES("decode", "decode.gemv.uq"), stack_prof_batch = NAMES("decode_batch", "decode_batch.linear");
#undef NAMES

static int round_up(int a, int b) { return (a + b - 1) / b * b; }
static size_t up256(size_t b) { return (b + 255) / 256 * 256; }

size_t Stack::ws_bytes(int rows, int H, int es, bool decode) const {
    const size_t r = (size_t)rows;
    return (decode ? up256(r * q_n * es) + 2 * up256(r * lat_n * es) : 0) + up256(r * moe_act * es) + up256(r * moe_top * H * es) + 2 * up256(r * moe_top * 4) +
           (moe_top ? up256(group_plan_bytes(rows * moe_top)) : 0) + (c.loop_mix ? up256(r * 2 * H * es) : 0);
}

StackWs Stack::ws(void* base, int rows, int H, int es, bool decode) const {
    char* p = static_cast<char*>(base);
    const size_t r = (size_t)rows;
    auto take = [&](size_t bytes) -> void* { void* q = p; p += up256(bytes); return q; };
    StackWs w{};
    if (decode) { w.q = take(r * q_n * es); w.qlat = take(r * lat_n * es); w.olat = take(r * lat_n * es); }
    w.act = take(r * moe_act * es);
    w.slots = take(r * moe_top * H * es);
    w.ids = static_cast<int*>(take(r * moe_top * 4));
    w.wt = static_cast<float*>(take(r * moe_top * 4));
    if (moe_top) w.plan = take(group_plan_bytes(rows * moe_top));
    if (c.loop_mix) w.cat = take(r * 2 * H * es);
    return w;
}

// ---------------------------------------------------------------------------------------------------------------
// prompt rows
// ---------------------------------------------------------------------------------------------------------------
// keys [k0, end) that the rows of a segment can see, k0 on a 64-key boundary
static int first_key(const lmx_layer_config& d, int pos0) { return d.window > 0 && pos0 - d.window + 1 > 0 ? (pos0 - d.window + 1) & ~63 : 0; }

// several prompts from their first rows on, all in one launch each of norm, expansion, caches and attention (32 prompts of 29 .. 64 rows, a latent layer of 4096: 32 x (3.4 + 9.7 + 4.6 +
// 8.4) us -> 6.5 + 27.7 + 18.0 + 19.2).  Rows that go on behind cached ones see keys that are no rows of the piece: those pieces take the segments one after the other
static bool fresh_together(int dtype, int D, const std::vector<Model::Segment>& seg) {
    if (dtype == kF32 || D > 128 || seg.size() < 2) return false;
    for (const Model::Segment& g : seg) if (g.pos0) return false;
    return true;
}

// Rows whose keys and values are there at a time, of whole prompts: 8192 or the longest prompt (`keys` bounds it).  5 x their heads' width stands in scratch: 32 prompts of 2000 rows at 4096
// would take 2.76 GB all at once, 0.92 so, and a product of 8192 rows fills the chip as well as one of 64000
static int together_rows(int rows, int keys) { return std::min(rows, std::max(keys, 8192)); }

size_t latent_prefill_scratch(int an, int R, int es, int window, int rows, int keys, int n) {
    const int nk = window > 0 ? std::min(keys, rows + window + 64) : keys;
    const size_t q = up256((size_t)rows * an * es), apart = q + up256((size_t)nk * 2 * an * es) + 2 * up256((size_t)round_up(nk, 128) * an * es);
    if (n < 2) return apart;
    const int t = together_rows(rows, keys);                 // fresh_together: latents of all rows, of t rows keys and values by row and caches of whole 128 keys each
    return std::max(apart, q + up256((size_t)rows * R * es) + up256((size_t)t * 2 * an * es) + 2 * up256((size_t)(t + 127 * std::min(n, ROW_SEGS)) * an * es));
}

// scratch of the widest mixer; keys: longest context of the call, n: sequences
size_t Model::stack_mix_scratch(int rows, int keys, int n) const {
    size_t most = 0;
    for (const StackLayer& l : stk->layers) {
        size_t b = 0;
        if (l.c.mixer == LMX_MIXER_LATENT) b = latent_prefill_scratch(l.an, l.R, es, l.c.window, rows, keys, n);
        else if (l.c.mixer == LMX_MIXER_DELTA) b = up256((size_t)rows * l.ds.H * (l.ds.DK + l.ds.DV) * es) + delta_scratch_bytes(l.ds, rows, es);
        most = std::max(most, b);
    }
    return most;
}

void Model::stack_mix_prefill(int r, Seq* const* seqs, const std::vector<Segment>& seg, int fill, const void* x, void* qkv, void* mix, void* scratch, const DevBuf& skw, hipStream_t st) {
    Stack& S = *stk;
    const StackRun& run = S.runs[(size_t)r];
    const StackLayer& l = S.layers[(size_t)run.layer];
    const lmx_layer_config& d = l.c;
    const int dt = cfg.dtype, gv = cfg.gemm_variant;
    char* p = static_cast<char*>(scratch);
    auto take = [&](size_t bytes) -> char* { char* q = p; p += up256(bytes); return q; };
    auto gemm = [&](const char* name, GemmArgs g) { LMX_PROF_K(name);
        // inner sizes of a few K-steps: the time is the launch's fixed part and the output; the smaller tiles write it sooner than the large ones
        const int v = gv == 0 && dt != kF32 && g.K <= 512 ? (g.K <= 256 ? 5 : 18) : gv;
        if (g.K >= 1024) g.scratch(skw.p, skw.bytes);
        launch_gemm(dt, g, v, st); };
    if (d.mixer == LMX_MIXER_DELTA) {
        DeltaPrefillArgs a{};
        a.s = l.ds; a.w = DeltaWeights{l.conv, l.a_log, l.dt_bias, l.onorm};
        a.proj = qkv; a.ld = l.qkv_n;
        const int agn = l.ds.H * (l.ds.DK + l.ds.DV), k = l.ra + l.rg;
        void* ag = take((size_t)fill * agn * es);
        gemm("prefill.gemm.decay_gate", GemmArgs{static_cast<char*>(qkv) + (size_t)l.a_off() * es, l.wag, ag, nullptr, nullptr, fill, agn, k, l.qkv_n, k, agn, 0, kActNone});
        a.ag = ag; a.ag_ld = agn;
        delta_carve(a, p, fill, es);
        a.out = mix; a.out_ld = l.out_k; a.eps = S.c.norm_eps;
        for (size_t s0 = 0; s0 < seg.size(); s0 += DELTA_MAX_SEG) {
            a.n_seg = (int)std::min(seg.size() - s0, (size_t)DELTA_MAX_SEG);
            for (int i = 0, chunks = 0; i < a.n_seg; ++i) {
                const Segment& g = seg[s0 + (size_t)i];
                char* rs = seqs[g.seq]->rs.as<char>();
                a.seg[i] = DeltaSeg{g.dst0, g.n, g.pos0, chunks, reinterpret_cast<float*>(rs + run.s_off), rs + run.r_off};
                chunks += (g.n + 15) / 16;
            }
            { LMX_PROF_K("prefill.delta.prep"); launch_delta_prep(dt, a, st); }
            { LMX_PROF_K("prefill.delta.scan"); launch_delta_scan(dt, a, st); }
            { LMX_PROF_K("prefill.delta.gate"); launch_delta_gate(dt, a, st); }
        }
        return;
    }
    if (fresh_together(dt, l.D, seg)) {
        // every key is a row of this piece: one product makes the keys and values of many prompts
        int longest = 0;
        for (const Segment& g : seg) longest = std::max(longest, g.n);
        const int most = together_rows(fill, longest);
        char* q = take((size_t)fill * l.an * es);
        char* lat = take((size_t)fill * l.R * es);
        char* kv = take((size_t)most * 2 * l.an * es);
        const size_t cache = (size_t)(most + 127 * std::min((int)seg.size(), ROW_SEGS)) * l.an * es;
        char *kc = take(cache), *vt = take(cache);
        auto groups = [&](size_t s0, size_t end, auto&& f) {             // as many segments as a launch takes
            for (; s0 < end; s0 += ROW_SEGS) {
                RowSegs g{};
                g.n = (int)std::min(end - s0, (size_t)ROW_SEGS);
                f(g, seg.data() + s0);
            }
        };
        groups(0, seg.size(), [&](RowSegs& g, const Segment* s) {
            LMX_PROF("prefill.latent_norm");
            for (int i = 0; i < g.n; ++i) g.s[i] = RowSeg{s[i].dst0, s[i].n, 0, s_max, 0, seqs[s[i].seq]->kc.as<char>() + run.k_off, nullptr};
            LatentNormArgs n{qkv, l.qkv_n, l.Q, d.q_rank, l.R, d.kv_rank, l.qn_lat, l.kn_lat, nullptr, 0};
            n.eps = S.c.norm_eps; n.lat = lat;
            launch_latent_norm_segs(dt, n, g, st);
        });
        gemm("prefill.gemm.uq", GemmArgs{qkv, l.wuq, q, nullptr, nullptr, fill, l.an, l.Q, l.qkv_n, l.Q, l.an, 0, kActNone});
        for (size_t s0 = 0, s1; s0 < seg.size(); s0 = s1) {
            const int first = seg[s0].dst0;
            int rows = 0;
            for (s1 = s0; s1 < seg.size() && rows + seg[s1].n <= most; ++s1) rows += seg[s1].n;
            gemm("prefill.gemm.ukv", GemmArgs{lat + (size_t)first * l.R * es, l.wukv, kv, nullptr, nullptr, rows, 2 * l.an, l.R, l.R, l.R, 2 * l.an, 0, kActNone});
            groups(s0, s1, [&](RowSegs& g, const Segment* s) {
                size_t at = 0;
                for (int i = 0; i < g.n; ++i) {
                    const int cap = round_up(s[i].n, 128);
                    g.s[i] = RowSeg{s[i].dst0 - first, s[i].n, 0, cap, cap, kc + at, vt + at};      // the attention tiles are whole: what lies behind the last key must not be NaN bits
                    at += (size_t)cap * l.an * es;
                }
                {
                    LMX_PROF("prefill.kv_rows");
                    launch_qkv_norm_rope_segs(dt, l.D, QkvNormRopeArgs{kv, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 2 * l.an, 0, d.n_heads, 0, l.D, 0, S.c.norm_eps}, g, st);
                }
                LMX_PROF("prefill.attn");
                FlashArgs fa{q + (size_t)first * l.an * es, static_cast<char*>(mix) + (size_t)first * l.out_k * es, nullptr, nullptr, 0, 0, 0, l.an, l.out_k, d.n_heads, d.n_heads, 0, d.attn_scale, 1};
                fa.win = 1; fa.window = d.window; fa.sink = d.softmax_sink;
                launch_flash_segs(dt, l.D, fa, g, st);
            });
        }
        return;
    }
    // latent attention: latents into the cache, queries, then per segment the keys and values its rows can see
    for (const Segment& g : seg) {
        LMX_PROF("prefill.latent_norm");
        LatentNormArgs n{static_cast<char*>(qkv) + (size_t)g.dst0 * l.qkv_n * es, l.qkv_n, l.Q, d.q_rank, l.R, d.kv_rank, l.qn_lat, l.kn_lat, seqs[g.seq]->kc.as<char>() + run.k_off, g.pos0};
        n.s_max = s_max; n.eps = S.c.norm_eps;
        launch_latent_norm(dt, n, g.n, st);
    }
    void* q = take((size_t)fill * l.an * es);
    gemm("prefill.gemm.uq", GemmArgs{qkv, l.wuq, q, nullptr, nullptr, fill, l.an, l.Q, l.qkv_n, l.Q, l.an, 0, kActNone});
    char* const base = p;
    for (const Segment& g : seg) {
        p = base;
        const int k0 = first_key(d, g.pos0), nk = g.pos0 + g.n - k0, cap = round_up(nk, 128);
        const char* lat = seqs[g.seq]->kc.as<char>() + run.k_off + (size_t)k0 * l.R * es;
        void* kv = take((size_t)nk * 2 * l.an * es);
        void *kc = take((size_t)cap * l.an * es), *vt = take((size_t)cap * l.an * es);
        gemm("prefill.gemm.ukv", GemmArgs{lat, l.wukv, kv, nullptr, nullptr, nk, 2 * l.an, l.R, l.R, l.R, 2 * l.an, 0, kActNone});
        {
            LMX_PROF("prefill.kv_rows");
            QkvNormRopeArgs ra{kv, kc, vt, nullptr, nullptr, nullptr, nk, 0, 2 * l.an, 0, d.n_heads, cap, l.D, 0, S.c.norm_eps};
            ra.zero_to = cap;                                // the attention tiles are whole: what lies behind the last key must not be NaN bits
            launch_qkv_norm_rope_kv(dt, l.D, ra, st);
        }
        LMX_PROF("prefill.attn");
        FlashArgs fa{static_cast<char*>(q) + (size_t)g.dst0 * l.an * es, static_cast<char*>(mix) + (size_t)g.dst0 * l.out_k * es, kc, vt, g.n, nk, g.pos0 - k0, l.an, l.out_k, d.n_heads, d.n_heads, cap,
                     d.attn_scale, 1};
        fa.win = 1; fa.window = d.window; fa.sink = d.softmax_sink;
        if (dt == kF32 || l.D > 128) launch_rows_attn(dt, l.D, fa, st); else launch_flash_prefill(dt, l.D, fa, st);
    }
}

// ---------------------------------------------------------------------------------------------------------------
// one new token per sequence
// ---------------------------------------------------------------------------------------------------------------
bool Model::stack_mix_decode(int r, const DecodeFusedSeq* tab, const DecodeFusedSeq& one, int n, int max_len, const void* x, void* qkv, void* mix, const StackWs& w, Batch* b, hipStream_t st, const GemvArgs* beside) {
    Stack& S = *stk;
    const StackLayer& l = S.layers[(size_t)S.runs[(size_t)r].layer];
    const lmx_layer_config& d = l.c;
    const int dt = cfg.dtype;
    const StackProf& pn = b ? stack_prof_batch : stack_prof_decode;
    // a parallel layer's mixture reads the mixer's input row: its choice is one workgroup more of the mixer's longest launch.  A launch of its own takes 8 us for 64 KB of router rows
    const MoeRouterArgs router = l.parallel() && l.moe() && opt_stack_fuse ? stack_router(l, x, w) : MoeRouterArgs{};
    if (d.mixer == LMX_MIXER_DELTA) {
        DeltaDecodeArgs a{};
        a.s = l.ds; a.w = DeltaWeights{l.conv, l.a_log, l.dt_bias, l.onorm};
        a.proj = qkv; a.ld = l.qkv_n; a.a_off = l.a_off(); a.ra = l.ra; a.rg = l.rg;
        a.wag = l.wag; a.wag_ld = l.ra + l.rg; a.out = mix; a.out_ld = l.out_k;
        a.tab = tab; a.one = one; a.n_seq = n; a.eps = S.c.norm_eps;
        if (delta_decode_routes(l.ds, n)) a.router = router;
        LMX_PROF_K(beside ? "decode.delta_gate_up" : pn.delta);
        if (beside) launch_delta_decode_linear(dt, a, *beside, st); else launch_delta_decode(dt, a, st);
        return a.router.x;
    }
    const bool routes = router.x && latent_decode_routes(dt, l.R);
    {
        LMX_PROF_K(pn.norm);
        LatentNormArgs a{qkv, l.qkv_n, l.Q, d.q_rank, l.R, d.kv_rank, l.qn_lat, l.kn_lat, one.K, 0};
        a.tab = tab; a.pos_ptr = tab ? nullptr : one.pos_ptr; a.s_max = s_max; a.eps = S.c.norm_eps;
        launch_latent_norm(dt, a, n, st);
    }
    {
        LMX_PROF_K(pn.uq);
        if (b) stack_batch_linear(b, GemmArgs{qkv, l.wuq, w.q, nullptr, nullptr, n, l.an, l.Q, l.qkv_n, l.Q, l.an, 0, kActNone}, l.sw_uq, st);
        else launch_gemv(dt, GemvArgs{qkv, l.wuq, w.q, nullptr, nullptr, nullptr, 0.f, l.an, l.Q, l.qkv_n, l.Q, l.an, 0, kActNone}, 1, st);
    }
    // q W_uk of every head: the scores against all cached latents are then plain dot products
    GroupGemvArgs g{w.q, l.wuk_t, w.qlat, l.R, l.D, l.an, l.D, d.n_heads * l.R, (size_t)l.R * l.D};
    g.groups = d.n_heads; g.x_group = l.D; g.c_group = l.R;
    { LMX_PROF_K(pn.qlat); stack_heads(g, n, st); }
    {
        LMX_PROF_K(pn.attn);
        LatentDecodeArgs a;
        a.q = w.qlat; a.out = w.olat; a.tab = tab; a.one = one; a.n_seq = n; a.H = d.n_heads; a.R = l.R; a.s_max = s_max; a.window = d.window; a.scale = d.attn_scale;
        int span = max_len + 1;
        if (d.window > 0 && d.window < span) span = d.window;
        a.n_split = latent_decode_split(dt, l.R, d.n_heads, n, span);
        if (routes) a.router = router;
        launch_latent_decode(dt, a, st);
    }
    GroupGemvArgs o{w.olat, static_cast<char*>(l.wukv) + (size_t)l.an * l.R * es, mix, l.D, l.R, d.n_heads * l.R, l.R, l.out_k, (size_t)l.D * l.R};
    o.groups = d.n_heads; o.x_group = l.R; o.c_group = l.D;
    { LMX_PROF_K(pn.olat); stack_heads(o, n, st); }
    return routes;
}

// every head's rows through the head's own weight
void Model::stack_heads(const GroupGemvArgs& g, int n, hipStream_t st) {
    const int dt = cfg.dtype;
    if (dt == kF32 || n < 4) { launch_group_gemv(dt, g, n * g.groups, st); return; }
    GroupGemmArgs a{g.X, g.W, g.C, g.N, g.K, g.ldx, g.ldw, g.ldc, g.w_group, n, g.groups};
    a.x_group = g.x_group; a.c_group = g.c_group;
    launch_group_gemm(dt, a, n <= 32 ? 32 : 64, st);
}

// ---------------------------------------------------------------------------------------------------------------
// mixture of experts: choices, then both products with the rows as they are (few: weights streamed per row) or sorted by expert (MFMA tiles)
// ---------------------------------------------------------------------------------------------------------------
MoeRouterArgs Model::stack_router(const StackLayer& l, const void* x, const StackWs& w) const { return MoeRouterArgs{x, l.wr, l.br, H, H, l.c.experts, l.c.top_experts, w.ids, w.wt}; }
GroupGemvArgs Model::stack_moe_first(const StackLayer& l, const void* x, const StackWs& w) const {
    GroupGemvArgs g{x, l.wgu, w.act, 2 * l.ff, H, H, H, l.ff, (size_t)2 * l.ff * H};
    g.act = l.act(); g.ids = w.ids; g.per_row = l.c.top_experts;
    return g;
}
void Model::stack_moe(const StackLayer& l, const void* x, int rows, const StackWs& w, const StackProf& pn, hipStream_t st, bool routed, const GemvArgs* beside) {
    const int dt = cfg.dtype, top = l.c.top_experts, E = l.c.experts, slots = rows * top;
    if (!routed) { LMX_PROF_K(pn.router); launch_moe_router(dt, stack_router(l, x, w), rows, st); }
    if (group_gemm_applies(dt, slots, E)) {
        GroupGemmArgs p[2] = {{x, l.wgu, w.act, 2 * l.ff, H, H, H, l.ff, (size_t)2 * l.ff * H, slots, E}, {w.act, l.wd, w.slots, H, l.ff, l.ff, l.ff, H, (size_t)H * l.ff, slots, E}};
        p[0].act = l.act(); p[0].per_row = top;
        p[0].plan = p[1].plan = group_plan_at(w.plan, slots);
        const int bm = group_gemm_bm(p, 2);
        { LMX_PROF_K(pn.plan); launch_group_plan(w.ids, slots, E, bm, p[0].plan, st); }
        { LMX_PROF_K(pn.gate_up); launch_group_gemm(dt, p[0], bm, st); }
        { LMX_PROF_K(pn.down); launch_group_gemm(dt, p[1], bm, st); }
        return;
    }
    const GroupGemvArgs g = stack_moe_first(l, x, w);
    { LMX_PROF_K(beside ? "decode.moe.gate_up_o" : pn.gate_up); if (beside) launch_group_gemv_linear(dt, g, slots, *beside, st); else launch_group_gemv(dt, g, slots, st); }
    GroupGemvArgs o{w.act, l.wd, w.slots, H, l.ff, l.ff, l.ff, H, (size_t)H * l.ff};
    o.ids = w.ids;
    { LMX_PROF_K(pn.down); launch_group_gemv(dt, o, slots, st); }
}

}  // namespace lmx
