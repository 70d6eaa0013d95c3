// Attention kernels for gfx950.
//
// Contract reproduced (reference = third-party HF code the reference repo calls, plus its own statement of the fused
// contract): scores = q·kᵀ / sqrt(D) (+ causal mask), softmax in fp32, probabilities · V.
//   HF5:models/llama/modeling_llama.py:191-214 (eager_attention_forward), :243-281 (LlamaAttention.forward)
//   HF5:models/clip/modeling_clip.py:259-335  (CLIP attention, non-causal, d=64)
//   llava/train/llama_flash_attn_monkey_patch.py:79-91 (causal=True, softmax_scale=1/sqrt(d), dropout 0)
//
// flash_prefill2_kernel (16-bit, MFMA 32x32x16): one workgroup = 4 waves on 64 query rows or 8 on 128; tiles of K and Vᵀ go by LDS-DMA into an XOR-swizzled
//   ring.  Both products keep the query index on the MFMA *column* (lane&31): Sᵀ = K·Qᵀ and Oᵀ = Vᵀ·Pᵀ, so the running max /
//   sum / rescale are per-lane scalars and P goes from the score accumulators straight into the next MFMA's B operand
//   with no cross-lane traffic (the key order inside each 16-key MFMA step is permuted identically for P and Vᵀ).
// decode_attn_kernel    (any dtype, VALU): one workgroup per (row, head, key-split); used for single-token decode
//   (HBM-bound KV streaming) and as the fp32 verification-mode attention for whole prompts.
#include <algorithm>
#include <cstdlib>
#include <functional>
#include <type_traits>
#include <vector>
#include "common.h"
#include "kernels.h"
#include "attention_decode.h"
#include "attention_mfma.h"
#include "attention_batch.h"

namespace lmx {

// flash_prefill2_kernel: the KEYS of a query block split over two wave groups: group g walks the key tiles of parity g, RW waves over the query rows, 32 each.  Tiles are staged in rounds
// (a tile of each group, by the group's own waves) into a ring of two rounds, one workgroup barrier a round.  At the end group 1 hands its (O, m, l) to group 0 through the (then free)
// ring and group 0 merges the two online-softmax states per lane: m = max(m0, m1), O = O0 2^(m0 - m) + O1 2^(m1 - m), l likewise.
// Bound: neither matrix cores nor memory alone.  128 rows x 128 keys of D = 128 take a CU 0.9 us of products, as much of exponentials and their sums and 0.6 - 1.2 us of LDS (fragments; the
// L2s would deliver the tiles four times as fast), and waves that a barrier keeps in step take them one after the other: 2.0 us.  So
//   * D = 128 takes K a round ahead of Vᵀ: a tile's exponentials stand between the next tile's score products, whose results they do not wait for, in one instruction stream (turn), with
//     the LDS reads some products ahead.  8 waves on 128 rows, 64-key tiles: 2.0 -> 1.85 us;
//   * where blocks of 128 rows leave CUs idle (flash_wide), 64 rows and 32-key tiles: four waves, two workgroups a CU, in step with nobody but themselves.
// The launch alone, repeated: 1087 causal rows of 32 heads 25.0 -> 22.5 us (inside a prompt's pass 27 -> 24.1), 139 rows on 1347 keys (with the merge of their slices) 26.8 -> 20.0, 2048
// rows of 16 heads with 4 kv heads 39.6 -> 33.2 (41 -> 35.0), D = 64: four images of 577 rows, 16 heads, 18.6 -> 17.7 (the scale in the exponential's own multiply-add).  Behind 9216 keys,
// 256 heads, 128 rows: 163 -> 153.
// WIN (FlashArgs::win): sliding window, softmax sink and output gate of the windowed decoders.  Only the key tiles a query block can see are walked: the tile
// range starts at the tile of the first row's oldest visible key, so the work per block is bounded by the window.
// Without a causal limit every row's position lies behind the last key (launch_flash_prefill): the same code, and fewer registers than a form of its own took.
// D = 64: two workgroups a CU (128 registers), which leaves no room for the next tile's scores.
constexpr int FA_SLICES_MAX = 8;
template <int D, int RW> struct FlashShape {
    static constexpr int KT = D == 128 && RW == 2 ? 32 : 64;     // keys of a tile
    static constexpr int QB = 32 * RW, THREADS = 128 * RW;       // query rows, threads of a workgroup: RW waves over the rows, 32 each, in two key groups
    static constexpr int TILE = 2 * KT * D;                      // bytes of a K or a Vᵀ tile
    static constexpr int LDS = 2 * 2 * 2 * TILE;                 // two rounds, a round being a tile of each key group
};
// block: of the launch's query blocks of every head (a.q_len rows); bz: problem of a batch
template <typename T, int D, int RW, bool WIN>
__device__ __forceinline__ void flash_body(const FlashArgs& a, const int block, const int nqb, const size_t bz, char* smem) {
    using SH = FlashShape<D, RW>;
    constexpr int KT = SH::KT, KB = KT / 32;
    constexpr int KSTEPS = D / 16;        // MFMA k-steps over the head dim (QKᵀ)
    constexpr int DB = D / 32;            // 32-row blocks of Oᵀ
    constexpr int KROWS_PP = 1024 / (D * 2);      // K rows per 1-KiB DMA piece (4 for D=128, 8 for D=64)
    constexpr int KCPR = D / 8;                   // 16-byte chunks per K row
    constexpr int KPPW = SH::TILE / 1024 / RW;    // K pieces per wave per tile
    constexpr int VPPW = SH::TILE / 1024 / RW;    // Vᵀ pieces per wave per tile
    constexpr int VROWS_PP = 1024 / (KT * 2);     // Vᵀ rows per piece
    constexpr int VCPR = KT / 8;                  // 16-byte chunks per Vᵀ row
    constexpr bool PIPE = D == 128;               // the next tile's scores beside this tile's exponentials

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wave8 % RW, grp = wave8 / RW;        // query-row wave, key group
    const int hi = lane >> 5, l31 = lane & 31;
    // 1-D grid ordered by work: ALL heads' heaviest (latest) causal query block first, then the next one, ... so the workgroups
    // that do not fit the first round (grid > CUs) are the lightest ones, not a few heads' full set
    const int head = block % a.n_heads;
    const int kvh = head / (a.n_heads / a.n_kv_heads);
    const int qb = nqb - 1 - block / a.n_heads;
    const int q0 = qb * SH::QB + wave * 32;               // this wave's first query row
    const int qrow = q0 + l31;                           // this lane's query row (column of both products)
    const int krow_pi = fa_key_perm(l31);                // key row this lane feeds to QKᵀ as tile row l31

    // scores in the log2 domain: factor behind the products
    const float sc = (a.scale != 0.f ? fabsf(a.scale) : 1.f) * 1.4426950408889634f;

    const T* __restrict__ Q = reinterpret_cast<const T*>(a.Q) + bz * a.q_batch;
    const T* __restrict__ Kc = reinterpret_cast<const T*>(a.K) + bz * a.kv_batch + (size_t)kvh * a.s_max * D;
    const T* __restrict__ Vt = reinterpret_cast<const T*>(a.VT) + bz * a.kv_batch + (size_t)kvh * D * a.s_max;

    // ---- Q fragments: B operand, lane holds Q[qrow][s*16 + hi*8 .. +8) ----------------------------------------
    uint4 qf[KSTEPS];
    {
        const int qr = qrow < a.q_len ? qrow : a.q_len - 1;
        const T* qp = Q + (size_t)qr * a.q_stride + head * D + hi * 8;
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) qf[s] = *reinterpret_cast<const uint4*>(qp + s * 16);
        // the products need a positive factor behind the maximum; others turn the queries' signs, or take them as zeros
        if (a.scale <= 0.f) {
#pragma unroll
            for (int s = 0; s < KSTEPS; ++s) {
                const uint32_t keep = a.scale < 0.f ? 0xffffffffu : 0u, turn = a.scale < 0.f ? 0x80008000u : 0u;
                qf[s] = uint4{(qf[s].x & keep) ^ turn, (qf[s].y & keep) ^ turn, (qf[s].z & keep) ^ turn, (qf[s].w & keep) ^ turn};
            }
        }
    }

    // number of key tiles this workgroup needs
    int kv_end = a.kv_len;
    {
        const int last_q = qb * SH::QB + SH::QB - 1;
        const int lim = a.q_pos0 + (last_q < a.q_len ? last_q : a.q_len - 1) + 1;
        kv_end = lim < kv_end ? lim : kv_end;
    }
    // first tile of the walk (tile indices below are relative to it)
    int tile0 = 0;
    if constexpr (WIN) {
        const int oldest = a.window > 0 ? a.q_pos0 + qb * SH::QB - a.window + 1 : 0;
        tile0 = oldest > 0 ? oldest / KT : 0;
    }
    int ntiles = (kv_end + KT - 1) / KT - tile0;
    if (a.part) {                                        // this workgroup's slice of the keys (blockIdx.z); 0 tiles: a partial row of weight 0
        const int lo = ntiles * (int)blockIdx.z / (int)gridDim.z;
        ntiles = ntiles * ((int)blockIdx.z + 1) / (int)gridDim.z - lo;
        tile0 += lo;
    }
    const int nrounds = (ntiles + 1) / 2;

    f32x16 oacc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
    // running maximum, in units of log2 (scores times sc), and sum
    float m_run = -1e30f, l_run = 0.f;
    const int my_pos = a.q_pos0 + qrow;                   // causal limit of this lane's row

    // ---- K / Vᵀ tiles by LDS-DMA into a ring of two rounds (inline asm: see gemm_pipe_kernel for why) -----------------------
    // per-lane source offsets (bytes) inside a tile; the swizzle lives in the SOURCE address, the LDS image is lane-linear.
    // Vᵀ tile in LDS: [D rows][KT keys], KT / 8 chunks of 16 bytes (8 keys) a row, chunk c of row r at c ^ (r >> 1) (64 keys) or c ^ (r >> 2) (32 keys) in the chunk's bits: a product of
    // probabilities reads whole chunks, the keys of a 32-key block being fed to QKᵀ in the order fa_key_perm, and the 16 lanes of every ds_read_b128 service group hit 16 distinct slots
    uint32_t ksrc[KPPW], vsrc[VPPW];
#pragma unroll
    for (int i = 0; i < KPPW; ++i) {
        const int row = (wave + RW * i) * KROWS_PP + lane / KCPR;         // key row inside the tile
        ksrc[i] = (uint32_t)(row * D + (((lane % KCPR) ^ (D == 128 ? row : row >> 1)) & (KCPR - 1)) * 8) * 2u;
    }
#pragma unroll
    for (int i = 0; i < VPPW; ++i) {
        const int row = (wave + RW * i) * VROWS_PP + lane / VCPR;         // d row
        vsrc[i] = ((uint32_t)row * (uint32_t)a.s_max + (((lane % VCPR) ^ (row / (16 / VCPR))) & (VCPR - 1)) * 8) * 2u;
    }
    const unsigned lds_base = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * 1024);
    auto dma = [&](const T* src, uint32_t off, unsigned dst) {
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(src), "s"(dst) : "memory");
    };
    // this wave's group stages its tile 2 r + grp of round r into slot 2 (r % 2) + grp of the ring (nothing if that tile does not exist)
    auto stage_k = [&](int r) {
        const int t = 2 * r + grp;
        if (t >= ntiles) return;
        const T* kt = Kc + (size_t)(tile0 + t) * KT * D;
        const unsigned base = lds_base + ((r & 1) * 2 + grp) * 2 * SH::TILE;
#pragma unroll
        for (int i = 0; i < KPPW; ++i) dma(kt, ksrc[i], base + i * RW * 1024);
    };
    auto stage_v = [&](int r) {
        const int t = 2 * r + grp;
        if (t >= ntiles) return;
        const T* vt = Vt + (size_t)(tile0 + t) * KT;
        const unsigned base = lds_base + ((r & 1) * 2 + grp) * 2 * SH::TILE + SH::TILE;
#pragma unroll
        for (int i = 0; i < VPPW; ++i) dma(vt, vsrc[i], base + i * RW * 1024);
    };
    auto ring_at = [&](int r) { return ((r & 1) * 2 + grp) * 2 * SH::TILE; };

    // fragment f of the stream that a tile's products read: Sᵀ = K · Qᵀ takes K rows kb 32 .. + 31, dims 16 s .. + 15 (f = 2 s + kb: two accumulator chains), Oᵀ += Vᵀ · Pᵀ takes
    // Vᵀ rows db 32 .. + 31, keys 16 step .. + 15 (f = DB step + db: DB chains; slot e of step is key 16 step + 8 hi + e of the tile, see fa_key_perm: one 16-byte read).  The chunk of
    // s or step is an xor of address bits that nothing else sets: one register of address for K and one for Vᵀ
    const int k_lane = k_lds_off<D>(krow_pi, hi), v_lane = SH::TILE + l31 * KT * 2 + (((hi ^ (l31 / (16 / VCPR))) & (VCPR - 1)) << 4);
    auto k_frag = [&](int ring, int f) { return *reinterpret_cast<const uint4*>(smem + ((ring + k_lane) ^ ((f / KB) << 5)) + f % KB * 64 * D); };
    auto v_frag = [&](int ring, int f) { return *reinterpret_cast<const uint4*>(smem + ((ring + v_lane) ^ ((f / DB) << 5)) + (f % DB) * 64 * KT); };
    auto scores = [&](f32x16 (&s)[KB], int f, const uint4& kf) { s[f % KB] = Mfma32<T>::run(kf, qf[f / KB], f < KB ? f32x16{} : s[f % KB]); };

    // s[kb][r] = score of key = tile * KT + kb * 32 + 16 (r >> 3) + 8 hi + (r & 7) and row qrow, before the scale.  What a row does not see becomes -inf (masking only on tiles that
    // can hold an invisible key for some row of this wave: a wave-uniform test); the running maximum follows.
    auto see = [&](f32x16 (&s)[KB], int t) {
        const int tile_first = (tile0 + t) * KT, tile_last = tile_first + KT - 1;
        if (tile_last >= a.kv_len || tile_last > a.q_pos0 + q0) {
            const int last = (my_pos < a.kv_len - 1 ? my_pos : a.kv_len - 1) - tile_first - 8 * hi;      // of the lane's keys
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r) s[kb][r] = kb * 32 + 16 * (r >> 3) + (r & 7) <= last ? s[kb][r] : -INFINITY;
        }
        if constexpr (WIN) {
            if (a.window > 0 && tile_first <= a.q_pos0 + q0 + 31 - a.window) {
                const int first = my_pos - a.window + 1 - tile_first - 8 * hi;
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[kb][r] = kb * 32 + 16 * (r >> 3) + (r & 7) >= first ? s[kb][r] : -INFINITY;
            }
        }
        float tmax = s[0][0];
#pragma unroll
        for (int i = 1; i < KT / 2; ++i) tmax = fmaxf(tmax, s[i >> 4][i & 15]);
        tmax = fold32(tmax, OpMax{}) * sc;
        // defer-max: keep the old running max (no O / l rescale) while no row of the wave grew by more than 2^FA_DEFER;
        // P is then bounded by 2^FA_DEFER instead of 1, which fp32 sums and 16-bit P fragments absorb.  m_run starts at
        // -1e30, so the first tile always takes the rescale branch (alpha = 0 on zero accumulators).
        if (!__all(tmax - m_run <= FA_DEFER)) {
            const float m_new = fmaxf(m_run, tmax), alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (int i = 0; i < DB; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[i][r] *= alpha;
            m_run = m_new;
        }
    };

    // Probabilities of a tile from its scores, Oᵀ += Vᵀ Pᵀ, and (NEXT) the scores of the group's next tile, as one stream of 32 slots: an exponential each, beside products of the
    // matrix cores that do not wait for it (the next tile's scores, then the products of probabilities at least a slot back), each with the LDS read of the fragment AHEAD products on.
    constexpr int AHEAD = 4;
    uint4 fr[AHEAD];
    auto read = [&](auto next_c, int kn, int vr, int m) {
        constexpr int NS = decltype(next_c)::value ? KB * KSTEPS : 0;
        if (m < NS + 2 * KB * DB) fr[m % AHEAD] = m < NS ? k_frag(kn, m) : v_frag(vr, m - NS);
    };
    auto read_ahead = [&](auto next_c, int kn, int vr) {
#pragma unroll
        for (int m = 0; m < AHEAD; ++m) read(next_c, kn, vr, m);
    };
    auto turn = [&](auto next_c, const f32x16 (&s)[KB], f32x16 (&sn)[KB], int kn, int vr) {
        constexpr bool NEXT = decltype(next_c)::value;
        constexpr int NS = NEXT ? KB * KSTEPS : 0, NP = 2 * KB * DB;
        uint4 pf[2 * KB];
        auto product = [&](int m) {
            if (m < NS) scores(sn, m, fr[m % AHEAD]);
            else oacc[(m - NS) % DB] = Mfma32<T>::run(fr[m % AHEAD], pf[(m - NS) / DB], oacc[(m - NS) % DB]);
            read(next_c, kn, vr, m + AHEAD);
        };
        float psum = 0.f, e[KT / 2];
        auto pack = [&](int j) { pf[j] = uint4{pack2<T>(e[8 * j], e[8 * j + 1]), pack2<T>(e[8 * j + 2], e[8 * j + 3]), pack2<T>(e[8 * j + 4], e[8 * j + 5]), pack2<T>(e[8 * j + 6], e[8 * j + 7])}; };
        if constexpr (PIPE) {
            static_assert(KSTEPS == 8 && DB == 4, "slots and products of the stream");
#pragma unroll
            for (int i = 0; i <= KT / 2; ++i) {
                // products of slot i: the next tile's scores one a slot, then those of the probabilities 8 j .. + 7 from slot 8 j + 9 on, one a slot or one in two, the last step's behind the
                // last slot
                if (i < KT / 2) e[i] = __builtin_amdgcn_exp2f(fmaf(s[i >> 4][i & 15], sc, -m_run));
                if (i > 0) psum += e[i - 1];                 // (a slot behind the exponential)
                if (i > 0 && i % 8 == 0) pack(i / 8 - 1);
                if (i < KT / 2) {
                    if (NEXT && i < NS) product(i);
                    else if (NEXT && KB == 2 && i < 24) product(i);
                    else if (i > 8 && (i & 1)) product(KB == 2 ? (NEXT ? 24 + (i - 25) / 2 : (i - 9) / 2) : NS + (i - 9) / 2);
                } else {
#pragma unroll
                    for (int m = NS + NP - DB; m < NS + NP; ++m) product(m);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < KT / 2; ++i) {
                e[i] = __builtin_amdgcn_exp2f(fmaf(s[i >> 4][i & 15], sc, -m_run));
                psum += e[i];
                if (i % 8 == 7) pack(i / 8);
            }
#pragma unroll
            for (int m = 0; m < NP; ++m) oacc[m % DB] = Mfma32<T>::run(v_frag(vr, m), pf[m / DB], oacc[m % DB]);
        }
        l_run += psum;
    };

    stage_k(0);
    stage_v(0);
    if constexpr (PIPE) stage_k(1);
    // Q's are the only vector-memory loads the COMPILER knows of (the DMAs are inline asm).  Waited for here, with an instruction that its wait-count pass sees, they leave the loop with
    // the one wait a round that is meant: left pending, their first use there would carry counts that also cover the DMAs on their way.
    __builtin_amdgcn_s_waitcnt(0x0F70);              // vmcnt(0); expcnt / lgkmcnt untouched
    if constexpr (PIPE) {
        // In round r K of round r + 1 and Vᵀ of round r have landed and the scores of round r are in registers: K runs a round ahead of Vᵀ in its two slots
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        f32x16 sa[KB], sb[KB];
        if (grp < ntiles) {
#pragma unroll
            for (int f = 0; f < KB * KSTEPS; ++f) scores(sa, f, k_frag(ring_at(0), f));
        }
        auto round = [&](auto next_c, f32x16 (&s)[KB], f32x16 (&sn)[KB], int r) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // everything this wave staged in the round before has landed
            __builtin_amdgcn_s_barrier();      // ... and every wave's; everyone is done with K of round r and Vᵀ of round r - 1, whose slots are free
            asm volatile("" ::: "memory");
            stage_v(r + 1);
            stage_k(r + 2);
            if constexpr (KB == 1) read_ahead(next_c, ring_at(r + 1), ring_at(r));      // on their way while the maximum is found
            see(s, 2 * r + grp);
            if constexpr (KB == 2) read_ahead(next_c, ring_at(r + 1), ring_at(r));
            turn(next_c, s, sn, ring_at(r + 1), ring_at(r));
        };
        const int mine = (ntiles + 1 - grp) / 2;              // rounds in which this wave's group has a tile
        const std::true_type next{};
        const std::false_type last{};
        int r = 0;
#pragma unroll 1
        for (; r + 2 < mine; r += 2) {
            round(next, sa, sb, r);
            round(next, sb, sa, r + 1);
        }
        // One round without a next tile for odd and even counts.  With one of each behind the loop, 128 rows took 256 registers and spilled 23, whose reloads waited for the DMAs; this form
        // takes 238 (windowed 244), 64 rows 197 for 241.  The loop is the same, the copy is 32 registers once
        if (r + 1 < mine) {
            round(next, sa, sb, r);
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) sa[kb] = sb[kb];
            ++r;
        }
        if (r < mine) round(last, sa, sb, r);
        if (mine < nrounds) {                  // an odd tile count: group 1 sits out the last round
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
        }
    } else {
#pragma unroll 1
        for (int r = 0; r < nrounds; ++r) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // everything this wave staged for round r has landed
            __builtin_amdgcn_s_barrier();      // round r visible to every wave; everyone is done with round r - 1 (its slots are free)
            asm volatile("" ::: "memory");
            stage_k(r + 1);
            stage_v(r + 1);
            const int t = 2 * r + grp;
            if (t >= ntiles) continue;
            f32x16 s[KB];
#pragma unroll
            for (int f = 0; f < KB * KSTEPS; ++f) scores(s, f, k_frag(ring_at(r), f));
            see(s, t);
            turn(std::false_type{}, s, s, 0, ring_at(r));
        }
    }

    // ---- merge the two key groups (group 1 -> LDS -> group 0), then O[q][d] = oacc / l ---------------------------------------------------
    __builtin_amdgcn_s_barrier();              // every wave is done with the ring
    float* mg = reinterpret_cast<float*>(smem) + (size_t)wave * (DB * 16 + 2) * 64;       // [reg][lane] of this query-row wave
    if (grp == 1) {
#pragma unroll
        for (int i = 0; i < DB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) mg[(i * 16 + r) * 64 + lane] = oacc[i][r];
        mg[(DB * 16) * 64 + lane] = m_run;
        mg[(DB * 16 + 1) * 64 + lane] = l_run;
    }
    __syncthreads();
    if (grp == 1) return;
    {
        const float m1 = mg[(DB * 16) * 64 + lane], l1 = mg[(DB * 16 + 1) * 64 + lane];
        const float m = fmaxf(m_run, m1);
        const float a0 = __builtin_amdgcn_exp2f(m_run - m), a1 = __builtin_amdgcn_exp2f(m1 - m);
        l_run = l_run * a0 + l1 * a1;
        m_run = m;
#pragma unroll
        for (int i = 0; i < DB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[i][r] = oacc[i][r] * a0 + mg[(i * 16 + r) * 64 + lane] * a1;
    }
    const float l_tot = fold32(l_run, OpSum{});
    if (a.part) {                                        // sums as they are, with their maximum: flash_merge_kernel
        if (qrow >= a.q_len) return;
        float* pp = a.part + (((size_t)blockIdx.z * a.q_len + qrow) * a.n_heads + head) * (D + 4);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
                *reinterpret_cast<float4*>(pp + db * 32 + 8 * q4 + 4 * hi) = float4{oacc[db][4 * q4], oacc[db][4 * q4 + 1], oacc[db][4 * q4 + 2], oacc[db][4 * q4 + 3]};
        if (hi == 0) { pp[D] = m_run; pp[D + 1] = l_tot; }
        return;
    }
    float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    if constexpr (WIN) {
        if (a.sink) {                          // the running maximum may lie below the sink's score 0: bring both sums to max(m, 0)
            const float m2 = fmaxf(m_run, 0.f), f = __builtin_amdgcn_exp2f(m_run - m2);
            inv = f / (l_tot * f + __builtin_amdgcn_exp2f(-m2));
        }
        if (a.gate && qrow < a.q_len) {
            const float g = to_f32(reinterpret_cast<const T*>(a.gate)[(size_t)qrow * a.q_stride + head]);
            inv *= 1.f / (1.f + __expf(-g));
        }
    }
    if (a.lse && hi == 0 && qrow < a.q_len) a.lse[(size_t)head * a.lse_stride + qrow] = m_run + __builtin_amdgcn_logf(l_tot);      // v_log_f32 = log2
    if (qrow < a.q_len) {
        T* op = reinterpret_cast<T*>(a.O) + bz * a.o_batch + (size_t)qrow * a.o_stride + head * D;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const int d = db * 32 + 8 * q4 + 4 * hi;
                uint2 u;
                u.x = pack2<T>(oacc[db][4 * q4 + 0] * inv, oacc[db][4 * q4 + 1] * inv);
                u.y = pack2<T>(oacc[db][4 * q4 + 2] * inv, oacc[db][4 * q4 + 3] * inv);
                *reinterpret_cast<uint2*>(op + d) = u;
            }
    }
}

template <typename T, int D, int RW, bool WIN>
__global__ __launch_bounds__((FlashShape<D, RW>::THREADS), D == 64 && !WIN ? 4 : 2) void flash_prefill2_kernel(FlashArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    flash_body<T, D, RW, WIN>(a, blockIdx.x, gridDim.x / a.n_heads, blockIdx.y, smem);
}

// Bound: a launch of one short prompt leaves most CUs idle.  32 prompts of 29 .. 64 rows, 32 heads: 8.4 us each, 268 in all -> 19.2 together; three of 1100, 894
// and 688, 16 heads: 54 -> 29 (64-row blocks; the larger ones, flash_segs_wide, were not timed in this launch)
template <typename T, int D, int RW>
__global__ __launch_bounds__((FlashShape<D, RW>::THREADS), 2) void flash_segs_kernel(FlashArgs a, RowSegs g) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int block = blockIdx.x;
    const RowSeg& s = g.s[row_segs_at(g, block)];
    const int nqb = (s.n + FlashShape<D, RW>::QB - 1) / FlashShape<D, RW>::QB;
    a.Q = reinterpret_cast<const T*>(a.Q) + (size_t)s.row0 * a.q_stride;
    a.O = reinterpret_cast<T*>(a.O) + (size_t)s.row0 * a.o_stride;
    if (a.gate) a.gate = reinterpret_cast<const T*>(a.gate) + (size_t)s.row0 * a.q_stride;
    a.K = s.K; a.VT = s.VT; a.q_len = s.n; a.kv_len = s.pos0 + s.n; a.q_pos0 = s.pos0; a.s_max = s.s_max;
    flash_body<T, D, RW, true>(a, block, nqb, 0, smem);
}

// the slices' partial rows of one (query row, head), in slice order: four dims a thread
template <typename T, int D>
__global__ __launch_bounds__(256) void flash_merge_kernel(FlashArgs a, int slices) {
    const int i = blockIdx.x * 256 + threadIdx.x, pair = i / (D / 4), d = i % (D / 4) * 4;
    if (pair >= a.q_len * a.n_heads) return;
    const size_t step = (size_t)a.q_len * a.n_heads * (D + 4);
    const float* p = a.part + (size_t)pair * (D + 4);
    float m[FA_SLICES_MAX], l[FA_SLICES_MAX];
    float4 o[FA_SLICES_MAX];
#pragma unroll
    for (int s = 0; s < FA_SLICES_MAX; ++s) {
        const float* ps = p + (s < slices ? s : 0) * step;
        m[s] = s < slices ? ps[D] : -INFINITY; l[s] = ps[D + 1]; o[s] = *reinterpret_cast<const float4*>(ps + d);
    }
    float M = m[0];
#pragma unroll
    for (int s = 1; s < FA_SLICES_MAX; ++s) M = fmaxf(M, m[s]);
    float lt = 0.f, t[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < FA_SLICES_MAX; ++s) {
        const float w = __builtin_amdgcn_exp2f(m[s] - M);
        lt = fmaf(w, l[s], lt); t[0] = fmaf(w, o[s].x, t[0]); t[1] = fmaf(w, o[s].y, t[1]); t[2] = fmaf(w, o[s].z, t[2]); t[3] = fmaf(w, o[s].w, t[3]);
    }
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    uint2 u;
    u.x = pack2<T>(t[0] * inv, t[1] * inv); u.y = pack2<T>(t[2] * inv, t[3] * inv);
    *reinterpret_cast<uint2*>(reinterpret_cast<T*>(a.O) + (size_t)(pair / a.n_heads) * a.o_stride + (pair % a.n_heads) * D + d) = u;
}

// Key slices of a launch: where its workgroups leave half of the places on the CUs empty or more, as many as fill them, of at least four 64-key tiles each.
// 139 rows on 1347 keys, 32 heads of 128 (64 workgroups of 11 rounds): 30.5 us -> 17.5 with four slices and 5.0 for the merge.
static int flash_slices(int D, const FlashArgs& a, int workgroups, bool wide) {
    if (!a.part || a.win || a.lse || a.n_batch != 1) return 1;
    int s = std::min(std::min((D == 128 && wide ? 256 : 512) / workgroups, cdiv(a.kv_len, FA_KT) / 4), FA_SLICES_MAX);
    while (s > 1 && (size_t)s * a.q_len * a.n_heads * (D + 4) * sizeof(float) > a.part_bytes) --s;
    return std::max(s, 1);
}

// Which query blocks, D = 128.  128 rows (eight waves, a workgroup a CU) read K and Vᵀ from L2 and LDS for twice the rows, 64 rows (four waves, two workgroups a CU whose barriers are
// their own) divide the work twice as finely, and the matrix cores of one workgroup run beside the exponentials of the other.  The larger blocks where they keep the chip busy to the end:
// their work over 256 CUs against what the busiest CU has, the block with the most tiles or, in a second round (heaviest first), what the last of the first and the first of the second
// take together.  us, 128 -> 64 rows:  1087 causal rows, 32 heads (0.65 of the time busy) 25.0 -> 22.5;  1100, 16 heads (0.31) 22.6 -> 19.8;  2048, 16 heads (0.53) 36.6 -> 33.2;  2048 in a
// window of 1024, 32 heads (0.79) 50.5 -> 45.5;  2048, 32 heads (1.0) 52.9 -> 55.8;  128 rows behind 9216, 256 heads (1.0) 159 -> 172.  The line lies between 0.79 and 1.0.  Past two rounds,
// 512 blocks, always 128 rows, as before there were smaller ones: a third round of a few blocks (513 .. 767) was not compared.  The 128-row figures are of a form that spilled 23 registers.
static bool flash_wide(int D, const FlashArgs& a) {
    if (D != 128) return true;
    const int nqb = cdiv(a.q_len, 128);
    auto tiles = [&](int qb) {                               // 64-key tiles of a block
        int end = a.kv_len, first = 0;
        if (a.causal) end = std::min(end, a.q_pos0 + std::min(128 * (qb + 1), a.q_len));
        if (a.win && a.window > 0) first = std::max(0, a.q_pos0 + qb * 128 - a.window + 1) / FA_KT;
        return cdiv(end, FA_KT) - first;
    };
    const long heads = (long)a.n_heads * a.n_batch, blocks = nqb * heads;
    if (blocks < 256) return false;
    long all = 0;
    for (int qb = 0; qb < nqb; ++qb) all += tiles(qb) * heads;
    auto nth = [&](long i) { return i < blocks ? tiles(nqb - 1 - (int)(i / heads)) : 0; };
    const int busiest = blocks > 512 ? 0 : std::max(nth(0), nth(255) + nth(256));
    return all >= 0.9 * 256 * busiest;
}

void launch_flash_prefill(int dtype, int D, const FlashArgs& a, hipStream_t st) {
    LMX_REQUIRE(dtype == kBF16 || dtype == kF16, "flash prefill is the 16-bit path (fp32 verification uses decode_attn)");
    LMX_REQUIRE(D == 64 || D == 128, "head_dim must be 64 or 128");
    LMX_REQUIRE(a.s_max % 64 == 0, "KV cache length must be a multiple of 64");
    LMX_REQUIRE(a.kv_len <= a.s_max && a.q_len > 0, "bad lengths");
    LMX_REQUIRE(a.q_stride % 8 == 0 && a.o_stride % 4 == 0, "q/o strides must keep 16-byte alignment");
    LMX_REQUIRE(a.n_batch >= 1 && (a.n_batch == 1 || (!a.win && !a.lse && a.q_batch % 8 == 0 && a.o_batch % 4 == 0 && a.kv_batch % 8 == 0)), "flash prefill: a batch is of plain problems, 16 bytes apart");
    const bool wide = flash_wide(D, a);
    const int qblocks = cdiv(a.q_len, wide ? 128 : 64), slices = flash_slices(D, a, qblocks * a.n_heads, wide);
    const dim3 grid(qblocks * a.n_heads, a.n_batch, slices);
    {
#define LMX_FA2_LAUNCH(TT, DD, RW, WW)                                                                              \
    do {                                                                                                            \
        using SH = FlashShape<DD, RW>;                                                                              \
        auto kern = flash_prefill2_kernel<TT, DD, RW, WW>;                                                          \
        static bool attr_set = false;                                                                               \
        if (!attr_set) {                                                                                            \
            LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SH::LDS)); \
            attr_set = true;                                                                                        \
        }                                                                                                           \
        hipLaunchKernelGGL(kern, grid, dim3(SH::THREADS), SH::LDS, st, b);                                          \
    } while (0)
#define LMX_FA2_D(TT, WW) do { if (D == 64) LMX_FA2_LAUNCH(TT, 64, 4, WW); else if (wide) LMX_FA2_LAUNCH(TT, 128, 4, WW); else LMX_FA2_LAUNCH(TT, 128, 2, WW); } while (0)
        FlashArgs b = a;
        if (!a.causal) b.q_pos0 = a.kv_len;                  // every row sees every key
        if (slices == 1) b.part = nullptr;
        if (a.win) {
            LMX_REQUIRE(a.causal && !a.lse, "flash prefill: the windowed form is causal and keeps no log-sum-exp");
            if (dtype == kBF16) LMX_FA2_D(bf16_t, true); else LMX_FA2_D(f16_t, true);
        } else if (dtype == kBF16) LMX_FA2_D(bf16_t, false);
        else LMX_FA2_D(f16_t, false);
#undef LMX_FA2_D
#undef LMX_FA2_LAUNCH
        if (slices > 1) {
            const dim3 mgrid(cdiv(a.q_len * a.n_heads * (D / 4), 256));
#define LM(TT, DD) hipLaunchKernelGGL((flash_merge_kernel<TT, DD>), mgrid, dim3(256), 0, st, b, slices)
            if (dtype == kBF16) { if (D == 128) LM(bf16_t, 128); else LM(bf16_t, 64); } else { if (D == 128) LM(f16_t, 128); else LM(f16_t, 64); }
#undef LM
        }
        LMX_CHECK_HIP(hipGetLastError());
        return;
    }
}

// Which query blocks of several prompts' rows, D = 128: 128 rows as flash_wide has it, all blocks taken as heaviest first, and only where their partly empty rows cost less than the smaller
// blocks do.  With the chip full those take 1.08 times as long for the same tiles (flash_wide's last two figures: 55.8 us for 528 x 32 tiles of 64 x 64 against 52.9 for 544 x 32, 172 against
// 159 for equally many).  That holds for a few long prompts, 2 x 2048 rows of 32 heads, not for 4 x 900 (142 against 120) nor for 32 of 64.
static bool flash_segs_wide(int n_heads, int window, const RowSegs& g) {
    std::vector<int> tiles;                                  // 64-key tiles of every block of 128 rows of a head
    long all = 0, halves = 0;                                // of these, and of the blocks of 64 rows
    for (int i = 0; i < g.n; ++i) {
        const RowSeg& s = g.s[i];
        auto keys = [&](int r0, int rows) { return cdiv(s.pos0 + std::min(r0 + rows, s.n), FA_KT) - (window > 0 ? std::max(0, s.pos0 + r0 - window + 1) / FA_KT : 0); };
        for (int r = 0; r < s.n; r += 128) { tiles.push_back(keys(r, 128)); all += tiles.back(); }
        for (int r = 0; r < s.n; r += 64) halves += keys(r, 64);
    }
    const long blocks = (long)tiles.size() * n_heads;
    if (blocks < 256 || 2.0 * all > 1.08 * halves) return false;
    if (blocks > 512) return true;
    std::sort(tiles.begin(), tiles.end(), std::greater<int>());
    auto nth = [&](long i) { return i < blocks ? tiles[(size_t)(i / n_heads)] : 0; };
    return (double)all * n_heads >= 0.9 * 256 * std::max(nth(0), nth(255) + nth(256));
}

// the segments with the most keys first, as a segment's own blocks go: a long prompt that the caller names last does not begin last
FlashSegsPlan flash_segs_plan(int D, int n_heads, int window, RowSegs& g) {
    const int rows = D == 64 || flash_segs_wide(n_heads, window, g) ? 128 : 64;
    std::stable_sort(g.s, g.s + g.n, [](const RowSeg& x, const RowSeg& y) { return x.pos0 + x.n > y.pos0 + y.n; });
    return {rows, row_segs_blocks(g, [&](const RowSeg& s) { return cdiv(s.n, rows) * n_heads; })};
}

void launch_flash_segs(int dtype, int D, const FlashArgs& a, const RowSegs& segs, hipStream_t st) {
    RowSegs g = segs;
    LMX_REQUIRE(dtype == kBF16 || dtype == kF16, "flash prefill is the 16-bit path");
    LMX_REQUIRE(D == 64 || D == 128, "head_dim must be 64 or 128");
    LMX_REQUIRE(a.win && a.causal && !a.lse && !a.part && a.n_batch == 1, "flash segments: the windowed form");
    LMX_REQUIRE(a.q_stride % 8 == 0 && a.o_stride % 4 == 0, "q/o strides must keep 16-byte alignment");
    LMX_REQUIRE(g.n >= 0 && g.n <= ROW_SEGS, "flash segments: too many");
    for (int i = 0; i < g.n; ++i) {
        const RowSeg& s = g.s[i];
        LMX_REQUIRE(s.K && s.VT && s.n >= 1 && s.row0 >= 0 && s.pos0 >= 0 && s.s_max % 64 == 0 && s.pos0 + s.n <= s.s_max, "flash segments: bad lengths");
    }
    if (g.n == 0) return;
    const FlashSegsPlan plan = flash_segs_plan(D, a.n_heads, a.window, g);
#define L(TT, DD, RW) do {                                                                                                               \
        using SH = FlashShape<DD, RW>;                                                                                                   \
        auto kern = flash_segs_kernel<TT, DD, RW>;                                                                                       \
        static bool attr_set = false;                                                                                                    \
        if (!attr_set) { LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SH::LDS)); attr_set = true; } \
        hipLaunchKernelGGL(kern, dim3(plan.blocks), dim3(SH::THREADS), SH::LDS, st, a, g);                                                \
    } while (0)
#define LD(TT) do { if (D == 64) L(TT, 64, 4); else if (plan.rows == 128) L(TT, 128, 4); else L(TT, 128, 2); } while (0)
    if (dtype == kBF16) LD(bf16_t); else LD(f16_t);
#undef LD
#undef L
    LMX_CHECK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------------------------
// decode / verification attention: grid (n_heads, n_split, n_rows), 256 threads.
//   phase 1  scores: D/8 lanes per key (16-byte K loads), shuffle-reduced, written to LDS in the log2 domain
//   phase 2  block max, exp2, block sum
//   phase 3  o[d] = sum_k p[k] * Vᵀ[d][k]: 8 lanes per d row read one 128-byte line of 64 keys per step
//   partial (m, l, o[D]) -> workspace; combine kernel merges the splits.
// ---------------------------------------------------------------------------------------------------------------
template <typename T, int D>
__global__ __launch_bounds__(256) void decode_attn_kernel(DecodeAttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float* sc_lds = reinterpret_cast<float*>(smem);      // [lds_keys] scores / probabilities of this split

    const int tid = threadIdx.x, lane = tid & 63;
    const int head = blockIdx.x, split = blockIdx.y, row = blockIdx.z;
    const int kvh = head / (a.n_heads / a.n_kv_heads);
    const int pos0 = a.pos_ptr ? *a.pos_ptr : a.pos0;
    const int kv_len = a.causal ? (pos0 + row + 1) : a.kv_total;
    // key range of this split: chunks are multiples of 64 keys
    const int chunk = ((((kv_len + a.n_split - 1) / a.n_split) + 63) / 64) * 64;
    const int k_begin = split * chunk;
    int k_end = k_begin + chunk; k_end = k_end < kv_len ? k_end : kv_len;
    const int nk = k_end > k_begin ? k_end - k_begin : 0;
    // LDS carve: scores live in [0, lds_keys) floats, reduction scratch after them
    const int lds_keys = a.causal ? a.s_max : ((a.kv_total + 63) & ~63);
    float* red = sc_lds + lds_keys;

    const T* __restrict__ Q = reinterpret_cast<const T*>(a.Q) + (size_t)row * a.q_stride + head * D;
    const T* __restrict__ Kc = reinterpret_cast<const T*>(a.K) + (size_t)kvh * a.s_max * D;
    const T* __restrict__ Vt = reinterpret_cast<const T*>(a.VT) + (size_t)kvh * D * a.s_max;
    float* ws = a.ws + ((size_t)(row * a.n_heads + head) * a.n_split + split) * (D + 2);

    constexpr int LPK = D / 8;            // lanes per key
    constexpr int KPW = 64 / LPK;         // keys per wave-iteration
    const float scl = a.scale * 1.4426950408889634f;

    // ---- phase 1: scores -------------------------------------------------------------------------------------
    {
        const int sub = lane % LPK, kslot = lane / LPK;
        float qv[8]; load8<T>(Q + sub * 8, qv);
        const int wave = tid >> 6;
        for (int k0 = wave * KPW; k0 < nk; k0 += 4 * KPW) {
            const int kl = k0 + kslot;
            const int key = k_begin + (kl < nk ? kl : nk - 1);
            float kv[8]; load8<T>(Kc + (size_t)key * D + sub * 8, kv);
            float s = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) s = fmaf(qv[e], kv[e], s);
            s = group_sum<LPK>(s);
            if (sub == 0 && kl < nk) sc_lds[kl] = s * scl;
        }
    }
    __syncthreads();

    // ---- phase 2: softmax statistics ---------------------------------------------------------------------------
    float mx = -INFINITY;
    for (int k = tid; k < nk; k += 256) mx = fmaxf(mx, sc_lds[k]);
    mx = block_max<4>(mx, red);
    float sum = 0.f;
    const int nk_pad = (nk + 63) & ~63;
    for (int k = tid; k < nk_pad; k += 256) {
        float e = 0.f;
        if (k < nk) e = __builtin_amdgcn_exp2f(sc_lds[k] - mx);
        sc_lds[k] = e;                          // zero-fills the tail of the last 64-key line
        sum += e;
    }
    sum = block_sum<4>(sum, red);
    __syncthreads();

    // ---- phase 3: o = P · V ---------------------------------------------------------------------------------------
    {
        const int sub = tid & 7, drow = tid >> 3;            // 32 d rows per pass
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
            const int d = db * 32 + drow;
            float acc = 0.f;
            for (int kb = 0; kb < nk_pad; kb += 64) {
                float vv[8]; load8<T>(Vt + (size_t)d * a.s_max + k_begin + kb + sub * 8, vv);
                const float4 p0 = *reinterpret_cast<const float4*>(sc_lds + kb + sub * 8);
                const float4 p1 = *reinterpret_cast<const float4*>(sc_lds + kb + sub * 8 + 4);
                if (kb + 64 > nk) {                          // behind the last key the cache may hold Inf or NaN: 0 x NaN is NaN
#pragma unroll
                    for (int e = 0; e < 8; ++e) vv[e] = kb + sub * 8 + e < nk ? vv[e] : 0.f;
                }
                acc = fmaf(p0.x, vv[0], acc); acc = fmaf(p0.y, vv[1], acc);
                acc = fmaf(p0.z, vv[2], acc); acc = fmaf(p0.w, vv[3], acc);
                acc = fmaf(p1.x, vv[4], acc); acc = fmaf(p1.y, vv[5], acc);
                acc = fmaf(p1.z, vv[6], acc); acc = fmaf(p1.w, vv[7], acc);
            }
            acc = sum8(acc);
            if (sub == 0) ws[2 + d] = acc;
        }
    }
    if (tid == 0) { ws[0] = nk > 0 ? mx : -INFINITY; ws[1] = sum; }
}

template <typename T, int D>
__global__ __launch_bounds__(D) void decode_attn_combine_kernel(DecodeAttnArgs a) {
    const int head = blockIdx.x, row = blockIdx.y, d = threadIdx.x;
    const float* ws = a.ws + (size_t)(row * a.n_heads + head) * a.n_split * (D + 2);
    float M = -INFINITY;
    for (int s = 0; s < a.n_split; ++s) M = fmaxf(M, ws[s * (D + 2)]);
    float l = 0.f, o = 0.f;
    for (int s = 0; s < a.n_split; ++s) {
        const float m = ws[s * (D + 2)];
        if (m == -INFINITY) continue;
        const float w = __builtin_amdgcn_exp2f(m - M);
        l += w * ws[s * (D + 2) + 1];
        o += w * ws[s * (D + 2) + 2 + d];
    }
    T* op = reinterpret_cast<T*>(a.O) + (size_t)row * a.o_stride + head * D;
    op[d] = from_f32<T>(l > 0.f ? o / l : 0.f);
}

size_t decode_attn_ws_floats(int n_rows, int n_heads, int n_split, int D) {
    return (size_t)n_rows * n_heads * n_split * (D + 2);
}

template <typename T, int D>
static void launch_decode_attn_t(const DecodeAttnArgs& a, hipStream_t st) {
    const int lds_keys = a.causal ? a.s_max : ((a.kv_total + 63) & ~63);
    const size_t smem = (size_t)lds_keys * 4 + 64;
    auto kern = decode_attn_kernel<T, D>;
    static bool attr_set = false;
    if (!attr_set) {
        LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        attr_set = true;
    }
    hipLaunchKernelGGL(kern, dim3(a.n_heads, a.n_split, a.n_rows), dim3(256), smem, st, a);
    LMX_CHECK_HIP(hipGetLastError());
    hipLaunchKernelGGL((decode_attn_combine_kernel<T, D>), dim3(a.n_heads, a.n_rows), dim3(D), 0, st, a);
    LMX_CHECK_HIP(hipGetLastError());
}

void launch_decode_attn(int dtype, int D, const DecodeAttnArgs& a, hipStream_t st) {
    LMX_REQUIRE(D == 64 || D == 128, "head_dim must be 64 or 128");
    LMX_REQUIRE(a.s_max % 64 == 0, "KV cache length must be a multiple of 64");
    LMX_REQUIRE(a.n_split >= 1 && a.ws != nullptr, "decode attention needs a workspace");
    LMX_REQUIRE((size_t)(a.causal ? a.s_max : a.kv_total + 64) * 4 + 64 <= 160 * 1024, "score row does not fit LDS");
#define LMX_DA(TT)                                                                                     \
    do { if (D == 128) launch_decode_attn_t<TT, 128>(a, st); else launch_decode_attn_t<TT, 64>(a, st); } while (0)
    if (dtype == kBF16) LMX_DA(bf16_t);
    else if (dtype == kF16) LMX_DA(f16_t);
    else if (dtype == kF32) LMX_DA(float);
    else throw Error{"decode_attn: bad dtype"};
#undef LMX_DA
}

}  // namespace lmx

// ---------------------------------------------------------------------------------------------------------------
// Fused single-token decode attention: RoPE(q, k_new) + KV append + split-K partials in one launch.
// grid (n_heads, n_split), 256 threads.  The newest key/value never round-trips through the cache inside this launch:
// every block whose key range contains `pos` rotates k_new / reads v_new straight from the qkv row, and exactly one block
// per kv head (first q head of the group, owning split) writes them to the caches for later steps.
// ---------------------------------------------------------------------------------------------------------------
namespace lmx {

template <typename T, int D>
__global__ __launch_bounds__(256) void decode_fused_kernel(DecodeFusedArgs a) {
    decode_fused_body<T, D>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

size_t decode_fused_ws_floats(int n_heads, int n_split, int D) { return (size_t)n_heads * n_split * (D + 4); }

// Order of the sequences of a launch of n_heads workgroups each.  Two workgroups share a CU from the start (registers), the k-th and the (k + 256)-th, and all later ones start where
// one ends: the longest first, the second 256 the other way round, so that the longest and the shortest of the first 512 meet, then again the longest first.  (16 sequences of 1087 ..
// 516 keys already sorted, 32 heads: the pairs (1087, 782) .. (820, 514) of the order as it is take 43.2 us, (1087, 514) .. (820, 782) 40.9.)  16 .. 64 heads, 7 .. 64 sequences, us a launch
// as they come -> in this order:  32 heads of 16 random lengths 36.0 -> 31.2, 32 66.4 -> 61.8;  40 heads of 10 34.0 -> 32.5, of 18 55.0 -> 46.2;  16 heads of 32 36.9 -> 33.0;  up to 256 workgroups,
// and sorted lengths past them but for 16 x 32, within 3 % either way.
void batch_attn_order(const int* len, int n_seq, int n_heads, uint8_t* order) {
    for (int i = 0; i < n_seq; ++i) order[i] = (uint8_t)i;
    std::stable_sort(order, order + n_seq, [&](uint8_t a, uint8_t b) { return len[a] > len[b]; });
    const int half = std::min(n_seq, (256 + n_heads - 1) / n_heads);
    std::reverse(order + half, order + std::min(n_seq, 2 * half));
}

// Where the heads do not divide 256 the reversed ones can be the last of the launch and reach past the first 512 workgroups: the longest of them would start when others end.  40 heads, 14
// sequences (560 workgroups), as they come / in order: 38.7 / 44.4 us with random lengths, 46.6 / 48.4 sorted.
bool batch_attn_ordered(int n_seq, int n_heads) { return n_seq * n_heads <= 512 || n_seq > 2 * ((256 + n_heads - 1) / n_heads); }

void launch_decode_fused(int dtype, int D, const DecodeFusedArgs& a, hipStream_t st) {
    LMX_REQUIRE(D == 64 || D == 128, "head_dim must be 64 or 128");
    LMX_REQUIRE(a.s_max % DF_CHUNK == 0 || a.s_max % 64 == 0, "KV cache length must be a multiple of 64");
    // n_split = the caller's count of 128-key chunks to visit: at least every chunk that holds a key of the longest sequence (the host mirrors the positions)
    LMX_REQUIRE(a.n_split >= 1 && a.n_split <= DF_MAX_SPLIT && (a.n_split - 1) * DF_CHUNK < a.s_max, "decode_fused: n_split must be 1..32 chunks of 128 keys inside the cache");
    LMX_REQUIRE(a.cos_sin && a.O && (a.tab ? a.n_seq >= 1 : (a.ws && a.pos_ptr && a.counters)), "decode_fused: bad arguments");
    if (a.tab && D == 128 && (dtype == kBF16 || dtype == kF16) && a.s_max % BA_PIECE == 0) {
        // the decode batch of 16-bit models with head_dim 128 (attention_batch.h): one workgroup per (sequence, head), waves stream the keys — 44.8 -> 38.9 us per
        // layer at 8 sequences, 143 -> 134 at 32 against the chunked launch below (profiles/r05_batch_attn_wave.jsonl)
        if (dtype == kBF16) launch_decode_attn_wave_t<bf16_t>(a, st); else launch_decode_attn_wave_t<f16_t>(a, st);
        LMX_CHECK_HIP(hipGetLastError());
        return;
    }
#define LMX_DF(TT, DD) hipLaunchKernelGGL((decode_fused_kernel<TT, DD>), dim3(a.n_heads, a.n_split, a.tab ? a.n_seq : 1), dim3(256), 0, st, a)
    if (dtype == kBF16) { if (D == 128) LMX_DF(bf16_t, 128); else LMX_DF(bf16_t, 64); }
    else if (dtype == kF16) { if (D == 128) LMX_DF(f16_t, 128); else LMX_DF(f16_t, 64); }
    else if (dtype == kF32) { if (D == 128) LMX_DF(float, 128); else LMX_DF(float, 64); }
    else throw Error{"decode_fused: bad dtype"};
#undef LMX_DF
    LMX_CHECK_HIP(hipGetLastError());
}

}  // namespace lmx

// ---------------------------------------------------------------------------------------------------------------
// output_attentions: one workgroup per (query row, head); wave w takes keys w, w + 4, ... (a key row is one coalesced 64-lane read), the scores wait in LDS for
// the row's softmax.  Rounding points of the eager path (kernels.h: AttnProbsArgs).
// ---------------------------------------------------------------------------------------------------------------
namespace lmx {

template <typename T, int D>
__global__ __launch_bounds__(256) void attn_probs_kernel(AttnProbsArgs a) {
    extern __shared__ float ap_sc[];                          // [kv_total] scores, then 4 floats for the reductions
    float* red = ap_sc + a.kv_total;
    const int i = blockIdx.x, h = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int kvh = h / (a.n_heads / a.n_kv_heads);
    const int n_keys = min(a.pos0 + i + 1, a.kv_total);
    constexpr int E = D / 64;
    const T* q = reinterpret_cast<const T*>(a.Q) + (size_t)i * a.q_stride + (size_t)h * D + lane * E;
    const T* K = reinterpret_cast<const T*>(a.K) + (size_t)kvh * a.s_max * D + lane * E;
    float qv[E];
#pragma unroll
    for (int e = 0; e < E; ++e) qv[e] = to_f32(q[e]);
    for (int j = wave; j < n_keys; j += 4) {
        const T* kr = K + (size_t)j * D;
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) s = fmaf(qv[e], to_f32(kr[e]), s);
        s = wave_sum(s);
        if (lane == 0) ap_sc[j] = round_to<T>(round_to<T>(s) * a.scale);
    }
    __syncthreads();
    float m = -INFINITY;
    for (int j = tid; j < n_keys; j += 256) m = fmaxf(m, ap_sc[j]);
    m = block_max<4>(m, red);
    float l = 0.f;
    for (int j = tid; j < n_keys; j += 256) { const float p = expf(ap_sc[j] - m); ap_sc[j] = p; l += p; }
    l = block_sum<4>(l, red);
    T* out = reinterpret_cast<T*>(a.P) + ((size_t)h * a.rows_total + a.row0 + i) * a.kv_total;
    for (int j = tid; j < a.kv_total; j += 256) out[j] = from_f32<T>(j < n_keys ? ap_sc[j] / l : 0.f);
}

void launch_attn_probs(int dtype, int D, const AttnProbsArgs& a, hipStream_t st) {
    LMX_REQUIRE(D == 64 || D == 128, "head_dim must be 64 or 128");
    LMX_REQUIRE(a.Q && a.K && a.P && a.n_rows >= 1 && a.row0 >= 0 && a.row0 + a.n_rows <= a.rows_total, "attn_probs: bad arguments");
    LMX_REQUIRE(a.pos0 >= 0 && a.pos0 + a.n_rows <= a.kv_total && a.kv_total <= a.s_max, "attn_probs: rows past the key range");
    LMX_REQUIRE(a.n_kv_heads >= 1 && a.n_heads % a.n_kv_heads == 0, "attn_probs: heads must be a multiple of kv heads");
    const size_t smem = ((size_t)a.kv_total + 8) * sizeof(float);
    LMX_REQUIRE(smem <= 64 * 1024, "attn_probs: score row does not fit LDS");
#define LMX_AP(TT, DD) hipLaunchKernelGGL((attn_probs_kernel<TT, DD>), dim3(a.n_rows, a.n_heads), dim3(256), smem, st, a)
    if (dtype == kBF16) { if (D == 128) LMX_AP(bf16_t, 128); else LMX_AP(bf16_t, 64); }
    else if (dtype == kF16) { if (D == 128) LMX_AP(f16_t, 128); else LMX_AP(f16_t, 64); }
    else if (dtype == kF32) { if (D == 128) LMX_AP(float, 128); else LMX_AP(float, 64); }
    else throw Error{"attn_probs: bad dtype"};
#undef LMX_AP
    LMX_CHECK_HIP(hipGetLastError());
}

}  // namespace lmx
