// Grouped linears and mixtures of experts.
//
//   moe_router_kernel    fp32 router logits, the `top` largest and the softmax over them
//   group_plan_kernel    rows of every expert side by side, cut into tiles
//   group_gemm_kernel    the rows of a group times its weight on MFMA tiles (16-bit), groups of up to 64 rows (more of them: gemm4w.h)
//   group_gemv_kernel    one row through the weight of its group (an expert, or a head), weights streamed straight into the vector ALUs
#include <algorithm>

#include "common.h"
#include "kernels.h"
#include "gemm_common.h"
#include "moe_pick.h"
#include "gemv2.h"

namespace lmx {

// grid (rows), 64 NW threads
template <typename T, int NW>
__global__ __launch_bounds__(64 * NW) void moe_router_kernel(MoeRouterArgs a) { moe_router_row<T, NW>(a, blockIdx.x); }

void launch_moe_router(int dtype, const MoeRouterArgs& a, int rows, hipStream_t st) {
    LMX_REQUIRE(a.x, "moe_router: bad arguments");
    check_router(a);
    if (rows <= 0) return;
#define L(TT) do { if (rows <= 64) LMX_LAUNCH((moe_router_kernel<TT, 16>), dim3(rows), dim3(1024), 0, st, a); else LMX_LAUNCH((moe_router_kernel<TT, 4>), dim3(rows), dim3(256), 0, st, a); } while (0)
    if (dtype == kBF16) L(bf16_t); else if (dtype == kF16) L(f16_t); else L(float);
#undef L
    LMX_CHECK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------------------------
// plan of a grouped product: slots sorted by expert (order) and the tiles of `bm` rows they make.  One workgroup
// ---------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void group_plan_kernel(const int* ids, int slots, int E, int bm, GroupPlan p) {
    __shared__ int cnt[MOE_MAX_E], pos[MOE_MAX_E], scan[2][MOE_MAX_E], tsum[2][MOE_MAX_E];
    const int tid = threadIdx.x;
    if (tid < MOE_MAX_E) cnt[tid] = 0;
    __syncthreads();
    for (int i = tid; i < slots; i += 1024) atomicAdd(&cnt[ids[i]], 1);
    __syncthreads();
    if (tid < MOE_MAX_E) { scan[0][tid] = cnt[tid]; tsum[0][tid] = (cnt[tid] + bm - 1) / bm; }
    __syncthreads();
    int b = 0;
    for (int o = 1; o < MOE_MAX_E; o <<= 1, b ^= 1) {
        if (tid < MOE_MAX_E) {
            scan[b ^ 1][tid] = scan[b][tid] + (tid >= o ? scan[b][tid - o] : 0);
            tsum[b ^ 1][tid] = tsum[b][tid] + (tid >= o ? tsum[b][tid - o] : 0);
        }
        __syncthreads();
    }
    if (tid < E) {
        const int n = cnt[tid], nt = (n + bm - 1) / bm, r0 = scan[b][tid] - n, t0 = tsum[b][tid] - nt;
        pos[tid] = r0;
        for (int t = 0; t < nt; ++t) p.tiles[t0 + t] = GroupTile{tid, r0 + t * bm, n - t * bm < bm ? n - t * bm : bm, t0, nt, {0, 0, 0}};
    }
    if (tid == MOE_MAX_E - 1) *p.n_tiles = tsum[b][tid];
    __syncthreads();
    for (int i = tid; i < slots; i += 1024) p.order[atomicAdd(&pos[ids[i]], 1)] = i;
}

size_t group_plan_bytes(int slots) { return 256 + ((size_t)slots * 4 + 255) / 256 * 256 + ((size_t)slots / GROUP_MIN_BM + MOE_MAX_E + 1) * sizeof(GroupTile); }
GroupPlan group_plan_at(void* base, int slots) {
    char* p = static_cast<char*>(base);
    return GroupPlan{reinterpret_cast<int*>(p + 256), reinterpret_cast<GroupTile*>(p + 256 + ((size_t)slots * 4 + 255) / 256 * 256), reinterpret_cast<int*>(p)};
}
// Rows of a tile.  From 65 rows a group on the four-wave tiles (gemm4w.h) that make the cheapest rounds; below them 32 or 64 rows, what an average group fills.  us of both
// products of a mixture of 16, tiles of 64 rows (or, the best before, 128 and 256 rows of eight waves and a ring of two) / four-wave tiles:
//   2048 wide, experts of 1408: 50 rows a group 51 / 50   75: 62 / 51   130: 75 / 55   250: 103 / 81   385: 157 / 111   670: 239 / 184
//   4096 wide, experts of 2752: 50 rows a group 215 / 212   75: 264 / 229   130: 316 / 249   250: 399 / 322   385: 516 / 384   670: 787 / 618
int group_gemm_bm(const GroupGemmArgs* a, int n) {
    const int avg = a->rows / a->groups;
    bool four = avg > 64;
    for (int i = 0; i < n; ++i) four = four && group_gemm4w_applies(a[i]);
    return four ? group_gemm4w_bm(a, n) : avg <= 24 ? 32 : 64;
}
bool group_gemm_applies(int dtype, int slots, int groups) { return dtype != kF32 && slots >= 16 && slots >= groups; }
void launch_group_plan(const int* ids, int slots, int E, int bm, const GroupPlan& p, hipStream_t st) {
    LMX_REQUIRE(ids && slots >= 1 && E >= 1 && E <= MOE_MAX_E && bm >= GROUP_MIN_BM && p.order && p.tiles && p.n_tiles, "group_plan: bad arguments");
    LMX_LAUNCH(group_plan_kernel, dim3(1), dim3(1024), 0, st, ids, slots, E, bm, p);
    LMX_CHECK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------------------------
// MFMA tiles of a grouped product: the LDS ring of gemm_pipe_kernel (gemm.hip) with a row list.  Logical tiles run group by group, a group's row tiles next to each
// other for one panel of its weight.  The grid is an upper bound: workgroups past the plan's tile count leave at once.
// ---------------------------------------------------------------------------------------------------------------
template <typename T, int BM, int BN, int WM, int WN, int NSTAGE, bool STREAM>
__global__ __launch_bounds__(WM * WN * 64) void group_gemm_kernel(GroupGemmArgs a) {
    constexpr int NW = WM * WN, TM = BM / WM, TN = BN / WN, MT = TM / 32, NTL = TN / 32, PIECES = (BM + BN) / 8, PPW = PIECES / NW;
    constexpr int BUF_BYTES = (BM + BN) * GEMM_ROWB;
    static_assert(PIECES % NW == 0 && NTL % 2 == 0 && NSTAGE >= 2 && NSTAGE <= 4 && (NSTAGE - 2) * PPW <= 63, "tile");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, hi = lane >> 5, l31 = lane & 31;
    const int nt = (a.N + BN - 1) / BN;
    int grp, row0, rows, tile_n;
    if (a.plan.n_tiles) {
        const int total = *a.plan.n_tiles * nt;
        if ((int)blockIdx.x >= total) return;
        const int lid = xcd_remap(blockIdx.x, total);
        const GroupTile t = a.plan.tiles[lid / nt];
        const int rel = lid - t.first * nt;
        const GroupTile u = a.plan.tiles[t.first + rel % t.n_tiles];
        grp = u.group; row0 = u.row0; rows = u.rows; tile_n = rel / t.n_tiles;
    } else {
        const int mt = (a.rows + BM - 1) / BM, lid = xcd_remap(blockIdx.x, a.groups * mt * nt), rel = lid % (mt * nt);
        grp = lid / (mt * nt); tile_n = rel / mt; row0 = rel % mt * BM;
        rows = a.rows - row0 < BM ? a.rows - row0 : BM;
    }
    grp = __builtin_amdgcn_readfirstlane(grp); row0 = __builtin_amdgcn_readfirstlane(row0); rows = __builtin_amdgcn_readfirstlane(rows); tile_n = __builtin_amdgcn_readfirstlane(tile_n);
    const int n0 = tile_n * BN;
    const T* X = reinterpret_cast<const T*>(a.X) + (size_t)grp * a.x_group;
    const T* W = reinterpret_cast<const T*>(a.W) + (size_t)grp * a.w_group;
    const T* gsrc[PPW];
#pragma unroll
    for (int i = 0; i < PPW; ++i) {
        const int row = (wave + NW * i) * 8 + (lane >> 3), chunk = ((lane & 7) ^ (row >> 1)) & 7;
        if (row < BM) {
            int m = row0 + (row < rows ? row : rows - 1);
            if (a.plan.order) m = a.plan.order[m] / a.per_row;
            gsrc[i] = X + (size_t)m * a.ldx + chunk * 8;
        } else {
            int n = n0 + row - BM; n = n < a.N ? n : a.N - 1;
            gsrc[i] = W + (size_t)n * a.ldw + chunk * 8;
        }
    }
    f32x16 acc[NTL][MT];
#pragma unroll
    for (int i = 0; i < NTL; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    const int nk = a.K / GEMM_BK;
    const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    const int rot = STREAM ? (tile_n * 5 + grp * 3) % nk : 0;      // (in step, all tiles ask for the same 128 bytes of every weight row at a time)
    auto stage = [&](int kt, unsigned buf_off) {             // (inline asm for the reason given in gemm_pipe_kernel: ordering is the counted vmcnt + s_barrier below)
        int k = kt;
        if constexpr (STREAM) { k += rot; k = k < nk ? k : k - nk; }
#pragma unroll
        for (int i = 0; i < PPW; ++i) {
            const unsigned dst = __builtin_amdgcn_readfirstlane(lds_base + buf_off + (wave + NW * i) * 1024);
            const T* src = gsrc[i] + (size_t)k * GEMM_BK;
            unsigned keep;
            if (STREAM && (wave + NW * i) * 8 >= BM)         // (wave-uniform)
                asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt\n\ts_mov_b32 m0, %0"
                             : "=&s"(keep) : "v"(src), "s"(dst) : "memory");
            else
                asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                             : "=&s"(keep) : "v"(src), "s"(dst) : "memory");
        }
    };
#pragma unroll
    for (int i = 0; i < NSTAGE - 1; ++i) if (i < nk) stage(i, i * BUF_BYTES);
    int slot = 0;
    for (int kt = 0; kt < nk; ++kt) {
        const int rem = nk - 1 - kt;                         // tiles allowed to stay in flight past this wait: min(NSTAGE - 2, rem)
        if (NSTAGE >= 4 && rem >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NSTAGE >= 4 ? 2 * PPW : 0) : "memory");
        else if (NSTAGE >= 3 && rem >= 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PPW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();                        // tile kt visible to every wave; everyone is done reading the slot that is filled next
        if (kt + NSTAGE - 1 < nk) { int s2 = slot + NSTAGE - 1; s2 = s2 >= NSTAGE ? s2 - NSTAGE : s2; stage(kt + NSTAGE - 1, s2 * BUF_BYTES); }
        const char* buf = smem + slot * BUF_BYTES;
#pragma unroll
        for (int ks = 0; ks < GEMM_BK / 16; ++ks) {
            uint4 wf[NTL], xf[MT];
#pragma unroll
            for (int i = 0; i < NTL; ++i) wf[i] = *reinterpret_cast<const uint4*>(buf + lds_chunk_off(BM + wn * TN + i * 32 + l31, ks * 2 + hi));
#pragma unroll
            for (int j = 0; j < MT; ++j) xf[j] = *reinterpret_cast<const uint4*>(buf + lds_chunk_off(wm * TM + j * 32 + l31, ks * 2 + hi));
#pragma unroll
            for (int i = 0; i < NTL; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) acc[i][j] = Mfma32x32x16<T>::run(wf[i], xf[j], acc[i][j]);
        }
        slot = slot + 1 == NSTAGE ? 0 : slot + 1;
    }
    const bool gated = act_gated(a.act);
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int r = wm * TM + j * 32 + l31;
        if (r >= rows) continue;
        const int m = a.plan.order ? a.plan.order[row0 + r] : row0 + r;
        T* C = reinterpret_cast<T*>(a.C) + (size_t)m * a.ldc + (size_t)grp * a.c_group;
#pragma unroll
        for (int i = 0; i < NTL; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + wn * TN + i * 32 + 8 * q + 4 * hi;      // (gated: 32 gate rows, then 32 up rows)
                if (n >= a.N || (gated && (i & 1))) continue;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = gated ? gate_mul(a.act, acc[i][j][4 * q + e], acc[i | 1][j][4 * q + e]) : acc[i][j][4 * q + e];
                store4<T>(C + (gated ? (n - 8 * q - 4 * hi) / 2 + 8 * q + 4 * hi : n), v);
            }
    }
}

template <typename T, int BM, int BN, int WM, int WN, int NSTAGE, bool STREAM>
static void launch_group_gemm_cfg(const GroupGemmArgs& a, int m_tiles, hipStream_t st) {
    constexpr int smem = NSTAGE * (BM + BN) * GEMM_ROWB;
    static_assert(smem <= 160 * 1024, "LDS ring does not fit");
    auto kern = group_gemm_kernel<T, BM, BN, WM, WN, NSTAGE, STREAM>;
    static bool attr_set = false;
    if (!attr_set) { LMX_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem)); attr_set = true; }
    LMX_LAUNCH(kern, dim3(m_tiles * cdiv(a.N, BN)), dim3(WM * WN * 64), smem, st, a);
    LMX_CHECK_HIP(hipGetLastError());
}
// Tiles of 32 and 64 rows.  Weights that nearly always have one reader, groups filling four fifths of a tile in the mean or less, are marked streaming, so that the rows stay in L2, and every
// workgroup walks K from a place of its own.  Both pay where the workgroups fill the chip (counted as if the rows were spread evenly: the grid itself is an upper bound); a few of them wait
// longer for a line that is fetched again for its second half.  320 products of 4 .. 64 groups at 3 .. 63 rows a group, weights cold, time of plain loads over streaming:  528 .. 1024
// workgroups 1.04 .. 1.43, 240 .. 512 1.03 .. 1.39, 224 0.98 .. 1.25, 208 0.97, 192 1.03 .. 1.17 with K a multiple of 2048 (rows on the same channels) and 0.93 .. 1.05 without, fewer
// 0.69 .. 1.02 (704 x 6528 in 4 groups 46 us : 67, 576 x 6144 in 6 43 : 62).  32 rows x 4 of 16 experts: 5504 x 4096 gated 135 -> 120 us, 2816 x 2048 43 -> 33.5.
// Two slabs instead of four: past what four let reside (512 workgroups) up to all that two do (1024).  5504 x 4096 (688) 120 -> 110 us, 6.5 TB/s of weights; two / four of 320 .. 416
// workgroups 0.89 .. 0.95, of 528 .. 992 1.00 .. 1.23, of 1040 .. 1536 0.85 .. 0.96, from 1800 on level.
GroupGemmForm group_gemm_form(const GroupGemmArgs& a, int bm) {
    if (bm > 64) return GroupGemmForm{false, 0};
    const int nt = cdiv(a.N, 128), wgs = a.groups * cdiv(a.rows, a.plan.n_tiles ? a.groups * bm : bm) * nt;
    const bool lone = a.plan.n_tiles ? a.rows * 5 <= a.groups * bm * 4 : a.rows <= bm;
    const bool stream = lone && wgs >= (a.K % 2048 == 0 ? 192 : 224);
    return GroupGemmForm{stream, bm == 64 ? 3 : a.plan.n_tiles && stream && wgs > 512 && wgs <= 1024 ? 2 : 4};
}
void launch_group_gemm(int dtype, const GroupGemmArgs& a, int bm, hipStream_t st, int nb) {
    LMX_REQUIRE(a.X && a.W && a.C && a.rows >= 1 && a.groups >= 1 && a.N >= 1 && a.K >= 64 && a.K % 64 == 0 && a.per_row >= 1, "group_gemm: bad arguments");
    LMX_REQUIRE(a.ldx % 8 == 0 && a.ldw % 8 == 0 && a.ldc % 4 == 0 && a.w_group % 8 == 0 && a.x_group % 8 == 0 && a.c_group % 4 == 0 && a.N % 4 == 0, "group_gemm: 16-byte rows");
    LMX_REQUIRE(!act_gated(a.act) || a.N % 64 == 0, "group_gemm: gated rows come in groups of 64");
    // with a plan: every group's last tile may be part empty; no more tiles than rows
    const int m_tiles = a.plan.n_tiles ? std::min(a.rows, a.rows / bm + a.groups) : a.groups * cdiv(a.rows, bm);
    const GroupGemmForm f = group_gemm_form(a, bm);
    const bool stream = f.stream, two = f.slabs == 2;
#define L(TT) do { if (bm == 32 && two) launch_group_gemm_cfg<TT, 32, 128, 1, 2, 2, true>(a, m_tiles, st); \
                    else if (bm == 32) { if (stream) launch_group_gemm_cfg<TT, 32, 128, 1, 2, 4, true>(a, m_tiles, st); else launch_group_gemm_cfg<TT, 32, 128, 1, 2, 4, false>(a, m_tiles, st); } \
                    else if (bm == 64) { if (stream) launch_group_gemm_cfg<TT, 64, 128, 2, 2, 3, true>(a, m_tiles, st); else launch_group_gemm_cfg<TT, 64, 128, 2, 2, 3, false>(a, m_tiles, st); } \
                    else throw Error{"group_gemm: tiles of 32, 64 or 128 .. 256 rows"}; } while (0)
    if (bm > 64 && dtype != kF32) { launch_group_gemm4w(dtype, a, bm, nb, m_tiles, st); return; }
    if (dtype == kBF16) L(bf16_t); else if (dtype == kF16) L(f16_t); else throw Error{"group_gemm: 16-bit models"};
#undef L
}

// ---------------------------------------------------------------------------------------------------------------
// grid (slots, ceil(outputs / outputs per workgroup)), 256 threads.  `lpr` lanes own one weight row (a power of two with 8 lpr <= K): short rows leave no lane idle.
// Gated: a lane group takes the gate row and the up row of its output.
// ---------------------------------------------------------------------------------------------------------------
template <typename T, bool GATED, int U>
__device__ __forceinline__ void group_gemv_body(const GroupGemvArgs& a, int lpr, int opw, int slot, int part, char* smem) {
    T* xs = reinterpret_cast<T*>(smem);
    const int tid = threadIdx.x;
    const int grp = a.ids ? a.ids[slot] : slot % a.groups;
    const size_t xr = a.ids ? slot / a.per_row : slot / a.groups, cr = a.ids ? slot : slot / a.groups;
    const T* x = reinterpret_cast<const T*>(a.X) + xr * a.ldx + (a.ids ? 0 : grp * a.x_group);
    const T* W = reinterpret_cast<const T*>(a.W) + (size_t)grp * a.w_group;
    T* C = reinterpret_cast<T*>(a.C) + cr * a.ldc + (a.ids ? 0 : grp * a.c_group);
    const int outs = GATED ? a.N / 2 : a.N, sub = tid % lpr, per = 256 / lpr;
    const int o0 = part * opw, o1 = o0 + opw < outs ? o0 + opw : outs;
    // U pieces of a row (both rows, gated) are on their way together, the first ones ahead of the staging of x: piece by piece a row of 2048 was four memory latencies.  Pieces
    // past the row's end re-read its first one and count as zeros.  (us a launch, four slots: 2 x 1408 rows of 2048 12.2 -> 11.6, 2048 rows of 1408 8.1 -> 6.7)
    Chunk8<T> g[U], u[GATED ? U : 1];
    const int step = U * lpr * 8;
    for (int ob = o0; ob < o1; ob += per) {                  // every lane stays: the sums run over whole lane groups
        const int o = ob + tid / lpr, oc = o < o1 ? o : o1 - 1;
        const T* w0 = W + (size_t)(GATED ? 64 * (oc >> 5) + (oc & 31) : oc) * a.ldw;
        const T* w1 = w0 + (size_t)32 * a.ldw;
        float s0 = 0.f, s1 = 0.f;
        for (int cb = 0; cb < a.K; cb += step) {
#pragma unroll
            for (int k = 0; k < U; ++k) {
                int c = cb + sub * 8 + k * lpr * 8; c = c < a.K ? c : 0;
                g[k].load(w0 + c);
                if (GATED) u[k].load(w1 + c);
            }
            if (ob == o0 && cb == 0) {
                for (int c = tid * 8; c < a.K; c += 2048) { Chunk8<T> v; v.load(x + c); *reinterpret_cast<Chunk8<T>*>(xs + c) = v; }
                __syncthreads();
            }
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const int c = cb + sub * 8 + k * lpr * 8;
                const bool in = c < a.K;
                float v[8], f[8]; load8<T>(xs + (in ? c : 0), v); g[k].get(f);
#pragma unroll
                for (int i = 0; i < 8; ++i) s0 = in ? fmaf(f[i], v[i], s0) : s0;
                if (GATED) {
                    u[k].get(f);
#pragma unroll
                    for (int i = 0; i < 8; ++i) s1 = in ? fmaf(f[i], v[i], s1) : s1;
                }
            }
        }
        if (lpr == 64) { s0 = group_sum<64>(s0); if (GATED) s1 = group_sum<64>(s1); }
        else for (int d = lpr >> 1; d > 0; d >>= 1) { s0 += __shfl_xor(s0, d, 64); if (GATED) s1 += __shfl_xor(s1, d, 64); }
        if (sub == 0 && o < o1) C[o] = from_f32<T>(GATED ? gate_mul<T>(a.act, s0, s1) : s0);
    }
}
template <typename T, bool GATED, int U>
__global__ __launch_bounds__(256) void group_gemv_kernel(GroupGemvArgs a, int lpr, int opw) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    group_gemv_body<T, GATED, U>(a, lpr, opw, blockIdx.x, blockIdx.y, smem);
}

// The same beside a small linear that neither reads nor writes what it does (a parallel layer's output projection beside its experts): the linear's workgroups first
template <typename T, bool GATED, int U>
__global__ __launch_bounds__(256) void group_gemv_linear_kernel(GroupGemvArgs a, int lpr, int opw, int slots, GemvArgs g, int linear_wgs) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int b = (int)blockIdx.x - linear_wgs;
    if (b < 0) gemv2_body<T, 1, 2, 2, false>(g, blockIdx.x, smem, nullptr, 0u);
    else group_gemv_body<T, GATED, U>(a, lpr, opw, b % slots, b / slots, smem);
}

struct GroupGemvForm { int lpr, opw, parts, U; };
static GroupGemvForm group_gemv_form(const GroupGemvArgs& a, int slots) {
    int lpr = 64;
    while (lpr > 1 && lpr * 8 > a.K) lpr >>= 1;
    const int outs = act_gated(a.act) ? a.N / 2 : a.N, per = 256 / lpr;
    int opw = per;                                           // outputs of a workgroup: more of them while the grid stays large enough
    while (opw < 64 && (long)slots * cdiv(outs, opw * 2) >= 1024) opw *= 2;
    const int parts = cdiv(outs, opw);
    // pieces together: up to four, as many as leave the fewest past the end of a row of this length, and one by one where so many workgroups follow each other that their latencies do not
    // count.  us a launch one by one / four always / now, fp32 (16-bit models have few slots here): 16 rows x 16 heads of 512 columns 10.9 / 12.6 / 8.5 and of 128 8.2 / 13.8 / 8.3,
    // 32 rows x 32 heads 22 / 40 / 16.5 and 24 / 40 / 23, 128 slots x 4096 rows of 2752 576 / 618 / 599, 3600 slots x 2048 rows of 1408 1925 / 2128 / 1950 and x 2 x 1408 rows
    // of 2048 7934 / 8181 / 7916
    const int pieces = cdiv(a.K, lpr * 8);
    const int U = (long)slots * parts > 4096 ? 1 : pieces <= 4 ? pieces : cdiv(pieces, 3) * 3 < cdiv(pieces, 4) * 4 ? 3 : 4;
    return GroupGemvForm{lpr, opw, parts, U};
}
static void group_gemv_check(int dtype, const GroupGemvArgs& a) {
    LMX_REQUIRE(a.X && a.W && a.C && a.N >= 1 && a.K >= 64 && a.K % 8 == 0 && a.ldx % 8 == 0 && a.ldw % 8 == 0 && a.w_group % 8 == 0 && a.x_group % 8 == 0, "group_gemv: bad arguments");
    LMX_REQUIRE(!act_gated(a.act) || a.N % 64 == 0, "group_gemv: gated rows come in groups of 64");
    LMX_REQUIRE(a.per_row >= 1 && a.groups >= 1 && (size_t)a.K * dtype_size(dtype) <= 64 * 1024, "group_gemv: bad groups");
}
void launch_group_gemv(int dtype, const GroupGemvArgs& a, int slots, hipStream_t st) {
    group_gemv_check(dtype, a);
    if (slots <= 0) return;
    const GroupGemvForm f = group_gemv_form(a, slots);
    const dim3 grid(slots, f.parts);
#define L1(TT, G, UU) LMX_LAUNCH((group_gemv_kernel<TT, G, UU>), grid, dim3(256), (size_t)a.K * sizeof(TT), st, a, f.lpr, f.opw)
#define LU(TT, G) do { if (f.U == 4) L1(TT, G, 4); else if (f.U == 3) L1(TT, G, 3); else if (f.U == 2) L1(TT, G, 2); else L1(TT, G, 1); } while (0)
#define L(TT) do { if (act_gated(a.act)) LU(TT, true); else LU(TT, false); } while (0)
    if (dtype == kBF16) L(bf16_t); else if (dtype == kF16) L(f16_t); else L(float);
#undef L
#undef LU
#undef L1
    LMX_CHECK_HIP(hipGetLastError());
}

// Where the shared launch takes less than the two (us a layer of one token, two launches -> one):  rows of up to 3072  4 slots of 2 x 1408 x 2048 42.7 -> 39.8, 2 x 4096 x 2048 72.6 -> 68.7,
// 2 x 4096 x 3072 96.6 -> 94.0, 8 slots 149.2 -> 146.3.  Longer rows while a workgroup has few of them and there are more than four workgroups a CU (the linear's go first, and what follows
// in one even round ends as late as they began): 4 slots of 2 x 2752 x 4096 106.4 -> 104.4, 2 x 3328 x 4096 115.0 -> 111.6, 8 of 2 x 1408 103.5 -> 102.2, 2 of 2 x 5632 106.9 -> 104.6, but
// 4 of 2 x 4096 128.1 : 131.9, 2 x 8192 197.9 : 208.5, 2 of 2 x 4096 92.7 : 94.5, 8 of 2 x 2048 133.2 : 134.2; rows of 6144 .. 8192 99 .. 283 us, 0.9 % less to 5.6 % more.
bool group_gemv_joins(int dtype, const GroupGemvArgs& a, int slots, const GemvArgs& g) {
    if (g.K > 4096 || g.K % 8 != 0 || (size_t)g.N * g.K > ((size_t)1 << 25) || g.norm_w || !gemv2_applies(dtype, g)) return false;
    if (a.K <= 3072) return true;
    const GroupGemvForm f = group_gemv_form(a, slots);
    return a.K <= 4096 && (f.opw <= 4 || (f.opw <= 8 && slots * f.parts > 1024));
}
void launch_group_gemv_linear(int dtype, const GroupGemvArgs& a, int slots, const GemvArgs& g, hipStream_t st) {
    group_gemv_check(dtype, a);
    LMX_REQUIRE(slots >= 1 && act_gated(a.act) && !act_gated(g.act) && group_gemv_joins(dtype, a, slots, g), "group_gemv_linear: a gated grouped product and a small plain linear");
    const GroupGemvForm f = group_gemv_form(a, slots);
    const int linear_wgs = cdiv(g.N, 4);
    const dim3 grid(linear_wgs + slots * f.parts);
    const size_t smem = std::max((size_t)a.K * 2, gemv2_smem_bytes(g.K, 2));
#define L1(TT, UU) LMX_LAUNCH((group_gemv_linear_kernel<TT, true, UU>), grid, dim3(256), smem, st, a, f.lpr, f.opw, slots, g, linear_wgs)
#define L(TT) do { if (f.U == 4) L1(TT, 4); else if (f.U == 3) L1(TT, 3); else if (f.U == 2) L1(TT, 2); else L1(TT, 1); } while (0)
    if (dtype == kBF16) L(bf16_t); else L(f16_t);
#undef L
#undef L1
    LMX_CHECK_HIP(hipGetLastError());
}

}  // namespace lmx
