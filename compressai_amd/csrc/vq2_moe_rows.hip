// vq2_moe_rows.hip -- the MoE experts for many tokens: the pairs of one expert
// share each gathered centroid (gfx950 matrix cores).
//
//   gu    = VQ(gate_up[e]) . RHT_H(h_t)                       [2I]
//   act   = RHT_I(silu(gu[:I]) * gu[I:])                      [I]
//   out_t = sum_k w[t, k] * VQ(down[e]) . act                 [H]
//
// for the pairs (t, k), e = ids[t, k] (vq2/paged_runtime.py:495-510), from the
// reference-layout pools.  The one-pair kernels (vq2_sorted_moe.hip) gather an
// expert's codes once per pair, ~0.8 us each; a prompt's chunk of 512 tokens
// has 18 pairs an expert.  Here the pairs are grouped by expert and a
// workgroup multiplies up to 32 or 64 of them by 128 rows of the expert, so an
// expert's codes are gathered once per such tile: at least one per expert
// that has pairs, and ceil(T / tile) for one that every token names, as the
// shared expert.  Bound by those gathers: 393 K codes a tile at the ~240 G/s that
// the L2s serve, 0.45 ms for the 272 tiles of 512 tokens over 257 experts.
// Five launches:
//  1. moe_prep: workgroup 0 sorts the pairs by expert (a slot each) and cuts
//     them into tiles; the others rotate a token each and pack it.
//  2. moe_gemm, gate_up: gu[slot] = row sums * row scale, fp32.
//  3. moe_act: silu(gate) * up of a slot, rotated and packed.
//  4. moe_gemm, down: share[slot] = w * (row sums * row scale).
//  5. moe_rows_combine: out_t = the sum of its pairs' shares, in pair order.
// A pair whose expert id is outside the pool gives NaN.
//
// Precision: the one-pair kernels multiply fp32 activations by the centroids
// in fp32.  The matrix cores take 16-bit operands, so the activation is split
// into three addends of 8 bits each, which keep its 24 bits: bf16 with a bf16
// codebook, and with an fp16 codebook the same values as fp16 under a
// power-of-two scale per row (divided out exactly).  The centroids enter as
// they are; a stage's sums are added to the total in fp32 with the rounding
// error carried along.  Error against 64 bits (2-norm, 35B shape, 3 to 2048
// tokens): 1.9e-7 (bf16) and 2.1e-7 (fp16), the one-pair kernels 2.2e-7 to
// 2.4e-7.  Two fp16 addends of 11 bits took one product fewer but lost bits
// inside the instruction (2.6e-7), and one chain of instructions over all of K
// 7e-7.
//
// Measured (35B shape, us a layer, router included, one-pair kernels before):
// 73 tokens 510 -> 462, 128 tokens 883 -> 489, 512 tokens 3432 -> 574 (graph
// replays; bf16 codebook 561); at 512 tokens gate_up takes 0.35 ms, down 0.2
// (with all codes alike 0.17 and 0.12).
#include <algorithm>
#include <mutex>

#include "vq2_common.hpp"
#include "vq2_internal.hpp"
#include "vq2_rot_row.hpp"

namespace vq2 {

constexpr int MR_TILE_G = 32;   // groups per k tile, as in vq2_rows.hip
constexpr int MR_NS = 3;        // addends of an activation value
constexpr int MR_TS = 4;        // steps of a stage
// 16-byte units between staged rows in LDS; odd, so that the 16 rows of an
// operand start in 16 bank groups and every operand lies at a constant offset
// from the lane's first (a permutation of the units instead of the odd stride
// took an address register for each and spilled)
constexpr int MR_LROW = MR_TS * 4 * MR_NS + 1;
constexpr int MR_WAVES = 8;
constexpr int MR_THREADS = 64 * MR_WAVES;
constexpr int MR_COLS = 16 * MR_WAVES;  // expert rows of a workgroup
constexpr int MR_MAX_E = 4096;  // pool entries the sorting workgroup counts in LDS
constexpr int MR_PLAN_T = 256;  // its threads that scan the counts

struct MoeTile {
    int expert;
    int slot0;
    int count;
    int pad;
};

// ---------------------------------------------------------------- packing
// A row's 8 values of group g as NS operands of 8 16-bit addends, stored at
// unit ((kt * 8 + t) * NS + s) * 4 + q of the row (kt = g / 32, q = g / 8 % 4,
// t = g % 8: the k tile, k block and step of vq2_rows.hip), so that the
// operands of a few consecutive steps are contiguous.
template <int F16>
__device__ __forceinline__ void split_store(u32x4* row, int g, const float (&v)[8], int e)
{
    const int kt = g / MR_TILE_G, t = g & 7, q = (g >> 3) & 3;
    u32x4* u = row + (kt * 8 + t) * MR_NS * 4 + q;
    u32x4 o[MR_NS];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        float r = F16 ? ldexpf(v[k], e) : v[k];
        const bool fin = fabsf(r) < __builtin_inff();
#pragma unroll
        for (int s = 0; s < MR_NS; s++) {
            const uint32_t b = f32_to_bf16_bits(r);
            const uint32_t w = F16 ? f32_to_f16_bits(bf16_bits_to_f32(b)) : b;
            r = fin ? r - bf16_bits_to_f32(b) : 0.0f;
            if (k & 1) o[s][k >> 1] |= w << 16;
            else o[s][k >> 1] = w;
        }
    }
#pragma unroll
    for (int s = 0; s < MR_NS; s++) u[4 * s] = o[s];
}

struct MoePackArgs {
    const void* x;   // moe_prep: h [tokens, n]; moe_act: gu [slots, 2n] fp32
    int x_dt;
    int x_vec;
    int n;
    int kt;
    int hb_log2;
    const int32_t* perm;
    const int8_t* sign;
    float scale;
    u32x4* a;  // packed rows
    int* e;    // their exponents (F16)
};

struct MoePlanArgs {
    const void* ids;
    int ids_i64;
    int pairs;
    int P;
    int n_experts;
    int* slot_tok;    // [pairs] token of a slot
    int* slot_pair;   // [pairs]
    int* pair_slot;   // [pairs]; -1: id outside the pool
    MoeTile* tiles;
    int* n_tiles;
    int rows;         // pairs of a tile at most
};

// The rotated row's 8 values of this thread, packed (every thread of the
// workgroup calls it).  s_x holds the natural row.
template <int F16>
__device__ __forceinline__ void pack_row(const MoePackArgs& a, float* s_x, float* s_max, int64_t row,
                                         const int32_t (&pw)[8], const uint32_t (&sg)[2])
{
    const int T = (int)blockDim.x, tid = threadIdx.x;
    const bool g_ok = tid < a.n / 8;
    float v[8];
    rot_gather(s_x, pw, sg, a.n, g_ok, v);
    rot_transform(v, s_x, tid, T, a.hb_log2);
    float am = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        v[k] *= a.scale;
        am = fmaxf(am, fabsf(v[k]));
    }
    int e = 0;
    if constexpr (F16) {
        e = rot_row_exponent(am, s_max, tid, T);
        if (tid == 0) a.e[row] = e;
    }
    if (tid / MR_TILE_G < a.kt) split_store<F16>(a.a + row * a.kt * (32 * MR_NS), tid, v, e);
}

__device__ __forceinline__ int64_t moe_pair_id(const MoePlanArgs& p, int i)
{
    return p.ids_i64 ? ((const int64_t*)p.ids)[i] : (int64_t)((const int32_t*)p.ids)[i];
}

// Pairs by expert: counts, their prefix sums, a slot per pair, the tiles.
// The order of one expert's pairs is that of the atomics: every result
// depends on its own pair's row alone.
__device__ void moe_plan(const MoePlanArgs& p, int* s_cnt)
{
    __shared__ int s_sum[2][MR_PLAN_T];
    const int T = (int)blockDim.x, tid = threadIdx.x, E = p.n_experts;
    for (int i = tid; i < E; i += T) s_cnt[i] = 0;
    __syncthreads();
    // ids in batches, so that their loads are in flight together; one batch
    // (up to 5120 pairs with 256 threads) stays in registers for both passes
    // (one load at a time the two passes over 4608 pairs took ~12 us)
    constexpr int NB = 20;
    int e[NB];
    auto load_ids = [&](int i0) {
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const int64_t id = moe_pair_id(p, min(i0 + j * T, p.pairs - 1));
            e[j] = i0 + j * T < p.pairs && id >= 0 && id < E ? (int)id : -1;
        }
    };
    for (int i0 = tid; i0 - tid < p.pairs; i0 += NB * T) {
        load_ids(i0);
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (e[j] >= 0) atomicAdd(&s_cnt[e[j]], 1);
    }
    __syncthreads();
    // thread t scans the experts [t * per, t * per + per)
    const int per = (E + MR_PLAN_T - 1) / MR_PLAN_T;
    int c = 0, n = 0;
    if (tid < MR_PLAN_T) {
        for (int e = tid * per; e < min(E, (tid + 1) * per); e++) {
            c += s_cnt[e];
            n += (s_cnt[e] + p.rows - 1) / p.rows;
        }
        s_sum[0][tid] = c;
        s_sum[1][tid] = n;
    }
    __syncthreads();
    for (int d = 1; d < MR_PLAN_T; d <<= 1) {
        int a0 = 0, a1 = 0;
        if (tid < MR_PLAN_T && tid >= d) { a0 = s_sum[0][tid - d]; a1 = s_sum[1][tid - d]; }
        __syncthreads();
        if (tid < MR_PLAN_T) { s_sum[0][tid] += a0; s_sum[1][tid] += a1; }
        __syncthreads();
    }
    if (tid < MR_PLAN_T) {
        int slot = s_sum[0][tid] - c, tile = s_sum[1][tid] - n;
        for (int e = tid * per; e < min(E, (tid + 1) * per); e++) {
            const int cnt = s_cnt[e];
            s_cnt[e] = slot;  // the next slot of this expert
            for (int o = 0; o < cnt; o += p.rows) p.tiles[tile++] = MoeTile{e, slot + o, min(p.rows, cnt - o), 0};
            slot += cnt;
        }
        if (tid == MR_PLAN_T - 1) *p.n_tiles = s_sum[1][tid];
    }
    __syncthreads();
    for (int i0 = tid; i0 - tid < p.pairs; i0 += NB * T) {
        if (p.pairs > NB * T) load_ids(i0);
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const int i = i0 + j * T;
            if (i >= p.pairs) break;
            int slot = -1;
            if (e[j] >= 0) {
                slot = atomicAdd(&s_cnt[e[j]], 1);
                p.slot_tok[slot] = i / p.P;
                p.slot_pair[slot] = i;
            }
            p.pair_slot[i] = slot;
        }
    }
}

template <int F16>
__global__ void __launch_bounds__(ROT_ROW_MAX_T) moe_prep_kernel(const MoePackArgs a, const MoePlanArgs p)
{
    extern __shared__ __align__(16) float s_x[];
    __shared__ float s_max[ROT_ROW_MAX_T / 64];
    if (blockIdx.x == 0) {
        moe_plan(p, (int*)s_x);
        return;
    }
    const int64_t row = blockIdx.x - 1;
    const int T = (int)blockDim.x, tid = threadIdx.x;
    int32_t pw[8];
    uint32_t sg[2];
    rot_tables(a.perm, a.sign, tid < a.n / 8 ? tid : 0, pw, sg);
    rot_stage_row(a.x, a.x_dt, a.x_vec, row * a.n, a.n, s_x, tid, T);
    __syncthreads();
    pack_row<F16>(a, s_x, s_max, row, pw, sg);
}

template <int F16>
__global__ void __launch_bounds__(ROT_ROW_MAX_T) moe_act_kernel(const MoePackArgs a)
{
    extern __shared__ __align__(16) float s_x[];
    __shared__ float s_max[ROT_ROW_MAX_T / 64];
    const int64_t row = blockIdx.x;
    const int T = (int)blockDim.x, tid = threadIdx.x;
    int32_t pw[8];
    uint32_t sg[2];
    rot_tables(a.perm, a.sign, tid < a.n / 8 ? tid : 0, pw, sg);
    const float* gu = (const float*)a.x + row * 2 * a.n;
    for (int c = tid; c < a.n / 4; c += T) {
        const f32x4_t g = *((const f32x4_t*)gu + c), u = *((const f32x4_t*)(gu + a.n) + c);
        f32x4_t s;
#pragma unroll
        for (int k = 0; k < 4; k++) s[k] = g[k] / (1.0f + expf(-g[k])) * u[k];
        *((f32x4_t*)s_x + c) = s;
    }
    __syncthreads();
    pack_row<F16>(a, s_x, s_max, row, pw, sg);
}

// ------------------------------------------------------------- the product
struct MoeGemmArgs {
    const u32x4* a;      // packed rows
    const int* e;        // their exponents (F16)
    const int* row_of;   // packed row of a slot (null: the slot)
    const MoeTile* tiles;
    const int* n_tiles;
    const int16_t* idx;  // pool [n_experts, rows, ng]
    const u32x4* cb;     // fp16 (F16) or bf16 codebook
    const void* scale;   // [n_experts, rows]
    int s_dt;
    int rows;
    int ng;
    int kt;
    int col_blocks;      // MR_COLS-row blocks of an expert
    const float* w;      // combine weight of a pair (null: 1)
    const int* slot_pair;
    float* y;            // [slots][rows]
};

// Workgroup: one tile of up to 16 MT pairs x 128 rows of its expert, a wave 16
// rows.  Per stage (MR_TS steps of a k tile) the waves gather their own
// operands into registers, one stage ahead, and stage the pairs' packed
// operands in LDS for all of them (two buffers, one barrier a stage): fetched
// by each wave for itself they would double the L2 requests the gathers wait
// for.  Two workgroups a CU at MT = 2 (126 VGPRs); held to three (80 VGPRs) it
// spills and takes twice the time, with 2 steps a stage 5 % longer.  A tile
// multiplies all its 16 MT rows: a branch per 16 rows made the compiler
// specialise the loop and spill.
template <int F16, int MT>
__global__ void __launch_bounds__(MR_THREADS, MT == 2 ? 4 : 2) moe_gemm_kernel(const MoeGemmArgs a)
{
    constexpr int NS = MR_NS, TS = MR_TS, ROWS = 16 * MT;
    constexpr int HS = 8 / TS;             // stages of a k tile
    constexpr int UR = TS * 4 * NS;        // 16-byte units of a row and stage
    constexpr int LR = MR_LROW;
    constexpr int NL = ROWS * UR / MR_THREADS;  // staging loads of a thread
    static_assert(HS % 2 == 0 && NL * MR_THREADS == ROWS * UR, "two buffers in turn, whole rounds of staging loads");
    extern __shared__ __align__(16) u32x4 s_dyn[];
    u32x4 (*s_a)[ROWS * LR] = (u32x4 (*)[ROWS * LR])s_dyn;
    const int tile_i = (int)blockIdx.x / a.col_blocks, cb0 = (int)blockIdx.x % a.col_blocks;
    if (tile_i >= *a.n_tiles) return;
    const MoeTile tile = a.tiles[tile_i];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 15, q = lane >> 4;
    const int col = cb0 * MR_COLS + wave * 16 + nl;
    const bool col_ok = col < a.rows;
    const int nmt = (tile.count + 15) / 16;
    const int64_t colr = (int64_t)tile.expert * a.rows + (col_ok ? col : 0);
    const int16_t* ix = a.idx + colr * a.ng;
    const u32x4 zero = {0, 0, 0, 0};

    auto load_idx = [&](int kt) {
        const int g = min(kt, a.kt - 1) * MR_TILE_G + q * 8;
        return __builtin_nontemporal_load((const u32x4*)(ix + (g < a.ng ? g : 0)));
    };
    u32x4 w0 = load_idx(0), w1 = load_idx(1);

    // this thread's units of the staged operands: row u / UR, unit u % UR
    const u32x4* src[NL];
    int dst[NL];
    bool st[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int u = tid + i * MR_THREADS, r = u / UR, c = u % UR;
        st[i] = r < nmt * 16;
        const int slot = tile.slot0 + min(r, tile.count - 1);
        const int64_t ar = a.row_of ? a.row_of[slot] : slot;
        src[i] = a.a + ar * a.kt * (32 * NS) + c;
        dst[i] = r * LR + c;
    }
    u32x4 sa[NL];
    auto load_a = [&](int step) {
#pragma unroll
        for (int i = 0; i < NL; i++)
            if (st[i]) sa[i] = src[i][(int64_t)step * UR];
    };
    auto code = [](const u32x4& w, int t) { return (w[t >> 1] >> (16 * (t & 1))) & 0xFFFFu; };

    f32x4_t acc[MT], err[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i] = err[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    u32x4 b[TS], bn[TS];
    load_a(0);
#pragma unroll
    for (int j = 0; j < TS; j++) b[j] = a.cb[code(w0, j)];

    for (int kt = 0; kt < a.kt; kt++) {
        const bool g_ok = kt * MR_TILE_G + q * 8 < a.ng;  // a short last k tile lacks whole k blocks
#pragma unroll
        for (int h = 0; h < HS; h++) {
            const int step = kt * HS + h;
#pragma unroll
            for (int i = 0; i < NL; i++)
                if (st[i]) s_a[h & 1][dst[i]] = sa[i];
            __syncthreads();
            const bool more = h + 1 < HS || kt + 1 < a.kt;
            if (more) {
                load_a(step + 1);
#pragma unroll
                for (int j = 0; j < TS; j++)
                    bn[j] = a.cb[h + 1 < HS ? code(w0, (h + 1) * TS + j) : code(w1, j)];
            }
            if (h + 1 == HS) {
                w0 = w1;
                w1 = load_idx(kt + 2);
            }
            // a stage's products in two short chains, the leading addends and
            // the small ones, added to the sums in fp32: in one chain over all
            // of K the error against 64 bits was three times as large
#pragma unroll
            for (int j = 0; j < TS; j++) b[j] = g_ok ? b[j] : zero;
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const int r = i * 16 + nl;
                f32x4_t big = {0.0f, 0.0f, 0.0f, 0.0f}, small = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < TS; j++) {
#pragma unroll
                    for (int s = 0; s < NS; s++) {
                        const u32x4 x = s_a[h & 1][r * LR + (j * NS + s) * 4 + q];
                        if (s == 0) big = mfma_16<F16>(x, b[j], big);
                        else small = mfma_16<F16>(x, b[j], small);
                    }
                }
                // acc + err: the exact sum of acc and big (two-sum)
                const f32x4_t sum = acc[i] + big, bv = sum - acc[i];
                err[i] += ((acc[i] - (sum - bv)) + (big - bv)) + small;
                acc[i] = sum;
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < TS; j++) b[j] = bn[j];
        }
    }

    // D[i][j]: pair 4 (l / 16) + e of the 16, expert row l % 16
    if (!col_ok) return;
    const float s = load_as_f32(a.scale, a.s_dt, colr);
#pragma unroll
    for (int i = 0; i < MT; i++) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int r = i * 16 + q * 4 + e;
            if (r >= tile.count) continue;
            const int slot = tile.slot0 + r;
            // (an infinite sum stays one: its two-sum error is NaN)
            float v = acc[i][e];
            if (fabsf(v) < __builtin_inff()) v += err[i][e];
            if constexpr (F16) v = ldexpf(v, -a.e[a.row_of ? a.row_of[slot] : slot]);
            v *= s;
            if (a.w) v *= a.w[a.slot_pair[slot]];
            a.y[(int64_t)slot * a.rows + col] = v;
        }
    }
}

// out[t][4c .. 4c + 3] = the token's shares in pair order
__global__ void __launch_bounds__(256) moe_rows_combine_kernel(const float* share, const int* pair_slot, int P, int H,
                                                               void* out, int out_dt)
{
    const int t = blockIdx.y, c = (int)blockIdx.x * 256 + threadIdx.x;
    if (c * 4 >= H) return;
    f32x4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int NB = 12;  // pairs whose loads are in flight together
    for (int k0 = 0; k0 < P; k0 += NB) {
        f32x4_t v[NB];
        int slot[NB];
#pragma unroll
        for (int k = 0; k < NB; k++) slot[k] = pair_slot[(int64_t)t * P + min(k0 + k, P - 1)];
#pragma unroll
        for (int k = 0; k < NB; k++) v[k] = *((const f32x4_t*)(share + (int64_t)max(slot[k], 0) * H) + c);
#pragma unroll
        for (int k = 0; k < NB; k++) {
            if (k0 + k >= P) continue;
            const float bad = __builtin_nanf("");
            sum += slot[k] >= 0 ? v[k] : f32x4_t{bad, bad, bad, bad};
        }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) store_from_f32(out, out_dt, (int64_t)t * H + c * 4 + k, sum[k]);
}

// ------------------------------------------------------------------ launch
struct MoeRowsPlan {
    int kt_h, kt_i;
    int mt;  // 16-row tiles of a workgroup's pairs
    int64_t pairs, max_tiles;
    size_t slot_tok, slot_pair, pair_slot, tiles, n_tiles, e_h, e_i, a_h, a_i, gu, share, total;
};

static MoeRowsPlan moe_rows_plan(const MoeRowsCall& c)
{
    MoeRowsPlan p{};
    p.kt_h = (int)((c.hidden / 8 + MR_TILE_G - 1) / MR_TILE_G);
    p.kt_i = (int)((c.inter / 8 + MR_TILE_G - 1) / MR_TILE_G);
    p.pairs = c.tokens * c.P;
    // every expert may end with a short tile
    // 64 pairs a tile from 28 an expert on (35B shape, us a layer at 32 / 64
    // pairs when the line was set, before the router and the sorting took 20
    // us less: 512 tokens, 18 an expert 610 / 777; 1024 tokens 939 / 846; 2048
    // tokens 1533 / 1333)
    p.mt = p.pairs >= 28 * c.n_experts ? 4 : 2;
    p.max_tiles = p.pairs / (16 * p.mt) + std::min<int64_t>(p.pairs, c.n_experts);
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o += (bytes + 255) / 256 * 256;
        return at;
    };
    p.slot_tok = take(p.pairs * sizeof(int));
    p.slot_pair = take(p.pairs * sizeof(int));
    p.pair_slot = take(p.pairs * sizeof(int));
    p.tiles = take(p.max_tiles * sizeof(MoeTile));
    p.n_tiles = take(sizeof(int));
    p.e_h = take(c.tokens * sizeof(int));
    p.e_i = take(p.pairs * sizeof(int));
    p.a_h = take((size_t)c.tokens * p.kt_h * 32 * MR_NS * sizeof(u32x4));
    p.a_i = take((size_t)p.pairs * p.kt_i * 32 * MR_NS * sizeof(u32x4));
    p.gu = take((size_t)p.pairs * 2 * c.inter * sizeof(float));
    p.share = take((size_t)p.pairs * c.hidden * sizeof(float));
    p.total = o;
    return p;
}

static int moe_rows_check(const MoeRowsCall& c)
{
    if (c.tokens < 1 || c.P < 1) return set_error(VQ2_ERR_ARG, "vq2_moe_rows: tokens and pairs per token must be >= 1");
    if (c.hidden % 64 || c.inter % 64 || c.hidden < 64 || c.inter < 64 || c.hidden > 8 * ROT_ROW_MAX_T ||
        c.inter > 8 * ROT_ROW_MAX_T)
        return set_error(VQ2_ERR_UNSUPPORTED, "vq2_moe_rows: hidden=%lld / inter=%lld must be multiples of 64 up to %d",
                         (long long)c.hidden, (long long)c.inter, 8 * ROT_ROW_MAX_T);
    if (c.cb_dt != VQ2_DT_F16 && c.cb_dt != VQ2_DT_BF16)
        return set_error(VQ2_ERR_UNSUPPORTED, "vq2_moe_rows: fp16 / bf16 codebooks only");
    if (c.tokens > 1 << 20 || c.tokens * c.P > 1 << 20)
        return set_error(VQ2_ERR_UNSUPPORTED, "vq2_moe_rows: too many pairs");
    if (c.n_experts < 1 || c.n_experts > MR_MAX_E)
        return set_error(VQ2_ERR_UNSUPPORTED, "vq2_moe_rows: %lld pool entries outside 1..%d", (long long)c.n_experts,
                         MR_MAX_E);
    return VQ2_OK;
}

size_t moe_rows_workspace_bytes(const MoeRowsCall& c)
{
    return moe_rows_check(c) == VQ2_OK ? moe_rows_plan(c).total : 0;
}

template <int F16, int MT>
static hipError_t launch_gemm_t(const MoeGemmArgs& g, const MoeRowsPlan& p, hipStream_t st)
{
    // opt in to more than 64 KiB of dynamic LDS, once per instantiation
    constexpr int SHM = 2 * 16 * MT * MR_LROW * (int)sizeof(u32x4);
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    std::call_once(once, [] {
        attr = hipFuncSetAttribute((const void*)moe_gemm_kernel<F16, MT>, hipFuncAttributeMaxDynamicSharedMemorySize, SHM);
    });
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL((moe_gemm_kernel<F16, MT>), dim3((unsigned)(p.max_tiles * g.col_blocks)), dim3(MR_THREADS), SHM, st,
                       g);
    return hipGetLastError();
}

template <int F16>
static hipError_t launch_gemm(const MoeGemmArgs& g, const MoeRowsPlan& p, hipStream_t st)
{
    return p.mt == 2 ? launch_gemm_t<F16, 2>(g, p, st) : launch_gemm_t<F16, 4>(g, p, st);
}

template <int F16>
static hipError_t moe_rows_launches(const MoeRowsCall& c, const MoeRowsPlan& p, int hl_h, int hl_i)
{
    char* ws = (char*)c.workspace;
    hipStream_t st = (hipStream_t)c.stream;
    const int T_h = std::max(MR_PLAN_T, (p.kt_h * MR_TILE_G + 63) / 64 * 64), T_i = std::max(64, (p.kt_i * MR_TILE_G + 63) / 64 * 64);

    MoePlanArgs pl{c.ids, c.ids_i64, (int)p.pairs, c.P, (int)c.n_experts, (int*)(ws + p.slot_tok),
                   (int*)(ws + p.slot_pair), (int*)(ws + p.pair_slot), (MoeTile*)(ws + p.tiles), (int*)(ws + p.n_tiles), 16 * p.mt};
    MoePackArgs k{};
    k.x = c.h;
    k.x_dt = c.h_dt;
    k.x_vec = (uintptr_t)c.h % 16 == 0;
    k.n = (int)c.hidden;
    k.kt = p.kt_h;
    k.hb_log2 = hl_h;
    k.perm = c.rot_h.perm;
    k.sign = c.rot_h.sign;
    k.scale = c.rot_h.scale;
    k.a = (u32x4*)(ws + p.a_h);
    k.e = (int*)(ws + p.e_h);
    const size_t shm_h = std::max((size_t)T_h * 8 * sizeof(float), (size_t)c.n_experts * sizeof(int));
    hipLaunchKernelGGL(moe_prep_kernel<F16>, dim3((unsigned)(c.tokens + 1)), dim3(T_h), shm_h, st, k, pl);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;

    MoeGemmArgs g{};
    g.a = k.a;
    g.e = k.e;
    g.row_of = pl.slot_tok;
    g.tiles = pl.tiles;
    g.n_tiles = pl.n_tiles;
    g.idx = c.gu_idx;
    g.cb = (const u32x4*)c.cb;
    g.scale = c.gu_scale;
    g.s_dt = c.gu_s_dt;
    g.rows = (int)(2 * c.inter);
    g.ng = (int)(c.hidden / 8);
    g.kt = p.kt_h;
    g.col_blocks = (int)((2 * c.inter + MR_COLS - 1) / MR_COLS);
    g.y = (float*)(ws + p.gu);
    if ((err = launch_gemm<F16>(g, p, st)) != hipSuccess) return err;

    k.x = g.y;
    k.n = (int)c.inter;
    k.kt = p.kt_i;
    k.hb_log2 = hl_i;
    k.perm = c.rot_i.perm;
    k.sign = c.rot_i.sign;
    k.scale = c.rot_i.scale;
    k.a = (u32x4*)(ws + p.a_i);
    k.e = (int*)(ws + p.e_i);
    hipLaunchKernelGGL(moe_act_kernel<F16>, dim3((unsigned)p.pairs), dim3(T_i), (size_t)T_i * 8 * sizeof(float), st, k);
    if ((err = hipGetLastError()) != hipSuccess) return err;

    g.a = k.a;
    g.e = k.e;
    g.row_of = nullptr;
    g.idx = c.dn_idx;
    g.scale = c.dn_scale;
    g.s_dt = c.dn_s_dt;
    g.rows = (int)c.hidden;
    g.ng = (int)(c.inter / 8);
    g.kt = p.kt_i;
    g.col_blocks = (int)((c.hidden + MR_COLS - 1) / MR_COLS);
    g.w = c.w;
    g.slot_pair = pl.slot_pair;
    g.y = (float*)(ws + p.share);
    if ((err = launch_gemm<F16>(g, p, st)) != hipSuccess) return err;

    hipLaunchKernelGGL(moe_rows_combine_kernel, dim3((unsigned)((c.hidden / 4 + 255) / 256), (unsigned)c.tokens), dim3(256), 0,
                       st, g.y, pl.pair_slot, c.P, (int)c.hidden, c.out, c.out_dt);
    return hipGetLastError();
}

int moe_rows_launch(const MoeRowsCall& c)
{
    if (int r = moe_rows_check(c)) return r;
    if (c.tokens > 65535) return set_error(VQ2_ERR_UNSUPPORTED, "vq2_moe_rows: more than 65535 tokens");
    auto log2_of = [](int64_t hb, int64_t n) {
        int l = 0;
        while ((int64_t(1) << l) < hb) l++;
        return hb >= 64 && (int64_t(1) << l) == hb && n % hb == 0 ? l : -1;
    };
    const int hl_h = log2_of(c.rot_h.hb, c.hidden), hl_i = log2_of(c.rot_i.hb, c.inter);
    if (hl_h < 0 || hl_i < 0)
        return set_error(VQ2_ERR_ARG, "vq2_moe_rows: rotation blocks must be powers of two of at least 64 dividing the widths");
    if (((uintptr_t)c.rot_h.perm | (uintptr_t)c.rot_i.perm) % 16 || ((uintptr_t)c.rot_h.sign | (uintptr_t)c.rot_i.sign) % 8)
        return set_error(VQ2_ERR_ARG, "vq2_moe_rows: perm 16-byte, sign 8-byte aligned");
    if (((uintptr_t)c.gu_idx | (uintptr_t)c.dn_idx) % 16 || (uintptr_t)c.cb % 16)
        return set_error(VQ2_ERR_UNSUPPORTED, "vq2_moe_rows: pools and codebook must be 16-byte aligned");
    const MoeRowsPlan p = moe_rows_plan(c);
    if (p.max_tiles * ((std::max(2 * c.inter, c.hidden) + MR_COLS - 1) / MR_COLS) > 0x7FFFFFFF)
        return set_error(VQ2_ERR_UNSUPPORTED, "vq2_moe_rows: grid too large");
    if (!c.workspace || c.ws_bytes < p.total || (uintptr_t)c.workspace % 256)
        return set_error(VQ2_ERR_ARG, "vq2_moe_rows: workspace of %zu bytes (256-byte aligned) needed, got %zu", p.total,
                         c.ws_bytes);
    const hipError_t err = c.cb_dt == VQ2_DT_F16 ? moe_rows_launches<1>(c, p, hl_h, hl_i) : moe_rows_launches<0>(c, p, hl_h, hl_i);
    if (err != hipSuccess) return set_hip_error(err, "vq2_moe_rows launch");
    return VQ2_OK;
}

}  // namespace vq2
