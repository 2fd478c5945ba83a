// vq2_rows.hip -- several activation rows times up to 4 VQ matrices on the
// gfx950 matrix cores, the rotation included.
//
//   y_s[m, r] = (sum_k RHT(x)[m, k] * W_s[r, k]) * scale_s[r] * rs,
//   W[r, 8g + j] = cb0[i0[r, g]][j] (+ cb1[i1[r, g]][j]).
//
// Two or three launches for any number of rows:
//  1. rows_pack_kernel: one workgroup per activation row rotates it (or takes
//     it rotated), finds the row's power-of-two scale and writes it as fp16
//     in the order the second launch's matrix instructions read (below).
//     Up to RW_BF_ROWS rows a bf16 codebook is multiplied as it is, in bf16:
//     each fp16 value of a row goes in as two bf16 addends, which hold its 11
//     bits exactly, in two packed rows whose sums the product adds.
//  2. rows_gemm_kernel, or for many rows rows_wide_kernel (and rows_sum_kernel
//     where its k tiles are shared): the product.  rows_gemm_kernel rounds
//     codebooks that are not fp16 to fp16 as it gathers them.  For
//     rows_wide_kernel, and fp32 ones of many gathers (RW_F32_GATHERS),
//     further workgroups of the first launch round them, once per call.
//
// Why two launches and this layout.  The products are bound by the random
// 16-byte centroid gathers, which the L2s serve at ~240 G/s whatever else the
// chip does (bench_gather.hip), so a code must be gathered as few times as
// possible, by a kernel with nothing else on its way.  A workgroup that
// stages and converts its own activation (vq2_gemm_mfma.hip) does so once
// per 64 output rows and K split and needs a third launch for the splits'
// sum; here the activation is converted once, a wave reads its operand
// fragments as whole 1 KiB lines straight into registers, and the K split
// lies inside the workgroup (waves take k tiles in turn and their sums meet
// in LDS), so nothing is written but y.  Measured, us a call, rotation
// included (before: vq2_rht, vq2_gemm_small_m per 64 rows and its reduce
// launch): 2048 x 6144 at 4 bpw, 16 rows 34.0 -> 25.7; two 6144 x 2048 at
// 3 bpw, 64 rows, bf16 75.2 -> 30.1; 2999 x 4096 at 2 bpw, 100 rows 52.0 ->
// 33.2; two 6144 x 2048 at 4 bpw, 1024 rows 979 -> 173.  In graph replays,
// without the launches' host time (fp16 codebooks): 2048 x 6144 at 4 bpw, 3 /
// 16 / 64 rows 25.3 / 26.7 / 36.3 -> 24.5 / 25.2 / 30.4; 6144 x 2048 24.2 /
// 25.9 / 35.8 -> 22.4 / 22.8 / 27.2; 2048 x 2048 at 2 bpw, 16 rows 14.0 ->
// 10.9.  Left behind them: 17 rows of 6144 x 6144 and 6144 x 4096 at 4 bpw (60.1
// / 42.3 -> 62.3 / 43.3), 3 rows of the former (57.7 -> 58.4).  Bound by the gathers (13 us
// of a 6144 x 2048 call at 4 bpw) and, below about a million codes, by the
// two launches' latency (~12 us).
//
// Fragment layout: v_mfma_f32_16x16x32_f16 takes 8 consecutive k of row
// l % 16 from lane l, k block l / 16.  A k tile is 32 groups (256 k); its
// step t (0..7) multiplies the groups 8q + t, q = 0..3, so that a lane's 8
// codes of one matrix row and k tile are one 16-byte index load and step t's
// gather is that lane's B operand as it arrives.  The packed activation holds,
// for 16-row tile mt, k tile kt and step t, the 64 lanes' 16-byte operands in
// lane order: chunk (((mt * KT + kt) * 8 + t) * 64 + q * 16 + row % 16).
//
// Precision: as vq2_gemm_mfma.hip: the rotation in fp32, one rounding to fp16
// under a power-of-two scale per row (divided out of the fp32 sum exactly),
// fp16 centroids as they are, fp32 accumulation.  Up to RW_BF_ROWS rows bf16
// centroids as they are too, as in the sorted batch kernel; above, rounded to
// fp16 as in vq2_gemm_mfma.hip.
//
// Semantics: the PackedLinear fallback for batch > 1, rotate, dequantize,
// F.linear (vq2/runtime.py:82-89, 105-110), for (16,), (16,8) and (16,16).
#include <algorithm>
#include <mutex>

#include "vq2_common.hpp"
#include "vq2_internal.hpp"
#include "vq2_rot_row.hpp"

namespace vq2 {

constexpr int RW_TILE_G = 32;      // groups per k tile
constexpr int RW_PACK_MAX = ROT_ROW_MAX_T;
constexpr int64_t RW_MAX_N = 8 * RW_PACK_MAX;
constexpr int RW_CB_ROWS = 65536;
// bf16 codebooks: up to this many rows are packed as two bf16 addends each,
// which fit one 16-row tile, so the centroids need no rounding.  More rows
// round them as gathered: rounding the codebooks first, in every call, cost up
// to 4 us of it.  Graph replays, us a call, first / now (vq2_rht and
// vq2_gemm_small_m before): 8 rows 6144 x 2048 at 4 bpw 25.5 / 22.8 (25.2),
// 2048 x 6144 27.6 / 25.6 (26.3), 512 x 6144 19.9 / 16.2 (16.6); 17 rows 512 x
// 2048 at 4 bpw 18.2 / 15.0 (15.4), 64 rows 6144 x 2048 at 3 bpw 22.0 / 21.1
// (31.7).  Left behind the launches before: 9 to 17 rows of 512 x 6144 (9 rows
// 17.5 / 17.1) and of 6144 x 4096 (43.1 / 41.4) at 4 bpw.
constexpr int64_t RW_BF_ROWS = 8;
static_assert(RW_BF_ROWS <= 8, "both addends of every row in one row tile");

// fp32 codebooks: with one 16-bit stage and up to this many gathers they are
// rounded as gathered, 32 bytes a code, else once per call by the packing
// launch.  Graph replays, us a call, once per call / as gathered: 512 x 2048
// at 2 bpw, 8 rows 13.8 / 12.1, 1024 x 2048 13.7 / 11.9; 17 rows 2048 x 6144
// (1.5 M codes) 21.1 / 21.8; with two 16-bit stages 512 x 2048 15.5 / 16.8,
// 6144 x 2048 24.6 / 31.2.
constexpr int64_t RW_F32_GATHERS = 1 << 20;

// ------------------------------------------------------------- the packing
struct RowsPackArgs {
    const void* x;
    int x_dt;
    int x_vec;  // rows are 16-byte aligned
    int64_t x_stride;
    int64_t m;
    int n;
    int kt;       // k tiles
    int hb_log2;  // 0: x is rotated
    const int32_t* perm;
    const int8_t* sign;
    float scale;
    int act_dt;  // type the rotated activation is rounded to first
    half8_t* a;  // packed activation
    int* e;      // exponent of each row's scale
    uint32_t* cnt;  // arrival counters of the product, to be cleared
    int n_cnt;
    // codebooks to round to fp16 (null: none)
    const void* cb0;
    const void* cb1;
    int cb_dt;
    int cb1_rows;
    half8_t* h0;
    half8_t* h1;
};

__device__ __forceinline__ float rows_round_act(float v, int dt)
{
    if (dt == VQ2_DT_F16) return (float)(_Float16)v;
    if (dt == VQ2_DT_BF16) return bf16_bits_to_f32(f32_to_bf16_bits(v));
    return v;
}

__device__ __forceinline__ half8_t rows_bf16_to_half(u32x4 u)
{
    half8_t h;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        h[2 * k] = (_Float16)__uint_as_float(u[k] << 16);
        h[2 * k + 1] = (_Float16)__uint_as_float(u[k] & 0xFFFF0000u);
    }
    return h;
}

__device__ __forceinline__ half8_t rows_f32_to_half(u32x4 lo, u32x4 hi)
{
    half8_t h;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        h[k] = (_Float16)__uint_as_float(lo[k]);
        h[4 + k] = (_Float16)__uint_as_float(hi[k]);
    }
    return h;
}

// Centroid i of cb0, then cb1, rounded to fp16.
__device__ __forceinline__ void rows_cvt_codebook(const RowsPackArgs& a, int64_t i)
{
    const void* src = a.cb0;
    half8_t* dst = a.h0;
    if (i >= RW_CB_ROWS) {
        i -= RW_CB_ROWS;
        src = a.cb1;
        dst = a.h1;
        if (i >= a.cb1_rows) return;
    }
    const half8_t h = a.cb_dt == VQ2_DT_BF16 ? rows_bf16_to_half(*((const u32x4*)src + i))
                                             : rows_f32_to_half(*((const u32x4*)src + 2 * i), *((const u32x4*)src + 2 * i + 1));
    dst[i] = h;
}

// Workgroup b < m: row b, one thread per group (vq2_rot_row.hpp).  BF: two
// bf16 addends a value, the second in row 8 + b of the one tile.
template <int BF>
__global__ void __launch_bounds__(RW_PACK_MAX) rows_pack_kernel(const RowsPackArgs a)
{
    extern __shared__ __align__(16) float s_x[];  // the row; later the exchanges
    __shared__ float s_max[RW_PACK_MAX / 64];
    const int T = (int)blockDim.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row = blockIdx.x;
    if (row >= a.m) {
        rows_cvt_codebook(a, (row - a.m) * T + tid);
        return;
    }
    // the product's arrival counters
    if (row == 0)
        for (int i = tid; i < a.n_cnt; i += T) a.cnt[i] = 0u;
    const int ng = a.n / 8;
    const bool rot = a.hb_log2 > 0;
    const bool g_ok = tid < ng;

    // this thread's permutation and sign words, then the row into LDS
    int32_t pw[8];
    uint32_t sg[2];
    if (rot) rot_tables(a.perm, a.sign, g_ok ? tid : 0, pw, sg);
    rot_stage_row(a.x, a.x_dt, a.x_vec, row * a.x_stride, a.n, s_x, tid, T);
    __syncthreads();

    float v[8];
    if (rot) {
        rot_gather(s_x, pw, sg, a.n, g_ok, v);
        rot_transform(v, s_x, tid, T, a.hb_log2);
    } else {
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = g_ok ? s_x[tid * 8 + k] : 0.0f;
    }
    float am = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        if (rot) v[k] = rows_round_act(v[k] * a.scale, a.act_dt);
        am = fmaxf(am, fabsf(v[k]));  // skips NaN, which reaches its output row through the product
    }
    const int e = rot_row_exponent(am, s_max, tid, T);
    if (tid == 0) a.e[row] = e;
    const int kt = tid / RW_TILE_G, t = tid & 7, q = (tid >> 3) & 3;
    if (kt >= a.kt) return;
    half8_t h;
#pragma unroll
    for (int k = 0; k < 8; k++) h[k] = (_Float16)ldexpf(v[k], e);
    auto put = [&](int64_t r, half8_t w) { a.a[(((r >> 4) * a.kt + kt) * 8 + t) * 64 + q * 16 + (r & 15)] = w; };
    if constexpr (!BF) {
        put(row, h);
        return;
    }
    // the upper 8 of a value's 11 bits, and the rest (nothing of an infinity)
    u32x4 hi, lo;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        uint32_t u[2], r[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float f = (float)h[2 * k + j];
            u[j] = __float_as_uint(f) & 0xFFFF0000u;
            r[j] = fabsf(f) < __builtin_inff() ? __float_as_uint(f - __uint_as_float(u[j])) : 0u;
        }
        hi[k] = (u[0] >> 16) | u[1];
        lo[k] = (r[0] >> 16) | (r[1] & 0xFFFF0000u);
    }
    put(row, __builtin_bit_cast(half8_t, hi));
    put(8 + row, __builtin_bit_cast(half8_t, lo));
}

// ------------------------------------------------------------- the product
struct RowsSeg {
    const int16_t* idx0;
    const void* idx1;
    const void* scale;
    void* y;
    int64_t y_stride;
    int rows;
    int tile0;  // first column tile of this matrix
};

struct RowsArgs {
    const half8_t* a;  // packed activation
    const int* e;
    int m;
    int kt;  // k tiles
    int ng;
    const void* cb0;  // codebooks (rows_wide_kernel: fp16)
    const void* cb1;
    int s_dt;
    int y_dt;
    float rs;
    int nseg;
    int kw;  // waves of a workgroup that share a column tile's k tiles
    int nc;  // column tiles of a workgroup of rows_gemm_kernel
    int nz;  // workgroups that share a tile's k tiles (gridDim.z); nc is 1 then
    float* part;    // nz > 1: [row block][column tile][nz][16 MT][16] sums
    uint32_t* cnt;  // nz > 1: arrivals per [row block][column tile], zero
    int tiles;      // column tiles of all matrices
    RowsSeg seg[4];
};

// A wave's codes of one column (16 columns a wave, lane l: column l % 16)
// and k tile: the 8 groups 8 (l / 16) + t.
template <int S2>
struct RowCodes {
    u32x4 w0;
    u32x4 w1;  // (16,8): the first two words
    __device__ __forceinline__ void load(const RowsSeg& s, int64_t off)
    {
        w0 = __builtin_nontemporal_load((const u32x4*)(s.idx0 + off));
        if constexpr (S2 == VQ2_S2_U16) w1 = __builtin_nontemporal_load((const u32x4*)((const int16_t*)s.idx1 + off));
        if constexpr (S2 == VQ2_S2_U8) {
            const u32x2 w = __builtin_nontemporal_load((const u32x2*)((const uint8_t*)s.idx1 + off));
            w1[0] = w.x;
            w1[1] = w.y;
        }
    }
    __device__ __forceinline__ uint32_t c0(int t) const { return (w0[t >> 1] >> (16 * (t & 1))) & 0xFFFFu; }
    __device__ __forceinline__ uint32_t c1(int t) const
    {
        if constexpr (S2 == VQ2_S2_U8) return (w1[t >> 2] >> (8 * (t & 3))) & 0xFFu;
        else return (w1[t >> 1] >> (16 * (t & 1))) & 0xFFFFu;
    }
};

// How rows_gemm_kernel takes its codebooks: the dtype codes (bf16 and fp32
// rounded to fp16 as gathered), or bf16 as it is.
constexpr int RW_CB_BF = 3;

// A centroid as gathered, and as the matrix instruction's operand.
template <int CB>
struct RowCentroid {
    half8_t h;
    __device__ __forceinline__ void load(const void* cb, uint32_t code) { h = ((const half8_t*)cb)[code]; }
    __device__ __forceinline__ half8_t operand() const { return h; }
};

template <>
struct RowCentroid<VQ2_DT_BF16> {
    u32x4 u;
    __device__ __forceinline__ void load(const void* cb, uint32_t code) { u = ((const u32x4*)cb)[code]; }
    __device__ __forceinline__ half8_t operand() const { return rows_bf16_to_half(u); }
};

template <>
struct RowCentroid<VQ2_DT_F32> {
    u32x4 lo, hi;
    __device__ __forceinline__ void load(const void* cb, uint32_t code)
    {
        lo = ((const u32x4*)cb)[2 * (size_t)code];
        hi = ((const u32x4*)cb)[2 * (size_t)code + 1];
    }
    __device__ __forceinline__ half8_t operand() const { return rows_f32_to_half(lo, hi); }
};

__device__ __forceinline__ const RowsSeg& rows_seg(const RowsArgs& a, int tile)
{
    int s = 0;
    for (int i = 1; i < a.nseg; i++) s += tile >= a.seg[i].tile0 ? 1 : 0;
    return a.seg[s];
}

constexpr int RW_MAX_WAVES = 16;
constexpr int RW_MAX_MT = 4;     // 16-row tiles of a wave of rows_gemm_kernel
constexpr int RW_WIDE_WAVES = 4; // waves of a rows_wide_kernel workgroup
constexpr int RW_MAX_Z = 4;  // workgroups that share a tile's k tiles

// Up to 16 * MT rows: a workgroup is nc column tiles of 16 columns x kw waves
// over the k tiles; blockIdx.y counts blocks of 16 * MT rows.  CB: the
// codebooks (RowCentroid); with RW_CB_BF the packed rows are bf16 too, the
// addends of row r in rows r and 8 + r of the one tile.
template <int S2, int MT, int CB>
__global__ void __launch_bounds__(64 * RW_MAX_WAVES) rows_gemm_kernel(const RowsArgs a)
{
    touch_kernargs(a);
    extern __shared__ __align__(16) float s_red[];  // [waves][16 MT][17]
    __shared__ half8_t s_c1[S2 == VQ2_S2_U8 ? 256 : 1];
    __shared__ int s_e[16 * MT];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 15, q = lane >> 4;
    const int kw = a.kw, nc = a.nc;
    const int ct0 = nc == 1 ? 0 : wave / kw;  // this wave's column tile of the workgroup
    const int tile = (int)blockIdx.x * nc + ct0;
    const int k0 = (int)blockIdx.z * kw + wave - ct0 * kw, kstep = kw * a.nz;
    const RowsSeg& sg = rows_seg(a, tile);
    const int col0 = (tile - sg.tile0) * 16;  // may lie past the last matrix's rows (tail workgroup)
    const int mt0 = (int)blockIdx.y * MT;
    const half8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    auto mfma = [](half8_t x, half8_t b, f32x4_t c) {
        return mfma_16<CB != RW_CB_BF>(__builtin_bit_cast(u32x4, x), __builtin_bit_cast(u32x4, b), c);
    };

    // what the epilogue needs, loaded ahead of everything else: the rows'
    // exponents and (one column tile: a thread keeps its column) the scale.
    // Finding the matrix of each output again, with its divisions and its
    // loads, took 4.4 of 35.9 us for gate and up of 6144 x 2048 at 3 bpw and 64 rows.
    const int e_pre = tid < 16 * MT ? a.e[min(mt0 * 16 + tid, a.m - 1)] : 0;
    const int ecol = min(col0 + tid % 16, sg.rows - 1);
    const uint32_t s_pre = nc == 1 ? load_raw(sg.scale, a.s_dt, ecol) : 0u;

    const int64_t rowoff = (int64_t)(col0 + nl < sg.rows ? col0 + nl : 0) * a.ng;
    // row tiles past the last one read tile mt_last again (results dropped)
    const int mt_last = (a.m - 1) >> 4;
    const half8_t* ap[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) ap[i] = a.a + (int64_t)min(mt0 + i, mt_last) * a.kt * 512 + lane;

    f32x4_t acc[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    RowCodes<S2> cd;
    auto load_codes = [&](int kt) {
        // the last k tile may be short: whole k blocks of 8 groups are missing
        const int g = kt * RW_TILE_G + q * 8;
        cd.load(sg, rowoff + (g < a.ng ? g : 0));
    };
    if (k0 < a.kt) load_codes(k0);
    if constexpr (S2 == VQ2_S2_U8) {
        for (int i = tid; i < 256; i += (int)blockDim.x) {
            RowCentroid<CB> c;
            c.load(a.cb1, i);
            s_c1[i] = c.operand();
        }
        __syncthreads();
    }
    for (int kt = k0; kt < a.kt; kt += kstep) {
        const bool g_ok = kt * RW_TILE_G + q * 8 < a.ng;
        // steps whose gathers are in flight together: as many as the 128 registers of a lane hold
        constexpr int TS = CB == VQ2_DT_F32 || (CB == VQ2_DT_BF16 && S2 == VQ2_S2_U8 && MT >= 3) ? 4 : 8;
#pragma unroll
        for (int t0 = 0; t0 < 8; t0 += TS) {
            RowCentroid<CB> b0[TS];
            RowCentroid<S2 == VQ2_S2_U8 ? VQ2_DT_F16 : CB> b1[TS];  // (16,8): from LDS, as operands
#pragma unroll
            for (int t = 0; t < TS; t++) {
                b0[t].load(a.cb0, cd.c0(t0 + t));
                if constexpr (S2 == VQ2_S2_U16) b1[t].load(a.cb1, cd.c1(t0 + t));
                if constexpr (S2 == VQ2_S2_U8) b1[t].h = s_c1[cd.c1(t0 + t)];
            }
            if (t0 + TS == 8 && kt + kstep < a.kt) load_codes(kt + kstep);
#pragma unroll
            for (int t = 0; t < TS; t++) {
                half8_t av[MT];
#pragma unroll
                for (int i = 0; i < MT; i++) av[i] = ap[i][((int64_t)kt * 8 + t0 + t) * 64];
                const half8_t bb = g_ok ? b0[t].operand() : zero8;
#pragma unroll
                for (int i = 0; i < MT; i++) acc[i] = mfma(av[i], bb, acc[i]);
                if constexpr (S2 != VQ2_S2_NONE) {
                    const half8_t bc = g_ok ? b1[t].operand() : zero8;
#pragma unroll
                    for (int i = 0; i < MT; i++) acc[i] = mfma(av[i], bc, acc[i]);
                }
            }
        }
    }

    // rows r and 8 + r of a tile lie 32 lanes apart: the sum of the two addends
    if constexpr (CB == RW_CB_BF)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[0][e] += xor32(acc[0][e]);

    // D[i][j]: activation row 4 (l / 16) + e of the tile, column l % 16; the
    // waves' sums meet in LDS and are added in wave order
    constexpr int LD = 17, TILE = 16 * MT * LD;
    float* mine = s_red + wave * TILE;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) mine[(i * 16 + q * 4 + e) * LD + nl] = acc[i][e];
    if (tid < 16 * MT) s_e[tid] = e_pre;
    __syncthreads();
    const int mrows = min(16 * MT, a.m - mt0 * 16);
    const float* red = s_red;
    int nred = kw;
    if (a.nz > 1) {
        // this workgroup's sums; the last of the tile's workgroups adds them
        // in order (arrive_last)
        const int64_t unit = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
        float* pt = a.part + (unit * a.nz + blockIdx.z) * (256 * MT);
        for (int t = tid; t < 256 * MT; t += (int)blockDim.x) {
            const float* p = s_red + t / 16 * LD + t % 16;
            float sum = 0.0f;
            for (int w = 0; w < kw; w++) sum += p[w * TILE];
            share_store(pt + t, sum);
        }
        if (!arrive_last(a.cnt + unit, (uint32_t)a.nz)) return;
        pt = a.part + unit * a.nz * (256 * MT);
        for (int t = tid; t < 256 * MT; t += (int)blockDim.x) {
            // at most RW_MAX_Z partials, their loads in flight together
            float v[RW_MAX_Z], sum = 0.0f;
#pragma unroll
            for (int z = 0; z < RW_MAX_Z; z++) v[z] = share_load(pt + min(z, a.nz - 1) * (256 * MT) + t);
#pragma unroll
            for (int z = 0; z < RW_MAX_Z; z++) sum += z < a.nz ? v[z] : 0.0f;
            s_red[t / 16 * LD + t % 16] = sum;
        }
        __syncthreads();
        nred = 1;
    }
    if (nc == 1) {
        // (blockDim is a multiple of 16: the thread's column stays)
        const int c = tid % 16;
        const float s = raw_as_f32(s_pre, a.s_dt);
        if (col0 + c >= sg.rows) return;
        for (int r = tid / 16; r < mrows; r += (int)blockDim.x / 16) {
            const float* p = red + r * LD + c;
            float sum = 0.0f;
            for (int w = 0; w < nred; w++) sum += p[w * TILE];
            store_from_f32(sg.y, a.y_dt, (int64_t)(mt0 * 16 + r) * sg.y_stride + col0 + c, (ldexpf(sum, -s_e[r]) * s) * a.rs);
        }
        return;
    }
    for (int t = tid; t < nc * mrows * 16; t += (int)blockDim.x) {
        const int c = t % 16, u = t / 16;
        const int r = u % mrows, ct = u / mrows;
        const int tl = (int)blockIdx.x * nc + ct;
        const RowsSeg& so = rows_seg(a, tl);
        const int col = (tl - so.tile0) * 16 + c;
        if (col >= so.rows) continue;
        const float* p = red + ct * kw * TILE + r * LD + c;
        float sum = 0.0f;
        for (int w = 0; w < nred; w++) sum += p[w * TILE];
        const float s = load_as_f32(so.scale, a.s_dt, col);
        store_from_f32(so.y, a.y_dt, (int64_t)(mt0 * 16 + r) * so.y_stride + col, (ldexpf(sum, -s_e[r]) * s) * a.rs);
    }
}

// Many rows: a workgroup is 4 waves of 16 columns x 16 * MT rows and walks
// all k tiles of its share (blockIdx.z of nz).  Per stage of TS steps the waves
// gather their own operands into registers, a stage ahead, and stage the rows'
// packed operands in LDS for all of them, two buffers in turn.  So a code is
// gathered once per 128 or 256 rows instead of 64.  Bound by those gathers and,
// as a wave reads every operand of the rows from LDS for its 16 columns, by
// the LDS rate (with all codes alike, two 6144 x 2048 matrices at 4 bpw and
// 1024 rows took 133 us of the 192 of a graph replay; 173 a call now).
// Measured there, us a replay: 8 waves and 4 steps a stage 208, 8 and 2 205,
// 4 and 2 192; 32 columns a wave, which halves
// the LDS reads, spills at 256 rows (266), and so do 512 rows (216).
template <int S2, int MT, int TS>
__global__ void __launch_bounds__(64 * RW_WIDE_WAVES, 2) rows_wide_kernel(const RowsArgs a)
{
    touch_kernargs(a);
    constexpr int NW = RW_WIDE_WAVES;
    constexpr int HS = 8 / TS, NF = MT * TS;  // stages of a k tile, operands of a stage
    constexpr int NL = (NF + NW - 1) / NW;    // operands a wave stages
    static_assert(HS % 2 == 0, "two buffers in turn");
    extern __shared__ __align__(16) half8_t s_wide[];
    __shared__ half8_t s_c1[S2 == VQ2_S2_U8 ? 256 : 1];
    half8_t (*s_a)[NF][64] = (half8_t (*)[NF][64])s_wide;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 15, q = lane >> 4;
    const int tile = (int)blockIdx.x * NW + wave;
    const RowsSeg& sg = rows_seg(a, tile);
    const int col = (tile - sg.tile0) * 16 + nl;  // may lie past the last matrix's rows
    const bool col_ok = col < sg.rows;
    const int mt0 = (int)blockIdx.y * MT, mt_last = (a.m - 1) >> 4;
    const int kt0 = (int)((int64_t)a.kt * blockIdx.z / a.nz), kt1 = (int)((int64_t)a.kt * (blockIdx.z + 1) / a.nz);
    const half8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
    const int64_t rowoff = (int64_t)(col_ok ? col : 0) * a.ng;

    RowCodes<S2> c0, c1;
    auto load_codes = [&](RowCodes<S2>& c, int kt) {
        const int g = min(kt, a.kt - 1) * RW_TILE_G + q * 8;
        c.load(sg, rowoff + (g < a.ng ? g : 0));
    };
    load_codes(c0, kt0);
    if constexpr (S2 == VQ2_S2_U8) {
        for (int i = tid; i < 256; i += 64 * NW) s_c1[i] = ((const half8_t*)a.cb1)[i];
        __syncthreads();
    }

    // this wave stages the operands f = wave + NW i of every stage: row tile
    // f / TS, step f % TS
    const half8_t* src[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int f = min(wave + NW * i, NF - 1);
        src[i] = a.a + (int64_t)min(mt0 + f / TS, mt_last) * a.kt * 512 + f % TS * 64;
    }
    half8_t sa[NL];
    auto load_a = [&](int stage) {
#pragma unroll
        for (int i = 0; i < NL; i++) sa[i] = (src[i] + stage * (64 * TS))[(uint32_t)lane];
    };
    f32x4_t acc[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    half8_t b0[TS], b1[TS], n0[TS], n1[TS];
    auto gather = [&](const RowCodes<S2>& c, int t0, half8_t (&g0)[TS], half8_t (&g1)[TS]) {
#pragma unroll
        for (int j = 0; j < TS; j++) {
            g0[j] = ((const half8_t*)a.cb0)[c.c0(t0 + j)];
            if constexpr (S2 == VQ2_S2_U16) g1[j] = ((const half8_t*)a.cb1)[c.c1(t0 + j)];
            if constexpr (S2 == VQ2_S2_U8) g1[j] = s_c1[c.c1(t0 + j)];
        }
    };
    load_a(kt0 * HS);
    gather(c0, 0, b0, b1);
    load_codes(c1, kt0 + 1);

    for (int kt = kt0; kt < kt1; kt++) {
        const bool g_ok = kt * RW_TILE_G + q * 8 < a.ng;
#pragma unroll
        for (int h = 0; h < HS; h++) {
#pragma unroll
            for (int i = 0; i < NL; i++)
                if (NF % NW == 0 || wave + NW * i < NF) s_a[h & 1][wave + NW * i][lane] = sa[i];
            __syncthreads();
            if (h + 1 < HS || kt + 1 < kt1) {
                load_a(kt * HS + h + 1);
                if (h + 1 < HS) gather(c0, (h + 1) * TS, n0, n1);
                else gather(c1, 0, n0, n1);
            }
            if (h + 1 == HS) {
                c0 = c1;
                load_codes(c1, kt + 2);
            }
            // operands in batches, the next one's LDS reads before this one's
            // products (left to itself the compiler waits for each read and
            // issues the stage's loads after its products)
            __builtin_amdgcn_sched_barrier(0);
            constexpr int FB = 4, NB = NF / FB;
            half8_t fr[2][FB];
            // operand u: step u / MT, row tile u % MT
            auto read = [&](int bt, half8_t (&r)[FB]) {
#pragma unroll
                for (int f = 0; f < FB; f++) {
                    const int u = bt * FB + f;
                    r[f] = s_a[h & 1][u % MT * TS + u / MT][lane];
                }
            };
            read(0, fr[0]);
#pragma unroll
            for (int j = 0; j < TS; j++) {
                b0[j] = g_ok ? b0[j] : zero8;
                if constexpr (S2 != VQ2_S2_NONE) b1[j] = g_ok ? b1[j] : zero8;
            }
#pragma unroll
            for (int bt = 0; bt < NB; bt++) {
                if (bt + 1 < NB) read(bt + 1, fr[(bt + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int f = 0; f < FB; f++) {
                    const int i = (bt * FB + f) % MT, j = (bt * FB + f) / MT;
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fr[bt & 1][f], b0[j], acc[i], 0, 0, 0);
                }
                if constexpr (S2 != VQ2_S2_NONE) {
#pragma unroll
                    for (int f = 0; f < FB; f++) {
                        const int i = (bt * FB + f) % MT, j = (bt * FB + f) / MT;
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fr[bt & 1][f], b1[j], acc[i], 0, 0, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int j = 0; j < TS; j++) {
                b0[j] = n0[j];
                b1[j] = n1[j];
            }
        }
    }

    if (!col_ok) return;
    const float s = a.nz > 1 ? 0.0f : load_as_f32(sg.scale, a.s_dt, col);
#pragma unroll
    for (int u = 0; u < MT * 4; u++) {
        const int i = u / 4, e = u % 4;
        const int row = (mt0 + i) * 16 + q * 4 + e;
        if (row >= a.m) continue;
        const float p = ldexpf(acc[i][e], -a.e[row]);
        if (a.nz > 1)
            a.part[((int64_t)blockIdx.z * a.m + row) * (a.tiles * 16) + tile * 16 + nl] = p;
        else
            store_from_f32(sg.y, a.y_dt, (int64_t)row * sg.y_stride + col, (p * s) * a.rs);
    }
}

// y = (the shares of the k tiles added in order) * scale * rs, for nz > 1
__global__ void __launch_bounds__(256) rows_sum_kernel(const RowsArgs a)
{
    const int c4 = (int)blockIdx.x * 256 + threadIdx.x, row = blockIdx.y;
    if (c4 >= a.tiles * 4) return;
    const int64_t ld = (int64_t)a.tiles * 16;
    const float* p = a.part + row * ld + c4 * 4;
    f32x4_t v[RW_MAX_Z], sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int z = 0; z < RW_MAX_Z; z++) v[z] = *(const f32x4_t*)(p + (int64_t)min(z, a.nz - 1) * a.m * ld);
#pragma unroll
    for (int z = 0; z < RW_MAX_Z; z++)
        if (z < a.nz) sum += v[z];
    const int tile = c4 / 4;
    const RowsSeg& sg = rows_seg(a, tile);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int col = (tile - sg.tile0) * 16 + (c4 % 4) * 4 + k;
        if (col < sg.rows)
            store_from_f32(sg.y, a.y_dt, (int64_t)row * sg.y_stride + col, (sum[k] * load_as_f32(sg.scale, a.s_dt, col)) * a.rs);
    }
}

// ------------------------------------------------------------------ launch
struct RowsPlan {
    int cb;            // codebooks of rows_gemm_kernel (RowCentroid)
    int cvt;           // rounded to fp16 by the packing launch (cb = VQ2_DT_F16)
    int kt;
    int mt;            // 16-row tiles of a wave
    int kw, nc, nz;    // waves and workgroups over a column tile's k tiles; column tiles of a workgroup
    int wide;          // rows_wide_kernel
    int64_t tiles;     // column tiles of all matrices
    int64_t grid_x, grid_y;
    // workspace: arrival counters, the rows' exponents, the packed
    // activation, fp16 codebooks, the partial sums of nz > 1
    size_t e, a, h0, h1, part, total;
};

static size_t up256(size_t b) { return (b + 255) / 256 * 256; }

// Above 64 rows: rows_wide_kernel where a model of both kernels puts it ahead.
// L2 requests are what both wait for: a gather per code and row block, and the
// packed activation's lines, read once per 16 columns (rows_gemm_kernel) or
// per workgroup of 64 (rows_wide_kernel).  Rates in requests a ns, measured
// (MI355X): rows_gemm_kernel 235; rows_wide_kernel a workgroup 1.0 with 128
// rows and 0.75 with 256, all of them 200 and 160; nz > 1 adds the partials'
// launch (4 us) and their traffic (5 TB/s).  It serves to order the plans, not
// to tell their times: a CU with less than two workgroups and the rows that
// pad a tile are not in it (2048 + 512 + 512 rows x 2048, 2, 333 rows: 21 us
// for a launch of 33).  Over fourteen shapes and 70 to 1024 rows the choice
// is the fastest of the seven or within 1 % of it (graph replays, us a call,
// rows x n, bits, activation rows: rows_gemm / chosen / the next best): 2 x
// 6144 x 2048, 4, 100 rows 73 / 53 / 56, 1024 rows 523 / 175 / 231; 2048 x
// 6144, 4, 256 rows 81 / 59 / 62, 1024 297 / 118 / 118; 2048 + 512 + 512 x
// 2048, 2, 333 rows 41.8 / 39.7 / 40.0; 2999 x 4096, 2, 100 rows 34.1 / 33.2 /
// 36.1; 512 x 2048, 2, stays (1024 rows 29.3, the best wide plan 34.5).
static void rows_plan_wide(const RowsCall& c, RowsPlan& p)
{
    const double stages = c.s2 == VQ2_S2_U16 ? 2 : 1, m = (double)c.m;
    double codes = 0, rows = 0;
    for (int s = 0; s < c.nseg; s++) rows += (double)c.seg[s].rows;
    codes = rows * (double)(c.n / 8) * stages;
    const double a_lines = m * (double)c.n * 2 / 128;
    const double t_rows = (codes * (double)p.grid_y + a_lines * (double)p.tiles) / 235e3;
    double best = t_rows;
    const int64_t blocks = (p.tiles + RW_WIDE_WAVES - 1) / RW_WIDE_WAVES;
    for (int mt = 8; mt <= 16; mt += 8) {
        const int64_t rb = (c.m + 16 * mt - 1) / (16 * mt);
        const double req = codes * (double)rb + a_lines * (double)blocks;
        for (int nz = 1; nz <= std::min(RW_MAX_Z, p.kt); nz *= 2) {
            const double rate = std::min((double)(blocks * rb * nz) * (mt == 8 ? 1.0 : 0.75), mt == 8 ? 200.0 : 160.0);
            const double t = req / (rate * 1e3) + (nz > 1 ? 4.0 + nz * m * rows * 8 / 5e6 : 0.0) + 1.0;
            if (t >= best) continue;
            best = t;
            p.wide = 1;
            p.mt = mt;
            p.nz = nz;
            p.nc = RW_WIDE_WAVES;
            p.kw = 1;
            p.grid_y = rb;
        }
    }
}

static RowsPlan rows_plan(const RowsCall& c)
{
    RowsPlan p{};
    p.kt = (int)((c.n / 8 + RW_TILE_G - 1) / RW_TILE_G);
    p.cb = c.cb_dt == VQ2_DT_BF16 && c.m <= RW_BF_ROWS ? RW_CB_BF : c.cb_dt;
    // row blocks of at most 64 rows, as even as whole tiles allow
    const int64_t mtiles = (c.m + 15) / 16, blocks = (mtiles + RW_MAX_MT - 1) / RW_MAX_MT;
    p.mt = (int)((mtiles + blocks - 1) / blocks);
    for (int s = 0; s < c.nseg; s++) p.tiles += (c.seg[s].rows + 15) / 16;
    p.grid_y = (c.m + 16 * p.mt - 1) / (16 * p.mt);
    // Few column tiles leave CUs idle, and a CU gathers at most ~0.9 codes a
    // ns however few others do: several workgroups then share a tile's k
    // tiles, while a workgroup has 6144 gathers or more (below that the
    // sum over workgroups costs more, ~1.5 us: 2048 x 2048 at 2 bpw, 16 rows,
    // 4096 gathers 13.7 us a call, two workgroups 14.4; at 4 bpw 18.3 / 17.5;
    // 2048 x 6144 at 4 bpw 34.5 / 28.3; 512 x 6144 40.1 / 26.3 / 20.7 with
    // four) and the launch stays within a workgroup per CU.
    const int64_t gathers = 16 * (c.n / 8) * (c.s2 == VQ2_S2_U16 ? 2 : 1);
    p.nz = 1;
    while (2 * p.nz <= std::min(RW_MAX_Z, p.kt) && 2 * p.nz * p.tiles * p.grid_y <= device_cu_count() &&
           gathers / p.nz >= 6144)
        p.nz *= 2;
    // the k tiles over up to 16 waves, as evenly as whole tiles allow; short
    // reductions put several column tiles into a workgroup of 8 waves where
    // every CU still has one (1024 x 1024 at 4 bpw in 32 workgroups of two
    // tiles took 18.6 us a call, in 64 of one 13.9)
    const int per = (p.kt + p.nz - 1) / p.nz, rounds = (per + RW_MAX_WAVES - 1) / RW_MAX_WAVES;
    p.kw = (per + rounds - 1) / rounds;
    p.nc = (int)std::max<int64_t>(1, std::min<int64_t>(8 / p.kw, p.tiles * p.grid_y / device_cu_count()));
    if (c.m > 16 * RW_MAX_MT) rows_plan_wide(c, p);
    p.grid_x = (p.tiles + p.nc - 1) / p.nc;
    int64_t codes = 0;
    for (int s = 0; s < c.nseg; s++) codes += c.seg[s].rows * (c.n / 8);
    p.cvt = c.cb_dt == VQ2_DT_BF16 ? p.wide
            : c.cb_dt == VQ2_DT_F32 && (p.wide || c.s2 == VQ2_S2_U16 || codes * p.grid_y > RW_F32_GATHERS);
    if (p.cvt) p.cb = VQ2_DT_F16;
    const int64_t units = p.nz > 1 && !p.wide ? p.grid_x * p.grid_y : 0;
    p.e = up256((size_t)units * sizeof(uint32_t));
    p.a = p.e + up256((size_t)c.m * sizeof(int));
    p.h0 = p.a + (size_t)((c.m + 15) / 16) * p.kt * 512 * sizeof(half8_t);
    p.h1 = p.h0 + (p.cvt ? (size_t)RW_CB_ROWS * sizeof(half8_t) : 0);
    p.part = p.h1 + (!p.cvt || c.s2 == VQ2_S2_NONE ? 0 : (size_t)(c.s2 == VQ2_S2_U8 ? 256 : RW_CB_ROWS) * sizeof(half8_t));
    p.total = p.part + (p.wide && p.nz > 1 ? (size_t)p.nz * c.m * p.tiles * 16 : (size_t)units * p.nz * 256 * p.mt) *
                           sizeof(float);
    return p;
}

static int rows_check(const RowsCall& c)
{
    if (c.n > RW_MAX_N || c.n < 64 || c.n % 64)
        return set_error(VQ2_ERR_UNSUPPORTED, "vq2_rows_gemm: n=%lld must be a multiple of 64 up to %lld", (long long)c.n,
                         (long long)RW_MAX_N);
    if (c.m < 1 || c.m > 1 << 20)
        return set_error(VQ2_ERR_UNSUPPORTED, "vq2_rows_gemm: %lld activation rows outside 1..2^20", (long long)c.m);
    for (int s = 0; s < c.nseg; s++)
        if (c.seg[s].rows < 0 || c.seg[s].rows > 0x0FFFFFFF)
            return set_error(VQ2_ERR_UNSUPPORTED, "vq2_rows_gemm: matrix %d has %lld rows", s, (long long)c.seg[s].rows);
    return VQ2_OK;
}

size_t rows_workspace_bytes(const RowsCall& c)
{
    return rows_check(c) == VQ2_OK ? rows_plan(c).total : 0;
}

template <int S2, int MT, int CB>
static hipError_t rows_launch_t(const RowsArgs& a, dim3 grid, int waves, hipStream_t st)
{
    // opt in to more than 64 KiB of dynamic LDS, once per instantiation
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    constexpr size_t SHM_WAVE = 16 * MT * 17 * sizeof(float);
    std::call_once(once, [] {
        attr = hipFuncSetAttribute((const void*)rows_gemm_kernel<S2, MT, CB>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)(RW_MAX_WAVES * SHM_WAVE));
    });
    if (attr != hipSuccess) return attr;
    const size_t shm = waves * SHM_WAVE;
    hipLaunchKernelGGL((rows_gemm_kernel<S2, MT, CB>), grid, dim3(64 * waves), shm, st, a);
    return hipGetLastError();
}

template <int S2, int CB>
static hipError_t rows_launch_c(int mt, const RowsArgs& a, dim3 grid, int waves, hipStream_t st)
{
    if constexpr (CB == RW_CB_BF) {
        return rows_launch_t<S2, 1, CB>(a, grid, waves, st);
    } else {
        switch (mt) {
        case 1: return rows_launch_t<S2, 1, CB>(a, grid, waves, st);
        case 2: return rows_launch_t<S2, 2, CB>(a, grid, waves, st);
        case 3: return rows_launch_t<S2, 3, CB>(a, grid, waves, st);
        default: return rows_launch_t<S2, 4, CB>(a, grid, waves, st);
        }
    }
}

template <int S2>
static hipError_t rows_launch_s(int mt, int cb, const RowsArgs& a, dim3 grid, int waves, hipStream_t st)
{
    switch (cb) {
    case VQ2_DT_F16: return rows_launch_c<S2, VQ2_DT_F16>(mt, a, grid, waves, st);
    case VQ2_DT_BF16: return rows_launch_c<S2, VQ2_DT_BF16>(mt, a, grid, waves, st);
    case RW_CB_BF: return rows_launch_c<S2, RW_CB_BF>(mt, a, grid, waves, st);
    default:
        // fp32: rows_plan gathers only single 16-bit stages of it
        if constexpr (S2 != VQ2_S2_U16) return rows_launch_c<S2, VQ2_DT_F32>(mt, a, grid, waves, st);
        else return hipErrorInvalidValue;
    }
}

template <int S2, int MT, int TS>
static hipError_t rows_wide_t(const RowsArgs& a, dim3 grid, hipStream_t st)
{
    // opt in to more than 64 KiB of dynamic LDS, once per instantiation
    constexpr int SHM = 2 * MT * TS * 64 * (int)sizeof(half8_t);
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    std::call_once(once, [] {
        attr = hipFuncSetAttribute((const void*)rows_wide_kernel<S2, MT, TS>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, SHM);
    });
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL((rows_wide_kernel<S2, MT, TS>), grid, dim3(64 * RW_WIDE_WAVES), SHM, st, a);
    return hipGetLastError();
}

template <int S2>
static hipError_t rows_wide_s(int mt, const RowsArgs& a, dim3 grid, hipStream_t st)
{
    return mt == 8 ? rows_wide_t<S2, 8, 4>(a, grid, st) : rows_wide_t<S2, 16, 2>(a, grid, st);
}

static hipError_t rows_pack_launch(const RowsPackArgs& p, int bf, hipStream_t st)
{
    const int T = std::max(64, (p.kt * RW_TILE_G + 63) / 64 * 64);
    int64_t blocks = p.m;
    if (p.cb0) blocks += (RW_CB_ROWS + p.cb1_rows + T - 1) / T;
    const size_t shm = (size_t)T * 8 * sizeof(float);
    if (bf) hipLaunchKernelGGL(rows_pack_kernel<1>, dim3((unsigned)blocks), dim3(T), shm, st, p);
    else hipLaunchKernelGGL(rows_pack_kernel<0>, dim3((unsigned)blocks), dim3(T), shm, st, p);
    return hipGetLastError();
}

int rows_launch(const RowsCall& c)
{
    if (int r = rows_check(c)) return r;
    int hl = 0;
    while ((1LL << hl) < c.hb) hl++;
    if (c.hb && ((1LL << hl) != c.hb || c.hb < 64 || c.n % c.hb))
        return set_error(VQ2_ERR_ARG, "vq2_rows_gemm: hb=%lld must be 0 or a power of two of at least 64 dividing n",
                         (long long)c.hb);
    for (int s = 0; s < c.nseg; s++) {
        const RowsSegCall& g = c.seg[s];
        const uintptr_t al = (uintptr_t)g.idx0 | (c.s2 == VQ2_S2_U16 ? (uintptr_t)g.idx1 : 0);
        if (al % 16 || (c.s2 == VQ2_S2_U8 && (uintptr_t)g.idx1 % 8))
            return set_error(VQ2_ERR_UNSUPPORTED, "vq2_rows_gemm: index planes must be 16-byte aligned");
    }
    const RowsPlan p = rows_plan(c);
    if (p.tiles == 0) return VQ2_OK;
    if (p.grid_x > 0x3FFFFFFF || p.grid_y > 65535)
        return set_error(VQ2_ERR_UNSUPPORTED, "vq2_rows_gemm: grid too large");
    if (!c.workspace || c.ws_bytes < p.total || (uintptr_t)c.workspace % 256)
        return set_error(VQ2_ERR_ARG, "vq2_rows_gemm: workspace of %zu bytes (256-byte aligned) needed, got %zu", p.total,
                         c.ws_bytes);
    char* ws = (char*)c.workspace;
    hipStream_t st = (hipStream_t)c.stream;

    RowsPackArgs k{};
    k.x = c.x;
    k.x_dt = c.x_dt;
    k.x_vec = (uintptr_t)c.x % 16 == 0 && (c.x_stride * dt_size(c.x_dt)) % 16 == 0;
    k.x_stride = c.x_stride;
    k.m = c.m;
    k.n = (int)c.n;
    k.kt = p.kt;
    k.hb_log2 = c.hb ? hl : 0;
    k.perm = c.perm;
    k.sign = c.sign;
    k.scale = c.xscale;
    k.act_dt = c.act_dt;
    k.a = (half8_t*)(ws + p.a);
    k.e = (int*)(ws + p.e);
    k.cnt = (uint32_t*)ws;
    k.n_cnt = p.nz > 1 && !p.wide ? (int)(p.grid_x * p.grid_y) : 0;
    if (p.cvt) {
        k.cb0 = c.cb0;
        k.cb1 = c.cb1;
        k.cb_dt = c.cb_dt;
        k.cb1_rows = c.s2 == VQ2_S2_NONE ? 0 : (c.s2 == VQ2_S2_U8 ? 256 : RW_CB_ROWS);
        k.h0 = (half8_t*)(ws + p.h0);
        k.h1 = (half8_t*)(ws + p.h1);
    }
    hipError_t err = rows_pack_launch(k, p.cb == RW_CB_BF, st);
    if (err != hipSuccess) return set_hip_error(err, "vq2_rows_gemm packing launch");

    RowsArgs a{};
    a.a = k.a;
    a.e = k.e;
    a.m = (int)c.m;
    a.ng = (int)(c.n / 8);
    a.kt = p.kt;
    a.cb0 = p.cvt ? k.h0 : c.cb0;
    a.cb1 = p.cvt ? k.h1 : c.cb1;
    a.s_dt = c.s_dt;
    a.y_dt = c.y_dt;
    a.rs = c.rs;
    a.kw = p.kw;
    a.nc = p.nc;
    a.nz = p.nz;
    a.part = (float*)(ws + p.part);
    a.cnt = k.cnt;
    int64_t tile = 0;
    for (int s = 0; s < c.nseg; s++) {
        const RowsSegCall& g = c.seg[s];
        if (g.rows == 0) continue;
        a.seg[a.nseg++] = RowsSeg{g.idx0, g.idx1, g.scale, g.y, g.y_stride, (int)g.rows, (int)tile};
        tile += (g.rows + 15) / 16;
    }
    a.tiles = (int)p.tiles;
    const dim3 grid((unsigned)p.grid_x, (unsigned)p.grid_y, (unsigned)p.nz);
    if (p.wide) {
        switch (c.s2) {
        case VQ2_S2_U8: err = rows_wide_s<VQ2_S2_U8>(p.mt, a, grid, st); break;
        case VQ2_S2_U16: err = rows_wide_s<VQ2_S2_U16>(p.mt, a, grid, st); break;
        default: err = rows_wide_s<VQ2_S2_NONE>(p.mt, a, grid, st); break;
        }
        if (err == hipSuccess && p.nz > 1) {
            hipLaunchKernelGGL(rows_sum_kernel, dim3((unsigned)((p.tiles * 4 + 255) / 256), (unsigned)c.m), dim3(256), 0, st,
                               a);
            err = hipGetLastError();
        }
        if (err != hipSuccess) return set_hip_error(err, "vq2_rows_gemm launch");
        return VQ2_OK;
    }
    switch (c.s2) {
    case VQ2_S2_U8: err = rows_launch_s<VQ2_S2_U8>(p.mt, p.cb, a, grid, p.kw * p.nc, st); break;
    case VQ2_S2_U16: err = rows_launch_s<VQ2_S2_U16>(p.mt, p.cb, a, grid, p.kw * p.nc, st); break;
    default: err = rows_launch_s<VQ2_S2_NONE>(p.mt, p.cb, a, grid, p.kw * p.nc, st); break;
    }
    if (err != hipSuccess) return set_hip_error(err, "vq2_rows_gemm launch");
    return VQ2_OK;
}

}  // namespace vq2
