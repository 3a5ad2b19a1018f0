// W8A8 projection for gfx950: the engine's linear() with a QuantizedWeight
// (operator/linear.hpp:106-132). Input rows are quantized per row (quantize_rows,
// quant.hpp:112-133, by the per-token kernel), the int8 rows times the int8
// weight [out, in] are exact int32 sums on v_mfma_i32_16x16x64_i8, and the
// epilogue applies y = float(sum) * (row_scale * weight_scale) (+ bias), the
// engine's float steps in its order, each rounded on its own (no contraction),
// so the outputs are bit-identical.
//
// Two kernels. Many rows: output tiles of BM rows x BN features, one workgroup of four or
// eight waves per tile and compute unit, K in 128-byte steps through a ring of LDS stages
// filled by direct-to-LDS buffer loads. Few rows (a decode batch): the weight is read
// once, straight into the matrix instructions' operand registers, by workgroups that
// own a few features and split K over their waves.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "reef_common.hpp"

namespace reef {
namespace {

constexpr int kXcds = 8;
constexpr int kBK = 128;      // bytes of K per step of the tile kernel

struct GemmArgs {
    const int8_t *x;  // [rows, in] quantized rows, row stride in
    const float *xs;  // [rows]
    const int8_t *w;  // [out, in]
    const float *ws;  // [out]
    const float *bias;  // [out] or null
    float *y;
    int64_t y_stride;
    int32_t rows, in, out;
    int32_t m_tiles, n_tiles;
    int32_t y_vec;  // rows of y start on 16 bytes
    uint32_t *status;
};

// The epilogue of one 16 x 16 block: lane l holds, in register i, feature
// n0 + 4 (l / 16) + i of row m0 + l % 16, so a lane's four values are consecutive.
// The engine's float steps, each rounded on its own: safe_multiply(row scale, column
// scale), safe_multiply(sum, scale), add_bias. True when a result is not finite.
__device__ __forceinline__ bool store_block(const GemmArgs &a, int m, int n, float xs,
                                            const float (&ws)[4], const float (&bias)[4],
                                            const i32x4 &acc) {
    bool bad = false;
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma clang fp contract(off)
        const float scale = xs * ws[i];
        float r = (float)acc[i] * scale;
        if (a.bias) r = r + bias[i];
        v[i] = r;
        bad |= n + i < a.out && !__builtin_isfinite(r);
    }
    if (m >= a.rows) return false;
    float *y = a.y + (int64_t)m * a.y_stride + n;
    if (a.y_vec && n + 3 < a.out) {
        *reinterpret_cast<f32x4 *>(y) = v;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n + i < a.out) y[i] = v[i];
    }
    return bad;
}

// Column scales and biases of features n .. n + 3 (zeros past the end).
__device__ __forceinline__ void load_columns(const GemmArgs &a, int n, float (&ws)[4],
                                             float (&bias)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ws[i] = n + i < a.out ? a.ws[n + i] : 0.0f;
        bias[i] = a.bias && n + i < a.out ? a.bias[n + i] : 0.0f;
    }
}

// ---- many rows: tiles ------------------------------------------------------------------
//
// What bounds a tile: its products, and beside them the way of its operands, BM + BN rows
// through the unit's 64 bytes a cycle from L2 into LDS and from LDS to every wave that
// needs them (together about the time of the products at 256 x 128). So a workgroup
// has a compute unit alone, its stages fill the LDS (112 to 160 KB, for an L2 or
// memory round trip of several steps), each half step's operands are read while the
// half step before is multiplied (two register sets), and the reads and direct loads
// are issued one by one between the products. Measured (8192 x 8192 -> 8192): 489 us,
// 2.25 POP/s, where 128 x 128 tiles with two workgroups a unit and no interleaving took
// 740; 4096 x 4096 -> 6144: 103 against 147; 4096 x 8192 -> 1280: 46 against 62. Eight
// waves, two per SIMD, fill each other's waits: 4096 x 8192 -> 1280 in 256 x 128 tiles
// takes 50.8 us with eight, 58.2 with four; in 128 x 160 tiles 46 and 48.5.
//
// Chunk c (16 bytes) of tile row r sits at chunk_pos in its 128-byte LDS row: the 16
// lanes that read one chunk of 16 consecutive rows hit 16 distinct bank groups.
__device__ __forceinline__ int chunk_pos(int r, int c) { return c ^ ((r >> 1) & 7); }

template <int BM, int BN, int WM, int WN, int ST>
__device__ __forceinline__ void gemm_tile(const GemmArgs &a, int8_t *smem) {
    constexpr int W = WM * WN;                          // waves, WM x WN over the tile
    constexpr int MI = BM / WM / 16, NJ = BN / WN / 16;  // 16 x 16 blocks per wave
    constexpr int TA = BM * kBK, TB = BN * kBK;         // operand tiles of a stage
    constexpr int PA = BM / 8 / W, PB = (BN / 8 + W - 1) / W;  // 1 KB direct loads per wave
    constexpr int kLoads = PA + PB, kFirst = kLoads / 2;
    constexpr int kInFlight = kLoads * (ST - 2);        // loads of the stages after the next
    static_assert(BM % (8 * W) == 0 && BN % 16 == 0 && W % 2 == 0, "whole loads");
    static_assert(BN / 8 >= W, "every wave has a block of the weight tile");
    static_assert(kInFlight + kFirst < 64, "vmcnt fits");

    // Workgroup g runs on XCD g % 8: each XCD takes a contiguous run of tiles, in panels
    // of 8 feature tiles, features fastest, so the tiles an XCD works on at a time share
    // their rows and features in its L2.
    const int g = (int)blockIdx.x, count = (int)gridDim.x;
    const int x = g % kXcds, per = count / kXcds, rem = count % kXcds;
    const int t = x * per + min(x, rem) + g / kXcds;
    constexpr int kPanel = 8;
    const int panel = t / (kPanel * a.m_tiles), first = panel * kPanel;
    const int width = min(kPanel, a.n_tiles - first), r0 = t - first * a.m_tiles;
    const int m0 = r0 / width * BM, n0 = (first + r0 % width) * BN;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int col = lane & 15, grp = lane >> 4;

    // Direct loads: wave w fills 1 KB blocks w, w + W, ... of each operand tile; lane L
    // of block b writes tile row 8 b + L / 8 at position L % 8. Rows past the end and
    // chunks past `in` read zeros: their offset is set beyond the buffer.
    const uint32_t xbytes = (uint32_t)((int64_t)a.rows * a.in);
    const uint32_t wbytes = (uint32_t)((int64_t)a.out * a.in);
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(a.x, xbytes);
    const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(a.w, wbytes);
    uint32_t off[kLoads];
    // Where the weight tile's blocks do not divide by the waves, a wave without an i-th
    // block loads its first once more (the same bytes), so that all count the same loads.
    auto b_block = [&](int i) {
        return BN / 8 % W == 0 || wave + W * i < BN / 8 ? wave + W * i : wave;
    };
    // (a wave's blocks are a multiple of 16 rows apart: one chunk position, one k offset)
    const int kch = 16 * chunk_pos(8 * wave + lane / 8, lane % 8);
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        const int r = m0 + 8 * (wave + W * i) + lane / 8;
        off[i] = r < a.rows ? (uint32_t)((int64_t)r * a.in + kch) : xbytes;
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const int r = n0 + 8 * b_block(i) + lane / 8;
        off[PA + i] = r < a.out ? (uint32_t)((int64_t)r * a.in + kch) : wbytes;
    }
    const int steps = (a.in + kBK - 1) / kBK;
    // Direct load i of this wave (PA of x, then PB of the weight) for K step s (clamped
    // to the last) into a stage.
    auto issue = [&](int i, int s, int slot) {
        const int k0 = min(s, steps - 1) * kBK;
        int8_t *st = smem + slot * (TA + TB) + 1024 * wave;
        const bool in_k = k0 + kch < a.in;
        if (i < PA)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                xr, (__attribute__((address_space(3))) void *)(st + 1024 * W * i), 16,
                in_k ? off[i] : xbytes, k0, 0, 0);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                wr, (__attribute__((address_space(3))) void *)(st + TA + 1024 * (b_block(i - PA) - wave)), 16,
                in_k ? off[i] : wbytes, k0, 0, 0);
    };

    // Operand reads: row (BM/WM) wm + 16 i + col of A, (BN/WN) wn + 16 j + col of B,
    // chunk 4 half + grp.
    struct Operands {
        i32x4 x[MI], w[NJ];
    };
    const int arow = ((BM / WM) * wm + col) * kBK, brow = TA + ((BN / WN) * wn + col) * kBK;
    auto read = [&](Operands &o, int r, const int8_t *st) {  // read r of MI + NJ
        if (r < NJ)
            o.w[r < NJ ? r : 0] = *reinterpret_cast<const i32x4 *>(st + brow + 16 * r * kBK);
        else
            o.x[r < NJ ? 0 : r - NJ] =
                *reinterpret_cast<const i32x4 *>(st + arow + 16 * (r - NJ) * kBK);
    };
    auto half_of = [&](int slot, int half) {
        return smem + slot * (TA + TB) + 16 * chunk_pos(col, 4 * half + grp);
    };
    i32x4 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = i32x4{};
    // The products of one half step (D rows: features, D columns: rows of x), with the
    // LDS reads of the next half step's operands and the direct loads [l0, l1) of step s
    // spread between them. Both kinds wait for their place in a queue that the other
    // waves fill as well; issued in one block they kept the matrix core idle for that
    // time, and a step took the sum of its products, reads and loads (4096 x 8192 -> 1280,
    // 256 x 128, four waves: 72.6 us; loads spread 62.5; both spread 58.2).
    auto half_step = [&](const Operands &o, Operands &next, const int8_t *st, auto l0_tag,
                         auto l1_tag, int s, int slot) {
        constexpr int l0 = decltype(l0_tag)::value, L = decltype(l1_tag)::value - l0;
        constexpr int N = MI * NJ, T = MI + NJ + L;  // operation t goes before product t N / T
#pragma unroll
        for (int m = 0; m < N; ++m) {
#pragma unroll
            for (int t = (m * T + N - 1) / N; t < ((m + 1) * T + N - 1) / N; ++t) {
                const int l = t * L / T;  // loads among the operations before t
                if ((t + 1) * L / T > l) issue(l0 + l, s, slot);
                else read(next, t - l, st);
                __builtin_amdgcn_sched_barrier(0);
            }
            acc[m / NJ][m % NJ] = mfma_16x16x64_i8(o.w[m % NJ], o.x[m / NJ], acc[m / NJ][m % NJ]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    using Zero = std::integral_constant<int, 0>;
    using First = std::integral_constant<int, kFirst>;
    using All = std::integral_constant<int, kLoads>;

    // Stages 0 .. ST - 2 and the first loads of stage ST - 1.
#pragma unroll
    for (int s = 0; s < ST; ++s)
#pragma unroll
        for (int i = 0; i < (s < ST - 1 ? kLoads : kFirst); ++i) issue(i, s, s);
    constexpr int kWait0 = kInFlight + kFirst;
    __builtin_amdgcn_s_waitcnt(0xf70 | (kWait0 & 15) | ((kWait0 >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    Operands o0, o1;
#pragma unroll
    for (int r = 0; r < MI + NJ; ++r) read(o0, r, half_of(0, 0));
    int slot = 0, prev = ST - 1;  // stage k sits in `slot`, stage k - 1 sat in `prev`
    for (int k = 0; k < steps; ++k) {
        const int after = slot + 1 == ST ? 0 : slot + 1;
        half_step(o0, o1, half_of(slot, 1), First{}, All{}, k - 1 + ST, prev);
        // This wave's loads of step k + 1 have landed (those of the ST - 2 steps after it
        // may still fly) and its reads of step k are done, so past the barrier stage
        // k + 1 is whole and stage k is free. (s_waitcnt fields: vmcnt in bits 3:0 and
        // 15:14, expcnt 6:4 unconstrained, lgkmcnt 11:8. A bare barrier: __syncthreads()
        // would wait for every load in flight.)
        __builtin_amdgcn_s_waitcnt(0x070 | (kInFlight & 15) | ((kInFlight >> 4) << 14));
        __builtin_amdgcn_s_barrier();
        half_step(o1, o0, half_of(after, 0), Zero{}, First{}, k + ST, slot);
        prev = slot;
        slot = after;
    }
    // The trailing loads of the clamped last steps must land before the workgroup's
    // LDS can be handed to another workgroup.
    __builtin_amdgcn_s_waitcnt(0x070);

    bool bad = false;
    float xs[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int m = m0 + (BM / WM) * wm + 16 * i + col;
        xs[i] = m < a.rows ? a.xs[m] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int n = n0 + (BN / WN) * wn + 16 * j + 4 * grp;
        float ws[4], bias[4];
        load_columns(a, n, ws, bias);
#pragma unroll
        for (int i = 0; i < MI; ++i)
            bad |= store_block(a, m0 + (BM / WM) * wm + 16 * i + col, n, xs[i], ws, bias, acc[i][j]);
    }
    if (bad) flag_status(a.status, REEF_STATUS_BIT_OVERFLOW);
}

template <int BM, int BN, int WM, int WN, int ST>
__global__ __launch_bounds__(64 * WM * WN, 1) void gemm_tile_kernel(GemmArgs a) {
    static_assert(ST * (BM + BN) * kBK <= 160 * 1024, "LDS fits");
    __shared__ __attribute__((aligned(1024))) int8_t smem[ST * (BM + BN) * kBK];
    gemm_tile<BM, BN, WM, WN, ST>(a, smem);
}

// ---- few rows: the weight streamed once -----------------------------------------------
//
// A workgroup of W waves owns 16 NT features and 16 MT rows of x (rows past the end are
// zeros) and splits K over its waves in 128-byte units, wave w taking units w, w + W,
// ...: together the waves read runs of 128 W bytes of each weight row. Weight and x
// fragments go from memory into operand registers (x from L2: it is small), the next
// unit's loads in flight while one is multiplied; the waves' int32 sums are added
// through LDS, exactly, in any order.
template <int MT, int NT, int W>
__global__ __launch_bounds__(64 * W, 1) void gemm_rows_kernel(GemmArgs a) {
    __shared__ i32x4 part[W][MT * NT][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int n0 = (int)blockIdx.x * 16 * NT, m0 = (int)blockIdx.y * 16 * MT;
    const uint32_t xbytes = (uint32_t)((int64_t)a.rows * a.in);
    const uint32_t wbytes = (uint32_t)((int64_t)a.out * a.in);
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(a.x, xbytes);
    const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(a.w, wbytes);
    uint32_t woff[NT], xoff[MT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int n = n0 + 16 * j + col;
        woff[j] = n < a.out ? (uint32_t)((int64_t)n * a.in + 16 * grp) : wbytes;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = m0 + 16 * i + col;
        xoff[i] = m < a.rows ? (uint32_t)((int64_t)m * a.in + 16 * grp) : xbytes;
    }
    const int units = (a.in + kBK - 1) / kBK;
    struct Unit {
        i32x4 w[2][NT], x[2][MT];
    };
    // Unit k; chunks past `in` read zeros. The range check compares a lane's offset with the
    // buffer's size less the scalar offset, so that one stays inside a row: the units past
    // the last and the upper half of a partial one would carry it past the end of a buffer
    // of one row (only offsets past `in` move: lanes inside it imply k0 <= in - 16).
    auto load = [&](Unit &u, int k) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int k0 = k * kBK + 64 * half, at = min(k0, a.in - 16);
            const bool in_k = k0 + 16 * grp < a.in;
#pragma unroll
            for (int j = 0; j < NT; ++j)
                u.w[half][j] = __builtin_bit_cast(
                    i32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, in_k ? woff[j] : wbytes, at, 0));
#pragma unroll
            for (int i = 0; i < MT; ++i)
                u.x[half][i] = __builtin_bit_cast(
                    i32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, in_k ? xoff[i] : xbytes, at, 0));
        }
    };
    i32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = i32x4{};
    auto multiply = [&](const Unit &u) {
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = mfma_16x16x64_i8(u.w[half][j], u.x[half][i], acc[i][j]);
    };
    if (wave < units) {
        Unit u0, u1;
        load(u0, wave);
        int k = wave;
        for (; k + W < units; k += 2 * W) {
            load(u1, k + W);
            multiply(u0);
            load(u0, k + 2 * W);  // past the last unit: zeros
            multiply(u1);
        }
        if (k < units) multiply(u0);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) part[wave][i * NT + j][lane] = acc[i][j];
    __syncthreads();
    bool bad = false;
    for (int b = wave; b < MT * NT; b += W) {
        i32x4 sum = part[0][b][lane];
#pragma unroll
        for (int w = 1; w < W; ++w) sum += part[w][b][lane];
        const int m = m0 + 16 * (b / NT) + col, n = n0 + 16 * (b % NT) + 4 * grp;
        float ws[4], bias[4];
        load_columns(a, n, ws, bias);
        bad |= store_block(a, m, n, m < a.rows ? a.xs[m] : 0.0f, ws, bias, sum);
    }
    if (bad) flag_status(a.status, REEF_STATUS_BIT_OVERFLOW);
}

template <int BM, int BN, int WM, int WN, int ST>
void launch_tiles(GemmArgs &a, hipStream_t stream) {
    a.m_tiles = (int32_t)ceil_div(a.rows, BM);
    a.n_tiles = (int32_t)ceil_div(a.out, BN);
    hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WM, WN, ST>),
                       dim3((unsigned)(a.m_tiles * a.n_tiles)), dim3(64 * WM * WN), 0, stream, a);
}

template <int MT, int NT, int W>
void launch_rows_kernel(const GemmArgs &a, hipStream_t stream) {
    hipLaunchKernelGGL((gemm_rows_kernel<MT, NT, W>),
                       dim3((unsigned)ceil_div(a.out, 16 * NT), (unsigned)ceil_div(a.rows, 16 * MT)),
                       dim3(64 * W), 0, stream, a);
}

// Tiles of BM x BN with WM x WN waves, and the time of one K step (128 bytes) of a
// workgroup when every compute unit has one, in ns (8192 x 8192 -> 8192 and
// 4096 x 8192 -> 1280 among others). The larger the tile, the fewer operand bytes per
// product; the smaller, the more units a small output occupies (64 x 4096 -> 6144: 10.1 us
// in 192 tiles of 64 x 32, 11.4 in 96 of 64 x 64). A call takes the tile
// with the least rounds x step time, rounds = ceil(tiles / units).
struct TileChoice {
    int32_t bm, bn, step_ns;
    void (*launch)(GemmArgs &, hipStream_t);
};
const TileChoice kTiles[] = {
    {256, 256, 1880, launch_tiles<256, 256, 2, 4, 2>}, {256, 192, 1600, launch_tiles<256, 192, 4, 2, 2>},
    {256, 128, 970, launch_tiles<256, 128, 4, 2, 3>},  {128, 160, 690, launch_tiles<128, 160, 4, 2, 4>},
    {128, 128, 610, launch_tiles<128, 128, 2, 4, 5>},  {128, 64, 410, launch_tiles<128, 64, 2, 2, 6>},
    {64, 64, 300, launch_tiles<64, 64, 2, 2, 8>},      {64, 32, 240, launch_tiles<64, 32, 2, 2, 10>},
};

reef_status launch_gemm(const int8_t *xq, const float *xs, int64_t rows, int64_t in,
                        const int8_t *w, const float *ws, const float *bias, int64_t out,
                        float *y, int64_t y_stride, uint32_t *status, hipStream_t stream) {
    GemmArgs a;
    a.x = xq;
    a.xs = xs;
    a.w = w;
    a.ws = ws;
    a.bias = bias;
    a.y = y;
    a.y_stride = y_stride;
    a.rows = (int32_t)rows;
    a.in = (int32_t)in;
    a.out = (int32_t)out;
    a.m_tiles = a.n_tiles = 0;
    a.y_vec = aligned(y, 16) && y_stride % 4 == 0;
    a.status = status;
    const int64_t cus = compute_units();
    // Few rows and features: while 16-feature workgroups with 16 or 32 rows each fit the
    // units at once, every wave's share of K is short and a tile's serial K loop is not
    // (32 rows, 8192 -> 1280: 9.9 us against 14.8 in tiles; 64 rows, 4096 -> 512: 6.5
    // against 9.4). At most 16 rows take 32 features per workgroup up to three quarters of
    // the units (4 rows, 2048 -> 6144: 5.4 against 6.5; 8 rows, 8192 -> 6144: 13.8 against
    // 15.1; 16 rows, 4096 -> 6144: 9.1 against 9.3). With more features it is 4 to 6 %
    // faster at 4096 values a row and 12 % slower at 8192 (-> 8192: 9.0 against 9.6 and 18.0
    // against 16.0), and past one workgroup a unit slower (4096 -> 11008: 15.2 against 11.3).
    const int64_t nb = ceil_div(out, 16);
    if (ceil_div(rows, 16) * nb <= cus) {
        launch_rows_kernel<1, 1, 8>(a, stream);
    } else if (ceil_div(rows, 32) * nb <= cus) {
        launch_rows_kernel<2, 1, 8>(a, stream);
    } else if (rows <= 16 && 4 * ceil_div(out, 32) <= 3 * cus) {
        launch_rows_kernel<1, 2, 8>(a, stream);
    } else {
        const TileChoice *best = nullptr;
        int64_t least = 0;
        for (const TileChoice &t : kTiles) {
            const int64_t cost = ceil_div(ceil_div(rows, t.bm) * ceil_div(out, t.bn), cus) * t.step_ns;
            if (!best || cost < least) {
                best = &t;
                least = cost;
            }
        }
        best->launch(a, stream);
    }
    return launch_status();
}

reef_status validate_gemm(const void *x, const float *xs, int64_t rows, int64_t in,
                          const int8_t *w, const float *ws, int64_t out, float *y,
                          int64_t y_stride) {
    if (!x || !xs || !w || !ws || !y || rows <= 0 || in <= 0 || out <= 0 || y_stride < out)
        return REEF_INVALID_ARGUMENT;
    if (in % 16 != 0 || !aligned(w, 16)) return REEF_UNSUPPORTED;
    if (rows * in >= (int64_t(1) << 31) || out * in >= (int64_t(1) << 31) ||
        ceil_div(rows, 128) * ceil_div(out, 128) >= (int64_t(1) << 31))
        return REEF_UNSUPPORTED;
    return REEF_OK;
}

}  // namespace
}  // namespace reef

using namespace reef;

extern "C" size_t reef_linear_w8a8_workspace_bytes(int64_t rows, int64_t in_features) {
    if (rows <= 0 || in_features <= 0) return 0;
    // quantized rows (16-byte aligned), then one scale per row
    return (size_t)(ceil_div(rows * in_features, 16) * 16 + rows * 4);
}

extern "C" reef_status reef_gemm_w8a8(const int8_t *xq, const float *x_scales, int64_t rows,
                                      int64_t in_features, const int8_t *weight,
                                      const float *w_scales, const float *bias,
                                      int64_t out_features, float *y, int64_t y_row_stride,
                                      uint32_t *status_word, hipStream_t stream) {
    const reef_status s = validate_gemm(xq, x_scales, rows, in_features, weight, w_scales,
                                        out_features, y, y_row_stride);
    if (s != REEF_OK) return s;
    if (!aligned(xq, 16)) return REEF_UNSUPPORTED;
    return launch_gemm(xq, x_scales, rows, in_features, weight, w_scales, bias, out_features, y,
                       y_row_stride, status_word, stream);
}

extern "C" reef_status reef_linear_w8a8(const float *x, int64_t rows, int64_t in_features,
                                        int64_t x_row_stride, const int8_t *weight,
                                        const float *w_scales, const float *bias,
                                        int64_t out_features, float *y, int64_t y_row_stride,
                                        void *workspace, size_t workspace_bytes,
                                        uint32_t *status_word, hipStream_t stream) {
    reef_status s = validate_gemm(x, w_scales, rows, in_features, weight, w_scales, out_features,
                                  y, y_row_stride);
    if (s != REEF_OK) return s;
    if (!workspace || !aligned(workspace, 16) ||
        workspace_bytes < reef_linear_w8a8_workspace_bytes(rows, in_features))
        return REEF_INVALID_ARGUMENT;
    int8_t *xq = static_cast<int8_t *>(workspace);
    float *xs = reinterpret_cast<float *>(xq + ceil_div(rows * in_features, 16) * 16);
    s = reef_quantize_int8_per_token(x, rows, in_features, x_row_stride, xq, xs, status_word,
                                     stream);
    if (s != REEF_OK) return s;
    return launch_gemm(xq, xs, rows, in_features, weight, w_scales, bias, out_features, y,
                       y_row_stride, status_word, stream);
}
