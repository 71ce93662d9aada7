// Quantised weights times several f32 vectors on gfx950's bf16 matrix cores:
// prompt prefill (qmm.matMulQ8_0's role, qmm.zig:58-138) and the MoE experts
// of a batch grouped by expert (moeFFN over forwardBatch's tokens,
// inference.zig:346-351, 886-1188; gate, up and silu(gate) * up in one launch).
//
// The integer weights of both formats (int8 codes; grid magnitudes with their
// signs) are exact in bf16, and a vector element is two bf16 numbers
// (split_bf16), so a 32-column block of 16 weight rows times 16 vectors is two
// v_mfma_f32_16x16x32_bf16 and one multiply-add per output with the block's
// scale. Int8 digit planes need four vector instructions per output and block
// (combine the digits, convert, scale twice), and their quantisation is a
// launch of its own.
//
// Bound: vector instructions (per block 64 for the split of 32 vectors, 48 for
// four tiles of int8 -> bf16, 32 for the sums), then the launch's fixed cost.
// A workgroup's waves split the columns of one tile, so no wave waits for
// another before the sums: each reads its vectors in whole rows (16-byte loads
// straight into the operand layout took 64 address cycles each, [768 x 2048]
// times 32: 16.7 us against 12.9), splits them and turns them into operands
// through LDS of its own, and reads weights as the record layout has them.
// Four projections of a layer (768 / 3840 / 576 / 2048 rows): Q8_0 at 256
// tokens 83.7 -> 45.6 us, IQ2_XXS at 77 tokens 54.1 -> 34.6 us. Q8_0 MoE layer
// (64 experts of 1536 and a shared one, hidden 2048) at 256 tokens 405 -> 184
// us, there between the vector instructions (half of the launch) and the L2's
// traffic (12 TB/s: every item reads its weights again).
#include "device_common.hpp"
#include "gemm_tile_ops.hpp"
#include "kernels.hpp"

namespace mmhip {

namespace {

// Waves of a workgroup split the columns: wave v takes the v-th share of the
// tile's column turns and the shares are added at the end. Four waves per SIMD
// (128 registers) where a wave holds 16 rows of x; 32 need 192 and more.
// Experts: the items of a.work over packed rows; gate/up leaves packed rows too.
template <int FMT, int MT, int NJ, int KS, bool GU, bool EXPERTS>
__global__ __launch_bounds__(KS * 64, MT == 1 ? 4 : 2) void gemm_tile_kernel(GemmTileArgs a) {
    // The waves' activation copies and the IQ2_XXS tables, then the sums.
    constexpr uint32_t kSlot = MT * NJ * 4 * 64;  // floats of a wave's sums
    constexpr uint32_t kRed = KS / 2 * kSlot * 4, kX = tile_lds_bytes<MT>();
    constexpr uint32_t kMain = KS * kX + (FMT == kFmtIq2 ? kIq2BfWords * 4 : 0);
    __shared__ __align__(16) uint8_t lds[kRed > kMain ? kRed : kMain];
    uint32_t* const tab = reinterpret_cast<uint32_t*>(lds + KS * kX);

    // Block b: one of eight consecutive blocks per XCD. Tile group tg always
    // runs on XCD tg % 8, so each XCD's L2 holds one eighth of a matrix for all
    // of its items.
    const uint32_t xcd = blockIdx.x & 7, r8 = blockIdx.x >> 3;
    uint32_t item, tg;
    if (EXPERTS) {  // item-major: the items of one expert follow each other
        item = r8 / a.groups8;
        tg = (r8 % a.groups8) * 8 + xcd;
    } else {
        item = r8 % a.n_items;
        tg = (r8 / a.n_items) * 8 + xcd;
    }
    if (tg >= a.groups) return;  // whole workgroup

    uint32_t first, count;
    uint64_t mat, mat2;
    if (EXPERTS) {
        // The count and the item in one round trip (the grid stays within
        // the list).
        uint32_t n_work = *a.n_work;
        QmmWork w = a.work[item];
        asm volatile("" : "+s"(n_work), "+s"(w.mat), "+s"(w.slot), "+s"(w.count), "+s"(w.pad));
        if (item >= n_work) return;
        first = w.slot;
        count = w.count;
        mat = w.mat;
        mat2 = w.pad;
    } else {
        first = item * (MT * 16);
        count = min(a.batch - first, MT * 16u);
        mat = a.mat;
        mat2 = a.mat + 1;
    }

    const uint32_t lane = threadIdx.x & 63;
    const uint32_t n = lane & 15, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    if (FMT == kFmtIq2) iq2_bf_table_load<KS * 64>(tab);

    f32x4 acc[MT][NJ];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[m][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    TileStream<FMT, MT, NJ, GU, EXPERTS> st;
    st.init_w(a, mat, mat2, tg, lane);
    uint8_t* const xs = lds + wave * kX;
    const uint32_t s0 = a.turns * wave / KS, s1 = a.turns * (wave + 1) / KS;
    if (s0 < s1) {
        // The weights first: the rows of x wait for their list.
        st.load_d(s0, s1);
        st.load_w(s0, s1, 0);
        if (FMT == kFmtQ8) st.load_w(s0, s1, 1);
    }
    st.init_x(a, first, count, lane);
    if (s0 < s1) {
        st.load_x(s0, s1, 0);
        st.load_x(s0, s1, 1);
    }
    if (FMT == kFmtIq2) lds_barrier();
    for (uint32_t s = s0; s < s1; ++s) {
        float c[4][4];
        st.scales(c);
        st.load_d(s + 1, s1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            st.stage(h, xs);
            st.load_x(s + 1, s1, h);
            wave_lds_order();
            st.products(h, xs, tab, c, acc);
            wave_lds_order();
            if (FMT == kFmtQ8 || h == 1) st.load_w(s + 1, s1, h);
        }
    }

    // Sum of the waves' shares: the upper half of the waves hands over to the
    // lower half, which hands its sums to whoever stores them.
    lds_barrier();  // the sums take the memory over
    float* red = reinterpret_cast<float*>(lds);
    float* mine = red + (wave % (KS / 2)) * kSlot + lane;
    if (wave >= KS / 2) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) mine[((m * NJ + j) * 4 + r) * 64] = acc[m][j][r];
    }
    lds_barrier();
    if (wave < KS / 2) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) mine[((m * NJ + j) * 4 + r) * 64] += acc[m][j][r];
    }
    lds_barrier();
    auto sum = [&](uint32_t m, uint32_t j, uint32_t r) {
        const float* p = red + ((m * NJ + j) * 4 + r) * 64 + lane;
        float v = p[0];
#pragma unroll
        for (int k = 1; k < KS / 2; ++k) v += p[k * kSlot];
        return v;
    };
    constexpr uint32_t kOut = GU ? NJ / 2 : NJ;
    for (uint32_t e = wave; e < MT * kOut; e += KS) {
        const uint32_t m = e / kOut, j = e % kOut;
        const uint32_t row = (tg * kOut + j) * 16 + n;
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
            float v = sum(m, j, r);
            // expertFFN's activation (inference.zig:1179-1180).
            if (GU) v = silu(v) * sum(m, j + kOut, r);
            const uint32_t t = m * 16 + 4 * g + r;
            if (t >= count || row >= a.rows) continue;
            float* const out = a.y + (uint64_t)(first + t) * a.y_slot;
            if (GU && EXPERTS)
                pack_row(out, a.rows, row, v);
            else
                out[(uint64_t)row * a.y_row] = v;
        }
    }
}

// A launch's tile: 16 mt rows of x by 16 nj weight rows per workgroup of ks
// waves.
struct TileShape {
    int mt, nj, ks;
};

template <int FMT, bool GU>
const void* dense_fn(const TileShape& t) {
    if (t.mt == 1)
        return t.nj == 2 ? reinterpret_cast<const void*>(&gemm_tile_kernel<FMT, 1, 2, 8, GU, false>)
                         : reinterpret_cast<const void*>(&gemm_tile_kernel<FMT, 1, 4, 8, GU, false>);
    return t.ks == 8 ? reinterpret_cast<const void*>(&gemm_tile_kernel<FMT, 2, 4, 8, GU, false>)
                     : reinterpret_cast<const void*>(&gemm_tile_kernel<FMT, 2, 4, 4, GU, false>);
}
template <int FMT, bool GU>
const void* experts_fn(const TileShape& t) {
    return t.nj == 2 ? reinterpret_cast<const void*>(&gemm_tile_kernel<FMT, 1, 2, 4, GU, true>)
                     : reinterpret_cast<const void*>(&gemm_tile_kernel<FMT, 1, 4, 4, GU, true>);
}
template <bool GU>
const void* tile_fn(uint32_t fmt, bool experts, const TileShape& t) {
    if (fmt == kFmtIq2) return experts ? experts_fn<kFmtIq2, GU>(t) : dense_fn<kFmtIq2, GU>(t);
    return experts ? experts_fn<kFmtQ8, GU>(t) : dense_fn<kFmtQ8, GU>(t);
}

uint32_t groups_of(uint32_t tiles, bool gu, const TileShape& t) {
    const uint32_t per = gu ? t.nj / 2 : t.nj;
    return (tiles + per - 1) / per;
}

// Dense launches. A workgroup's time is its column turns' conversions and
// products, so the smallest tile whose workgroups all run at once (one per
// CU) ends first; past one per CU a larger tile costs less than a second
// round, and four waves let two workgroups share a CU. Measured, us with tiles
// 16x32 / 16x64 / 32x64 by eight waves / 32x64 by four: Q8_0 [2048 x 2560]
// times 64 rows 8.1 / 10.1 / 14.8 / 15.2, [3840 x 768] times 48 6.2 / 5.8 /
// 7.7 / 8.7, [1536 x 2048] times 256 12.9 / 15.2 / 11.9 / 13.1, [3840 x 768]
// times 256 16.7 / 18.0 / 14.3 / 11.3; IQ2_XXS [8192 x 4096] times 48 21.2 /
// 25.4 / 20.3 / 26.2, times 256 97.6 / 96.8 / 75.4 / 65.8.
TileShape dense_shape(uint32_t tiles, bool gu, uint32_t batch, int num_cu) {
    const TileShape shapes[4] = {{1, 2, 8}, {1, 4, 8}, {2, 4, 8}, {2, 4, 4}};
    for (int i = 0; i < 3; ++i) {
        const uint64_t items = (batch + shapes[i].mt * 16 - 1) / (shapes[i].mt * 16);
        if (groups_of(tiles, gu, shapes[i]) * items <= (uint64_t)num_cu) return shapes[i];
    }
    return shapes[3];
}

hipError_t launch(GemmTileArgs& a, uint32_t fmt, bool gu, const TileShape& t, uint32_t items, hipStream_t s) {
    if (items == 0 || a.tiles == 0) return hipSuccess;
    a.groups = groups_of(a.tiles, gu, t);
    a.groups8 = (a.groups + 7) / 8;
    a.n_items = items;
    const uint64_t blocks = (uint64_t)a.groups8 * items * 8;
    if (blocks > 0x7FFFFFFFu) return hipErrorInvalidValue;
    const bool experts = a.work != nullptr;
    const void* fn = gu ? tile_fn<true>(fmt, experts, t) : tile_fn<false>(fmt, experts, t);
    void* args[] = {&a};
    return hipLaunchKernel(fn, dim3((unsigned)blocks), dim3(t.ks * 64), args, 0, s);
}

GemmTileArgs base(const uint4* recs, const uint16_t* dvals, const TileGeom& g, const float* x, uint64_t x_stride,
                  uint64_t x_rows, float* y) {
    GemmTileArgs a{};
    a.recs = recs;
    a.dvals = dvals;
    a.rec_stride = g.rec_stride;
    a.d_stride = g.d_stride;
    a.d_row = (uint32_t)g.d_row;
    a.x = x;
    a.x_stride = (uint32_t)x_stride;
    a.x_bytes = (uint32_t)(((x_rows - 1) * x_stride + g.cols) * 4);
    a.cols = (uint32_t)g.cols;
    a.turns = (uint32_t)((g.cols + kTileTurn - 1) / kTileTurn);
    a.y = y;
    a.tiles = (uint32_t)g.tiles;
    a.units = (uint32_t)g.units;
    a.rows = (uint32_t)g.rows;
    return a;
}

}  // namespace

bool gemm_tile_fits(const TileGeom& g, uint64_t x_rows, uint64_t x_stride) {
    if (g.cols % 32 || x_rows == 0 || x_stride < g.cols || x_rows > 0x7FFFFFFFu / 4 / x_stride) return false;
    // A launch of 2^32 threads or more does not run: the largest dense calls are
    // 32x64 tiles of 256 threads (3.4e10 results, 137 GB).
    return (g.tiles / 4 + 8) * ((x_rows + 31) / 32) < 1u << 24;
}

hipError_t launch_gemm_tile(const uint4* recs, const uint16_t* dvals, const TileGeom& g, uint64_t mat, bool gate_up,
                            const float* x, uint64_t x_stride, uint32_t batch, float* y, uint64_t y_slot,
                            uint64_t y_row, int num_cu, hipStream_t s) {
    if (batch == 0) return hipSuccess;
    if (!gemm_tile_fits(g, batch, x_stride)) return hipErrorInvalidValue;
    GemmTileArgs a = base(recs, dvals, g, x, x_stride, batch, y);
    a.mat = mat;
    a.batch = batch;
    a.y_slot = y_slot;
    a.y_row = y_row;
    const TileShape t = dense_shape(a.tiles, gate_up, batch, num_cu > 0 ? num_cu : 256);
    return launch(a, g.fmt, gate_up, t, (batch + t.mt * 16 - 1) / (t.mt * 16), s);
}

hipError_t launch_gemm_tile_experts(const uint4* recs, const uint16_t* dvals, const TileGeom& g, bool gate_up,
                                    const float* x, uint64_t x_stride, uint64_t x_rows, const uint32_t* x_row,
                                    const QmmWork* work, const uint32_t* n_work, uint32_t max_work, uint32_t n_tokens, float* y,
                                    uint64_t y_slot, hipStream_t s) {
    if (!gemm_tile_fits(g, x_rows, x_stride)) return hipErrorInvalidValue;
    GemmTileArgs a = base(recs, dvals, g, x, x_stride, x_rows, y);
    a.x_row = x_row;
    a.work = work;
    a.n_work = n_work;
    a.y_slot = y_slot;
    a.y_row = 1;
    // Items of 16 rows and four waves: the many short workgroups need the CU's
    // other workgroups to cover their start and end (four a CU; 32-row items
    // leave room for two and halve the weights' conversions, the same 190 us for
    // the Q8_0 layer above at 256 tokens and 103 against 91 at 64). A call of few
    // tokens has few items: half tiles give it twice the workgroups (Q8_0 2
    // tokens 32.3 us against 34.8, 16 tokens 50.6 against 55.7, 64 tokens 101.5
    // against 90.6; IQ2_XXS 2 tokens 32.5 against 35.7, 12 tokens 43.7 against
    // 41.9).
    const uint32_t few = g.fmt == kFmtIq2 ? 8 : 16;
    return launch(a, g.fmt, gate_up, TileShape{1, n_tokens <= few ? 2 : 4, 4}, max_work, s);
}

}  // namespace mmhip
