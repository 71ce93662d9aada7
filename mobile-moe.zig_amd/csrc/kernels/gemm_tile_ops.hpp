// Per-wave pieces of the bf16 matrix-core products of gemm_tile.hip: the
// loads of one column step, its operands and its sums.
#pragma once

#include "device_common.hpp"
#include "kernels.hpp"

namespace mmhip {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Columns of one turn of a wave's loop: two Q8_0 record units, or half an
// IQ2_XXS record unit (four sub-blocks; a lane's first or last two dwords,
// which also carry those sub-blocks' scales). A turn is two halves of 64.
constexpr uint32_t kTileTurn = 128;

struct GemmTileArgs {
    const uint4* recs;
    const uint16_t* dvals;
    uint64_t rec_stride, d_stride;
    uint32_t d_row;
    const float* x;
    uint32_t x_stride;              // floats between rows
    uint32_t x_bytes;               // readable bytes of x (< 2^31)
    const uint32_t* x_row;          // slot -> row of x (grouped), or null
    float* y;
    uint64_t y_slot, y_row;         // y[slot * y_slot + row * y_row]
    const QmmWork* work;            // grouped when non-null; pad = the up matrix (gate/up)
    const uint32_t* n_work;
    uint64_t mat;                   // dense: matrix (gate/up: gate, up = mat + 1)
    uint32_t batch;                 // dense: rows of x
    uint32_t cols, turns, tiles, units, rows;
    uint32_t groups, groups8, n_items;  // set by the launch
};

// Activations enter the products times 2^-12, so that a block's 32 products of at
// most 128 x (a code of -128) stay within f32 for every finite x: their sum
// reaches 2^128 only where the first parts round up to it, and there the second
// parts, which are summed before them, have the other sign. The weight scales
// carry the 2^12.
constexpr float kActScale = 0x1p-12f, kActUnscale = 0x1p12f;

// Four f32 values as two times four bf16: the nearest bf16 and the nearest
// bf16 to what is left, 16 bits of significand and more (error at most 2^-17
// of the value, down to values of 2^-105; below, where the second part is a
// subnormal number, at most 2^-122; the int8 digit planes give 2^-16 of the
// block's largest and zeros for blocks below 2^-100). An
// infinity leaves a NaN in the second part: it poisons its row's outputs, as a
// NaN does.
__device__ __forceinline__ void split_bf16(const uint4& q, uint2& hi, uint2& lo) {
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    uint32_t h[2], l[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const f32x2 v = {__uint_as_float(w[2 * i]) * kActScale, __uint_as_float(w[2 * i + 1]) * kActScale};
        h[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
        const f32x2 d = {v[0] - __uint_as_float(h[i] << 16), v[1] - __uint_as_float(h[i] & 0xFFFF0000u)};
        l[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(d, bf16x2));
    }
    hi = make_uint2(h[0], h[1]);
    lo = make_uint2(l[0], l[1]);
}

// A packed row of `cols` values takes the bytes of its f32 row: cols bf16 of
// the first parts, then cols bf16 of the second.
__device__ __forceinline__ void pack_row(float* row, uint32_t cols, uint32_t col, float v) {
    const f32x2 p = {v * kActScale, 0.0f};
    const uint16_t h = (uint16_t)__builtin_bit_cast(uint32_t, __builtin_convertvector(p, bf16x2));
    const f32x2 d = {p[0] - __uint_as_float((uint32_t)h << 16), 0.0f};
    uint16_t* r16 = reinterpret_cast<uint16_t*>(row);
    r16[col] = h;
    r16[cols + col] = (uint16_t)__builtin_bit_cast(uint32_t, __builtin_convertvector(d, bf16x2));
}

// Eight int8 weights as bf16 (exact: at most eight significant bits). The
// conversions leave zeros below the upper half, which v_perm_b32 picks.
__device__ __forceinline__ bf16x8 q8_bop(uint32_t w0, uint32_t w1) {
    uint32_t b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = i < 2 ? w0 : w1;
        const float f0 = (float)(int8_t)(w >> (16 * (i & 1))), f1 = (float)(int8_t)(w >> (16 * (i & 1) + 8));
        b[i] = __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
    }
    return __builtin_bit_cast(bf16x8, make_uint4(b[0], b[1], b[2], b[3]));
}

// IQ2_XXS operand tables (4.5 KiB): entry idx of the grid as eight bf16
// magnitudes, then for each of 128 sign keys (b012 | P << 3 | hi3 << 4 of the
// record, device_common.hpp) the eight signs in one word: columns 2 c and
// 2 c + 1 at bits 15 - c and 31 - c, a shift by c away from their bf16 sign bits
// (a second 16-byte read per record instead of the shifts: the IQ2_XXS experts
// below were LDS bound).
constexpr uint32_t kIq2BfGridWords = 256 * 4, kIq2BfWords = kIq2BfGridWords + 128;
struct Iq2BfTables {
    uint32_t w[kIq2BfWords];
};
constexpr uint32_t small_bf16(uint32_t v) {  // 8, 25, 43
    return v == 8 ? 0x4100u : v == 25 ? 0x41C8u : 0x422Cu;
}
constexpr Iq2BfTables make_iq2_bf_tables() {
    Iq2BfTables t{};
    for (uint32_t e = 0; e < 256; ++e)
        for (uint32_t c = 0; c < 4; ++c)
            t.w[e * 4 + c] = small_bf16((uint32_t)(kIq2Grid[e] >> (16 * c)) & 0xFFu) |
                             small_bf16((uint32_t)(kIq2Grid[e] >> (16 * c + 8)) & 0xFFu) << 16;
    for (uint32_t k = 0; k < 128; ++k) {
        const uint32_t b012 = k & 7u, par = (k >> 3) & 1u, h = k >> 4;
        const uint32_t s = b012 | ((par ^ parity3(b012)) << 3) | (h << 4) | ((par ^ parity3(h)) << 7);
        for (uint32_t c = 0; c < 4; ++c)
            t.w[kIq2BfGridWords + k] |= ((s >> (2 * c)) & 1u) << (15 - c) | ((s >> (2 * c + 1)) & 1u) << (31 - c);
    }
    return t;
}
static __constant__ Iq2BfTables c_iq2_bf = make_iq2_bf_tables();

template <int WG>
__device__ __forceinline__ void iq2_bf_table_load(uint32_t* tab) {
    const uint4* src = reinterpret_cast<const uint4*>(c_iq2_bf.w);
    for (uint32_t i = threadIdx.x; i < kIq2BfWords / 4; i += WG) reinterpret_cast<uint4*>(tab)[i] = src[i];
}

__device__ __forceinline__ bf16x8 iq2_bop_bf16(uint32_t grid_off, uint32_t sign_off, const uint32_t* tab) {
    const char* t = reinterpret_cast<const char*>(tab);
    const uint4 m = *reinterpret_cast<const uint4*>(t + grid_off);
    const uint32_t s = *reinterpret_cast<const uint32_t*>(t + kIq2BfGridWords * 4 + sign_off);
    constexpr uint32_t k = 0x80008000u;
    return __builtin_bit_cast(bf16x8, make_uint4(m.x ^ (s & k), m.y ^ ((s << 1) & k), m.z ^ ((s << 2) & k),
                                                 m.w ^ ((s << 3) & k)));
}

// A wave's LDS copy of one half turn of its activations, as the products read
// it: per 16 rows and plane eight runs (block b, column group g), each the 16
// rows' eight columns. Runs are 272 bytes apart: the 8-byte writes (16 lanes
// to a row) would otherwise all meet in four banks.
constexpr uint32_t kRunBytes = 16 * 16 + 16;
constexpr uint32_t kPlaneBytes = 8 * kRunBytes;
template <int MT>
constexpr uint32_t tile_lds_bytes() { return MT * 2 * kPlaneBytes; }

// Orders a wave's LDS writes before its other lanes' reads (and reads before
// the next writes). The LDS serves a wave in order: nothing to wait for.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// v of lane 16 j + n, for j = 0..3, in every lane (n, g).
__device__ __forceinline__ void broadcast_rows4(float v, float (&out)[4]) {
    const uint32_t u = __float_as_uint(v);
    const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);        // rows (0,1,0,1), (2,3,2,3)
    const auto a = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);  // rows 0, 1
    const auto b = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);  // rows 2, 3
    out[0] = __uint_as_float(a[0]);
    out[1] = __uint_as_float(a[1]);
    out[2] = __uint_as_float(b[0]);
    out[3] = __uint_as_float(b[1]);
}

// NJ 16-row weight tiles per wave; GU: the first half gate tiles, the others
// the up tiles of the same rows.
// PACKED: x rows hold two bf16 planes (pack_row) instead of f32 values.
template <int FMT, int MT, int NJ, bool GU, bool PACKED>
struct TileStream {
    static constexpr uint32_t kRowTiles = GU ? NJ / 2 : NJ;
    // Loads in flight: both halves' activations (lane l: f32 rows 4 i + l / 16,
    // columns 4 (l % 16) .. + 3; packed plane i % 2 of rows 8 (i / 2) + l / 8,
    // columns 8 (l % 8) .. + 7) and weights of a turn, and the scales of the
    // wave's 64 weight rows (lane l: row l).
    uint4 x[2][MT * 4];
    uint4 q8[2][FMT == kFmtQ8 ? NJ : 1];
    uint2 iq[FMT == kFmtIq2 ? NJ : 1];
    uint2 d;

    BufRsrc x_r, rec_r, rec2_r;
    const uint16_t* d_lane;
    static constexpr uint32_t kRowLanes = PACKED ? 8 : 16;
    static constexpr int kXRows = PACKED ? MT * 2 : MT * 4;
    uint32_t x_voff[kXRows];
    uint32_t rec_voff, col_lane, tile0, tiles, units, cols;

    __device__ __forceinline__ void init_w(const GemmTileArgs& a, uint64_t mat, uint64_t mat2, uint32_t tg,
                                           uint32_t lane) {
        rec_r = make_rsrc(a.recs + mat * a.rec_stride, (uint32_t)(a.rec_stride * 16));
        if (GU) rec2_r = make_rsrc(a.recs + mat2 * a.rec_stride, (uint32_t)(a.rec_stride * 16));
        rec_voff = lane * 16;
        tile0 = tg * kRowTiles;
        tiles = a.tiles;
        units = a.units;
        // Tiles past the matrix read its last tile's scales (their weights
        // read as zeros).
        const uint32_t j = min(lane >> 4, NJ - 1u);
        const uint32_t t = min(tile0 + j % kRowTiles, tiles - 1);
        d_lane = a.dvals + (j >= kRowTiles ? mat2 : mat) * a.d_stride + (uint64_t)(t * 16 + (lane & 15)) * a.d_row;
    }
    __device__ __forceinline__ void init_x(const GemmTileArgs& a, uint32_t first, uint32_t count, uint32_t lane) {
        x_r = make_rsrc(a.x, a.x_bytes);
        col_lane = lane % kRowLanes * (64 / kRowLanes);
        cols = a.cols;
        // Rows past the item read zeros (no memory access).
#pragma unroll
        for (int i = 0; i < kXRows; ++i) {
            const uint32_t j = 64 / kRowLanes * i + lane / kRowLanes;
            const bool ok = j < count;
            uint32_t row = first + (ok ? j : 0);
            if (a.x_row) row = a.x_row[row];
            x_voff[i] = ok ? row * (a.x_stride * 4) + lane % kRowLanes * 16 : kBufOob;
        }
    }

    // Half h of turn s; a turn at or past `end` loads nothing (zeros, no
    // memory access).
    __device__ __forceinline__ void load_x(uint32_t s, uint32_t end, int h) {
        const uint32_t col = s * kTileTurn + 64 * h;
        const bool in = s < end && col + col_lane < cols;
#pragma unroll
        for (int i = 0; i < MT * 4; ++i) {
            if constexpr (PACKED)
                x[h][i] = buf_load_b128(x_r, in ? x_voff[i >> 1] : kBufOob, col * 2 + (i & 1) * (cols * 2));
            else
                x[h][i] = buf_load_b128(x_r, in ? x_voff[i] : kBufOob, col * 4);
        }
    }
    __device__ __forceinline__ void load_w(uint32_t s, uint32_t end, int h) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const uint32_t t = tile0 + j % kRowTiles;
            const bool ok = s < end && t < tiles;
            const BufRsrc rr = j >= (int)kRowTiles ? rec2_r : rec_r;
            if constexpr (FMT == kFmtIq2) {
                iq[j] = buf_load_b64(rr, rec_voff, ok ? (t * units + (s >> 1)) * 1024 + 8 * (s & 1) : kBufOob);
            } else {
                const uint32_t u = 2 * s + h;
                q8[h][j] = buf_load_b128(rr, rec_voff, ok && u < units ? (t * units + u) * 1024 : kBufOob);
            }
        }
    }
    __device__ __forceinline__ void load_d(uint32_t s, uint32_t end) {
        s = min(s, end - 1);
        if constexpr (FMT == kFmtIq2)
            d.x = d_lane[s >> 1];
        else
            d = *reinterpret_cast<const uint2*>(d_lane + 4 * s);  // rows hold a multiple of 8 scales
    }

    // The turn's weight scales: lane (n, g) gets c[b][j] for block b of
    // weight row n of tile j. Uses d (and, IQ2_XXS, the records in iq).
    __device__ __forceinline__ void scales(float (&c)[4][4]) const {
        if constexpr (FMT == kFmtIq2) {
            const uint32_t g = (threadIdx.x & 63) >> 4;
            // (0.5 + ls) / 4 = (2 ls + 1) / 8 of the row's scale (dequant.zig:336),
            // as one product: ls (2 / 8) + 1 / 8 is a NaN for an infinite
            // scale and ls = 0.
            float d8[4];
            broadcast_rows4(f16_scale((uint16_t)d.x) * (0.125f * kActUnscale), d8);
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                // Byte b: 2 ls + 1 of sub-block b of the half unit, gathered
                // from the row's four lane groups.
                const uint32_t ls2 = ((iq[j].x >> 29) & 6u) | ((iq[j].y >> 27) & 0x18u) | 1u;
                const uint32_t mine = ls2 << (8 * g);
                const auto p = __builtin_amdgcn_permlane16_swap(mine, mine, false, false);
                const uint32_t pair = p[0] | p[1];
                const auto q = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
                const uint32_t ls = q[0] | q[1];
#pragma unroll
                for (int b = 0; b < 4; ++b) c[b][j] = (float)((ls >> (8 * b)) & 0xFFu) * d8[j];
            }
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b)
                broadcast_rows4(f16_scale((uint16_t)((b < 2 ? d.x : d.y) >> (16 * (b & 1)))) * kActUnscale, c[b]);
        }
    }

    // Half h's activations into the wave's LDS copy.
    __device__ __forceinline__ void stage(int h, uint8_t* xs) const {
        if constexpr (PACKED) {
            const uint32_t lane = threadIdx.x & 63;
            uint8_t* dst = xs + (lane & 7) * kRunBytes + (lane >> 3) * 16;
#pragma unroll
            for (int i = 0; i < MT * 4; ++i)
                *reinterpret_cast<uint4*>(dst + ((i >> 2) * 2 + (i & 1)) * kPlaneBytes + ((i >> 1) & 1) * 128) = x[h][i];
            return;
        }
        const uint32_t lane = threadIdx.x & 63, cq = lane & 15;
        uint8_t* dst = xs + (cq >> 1) * kRunBytes + (lane >> 4) * 16 + (cq & 1) * 8;
#pragma unroll
        for (int i = 0; i < MT * 4; ++i) {
            uint2 hi, lo;
            split_bf16(x[h][i], hi, lo);
            uint8_t* p = dst + (i >> 2) * (2 * kPlaneBytes) + (i & 3) * 64;
            *reinterpret_cast<uint2*>(p) = hi;
            *reinterpret_cast<uint2*>(p + kPlaneBytes) = lo;
        }
    }

    // Half h's products: w[j] the half's weights, two blocks each.
    __device__ __forceinline__ void products(int h, const uint8_t* xs, const uint32_t* tab, const float (&c)[4][4],
                                             f32x4 (&acc)[MT][NJ]) const {
        const uint32_t lane = threadIdx.x & 63;
        const uint8_t* src = xs + (lane >> 4) * kRunBytes + (lane & 15) * 16;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            bf16x8 hi[MT], lo[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const uint8_t* p = src + m * (2 * kPlaneBytes) + b * 4 * kRunBytes;
                hi[m] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
                lo[m] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p + kPlaneBytes));
            }
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                bf16x8 w;
                if constexpr (FMT == kFmtIq2) {
                    const uint32_t dw = h ? iq[j].y : iq[j].x;
                    w = b ? iq2_bop_bf16((dw >> 18) & 0xFF0u, ((dw >> 16) & 0x3Cu) | ((dw << 6) & 0x1C0u), tab)
                          : iq2_bop_bf16((dw >> 3) & 0xFF0u, ((dw >> 1) & 0x3Cu) | ((dw >> 9) & 0x1C0u), tab);
                } else {
                    w = b ? q8_bop(q8[h][j].z, q8[h][j].w) : q8_bop(q8[h][j].x, q8[h][j].y);
                }
                const float cb = c[2 * h + b][j];
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    f32x4 p = {0.0f, 0.0f, 0.0f, 0.0f};
                    p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo[m], w, p, 0, 0, 0);
                    p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi[m], w, p, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[m][j][e] = fmaf(p[e], cb, acc[m][j][e]);
                }
            }
        }
    }
};

}  // namespace mmhip
