// f32 / f16 weights times several vectors (the router of a prefill call,
// batchMatMulUnified's f32 branch, inference.zig:1231-1264): one matrix,
// every output summed in math.matVecMul's order, bit for bit (four lane
// chains of unfused products, ((a0 + a1) + a2) + a3, then the last cols % 4
// products; gemv_strict_kernel has the single-vector form).
//
// Bound: VALU. The order forbids fused multiply-adds and matrix
// instructions, so an output costs 2 cols instructions. A workgroup of four
// waves owns a tile of 4 PR rows x 16 PV vectors; lane (v, l) of a wave holds
// the partial sums of chain l for PR rows and PV vectors. Per chunk of columns
// the tile's rows and vectors are staged in LDS split by chain, so that one
// 16-byte read brings four consecutive terms of a chain: PR + PV reads feed
// 8 PR PV VALU instructions. The next chunk's global loads are issued before
// the current one is summed. [2560 x 512] times 300 vectors: 388 us as one
// workgroup per row and 16 vectors (its products went through LDS and 64 of 256
// threads summed), 27 us here, 29 M VALU instructions per us of the chip's 39 M.
#include "device_common.hpp"
#include "kernels.hpp"

namespace mmhip {

namespace {

constexpr uint32_t kThreads = 256;

template <typename WT, int PR, int PV, uint32_t KC>
__global__ __launch_bounds__(kThreads) void gemm_strict_kernel(const WT* __restrict__ w, const float* __restrict__ x,
                                                               uint64_t x_stride, float* __restrict__ y,
                                                               uint64_t y_stride, uint32_t n_vecs, uint32_t rows,
                                                               uint32_t cols) {
#pragma clang fp contract(off)
    constexpr uint32_t TR = 4 * PR, TV = 16 * PV;
    // LDS rows [chain][row][KC / 4 terms]; the pads keep the 16 vectors of a
    // chain, and the four chains of a weight row, on separate banks.
    constexpr uint32_t kRun = KC / 4 + 4;
    constexpr uint32_t kWChain = TR * kRun + 8, kXChain = TV * kRun + 8;
    constexpr uint32_t kQuads = KC / 4;                       // column quads of a chunk
    constexpr uint32_t kRowsPerPass = kThreads / kQuads;
    constexpr uint32_t kWPass = (TR + kRowsPerPass - 1) / kRowsPerPass;
    constexpr uint32_t kXPass = (TV + kRowsPerPass - 1) / kRowsPerPass;
    constexpr int kUnroll = PR * PV == 1 ? 8 : PR * PV == 2 ? 4 : 2;
    static_assert(kThreads % kQuads == 0 && TR % kRowsPerPass == 0 && TV % kRowsPerPass == 0, "staging covers the tile");
    __shared__ __align__(16) float ws[4 * kWChain];
    __shared__ __align__(16) float xs[4 * kXChain];
    __shared__ float ys[TV][TR + 1];

    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t v = lane & 15, l = lane >> 4;
    const uint32_t r0 = blockIdx.x * TR, v0 = blockIdx.y * TV;
    const uint32_t cols4 = cols & ~3u;
    const uint32_t n_r = min(rows - r0, TR), n_v = min(n_vecs - v0, TV);
    // Byte offsets inside the tile stay below 2^31 (launch_gemm_strict).
    const BufRsrc wr = make_rsrc(w + (uint64_t)r0 * cols, n_r * cols * (uint32_t)sizeof(WT));
    const BufRsrc xr = make_rsrc(x + (uint64_t)v0 * x_stride, ((n_v - 1) * (uint32_t)x_stride + cols) * 4);
    const uint32_t sq = tid % kQuads, sr = tid / kQuads;  // staging: quad and first row

    uint4 wq[kWPass], xq[kXPass];
    auto load = [&](uint32_t c0) {
        const uint32_t col = c0 + 4 * sq;
        const bool ok = col < cols4;
#pragma unroll
        for (uint32_t p = 0; p < kWPass; ++p) {
            const uint32_t r = sr + p * kRowsPerPass;
            const uint32_t off = ok && r < n_r ? (r * cols + col) * (uint32_t)sizeof(WT) : kBufOob;
            if constexpr (sizeof(WT) == 2) {
                const uint2 h = buf_load_b64(wr, off, 0);
                wq[p] = make_uint4(h.x, h.y, 0, 0);
            } else {
                wq[p] = buf_load_b128(wr, off, 0);
            }
        }
#pragma unroll
        for (uint32_t p = 0; p < kXPass; ++p) {
            const uint32_t m = sr + p * kRowsPerPass;
            xq[p] = buf_load_b128(xr, ok && m < n_v ? (m * (uint32_t)x_stride + col) * 4 : kBufOob, 0);
        }
    };
    auto store = [&]() {
#pragma unroll
        for (uint32_t p = 0; p < kWPass; ++p) {
            float* d = ws + (sr + p * kRowsPerPass) * kRun + sq;
            if constexpr (sizeof(WT) == 2) {
                d[0] = f16_bits_to_f32(wq[p].x & 0xFFFFu);
                d[kWChain] = f16_bits_to_f32(wq[p].x >> 16);
                d[2 * kWChain] = f16_bits_to_f32(wq[p].y & 0xFFFFu);
                d[3 * kWChain] = f16_bits_to_f32(wq[p].y >> 16);
            } else {
                d[0] = __uint_as_float(wq[p].x);
                d[kWChain] = __uint_as_float(wq[p].y);
                d[2 * kWChain] = __uint_as_float(wq[p].z);
                d[3 * kWChain] = __uint_as_float(wq[p].w);
            }
        }
#pragma unroll
        for (uint32_t p = 0; p < kXPass; ++p) {
            float* d = xs + (sr + p * kRowsPerPass) * kRun + sq;
            d[0] = __uint_as_float(xq[p].x);
            d[kXChain] = __uint_as_float(xq[p].y);
            d[2 * kXChain] = __uint_as_float(xq[p].z);
            d[3 * kXChain] = __uint_as_float(xq[p].w);
        }
    };

    // A chain's terms past cols4 are products of zeros: the sum starts at +0
    // and so is never -0, and adding +0 leaves every other value as it is.
    float acc[PR][PV];
#pragma unroll
    for (int i = 0; i < PR; ++i)
#pragma unroll
        for (int j = 0; j < PV; ++j) acc[i][j] = 0.0f;
    const float4* wp = reinterpret_cast<const float4*>(ws + l * kWChain + wave * PR * kRun);
    const float4* xp = reinterpret_cast<const float4*>(xs + l * kXChain + v * kRun);
    load(0);
    for (uint32_t c0 = 0; c0 < cols4; c0 += KC) {
        store();
        lds_barrier();
        if (c0 + KC < cols4) load(c0 + KC);
        const uint32_t n16 = (min(KC, cols4 - c0) + 15) / 16;
#pragma unroll(kUnroll)
        for (uint32_t i = 0; i < n16; ++i) {
            float4 a[PR], b[PV];
#pragma unroll
            for (int p = 0; p < PR; ++p) a[p] = wp[p * (kRun / 4) + i];
#pragma unroll
            for (int p = 0; p < PV; ++p) b[p] = xp[p * 16 * (kRun / 4) + i];
#pragma unroll
            for (int p = 0; p < PR; ++p)
#pragma unroll
                for (int q = 0; q < PV; ++q) {
                    float s = acc[p][q];
                    s = s + a[p].x * b[q].x;
                    s = s + a[p].y * b[q].y;
                    s = s + a[p].z * b[q].z;
                    s = s + a[p].w * b[q].w;
                    acc[p][q] = s;
                }
        }
        lds_barrier();
    }
#pragma unroll
    for (int p = 0; p < PR; ++p)
#pragma unroll
        for (int q = 0; q < PV; ++q) {
            const float a0 = acc[p][q];
            const float a1 = __shfl(a0, v + 16, kWave), a2 = __shfl(a0, v + 32, kWave), a3 = __shfl(a0, v + 48, kWave);
            if (l == 0) {
                const uint32_t r = wave * PR + p, m = q * 16 + v;
                float sum = ((a0 + a1) + a2) + a3;
                if (r < n_r && m < n_v) {
                    const WT* wt = w + (uint64_t)(r0 + r) * cols;
                    const float* xt = x + (uint64_t)(v0 + m) * x_stride;
                    for (uint32_t c = cols4; c < cols; ++c) {
                        float wv;
                        if constexpr (sizeof(WT) == 2)
                            wv = f16_bits_to_f32(wt[c]);
                        else
                            wv = wt[c];
                        sum = sum + wv * xt[c];
                    }
                }
                ys[m][r] = sum;
            }
        }
    lds_barrier();
    for (uint32_t i = tid; i < TR * TV; i += kThreads) {
        const uint32_t m = i / TR, r = i % TR;
        if (m < n_v && r < n_r) y[(uint64_t)(v0 + m) * y_stride + r0 + r] = ys[m][r];
    }
}

template <int PR, int PV, uint32_t KC>
void launch_tile(const void* w, bool f16, const float* x, uint64_t x_stride, float* y, uint64_t y_stride, uint32_t n,
                 uint32_t rows, uint32_t cols, hipStream_t s) {
    const dim3 grid((rows + 4 * PR - 1) / (4 * PR), (n + 16 * PV - 1) / (16 * PV));
    if (f16)
        gemm_strict_kernel<uint16_t, PR, PV, KC>
            <<<grid, kThreads, 0, s>>>((const uint16_t*)w, x, x_stride, y, y_stride, n, rows, cols);
    else
        gemm_strict_kernel<float, PR, PV, KC>
            <<<grid, kThreads, 0, s>>>((const float*)w, x, x_stride, y, y_stride, n, rows, cols);
}

}  // namespace

// The row kernel (gemv_strict_kernel with 16 vectors, one workgroup per row and
// a CU's LDS each) stays the faster one while its workgroups fit one round of
// the CUs: [64 x 2048] times 2..64 vectors takes 5.6-6.0 us there and 7.3-7.5
// here, times 256 (four rounds) 19.8 and 7.9; [1500 x 512] times 12, 13.4 and
// 4.3. Tiles are addressed with 32-bit byte offsets: 32 rows of 2^24 floats.
bool gemm_strict_fits(uint32_t n, uint32_t rows, uint32_t cols, uint64_t x_stride, int num_cu) {
    return (uint64_t)rows * ((n + 15) / 16) > (uint64_t)(num_cu > 0 ? num_cu : 256) && cols < (1u << 24) &&
           x_stride < (1u << 24) && (n + 15) / 16 < 65536;
}

hipError_t launch_gemm_strict(const void* w, uint32_t type, const float* x, uint64_t x_stride, float* y,
                              uint64_t y_stride, uint32_t n, uint32_t rows, uint32_t cols, int num_cu, hipStream_t s) {
    if ((uint64_t)n * rows == 0) return hipSuccess;
    const bool h = type != 0;
    // The largest tile that still gives 7/4 workgroups per CU. Measured (us
    // with 4 x 2, 2 x 1, 1 x 1): [2560 x 512] times 300 vectors 27.0, 34.6,
    // 47.5 (1600 workgroups of the largest); [1024 x 3072] times 50 42.1, 19.9,
    // 26.7 (128, 512 and 1024 workgroups); [64 x 2048] times 256 28.8, 12.8,
    // 7.9 (32, 128 and 256). Long chunks help where few workgroups share a
    // CU: that last one takes 9.5 with 256-column chunks, 7.9 with 512.
    const uint64_t enough = (uint64_t)(num_cu > 0 ? num_cu : 256) * 7 / 4;
    auto wgs = [&](uint64_t tr, uint64_t tv) { return (rows + tr - 1) / tr * ((n + tv - 1) / tv); };
    if (wgs(16, 32) >= enough)
        launch_tile<4, 2, 128>(w, h, x, x_stride, y, y_stride, n, rows, cols, s);
    else if (wgs(8, 16) >= enough)
        launch_tile<2, 1, 128>(w, h, x, x_stride, y, y_stride, n, rows, cols, s);
    else
        launch_tile<1, 1, 512>(w, h, x, x_stride, y, y_stride, n, rows, cols, s);
    return hipGetLastError();
}

}  // namespace mmhip
