// MoE routing and combine on gfx950 (moeFFN, inference.zig:886-1010).
//
// route_kernel: workgroups of 16 tokens route (four tokens per wave, one per
// 16-lane row); further workgroups quantise the hidden states for the grouped
// IQ2_XXS gate/up meanwhile (one wave per token and 256-column unit). Each
// token runs Scheduler.route exactly as the CPU path does (math.topK's size-k
// min-heap, softmax over the selected logits, throttle scaling, the
// heavy-throttle top-1 fallback). The routing workgroup that ends last counts
// the experts (ExpertStats.counts), lays out the activation slots of the call
// and writes the work items that the expert kernels read on the device, so no
// routing result travels back to the host: assignments sorted by expert
// (tokens in order) and cut into items of <= item_rows rows.
//
// Bound: a token's selection is ~600 dependent vector instructions, so one
// workgroup for all tokens was bound by its CU (256 tokens 21.5 us, 64 tokens
// 7.9); sixteen tokens per CU leave one wave per SIMD.
// combine_kernel: the weighted sum in route order, the shared expert and the
// deferral bias, with products and sums rounded separately as on the CPU.
#include "device_common.hpp"
#include "gemm_tile_ops.hpp"
#include "kernels.hpp"
#include "route_ops.hpp"

namespace mmhip {

namespace {

constexpr int kRouteThreads = 256;   // 4 waves, 4 tokens each
constexpr uint32_t kRouteTokens = kRouteThreads / 64 * 4;
constexpr int kMaxTokens = 256;      // MMHIP_MOE_MAX_TOKENS
constexpr int kMaxExperts = 256;

// LDS of a routing workgroup.
struct RouteLds {
    uint64_t tok[kMaxTokens];    // routed tokens: ids (a byte each), then act from bit 32
    uint32_t cnt[kMaxExperts];   // assignments per expert
    uint32_t rec[kMaxExperts];   // experts recorded in the statistics this call
    uint32_t off[kMaxExperts];   // first slot of each expert
    uint32_t choff[kMaxExperts]; // first work item (chunk) of each expert
    uint32_t rank[kMaxTokens * kMaxK];
    uint32_t nchunks, last;
};

// Routes this workgroup's tokens; true in the workgroup that ends last, with
// every token's word in L.tok.
__device__ bool route_tokens(const RouteBatchArgs& a, RouteLds& L) {
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t T = a.n_tokens, E = a.n_experts, k = a.k;
    const uint32_t n_wg = (T + kRouteTokens - 1) / kRouteTokens;
    const uint32_t t = blockIdx.x * kRouteTokens + (tid >> 6) * 4 + (lane >> 4);
    const bool mine = (lane & 15) == 0 && t < T;
    uint32_t ids[kMaxK], act, deferred;
    float ts[kMaxK];
    if (E <= 64)
        route_select_row16<4>(a, t, ids, ts);
    else
        route_select_row16<16>(a, t, ids, ts);
    route_active(a, act, deferred);
    // The row's first lane writes the token's results.
    if (mine) {
        uint32_t packed = 0;
#pragma unroll
        for (uint32_t i = 0; i < kMaxK; ++i) packed |= (ids[i] & 0xFFu) << (8 * i);
        const uint64_t word = (uint64_t)act << 32 | packed;
        if (n_wg > 1)
            __hip_atomic_store(a.tok + t, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else
            L.tok[t] = word;
    }
    if (n_wg > 1) {
        // The ticket once the words' device-scope stores are performed
        // (stores count in vmcnt on gfx950).
        vm_wait_all();
        lds_barrier();
        if (tid == 0) {
            const uint32_t ended = __hip_atomic_fetch_add(a.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            L.last = ended == n_wg - 1;
            if (L.last) __hip_atomic_store(a.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // The weights while the ticket is on its way.
    const TokenRoute tr = finish_route(a, ids, ts);
    if (mine) {
        // RouteResult as moeFFN sees it (after the fallback).
#pragma unroll
        for (uint32_t i = 0; i < kMaxK; ++i) {
            if (a.route_ids) a.route_ids[t * kMaxK + i] = i < k ? tr.ids[i] : 0xFFFFFFFFu;
            if (a.route_w) a.route_w[t * kMaxK + i] = i < k ? tr.w[i] : 0.0f;
            a.assign_w[t * kMaxK + i] = ((tr.act >> i) & 1u) ? tr.w[i] : 0.0f;
        }
        a.deferred[t] = tr.deferred;
        a.shared_slot[t] = a.shared ? (int32_t)(4 * T + t) : -1;
        a.slot_tok[4 * T + t] = t;
    }
    if (n_wg > 1) {
        lds_barrier();
        if (!L.last) return false;
        for (uint32_t p = tid; p < T; p += kRouteThreads)
            L.tok[p] = __hip_atomic_load(a.tok + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return true;
}

__device__ void route_layout(const RouteBatchArgs& a, RouteLds& L) {
    uint32_t* const s_cnt = L.cnt;
    uint32_t* const s_rec = L.rec;
    uint32_t* const s_off = L.off;
    uint32_t* const s_choff = L.choff;
    uint32_t* const s_rank = L.rank;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t T = a.n_tokens, E = a.n_experts, k = a.k;
    auto id_of = [&](uint32_t t, uint32_t i) { return (uint32_t)(L.tok[t] >> (8 * i)) & 0xFFu; };
    auto active = [&](uint32_t t, uint32_t i) { return i < k && ((L.tok[t] >> (32 + i)) & 1u); };
    for (uint32_t e = tid; e < E; e += kRouteThreads) {
        s_cnt[e] = 0;
        s_rec[e] = 0;
    }
    // Every barrier here orders LDS only: no phase reads what an earlier one
    // stored to global memory, and __syncthreads() would also wait for every
    // wave's outstanding global stores and statistics atomics (~1 us each).
    lds_barrier();

    // Prefill: assignments grouped by expert. An assignment's rank inside its
    // expert group comes from an LDS counter; rows of a group are independent,
    // so the order inside a group does not change any result.
    for (uint32_t p = tid; p < T * kMaxK; p += kRouteThreads) {
        const uint32_t t = p / kMaxK, i = p % kMaxK;
        if (i < k) atomicAdd(&s_rec[id_of(t, i)], 1u);  // stats.record (220-222)
        if (active(t, i)) s_rank[p] = atomicAdd(&s_cnt[id_of(t, i)], 1u);
    }
    lds_barrier();
    // Statistics: one device atomic per recorded expert.
    for (uint32_t e = tid; e < E; e += kRouteThreads)
        if (s_rec[e]) atomicAdd(a.counts + e, (unsigned long long)s_rec[e]);
    if (wave == 0) {
        // Exclusive scans over experts: slot offsets and chunk (work item) offsets.
        uint32_t carry = 0, carry_ch = 0;
        for (uint32_t base = 0; base < E; base += 64) {
            const uint32_t e = base + lane;
            const uint32_t c = e < E ? s_cnt[e] : 0u;
            const uint32_t ch = (c + a.item_rows - 1) / a.item_rows;
            uint32_t inc = c, inc_ch = ch;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t u = (uint32_t)__shfl_up((int)inc, off, 64);
                const uint32_t uch = (uint32_t)__shfl_up((int)inc_ch, off, 64);
                if (lane >= (uint32_t)off) {
                    inc += u;
                    inc_ch += uch;
                }
            }
            if (e < E) {
                s_off[e] = carry + inc - c;
                s_choff[e] = carry_ch + inc_ch - ch;
            }
            carry += (uint32_t)__shfl((int)inc, 63, 64);
            carry_ch += (uint32_t)__shfl((int)inc_ch, 63, 64);
        }
        if (lane == 0) L.nchunks = carry_ch;
    }
    lds_barrier();
    for (uint32_t p = tid; p < T * kMaxK; p += kRouteThreads) {
        const uint32_t t = p / kMaxK, i = p % kMaxK;
        int32_t slot = -1;
        if (active(t, i)) {
            slot = (int32_t)(s_off[id_of(t, i)] + s_rank[p]);
            a.slot_tok[slot] = t;
        }
        a.assign_slot[p] = slot;
    }
    // Work items: chunk c of expert e is item s_choff[e] + c; the shared
    // expert's chunks follow.
    auto put = [&](uint32_t q, uint32_t gate, uint32_t up, uint32_t down, uint32_t slot, uint32_t m) {
        if (a.paired) {
            a.work_gu[q] = QmmWork{gate, slot, m, up};
        } else {
            a.work_gu[2 * q] = QmmWork{gate, slot, m, 0};
            a.work_gu[2 * q + 1] = QmmWork{up, slot, m, a.inter};
        }
        a.work_dn[q] = QmmWork{down, slot, m, 0};
    };
    for (uint32_t e = tid; e < E; e += kRouteThreads) {
        const uint32_t c = s_cnt[e], off = s_off[e], ch0 = s_choff[e];
        for (uint32_t c0 = 0, q = ch0; c0 < c; c0 += a.item_rows, ++q)
            put(q, e, E + e, e, off + c0, min(a.item_rows, c - c0));
    }
    const uint32_t nch = L.nchunks;
    const bool sh = a.shared && a.shared_merged;
    const uint32_t sh_chunks = sh ? (T + a.item_rows - 1) / a.item_rows : 0;
    for (uint32_t c = tid; c < sh_chunks; c += kRouteThreads) {
        const uint32_t c0 = c * a.item_rows;
        put(nch + c, 2 * E, 2 * E + 1, E, 4 * T + c0, min(a.item_rows, T - c0));
    }
    if (tid == 0) {
        a.n_work[0] = (a.paired ? 1 : 2) * (nch + sh_chunks);
        a.n_work[1] = nch + sh_chunks;
    }
}

__global__ __launch_bounds__(kRouteThreads) void route_kernel(RouteBatchArgs a) {
    __shared__ RouteLds L;
    const uint32_t n_wg = (a.n_tokens + kRouteTokens - 1) / kRouteTokens;
    if (blockIdx.x >= n_wg) {
        if (a.px) {
            // Hidden states as bf16 pairs.
            const uint64_t i = (uint64_t)(blockIdx.x - n_wg) * kRouteThreads + threadIdx.x;
            if (i < (uint64_t)a.n_tokens * a.px_cols) {
                const uint32_t t = (uint32_t)(i / a.px_cols), col = (uint32_t)(i % a.px_cols);
                pack_row(a.px_out + (uint64_t)t * a.px_cols, a.px_cols, col, a.px[i]);
            }
            return;
        }
        // Hidden-state quantisation: one wave per (token, 256-column unit).
        const uint64_t unit = (uint64_t)(blockIdx.x - n_wg) * (kRouteThreads / 64) + (threadIdx.x >> 6);
        if (unit < (uint64_t)a.n_tokens * a.q_units)
            quantize_unit_wave<false>(a.qx, a.qx_stride, 0, unit / a.q_units, (uint32_t)(unit % a.q_units), a.q_cols,
                                      a.qa.hi, a.qa.lo, a.qa.scale, a.qa.stride, a.qa.scale_stride);
        return;
    }
    if (route_tokens(a, L)) route_layout(a, L);  // uniform over the workgroup
}

// Four columns of one token per thread (VEC: rows of a multiple of four
// columns, 16-byte aligned), so the token's slots and weights are uniform and
// its expert rows load together; one column at a time took 2.4 us for one token of
// 2048 columns against 1.4, 3.9 for 64 against 3.0 and 5.2 for 256 against 4.6.
template <int VEC>
__global__ __launch_bounds__(256) void combine_kernel(const float* __restrict__ eo, const int32_t* __restrict__ assign_slot,
                               const float* __restrict__ assign_w, const int32_t* __restrict__ shared_slot,
                               const uint32_t* __restrict__ deferred, const float* __restrict__ bias,
                               float* __restrict__ out, uint32_t hidden) {
    typedef float vf __attribute__((ext_vector_type(VEC)));
    const uint32_t t = blockIdx.y, j = (blockIdx.x * 256 + threadIdx.x) * VEC;
    if (j >= hidden) return;
    int32_t s[kMaxK + 1];
    float w[kMaxK];
#pragma unroll
    for (int i = 0; i < kMaxK; ++i) {
        s[i] = assign_slot[t * kMaxK + i];
        w[i] = assign_w[t * kMaxK + i];
    }
    s[kMaxK] = shared_slot[t];
    const bool with_bias = bias && deferred[t];
    vf v[kMaxK + 1];
#pragma unroll
    for (int i = 0; i <= kMaxK; ++i)
        if (s[i] >= 0) v[i] = *reinterpret_cast<const vf*>(eo + (uint64_t)s[i] * hidden + j);
    vf o = 0.0f;
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
#pragma unroll
        for (int i = 0; i < kMaxK; ++i)
            if (s[i] >= 0) o[e] = __fadd_rn(o[e], __fmul_rn(w[i], v[i][e]));
        if (s[kMaxK] >= 0) o[e] = __fadd_rn(o[e], v[kMaxK][e]);
        if (with_bias) o[e] = __fadd_rn(o[e], bias[j + e]);
    }
    *reinterpret_cast<vf*>(out + (uint64_t)t * hidden + j) = o;
}

}  // namespace

uint32_t route_max_work(uint32_t n_tokens, uint32_t n_experts, uint32_t item_rows) {
    const uint32_t routed = 4 * n_tokens;
    const uint32_t chunks = (n_experts < routed ? n_experts : routed) + (routed + item_rows - 1) / item_rows +
                            (n_tokens + item_rows - 1) / item_rows;
    return 2 * chunks;
}

hipError_t launch_route(const RouteBatchArgs& a, hipStream_t s) {
    if (a.n_tokens < 2 || a.n_tokens > kMaxTokens || a.n_experts > kMaxExperts || a.k == 0 || a.k > kMaxK ||
        a.k > a.n_experts)
        return hipErrorInvalidValue;
    const uint64_t q_waves = a.qx ? (uint64_t)a.n_tokens * a.q_units : 0;
    const uint64_t p_waves = a.px ? ((uint64_t)a.n_tokens * a.px_cols + 63) / 64 : 0;
    const unsigned q_wgs = (unsigned)((q_waves + p_waves + kRouteThreads / 64 - 1) / (kRouteThreads / 64));
    const unsigned r_wgs = (a.n_tokens + kRouteTokens - 1) / kRouteTokens;
    route_kernel<<<r_wgs + q_wgs, kRouteThreads, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_combine(const float* eo, const int32_t* assign_slot, const float* assign_w,
                          const int32_t* shared_slot, const uint32_t* deferred, const float* bias, float* out,
                          uint32_t n_tokens, uint32_t hidden, hipStream_t s) {
    if (n_tokens == 0 || hidden == 0) return hipSuccess;
    const bool vec = hidden % 4 == 0 && (reinterpret_cast<uintptr_t>(eo) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
    const uint32_t per = vec ? 1024 : 256;
    const dim3 grid((hidden + per - 1) / per, n_tokens);
    if (vec)
        combine_kernel<4><<<grid, 256, 0, s>>>(eo, assign_slot, assign_w, shared_slot, deferred, bias, out, hidden);
    else
        combine_kernel<1><<<grid, 256, 0, s>>>(eo, assign_slot, assign_w, shared_slot, deferred, bias, out, hidden);
    return hipGetLastError();
}

}  // namespace mmhip
