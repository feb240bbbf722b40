// qw_topk.hpp -- softmax, exact top-k and weight normalisation of one token's
// router logits, for one wave (ggml_soft_max, ARGSORT + top-k, sum/clamp/div of
// core/runtime.cpp:869-897; bit-identical to the reference CPU path), with the
// resident-decode routing of core/runtime.cpp:870-881: want = the top k of the
// raw logits (ggml_argsort_top_k), then logits + mask (ggml_add of the layer's
// 0 / -inf row) before the softmax.
#pragma once

#include "qw_kernels.hpp"
#include "qw_sort.hpp"

namespace qw {

// A barrier for LDS traffic between the lanes of one wave.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float lane_value(float v, int lane) {   // lane: uniform
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// ARGSORT (descending) of the E values in p, first k into order[0..k): ranks by
// count of strictly larger values.  Tied values share a rank, so when exactly k
// values rank below k and they fill all k places, no tie (and no NaN, which nothing
// is larger than) reaches into the first k; else the order is std::sort's to say,
// which is then replayed exactly (and reported as status bit 0).  Ends synchronised.
template <bool WAVE>
__device__ __forceinline__ void topk_order(const float* p, int64_t E, int64_t k, int32_t* order,
                                           SortRange* sort_stack, int32_t* __restrict__ status, int lane) {
    auto sync = [] {
        if constexpr (WAVE) wave_sync();
        else __syncthreads();
    };
    for (int64_t r = lane; r < k; r += 64) order[r] = -1;
    sync();
    // (p is 16-byte aligned and E % 8 == 0: four values per LDS read)
    int found = 0;
    for (int64_t i0 = 0; i0 < E; i0 += 64) {
        const int64_t i = i0 + lane;
        const bool valid = i < E;
        const float pi = p[valid ? i : 0];
        int gt = 0;
#pragma unroll 8
        for (int64_t j = 0; j < E; j += 4) {
            const float4 q = *(const float4*) (p + j);
            gt += (q.x > pi) + (q.y > pi) + (q.z > pi) + (q.w > pi);
        }
        const bool in = valid && gt < k;
        if (in) order[gt] = (int32_t) i;
        found += __popcll(__ballot(in));
    }
    sync();
    bool bad = found != k;
    for (int64_t r = lane; r < k; r += 64) bad = bad || order[r] < 0;
    if (__any(bad)) {
        if (lane == 0) {
            for (int64_t i = 0; i < E; ++i) order[i] = (int32_t) i;
            libstdcxx_sort_desc(order, (int) E, p, sort_stack);
            if (status) atomicOr(status, 1);
        }
        sync();
    }
}

// One wave (lane 0..63) handles token t.  p (16-byte aligned), order: E <= 512 entries;
// sort_stack: SORT_STACK (all in LDS, private to the wave when WAVE is set, else to a
// 64-thread workgroup).  The ordered double sums take their terms by lane reads, not
// through LDS on one lane (with the grouping, 128 experts, top 8: 7.6 us at T = 1, 9.7 at
// T = 10, which was 16 with the sums on one lane and the grouping by the whole workgroup).  mask: [E] added to the
// logits before the softmax, or null; want: [T][k] top k of the raw logits, or null.
template <bool WAVE>
__device__ __forceinline__ void topk_token(const float* __restrict__ logits, int64_t E, int64_t k, int64_t t,
                                           float clamp_min, float scale, int32_t* __restrict__ ids,
                                           float* __restrict__ weights, float* __restrict__ probs_out,
                                           int32_t* __restrict__ status, float* p, int32_t* order,
                                           SortRange* sort_stack, int lane,
                                           const float* __restrict__ mask = nullptr, int32_t* __restrict__ want = nullptr) {
    auto sync = [] {
        if constexpr (WAVE) wave_sync();
        else __syncthreads();
    };
    const float* l = logits + t * E;
    if (want) {
        for (int64_t i = lane; i < E; i += 64) p[i] = l[i];
        sync();
        topk_order<WAVE>(p, E, k, order, sort_stack, status, lane);
        for (int64_t i = lane; i < k; i += 64) want[t * k + i] = order[i];
        sync();
    }
    auto lm = [&](int64_t i) { return mask ? l[i] + mask[i] : l[i]; };
    float mx = -INFINITY;
    for (int64_t i = lane; i < E; i += 64) mx = fmaxf(mx, lm(i));
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    for (int64_t i = lane; i < E; i += 64) p[i] = v_expf(lm(i) - mx);
    sync();
    const int ng = (int) (E / 8);   // at most 64 groups: lane gi holds group gi's sum
    const float gs = lane < ng ? hsum8(&p[8 * lane]) : 0.0f;
    double sum = 0.0;
    for (int gi = 0; gi < ng; ++gi) sum += (double) lane_value(gs, gi);
    sync();
    const float inv = (float) (1.0 / sum);
    for (int64_t i = lane; i < E; i += 64) p[i] = p[i] * inv;
    sync();
    if (probs_out)
        for (int64_t i = lane; i < E; i += 64) probs_out[t * E + i] = p[i];
    // the order of the probabilities.  NaNs go to the sort replay (they fill one place only):
    // softmax makes every probability NaN then, which std::sort treats as all
    // equivalent.
    topk_order<WAVE>(p, E, k, order, sort_stack, status, lane);
    double s = 0.0;
    for (int64_t i0 = 0; i0 < k; i0 += 64) {
        const float pv = i0 + lane < k ? p[order[i0 + lane]] : 0.0f;
        const int n = (int) (k - i0 < 64 ? k - i0 : 64);
        for (int i = 0; i < n; ++i) s += (double) lane_value(pv, i);
    }
    float wsum = (float) s;
    wsum = fmaxf(fminf(wsum, INFINITY), clamp_min);
    for (int64_t i = lane; i < k; i += 64) {
        float wi = p[order[i]] / wsum;
        if (scale != 0.0f && scale != 1.0f) wi = wi * scale;
        ids[t * k + i] = order[i];
        weights[t * k + i] = wi;
    }
}

}  // namespace qw
