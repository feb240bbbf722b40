// quantize.hip -- block quantizers on the GPU, bit-identical to ggml's CPU code.
//
// Activation quantizers (what ggml_compute_forward_mul_mat_id runs on src1,
// ggml/src/ggml-cpu/ggml-cpu.c:1585-1620, through type_traits_cpu.from_float):
//   Q8_K: quantize_row_q8_K_ref      ggml/src/ggml-quants.c:2768-2803
//   Q8_0: x86 quantize_row_q8_0      ggml/src/ggml-cpu/arch/x86/quants.c:302-404
// Weight quantizers (ggml_quantize_chunk with no imatrix, ggml/src/ggml.c:7919-8000):
//   Q4_K: quantize_row_q4_K_ref      ggml-quants.c:1457-1527 (+ make_qkx2_quants 799-878)
//   Q6_K: quantize_row_q6_K_ref      ggml-quants.c:1869-1937 (+ make_qx_quants 628-700)
//   Q8_0: quantize_row_q8_0_ref      ggml-quants.c:276-297
// Division and sqrt are IEEE correctly rounded (HIP default), no contraction.
#include "qw_kernels.hpp"

namespace qw {

// ---------------------------------------------------------------------------
// Activation Q8_K: one wave per 256-value block, 4 values per lane.
// src rows may be strided (ggml nb1/nb2 in bytes); dst rows are dense.
__global__ void __launch_bounds__(256) k_quant_q8K(const float* __restrict__ src, int64_t K, int64_t ne1,
                                                   int64_t nrows, size_t nb1, size_t nb2,
                                                   BlockQ8_K* __restrict__ dst, _Float16* __restrict__ hout) {
    const int lane = threadIdx.x & 63;
    const int64_t nb = K / QK_K;
    const int64_t blk = (int64_t) blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
    if (blk >= nb * nrows) return;
    const int64_t row = blk / nb, ib = blk % nb;
    const int64_t i1 = row % ne1, i2 = row / ne1;
    const float* x = (const float*) ((const char*) src + i1 * nb1 + i2 * nb2) + ib * QK_K;
    const float4 q = *(const float4*) (x + 4 * lane);
    const float v[4] = {q.x, q.y, q.z, q.w};
    quant_q8K_wave(v, lane, dst + blk, hout ? hout + (size_t) blk * QK_K : nullptr,
                   hout ? hout + (size_t) (nb * nrows) * QK_K + (size_t) blk * 16 : nullptr);
}

// SwiGLU (ggml_swiglu_split: silu(gate) * up, ops.cpp:3182-3238) of n_rows dense
// rows of F values, quantized straight to Q8_K as the down projection reads it:
// one wave per 256-value block, the same values and quantizer as k_swiglu then
// k_quant_q8K, without the fp32 round trip.
__global__ void __launch_bounds__(256) k_swiglu_q8K(const float* __restrict__ gate, const float* __restrict__ up,
                                                    int64_t F, int64_t n_rows, BlockQ8_K* __restrict__ dst,
                                                    _Float16* __restrict__ hout) {
    const int lane = threadIdx.x & 63;
    const int64_t nb = F / QK_K;
    const int64_t blk = (int64_t) blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
    if (blk >= nb * n_rows) return;
    const int64_t off = (blk / nb) * F + (blk % nb) * QK_K + 4 * lane;
    const float4 g = *(const float4*) (gate + off);
    const float4 u = *(const float4*) (up + off);
    const float v[4] = {v_silu(g.x) * u.x, v_silu(g.y) * u.y, v_silu(g.z) * u.z, v_silu(g.w) * u.w};
    quant_q8K_wave(v, lane, dst + blk, hout ? hout + (size_t) blk * QK_K : nullptr,
                   hout ? hout + (size_t) (nb * n_rows) * QK_K + (size_t) blk * 16 : nullptr);
}

int launch_swiglu_q8K(const float* gate, const float* up, int64_t F, int64_t n_rows, void* dst, hipStream_t stream,
                      uint16_t* h_out) {
    if (F % QK_K) return -2;
    const int64_t nblk = (F / QK_K) * n_rows;
    if (nblk == 0) return 0;
    hipLaunchKernelGGL(k_swiglu_q8K, dim3((unsigned) ((nblk + 3) / 4)), dim3(256), 0, stream, gate, up, F, n_rows,
                       (BlockQ8_K*) dst, (_Float16*) h_out);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

__global__ void __launch_bounds__(256) k_quant_q8_0_act(const float* __restrict__ src, int64_t K, int64_t ne1,
                                                        int64_t nrows, size_t nb1, size_t nb2,
                                                        BlockQ8_0* __restrict__ dst, _Float16* __restrict__ h,
                                                        float* __restrict__ hd) {
    const int64_t nb = K / QK8_0;
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t blk = gid >> 3;
    const int sub = threadIdx.x & 7;
    const bool valid = blk < nb * nrows;
    const int64_t b = valid ? blk : 0;
    const int64_t row = b / nb, ib = b % nb;
    const int64_t i1 = row % ne1, i2 = row / ne1;
    const float* x = (const float*) ((const char*) src + i1 * nb1 + i2 * nb2) + ib * QK8_0;
    quant_q80_lane8(*(const float4*) (x + 4 * sub), valid, blk, sub, dst, h, hd);
}

// SwiGLU of dense rows straight into Q8_0 (k_swiglu's values, k_quant_q8_0_act's
// quantizer), without the fp32 round trip and its launch.
__global__ void __launch_bounds__(256) k_swiglu_q80(const float* __restrict__ gate, const float* __restrict__ up,
                                                    int64_t nblk, BlockQ8_0* __restrict__ dst,
                                                    _Float16* __restrict__ h, float* __restrict__ hd) {
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t blk = gid >> 3;
    const int sub = threadIdx.x & 7;
    const bool valid = blk < nblk;
    const int64_t off = QK8_0 * (valid ? blk : 0) + 4 * sub;
    const float4 g = *(const float4*) (gate + off);
    const float4 u = *(const float4*) (up + off);
    quant_q80_lane8(float4{v_silu(g.x) * u.x, v_silu(g.y) * u.y, v_silu(g.z) * u.z, v_silu(g.w) * u.w}, valid, blk, sub,
                    dst, h, hd);
}

int launch_swiglu_q80(const float* gate, const float* up, int64_t F, int64_t n_rows, void* dst, hipStream_t stream,
                      uint16_t* h_out, float* hd_out) {
    if (F % QK8_0 || (((uintptr_t) gate | (uintptr_t) up) & 15) || !h_out != !hd_out) return -2;
    const int64_t nblk = (F / QK8_0) * n_rows;
    if (nblk == 0) return 0;
    hipLaunchKernelGGL(k_swiglu_q80, dim3((unsigned) ((8 * nblk + 255) / 256)), dim3(256), 0, stream, gate, up, nblk,
                       (BlockQ8_0*) dst, (_Float16*) h_out, hd_out);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

int launch_quantize_act(int vdt, const float* src, int64_t K, int64_t ne1, int64_t nrows, size_t nb1, size_t nb2,
                        void* dst, hipStream_t stream, uint16_t* h_out, float* hd_out) {
    if (h_out && vdt == T_Q8_0 && !hd_out) return -2;
    if (vdt == T_Q8_K) {
        const int64_t nblk = (K / QK_K) * nrows;
        if (nblk == 0) return 0;
        hipLaunchKernelGGL(k_quant_q8K, dim3((unsigned) ((nblk + 3) / 4)), dim3(256), 0, stream, src, K, ne1, nrows,
                           nb1, nb2, (BlockQ8_K*) dst, (_Float16*) h_out);
    } else if (vdt == T_Q8_0) {
        const int64_t nthr = (K / QK8_0) * nrows * 8;
        if (nthr == 0) return 0;
        hipLaunchKernelGGL(k_quant_q8_0_act, dim3((unsigned) ((nthr + 255) / 256)), dim3(256), 0, stream, src, K, ne1,
                           nrows, nb1, nb2, (BlockQ8_0*) dst, (_Float16*) h_out, hd_out);
    } else {
        return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

// ---------------------------------------------------------------------------
// Weight quantizers.  One thread per 32-value sub-block (Q4_K) or 16-value
// sub-block (Q6_K), everything in registers; the super-block finalisation is done
// after exchanging the sub-block results through shuffles.
//
// Bound: VALU issue -- the reference's searches are 21 (18) passes over a
// sub-block with float sums in element order, which leaves one thread per
// sub-block and about 17 (9) instructions per value and pass.  So the searches
// keep the quants as floats (nearest_int's magic addend added and taken off
// again, clamped in between), and instead of copying a candidate's quants when it
// wins they remember what produced it: those quants are read only for a
// sub-block whose stored scale rounds to 0.  Both need every value finite and
// every scaled value below 2^21, as ggml's nearest_int asserts 2^22; the few sub-blocks
// that are not go through the general form, which repeats the reference's integer
// steps.  12288 x 2048 values: Q4_K 2056 -> 234 us,
// Q6_K 188 -> 113 us.

constexpr float QMAGIC = 12582912.f;   // 1.5 * 2^23: nearest_int's addend

// make_qkx2_quants(32, 15, x, weights, L, &min, Laux, -1, 0.1, 20, false) of the 32
// values at x (weights av_x + |x|), step for step with ggml's integer quants: the
// general form, values read from memory in rolled loops (no registers held for it).
// The quants are those of nearest_int(l_iscale * (x - l_min)).
__device__ __forceinline__ void qkx2_32_general(const float* x, float av_x, float& scale_out, float& min_out,
                                                float& l_iscale, float& l_min) {
    const int n = 32, nmax = 15;
    const float rmin = -1.f, rdelta = 0.1f;
    const int nstep = 20;
    auto w = [&](int i) { return av_x + __builtin_fabsf(x[i]); };
    float min = x[0], max = x[0];
    float sum_w = w(0);
    float sum_x = sum_w * x[0];
#pragma unroll 1
    for (int i = 1; i < n; ++i) {
        if (x[i] < min) min = x[i];
        if (x[i] > max) max = x[i];
        const float wi = w(i);
        sum_w += wi;
        sum_x += wi * x[i];
    }
    if (min > 0) min = 0;
    if (max == min) {
        scale_out = 0.f;
        min_out = -min;
        l_iscale = 0.f;
        l_min = min;
        return;
    }
    auto quant = [&](float is, float mn, int i) {
        const int l = nearest_int(is * (x[i] - mn));
        return l < 0 ? 0 : (l > nmax ? nmax : l);
    };
    float iscale = nmax / (max - min);
    float scale = 1 / iscale;
    float best_error = 0;
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
        float diff = scale * quant(iscale, min, i) + min - x[i];
        diff = diff * diff;
        best_error += w(i) * diff;
    }
    l_iscale = iscale;
    l_min = min;
#pragma unroll 1
    for (int is = 0; is <= nstep; ++is) {
        iscale = (rmin + rdelta * is + nmax) / (max - min);
        float sum_l = 0, sum_l2 = 0, sum_xl = 0;
#pragma unroll 1
        for (int i = 0; i < n; ++i) {
            const int l = quant(iscale, min, i);
            const float wi = w(i);
            sum_l += wi * l;
            sum_l2 += wi * l * l;
            sum_xl += wi * l * x[i];
        }
        const float D = sum_w * sum_l2 - sum_l * sum_l;
        if (D > 0) {
            float this_scale = (sum_w * sum_xl - sum_x * sum_l) / D;
            float this_min = (sum_l2 * sum_x - sum_l * sum_xl) / D;
            if (this_min > 0) {
                this_min = 0;
                this_scale = sum_xl / sum_l2;
            }
            float cur_error = 0;
#pragma unroll 1
            for (int i = 0; i < n; ++i) {
                float diff = this_scale * quant(iscale, min, i) + this_min - x[i];
                diff = diff * diff;
                cur_error += w(i) * diff;
            }
            if (cur_error < best_error) {
                best_error = cur_error;
                scale = this_scale;
                l_iscale = iscale;
                l_min = min;
                min = this_min;
            }
        }
    }
    scale_out = scale;
    min_out = -min;
}

// The same search with float quants (see above): the scale, *the_min, and what
// the winning quants come from (iscale and the min they were taken against).
// Returns false (nothing written) where the general form has to run.
__device__ __forceinline__ bool qkx2_32_fast(const float* x, const float* w, float& scale_out, float& min_out,
                                             float& l_iscale, float& l_min) {
    const float nmax = 15.f, rmin = -1.f, rdelta = 0.1f;
    float min = x[0], max = x[0], fin = x[0] * 0.0f;
    float sum_w = w[0];
    float sum_x = sum_w * x[0];
#pragma unroll
    for (int i = 1; i < 32; ++i) {
        if (x[i] < min) min = x[i];
        if (x[i] > max) max = x[i];
        fin = __builtin_fmaf(x[i], 0.0f, fin);
        sum_w += w[i];
        sum_x += w[i] * x[i];
    }
    const float lo = min;   // the smallest value (min may be clamped to 0, then moves)
    if (min > 0) min = 0;
    if (!(fin == 0.0f)) return false;
    if (max == min) {
        scale_out = 0.f;
        min_out = -min;
        l_iscale = 0.f;     // quants all 0
        l_min = min;
        return true;
    }
    float iscale = nmax / (max - min);
    float scale = 1 / iscale;
    auto in_range = [&](float is, float mn) {   // x -> is * (x - mn) is monotonic: its ends bound it
        return __builtin_fabsf(is * (max - mn)) < 2097152.f && __builtin_fabsf(is * (lo - mn)) < 2097152.f;
    };
    auto quant = [&](float xi, float is, float mn) {
        return __builtin_amdgcn_fmed3f(is * (xi - mn) + QMAGIC, QMAGIC, QMAGIC + 15.f) - QMAGIC;
    };
    if (!in_range(iscale, min)) return false;
    float best_error = 0;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        float diff = scale * quant(x[i], iscale, min) + min - x[i];
        diff = diff * diff;
        best_error += w[i] * diff;
    }
    l_iscale = iscale;
    l_min = min;
    bool ok = true;
#pragma unroll 1
    for (int is = 0; is <= 20; ++is) {
        iscale = (rmin + rdelta * is + nmax) / (max - min);
        ok = ok && in_range(iscale, min);
        float sum_l = 0, sum_l2 = 0, sum_xl = 0;
        float l[32];
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            l[i] = quant(x[i], iscale, min);
            const float wl = w[i] * l[i];
            sum_l += wl;
            sum_l2 += wl * l[i];
            sum_xl += wl * x[i];
        }
        const float D = sum_w * sum_l2 - sum_l * sum_l;
        if (D > 0) {
            float this_scale = (sum_w * sum_xl - sum_x * sum_l) / D;
            float this_min = (sum_l2 * sum_x - sum_l * sum_xl) / D;
            if (this_min > 0) {
                this_min = 0;
                this_scale = sum_xl / sum_l2;
            }
            float cur_error = 0;
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                float diff = this_scale * l[i] + this_min - x[i];
                diff = diff * diff;
                cur_error += w[i] * diff;
            }
            if (cur_error < best_error) {
                best_error = cur_error;
                scale = this_scale;
                l_iscale = iscale;
                l_min = min;
                min = this_min;
            }
        }
    }
    scale_out = scale;
    min_out = -min;
    return ok;
}

// 8 threads per Q4_K super-block; thread j owns sub-block j (32 values).
// AL: src and dst 16-byte aligned (16-byte loads, 16-byte stores of the quants).
template <bool AL>
__global__ void __launch_bounds__(256) k_quant_w_q4K(const float* __restrict__ src, int64_t nblocks,
                                                     BlockQ4_K* __restrict__ dst) {
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t blk = gid >> 3;
    const int j = (int) (gid & 7);
    const bool valid = blk < nblocks;
    const float* x = src + (valid ? blk : 0) * QK_K + 32 * j;
    float xv[32], wv[32];
    float sum_x2 = 0;
#pragma unroll
    for (int l = 0; l < 32; l += 4) {
        if constexpr (AL) {
            const float4 v = *(const float4*) (x + l);
            xv[l] = v.x; xv[l + 1] = v.y; xv[l + 2] = v.z; xv[l + 3] = v.w;
        } else {
            for (int u = 0; u < 4; ++u) xv[l + u] = x[l + u];
        }
    }
#pragma unroll
    for (int l = 0; l < 32; ++l) sum_x2 += xv[l] * xv[l];
    const float av_x = sqrtf(sum_x2 / 32);
#pragma unroll
    for (int l = 0; l < 32; ++l) wv[l] = av_x + __builtin_fabsf(xv[l]);
    float sc, mn, l_iscale, l_min;
    const bool fast = qkx2_32_fast(xv, wv, sc, mn, l_iscale, l_min);
    if (!fast) qkx2_32_general(x, av_x, sc, mn, l_iscale, l_min);
    // super-block maxima over the 8 sub-blocks, in sub-block order (strict >)
    float max_scale = 0, max_min = 0;
    float scales[8], mins[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        scales[t] = __shfl(sc, (threadIdx.x & ~7) + t);
        mins[t] = __shfl(mn, (threadIdx.x & ~7) + t);
        if (scales[t] > max_scale) max_scale = scales[t];
        if (mins[t] > max_min) max_min = mins[t];
    }
    if (!valid) return;
    const float inv_scale = max_scale > 0 ? 63.f / max_scale : 0.f;
    const float inv_min = max_min > 0 ? 63.f / max_min : 0.f;
    uint8_t sbytes[12];
#pragma unroll
    for (int t = 0; t < 12; ++t) sbytes[t] = 0;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        uint8_t ls = (uint8_t) nearest_int(inv_scale * scales[t]);
        uint8_t lm = (uint8_t) nearest_int(inv_min * mins[t]);
        ls = ls < 63 ? ls : 63;
        lm = lm < 63 ? lm : 63;
        if (t < 4) {
            sbytes[t] = ls;
            sbytes[t + 4] = lm;
        } else {
            sbytes[t + 4] = (uint8_t) ((ls & 0xF) | ((lm & 0xF) << 4));
            sbytes[t - 4] |= (uint8_t) ((ls >> 4) << 6);
            sbytes[t - 0] |= (uint8_t) ((lm >> 4) << 6);
        }
    }
    const uint16_t dh = f2h(max_scale / 63.f), mh = f2h(max_min / 63.f);
    // sub-block j's 6-bit scale and min out of the packed bytes (selects, so that
    // the bytes stay in registers)
    int scj = 0, mj = 0;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        int s_, m_;
        scale_min_k4(t, sbytes, s_, m_);
        scj = j == t ? s_ : scj;
        mj = j == t ? m_ : mj;
    }
    const float d = h2f(dh) * scj, dm = h2f(mh) * mj;
    uint32_t L4[8];   // the quants, four bytes per word; the search's own where the scale rounds to 0
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        uint32_t w4 = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float xi = xv[4 * q + u];
            int l = nearest_int(d != 0.0f ? (xi + dm) / d : l_iscale * (xi - l_min));
            l = l < 0 ? 0 : (l > 15 ? 15 : l);
            w4 |= (uint32_t) l << (8 * u);
        }
        L4[q] = w4;
    }
    // sub-block j = 2 c + h: nibble h of qs[32 c ..].  The pair's threads exchange
    // their quants; thread h writes bytes 16 h .. 16 h + 15 of the 32.
    BlockQ4_K* y = dst + blk;
    const int c = j >> 1, h = j & 1;
    uint32_t o4[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t lo_mine = L4[q], hi_mine = L4[q + 4];
        const uint32_t send = h ? lo_mine : hi_mine;            // what the partner writes
        const uint32_t keep = h ? hi_mine : lo_mine;
        const uint32_t got = (uint32_t) dpp_i<DPP_XOR1>((int) send);
        o4[q] = h ? (got | (keep << 4)) : (keep | (got << 4));
    }
    if constexpr (AL) {
        *(u32x4*) &y->qs[32 * c + 16 * h] = u32x4{o4[0], o4[1], o4[2], o4[3]};
    } else {
        for (int l = 0; l < 16; ++l) y->qs[32 * c + 16 * h + l] = (uint8_t) (o4[l >> 2] >> (8 * (l & 3)));
    }
    if (j == 0) {
        y->d = dh;
        y->dmin = mh;
        for (int t = 0; t < 12; ++t) y->scales[t] = sbytes[t];
    }
}

// make_qx_quants(16, 32, x, L, rmse_type = 1, NULL) of the 16 values at x, step for
// step with ggml's integer quants: the general form (rolled loops over memory).  The
// quants are those of nearest_int(l_iscale * x) + 32, or all 0 (zero).
__device__ __forceinline__ void qx_16_general(const float* x, float& scale_out, float& l_iscale, bool& zero) {
    const int n = 16, nmax = 32;
    float max = 0, amax = 0;
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
        const float ax = __builtin_fabsf(x[i]);
        if (ax > amax) { amax = ax; max = x[i]; }
    }
    scale_out = 0.f;
    l_iscale = 0.f;
    zero = amax < 1e-15f;
    if (zero) return;
    auto sums = [&](float is, float& sumlx, float& suml2) {
        sumlx = suml2 = 0;
#pragma unroll 1
        for (int i = 0; i < n; ++i) {
            int l = nearest_int(is * x[i]);
            l = l < -nmax ? -nmax : (l > nmax - 1 ? nmax - 1 : l);
            const float w = x[i] * x[i];
            sumlx += w * x[i] * l;
            suml2 += w * l * l;
        }
    };
    float iscale = -nmax / max, sumlx, suml2;
    sums(iscale, sumlx, suml2);
    l_iscale = iscale;
    float scale = suml2 ? sumlx / suml2 : 0.0f;
    float best = scale * sumlx;
#pragma unroll 1
    for (int is = -9; is <= 9; ++is) {
        if (is == 0) continue;
        iscale = -(nmax + 0.1f * is) / max;
        sums(iscale, sumlx, suml2);
        if (suml2 > 0 && sumlx * sumlx > best * suml2) {
            l_iscale = iscale;
            scale = sumlx / suml2;
            best = scale * sumlx;
        }
    }
    scale_out = scale;
}

// The same search with float quants: the scale and the winning quants' iscale.
// False where the general form has to run (a value that is not finite; a finite
// one's scaled value is at most 33 in magnitude).
__device__ __forceinline__ bool qx_16_fast(const float* x, float& scale_out, float& l_iscale, bool& zero) {
    const float nmax = 32.f;
    float max = 0, amax = 0, fin = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float ax = __builtin_fabsf(x[i]);
        if (ax > amax) { amax = ax; max = x[i]; }
        fin = __builtin_fmaf(x[i], 0.0f, fin);
    }
    if (!(fin == 0.0f)) return false;
    scale_out = 0.f;
    l_iscale = 0.f;
    zero = amax < 1e-15f;
    if (zero) return true;
    float w[16], wx[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        w[i] = x[i] * x[i];
        wx[i] = w[i] * x[i];
    }
    float iscale = -nmax / max;
    auto sums = [&](float is, float& sumlx, float& suml2) {
        sumlx = suml2 = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float l = __builtin_amdgcn_fmed3f(is * x[i] + QMAGIC, QMAGIC - 32.f, QMAGIC + 31.f) - QMAGIC;
            sumlx += wx[i] * l;
            suml2 += w[i] * l * l;
        }
    };
    float sumlx, suml2;
    sums(iscale, sumlx, suml2);
    l_iscale = iscale;
    float scale = suml2 ? sumlx / suml2 : 0.0f;
    float best = scale * sumlx;
#pragma unroll 1
    for (int is = -9; is <= 9; ++is) {
        if (is == 0) continue;
        iscale = -(nmax + 0.1f * is) / max;
        sums(iscale, sumlx, suml2);
        if (suml2 > 0 && sumlx * sumlx > best * suml2) {
            l_iscale = iscale;
            scale = sumlx / suml2;
            best = scale * sumlx;
        }
    }
    scale_out = scale;
    return true;
}

// 16 threads per Q6_K super-block; thread ib owns sub-block ib (16 values).
// AL: src 16-byte and dst 2-byte aligned.
template <bool AL>
__global__ void __launch_bounds__(256) k_quant_w_q6K(const float* __restrict__ src, int64_t nblocks,
                                                     BlockQ6_K* __restrict__ dst) {
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t blk = gid >> 4;
    const int ib = (int) (gid & 15);
    const bool valid = blk < nblocks;
    const float* x = src + (valid ? blk : 0) * QK_K + 16 * ib;
    float xv[16];
#pragma unroll
    for (int l = 0; l < 16; l += 4) {
        if constexpr (AL) {
            const float4 v = *(const float4*) (x + l);
            xv[l] = v.x; xv[l + 1] = v.y; xv[l + 2] = v.z; xv[l + 3] = v.w;
        } else {
            for (int u = 0; u < 4; ++u) xv[l + u] = x[l + u];
        }
    }
    float sc, l_iscale;
    bool zero;
    if (!qx_16_fast(xv, sc, l_iscale, zero)) qx_16_general(x, sc, l_iscale, zero);
    float max_scale = 0, max_abs_scale = 0;
    const int base = threadIdx.x & ~15;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const float s = __shfl(sc, base + t);
        const float as = __builtin_fabsf(s);
        if (as > max_abs_scale) { max_abs_scale = as; max_scale = s; }
    }
    if (!valid) return;
    BlockQ6_K* y = dst + blk;
    int8_t my_scale = 0;
    uint16_t dh = 0;
    uint32_t L4[4] = {0u, 0u, 0u, 0u};   // the quants (+ 32), four bytes per word
    if (max_abs_scale < 1e-15f) {
        dh = f2h(0.f);   // block is all zeros (memset in the reference)
    } else {
        const float iscale = -128.f / max_scale;
        dh = f2h(1 / iscale);
        const int q = nearest_int(iscale * sc);
        my_scale = (int8_t) (q < 127 ? q : 127);
        const float d = h2f(dh) * my_scale;
        // (the search's own quants where the scale rounds to 0)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t w4 = 0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float xi = xv[4 * k + u];
                int l = nearest_int(d != 0.0f ? xi / d : l_iscale * xi);
                l = l < -32 ? -32 : (l > 31 ? 31 : l);
                w4 |= (uint32_t) (l + 32) << (8 * u);
            }
            L4[k] = d == 0.0f && zero ? 0u : w4;
        }
    }
    // Packing (quantize_row_q6_K_ref): element e = 128*jj + 32*m + l (l < 32) ->
    // ql[64*jj + 32*(m&1) + l] nibble (m>>1), qh[32*jj + l] bits 2m..2m+1.
    // Thread ib holds elements 16*ib .. 16*ib+15: jj = ib/8, m = (ib%8)/2, l0 = 16*(ib&1).
    const int jj = ib >> 3, m = (ib & 7) >> 1, l0 = 16 * (ib & 1);
    // The four m-threads sharing (jj, l0) see each other's quants; m = 0 and 1 write
    // ql's 16 bytes of their half (with m + 2's high nibbles), m = 2 writes qh's.
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int v = (int) L4[k], s0 = base + jj * 8 + (ib & 1);
        const uint32_t v0 = (uint32_t) __shfl(v, s0), v1 = (uint32_t) __shfl(v, s0 + 2);
        const uint32_t v2 = (uint32_t) __shfl(v, s0 + 4), v3 = (uint32_t) __shfl(v, s0 + 6);
        const uint32_t lo = m & 1 ? v1 : v0, hi = m & 1 ? v3 : v2;
        const uint32_t qlw = (lo & 0x0F0F0F0Fu) | ((hi & 0x0F0F0F0Fu) << 4);
        const uint32_t qhw = ((v0 >> 4) & 0x03030303u) | (((v1 >> 4) & 0x03030303u) << 2) |
                             (((v2 >> 4) & 0x03030303u) << 4) | (((v3 >> 4) & 0x03030303u) << 6);
        const uint32_t w4 = m == 2 ? qhw : qlw;
        uint8_t* o = (m == 2 ? y->qh + 32 * jj + l0 : y->ql + 64 * jj + 32 * (m & 1) + l0) + 4 * k;
        if (m < 3) {
            if constexpr (AL) {   // 210-byte blocks: 2-byte aligned
                ((uint16_t*) o)[0] = (uint16_t) w4;
                ((uint16_t*) o)[1] = (uint16_t) (w4 >> 16);
            } else {
                for (int u = 0; u < 4; ++u) o[u] = (uint8_t) (w4 >> (8 * u));
            }
        }
    }
    y->scales[ib] = my_scale;
    if (ib == 0) y->d = dh;
}

// Q8_0 weights (quantize_row_q8_0_ref): one thread per 32-value block.
__global__ void __launch_bounds__(256) k_quant_w_q8_0(const float* __restrict__ src, int64_t nblocks,
                                                      BlockQ8_0* __restrict__ dst) {
    const int64_t blk = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (blk >= nblocks) return;
    const float* x = src + blk * QK8_0;
    float amax = 0.0f;
    for (int j = 0; j < QK8_0; j++) amax = fmaxf(amax, __builtin_fabsf(x[j]));
    const float d = amax / ((1 << 7) - 1);
    const float id = d ? 1.0f / d : 0.0f;
    BlockQ8_0* y = dst + blk;
    y->d = f2h(d);
    for (int j = 0; j < QK8_0; ++j) y->qs[j] = (int8_t) roundf(x[j] * id);
}

int launch_quantize_weights(int type, const float* src, int64_t n, void* dst, hipStream_t stream) {
    if (type == T_Q4_K) {
        const int64_t nb = n / QK_K;
        const dim3 grid((unsigned) ((nb * 8 + 255) / 256));
        if ((((uintptr_t) src | (uintptr_t) dst) & 15) == 0)
            hipLaunchKernelGGL(k_quant_w_q4K<true>, grid, dim3(256), 0, stream, src, nb, (BlockQ4_K*) dst);
        else
            hipLaunchKernelGGL(k_quant_w_q4K<false>, grid, dim3(256), 0, stream, src, nb, (BlockQ4_K*) dst);
    } else if (type == T_Q6_K) {
        const int64_t nb = n / QK_K;
        const dim3 grid((unsigned) ((nb * 16 + 255) / 256));
        if (((uintptr_t) src & 15) == 0 && ((uintptr_t) dst & 1) == 0)
            hipLaunchKernelGGL(k_quant_w_q6K<true>, grid, dim3(256), 0, stream, src, nb, (BlockQ6_K*) dst);
        else
            hipLaunchKernelGGL(k_quant_w_q6K<false>, grid, dim3(256), 0, stream, src, nb, (BlockQ6_K*) dst);
    } else if (type == T_Q8_0) {
        const int64_t nb = n / QK8_0;
        hipLaunchKernelGGL(k_quant_w_q8_0, dim3((unsigned) ((nb + 255) / 256)), dim3(256), 0, stream, src, nb,
                           (BlockQ8_0*) dst);
    } else {
        return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

// ---------------------------------------------------------------------------
// Dequantizers (dequantize_row_q8_0 / _q4_K / _q6_K, ggml-quants.c:553-566,
// 1529-1551, 1939-1968).  A thread forms 8 (Q4_K: four bytes' low and high nibbles;
// Q8_0) or 16 values (Q6_K: the four values of four positions) and writes them as
// 16-byte stores; k_dequant, one thread per value, where y is not 16-byte
// or the blocks not 2-byte (Q4_K 4-byte) aligned.  Bound: HBM.  12288 x 2048 values
// of Q4_K: 55 -> 19 us (115 MB; Q6_K 61 -> 20, Q8_0 36 -> 21).
__device__ __forceinline__ uint32_t ld32_a2(const void* p) {   // a 2-byte aligned word
    const uint16_t* q = (const uint16_t*) p;
    return (uint32_t) q[0] | ((uint32_t) q[1] << 16);
}

template <int TYPE>
__global__ void __launch_bounds__(256) k_dequant_v(const uint8_t* __restrict__ x, float* __restrict__ y, int64_t n) {
    constexpr int PER = TYPE == T_Q6_K ? 16 : 8;   // values per thread
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (i * PER >= n) return;
    if constexpr (TYPE == T_Q8_0) {
        const int64_t blk = i >> 2;
        const int s = (int) (i & 3);
        const uint8_t* b = x + 34 * blk;
        const float d = h2f(*(const uint16_t*) b);
        const uint32_t w0 = ld32_a2(b + 2 + 8 * s), w1 = ld32_a2(b + 6 + 8 * s);
        auto v = [&](uint32_t w, int k) { return (float) (int8_t) (w >> (8 * k)) * d; };
        float4* o = (float4*) (y + 8 * i);
        o[0] = float4{v(w0, 0), v(w0, 1), v(w0, 2), v(w0, 3)};
        o[1] = float4{v(w1, 0), v(w1, 1), v(w1, 2), v(w1, 3)};
    } else if constexpr (TYPE == T_Q4_K) {
        const int64_t blk = i >> 5;
        const int c = (int) (i & 31) >> 3, j = (int) (i & 7);
        const BlockQ4_K* b = (const BlockQ4_K*) (x + 144 * blk);
        const uint32_t w = *(const uint32_t*) (b->qs + 32 * c + 4 * j);
        const uint32_t h = *(const uint32_t*) b;
        int s0, m0, s1, m1;
        scale_min_k4(2 * c, b->scales, s0, m0);
        scale_min_k4(2 * c + 1, b->scales, s1, m1);
        const float dd = h2f((uint16_t) (h & 0xffffu)), dm = h2f((uint16_t) (h >> 16));
        const float d0 = dd * s0, n0 = dm * m0, d1 = dd * s1, n1 = dm * m1;
        auto lo = [&](int k) { return d0 * (float) (int) ((w >> (8 * k)) & 0xFu) - n0; };
        auto hi = [&](int k) { return d1 * (float) (int) ((w >> (8 * k + 4)) & 0xFu) - n1; };
        float* o = y + 256 * blk + 64 * c + 4 * j;
        *(float4*) o = float4{lo(0), lo(1), lo(2), lo(3)};
        *(float4*) (o + 32) = float4{hi(0), hi(1), hi(2), hi(3)};
    } else {
        const int64_t blk = i >> 4;
        const int half = (int) (i & 15) >> 3, j = (int) (i & 7);   // positions l = 4 j .. + 3
        const BlockQ6_K* b = (const BlockQ6_K*) (x + 210 * blk);
        const uint32_t a = ld32_a2(b->ql + 64 * half + 4 * j), c = ld32_a2(b->ql + 64 * half + 32 + 4 * j);
        const uint32_t h = ld32_a2(b->qh + 32 * half + 4 * j);
        const float d = h2f(*(const uint16_t*) &b->d);
        float* o = y + 256 * blk + 128 * half + 4 * j;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const uint32_t q = (((m & 1 ? c : a) >> (m >= 2 ? 4 : 0)) & 0x0F0F0F0Fu) | (((h >> (2 * m)) & 0x03030303u) << 4);
            const float s = d * b->scales[8 * half + (j >> 2) + 2 * m];
            auto v = [&](int k) { return s * (float) ((int) ((q >> (8 * k)) & 63u) - 32); };
            *(float4*) (o + 32 * m) = float4{v(0), v(1), v(2), v(3)};
        }
    }
}

// One thread per output value.
__global__ void k_dequant(int type, const uint8_t* __restrict__ x, float* __restrict__ y, int64_t n) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (type == T_Q8_0) {
        const BlockQ8_0* b = (const BlockQ8_0*) x + i / QK8_0;
        y[i] = b->qs[i % QK8_0] * h2f(b->d);
    } else if (type == T_Q4_K) {
        const BlockQ4_K* b = (const BlockQ4_K*) x + i / QK_K;
        const int e = (int) (i % QK_K);
        const int c = e / 64, within = e % 64, hi = within >= 32, l = within & 31;
        int sc, m;
        scale_min_k4(2 * c + hi, b->scales, sc, m);
        const float d = h2f(b->d) * sc, mn = h2f(b->dmin) * m;
        const int q = hi ? (b->qs[32 * c + l] >> 4) : (b->qs[32 * c + l] & 0xF);
        y[i] = d * q - mn;
    } else if (type == T_Q6_K) {
        const BlockQ6_K* b = (const BlockQ6_K*) x + i / QK_K;
        const int e = (int) (i % QK_K);
        const int half = e / 128, r = e % 128, m = r / 32, l = r % 32;
        const uint8_t* ql = b->ql + 64 * half;
        const uint8_t* qh = b->qh + 32 * half;
        int q;
        switch (m) {
            case 0: q = (ql[l] & 0xF) | (((qh[l] >> 0) & 3) << 4); break;
            case 1: q = (ql[l + 32] & 0xF) | (((qh[l] >> 2) & 3) << 4); break;
            case 2: q = (ql[l] >> 4) | (((qh[l] >> 4) & 3) << 4); break;
            default: q = (ql[l + 32] >> 4) | (((qh[l] >> 6) & 3) << 4); break;
        }
        const int is = l / 16;
        y[i] = h2f(b->d) * b->scales[8 * half + is + 2 * m] * (float) (q - 32);
    }
}

int launch_dequantize(int type, const void* x, float* y, int64_t n, hipStream_t stream) {
    if (n <= 0) return 0;
    if (((uintptr_t) y & 15) == 0 && ((uintptr_t) x & (type == T_Q4_K ? 3 : 1)) == 0) {
        const int64_t thr = n / (type == T_Q6_K ? 16 : 8);   // (n is whole blocks)
        const dim3 grid((unsigned) ((thr + 255) / 256));
        const uint8_t* xb = (const uint8_t*) x;
        if (type == T_Q4_K) hipLaunchKernelGGL(k_dequant_v<T_Q4_K>, grid, dim3(256), 0, stream, xb, y, n);
        else if (type == T_Q6_K) hipLaunchKernelGGL(k_dequant_v<T_Q6_K>, grid, dim3(256), 0, stream, xb, y, n);
        else hipLaunchKernelGGL(k_dequant_v<T_Q8_0>, grid, dim3(256), 0, stream, xb, y, n);
        return hipGetLastError() == hipSuccess ? 0 : -3;
    }
    hipLaunchKernelGGL(k_dequant, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, stream, type, (const uint8_t*) x,
                       y, n);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

// ---------------------------------------------------------------------------
// Seeded N(mean, std) fp32 generator for synthetic weights and inputs:
// splitmix64 over (seed, index) and a Box-Muller pair.  Deterministic on the
// GPU for a given seed; not meant to match any CPU generator bit for bit.
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__global__ void k_randn(float* __restrict__ y, int64_t n, uint64_t seed, float mean, float stddev) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t pair = i >> 1;
    if (2 * pair >= n) return;
    const uint64_t r = splitmix64(seed * 0x9e3779b97f4a7c15ull ^ splitmix64((uint64_t) pair));
    const float u1 = ((float) (r >> 40) + 1.0f) * (1.0f / 16777216.0f);  // (0, 1]
    const float u2 = (float) ((r >> 16) & 0xffffff) * (1.0f / 16777216.0f);
    const float rad = sqrtf(-2.0f * logf(u1));
    const float ang = 6.283185307179586f * u2;
    const float z = (i & 1) ? rad * sinf(ang) : rad * cosf(ang);
    if (i < n) y[i] = mean + stddev * z;
}

int launch_randn(float* y, int64_t n, uint64_t seed, float mean, float stddev, hipStream_t stream) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_randn, dim3((unsigned) ((n + 1 + 255) / 256)), dim3(256), 0, stream, y, n, seed, mean, stddev);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace qw
