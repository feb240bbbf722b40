// attn.hip -- the attention half of a Qwen3 decoder layer's Seg A
// (core/runtime.cpp:1976-2030, build_attn 681-734 on its manual path, RoPE by
// apply_rope 290-300): per-head RMSNorm and NEOX RoPE of Q and K, the f16 KV
// cache write, causal GQA scores, ggml's soft_max_ext and the P.V product,
// then the residual and the FFN input norm.  The four projections run on the
// quantized mul_mat kernels (a one-expert mul_mat_id; api.cpp).
//
// Layout in HBM: Q [T][n_head][128] f16 after RoPE; the caller's caches
// [n_ctx][n_head_kv * 128] f16 (ggml's k_cache / v_cache rows); each row's softmax
// statistics per key split, and the P.V sums [split][T][n_head][128].
//
// ggml converts the second operand of a mul_mat with an f16 first operand to
// f16 (vec_dot_type), so Q is rounded to f16 before the scores and the
// normalized probabilities before P.V, as here; sums run in fp32.  Outputs agree with the CPU backend to float
// rounding of the fp32 sums (the 1e-3 bar); they are not bit-identical.
#include <hip/hip_fp16.h>

#include <type_traits>

#include "qw_mfma.hpp"

namespace qw {

namespace {

constexpr int AD = 128;   // head dimension (Qwen3: n_embd_head_k = n_embd_head_v = 128)

typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

// Head rows of one token: Q and K heads get ggml_rms_norm (sum of squares in
// double) * norm weight and NEOX RoPE; K and V heads go to the caches at row
// n_past + t.  A wave per head row, lane i holds elements i and i + 64: NEOX's
// pair.  Block (t, y) takes head rows y * hpb ..; its cosines and sines (the same
// for every head) are formed once, in LDS.  A wave takes RB rows at a time, whose
// loads and double sums overlap: a row alone is a load and six dependent shuffles of
// a double.  T = 512, 40 head rows: 13.2 us a row at a time, a block per
// token -> 8.8, five rows at a time, two blocks.  Few tokens take a row per wave.
template <int RB>
__global__ void __launch_bounds__(256) k_attn_qk_rope(AttnArgs a, int hpb) {
    __shared__ float s_c[AD / 2], s_s[AD / 2];
    const int t = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nq = a.n_head, nk = a.n_head_kv, gqa = nk * AD;
    const int64_t pos = a.n_past + t;
    const int r0 = blockIdx.y * hpb, r1 = min(r0 + hpb, nq + 2 * nk);
    if (w == 0 && r0 < nq + nk) {
        // ggml_rope_cache_init: theta_0 = pos, theta_{i+1} = theta_i * theta_scale (fp32, in order)
        float th = (float) pos;
        for (int i = 0; i < lane; ++i) th = th * a.theta_scale;
        s_c[lane] = cosf(th);
        s_s[lane] = sinf(th);
    }
    __syncthreads();
    const float wq0 = a.q_norm[lane], wq1 = a.q_norm[lane + 64], wk0 = a.k_norm[lane], wk1 = a.k_norm[lane + 64];
    for (int rb = r0 + w; rb < r1; rb += 4 * RB) {
        float x0[RB], x1[RB];
        double s[RB];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const int r = min(rb + 4 * i, r1 - 1);
            const float* src = r < nq        ? a.q + ((int64_t) t * nq + r) * AD
                               : r < nq + nk ? a.k + (int64_t) t * gqa + (r - nq) * AD
                                             : a.v + (int64_t) t * gqa + (r - nq - nk) * AD;
            x0[i] = src[lane];
            x1[i] = src[lane + 64];
        }
#pragma unroll
        for (int i = 0; i < RB; ++i) s[i] = (double) (x0[i] * x0[i]) + (double) (x1[i] * x1[i]);
        for (int off = 32; off >= 1; off >>= 1) {
#pragma unroll
            for (int i = 0; i < RB; ++i) s[i] += __shfl_xor(s[i], off);
        }
        const float c = s_c[lane], sn = s_s[lane];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const int r = rb + 4 * i;
            if (r >= r1) break;
            float o0 = x0[i], o1 = x1[i];
            if (r < nq + nk) {
                const float mean = (float) (s[i] / (double) AD);
                const float scale = 1.0f / sqrtf(mean + a.eps);
                const float y0 = (o0 * scale) * (r < nq ? wq0 : wk0), y1 = (o1 * scale) * (r < nq ? wq1 : wk1);
                o0 = y0 * c - y1 * sn;
                o1 = y0 * sn + y1 * c;
            }
            __half* dst = r < nq        ? (__half*) a.qr + ((int64_t) t * nq + r) * AD
                          : r < nq + nk ? (__half*) a.kc + pos * gqa + (r - nq) * AD
                                        : (__half*) a.vc + pos * gqa + (r - nq - nk) * AD;
            dst[lane] = __float2half_rn(o0);
            dst[lane + 64] = __float2half_rn(o1);
        }
    }
}

// ---- scores, softmax and P.V on the matrix cores --------------------------------
//
// Rows r = t R + h (token-major) of kv head g, 32 per wave; a workgroup of NW waves
// takes 32 NW rows and one split of the keys, 64 keys at a time.  Two kernels: the
// statistics (each row's maximum and sum of exponentials over a split), then, with
// every split's statistics known, the scores again beside P.V -- ggml rounds the
// normalized probabilities to f16, so the sum has to be known before the first
// product, and forming scores twice costs less than writing them (4 n_head T n_kv
// bytes).  A third adds the splits (k_attn_combine).
//
// Scores are formed transposed, S^T = K Q^T, by v_mfma_f32_32x32x16_f16: lane l of
// A holds key l % 32, dims 8 (l / 32) .. + 7 of a 16-dim step; B the row l % 32
// likewise; D register i of lane l is key 8 (i / 4) + 4 (l / 32) + i % 4 of row l % 32.
// A lane so holds scores of one row: maximum, sum and normalisation are lane
// scalars.  The probabilities, as they lie in D, are the B operand of O^T = V^T P^T with
// the keys of a 16-key step in the order (4 h .. + 3, 8 + 4 h .. + 3) for lane half h;
// V^T is read in that order.
//
// K rows are copied straight into LDS one chunk ahead (two buffers), 16-byte chunk
// c of key k at position c ^ (k % 16): 32 lanes reading one chunk of 32 keys hit
// distinct banks.  V rows come through registers, also a chunk ahead, and are
// stored transposed, four keys of a dim as one 8-byte store at quad position
// q ^ (dim / 2 % 16).
//
// The probabilities are ggml's: ggml_v_expf of score / sqrt(D) less the row's maximum,
// times 1 / S, S in double over the splits (k_attn_stat).
//
// Bound: latency and VALU (the exponentials), not memory or matrix cores.  30B
// heads, T = 512 behind 1037 keys: 233 us (16-row tiles of v_mfma_f32_16x16x16_f16 and
// one workgroup per CU) -> 61 us for the three (15.7, 36.0, 9.4; 52 with the hardware's
// exp2 of a fused product for ggml_v_expf, which moved one probability in 500 by an f16
// step); T = 1 at 3000 keys: 34.1 us (dot products on the VALU, scores through memory) ->
// 18.8 us (5.0, 9.4, 4.4).
constexpr int FK = 64;   // keys per chunk

// What both kernels know of a wave's rows and its workgroup's keys.
struct AttnTile {
    int64_t row_id;    // t * n_head + head of this lane's row
    int64_t k0;        // first key of the split
    int nkeys;         // keys of the split some row of the workgroup sees (<= 0: none)
    int vis;           // this lane's row: the last key it sees, relative to k0 (rows past the end: -1)
    int vis_all;       // keys up to here are visible to every row of the workgroup
    int wrows;         // rows of this wave (<= 0: none)
    bool row_ok;
};
template <int NW>
__device__ __forceinline__ AttnTile attn_tile(const AttnArgs& a, int w, int li, int64_t k0, int64_t keys) {
    const int g = blockIdx.x, nq = a.n_head, R = nq / a.n_head_kv;
    const int64_t rows = (int64_t) a.T * R, row0 = (int64_t) blockIdx.y * (32 * NW), r = row0 + 32 * w + li;
    AttnTile x;
    x.row_ok = r < rows;
    x.wrows = (int) min(rows - row0 - 32 * w, (int64_t) 32);
    const int t = x.row_ok ? (int) (r / R) : 0, hd = x.row_ok ? g * R + (int) (r % R) : 0;
    x.row_id = (int64_t) t * nq + hd;
    const int t_last = (int) ((min(rows, row0 + 32 * NW) - 1) / R);
    x.k0 = k0;
    // keys past klim are masked for every row
    const int64_t klim = min(min(a.n_kv, k0 + keys), a.n_past + t_last + 1);
    x.nkeys = (int) max(klim - k0, (int64_t) 0);
    x.vis = x.row_ok ? (int) max(min((int64_t) x.nkeys - 1, a.n_past + t - k0), (int64_t) -1) : -1;
    x.vis_all = (int) max(min((int64_t) x.nkeys - 1, a.n_past + row0 / R - k0), (int64_t) -1);
    return x;
}

// The row's Q as the B operand of S^T.
__device__ __forceinline__ void attn_load_q(const AttnArgs& a, const AttnTile& x, int h, h8 (&qb)[8]) {
    const h8* q = (const h8*) ((const _Float16*) a.qr + x.row_id * AD + 8 * h);
#pragma unroll
    for (int st = 0; st < 8; ++st) qb[st] = x.row_ok ? q[2 * st] : h8{0, 0, 0, 0, 0, 0, 0, 0};
}

// Copies of a chunk's K rows into LDS: instruction j of 16 brings keys 4 j .. 4 j + 3.
// Keys past nkeys are past the buffer's end (no access).
template <int NW>
struct AttnKCopy {
    static constexpr int KI = 16 / NW;
    i32x4 rsrc;
    uint32_t off[KI];
    uint32_t row_bytes;
    int w;
    __device__ __forceinline__ void init(const AttnArgs& a, const AttnTile& x, int w_, int l) {
        const int gqa = a.n_head_kv * AD;
        w = w_;
        row_bytes = 2u * (uint32_t) gqa;
        const i32x4 r = rsrc_words((const _Float16*) a.kc + x.k0 * gqa, (uint32_t) x.nkeys * row_bytes);
        rsrc = i32x4{__builtin_amdgcn_readfirstlane(r.x), __builtin_amdgcn_readfirstlane(r.y),
                     __builtin_amdgcn_readfirstlane(r.z), __builtin_amdgcn_readfirstlane(r.w)};
#pragma unroll
        for (int j = 0; j < KI; ++j) {
            const int key = 4 * (w + NW * j) + (l >> 4);
            off[j] = (uint32_t) key * row_bytes + (uint32_t) (2 * (int) blockIdx.x * AD + 16 * ((l & 15) ^ (key & 15)));
        }
    }
    __device__ __forceinline__ void issue(uint8_t* sk, int c0) const {
        uint32_t lb = (uint32_t) (uintptr_t) sk;
        asm volatile("" : "+s"(lb));
        // (the chunk's offset in the lane offset: it counts for the bounds check)
#pragma unroll
        for (int j = 0; j < KI; ++j) dma_b128(rsrc, lb + 1024u * (uint32_t) (w + NW * j), off[j] + (uint32_t) c0 * row_bytes, 0u);
    }
};

// S^T of 32 keys (32 kk .. of a chunk) and the wave's rows.
__device__ __forceinline__ f16v attn_scores(const uint8_t* sk, int kk, int li, int h, const h8 (&qb)[8]) {
    f16v s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
    for (int st = 0; st < 8; ++st) {
        const h8 ka = *(const h8*) (sk + (32 * kk + li) * (2 * AD) + 16 * ((2 * st + h) ^ (li & 15)));
        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, qb[st], s, 0, 0, 0);
    }
    return s;
}

// v_expf for -80 <= x <= 0, its bits without its branches.  Scores further below the
// maximum are raised to -80: 0 as an f16 probability, and nothing beside a double sum
// of at least 1.
__device__ __forceinline__ float exp_score(float x) {
    const float z = __builtin_fmaf(x, 0x1.715476p+0f, 0x1.8p23f);
    const float n = z - 0x1.8p23f;
    const float b = __builtin_fmaf(-n, 0x1.7f7d1cp-20f, __builtin_fmaf(-n, 0x1.62e4p-1f, x));
    const float k = bitsf((fbits(z) << 23) + 0x3f800000u);
    const float u = b * b;
    const float j = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(0x1.0e4020p-7f, b, 0x1.573e2ep-5f), u,
                                                  __builtin_fmaf(0x1.555e66p-3f, b, 0x1.fffdb6p-2f)),
                                   u, 0x1.ffffecp-1f * b);
    return __builtin_fmaf(k, j, k);
}

// Per row and split of a.split keys: the maximum of its scores and, in double, the sum
// of exponentials (stored as a float); a maximum of -inf where the row sees none of its keys.
// Up to 64 rows (decode, verify) the exponentials are ggml_v_expf's, each added in
// double; more rows form them with the hardware's exp and add sixteen in fp32 first
// (they only normalize: S moves by ~1e-7 of itself, far below the f16 step of p).
template <int NW>
__global__ void __launch_bounds__(64 * NW) k_attn_stat(AttnArgs a) {
    constexpr bool EXACT = NW <= 2;
    __shared__ __align__(16) uint8_t s_k[2][FK * 2 * AD];
    const int l = threadIdx.x & 63, li = l & 31, h = l >> 5;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const AttnTile x = attn_tile<NW>(a, w, li, (int64_t) blockIdx.z * a.split, a.split);
    float* stat = a.stat + 2 * ((int64_t) blockIdx.z * a.T * a.n_head + x.row_id);
    float m = -INFINITY;   // the row's maximum so far (both lanes that hold it)
    double lsum = 0.0;     // over this lane's keys
    if (x.nkeys > 0) {
        h8 qb[8];
        attn_load_q(a, x, h, qb);
        AttnKCopy<NW> kc;
        kc.init(a, x, w, l);
        kc.issue(s_k[0], 0);
        int buf = 0;
        for (int c0 = 0; c0 < x.nkeys; c0 += FK) {
            vm_wait<0>();
            lds_barrier();   // this chunk's copies are there; the other buffer's readers are done
            if (c0 + FK < x.nkeys) kc.issue(s_k[buf ^ 1], c0 + FK);
            f16v s[2];
            float mc = -INFINITY;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                s[kk] = attn_scores(s_k[buf], kk, li, h, qb);
#pragma unroll
                for (int i = 0; i < 16 && EXACT; ++i) s[kk][i] *= a.kq_scale;
                if (c0 + FK - 1 > x.vis_all) {   // uniform
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        s[kk][i] = c0 + 32 * kk + 8 * (i >> 2) + 4 * h + (i & 3) <= x.vis ? s[kk][i] : -INFINITY;
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) mc = fmaxf(mc, s[kk][i]);
            }
            if constexpr (!EXACT) mc *= a.kq_scale;
            mc = fmaxf(mc, __shfl_xor(mc, 32));   // (lane l ^ 32 holds the row's other keys)
            const float mn = fmaxf(m, mc), mu = mn == -INFINITY ? 0.0f : mn;   // (no key yet: every exponential is 0)
            if (__any(mn > m && m != -INFINITY))
                lsum *= m == -INFINITY ? 0.0 : EXACT ? exp((double) m - (double) mn) : (double) __expf(m - mn);
            m = mn;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                if constexpr (EXACT) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const float d = s[kk][i] - mu;
                        lsum += (double) exp_score(d < -80.0f ? -80.0f : d);   // (a NaN stays)
                    }
                } else {
                    float e0 = 0.0f, e1 = 0.0f;
#pragma unroll
                    for (int i = 0; i < 16; i += 2) {
                        e0 += __expf(__builtin_fmaf(s[kk][i], a.kq_scale, -mu));
                        e1 += __expf(__builtin_fmaf(s[kk][i + 1], a.kq_scale, -mu));
                    }
                    lsum += (double) (e0 + e1);
                }
            }
            buf ^= 1;
        }
        lsum += __shfl_xor(lsum, 32);
    }
    if (x.row_ok && h == 0) *(float2*) stat = float2{m, (float) lsum};
}

// P.V sums over a PV split (merge statistics splits of a.split keys each).
template <int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 4 ? 2 : 1, 2))) k_attn_pv(AttnArgs a, int n_split,
                                                                                             int merge) {
    __shared__ __align__(16) uint8_t s_k[2][FK * 2 * AD];
    __shared__ __align__(16) uint8_t s_v[AD * 2 * FK];
    const int tid = threadIdx.x, l = tid & 63, li = l & 31, h = l >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gqa = a.n_head_kv * AD;
    const int64_t keys = a.split * merge, heads = (int64_t) a.T * a.n_head;
    const AttnTile x = attn_tile<NW>(a, w, li, (int64_t) blockIdx.z * keys, keys);
    float* dst = a.part + ((int64_t) blockIdx.z * heads + x.row_id) * AD + 4 * h;
    f16v o[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
    if (x.nkeys > 0) {
        AttnKCopy<NW> kc;
        kc.init(a, x, w, l);
        kc.issue(s_k[0], 0);
        // V units of 4 keys x 4 dims: dims 4 (tid % 32), keys 4 (tid / 32 + 2 NW u)
        constexpr int VU = 8 / NW;
        const _Float16* vbase = (const _Float16*) a.vc + x.k0 * gqa + (int) blockIdx.x * AD + 4 * (tid & 31);
        uint2 vr[VU][4];
        auto load_v = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < VU; ++u)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int key = c0 + 4 * ((tid >> 5) + 2 * NW * u) + k;
                    const uint2 v = *(const uint2*) (vbase + (int64_t) min(key, x.nkeys - 1) * gqa);
                    vr[u][k] = key < x.nkeys ? v : uint2{0u, 0u};
                }
        };
        auto store_v = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                const int kq = (tid >> 5) + 2 * NW * u;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int dim = 4 * (tid & 31) + j;
                    const uint32_t sel = j & 1 ? 0x07060302u : 0x05040100u;   // the odd / even halves of two words
                    auto wd = [&](const uint2& v) { return j & 2 ? v.y : v.x; };
                    const uint2 p = uint2{__builtin_amdgcn_perm(wd(vr[u][1]), wd(vr[u][0]), sel),
                                          __builtin_amdgcn_perm(wd(vr[u][3]), wd(vr[u][2]), sel)};
                    *(uint2*) (s_v + dim * (2 * FK) + 8 * (kq ^ ((dim >> 1) & 15))) = p;
                }
            }
        };
        load_v(0);
        h8 qb[8];
        attn_load_q(a, x, h, qb);
        // each row's maximum M and 1 / S, S = sum_s exp(m_s - M) l_s in double over the
        // splits: 64 / p2 lanes per row, p2 the power of two that holds the wave's rows
        int p2 = 32;
        while (p2 / 2 >= x.wrows && p2 > 1) p2 /= 2;   // uniform
        const int mine = l & (p2 - 1);
        const int64_t rid = __shfl(x.row_id, mine);
        const float2* st = (const float2*) a.stat + rid;
        float M = -INFINITY;
#pragma unroll 4
        for (int s = l / p2; s < n_split; s += 64 / p2) M = fmaxf(M, st[s * heads].x);
        for (int off = p2; off < 64; off <<= 1) M = fmaxf(M, __shfl_xor(M, off));
        double S = 0.0;
#pragma unroll 1
        for (int s = l / p2; s < n_split; s += 64 / p2) {
            const float2 v = st[s * heads];
            if (v.x != -INFINITY) S += exp((double) v.x - (double) M) * (double) v.y;
        }
        for (int off = p2; off < 64; off <<= 1) S += __shfl_xor(S, off);
        // (every score -inf: probabilities 0)
        const float inv1 = __shfl(S == 0.0 ? 0.0f : (float) (1.0 / S), li & (p2 - 1));
        M = __shfl(M == -INFINITY ? 0.0f : M, li & (p2 - 1));
        const float inv = x.row_ok ? inv1 : 0.0f;
        int buf = 0;
        for (int c0 = 0; c0 < x.nkeys; c0 += FK) {
            vm_wait<0>();      // this chunk's K copies and V rows
            lds_barrier();     // every wave is done with the previous chunk
            store_v();
            lds_barrier();
            if (c0 + FK < x.nkeys) {
                kc.issue(s_k[buf ^ 1], c0 + FK);
                load_v(c0 + FK);
            }
#pragma unroll 1
            for (int kk = 0; kk < 2; ++kk) {
                f16v s = attn_scores(s_k[buf], kk, li, h, qb);
#pragma unroll
                for (int i = 0; i < 16; ++i) 
                    s[i] = exp_score(fmaxf(s[i] * a.kq_scale - M, -80.0f)) * inv;   // (a NaN: inv is one too)
                if (c0 + FK - 1 > x.vis_all) {   // uniform
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        s[i] = c0 + 32 * kk + 8 * (i >> 2) + 4 * h + (i & 3) <= x.vis ? s[i] : 0.0f;
                }
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    h8 p;
#pragma unroll
                    for (int i = 0; i < 8; ++i) p[i] = (_Float16) s[8 * ks + i];
#pragma unroll
                    for (int dt = 0; dt < 4; ++dt) {
                        const int dim = 32 * dt + li, q0 = 8 * kk + 4 * ks + h, f = (dim >> 1) & 15;
                        const h4 v0 = *(const h4*) (s_v + dim * (2 * FK) + 8 * (q0 ^ f));
                        const h4 v1 = *(const h4*) (s_v + dim * (2 * FK) + 8 * ((q0 + 2) ^ f));
                        const h8 va = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, p, o[dt], 0, 0, 0);
                    }
                }
            }
            buf ^= 1;
        }
    }
    if (!x.row_ok) return;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *(float4*) (dst + 32 * dt + 8 * j) = float4{o[dt][4 * j], o[dt][4 * j + 1], o[dt][4 * j + 2], o[dt][4 * j + 3]};
}

// att = the sum of the PV splits, a 256-value block per WV waves: wave v adds splits
// v, v + WV, ... in order, then the waves' sums are added in order.  Then the Q8_K of
// the block (and its f16 copy), the attn_output projection's input, or the f32
// values (att).
template <int WV>
__global__ void __launch_bounds__(256) k_attn_combine(AttnArgs a, int n_split) {
    __shared__ float4 s_p[WV > 1 ? 4 : 1][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, v = wv % WV;
    const int64_t n = (int64_t) a.T * a.n_head * AD;   // (an odd number of heads leaves the last block half)
    const int64_t blk = (int64_t) blockIdx.x * (4 / WV) + wv / WV, i0 = blk * 256 + 4 * lane;
    float4 acc = float4{0.0f, 0.0f, 0.0f, 0.0f};
    if (i0 < n) {
#pragma unroll 8
        for (int s = v; s < n_split; s += WV) {
            const float4 x = *(const float4*) (a.part + s * n + i0);
            acc.x += x.x;
            acc.y += x.y;
            acc.z += x.z;
            acc.w += x.w;
        }
    }
    if constexpr (WV > 1) {
        s_p[wv][lane] = acc;
        __syncthreads();
        if (wv > 0) return;
#pragma unroll
        for (int u = 1; u < WV; ++u) {
            const float4 x = s_p[u][lane];
            acc.x += x.x;
            acc.y += x.y;
            acc.z += x.z;
            acc.w += x.w;
        }
    }
    if (blk * 256 >= n) return;
    if (a.att_q8K) {   // (n is a multiple of 256)
        const float vv[4] = {acc.x, acc.y, acc.z, acc.w};
        _Float16* hh = (_Float16*) a.att_h;
        quant_q8K_wave(vv, lane, (BlockQ8_K*) a.att_q8K + blk, hh ? hh + (size_t) blk * QK_K : nullptr,
                       hh ? hh + (size_t) n + (size_t) blk * 16 : nullptr);
    } else if (i0 < n) {
        *(float4*) (a.att + i0) = acc;
    }
}

// resid = x + y (ggml_add), out = rms_norm(resid) * w (k_rms_norm's order); one
// 256-thread block per row of n.
__global__ void __launch_bounds__(256) k_add_rms_norm_mul(const float* __restrict__ x, const float* __restrict__ y,
                                                          float* __restrict__ resid, float* __restrict__ out,
                                                          int64_t n, float eps, const float* __restrict__ w) {
    __shared__ double part[4];
    const int64_t o = (int64_t) blockIdx.x * n;
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += 256) {
        const float v = x[o + i] + y[o + i];
        resid[o + i] = v;
        s += (double) (v * v);
    }
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (!out) return;
    const double tot = (part[0] + part[1]) + (part[2] + part[3]);
    const float mean = (float) (tot / (double) n);
    const float scale = 1.0f / sqrtf(mean + eps);
    for (int64_t i = threadIdx.x; i < n; i += 256) out[o + i] = (resid[o + i] * scale) * w[i];
}

// Row t's part of the groupings (one thread per row).
__device__ __forceinline__ void row_groups(const RowGroups& g, int t, int T) {
    if (g.rows) {
        g.rows[2 * t] = 0;
        g.rows[2 * t + 1] = t;
        if (t == 0) {
            g.active[0] = 0;
            g.active_off[0] = 0;
            g.active_off[1] = T;
            *g.n_active = 1;
        }
    }
    if (g.trows) {
        g.trows[2 * t] = 0;
        g.trows[2 * t + 1] = t;
        const int nb = (T + g.tpb - 1) / g.tpb;
        if (t % g.tpb == 0) {
            g.tactive[t / g.tpb] = t / g.tpb;
            g.toff[t / g.tpb] = t;
            g.tslot[t / g.tpb] = 0;
        }
        if (t == 0) {
            g.toff[nb] = T;
            *g.tn = nb;
        }
    }
}
__global__ void k_row_groups(RowGroups g, int T) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < T) row_groups(g, t, T);
}

// attn_norm and the Q8_K quantisation of its output in one launch, one
// 256-thread block per row of n (a multiple of 256): the sum of squares and
// scale exactly as k_rms_norm, each value (x * scale) * w as it writes them, and
// each 256-value block quantized by one wave as k_quant_q8K does.
__global__ void __launch_bounds__(256) k_rms_norm_q8K(const float* __restrict__ x, int64_t n, float eps,
                                                      const float* __restrict__ w, BlockQ8_K* __restrict__ dst,
                                                      _Float16* __restrict__ hout, BlockQ8_0* __restrict__ dst0,
                                                      RowGroups g) {
    __shared__ double part[4];
    if (threadIdx.x == 0) row_groups(g, blockIdx.x, gridDim.x);
    const float* xr = x + (int64_t) blockIdx.x * n;
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += 256) {
        const float v = xr[i];
        s += (double) (v * v);
    }
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    const double tot = (part[0] + part[1]) + (part[2] + part[3]);
    const float mean = (float) (tot / (double) n);
    const float scale = 1.0f / sqrtf(mean + eps);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t nb = n / QK_K;
    for (int64_t ib = wv; ib < nb; ib += 4) {
        const float4 q = *(const float4*) (xr + ib * QK_K + 4 * lane);
        const float4 ww = *(const float4*) (w + ib * QK_K + 4 * lane);
        const float v[4] = {(q.x * scale) * ww.x, (q.y * scale) * ww.y, (q.z * scale) * ww.z, (q.w * scale) * ww.w};
        const int64_t blk = (int64_t) blockIdx.x * nb + ib;
        quant_q8K_wave(v, lane, dst + blk, hout ? hout + (size_t) blk * QK_K : nullptr,
                       hout ? hout + (size_t) (nb * gridDim.x) * QK_K + (size_t) blk * 16 : nullptr);
        if (dst0)
            quant_q80_lane8(float4{v[0], v[1], v[2], v[3]}, true, 8 * blk + (lane >> 3), lane & 7, dst0, nullptr, nullptr);
    }
}

__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v) {
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = v;
}

}  // namespace

int launch_attn_core(const AttnArgs& a, hipStream_t st) {
    if (a.T <= 0) return 0;
    const int nq = a.n_head, nk = a.n_head_kv;
    const int64_t rows = (int64_t) a.T * (nq / nk), n = (int64_t) a.T * nq * AD;
    const int n_split = a.split > 0 ? (int) ((a.n_kv + a.split - 1) / a.split) : 0;
    const int n_pv = a.merge > 0 ? (n_split + a.merge - 1) / a.merge : 0;
    if (n_split <= 0 || n_split > 65535 || n_pv <= 0 || a.split % FK || !a.stat || !a.part || (a.att_q8K && n % QK_K) ||
        (!a.att_q8K && !a.att) || a.split * a.merge * (int64_t) nk * AD * 2 >= (int64_t(1) << 31))
        return -2;
    // head rows per block: five per wave for many tokens, one for few (T = 1: 4.8 us)
    const int hpb = a.T >= 128 ? 20 : 4;
    const dim3 gr((unsigned) a.T, (unsigned) ((nq + 2 * nk + hpb - 1) / hpb));
    if (hpb == 4) hipLaunchKernelGGL(k_attn_qk_rope<1>, gr, dim3(256), 0, st, a, hpb);
    else hipLaunchKernelGGL(k_attn_qk_rope<5>, gr, dim3(256), 0, st, a, hpb);
    const int nw = attn_waves(rows);
    const unsigned rb = (unsigned) ((rows + 32 * nw - 1) / (32 * nw));
    const dim3 gs((unsigned) nk, rb, (unsigned) n_split), gp((unsigned) nk, rb, (unsigned) n_pv);
    if (nw == 1) {
        hipLaunchKernelGGL(k_attn_stat<1>, gs, dim3(64), 0, st, a);
        hipLaunchKernelGGL(k_attn_pv<1>, gp, dim3(64), 0, st, a, n_split, a.merge);
    } else if (nw == 2) {
        hipLaunchKernelGGL(k_attn_stat<2>, gs, dim3(128), 0, st, a);
        hipLaunchKernelGGL(k_attn_pv<2>, gp, dim3(128), 0, st, a, n_split, a.merge);
    } else {
        hipLaunchKernelGGL(k_attn_stat<4>, gs, dim3(256), 0, st, a);
        hipLaunchKernelGGL(k_attn_pv<4>, gp, dim3(256), 0, st, a, n_split, a.merge);
    }
    const unsigned nblk = (unsigned) ((n + QK_K - 1) / QK_K);
    if (n_pv <= 4) hipLaunchKernelGGL(k_attn_combine<1>, dim3((nblk + 3) / 4), dim3(256), 0, st, a, n_pv);
    else hipLaunchKernelGGL(k_attn_combine<4>, dim3(nblk), dim3(256), 0, st, a, n_pv);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

int launch_rms_norm_q8K(const float* x, int64_t n, int64_t rows, float eps, const float* w, void* dst,
                        hipStream_t st, uint16_t* h_out, void* dst0, const RowGroups* g) {
    if (n % QK_K || !w || (((uintptr_t) x | (uintptr_t) w) & 15)) return -2;
    if (rows == 0) return 0;
    hipLaunchKernelGGL(k_rms_norm_q8K, dim3((unsigned) rows), dim3(256), 0, st, x, n, eps, w, (BlockQ8_K*) dst,
                       (_Float16*) h_out, (BlockQ8_0*) dst0, g ? *g : RowGroups{});
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

int launch_row_groups(const RowGroups& g, int64_t T, hipStream_t st) {
    if (T <= 0 || T >= (int64_t(1) << 30)) return -2;
    hipLaunchKernelGGL(k_row_groups, dim3((unsigned) ((T + 255) / 256)), dim3(256), 0, st, g, (int) T);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

int launch_add_rms_norm_mul(const float* x, const float* y, float* resid, float* out, int64_t n, int64_t rows,
                            float eps, const float* w, hipStream_t st) {
    if (rows == 0) return 0;
    hipLaunchKernelGGL(k_add_rms_norm_mul, dim3((unsigned) rows), dim3(256), 0, st, x, y, resid, out, n, eps, w);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

int launch_fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t st) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_fill_i32, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, st, p, n, v);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace qw
