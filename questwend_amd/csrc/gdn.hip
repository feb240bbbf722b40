// gdn.hip -- the recurrent half of Seg A for the gated-delta-net layers of
// qwen3next / qwen35moe (core/runtime.cpp:1976-1995 with build_gdn, 737-859):
// the causal depthwise conv over [conv_state | qkv] with its state update,
// SiLU, the per-head L2 norms of q and k, beta = sigmoid, g = softplus(alpha +
// dt_bias) * ssm_a, ggml_gated_delta_net's recurrence over the tokens with the
// state update, and the gated RMSNorm.  The five projections (attn_qkv,
// attn_gate, ssm_beta, ssm_alpha, ssm_out) run on the quantized mul_mat kernels
// as one-expert mul_mat_ids (api.cpp).
//
// Layout in HBM: qkv, conv [T][conv_ch] f32 (conv_ch = H_v S + 2 H_k S: q heads,
// then k heads, then v heads); conv_state [conv_ch][d_conv - 1] and the state
// [H_v][S][S] f32 in ggml's layouts (state[h][j][i] = S_h[i][j], ops.cpp:
// 10840-10842); qn, kn [T][H_k][S]; bg [T][H_v][2] (beta, g); o [T][H_v][S];
// y [T][H_v S].
//
// The float steps follow ggml's CPU ops: ggml_compute_forward_ssm_conv_f32
// (ops.cpp:9557-9610: a float sum over the d_conv taps in order), silu as
// ggml_v_silu, l2_norm with a double sum of squares (ops.cpp:4174-4219),
// sigmoid and softplus (threshold 20) as unary-ops.cpp:31-33 and 80-82, the
// recurrence as ggml_compute_forward_gated_delta_net_one_chunk (ops.cpp:
// 10734-10887; scalar gate), rms_norm with a double sum.  The recurrence's dots
// are summed in another order than ggml's vec_dot_f32, so results agree with
// the CPU backend to float rounding (the 1e-3 bar), not bit for bit.
#include "qw_kernels.hpp"

namespace qw {

namespace {

constexpr int GS = 128;        // state size S (ssm.state_size of the Qwen3-Next family)
constexpr int GJB = 32;        // state rows j per workgroup of the token-by-token recurrence (8 lanes per row)

// Four channels and CT tokens per thread: the DC-tap windows over [conv_state |
// qkv rows] ending at each token (x_0 .. x_{DC-2} are the state, x_{DC-1+t} =
// qkv[t]), then SiLU.  A row of x is loaded once for the DC tokens it reaches.
// T = 300, 8192 channels: 14.7 (a thread per output) -> 10.5 us.
constexpr int CT = 4;
template <int DC>
__global__ void __launch_bounds__(256) k_gdn_conv(GdnArgs a) {
    const int64_t c = ((int64_t) blockIdx.x * 64 + (threadIdx.x & 63)) * 4;
    const int t0 = ((int) blockIdx.y * 4 + (int) (threadIdx.x >> 6)) * CT;
    if (c >= a.conv_ch || t0 >= a.T) return;
    float4 x[CT + DC - 1];
#pragma unroll
    for (int i = 0; i < CT + DC - 1; ++i) {
        const int xi = t0 + i;
        if (xi < DC - 1) {
            const float* s = a.conv_state + c * (DC - 1) + xi;
            x[i] = float4{s[0], s[DC - 1], s[2 * (DC - 1)], s[3 * (DC - 1)]};
        } else {
            x[i] = *(const float4*) (a.qkv + (int64_t) min(xi - (DC - 1), a.T - 1) * a.conv_ch + c);
        }
    }
    float w[4][DC];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < DC; ++j) w[q][j] = a.conv1d[(c + q) * DC + j];
#pragma unroll
    for (int k = 0; k < CT; ++k) {
        if (t0 + k >= a.T) break;
        float4 s = float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < DC; ++j) {
            s.x = __builtin_fmaf(x[k + j].x, w[0][j], s.x);
            s.y = __builtin_fmaf(x[k + j].y, w[1][j], s.y);
            s.z = __builtin_fmaf(x[k + j].z, w[2][j], s.z);
            s.w = __builtin_fmaf(x[k + j].w, w[3][j], s.w);
        }
        *(float4*) (a.conv + (int64_t) (t0 + k) * a.conv_ch + c) = float4{v_silu(s.x), v_silu(s.y), v_silu(s.z), v_silu(s.w)};
    }
}

// The conv state after the call: x_T .. x_{T+d_conv-2}, one thread per channel
// (in the launch after k_gdn_conv, which reads the old state).
__device__ __forceinline__ void gdn_conv_state(const GdnArgs& a, int64_t c) {
    if (c >= a.conv_ch) return;
    const int dc = a.d_conv, T = a.T;
    float nw[GDN_MAX_CONV];
#pragma unroll
    for (int j = 0; j + 1 < GDN_MAX_CONV; ++j)
        if (j < dc - 1) {
            const int xi = T + j;
            nw[j] = xi < dc - 1 ? a.conv_state[c * (dc - 1) + xi] : a.qkv[(int64_t) (xi - (dc - 1)) * a.conv_ch + c];
        }
#pragma unroll
    for (int j = 0; j + 1 < GDN_MAX_CONV; ++j)
        if (j < dc - 1) a.conv_state[c * (dc - 1) + j] = nw[j];
}

// Block t (H_k + 1) + hk: q and k of token t's key head hk divided by max(||.||,
// eps) (the sum of squares in double, as ggml_l2_norm); with hk = H_k instead beta
// and g of every value head; the blocks past the tokens' the conv state.
__global__ void __launch_bounds__(GS) k_gdn_prep(GdnArgs a) {
    const int per = a.H_k + 1, t = blockIdx.x / per, hk = blockIdx.x % per, i = threadIdx.x;
    if (t >= a.T) {
        gdn_conv_state(a, (int64_t) ((int) blockIdx.x - a.T * per) * GS + i);
        return;
    }
    __shared__ double s_red[2][GS / 64];
    if (hk == a.H_k) {
        for (int hv = i; hv < a.H_v; hv += GS) {
            const float b = a.braw[(int64_t) t * a.H_v + hv];
            const float al = a.araw[(int64_t) t * a.H_v + hv] + a.dt_bias[hv];
            const float sp = al > 20.0f ? al : logf(1.0f + expf(al));
            a.bg[((int64_t) t * a.H_v + hv) * 2] = 1.0f / (1.0f + expf(-b));
            a.bg[((int64_t) t * a.H_v + hv) * 2 + 1] = sp * a.ssm_a[hv];
        }
        return;
    }
    const int64_t key_dim = (int64_t) a.H_k * GS;
    const float q = a.conv[(int64_t) t * a.conv_ch + hk * GS + i];
    const float k = a.conv[(int64_t) t * a.conv_ch + key_dim + hk * GS + i];
    double sq = (double) (q * q), sk = (double) (k * k);
    for (int off = 32; off >= 1; off >>= 1) {
        sq += __shfl_xor(sq, off);
        sk += __shfl_xor(sk, off);
    }
    if ((i & 63) == 0) {
        s_red[0][i >> 6] = sq;
        s_red[1][i >> 6] = sk;
    }
    __syncthreads();
    double tq = 0.0, tk = 0.0;
#pragma unroll
    for (int w = 0; w < GS / 64; ++w) {
        tq += s_red[0][w];
        tk += s_red[1][w];
    }
    const float scq = 1.0f / fmaxf(sqrtf((float) tq), a.eps), sck = 1.0f / fmaxf(sqrtf((float) tk), a.eps);
    a.qn[((int64_t) t * a.H_k + hk) * GS + i] = q * scq;
    a.kn[((int64_t) t * a.H_k + hk) * GS + i] = k * sck;
}

// The recurrence token by token, for batches of fewer than GCHUNK_MIN tokens.
// Workgroup (value head hv, rows j0 .. j0 + GJB - 1 of its state M = S^T): 8 lanes per
// row, each holding 16 of its 128 columns in registers for all tokens.  Per token, as
// ggml: M *= exp(g); delta_j = (v_j - M_j . k) beta; M_j += delta_j k; o_j = (M_j . q) /
// sqrt(S).  A row's dots are reduced over its 8 lanes by DPP (quad xor 1, xor 2, half-row
// mirror).  Nothing of a token's steps depends on where it stands in the call, so a call
// gives the bits that calls of its parts give (decode steps and a verify batch agree).
// q, k (the key head), v (the workgroup's rows), beta and exp(g) sit in LDS.
//
// Bound: the chain of the two row reductions per token, with a wave per SIMD.  Four tokens
// per step, whose reductions are independent, gain little at this length and round each
// token by its place in the call (us per call, H_v = 32, token by token / four per step:
// 49.8 / 51.0 at T = 1, 71.0 / 71.4 at 4, 81.2 / 81.3 at 16, 86.3 / 85.3 at 31).
typedef float fx4 __attribute__((ext_vector_type(4)));   // (arrays of it stay in registers)
constexpr int GTB = 32;   // tokens staged
__global__ void __launch_bounds__(256) k_gdn_delta(GdnArgs a) {
    const int hv = blockIdx.x, tid = threadIdx.x, r = tid >> 3, l = tid & 7;
    const int j0 = blockIdx.y * GJB, j = j0 + r, hk = hv % a.H_k;
    __shared__ __align__(16) float s_q[GTB][GS];
    __shared__ __align__(16) float s_k[GTB][GS];
    __shared__ float s_v[GTB][GJB];
    __shared__ float s_b[GTB], s_e[GTB];
    static_assert(GJB * 8 == 256 && GTB * GS / 4 == 4 * 256 && GTB * GJB == 4 * 256, "the loads' split over 256 threads");
    float* st = a.state + ((int64_t) hv * GS + j) * GS + 16 * l;
    fx4 m[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = *(const fx4*) (st + 4 * i);
    const float scale = 1.0f / sqrtf((float) GS);
    const int64_t vbase = 2 * (int64_t) a.H_k * GS + (int64_t) hv * GS + j0;
    const int qcol = 4 * (tid % (GS / 4));
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int tq = tid / (GS / 4) + 8 * u, tv = tid / GJB + 8 * u;
        const int64_t row = ((int64_t) min(tq, a.T - 1) * a.H_k + hk) * GS + qcol;
        *(fx4*) &s_q[tq][qcol] = *(const fx4*) (a.qn + row);
        *(fx4*) &s_k[tq][qcol] = *(const fx4*) (a.kn + row);
        s_v[tv][tid % GJB] = a.conv[(int64_t) min(tv, a.T - 1) * a.conv_ch + vbase + tid % GJB];
    }
    if (tid < 2 * GTB) {
        const float bg = a.bg[((int64_t) min(tid >> 1, a.T - 1) * a.H_v + hv) * 2 + (tid & 1)];
        if (tid & 1) s_e[tid >> 1] = expf(bg);
        else s_b[tid >> 1] = bg;
    }
    auto red8 = [](float x) __attribute__((always_inline)) {
        x = x + dpp_f<DPP_XOR1>(x);
        x = x + dpp_f<DPP_XOR2>(x);
        return x + dpp_f<DPP_HALF_MIRROR>(x);
    };
    __syncthreads();
#pragma unroll 1
    for (int t = 0; t < a.T; ++t) {
        const float e = s_e[t];
        fx4 q[4], k[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            q[i] = *(const fx4*) &s_q[t][16 * l + 4 * i];
            k[i] = *(const fx4*) &s_k[t][16 * l + 4 * i];
        }
        float d0 = 0.0f, d1 = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            m[i] *= e;
            d0 = __builtin_fmaf(m[i].x, k[i].x, d0);
            d1 = __builtin_fmaf(m[i].y, k[i].y, d1);
            d0 = __builtin_fmaf(m[i].z, k[i].z, d0);
            d1 = __builtin_fmaf(m[i].w, k[i].w, d1);
        }
        const float delta = (s_v[t][r] - red8(d0 + d1)) * s_b[t];
        float o0 = 0.0f, o1 = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int c = 0; c < 4; ++c) m[i][c] = __builtin_fmaf(k[i][c], delta, m[i][c]);
            o0 = __builtin_fmaf(m[i].x, q[i].x, o0);
            o1 = __builtin_fmaf(m[i].y, q[i].y, o1);
            o0 = __builtin_fmaf(m[i].z, q[i].z, o0);
            o1 = __builtin_fmaf(m[i].w, q[i].w, o1);
        }
        const float o = red8(o0 + o1);
        if (l == 0) a.o[((int64_t) t * a.H_v + hv) * GS + j] = o * scale;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) *(fx4*) (st + 4 * i) = m[i];
}

// ---- batches of GCHUNK_MIN tokens and more: sixteen tokens per step, on the matrix cores ----
//
// With D the deltas of a chunk's 16 tokens (a row per token), V, K, Q its rows, M the
// state before it, E_b = e_1 .. e_b and E_{a,b} = e_{a+1} .. e_b, the recurrence reads
//     (I + A) D = R = beta (V - E K M^T),     A[b][a] = beta_b E_{a,b} (k_a . k_b), a < b
//     O sqrt(S) = E Q M^T + P D,              P[b][a] = E_{a,b} (k_a . q_b),        a <= b
//     M^T after = E_16 M^T + K^T (E_{a,16} D)
// A and P hold nothing of the state: k_gdn_chunk forms P and T = (I + A)^-1 (16 x 16,
// forward substitution) for every chunk and head at once, and the serial kernel is left
// with five small fp32 matrix products per chunk.
// The same sums in another order, all in fp32: a call of 32 tokens and more equals calls
// of its parts to fp32 rounding.  From 32 tokens on (us per call, token by token / chunks,
// H_v = 32): 81.4 / 83.1 at T = 16, 84.9 / 85.4 at 24, 87.2 / 86.2 at 31; H_v = 16: 74.2 /
// 75.2, 76.8 / 76.7, 78.9 / 77.1.
constexpr int GCHUNK_MIN = 32;
constexpr int GCK = 16;              // tokens per chunk
constexpr int GCK_P = 256, GCK_E = 512, GCK_E2 = 528, GCK_B = 544;   // record: T, P / sqrt(S), E_b, E_{a,16}, beta
constexpr int GCK_REC = 576;         // floats per record (chunk, value head), in the y rows, written only later
static_assert(GCHUNK_MIN - 1 <= GTB, "the token-by-token form stages one block of tokens");
static_assert(GCHUNK_MIN >= GCK && 2 * GCK_REC <= (GCK + 1) * GS, "the records of ceil(T / 16) chunks fit T rows of y");

__device__ __forceinline__ fx4 mfma_f32(float x, float y, fx4 c) {   // D[16][16] += A[16][4] B[4][16]
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0);
}

// Block c H_k + hk: k_gdn_prep's norms for chunk c of key head hk, and the records of the
// value heads that read it; the blocks past the chunks' the conv state.
__global__ void __launch_bounds__(256) k_gdn_chunk(GdnArgs a) {
    const int n_ch = (a.T + GCK - 1) / GCK, c = blockIdx.x / a.H_k, hk = blockIdx.x % a.H_k, tid = threadIdx.x;
    if (c >= n_ch) {
        gdn_conv_state(a, (int64_t) ((int) blockIdx.x - n_ch * a.H_k) * 256 + tid);
        return;
    }
    constexpr int HS = 16;   // value heads at a time
    __shared__ __align__(16) float s_q[GCK][GS + 4], s_k[GCK][GS + 4];
    __shared__ float s_p[2][4][256];
    __shared__ __align__(16) float s_e[HS][GCK], s_b[HS][GCK];
    __shared__ __align__(16) float s_A[HS][GCK * GCK + 4];
    const int t0 = c * GCK, w = tid >> 6, lane = tid & 63;
    const int64_t key_dim = (int64_t) a.H_k * GS;
    {   // 32 lanes per token, two rounds
        const int col = 4 * (lane & 31);
        fx4 q[2], k[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const float* row = a.conv + (int64_t) min(t0 + 4 * w + 2 * u + (lane >> 5), a.T - 1) * a.conv_ch + hk * GS + col;
            q[u] = *(const fx4*) row;
            k[u] = *(const fx4*) (row + key_dim);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int b = 4 * w + 2 * u + (lane >> 5);
            double sq = 0.0, sk = 0.0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sq += (double) (q[u][i] * q[u][i]);
                sk += (double) (k[u][i] * k[u][i]);
            }
            for (int off = 16; off >= 1; off >>= 1) {
                sq += __shfl_xor(sq, off);
                sk += __shfl_xor(sk, off);
            }
            const float scq = 1.0f / fmaxf(sqrtf((float) sq), a.eps), sck = 1.0f / fmaxf(sqrtf((float) sk), a.eps);
            const fx4 qn = q[u] * scq, kn = k[u] * sck;
            *(fx4*) &s_q[b][col] = qn;
            *(fx4*) &s_k[b][col] = kn;
            if (t0 + b < a.T) {
                *(fx4*) (a.qn + ((int64_t) (t0 + b) * a.H_k + hk) * GS + col) = qn;
                *(fx4*) (a.kn + ((int64_t) (t0 + b) * a.H_k + hk) * GS + col) = kn;
            }
        }
    }
    __syncthreads();
    {   // k_b . k_a and q_b . k_a over the wave's 32 columns; the contraction takes them in any order
        const int n = lane & 15, g = lane >> 4;
        fx4 gk = fx4{0.0f, 0.0f, 0.0f, 0.0f}, gq = gk;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const fx4 kf = *(const fx4*) &s_k[n][32 * w + 16 * u + 4 * g], qf = *(const fx4*) &s_q[n][32 * w + 16 * u + 4 * g];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                gk = mfma_f32(kf[r], kf[r], gk);
                gq = mfma_f32(qf[r], kf[r], gq);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s_p[0][w][(4 * g + r) * GCK + n] = gk[r];
            s_p[1][w][(4 * g + r) * GCK + n] = gq[r];
        }
    }
    __syncthreads();
    const int hi = tid >> 4, lo = tid & 15;
    const float gk = (s_p[0][0][tid] + s_p[0][1][tid]) + (s_p[0][2][tid] + s_p[0][3][tid]);
    const float gq = (s_p[1][0][tid] + s_p[1][1][tid]) + (s_p[1][2][tid] + s_p[1][3][tid]);
    const float scale = 1.0f / sqrtf((float) GS);
    const int rep = a.H_v / a.H_k;
    for (int m0 = 0; m0 < rep; m0 += HS) {
        const int nm = rep - m0 < HS ? rep - m0 : HS;
        if (hi < nm) {   // head m0 + hi, token lo
            const int hv = hk + (m0 + hi) * a.H_k, t = t0 + lo;
            float e = 1.0f, be = 0.0f;
            if (t < a.T) {
                const float al = a.araw[(int64_t) t * a.H_v + hv] + a.dt_bias[hv];
                const float sp = al > 20.0f ? al : logf(1.0f + expf(al));
                e = expf(sp * a.ssm_a[hv]);
                be = 1.0f / (1.0f + expf(-a.braw[(int64_t) t * a.H_v + hv]));
            }
            s_e[hi][lo] = e;
            s_b[hi][lo] = be;
        }
        __syncthreads();
        for (int m = 0; m < nm; ++m) {   // token hi against token lo
            float* rec = a.y + ((int64_t) c * a.H_v + hk + (m0 + m) * a.H_k) * GCK_REC;
            float ev[GCK], E = 1.0f;
#pragma unroll
            for (int y = 0; y < GCK; y += 4) *(fx4*) &ev[y] = *(const fx4*) &s_e[m][y];
#pragma unroll
            for (int y = 1; y < GCK; ++y) E = y > lo && y <= hi ? E * ev[y] : E;
            const float be = s_b[m][hi];
            s_A[m][tid] = lo < hi && t0 + hi < a.T ? (be * E) * gk : 0.0f;
            rec[GCK_P + tid] = lo <= hi ? (E * gq) * scale : 0.0f;
            if (lo == 0) {
                rec[GCK_E + hi] = ev[0] * E;
                rec[GCK_B + hi] = be;
            }
            if (hi == GCK - 1) rec[GCK_E2 + lo] = E;
        }
        __syncthreads();
        if (hi < nm) {   // head m0 + hi, column lo of T
            float* rec = a.y + ((int64_t) c * a.H_v + hk + (m0 + hi) * a.H_k) * GCK_REC;
            float tc[GCK];
#pragma unroll
            for (int b = 0; b < GCK; ++b) {
                float s = b == lo ? 1.0f : 0.0f;
#pragma unroll
                for (int y = 0; y < b; ++y) s = __builtin_fmaf(-s_A[hi][b * GCK + y], tc[y], s);
                tc[b] = lo > b ? 0.0f : s;
                rec[b * GCK + lo] = tc[b];
            }
        }
        __syncthreads();
    }
}

// C[b][j] += sum_{a <= b} L[b][a] x[a][j] for values that are not all finite: the product over
// whole rows would carry a token's infinity or NaN to the tokens before it as 0 * inf.
__device__ __forceinline__ fx4 gdn_tri(const float* __restrict__ L, fx4 x, fx4 acc) {
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
#pragma unroll 1
    for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const float xa = __shfl(x[y], h * 16 + n);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * h + y <= 4 * g + r) acc[r] = __builtin_fmaf(L[(4 * g + r) * GCK + 4 * h + y], xa, acc[r]);
        }
    return acc;
}

// Workgroup (value head hv, rows j0 .. j0 + 15 of M), wave w its columns 32 w .. + 31 as two
// accumulator tiles of M^T: lane (g, n) = (lane / 16, lane % 16) holds M[j0 + n][i0 + 4 g + r]
// in register r.  Register r is at once the operand B of a product that contracts the
// columns 4 g + r of step r, so the state never changes its layout; nor do X = K M^T, R
// and D, which come out as [token 4 g + r][row n] and are contracted over the tokens the
// same way.  K M^T and Q M^T are summed over the four waves through LDS (one barrier per
// chunk); R and D are formed by every wave, O by one of them in turn.  Operands are
// loaded two chunks ahead.  H_v = 32, T = 300, with k_gdn_chunk (7.4) in place of k_gdn_prep
// (6.0): 74 us four tokens a step, 39 loading one chunk ahead, 32 now: 1.3 us a chunk, the
// chain of products, exchange and elementwise steps with one wave per SIMD (26 us without
// any load).  Buffer loads with scalar bases, O split over all waves and loads placed
// between the products: 33 each.
__global__ void __launch_bounds__(256) k_gdn_delta_chunk(GdnArgs a) {
    const int hv = blockIdx.x, j0 = blockIdx.y * 16, hk = hv % a.H_k;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int n_ch = (a.T + GCK - 1) / GCK;
    __shared__ fx4 s_x[2][2][4][64];
    float* st = a.state + ((int64_t) hv * GS + j0 + n) * GS + 32 * w + 4 * g;
    fx4 m[2] = {*(const fx4*) st, *(const fx4*) (st + 16)};
    const float scale = 1.0f / sqrtf((float) GS);
    const int64_t vcol = 2 * (int64_t) a.H_k * GS + (int64_t) hv * GS + j0 + n;
    struct Chunk {
        fx4 kf[2], qf[2], kt[2], v, T, P, E, E2, b;
        float e;
    };
    auto load = [&](int c) __attribute__((always_inline)) {
        Chunk x;
        const int t0 = c * GCK, last = a.T - 1;
        const int64_t row = ((int64_t) min(t0 + n, last) * a.H_k + hk) * GS + 32 * w + 4 * g;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            x.kf[u] = *(const fx4*) (a.kn + row + 16 * u);
            x.qf[u] = *(const fx4*) (a.qn + row + 16 * u);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t t = min(t0 + 4 * g + r, last);
            x.v[r] = a.conv[t * a.conv_ch + vcol];
#pragma unroll
            for (int u = 0; u < 2; ++u) x.kt[u][r] = a.kn[(t * a.H_k + hk) * GS + 32 * w + 16 * u + n];
        }
        const float* rec = a.y + ((int64_t) c * a.H_v + hv) * GCK_REC;
        x.T = *(const fx4*) (rec + n * GCK + 4 * g);
        x.P = *(const fx4*) (rec + GCK_P + n * GCK + 4 * g);
        x.E = *(const fx4*) (rec + GCK_E + 4 * g);
        x.E2 = *(const fx4*) (rec + GCK_E2 + 4 * g);
        x.b = *(const fx4*) (rec + GCK_B + 4 * g);
        x.e = rec[GCK_E + GCK - 1];
        return x;
    };
    auto finite = [](fx4 x) __attribute__((always_inline)) {
        bool f = true;
#pragma unroll
        for (int r = 0; r < 4; ++r) f = f && __builtin_fabsf(x[r]) < INFINITY;
        return (bool) __all(f);
    };
    const fx4 zero = fx4{0.0f, 0.0f, 0.0f, 0.0f};
    auto step = [&](int c, const Chunk& x) __attribute__((always_inline)) {
        const float* rec = a.y + ((int64_t) c * a.H_v + hv) * GCK_REC;
        fx4 X[2] = {zero, zero}, Y[2] = {zero, zero};
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                X[u] = mfma_f32(x.kf[u][r], m[u][r], X[u]);
                Y[u] = mfma_f32(x.qf[u][r], m[u][r], Y[u]);
            }
        s_x[c & 1][0][w][lane] = X[0] + X[1];
        s_x[c & 1][1][w][lane] = Y[0] + Y[1];
        __syncthreads();   // (a wave that writes these words again has passed the next barrier)
        const fx4(*sx)[64] = s_x[c & 1][0];
        const fx4 Xs = (sx[0][lane] + sx[1][lane]) + (sx[2][lane] + sx[3][lane]);
        fx4 R, D = zero;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            R[r] = c * GCK + 4 * g + r < a.T ? (x.v[r] - x.E[r] * Xs[r]) * x.b[r] : 0.0f;
        if (finite(R)) {
#pragma unroll
            for (int r = 0; r < 4; ++r) D = mfma_f32(x.T[r], R[r], D);
        } else {
            D = gdn_tri(rec, R, D);
        }
        const fx4 De = D * x.E2;
#pragma unroll
        for (int u = 0; u < 2; ++u) m[u] *= x.e;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int u = 0; u < 2; ++u) m[u] = mfma_f32(x.kt[u][r], De[r], m[u]);
        if ((c & 3) == w) {
            const fx4(*sy)[64] = s_x[c & 1][1];
            fx4 O = ((sy[0][lane] + sy[1][lane]) + (sy[2][lane] + sy[3][lane])) * x.E * scale;
            if (finite(D)) {
#pragma unroll
                for (int r = 0; r < 4; ++r) O = mfma_f32(x.P[r], D[r], O);
            } else {
                O = gdn_tri(rec + GCK_P, D, O);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = c * GCK + 4 * g + r;
                if (t < a.T) a.o[((int64_t) t * a.H_v + hv) * GS + j0 + n] = O[r];
            }
        }
    };
    Chunk x0 = load(0), x1 = load(min(1, n_ch - 1)), x2;
#pragma unroll 1
    for (int c = 0; c < n_ch; c += 3) {
        x2 = load(min(c + 2, n_ch - 1));
        step(c, x0);
        if (c + 1 >= n_ch) break;
        x0 = load(min(c + 3, n_ch - 1));
        step(c + 1, x1);
        if (c + 2 >= n_ch) break;
        x1 = load(min(c + 4, n_ch - 1));
        step(c + 2, x2);
    }
    *(fx4*) st = m[0];
    *(fx4*) (st + 16) = m[1];
}

// Block (t, value head): rms_norm of the head's 128 outputs (double sum) times
// ssm_norm, times silu(z) of the same elements: ggml_mul(ggml_mul(rms_norm(o),
// ssm_norm), ggml_silu(z)), each product rounded as there.
__global__ void __launch_bounds__(GS) k_gdn_gate_norm(GdnArgs a) {
    const int t = blockIdx.x, hv = blockIdx.y, i = threadIdx.x;
    __shared__ double s_red[GS / 64];
    const int64_t e = ((int64_t) t * a.H_v + hv) * GS + i;
    const float x = a.o[e];
    double s = (double) (x * x);
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
    if ((i & 63) == 0) s_red[i >> 6] = s;
    __syncthreads();
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < GS / 64; ++w) tot += s_red[w];
    const float mean = (float) (tot / (double) GS);
    const float sc = 1.0f / sqrtf(mean + a.eps);
    const float zn = (x * sc) * a.ssm_norm[i];
    a.y[e] = zn * v_silu(a.z[e]);
}

// The same, two heads (256 values) per wave and straight into Q8_K (and its f16
// copy): the output projection's input.
__global__ void __launch_bounds__(256) k_gdn_gate_norm_q8K(GdnArgs a) {
    const int lane = threadIdx.x & 63;
    const int64_t nblk = (int64_t) a.T * a.H_v / 2, blk = (int64_t) blockIdx.x * 4 + (threadIdx.x >> 6);
    if (blk >= nblk) return;
    const int64_t e = blk * 256 + 4 * lane;
    const float4 x = *(const float4*) (a.o + e), z = *(const float4*) (a.z + e);
    const float* nw = a.ssm_norm + 4 * (lane & 31);   // (the caller's: any alignment)
    double s = ((double) (x.x * x.x) + (double) (x.y * x.y)) + ((double) (x.z * x.z) + (double) (x.w * x.w));
    for (int off = 16; off >= 1; off >>= 1) s += __shfl_xor(s, off);   // the head's 32 lanes
    const float mean = (float) (s / (double) GS);
    const float sc = 1.0f / sqrtf(mean + a.eps);
    const float v[4] = {((x.x * sc) * nw[0]) * v_silu(z.x), ((x.y * sc) * nw[1]) * v_silu(z.y),
                        ((x.z * sc) * nw[2]) * v_silu(z.z), ((x.w * sc) * nw[3]) * v_silu(z.w)};
    _Float16* h = (_Float16*) a.y_h;
    quant_q8K_wave(v, lane, (BlockQ8_K*) a.y_q8K + blk, h ? h + (size_t) blk * QK_K : nullptr,
                   h ? h + (size_t) nblk * QK_K + (size_t) blk * 16 : nullptr);
}

}  // namespace

bool gdn_shape_ok(int64_t S, int64_t H_k, int64_t H_v, int64_t d_conv) {
    return S == GS && H_k > 0 && H_v > 0 && H_v % H_k == 0 && H_v <= 4096 && d_conv >= 2 && d_conv <= GDN_MAX_CONV;
}

int launch_gdn_core(const GdnArgs& a, hipStream_t stream) {
    if (!gdn_shape_ok(GS, a.H_k, a.H_v, a.d_conv) || a.T <= 0 || (a.y_q8K && a.H_v % 2)) return -2;
    const int64_t prep = (int64_t) a.T * (a.H_k + 1) + (a.conv_ch + GS - 1) / GS;
    if (prep > INT32_MAX) return -2;
    const dim3 gc((unsigned) ((a.conv_ch + 255) / 256), (unsigned) ((a.T + 4 * CT - 1) / (4 * CT)));
    switch (a.d_conv) {
        case 2: hipLaunchKernelGGL(k_gdn_conv<2>, gc, dim3(256), 0, stream, a); break;
        case 3: hipLaunchKernelGGL(k_gdn_conv<3>, gc, dim3(256), 0, stream, a); break;
        case 4: hipLaunchKernelGGL(k_gdn_conv<4>, gc, dim3(256), 0, stream, a); break;
        case 5: hipLaunchKernelGGL(k_gdn_conv<5>, gc, dim3(256), 0, stream, a); break;
        case 6: hipLaunchKernelGGL(k_gdn_conv<6>, gc, dim3(256), 0, stream, a); break;
        case 7: hipLaunchKernelGGL(k_gdn_conv<7>, gc, dim3(256), 0, stream, a); break;
        default: hipLaunchKernelGGL(k_gdn_conv<8>, gc, dim3(256), 0, stream, a); break;
    }
    if (a.T >= GCHUNK_MIN) {
        const int64_t chunks = (int64_t) ((a.T + GCK - 1) / GCK) * a.H_k + (a.conv_ch + 255) / 256;
        hipLaunchKernelGGL(k_gdn_chunk, dim3((unsigned) chunks), dim3(256), 0, stream, a);
        hipLaunchKernelGGL(k_gdn_delta_chunk, dim3((unsigned) a.H_v, (unsigned) (GS / 16)), dim3(256), 0, stream, a);
    } else {
        hipLaunchKernelGGL(k_gdn_prep, dim3((unsigned) prep), dim3(GS), 0, stream, a);
        hipLaunchKernelGGL(k_gdn_delta, dim3((unsigned) a.H_v, (unsigned) (GS / GJB)), dim3(256), 0, stream, a);
    }
    if (a.y_q8K)
        hipLaunchKernelGGL(k_gdn_gate_norm_q8K, dim3((unsigned) (((int64_t) a.T * a.H_v / 2 + 3) / 4)), dim3(256), 0,
                           stream, a);
    else
        hipLaunchKernelGGL(k_gdn_gate_norm, dim3((unsigned) a.T, (unsigned) a.H_v), dim3(GS), 0, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace qw
