// mmid_q80.hip -- ggml_mul_mat_id of Q8_0 weights: the matrix-core form for bins
// with many routed rows, and the GEMV that copies whole rows straight into LDS.
//
// Reference: ggml_vec_dot_q8_0_q8_0, AVX2 branch (ggml/src/ggml-cpu/arch/x86/
// quants.c).  Per (weight row, activation row) and 32-value block i it keeps eight
// int32 lanes, lane L the sum over elements 4 L .. 4 L + 3, and eight float chains
// acc_L = fma(fp16(x.d) * fp16(y.d), (float) sumi_L, acc_L) over the blocks in
// order; the result is hsum_float_8(acc).  Both kernels form those integers and
// replay those float steps, so their outputs equal ggml's bit for bit.
#include "qw_mfma.hpp"
#include "qw_rowdot.hpp"

#include <type_traits>

namespace qw {

typedef _Float16 q80_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 q80_h4 __attribute__((ext_vector_type(4)));
typedef _Float16 q80_h8 __attribute__((ext_vector_type(8)));
typedef float q80_f16 __attribute__((ext_vector_type(16)));

// ---- matrix cores ------------------------------------------------------------
//
// v_mfma_f32_16x16x4_4b_f16 forms four independent 16 x 16 x 4 products: lane l of
// A holds row l % 16, k = 0 .. 3 of product l / 16; B the column l % 16 likewise; D
// register 4 p + r of lane l is row 4 (l / 16) + r, column l % 16 of product p.
// With product p = AVX lane p (first instruction) or 4 + p (second), D is exactly
// the reference's integer lane sums as f32 (int8 products: below 2^17), one
// instruction per four lanes, with neither an integer dot nor a conversion; what
// is left on the VALU is the reference's own 32 fma per 16 x 16 tile and block
// (a lane: four rows x eight chains) and four products of the block scales.
//
// A = activation rows (an f16 copy of the Q8_0 rows, written by the launch that
// quantizes them: launch_q80_to_f16's layout), B = weight rows (converted here: a
// byte q ^ 0x80 under exponent byte 0x64 is the f16 1152 + q).  A lane then has
// one weight row, whose block scale it converts once for all its activation rows;
// those rows' scales are one 16-byte LDS read.
//
// Workgroup: 64 weight rows (a wave per 16) x one item of up to 16 routed rows.
// Eight blocks (272 weight bytes, 17 x 16) per step are copied straight into LDS one
// step ahead (two buffers).  52.7 KB and 112 VGPRs: three workgroups per CU, whose
// products and fp32 steps cover each other's waits for copies.  Items of 32 rows (two
// tiles share each weight operand, but 70 KB and 177 VGPRs leave two per CU) were slower
// up to 32 rows per bin and no faster at 64; us per 30B layer, 32 / 16 rows per item: 97.5 /
// 86.6 at T = 8, 207 / 184 at 33, 244 / 217 at 128, 308 / 282 at 251 (Zipf-skewed), 426 / 424 at
// 512, 702 / 707 and 713 / 709 at 1024 (skewed, not); H = 1024, 64 experts: 99.1 / 88.5 at 400.
// Weight rows sit 272 bytes apart, activation rows in pairs 1040 bytes apart, the odd
// row's 16-byte chunk c at position c ^ 8: 16 rows read at one chunk hit distinct banks.
//
// Bound: VALU issue (about 46 instructions per tile and block against 64 cycles of
// matrix core), 77 % of the cycles of gate and up at T = 251 (down 68 %), with waves waiting
// 36 % (45 %) of theirs; 607 MB read past the L2s there, of 430 MB of weights.  The GEMV alone
// took 1.8 ms per launch at T = 251, the layer 2509 us.
constexpr uint32_t Q80_WS = 272;     // LDS bytes of a staged weight row (8 blocks)
constexpr uint32_t Q80_HS = 1040;    // LDS bytes of an activation copy instruction (rows 2 i, 2 i + 1, pad)
constexpr int Q80_NR = 16;           // activation rows per item
constexpr int Q80_WDMA = MF_M * 17 / 64;   // weight copy instructions per step

__device__ __forceinline__ q80_h4 q80_to_h4(uint32_t q) {
    const uint32_t u = q ^ 0x80808080u;
    const q80_h2 lo = __builtin_bit_cast(q80_h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - q80_h2{1152, 1152};
    const q80_h2 hi = __builtin_bit_cast(q80_h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - q80_h2{1152, 1152};
    return q80_h4{lo.x, lo.y, hi.x, hi.y};
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) k_mmid_mfma_q80(MfLaunch lp) {
    const uint32_t zm = blockIdx.x >= lp.groups ? 1u : 0u;   // uniform: which matrix
    const MmidArgs& m = lp.m[zm];
    const uint32_t bid = blockIdx.x - zm * lp.groups;
    __shared__ __align__(16) uint8_t s_w0[MF_M * Q80_WS];
    __shared__ __align__(16) uint8_t s_w1[MF_M * Q80_WS];
    __shared__ __align__(16) uint8_t s_h0[8 * Q80_HS];
    __shared__ __align__(16) uint8_t s_h1[8 * Q80_HS];
    __shared__ __align__(16) float s_d0[8 * Q80_NR];   // activation block scales [block][row]
    __shared__ __align__(16) float s_d1[8 * Q80_NR];
    __shared__ int32_t s_arow[Q80_NR];
    __shared__ int32_t s_et[Q80_NR][2];
    __shared__ int s_item[2];
    const int tiles = (int) (m.N / MF_M);
    const int tile = (int) (bid % (uint32_t) tiles);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    mf_item(m, (int) (bid / (uint32_t) tiles), Q80_NR, wave, lane, s_item);
    const int g = s_item[0];
    if (g < 0) return;   // past the last item
    const int p0 = m.active_off[g] + Q80_NR * s_item[1], p1 = min(m.active_off[g + 1], p0 + Q80_NR);
    const int bin = m.active[g];
    int64_t mat = bin;
    if (m.slot_of) mat = (bin < m.n_slot_of) ? m.slot_of[bin] : -1;
    if (mat < 0 || mat >= m.n_as) {
        if (threadIdx.x == 0 && m.status) atomicOr(m.status, 4);
        return;
    }
    const int64_t r0 = (int64_t) tile * MF_M;
    const int lr = lane & 15, gq = lane >> 4;
    const int steps = (int) (m.K / 256);
    const uint8_t* wtile = m.w + (size_t) mat * m.nb2 + (size_t) r0 * m.nb1;
    const i32x4 wrsrc = rsrc_words(wtile, (uint32_t) (MF_M * m.nb1));
    const i32x4 hrsrc = rsrc_words(m.act_h, 0x7fffffffu);
    const i32x4 drsrc = rsrc_words(m.act_hd, 0x7fffffffu);
    const int ntok = p1 - p0;   // 1 .. Q80_NR
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    if (tid < Q80_NR) {
        const int pp = p0 + (tid < ntok ? tid : 0);   // rows past ntok are staged from row 0, never written
        const int e = m.rows[2 * pp], t = m.rows[2 * pp + 1];
        s_et[tid][0] = e;
        s_et[tid][1] = t;
        s_arow[tid] = (int) ((int64_t) (e % m.b_ne1) + (int64_t) t * m.b_ne1);
    }
    lds_barrier();
    uint32_t woff[5], hoff[2];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        const int q = 64 * (wave + 4 * k) + lane;
        const int qc = q < MF_M * 17 ? q : 0;
        woff[k] = (uint32_t) (qc / 17) * (uint32_t) m.nb1 + 16u * (uint32_t) (qc % 17);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int up = lane >> 5, n = 2 * (wave + 4 * k) + up;
        hoff[k] = (uint32_t) s_arow[n] * (uint32_t) (2 * m.K) + 16u * (uint32_t) ((lane & 31) ^ (8 * up));
    }
    // block scales: instruction w (of two) brings blocks 4 w .. 4 w + 3 of the step, all rows
    const uint32_t doff = (uint32_t) s_arow[lr] * (uint32_t) (m.K / 8) + 4u * (uint32_t) (4 * wave + gq);
    auto issue = [&](uint8_t* sw, uint8_t* sh, float* sd, int i) __attribute__((always_inline)) {
        uint32_t lw = (uint32_t) (uintptr_t) sw, lh = (uint32_t) (uintptr_t) sh, ld = (uint32_t) (uintptr_t) sd;
        asm volatile("" : "+s"(lw), "+s"(lh), "+s"(ld));
#pragma unroll
        for (int k = 0; k < 5; ++k)
            if (wv + 4 * k < Q80_WDMA) dma_b128(wrsrc, lw + 1024u * (uint32_t) (wv + 4 * k), woff[k], 272u * (uint32_t) i);
#pragma unroll
        for (int k = 0; k < 2; ++k) dma_b128(hrsrc, lh + Q80_HS * (uint32_t) (wv + 4 * k), hoff[k], 512u * (uint32_t) i);
        if (wv < 2) dma_b32(drsrc, ld + 256u * (uint32_t) wv, doff, 32u * (uint32_t) i);
    };
    float acc[4][8];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int L = 0; L < 8; ++L) acc[r][L] = 0.0f;
    auto compute = [&](const uint8_t* sw, const uint8_t* sh, const float* sd) __attribute__((always_inline)) {
        const uint32_t* wr = (const uint32_t*) (sw + (16 * wave + lr) * Q80_WS);
        const uint8_t* ah = sh + Q80_HS * (uint32_t) (lr >> 1) + 512 * (lr & 1) + 16 * gq;
        const int odd = 128 * (lr & 1);   // (chunk 4 i + gq at position ^ 8)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            // two blocks, 17 dwords: the even block's quants start 2 bytes into a dword
            const uint32_t e0 = wr[17 * p + gq], e1 = wr[17 * p + gq + 1];
            const uint32_t e2 = wr[17 * p + gq + 4], e3 = wr[17 * p + gq + 5];
            const uint32_t o0 = wr[17 * p + gq + 9], o1 = wr[17 * p + gq + 13];
            const uint32_t dd[2] = {wr[17 * p], wr[17 * p + 8]};
            const uint32_t q0[2] = {__builtin_amdgcn_alignbyte(e1, e0, 2), o0};
            const uint32_t q1[2] = {__builtin_amdgcn_alignbyte(e3, e2, 2), o1};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int i = 2 * p + h;
                const float dx = h2f((uint16_t) (h ? dd[h] >> 16 : dd[h] & 0xffffu));
                const q80_h4 b0 = q80_to_h4(q0[h]), b1 = q80_to_h4(q1[h]);
                const q80_h8 a = *(const q80_h8*) (ah + (i & 2 ? -odd : odd) + 64 * i);
                const float4 dy = *(const float4*) (sd + Q80_NR * i + 4 * gq);
                const q80_h4 a0 = {a[0], a[1], a[2], a[3]}, a1 = {a[4], a[5], a[6], a[7]};
                q80_f16 z;
#pragma unroll
                for (int k = 0; k < 16; ++k) z[k] = 0.0f;
                const q80_f16 s0 = __builtin_amdgcn_mfma_f32_16x16x4f16(a0, b0, z, 0, 0, 0);
                const q80_f16 s1 = __builtin_amdgcn_mfma_f32_16x16x4f16(a1, b1, z, 0, 0, 0);
                const float d[4] = {dx * dy.x, dx * dy.y, dx * dy.z, dx * dy.w};
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int L = 0; L < 4; ++L) {
                        acc[r][L] = __builtin_fmaf(d[r], s0[4 * L + r], acc[r][L]);
                        acc[r][4 + L] = __builtin_fmaf(d[r], s1[4 * L + r], acc[r][4 + L]);
                    }
            }
        }
    };
    issue(s_w0, s_h0, s_d0, 0);
    for (int i = 0; i < steps; i += 2) {
        vm_wait<0>();
        lds_barrier();
        if (i + 1 < steps) issue(s_w1, s_h1, s_d1, i + 1);
        compute(s_w0, s_h0, s_d0);
        if (i + 1 >= steps) break;
        vm_wait<0>();
        lds_barrier();
        if (i + 2 < steps) issue(s_w0, s_h0, s_d0, i + 2);
        compute(s_w1, s_h1, s_d1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 4 * gq + r;
        const float* a = acc[r];
        const float o = ((a[4] + a[0]) + (a[6] + a[2])) + ((a[5] + a[1]) + (a[7] + a[3]));
        if (row < ntok) {
            const int e = s_et[row][0], tt = s_et[row][1];
            float* dp = (float*) ((char*) m.dst + (size_t) e * m.dst_nb1 + (size_t) tt * m.dst_nb2);
            dp[r0 + 16 * wave + lr] = o;
        }
    }
}

// Rows of 16-byte aligned groups of eight blocks; 64-row tiles.
bool mf_q80_supported(const MmidArgs& m) {
    return m.type == T_Q8_0 && m.nb1 % 16 == 0 && m.nb2 % 16 == 0 && ((uintptr_t) m.w & 15) == 0 && m.K % 256 == 0 &&
           m.N % MF_M == 0 && (uint64_t) MF_M * m.nb1 < (1ull << 31) && m.dst_nb1 % 4 == 0 && m.dst_nb2 % 4 == 0;
}

int64_t mf_q80_groups(const MmidArgs& m) { return mf_max_items(m, Q80_NR) * (m.N / MF_M); }

int launch_mf_q80(const MfLaunch& lp, int nz, hipStream_t stream) {
    for (int z = 0; z < nz; ++z)
        if (!lp.m[z].act_h || !lp.m[z].act_hd) return -2;
    hipLaunchKernelGGL(k_mmid_mfma_q80, dim3(lp.groups * (unsigned) nz), dim3(256), 0, stream, lp);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

// Four lanes' worth of a row's f16 copy per thread: chunk c of block b.
__global__ void __launch_bounds__(256) k_q80_to_h(const uint8_t* __restrict__ q, int64_t nblk, _Float16* __restrict__ h,
                                                  float* __restrict__ hd) {
    const int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x;
    const int64_t b = i >> 2;
    if (b >= nblk) return;
    const int c = (int) (i & 3);
    const uint8_t* src = q + 34 * (size_t) b;
    q80_h8 v;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = (_Float16) (float) (int8_t) src[2 + 4 * c + k];
        v[4 + k] = (_Float16) (float) (int8_t) src[18 + 4 * c + k];
    }
    *(q80_h8*) (h + 32 * (size_t) b + 8 * c) = v;
    if (c == 0) hd[b] = h2f(ld_unaligned<uint16_t>(src));
}

int launch_q80_to_f16(const uint8_t* q, int64_t K, int64_t n_rows, uint16_t* h, float* hd, hipStream_t stream) {
    if (K % 32 || n_rows <= 0 || ((uintptr_t) h & 15)) return -2;
    const int64_t nblk = n_rows * (K / 32);
    hipLaunchKernelGGL(k_q80_to_h, dim3((unsigned) ((4 * nblk + 255) / 256)), dim3(256), 0, stream, q, nblk,
                       (_Float16*) h, hd);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

// ---- GEMV -----------------------------------------------------------------------
//
// A wave takes 8 weight rows, lane (row, n) the AVX lane n of its row.  The rows'
// whole bytes are copied straight into LDS by buffer loads that are all in flight
// at once (K = 2048: 19 instructions of 1 KB per wave), so a row costs one memory
// latency however long it is; the waves share the bin's activation rows (quants as
// dwords, scales as f32, 36 bytes per block) and nothing else.  The LDS row stride
// is 32 bytes past a multiple of 256: the 64 lanes' reads at one block fall on
// distinct banks.  16 rows per workgroup: 768 workgroups for a T = 1 gate + up
// launch, three resident per CU.  Bound: the chain grouping -> slot -> rows, then
// HBM.  T = 1, 30B layer: 17.6 us per launch (k_mmid_gemv, rows staged through
// registers in three rounds) -> 9.1 us, 26.7 MB of gate + up in 2.9 TB/s.
constexpr int QG_WAVES = 2;    // waves per workgroup (16 rows)
constexpr int QG_CT = 4;       // activation rows staged per pass, at most
constexpr uint32_t QG_LDS = 80 * 1024;   // LDS per workgroup, at most (two per CU)

// 16-byte chunks of a staged row: its bytes, then padding up to 2 mod 16
__host__ __device__ inline uint32_t qg_chunks(int64_t K) {
    const uint32_t n = (uint32_t) (K / 32 * 34 / 16);
    return n + ((18u - (n & 15u)) & 15u);
}
// bytes of a wave's weight region: whole copy instructions
__host__ __device__ inline uint32_t qg_wave_bytes(int64_t K) { return (8u * qg_chunks(K) + 63u) / 64u * 1024u; }
__host__ __device__ inline uint32_t qg_lds(int64_t K, int ct) {
    return QG_WAVES * qg_wave_bytes(K) + (uint32_t) ct * (uint32_t) (K / 32) * 36u;
}
// activation rows staged per pass: no more than a bin can hold, or than fit
__host__ __device__ inline int qg_stage_rows(int64_t max_rows, int64_t K) {
    int ct = max_rows < 1 ? 1 : max_rows < QG_CT ? (int) max_rows : QG_CT;
    while (ct > 1 && qg_lds(K, ct) > QG_LDS) --ct;
    return ct;
}

struct QgPair {
    MmidArgs m[2];
};

__global__ void __launch_bounds__(QG_WAVES * 64) k_mmid_gemv_q80(QgPair pr) {
    const MmidArgs& m = pr.m[blockIdx.z];
    extern __shared__ __align__(16) uint32_t lds[];
    __shared__ int s_chunk[QG_CT][3];   // (e, t, activation row) of the staged rows
    const int g = blockIdx.y;
    const int64_t r0 = (int64_t) blockIdx.x * (8 * QG_WAVES);
    if (r0 >= m.N) return;
    const int n_act = *m.n_active;
    const int p0 = m.active_off[g], p1 = m.active_off[g + 1];
    const int bin = m.active[g];
    if (g >= n_act) return;
    if (m.mfma_min_rows > 0 && p1 - p0 >= m.mfma_min_rows) return;   // matrix cores take it
    int64_t mat = bin;
    if (m.slot_of) mat = (bin < m.n_slot_of) ? m.slot_of[bin] : -1;
    const int CT = qg_stage_rows(m.max_rows, m.K);
    int pe = 0, pt = 0;
    if ((int) threadIdx.x < min(p1 - p0, CT)) {
        pe = m.rows[2 * (p0 + threadIdx.x)];
        pt = m.rows[2 * (p0 + threadIdx.x) + 1];
    }
    if (mat < 0 || mat >= m.n_as) {
        if (threadIdx.x == 0 && m.status) atomicOr(m.status, 4);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb = (int) (m.K / QK8_0);
    const uint32_t nch = (uint32_t) nb * 34u / 16u, c16 = qg_chunks(m.K);
    const int64_t wr0 = r0 + 8 * wave;
    const int wrows = (int) (m.N - wr0 < 8 ? (m.N - wr0 > 0 ? m.N - wr0 : 0) : 8);
    const uint32_t wbytes = qg_wave_bytes(m.K);
    {   // this wave's rows, all copies in flight; slots of no row are past the buffer's end (no access)
        const uint8_t* wp = m.w + (size_t) __builtin_amdgcn_readfirstlane((int) mat) * m.nb2 + (size_t) (wrows > 0 ? wr0 : r0) * m.nb1;
        const i32x4 w4 = rsrc_words(wp, wrows > 0 ? (uint32_t) (wrows - 1) * (uint32_t) m.nb1 + 16u * nch : 0u);
        const i32x4 wrsrc = i32x4{__builtin_amdgcn_readfirstlane(w4.x), __builtin_amdgcn_readfirstlane(w4.y),
                                  __builtin_amdgcn_readfirstlane(w4.z), __builtin_amdgcn_readfirstlane(w4.w)};
        const uint32_t l0 = (uint32_t) (uintptr_t) lds + (uint32_t) wave * wbytes;
        uint32_t row = (uint32_t) lane / c16, c = (uint32_t) lane - row * c16;
        for (uint32_t o = 0; o < wbytes; o += 1024u) {
            const bool ok = row < (uint32_t) wrows && c < nch;
            dma_b128(wrsrc, l0 + o, ok ? row * (uint32_t) m.nb1 + 16u * c : 0x7ffffff0u, 0u);
            c += 64u;
            while (c >= c16) {
                c -= c16;
                ++row;
            }
        }
    }
    const uint32_t AB = QG_WAVES * wbytes / 4;                  // staged quants [CT][8 nb] dwords
    const uint32_t DB = AB + (uint32_t) CT * 8u * (uint32_t) nb;   // staged scales [CT][nb]
    const int rl = lane >> 3, n = lane & 7;
    const uint32_t* wl = lds + (uint32_t) wave * wbytes / 4 + (uint32_t) rl * c16 * 4u;
    for (int pc = p0; pc < p1; pc += CT) {
        const int cnt = (p1 - pc) < CT ? (p1 - pc) : CT;
        __syncthreads();   // previous rows consumed
        if ((int) threadIdx.x < cnt) {
            const int e = pc == p0 ? pe : m.rows[2 * (pc + threadIdx.x)];
            const int t = pc == p0 ? pt : m.rows[2 * (pc + threadIdx.x) + 1];
            s_chunk[threadIdx.x][0] = e;
            s_chunk[threadIdx.x][1] = t;
            s_chunk[threadIdx.x][2] = (int) ((int64_t) (e % m.b_ne1) + (int64_t) t * m.b_ne1);
        }
        __syncthreads();
        for (int tk = 0; tk < cnt; ++tk) {
            const uint8_t* y = m.act_q + (size_t) s_chunk[tk][2] * m.act_row_bytes;
#pragma unroll 4
            for (int idx = threadIdx.x; idx < 8 * nb; idx += QG_WAVES * 64)
                lds[AB + (uint32_t) (tk * 8 * nb + idx)] = ld_unaligned<uint32_t>(y + 34 * (idx >> 3) + 2 + 4 * (idx & 7));
            for (int b = threadIdx.x; b < nb; b += QG_WAVES * 64)
                lds[DB + (uint32_t) (tk * nb + b)] = fbits(h2f(ld_unaligned<uint16_t>(y + 34 * b)));
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the copies into LDS are not the compiler's to wait for)
        __syncthreads();
        auto rows_dot = [&](auto nt_tag, int tk0) {
            constexpr int NT = decltype(nt_tag)::value;
            float acc[NT], v[NT];
#pragma unroll
            for (int u = 0; u < NT; ++u) acc[u] = 0.0f;
#pragma unroll 4
            for (int p = 0; p < nb / 2; ++p) {
                const uint32_t e0 = wl[17 * p + n], e1 = wl[17 * p + n + 1], o0 = wl[17 * p + n + 9];
                const uint32_t d0 = wl[17 * p], d1 = wl[17 * p + 8];
                const int q0 = (int) __builtin_amdgcn_alignbyte(e1, e0, 2), q1 = (int) o0;
                const float w0 = h2f((uint16_t) (d0 & 0xffffu)), w1 = h2f((uint16_t) (d1 >> 16));
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    const uint32_t* ya = lds + AB + (uint32_t) ((tk0 + u) * 8 * nb + 16 * p + n);
                    const float2 yd = *(const float2*) (lds + DB + (uint32_t) ((tk0 + u) * nb + 2 * p));
                    const int s0 = sdot4(q0, (int) ya[0], 0), s1 = sdot4(q1, (int) ya[8], 0);
                    acc[u] = __builtin_fmaf(w0 * yd.x, (float) s0, acc[u]);
                    acc[u] = __builtin_fmaf(w1 * yd.y, (float) s1, acc[u]);
                }
            }
            reduce8_mt<NT>(acc, v);
            if (n == 0 && rl < wrows) {
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    const int e = s_chunk[tk0 + u][0], t = s_chunk[tk0 + u][1];
                    float* d = (float*) ((char*) m.dst + (size_t) e * m.dst_nb1 + (size_t) t * m.dst_nb2);
                    d[wr0 + rl] = v[u];
                }
            }
        };
        if (cnt == 4) {
            rows_dot(std::integral_constant<int, 4>{}, 0);
        } else {
            int tk0 = 0;
            if (cnt >= 2) {
                rows_dot(std::integral_constant<int, 2>{}, 0);
                tk0 = 2;
            }
            if (tk0 < cnt) rows_dot(std::integral_constant<int, 1>{}, tk0);
        }
    }
}

int launch_gemv_q80(const MmidArgs* m, int nz, hipStream_t stream) {
    const MmidArgs& a = m[0];
    for (int z = 0; z < nz; ++z) {
        const MmidArgs& b = m[z];
        // K % 256: rows are whole 16-byte chunks (272 bytes per 256 values)
        if (b.type != T_Q8_0 || b.K % 256 || ((uintptr_t) b.w & 15) || b.nb1 % 16 || b.nb2 % 16 ||
            (uint64_t) b.nb1 * 8 >= (1ull << 30) || b.act_row_bytes != (size_t) (b.K / 32) * 34 || b.n_as > 0x7fffffff ||
            b.swiglu_gate)
            return -2;
    }
    if (a.K > 8192) return -2;
    const uint32_t lds_bytes = qg_lds(a.K, qg_stage_rows(a.max_rows, a.K));
    if (lds_bytes > QG_LDS) return -2;
    const dim3 grid((unsigned) ((a.N + 8 * QG_WAVES - 1) / (8 * QG_WAVES)), (unsigned) a.max_active, (unsigned) nz);
    if (grid.y == 0) return 0;
    QgPair pr;
    pr.m[0] = a;
    pr.m[1] = m[nz - 1];
    hipLaunchKernelGGL(k_mmid_gemv_q80, grid, dim3(QG_WAVES * 64), lds_bytes, stream, pr);
    return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace qw
