// qw_mfma.hpp -- what the matrix-core mul_mat_id kernels share: copies straight
// into LDS, the work items of a launch, the launch arguments.
#pragma once

#include <algorithm>

#include "qw_kernels.hpp"

namespace qw {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4m __attribute__((ext_vector_type(4)));

constexpr int MF_M = 64;          // weight rows per workgroup (4 waves x 16)

// Waits until at most N of this wave's vector memory operations are in flight.
template <int N>
__device__ __forceinline__ void vm_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Buffer resource words over [base, base + bytes) (the layout
// __builtin_amdgcn_make_buffer_rsrc builds; loads past the end return zeros).
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ i32x4 rsrc_words(const void* base, uint32_t bytes) {
    const uint64_t a = (uint64_t) base;
    return i32x4{(int) (uint32_t) a, (int) ((uint32_t) (a >> 32) & 0xffffu), (int) bytes, 0x00020000};
}

// Buffer loads straight into LDS: lane l's 16 (4) bytes from voff + soff land at
// LDS byte lds_base + 16 l (4 l).  Written as instructions, not through the
// compiler's builtin: the compiler then inserts no wait of its own before the
// LDS reads (it would wait for every copy in flight, the prefetched stages
// included); the kernel waits with vm_wait and orders waves with a barrier.
// M0 holds the LDS base for the instruction and is restored after it.
__device__ __forceinline__ void dma_b128(i32x4 rsrc, uint32_t lds_base, uint32_t voff, uint32_t soff) {
    uint32_t keep;
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
        : "=&s"(keep)
        : "s"(lds_base), "v"(voff), "s"(rsrc), "s"(soff)
        : "memory");
}
__device__ __forceinline__ void dma_b32(i32x4 rsrc, uint32_t lds_base, uint32_t voff, uint32_t soff) {
    uint32_t keep;
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dword %2, %3, %4 offen lds\n\ts_mov_b32 m0, %0"
        : "=&s"(keep)
        : "s"(lds_base), "v"(voff), "s"(rsrc), "s"(soff)
        : "memory");
}

// Work items: the routed rows of each heavy expert (at least mfma_min_rows)
// cut into chunks of R rows; item i is chunk c of active expert g, items in
// expert order.  Wave 0 scans the active experts' chunk counts 64 at a time and
// leaves (g, c) in s_item, g = -1 past the last item.  Splitting an expert's
// rows over workgroups keeps the longest workgroup at R rows whatever the skew
// of the routing (one expert can hold every token of the batch).
__device__ __forceinline__ void mf_item(const MmidArgs& m, int item, int R, int wave, int lane, int* s_item) {
    if (wave == 0) {
        const int n = *m.n_active;
        int run = 0, fg = -1, fc = 0;
        for (int base = 0; base < n; base += 64) {
            const int j = base + lane;
            int ch = 0;
            if (j < n) {
                const int cnt = m.active_off[j + 1] - m.active_off[j];
                ch = cnt >= m.mfma_min_rows ? (cnt + R - 1) / R : 0;
            }
            int incl = ch;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(incl, o);
                if (lane >= o) incl += v;
            }
            const int excl = incl - ch;
            const uint64_t hit = __ballot(item >= run + excl && item < run + incl);
            if (hit) {   // uniform
                const int src = __ffsll((unsigned long long) hit) - 1;
                fg = base + src;
                fc = item - run - __shfl(excl, src);
                break;
            }
            run += __shfl(incl, 63);
        }
        if (lane == 0) {
            s_item[0] = fg;
            s_item[1] = fc;
        }
    }
    __syncthreads();
}

// Upper bound on the items of a launch: at most min(max_active, n_pairs /
// mfma_min_rows) heavy experts, each with at most one partial chunk.
inline int64_t mf_max_items(const MmidArgs& m, int R) {
    const int64_t heavy = std::min<int64_t>(m.max_active, m.n_pairs / std::max(m.mfma_min_rows, 1));
    return heavy + m.n_pairs / R;
}

// One launch runs the matrix-core part of one mul_mat_id, or of two of the same
// type, shape and grouping (gate and up of an FFN): workgroups [0, groups) take
// m[0], [groups, 2 groups) m[1], so the second matrix's workgroups fill the CUs
// the first one's last round leaves idle.
struct MfLaunch {
    MmidArgs m[2];
    uint32_t groups;   // workgroups per matrix
};

// mmid_q80.hip: the Q8_0 form of a launch (mmid_mfma_supported and act_h / act_hd set)
int launch_mf_q80(const MfLaunch& lp, int nz, hipStream_t stream);
int64_t mf_q80_groups(const MmidArgs& m);
bool mf_q80_supported(const MmidArgs& m);

}  // namespace qw
