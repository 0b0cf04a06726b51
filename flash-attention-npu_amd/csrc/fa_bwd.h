// fa_bwd.h -- what the backward kernels share: the sequences of a call and
// the list of work items that every workgroup builds from them.
#pragma once
#include "fa_common.h"
#include "fa_kernel_args.h"

#include <type_traits>

namespace fa {

namespace bw {
constexpr int kMaxBatch = 2048;
}  // namespace bw

struct BwBatch {
    int sq, sk, rows;  // query positions, keys, packed rows (sq * g)
};

__device__ __forceinline__ BwBatch bw_batch(const BwdArgs& a, int b) {
    BwBatch r;
    int sq = a.cu_seqlens_q ? a.cu_seqlens_q[b + 1] - a.cu_seqlens_q[b] : a.Sq;
    int sk = a.cu_seqlens_k ? a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b] : a.Sk;
    r.sq = min(max(sq, 0), a.Sq);
    r.sk = min(max(sk, 0), a.Sk);
    r.rows = r.sq * a.g;
    return r;
}

// Per-batch item prefix in LDS (s_pref[0..B]); items(b) is the work item
// count of batch b. Every workgroup computes the same table.
template <int NT, class F>
__device__ __forceinline__ int bw_prefix(const BwdArgs& a, int* s_pref, F items) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int b = tid; b < a.B; b += NT) s_pref[b + 1] = items(b);
    __syncthreads();
    if (wave == 0) {
        const int seg = (a.B + 63) / 64, b0 = lane * seg;
        int local = 0;
        for (int k = 0; k < seg; ++k)
            if (b0 + k < a.B) local += s_pref[b0 + k + 1];
        int incl = local;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            int v = __shfl_up(incl, o);
            if (lane >= o) incl += v;
        }
        int run = incl - local;
        for (int k = 0; k < seg; ++k)
            if (b0 + k < a.B) {
                run += s_pref[b0 + k + 1];
                s_pref[b0 + k + 1] = run;
            }
        if (lane == 0) s_pref[0] = 0;
    }
    __syncthreads();
    return s_pref[a.B];
}

// The same with the sequences of a small ragged batch in order of falling item
// count (s_ord[p]: sequence at place p of the list), so that the long ones do
// not come last; others keep their order. s_pref then goes by place.
constexpr int kOrdered = 64;
template <int NT, class F>
__device__ __forceinline__ int bw_ordered_prefix(const BwdArgs& a, int* s_pref, int* s_ord, F items) {
    if (!a.cu_seqlens_q || a.B > kOrdered) return bw_prefix<NT>(a, s_pref, items);
    const int lane = threadIdx.x & 63;
    if (threadIdx.x < 64) {
        const int n = lane < a.B ? items(lane) : -1;
        int place = 0, before = 0;
        for (int c = 0; c < a.B; ++c) {
            const int m = __shfl(n, c);
            const bool first = m > n || (m == n && c < lane);
            place += first ? 1 : 0;
            before += first ? m : 0;
        }
        if (lane < a.B) {
            s_ord[place] = lane;
            s_pref[place] = before;
            if (place == a.B - 1) s_pref[a.B] = before + n;
        }
    }
    __syncthreads();
    return s_pref[a.B];
}

__device__ __forceinline__ int bw_find_batch(const int* s_pref, int B, int w) {
    int bl = 0, bh = B;
    while (bh - bl > 1) {
        const int mid = (bl + bh) >> 1;
        if (s_pref[mid] <= w) bl = mid;
        else bh = mid;
    }
    return bl;
}

// dQ and dsum without ALiBi or chunks (fa_bwd_dq.hip); 128-row items
bool bwd_dq_takes(const BwdArgs& a);
void launch_bwd_dq(const BwdArgs& a, int dtype, int d, int grid, hipStream_t stream);

// dK and dV at head dims 65..128 without soft cap, ALiBi or chunks (fa_bwd_kv.hip)
bool bwd_kv_takes(const BwdArgs& a);
void launch_bwd_kv(const BwdArgs& a, int dtype, int grid, hipStream_t stream);

}  // namespace fa
