// fa_fwd.h -- what the prefill kernels share: the sequences of a call, the
// split plan and the list of work items that every workgroup builds from them.
#pragma once
#include "fa_common.h"
#include "fa_kernel_args.h"

#include <type_traits>

namespace fa {

constexpr int kMaxBatchLds = 2048;

struct BatchInfo {
    int sq, sk, rows, mt, lo, hi;
    int len0;  // kvcache: cache_seqlens[b] before this call's append, else 0
    int lp;    // kvcache: cache_leftpad[b] (key j is cache row lp + j), else 0
};

template <int BM>
__device__ __forceinline__ void batch_info(const FwdArgs& a, int b, BatchInfo& bi) {
    int sq = a.cu_seqlens_q ? a.cu_seqlens_q[b + 1] - a.cu_seqlens_q[b] : a.Sq;
    int sk;
    bi.len0 = a.seqlens_k ? a.seqlens_k[b] : 0;
    bi.lp = a.leftpad ? min(max(a.leftpad[b], 0), a.kv_capacity) : 0;
    if (a.seqlens_k)  // cache_seqlens (+ this call's new tokens) / seqused_k
        sk = bi.len0 + (a.cu_knew ? a.cu_knew[b + 1] - a.cu_knew[b] : a.seqlen_new) - bi.lp;
    else if (a.cu_seqlens_k) sk = a.cu_seqlens_k[b + 1] - a.cu_seqlens_k[b];
    else sk = a.Sk;
    sq = min(max(sq, 0), a.Sq);  // Sq is max_seqlen_q for varlen: bounds the tiles
    sk = min(max(sk, 0), a.kv_capacity - bi.lp);
    bi.sq = sq;
    bi.sk = sk;
    bi.rows = sq * a.g;
    bi.mt = (bi.rows + BM - 1) / BM;
    // union of the keys visible to any row of this sequence
    const int lo = max(0, key_lo(sk - sq, a.wl, a.chunk));
    const int hi = min(sk, key_hi(sk - 1, a.wr, a.chunk) + 1);
    bi.lo = lo;
    bi.hi = max(hi, lo);
}

__device__ __forceinline__ void split_of(const FwdArgs& a, int range, int chunk_auto, int& ns, int& chunk) {
    if (!a.allow_split || range <= 0) {
        ns = 1;
        chunk = max(range, 1);
    } else if (a.num_splits > 0) {
        ns = a.num_splits;
        chunk = (range + ns - 1) / ns;
    } else {
        chunk = chunk_auto;
        ns = (range + chunk - 1) / chunk;
    }
}

// Builds the per-batch work prefix in LDS. Every workgroup computes the same
// plan; workgroup 0 also publishes it for the combine kernel.
template <int BM, int BN, int NT, int NW>
__device__ void build_schedule(const FwdArgs& a, int* s_pref, long long* s_red, int& total, int& chunk_auto) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    long long work = 0, base = 0;
    for (int b = tid; b < a.B; b += NT) {
        BatchInfo bi;
        batch_info<BM>(a, b, bi);
        long long tiles = (long long)a.Hk * bi.mt;
        base += tiles;
        work += tiles * (bi.hi - bi.lo);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        work += __shfl_xor(work, o);
        base += __shfl_xor(base, o);
    }
    if (lane == 0) {
        s_red[wave * 2] = work;
        s_red[wave * 2 + 1] = base;
    }
    __syncthreads();
    work = 0;
    base = 0;
    for (int w = 0; w < NW; ++w) {
        work += s_red[w * 2];
        base += s_red[w * 2 + 1];
    }
    int ca = 0x3fffffff;
    if (a.allow_split && a.num_splits <= 0 && base < a.target_items) {
        long long c = (work + a.target_items - 1) / a.target_items;
        c = c < a.min_chunk ? a.min_chunk : c;
        c = (c + BN - 1) / BN * BN;
        ca = (int)(c > 0x3fffffff ? 0x3fffffff : c);
    }
    chunk_auto = ca;
    for (int b = tid; b < a.B; b += NT) {
        BatchInfo bi;
        batch_info<BM>(a, b, bi);
        int ns, chunk;
        split_of(a, bi.hi - bi.lo, ca, ns, chunk);
        s_pref[b + 1] = a.Hk * bi.mt * ns;
        if (blockIdx.x == 0 && a.sched) a.sched[a.B + 1 + b] = ns;
    }
    __syncthreads();
    if (wave == 0) {
        const int seg = (a.B + 63) / 64;
        const int b0 = lane * seg;
        int local = 0;
        for (int k = 0; k < seg; ++k) {
            int b = b0 + k;
            if (b < a.B) local += s_pref[b + 1];
        }
        int incl = local;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            int v = __shfl_up(incl, o);
            if (lane >= o) incl += v;
        }
        int run = incl - local;
        for (int k = 0; k < seg; ++k) {
            int b = b0 + k;
            if (b < a.B) {
                run += s_pref[b + 1];
                s_pref[b + 1] = run;
            }
        }
        if (lane == 0) s_pref[0] = 0;
    }
    __syncthreads();
    total = s_pref[a.B];
    if (blockIdx.x == 0 && a.sched) {
        for (int b = tid; b <= a.B; b += NT) a.sched[b] = s_pref[b];
    }
}

// Without a split: the item list of a small ragged batch with the sequences in
// order of falling item count (s_ord[p]: sequence at place p of the list, by
// which s_pref goes), so that the long ones do not come last.
constexpr int kOrdered = 64;
__device__ __forceinline__ bool ordered(const FwdArgs& a) { return a.cu_seqlens_q && a.B <= kOrdered && !a.allow_split; }
template <int BM>
__device__ int ordered_schedule(const FwdArgs& a, int* s_pref, int* s_ord) {
    const int lane = threadIdx.x & 63;
    if (threadIdx.x < 64) {
        int n = -1;
        if (lane < a.B) {
            BatchInfo bi;
            batch_info<BM>(a, lane, bi);
            n = a.Hk * bi.mt;
        }
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

// The pipelined prefill (fa_fwd_pipe.h) by kernel head dim
void launch_prefill_pipe_fp8(const FwdArgs& a, int grid, hipStream_t stream);
void launch_prefill_pipe64(const FwdArgs& a, int dtype, int grid, hipStream_t stream);
void launch_prefill_pipe128(const FwdArgs& a, int dtype, int grid, hipStream_t stream);
void launch_prefill_pipe256(const FwdArgs& a, int dtype, int grid, hipStream_t stream);

}  // namespace fa
