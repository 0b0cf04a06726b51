// fa_fwd_pipe.h -- the prefill forward with one wave per SIMD (compiled per head
// dim by fa_fwd_pipe64 / 128 / 256.hip).
//
// The work items, masks and split of fa_fwd.hip; another inner loop. Four waves
// of RB x 32 packed rows; K and V tiles go straight from memory into four LDS
// buffers, two tiles ahead. Per 32 keys a wave forms S^T = K.Q^T and
// O^T += V^T.P^T with 32x32x16 MFMA (a lane holds one row and 16 keys, which is
// the packed P^T operand; V^T by transpose reads).
//   * Two waves per SIMD of 32 rows each (fa_fwd.hip) read an operand from LDS
//     for two products and do their products and their softmax mostly one after
//     the other. 64 rows to a wave halve the LDS reads and take the registers of
//     the whole SIMD, so the wave overlaps by itself: while the softmax of 32
//     keys runs, the scores of the next 32 are formed, and their maximum is
//     taken under the P.V products, in slots of one MFMA and a share of the
//     vector work (unit()).
//   * The running maximum moves only when a score exceeds it by 2^8 (raise()),
//     between two units, when no product is in flight that it would change.
// bf16, one box: B4 S4096 H32/8 D128 full mask 1082 -> 977 us (1.13 PFLOP/s; an
// 8192^3 matrix product reaches 1.24 on this card), causal 593 -> 540; chunked
// prefill B4 2048 onto 6144 895 -> 813, with rotary and append 953 -> 860.
// Without the softmax 785 us, with products alone 730 (of 920, another box).
// Head dim 256 (32 rows per wave, 32-key tiles), window 1024 and soft cap, B2 S4096
// H16/8: 281 -> 190 us; head dim 64 (bound by the softmax, whose share of the
// products is twice as large), B8 S1025 H16 fp16: 102 -> 97 (then 4 more for the
// part tile that every item ends in, clear_v).
#pragma once
#include "fa_fwd.h"
#include "fa_pipe.h"
#include "fa_rope.h"

namespace fa {
namespace pipe {

constexpr int NT = 256, NBUF = 4;
constexpr float kLazy = 8.f;  // log2 headroom before the running maximum moves

// Slot of chunk c in row r: fa_pipe.h's; 128-byte rows (two to a line of LDS
// banks) take theirs from the row pair, conflict free for the same reads.
template <int ROW>
__device__ __forceinline__ int slot_of(int r, int c) {
    return ROW == 128 ? c ^ ((((r >> 1) & 1) << 2) | ((r >> 2) & 3)) : swz(r, c);
}

// EB: bytes per element of q, K and V
template <int HD, int RBLK, int EB>
struct PipeCfg {
    static constexpr int RB = RBLK;            // 32-row blocks per wave
    static constexpr int BM = 4 * RB * 32;     // packed rows per work tile
    static constexpr int ROW = EB * HD;        // bytes
    static constexpr int NH = 512 / ROW;       // 32-key halves per LDS tile
    static constexpr int BN = 32 * NH;
    static constexpr int KS = ROW / 32;        // K operand reads: 16 bytes of each half wave
    static constexpr int DB = HD / 32;         // 32-dim blocks of O
    static constexpr int CH = ROW / 16;        // 16-byte chunks per row
    static constexpr int RPL = 64 / CH;        // rows per LDS load
    static constexpr int KT = BN * ROW;        // bytes of a K (or V) tile
    static constexpr int TILE = 2 * KT;
};

// CAP: soft cap (scores are capped and in log2 units once their maximum is taken)
template <int DT, int HD, int RBLK, bool PAGED, bool ROT, bool CAP>
__global__ void __launch_bounds__(NT, 1) fa_prefill_pipe_kernel(FwdArgs a) {
    constexpr bool F8 = DT == DT_FP8;
    constexpr int EB = F8 ? 1 : 2;
    static_assert(!(F8 && ROT), "no rotary with FP8");
    using C = PipeCfg<HD, RBLK, EB>;
    constexpr int RB = C::RB, BM = C::BM, BN = C::BN, NH = C::NH, KS = C::KS, DB = C::DB, CH = C::CH, ROW = C::ROW,
                  KT = C::KT, TILE = C::TILE, NE = 16 * RB;
    // slots: S products, then the P.V products of the first and the last 16 keys
    constexpr int QS = KS * 2 / EB;  // S products per row block: an FP8 read is two bf16 operands
    constexpr int SS = QS * RB, SP = DB * RB;
    static_assert(KT == 4 * 4 * 1024, "four loads of four waves bring a tile");
    __shared__ __attribute__((aligned(256))) char s_t[NBUF * TILE];
    __shared__ int s_pref[kMaxBatchLds + 1], s_ord[kOrdered];
    __shared__ long long s_red[8];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hi = lane >> 5;
    // K chunks past the head dim are 0 and stay so (no load writes them): q is 0
    // there, but another chunk's infinity times 0 is not. e4m3 has no infinity.
    if (!F8 && a.hd < HD) {
#pragma unroll
        for (int x = 0; x < NBUF; ++x)
            for (int at = tid * 16; at < KT; at += NT * 16) row_write(lds_addr(s_t) + x * TILE + at, u32x4{0u, 0u, 0u, 0u});
        __syncthreads();
    }
    int total, chunk_auto = 0;
    if (ordered(a)) total = ordered_schedule<BM>(a, s_pref, s_ord);
    else build_schedule<BM, C::BN, NT, 4>(a, s_pref, s_red, total, chunk_auto);

    const unsigned lds0 = lds_addr(s_t);
    const unsigned rowa = lds0 + col * ROW + (slot_of<ROW>(col, hi) << 4);  // chunk 2s + hi: ^ (s << 5)
    const int tr_r = 4 * hi + ((lane & 15) >> 2), tr_c = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    // dim block db: ^ (db << 6). FP8: a group of 16 lanes reads 8 rows of one chunk,
    // those of a whole operand: rows 4hi .. + 3 and 8 + 4hi .. + 3; db: ^ (db << 5)
    const int tr8_r = 4 * hi + ((lane >> 1) & 3) + 8 * ((lane >> 3) & 1);
    const unsigned tra = lds0 + KT + (lane & 1) * 8 +
                         (F8 ? tr8_r * ROW + (slot_of<ROW>(tr8_r, (lane >> 4) & 1) << 4)
                             : tr_r * ROW + (slot_of<ROW>(tr_r, tr_c) << 4));

    const char* qp = static_cast<const char*>(a.q);
    uint16_t* op = static_cast<uint16_t*>(a.out);
    float cs = CAP ? 1.f : a.scale_log2;  // (FP8: times the item's descales)
    // cap * tanh(scale s / cap) in log2 units = c1 - 2 c1 / (2^(c0 s) + 1)
    [[maybe_unused]] float c0 = CAP ? 2.f * a.scale_log2 / a.softcap : 0.f;
    [[maybe_unused]] const float c1 = a.softcap * kLog2e;

    for (int k = 0; k * (int)gridDim.x < total; ++k) {
        const int w = k * (int)gridDim.x + ((k & 1) ? (int)gridDim.x - 1 - (int)blockIdx.x : (int)blockIdx.x);
        if (w >= total) continue;
        int bl = 0, bh = a.B;
        while (bh - bl > 1) {
            const int mid = (bl + bh) >> 1;
            if (s_pref[mid] <= w) bl = mid;
            else bh = mid;
        }
        const int b = __builtin_amdgcn_readfirstlane(ordered(a) ? s_ord[bl] : bl);
        BatchInfo bi;
        batch_info<BM>(a, b, bi);
        int ns, chunk;
        split_of(a, bi.hi - bi.lo, chunk_auto, ns, chunk);
        const int local = w - __builtin_amdgcn_readfirstlane(s_pref[bl]);
        const int hk = local % a.Hk;
        const int split = (local / a.Hk) % ns;
        const int mt = bi.mt - 1 - local / a.Hk / ns;  // heaviest causal tiles first
        const bool final_out = ns == 1;
        const int crow = a.batch_idx ? min(max(a.batch_idx[b], 0), (a.block_table ? a.bt_rows : a.batch_cache) - 1) : b;
        const int g = a.g;
        const int diag0 = bi.sk - bi.sq;

        const int tile_row0 = mt * BM, tile_rows = min(BM, bi.rows - tile_row0);
        const int i_lo = tile_row0 / g, i_hi = (tile_row0 + tile_rows - 1) / g;
        int k_lo = max(0, key_lo(i_lo + diag0, a.wl, a.chunk));
        int k_hi = min(bi.sk, key_hi(i_hi + diag0, a.wr, a.chunk) + 1);
        if (ns > 1) {
            const int c0 = bi.lo + split * chunk;
            k_lo = max(k_lo, c0);
            k_hi = min(k_hi, c0 + chunk);
        }
        if (k_hi < k_lo) k_hi = k_lo;
        const int base = PAGED ? k_lo & ~(BN - 1) : k_lo;  // key of tile 0: a tile lies in one page
        const int ntiles = k_hi > k_lo ? (k_hi - base + BN - 1) / BN : 0;
        // tiles all of whose keys are visible to all rows: [t1, t2)
        const int f_lo = max(k_lo, key_lo(i_hi + diag0, a.wl, a.chunk)), f_hi = min(k_hi, key_hi(i_lo + diag0, a.wr, a.chunk) + 1);
        const int t1 = min(ntiles, (f_lo - base + BN - 1) / BN), t2 = max(t1, (f_hi - base) / BN);

        // ---- K / V tiles straight into LDS -------------------------------------------------
        const int kvh = hk / a.kvdiv;
        const char* kb = static_cast<const char*>(a.k) + EB * (int64_t)kvh * a.k_sh;
        const char* vb = static_cast<const char*>(a.v) + EB * (int64_t)kvh * a.v_sh;
        [[maybe_unused]] const int* btrow = nullptr;
        if constexpr (PAGED) {
            btrow = a.block_table + (int64_t)crow * a.bt_stride;
        } else if (a.cu_seqlens_k) {
            kb += EB * ((int64_t)a.cu_seqlens_k[b] + base) * a.k_si;
            vb += EB * ((int64_t)a.cu_seqlens_k[b] + base) * a.v_si;
        } else {
            kb += EB * ((int64_t)crow * a.k_sb + (int64_t)(bi.lp + base) * a.k_si);
            vb += EB * ((int64_t)crow * a.v_sb + (int64_t)(bi.lp + base) * a.v_si);
        }
        // Load u of the wave brings rows RPL * (4 wave + u) .., lane l chunk slot
        // l % CH of row l / CH (the swizzle is in the address read). Rows past
        // the last key of the item load that key: second set, for the last tile.
        unsigned ko[2][4], vo[2][4];
        [[maybe_unused]] uint64_t in_hd[4];  // K load u: lanes whose chunk lies in the head dim
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int r = C::RPL * (4 * wave + u) + lane / CH;
            const int c = min(slot_of<ROW>(r, lane % CH), EB * a.hd / 16 - 1);  // V: what is past the head dim is not written out
            in_hd[u] = __ballot(slot_of<ROW>(r, lane % CH) < EB * a.hd / 16);
            const int rl = min(r, k_hi - 1 - base - (ntiles - 1) * BN);
            ko[0][u] = (unsigned)(EB * r * (int)a.k_si + c * 16) + (3 - u) * 1024;
            vo[0][u] = (unsigned)(EB * r * (int)a.v_si + c * 16) + (3 - u) * 1024;
            ko[1][u] = (unsigned)(EB * rl * (int)a.k_si + c * 16) + (3 - u) * 1024;
            vo[1][u] = (unsigned)(EB * rl * (int)a.v_si + c * 16) + (3 - u) * 1024;
        }
        // Tiles are asked for in order; tiles past the end are the last one again.
        // Paged: page, first row in it and (read one tile early) block of the next.
        [[maybe_unused]] int pg = 0, in = 0, blk = 0;
        [[maybe_unused]] auto read_block = [&]() {
            blk = __builtin_amdgcn_readfirstlane(min(max(btrow[pg], 0), a.num_blocks - 1));
        };
        if constexpr (PAGED) {
            if (ntiles > 0) {
                pg = base / a.page;
                in = base - pg * a.page;
                read_block();
            }
        }
        auto load_tile = [&](int t, int buf, [[maybe_unused]] auto first) {
            const bool last = t >= ntiles - 1;
            int64_t ok, ov;
            if constexpr (PAGED) {
                ok = (int64_t)blk * a.k_sb + (int64_t)in * a.k_si;
                ov = (int64_t)blk * a.v_sb + (int64_t)in * a.v_si;
                in = last ? in : in + BN;
                pg = in == a.page ? pg + 1 : pg;
                in = in == a.page ? 0 : in;
                read_block();
            } else {
                ok = (int64_t)min(t, ntiles - 1) * BN * a.k_si;
                ov = (int64_t)min(t, ntiles - 1) * BN * a.v_si;
            }
            unsigned k4[4], v4[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                k4[u] = last ? ko[1][u] : ko[0][u];
                v4[u] = last ? vo[1][u] : vo[0][u];
                if constexpr (decltype(first)::value && PAGED) {  // rows before the item's first key load that key
                    const unsigned up = (unsigned)max(0, k_lo - base - (C::RPL * (4 * wave + u) + lane / CH));
                    k4[u] += EB * up * (unsigned)a.k_si;
                    v4[u] += EB * up * (unsigned)a.v_si;
                }
            }
            const unsigned wb = lds0 + TILE * buf + wave * 4096;
            if constexpr (F8) dma16x4(wb, kb + EB * ok - 3072, k4);
            else dma16x4(wb, kb + EB * ok - 3072, k4, in_hd);
            dma16x4(wb + KT, vb + EB * ov - 3072, v4);
        };
        if (ntiles > 0) {
            load_tile(0, 0, std::true_type{});
            load_tile(1, 1, std::false_type{});
            load_tile(2, 2, std::false_type{});
        }

        // V rows of a tile outside [begin, end) are no keys of the item: made 0 once
        // they are there, for 0 weight times an infinity of the repeated key is no
        // number (e4m3 has none). As masked loads it cost the whole loop 2.5 %; so, 1 %
        // where the last tile is a part one.
        [[maybe_unused]] auto clear_v = [&](int buf, int begin, int end) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int r = C::RPL * (4 * wave + u) + lane / CH;
                if (r < begin || r >= end) row_write(lds0 + TILE * buf + KT + wave * 4096 + 1024 * u + 16 * lane, u32x4{0u, 0u, 0u, 0u});
            }
        };
        const int last_end = k_hi - base - (ntiles - 1) * BN;
        const int part_tile = __builtin_amdgcn_readfirstlane(!F8 && last_end < BN ? ntiles - 1 : -1);

        [[maybe_unused]] float sc_v = 1.f;
        [[maybe_unused]] uint32_t flip = 0;
        if constexpr (F8) {
            const float qk = descale_at(a.qd, a.qd_sb, a.qd_sh, b, kvh) * descale_at(a.kd, a.kd_sb, a.kd_sh, b, kvh);
            sc_v = descale_at(a.vd, a.vd_sb, a.vd_sh, b, kvh);
            if constexpr (CAP) {
                c0 = 2.f * a.scale_log2 * qk / a.softcap;
            } else {
                // a negative factor goes to the signs of q; 0 must not meet the masks' infinity
                cs = a.scale_log2 * qk;
                flip = cs < 0.f ? 0x80008000u : 0u;
                cs = cs == 0.f ? 1e-30f : fabsf(cs);
            }
        }
        // ---- q as B operands: lane holds row col, chunks 2s + hi -------------------------------
        const int wrow0 = tile_row0 + wave * RB * 32;
        u32x4 qreg[RB][QS];
        int rlo[RB], rhi[RB];  // the row's visible keys, as offsets from the item's first tile
        [[maybe_unused]] int qi[RB];
        [[maybe_unused]] const uint16_t* qrows[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int r = wrow0 + rb * 32 + col;
            const bool ok = r < bi.rows;
            const int i = ok ? r / g : 0, h = hk * g + (ok ? r % g : 0);
            rlo[rb] = max(k_lo, key_lo(i + diag0, a.wl, a.chunk)) - base - 4 * hi;
            rhi[rb] = min(k_hi - 1, key_hi(i + diag0, a.wr, a.chunk)) - base - 4 * hi;
            const char* qrow = qp + EB * ((a.cu_seqlens_q ? ((int64_t)a.cu_seqlens_q[b] + i) * a.q_si
                                                          : (int64_t)b * a.q_sb + (int64_t)i * a.q_si) + (int64_t)h * a.q_sh);
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int c = 2 * s + hi;
                const u32x4 x = ok && c * 16 < EB * a.hd ? *reinterpret_cast<const u32x4*>(qrow + c * 16) : u32x4{0u, 0u, 0u, 0u};
                if constexpr (F8) {
                    qreg[rb][2 * s] = fp8x8_to_bf16(u32x2{x[0], x[1]}) ^ flip;
                    qreg[rb][2 * s + 1] = fp8x8_to_bf16(u32x2{x[2], x[3]}) ^ flip;
                } else {
                    qreg[rb][s] = x;
                }
            }
            if constexpr (ROT) {
                qi[rb] = i;
                qrows[rb] = reinterpret_cast<const uint16_t*>(qrow);
            }
        }
        if constexpr (ROT) {
            // q[b, i] is rotated at rot_pos / cache_seqlens[b] (+ i when causal or local)
            const int clast = (a.rot_dim >> 3) - 1;
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                int pos = (a.rot_pos ? a.rot_pos[b] : bi.len0) + (a.rot_same_pos ? 0 : qi[rb]);
                pos = min(max(pos, 0), a.seqlen_ro - 1);
                const uint16_t* rc = static_cast<const uint16_t*>(a.rot_cos) + (int64_t)pos * (a.rot_dim >> 1);
                const uint16_t* rs = static_cast<const uint16_t*>(a.rot_sin) + (int64_t)pos * (a.rot_dim >> 1);
                const bool ok = wrow0 + rb * 32 + col < bi.rows;
                auto rotate = [&](auto inter) {
                    constexpr bool I = decltype(inter)::value;
#pragma unroll
                    for (int s = 0; s < KS; ++s) {
                        const int c = 2 * s + hi;
                        const RopeOps r = rope_load(qrows[rb], min(c, clast), a.rot_dim, I, rc, rs);
                        const u32x4 x = rope_apply<DT>(qreg[rb][s], r, c, a.rot_dim, I);
                        if (ok && c <= clast) qreg[rb][s] = x;
                    }
                };
                if (a.rot_interleaved) rotate(std::true_type{});
                else rotate(std::false_type{});
            }
        }

        // q in accumulation registers, one tuple per operand (rotated in pieces, it would be put
        // together again before every product)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int s = 0; s < QS; ++s) asm volatile("" : "+a"(qreg[rb][s]));

        f32x16 o[RB][DB];
        float m[RB], l[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            m[rb] = -1e30f;  // finite floor: exp2(x - m) never forms inf - inf
            l[rb] = 0.f;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[rb][db][i] = 0.f;
        }

        // LDS addresses of this lane's operands in the tile read next, moved on
        // with the tile; opaque, so that the rest goes into the instructions' offsets
        unsigned ra[KS], ta[DB], tb[DB];
#pragma unroll
        for (int s = 0; s < KS; ++s) ra[s] = rowa ^ (s << 5);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            ta[db] = tra ^ (db << (F8 ? 5 : 6));
            tb[db] = (tra ^ (db << 6) ^ 32) + 8 * ROW;  // (FP8: one read)
        }
        auto move_on = [&](unsigned& x, unsigned by) {
            x += by;
            asm volatile("" : "+v"(x));
        };
        u32x4 kop[KS];
        std::conditional_t<F8, u32x2, u32x4> vop[2 * DB];
        auto read_rows = [&](int h, int s) {  // steps s and s + 1
            kop[s] = row_read(ra[s] + h * 32 * ROW);
            kop[s + 1] = row_read(ra[s + 1] + h * 32 * ROW);
        };
        auto read_tr = [&](int h, int x) {  // x, x + 1: step of 16 keys, then dim block
#pragma unroll
            for (int i = x; i < x + 2; ++i) {
                const int o_ = (h * 32 + i / DB * 16) * ROW;
                if constexpr (F8) vop[i] = tr8_read(ta[i % DB] + o_);
                else vop[i] = tr_read(ta[i % DB] + o_, tb[i % DB] + o_);
            }
        };

        float peak[RB];
        [[maybe_unused]] auto cap = [&](float x) {
            return __builtin_fmaf(-2.f * c1, __builtin_amdgcn_rcpf(fast_exp2(x * c0) + 1.f), c1);
        };
        auto visible = [&](f32x16 (&ns_)[RB], int e, int s0) {  // s0: key offset of the half
            const int rb = e / 16, i = e % 16, j = s0 + 8 * (i / 4) + i % 4;
            ns_[rb][i] = j >= rlo[rb] && j <= rhi[rb] ? ns_[rb][i] : -INFINITY;
        };
        // moves the running maximum to that of the scores where they exceed it by 2^8
        auto raise = [&](bool live) {
            bool need = false;
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) need |= peak[rb] * cs > m[rb] + kLazy;
            if (live && __ballot(need)) {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const float mn = fmaxf(m[rb], fmaxf(peak[rb], __shfl_xor(peak[rb], 32)) * cs);
                    const float alpha = fast_exp2(m[rb] - mn);
                    m[rb] = mn;
                    l[rb] *= alpha;
#pragma unroll
                    for (int db = 0; db < DB; ++db) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) o[rb][db][i] *= alpha;
                    }
                }
            }
        };
        // operand d of the reads s and s + 1
        auto k_operand = [&](const u32x4 (&x)[KS], int s, int d) -> u32x4 {
            if constexpr (F8) {
                const u32x4 r = x[s + d / 2];
                return fp8x8_to_bf16(d & 1 ? u32x2{r[2], r[3]} : u32x2{r[0], r[1]});
            } else {
                return x[s + d];
            }
        };
        const f32x16 zero = {};

        // One half tile: its softmax and P.V while the scores of the next are
        // formed (n_), one MFMA to a slot. Each score takes three slots: scaled, its
        // exponential, summed and packed; they are spread evenly up to the last
        // keys' P.V products.
        u32x4 pk[RB][2];
        float px[NE];
        auto unit = [&](f32x16 (&c_)[RB], f32x16 (&n_)[RB], auto ha, auto hb, int s0n, auto mask, auto more, auto ahead) {
            constexpr int A = decltype(ha)::value, B = decltype(hb)::value;
            int slot = 0;
            auto next = [&]() {
#pragma unroll
                for (int q = 0; q < NE; ++q) {
                    // q-th score: the first 16 keys of every row block, then the others
                    const int ks = q / (8 * RB), rb = q / 8 % RB, i = 8 * ks + q % 8;
                    const int at = q * (SS + SP - 2) / NE;
                    if (slot == at) px[q] = __builtin_fmaf(c_[rb][i], cs, -m[rb]);
                    if (slot == at + 1) px[q] = fast_exp2(px[q]);
                    if (slot == at + 2) {
                        l[rb] += px[q];
                        if (q & 1) pk[rb][ks][q / 2 % 4] = pack2<DT>(px[q - 1], px[q]);
                    }
                }
#pragma unroll
                for (int e = 0; e < NE; ++e) {
                    if (slot != SS + 2 + e * (2 * SP - 4) / NE) continue;
                    if constexpr (CAP) n_[e / 16][e % 16] = cap(n_[e / 16][e % 16]);
                    if constexpr (decltype(mask)::value) visible(n_, e, s0n);
                    if (e % 16 == 0) peak[e / 16] = n_[e / 16][0];
                    else peak[e / 16] = fmaxf(peak[e / 16], n_[e / 16][e % 16]);
                }
                ++slot;
                fence();
            };
            // operands are read two steps ahead, the last one read is used first
#pragma unroll
            for (int s = 0; s < KS; s += 2) {
#pragma unroll
                for (int d = 4 / EB - 1; d >= 0; --d) {
                    const u32x4 ka = k_operand(kop, s, d);
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) {
                        n_[rb] = mfma32<DT>(ka, qreg[rb][s * 2 / EB + d], s == 0 && d == 4 / EB - 1 ? zero : n_[rb]);
                        if (d == 4 / EB - 1 && rb == 0) {
                            if (s + 2 < KS) read_rows(A, s + 2);
                            else read_tr(B, 0);
                        }
                        next();
                    }
                }
            }
#pragma unroll
            for (int x = 0; x < 2 * DB; x += 2) {
#pragma unroll
                for (int d = 1; d >= 0; --d) {
                    u32x4 vt;
                    if constexpr (F8) vt = fp8x8_to_bf16(vop[x + d]);
                    else vt = vop[x + d];
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) {
                        o[rb][(x + d) % DB] = mfma32<DT>(vt, pk[rb][(x + d) / DB], o[rb][(x + d) % DB]);
                        if (d == 1 && rb == 0) {
                            if (x + 2 < 2 * DB) read_tr(B, x + 2);
                            else ahead();
                        }
                        more(x * RB + (1 - d) * RB + rb);
                        next();
                    }
                }
            }
        };

        if (ntiles > 0) {
            using H0 = std::integral_constant<int, 0>;
            wait_loads<0>();  // (with the q rows, which the compiler waits for)
            if constexpr (PAGED && !F8) {
                if (k_lo > base) clear_v(0, k_lo - base, BN);
            }
            __syncthreads();
            f32x16 s0[RB], s1[RB];
#pragma unroll
            for (int s = 0; s < KS; s += 2) read_rows(0, s);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                s0[rb] = zero;
#pragma unroll
                for (int s = 0; s < KS; s += 2)
#pragma unroll
                    for (int d = 0; d < 4 / EB; ++d)
                        s0[rb] = mfma32<DT>(k_operand(kop, s, d), qreg[rb][s * 2 / EB + d], s0[rb]);
            }
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                if constexpr (CAP) s0[e / 16][e % 16] = cap(s0[e / 16][e % 16]);
                visible(s0, e, 0);
                if (e % 16 == 0) peak[e / 16] = s0[e / 16][0];
                else peak[e / 16] = fmaxf(peak[e / 16], s0[e / 16][e % 16]);
            }
            raise(true);
            if constexpr (NH == 1) {
#pragma unroll
                for (int s = 0; s < KS; ++s) move_on(ra[s], TILE);
            }
            read_rows(NH > 1 ? 1 : 0, 0);
            int t = 0, nb = 1, fb = 3;  // buffers of tiles t + 1 and t + 3
            auto next_buf = [](int x) { return x == NBUF - 1 ? 0 : x + 1; };
            auto step_to = [](int x) { return x == 0 ? 0u - (NBUF - 1) * (unsigned)TILE : (unsigned)TILE; };
            auto ask = [&]() { load_tile(t + 3, fb, std::false_type{}); };  // into the buffer of tile t - 1
            constexpr int LAST = (2 * DB - 2) * RB;  // first product of the last operand pair: `ahead` runs there
            auto tile = [&](auto mask) {
                const unsigned by = step_to(nb);  // from tile t's buffer to the next
                const int s0k = t * BN;
                if constexpr (NH > 1) {
                    auto half = [&](auto hh) {  // the next unit's scores: half (h + 1) % NH, the one's after it (h + 2) % NH
                        constexpr int H = decltype(hh)::value;
                        unit(H % 2 ? s1 : s0, H % 2 ? s0 : s1, std::integral_constant<int, (H + 1) % NH>{}, hh,
                             s0k + 32 * (H + 1), mask,
                             [&](int x) {
                                 if (H == NH - 2 && x == SP / 2) {
#pragma unroll
                                     for (int s = 0; s < KS; ++s) move_on(ra[s], by);
                                 }
                                 if (H == NH - 2 && x == LAST - 1) {
                                     wait_loads<8>();
                                     __syncthreads();
                                 }
                                 if (H == NH - 1 && x == 0) ask();
                                 if (H == NH - 1 && x == LAST) {
#pragma unroll
                                     for (int db = 0; db < DB; ++db) {
                                         move_on(ta[db], by);
                                         move_on(tb[db], by);
                                     }
                                 }
                             },
                             [&]() { read_rows((H + 2) % NH, 0); });
                        if constexpr (H < NH - 1) raise(true);
                    };
                    half(std::integral_constant<int, 0>{});
                    half(std::integral_constant<int, 1>{});
                    if constexpr (NH == 4) {
                        half(std::integral_constant<int, 2>{});
                        half(std::integral_constant<int, 3>{});
                    }
                } else {
                    const unsigned by2 = step_to(next_buf(nb));  // from tile t + 1's buffer to the next
                    unit(s0, s1, H0{}, H0{}, s0k + 32, mask,
                         [&](int x) {
                             if (x == SP / 2) {
#pragma unroll
                                 for (int s = 0; s < KS; ++s) move_on(ra[s], by2);
                             }
                             if (x == LAST - 1) {
                                 wait_loads<0>();
                                 __syncthreads();
                             }
                             if (x == LAST) {
                                 ask();
#pragma unroll
                                 for (int db = 0; db < DB; ++db) {
                                     move_on(ta[db], by);
                                     move_on(tb[db], by);
                                 }
                             }
                         },
                         [&]() { read_rows(0, 0); });
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) s0[rb] = s1[rb];
                }
                nb = next_buf(nb);
                fb = next_buf(fb);
                ++t;
                raise(t < ntiles);
            };
            // a tile's mask covers the scores formed in it: those of its second
            // half and of the next tile's first
            for (int part = 0; part < 2; ++part) {
                const int tm = part == 0 ? t1 : ntiles;
                while (t < tm) {
                    if (__builtin_expect(t == part_tile, 0)) {
                        clear_v(nb == 0 ? NBUF - 1 : nb - 1, 0, last_end);
                        __syncthreads();
                    }
                    tile(std::true_type{});
                }
                while (t + 1 < t2) tile(std::false_type{});
            }
        }
        wait_loads<0>();
        __syncthreads();  // the next item's tiles go where other waves may still read

        // ---- epilogue: lane holds O^T [dims 32db + 8q + 4hi + i][row col] --------------------------
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int r = wrow0 + rb * 32 + col;
            const float lrow = l[rb] + __shfl_xor(l[rb], 32);
            const bool nonempty = lrow > 0.f;
            const float inv = nonempty ? (F8 ? sc_v / lrow : 1.f / lrow) : 0.f;
            const float lse = nonempty ? (m[rb] + fast_log2(lrow)) * kLn2 : (final_out ? INFINITY : -INFINITY);
            if (r >= bi.rows) continue;
            const int i = r / g, h = hk * g + r % g;
            if (final_out) {
                uint16_t* orow = a.cu_seqlens_q ? op + ((int64_t)a.cu_seqlens_q[b] + i) * a.o_si + (int64_t)h * a.o_sh
                                                : op + (int64_t)b * a.o_sb + (int64_t)i * a.o_si + (int64_t)h * a.o_sh;
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int d = 32 * db + 8 * q + 4 * hi;
                        if (d >= a.hd) continue;
                        const u32x2 x = {pack2<DT>(o[rb][db][4 * q] * inv, o[rb][db][4 * q + 1] * inv),
                                         pack2<DT>(o[rb][db][4 * q + 2] * inv, o[rb][db][4 * q + 3] * inv)};
                        *reinterpret_cast<u32x2*>(orow + d) = x;
                    }
                if (hi == 0) {
                    const int64_t off = a.cu_seqlens_q ? (int64_t)h * a.lse_sh + a.cu_seqlens_q[b] + i
                                                       : (int64_t)b * a.lse_sb + (int64_t)h * a.lse_sh + i;
                    a.lse[off] = lse;
                }
            } else {
                const int64_t prow = (int64_t)w * BM + (r - tile_row0);
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<f32x4*>(a.part_o + prow * HD + 32 * db + 8 * q + 4 * hi) =
                            f32x4{o[rb][db][4 * q] * inv, o[rb][db][4 * q + 1] * inv, o[rb][db][4 * q + 2] * inv,
                                  o[rb][db][4 * q + 3] * inv};
                if (hi == 0) a.part_lse[prow] = lse;
            }
        }
    }
}

template <int DT, int HD, int RB>
void launch_t(const FwdArgs& a, int grid, hipStream_t stream) {
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(NT), 0, stream, a); };
    if (a.softcap > 0.f) {
        if (a.block_table) go(fa_prefill_pipe_kernel<DT, HD, RB, true, false, true>);
        else go(fa_prefill_pipe_kernel<DT, HD, RB, false, false, true>);
    } else if constexpr (DT == DT_FP8) {
        if (a.block_table) go(fa_prefill_pipe_kernel<DT, HD, RB, true, false, false>);
        else go(fa_prefill_pipe_kernel<DT, HD, RB, false, false, false>);
    } else if (a.block_table) {
        if (a.rot_cos) go(fa_prefill_pipe_kernel<DT, HD, RB, true, true, false>);
        else go(fa_prefill_pipe_kernel<DT, HD, RB, true, false, false>);
    } else {
        if (a.rot_cos) go(fa_prefill_pipe_kernel<DT, HD, RB, false, true, false>);
        else go(fa_prefill_pipe_kernel<DT, HD, RB, false, false, false>);
    }
}

template <int HD, int RB>
void launch_d(const FwdArgs& a, int dtype, int grid, hipStream_t stream) {
    if (dtype == DT_BF16) launch_t<DT_BF16, HD, RB>(a, grid, stream);
    else launch_t<DT_FP16, HD, RB>(a, grid, stream);
}

}  // namespace pipe
}  // namespace fa
