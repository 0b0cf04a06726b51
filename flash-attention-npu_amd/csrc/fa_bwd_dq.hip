// fa_bwd_dq.hip -- dQ and dsum of the backward with one wave per SIMD (no ALiBi
// or attention chunk).
//
// The loop of the pipelined prefill (fa_fwd_pipe.h) with 32 rows per wave, whose
// q and dout stay in registers: S^T = K.Q^T and dP^T = V.dO^T of the next 32 keys
// are formed while dS = P (dP - dsum) of the current ones is, then
// dQ^T += K^T.dS^T (K^T by transpose reads). 64 rows per wave would halve the LDS
// reads, but their q, dout, dQ and two sets of scores do not fit 512 registers at
// head dim 128 (nor compile well at 64).
// Whole backward, same box (dK/dV changed as well at head dim 128), us: head dim
// 128 B4 S4096 H32/8 causal 2138 -> 1782, soft-capped B2 1705 -> 1431; head dim 256
// B2 S4096 H16/8, window and soft cap 1419 -> 996; head dim 64 B8 S1025 H16 fp16
// 244 -> 229 (bound by the softmax gradient's vector work).
#include "fa_bwd.h"
#include "fa_pipe.h"

namespace fa {
namespace {

constexpr int NT = 256, NBUF = 4;

// Slot of chunk c in row r (128-byte rows: from the row pair)
template <int HD>
__device__ __forceinline__ int slot_of(int r, int c) {
    return HD == 64 ? c ^ ((((r >> 1) & 1) << 2) | ((r >> 2) & 3)) : swz(r, c);
}

template <int HD>
struct DqCfg {
    static constexpr int RB = 1;                   // 32-row blocks per wave
    static constexpr int BM = 4 * RB * 32;
    static constexpr int NH = 256 / HD;           // 32-key halves per LDS tile
    static constexpr int BN = 32 * NH;
    static constexpr int KS = HD / 16, DB = HD / 32, CH = HD / 8, RPL = 64 / CH;
    static constexpr int ROW = 2 * HD, KT = BN * ROW, TILE = 2 * KT;
};

// PART: the head dim is below HD. A template argument: the masks of its loads
// cost the others 1-2 % (B2 S4096 D256 with window and cap 1176 -> 1203 us).
template <int DT, int HD, bool CAP, bool PART>
__global__ void __launch_bounds__(NT, 1) fa_bwd_dq_pipe_kernel(BwdArgs a) {
    using C = DqCfg<HD>;
    constexpr int RB = C::RB, BM = C::BM, BN = C::BN, NH = C::NH, KS = C::KS, DB = C::DB, CH = C::CH, ROW = C::ROW,
                  KT = C::KT, TILE = C::TILE, NE = 16 * RB;
    constexpr int SS = 2 * KS * RB, SP = DB * RB;  // slots: S and dP products, then dQ's of the first and the last 16 keys
    static_assert(KT == 4 * 4 * 1024, "four loads of four waves bring a tile");
    __shared__ __attribute__((aligned(256))) char s_t[NBUF * TILE];
    __shared__ int s_pref[bw::kMaxBatch + 1], s_ord[kOrdered];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hi = lane >> 5;
    if constexpr (PART) {  // chunks past the head dim are 0 and stay so, as in the prefill (barrier: in the prefix)
#pragma unroll
        for (int x = 0; x < NBUF; ++x)
            for (int at = tid * 16; at < TILE; at += NT * 16) row_write(lds_addr(s_t) + x * TILE + at, u32x4{0u, 0u, 0u, 0u});
    }
    const int total = bw_ordered_prefix<NT>(a, s_pref, s_ord, [&](int b) {
        const BwBatch bb = bw_batch(a, b);
        return a.Hk * ((bb.rows + BM - 1) / BM);
    });

    const unsigned lds0 = lds_addr(s_t);
    const unsigned rowa = lds0 + col * ROW + (slot_of<HD>(col, hi) << 4);  // chunk 2s + hi: ^ (s << 5)
    const int tr_r = 4 * hi + ((lane & 15) >> 2), tr_c = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    const unsigned tra = lds0 + tr_r * ROW + (slot_of<HD>(tr_r, tr_c) << 4) + (lane & 1) * 8;  // dim block db: ^ (db << 6)

    const uint16_t* qp = static_cast<const uint16_t*>(a.q);
    const uint16_t* dop = static_cast<const uint16_t*>(a.dout);
    const uint16_t* outp = static_cast<const uint16_t*>(a.out);
    const float sc = a.scale_log2;
    // cap * tanh(scale s / cap) in log2 units = c1 t, t = 1 - 2 / (2^(c0 s) + 1)
    [[maybe_unused]] const float c0 = CAP ? 2.f * a.scale_log2 / a.softcap : 0.f, c1 = a.softcap * kLog2e;

    // pass k takes item k * grid + blockIdx.x, the other way round on odd
    // passes (a heavy item of one pass pairs with a light one of the next)
    for (int k = 0; k * (int)gridDim.x < total; ++k) {
        const int w = k * (int)gridDim.x + ((k & 1) ? (int)gridDim.x - 1 - (int)blockIdx.x : (int)blockIdx.x);
        if (w >= total) continue;
        const int place = bw_find_batch(s_pref, a.B, w);
        const int b = __builtin_amdgcn_readfirstlane(a.cu_seqlens_q && a.B <= kOrdered ? s_ord[place] : place);
        const BwBatch bb = bw_batch(a, b);
        const int local = w - __builtin_amdgcn_readfirstlane(s_pref[place]);
        const int hk = local % a.Hk;
        // heavy first: with a right window bound (causal) later row tiles see more keys
        const int nmt = (bb.rows + BM - 1) / BM;
        const int mt = a.wr >= 0 ? nmt - 1 - local / a.Hk : local / a.Hk;
        const int g = a.g;
        const int diag0 = bb.sk - bb.sq;
        const int tile_row0 = mt * BM, tile_rows = min(BM, bb.rows - tile_row0);
        const int i_lo = tile_row0 / g, i_hi = (tile_row0 + tile_rows - 1) / g;
        const int k_lo = max(0, key_lo(i_lo + diag0, a.wl, 0));
        const int k_hi = max(k_lo, min(bb.sk, key_hi(i_hi + diag0, a.wr, 0) + 1));
        const int ntiles = (k_hi - k_lo + BN - 1) / BN;
        // tiles all of whose keys are visible to all rows: [t1, t2)
        const int f_lo = max(k_lo, key_lo(i_hi + diag0, a.wl, 0)), f_hi = min(k_hi, key_hi(i_lo + diag0, a.wr, 0) + 1);
        const int t1 = min(ntiles, (f_lo - k_lo + BN - 1) / BN), t2 = max(t1, (f_hi - k_lo) / BN);
        const int64_t q0 = a.cu_seqlens_q ? (int64_t)a.cu_seqlens_q[b] : 0;
        const int64_t k0 = (a.cu_seqlens_k ? (int64_t)a.cu_seqlens_k[b] : 0) + k_lo;

        // ---- K / V tiles straight into LDS (as in the prefill, fa_fwd_pipe.h) -----------------
        const char* kb = static_cast<const char*>(a.k) + 2 * ((a.cu_seqlens_k ? 0 : (int64_t)b * a.k_sb) + k0 * a.k_si + (int64_t)hk * a.k_sh);
        const char* vb = static_cast<const char*>(a.v) + 2 * ((a.cu_seqlens_k ? 0 : (int64_t)b * a.v_sb) + k0 * a.v_si + (int64_t)hk * a.v_sh);
        unsigned ko[2][4], vo[2][4];
        [[maybe_unused]] uint64_t in_hd[4];  // load u: lanes whose chunk lies in the head dim
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int r = C::RPL * (4 * wave + u) + lane / CH;
            const int c = slot_of<HD>(r, lane % CH);
            if constexpr (PART) in_hd[u] = __ballot(c < (a.hd >> 3));
            const int rl = min(r, k_hi - 1 - k_lo - (ntiles - 1) * BN);   // the last tile's rows past the last key load it
            ko[0][u] = 2u * (unsigned)(r * (int)a.k_si + c * 8) + (3 - u) * 1024;
            vo[0][u] = 2u * (unsigned)(r * (int)a.v_si + c * 8) + (3 - u) * 1024;
            ko[1][u] = 2u * (unsigned)(rl * (int)a.k_si + c * 8) + (3 - u) * 1024;
            vo[1][u] = 2u * (unsigned)(rl * (int)a.v_si + c * 8) + (3 - u) * 1024;
        }
        auto load_tile = [&](int t, int buf) {  // tiles past the end: the last one
            const bool last = t >= ntiles - 1;
            const int64_t j = (int64_t)min(t, ntiles - 1) * BN;
            unsigned k4[4], v4[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                k4[u] = last ? ko[1][u] : ko[0][u];
                v4[u] = last ? vo[1][u] : vo[0][u];
            }
            const unsigned wb = lds0 + TILE * buf + wave * 4096;
            if constexpr (PART) {
                dma16x4(wb, kb + 2 * j * a.k_si - 3072, k4, in_hd);
                dma16x4(wb + KT, vb + 2 * j * a.v_si - 3072, v4, in_hd);
            } else {
                dma16x4(wb, kb + 2 * j * a.k_si - 3072, k4);
                dma16x4(wb + KT, vb + 2 * j * a.v_si - 3072, v4);
            }
        };
        if (ntiles > 0) {
            load_tile(0, 0);
            load_tile(1, 1);
            load_tile(2, 2);
        }

        // ---- q and dout as B operands, dsum = rowsum(dout * out) --------------------------------
        u32x4 qreg[RB][KS], dreg[RB][KS];
        float lse2[RB], dsv[RB];
        int rlo[RB], rhi[RB];  // the row's visible keys, as offsets from k_lo
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int r = tile_row0 + (wave * RB + rb) * 32 + col;
            const bool ok = r < bb.rows;
            const int i = ok ? r / g : 0, h = hk * g + (ok ? r % g : 0);
            rlo[rb] = max(k_lo, key_lo(i + diag0, a.wl, 0)) - k_lo - 4 * hi;
            rhi[rb] = min(k_hi - 1, key_hi(i + diag0, a.wr, 0)) - k_lo - 4 * hi;
            const int64_t lo = a.cu_seqlens_q ? (int64_t)h * a.lse_sh + q0 + i
                                              : (int64_t)b * a.lse_sb + (int64_t)h * a.lse_sh + i;
            lse2[rb] = ok ? a.lse[lo] * kLog2e : INFINITY;
            const uint16_t* qrow = qp + (a.cu_seqlens_q ? q0 * a.q_si : (int64_t)b * a.q_sb) + (int64_t)i * a.q_si + (int64_t)h * a.q_sh;
            const uint16_t* drow = dop + (a.cu_seqlens_q ? q0 * a.do_si : (int64_t)b * a.do_sb) + (int64_t)i * a.do_si + (int64_t)h * a.do_sh;
            const uint16_t* orow = outp + (a.cu_seqlens_q ? q0 * a.o_si : (int64_t)b * a.o_sb) + (int64_t)i * a.o_si + (int64_t)h * a.o_sh;
            float acc = 0.f;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int c = 2 * s + hi;
                const bool in = ok && c * 8 < a.hd;
                qreg[rb][s] = in ? *reinterpret_cast<const u32x4*>(qrow + c * 8) : u32x4{0u, 0u, 0u, 0u};
                dreg[rb][s] = in ? *reinterpret_cast<const u32x4*>(drow + c * 8) : u32x4{0u, 0u, 0u, 0u};
                const u32x4 x = in ? *reinterpret_cast<const u32x4*>(orow + c * 8) : u32x4{0u, 0u, 0u, 0u};
                uint16_t oh[8], dh[8];
                __builtin_memcpy(oh, &x, 16);
                __builtin_memcpy(dh, &dreg[rb][s], 16);
#pragma unroll
                for (int e = 0; e < 8; ++e) acc += f16_to_32<DT>(oh[e]) * f16_to_32<DT>(dh[e]);
            }
            acc += __shfl_xor(acc, 32);
            dsv[rb] = ok ? acc : 0.f;
            if (hi == 0 && ok) a.dsum[lo] = acc;
        }
        // in accumulation registers, one tuple per operand
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int s = 0; s < KS; ++s) asm volatile("" : "+a"(qreg[rb][s]), "+a"(dreg[rb][s]));

        f32x16 dq[RB][DB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) dq[rb][db][i] = 0.f;

        // LDS addresses of this lane's operands in the tile read next, moved on
        // with the tile; opaque, so that the rest goes into the instructions' offsets
        unsigned ra[KS], ta[DB], tb[DB];
#pragma unroll
        for (int s = 0; s < KS; ++s) ra[s] = rowa ^ (s << 5);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            ta[db] = tra ^ (db << 6);
            tb[db] = (tra ^ (db << 6) ^ 32) + 8 * ROW;
        }
        auto move_on = [&](unsigned& x, unsigned by) {
            x += by;
            asm volatile("" : "+v"(x));
        };
        u32x4 kop[KS], vop[KS], top[2 * DB];
        auto read_rows = [&](int h, int s) {  // steps s and s + 1
#pragma unroll
            for (int i = s; i < s + 2; ++i) {
                kop[i] = row_read(ra[i] + h * 32 * ROW);
                vop[i] = row_read(ra[i] + h * 32 * ROW + KT);
            }
        };
        auto read_tr = [&](int h, int x) {  // x, x + 1: step of 16 keys, then dim block
#pragma unroll
            for (int i = x; i < x + 2; ++i) {
                const int o = (h * 32 + i / DB * 16) * ROW;
                top[i] = tr_read(ta[i % DB] + o, tb[i % DB] + o);
            }
        };

        const f32x16 zero = {};
        u32x4 dsk[RB][2];
        float px[NE], dx[NE];
        [[maybe_unused]] float tx[NE];
        // One half tile: its softmax gradient and dQ products while the scores and
        // dP of the next are formed (n_, np_), one MFMA to a slot.
        auto unit = [&](f32x16 (&c_)[RB], f32x16 (&cp_)[RB], f32x16 (&n_)[RB], f32x16 (&np_)[RB], auto ha, auto hb, int s0,
                        auto mask, auto more, auto ahead) {
            constexpr int A = decltype(ha)::value, B = decltype(hb)::value;
            int slot = 0;
            auto next = [&]() {
#pragma unroll
                for (int q = 0; q < NE; ++q) {
                    // q-th score: the first 16 keys of every row block, then the others
                    const int ks = q / (8 * RB), rb = q / 8 % RB, i = 8 * ks + q % 8;
                    constexpr int ST = CAP ? 5 : 3;  // slots from first to last
                    const int at = q * (SS + SP - ST + 1) / NE;
                    if constexpr (CAP) {
                        if (slot == at) tx[q] = fast_exp2(c_[rb][i] * c0);
                        if (slot == at + 1) tx[q] = __builtin_amdgcn_rcpf(tx[q] + 1.f);
                        if (slot == at + 2) {
                            tx[q] = __builtin_fmaf(-2.f, tx[q], 1.f);
                            px[q] = __builtin_fmaf(tx[q], c1, -lse2[rb]);
                        }
                    } else {
                        if (slot == at) px[q] = __builtin_fmaf(c_[rb][i], sc, -lse2[rb]);
                    }
                    if (slot == at + ST - 2) {
                        px[q] = fast_exp2(px[q]);
                        dx[q] = cp_[rb][i] - dsv[rb];
                        if constexpr (CAP) dx[q] *= __builtin_fmaf(-tx[q], tx[q], 1.f);
                    }
                    if (slot == at + ST - 1) {
                        if constexpr (decltype(mask)::value) {
                            const int j = s0 + 8 * (i / 4) + i % 4;
                            px[q] = j >= rlo[rb] && j <= rhi[rb] ? px[q] : 0.f;
                        }
                        dx[q] *= px[q];
                        if (q & 1) dsk[rb][ks][q / 2 % 4] = pack2<DT>(dx[q - 1], dx[q]);
                    }
                }
                ++slot;
                fence();
            };
            // operands are read two steps ahead, the last one read is used first
#pragma unroll
            for (int s = 0; s < KS; s += 2) {
#pragma unroll
                for (int d = 1; d >= 0; --d)
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) {
                        np_[rb] = mfma32<DT>(vop[s + d], dreg[rb][s + d], s == 0 && d == 1 ? zero : np_[rb]);
                        if (d == 1 && rb == 0) {
                            if (s + 2 < KS) read_rows(A, s + 2);
                            else read_tr(B, 0);
                        }
                        next();
                        n_[rb] = mfma32<DT>(kop[s + d], qreg[rb][s + d], s == 0 && d == 1 ? zero : n_[rb]);
                        next();
                    }
            }
#pragma unroll
            for (int x = 0; x < 2 * DB; x += 2) {
#pragma unroll
                for (int d = 1; d >= 0; --d)
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) {
                        dq[rb][(x + d) % DB] = mfma32<DT>(top[x + d], dsk[rb][(x + d) / DB], dq[rb][(x + d) % DB]);
                        if (d == 1 && rb == 0) {
                            if (x + 2 < 2 * DB) read_tr(B, x + 2);
                            else ahead();
                        }
                        more(x * RB + (1 - d) * RB + rb);
                        next();
                    }
            }
        };

        if (ntiles > 0) {
            using H0 = std::integral_constant<int, 0>;
            wait_loads<0>();
            __syncthreads();
            f32x16 s0[RB], p0[RB], s1[RB], p1[RB];
#pragma unroll
            for (int s = 0; s < KS; s += 2) read_rows(0, s);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                s0[rb] = p0[rb] = zero;
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    s0[rb] = mfma32<DT>(kop[s], qreg[rb][s], s0[rb]);
                    p0[rb] = mfma32<DT>(vop[s], dreg[rb][s], p0[rb]);
                }
            }
            if constexpr (NH == 1) {
#pragma unroll
                for (int s = 0; s < KS; ++s) move_on(ra[s], TILE);
            }
            read_rows(NH > 1 ? 1 : 0, 0);
            int t = 0, nb = 1, fb = 3;  // buffers of tiles t + 1 and t + 3
            auto next_buf = [](int x) { return x == NBUF - 1 ? 0 : x + 1; };
            auto step_to = [](int x) { return x == 0 ? 0u - (NBUF - 1) * (unsigned)TILE : (unsigned)TILE; };
            auto ask = [&]() { load_tile(t + 3, fb); };  // into the buffer of tile t - 1
            constexpr int LAST = (2 * DB - 2) * RB;  // first product of the last operand pair: `ahead` runs there
            auto tile = [&](auto mask) {
                const unsigned by = step_to(nb);  // from tile t's buffer to the next
                const int s0k = t * BN;
                if constexpr (NH > 1) {
                    auto half = [&](auto hh) {
                        constexpr int H = decltype(hh)::value;
                        unit(H % 2 ? s1 : s0, H % 2 ? p1 : p0, H % 2 ? s0 : s1, H % 2 ? p0 : p1,
                             std::integral_constant<int, (H + 1) % NH>{}, hh, s0k + 32 * H, mask,
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
                    };
                    half(std::integral_constant<int, 0>{});
                    half(std::integral_constant<int, 1>{});
                    if constexpr (NH == 4) {
                        half(std::integral_constant<int, 2>{});
                        half(std::integral_constant<int, 3>{});
                    }
                } else {
                    const unsigned by2 = step_to(next_buf(nb));  // from tile t + 1's buffer to the next
                    unit(s0, p0, s1, p1, H0{}, H0{}, s0k, mask,
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
                    for (int rb = 0; rb < RB; ++rb) {
                        s0[rb] = s1[rb];
                        p0[rb] = p1[rb];
                    }
                }
                nb = next_buf(nb);
                fb = next_buf(fb);
                ++t;
            };
            for (int part = 0; part < 2; ++part) {
                const int tm = part == 0 ? t1 : ntiles;
                while (t < tm) tile(std::true_type{});
                while (t < t2) tile(std::false_type{});
            }
        }
        wait_loads<0>();
        __syncthreads();  // the next item's tiles go where other waves may still read

        // lane holds dQ^T [dims 32db + 8q + 4hi + i][row col]
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int r = tile_row0 + (wave * RB + rb) * 32 + col;
            if (r >= bb.rows) continue;
            const int i = r / g, h = hk * g + r % g;
            uint16_t* row = static_cast<uint16_t*>(a.dq) + (a.cu_seqlens_q ? q0 * a.dq_si : (int64_t)b * a.dq_sb) +
                            (int64_t)i * a.dq_si + (int64_t)h * a.dq_sh;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int d = 32 * db + 8 * q + 4 * hi;
                    if (d >= a.hd) continue;
                    const u32x2 x = {pack2<DT>(dq[rb][db][4 * q] * a.scale, dq[rb][db][4 * q + 1] * a.scale),
                                     pack2<DT>(dq[rb][db][4 * q + 2] * a.scale, dq[rb][db][4 * q + 3] * a.scale)};
                    *reinterpret_cast<u32x2*>(row + d) = x;
                }
        }
    }
}

template <int DT, int HD>
void launch_t(const BwdArgs& a, int grid, hipStream_t stream) {
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(NT), 0, stream, a); };
    const bool part = a.hd < HD;
    if (a.softcap > 0.f) part ? go(fa_bwd_dq_pipe_kernel<DT, HD, true, true>) : go(fa_bwd_dq_pipe_kernel<DT, HD, true, false>);
    else part ? go(fa_bwd_dq_pipe_kernel<DT, HD, false, true>) : go(fa_bwd_dq_pipe_kernel<DT, HD, false, false>);
}

template <int DT>
void launch_d(const BwdArgs& a, int d, int grid, hipStream_t stream) {
    if (d == 64) launch_t<DT, 64>(a, grid, stream);
    else if (d == 128) launch_t<DT, 128>(a, grid, stream);
    else launch_t<DT, 256>(a, grid, stream);
}

}  // namespace

// Which calls can run here; the others keep the kernel of fa_bwd.hip. The rows of a
// tile (16 KB) have 32-bit byte offsets.
bool bwd_dq_takes(const BwdArgs& a) {
    auto fits = [](int64_t si) { return si >= 0 && si < (1 << 22); };
    return a.chunk == 0 && !a.alibi && a.scale > 0.f && fits(a.k_si) && fits(a.v_si);
}

void launch_bwd_dq(const BwdArgs& a, int dtype, int d, int grid, hipStream_t stream) {
    if (dtype == DT_BF16) launch_d<DT_BF16>(a, d, grid, stream);
    else launch_d<DT_FP16>(a, d, grid, stream);
}

}  // namespace fa
