// fa_bwd_kv.hip -- dK and dV of the plain backward at head dims 65..128 (no
// soft cap, ALiBi or attention chunk; query heads per kv head a power of two).
//
// One workgroup per (batch, kv head, 128-key block), four waves of 32 keys, one
// wave per SIMD. A wave keeps its keys' K and V (64 registers) and its dK and dV
// (128) and streams the packed (position, head) rows through LDS tiles of 64:
//   S = Q.K^T, dP = dO.V^T; P = exp(S - lse), dS = P (dP - dsum);
//   dV^T += dO^T.P, dK^T += Q^T.dS  (dO^T, Q^T by transpose reads of the tile)
// with 32x32x16 MFMA, whose result (one key, 16 rows per lane) is the packed
// operand of the last two.
//   * 32 keys to a wave instead of 16 halve the LDS reads per product, which
//     take the registers of a whole SIMD. With no second wave to fill in, the
//     wave overlaps by itself: the scores of half tile h + 1 are formed between
//     the vector work of half tile h and its dK / dV products, in slots of one
//     MFMA and a share of everything else (unit()).
//   * A wave issues one instruction in four cycles whatever its kind, so the
//     loop is counted in instructions: -lse / scale and -dsum enter the
//     accumulators as one product each with a row of ones (three bf16 terms
//     hold an fp32 value exactly), tiles go straight from memory to LDS two
//     tiles ahead, operand reads wait once per four products.
//   * Tile rows are 256 bytes with 16-byte chunk c of row r in slot
//     c ^ ((r & 3) << 2 | (r >> 2) & 3): conflict free for ds_read_b128 of 32
//     rows (about 200 bytes a cycle; 127 with c ^ (r & 15) and 16-row operands)
//     and for the transpose reads of 4 rows x 4 chunks.
// B4 S4096 H32/8 D128 causal bf16: 1463 -> 1079 us against the kernel of
// fa_bwd.hip (kernel trace), 0.75 -> 1.02 PFLOP/s of its four products; whole
// backward 2165 -> 1830 us. Its MFMAs alone (no vector work, LDS reads, loads)
// take 650 us at 1.8 GHz, the power limit; the clock is 1.9 GHz with all of it.
#include "fa_bwd.h"
#include "fa_pipe.h"

namespace fa {
namespace {

constexpr int D = 128, DCH = 16, NT = 256, BK = 128, BQ = 64;
constexpr int KS = D / 16;                 // 16-dim steps of S and dP
constexpr int DB = D / 32;                 // 32-dim blocks of dK and dV
constexpr int CPQ = BQ * DCH / NT;         // staged 16-byte chunks per thread of each tile
constexpr int QT = BQ * D;                 // elements per q (and dout) tile
constexpr int ST = BQ * 8;                 // elements per row constant (one 16-byte operand row each)
constexpr int RAW = BQ * 4;                // elements of the raw lse and dsum
constexpr int TILE = 2 * QT + 2 * ST + RAW;  // q, dout, -lse, -dsum, raw lse and dsum
constexpr int NBUF = 4;
constexpr int DMA = 2 * CPQ + 1;           // loads of a wave per tile

// v as the sum of three bf16 values (exact), the first three slots of an operand row
__device__ __forceinline__ u32x2 split3(float v) {
    const uint32_t h = f32_to_16<DT_BF16>(v);
    const float r1 = v - f16_to_32<DT_BF16>((uint16_t)h);
    const uint32_t m = f32_to_16<DT_BF16>(r1);
    const float r2 = r1 - f16_to_32<DT_BF16>((uint16_t)m);
    const uint32_t l = f32_to_16<DT_BF16>(r2);
    return u32x2{h | (m << 16), l};
}

// PART: the head dim is below 128 (see fa_bwd_dq.hip)
template <int DT, bool PART>
__global__ void __launch_bounds__(NT, 1) fa_bwd_kv_kernel(BwdArgs a) {
    __shared__ __attribute__((aligned(256))) uint16_t s_t[NBUF * TILE];
    __shared__ int s_pref[bw::kMaxBatch + 1], s_ord[kOrdered];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, hi = lane >> 5;
    if constexpr (PART) {  // q and dout chunks past the head dim are 0 and stay so, as K and V are there (barrier: in the prefix)
#pragma unroll
        for (int x = 0; x < NBUF; ++x)
            for (int at = tid * 16; at < 4 * QT; at += NT * 16)
                row_write(lds_addr(s_t) + x * 2 * TILE + at, u32x4{0u, 0u, 0u, 0u});
    }
    const int total = bw_ordered_prefix<NT>(a, s_pref, s_ord, [&](int b) {
        const BwBatch bb = bw_batch(a, b);
        return a.Hk * ((bb.sk + BK - 1) / BK);
    });
    const int gs = __builtin_ctz(a.g);  // g is a power of two, at most BQ
    const int g = a.g;
    const float sc = a.scale_log2;
    const float lscale = kLog2e / sc;

    const unsigned lds0 = lds_addr(s_t);
    // operand addresses within a tile: rows (chunk 2s + hi of row col) and
    // transposed (rows 4hi.., dims 32db + col), lo: rows +0..3, hi: +8..11
    const unsigned rowa = lds0 + col * (2 * D) + (swz(col, hi) << 4);  // chunk 2s + hi: ^ (s << 5)
    const int tr_r = 4 * hi + ((lane & 15) >> 2), tr_c = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    const unsigned tra = lds0 + tr_r * (2 * D) + (swz(tr_r, tr_c) << 4) + (lane & 1) * 8;  // dim block db: ^ (db << 6)
    const u32x4 ones = hi == 0 ? u32x4{0x3f803f80u, 0x00003f80u, 0u, 0u} : u32x4{0u, 0u, 0u, 0u};

    const char* qp = static_cast<const char*>(a.q);
    const uint16_t* kp = static_cast<const uint16_t*>(a.k);
    const uint16_t* vp = static_cast<const uint16_t*>(a.v);
    const char* dop = static_cast<const char*>(a.dout);

    for (int k = 0; k * (int)gridDim.x < total; ++k) {
        const int w = k * (int)gridDim.x + ((k & 1) ? (int)gridDim.x - 1 - (int)blockIdx.x : (int)blockIdx.x);
        if (w >= total) continue;
        const int place = bw_find_batch(s_pref, a.B, w);
        const int b = __builtin_amdgcn_readfirstlane(a.cu_seqlens_q && a.B <= kOrdered ? s_ord[place] : place);
        const BwBatch bb = bw_batch(a, b);
        const int local = w - __builtin_amdgcn_readfirstlane(s_pref[place]);
        const int hk = local % a.Hk;
        const int nkt = (bb.sk + BK - 1) / BK;
        const int kt = (a.wl >= 0 && a.wr < 0) ? nkt - 1 - local / a.Hk : local / a.Hk;
        const int j0 = kt * BK;
        const int diag0 = bb.sk - bb.sq;
        const int64_t q0 = a.cu_seqlens_q ? (int64_t)a.cu_seqlens_q[b] : 0;
        const int64_t k0 = a.cu_seqlens_k ? (int64_t)a.cu_seqlens_k[b] : 0;

        // rows that see some key of the block, [i_lo, i_hi]
        int i_lo = 0, i_hi = bb.sq - 1;
        if (a.wr >= 0) i_lo = max(0, j0 - diag0 - a.wr);
        if (a.wl >= 0) i_hi = min(bb.sq - 1, j0 + BK - 1 - diag0 + a.wl);
        const int r_lo = i_lo << gs;
        const int nrows = i_hi >= i_lo ? (i_hi + 1 - i_lo) << gs : 0;
        const int ntiles = (nrows + BQ - 1) / BQ;

        // the wave's 32 keys as B operands
        const int jw = j0 + 32 * wave, jl = jw + col;
        const bool key_ok = jl < bb.sk;
        u32x4 kreg[KS], vreg[KS];
        {
            const uint16_t* kr = kp + (a.cu_seqlens_k ? k0 * a.k_si : (int64_t)b * a.k_sb) + (int64_t)jl * a.k_si + (int64_t)hk * a.k_sh;
            const uint16_t* vr = vp + (a.cu_seqlens_k ? k0 * a.v_si : (int64_t)b * a.v_sb) + (int64_t)jl * a.v_si + (int64_t)hk * a.v_sh;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const int c = 2 * s + hi;
                const bool in = key_ok && c * 8 < a.hd;
                kreg[s] = in ? *reinterpret_cast<const u32x4*>(kr + c * 8) : u32x4{0u, 0u, 0u, 0u};
                vreg[s] = in ? *reinterpret_cast<const u32x4*>(vr + c * 8) : u32x4{0u, 0u, 0u, 0u};
            }
        }

        // staged rows: tile base (uniform) + this thread's byte offsets
        const char* qt = qp + 2 * ((a.cu_seqlens_q ? q0 * a.q_si : (int64_t)b * a.q_sb) + (int64_t)i_lo * a.q_si + (int64_t)hk * g * a.q_sh);
        const char* dt = dop + 2 * ((a.cu_seqlens_q ? q0 * a.do_si : (int64_t)b * a.do_sb) + (int64_t)i_lo * a.do_si + (int64_t)hk * g * a.do_sh);
        const int64_t q2 = 2 * a.q_si, d2 = 2 * a.do_si;
        // row constants: every thread loads one, waves 2 and 3 the same as 0 and 1
        const char* lt = (const char*)(((wave & 1) == 0 ? a.lse : (const float*)a.dsum) +
                                       (a.cu_seqlens_q ? q0 : (int64_t)b * a.lse_sb) + i_lo + (int64_t)hk * g * a.lse_sh);
        // Tile t holds rows row0(t) .. + 63 of the block's; the last one is moved
        // back to end at the last row, and the rows it repeats count for nothing
        // (store_stat), so no load needs a bound of its own (fewer than 64 rows:
        // the positions past the end load the last one).
        auto row0 = [&](int t) { return max(0, min(t * BQ, nrows - BQ)); };
        // The wave's share of a tile: load u brings rows 16 wave + 4u .. + 3, lane
        // l the 16 bytes of slot l % 16 of row l / 16 (the swizzle is in the
        // address read).
        unsigned qo[CPQ], dof[CPQ];
        [[maybe_unused]] uint64_t in_hd[CPQ];  // load u: lanes whose chunk lies in the head dim
#pragma unroll
        for (int u = 0; u < CPQ; ++u) {
            const int r = 16 * wave + 4 * u + (lane >> 4);
            const int c = swz(r, lane & 15);
            if constexpr (PART) in_hd[u] = __ballot(c < (a.hd >> 3));
            const int i = min(r >> gs, i_hi - i_lo), j = r & (g - 1);
            qo[u] = 2u * (unsigned)(i * (int)a.q_si + j * (int)a.q_sh + c * 8) + (3 - u) * 1024;
            dof[u] = 2u * (unsigned)(i * (int)a.do_si + j * (int)a.do_sh + c * 8) + (3 - u) * 1024;
        }
        const unsigned so = 4u * (unsigned)((lane & (g - 1)) * (int)a.lse_sh + min(lane >> gs, i_hi - i_lo));
        auto load_tile = [&](int t, int buf) {  // tiles past the end: the last one
            const int64_t i = row0(min(t, ntiles - 1)) >> gs;
            const unsigned base = lds0 + 2 * TILE * buf, wb = base + wave * 16 * 2 * D;
            if constexpr (PART) {
                dma16x4(wb, qt + i * q2 - 3072, qo, in_hd);
                dma16x4(wb + 2 * QT, dt + i * d2 - 3072, dof, in_hd);
            } else {
                dma16x4(wb, qt + i * q2 - 3072, qo);
                dma16x4(wb + 2 * QT, dt + i * d2 - 3072, dof);
            }
            dma4(base + 4 * QT + 4 * ST + (wave & 1) * RAW, lt + 4 * i, so);
        };
        // this wave's row constants of tile t, once its loads are there
        unsigned wsa = lds0 + 4 * QT + (tid & (2 * BQ - 1)) * 16, rsa = lds0 + 4 * QT + 4 * ST + (tid & (2 * BQ - 1)) * 4;
        float st = 0.f;
        const int is_lse = (wave & 1) ^ 1;
        const float smul = is_lse ? -lscale : -1.f;
        auto store_stat = [&](int t) {
            // rows of the tile before, rows past the end and rows without a visible key (lse = +inf): P = 0
            const int r = row0(t) + lane;
            const int drop = is_lse & ((r < t * BQ) | (r >= nrows) | (st >= 1e30f));
            const u32x2 x = split3(drop ? -1e30f : st * smul);
            row_write(wsa, u32x4{x[0], x[1], 0u, 0u});
        };

        f32x16 dv[DB], dk[DB];
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) dv[db][i] = dk[db][i] = 0.f;

        // visible rows of this lane's key, relative to r_lo: [vlo, vhi). In positions the
        // bounds are cut to the sequence first: a window past it has no 32-bit row.
        auto row_of = [&](int i) { return (min(max(i, 0), bb.sq) << gs) - r_lo; };
        const int vlo = a.wr >= 0 ? row_of(jl - diag0 - a.wr) : -0x40000000;
        const int vhi = a.wl >= 0 ? row_of(jl - diag0 + a.wl + 1) : 0x40000000;
        // tiles all of whose rows see all keys of the block: [t1, t2)
        const int flo = a.wr >= 0 ? row_of(j0 + BK - 1 - diag0 - a.wr) : 0;
        const int fhi = a.wl >= 0 ? row_of(j0 - diag0 + a.wl + 1) : nrows;
        const int t1 = min(ntiles, max(0, (flo + BQ - 1) / BQ));
        const int t2 = max(t1, a.wl >= 0 ? min(ntiles, max(0, fhi) / BQ) : ntiles);

        // LDS addresses of this lane's operands in the tile that they are read
        // from next, moved on with the tile; opaque, so that the rest goes into
        // the instructions' offsets
        unsigned ra[KS], ta[DB], tb[DB], sa = lds0 + 4 * QT + col * 16;
#pragma unroll
        for (int s = 0; s < KS; ++s) ra[s] = rowa ^ (s << 5);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            ta[db] = tra ^ (db << 6);
            tb[db] = (tra ^ (db << 6) ^ 32) + 8 * 2 * D;
        }
        auto move_on = [&](unsigned& x, unsigned by) {
            x += by;
            asm volatile("" : "+v"(x));
        };

        u32x4 aq[KS], ad[KS], al, adx;   // S / dP operands of the next half, in flight
        u32x4 xd[2 * DB], xq[2 * DB];    // dV / dK operands of the current half
        auto read_stat = [&](int h) {
            al = row_read(sa + h * 32 * 16);
            adx = row_read(sa + h * 32 * 16 + 2 * ST);
        };
        auto read_rows = [&](int h, int s) {  // steps s and s + 1
#pragma unroll
            for (int i = s; i < s + 2; ++i) {
                aq[i] = row_read(ra[i] + h * 32 * 2 * D);
                ad[i] = row_read(ra[i] + h * 32 * 2 * D + 2 * QT);
            }
        };
        auto read_tr = [&](int h, int x) {  // x, x + 1: step of 16 rows, then dim block
#pragma unroll
            for (int i = x; i < x + 2; ++i) {
                const int db = i % DB, o = (h * 32 + i / DB * 16) * 2 * D;
                xd[i] = tr_read(ta[db] + o + 2 * QT, tb[db] + o + 2 * QT);
                xq[i] = tr_read(ta[db] + o, tb[db] + o);
            }
        };

        // One half tile: dK / dV of the current half (scores in cs / cp) while
        // the scores of the next (ns / np) are formed, one MFMA to a slot. The
        // vector work of score e is spread over the slots from FIRST(e) on:
        // scaled in one, its exponential in the next, dS in the third.
        u32x4 pk[2], dsk[2];
        float px[16], de[16];
        auto score = [&](f32x16& cs, const f32x16& cp, int slot, int m0, auto mask) {
            auto at = [&](int e, int k) { return slot == e * 3 / 2 + k; };
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                if (at(e, 0)) px[e] = cs[e] * sc;
                if (at(e, 1)) px[e] = fast_exp2(px[e]);
                if (at(e, 2)) {
                    if constexpr (decltype(mask)::value) {
                        const int r = m0 + 8 * (e / 4) + e % 4;
                        px[e] = r >= vlo && r < vhi ? px[e] : 0.f;
                    }
                    de[e] = px[e] * cp[e];
                    if (e & 1) {
                        pk[e / 8][e / 2 % 4] = pack2<DT>(px[e - 1], px[e]);
                        dsk[e / 8][e / 2 % 4] = pack2<DT>(de[e - 1], de[e]);
                    }
                }
            }
        };
        const f32x16 zero = {};
        // A: half of the next scores within their tile; B: half of the current
        // rows within theirs; `more` issues the staging of its slot, `ahead` the
        // reads of the next unit's first operands
        auto unit = [&](f32x16& cs, f32x16& cp, f32x16& ns, f32x16& np, auto ha, auto hb, int m0, auto mask, auto more,
                        auto ahead) {
            constexpr int A = decltype(ha)::value, B = decltype(hb)::value;
            int slot = 0;
            auto next = [&]() {
                score(cs, cp, slot, m0, mask);
                ++slot;
                fence();
            };
            // Operands are read two steps at a time, a group ahead of their use,
            // and the last one read is the first one used: one wait per group.
            np = mfma32<DT_BF16>(adx, ones, zero);
            next();
            ns = mfma32<DT_BF16>(al, ones, zero);
            next();
#pragma unroll
            for (int s = 0; s < KS; s += 2) {
                np = mfma32<DT>(ad[s + 1], vreg[s + 1], np);
                if (s + 2 < KS) read_rows(A, s + 2);
                else read_tr(B, 0);
                next();
                ns = mfma32<DT>(aq[s + 1], kreg[s + 1], ns);
                next();
                np = mfma32<DT>(ad[s], vreg[s], np);
                next();
                ns = mfma32<DT>(aq[s], kreg[s], ns);
                next();
            }
#pragma unroll
            for (int x = 0; x < 2 * DB; x += 2) {
                dk[(x + 1) % DB] = mfma32<DT>(xq[x + 1], dsk[x / DB], dk[(x + 1) % DB]);
                if (x + 2 < 2 * DB) read_tr(B, x + 2);
                else ahead();
                next();
                dv[(x + 1) % DB] = mfma32<DT>(xd[x + 1], pk[x / DB], dv[(x + 1) % DB]);
                more(2 * x);
                next();
                dk[x % DB] = mfma32<DT>(xq[x], dsk[x / DB], dk[x % DB]);
                more(2 * x + 1);
                next();
                dv[x % DB] = mfma32<DT>(xd[x], pk[x / DB], dv[x % DB]);
                more(2 * x + 2);
                next();
            }
        };

        if (ntiles > 0) {
            using H0 = std::integral_constant<int, 0>;
            using H1 = std::integral_constant<int, 1>;
            load_tile(0, 0);
            load_tile(1, 1);
            load_tile(2, 2);
            wait_loads<2 * DMA>();
            st = float_read(rsa);
            store_stat(0);
            __syncthreads();
            f32x16 s0, p0, s1, p1;
            read_stat(0);
#pragma unroll
            for (int s = 0; s < KS; s += 2) read_rows(0, s);
            s0 = mfma32<DT_BF16>(al, ones, zero);
            p0 = mfma32<DT_BF16>(adx, ones, zero);
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                s0 = mfma32<DT>(aq[s], kreg[s], s0);
                p0 = mfma32<DT>(ad[s], vreg[s], p0);
            }
            read_stat(1);
            read_rows(1, 0);
            // Tile t: its first half while the scores of its second are formed and
            // tile t + 1 arrives; then its second half while the scores of the next
            // tile are formed and tile t + 3 is asked for, into the buffer of tile
            // t - 1, which no wave reads after the barrier in between.
            int t = 0, nb = 1, fb = 3;  // buffers of tiles t + 1 and t + 3
            auto tile = [&](auto mask) {
                const int m0 = row0(t) + 4 * hi;
                const unsigned by = nb == 0 ? 0u - 2u * (NBUF - 1) * TILE : 2u * TILE;  // from tile t's buffer to it
                unit(s0, p0, s1, p1, H1{}, H0{}, m0, mask,
                     [&](int k) {
                         if (k == 0) {
                             wait_loads<DMA>();
                             move_on(rsa, by);
                             st = float_read(rsa);
                         }
                         if (k == 2) {
                             move_on(wsa, by);
                             store_stat(t + 1);
                         }
                         if (k == 6) {
                             move_on(sa, by);
#pragma unroll
                             for (int s = 0; s < KS; ++s) move_on(ra[s], by);
                         }
                         if (k == 4 * DB - 6) __syncthreads();
                     },
                     [&]() {
                         read_stat(0);
                         read_rows(0, 0);
                     });
                unit(s1, p1, s0, p0, H0{}, H1{}, m0 + 32, mask,
                     [&](int k) {
                         if (k == 0) load_tile(t + 3, fb);
                         if (k == 4 * DB - 6) {
#pragma unroll
                             for (int db = 0; db < DB; ++db) {
                                 move_on(ta[db], by);
                                 move_on(tb[db], by);
                             }
                         }
                     },
                     [&]() {
                         read_stat(1);
                         read_rows(1, 0);
                     });
                nb = nb == NBUF - 1 ? 0 : nb + 1;
                fb = fb == NBUF - 1 ? 0 : fb + 1;
                ++t;
            };
            for (int part = 0; part < 2; ++part) {
                const int tm = part == 0 ? t1 : ntiles;
                while (t < tm) tile(std::true_type{});
                while (t < t2) tile(std::false_type{});
            }
        }

        // lane holds dK^T / dV^T [dims 32db + 8q + 4hi + i][key jl]
        if (key_ok) {
            uint16_t* dkp = static_cast<uint16_t*>(a.dk) + (a.cu_seqlens_k ? k0 * a.dk_si : (int64_t)b * a.dk_sb) +
                            (int64_t)jl * a.dk_si + (int64_t)hk * a.dk_sh;
            uint16_t* dvp = static_cast<uint16_t*>(a.dv) + (a.cu_seqlens_k ? k0 * a.dv_si : (int64_t)b * a.dv_sb) +
                            (int64_t)jl * a.dv_si + (int64_t)hk * a.dv_sh;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int d = 32 * db + 8 * q + 4 * hi;
                    if (d >= a.hd) continue;
                    uint16_t k4[4], v4[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        k4[i] = f32_to_16<DT>(dk[db][4 * q + i] * a.scale);
                        v4[i] = f32_to_16<DT>(dv[db][4 * q + i]);
                    }
                    *reinterpret_cast<u32x2*>(dkp + d) = __builtin_bit_cast(u32x2, k4);
                    *reinterpret_cast<u32x2*>(dvp + d) = __builtin_bit_cast(u32x2, v4);
                }
        }
        wait_loads<0>();
        __syncthreads();  // the next item's tiles go where other waves may still read
    }
}

}  // namespace

// Which calls can run here; the others keep the kernel of fa_bwd.hip.
// The rows of a tile are BQ / g positions of all g heads, so g divides BQ; their
// byte offsets within a tile are 32-bit; -lse / scale stays in range.
bool bwd_kv_takes(const BwdArgs& a) {
    auto fits = [&](int64_t si, int64_t sh) {
        return si >= 0 && sh >= 0 && si < (1 << 23) && sh < (1 << 29) / a.g && si * (BQ / a.g) < (1 << 28);
    };
    return a.chunk == 0 && a.g <= BQ && (a.g & (a.g - 1)) == 0 && a.scale >= 1e-6f && fits(a.q_si, a.q_sh) &&
           fits(a.do_si, a.do_sh) && a.lse_sh < (1 << 28) / a.g;
}

void launch_bwd_kv(const BwdArgs& a, int dtype, int grid, hipStream_t stream) {
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(NT), 0, stream, a); };
    const bool part = a.hd < D;
    if (dtype == DT_BF16) part ? go(fa_bwd_kv_kernel<DT_BF16, true>) : go(fa_bwd_kv_kernel<DT_BF16, false>);
    else part ? go(fa_bwd_kv_kernel<DT_FP16, true>) : go(fa_bwd_kv_kernel<DT_FP16, false>);
}

}  // namespace fa
