"""GPU parity of the pipelined prefill kernel where its tiling can go wrong:
row tiles of 128 and 256 and key tiles of 64 met, missed by one and undershot,
row blocks of the last wave empty, every window edge inside and between tiles,
paged caches at the smallest page it takes and one it does not, splits of the
keys (whole and forced) and none, ragged batches, head dims below 128, scores
that move the running maximum late. Reference and bar are those of the forward
oracle tests."""
import numpy as np
import pytest
import torch

from oracle import fa_oracle as orc
from tests._util import assert_close_lse, assert_close_out, bits, odt

pytestmark = pytest.mark.gpu
NT = 16


def inputs(seed, dtype, *shapes, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return [(torch.randn(s, generator=g) * scale).to(dtype) for s in shapes]


def dense(dtype, B, H, Hk, Sq, Sk, D, causal=False, window=(-1, -1), softcap=0.0, seed=0, grow=False):
    import flash_attn_npu_v2
    print(f"case pipe dense {dtype} B{B} H{H}/{Hk} {Sq}x{Sk} D{D} causal={causal} window={window} softcap={softcap}", flush=True)
    q, k, v = inputs(seed, dtype, (B, Sq, H, D), (B, Sk, Hk, D), (B, Sk, Hk, D))
    if grow:  # later keys score higher, so the running maximum moves again and again
        k = (k.float() * torch.linspace(0.1, 6.0, Sk)[None, :, None, None]).to(dtype)
    out, lse, _ = flash_attn_npu_v2.flash_attn_func(q.cuda(), k.cuda(), v.cuda(), causal=causal, window_size=window,
                                                    softcap=softcap, return_attn_probs=True)
    ro, rl = orc.attention(bits(q), bits(k), bits(v), dtype=odt(dtype), scale=D ** -0.5, softcap=softcap, causal=causal,
                           window=window, nthreads=NT)
    assert_close_out(out, ro, dtype)
    assert_close_lse(lse, rl)


@pytest.mark.parametrize("sq,sk", [(1, 1), (5, 64), (31, 65), (128, 63), (129, 129), (257, 128), (300, 1000), (64, 1025)])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("causal", [False, True])
def test_tile_edges(sq, sk, d, causal):
    dense(torch.bfloat16, 2, 6, 2, sq, sk, d, causal, seed=sq + sk)


@pytest.mark.parametrize("b,sq", [(1, 700), (24, 600)])  # row tiles of the small and of the large kind
@pytest.mark.parametrize("d", [40, 72, 96, 160])
def test_head_dims(b, sq, d):
    dense(torch.float16, b, 4, 4, sq, 130, d, seed=d)


@pytest.mark.parametrize("d", [40, 64, 72, 120, 128, 160])
def test_infinite_key(d):
    """A key of -inf in the last dimension, against positive q: weight 0, nothing else touched."""
    import flash_attn_npu_v2
    print(f"case pipe -inf key D{d}", flush=True)
    q, k, v = inputs(d, torch.bfloat16, (2, 150, 4, d), (2, 200, 2, d), (2, 200, 2, d))
    q[..., -1] = 1.0
    k[:, 77, :, -1] = -float("inf")
    out, lse, _ = flash_attn_npu_v2.flash_attn_func(q.cuda(), k.cuda(), v.cuda(), return_attn_probs=True)
    keep = [j for j in range(200) if j != 77]
    ro, rl = orc.attention(bits(q), bits(k[:, keep].contiguous()), bits(v[:, keep].contiguous()), dtype=odt(torch.bfloat16),
                           scale=d ** -0.5, nthreads=NT)
    assert_close_out(out, ro, torch.bfloat16)
    assert_close_lse(lse, rl)


@pytest.mark.parametrize("window", [(0, 0), (63, 0), (64, 3), (100, -1), (-1, 70)])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_windows(window, d):
    dense(torch.float16, 1, 4, 2, 260, 300, d, window=window, seed=9)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_rising_scores(d, softcap):
    dense(torch.bfloat16, 1, 2, 2, 200, 700, d, causal=True, softcap=softcap, seed=4, grow=True)


def kvcache(dtype, B, H, Hk, Sq, lens, D, page, num_splits=0, window=(-1, -1), rotary=False, seed=0):
    import flash_attn_npu_v2
    print(f"case pipe kvcache {dtype} B{B} H{H}/{Hk} Sq{Sq} lens={lens} D{D} page={page} splits={num_splits}", flush=True)
    g = torch.Generator().manual_seed(seed)
    sl = torch.tensor(lens, dtype=torch.int32)
    new = Sq if rotary else 0
    cap = max(lens) + new
    bt = None
    if page:
        nb = -(-cap // page)
        bt = torch.randperm(B * nb + 2, generator=g)[:B * nb].view(B, nb).to(torch.int32)
        kv = (B * nb + 2, page, Hk, D)
    else:
        kv = (B, cap, Hk, D)
    q, kc, vc, kn, vn = inputs(seed, dtype, (B, Sq, H, D), kv, kv, (B, Sq, Hk, D), (B, Sq, Hk, D))
    more, ref = {}, {}
    if rotary:
        ang = torch.arange(cap)[:, None] * 10000.0 ** (-torch.arange(0, D, 2) / D)
        cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
        more = dict(k=kn.cuda(), v=vn.cuda(), rotary_cos=cos.cuda(), rotary_sin=sin.cuda(), rotary_interleaved=False)
        ref = dict(k=bits(kn), v=bits(vn), rotary_cos=bits(cos), rotary_sin=bits(sin), rotary_interleaved=False)
    kd, vd = kc.cuda(), vc.cuda()
    out, lse = flash_attn_npu_v2.flash_attn_with_kvcache(
        q.cuda(), kd, vd, cache_seqlens=sl.cuda(), block_table=None if bt is None else bt.cuda(), causal=True,
        window_size=window, num_splits=num_splits, return_softmax_lse=True, **more)
    ro, rl, rk, _ = orc.kvcache_forward(bits(q), bits(kc), bits(vc), dtype=odt(dtype), cache_seqlens=sl.numpy(),
                                        block_table=None if bt is None else bt.numpy(), causal=True, window=window, **ref)
    assert_close_out(out, ro, dtype)
    assert_close_lse(lse, rl)
    assert np.array_equal(bits(kd), rk)


@pytest.mark.parametrize("page", [0, 16, 64, 192])
@pytest.mark.parametrize("num_splits", [0, 1, 3])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_split_and_paged(page, num_splits, d):
    kvcache(torch.bfloat16, 2, 8, 2, 70, [1500, 333], d, page, num_splits, seed=page + num_splits)


@pytest.mark.parametrize("page", [0, 64])
def test_paged_window(page):
    kvcache(torch.bfloat16, 1, 8, 2, 90, [900], 128, page, window=(130, 0), seed=1)


@pytest.mark.parametrize("page", [0, 128])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_rotary(page, d):
    kvcache(torch.bfloat16, 2, 8, 2, 100, [37, 250], d, page, rotary=True, seed=2)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_ragged(causal, d):
    import flash_attn_npu_v3
    lens = [1, 300, 0, 64, 129, 700]
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    q, k, v = inputs(3, torch.bfloat16, (cu[-1], 4, d), (cu[-1], 2, d), (cu[-1], 2, d))
    c = torch.from_numpy(cu).cuda()
    out, lse = flash_attn_npu_v3.flash_attn_varlen_func(q.cuda(), k.cuda(), v.cuda(), c, c, 700, 700, causal=causal,
                                                        return_attn_probs=True)
    ro, rl = orc.attention(bits(q), bits(k), bits(v), dtype=orc.BF16, scale=d ** -0.5, causal=causal, cu_seqlens_q=cu,
                           cu_seqlens_k=cu, max_seqlen_q=700, nthreads=NT)
    assert_close_out(out, ro, torch.bfloat16)
    assert_close_lse(lse, rl)


@pytest.mark.parametrize("b,sq,sk", [(1, 17, 40), (1, 128, 128), (2, 257, 129), (3, 300, 1100), (16, 520, 513)])
@pytest.mark.parametrize("d", [80, 128])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_fp8(b, sq, sk, d, softcap):
    """e4m3 inputs with descales of either sign and zero, row tiles of both kinds."""
    import flash_attn_npu_v3
    print(f"case pipe fp8 B{b} {sq}x{sk} D{d} softcap={softcap}", flush=True)
    f8 = torch.float8_e4m3fn
    q, k, v = inputs(sq, torch.bfloat16, (b, sq, 8, d), (b, sk, 2, d), (b, sk, 2, d))
    q, k, v = q.to(f8), k.to(f8), v.to(f8)
    g = torch.Generator().manual_seed(1)
    qd, kd, vd = (0.5 + torch.rand((b, 2), generator=g) for _ in range(3))
    qd[0, 0], kd[b - 1, 1] = -1.25, 0.0
    out, lse = flash_attn_npu_v3.flash_attn_func(q.cuda(), k.cuda(), v.cuda(), causal=True, softcap=softcap,
                                                 q_descale=qd.cuda(), k_descale=kd.cuda(), v_descale=vd.cuda(),
                                                 return_attn_probs=True)
    by = lambda x: x.view(torch.uint8).numpy()
    ro, rl = orc.attention_fp8(by(q), by(k), by(v), scale=d ** -0.5, q_descale=qd.numpy(), k_descale=kd.numpy(),
                               v_descale=vd.numpy(), causal=True, softcap=softcap, nthreads=NT)
    err = (out.float().cpu() - torch.from_numpy(ro)).abs()
    # 1e-2 + one bf16 ulp of the reference, as for bf16 inputs (outputs here reach v_descale x 4)
    assert bool((err <= 1e-2 + 2.0 ** -7 * torch.from_numpy(ro).abs()).all()), float(err.max())
    assert_close_lse(lse, rl)


@pytest.mark.parametrize("page", [0, 64, 128, 256])
def test_fp8_kvcache(page):
    """A cache of e4m3 rows, paged where a tile lies in one page and where it does not, and a split of the keys."""
    import flash_attn_npu_v3
    f8 = torch.float8_e4m3fn
    B, Sq, Hk, D, lens = 2, 70, 2, 128, [1500, 333]
    q, k, v = inputs(page, torch.bfloat16, (B, Sq, 8, D), (B, 1536, Hk, D), (B, 1536, Hk, D))
    q, k, v = q.to(f8), k.to(f8), v.to(f8)
    by = lambda x: x.view(torch.uint8).numpy()
    ro, rl = orc.attention_fp8(by(q), by(k), by(v), scale=D ** -0.5, causal=True, nthreads=NT,
                               seqlens_k=np.array(lens, np.int32))
    more = {}
    kc, vc = k.cuda(), v.cuda()
    if page:
        n = 1536 // page
        more["page_table"] = torch.arange(B * n, dtype=torch.int32).view(B, n).cuda()
        kc, vc = (x.reshape(B * n, page, Hk, D) for x in (kc, vc))
    for ns in (0, 3):
        out, lse, _, _ = flash_attn_npu_v3.flash_attn_with_kvcache(
            q.cuda(), kc, vc, cache_seqlens=torch.tensor(lens, dtype=torch.int32).cuda(), causal=True, num_splits=ns,
            return_softmax_lse=True, **more)
        err = (out.float().cpu() - torch.from_numpy(ro)).abs()
        assert bool((err <= 1e-2 + 2.0 ** -7 * torch.from_numpy(ro).abs()).all()), float(err.max())
        assert_close_lse(lse, rl)


@pytest.mark.parametrize("sq", [1, 4, 70])
@pytest.mark.parametrize("page", [0, 64])
def test_window_past_the_cache(sq, page):
    """The widest windows there are hide nothing, in decode and prefill: the bounds are added to positions in 32 bits."""
    import flash_attn_npu_v2
    q, k, v = (x.cuda() for x in inputs(sq, torch.bfloat16, (2, sq, 8, 128), (2, 256, 2, 128), (2, 256, 2, 128)))
    more = dict(cache_seqlens=torch.tensor([201, 33], dtype=torch.int32).cuda(), return_softmax_lse=True)
    if page:
        k, v = (x.reshape(-1, page, 2, 128) for x in (k, v))
        more["block_table"] = torch.arange(512 // page, dtype=torch.int32).view(2, -1).cuda()
    big = (1 << 31) - 1
    for window, same in (((big, big), (-1, -1)), ((-1, big), (-1, -1)), ((big, 0), (-1, 0))):
        print(f"case window {window} sq{sq} page{page}", flush=True)
        got, want = (flash_attn_npu_v2.flash_attn_with_kvcache(q, k, v, window_size=w, **more) for w in (window, same))
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("d", [64, 96, 128, 256])
@pytest.mark.parametrize("page", [0, 64])
def test_infinity_in_v(d, page):
    """An infinity in V of the first or the last key that the rows see stays that infinity: the rows of a tile that
    are no keys of the call are 0, not that key again (0 times infinity)."""
    import flash_attn_npu_v2
    q, k, v = inputs(d, torch.bfloat16, (1, 1, 36, d), (1, 256, 2, d), (1, 256, 2, d))
    seen, left = 150, 129  # one position, keys 20 .. 149
    v[0, seen - 1, :, 3] = float("inf")
    v[0, seen - 1 - left, :, 5] = -float("inf")
    kd, vd = k.cuda(), v.cuda()
    more = {}
    if page:
        kd, vd = (x.reshape(-1, page, 2, d) for x in (kd, vd))
        more["block_table"] = torch.arange(256 // page, dtype=torch.int32).view(1, -1).cuda()
    print(f"case infinity in v d{d} page{page}", flush=True)
    out = flash_attn_npu_v2.flash_attn_with_kvcache(
        q.cuda(), kd, vd, cache_seqlens=torch.tensor([seen], dtype=torch.int32).cuda(), window_size=(left, 0),
        causal=True, num_splits=1, **more).float().cpu()
    assert bool((out[..., 3] == float("inf")).all()) and bool((out[..., 5] == -float("inf")).all())
    assert bool(out[..., [i for i in range(d) if i not in (3, 5)]].isfinite().all())
