"""GPU parity of the dK/dV kernel of the plain backward at head dims 65..128
(64-row tiles in four LDS buffers, 128-key blocks) where its tiling can go
wrong: fewer rows than a tile, one row more or less than whole tiles and
blocks, few and many tiles, every group size it takes and one it does not,
windows that hide rows at either end, head dims below 128, rows with no
visible key, ragged batches and transposed layouts. Reference and bar are
those of test_gpu_bwd.py."""
import numpy as np
import pytest
import torch

from tests.test_gpu_bwd import check, rand_inputs, run_dense, run_varlen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sq,sk", [(1, 1), (3, 130), (16, 127), (17, 128), (63, 129), (64, 64), (65, 257), (129, 31),
                                   (256, 256), (333, 300)])
@pytest.mark.parametrize("h,hk", [(4, 4), (8, 2)])
@pytest.mark.parametrize("causal", [False, True])
def test_tile_edges(sq, sk, h, hk, causal):
    run_dense(torch.bfloat16, 2, h, hk, sq, sk, 128, causal, seed=sq * 1000 + sk)


@pytest.mark.parametrize("g", [1, 2, 3, 8, 16, 64])
def test_group_sizes(g):
    run_dense(torch.bfloat16, 1, 2 * g, 2, 45, 70, 128, True, seed=g)


@pytest.mark.parametrize("window", [(5, 0), (40, 9), (-1, 20), (70, -1), (0, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_windows(window, dtype):
    run_dense(dtype, 1, 4, 1, 200, 210, 128, False, window=window, seed=7)


@pytest.mark.parametrize("sides", [(1, None), (1, 0), (None, 1), (1, 1)], ids=["left", "left_causal", "right", "both"])
@pytest.mark.parametrize("g", [1, 2, 4, 8, 64])
@pytest.mark.parametrize("w", [1 << 25, 1 << 28, 10**9, 1 << 30, (1 << 31) - 1])
def test_windows_past_the_sequence(w, g, sides):
    """A window wider than the sequence hides nothing: the results of an
    unbounded one bit for bit, also where the bound times the query heads per kv
    head, or plus a position, is past 32 bits."""
    import flash_attn_npu_v2
    gen = torch.Generator().manual_seed(g)
    for sq, sk in ((150, 150), (40, 200), (200, 40)):
        q, do = (rand_inputs((1, sq, g, 128), torch.bfloat16, gen).cuda() for _ in range(2))
        k, v = (rand_inputs((1, sk, 1, 128), torch.bfloat16, gen).cuda() for _ in range(2))

        def run(window):
            print(f"case wide window {window} g{g} {sq}x{sk}", flush=True)
            parts = [x.detach().requires_grad_(True) for x in (q, k, v)]
            out, lse, _ = flash_attn_npu_v2.flash_attn_func(*parts, window_size=window, return_attn_probs=True)
            return (out, lse) + torch.autograd.grad(out, parts, do)

        want = run(tuple(0 if x == 0 else -1 for x in sides))
        got = run(tuple(-1 if x is None else x * w for x in sides))
        for name, x, ref in zip(("out", "lse", "dq", "dk", "dv"), got, want):
            assert torch.equal(x, ref), name


@pytest.mark.parametrize("d", [72, 96, 120])
def test_head_dims(d):
    run_dense(torch.float16, 2, 4, 2, 150, 140, d, True, seed=d, api="v3")


@pytest.mark.parametrize("causal", [False, True])
def test_ragged(causal):
    run_varlen(torch.bfloat16, 8, 2, [1, 200, 64, 0, 129, 17], [130, 200, 1, 40, 128, 5], 128, causal, seed=3)


def test_layouts():
    """Heads outside positions and a packed qkv: the same gradients, bit for bit, as contiguous copies."""
    import flash_attn_npu_v2
    g = torch.Generator().manual_seed(5)
    qkv = rand_inputs((2, 100, 3, 4, 128), torch.bfloat16, g).cuda()
    do = rand_inputs((2, 100, 4, 128), torch.bfloat16, g).cuda()
    outer = [x.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for x in qkv.unbind(2)]

    def grads(parts, dout):
        parts = [x.detach().requires_grad_(True) for x in parts]
        return torch.autograd.grad(flash_attn_npu_v2.flash_attn_func(*parts, causal=True), parts, dout)

    want = grads([x.contiguous() for x in qkv.unbind(2)], do)
    for parts, dout in ((outer, do.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3)), (qkv.unbind(2), do)):
        for got, w, p in zip(grads(parts, dout), want, parts):
            assert torch.equal(got, w)
            assert got.stride() == torch.empty_like(p).stride()


@pytest.mark.parametrize("sq,sk", [(1, 33), (127, 64), (129, 257), (300, 31)])
@pytest.mark.parametrize("d", [40, 64, 128, 160, 256])
@pytest.mark.parametrize("softcap", [0.0, 20.0])
def test_dq_tiles(sq, sk, d, softcap):
    """The dQ kernel's 128-row items and 32- to 128-key tiles at every head dim, plain and with a soft cap."""
    run_dense(torch.bfloat16, 1, 6, 2, sq, sk, d, True, softcap=softcap, seed=sq + d)


@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("window", [(40, 9), (-1, 20), (70, -1)])
def test_dq_windows(d, window):
    run_dense(torch.float16, 1, 4, 1, 200, 210, d, False, window=window, softcap=15.0, seed=8)
    run_varlen(torch.bfloat16, 8, 2, [1, 200, 64, 0, 129], [130, 200, 1, 40, 128], d, False, window=window, seed=4)


@pytest.mark.parametrize("where", ["q", "k", "v", "do"])
@pytest.mark.parametrize("d", [40, 72, 96, 120, 160])
def test_infinity_below_the_kernel_head_dim(d, where):
    """An infinity in the last dims of a row goes where it goes in the same
    tensors with zeros up to the kernel's head dim (NaN for NaN), and no further:
    what the kernels hold past the head dim is 0. The other tensors are
    positive there, so that a key of -inf has weight 0 and its rows stay finite."""
    import flash_attn_npu_v2
    full = 64 if d <= 64 else 128 if d <= 128 else 256
    g = torch.Generator().manual_seed(d)
    x = {n: rand_inputs((1, 150, 2 if n in ("q", "do") else 1, d), torch.bfloat16, g) for n in ("q", "k", "v", "do")}
    for t in x.values():
        t[..., d - 3] = t[..., d - 3].abs() + 0.5
    x[where][0, 70, 0, d - 3] = -float("inf")
    print(f"case infinity in {where} d{d}", flush=True)

    def grads(width):
        q, k, v, do = (torch.nn.functional.pad(t, (0, width - d)).cuda() for t in x.values())
        parts = [t.requires_grad_(True) for t in (q, k, v)]
        out = flash_attn_npu_v2.flash_attn_func(*parts, softmax_scale=d ** -0.5, causal=True)
        return [t.detach()[..., :d].float().cpu() for t in (out, *torch.autograd.grad(out, parts, do))]

    for name, got, want in zip(("out", "dq", "dk", "dv"), grads(d), grads(full)):
        same = (got == want) | (got.isnan() & want.isnan())
        assert bool(same.all()), f"{name}: {int((~same).sum())} elements differ, {int(got.isnan().sum())} NaN, {int(want.isnan().sum())} wanted"
