"""Attention calls of few tiles, where two or four wavefronts share a tile's list and merge."""

import numpy as np
import pytest
import torch

from block_attn import block_sparse_attn, block_sparse_attn_v2
from oracle import attention as OA
from parity import f32np

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
MAX_ABS, MEAN_ABS = 2e-2, 2e-3      # the bar of the attention tests


def qkv(seed, B, H, Hk, M, D, dtype):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(B, h, M, D, generator=g).to(dtype) for h in (H, Hk, Hk))


def check(out, ref):
    err = np.abs(f32np(out) - ref)
    assert err.max() <= MAX_ABS and err.mean() <= MEAN_ABS, (err.max(), err.mean())


# (H, M) with one, two and four wavefronts per tile at every head_dim that has them, for lists as
# wide as the context and for row masks (test_layer_route_cpu.py asks the library which each takes)
LISTS = [(4, 190), (4, 1150), (20, 1101), (40, 1150), (56, 1101)]
ROWS = [(4, 190), (4, 1150), (28, 1101), (56, 1101)]


# lists from none to every visible block, so runs of no, one and several blocks, and one list in
# slot order (repeats)
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (64, torch.float16),
                                     (128, torch.bfloat16), (128, torch.float16),
                                     (256, torch.bfloat16), (256, torch.float16)])
@pytest.mark.parametrize("H,M", LISTS)
def test_tile_lists(hip_lib, D, dtype, H, M):
    print(f"[case] split lists D={D} {dtype} H={H} M={M}", flush=True)
    q, k, v = qkv(H + M + D, 1, H, H // 2, M, D, dtype)
    nb = qt = (M + 63) // 64
    g = torch.Generator().manual_seed(M)
    kv = torch.full((1, H, qt, nb), nb, dtype=torch.int32)
    for h in range(H):
        for t in range(qt):
            n = (h + t) % (t + 2)                       # 0 .. t + 1 blocks
            pick = torch.randperm(t + 1, generator=g)[:n].to(torch.int32)
            at = torch.randperm(nb, generator=g)[:n]    # sentinels between them
            kv[0, h, t, at] = pick
    if nb >= 5:
        kv[0, 1, 4] = nb
        kv[0, 1, 4, :5] = torch.tensor([3, 0, 3, 4, 0], dtype=torch.int32)
    out = torch.full((1, H, M, D), float("nan"), dtype=dtype, device=DEV)
    block_sparse_attn_v2(q.to(DEV), k.to(DEV), v.to(DEV), kv.to(DEV), D ** -0.5, out=out)
    ref = OA.gathered_attention(f32np(q), f32np(k), f32np(v), kv.numpy(), D ** -0.5)
    check(out, ref)
    for h in range(min(H, 4)):
        for t in range(qt):
            if (h + t) % (t + 2) == 0 and (h, t) != (1, 4):
                assert (out[0, h, 64 * t:64 * t + 64] == 0).all()


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("H,M", ROWS)
def test_row_masks(hip_lib, D, H, M):
    print(f"[case] split row masks D={D} H={H} M={M}", flush=True)
    q, k, v = qkv(H + M + D, 1, H, H // 2, M, D, torch.bfloat16)
    nb = (M + 63) // 64
    g = torch.Generator().manual_seed(M)
    rows = torch.arange(M)
    keep = torch.rand(1, H, M, nb, generator=g) < 0.4
    keep[0, :, rows, rows // 64] = True
    out = block_sparse_attn(q.to(DEV), k.to(DEV), v.to(DEV), keep.to(DEV), D ** -0.5)
    keep &= torch.arange(nb) <= (rows // 64)[:, None]
    check(out, OA.keep_attention(f32np(q), f32np(k), f32np(v), keep.numpy(), D ** -0.5))


@pytest.mark.parametrize("D", [64, 128, 256])
def test_offsets_far_apart(hip_lib, D):
    """Runs whose row maxima differ by hundreds of log2 units merge without overflow."""
    H, M = 4, 1150
    q, k, v = qkv(7, 1, H, H, M, D, torch.bfloat16)
    k[:, :, 640:704] *= 40.0
    nb = qt = (M + 63) // 64
    kv = torch.full((1, H, qt, nb), nb, dtype=torch.int32)
    for t in range(qt):
        kv[0, :, t, :t + 1] = torch.arange(t + 1, dtype=torch.int32)
    out = block_sparse_attn_v2(q.to(DEV), k.to(DEV), v.to(DEV), kv.to(DEV), D ** -0.5)
    check(out, OA.gathered_attention(f32np(q), f32np(k), f32np(v), kv.numpy(), D ** -0.5))


# past 512 blocks, where only head_dim 64 splits: lists of none to 40 blocks, a ragged last tile
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H", [1, 2])
def test_long_context_of_few_tiles(hip_lib, D, H):
    print(f"[case] split lists past 512 blocks D={D} H={H}", flush=True)
    M = 64 * 530 - 9
    q, k, v = qkv(M + D + H, 1, H, 1, M, D, torch.bfloat16)
    nb = qt = 530
    g = torch.Generator().manual_seed(H)
    kv = torch.full((1, H, qt, 40), nb, dtype=torch.int32)
    for h in range(H):
        for t in range(qt):
            n = min((h + t) % 41, t + 1)
            kv[0, h, t, torch.randperm(40, generator=g)[:n]] = torch.randperm(t + 1, generator=g)[:n].to(torch.int32)
    ref = OA.gathered_attention(f32np(q), f32np(k), f32np(v), kv.numpy(), D ** -0.5)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    check(block_sparse_attn_v2(qd, kd, vd, kv.to(DEV), D ** -0.5), ref)
    # the same lists as row masks that every row of a tile shares
    keep = torch.zeros(1, H, qt, nb + 1, dtype=torch.bool).scatter_(3, kv.long(), True)[..., :nb]
    keep = keep.repeat_interleave(64, dim=2)[:, :, :M].contiguous()
    check(block_sparse_attn(qd, kd, vd, keep.to(DEV), D ** -0.5), ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kept", [1500, 1600])
def test_long_row_lists(hip_lib, dtype, kept):
    """Head_dim 64, row-masked lists on either side of the length (1575 slots) where another form
    of the kernel takes over; the tiles that hold them and some others against fp32."""
    print(f"[case] long row lists {dtype} kept={kept}", flush=True)
    nb, D = 1610, 64
    M = 64 * nb - 30
    q, k, v = (t.to(DEV) for t in qkv(kept, 1, 2, 1, M, D, dtype))
    g = torch.Generator(device=DEV).manual_seed(kept)
    tile = torch.arange(M, device=DEV) // 64
    keep = torch.rand(1, 2, M, nb, device=DEV, generator=g) < 0.004
    keep[0, :, torch.arange(M, device=DEV), tile] = True
    full = (1605, nb - 1)                                   # whole and ragged tiles with long lists
    for t in full:
        rows = slice(64 * t, min(M, 64 * t + 64))
        keep[0, :, rows, :kept - 1] |= torch.rand(M, device=DEV, generator=g)[rows, None] < 0.7
        keep[0, :, rows, kept - 1:t] = False
    keep = keep & (torch.arange(nb, device=DEV) <= tile[:, None])
    out = block_sparse_attn(q, k, v, keep, D ** -0.5).float()
    for h in range(2):
        for t in (0, 1, 700, 1604) + full:
            rows = slice(64 * t, min(M, 64 * t + 64))
            s = (q[0, h, rows].float() @ k[0, 0].float().t().contiguous()) * D ** -0.5
            on = keep[0, h, rows].repeat_interleave(64, dim=1)[:, :M]
            on = on & (torch.arange(M, device=DEV) <= torch.arange(M, device=DEV)[rows, None])
            want = torch.softmax(s.masked_fill(~on, float("-inf")), -1) @ v[0, 0].float()
            check(out[0, h, rows], f32np(want))


@pytest.mark.parametrize("slots", [4600, 4800])
def test_long_plain_lists(hip_lib, slots):
    """Head_dim 64, lists on either side of the length (4700 slots) where that form takes over, their
    blocks anywhere among the sentinels."""
    print(f"[case] long plain lists slots={slots}", flush=True)
    M, D = 64 * 40 - 7, 64
    q, k, v = qkv(slots, 1, 2, 1, M, D, torch.bfloat16)
    g = torch.Generator().manual_seed(slots)
    short = torch.full((1, 2, 40, 40), 40, dtype=torch.int32)
    kv = torch.full((1, 2, 40, slots), 40, dtype=torch.int32)
    for h in range(2):
        for t in range(40):
            pick = torch.randperm(t + 1, generator=g)[:(7 * t + h) % (t + 2)].to(torch.int32)
            short[0, h, t, :len(pick)] = pick
            kv[0, h, t, torch.randperm(slots, generator=g)[:len(pick)]] = pick
    out = block_sparse_attn_v2(q.to(DEV), k.to(DEV), v.to(DEV), kv.to(DEV), D ** -0.5)
    check(out, OA.gathered_attention(f32np(q), f32np(k), f32np(v), short.numpy(), D ** -0.5))


@pytest.mark.parametrize("D", [64, 128, 256])
def test_tile_order_of_row_masks(hip_lib, D):
    """Tiles ranked by their work or by descending index: the same bits, lists that do not grow."""
    H, M = 40, 64 * 60 - 11                             # 2400 tiles, more than start at once
    q, k, v = (t.to(DEV) for t in qkv(D, 1, H, 4, M, D, torch.bfloat16))
    tile, nbs = torch.arange(M, device=DEV) // 64, torch.arange(60, device=DEV)
    keep = (tile[:, None] == nbs) | ((tile % 8 == 1)[:, None] & (nbs <= tile[:, None]))
    keep = keep.expand(1, H, M, 60).contiguous()
    ranked = block_sparse_attn(q, k, v, keep, D ** -0.5)
    assert torch.equal(ranked, block_sparse_attn(q, k, v, keep, D ** -0.5, lists_grow=True))
    check(ranked[:, :1], OA.keep_attention(f32np(q[:, :1]), f32np(k[:, :1]), f32np(v[:, :1]),
                                           keep[:, :1].cpu().numpy(), D ** -0.5))


def test_row_masks_in_a_graph(hip_lib):
    """A context whose lists are worth asking the device for their longest is captured without."""
    M, D = 64 * 700, 256
    q, k, v = (t.to(DEV) for t in qkv(9, 1, 2, 1, M, D, torch.bfloat16))
    tile, nbs = torch.arange(M, device=DEV) // 64, torch.arange(700, device=DEV)
    keep = ((tile[:, None] == nbs) | (nbs == 0)).expand(1, 2, M, 700).contiguous()
    eager = block_sparse_attn(q, k, v, keep, D ** -0.5)
    out, graph = torch.empty_like(q), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        block_sparse_attn(q, k, v, keep, D ** -0.5, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert torch.equal(block_sparse_attn(q, k, v, keep, D ** -0.5), eager)
