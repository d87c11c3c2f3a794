"""Per-row selection at the edges of its register layouts (1, 2, 4, .. blocks per lane), with ties,
NaN scores and margins at other ranks than the budget, against the oracle on the kernel's scores;
the lists and row masks made of keep masks, and the cached block means."""

import numpy as np
import pytest
import torch

import _capi
import sparse_attention as sa
from block_attn import keep_kv_idx
from oracle import attention as OA
from test_gpu_select_v1 import check_on_kernel_scores, make_sel

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def check(mode, kw, q, k):
    sel = make_sel(mode=mode, **kw)
    res = sa.select_mask_v1(q.to(DEV), k.to(DEV), q.shape[-1] ** -0.5, sel=sel, want_scores=True)
    check_on_kernel_scores(res, sel, k.shape[2])


# blocks at and around one, two and four per lane and 8-, 4-, 2- and 1-byte keep stores; budgets
# below, at and above the visible blocks; k_min 8 makes the kept rank differ from the margin's
@pytest.mark.parametrize("nb", [2, 9, 63, 64, 65, 66, 100, 128, 129, 260])
@pytest.mark.parametrize("mode,kw", [("topk", dict(budget_blocks=16)),
                                     ("router", dict(budget_blocks=4, router_mode="quantile")),
                                     ("router", dict(budget_blocks=40, router_grain="row")),
                                     ("belief", dict(top_p=0.6, k_min=1)),
                                     ("belief", dict(top_p=0.99, k_min=100, k_max=200))])
def test_keep_and_margin(hip_lib, nb, mode, kw):
    print(f"[case] rows nb={nb} {mode} {kw}", flush=True)
    S = 64 * nb - (nb * 7) % 64
    g = torch.Generator().manual_seed(nb)
    q = torch.randn(1, 2, S, 64, generator=g).to(torch.bfloat16)
    k = (0.2 * torch.randn(1, 1, S, 64, generator=g)).to(torch.bfloat16)
    check(mode, kw, q, k)


# a mass that is never reached: every row keeps the k_max best ranks, rows of fewer visible blocks
# than that too (their total is 1 within 1e-6, so no row sits near either top_p)
@pytest.mark.parametrize("nb,k_max", [(66, 66), (157, 112), (157, 64), (300, 200)])
@pytest.mark.parametrize("top_p", [1.00002, 1.5])
def test_belief_mass_never_reached(hip_lib, nb, k_max, top_p):
    print(f"[case] belief nb={nb} k_max={k_max} top_p={top_p}", flush=True)
    g = torch.Generator().manual_seed(nb)
    q = torch.randn(1, 2, 64 * nb, 64, generator=g).to(torch.bfloat16)
    k = (0.2 * torch.randn(1, 1, 64 * nb, 64, generator=g)).to(torch.bfloat16)
    sel = make_sel(mode="belief", top_p=top_p, k_min=1, k_max=k_max)
    res = sa.select_mask_v1(q.to(DEV), k.to(DEV), 0.125, sel=sel, want_scores=True)
    check_on_kernel_scores(res, sel, 64 * nb)
    assert res.keep[0, 0, 0].sum() == k_max        # one visible block, the rest lowest first


# the sort sizes (64, 128, 256, 512 keys) on either side of each, rows of fewer blocks among them
@pytest.mark.parametrize("k_max", [64, 65, 128, 129, 256, 257, 400])
def test_belief_sort_sizes(hip_lib, k_max):
    print(f"[case] belief sort k_max={k_max}", flush=True)
    g = torch.Generator().manual_seed(k_max)
    q = torch.randn(1, 1, 64 * 300, 64, generator=g).to(torch.bfloat16)
    k = (0.2 * torch.randn(1, 1, 64 * 300, 64, generator=g)).to(torch.bfloat16)
    check("belief", dict(top_p=0.8, k_min=1, k_max=k_max), q, k)


@pytest.mark.parametrize("nb", [40, 100, 300])
@pytest.mark.parametrize("mode,kw", [("topk", dict(budget_blocks=16)),
                                     ("router", dict(budget_blocks=24))])
def test_ties(hip_lib, nb, mode, kw):
    """Blocks of a few distinct means: most rows cut inside a run of equal scores."""
    g = torch.Generator().manual_seed(nb)
    base = torch.randn(5, 64, generator=g)
    k = base[torch.randint(0, 5, (nb,), generator=g)].repeat_interleave(64, 0)[None, None]
    q = torch.randn(1, 2, 64 * nb, 64, generator=g).to(torch.bfloat16)
    check(mode, kw, q, k.to(torch.bfloat16))
    check(mode, kw, torch.zeros_like(q), k.to(torch.bfloat16))     # all scores equal


def test_nan_and_infinite_scores(hip_lib):
    """NaN ranks above every score and infinities where they belong, as in the total order."""
    nb = 90
    g = torch.Generator().manual_seed(1)
    q = torch.randn(1, 2, 64 * nb, 64, generator=g).to(torch.bfloat16)
    k = torch.randn(1, 1, 64 * nb, 64, generator=g).to(torch.bfloat16)
    for blk, value in ((3, float("nan")), (7, float("inf")), (11, float("-inf"))):
        k[0, 0, 64 * blk, 5] = value
    for mode, kw in (("quest", dict(budget_blocks=16)),
                     ("router", dict(budget_blocks=12, router_score="quest"))):
        check(mode, kw, q, k)


# 1-, 4- and 8-byte words, one block, part of a 64-block step, one and several 1024-block sections
@pytest.mark.parametrize("nb", [1, 5, 64, 100, 132, 256, 260, 1024, 1025, 1032, 2056])
@pytest.mark.parametrize("block_m", [64, 32])
def test_keep_lists(hip_lib, nb, block_m):
    print(f"[case] keep lists nb={nb} block_m={block_m}", flush=True)
    g = torch.Generator().manual_seed(nb)
    M = 150                                             # a ragged last tile
    keep = torch.rand(2, 3, M, nb, generator=g) < 0.02
    keep[0, 1, 64:128] = False                          # a tile that keeps nothing
    want, want_max = OA.compute_kv_idx(keep.numpy(), block_m)
    odd = torch.empty(keep.numel() + 1, dtype=torch.bool, device=DEV)[1:].view(keep.shape)
    odd.copy_(keep)                                     # no word of it is aligned
    for dev in (keep.to(DEV), odd):
        kv, rm, most = keep_kv_idx(dev, block_m)
        assert most == want_max
        got = kv.cpu().numpy()
        assert np.array_equal(got[..., :most], want) and (got[..., most:] == nb).all()
        masks = rm.cpu().numpy().view(np.uint64)
        for t in range(got.shape[2]):
            rows = keep[:, :, t * block_m:(t + 1) * block_m].numpy()
            bits = (rows.astype(np.uint64) << np.arange(rows.shape[2], dtype=np.uint64)[:, None]).sum(2)
            pad = np.concatenate([bits, np.zeros_like(bits[..., :1])], -1)       # the sentinel: none
            assert np.array_equal(masks[:, :, t], np.take_along_axis(pad, got[:, :, t], -1))


def test_keep_lists_of_many_tiles(hip_lib):
    """More tiles than one launch dimension holds at a workgroup each."""
    B, H = 8700, 2000                                   # 17.4 million one-row tiles of two blocks
    keep = torch.zeros(B, H, 1, 2, dtype=torch.bool, device=DEV)
    keep[..., 1] = torch.arange(B * H, device=DEV).view(B, H, 1) % 3 == 0
    kv, _, most = keep_kv_idx(keep, 64, want_rowmask=False)
    on = keep[..., 1]
    assert most == 1
    assert torch.equal(kv[..., 0], torch.where(on, 1, 2).to(torch.int32)) and (kv[..., 1] == 2).all()


@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16), (256, torch.bfloat16)])
def test_cached_block_means(hip_lib, D, dtype):
    """k_pool_at holds the means of the summary planes in the model's dtype, once per query head."""
    g = torch.Generator().manual_seed(D)
    q = torch.randn(2, 4, 300, D, generator=g).to(dtype).to(DEV)
    k = torch.randn(2, 2, 300, D, generator=g).to(dtype).to(DEV)
    sel = make_sel(mode="topk")
    sa.select_mask_v1(q, k, 0.1, sel=sel, layer_idx=7)
    planes = sa.block_summary(k, _capi.MODE_MEAN)
    want = sa.block_means(planes, 2, 2, 5, D).repeat_interleave(2, dim=1).to(dtype)
    assert torch.equal(sel.k_pool_at[7], want)
