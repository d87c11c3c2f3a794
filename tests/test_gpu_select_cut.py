"""The tile selector's cut and sort at every row length up to and past its register layouts (512,
1024 and 2048 visible blocks) and sort sizes (64 to 512 winners): a causal context has a row of each
length, so one call per context covers them, against the oracle on the kernel's own scores."""

import numpy as np
import pytest
import torch

import sparse_attention as sa
from oracle import selector as OS

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def check(q, k, mode, budget, score="quest"):
    sel = sa.Selector()
    sel.mode, sel.budget_blocks, sel.router_score = mode, budget, score
    sel.router_mode, sel.router_grain, sel.router_quantile = "quantile", "cell", 0.3
    res = sa.select_v2(q.to(DEV), k.to(DEV), 0.125, sel=sel, want_tile_score=True)
    ref = OS.select_from_tile_scores(res.tile_score.cpu().numpy(), OS.SelectorConfig.from_selector(sel))
    assert np.array_equal(res.kv_idx.cpu().numpy(), ref.kv_idx)


@pytest.mark.parametrize("nb,budget", [(66, 8), (130, 16), (260, 32), (520, 64), (530, 112),
                                       (1030, 32), (2060, 48)])
@pytest.mark.parametrize("mode", ["router", "quest"])
def test_every_row_length(hip_lib, nb, budget, mode):
    print(f"[case] select cut nb={nb} budget={budget} {mode}", flush=True)
    g = torch.Generator().manual_seed(nb)
    q = torch.randn(1, 2, 64 * nb - 5, 64, generator=g).to(torch.bfloat16)
    k = torch.randn(1, 1, 64 * nb - 5, 64, generator=g).to(torch.bfloat16)
    check(q, k, mode, budget)


@pytest.mark.parametrize("nb", [100, 600])
def test_ties_and_signs(hip_lib, nb):
    """Few distinct scores (cuts inside runs of equal keys), all equal ones, and scores of both
    signs and of magnitudes apart (no common prefix)."""
    g = torch.Generator().manual_seed(nb)
    base = torch.randn(7, 64, generator=g)
    k = base[torch.randint(0, 7, (nb,), generator=g)].repeat_interleave(64, 0)[None, None]
    q = torch.randn(1, 2, 64, 64, generator=g).repeat(1, 1, nb, 1)
    for qq, kk in ((q, k), (torch.zeros_like(q), k),
                   (q[:, :, :1].expand_as(q), k * 2.0 ** torch.arange(nb).remainder(37).repeat_interleave(64)[:, None])):
        check(qq.to(torch.bfloat16), kk.to(torch.bfloat16), "router", 8)
        check(qq.to(torch.bfloat16), kk.to(torch.bfloat16), "topk", 16)
