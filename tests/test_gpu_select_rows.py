"""Per-row selection at the edges of its register layouts (1, 2, 4, .. blocks per lane), with ties,
NaN scores and margins at other ranks than the budget, against the oracle on the kernel's scores."""

import pytest
import torch

import sparse_attention as sa
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
