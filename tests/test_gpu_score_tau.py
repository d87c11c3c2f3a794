"""The dump's noise estimate where its split over workgroups has edges: block ranges and pair
groups from one to several, ragged last ones, fewer scratch places than ranges wanted."""

import numpy as np
import pytest
import torch

import dump_block_scores as dbs
import sparse_attention as sa
import synth
from oracle import score_dump as OD
from parity import f32np, same_float_bits

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


# 5 blocks (the fewest a dump of budget 1 records) up to three 32-block chunks and all 1024 pairs;
# head_dim 256 takes 16 pairs a pass with Quest planes, 32 elsewhere
@pytest.mark.parametrize("S", [258, 513, 1025, 2049, 4160])
@pytest.mark.parametrize("D,mode,score,dtype", [(64, "topk", "mean", torch.bfloat16),
                                                (128, "quest", "quest", torch.float16),
                                                (128, "router", "mean", torch.bfloat16),
                                                (256, "quest", "quest", torch.bfloat16),
                                                (256, "topk", "mean", torch.float16)])
def test_tau_splits(hip_lib, S, D, mode, score, dtype):
    print(f"[case] tau S={S} D={D} {mode} {score} {dtype}", flush=True)
    q, k, _ = synth.make_layer(synth.CONFIGS["c1"], 3, S=S, Hq=4, Hkv=2, D=D, dtype=dtype)
    sel = sa.Selector()
    sel.mode, sel.router_score, sel.budget_blocks = mode, score, 1
    shard = dbs.record(q.to(DEV), k.to(DEV), D ** -0.5, sel=sel, want_tile_score=True)
    ref = OD.tau_hat(f32np(q), f32np(k), D ** -0.5, sa.use_quest(sel))
    # fp32 scores of both: a difference of two rows' scores, of the scores' own size, carries
    # at most a few times D 2^-24 of it, and the mean of their squares less
    np.testing.assert_allclose(shard["tau_hat"], ref, rtol=1e-4)
    # no partial sum left in g or r, the tiles past the valid ones among them: the order
    # statistics of the kernel's own scores, bit for bit
    T = shard["tile_score"].cpu().numpy()
    with np.errstate(invalid="ignore"):
        stats = OD.order_stats(T, *OD.dump_budgets(sel.budget_blocks, T.shape[-1]))
    for name, want in zip(("g", "r", "sigma", "g_rho"), stats):
        assert same_float_bits(shard[name], want), name
    again = dbs.record(q.to(DEV), k.to(DEV), D ** -0.5, sel=sel)
    for name in ("g", "r", "sigma", "g_rho", "valid", "tau_hat"):
        assert np.array_equal(shard[name], again[name], equal_nan=True), name


@pytest.mark.parametrize("mode,score,size", [("quest", "quest", 3e17), ("topk", "mean", 3e18),
                                             ("quest", "quest", 1e-15), ("topk", "mean", 1e-15)])
def test_tau_of_large_and_small_scores(hip_lib, mode, score, size):
    """Squares whose sum over a workgroup leaves fp32's range while their mean does not."""
    print(f"[case] tau of scores {size} {mode}", flush=True)
    g = torch.Generator().manual_seed(5)
    q = torch.randn(1, 4, 1025, 64, generator=g).to(torch.bfloat16)
    k = (size * torch.randn(1, 2, 1025, 64, generator=g)).to(torch.bfloat16)
    sel = sa.Selector()
    sel.mode, sel.router_score, sel.budget_blocks = mode, score, 1
    ref = OD.tau_hat(f32np(q), f32np(k), 0.5, sa.use_quest(sel))
    if size > 1:                                     # 256 pairs x 17 blocks: one workgroup's sum
        assert (256 * 17 * 2 * ref.astype(np.float64) ** 2 > 4 * float(np.finfo(np.float32).max)).all()
    shard = dbs.record(q.to(DEV), k.to(DEV), 0.5, sel=sel)
    np.testing.assert_allclose(shard["tau_hat"], ref, rtol=1e-4)
