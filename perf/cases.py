"""The work this package is measured on: sparse prefill and decode calls as a program makes them.

Layers go through ``sparse_attention.block_sparse_attention``, the function that transformers
calls for every attention layer of a model loaded with ``attn_implementation="block_sparse"``:
query, key and value are ``[B, S, heads, head_dim]`` projections viewed as ``[B, heads, S,
head_dim]``, and ``SEL`` holds the policy.  Beside them: the selector alone
(``_block_select_kv_idx_v2``), which harnesses wrap and time by itself, and the score-dump
diagnostic (``dump_block_scores.record``).

Shapes are the ones of this repository's benchmark layers (28/4, 40/8 and 16/2 heads at 32K to
128K tokens, ``synth.CONFIGS``), of its tests (8/2 and 4/2 heads, head_dim 64, ragged lengths,
fp16, both selector paths), and the same layers at the short prompts a served model sees most.
"""

from __future__ import annotations

import math
import os
import sys
from types import SimpleNamespace

import torch

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "uncertainty-gated-block-sparse-attention_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import dump_block_scores  # noqa: E402
import sparse_attention as sa  # noqa: E402

BLOCK = 64
K_MIN, K_MAX, TOP_P = 8, 112, 0.9       # Selector defaults
DEV = "cuda"

# A layer and its policy where a case says nothing else: a router layer as the benchmark runs it.
BASE = dict(kind="layer", B=1, H=28, Hk=4, S=4096, D=128, dtype="bf16", path="v2",
            mode="router", score="quest", budget=32, grain="row", rmode="quantile",
            quantile=0.25, planted=True, outliers=False, qk_norm=False)


def _case(**kw):
    return {**BASE, **kw}


def listed():
    return [
        # a short prompt through a 7B-sized layer: every block is kept, launches and host work count
        _case(name="layer_512", S=512),
        # a ragged fp16 prompt on a small model, absolute trigger per cell
        _case(name="layer_2k_ragged_fp16", H=8, Hk=2, S=1999, dtype="fp16", score="mean",
              budget=8, grain="cell", rmode="abs"),
        # two sequences of 8K at head_dim 64, plain Quest selection
        _case(name="layer_8k_hd64_b2", B=2, H=16, Hk=4, S=8192, D=64, mode="quest", budget=16),
        # the benchmark's headline layer: 32K tokens, router on Quest, 64 -> 128 blocks
        _case(name="layer_32k", S=32768),
        # the 14B-sized layer at 64K, top-96 on K means, outlier channels
        _case(name="layer_64k_topk_mean", H=40, Hk=8, S=65536, mode="topk", score="mean",
              budget=48, planted=False, outliers=True),
        # the 7B-sized layer at 128K, 128 -> 256 blocks: the largest call
        _case(name="layer_128k", S=131072, budget=64),
        # head_dim 256 with QK-norm at 64K, router on K means, 128 -> 256 blocks
        _case(name="layer_64k_hd256", H=16, Hk=2, S=65536, D=256, score="mean", budget=64,
              qk_norm=True),
        # the per-row selector (Selector.kernel_v2 False, its default) with the router
        _case(name="rows_layer_4k_router", path="v1", S=4096, score="mean", budget=16),
        # the per-row selector with budgets from the belief mass, a ragged length
        _case(name="rows_layer_10k_belief", path="v1", H=8, Hk=2, S=10007, mode="belief",
              score="mean"),
        # the selector alone at 16K on the 14B-sized layer
        _case(name="select_16k", kind="select", H=40, Hk=8, S=16384, score="mean", budget=48),
        # the score-dump diagnostic beside a 32K layer
        _case(name="dump_32k", kind="dump", S=32768),
        # one generated token against a 32K cache (Q == 1 is dense attention)
        _case(name="decode_32k", kind="decode", S=32768),
    ]


_SHAPES = [(28, 4, 128), (28, 4, 128), (40, 8, 128), (8, 2, 128), (16, 2, 256), (4, 2, 256),
           (16, 4, 64), (8, 8, 64)]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more call of the listed kinds: the same layers at other lengths, batches and policies."""
    cap = max(work(c)["flops"] for c in listed())
    while True:
        kind = rng.choice(["layer", "layer", "layer", "layer", "rows", "rows", "select", "dump",
                           "decode"])
        H, Hk, D = rng.choice(_SHAPES)
        c = _case(kind=kind, H=H, Hk=Hk, D=D, dtype=rng.choice(["bf16", "bf16", "bf16", "fp16"]),
                  B=rng.choice([1, 1, 1, 2, 3]), grain=rng.choice(["row", "row", "cell"]),
                  rmode=rng.choice(["quantile", "quantile", "quantile", "abs"]),
                  quantile=rng.choice([0.1, 0.2, 0.25, 0.4]), score=rng.choice(["mean", "quest"]),
                  mode=rng.choice(["router", "router", "topk", "quest"]),
                  budget=_log_int(rng, 8, 96), planted=rng.random() < 0.7,
                  outliers=rng.random() < 0.3, qk_norm=D == 256)
        if kind == "layer":
            c["S"] = _log_int(rng, 64, 131072)
        elif kind == "rows":
            c.update(kind="layer", path="v1", S=_log_int(rng, 64, 16384),
                     mode=rng.choice(["topk", "quest", "router", "router", "belief"]))
        elif kind == "select":
            c["S"] = _log_int(rng, 512, 131072)
        elif kind == "dump":
            c["S"] = _log_int(rng, 4096, 65536)
            c["budget"] = min(c["budget"], (c["S"] // BLOCK - 1) // 4)    # room for its deepest rank
        else:
            c.update(S=_log_int(rng, 128, 131072), B=rng.choice([1, 1, 2, 4, 8]))
        if rng.random() < 0.5 and kind != "decode":
            c["S"] = max(BLOCK, c["S"] // BLOCK * BLOCK)
        if c["B"] * c["S"] > 262144 or (c["path"] == "v1" and c["B"] * c["H"] * c["S"] > 1 << 19):
            c["B"] = 1
        if work(c)["flops"] <= cap and not (c["path"] == "v1" and c["H"] * c["S"] > 1 << 19):
            return c


# ---- inputs ---------------------------------------------------------------

def _inputs(case, seed):
    """q [B, S, H, D], k and v [B, S, Hk, D] fp32-drawn, cast to the case's dtype: N(0, 1), most
    key blocks aligned with the mean query of a later tile (near-tied cut-offs, as retrieval heads
    show), a few outlier key channels or QK-norm where the layer has them."""
    B, H, Hk, S, D = (case[n] for n in ("B", "H", "Hk", "S", "D"))
    g = torch.Generator(device=DEV).manual_seed(7919 * (seed % (1 << 40)) + 13)
    n_q = 1 if case["kind"] == "decode" else S
    q = torch.randn(B, n_q, H, D, generator=g, device=DEV)
    k = torch.randn(B, S, Hk, D, generator=g, device=DEV)
    v = torch.randn(B, S, Hk, D, generator=g, device=DEV)
    tiles = S // BLOCK
    if case["planted"] and n_q > 1 and tiles > 2:
        full = tiles * BLOCK
        qm = q[:, :full].reshape(B, tiles, BLOCK, Hk, H // Hk, D).mean(dim=(2, 4))   # [B, tiles, Hk, D]
        blk = torch.arange(tiles, device=DEV).view(1, tiles, 1)
        u = torch.rand(B, tiles, Hk, generator=g, device=DEV)
        tile = blk + 1 + (u * (tiles - 1 - blk)).long()             # a later tile
        hit = (torch.rand(B, tiles, Hk, generator=g, device=DEV) < 0.9) & (blk >= 1) & (tile < tiles)
        src = torch.gather(qm, 1, tile.clamp(max=tiles - 1).unsqueeze(-1).expand(B, tiles, Hk, D))
        kb = k[:, :full].reshape(B, tiles, BLOCK, Hk, D)
        noise = torch.randn(kb.shape, generator=g, device=DEV)
        kb = torch.where(hit[:, :, None, :, None], 0.8 * src[:, :, None] + 0.6 * noise, kb)
        k[:, :full] = kb.reshape(B, full, Hk, D)
        del kb, noise, src
    if case["outliers"]:
        k[..., torch.randperm(D, generator=g, device=DEV)[:max(1, round(0.05 * D))]] *= 4.0
    if case["qk_norm"]:
        q = q * torch.rsqrt(q.square().mean(-1, keepdim=True) + 1e-6)
        k = k * torch.rsqrt(k.square().mean(-1, keepdim=True) + 1e-6)
    dt = torch.float16 if case["dtype"] == "fp16" else torch.bfloat16
    return q.to(dt), k.to(dt), v.to(dt)


def _policy(case):
    return dict(mode=case["mode"], budget_blocks=case["budget"], router_mode=case["rmode"],
                router_grain=case["grain"], router_quantile=case["quantile"], router_tau=0.10,
                router_score=case["score"], kernel_v2=case["path"] == "v2", k_min=K_MIN,
                k_max=K_MAX, top_p=TOP_P)


def prepare(case, seed):
    q, k, v = (t.transpose(1, 2) for t in _inputs(case, seed))
    if case["kind"] == "decode":            # the cache holds [B, Hk, N, D]
        k, v = k.contiguous(), v.contiguous()
    elif case["kind"] != "layer":           # harnesses call the selector with contiguous tensors
        q, k, v = q.contiguous(), k.contiguous(), None
    return SimpleNamespace(kind=case["kind"], q=q, k=k, v=v, scaling=case["D"] ** -0.5,
                           policy=_policy(case), module=SimpleNamespace(layer_idx=0))


def run(state):
    sel = sa.SEL
    for name, value in state.policy.items():
        setattr(sel, name, value)
    if state.kind == "select":
        return sa._block_select_kv_idx_v2(state.q, state.k, state.scaling)
    if state.kind == "dump":
        shard = dump_block_scores.record(state.q, state.k, state.scaling)
        return {n: shard[n] for n in ("g", "r", "sigma", "g_rho", "valid", "tau_hat")}
    return sa.block_sparse_attention(state.module, state.q, state.k, state.v, None, state.scaling)[0]


# ---- what a pass cannot do without ----------------------------------------

def _budgets(case, nb):
    k_row = max(min(K_MAX, case["budget"]), K_MIN)
    k_base = min(2 * k_row, nb)
    k_slots = min(2 * k_base, nb) if case["mode"] == "router" else k_base
    return k_base, k_slots


def work(case):
    B, H, Hk, S, D = (case[n] for n in ("B", "H", "Hk", "S", "D"))
    nb = -(-S // BLOCK)
    if case["kind"] == "decode":
        return {"bytes": 2.0 * B * D * (2 * Hk * S + 2 * H), "flops": 4.0 * B * H * S * D}
    quest = case["mode"] == "quest" or (case["mode"] == "router" and case["score"] == "quest")
    # one dot product per query row and visible block (two with Quest's max and min)
    flops = (2 if quest else 1) * 2.0 * B * H * D * BLOCK * nb * (nb + 1) / 2
    read = 2.0 * B * S * D * (H + Hk)
    k_base, k_slots = _budgets(case, nb)
    if case["kind"] == "select":
        return {"bytes": read + 4.0 * B * H * nb * k_slots, "flops": flops}
    if case["kind"] == "dump":
        # the score noise reads 1024 row pairs against every block
        return {"bytes": read + 17.0 * B * H * nb,
                "flops": flops + (2 if quest else 1) * 2.0 * B * H * D * 2 * min(1024, S - 1) * nb}
    if case["path"] == "v2":
        share = 0.0
        if case["mode"] == "router":
            share = 1.0 if case["rmode"] == "abs" else case["quantile"]   # tiles over both budgets
        blocks = sum((1 - share) * min(t + 1, k_base) + share * min(t + 1, k_slots) for t in range(nb))
    else:
        k = max(K_MIN, min(K_MAX, case["budget"], nb))
        if case["mode"] == "belief":
            blocks = sum(max(min(t + 1, K_MIN), min(TOP_P * (t + 1), K_MAX)) for t in range(nb))
        else:
            share = case["quantile"] if case["mode"] == "router" and case["rmode"] == "quantile" else 0.0
            blocks = sum((1 - share) * min(t + 1, k) + share * (t + 1) for t in range(nb))
    flops += 4.0 * B * H * D * BLOCK * BLOCK * blocks
    return {"bytes": 2.0 * B * S * D * (2 * H + 2 * Hk), "flops": flops}


def _trigger_ranks_denormals(case):
    """Whether the layer's result hangs on the order of the tile selector's quantile margins.  Their
    denominator is FLT_MAX (the sink is forced), so they are fp32 denormals of a few hundred levels
    that many tiles share: the last bit of one score moves whole tiles across the threshold, and
    64-bit scores trigger other tiles than any 32-bit ones."""
    k_base, k_slots = _budgets(case, -(-case["S"] // BLOCK))
    return (case["path"] == "v2" and case["mode"] == "router" and case["rmode"] == "quantile"
            and k_base < k_slots)


def tolerance(case):
    if case["kind"] == "select":
        return {"differ": 1e-2}             # near ties change places; see _trigger_ranks_denormals
    if case["kind"] == "dump":
        return {"rel": 1e-3, "max": 0.1}
    return {"rel": 1e-2, "max": 0.3}


# ---- the same results in 64 bits ------------------------------------------

def _row_scores(q, k, quest, scaling):
    """Per-row block scores [H, M, NB] of one sequence, q [H, M, D], k [Hk, N, D] in fp64."""
    H, M, D = q.shape
    Hk, N, _ = k.shape
    nb = -(-N // BLOCK)
    kb = torch.cat([k, k.new_zeros(Hk, nb * BLOCK - N, D)], 1).view(Hk, nb, BLOCK, D)
    qg = q.reshape(Hk, H // Hk * M, D)
    if quest:
        s = torch.bmm(qg.clamp(min=0), kb.amax(2).transpose(1, 2).contiguous())
        s += torch.bmm(qg.clamp(max=0), kb.amin(2).transpose(1, 2).contiguous())
    else:
        s = torch.bmm(qg, kb.mean(2).transpose(1, 2).contiguous())
    return (s * scaling).view(H, M, nb)


def _tile_scores(q, k, quest, scaling):
    """Tile scores [H, Qt, NB]: the maximum over a tile's rows (rows past the end score 0), blocks
    after the tile -inf."""
    H, M, _ = q.shape
    Hk = k.shape[0]
    nb = -(-k.shape[1] // BLOCK)
    out = torch.empty(H, nb, nb, dtype=torch.float64, device=q.device)
    step = max(BLOCK, (1 << 28) // (8 * H * nb) * 8 // BLOCK * BLOCK)
    for r0 in range(0, M, step):
        s = _row_scores(q[:, r0:r0 + step].reshape(H, -1, q.shape[-1]), k, quest, scaling)
        pad = -s.shape[1] % BLOCK
        if pad:
            s = torch.cat([s, s.new_zeros(H, pad, nb)], 1)
        out[:, r0 // BLOCK:r0 // BLOCK + s.shape[1] // BLOCK] = s.view(H, -1, BLOCK, nb).amax(2)
    vis = torch.arange(nb, device=q.device) <= torch.arange(nb, device=q.device)[:, None]
    return out.masked_fill_(~vis, -math.inf)


def _kv_idx(case, q, k):
    """kv_idx [B, H, Qt, k_slots] of the tile selector.  The margin is defined on fp32 scores (its
    denominator is FLT_MAX, so its values are fp32 denormals), and so it is formed in fp32."""
    B, H, S, _ = q.shape
    nb = -(-S // BLOCK)
    k_base, k_slots = _budgets(case, nb)
    quest = case["mode"] == "quest" or (case["mode"] == "router" and case["score"] == "quest")
    router = case["mode"] == "router" and k_base < k_slots
    eye = torch.arange(nb, device=q.device)
    fmax = torch.finfo(torch.float32).max
    idx, sig = [], []
    for b in range(B):
        t = _tile_scores(q[b], k[b], quest, case["D"] ** -0.5)
        t[:, :, 0] = fmax
        t[:, eye, eye] = fmax
        val, order = t.sort(dim=-1, descending=True, stable=True)
        idx.append(order[..., :k_slots].to(torch.int32))
        if router:
            v = val.float()
            spread = (v[..., 0] - v[..., k_base]).clamp(min=1e-6)
            sig.append((v[..., k_base - 1] - v[..., k_base]) / spread)
    idx = torch.stack(idx)
    if router:
        sigma = torch.stack(sig)
        if case["grain"] == "row":
            acc = sigma[:, 0].clone()
            for h in range(1, H):
                acc += sigma[:, h]
            sigma = (acc / H)[:, None].expand(B, H, nb)
        if case["rmode"] == "quantile":
            kq = max(1, int(case["quantile"] * sigma.numel()))
            uncertain = sigma <= sigma.reshape(-1).sort().values[kq - 1]
        else:
            uncertain = sigma < 0.10
        tail = idx[..., k_base:]
        tail.masked_fill_(~uncertain[..., None], nb)
    return idx


def _attend_tiles(q, k, v, idx, scaling):
    """Attention of one sequence over kv_idx [H, Qt, slots]: out [H, M, D] fp64."""
    H, M, D = q.shape
    Hk, N, _ = k.shape
    nb = -(-N // BLOCK)
    slots = idx.shape[-1]
    pad = nb * BLOCK - N
    kb = torch.cat([k, k.new_zeros(Hk, pad, D)], 1).view(Hk, nb, BLOCK, D)
    vb = torch.cat([v, v.new_zeros(Hk, pad, D)], 1).view(Hk, nb, BLOCK, D)
    qb = torch.cat([q, q.new_zeros(H, pad, D)], 1).view(H, nb, BLOCK, D)
    out = torch.empty(H, nb, BLOCK, D, dtype=torch.float64, device=q.device)
    lane = torch.arange(BLOCK, device=q.device)
    step = max(1, (1 << 31) // (slots * BLOCK * D * 8))
    for h in range(H):
        for t0 in range(0, nb, step):
            ix = idx[h, t0:t0 + step].long()
            t = torch.arange(t0, t0 + ix.shape[0], device=q.device)
            key = (ix[..., None] * BLOCK + lane).view(ix.shape[0], 1, slots * BLOCK)
            row = (t[:, None] * BLOCK + lane).view(-1, BLOCK, 1)
            safe = ix.clamp(max=nb - 1)
            kk = kb[h * Hk // H][safe].view(-1, slots * BLOCK, D)
            s = torch.bmm(qb[h, t0:t0 + step], kk.transpose(1, 2)) * scaling
            del kk
            s.masked_fill_((key > row) | (key >= N), -math.inf)
            s = torch.softmax(s, -1)
            out[h, t0:t0 + step] = torch.bmm(s, vb[h * Hk // H][safe].view(-1, slots * BLOCK, D))
    return out.view(H, nb * BLOCK, D)[:, :M]


def _keep_rows(case, q, k):
    """Blocks each row of one sequence attends to, bool [B, H, M, NB] (per-row selector)."""
    B, H, S, _ = q.shape
    nb = -(-S // BLOCK)
    quest = case["mode"] == "quest" or (case["mode"] == "router" and case["score"] == "quest")
    blk, own = torch.arange(nb, device=q.device), torch.arange(S, device=q.device) // BLOCK
    vis = blk <= own[:, None]
    k_bud = min(max(min(K_MAX, case["budget"]), K_MIN), nb)
    k_eff = max(1, min(case["budget"], nb - 1))
    keep = torch.empty(B, H, S, nb, dtype=torch.bool, device=q.device)
    margin = torch.zeros(B, H, S, dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(H):
            s = _row_scores(q[b, h:h + 1], k[b, h * k.shape[1] // H][None], quest, case["D"] ** -0.5)[0]
            s.masked_fill_(~vis, -math.inf)
            val, order = s.sort(dim=-1, descending=True, stable=True)
            if case["mode"] == "belief":
                mass = torch.softmax(val, -1).cumsum(-1)[:, :min(K_MAX, nb)]
                count = ((mass < TOP_P).sum(-1) + 1).clamp(K_MIN, K_MAX)
            else:
                count = torch.full((S,), k_bud, device=q.device)
            keep[b, h] = torch.zeros(S, nb, dtype=torch.bool, device=q.device).scatter_(
                1, order, blk < count[:, None])
            if case["mode"] == "router" and nb > 1:
                margin[b, h] = (val[:, k_eff - 1] - val[:, k_eff]) / (val[:, 0] - val[:, k_eff]).clamp(min=1e-6)
    keep[..., 0] = True
    keep |= blk == own[:, None]
    if case["mode"] == "router" and nb > 1:
        elig = torch.arange(S, device=q.device) >= BLOCK * k_eff
        row = case["grain"] == "row"
        m = margin.mean(1, keepdim=True) if row else margin
        if case["rmode"] == "quantile":
            n = int(elig.sum()) * (1 if row else B * H)
            safe = torch.where(elig & ~m.isnan(), m, math.inf)
            unc = torch.zeros_like(m, dtype=torch.bool)
            if n:
                unc = (safe <= safe.reshape(-1).sort().values[max(1, int(case["quantile"] * n)) - 1]) & elig
        else:
            unc = (m < 0.10) & elig
        keep |= unc[..., None]
    return keep & vis


def exact(case, seed):
    q, k, v = (t.transpose(1, 2).double() for t in _inputs(case, seed))
    B, H, S, D = case["B"], case["H"], case["S"], case["D"]
    rep = H // case["Hk"]
    if case["kind"] == "decode":
        out = torch.empty(B, 1, H, D, dtype=torch.float64, device=DEV)
        for b in range(B):
            for g in range(case["Hk"]):
                qg = q[b, g * rep:(g + 1) * rep, 0]
                p = torch.softmax(qg @ k[b, g].t().contiguous() * D ** -0.5, -1)
                out[b, 0, g * rep:(g + 1) * rep] = p @ v[b, g]
        return out
    if case["kind"] == "dump":
        return _exact_dump(case, q, k)
    if case["kind"] == "select" or _trigger_ranks_denormals(case):
        return None                         # whole numbers; no value in 64 bits
    out = torch.empty(B, S, H, D, dtype=torch.float64, device=DEV)
    if case["path"] == "v2":
        idx = _kv_idx(case, q, k)
        for b in range(B):
            out[b] = _attend_tiles(q[b], k[b], v[b], idx[b], D ** -0.5).transpose(0, 1)
        return out
    keep = _keep_rows(case, q, k)
    key = torch.arange(S, device=DEV)
    for b in range(B):
        for h in range(H):
            for r0 in range(0, S, 4096):
                r1 = min(S, r0 + 4096)
                s = q[b, h, r0:r1] @ k[b, h // rep, :r1].t().contiguous() * D ** -0.5
                on = keep[b, h, r0:r1].repeat_interleave(BLOCK, dim=-1)[:, :r1]
                s.masked_fill_(~(on & (key[:r1] <= key[r0:r1, None])), -math.inf)
                out[b, r0:r1, h] = torch.softmax(s, -1) @ v[b, h // rep, :r1]
    return out


def _exact_dump(case, q, k):
    """The shard's arrays; sigma, g_rho and g of tiles whose ranks reach past the visible blocks
    hold -inf and NaN, which the fp32 definition gives too."""
    B, H, S, D = q.shape
    nb = -(-S // BLOCK)
    quest = case["mode"] == "quest" or (case["mode"] == "router" and case["score"] == "quest")
    k_b = min(2 * case["budget"], nb)
    rho = min(2 * k_b, nb)
    names = ("g", "r", "sigma", "g_rho")
    out = {n: torch.empty(B, H, nb, dtype=torch.float64, device=DEV) for n in names}
    tau = torch.empty(B, H, dtype=torch.float64, device=DEV)
    pairs = min(1024, S - 1)
    i = (torch.arange(pairs, device=DEV) * max(1, (S - 1) // pairs)).clamp(max=S - 2)
    for b in range(B):
        val = _tile_scores(q[b], k[b], quest, D ** -0.5).sort(dim=-1, descending=True).values
        g = val[..., k_b - 1] - val[..., k_b]
        r = val[..., 0] - val[..., k_b]
        r = torch.where(r < 1e-9, torch.full_like(r, 1e-9), r)
        out["g"][b], out["r"][b] = g, r
        out["sigma"][b] = (g / r).clamp(0, 2)
        out["g_rho"][b] = val[..., rho - 1] - val[..., rho]
        d = (_row_scores(q[b][:, i + 1], k[b], quest, D ** -0.5)
             - _row_scores(q[b][:, i], k[b], quest, D ** -0.5))
        tau[b] = (0.5 * d.square().mean(dim=(1, 2))).clamp(min=0).sqrt()
    out["valid"] = None                     # whole values
    out["tau_hat"] = tau
    return out
