"""Which entry points a sparse layer calls, with what, without a GPU: host tensors that pass for
device ones, and a library that records its calls and launches nothing."""

import ctypes

import pytest
import torch

import _capi
import sparse_attention as sa
from block_attn import block_sparse_attn

LAUNCHES = {name for name, (res, args) in _capi.SIGNATURES.items()
            if res is _capi._i and args}              # the rest are host-side queries


class Dev(torch.Tensor):
    is_cuda = True


class Recorder:
    """The library with its launches recorded as (name, arguments); ``on[name]`` runs with each and
    may return the call's status."""

    def __init__(self, real):
        self.real, self.calls, self.on = real, [], {}

    def __getattr__(self, name):
        if name not in LAUNCHES:
            return getattr(self.real, name)

        def launch(*args):
            self.calls.append((name, args))
            return self.on.get(name, lambda *a: 0)(*args) or 0
        return launch

    def names(self):
        return [name for name, _ in self.calls]

    def args(self, name):
        found = [args for n, args in self.calls if n == name]
        assert len(found) == 1, (name, self.names())
        return found[0]


@pytest.fixture
def rec(monkeypatch):
    rec = Recorder(_capi.lib())
    monkeypatch.setattr(_capi, "lib", lambda: rec)
    monkeypatch.setattr(_capi, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(sa, "SEL", sa.Selector())
    sa.SEL.mode, sa.SEL.kernel_v2, sa.SEL.budget_blocks = "router", True, 8
    sa.SEL.k_min = 2
    return rec


def qkv(B=1, H=4, Hk=2, S=2048, D=64):
    return tuple(torch.zeros(B, h, S, D, dtype=torch.bfloat16).as_subclass(Dev)
                 for h in (H, Hk, Hk))


@pytest.mark.parametrize("before,after", [("quest", "mean"), ("mean", "quest")])
def test_policy_changed_between_preparation_and_selection(rec, before, after):
    """The planes are read as what they were made as, whatever SEL has become since."""
    sa.SEL.router_score = before
    rec.on["ugbsa_prepare_layer"] = lambda *a: setattr(sa.SEL, "router_score", after)
    sa.block_sparse_attention(None, *qkv(), None, 0.125)
    made, read = rec.args("ugbsa_prepare_layer"), rec.args("ugbsa_select")
    assert made[15:17] == (read[13], made[16]) and read[5] == made[16]
    assert read[13] == (_capi.MODE_QUEST if before == "quest" else _capi.MODE_MEAN)


def test_planes_of_another_mode_are_refused(rec):
    q, k, _ = qkv()
    sa.SEL.router_score = "mean"
    planes = sa.block_summary(k, _capi.MODE_QUEST)
    with pytest.raises(AssertionError):
        sa.select_v2(q, k, 0.125, planes=planes)
    assert "ugbsa_select" not in rec.names()
    sa.select_v2(q, k, 0.125, planes=planes, mode=_capi.MODE_QUEST)
    assert rec.args("ugbsa_select")[13] == _capi.MODE_QUEST


class Buckets:
    """A profiler that notes its buckets among the recorded calls."""
    enabled = True

    def __init__(self, rec):
        self.rec = rec

    def start(self, name):
        self.rec.calls.append((name, ()))
        return name

    def stop(self, name):
        self.rec.calls.append(("end " + name, ()))


@pytest.mark.parametrize("wrapped", [False, True])
def test_profiler_buckets(rec, monkeypatch, wrapped):
    """v2_select holds the selector and v2_kernel all of the attention, the K/V operand copies
    included, whether or not a harness wraps the selector."""
    monkeypatch.setattr(sa, "PROF", Buckets(rec))
    if wrapped:
        inner = sa._block_select_kv_idx_v2
        monkeypatch.setattr(sa, "_block_select_kv_idx_v2", lambda *a, **kw: inner(*a, **kw))
    q, k, v = qkv()
    sa.block_sparse_attention(None, q, k, v, None, 0.125)
    assert rec.names() == ["v2_select", "ugbsa_block_summary", "ugbsa_select", "ugbsa_router",
                           "end v2_select", "v2_kernel", "ugbsa_attn_fwd", "end v2_kernel"]
    assert rec.args("ugbsa_attn_fwd")[10] == v.data_ptr()      # not prepared: copied in this call


def test_layer_without_profiler_prepares_in_one_launch(rec):
    sa.block_sparse_attention(None, *qkv(), None, 0.125)
    assert rec.names() == ["ugbsa_prepare_layer", "ugbsa_select", "ugbsa_router", "ugbsa_attn_fwd"]
    assert rec.args("ugbsa_attn_fwd")[10] is None


# a list with masks beside Q's fragments fills an eighth (head_dim 64) or a quarter of a CU's LDS
@pytest.mark.parametrize("D,widest", [(64, 1013), (128, 1024), (256, 675)])
def test_row_lists_as_wide_as_the_mask_keep_the_wavefronts(rec, D, widest):
    waves = 8 if D == 64 else 4
    for nb in (widest, widest + 1):
        S = 64 * nb
        q, k, v = qkv(1, 1, 1, S, D)
        keep = torch.zeros(1, 1, S, nb, dtype=torch.bool).as_subclass(Dev)
        rec.calls.clear()
        rec.on["ugbsa_keep_kv_idx"] = lambda *a: ctypes.memset(a[8], 0, 4 * nb) and 0
        block_sparse_attn(q, k, v, keep, 0.125)
        slots = rec.args("ugbsa_attn_fwd_rows")[29]
        assert slots == (nb if nb == widest else 1)       # past it: the longest list (none here)
        listed = (nb + (nb + 31) // 32 + 1) // 2 * 2 * 4 + 8 * nb
        fits = waves * ((listed + (0 if D == 128 else 128 * D)) + 15 & ~15) <= 160 * 1024
        assert fits == (nb == widest) or D == 128         # (there 1024 is a cap on the copy to LDS)


def test_refused_call_caches_no_block_means(rec):
    """k_pool_at holds means that were computed, never the buffer of a call that failed."""
    q, k, _ = qkv()
    sa.SEL.mode = "topk"
    rec.on["ugbsa_block_summary_means"] = lambda *a: -1
    with pytest.raises(AssertionError):
        sa.select_mask_v1(q, k, 0.125, layer_idx=3)
    assert sa.SEL.k_pool_at == {}
    del rec.on["ugbsa_block_summary_means"]
    sa.select_mask_v1(q, k, 0.125, layer_idx=3)
    means = sa.SEL.k_pool_at[3]
    assert rec.calls[1][1][12] == means.data_ptr() and means.shape == (1, 4, 32, 64)


def test_row_masked_calls_say_whether_their_lists_grow(rec, monkeypatch):
    """A per-row layer's lists do; a caller's own masks may be any, so its tiles are ranked."""
    q, k, v = qkv()
    sa.SEL.kernel_v2 = False
    module = type("Layer", (), {"layer_idx": 0})
    keep = torch.zeros(1, 4, 2048, 32, dtype=torch.bool).as_subclass(Dev)
    monkeypatch.setattr(sa, "_block_select_mask", lambda *a: keep)
    sa.block_sparse_attention(module, q, k, v, None, 0.125)
    assert "ugbsa_attn_fwd_rows_grow" in rec.names() and "ugbsa_attn_fwd_rows" not in rec.names()
    rec.calls.clear()
    block_sparse_attn(q, k, v, keep, 0.125)
    assert "ugbsa_attn_fwd_rows" in rec.names()
    seen = []
    monkeypatch.setattr(sa, "block_sparse_attn",
                        lambda q, k, v, keep, scale, block_n, out, workspace: seen.append(1))
    sa.block_sparse_attention(module, q, k, v, None, 0.125)
    assert seen == [1]


@pytest.mark.parametrize("D", [64, 128, 256])
def test_split_shapes_cover_every_form(D):
    """The calls of test_gpu_attention_split.py launch every number of wavefronts per tile."""
    import test_gpu_attention_split as split
    lib = _capi.lib()

    def forms(shapes, row_masks):
        return {lib.ugbsa_attn_tile_waves(1, H, M, D, (M + 63) // 64, row_masks) for H, M in shapes}
    assert forms(split.LISTS, 0) == {1, 2, 4}
    assert forms(split.ROWS, 1) == ({1, 2, 4} if D < 256 else {1})     # no split row-masked form there
    past = lib.ugbsa_attn_tile_waves(1, 1, 64 * 530 - 9, D, 40, 0)     # its long contexts
    assert past == (4 if D == 64 else 1)
