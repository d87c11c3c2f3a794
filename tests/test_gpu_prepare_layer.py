"""Summary planes and K/V operand copies from one launch: the bits of the two separate ones, and
the dispatcher's layer through it equal to the layer through the separate entry points."""

import pytest
import torch

import _capi
import sparse_attention as sa
from block_attn import attn_workspace, block_sparse_attn_v2

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def qkv(seed, B, H, Hk, S, D, dtype):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return tuple(torch.randn(B, S, h, D, generator=g, device=DEV).to(dtype).transpose(1, 2)
                 for h in (H, Hk, Hk))


# one row, a partial block, whole blocks, a ragged last one
@pytest.mark.parametrize("N", [1, 63, 128, 1001])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype,mode", [(torch.bfloat16, _capi.MODE_MEAN), (torch.float16, _capi.MODE_MEAN),
                                        (torch.bfloat16, _capi.MODE_QUEST), (torch.float16, _capi.MODE_QUEST)])
def test_same_bits(hip_lib, N, D, dtype, mode):
    print(f"[case] prepare_layer N={N} D={D} {dtype} mode={mode}", flush=True)
    B, Hk = 2, 3
    _, k, v = qkv(N + D, B, Hk, Hk, N, D, dtype)
    lib, code, st = _capi.lib(), _capi.dtype_code(dtype), _capi.stream_ptr(DEV)
    planes = sa.block_summary(k, mode)
    copies = 2 * B * Hk * ((N + 63) // 64) * 64 * D          # the schedule after them is written later
    ws = attn_workspace(B, Hk, N, D, DEV)
    _capi.check(lib.ugbsa_attn_prepare_kv(k.data_ptr(), *k.stride(), v.data_ptr(), *v.stride(), B, Hk, N,
                                          D, code, 64, ws.data_ptr(), ws.numel(), st), "prepare_kv")
    planes2, ws2 = torch.empty_like(planes), torch.empty_like(ws)
    _capi.check(lib.ugbsa_prepare_layer(k.data_ptr(), *k.stride(), v.data_ptr(), *v.stride(), B, Hk, N, D,
                                        code, mode, planes2.data_ptr(), ws2.data_ptr(), ws2.numel(), st),
                "prepare_layer")
    assert torch.equal(planes.view(torch.int16), planes2.view(torch.int16))
    assert torch.equal(ws[:copies].view(torch.int16), ws2[:copies].view(torch.int16))


@pytest.mark.parametrize("policy", [("router", "quest"), ("router", "mean"), ("topk", "mean")])
@pytest.mark.parametrize("D,S,dtype", [(64, 777, torch.float16), (128, 2048, torch.bfloat16),
                                       (256, 1500, torch.bfloat16)])
def test_layer_equals_separate_entry_points(hip_lib, monkeypatch, policy, D, S, dtype):
    q, k, v = qkv(S, 2, 8, 2, S, D, dtype)
    monkeypatch.setattr(sa, "SEL", sa.Selector())
    sa.SEL.mode, sa.SEL.router_score = policy
    sa.SEL.kernel_v2, sa.SEL.budget_blocks, sa.SEL.router_mode = True, 8, "quantile"
    out, _ = sa.block_sparse_attention(None, q, k, v, None, D ** -0.5)
    kv = sa._block_select_kv_idx_v2(q, k, D ** -0.5)
    assert torch.equal(out, block_sparse_attn_v2(q, k, v, kv, D ** -0.5).transpose(1, 2))
    # a wrapped selector sees the call and its result is used
    seen = []
    inner = sa._block_select_kv_idx_v2
    monkeypatch.setattr(sa, "_block_select_kv_idx_v2", lambda *a, **kw: (seen.append(1), inner(*a, **kw))[1])
    again, _ = sa.block_sparse_attention(None, q, k, v, None, D ** -0.5)
    assert seen == [1] and torch.equal(again, out)
    # a layout the kernels cannot read in place
    odd = torch.empty(*k.shape[:3], D + 1, dtype=dtype, device=DEV)[..., 1:].copy_(k)
    monkeypatch.setattr(sa, "_block_select_kv_idx_v2", inner)
    strided, _ = sa.block_sparse_attention(None, q, odd, v, None, D ** -0.5)
    assert torch.equal(strided, out)


def test_mismatched_layers_are_refused_as_before(hip_lib):
    q, k, v = qkv(3, 1, 4, 2, 256, 64, torch.bfloat16)
    saved = dict(vars(sa.SEL))
    try:
        sa.SEL.mode, sa.SEL.kernel_v2 = "topk", True
        for bad in ((q, k, v[:, :1]), (q, k, v.half()), (q.half(), k, v), (q, k[:, :, :200], v),
                    (q[:, :3], k, v)):
            with pytest.raises(AssertionError):
                sa.block_sparse_attention(None, *bad, None, 0.125)
    finally:
        sa.SEL.__dict__.update(saved)
