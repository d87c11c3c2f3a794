"""Decode attention (Q == 1) against 64-bit softmax attention on the same inputs."""

import pytest
import torch

import sparse_attention as sa
from block_attn import decode_attn

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def qkv(seed, B, H, Hk, N, D, dtype):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q = torch.randn(B, 1, H, D, generator=g, device=DEV).to(dtype).transpose(1, 2)
    k = torch.randn(B, Hk, N, D, generator=g, device=DEV).to(dtype)
    v = torch.randn(B, Hk, N, D, generator=g, device=DEV).to(dtype)
    return q, k, v


def exact(q, k, v, scale):
    """(out, sum of p |v|) [B, 1, H, D] in fp64."""
    rep = q.shape[1] // k.shape[1]
    kd = k.double().repeat_interleave(rep, 1)
    vd = v.double().repeat_interleave(rep, 1)
    p = torch.softmax((q.double() * kd).sum(-1) * scale, -1).unsqueeze(-1)
    return (p * vd).sum(2).unsqueeze(1), (p * vd.abs()).sum(2).unsqueeze(1)


def bound(ref, mass, dtype):
    """P and the output are rounded once each to the element format: half a unit in the last place
    is 2^-8 of the value for bf16's 8 significant bits, 2^-11 for fp16's 11 (a weight below fp16's
    normal range moves by 2^-25 of the largest instead).  fp32 scores and sums move a weight by
    less than 1e-5 of itself, and the normaliser with them."""
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    return u * (mass + ref.abs()) + 2e-5 * mass + 1e-7


# One step, its edges, one and several splits, a ragged last split; one query head per KV head,
# a whole group, and a group past the MFMA's 16 columns.
@pytest.mark.parametrize("N", [1, 31, 33, 129, 511, 512, 4097])
@pytest.mark.parametrize("D,H,Hk,B,dtype", [(64, 8, 8, 3, torch.bfloat16), (64, 8, 2, 1, torch.float16),
                                            (128, 28, 4, 1, torch.bfloat16),
                                            (128, 34, 2, 2, torch.float16),
                                            (256, 16, 2, 1, torch.bfloat16),
                                            (256, 9, 1, 2, torch.float16)])
def test_decode_matches_fp64(hip_lib, N, D, H, Hk, B, dtype):
    print(f"[case] decode N={N} D={D} H={H}/{Hk} B={B} {dtype}", flush=True)
    q, k, v = qkv(N + D, B, H, Hk, N, D, dtype)
    out, _ = sa.block_sparse_attention(None, q, k, v, None, D ** -0.5)
    assert out.shape == (B, 1, H, D) and out.is_contiguous()
    ref, mass = exact(q, k, v, D ** -0.5)
    assert ((out.double() - ref).abs() <= bound(ref, mass, dtype)).all()


def test_decode_special_values(hip_lib):
    """An infinite value in the last key's row stays infinite (rows past the end add nothing), a
    NaN key touches only its own KV head, and keys of score -inf weigh nothing."""
    q, k, v = qkv(3, 1, 8, 2, 130, 128, torch.bfloat16)
    v[0, 0, 129, 5] = float("inf")
    k[0, 1, 7, 3] = float("nan")
    out, _ = sa.block_sparse_attention(None, q, k, v, None, 128 ** -0.5)
    assert torch.isposinf(out[0, 0, :4, 5]).all() and torch.isnan(out[0, 0, 4:]).all()
    assert torch.isfinite(out[0, 0, :4, :5]).all() and torch.isfinite(out[0, 0, :4, 6:]).all()
    q, k, v = qkv(4, 1, 4, 1, 200, 64, torch.float16)
    q[..., 0] = 1.0
    k[0, 0, :100, 0] = float("-inf")        # the first wavefronts' steps hold no finite score
    out, _ = sa.block_sparse_attention(None, q, k, v, None, 0.125)
    ref, mass = exact(q, k[:, :, 100:], v[:, :, 100:], 0.125)
    assert ((out.double() - ref).abs() <= bound(ref, mass, q.dtype)).all()


def test_decode_strided_cache_and_graph(hip_lib):
    """K/V views of a longer cache ([B, S, Hk, D] memory), replayed from a graph."""
    q, kc, vc = qkv(5, 2, 8, 2, 700, 128, torch.bfloat16)
    k, v = (t.transpose(1, 2).contiguous().transpose(1, 2)[:, :, 13:650] for t in (kc, vc))
    eager = decode_attn(q, k, v, 0.1)
    ref, mass = exact(q, k, v, 0.1)
    assert ((eager.double() - ref).abs() <= bound(ref, mass, q.dtype)).all()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = decode_attn(q, k, v, 0.1)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert torch.equal(decode_attn(q, k, v, 0.1), eager)


def test_other_calls_stay_with_sdpa(hip_lib):
    q, k, v = qkv(6, 1, 4, 2, 64, 128, torch.bfloat16)
    assert decode_attn(q, k, v, 0.1) is not None
    assert decode_attn(q, k, v, None) is None
    assert decode_attn(q.float(), k.float(), v.float(), 0.1) is None
    assert decode_attn(q, k.half(), v, 0.1) is None
    assert decode_attn(q.cpu(), k.cpu(), v.cpu(), 0.1) is None
    assert decode_attn(q, k[..., :96], v[..., :96], 0.1) is None
    assert decode_attn(q[..., :96], k[..., :96], v[..., :96], 0.1) is None
    assert decode_attn(q, k[:, :, :0], v[:, :, :0], 0.1) is None
    odd = torch.empty(1, 2, 64, 129, device=DEV, dtype=q.dtype)[..., 1:]
    assert decode_attn(q, odd, v, 0.1) is None                            # misaligned rows
    assert decode_attn(q, k.transpose(2, 3).contiguous().transpose(2, 3), v, 0.1) is None
    grad = q.detach().requires_grad_()
    assert decode_attn(grad, k, v, 0.1) is None
    with torch.no_grad():
        assert decode_attn(grad, k, v, 0.1) is not None
    with torch.autocast("cuda", dtype=torch.float16):
        assert decode_attn(q, k, v, 0.1) is None
    with torch.autograd.forward_ad.dual_level():
        assert decode_attn(q, k, v, 0.1) is None
    seen = []
    torch.func.vmap(lambda x: (seen.append(decode_attn(x, k, v, 0.1)), x)[1])(torch.stack([q, q]))
    assert seen == [None]


@pytest.mark.parametrize("which", ["q", "k", "v"])
def test_negated_views_are_read_as_their_values(hip_lib, which):
    """A view whose negation is put off (the imaginary part of a conjugate is one) is SDPA's."""
    ops = dict(zip("qkv", qkv(8, 1, 4, 2, 200, 128, torch.float16)))
    want, _ = sa.block_sparse_attention(None, *ops.values(), None, 0.1)
    ops[which] = torch._neg_view(-ops[which])
    got, _ = sa.block_sparse_attention(None, *ops.values(), None, 0.1)
    # SDPA's rounding against the kernel's: P and the output once each, as in bound()
    ref, mass = exact(*(t.resolve_neg() for t in ops.values()), 0.1)
    for out in (got, want):         # the same values
        assert ((out.double() - ref).abs() <= 4 * bound(ref, mass, torch.float16)).all()
    assert decode_attn(*ops.values(), 0.1) is None


def test_many_short_sequences_stay_with_sdpa(hip_lib):
    def taken(H, Hk, N, B, D=256):
        return decode_attn(*qkv(9, B, H, Hk, N, D, torch.bfloat16), 0.1) is not None
    assert not taken(8, 8, 32, 128) and not taken(8, 8, 1, 128)
    assert taken(8, 8, 33, 128) and taken(8, 8, 32, 127) and taken(8, 4, 32, 128) and taken(8, 8, 32, 128, 128)
    q, k, v = qkv(9, 128, 8, 8, 32, 256, torch.bfloat16)
    out, _ = sa.block_sparse_attention(None, q, k, v, None, 0.1)
    ref, mass = exact(q, k, v, 0.1)
    assert ((out.double() - ref).abs() <= 4 * bound(ref, mass, q.dtype)).all()   # SDPA's rounding
