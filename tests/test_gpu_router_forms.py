"""The router's forms: one launch, one workgroup plus fill, and the row fill.

The one-launch form ranks up to 2048 values of up to 65536 cells in
registers, where sigma_eff lies apart from sigma; the row fill writes many
short rows as one run of words.  Each side of these lines, in both grains,
against the mean and rank formed on the host: every value is exact.
"""

import numpy as np
import pytest
import torch

import _capi
from oracle import selector as OS
from parity import same_float_bits

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def ptrs(*ts):
    return [t.data_ptr() for t in ts]


@pytest.mark.parametrize("B,H,Qt", [(1, 1, 1), (2, 3, 65), (1, 4, 512), (1, 2, 513), (1, 32, 2048),
                                    (1, 33, 2048), (1, 2, 2049), (1, 1, 4097), (3, 5, 1400)])
@pytest.mark.parametrize("grain", [_capi.GRAIN_ROW, _capi.GRAIN_CELL])
@pytest.mark.parametrize("values", ["floats", "ties"])
@pytest.mark.parametrize("in_place", [False, True])
def test_router_forms(hip_lib, B, H, Qt, grain, values, in_place):
    print(f"[case] router {B} {H} {Qt} {grain} {values} {in_place}", flush=True)
    rng = np.random.default_rng(B * 1000 + H * 10 + Qt)
    sig = rng.standard_normal((B, H, Qt)).astype(np.float32)
    if values == "ties":
        sig = rng.integers(-2, 3, (B, H, Qt)).astype(np.float32)
        sig[rng.random(sig.shape) < 0.01] = np.inf
        sig[rng.random(sig.shape) < 0.01] = np.nan
    want_eff = OS.head_mean(sig) if grain == _capi.GRAIN_ROW else sig
    kb, ks, nb = 3, 5, 70
    for rmode, frac in ((_capi.ROUTER_QUANTILE, 0.0), (_capi.ROUTER_QUANTILE, 0.25),
                        (_capi.ROUTER_QUANTILE, 1.0), (_capi.ROUTER_ABS, 0.0)):
        kq = max(1, int(frac * sig.size))
        sd = torch.from_numpy(sig).to(DEV)
        eff = sd if in_place else torch.empty_like(sd)
        unc = torch.empty(sd.shape, dtype=torch.uint8, device=DEV)
        kv = torch.arange(ks, dtype=torch.int32, device=DEV).repeat(B, H, Qt, 1)
        thr = torch.empty(1, device=DEV)
        _capi.check(_capi.lib().ugbsa_router(sd.data_ptr(), B, H, Qt, grain, rmode, 0.125, kq,
                                             kv.data_ptr(), kb, ks, nb,
                                             *ptrs(eff, unc, thr), _capi.stream_ptr(DEV)), "router")
        assert same_float_bits(eff.cpu().numpy(), want_eff)
        with np.errstate(invalid="ignore"):
            if rmode == _capi.ROUTER_QUANTILE:
                want_thr = OS.kth_smallest(want_eff, kq)
                got = thr.cpu().numpy()[0]
                assert got == want_thr or (np.isnan(got) and np.isnan(want_thr))
                want_unc = want_eff <= want_thr
            else:
                want_unc = want_eff < np.float32(0.125)
        assert np.array_equal(unc.cpu().numpy().astype(bool), want_unc)
        want_kv = np.tile(np.arange(ks, dtype=np.int32), (B, H, Qt, 1))
        want_kv[~want_unc, kb:] = nb
        assert np.array_equal(kv.cpu().numpy(), want_kv)


@pytest.mark.parametrize("B,H,M,NB", [(1, 2, 50, 8), (2, 3, 700, 16), (1, 2, 1024, 13), (1, 3, 1025, 24),
                                      (1, 1, 4096, 64), (1, 2, 4097, 72), (1, 1, 640, 520)])
@pytest.mark.parametrize("grain", [_capi.GRAIN_ROW, _capi.GRAIN_CELL])
@pytest.mark.parametrize("frac", [0.02, 0.6, 1.0])
def test_router_rows_forms(hip_lib, B, H, M, NB, grain, frac):
    print(f"[case] router rows {B} {H} {M} {NB} {grain} {frac}", flush=True)
    rng = np.random.default_rng(M + NB)
    margin = rng.integers(0, 200, (B, H, M)).astype(np.float32) / 64
    margin[rng.random(margin.shape) < 0.01] = np.nan
    k_eff = 1 if M < 1000 else 4
    row0 = min(64 * k_eff, M)
    eff = OS.head_mean(margin) if grain == _capi.GRAIN_ROW else margin
    elig = np.broadcast_to(np.arange(M) >= row0, eff.shape)
    safe = np.where(elig & ~np.isnan(eff), eff, np.float32(np.inf))
    ranked = safe[:, 0] if grain == _capi.GRAIN_ROW else safe
    n_elig = (M - row0) * B * (1 if grain == _capi.GRAIN_ROW else H)
    kq = max(1, int(frac * n_elig)) if n_elig else 0
    want_thr = OS.kth_smallest(ranked, kq) if kq else np.float32("nan")
    want_unc = (safe <= want_thr) & elig
    keep0 = rng.integers(0, 2, (B, H, M, NB)).astype(np.uint8)
    visible = np.arange(NB)[None] <= (np.arange(M) // 64)[:, None]
    want_keep = np.where(want_unc[..., None], visible, keep0)
    md, keep = torch.from_numpy(margin).to(DEV), torch.from_numpy(keep0).to(DEV)
    me = torch.empty_like(md)
    unc = torch.empty(md.shape, dtype=torch.uint8, device=DEV)
    thr = torch.empty(1, device=DEV)
    _capi.check(_capi.lib().ugbsa_router_rows(md.data_ptr(), B, H, M, NB, grain,
                                              _capi.ROUTER_QUANTILE, 0.0, kq, k_eff,
                                              *ptrs(keep, me, unc, thr), _capi.stream_ptr(DEV)),
                "router_rows")
    assert same_float_bits(me.cpu().numpy(), eff)
    assert same_float_bits(thr.cpu().numpy(), np.array([want_thr]))
    assert np.array_equal(unc.cpu().numpy().astype(bool), want_unc)
    assert np.array_equal(keep.cpu().numpy(), want_keep)
