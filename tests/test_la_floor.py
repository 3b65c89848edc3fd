"""The SINR floors below which the link adaptation does not search (PhyTables.la_floor, la_line): just below an MCS's
floor no PRB count meets the BLER target (host tables, every row of the link-adaptation table), the line lies below the
floors, and on the GPU the bounded search gives the bits of the full one, over SINRs from far below to far above the
table, NaN and infinities."""
import numpy as np
import pytest
import torch

import isaac_net_amd as P

DEV = "cuda:0"


@pytest.mark.parametrize("table,target,nprb,nsym", [(1, 0.1, 52, 12), (2, 0.1, 106, 12), (1, 0.01, 273, 2),
                                                    (2, 0.5, 24, 10), (1, 1e-4, 51, 12)])
def test_no_tb_passes_below_the_floor(table, target, nprb, nsym):
    t = P.PhyTables(table, target, 4, None)
    tbs, ci0, wi, ncb = t.la_tables(nprb, nsym)
    f = t.la_floor()
    assert f.shape == (t.M,) and np.isfinite(f).any()
    for m in range(t.M):
        if not np.isfinite(f[m]):
            continue
        xg = np.float32(min(max((f[m] + 1e-3 - t.s0) / t.ds, 0.0), t.G - 1)) - np.float32(1e-4)
        j0 = int(min(np.floor(xg), t.G - 2))
        wj = np.float32(xg - j0)
        p = t.bler[m]
        for n in range(1, nprb + 1):
            if tbs[n, m] <= 0:
                continue
            lo = p[ci0[n, m], j0] * (1 - wj) + p[ci0[n, m], j0 + 1] * wj
            hi = p[ci0[n, m] + 1, j0] * (1 - wj) + p[ci0[n, m] + 1, j0 + 1] * wj
            b = lo * (np.float32(1) - wi[n, m]) + hi * wi[n, m]
            assert 1.0 - (1.0 - float(b)) ** float(ncb[n, m]) > target, (m, n)
    line = t.la_line()
    assert line is not None
    for m in range(t.M):
        assert line[0] + m / line[1] < f[m] - 1e-3, m


@pytest.mark.parametrize("table", [1, 2])
@pytest.mark.parametrize("target", [1e-5, 1e-3, 0.01, 0.1, 0.3, 0.5, 0.9, 0.99])
def test_line_takes_the_rounding_before_the_olla_offset(table, target):
    """An effective SINR's float32 rounding, at most 1e-5 beta (linear), is there before the OLLA offset of up to 10 dB:
    the largest SINR that this rounding and that offset can lift to an MCS's floor still lies above the line."""
    t = P.PhyTables(table, target, 4, None)
    a, k = t.la_line()
    f = t.la_floor()
    for m in range(t.M):
        if np.isfinite(f[m]):
            least = 10 * np.log10(10 ** ((f[m] - 10.0) / 10) - 1e-5 * float(t.beta[m])) + 10.0
            assert float(a) + m / float(k) < least - 1e-3, m


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [dict(), dict(mcs_table=2, ul_mcs_max=20), dict(eff_sinr="mean_db"),
                                dict(n_prb=273, rbg_size=35), dict(ul_amc_alloc="previous", ul_power="whole_band"),
                                dict(olla_up_db=1.0, bler_target=0.3)])
def test_search_from_the_floor_equals_the_full_search(kw):
    cfg = P.NRConfig(control_step_ms=20.0, msg_sizes=(3000.0,), n_harq=4, seed=0, **kw)
    E, R, S = 32, 24, cfg.n_subbands
    print(f"link adaptation from the floor, {kw}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(3)
    a, b = (P.make_engine("L2", E, R, DEV, cfg, seed=5) for _ in range(2))
    assert a._ctab.thr_ext == 1
    b._ctab.thr_ext = 0
    mean = torch.rand(E, R, 1, generator=g, device=DEV) * 70.0 - 30.0
    for s in range(4):
        snr = mean + torch.randn(E, R, S, generator=g, device=DEV) * 6.0
        if s == 2:
            snr[3, 5, 1] = float("nan")
            snr[4, 6] = float("inf")
            snr[4, 7] = -float("inf")
        c = (torch.rand(E, R, 1, generator=g, device=DEV) < 0.7).to(torch.uint8)
        oa, ob = a.step(None, snr_db=snr, arrivals=c), b.step(None, snr_db=snr, arrivals=c)
        for k in oa:
            assert torch.equal(oa[k].nan_to_num(-7.0) if oa[k].is_floating_point() else oa[k],
                               ob[k].nan_to_num(-7.0) if ob[k].is_floating_point() else ob[k]), (s, k)
    for k in ("h_meta", "h_tbs", "sent", "csi", "olla", "ctr"):
        assert torch.equal(a.st[k].nan_to_num(-7.0) if a.st[k].is_floating_point() else a.st[k],
                           b.st[k].nan_to_num(-7.0) if b.st[k].is_floating_point() else b.st[k]), k
    assert int(a.st["ctr"][:, 0].sum()) > 100


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [dict(), dict(mcs_table=2), dict(n_prb=273, bler_target=0.5)])
def test_search_from_the_floor_at_the_largest_olla_offset(kw):
    """Robots at OLLA offsets of +10, 9.7 and -9.7 dB with reference SINRs from -28 to -4 dB: the lowest MCS passes at raw
    SINRs where the rounding of the log-sum-exp weighs the most."""
    cfg = P.NRConfig(control_step_ms=20.0, msg_sizes=(3000.0,), n_harq=4, seed=0, **kw)
    E, R, S = 16, 48, cfg.n_subbands
    print(f"link adaptation at the largest OLLA offset, {kw}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(4)
    a, b = (P.make_engine("L2", E, R, DEV, cfg, seed=5) for _ in range(2))
    b._ctab.thr_ext = 0
    for s in range(4):
        off = torch.full((E, R), 10.0, device=DEV)
        off[:, 1::4], off[:, 2::4] = 9.7, -9.7
        for e in (a, b):
            e.st["olla"].copy_(off)
        # (SNR input is the reference SINR: the power split over the PRBs and the fading come on top)
        snr = torch.rand(E, R, 1, generator=g, device=DEV) * 24.0 - 28.0
        snr = (snr + torch.randn(E, R, S, generator=g, device=DEV) * 0.5).contiguous()
        c = torch.ones(E, R, 1, dtype=torch.uint8, device=DEV)
        oa, ob = a.step(None, snr_db=snr, arrivals=c), b.step(None, snr_db=snr, arrivals=c)
        for k in oa:
            assert torch.equal(oa[k].nan_to_num(-7.0) if oa[k].is_floating_point() else oa[k],
                               ob[k].nan_to_num(-7.0) if ob[k].is_floating_point() else ob[k]), (s, k)
        for k in ("h_meta", "h_tbs", "sent", "csi", "olla", "ctr"):
            assert torch.equal(a.st[k], b.st[k]), (s, k)
    mcs = (a.st["h_meta"] >> 16) & 0xff
    assert int(a.st["ctr"][:, 0].sum()) > 50 and int((mcs == 0).sum()) > 0 and int((mcs > 0).sum()) > 20
