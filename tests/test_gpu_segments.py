"""The lanes that an env takes of a wavefront follow the batch size (few envs: one per wavefront; many: next_pow2(R)
lanes each), and an env's results do not: the first envs of a batch large enough for the narrow segments equal, bit for
bit, an engine of those envs alone, over the common configuration's builds and the general ones, the uplink, the
downlink, HARQ-IR and several cells, through a partial reset."""
import pytest
import torch

import isaac_net_amd as P
from isaac_net_amd import scenarios as S

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENA = dict(pf_update="rbg", pf_avg_idle="freeze", ul_retx_sched="tdma", ul_amc_alloc="previous",
            harq_combining="ir_lena", tr38901_los="stochastic")
# name -> config, R, envs of the large batch: more wavefronts at the next width than are resident (one cell 2048,
# several cells 1024)
CASES = {
    "plumbing R=5": (lambda: S.plumbing_config(), 5, 8200),                       # 8 lanes against 64
    "plumbing R=8, 16 lanes": (lambda: S.plumbing_config(), 8, 4100),
    "default R=16": (lambda: P.NRConfig(control_step_ms=10.0, seed=0), 16, 4100),  # 16 lanes against 64
    "default R=17, 32 lanes": (lambda: P.NRConfig(control_step_ms=10.0, seed=0), 17, 2050),
    "rl_scale R=32": (lambda: S.rl_scale_config(), 32, 2050),
    "rl_scale R=20, 106 PRB": (lambda: S.rl_scale_config(n_prb=106, n_harq=16), 20, 2050),
    "rl_scale downlink R=24": (lambda: S.rl_scale_config(dl=True), 24, 2050),
    "lena R=12": (lambda: S.rl_scale_config(fading_rician=False, **LENA), 12, 4100),
    "three cells R=16": (lambda: S.mc_interf_config(), 16, 2050),
    "three cells R=32": (lambda: S.mc_interf_config(), 32, 1030),
}


def bits(a):
    return a.contiguous().view(torch.int32) if a.dtype == torch.float32 else a


@pytest.mark.parametrize("name", list(CASES))
def test_segment_width_does_not_change_results(name):
    make, R, E = CASES[name]
    n, steps = 6, 5
    print(f"{name}: {n} envs of {R} robots alone against {E} envs, {steps} steps", flush=True)
    cfg = make()
    g = torch.Generator(device=DEV).manual_seed(4)
    big, few = (P.make_engine("L2", e, R, DEV, cfg, seed=9) for e in (E, n))
    nc = len(cfg.msg_sizes)
    x = torch.rand(E, R, 2, generator=g, device=DEV) * 200.0
    for s in range(steps):
        if s == 3:
            big.reset([1, 4])
            few.reset([1, 4])
        x = (x + torch.randn(E, R, 2, generator=g, device=DEV) * 0.05).clamp(0.0, 200.0)
        c = torch.poisson(torch.full((E, R, nc), 0.6, device=DEV), generator=g).clamp(max=3).to(torch.uint8)
        if cfg.dl:
            b = torch.where(torch.rand(E, R, generator=g, device=DEV) < 0.5, 2000.0, 0.0)
            big.add_dl_frames(None, b)
            few.add_dl_frames(None, b[:n].contiguous())
        ob = big.step(None, x, arrivals=c)
        of = few.step(None, x[:n].contiguous(), arrivals=c[:n].contiguous())
        for k in of:
            assert torch.equal(bits(of[k]), bits(ob[k][:n])), (s, k)
    for a, b in [(few.st, big.st)] + ([(few.dst, big.dst)] if cfg.dl else []):
        for k in a:
            if k != "clock" and a[k].shape[:1] == (n,):
                assert torch.equal(bits(a[k]), bits(b[k][:n])), k
    assert int(few.st["ctr"][:, 0].sum()) > 0


@pytest.mark.parametrize("level,E,R,epw", [("WIFI", 1500, 16, 4), ("WIFI", 4200, 6, 8), ("WIFI", 1030, 30, 2),
                                           ("WIFI_DCF", 2100, 16, 2), ("WIFI_DCF", 8200, 5, 8)])
def test_wifi_envs_per_wave_do_not_change_results(level, E, R, epw):
    n, steps = 5, 4
    print(f"{level}: {n} envs of {R} stations alone against {E} envs, {epw} envs per wavefront", flush=True)
    cfg = S.wifi_dcf_config()
    g = torch.Generator(device=DEV).manual_seed(4)
    big, few = (P.make_engine(level, e, R, DEV, cfg, seed=9) for e in (E, n))
    assert (big.envs_per_wave, few.envs_per_wave) == (epw, 1)
    x = (torch.rand(E, R, 2, generator=g, device=DEV) - 0.5) * 70.0
    for s in range(steps):
        c = torch.poisson(torch.full((E, R, 1), 0.8, device=DEV), generator=g).clamp(max=3).to(torch.uint8)
        c[:, 0] = 1                                    # (both batches make the same number of submit calls)
        c[:, 1:] = c[:, 1:].clamp(max=1)
        ob = big.step(None, x, counts=c)
        of = few.step(None, x[:n].contiguous(), counts=c[:n].contiguous())
        for k in of:
            assert torch.equal(bits(of[k]), bits(ob[k][:n])), (s, k)
