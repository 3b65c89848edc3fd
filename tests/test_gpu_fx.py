"""The step kernels built for the common configurations (PF, chase combining, EESM, RLC AM, OLLA, PHR cap, retx
priority, fading, with a fixed Rician phasor or without: every RBG count, 8 and 16 HARQ processes, envs in 32 and 64
lanes and on two wavefronts, UL and DL; config 3's three-cell kernel at 14 RBGs) equal the general builds bit for bit:
outputs and every state tensor, the frames' completion slots among them, through a partial reset. INET_NR_GENERIC=1
makes the library launch the general build for the same call, INET_NR_LANES sets the lanes per env."""
import os

import numpy as np
import pytest
import torch

import isaac_net_amd as P

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def run(name, E, R, steps, generic):
    from isaac_net_amd import scenarios as S
    os.environ["INET_NR_GENERIC"] = "1" if generic else "0"
    try:
        wl = S.Workload(E, R, steps, seed=2, name=name, device=DEV)
        eng = P.make_engine("L2", E, R, DEV, wl.cfg, seed=2)
        outs = []
        for s in range(steps):
            if s == steps // 2:
                eng.reset([1, E - 2])
            if name == "rl_scale_dl":
                for i in range(wl.dl_bytes.shape[1]):
                    eng.add_dl_frames(None, wl.dl_bytes[s, i])
            o = eng.step(None, wl.poses[s], arrivals=wl.counts[s])
            outs.append({k: v.detach().cpu() for k, v in o.items()})
        st = {k: v.detach().cpu() for k, v in eng.owner_state().items()}
        return outs, st
    finally:
        os.environ.pop("INET_NR_GENERIC", None)


def same(a, b):
    if a.is_floating_point():
        return torch.equal(a.nan_to_num(-7.0).view(torch.int32) if a.dtype == torch.float32 else a.nan_to_num(-7.0),
                           b.nan_to_num(-7.0).view(torch.int32) if b.dtype == torch.float32 else b.nan_to_num(-7.0))
    return torch.equal(a, b)


@pytest.mark.parametrize("name", ["rl_scale", "rl_scale_dl", "freq_sel", "mc_interf"])
def test_common_configuration_build_equals_general_build(name):
    E, R, steps = {"freq_sel": (16, 128, 4), "mc_interf": (16, 64, 6)}.get(name, (64, 32, 8))
    print(f"{name} {E}x{R}, {steps} steps: common-configuration build vs general build", flush=True)
    o_fx, st_fx = run(name, E, R, steps, generic=False)
    o_gen, st_gen = run(name, E, R, steps, generic=True)
    for s in range(steps):
        for k in o_fx[s]:
            assert same(o_fx[s][k], o_gen[s][k]), (s, k)
    for k in st_fx:
        assert same(st_fx[k], st_gen[k]), k
    assert int(st_fx["ul.q.enq"].sum()) > 0


# RBG count -> n_prb (the 38.101 carriers at 30 kHz; 8 RBGs: 273 PRB in RBGs of 35)
PRB = {8: 273, 10: 78, 11: 162, 12: 24, 13: 52, 14: 106, 16: 245, 17: 133, 18: 273}


def _run(cfg, E, R, steps, generic, monkeypatch):
    """Outputs and state of a run with frames of 0 bytes, frames of several TBs, full queues, time-outs and robots at
    the cell edge (retransmissions over several steps, TBs that start over)."""
    monkeypatch.setenv("INET_NR_GENERIC", "1" if generic else "0")
    g = torch.Generator(device=DEV).manual_seed(17 * R + cfg.n_subbands)
    eng = P.make_engine("L2", E, R, DEV, cfg, seed=2)
    snr = torch.rand(E, R, generator=g, device=DEV) * 20.0 - 6.0
    outs = []
    for s in range(steps):
        if s == steps // 2:
            eng.reset([1, E - 2])
        c = (torch.rand(E, R, 3, generator=g, device=DEV) < 0.4).to(torch.uint8)
        if s % 4 == 2:
            c[:, 1::2] = 0
        if cfg.dl:
            b = torch.where(torch.rand(E, R, generator=g, device=DEV) < 0.5, 1800.0, 0.0)
            b[:, ::5] = 0.3
            eng.add_dl_frames(None, b)
        o = eng.step(None, snr, arrivals=c)
        outs.append({k: v.detach().cpu() for k, v in o.items()})
    return outs, {k: v.detach().cpu() for k, v in eng.owner_state().items()}


@pytest.mark.parametrize("lanes", [32, 64, 128])
@pytest.mark.parametrize("n_harq", [8, 16])
@pytest.mark.parametrize("S", sorted(PRB))
def test_every_common_build_equals_the_general_build(S, n_harq, lanes, monkeypatch):
    R = {32: 19, 64: 37, 128: 70}[lanes] if S % 2 else {32: 32, 64: 24, 128: 97}[lanes]
    if lanes < 128:
        monkeypatch.setenv("INET_NR_LANES", str(lanes))
    for dl, fade in ((False, dict(fading_rician=True, fading_rho_per_ms=0.0)), (True, dict(fading_rician=True)),
                     (False, {}), (True, dict(fading_rho_per_ms=0.0))):
        kw = dict(fade, rbg_size=35) if S == 8 else dict(fade)
        cfg = P.NRConfig(n_prb=PRB[S], control_step_ms=10.0, msg_sizes=(0.3, 700.0, 4000.0), n_harq=n_harq,
                         max_harq_tx=3, frame_buffer=8, timeout_steps=4, dl=dl, seed=0, **kw)
        assert cfg.n_subbands == S
        print(f"{S} RBGs, {n_harq} processes, {lanes} lanes, R={R}, dl={dl}, {fade}", flush=True)
        o_fx, st_fx = _run(cfg, 5, R, 8, False, monkeypatch)
        o_gen, st_gen = _run(cfg, 5, R, 8, True, monkeypatch)
        for s in range(8):
            for k in o_fx[s]:
                assert same(o_fx[s][k], o_gen[s][k]), (dl, fade, s, k)
        for k in st_fx:
            assert same(st_fx[k], st_gen[k]), (dl, fade, k)
        assert {"ul.q.fin", "ul.h_comb", "ul.h_lo", "ul.h_hi"} <= set(st_fx)
        assert any(bool(o["delivered"].any()) for o in o_fx) and any(bool(o["timed_out"].any()) for o in o_fx)
