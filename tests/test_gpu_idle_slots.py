"""Slots in which nobody has anything to send, and the HARQ words that stay in memory between transmissions: steps with
no message at all, with one robot sending, with messages that round to 0 bytes (complete at the first data slot without a
transmission), and with all robots sending at the cell edge (retransmissions over several steps), against the oracle
on one, two and four wavefronts per env, UL and DL, chase combining and HARQ-IR, dropped and restarted TBs."""
import pytest
import torch

import isaac_net_amd as P
from oracle import nr_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
KEYS = ("newest", "delivered", "timed_out", "dropped", "cap", "cls", "queue_len", "queue_bytes", "dl_newest",
        "dl_queue_len")


@pytest.mark.parametrize("R,kw", [
    (5, dict(dl=True, n_harq=4)), (40, dict(dl=True, n_harq=16)), (100, dict(dl=True, n_harq=8)),
    (150, dict(n_harq=2)), (9, dict(dl=True, harq_combining="ir_lena", n_harq=16)),
    (70, dict(harq_combining="ir_lena", harq_fail="drop")), (12, dict(dl=True, harq_fail="drop", n_harq=8)),
    (33, dict(fading_rho_per_ms=0.0, n_harq=8)), (3, dict(fading=False, n_harq=8, scheduler="rr"))])
def test_idle_and_busy_slots_equal_the_oracle(R, kw):
    print(f"idle slots R={R} {kw}", flush=True)
    cfg = P.NRConfig(control_step_ms=10.0, msg_sizes=(0.3, 2500.0), max_harq_tx=3, seed=0, **kw)
    E, steps = 3, 8
    g = torch.Generator().manual_seed(R)
    eng, ora = P.make_engine("L2", E, R, DEV, cfg, seed=3), O.OracleEngine(E, R, cfg, seed=3)
    snr = torch.rand(E, R, generator=g) * 12.0 - 4.0
    for s in range(steps):
        send = torch.zeros(E, R, dtype=torch.long)
        if s == 1:
            send[1, R // 2] = 2
        elif s == 3:
            send[:, ::2] = 1                           # 0.3 B: a frame of 0 bytes
        elif s in (4, 5):
            send = torch.where(torch.rand(E, R, generator=g) < 0.5, 2, 0)
        assert torch.equal(eng.submit(None, P.Requests(send.to(DEV))).cpu(), ora.submit(None, send))
        if cfg.dl:
            nb = torch.where(send > 0, torch.where(send == 1, 0.3, 1500.0), 0.0)
            assert torch.equal(eng.add_dl_frames(None, nb.to(DEV)).cpu(), ora.add_dl_frames(None, nb))
        og, oo = eng.step(None, snr.to(DEV)), ora.step(None, snr)
        for k in KEYS:
            if k in oo:
                assert torch.equal(og[k].cpu().to(oo[k].dtype), oo[k]), (s, k)
    assert int(eng.st["ctr"][:, 1].sum()) > 0          # (retransmissions were sent)
