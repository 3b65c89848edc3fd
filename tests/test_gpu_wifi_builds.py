"""The mean-field step's builds without a lane for every background station (65 stations: 64 robots at one AP, 63 at two)
and with the general stage sums (8 and more attempts), free running against the oracle: busy and idle steps (sub-steps in
which no station of the wavefront contends take a short form), a background station that sends, both access noises, the
enqueue in the step and as its own launch. The bounds are test_gpu_wifi's."""
import numpy as np
import pytest
import torch

import isaac_net_amd as P
import test_gpu_wifi as W
from isaac_net_amd.wifi_config import WifiConfig
from oracle.wifi_oracle import WifiOracle

pytestmark = pytest.mark.gpu
TWO_APS = ((-20.0, 0.0), (20.0, 0.0))


class _Ref(dict):
    files = property(lambda self: list(self.keys()))


@pytest.mark.parametrize("R,kw", [
    (64, {}), (64, dict(max_tx=9)), (64, dict(access_category="BE", bg_stations=2)),
    (64, dict(access_category="BE", bg_stations=2, max_tx=10)), (64, dict(access_noise="mean", max_tx=12)),
    (63, dict(ap_positions_m=TWO_APS)), (63, dict(ap_positions_m=TWO_APS, max_tx=8)),
    (5, dict(max_tx=8)), (16, dict(max_tx=12)), (16, dict(max_tx=16, bg_stations=2)),
    (16, dict(max_tx=8, access_category="BE", bg_stations=2)), (7, dict(max_tx=8, ap_positions_m=TWO_APS)),
    (6, dict(max_tx=10, ap_positions_m=TWO_APS, ap_channels=(1, 6))),
    (8, dict(max_tx=9, access_category="VO", bg_stations=2, bg_ac="BE"))])
@pytest.mark.parametrize("in_step", [False, True])
def test_free_running_against_the_oracle(R, kw, in_step):
    print(f"wifi R={R} {kw} enqueue in the step: {in_step}", flush=True)
    E, T = 3, 7
    cfg = P.NRConfig(control_step_ms=10.0, msg_sizes=(1500.0, 9000.0), frame_buffer=12, seed=0,
                     cell_positions_m=((0.0, 0.0),), wifi=WifiConfig(**dict(dict(access_category="DCF"), **kw)))
    rs = np.random.default_rng(R + len(kw))
    eng, orc = P.make_engine("WIFI", E, R, "cuda:0", cfg, seed=3), WifiOracle(E, R, cfg, seed=3)
    pos = rs.uniform(-35.0, 35.0, (E, R, 2)).astype(np.float32)
    bad = []
    for s in range(T):
        counts = np.stack([rs.poisson(0.4, (E, R)), rs.poisson(0.05, (E, R))], -1).astype(np.uint8)
        if s in (3, 4):
            counts[:] = 0                                   # the queues empty: idle steps
        if s == 5:
            counts[1:] = 0                                  # one env sends
        for c in range(2):
            for i in range(int(counts[..., c].max())):
                orc.submit(None, torch.from_numpy(np.where(counts[..., c] > i, c + 1, 0).astype(np.int64)))
        cnt, x = torch.from_numpy(counts).to("cuda:0"), torch.from_numpy(pos)
        if in_step:
            og = eng.step(None, x.to("cuda:0"), counts=cnt)
        else:
            eng.submit_counts(cnt)
            og = eng.step(None, x.to("cuda:0"))
        oo = orc.step(None, x)
        ref = _Ref({f"s/out.{k}": v.numpy() for k, v in oo.items()})
        ref.update({f"s/{k}": v.numpy() for k, v in orc.state().items()})
        b = W.compare(ref, "s", {"out." + k: v for k, v in og.items()})
        b.update(W.compare(ref, "s", eng.state_dict()))
        if b:
            bad.append((s, b))
        pos = pos + rs.normal(0, 0.5, pos.shape).astype(np.float32)
    print(f"max |deviation| { {k: f'{v:.2e}' for k, v in W.MAX_DEV.items()} }", flush=True)
    W.MAX_DEV.clear()
    assert not bad, bad[:5]
