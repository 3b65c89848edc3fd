"""The Wi-Fi steps' forms that depend on what a wavefront holds, against each other, bit for bit, on every output and
state word: sub-steps in which no station of the wavefront contends take a short form, and the end of step leaves the
frames of a wavefront in place when none has to move. With one env per wavefront the quiet envs take the short forms;
with several, beside envs that always have frames queued, the general ones. Sizes around whole blocks of 8 stations and
frame slots (the row sums read blocks of 8; the frame outputs go out in blocks of 8 where they are whole)."""
import pytest
import torch

import isaac_net_amd as P
from isaac_net_amd.wifi_config import WifiConfig
from isaac_net_amd.wifi_engine import HipWifiDcfEngine, HipWifiEngine

pytestmark = pytest.mark.gpu


def _cfg(F, **kw):
    nr = {k: kw.pop(k) for k in list(kw) if k in P.NRConfig.__dataclass_fields__}
    return P.NRConfig(msg_sizes=(1500.0, 40000.0), frame_buffer=F, seed=0, wifi=WifiConfig(**kw), **nr)


def _same(a, b):
    a, b = a.reshape(-1), b.reshape(-1)
    return torch.equal(torch.nan_to_num(a.double(), nan=-7.5), torch.nan_to_num(b.double(), nan=-7.5))


@pytest.mark.parametrize("level,R,F,kw", [
    ("WIFI", 2, 3, {}), ("WIFI", 4, 8, {}), ("WIFI", 7, 12, {}), ("WIFI", 8, 16, {}), ("WIFI", 15, 7, {}),
    ("WIFI", 16, 17, dict(access_noise="mean")), ("WIFI", 23, 64, {}), ("WIFI", 31, 40, {}),
    ("WIFI", 5, 16, dict(ap_positions_m=((0.0, 0.0), (40.0, 0.0)))),
    ("WIFI", 5, 16, dict(ap_positions_m=((0.0, 0.0), (40.0, 0.0)), ap_channels=(1, 6))),
    ("WIFI_DCF", 3, 5, dict(access_category="DCF")), ("WIFI_DCF", 16, 16, dict(access_category="DCF"))])
def test_quiet_and_busy_wavefronts_agree(level, R, F, kw):
    print(f"{level} R={R} F={F} {kw}", flush=True)
    E, T = 8, 10
    cls = HipWifiEngine if level == "WIFI" else HipWifiDcfEngine
    cfg = _cfg(F, control_step_ms=20.0, **kw)
    n_st = R if level == "WIFI_DCF" else R + len(kw.get("ap_positions_m", ((0.0, 0.0),)))
    rb, seg = 1 << (R - 1).bit_length(), 1 << (n_st - 1).bit_length()
    # (the mean-field launch regroups envs_per_wave segments of next_pow2(R) lanes into segments of next_pow2(R + A))
    one = cls(E, R, "cuda:0", cfg, seed=1, envs_per_wave=max(1, seg // rb))
    many = cls(E, R, "cuda:0", cfg, seed=1, envs_per_wave=64 // rb)
    g = torch.Generator().manual_seed(R * 100 + F)
    pos = (torch.rand(E, R, 2, generator=g) - 0.5) * 60.0
    bad = []
    for s in range(T):
        cnt = torch.poisson(torch.full((E, R, 2), 0.3 if s % 3 == 0 else 0.0), generator=g)
        cnt[..., 1] = 0
        cnt[1::2, :, 1] = 2                            # every second env is never empty
        cnt = cnt.to(torch.uint8).to("cuda:0")
        x = (pos + 0.05 * s).to("cuda:0")
        oa, ob = one.step(None, x, counts=cnt), many.step(None, x, counts=cnt)
        bad += [(s, "out." + k) for k in oa if not _same(oa[k], ob[k])]
        sa, sb = one.state_dict(), many.state_dict()
        bad += [(s, k) for k, v in sa.items() if torch.is_tensor(v) and not _same(v, sb[k])]
    assert not bad, bad[:8]
