"""The global submit calls of the counts form (per class its largest count over every env and robot, summed), counted
by the step's own workgroup and by submit_counts' kernel, at counts that begin on and off a 16-byte boundary, with class
counts that divide 16 and that do not, and with fewer bytes than one 16-byte word; the largest count lies at every byte in
turn of the small sizes."""
import pytest
import torch

import isaac_net_amd as P
from isaac_net_amd.wifi_config import WifiConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,R,n_cls", [(1, 2, 3), (3, 5, 1), (5, 3, 2), (7, 11, 3), (40, 16, 5), (300, 11, 1),
                                       (301, 13, 7), (9, 4, 16)])
@pytest.mark.parametrize("shift", [0, 1, 7, 8])
def test_calls_at_any_alignment(E, R, n_cls, shift):
    print(f"calls E={E} R={R} n_cls={n_cls} shift={shift}", flush=True)
    cfg = P.NRConfig(msg_sizes=(200.0,) * n_cls, frame_buffer=4, seed=0, wifi=WifiConfig())
    eng = P.make_engine("WIFI", E, R, "cuda:0", cfg, seed=0)
    x = torch.full((E, R), 20.0, device="cuda:0")
    n = E * R * n_cls
    g = torch.Generator().manual_seed(n + shift)
    buf = torch.zeros(n + 64, dtype=torch.uint8, device="cuda:0")
    want = int(eng.state_dict()["rng.ctr[1]"][0])
    for i in range(min(n, 24)):
        c = torch.randint(0, 2, (n,), generator=g, dtype=torch.uint8)
        c[(i * 5 if n > 120 else i) % n if i % 2 else n - 1 - i] = 3 + i % 3
        buf.fill_(255)                                  # (bytes outside the counts must not count)
        v = buf[shift:shift + n]
        v.copy_(c)
        v = v.view(E, R, n_cls)
        if i % 3 == 0:
            eng.submit_counts(v)
            eng.step(None, x)
        else:
            eng.step(None, x, counts=v)
        want += int(c.view(-1, n_cls).amax(0).int().sum())
        got = eng.state_dict()["rng.ctr[1]"]
        assert bool((got == want).all()), (i, got[:4].tolist(), want)
