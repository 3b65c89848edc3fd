"""The step kernels at the lanes per env that large batches take. The launch gives a small batch a whole wavefront per
env, so the reference trajectories, whose batches are small, run that layout alone by default; here they run in every
narrower one (INET_NR_LANES: several envs per wavefront, the segment's reductions and exchanges over part of it, each
lane's own terms of several cells' interference, the 32-lane builds): teacher-forced and free running on every
one-wavefront trajectory, with the bounds of the trajectories' own tests, and the idle and busy slots against the
oracle."""
import pytest
import torch

import isaac_net_amd as P
import test_gpu_idle_slots as idle
import test_gpu_parity as parity
from conftest import CASES, DL_CASES, MC_CASES
from gpu_util import load

pytestmark = pytest.mark.gpu


def _widths(R):
    """The widths below 64 of envs of R robots."""
    n = 1 << max(0, (R - 1).bit_length())
    return [w for w in (1, 2, 4, 8, 16, 32) if w >= n]


WIDTHS = [(n, w) for n in CASES + DL_CASES + MC_CASES for w in _widths(int(load(n)[0]["R"]))]


@pytest.mark.parametrize("name,lanes", WIDTHS)
def test_teacher_forced_bit_exact(name, lanes, monkeypatch):
    print(f"{lanes} lanes per env:", flush=True)
    monkeypatch.setenv("INET_NR_LANES", str(lanes))
    parity.test_teacher_forced_bit_exact(name)


@pytest.mark.parametrize("name,lanes", [(n, w) for n, w in WIDTHS if w == _widths(int(load(n)[0]["R"]))[0]])
def test_free_running_bit_exact(name, lanes, monkeypatch):
    print(f"{lanes} lanes per env:", flush=True)
    monkeypatch.setenv("INET_NR_LANES", str(lanes))
    parity.test_free_running_bit_exact(name)


SLOTS = next(m for m in idle.test_idle_and_busy_slots_equal_the_oracle.pytestmark if m.name == "parametrize").args[1]


@pytest.mark.parametrize("R,kw,lanes", [(R, kw, w) for R, kw in SLOTS if R <= 32 for w in _widths(R)])
def test_idle_and_busy_slots_equal_the_oracle(R, kw, lanes, monkeypatch):
    print(f"{lanes} lanes per env:", flush=True)
    monkeypatch.setenv("INET_NR_LANES", str(lanes))
    idle.test_idle_and_busy_slots_equal_the_oracle(R, kw)


@pytest.mark.parametrize("R,lanes", [(9, 8), (9, 12), (3, 128), (3, 0), (64, 32)])
def test_other_widths_are_refused(R, lanes, monkeypatch):
    monkeypatch.setenv("INET_NR_LANES", str(lanes))
    eng = P.make_engine("L2", 2, R, "cuda:0", P.NRConfig(control_step_ms=10.0, seed=0), seed=0)
    with pytest.raises(RuntimeError, match="invalid argument"):
        eng.step(None, torch.zeros(2, R, 2, device="cuda:0"))
