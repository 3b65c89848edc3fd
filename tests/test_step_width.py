"""The lanes per env that the step launch gives a batch (csrc/step_width.h, compiled for the host with g++): wider than
next_pow2(R) only while every wavefront of the batch is resident, by its registers and by its LDS; and the LDS that
this counts on, against what the compiled kernels hold."""
import ctypes
import os
import re
import struct
import subprocess

import pytest
import torch

from conftest import ROOT
from isaac_net_amd import _lib

CSRC = os.path.join(ROOT, "isaac-net_amd", "csrc")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"

DRIVER = r"""
#include <cstdio>
#include "step_width.h"
int main() {
    int E, rb0, occ, n_ul, drop, max_tx, nc, S, ir, common, W;
    while (scanf("%d %d %d %d %d %d %d %d %d %d %d", &E, &rb0, &occ, &n_ul, &drop, &max_tx, &nc, &S, &ir, &common,
                 &W) == 11) {
        auto lds = [&](int w) {
            return inet::step_lds_static(S, nc, ir, common, W) + inet::step_lds_bytes(n_ul, drop, w, max_tx, nc, S);
        };
        const int rb = inet::seg_width(E, rb0, occ, lds);
        printf("%d", rb);
        for (int w = 1; w <= 64; w *= 2) printf(" %zu", lds(w));
        printf("\n");
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def width(tmp_path_factory):
    d = tmp_path_factory.mktemp("step_width")
    (d / "drv.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{CSRC}", "-o", str(d / "drv"), str(d / "drv.cpp")], check=True)

    def run(rows):
        """[(lanes, {width: LDS bytes of a wavefront})] of rows (E, rb0, occ, n_ul, drop, max_tx, nc, S, ir, common[,
        waves])."""
        text = "\n".join(" ".join(str(int(v)) for v in (tuple(r) + (1,))[:11]) for r in rows)
        out = subprocess.run([str(d / "drv")], input=text,
                             capture_output=True, text=True, check=True).stdout.split("\n")
        vals = [[int(v) for v in line.split()] for line in out if line]
        return [(v[0], {1 << i: b for i, b in enumerate(v[1:])}) for v in vals]
    return run


def _waves(E, w):
    return -(-E * w // 64)


def _resident(lds, occ):
    return 256 * min(4 * occ, 160 * 1024 // (-(-lds // 1280) * 1280))


def test_wavefronts_of_a_widened_batch_are_resident(width):
    rows = [(E, rb0, 1 if nc > 1 else 2, n_ul, drop, 4, nc, S, ir, 0)
            for E in (1, 64, 500, 512, 513, 768, 1000, 1024, 1025, 1500, 2048, 2500, 4096, 9000, 16384)
            for rb0 in (1, 4, 8, 16, 32, 64) for S, nc in ((8, 1), (13, 1), (18, 1), (8, 2), (14, 3), (14, 4), (13, 7), (14, 7))
            for n_ul, drop in ((8, 0), (20, 0), (20, 1), (60, 1)) for ir in (0, 1)]
    got = width(rows)
    assert len(got) == len(rows)
    for r, (rb, lds) in zip(rows, got):
        E, rb0, occ = r[:3]
        assert rb0 <= rb <= 64 and rb & (rb - 1) == 0, r
        fits = lambda w: lds[w] + 16384 <= 160 * 1024  # noqa: E731
        assert rb == rb0 or _waves(E, rb) <= _resident(lds[rb], occ) or not fits(rb // 2), r
        assert rb == 64 or fits(rb), r
        if rb < 64:                                        # (the next width would not be)
            assert _waves(E, 2 * rb) > _resident(lds[2 * rb], occ), r


@pytest.mark.parametrize("row,lanes", [
    ((2048, 32, 2, 20, 1, 4, 1, 13, 0, 0), 32),    # the losses of 20 slots in LDS: 1280 wavefronts are resident
    ((1024, 32, 2, 20, 1, 4, 1, 13, 0, 0), 64),
    ((4096, 8, 2, 20, 1, 4, 1, 13, 0, 0), 16),
    ((2048, 32, 2, 20, 0, 4, 1, 13, 0, 0), 64),
    ((1024, 32, 1, 10, 0, 5, 7, 13, 0, 0), 32),    # seven cells: 512
    ((2048, 8, 1, 10, 0, 5, 7, 13, 0, 0), 16),
    ((1024, 16, 1, 10, 0, 5, 4, 14, 0, 0), 32),    # four cells: 768
    ((1024, 16, 1, 10, 0, 5, 3, 14, 0, 0), 64),    # three cells: one per SIMD
    ((256, 16, 2, 20, 0, 4, 1, 13, 0, 1), 64),
    ((4096, 32, 2, 10, 0, 5, 1, 13, 0, 1), 32),
    ((4096, 8, 2, 0, 0, 5, 1, 13, 0, 1), 32),         # (the downlink: no history)
    ((2048, 8, 2, 10, 0, 5, 1, 13, 0, 1), 64),
    ((50000, 1, 1, 60, 1, 4, 7, 14, 0, 0), 2)])         # (64 envs per wavefront: their N+I rows exceed the CU)
def test_measured_batches(width, row, lanes):
    assert width([row])[0][0] == lanes


def _kernels():
    """{kernel name: static LDS bytes} of the library's code objects (the offload bundles of libinet_nr.so)."""
    data = open(_lib.LIB_PATH, "rb").read()
    magic, out, pos = b"__CLANG_OFFLOAD_BUNDLE__", {}, 0
    tmp = f"/tmp/inet_co_{os.getpid()}"
    while (pos := data.find(magic, pos)) >= 0:
        n, q = struct.unpack_from("<Q", data, pos + 24)[0], pos + 32
        for _ in range(n if n < 16 else 0):
            off, size, ln = struct.unpack_from("<QQQ", data, q)
            name = data[q + 24:q + 24 + ln]
            q += 24 + ln
            if b"gfx950" in name and size:
                with open(tmp, "wb") as f:
                    f.write(data[pos + off:pos + off + size])
                notes = subprocess.run([READELF, "--notes", tmp], capture_output=True, text=True, check=True).stdout
                for k in notes.split(".group_segment_fixed_size:")[1:]:
                    out[re.search(r"\.name:\s+(\S+)", k).group(1)] = int(k.split(None, 1)[0])
        pos += len(magic)
    if os.path.exists(tmp):
        os.remove(tmp)
    return out


@pytest.mark.skipif(not os.path.exists(READELF) or not os.path.exists(_lib.LIB_PATH), reason="no readelf or no library")
def test_static_lds_covers_the_compiled_kernels(width):
    # <S, P, IR, VREF, RBT, link, NC, FX> in the mangled name
    pat = re.compile(r"nr_step_kernelILi(\d+)ELi(\d+)ELb([01])ELb([01])ELi(\d+)E.*?Li(\d+)ELi(\d+)EE")
    found = {}
    for name, lds in _kernels().items():
        m = pat.search(name)
        if m:
            S, _, ir, _, rbt, nc, fx = (int(v) for v in m.groups())
            found.setdefault((S, nc, ir, int(fx != 0), max(1, rbt // 64)), set()).add(lds)
    assert {k[4] for k in found} == {1, 2, 4} and {k[1] for k in found} == {1, 2, 3, 4, 5, 6, 7}
    assert {k[0] for k in found if k[1] == 1} >= {8, 13, 18}
    rows = [(1, 64, 1, 0, 0, -1, nc, S, ir, common, W) for S, nc, ir, common, W in found]
    for (k, have), (_, lds) in zip(found.items(), width(rows)):
        want = lds[64] - (8 * k[1] * k[0] if k[1] > 1 else 0)      # (less the N+I rows, dynamic)
        assert max(have) <= want <= min(have) + 128, (k, have, want)


@pytest.mark.skipif(torch.cuda.is_available(), reason="a refusal of the host's checks, tested where nothing can launch")
@pytest.mark.parametrize("R,S,n_data,drop,rc", [(200, 16, 60, 1, -2), (200, 16, 20, 1, -3), (200, 18, 64, 0, -3),
                                                (150, 13, 40, 1, -2), (100, 18, 64, 1, -3), (20, 18, 64, 1, -3)])
def test_launch_beyond_the_lds_is_refused(R, S, n_data, drop, rc):
    """Four wavefronts per env with RLC UM keep 3 KB of LDS per UL slot: with many slots the workgroup needs more than
    a CU has, and the call is refused (-2) before the launch; what fits goes on to the launch (-3: no GPU here)."""
    lib = _lib.load()
    st, tb, pm, out = _lib.InetNrState(), _lib.InetNrTables(), _lib.InetNrParams(), _lib.InetNrOutputs()
    tb.M, tb.C, tb.G, tb.EQW, tb.mcs_max, tb.NPRB = 29, 4, 8, 5, 28, 52
    pm.E, pm.R, pm.S, pm.P, pm.F, pm.N = 2, R, S, 8, 16, 100
    pm.max_tx, pm.input_kind, pm.harq_drop, pm.n_data, pm.n_cells = 4, 1, drop, n_data, 1
    got = lib.inet_nr_step(ctypes.byref(st), ctypes.byref(tb), ctypes.byref(pm), ctypes.c_void_p(16), n_data, 0,
                           ctypes.c_void_p(16), None, ctypes.byref(out), None)
    assert got == rc
