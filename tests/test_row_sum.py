"""The row sums of the Wi-Fi step kernels (csrc/row_sum.h, torch's CPU order for a length that only the launch knows)
against torch's sum and against that order written out, at every length that a step can have (1 .. 65 elements), bit
for bit. Rows lie in memory as the kernel's do: zeros up to whole blocks of 8 (the FIFO columns), or up to the next
power of two with other envs' values behind (the station rows), which must not enter the sum. Compiled for the host
with g++ (the header is plain C++)."""
import os
import subprocess

import numpy as np
import pytest
import torch

HDR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "isaac-net_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include <cstring>
#include <vector>
#include "row_sum.h"
int main() {
    int t;
    if (scanf("%d", &t) != 1) return 1;
    while (t--) {
        int n, pad;
        if (scanf("%d %d", &n, &pad) != 2) return 1;
        std::vector<float> k(pad + 64, __builtin_nanf(""));
        for (int i = 0; i < pad; ++i) k[i] = 0.0f;
        for (int i = 0; i < n; ++i) {
            unsigned u;
            if (scanf("%x", &u) != 1) return 1;
            memcpy(&k[i], &u, 4);
        }
        float s = inet::aten_sum_padded(n, [&](int i) { return k[i]; },
                                        [&](int b) { inet::Row8 v; memcpy(&v, &k[8 * b], 32); return v; });
        unsigned u;
        memcpy(&u, &s, 4);
        printf("%x\n", u);
    }
    return 0;
}
"""


def _order(x):
    """torch's order, element by element in float32 (SumKernel.cpp)."""
    f = np.float32
    n = len(x)
    if n < 8:
        a = [f(0)] * 4
        for i in range(n // 4 * 4):
            a[i % 4] += x[i]
        for i in range(n // 4 * 4, n):
            a[0] += x[i]
        return ((a[0] + a[1]) + a[2]) + a[3]
    nv, fin = n // 8, f(0)
    for i in range(nv * 8, n):
        fin += x[i]
    for lane in range(8):
        a = [f(0)] * 4
        for i in range(nv // 4 * 4):
            a[i % 4] += x[i * 8 + lane]
        for i in range(nv // 4 * 4, nv):
            a[0] += x[i * 8 + lane]
        fin += ((a[0] + a[1]) + a[2]) + a[3]
    return fin


@pytest.fixture(scope="module")
def summer(tmp_path_factory):
    d = tmp_path_factory.mktemp("row_sum")
    src, exe = d / "drv.cpp", d / "drv"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-std=c++17", "-Wno-psabi", f"-I{HDR}", "-o", str(exe), str(src)], check=True)
    return exe


def test_matches_torch_order_at_every_length(summer):
    rs = np.random.default_rng(3)
    rows, lines = [], []
    for n in range(1, 66):
        blocks, pow2 = -(-n // 8) * 8, 1 << (n - 1).bit_length()
        # FIFO columns of any length; station rows from two stations on (65: the last station's value is not in the row)
        for pad in {blocks, *([pow2] if n > 1 else [])}:
            for kind in range(6):
                x = (rs.standard_normal(n) * 10.0 ** rs.integers(-6, 7, n)).astype(np.float32)
                if kind == 1:
                    x[rs.random(n) < 0.7] = 0.0
                if kind == 2:
                    x = np.where(rs.random(n) < 0.5, np.float32(-0.0), np.float32(0.0))
                if kind == 3:
                    x[:] = -0.0
                if kind == 4:
                    x = -np.abs(x)
                rows.append(x)
                lines.append(f"{n} {pad} " + " ".join(f"{b:x}" for b in x.view(np.uint32)))
    out = subprocess.run([str(summer)], input=f"{len(rows)}\n" + "\n".join(lines) + "\n", capture_output=True,
                         text=True, check=True).stdout.split()
    got = np.array([int(v, 16) for v in out], np.uint32)
    want = np.array([_order(x) for x in rows], np.float32).view(np.uint32)
    assert np.array_equal(got, want), [len(rows[i]) for i in np.nonzero(got != want)[0]]
    for x, g in zip(rows, got.view(np.float32)):
        assert g == torch.from_numpy(x[None].copy()).sum(-1).item(), len(x)
