"""The order of the correction's windows over the XCDs (gg_runs.h), with the rule compiled for the host: every
window once, and the work of boxes of equal sides in a row spread evenly.  A run's work is taken as its layers
times their share of a ball's shell, so the outer runs of a box cost less than the middle ones."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gragles_3d_amd", "csrc")
XCDS = 8
NMAX = {8: 32, 4: 48, 2: 64, 1: 96}  # largest side of the class with runs of so many layers


@pytest.fixture(scope="module")
def run_window(tmp_path_factory):
    d = tmp_path_factory.mktemp("runs")
    src = d / "runs.cpp"
    src.write_text('#include "gg_runs.h"\nextern "C" int w(int u, int chunk) { return gg::run_window(u, chunk); }\n'
                   'extern "C" int chunk(int nmax, int zt) { return gg::run_chunk(nmax, zt); }\n')
    so = str(d / "runs.so")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(src), "-o", so], check=True)
    lib = ctypes.CDLL(so)

    def order(n, zt):
        """The windows of positions 0 .. m - 1, m the next multiple of the rule's period from n on."""
        chunk = lib.chunk(NMAX[zt], zt)
        m = -(-n // (XCDS * chunk)) * XCDS * chunk
        return np.array([lib.w(u, chunk) for u in range(m)])

    return order


@pytest.mark.parametrize("zt", [8, 4, 2, 1])
@pytest.mark.parametrize("n", [1, 8, 64, 4096, 80000])
def test_every_window_once(run_window, n, zt):
    w = run_window(n, zt)
    assert w.size >= n and np.array_equal(np.sort(w), np.arange(w.size))


@pytest.mark.parametrize("side,zt", [(9, 8), (17, 8), (24, 8), (28, 8), (31, 8), (32, 8), (33, 4), (36, 4), (40, 4),
                                     (48, 4), (50, 2), (56, 2), (64, 2), (72, 1), (96, 1)])
def test_equal_sides_spread_evenly(run_window, side, zt):
    grains = 2000
    layer = np.tile(np.arange(side), grains)
    z = (np.arange(side) - (side - 1) / 2.0) / (side / 2.0)
    cost = 0.2 + np.sqrt(np.maximum(0.0, 1.0 - z * z))  # of a layer
    run_cost = np.array([cost[k:k + zt].sum() for k in range(0, side, zt)])
    at = np.nonzero(layer % zt == 0)[0]  # first tiles of the runs, in plan order
    w = run_window(-(-layer.size // zt), zt)
    xcd = np.empty(w.size, dtype=np.int64)
    xcd[w] = np.arange(w.size) % XCDS
    work = np.bincount(xcd[at // zt], weights=np.tile(run_cost, grains), minlength=XCDS)
    assert work.max() <= 1.05 * work.mean(), work / work.mean()
