"""The mlp line's rate and roofline describe the same run: the GEMM operations of a step over the measured step, whatever the
separately timed per-layer kernels take.  CPU only (a stand-in for the library whose steps take a known time)."""
import argparse
import json
import os
import sys
import time

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


class Net:
    def __init__(self, n_in, width, hidden, n_out, seed):
        self.dims = [n_in] + [width] * hidden + [n_out]
        self.timed = False

    def layers(self):
        return list(zip(self.dims[1:], self.dims[:-1]))

    def set_data(self, X, T):
        pass

    def train(self, steps, batch=8192, lr=1e-3, graph=True):
        time.sleep(steps * 5e-3)

    def timing(self, on=True):
        self.timed = on

    def timing_reset(self):
        pass

    def timing_get(self, k):
        assert self.timed
        return 7, 1e4, 1.0  # ten seconds of other kernels

    def close(self):
        pass


class Library:
    MLP = Net
    MLP_KERNEL_NAMES = {0: "k_gemm forward"}


def test_roofline_is_of_the_timed_steps(capsys):
    bench.bench_mlp(Library, argparse.Namespace(steps=10, warmup=1))
    d = json.loads(capsys.readouterr().out)
    weights = 4 * 128 + 3 * 128 * 128 + 128 * 4
    flop = 2 * 8192 * (weights + weights + weights - 4 * 128)  # forward, weight gradients, activation gradients
    r = d["roofline"]
    assert r["achieved"] == pytest.approx(flop / (d["ms_per_step"] * 1e-3) / 1e12, rel=1e-12)
    assert r["frac"] == pytest.approx(r["achieved"] / r["peak"], rel=1e-12)
    assert d["value"] == pytest.approx(1e3 / d["ms_per_step"], rel=1e-12)
    assert "k_net" in r["kernel"] and "graph" not in d["metric"] and "kernels" not in d
