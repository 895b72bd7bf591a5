"""CPU: host-side logic of the package that needs no device."""
import os

import numpy as np
import pytest

from oracle import pyoracle as orc
from tscale_amd.attention import alibi_layer_schedule

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("wide", [1024, 4096])
def test_layer_schedule_matches_the_oracle(wide):
    # the oracle's schedule is itself pinned against the reference-built InitModelDescr
    for depth in list(range(1, 41)) + [64, 96]:
        w, s = orc.init_alibi(depth, wide)
        got = alibi_layer_schedule(depth, wide)
        assert [g[0] for g in got] == w.tolist(), depth
        assert np.allclose([g[1] for g in got], s), depth


def test_layer_schedule_of_the_documented_models():
    # 12 layers: one pair of width-1 layers, then 5 x (64 with slope 0.5, wide)
    sched = alibi_layer_schedule(12, 1024)
    assert sched[:2] == [(1, 0.0), (1, 0.0)] and sched[2:4] == [(64, 0.5), (1024, 0.0)] and len(sched) == 12
    # 24 layers: two leading pairs of width 1, ten alternating pairs
    sched = alibi_layer_schedule(24, 2048)
    assert [w for w, _ in sched].count(1) == 4 and [w for w, _ in sched].count(64) == 10 and len(sched) == 24


def test_matrix_scales_of_every_form():
    """A layer's scales: Python numbers, numpy scalars and arrays of one, tensors of one -- whose value at the time of the call counts."""
    import torch
    from tscale_amd.attention import VEC_SCALE, _product_scale
    want = lambda x, n: float(np.float32(x) * np.float32(VEC_SCALE) * np.float32(np.sqrt(np.float32(1.0) / np.float32(n))))
    for x in (0.3, 2, np.float32(0.3), np.float64(0.3), np.array(0.3), np.array(0.3, np.float32), torch.tensor(0.3), torch.tensor(0.3, dtype=torch.float64)):
        assert _product_scale(x, 768) == want(float(x), 768) == _product_scale(x, 768)
    t = torch.tensor(0.5)
    assert _product_scale(t, 64) == want(0.5, 64)
    t.fill_(0.25)
    assert _product_scale(t, 64) == want(0.25, 64)
    a = np.array(0.5)
    a[...] = 0.75
    assert _product_scale(a, 64) == want(0.75, 64)


def test_prefill_workgroup_mapping_visits_every_head_and_tile_once(tmp_path):
    """tests/cpp/test_wg_map.cpp walks the launch mapping of tscale_amd/csrc/wg_map.h (the code the kernel runs) over
    ~1500 launch shapes on the CPU, divisors of 1 (one query tile, one sequence, one unit per group) included."""
    import subprocess
    exe = tmp_path / "test_wg_map"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), os.path.join(ROOT, "tests", "cpp", "test_wg_map.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    assert r.stdout.startswith("OK")


def test_decode_splits(tmp_path):
    """tests/cpp/test_decode_splits.cpp holds the choice of tscale_amd/csrc/decode_splits.h against measured launches."""
    import subprocess
    exe = tmp_path / "test_decode_splits"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), os.path.join(ROOT, "tests", "cpp", "test_decode_splits.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    assert r.stdout.startswith("OK")


def test_stream_walk(tmp_path):
    """tests/cpp/test_stream_walk.cpp: the requests of the streamed product, those past a wave's share included."""
    import subprocess
    exe = tmp_path / "test_stream_walk"
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), os.path.join(ROOT, "tests", "cpp", "test_stream_walk.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    assert r.stdout.startswith("OK")
