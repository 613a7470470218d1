"""Which xLSTM groups and scans a tick's run lengths take (Engine.tick_route,
default widths), on both sides of each line of the rules. Results on either
side are checked by the parity tests of the ticks and scans."""

import numpy as np
import pytest

import bench
from hackathon_amd import spec

pytestmark = pytest.mark.gpu

CFG = spec.ModelConfig(tower_depth=1)


@pytest.fixture(scope="module", params=["bf16", "fp32"])
def engine(request, dev):
    from hackathon_amd.engine import Engine

    eng = Engine(CFG, capacity=1, max_rows=1, linear_dtype=request.param)
    yield eng
    eng.close()


@pytest.mark.parametrize("steps,line", [(24, 64), (32, 64), (48, 80)])
def test_small_second_group_keeps_the_general_scan(engine, steps, line):
    """The second group of a split tick streams its tiles from 64 runs up, and
    from 32 more runs than the tick has steps (at eight heads of 512 columns 32
    runs fill the device)."""
    seen = {}
    for n in range(40, 220):
        r = engine.tick_route([steps] + [1] * (n - 1))
        if r["split"] < n:
            seen[n - r["split"]] = r["xlstm2"]
    assert seen[line - 1] == 0 and seen[line - 10] == 0
    assert seen[line] == line and seen[line + 6] == line + 6


def test_one_group_streams_from_32_runs(engine):
    """(2 x 8 x 32 work-groups of 256 columns.)"""
    assert engine.tick_route([1] * 31)["xlstm1"] == 0
    assert engine.tick_route([8] + [1] * 31)["xlstm1"] == 32


def test_groups_are_the_benchmark_replicas(engine):
    """Ticks of short runs stay whole below 192 runs; the line for the longest
    run is 9 with 16-bit linears and 16 in fp32. The whole rule, cost model
    included, is the one that bench.py replays."""
    lowp = engine.linear_dtype != "fp32"
    line = 9 if lowp else 16
    for n in (24, 64, 128):
        assert engine.tick_route([line - 1] + [1] * (n - 1))["split"] == n
    assert engine.tick_route([line] + [1] * 63)["split"] < 64
    assert engine.tick_route([1] * 191)["split"] == 191
    assert engine.tick_route([1] * 192)["split"] == 96
    assert engine.tick_route([line - 1] + [1] * 191)["split"] < 192
    weight_us = bench.xlstm_layer_weight_us(CFG, lowp)
    rng = np.random.default_rng(0)
    for _ in range(300):
        n = int(np.exp(rng.uniform(0, np.log(700))))
        lens = np.sort(rng.zipf(rng.uniform(1.3, 4.0), n).clip(max=rng.integers(1, 60)))[::-1]
        off = np.concatenate([[0], np.cumsum(lens)])
        assert engine.tick_route(lens)["split"] == bench.xlstm_split_point(off, weight_us, lowp), lens.tolist()
