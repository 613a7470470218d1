"""Which xLSTM groups and scans a tick's run lengths take (Engine.tick_route,
default widths), on both sides of each line of the rules. Results on either
side are checked by the parity tests of the ticks and scans."""

import pytest

from hackathon_amd import spec

pytestmark = pytest.mark.gpu

CFG = spec.ModelConfig(tower_depth=1)


@pytest.fixture(scope="module", params=["bf16", "fp32"])
def engine(request, dev):
    from hackathon_amd.engine import Engine

    eng = Engine(CFG, capacity=1, max_rows=1, linear_dtype=request.param)
    yield eng
    eng.close()


def test_small_second_group_keeps_the_general_scan(engine):
    """The second group of a split tick streams its tiles from 64 runs up (at
    eight heads of 512 columns 32 runs fill the device)."""
    seen = {}
    for n in range(40, 160):
        r = engine.tick_route([24] + [1] * (n - 1))
        if r["split"] < n:
            seen[n - r["split"]] = r["xlstm2"]
    assert seen[63] == 0 and seen[40] == 0
    assert seen[64] == 64 and seen[70] == 70
    # one group: from 32 runs up
    assert engine.tick_route([1] * 31)["xlstm1"] == 0
    assert engine.tick_route([8] + [1] * 31)["xlstm1"] == 32
