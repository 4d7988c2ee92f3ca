"""The launch tuner starts from the engine's own defaults at every size, and
times no two settings of the same launch."""
import os
import re

import pytest

from protomol3_amd import pmx, tune

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


class Recorder:
    def __init__(self, n):
        self.n, self.shape, self.seen = n, {}, []

    def set_tuning(self, knob, value):
        self.shape[knob] = value

    def md_set_state(self, x, v):
        pass

    def md_run(self, steps):
        self.seen.append(dict(self.shape))


def engine_constant(name):
    src = open(os.path.join(ROOT, "protomol3_amd", "csrc", "pmx.hip")).read()
    return int(re.search(rf"constexpr int {name} = (\d+);", src).group(1))


@pytest.mark.parametrize("n", [1500, 9999, 10000, 26000, 99999, 100000, 1000000])
def test_every_knob_is_timed_at_the_others_defaults(n):
    spread = int(n >= engine_constant("kSpread2From"))
    fixup = int(n < engine_constant("kFixupMainBelow"))
    default = {pmx.TUNE_PAIR_SCHEDULE: 0, pmx.TUNE_LIST_PRUNE: 1, pmx.TUNE_FIXUP_STREAM: fixup,
               pmx.TUNE_PAIR_BLOCKS_PER_CU: 0, pmx.TUNE_FFT_LINES: 16, pmx.TUNE_FFT_PLANES: 1,
               pmx.TUNE_SPREAD_STREAM: spread}
    sy = Recorder(n)
    tune.tune_launch(sy, None, None, rounds=1)
    assert sy.seen
    for shape in sy.seen:
        assert set(shape) == set(default)  # no knob without effect
        assert sum(shape[k] != default[k] for k in default) <= 1
    # one to eight lines a block: 16, the default, is the launch of 8
    lines = {min(8, s[pmx.TUNE_FFT_LINES]) for s in sy.seen}
    assert len(lines) == len({s[pmx.TUNE_FFT_LINES] for s in sy.seen})
