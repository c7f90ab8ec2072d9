"""Results that kernels hand over in mapped host memory, at the sizes where the hand-over
splits: fired-neuron lists against the spike rows."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def input_env(pkg, n_input, hz):
    """An INPUT population of n_input neurons, each its own stimulus entry, and one cell."""
    env = pkg.NetworkEnvironment(1, 2, 0, 1)
    env.set_neuron_params(0, "cell", 0, 1, 10.0, -65.0, 2.0, 0.0, -70.0, -50.0, 1.0, pkg.NORMAL,
                          [1.0, 0.0, 0.1, 5.0])
    index = env.set_neuron_params(1, "input", 0, n_input, 0, 0, 0, 0, 0, 0, 0, pkg.INPUT, [])
    f = pkg.StimFunc()
    f.poisson_hz, f.poisson_on, f.poisson_off, f.seed = hz, 0.0, math.inf, 5
    env.set_input_stim_ids(index, np.arange(n_input), f)
    env.initialize(50, 25)
    return env


@pytest.mark.parametrize("n_input,hz", [
    (1, 10000.0),        # one word, one bit
    (130, 0.0),          # no spike at all
    (65536, 10000.0),    # a tile's words full: more ids than are collected at a time
    (65537, 300.0),      # one word past a tile
    (300001, 10000.0),   # more ids than are handed over at a time
    (300001, 20.0),
])
def test_fired_lists_match_rows(pkg, n_input, hz):
    env = input_env(pkg, n_input, hz)
    env.loop_n_steps(0, 3, want_output=False)
    for step in (0, 2):
        want = np.flatnonzero(env.spike_row(step))
        got, n = env.fired(step)
        assert n == want.size and np.array_equal(got, want)
        for cap in {0, 1, min(want.size, 8192), max(0, want.size - 1)}:
            got, n = env.fired(step, cap=cap)
            assert n == want.size and np.array_equal(got, want[:cap])
    env.finalize()
