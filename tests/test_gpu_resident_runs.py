"""Which calls run resident (one launch per run), by the engine's own counts of those
runs, with their results against the oracle bit for bit."""
import math

import numpy as np
import pytest

from conftest import new_env
from test_gpu_resident import bits, compare, small_env

pytestmark = pytest.mark.gpu


def runs(env):
    return env.get_option("resident_runs"), env.get_option("runs_given_up")


@pytest.mark.parametrize("options", [
    {},
    {"stage_spikes": 0},
    {"lane_max_fanin": 4096, "lane_synapses": 8},
    {"lane_synapses": 1},
    {"word_groups": 0, "index_bits": 16, "weight_precision": 2},
    {"index_bits": 16, "weight_precision": 1},
], ids=["default", "ring", "lanes", "wide", "fp8_idx16", "bf16_idx16"])
def test_layouts_run_resident(pkg, options):
    env = small_env(pkg, 1, **options)
    assert runs(env) == (0, 0)
    env.initialize(50, 25)
    for t in range(0, 75, 25):
        env.loop_n_steps(t, 25, want_output=False)
    assert runs(env) == (3, 0)
    env.finalize()


def test_teams_only_run_resident(pkg, orc):
    """Every population in narrow teams, 16 to a block, of a network small enough."""
    env = new_env(pkg, 1, scale=0.02, burst_n_mf=1)
    env.set_option("lane_max_fanin", 0)
    env.set_option("lane_synapses", 64)
    env.initialize(50, 25)
    compare(env, orc.OracleSim.from_env(env), [25, 25, 100], 25)
    assert runs(env)[0] > 0 and runs(env)[1] == 0
    env.finalize()


def test_largest_grids_run_resident(pkg, orc):
    """48k cells: a block on nearly every compute unit."""
    env = new_env(pkg, 1, scale=0.5, burst_n_mf=25)
    env.initialize(50, 25)
    assert 240 <= env.info().n_blocks <= 256
    compare(env, orc.OracleSim.from_env(env), [25, 30], 25)
    assert runs(env)[0] > 0 and runs(env)[1] == 0
    env.finalize()


@pytest.mark.parametrize("n", [128, 260, 380])
def test_one_step_projections_of_many_blocks(pkg, orc, n):
    """A population of wide teams (two neurons to a block) that projects onto itself in one
    step: every block reads the spikes of n / 2 others (up to 64, 128 and 192)."""
    env = pkg.NetworkEnvironment(1, 2, 2, 1)
    env.set_neuron_params(0, "cell", 0, n, 14.6, -68.0, 1.6, 16.0, -78.0, -53.0, 1.6, pkg.NORMAL,
                          [1.0, 0.0, 0.5, 5.0, 1.0, -82.0, 0.5, 9.0])
    pin = env.set_neuron_params(1, "input", 0, 640, 0, 0, 0, 0, 0, 0, 0, pkg.INPUT, [])
    rng = np.random.default_rng(n)
    for k, (pre_n, pre, fan, w, delay) in enumerate(((640, pin, 400, 0.02, 4.0), (n, 0, 40, -0.05, 1.0))):
        col = np.stack([np.sort(rng.choice(pre_n, fan, replace=False)) for _ in range(n)]).astype(np.int32)
        env.set_connectivity_csr(k, pre_n, n, pre, 0, w, delay, np.arange(0, n * fan + 1, fan, dtype=np.int64),
                                 np.ascontiguousarray(col.reshape(-1)), None)
    f = pkg.StimFunc()
    f.poisson_hz, f.poisson_on, f.poisson_off, f.seed = 30.0, 0.0, math.inf, 7
    env.set_input_stim_ids(pin, np.arange(640), f)
    env.set_option("lane_max_fanin", 0)
    env.set_option("lane_synapses", 1)
    env.initialize(50, 25)
    assert env.info().n_blocks >= n // 2
    ref = orc.OracleSim.from_env(env)
    ref.initialize()
    for t in range(0, 150, 50):
        env.loop_n_steps(t, 50, want_output=False)
        ref.run(t, 50)
        for s in range(t, t + 50):
            assert np.array_equal(env.spike_row(s), ref.spike_row(s)), f"raster differs at step {s}"
    for x, y in zip(env.state(), ref.state()):
        assert np.array_equal(bits(x), bits(y))
    assert env.totals()[0][0] > 0 and runs(env)[0] > 0 and runs(env)[1] == 0
    env.finalize()


def test_given_up_run_is_counted(pkg, orc):
    """Given up once; a kernel per step from then on."""
    env = small_env(pkg, 3, run_polls=0)
    env.initialize(50, 25)
    compare(env, orc.OracleSim.from_env(env), [25, 50], 25)
    assert runs(env) == (1, 1)
    env.finalize()


@pytest.mark.parametrize("T_print,T,graph_steps,calls", [
    # calls of (steps, resident runs): short last runs joined to the others, equal cuts
    (50, 25, 25, [(15, 0), (16, 1), (26, 1), (40, 1), (41, 2), (51, 2), (100, 4), (1, 0)]),
    (50, 25, 3, [(25, 0), (16, 0), (50, 0)]),        # runs too short to pay
    (50, 25, 5, [(25, 4), (16, 3), (50, 9)]),
    (50, 25, 10, [(25, 2), (50, 4), (16, 1)]),
    (12, 12, 25, [(18, 1), (19, 2), (36, 2), (40, 3)]),  # a ring with room for 18 steps
])
def test_call_lengths_in_runs(pkg, orc, T_print, T, graph_steps, calls):
    env = small_env(pkg, 2, graph_steps=graph_steps)
    env.initialize(T_print, T)
    counts, loop = [], env.loop_n_steps
    def counted(t, n):
        before = runs(env)[0]
        out = loop(t, n)
        counts.append((n, runs(env)[0] - before))
        return out
    env.loop_n_steps = counted
    compare(env, orc.OracleSim.from_env(env), [n for n, _ in calls], T)
    assert counts == calls and runs(env)[1] == 0
    env.finalize()


def test_short_runs_of_a_large_grid(pkg):
    """24k cells in runs of 6 or 7 steps: a launch per step is faster there."""
    env = new_env(pkg, 1, scale=0.25, burst_n_mf=12)
    env.set_option("graph_steps", 5)
    env.initialize(50, 25)
    assert env.info().n_blocks > 128
    env.loop_n_steps(0, 50, want_output=False)
    assert runs(env) == (0, 0)
    env.set_option("graph_steps", 8)
    env.loop_n_steps(50, 50, want_output=False)
    assert runs(env) == (6, 0)
    env.finalize()


def test_given_up_run_is_not_timed(pkg):
    """What is timed are the steps launched again, and the step timer leaves the call out."""
    env = small_env(pkg, 3, run_polls=0)
    env.initialize(50, 25)
    env.step_timer(1)
    env.loop_n_steps(0, 25, want_output=False)
    assert env.step_timer() == (0.0, 0)
    env.loop_n_steps(25, 25, want_output=False)
    ms, launches = env.step_timer(0)
    assert ms > 0.0 and launches == 25
    env.finalize()
    env = small_env(pkg, 3, run_polls=0)
    env.initialize(50, 25)
    given_up, later = env.time_steps(200), env.time_steps(200)
    assert runs(env)[1] == 1 and env.info().current_step == 400
    assert 0.5 * later < given_up < 2.0 * later
    env.finalize()


def test_lane_synapses_as_given(pkg):
    """A given team width holds whether runs may be resident or not; the default is wider
    where they are."""
    def blocks(**options):
        env = small_env(pkg, 1, **options)
        env.initialize(50, 25)
        n = env.info().n_blocks
        env.finalize()
        return n

    assert blocks(lane_synapses=8) == blocks(lane_synapses=8, resident=0)
    assert blocks(lane_synapses=2) == blocks(lane_synapses=2, resident=0)
    assert blocks() > blocks(resident=0) == blocks(lane_synapses=8)
