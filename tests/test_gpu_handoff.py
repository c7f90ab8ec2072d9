"""What kernels hand over in mapped host memory and take as arguments, at the sizes where
that splits: fired-neuron lists, output trains and counts against the spike rows, rates
against the spikes they set."""
import math
import time

import numpy as np
import pytest

from conftest import new_env

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


@pytest.mark.parametrize("n_stims", [1, 8, 9, 17])
def test_rates_take_their_place_between_runs(pkg, n_stims):
    """Stimulus i fires all its neurons or none, as the rates of each window say."""
    env = pkg.NetworkEnvironment(1, n_stims + 1, 0, n_stims)
    env.set_neuron_params(0, "cell", 0, 1, 10.0, -65.0, 2.0, 0.0, -70.0, -50.0, 1.0, pkg.NORMAL,
                          [1.0, 0.0, 0.1, 5.0])
    pops = []
    for i in range(n_stims):
        index = env.set_neuron_params(1 + i, f"in{i}", 0, 3 + i, 0, 0, 0, 0, 0, 0, 0, pkg.INPUT, [])
        f = pkg.StimFunc()
        f.poisson_hz, f.poisson_on, f.poisson_off, f.seed = 0.0, 0.0, math.inf, 5 + i
        f.poisson_hz_from_freq = 1
        env.set_input_stim_ids(index, np.arange(3 + i), f)
        pops.append(index)
    env.initialize(50, 25)
    rng = np.random.default_rng(n_stims)
    t = 0
    for _ in range(4):
        on = rng.integers(0, 2, n_stims)
        env.set_input_freq([10000.0 * x for x in on])
        env.loop_n_steps(t, 2, want_output=False)
        t += 2
        for step in (t - 2, t - 1):
            counts, _ = env.counts(step)
            assert [counts[p] for p in pops] == [x * (3 + i) for i, x in enumerate(on)]
    spikes, _ = env.totals()
    assert spikes.sum() == sum(env.counts(s)[0].sum() for s in range(t))
    env.finalize()


@pytest.mark.parametrize("T", [1, 40, 47, 100])
def test_trains_match_rows(pkg, T):
    """Trains of one and of several blocks, handed over by calls of one window and of several."""
    env = new_env(pkg, 0)
    env.initialize(2 * T, T)
    t = 0
    for n in (T, T, 2 * T if T > 1 else 30):
        out = np.array(env.loop_n_steps(t, n))
        t += n
        rows = np.stack([env.spike_row(s) for s in range(t - T, t)])
        base = [env.population(i).base_id for i in range(env.info().n_populations)
                if env.population(i).device_type == pkg.OUTPUT]
        assert np.array_equal(out, rows[:, base[0]:base[0] + out.shape[1]])
    env.finalize()


def test_rates_set_before_a_batch_runs(pkg):
    """A batch runs on a stream of its own: the rates set on its networks come first."""
    def rates(env, hz):
        env.set_input_freq([hz] * env.info().n_stimuli)

    one, alone = new_env(pkg, 0), new_env(pkg, 0)
    for e in (one, alone):
        e.initialize(50, 25)
    batch = pkg.Batch([one])
    for w, hz in enumerate((3.0, 25.0, 1.0)):
        rates(one, hz)
        batch.run(25)
        rates(alone, hz)
        alone.loop_n_steps(25 * w, 25, want_output=False)
    assert np.array_equal(one.totals()[0], alone.totals()[0]) and one.totals()[1] == alone.totals()[1]
    for s in range(60, 75):
        assert np.array_equal(one.counts(s)[0], alone.counts(s)[0])
    for x, y in zip(one.state(), alone.state()):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    batch.destroy()
    one.finalize()
    alone.finalize()


@pytest.mark.parametrize("n_input", [1, 16382, 16384, 65537, 131070, 131071, 300001])
def test_state_read_back_in_parts(pkg, n_input):
    """The state that was set, read back whole, in parts, and in parts copied by threads."""
    env = input_env(pkg, n_input, 0.0)
    n = n_input + 1
    rng = np.random.default_rng(n)
    V, g = rng.standard_normal(n).astype(np.float32), rng.standard_normal(2 * n).astype(np.float32)
    refr = rng.integers(0, 1 << 30, n).astype(np.int32)
    env.set_state(V, g, refr)
    for _ in range(2):
        for got, want in zip(env.state(), (V, g, refr)):
            assert np.array_equal(got, want)
    env.finalize()


@pytest.mark.parametrize("preset", [0, 1])
def test_multipliers_read_back_in_parts(pkg, preset):
    """A plastic projection's multipliers as they were set, read back in parts and (1.97M
    synapses) in parts copied by threads."""
    env = new_env(pkg, preset, plasticities=1)
    idx = {env.projection(i).type: i for i in range(env.info().n_projections)}
    want = env.projection_csr(idx[0])[2].copy()
    env.set_plasticity(rule=pkg.STDP_TEACHER, target=idx[0], teacher=idx[11],
                       coefficients={pkg.A1_J: 0.0, pkg.A2_JI: -0.01}, time_window=50)
    env.initialize(50, 25)
    for _ in range(2):
        assert np.array_equal(env.projection_csr(idx[0])[2], want)
    env.finalize()


def test_batch_after_a_call_on_one_of_its_networks(pkg):
    """The batch's steps follow on from where a network's own calls left its ring."""
    one, other, alone = (new_env(pkg, 0) for _ in range(3))
    for e in (one, other, alone):
        e.initialize(50, 25)
    batch = pkg.Batch([one, other])
    batch.run(25)
    one.loop_n_steps(25, 17, want_output=False)
    batch.run(60)
    alone.loop_n_steps(0, 102, want_output=False)
    for s in range(90, 102):
        assert np.array_equal(one.spike_row(s), alone.spike_row(s))
    for x, y in zip(one.state(), alone.state()):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    batch.destroy()
    for e in (one, other, alone):
        e.finalize()


def test_statistics_of_uneven_batches(pkg):
    """Counts, events and totals of every network of a batch, as its own calls give them:
    networks of one and of several statistics blocks a row, of few and of many rows."""
    def nets():
        envs = [input_env(pkg, n, hz) for n, hz in ((140000, 20.0), (3, 900.0), (131073, 0.0))]
        for k in range(9):
            e = new_env(pkg, 0, stim_seed=300 + k)
            e.initialize(50, 25)
            envs.append(e)
        return envs

    one, alone = nets(), nets()
    batch = pkg.Batch(one)
    t = 0
    for n in (1, 60, 25):
        batch.run(n)
        for e in alone:
            e.loop_n_steps(t, n, want_output=False)
        t += n
        for a, b in zip(one, alone):
            assert np.array_equal(a.totals()[0], b.totals()[0]) and a.totals()[1] == b.totals()[1]
            for s in range(t - n, t):
                ca, ea = a.counts(s)
                cb, eb = b.counts(s)
                assert np.array_equal(ca, cb) and ea == eb
    assert all(e.totals()[1] > 0 for e in one[3:])
    batch.destroy()
    for e in one + alone:
        e.finalize()


def test_batch_run_does_not_grow_with_every_network(pkg):
    """A one-step run of 64 small networks is bound by launches, like one of 8: their
    statistics are closed side by side (one after another, 3.3 times as long)."""
    def median(n):
        envs = [new_env(pkg, 1, scale=0.03, burst_n_mf=2, seed=400 + k) for k in range(n)]
        for e in envs:
            e.initialize(50, 25)
        batch = pkg.Batch(envs)
        for _ in range(20):
            batch.run(1)
        times = []
        for _ in range(101):
            t0 = time.perf_counter()
            batch.run(1)
            times.append(time.perf_counter() - t0)
        batch.destroy()
        for e in envs:
            e.finalize()
        return sorted(times)[50]

    assert median(64) < 2.4 * median(8)


def test_batches_that_share_a_network(pkg):
    """Each batch follows on from what the other, the network's own calls, jumps of the step
    count and timed steps made of its ring."""
    one, other, alone = (new_env(pkg, 0) for _ in range(3))
    for e in (one, other, alone):
        e.initialize(50, 25)
    both, single = pkg.Batch([one, other]), pkg.Batch([one])
    both.run(7)
    both.run(7)
    single.run(5)
    both.run(6)
    one.time_steps(9, kernel_mean=True)
    both.run(4)
    one.loop_n_steps(1000, 3, want_output=False)
    both.run(8)
    alone.loop_n_steps(0, 38, want_output=False)
    alone.loop_n_steps(1000, 11, want_output=False)
    assert one.info().current_step == alone.info().current_step == 1011
    for s in range(1000, 1011):
        assert np.array_equal(one.spike_row(s), alone.spike_row(s))
        assert np.array_equal(one.counts(s)[0], alone.counts(s)[0])
    for x, y in zip(one.state(), alone.state()):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    both.destroy()
    single.destroy()
    for e in (one, other, alone):
        e.finalize()


def many_stimuli(pkg, n):
    """n stimuli of one neuron each, over 20 INPUT populations, in index order."""
    n_pops, per = 20, -(-n // 20)
    env = pkg.NetworkEnvironment(1, n_pops + 1, 0, n)
    env.set_neuron_params(0, "cell", 0, 1, 10.0, -65.0, 2.0, 0.0, -70.0, -50.0, 1.0, pkg.NORMAL,
                          [1.0, 0.0, 0.1, 5.0])
    pops = [env.set_neuron_params(1 + i, f"in{i}", 0, per, 0, 0, 0, 0, 0, 0, 0, pkg.INPUT, []) for i in range(n_pops)]
    for k in range(n):
        f = pkg.StimFunc()
        f.poisson_hz, f.poisson_on, f.poisson_off, f.seed = 0.0, 0.0, math.inf, 5 + k
        f.poisson_hz_from_freq = 1
        env.set_input_stim_ids(pops[k // per], np.array([k % per]), f)
    env.initialize(50, 25)
    base = [env.population(p).base_id for p in pops]
    return env, np.array([base[k // per] + k % per for k in range(n)])


@pytest.mark.parametrize("n", [40, 41, 300])
def test_rates_of_many_stimuli(pkg, n):
    env, ids = many_stimuli(pkg, n)
    rng = np.random.default_rng(n)
    t = 0
    for _ in range(4):
        on = rng.integers(0, 2, n)
        env.set_input_freq([10000.0 * x for x in on])
        env.loop_n_steps(t, 2, want_output=False)
        t += 2
        for step in (t - 2, t - 1):
            assert np.array_equal(env.spike_row(step)[ids], on)
    env.finalize()


def test_rates_do_not_grow_with_every_stimulus(pkg):
    """New rates before a one-step exchange: 1024 stimuli took 23 times as long as 8 when
    each 8 of them were a launch."""
    def median(n):
        env, _ = many_stimuli(pkg, n)
        times = []
        for t in range(101):
            freqs = [4.0 + t % 2] * n
            t0 = time.perf_counter()
            env.set_input_freq(freqs)
            env.loop_n_steps(t, 1, want_output=False)
            times.append(time.perf_counter() - t0)
        env.finalize()
        return sorted(times)[50]

    assert median(1024) < 10.0 * median(8)


@pytest.mark.parametrize("n_input,hz", [
    (65600, 10000.0),     # two words a thread, every bit set, the last thread's words past the end
    (262144, 3000.0),     # four words a thread, one whole tile
    (262209, 50.0),       # a word past it
    (600000, 4.0),        # three tiles
])
def test_fired_lists_by_parts_of_a_tile(pkg, n_input, hz):
    """Lists cut short inside a tile, at its end and in the next, both ways of asking."""
    env = input_env(pkg, n_input, hz)
    env.loop_n_steps(0, 2, want_output=False)
    want = np.flatnonzero(env.spike_row(1))
    for cap in sorted({0, 1, 5, 4095, 8192, 8193, want.size - 1, want.size, want.size + 7}):
        if cap < 0:
            continue
        for query in (env.fired, env.fired_noalloc):
            got, n = query(1, cap)
            assert n == want.size and np.array_equal(got, want[:cap])
    env.finalize()
