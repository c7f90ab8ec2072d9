"""Resident runs (one launch per run, blocks that stay on their CUs) against the oracle:
rasters, state and output trains bit for bit, over layouts, run lengths and rings."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def small_env(pkg, seed, **options):
    """A 9.9k-cell scaffold with its own connectome and streams."""
    env = pkg.NetworkEnvironment(1, 7, 16, 2)
    cfg = pkg.synth_preset(0)
    cfg.seed = 100 + seed
    cfg.stim_seed = 900 + seed
    cfg.mf_rate_hz = 8.0
    env.describe_synthetic(cfg)
    for k, v in options.items():
        env.set_option(k, v)
    return env


def compare(env, ref, calls, T):
    ref.initialize()
    t = 0
    for n in calls:
        out = env.loop_n_steps(t, n)
        ref.run(t, n)
        R = env.info().ring_rows
        for s in range(max(t, t + n - R + 1), t + n):
            assert np.array_equal(env.spike_row(s), ref.spike_row(s)), f"raster differs at step {s}"
        t += n
        if (t // T) * T > t - n:  # the call completed a window
            last = (t // T) * T
            if last - T > t - R:
                n_out = out.shape[1]
                rows = np.stack([ref.spike_row(s) for s in range(last - T, last)])
                base = [env.population(i).base_id for i in range(env.info().n_populations)
                        if env.population(i).device_type == 2]
                assert np.array_equal(out, rows[:, base[0]:base[0] + n_out])
    for x, y in zip(env.state(), ref.state()):
        assert np.array_equal(bits(x), bits(y))
    assert env.totals()[0].sum() > 0


@pytest.mark.parametrize("options", [
    {},                                                      # default layout
    {"stage_spikes": 0},                                     # every spike word from the ring
    {"lane_max_fanin": 4096, "lane_synapses": 8},            # lanes wherever 3 slices suffice
    {"lane_max_fanin": 0, "lane_synapses": 64},              # teams only, narrow
    {"lane_synapses": 1},                                    # widest teams (a neuron per block)
    {"word_groups": 0, "index_bits": 16, "weight_precision": 2},
    {"index_bits": 16, "weight_precision": 1},
], ids=["default", "ring", "lanes", "teams", "wide", "fp8_idx16", "bf16_idx16"])
def test_layouts_bit_exact(pkg, orc, options):
    env = small_env(pkg, 1, **options)
    env.initialize(50, 25)
    compare(env, orc.OracleSim.from_env(env), [25, 25, 100], 25)
    env.finalize()


@pytest.mark.parametrize("T_print,T,calls", [
    (50, 25, [16, 9, 15, 17, 3, 1, 60, 26]),  # shortest runs, per-step calls between, short last runs
    (4, 2, [2, 8, 30, 5]),                    # a ring of 8 rows: no room for a run
    (12, 12, [12, 48, 7, 40]),                # runs as long as the ring allows
])
def test_run_lengths_and_rings_bit_exact(pkg, orc, T_print, T, calls):
    env = small_env(pkg, 2)
    env.initialize(T_print, T)
    compare(env, orc.OracleSim.from_env(env), calls, T)
    env.finalize()


def test_given_up_run_is_launched_again(pkg, orc):
    """Waits of one poll: the run is given up on the device, nothing of it is kept, and the
    same call launches its steps again."""
    env = small_env(pkg, 3, run_polls=0)
    env.initialize(50, 25)
    compare(env, orc.OracleSim.from_env(env), [25, 50, 20, 25], 25)
    env.finalize()


def test_two_networks_in_turn_bit_exact(pkg, orc):
    """Two environments on streams of their own, called in turn."""
    envs = [small_env(pkg, 4), small_env(pkg, 5, index_bits=16)]
    refs = []
    for e in envs:
        e.initialize(50, 25)
        r = orc.OracleSim.from_env(e)
        r.initialize()
        refs.append(r)
    for t in range(0, 100, 25):
        for e, r in zip(envs, refs):
            e.loop_n_steps(t, 25, want_output=False)
            r.run(t, 25)
    for e, r in zip(envs, refs):
        for x, y in zip(e.state(), r.state()):
            assert np.array_equal(bits(x), bits(y))
        e.finalize()
