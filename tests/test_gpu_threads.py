"""Networks called from threads of their own: the same results as alone, and runs side by
side where the networks fit the chip together."""
import threading
import time

import numpy as np
import pytest

from conftest import new_env
from test_gpu_resident import bits, small_env
from test_gpu_resident_runs import runs

pytestmark = pytest.mark.gpu

WINDOWS = 120


def quarter_env(pkg, seed, **options):
    env = new_env(pkg, 1, scale=0.25, burst_n_mf=12, seed=500 + seed, stim_seed=700 + seed)
    for k, v in options.items():
        env.set_option(k, v)
    return env


def together(jobs):
    """Seconds that the jobs, a thread each, take from a common start."""
    gate, errors = threading.Barrier(len(jobs) + 1), []

    def body(job):
        try:
            gate.wait()
            job()
        except Exception as e:  # noqa: BLE001 (reported by the test's own thread)
            errors.append(e)
    threads = [threading.Thread(target=body, args=(j,)) for j in jobs]
    for t in threads:
        t.start()
    gate.wait()
    t0 = time.perf_counter()
    for t in threads:
        t.join()
    assert not errors, errors
    return time.perf_counter() - t0


def windows(env, n=WINDOWS):
    def job():
        t = env.info().current_step
        for _ in range(n):
            env.loop_n_steps(t, 25)
            t += 25
    return job


def same_state(env, alone):
    for x, y in zip(env.state(), alone.state()):
        assert np.array_equal(bits(x), bits(y))
    assert np.array_equal(env.totals()[0], alone.totals()[0]) and env.totals()[1] == alone.totals()[1]


@pytest.mark.parametrize("make,fit,most", [
    (small_env, True, 1.6),     # 96 of 256 blocks each: side by side
    (quarter_env, False, 1.8),  # 224 each: step by step while the other is under way
], ids=["fit", "too_large"])
def test_two_networks_on_two_threads(pkg, make, fit, most):
    """Two networks on two threads take less than twice as long as one of them (one run after
    another: 2.0 to 2.1 times), and each of them gives what it gives alone."""
    envs = [make(pkg, k) for k in (1, 2)]
    alone = [make(pkg, k, resident=0) for k in (1, 2)]
    for e in envs + alone:
        e.initialize(50, 25)
    one = together([windows(envs[0])])
    before = [runs(e)[0] for e in envs]
    both = together([windows(e) for e in envs])
    resident = [runs(e)[0] - b for e, b in zip(envs, before)]
    assert all(runs(e)[1] == 0 for e in envs)
    assert sum(resident) == 2 * WINDOWS if fit else sum(resident) < 2 * WINDOWS
    windows(alone[0], 2 * WINDOWS)()
    windows(alone[1])()
    for e, a in zip(envs, alone):
        same_state(e, a)
        e.finalize()
        a.finalize()
    assert both < most * one


def test_batch_graphs_and_resident_runs_on_threads(pkg):
    """A batch, a network that replays graphs (captured meanwhile) and resident networks."""
    def nets():
        envs = [small_env(pkg, 11), small_env(pkg, 12, graph=1), quarter_env(pkg, 13), small_env(pkg, 14),
                small_env(pkg, 15)]
        for e in envs:
            e.initialize(50, 25)
        return envs

    envs, alone = nets(), nets()
    batch = pkg.Batch(envs[3:])

    def batch_job():
        for n in (25, 7, 100, 25, 60, 33):
            batch.run(n)

    def graph_job():
        t = 0
        for n in (25, 50, 30, 25, 120):
            envs[1].set_option("graph_steps", 25 if t % 2 else 10)  # captured again
            envs[1].loop_n_steps(t, n)
            t += n
    together([windows(envs[0]), graph_job, windows(envs[2]), batch_job])
    for e in (alone[0], alone[2]):
        windows(e)()
    for e, n in ((alone[1], 250), (alone[3], 250), (alone[4], 250)):
        e.loop_n_steps(0, n, want_output=False)
    for e, a in zip(envs, alone):
        same_state(e, a)
    batch.destroy()
    for e in envs + alone:
        e.finalize()
