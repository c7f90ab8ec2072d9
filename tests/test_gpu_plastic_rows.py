"""Teacher rules on rows shorter than a wavefront, whose synapses share wavefronts across
rows: some of a wavefront's rows triggered, none, all."""
import math

import numpy as np
import pytest

from test_gpu_resident import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per,n_rows", [(5, 301), (40, 130), (63, 65)])
@pytest.mark.parametrize("teacher_hz", [0.0, 20.0, 10000.0])
def test_teacher_rows_bit_exact(pkg, orc, per, n_rows, teacher_hz):
    n_pre = 200
    rng = np.random.default_rng(per)
    env = pkg.NetworkEnvironment(1, 3, 2, 2, 1)
    env.set_neuron_params(0, "cell", 0, n_rows, 10.0, -65.0, 2.0, 0.0, -70.0, -50.0, 1.0, pkg.NORMAL,
                          [1.0, 0.0, 0.1, 5.0])
    teach = env.set_neuron_params(1, "teach", 0, n_rows, 0, 0, 0, 0, 0, 0, 0, pkg.INPUT, [])
    pre = env.set_neuron_params(2, "pre", 0, n_pre, 0, 0, 0, 0, 0, 0, 0, pkg.INPUT, [])
    col = np.sort(np.stack([rng.choice(n_pre, per, replace=False) for _ in range(n_rows)]), axis=1).astype(np.int32)
    target = env.set_connectivity_csr(0, n_pre, n_rows, pre, 0, 0.02, 1.0,
                                      np.arange(0, n_rows * per + 1, per, dtype=np.int64),
                                      np.ascontiguousarray(col.reshape(-1)),
                                      rng.uniform(0.8, 1.2, n_rows * per).astype(np.float32))
    teacher = env.set_connectivity_csr(1, n_rows, n_rows, teach, 0, 0.02, 1.0, np.arange(n_rows + 1, dtype=np.int64),
                                       np.arange(n_rows, dtype=np.int32), None)
    for pop, n, hz, seed in ((teach, n_rows, teacher_hz, 5), (pre, n_pre, 60.0, 9)):
        f = pkg.StimFunc()
        f.poisson_hz, f.poisson_on, f.poisson_off, f.seed = hz, 0.0, math.inf, seed
        env.set_input_stim_ids(pop, np.arange(n), f)
    coefficients = {pkg.A1_J: 0.0, pkg.A2_JI: -0.01}
    env.set_plasticity(rule=pkg.STDP_TEACHER, target=target, teacher=teacher, coefficients=coefficients,
                       time_window=50)
    before = env.projection_csr(target)[2].copy()
    env.initialize(50, 25)
    ref = orc.OracleSim.from_env(env)
    ref.initialize()
    ref.add_plasticity(pkg.STDP_TEACHER, target, teacher, coefficients, 50, env.projection(target).grid_exp)
    env.loop_n_steps(0, 120, want_output=False)
    ref.run(0, 120)
    after = env.projection_csr(target)[2]
    assert np.array_equal(bits(after), bits(ref.multipliers(target)))
    assert np.array_equal(after, before) == (teacher_hz == 0.0)
    for x, y in zip(env.state(), ref.state()):
        assert np.array_equal(bits(x), bits(y))
    env.finalize()
