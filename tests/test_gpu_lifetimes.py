"""Contexts, batches and downloads against the order in which a program gives them up."""
import numpy as np
import pytest

import lbdem
import workloads

pytestmark = pytest.mark.gpu


def _small(lib, seed, steps=12):
    run = workloads.random_impact_run(np.random.default_rng(seed), (32,), 60, relax=60)
    sim = lbdem.Simulation(lib, lbdem.params_from_values(run.values, lbdem.PREC_FP32), run.particles, run.objects)
    sim.init()
    sim.set_tile(8)
    sim.cycle(steps)
    return sim


def test_member_destroyed_before_its_batch(gpu_lib):
    """The batch refuses further steps, its end touches the remaining members only, and those go on alone
    with the results of a run that was never in a batch (tolerances of test_pool)."""
    ref, a, b = _small(gpu_lib, 3), _small(gpu_lib, 3), _small(gpu_lib, 4)
    batch = lbdem.Batch(gpu_lib, [a, b])
    batch.cycle(10)
    b.close()
    with pytest.raises(lbdem.LbdemError, match="destroyed"):
        batch.cycle(2)
    with pytest.raises(lbdem.LbdemError, match="destroyed"):
        batch.set_tile(4)
    batch.synchronize()
    batch.close()
    a.cycle(9)
    ref.cycle(19)
    for x, y in ((a.objects(), ref.objects()), (a.walls(), ref.walls())):
        assert np.abs(x - y).max() <= 1e-9 * np.abs(y).max()
    assert a.info()["nActive"] == ref.info()["nActive"] and a.info()["lbTime"] == 31
    a.close()
    ref.close()
