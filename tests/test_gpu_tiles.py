"""The tile that a run reports against the same tile fixed by the caller, with 2-byte storage, where the
number of nodes that share one 32-bit particle sum shows in the results."""
import numpy as np
import pytest

import lbdem
import workloads

pytestmark = pytest.mark.gpu

# the same sums of nodes in 32 bits, added in FP64 in an order that atomics decide, differ by less than
# 1e-12 of the largest force (thousands of terms); sums over other groups of nodes by some 1e-8
SAME = 1e-12


def _forces(sim):
    return sim.particles()[:, 9:15]


def _close(a, b):
    return np.abs(a - b).max() <= SAME * np.abs(b).max()


def test_fixed_tile_repeats_a_tuned_run(gpu_lib):
    """A run whose walk the timing picked, and a run that fixes the tile the first one reports; before that it
    runs the walks that the tuner times, in its order."""
    v, ps, obs = workloads.impact_box(**workloads.HEADLINE)
    a, b = (lbdem.Simulation(gpu_lib, lbdem.params_from_values(v, lbdem.PREC_FP16), ps, obs) for _ in range(2))
    a.init()
    b.init()
    assert a.info()["lbTime"] == 0
    a.cycle(8)
    for z in (8, 4, 2, 1):
        b.set_tile(z)
        b.cycle(2)
    assert _close(_forces(a), _forces(b))
    a.cycle(1)  # the pick
    t = a.tuning()
    assert t["tuned"]
    b.set_tile(t["tile"][2])
    assert b.tuning()["tile"] == t["tile"]
    b.cycle(1)
    a.cycle(3)
    b.cycle(3)
    print("picked", t, flush=True)
    assert _close(_forces(a), _forces(b))
    a.close()
    b.close()


@pytest.mark.parametrize("size", [(70, 64, 62), (256, 200, 200)])
def test_batch_tile_repeats_alone(gpu_lib, size):
    """A batch that times its walk gives each member what it has alone with the tile that the batch reports,
    whichever walk was the fastest; on either side of the size at which a fixed tile of two changes its walk."""
    X, Y, Z = size
    v, ps, obs = workloads.impact_box(size=size, fluid_height=0.75 * Y, n_spheres=X * Y * Z // 6000, r=4.0, r_imp=8.0,
                                      y_imp=0.75 * Y + 4.0, speed=0.01, relax=60, bed_top=0.75 * Y - 6.0)
    sims = []
    for _ in range(2):
        s = lbdem.Simulation(gpu_lib, lbdem.params_from_values(v, lbdem.PREC_FP16), ps, obs)
        s.init()
        s.set_tile(8)
        s.cycle(4)
        sims.append(s)
    batch = lbdem.Batch(gpu_lib, sims[:1])
    batch.set_tile(0)
    batch.cycle(8)
    tile = batch.tile()
    assert tile["tuned"]
    batch.synchronize()
    batch.close()
    sims[1].set_tile(tile["tileZ"])
    sims[1].cycle(8)
    print("batch tile", tile, flush=True)
    assert _close(_forces(sims[0]), _forces(sims[1]))
    sims[0].cycle(2)  # alone again, on the batch's tile
    sims[1].cycle(2)
    assert sims[0].tuning()["tile"] == sims[1].tuning()["tile"]
    assert _close(_forces(sims[0]), _forces(sims[1]))
    for s in sims:
        s.close()
