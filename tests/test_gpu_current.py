"""The one-launch current update on grids that need not be periodic against
the stages it stands for (guard add, guard copy, filter), bit for bit, on
random deposits with inconsistent guards: tiles down to the narrowest it
takes, filters on both sides of the register form's limit of five passes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ENDS = {"periodic": ("periodic", "periodic"), "none": ("none", "none")}


@pytest.mark.parametrize("x", ENDS)
@pytest.mark.parametrize("y", ENDS)
@pytest.mark.parametrize("ntiles,nx,filt", [
    ((1, 1), (3, 3), None),
    ((3, 2), (16, 16), None),
    ((1, 3), (4, 5), ("binomial", 0, 1)),
    ((3, 1), (8, 7), ("compensated", 0, 4)),     # 5 passes, the narrowest tile
    ((4, 3), (17, 6), ("binomial", 0, 5)),
    ((2, 2), (9, 4), ("compensated", 0, 5)),     # 6 passes
    ((2, 3), (30, 9), ("binomial", 0, 2)),
    ((70, 60), (4, 3), ("binomial", 0, 1)),      # more tiles than workgroups of one tile each
])
def test_current_update_matches_stages(ntiles, nx, filt, x, y):
    import pyzpic as zp
    rng = np.random.default_rng(3)
    out = []
    J = None
    for one in (True, False):
        sim = zp.Simulation(ntiles, nx, (ntiles[0] * nx[0] * 0.1, ntiles[1] * nx[1] * 0.1), 0.05, filter=filt)
        sim.set_current_bc(ENDS[x], ENDS[y])
        if J is None:
            J = rng.normal(0, 1, (sim.ntiles * sim.geom.tile_vol, 3)).astype(np.float32)
        sim.set_field("J", J)
        for stage in (("current",) if one else ("add_gc", "copy_gc", "filter")):
            sim.stage(stage)
        out.append(sim.field("J"))
        sim.close()
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
