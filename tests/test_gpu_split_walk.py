"""Split storage: the kick walk, with the limits, the potential and the fold in its
launches, rounds what the fused step's cell passes store, so that a small disk's
fields are the same bit for bit through either; on grids at the edges of the walk's
59-sector segments and of its tiles, Euler and LeapFrog, each rounding mode, stepwise
and in graphs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ["SIGMA", "VRAD", "VAZI", "ENERGY", "PRESSURE", "SOUNDSPEED", "SCALE_HEIGHT",
          "VISCOSITY", "TEMPERATURE", "QPLUS", "QMINUS", "POTENTIAL"]


def _disk(name, nr, nphi, integrator, tile, rounding):
    import dataclasses
    from fargocpt_amd import workloads as W
    from fargocpt_amd.capi import Disk
    from fargocpt_amd.ic import initial_state, log_radii
    cfg = W.disk_config(name, 1)
    cfg.update({"nr": nr, "nphi": nphi, "radii": log_radii(nr, cfg["rmin"], cfg["rmax"]), "integrator": integrator})
    d = Disk(cfg)
    ic = initial_state(dataclasses.replace(W.setup(name), nr=nr, nphi=nphi))
    d.upload_reference(ic["sigma"], ic["vrad"], ic["vazi"], ic["energy"])
    d.upload_state(ic["sigma"], ic["vrad"], ic["vazi"], ic["energy"])
    d.set_time(0.0, 0.1, 0)
    d.calculate_timestep()
    d.set_step_params(*W.planet_inputs(name))
    d.set_split_rounding(rounding)
    d.set_kick_tile(tile)
    return d


@pytest.mark.parametrize("rounding", [0, 1, 2])
@pytest.mark.parametrize("integrator", [0, 1])
@pytest.mark.parametrize("name", ["iso_128x384", "adi_512x1536", "adi_beta_4096x12288"])
def test_walk_rounds_as_passes(name, integrator, rounding):
    for nr, nphi in ((8, 4), (25, 59), (26, 60), (40, 97), (67, 119)):
        print(f"{name} {nr} x {nphi} integrator {integrator} rounding {rounding}", flush=True)
        a, b = (_disk(name, nr, nphi, integrator, t, rounding) for t in (0, 1))
        a.run_steps(9)
        for _ in range(9):
            b.run_step()
        # the limits and the force between steps read the fields as the last step rounded them
        assert a.calculate_timestep() == b.calculate_timestep()
        for d in (a, b):
            d.run_step()
        bodies = [(0.0, 0.0, 0.0, 0.0), (1.0, 0.1, 1.005, 0.0)]
        assert np.array_equal(a.disk_on_planet_accel(bodies), b.disk_on_planet_accel(bodies))
        assert a.calculate_timestep() == b.calculate_timestep()
        assert a.get_time() == b.get_time()
        for f in FIELDS:
            x, y = a.download_field(f), b.download_field(f)
            assert np.array_equal(x, y), (nr, nphi, f, float(np.max(np.abs(x - y))))
