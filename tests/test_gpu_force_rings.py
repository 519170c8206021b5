"""The disk's pull on the bodies, one block per ring, where a ring has fewer
sectors than the block has threads, as many, one more, and two rounds and a
remainder, for one and for the most bodies; and the clock of a step, which the
step's last kernel writes to the host, against the one read from the device.
The bound is that of test_gpu_force.py (summation order only).
"""
import numpy as np
import pytest

from fixtures import disk_config, initial_condition, load_case
from test_gpu_force import FP64_TOL, _check_against_oracle

pytestmark = pytest.mark.gpu


def _disk(case, nr, ns, integrator=0, fused=True):
    from fargocpt_amd.capi import Disk
    meta, _ = load_case(case)
    meta = dict(meta, Nr=nr, Nphi=ns)
    cfg = dict(disk_config(meta), integrator=integrator)
    d = Disk(cfg)
    d.set_fused_step(fused)
    ic = initial_condition(dict(meta))
    rng = np.random.default_rng(ns)
    ic["sigma"] = ic["sigma"] * (1.0 + 0.3 * rng.random((nr, ns)))
    d.upload_reference(ic["sigma"], ic["vrad"], ic["vazi"], ic["energy"])
    d.upload_state(ic["sigma"], ic["vrad"], ic["vazi"], ic["energy"])
    return d, cfg, meta


@pytest.mark.parametrize("case", ["c1_small", "c2_small"])
@pytest.mark.parametrize("nr,ns", [(8, 4), (9, 255), (10, 256), (11, 257), (20, 515)])
def test_ring_remainders(case, nr, ns):
    from fargocpt_amd.capi import FORCE_CORRECT_SELFGRAVITY
    d, cfg, meta = _disk(case, nr, ns)
    for n in (1, 8):
        bodies = [(0.0, 0.0, 0.0, 0.0)] + [(0.4 + 0.2 * k, 0.1 * k, float(np.hypot(0.4 + 0.2 * k, 0.1 * k)), 0.05 * k)
                                           for k in range(1, n)]
        for flags in (0, FORCE_CORRECT_SELFGRAVITY):
            _check_against_oracle(d, cfg, bodies, flags, meta["G"], meta["thickness_smoothing"], FP64_TOL,
                                  f"{case} {nr} x {ns}, {n} bodies, flags {flags}")
    d.close()


@pytest.mark.parametrize("integrator,fused", [(0, True), (0, False), (1, True), (1, False)])
def test_step_reports_its_clock(integrator, fused):
    d, _, _ = _disk("c2_small", 16, 48, integrator, fused)
    print(f"integrator {integrator} fused {fused}", flush=True)
    d.set_time(0.0, 1e-3, 0)
    d.set_step_params([(0.0, 0.0, 1.0, 0.0), (0.8, 0.3, 1e-3, 0.0)])
    for _ in range(3):
        before = d.get_time()[0]
        dt = d.run_step()
        assert dt > 0.0 and d.get_time()[0] == before + dt
    d.close()
