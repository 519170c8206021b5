"""Derived fields that a fused step has left to be formed are stored before
anything reads them: a change of a launch parameter, a batch whose plan differs
from the disk's own step, the disk's force.  Against the separate kernels, bit
for bit in FP64 storage.
"""
import numpy as np
import pytest

from test_gpu_kick_walk import _disk, _same

pytestmark = pytest.mark.gpu

NAMES = {"iso": "iso_128x384", "adi": "adi_512x1536"}
BODIES = [(0.0, 0.0, 0.0, 0.0), (1.0, 0.1, 1.005, 0.0)]
CHANGES = {"fused": lambda d: d.set_fused_step(False), "kick": lambda d: d.set_kick_tile(1),
           "visc": lambda d: d.set_visc_tile(1)}


def _pair(physics, integrator=0):
    return [_disk(NAMES[physics], 40, 97, integrator, fused=f) for f in (True, False)]


def _force(a, b):
    assert np.array_equal(a.disk_on_planet_accel(BODIES), b.disk_on_planet_accel(BODIES))


@pytest.mark.parametrize("change", list(CHANGES))
@pytest.mark.parametrize("integrator", [0, 1])
@pytest.mark.parametrize("physics", ["iso", "adi"])
def test_parameter_after_steps(physics, integrator, change):
    for how in ("run_step", "run_steps"):
        print(f"{physics} integrator {integrator} {change} {how}", flush=True)
        a, b = _pair(physics, integrator)
        for d in (a, b):
            d.run_steps(5)
        CHANGES[change](a)
        _force(a, b)
        for d in (a, b):
            if how == "run_step":
                for _ in range(3):
                    d.run_step()
            else:
                d.run_steps(3)
        _same(a, b, (physics, integrator, change, how))
        assert a.get_time() == b.get_time()


@pytest.mark.parametrize("change", list(CHANGES))
@pytest.mark.parametrize("physics", ["iso", "adi"])
def test_parameter_before_batch(physics, change):
    """A batch runs the step it was planned with, whatever the disk's own
    parameters are by then."""
    from fargocpt_amd.capi import Batch
    print(f"{physics} {change}", flush=True)
    a, b = _pair(physics)
    batch = Batch([a])
    CHANGES[change](a)
    batch.run_steps(5)
    b.run_steps(5)
    _force(a, b)
    for d in (a, b):
        d.run_steps(3)
    _same(a, b, (physics, change))
    batch.close()


@pytest.mark.parametrize("physics", ["iso", "adi"])
def test_batch_of_separate_passes(physics):
    """A member planned with the kick as separate passes, stepped alone by the
    walk before the batch reads its fields."""
    from fargocpt_amd.capi import Batch
    print(physics, flush=True)
    a, b = _pair(physics)
    a.set_kick_tile(1)
    batch = Batch([a])
    a.set_kick_tile(0)
    for n in (4, 3):
        a.run_steps(n)
        batch.run_steps(n)
        batch.synchronize()
        b.run_steps(2 * n)
        _force(a, b)
    _same(a, b, physics)
    batch.close()


@pytest.mark.parametrize("field", ["PRESSURE", "ENERGY", "SCALE_HEIGHT"])
def test_autotune_keeps_uploaded_field(field):
    """The autotuner's trials leave the next step a field of the caller's own
    to read."""
    print(field, flush=True)
    disks = [_disk(NAMES["adi"], 40, 97, fused=f) for f in (True, True, False)]
    for d in disks:
        d.run_steps(3)
        d.upload_field(field, d.download_field(field) * 1.01)
    disks[0].autotune_walks(2)
    for d in disks:
        d.run_steps(3)
    _same(disks[1], disks[2], field)
    _same(disks[0], disks[2], field)


@pytest.mark.parametrize("integrator", [0, 1])
@pytest.mark.parametrize("how", ["pressure", "damping"])
def test_own_fields_keep_the_fused_passes(integrator, how):
    """A step that reads the fields as the caller left them is still a fused
    one: the tensors that only the separate kernels store keep their marks."""
    print(f"integrator {integrator} {how}", flush=True)
    a, b = _pair("adi", integrator)
    for d in (a, b):
        d.run_step()
        if how == "pressure":
            d.upload_field("PRESSURE", d.download_field("PRESSURE") * 1.01)
        else:
            d.apply_boundary_condition(1e-3, True)
    mark = np.full((40, 97), 7.0)
    for f in ("Q_R", "Q_PHI"):
        a.upload_field(f, mark)
    for d in (a, b):
        d.run_step()
    for f in ("Q_R", "Q_PHI"):
        assert np.array_equal(a.download_field(f), mark), f
    _same(a, b, (integrator, how))
