"""The CFL limits with the potential in one launch and their fold inside the
kick walk, against the separate kernels: the same time steps and fields, bit
for bit in FP64 storage, where the rings fill a wavefront's lanes, leave a
remainder, are the most the walk folds (512) and one more; with the monitor
clip, after a boundary call of the caller's, and with a limit that is not finite.
"""
import numpy as np
import pytest

from test_gpu_kick_walk import FIELDS, _disk

pytestmark = pytest.mark.gpu


def _steps(d, n=4):
    d.apply_boundary_condition(0.0, False)
    return [d.run_step() for _ in range(n)]


@pytest.mark.parametrize("name", ["iso_128x384", "adi_512x1536", "adi_beta_4096x12288"])
@pytest.mark.parametrize("nr,nphi", [(8, 4), (64, 13), (65, 70), (511, 12), (512, 12), (513, 12)])
def test_folds_and_potential(name, nr, nphi):
    for integrator in (0, 1):
        print(f"{name} {nr} x {nphi} integrator {integrator}", flush=True)
        a = _disk(name, nr, nphi, integrator)
        b = _disk(name, nr, nphi, integrator, fused=False)
        assert _steps(a) == _steps(b)
        assert a.get_time() == b.get_time()
        for f in FIELDS + ["POTENTIAL"]:
            assert np.array_equal(a.download_field(f), b.download_field(f)), f


def test_monitor_clip():
    """Steps that end on a monitor time, one at a time and in a graph."""
    disks = [_disk("iso_128x384", 40, 60, fused=f) for f in (True, True, False)]
    for d in disks:
        d.set_time(0.0, 1e3, 0)
    for _ in range(24):
        disks[0].run_step()
        disks[2].run_step()
    disks[1].run_steps(24, True)
    times = [d.get_time() for d in disks]
    assert times[0] == times[1] == times[2] and times[0][2] > 0
    for f in ("SIGMA", "VRAD", "VAZI"):
        x = [d.download_field(f) for d in disks]
        assert np.array_equal(x[0], x[2]) and np.array_equal(x[1], x[2]), f


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_limit_not_finite(value):
    """An infinite velocity makes the limit zero (an error); a NaN one is no
    limit at all.  As the separate kernels."""
    seen = []
    for fused in (True, False):
        d = _disk("iso_128x384", 40, 60, fused=fused)
        v = d.download_field("VRAD")
        v[20, 30] = value
        d.upload_field("VRAD", v)
        try:
            seen.append(d.run_step())
        except RuntimeError as e:
            seen.append(str(e))
        d.close()
    assert seen[0] == seen[1]
