"""The transport's sweeps (radial and azimuthal in one walk) against the
oracle's separate loops, in FP64 storage.

Grids at the edges of the walk's 57-sector segments and of its ring tiles, the
smallest grid, disks small enough for one quantity per block; shifts in both
directions beyond the ring, uniform residuals of both signs on neighbouring
rings; Sigma and E outside the range of the shared reciprocals; an infinite E.

The sweeps' expressions are the oracle's, so only the order of the ring's
v_phi sum differs: the mean moves by at most n 2^-53 of itself (2e-14 at 177
sectors), the residual velocity by that times |v_phi|, and the transported
values by the fraction of a cell that this crosses, below 1e-12 of the largest
here (|v_phi| dt < 2.1 rings of 177 cells).  Bound: 1e-10.
"""
import numpy as np
import pytest

from fixtures import disk_config, load_case
from oracle import OracleDisk

pytestmark = pytest.mark.gpu
DT = 0.01


def _state(nr, ns, rmed, scale):
    rng = np.random.default_rng(nr * 1000 + ns)
    sigma = scale * (1.0 + 0.5 * rng.random((nr, ns)))
    width = np.diff(rmed).min()
    vrad = 0.4 * width / DT * rng.uniform(-1.0, 1.0, (nr + 1, ns))
    vrad[nr // 2] = 0.0
    dphi = 2 * np.pi / ns
    shift = (np.arange(nr) % 5 - 2) * ns + rng.uniform(-0.5, 0.5, nr)
    vazi = (rmed * dphi / DT)[:, None] * (shift[:, None] + 0.3 * rng.uniform(-1.0, 1.0, (nr, ns)))
    energy = sigma * (1e-3 + 1e-3 * rng.random((nr, ns)))
    return sigma, vrad, vazi, energy


def _check(case, nr, ns, tile, scale=1.0, bad=None):
    from fargocpt_amd.capi import Disk
    meta, _ = load_case(case)
    cfg = disk_config(dict(meta, Nr=nr, Nphi=ns))
    print(f"{case} {nr} x {ns} tile {tile} Sigma scaled by {scale} {bad}", flush=True)
    gpu, cpu = Disk(cfg), OracleDisk(cfg)
    gpu.set_radial_tile(tile)
    st = _state(nr, ns, cpu.geom("Rmed", nr), scale)
    if bad is not None:
        st[3][nr // 2, ns // 2] = bad
    for d in (gpu, cpu):
        d.upload_state(*st)
        d.transport(DT)
    assert np.array_equal(gpu.nshift(), cpu.nshift())
    for f in ("SIGMA", "VRAD", "VAZI") + (("ENERGY",) if meta["adiabatic"] else ()):
        x, y = gpu.download_field(f), cpu.download_field(f)
        ok = np.isfinite(y)
        assert np.array_equal(np.isfinite(x), ok), f
        assert np.max(np.abs(x[ok] - y[ok])) <= 1e-10 * np.max(np.abs(y[ok])), f
    gpu.close()
    cpu.close()


@pytest.mark.parametrize("case", ["c1_small", "c2_small"])
@pytest.mark.parametrize("nr,ns,tile", [(8, 4, 0), (9, 56, 2), (10, 57, 3), (11, 58, 11), (33, 114, 0), (67, 115, 64),
                                        (40, 177, 1), (70, 171, 5)])
def test_segments_and_tiles(case, nr, ns, tile):
    _check(case, nr, ns, tile)


@pytest.mark.parametrize("scale", [2.0 ** -99, 2.0 ** -110, 2.0 ** 99, 2.0 ** 112])
def test_quotients_out_of_range(scale):
    for case in ("c1_small", "c2_small"):
        _check(case, 24, 97, 4, scale=scale)


def test_infinite_energy():
    _check("c2_small", 24, 97, 4, bad=np.inf)
