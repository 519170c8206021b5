"""Fields to the host: the single-kernel copy below and above the size from
which several threads move it, and the pieced copy above the staging slots,
with pieces that end inside rows, for both storages; two disks at once from
two threads; and copies after every other disk is gone (the slots with it).

FP64 storage returns what was uploaded bit for bit; split storage within the
FP32 rounding of the deviation from the ring mean, and the same values through
every route (a field alone, the state as a whole).
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("SIGMA", "VRAD", "VAZI", "ENERGY")


def _disk(nr, nphi, precision):
    from fargocpt_amd import workloads as W
    from fargocpt_amd.capi import Disk
    from fargocpt_amd.ic import log_radii
    cfg = W.disk_config("adi_512x1536", precision)
    cfg.update({"nr": nr, "nphi": nphi, "radii": log_radii(nr, cfg["rmin"], cfg["rmax"])})
    return Disk(cfg)


def _upload(d, nr, nphi, seed):
    rng = np.random.default_rng(seed)
    x = [1.0 + 0.1 * rng.standard_normal((nr + (f == "VRAD"), nphi)) ** 2 for f in FIELDS]
    d.upload_state(*x)
    return x


def _check(x, got, precision):
    for f, a, b in zip(FIELDS, x, got):
        if precision == 0:
            assert np.array_equal(a, b), f
        else:
            dev = np.abs(a - a.mean(axis=1, keepdims=True))
            assert np.all(np.abs(b - a) <= 1.01 * (2.0 ** -24 * dev + 2.0 ** -52 * np.abs(a))), f


# state sizes: 34 KB, 0.98 MB and 1.05 MB (one buffer / the slots), 48 MB from
# below and above (one kernel / pieces), 130 MB (more pieces than slots)
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nr,nphi", [(8, 131), (101, 303), (105, 313), (1001, 1571), (1001, 1573), (1999, 2039)])
def test_state_and_fields(nr, nphi, precision):
    print(f"{nr} x {nphi} precision {precision}", flush=True)
    d = _disk(nr, nphi, precision)
    x = _upload(d, nr, nphi, 3)
    got = d.download_state()
    _check(x, got, precision)
    for f, b in zip(FIELDS, got):
        assert np.array_equal(d.download_field(f), b), f
    d.close()


def test_two_threads():
    sizes = [(1001, 1573), (301, 701)]
    disks = [_disk(nr, nphi, k) for k, (nr, nphi) in enumerate(sizes)]
    xs = [_upload(d, nr, nphi, 5 + k) for k, (d, (nr, nphi)) in enumerate(zip(disks, sizes))]
    got = [[], []]

    def work(k):
        for _ in range(4):
            got[k].append(disks[k].download_state())

    threads = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in (0, 1):
        for g in got[k]:
            _check(xs[k], g, k)
    for d in disks:
        d.close()
    test_state_and_fields(101, 303, 0)
