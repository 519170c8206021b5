"""A batch whose members have fields of their caller's own: the host waits no more
often than for any other batched run (tests/cpp/batch_check counts), and the
members' fields are those of disks stepped alone, bit for bit."""
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "batch_check.bin")


@pytest.mark.parametrize("name", ["iso_128x384", "adi_512x1536"])
def test_host_waits(tmp_path, name):
    from fargocpt_amd import workloads as W
    from fargocpt_amd.capi import desc_from_dict
    from fargocpt_amd.ic import initial_state
    assert os.path.exists(EXE), "build tests/cpp/batch_check with __graft_entry__.build()"
    desc, radii = desc_from_dict(W.disk_config(name))
    (tmp_path / "desc.bin").write_bytes(bytes(desc))
    radii.tofile(str(tmp_path / "radii.bin"))
    ic = initial_state(W.setup(name))
    for f in ("sigma", "vrad", "vazi", "energy"):
        ic[f].tofile(str(tmp_path / f"{f}.bin"))
    print(name, flush=True)
    r = subprocess.run([EXE, str(tmp_path), "3"], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert [int(w) for w in r.stdout.split()] == [3, 3, 3]  # one per member


@pytest.mark.parametrize("field", ["SIGMA", "PRESSURE", "ENERGY"])
def test_fields(field):
    from fargocpt_amd.capi import Batch
    from test_gpu_kick_walk import _disk, _same
    print(field, flush=True)
    names = ["iso_128x384", "adi_512x1536", "adi_beta_4096x12288"]
    alone, batched = ([_disk(n, 40 + k, 97) for k, n in enumerate(names)] for _ in range(2))
    batch = Batch(batched)
    for n in (3, 2):
        batch.run_steps(n)
        for d in alone:
            d.run_steps(n)
        for disks in (alone, batched):
            for d in disks[:2]:
                d.upload_field(field, d.download_field(field) * 1.01)
    batch.run_steps(4)
    for a, b in zip(alone, batched):
        a.run_steps(4)
        _same(a, b, field)
        assert a.get_time() == b.get_time()
    batch.close()
