"""Names that programs time kernels by: the radial and the azimuthal sweep run as
one kernel, and both names, with the combined one, time it."""
import pytest

from fargocpt_amd import capi
from fargocpt_amd import workloads as W


@pytest.mark.parametrize("kernels", [capi.KERNELS, capi.BATCH_KERNELS])
def test_sweep_names(kernels):
    assert kernels["radial_sweep"] == 0 and kernels["azimuthal_sweep"] == 1 and kernels["sweeps"] == 0
    assert "radial_sweep" in kernels and kernels.get("azimuthal_sweep") == 1
    # one entry per kernel that can be timed
    assert [k for k in kernels if "sweep" in k] == ["sweeps"]
    assert "stress" not in kernels and kernels.get("stress") is None
    with pytest.raises(KeyError):
        kernels["stress"]


def test_sweep_bytes():
    for adiabatic in (False, True):
        for element in (4, 8):
            want = W.algorithmic_bytes("sweeps", adiabatic, element)
            assert W.algorithmic_bytes("radial_sweep", adiabatic, element) == want
            assert W.algorithmic_bytes("azimuthal_sweep", adiabatic, element) == want
