"""Fields to the host in one piece, in several with a ragged last one, and
without device memory for a staging buffer: the same bytes, and what the buffer
holds is counted."""
import numpy as np
import pytest

from test_adv2d_resident_gpu import _model as adv2d_model
from test_hpe_gpu import _pair as hpe_pair
from test_sw2d_resident_gpu import _model as sw2d_model

pytestmark = pytest.mark.gpu


def _sw2d():
    m = sw2d_model(N=5, nX=9, nY=7, precision="fp64")
    m.ForwardStepRK3(0.0, 1)
    return m


def _adv2d():
    return adv2d_model(N=4, nX=9, nY=7, nq=3)


def _hpe():
    m = hpe_pair(dict(N=3, n=(3, 2, 5), periodic=(False, True), warp=0.02, dp=True), dt=2e-3)[1]
    m.ForwardStepRK3(1)
    return m


@pytest.mark.parametrize("make", [_sw2d, _adv2d, _hpe])
def test_every_way_gives_the_same_bytes(gpu_lib, make, monkeypatch):
    m = make()
    monkeypatch.setenv("SELF_AMD_STAGE_DOUBLES", "0")
    want = m.GetSolution()
    assert np.isfinite(want).all() and want.any()
    for most in ("1", "700", "1000000"):  # an element a piece, a few, all
        monkeypatch.setenv("SELF_AMD_STAGE_DOUBLES", most)
        assert np.array_equal(m.GetSolution(), want), most
    monkeypatch.delenv("SELF_AMD_STAGE_DOUBLES")
    assert np.array_equal(m.GetSolution(), want)


def test_device_bytes_count_the_staging_buffer(gpu_lib, monkeypatch):
    m = _sw2d()
    before = m.DeviceBytes()
    monkeypatch.setenv("SELF_AMD_STAGE_DOUBLES", "0")
    n = m.GetSolution().nbytes
    assert m.DeviceBytes() == before
    monkeypatch.delenv("SELF_AMD_STAGE_DOUBLES")
    m.GetSolution()
    assert m.DeviceBytes() == before + n
