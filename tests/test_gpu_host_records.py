"""Host records to the device and back, to the last byte, around the sizes
where the transfer takes pinned slots and where it needs another one."""
import numpy as np
import pytest

from raypier_optics_amd import _abi, _device
from raypier_optics_amd._device import DeviceRays, DeviceRaysView

pytestmark = pytest.mark.gpu


def _records(n, dt):
    """Every byte of every field random (finite or not: the copies are exact)."""
    a = np.frombuffer(np.random.default_rng(n).bytes(n * dt.itemsize), dt).copy()
    return a


@pytest.mark.parametrize("gausslet", [False, True])
@pytest.mark.parametrize("edge", [0.25, 1.0, 2.0, 3.0])
@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_records_round_trip(gpu, gausslet, edge, extra):
    dt = _abi.gausslet_dtype if gausslet else _abi.ray_dtype
    n = int(edge * _device._SLOT) // dt.itemsize + extra
    a = _records(n, dt)
    d = DeviceRays(n + 7, gausslet=gausslet)
    d.upload(a)
    back = d.download(n)
    assert back.dtype == dt and back.flags.owndata and back.flags.writeable
    assert back.tobytes() == a.tobytes()
    part = DeviceRaysView(d, 3, n - 3).download(n - 3)
    assert part.tobytes() == a[3:].tobytes()


@pytest.mark.parametrize("n", [10, 30000])
def test_read_only_and_strided_records(gpu, n):
    a = _records(2 * n, _abi.ray_dtype)
    b = a[::2]
    d = DeviceRays(n)
    d.upload(b)
    assert d.download(n).tobytes() == b.tobytes()
    b = a[:n].copy()
    b.flags.writeable = False
    d.upload(b)
    assert d.download(n).tobytes() == b.tobytes()


def test_records_with_a_default_device(gpu):
    """The pinned slots are host memory whatever torch's default device is."""
    a = _records(20000, _abi.ray_dtype)     # 3.8 MB
    d = DeviceRays(len(a))
    with gpu.device("cuda"):
        d.upload(a)
        assert d.download(len(a)).tobytes() == a.tobytes()
