"""The range check of a map's entries on the device: sizes around a wave, a
workgroup and the whole grid, and maps on both sides of the size where the
check moves to the device."""
import numpy as np
import pytest

from pyop2_amd import device as dev, exceptions as ex, op2
from pyop2_amd.types import map as map_module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 65535, 65536, 65537, 300001])
def test_entry_range(device, n):
    rng = np.random.default_rng(n)
    v = rng.integers(-2 ** 31, 2 ** 31, n).astype(np.int32)
    for at in (0, n // 2, n - 1):
        w = v // 2
        w[at] = 2 ** 31 - 1
        assert dev.entry_range(dev.to_device(w)) == (w.min(), 2 ** 31 - 1)
        w[at] = -2 ** 31
        assert dev.entry_range(dev.to_device(w)) == (-2 ** 31, w.max())


@pytest.mark.parametrize("least", [1, 1 << 30])
def test_maps_on_both_sides(device, monkeypatch, least):
    monkeypatch.setattr(map_module, "_RANGE_ON_DEVICE", least)
    it, to = op2.Set(500), op2.Set(77)
    v = np.random.default_rng(5).integers(0, 77, (500, 3)).astype(np.int32)
    m = op2.Map(it, to, 3, v)
    assert not m.has_negative and np.array_equal(dev.to_host(m.device_values).reshape(v.shape), v)
    v[499, 2] = -1
    assert op2.Map(it, to, 3, v).has_negative
    v[0, 0] = 77
    m = op2.Map(it, to, 3, v)
    for _ in range(2):
        with pytest.raises(ex.MapValueError):
            m.device_values
    empty = op2.Map(op2.Set(0), to, 3, np.empty((0, 3), np.int32))
    assert not empty.has_negative and empty.device_values.numel() == 0
