"""The sizes at which a kernel or a rule of a dispatch can go wrong: edges of tiles, remainders, both sides of a
threshold - against the oracle or numpy."""
import numpy as np
import pytest

from comet_amd import gen
from comet_amd import runtime as rt
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, scope="module")
def _device():
    rt.init(0)


@pytest.mark.parametrize("nbytes", [1, 512, 513, 8192, 8193, 1 << 20, (1 << 20) + 8, 37_000_001])
def test_freed_blocks_come_back_only_when_nothing_uses_them(nbytes):
    a = rt.DeviceArray(nbytes, np.uint8)
    a.free()
    b, c = rt.DeviceArray(nbytes, np.uint8), rt.DeviceArray(nbytes, np.uint8)
    assert b.ptr != c.ptr
    ones, twos = np.full(nbytes, 1, np.uint8), np.full(nbytes, 2, np.uint8)
    for d, v in ((b, ones), (c, twos)):
        rt._check(rt.lib().comet_hip_memcpy(d.ptr, rt._vptr(v), nbytes, 0))
    assert np.array_equal(b.to_numpy(), ones) and np.array_equal(c.to_numpy(), twos)
    old = b.ptr
    b.free()
    assert rt.lib().comet_hip_free(old) != 0          # a second time
    assert np.array_equal(c.to_numpy(), twos)
