"""The one-workgroup sort (up to 4096 keys, csrc/kernels/binning.hip) at the edges of its waves and rounds, against
numpy's stable argsort; the same keys with a second value array take the general passes and must agree too."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_sort import _expect, _sort


@pytest.mark.parametrize("n", [1, 63, 65, 255, 257, 1200, 4095, 4096, 4097])
@pytest.mark.parametrize("begin,end", [(0, 32), (3, 14), (0, 1), (24, 32)])
@pytest.mark.parametrize("keys", ["rand", "dup", "culled"])
def test_one_workgroup_sort(n, begin, end, keys):
    rng = np.random.default_rng(n * 37 + begin)
    k = rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)
    if keys == "dup":
        k &= np.uint32(0x01010109)
    elif keys == "culled":
        k[rng.random(n) < 0.8] = 0xFFFFFFFF
    v, v2 = (rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(2))
    for vals in (v, None):
        ko, vo, _ = _sort(k, vals, None, begin, end)
        ek, ev, _ = _expect(k, vals, None, begin, end)
        assert np.array_equal(ko, ek) and np.array_equal(vo, ev)
    ko, vo, v2o = _sort(k, v, v2, begin, end)
    ek, ev, ev2 = _expect(k, v, v2, begin, end)
    assert np.array_equal(ko, ek) and np.array_equal(vo, ev) and np.array_equal(v2o, ev2)
