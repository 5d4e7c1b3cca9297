"""The small sorts of csrc/kernels/binning.hip: one workgroup (up to 4096 keys) at the edges of its waves and rounds, up to
64 tiles without a digit scan, and the change from 2048- to 4096-key tiles, against
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


@pytest.mark.parametrize("n", [4097, 6144, 6145, 131_071, 131_072, 131_073])
@pytest.mark.parametrize("begin,end,two", [(0, 32, False), (5, 18, True), (0, 8, False)])
def test_scatter_sums_the_tiles_before_it(n, begin, end, two):
    """Sorts of up to 64 tiles of 2048 keys have no digit scan; one key more has."""
    rng = np.random.default_rng(n + end)
    k, v, v2 = (rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3))
    k[rng.random(n) < 0.3] = 0xFFFFFFFF
    got, want = _sort(k, v, v2 if two else None, begin, end), _expect(k, v, v2 if two else None, begin, end)
    for g, w in zip(got, want):
        assert (g is None and w is None) or np.array_equal(g, w)


@pytest.mark.parametrize("n", [(5 << 19) - 1, 5 << 19, (5 << 19) + 4097])
@pytest.mark.parametrize("begin,end,two", [(0, 32, False), (0, 17, True)])
def test_both_sides_of_the_large_tiles(n, begin, end, two):
    """From 5 2^19 keys on a tile holds 4096 instead of 2048 of them, and 17 bits are two passes instead of three."""
    rng = np.random.default_rng(n + end)
    k, v, v2 = (rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3))
    got, want = _sort(k, v, v2 if two else None, begin, end), _expect(k, v, v2 if two else None, begin, end)
    for g, w in zip(got, want):
        assert (g is None and w is None) or np.array_equal(g, w)
