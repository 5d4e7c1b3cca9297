"""The device-side rows of download_evidence and download_labels against the same formulas in numpy, over
accumulators with zeros, ties, single votes and counts around the workgroup size."""
import ctypes as C

import numpy as np
import pytest

from b2ctrain_amd import _native

pytestmark = pytest.mark.gpu

BINS, STRIDE = 32, 8


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1000])
def test_export_rows(n):
    rng = np.random.default_rng(n)
    ev = (rng.random((n, STRIDE)) * rng.choice([0.0, 1.0, 1e-20, 1e6], (n, 1))).astype(np.float32)
    ev[::3, 7] = 0.0
    votes = np.where(rng.random((n, BINS)) < 0.2, rng.integers(0, 4, (n, BINS)), 0).astype(np.float32)  # ties
    votes[1::4] = 0.0
    votes[2::5, -1] = 7.5
    L = _native.lib()
    d_ev, d_lab = _native.DeviceArray(ev), _native.DeviceArray(votes)
    o_ev, o_lab = _native.DeviceArray(np.full((n, 7), np.nan, np.float32)), _native.DeviceArray(np.full((n, 2), np.nan, np.float32))
    _native.check(L.b2c_hip_evidence_export(n, C.c_void_p(d_ev.ptr), C.c_void_p(o_ev.ptr), None))
    _native.check(L.b2c_hip_label_export(n, C.c_void_p(d_lab.ptr), C.c_void_p(o_lab.ptr), None))
    with np.errstate(divide="ignore", invalid="ignore"):
        ratio = np.where(ev[:, 7] > 0, ev[:, 0] * ev[:, 0] / ev[:, 7], np.float32(0))
    want = np.concatenate([ev[:, :3], ratio[:, None], ev[:, 4:7]], 1).astype(np.float32)
    np.testing.assert_array_equal(o_ev.download(np.float32, (n, 7)), want)
    total = np.zeros(n, np.float32)
    for k in range(BINS):
        total = total + votes[:, k]
    win = votes.argmax(1)  # the first of equal votes
    lab = np.zeros((n, 2), np.float32)
    on = total > 0
    lab[on, 0] = win[on]
    lab[on, 1] = votes.max(1)[on] / total[on]
    np.testing.assert_array_equal(o_lab.download(np.float32, (n, 2)), lab)
