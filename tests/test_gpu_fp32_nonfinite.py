"""The fp32 backward on a pixel whose alpha gradient is infinite: the quotient Q / (1 - alpha) of an infinite remainder is
infinite, as a division gives it, so the opacity gradients of the pixel's splats are infinite with its sign and not NaN,
and those of all other splats zero."""
import numpy as np
import pytest

from b2ctrain_amd import _native
from b2ctrain_amd import scenes as S
from tests.gpu_harness import emit

pytestmark = pytest.mark.gpu

OPACITY = 8  # v_splat's opacity lane


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_infinite_alpha_gradient(sign):
    sc = S.pixel_centred_scene()
    emit(f"fp32 backward, v_out {sign:+.0f} inf at five pixels")
    r = _native.Renderer(sc)
    try:
        r.forward()
        xy = r.read("proj0")[:5, :2].astype(int)
        v = np.zeros((sc.W * sc.H, 4), np.float32)
        v[xy[:, 1] * sc.W + xy[:, 0], 3] = sign * np.inf
        r.write("v_out", v)
        r.zero("v_splat")
        r.zero("vis_flag")
        r.backward(mode=0, grad_scale=1.0)
        g = r.read("v_splat").reshape(-1, 13)[:sc.n, OPACITY]
    finally:
        r.close()
    assert not np.isnan(g).any(), np.flatnonzero(np.isnan(g))
    assert (g[:5] == sign * np.inf).all()
    assert np.isin(g, [0.0, sign * np.inf]).all()
