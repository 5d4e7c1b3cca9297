"""A replayed fragment carries the blend weight that the render gave it, bit for bit: 40 splats over one 8x8 tile, one
pixel with a weight, so a splat's w_all is its blend weight there; and the render in which that splat alone has a colour
gives the pixel weight times colour."""
import numpy as np
import pytest

from b2ctrain_amd import _native
from b2ctrain_amd import scenes as S
from tests.gpu_harness import emit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pixel", [27, 0, 61])
def test_evidence_takes_the_renders_weights(pixel):
    rng = np.random.default_rng(pixel)
    n, W, H = 40, 8, 8
    pos = np.stack([rng.uniform(-0.03, 0.03, n), rng.uniform(-0.03, 0.03, n), 2.0 + 0.01 * rng.permutation(n)], 1)
    pos_op = np.concatenate([pos, rng.uniform(-2.5, -1.0, (n, 1))], 1).astype(np.float32)
    lscale = np.zeros((n, 4), np.float32)
    lscale[:, :3] = rng.uniform(-2.3, -1.8, (n, 3))
    black = np.full((n, 1, 3), -0.5 / S.SH_C0 - 0.1, np.float32)
    cam = S.Camera(W, H, 64.0, 64.0, 4.0, 4.0, np.eye(3, dtype=np.float32).reshape(9), np.zeros(3, np.float32))
    weights = np.zeros(W * H, np.uint8)
    weights[pixel] = 255
    gt = S._pack_rgba(*rng.random((3, H * W)), np.ones(H * W))
    q = rng.standard_normal((n, 4)).astype(np.float32)
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    sc = S.Scene("one tile", 0, pos_op, q, lscale, black, cam, gt, weights)
    emit(f"blend weights at pixel {pixel}")
    r = _native.Renderer(sc)
    v = _native.View(W, H, gt, weights, has_alpha=True)
    try:
        w_all = r.compute_evidence([v], [cam])[:, 1]
        want = np.zeros(n, np.float32)
        for i in range(n):
            sc.sh = black.copy()
            sc.sh[i] = 0.6
            r.upload(sc)
            r.forward(bg=(0.0, 0.0, 0.0))
            colour = r.read("proj2")[i, 0]
            want[i] = r.read("out_rgba")[pixel, 0]
            assert colour > 0.5
            w_all[i] *= colour
    finally:
        v.close()
        r.close()
    assert (want > 0).sum() >= 30
    np.testing.assert_array_equal(w_all, want)
