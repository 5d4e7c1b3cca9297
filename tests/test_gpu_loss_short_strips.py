"""The fused loss on small images, whose strips are shorter than the 35 rows of large ones (pick_strip_rows in
b2ctrain_amd/csrc/kernels/loss.hip): value and per-pixel gradient against the CPU oracle, at widths around one
54-column strip and heights from one row to several short strips with a ragged last one."""
import numpy as np
import pytest

from b2ctrain_amd import _native
from b2ctrain_amd import scenes as S
from tests.gpu_harness import check_loss, emit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(1, 1), (54, 1), (55, 2), (7, 97), (64, 64), (109, 37), (230, 219), (400, 301)])
def test_loss_short_strips(W, H):
    sc = S.config1()
    rng = np.random.default_rng(W * 1000 + H)
    sc.cam = S.Camera(W, H, float(W), float(W), W / 2, H / 2, sc.cam.R, sc.cam.t)
    c = rng.random((H * W, 3))
    sc.gt = S._pack_rgba(c[:, 0], c[:, 1], c[:, 2], np.ones(H * W))
    bg = (0.3, 0.6, 0.2)
    emit(f"loss at {W}x{H}")
    r = _native.Renderer(sc)
    try:
        r.project(bg=bg)
        r.bin()
        r.raster_fwd(bg=bg)
        check_loss(r, sc, r.read("out_rgba"), 3.0 * W * H, bg)
    finally:
        r.close()
