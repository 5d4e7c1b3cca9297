"""The eval metrics (b2ctrain_amd/csrc/kernels/aux_loss.hip) against the CPU oracle, with and without the target's alpha as
weight: the tile kernel of small and of narrow images at sizes around one 16x16 tile, and the strip kernel at strip heights
of 23, 34, 67 and 122 rows with ragged last strips in either direction. Bound: the sums
are of at most W H terms in [-1, 1]; a term's fp32 blurs differ from the oracle's by roundings (1e-5 of it), its
squared error by none that matters."""
import numpy as np
import pytest

from b2ctrain_amd import _native
from b2ctrain_amd import scenes as S
from oracle import oracle as O
from tests.gpu_harness import emit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(1, 1), (7, 97), (54, 23), (55, 24), (53, 46), (109, 131), (640, 363),
                                 (16, 16), (17, 15), (16, 30000),
                                 (600, 610), (163, 3001), (54, 9001), (1600, 900), (2001, 1201), (3800, 2155)])
@pytest.mark.parametrize("mask_weighted", [False, True])
def test_eval_strips(W, H, mask_weighted):
    sc = S.config1()
    rng = np.random.default_rng(W * 1000 + H)
    sc.cam = S.Camera(W, H, float(W), float(W), W / 2, H / 2, sc.cam.R, sc.cam.t)
    c = rng.random((H * W, 4))
    sc.gt = S._pack_rgba(c[:, 0], c[:, 1], c[:, 2], c[:, 3])
    emit(f"eval at {W}x{H} mask_weighted={mask_weighted}")
    r = _native.Renderer(sc)
    try:
        r.forward(bg=(0.0, 0.0, 0.0))
        r.zero("loss_accum")
        r.eval_metrics(mask_weighted=mask_weighted)
        got = r.read("loss_accum")
        se, ss = O.eval_metrics(W, H, r.read("out_rgba"), sc.gt, mask_weighted)
    finally:
        r.close()
    assert abs(got[4] - se) <= 1e-5 * se + 1e-6
    assert abs(got[5] - ss) <= 1e-5 * 3 * W * H
