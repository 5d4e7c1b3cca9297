"""The eval metrics (eval_kernel in b2ctrain_amd/csrc/kernels/aux_loss.hip) at sizes around one 54-column strip and the
ends of its strip heights, with and without the target's alpha as weight, against the CPU oracle. Bound: the sums
are of at most W H terms in [-1, 1]; a term's fp32 blurs differ from the oracle's by roundings (1e-5 of it), its
squared error by none that matters."""
import numpy as np
import pytest

from b2ctrain_amd import _native
from b2ctrain_amd import scenes as S
from oracle import oracle as O
from tests.gpu_harness import emit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(1, 1), (7, 97), (54, 23), (55, 24), (53, 46), (109, 131), (640, 363)])
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
