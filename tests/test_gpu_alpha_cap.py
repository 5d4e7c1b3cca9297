"""The MFMA backward's two replays: groups of eight splats that may reach the 0.999 alpha cap, and groups that cannot
(which leave the cap out). Opacities on both sides of the cap and of the bound that tells the groups apart
(log2 opacity near -0.0015, logits 6.4 to 6.9), list lengths around the group of 8 and the batch of 48, splats
centred on pixel centres (where sigma rounds about 0): every stage against the oracle, in both backward modes."""
import numpy as np
import pytest

from b2ctrain_amd import scenes as S
from tests.gpu_harness import emit, full_check

pytestmark = pytest.mark.gpu

LOGITS = np.array([2.0, 6.3, 6.5, 6.8, 6.86, 6.9, 6.906, 6.92, 7.5, 9.0, 16.0], np.float32)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,every", [(7, 1), (9, 1), (47, 1), (49, 3), (120, 9)])
def test_opacities_about_the_cap(n, every, mode):
    sc = S.pixel_centred_scene(n)
    rng = np.random.default_rng(n)
    pick = rng.permutation(sc.n)[:min(n, sc.n)]
    sc.pos_op, sc.quat, sc.lscale, sc.sh = (a[pick].copy() for a in (sc.pos_op, sc.quat, sc.lscale, sc.sh))
    sc.pos_op[:, 3] = rng.uniform(-2.0, 2.0, sc.n)
    sc.pos_op[::every, 3] = rng.choice(LOGITS, sc.pos_op[::every].shape[0])
    sc.bg = (0.25, 0.5, 0.75)
    emit(f"alpha cap n={sc.n} every={every} mode={mode}")
    full_check(sc, mode=mode)
