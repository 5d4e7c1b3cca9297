"""The workgroup-to-tile mapping of the raster kernels (4x4-tile blocks dealt to the XCDs in turn, 2x2 or single
tiles on small images): every tile of an image must be rendered and replayed once, whatever its size. The
sizes sit at the mapping's edges: one tile, fewer tiles than XCDs, ragged last blocks in either direction, one
row of tiles, and both sides of each block-size change (128 blocks)."""
import numpy as np
import pytest

from b2ctrain_amd import scenes as S
from tests.gpu_harness import emit, full_check

pytestmark = pytest.mark.gpu


def _scene(W, H, n=150):
    sc = S.fd_scene(1234 + W * 3 + H, n=n)
    f = 0.85 * max(W, H)
    sc.cam = S.Camera(W, H, f, f, W / 2.0, H / 2.0, sc.cam.R, sc.cam.t)
    rng = np.random.default_rng(W * 10007 + H)
    sc.pos_op[:, 0] = ((rng.random(n) - 0.5) * 2.0 * W / f).astype(np.float32)
    sc.pos_op[:, 1] = ((rng.random(n) - 0.5) * 2.0 * H / f).astype(np.float32)
    sc.lscale[:, :3] -= np.float32(0.7)
    rgba = rng.integers(0, 256, (W * H, 4)).astype(np.uint32)
    sc.gt = (rgba[:, 0] | (rgba[:, 1] << 8) | (rgba[:, 2] << 16) | (rgba[:, 3] << 24)).astype(np.uint32)
    sc.weights = rng.integers(64, 256, W * H).astype(np.uint8)
    sc.name = f"blocks{W}x{H}"
    return sc


# tiles: 1x1, 3x2, 44x44 (121 blocks of 4x4: 2x2 blocks), 48x44 (132), 31x16 (128 blocks of 2x2), 30x16 (120: single
# tiles), 257x2 and 125x1 (one row of blocks)
@pytest.mark.parametrize("W,H", [(8, 8), (21, 13), (352, 352), (383, 345), (245, 128), (240, 121), (2055, 9), (1000, 5)])
def test_every_tile_once(W, H):
    sc = _scene(W, H)
    emit(f"{sc.name}")
    full_check(sc, mode=1)
