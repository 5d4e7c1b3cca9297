"""The label vote of tiles that hold several classes (evidence_kernel in b2ctrain_amd/csrc/kernels/replay.hip): up to four
classes a tile have pixel vectors of their own, the others a masked sum each. Label maps that put two to four, five to
nine and up to 40 classes into one 8x8 tile, ids of 32 and more (ignored) and pixels of weight zero among them, on lists
of any length and on an image that ends inside a tile; winners and shares against the CPU oracle at the bars of
test_gpu_replay.py."""
import numpy as np
import pytest

from b2ctrain_amd import _native
from b2ctrain_amd import scenes as S
from oracle import oracle as O
from tests.gpu_harness import emit
from tests.test_gpu_replay import _oracle_evidence, _views

pytestmark = pytest.mark.gpu

MAPS = {  # class of a pixel, the most voting classes in a tile
    "halves_of_tiles": (lambda x, y: (x + 4) // 8 % 2 * 5 + 3, 2),
    "blocks8_shifted3": (lambda x, y: ((x + 3) // 8 * 7 + (y + 3) // 8 * 3) % 31, 4),
    "three": (lambda x, y: (x + y) % 3 * 15, 3),
    "four": (lambda x, y: (x + 2 * y) % 4 * 10 + 1, 4),
    "five": (lambda x, y: (x + y) % 5 * 7 + 3, 5),
    "blocks5": (lambda x, y: (x // 5 * 7 + y // 5 * 3) % 40, 9),
    "pixels": (lambda x, y: (x * 7 + y * 3) % 40, 24),
}


def _most_in_a_tile(labels, weights, W, H):
    y, x = np.divmod(np.arange(W * H), W)
    on = (labels < 32) & (weights > 0)
    seen = np.zeros(((H + 7) // 8, (W + 7) // 8, 32), bool)
    seen[y[on] // 8, x[on] // 8, labels[on]] = True
    return int(seen.sum(2).max())


@pytest.mark.parametrize("name", MAPS)
@pytest.mark.parametrize("scene", ["ragged", "config2"])
def test_classes_inside_one_tile(scene, name):
    sc = S.fd_scene(11, n=90) if scene == "ragged" else S.config2(n=12_000)
    if scene == "ragged":
        sc.cam = S.Camera(45, 37, 40.0, 40.0, 22.5, 18.5, sc.cam.R, sc.cam.t)
        sc.gt = sc.gt[:45 * 37].copy()
    emit(f"labels {sc.name} {sc.W}x{sc.H} {name}")
    rng = np.random.default_rng(len(name))
    weights = rng.integers(64, 256, sc.W * sc.H).astype(np.uint8)
    weights[rng.random(sc.W * sc.H) < 0.1] = 0
    y, x = np.divmod(np.arange(sc.W * sc.H), sc.W)
    labels = MAPS[name][0](x, y).astype(np.uint8)
    assert _most_in_a_tile(labels, weights, sc.W, sc.H) >= MAPS[name][1]
    spec = dict(gt=sc.gt, weights=weights, labels=labels)
    r = _native.Renderer(sc)
    vs = _views(sc, [spec])
    try:
        ev = r.compute_evidence(vs, [sc.cam], export_labels=True)
        lv = r.download_labels()
        fw = dict(tile_ranges=r.read("tile_ranges"), out_rgba=r.read("out_rgba"), last_idx=r.read("last_idx"))
    finally:
        for v in vs:
            v.close()
        r.close()
    want, lab = _oracle_evidence(sc, [sc.cam], [spec], fws=[fw])
    assert (np.abs(ev - want).max(0) <= 1e-4 * (np.abs(want).max(0) + 1e-30)).all()
    win = O.label_winners(lab)
    srt = np.sort(lab, 1)
    clear = (srt[:, -1] - srt[:, -2]) > 1e-3 * np.maximum(srt[:, -1], 1e-30)
    emit(f"    voting splats {(win[:, 1] > 0).sum()}, clear winners {clear.sum()}")
    assert clear.sum() > (20 if scene == "ragged" else 1000)
    assert (lv[clear, 0] == win[clear, 0]).all()
    np.testing.assert_allclose(lv[:, 1], win[:, 1], atol=1e-4)
