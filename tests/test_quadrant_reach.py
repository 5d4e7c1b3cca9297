"""The raster's quadrant test by nearest lines (quadrant_reach in b2ctrain_amd/csrc/kernels/raster_common.h), restated
in float32 numpy with the hardware reciprocal and square root anywhere within 1 ulp, over the splats of
quadrant_util.py: a quadrant with a pixel that passes the cutoff is kept, pixels exactly on the cutoff
included, and no more is kept than by the minimum over each quadrant's edges but for the margins. The GPU parity tests
check the device code itself (a wrongly culled fragment changes the rendered colour by at least alpha = 1/255 of
its weight)."""
import numpy as np
import pytest

from tests.quadrant_util import _splats, pixel_truth, quadrant_mask_all_edges, sigma_at

f32 = np.float32


def _fma(a, b, c):
    return (np.asarray(a, np.float64) * b + np.asarray(c, np.float64)).astype(f32)


def _approx(x, rng):  # within 1 ulp
    x = x.astype(f32)
    d = rng.integers(-1, 2, x.shape)
    return np.where(d < 0, np.nextafter(x, f32(-np.inf)), np.where(d > 0, np.nextafter(x, f32(np.inf)), x))


def quadrant_reach(mx, my, ah, b, ch, power, x0, y0, rng):
    with np.errstate(all="ignore"):
        ra, rc = _approx(f32(1) / (ah + ah), rng), _approx(f32(1) / (ch + ch), rng)
        ky, kx = -b * rc, -b * ra
        qv, qh = _fma(f32(0.5) * b, ky, ah), _fma(f32(0.5) * b, kx, ch)
        dx0, dy0 = x0 - mx, y0 - my
        mxr, myr, bb = np.abs(dx0 + f32(3.5)), np.abs(dy0 + f32(3.5)), np.abs(b)
        scale = (((ah * mxr + bb * myr) * mxr + ch * myr * myr) +
                 f32(3.5) * ((f32(2) * ah + bb) * mxr + (bb + f32(2) * ch) * myr) + f32(12.25) * (ah + bb + ch))
        pw = _fma(f32(2e-5), scale, power)
        keep = ~((ah > 0) & (ch > 0)) | ~(np.abs(scale + (qv + qh)) < np.inf)
        q = [keep.copy() for _ in range(4)]
        for k in range(2):
            xlo, ylo = dx0 + f32(4 * k), dy0 + f32(4 * k)
            xe = np.clip(f32(0), xlo, xlo + f32(3)).astype(f32)
            ye = np.clip(f32(0), ylo, ylo + f32(3)).astype(f32)
            rv = _approx(np.sqrt(_fma(-qv * xe, xe, pw) * (rc + rc)), rng) + f32(1.5)
            rh = _approx(np.sqrt(_fma(-qh * ye, ye, pw) * (ra + ra)), rng) + f32(1.5)
            cv, cz = _fma(ky, xe, f32(-1.5) - dy0), _fma(kx, ye, f32(-1.5) - dx0)
            for o in range(2):
                q[2 * o + k] |= np.abs(cv - f32(4 * o)) <= rv
                q[2 * k + o] |= np.abs(cz - f32(4 * o)) <= rh
        return sum(np.where(m, np.uint32(1 << k), np.uint32(0)) for k, m in enumerate(q)).astype(np.uint32)


@pytest.mark.parametrize("spread,ratio", [(3.0, 2.0), (10.0, 5.0), (1.0, 9.2), (5.0, 11.5), (30.0, 9.2), (40.0, 9.2),
                                          (100.0, 11.5), (1000.0, 11.5)])
@pytest.mark.parametrize("on_cutoff", [False, True])
def test_quadrant_reach_is_conservative(spread, ratio, on_cutoff):
    rng = np.random.default_rng(int(spread) + 100 * on_cutoff)
    mx, my, c00, c01, c11, power, x0, y0 = _splats(rng, 200_000, spread, ratio)
    if on_cutoff:  # one pixel of each splat passes with sigma == power (one rounded below 0, against power 0)
        i, j = rng.integers(0, 8, mx.size), rng.integers(0, 8, mx.size)
        sig = sigma_at(mx, my, c00, c01, c11, x0, y0, i.astype(f32), j.astype(f32))
        power = np.maximum(sig, f32(0)).astype(f32)
    ah, ch = f32(0.5) * c00, f32(0.5) * c11
    got = quadrant_reach(mx, my, ah, c01, ch, power, x0, y0, rng)
    truth = pixel_truth(mx, my, c00, c01, c11, power, x0, y0)
    missed = truth & ~got
    assert not missed.any(), f"culled a reachable quadrant: {np.flatnonzero(missed)[:5]}"
    if on_cutoff:
        on = sig <= power
        assert ((truth & (np.uint32(1) << (2 * (j // 4) + i // 4).astype(np.uint32))) != 0)[on].all() and on.any()
        return
    old = quadrant_mask_all_edges(mx, my, ah, c01, ch, power, x0, y0)
    assert np.count_nonzero(got & ~old) <= 1e-3 * mx.size
    if spread <= 40.0:  # both outcomes occur
        assert np.count_nonzero(truth) > 10_000 and np.count_nonzero(~got & np.uint32(0xF)) > 10_000


def test_quadrant_reach_centre_inside():
    mx, my, ah, b, ch, power = (np.array([v], f32) for v in (101.0, 101.0, 0.5, 0.0, 0.5, 0.0))
    got = quadrant_reach(mx, my, ah, b, ch, power, f32(96.5), f32(96.5), np.random.default_rng(0))
    assert got[0] == 1 << 3  # the centre is a pixel centre of quadrant (1, 1), and nothing else is reached


def test_quadrant_reach_degenerate():
    rng = np.random.default_rng(1)
    for bad in [(np.nan, 1, 0.5, 0, 0.5), (np.inf, 1, 0.5, 0, 0.5), (1, 1, 0, 0, 0.5), (1, 1, 0.5, 0, -1), (1, 1, np.inf, 0, 1),
                (1, 1, 0.5, np.nan, 0.5), (1, 1, 1e-45, 0, 0.5)]:
        mx, my, ah, b, ch = (np.array([v], f32) for v in bad)
        assert quadrant_reach(mx, my, ah, b, ch, np.array([1], f32), f32(0.5), f32(0.5), rng)[0] == 0xF
