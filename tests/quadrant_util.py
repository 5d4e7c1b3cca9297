"""Splats, pixel truth and a second culling bound for test_quadrant_reach.py. Splats are random, among them needle-thin
ellipses (axis ratio up to 1e5) whose terms cancel, centred inside, on the edges and far outside the tile. The truth is
taken by brute force over all 64 pixel centres with the raster kernels' fp32 sigma (the quadratic about the tile
centre of sigma_coefs / poly_sigma, five fused multiply-adds, evaluated by the oracle's C restatement; the reference's
src/gpu/raster_fwd.cu:44-50 rounds the same quantity differently)."""
import numpy as np

from oracle import oracle as O

f32 = np.float32


def edge_lb(ah, b, ch, dx, dy):
    t1 = ah * dx * dx
    t2 = ch * dy * dy
    t3 = b * dx * dy
    return (t1 + t2 + t3) - f32(1e-5) * (np.abs(t1) + np.abs(t2) + np.abs(t3))


def poly_slack_power(mx, my, ah, b, ch, power, x0, y0):
    """power raised by 1e-5 of the magnitude of the tile-centred quadratic's terms over the tile, far above the
    rounding of the per-pixel sigma."""
    mxr, myr, bb = np.abs(mx - (x0 + f32(3.5))), np.abs(my - (y0 + f32(3.5))), np.abs(b)
    scale = (((ah * mxr + bb * myr) * mxr + ch * myr * myr) +
             f32(3.5) * ((f32(2) * ah + bb) * mxr + (bb + f32(2) * ch) * myr) + f32(12.25) * (ah + bb + ch))
    return power + f32(1e-5) * scale


def quadrant_mask_all_edges(mx, my, ah, b, ch, power, x0, y0):
    """Per quadrant, the centre inside the box, or the clamped minimum of sigma on one of the box's four edges, within a
    margin of 1e-5 of its terms: the bound by edges that quadrant_reach, which goes by lines, is measured against."""
    with np.errstate(all="ignore"):
        power = poly_slack_power(mx, my, ah, b, ch, power, x0, y0)
        ky = -b / (f32(2) * ch)
        kx = -b / (f32(2) * ah)
        ex = [x0 - mx, x0 + f32(3) - mx, x0 + f32(4) - mx, x0 + f32(7) - mx]
        ey = [y0 - my, y0 + f32(3) - my, y0 + f32(4) - my, y0 + f32(7) - my]
        mask = np.zeros(mx.shape, np.uint32)
        for qy in range(2):
            for qx in range(2):
                xlo, xhi, ylo, yhi = ex[2 * qx], ex[2 * qx + 1], ey[2 * qy], ey[2 * qy + 1]
                inside = (xlo <= 0) & (xhi >= 0) & (ylo <= 0) & (yhi >= 0)
                reach = inside.copy()
                for xe in (xlo, xhi):
                    reach |= ~(edge_lb(ah, b, ch, xe, np.fmin(np.fmax(ky * xe, ylo), yhi)) > power)
                for ye in (ylo, yhi):
                    reach |= ~(edge_lb(ah, b, ch, np.fmin(np.fmax(kx * ye, xlo), xhi), ye) > power)
                mask |= np.where(reach, np.uint32(1 << (2 * qy + qx)), np.uint32(0))
        return np.where(~((ah > 0) & (ch > 0)), np.uint32(0xF), mask)


def sigma_at(mx, my, c00, c01, c11, x0, y0, i, j):
    return O.frag_sigma(mx, my, c00, c01, c11, x0 + f32(i), y0 + f32(j))


def pixel_truth(mx, my, c00, c01, c11, power, x0, y0):
    """Per quadrant: does any pixel centre pass the reference's cutoff (fp32, uncontracted)?"""
    truth = np.zeros(mx.shape, np.uint32)
    for j in range(8):
        for i in range(8):
            sig = sigma_at(mx, my, c00, c01, c11, x0, y0, i, j)
            hit = sig <= power
            truth |= np.where(hit, np.uint32(1 << (2 * (j // 4) + i // 4)), np.uint32(0))
    return truth


def _splats(rng, n, spread, log_ratio_max):
    theta = rng.uniform(0, np.pi, n)
    s1 = np.exp(rng.uniform(-1.0, 4.0, n))
    s2 = s1 * np.exp(-rng.uniform(0, log_ratio_max, n))
    c, s = np.cos(theta), np.sin(theta)
    # covariance R diag(s1^2, s2^2) R^T (+0.3 px dilation as the projection adds), conic = inverse
    a = c * c * s1**2 + s * s * s2**2 + 0.3
    bb = c * s * (s1**2 - s2**2)
    d = s * s * s1**2 + c * c * s2**2 + 0.3
    det = a * d - bb * bb
    c00, c01, c11 = (d / det).astype(f32), (-bb / det).astype(f32), (a / det).astype(f32)
    x0, y0 = f32(8 * 37 + 0.5), f32(8 * 11 + 0.5)
    mx = (x0 + 3.5 + rng.normal(0, spread, n)).astype(f32)
    my = (y0 + 3.5 + rng.normal(0, spread, n)).astype(f32)
    power = rng.uniform(0.0, 8.0, n).astype(f32)
    return mx, my, c00, c01, c11, power, x0, y0
