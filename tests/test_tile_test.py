"""The tile test's arithmetic (kernels/device_math.h, tile_hit): the quotient by the splat's rounded reciprocal and
the edge clamp of that form, restated in numpy fp32, against the reference's form (splat_math.cuh:27-41: two
divisions by the scaled edge) bit for bit: the nearest point and the decision, over tiles on every side of the
centre, centres on tile edges, thin, tiny and huge conics, and powers next to the sigma of the point. And the row of a
tile number in a bounding box by one multiplication, over every box width up to 512 and numbers at row edges."""
import numpy as np

f = np.float32


def _sigma(px, py, a, b, c, mx, my):
    dx, dy = px - mx, py - my
    return f(0.5) * (a * dx * dx + c * dy * dy) + b * dx * dy


def _reference(rx, ry, mx, my, a, b, c, power):
    Rx, Ry = rx + f(8), ry + f(8)
    xl, xr, ya, yb = mx < rx, mx > Rx, my < ry, my > Ry
    in_x, in_y = ~(xl | xr), ~(ya | yb)
    cx, cy = np.where(xl, rx, Rx), np.where(ya, ry, Ry)
    dxf, dyf = np.where(xl, f(8), f(-8)), np.where(ya, f(8), f(-8))
    ex, ey = mx - cx, my - cy
    tx = (dxf * a * ex + dxf * b * ey) / (dxf * a * dxf)
    ty = (dyf * b * ex + dyf * c * ey) / (dyf * c * dyf)
    tx = np.where(in_y, f(0), np.clip(tx, f(0), f(1)))
    ty = np.where(in_x, f(0), np.clip(ty, f(0), f(1)))
    px, py = cx + tx * dxf, cy + ty * dyf
    s = _sigma(px, py, a, b, c, mx, my)
    return px, py, s, (in_x & in_y) | (s <= power)


def _fma(x, y, z):  # exact in double here: 48-bit products, sums that cancel to fewer bits or dominate
    return (x.astype(np.float64) * y.astype(np.float64) + z.astype(np.float64)).astype(f)


def _quotient(n, c):
    r = np.where((c >= f(2.0**-40)) & (c <= f(2.0**40)), f(1) / c, f(0))
    q0 = n * r
    q = _fma(_fma(-c, q0, n), r, q0)
    return np.where(r == 0, n / c, q)


def _kernel(rx, ry, mx, my, a, b, c, power):
    Rx, Ry = rx + f(8), ry + f(8)
    xl, xr, ya, yb = mx < rx, mx > Rx, my < ry, my > Ry
    in_x, in_y = ~(xl | xr), ~(ya | yb)
    cx, cy = np.where(xl, rx, Rx), np.where(ya, ry, Ry)
    ex, ey = mx - cx, my - cy
    lx, ly = np.where(xl, f(0), f(-8)), np.where(ya, f(0), f(-8))
    qx, qy = _quotient(a * ex + b * ey, a), _quotient(b * ex + c * ey, c)
    px = cx + np.where(in_y, f(0), np.minimum(np.maximum(qx, lx), lx + f(8)))
    py = cy + np.where(in_x, f(0), np.minimum(np.maximum(qy, ly), ly + f(8)))
    s = _sigma(px, py, a, b, c, mx, my)
    return px, py, s, (in_x & in_y) | (s <= power)


def _conics(rng, n, kind):
    if kind == "thin":
        l1, l2 = 10.0 ** rng.uniform(-1, 6, n), 0.3 + 10.0 ** rng.uniform(-3, 0, n)
    elif kind == "huge":
        l1, l2 = 10.0 ** rng.uniform(6, 17, n), 10.0 ** rng.uniform(-1, 17, n)
    else:
        l1, l2 = 0.3 + 10.0 ** rng.uniform(-3, 3, n), 0.3 + 10.0 ** rng.uniform(-3, 3, n)
    th = rng.uniform(0, np.pi, n)
    cs, sn = np.cos(th), np.sin(th)
    a, b, c = cs * cs / l1 + sn * sn / l2, cs * sn * (1 / l1 - 1 / l2), sn * sn / l1 + cs * cs / l2
    return a.astype(f), b.astype(f), c.astype(f)


def test_tile_test_matches_the_reference_form():
    rng = np.random.default_rng(11)
    for kind in ("thin", "huge", "plain"):
        n = 400_000
        a, b, c = _conics(rng, n, kind)
        rx, ry = (8.0 * rng.integers(0, 480, n)).astype(f), (8.0 * rng.integers(0, 270, n)).astype(f)
        reach = 10.0 ** rng.uniform(-2, 3.3, n)
        mx = (rx + 4 + reach * rng.uniform(-1, 1, n)).astype(f)
        my = (ry + 4 + reach * rng.uniform(-1, 1, n)).astype(f)
        edge = rng.random(n) < 0.1  # centres on tile edges
        mx[edge] = rx[edge] + f(8) * rng.integers(-1, 3, int(edge.sum())).astype(f)
        p = rng.uniform(0, 5.6, n).astype(f)
        _, _, s, _ = _reference(rx, ry, mx, my, a, b, c, p)
        near = rng.random(n) < 0.5  # powers at and next to the point's sigma
        p[near] = np.nextafter(s[near], s[near] + rng.integers(-1, 2, int(near.sum())).astype(f)).astype(f)
        want, got = _reference(rx, ry, mx, my, a, b, c, p), _kernel(rx, ry, mx, my, a, b, c, p)
        for w, g in zip(want, got):
            np.testing.assert_array_equal(w, g)


def test_row_of_a_tile_number():
    for bw in list(range(1, 513)) + [777, 1024, 4096]:
        rows = min(2048, (1 << 20) // bw)
        row = np.unique(np.concatenate([np.arange(min(rows, 64)), np.linspace(0, rows - 1, 200).astype(np.int64)]))
        b = np.concatenate([row * bw, row * bw + bw - 1, row * bw + bw // 2])
        inv = f(1) / f(bw)
        got = ((b.astype(f) + f(0.5)) * inv).astype(np.int64)
        np.testing.assert_array_equal(got, b // bw)
