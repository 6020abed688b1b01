"""The render backward's entry sums (four entries' pixel rows summed
together) at the edges of their grouping, against the blend's gradient written
out in float64.

n Gaussians that every pixel of a 40x24 image blends (partial tiles on two
edges), so that each quadrant's walk has n entries: remainders of four, of the
64 staged at a time and of the 64-position list words; ones as wide as the
image and ten times wider, some with their means far outside it.  (Narrow ones,
of a few pixels each, are test_gpu_backward_narrow.py's.)

Tolerance, element by element: |difference| <= (2e-6 + 3e-7 n) times the sum
of the terms' magnitudes.  The device recovers T in front of entry k by n - k
products with 1 / (1 - alpha), each within about 2 ulp, i.e. 2.4e-7 n
relative; the falloff's exp is within 5e-7, its exponent (below 1 here) and
the sums of 960 pixels within a few ulp.
"""
import numpy as np
import pytest
import torch

from blitzgs_amd import _lib, rasterizer
from tests.gpu_helpers import np_, to_dev

pytestmark = pytest.mark.gpu

W, H = 40, 24


def _inputs(n, seed=7):
    rng = np.random.default_rng(seed)
    m = np.stack([rng.uniform(0, W, n), rng.uniform(0, H, n)], 1)
    wide = rng.random(n) < 0.5
    m[wide] += rng.uniform(-150, 150, (int(wide.sum()), 2))
    s = np.where(wide, 400.0, 60.0)
    th = rng.uniform(0, np.pi, n)
    l1, l2 = 1 / s ** 2, 1 / (0.6 * s) ** 2
    a = l1 * np.cos(th) ** 2 + l2 * np.sin(th) ** 2
    c = l1 * np.sin(th) ** 2 + l2 * np.cos(th) ** 2
    b = (l1 - l2) * np.sin(th) * np.cos(th)
    op = rng.uniform(0.012, 0.03, n)
    return dict(means2D=m.astype(np.float32), conic=np.stack([a, b, c, op], 1).astype(np.float32),
                rgb=rng.uniform(0, 1, (n, 3)).astype(np.float32), radii=np.full(n, 2000, np.int32),
                depths=rng.permutation(n).astype(np.float32) + 1, bg=np.array([0.3, 0.1, 0.2], np.float32),
                dL=rng.standard_normal((3, H, W)).astype(np.float32))


def _reference(x, tiles=None):
    """(gradients, magnitudes): dmeans2D (scaled by W/2, H/2), |dmeans2D|, dconic
    a b c + dopacity (the b term halved, as the render backward leaves it) and
    drgb; tiles: mask of the tiles that take part."""
    o = np.argsort(x["depths"], kind="stable")
    m, con, rgb = (x[k][o].astype(np.float64) for k in ("means2D", "conic", "rgb"))
    py, px = np.mgrid[0:H, 0:W].reshape(2, -1).astype(np.float64)
    on = np.ones(H * W) if tiles is None else np.repeat(np.repeat(tiles, 16, 0), 16, 1)[:H, :W].reshape(-1)
    dL = x["dL"].reshape(3, -1).astype(np.float64) * on
    dx, dy = m[:, :1] - px, m[:, 1:] - py
    A, B, C, op = (con[:, k:k + 1] for k in range(4))
    G = np.exp(-0.5 * (A * dx * dx + C * dy * dy) - B * dx * dy)
    al = np.minimum(0.99, op * G)
    assert (al >= 1.05 / 255).all()
    after = np.cumprod(1 - al, 0)
    assert after[-1].min() > 1e-3
    T = after / (1 - al)
    out = []
    for ab in (lambda v: v, np.abs):
        cd = ab(rgb) @ ab(dL)
        w = al * T * cd
        behind = np.cumsum(w[::-1], 0)[::-1] - w + after[-1] * (ab(x["bg"].astype(np.float64)) @ ab(dL))
        da = T * cd - behind / (1 - al) if ab is not np.abs else T * cd + behind / (1 - al)
        g = G * op * da
        fx, fy = -(A * dx + B * dy), -(C * dy + B * dx)
        mean = np.stack([(g * ab(fx)).sum(1) * W / 2, (g * ab(fy)).sum(1) * H / 2], 1)
        mabs = np.stack([np.abs(g * fx).sum(1) * W / 2, np.abs(g * fy).sum(1) * H / 2], 1)
        c4 = np.stack([-0.5 * (g * dx * dx).sum(1), -0.5 * (g * ab(dx * dy)).sum(1), -0.5 * (g * dy * dy).sum(1),
                       (G * da).sum(1)], 1)
        r = dict(m2=mean, m2a=mabs, con=ab(c4), col=(al * T) @ ab(dL).T)
        back = np.empty_like(o)
        back[o] = np.arange(len(o))
        out.append({k: v[back] for k, v in r.items()})
    return out


def _gpu(x, capacity=None, cl_bwd=None):
    """capacity: None, the exact two-call forward; else the one-call forward
    with a buffer laid out for that many instances."""
    dev = torch.device("cuda:0")
    keep = _lib.RESERVE
    _lib.RESERVE = _lib.InstanceReserve()
    if capacity is not None:
        _lib.RESERVE.update(dev, capacity)
    try:
        m, c, g, bg = (to_dev(x[k]) for k in ("means2D", "conic", "rgb", "bg"))
        out = rasterizer._render_forward_raw(bg, H, W, m, to_dev(x["depths"]), to_dev(x["radii"]), c, g, None)
        R, geom, binning, img = out[0], out[6], out[7], out[8]
        cl = None if cl_bwd is None else to_dev(cl_bwd).bool()
        m2, m2a, con, col, _ = rasterizer._render_backward_raw(bg, R, H, W, m, c, g, cl, geom, binning, img,
                                                               to_dev(x["dL"]))
    finally:
        _lib.RESERVE = keep
    return out, dict(m2=m2, m2a=m2a[:, :2], con=con, col=col)


def _check(got, want, n):
    ref, mag = want
    for k in ref:
        g = np_(got[k]).astype(np.float64)
        e = np.abs(g - ref[k]) / mag[k]
        assert np.isfinite(g).all() and e.max() <= 2e-6 + 3e-7 * n, (k, n, e.max(), np.unravel_index(e.argmax(), e.shape))


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 63, 64, 65, 127, 128, 130, 200])
def test_entry_sums(gpu, n):
    x = _inputs(n)
    _check(_gpu(x)[1], _reference(x), n)


def test_large_capacity_and_masked_backward(gpu):
    """The lists in a buffer laid out for far more instances than there are;
    then the backward over half the tiles the forward rendered."""
    x = _inputs(130)
    _check(_gpu(x, capacity=500000)[1], _reference(x), 130)
    cl = np.zeros((2, 3), np.uint8)
    cl[1, :] = 1
    _check(_gpu(x, capacity=1000, cl_bwd=cl)[1], _reference(x, cl), 130)


def test_infinite_colour_stays_with_its_pixels(gpu):
    """A Gaussian of infinite colour that reaches only part of a quadrant
    leaves the gradients of one that shares the quadrant but no pixel as they
    were."""
    x = _inputs(2)
    x["means2D"][:] = [[1.0, 1.0], [6.0, 6.0]]
    x["conic"][:] = [[1.0, 0.0, 1.0, 0.5], [1.0, 0.0, 1.0, 0.5]]
    x["depths"][:] = [1.0, 2.0]
    x["radii"][:] = 8
    want = _gpu(x)[1]
    x["rgb"][0] = np.inf
    got = _gpu(x)[1]
    for k in want:
        # the quadrants' sums meet in any order: three additions of 6e-8, on sums up to 30 times the result
        a, b = np_(got[k])[1], np_(want[k])[1]
        assert np.isfinite(a).all() and (np.abs(a - b) <= 6e-6 * np.abs(b)).all(), k
