"""The render backward's gradients for narrow Gaussians (sigma from the
low-pass limit sqrt(0.3) px up to 2 px, opacities from just above 1/255 to 0.5,
sub-pixel mean offsets): one or a few blended pixels per Gaussian, so that a
sum of offsets from the mean must not cancel.  The split, the full-image and the
render_geo backward, against the blend's gradient written out in float64 with
the 1/255 cut and the 0.99 clamp (which in the full-image path also drops the
conic and opacity gradients).

Tolerance, element by element: |difference| <= the sum over the pixels of e
times the magnitude of the pixel's terms (A dx and B dy taken separately), with
e = 3e-6 + 3e-7 n + 6e-7 sum alpha / (1 - alpha) over the pixel's n blended
entries.  The exponent is a sum of terms below 12 in magnitude, each rounded
twice, and the exp2 takes it times log2(e): 2e-6 of the falloff together; sums,
colour dot products and the final scale a few ulp; the transmittance is
recovered by n products with 1 / (1 - alpha), each within 2 ulp, and an error
of 6e-7 of alpha (of which the forward's T holds the same) is amplified by
alpha / (1 - alpha).
"""
import ctypes as C

import numpy as np
import pytest
import torch

from blitzgs_amd import _lib, rasterizer
from tests.gpu_helpers import np_, to_dev

pytestmark = pytest.mark.gpu

W, H = 40, 24
CUT, CLAMP = 1 / 255, np.float64(np.float32(0.99))


def _inputs(seed, n=240, clamped=False, faint=False):
    rng = np.random.default_rng(seed)
    m = np.stack([rng.uniform(-1, W, n), rng.uniform(-1, H, n)], 1)
    s = rng.choice([np.sqrt(0.3), 0.8, 1.2, 2.0], n)
    op = rng.uniform(0.03, 0.5, n)
    faint = np.ones(n, bool) if faint else rng.random(n) < 0.5
    op[faint] = rng.uniform(1.02, 3.0, int(faint.sum())) / 255
    # some means almost on a pixel centre, where one offset is far below the others
    on = rng.random(n) < 0.3
    m[on] = np.round(m[on]) + rng.uniform(-0.02, 0.02, (int(on.sum()), 2))
    depths = rng.permutation(n).astype(np.float32) + 1
    if clamped:   # opaque ones in front, on pixels of their own, above the clamp at the centre pixel
        k = 24
        cells = rng.permutation((W // 8) * (H // 4))[:k]
        m[:k] = np.stack([8 * (cells % (W // 8)) + 3, 4 * (cells // (W // 8)) + 1], 1) + rng.uniform(-0.03, 0.03, (k, 2))
        op[:k], s[:k], depths[:k] = 1.0, np.sqrt(0.3), -1 - np.arange(k)
        depths += k + 2
    th = rng.uniform(0, np.pi, n)
    l1, l2 = 1 / s ** 2, 1 / (rng.uniform(0.8, 1.0, n) * s) ** 2
    a = l1 * np.cos(th) ** 2 + l2 * np.sin(th) ** 2
    c = l1 * np.sin(th) ** 2 + l2 * np.cos(th) ** 2
    b = (l1 - l2) * np.sin(th) * np.cos(th)
    return dict(means2D=m.astype(np.float32), conic=np.stack([a, b, c, op], 1).astype(np.float32),
                rgb=rng.uniform(0, 1, (n, 3)).astype(np.float32), maps=rng.standard_normal((n, 5)).astype(np.float32),
                radii=np.full(n, 14, np.int32), depths=depths, bg=np.array([0.3, 0.1, 0.2], np.float32),
                dL=rng.standard_normal((3, H, W)).astype(np.float32),
                dmap=rng.standard_normal((5, H, W)).astype(np.float32))


def _reference(x, full, geo):
    """(gradients, bounds), as the render backward leaves them."""
    o = np.argsort(x["depths"], kind="stable")
    m, con, col = (x[k][o].astype(np.float64) for k in ("means2D", "conic", "rgb"))
    dL, bg = x["dL"].reshape(3, -1).astype(np.float64), x["bg"].astype(np.float64)
    if geo:
        col = np.concatenate([col, x["maps"][o].astype(np.float64)], 1)
        dL = np.concatenate([dL, x["dmap"].reshape(5, -1).astype(np.float64)], 0)
        bg = np.concatenate([bg, np.zeros(5)])
    py, px = np.mgrid[0:H, 0:W].reshape(2, -1).astype(np.float64)
    dx, dy = m[:, :1] - px, m[:, 1:] - py
    A, B, Cc, op = (con[:, k:k + 1] for k in range(4))
    G = np.exp(-0.5 * (A * dx * dx + Cc * dy * dy) - B * dx * dy)
    oG = op * G
    # no decision within the rounding of either side, no pixel that stops early
    assert np.abs(oG / CUT - 1).min() > 1e-5 and np.abs(oG / CLAMP - 1).min() > 1e-5
    use = oG >= CUT
    al = np.where(use, np.minimum(CLAMP, oG), 0.0)
    after = np.cumprod(1 - al, 0)
    assert after[-1].min() > 3e-4
    T = after / (1 - al)
    e = 3e-6 + 3e-7 * use.sum(0) + 6e-7 * (al / (1 - al)).sum(0)
    free = use & (oG <= CLAMP) if full else use
    out = []
    for ab in (lambda v: v, np.abs):
        cd = ab(col) @ ab(dL)
        w = al * T * cd
        behind = np.cumsum(w[::-1], 0)[::-1] - w + after[-1] * (ab(bg) @ ab(dL))
        da = np.where(use, T * cd + (behind if ab is np.abs else -behind) / (1 - al), 0.0)
        if ab is np.abs:
            da, T = da * e, T * e
        g = oG * da
        fx = (A * ab(dx) + ab(B) * ab(dy)) if ab is np.abs else -(A * dx + B * dy)
        fy = (Cc * ab(dy) + ab(B) * ab(dx)) if ab is np.abs else -(Cc * dy + B * dx)
        gc = g * free
        r = dict(m2=np.stack([(g * fx).sum(1) * W / 2, (g * fy).sum(1) * H / 2], 1),
                 con=ab(np.stack([-0.5 * (gc * dx * dx).sum(1), -0.5 * (gc * ab(dx * dy)).sum(1),
                                  -0.5 * (gc * dy * dy).sum(1), (G * da * free).sum(1)], 1)))
        c8 = (al * T) @ ab(dL).T
        r["col"] = c8[:, :3]
        if geo:
            r["map"] = c8[:, 3:]
        if not full:
            fa = [np.abs(A * dx + B * dy), np.abs(Cc * dy + B * dx)] if ab is not np.abs else [fx, fy]
            r["m2a"] = np.stack([(np.abs(g) * fa[0]).sum(1) * W / 2, (np.abs(g) * fa[1]).sum(1) * H / 2], 1)
        back = np.empty_like(o)
        back[o] = np.arange(len(o))
        out.append({k: v[back] for k, v in r.items()})
    return out


def _split(x, geo):
    m, c, g, bg = (to_dev(x[k]) for k in ("means2D", "conic", "rgb", "bg"))
    maps = to_dev(x["maps"])
    out = rasterizer._render_forward_raw(bg, H, W, m, to_dev(x["depths"]), to_dev(x["radii"]), c, g, None,
                                         geo=(1.0, 1.0, maps) if geo else None)
    R, geom, binning, img = out[0], out[6], out[7], out[8]
    back = rasterizer._render_backward_raw(bg, R, H, W, m, c, g, None, geom, binning, img, to_dev(x["dL"]),
                                           geo=(1.0, 1.0, out[10], maps, to_dev(x["dmap"]), None) if geo else None)
    r = dict(m2=back[0], m2a=back[1][:, :2], con=back[2], col=back[3])
    if geo:
        r["map"] = back[5]
    return r


def _full(x, dL=None):
    lib, ptr, check = _lib.load(), _lib.ptr, _lib.check
    dev = torch.device("cuda:0")
    s = _lib.stream_of(dev)
    m, c, g, bg, d, rad = (to_dev(x[k]) for k in ("means2D", "conic", "rgb", "bg", "depths", "radii"))
    P = m.shape[0]
    rects = rad.float()[:, None].expand(P, 2).contiguous()
    buf = lambda n: torch.empty(int(n), device=dev, dtype=torch.uint8)  # noqa: E731
    f32 = lambda *shape: torch.empty(shape, device=dev)  # noqa: E731
    geom, img, color = buf(lib.gs_render_geom_bytes(P, W, H)), buf(lib.gs_render_img_bytes(W, H)), f32(3, H, W)
    R = C.c_int64(0)
    check(lib.gs_render_full_count(P, W, H, ptr(m), ptr(rad), ptr(rects), ptr(c), ptr(geom), C.byref(R), s), "count")
    binning = buf(lib.gs_render_binning_bytes(R.value))
    check(lib.gs_render_full_forward(P, R.value, W, H, ptr(bg), ptr(m), ptr(d), ptr(rad), ptr(rects), ptr(c), ptr(g),
                                     ptr(geom), ptr(binning), ptr(img), ptr(color), None, None, None, s), "forward")
    dm, dc, dg = f32(P, 3), f32(P, 4), f32(P, 3)
    dL = to_dev(x["dL"] if dL is None else dL)
    check(lib.gs_render_full_backward(P, R.value, W, H, ptr(bg), ptr(m), ptr(c), ptr(geom), ptr(binning), ptr(img),
                                      ptr(dL), ptr(dm), ptr(dc), ptr(dg), s), "backward")
    return dict(m2=dm[:, :2], con=dc, col=dg)


def _check(x, path):
    full, geo = path == "full", path == "geo"
    ref, bound = _reference(x, full, geo)
    got = _full(x) if full else _split(x, geo)
    assert set(got) == set(ref)
    for k in ref:
        g = np_(got[k]).astype(np.float64)
        assert np.isfinite(g).all(), k
        bad = np.abs(g - ref[k]) > bound[k]
        i = np.unravel_index((np.abs(g - ref[k]) / np.maximum(bound[k], 1e-300)).argmax(), g.shape)
        assert int(bad.sum()) == 0, (k, int(bad.sum()), i, g[i], ref[k][i], bound[k][i])


@pytest.mark.parametrize("path", ["split", "geo", "full"])
@pytest.mark.parametrize("seed,faint", [(0, False), (1, True), (2, True)])
def test_narrow(gpu, path, seed, faint):
    _check(_inputs(seed, clamped=path == "full", faint=faint), path)


@pytest.mark.parametrize("path", ["split", "geo", "full"])
def test_blended_entries_far_apart_in_a_long_list(gpu, path):
    """130 Gaussians that every pixel blends among 9000 that lie between pixel
    centres of one quadrant of two tiles and are blended by none: lists of more
    than 64 batches of 64, most of whose marks are empty (split) or staged in vain
    (full)."""
    n, wide = 9130, 130
    rng = np.random.default_rng(5)
    x = _inputs(5, n=n)
    m = np.where(np.arange(n)[:, None] % 2 == 0, [3.5, 3.5], [35.5, 19.5]) + rng.uniform(-0.1, 0.1, (n, 2))
    s = 1 / 0.3
    conic = np.stack([np.full(n, s), np.zeros(n), np.full(n, s), rng.uniform(1.05, 1.3, n) / 255], 1)
    radii = np.full(n, 2, np.int32)
    at = rng.choice(n, wide, replace=False)
    m[at] = rng.uniform([0, 0], [W, H], (wide, 2))
    conic[at] = np.stack([np.full(wide, 1 / 60 ** 2), np.zeros(wide), np.full(wide, 1 / 45 ** 2),
                          rng.uniform(0.012, 0.03, wide)], 1)
    radii[at] = 2000
    x.update(means2D=m.astype(np.float32), conic=conic.astype(np.float32), radii=radii)
    _check(x, path)


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("n", [1, 4, 6, 70])
def test_full_path_unblended_entries_take_no_gradient(gpu, n, value):
    """Full-image path: faint Gaussians whose means lie between pixel centres
    are staged (the test that drops entries is against the quadrant's rectangle)
    and blended by no pixel.  Beside blended ones and with an image gradient that
    is not finite in their quadrant they take no gradient, and the blended ones of
    the other quadrants take what they take without it."""
    rng = np.random.default_rng(n)
    m = rng.integers(0, 6, (n, 2)) + 0.5
    op = np.full(n, 1.2 / 255)
    seen = np.arange(n) % 3 == 1     # these are blended, every other one in the quadrant at (8, 0)
    op[seen] = 0.4
    m[seen] += np.where(np.arange(int(seen.sum())) % 2 == 1, 8.0, 0.0)[:, None] * [[1.0, 0.0]] + 0.5
    other = seen & (m[:, 0] > 8)
    m[other] = [12.0, 4.0]
    s = 1 / 0.3
    x = dict(means2D=m.astype(np.float32), conic=np.stack([np.full(n, s), np.zeros(n), np.full(n, s), op], 1).astype(np.float32),
             rgb=rng.uniform(0, 1, (n, 3)).astype(np.float32), radii=np.full(n, 4, np.int32),
             depths=np.arange(n, dtype=np.float32) + 1, bg=np.zeros(3, np.float32),
             dL=rng.standard_normal((3, H, W)).astype(np.float32))
    x["conic"][other, 0] = x["conic"][other, 2] = 2.0   # within 8 .. 15
    want = _full(x)
    bad = x["dL"].copy()
    bad[:, 2, 3] = value
    got = _full(x, dL=bad)
    for k in got:
        a, b = np_(got[k]), np_(want[k])
        assert not a[~seen].any() and not b[~seen].any(), k
        # three additions in another order
        assert (np.abs(a[other] - b[other]) <= 6e-7 * np.abs(b[other]).max(initial=0.0)).all(), k
