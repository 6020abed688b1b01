"""The split render without gradients (gs_render_view, gs_render_view_reserved):
the outputs are the forward's bit for bit, and a backward over its buffers
returns zeros."""
import numpy as np
import pytest
import torch

from blitzgs_amd import _lib, rasterizer
from tests.gpu_helpers import np_, settings_for, to_dev

pytestmark = pytest.mark.gpu

W, H = 150, 70


def _inputs(n=900, seed=3):
    rng = np.random.default_rng(seed)
    s = np.exp(rng.uniform(np.log(0.6), np.log(30.0), n))
    conic = np.stack([1 / s ** 2, np.zeros(n), 1 / (0.7 * s) ** 2, rng.uniform(0.02, 0.95, n)], 1)
    return dict(means2D=to_dev(rng.uniform(-10, [W + 10, H + 10], (n, 2)).astype(np.float32)),
                conic=to_dev(conic.astype(np.float32)), rgb=to_dev(rng.uniform(0, 1, (n, 3)).astype(np.float32)),
                depths=to_dev(rng.uniform(1, 5, n).astype(np.float32)), radii=to_dev(np.ceil(3 * s).astype(np.int32)))


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("capacity", [None, 500, 200000])
def test_view_equals_forward(gpu, capacity, masked):
    """capacity: None, the exact call; 500 does not fit (the exact call follows); 200000 fits."""
    x = _inputs()
    dev = torch.device("cuda:0")
    cl = (to_dev(np.arange(50).reshape(5, 10) % 3 > 0)) if masked else None
    bg = to_dev(np.array([0.2, 0.4, 0.1], np.float32))
    keep, outs = _lib.RESERVE, []
    try:
        for backward in (True, False):
            _lib.RESERVE = _lib.InstanceReserve()
            if capacity is not None:
                _lib.RESERVE.update(dev, capacity)
            zero = torch.full((640,), 7.0, device=dev)
            outs.append(rasterizer._render_forward_raw(bg, H, W, x["means2D"], x["depths"], x["radii"], x["conic"],
                                                       x["rgb"], cl, clear=zero, backward=backward))
            assert not np_(zero).any()
    finally:
        _lib.RESERVE = keep
    a, b = outs
    assert a[0] == b[0] > 500
    for k in range(1, 6):
        assert torch.equal(a[k], b[k]), k
    R, geom, binning, img = b[0], b[6], b[7], b[8]
    dL = torch.ones((3, H, W), device=dev)
    for g in rasterizer._render_backward_raw(bg, R, H, W, x["means2D"], x["conic"], x["rgb"], cl, geom, binning, img, dL)[:4]:
        assert not np_(g).any()


def test_no_grad_render_equals_grad_render(gpu):
    x = _inputs(seed=4)
    cam = dict(H=H, W=W, tanfovx=1.0, tanfovy=0.5, viewmatrix=np.eye(4), projmatrix=np.eye(4), campos=np.zeros(3))
    rs = settings_for(cam, bg=(0.2, 0.4, 0.1))
    n = x["means2D"].shape[0]
    means2D = x["means2D"].requires_grad_(True)
    conic, rgb = x["conic"].requires_grad_(True), x["rgb"].requires_grad_(True)
    absgrad, maps = torch.zeros((n, 3), device="cuda", requires_grad=True), torch.zeros((n, 5), device="cuda")
    call = lambda: rasterizer.render_gaussians(means2D, absgrad, conic, rgb, maps, x["depths"], x["radii"], None,  # noqa: E731
                                               None, rs, {})
    with torch.no_grad():
        view = call()
    grad = call()
    for k, (a, b) in enumerate(zip(view, grad)):
        assert torch.equal(a, b.detach()), k
    grad[0].sum().backward()
    assert all(bool(t.grad.abs().sum() > 0) for t in (means2D, conic, rgb, absgrad))
