"""The calls that a training program makes of this package, as measurable cases.

Six kinds of work, each through the entry points such a program uses:
  step      one training step of the split rasterizer: preprocess, render,
            backward (image gradients given, or the L1 + SSIM loss)
  eval      one evaluation view of the full-image rasterizer, no gradients
  full      the full-image rasterizer forward and backward, with the max-count
            output that pruning reads
  ssim      the SSIM loss over a batch, forward and backward
  knn       distCUDA2, which seeds the Gaussians' scales from a point cloud
  adam      one sparse Adam step over the visible Gaussians
  exchange  one rank's side of the screen-space exchange: routing, packing of
            the rows it sends, unpacking of those it gets, and the way back
            of their gradients

listed() holds the sizes; draw() takes more from the same ranges."""
import math

import numpy as np
import torch

DEV = "cuda"
TILE = 16

# ------------------------------------------------------------------- the cases

# Gaussians a camera of each family sees, of all; list entries it blends per
# pixel, both rounded from the listed scenes (they size work() only)
SEEN = {"cube": 1.0, "cluster": 0.5, "aerial": 0.19}
BLENDED = {"cube": 25, "cluster": 60, "aerial": 45}


def listed():
    return [
        # a small object in a small image: latency and launches
        dict(name="step_16k_256", kind="step", family="cube", P=16384, W=256, H=256, degree=3, loss="given", rows=1,
             white=False),
        # early in training: few Gaussians, low SH degree, odd image size, white background
        dict(name="step_218k_979x546", kind="step", family="aerial", P=217853, W=979, H=546, degree=1, loss="given",
             rows=1, white=True),
        # an object-scale scene of wide Gaussians with the training loss
        dict(name="step_1m_1080p_loss", kind="step", family="cluster", P=1000000, W=1920, H=1080, degree=3,
             loss="l1_ssim", rows=1, white=False),
        # the city-scale aerial step that the benchmark times
        dict(name="step_6m_1600x1066", kind="step", family="aerial", P=6000000, W=1600, H=1066, degree=3,
             loss="given", rows=1, white=False),
        # one of four ranks' share of a 4K image: a block of tile rows
        dict(name="step_8m_4k_rows", kind="step", family="aerial", P=8000000, W=4096, H=2730, degree=3, loss="given",
             rows=4, white=False),
        # a test view of a trained city-scale scene
        dict(name="eval_6m_1600x1066", kind="eval", family="aerial", P=6000000, W=1600, H=1066, degree=3,
             white=False),
        # full-image training step of a middle-sized scene, with the counts that pruning reads
        dict(name="full_2m_1237x822", kind="full", family="aerial", P=2000000, W=1237, H=822, degree=3, white=False),
        # the SSIM term over a batch of full-HD images
        dict(name="ssim_8x3x1080x1920", kind="ssim", B=8, C=3, W=1920, H=1080, padding="same"),
        # scene initialisation from a large point cloud, and from a usual SfM one
        dict(name="knn_10m", kind="knn", family="aerial", P=10000000),
        dict(name="knn_100k", kind="knn", family="cluster", P=100003),
        # the optimiser step of the city-scale scene
        dict(name="adam_6m", kind="adam", P=6000000, seen=0.19),
        # rank 1 of 4's exchange of a 4K view
        dict(name="exchange_8m_4", kind="exchange", P=8000000, W=4096, H=2730, ranks=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "eval", "full", "ssim", "knn", "knn", "adam", "exchange"])
    image = dict(W=rng.randint(200, 2000), H=rng.randint(150, 1200))
    if kind == "step":
        family = rng.choice(["cube", "cluster", "aerial", "aerial"])
        top = {"cube": 60000, "cluster": 800000, "aerial": 6000000}[family]
        return dict(kind=kind, family=family, P=_log(rng, 5000, top), **image, degree=rng.randint(0, 3),
                    loss=rng.choice(["given", "l1_ssim"]), rows=rng.choice([1, 1, 2, 4]), white=rng.random() < 0.3)
    if kind in ("eval", "full"):
        return dict(kind=kind, family=rng.choice(["cluster", "aerial"]), P=_log(rng, 5000, 1000000), **image,
                    degree=rng.randint(0, 3), white=rng.random() < 0.3)
    if kind == "ssim":
        return dict(kind=kind, B=rng.randint(1, 6), C=rng.choice([1, 3]), **image,
                    padding=rng.choice(["same", "valid"]))
    if kind == "knn":
        return dict(kind=kind, family=rng.choice(["cube", "cluster", "aerial"]), P=_log(rng, 3000, 8000000))
    if kind == "adam":
        return dict(kind=kind, P=_log(rng, 10000, 6000000), seen=round(rng.uniform(0.05, 1.0), 3))
    return dict(kind=kind, P=_log(rng, 20000, 6000000), **image, ranks=rng.randint(2, 8))


# ---------------------------------------------------------------------- scenes

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device=DEV) * (hi - lo) + lo


def _means(family, P, g):
    """Points of a unit cube; of 64 anisotropic clusters in a 10 m box; or of a
    400 m ground plane with 30 % of the points in 200 clusters of 10 m."""
    if family == "cube":
        return _uniform(g, (P, 3), -1.0, 1.0)
    if family == "cluster":
        centre = _uniform(g, (64, 3), -4.0, 4.0)
        axes = torch.exp(math.log(0.6) + 0.4 * torch.randn((64, 3), generator=g, device=DEV))
        turn = torch.linalg.qr(torch.randn((64, 3, 3), generator=g, device=DEV))[0] * axes[:, None, :]
        which = torch.randint(0, 64, (P,), generator=g, device=DEV)
        local = torch.randn((P, 3), generator=g, device=DEV)
        return (centre[which] + (turn[which] * local[:, None, :]).sum(2)).clamp_(-5.0, 5.0)
    m = _uniform(g, (P, 3), -200.0, 200.0)
    m[:, 2] = torch.randn(P, generator=g, device=DEV).abs_() * 15.0
    centre = _uniform(g, (200, 3), -200.0, 200.0)
    centre[:, 2] = 10.0
    n = int(round(0.3 * P))
    d = torch.nn.functional.normalize(torch.randn((n, 3), generator=g, device=DEV), dim=1)
    r = 10.0 * torch.rand((n, 1), generator=g, device=DEV) ** (1.0 / 3.0)
    m[P - n:] = centre[torch.randint(0, 200, (n,), generator=g, device=DEV)] + d * r
    return m


def _camera(family, W, H):
    """View and projection as row-major transposes (points multiply from the left), in float32."""
    if family == "cube":
        at, fwd, right, fov = np.array([0.0, 0.0, -4.0]), np.array([0.0, 0.0, 1.0]), np.array([1.0, 0.0, 0.0]), 60.0
    else:
        if family == "cluster":
            az, el = math.radians(30.0), math.radians(20.0)
            at, fov = 8.0 * np.array([math.cos(el) * math.cos(az), math.cos(el) * math.sin(az), math.sin(el)]), 50.0
        else:
            at, fov = np.array([0.0, -150.0 * math.tan(math.radians(30.0)), 150.0]), 60.0
        fwd = -at / np.linalg.norm(at)
        right = np.cross(fwd, [0.0, 0.0, 1.0])
        right /= np.linalg.norm(right)
    R = np.stack([right, np.cross(fwd, right), fwd], axis=1)
    view = np.eye(4)
    view[:3, :3], view[:3, 3] = R.T, -R.T @ at
    tx = math.tan(math.radians(fov) / 2)
    ty = tx * H / W
    near, far = 0.01, 100.0
    proj = np.zeros((4, 4))
    proj[0, 0], proj[1, 1], proj[3, 2] = 1 / tx, 1 / ty, 1.0
    proj[2, 2], proj[2, 3] = far / (far - near), -far * near / (far - near)
    v = view.T.astype(np.float32)
    on = lambda a: torch.tensor(np.ascontiguousarray(a, np.float32), device=DEV)  # noqa: E731
    return dict(tanfovx=tx, tanfovy=ty, view=on(v), proj=on(v @ proj.T.astype(np.float32)), campos=on(at))


SCALE = {"cube": (-4.0, 0.5, 0.0, 1.0), "cluster": (-3.5, 0.7, 0.0, 1.5), "aerial": (-1.5, 0.8, 0.5, 1.5)}


def _scene(case, seed):
    """Activated parameters as a Gaussian model hands them over, the camera, and the image gradient or target."""
    g, P, W, H = _gen(seed), case["P"], case["W"], case["H"]
    mu, sd, op_mu, op_sd = SCALE[case["family"]]
    s = dict(means3D=_means(case["family"], P, g))
    s["scales"] = torch.exp(mu + sd * torch.randn((P, 3), generator=g, device=DEV))
    s["rotations"] = torch.nn.functional.normalize(torch.randn((P, 4), generator=g, device=DEV), dim=1)
    s["opacities"] = torch.sigmoid(op_mu + op_sd * torch.randn((P, 1), generator=g, device=DEV))
    s["sh"] = torch.randn((P, 16, 3), generator=g, device=DEV)
    s["sh"][:, 0] *= 0.5
    s["sh"][:, 1:] *= 0.05
    image = (3, H, W)
    pix = _uniform(g, image, 0.0, 1.0) if case.get("loss") == "l1_ssim" else torch.randn(image, generator=g, device=DEV)
    mask = None
    gy, gx = (H + TILE - 1) // TILE, (W + TILE - 1) // TILE
    if case.get("rows", 1) > 1:
        per = -(-gy // case["rows"])
        mask = torch.zeros((gy, gx), dtype=torch.bool, device=DEV)
        mask[per:2 * per] = True   # rank 1's block
    return s, _camera(case["family"], W, H), pix, mask


def _settings(case, cam):
    from blitzgs_amd.rasterizer import GaussianRasterizationSettings
    return GaussianRasterizationSettings(
        image_height=case["H"], image_width=case["W"], tanfovx=cam["tanfovx"], tanfovy=cam["tanfovy"],
        bg=torch.full((3,), 1.0 if case["white"] else 0.0, device=DEV), scale_modifier=1.0, viewmatrix=cam["view"],
        projmatrix=cam["proj"], sh_degree=case["degree"], campos=cam["campos"], prefiltered=False, debug=False)


# --------------------------------------------------------------------- prepare

ADAM_WIDTHS = {"xyz": 3, "f_dc": 3, "f_rest": 45, "opacity": 1, "scaling": 3, "rotation": 4}
ROW_WIDTHS = [2, 3, 4, 1, 1, 3, 3, 4]   # means2D, rgb, conic_opacity, radii, depths, means3D, scales, rotation


def _exchange_inputs(case, seed):
    """Screen-space rows of which a fifth are visible, and the tile-row
    strategy's bounds.  Every seed has the same rows and radii, at other
    Gaussians, so that as many rows travel."""
    g, P, W, H = _gen(seed), case["P"], case["W"], case["H"]
    same, n = _gen(P), P // 5
    at = torch.randperm(P, generator=g, device=DEV)[:n]
    fields = [torch.randn((P, w), generator=g, device=DEV) for w in ROW_WIDTHS]
    fields[0] = torch.zeros((P, 2), device=DEV)
    fields[0][at, 0] = _uniform(g, (n,), 0.0, 1.0) * (W - 1)
    fields[0][at, 1] = _uniform(same, (n,), 0.0, 1.0) * (H - 1)
    fields[3] = torch.zeros(P, dtype=torch.int32, device=DEV)
    fields[3][at] = torch.exp(2.0 + 0.8 * torch.randn(n, generator=same, device=DEV)).ceil().int()
    fields[4] = fields[4].reshape(P)
    gy, gx = (H + TILE - 1) // TILE, (W + TILE - 1) // TILE
    per = -(-gy // case["ranks"])
    bounds = [min(gy, per * r) * gx for r in range(case["ranks"] + 1)]
    return fields, torch.tensor(bounds, dtype=torch.int32, device=DEV)


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("step", "eval", "full"):
        from blitzgs_amd.rasterizer import GaussianRasterizer
        s, cam, st["pix"], st["mask"] = _scene(case, seed)
        st["rast"] = GaussianRasterizer(_settings(case, cam))
        if kind != "step":
            s["dc"], s["rest"] = s["sh"][:, :1].contiguous(), s["sh"][:, 1:].contiguous()
            del s["sh"]
        st["params"] = {k: v.requires_grad_(kind != "eval") for k, v in s.items()}
        st["screen"] = torch.zeros((case["P"], 3), device=DEV, requires_grad=kind != "eval")
        if kind == "step":
            st["all_map"] = torch.zeros((case["P"], 5), device=DEV)
        else:
            st["culling"] = torch.zeros(case["P"], dtype=torch.bool, device=DEV)
    elif kind == "ssim":
        g, shape = _gen(seed), (case["B"], case["C"], case["H"], case["W"])
        st["img1"] = torch.rand(shape, generator=g, device=DEV)
        # the target: the rendered image's neighbour, as late in training
        st["img2"] = (st["img1"] + 0.2 * torch.randn(shape, generator=g, device=DEV)).clamp_(0.0, 1.0)
        st["img1"].requires_grad_(True)
    elif kind == "knn":
        st["points"] = _means(case["family"], case["P"], _gen(seed))
    elif kind == "adam":
        from blitzgs_amd.adam import SparseGaussianAdam
        g, P = _gen(seed), case["P"]
        st["params"] = {}
        for k, w in ADAM_WIDTHS.items():
            p = torch.randn((P, w), generator=g, device=DEV).requires_grad_(True)
            p.grad = torch.randn((P, w), generator=g, device=DEV) * 1e-3
            st["params"][k] = p
        st["seen"] = torch.rand(P, generator=g, device=DEV) < case["seen"]
        st["opt"] = SparseGaussianAdam([{"params": [p], "lr": 1e-3, "name": k} for k, p in st["params"].items()],
                                       lr=0.0, eps=1e-15)
    else:
        st["fields"], st["bounds"] = _exchange_inputs(case, seed)
    return st


# ------------------------------------------------------------------------- run

def run(st):
    return _RUN[st["case"]["kind"]](st)


def _loss(case, color, pix):
    from blitzgs_amd.ssim import fused_ssim
    return 0.8 * (color - pix).abs().mean() + 0.2 * (1.0 - fused_ssim(color[None], pix[None]))


def _run_step(st):
    case, p, rast = st["case"], st["params"], st["rast"]
    for v in list(p.values()) + [st["screen"]]:
        v.grad = None
    args = {"avoid_pixel_all2all": False}
    means2D, rgb, conic, radii, depths = rast.preprocess_gaussians(p["means3D"], p["scales"], p["rotations"], p["sh"],
                                                                   p["opacities"], args)
    means2D.retain_grad()
    color, _, _, _, observe, _, _ = rast.render_gaussians(means2D, st["screen"], conic, rgb, st["all_map"], depths,
                                                          radii, st["mask"], st["mask"], args)
    if case["loss"] == "given":
        color.backward(st["pix"])
    else:
        _loss(case, color, st["pix"]).backward()
    return dict(color=color, radii=radii, observe=observe, means2D=means2D.grad, means2D_abs=st["screen"].grad,
                grads={k: v.grad for k, v in p.items()})


def _full(st, counts):
    p = st["params"]
    return st["rast"](means3D=p["means3D"], means2D=st["screen"], opacities=p["opacities"], culling=st["culling"],
                      dc=p["dc"], shs=p["rest"], scales=p["scales"], rotations=p["rotations"], flag_max_count=counts)


def _run_eval(st):
    with torch.no_grad():
        color, radii, _ = _full(st, False)
    return dict(color=color, radii=radii)


def _run_full(st):
    for v in list(st["params"].values()) + [st["screen"]]:
        v.grad = None
    color, radii, counts = _full(st, True)
    color.backward(st["pix"])
    return dict(color=color, radii=radii, counts=counts, means2D=st["screen"].grad,
                grads={k: v.grad for k, v in st["params"].items()})


def _run_ssim(st):
    from blitzgs_amd.ssim import fused_ssim
    st["img1"].grad = None
    loss = 1.0 - fused_ssim(st["img1"], st["img2"], padding=st["case"]["padding"])
    loss.backward()
    return dict(loss=loss, grad=st["img1"].grad)


def _run_knn(st):
    from blitzgs_amd.knn import distCUDA2
    return distCUDA2(st["points"])


def _run_adam(st):
    st["opt"].step(st["seen"], st["case"]["P"])
    return {k: dict(p=p, m=st["opt"].state[p]["exp_avg"], v=st["opt"].state[p]["exp_avg_sq"])
            for k, p in st["params"].items()}


def _run_exchange(st):
    from blitzgs_amd import routing
    case, fields = st["case"], st["fields"]
    ids, counts, _ = routing.local2j_ids_concat(fields[0], fields[3], case["H"], case["W"], st["bounds"],
                                                case["ranks"])
    sent = routing.pack_rows(ids, fields)
    lo, n = counts[0], counts[1]
    types = [torch.int32 if k == 3 else torch.float32 for k in range(len(fields))]
    got = routing.unpack_rows(sent[lo:lo + n], ROW_WIDTHS, types)
    # the way back: the differentiable fields' gradients (rows of those shapes) to their Gaussians
    back = routing.scatter_rows(ids[lo:lo + n], [r for k, r in enumerate(got) if k not in (3, 4)], case["P"])
    return dict(ids=ids, sent=sent, got=got, back=back)


_RUN = dict(step=_run_step, eval=_run_eval, full=_run_full, ssim=_run_ssim, knn=_run_knn, adam=_run_adam,
            exchange=_run_exchange)


# ------------------------------------------------------------- work, tolerance

def work(case):
    kind, P = case["kind"], case.get("P", 0)
    if kind in ("step", "eval", "full"):
        share = 1.0 / case.get("rows", 1)
        px, seen = case["W"] * case["H"] * share, P * SEEN[case["family"]]
        sh = 12 * (case["degree"] + 1) ** 2
        # parameters (SH of what is seen), image and radii; then the image's gradient and every dense gradient
        b = 44 * P + sh * seen + 12 * px + 4 * P
        f = seen * 400 + px * BLENDED[case["family"]] * 20
        if kind != "eval":
            b += 12 * px + sh * seen + (44 + 192 + 12) * P + (8 * P if kind == "step" else 0)
            f += seen * 900 + px * BLENDED[case["family"]] * 60
        return dict(bytes=b, flops=f)
    if kind == "ssim":
        n = case["B"] * case["C"] * case["H"] * case["W"]
        return dict(bytes=4 * n * (2 + 1), flops=n * (2 * 11 * 2 * 8 + 60))
    if kind == "knn":
        return dict(bytes=16 * P, flops=P * 8 * 30)
    if kind == "adam":
        w = sum(ADAM_WIDTHS.values())
        return dict(bytes=P + 28 * w * case["seen"] * P, flops=15 * w * case["seen"] * P)
    w = sum(ROW_WIDTHS)
    sent = 0.25 * P
    return dict(bytes=12 * P + sent * (8 + 8 * w) + sent / case["ranks"] * 8 * w + 76 * P, flops=0)


def tolerance(case):
    """Single precision: sums in another order, and the blend's decisions (an
    entry's 1/255 cut, a pixel's stop at 1e-4) falling the other way at the few
    places that are within rounding of them."""
    kind = case["kind"]
    if kind in ("step", "full"):
        return {"rel": 2e-3, "max": 0.5, "differ": 1e-3}
    if kind == "eval":
        return {"rel": 7e-5, "max": 1e-2, "differ": 1e-5}
    if kind == "ssim":
        return {"rel": 2e-6, "max": 1e-4}
    if kind == "knn":
        return {"rel": 2e-7, "max": 1e-6}
    if kind == "adam":
        return {"rel": 5e-5, "max": 1e-3}
    return "exact"


# ----------------------------------------------------------------------- exact

def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "eval", "full"):
        return _exact_raster(case, seed)
    st = prepare(case, seed) if kind in ("ssim", "knn", "adam") else None
    if kind == "ssim":
        x = st["img1"].detach().double().requires_grad_(True)
        m = _ssim_map64(x, st["img2"].double())
        m = m[..., 5:-5, 5:-5] if case["padding"] == "valid" else m
        loss = 1.0 - m.mean()
        loss.backward()
        return dict(loss=loss.detach(), grad=x.grad)
    if kind == "knn":
        return _exact_knn(st["points"]) if case["P"] <= 250000 else None
    if kind == "adam":
        out, seen = {}, st["seen"][:, None]
        lr = 1e-3 * math.sqrt(1 - 0.999) / (1 - 0.9)
        for k, p in st["params"].items():
            g = p.grad.double()
            m, v = torch.where(seen, 0.1 * g, 0.0), torch.where(seen, 0.001 * g * g, 0.0)
            out[k] = dict(p=torch.where(seen, p.detach().double() - lr * m / (v.sqrt() + 1e-15), p.detach().double()),
                          m=m, v=v)
        return out
    return None   # rows are moved, not computed


def _exact_knn(points):
    x = points.double()
    out = []
    for a in x.split(2048):
        d = sum((a[:, k:k + 1] - x[None, :, k]) ** 2 for k in range(3))
        out.append(d.topk(4, largest=False).values[:, 1:].mean(1))
    return torch.cat(out)


def _ssim_map64(a, b):
    w = torch.exp(-torch.arange(-5, 6, dtype=torch.float64, device=a.device) ** 2 / 4.5)
    w = w / w.sum()

    def blur(t):
        n, c, h, wd = t.shape
        t = t.reshape(n * c, 1, h, wd)
        t = torch.nn.functional.pad(t, (5, 5, 5, 5))
        t = sum(w[k] * t[..., k:k + wd] for k in range(11))
        t = sum(w[k] * t[..., k:k + h, :] for k in range(11))
        return t.reshape(n, c, h, wd)

    mu1, mu2 = blur(a), blur(b)
    s1, s2, s12 = blur(a * a) - mu1 * mu1, blur(b * b) - mu2 * mu2, blur(a * b) - mu1 * mu2
    c1, c2 = 0.01 ** 2, 0.03 ** 2
    return ((2 * mu1 * mu2 + c1) * (2 * s12 + c2)) / ((mu1 * mu1 + mu2 * mu2 + c1) * (s1 + s2 + c2))


def _sh_basis(deg, d):
    x, y, z = d.unbind(1)
    one = torch.ones_like(x)
    b = [0.28209479177387814 * one]
    if deg > 0:
        c = 0.4886025119029199
        b += [-c * y, c * z, -c * x]
    if deg > 1:
        b += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
              0.31539156525252005 * (2 * z * z - x * x - y * y), -1.0925484305920792 * x * z,
              0.5462742152960396 * (x * x - y * y)]
    if deg > 2:
        b += [-0.5900435899266435 * y * (3 * x * x - y * y), 2.890611442640554 * x * y * z,
              -0.4570457994644658 * y * (4 * z * z - x * x - y * y),
              0.3731763325901154 * z * (2 * z * z - 3 * x * x - 3 * y * y),
              -0.4570457994644658 * x * (4 * z * z - x * x - y * y), 1.445305721320277 * z * (x * x - y * y),
              -0.5900435899266435 * x * (x * x - 3 * y * y)]
    return torch.stack(b, 1)


def _exact_raster(case, seed):
    """The rasterizer in 64 bits: projection by torch's autograd, the blend as
    dense products over padded tile lists with its gradient written out."""
    s, cam, pix, mask = _scene(case, seed)
    P, W, H, deg, full = case["P"], case["W"], case["H"], case["degree"], case["kind"] != "step"
    V, PM = cam["view"].double(), cam["proj"].double()
    f32 = lambda v: float(np.float32(v))  # noqa: E731
    tx, ty = f32(cam["tanfovx"]), f32(cam["tanfovy"])
    gx, gy = (W + TILE - 1) // TILE, (H + TILE - 1) // TILE

    def project(v):
        m = v["means3D"]
        t = m @ V[:3, :3] + V[3, :3]
        h = m @ PM[:3] + PM[3]
        w = 1.0 / (h[:, 3] + 1e-7)
        xy = torch.stack([((h[:, 0] * w + 1) * W - 1) * 0.5, ((h[:, 1] * w + 1) * H - 1) * 0.5], 1)
        r, x, y, z = v["rotations"].unbind(1)
        R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - r * z), 2 * (x * z + r * y),
                         2 * (x * y + r * z), 1 - 2 * (x * x + z * z), 2 * (y * z - r * x),
                         2 * (x * z - r * y), 2 * (y * z + r * x), 1 - 2 * (x * x + y * y)], 1).reshape(-1, 3, 3)
        M = R * v["scales"][:, None, :]
        # outside 1.3 times the field of view the clamped coordinate is a constant of the gradient
        tz, fx, fy = t[:, 2], W / (2 * tx), H / (2 * ty)
        held = [torch.where((t[:, k] / tz).abs() > 1.3 * lim,
                            ((t[:, k] / tz).clamp(-1.3 * lim, 1.3 * lim) * tz).detach(), t[:, k])
                for k, lim in ((0, tx), (1, ty))]
        u = (fx / tz)[:, None] * V[:3, 0] - (fx * held[0] / tz ** 2)[:, None] * V[:3, 2]
        q = (fy / tz)[:, None] * V[:3, 1] - (fy * held[1] / tz ** 2)[:, None] * V[:3, 2]
        Mu, Mq = (M * u[:, :, None]).sum(1), (M * q[:, :, None]).sum(1)
        cov = torch.stack([(Mu * Mu).sum(1) + 0.3, (Mu * Mq).sum(1), (Mq * Mq).sum(1) + 0.3], 1)
        d = torch.nn.functional.normalize(m - cam["campos"].double(), dim=1)
        n = (deg + 1) ** 2
        rgb = ((_sh_basis(deg, d)[:, :, None] * v["sh"][:, :n]).sum(1) + 0.5).clamp_min(0.0)
        return t[:, 2], xy, cov, rgb

    def extents(cov, op):
        o = 2 * torch.log(op * 255.0)
        ext = torch.where(o > 0, o.clamp_min(0).sqrt().clamp_max(3.33), 3.33)
        det, mid = cov[:, 0] * cov[:, 2] - cov[:, 1] ** 2, 0.5 * (cov[:, 0] + cov[:, 2])
        rad = ext * (mid + (mid * mid - det).clamp_min(0.01).sqrt()).sqrt()
        return rad, torch.minimum(ext * cov[:, 0].sqrt(), rad), torch.minimum(ext * cov[:, 2].sqrt(), rad)

    def box(lo, hi, n):
        return lo.clamp(0, n).long(), hi.clamp(0, n).long()

    names = ["means3D", "scales", "rotations", "opacities", "sh"]
    seen = []
    with torch.no_grad():
        for ids in torch.arange(P, device=DEV).split(1 << 20):
            ids = ids[(s["means3D"][ids].double() @ V[:3, 2] + V[3, 2]) > 0.2]
            v = {k: s[k][ids].double() for k in names}
            _, xy, cov, _ = project(v)
            _, ex, ey = extents(cov, v["opacities"][:, 0])
            x0, x1 = box(((xy[:, 0] - ex) / TILE).floor(), ((xy[:, 0] + ex) / TILE).ceil(), gx)
            y0, y1 = box(((xy[:, 1] - ey) / TILE).floor(), ((xy[:, 1] + ey) / TILE).ceil(), gy)
            seen.append(ids[(x1 > x0) & (y1 > y0)])
    seen = torch.cat(seen)
    v = {k: s[k][seen].double().requires_grad_(True) for k in names}
    depth, xy, cov, rgb = project(v)
    covl = cov.detach().requires_grad_(True)
    det = covl[:, 0] * covl[:, 2] - covl[:, 1] ** 2
    conic = torch.stack([covl[:, 2] / det, -covl[:, 1] / det, covl[:, 0] / det], 1)
    op = v["opacities"].detach()[:, 0]
    with torch.no_grad():
        rad, ex, ey = extents(covl, op)
        if full:
            x0, x1 = box(((xy[:, 0] - ex) / TILE).floor(), ((xy[:, 0] + ex) / TILE).ceil(), gx)
            y0, y1 = box(((xy[:, 1] - ey) / TILE).floor(), ((xy[:, 1] + ey) / TILE).ceil(), gy)
        else:
            r = rad.ceil()
            x0, x1 = box(((xy[:, 0] - r) / TILE).trunc(), ((xy[:, 0] + r + TILE - 1) / TILE).trunc(), gx)
            y0, y1 = box(((xy[:, 1] - r) / TILE).trunc(), ((xy[:, 1] + r + TILE - 1) / TILE).trunc(), gy)
        wx = x1 - x0
        n = wx * (y1 - y0)
        who = torch.repeat_interleave(torch.arange(len(seen), device=DEV), n)
        k = torch.arange(len(who), device=DEV) - (n.cumsum(0) - n)[who]
        tile = (y0[who] + k // wx[who]) * gx + x0[who] + k % wx[who]
        if mask is not None:
            on = mask.reshape(-1)[tile]
            who, tile = who[on], tile[on]
        order = torch.argsort(depth.detach()[who], stable=True)
        order = order[torch.argsort(tile[order], stable=True)]
        who, tile = who[order], tile[order]
        length = torch.bincount(tile, minlength=gx * gy)
        start = length.cumsum(0) - length
        g2 = dict(xy=xy.detach(), conic=conic.detach(), op=op, rgb=rgb.detach())
        color = torch.zeros((3, gy * TILE, gx * TILE), dtype=torch.float64, device=DEV)
        color += 1.0 if case["white"] else 0.0
        if mask is not None:
            color *= mask.repeat_interleave(TILE, 0).repeat_interleave(TILE, 1)
    tiles = torch.nonzero(length)[:, 0]
    tiles = tiles[torch.argsort(length[tiles], descending=True)]
    lens = length[tiles].tolist()
    batches, at = [], 0
    while at < len(lens):
        k = max(1, (1 << 26) // (256 * lens[at]))
        batches.append(tiles[at:at + k])
        at += k
    inner = torch.arange(256, device=DEV)

    def lists(b):
        L = int(length[b[0]])
        pos = torch.arange(L, device=DEV)[None]
        ok = pos < length[b][:, None]
        idx = who[(start[b][:, None] + pos).clamp_max(len(who) - 1)]
        px = (b % gx)[:, None] * TILE + inner % TILE
        py = (b // gx)[:, None] * TILE + inner // TILE
        dx = g2["xy"][idx, 0][:, :, None] - px[:, None, :]
        dy = g2["xy"][idx, 1][:, :, None] - py[:, None, :]
        con, o = g2["conic"][idx], g2["op"][idx][:, :, None]
        A, B, C = con[..., 0:1], con[..., 1:2], con[..., 2:3]
        power = -0.5 * (A * dx * dx + C * dy * dy) - B * dx * dy
        G = power.exp()
        alpha = (o * G).clamp_max(0.99)
        alpha = torch.where((power <= 0) & (alpha >= 1 / 255) & ok[:, :, None], alpha, 0.0)
        alpha = torch.where((1 - alpha).cumprod(1) >= 1e-4, alpha, 0.0)
        after = (1 - alpha).cumprod(1)
        return idx, px, py, dx, dy, A, B, C, o, G, alpha, after

    with torch.no_grad():
        for b in batches:
            idx, px, py, *_, alpha, after = lists(b)
            w = alpha * after / (1 - alpha)
            c = torch.bmm(w.transpose(1, 2).contiguous(), g2["rgb"][idx])
            color[:, py, px] = c.permute(2, 0, 1) + after[:, -1] * (1.0 if case["white"] else 0.0)
    color = color[:, :H, :W].contiguous()
    out = dict(color=color, radii=None)
    if case["kind"] == "eval":
        return out
    if case.get("loss") == "l1_ssim":
        x = color.clone().requires_grad_(True)
        t = pix.double()
        (0.8 * (x - t).abs().mean() + 0.2 * (1 - _ssim_map64(x[None], t[None]).mean())).backward()
        pix = x.grad
    dpad = torch.nn.functional.pad(pix.double(), (0, gx * TILE - W, 0, gy * TILE - H))
    with torch.no_grad():
        N = len(seen)
        acc = torch.zeros((N, 11), dtype=torch.float64, device=DEV)
        for b in batches:
            idx, px, py, dx, dy, A, B, C, o, G, alpha, after = lists(b)
            d = dpad[:, py, px].permute(1, 2, 0)                     # tiles, pixels, 3
            before = after / (1 - alpha)
            w = alpha * before
            cd = torch.bmm(g2["rgb"][idx], d.transpose(1, 2).contiguous())
            wcd = w * cd
            behind = wcd.flip(1).cumsum(1).flip(1) - wcd
            if case["white"]:
                behind = behind + (after[:, -1] * d.sum(2))[:, None, :]
            da = torch.where(alpha > 0, before * cd - behind / (1 - alpha), 0.0)
            gw = G * o * da
            gmx, gmy = gw * -(A * dx + B * dy), gw * -(C * dy + B * dx)
            if full:   # no conic or opacity gradient where the clamp at 0.99 holds
                da = torch.where(o * G > 0.99, 0.0, da)
                gw = G * o * da
            rows = torch.stack([gmx.sum(2), gmy.sum(2), gmx.abs().sum(2), gmy.abs().sum(2),
                                (-0.5 * gw * dx * dx).sum(2), (-gw * dx * dy).sum(2), (-0.5 * gw * dy * dy).sum(2),
                                (G * da).sum(2)], 2)
            rows = torch.cat([rows, torch.bmm(w, d.contiguous())], 2)
            acc.index_add_(0, idx.reshape(-1), rows.reshape(-1, 11))
    conic.backward(acc[:, 4:7])
    # the reference's inverse carries 1e-7 under the squared determinant
    det2 = det.detach() ** 2
    gcov = covl.grad * (det2 / (det2 + 1e-7))[:, None]
    torch.autograd.backward([cov, xy, rgb], [gcov, acc[:, 0:2].contiguous(), acc[:, 8:11].contiguous()])

    def dense(t, shape):
        g = torch.zeros((P,) + shape, dtype=torch.float64, device=DEV)
        g[seen] = t
        return g

    half = torch.tensor([0.5 * W, 0.5 * H], dtype=torch.float64, device=DEV)
    pad = lambda t: torch.nn.functional.pad(t, (0, 1))  # noqa: E731
    grads = {k: dense(v[k].grad, tuple(v[k].shape[1:])) for k in ("means3D", "scales", "rotations", "sh")}
    grads["opacities"] = dense(acc[:, 7:8], (1,))
    if full:
        sh = grads.pop("sh")
        grads["dc"], grads["rest"] = sh[:, :1], sh[:, 1:]
        return dict(out, counts=None, means2D=dense(pad(acc[:, 0:2] * half), (3,)), grads=grads)
    return dict(out, observe=None, means2D=dense(acc[:, 0:2] * half, (2,)),
                means2D_abs=dense(pad(acc[:, 2:4] * half), (3,)), grads=grads)
