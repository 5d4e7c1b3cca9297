"""The work that users of this framework have it do, as cases to be timed and compared.

A case is a dict of plain values: `op` (what one pass does), `family` (the kind of splat cloud), its sizes and
options. Clouds, cameras and targets follow the distributions of b2ctrain_amd/scenes.py's workloads, at other
sizes too (the focal length scales with the image), drawn on the GPU from the seed.

  op        one pass
  train     a training step ending in parameter gradients, over `views` poses with the gradients accumulated
  features  the same with the pseudo-normal lanes, the normal-map loss and the hollow loss
  adam      a training iteration ending in the fused update (dense, or lazy sparse Adam)
  eval      a held-out view: a render without backward data, then the squared-error and SSIM sums
  loss      the photometric loss and its gradient on a rendered image
  evidence  the evidence pass with the label vote over `views` views, and its download

  family    after
  cube      scenes.config1: a unit cube of splats ahead of the camera
  ball      scenes.config2: an object in front of an empty background
  box       scenes.config3: a scene around the camera, four splats in ten outside the frustum
  slab      scenes.config4: a deep stack of faint splats on a wall
  wide      scenes.config5: mostly sub-pixel splats, one in twenty a large anisotropic one
"""
import ctypes
import math
from types import SimpleNamespace

import numpy as np
import torch

from b2ctrain_amd import _native
from b2ctrain_amd import scenes as S

C0 = S.SH_C0

# Composited fragments per pixel, and the share of the splats that project into the image, at the sizes of the
# scenes.py workload of each family: (splats, fragments per pixel, most fragments per pixel before a pixel is
# opaque, visible share).
DEPTH = {"cube": (1024, 10.0, 60.0, 1.0), "ball": (100_000, 39.0, 60.0, 0.97), "box": (1_000_000, 69.0, 75.0, 0.63),
         "slab": (3_000_000, 190.0, 190.0, 0.95), "wide": (500_000, 69.0, 75.0, 0.93)}
FLOPS_FWD, FLOPS_BWD = 25, 60  # per composited fragment: sigma, exponential, blend; replay and gradient terms
FLOPS_LOSS = 3 * 2 * (2 * 5 + 2 * 3) * 11  # per pixel: eight maps blurred along both axes by 11 taps, three channels


def _case(name, op, family, n, w, h, degree, fp16=False, view="opaque", views=1, sparse=False, mode=1):
    return dict(name=name, op=op, family=family, n=n, w=w, h=h, degree=degree, fp16=fp16, view=view, views=views,
                sparse=sparse, mode=mode)


def listed():
    return [
        # the smallest call: a unit-sized scene, as in a smoke run or the first steps from a sparse init
        _case("train_tiny", "train", "cube", 1024, 64, 64, 0),
        # an object capture (synthetic turntable views): the ordinary small step
        _case("train_object", "train", "ball", 100_000, 800, 800, 3),
        # the headline step: a full scene at 1080p with soft alpha, weights and a random background
        _case("train_scene", "train", "box", 1_000_000, 1920, 1080, 3, view="transparent"),
        # a mid-sized step at odd sizes from masked photographs, half-precision SH bands, degree 2
        _case("train_masked_odd", "train", "box", 333_333, 1279, 717, 2, fp16=True, view="masked"),
        # a late step on a dense model (deep tile lists), degree 4, two poses accumulated
        _case("train_dense", "train", "slab", 3_000_000, 1920, 1080, 4, views=2),
        # 4K frames with large background splats, half-precision bands
        _case("train_4k", "train", "wide", 500_000, 3840, 2160, 3, fp16=True),
        # normal-map and depth supervision
        _case("train_normals", "features", "ball", 200_000, 1237, 822, 3),
        # the reference's fp32 backward (--backward warp), chosen where gradients are audited
        _case("train_fp32", "train", "ball", 150_000, 960, 540, 1, mode=0),
        # complete iterations with the fused optimizer: dense, and lazy sparse with half-precision bands
        _case("adam_dense", "adam", "box", 1_000_000, 1920, 1080, 3, view="transparent"),
        _case("adam_sparse", "adam", "ball", 250_000, 980, 545, 3, fp16=True, sparse=True),
        # PSNR / SSIM of held-out views during training
        _case("eval_scene", "eval", "box", 600_000, 1600, 900, 3),
        # the per-splat evidence and label vote after training, over a few views
        _case("evidence", "evidence", "ball", 200_000, 960, 720, 3, view="masked", views=8),
    ]


def draw(rng):
    op = rng.choice(["train", "train", "train", "adam", "adam", "features", "eval", "loss", "evidence"])
    family = rng.choice(["cube", "ball", "ball", "box", "box", "slab", "wide"])
    pick = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    w = pick(64, 2600)
    h = max(48, min(1600, int(w * rng.uniform(0.45, 1.3))))
    most = {"cube": 20_000, "ball": 400_000, "box": 1_500_000, "slab": 1_000_000, "wide": 300_000}[family]
    n = pick(900, most)
    if family in ("cube", "slab", "wide"):  # large footprints: fewer pixels keep the lists within the listed range
        w, h = min(w, 1600), min(h, 1000)
    degree = rng.choice([0, 1, 2, 3, 3, 3, 4])
    c = _case("", op, family, n, w, h, degree, fp16=degree > 0 and rng.random() < 0.4,
              view=rng.choice(["opaque", "transparent", "masked"]), views=1, sparse=op == "adam" and rng.random() < 0.5)
    if op == "train" and rng.random() < 0.25:
        c["views"] = 2
    if op == "evidence":
        c["views"] = 4
        c["n"] = min(n, 200_000)
    del c["name"]
    return c


# ---- inputs ----------------------------------------------------------------------------------------------

def _rotations(n, g):
    q = torch.randn(n, 4, generator=g, device="cuda")
    return q / q.norm(dim=1, keepdim=True)


def _cloud(c, g):
    """(positions, opacity logits, log scales, rotations, SH [n][K][3]) of the case's family."""
    n, fam = c["n"], c["family"]
    U = lambda *s: torch.rand(*s, generator=g, device="cuda")  # noqa: E731
    R = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    box = lambda lo, hi: torch.tensor(lo, device="cuda") + U(n, 3) * (torch.tensor(hi, device="cuda") - torch.tensor(lo, device="cuda"))  # noqa: E731
    if fam == "cube":
        pos, op, ls = box([-0.5, -0.5, 2.5], [0.5, 0.5, 3.5]), R(n), -3.0 + 0.5 * R(n, 3)
    elif fam == "ball":
        pos = R(n, 3)
        r = pos.norm(dim=1, keepdim=True)
        pos = torch.where(r > 2, pos / r * 2 * U(n, 1) ** (1 / 3), pos)
        op, ls = -1.0 + 1.5 * R(n), -4.5 + 0.6 * R(n, 3)
    elif fam == "box":
        pos, op, ls = box([-3.0, -2.0, 0.0], [3.0, 2.0, 6.0]), -0.5 + 2.0 * R(n), -5.0 + 0.7 * R(n, 3)
    elif fam == "slab":
        pos, op, ls = box([-2.2, -1.25, -0.25], [2.2, 1.25, 0.25]), -2.0 + R(n), -4.0 + 0.5 * R(n, 3)
    else:
        pos, op, ls = box([-3.0, -1.8, 1.0], [3.0, 1.8, 7.0]), 2.0 * R(n), -7.0 + 0.3 * R(n, 3)
        big = U(n) < 0.05
        axes = torch.tensor([-1.0, -3.0, -6.0], device="cuda")[torch.randint(0, 3, (n, 3), generator=g, device="cuda")]
        ls = torch.where(big[:, None], axes, ls)
    K = (c["degree"] + 1) ** 2
    sh = R(n, K, 3) * 0.05
    sh[:, 0] = (U(n, 3) - 0.5) / C0
    if c["fp16"]:
        sh[:, 1:] = sh[:, 1:].half().float()
    return pos, op, ls, _rotations(n, g), sh


def _cameras(c):
    """`views` poses: the family's own, then small turns about it."""
    w, h = c["w"], c["h"]
    cams = []
    for v in range(c["views"]):
        a = math.radians(4.0 * ((v + 1) // 2) * (-1 if v % 2 else 1))
        if c["family"] == "cube":
            f, eye, at = float(w), (3.0 * math.sin(a), 0.0, 3.0 - 3.0 * math.cos(a)), (0.0, 0.0, 3.0)
        elif c["family"] == "ball":
            f, eye, at = 0.5 * w / math.tan(math.radians(25.0)), (4.0 * math.sin(a), 0.0, -4.0 * math.cos(a)), (0.0, 0.0, 0.0)
        elif c["family"] == "box":
            f, eye, at = 1000.0 * w / 1920, (0.0, 0.0, -0.05), (3.0 * math.sin(a), 0.0, 3.0 * math.cos(a))
        elif c["family"] == "slab":
            f, eye, at = 1000.0 * w / 1920, (2.4 * math.sin(a), 0.1, -2.4 * math.cos(a)), (0.0, 0.0, 0.0)
        else:
            f, eye, at = 2000.0 * w / 3840, (0.0, 0.0, -1.0), (3.0 * math.sin(a), 0.0, 4.0)
        R, t = S.look_at(eye, at)
        cams.append(S.Camera(w, h, f, f, w / 2.0, h / 2.0, R, t))
    return cams


def _bytes(x):
    return torch.floor(x.clamp(0, 1) * 255.0 + 0.5).to(torch.int64)


def _packed(rgb, a):
    """[h][w] RGBA8 words of [h][w][3] colours and [h][w] alpha, as uint32 on the host."""
    q, qa = _bytes(rgb), _bytes(a)
    word = q[..., 0] | (q[..., 1] << 8) | (q[..., 2] << 16) | (qa << 24)
    return word.reshape(-1).cpu().numpy().astype(np.uint32)


def _picture(w, h, g):
    """A photograph-like target: smooth blobs with a little noise, [h][w][3] in [0, 1]."""
    y, x = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float32), torch.arange(w, device="cuda", dtype=torch.float32), indexing="ij")
    u = torch.rand(24, 6, generator=g, device="cuda")
    img = torch.zeros(h, w, 3, device="cuda")
    for k in range(24):
        s = (0.05 + 0.2 * u[k, 2]) * min(w, h)
        img += torch.exp(-((x - u[k, 0] * w) ** 2 + (y - u[k, 1] * h) ** 2) / (2 * s * s))[..., None] * u[k, 3:]
    img = img / img.max().clamp_min(1e-6)
    return (img + 0.02 * torch.randn(h, w, 3, generator=g, device="cuda")).clamp(0, 1)


def _inside(w, h):
    y, x = torch.meshgrid(torch.arange(h, device="cuda") + 0.5, torch.arange(w, device="cuda") + 0.5, indexing="ij")
    return ((((x - w / 2) / (0.4 * w)) ** 2 + ((y - h / 2) / (0.4 * h)) ** 2) <= 1.0).float()


def _inputs(c, seed):
    """The case's scene (host arrays, as a loaded dataset and model have them) and what its options add."""
    g = torch.Generator(device="cuda")
    g.manual_seed(0xB2C0 + int(seed))
    w, h = c["w"], c["h"]
    pos, op, ls, q, sh = _cloud(c, g)
    pic, weights, alpha = _picture(w, h, g), None, torch.ones(h, w, device="cuda")
    if c["view"] != "opaque":
        alpha = _inside(w, h)
        weights = torch.randint(85, 256, (h * w,), generator=g, device="cuda").to(torch.uint8).cpu().numpy()
    if c["view"] == "transparent":
        pic = pic * alpha[..., None]
    zero = torch.zeros(c["n"], 1, device="cuda")
    cams = _cameras(c)
    bg = tuple(torch.rand(3, generator=g, device="cuda").tolist()) if c["view"] == "transparent" else (0.0, 0.0, 0.0)
    host = lambda x: x.contiguous().cpu().numpy()  # noqa: E731
    sc = S.Scene("case", c["degree"], host(torch.cat([pos, op[:, None]], 1)), host(q), host(torch.cat([ls, zero], 1)), host(sh),
                 cams[0], _packed(pic, alpha), weights, sh_fp16=c["fp16"], composite=c["view"] == "transparent",
                 mask=c["view"] == "masked", alpha_lane=c["view"] == "transparent",
                 scale=1.5 if c["view"] != "opaque" else 1.0, bg=bg, extra_cams=cams)
    if c["op"] == "features":
        y, x = torch.meshgrid(torch.linspace(-1, 1, h, device="cuda"), torch.linspace(-1, 1, w, device="cuda"), indexing="ij")
        nm = torch.stack([0.6 * torch.sin(3 * x), 0.6 * torch.cos(2 * y), torch.ones_like(x)], -1)
        nm = 0.5 + 0.5 * nm / nm.norm(dim=-1, keepdim=True)
        near = {"cube": 3.0, "ball": 3.6, "box": 2.0, "slab": 2.4, "wide": 3.0}[c["family"]]
        z = near + 0.2 * torch.sin(5 * x) + 0.2 * torch.cos(4 * y)
        sc.normals = _packed(nm, _inside(w, h))
        sc.feat_mode, sc.normal_scale = 1, 0.05 / max(1.0, float(_inside(w, h).sum()))
        sc.hollow_z = host(torch.where(_inside(w, h) > 0, z, torch.inf).reshape(-1))
        sc.hollow_margin, sc.hollow_lam = 0.05, 0.7 / (w * h)
    return sc


class _Raw:
    """A device buffer of a Renderer's context or model, which the tensors made over it keep alive."""

    def __init__(self, owner, ptr, shape, typ):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typ, "data": (ptr, False), "version": 3}


class _Outputs(dict):
    """The outputs of a pass; holds the Renderer whose buffers they are."""

    owner = None


def _tensor(r, field, shape, model=False, typ="<f4"):
    """A tensor over one of the context's (or the model's) device buffers, without a copy."""
    ptr, _ = r.device_ptr(field, model=model)
    return torch.as_tensor(_Raw(r, ptr, shape, typ), device="cuda")


def _planes(r, field):
    """A planar [lanes][capacity] array of the model."""
    ptr, size = r.device_ptr(field, model=True)
    half = field.endswith("_hi")
    return torch.as_tensor(_Raw(r, ptr, (size // (2 if half else 4),), "<f2" if half else "<f4"), device="cuda")


def prepare(case, seed):
    sc = _inputs(case, seed)
    r = _native.Renderer(sc)
    s = SimpleNamespace(case=case, r=r, cams=sc.extra_cams, bg=sc.bg, out=None)
    w, h = case["w"], case["h"]
    if case["op"] == "adam":
        s.opts = _native.adam_opts(sparse=int(case["sparse"]), lr_mean=2e-5, noise_weight=1e-3, noise_clamp=0.01, seed=7)
    elif case["op"] == "loss":  # a render close to its target, as after some training
        g = torch.Generator(device="cuda")
        g.manual_seed(int(seed) + 17)
        r.write("out_rgba", _rendered(sc, g).cpu().numpy())
        s.lo = r.loss_opts(3.0 * w * h)
    elif case["op"] == "evidence":
        yy, xx = np.divmod(np.arange(w * h), w)
        labels = ((xx // 64 + 3 * (yy // 64)) % 29).astype(np.uint8)
        s.views = [_native.View(w, h, sc.gt, sc.weights, labels=labels, has_alpha=True, masked=True) for _ in s.cams]
    return s


def _rendered(sc, g):
    word = torch.from_numpy(sc.gt.astype(np.int64)).cuda()
    rgba = torch.stack([(word >> k) & 255 for k in (0, 8, 16, 24)], -1).float() / 255.0
    return (rgba + 0.08 * torch.randn(rgba.shape, generator=g, device="cuda")).contiguous()


# ---- one pass ----------------------------------------------------------------------------------------------

def _outputs(s):
    c, r = s.case, s.r
    P, n = c["w"] * c["h"], c["n"]
    if c["op"] == "loss":
        return {"loss": _tensor(r, "loss_accum", (1,)), "v_out": _tensor(r, "v_out", (P, 4))}
    if c["op"] == "eval":
        return {"image": _tensor(r, "out_rgba", (P, 4)), "sums": _tensor(r, "loss_accum", (16,))[4:6]}
    out = {"image": _tensor(r, "out_rgba", (P, 4)), "loss": _tensor(r, "loss_accum", (16,))[:4]}
    if c["op"] != "adam":
        out["grads"] = _tensor(r, "grads", (n, 11 + 3 * (c["degree"] + 1) ** 2))
        return out
    for f in ("pos_op", "quat", "lscale", "m_pos_op", "v_pos_op", "m_quat", "m_lscale"):
        out[f] = _tensor(r, f, (n, 4), model=True)
    bands = ([] if c["degree"] == 0 else ["sh_hi", "m_sh_hi"] if c["fp16"] else ["sh_hi32", "m_sh_hi32"])
    for f in ["sh_dc", "m_sh_dc"] + bands:
        out[f] = _planes(r, f)
    return out


def run(state):
    s, r, c = state, state.r, state.case
    if c["op"] == "evidence":
        e = r.compute_evidence(s.views, s.cams, export_labels=True)
        votes = r.download_labels()
        return {"evidence": e, "class": votes[:, 0].astype(np.int32), "share": votes[:, 1].copy()}
    if c["op"] in ("train", "features"):
        for v, cam in enumerate(s.cams):
            r.step(mode=c["mode"], cam=cam, bg=s.bg, accumulate=v > 0)
    elif c["op"] == "adam":
        s.opts.step += 1
        r.step_adam(s.opts, mode=c["mode"], cam=s.cams[0], bg=s.bg)
    elif c["op"] == "eval":
        r.zero("loss_accum")
        r.forward(cam=s.cams[0], bg=s.bg, bwd_info=False)
        r.eval_metrics(mask_weighted=c["view"] == "masked")
    else:
        r.zero("loss_accum")
        _native.check(r.L.b2c_photometric_loss(r.ctx, r.view, ctypes.byref(s.lo)), "photometric_loss")
    if s.out is None:  # the buffers stay where they are from the first pass on
        s.out = _Outputs(_outputs(s))
        s.out.owner = r
    return s.out


# ---- what a pass cannot do without ---------------------------------------------------------------------------

def work(case):
    n, P, K = case["n"], case["w"] * case["h"], (case["degree"] + 1) ** 2
    op, views = case["op"], case["views"]
    sh = 12 + (2 if case["fp16"] else 4) * 3 * (K - 1)
    n0, per_px, most, seen = DEPTH[case["family"]]
    frags = min(most, per_px * n / n0) * P * views
    target = (4 if case["view"] == "opaque" else 5) * P  # RGBA8 and, with weights, a byte
    if op == "loss":
        return {"bytes": 16 * P + target + 16 * P, "flops": FLOPS_LOSS * P}
    model = 48 * n + sh * seen * n  # parameters in; the bands of the splats in view
    if op == "eval":
        return {"bytes": model + 16 * P + target, "flops": FLOPS_FWD * frags + 3 * 2 * 2 * 5 * 11 * P}
    if op == "evidence":
        return {"bytes": model * views + (target + P) * views + 36 * n, "flops": (2 * FLOPS_FWD + 8) * frags}
    flops = (FLOPS_FWD + FLOPS_BWD) * frags + FLOPS_LOSS * P * views
    per_view = model + target + 16 * P  # and the image
    if op == "adam":  # parameters, moments and the SH's, each read and written
        touched = seen * n if case["sparse"] else n
        return {"bytes": per_view + touched * 2 * (48 + 96 + 2 * sh + 4), "flops": flops}
    if op == "features":
        per_view += 8 * P  # the normal map and the reference depth
    return {"bytes": per_view * views + 4 * n * (11 + 3 * K), "flops": flops}


def tolerance(case):
    op = case["op"]
    if op == "loss":
        return {"rel": 2e-3, "max": 0.9}  # a pixel at its target takes either sign of the L1 term
    if op == "eval":
        return {"rel": 1e-4, "max": 0.02}
    if op == "evidence":
        return {"rel": 1e-3, "max": 0.1, "differ": 1e-4}
    # gradients: a fragment at the 1/255 cutoff, or a pixel at the transmittance stop, falls on either side of it
    # with another rounding, and takes its whole share of one splat's gradient with it (positions moved by one
    # rounding: 1e-6 to 8e-4 over the listed cases, single entries by more than their size)
    return {"rel": 3e-3, "max": 0.95}


# ---- the same in 64 bits -------------------------------------------------------------------------------------

def _basis(d, degree):
    x, y, z = d.unbind(1)
    b = [torch.full_like(x, C0)]
    if degree >= 1:
        b += [-0.48860251190292 * y, 0.48860251190292 * z, -0.48860251190292 * x]
    if degree >= 2:
        b += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z, 0.94617469575756 * z * z - 0.31539156525252,
              -1.0925484305920792 * x * z, 0.5462742152960396 * (x * x - y * y)]
    if degree >= 3:
        b += [-0.5900435899266435 * y * (3 * x * x - y * y), 2.890611442640554 * x * y * z,
              -0.4570457994644658 * y * (5 * z * z - 1), 0.3731763325901154 * z * (5 * z * z - 3),
              -0.4570457994644658 * x * (5 * z * z - 1), 1.445305721320277 * z * (x * x - y * y),
              -0.5900435899266435 * x * (x * x - 3 * y * y)]
    return torch.stack(b, 1)


def _blur(x):
    """The 11-tap Gaussian (sigma 1.5) along both axes of [3][h][w], zero outside."""
    k = torch.exp(-(torch.arange(11, device=x.device, dtype=x.dtype) - 5) ** 2 / (2 * 1.5 * 1.5))
    k = k / k.sum()
    x = torch.nn.functional.pad(x, (5, 5, 5, 5))
    h, w = x.shape[1] - 10, x.shape[2] - 10
    x = sum(k[d] * x[:, :, d:d + w] for d in range(11))
    return sum(k[d] * x[:, d:d + h] for d in range(11))


def _loss64(sc, rgba):
    """The photometric loss of [P][4] rendered pixels: weighted L1 and SSIM, and the alpha match."""
    w, h = sc.W, sc.H
    word = torch.from_numpy(sc.gt.astype(np.int64)).cuda()
    gt = torch.stack([(word >> k) & 255 for k in (0, 8, 16, 24)], -1).double() / 255.0
    bg = torch.tensor([float(np.float32(b)) for b in sc.bg], dtype=torch.float64, device="cuda")
    target = gt[:, :3] + (1 - gt[:, 3:]) * bg if sc.composite else gt[:, :3]
    wp = torch.ones(w * h, dtype=torch.float64, device="cuda") if sc.weights is None else torch.from_numpy(sc.weights).cuda().double() / 255.0
    m = (wp * (gt[:, 3] if sc.mask else 1.0)) * sc.scale / (3.0 * w * h)
    p, t = (x.t().reshape(3, h, w) for x in (rgba[:, :3], target))
    mu1, mu2 = _blur(p), _blur(t)
    s1, s2, s12 = (_blur(p * p) - mu1 * mu1).clamp_min(0), (_blur(t * t) - mu2 * mu2).clamp_min(0), _blur(p * t) - mu1 * mu2
    ssim = ((2 * mu1 * mu2 + 1e-4) * (2 * s12 + 9e-4)) / ((mu1 * mu1 + mu2 * mu2 + 1e-4) * (s1 + s2 + 9e-4))
    each = sc.l1_w * (p - t).abs() + sc.ssim_w * ssim.clamp(-1, 1)
    loss = (m.reshape(h, w) * each).sum()
    if sc.alpha_lane:
        loss = loss + (wp * (rgba[:, 3] - gt[:, 3]).abs()).sum() * sc.match_alpha_weight * sc.scale / (w * h)
    return loss


def _render64(sc, cam, par):
    """[P][4] pixels by brute force: every splat at every pixel, front to back."""
    f64 = lambda a: torch.from_numpy(np.asarray(a, np.float32)).cuda().double()  # noqa: E731
    pos, logit, q, ls, sh = par
    g = S.camera_gpu(cam)
    R, o = f64(g["R"]).reshape(3, 3), f64(g["pos"])
    fx, fy, cx, cy = (float(g[k]) for k in ("fx", "fy", "cx", "cy"))
    d = pos - o
    c = d @ R.t()
    z = c[:, 2]
    seen = z >= 0.01
    z = torch.where(seen, z, torch.ones_like(z))
    x, y = c[:, 0] / z, c[:, 1] / z
    tx = x.clamp(float(g["lim_neg_x"]), float(g["lim_pos_x"]))
    ty = y.clamp(float(g["lim_neg_y"]), float(g["lim_pos_y"]))
    qw, qx, qy, qz = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    rot = torch.stack([1 - 2 * (qy * qy + qz * qz), 2 * (qx * qy - qw * qz), 2 * (qx * qz + qw * qy),
                       2 * (qx * qy + qw * qz), 1 - 2 * (qx * qx + qz * qz), 2 * (qy * qz - qw * qx),
                       2 * (qx * qz - qw * qy), 2 * (qy * qz + qw * qx), 1 - 2 * (qx * qx + qy * qy)], 1).reshape(-1, 3, 3)
    ax = (R @ rot) * torch.exp(ls)[:, None, :]
    ux = (fx / z)[:, None] * (ax[:, 0] - tx[:, None] * ax[:, 2])
    uy = (fy / z)[:, None] * (ax[:, 1] - ty[:, None] * ax[:, 2])
    a, b, e = (ux * ux).sum(1) + 0.3, (ux * uy).sum(1), (uy * uy).sum(1) + 0.3
    det = a * e - b * b
    k00, k01, k11 = e / det, -b / det, a / det
    op = torch.sigmoid(logit)
    colour = (_basis(d / d.norm(dim=1, keepdim=True), sc.degree)[:, :, None] * sh).sum(1) + 0.5
    colour = colour.clamp_min(0)
    w, h = sc.W, sc.H
    yy, xx = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float64) + 0.5, torch.arange(w, device="cuda", dtype=torch.float64) + 0.5, indexing="ij")
    order = torch.argsort(z.detach(), stable=True)
    dx = xx.reshape(-1, 1) - (fx * x + cx)[order]
    dy = yy.reshape(-1, 1) - (fy * y + cy)[order]
    sigma = 0.5 * (k00[order] * dx * dx + k11[order] * dy * dy) + k01[order] * dx * dy
    raw = op[order] * torch.exp(-sigma)
    alpha = torch.where((raw >= 1.0 / 255.0) & seen[order], raw.clamp_max(float(np.float32(0.999))), torch.zeros_like(raw))
    after = torch.cumprod(1 - alpha, 1)
    keep = after > 1e-4  # a fragment that would leave less ends the pixel, uncomposited
    before = torch.cat([torch.ones_like(after[:, :1]), after[:, :-1]], 1)
    vis = torch.where(keep, alpha * before, torch.zeros_like(alpha))
    left = torch.where(keep, 1 - alpha, torch.ones_like(alpha)).prod(1)
    bg = torch.tensor([float(np.float32(v)) for v in sc.bg], dtype=torch.float64, device="cuda")
    return torch.cat([vis @ colour[order] + left[:, None] * bg, 1 - left[:, None]], 1)


def exact(case, seed):
    P = case["w"] * case["h"]
    if case["op"] == "loss":
        sc = _inputs(case, seed)
        g = torch.Generator(device="cuda")
        g.manual_seed(int(seed) + 17)
        rgba = _rendered(sc, g).double().requires_grad_()
        loss = _loss64(sc, rgba)
        loss.backward()
        return {"loss": loss.detach().reshape(1), "v_out": rgba.grad * (3.0 * P)}
    if case["op"] != "train" or case["views"] != 1 or case["degree"] > 3 or case["n"] * P > 20_000_000:
        return None
    sc = _inputs(case, seed)
    f64 = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda().double().requires_grad_()  # noqa: E731
    par = [f64(sc.pos_op[:, :3]), f64(sc.pos_op[:, 3]), f64(sc.quat), f64(sc.lscale[:, :3]), f64(sc.sh)]
    rgba = _render64(sc, sc.extra_cams[0], par)
    loss = _loss64(sc, rgba)
    loss.backward()
    grads = torch.cat([p.grad.reshape(case["n"], -1) for p in par], 1)
    value = loss.detach().reshape(1)
    return {"image": rgba.detach(), "loss": torch.cat([value, 0 * value, value, 0 * value + 1]), "grads": grads}
