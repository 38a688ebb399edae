"""The work whose speed is followed: what a program built on this framework has it do.

Every case is a dict of plain values.  `prepare(case, seed)` makes what such a program has in
hand (a trainer with its views, a batch, host arrays), `run(state)` is one pass through the
public Python mirror of the C ABI (splatrs_amd.abi), and `exact(case, seed)` is the same
result from plain torch in binary64, where that can be computed in reasonable time.

The kinds of work:

  steps      training iterations on a resident model (the inner loop of train()), then the
             download of the model that a save does
  train      the whole train() loop from a fresh model: steps, densification, opacity reset,
             progress records, in the reference's summation order
  batch      iterations of many scenes and views at once, then the download of every scene
  evaluate   PSNR over held-out views of a resident model, and one rendered image
  functions  the reference's functions with host arrays, one after the other, as a program
             that replaces them one by one calls them
  loss       the photometric loss on device buffers
  points     a model from a point cloud
  scorer     the learned densification's online update: a fit, then the logits of a model

Scenes follow the repository's synthetic configurations: Gaussians in a box seen from outside
("object"), from close by ("room"), or on ellipsoid surfaces ("surface"), with a median screen
size of about 1.4 pixels.
"""
import math

import numpy as np
import torch

from splatrs_amd import abi, scenes
from splatrs_amd import records as rec

DEVICE = "cuda:0"
SH_C0 = 0.28209479177387814

_CTX = None


def context():
    """The process's context: a program holds one, and everything it makes shares it."""
    global _CTX
    if _CTX is None:
        _CTX = abi.Context(0)
    return _CTX


# ---- the cases --------------------------------------------------------------------------

STEPS = dict(kind="steps", sh=3, stats=True, absgrad=False, antialias=False, white=False,
             moments=False, tune=False)


def listed():
    return [
        # 10k Gaussians, 8 views of 256x256 (the small configuration): every launch is short,
        # so launch latency and the chain of small kernels count.  Saved with the optimizer.
        dict(STEPS, name="steps_10k_256", layout="object", n=10_000, width=256, height=256,
             views=8, steps=20, moments=True),
        # an odd-sized model and view with the options that change the step: AbsGS statistics,
        # antialiasing, a white background, a lower active SH degree
        dict(STEPS, name="steps_61k_options", layout="object", n=61_003, width=643, height=481,
             views=3, steps=24, sh=2, absgrad=True, antialias=True, white=True),
        # full training at the size of a real capture: 300k Gaussians on surfaces, 1297x840
        dict(STEPS, name="steps_300k_1297x840", layout="surface", n=300_000, width=1297,
             height=840, views=4, steps=24),
        # the headline: 1M Gaussians at 1920x1080, launch shapes tuned
        dict(STEPS, name="steps_1m_1080p", layout="room", n=1_000_000, width=1920, height=1080,
             views=1, steps=40, stats=False, tune=True),
        # train() as a whole on a small capture, in the reference's summation order
        dict(kind="train", name="train_6k_200x150", n=6_000, width=200, height=150, views=6,
             iterations=120),
        # many scenes and views of uneven size in one step
        dict(kind="batch", name="batch_6x3", scenes=6, per_scene=3, n_lo=20_000, n_hi=200_000,
             steps=6, tune=True),
        # held-out views of a trained model
        dict(kind="evaluate", name="evaluate_300k", layout="surface", n=300_000, width=1297,
             height=840, views=6, sh=3, antialias=False),
        # the reference's functions one by one
        dict(kind="functions", name="functions_20k_400x304", n=20_000, width=400, height=304,
             sh=3, ordered=False),
        # the loss alone, on small training images and on the largest the entry point takes
        dict(kind="loss", name="loss_256", width=256, height=256),
        dict(kind="loss", name="loss_1080p", width=1920, height=1080),
        # a sparse reconstruction's points
        dict(kind="points", name="points_150k", n=150_000),
        # one online update of the learned densification
        dict(kind="scorer", name="scorer_64k", samples=65_536, rows=300_000, batch=4096,
             epochs=4),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed kinds, over their ranges; it costs no more than the largest
    listed one (the model grows with the image, and large models take fewer steps)."""
    kind = rng.choice(["steps", "steps", "steps", "train", "batch", "evaluate", "functions",
                       "loss", "points", "scorer"])
    if kind == "loss":
        pixels = _log_uniform(rng, 48 * 40, 1 << 21)
        width = max(16, min(3000, int(math.sqrt(pixels) * rng.uniform(0.7, 1.8))))
        return dict(kind=kind, width=width, height=max(16, pixels // width))
    if kind == "points":
        return dict(kind=kind, n=_log_uniform(rng, 500, 150_000))
    if kind == "scorer":
        return dict(kind=kind, samples=_log_uniform(rng, 3000, 65_536),
                    rows=_log_uniform(rng, 10_000, 500_000),
                    batch=rng.choice([1024, 2048, 4096]), epochs=rng.randint(1, 4))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(2, 6), per_scene=rng.randint(1, 3),
                    n_lo=_log_uniform(rng, 2000, 20_000), n_hi=_log_uniform(rng, 25_000, 200_000),
                    steps=rng.randint(2, 6), tune=rng.random() < 0.5)
    # an image, and a model of 0.05 to 0.5 Gaussians per pixel
    top = {"train": 40_000, "functions": 300_000, "evaluate": 1_500_000}.get(kind, 1920 * 1080)
    pixels = _log_uniform(rng, 90 * 70, top)
    width = max(64, min(1920, int(math.sqrt(pixels) * rng.uniform(0.8, 1.4))))
    height = max(48, pixels // width)
    n = max(500, int(pixels * rng.uniform(0.05, 0.48)))
    if kind == "train":
        return dict(kind=kind, n=n, width=width, height=height, views=rng.randint(2, 8),
                    iterations=rng.randint(60, 120))
    if kind == "functions":
        return dict(kind=kind, n=n, width=width, height=height, sh=rng.randint(0, 3),
                    ordered=rng.random() < 0.5)
    layout = rng.choice(["object", "surface", "room"])
    if kind == "evaluate":
        return dict(kind=kind, layout=layout, n=min(n, 500_000), width=width, height=height,
                    views=rng.randint(1, 6), sh=rng.randint(0, 3), antialias=rng.random() < 0.3)
    stats = rng.random() < 0.6
    moments = n < 50_000 and rng.random() < 0.5
    return dict(STEPS, layout=layout, n=n, width=width, height=height, views=rng.randint(1, 6),
                steps=rng.randint(8, 16) if moments else rng.randint(12, 28),
                sh=rng.randint(0, 3), stats=stats, absgrad=stats and rng.random() < 0.3,
                antialias=rng.random() < 0.3, white=rng.random() < 0.3, moments=moments,
                tune=rng.random() < 0.3)


# ---- inputs -----------------------------------------------------------------------------

class _Draws:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(int(seed) * 7919 + 12345)

    def uniform(self, shape, lo, hi):
        return torch.rand(shape, generator=self.gen, device=DEVICE) * (hi - lo) + lo

    def normal(self, shape, mu=0.0, sigma=1.0):
        return torch.randn(shape, generator=self.gen, device=DEVICE) * sigma + mu


def _gaussians(d, n, layout, sigma_world):
    """Records on the device: log-scales N(ln sigma_world, 0.6), random rotations, opacities
    and colours of the repository's generators."""
    g = torch.empty((n, rec.NUM_PARAMS), device=DEVICE)
    if layout == "surface":
        centre, radii = d.uniform((20, 3), -0.8, 0.8), d.uniform((20, 3), 0.1, 0.4)
        which = torch.randint(0, 20, (n,), generator=d.gen, device=DEVICE)
        ray = torch.nn.functional.normalize(d.normal((n, 3)), dim=1)
        g[:, 0:3] = centre[which] + ray * radii[which]
        g[:, 10] = d.normal((n,), 2.0, 0.5)
    else:
        half = 5.0 if layout == "room" else 1.0
        g[:, 0:3] = d.uniform((n, 3), -half, half)
        g[:, 10] = d.normal((n,))
    g[:, 3:6] = d.normal((n, 3), math.log(sigma_world), 0.6)
    g[:, 6:10] = torch.nn.functional.normalize(d.normal((n, 4)), dim=1)
    g[:, 11:14] = d.normal((n, 3), 0.5, 0.3)
    g[:, 14:] = d.normal((n, 45), 0.0, 0.05)
    return g


def _model_near(d, g):
    """A model on its way to g: what training starts an iteration from."""
    m = g.clone()
    m[:, 0:3] += d.normal((len(g), 3), 0.0, 0.004)
    m[:, 3:6] += d.normal((len(g), 3), 0.0, 0.1)
    m[:, 10] += d.normal((len(g),), 0.0, 0.3)
    m[:, 11:14] += d.normal((len(g), 3), 0.0, 0.15)
    return m


def _cameras(layout, views, width, height):
    """Cameras on a sphere around an object, or in front of a room it looks into."""
    focal, dist = _focal(layout, width), _distance(layout)
    cams = []
    for k, u in enumerate(scenes.fibonacci_sphere(max(views, 2))[:views]):
        if layout == "room":
            eye, up = (0.6 * u[0], 0.6 * u[1], -dist), (0.0, -1.0, 0.0)
        else:
            eye = (dist * u[0], dist * u[1], dist * u[2])
            up = (0.0, -1.0, 0.0) if abs(u[1]) < 0.99 else (0.0, 0.0, 1.0)
        cams.append(scenes.look_at(width, height, focal, focal, eye, (0.0, 0.0, 0.0), up))
    return cams


def _focal(layout, width):
    return (0.833 if layout == "room" else 1.17) * width


def _distance(layout):
    return 8.0 if layout == "room" else 4.0


def _sigma_world(layout, width):
    return 1.37 * _distance(layout) / _focal(layout, width)


def _renders(ctx, g, cams, sh=3, antialias=False, background=(0.0, 0.0, 0.0)):
    """RGB8 images of the records g (host array) through cams: a capture of the scene."""
    t = abi.Trainer(ctx, g)
    out = []
    for k, c in enumerate(cams):
        t.add_view(c, np.zeros((int(c["height"]), int(c["width"]), 3), np.uint8))
        image = t.render(k, sh, antialias, background)
        out.append((np.clip(image, 0.0, 1.0) * 255.0 + 0.5).astype(np.uint8))
    t.close()
    return out


def _scene(ctx, case, seed):
    """(model to train, cameras, images) of a steps / evaluate case."""
    d = _Draws(seed)
    layout, w, h = case["layout"], case["width"], case["height"]
    truth = _gaussians(d, case["n"], layout, _sigma_world(layout, w))
    model = _model_near(d, truth).cpu().numpy()
    cams = _cameras(layout, case["views"], w, h)
    bg = (1.0, 1.0, 1.0) if case.get("white") else (0.0, 0.0, 0.0)
    images = _renders(ctx, truth.cpu().numpy(), cams, case["sh"], case["antialias"], bg)
    return model, cams, images


def _step_params(case, extent):
    bg = (1.0, 1.0, 1.0) if case["white"] else (0.0, 0.0, 0.0)
    lr = rec.learning_rates(rec.position_lr(1, extent))
    return rec.step_params(case["sh"], lr, accumulate_stats=case["stats"],
                           absgrad=case["absgrad"], antialias=case["antialias"],
                           want_loss=True, background=bg)


def _padded(a, rows):
    """The array with zeros after it, so that every run's has the same shape."""
    out = np.zeros((max(rows, len(a)),) + a.shape[1:], a.dtype)
    out[:len(a)] = a
    return out


def prepare(case, seed):
    return _KINDS[case["kind"]].prepare(case, seed)


def run(state):
    return _KINDS[state["kind"]].run(state)


def work(case):
    return _KINDS[case["kind"]].work(case)


def tolerance(case):
    return _KINDS[case["kind"]].tolerance(case)


def exact(case, seed):
    return _KINDS[case["kind"]].exact(case, seed)


# Pairs of a Gaussian and a pixel that reach it, per Gaussian in view: the ellipse of a
# median Gaussian of 1.4 pixels out to an alpha of 1/255 (the 1M-Gaussian step evaluates 114
# per visible Gaussian).  A pair costs 30 operations forward and 70 backward.
PAIRS = 110


# ---- training steps ---------------------------------------------------------------------

class Steps:
    @staticmethod
    def prepare(case, seed):
        ctx = context()
        model, cams, images = _scene(ctx, case, seed)
        t = abi.Trainer(ctx, model)
        for cam, image in zip(cams, images):
            t.add_view(cam, image)
        params = _step_params(case, scenes.scene_extent(cams))
        if case["tune"]:
            t.tune(0, params)
        return dict(kind="steps", trainer=t, params=params, views=len(cams),
                    steps=case["steps"], moments=case["moments"], stats=case["stats"])

    @staticmethod
    def run(s):
        t = s["trainer"]
        for k in range(s["steps"] - 1):
            t.step(k % s["views"], s["params"], result=False)
        r = t.step((s["steps"] - 1) % s["views"], s["params"])
        out = t.download(moments=s["moments"], stats=s["moments"] and s["stats"])
        out["loss"] = float(r["loss"])
        # counts of the last step: after many steps a Gaussian on the edge of the view may
        # fall on either side, so they are compared as amounts
        out["visible"], out["entries"] = float(r["num_visible"]), float(r["num_entries"])
        return out

    @staticmethod
    def work(case):
        n, px, k = case["n"], case["width"] * case["height"], case["steps"]
        # parameters and both moments read and written once a step (the target image read);
        # the records that a save writes
        seen = n * (0.5 if case["layout"] == "room" else 1.0)
        return dict(bytes=k * (6 * 236 * n + 3 * px) + 236 * n * (3 if case["moments"] else 1),
                    flops=k * 100 * PAIRS * seen)

    @staticmethod
    def tolerance(case):
        # The updates of Adam from a first step are nearly +-lr whatever the gradient's size,
        # so a gradient that cancels to rounding error moves a parameter either way, and the
        # steps that follow see it.  Between the two summation orders of the backward pass,
        # which differ by rounding alone, the parameters are up to 9e-4 apart and the moments,
        # which are gradients, 6e-3 (the largest single differences 0.2 and 1 of the values'
        # root mean square).
        if case["moments"]:
            return dict(rel=2.4e-2, max=0.99, differ=2e-3)
        return dict(rel=3.5e-3, max=0.99, differ=2e-3)

    @staticmethod
    def exact(case, seed):
        px, k = case["width"] * case["height"], case["steps"]
        if k * px > 8e6 or k * case["n"] > 1.1e6:
            return None  # minutes in binary64
        model, cams, images = _scene(context(), case, seed)
        p = _step_params(case, scenes.scene_extent(cams))
        ref = _Ref(model, case["sh"], case["antialias"], p["background"])
        adam = _Adam64(ref.g, p["lr"])
        accum = torch.zeros(case["n"], dtype=torch.float64, device=DEVICE)
        for i in range(k):
            v = i % len(cams)
            loss, grad, mean2d = ref.loss_grad(cams[v], images[v], 0.2)
            scale = torch.tensor([case["width"] * 0.5, case["height"] * 0.5],
                                 dtype=torch.float64, device=DEVICE)
            accum += (mean2d * scale).norm(dim=1)
            ref.g = adam.step(ref.g, grad)
        out = dict(params=ref.g, loss=torch.tensor(loss, dtype=torch.float64))
        if case["moments"]:
            out.update(m=adam.m, v=adam.v)
            if case["stats"] and not case["absgrad"]:
                out["grad_accum"] = accum
        return out


# ---- the train loop ---------------------------------------------------------------------

class Train:
    @staticmethod
    def prepare(case, seed):
        ctx = context()
        d = _Draws(seed)
        w, h, n = case["width"], case["height"], case["n"]
        truth = _gaussians(d, 2 * n, "surface", _sigma_world("object", w))
        cams = _cameras("object", case["views"], w, h)
        images = _renders(ctx, truth.cpu().numpy(), cams)
        # the initial model: one Gaussian per point of a reconstruction of the surfaces
        pick = torch.randperm(2 * n, generator=d.gen, device=DEVICE)[:n]
        xyz = (truth[pick, 0:3] + d.normal((n, 3), 0.0, 0.003)).cpu().numpy()
        rgb = (torch.clamp(truth[pick, 11:14] * SH_C0 + 0.5, 0, 1) * 255).to(torch.uint8)
        init = ctx.from_points(xyz, rgb.cpu().numpy())
        t = abi.Trainer(ctx, init, 3 * n)
        for cam, image in zip(cams, images):
            t.add_view(cam, image)
        it = case["iterations"]
        cfg = abi.TrainConfig.default(
            iterations=it, densify_from_iter=it // 8, densify_until_iter=it - it // 8,
            densification_interval=max(5, it // 6), opacity_reset_interval=it // 2,
            sh_degree_interval=max(1, it // 4), log_interval=max(1, it // 3), seed=seed,
            ordered_backward=1)
        return dict(kind="train", trainer=t, init=init, cfg=cfg,
                    extent=float(scenes.scene_extent(cams)))

    @staticmethod
    def run(s):
        t = s["trainer"]
        t.restore({"params": s["init"]}, 0)
        progress = []
        t.train(s["extent"], s["cfg"], lambda p: progress.append(
            [p.iteration, p.loss, p.ema_loss, p.psnr, p.num_gaussians, p.cloned, p.split,
             p.pruned]))
        out = t.download(moments=True, stats=True)
        rows = len(out["params"])
        out = {k: _padded(a, 6 * len(s["init"])) for k, a in out.items()}
        out["rows"], out["progress"] = rows, np.array(progress, np.float64)
        return out

    @staticmethod
    def work(case):
        n, px, k = case["n"], case["width"] * case["height"], case["iterations"]
        return dict(bytes=k * (6 * 236 * n + 3 * px) + 4 * 236 * n, flops=k * 100 * PAIRS * n)

    @staticmethod
    def tolerance(case):
        # the reference's order fixes every sum, so runs agree to the rounding of binary32
        return dict(rel=1e-5, max=1e-3, differ=1e-4)

    @staticmethod
    def exact(case, seed):
        return None  # which rows are cloned turns on the last bits of the statistics


# ---- batched steps ----------------------------------------------------------------------

class BatchSteps:
    @staticmethod
    def _sizes(case):
        lo, hi, k = math.log(case["n_lo"]), math.log(case["n_hi"]), case["scenes"]
        return [int(math.exp(lo + (hi - lo) * (s + 0.5) / k)) for s in range(k)]

    @staticmethod
    def _views(case):
        """[(scene, width, height)]: resolutions of the batched configuration, larger ones for
        larger scenes."""
        out = []
        for s, n in enumerate(BatchSteps._sizes(case)):
            for j in range(case["per_scene"]):
                fit = [r for r in scenes.RESOLUTIONS if r[0] * r[1] < 14 * n] or \
                    scenes.RESOLUTIONS[:1]
                w, h = fit[-1 - (j % min(3, len(fit)))]
                out.append((s, w, h))
        return out

    @staticmethod
    def prepare(case, seed):
        ctx = context()
        d = _Draws(seed)
        b = abi.Batch(ctx)
        views = BatchSteps._views(case)
        dirs = scenes.fibonacci_sphere(case["per_scene"] + 1)
        for s, n in enumerate(BatchSteps._sizes(case)):
            mine = [(w, h) for ps, w, h in views if ps == s]
            truth = _gaussians(d, n, "object", _sigma_world("object", max(mine)[0]))
            b.add_scene(_model_near(d, truth).cpu().numpy())
            cams = []
            for k, (w, h) in enumerate(mine):
                eye = tuple(4.0 * x for x in dirs[k])
                cams.append(scenes.look_at(w, h, 1.17 * w, 1.17 * w, eye, (0.0, 0.0, 0.0),
                                           (0.0, 0.0, 1.0)))
            for cam, image in zip(cams, _renders(ctx, truth.cpu().numpy(), cams)):
                b.add_view(s, cam, image)
        p = rec.batch_step_params(3, rec.learning_rates(0.0))
        order = list(range(len(views)))
        if case["tune"]:
            b.tune(order, p)
        return dict(kind="batch", batch=b, params=p, order=order, steps=case["steps"],
                    lr_mean=[1.6e-4 * 4.0] * case["scenes"], scenes=case["scenes"])

    @staticmethod
    def run(s):
        b = s["batch"]
        for k in range(s["steps"] - 1):
            b.step(s["order"], s["params"], s["lr_mean"], want_losses=False)
        losses = b.step(s["order"], s["params"], s["lr_mean"])
        return dict(losses=losses,
                    models=[b.download(k)["params"] for k in range(s["scenes"])])

    @staticmethod
    def work(case):
        sizes = BatchSteps._sizes(case)
        px = sum(w * h for _, w, h in BatchSteps._views(case))
        pairs = sum(PAIRS * sizes[s] for s, _, _ in BatchSteps._views(case))
        return dict(bytes=case["steps"] * (6 * 236 * sum(sizes) + 3 * px) + 236 * sum(sizes),
                    flops=case["steps"] * 100 * pairs)

    @staticmethod
    def tolerance(case):
        return dict(rel=3.5e-3, max=0.99, differ=2e-3)  # as for the single-view steps

    @staticmethod
    def exact(case, seed):
        return None  # the listed sizes take over a minute in binary64


# ---- evaluation -------------------------------------------------------------------------

class Evaluate:
    @staticmethod
    def prepare(case, seed):
        ctx = context()
        model, cams, images = _scene(ctx, case, seed)
        t = abi.Trainer(ctx, model)
        for cam, image in zip(cams, images):
            t.add_view(cam, image)
        return dict(kind="evaluate", trainer=t, views=list(range(len(cams))), sh=case["sh"],
                    antialias=case["antialias"])

    @staticmethod
    def run(s):
        mean, each = s["trainer"].evaluate(s["views"], s["sh"], s["antialias"])
        image = s["trainer"].render(s["views"][-1], s["sh"], s["antialias"])
        return dict(mean=float(mean), psnr=each, image=image)

    @staticmethod
    def work(case):
        n, px, k = case["n"], case["width"] * case["height"], case["views"]
        # every view reads the records' active part and its target, one image is written
        words = 11 + 3 * (case["sh"] + 1) ** 2
        return dict(bytes=(k + 1) * 4 * words * n + k * 3 * px + 12 * px,
                    flops=(k + 1) * 30 * PAIRS * n)

    @staticmethod
    def tolerance(case):
        return dict(rel=1e-5, max=1e-3)

    @staticmethod
    def exact(case, seed):
        model, cams, images = _scene(context(), case, seed)
        ref = _Ref(model, case["sh"], case["antialias"], (0.0, 0.0, 0.0))
        each = []
        for cam, image in zip(cams, images):
            got = ref.render(cam)
            want = _target64(image)
            mse = ((got.clamp(0, 1) - want) ** 2).mean()
            each.append(-10.0 * torch.log10(mse))
        each = torch.stack(each)
        return dict(mean=each.mean(), psnr=each, image=got)


# ---- the reference's functions ----------------------------------------------------------

class Functions:
    @staticmethod
    def prepare(case, seed):
        d = _Draws(seed)
        w, h, n = case["width"], case["height"], case["n"]
        truth = _gaussians(d, n, "object", _sigma_world("object", w))
        cam = _cameras("object", 1, w, h)[0]
        target = _renders(context(), truth.cpu().numpy(), [cam], case["sh"])[0]
        return dict(kind="functions", ctx=context(), g=_model_near(d, truth).cpu().numpy(),
                    cam=cam, target=target.astype(np.float32) / np.float32(255.0), width=w,
                    height=h, opts=rec.proj_opts(case["sh"]), ordered=case["ordered"],
                    lr=rec.learning_rates(1.6e-4 * 4.0))

    @staticmethod
    def run(s):
        ctx, g, w, h = s["ctx"], s["g"], s["width"], s["height"]
        settings = rec.raster_settings(w, h)
        proj = ctx.project_all(g, s["cam"], s["opts"])
        b = ctx.bin(proj, w, h)
        image, final_t, n_contrib = ctx.rasterize_forward(proj, b, settings)
        loss, dimage = ctx.photometric_loss(image, s["target"], w, h, 0.2)
        pg, absg = ctx.rasterize_backward(proj, b, settings, final_t, n_contrib, dimage,
                                          ordered=s["ordered"])
        grads = ctx.project_backward_all(g, s["cam"], s["opts"], pg)
        n = len(g)
        acc, denom, radii = (np.zeros(n, t) for t in (np.float32, np.uint32, np.uint32))
        ctx.stats_accumulate(proj, pg, None, w, h, acc, denom, radii)
        p, m, v = g.copy(), np.zeros_like(g), np.zeros_like(g)
        ctx.adam_step(p, grads, m, v, rec.adam_state(), s["lr"])
        words = np.ascontiguousarray(proj).view(np.uint32).reshape(n, 15)
        return dict(screen=words[:, 0:6].view(np.float32).copy(),
                    radius=words[:, 6].astype(np.int64),
                    color=words[:, 7:11].copy().view(np.float32),
                    tiles=words[:, 11:15].astype(np.int64),
                    entries=_padded(b.sorted_entries, 16 * n).astype(np.int64),
                    num_entries=b.num_entries, ranges=b.tile_range.astype(np.int64), image=image, final_t=final_t,
                    n_contrib=n_contrib.astype(np.int64), loss=loss, dimage=dimage,
                    proj_grads=np.ascontiguousarray(pg).view(np.float32).reshape(n, 9),
                    abs_grads=absg, grads=grads, accum=acc, params=p, m=m, v=v)

    @staticmethod
    def work(case):
        n, px = case["n"], case["width"] * case["height"]
        e = 5 * n  # tile entries
        # each function's arrays in and out once
        return dict(bytes=n * (236 + 60) + (60 * n + 16 * e) + (60 * n + 8 * e + 20 * px)
                    + 36 * px + (60 * n + 8 * e + 20 * px + 44 * n) + n * (236 + 36 + 236)
                    + n * (96 + 24) + 7 * 236 * n,
                    flops=100 * PAIRS * n)

    @staticmethod
    def tolerance(case):
        # gradients that cancel: the two summation orders of the backward pass, per array
        return dict(rel=1e-4, max=0.1, differ=1e-3)

    @staticmethod
    def exact(case, seed):
        s = Functions.prepare(case, seed)
        n = case["n"]
        ref = _Ref(s["g"], case["sh"], False, (0.0, 0.0, 0.0))
        loss, grad, leaves, proj, image, dimage = ref.loss_grad(
            s["cam"], torch.from_numpy(s["target"]).to(DEVICE).double(), 0.2, everything=True)
        adam = _Adam64(ref.g, s["lr"])
        p = adam.step(ref.g, grad)
        rows = proj["rows"]

        def full(x):
            out = torch.zeros((n,) + x.shape[1:], dtype=torch.float64, device=DEVICE)
            out[rows] = x
            return out
        screen = full(torch.cat([proj["mean"], proj["conic"], proj["depth"][:, None]], 1))
        color = full(torch.cat([proj["opacity"][:, None], proj["color"]], 1))
        pg = full(torch.cat([leaves[0], leaves[1], leaves[2][:, None], leaves[3]], 1))
        scale = torch.tensor([case["width"] * 0.5, case["height"] * 0.5], dtype=torch.float64,
                             device=DEVICE)
        return dict(screen=screen, color=color, image=image, dimage=dimage,
                    loss=torch.tensor(loss, dtype=torch.float64), proj_grads=pg, grads=grad,
                    accum=(pg[:, 0:2] * scale).norm(dim=1), params=p, m=adam.m, v=adam.v)


# ---- the loss on device buffers ---------------------------------------------------------

class Loss:
    @staticmethod
    def prepare(case, seed):
        d = _Draws(seed)
        w, h = case["width"], case["height"]
        # a smooth picture with detail, and a rendering that is close to it
        low = d.uniform((1, 3, max(2, h // 16), max(2, w // 16)), 0.0, 1.0)
        target = torch.nn.functional.interpolate(low, (h, w), mode="bilinear")[0]
        target = (target.permute(1, 2, 0) + d.normal((h, w, 3), 0.0, 0.05)).clamp(0, 1)
        target = torch.round(target * 255.0) / 255.0
        pred = target + d.normal((h, w, 3), 0.0, 0.04)
        return dict(kind="loss", ctx=context(), pred=pred.contiguous(),
                    target=target.contiguous(), width=w, height=h,
                    loss=torch.zeros(1, device=DEVICE),
                    grad=torch.zeros((h, w, 3), device=DEVICE))

    @staticmethod
    def run(s):
        s["ctx"].photometric_loss_device_noalloc(
            s["pred"].data_ptr(), s["target"].data_ptr(), s["width"], s["height"], 0.2,
            s["loss"].data_ptr(), s["grad"].data_ptr())
        return dict(loss=s["loss"], grad=s["grad"])

    @staticmethod
    def work(case):
        px = case["width"] * case["height"]
        # two images read, the gradient written; 5 + 3 blurred maps of 2 x 11 taps, and the
        # SSIM terms, per channel
        return dict(bytes=36 * px, flops=3 * px * (8 * 44 + 60))

    @staticmethod
    def tolerance(case):
        return dict(rel=1e-4, max=1e-2)

    @staticmethod
    def exact(case, seed):
        s = Loss.prepare(case, seed)
        loss, grad = _loss64(s["pred"].double(), s["target"].double(), 0.2)
        return dict(loss=torch.tensor([loss], dtype=torch.float64), grad=grad)


# ---- a model from points ----------------------------------------------------------------

class Points:
    @staticmethod
    def _cloud(case, seed):
        """Points of a reconstruction: surfaces of uneven density, a few far outliers, a few
        points reported twice."""
        d = _Draws(seed)
        n = case["n"]
        on = _gaussians(d, n, "surface", 0.01)[:, 0:3]
        xyz = on + d.normal((n, 3), 0.0, 0.004)
        far = torch.rand((n, 1), generator=d.gen, device=DEVICE) < 0.02
        xyz = torch.where(far, d.uniform((n, 3), -6.0, 6.0), xyz)
        k = n // 200
        xyz[n - k:] = xyz[:k]
        rgb = torch.randint(0, 256, (n, 3), generator=d.gen, device=DEVICE, dtype=torch.uint8)
        return xyz, rgb

    @staticmethod
    def prepare(case, seed):
        xyz, rgb = Points._cloud(case, seed)
        return dict(kind="points", ctx=context(), xyz=xyz.cpu().numpy(), rgb=rgb.cpu().numpy())

    @staticmethod
    def run(s):
        return s["ctx"].from_points(s["xyz"], s["rgb"])

    @staticmethod
    def work(case):
        n = case["n"]
        # points read, records written; a k-d tree's neighbour search visits a few dozen
        # points per query
        return dict(bytes=n * (15 + 236), flops=n * 40 * 8)

    @staticmethod
    def tolerance(case):
        return dict(rel=1e-6, max=1e-5)

    @staticmethod
    def exact(case, seed):
        xyz, rgb = Points._cloud(case, seed)
        x = xyz.double()
        n = len(x)
        d2 = torch.empty(n, dtype=torch.float64, device=DEVICE)
        for a in range(0, n, 512):
            q = x[a:a + 512]
            d = sum((q[:, None, c] - x[None, :, c]) ** 2 for c in range(3))
            d[torch.arange(len(q)), torch.arange(a, a + len(q))] = math.inf  # not itself
            d2[a:a + 512] = d.topk(min(3, n - 1), dim=1, largest=False).values.mean(1)
        g = torch.zeros((n, rec.NUM_PARAMS), dtype=torch.float64, device=DEVICE)
        g[:, 0:3] = x
        g[:, 3:6] = torch.log(torch.sqrt(d2.clamp(min=1e-7)))[:, None]
        g[:, 6] = 1.0
        g[:, 10] = math.log(0.1 / 0.9)
        g[:, 11:14] = (rgb.double() / 255.0 - 0.5) / SH_C0
        return g


# ---- the learned scorer -----------------------------------------------------------------

class ScorerUpdate:
    @staticmethod
    def _inputs(case, seed):
        d = _Draws(seed)

        def features(n):
            x = d.normal((n, rec.SCORER_FEATURES), 0.0, 0.4)
            x[:, 2] = x[:, 2].abs().clamp(max=1.0)
            x[:, 6] = torch.sigmoid(3.0 * x[:, 6])
            return x
        x = features(case["samples"])
        push = torch.stack([x[:, 0] + 0.5 * x[:, 6], x[:, 11] - x[:, 1], 0.4 - x[:, 6]], 1)
        bits = (push + d.normal(tuple(push.shape), 0.0, 0.3)) > 0
        label = (bits * torch.tensor([1, 2, 4], device=DEVICE)).sum(1).to(torch.uint8)
        weight = d.uniform((case["samples"],), 0.5, 2.0)
        return [a.cpu().numpy() for a in (x, label, weight, features(case["rows"]))]

    @staticmethod
    def prepare(case, seed):
        x, y, w, rows = ScorerUpdate._inputs(case, seed)
        s = abi.Scorer(context(), seed=seed)
        return dict(kind="scorer", scorer=s, init=s.params(), x=x, y=y, w=w, rows=rows,
                    cfg=rec.scorer_fit_config(case["epochs"], case["batch"], seed=seed))

    @staticmethod
    def run(s):
        s["scorer"].set_params(s["init"])
        loss = s["scorer"].fit(s["x"], s["y"], s["w"], s["cfg"])
        return dict(loss=loss, params=s["scorer"].params(),
                    logits=s["scorer"].forward(s["rows"]))

    @staticmethod
    def work(case):
        mac = 12 * 64 + 2 * 64 * 64 + 3 * 64
        k = case["samples"]
        return dict(bytes=53 * k + 60 * case["rows"],
                    flops=case["epochs"] * 6 * mac * k + 2 * mac * case["rows"])

    @staticmethod
    def tolerance(case):
        return dict(rel=1e-2, max=0.3)  # bfloat16 operands through a few dozen updates

    @staticmethod
    def exact(case, seed):
        """The same fit in binary64 without bfloat16 operands (its minibatch order is the
        documented SplitMix64 Fisher-Yates shuffle)."""
        x, y, w, rows = ScorerUpdate._inputs(case, seed)
        s = ScorerUpdate.prepare(dict(case, samples=16, rows=16), seed)["init"]
        p = torch.from_numpy(s).double().requires_grad_(True)
        x, w, rows = (torch.from_numpy(a).double() for a in (x, w, rows))
        bits = torch.from_numpy((y[:, None] >> np.arange(3)) & 1).double()
        n, batch = len(x), min(case["batch"], len(x))
        m, v = torch.zeros_like(p), torch.zeros_like(p)
        state, mask, step, loss = seed, (1 << 64) - 1, 0, 0.0
        for _ in range(case["epochs"]):
            perm = list(range(n))
            for i in range(n - 1, 0, -1):
                state = (state + 0x9e3779b97f4a7c15) & mask
                z = ((state ^ (state >> 30)) * 0xbf58476d1ce4e5b9) & mask
                z = ((z ^ (z >> 27)) * 0x94d049bb133111eb) & mask
                j = (z ^ (z >> 31)) % (i + 1)
                perm[i], perm[j] = perm[j], perm[i]
            losses = []
            for b in range(0, n - batch + 1, batch):
                at = torch.tensor(perm[b:b + batch])
                z = _mlp64(p, x[at])
                each = (torch.nn.functional.softplus(z) - bits[at] * z).sum(1)
                value = (w[at] * each).sum() / batch
                g, = torch.autograd.grad(value, p)
                step += 1
                with torch.no_grad():
                    m.mul_(0.9).add_(0.1 * g)
                    v.mul_(0.999).add_(0.001 * g * g)
                    p -= case.get("lr", 1e-3) * (m / (1 - 0.9 ** step)) / (
                        torch.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
                losses.append(float(value))
            loss = sum(losses) / max(1, len(losses))
        with torch.no_grad():
            return dict(loss=torch.tensor(loss, dtype=torch.float64), params=p.detach(),
                        logits=_mlp64(p, rows))


def _mlp64(p, x):
    at = 0

    def layer(a, nout):
        nonlocal at
        nin = a.shape[1]
        wt = p[at:at + nout * nin].reshape(nout, nin)
        at += nout * nin
        b = p[at:at + nout]
        at += nout
        return a @ wt.T + b
    a = x
    for _ in range(3):
        a = torch.nn.functional.gelu(layer(a, 64), approximate="tanh")
    return layer(a, 3)


_KINDS = dict(steps=Steps, train=Train, batch=BatchSteps, evaluate=Evaluate,
              functions=Functions, loss=Loss, points=Points, scorer=ScorerUpdate)


# ---- the path in binary64 ---------------------------------------------------------------

def _target64(image):
    if isinstance(image, torch.Tensor):
        return image
    return torch.from_numpy(image).to(DEVICE).double() / 255.0


def _blur_matrix(n):
    """11 taps of a Gaussian of sigma 1.5, zero outside the image."""
    x = torch.arange(-5, 6, dtype=torch.float64, device=DEVICE)
    k = torch.exp(-x * x / 4.5)
    k = k / k.sum()
    m = torch.zeros((n, n), dtype=torch.float64, device=DEVICE)
    for t in range(11):
        o = t - 5
        if abs(o) < n:
            m.diagonal(o).fill_(float(k[t]))
    return m


def _loss64(pred, target, lam):
    """(1 - lam) L1 + lam (1 - SSIM) of height x width x 3 images, and d/dpred."""
    h, w, _ = pred.shape
    bh, bw = _blur_matrix(h), _blur_matrix(w)
    x = pred.permute(2, 0, 1).contiguous().requires_grad_(True)
    y = target.permute(2, 0, 1).contiguous()

    def blur(a):
        return torch.stack([bh @ a[c] @ bw for c in range(3)])
    mx, my = blur(x), blur(y)
    sx, sy, sxy = blur(x * x) - mx * mx, blur(y * y) - my * my, blur(x * y) - mx * my
    c1, c2 = 0.01 ** 2, 0.03 ** 2
    ssim = ((2 * mx * my + c1) * (2 * sxy + c2)) / ((mx * mx + my * my + c1) * (sx + sy + c2))
    loss = (1 - lam) * (x - y).abs().mean() + lam * (1 - ssim.mean())
    g, = torch.autograd.grad(loss, x)
    return float(loss), g.permute(1, 2, 0).contiguous()


class _Adam64:
    def __init__(self, g, lr):
        rate = [float(lr[k]) for k in ("mean", "log_scale", "quat", "opacity", "sh_dc", "sh_rest")]
        per = [rate[0]] * 3 + [rate[1]] * 3 + [rate[2]] * 4 + [rate[3]] + [rate[4]] * 3 \
            + [rate[5]] * 45
        self.rate = torch.tensor(per, dtype=torch.float64, device=DEVICE)
        self.m, self.v, self.t = torch.zeros_like(g), torch.zeros_like(g), 0

    def step(self, p, g):
        self.t += 1
        self.m = 0.9 * self.m + 0.1 * g
        self.v = 0.999 * self.v + 0.001 * g * g
        mh, vh = self.m / (1 - 0.9 ** self.t), self.v / (1 - 0.999 ** self.t)
        return p - self.rate * mh / (vh.sqrt() + 1e-15)


def _sh_basis(degree, d):
    x, y, z = d.unbind(1)
    out = [torch.full_like(x, SH_C0)]
    if degree >= 1:
        out += [-0.4886025119029199 * y, 0.4886025119029199 * z, -0.4886025119029199 * x]
    if degree >= 2:
        xx, yy, zz, xy, yz, xz = x * x, y * y, z * z, x * y, y * z, x * z
        out += [1.0925484305920792 * xy, -1.0925484305920792 * yz,
                0.31539156525252005 * (2 * zz - xx - yy), -1.0925484305920792 * xz,
                0.5462742152960396 * (xx - yy)]
    if degree >= 3:
        out += [-0.5900435899266435 * y * (3 * xx - yy), 2.890611442640554 * xy * z,
                -0.4570457994644658 * y * (4 * zz - xx - yy),
                0.3731763325901154 * z * (2 * zz - 3 * xx - 3 * yy),
                -0.4570457994644658 * x * (4 * zz - xx - yy),
                1.445305721320277 * z * (xx - yy), -0.5900435899266435 * x * (xx - 3 * yy)]
    return torch.stack(out, 1)


class _Ref:
    """Projection, tile lists and front-to-back compositing in binary64; gradients by
    autograd."""

    def __init__(self, model, sh, antialias, background):
        self.g = torch.from_numpy(np.asarray(model)).to(DEVICE).double()
        self.sh, self.antialias = sh, antialias
        self.bg = torch.tensor([float(b) for b in background], dtype=torch.float64,
                               device=DEVICE)

    def _project(self, g, cam):
        w, h = int(cam["width"]), int(cam["height"])
        fx, fy, cx, cy = (float(cam[k]) for k in ("fx", "fy", "cx", "cy"))
        rot = torch.from_numpy(np.asarray(cam["rot"], np.float64)).to(DEVICE).reshape(3, 3)
        trans = torch.from_numpy(np.asarray(cam["trans"], np.float64)).to(DEVICE)
        t = g[:, 0:3] @ rot.T + trans
        rows = torch.nonzero(t[:, 2].detach() > 0.2)[:, 0]
        g, t = g[rows], t[rows]
        s = torch.exp(g[:, 3:6])
        qw, qx, qy, qz = torch.nn.functional.normalize(g[:, 6:10], dim=1).unbind(1)
        r = torch.stack([1 - 2 * (qy * qy + qz * qz), 2 * (qx * qy - qw * qz),
                         2 * (qx * qz + qw * qy), 2 * (qx * qy + qw * qz),
                         1 - 2 * (qx * qx + qz * qz), 2 * (qy * qz - qw * qx),
                         2 * (qx * qz - qw * qy), 2 * (qy * qz + qw * qx),
                         1 - 2 * (qx * qx + qy * qy)], 1).reshape(-1, 3, 3)
        m = r * s[:, None, :]
        z = t[:, 2]
        rx, ry = t[:, 0] / z, t[:, 1] / z
        tx, ty = 0.3 * 0.5 * w / fx, 0.3 * 0.5 * h / fy
        cxr = rx.clamp(-(cx / fx + tx), (w - cx) / fx + tx) * z
        cyr = ry.clamp(-(cy / fy + ty), (h - cy) / fy + ty) * z
        zero = torch.zeros_like(z)
        j = torch.stack([fx / z, zero, -fx * cxr / (z * z), zero, fy / z, -fy * cyr / (z * z)],
                        1).reshape(-1, 2, 3)
        u = torch.bmm((j @ rot), m)
        a0 = (u[:, 0] * u[:, 0]).sum(1)
        b = (u[:, 0] * u[:, 1]).sum(1)
        c0 = (u[:, 1] * u[:, 1]).sum(1)
        a, c = a0 + 0.3, c0 + 0.3
        det = a * c - b * b
        conic = torch.stack([c / det, -b / det, a / det], 1)
        opacity = torch.sigmoid(g[:, 10])
        if self.antialias:
            opacity = opacity * torch.sqrt((a0 * c0 - b * b).clamp(min=0) / det)
        mid = 0.5 * (a + c)
        radius = torch.ceil(3 * torch.sqrt(mid + torch.sqrt((mid * mid - det).clamp(min=0.1))))
        mean = torch.stack([fx * rx + cx, fy * ry + cy], 1)
        centre = -(rot.T @ trans)
        ray = torch.nn.functional.normalize(g[:, 0:3] - centre, dim=1)
        k = (self.sh + 1) ** 2
        color = (0.5 + (_sh_basis(self.sh, ray)[:, :, None]
                        * g[:, 11:11 + 3 * k].reshape(-1, k, 3)).sum(1)).clamp(min=0)
        tiles_x, tiles_y = (w + 15) // 16, (h + 15) // 16
        with torch.no_grad():
            lim = torch.tensor([tiles_x, tiles_y], dtype=torch.float64, device=DEVICE)
            lo = torch.minimum(torch.floor((mean - radius[:, None]) / 16).clamp(min=0), lim)
            hi = torch.minimum(torch.ceil((mean + radius[:, None]) / 16).clamp(min=0), lim)
            seen = torch.nonzero((hi > lo).all(1))[:, 0]
        return dict(rows=rows[seen], mean=mean[seen], conic=conic[seen], opacity=opacity[seen],
                    color=color[seen], depth=z[seen], lo=lo[seen].long(), hi=hi[seen].long(),
                    width=w, height=h, tiles_x=tiles_x, tiles_y=tiles_y)

    @staticmethod
    def _tiles(p):
        """Chunks of (tiles, Gaussians of each tile front to back, padded with -1)."""
        span = p["hi"] - p["lo"]
        count = span[:, 0] * span[:, 1]
        who = torch.repeat_interleave(torch.arange(len(count), device=DEVICE), count)
        first = torch.cumsum(count, 0) - count
        k = torch.arange(len(who), device=DEVICE) - first[who]
        tile = (p["lo"][who, 1] + k // span[who, 0]) * p["tiles_x"] + p["lo"][who, 0] \
            + k % span[who, 0]
        by_depth = torch.argsort(p["depth"].detach()[who], stable=True)
        order = by_depth[torch.argsort(tile[by_depth], stable=True)]
        who, tile = who[order], tile[order]
        total = p["tiles_x"] * p["tiles_y"]
        per = torch.bincount(tile, minlength=total)
        start = torch.cumsum(per, 0) - per
        by_size = torch.argsort(per)
        sizes = per[by_size].tolist()
        a = 0
        while a < total:
            b = a + 1
            while b < total and (b + 1 - a) * max(1, sizes[b]) * 256 <= 3e7:
                b += 1
            tiles, most = by_size[a:b], max(1, sizes[b - 1])
            slot = torch.arange(most, device=DEVICE)
            at = (start[tiles][:, None] + slot).clamp(max=max(0, len(who) - 1))
            idx = torch.where(slot < per[tiles][:, None], who[at] if len(who) else at, -1)
            yield tiles, idx
            a = b

    def _composite(self, p, tiles, idx):
        """Colour (tiles x 256 x 3) of the tiles' pixels."""
        q = torch.arange(256, device=DEVICE)
        px = ((tiles % p["tiles_x"]) * 16)[:, None] + q % 16 + 0.5
        py = ((tiles // p["tiles_x"]) * 16)[:, None] + q // 16 + 0.5
        live = idx >= 0
        at = idx.clamp(min=0)
        mean, conic, o = p["mean"][at], p["conic"][at], p["opacity"][at]
        dx = px[:, None, :] - mean[:, :, 0:1]
        dy = py[:, None, :] - mean[:, :, 1:2]
        sigma = 0.5 * (conic[:, :, 0:1] * dx * dx + conic[:, :, 2:3] * dy * dy) \
            + conic[:, :, 1:2] * dx * dy
        og = o[:, :, None] * torch.exp(-sigma)
        with torch.no_grad():
            on = live[:, :, None] & (sigma >= 0) & (og >= 1.0 / 255.0)
        alpha = torch.where(on, og.clamp(max=0.99), torch.zeros_like(og))
        after = torch.cumprod(1 - alpha, 1)
        with torch.no_grad():
            on = on & (after >= 1e-4)
        alpha = torch.where(on, alpha, torch.zeros_like(alpha))
        after = torch.cumprod(1 - alpha, 1)
        before = torch.cat([torch.ones_like(after[:, :1]), after[:, :-1]], 1)
        weight = (alpha * before).transpose(1, 2).contiguous()
        return torch.bmm(weight, p["color"][at]) + after[:, -1, :, None] * self.bg

    @staticmethod
    def _place(p, tiles):
        q = torch.arange(256, device=DEVICE)
        x = ((tiles % p["tiles_x"]) * 16)[:, None] + q % 16
        y = ((tiles // p["tiles_x"]) * 16)[:, None] + q // 16
        return x, y, (x < p["width"]) & (y < p["height"])

    def _image(self, p):
        image = torch.zeros((p["height"], p["width"], 3), dtype=torch.float64, device=DEVICE)
        for tiles, idx in self._tiles(p):
            x, y, inside = self._place(p, tiles)
            image[y[inside], x[inside]] = self._composite(p, tiles, idx)[inside]
        return image

    def render(self, cam):
        with torch.no_grad():
            return self._image(self._project(self.g, cam))

    def loss_grad(self, cam, target, lam, everything=False):
        """(loss, d/drecords, d/dmean2d per record)."""
        g = self.g.detach().requires_grad_(True)
        p = self._project(g, cam)
        keys = ("mean", "conic", "opacity", "color")
        leaf = {k: p[k].detach().requires_grad_(True) for k in keys}
        cut = dict(p, **leaf)
        with torch.no_grad():
            image = self._image(cut)
        loss, dimage = _loss64(image, _target64(target), lam)
        for tiles, idx in self._tiles(cut):
            x, y, inside = self._place(cut, tiles)
            out = self._composite(cut, tiles, idx)
            d = torch.zeros_like(out)
            d[inside] = dimage[y[inside], x[inside]]
            out.backward(d)
        grads = [leaf[k].grad if leaf[k].grad is not None else torch.zeros_like(leaf[k])
                 for k in keys]
        grad, = torch.autograd.grad([p[k] for k in keys], g, grads)
        mean2d = torch.zeros((len(g), 2), dtype=torch.float64, device=DEVICE)
        mean2d[p["rows"]] = grads[0]
        if everything:
            p = {k: v.detach() if isinstance(v, torch.Tensor) else v for k, v in p.items()}
            return loss, grad.detach(), grads, p, image, dimage
        return loss, grad.detach(), mean2d
