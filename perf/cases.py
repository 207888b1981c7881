"""Workloads that users of the renderer run, each through its public entry points.

A case is a dict of plain values.  Its "kind" names the entry point:

  render   ``pyrenderer.Renderer.render_forward``: images of one volume
  step     ``diffdvr.Renderer`` forward, MSE image loss, backward (the training
           step of a torch program); "wrt" says what is optimised: the transfer
           function, the densities, the cameras, or a pre-shaded colour volume
  forward  ``diffdvr.Renderer(gradient_method="forward")``: the same step with
           forward-mode derivatives of the transfer function
  batch    ``batch.BatchPlan.run``: many views of several volumes, image loss and
           gradients in one persistent launch

Volumes are sums of Gaussian blobs in [0, 1] (optionally with noise), rendered
in the box [-0.5, 0.5]^3 from cameras on a sphere of radius 2.5 looking at its
centre with a vertical field of view of 45 degrees.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

FOV_Y = math.radians(45.0)
RADIUS = 2.5
EARLY_OUT = 1.0 - 1e-5
IDENTITY, TEXTURE, LINEAR, GAUSSIAN, PRESHADED = 0, 1, 2, 3, 5
TF_COLUMNS = {IDENTITY: 2, TEXTURE: 4, LINEAR: 5, GAUSSIAN: 6}
NEAREST, TRILINEAR = 0, 1
BEER_LAMBERT, ALPHA = 0, 1


def _case(name, kind, sizes, views, image, tf, *, rows=1, step=0.5, wrt="", blend=BEER_LAMBERT, filter=TRILINEAR,
          opacity=1.0, noise=0.0, interval=16, loss="l2"):
    """sizes: "XxYxZ" of every volume, separated by spaces; views per volume; image: "WxH" of the views, cycled
    over all views; step in voxels of the volume's x axis; opacity scales the transfer functions' absorption."""
    return dict(name=name, kind=kind, sizes=sizes, views=views, image=image, tf=tf, rows=rows, step=step, wrt=wrt,
                blend=blend, filter=filter, opacity=opacity, noise=noise, interval=interval, loss=loss)


def listed():
    return [
        # one preview image of a small volume: the interactive call, bound by launches and latency
        _case("render_small", "render", "64x64x64", 1, "128x128", LINEAR, rows=5),
        # final images of a large volume with an opaque transfer function (rays end early), alpha blending
        _case("render_large", "render", "256x256x256", 2, "1024x768", TEXTURE, rows=64, blend=ALPHA, opacity=20.0),
        # a training step on a single small view: the per-view loop of the reference's scripts
        _case("step_tf_single", "step", "64x64x64", 1, "128x128", LINEAR, rows=5, wrt="tf"),
        # transfer-function reconstruction from eight views, quarter-voxel steps
        _case("step_tf", "step", "128x128x128", 8, "256x256", TEXTURE, rows=64, step=0.25, wrt="tf"),
        # density reconstruction of a large noisy volume, a mini-batch of views
        _case("step_volume", "step", "256x256x256", 8, "256x256", IDENTITY, wrt="volume", opacity=10.0, noise=0.02),
        # camera calibration: gradients of the viewports through the per-pixel rays; images of odd sizes
        _case("step_camera", "step", "128x128x128", 4, "237x181", GAUSSIAN, rows=4, wrt="camera"),
        # reconstruction of a pre-shaded (colour) volume, a mini-batch of views
        _case("step_preshaded", "step", "128x128x128", 4, "256x256", PRESHADED, wrt="volume"),
        # forward-mode derivatives of a small Gaussian transfer function
        _case("forward_tf", "forward", "96x112x80", 2, "160x160", GAUSSIAN, rows=4, wrt="tf"),
        # the batched launch on the transfer-function reconstruction, L1 loss
        _case("batch_tf", "batch", "128x128x128", 8, "256x256", TEXTURE, rows=64, step=0.25, wrt="tf", loss="l1"),
        # the batched launch on a density reconstruction from many views
        _case("batch_volume", "batch", "256x256x256", 24, "256x256", IDENTITY, wrt="volume", opacity=10.0, noise=0.02,
              interval=8),
        # joint density and transfer-function reconstruction of several volumes, views of uneven sizes
        _case("batch_joint", "batch", "64x64x64 96x96x96 128x128x128 160x160x160 192x192x192", 8,
              "128x128 512x512 256x256 384x384 160x160 320x320 192x192", LINEAR, rows=5, wrt="volume+tf", interval=4),
        # calibration of many cameras of uneven sizes
        _case("batch_camera", "batch", "128x128x128", 96, "64x64 256x256 128x128 512x512 256x256", GAUSSIAN, rows=4,
              wrt="camera", interval=8),
    ]


def draw(rng):
    """One more case of the same kinds, sizes spread over the ranges the listed ones span."""
    limit = max(_cost(c) for c in listed())
    while True:
        kind, wrt = rng.choice([("render", ""), ("render", ""), ("step", "tf"), ("step", "volume"), ("step", "camera"),
                                ("step", "preshaded"), ("step", "volume+tf"), ("forward", "tf"), ("batch", "tf"),
                                ("batch", "volume"), ("batch", "volume+tf"), ("batch", "camera")])
        log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        tf = rng.choice([IDENTITY, TEXTURE, LINEAR, GAUSSIAN])
        rows = {IDENTITY: 1, TEXTURE: rng.choice([16, 33, 64, 256]), LINEAR: rng.randint(2, 9),
                GAUSSIAN: rng.randint(1, 8)}[tf]
        if kind == "forward" and tf == TEXTURE:
            rows = rng.randint(2, 12)
        if wrt == "preshaded":
            tf, rows, wrt = PRESHADED, 1, "volume"
        elif wrt == "camera":
            tf, rows = GAUSSIAN, rng.randint(1, 6)
        n_volumes = rng.randint(1, 4) if kind == "batch" and wrt != "camera" else 1
        top = {"render": 288, "step": 224, "forward": 128, "batch": 208}[kind]
        sizes = []
        for _ in range(n_volumes):
            n = log(24, top)
            sizes.append("%dx%dx%d" % (n, max(16, int(n * rng.uniform(0.7, 1.3))), max(16, int(n * rng.uniform(0.7, 1.3)))))
        views = {"render": rng.randint(1, 3), "step": rng.randint(1, 8), "forward": rng.randint(1, 2),
                 "batch": rng.randint(2, 24)}[kind]
        big = {"render": 1024, "step": 288, "forward": 192, "batch": 400}[kind]
        image = " ".join("%dx%d" % (log(48, big), log(48, big)) for _ in range(rng.randint(2, 5) if kind == "batch" else 1))
        c = _case("", kind, " ".join(sizes), views, image, tf, rows=rows, step=rng.choice([0.25, 0.4, 0.5, 0.7, 1.0]),
                  wrt=wrt, blend=rng.choice([BEER_LAMBERT, BEER_LAMBERT, ALPHA]),
                  filter=NEAREST if kind in ("render", "step") and tf != PRESHADED and wrt != "camera"
                  and rng.random() < 0.15 else TRILINEAR,
                  opacity=rng.choice([1.0, 5.0, 10.0]), noise=rng.choice([0.0, 0.02]),
                  interval=rng.choice([4, 8, 16]) if kind == "batch" else 16, loss=rng.choice(["l1", "l2"])
                  if kind == "batch" else "l2")
        if _cost(c) <= limit:
            del c["name"]
            return c


# ---------------------------------------------------------------------------
# the scene of a case: plain torch, used by prepare and by exact
# ---------------------------------------------------------------------------
def _dims(text):
    return [tuple(int(v) for v in s.split("x")) for s in text.split()]


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _view_list(case):
    """(volume index, width, height) of every view, in order."""
    images, n_volumes = _dims(case["image"]), len(_dims(case["sizes"]))
    return [(i // case["views"], *images[i % len(images)]) for i in range(n_volumes * case["views"])]


def _viewport_rows(i, n, lat_shift=0.0):
    """eye, right, up of camera i of n, spread over the sphere on a golden-angle spiral (numpy float64)."""
    lat = math.asin(max(-0.9, min(0.9, -1.0 + 2.0 * (i + 1) / (n + 1) + 0.13))) + lat_shift
    lon = (i + 1) * math.pi * (3.0 - math.sqrt(5.0)) + 0.4
    eye = RADIUS * np.array([math.cos(lat) * math.cos(lon), math.sin(lat), math.cos(lat) * math.sin(lon)])
    front = -eye / np.linalg.norm(eye)
    right = np.cross(front, np.array([0.0, 1.0, 0.0]))
    right /= np.linalg.norm(right)
    return np.stack([eye, right, np.cross(right, front)])


def _viewports(case):
    n = len(_view_list(case))
    return torch.tensor(np.stack([_viewport_rows(i, n) for i in range(n)]), dtype=torch.float32)


def _blobs(size, gen, noise):
    """X x Y x Z float32 sum of blobs (plus uniform noise in [0, noise]), clamped to [0, 1], on the GPU."""
    dev = _device()
    k = 16
    centre = 0.2 + 0.6 * torch.rand(k, 3, generator=gen, device=dev, dtype=torch.float64)
    width = 0.05 + 0.1 * torch.rand(k, generator=gen, device=dev, dtype=torch.float64)
    height = 0.3 + 0.7 * torch.rand(k, generator=gen, device=dev, dtype=torch.float64)
    f = []
    for axis, n in enumerate(size):
        p = torch.arange(n, dtype=torch.float64, device=dev) / (n - 1)
        f.append(torch.exp(-(p[None] - centre[:, axis:axis + 1]) ** 2 / (2.0 * width[:, None] ** 2)))
    vol = torch.einsum("kxy,kz->xyz", (height[:, None] * f[0])[:, :, None] * f[1][:, None, :], f[2])
    if noise > 0:
        vol += noise * torch.rand(vol.shape, generator=gen, device=dev, dtype=torch.float64)
    return vol.clamp_(0.0, 1.0).float().contiguous()


def _transfer_function(case, gen):
    """R x C float32: random colours; control points and means spread over [0, 1]."""
    dev, tf, R, opacity = _device(), case["tf"], case["rows"], case["opacity"]
    u = lambda *s: torch.rand(*s, generator=gen, device=dev, dtype=torch.float64)
    if tf == IDENTITY:
        return torch.tensor([[opacity, opacity]], device=dev, dtype=torch.float32)
    rgba = u(R, 4)
    rgba[:, 3] *= opacity
    if tf == TEXTURE:
        return rgba.float().contiguous()
    at = (torch.arange(R, device=dev, dtype=torch.float64) + 0.5 + 0.4 * (u(R) - 0.5)) / R
    if tf == LINEAR:
        at[0], at[-1] = 0.0, 1.0
        return torch.cat([rgba, at[:, None]], 1).float().contiguous()
    return torch.cat([rgba, at[:, None], 0.02 + 0.08 * u(R, 1)], 1).float().contiguous()


def _scene(case, seed):
    """volumes, transfer functions (one per volume), viewports and target images of a case."""
    gen = torch.Generator(device=_device())
    gen.manual_seed(seed)
    sizes = _dims(case["sizes"])
    if case["tf"] == PRESHADED:
        channels = [_blobs(sizes[0], gen, case["noise"]) for _ in range(4)]
        channels[3] = channels[3] * case["opacity"]
        volumes = [torch.stack(channels).contiguous()]
        tfs = [torch.ones(1, 2, device=_device())]
    else:
        volumes = [_blobs(s, gen, case["noise"]) for s in sizes]
        tfs = [_transfer_function(case, gen) for _ in sizes]
    targets = [torch.rand(h, w, 4, generator=gen, device=_device()) for _, w, h in _view_list(case)]
    return volumes, tfs, _viewports(case).to(_device()), targets


def _step(case, volume_index=0):
    return float(np.float32(case["step"] / _dims(case["sizes"])[volume_index][0]))


# ---------------------------------------------------------------------------
# a user's program
# ---------------------------------------------------------------------------
def prepare(case, seed):
    from diffdvr_amd import batch, diffdvr, pyrenderer as pr

    volumes, tfs, viewports, targets = _scene(case, seed)
    views = _view_list(case)
    state = {"kind": case["kind"]}
    if case["kind"] == "batch":
        wrt = case["wrt"]
        like = lambda on, t: torch.zeros_like(t) if on in wrt else None
        vols = [batch.BatchVolume(v, grad=like("volume", v)) for v in volumes]
        luts = [batch.BatchTf(t, grad=like("tf", t)) for t in tfs]
        # the images of all views lie one after the other in one buffer
        first = np.concatenate([[0], np.cumsum([w * h for _, w, h in views])]).tolist()
        color = torch.empty(first[-1], 4, device=_device())
        term = torch.empty(first[-1], dtype=torch.int32, device=_device())
        camera_grad = like("camera", viewports)
        bv = [batch.BatchView(volume=k, tf=k, width=w, height=h, camera=viewports[i], fov_y=FOV_Y, step=_step(case, k),
                              color=color[first[i]:first[i + 1]].view(h, w, 4),
                              termination=term[first[i]:first[i + 1]].view(h, w), target=targets[i],
                              camera_grad=None if camera_grad is None else camera_grad[i])
              for i, (k, w, h) in enumerate(views)]
        loss = torch.zeros(1, device=_device())
        plan = batch.BatchPlan(vols, luts, bv, volume_filter_mode=case["filter"], tf_mode=case["tf"],
                               blend_mode=case["blend"], blending_early_out=EARLY_OUT, loss=case["loss"], loss_out=loss,
                               checkpoint_interval=case["interval"])
        state.update(plan=plan, loss=loss, color=color, term=term,
                     grads=[g for g in [v.grad for v in vols] + [t.grad for t in luts] + [camera_grad] if g is not None])
        return state

    _, W, H = views[0]
    s = pr.RendererInputs()
    s.screen_size = pr.int2(W, H)
    preshaded = case["tf"] == PRESHADED
    volume = volumes[0] if preshaded else volumes[0].unsqueeze(0)
    tf = tfs[0].unsqueeze(0)
    s.volume = volume
    s.volume_filter_mode = pr.VolumeFilterMode.Preshaded if preshaded else pr.VolumeFilterMode(case["filter"])
    s.box_min, s.box_size = pr.real3(-0.5, -0.5, -0.5), pr.real3(1, 1, 1)
    s.step_size = _step(case)
    s.tf_mode = pr.TFMode(case["tf"])
    s.tf = tf
    s.blend_mode = pr.BlendMode(case["blend"])
    s.blending_early_out = EARLY_OUT
    s.camera_mode = pr.CameraMode.ReferenceFrame
    s.camera = pr.CameraReferenceFrame(viewports, FOV_Y)
    if case["kind"] == "render":
        color = torch.empty(len(views), H, W, 4, device=_device())
        term = torch.empty(len(views), H, W, dtype=torch.int32, device=_device())
        state.update(inputs=s, color=color, term=term, outputs=pr.RendererOutputs(color, term))
        return state
    wrt = case["wrt"]
    leaves = {"tf": tf, "volume": volume, "camera": viewports}
    for name, t in leaves.items():
        t.requires_grad_(name in wrt)
    state["renderer"] = diffdvr.Renderer(s, optimize_tf="tf" in wrt, optimize_volume="volume" in wrt,
                                         optimize_camera="camera" in wrt,
                                         gradient_method="forward" if case["kind"] == "forward" else "adjoint")
    state.update(target=torch.stack(targets), viewports=viewports, tf=tf, volume=volume,
                 leaves=[t for t in (volume, tf, viewports) if t.requires_grad])
    return state


def run(state):
    if state["kind"] == "render":
        from diffdvr_amd import pyrenderer as pr
        pr.Renderer.render_forward(state["inputs"], state["outputs"])
        return {"color": state["color"], "term": state["term"]}
    if state["kind"] == "batch":
        state["plan"].run()
        return {"color": state["color"], "term": state["term"], "loss": state["loss"], "grads": state["grads"]}
    image = state["renderer"](camera=state["viewports"], fov_y_radians=FOV_Y, tf=state["tf"], volume=state["volume"])
    loss = torch.nn.functional.mse_loss(image, state["target"])
    grads = torch.autograd.grad(loss, state["leaves"])
    return {"color": image.detach(), "grads": list(grads)}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=256)
def _view_samples(i, n, W, H, step):
    """Samples of one view's rays inside the box (numpy, every fourth pixel in x and y)."""
    eye, right, up = _viewport_rows(i, n)
    front = np.cross(up, right)
    sx, sy = max(1, W // 64), max(1, H // 64)
    x, y = np.meshgrid(np.arange(sx // 2, W, sx), np.arange(sy // 2, H, sy))
    fx = (2.0 * (x + 0.5) / W - 1.0) * math.tan(FOV_Y * W / H / 2.0)
    fy = (2.0 * (y + 0.5) / H - 1.0) * math.tan(FOV_Y / 2.0)
    d = front + fx[..., None] * right + fy[..., None] * up
    d /= np.linalg.norm(d, axis=-1, keepdims=True)
    with np.errstate(divide="ignore"):
        a, b = (-0.5 - eye) / d, (0.5 - eye) / d
    t0, t1 = np.minimum(a, b).max(-1), np.maximum(a, b).min(-1)
    count = np.where(t1 >= t0, np.floor((t1 - t0) / step) + 1.0, 0.0)
    return float(count.mean()) * W * H


def _samples(case):
    views = _view_list(case)
    return sum(_view_samples(i, len(views), w, h, _step(case, k)) for i, (k, w, h) in enumerate(views))


def _flops(case):
    """Arithmetic per sample of the formulas: position 6, trilinear form 21 (per channel), transfer function (lerp of
    four channels 15, Gaussian 15 a row), blend 20; the adjoint of a sample costs about twice its value, and the
    gradient of the eight corners 32 more (per channel)."""
    channels = 4 if case["tf"] == PRESHADED else 1
    tf = {IDENTITY: 6, TEXTURE: 15, LINEAR: 18, GAUSSIAN: 15 * case["rows"], PRESHADED: 0}[case["tf"]]
    value = 6 + 21 * channels + tf + 20
    if case["kind"] == "render":
        return value
    if case["kind"] == "forward":
        return value + 16 * case["rows"] * TF_COLUMNS[case["tf"]]
    return 3 * value + (32 * channels if "volume" in case["wrt"] else 0) + (24 if "camera" in case["wrt"] else 0)


def _cost(case):
    """Relative cost of a case for draw: samples, weighted by what the pass does with each."""
    weight = {"render": 1.0, "step": 3.0, "batch": 3.0,
              "forward": 2.0 + case["rows"] * TF_COLUMNS.get(case["tf"], 1) / 8.0}[case["kind"]]
    if "volume" in case["wrt"]:
        weight *= 8.0 if case["tf"] == PRESHADED else 2.0
    return weight * _samples(case)


def work(case):
    pixels = sum(w * h for _, w, h in _view_list(case))
    channels = 4 if case["tf"] == PRESHADED else 1
    voxels = channels * sum(x * y * z for x, y, z in _dims(case["sizes"]))
    size = 4 * voxels + pixels * 20                          # volumes read, colours and sample counts written
    if case["kind"] != "render":
        size += 16 * pixels                                  # target images
        if "volume" in case["wrt"]:
            size += 4 * voxels
    return {"bytes": int(size), "flops": int(_flops(case) * _samples(case))}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _fetch64(vol, p, filter):
    """vol: C x X x Y x Z float64; p: rays x samples x 3 voxel positions -> C values of that shape."""
    C, X, Y, Z = vol.shape
    flat = vol.reshape(C, -1)
    take = lambda idx: torch.stack([flat[c].index_select(0, idx.reshape(-1)).reshape(idx.shape) for c in range(C)])
    if filter == NEAREST:
        n = torch.tensor([X, Y, Z], dtype=torch.float64, device=p.device)
        i = torch.floor(torch.minimum(p.detach().clamp(min=1e-7), n - (1.0 + 1e-7)) + 0.5).long()
        return take((i[..., 0] * Y + i[..., 1]) * Z + i[..., 2])
    i = p.detach().to(torch.int64)                           # truncation, as the renderer's cell index
    f = p - i.double()
    lo = [i[..., a].clamp(0, n - 1) for a, n in enumerate((X, Y, Z))]
    hi = [(i[..., a] + 1).clamp(0, n - 1) for a, n in enumerate((X, Y, Z))]
    corner = lambda x, y, z: take((x * Y + y) * Z + z)
    lerp = lambda u, v, t: u + t * (v - u)                   # exact where both ends are equal
    rod = lambda y, z: lerp(corner(lo[0], y, z), corner(hi[0], y, z), f[..., 0])
    face = lambda z: lerp(rod(lo[1], z), rod(hi[1], z), f[..., 1])
    return lerp(face(lo[2]), face(hi[2]), f[..., 2])


def _shade64(case, tf, d):
    """Colour and absorption (a list of four) of the densities d through the R x C float64 table."""
    R = tf.shape[0]
    if case["tf"] == IDENTITY:
        inside = (d.detach() > 0) & (d.detach() < 1)
        c = torch.where(inside, d, d.detach().clamp(0, 1))
        return [c * tf[0, 1]] * 3 + [c * tf[0, 0]]
    if case["tf"] == GAUSSIAN:
        out = [0.0] * 4
        for r in range(R):
            g = torch.exp(-(d - tf[r, 4]) ** 2 / (2.0 * tf[r, 5] ** 2))
            out = [o + tf[r, c] * g for c, o in enumerate(out)]
        return out
    # each sample reads one of many copies of the table, so that few of the backward's sums meet on one address
    copies = 1 << 15
    lane = torch.arange(d.numel(), device=d.device).remainder_(copies).reshape(d.shape)
    wide = [tf[:, c, None].expand(R, copies).reshape(-1) for c in range(tf.shape[1])]
    pick = lambda c, idx: wide[c].index_select(0, (idx * copies + lane).reshape(-1)).reshape(idx.shape)
    if case["tf"] == TEXTURE:
        x = d * R - 0.5
        i = torch.floor(x.detach()).long()
        f = x - i.double()
        a, b = i.clamp(0, R - 1), (i + 1).clamp(0, R - 1)
    else:
        a = (torch.searchsorted(tf[:, 4].detach().contiguous(), d.detach().contiguous(), right=True) - 1).clamp(0, R - 2)
        b = a + 1
        f = (d - pick(4, a)) / (pick(4, b) - pick(4, a))
    return [pick(c, a) + f * (pick(c, b) - pick(c, a)) for c in range(4)]


def _march64(case, vol, tf, viewport, W, H, step, rows):
    """Colours (rows of the image as a slice) of one view in float64: len(rows) * W x 4."""
    dev = vol.device
    y, x = torch.meshgrid(rows.double(), torch.arange(W, device=dev, dtype=torch.float64), indexing="ij")
    fx = ((2.0 * (x + 0.5) / W - 1.0) * math.tan(FOV_Y32 * W / H / 2.0)).reshape(-1, 1)
    fy = ((2.0 * (y + 0.5) / H - 1.0) * math.tan(FOV_Y32 / 2.0)).reshape(-1, 1)
    eye, right, up = viewport[0], viewport[1], viewport[2]
    dirs = torch.linalg.cross(up, right)[None] + fx * right[None] + fy * up[None]
    dirs = dirs / dirs.norm(dim=1, keepdim=True)
    with torch.no_grad():
        a, b = (-0.5 - eye)[None] / dirs, (0.5 - eye)[None] / dirs
        t0 = torch.minimum(a, b).amax(1).clamp(min=0.0)
        t1 = torch.maximum(a, b).amin(1)
        # the sample schedule of the renderer: t0, t1 and t0 + i * step rounded to float
        t0f, t1f = t0.float(), t1.float()
        n = torch.where(t1f >= t0f, ((t1f - t0f).double() / step).floor() + 3.0, torch.zeros_like(t0))
        live = torch.nonzero(t1f >= t0f).reshape(-1)
    out = torch.zeros(dirs.shape[0], 4, dtype=torch.float64, device=dev)
    if live.numel() == 0:
        return out
    count = int(n.max().item())
    i = torch.arange(count, device=dev, dtype=torch.float64)[None]
    t = t0[live, None] + i * step
    taken = (t0f[live, None].double() + i * step).float() <= t1f[live, None]
    dims = torch.tensor(vol.shape[1:], dtype=torch.float64, device=dev)
    p = (eye[None, None] + t[..., None] * dirs[live, None, :] + 0.5) * (dims - 1.0)
    value = _fetch64(vol, p, case["filter"])
    c = list(value) if case["tf"] == PRESHADED else _shade64(case, tf, value[0])
    od = torch.where(taken, c[3] * step, torch.zeros_like(c[3]))
    if case["blend"] == BEER_LAMBERT:
        before = torch.cumsum(od, 1)
        before = torch.exp(-torch.cat([torch.zeros_like(before[:, :1]), before[:, :-1]], 1))
        alpha = -torch.expm1(-od)
    else:
        alpha = od.clamp(max=1.0)
        before = torch.cumprod(1.0 - alpha, 1)
        before = torch.cat([torch.ones_like(before[:, :1]), before[:, :-1]], 1)
    w = torch.where(before.detach() >= 1.0 - float(np.float32(EARLY_OUT)), before * alpha, torch.zeros_like(alpha))
    sums = torch.stack([(w * c[0]).sum(1), (w * c[1]).sum(1), (w * c[2]).sum(1), w.sum(1)], 1)
    return out.index_copy(0, live, sums)


FOV_Y32 = float(np.float32(FOV_Y))


def exact(case, seed):
    if _samples(case) * (4 if case["tf"] == PRESHADED else 1) * (case["rows"] if case["tf"] == GAUSSIAN else 1) > 4e9:
        return None
    volumes, tfs, viewports, targets = _scene(case, seed)
    wrt = case["wrt"]
    vols = [(v if v.dim() == 4 else v.unsqueeze(0)).double().requires_grad_("volume" in wrt) for v in volumes]
    luts = [t.double().requires_grad_("tf" in wrt) for t in tfs]
    cams = [viewports[i].double().requires_grad_("camera" in wrt) for i in range(viewports.shape[0])]
    views = _view_list(case)
    elements = 4.0 * sum(w * h for _, w, h in views)
    colors, loss = [], 0.0
    for i, (k, W, H) in enumerate(views):
        longest = 1.7321 / _step(case, k) + 3
        chunk = max(1, int(6e6 / (longest * W * (4 if case["tf"] == PRESHADED else 1))))
        parts = []
        for y0 in range(0, H, chunk):
            rows = torch.arange(y0, min(H, y0 + chunk), device=_device())
            with torch.set_grad_enabled(case["kind"] != "render"):
                c = _march64(case, vols[k], luts[k], cams[i], W, H, _step(case, k), rows).reshape(len(rows), W, 4)
                if case["kind"] != "render":
                    diff = c - targets[i][y0:y0 + chunk].double()
                    part = (diff.abs() if case["loss"] == "l1" else diff * diff).sum() / elements
                    if part.requires_grad:
                        part.backward()
                    loss += float(part.detach())
            parts.append(c.detach())
        colors.append(torch.cat(parts))
    if case["kind"] == "render":
        return {"color": torch.stack(colors), "term": None}
    grad = lambda ts: [t.grad if t.grad is not None else torch.zeros_like(t) for t in ts if t.requires_grad]
    if case["kind"] == "batch":
        return {"color": torch.cat([c.reshape(-1, 4) for c in colors]), "term": None,
                "loss": torch.tensor([loss], dtype=torch.float64, device=_device()),
                "grads": [g.reshape(v.shape) for g, v in zip(grad(vols), volumes)] + grad(luts)
                + ([torch.stack(grad(cams))] if "camera" in wrt else [])}
    grads = [g.reshape(volumes[0].shape if case["tf"] == PRESHADED else (1, *volumes[0].shape)) for g in grad(vols)]
    grads += [g.unsqueeze(0) for g in grad(luts)]
    if "camera" in wrt:
        grads.append(torch.stack(grad(cams)))
    return {"color": torch.stack(colors), "grads": grads}
