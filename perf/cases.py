"""The workloads whose speed this framework is judged by, each through its public Python entry points.

    listed()              the fixed cases
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   inputs and engine, as a program holds them before the call
    run(state)            one pass; returns its outputs
    work(case)            bytes and operations no implementation can do without
    exact(case, seed)     the outputs in 64-bit arithmetic, by plain torch

Scenes are seeded random Gaussians of the two layouts of torpedo_amd/scenes.py (uniform in a cube, or
64 anisotropic clusters), made on the GPU; sizes are those of the benchmark, the tests and the smoke
test, and sizes between them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from torpedo_amd.autograd import rasterize
from torpedo_amd.engine import (GaussianEngine, PerspectiveCamera, Scene, Settings, sort_pairs_device,
                                sort_pairs_device_noalloc)

DEV = "cuda"


def listed():
    return [
        # One small frame, the smoke test's: an icon, a thumbnail, a unit test.  Launches and waits.
        dict(name="frame-4k-256x144", kind="frame", layout="uniform", n=4_000, width=256, height=144,
             log_scale=-4.5, degree=3),
        # The viewer's ordinary frame: 100k Gaussians at 720p.
        dict(name="frame-100k-720p", kind="frame", layout="uniform", n=100_000, width=1280, height=720,
             log_scale=-4.5, degree=3),
        # A compiled scene of three entities with transforms, an odd size and a low SH degree, presented
        # as RGBA8: what an editor shows.
        dict(name="present-250k-3ent-801x603", kind="present", layout="clusters", n=250_007, width=801, height=603,
             log_scale=-4.5, degree=1, entities=3),
        # A captured scene at full HD, one camera.
        dict(name="frame-1m-1080p", kind="frame", layout="clusters", n=1_000_000, width=1920, height=1080,
             log_scale=-4.5, degree=3),
        # The same with large splats (about 20 tiles each): the sort-bound frame.
        dict(name="frame-1m-dense-1080p", kind="frame", layout="clusters", n=1_000_000, width=1920, height=1080,
             log_scale=-3.0, degree=3),
        # A small training step through torch.autograd: fitting a single object.
        dict(name="train-20k-320x200", kind="autograd", layout="uniform", n=20_000, width=320, height=200,
             log_scale=-3.5, degree=3),
        # A training step of a large scene, one full-HD view, on the engine's own buffers.
        dict(name="train-3m-1080p", kind="train", layout="clusters", n=3_000_000, width=1920, height=1080,
             log_scale=-4.5, degree=3),
        # Eight small views whose cameras move every frame: a simulator's sensors.
        dict(name="moving-8x100k-512", kind="moving", layout="uniform", n=100_000, views=8, width=512, height=512,
             log_scale=-4.5, degree=3),
        # The benchmark's batch: a fixed rig of 32 cameras, 256x256 to 1920x1080, tuned once.
        dict(name="batch-32x1m", kind="batch", layout="clusters", n=1_000_000, views=32, log_scale=-4.5, degree=3),
        # The benchmark's training step over many scenes: 16 scenes of 50k to 2M Gaussians, 4 views each.
        dict(name="step-16x4", kind="step", layout="clusters", n=50_000, n_max=2_000_000, scenes=16, views=4,
             log_scale=-4.5, degree=3),
        # The stand-alone sort in a loop that may not allocate.
        dict(name="sort-200k-noalloc", kind="sort", n=200_000, key_bits=43, noalloc=True),
        # The stand-alone sort of a large frame's (tile, depth) pairs.
        dict(name="sort-20m", kind="sort", n=20_000_000, key_bits=45, noalloc=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "present", "autograd", "train", "moving", "batch", "step", "sort", "sort"])
    if kind == "sort":
        noalloc = rng.random() < 0.5
        return dict(kind=kind, n=_log(rng, 1_000, 4_000_000 if noalloc else 20_000_000),
                    key_bits=rng.randint(33, 64) if rng.random() < 0.8 else rng.randint(8, 32), noalloc=noalloc)
    case = dict(kind=kind, layout=rng.choice(["uniform", "clusters"]), log_scale=round(rng.uniform(-5.0, -3.2), 3),
                degree=rng.choice([0, 1, 2, 3, 3, 3]))
    if kind == "batch":
        return dict(case, n=_log(rng, 20_000, 500_000), views=rng.randint(2, 32))
    if kind == "step":
        n = _log(rng, 5_000, 50_000)
        return dict(case, n=n, n_max=4 * n, scenes=rng.randint(1, 12), views=rng.randint(1, 4))
    height = _log(rng, 96, 1080 if kind in ("frame", "train", "present") else 540)
    case.update(width=max(1, int(height * rng.uniform(0.8, 1.78))), height=height)
    if kind == "moving":
        return dict(case, n=_log(rng, 2_000, 200_000), views=rng.randint(1, 12))
    top = {"frame": 2_000_000, "present": 400_000, "autograd": 300_000, "train": 2_000_000}[kind]
    case["n"] = _log(rng, 2_000, top)
    if kind == "present":
        case["entities"] = rng.randint(1, 8)
    return case


# ------------------------------------------------------------------ scenes and cameras

def _generator(seed, part):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1009 + part)


def _rotations(q):
    x, y, z, w = q.unbind(-1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1).reshape(-1, 3, 3)


def _params(layout, n, log_scale, seed, part=0):
    """means, log-scales, unit quaternions (xyzw), opacity logits and 48 SH coefficients of n Gaussians."""
    gen = _generator(seed, part)
    normal = lambda *s: torch.randn(*s, device=DEV, generator=gen)  # noqa: E731
    if layout == "uniform":
        means = 2.0 * torch.rand(n, 3, device=DEV, generator=gen) - 1.0
    else:
        centres = 10.0 * torch.rand(64, 3, device=DEV, generator=gen) - 5.0
        stds = 0.1 + 0.9 * torch.rand(64, 3, device=DEV, generator=gen)
        rots = _rotations(torch.nn.functional.normalize(normal(64, 4), dim=1))
        member = torch.randint(64, (n,), device=DEV, generator=gen)
        axes = (rots * stds[:, None, :])[member]
        means = (axes * normal(n, 1, 3)).sum(-1) + centres[member]
    log_scales = log_scale + 0.5 * normal(n, 3)
    quats = torch.nn.functional.normalize(normal(n, 4), dim=1)
    logits = normal(n)
    sh = 0.2 * normal(n, 48)
    sh[:, :3] += 0.5
    return means, log_scales, quats, logits, sh


def _records(params):
    means, log_scales, quats, logits, sh = params
    return torch.cat([means, torch.sigmoid(logits)[:, None], quats, torch.exp(log_scales),
                      torch.ones_like(logits)[:, None], sh], 1).contiguous()


def _eye(layout):
    return (0.0, 0.0, -3.0) if layout == "uniform" else (0.0, 0.0, -8.0)


def _camera(eye, up, width, height):
    cam = PerspectiveCamera(width, height)
    cam.lookAt(list(eye), [0.0, 0.0, 0.0], list(up))
    return cam


RESOLUTIONS = [(256, 256), (512, 512), (640, 480), (800, 600), (1024, 768), (1280, 720), (1600, 900), (1920, 1080)]


def _rig(case, seed, part=0):
    """(eye, width, height) of a case's views: eyes on a Fibonacci sphere around the scene."""
    count = case["views"]
    radius = 3.0 if case["layout"] == "uniform" else 8.0
    rng = np.random.default_rng([int(seed), 7, part])
    # the sizes of a rig belong to the case, not to the seed: every seed is the same amount of work
    sizes = np.random.default_rng([count, part, case["n"]])
    turn = rng.uniform(0.0, 2.0 * math.pi)
    out = []
    for k in range(count):
        z = min(0.95, max(-0.95, 1.0 - 2.0 * (k + 0.5) / count))
        r, phi = math.sqrt(1.0 - z * z), turn + k * math.pi * (3.0 - math.sqrt(5.0))
        if "width" in case:
            w, h = case["width"], case["height"]
        elif case["kind"] == "step":
            w, h = int(sizes.integers(512, 1601)), int(sizes.integers(512, 901))
        else:
            w, h = RESOLUTIONS[int(sizes.integers(len(RESOLUTIONS)))]
        out.append(((radius * r * math.cos(phi), radius * r * math.sin(phi), radius * z), w, h))
    return out


def _scene_sizes(case):
    """Gaussians per scene of a step, log-spaced between n and n_max."""
    s = case["scenes"]
    return [int(case["n"] * (case["n_max"] / case["n"]) ** ((k + 0.5) / s)) for k in range(s)]


def _entity_transforms(case, seed):
    """Model matrices of a presented scene's entities: a turn about y and a shift."""
    rng = np.random.default_rng([int(seed), 11])
    out = []
    for _ in range(case["entities"]):
        a = rng.uniform(-0.5, 0.5)
        m = np.eye(4, dtype=np.float32)
        m[0, 0] = m[2, 2] = math.cos(a)
        m[0, 2], m[2, 0] = math.sin(a), -math.sin(a)
        m[:3, 3] = rng.uniform(-0.3, 0.3, 3)
        out.append(m)
    return out


class _DeviceArray:
    """An engine-owned device buffer as a torch tensor sees it.  The tensor holds this object, and with
    it the engine, so that the buffer outlives every tensor over it."""

    def __init__(self, eng, ptr, shape):
        self.owner = eng
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False), version=2)


def _batch_images(eng):
    ptr, pixels = eng.batchImagesPtr()
    return torch.as_tensor(_DeviceArray(eng, ptr, (pixels, 3)), device=DEV)


# ------------------------------------------------------------------ preparation

def prepare(case, seed):
    kind = case["kind"]
    state = dict(case=case, kind=kind, eng=GaussianEngine(device=torch.cuda.current_device()))
    _PREPARE[kind](state, case, seed)
    torch.cuda.synchronize()
    return state


def _prepare_frame(state, case, seed):
    w, h = case["width"], case["height"]
    state["rec"] = _records(_params(case["layout"], case["n"], case["log_scale"], seed))
    state["cam"] = _camera(_eye(case["layout"]), (0, -1, 0), w, h)
    state["img"] = torch.empty(h, w, 3, device=DEV)
    torch.cuda.synchronize()
    state["eng"].bindDeviceScene(state["rec"].data_ptr(), case["n"], case["degree"])


def _prepare_present(state, case, seed):
    rec = _records(_params(case["layout"], case["n"], case["log_scale"], seed)).cpu().numpy()
    scene = Scene()
    ents = [scene.add(part) for part in np.array_split(rec, case["entities"])]
    state["eng"].compile(scene, Settings(case["degree"]))
    for e, m in zip(ents, _entity_transforms(case, seed)):
        state["eng"].getTransformHost().transform(e, m)
    state["cam"] = _camera(_eye(case["layout"]), (0, -1, 0), case["width"], case["height"])
    state["surface"] = torch.empty(case["height"], case["width"], 4, dtype=torch.uint8, device=DEV)


def _upstream(pixels, seed):
    return torch.randn(pixels, 3, device=DEV, generator=_generator(seed, 501))


def _prepare_autograd(state, case, seed):
    w, h = case["width"], case["height"]
    params = _params(case["layout"], case["n"], case["log_scale"], seed)
    state["params"] = [p.requires_grad_(True) for p in params]
    state["cam"] = _camera(_eye(case["layout"]), (0, -1, 0), w, h)
    state["up"] = _upstream(w * h, seed).reshape(h, w, 3)
    state["stream"] = torch.cuda.Stream()


def _prepare_train(state, case, seed):
    _prepare_frame(state, case, seed)
    state["up"] = _upstream(case["width"] * case["height"], seed)
    state["grads"] = [torch.empty(case["n"], k, device=DEV) for k in (3, 3, 4, 1, 48)]


def _prepare_views(state, case, seed):
    eng = state["eng"]
    state["rec"] = _records(_params(case["layout"], case["n"], case["log_scale"], seed))
    torch.cuda.synchronize()
    sid = eng.addDeviceScene(state["rec"].data_ptr(), case["n"], case["degree"])
    state["views"] = [(sid, _camera(eye, (0, 0, 1), w, h)) for eye, w, h in _rig(case, seed)]
    eng.setViews(state["views"])
    if case["kind"] == "batch":  # a fixed rig: its radix shapes are tuned before the loop, as the benchmark does
        eng.rasterBatch()
        eng.syncBatch()
        eng.autotuneBatch()


def _prepare_step(state, case, seed):
    eng = state["eng"]
    sizes = _scene_sizes(case)
    state["recs"], views, pixels = [], [], 0
    for s, n in enumerate(sizes):
        state["recs"].append(_records(_params(case["layout"], n, case["log_scale"], seed, s)))
    torch.cuda.synchronize()
    for s, n in enumerate(sizes):
        sid = eng.addDeviceScene(state["recs"][s].data_ptr(), n, case["degree"])
        for eye, w, h in _rig(case, seed, s):
            views.append((sid, _camera(eye, (0, 0, 1), w, h)))
            pixels += w * h
    eng.setViews(views)
    state["up"] = _upstream(pixels, seed)
    state["grads"] = [torch.empty(sum(sizes), k, device=DEV) for k in (3, 3, 4, 1, 48)]
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    state["table"] = [tuple(g.data_ptr() + int(a) * g.shape[1] * 4 for g in state["grads"]) for a in starts]


def _prepare_sort(state, case, seed):
    n, bits = case["n"], case["key_bits"]
    gen = _generator(seed, 601)
    low = torch.randint(0, 1 << min(bits, 32), (n,), device=DEV, generator=gen, dtype=torch.int64)
    high = torch.randint(0, 1 << max(bits - 32, 0), (n,), device=DEV, generator=gen, dtype=torch.int64)
    state["keys"] = (high << 32) | low
    state["vals"] = torch.arange(n, device=DEV, dtype=torch.int32)
    state["work"] = [torch.empty_like(t) for t in (state["keys"], state["vals"]) for _ in range(2)]
    state["stream"] = torch.cuda.Stream()


_PREPARE = dict(frame=_prepare_frame, present=_prepare_present, autograd=_prepare_autograd, train=_prepare_train,
                moving=_prepare_views, batch=_prepare_views, step=_prepare_step, sort=_prepare_sort)


# ------------------------------------------------------------------ one pass

def run(state):
    return _RUN[state["kind"]](state)


def _run_frame(st):
    st["eng"].rasterFrame(st["cam"])
    st["eng"].copyImageTo(st["img"].data_ptr())
    st["eng"].waitIdle()  # the engine's stream is its own: the image is read on another
    return st["img"]


def _run_present(st):
    st["eng"].rasterFrame(st["cam"])
    st["eng"].presentTo(st["surface"].data_ptr())
    st["eng"].waitIdle()
    return st["surface"]


def _run_autograd(st):
    now, side = torch.cuda.current_stream(), st["stream"]
    side.wait_stream(now)
    with torch.cuda.stream(side):
        img = rasterize(*st["params"], st["eng"], st["cam"], st["case"]["degree"])
        out = (img.detach(), *torch.autograd.grad(img, st["params"], st["up"]))
    now.wait_stream(side)
    for t in out:
        t.record_stream(now)
    return out


def _run_train(st):
    eng = st["eng"]
    eng.rasterFrame(st["cam"])
    eng.backward(st["up"].data_ptr(), *[g.data_ptr() for g in st["grads"]])
    eng.copyImageTo(st["img"].data_ptr())
    eng.waitIdle()
    return (st["img"], *st["grads"])


def _run_moving(st):
    st["eng"].setViews(st["views"])
    return _run_batch(st)


def _run_batch(st):
    st["eng"].rasterBatch()
    st["eng"].syncBatch()
    return _batch_images(st["eng"])


def _run_step(st):
    st["eng"].batchStep(st["up"].data_ptr(), st["table"])
    st["eng"].syncBatch()
    return (_batch_images(st["eng"]), *st["grads"])


def _run_sort(st):
    case = st["case"]
    now, side = torch.cuda.current_stream(), st["stream"]
    keys, keys_alt, vals, vals_alt = st["work"]
    sort = sort_pairs_device_noalloc if case["noalloc"] else sort_pairs_device
    side.wait_stream(now)
    with torch.cuda.stream(side):  # the sort works in place: a pass sorts a fresh copy
        keys.copy_(st["keys"])
        vals.copy_(st["vals"])
        in_alt = sort(st["eng"], keys.data_ptr(), vals.data_ptr(), keys_alt.data_ptr(), vals_alt.data_ptr(),
                      case["n"], case["key_bits"], side.cuda_stream)
    now.wait_stream(side)
    return (keys_alt, vals_alt) if in_alt else (keys, vals)


_RUN = dict(frame=_run_frame, present=_run_present, autograd=_run_autograd, train=_run_train, moving=_run_moving,
            batch=_run_batch, step=_run_step, sort=_run_sort)


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    """Bytes: records (and upstream gradients) read once, images and gradients written once.  Operations:
    the projection of every Gaussian in every view (about 400, half again as many for its gradient twice
    over); how many pixels a splat is evaluated for depends on the picture and is not counted."""
    kind = case["kind"]
    if kind == "sort":
        return {"bytes": 24.0 * case["n"], "flops": 0.0}
    if kind == "step":
        sizes = _scene_sizes(case)
        pixels = sum(w * h for s in range(len(sizes)) for _, w, h in _rig(case, 0, s))
        n = sum(sizes)
        return {"bytes": (240.0 + 236.0) * n + (16.0 + 12.0) * pixels, "flops": 1600.0 * n * case["views"]}
    n = float(case["n"])
    if "views" in case:
        pixels = sum(w * h for _, w, h in _rig(case, 0))
        return {"bytes": 240.0 * n + 16.0 * pixels, "flops": 400.0 * n * case["views"]}
    pixels = case["width"] * case["height"]
    if kind in ("train", "autograd"):
        return {"bytes": (240.0 + 236.0) * n + (12.0 + 12.0) * pixels, "flops": 1600.0 * n}
    return {"bytes": 240.0 * n + (4.0 if kind == "present" else 12.0) * pixels, "flops": 400.0 * n}


# ------------------------------------------------------------------ the same in 64 bits

def _look_at(eye, up):
    eye, up = np.asarray(eye, np.float64), np.asarray(up, np.float64)
    z = -eye / np.linalg.norm(eye)
    x = np.cross(z, up)
    x /= np.linalg.norm(x)
    y = np.cross(z, x)
    y /= np.linalg.norm(y)
    view = np.eye(4)
    view[:3, :3] = [x, y, z]
    view[:3, 3] = [-x @ eye, -y @ eye, -z @ eye]
    return view


def _projection(width, height, near=0.01, far=100.0):
    fy = math.sqrt(3.0)
    p = np.zeros((4, 4))
    p[0, 0], p[1, 1] = fy * height / width, fy
    p[2, 2], p[2, 3], p[3, 2] = near / (near - far), near * far / (far - near), 1.0
    return p


def _sh_colour(sh, d, degree):
    """SH colour plus 0.5, at least 0; coefficient 12 enters without its basis function, as in the original."""
    x, y, z = d.unbind(-1)
    one, zero = torch.ones_like(x), torch.zeros_like(x)
    basis = [0.28209479177387814 * one]
    if degree > 0:
        c = 0.4886025119029199
        basis += [-c * y, c * z, -c * x]
    if degree > 1:
        basis += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
                  0.31539156525252005 * (2 * z * z - x * x - y * y), -1.0925484305920792 * x * z,
                  0.5462742152960396 * (x * x - y * y)]
    extra = zero
    if degree > 2:
        basis += [-0.5900435899266435 * y * (3 * x * x - y * y), 2.890611442640554 * x * y * z,
                  -0.4570457994644658 * y * (4 * z * z - x * x - y * y), one,
                  -0.4570457994644658 * x * (4 * z * z - x * x - y * y), 1.445305721320277 * z * (x * x - y * y),
                  -0.5900435899266435 * x * (x * x - 3 * y * y)]
        extra = 0.3731763325901154 * z * (2 * z * z - 3 * x * x - 3 * y * y)
    k = len(basis)
    coef = torch.cat([sh[:, :3, None], sh[:, 3:].reshape(-1, 3, 15)[:, :, :k - 1]], 2)  # (N, 3, k)
    out = (coef * torch.stack(basis, -1)[:, None, :]).sum(-1) + extra[:, None]
    return torch.clamp(out + 0.5, min=0.0)


def _project(means, scales, quats, opacity, sh, view, proj, width, height, degree):
    """Screen-space splats of every Gaussian: (N, 9) of x, y, conic a, b, c, r, g, b, opacity; the depth,
    the tile rectangle, and whether the Gaussian is seen at all (its other values are meaningless if not)."""
    V = torch.tensor(view, device=DEV)
    PV = torch.tensor(proj @ view, device=DEV)
    p = means @ V[:3, :3].T + V[:3, 3]
    clip = means @ PV[:, :3].T + PV[:, 3]
    w = clip[:, 3]
    depth = p[:, 2]
    seen = ((depth > 0) & (clip[:, 0].abs() <= 1.3 * w) & (clip[:, 1].abs() <= 1.3 * w) & (clip[:, 2] >= 0)
            & (clip[:, 2] <= w))
    depth_ok = torch.where(seen, depth, torch.ones_like(depth))
    w_ok = torch.where(seen, w, torch.ones_like(w))
    fx, fy = 0.5 * width * proj[0, 0], 0.5 * height * proj[1, 1]
    M = _rotations(quats) * scales[:, None, :]
    cov = M @ M.transpose(1, 2)
    zero = torch.zeros_like(depth)
    J = torch.stack([fx / depth_ok, zero, -fx * p[:, 0] / depth_ok ** 2,
                     zero, fy / depth_ok, -fy * p[:, 1] / depth_ok ** 2], -1).reshape(-1, 2, 3)
    T = J @ V[:3, :3]
    c2 = T @ cov @ T.transpose(1, 2)
    a, b, c = c2[:, 0, 0] + 0.3, c2[:, 1, 0], c2[:, 1, 1] + 0.3
    det = a * c - b * b
    seen = seen & (det != 0)
    det = torch.where(seen, det, torch.ones_like(det))
    with torch.no_grad():
        mid = 0.5 * (a + c)
        root = torch.sqrt(torch.clamp(mid * mid - det, min=0.1))
        radius = torch.ceil(3.0 * torch.sqrt(torch.clamp(mid + root, min=0.0)))
    x = ((clip[:, 0] / w_ok + 1.0) * width - 1.0) * 0.5
    y = ((clip[:, 1] / w_ok + 1.0) * height - 1.0) * 0.5
    with torch.no_grad():
        gx, gy = (width + 15) // 16, (height + 15) // 16
        rect = [torch.trunc((x - radius) / 16).clamp(0, gx), torch.trunc((y - radius) / 16).clamp(0, gy),
                torch.trunc((x + radius + 15) / 16).clamp(0, gx), torch.trunc((y + radius + 15) / 16).clamp(0, gy)]
        rect = [torch.nan_to_num(r).long() for r in rect]
        seen = seen & (rect[2] > rect[0]) & (rect[3] > rect[1])
    eye = -(V[:3, :3].T @ V[:3, 3])
    colour = _sh_colour(sh, torch.nn.functional.normalize(means - eye, dim=1), degree)
    splats = torch.cat([torch.stack([x, y, c / det, -b / det, a / det], -1), colour, opacity[:, None]], 1)
    return splats, depth, rect, seen


def _tile_lists(depth, rect, seen, gx, gy):
    """Splat indices by (tile, depth) and each tile's range in them."""
    ids = torch.nonzero(seen)[:, 0]
    ids = ids[torch.sort(depth[ids], stable=True)[1]]
    x0, y0, x1, y1 = (r[ids] for r in rect)
    w, count = x1 - x0, (x1 - x0) * (y1 - y0)
    owner = torch.repeat_interleave(torch.arange(ids.numel(), device=DEV), count)
    k = torch.arange(owner.numel(), device=DEV) - (torch.cumsum(count, 0) - count)[owner]
    tile = (y0[owner] + k // w[owner]) * gx + x0[owner] + k % w[owner]
    tile, order = torch.sort(tile, stable=True)
    length = torch.bincount(tile, minlength=gx * gy)
    return ids[owner[order]], torch.cumsum(length, 0) - length, length


def _blend(splats, lists, width, height, upstream=None):
    """The front-to-back composite in chunks of every tile's list; with upstream (H, W, 3) also the
    gradients of the splats' nine values."""
    values, start, length = lists
    gx, gy = (width + 15) // 16, (height + 15) // 16
    ntiles, K, most = gx * gy, 32, 8192
    tiles = torch.arange(ntiles, device=DEV)
    lane = torch.arange(256, device=DEV)
    px, py = (tiles % gx)[:, None] * 16 + lane % 16, (tiles // gx)[:, None] * 16 + lane // 16
    inside = (px < width) & (py < height)
    colour = torch.zeros(ntiles, 256, 3, device=DEV, dtype=torch.float64)
    grads = up = total = None
    if upstream is not None:
        up = torch.zeros_like(colour)
        up[inside] = upstream.double()[py[inside], px[inside]]
        grads = torch.zeros(splats.shape[0], 9, device=DEV, dtype=torch.float64)
    for backward in ([False] if upstream is None else [False, True]):
        if backward:
            total = (colour * up).sum(-1)
        T = inside.double()  # 0 for a pixel that takes no more splats
        behind = torch.zeros_like(T)  # sum of weight * (colour . upstream) so far
        for c in range(0, int(length.max()) if length.numel() else 0, K):
            live = torch.nonzero((length > c) & (T > 0).any(1))[:, 0]
            if live.numel() == 0:
                break
            for t in live.split(most):
                at = c + torch.arange(K, device=DEV)
                valid = at[None, :] < length[t][:, None]
                g = values[torch.where(valid, start[t][:, None] + at, torch.zeros_like(at))]
                s = splats[g]  # (B, K, 9)
                dx, dy = s[..., 0, None] - px[t][:, None, :], s[..., 1, None] - py[t][:, None, :]
                power = -0.5 * (s[..., 2, None] * dx * dx + s[..., 4, None] * dy * dy) - s[..., 3, None] * dx * dy
                raw = s[..., 8, None] * torch.exp(power)
                alpha = torch.clamp(raw, max=0.99)
                alpha = torch.where(valid[..., None] & (power <= 0) & (alpha >= 1.0 / 255.0), alpha, 0.0)
                after = T[t][:, None, :] * torch.cumprod(1.0 - alpha, 1)
                stopped = after < 1e-4
                alpha = torch.where(stopped, 0.0, alpha)
                before = torch.cat([T[t][:, None, :], after[:, :-1]], 1)
                weight = torch.where(stopped, 0.0, alpha * before)
                if not backward:
                    colour[t] += weight.transpose(1, 2) @ s[..., 5:8]
                else:
                    shade = s[..., 5:8] @ up[t].transpose(1, 2)  # (B, K, 256)
                    front = behind[t][:, None, :] + torch.cumsum(weight * shade, 1)
                    d_alpha = before * shade - (total[t][:, None, :] - front) / (1.0 - alpha)
                    d_alpha = torch.where(weight > 0, d_alpha, 0.0)
                    d_raw = torch.where(raw < 0.99, d_alpha, 0.0)
                    d_power = d_raw * alpha
                    a, b, cc = s[..., 2], s[..., 3], s[..., 4]
                    mx, my = (d_power * dx).sum(-1), (d_power * dy).sum(-1)
                    out = torch.stack([-a * mx - b * my, -cc * my - b * mx, -0.5 * (d_power * dx * dx).sum(-1),
                                       -(d_power * dx * dy).sum(-1), -0.5 * (d_power * dy * dy).sum(-1)], -1)
                    out = torch.cat([out, weight @ up[t], (d_power.sum(-1) / s[..., 8])[..., None]], -1)
                    grads.index_add_(0, g[valid], out[valid])
                    behind[t] = front[:, -1]
                T[t] = torch.where(stopped.any(1), 0.0, after[:, -1])
    image = torch.zeros(height, width, 3, device=DEV, dtype=torch.float64)
    image[py[inside], px[inside]] = colour[inside]
    return image, grads


def _render64(params, view, proj, width, height, degree, upstream=None):
    """The image, and with upstream the gradients of the five parameter groups."""
    p = [t.detach().double().requires_grad_(upstream is not None) for t in params]
    means, log_scales, quats, logits, sh = p
    splats, depth, rect, seen = _project(means, torch.exp(log_scales), quats, torch.sigmoid(logits), sh, view, proj,
                                         width, height, degree)
    with torch.no_grad():
        lists = _tile_lists(depth, rect, seen, (width + 15) // 16, (height + 15) // 16)
        image, grads = _blend(splats, lists, width, height, upstream)
    if upstream is None:
        return image, None
    return image, torch.autograd.grad(splats, p, grads)


def _render64_step(case, seed):
    """Every scene's views: all images, and each parameter group's gradients summed over the views."""
    sizes = _scene_sizes(case)
    rigs = [_rig(case, seed, s) for s in range(len(sizes))]
    up = _upstream(sum(w * h for rig in rigs for _, w, h in rig), seed)
    images, groups, at = [], [[] for _ in range(5)], 0
    for s, n in enumerate(sizes):
        params = _params(case["layout"], n, case["log_scale"], seed, s)
        total = None
        for eye, w, h in rigs[s]:
            image, grads = _render64(params, _look_at(eye, (0, 0, 1)), _projection(w, h), w, h, case["degree"],
                                     up[at:at + w * h].reshape(h, w, 3))
            at += w * h
            images.append(image.reshape(-1, 3))
            total = grads if total is None else [a + b for a, b in zip(total, grads)]
        for group, g in zip(groups, total):
            group.append(g.reshape(n, -1))
    return (torch.cat(images), *(torch.cat(g) for g in groups))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("present", "sort"):  # bytes and whole numbers
        return None
    if kind == "step":
        return _render64_step(case, seed) if sum(_scene_sizes(case)) * case["views"] < 8_000_000 else None
    params = _params(case["layout"], case["n"], case["log_scale"], seed)
    if "views" in case:
        return torch.cat([_render64(params, _look_at(eye, (0, 0, 1)), _projection(w, h), w, h,
                                    case["degree"])[0].reshape(-1, 3) for eye, w, h in _rig(case, seed)])
    w, h = case["width"], case["height"]
    up = _upstream(w * h, seed).reshape(h, w, 3) if kind in ("autograd", "train") else None
    image, grads = _render64(params, _look_at(_eye(case["layout"]), (0, -1, 0)), _projection(w, h), w, h,
                             case["degree"], up)
    if up is None:
        return image
    return (image, *(g.reshape(case["n"], -1) if kind == "train" else g for g in grads))
