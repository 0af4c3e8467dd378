"""The work a user of the permutohedral-lattice filter has it do, as cases that can be timed.

Every case goes through the package's public entry points the way a program that uses them does:

* ``op``      ``lattice_filter`` on a batch of images or volumes (inference);
* ``train``   ``lattice_filter`` and its registered gradient, through autograd;
* ``filter``  a lattice object that filters forward and reverse under given positions;
* ``apply``   a lattice that was built once and filters new values, forward and reverse;
* ``static``  ``filter_static``, the entry point that allocates nothing;
* ``crf``     the dense-CRF harness: lattices rebuilt for new guides, five mean-field iterations
  and the gradient pass;
* ``cloud``   a lattice object on an unordered list of points.

``listed()`` names twelve of them, ``draw(rng)`` gives others of the same ranges.
"""
import math

import torch

import permutohedral_lattice_amd as pla
from permutohedral_lattice_amd.crf import MeanField

DEVICE = "cuda"


def _image(name, path, height, width, *, depth=0, batch=1, values=3, guide=3, dtype="float32",
           alpha=8.0, beta=0.125):
    """A case on a row-major image (depth 0) or volume.  ``guide``: channels of the reference image;
    0 filters under the coordinates alone (alpha is then the op's theta_gamma)."""
    case = {"path": path, "batch": batch, "depth": depth, "height": height, "width": width,
            "values": values, "guide": guide, "dtype": dtype, "alpha": alpha, "beta": beta}
    return dict(case, name=name) if name else case


def _cloud(name, points, features, values=3):
    case = {"path": "cloud", "points": points, "features": features, "values": values}
    return dict(case, name=name) if name else case


def listed():
    return [
        # A thumbnail through the op: what one smallest call costs, launches and host work.
        _image("thumbnail_op", "op", 64, 64),
        # A patch of a serving loop that must not allocate.
        _image("patch_static", "static", 120, 160),
        # Colour image under itself, forward and reverse: the filter call of a lattice object.
        _image("rgb_filter", "filter", 1024, 1024),
        # The same lattice kept for many right-hand sides (the build is behind the program).
        _image("rgb_apply", "apply", 1024, 1024),
        # A photograph through the op; sides that are no powers of two.
        _image("photo_op", "op", 800, 1200),
        # Plain Gaussian smoothing of a grey image: two features, little per vertex.
        _image("spatial_op", "op", 1024, 1024, values=1, guide=0),
        # Training step of a joint bilateral layer: grey values under a colour guide, batch of 4.
        _image("guided_train", "train", 1024, 1024, batch=4, values=1),
        # A scan filtered under its own intensities: the largest call.
        _image("volume_op", "op", 256, 256, depth=128, values=1, guide=1, alpha=5.0, beta=0.1),
        # Dense-CRF inference and gradient over 21 labels, guides in 0..255, new guides each step.
        _image("crf", "crf", 512, 512, batch=2, values=21, alpha=80.0, beta=13.0),
        # A message-passing layer of a segmentation network: 21 label maps under a colour guide,
        # odd sides, forward and gradient through the op.
        _image("labels_train", "train", 321, 481, batch=2, values=21),
        # A scanned point cloud in no order, its colours smoothed along the surfaces.
        _cloud("cloud_filter", 500009, 3),
        # The op in double precision, as a numerical check of a training program runs it.
        _image("double_op", "op", 601, 803, dtype="float64"),
    ]


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _sides(rng, low, high):
    """Height and width of an image of low..high pixels, up to 5:3 either way."""
    pixels, aspect = _log_uniform(rng, low, high), _log_uniform(rng, 0.6, 1.0 / 0.6)
    height = max(8, int(math.sqrt(pixels * aspect)))
    return height, max(8, int(pixels / height))


def draw(rng):
    path = rng.choice(("op", "op", "volume", "double", "train", "labels", "filter", "apply",
                       "static", "crf", "cloud"))
    alpha, beta = round(rng.uniform(6.0, 12.0), 2), round(rng.uniform(0.12, 0.2), 3)
    if path == "cloud":
        return _cloud(None, int(_log_uniform(rng, 5000, 1 << 20)), rng.choice((3, 4)))
    if path == "volume":
        scale = _log_uniform(rng, 0.15, 1.0)
        depth, height, width = (max(8, int(side * scale * rng.uniform(0.8, 1.0)))
                                for side in (128, 256, 256))
        return _image(None, "op", height, width, depth=depth, values=1, guide=1,
                      alpha=round(rng.uniform(4.0, 6.0), 2), beta=round(rng.uniform(0.08, 0.15), 3))
    if path == "static":
        height, width = _sides(rng, 500, 21000)
        return _image(None, "static", height, width, alpha=alpha, beta=beta)
    if path == "crf":
        height, width = _sides(rng, 5000, 1 << 18)
        return _image(None, "crf", height, width, batch=rng.choice((1, 2)), values=rng.choice((5, 21)),
                      alpha=round(rng.uniform(40.0, 80.0), 1), beta=round(rng.uniform(10.0, 16.0), 1))
    if path == "labels":
        height, width = _sides(rng, 5000, 180000)
        return _image(None, "train", height, width, batch=rng.choice((1, 2)),
                      values=rng.choice((7, 21)), alpha=alpha, beta=beta)
    if path == "train":
        height, width = _sides(rng, 5000, 1 << 20)
        return _image(None, "train", height, width, batch=rng.choice((1, 2, 4)),
                      values=rng.choice((1, 3)), alpha=alpha, beta=beta)
    if path == "double":
        height, width = _sides(rng, 2000, 500000)
        return _image(None, "op", height, width, dtype="float64", alpha=alpha, beta=beta)
    height, width = _sides(rng, 2000, 1 << 20)
    if path == "op":
        return _image(None, "op", height, width, batch=rng.choice((1, 2)), values=rng.choice((1, 3)),
                      guide=rng.choice((0, 1, 3)), alpha=alpha, beta=beta)
    return _image(None, path, height, width, alpha=alpha, beta=beta)


# ---- inputs ---------------------------------------------------------------------------------------


def _scene(gen, sides, channels):
    """Channels-last image or volume in [0, 1]: smooth blobs (sigma 20..80 pixels, as in the
    package's synthetic images), solid shapes with hard edges, noise."""
    axes = [torch.arange(s, dtype=torch.float32, device=DEVICE) for s in sides]
    k = len(sides)
    scene = torch.zeros(tuple(sides) + (channels,), device=DEVICE)

    def distance(centre, radius):
        d = 0.0
        for i, axis in enumerate(axes):
            shape = [1] * k
            shape[i] = -1
            d = d + (((axis - centre[i] * sides[i]) / radius[i]) ** 2).view(shape)
        return d

    for _ in range(12):
        u = torch.rand(1 + k + channels, generator=gen, device=DEVICE)
        sigma = (20.0 + 60.0 * u[0]).expand(k)
        scene += torch.exp(-0.5 * distance(u[1:1 + k], sigma))[..., None] * u[1 + k:]
    for _ in range(6):
        u = torch.rand(2 * k + channels, generator=gen, device=DEVICE)
        inside = distance(u[:k], 10.0 + 90.0 * u[k:2 * k]) <= 1.0
        scene = torch.where(inside[..., None], u[2 * k:], scene)
    scene += 0.1 * torch.rand(scene.shape, generator=gen, device=DEVICE) - 0.05
    return scene.clamp_(0.0, 1.0)


def _surfaces(gen, points, features):
    """Positions (in units of the filter's widths) and colours of points sampled from eight spheres,
    in no order.  The filter is 6 sample spacings wide, so that a unit of area holds 36 points; a
    fourth feature is the brightness, with 0.15 of full scale as its width."""
    u = torch.rand((8, 8), generator=gen, device=DEVICE)
    radius = 0.5 + 0.5 * u[:, 3]
    radius = radius * (points / 36.0 / (4.0 * math.pi * (radius * radius).sum())).sqrt()
    extent = 4.0 * radius.max()
    which = torch.multinomial(radius * radius, points, replacement=True, generator=gen)
    v = torch.randn((points, 3), generator=gen, device=DEVICE)
    v = v / v.norm(dim=1, keepdim=True).clamp_min(1e-6)
    xyz = extent * u[which, 0:3] + radius[which, None] * v
    xyz = xyz + 0.05 * torch.randn(v.shape, generator=gen, device=DEVICE)
    colour = u[which, 4:7] * (0.75 + 0.25 * v)
    colour = (colour + 0.03 * torch.randn(v.shape, generator=gen, device=DEVICE)).clamp_(0.0, 1.0)
    if features == 4:
        xyz = torch.cat((xyz, colour.mean(dim=1, keepdim=True) / 0.15), dim=1)
    return xyz.contiguous(), colour.contiguous()


def _sdims(case):
    sides = (case["height"], case["width"])
    return (case["depth"],) + sides if case["depth"] else sides


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    if case["path"] == "cloud":
        position, colour = _surfaces(gen, case["points"], case["features"])
        lattice = pla.PermutohedralLattice(case["features"], case["values"] + 1, case["points"])
        return {"case": case, "lattice": lattice, "positions": position, "input": colour,
                "output": torch.empty_like(colour)}

    sides, batch, values, guide = _sdims(case), case["batch"], case["values"], case["guide"]
    dtype = getattr(torch, case["dtype"])
    shape = (batch,) + sides
    state = {"case": case}
    if guide:
        state["guide"] = torch.stack([_scene(gen, sides, guide) for _ in range(batch)]).to(dtype)
    if case["path"] == "crf":
        state["guide"] *= 255.0
        state["logits"] = torch.randn(shape + (values,), generator=gen, device=DEVICE)
        state["upstream"] = torch.randn(shape + (values,), generator=gen, device=DEVICE)
        state["field"] = MeanField(state["guide"], values, case["alpha"], case["beta"])
        return state
    if values == guide and case["path"] != "train":
        state["input"] = state["guide"]             # an image filtered under itself
    elif values > 4:
        state["input"] = torch.softmax(torch.randn(shape + (values,), generator=gen, device=DEVICE,
                                                   dtype=dtype), dim=-1)
    else:
        state["input"] = torch.rand(shape + (values,), generator=gen, device=DEVICE, dtype=dtype)
    if case["path"] == "train":
        state["input"].requires_grad_(True)
        state["upstream"] = torch.randn(shape + (values,), generator=gen, device=DEVICE, dtype=dtype)
        return state
    if case["path"] == "op":
        return state

    n = math.prod(sides)
    state["input"] = state["input"].reshape(n, values)
    state["output"], state["reverse"] = torch.empty_like(state["input"]), torch.empty_like(state["input"])
    state["positions"] = pla.compute_positions(state["guide"][0], sides, case["alpha"], case["beta"])
    if case["path"] == "static":
        return state
    lattice = pla.PermutohedralLattice(state["positions"].shape[1], values + 1, n)
    lattice.set_point_grid(sides)
    if case["path"] == "apply":
        lattice.build(state["positions"])
    state["lattice"] = lattice
    return state


def run(state):
    case = state["case"]
    path = case["path"]
    if path in ("op", "train"):
        out = pla.lattice_filter(state["input"], state.get("guide"), bilateral=case["guide"] > 0,
                                 theta_alpha=case["alpha"], theta_beta=case["beta"],
                                 theta_gamma=case["alpha"])
        if path == "op":
            return out
        (grad,) = torch.autograd.grad(out, state["input"], state["upstream"])
        return out.detach(), grad
    if path == "crf":
        field = state["field"]
        field.rebuild(state["guide"])
        return field.infer(state["logits"], 5), field.reverse(state["upstream"])
    if path == "static":
        return pla.filter_static(state["output"], state["input"], state["positions"],
                                 state["positions"].shape[1], case["values"] + 1)
    lattice = state["lattice"]
    if path == "cloud":
        return lattice.filter(state["output"], state["input"], state["positions"])
    if path == "apply":
        return (lattice.apply(state["output"], state["input"]),
                lattice.apply(state["reverse"], state["input"], reverse=True))
    return (lattice.filter(state["output"], state["input"], state["positions"]),
            lattice.filter(state["reverse"], state["input"], state["positions"], reverse=True))


def work(case):
    """Inputs read once, outputs written once; the multiplications and additions of embedding the
    points, splatting and slicing (the vertices and their blur depend on the data)."""
    path = case["path"]
    if path == "cloud":
        n, pd, read = case["points"], case["features"], case["features"]
    else:
        n = case["batch"] * math.prod(_sdims(case))
        pd = len(_sdims(case)) + case["guide"]
        read = pd if path in ("filter", "static") else (0 if path == "apply" else case["guide"])
    size = 8 if case.get("dtype") == "float64" else 4
    values = case["values"]
    filters = {"filter": 2, "apply": 2, "train": 2, "crf": 6}.get(path, 1)
    # filter and apply read one input for both directions, the others an input for each output
    streams = {"filter": 3, "apply": 3, "train": 4, "crf": 4}.get(path, 2)
    embed = 0 if path == "apply" else 2 * pd * (pd + 1)
    move = 4 * (pd + 1) * (values + 1)
    if path == "crf":                               # and the lattice of the coordinates alone
        embed += 2 * 2 * 3
        move += 4 * 3 * (values + 1)
    return {"bytes": size * n * (read + streams * values), "flops": n * (embed + filters * move)}


def tolerance(case):
    """What another order of the additions does to the outputs (with and without tiles merged in a
    workgroup, points in their own order and in the order of space, sums gathered and added
    atomically): at most 1.2e-7 and 9e-7 in single precision, 1.5e-16 and 1.1e-15 in double."""
    if case.get("dtype") == "float64":
        return {"rel": 6e-16, "max": 5e-15}
    return {"rel": 5e-7, "max": 4e-6}
