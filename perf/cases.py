"""Performance cases: the work that users of this framework have it do, through its Python binding.

Each case is one program's steady work.  A fluid program restores or keeps a model's state on the device and
advances it by substeps; a boids or Clouds program loads its particles and runs a number of steps; a
warm-start program trains the network on host arrays.  Model states are compared bit for bit: every launch
shape and walk of this framework gives the same bits, and a trajectory of many steps amplifies any change of
rounding until nothing could be compared.
"""
import math

import numpy as np
import torch

from realtimeparticles_amd import capi, learned, scenes

# Launch shapes a program keeps once rtp_fluids_autotune / rtp_batch_autotune has chosen them.
LITERAL_LARGE = (64, capi.LAUNCH_XCD_MAP | capi.LAUNCH_RESORT | capi.LAUNCH_NB_LIST | capi.LAUNCH_BRICKS, 9, 16)
STABLE_LARGE = (64, capi.LAUNCH_XCD_MAP | capi.LAUNCH_NB_LIST, 9, 16)
SMALL_RUN = (64, capi.LAUNCH_QUAD | capi.LAUNCH_NB_LIST, 0, 16)
SHAPES = {"default": None, "literal-large": LITERAL_LARGE, "stable-large": STABLE_LARGE, "small-run": SMALL_RUN}


def listed():
    return [
        # a small interactive fluid (the app's 8,192-particle setting), one substep a frame: launch latency
        fluids("fluids-8k-frame", 32, 16, 16, mapping="stable"),
        # the app's largest fluid, its default parameters and its rendering steps (camera sort, colours)
        fluids("fluids-131k-app-frame", 64, 64, 32, mapping="app", iters=2, render=True),
        # the 300-frame run of the 65,536-particle dam break, from its half-way state on
        fluids("fluids-65k-run", 64, 32, 32, steps=10, age=300, shape="small-run"),
        # the benchmark's workload: the 1,048,576-particle dam break's substep
        fluids("fluids-1m-substep", 128, 128, 64, shape="literal-large"),
        # an uneven large scene under the stable coefficients, a frame of two substeps
        fluids("fluids-968k-stable-frame", 125, 127, 61, mapping="stable", steps=2, shape="stable-large"),
        # the largest dam break
        fluids("fluids-4m-substep", 256, 128, 128, shape="literal-large"),
        # the learned warm start with its per-particle fallback on the 1M scene
        fluids("learned-1m-substep", 128, 128, 64, mapping="stable", shape="stable-large", learned=True),
        # uneven scenes advanced together
        {"name": "batch-24-scenes", "kind": "batch", "count": 24, "n_lo": 2048, "n_hi": 65536, "steps": 10},
        # the flock of the boids configuration, its 200 steps
        {"name": "boids-8k-run", "kind": "boids", "n": 8192, "box": 2.0, "res": 20, "steps": 200, "app": False},
        # the app's largest flock with its default rules
        {"name": "boids-131k-run", "kind": "boids", "n": 131072, "box": 10.0, "res": 30, "steps": 60, "app": True},
        # the app's cumulus cloud
        {"name": "clouds-65k-run", "kind": "clouds", "n": 65536, "steps": 50, "fill": 0.25, "iters": 2},
        # training the warm-start network (forward, backward, Adam) on teacher rows
        {"name": "train-256k-rows", "kind": "train", "rows": 262144, "batch": 65536, "epochs": 20},
    ]


def fluids(name, lx, ly, lz, mapping="literal", iters=4, steps=1, age=0, shape="default", render=False, learned=False):
    return {"name": name, "kind": "fluids", "lx": lx, "ly": ly, "lz": lz, "mapping": mapping, "iters": iters,
            "steps": steps, "age": age, "shape": shape, "render": render, "learned": learned}


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def lattice(rng, n):
    """Sides of about n particles, aspect ratios up to 1:3, odd sides among them."""
    a, b = rng.uniform(1.0, 3.0), rng.uniform(1.0, 2.0)
    s = (n / (a * b)) ** (1.0 / 3.0)
    return max(4, int(a * s)), max(4, int(b * s)), max(4, int(s))


def draw(rng):
    kind = rng.choice(["small", "small", "large", "large", "learned", "batch", "flock", "boids", "clouds", "train"])
    if kind == "small":  # default shapes, with and without what the app adds
        c = fluids("", *lattice(rng, log_int(rng, 1500, 250000)), mapping=rng.choice(["literal", "stable", "app"]),
                   iters=rng.choice([1, 2, 3, 4]), steps=rng.choice([1, 2, 5]), render=rng.random() < 0.3)
    elif kind == "large":
        m = rng.choice(["literal", "stable"])
        c = fluids("", *lattice(rng, log_int(rng, 270000, 3900000)), mapping=m, steps=rng.choice([1, 1, 2]) if m == "stable" else 1,
                   shape=m + "-large")
    elif kind == "learned":
        c = fluids("", *lattice(rng, log_int(rng, 270000, 1500000)), mapping="stable", shape="stable-large", learned=True)
    elif kind == "batch":
        c = {"kind": "batch", "count": rng.randint(3, 24), "n_lo": 1000, "n_hi": log_int(rng, 8000, 65536), "steps": rng.choice([4, 8])}
    elif kind == "flock":
        c = {"kind": "boids", "n": log_int(rng, 500, 16000), "box": 2.0, "res": 20, "steps": rng.choice([50, 101]), "app": False}
    elif kind == "boids":
        c = {"kind": "boids", "n": log_int(rng, 16000, 131000), "box": 10.0, "res": 30, "steps": rng.choice([20, 33]), "app": True}
    elif kind == "clouds":
        c = {"kind": "clouds", "n": log_int(rng, 8000, 65000), "steps": rng.choice([10, 21]), "fill": rng.choice([0.25, 0.5, 1.0]),
             "iters": rng.choice([1, 2, 3])}
    else:
        rows = log_int(rng, 20000, 262144)
        c = {"kind": "train", "rows": rows, "batch": rng.choice([4096, 16384, 65536]), "epochs": rng.choice([0, 4])}
    c.pop("name", None)
    return c


class DeviceArray:
    """Device memory of a model as a tensor's storage; it keeps the model alive."""

    def __init__(self, owner, ptr, shape, typestr="<f4"):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 3, "strides": None}


def tensor(owner, ptr, shape, typestr="<f4"):
    return torch.as_tensor(DeviceArray(owner, ptr, shape, typestr), device="cuda")


def scene(case, seed):
    lat = (case["lx"], case["ly"], case["lz"])
    res = tuple(max(4, int(math.ceil(side * 0.5 / 0.8))) for side in lat)
    box = tuple(float(np.float32(r * 0.1)) for r in res)
    return scenes.dam_break(lat, box, res, seed=seed)


def fluid_params(case, sc):
    """The dam break's coefficients ("literal"), their stable variant, or the app's own defaults."""
    if case["mapping"] == "app":
        return dict(capi.FLUID_DEFAULTS, restDensity=float(np.float32(sc.rest_density)))
    return sc.params(case["mapping"])


def warm_start_network(model, sc, iters):
    """A network whose output is the plain lambda input, amplified (GELU(z) - GELU(-z) = z): what a trained
    one does to first order, without the minutes of training it.  Normalised on the scene's own rows."""
    feat, target = model.record_teacher(iters)
    norm = learned.fit_normalization(feat, target)
    lam = feat[:, 1].astype(np.float64)
    gain = float((lam * target).sum() / (lam * lam).sum())
    w1, w2, w3 = np.zeros((8, 64)), np.zeros((64, 64)), np.zeros(64)
    w1[1, 0], w1[1, 1] = 1.0, -1.0
    w2[0, 0], w2[1, 0], w2[0, 1], w2[1, 1] = 1.0, -1.0, -1.0, 1.0
    k = gain * float(norm.sigma[1]) / norm.out_scale
    w3[0], w3[1] = k, -k
    b3 = gain * float(norm.mu[1]) / norm.out_scale
    net = capi.Mlp(seed=1)
    net.set_params(np.concatenate([w1.ravel(), np.zeros(64), w2.ravel(), np.zeros(64), w3, [b3]]).astype(np.float32))
    net.set_normalization(norm.mu, norm.sigma, norm.out_scale)
    return net


def prepare_fluids(case, seed):
    sc = scene(case, seed)
    m = capi.Fluids(sc.max_n, sc.n, sc.box, sc.res, gravity=sc.gravity)
    m.set_params(**fluid_params(case, sc))
    m.set_nb_jacobi_iters(case["iters"])
    if SHAPES[case["shape"]]:
        m.set_tuning(*SHAPES[case["shape"]])
    m.load_state(sc.pos, sc.vel)
    net = None
    if case["learned"]:
        m.save_checkpoint()
        net = warm_start_network(m, sc, case["iters"])
        m.restore_checkpoint()
        m.set_warm_start(net, 1, 4, 0.2)
    if case["render"]:
        m.set_render(True)
        m.set_camera((0.0, 4.0, 12.0))
    if case["age"]:
        m.update(case["age"])
    m.save_checkpoint()
    m.sync()
    return {"case": case, "model": m, "net": net}


def run_fluids(s):
    m = s["model"]
    m.restore_checkpoint()
    m.update(s["case"]["steps"])
    pos, vel = m.device_state()
    out = {"pos": tensor(s, pos, (m.n, 4)), "vel": tensor(s, vel, (m.n, 4))}
    if s["case"]["render"]:
        col, dist, _ = m.device_render()
        out["color"] = tensor(s, col, (m.n, 4))
        out["camera"] = tensor(s, dist, (m.n,), "<i4")
    return out


def prepare_batch(case, seed):
    scs = scenes.batch_scenes(case["count"], n_lo=case["n_lo"], n_hi=case["n_hi"])
    for k, sc in enumerate(scs):  # these scenes' boxes and gravity, the seed's particles in them
        inside = scenes.dam_break(sc.lattice, sc.box, sc.res, seed=seed * 1009 + k)
        sc.pos, sc.vel = inside.pos, inside.vel
    b = capi.Batch(scs)
    for k, sc in enumerate(scs):
        b.set_params(k, **sc.params("stable"))
        b.load_state(k, sc.pos, sc.vel)
    b.set_nb_jacobi_iters(4)
    b.set_tuning(256, 9, 24, capi.LAUNCH_NB_LIST)
    b.save_checkpoint()
    b.sync()
    return {"case": case, "batch": b}


def run_batch(s):
    b = s["batch"]
    b.restore_checkpoint()
    b.update(s["case"]["steps"])
    states = [b.read_state(k) for k in range(len(b.sizes))]
    return {"pos": np.concatenate([p for p, _ in states]), "vel": np.concatenate([v for _, v in states])}


def prepare_boids(case, seed):
    sc = scenes.boids_flock(case["n"], seed=seed, box=case["box"], res=case["res"])
    m = capi.Boids(sc.max_n, sc.n, sc.box, sc.res)
    if case["app"]:
        m.set_params()
        m.set_time_step(0.1)
    else:
        m.set_params(sc.velocity_scale, sc.alignment, sc.separation, sc.cohesion)
        m.set_time_step(sc.time_step)
    return {"case": case, "model": m, "pos": sc.pos, "vel": sc.vel}


def prepare_clouds(case, seed):
    box = (10.0, 20.0, 10.0)
    n = case["n"]
    lo = np.array([-5.0, -10.0, -5.0], np.float32)
    span = np.array([10.0, 20.0 * case["fill"], 10.0], np.float32)
    pos, vel = np.zeros((n, 4), np.float32), np.zeros((n, 4), np.float32)
    pos[:, :3] = scenes.uniform24(seed, 0, 3 * n).reshape(n, 3) * span + lo
    like = scenes.CloudScene("", box, (30, 60, 30), n, n, pos, vel)
    m = capi.Clouds(131072, n, box, (30, 60, 30))
    m.set_params(like.params(), like.cloud_params())
    m.set_nb_jacobi_iters(case["iters"])
    return {"case": case, "model": m, "pos": pos, "vel": vel}


def run_particles(s):
    """A boids or Clouds run: the particles loaded, the steps, the state read back."""
    m = s["model"]
    m.load_state(s["pos"], s["vel"])
    m.update(s["case"]["steps"])
    pos, vel = m.read_state()
    if s["case"]["kind"] == "boids":
        return {"pos": pos, "vel": vel}
    return {"pos": pos, "vel": vel, "temperature": m.read_field(capi.FIELD_TEMPERATURE), "cloud": m.read_field(capi.FIELD_CLOUD_DENSITY)}


def prepare_train(case, seed):
    """Rows with the spread of the solver's eight inputs and a smooth target of them."""
    rng = np.random.default_rng(seed)
    n = case["rows"]
    feat = (rng.standard_normal((n, 8)) * np.array([0.1, 2e-4, 8.0, 0.3, 0.2, 0.5, 0.4, 0.8]) +
            np.array([-0.05, 1e-4, 27.0, 0.5, 0.1, 0.3, 0.8, 1.5])).astype(np.float32)
    target = (2.0 * feat[:, 1] - 3e-4 * np.tanh(4.0 * feat[:, 0]) + 1e-4 * feat[:, 4] * feat[:, 6]).astype(np.float32)
    norm = learned.fit_normalization(feat, target)
    net = capi.Mlp(seed=3)
    net.set_normalization(norm.mu, norm.sigma, norm.out_scale)
    return {"case": case, "net": net, "start": net.params(), "feat": feat, "target": target, "norm": norm}


def run_train(s):
    """Training from the initial weights, or (no epochs) the inference and gradients a trainer of its own asks for."""
    net, case = s["net"], s["case"]
    net.set_params(s["start"])
    if case["epochs"] == 0:
        grad, loss = net.gradients(s["feat"], s["target"])
        return {"grad": grad, "loss": loss, "out": net.forward(s["feat"])}
    hist = net.train(s["feat"], s["target"], epochs=case["epochs"], batch=case["batch"], lr=2e-3, seed=5)
    return {"params": net.params(), "history": hist}


PREPARE = {"fluids": prepare_fluids, "batch": prepare_batch, "boids": prepare_boids, "clouds": prepare_clouds, "train": prepare_train}
RUN = {"fluids": run_fluids, "batch": run_batch, "boids": run_particles, "clouds": run_particles, "train": run_train}


def prepare(case, seed):
    return PREPARE[case["kind"]](case, seed)


def run(state):
    return RUN[state["case"]["kind"]](state)


def work(case):
    """State read and written once per step (32 bytes a particle each way), and the arithmetic of the true
    neighbour pairs: about 29 neighbours on the dam-break lattice, 20 operations a pair and sum."""
    if case["kind"] == "train":
        rows = case["rows"] * max(1, case["epochs"])
        return {"bytes": 36.0 * rows, "flops": rows * (3 if case["epochs"] else 4) * 2.0 * (8 * 64 + 64 * 64 + 64)}
    if case["kind"] == "fluids":
        n = case["lx"] * case["ly"] * case["lz"]
        pairs = 29.0 * (2 * (5 if case["learned"] else case["iters"]) + 3)
    elif case["kind"] == "batch":
        n = case["count"] * (case["n_hi"] - case["n_lo"]) / math.log(case["n_hi"] / case["n_lo"])
        pairs = 29.0 * 11
    elif case["kind"] == "boids":
        n = case["n"]
        pairs = n * 4.18879 / case["res"] ** 3
    else:
        n = case["n"]
        pairs = 5.2 / case["fill"] * (2 * case["iters"] + 5)
    return {"bytes": 64.0 * n * case["steps"], "flops": 20.0 * pairs * n * case["steps"]}


def tolerance(case):
    # The training kernels add gradients with atomics, whose order differs from run to run: two runs differ by 5e-6 after
    # 20 epochs of Adam and by 5e-7 in one gradient.  Another order inside a tile's 32-bit sums also moves a few of the
    # activations and errors that are rounded to bf16 to the other neighbour.
    if case["kind"] == "train":
        return {"rel": 5e-4, "max": 0.02} if case["epochs"] else {"rel": 2e-5, "max": 1e-3}
    return "exact"


def exact(case, seed):
    """One substep of a small scene, or a network's outputs and gradients, in 64 bits.  None elsewhere: over
    several steps 32 and 64 bits part exponentially, and the sorted order with them."""
    if case["kind"] == "train" and case["epochs"] == 0:
        return exact_network(case, seed)
    if case["kind"] == "fluids" and case["steps"] == 1 and not (case["age"] or case["render"] or case["learned"]):
        n = case["lx"] * case["ly"] * case["lz"]
        if n <= 20000 and case["mapping"] != "literal":
            return exact_substep(case, seed)
    return None


def exact_network(case, seed):
    s = prepare_train(case, seed)
    norm, p = s["norm"], torch.tensor(s["start"], dtype=torch.float64, requires_grad=True)
    x = (torch.tensor(s["feat"], dtype=torch.float64) - torch.tensor(norm.mu).double()) / torch.tensor(norm.sigma).double()
    w1, b1, w2, b2, w3, b3 = p[:512].view(8, 64), p[512:576], p[576:4672].view(64, 64), p[4672:4736], p[4736:4800], p[4800]
    gelu = torch.nn.functional.gelu
    y = gelu(gelu(x @ w1 + b1, approximate="tanh") @ w2 + b2, approximate="tanh") @ w3 + b3
    loss = ((y - torch.tensor(s["target"]).double() / norm.out_scale) ** 2).mean()
    loss.backward()
    return {"grad": p.grad.numpy(), "loss": float(loss.detach()), "out": (y.detach() * norm.out_scale).numpy()}


def exact_substep(case, seed):
    sc = scene(case, seed)
    prm = {**capi.FLUID_DEFAULTS, **fluid_params(case, sc)}
    d = dict(dtype=torch.float64, device="cuda")
    pos, vel = torch.tensor(sc.pos[:, :3], **d), torch.tensor(sc.vel[:, :3], **d)
    h, dt, rho0 = float(np.float32(sc.box[0] / sc.res[0])), prm["timeStep"], prm["restDensity"]
    wall = torch.tensor(sc.box, **d) / 2
    res = torch.tensor(sc.res, device="cuda")
    poly = lambda r2: torch.where(r2 < h * h, 315 / (64 * math.pi * h ** 9) * (h * h - r2) ** 3, 0.0)  # noqa: E731

    def cells(p):
        return torch.floor((torch.minimum(torch.maximum(p, -wall), wall) + wall) / h).long()

    pred = pos + (vel + torch.tensor([0.0, -sc.gravity * dt, 0.0], **d)) * dt
    cell = cells(pred)
    order = torch.sort((cell[:, 0] * res[1] + cell[:, 1]) * res[2] + cell[:, 2], stable=True).indices
    pos, pred, cell = pos[order], pred[order], cell[order]
    seen = torch.arange(len(order), device="cuda") > 0  # the first sorted particle is in no cell's list

    def sums(p, f):
        """f(rows, difference, r2, gradient of the spiky kernel) over the listed neighbours, in blocks of particles."""
        mine, out = cells(p), []
        for i in range(0, len(p), 512):
            rows = slice(i, i + 512)
            diff = p[rows, None] - p[None]
            r2 = (diff * diff).sum(-1)
            away = (cell[None] - mine[rows, None]).abs()
            near = (torch.minimum(away, res - away) <= 1).all(-1) & seen & (r2 < h * h)
            r = r2.sqrt()
            grad = torch.where((near & (r > 1e-8))[..., None], -45 / (math.pi * h ** 6) * ((h - r) ** 2 / r.clamp_min(1e-30))[..., None] * diff, 0.0)
            out.append(f(rows, torch.where(near, poly(r2), 0.0), grad))
        return torch.cat(out)

    for _ in range(case["iters"]):
        pred = torch.minimum(torch.maximum(pred, -wall + 0.01), wall - 0.1)
        both = sums(pred, lambda rows, w, g: torch.cat([w.sum(1, True), g.sum(1), (g * g).sum((1, 2))[:, None]], 1))
        lam = -(both[:, 0] / rho0 - 1) / ((both[:, 4] + (both[:, 1:4] ** 2).sum(1)) / rho0 ** 2 + prm["relaxCFM"])
        wdq = float(poly(torch.tensor((prm["artPressureRadius"] * h) ** 2, **d)))
        pred = pred + sums(pred, lambda rows, w, g: ((lam[rows, None] + lam[None] - prm["artPressureCoeff"] *
                                                      (w / wdq) ** prm["artPressureExp"])[..., None] * g).sum(1)) / rho0
    vel = ((pred - pos) / (dt + 1e-8)).clamp(-30.0, 30.0)
    cross = torch.linalg.cross
    vort = sums(pred, lambda rows, w, g: cross(vel[None] - vel[rows, None], g, dim=-1).sum(1))
    size = vort.norm(dim=1)
    way = torch.nn.functional.normalize(sums(pred, lambda rows, w, g: (size[None, :, None] * g).sum(1)), dim=1, eps=1e-300)
    vel = vel + prm["vorticityConfCoeff"] * dt * cross(way, vort, dim=-1)
    vel = vel + prm["xsphViscosityCoeff"] * sums(pred, lambda rows, w, g: (w[..., None] * (vel[None] - vel[rows, None])).sum(1))
    pad = lambda v: torch.nn.functional.pad(v, (0, 1))  # noqa: E731
    return {"pos": pad(pred), "vel": pad(vel)}
