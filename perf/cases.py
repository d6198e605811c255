"""Workloads of the framework, as a user's program runs them.

Every case goes through the public Python entry points (``fdModel``,
``Batch``, ``autograd.misfit``, ``precond.HipUNet`` / ``HipUNetTrainer``):

* ``sample``: one Monte-Carlo sample of one model -- a new model vector, the
  forward of every shot without stored wavefields, the L2 misfit;
* ``calls``: one FWI gradient by the per-shot calls of a descent loop;
* ``run_model``: one FWI gradient by the single driver call;
* ``autograd``: misfit and gradient of torch tensors;
* ``batch`` / ``batch_gradient``: many models advanced together;
* ``infer`` / ``train``: the learned preconditioner's network.

``exact`` restates each of them in plain torch in 64 bits.
"""
import math

import numpy as np
import torch

C1, C2 = 9.0 / 8.0, 1.0 / 24.0
WIDTHS = (32, 48, 64, 128)  # the network's default channel widths


# --- cases ----------------------------------------------------------------

def _fd(name, kind, nxi, nzi, npb, nt, shots, nr, si=10, edge_x=0, edge_z=0, dx=5.0, dt=5e-4,
        freq=10.0, medium="grf", models=1, every=1, per_shot=1):
    """A finite-difference case: nxi x nzi inner points inside an npb-point
    absorbing taper, nt steps, shots of per_shot sources each, nr receivers,
    a snapshot every si steps; kernels edge_x / edge_z points inside."""
    return dict(name=name, kind=kind, nxi=nxi, nzi=nzi, npb=npb, nt=nt, shots=shots, nr=nr, si=si,
                edge_x=edge_x, edge_z=edge_z, dx=dx, dt=dt, freq=freq, medium=medium,
                models=models, every=every, per_shot=per_shot)


def listed():
    return [
        # a toy model, as in a first script or a unit test: launches and
        # latency are all of it
        _fd("toy_sample", "sample", 70, 41, 10, 200, 1, 4, si=5, dx=1.25, dt=2.5e-4, freq=60.0),
        # Monte-Carlo sample on the reference's test configuration: 250 x 150
        # points, 8000 steps, one shot of four sources, 19 receivers
        _fd("test_configuration_sample", "sample", 200, 100, 25, 8000, 1, 19, edge_x=10, edge_z=20,
            dx=1.249, dt=2.5e-4, freq=50.0, per_shot=4),
        # the small CPU-sized workload (300 x 200, two shots), one descent
        # gradient by the per-shot calls
        _fd("small_calls", "calls", 200, 100, 50, 4000, 2, 19, edge_x=10, edge_z=20, dx=1.25,
            dt=2.5e-4, freq=50.0),
        # one iteration of the preconditioner's FWI loop: 316 x 188, six shots
        _fd("fwi_gradient", "run_model", 256, 128, 30, 2500, 6, 48, edge_z=8, dx=10.0, dt=1e-3, freq=8.0),
        # the differentiable path: 680 x 380, four shots, full snapshot store
        _fd("autograd_gradient", "autograd", 600, 300, 40, 4000, 4, 64, edge_x=10, edge_z=10),
        # the same with a checkpoint every eighth snapshot, for less memory
        _fd("checkpointed_gradient", "run_model", 600, 300, 40, 4000, 4, 64, edge_x=10, edge_z=10,
            every=8),
        # the benchmark's grid (1800 x 450, layered, 300 receivers), two of
        # its eight shots
        _fd("large_gradient", "run_model", 1700, 350, 50, 6000, 2, 300, edge_z=20, dt=3e-4,
            medium="layered"),
        # a forward of a survey-sized grid, 2400 x 1237 points
        _fd("survey_sample", "sample", 2300, 1137, 50, 1000, 2, 240),
        # Monte-Carlo forwards of 16 models of uneven size in one batch
        _fd("batch_forward", "batch", 800, 400, 30, 3000, 2, 32, models=16),
        # training pairs: the gradients of eight models at once
        _fd("batch_gradients", "batch_gradient", 256, 128, 30, 2500, 6, 48, edge_z=8, dx=10.0, dt=1e-3,
            freq=8.0, models=8),
        # the network's prediction for one gradient of a 316 x 188 grid
        dict(name="network_infer", kind="infer", nx=316, nz=188, images=1),
        # one training pass (loss and parameter gradients) on a batch of 16
        dict(name="network_train", kind="train", nx=316, nz=188, images=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sample", "sample", "calls", "run_model", "run_model", "autograd", "batch",
                       "batch_gradient", "infer", "train"])
    if kind in ("infer", "train"):
        return dict(kind=kind, nx=_log_int(rng, 40, 330), nz=_log_int(rng, 40, 200),
                    images=1 if kind == "infer" else rng.randint(1, 16))
    forward = kind in ("sample", "batch")
    npb = rng.randint(10, 50)
    nxi, nzi = _log_int(rng, 60, 2300 if kind == "sample" else 800), _log_int(rng, 40, 1137 if kind == "sample" else 400)
    shots = rng.randint(1, 6) if not forward else rng.randint(1, 3)
    si = rng.choice([5, 10, 10, 20])
    models = rng.randint(2, 12) if kind.startswith("batch") else 1
    points = (nxi + 2 * npb) * (nzi + 2 * npb) * shots * models * (1 if forward else 2)
    most = 1.0e10 if forward else 4.0e9  # point updates of a drawn case
    nt = max(20, min(_log_int(rng, 300, 4000), int(most / points)) // 20) * 20
    every = rng.choice([1, 1, 1, 4]) if kind == "run_model" else 1
    medium = rng.choice(["grf", "grf", "layered"])
    # kernels stay below the water, as in the listed cases
    edge_z = rng.randint(nzi // 18, nzi // 18 + 4) if medium == "layered" else rng.randint(0, 8)
    case = _fd("", kind, nxi, nzi, npb, nt, shots, rng.randint(1, 120), si=si, edge_x=rng.randint(0, 8),
               edge_z=edge_z, medium=medium, models=models, every=every, per_shot=rng.randint(1, 3), dt=4e-4)
    del case["name"]
    return case


def _sizes(case):
    """Inner sizes of the members: the case's own, or for the forward batch
    uneven ones from a quarter of it up."""
    if case["kind"] != "batch":
        return [(case["nxi"], case["nzi"])] * case["models"]
    rng = np.random.default_rng([case["nxi"], case["nzi"], case["models"]])
    return [(int(rng.integers(case["nxi"] // 4, case["nxi"] + 1)),
             int(rng.integers(case["nzi"] // 4, case["nzi"] + 1))) for _ in range(case["models"])]


def _config(case, nxi, nzi):
    k, p = case["shots"], case["per_shot"]
    n = k * p
    return {
        "domain": dict(nt=case["nt"], nx_inner=nxi, nz_inner=nzi, nx_inner_boundary=case["edge_x"],
                       nz_inner_boundary=case["edge_z"], dx=case["dx"], dz=case["dx"], dt=case["dt"]),
        "boundary": dict(np_boundary=case["npb"], np_factor=0.015),
        "medium": dict(scalar_rho=1800.0, scalar_vp=2400.0, scalar_vs=1200.0),
        "sources": dict(peak_frequency=case["freq"], n_sources=n, n_shots=k, source_timeshift=0.0,
                        delay_cycles_per_shot=2, moment_angles=[30.0 + 25.0 * i for i in range(n)],
                        ix_sources=[int((i + 0.5) * nxi / n) for i in range(n)],
                        iz_sources=[min(25, nzi // 8)] * n,
                        which_source_to_fire_in_which_shot=[list(range(s * p, s * p + p)) for s in range(k)]),
        "receivers": dict(nr=case["nr"],
                          ix_receivers=[int((i + 0.5) * nxi / case["nr"]) for i in range(case["nr"])],
                          iz_receivers=[min(20, nzi // 10)] * case["nr"]),
        "inversion": dict(snapshot_interval=case["si"]),
        "basis": dict(npx=1, npz=1),
        "output": dict(observed_data_folder=".", stf_folder="."),
    }


# --- inputs ---------------------------------------------------------------

def _smooth(shape, corr, rng):
    """A Gaussian random field of correlation length corr points, scaled to
    [0, 1]."""
    n, m = (-(-k // 32) * 32 for k in shape)
    noise = np.fft.rfft2(rng.standard_normal((n, m)))
    gauss = [np.exp(-0.5 * (np.pi * corr * k) ** 2) for k in (np.fft.fftfreq(n), np.fft.rfftfreq(m))]
    f = np.fft.irfft2(noise * np.outer(*gauss), (n, m))[:shape[0], :shape[1]]
    return (f - f.min()) / (f.max() - f.min())


def _media(case, nxi, nzi, rng):
    """(start, true) models: smooth random fields, or layers of growing
    velocity under a water layer; the true one perturbed by +-5 %."""
    npb = case["npb"]
    shape = (nxi + 2 * npb, nzi + 2 * npb)
    if case["medium"] == "layered":
        n = max(3, min(40, nzi // 6))
        vps = np.sort(rng.uniform(1500.0, 5500.0, n))
        tops = np.sort(rng.uniform(0.0, nzi, n - 1))
        rows = np.clip(np.arange(shape[1]) - npb, 0, nzi - 1)
        dip = (12.0 * (_smooth((shape[0], 4), 200, rng)[:, :1] - 0.5))
        vp = vps[np.searchsorted(tops, rows[None, :] + dip, side="right")]
        water = rows < nzi // 18
        vp[:, water] = 1500.0
        vs = vp / 1.73
        vs[:, water] = 0.0
        rho = 310.0 * vp ** 0.25
    else:
        vp = 2000.0 + 800.0 * _smooth(shape, 20, rng)
        vs = vp * (0.45 + 0.10 * _smooth(shape, 20, rng))
        rho = 1500.0 + 500.0 * _smooth(shape, 20, rng)
    p = 0.1 * (_smooth(shape, 12, rng) - 0.5)
    true = (np.minimum(vp * (1 + p), 5500.0), vs * (1 + p), rho * (1 + 0.5 * p))
    return (vp, vs, rho), true


def _members(case, seed):
    """Per member: its configuration, start model and true model."""
    rng = np.random.default_rng([seed, 17])
    out = []
    for nxi, nzi in _sizes(case):
        start, true = _media(case, nxi, nzi, rng)
        out.append((_config(case, nxi, nzi), start, true))
    return out


def _weights(seed):
    """The network's parameters by name, scaled as for training."""
    g = torch.Generator().manual_seed(seed)
    c = WIDTHS
    convs = {"enc.0.0": (3, c[0]), "enc.0.2": (c[0], c[0]), "enc.1.0": (c[0], c[1]),
             "enc.1.2": (c[1], c[1]), "enc.2.0": (c[1], c[2]), "enc.2.2": (c[2], c[2]),
             "mid.0": (c[2], c[3]), "mid.2": (c[3], c[3]), "dec.0.0": (2 * c[2], c[2]),
             "dec.0.2": (c[2], c[2]), "dec.1.0": (2 * c[1], c[1]), "dec.1.2": (c[1], c[1]),
             "dec.2.0": (2 * c[0], c[0]), "dec.2.2": (c[0], c[0])}
    w = {}
    for k, (ci, co) in convs.items():
        w[k + ".weight"] = torch.randn(co, ci, 3, 3, generator=g) * (2.0 / (9 * ci)) ** 0.5
        w[k + ".bias"] = torch.randn(co, generator=g) * 0.05
    for i, (ci, co) in enumerate(((c[3], c[2]), (c[2], c[1]), (c[1], c[0]))):
        w[f"up.{i}.weight"] = torch.randn(ci, co, 2, 2, generator=g) * (1.0 / ci) ** 0.5
        w[f"up.{i}.bias"] = torch.randn(co, generator=g) * 0.05
    w["out.weight"] = torch.randn(3, c[0], 1, 1, generator=g) * (1.0 / c[0]) ** 0.5
    w["out.bias"] = torch.randn(3, generator=g) * 0.05
    return w


def _images(case, seed):
    """Normalised gradients, perturbations and the kernel-region mask."""
    rng = np.random.default_rng([seed, 29])
    shape = (case["nx"], case["nz"])
    x = np.stack([[_smooth(shape, 6, rng) - 0.5 for _ in range(3)] for _ in range(case["images"])])
    x /= np.sqrt(np.mean(x * x, axis=(2, 3), keepdims=True))
    y = np.stack([[0.1 * (_smooth(shape, 12, rng) - 0.5) for _ in range(3)] for _ in range(case["images"])])
    mask = np.zeros(shape)
    mx, mz = shape[0] // 10, shape[1] // 6
    mask[mx:-mx, mz:-mz] = 1.0
    return [torch.tensor(a, dtype=torch.float32) for a in (x, y, mask)]


# --- the passes -----------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("infer", "train"):
        from psvwave_amd import precond
        net = precond.make_unet(WIDTHS)
        net.load_state_dict(_weights(seed))
        x, y, mask = (t.cuda() for t in _images(case, seed))
        if kind == "infer":
            return dict(kind=kind, net=precond.HipUNet(net.eval()), x=x[0])
        return dict(kind=kind, trainer=precond.HipUNetTrainer(net), x=x, y=y, mask=mask)
    import psvwave_amd
    members = _members(case, seed)
    if kind in ("batch", "batch_gradient"):
        batch = psvwave_amd.Batch([cfg for cfg, _, _ in members])
        for m, (_, _, true) in enumerate(members):
            batch.set_parameter_fields(m, *true)
        batch.forward_all()
        for m in range(len(members)):
            batch.set_observed_data(m, *batch.get_synthetic_data(m))
        return dict(kind=kind, batch=batch, starts=[start for _, start, _ in members])
    cfg, start, true = members[0]
    model = psvwave_amd.fdModel(cfg)
    model.set_parameter_fields(*true)
    for s in range(case["shots"]):
        model.forward_simulate(s, store_fields=False)
    model.set_observed_data(*model.get_synthetic_data())
    model.set_parameter_fields(*start)
    state = dict(kind=kind, model=model, start=start)
    if kind == "sample":
        state["vector"] = model.get_model_vector()
    if kind == "autograd":
        state["fields"] = [torch.tensor(f, device="cuda", requires_grad=True) for f in start]
    if case["every"] > 1:
        model.set_checkpointing(case["every"])
    return state


def run(state):
    kind = state["kind"]
    if kind == "infer":
        return state["net"](state["x"])
    if kind == "train":
        loss, grads = state["trainer"].loss_and_grads(state["x"], state["y"], state["mask"])
        return [loss] + [g for _, gw, gb in grads for g in (gw, gb)]
    if kind == "batch":
        batch = state["batch"]
        for m, start in enumerate(state["starts"]):
            batch.set_parameter_fields(m, *start)
        batch.forward_all()
        return [batch.misfits()] + [batch.get_synthetic_data(m) for m in range(len(batch))]
    if kind == "batch_gradient":
        batch = state["batch"]
        for m, start in enumerate(state["starts"]):
            batch.set_parameter_fields(m, *start)
        return [batch.gradients()] + [batch.get_kernels(m) for m in range(len(batch))]
    model = state["model"]
    if kind == "sample":
        model.set_model_vector(state["vector"])
        for s in range(model.n_shots):
            model.forward_simulate(s, store_fields=False)
        model.calculate_l2_misfit()
        return [model.misfit, *model.get_synthetic_data()]
    if kind == "autograd":
        from psvwave_amd import autograd
        f = autograd.misfit(*state["fields"], model)
        return [f.detach(), *torch.autograd.grad(f, state["fields"])]
    model.set_parameter_fields(*state["start"])
    if kind == "run_model":
        model.run_model(False, True)
        return [model.misfit, *model.get_kernels(), *model.get_synthetic_data()]
    for s in range(model.n_shots):
        model.forward_simulate(s)
    model.calculate_l2_misfit()
    model.calculate_l2_adjoint_sources()
    model.reset_kernels()
    for s in range(model.n_shots):
        model.adjoint_simulate(s)
    model.map_kernels_to_velocity()
    return [model.misfit, model.get_gradient_vector(), *model.get_synthetic_data()]


def work(case):
    """Bytes of the inputs and outputs of the call (parameters, observed and
    synthetic data, kernels; network inputs, parameters and outputs) and the
    stencil's (87 per point and step) or the convolutions' operations."""
    if case["kind"] in ("infer", "train"):
        train = case["kind"] == "train"
        px = [case["images"] * case["nx"] * case["nz"] / 4.0 ** k for k in range(4)]
        c = WIDTHS
        macs = px[0] * (9 * (3 * c[0] + c[0] * c[0]) + 9 * (2 * c[0] * c[0] + c[0] * c[0]) + 3 * c[0])
        macs += px[1] * 9 * (c[0] * c[1] + c[1] * c[1] + 2 * c[1] * c[1] + c[1] * c[1])
        macs += px[2] * 9 * (c[1] * c[2] + c[2] * c[2] + 2 * c[2] * c[2] + c[2] * c[2])
        macs += px[3] * 9 * (c[2] * c[3] + c[3] * c[3])
        macs += px[3] * 4 * c[3] * c[2] + px[2] * 4 * c[2] * c[1] + px[1] * 4 * c[1] * c[0]
        weights = sum(v.numel() for v in _weights(0).values())
        images = 4 * 3 * px[0] * 2
        return {"bytes": images + 4 * weights * (2 if train else 1), "flops": 2 * macs * (3 if train else 1)}
    grad = case["kind"] not in ("sample", "batch")
    points = traces = 0
    for nxi, nzi in _sizes(case):
        points += (nxi + 2 * case["npb"]) * (nzi + 2 * case["npb"])
        traces += 2 * case["shots"] * case["nr"] * case["nt"]
    updates = points * case["shots"] * case["nt"] * (2 if grad else 1)
    return {"bytes": 8 * (points * (6 if grad else 3) + 2 * traces), "flops": 87 * updates}


# --- the same in plain torch, 64 bits -------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Survey:
    """Time loops of every shot of models of one size, side by side on the
    first axis: fields are (models * shots, nx, nz)."""

    def __init__(self, cfg, models):
        dev = self.dev = _device()
        d, npb = cfg["domain"], cfg["boundary"]["np_boundary"]
        src, rec = cfg["sources"], cfg["receivers"]
        self.nt, self.dt, self.dx, self.si = d["nt"], d["dt"], d["dx"], cfg["inversion"]["snapshot_interval"]
        self.nx, self.nz = d["nx_inner"] + 2 * npb, d["nz_inner"] + 2 * npb
        self.shots, self.models, self.nr = src["n_shots"], models, rec["nr"]
        self.L = models * self.shots
        ex, ez = npb + d["nx_inner_boundary"], npb + d["nz_inner_boundary"]
        self.kx, self.kz = slice(ex, self.nx - ex), slice(ez, self.nz - ez)
        x = torch.arange(self.nx, device=dev).view(-1, 1)
        z = torch.arange(self.nz, device=dev).view(1, -1)
        depth = torch.minimum(torch.minimum(x, self.nx - 1 - x), torch.minimum(z, self.nz - 1 - z)) + 1
        arg = cfg["boundary"]["np_factor"] * (npb - depth.clamp(max=npb)).double()
        self.taper = torch.exp(-arg * arg)[2:-2, 2:-2]
        self.rx = torch.tensor(rec["ix_receivers"], device=dev) + npb
        self.rz = torch.tensor(rec["iz_receivers"], device=dev) + npb
        # the moment-tensor terms of every loop: loop, component, point, weight, wavelet
        terms = {0: [], 1: []}
        self.waves = torch.empty(self.nt, src["n_sources"], dtype=torch.float64, device=dev)
        t = torch.arange(self.nt, dtype=torch.float64, device=dev) * self.dt
        f = src["peak_frequency"]
        for s, fired in enumerate(src["which_source_to_fire_in_which_shot"]):
            for place, i in enumerate(fired):
                a = math.pi * f * (t - 1.4 / f - src["delay_cycles_per_shot"] * place / f)
                self.waves[:, i] = (1 - 2 * a * a) * torch.exp(-a * a)
                angle = src["moment_angles"][i] * 3.14159265 / 180.0
                m0, m1 = math.cos(angle) * 1e15, -math.sin(angle) * 1e15
                px, pz = src["ix_sources"][i] + npb, src["iz_sources"][i] + npb
                for m in range(models):
                    k = m * self.shots + s
                    terms[0] += [(k, px - 1, pz, i, -m0), (k, px, pz, i, m0)]
                    terms[1] += [(k, px, pz - 1, i, m0), (k, px, pz, i, -m0)]
                    for ox, oz, q in ((-1, 1, m1), (0, 1, m1), (-1, -1, -m1), (0, -1, -m1)):
                        terms[0].append((k, px + ox, pz + oz, i, 0.25 * q))
                    for ox, oz, q in ((1, -1, m1), (1, 0, m1), (-1, -1, -m1), (-1, 0, -m1)):
                        terms[1].append((k, px + ox, pz + oz, i, 0.25 * q))
        self.terms = []
        for c in (0, 1):
            cols = list(zip(*terms[c]))
            self.terms.append([torch.tensor(v, device=dev) for v in cols[:4]]
                              + [torch.tensor(cols[4], dtype=torch.float64, device=dev)])

    def fields(self, models):
        """Lame parameters and buoyancy of every loop from (vp, vs, rho) per model."""
        put = [torch.stack([torch.tensor(m[k], dtype=torch.float64, device=self.dev) for m in models])
               .repeat_interleave(self.shots, 0) for k in range(3)]
        vp, vs, rho = put
        self.vp, self.vs, self.rho = put
        self.lm, self.mu, self.b = vp * vp * rho, vs * vs * rho, 1.0 / rho
        self.la = self.lm - 2 * self.mu
        inner = [a[:, 2:-2, 2:-2] for a in (self.lm, self.la, self.mu, self.b)]
        self.ilm, self.ila, self.imu, self.ib = inner
        self.sign = 0
        for c in (0, 1):
            k, px, pz, i, w = self.terms[c][:5]
            self.terms[c][5:] = [w * self.dt * self.b[k, px, pz] / self.dx ** 4]

    def zero(self):
        return [torch.zeros(self.L, self.nx, self.nz, dtype=torch.float64, device=self.dev) for _ in range(5)]

    def advance(self, state, sign):
        vx, vz, xx, zz, xz = state
        if self.sign != sign:
            self.sign = sign
            self.dtmu, self.dtb = sign * self.dt * self.imu, sign * self.dt * self.ib
            self.dtlm, self.dtla = sign * self.dt * self.ilm, sign * self.dt * self.ila
        n, m = self.nx, self.nz

        def dif(f, axis, back):  # centred between the points: ahead of each point, or behind it
            if axis == 0:
                at = lambda o: f[:, 2 + o:n - 2 + o, 2:-2]  # noqa: E731
            else:
                at = lambda o: f[:, 2:-2, 2 + o:m - 2 + o]  # noqa: E731
            o = -1 if back else 0
            return (at(1 + o) - at(o)).mul_(C1 / self.dx).add_(at(o - 1) - at(2 + o), alpha=C2 / self.dx)

        exx, ezz = dif(vx, 0, False), dif(vz, 1, True)
        exz = dif(vx, 1, False).add_(dif(vz, 0, True))
        t = self.taper
        i = (slice(None), slice(2, -2), slice(2, -2))
        xx[i] = torch.addcmul(xx[i], self.dtlm, exx).addcmul_(self.dtla, ezz).mul_(t)
        zz[i] = torch.addcmul(zz[i], self.dtla, exx).addcmul_(self.dtlm, ezz).mul_(t)
        xz[i] = torch.addcmul(xz[i], self.dtmu, exz).mul_(t)
        vx[i] = torch.addcmul(vx[i], self.dtb, dif(xx, 0, True).add_(dif(xz, 1, True))).mul_(t)
        vz[i] = torch.addcmul(vz[i], self.dtb, dif(xz, 0, False).add_(dif(zz, 1, False))).mul_(t)

    def forward(self, keep):
        """Traces (models, shots, nr, nt) of both components, and with
        `keep` the snapshots on the kernel region."""
        state, snaps = self.zero(), []
        rec = torch.empty(2, self.nt, self.L, self.nr, dtype=torch.float64, device=self.dev)
        for it in range(self.nt):
            for c in (0, 1):
                rec[c, it] = state[c][:, self.rx, self.rz]
            if keep and it % self.si == 0:
                snaps.append([f[:, self.kx, self.kz].clone() for f in state])
            self.advance(state, 1)
            for c in (0, 1):
                k, px, pz, i, _, w = self.terms[c]
                state[c].index_put_((k, px, pz), w * self.waves[it, i], accumulate=True)
        rec = torch.cumsum(rec * (self.dt / self.dx ** 2), 1).permute(0, 2, 3, 1)
        return rec.reshape(2, self.models, self.shots, self.nr, self.nt).contiguous(), snaps

    def adjoint(self, residual, snaps):
        """Velocity kernels (vp, vs, rho) per model from the residual traces."""
        res = residual.reshape(2, self.L, self.nr, self.nt)
        region = (slice(None), self.kx, self.kz)
        lm, mu, la = self.lm[region], self.mu[region], self.la[region]
        d = lm - la * la / lm
        w = self.si * self.dt
        kr, kl, km = (torch.zeros_like(lm) for _ in range(3))
        ratio, inv, shear = la / lm, w / (d * d), w / (mu * mu)
        k = torch.arange(self.L, device=self.dev).view(-1, 1).expand(-1, self.nr)
        px, pz = self.rx.expand(self.L, -1), self.rz.expand(self.L, -1)
        weight = self.dt * self.b[k, px, pz] / self.dx ** 2
        state = self.zero()
        for it in range(self.nt - 1, -1, -1):
            if it % self.si == 0:
                vx, vz, xx, zz, xz = snaps[it // self.si]
                ax, az, axx, azz, axz = [f[region] for f in state]
                kr -= w * (ax * vx + az * vz)
                qa, qb = axx - azz * ratio, azz - axx * ratio
                p, q = xx - zz * ratio, zz - xx * ratio
                kl += inv * (qa + qb) * (p + q)
                km += 2 * inv * (p * qa + q * qb) + shear * (xz * axz)
            self.advance(state, -1)
            for c in (0, 1):
                state[c].index_put_((k, px, pz), weight * res[c, :, :, it], accumulate=True)
        out = []
        total = lambda a: a.view(self.models, self.shots, *a.shape[1:]).sum(1)  # noqa: E731
        kr, kl, km = total(kr), total(kl), total(km)
        vp, vs, rho = (a[::self.shots][region] for a in (self.vp, self.vs, self.rho))
        for part in (2 * vp * kl * rho, (2 * vs * km - 4 * vs * kl) * rho,
                     kr + (vp * vp - 2 * vs * vs) * kl + vs * vs * km):
            full = torch.zeros(self.models, self.nx, self.nz, dtype=torch.float64, device=self.dev)
            full[region] = part
            out.append(full)
        return out


def _exact_survey(cfg, starts, trues, gradient):
    s = _Survey(cfg, len(starts))
    s.fields(trues)
    observed, _ = s.forward(False)
    s.fields(starts)
    synthetic, snaps = s.forward(gradient)
    residual = synthetic - observed
    misfit = 0.5 * s.dt * (residual * residual).sum(dim=(0, 2, 3, 4))
    return misfit, synthetic, s.adjoint(residual, snaps) if gradient else None, s


def _exact_network(case, seed):
    dev = _device()
    w = {k: v.double().to(dev).requires_grad_(True) for k, v in _weights(seed).items()}
    x, y, mask = (t.double().to(dev) for t in _images(case, seed))
    ph, pw = (-case["nx"]) % 16, (-case["nz"]) % 16
    a = torch.nn.functional.pad(x, (0, pw, 0, ph)).permute(0, 2, 3, 1)

    def conv(a, k, gelu=True):  # one matrix product over the gathered taps
        wt = w[k + ".weight"]
        r = wt.shape[-1] // 2
        h, v = a.shape[1:3]
        p = torch.nn.functional.pad(a, (0, 0, r, r, r, r))
        taps = torch.cat([p[:, i:i + h, j:j + v] for i in range(2 * r + 1) for j in range(2 * r + 1)], -1)
        o = taps.reshape(-1, taps.shape[-1]) @ wt.permute(2, 3, 1, 0).reshape(-1, wt.shape[0]) + w[k + ".bias"]
        o = o.reshape(*a.shape[:3], -1)
        return torch.nn.functional.gelu(o) if gelu else o

    def half(a):
        b, h, v, c = a.shape
        return a.reshape(b, h // 2, 2, v // 2, 2, c).amax(dim=(2, 4))

    def up(a, k):
        b, h, v, c = a.shape
        wt = w[k + ".weight"]
        o = (a.reshape(-1, c) @ wt.permute(0, 2, 3, 1).reshape(c, -1)).reshape(b, h, v, 2, 2, -1) + w[k + ".bias"]
        return o.permute(0, 1, 3, 2, 4, 5).reshape(b, 2 * h, 2 * v, -1)

    skips = []
    for i in range(3):
        a = conv(conv(a, f"enc.{i}.0"), f"enc.{i}.2")
        skips.append(a)
        a = half(a)
    a = conv(conv(a, "mid.0"), "mid.2")
    for i in range(3):
        a = torch.cat([up(a, f"up.{i}"), skips[2 - i]], -1)
        a = conv(conv(a, f"dec.{i}.0"), f"dec.{i}.2")
    pred = conv(a, "out", gelu=False)[:, :case["nx"], :case["nz"]].permute(0, 3, 1, 2)
    if case["kind"] == "infer":
        return pred[0].detach().contiguous()
    loss = (((pred - y) * mask) ** 2).mean() / (mask.mean() * 1e-3)
    loss.backward()
    # in the order in which the backward pass meets the layers
    order = ["out"]
    for i in (2, 1, 0):
        order += [f"dec.{i}.2", f"dec.{i}.0", f"up.{i}"]
    order += ["mid.2", "mid.0"]
    for i in (2, 1, 0):
        order += [f"enc.{i}.2", f"enc.{i}.0"]
    return [loss.detach()] + [w[f"{k}.{p}"].grad for k in order for p in ("weight", "bias")]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("infer", "train"):
        return _exact_network(case, seed)
    members = _members(case, seed)
    if kind == "batch":
        misfits, traces = [], []
        for cfg, start, true in members:
            f, syn, _, _ = _exact_survey(cfg, [start], [true], False)
            misfits.append(f)
            traces.append((syn[0, 0], syn[1, 0]))
        return [torch.cat(misfits)] + traces
    starts, trues = [m[1] for m in members], [m[2] for m in members]
    misfit, syn, kernels, s = _exact_survey(members[0][0], starts, trues, kind != "sample")
    if kind == "batch_gradient":
        return [misfit] + [tuple(k[m] for k in kernels) for m in range(len(members))]
    if kind == "sample":
        return [misfit[0], syn[0, 0], syn[1, 0]]
    if kind == "autograd":
        return [misfit[0]] + [k[0] for k in kernels]
    if kind == "run_model":
        return [misfit[0], *(k[0] for k in kernels), syn[0, 0], syn[1, 0]]
    # the gradient vector: free points with x fastest, one block per parameter
    vector = torch.cat([k[0][s.kx, s.kz].t().reshape(-1) for k in kernels])
    return [misfit[0], vector, syn[0, 0], syn[1, 0]]
