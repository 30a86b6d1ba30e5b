"""Performance cases of the compact-difference framework: the work its users have it do.

Families
  lines      derivative and filter operators along grid lines (ops.LineOp)
  solver     one full time step of a box (solver.Solver)
  ensemble   several steps of many small boxes advanced together (ensemble.Ensemble)
  sgs        the Vreman / dynamic Smagorinsky models over caller-owned fields (sgs.Sgs)
  learned    the learned closure over caller-owned fields (sgs.Sgs)
  train      minibatch training of the closure network (closure.Closure)
  gradient   one gradient of the closure network and its Adam update (closure.Closure)
  infer      evaluation of the closure network on given samples (closure.Closure)

``exact`` restates every result in 64 bits with plain torch: line operators as
dense matrices A^-1 B built from the schemes' published coefficients, the time
step and the SGS models from their equations.
"""
import math

import numpy as np
import torch

GAMMA = 1.4
R_GAS = 1.0 / GAMMA
CP = R_GAS * GAMMA / (GAMMA - 1.0)
PRANDTL = 0.7
SCHEMES = {"cd2": ("deriv", 0, 0.0), "pade6": ("deriv", 1, 0.0), "penta10": ("deriv", 2, 0.0),
           "compact8": ("filter", 0, 0.49), "compact10": ("filter", 1, 0.49),
           "commn5pade": ("filter", 2, 0.0), "commn5exp": ("filter", 3, 0.0)}
LAYOUT = {"x": 0, "y": 1, "z": 2}
N_PARAMS = 8962  # 7-64-64-64-2


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    def lines(name, schemes, n, walls, fields, pencil="x"):
        return dict(name=name, family="lines", schemes=schemes, nx=n[0], ny=n[1], nz=n[2], walls=walls,
                    fields=fields, pencil=pencil)

    def solver(name, n, fd, filt, rk, les, avg, walls=""):
        return dict(name=name, family="solver", nx=n[0], ny=n[1], nz=n[2], fd=fd, filt=filt, rk=rk, les=les, avg=avg,
                    walls=walls)

    return [
        # gradients of the four primitive fields on a small box: launches and latency
        lines("grad_32", "penta10", (32, 32, 32), "", 4),
        # the kernel-level pass of the operator benchmark: derivatives and the filter in every
        # direction on five conserved fields, periodic in x and one-sided closures in y and z
        lines("pass_256", "penta10+compact8", (256, 256, 256), "yz", 5),
        # a walled box whose sizes no chunk length splits evenly
        lines("ragged_150", "pade6+compact10", (150, 131, 165), "xz", 5),
        # channel-like box with long lines in x and z and a prime wall-normal size, in the
        # pencil that callers keep for the wall-normal direction
        lines("channel_640", "penta10+compact8", (640, 193, 384), "y", 3, "y"),
        # the headline workload: decaying isotropic turbulence, LES with the Vreman model
        solver("les_256", (256, 256, 256), "PENTA10", "COMPACT8", "KENRK4", "VREMAN", "LOCAL"),
        # a small box of the reference's own decaying-turbulence deck, run by itself
        solver("box_64", (64, 64, 64), "PADE6", "COMPACT10", "RK4", "NOMODEL", "NONE"),
        # wall-bounded flow on a stretched grid, odd wall-normal size
        solver("walls_160", (160, 129, 144), "PENTA10", "COMPACT8", "RK4", "VREMAN", "LOCAL", "y"),
        # dynamic Smagorinsky model with the line-averaged coefficients
        dict(name="dsm_160", family="sgs", nx=160, ny=160, nz=160, model="DSM", avg="XI1_AVG", testfilter=1,
             pencil="x"),
        # boxes of uneven sizes advanced together for some steps, then read back
        dict(name="ensemble_6", family="ensemble", sizes="32,48,48,64,64,96", steps=10, seed=11),
        # the learned closure in place of the model above, point-wise features
        dict(name="learned_160", family="learned", nx=160, ny=160, nz=160, pencil="x"),
        # closure training as the studies run it: batches of 8192 pairs
        dict(name="train_8192", family="train", samples=262144, batch=8192, epochs=4),
        # one training step on a ragged batch, gradient and update by hand
        dict(name="gradient_5000", family="gradient", samples=5000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi, cap):
    """Three sizes in lo..hi (over the logarithm) with at most cap points; half of them even splits."""
    while True:
        n = [_log_int(rng, lo, hi) for _ in range(3)]
        if rng.random() < 0.5:
            n = [max(lo, 16 * round(v / 16)) if v >= 24 else v for v in n]
        if n[0] * n[1] * n[2] <= cap:
            return n


def draw(rng):
    family = rng.choice(["lines"] * 4 + ["solver"] * 3 + ["sgs"] * 2 +
                        ["learned", "ensemble", "train", "gradient", "infer"])
    if family == "lines":
        n = _box(rng, 24, 768, 30_000_000)
        deriv = rng.choice(["penta10", "pade6", "penta10", "pade6", "cd2"])
        filt = rng.choice(["compact8", "compact10", "compact8", "compact10", "commn5pade", "commn5exp"])
        schemes = rng.choice([deriv, filt, deriv + "+" + filt])
        walls = "".join(d for d in "xyz" if rng.random() < 0.4)
        return dict(family=family, schemes=schemes, nx=n[0], ny=n[1], nz=n[2], walls=walls,
                    fields=rng.randint(1, 5), pencil=rng.choice(["x", "x", "y", "z"]))
    if family == "solver":
        n = _box(rng, 32, 256, 8_000_000)
        les, avg = rng.choice([("NOMODEL", "NONE"), ("VREMAN", "LOCAL"), ("VREMAN", "NONE")])
        return dict(family=family, nx=n[0], ny=n[1], nz=n[2], fd=rng.choice(["PADE6", "PENTA10"]),
                    filt=rng.choice(["COMPACT8", "COMPACT10"]), rk=rng.choice(["TVDRK3", "RK4", "KENRK4"]),
                    les=les, avg=avg, walls=rng.choice(["", "", "y"]))
    if family == "sgs":
        n = _box(rng, 32, 224, 5_000_000)
        model = rng.choice(["DSM", "DSM", "VREMAN"])
        avg = rng.choice(["GLOBAL", "XI1_AVG", "XI3_AVG"]) if model == "DSM" else rng.choice(["LOCAL", "NONE"])
        return dict(family=family, nx=n[0], ny=n[1], nz=n[2], model=model, avg=avg, testfilter=rng.choice([1, 2]),
                    pencil=rng.choice(["x", "y"]))
    if family == "learned":
        n = _box(rng, 32, 224, 5_000_000)
        return dict(family=family, nx=n[0], ny=n[1], nz=n[2], pencil=rng.choice(["x", "y"]))
    if family == "ensemble":
        sizes = sorted(rng.choice([32, 40, 48, 64, 80, 96]) for _ in range(rng.randint(3, 8)))
        return dict(family=family, sizes=",".join(map(str, sizes)), steps=rng.randint(4, 10),
                    seed=rng.randint(1, 10**6))
    if family == "train":
        return dict(family=family, samples=_log_int(rng, 10_000, 300_000),
                    batch=rng.choice([1024, 2048, 4096, 5000, 8192, 16384]), epochs=rng.randint(1, 4))
    if family == "gradient":
        return dict(family=family, samples=_log_int(rng, 300, 40_000))
    return dict(family="infer", samples=_log_int(rng, 1000, 4_000_000))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cpu")
    g.manual_seed(int(seed))
    return g


def _modes(seed, n, count=20):
    """Wave vectors, phases and solenoidal amplitudes of a turbulence-like field on a grid of n points a side:
    wave numbers spread over their logarithm up to six points a wave, energy falling as k^(-5/3)."""
    r = np.random.default_rng(seed)
    out = []
    while len(out) < count:
        mag = math.exp(r.uniform(0.0, math.log(max(2.0, n / 6.0))))
        dirn = r.standard_normal(3)
        k = np.rint(mag * dirn / np.linalg.norm(dirn)).astype(int)
        k2 = float(k @ k)
        if k2 < 1.0:
            continue
        a = r.standard_normal(3)
        a -= k * (a @ k) / k2
        out.append((k, r.uniform(0, 2 * math.pi), k2 ** (-1.0 / 6.0) * a / np.linalg.norm(a)))
    return out


class _Grid:
    """Angles 2 pi xi of the grid points as broadcastable tensors; tensors are laid out in the pencil's axis order."""

    def __init__(self, dims, walls="", pencil="x"):
        r = LAYOUT[pencil]
        fast = [m for m in ((0 + r) % 3, (1 + r) % 3, (2 + r) % 3)]
        self.dims = tuple(dims)
        self.axis = [2 - fast.index(d) for d in range(3)]  # tensor axis of direction d
        self.shape = tuple(dims[fast[2 - a]] for a in range(3))
        self.walls = [c in walls for c in "xyz"]
        self.xi = []
        for d in range(3):
            n = dims[d]
            x = torch.arange(n, dtype=torch.float64, device="cuda") / (n - 1 if self.walls[d] else n)
            s = [1, 1, 1]
            s[self.axis[d]] = n
            self.xi.append((2.0 * math.pi * x).reshape(s))

    def waves(self, modes):
        """cos and sin of every mode, one at a time."""
        for k, ph, a in modes:
            c = torch.polar(torch.ones_like(self.xi[0]), float(k[0]) * self.xi[0] + ph)
            for d in (1, 2):
                c = c * torch.polar(torch.ones_like(self.xi[d]), float(k[d]) * self.xi[d])
            yield k, a, c.real, c.imag


def _flow(grid, seed, mach=0.3, gradients=False):
    """rho, velocities, p, T of a compressible field with a turbulence-like spectrum (and Cartesian gradients
    of velocity and temperature on the 2 pi box)."""
    modes = _modes(seed, min(grid.dims))
    u = [torch.zeros(grid.shape, dtype=torch.float64, device="cuda") for _ in range(3)]
    th = torch.zeros(grid.shape, dtype=torch.float64, device="cuda")
    gu = [[torch.zeros_like(th) for _ in range(3)] for _ in range(3)] if gradients else None
    gt = [torch.zeros_like(th) for _ in range(3)] if gradients else None
    total = math.sqrt(sum(0.5 * float(a @ a) for _, _, a in modes))
    for m, (k, a, c, s) in enumerate(grid.waves(modes)):
        b = 0.03 * math.cos(1.0 + m) * float(a @ a)
        for i in range(3):
            u[i] += (mach * float(a[i]) / total) * c
            if gradients:
                for j in range(3):
                    if k[j]:
                        gu[i][j] -= (mach * float(a[i]) / total * float(k[j])) * s
        th += b * s
        if gradients:
            for j in range(3):
                if k[j]:
                    gt[j] += (b * float(k[j])) * c
    rho = 1.0 + 0.3 * th
    return dict(rho=rho, u=u, T=1.0 + th, p=rho * R_GAS * (1.0 + th), gu=gu, gt=gt)


def _spacing(dims, walls):
    return [1.0 / (n - 1) if c in walls else 1.0 / n for n, c in zip(dims, "xyz")]


def _metrics(grid):
    """J, J11 .. J33 of the 2 pi box; walled directions are stretched, x = 2 pi (xi - 0.06 sin(4 pi xi) / (4 pi))."""
    full = []
    for d in range(3):
        h = 2.0 * math.pi * torch.ones_like(grid.xi[d])
        if grid.walls[d]:
            h = h * (1.0 - 0.06 * torch.cos(2.0 * grid.xi[d]))
        full.append((1.0 / h).expand(grid.shape).contiguous())
    zero = torch.zeros(grid.shape, dtype=torch.float64, device="cuda")
    J = full[0] * full[1] * full[2]
    return [J, full[0], zero, zero, zero, full[1], zero, zero, zero, full[2]]


def _deck(dims, fd, filt, rk, les, avg, mu, walls="", testfilter=1):
    from mpi_3dcompact_amd import hit
    faces = {f: "ADIABATIC_WALL" for c in walls.upper() for f in (c + "0", c + "1")} or None
    return hit.options_text(dims[0], fd=fd, filt=filt, rk=rk, les=les, les_avg=avg, mu_ref=mu, dims=tuple(dims),
                            faces=faces, dsm_filter=testfilter)


class _DeviceField:
    """A solver's field as a device array; keeps the solver alive."""

    def __init__(self, solver, name):
        self.solver = solver
        self.__cuda_array_interface__ = dict(shape=tuple(solver.shape), typestr="<f8", strides=None, version=2,
                                             data=(solver.device_ptr(name), False))


CONSERVED = ("rho", "rhoU", "rhoV", "rhoW", "rhoE")


def _dims(case):
    return (case["nx"], case["ny"], case["nz"])


def _solver_flow(case, seed):
    grid = _Grid(_dims(case), case.get("walls", ""))
    f = _flow(grid, seed)
    for d in range(3):
        if grid.walls[d]:  # no slip at the walls
            for i in range(3):
                f["u"][i] *= torch.sin(0.5 * grid.xi[d])
    return grid, f


def _pairs(seed, n):
    """Standardised features and targets like the sampled training pairs."""
    g = _generator(seed)
    x = torch.randn((n, 7), generator=g)
    t = torch.stack([torch.sin(x[:, 0]) + x[:, 1] * x[:, 2], torch.tanh(x[:, 3] - x[:, 4])], dim=1)
    return x.cuda(), (t + 0.3 * torch.randn((n, 2), generator=g)).cuda()


def _network(seed):
    """Uniform initial weights with variance 1 / fan-in and small biases."""
    r = np.random.default_rng(seed)
    parts = []
    for fan, out in ((7, 64), (64, 64), (64, 64), (64, 2)):
        s = math.sqrt(3.0 / fan)
        parts.append([r.uniform(-s, s, (out, fan)), 0.1 * r.standard_normal(out)])
    return parts


def _pack(parts):
    """Parameter vector: the four weight matrices and biases, layer by layer."""
    return np.concatenate([np.concatenate([w.reshape(-1), b]) for w, b in parts]).astype(np.float32)


def _unpack(flat):
    out, at = [], 0
    for fan, n in ((7, 64), (64, 64), (64, 64), (64, 2)):
        out.append((flat[at:at + n * fan].reshape(n, fan), flat[at + n * fan:at + n * fan + n]))
        at += n * fan + n
    return out


def _feature_scaling(case, flow):
    """Standardisation of the closure's inputs from a sample of the field's own features."""
    f, _ = _features(case, flow, sample=True)
    mean = [float(v.mean()) for v in f]
    std = [max(float(v.std()), 1e-3) for v in f]
    return dict(in_mean=mean, in_std=std, out_mean=[0.02, 0.03], out_std=[0.01, 0.02],
                lo=[m - 5.0 * s for m, s in zip(mean, std)], hi=[m + 5.0 * s for m, s in zip(mean, std)])


def prepare(case, seed):
    fam = case["family"]
    st = {"case": case}
    if fam == "lines":
        from mpi_3dcompact_amd.ops import LineOp
        dims = _dims(case)
        grid = _Grid(dims, case["walls"], case["pencil"])
        dd = _spacing(dims, case["walls"])
        bc3 = tuple(int(w) for w in grid.walls)
        lay = LAYOUT[case["pencil"]]
        st["ins"] = _line_inputs(case, grid, seed)
        st["deriv"], st["filter"], st["outs"], st["filtered"] = [], [], [], []
        for s in case["schemes"].split("+"):
            cls, kind, af = SCHEMES[s]
            if cls == "deriv":
                st["deriv"] = [LineOp.deriv(kind, d, bc3[d], dims, dd[d], lay) for d in range(3)]
                st["outs"] = [[torch.empty_like(f) for f in st["ins"]] for _ in range(3)]
            else:
                st["filter"] = [LineOp.filter(kind, af, d, bc3, dims, lay) for d in range(3)]
                st["filtered"] = [torch.empty_like(f) for f in st["ins"]]
    elif fam == "solver":
        from mpi_3dcompact_amd.solver import Solver
        dims = _dims(case)
        grid, f = _solver_flow(case, seed)
        s = Solver(_deck(dims, case["fd"], case["filt"], case["rk"], case["les"], case["avg"], 1.0 / 1600.0,
                         case["walls"]), grid.shape)
        s.set_metrics([m.cpu().numpy() for m in _metrics(grid)])
        s.set_initial(dict(rho=f["rho"].cpu().numpy(), p=f["p"].cpu().numpy(),
                           **{n: v.cpu().numpy() for n, v in zip("UVW", f["u"])}))
        st["solver"] = s
        st["fields"] = {n: torch.as_tensor(_DeviceField(s, n), device="cuda") for n in CONSERVED}
    elif fam == "ensemble":
        from mpi_3dcompact_amd.ensemble import Ensemble
        sizes, mu = _members(case)
        e = Ensemble(_deck((sizes[0],) * 3, "PADE6", "COMPACT10", "RK4", "NOMODEL", "NONE", 1.0 / 1600.0),
                     [(n, n, n) for n in sizes], mu_ref=mu)
        for m, n in enumerate(sizes):
            grid = _Grid((n, n, n))
            f = _flow(grid, seed * 64 + m, mach=0.1 + 0.3 * m / len(sizes))
            e.set_metrics(m, [v.cpu().numpy() for v in _metrics(grid)])
            e.set_initial(m, dict(rho=f["rho"].cpu().numpy(), p=f["p"].cpu().numpy(),
                                  **{k: v.cpu().numpy() for k, v in zip("UVW", f["u"])}))
        st["ensemble"] = e
    elif fam in ("sgs", "learned"):
        from mpi_3dcompact_amd.sgs import Sgs
        dims = _dims(case)
        grid = _Grid(dims, "", case["pencil"])
        f = _flow(grid, seed, gradients=True)
        model = case["model"] if fam == "sgs" else "LEARNED"
        st["J"] = torch.full(grid.shape, (2.0 * math.pi) ** -3, dtype=torch.float64, device="cuda")
        deck = _deck(dims, "PENTA10", "COMPACT8", "KENRK4", model, case.get("avg", "NONE"), 1e-4,
                     testfilter=case.get("testfilter", 1))
        if fam == "learned":
            deck = deck.replace("CLOSUREFALLBACK = TRUE", "CLOSUREFALLBACK = FALSE") + "CLOSUREFEATURES = POINT\n"
        st["gradU"] = [f["gu"][i][j] for i in range(3) for j in range(3)]
        st["gradT"], st["rho"], st["T"] = f["gt"], f["rho"], f["T"]
        st["m"] = [f["rho"] * v for v in f["u"]]
        st["sgs"] = Sgs(deck, st["J"], layout=LAYOUT[case["pencil"]])
        st["out"] = [torch.empty_like(f["rho"]) for _ in range(3)]
        if fam == "learned":
            from mpi_3dcompact_amd.closure import Closure
            net = Closure(0)
            net.set_params(_pack(_network(3)))
            net.set_scaling(**_feature_scaling(case, f))
            st["sgs"].set_closure(net)
    else:
        from mpi_3dcompact_amd.closure import Closure
        st["net"] = Closure(0)
        st["net"].set_params(_pack(_network(seed)))
        st["X"], st["T"] = _pairs(seed, case["samples"])
    return st


def _line_inputs(case, grid, seed):
    f = _flow(grid, seed)
    rhoE = f["p"] / (GAMMA - 1.0) + 0.5 * f["rho"] * (f["u"][0] ** 2 + f["u"][1] ** 2 + f["u"][2] ** 2)
    return [f["rho"], f["u"][0], f["u"][1], f["u"][2], rhoE][:case["fields"]]


def _members(case):
    sizes = [int(v) for v in case["sizes"].split(",")]
    r = np.random.default_rng(case["seed"])
    return sizes, [float(r.uniform(1.0 / 3200.0, 1.0 / 800.0)) for _ in sizes]


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    case = st["case"]
    fam = case["family"]
    if fam == "lines":
        for d, op in enumerate(st["deriv"]):
            op.apply(st["ins"], st["outs"][d])
        if st["filter"]:
            st["filter"][0].apply(st["ins"], st["filtered"])
            st["filter"][1].apply(st["filtered"], st["filtered"])  # in place, as the solver filters
            st["filter"][2].apply(st["filtered"], st["filtered"])
        return dict(deriv=st["outs"], filtered=st["filtered"])
    if fam == "solver":
        st["solver"].step(1)
        return st["fields"]
    if fam == "ensemble":
        e = st["ensemble"]
        e.step(case["steps"])
        e.sync()
        return [[e.field(m, n) for n in CONSERVED] for m in range(len(e))]
    if fam == "sgs":
        mu, tau, k = st["out"]
        s = st["sgs"]
        if case["model"] == "VREMAN":
            s.vreman(st["gradU"], st["rho"], mu)
            return dict(mu=mu)
        s.dsm_mu_taukk(st["gradU"], st["rho"], *st["m"], mu, tau)
        s.dsm_ksgs(st["gradT"], st["rho"], *st["m"], st["T"], k)
        return dict(mu=mu, taukk=tau, k=k)
    if fam == "learned":
        mu, _, k = st["out"]
        st["sgs"].learned(st["gradU"], st["rho"], mu, k)
        return dict(mu=mu, k=k)
    if fam == "train":
        losses = st["net"].train(st["X"], st["T"], epochs=case["epochs"], batch=case["batch"], lr=1e-3, seed=5)
        return dict(losses=np.array(losses), params=st["net"].params())
    if fam == "gradient":
        g, loss = st["net"].gradient(st["X"], st["T"])
        st["net"].adam_step(g, lr=1e-3)
        return dict(grad=g, loss=loss)
    return dict(y=st["net"].infer(st["X"]))


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how exact its results are
# ---------------------------------------------------------------------------
FLOP_PER_PAIR = 2 * (7 * 64 + 64 * 64 + 64 * 64 + 64 * 2)  # forward pass of the network
STAGES = {"TVDRK3": 3, "RK4": 4, "KENRK4": 5}


def work(case):
    fam = case["family"]
    if fam == "lines":
        n = case["nx"] * case["ny"] * case["nz"] * case["fields"]
        arrays, flops = 1, 0
        for s in case["schemes"].split("+"):
            arrays += 3 if SCHEMES[s][0] == "deriv" else 1
            flops += 3 * {"cd2": 4, "pade6": 14, "penta10": 24, "compact8": 24, "compact10": 28, "commn5pade": 30,
                          "commn5exp": 14}[s]
        return dict(bytes=8.0 * n * arrays, flops=float(flops) * n)
    if fam == "solver":
        # state (5) and the previous momentum increments (3) in and out, ten metric fields in
        n = case["nx"] * case["ny"] * case["nz"]
        return dict(bytes=8.0 * n * 26, flops=900.0 * STAGES[case["rk"]] * n)
    if fam == "ensemble":
        n = sum(int(v) ** 3 for v in case["sizes"].split(","))
        return dict(bytes=8.0 * n * 26 * case["steps"], flops=900.0 * 4 * case["steps"] * n)
    if fam == "sgs":
        # in: 9 velocity gradients, rho, J, and for the dynamic model 3 momenta, 3 temperature gradients, T
        n = case["nx"] * case["ny"] * case["nz"]
        return dict(bytes=8.0 * n * (12 if case["model"] == "VREMAN" else 21),
                    flops=(150.0 if case["model"] == "VREMAN" else 4000.0) * n)
    if fam == "learned":
        n = case["nx"] * case["ny"] * case["nz"]
        return dict(bytes=8.0 * n * 13, flops=(FLOP_PER_PAIR + 300.0) * n)
    if fam == "train":
        n = case["samples"] * case["epochs"]
        return dict(bytes=4.0 * 10 * n, flops=3.0 * FLOP_PER_PAIR * n)
    if fam == "gradient":
        return dict(bytes=4.0 * (9 * case["samples"] + 6 * N_PARAMS), flops=3.0 * FLOP_PER_PAIR * case["samples"])
    return dict(bytes=4.0 * 9 * case["samples"], flops=float(FLOP_PER_PAIR) * case["samples"])


def tolerance(case):
    """About four times the errors measured against exact() (for the training, the spread under a change of the
    initial weights by one part in 10^7)."""
    fam = case["family"]
    if fam == "lines":  # derivatives of a density that varies by a percent lose two digits
        return {"rel": 8e-12, "max": 1e-9}
    if fam in ("solver", "ensemble"):
        return {"rel": 1e-13, "max": 1e-11}
    if fam == "sgs":  # ratios of averaged contractions
        return {"rel": 1e-10, "max": 1e-8}
    if fam == "learned":  # bf16 products
        return {"rel": 2.5e-3, "max": 0.05}
    if fam == "train":
        return {"rel": 1e-3, "max": 0.02}
    if fam == "gradient":
        return {"rel": 1.4e-2, "max": 0.3}
    return {"rel": 1e-2, "max": 0.2}


# ---------------------------------------------------------------------------
# 64-bit restatement
# ---------------------------------------------------------------------------
def _cyclic(n, taps):
    m = np.zeros((n, n))
    i = np.arange(n)
    for off, v in taps.items():
        m[i, (i + off) % n] += v
    return m


def _sym(c):
    return {s * k: v for k, v in enumerate(c) for s in ((1,) if k == 0 else (1, -1))}


def _odd(c):
    return {s * (k + 1): s * v for k, v in enumerate(c) for s in (1, -1)}


def _one_sided(m, r0, rows, sign):
    """Boundary rows r0, r0 + 1, .. of m over the first points, mirrored (times sign) at the far end."""
    n = m.shape[0]
    for r, c in enumerate(rows):
        m[r0 + r] = 0.0
        m[n - 1 - r0 - r] = 0.0
        for j, v in enumerate(c):
            m[r0 + r, j] += v
            m[n - 1 - r0 - r, n - 1 - j] += sign * v


def _compact8_rows(a):
    return [
        [1 / 256 + 127 * a / 128, 31 / 32 + a / 16, 7 / 64 + 25 * a / 32, -7 / 32 + 7 * a / 16,
         7 * (5 - 10 * a) / 128, -7 / 32 + 7 * a / 16, 7 / 64 - 7 * a / 32, -1 / 32 + a / 16, 1 / 256 - a / 128],
        [-1 / 256 + a / 128, 1 / 32 + 15 * a / 16, 57 / 64 + 7 * a / 32, 7 / 32 + 9 * a / 16,
         7 * (-5 + 10 * a) / 128, 7 / 32 - 7 * a / 16, -7 / 64 + 7 * a / 32, 1 / 32 - a / 16, -1 / 256 + a / 128],
        [1 / 256 - a / 128, -1 / 32 + a / 16, 7 / 64 + 25 * a / 32, 25 / 32 + 7 * a / 16,
         35 / 128 + 29 * a / 64, -7 / 32 + 7 * a / 16, 7 / 64 - 7 * a / 32, -1 / 32 + a / 16, 1 / 256 - a / 128]]


def _compact10_rows(a):
    """Row r = 1 .. 4: the tenth difference at the wall, weighted so that the filter passes polynomials of degree 9:
    row_r = A_r + (1 - 2 a) / 1024 (-1)^(r) delta, delta the alternating binomials of 10."""
    rows = []
    for r in range(1, 5):
        c = [(-1) ** (r + 1 + j) * math.comb(10, j) * (1 - 2 * a) / 1024 for j in range(11)]
        c[r - 1] += a
        c[r] += 1.0
        c[r + 1] += a
        rows.append(c)
    return rows


def _matrix(scheme, n, wall, dd=1.0):
    """Dense operator of one line: derivative (divided by dd) or filter."""
    cls, kind, af = SCHEMES[scheme]
    return _matrix_of(scheme, n, wall, dd, af)


def _matrix_of(scheme, n, wall, dd, af):
    ident = np.eye(n)
    if scheme == "cd2":
        # the interior carries the opposite sign of the end rows
        b = _cyclic(n, {1: -0.5, -1: 0.5})
        if wall:
            _one_sided(b, 0, [[-1.5, 2.0, -0.5]], 1.0)
        else:
            b[0] *= -1.0
            b[n - 1] *= -1.0
        return b / dd
    if scheme == "pade6":
        a, b = _cyclic(n, _sym([1.0, 1.0 / 3.0])), _cyclic(n, _odd([7.0 / 9.0, 1.0 / 36.0]))
        if wall:
            _one_sided(a, 0, [[1.0, 2.0], [1.0 / 6.0, 1.0, 0.5]], 1.0)
            _one_sided(b, 0, [[-2.5, 2.0, 0.5], [-5.0 / 9.0, -0.5, 1.0, 1.0 / 18.0]], -1.0)
        return np.linalg.solve(a, b) / dd
    if scheme == "penta10":
        a = _cyclic(n, _sym([1.0, 0.5, 0.05]))
        b = _cyclic(n, _odd([17.0 / 24.0, 101.0 / 600.0, 1.0 / 600.0]))
        if wall:
            _one_sided(a, 0, [[1.0, 5.0], [1.0 / 12.0, 1.0, 1.25], [1.0 / 36.0, 4.0 / 9.0, 1.0, 4.0 / 9.0, 1.0 / 36.0]],
                       1.0)
            _one_sided(b, 0, [[-197.0 / 60.0, -5.0 / 12.0, 5.0, -5.0 / 3.0, 5.0 / 12.0, -1.0 / 20.0],
                              [-79.0 / 240.0, -77.0 / 60.0, 55.0 / 48.0, 5.0 / 9.0, -5.0 / 48.0, 1.0 / 60.0,
                               -1.0 / 720.0],
                              [-25.0 / 216.0, -20.0 / 27.0, 0.0, 20.0 / 27.0, 25.0 / 216.0]], -1.0)
        return np.linalg.solve(a, b) / dd
    if scheme == "compact8":
        a = _cyclic(n, _sym([1.0, af]))
        b = _cyclic(n, _sym([(93 + 70 * af) / 128, (7 + 18 * af) / 32, (-7 + 14 * af) / 64, (1 - 2 * af) / 32,
                             (-1 + 2 * af) / 256]))
        if wall:
            _one_sided(a, 0, [[1.0]], 1.0)
            _one_sided(b, 0, [[1.0]] + _compact8_rows(af), 1.0)
        return np.linalg.solve(a, b)
    if scheme == "compact10":
        a = _cyclic(n, _sym([1.0, af]))
        b = _cyclic(n, _sym([(193 + 126 * af) / 256, (105 + 302 * af) / 512, (-15 + 30 * af) / 128,
                             (45 - 90 * af) / 1024, (-5 + 10 * af) / 512, (1 - 2 * af) / 1024]))
        if wall:
            _one_sided(a, 0, [[1.0]], 1.0)
            _one_sided(b, 0, [[1.0]] + _compact10_rows(af), 1.0)
        return np.linalg.solve(a, b)
    exp = [11.0 / 16.0, 15.0 / 64.0, -3.0 / 32.0, 1.0 / 64.0]
    ends = [[31 / 32, 5 / 32, -5 / 16, 5 / 16, -5 / 32, 1 / 32], [1 / 32, 27 / 32, 5 / 16, -5 / 16, 5 / 32, -1 / 32],
            [-1 / 32, 5 / 32, 11 / 16, 5 / 16, -5 / 32, 1 / 32]]
    if scheme == "commn5exp":
        b = _cyclic(n, _sym(exp))
        if wall:
            _one_sided(b, 0, ends, 1.0)
        return b
    a = _cyclic(n, {0: 7.0 / 12.0, 2: 5.0 / 24.0, -2: 5.0 / 24.0})
    b = _cyclic(n, _sym([7.0 / 24.0, 175.0 / 768.0, 5.0 / 48.0, 35.0 / 1536.0, 0.0, -1.0 / 1536.0]))
    if wall:
        inner = [exp[3], exp[2], exp[1], exp[0], exp[1], exp[2], exp[3]]
        _one_sided(b, 0, ends + [inner, [0.0] + inner], 1.0)
        for r in range(5):
            a[r], a[n - 1 - r] = ident[r], ident[n - 1 - r]
    return np.linalg.solve(a, b)


def _along(m, f, axis):
    """The matrix m applied along a tensor axis."""
    if axis == 2:
        return torch.matmul(f, m.T)
    if axis == 0:
        return torch.matmul(m, f.reshape(f.shape[0], -1)).reshape(f.shape)
    return torch.stack([torch.matmul(m, s) for s in f])


def _cuda(m):
    return torch.from_numpy(np.ascontiguousarray(m)).cuda()


def _filter_along(grid, m, f, d):
    """The filter along direction d; lines on a walled face of another direction keep their values."""
    out = _along(m, f, grid.axis[d])
    for e in range(3):
        if e != d and grid.walls[e]:
            for i in (0, grid.dims[e] - 1):
                out.select(grid.axis[e], i).copy_(f.select(grid.axis[e], i))
    return out


def _exact_lines(case, seed):
    dims = _dims(case)
    grid = _Grid(dims, case["walls"], case["pencil"])
    ins = _line_inputs(case, grid, seed)
    dd = _spacing(dims, case["walls"])
    deriv, filtered = [], []
    for s in case["schemes"].split("+"):
        m = [_cuda(_matrix(s, dims[d], grid.walls[d], dd[d])) for d in range(3)]
        if SCHEMES[s][0] == "deriv":
            deriv = [[_along(m[d], f, grid.axis[d]) for f in ins] for d in range(3)]
        else:
            for f in ins:
                for d in range(3):
                    f = _filter_along(grid, m[d], f, d)
                filtered.append(f)
    return dict(deriv=deriv, filtered=filtered)


def _vreman(g, rho, delta2):
    """Eddy viscosity from g[i][j] = du_i/dx_j; the norm counts dw/dy twice and dv/dz not at all."""
    b = [[delta2 * (g[i][0] * g[j][0] + g[i][1] * g[j][1] + g[i][2] * g[j][2]) for j in range(3)] for i in range(3)]
    ab = (g[0][0] ** 2 + g[1][0] ** 2 + g[2][0] ** 2 + g[0][1] ** 2 + g[1][1] ** 2 + 2.0 * g[2][1] ** 2 +
          g[0][2] ** 2 + g[2][2] ** 2)
    bb = (b[0][0] * b[1][1] - b[0][1] ** 2 + b[0][0] * b[2][2] - b[0][2] ** 2 + b[1][1] * b[2][2] - b[1][2] ** 2)
    mu = 2.5 * 0.17 * 0.17 * rho * torch.sqrt(bb.clamp_min(1e-12) / (ab + 1e-12))
    return torch.minimum(mu, 0.05 * delta2 * torch.sqrt(2.0 * ab))


class _Box64:
    """Time steps of a periodic 2 pi box in 64 bits."""

    def __init__(self, dims, fd, filt, rk, les, avg, mu_ref, flow):
        self.grid = _Grid(dims)
        self.dims, self.rk, self.les, self.mu_ref = dims, rk, les, mu_ref
        self.D = [_cuda(_matrix(fd.lower(), dims[d], False, 1.0 / dims[d])) for d in range(3)]
        self.F = [_cuda(_matrix(filt.lower(), dims[d], False)) for d in range(3)]
        self.A = [_cuda(_matrix_of("compact10", dims[d], False, 1.0, -0.49)) for d in range(3)] if avg == "LOCAL" else None
        rho, u, p = flow["rho"], flow["u"], flow["p"]
        self.q = [rho, rho * u[0], rho * u[1], rho * u[2],
                  p / (GAMMA - 1.0) + 0.5 * rho * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)]
        self.k2 = [torch.zeros_like(rho) for _ in range(3)]

    def d(self, f, i):
        return _along(self.D[i], f, self.grid.axis[i])

    def three(self, m, f):
        for i in (1, 2, 0):
            f = _along(m[i], f, self.grid.axis[i])
        return f

    @staticmethod
    def prim(q):
        u = [q[i] / q[0] for i in (1, 2, 3)]
        p = (GAMMA - 1.0) * (q[4] - 0.5 * q[0] * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2))
        return u, p, p / (q[0] * R_GAS)

    def divergence(self, q):
        L = 2.0 * math.pi
        u, p, T = self.prim(q)
        mu = self.mu_ref * T ** 0.76
        g = [[self.d(u[i], j) / L for j in range(3)] for i in range(3)]
        gT = [self.d(T, j) / L for j in range(3)]
        mu_eff, k_eff = mu, CP / PRANDTL * mu
        if self.les == "VREMAN":
            delta2 = (L ** 3 / (self.dims[0] * self.dims[1] * self.dims[2])) ** (2.0 / 3.0)
            ms = _vreman(g, q[0], delta2)
            if self.A is not None:
                ms = self.three(self.A, ms)
            mu_eff = (mu + ms).clamp_min(0.0)
            k_eff = (CP * (mu / PRANDTL + ms / 0.9)).clamp_min(0.0)
        tr = (g[0][0] + g[1][1] + g[2][2]) * (2.0 / 3.0)
        div = [torch.zeros_like(p) for _ in range(5)]
        for j in range(3):
            tau = [mu_eff * (g[i][j] + g[j][i] - (tr if i == j else 0.0)) for i in range(3)]
            heat = k_eff * gT[j] + sum(u[i] * tau[i] for i in range(3))
            flux = [q[0] * u[j]] + [q[1 + i] * u[j] + (p if i == j else 0.0) - tau[i] for i in range(3)]
            flux.append((q[4] + p) * u[j] - heat)
            for e in range(5):
                div[e] += self.d(flux[e] * L ** 2, j)  # J_jj / J = L^2
        return div

    def step(self):
        L = 2.0 * math.pi
        u, p, _ = self.prim(self.q)
        c = torch.sqrt(GAMMA * p / self.q[0])
        dt = 0.5 / float(sum((u[i].abs() + c) / L * self.dims[i] for i in range(3)).max())
        dtJ = dt / L ** 3
        stages = STAGES[self.rk]
        q1 = self.q
        rk, acc, reg = q1, None, None
        for s in range(stages):
            div = self.divergence(rk)
            # momentum increments carry the previous stage's increment
            k = [-dtJ * div[0]] + [(self.k2[i] - div[1 + i]) * dtJ for i in range(3)] + [-dtJ * div[4]]
            self.k2 = k[1:4]
            if self.rk == "TVDRK3":
                a, b, w = ((0.0, 1.0, 1.0), (0.75, 0.25, 0.25), (1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0))[s]
                rk = [a * x + b * y + w * z for x, y, z in zip(q1, rk, k)]
            elif self.rk == "RK4":
                a, b = (1 / 6, 1 / 3, 1 / 3, 1 / 6)[s], (0.5, 0.5, 1.0, 0.0)[s]
                acc = [x + a * z for x, z in zip(q1 if acc is None else acc, k)]
                rk = [x + b * z for x, z in zip(q1, k)] if s < 3 else acc
            else:
                a = (0.0, -6234157559845.0 / 12983515589748.0, -6194124222391.0 / 4410992767914.0,
                     -31623096876824.0 / 15682348800105.0, -12251185447671.0 / 11596622555746.0)[s]
                b = (494393426753.0 / 4806282396855.0, 4047970641027.0 / 5463924506627.0,
                     9795748752853.0 / 13190207949281.0, 4009051133189.0 / 8539092990294.0,
                     1348533437543.0 / 7166442652324.0)[s]
                reg = k if reg is None else [z + a * x for x, z in zip(reg, k)]
                rk = [x + b * z for x, z in zip(rk, reg)]
        self.q = [self.three(self.F, x) for x in rk]


def _exact_sgs(case, seed):
    dims = _dims(case)
    grid = _Grid(dims, "", case["pencil"])
    f = _flow(grid, seed, gradients=True)
    rho, g, gT, T = f["rho"], f["gu"], f["gt"], f["T"]
    delta2 = ((2.0 * math.pi) ** 3 / (dims[0] * dims[1] * dims[2])) ** (2.0 / 3.0)

    def three(mats, x):
        for d in (1, 2, 0):
            x = _along(mats[d], x, grid.axis[d])
        return x

    if case["model"] == "VREMAN":
        mu = _vreman(g, rho, delta2)
        if case["avg"] == "LOCAL":
            mu = three([_cuda(_matrix_of("compact10", n, False, 1.0, -0.49)) for n in dims], mu)
        return dict(mu=mu)
    name = "commn5pade" if case["testfilter"] == 1 else "commn5exp"
    mats = [_cuda(_matrix(name, n, False)) for n in dims]

    def hat(x):
        return three(mats, x)

    def avg(x):
        if case["avg"] == "GLOBAL":
            return x.mean()
        return x.mean(dim=grid.axis[0 if case["avg"] == "XI1_AVG" else 2], keepdim=True)

    pairs = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]
    S = {ij: 0.5 * (g[ij[0]][ij[1]] + g[ij[1]][ij[0]]) for ij in pairs}
    smag = torch.sqrt(2.0 * sum((1.0 if i == j else 2.0) * S[i, j] ** 2 for i, j in pairs))

    def dev(X):
        tr = (X[0, 0] + X[1, 1] + X[2, 2]) / 3.0
        return {ij: X[ij] - tr if ij[0] == ij[1] else X[ij] for ij in pairs}

    Sd, Shd = dev(S), dev({ij: hat(S[ij]) for ij in pairs})
    rho_h, smag_h = hat(rho), hat(smag)
    M = {ij: hat(2.0 * rho * smag * Sd[ij]) - 8.0 * rho_h * smag_h * Shd[ij] for ij in pairs}
    m = [rho * v for v in f["u"]]
    mh = [hat(v) for v in m]
    Lm = {(i, j): hat(m[i] * m[j] / rho) - mh[i] * mh[j] / rho_h for i, j in pairs}
    Ld = dev(Lm)
    LM = avg(sum((1.0 if i == j else 2.0) * Ld[i, j] * M[i, j] for i, j in pairs))
    MM = avg(sum((1.0 if i == j else 2.0) * M[i, j] ** 2 for i, j in pairs))
    mu = rho * smag * LM / MM
    ci = avg(8.0 * rho_h * smag_h ** 2 - hat(2.0 * rho * smag ** 2))
    tau = 2.0 * rho * smag ** 2 * avg(Lm[0, 0] + Lm[1, 1] + Lm[2, 2]) / ci
    nv = [4.0 * rho_h * smag_h * hat(gT[i]) - hat(rho * smag * gT[i]) for i in range(3)]
    rTh = hat(rho * T)
    kv = [hat(m[i] * T) - mh[i] * rTh / rho for i in range(3)]
    k = -CP * avg(sum(a * b for a, b in zip(nv, kv))) / avg(sum(a * a for a in nv)) * rho * smag
    return dict(mu=mu, taukk=tau, k=k)


def _features(case, f, sample=False):
    """The seven invariants of the velocity gradient with |S| and Delta^2."""
    dims = _dims(case)
    g = torch.stack([torch.stack([f["gu"][i][j].reshape(-1) for j in range(3)], -1) for i in range(3)], -2)
    if sample:
        g = g[:: max(1, g.shape[0] // 4096)]
    S, W = 0.5 * (g + g.transpose(1, 2)), 0.5 * (g - g.transpose(1, 2))

    def dot(a, b):
        return (a * b.transpose(1, 2)).sum((1, 2))

    def product(a, b):
        return (a.unsqueeze(3) * b.unsqueeze(1)).sum(2)

    SS, WW = product(S, S), product(W, W)
    s2, w2 = (S * S).sum((1, 2)), (W * W).sum((1, 2))
    a = torch.sqrt(s2 + w2)
    log_delta = math.log((2.0 * math.pi) ** 3 / (dims[0] * dims[1] * dims[2])) / 3.0
    feats = [g.diagonal(dim1=1, dim2=2).sum(1) / a, (s2 - w2) / a ** 2, dot(SS, S) / a ** 3, dot(S, WW) / a ** 3,
             dot(SS, WW) / a ** 4, torch.log(a), torch.full_like(a, log_delta)]
    return feats, (torch.sqrt(2.0 * s2), math.exp(2.0 * log_delta))


def _mlp(parts, x):
    for i, (w, b) in enumerate(parts):
        x = x @ w.T + b
        if i < 3:
            x = 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))
    return x


def _params64(flat):
    return [(w.clone().requires_grad_(True), b.clone().requires_grad_(True))
            for w, b in _unpack(torch.from_numpy(flat.astype(np.float64)).cuda())]


def exact(case, seed):
    fam = case["family"]
    if fam == "lines":
        return _exact_lines(case, seed)
    if fam == "solver":
        if case["walls"]:
            return None  # no restatement of the wall treatment
        _, f = _solver_flow(case, seed)
        box = _Box64(_dims(case), case["fd"], case["filt"], case["rk"], case["les"], case["avg"], 1.0 / 1600.0, f)
        box.step()
        return dict(zip(CONSERVED, box.q))
    if fam == "ensemble":
        sizes, mu = _members(case)
        out = []
        for m, n in enumerate(sizes):
            f = _flow(_Grid((n, n, n)), seed * 64 + m, mach=0.1 + 0.3 * m / len(sizes))
            box = _Box64((n, n, n), "PADE6", "COMPACT10", "RK4", "NOMODEL", "NONE", mu[m], f)
            for _ in range(case["steps"]):
                box.step()
            out.append([q.cpu().numpy() for q in box.q])
        return out
    if fam == "sgs":
        return _exact_sgs(case, seed)
    if fam == "learned":
        grid = _Grid(_dims(case), "", case["pencil"])
        f = _flow(grid, seed, gradients=True)
        sc = {k: torch.tensor(np.float32(v).astype(np.float64), device="cuda")
              for k, v in _feature_scaling(case, f).items()}
        feats, (smag, delta2) = _features(case, f)
        x = torch.minimum(torch.maximum(torch.stack(feats, 1), sc["lo"]), sc["hi"])
        with torch.no_grad():
            y = _mlp(_params64(_pack(_network(3))), (x - sc["in_mean"]) / sc["in_std"]) * sc["out_std"] + sc["out_mean"]
        base = f["rho"].reshape(-1) * delta2 * smag
        return dict(mu=(base * y[:, 0]).reshape(grid.shape), k=(CP * base * y[:, 1]).reshape(grid.shape))
    if fam == "train":
        return None  # the visiting order is the library's own
    X, T = _pairs(seed, case["samples"])
    parts = _params64(_pack(_network(seed)))
    if fam == "infer":
        with torch.no_grad():
            return dict(y=_mlp(parts, X.double()))
    loss = ((_mlp(parts, X.double()) - T.double()) ** 2).mean()
    loss.backward()
    return dict(grad=torch.cat([torch.cat([w.grad.reshape(-1), b.grad]) for w, b in parts]), loss=float(loss))
