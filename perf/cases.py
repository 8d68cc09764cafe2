"""Workloads of the batched propagator for timing and comparing two builds.

Every case goes through the package's public entry points (crpropa3_amd.capi and
crpropa3_amd.adjoint) as a steering program uses them:

* "eval": Field.eval of host positions (a line of sight, a plotted map);
* "run": a Batch is reset from the uploaded start state, propagated, and its final state (and the
  observer's detections) downloaded;
* "adjoint": the loss of differentiable Boris propagation and its gradients.

listed() holds the cases, draw(rng) gives more from the same ranges, prepare/run/work/tolerance/exact
describe one case.  Fields and particles are made here from the seed: a transverse Gaussian random field
with a Kolmogorov spectrum on the grid, a plane-wave mode table, power-law energies and isotropic
directions.
"""
import math

import numpy as np
import torch

from crpropa3_amd import capi

PC = 648000 / math.pi * 149597870700.0
KPC, MPC = 1e3 * PC, 1e6 * PC
EPLUS = 1.602176487e-19
EV = EPLUS
EEV = 1e18 * EV
C_LIGHT = 2.99792458e8
NG, MUG = 1e-13, 1e-10

# ---------------------------------------------------------------------------- cases


def listed():
    return [
        # the field along a line of sight: a thousand positions of a small grid, the shortest call there is
        dict(name="eval_sightline", kind="eval", field="grid", nx=64, ny=64, nz=64, spacing=50 * KPC, n=1000,
             precision="fp64"),
        # a few thousand protons with fixed Boris steps in a 64^3 grid: fewer particles than the GPU has lanes
        dict(name="bp_grid64", kind="run", prop="BP", field="grid", nx=64, ny=64, nz=64, spacing=50 * KPC, n=4096,
             steps=2000, min_step=100 * KPC, max_step=100 * KPC, emin=1, emax=100, nuclei=0, precision="fp64"),
        # adaptive Boris steps of nuclei in a reflective grid of odd shape, stopped by a sphere or the length
        # limit, with snapshots of an observer on the way
        dict(name="bp_adaptive_observer", kind="run", prop="BP", field="grid", nx=97, ny=80, nz=101, spacing=20 * KPC,
             reflective=1, n=20011, min_step=1 * KPC, max_step=200 * KPC, tol=1e-3, max_length=20 * MPC, snapshots=4,
             sphere=10 * MPC, emin=1, emax=100, nuclei=1, precision="fp64"),
        # fixed Boris steps through a grid read with tricubic interpolation
        dict(name="bp_tricubic128", kind="run", prop="BP", field="grid", nx=128, ny=128, nz=128, spacing=20 * KPC,
             interpolation="TRICUBIC", n=65536, steps=300, min_step=20 * KPC, max_step=20 * KPC, emin=1, emax=100,
             nuclei=0, precision="fp64"),
        # the benchmark's default: a million nuclei, adaptive Cash-Karp to 100 Mpc in a 256^3 grid
        dict(name="ck_grid256", kind="run", prop="CK", field="grid", nx=256, ny=256, nz=256, spacing=20 * KPC,
             n=2 ** 20, min_step=1 * KPC, max_step=1 * MPC, tol=1e-4, max_length=100 * MPC, emin=1, emax=300, nuclei=1,
             precision="fp64"),
        # the mixed-precision path with FP16 bricks: high-rigidity protons, a fixed number of adaptive steps
        dict(name="ck_mixed_fp16", kind="run", prop="CK", field="grid", nx=256, ny=256, nz=256, spacing=20 * KPC,
             n=2 ** 19, steps=200, min_step=1 * KPC, max_step=100 * KPC, tol=1e-4, emin=10, emax=300, nuclei=0,
             precision="mixed", storage="fp16"),
        # two million protons in a 512^3 grid, whose cell table outgrows the address translation caches
        dict(name="bp_grid512", kind="run", prop="BP", field="grid", nx=512, ny=512, nz=512, spacing=10 * KPC,
             n=2 ** 21, steps=1000, min_step=20 * KPC, max_step=20 * KPC, emin=1, emax=100, nuclei=0,
             precision="fp64"),
        # plane-wave turbulence summed on the fly, exact path
        dict(name="planewave_fp64", kind="run", prop="BP", field="planewave", nm=256, lmin=1 * PC, lmax=100 * PC,
             brms=1 * MUG, n=2 ** 18, steps=300, min_step=0.05 * PC, max_step=0.05 * PC, emin=1e-3, emax=1, nuclei=0,
             precision="fp64"),
        # the same model on the mixed-precision path
        dict(name="planewave_mixed", kind="run", prop="BP", field="planewave", nm=256, lmin=1 * PC, lmax=100 * PC,
             brms=1 * MUG, n=2 ** 19, steps=1500, min_step=0.05 * PC, max_step=0.05 * PC, emin=3e-2, emax=1, nuclei=0,
             precision="mixed"),
        # stochastic transport along the field lines
        dict(name="sde_grid256", kind="run", prop="SDE", field="grid", nx=256, ny=256, nz=256, spacing=1 * PC,
             n=2 ** 20, min_step=0.1 * PC, max_step=10 * PC, tol=1e-4, max_length=1 * KPC, emin=1e-6, emax=1e-3,
             nuclei=0, precision="fp64"),
        # back-tracking antiprotons through the Galactic model with its striated and turbulent grids
        dict(name="ck_jf12", kind="run", prop="CK", field="jf12", n=2 ** 16, steps=1500, min_step=0.1 * PC,
             max_step=0.1 * PC, emin=1, emax=1.0001, nuclei=-1, precision="fp64"),
        # loss and gradients of the differentiable Boris push
        dict(name="adjoint_grid128", kind="adjoint", nx=128, ny=128, nz=128, spacing=20 * KPC, n=65536, steps=4096,
             checkpoint=64, step=10 * KPC, emin=20, emax=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, lo, hi):
    """A grid shape: mostly cubes, else three sizes of their own."""
    n = _log_int(rng, lo, hi)
    if rng.random() < 0.6:
        return dict(nx=n, ny=n, nz=n)
    return dict(nx=n, ny=max(4, int(n * rng.uniform(0.7, 1.0))), nz=max(4, int(n * rng.uniform(0.7, 1.0))))


def draw(rng):
    kind = rng.choice(["eval", "bp", "bp", "bp_adaptive", "tricubic", "ck", "ck", "ck_mixed", "grid512", "planewave",
                       "planewave", "sde", "jf12", "adjoint"])
    if kind == "eval":
        return dict(kind="eval", field="grid", spacing=50 * KPC, n=_log_int(rng, 1, 200000),
                    precision=rng.choice(["fp64", "mixed"]), reflective=int(rng.random() < 0.3), **_shape(rng, 8, 128))
    if kind == "bp":
        precision = rng.choice(["fp64", "fp64", "mixed"])
        return dict(kind="run", prop="BP", field="grid", spacing=50 * KPC, n=_log_int(rng, 500, 300000),
                    steps=_log_int(rng, 50, 1000 if precision == "fp64" else 60), min_step=20 * KPC, max_step=20 * KPC,
                    emin=1 if precision == "fp64" else 10, emax=100, nuclei=0, precision=precision,
                    reflective=int(rng.random() < 0.3), **_shape(rng, 16, 160))
    if kind == "bp_adaptive":
        return dict(kind="run", prop="BP", field="grid", spacing=20 * KPC, reflective=int(rng.random() < 0.5),
                    n=_log_int(rng, 500, 60000), min_step=1 * KPC, max_step=200 * KPC, tol=1e-3,
                    max_length=rng.uniform(5, 20) * MPC, snapshots=rng.choice([0, 1, 4, 7]),
                    sphere=rng.choice([0, 10 * MPC]), emin=1, emax=100, nuclei=1, precision="fp64",
                    **_shape(rng, 16, 128))
    if kind == "tricubic":
        return dict(kind="run", prop="BP", field="grid", spacing=20 * KPC, interpolation="TRICUBIC",
                    reflective=int(rng.random() < 0.3), n=_log_int(rng, 500, 65536), steps=_log_int(rng, 50, 300),
                    min_step=20 * KPC, max_step=20 * KPC, emin=1, emax=100, nuclei=0, precision="fp64",
                    **_shape(rng, 16, 128))
    if kind == "ck":
        return dict(kind="run", prop="CK", field="grid", spacing=20 * KPC, n=_log_int(rng, 1000, 300000),
                    min_step=1 * KPC, max_step=1 * MPC, tol=1e-4, max_length=rng.uniform(5, 50) * MPC, emin=1, emax=300,
                    nuclei=1, precision="fp64", reflective=int(rng.random() < 0.2), **_shape(rng, 32, 256))
    if kind == "ck_mixed":
        return dict(kind="run", prop="CK", field="grid", spacing=20 * KPC, n=_log_int(rng, 1000, 500000),
                    steps=_log_int(rng, 50, 200), min_step=1 * KPC, max_step=100 * KPC, tol=1e-4, emin=10, emax=300,
                    nuclei=0, precision="mixed", storage=rng.choice(["fp32", "fp16"]), **_shape(rng, 32, 256))
    if kind == "grid512":
        n = rng.randint(300, 512)
        return dict(kind="run", prop="BP", field="grid", nx=n, ny=n, nz=n, spacing=10 * KPC,
                    n=_log_int(rng, 100000, 2 ** 20), steps=_log_int(rng, 200, 1000), min_step=20 * KPC,
                    max_step=20 * KPC, emin=1, emax=100, nuclei=0, precision="fp64")
    if kind == "planewave":
        precision = rng.choice(["fp64", "mixed"])
        nm = _log_int(rng, 20, 400)
        budget = 2e10 if precision == "fp64" else 2e11  # particles x steps x modes
        n = _log_int(rng, 2000, 300000)
        steps = max(20, min(_log_int(rng, 50, 1500), int(budget / (n * nm))))
        return dict(kind="run", prop="BP", field="planewave", nm=nm, lmin=1 * PC, lmax=100 * PC, brms=1 * MUG, n=n,
                    steps=steps, min_step=0.05 * PC, max_step=0.05 * PC, emin=1e-3 if precision == "fp64" else 3e-2,
                    emax=1, nuclei=0, precision=precision)
    if kind == "sde":
        return dict(kind="run", prop="SDE", field="grid", spacing=1 * PC, n=_log_int(rng, 1000, 500000),
                    min_step=0.1 * PC, max_step=10 * PC, tol=1e-4, max_length=rng.uniform(0.1, 1) * KPC, emin=1e-6,
                    emax=1e-3, nuclei=0, precision="fp64", **_shape(rng, 32, 256))
    if kind == "jf12":
        return dict(kind="run", prop=rng.choice(["BP", "CK"]), field="jf12", n=_log_int(rng, 1000, 65536),
                    steps=_log_int(rng, 500, 1500), min_step=0.1 * PC, max_step=0.1 * PC, emin=1, emax=10,
                    nuclei=-1, precision="fp64")
    return dict(kind="adjoint", spacing=20 * KPC, n=_log_int(rng, 1000, 65536), steps=_log_int(rng, 64, 1024),
                checkpoint=rng.choice([16, 50, 64, 100]), step=10 * KPC, emin=3, emax=100, **_shape(rng, 16, 160))


# ---------------------------------------------------------------------------- inputs


def _dev():
    return torch.device("cuda:0")


def _grid(case, seed, brms):
    """(nx, ny, nz, 3) float32 transverse Gaussian random field, <|B(k)|^2> ~ k^-11/3 between 2 cells and half
    the box, rms |B| = brms."""
    n = (case["nx"], case["ny"], case["nz"])
    gen = torch.Generator(device=_dev())
    gen.manual_seed(1000003 * seed + 17)
    k = [torch.fft.fftfreq(n[0], device=_dev()), torch.fft.fftfreq(n[1], device=_dev()),
         torch.fft.rfftfreq(n[2], device=_dev())]
    kx, ky, kz = k[0][:, None, None], k[1][None, :, None], k[2][None, None, :]
    k2 = kx * kx + ky * ky + kz * kz
    band = (k2 <= 0.25) & (k2 >= (2.0 / max(n)) ** 2)
    amp = torch.where(band, k2.clamp_min(1e-12) ** (-11.0 / 12.0), torch.zeros((), device=_dev()))
    v = []
    for _ in range(3):
        c = torch.fft.rfftn(torch.randn(n, generator=gen, device=_dev()))
        v.append(c.mul_(amp))
    div = (kx * v[0] + ky * v[1] + kz * v[2]) / k2.clamp_min(1e-12)
    out = torch.empty(n + (3,), dtype=torch.float32, device=_dev())
    for a, ka in enumerate((kx, ky, kz)):
        out[..., a] = torch.fft.irfftn(v[a] - ka * div, s=n)
        v[a] = None
    rms = math.sqrt((out.double() ** 2).sum().item() / (n[0] * n[1] * n[2]))
    return out.mul_(brms / rms)


def _brms(case):
    return 1 * MUG if case.get("prop") == "SDE" else 1 * NG


def _planewave(case, seed):
    """Mode table as PlaneWaveTurbulence draws it: logarithmic k, isotropic directions, random polarisations."""
    rng = np.random.default_rng([seed, 29])
    nm = case["nm"]
    kmin, kmax = 2 * math.pi / case["lmax"], 2 * math.pi / case["lmin"]
    k = kmin * (kmax / kmin) ** (np.arange(nm) / (nm - 1))
    ak = k ** (-5 / 3.) * k
    ak = np.sqrt(2 * ak / ak.sum()) * case["brms"]
    ph, ct = rng.uniform(-math.pi, math.pi, nm), rng.uniform(-1, 1, nm)
    st = np.sqrt(1 - ct * ct)
    al, beta = rng.uniform(0, 2 * math.pi, nm), rng.uniform(0, 2 * math.pi, nm)
    kappa = np.stack([st * np.cos(ph), st * np.sin(ph), ct], 1)
    xi = np.stack([ct * np.cos(ph) * np.cos(al) + np.sin(ph) * np.sin(al),
                   ct * np.sin(ph) * np.cos(al) - np.cos(ph) * np.sin(al), -st * np.cos(al)], 1)
    return dict(k=k, Ak=ak, xi=xi, kappa=kappa, beta=beta)


def _particles(case, seed):
    """Start positions [m], unit directions, energies [J] and charges [C]."""
    rng = np.random.default_rng([seed, 31])
    n = case["n"]
    E = case["emin"] * (case["emax"] / case["emin"]) ** rng.random(n) * EEV
    d = rng.normal(size=(n, 3))
    d /= np.sqrt((d * d).sum(1))[:, None]
    if case["kind"] == "run" and case["nuclei"] == 1:
        z = rng.choice([1., 2., 7., 14., 26.], size=n, p=[0.5, 0.2, 0.15, 0.1, 0.05])
    else:
        z = np.full(n, -1.0 if case.get("nuclei") == -1 else 1.0)
    field = case.get("field", "grid")
    if field == "jf12":
        pos = np.tile([-8.5 * KPC, 0.0, 0.0], (n, 1))
    elif field == "planewave":
        pos = np.zeros((n, 3))
    else:
        pos = np.tile([0.5 * case[a] * case["spacing"] for a in ("nx", "ny", "nz")], (n, 1))
    return pos, d, E, z * EPLUS


def _positions(case, seed):
    """Points along a line through the box and a little beyond it."""
    rng = np.random.default_rng([seed, 37])
    L = np.array([case[a] * case["spacing"] for a in ("nx", "ny", "nz")])
    a, b = rng.uniform(-0.3, 1.3, 3) * L, rng.uniform(-0.3, 1.3, 3) * L
    t = np.linspace(0, 1, case["n"])[:, None]
    return a * (1 - t) + b * t


def _field(case, seed):
    """The device field and the data it was made from."""
    if case["field"] == "planewave":
        m = _planewave(case, seed)
        return capi.Field.planewave(m["k"], m["Ak"], m["xi"], m["kappa"], m["beta"]), m
    if case["field"] == "jf12":
        rng = np.random.default_rng([seed, 41])
        striated = (2 * rng.integers(0, 2, (100, 100, 100)) - 1).astype(np.float32)
        turb = _grid(dict(nx=256, ny=256, nz=256), seed, 1.0).cpu().numpy()
        return capi.Field.jf12(striated=striated, striated_spacing=0.1 * KPC, turbulent=turb,
                               turbulent_spacing=4 * PC), None
    g = _grid(case, seed, _brms(case))
    torch.cuda.synchronize()
    f = capi.Field.grid3f_device(g.data_ptr(), tuple(g.shape[:3]), [0, 0, 0], [case["spacing"]] * 3,
                                 reflective=bool(case.get("reflective")), keep=g)
    if case.get("interpolation"):
        f.set_interpolation(case["interpolation"])
    if case.get("storage") == "fp16":
        f.set_storage("fp16")
    return f, g


def _snapshot_times(case):
    return [case["max_length"] * (i + 1) / (case["snapshots"] + 1) for i in range(case["snapshots"])]


def prepare(case, seed):
    if case["kind"] == "adjoint":
        _, d, E, _ = _particles(case, seed)
        pos = np.tile([0.5 * case[a] * case["spacing"] for a in ("nx", "ny", "nz")], (case["n"], 1))
        t = np.random.default_rng([seed, 43]).normal(size=d.shape)
        t /= np.sqrt((t * t).sum(1))[:, None]
        dev = _dev()
        return dict(case=case, grid=_grid(case, seed, 1 * NG).requires_grad_(True), x0=torch.tensor(pos, device=dev),
                    u0=torch.tensor(d, device=dev, requires_grad=True), E=torch.tensor(E, device=dev),
                    target=torch.tensor(t, device=dev),
                    scale=torch.tensor(1.0, dtype=torch.float64, device=dev, requires_grad=True))
    field, _ = _field(case, seed)
    mixed = capi.PRECISION_MIXED if case["precision"] == "mixed" else capi.PRECISION_FP64
    if case["kind"] == "eval":
        return dict(case=case, field=field, pos=_positions(case, seed), precision=mixed)
    kw = dict(max_length=case.get("max_length", 0.0), precision=mixed)
    if case["prop"] == "SDE":
        kw.update(epsilon=0.1, alpha=1 / 3., scale=1.0, seed=seed + 11)
    prop = capi.Propagator(case["prop"], field, case.get("tol", 0.42 if case["prop"] == "BP" else 1e-4),
                           case["min_step"], case["max_step"], **kw)
    if case.get("snapshots"):
        prop.set_observer(_snapshot_times(case))
    pos, d, E, q = _particles(case, seed)
    if case.get("sphere"):
        prop.set_spherical_boundary(pos[0], case["sphere"])
    init, work_ = capi.Batch(case["n"]), capi.Batch(case["n"])
    init.upload(pos, d, E, q)
    return dict(case=case, field=field, prop=prop, init=init, work=work_)


# ---------------------------------------------------------------------------- one pass


def run(state):
    case = state["case"]
    if case["kind"] == "eval":
        return state["field"].eval(state["pos"], state["precision"])
    if case["kind"] == "adjoint":
        from crpropa3_amd.adjoint import boris_grid_propagate
        grid, u0, scale = state["grid"], state["u0"], state["scale"]
        grid.grad = u0.grad = scale.grad = None
        x, u = boris_grid_propagate(grid, state["x0"], u0, state["E"], EPLUS, [0, 0, 0], [case["spacing"]] * 3,
                                    case["step"], case["steps"], case["checkpoint"], scale=scale)
        loss = ((u - state["target"]) ** 2).sum()
        loss.backward()
        return dict(x=x.detach(), u=u.detach(), loss=loss.detach(), grid_grad=grid.grad, u0_grad=u0.grad,
                    scale_grad=scale.grad)
    state["work"].copy_from(state["init"])
    st = state["prop"].propagate(state["work"], max_steps=case.get("steps", -1))
    out = state["work"].download()
    if case["precision"] == "fp64":  # step counts of adaptive mixed runs follow their rounding
        out["accepted_steps"] = int(st.accepted_steps)
        out["rejected_trials"] = int(st.rejected_trials)
        out["finished"] = int(st.finished)
    if case.get("snapshots"):
        out["detections"] = np.nan_to_num(state["work"].detections(case["snapshots"]), nan=-1.0)
    return out


# ---------------------------------------------------------------------------- what a pass needs


def _process_calls(case):
    """Steps of one particle: the budget, or the length limit over the mean step that these fields give."""
    if case.get("steps"):
        return case["steps"]
    mean = dict(CK=60 * KPC, BP=40 * KPC, SDE=4.2 * PC)[case["prop"]]
    return case["max_length"] / min(mean, case["max_step"])


def work(case):
    """Each input read and each output written once (grid, particles, results); operations of the steps: an
    interpolation, a mode or a model evaluation, and the push or the six stages around it."""
    grid = 12.0 * case["nx"] * case["ny"] * case["nz"] if "nx" in case else 0.0
    n = case["n"]
    if case["kind"] == "eval":
        return dict(bytes=48.0 * n + min(grid, 96.0 * n), flops=150.0 * n)
    if case["kind"] == "adjoint":
        # forward and reverse step; the grid, its gradient, states and their gradients
        return dict(bytes=2 * grid + 8.0 * n * 20, flops=float(n) * case["steps"] * (230 + 600))
    field_flops = {"grid": 150.0, "planewave": 0.0, "jf12": 700.0 + 128 * 3 * 12 / 256.}[case["field"]]
    if case.get("interpolation") == "TRICUBIC":
        field_flops = 21 * 3 * 17.0
    if case["field"] == "planewave":
        field_flops = case["nm"] * (16 + 20.0)
    if case["field"] == "jf12":
        grid = 12.0 * 256 ** 3 + 4e6
    evals = dict(BP=1 if case["min_step"] == case["max_step"] else 3, CK=6, SDE=13.3)[case["prop"]]
    step = dict(BP=80.0, CK=250.0, SDE=400.0)[case["prop"]]
    calls = float(n) * _process_calls(case)
    out = (18 * 8 + 12 + case.get("snapshots", 0) * 72) * n
    return dict(bytes=grid + 18.0 * 8 * n + out, flops=calls * (evals * field_flops + step))


def tolerance(case):
    """The FP64 path reproduces the reference's operations bit for bit, and so do two builds of it.

    The other bounds are about four times the largest relative difference measured against exact() and against
    the same run from directions changed in their last bit (FP32's on the mixed path, FP64's for the adjoint):
    6e-8 for a mixed field value, 1.4e-7 and 1.8e-6 for mixed Boris runs in grids and in plane waves, 2.6e-3 for
    the last step sizes of mixed adaptive runs (a trial accepted on one side and repeated on the other), 4e-8 for
    gradients stored in FP32 and 1e-8 per rounding for those that 4096 steps amplify."""
    if case["kind"] == "adjoint":
        return dict(rel=2e-6)
    if case["precision"] == "fp64":
        return "exact"
    if case["kind"] == "eval":
        return dict(rel=3e-7)
    if case["prop"] == "CK":
        return dict(rel=1e-2)
    return dict(rel=1e-5 if case["field"] == "planewave" else 1e-6)


# ---------------------------------------------------------------------------- the same in plain torch, 64 bits


def _wrap(r, n, reflective):
    if reflective:
        p = 2 * n
        m = torch.remainder(r + 0.5, p) - 0.5
        r = torch.where(m > n - 0.5, p - 1 - m, m)
        lo = torch.floor(r)
        f = r - lo
        hi = torch.clamp(lo + 1, max=n - 1)
        lo = torch.clamp(lo, min=0)
        hi = torch.where(r < 0, torch.zeros_like(hi), hi)
        return lo.long(), hi.long(), f
    lo = torch.floor(r)
    f = r - lo
    i = torch.remainder(lo, n).long()
    return i, torch.remainder(i + 1, n), f


def _trilinear(g, spacing, reflective, p):
    n = g.shape[:3]
    w = [_wrap(p[:, a] / spacing - 0.5, n[a], reflective) for a in range(3)]
    b = 0.0
    for cx in (0, 1):
        for cy in (0, 1):
            for cz in (0, 1):
                wt = 1.0
                for c, (_, _, f) in zip((cx, cy, cz), w):
                    wt = wt * (f if c else 1 - f)
                b = b + g[w[0][cx], w[1][cy], w[2][cz]].double() * wt[:, None]
    return b


def _tricubic(g, spacing, reflective, p):
    n = g.shape[:3]
    idx, wts = [], []
    for a in range(3):
        r = p[:, a] / spacing - 0.5
        lo = torch.floor(r)
        t = r - lo
        ia = []
        for d in (-1, 0, 1, 2):
            j = lo.long() + d
            if reflective:
                j = torch.remainder(j, 2 * n[a])
                j = torch.where(j < n[a], j, 2 * n[a] - 1 - j)
            else:
                j = torch.remainder(j, n[a])
            ia.append(j)
        idx.append(ia)
        t2, t3 = t * t, t * t * t
        wts.append([-0.5 * t + t2 - 0.5 * t3, 1 - 2.5 * t2 + 1.5 * t3, 0.5 * t + 2 * t2 - 1.5 * t3,
                    -0.5 * t2 + 0.5 * t3])
    b = 0.0
    for x in range(4):
        for y in range(4):
            for z in range(4):
                wt = wts[0][x] * wts[1][y] * wts[2][z]
                b = b + g[idx[0][x], idx[1][y], idx[2][z]].double() * wt[:, None]
    return b


def _exact_field(case, data):
    if case["field"] == "planewave":
        t = {k: torch.tensor(v, device=_dev()) for k, v in data.items()}
        kv, a = t["k"][:, None] * t["kappa"], t["Ak"][:, None] * t["xi"]

        def pw(p):
            return torch.cat([torch.cos(q @ kv.T + t["beta"]) @ a for q in p.split(1 << 17)])
        return pw
    fn = _tricubic if case.get("interpolation") == "TRICUBIC" else _trilinear
    return lambda p: fn(data, case["spacing"], bool(case.get("reflective")), p)


def _unit(v):
    return v / v.norm(dim=1, keepdim=True)


def _boris(field, x, u, h, q, E):
    """One Boris step of length h [n]: half drift, rotation by the field there, half drift."""
    x1 = x + u * (h / 2)[:, None]
    t = field(x1) * (q * C_LIGHT * h / (2 * E))[:, None]
    s = t * (2 / (1 + (t * t).sum(1)))[:, None]
    v = u + torch.linalg.cross(u, t)
    w = u + torch.linalg.cross(v, s)
    return x1 + w * (h / 2)[:, None], w


_CK_A = [[], [1 / 5], [3 / 40, 9 / 40], [3 / 10, -9 / 10, 6 / 5], [-11 / 54, 5 / 2, -70 / 27, 35 / 27],
         [1631 / 55296, 175 / 512, 575 / 13824, 44275 / 110592, 253 / 4096]]
_CK_B = [37 / 378, 0, 250 / 621, 125 / 594, 0, 512 / 1771]
_CK_S = [2825 / 27648, 0, 18575 / 48384, 13525 / 55296, 277 / 14336, 1 / 4]


def _cash_karp(field, x, u, h, q, E):
    """One Cash-Karp step of length h [n]: the new state and the norm of the direction's error."""
    kx, ku = [], []
    for row in _CK_A:
        xs, us = x, u
        for a, bx, bu in zip(row, kx, ku):
            xs, us = xs + bx * (a * h)[:, None], us + bu * (a * h)[:, None]
        n = _unit(us)
        kx.append(n)
        ku.append(torch.linalg.cross(n, field(xs)) * (q * C_LIGHT / E)[:, None])
    e = 0.0
    xo, uo = x, u
    for b, s, bx, bu in zip(_CK_B, _CK_S, kx, ku):
        xo, uo = xo + bx * (b * h)[:, None], uo + bu * (b * h)[:, None]
        e = e + bu * ((b - s) * h)[:, None]
    return xo, uo, e.norm(dim=1)


def _exact_run(case, seed):
    field = _exact_field(case, _planewave(case, seed) if case["field"] == "planewave"
                         else _grid(case, seed, _brms(case)))
    pos, d, E_, q_ = (torch.tensor(a, device=_dev()) for a in _particles(case, seed))
    n, ck = case["n"], case["prop"] == "CK"
    lo, hi, tol = case["min_step"], case["max_step"], case.get("tol", 1e-4)
    x, u, E, q = pos.clone(), d.clone(), E_, q_
    nxt = torch.zeros(n, dtype=torch.float64, device=_dev())
    cur, length, px, pu = nxt.clone(), nxt.clone(), x.clone(), u.clone()
    for _ in range(case["steps"]):
        px, pu = x, u
        h = torch.clamp(nxt, lo, hi)
        if lo == hi:
            if ck:
                x, u, _ = _cash_karp(field, x, u, h, q, E)
            else:
                x, u = _boris(field, x, u, h, q, E)
            nxt = h
        else:
            todo = torch.arange(n, device=_dev())
            x, u, nxt, cur = px.clone(), pu.clone(), h.clone(), h.clone()
            while len(todo):
                ht = h[todo]
                xo, uo, err = _cash_karp(field, px[todo], pu[todo], ht, q[todo], E[todo])
                r = err / tol
                new = 0.95 * ht * r.clamp_min(1e-300) ** -0.2
                shrink = torch.clamp(torch.maximum(new, 0.1 * ht), min=lo)
                grow = torch.where(ht == hi, ht, torch.clamp(torch.minimum(new, 5 * ht), max=hi))
                ok = (r <= 1) | (ht == lo)
                w = todo[ok]
                x[w], u[w], cur[w] = xo[ok], uo[ok], ht[ok]
                nxt[w] = torch.where(r[ok] <= 1, grow[ok], ht[ok])
                h[todo[~ok]] = shrink[~ok]
                todo = todo[~ok]
            h = cur
        cur = h
        u = _unit(u)
        length = length + h
    out = dict(pos=x, dir=u, energy=E, charge=q, current_step=cur, next_step=nxt, trajectory_length=length,
               time=length / C_LIGHT, prev_pos=px, prev_dir=pu, source_pos=pos, created_pos=pos)
    out = {k: v.cpu().numpy() for k, v in out.items()}
    out.update(active=np.ones(n, dtype=np.int32), detection_index=np.zeros(n, dtype=np.int32),
               sde_step=np.zeros(n, dtype=np.uint32))
    if case["precision"] == "fp64":
        out.update(accepted_steps=n * case["steps"], rejected_trials=None, finished=0)
    return out


def _exact_adjoint(case, seed):
    s = prepare(case, seed)
    grid = s["grid"].detach().double().requires_grad_(True)
    u0, scale, n, K = s["u0"].detach(), torch.tensor(1.0, dtype=torch.float64, device=_dev()), case["n"], 16
    h = torch.full((n,), case["step"], dtype=torch.float64, device=_dev())
    q = torch.full((n,), EPLUS, dtype=torch.float64, device=_dev())

    def segment(g, sc, x, u, steps):
        for _ in range(steps):
            x, u = _boris(lambda p: _trilinear(g, case["spacing"], False, p) * sc, x, u, h, q, s["E"])
            u = _unit(u)
        return x, u

    states = [(s["x0"], u0)]
    counts = [min(K, case["steps"] - i) for i in range(0, case["steps"], K)]
    with torch.no_grad():
        for c in counts:
            states.append(segment(grid, scale, *states[-1], c))
    x, u = states[-1]
    loss = ((u - s["target"]) ** 2).sum()
    ax, au = torch.zeros_like(x), 2 * (u - s["target"])
    gg, gs = torch.zeros_like(grid), torch.zeros_like(scale)
    for (xs, us), c in zip(reversed(states[:-1]), reversed(counts)):
        leaf = [grid, scale.clone().requires_grad_(True), xs.clone().requires_grad_(True),
                us.clone().requires_grad_(True)]
        xo, uo = segment(*leaf, c)
        g = torch.autograd.grad([xo, uo], leaf, [ax, au])
        gg, gs, ax, au = gg + g[0], gs + g[1], g[2], g[3]
    return dict(x=x, u=u, loss=loss, grid_grad=gg, u0_grad=au, scale_grad=gs)


def exact(case, seed):
    """What run returns, in 64 bits and plain torch.  None for the Galactic model, stochastic transport and
    runs to a length limit (thousands of masked trials) and for the long adjoint: each takes longer than 20 s
    that way; and for grid runs over more than 30 Mpc, where the low-energy particles have turned around so
    often that a difference of the last FP32 bit in the interpolation has grown to the size of the result."""
    if case["kind"] == "eval":
        g = _grid(case, seed, _brms(case))
        return _exact_field(case, g)(torch.tensor(_positions(case, seed), device=_dev())).cpu().numpy()
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, seed) if case["steps"] <= 512 else None
    if case["prop"] == "SDE" or case["field"] == "jf12" or case.get("max_length"):
        return None
    if case["field"] == "planewave" and float(case["n"]) * case["nm"] * case["steps"] > 2.2e11:
        return None
    if case["field"] == "grid" and case["steps"] * case["max_step"] > 30 * MPC:
        return None
    return _exact_run(case, seed)
