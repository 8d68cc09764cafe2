"""Adjoint of the Boris push through a periodic grid (crp_adjoint_*), behind
torch.autograd: checked against the oracle's FP64 CPU reference gradient (an
independent implementation that tapes every state instead of checkpointing,
itself pinned by finite differences) and against central finite differences
of the GPU forward pass."""
import numpy as np
import pytest

import oracle_ctypes as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def setup(n=64, N=16, nsteps=300, K=32, seed=3):
    from crpropa3_amd.turbulence import simple_grid_turbulence
    sp = 20 * O.kpc
    grid = simple_grid_turbulence(N, sp, 1 * O.nG, 2 * sp, N * sp, seed).astype(np.float32)
    rng = np.random.default_rng(seed)
    _, E, d = O.sample_particles(seed + 1, n, 1 * O.EeV, 100 * O.EeV)
    u0 = O.normalise(d)
    x0 = rng.uniform(0, N * sp, size=(n, 3))
    target = O.normalise(rng.normal(size=(n, 3)))
    wx = rng.normal(size=(n, 3)) / (N * sp)
    h = 10 * O.kpc
    kq = O.eplus * O.c_light * h / (2 * E)
    return dict(grid=grid, sp=sp, x0=x0, u0=u0, E=E, kq=kq, target=target, wx=wx, h=h, nsteps=nsteps, K=K, N=N)


def oracle_grad(s, scale=1.0):
    o, sp = np.zeros(3), np.full(3, s["sp"])
    xo, uo = O.adjoint_forward(s["grid"], o, sp, scale, s["h"], s["nsteps"], s["x0"], s["u0"], s["kq"])
    gg, gx0, gu0, gs = O.adjoint_backward(s["grid"], o, sp, scale, s["h"], s["nsteps"], s["x0"], s["u0"], s["kq"],
                                          s["wx"], 2 * (uo - s["target"]))
    loss = np.sum((uo - s["target"]) ** 2) + np.sum(s["wx"] * xo)
    return loss, xo, uo, gg, gx0, gu0, gs


def gpu_run(s, scale=1.0, grad=True, grid=None, u0=None):
    from crpropa3_amd.adjoint import boris_grid_propagate
    dev = torch.device("cuda:0")
    g = torch.tensor(s["grid"] if grid is None else grid, dtype=torch.float32, device=dev, requires_grad=grad)
    x0 = torch.tensor(s["x0"], dtype=torch.float64, device=dev, requires_grad=grad)
    u0 = torch.tensor(s["u0"] if u0 is None else u0, dtype=torch.float64, device=dev, requires_grad=grad)
    sc = torch.tensor(scale, dtype=torch.float64, device=dev, requires_grad=grad)
    tgt = torch.tensor(s["target"], dtype=torch.float64, device=dev)
    wx = torch.tensor(s["wx"], dtype=torch.float64, device=dev)
    with torch.set_grad_enabled(grad):
        xo, uo = boris_grid_propagate(g, x0, u0, torch.tensor(s["E"], device=dev), O.eplus, [0, 0, 0],
                                      [s["sp"]] * 3, s["h"], s["nsteps"], s["K"], scale=sc)
        loss = ((uo - tgt) ** 2).sum() + (wx * xo).sum()
    if not grad:
        return loss.item()
    loss.backward()
    torch.cuda.synchronize()
    return (loss.item(), xo.detach().cpu().numpy(), uo.detach().cpu().numpy(), g.grad.double().cpu().numpy(),
            x0.grad.cpu().numpy(), u0.grad.cpu().numpy(), sc.grad.item())


def test_adjoint_forward_and_gradients_match_cpu_reference():
    s = setup()
    ref = oracle_grad(s)
    got = gpu_run(s)
    print("loss %.6e, forward max |dx| %.2e m, grid-gradient max rel %.2e" % (
        got[0], np.abs(got[1] - ref[1]).max(), np.abs(got[3] - ref[3]).max() / np.abs(ref[3]).max()))
    # the GPU divides by multiplying with reciprocals: agreement to rounding, not bit-exact
    assert got[0] == pytest.approx(ref[0], rel=1e-10)
    assert np.allclose(got[1], ref[1], rtol=1e-10, atol=0)
    assert np.allclose(got[2], ref[2], rtol=0, atol=1e-10)
    # the grid gradient comes back in the grid's dtype (float32)
    assert np.max(np.abs(got[3] - ref[3])) < 1e-6 * np.abs(ref[3]).max()
    assert np.allclose(got[4], ref[4], rtol=1e-7, atol=1e-8 * np.abs(ref[4]).max())
    assert np.allclose(got[5], ref[5], rtol=1e-7, atol=1e-8 * np.abs(ref[5]).max())
    assert got[6] == pytest.approx(ref[6], rel=1e-8)


def test_adjoint_partial_segment_and_no_position_adjoint():
    """nsteps not a multiple of K; loss on directions only (no adjoint of x_final)."""
    from crpropa3_amd.adjoint import boris_grid_propagate
    s = setup(n=100, nsteps=77, K=10)
    o, sp = np.zeros(3), np.full(3, s["sp"])
    xo, uo = O.adjoint_forward(s["grid"], o, sp, 1.0, s["h"], s["nsteps"], s["x0"], s["u0"], s["kq"])
    gg, gx0, gu0, gs = O.adjoint_backward(s["grid"], o, sp, 1.0, s["h"], s["nsteps"], s["x0"], s["u0"], s["kq"],
                                          None, 2 * (uo - s["target"]))
    dev = torch.device("cuda:0")
    g = torch.tensor(s["grid"], device=dev, requires_grad=True)
    u0 = torch.tensor(s["u0"], device=dev, requires_grad=True)
    x0 = torch.tensor(s["x0"], device=dev)
    _, ug = boris_grid_propagate(g, x0, u0, torch.tensor(s["E"], device=dev), O.eplus, [0, 0, 0], [s["sp"]] * 3,
                                 s["h"], s["nsteps"], s["K"])
    ((ug - torch.tensor(s["target"], device=dev)) ** 2).sum().backward()
    assert np.max(np.abs(g.grad.double().cpu().numpy() - gg)) < 1e-6 * np.abs(gg).max()
    assert np.allclose(u0.grad.cpu().numpy(), gu0, rtol=1e-7, atol=1e-8 * np.abs(gu0).max())


def test_adjoint_matches_finite_differences_of_gpu_forward():
    """Central differences of the GPU forward on 256 grid values, 12 initial directions and the scale."""
    s = setup(n=48, nsteps=200, K=16)
    got = gpu_run(s)
    rng = np.random.default_rng(11)
    flat = s["grid"].reshape(-1)
    order = np.argsort(-np.abs(got[3].reshape(-1)))
    picks = np.concatenate([order[:192], rng.choice(order[:2000], 64, replace=False)])
    # central differences converge as e^2: at 1e-3 of the largest value the truncation error is ~3e-3 of
    # the largest gradient, at 1e-5 it is ~3e-8 (measured on the oracle)
    e = np.float32(1e-5) * np.abs(flat).max()
    fd = []
    for j in picks:
        gp = flat.copy()
        gm = flat.copy()
        gp[j] = np.float32(flat[j] + e)
        gm[j] = np.float32(flat[j] - e)
        lp = gpu_run(s, grad=False, grid=gp.reshape(s["grid"].shape))
        lm = gpu_run(s, grad=False, grid=gm.reshape(s["grid"].shape))
        fd.append((lp - lm) / (float(gp[j]) - float(gm[j])))
    fd = np.array(fd)
    ad = got[3].reshape(-1)[picks]
    err = np.abs(ad - fd) / np.abs(got[3]).max()
    big = np.abs(fd) > 1e-2 * np.abs(fd).max()
    rel = np.abs(ad[big] - fd[big]) / np.abs(fd[big])
    print("grid FD: %d values, max err %.2e of the largest gradient; %d large ones: max rel err %.2e"
          % (len(picks), err.max(), big.sum(), rel.max()))
    assert err.max() < 1e-6
    assert rel.max() < 1e-4
    # steps measured on the oracle for this grid: a direction step of 1e-6 leaves a truncation error of
    # 4e-4 relative (the 300-step trajectories are strongly curved), 1e-7 of 1e-7; for the scale,
    # 1e-5 gives 0.16 and 1e-6 gives 7e-9
    for i in range(12):
        for a in range(3):
            d = 1e-7
            up = s["u0"].copy()
            um = s["u0"].copy()
            up[i, a] += d
            um[i, a] -= d
            fdv = (gpu_run(s, grad=False, u0=up) - gpu_run(s, grad=False, u0=um)) / (2 * d)
            assert got[5][i, a] == pytest.approx(fdv, rel=1e-5, abs=1e-6 * np.abs(got[5]).max())
    d = 1e-6
    fds = (gpu_run(s, 1 + d, grad=False) - gpu_run(s, 1 - d, grad=False)) / (2 * d)
    assert got[6] == pytest.approx(fds, rel=1e-6)


def test_adjoint_checkpoint_interval_does_not_change_results():
    s = setup(n=32, nsteps=100, K=7)
    a = gpu_run(s)
    s["K"] = 100
    b = gpu_run(s)
    s["K"] = 1
    c = gpu_run(s)
    assert np.array_equal(a[2], b[2]) and np.array_equal(a[2], c[2])
    for r in (a, c):
        assert np.allclose(r[3], b[3], rtol=1e-6, atol=1e-6 * np.abs(b[3]).max())
        assert np.array_equal(r[5], b[5])


def test_adjoint_rejects_bad_input():
    from crpropa3_amd import capi
    from crpropa3_amd.adjoint import boris_grid_propagate
    s = setup(n=4, nsteps=10, K=4)
    dev = torch.device("cuda:0")
    g = torch.tensor(s["grid"], device=dev)
    x0 = torch.tensor(s["x0"], device=dev)
    u0 = torch.tensor(s["u0"], device=dev)
    with pytest.raises(capi.CrpError):
        boris_grid_propagate(g, x0, u0, 1 * O.EeV, O.eplus, [0, 0, 0], [s["sp"]] * 3, s["h"], 10, 0)
    with pytest.raises(ValueError):
        boris_grid_propagate(g.double(), x0, u0, 1 * O.EeV, O.eplus, [0, 0, 0], [s["sp"]] * 3, s["h"], 10, 4)


@pytest.mark.parametrize("budget,shift", [(None, None), ("3e4", None), ("0", None), (None, "4"), ("3e4", "4")])
def test_adjoint_backward_paths(budget, shift, monkeypatch):
    """The backward's three schedules against the oracle on a 20^3 grid (tiles cut by the grid's end):
    the default blocks (17 segments of 8 steps in 6 blocks of at most 3, each recomputed in runs of 8
    steps from sub-checkpoints), one segment per block with the adjoint carried between 17 blocks (a
    small per-block budget), and per-step atomics (budget 0); the blocked ones with 8^3-cell tiles and
    with the 16^3-cell tiles of large grids.  (One block in all: nsteps = K in
    test_adjoint_checkpoint_interval_does_not_change_results.)"""
    if budget is not None:
        monkeypatch.setenv("CRP_ADJOINT_BLOCK_BYTES", budget)
    if shift is not None:
        monkeypatch.setenv("CRP_ADJOINT_TILE_SHIFT", shift)
    s = setup(n=96, N=20, nsteps=130, K=8, seed=9)
    ref = oracle_grad(s)
    got = gpu_run(s)
    rel = np.abs(got[3] - ref[3]).max() / np.abs(ref[3]).max()
    print("budget %s, tile shift %s: grid-gradient max rel %.2e" % (budget, shift, rel))
    assert rel < 1e-6
    assert np.allclose(got[4], ref[4], rtol=1e-7, atol=1e-8 * np.abs(ref[4]).max())
    assert np.allclose(got[5], ref[5], rtol=1e-7, atol=1e-8 * np.abs(ref[5]).max())
    assert got[6] == pytest.approx(ref[6], rel=1e-8)


def test_adjoint_several_particle_groups():
    """600 particles: two full groups of 256 and a partial third one (their tile counts, offsets and
    carried adjoints kept apart), 9 segments of 13 steps (the last of 7) in 5 blocks: runs of 8, 8, 8
    and 2 steps that cross the segments' ends, and one run of 7 in the last block; against the oracle."""
    s = setup(n=600, N=16, nsteps=111, K=13, seed=21)
    ref = oracle_grad(s)
    got = gpu_run(s)
    rel = np.abs(got[3] - ref[3]).max() / np.abs(ref[3]).max()
    print("600 particles: grid-gradient max rel %.2e" % rel)
    assert rel < 1e-6
    assert np.allclose(got[4], ref[4], rtol=1e-7, atol=1e-8 * np.abs(ref[4]).max())
    assert np.allclose(got[5], ref[5], rtol=1e-7, atol=1e-8 * np.abs(ref[5]).max())
    assert got[6] == pytest.approx(ref[6], rel=1e-8)


def test_adjoint_large_grid_uses_16_cell_tiles():
    """A 176^3 grid has 10648 tiles of 8^3 cells, more than the blocked backward takes: it runs with
    16^3-cell tiles (1331) and matches the oracle."""
    s = setup(n=64, N=176, nsteps=60, K=8, seed=12)
    ref = oracle_grad(s)
    got = gpu_run(s)
    rel = np.abs(got[3] - ref[3]).max() / np.abs(ref[3]).max()
    print("176^3: grid-gradient max rel %.2e" % rel)
    assert rel < 1e-6
    assert np.allclose(got[5], ref[5], rtol=1e-7, atol=1e-8 * np.abs(ref[5]).max())
    assert got[6] == pytest.approx(ref[6], rel=1e-8)


@pytest.mark.parametrize("n,nsteps,K,budget", [(1, 1, 1, None), (256, 64, 8, None), (257, 111, 13, None), (600, 111, 13, None),
                                               (600, 111, 13, "4e5"), (257, 111, 13, "1.5e5")])
def test_adjoint_kept_and_recomputed_sub_checkpoints(n, nsteps, K, budget, monkeypatch):
    """The forward keeps the blocks' sub-checkpoints and tile counts where they fit the buffer budget;
    beyond it (4e5 bytes where the states of 600 particles take 5.2e5; 1.5e5 of 2.2e5) the backward
    recomputes them.  Both against the oracle at full and partial particle groups, with segments that are no
    multiple of the 8 steps of a run, and down to one step; a second backward of the same graph finds what the
    forward left unchanged, so it gives the gradients of the first (those of the grid up to the order of the
    FP64 sums)."""
    from crpropa3_amd.adjoint import boris_grid_propagate
    if budget is not None:
        monkeypatch.setenv("CRP_ADJOINT_BLOCK_BYTES", budget)
    s = setup(n=n, N=16, nsteps=nsteps, K=K, seed=31)
    ref = oracle_grad(s)
    dev = torch.device("cuda:0")
    g = torch.tensor(s["grid"], dtype=torch.float32, device=dev, requires_grad=True)
    x0 = torch.tensor(s["x0"], device=dev, requires_grad=True)
    u0 = torch.tensor(s["u0"], device=dev, requires_grad=True)
    sc = torch.tensor(1.0, dtype=torch.float64, device=dev, requires_grad=True)
    xo, uo = boris_grid_propagate(g, x0, u0, torch.tensor(s["E"], device=dev), O.eplus, [0, 0, 0], [s["sp"]] * 3,
                                  s["h"], s["nsteps"], s["K"], scale=sc)
    loss = ((uo - torch.tensor(s["target"], device=dev)) ** 2).sum() + (torch.tensor(s["wx"], device=dev) * xo).sum()
    one = [t.double().cpu().numpy() for t in torch.autograd.grad(loss, (g, x0, u0, sc), retain_graph=True)]
    two = [t.double().cpu().numpy() for t in torch.autograd.grad(loss, (g, x0, u0, sc))]
    assert np.allclose(one[0], ref[3], rtol=0, atol=1e-6 * np.abs(ref[3]).max())
    for a, b in ((one[1], ref[4]), (one[2], ref[5])):
        assert np.allclose(a, b, rtol=1e-7, atol=1e-8 * np.abs(b).max())
    assert float(one[3]) == pytest.approx(ref[6], rel=1e-8)
    assert np.array_equal(one[1], two[1]) and np.array_equal(one[2], two[2])
    # the grid gradient is rounded to float32 after the FP64 sums: at most an ulp apart
    assert np.allclose(one[0], two[0], rtol=2.0 ** -23, atol=1e-12 * np.abs(one[0]).max())


@pytest.mark.parametrize("before,after", [({}, dict(CRP_ADJOINT_BLOCK_BYTES="0")),
                                          ({}, dict(CRP_ADJOINT_BLOCK_BYTES="3e4")),
                                          ({}, dict(CRP_ADJOINT_TILE_SHIFT="4")),
                                          (dict(CRP_ADJOINT_BLOCK_BYTES="4e5"), {}),
                                          (dict(CRP_ADJOINT_TILE_SHIFT="4"), {})])
def test_adjoint_environment_changes_between_forward_and_backward(before, after, monkeypatch):
    """The buffers' layout is fixed by the forward: another environment at the backward changes nothing."""
    from crpropa3_amd.adjoint import boris_grid_propagate
    s = setup(n=600, N=20, nsteps=111, K=13, seed=41)
    ref = oracle_grad(s)
    dev = torch.device("cuda:0")
    g = torch.tensor(s["grid"], dtype=torch.float32, device=dev, requires_grad=True)
    x0 = torch.tensor(s["x0"], device=dev, requires_grad=True)
    u0 = torch.tensor(s["u0"], device=dev, requires_grad=True)
    for k, v in before.items():
        monkeypatch.setenv(k, v)
    xo, uo = boris_grid_propagate(g, x0, u0, torch.tensor(s["E"], device=dev), O.eplus, [0, 0, 0], [s["sp"]] * 3,
                                  s["h"], s["nsteps"], s["K"])
    for k in before:
        monkeypatch.delenv(k)
    for k, v in after.items():
        monkeypatch.setenv(k, v)
    loss = ((uo - torch.tensor(s["target"], device=dev)) ** 2).sum() + (torch.tensor(s["wx"], device=dev) * xo).sum()
    loss.backward()
    assert np.allclose(g.grad.double().cpu().numpy(), ref[3], rtol=0, atol=1e-6 * np.abs(ref[3]).max())
    for a, b in ((x0.grad, ref[4]), (u0.grad, ref[5])):
        assert np.allclose(a.cpu().numpy(), b, rtol=1e-7, atol=1e-8 * np.abs(b).max())


@pytest.mark.parametrize("factor", [-3.0, 1e6, float("nan")])
def test_adjoint_backward_with_other_charges_stays_in_its_scratch(factor):
    """A backward whose kq is not the forward's finds other tiles than the forward counted: its gradients mean
    nothing, but nothing outside the plan's scratch is written, and the next correct backward is unharmed."""
    import ctypes as C
    from crpropa3_amd import adjoint, capi
    s = setup(n=300, N=32, nsteps=100, K=10, seed=5)
    dev = torch.device("cuda:0")
    L = adjoint._bind()
    g = torch.tensor(s["grid"], device=dev)
    x0, u0, kq, gu = (torch.tensor(s[k], device=dev) for k in ("x0", "u0", "kq", "target"))
    cfg = adjoint._config(g, [0, 0, 0], [s["sp"]] * 3, 1.0, s["h"], s["nsteps"], s["K"])
    plan = adjoint.AdjointPlan()
    capi.check(L.crp_adjoint_plan_make(C.byref(cfg), 300, 1, C.byref(plan)))
    assert plan.keep_states == 1
    ckpt = torch.empty(plan.checkpoint_bytes // 8, dtype=torch.float64, device=dev)
    xo, uo, gx0, gu0 = (torch.empty_like(x0) for _ in range(4))
    size = -(-plan.scratch_bytes // 8)
    guard = 1 << 20
    scratch = torch.full((size + guard,), 7.0, dtype=torch.float64, device=dev)
    gg = torch.zeros(g.numel() + 4096, dtype=torch.float64, device=dev)
    gs = torch.zeros(1, dtype=torch.float64, device=dev)
    p = adjoint._ptr
    capi.check(L.crp_adjoint_forward_planned(C.byref(cfg), 300, C.byref(plan), p(x0), p(u0), p(kq), p(ckpt), p(xo), p(uo),
                                             None))
    kept = ckpt.clone()
    res = []
    for k in (kq, kq * factor, kq):
        gg.zero_()
        capi.check(L.crp_adjoint_backward_planned(C.byref(cfg), 300, C.byref(plan), p(k), p(ckpt), None, p(gu), p(scratch),
                                                  p(gg), p(gx0), p(gu0), p(gs), None))
        torch.cuda.synchronize()
        assert (scratch[size:] == 7.0).all() and (gg[g.numel():] == 0).all()
        assert torch.equal(ckpt.view(torch.int64), kept.view(torch.int64))
        res.append((gx0.clone(), gu0.clone(), gg.clone()))
    assert torch.equal(res[0][0], res[2][0]) and torch.equal(res[0][1], res[2][1])
    assert torch.allclose(res[0][2], res[2][2], rtol=0, atol=1e-12 * float(res[0][2].abs().max()))


def test_adjoint_checkpoint_interval_bounds_memory():
    """What a graph holds until its backward: with keep_states False the states every K steps and the cell table;
    without a backward to come nothing more is written either, and the default keeps 6 bytes a step.  The values
    are the same bits (the grid gradient's FP64 sums in another order, then rounded to float32)."""
    from crpropa3_amd import adjoint
    n, nsteps, K, N = 4096, 256, 64, 16
    s = setup(n=n, N=N, nsteps=nsteps, K=K, seed=51)
    dev = torch.device("cuda:0")
    E, target = torch.tensor(s["E"], device=dev), torch.tensor(s["target"], device=dev)
    g = torch.tensor(s["grid"], dtype=torch.float32, device=dev, requires_grad=True)
    x0 = torch.tensor(s["x0"], device=dev, requires_grad=True)
    u0 = torch.tensor(s["u0"], device=dev, requires_grad=True)
    few, many = 48 * n * (nsteps // K) + 128 * N ** 3, 6 * n * nsteps + 128 * N ** 3
    slack = 48 * n * 3  # x, u, kq and the like

    def run(**kw):
        return adjoint.boris_grid_propagate(g, x0, u0, E, O.eplus, [0, 0, 0], [s["sp"]] * 3, s["h"], nsteps, K, **kw)

    res = {}
    for keep in (None, False, True):
        before = torch.cuda.memory_allocated()
        x, u = run(keep_states=keep)
        held = torch.cuda.memory_allocated() - before
        want = few if keep is False else many
        assert want <= held <= want + slack + 4 * 8 * (n // 256) * 8, (keep, held)
        res[keep] = (x.detach(), u.detach()) + torch.autograd.grad(((u - target) ** 2).sum(), (g, x0, u0))
        del x, u
    for keep in (False, True):
        for a, b in zip(res[None], res[keep]):
            if a.dtype == torch.float64:
                assert torch.equal(a, b)
            else:
                assert torch.allclose(a, b, rtol=2.0 ** -23, atol=1e-12 * float(a.abs().max()))
    with torch.no_grad():
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        x, u = run()
        assert torch.cuda.max_memory_allocated() - before <= few + slack
        assert torch.equal(x, res[None][0]) and torch.equal(u, res[None][1])


def test_adjoint_keeps_no_states_on_a_full_card(monkeypatch):
    """The default keeps the states only where the card has eight times their size free."""
    from crpropa3_amd import adjoint
    dev = torch.device("cuda:0")
    assert adjoint._roomy(1 << 20, dev)
    assert adjoint._roomy(1 << 30, dev)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: (3 << 30, 288 << 30))
    unused = torch.cuda.memory_reserved(dev) - torch.cuda.memory_allocated(dev)
    assert not adjoint._roomy((3 << 30) + unused, dev)
    assert adjoint._roomy(1 << 28, dev)


@pytest.mark.parametrize("before,after", [({}, {}), ({}, dict(CRP_ADJOINT_BLOCK_BYTES="0")),
                                          ({}, dict(CRP_ADJOINT_BLOCK_BYTES="3e4")),
                                          (dict(CRP_ADJOINT_TILE_SHIFT="4"), {})])
def test_adjoint_calls_without_a_plan(before, after, monkeypatch):
    """crp_adjoint_forward and crp_adjoint_backward with checkpoints of the documented size and a scratch sized at
    the backward: the environment may change in between, and nothing past the buffers is written."""
    import ctypes as C
    from crpropa3_amd import adjoint, capi
    n, N, nsteps, K = 300, 20, 111, 13
    s = setup(n=n, N=N, nsteps=nsteps, K=K, seed=61)
    ref = oracle_grad(s)
    dev = torch.device("cuda:0")
    L, p = adjoint._bind(), adjoint._ptr
    g = torch.tensor(s["grid"], device=dev)
    x0, u0, kq, wx = (torch.tensor(s[k], device=dev) for k in ("x0", "u0", "kq", "wx"))
    cfg = adjoint._config(g, [0, 0, 0], [s["sp"]] * 3, 1.0, s["h"], nsteps, K)
    states = (-(-nsteps // K) * 48 * n + 255) // 256 * 32
    size, guard = states + 16 * N ** 3, 4096
    ckpt = torch.full((size + guard,), 7.0, dtype=torch.float64, device=dev)
    xo, uo, gx0, gu0 = (torch.empty_like(x0) for _ in range(4))
    for k, v in before.items():
        monkeypatch.setenv(k, v)
    capi.check(L.crp_adjoint_forward(C.byref(cfg), n, p(x0), p(u0), p(kq), p(ckpt), p(xo), p(uo), None))
    for k in before:
        monkeypatch.delenv(k)
    for k, v in after.items():
        monkeypatch.setenv(k, v)
    sb = C.c_size_t(0)
    capi.check(L.crp_adjoint_workspace(C.byref(cfg), n, None, C.byref(sb)))
    scratch = torch.full((-(-sb.value // 8) + guard,), 7.0, dtype=torch.float64, device=dev)
    gg, gs = torch.zeros(g.numel(), dtype=torch.float64, device=dev), torch.zeros(1, dtype=torch.float64, device=dev)
    gu = 2 * (uo - torch.tensor(s["target"], device=dev))
    capi.check(L.crp_adjoint_backward(C.byref(cfg), n, p(kq), p(ckpt), p(wx), p(gu), p(scratch), p(gg), p(gx0), p(gu0),
                                      p(gs), None))
    torch.cuda.synchronize()
    assert (ckpt[size:] == 7.0).all() and (scratch[-guard:] == 7.0).all()
    assert np.allclose(gg.cpu().numpy().reshape(ref[3].shape), ref[3], rtol=0, atol=1e-6 * np.abs(ref[3]).max())
    for a, b in ((gx0, ref[4]), (gu0, ref[5])):
        assert np.allclose(a.cpu().numpy(), b, rtol=1e-7, atol=1e-8 * np.abs(b).max())
    assert gs.item() == pytest.approx(ref[6], rel=1e-8)
