"""The straight-line forms of the FP64 steps (range tests merged, repeated with the tested form where one
fails), the folded mirror boundary, small batches spread over the GPU, quads of lanes on tricubic grids and the
pinned transfers: bit for bit against the oracle, at the operands and sizes where each can go wrong."""
import numpy as np
import pytest

import oracle_ctypes as O
from crpropa3_amd import capi

pytestmark = pytest.mark.gpu

KPC = 3.0856775814913674e19
EPLUS = 1.602176487e-19
EEV = 1e18 * EPLUS


def same(a, b):
    a = np.ascontiguousarray(a, dtype=np.float64)
    b = np.ascontiguousarray(b, dtype=np.float64)
    return np.array_equal(a.view(np.uint64), b.view(np.uint64))


def noise(shape, seed=3):
    return (np.random.default_rng(seed).normal(size=tuple(shape) + (3,)) * 1e-13).astype(np.float32)


def compare(field, ofield, kind, pos, d, E, q, steps, lo, hi, tol):
    ref = O.OracleState(pos, d, E, q)
    O.propagate(ofield, O.PROP_BP if kind == "BP" else O.PROP_CK, ref, steps, tolerance=tol, min_step=lo, max_step=hi,
                libm=O.LIBM_CR)
    p = capi.Propagator(kind, field, tol, lo, hi)
    b = capi.Batch(len(E))
    b.upload(pos, O.normalise(d), E, q)
    p.propagate(b, max_steps=steps)
    out = b.download()
    for k in ("pos", "dir", "prev_pos", "prev_dir", "current_step", "next_step", "trajectory_length", "time"):
        assert same(out[k], getattr(ref, k)), k
    return out


def special_particles():
    """Directions with zero, negative-zero and tiny components, energies and charges from far below to far above
    the bounds of the straight line, positions at the origin and far away, between ordinary ones."""
    dirs = [(1, 0, 0), (0, -1, 0), (-0.0, 0.0, 1), (1, 1e-170, 0), (1e-300, 1, 1), (1, 2, 3), (3, -2, 1e-160),
            (1e-308, 1e-308, 1)]
    es = [1e-60, 1e-30, 1e-10, 1 * EEV, 1e3 * EEV, 1e40, 1e90]
    qs = [EPLUS, -EPLUS, 26 * EPLUS, 1e-40, 1e30, 0.0]
    ps = [(0, 0, 0), (-0.0, 1e-200, 3e20), (1e21, -2e21, 5e20), (1e28, 1e21, 1e21), (3e19, 3e19, 3e19)]
    rows = [(p, d, e, q) for p in ps for d in dirs for e in es for q in qs]
    P, D, E, Q = (np.array(x, dtype=np.float64) for x in zip(*rows))
    return P, D, E, Q


@pytest.mark.parametrize("reflective", [False, True])
@pytest.mark.parametrize("kind,fixed", [("BP", True), ("BP", False), ("CK", True), ("CK", False)])
def test_extreme_operands(kind, fixed, reflective):
    g = noise((7, 5, 6))
    g[0, 0, 0] = 0.0  # cells with zero, tiny and huge values
    g[1, 1, 1] = (1e-45, -1e-40, 0.0)
    g[3, 2, 2] = (1e30, -1e20, 1e-20)
    P, D, E, Q = special_particles()
    if reflective:  # the reference's mirror loop takes a pass per box length
        keep = np.abs(P).max(axis=1) < 1e25
        P, D, E, Q = P[keep], D[keep], E[keep], Q[keep]
    sp = [2e19, 3e19, 1e19]
    f = capi.Field.grid3f(g, [-1e19, 0, 0], sp, reflective=reflective)
    of = O.OracleField.grid(g, [-1e19, 0, 0], sp, reflective)
    lo, hi = (1e19, 1e19) if fixed else (1e17, 1e20)
    ref = O.OracleState(P, D, E, Q)
    O.propagate(of, O.PROP_BP if kind == "BP" else O.PROP_CK, ref, 3, tolerance=1e-3, min_step=lo, max_step=hi,
                libm=O.LIBM_CR)
    b = capi.Batch(len(E))
    b.upload(P, O.normalise(D), E, Q)
    capi.Propagator(kind, f, 1e-3, lo, hi).propagate(b, max_steps=3)
    out = b.download()
    for k in ("pos", "dir", "current_step", "next_step"):
        a, r = out[k], getattr(ref, k)
        ok = (a.view(np.uint64) == r.view(np.uint64)) | (np.isnan(a) & np.isnan(r))
        assert ok.all(), (k, np.argwhere(~ok)[:4], a[~ok][:4], r[~ok][:4])


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 3, 1), (5, 8, 7), (97, 4, 33)])
def test_mirror_fold(shape):
    """Reflective positions inside, on and around the mirrors, up to 3000 boxes away."""
    rng = np.random.default_rng(7)
    g = noise(shape)
    sp, o = 1.5, [0.25, -3.0, 7.0]
    n = np.array(shape)
    half = rng.integers(-40, 40, (4000, 3)) * 0.5 * n + rng.choice([0, 0.5, -0.5, 1e-9, -1e-9, 1e-16], (4000, 3))
    cells = np.concatenate([half, rng.uniform(-3, 4, (4000, 3)) * n, rng.uniform(-3000, 3000, (2000, 3)) * n])
    pos = np.array(o) + 0.5 * sp + cells * sp
    pos = np.concatenate([pos, np.nextafter(pos[:4000], 1e9), np.nextafter(pos[:4000], -1e9)])
    want = O.OracleField.grid(g, o, sp, True).eval(pos)
    assert same(capi.Field.grid3f(g, o, sp, reflective=True).eval(pos), want)


@pytest.mark.parametrize("n", [1, 5, 63, 1023, 1025, 4095, 4096, 4097, 66000])
@pytest.mark.parametrize("kind", ["BP", "CK"])
def test_spread_batches(kind, n):
    """A particle's steps do not depend on how many share its wave."""
    rng = np.random.default_rng(11)
    m = 4097
    g = noise((16, 16, 16))
    sp = [50 * KPC] * 3
    d = rng.normal(size=(m, 3))
    pos = rng.uniform(0, 800 * KPC, (m, 3))
    E = 10 ** rng.uniform(0, 2, m) * EEV
    q = np.where(np.arange(m) % 5 == 0, 0.0, EPLUS)
    if n <= m:
        pos, d, E, q = pos[:n], d[:n], E[:n], q[:n]
    else:
        pos, d, E, q = (np.concatenate([x] * (n // m + 1))[:n] for x in (pos, d, E, q))
    ref = O.OracleState(pos[:m], d[:m], E[:m], q[:m])
    O.propagate(O.OracleField.grid(g, [0, 0, 0], sp), O.PROP_BP if kind == "BP" else O.PROP_CK, ref, 20,
                tolerance=1e-3, min_step=KPC, max_step=100 * KPC, libm=O.LIBM_CR)
    b = capi.Batch(n)
    b.upload(pos, O.normalise(d), E, q)
    st = capi.Propagator(kind, capi.Field.grid3f(g, [0, 0, 0], sp), 1e-3, KPC, 100 * KPC).propagate(b, max_steps=20)
    out = b.download()
    assert st.accepted_steps == 20 * n
    for i in range(0, n, m):
        k = min(m, n - i)
        assert same(out["pos"][i:i + k], ref.pos[:k]) and same(out["next_step"][i:i + k], ref.next_step[:k])


@pytest.mark.parametrize("shape,reflective,clip", [((1, 1, 1), False, False), ((2, 3, 5), True, False),
                                                   ((4, 4, 4), False, True), ((33, 6, 19), False, False),
                                                   ((33, 6, 19), True, True)])
@pytest.mark.parametrize("kind,fixed", [("BP", True), ("BP", False), ("CK", True), ("CK", False)])
def test_tricubic_quads(kind, fixed, shape, reflective, clip):
    """Four lanes to a particle: every wrap of a row, ragged quads and waves, neutral particles among them."""
    rng = np.random.default_rng(13)
    n = 1003
    g = noise(shape)
    sp = [20 * KPC] * 3
    f = capi.Field.grid3f(g, [0, 0, 0], sp, reflective=reflective, clip_volume=clip)
    f.set_interpolation("TRICUBIC")
    of = O.OracleField.grid(g, [0, 0, 0], sp, reflective, clip, interp=O.GRID_TRICUBIC)
    L = np.array(shape) * 20 * KPC
    pos = rng.uniform(-0.6, 1.6, (n, 3)) * L
    q = np.where(np.arange(n) % 6 == 1, 0.0, EPLUS)
    lo, hi = (20 * KPC, 20 * KPC) if fixed else (KPC, 60 * KPC)
    compare(f, of, kind, pos, rng.normal(size=(n, 3)), 10 ** rng.uniform(0, 2, n) * EEV, q, 12, lo, hi, 1e-3)


@pytest.mark.parametrize("n", [1, 10279, 10281, 250001])
def test_download_returns_what_was_uploaded(n):
    """One chunk, a chunk's edges and several threads."""
    rng = np.random.default_rng(n)
    v = {k: rng.normal(size=(n, 3)) for k in ("pos", "dir", "source_pos", "created_pos")}
    s = {k: rng.normal(size=n) for k in ("energy", "charge", "current_step", "next_step", "trajectory_length", "time")}
    w = dict(active=rng.integers(0, 2, n).astype(np.int32), detection_index=rng.integers(0, 9, n).astype(np.int32),
             sde_step=rng.integers(0, 2 ** 32, n).astype(np.uint32))
    b = capi.Batch(n)
    b.upload(v["pos"], v["dir"], s["energy"], s["charge"], **{k: s[k] for k in list(s)[2:]}, **w,
             source_pos=v["source_pos"], created_pos=v["created_pos"])
    out = b.download()
    for k, a in {**v, **s, **w, "prev_pos": v["pos"], "prev_dir": v["dir"]}.items():
        assert np.array_equal(out[k].view(np.uint8), a.view(np.uint8)), k


@pytest.mark.parametrize("precision", [capi.PRECISION_FP64, capi.PRECISION_MIXED])
@pytest.mark.parametrize("n", [1, 255, 257, 43690, 43691, 100003])
def test_staged_eval(n, precision):
    """Positions that fill a slot and one more, against calls of 1000."""
    g = noise((9, 11, 10))
    f = capi.Field.grid3f(g, [0, 0, 0], 1.0)
    pos = np.random.default_rng(n).uniform(-20, 30, (n, 3))
    got = f.eval(pos, precision)
    want = np.concatenate([f.eval(pos[i:i + 1000], precision) for i in range(0, n, 1000)])
    assert same(got, want)
    if precision == capi.PRECISION_FP64:
        assert same(got, O.OracleField.grid(g, [0, 0, 0], 1.0).eval(pos))


@pytest.mark.parametrize("shape,clip", [((1, 1, 1), False), ((2, 3, 5), False), ((4, 4, 4), True), ((9, 6, 19), False)])
@pytest.mark.parametrize("kind,fixed", [("BP", True), ("BP", False), ("CK", True), ("CK", False)])
def test_tricubic_row_table(kind, fixed, shape, clip):
    """Batches that fill the chip read a table of row pairs built by the run: copies of the same particles, every
    wrap; then the caller's grid changes and the next run of the same batch sees it."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(17)
    m, n = 1003, 33100
    sp = [20 * KPC] * 3
    L = np.array(shape) * 20 * KPC
    pos, d, E = rng.uniform(-0.6, 1.6, (m, 3)) * L, rng.normal(size=(m, 3)), 10 ** rng.uniform(0, 2, m) * EEV
    q = np.where(np.arange(m) % 6 == 1, 0.0, EPLUS)
    lo, hi = (20 * KPC, 20 * KPC) if fixed else (KPC, 60 * KPC)
    idx = np.arange(n) % m
    dev = torch.empty(tuple(shape) + (3,), dtype=torch.float32, device="cuda:0")
    f = capi.Field.grid3f_device(dev.data_ptr(), shape, [0, 0, 0], sp, clip_volume=clip, keep=dev)
    f.set_interpolation("TRICUBIC")
    p, b = capi.Propagator(kind, f, 1e-3, lo, hi), capi.Batch(n)
    for seed in (3, 4):
        g = noise(shape, seed)
        dev.copy_(torch.from_numpy(g))
        torch.cuda.synchronize()
        ref = O.OracleState(pos, d, E, q)
        O.propagate(O.OracleField.grid(g, [0, 0, 0], sp, False, clip, interp=O.GRID_TRICUBIC),
                    O.PROP_BP if kind == "BP" else O.PROP_CK, ref, 8, tolerance=1e-3, min_step=lo, max_step=hi,
                    libm=O.LIBM_CR)
        b.upload(pos[idx], O.normalise(d)[idx], E[idx], q[idx])
        p.propagate(b, max_steps=8)
        out = b.download()
        for k in ("pos", "dir", "next_step", "trajectory_length"):
            assert same(out[k], getattr(ref, k)[idx]), k


def test_transfers_without_pinned_memory(monkeypatch):
    """With no pinned memory to be had, downloads, detections and field samples return the same bytes; a batch
    without detections needs none."""
    rng = np.random.default_rng(41)
    n = 25001
    f = capi.Field.grid3f(noise((8, 9, 7)), [0, 0, 0], [20 * KPC] * 3)
    pos = rng.uniform(0, 150 * KPC, (n, 3))
    p = capi.Propagator("BP", f, 1e-3, 5 * KPC, 5 * KPC, max_length=60 * KPC)
    p.set_observer([12 * KPC, 31 * KPC, 49 * KPC, 200 * KPC])
    b, empty = capi.Batch(n), capi.Batch(n)
    for x in (b, empty):
        x.upload(pos, O.normalise(rng.normal(size=(n, 3))), 10 ** rng.uniform(0, 2, n) * EEV, np.full(n, EPLUS))
    p.propagate(b, max_steps=8)
    got = [b.download(), b.detections(4), empty.detections(2), f.eval(pos)]
    monkeypatch.setenv("CRP_PINNED_SLOTS", "0")
    ref = [b.download(), b.detections(4), empty.detections(2), f.eval(pos)]
    assert np.isnan(got[2]).all() and np.isfinite(got[1][0]).all() and np.isnan(got[1][3]).all()
    for k in got[0]:
        assert np.array_equal(got[0][k].view(np.uint8), ref[0][k].view(np.uint8)), k
    for a, c in zip(got[1:], ref[1:]):
        assert np.array_equal(a.view(np.uint64), c.view(np.uint64))


@pytest.mark.parametrize("n", [1, 31, 33, 4095, 4097, 16383, 16385, 33000])
@pytest.mark.parametrize("name,kind,steps", [("grid", "BP", 20), ("grid", "BP", 520), ("grid", "CK", 20), ("reflective", "CK", 220),
                                             ("uniform", "BP", 20), ("uniform", "CK", 20)])
def test_fixed_steps_of_small_batches(name, kind, steps, n):
    """Fixed steps fill their waves fuller, by batch, field and length of the run: a particle's steps do not depend
    on it, on either path."""
    rng = np.random.default_rng(29)
    m = 97
    g, sp = noise((16, 16, 16)), [50 * KPC] * 3
    pos, d, E = rng.uniform(-100 * KPC, 900 * KPC, (m, 3)), rng.normal(size=(m, 3)), 10 ** rng.uniform(0, 2, m) * EEV
    q = np.where(np.arange(m) % 5 == 0, 0.0, EPLUS)
    if name == "uniform":
        B = (1e-13, -2e-13, 3e-14)
        f, of = capi.Field.uniform(B), O.OracleField.uniform(B)
    else:
        r = name == "reflective"
        f, of = capi.Field.grid3f(g, [0, 0, 0], sp, reflective=r), O.OracleField.grid(g, [0, 0, 0], sp, r)
    i, h = np.arange(n) % m, 20 * KPC
    ref = O.OracleState(pos, d, E, q)
    O.propagate(of, O.PROP_BP if kind == "BP" else O.PROP_CK, ref, steps, min_step=h, max_step=h, libm=O.LIBM_CR)
    for precision in (capi.PRECISION_FP64, capi.PRECISION_MIXED):
        b = capi.Batch(n)
        b.upload(pos[i], O.normalise(d)[i], E[i], q[i])
        st = capi.Propagator(kind, f, 1e-3, h, h, precision=precision).propagate(b, max_steps=steps)
        out = b.download()
        assert st.accepted_steps == steps * n
        for k in ("pos", "dir", "next_step", "trajectory_length"):
            if precision == capi.PRECISION_FP64:
                assert same(out[k], getattr(ref, k)[i]), k
            else:
                assert same(out[k], out[k][:m][i]), k


@pytest.mark.parametrize("n", [22528, 22529, 32768, 32769])
@pytest.mark.parametrize("shape", [(73, 72, 71), (33, 6, 19)])
@pytest.mark.parametrize("kind,fixed", [("BP", True), ("CK", False)])
def test_tricubic_switch_from_quads_to_the_row_table(kind, fixed, shape, n):
    """Either side of both lines (points beyond and within 4 MB): copies of the same particles against the oracle."""
    rng = np.random.default_rng(19)
    m = 257
    sp, steps = [20 * KPC] * 3, 40 if fixed else 7
    g = noise(shape)
    pos, d, E = rng.uniform(-0.6, 1.6, (m, 3)) * np.array(shape) * 20 * KPC, rng.normal(size=(m, 3)), \
        10 ** rng.uniform(0, 2, m) * EEV
    q = np.where(np.arange(m) % 6 == 1, 0.0, EPLUS)
    lo, hi = (20 * KPC, 20 * KPC) if fixed else (KPC, 60 * KPC)
    f = capi.Field.grid3f(g, [0, 0, 0], sp)
    f.set_interpolation("TRICUBIC")
    ref = O.OracleState(pos, d, E, q)
    O.propagate(O.OracleField.grid(g, [0, 0, 0], sp, interp=O.GRID_TRICUBIC), O.PROP_BP if kind == "BP" else O.PROP_CK,
                ref, steps, tolerance=1e-3, min_step=lo, max_step=hi, libm=O.LIBM_CR)
    idx = np.arange(n) % m
    b = capi.Batch(n)
    b.upload(pos[idx], O.normalise(d)[idx], E[idx], q[idx])
    capi.Propagator(kind, f, 1e-3, lo, hi).propagate(b, max_steps=steps)
    out = b.download()
    for k in ("pos", "dir", "next_step", "trajectory_length"):
        assert same(out[k], getattr(ref, k)[idx]), k


@pytest.mark.parametrize("kind,fixed", [("BP", True), ("BP", False), ("CK", True), ("CK", False)])
def test_tricubic_quads_with_boundaries_and_observer(kind, fixed):
    """Four lanes to a particle in a periodic box that shifts source and created positions, a sphere, a length limit
    and an observer: the same bits and counts as one lane to a particle (33100 copies, the row table)."""
    rng = np.random.default_rng(23)
    m = 331
    sp, L = [20 * KPC] * 3, np.array([120, 140, 100]) * KPC
    f = capi.Field.grid3f(noise((6, 7, 5)), [0, 0, 0], sp)
    f.set_interpolation("TRICUBIC")
    pos, d, E = rng.uniform(0, 1, (m, 3)) * L, O.normalise(rng.normal(size=(m, 3))), 10 ** rng.uniform(0, 2, m) * EEV
    q = np.where(np.arange(m) % 6 == 1, 0.0, EPLUS)
    src, made = rng.normal(size=(m, 3)) * KPC, rng.normal(size=(m, 3)) * KPC
    lo, hi = (15 * KPC, 15 * KPC) if fixed else (KPC, 60 * KPC)
    res = []
    for n in (m, 33100):
        p = capi.Propagator(kind, f, 1e-3, lo, hi, max_length=700 * KPC)
        p.set_observer([40 * KPC, 130 * KPC, 390 * KPC])
        p.set_periodic_box([0, 0, 0], L)
        p.set_spherical_boundary(L / 2, 95 * KPC, 1 * KPC)
        b, i = capi.Batch(n), np.arange(n) % m
        b.upload(pos[i], d[i], E[i], q[i], source_pos=src[i], created_pos=made[i])
        st = p.propagate(b, max_steps=60)
        res.append((b.download(), b.detections(3), st))
    (a, da, sa), (c, dc, sc) = res
    assert not same(a["source_pos"], src) and (a["detection_index"] > 0).any() and (a["active"] == 0).any()
    for k in a:
        assert np.array_equal(a[k].view(np.uint8), c[k][:m].view(np.uint8)), k
        assert np.array_equal(c[k][:m].view(np.uint8), c[k][m:2 * m].view(np.uint8)), k
    assert np.array_equal(da.view(np.uint64), dc[:, :m].view(np.uint64))
    assert sc.accepted_steps == 100 * sa.accepted_steps and sc.finished == 100 * sa.finished
