"""Cell tables beyond the reach of the first-level address translation (3 GB): batches of 44 particles to a SIMD and
more (45056 on 256 compute units) are gathered by waves together, smaller ones read by each lane.  The same bits as
the point layout's eight scattered reads, for every step kind, with ragged batches, neutral and inactive particles
and positions outside a clipped volume; the tests with 45055 particles and more take both sides of the line, those
with up to 1000 the lanes' loads."""
import numpy as np
import pytest

from crpropa3_amd import capi

pytestmark = pytest.mark.gpu

KPC = 3.0856775814913674e19
EPLUS = 1.602176487e-19
EEV = 1e18 * EPLUS
SHAPE = (301, 277, 283)  # 3.02 GB of 128-byte cells


@pytest.fixture(scope="module")
def fields():
    torch = pytest.importorskip("torch")
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(5)
    g = torch.randn(SHAPE + (3,), generator=gen, device="cuda:0") * 1e-13
    torch.cuda.synchronize()
    out = {}
    for clip in (False, True):
        for layout in ("cells", "points"):
            f = capi.Field.grid3f_device(g.data_ptr(), SHAPE, [0, 0, 0], [20 * KPC] * 3, clip_volume=clip, keep=g)
            out[clip, layout] = f.set_layout(layout)
    return out


def _run(field, kind, fixed, n, steps, precision):
    rng = np.random.default_rng(n)
    L = np.array(SHAPE) * 20 * KPC
    pos = rng.uniform(-0.2, 1.2, (n, 3)) * L
    d = rng.normal(size=(n, 3))
    d /= np.sqrt((d * d).sum(1))[:, None]
    q = np.where(np.arange(n) % 7 == 3, 0.0, EPLUS)
    act = (np.arange(n) % 11 != 5).astype(np.int32)
    lo, hi = (10 * KPC, 10 * KPC) if fixed else (1 * KPC, 50 * KPC)
    p = capi.Propagator(kind, field, 1e-3 if kind == "BP" else 1e-4, lo, hi, precision=precision)
    b = capi.Batch(n)
    b.upload(pos, d, 10 ** rng.uniform(0, 2, n) * EEV, q, active=act)
    st = p.propagate(b, max_steps=steps)
    return b.download(), st


@pytest.mark.parametrize("n", [1, 63, 1000])
@pytest.mark.parametrize("clip", [False, True])
@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("kind", ["BP", "CK"])
def test_wave_gather_equals_point_layout(fields, kind, fixed, clip, n):
    print(kind, fixed, clip, n, flush=True)
    a, sa = _run(fields[clip, "cells"], kind, fixed, n, 20, capi.PRECISION_FP64)
    b, sb = _run(fields[clip, "points"], kind, fixed, n, 20, capi.PRECISION_FP64)
    assert sa.accepted_steps == sb.accepted_steps and sa.rejected_trials == sb.rejected_trials
    for k in a:
        assert np.array_equal(a[k].view(np.uint8), b[k].view(np.uint8)), k


@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("kind", ["BP", "CK"])
def test_wave_gather_mixed(fields, kind, fixed):
    """The mixed path against the FP64 path: three fixed 10 kpc steps, or the first adaptive step (its size is
    the minimum; later sizes follow the rounding of the error estimate, a difference of nearly equal terms).
    FP32 rounding of field values and directions, 2^-24 each over at most 3 x 6 evaluations: below 2e-6 of a
    step, a step below 1/500 of the largest position."""
    print(kind, fixed, flush=True)
    steps = 3 if fixed else 1
    a, _ = _run(fields[False, "cells"], kind, fixed, 1000, steps, capi.PRECISION_MIXED)
    b, _ = _run(fields[False, "cells"], kind, fixed, 1000, steps, capi.PRECISION_FP64)
    err = np.abs(a["pos"] - b["pos"]).max(axis=1) / np.abs(b["pos"]).max()
    assert err.max() < 1e-8


@pytest.mark.parametrize("n", [45055, 45056, 45057, 66001])
@pytest.mark.parametrize("clip", [False, True])
@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("kind", ["BP", "CK"])
def test_batches_around_the_switch_to_wave_gathers(fields, kind, fixed, clip, n):
    """Waves gather from 176 particles to a compute unit on (45056 on 256 units), the lanes' own loads serve smaller
    batches: either side of the line, a ragged last wave, and enough particles that lanes take a second one."""
    print(kind, fixed, clip, n, flush=True)
    a, sa = _run(fields[clip, "cells"], kind, fixed, n, 6, capi.PRECISION_FP64)
    b, sb = _run(fields[clip, "points"], kind, fixed, n, 6, capi.PRECISION_FP64)
    assert sa.accepted_steps == sb.accepted_steps and sa.rejected_trials == sb.rejected_trials
    for k in a:
        assert np.array_equal(a[k].view(np.uint8), b[k].view(np.uint8)), k


@pytest.mark.parametrize("n", [45055, 45056, 66001])
@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("kind", ["BP", "CK"])
def test_wave_gather_mixed_large_batches(fields, kind, fixed, n):
    """test_wave_gather_mixed's bound where the waves gather."""
    print(kind, fixed, n, flush=True)
    steps = 3 if fixed else 1
    a, _ = _run(fields[False, "cells"], kind, fixed, n, steps, capi.PRECISION_MIXED)
    b, _ = _run(fields[False, "points"], kind, fixed, n, steps, capi.PRECISION_FP64)
    err = np.abs(a["pos"] - b["pos"]).max(axis=1) / np.abs(b["pos"]).max()
    assert err.max() < 1e-8
