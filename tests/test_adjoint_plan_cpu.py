"""Sizes and layout of the adjoint's buffers: what crp_adjoint_workspace documents, and a plan that the environment
does not change once it is made."""
import ctypes as C

import pytest

from crpropa3_amd import adjoint, capi

SETTINGS = [dict(), dict(CRP_ADJOINT_BLOCK_BYTES="0"), dict(CRP_ADJOINT_BLOCK_BYTES="3e4"),
            dict(CRP_ADJOINT_BLOCK_BYTES="1e12"), dict(CRP_ADJOINT_TILE_SHIFT="4")]


def config(N=20, nsteps=130, K=8):
    cfg = adjoint.AdjointConfig()
    cfg.grid, cfg.nx, cfg.ny, cfg.nz, cfg.nsteps, cfg.checkpoint_every = 1, N, N, N, nsteps, K
    for a in range(3):
        cfg.spacing[a] = 1.0
    return cfg


@pytest.mark.parametrize("env", SETTINGS)
@pytest.mark.parametrize("N,n,nsteps,K", [(20, 96, 130, 8), (16, 1, 1, 64), (128, 65536, 4096, 64), (176, 1000, 77, 10)])
def test_checkpoints_have_the_documented_size(env, N, n, nsteps, K, monkeypatch):
    """A state every K steps and the cell table, whatever the environment: a caller may size the buffer by the
    header's formula."""
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    size = C.c_size_t(0)
    capi.check(adjoint._bind().crp_adjoint_workspace(C.byref(config(N, nsteps, K)), n, C.byref(size), None))
    assert size.value == (-(-nsteps // K) * 48 * n + 255) // 256 * 256 + 128 * N ** 3


def test_plan_is_checked_against_its_configuration():
    L = adjoint._bind()
    plan = adjoint.AdjointPlan()
    capi.check(L.crp_adjoint_plan_make(C.byref(config()), 96, 1, C.byref(plan)))
    assert plan.keep_states == 1 and plan.checkpoint_bytes >= 6 * 96 * 130 + 128 * 20 ** 3
    one = C.c_void_p(256)  # never read: the calls fail before
    for cfg, n in ((config(nsteps=131, K=8), 96), (config(K=9), 96), (config(N=40), 96), (config(), 97)):
        with pytest.raises(capi.CrpError):
            capi.check(L.crp_adjoint_forward_planned(C.byref(cfg), n, C.byref(plan), *[one] * 7))
        with pytest.raises(capi.CrpError):
            capi.check(L.crp_adjoint_backward_planned(C.byref(cfg), n, C.byref(plan), *[one] * 10))
    for bad in (None, C.byref(adjoint.AdjointPlan())):
        with pytest.raises(capi.CrpError):
            capi.check(L.crp_adjoint_forward_planned(C.byref(config()), 96, bad, *[one] * 7))
