"""Differentiable fixed-step Boris propagation through a periodic Grid3f.

`BorisGridFunction` is a torch.autograd.Function whose forward and backward
are the HIP kernels behind crp_adjoint_forward_planned / crp_adjoint_backward_planned
(include/crpropa3_amd.h): the forward keeps the states every 8 steps (the state
every K steps where those take too much), the backward recomputes each run of
steps from the state before it, runs the hand-written reverse step and
accumulates the grid gradient in FP64.  One plan of the buffers, made in the
forward, serves both.

Model (per step h; PropagationBP::dY, src/module/PropagationBP.cpp:19-39, and
the two direction normalisations of :121 and src/ParticleState.cpp:30-32):
B = scale * trilinear(grid) in FP64.  Gradients are returned for the grid
values, the initial positions and directions, and the field scale.
Tensors live on the GPU; torch only supplies device memory and the stream.
"""
import ctypes as C

import torch

from . import capi

C_LIGHT = 2.99792458e8


class AdjointConfig(C.Structure):
    _fields_ = [("grid", C.c_void_p), ("nx", C.c_int), ("ny", C.c_int), ("nz", C.c_int),
                ("origin", C.c_double * 3), ("spacing", C.c_double * 3), ("scale", C.c_double),
                ("step", C.c_double), ("nsteps", C.c_int), ("checkpoint_every", C.c_int)]


class AdjointPlan(C.Structure):
    """crp_adjoint_plan: the buffers' layout, fixed once for a forward and its backward"""
    _fields_ = [("block_bytes", C.c_uint64), ("checkpoint_bytes", C.c_uint64), ("scratch_bytes", C.c_uint64),
                ("tile_shift", C.c_int32), ("keep_states", C.c_int32)]


def _bind():
    L = capi.lib()
    if getattr(L, "_adjoint_bound", False):
        return L
    P = C.POINTER(AdjointConfig)
    vp = C.c_void_p
    L.crp_adjoint_workspace.argtypes = [P, C.c_size_t, C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    L.crp_adjoint_forward.argtypes = [P, C.c_size_t, vp, vp, vp, vp, vp, vp, vp]
    L.crp_adjoint_backward.argtypes = [P, C.c_size_t, vp, vp, vp, vp, vp, vp, vp, vp, vp, vp]
    Q = C.POINTER(AdjointPlan)
    L.crp_adjoint_plan_make.argtypes = [P, C.c_size_t, C.c_int, Q]
    L.crp_adjoint_forward_planned.argtypes = [P, C.c_size_t, Q, vp, vp, vp, vp, vp, vp, vp]
    L.crp_adjoint_backward_planned.argtypes = [P, C.c_size_t, Q, vp, vp, vp, vp, vp, vp, vp, vp, vp, vp]
    L._adjoint_bound = True
    return L


def _ptr(t):
    return C.c_void_p(t.data_ptr()) if t is not None else None


def _config(grid, origin, spacing, scale, step, nsteps, K):
    cfg = AdjointConfig()
    cfg.grid = grid.data_ptr()
    cfg.nx, cfg.ny, cfg.nz = grid.shape[:3]
    for a in range(3):
        cfg.origin[a] = float(origin[a])
        cfg.spacing[a] = float(spacing[a])
    cfg.scale = float(scale)
    cfg.step = float(step)
    cfg.nsteps = int(nsteps)
    cfg.checkpoint_every = int(K)
    return cfg


def _roomy(nbytes, device):
    """Whether a buffer that lives until the backward leaves the card room: an eighth of what is free at most (small
    ones always), so that many of them alive at once do not fill it and the rest of a program finds its memory."""
    if nbytes <= 1 << 28 or torch.cuda.is_current_stream_capturing():
        return True
    free = torch.cuda.mem_get_info(device)[0]
    if 8 * nbytes <= free:
        return True
    return 8 * nbytes <= free + torch.cuda.memory_reserved(device) - torch.cuda.memory_allocated(device)


class BorisGridFunction(torch.autograd.Function):
    """(grid, x0, u0, scale) -> (x_final, u_final); see the module docstring."""

    @staticmethod
    def forward(ctx, grid, x0, u0, scale, kq, origin, spacing, step, nsteps, K, keep_states=None):
        if not (grid.is_cuda and x0.is_cuda and u0.is_cuda and kq.is_cuda):
            raise ValueError("BorisGridFunction: tensors must be on the GPU")
        grid = grid.detach().contiguous()
        if grid.dtype != torch.float32 or grid.dim() != 4 or grid.shape[3] != 3:
            raise ValueError("grid must be float32 of shape (nx, ny, nz, 3)")
        x0c = x0.detach().to(torch.float64).contiguous()
        u0c = u0.detach().to(torch.float64).contiguous()
        kqc = kq.detach().to(torch.float64).contiguous()
        n = x0c.shape[0]
        L = _bind()
        cfg = _config(grid, origin, spacing, float(scale), step, nsteps, K)
        plan = AdjointPlan()
        keep = any(ctx.needs_input_grad) if keep_states is None else bool(keep_states)
        capi.check(L.crp_adjoint_plan_make(C.byref(cfg), n, int(keep), C.byref(plan)))
        if keep_states is None and plan.keep_states and not _roomy(plan.checkpoint_bytes, grid.device):
            capi.check(L.crp_adjoint_plan_make(C.byref(cfg), n, 0, C.byref(plan)))
        ckpt = torch.empty(max(plan.checkpoint_bytes // 8, 1), dtype=torch.float64, device=grid.device)
        xo = torch.empty_like(x0c)
        uo = torch.empty_like(u0c)
        stream = C.c_void_p(torch.cuda.current_stream(grid.device).cuda_stream)
        capi.check(L.crp_adjoint_forward_planned(C.byref(cfg), n, C.byref(plan), _ptr(x0c), _ptr(u0c), _ptr(kqc),
                                                 _ptr(ckpt), _ptr(xo), _ptr(uo), stream))
        ctx.save_for_backward(grid, kqc, ckpt)
        ctx.meta = (origin, spacing, float(scale), step, nsteps, K, plan, grid.dtype)
        ctx.scale_is_tensor = torch.is_tensor(scale)
        return xo, uo

    @staticmethod
    def backward(ctx, gx, gu):
        grid, kqc, ckpt = ctx.saved_tensors
        origin, spacing, scale, step, nsteps, K, plan, gdtype = ctx.meta
        n = kqc.shape[0]
        dev = grid.device
        L = _bind()
        cfg = _config(grid, origin, spacing, scale, step, nsteps, K)
        gu = torch.zeros((n, 3), dtype=torch.float64, device=dev) if gu is None else gu.to(torch.float64).contiguous()
        gx = None if gx is None else gx.to(torch.float64).contiguous()
        scratch = torch.empty(max(plan.scratch_bytes // 8, 1), dtype=torch.float64, device=dev)
        ggrid = torch.zeros(grid.numel(), dtype=torch.float64, device=dev)
        gscale = torch.zeros(1, dtype=torch.float64, device=dev)
        gx0 = torch.empty((n, 3), dtype=torch.float64, device=dev)
        gu0 = torch.empty((n, 3), dtype=torch.float64, device=dev)
        stream = C.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
        capi.check(L.crp_adjoint_backward_planned(C.byref(cfg), n, C.byref(plan), _ptr(kqc), _ptr(ckpt), _ptr(gx),
                                                  _ptr(gu), _ptr(scratch), _ptr(ggrid), _ptr(gx0), _ptr(gu0),
                                                  _ptr(gscale), stream))
        gs = gscale.view(()) if ctx.scale_is_tensor else None
        return (ggrid.view(grid.shape).to(gdtype), gx0, gu0, gs, None, None, None, None, None, None, None)


def boris_grid_propagate(grid, x0, u0, energy, charge, origin, spacing, step, nsteps, checkpoint_every=64,
                         scale=1.0, keep_states=None):
    """Differentiable fixed-step Boris push of particles through `scale * grid`.

    grid: (nx, ny, nz, 3) float32 CUDA tensor (periodic Grid3f values); x0, u0: (n, 3)
    float64 CUDA tensors (positions [m], unit directions); energy [J], charge [C]: (n,)
    tensors or floats.  `scale` may be a float or a 0-d tensor requiring grad.
    Between forward and backward the graph holds the state every `checkpoint_every` (K) steps, 48/K bytes a step
    and particle, and the grid's cell table; or, with `keep_states`, the states every 8 steps, 6 bytes a step and
    particle whatever K is, for a shorter backward (the same values).  keep_states None keeps them where a
    backward can follow, they take at most 4 GiB and the card has eight times that free; False leaves K to bound
    the memory.  Returns (x_final, u_final)."""
    dev = grid.device
    E = torch.as_tensor(energy, dtype=torch.float64, device=dev).expand(x0.shape[0])
    q = torch.as_tensor(charge, dtype=torch.float64, device=dev).expand(x0.shape[0])
    kq = (q * C_LIGHT * step / (2 * E)).contiguous()
    if not torch.is_tensor(scale):
        scale = torch.tensor(float(scale), dtype=torch.float64, device=dev)
    if keep_states is None and not torch.is_grad_enabled():
        keep_states = False
    return BorisGridFunction.apply(grid, x0, u0, scale, kq, origin, spacing, step, nsteps, checkpoint_every,
                                   keep_states)
