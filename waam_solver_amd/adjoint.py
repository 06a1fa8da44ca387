"""The differentiation form: gradients of the thermal sub-step through many steps.

Forward: the coupled step's thermal chain with frozen flags (and phi) and zero velocity, on a
copy of a twin's state (reference solvers/coupled_step.py:97-160, the flow and the free surface
held): Gaussian2D arc injection, enthalpy ceiling, conduction from the step's starting
temperature, boundary losses, enthalpy floor, phase map, ceiling, phase map — the product's own
kernels, one launch each. Parameters theta = (eta, s_h, s_sigma): the arc efficiency, a factor
on both loss coefficients (the calibration overlay's heat-loss factor) and a factor on the arc
radius (its sigma scale).

Backward: hand-written adjoint kernels (``csrc/adjoint.hip``) step the adjoint state
lambda = dL/dH back through each step and accumulate dL/dtheta in binary64. The forward keeps
the enthalpy every ``checkpoint_every`` steps; the backward recomputes each segment from its
checkpoint (keeping the step's enthalpy after the arc, before and after the floor, and its
starting f_l), then runs the segment's adjoint steps in reverse. ``ThermalRolloutFn`` wraps the
pair as a ``torch.autograd.Function`` of theta returning the final (T, f_l), so any loss written
in torch differentiates through it; ``fit_calibration`` runs gradient descent on it.

Derivatives at the piecewise points are one-sided (a clamped value has derivative 0; the phase
map's slope is the one of the branch the enthalpy is on); f_l enters the arc's surface weight
only through a step at 0.55, whose derivative is 0.
"""

from __future__ import annotations

import ctypes

import numpy as np
import torch

from . import kernels
from ._lib import lib
from .field import P, tensor_of
from .physics import weld_forces
from .solvers.coupled_step import resolve_arc_k

_f = ctypes.c_float


class AdjConsts(ctypes.Structure):
    _fields_ = [(n, _f) for n in (
        "cp_rho", "L_rho", "T_s", "T_l", "T_cap", "T_floor", "alpha_lu", "T_amb", "h_conv0",
        "eps_rad0", "sigma_sb", "dt", "dx", "loss_scale", "arc_i", "arc_j", "arc_k", "sigma",
        "sigma0", "Q_w", "eta", "dx3", "pen")] + [(n, ctypes.c_int32) for n in (
            "enable_cap", "enable_loss", "enable_arc", "enable_conv", "enable_rad",
            "surface_weight")]


class RolloutC(ctypes.Structure):
    """include/waam_hip.h waam_rollout."""

    _fields_ = ([("c", AdjConsts)] + [(n, _f) for n in (
        "h_conv", "eps_rad", "gamma_lu", "cos_t", "sin_t", "dgamma", "p_sigma", "p_pa",
        "rho_phys", "g_lu", "beta", "F_cap", "u_cap", "omega_s", "omega_b", "C_darcy")] +
        [(n, ctypes.c_int32) for n in (
            "flow", "enable_csf", "wetting", "enable_hydro", "nx", "ny", "nz", "layout", "stack",
            "slot0", "n_active")] +
        [(n, ctypes.c_void_p) for n in (
            "H", "T", "fl", "u", "f", "flags", "phi", "active", "A", "B", "E", "F", "Fr", "Fc",
            "sums", "depth", "scratch")])


class RollbackC(ctypes.Structure):
    """include/waam_hip.h waam_rollback."""

    _fields_ = [(n, ctypes.c_void_p) for n in (
        "lam_H", "lam_u", "lam_f", "lam_T1", "lam_fl1", "G", "lamC", "lamB", "parts",
        "step_totals", "grads")] + [(n, ctypes.c_double) for n in (
            "omega_s", "omega_b", "C_darcy", "u_cap", "F_cap", "g_lu", "beta", "T_l",
            "dgamma")] + [("slot", ctypes.c_int32)]


class ThermalRollout:
    """n_steps of the thermal sub-step from the twin's current state along ``path``
    (step -> torch (x_m, y_m)), differentiable in theta."""

    def __init__(self, twin, n_steps: int, path, checkpoint_every: int = 50,
                 is_welding: bool = True):
        if type(twin.arc_source).__name__ != "Gaussian2D":
            raise NotImplementedError("the differentiation form covers the Gaussian2D arc")
        twin.sync()
        self.tw, g = twin, twin.grid
        self.n_steps, self.K = int(n_steps), max(1, int(checkpoint_every))
        self.path, self.is_welding = path, bool(is_welding)
        f = lambda: g.field(torch.float32)  # noqa: E731
        # the starting state is the twin's enthalpy with T and f_l from the phase map, as at
        # every later step boundary (and as the checkpoints restore it)
        self.H0, self.T0, self.fl0 = f(), f(), f()
        tensor_of(self.H0).copy_(tensor_of(g.H))
        kernels.update_phase(self.H0, self.T0, self.fl0, twin.cp_rho, twin.L_rho,
                             twin.mat.T_solidus, twin.mat.T_liquidus)
        # the rollout's own copies of the frozen flags and phi: the twin may step (and the fused
        # step updates phi in place and swaps its flag buffers) between forward and backward
        self.flags = g.field(torch.uint8, np_dtype=np.int32)
        self.phi = f()
        tensor_of(self.flags).copy_(tensor_of(g.flags))
        tensor_of(self.phi).copy_(tensor_of(g.phi))
        self.h_conv0, self.eps0 = float(twin.h_conv), float(twin.eps_rad)
        self.sigma0 = float(twin.sigma_cells)
        x0, y0 = path(0)
        self.arc_k = resolve_arc_k(twin, g, x0 / g.dx, y0 / g.dx)
        self.shape = tuple(tensor_of(self.H0).shape)
        self._slots = {k: self._new(2) for k in ("H", "T", "fl")}
        self._sums = torch.empty(2, dtype=torch.float64, device=g.device)
        self._depth = torch.empty(g.nz, dtype=torch.float32, device=g.device)
        self.ckpt: list[torch.Tensor] = []
        self.theta = None

    def _new(self, *lead) -> torch.Tensor:
        """Uninitialised fp32 storage of `lead` fields."""
        return torch.empty(tuple(lead) + self.shape, dtype=torch.float32,
                           device=self.tw.grid.device)

    def _arcs(self, s0: int, n: int):
        """The arc centres (cells) of steps s0 .. s0 + n - 1, as two double arrays."""
        dx = self.tw.grid.dx
        pos = [self.path(s) for s in range(s0, s0 + n)]
        return ((ctypes.c_double * n)(*[p[0] / dx for p in pos]),
                (ctypes.c_double * n)(*[p[1] / dx for p in pos]))

    def _rollout(self, bufs: dict, stack: bool, slot0: int) -> RolloutC:
        """The call's parameters; bufs holds the state's slots and, for the backward, the saved
        fields (the caller keeps it until the call returns)."""
        tw, g = self.tw, self.tw.grid
        r = RolloutC(c=self._consts(0), h_conv=self.h_conv0 * self.theta[1],
                     eps_rad=self.eps0 * self.theta[1], nx=g.nx, ny=g.ny, nz=g.nz,
                     layout=g.layout, stack=int(stack), slot0=slot0, flags=P(self.flags),
                     phi=P(self.phi), sums=P(self._sums), depth=P(self._depth),
                     scratch=P(g.scratch))
        for name, t in bufs.items():
            setattr(r, name, P(t))
        return r

    def _run(self, s0: int, n: int, bufs: dict, stack: bool = False, slot0: int = 0) -> None:
        # locals, as the arcs: addressof keeps no reference
        r = self._rollout(bufs, stack, slot0)
        ai, aj = self._arcs(s0, n)
        lib().call("waam_rollout_forward", ctypes.addressof(r),
                   ctypes.addressof(ai), ctypes.addressof(aj), n,
                   torch.cuda.current_stream().cuda_stream)

    def _segments(self):
        return [(s0, min(self.K, self.n_steps - s0)) for s0 in range(0, self.n_steps, self.K)]

    # ------------------------------------------------------------------ forward
    def forward(self, theta) -> tuple[torch.Tensor, torch.Tensor]:
        """Final (T, f_l) (storage order) after n_steps with parameters theta."""
        self.theta = tuple(float(v) for v in theta)
        self.ckpt = []
        sl = self._slots
        for name, src in (("H", self.H0), ("T", self.T0), ("fl", self.fl0)):
            sl[name][0].copy_(tensor_of(src))
        slot = 0
        for s0, n in self._segments():
            self.ckpt.append(sl["H"][slot].clone())
            self._run(s0, n, sl, slot0=slot)
            slot = (slot + n) & 1
        self.H_final = sl["H"][slot].clone()
        return sl["T"][slot].clone(), sl["fl"][slot].clone()

    # ------------------------------------------------------------------ backward
    def _consts(self, n: int) -> AdjConsts:
        tw, g = self.tw, self.tw.grid
        eta, s_h, s_sig = self.theta
        x, y = self.path(n)
        m = tw.mat
        c = AdjConsts(cp_rho=tw.cp_rho, L_rho=tw.L_rho, T_s=m.T_solidus, T_l=m.T_liquidus,
                      T_cap=tw.T_vapor_cap_K, T_floor=tw.T_amb, alpha_lu=tw.alpha_lu,
                      T_amb=tw.T_amb, h_conv0=self.h_conv0, eps_rad0=self.eps0,
                      sigma_sb=tw.sigma_sb, dt=g.dt, dx=g.dx, loss_scale=s_h, arc_i=x / g.dx,
                      arc_j=y / g.dx, arc_k=self.arc_k, sigma=self.sigma0 * s_sig,
                      sigma0=self.sigma0, Q_w=tw.Q_w, eta=eta, dx3=g.dx ** 3,
                      pen=tw.arc_penetration_m / g.dx)
        c.enable_cap = 1 if tw.enable_enthalpy_cap else 0
        c.enable_loss = 1 if tw.enable_heat_loss else 0
        c.enable_arc = 1 if self.is_welding else 0
        c.enable_conv = 1 if tw.enable_convection else 0
        c.enable_rad = 1 if tw.enable_radiation else 0
        c.surface_weight = 1 if tw.arc_surface_weighting else 0
        return c

    def backward(self, grad_T: torch.Tensor, grad_fl: torch.Tensor) -> np.ndarray:
        """dL/dtheta (float64) given dL/dT and dL/df_l at the final step."""
        if self.theta is None:
            raise RuntimeError("backward before forward")
        tw, g = self.tw, self.tw.grid
        st = torch.cuda.current_stream().cuda_stream
        dev = g.device
        L = min(self.K, self.n_steps)
        lam = self._new(2)
        grads = torch.zeros(3, dtype=torch.float64, device=dev)
        parts = torch.empty(L * 6 * 1024, dtype=torch.float64, device=dev)
        totals = torch.empty(L * 3, dtype=torch.float64, device=dev)
        c_last = self._consts(self.n_steps - 1)
        # P() hands over a bare address: the converted seeds are held in locals until the
        # kernels that read them are queued (a temporary would be freed, and its memory reused,
        # before the call)
        gT = grad_T.float().contiguous()
        gfl = grad_fl.float().contiguous()
        lib().call("waam_adj_terminal", P(self.H_final), P(gT), P(gfl), P(self.flags),
                   ctypes.addressof(c_last), P(lam), g.n_cells, st)
        # a segment's state and saved fields, one slot a step (T, which only the forward reads: two
        # in turn), reused from segment to segment
        sv = {k: self._new(2 if k == "T" else L + 1) for k in ("H", "T", "fl")}
        sv.update({k: self._new(L) for k in ("A", "E", "F")})
        sv["sums"] = torch.empty(2 * L, dtype=torch.float64, device=dev)
        slot = 0
        for (s0, n), H in zip(reversed(self._segments()), reversed(self.ckpt)):
            sv["H"][0].copy_(H)
            lib().call("waam_update_phase", P(sv["H"]), P(sv["T"]), P(sv["fl"]), tw.cp_rho,
                       tw.L_rho, tw.mat.T_solidus, tw.mat.T_liquidus, g.n_cells, st)
            self._run(s0, n, sv, stack=True)
            ai, aj = self._arcs(s0, n)
            r = self._rollout(sv, True, 0)
            lib().call("waam_adj_rollback", ctypes.addressof(r),
                       ctypes.addressof(ai), ctypes.addressof(aj), n, P(lam), slot, P(parts),
                       P(totals), P(grads), st)
            slot = (slot + n) & 1
        self.lam0 = lam[slot]
        return grads.cpu().numpy()


class ThermalRolloutFn(torch.autograd.Function):
    """(T_final, f_l_final) = rollout(theta), differentiable in theta (a length-3 tensor)."""

    @staticmethod
    def forward(ctx, theta: torch.Tensor, rollout: ThermalRollout):
        T, fl = rollout.forward(theta.detach().double().cpu().numpy())
        ctx.rollout = rollout
        ctx.theta_dtype, ctx.theta_device = theta.dtype, theta.device
        return T, fl

    @staticmethod
    def backward(ctx, grad_T, grad_fl):
        g = ctx.rollout.backward(grad_T.float(), grad_fl.float())
        return torch.tensor(g, dtype=ctx.theta_dtype, device=ctx.theta_device), None


def field_loss(T, fl, T_target, fl_target, T_scale: float = 100.0):
    """Mean squared error of the final temperature (scaled) and liquid fraction fields."""
    return (((T - T_target) / T_scale) ** 2).mean() + ((fl - fl_target) ** 2).mean()


def fit_calibration(rollout: ThermalRollout, T_target, fl_target, theta0, iters: int = 20,
                    lr: float = 0.02) -> dict:
    """Gradient descent (Adam) on theta = (eta, s_h, s_sigma) against target fields; returns the
    parameter and loss history."""
    theta = torch.tensor(theta0, dtype=torch.float64, requires_grad=True)
    opt = torch.optim.Adam([theta], lr=lr)
    hist = {"theta": [], "loss": []}
    for _ in range(iters):
        opt.zero_grad()
        T, fl = ThermalRolloutFn.apply(theta, rollout)
        loss = field_loss(T, fl, T_target, fl_target)
        loss.backward()
        hist["theta"].append(theta.detach().numpy().copy())
        hist["loss"].append(float(loss))
        opt.step()
    return hist


# ---------------------------------------------------------------------------- Marangoni forcing
def marangoni_force(T: torch.Tensor, phi: torch.Tensor, f_l: torch.Tensor, flags: torch.Tensor,
                    dgamma: float, dims: tuple[int, int, int], layout: int):
    """The thermocapillary force (reference kernels.py:2158-2217) on device tensors, through the
    product kernel: (Fx, Fy, Fz), zero where it does not apply."""
    nx, ny, nz = dims
    F = [torch.zeros_like(T) for _ in range(3)]
    st = torch.cuda.current_stream().cuda_stream
    lib().call("waam_compute_marangoni_force", T.data_ptr(), phi.data_ptr(), f_l.data_ptr(),
               F[0].data_ptr(), F[1].data_ptr(), F[2].data_ptr(), flags.data_ptr(), float(dgamma),
               nx, ny, nz, layout, st)
    return tuple(F)


def marangoni_force_vjp(T, phi, f_l, flags, lam, dgamma: float, dims, layout: int):
    """Hand-written adjoint (``waam_adj_marangoni``) of ``marangoni_force`` with phi, f_l and
    the flags held: for lam = (dL/dFx, dL/dFy, dL/dFz), returns dL/dT (binary64, shaped like
    T) and dL/d(dgamma) (a binary64 sum over the cells)."""
    nx, ny, nz = dims
    lam = [x.contiguous().float() for x in lam]
    T_adj = torch.zeros(T.shape, dtype=torch.float64, device=T.device)
    s_cell = torch.empty(T.shape, dtype=torch.float64, device=T.device)
    G = torch.empty((3,) + tuple(T.shape), dtype=torch.float64, device=T.device)
    st = torch.cuda.current_stream().cuda_stream
    lib().call("waam_adj_marangoni", T.data_ptr(), phi.data_ptr(), f_l.data_ptr(),
               flags.data_ptr(), lam[0].data_ptr(), lam[1].data_ptr(), lam[2].data_ptr(),
               float(dgamma), T_adj.data_ptr(), s_cell.data_ptr(), G.data_ptr(), nx, ny, nz,
               layout, st)
    return T_adj, s_cell.sum()


class MarangoniForceFn(torch.autograd.Function):
    """(T, dgamma) -> (Fx, Fy, Fz) as a ``torch.autograd.Function``: forward through the
    product kernel, backward through the adjoint kernels (phi, f_l and the flags held, as the
    thermal rollout holds them)."""

    @staticmethod
    def forward(ctx, T, dgamma, phi, f_l, flags, dims, layout):
        ctx.save_for_backward(T, phi, f_l, flags)
        ctx.dgamma, ctx.dims, ctx.layout = float(dgamma), dims, layout
        return marangoni_force(T, phi, f_l, flags, float(dgamma), dims, layout)

    @staticmethod
    def backward(ctx, gx, gy, gz):
        T, phi, f_l, flags = ctx.saved_tensors
        zero = torch.zeros_like(T)
        lam = [g if g is not None else zero for g in (gx, gy, gz)]
        T_adj, d_dg = marangoni_force_vjp(T, phi, f_l, flags, lam, ctx.dgamma, ctx.dims,
                                          ctx.layout)
        g_T = T_adj.to(T.dtype) if ctx.needs_input_grad[0] else None
        g_dg = d_dg.reshape(()) if ctx.needs_input_grad[1] else None
        return g_T, g_dg, None, None, None, None, None


# ---------------------------------------------------------------------------- collision
def collide_srt_vjp(f_src, Fx, Fy, Fz, f_l, flags, lam, omega: float, C_darcy: float):
    """Hand-written adjoint (``waam_adj_collide_srt``) of the BGK collision with Guo forcing and
    the Carman-Kozeny drag (reference kernels.py:2815-2885), f_l and the flags held: for
    lam = dL/d(post-collision populations) (19 q-major n-cell arrays), returns dL/d(f_src)
    (float64, like f_src) and dL/d(Fx, Fy, Fz) (float64, (3,) + the field shape)."""
    n = f_l.numel()
    lam = lam.contiguous().float()
    lam_f = torch.empty(f_src.shape, dtype=torch.float64, device=f_src.device)
    lam_F = torch.empty((3,) + tuple(f_l.shape), dtype=torch.float64, device=f_src.device)
    st = torch.cuda.current_stream().cuda_stream
    lib().call("waam_adj_collide_srt", f_src.data_ptr(), Fx.data_ptr(), Fy.data_ptr(),
               Fz.data_ptr(), f_l.data_ptr(), flags.data_ptr(), lam.data_ptr(), float(omega),
               float(C_darcy), lam_f.data_ptr(), lam_F.data_ptr(), n, st)
    return lam_f, lam_F


# ---------------------------------------------------------------------------- the coupled step
class CoupledRollout:
    """n_steps of the coupled step with the flags and phi frozen, from the twin's current state
    along ``path`` (step -> torch (x_m, y_m)), differentiable in theta = (eta, s_h, s_sigma).

    Forward, per step (reference solvers/coupled_step.py:97-409 with the free surface, the flags,
    deposition and the stream held), the product's own kernels: arc injection and ceiling,
    conduction and enthalpy advection by the step's starting velocity, boundary losses, floor,
    phase map, ceiling, phase map; clear forces, CSF, Marangoni, arc pressure, hydrostatic
    gravity, buoyancy, force clamp; MRT collision and Mach clamp. With frozen flags the stream
    never feeds a collided cell (the next collision reads the cell's own post-collision
    populations), so the populations ping-pong between two buffers without it.

    Backward (``csrc/adjoint_coupled.hip``): the adjoint state (lambda_H, lambda_f, lambda_u) in
    binary64 runs back through each step — collision with the Mach clamp, forces with the force
    clamp, the phase map, the thermal chain with advection — and accumulates dL/dtheta in
    binary64. The forward keeps the state every ``checkpoint_every`` steps and the backward
    recomputes each segment from its checkpoint."""

    ADVECTION = ("flow", "frozen", "none")

    def __init__(self, twin, n_steps: int, path, checkpoint_every: int = 50,
                 is_welding: bool = True, advection: str = "flow"):
        """advection: "flow" — the enthalpy is advected by the velocity each step's collision
        produces (the coupled step); "frozen" — by the starting velocity throughout, with the
        forces and the collision left out; "none" — not at all (the thermal chain alone)."""
        if advection not in self.ADVECTION:
            raise ValueError(f"advection {advection!r} (one of {self.ADVECTION})")
        self.advection = advection
        if type(twin.arc_source).__name__ != "Gaussian2D":
            raise NotImplementedError("the differentiation form covers the Gaussian2D arc")
        if twin.use_srt or twin.use_material_tables:
            raise NotImplementedError("the coupled adjoint covers the scalar-material MRT step")
        if twin.enable_recoil or twin.enable_gas_shear or twin.enable_lorentz:
            raise NotImplementedError("the coupled adjoint covers the flow-tier forces")
        twin.sync()
        self.tw, g = twin, twin.grid
        self.n_steps, self.K = int(n_steps), max(1, int(checkpoint_every))
        self.path, self.is_welding = path, bool(is_welding)
        self.flags = g.field(torch.uint8, np_dtype=np.int32)
        self.phi = g.field(torch.float32)
        tensor_of(self.flags).copy_(tensor_of(g.flags))
        tensor_of(self.phi).copy_(tensor_of(g.phi))
        # the starting state: the twin's enthalpy (T, f_l from the phase map), populations and
        # velocity
        self.H0 = tensor_of(g.H).clone()
        self.f0 = tensor_of(g.f_src).clone()
        self.u0 = [tensor_of(x).clone() for x in (g.ux, g.uy, g.uz)]
        self.shape = tuple(self.H0.shape)
        # the FLUID/IFACE cells (the flags are held): the flow runs over them, and populations
        # and velocity are only read and written there
        fl = tensor_of(self.flags).reshape(-1)
        self._cells = torch.nonzero((fl == g.FLAG_FLUID) | (fl == g.FLAG_IFACE)).reshape(-1)
        self._active = self._cells.to(torch.int32)
        self._slots = {k: self._new(2) for k in ("H", "T", "fl")}
        if advection == "flow":
            self._slots["u"], self._slots["f"] = self._new(2, 3), self._new(2, 19)
        elif advection == "frozen":
            # the velocity the enthalpy is advected by when it does not evolve
            self._slots["u"] = torch.stack(self.u0)
        self._sums = torch.empty(2, dtype=torch.float64, device=g.device)
        self._depth = torch.empty(g.nz, dtype=torch.float32, device=g.device)
        self.h_conv0, self.eps0 = float(twin.h_conv), float(twin.eps_rad)
        self.sigma0 = float(twin.sigma_cells)
        x0, y0 = path(0)
        self.arc_k = resolve_arc_k(twin, g, x0 / g.dx, y0 / g.dx)
        self.u_cap = float(getattr(twin, "u_mach_limit_lu", 0.08))
        self.F_cap = float(getattr(twin, "force_limit_lu", 0.05))
        self.ckpt: list = []
        self.theta = None

    def _rollout(self, bufs: dict, stack: bool, slot0: int) -> RolloutC:
        r = ThermalRollout._rollout(self, bufs, stack, slot0)
        tw = self.tw
        r.flow = {"none": 0, "frozen": 1, "flow": 2}[self.advection]
        r.active, r.n_active = P(self._active), self._active.numel()
        r.enable_csf, r.wetting = int(bool(tw.enable_csf_tension)), int(bool(tw.enable_wetting))
        r.enable_hydro = int(bool(tw.enable_hydrostatic_gravity))
        r.gamma_lu, r.dgamma = tw.gamma_lu, tw.dgamma_dT_lu
        r.cos_t, r.sin_t = kernels.contact_angle_cos_sin(tw.theta_rad)
        r.p_sigma = weld_forces.arc_pressure_sigma_cells(tw)
        r.p_pa = weld_forces.arc_pressure_peak_pa(tw)
        r.rho_phys, r.g_lu, r.beta = tw.mat.rho, tw.g_lu, tw.beta_T
        r.F_cap, r.u_cap = self.F_cap, self.u_cap
        r.omega_s, r.omega_b, r.C_darcy = tw.omega, tw.omega_bulk, tw.C_darcy
        return r

    def _rollback(self, lam: dict, slot: int) -> RollbackC:
        """The backward call's parameters; lam holds its buffers (kept by the caller). The flow's
        coefficients go in binary64: the adjoint is one of the step's equations, whose forward
        alone is fp32."""
        tw = self.tw
        return RollbackC(omega_s=tw.omega, omega_b=tw.omega_bulk, C_darcy=tw.C_darcy,
                         u_cap=self.u_cap, F_cap=self.F_cap, g_lu=tw.g_lu, beta=tw.beta_T,
                         T_l=tw.mat.T_liquidus, dgamma=tw.dgamma_dT_lu, slot=slot,
                         **{k: P(v) for k, v in lam.items()})

    def _cells_of(self, t: torch.Tensor) -> torch.Tensor:
        """The listed cells' values of a stack of fields, (fields, cells)."""
        return t.reshape(-1, self.tw.grid.n_cells)[:, self._cells]

    def _put(self, bufs: dict, H, fc, uc) -> None:
        """A state (H, and with the flow the listed cells' populations and velocity) into slot 0:
        T and f_l from the phase map."""
        tw, g = self.tw, self.tw.grid
        bufs["H"][0].copy_(H)
        lib().call("waam_update_phase", P(bufs["H"]), P(bufs["T"]), P(bufs["fl"]), tw.cp_rho,
                   tw.L_rho, tw.mat.T_solidus, tw.mat.T_liquidus, g.n_cells,
                   torch.cuda.current_stream().cuda_stream)
        if self.advection == "flow":
            for name, v in (("f", fc), ("u", uc)):
                bufs[name][0].reshape(-1, g.n_cells)[:, self._cells] = v

    # ------------------------------------------------------------------ forward
    def forward(self, theta) -> tuple[torch.Tensor, torch.Tensor]:
        """Final (T, f_l) (storage order) after n_steps with parameters theta."""
        self.theta = tuple(float(v) for v in theta)
        self.ckpt = []
        sl, flow = self._slots, self.advection == "flow"
        self._put(sl, self.H0, self._cells_of(self.f0), self._cells_of(torch.stack(self.u0)))
        slot = 0
        for s0, n in self._segments():
            self.ckpt.append((sl["H"][slot].clone(),) + (
                (self._cells_of(sl["f"][slot]), self._cells_of(sl["u"][slot])) if flow
                else (None, None)))
            self._run(s0, n, sl, slot0=slot)
            slot = (slot + n) & 1
        self.H_final = sl["H"][slot].clone()
        return sl["T"][slot].clone(), sl["fl"][slot].clone()

    # ------------------------------------------------------------------ backward
    def backward(self, grad_T: torch.Tensor, grad_fl: torch.Tensor) -> np.ndarray:
        """dL/dtheta (float64) given dL/dT and dL/df_l at the final step."""
        if self.theta is None:
            raise RuntimeError("backward before forward")
        g = self.tw.grid
        st = torch.cuda.current_stream().cuda_stream
        shp = self.shape
        d64 = dict(dtype=torch.float64, device=g.device)
        flow, adv = self.advection == "flow", self.advection != "none"
        L = min(self.K, self.n_steps)
        z = lambda *lead: torch.zeros(lead + shp, **d64)  # noqa: E731
        lam = {"lam_H": z(2), "lamC": torch.empty(shp, **d64), "lamB": torch.empty(shp, **d64),
               "parts": torch.empty(L * 6 * 1024, **d64), "step_totals": torch.empty(3 * L, **d64),
               "grads": torch.zeros(3, **d64)}
        if adv:
            lam["lam_u"] = z(2, 3)
        if flow:
            # zero outside the listed cells, and never written there
            lam.update(lam_f=z(2, 19), lam_T1=z(), lam_fl1=z(), G=z(3))
        c_last = self._consts(self.n_steps - 1)
        # the binary64 seeds live in locals while their kernel is queued (P() keeps no reference)
        gT = grad_T.double().contiguous()
        gfl = grad_fl.double().contiguous()
        lib().call("waam_cadj_phase", P(self.H_final), P(self.flags), ctypes.addressof(c_last),
                   P(gT), P(gfl), P(lam["lam_H"]), g.n_cells, st)
        # a segment's state and saved fields, one slot a step, reused from segment to segment
        # (T: two in turn where only the forward reads it)
        sv = {k: self._new(2 if k == "T" and not flow else L + 1) for k in ("H", "T", "fl")}
        sv.update({k: self._new(L) for k in (("A", "B", "E", "F") if adv else ("A", "E", "F"))})
        if flow:
            sv.update(u=self._new(L + 1, 3), f=self._new(L + 1, 19), Fr=self._new(L, 3),
                      Fc=self._new(L, 3))
        elif adv:
            sv["u"] = self._slots["u"]
        sv["sums"] = torch.empty(2 * L, **d64)
        slot = 0
        for (s0, n), state in zip(reversed(self._segments()), reversed(self.ckpt)):
            self._put(sv, *state)
            self._run(s0, n, sv, stack=True)
            ai, aj = self._arcs(s0, n)
            b = self._rollback(lam, slot)
            r = self._rollout(sv, True, 0)
            lib().call("waam_cadj_rollback", ctypes.addressof(r),
                       ctypes.addressof(b), ctypes.addressof(ai), ctypes.addressof(aj), n, st)
            slot = (slot + n) & 1
        self.lam0 = lam["lam_H"][slot]
        return lam["grads"].cpu().numpy()

    _new, _arcs = ThermalRollout._new, ThermalRollout._arcs
    _run, _segments = ThermalRollout._run, ThermalRollout._segments

    def _consts(self, n: int) -> AdjConsts:
        return ThermalRollout._consts(self, n)


class CoupledRolloutFn(torch.autograd.Function):
    """(T_final, f_l_final) = coupled rollout(theta), differentiable in theta (length 3)."""

    @staticmethod
    def forward(ctx, theta: torch.Tensor, rollout: CoupledRollout):
        T, fl = rollout.forward(theta.detach().double().cpu().numpy())
        ctx.rollout = rollout
        ctx.theta_dtype, ctx.theta_device = theta.dtype, theta.device
        return T, fl

    @staticmethod
    def backward(ctx, grad_T, grad_fl):
        g = ctx.rollout.backward(grad_T, grad_fl)
        return torch.tensor(g, dtype=ctx.theta_dtype, device=ctx.theta_device), None


def pool_wd_surrogate(fl: torch.Tensor, i_c: int, nz_solid: int, layout: int, dx: float,
                      tau: float = 0.1) -> tuple[torch.Tensor, torch.Tensor]:
    """Smoothed pool width and depth (m) on the cross-section x = i_c, differentiable in f_l.

    The reference's telemetry (twin.py:716-744) counts, on the cross-section through the pool,
    the y-extent of f_l > 0.5 and the plate layers down to the deepest f_l > 0.5: step functions
    of f_l. The surrogate replaces each column's and each plate layer's indicator with a logistic
    of its largest liquid fraction: W = dx * sum_j s((max_k f_l(i_c, j, k) - 0.5) / tau),
    D = dx * sum_{k < nz_solid} s((max_j f_l(i_c, j, k) - 0.5) / tau), s the logistic function;
    as tau -> 0 these become the cell counts of a pool without holes."""
    sec = fl[:, :, i_c] if layout == 1 else fl[i_c].transpose(0, 1)  # (nz, ny)
    col = sec.max(dim=0).values            # per j: the column's largest f_l
    lay = sec[:nz_solid].max(dim=1).values  # per plate layer
    W = dx * torch.sigmoid((col - 0.5) / tau).sum()
    D = dx * torch.sigmoid((lay - 0.5) / tau).sum()
    return W, D
