"""Proximal gradient methods (``scico/optimize/_pgm.py:30-252``,
``scico/optimize/_pgmaux.py:23-62``).

``PGM`` / ``AcceleratedPGM`` follow the reference algorithm for any
``f`` with a gradient and ``g`` with a prox.  For the deconvolution
structure

    f = SquaredL2Loss(y, CircularConvolve (one real image, both axes of 3 or
                      more pixels), scale=0.5),
    g = lam * IsotropicTVNorm() or lam * AnisotropicTVNorm()  (2D),
    constant step size,

the iteration runs through fused kernels (:class:`_FusedDeconv`): the
prox writes x, the partials of the residual and of TV(x) and the
extrapolated point in one pass, and one FFT convolution by ``G = A^T A`` per iteration gives both
the next gradient (``G v = (1 + c) G x - c G x_prev`` by linearity) and,
on the way through the spectrum, the objective (Parseval).  The reference
evaluates three convolutions per iteration (``A v``, ``A^T r`` and
``A x`` for the objective).
"""

from __future__ import annotations

from typing import List

import numpy as np
import torch

from .. import _device as dev
from .. import _vec as vec
from .._lib import SCXR_ERR_UNSUPPORTED, ScxrError, call, load
from ._common import Optimizer


class PGMStepSize:
    """Constant reciprocal step size ``L`` (``_pgmaux.py:23-62``)."""

    def internal_init(self, pgm):
        self.pgm = pgm

    def update(self, v):
        return self.pgm.L


class PGM(Optimizer):
    def __init__(self, f, g, L0: float, x0, step_size=None, **kwargs):
        self.f = f
        if g.has_prox is not True:
            raise ValueError(f"Functional 'g' ({type(g)}) must have a prox method.")
        self.g = g
        if step_size is None:
            step_size = PGMStepSize()
        if type(step_size) is not PGMStepSize:
            raise NotImplementedError("Only the constant PGMStepSize is supported.")
        self.step_size = step_size
        self.step_size.internal_init(self)
        self.L = float(L0)
        self.fixed_point_residual = float("inf")
        self.x = dev.as_device(x0).clone()
        super().__init__(**kwargs)

    def x_step(self, v, L):
        """``g.prox(v - (1/L) grad f(v), 1/L)`` (``_pgm.py:106-117``)."""
        u = vec.axpby(1.0, v, -(1.0 / L), self.f.grad(v))
        return self.g.prox(u, 1.0 / L)

    def _working_vars_finite(self) -> bool:
        return bool(torch.isfinite(self.x).all().item())

    def _objective_evaluatable(self):
        return self.f.has_eval and self.g.has_eval

    def _itstat_extra_fields(self):
        return {"L": "%9.3e", "Residual": "%9.3e"}, ["L", "norm_residual()"]

    def _state_variable_names(self) -> List[str]:
        return ["x", "L"]

    def minimizer(self):
        return self.x

    def objective(self, x=None):
        """``f(x) + g(x)`` (``_pgm.py:151-156``), device float64."""
        fused = getattr(self, "_fused", None)
        if x is None and fused is not None and fused.has_row():
            return fused.stat(0)
        x = self.x if x is None else x
        return self.f(x) + self.g(x)

    def norm_residual(self):
        return self.fixed_point_residual

    def _momentum(self):
        """Extrapolation coefficient of the step (0 for PGM)."""
        return 0.0

    def step(self):
        if getattr(self, "_fused", None) is not None:
            self._fused.step(self._momentum())
            return
        self.L = self.step_size.update(self.x)
        x = self.x_step(self.x, self.L)
        self.fixed_point_residual = vec.reduce(vec.RED_SQDIST, self.x, x, post=vec.POST_SQRT)
        self.x = x


class AcceleratedPGM(PGM):
    """FISTA (``_pgm.py:183-252``)."""

    def __init__(self, f, g, L0: float, x0, step_size=None, **kwargs):
        super().__init__(f=f, g=g, L0=L0, x0=x0, step_size=step_size, **kwargs)
        self.v = self.x.clone()
        self.t = 1.0
        self._fused = _FusedDeconv.build(self)

    def _momentum(self):
        # t_{k+1} = (1 + sqrt(1 + 4 t_k^2)) / 2 in float32, as the reference
        # evaluates it after the first step (data independent: host side)
        t_old = self.t
        f32 = np.float32
        self.t = float(f32(0.5) * (f32(1) + np.sqrt(f32(1) + f32(4) * f32(t_old) ** 2)))
        return float(f32(f32(t_old) - f32(1)) / f32(self.t))

    def _after_load_state(self):
        if getattr(self, "_fused", None) is not None:
            self._fused.adopt_state()

    def step(self):
        if self._fused is not None:
            self._fused = self._fused.current()
        if self._fused is not None:
            self._fused.step(self._momentum())
            return
        x_old = self.x
        self.L = self.step_size.update(self.v)
        self.x = self.x_step(self.v, self.L)
        self.fixed_point_residual = vec.reduce(vec.RED_SQDIST, self.x, self.v,
                                               post=vec.POST_SQRT)
        # t_{k+1} = (1 + sqrt(1 + 4 t_k^2)) / 2 in float32, as the reference
        # evaluates it after the first step (the sequence does not depend on
        # the data, so it is computed on the host).
        t_old = self.t
        f32 = np.float32
        self.t = float(f32(0.5) * (f32(1) + np.sqrt(f32(1) + f32(4) * f32(t_old) ** 2)))
        c = float(f32(f32(t_old) - f32(1)) / f32(self.t))
        self.v = vec.axpby(1.0, self.x, c, vec.add(self.x, -1.0, x_old))

    def _working_vars_finite(self) -> bool:
        return bool(torch.isfinite(self.x).all().item()) and bool(torch.isfinite(self.v).all().item())

    def _state_variable_names(self) -> List[str]:
        return ["x", "v", "t", "L"]


def _version(t):
    """torch's count of a tensor's in-place changes; None where there is none
    (inference tensors, host arrays)."""
    if not isinstance(t, torch.Tensor) or t.is_inference():
        return None
    return t._version


class _FusedDeconv:
    """Fused device implementation of AcceleratedPGM-TV deconvolution."""

    enabled = True  # tests switch this off to run the generic path

    @staticmethod
    def build(pgm: AcceleratedPGM):
        from ..functional import ScaledFunctional
        from ..functional._tvnorm import TVNorm
        from ..linop import CircularConvolve
        from ..loss import SquaredL2Loss

        if not _FusedDeconv.enabled or not torch.cuda.is_available():
            return None
        f, g = pgm.f, pgm.g
        if not (type(f) is SquaredL2Loss and f.scale == 0.5 and type(f.A) is CircularConvolve):
            return None
        A = f.A
        if not (A.ndims == 2 and A.input_shape == A.fft_shape and
                tuple(f.y.shape) == A.input_shape):
            return None
        scale, base = (g.scale, g.functional) if isinstance(g, ScaledFunctional) else (1.0, g)
        if not isinstance(base, TVNorm) or base.axes is not None:
            return None
        if tuple(pgm.x.shape) != A.input_shape or pgm.x.dtype != torch.float32:
            return None
        try:
            if int(load().scxr_cconv_apgm_parts(A.plan)) <= 0:
                return None
        except ScxrError as e:
            if e.code != SCXR_ERR_UNSUPPORTED:
                raise
            return None  # no plan for this size: the generic path reports it when used
        return _FusedDeconv(pgm, float(scale), base)

    @staticmethod
    def _inputs(pgm):
        """What the set-up is made from: the objects, and with their identities
        the values that change in place (torch counts a tensor's changes,
        except those of a y made in inference mode, which are not followed)."""
        f, g = pgm.f, pgm.g
        A, y, base = getattr(f, "A", None), getattr(f, "y", None), getattr(g, "functional", g)
        return (f, A, y, g, base), (id(f), id(A), id(y), id(g), id(base),
                                    getattr(f, "scale", None), _version(y),
                                    getattr(g, "scale", 1.0), getattr(base, "isotropic", None),
                                    getattr(base, "circular", None))

    def _same_problem(self):
        # (the objects are held, so that no other can have one's identity)
        return self._inputs(self.pgm)[1] == self._made_from[1]

    def has_row(self):
        """Whether the last statistics row is that of the solver's present x
        (not replaced, modified or loaded since the step) and problem."""
        return self._stepped and self.pgm.x is self.x and \
            self.x._version == self._versions[0] and self._same_problem()

    def current(self):
        """This object if the solver's problem and state are the ones that it
        left, itself brought up to date if only the state was replaced or
        modified (or L), else what the new problem calls for (host checks)."""
        if not self._same_problem():
            return _FusedDeconv.build(self.pgm)
        p = self.pgm
        if p.x is not self.x or p.v is not self.v or float(p.L) != self._L or \
                (self.x._version, self.v._version) != self._versions:
            self.adopt_state()
        return self

    def __init__(self, pgm: AcceleratedPGM, lam: float, tv):
        self.pgm = pgm
        self.A = pgm.f.A
        self.lam = lam
        self.iso = int(tv.isotropic)
        self.circ = int(tv.circular)
        self.M, self.N = self.A.input_shape
        n = self.M * self.N
        lib = load()
        f32 = dict(dtype=torch.float32, device=dev.DEVICE)
        f64 = dict(dtype=torch.float64, device=dev.DEVICE)
        y = dev.as_device(pgm.f.y)
        self._made_from = self._inputs(pgm)
        # the half-grid spectra of G = A^T A and of y, and A^T y, formed in
        # float64 on the device and rounded once (host FFTs took 15 ms of a new
        # 1024 x 1024 problem; the rounding of A^T y stays in every gradient)
        H1 = self.N // 2 + 1
        self.gs = torch.empty(self.M * H1, **f32)
        self.Yh = torch.empty(2 * self.M * H1, **f32)
        ws = torch.empty(int(lib.scxr_cconv_apgm_setup_ws(self.A.plan)), **f64)
        self.aty = torch.empty((self.M, self.N), **f32)
        call("scxr_cconv_apgm_setup_aty", self.A.plan, y.data_ptr(), self.gs.data_ptr(),
             self.Yh.data_ptr(), self.aty.data_ptr(), ws.data_ptr(), dev.stream())
        self.n_obj = int(lib.scxr_cconv_apgm_parts(self.A.plan))
        self.n_res = int(lib.scxr_tv_prox_apgm_parts(self.M, self.N))
        self.n_tv = self.n_res  # the prox kernel's TV partials, one per workgroup
        self.ws_obj = torch.empty(self.n_obj, **f64)
        self.ws_res = torch.empty(self.n_res, **f64)
        self.ws_tv = torch.empty(self.n_tv, **f64)
        self.u = torch.empty((self.M, self.N), **f32)
        self.gx = torch.zeros((self.M, self.N), **f32)
        self.obj_scale = 0.5 / float(n)
        self.hist_cap = 0
        self.hist = None
        self.counter = torch.zeros(1, dtype=torch.int32, device=dev.DEVICE)
        self.n_steps = 0
        self._consts_of = (None, 0.0, 0.0)  # L and the b and tau of it
        self._reserve(max(64, pgm.maxiter))
        self.adopt_state(same=getattr(pgm, "itnum", 0) == 0 and pgm.t == 1.0)

    def _reserve(self, rows: int):
        if rows <= self.hist_cap:
            return
        new = torch.zeros((rows, 2), dtype=torch.float64, device=dev.DEVICE)
        if self.hist is not None:
            new[: self.hist_cap] = self.hist
        self.hist, self.hist_cap = new, rows

    def stat(self, col: int):
        return self.hist[self.n_steps - 1, col]

    def _consts(self):
        L = float(self.pgm.L)
        if L != self._consts_of[0]:
            lam_eff = (1.0 / L) * self.lam  # ScaledFunctional.prox(v, 1/L)
            tau = float(np.float32(np.float32(np.sqrt(np.float32(2.0))) * np.float32(4)) *
                        np.float32(lam_eff))
            self._consts_of = (L, -(1.0 / L), tau)
        return self._consts_of[1:]

    def adopt_state(self, same: bool = False):
        """Own contiguous x and v, and the first gradient step from them
        (``same``: v is known to equal x, as in a new solver).  The kernels take
        pointers, so both are brought to the device and to float32, and one of
        another shape is refused."""
        p = self.pgm
        self._stepped = False
        x = dev.input_array(p.x, (self.M, self.N), "x")
        v = dev.input_array(p.v, (self.M, self.N), "v") if hasattr(p, "v") else x
        with torch.inference_mode(False):  # (tensors with a count of their changes)
            self.x, self.v = x.clone(), v.clone()
        self._publish()
        self._L = float(p.L)
        self._prime(same)

    def _publish(self):
        self.pgm.x = self.x
        if hasattr(self.pgm, "v"):
            self.pgm.v = self.v
        self._versions = (self.x._version, self.v._version)

    def _prime(self, same: bool):
        """The state a step starts from: u = v - (1/L) grad f(v) and gx = G x
        (the step forms G v_next = (1 + c) G x_next - c gx)."""
        b, _ = self._consts()
        P = lambda t: t.data_ptr()
        s = dev.stream()
        vec.fill(self.gx, 0.0)
        call("scxr_cconv_apgm_grad", self.A.plan, P(self.v), P(self.gs), None, None, P(self.gx),
             P(self.v), P(self.aty), 0.0, b, P(self.u), None, s)
        if not same:  # a mid-run state: gx = G x as well (no look at the values: capturable)
            scratch = torch.empty_like(self.u)
            call("scxr_cconv_apgm_grad", self.A.plan, P(self.x), P(self.gs), None, None,
                 P(self.gx), P(self.x), P(self.aty), 0.0, b, P(scratch), None, s)

    def step(self, c: float):
        if self.n_steps >= self.hist_cap:
            self._reserve(2 * self.hist_cap)
        # An iterate once published keeps its values: a step makes new tensors.
        # A captured step updates the solver's own instead, so that each replay
        # goes on from the last one's results.
        if torch.cuda.is_current_stream_capturing():
            self.enqueue(c)
        elif torch.is_inference_mode_enabled():
            with torch.inference_mode(False):  # (tensors with a count of their changes)
                self.enqueue(c, torch.empty_like(self.x), torch.empty_like(self.v))
        else:
            self.enqueue(c, torch.empty_like(self.x), torch.empty_like(self.v))
        self.n_steps += 1
        self._stepped = True
        self._publish()
        self.pgm.fixed_point_residual = self.stat(1)

    def enqueue(self, c: float, x_new=None, v_new=None):
        """One iteration (no host synchronisation; capturable), of x and v in
        place or into new tensors."""
        b, tau = self._consts()
        P = lambda t: t.data_ptr()
        s = dev.stream()
        x, v = self.x, self.v
        if x_new is not None:
            self.x, self.v = x_new, v_new
        call("scxr_tv_prox_apgm_to", self.M, self.N, P(self.u), P(x), P(v), P(self.x), P(self.v),
             tau, self.iso, self.circ, c, P(self.ws_res), P(self.ws_tv), None, s)
        call("scxr_cconv_apgm_grad_itstat", self.A.plan, P(self.x), P(self.gs), P(self.Yh),
             P(self.ws_obj), P(self.gx), P(self.v), P(self.aty), c, b, P(self.u), self.obj_scale,
             P(self.ws_tv), self.n_tv, self.lam, P(self.ws_res), self.n_res, P(self.hist),
             P(self.counter), self.hist_cap, None, s)
