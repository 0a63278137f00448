"""Host side of the fused AcceleratedPGM deconvolution: what it takes over
from the solver, without a GPU (the device conversions and the kernels are
replaced)."""

import types

import numpy as np
import pytest
import torch

from scico_amd import _device as dev
from scico_amd.optimize import _pgm


@pytest.fixture
def fused(monkeypatch):
    """A fused iteration of a 4 x 5 problem with its kernels left out; calls
    that would launch are counted in ``primed``."""

    def as_device(x, dtype=np.float32):
        return torch.as_tensor(x).to(dev.torch_dtype(dtype)).contiguous()

    monkeypatch.setattr(dev, "as_device", as_device)
    f = object.__new__(_pgm._FusedDeconv)
    f.M, f.N = 4, 5
    y = torch.zeros(4, 5)
    f.pgm = types.SimpleNamespace(x=torch.zeros(4, 5), v=torch.zeros(4, 5), L=1.0,
                                  f=types.SimpleNamespace(A=object(), y=y, scale=0.5),
                                  g=types.SimpleNamespace(scale=1.0))
    f.primed = 0

    def prime(same):
        f.primed += 1

    f._prime = prime
    f._made_from = f._inputs(f.pgm)
    f.adopt_state()
    return f


@pytest.mark.parametrize("name", ["x", "v"])
@pytest.mark.parametrize("shape", [(4, 4), (5, 4), (20,), (1, 4, 5), ()])
def test_assigned_state_of_another_shape_is_refused(fused, name, shape):
    setattr(fused.pgm, name, torch.zeros(shape))
    with pytest.raises(ValueError, match="Shapes do not conform"):
        fused.current()
    assert fused.primed == 1
    assert fused.x.shape == fused.v.shape == (4, 5)


@pytest.mark.parametrize("given", [torch.ones(4, 5, dtype=torch.float64), np.ones((4, 5)),
                                   torch.ones(5, 4).T, torch.ones(4, 5, dtype=torch.int32)])
def test_assigned_state_is_converted(fused, given):
    fused.pgm.v = given
    assert fused.current() is fused and fused.primed == 2
    v = fused.pgm.v
    assert v is fused.v and v is not given
    assert v.dtype == torch.float32 and v.is_contiguous() and torch.equal(v, torch.ones(4, 5))


def test_replaced_problem_asks_for_another_path(fused, monkeypatch):
    """Functionals without the attributes of the fused structure, and changes
    of those it was made from, go back to the choice of a path."""
    built = []
    monkeypatch.setattr(_pgm._FusedDeconv, "build", staticmethod(lambda p: built.append(p)))
    assert fused.current() is fused and not built
    keep = fused.pgm.f, fused.pgm.g
    for f, g in ((object(), keep[1]), (keep[0], object()),
                 (types.SimpleNamespace(A=keep[0].A, y=np.zeros((4, 5)), scale=0.5), keep[1])):
        fused.pgm.f, fused.pgm.g = f, g
        assert fused.current() is None and len(built) == 1
        built.clear()
        fused.pgm.f, fused.pgm.g = keep
        assert fused.current() is fused and not built
    fused.pgm.f.y.add_(1.0)
    assert fused.current() is None and len(built) == 1


def test_inference_mode(fused):
    """In inference mode, and with data made there, the state is taken over
    and followed as elsewhere: torch keeps no count of changes for tensors of
    that mode, so the solver's own are made outside it."""
    with torch.inference_mode():
        fused.pgm.x = torch.ones(4, 5)
        fused.pgm.f.y = torch.ones(4, 5)
        fused._made_from = fused._inputs(fused.pgm)
        assert fused.current() is fused and fused.primed == 2
        assert fused.current() is fused and fused.primed == 2
        assert torch.equal(fused.x, torch.ones(4, 5))
        fused.pgm.v.mul_(2.0)
        assert fused.current() is fused and fused.primed == 3
    assert fused.current() is fused and fused.primed == 3


@pytest.mark.parametrize("code", [-6, -5, -4])
def test_plan_failures(monkeypatch, code):
    """Only a size without a plan declines the fused iteration; a plan that
    could not be made is reported."""
    from scico_amd._lib import ScxrError
    from scico_amd.functional import IsotropicTVNorm
    from scico_amd.linop import CircularConvolve
    from scico_amd.loss import SquaredL2Loss

    def plan(self):
        raise ScxrError("scxr_cconv_plan_create", code, "")

    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(_pgm, "load", lambda: types.SimpleNamespace(scxr_cconv_apgm_parts=int))
    monkeypatch.setattr(CircularConvolve, "plan", property(plan))
    A = object.__new__(CircularConvolve)
    A.ndims, A.input_shape, A.fft_shape = 2, (4, 5), (4, 5)
    f = object.__new__(SquaredL2Loss)
    f.A, f.y, f.scale = A, torch.zeros(4, 5), 0.5
    pgm = types.SimpleNamespace(f=f, g=IsotropicTVNorm(), x=torch.zeros(4, 5))
    if code == -6:
        assert _pgm._FusedDeconv.build(pgm) is None
    else:
        with pytest.raises(ScxrError) as e:
            _pgm._FusedDeconv.build(pgm)
        assert e.value.code == code
