"""GPU checks of the FP32 training kernels on the matrix instructions: the
forward step, the adjoint and the parameter gradient summed in it, against
the FP64 kernels, on cell counts below, at and off a wave's 64 cells and a
block's share, in both forms of the incoming adjoint."""
import pytest
import torch

import lettuce_amd as lt
from lettuce_amd import _native as N
from lettuce_amd.ext._training import _Problem
from tests.test_learned_oracle import _grid, _grid27, _theta

pytestmark = pytest.mark.gpu
F32, F64 = torch.float32, torch.float64
DEV = torch.device("cuda:0")


def _populations(shape):
    """near-equilibrium populations [Q, *shape], cut from a cubic field"""
    if len(shape) == 2:
        f = _grid(n=max(shape), seed=sum(shape))
        return f[:, :shape[0], :shape[1]].contiguous()
    f = _grid27(n=max(shape), seed=sum(shape))
    return f[:, :shape[0], :shape[1], :shape[2]].contiguous()


@pytest.mark.parametrize("gathered", [False, True])
@pytest.mark.parametrize("out_scale,lo,hi", [(0.3, 0.05, 1.95), (3.0, 0.9, 1.1)])
@pytest.mark.parametrize("shape", [(3, 4), (8, 8), (5, 13), (37, 61), (300, 257),
                                   (3, 3, 3), (4, 4, 4), (5, 3, 13), (31, 18, 23)])
def test_fused_step_and_gradient_match_fp64(shape, out_scale, lo, hi, gathered):
    # the rates read 100 x non-equilibrium moments, which FP32 populations
    # carry to about 100 * 2^-24 * 4 = 2e-5 each: rates and adjoints follow
    # to about 1e-4 of their size; at out_scale 3 ten times that, and the
    # odd rate that sits so close to a limit may fall on either side of it
    tol = 1e-3 if out_scale < 1 else 1e-2
    f = _populations(shape)
    theta = _theta(3, out_scale=out_scale)
    g = torch.Generator().manual_seed(7)
    lam = torch.rand(f.shape, generator=g, dtype=F64) - 0.5
    grad0 = torch.randn(N.LEARNED_PARAMS, generator=g, dtype=F64)
    cfg = lt.TrainConfig(tau=0.57, in_scale=100.0, rate_lo=lo, rate_hi=hi)
    res = {}
    for dt in (F64, F32):
        fd, ld = f.to(DEV, dt).contiguous(), lam.to(DEV, dt).contiguous()
        prob = _Problem(fd, theta.to(DEV, dt), cfg)
        nxt, mu = torch.full_like(fd, float("nan")), torch.full_like(fd, float("nan"))
        prob.step(fd, nxt)
        ws, grad = prob.grad_workspace(), torch.zeros(N.LEARNED_PARAMS, dtype=dt, device=DEV)
        base = grad0.to(DEV, dt)
        for out in (grad, base):
            if prob.fused_gradient:
                prob.adjoint_gradient(fd, ld, gathered, mu, ws, out)
            else:
                rec = torch.empty((N.LEARNED_RECORD, prob.cells), dtype=dt, device=DEV)
                prob.adjoint(fd, ld, gathered, mu, rec)
                prob.grad_reduce(rec, ws, out)
        # onto a gradient that is there: the same sum is added
        added = (base.double() - grad0.to(DEV, dt).double() - grad.double()).abs().max().item()
        assert added <= 1e-6 * (1 + grad.abs().max().item())
        res[dt] = [t.double().cpu() for t in (nxt, mu, grad)]
    assert prob.fused_gradient
    for a, b, t in zip(res[F64], res[F32], (1e-5 if out_scale < 1 else 1e-4, tol, tol)):
        err, size = (a - b).norm().item(), a.norm().item()
        assert err <= t * size, (err, size)


def test_fused_gradient_is_refused_in_fp64():
    f = _grid(n=8, seed=0).to(DEV).contiguous()
    theta = _theta(0).to(DEV)
    prob = _Problem(f, theta, lt.TrainConfig(tau=0.57))
    assert N.lib().lbm_learned_gradient_workspace(N.F64, prob.cells) < 0
    with pytest.raises(RuntimeError):
        prob.adjoint_gradient(f, f, False, torch.empty_like(f), theta, theta.clone())


@pytest.mark.parametrize("shape", [(5, 241, 251), (67, 65, 63)])
def test_waves_that_take_several_tiles(shape):
    """more cells than the kernels' waves hold at once (262144), with a rest:
    the waves' LDS areas are used again, their sums go on over their tiles.
    Each block of parameters against its own norm: the rates follow to about
    1e-4 of their size (see above), and a sum over cells to the same relative
    error as its terms; three times that."""
    f = torch.stack([_grid(n=max(shape[1:]), seed=b)[:, :shape[1], :shape[2]]
                     for b in range(shape[0])], dim=1) if shape[0] == 5 else _populations(shape)
    theta = _theta(3, out_scale=0.3)
    lam = torch.rand(f.shape, generator=torch.Generator().manual_seed(7), dtype=F64) - 0.5
    cfg = lt.TrainConfig(tau=0.57, in_scale=100.0, rate_lo=0.05, rate_hi=1.95)
    res = {}
    for dt in (F64, F32):
        fd, ld = f.to(DEV, dt).contiguous(), lam.to(DEV, dt).contiguous()
        prob = _Problem(fd, theta.to(DEV, dt), cfg)
        nxt, mu = torch.full_like(fd, float("nan")), torch.full_like(fd, float("nan"))
        prob.step(fd, nxt)
        ws, grad = prob.grad_workspace(), torch.zeros(N.LEARNED_PARAMS, dtype=dt, device=DEV)
        if prob.fused_gradient:
            prob.adjoint_gradient(fd, ld, True, mu, ws, grad)
        else:
            rec = torch.empty((N.LEARNED_RECORD, prob.cells), dtype=dt, device=DEV)
            prob.adjoint(fd, ld, True, mu, rec)
            prob.grad_reduce(rec, ws, grad)
        blocks = torch.split(grad, [32 * 6, 32, 32 * 32, 32, 3 * 32, 3])
        res[dt] = [t.double().cpu() for t in (nxt, mu, *blocks)]
    names = ("state", "adjoint", "W1", "b1", "W2", "b2", "W3", "b3")
    for name, a, b, tol in zip(names, res[F64], res[F32], [1e-5] + 7 * [3e-4]):
        err, size = (a - b).norm().item(), a.norm().item()
        assert err <= tol * size, (name, err, size)
