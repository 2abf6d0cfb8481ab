"""GPU checks of the enstrophy sum: whole-grid FP64 differences by torch.roll
on the CPU against lbm_enstrophy_f64, on extents below the stencil's width,
odd ones, and planes of more tiles than blocks."""
import ctypes

import pytest
import torch

from lettuce_amd import _native as N

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _d6(u, dim):
    return sum(w * (u.roll(-k, dim) - u.roll(k, dim))
               for k, w in ((1, 3 / 4), (2, -3 / 20), (3, 1 / 60)))


@pytest.mark.parametrize("shape", [
    (1, 1), (2, 3), (251, 187), (1030, 1024),
    (1, 1, 1), (2, 3, 5), (3, 1, 300), (7, 33, 9), (64, 64, 64), (130, 31, 17), (3, 1024, 520)])
def test_enstrophy_matches_rolled_differences(shape):
    # each difference is exact to a few roundings of values of order 1 and
    # the sum has positive terms only: relative error well below 1e-12
    g = torch.Generator().manual_seed(sum(shape))
    u = torch.rand((len(shape),) + shape, generator=g, dtype=torch.float64) - 0.5
    w = _d6(u[0], 1) - _d6(u[1], 0)
    ref = (w * w).sum()
    if len(shape) == 3:
        for w in (_d6(u[2], 1) - _d6(u[1], 2), _d6(u[0], 2) - _d6(u[2], 0)):
            ref += (w * w).sum()
    n = (ctypes.c_int64 * 3)(*((1,) * (3 - len(shape)) + shape))
    lib = N.lib()
    ud = u.to(DEV).contiguous()
    ws = torch.empty(lib.lbm_reduce_workspace_bytes(n), dtype=torch.uint8, device=DEV)
    out = torch.full((1,), -1.0, dtype=torch.float64, device=DEV)
    N.check(lib.lbm_enstrophy_f64(N.D2Q9 if len(shape) == 2 else N.D3Q19, n, ud.data_ptr(),
                                  out.data_ptr(), ws.data_ptr(), N.stream_handle(DEV)),
            "lbm_enstrophy_f64")
    assert abs(out.item() - ref.item()) <= 1e-12 * ref.item()
