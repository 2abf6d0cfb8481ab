"""The several-step kernel for 2D grids (csrc/lbm_tile2d.hip) against single
steps: periodic D2Q9 grids and channels with every boundary rule, extents
that are no multiple of the tile, the smallest extents a tile's halo fits,
both streaming orders, every storage format and both memory layouts.  Without
collision the streaming and the boundary rules must agree bit for bit;
otherwise to the rounding of the collision arithmetic, which the compiler may
contract differently in the two kernels (a few units in the last place of the
stored format per step)."""
import numpy as np
import pytest
import torch

import lettuce_amd as lt
from tests.test_parity_gpu import ArrayFlow
from tests.test_two_step_2d_gpu import COLLISIONS, ULPS, _channel, _periodic_f0

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64
PRE, POST = lt.StreamingStrategy.PRE_STREAMING, lt.StreamingStrategy.POST_STREAMING
TOL = dict(ULPS, f64=4 * 0.5 * 2.0 ** -52)


def _bits(flow):
    return flow._state.detach().cpu().contiguous().view(-1).view(torch.uint8).numpy()


def _compare(make, storage, coll, strategy, depth, tile, knobs, counts=(3, 4, 11, 14)):
    """`make()` gives a fresh flow; several-step launches against single steps"""
    for steps in counts:
        out = []
        for multi in (False, True):
            knobs(two_step=1 if multi else 0)
            knobs(multi_step=2, multi_step_depth=depth, multi_step_tile1=tile[0],
                  multi_step_tile2=tile[1])
            flow = make()
            sim = lt.Simulation(flow, COLLISIONS[coll](flow.units.relaxation_parameter_lu
                                                       if coll != "trt" else 0.7), [], strategy)
            several, two, single = sim._collide_and_stream.launches(steps)
            assert two == 0 and (several > 0) == multi, (several, two, single)
            assert (several + single - steps) % 2 == 0
            sim(steps)
            torch.cuda.synchronize()
            out.append((_bits(flow), flow.f.double().cpu().numpy()))
        if coll == "none":
            assert np.array_equal(out[0][0], out[1][0]), steps
        else:
            err = np.abs(out[0][1] - out[1][1]).max()
            tol = steps * TOL[storage] * (50 if coll == "kbc" else 1)
            assert err <= tol, (steps, err, tol)


@pytest.mark.parametrize("storage,layout,nx,ny,coll,depth,tile", [
    ("f32", "soa", 40, 64, "bgk", 4, (8, 16)),
    ("f32", "rows", 37, 131, "kbc", 3, (16, 32)),
    ("f64", "soa", 53, 29, "none", 5, (8, 8)),
    ("f64", "rows", 41, 50, "trt", 10, (8, 8)),
    ("f16_shifted", "soa", 33, 47, "none", 6, (12, 16)),
    ("bf16_shifted", "rows", 64, 40, "bgk", 2, (32, 32)),
    # the halo reaches once around the grid: tile + halo = extent
    ("f32", "soa", 11, 19, "none", 4, (8, 16)),
    # one tile, with cells past the grid's end
    ("f32", "soa", 9, 10, "bgk", 2, (8, 8))])
@pytest.mark.parametrize("strategy", [PRE, POST])
def test_periodic(storage, layout, nx, ny, coll, depth, tile, strategy, knobs):
    f0 = _periodic_f0(nx, ny)
    dtype = F64 if storage == "f64" else F32

    def make():
        ctx = lt.Context("cuda:0", dtype=dtype, storage=storage, layout=layout)
        return ArrayFlow(ctx, f0, lt.D2Q9())
    _compare(make, storage, coll, strategy, depth, tile, knobs)


@pytest.mark.parametrize("storage,nx,ny,outlet,solid,coll,depth,tile", [
    ("f32", 61, 45, "equilibrium", "halfway", "none", 4, (8, 16)),
    ("f32", 50, 64, "antibounceback", "fullway", "none", 3, (16, 16)),
    ("f32", 70, 51, "antibounceback", "halfway", "bgk", 5, (8, 32)),
    ("f64", 48, 40, "equilibrium", "fullway", "trt", 4, (8, 8)),
    ("f16_shifted", 64, 35, "equilibrium", "halfway", "kbc", 2, (24, 32)),
    ("bf16_shifted", 47, 96, "antibounceback", "halfway", "bgk", 6, (8, 16)),
    # a tile's halo spans inlet, outlet and walls at once
    ("f32", 24, 24, "equilibrium", "halfway", "none", 5, (16, 16))])
@pytest.mark.parametrize("strategy", [PRE, POST])
def test_channel(storage, nx, ny, outlet, solid, coll, depth, tile, strategy, knobs):
    def make():
        return _channel(None if storage == "f64" else storage, nx, ny, outlet, solid,
                        walls=outlet == "equilibrium" and solid == "halfway",
                        dtype=F64 if storage == "f64" else F32)
    _compare(make, storage, coll, strategy, depth, tile, knobs)


@pytest.mark.parametrize("strategy", [PRE, POST])
def test_stochastic_rounding_draws_the_same_bits(strategy, knobs):
    """BF16 storage rounded stochastically, without collision: the stored
    values of every step carry that step's bits, so the runs agree bit for
    bit (the post order keeps single launches at its ends)"""
    f0 = _periodic_f0(37, 41)
    out = []
    for multi in (False, True):
        knobs(two_step=1 if multi else 0)
        knobs(multi_step=2, multi_step_depth=4, multi_step_tile1=8, multi_step_tile2=16)
        flow = ArrayFlow(lt.Context("cuda:0", dtype=F32, storage="bf16_shifted",
                                    rounding="stochastic", rounding_seed=5), f0, lt.D2Q9())
        sim = lt.Simulation(flow, lt.NoCollision(), [], strategy)
        several, _, single = sim._collide_and_stream.launches(14)
        assert (several > 0) == multi and single == (0 if multi and strategy == PRE else
                                                     2 if multi else 14)
        sim(14)
        out.append(_bits(flow))
    assert np.array_equal(out[0], out[1])


def test_default_selection(knobs):
    """small grids of any extents run several steps per launch, grids smaller
    than a tile and its halo run single steps, and the row-sweeping kernel
    keeps the large channel"""
    def launches(flow, steps, strategy=PRE):
        sim = lt.Simulation(flow, lt.BGKCollision(0.6), [], strategy)
        return sim._collide_and_stream.launches(steps)
    ctx = lt.Context("cuda:0", dtype=F64)
    several, two, single = launches(ArrayFlow(ctx, _periodic_f0(251, 187), lt.D2Q9()), 200)
    assert 20 <= several <= 70 and two == 0 and single == 0
    several, two, single = launches(_channel("f32", 250, 125, "antibounceback", "fullway",
                                             walls=False), 200, POST)
    assert 20 <= several <= 100 and two == 0 and single == 0
    assert launches(ArrayFlow(ctx, _periodic_f0(5, 6), lt.D2Q9()), 10) == (0, 0, 10)
    assert launches(_channel("f32", 2048, 512, "equilibrium", "halfway"), 100) == (0, 50, 0)


@pytest.mark.parametrize("strategy", [PRE, POST])
def test_depth_of_one_step_leaves_the_kernel_out(strategy, knobs):
    """one step per launch: nothing for the kernel to fuse, and no launch
    without a stage (a post-order run has one stage more than steps)"""
    f0 = _periodic_f0(40, 50)
    for steps in (2, 3, 4, 7):
        out = []
        for depth in (1, 0):
            knobs(multi_step=2 if depth else 0, multi_step_depth=depth, two_step=1 if depth else 0)
            flow = ArrayFlow(lt.Context("cuda:0", dtype=F64), f0, lt.D2Q9())
            sim = lt.Simulation(flow, lt.NoCollision(), [], strategy)
            assert sim._collide_and_stream.launches(steps) == (0, 0, steps)
            sim(steps)
            out.append(_bits(flow))
        assert np.array_equal(out[0], out[1]), steps


@pytest.mark.parametrize("storage,nx,ny,coll,order,tiles,rows", [
    # small, or bound by memory: several steps per launch
    ("f32", 128, 128, "bgk", POST, True, False), ("f64", 1024, 1024, "bgk", PRE, True, False),
    ("f32", 700, 701, "kbc", PRE, True, False), ("f16_shifted", 512, 512, "kbc", PRE, True, False),
    # bound by arithmetic, which the tiles' overlap adds to: without it
    ("f16_shifted", 1500, 1100, "kbc", POST, False, False),
    ("f16_shifted", 3072, 4096, "kbc", PRE, False, False),
    ("f32", 4096, 256, "kbc", PRE, False, True), ("f32", 8192, 128, "kbc", PRE, False, True)])
def test_tiles_only_where_they_are_faster(storage, nx, ny, coll, order, tiles, rows):
    flow = lt.TaylorGreenVortex(
        lt.Context("cuda:0", dtype=F64 if storage == "f64" else F32, storage=storage),
        [nx, ny], 100, 0.05, lt.D2Q9())
    sim = lt.Simulation(flow, COLLISIONS[coll](0.6), [], order)
    several, two, single = sim._collide_and_stream.launches(40)
    assert (several > 0, two > 0) == (tiles, rows), (several, two, single)


def test_arrays_past_the_caches(knobs):
    """two arrays of 201 MB, whose stores bypass the caches, bit for bit"""
    f0 = _periodic_f0(1181, 1181)

    def make():
        return ArrayFlow(lt.Context("cuda:0", dtype=F64), f0, lt.D2Q9())
    _compare(make, "f64", "none", PRE, 3, (16, 32), knobs, counts=(4, 5))
