"""The row-sweeping two-step kernel for 2D grids (csrc/lbm_tb2d.hip) with the
several-step kernel, which takes small grids by default, left out: the cases
of test_two_step_2d_gpu, with plan() giving the launches that are made, and
captured graphs of both kernels."""
import pytest
import torch

import lettuce_amd as lt
from lettuce_amd._simulation import NativeStep
from tests import test_graph_gpu as G
from tests import test_two_step_2d_gpu as T

pytestmark = pytest.mark.gpu

PRE, POST = T.PRE, T.POST


@pytest.fixture
def rows_only(knobs, monkeypatch):
    def plan(self, nsteps):
        several, two, single = self.launches(nsteps)
        assert several == 0
        return two, single
    knobs(multi_step=0)
    monkeypatch.setattr(NativeStep, "plan", plan)
    return knobs


@pytest.mark.parametrize("storage,nx,ny,outlet,solid,coll,planes", [c for c in T.CASES if c[-1] == 0])
@pytest.mark.parametrize("strategy", [PRE, POST])
def test_channel(storage, nx, ny, outlet, solid, coll, planes, strategy, rows_only):
    T.test_two_step_2d_matches_single_steps(storage, nx, ny, outlet, solid, coll, planes, strategy,
                                            rows_only)


@pytest.mark.parametrize("storage,layout,nx,ny,coll", [
    ("f32", "soa", 40, 64, "bgk"), ("f32", "rows", 37, 128, "kbc"),
    ("f32", "soa", 24, 640, "trt"), ("f16_shifted", "soa", 33, 512, "bgk"),
    ("bf16_shifted", "rows", 20, 256, "none"), ("f32", "soa", 16, 128, "none")])
def test_periodic(storage, layout, nx, ny, coll, rows_only):
    T.test_two_step_2d_periodic_matches_single_steps(storage, layout, nx, ny, coll, rows_only)


@pytest.mark.parametrize("strategy", ["PRE_STREAMING", "POST_STREAMING"])
def test_channel_vs_oracle(strategy, rows_only):
    T.test_two_step_2d_channel_vs_oracle(strategy)


def test_default_obstacle_vs_oracle(rows_only):
    T.test_two_step_2d_default_obstacle_vs_oracle()


def test_stochastic_rounding(rows_only):
    T.test_two_step_2d_with_stochastic_rounding(rows_only)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_equilibrium_boundary_field_vs_oracle(dtype, rows_only):
    T.test_two_step_2d_equilibrium_boundary_field_vs_oracle(dtype, rows_only)


@pytest.mark.parametrize("multi_step,launches", [(0, (0, 2, 0)), (2, (2, 0, 0))])
def test_captured_steps_replay_like_eager_steps(multi_step, launches, knobs):
    knobs(multi_step=multi_step, multi_step_depth=2)
    flow, coll, _ = G._case("d2q9_kbc_channel_two_step")
    assert lt.Simulation(flow, coll, [], PRE)._collide_and_stream.launches(4) == launches
    G.test_captured_steps_replay_like_eager_steps("d2q9_kbc_channel_two_step")


def test_captured_run_in_the_default_order(knobs):
    """the several-step kernel with its first and last stages: 4 steps"""
    knobs(multi_step=2, multi_step_depth=3)
    flows = [G._case("d2q9_kbc_channel_two_step")[0] for _ in range(2)]
    flows[1]._state.copy_(flows[0]._state)
    sims = [lt.Simulation(f, lt.BGKCollision(0.6), [], POST) for f in flows]
    assert sims[0]._collide_and_stream.launches(4) == (2, 0, 0)
    graph = G._capture(sims[0], 4)
    for replay in range(3):
        graph.replay()
        sims[1](4)
        torch.cuda.synchronize()
        assert torch.equal(flows[0]._state, flows[1]._state), replay
