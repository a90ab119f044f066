"""Ray hand-out of the trace kernels: every ray is traced exactly once whatever
the rays per wave (16, 32, 64), the length of the runs a wave takes and the
leaves it holds back, and any-hit rays report the first hit of the reference's
traversal order.  Hits are compared bit for bit with the one-lane CPU oracle.
"""
import numpy as np
import pytest

import hippie_amd as hx
from hippie_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene_data():
    v, t = scenes.uniform_soup(3000, seed=31)
    return v, t, scenes.random_rays(300000, seed=32)


def _check(oracle, ctx, bvh, rays, any_hit, launch):
    rb = hx.RayBuffer(rays, closest_hit=not any_hit)
    rb.launch = launch
    rb.results.fill_(0x7F7F7F7F)  # a ray that no wave took keeps this
    res = hx.HipTracer(ctx, bvh).trace(rb).cpu().numpy()
    ref, _ = oracle.trace(bvh.nodes_host(), bvh.woop_host(), bvh.tri_indices_host(), rays, any_hit=any_hit)
    assert np.array_equal(res[:, :2], ref[:, :2])
    hit = res[:, 0] >= 0
    assert np.array_equal(res[hit, 2:], ref[hit, 2:])


# One block per CU is 1024 waves of 256 CUs: 16,384 rays are the most that 16
# rays a wave hold, 32,768 for 32, and above 65,536 waves take further runs.
@pytest.mark.parametrize("blocks", [0, 1])
@pytest.mark.parametrize("count", [1, 15, 17, 63, 64, 65, 257, 16384, 16385, 32768, 32769, 65537, 131073, 262145, 300000])
def test_ray_counts(oracle, ctx, scene_data, blocks, count):
    v, t, rays = scene_data
    bvh = hx.LBVHBuilder(ctx, morton_bits=60).build(hx.Scene(v, t))
    _check(oracle, ctx, bvh, rays[:count], False, {"trace_blocks_per_cu": blocks})


@pytest.mark.parametrize("postpone", [1, 2, 3, 4])
@pytest.mark.parametrize("ahead", [1, 2])
def test_any_hit_order(oracle, ctx, scene_data, postpone, ahead):
    v, t, rays = scene_data
    bvh = hx.LBVHBuilder(ctx, morton_bits=60).build(hx.Scene(v, t))
    _check(oracle, ctx, bvh, rays[:70001], True, {"trace_postpone": postpone, "trace_woop_ahead": ahead})


@pytest.mark.parametrize("layout", ["quad", "oct"])
@pytest.mark.parametrize("count", [1, 17, 65, 16385, 131073, 262145])
def test_wide_ray_counts(ctx, scene_data, layout, count):
    v, t, rays = scene_data
    out = []
    for lay in ("bin", layout):
        bvh = hx.LBVHBuilder(ctx, morton_bits=60, layout=lay).build(hx.Scene(v, t))
        rb = hx.RayBuffer(rays[:count])
        rb.launch = {"trace_blocks_per_cu": 1}
        out.append(hx.HipTracer(ctx, bvh).trace(rb).cpu().numpy())
    assert np.array_equal(*out)
