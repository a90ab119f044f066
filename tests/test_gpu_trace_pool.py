"""Ray hand-out of the trace kernels: every ray is traced exactly once whatever
the rays per wave (8 to 64), the length of the runs a wave takes and the
leaves it holds back, and any-hit rays report the first hit of the reference's
traversal order.  Hits are compared bit for bit with the one-lane CPU oracle.
"""
import numpy as np
import pytest
import torch

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


def _odd_rays(n, seed):
    """Random rays with the limits a merge of hits has to keep: negative tmin
    (hits behind the origin), empty, infinite and NaN intervals, dead rays."""
    rng = np.random.default_rng(seed)
    r = scenes.random_rays(n, seed=seed).copy()
    k = n // 8
    r[:k, 3] = -2.0
    r[k:2 * k, 7] = np.inf
    r[2 * k:3 * k, 7] = rng.uniform(0.0, 0.6, k)
    r[3 * k:3 * k + 40, 7] = np.nan
    r[3 * k + 40:3 * k + 80, 3] = np.nan
    r[4 * k:4 * k + 100, 7] = -1.0
    r[5 * k:5 * k + 100, 4:7] = 0.0
    return r


# Lanes share rays in the kernel with 16 stack entries in LDS; the one with 24
# does not.  Every triangle is there three times, so equal distances are common.
@pytest.mark.parametrize("n_rays", [1, 8, 65, 1000, 5000, 70000, 150000])
@pytest.mark.parametrize("postpone", [1, 2, 4])
def test_shared_rays_keep_hits(oracle, ctx, n_rays, postpone):
    v, t = scenes.merge(*[scenes.uniform_soup(700, seed=5)] * 3, scenes.ground_grid(12))
    bvh = hx.LBVHBuilder(ctx, morton_bits=60).build(hx.Scene(v, t))
    rays = _odd_rays(n_rays, seed=n_rays)
    out = []
    for depth in (16, 24):
        rb = hx.RayBuffer(rays)
        rb.launch = {"trace_lds_stack": depth, "trace_postpone": postpone}
        rb.results.fill_(0x7F7F7F7F)
        out.append(hx.HipTracer(ctx, bvh).trace(rb).cpu().numpy())
    assert np.array_equal(*out)
    ref, _ = oracle.trace(bvh.nodes_host(), bvh.woop_host(), bvh.tri_indices_host(), rays)
    assert np.array_equal(out[0][:, 0], ref[:, 0])


@pytest.mark.parametrize("sort", [False, True])
def test_shared_rays_deep_tree(oracle, ctx, sort):
    """A tree deeper than the stack's LDS part: entries beyond it are not given away."""
    n = 4000
    v, t = scenes.uniform_soup(n, seed=9)
    v = (v * np.exp2(-np.repeat(np.arange(n) % 19, 3)).astype(np.float32)[:, None]).astype(np.float32)
    bvh = hx.LBVHBuilder(ctx, morton_bits=60, adaptive_leaf_size=0, max_leaf_size=1).build(hx.Scene(v, t))
    rays = scenes.random_rays(20000, seed=10)
    rays[:10000, 4:7] = -rays[:10000, 0:3] / np.linalg.norm(rays[:10000, 0:3], axis=1, keepdims=True)
    rb = hx.RayBuffer(rays)
    tr = hx.HipTracer(ctx, bvh)
    res = (tr.trace_sort(rb) if sort else tr.trace(rb)).cpu().numpy()
    ref, ov = oracle.trace(bvh.nodes_host(), bvh.woop_host(), bvh.tri_indices_host(), rays)
    assert ov == 0 and ctx.overflow_count() == 0
    hit = ref[:, 0] >= 0
    assert np.array_equal(res[:, :2], ref[:, :2]) and np.array_equal(res[hit], ref[hit])


def _point_rays(n, seed, kind):
    """Rays from one point; "half": the second half from anywhere; "dead": every
    second ray's interval is empty; "nan": one ray in 5000 has no origin."""
    r = scenes.random_rays(n, seed=seed)
    k = n // 2 + 1 if kind == "half" else n
    r[:k, 0:3] = (0.5, 0.5, -0.8)
    if kind == "dead":
        r[::2, 7] = -1.0
    if kind == "nan":
        r[::5000, 0] = np.nan
    return r


# Sorted sets from 2 rays a lane slot on (the wide layouts: 4, sorted or not; input
# order: 12) are looked over for rays from one point, which are handed out refill by
# refill and read nodes by scalar loads: sizes around the lines, and sets that are
# only partly alike.
@pytest.mark.parametrize("layout", ["bin", "quad", "oct"])
@pytest.mark.parametrize("sort", [False, True])
@pytest.mark.parametrize("kind, extra", [("point", -1), ("point", 0), ("point", 77), ("half", 1), ("dead", 1), ("nan", 1)])
def test_rays_from_one_point(oracle, ctx, layout, sort, kind, extra):
    slots = torch.cuda.get_device_properties(0).multi_processor_count * 8 * 256
    n = slots * (4 if layout != "bin" else 2 if sort else 12) + extra
    v, t = scenes.uniform_soup(700, seed=41)
    bvh = hx.LBVHBuilder(ctx, morton_bits=60, layout=layout).build(hx.Scene(v, t))
    rays = _point_rays(n, 42, kind)
    rb = hx.RayBuffer(rays)
    rb.results.fill_(0x7F7F7F7F)
    tr = hx.HipTracer(ctx, bvh)
    res = (tr.trace_sort(rb) if sort else tr.trace(rb)).cpu().numpy()
    b = hx.LBVHBuilder(ctx, morton_bits=60).build(hx.Scene(v, t))
    ref, _ = oracle.trace(b.nodes_host(), b.woop_host(), b.tri_indices_host(), rays)
    assert np.array_equal(res[:, :2], ref[:, :2])
    hit = ref[:, 0] >= 0
    assert hit.any() and np.array_equal(res[hit], ref[hit])


@pytest.mark.parametrize("sort, per_slot", [(True, 4), (False, 12)])
def test_any_hit_rays_from_one_point(oracle, ctx, sort, per_slot):
    """Handed out refill by refill, any-hit rays still report the first hit of the
    reference's traversal order."""
    n = torch.cuda.get_device_properties(0).multi_processor_count * 8 * 256 * per_slot + 3
    v, t = scenes.uniform_soup(700, seed=43)
    bvh = hx.LBVHBuilder(ctx, morton_bits=60).build(hx.Scene(v, t))
    rays = _point_rays(n, 44, "point")
    rb = hx.RayBuffer(rays, closest_hit=False)
    rb.results.fill_(0x7F7F7F7F)
    tr = hx.HipTracer(ctx, bvh)
    res = (tr.trace_sort(rb) if sort else tr.trace(rb)).cpu().numpy()
    ref, _ = oracle.trace(bvh.nodes_host(), bvh.woop_host(), bvh.tri_indices_host(), rays, any_hit=True)
    hit = ref[:, 0] >= 0
    assert np.array_equal(res[:, :2], ref[:, :2]) and np.array_equal(res[hit], ref[hit])
