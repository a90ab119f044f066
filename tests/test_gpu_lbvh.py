"""GPU parity of the LBVH build (libhx through the C ABI) against the CPU oracle.

Bit-exact: Morton keys, sorted order, Karras left/right/parent, binary boxes,
the collapsed Bin tree in canonical DFS form, Woop rows.  FP64-summed SAH
cost within 1e-9 relative.
"""
import numpy as np
import pytest
import torch

import hippie_amd as hx
from hippie_amd import scenes

pytestmark = pytest.mark.gpu


def _area(b):
    d = b[3:6] - b[0:3]
    return float(np.float32(2.0) * (d[0] * d[1] + d[1] * d[2] + d[2] * d[0]))


def _oracle_build(oracle, v, t, bits, adaptive=True, max_leaf=8):
    sb = oracle.scene_box(v, t)
    bmin, bmax = oracle.setup_boxes(v, t)
    keys = oracle.morton_codes(bmin, bmax, sb, bits)
    sk, sv = oracle.sort_pairs(keys, np.arange(t.shape[0], dtype=np.int32), bits)
    left, right, parent = oracle.construct(sk)
    nmin, nmax = oracle.refit(sv, bmin, bmax, left, right, parent)
    nodes, tri, ni, nl = oracle.collapse(sv, left, right, parent, nmin, nmax, adaptive, max_leaf)
    woop = oracle.woopify(v, t, tri)
    return dict(sb=sb, keys=keys, sorted_keys=sk, sorted_tri=sv, left=left, right=right, parent=parent,
                nmin=nmin, nmax=nmax, nodes=nodes, tri=tri, n_interior=ni, n_leaves=nl, woop=woop)


def _gpu_build(ctx, v, t, bits, adaptive=True, max_leaf=8):
    scene = hx.Scene(v, t)
    b = hx.LBVHBuilder(ctx, morton_bits=bits, adaptive_leaf_size=int(adaptive), max_leaf_size=max_leaf,
                       keep_debug=1)
    bvh = b.build(scene)
    return scene, bvh


def _check_build(oracle, ctx, v, t, bits, adaptive=True, max_leaf=8, check_binary=True):
    ref = _oracle_build(oracle, v, t, bits, adaptive, max_leaf)
    scene, bvh = _gpu_build(ctx, v, t, bits, adaptive, max_leaf)
    n = t.shape[0]
    assert np.array_equal(bvh.scene_box(), ref["sb"]), "scene box"
    dbg = bvh.debug_host()
    assert np.array_equal(dbg["sorted_keys"], ref["sorted_keys"]), "sorted Morton keys"
    assert np.array_equal(dbg["sorted_tri"], ref["sorted_tri"]), "sorted order"
    if check_binary and n > 1:
        # The GPU numbers internal nodes by split position (the last leaf of
        # the left child); a Karras node's left child index is that position.
        L, R, P = ref["left"][: n - 1], ref["right"][: n - 1], ref["parent"]
        split = np.where(L < n - 1, L, L - (n - 1))
        assert np.array_equal(np.sort(split), np.arange(n - 1)), "split positions"
        node = np.concatenate([split, np.arange(n - 1, 2 * n - 1)])  # Karras index -> GPU index
        assert np.array_equal(dbg["left"][split], node[L]), "Karras left"
        assert np.array_equal(dbg["right"][split], node[R]), "Karras right"
        assert np.array_equal(dbg["parent"][node], np.where(P < 0, -1, node[np.maximum(P, 0)])), "Karras parent"
        for k in ("min", "max"):
            got = dbg["node_" + k][node][:, :3].view(np.uint32)
            assert np.array_equal(got, ref["n" + k][:, :3].view(np.uint32)), "box " + k
    nodes = bvh.nodes_host()
    tri = bvh.tri_indices_host()
    assert bvh.n_interior == ref["n_interior"] and bvh.n_leaves == ref["n_leaves"], "node counts"
    assert oracle.validate_bin(nodes, bvh.n_interior, bvh.n_leaves, tri, v, t) == 0, "validate"
    cg = oracle.bin_canonical(nodes, bvh.n_interior, bvh.n_leaves, tri)
    co = oracle.bin_canonical(ref["nodes"], ref["n_interior"], ref["n_leaves"], ref["tri"])
    assert np.array_equal(cg, co), "canonical Bin tree"
    woop = bvh.woop_host()
    assert np.array_equal(woop.view(np.uint32), oracle.woopify(v, t, tri).view(np.uint32)), "Woop rows"
    return ref, scene, bvh, nodes, tri, woop


@pytest.mark.parametrize("bits", [30, 60])
def test_lbvh_config1_shape(oracle, ctx, bits):
    """65,536-triangle uniform soup (config 1 geometry) at 30 and 60 bits."""
    v, t = scenes.uniform_soup(65536, seed=1)
    ref, scene, bvh, nodes, tri, woop = _check_build(oracle, ctx, v, t, bits)
    sa = _area(ref["sb"])
    c_gpu = bvh.get_cost()
    c_ref = oracle.cost(ref["nodes"], sa)
    assert abs(c_gpu - c_ref) <= 1e-9 * abs(c_ref)


@pytest.mark.parametrize("n", [2, 3, 5, 17, 64, 65, 1000, 4097])
def test_lbvh_small_sizes(oracle, ctx, n):
    v, t = scenes.uniform_soup(n, seed=10 + n)
    _check_build(oracle, ctx, v, t, 60)


def test_lbvh_single_triangle(oracle, ctx):
    v, t = scenes.uniform_soup(1, seed=3)
    ref, scene, bvh, nodes, tri, woop = _check_build(oracle, ctx, v, t, 60, check_binary=False)
    assert bvh.n_interior == 1 and bvh.n_leaves == 1


def test_lbvh_duplicate_keys(oracle, ctx):
    """All centroids equal: every Morton key ties; Karras ties break on index."""
    rng = np.random.default_rng(7)
    n = 3000
    base = np.array([[0.2, 0.3, 0.4], [0.25, 0.3, 0.4], [0.2, 0.35, 0.45]], np.float32)
    v = np.tile(base, (n, 1)).astype(np.float32)
    t = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    # one outlier so the scene box is not degenerate
    v[-3:] += np.float32(0.5)
    _check_build(oracle, ctx, v, t, 60)
    _check_build(oracle, ctx, v, t, 30)
    del rng


def test_lbvh_indexed_grid_and_degenerate(oracle, ctx):
    """Shared-vertex grid (flat in y) plus zero-area triangles."""
    gv, gt = scenes.ground_grid(40)
    dv = np.repeat(np.array([[0.5, 0.5, 0.5]], np.float32), 30, axis=0)
    dt = np.arange(30, dtype=np.int32).reshape(10, 3)
    v, t = scenes.merge((gv, gt), (dv, dt))
    _check_build(oracle, ctx, v, t, 60)


@pytest.mark.parametrize("max_leaf", [1, 4, 8])
def test_lbvh_fixed_leaf_size(oracle, ctx, max_leaf):
    v, t = scenes.uniform_soup(20000, seed=4)
    _check_build(oracle, ctx, v, t, 60, adaptive=False, max_leaf=max_leaf)


def test_lbvh_gaussian_mixture(oracle, ctx):
    v, t = scenes.config2_scene(n_mixture=50000, grid_cells=100, seed=2)
    _check_build(oracle, ctx, v, t, 60)


def test_rebuild_matches_build(oracle, ctx):
    v, t = scenes.uniform_soup(5000, seed=8)
    scene = hx.Scene(v, t)
    builder = hx.LBVHBuilder(ctx, morton_bits=60)
    bvh = builder.build(scene)
    a = oracle.bin_canonical(bvh.nodes_host(), bvh.n_interior, bvh.n_leaves, bvh.tri_indices_host())
    v2, t2 = scenes.uniform_soup(5000, seed=9)
    scene2 = hx.Scene(v2, t2)
    builder.rebuild(bvh, scene2)
    builder.rebuild(bvh, scene)
    b = oracle.bin_canonical(bvh.nodes_host(), bvh.n_interior, bvh.n_leaves, bvh.tri_indices_host())
    assert np.array_equal(a, b)


def test_morton_stage_entry(oracle, ctx):
    v, t = scenes.uniform_soup(10000, seed=12)
    scene = hx.Scene(v, t)
    box = hx.scene_box(ctx, scene)
    sb = oracle.scene_box(v, t)
    assert np.array_equal(box.cpu().numpy(), sb)
    bmin, bmax = oracle.setup_boxes(v, t)
    for bits in (6, 30, 45, 60):
        keys = hx.morton_codes(ctx, scene, box, bits).cpu().numpy().view(np.uint64)
        assert np.array_equal(keys, oracle.morton_codes(bmin, bmax, sb, bits)), bits


@pytest.mark.parametrize("n", [1, 2, 100, 4095, 4096, 4097, 100000, 1 << 20])
@pytest.mark.parametrize("kind", ["random", "dups", "sorted", "reversed", "equal"])
def test_sort_pairs(ctx, n, kind):
    rng = np.random.default_rng(n)
    bits = 60
    if kind == "random":
        k = rng.integers(0, 1 << bits, n, dtype=np.uint64)
    elif kind == "dups":
        k = rng.integers(0, 50, n, dtype=np.uint64) << np.uint64(20)
    elif kind == "sorted":
        k = np.sort(rng.integers(0, 1 << bits, n, dtype=np.uint64))
    elif kind == "reversed":
        k = np.sort(rng.integers(0, 1 << bits, n, dtype=np.uint64))[::-1].copy()
    else:
        k = np.full(n, 12345, np.uint64)
    vals = rng.permutation(n).astype(np.int32)
    kt = torch.from_numpy(k.view(np.int64).copy()).cuda()
    vt = torch.from_numpy(vals.copy()).cuda()
    hx.sort_pairs(ctx, kt, vt, bits)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(kt.cpu().numpy().view(np.uint64), k[order])
    assert np.array_equal(vt.cpu().numpy(), vals[order])


@pytest.mark.parametrize("run,limit", [(1, 64), (7, 64), (64, 64), (65, 64), (9, 8), (2, 1), (40, 2048), (1500, 2048)])
def test_sort_split_runs(ctx, run, limit):
    """Sorts of 60-bit keys with at least 2^18 keys rank each run of equal
    high 32 bits in place when no run exceeds sort_local_run keys, and run the
    low digit passes otherwise: both give the stable order, ties included."""
    n = 300007
    rng = np.random.default_rng(run * 1000 + limit)
    high = np.repeat(rng.integers(0, 1 << 32, n // run + 1, dtype=np.uint64), run)[:n]
    low = rng.integers(0, 4, n, dtype=np.uint64) * np.uint64(1 << 26) + rng.integers(0, 3, n, dtype=np.uint64)
    k = (high << np.uint64(28)) | low
    perm = rng.permutation(n)
    k = k[perm]
    vals = rng.permutation(n).astype(np.int32)
    old = ctx.get_tuning("sort_local_run")
    ctx.set_tuning("sort_local_run", limit)
    try:
        kt = torch.from_numpy(k.view(np.int64).copy()).cuda()
        vt = torch.from_numpy(vals.copy()).cuda()
        hx.sort_pairs(ctx, kt, vt, 60)
    finally:
        ctx.set_tuning("sort_local_run", old)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(kt.cpu().numpy().view(np.uint64), k[order])
    assert np.array_equal(vt.cpu().numpy(), vals[order])


@pytest.mark.parametrize("end_bit", [40, 52, 60, 63])
def test_sort_split_ignores_bits_above_end_bit(ctx, end_bit):
    """Key bits at and above end_bit are not part of the sort key: junk there
    must not split a run of equal [lo_bit, end_bit) bits in the local pass."""
    n = 300007
    rng = np.random.default_rng(end_bit)
    mask = np.uint64((1 << end_bit) - 1)
    k = rng.integers(0, 1 << 20, n, dtype=np.uint64) << np.uint64(end_bit - 20)
    k |= rng.integers(0, 4, n, dtype=np.uint64)
    junk = rng.integers(0, 1 << (64 - end_bit), n, dtype=np.uint64) << np.uint64(end_bit)
    kj = k | junk
    vals = rng.permutation(n).astype(np.int32)
    kt = torch.from_numpy(kj.view(np.int64).copy()).cuda()
    vt = torch.from_numpy(vals.copy()).cuda()
    hx.sort_pairs(ctx, kt, vt, end_bit)
    order = np.argsort(kj & mask, kind="stable")
    assert np.array_equal(vt.cpu().numpy(), vals[order])
    assert np.array_equal(kt.cpu().numpy().view(np.uint64), kj[order])


def test_lbvh_split_sort_off(oracle, ctx):
    """The LBVH build with every digit pass (sort_local_run 0) and with the
    split sort gives the same tree."""
    v, t = scenes.config2_scene(n_mixture=200000, grid_cells=256, seed=9)
    old = ctx.get_tuning("sort_local_run")
    try:
        ctx.set_tuning("sort_local_run", 0)
        _check_build(oracle, ctx, v, t, 60)
    finally:
        ctx.set_tuning("sort_local_run", old)
    _check_build(oracle, ctx, v, t, 60)


@pytest.mark.parametrize("end_bit", [4, 13, 30, 33, 64])
def test_sort_pairs_bit_ranges(ctx, end_bit):
    n = 50000
    rng = np.random.default_rng(end_bit)
    hi = np.uint64((1 << end_bit) - 1) if end_bit < 64 else np.uint64(0xFFFFFFFFFFFFFFFF)
    k = rng.integers(0, 1 << 63, n, dtype=np.uint64) & hi
    vals = np.arange(n, dtype=np.int32)
    kt = torch.from_numpy(k.view(np.int64).copy()).cuda()
    vt = torch.from_numpy(vals.copy()).cuda()
    hx.sort_pairs(ctx, kt, vt, end_bit)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(vt.cpu().numpy(), vals[order])


@pytest.fixture
def digits10(ctx):
    """Run a test with 10-bit radix digits, restoring the default after."""
    old = ctx.get_tuning("sort_digit_bits")
    ctx.set_tuning("sort_digit_bits", 10)
    yield ctx
    ctx.set_tuning("sort_digit_bits", old)


@pytest.mark.parametrize("n", [2, 4097, 300000])
@pytest.mark.parametrize("end_bit", [13, 30, 60, 64])
def test_sort_pairs_10bit_digits(digits10, n, end_bit):
    ctx = digits10
    rng = np.random.default_rng(n + end_bit)
    hi = np.uint64((1 << end_bit) - 1) if end_bit < 64 else np.uint64(0xFFFFFFFFFFFFFFFF)
    k = rng.integers(0, 1 << 63, n, dtype=np.uint64) & hi
    k[: n // 3] = k[0]  # duplicates
    vals = rng.permutation(n).astype(np.int32)
    kt = torch.from_numpy(k.view(np.int64).copy()).cuda()
    vt = torch.from_numpy(vals.copy()).cuda()
    hx.sort_pairs(ctx, kt, vt, end_bit)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(kt.cpu().numpy().view(np.uint64), k[order])
    assert np.array_equal(vt.cpu().numpy(), vals[order])


@pytest.mark.parametrize("bits", [30, 60])
def test_lbvh_10bit_digits(oracle, digits10, bits):
    v, t = scenes.gaussian_mixture_soup(100000, seed=bits)
    _check_build(oracle, digits10, v, t, bits)


@pytest.mark.parametrize("digits,items,lookback", [(d, i, lb) for d in (8, 10) for i in (8, 16, 32) for lb in (4, 8, 16)
                                                   if (d, i, lb) != (8, 16, 4)])
def test_sort_pairs_keys_per_thread(ctx, digits, items, lookback):
    """Every (digit width, keys per thread, look-back width) gives the stable order."""
    old = (ctx.get_tuning("sort_digit_bits"), ctx.get_tuning("sort_items"), ctx.get_tuning("sort_lookback"))
    ctx.set_tuning("sort_digit_bits", digits)
    ctx.set_tuning("sort_items", items)
    ctx.set_tuning("sort_lookback", lookback)
    try:
        for n, end_bit in ((5000, 30), (1000003, 60), (2, 64)):
            rng = np.random.default_rng(n + items)
            hi = np.uint64((1 << end_bit) - 1) if end_bit < 64 else np.uint64(0xFFFFFFFFFFFFFFFF)
            k = rng.integers(0, 1 << 63, n, dtype=np.uint64) & hi
            k[: n // 3] = k[0]
            vals = rng.permutation(n).astype(np.int32)
            kt = torch.from_numpy(k.view(np.int64).copy()).cuda()
            vt = torch.from_numpy(vals.copy()).cuda()
            hx.sort_pairs(ctx, kt, vt, end_bit)
            order = np.argsort(k, kind="stable")
            assert np.array_equal(kt.cpu().numpy().view(np.uint64), k[order])
            assert np.array_equal(vt.cpu().numpy(), vals[order])
    finally:
        ctx.set_tuning("sort_digit_bits", old[0])
        ctx.set_tuning("sort_items", old[1])
        ctx.set_tuning("sort_lookback", old[2])


def test_lbvh_sort_32_keys_per_thread(oracle, ctx):
    old = ctx.get_tuning("sort_items")
    ctx.set_tuning("sort_items", 32)
    try:
        v, t = scenes.gaussian_mixture_soup(200000, seed=5)
        _check_build(oracle, ctx, v, t, 60)
    finally:
        ctx.set_tuning("sort_items", old)


@pytest.mark.parametrize("seed", [1, 2])
def test_normalize_vertices_matches_oracle(oracle, ctx, seed):
    rng = np.random.default_rng(seed)
    v = (rng.normal(size=(100003, 3)) * np.array([0.3, 4.0, 1.5]) + 7.0).astype(np.float32)
    ref, rbox = oracle.normalize(v)
    vt = torch.from_numpy(v.copy()).cuda()
    box = hx.normalize_vertices(ctx, vt).cpu().numpy()
    assert np.array_equal(box, rbox)
    assert np.array_equal(vt.cpu().numpy().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("adaptive,max_leaf", [(True, 8), (False, 4), (False, 40)])
def test_leaf_stats(oracle, ctx, adaptive, max_leaf):
    """HipBVH::getAvgLeafSize / getLeafSizeHistogram inputs from the Bin leaves."""
    v, t = scenes.gaussian_mixture_soup(50000, seed=21)
    scene, bvh = _gpu_build(ctx, v, t, 60, adaptive, max_leaf)
    nodes = bvh.nodes_host()
    sizes = ~nodes[bvh.n_interior:bvh.n_interior + bvh.n_leaves, 14]
    hist, total = bvh.leaf_stats()
    assert total == sizes.sum() == t.shape[0]
    assert np.array_equal(hist, np.bincount(sizes[sizes <= 32], minlength=33)[:33])
    assert abs(bvh.avg_leaf_size() - t.shape[0] / bvh.n_leaves) < 1e-9


@pytest.mark.gpu
@pytest.mark.parametrize("method,presplit", [("lbvh", 0), ("ploc", 0), ("atr", 0), ("hlbvh", 0), ("insertion", 0),
                                             ("lbvh", 1)])
def test_validate(oracle, ctx, method, presplit):
    """HipBVH::validate on the device agrees with the oracle's validation of the same nodes."""
    v, t = scenes.merge(scenes.gaussian_mixture_soup(4000, seed=5), scenes.ground_grid(3))
    scene = hx.Scene(v, t)
    p = hx.BuildParams.from_env({"Bvh.method": method})
    p.presplitting, p.presplitter_beta = presplit, 0.3
    bvh = hx.BVHBuilder(ctx, params=p).build(scene)
    assert bvh.validate() == 0
    nodes, tri_idx = bvh.nodes_host(), bvh.tri_indices_host()
    assert oracle.validate_bin_refs(nodes, bvh.n_interior, bvh.n_leaves, tri_idx, v, t) == 0
    # Geometry moved after the build without a refit: the leaf boxes miss their
    # triangles and nothing else fails; a refit makes the BVH valid again.
    moved = hx.Scene(v + np.float32(100.0), t)
    bvh.update(moved)
    assert bvh.validate() == 0
    moved.vertices += 50.0
    assert bvh.validate() == 16
    bvh.update()
    assert bvh.validate() == 0


@pytest.mark.gpu
def test_validate_single_triangle(ctx):
    v = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32)
    t = np.array([[0, 1, 2]], np.int32)
    bvh = hx.LBVHBuilder(ctx).build(hx.Scene(v, t))
    assert bvh.validate() == 0


@pytest.mark.parametrize("n", [2, 63, 64, 65, 1023, 1024, 1025, 4099, 8191, 8192, 8193])
@pytest.mark.parametrize("bits", [1, 8, 9, 30, 39, 40, 41, 60, 64])
def test_sort_pairs_one_workgroup(ctx, n, bits):
    """Sorts of up to 8192 keys run in one workgroup (8193: the tiled passes):
    random keys, few distinct keys and keys whose bits above `bits` differ."""
    rng = np.random.default_rng(n * 100 + bits)
    for k in (rng.integers(0, 1 << 63, n, dtype=np.uint64) * np.uint64(2) + np.uint64(1),
              rng.integers(0, 7, n, dtype=np.uint64) << np.uint64(max(bits - 3, 0)), np.zeros(n, np.uint64)):
        vals = rng.permutation(n).astype(np.int32)
        kt = torch.from_numpy(k.view(np.int64).copy()).cuda()
        vt = torch.from_numpy(vals.copy()).cuda()
        hx.sort_pairs(ctx, kt, vt, bits)
        mask = np.uint64((1 << bits) - 1)
        order = np.argsort(k & mask, kind="stable")
        assert np.array_equal(kt.cpu().numpy().view(np.uint64), k[order])
        assert np.array_equal(vt.cpu().numpy(), vals[order])


def _edge_heavy_blocks(clusters):
    """Triangles whose sorted 60-bit codes agree in ever fewer bits from the
    edges of every 512-leaf block to its middle, so that ~57 nodes straddle
    each block (a random order has ~10)."""
    top = 60 - max(int(clusters).bit_length(), 5)
    alt = sum(1 << b for b in range(0, top, 2))
    keys = []
    for j in range(clusters + 1):
        c = (j << top) | alt
        below = [c & ~(1 << b) for b in range(0, top, 2)]
        above = [c | (1 << b) for b in range(1, top, 2)]
        per = 256 // (len(below) + 1)
        if j > 0:
            keys += below * per + [c] * (256 - per * len(below))
        if j < clusters:
            keys += above * per + [c] * (256 - per * len(above))
    k = np.array(keys, np.uint64)
    xyz = np.zeros((len(k), 3), np.int64)
    for b in range(20):
        for a in range(3):
            xyz[:, a] |= ((k >> np.uint64(3 * b + a)) & np.uint64(1)).astype(np.int64) << b
    v = np.repeat(((xyz + 0.5) / 1048575.0)[:, None, :], 3, 1)
    v[:, 1, 0] += 1e-7
    v[:, 2, 1] += 1e-7
    v[0, :], v[-1, :] = 0.0, 1.0  # the unit box
    return v.astype(np.float32).reshape(-1, 3), np.arange(3 * len(v), dtype=np.int32).reshape(-1, 3)


# 16 and 31 blocks fit one and two merge levels, 200 clusters overflow the first
# level's workgroups, 16 the last one's (640 entries; 16 x 57 of them).
@pytest.mark.parametrize("clusters", [1, 2, 16, 30, 200])
def test_lbvh_merge_of_straddling_nodes(oracle, ctx, clusters):
    v, t = _edge_heavy_blocks(clusters)
    bvh = hx.LBVHBuilder(ctx, morton_bits=60).build(hx.Scene(v, t))
    ref = oracle.build_lbvh(v, t, bits=60)
    a = oracle.bin_canonical(bvh.nodes_host(), bvh.n_interior, bvh.n_leaves, bvh.tri_indices_host())
    b = oracle.bin_canonical(ref["nodes"], ref["n_interior"], ref["n_leaves"], ref["tri_idx"])
    assert np.array_equal(a, b)


# Blocks of 512 leaves, merges of up to 16 lists (one level up to 8192 leaves).
@pytest.mark.parametrize("n", [2, 511, 512, 513, 1025, 8191, 8192, 8193, 131073])
@pytest.mark.parametrize("adaptive", [0, 1])
def test_lbvh_merge_level_edges(oracle, ctx, n, adaptive):
    v, t = scenes.uniform_soup(n, seed=n)
    bvh = hx.LBVHBuilder(ctx, morton_bits=60, adaptive_leaf_size=adaptive, max_leaf_size=3).build(hx.Scene(v, t))
    ref = oracle.build_lbvh(v, t, bits=60, adaptive=bool(adaptive), max_leaf_size=3)
    a = oracle.bin_canonical(bvh.nodes_host(), bvh.n_interior, bvh.n_leaves, bvh.tri_indices_host())
    b = oracle.bin_canonical(ref["nodes"], ref["n_interior"], ref["n_leaves"], ref["tri_idx"])
    assert np.array_equal(a, b)


# Sorts of fewer than 2560 keys a CU (10-bit digits: 1024) take smaller tiles and may
# need more status words than a larger sort: those are reserved with the larger one's.
@pytest.mark.parametrize("digits", [8, 10])
def test_smaller_sort_keeps_the_status_buffer(digits):
    c = hx.Context(0)
    c.set_tuning("sort_digit_bits", digits)
    line = torch.cuda.get_device_properties(0).multi_processor_count * (2560 if digits == 8 else 1024)
    rng = np.random.default_rng(digits)
    src = [torch.from_numpy(rng.integers(0, 1 << 62, n, dtype=np.int64)).cuda() for n in (line, line - 1)]
    keys = [k.clone() for k in src]
    vals = [torch.arange(k.numel(), dtype=torch.int32, device="cuda") for k in src]
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    c.set_stream(s)
    try:
        with torch.cuda.stream(s):
            hx.sort_pairs(c, keys[0], vals[0], 62)
            s.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                hx.sort_pairs(c, keys[1], vals[1], 62)
    finally:
        c.set_stream(torch.cuda.current_stream())
    order = torch.argsort(src[1], stable=True)
    for _ in range(3):
        keys[1].copy_(src[1])
        vals[1].copy_(torch.arange(src[1].numel(), dtype=torch.int32, device="cuda"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(keys[1].cpu().numpy(), src[1][order].cpu().numpy())
        assert np.array_equal(vals[1].cpu().numpy(), order.int().cpu().numpy())


# More than 640 entries of a merge go in runs that leave at most 258 nodes each: one
# run and a few entries, several runs, and three levels of them.
@pytest.mark.parametrize("clusters", [11, 12, 45, 300, 1200])
@pytest.mark.parametrize("adaptive", [0, 1])
def test_lbvh_merge_in_runs(oracle, ctx, clusters, adaptive):
    v, t = _edge_heavy_blocks(clusters)
    bvh = hx.LBVHBuilder(ctx, morton_bits=60, adaptive_leaf_size=adaptive, max_leaf_size=3).build(hx.Scene(v, t))
    ref = oracle.build_lbvh(v, t, bits=60, adaptive=bool(adaptive), max_leaf_size=3)
    a = oracle.bin_canonical(bvh.nodes_host(), bvh.n_interior, bvh.n_leaves, bvh.tri_indices_host())
    b = oracle.bin_canonical(ref["nodes"], ref["n_interior"], ref["n_leaves"], ref["tri_idx"])
    assert np.array_equal(a, b)


def test_lbvh_merge_in_runs_batched(oracle, ctx):
    meshes = [_edge_heavy_blocks(c) for c in (30, 1, 64)]
    hb = hx.HipBatch(ctx, hx.MeshBatch.from_meshes(meshes), morton_bits=60)
    for m, (v, t) in enumerate(meshes):
        got, ref = hb.mesh_host(m), oracle.build_lbvh(v, t, bits=60)
        a = oracle.bin_canonical(got["nodes"], got["n_interior"], got["n_leaves"], got["tri_idx"])
        b = oracle.bin_canonical(ref["nodes"], ref["n_interior"], ref["n_leaves"], ref["tri_idx"])
        assert np.array_equal(a, b), m


def test_lbvh_merge_in_runs_time(ctx):
    """1.5M triangles with ~50 nodes straddling each block: 0.68 ms for the climb; a single
    workgroup's climb of what is left over took 64 ms."""
    v, t = _edge_heavy_blocks(3000)
    scene, builder = hx.Scene(v, t), hx.LBVHBuilder(ctx, morton_bits=60)
    bvh = builder.build(scene)
    ctx.set_profiling(True)
    ctx.profile_reset()
    try:
        builder.rebuild(bvh, scene)
        ms = ctx.profile()["climb"][1]
    finally:
        ctx.set_profiling(False)
    assert ms < 10.0


# Both sides of the line from which a sort takes the tunable's keys per thread, the
# smallest tiled sort, and more keys than any clamp, with every instantiation.
@pytest.mark.parametrize("digits", [8, 10])
@pytest.mark.parametrize("items", [8, 16, 32])
@pytest.mark.parametrize("lookback", [4, 8, 16])
def test_sort_pairs_tiled_sizes(digits, items, lookback):
    c = hx.Context(0)
    for name, value in (("sort_digit_bits", digits), ("sort_items", items), ("sort_lookback", lookback)):
        c.set_tuning(name, value)
    line = torch.cuda.get_device_properties(0).multi_processor_count * (2560 if digits == 8 else 1024)
    for n, bits in ((8193, 64), (line - 1, 41), (line, 60), (2 * line + 12345, 33)):
        rng = np.random.default_rng(n + items)
        k = rng.integers(0, 1 << 63, n, dtype=np.uint64) >> np.uint64(63 - min(bits, 63))
        k[: n // 3] = k[0]
        vals = rng.permutation(n).astype(np.int32)
        kt = torch.from_numpy(k.view(np.int64).copy()).cuda()
        vt = torch.from_numpy(vals.copy()).cuda()
        hx.sort_pairs(c, kt, vt, bits)
        order = np.argsort(k, kind="stable")
        assert np.array_equal(kt.cpu().numpy().view(np.uint64), k[order])
        assert np.array_equal(vt.cpu().numpy(), vals[order])


@pytest.mark.parametrize("local_run", [1, 64])
def test_lbvh_large_sort_32_keys_per_thread(oracle, local_run):
    """32 keys per thread in a build whose sort is above the line; with runs of one key
    allowed the split sort falls back to the remaining passes."""
    c = hx.Context(0)
    c.set_tuning("sort_items", 32)
    c.set_tuning("sort_local_run", local_run)
    v, t = scenes.gaussian_mixture_soup(800000, seed=5)
    _check_build(oracle, c, v, t, 60)


@pytest.mark.parametrize("n", [64, 65, 66, 1000, 5000, 8192])
@pytest.mark.parametrize("run", [63, 64, 65, 66, 8192])
def test_sort_pairs_one_workgroup_runs(ctx, n, run):
    """Runs of equal high bits up to, at and over the longest one ranked in place (64)."""
    rng = np.random.default_rng(n + run)
    high = np.repeat(rng.permutation(n // run + 1), run)[:n].astype(np.uint64) << np.uint64(40)
    k = (high | rng.integers(0, 1 << 28, n, dtype=np.uint64))[rng.permutation(n)]
    vals = rng.permutation(n).astype(np.int32)
    kt = torch.from_numpy(k.view(np.int64).copy()).cuda()
    vt = torch.from_numpy(vals.copy()).cuda()
    hx.sort_pairs(ctx, kt, vt, 60)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(kt.cpu().numpy().view(np.uint64), k[order])
    assert np.array_equal(vt.cpu().numpy(), vals[order])
