"""GPU parity: the HIP engine, called through its C ABI, against the golden
vectors written by the real tay10r/lbvh and against the oracle.

Bar: bit-exact Morton codes, sorted order, topology and boxes; identical
hit/miss, primitive ids, t bits and uv bits for the reference intersector.
The watertight intersector is compared with the oracle's restatement of the
same test with a tolerance of 2 ulp on t (ids identical)."""
import numpy as np
import pytest

import lbvh_amd
import oracle
from lbvh_amd import workload as W
from conftest import golden_cases, nodes_u32

pytestmark = pytest.mark.gpu

CASES = golden_cases()
IDS = [c[0] for c in CASES]
VARIANTS = [(30, 0), (30, 1), (63, 0), (63, 1)]
VIDS = ["b30_ref", "b30_pid", "b63_ref", "b63_pid"]


def ulp_diff(a, b):
    ai = a.view(np.int32).astype(np.int64)
    bi = b.view(np.int32).astype(np.int64)
    ai = np.where(ai < 0, -(ai & 0x7FFFFFFF), ai)
    bi = np.where(bi < 0, -(bi & 0x7FFFFFFF), bi)
    return np.abs(ai - bi)


@pytest.mark.parametrize("case", CASES, ids=IDS)
@pytest.mark.parametrize("bits,leaf", VARIANTS, ids=VIDS)
def test_build_matches_golden(ctx, case, bits, leaf):
    name, rec = case
    tri = rec["tri"]
    bvh = ctx.build_triangles(tri, code_bits=bits, leaf_order=leaf, keep_codes=True)
    key = "b%d_l%d" % (bits, leaf)
    nodes = bvh.nodes()
    assert np.array_equal(nodes_u32(nodes), rec[key + "_nodes"]), "node array differs"
    sc, ids, bounds = bvh.codes()
    assert np.array_equal(sc, rec[key + "_sorted"]), "sorted codes differ"
    assert np.array_equal(bounds.view(np.uint32), rec["bounds"].view(np.uint32))
    # stable (code, id) order
    order = np.argsort(rec["codes%d" % bits], kind="stable").astype(np.uint32)
    assert np.array_equal(ids, order)
    bvh.destroy()


@pytest.mark.parametrize("case", CASES, ids=IDS)
@pytest.mark.parametrize("leaf", [0, 1], ids=["ref", "pid"])
@pytest.mark.parametrize("mode", [0, 1], ids=["first", "lowid"])
def test_trace_matches_golden(ctx, case, leaf, mode):
    name, rec = case
    bvh = ctx.build_triangles(rec["tri"], code_bits=30, leaf_order=leaf)
    p, t, uv = ctx.trace(bvh, rec["rays"], mode)
    key = "b30_l%d_m%d" % (leaf, mode)
    assert np.array_equal(p, rec[key + "_prim"])
    assert np.array_equal(t.view(np.uint32), rec[key + "_t"].view(np.uint32))
    hit = p != 0xFFFFFFFF
    assert np.array_equal(uv[hit].view(np.uint32), rec[key + "_uv"][hit].view(np.uint32))
    assert np.all(uv[~hit] == 0)
    bvh.destroy()


@pytest.mark.parametrize("nrays", [4096, 600000], ids=["rays4096", "rays600000"])
@pytest.mark.parametrize("mode", [0, 1], ids=["first", "lowid"])
def test_trace_deep_stacks_match_oracle(ctx, nrays, mode):
    """20,000 large, mutually overlapping triangles: most rays hit both
    children at many levels, so traversal stacks run far past the entries
    kept in registers and LDS into the private array (hundreds of pops per
    ray).  A dispatch that leaves most of the device idle and one that fills
    it, against the oracle, bit for bit."""
    print("deep-stack trace nrays=%d mode=%d" % (nrays, mode), flush=True)
    rng = np.random.default_rng(3)
    n = 20000
    c = rng.random((n, 3)) * 0.2 + 0.4
    v = np.concatenate([c + rng.normal(size=(n, 3)) * 0.3 for _ in range(3)], axis=1)
    tri = W.make_triangles(v.astype(np.float32))
    rays = W.box_rays(5, np.full(3, -0.5, np.float32), np.full(3, 1.5, np.float32), nrays)
    bvh = ctx.build_triangles(tri, code_bits=63, leaf_order=1)
    nodes, _, _, _ = oracle.build(tri, 63, 1)
    assert bvh.nodes().tobytes() == nodes.tobytes()
    p, t, uv = ctx.trace(bvh, rays, mode)
    op, ot, ouv = oracle.trace(nodes, tri, rays, mode)
    assert np.array_equal(p, op)
    assert np.array_equal(t.view(np.uint32), ot.view(np.uint32))
    hit = p != 0xFFFFFFFF
    assert np.array_equal(uv[hit].view(np.uint32), ouv[hit].view(np.uint32))
    bvh.destroy()


@pytest.mark.parametrize("n", [128, 256, 513, 1024, 70000, 131072])
def test_trace_stack_ring_depths_match_oracle(ctx, n):
    """Concentric triangles of one centre: equal codes, so a balanced tree of
    ceil(log2 n) levels, and every ray through the centre enters both children
    of every node, down to stacks just below, at and past the 8 entries of the
    LDS ring and past two rings."""
    s = (np.arange(1, n + 1, dtype=np.float64) * 2.0 ** -20)[:, None]
    corner = np.array([[-1, -1, -1], [1, -1, 0], [0, 1, 1]], dtype=np.float64)
    v = np.concatenate([0.5 + s * corner[k] for k in range(3)], axis=1).astype(np.float32)
    tri = W.make_triangles(v[np.random.default_rng(n).permutation(n)])
    rays = W.primary_rays(9, 7)
    rays[:, 3:6] = (0.5 - rays[:, 0:3]) + np.random.default_rng(1).normal(size=(63, 3)) * 2.0 ** -18
    bvh = ctx.build_triangles(tri, code_bits=30, leaf_order=1)
    nodes, _, _, _ = oracle.build(tri, 30, 1)
    assert bvh.nodes().tobytes() == nodes.tobytes()
    p, t, uv = ctx.trace(bvh, rays, 0)
    op, ot, ouv = oracle.trace(nodes, tri, rays, 0)
    assert (p != 0xFFFFFFFF).any()
    assert np.array_equal(p, op)
    assert np.array_equal(t.view(np.uint32), ot.view(np.uint32))
    assert np.array_equal(uv.view(np.uint32), ouv.view(np.uint32))
    bvh.destroy()


@pytest.mark.parametrize("n", [2, 3, 5, 33, 4097, 70001])
@pytest.mark.parametrize("bits,leaf", VARIANTS, ids=VIDS)
def test_build_matches_oracle_ragged(ctx, n, bits, leaf):
    v = W.cluster_vertices(1000 + n, n)
    tri = W.make_triangles(v)
    bvh = ctx.build_triangles(tri, code_bits=bits, leaf_order=leaf, keep_codes=True)
    on, ob, osc, oids = oracle.build(tri, bits, leaf)
    assert bvh.nodes().tobytes() == on.tobytes()
    sc, ids, bounds = bvh.codes()
    assert np.array_equal(sc, osc)
    assert np.array_equal(ids, oids)


@pytest.mark.parametrize("n", [2, 64, 65, 511, 513, 2049, 4095, 4096, 4097, 20001, 65535])
@pytest.mark.parametrize("dist", ["uniform", "clustered", "equal", "two"])
def test_small_builds_match_oracle(ctx, n, dist):
    """Builds below 65,536 primitives sort in one workgroup (up to 4,096) or
    in chunks that are merged: wave and block remainders, runs of a few dense
    spots, one code for everything, two far groups; triangles and boxes, both
    code widths and leaf orders."""
    rng = np.random.default_rng(n)
    if dist == "uniform":
        v = W.uniform_vertices(n, n, 0.01)
    elif dist == "clustered":
        v = W.cluster_vertices(n, n, 5, 0.0005, 0.0005)
    else:
        c = np.zeros((n, 1), np.float32) if dist == "equal" else (rng.integers(0, 2, (n, 1)) * 100.0)
        v = (np.tile(rng.random((1, 9)), (n, 1)) + c).astype(np.float32)
    tri = W.make_triangles(v)
    for bits, leaf in VARIANTS:
        bvh = ctx.build_triangles(tri, code_bits=bits, leaf_order=leaf, keep_codes=True)
        on, ob, osc, oids = oracle.build(tri, bits, leaf)
        sc, ids, bounds = bvh.codes()
        assert np.array_equal(sc, osc)
        assert np.array_equal(ids, oids)
        assert np.array_equal(bounds, np.asarray(ob, np.float32).reshape(-1))
        assert bvh.nodes().tobytes() == on.tobytes()
        bvh.destroy()
    p0, p1, p2 = tri[:, 0:3], tri[:, 0:3] - tri[:, 3:6], tri[:, 0:3] + tri[:, 6:9]
    boxes = np.concatenate([np.minimum(np.minimum(p0, p1), p2), np.maximum(np.maximum(p0, p1), p2)],
                           axis=1)
    for bits, leaf in VARIANTS:
        bvh = ctx.build_aabbs(boxes, code_bits=bits, leaf_order=leaf)
        assert bvh.nodes().tobytes() == oracle.build(tri, bits, leaf)[0].tobytes()
        bvh.destroy()


@pytest.mark.parametrize("kind", ["one-cluster-and-outlier", "duplicates", "two-clusters"])
@pytest.mark.parametrize("n", [4097, 5120, 8193, 16384, 16385, 32768, 32769, 65535])
def test_skewed_small_builds_sort_in_chunks(ctx, kind, n):
    """Builds of 4,097 to 65,535 primitives sort in chunks that are merged by
    ranks, at the sizes where the chunks change or the last one is short, and
    not by a global digit, whose fullest bucket would be one workgroup's work;
    equal codes stay in id order across chunks."""
    tri = _hybrid_edge_scene(kind, n, 700 + n)
    for bits, leaf in [(30, 1), (63, 1), (63, 0)]:
        bvh = ctx.build_triangles(tri, code_bits=bits, leaf_order=leaf, keep_codes=leaf == 1)
        info = bvh.info()
        assert (info.sort_strategy, info.sort_global_digits) == (3, 0)
        on, _, osc, oids = oracle.build(tri, bits, leaf)
        if leaf == 1:
            sc, ids, _ = bvh.codes()
            assert np.array_equal(sc, osc)
            assert np.array_equal(ids, oids)
        assert bvh.nodes().tobytes() == on.tobytes()
        bvh.destroy()
    p0, p1, p2 = tri[:, 0:3], tri[:, 0:3] - tri[:, 3:6], tri[:, 0:3] + tri[:, 6:9]
    box = np.concatenate([np.minimum(np.minimum(p0, p1), p2), np.maximum(np.maximum(p0, p1), p2)],
                         axis=1).astype(np.float64)
    for leaf in (0, 1):
        want, _, _ = oracle.build_f64(box, leaf)
        assert ctx.build_aabbs_f64(box, leaf).tobytes() == want.tobytes()


@pytest.mark.parametrize("extent", [0.01, 2.0 ** 24, 2.0 ** 25, 3e7, 1e8, 1e30])
@pytest.mark.parametrize("n", [200, 4096, 4097, 60000, 70000])
def test_every_sort_orders_all_code_bits(ctx, n, extent):
    """From an extent of 2^24 a centre at the far end of an axis falls into
    cell 2^20, so 63-bit codes use bits 60-62; codes of a small scene leave
    the top bits empty.  Every sort strategy, the untuned choice, the tuner's
    and the allocation-free build give the oracle's codes, ids and nodes."""
    print("code bits n=%d extent=%g" % (n, extent), flush=True)
    rng = np.random.default_rng(n)
    c = (rng.random((n, 1, 3)) * extent).astype(np.float32)
    c[0], c[n // 2], c[-1] = extent, 0.0, extent  # the far corner, out of input order
    tri = W.make_triangles(np.tile(c, (1, 3, 1)).reshape(n, 9))
    plain = lbvh_amd.Context(0)
    plain.set_autotune(False)
    for bits, leaf in [(63, 1), (63, 0), (30, 1)]:
        on, _, osc, oids = oracle.build(tri, bits, leaf)
        assert (bits == 63 and extent == 2.0 ** 24) <= bool((osc >> 60).any())
        builds = [(plain, {}), (ctx, {})]
        builds += [(plain, dict(sort_strategy=s, sort_digit_bits=d, sort_tile=t))
                   for s, d, t in SORT_CONFIGS]
        for c2, opts in builds:
            bvh = c2.build_triangles(tri, code_bits=bits, leaf_order=leaf, keep_codes=True, **opts)
            sc, ids, _ = bvh.codes()
            assert np.array_equal(sc, osc), opts
            assert np.array_equal(ids, oids), opts
            assert bvh.nodes().tobytes() == on.tobytes(), opts
            bvh.destroy()
        import ctypes
        from lbvh_amd.hip import DeviceArray
        d_tri, d_nodes = DeviceArray.from_host(tri), DeviceArray(32 * (n - 1), np.uint8)
        opts = lbvh_amd._make_opts(bits, leaf, False, 10, 4096, lbvh_amd.SORT_HYBRID)
        plain._check(lbvh_amd.lib().lbvh_build_triangles_noalloc(
            plain.handle, ctypes.c_void_p(d_tri.ptr), n, ctypes.byref(opts),
            ctypes.c_void_p(d_nodes.ptr)))
        plain.synchronize()
        assert d_nodes.numpy().tobytes() == on.tobytes()
    plain.close()


@pytest.mark.parametrize("slots", ["1", "200"])
@pytest.mark.parametrize("n", [9000, 70001, 300001])
@pytest.mark.parametrize("bits,leaf", [(30, 0), (63, 1)], ids=["b30_ref", "b63_pid"])
def test_split_tree_merges_match_oracle(ctx, monkeypatch, slots, n, bits, leaf):
    """The upper tree levels merge a group's lists 8 at a time (then the
    partial lists) when they hold more elements than a workgroup's slots.
    LBVH_TREE_GROUP_SLOTS lowers that limit so ordinary scenes take the
    split path (512-position level-0 workgroups, 64 per group): 18 level-0
    workgroups in one level-1 group (n = 9000), a partial last group
    (70001), ten level-1 workgroups under one top group (300001)."""
    monkeypatch.setenv("LBVH_TREE_GROUP_SLOTS", slots)
    v = W.cluster_vertices(2000 + n, n)
    tri = W.make_triangles(v)
    bvh = ctx.build_triangles(tri, code_bits=bits, leaf_order=leaf, keep_codes=True)
    on, ob, osc, oids = oracle.build(tri, bits, leaf)
    assert bvh.nodes().tobytes() == on.tobytes()
    sc, ids, bounds = bvh.codes()
    assert np.array_equal(sc, osc)
    assert np.array_equal(ids, oids)
    # the refit starts from the flags and links the tree kernels leave
    moved = W.make_triangles(W.perturb(7, v, 1e-4))
    ctx.refit_triangles(bvh, moved)
    assert bvh.nodes().tobytes() == oracle.fit(on, moved).tobytes()


SORT_CONFIGS = [(1, 8, 1024), (1, 8, 2048), (1, 8, 4096), (1, 10, 2048), (1, 10, 4096),
                (2, 8, 2048), (2, 8, 4096), (2, 10, 2048), (2, 10, 4096),
                (3, 8, 2048), (3, 8, 4096), (3, 10, 4096)]
SORT_NAMES = {1: "onesweep", 2: "rts", 3: "hybrid"}


@pytest.mark.parametrize("strategy,digit_bits,tile", SORT_CONFIGS,
                         ids=["%s-d%d-t%d" % (SORT_NAMES[c[0]], c[1], c[2])
                              for c in SORT_CONFIGS])
@pytest.mark.parametrize("bits", [30, 63])
def test_sort_configurations_agree(ctx, strategy, digit_bits, tile, bits):
    """Every sort strategy at every digit width and tile size gives the
    oracle's stable (code, id) order and tree."""
    v = W.cluster_vertices(77, 300000)
    tri = W.make_triangles(v)
    bvh = ctx.build_triangles(tri, code_bits=bits, leaf_order=1, keep_codes=True,
                              sort_digit_bits=digit_bits, sort_tile=tile, sort_strategy=strategy)
    on, _, osc, oids = oracle.build(tri, bits, 1)
    sc, ids, _ = bvh.codes()
    assert np.array_equal(sc, osc)
    assert np.array_equal(ids, oids)
    assert bvh.nodes().tobytes() == on.tobytes()


def _hybrid_edge_scene(kind, n, seed):
    """Key distributions that stress the hybrid sort's buckets."""
    rng = np.random.default_rng(seed)
    if kind == "one-cluster-and-outlier":
        # every code but one shares its top bits: one bucket of n - 1 keys,
        # sorted by the oversize-range path
        v = rng.random((n, 3, 3), dtype=np.float32) * np.float32(1e-3)
        v[-1] += np.float32(1e3)
    elif kind == "duplicates":
        # a handful of distinct triangles repeated: long runs of equal codes
        base = rng.random((7, 3, 3), dtype=np.float32)
        v = base[rng.integers(0, 7, n)]
    elif kind == "two-clusters":
        v = rng.random((n, 3, 3), dtype=np.float32) * np.float32(1e-2)
        v[n // 3:] += np.float32(5.0)
    else:  # "shells": clustered, buckets of every size
        v = W.cluster_vertices(seed, n)
    return W.make_triangles(v.reshape(n, 9))


@pytest.mark.parametrize("kind", ["one-cluster-and-outlier", "duplicates", "two-clusters",
                                  "shells"])
@pytest.mark.parametrize("n", [2, 3, 2049, 4097, 9000, 250001])
@pytest.mark.parametrize("bits", [30, 63])
def test_hybrid_sort_edge_distributions(ctx, kind, n, bits):
    """The hybrid sort on skewed keys (one bucket holding nearly every key,
    runs of equal codes, ragged sizes) gives the oracle's order and tree."""
    tri = _hybrid_edge_scene(kind, n, 600 + n)
    bvh = ctx.build_triangles(tri, code_bits=bits, leaf_order=1, keep_codes=True,
                              sort_strategy=lbvh_amd.SORT_HYBRID)
    assert bvh.info().sort_strategy == 3
    on, _, osc, oids = oracle.build(tri, bits, 1)
    sc, ids, _ = bvh.codes()
    assert np.array_equal(sc, osc)
    assert np.array_equal(ids, oids)
    assert bvh.nodes().tobytes() == on.tobytes()
    bvh.destroy()


def test_rejects_bad_arguments(ctx):
    tri = W.make_triangles(W.uniform_vertices(1, 10, 0.01))
    with pytest.raises(lbvh_amd.LbvhError) as e:
        ctx.build_triangles(tri[:1])
    assert e.value.status == 1
    with pytest.raises(lbvh_amd.LbvhError):
        ctx.build_triangles(tri, code_bits=31)
    with pytest.raises(lbvh_amd.LbvhError):
        ctx.build_triangles(tri, sort_digit_bits=7)


def test_uniform65536_hashes(ctx, hashes):
    e = hashes["uniform65536_seed1"]
    v, tri = W.scene_uniform(1, 65536, 0.01)
    assert oracle.fnv1a64(tri) == e["tri"]
    rays = W.primary_rays(256, 256)
    for leaf in (0, 1):
        bvh = ctx.build_triangles(tri, code_bits=30, leaf_order=leaf, keep_codes=True)
        assert oracle.fnv1a64(bvh.nodes()) == e["b30_l%d_nodes" % leaf]
        sc, _, _ = bvh.codes()
        assert oracle.fnv1a64(sc) == e["b30_l%d_sorted" % leaf]
        for mode in (0, 1):
            p, t, _ = ctx.trace(bvh, rays, mode)
            assert oracle.fnv1a64(np.concatenate([p, t.view(np.uint32)])) == \
                e["b30_l%d_m%d_hits" % (leaf, mode)]
        bvh.destroy()


def test_clustered1m_hashes(ctx, hashes):
    e = hashes["clustered1m_seed2"]
    v, tri = W.scene_clustered(2, 1 << 20)
    if oracle.fnv1a64(tri) != e["tri"]:
        pytest.skip("libm differs from the fixture host: compared in-run only")
    for bits in (30, 63):
        for leaf in (0, 1):
            bvh = ctx.build_triangles(tri, code_bits=bits, leaf_order=leaf, keep_codes=True)
            assert oracle.fnv1a64(bvh.nodes()) == e["b%d_l%d_nodes" % (bits, leaf)]
            sc, _, _ = bvh.codes()
            assert oracle.fnv1a64(sc) == e["b%d_l%d_sorted" % (bits, leaf)]
            bvh.destroy()


def test_uniform16m_hashes(ctx, hashes):
    e = hashes["uniform16m_seed3"]
    v, tri = W.scene_uniform(3, 1 << 24, 5e-4)
    del v
    assert oracle.fnv1a64(tri) == e["tri"]
    for bits in (30, 63):
        for leaf in (0, 1):
            bvh = ctx.build_triangles(tri, code_bits=bits, leaf_order=leaf, keep_codes=True)
            assert oracle.fnv1a64(bvh.nodes()) == e["b%d_l%d_nodes" % (bits, leaf)]
            sc, _, _ = bvh.codes()
            assert oracle.fnv1a64(sc) == e["b%d_l%d_sorted" % (bits, leaf)]
            bvh.destroy()


def test_clustered1m_primary_and_bounce_rays(ctx):
    """The 1,048,576-triangle clustered scene with 63-bit codes: primary rays
    and one diffuse bounce per hit, against the oracle traversal."""
    v, tri = W.scene_clustered(2, 1 << 20)
    bvh = ctx.build_triangles(tri, code_bits=63, leaf_order=1)
    nodes = bvh.nodes()
    rays = W.primary_rays(480, 270)
    for mode in (0, 1):
        p, t, uv = ctx.trace(bvh, rays, mode)
        op, ot, ouv = oracle.trace(nodes, tri, rays, mode)
        assert np.array_equal(p, op)
        assert np.array_equal(t.view(np.uint32), ot.view(np.uint32))
        assert np.array_equal(uv.view(np.uint32), ouv.view(np.uint32))
    b, src = W.bounce_rays(5, tri, rays, p, t)
    assert len(b) > 1000
    for mode in (0, 1):
        p2, t2, _ = ctx.trace(bvh, b, mode)
        op2, ot2, _ = oracle.trace(nodes, tri, b, mode)
        assert np.array_equal(p2, op2)
        assert np.array_equal(t2.view(np.uint32), ot2.view(np.uint32))


def test_watertight_matches_oracle(ctx):
    v, tri = W.scene_uniform(1, 65536, 0.01)
    bvh = ctx.build_triangles(tri, code_bits=30, leaf_order=1)
    nodes = bvh.nodes()
    rays = W.primary_rays(256, 256)
    p, t, uv = ctx.trace(bvh, rays, 2)
    op, ot, ouv = oracle.trace(nodes, tri, rays, 2)
    assert np.array_equal(p, op)
    hit = p != 0xFFFFFFFF
    assert ulp_diff(t[hit], ot[hit]).max() <= 2  # tolerance: 2 ulp on t
    t64 = oracle.t_fp64(tri, rays, p)
    rel = np.abs(t[hit] - t64[hit]) / np.abs(t64[hit])
    print("watertight t: max rel err vs FP64 %.3e over %d hits" % (rel.max(), hit.sum()))
    assert rel.max() < 1e-5


@pytest.mark.parametrize("leaf", [0, 1])
def test_refit_equals_oracle_fit(ctx, leaf):
    v, tri = W.scene_uniform(3, 200000, 5e-4)
    bvh = ctx.build_triangles(tri, code_bits=30, leaf_order=leaf)
    before = bvh.nodes()
    v2 = W.perturb(33, v, 1e-4)
    tri2 = W.make_triangles(v2)
    ctx.refit_triangles(bvh, tri2)
    after = bvh.nodes()
    assert np.array_equal(after["left"], before["left"])
    assert np.array_equal(after["right"], before["right"])
    expect = oracle.fit(before, tri2)
    assert after.tobytes() == expect.tobytes()
    # a second refit back to the original data restores the original boxes
    ctx.refit_triangles(bvh, tri)
    assert bvh.nodes().tobytes() == before.tobytes()


def test_refits_alternating_between_trees(ctx):
    """A context keeps the treelet list of the tree it last refitted: refits
    of A, B, A again and B again each equal the oracle's fit."""
    va, ta = W.scene_uniform(5, 150000, 5e-4)
    vb, tb = W.scene_clustered(6, 90000)
    a = ctx.build_triangles(ta, code_bits=63, leaf_order=1)
    b = ctx.build_triangles(tb, code_bits=30, leaf_order=0)
    na, nb = a.nodes(), b.nodes()
    for k in range(2):
        ma = W.make_triangles(W.perturb(40 + k, va, 1e-4))
        ctx.refit_triangles(a, ma)
        assert a.nodes().tobytes() == oracle.fit(na, ma).tobytes(), "A, round %d" % k
        mb = W.make_triangles(W.perturb(50 + k, vb.reshape(-1, 9), 1e-4))
        ctx.refit_triangles(b, mb)
        assert b.nodes().tobytes() == oracle.fit(nb, mb).tobytes(), "B, round %d" % k
    a.destroy()
    b.destroy()


@pytest.mark.parametrize("n", [2, 3, 5, 1023, 1024, 1025, 2049, 5000])
@pytest.mark.parametrize("bits,leaf", [(30, 0), (63, 1)], ids=["b30_ref", "b63_pid"])
def test_refit_small_and_treelet_edge_sizes(ctx, n, bits, leaf):
    """Refits of trees that are one treelet (n <= 1,024: the root is node 0)
    or a few treelets under a short top tree equal the oracle's fit."""
    v = W.cluster_vertices(3000 + n, n)
    bvh = ctx.build_triangles(W.make_triangles(v), code_bits=bits, leaf_order=leaf)
    before = bvh.nodes()
    moved = W.make_triangles(W.perturb(11, v, 1e-4))
    ctx.refit_triangles(bvh, moved)
    assert bvh.nodes().tobytes() == oracle.fit(before, moved).tobytes()
    bvh.destroy()


@pytest.mark.parametrize("leaf", [0, 1], ids=["ref", "pid"])
def test_refit_with_nan_vertices_equals_oracle_fit(ctx, leaf):
    """A refit whose new vertices hold NaNs (the topology is kept, so no
    code is computed from them): treelets with a NaN box are fitted in tree
    order, and every box equals the oracle's fit bit for bit."""
    v, tri = W.scene_uniform(8, 120000, 5e-4)
    bvh = ctx.build_triangles(tri, code_bits=30, leaf_order=leaf)
    before = bvh.nodes()
    v2 = W.perturb(9, v, 1e-4)
    rng = np.random.default_rng(10)
    bad = rng.choice(v2.shape[0], 40, replace=False)
    v2[bad, rng.integers(0, 9, 40)] = np.float32(np.nan)
    tri2 = W.make_triangles(v2)
    ctx.refit_triangles(bvh, tri2)
    assert bvh.nodes().tobytes() == oracle.fit(before, tri2).tobytes()


def test_device_path_equals_host_path(ctx):
    from lbvh_amd import hip
    v, tri = W.scene_uniform(1, 65536, 0.01)
    rays = W.primary_rays(128, 128)
    host = ctx.build_triangles(tri, code_bits=63, leaf_order=1)
    hp, ht, huv = ctx.trace(host, rays, 1)
    dtri = hip.DeviceArray.from_host(tri)
    drays = hip.DeviceArray.from_host(rays)
    dev = ctx.build_triangles(dtri, code_bits=63, leaf_order=1)
    dp, dt, duv = ctx.trace(dev, drays, 1)
    ctx.synchronize()
    assert dev.nodes().tobytes() == host.nodes().tobytes()
    assert np.array_equal(dp.numpy(), hp)
    assert np.array_equal(dt.numpy().view(np.uint32), ht.view(np.uint32))
    assert np.array_equal(duv.numpy().view(np.uint32), huv.view(np.uint32))
    # device refit from a device buffer, then trace again
    v2 = W.perturb(2, v, 1e-4)
    tri2 = W.make_triangles(v2)
    ctx.refit_triangles(dev, hip.DeviceArray.from_host(tri2))
    ctx.synchronize()
    assert dev.nodes().tobytes() == oracle.fit(host.nodes(), tri2).tobytes()


TORCH_INTEROP = r"""
import sys, numpy as np
import torch  # first: the engine then shares torch's HIP runtime
sys.path.insert(0, %r)
import lbvh_amd, oracle
from lbvh_amd import workload as W
v, tri = W.scene_uniform(1, 20000, 0.01)
rays = W.primary_rays(64, 64)
ctx = lbvh_amd.Context(0)
ctx.set_stream(torch.cuda.current_stream())
b = ctx.build_triangles(torch.from_numpy(tri).cuda(), code_bits=30, leaf_order=1)
prim = torch.empty(rays.shape[0], dtype=torch.int32, device="cuda")
t = torch.empty(rays.shape[0], dtype=torch.float32, device="cuda")
uv = torch.empty((rays.shape[0], 2), dtype=torch.float32, device="cuda")
ctx.trace(b, torch.from_numpy(rays).cuda(), 0, out=(prim, t, uv))
torch.cuda.synchronize()
on, _, _, _ = oracle.build(tri, 30, 1)
op, ot, _ = oracle.trace(on, tri, rays, 0)
assert b.nodes().tobytes() == on.tobytes()
assert np.array_equal(prim.cpu().numpy().view(np.uint32), op)
assert np.array_equal(t.cpu().numpy().view(np.uint32), ot.view(np.uint32))
print("torch interop ok")
"""


def test_torch_tensors_share_the_runtime(tmp_path):
    """torch CUDA tensors work as device arrays when torch is imported first
    (run in a fresh process: one HIP runtime per process)."""
    import subprocess
    import sys
    from conftest import ROOT
    r = subprocess.run([sys.executable, "-c", TORCH_INTEROP % ROOT], capture_output=True, text=True,
                       timeout=180)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "torch interop ok" in r.stdout


TORCH_ORDER = r"""
import sys, numpy as np
import torch
sys.path.insert(0, %r)
import lbvh_amd, oracle
from lbvh_amd import workload as W
v, tri = W.scene_uniform(1, 3000, 0.02)
rays = W.primary_rays(32, 32)
on, _, _, _ = oracle.build(tri, 30, 1)
op, ot, _ = oracle.trace(on, tri, rays, 0)
ctx = lbvh_amd.Context(0)
src_tri, src_rays = torch.from_numpy(tri).cuda(), torch.from_numpy(rays).cuda()
big = torch.randn(6144, 6144, device="cuda")
for stream in (torch.cuda.default_stream(), torch.cuda.Stream()):
    for k in range(3):
        d_tri, d_rays = torch.zeros_like(src_tri), torch.zeros_like(src_rays)
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            for _ in range(4):
                y = big @ big  # a few ms before the inputs are written
            d_tri.copy_(src_tri)
            b = ctx.build_triangles(d_tri, code_bits=30, leaf_order=1)
            for _ in range(4):
                y = big @ big
            d_rays.copy_(src_rays)
            prim, t, uv = ctx.trace(b, d_rays, 0)
        ctx.synchronize()
        assert b.nodes().tobytes() == on.tobytes()
        assert np.array_equal(prim.numpy(), op)
        assert np.array_equal(t.numpy().view(np.uint32), ot.view(np.uint32))
        torch.cuda.synchronize()
print("torch order ok")
"""


def test_torch_inputs_still_being_written_are_waited_for():
    """Calls on the context's own stream with torch tensors start after the
    work of torch's current stream, the default one or another."""
    import subprocess
    import sys
    from conftest import ROOT
    r = subprocess.run([sys.executable, "-c", TORCH_ORDER % ROOT], capture_output=True, text=True,
                       timeout=180)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "torch order ok" in r.stdout


TORCH_ORDER_MIXED = r"""
import sys, numpy as np
import torch
sys.path.insert(0, %r)
import lbvh_amd, oracle
from lbvh_amd import workload as W
from lbvh_amd.hip import DeviceArray
v, tri = W.scene_uniform(1, 3000, 0.02)
rays = W.primary_rays(32, 32)
ctx = lbvh_amd.Context(0)
big = torch.randn(6144, 6144, device="cuda")

def late(x):
    "x on the GPU, written only after a few ms of other work"
    src = torch.from_numpy(np.ascontiguousarray(x).view(np.uint8).reshape(-1)).cuda()
    d = torch.zeros_like(src)
    torch.cuda.synchronize()
    for _ in range(4):
        y = big @ big
    d.copy_(src)
    return d

def outputs(m, prim, t):
    "written by torch late: the hits have to come after that"
    o = tuple(torch.zeros(s, dtype=d, device="cuda") for s, d in ((m, prim), (m, t), ((m, 2), t)))
    torch.cuda.synchronize()
    for _ in range(4):
        y = big @ big
    for x in o:
        x.fill_(7)
    return o

# FP64: nodes, then triangles, then outputs still being written, the rest not torch's
boxes = np.concatenate([c.min(axis=1) if k == 0 else c.max(axis=1) for c in [v.reshape(-1, 3, 3)]
                        for k in (0, 1)], axis=1).astype(np.float64)
tri64, rays64 = tri.astype(np.float64), rays.astype(np.float64)
on, _, _ = oracle.build_f64(boxes, 1)
op, ot, ouv = oracle.trace_f64(on, tri64, rays64, 0)
for k in range(4):
    nodes, t64, out = (DeviceArray.from_host(on.view(np.uint64).reshape(-1)),
                       DeviceArray.from_host(tri64), None)
    r64 = DeviceArray.from_host(rays64)
    if k == 0:
        nodes = late(on).view(torch.int64)
    elif k == 1:
        t64 = late(tri64).view(torch.float64).reshape(-1, 12)
    elif k == 2:
        out = outputs(len(rays), torch.int64, torch.float64)
    else:
        d_boxes, nodes = DeviceArray.from_host(boxes), outputs(2999 * 8, torch.int64, torch.float64)[0]
        ctx.build_aabbs_f64(d_boxes, 1, out=nodes)
    prim, t, uv = ctx.trace_f64(nodes, t64, r64, out=out)
    ctx.synchronize()
    host = lambda x: x.cpu().numpy() if isinstance(x, torch.Tensor) else x.numpy()
    assert np.array_equal(host(prim).view(np.uint64), op), k
    assert np.array_equal(host(t).view(np.uint64), ot.view(np.uint64)), k
    torch.cuda.synchronize()
# a batch: ray offsets, then outputs
off = np.array([0, 1000, 3000], np.uint64)
roff = np.array([0, 500, 1024], np.uint64)
batch = ctx.build_batch(DeviceArray.from_host(tri), off, leaf_order=1)
want = batch.trace(rays, roff)
for k in range(2):
    d_rays, d_off, out = DeviceArray.from_host(rays), DeviceArray.from_host(roff), None
    if k == 0:
        d_off = late(roff).view(torch.int64)
    else:
        out = outputs(len(rays), torch.int32, torch.float32)
    prim, t, uv = batch.trace(d_rays, d_off, out=out)
    ctx.synchronize()
    assert np.array_equal(host(prim).view(np.uint32), want[0]), k
    assert np.array_equal(host(t).view(np.uint32), want[1].view(np.uint32)), k
    torch.cuda.synchronize()
print("torch mixed order ok")
"""


def test_any_torch_argument_orders_the_call():
    """Inputs and outputs alike: a call starts after torch's current stream
    when any one of its arrays is a torch tensor and the others are not."""
    import subprocess
    import sys
    from conftest import ROOT
    r = subprocess.run([sys.executable, "-c", TORCH_ORDER_MIXED % ROOT], capture_output=True,
                       text=True, timeout=180)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "torch mixed order ok" in r.stdout


def test_cpp_dropin_conformance(tmp_path):
    """The C++ drop-in header (include/lbvh_mi355x.hpp) used with the
    reference's call shapes: builder over triangles and over a user primitive
    with a lambda converter, host traverser, device tree; nodes and hits
    against the oracle."""
    import os
    import subprocess
    from lbvh_amd import build as B
    if not os.path.exists(B.DROPIN_BIN):
        pytest.skip("drop-in conformance program not built")
    out = tmp_path / "dropin.bin"
    r = subprocess.run([B.DROPIN_BIN, str(out)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    raw = out.read_bytes()
    n = int(np.frombuffer(raw[:8], np.uint64)[0])
    off = 8
    tri = np.frombuffer(raw[off:off + 48 * n], np.float32).reshape(n, 12)
    off += 48 * n
    nodes = np.frombuffer(raw[off:off + 32 * (n - 1)], oracle.NODE_DTYPE)
    off += 32 * (n - 1)
    m = int(np.frombuffer(raw[off:off + 8], np.uint64)[0])
    off += 8
    rays = np.frombuffer(raw[off:off + 32 * m], np.float32).reshape(m, 8)
    off += 32 * m
    hp = np.frombuffer(raw[off:off + 4 * m], np.uint32)
    off += 4 * m
    ht = np.frombuffer(raw[off:off + 4 * m], np.float32)
    on, _, _, _ = oracle.build(tri, 30, 0)
    assert nodes.tobytes() == on.tobytes()
    op, ot, _ = oracle.trace(on, tri, rays, 0)
    assert np.array_equal(hp, op)
    assert np.array_equal(ht.view(np.uint32), ot.view(np.uint32))
    # builder<double> over triangle<double> (its traversal is checked against
    # brute force inside the program)
    off += 4 * m + 64
    n64 = int(np.frombuffer(raw[off:off + 8], np.uint64)[0])
    off += 8
    tri64 = np.frombuffer(raw[off:off + 96 * n64], np.float64).reshape(n64, 12)
    off += 96 * n64
    nodes64 = np.frombuffer(raw[off:off + 64 * (n64 - 1)], oracle.NODE64_DTYPE)
    off += 64 * (n64 - 1)
    nodes64_pid = np.frombuffer(raw[off:off + 64 * (n64 - 1)], oracle.NODE64_DTYPE)
    assert off + 64 * (n64 - 1) == len(raw)
    boxes64 = oracle.triangle_aabb_f64(tri64)
    want, _, _ = oracle.build_f64(boxes64, 0)
    assert nodes64.tobytes() == want.tobytes()
    want_pid, _, _ = oracle.build_f64(boxes64, 1)
    assert nodes64_pid.tobytes() == want_pid.tobytes()


def test_aabb_build_equals_triangle_build(ctx):
    v, tri = W.scene_uniform(4, 50000, 0.01)
    boxes = oracle.triangle_aabb(tri)
    a = ctx.build_triangles(tri, code_bits=30, leaf_order=1)
    b = ctx.build_aabbs(boxes, code_bits=30, leaf_order=1)
    assert a.nodes().tobytes() == b.nodes().tobytes()


@pytest.mark.parametrize("leaf", [0, 1])
def test_tree_memory_reused_across_threads_and_contexts(leaf):
    """Freed trees' memory goes to the next trees of about their size.  Four
    threads with a context each build, trace and free trees whose sizes hand
    the blocks around; every node array and hit equals the oracle's, and a
    tree outlives the context that built it."""
    import threading
    sizes = [2, 3000, 2900, 4097, 70001, 3500, 65536, 2]
    rays = W.primary_rays(12, 8)
    want = {}
    for n in set(sizes):
        tri = W.make_triangles(W.cluster_vertices(5000 + n, n))
        nodes, _, _, _ = oracle.build(tri, 30, leaf)
        want[n] = (tri, nodes, oracle.trace(nodes, tri, rays, 0)) if leaf else (tri, nodes, None)
    bad = []

    def work(k):
        c = lbvh_amd.Context(0)
        left = None
        for r in range(3):
            for n in sizes[k:] + sizes[:k]:
                tri, nodes, hits = want[n]
                bvh = c.build_triangles(tri, code_bits=30, leaf_order=leaf)
                if bvh.nodes().tobytes() != nodes.tobytes():
                    bad.append((k, r, n, "nodes"))
                if hits is not None:
                    p, t, _ = c.trace(bvh, rays, 0)
                    if not (np.array_equal(p, hits[0]) and
                            np.array_equal(t.view(np.uint32), hits[1].view(np.uint32))):
                        bad.append((k, r, n, "hits"))
                left = bvh # the previous one is freed here
        c.close()
        left.destroy()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad


def test_trim_gives_kept_memory_back(ctx):
    """A freed tree's memory stays with the engine until it is trimmed."""
    from lbvh_amd import hip
    lbvh_amd.trim_memory()
    before = hip.mem_info()[0]
    tree = ctx.build_triangles(W.make_triangles(W.uniform_vertices(1, 1500000, 0.01)))
    held = tree.info().device_bytes
    tree.destroy()
    kept = hip.mem_info()[0]
    lbvh_amd.trim_memory()
    assert hip.mem_info()[0] - kept >= held
    assert kept <= before - held
    with pytest.raises(lbvh_amd.LbvhError):
        lbvh_amd.trim_memory(-1)


@pytest.mark.parametrize("mode", [0, 1, 2], ids=["global", "thread-local", "relaxed"])
@pytest.mark.parametrize("other_thread", [False, True], ids=["same-thread", "other-thread"])
def test_captures_survive_frees_and_stream_waits(ctx, mode, other_thread):
    """Destroying a tree and ordering a context after a stream leave a graph
    capture valid, in any capture mode and from any thread."""
    import ctypes
    import threading
    from lbvh_amd.hip import DeviceArray, check, hip
    P = ctypes.c_void_p
    L = hip()
    trees = [ctx.build_triangles(W.scene_uniform(1, n, 0.01)[1]) for n in (3000, 70001)]
    a, b = (DeviceArray.from_host(np.full(4096, v, np.uint32)) for v in (1, 2))
    cap, idle, graph, run = P(), P(), P(), P()
    for s in (cap, idle):
        check(L.hipStreamCreateWithFlags(ctypes.byref(s), 1), "stream")

    def copy():
        return L.hipMemcpyAsync(P(b.ptr), P(a.ptr), ctypes.c_size_t(16384), 3, cap)

    def disturb():
        for t in trees:
            t.destroy()
        ctx._check(lbvh_amd.lib().lbvh_ctx_wait_stream(ctx.handle, idle))

    print("capture mode=%d other_thread=%d" % (mode, other_thread), flush=True)
    check(L.hipStreamBeginCapture(cap, mode), "begin")
    rc = [copy()]
    if other_thread:
        t = threading.Thread(target=disturb)
        t.start()
        t.join()
    else:
        disturb()
    rc.append(copy())
    rc.append(L.hipStreamEndCapture(cap, ctypes.byref(graph)))
    assert rc == [0, 0, 0]
    check(L.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)), "graph")
    check(L.hipGraphLaunch(run, cap), "launch")
    check(L.hipStreamSynchronize(cap), "sync")
    assert (b.numpy() == 1).all()
    check(L.hipGraphExecDestroy(run), "destroy")
    check(L.hipGraphDestroy(graph), "destroy")
    for s in (cap, idle):
        check(L.hipStreamDestroy(s), "destroy")


def test_reported_bytes_are_those_held():
    """device_bytes counts the whole block that a tree took from a freed one,
    and its host-built triangles'."""
    c = lbvh_amd.Context(0)
    held = []
    for n in (61234, 60987, 30000):  # no other test's block lies between the first two
        bvh = c.build_triangles(W.make_triangles(W.uniform_vertices(n, n, 0.01)))
        held.append(bvh.info().device_bytes)
        bvh.destroy()
    assert held[1] == held[0] >= 61234 * (48 + 48)
    assert 30000 * (48 + 48) <= held[2] < held[0] // 2 + 65536
    c.close()


def test_phase_timing_reports_four_phases(ctx):
    v, tri = W.scene_uniform(1, 65536, 0.01)
    ctx.set_timing(True)
    bvh = ctx.build_triangles(tri, code_bits=30)
    ms = ctx.phase_ms()
    ctx.set_timing(False)
    assert len(ms) == 4 and all(x >= 0 for x in ms)


def test_autotuner_times_candidates_and_keeps_results_exact():
    """A fresh context tunes the sort on the first build of a size bucket:
    every candidate is timed, one is kept, and the tree equals the oracle's
    whatever configuration was picked."""
    c = lbvh_amd.Context(0)
    v = W.cluster_vertices(91, 200000)
    tri = W.make_triangles(v)
    bvh = c.build_triangles(tri, code_bits=63, leaf_order=1, keep_codes=True)
    log = c.tune_log()
    # 4 configurations each of reduce-then-scan, onesweep and the hybrid
    assert len(log) == 12 and all(r["ms"] > 0 for r in log)
    picked = [r for r in log if r["picked"]]
    assert len(picked) == 1
    inf = bvh.info()
    assert inf.sort_digit_bits == picked[0]["digit_bits"]
    assert inf.sort_tile == picked[0]["tile"]
    on, _, osc, oids = oracle.build(tri, 63, 1)
    assert bvh.nodes().tobytes() == on.tobytes()
    sc, ids, _ = bvh.codes()
    assert np.array_equal(sc, osc) and np.array_equal(ids, oids)
    # the same bucket again: no new tuning
    bvh2 = c.build_triangles(tri, code_bits=63, leaf_order=1)
    assert len(c.tune_log()) == 12
    assert bvh2.info().sort_tile == inf.sort_tile
    # a batch of the same size tunes its own candidates (no onesweep)
    sizes = W.loguniform_sizes(5, 64, 1000, 8000)
    btri, off = W.batched_scenes(seed=5, sizes=sizes)
    b = c.build_batch(btri, off, leaf_order=1)
    blog = [r for r in c.tune_log() if r["batch"]]
    assert len(blog) == 8 and sum(r["picked"] for r in blog) == 1
    for s in (0, 31, 63):
        on, _, _, _ = oracle.build(btri[int(off[s]):int(off[s + 1])], 30, 1)
        assert b.nodes(s).tobytes() == on.tobytes()
    # explicit options bypass the tuner
    c.set_autotune(False)
    bvh3 = c.build_triangles(W.make_triangles(W.cluster_vertices(92, 1 << 19)), code_bits=30)
    assert len(c.tune_log()) == 20
    assert bvh3.info().sort_strategy in (1, 2, 3)
    for x in (bvh, bvh2, bvh3, b):
        x.destroy()
    c.close()


def test_traversal_tuner_records_each_mode_and_keeps_results_exact():
    """The first traversal of a (mode, ray-count) bucket times every
    traversal configuration (rays as given or in key order, x 8, 6 or 4
    waves per SIMD) on its own rays; each mode is tuned apart, exactly one
    configuration is kept per bucket, and the hits equal the oracle's on the
    tuning call and on the calls that reuse the choice."""
    c = lbvh_amd.Context(0)
    tri = W.make_triangles(W.cluster_vertices(93, 100000))
    bvh = c.build_triangles(tri, code_bits=63, leaf_order=1)
    on, _, _, _ = oracle.build(tri, 63, 1)
    rays = W.primary_rays(256, 256)
    for mode in (0, 2):
        want = oracle.trace(on, tri, rays, mode)
        for _ in range(2):
            p, t, uv = c.trace(bvh, rays, mode)
            assert np.array_equal(p, want[0])
            if mode == 0:
                assert np.array_equal(t.view(np.uint32), want[1].view(np.uint32))
                assert np.array_equal(uv.view(np.uint32), want[2].view(np.uint32))
    log = [r for r in c.tune_log() if r["kind"] == "traversal"]
    assert len(log) == 12
    for mode in (0, 2):
        mine = [r for r in log if r["mode"] == mode]
        assert len(mine) == 6 and all(r["ms"] > 0 and r["log2_n"] == 16 for r in mine)
        assert sum(r["picked"] for r in mine) == 1
        assert sorted((r["reorder"], r["waves_per_simd"]) for r in mine) == \
            sorted((ro, w) for ro in (False, True) for w in (8, 6, 4))
    bvh.destroy()
    c.close()


@pytest.mark.parametrize("n", [2, 3, 5, 64])
@pytest.mark.parametrize("leaf", [0, 1], ids=["ref", "pid"])
def test_trace_edge_rays_match_oracle(ctx, n, leaf):
    """Tiny trees and degenerate rays (axis-aligned, in a triangle's plane,
    NaN and infinite components, tmin > tmax, zero direction) in every
    intersector mode: ids, t and uv equal the oracle's bit for bit."""
    from test_oracle import edge_rays32
    tri = W.make_triangles(W.uniform_vertices(80 + n, n, 0.2))
    bvh = ctx.build_triangles(tri, code_bits=30, leaf_order=leaf)
    on, _, _, _ = oracle.build(tri, 30, leaf)
    assert bvh.nodes().tobytes() == on.tobytes()
    rays = edge_rays32(tri)
    for mode in (0, 1, 2):
        p, t, uv = ctx.trace(bvh, rays, mode)
        op, ot, ouv = oracle.trace(on, tri, rays, mode)
        assert np.array_equal(p, op), "mode %d ids" % mode
        assert np.array_equal(t.view(np.uint32), ot.view(np.uint32)), "mode %d t" % mode
        assert np.array_equal(uv.view(np.uint32), ouv.view(np.uint32)), "mode %d uv" % mode
    bvh.destroy()
